"""drone_gcn_mod::GCN as a C++ program sees it (include/drone_gcn_modules.hpp): the state behind set_truth(), forward() and
metrics_async() that such a program reads, changes and passes on - truth_split, truth_count, ce->grad_scale, counts, l2_sum,
ce->d_loss.  The program is compiled by the host compiler against the library."""
import os
import shutil
import subprocess

import pytest

from drone_amd import _lib

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
ROCM = os.environ.get("ROCM_PATH", "/opt/rocm")

PROGRAM = r"""
#include <cmath>
#include <type_traits>

#include "drone_gcn_modules.hpp"

using drone_gcn_mod::GCN;
static_assert(std::is_same<decltype(GCN::truth_split), int>::value && std::is_same<decltype(GCN::truth_count), int>::value, "host numbers");
static_assert(std::is_same<decltype(GCN::counts), int *>::value && std::is_same<decltype(GCN::l2_sum), float *>::value, "arrays");
static_assert(std::is_same<decltype(&GCN::metrics_async), void (GCN::*)()>::value && std::is_same<decltype(&GCN::set_truth), void (GCN::*)(int)>::value, "calls");

template <typename T> T *up(const std::vector<T> &h)
{
    T *d = nullptr;
    DRONE_GCN_HIP(hipMalloc(&d, sizeof(T) * h.size()));
    DRONE_GCN_HIP(hipMemcpy(d, h.data(), sizeof(T) * h.size(), hipMemcpyHostToDevice));
    return d;
}
template <typename T> std::vector<T> down(const T *d, size_t n)
{
    std::vector<T> h(n);
    DRONE_GCN_HIP(hipDeviceSynchronize());
    DRONE_GCN_HIP(hipMemcpy(h.data(), d, sizeof(T) * n, hipMemcpyDeviceToHost));
    return h;
}
int failed = 0;
#define CHECK(cond) do { if (!(cond)) { printf("line %d: %s\n", __LINE__, #cond); failed = 1; } } while (0)

int main()
{
    const int N = 300, fin = 20, hid = 8, cls = 5;
    std::vector<int> rp(N + 1), ci, deg(N), label(N), split(N);
    for (int v = 0; v < N; ++v) {
        rp[v] = (int)ci.size();
        for (int d : {0, 1, 7}) ci.push_back((v + d) % N);
        deg[v] = 3;
        label[v] = v * 7 % cls;
        split[v] = v % 3 ? 1 : 2;
    }
    rp[N] = (int)ci.size();
    const int ones = 200, twos = 100;
    std::vector<float> X(N * fin), W1(fin * hid), W2(hid * cls);
    for (size_t i = 0; i < X.size(); ++i) X[i] = std::sin(0.37f * i);
    for (size_t i = 0; i < W1.size(); ++i) W1[i] = 0.3f * std::cos(0.91f * i);
    for (size_t i = 0; i < W2.size(); ++i) W2[i] = 0.3f * std::sin(1.7f * i);
    drone_gcn_mod::GCNParams p;
    p.localVertexSize = N; p.input_dim = fin; p.hidden_dim = hid; p.output_dim = cls;
    p.use_adam = false; p.mean_gradient = true; p.learning_rate = 0.0f;
    hipStream_t s;
    DRONE_GCN_HIP(hipStreamCreate(&s));
    GCN m(p, (int64_t)ci.size(), up(rp), up(ci), up(deg), up(deg), up(X), fin, up(label), up(split), up(W1), up(W2), s);

    // set_truth: the split and the number of its labelled rows are there when it returns, and so is the gradient's scale
    m.set_truth(1);
    CHECK(m.truth_split == 1 && m.truth_count == ones && m.ce->grad_scale == 1.0f / ones);
    m.set_truth(2);
    CHECK(m.truth_split == 2 && m.truth_count == twos && m.ce->grad_scale == 1.0f / twos);
    m.set_truth(7);
    CHECK(m.truth_count == 0 && m.ce->grad_scale == 1.0f);
    m.set_truth(1);

    // forward: counts and l2_sum hold this pass's numbers in the stream's order
    m.forward(true);
    const int ld = m.output->ld;
    const std::vector<float> z = down(m.output->data, (size_t)N * ld), grad = down(m.output->grad, (size_t)N * ld);
    int correct[3] = {0, 0, 0}, rows[3] = {0, 0, 0};
    for (int v = 0; v < N; ++v) {
        bool right = true;
        for (int c = 0; c < cls; ++c) right = right && !(z[v * ld + c] > z[v * ld + label[v]]);
        rows[split[v]]++;
        correct[split[v]] += right;
    }
    double squares = 0.0;
    for (float w : W1) squares += (double)w * w;
    std::vector<int> counts = down(m.counts, 2);
    CHECK(counts[0] == correct[1] && counts[1] == ones && rows[1] == ones);
    CHECK(std::fabs(down(m.l2_sum, 1)[0] - squares) <= 1e-6 * squares);
    const float loss = down(m.ce->d_loss, 1)[0];
    auto r = m.read_metrics();
    CHECK(r.second == (float)correct[1] / ones && r.first == loss + p.weight_decay * down(m.l2_sum, 1)[0] / 2);

    // a scale that the program sets holds until the split changes
    m.ce->grad_scale = 0.5f;
    m.set_truth(1);
    m.forward(true);
    const std::vector<float> scaled = down(m.output->grad, (size_t)N * ld);
    for (int v = 0; v < N; ++v)
        for (int c = 0; c < cls; ++c) CHECK(std::fabs(scaled[v * ld + c] - 0.5f * ones * grad[v * ld + c]) <= 1e-6f);
    m.set_truth(2);
    m.set_truth(1);
    m.forward(true);
    CHECK(down(m.output->grad, (size_t)N * ld) == grad);

    // metrics_async: the numbers of the logits, truth and weights as they are now; the loss is still the pass's
    m.set_truth(2);
    DRONE_GCN_HIP(hipMemset(m.layer1_weight->data, 0, m.layer1_weight->bytes()));
    DRONE_GCN_HIP(hipDeviceSynchronize());
    m.metrics_async();
    r = m.read_metrics();
    counts = down(m.counts, 2);
    CHECK(counts[0] == correct[2] && counts[1] == twos && r.first == loss && down(m.l2_sum, 1)[0] == 0.0f);
    CHECK(r.second == (float)correct[2] / twos);
    DRONE_GCN_HIP(hipMemcpy(m.layer1_weight->data, W1.data(), sizeof(float) * W1.size(), hipMemcpyHostToDevice));

    // what the program puts there (a sum over workers, say) is what read_metrics reports
    const int summed[2] = {3, 4};
    const float mean = 2.5f, none = 0.0f;
    DRONE_GCN_HIP(hipMemcpy(m.counts, summed, sizeof summed, hipMemcpyHostToDevice));
    DRONE_GCN_HIP(hipMemcpy(m.l2_sum, &none, sizeof none, hipMemcpyHostToDevice));
    DRONE_GCN_HIP(hipMemcpy(m.ce->d_loss, &mean, sizeof mean, hipMemcpyHostToDevice));
    r = m.read_metrics();
    CHECK(r.first == mean && r.second == 0.75f);

    // epochs and evaluations: the same state behind each of them, and the same gradient as with set_truth
    r = m.train_epoch();
    CHECK(m.truth_split == 1 && m.truth_count == ones && m.ce->grad_scale == 1.0f / ones && r.second == (float)correct[1] / ones);
    CHECK(down(m.output->grad, (size_t)N * ld) == grad);
    r = m.eval(2);
    CHECK(m.truth_split == 2 && m.truth_count == twos && m.ce->grad_scale == 1.0f / twos && r.second == (float)correct[2] / twos);

    // a captured set_truth to another split takes the scale from the device at every replay
    hipGraph_t graph;
    hipGraphExec_t exec;
    DRONE_GCN_HIP(hipStreamBeginCapture(s, hipStreamCaptureModeThreadLocal));
    m.set_truth(1);
    m.forward(true);
    DRONE_GCN_HIP(hipStreamEndCapture(s, &graph));
    DRONE_GCN_HIP(hipGraphInstantiate(&exec, graph, nullptr, nullptr, 0));
    for (int k = 0; k < 3; ++k) {
        DRONE_GCN_HIP(hipGraphLaunch(exec, s));
        r = m.read_metrics();
        CHECK(r.second == (float)correct[1] / ones && down(m.output->grad, (size_t)N * ld) == grad);
        CHECK(k > 0 || (m.truth_count == ones && m.ce->grad_scale == 1.0f / ones));  // (a replay is nothing the host sees)
        DRONE_GCN_HIP(hipMemset(m.output->grad, 0, sizeof(float) * (size_t)N * ld));
        m.eval(2);
    }
    DRONE_GCN_HIP(hipGraphExecDestroy(exec));
    DRONE_GCN_HIP(hipGraphDestroy(graph));
    if (!failed) printf("all as expected\n");
    fflush(stdout);
    return failed;
}
"""


# Programs that put their own modules and optimisers into a model, also at the addresses of the model's own.
REPLACED = r"""
#include <cmath>
#include <new>

#include "drone_gcn_modules.hpp"

using namespace drone_gcn_mod;

template <typename T> T *up(const std::vector<T> &h)
{
    T *d = nullptr;
    DRONE_GCN_HIP(hipMalloc(&d, sizeof(T) * h.size()));
    DRONE_GCN_HIP(hipMemcpy(d, h.data(), sizeof(T) * h.size(), hipMemcpyHostToDevice));
    return d;
}
std::vector<float> down(const Variable *v, const float *d)
{
    std::vector<float> h((size_t)v->rows * v->ld);
    DRONE_GCN_HIP(hipDeviceSynchronize());
    DRONE_GCN_HIP(hipMemcpy(h.data(), d, sizeof(float) * h.size(), hipMemcpyDeviceToHost));
    return h;
}
int failed = 0;
#define CHECK(cond) do { if (!(cond)) { printf("line %d: %s\n", __LINE__, #cond); failed = 1; } } while (0)

// Reads both weights' gradients, and steps by a rate of 0.
std::vector<float> seen1, seen2;
struct Reader : Optimizer {
    Variable *w1, *w2;
    char as_large_as_the_models_own[sizeof(SGD) - sizeof(Optimizer) - 2 * sizeof(Variable *)];
    Reader(Variable *a, Variable *b) : w1(a), w2(b) {}
    void step() override { seen1 = down(w1, w1->grad); seen2 = down(w2, w2->grad); }
};
static_assert(sizeof(Reader) == sizeof(SGD), "finds a place where one was");
// The same in the backward pass, in front of layer 1.
struct Last : Module {
    Variable *w2;
    explicit Last(Variable *w) : w2(w) {}
    void forward(bool) override {}
    void backward() override { seen2 = down(w2, w2->grad); }
};

int main()
{
    const int N = 3000, fin = 64, hid = 32, cls = 7;
    std::vector<int> rp(N + 1), ci, deg(N, 3), label(N), split(N);
    for (int v = 0; v < N; ++v) {
        rp[v] = (int)ci.size();
        for (int d : {0, 1, 7}) ci.push_back((v + d) % N);
        label[v] = v * 5 % cls;
        split[v] = v % 3 ? 1 : 2;
    }
    rp[N] = (int)ci.size();
    std::vector<float> X(N * fin), W1(fin * hid), W2(hid * cls);
    for (size_t i = 0; i < X.size(); ++i) X[i] = std::sin(0.37f * i);
    for (size_t i = 0; i < W1.size(); ++i) W1[i] = 0.3f * std::cos(0.91f * i);
    for (size_t i = 0; i < W2.size(); ++i) W2[i] = 0.3f * std::sin(1.7f * i);
    GCNParams p;
    p.localVertexSize = N; p.input_dim = fin; p.hidden_dim = hid; p.output_dim = cls;
    p.use_adam = false; p.learning_rate = 0.0f;
    GCN m(p, (int64_t)ci.size(), up(rp), up(ci), up(deg), up(deg), up(X), fin, up(label), up(split), up(W1), up(W2), nullptr);
    Variable *const w1 = m.layer1_weight, *const w2 = m.layer2_weight;
    CHECK(w1->sums_floats > 0 && w2->sums_floats > 0);  // or nothing here is to be seen

    m.set_truth(1);
    m.forward(true);
    m.backward();
    const std::vector<float> g1 = down(w1, w1->grad), g2 = down(w2, w2->grad);
    const auto forget = [&] {
        for (Variable *w : {w1, w2}) DRONE_GCN_HIP(hipMemset(w->grad, 0, sizeof(float) * (size_t)w->rows * w->ld));
        seen1.clear();
        seen2.clear();
    };
    // as built: the step leaves the gradients that backward() alone leaves
    for (int way = 0; way < 2; ++way) {
        forget();
        if (way) m.train_epoch(); else m.train_step_async();
        CHECK(down(w1, w1->grad) == g1 && down(w2, w2->grad) == g2);
    }
    // a module of the program's that reads a gradient during the backward pass
    forget();
    m.modules.insert(m.modules.begin(), std::unique_ptr<Module>(new Last(w2)));
    m.train_epoch();
    CHECK(seen2 == g2 && down(w1, w1->grad) == g1);
    m.modules.erase(m.modules.begin());
    // another optimiser's variables in the model's own: it steps layer 1 alone, and the gradient of layer 2 is there for the program
    forget();
    static_cast<SGD &>(*m.optimizer) = SGD({w1}, 0.0f, nullptr);
    m.train_epoch();
    CHECK(down(w1, w1->grad) == g1 && down(w2, w2->grad) == g2);
    // optimisers of the program's, one after the other, until one has the place of the model's own
    const void *const place = m.optimizer.get();
    bool taken = false;
    for (int i = 0; i < 100 && !taken; ++i) {
        m.optimizer.reset(new Reader(w1, w2));
        taken = m.optimizer.get() == place;
        forget();
        m.train_step_async();
        CHECK(seen1 == g1 && seen2 == g2);
    }
    CHECK(taken);
    if (!failed) printf("all as expected\n");
    fflush(stdout);
    return failed;
}
"""


def _compile(tmp_path, *extra, program=PROGRAM):
    cxx = shutil.which("g++") or shutil.which("c++")
    assert cxx, "no C++ compiler"
    src = tmp_path / "modules.cpp"
    src.write_text(program)
    subprocess.check_call([cxx, "-std=c++17", "-O1", "-Wall", "-Wno-unused-result", "-D__HIP_PLATFORM_AMD__", "-I", os.path.join(ROOT, "include"),
                           "-isystem", os.path.join(ROCM, "include"), str(src), *extra])


def test_module_header_keeps_what_programs_use(tmp_path):
    _compile(tmp_path, "-fsyntax-only")


def _run(tmp_path, program):
    exe, lib = str(tmp_path / "modules"), _lib.library_path()
    _compile(tmp_path, "-o", exe, lib, "-Wl,-rpath," + os.path.dirname(lib), "-L" + os.path.join(ROCM, "lib"),
             "-Wl,-rpath," + os.path.join(ROCM, "lib"), "-lamdhip64", program=program)
    done = subprocess.run([exe], capture_output=True, text=True, timeout=100)
    assert done.returncode == 0 and "all as expected" in done.stdout, done.stdout + done.stderr


@pytest.mark.gpu
def test_state_behind_the_model(tmp_path):
    _run(tmp_path, PROGRAM)


def test_programs_may_replace_what_a_model_has_built_compile(tmp_path):
    _compile(tmp_path, "-fsyntax-only", program=REPLACED)


@pytest.mark.gpu
def test_programs_may_replace_what_a_model_has_built(tmp_path):
    """The gradients are there for a module or an optimiser that is not the model's own, also where it lives at its address."""
    _run(tmp_path, REPLACED)
