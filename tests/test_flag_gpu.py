"""Waiting by a word of pinned memory: whatever was enqueued before the wait is done behind it, short or long, on any stream."""
import ctypes as C

import pytest

pytestmark = pytest.mark.gpu


class Flag(C.Structure):
    _fields_ = [("word", C.c_void_p), ("raised", C.c_uint)]


@pytest.mark.parametrize("elements", [1, 1000, 1 << 20, 1 << 27])  # 2^27: longer than the word is looked at
def test_everything_before_the_wait_is_done(elements):
    import torch
    from drone_amd._lib import check, lib
    word = torch.zeros(16, dtype=torch.int32, pin_memory=True)
    flag = Flag(word.data_ptr(), 0)
    streams = [torch.cuda.Stream() for _ in range(2)]
    x = [torch.zeros(elements, device="cuda") for _ in streams]
    torch.cuda.synchronize()
    other = torch.cuda.Stream()
    for i in range(20):
        for s, v in zip(streams, x):
            with torch.cuda.stream(s):
                v.add_(1.0)
            check(lib().drone_flag_wait(C.byref(flag), s.cuda_stream))
            with torch.cuda.stream(other):  # not ordered behind s but by the wait
                seen = v.min(), v.max()
            other.synchronize()
            assert (float(seen[0]), float(seen[1])) == (i + 1, i + 1)
    assert int(word[0]) == flag.raised == 40
