"""Arrays brought to and from the library's widths in one launch."""

import ctypes

import pytest
import torch
import torch.nn.functional as F

from tests.gpu_helpers import announce


def test_resize_refuses_bad_arrays():
    from mamba4_amd import _lib

    lib = _lib.load()
    one = _lib.ResizeArray(None, None, 1, 1, 4, 1, 8, 4, 0)
    for arrays, count in ((one, 0), (one, 9), (one, 1)):  # no array, too many, no pointers
        assert lib.m4mr_resize(ctypes.byref(arrays), count, None) == _lib.EINVAL
    for field, value in (("bytes", 8), ("outer", -1), ("dst_cols", -1)):
        bad = _lib.ResizeArray(1, 1, 1, 1, 4, 1, 8, 4, 0)
        setattr(bad, field, value)
        assert lib.m4mr_resize(ctypes.byref(bad), 1, None) == _lib.EINVAL


@pytest.mark.gpu
def test_resize_pads_and_cuts_like_torch(gpu_lib):
    from mamba4_amd.memory import _resized

    announce("resize of several arrays in one launch")
    gen = torch.Generator(device="cuda")
    gen.manual_seed(2)

    def normal(*shape, dtype=torch.float32):
        return torch.randn(*shape, device="cuda", generator=gen).to(dtype)

    a, b, c, d = normal(3, 5, 48), normal(2, 7, 33, dtype=torch.bfloat16), normal(4, 20, 13), normal(6)
    e, f, empty = normal(9, 64), normal(2, 3, 128, 64), normal(0, 5, 3)
    got = _resized((a, None, 64, 0), (b, None, 64, 0), (c, 64, 64, 0), (d, None, 64, 1),
                   (e, None, 1, 0), (f, 100, 48, 0), (empty, None, 64, 0), (None, 64, 64, 0),
                   (a, None, 48, 0))
    # Two-byte elements cut off: whole quads of columns, a ragged tail, and
    # rows that start off a quad's alignment.
    g, h = normal(5, 7, 64, dtype=torch.bfloat16), normal(3, 66, 70, dtype=torch.bfloat16)
    cut = _resized((g, None, 48, 0), (g, None, 33, 0), (g, None, 1, 0), (h, 65, 63, 0))
    torch.cuda.synchronize()
    for x, y in zip(cut, (g[..., :48], g[..., :33], g[..., :1], h[:, :65, :63])):
        assert x.is_contiguous() and x.dtype == y.dtype and torch.equal(x, y)
    want = [F.pad(a, (0, 16)), F.pad(b, (0, 31)), F.pad(c, (0, 51, 0, 44)),
            F.pad(d, (0, 58), value=1.0), e[:, :1], f[..., :100, :48], F.pad(empty, (0, 61))]
    for x, y in zip(got, want):
        assert x.is_contiguous() and x.dtype == y.dtype and torch.equal(x, y)
    assert got[7] is None and got[8] is a
