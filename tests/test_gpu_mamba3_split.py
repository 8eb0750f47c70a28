"""The Mamba-3 scan's chunk-boundary states formed in parallel and carried (few
sequences) against the walk (many): a batch row alone takes the first, in its
batch the second, with the same bits."""

import pytest
import torch

from tests.gpu_helpers import announce

pytestmark = pytest.mark.gpu

ROUTES = ("m3_walk", "m3_walk_bwd", "m3_local", "m3_carry", "m3_local_bwd", "m3_carry_bwd")


# (T, N, P, A): whole and ragged chunks; odd counts of angles (element loads),
# none, one per coordinate pair; narrow and odd widths.
@pytest.mark.parametrize("dtype,tolerance", [(torch.float32, 5e-6), (torch.bfloat16, 1e-3)])
@pytest.mark.parametrize("time,state,width,angles", [(300, 128, 64, 32), (320, 30, 9, 7),
                                                     (257, 62, 33, 0), (400, 128, 64, 64),
                                                     (449, 16, 8, 3), (1100, 128, 48, 36)])
def test_split_states_match_the_walk(gpu_lib, time, state, width, angles, dtype, tolerance):
    from mamba4_amd import _lib, mamba3_fused

    batch, heads, row = 16, 24, 11
    gen = torch.Generator(device="cuda")
    gen.manual_seed(time + state)

    def normal(*shape):
        return torch.randn(*shape, device="cuda", generator=gen)

    dt = torch.nn.functional.softplus(normal(batch, time, heads) - 1.0)
    x = [normal(batch, time, state).to(dtype), normal(batch, time, state).to(dtype),
         normal(batch, time, heads * width).to(dtype), -dt * normal(batch, time, heads).abs(), dt,
         normal(batch, time, heads), normal(batch, time, angles)]
    bias = [0.1 * normal(heads, 1, state), 0.1 * normal(heads, 1, state)]
    d_y, d_final = normal(batch, time, heads * width).to(dtype), normal(batch, heads, state, width)

    def run(rows):
        leaves = [t[rows].clone().requires_grad_(True) for t in x]
        _lib.profile_reset()
        _lib.profile_select(None)
        _lib.profile_enable(True)
        try:
            y, final = mamba3_fused(*leaves, q_bias=bias[0], k_bias=bias[1])
            grads = torch.autograd.grad([y, final], leaves if angles else leaves[:6],
                                        [d_y[rows], d_final[rows]])
            torch.cuda.synchronize()
        finally:
            _lib.profile_enable(False)
        launches = [_lib.profile_read(n)[1] for n in ROUTES]
        _lib.profile_reset()
        return launches, [y.detach(), final.detach(), *grads]

    announce(f"Mamba-3 split states T={time} N={state} P={width} A={angles} {dtype}")
    walks, many = run(slice(0, batch))
    splits, one = run(slice(row, row + 1))
    assert walks == [1, 1, 0, 0, 0, 0] and splits == [0, 0, 1, 1, 1, 1]
    # The shared rows' gradients (c, b, angles) are summed over groups of heads
    # that the batch size chooses: they agree to rounding, one of some thousands
    # of bfloat16 ones turned by it.  Everything else is equal to the bit.
    names = ["y", "final", "c", "b", "x", "adt", "dt", "trap", "angles"]
    for name, a, b in zip(names, many, one):
        if name in ("c", "b", "angles"):
            a, b = a[row].double(), b[0].double()
            assert (a - b).norm() <= tolerance * a.norm(), name
        else:
            assert torch.equal(a[row], b[0]), name


# A call of up to four chunks is bound by its launches: one walk, not three.
@pytest.mark.parametrize("time,split", [(1, False), (192, False), (256, False), (257, True)])
def test_short_sequences_are_walked(gpu_lib, time, split):
    from mamba4_amd import _lib, mamba3_fused

    gen = torch.Generator(device="cuda")
    gen.manual_seed(time)

    def normal(*shape):
        return torch.randn(*shape, device="cuda", generator=gen)

    heads, state, width, angles = 4, 128, 64, 32
    announce(f"Mamba-3 short sequence T={time}")
    _lib.profile_reset()
    _lib.profile_select(None)
    _lib.profile_enable(True)
    try:
        mamba3_fused(normal(1, time, state), normal(1, time, state), normal(1, time, heads * width),
                     -normal(1, time, heads).abs(), normal(1, time, heads).abs(),
                     normal(1, time, heads), normal(1, time, angles),
                     q_bias=normal(heads, 1, state), k_bias=normal(heads, 1, state))
        torch.cuda.synchronize()
    finally:
        _lib.profile_enable(False)
    launches = [_lib.profile_read(n)[1] for n in ("m3_walk", "m3_local", "m3_carry")]
    _lib.profile_reset()
    assert launches == ([0, 1, 1] if split else [1, 0, 0])
