"""The factor kernel's token spans: a small batch splits each sub-chunk into
spans whose evidence is brought up from the sub-chunk's start state, a full
chip walks whole sub-chunks.  Both apply the same updates in the same order,
so a batch row has the same bits in either, from states that the small batch
forms chunk by chunk and the large one walks."""

import pytest
import torch

from tests.gpu_helpers import announce

pytestmark = pytest.mark.gpu


# (time, chunk): whole and ragged 64-token chunks, sub-chunks of 24 (the
# last spans empty) and of 20 tokens, chunks shorter than a span count.
@pytest.mark.parametrize("time,chunk", [(1024, 64), (1013, 64), (1000, 48), (1001, 20), (500, 5)])
@pytest.mark.parametrize("mixer", [False, True])
def test_spans_give_the_whole_walks_bits(gpu_lib, time, chunk, mixer):
    import mamba4_amd as m4
    from mamba4_amd import memory

    batch, heads, row = 16, 8, 5
    gen = torch.Generator(device="cuda")
    gen.manual_seed(time + chunk)

    def normal(*shape):
        return torch.randn(*shape, device="cuda", generator=gen)

    k, q, v = (normal(batch, time, heads, 64) for _ in range(3))
    beta, decay = normal(batch, time, heads), normal(batch, time, heads) - 2.0
    floor = normal(heads, 64)

    def run(first, last):
        part = [t[first:last].contiguous() for t in (k, v, q, beta, decay)]
        if mixer:
            per_head = [torch.full((heads,), x, device="cuda") for x in (0.0, 0.0, 0.0, 0.5, 1.0)]
            with torch.no_grad():
                r = m4.mixer_read(*part, *per_head[:3], floor, *per_head[3:], chunk_size=chunk)
            return [r.output, r.variance]
        unit = [t / t.norm(dim=-1, keepdim=True) for t in (part[0], part[2])]
        out = memory.memread_forward(unit[0], part[1], unit[1], torch.sigmoid(part[3]),
                                     -torch.exp(part[4]), floor.abs() + 0.1, None, None, chunk)
        return [out[0], out[1], out[4], out[5]]

    announce(f"factor spans T={time} chunk={chunk} mixer={mixer}")
    whole = run(0, batch)
    small = run(row, row + 1)
    torch.cuda.synchronize()
    for i, (a, b) in enumerate(zip(whole, small)):
        assert torch.equal(a[row], b[0]), i


# (time, P): ragged chunks, and more than 64 steps in the carries (40 chunks of
# two sub-chunks).
@pytest.mark.parametrize("time,width", [(700, 128), (2500, 64)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_a_row_has_the_same_bits_at_any_batch_size(gpu_lib, dtype, time, width):
    """Memory read, forward and backward: alone, a row's states are formed chunk
    by chunk and its sub-chunks split into spans; in the batch its states are
    walked."""
    import mamba4_amd as m4
    from mamba4_amd import _lib

    batch, heads, row = 32, 4, 11
    gen = torch.Generator(device="cuda")
    gen.manual_seed(time)

    def normal(*shape):
        return torch.randn(*shape, device="cuda", generator=gen)

    def unit(*shape):
        x = normal(*shape)
        return x / x.norm(dim=-1, keepdim=True)

    half = normal(batch, heads, 64, 16)
    x = [unit(batch, time, heads, 64).to(dtype), normal(batch, time, heads, width).to(dtype),
         unit(batch, time, heads, 64).to(dtype), torch.sigmoid(normal(batch, time, heads)),
         -torch.exp(normal(batch, time, heads) - 3.0),
         torch.matmul(half, half.transpose(-1, -2).contiguous()) / 16,
         normal(batch, heads, width, 64)]
    floor = normal(heads, 64).abs() + 0.1
    cot = [normal(batch, time, heads, width), normal(batch, time, heads),
           normal(batch, heads, 64, 64), normal(batch, heads, width, 64)]

    def run(rows):
        leaves = [t[rows].clone().requires_grad_(True) for t in x]
        _lib.profile_reset()
        _lib.profile_select(None)
        _lib.profile_enable(True)
        try:
            r = m4.selective_gaussian_memory(*leaves[:5], floor,
                                             initial=m4.SelectiveState(*leaves[5:]))
            out = [r.output, r.variance, r.state.evidence, r.state.cross]
            grads = torch.autograd.grad(out, leaves, [c[rows] for c in cot])
            torch.cuda.synchronize()
        finally:
            _lib.profile_enable(False)
        walks = [_lib.profile_read(n)[1] for n in ("fwd_states", "bwd_states", "fwd_scan",
                                                   "bwd_scan")]
        _lib.profile_reset()
        return walks, [t.detach() for t in out] + list(grads)

    announce(f"row bits, memory read B{batch} T{time} H{heads} P{width} {dtype}")
    walks, many = run(slice(0, batch))
    carries, one = run(slice(row, row + 1))
    assert walks == [1, 1, 0, 0] and carries == [0, 0, 1, 1]
    for i, (a, b) in enumerate(zip(many, one)):
        assert torch.equal(a[row], b[0]), i
