"""The factor kernel's token spans: a small batch splits each sub-chunk into
spans whose evidence is brought up from the sub-chunk's start state, a full
chip walks whole sub-chunks.  Both apply the same updates in the same order,
so a batch row has the same bits in either; the state walk is forced to its
fused form, as the two forms sum in different orders."""

import pytest
import torch

from tests.gpu_helpers import announce

pytestmark = pytest.mark.gpu


# (time, chunk): whole and ragged 64-token chunks, sub-chunks of 24 (the
# last spans empty) and of 20 tokens, chunks shorter than a span count.
@pytest.mark.parametrize("time,chunk", [(1024, 64), (1013, 64), (1000, 48), (1001, 20), (500, 5)])
@pytest.mark.parametrize("mixer", [False, True])
def test_spans_give_the_whole_walks_bits(gpu_lib, monkeypatch, time, chunk, mixer):
    import mamba4_amd as m4
    from mamba4_amd import memory

    monkeypatch.setenv("M4MR_STATE_WALK", "fused")
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
