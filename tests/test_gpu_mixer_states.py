"""mixer_read's chunk-boundary states walked sequence by sequence against formed
chunk by chunk and carried: the gates, the shifted and normalised keys and the
read gate's weights enter both, and every result is the same bits."""

import pytest
import torch

from tests.gpu_helpers import announce

pytestmark = pytest.mark.gpu


# (T, P, chunk, key shift, cached key, initial state): whole and ragged chunks,
# one value tile and two, chunks of one and of two sub-chunks.
@pytest.mark.parametrize("time,width,chunk,shift,cached,initial", [
    (300, 64, 64, True, False, False), (257, 128, 64, True, True, True),
    (130, 64, 20, False, False, True), (64, 128, 48, True, False, True), (5, 64, 64, True, True, False),
    (400, 128, 5, True, True, True)])  # more than 64 steps in the carries
def test_walked_and_carried_states_agree(gpu_lib, monkeypatch, time, width, chunk, shift, cached,
                                         initial):
    import mamba4_amd as m4
    from mamba4_amd import _lib

    batch, heads = 2, 3
    gen = torch.Generator(device="cuda")
    gen.manual_seed(time)

    def normal(*shape):
        return torch.randn(*shape, device="cuda", generator=gen)

    x = [normal(batch, time, heads, 64), normal(batch, time, heads, width),
         normal(batch, time, heads, 64), normal(batch, time, heads),
         normal(batch, time, heads) - 2.0, normal(heads), normal(heads) - 2.0,
         0.3 * normal(heads), normal(heads, 64), normal(heads).abs(), normal(heads)]
    previous = normal(batch, heads, 64) if cached else None
    state = None
    if initial:
        half = normal(batch, heads, 64, 16)
        state = m4.SelectiveState(torch.matmul(half, half.transpose(-1, -2).contiguous()) / 16,
                                  normal(batch, heads, width, 64))
    cot = [normal(batch, time, heads, width), normal(batch, time, heads),
           normal(batch, heads, 64, 64), normal(batch, heads, width, 64)]

    def run(mode):
        monkeypatch.setenv("M4MR_STATE_WALK", mode)
        _lib.profile_reset()
        _lib.profile_select(None)
        _lib.profile_enable(True)
        leaves = [t.clone().requires_grad_(True) for t in x]
        extra = [t.clone().requires_grad_(True) for t in (state or ())]
        if cached:
            extra.append(previous.clone().requires_grad_(True))
        r = m4.mixer_read(*leaves, key_shift=shift, chunk_size=chunk,
                          previous=extra[-1] if cached else None,
                          initial=m4.SelectiveState(*extra[:2]) if initial else None)
        out = [r.output, r.variance, r.state.evidence, r.state.cross]
        grads = torch.autograd.grad(out, leaves + extra, cot)
        torch.cuda.synchronize()
        _lib.profile_enable(False)
        ran = [_lib.profile_read(n)[1] for n in ("fwd_states", "bwd_states", "fwd_stats",
                                                 "fwd_scan", "bwd_local", "bwd_scan")]
        _lib.profile_reset()
        assert ran == ([1, 1, 0, 0, 0, 0] if mode == "fused" else [0, 0, 1, 1, 1, 1])
        shifted = [] if r.shifted is None else [r.shifted.detach()]
        return [t.detach() for t in out] + shifted + list(grads)

    announce(f"mixer states T={time} P={width} chunk={chunk} shift={shift}")
    walked, carried = run("fused"), run("split")
    for i, (a, b) in enumerate(zip(walked, carried)):
        assert torch.equal(a, b), i
