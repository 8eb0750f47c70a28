"""The decode step's forms: a few states (eight waves each four) and many (one
wave), from a state to a new one or in place, give the same bits."""

import pytest
import torch

from tests.gpu_helpers import announce

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("value_dim", [64, 128])
def test_few_states_give_the_bits_of_many(gpu_lib, value_dim):
    import mamba4_amd as m4

    batch, heads = 351, 3  # 1,053 states: one wave per four; a few rows: eight
    gen = torch.Generator(device="cuda")
    gen.manual_seed(value_dim)

    def normal(*shape):
        return torch.randn(*shape, device="cuda", generator=gen)

    half = normal(batch, heads, 64, 16)
    state = m4.SelectiveState(torch.matmul(half, half.transpose(-1, -2).contiguous()),
                              normal(batch, heads, value_dim, 64))
    token = [normal(batch, heads, 64), normal(batch, heads, value_dim), normal(batch, heads, 64),
             torch.sigmoid(normal(batch, heads)), -normal(batch, heads).abs()]
    floor = normal(heads, 64).abs() + 0.1
    before = [t.clone() for t in state]
    announce(f"decode forms P={value_dim}")
    many = m4.selective_decode(state, *token, floor)
    torch.cuda.synchronize()
    for a, b in zip(state, before):  # the old state is left as it was
        assert torch.equal(a, b)
    # 1, 3 (a partial block) and 5 batch rows; the states also at an address
    # that is no multiple of 16, as a view of another tensor may be.
    for rows, skew in ((1, 0), (3, 1), (5, 3)):
        part = []
        for t in state:
            flat = torch.zeros(t[:rows].numel() + skew, device="cuda")
            flat[skew:] = t[:rows].reshape(-1)
            part.append(flat[skew:].view(t[:rows].shape))
        few = m4.selective_decode(m4.SelectiveState(*part), *(t[:rows] for t in token), floor)
        own = m4.SelectiveState(*(t[:rows].clone() for t in state))
        placed = m4.selective_decode_(own, *(t[:rows] for t in token), floor)
        torch.cuda.synchronize()
        for r in (few, placed):
            for a, b in zip((r.output, r.variance, *r.state),
                            (many.output, many.variance, *many.state)):
                assert torch.equal(a, b[:rows]), (rows, skew)
        assert placed.state.evidence is own.evidence


def test_narrow_decode_leaves_the_state_and_matches_padding(gpu_lib):
    """D = 64 with P = 40 pads the cross state alone; D = 20 pads both."""
    import torch.nn.functional as F

    import mamba4_amd as m4

    gen = torch.Generator(device="cuda")
    gen.manual_seed(9)
    for dim, width in ((64, 40), (20, 64), (20, 100)):
        half = torch.randn(2, 3, dim, 8, device="cuda", generator=gen)
        s = torch.matmul(half, half.transpose(-1, -2).contiguous())
        c = torch.randn(2, 3, width, dim, device="cuda", generator=gen)
        k, q = (torch.randn(2, 3, dim, device="cuda", generator=gen) for _ in range(2))
        v = torch.randn(2, 3, width, device="cuda", generator=gen)
        floor = torch.full((3, dim), 0.3, device="cuda")
        before = s.clone(), c.clone()
        announce(f"narrow decode D={dim} P={width}")
        got = m4.selective_decode(m4.SelectiveState(s, c), k, v, q, 0.5, -0.1, floor)
        full, pad = 64 if width <= 64 else 128, 64 - dim
        own = m4.SelectiveState(F.pad(s, (0, pad, 0, pad)), F.pad(c, (0, pad, 0, full - width)))
        want = m4.selective_decode_(own, F.pad(k, (0, pad)), F.pad(v, (0, full - width)),
                                    F.pad(q, (0, pad)), 0.5, -0.1, F.pad(floor, (0, pad), value=1.0))
        torch.cuda.synchronize()
        assert torch.equal(s, before[0]) and torch.equal(c, before[1])
        assert torch.equal(got.output, want.output[..., :width])
        assert torch.equal(got.state.evidence, want.state.evidence[..., :dim, :dim])
        assert torch.equal(got.state.cross, want.state.cross[..., :width, :dim])


def test_a_state_off_16_bytes_starts_a_prefill(gpu_lib):
    """An initial state that is a view at any address, as decode takes it."""
    import mamba4_amd as m4

    gen = torch.Generator(device="cuda")
    gen.manual_seed(4)
    k, q = (torch.randn(1, 5, 2, 64, device="cuda", generator=gen) / 8 for _ in range(2))
    v = torch.randn(1, 5, 2, 64, device="cuda", generator=gen)
    beta, decay = torch.full((1, 5, 2), 0.5, device="cuda"), torch.full((1, 5, 2), -0.1, device="cuda")
    floor = torch.ones(2, 64, device="cuda")
    state = torch.eye(64, device="cuda").repeat(1, 2, 1, 1), torch.randn(1, 2, 64, 64, device="cuda")
    skewed = []
    for t in state:
        flat = torch.zeros(t.numel() + 1, device="cuda")
        flat[1:] = t.reshape(-1)
        skewed.append(flat[1:].view(t.shape))
    for grad in (False, True):
        k = k.detach().requires_grad_(grad)
        announce(f"skewed initial state grad={grad}")
        want, got = (m4.selective_gaussian_memory(k, v, q, beta, decay, floor,
                                                  initial=m4.SelectiveState(*s))
                     for s in (state, skewed))
        assert torch.equal(want.output, got.output)
        assert torch.equal(want.state.cross, got.state.cross)


def test_decode_refuses_a_state_without_batch_and_head_axes(gpu_lib):
    import mamba4_amd as m4

    flat = m4.SelectiveState(torch.zeros(6, 64, 64, device="cuda"),
                             torch.zeros(6, 64, 64, device="cuda"))
    k, v, q = (torch.zeros(6, 1, 64, device="cuda") for _ in range(3))
    for step in (m4.selective_decode, m4.selective_decode_):
        with pytest.raises(ValueError):
            step(flat, k, v, q, 0.5, -0.1, torch.ones(1, 64, device="cuda"))
