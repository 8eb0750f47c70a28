"""selective_diagnostics on the GPU (m4mr_diagnostics) against the oracle.

The eigenvalue extremes come from a float64 tridiagonalisation of the float32
state and its Sturm counts, rounded to float32: they are checked to 2e-7 of themselves (fp32
rounding is 6e-8) plus 1e-10 of the state's largest eigenvalue, and the
condition number to 5e-7 relative; the finiteness flag, the cross maximum
and the floor range are exact.
"""

import numpy as np
import pytest
import torch

from oracle import memread as oracle
from tests.gpu_helpers import announce, run_gpu

pytestmark = pytest.mark.gpu


def _diagnose(evidence, cross, floor):
    from mamba4_amd import SelectiveState, selective_diagnostics

    dev = torch.device("cuda:0")
    state = SelectiveState(torch.tensor(evidence, dtype=torch.float32, device=dev),
                           torch.tensor(cross, dtype=torch.float32, device=dev))
    got = selective_diagnostics(state, torch.tensor(floor, dtype=torch.float32, device=dev))
    torch.cuda.synchronize()
    return {k: v.item() for k, v in got.items()}


def _check(got, want, scale):
    assert set(got) == set(oracle.DIAGNOSTIC_KEYS)
    for key in ("precision_min_eigenvalue", "precision_max_eigenvalue"):
        assert abs(got[key] - want[key]) <= 2e-7 * abs(want[key]) + 1e-10 * scale, (
            key, got[key], want[key])
    assert got["precision_max_condition"] == pytest.approx(want["precision_max_condition"], rel=5e-7)
    assert got["state_all_finite"] == want["state_all_finite"]
    for key in ("cross_max_abs", "floor_min", "floor_max"):
        assert got[key] == np.float32(want[key]), key


def _known_state(seed, batch, heads, dim, value_dim, low=1e-3, high=50.0):
    rng = np.random.default_rng(seed)
    mu = np.exp(rng.uniform(np.log(low), np.log(high), size=(batch, heads, dim)))
    q, _ = np.linalg.qr(rng.normal(size=(batch, heads, dim, dim)))
    precision = np.einsum("bhij,bhj,bhkj->bhik", q, mu, q)
    floor = rng.uniform(0.01, 0.5, size=(heads, dim)).astype(np.float32)
    evidence = (precision - floor[None, :, :, None] * np.eye(dim)).astype(np.float32)
    cross = rng.normal(size=(batch, heads, value_dim, dim)).astype(np.float32)
    return evidence, cross, floor


@pytest.mark.parametrize("dim", [1, 2, 17, 63, 64])
def test_diagnostics_match_oracle_on_known_spectra(gpu_lib, dim):
    announce(f"selective_diagnostics known spectra D={dim}")
    evidence, cross, floor = _known_state(dim, 3, 4, dim, 5)
    want = oracle.diagnostics(evidence, cross, floor)
    _check(_diagnose(evidence, cross, floor), want, want["precision_max_eigenvalue"])


def test_diagnostics_of_a_forward_end_state(gpu_lib):
    """The end state of a config-2-like forward (unit keys, sigmoid gates,
    floor 1e-2), as the mixer probes it (lm/models/mamba4.py:290-310)."""
    from mamba4_amd.inputs import synthetic_inputs

    data = synthetic_inputs(2, 256, 4, seed=42)
    announce("selective_diagnostics of a forward end state B2 T256 H4 D64")
    got = run_gpu(data, chunk=64)
    want = oracle.diagnostics(got["evidence"], got["cross"], data["floor"])
    _check(_diagnose(got["evidence"], got["cross"], data["floor"]), want,
           want["precision_max_eigenvalue"])


def test_diagnostics_symmetrise_broadcast_and_flag_non_finite(gpu_lib):
    announce("selective_diagnostics: skew part, shared floor, planted NaN and inf")
    evidence, cross, floor = _known_state(7, 2, 3, 12, 4)
    rng = np.random.default_rng(8)
    skew = rng.normal(size=evidence.shape).astype(np.float32)
    skew = skew - np.swapaxes(skew, -1, -2)
    want = oracle.diagnostics(evidence + skew, cross, floor)
    _check(_diagnose(evidence + skew, cross, floor), want, want["precision_max_eigenvalue"])
    # A floor shared by every head ([D]).
    shared = floor[0]
    want = oracle.diagnostics(evidence, cross, shared)
    _check(_diagnose(evidence, cross, shared), want, want["precision_max_eigenvalue"])
    # NaN in cross: not finite, NaN maximum, eigenvalues unaffected.
    bad = cross.copy()
    bad[1, 2, 0, 5] = np.nan
    got = _diagnose(evidence, bad, floor)
    assert got["state_all_finite"] is False and np.isnan(got["cross_max_abs"])
    assert np.isfinite(got["precision_min_eigenvalue"])
    # inf in evidence: not finite, NaN eigenvalue extremes and condition.
    bad = evidence.copy()
    bad[0, 1, 3, 4] = np.inf
    got = _diagnose(bad, cross, floor)
    assert got["state_all_finite"] is False
    assert np.isnan(got["precision_min_eigenvalue"]) and np.isnan(got["precision_max_condition"])
    assert np.isfinite(got["cross_max_abs"])


@pytest.mark.parametrize("dim", [1, 2, 3, 16, 17, 33, 64])
def test_diagnostics_of_degenerate_spectra(gpu_lib, dim):
    """Matrices whose tridiagonal decouples or repeats eigenvalues, and one
    that is indefinite: the extremes are eigvalsh's to float32 rounding (and
    float64 rounding of the largest eigenvalue)."""
    rng = np.random.default_rng(dim)
    dense = rng.normal(size=(dim, dim))
    blocks = np.zeros((dim, dim))
    half = (dim + 1) // 2
    blocks[:half, :half] = dense[:half, :half] @ dense[:half, :half].T
    vector = rng.normal(size=dim)
    cases = [
        np.zeros((dim, dim)),
        np.eye(dim) * 3.0,
        np.diag(np.logspace(-8, 3, dim)),
        blocks,                                    # half of it zero
        np.outer(vector, vector),                  # rank one
        dense + dense.T,                           # indefinite
        np.diag(rng.normal(size=dim)) * 1e30,      # squares past float32
        np.ones((dim, dim)) * 1e-30,
    ]
    floor = np.zeros(dim, np.float32)
    cross = np.ones((1, 1, 2, dim), np.float32)
    for i, matrix in enumerate(cases):
        evidence = matrix.astype(np.float32)
        announce(f"selective_diagnostics degenerate case {i} D={dim}")
        got = _diagnose(evidence[None, None], cross, floor)
        exact = evidence.astype(np.float64)
        want = np.linalg.eigvalsh(0.5 * (exact + exact.T))
        size = np.abs(want).max()
        for key, ref in (("precision_min_eigenvalue", want[0]),
                         ("precision_max_eigenvalue", want[-1])):
            assert abs(got[key] - ref) <= 1.2e-7 * abs(ref) + 1e-13 * size, (i, key, got[key], ref)


@pytest.mark.parametrize("dim", [2, 3, 17, 64])
@pytest.mark.parametrize("large", [1e6, 1e15, 1e30, -1e30])
def test_diagnostics_beside_a_large_coordinate(gpu_lib, dim, large):
    """One floor entry far above the rest: the extreme of the other coordinates
    is that of the precision without it, up to its coupling squared over the
    large entry (that second-order term included for 1e6), not lost in float64
    rounding of the large one."""
    evidence, cross, floor = _known_state(dim, 1, 1, dim, 2, low=1e-2, high=50.0)
    floor[0, dim // 2] = large
    announce(f"selective_diagnostics beside {large:g} D={dim}")
    got = _diagnose(evidence, cross, floor)
    exact = evidence[0, 0].astype(np.float64)
    exact = 0.5 * (exact + exact.T) + np.diag(floor[0].astype(np.float64))
    rest = np.arange(dim) != dim // 2
    coupling, top = exact[rest, dim // 2], exact[dim // 2, dim // 2]
    others = np.linalg.eigvalsh(exact[np.ix_(rest, rest)] - np.outer(coupling, coupling) / top)
    small = others[0] if large > 0 else others[-1]
    # The Schur complement's eigenvalues are off by its own size squared over the
    # large entry at most.
    bound = 2e-7 * abs(small) + 50.0 ** 3 / top ** 2 + 1e-12
    ends = ("precision_min_eigenvalue", "precision_max_eigenvalue")
    inner, outer = ends if large > 0 else ends[::-1]
    assert abs(got[inner] - small) <= bound, (got[inner], small)
    assert got[outer] == pytest.approx(top, rel=2e-7 + 50.0 ** 2 / top ** 2)
    if large > 0:
        assert got["precision_max_condition"] == pytest.approx(top / small, rel=1e-6 + bound / small)


@pytest.mark.parametrize("low,high", [(-3, 3), (0, 6), (-5, 5)])
def test_diagnostics_of_graded_precisions(gpu_lib, low, high):
    """Well-conditioned matrices scaled per coordinate over many orders of
    magnitude: the smallest eigenvalue (from the inverse, which the scaling makes
    accurate in float64) to float32 rounding."""
    rng = np.random.default_rng(high)
    for dim in (2, 9, 33, 64):
        x = rng.normal(size=(dim, 2 * dim))
        scale = 10.0 ** rng.uniform(low, high, size=dim)
        evidence = (scale[:, None] * (x @ x.T / (2 * dim)) * scale).astype(np.float32)
        announce(f"selective_diagnostics graded 1e{low}..1e{high} D={dim}")
        got = _diagnose(evidence[None, None], np.ones((1, 1, 2, dim), np.float32),
                        np.zeros(dim, np.float32))
        exact = evidence.astype(np.float64)
        exact = 0.5 * (exact + exact.T)
        root = np.sqrt(np.diag(exact))
        inverse = np.linalg.inv(exact / root[:, None] / root) / root[:, None] / root
        smallest = 1.0 / np.linalg.eigvalsh(0.5 * (inverse + inverse.T))[-1]
        assert got["precision_min_eigenvalue"] == pytest.approx(smallest, rel=1.2e-7)
        assert got["precision_max_eigenvalue"] == pytest.approx(np.linalg.eigvalsh(exact)[-1],
                                                                rel=1.2e-7)


def test_diagnostics_rejects_wide_states(gpu_lib):
    from mamba4_amd import SelectiveState, selective_diagnostics

    dev = torch.device("cuda:0")
    state = SelectiveState(torch.zeros(1, 1, 65, 65, device=dev), torch.zeros(1, 1, 4, 65, device=dev))
    with pytest.raises(ValueError):
        selective_diagnostics(state, torch.ones(65, device=dev))
