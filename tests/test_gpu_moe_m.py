"""The routed FFN on the matrix cores (k_moe_m) against the CPU oracle, <= 1e-5: every format it takes,
segments of more than one pass of 16 tokens, experts without tokens, odd numbers of 64-groups (slices and
halves of qNg64 units left empty), fewer groups than slices, non-finite tokens, and the calls that stay
with the other gathers."""
import numpy as np
import pytest

from golden.fixtures import seeded_normal
from oracle_ffi import moe_ffn
from test_gpu_moe import ctx, moe_setup, relerr, run_moe, say, torch_dev  # noqa: F401  (fixtures)

pytestmark = pytest.mark.gpu
TOL = 1e-5
FMTS = [(1, 0), (5, 0), (2, 0), (6, 4), (9, 4)] + [(4, n) for n in range(2, 16)]


def routing(rng, T, E, K, skew):
    """Most tokens on the first experts (segments over 16), the last expert without any."""
    idx = np.stack([rng.permutation(E - 1)[:K] for _ in range(T)]).astype(np.int32)
    idx[: int(T * skew), 0] = 0
    for t in range(T):
        if len(set(idx[t])) < K:
            idx[t] = np.arange(K)
    return idx, (rng.random((T, K)) + 0.1).astype(np.float32)


@pytest.mark.parametrize("fmt", FMTS)
def test_moe_m_formats(ctx, torch_dev, oracle, fmt):  # noqa: F811
    say("moe_m", fmt)
    E, H, I, K = 5, 192, 320, 2
    T = 40
    rng = np.random.default_rng(fmt[0] * 20 + fmt[1])
    sh = fmt if fmt[0] not in (6, 9) else (5, 0)
    gate, up, down, shared = moe_setup(oracle, 40 + fmt[1], E, H, I, 128, [fmt], sh_fmt=sh)
    idx, w = routing(rng, T, E, K, 0.8)
    x = seeded_normal(50 + fmt[1], (T, H))
    x[3] = 0.0
    x[5] *= 1e-3
    x[7, 10] = 3e4
    y = run_moe(ctx, torch_dev, gate, up, down, shared, x, idx, w)
    ref = moe_ffn(oracle, gate, up, down, shared, H, I, x, idx, w)
    for t in range(T):                             # token by token: their sizes differ
        assert relerr(y[t], ref[t]) <= TOL, t


@pytest.mark.parametrize("T,K,Ish", [(3, 2, 64), (16, 1, 0), (17, 3, 0), (64, 2, 128)])
def test_moe_m_shapes(ctx, torch_dev, oracle, T, K, Ish):  # noqa: F811
    """Mixed formats; one 64-group per row (all K slices but the first empty)."""
    say("moe_m shapes", T, K, Ish)
    E, H, I = 4, 64, 64
    rng = np.random.default_rng(T)
    gate, up, down, shared = moe_setup(oracle, 70 + T, E, H, I, Ish, [(1, 0), (4, 7), (4, 13), (2, 0)], [(4, 11), (5, 0)], sh_fmt=(4, 5))
    idx, w = routing(rng, T, E, K, 0.5)
    x = seeded_normal(80 + T, (T, H))
    y = run_moe(ctx, torch_dev, gate, up, down, shared, x, idx, w)
    assert relerr(y, moe_ffn(oracle, gate, up, down, shared, H, I, x, idx, w)) <= TOL


@pytest.mark.parametrize("fmt", [(1, 0), (6, 4), (4, 15)])
def test_moe_m_nonfinite_tokens(ctx, torch_dev, oracle, fmt):  # noqa: F811
    """NaN and +-Inf reach exactly the outputs that the reference's arithmetic gives them; the other
    tokens are untouched."""
    say("moe_m nonfinite", fmt)
    E, H, I, K, T = 4, 128, 128, 2, 20
    rng = np.random.default_rng(9)
    gate, up, down, _ = moe_setup(oracle, 95, E, H, I, 0, [fmt])
    idx, w = routing(rng, T, E, K, 0.5)
    x = seeded_normal(96, (T, H))
    x[2, 5], x[9, 100], x[11, 0] = np.nan, np.inf, -np.inf
    with np.errstate(all="ignore"):
        ref = moe_ffn(oracle, gate, up, down, None, H, I, x, idx, w)
    y = run_moe(ctx, torch_dev, gate, up, down, None, x, idx, w)
    bad = [2, 9, 11]
    good = [t for t in range(T) if t not in bad]
    assert relerr(y[good], ref[good]) <= TOL
    for t in bad:
        assert np.array_equal(np.isnan(y[t]), np.isnan(ref[t])), t
        inf = np.isinf(ref[t])
        assert np.array_equal(np.isinf(y[t]), inf) and np.array_equal(np.sign(y[t][inf]), np.sign(ref[t][inf])), t
