"""Finite fp32 activations of a wide range, through the kernels that split them into fp16 parts at few
columns (k_gemm_mfma at 2..15, k_moe_frag + k_moe_m): channels of up to 1e8 whose weights are zero, so that
the result comes from elements far below the largest one.  As exact digits (k_act_x24) such elements are
held to 2^-46 of their 64-group's largest; the fp16 parts alone reach 2^-38 of a whole K split's or row's
largest, so columns of a wide range are multiplied a second time by what the first parts leave over.  Bar: max|y - ref| / max|ref| <= 1e-5 per column, as everywhere."""
import numpy as np
import pytest

from golden.fixtures import seeded_normal
from oracle_ffi import moe_ffn
from test_gpu_moe import desc
from test_gpu_moe import run_moe as run_layer
from test_gpu_outliers import TOL, check_classes, context, make_weights, quant, relerr, run_dense, say, torch_dev  # noqa: F401

pytestmark = pytest.mark.gpu


def wide(name, K, M, seed):
    """(x [M][K], weight column factors): the large channels' weights are zero."""
    rng = np.random.default_rng(seed)
    x = seeded_normal(seed, (M, K))
    wmul = np.ones(K, np.float32)
    if name == "one_1e7":
        ch = [int(rng.integers(0, K))]
        x[:, ch] = np.float32(1e7)
    elif name == "group_1e8":                          # one channel in every group
        ch = np.arange(0, K, 64) + rng.integers(0, 64, K // 64)
        x[:, ch] = np.float32(1e8)
    elif name == "half_1e6":                           # whole groups far below the others
        ch = np.arange(K // 2)
        x[:, ch] *= np.float32(1e6)
    else:                                              # "few_small": and only a few nonzero elements in them
        ch = np.arange(64)
        x[:, 64:] *= (rng.random(K - 64) < 0.1).astype(np.float32)
        x[:, ch] *= np.float32(3e7)
    wmul[ch] = 0.0
    return x.astype(np.float32), wmul


NAMES = ["one_1e7", "group_1e8", "half_1e6", "few_small"]


@pytest.mark.parametrize("kind,bits", [(1, 0), (5, 0), (2, 0), (4, 3), (4, 7), (4, 10)])
@pytest.mark.parametrize("N,K", [(300, 4160), (1100, 576), (130, 192)])   # K split, and not
def test_few_columns(torch_dev, oracle, monkeypatch, kind, bits, N, K):  # noqa: F811
    """One column of ordinary range beside them: it takes no second product, and is as without them."""
    c = context(monkeypatch)
    for i, name in enumerate(NAMES):
        for M in (2, 7, 15):
            say("wide few columns", kind, bits, N, K, name, M)
            x, wmul = wide(name, K, M, 900 + i)
            x[M - 1] = seeded_normal(905 + i, (K,))
            pk, sc = make_weights(oracle, kind, bits, N, K, wmul, 910 + i)
            got = run_dense(c, torch_dev, kind, bits, pk, sc, N, K, x)
            ref = oracle.gemm_f32(kind, pk, sc, x, bits=bits)
            for m in range(M):
                assert relerr(got[m], ref[m]) <= TOL, (name, M, m, relerr(got[m], ref[m]))
    c.close()


@pytest.mark.parametrize("K", [128, 2112])
def test_few_columns_group(torch_dev, oracle, monkeypatch, K):  # noqa: F811
    """A fused group with biases; one column holds an Inf beside its wide range."""
    c = context(monkeypatch)
    M, outs = 5, (70, 200)
    say("wide few columns group", K)
    x, wmul = wide("one_1e7", K, M, 970)
    x[1, 3] = np.inf
    packed = [make_weights(oracle, 1, 0, o, K, wmul, 971 + o) for o in outs]
    bias = [seeded_normal(980 + o, (o,)) for o in outs]
    ts = [c.bind(1, p, s, o, K) for (p, s), o in zip(packed, outs)]
    dev = lambda a: torch_dev.from_numpy(np.ascontiguousarray(a)).cuda()  # noqa: E731
    xd, bd, ys = dev(x), [dev(b) for b in bias], [torch_dev.empty((M, o), device="cuda") for o in outs]
    torch_dev.cuda.synchronize()
    c.matmul_group(ts, xd, ys, biases=bd)
    c.sync()
    for (p, s), b, y in zip(packed, bias, ys):
        ref = oracle.gemm_f32(1, p, s, x) + b
        for m in range(M):
            check_classes(y[m].cpu().numpy(), ref[m], (K, m))
    for t in ts:
        t.free()
    c.close()


def layer(oracle, fmts, E, H, I, Ish, seed, wm_h, wm_i, up_rows=None):
    """Experts (gate, up, down) and shared ones: columns by wm_h (gate, up) and wm_i (down); up's rows
    by up_rows."""
    def one(kind, bits, o, i, s, wm, rows):
        w = seeded_normal(s, (o, i), 0.02) * wm[None, :].astype(np.float32)
        if rows is not None:
            w = w * rows[:, None]
        w = np.ascontiguousarray(w, np.float32)
        if kind == 6:                                  # int4 affine: codes 0..15 over each group's range
            g = w.reshape(o, -1, 64)
            b = g.min(-1)
            s_ = (g.max(-1) - b) / np.float32(15)
            q = np.rint((g - b[..., None]) / np.where(s_ > 0, s_, 1)[..., None]).astype(np.uint8).reshape(o, i)
            return (6, 4, np.ascontiguousarray(q[:, ::2] | (q[:, 1::2] << 4)), s_.astype(np.float32), b.astype(np.float32))
        if kind == 9:
            return desc(oracle, 9, 4, w)
        return (kind, bits, *quant(oracle, kind, w, bits))
    pick = lambda e: fmts[e % len(fmts)]  # noqa: E731
    gate = [one(*pick(e), I, H, seed + 3 * e, wm_h, None) for e in range(E)]
    up = [one(*pick(e), I, H, seed + 3 * e + 1, wm_h, up_rows) for e in range(E)]
    down = [one(*pick(e), H, I, seed + 3 * e + 2, wm_i, None) for e in range(E)]
    if not Ish:
        return gate, up, down, None
    k = fmts[0] if fmts[0][0] not in (6, 9) else (1, 0)
    sh = (one(*k, Ish, H, seed + 90, wm_h, None), one(*k, Ish, H, seed + 91, wm_h, None), one(*k, H, Ish, seed + 92, np.ones(Ish, np.float32), None))
    return gate, up, down, sh


@pytest.mark.parametrize("fmts", [[(1, 0)], [(5, 0), (2, 0)], [(4, 7), (4, 13)], [(6, 4)]])
@pytest.mark.parametrize("T,Ish,K", [(3, 128, 3), (9, 0, 3), (40, 192, 3), (10, 0, 1)])
def test_routed_rows(torch_dev, oracle, monkeypatch, fmts, T, Ish, K):  # noqa: F811
    """Token rows of a wide range (x), beside ordinary ones.  Affine int4 has no zero columns: its large
    channels fill whole groups, whose scale and bias are zero."""
    c = context(monkeypatch)
    E, H, I = 4, 320, 192
    for i, name in enumerate(NAMES):
        if fmts == [(6, 4)] and name != "half_1e6":
            continue
        say("wide routed rows", fmts, T, Ish, K, name)
        x, wmul = wide(name, H, T, 920 + i)
        if name == "half_1e6":
            wmul[:] = 1.0; wmul[:128] = 0.0
            x = seeded_normal(926, (T, H)); x[:, :128] *= np.float32(3e7)
        x[T - 1] = seeded_normal(927 + i, (H,))
        gate, up, down, sh = layer(oracle, fmts, E, H, I, Ish, 930 + 10 * i, wmul, np.ones(I, np.float32))
        idx, w = oracle.route(seeded_normal(940 + i, (T, E)), K, True)
        got = run_layer(c, torch_dev, gate, up, down, sh, x, idx, w)
        ref = moe_ffn(oracle, gate, up, down, sh, H, I, x, idx, w)
        for t in range(T):
            assert relerr(got[t], ref[t]) <= TOL, (name, t, relerr(got[t], ref[t]))
    c.close()


@pytest.mark.parametrize("fmts", [[(1, 0)], [(2, 0), (4, 14)], [(4, 9), (4, 5)]])
@pytest.mark.parametrize("T,Ish", [(4, 64), (12, 0)])
def test_routed_inner_rows(torch_dev, oracle, monkeypatch, fmts, T, Ish):  # noqa: F811
    """The same for h: every 64th value of the experts' up projection is 1e7 times the others, and the
    down projection's column there is zero."""
    c = context(monkeypatch)
    E, H, I, K = 4, 192, 320, 3
    say("wide inner rows", fmts, T, Ish)
    rows, wmul = np.ones(I, np.float32), np.ones(I, np.float32)
    rows[5::64] = 1e7
    wmul[5::64] = 0.0
    gate, up, down, sh = layer(oracle, fmts, E, H, I, Ish, 950, np.ones(H, np.float32), wmul, rows)
    x = seeded_normal(960, (T, H))
    idx, w = oracle.route(seeded_normal(961, (T, E)), K, True)
    got = run_layer(c, torch_dev, gate, up, down, sh, x, idx, w)
    ref = moe_ffn(oracle, gate, up, down, sh, H, I, x, idx, w)
    for t in range(T):
        assert relerr(got[t], ref[t]) <= TOL, (t, relerr(got[t], ref[t]))
    c.close()
