"""Finite fp32 activations of a wide range, through the kernels that split them into fp16 parts at few
columns (k_gemm_mfma at 2..15): channels of up to 1e8 whose weights are zero, so that the result comes
from elements far below the largest one.  As exact digits (k_act_x24) such elements are held to 2^-46 of
their 64-group's largest; the fp16 parts alone reach 2^-38 of a whole K split's largest, so columns of a
wide range are multiplied a second time by what the first parts leave over.  Bar: max|y - ref| / max|ref| <= 1e-5 per column, as everywhere."""
import numpy as np
import pytest

from golden.fixtures import seeded_normal
from test_gpu_outliers import TOL, check_classes, context, make_weights, relerr, run_dense, say, torch_dev  # noqa: F401

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
