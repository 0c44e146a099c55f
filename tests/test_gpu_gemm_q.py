"""W4A8 products of many columns or rows (k_gemm_q) against the CPU oracle, bit for bit: both tile
shapes, partly filled tiles and column blocks, K shorter than and around the load ring, several
launches, fused groups with biases, the SwiGLU chain, and weight scales at the ends of fp32."""
import sys

import numpy as np
import pytest

from golden.fixtures import seeded_normal

pytestmark = pytest.mark.gpu


def say(*a):
    print("[case]", *a, flush=True)
    sys.stdout.flush()


@pytest.fixture(scope="module")
def torch_dev():
    import torch
    assert torch.cuda.is_available(), "gpu tests need a GPU"
    return torch


@pytest.fixture(scope="module")
def ctx(torch_dev):
    import beglin_amd
    c = beglin_amd.Context(0)
    yield c
    c.sync()
    c.close()


def pack(oracle, kind, w):
    if kind == 1:
        return (*oracle.quantize_q4g64(w), None)
    if kind == 2:
        return (*oracle.quantize_q8g64(w), None)
    if kind == 10:                                 # plain g256: the q4 bytes, one scale per 256 values
        pk, s = oracle.quantize_q4g64(w)
        return pk, np.ascontiguousarray(s[:, ::4]), None
    return oracle.quantize_g256sf(w)


def columns(seed, M, inn):
    x = seeded_normal(seed, (M, inn), 1.0)
    x[M // 2, : inn // 2] *= 1e4
    x[M - 1] = 0.0
    return x


def run(ctx, torch, kind, packed, x, biases, shapes, bits_equal_to):
    ts = [ctx.bind(kind, p, s, p.shape[0], x.shape[1], sub=sub) for p, s, sub in packed]
    xd = torch.from_numpy(x).cuda()
    ys = [torch.full((x.shape[0], o), float("nan"), device="cuda") for o in shapes]
    bd = [torch.from_numpy(b).cuda() if b is not None else None for b in biases]
    torch.cuda.synchronize()
    ctx.matmul_group(ts, xd, ys, act=1, biases=bd)
    ctx.sync()
    for t, y, r in zip(ts, ys, bits_equal_to):
        assert np.array_equal(y.cpu().numpy().view(np.uint32), r.view(np.uint32))
        t.free()


# 16 x 16 tiles (few rows), then 32 x 32 tiles (512 and more of them); 65 and 130 columns take two
# and three launches
SHAPES = [(1, 77, 64, 17), (1, 200, 1024, 33), (1, 64, 4096, 65), (2, 130, 640, 48), (2, 50, 192, 130), (3, 65, 256, 64),
          (3, 100, 2304, 49), (10, 90, 1536, 31),
          (1, 16330, 192, 6), (3, 16400, 4096, 2), (3, 16400, 512, 9), (2, 90, 4160, 9),   # 2..16 columns
          (1, 16330, 192, 40), (1, 8200, 576, 64), (2, 16330, 320, 17), (3, 16400, 768, 64),
          # 32-row tiles in two launches (64 + 6 columns); a long K over few rows, its scales past 64 KB of
          # LDS (from K = 16192 in groups of 64), to the longest K that the W4A8 kernels take (34880; 140 KB)
          (1, 16400, 192, 70), (1, 70, 14336, 24), (1, 70, 16384, 33), (2, 40, 34880, 20), (3, 64, 49152, 17)]


@pytest.mark.parametrize("kind,out,inn,M", SHAPES)
def test_gemm_q_equals_oracle(ctx, torch_dev, oracle, kind, out, inn, M):
    say("gemm_q", kind, out, inn, M)
    w = seeded_normal(10 * kind + M, (out, inn), 0.02)
    x = columns(7 + M, M, inn)
    pk, sc, sub = pack(oracle, kind, w)
    ref = oracle.matmul_sdot(kind, pk, sc, x, sub=sub)
    run(ctx, torch_dev, kind, [(pk, sc, sub)], x, [None], [out], [ref])


def test_gemm_q_group_with_biases(ctx, torch_dev, oracle):
    say("gemm_q group")
    x = columns(3, 21, 512)
    outs = (130, 64, 40)
    packed = [pack(oracle, 1, seeded_normal(40 + o, (o, 512), 0.02)) for o in outs]
    bias = [seeded_normal(60 + o, (o,), 1.0) if i != 1 else None for i, o in enumerate(outs)]
    ref = [oracle.matmul_sdot(1, p, s, x, bias=b) for (p, s, _), b in zip(packed, bias)]
    run(ctx, torch_dev, 1, packed, x, bias, outs, ref)


@pytest.mark.parametrize("kind", [1, 2, 3])
@pytest.mark.parametrize("out,inn,M", [(70, 512, 20), (70, 512, 70), (16400, 256, 20)])
def test_gemm_q_nonfinite_columns(ctx, torch_dev, oracle, kind, out, inn, M):
    """Columns with NaN or +-Inf (every code of the group 0 and its scale NaN or Inf, so every output row NaN),
    with a group of zeros, and of values below 1e-8 (the floor of the scale); the finite columns bit for bit."""
    say("gemm_q nonfinite", kind, out, inn, M)
    pk, sc, sub = pack(oracle, kind, seeded_normal(820 + kind, (out, inn), 0.02))
    x = seeded_normal(821 + M, (M, inn), 1.0)
    x[1, 5], x[3, inn - 1], x[4, 70] = np.nan, np.inf, -np.inf
    x[5, 7], x[5, 9] = np.inf, np.nan
    x[7, :256], x[8, :256] = 0.0, x[8, :256] * np.float32(1e-10)
    x[M - 1, 100] = np.nan
    with np.errstate(all="ignore"):
        ref = oracle.matmul_sdot(kind, pk, sc, x, sub=sub)
    bad = [1, 3, 4, 5, M - 1]
    assert np.isnan(ref[bad]).all() and np.isfinite(np.delete(ref, bad, 0)).all()
    t = ctx.bind(kind, pk, sc, out, inn, sub=sub)
    xd, y = torch_dev.from_numpy(x).cuda(), torch_dev.zeros((M, out), device="cuda")
    torch_dev.cuda.synchronize()
    ctx.matmul(t, xd, y, act=1)
    ctx.sync()
    got = y.cpu().numpy()
    t.free()
    assert np.array_equal(np.isnan(got), np.isnan(ref))
    ok = ~np.isnan(ref)
    assert np.array_equal(got[ok].view(np.uint32), ref[ok].view(np.uint32))


@pytest.mark.parametrize("kind,out", [(1, 70), (3, 70), (1, 16384)])
def test_gemm_q_weight_scales_at_the_ends_of_fp32(ctx, torch_dev, oracle, kind, out):
    """16x sums with scales from subnormal to 1e37 (their products may leave fp32's range): the wave
    repeats such a tile with the sums shifted back."""
    say("gemm_q scales", kind, out)
    inn, M = 768, 20
    w = seeded_normal(5, (out, inn), 0.02)
    pk, sc, sub = pack(oracle, kind, w)
    sc = sc.copy()
    e = np.random.default_rng(1).integers(-149, 120, sc.shape)
    half = out // 2                                # the other rows keep ordinary scales
    sc[:half] = np.ldexp(np.float32(1.0) + sc[:half] % np.float32(0.5), e[:half]).astype(np.float32)
    sc[3] = 0.0
    x = columns(9, M, inn) * np.float32(0.01)
    with np.errstate(all="ignore"):
        ref = oracle.matmul_sdot(kind, pk, sc, x, sub=sub)
    t = ctx.bind(kind, pk, sc, out, inn, sub=sub)
    y = torch_dev.empty((M, out), device="cuda")
    xd = torch_dev.from_numpy(x).cuda()
    torch_dev.cuda.synchronize()
    ctx.matmul(t, xd, y, act=1)
    ctx.sync()
    got = y.cpu().numpy()
    t.free()
    assert np.array_equal(np.isnan(got), np.isnan(ref))
    ok = ~np.isnan(ref)
    assert np.array_equal(got[ok].view(np.uint32), ref[ok].view(np.uint32))


@pytest.mark.parametrize("kind,M", [(1, 17), (3, 40), (2, 70)])
def test_gemm_q_mlp_block(ctx, torch_dev, oracle, kind, M):
    """The MLP block: the down projection's quantization forms h; y and h bit for bit."""
    say("gemm_q mlp", kind, M)
    H, I = 512, 1280
    x = seeded_normal(M, (M, H), 1.0)
    ws = [pack(oracle, kind, seeded_normal(70 + i, s, 0.05)) for i, s in enumerate(((I, H), (I, H), (H, I)))]
    g, u = (oracle.matmul_sdot(kind, p, s, x, sub=sub) for p, s, sub in ws[:2])
    h = np.stack([oracle.swiglu(a, b) for a, b in zip(g, u)])
    ref = oracle.matmul_sdot(kind, ws[2][0], ws[2][1], h, sub=ws[2][2])
    ts = [ctx.bind(kind, p, s, p.shape[0], k, sub=sub) for (p, s, sub), k in zip(ws, (H, H, I))]
    y, hd = torch_dev.empty((M, H), device="cuda"), torch_dev.empty((M, I), device="cuda")
    xd = torch_dev.from_numpy(x).cuda()
    torch_dev.cuda.synchronize()
    ctx.mlp(*ts, xd, y, act=1, h_dev=hd)
    ctx.sync()
    assert np.array_equal(hd.cpu().numpy().view(np.uint32), h.view(np.uint32))
    assert np.array_equal(y.cpu().numpy().view(np.uint32), ref.view(np.uint32))
    for t in ts:
        t.free()


@pytest.mark.parametrize("kind,rows,inn,M", [(1, 100, 256, 20), (2, 16400, 256, 6), (3, 70, 512, 64)])
def test_gemm_q_leaves_prepared_operands(torch_dev, oracle, kind, rows, inn, M):
    """A W4A8 call over a short K took no prepared operands of its own, so what bgl_prep_act_dev left
    outlived it: k_gemm_q's codes lie elsewhere."""
    import beglin_amd
    say("gemm_q beside prepared operands", kind, rows, inn, M)
    c = beglin_amd.Context(0)
    packed = pack(oracle, kind, seeded_normal(800 + M, (rows, inn), 0.02))
    pp, ps = oracle.quantize_q4g64(seeded_normal(801, (90, 1024), 0.02))
    tp = c.bind(1, pp, ps, 90, 1024)
    x, xp = columns(802, M, inn), seeded_normal(803, (3, 1024))
    xpd, yp = torch_dev.from_numpy(xp).cuda(), torch_dev.empty((3, 90), device="cuda")
    for act in (0, 1):
        torch_dev.cuda.synchronize()
        c.prep_only(xpd, act, tp)
        run(c, torch_dev, kind, [packed], x, [None], [rows], [oracle.matmul_sdot(kind, packed[0], packed[1], x, sub=packed[2])])
        c.matmul_prepped(tp, yp, act=act, M=3)
        c.sync()
        ref = oracle.matmul_sdot(1, pp, ps, xp) if act else oracle.gemm_f32(1, pp, ps, xp)
        assert np.max(np.abs(yp.cpu().numpy() - ref)) <= 1e-5 * np.max(np.abs(ref))
    tp.free()
    c.close()
