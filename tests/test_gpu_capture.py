"""Graph capture and the context's per-call scratch, through the C-ABI.

A graph captured from a context's stream holds the raw addresses of the scratch its calls used
(activation digits, sort buffers, routing, partial sums).  These tests pin the contract stated in
include/beglin_qgemv.h:
* a later, larger eager call that outgrows the scratch does not free what a graph uses: replays
  after it still give the captured call's result, bit for bit;
* a captured call that would need more scratch than any eager call has sized fails with
  BGL_E_CAPTURE, enqueues nothing, and the context keeps working."""
import sys

import numpy as np
import pytest

from golden.fixtures import seeded_normal
from oracle_ffi import moe_ffn

pytestmark = pytest.mark.gpu


def say(*a):
    print("[case]", *a, flush=True)
    sys.stdout.flush()


@pytest.fixture(scope="module")
def torch_dev():
    import torch
    assert torch.cuda.is_available(), "gpu tests need a GPU"
    return torch


def dev(torch, a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def moe_stack(ctx, oracle, E, o, i, seed):
    ds = []
    for e in range(E):
        w = seeded_normal(seed + e, (o, i), 0.02)
        p, s = oracle.quantize_q4g32h(w) if e % 2 == 0 else oracle.quantize_qng64(w, 9)
        ds.append((5, 0, p, s) if e % 2 == 0 else (4, 9, p, s))
    return ctx.bind_experts(ds)


def test_moe_layer_graph_survives_larger_eager_call(torch_dev, oracle):
    import beglin_amd
    torch = torch_dev
    E, H, I, K = 16, 512, 256, 4
    say("capture moe layer T=1, eager T=64, replay")
    s = torch.cuda.Stream()
    c = beglin_amd.Context(0, stream=s.cuda_stream)
    g, u, d = moe_stack(c, oracle, E, I, H, 100), moe_stack(c, oracle, E, I, H, 200), moe_stack(c, oracle, E, H, I, 300)
    rw = dev(torch, seeded_normal(400, (E, H), 0.05))
    x1 = dev(torch, seeded_normal(401, (1, H)))
    x64 = dev(torch, seeded_normal(402, (64, H)))
    y1 = torch.zeros((1, H), device="cuda")
    y64 = torch.zeros((64, H), device="cuda")
    with torch.cuda.stream(s):
        c.moe_layer(rw, g, u, d, None, x1, K, y1)
    c.sync()
    eager = y1.cpu().numpy().copy()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=s):
        c.moe_layer(rw, g, u, d, None, x1, K, y1)
    for r in range(3):
        with torch.cuda.stream(s):
            c.moe_layer(rw, g, u, d, None, x64, K, y64)      # outgrows every scratch buffer the graph uses
        c.sync()
        y1.zero_()
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert np.array_equal(y1.cpu().numpy(), eager), r
    for t in (g, u, d):
        t.free()
    c.close()


def test_dense_graph_survives_larger_eager_call(torch_dev, oracle):
    """fp32 activations over a prepared-digit path (K > 4096) and a K-split launch (few tiles)."""
    import beglin_amd
    torch = torch_dev
    say("capture dense M=2, eager M=12, replay")
    s = torch.cuda.Stream()
    c = beglin_amd.Context(0, stream=s.cuda_stream)
    N, K = 96, 8192                                      # 2 tiles: split K over workgroups (partials)
    p, sc = oracle.quantize_qng64(seeded_normal(500, (N, K), 0.02), 6)
    t = c.bind(4, p, sc, N, K, bits=6)
    x2 = dev(torch, seeded_normal(501, (2, K)))
    x12 = dev(torch, seeded_normal(502, (12, K)))
    y2 = torch.zeros((2, N), device="cuda")
    y12 = torch.zeros((12, N), device="cuda")
    with torch.cuda.stream(s):
        c.matmul(t, x2, y2)
    c.sync()
    eager = y2.cpu().numpy().copy()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=s):
        c.matmul(t, x2, y2)
    for r in range(3):
        with torch.cuda.stream(s):
            c.matmul(t, x12, y12)
        c.sync()
        y2.zero_()
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert np.array_equal(y2.cpu().numpy(), eager), r
    t.free()
    c.close()


def test_capture_that_needs_more_scratch_is_refused(torch_dev, oracle):
    import beglin_amd
    torch = torch_dev
    say("capture needing growth -> BGL_E_CAPTURE")
    s = torch.cuda.Stream()
    c = beglin_amd.Context(0, stream=s.cuda_stream)
    N, K = 256, 8192
    p, sc = oracle.quantize_q4g32h(seeded_normal(600, (N, K), 0.02))
    t = c.bind(5, p, sc, N, K)
    x1 = dev(torch, seeded_normal(601, (1, K)))
    x8 = dev(torch, seeded_normal(602, (8, K)))
    y1 = torch.zeros((1, N), device="cuda")
    y8 = torch.zeros((8, N), device="cuda")
    with torch.cuda.stream(s):
        c.matmul(t, x1, y1)                               # sizes the scratch for one column
    c.sync()
    graph = torch.cuda.CUDAGraph()
    refused = None
    with torch.cuda.stream(s):
        graph.capture_begin()
        try:
            c.matmul(t, x8, y8)                           # eight columns' digits: more scratch
        except beglin_amd.BglError as e:
            refused = e
        graph.capture_end()
    assert refused is not None and "capture" in str(refused), refused
    with torch.cuda.stream(s):
        c.matmul(t, x8, y8)                               # eager: grows the scratch and runs
    c.sync()
    ref = oracle.gemm_f32(5, p, sc, x8.cpu().numpy())
    got = y8.cpu().numpy()
    assert np.max(np.abs(got - ref)) / np.max(np.abs(ref)) <= 1e-5
    t.free()
    c.close()


@pytest.mark.parametrize("H,I,fm,Ish", [(192, 9216, (5, 9), 0), (9216, 192, (5, 9), 0), (320, 256, (6,), 0), (9216, 192, (5, 9), 64)])
def test_routed_capture_at_fewer_tokens(torch_dev, oracle, H, I, fm, Ish):
    """A routed layer that ran at 16 tokens (matrix cores) may be captured at any fewer, also where the
    fewer tokens take another gather, whose prepared digits a width past 9k or affine int4 experts need."""
    import beglin_amd
    torch = torch_dev
    E, K = 8, 2
    s = torch.cuda.Stream()
    c = beglin_amd.Context(0, stream=s.cuda_stream)

    def desc(e, o, i, seed):
        f = fm[e % len(fm)]
        if f == 6:
            rng = np.random.default_rng(seed)
            return (6, 4, rng.integers(0, 256, (o, i // 2), dtype=np.uint8), rng.random((o, i // 64), dtype=np.float32) * np.float32(0.01),
                    rng.standard_normal((o, i // 64), dtype=np.float32) * np.float32(0.04))
        w = seeded_normal(seed, (o, i), 0.02)
        return (5, 0, *oracle.quantize_q4g32h(w)) if f == 5 else (4, 9, *oracle.quantize_qng64(w, 9))

    gate, up, down = ([desc(e, o, i, 700 + 100 * j + e) for e in range(E)] for j, (o, i) in enumerate(((I, H), (I, H), (H, I))))
    stacks = [c.bind_experts(d) for d in (gate, up, down)]
    shared = sh = None
    if Ish:
        shared = tuple((5, 0, *oracle.quantize_q4g32h(seeded_normal(1000 + j, oi, 0.02))) for j, oi in enumerate(((Ish, H), (Ish, H), (H, Ish))))
        sh = tuple(c.bind(5, d[2], d[3], d[2].shape[0], d[2].shape[1] * 2) for d in shared)
    x = seeded_normal(1010, (16, H))
    idx, w = oracle.route(seeded_normal(1011, (16, E)), K, True)
    ref = moe_ffn(oracle, gate, up, down, shared, H, I, x, idx, w)
    xd, idxd, wd = dev(torch, x), dev(torch, idx), dev(torch, w)
    y = torch.zeros((16, H), device="cuda")
    torch.cuda.synchronize()
    c.moe_ffn(*stacks, sh, xd, idxd, wd, y)
    c.sync()
    for T in (16, 7, 3, 2, 1):
        say("routed capture", H, I, fm, Ish, T)
        yt = torch.zeros((T, H), device="cuda")
        xt, it, wt = xd[:T].contiguous(), idxd[:T].contiguous(), wd[:T].contiguous()
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=s):
            c.moe_ffn(*stacks, sh, xt, it, wt, yt)
        for _ in range(2):
            yt.zero_()
            torch.cuda.synchronize()
            graph.replay()
            torch.cuda.synchronize()
            got = yt.cpu().numpy()
            assert np.max(np.abs(got - ref[:T])) / np.max(np.abs(ref[:T])) <= 1e-5, T
        del graph
    for t in stacks + list(sh or ()):
        t.free()
    c.close()


@pytest.mark.parametrize("kind,pre", [(1, 0), (4, 0), (1, 1)])
def test_one_column_captured_after_several_and_a_prep(torch_dev, oracle, kind, pre):
    """Operands prepared for another product (bgl_prep_act_dev) are in the context when a call of several
    columns runs: a capture of that call at one column, which needs prepared digits (K > 4096), still
    works, and the prepared operands are still the ones that were prepared."""
    import beglin_amd
    torch = torch_dev
    say("one column after a prep", kind, pre)
    s = torch.cuda.Stream()
    c = beglin_amd.Context(0, stream=s.cuda_stream)
    N, K = 96, 8192
    w = seeded_normal(520, (N, K), 0.02)
    p, sc = oracle.quantize_qng64(w, 6) if kind == 4 else oracle.quantize_q4g64(w)
    t = c.bind(kind, p, sc, N, K, bits=6 if kind == 4 else 0)
    pp, ps = oracle.quantize_q4g64(seeded_normal(521, (80, 512), 0.02))
    tp = c.bind(1, pp, ps, 80, 512)
    x, xp = seeded_normal(522, (5, K)), seeded_normal(523, (3, 512))
    xd, xpd = dev(torch, x), dev(torch, xp)
    y, yp = torch.zeros((5, N), device="cuda"), torch.zeros((3, 80), device="cuda")
    torch.cuda.synchronize()
    c.prep_only(xpd, pre, tp)
    c.matmul(t, xd, y)
    c.sync()
    y1 = torch.zeros((1, N), device="cuda")
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    c.matmul_prepped(tp, yp, act=pre, M=3)                # before the capture, which prepares its own
    with torch.cuda.graph(graph, stream=s):
        c.matmul(t, xd[:1], y1)
    ref = oracle.gemm_f32(kind, p, sc, x[:1], bits=6 if kind == 4 else 0)
    for _ in range(2):
        y1.zero_()
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert np.max(np.abs(y1.cpu().numpy() - ref)) / np.max(np.abs(ref)) <= 1e-5
    refp = oracle.gemm_f32(1, pp, ps, xp) if pre == 0 else oracle.matmul_sdot(1, pp, ps, xp)
    assert np.max(np.abs(yp.cpu().numpy() - refp)) / np.max(np.abs(refp)) <= 1e-5
    for q in (t, tp):
        q.free()
    c.close()
