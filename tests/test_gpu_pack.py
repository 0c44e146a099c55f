"""Device packers, repacks and the decoder at the edges of their workgroups: a last group of a partly
filled workgroup, tiles with missing rows, an odd number of groups, row ranges that start inside a tile;
bytes and decoded values bit for bit against the oracle."""
import sys

import numpy as np
import pytest

from golden.fixtures import seeded_normal
from test_gpu_gemv import ctx, ref_quant, torch_dev  # noqa: F401  (fixtures)

pytestmark = pytest.mark.gpu

CASES = [(1, 0), (2, 0), (3, 0), (5, 0)] + [(4, n) for n in range(2, 16)]


@pytest.mark.parametrize("kind,bits", CASES)
def test_pack_and_decode_edges(ctx, torch_dev, oracle, kind, bits):  # noqa: F811
    torch = torch_dev
    for out, inn in ((1, 256), (65, 256 if kind == 3 else 192), (130, 768 if kind == 3 else 832)):
        print("[case] pack", kind, bits, out, inn, flush=True)
        sys.stdout.flush()
        w = seeded_normal(900 + kind + bits + out, (out, inn), 0.02)
        w[0, :64] = 0.0
        pk, sc, sub = ref_quant(oracle, kind, w, bits)
        wd = torch.from_numpy(w).cuda()
        torch.cuda.synchronize()
        t, (gpk, gsc, gsub) = ctx.quantize(kind, wd, bits=bits, qng64_encoder=(bits != 4), want_ref=True)
        assert np.array_equal(gpk.view(np.uint8), np.asarray(pk).view(np.uint8))
        assert np.array_equal(gsc, sc) and (sub is None or np.array_equal(gsub, sub))
        ref = oracle.decode(kind, pk, sc, out, inn, bits=bits, sub=sub)
        for r0, nr in ((0, out), (out // 2, out - out // 2)):
            y = torch.full((nr, inn), float("nan"), device="cuda")
            torch.cuda.synchronize()
            ctx.dequant(t, r0, nr, y)
            ctx.sync()
            assert np.array_equal(y.cpu().numpy().view(np.uint32), ref[r0:r0 + nr].view(np.uint32))
        t.free()
