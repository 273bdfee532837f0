"""The row-parallel Q4_K and Q6_K weight encoders against the oracle, byte for byte: block counts off the four blocks of a
wave and the sixteen of a workgroup, a destination at 4-byte alignment only (Q6_K blocks are 210 bytes), ties between
equal magnitudes of either sign inside a sub-block and between sub-blocks, zero and one-valued blocks."""
import sys

import numpy as np
import pytest

from qdata import normal

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")
ov = pytest.importorskip("overfit_amd")


@pytest.mark.parametrize("fmt", ["q4k", "q6k"])
@pytest.mark.parametrize("n,k,offset", [(1, 256, 0), (3, 256, 4), (5, 768, 8), (17, 256, 4), (13, 1280, 12), (257, 256, 0)])
def test_encoder_block_counts_and_alignment(orc, fmt, n, k, offset):
    print("[case]", "encode", fmt, n, k, offset, flush=True, file=sys.stderr)
    rng = np.random.default_rng(n + k)
    w = normal(rng, (n, k), 0.02)
    w[0, :16] = [0.5, -0.5] * 8           # ties of either sign, and the next sub-block's against them
    w[0, 16:32] = [-0.5, 0.5] * 8
    w[n // 2, 64:96] = 0.25
    w[n - 1, 128:256] = 0.0
    w[n - 1, :128] = np.where(np.arange(128) % 3 == 0, -0.125, 0.125)
    ref = (orc.quantize_q4k(w) if fmt == "q4k" else orc.quantize_q6k(w)).reshape(-1)
    ctx = ov.default_context()
    src = torch.from_numpy(w).to("cuda:0")
    dst = torch.full((ref.size + 32,), 0xA5, dtype=torch.uint8, device="cuda:0")
    fn = ctx.lib.ovfq_quantize_weight_q4k_dev if fmt == "q4k" else ctx.lib.ovfq_quantize_weight_q6k_dev
    ctx.check(fn(ctx.handle, src.data_ptr(), k, n, dst.data_ptr() + offset))
    torch.cuda.synchronize()
    got = dst.cpu().numpy()
    assert np.array_equal(got[offset:offset + ref.size], ref)
    assert (got[:offset] == 0xA5).all() and (got[offset + ref.size:] == 0xA5).all()  # nothing beside the blocks
