"""The batch-1 attention merge in the O product, at chunk counts around its load groups (8, 16, then 16 at a time)."""
import numpy as np
import pytest

from lab import qwen_model as QM
from lab.hip import call, ptr
from oracle import quant as OQ

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T", [1, 3])
@pytest.mark.parametrize("nch,max_chunks", [(1, 1), (1, 64), (7, 7), (8, 9), (9, 9), (16, 17), (17, 32), (24, 64), (25, 64),
                                            (32, 32), (33, 64), (48, 64), (49, 64), (64, 64)])
def test_merge_of_n_chunks(cuda, nch, max_chunks, T):
    """h += Wo . Q8_1(merge): the merge in f64, so the quantizer sees the oracle's value to 1e-14 and the sum of exact
    block dots agrees to the fixed point (2^-48 a K slice; 1e-11 covers the f64 sums). Slots past the context hold NaN."""
    import torch
    nh, N = 6, 64
    K = nh * 128
    rng = np.random.default_rng(100 * nch + max_chunks + T)
    part = np.full((T, nh, max_chunks, 130), np.nan)
    part[:, :, :nch, :128] = rng.standard_normal((T, nh, nch, 128))
    part[:, :, :nch, 128] = rng.standard_normal((T, nh, nch)) * 3
    part[:, :, :nch, 129] = rng.random((T, nh, nch)) + 0.5
    p = part[:, :, :nch]
    w = np.exp(p[..., 128] - p[..., 128].max(2, keepdims=True))
    o = (w[..., None] * p[..., :128]).sum(2) / (w * p[..., 129]).sum(2)[..., None]
    q, d, _ = OQ.quantize_q8_1(o.reshape(T, K).astype(np.float32))
    wb = OQ.quantize_q4_0(rng.standard_normal((N, K)).astype(np.float32))
    W = QM.Q4Mat(wb, N, K, "cuda")
    h = torch.zeros(T, N, dtype=torch.int64, device=cuda)
    part_d = torch.from_numpy(part).cuda()
    pos = torch.full((T,), 64 * nch - 1, dtype=torch.int32, device=cuda)
    call("q355_attn_o_resid", ptr(W.qs), ptr(W.d), N, ptr(part_d), max_chunks, ptr(pos), nh, ptr(h), T)
    torch.cuda.synchronize()
    dw, qw = OQ.q4_0_blocks(wb)
    dense = ((qw.astype(np.float64) - 8) * dw.astype(np.float64).reshape(-1, 1)).reshape(N, K)
    ref = (q.astype(np.float64).reshape(T, -1, 32) * d.astype(np.float64).reshape(T, -1, 1)).reshape(T, K) @ dense.T
    got = h.cpu().numpy() / QM.FIX_SCALE
    assert np.abs(got - ref).max() <= 1e-11 * np.abs(ref).max() + 3 * 2.0 ** -48
