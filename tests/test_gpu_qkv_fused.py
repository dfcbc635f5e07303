"""Which QKV products of a prefill chunk run fused (q355_mmq_qkv_rope), over shapes on both sides of the rule."""
import numpy as np
import pytest

from lab import qwen_batched as QB
from lab import qwen_model as QM
from lab.hip import call, ptr

pytestmark = pytest.mark.gpu


# K past the register-resident form with 20 tokens, K % 128 != 0 with 50 and 100, and the shapes that do fuse
@pytest.mark.parametrize("H,NH,NKV,P", [(2048, 16, 2, 20), (2048, 16, 2, 100), (960, 8, 2, 50), (960, 8, 2, 100),
                                        (1088, 4, 1, 33), (1536, 12, 2, 20), (1536, 12, 2, 77), (896, 8, 2, 200),
                                        (1536, 12, 2, 300)])
def test_prefill_qkv_sums_as_the_split_product(cuda, H, NH, NKV, P):
    """A layer's K and V rows are those of the K-split product and q355_qkv_finish, bit for bit: both sum the same slices
    or in f64, so an fp16 rounding can differ with a chance of 2^-30 a value, where one fp32 chain over K moves about one
    value in 2,000."""
    import torch
    cfg = QM.Config(H=H, NH=NH, NKV=NKV, FFN=256, L=1, V=4096)
    m = QM.DeviceModel(QM.random_weights(cfg, seed=H + P), cfg, maxlen=512)
    dec = QM.Decoder(m, T=1, max_ctx=512)
    pf = QB.Prefill(dec, max_chunk=512)
    h = torch.from_numpy(np.round(np.random.default_rng(P).standard_normal((P, H)) * QM.FIX_SCALE).astype(np.int64)).cuda()
    pf.h[:P].copy_(h)
    pf.pos[:P].copy_(torch.arange(P, dtype=torch.int32))
    pf.layer(0, P, 0)
    L, W = m.layers[0], m.layers[0]["qkv"]
    xq = torch.zeros(P, H, dtype=torch.int8, device=cuda)
    xds = torch.zeros(P, H // 32, 2, dtype=torch.float16, device=cuda)
    acc = torch.zeros(P, W.N, dtype=torch.int64, device=cuda)
    q = torch.zeros(P, NH * 128, dtype=torch.float16, device=cuda)
    kc, vc = torch.zeros_like(dec.kc[0]), torch.zeros_like(dec.vc[0])
    call("q355_rmsnorm_fix_q8_1", ptr(h), ptr(L["ln1"]), ptr(xq), ptr(xds), P, H, cfg.eps)
    call("q355_mmq_q4_0_q8_1", ptr(W.qs), ptr(W.d), W.N, W.K, ptr(xq), ptr(xds), P, 6, None, ptr(acc), None, None, None,
         None)
    call("q355_qkv_finish", ptr(acc), ptr(L["qkv_b"]), ptr(m.cos), ptr(m.sin), ptr(pf.pos), ptr(dec.block_table),
         dec.max_chunks, 0, ptr(kc), ptr(vc), ptr(q), NH, NKV, P)
    torch.cuda.synchronize()
    assert int((vc != 0).sum()) > P * NKV * 100
    assert torch.equal(kc, dec.kc[0]) and torch.equal(vc, dec.vc[0])
