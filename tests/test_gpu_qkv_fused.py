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


@pytest.mark.parametrize("T", [20, 40, 100, 300])
def test_fused_qkv_keeps_large_and_non_finite_values(cuda, T):
    """Products past the residual stream's fixed point (2^15), past fp16, infinite and NaN come out of the fused call of
    every form as the float64 sum rounded to fp16."""
    import torch
    nh, nkv, K = 4, 1, 512
    N, nb = (nh + 2 * nkv) * 128, K // 32
    rng = np.random.default_rng(T)
    qs = np.full((N, nb, 16), 0x99, np.uint8)                             # every weight d (9 - 8)
    d = np.full((N, nb), 0.25, np.float16)
    row = {"large": (nh + nkv) * 128, "over": (nh + nkv) * 128 + 1, "inf": (nh + nkv) * 128 + 2, "nan": (nh + nkv) * 128 + 37}
    d[row["large"]], d[row["over"]] = 0.9, 20000
    d[row["inf"], nb // 2], d[row["nan"], nb - 1] = np.inf, np.nan
    W = QM.Q4Mat(np.concatenate([d.view(np.uint8).reshape(N, nb, 2), qs], 2).reshape(-1, 18), N, K, "cuda")
    xq = np.full((T, K), 100, np.int8) - rng.integers(0, 3, (T, K)).astype(np.int8)
    xds = np.ones((T, nb, 2), np.float16)
    with np.errstate(invalid="ignore", over="ignore"):
        dots = xq.reshape(T, nb, 32).astype(np.float64).sum(2)
        want = (dots[:, None] * d.astype(np.float64)[None]).sum(2).astype(np.float16)[:, (nh + nkv) * 128:]
    assert 2 ** 15 < want[0, 0] < 65504 and want[0, 1] == np.inf and want[0, 2] == np.inf and np.isnan(want[0, 37])
    t = lambda a: torch.from_numpy(a).cuda()  # noqa: E731
    pages = (T + 63) // 64
    kc = torch.zeros(pages, nkv, 64, 128, dtype=torch.float16, device=cuda)
    vc, q = torch.zeros_like(kc), torch.zeros(T, nh * 128, dtype=torch.float16, device=cuda)
    args = [t(xq), t(xds), t(np.zeros(N, np.float32)), t(np.ones((512, 64), np.float32)), t(np.zeros((512, 64), np.float32)),
            t(np.arange(T, dtype=np.int32)), t(np.arange(pages, dtype=np.int32))]
    p = [ptr(a) for a in args]
    call("q355_mmq_qkv_rope", ptr(W.qs), ptr(W.d), N, K, p[0], p[1], T, *p[2:], pages, 0, ptr(kc), ptr(vc), ptr(q), None, nh,
         nkv)
    torch.cuda.synchronize()
    got = vc.reshape(-1, 128)[:T].cpu().numpy()
    np.testing.assert_array_equal(got, want)


def test_fused_qkv_of_more_than_65535_tiles_of_32_tokens(cuda):
    """The call takes up to 65535 x 64 tokens, the grid's third dimension 65535 workgroups: past 65535 x 32 tokens the
    workgroups hold 64 tokens, and the last tokens come out as a short call gives them."""
    import torch
    nh, nkv, K, T = 4, 1, 32, 65535 * 32 + 33
    N = (nh + 2 * nkv) * 128
    rng = np.random.default_rng(3)
    d = np.full((N, 1), 0.01, np.float16)
    qs = rng.integers(0, 256, (N, 1, 16), dtype=np.uint8)
    W = QM.Q4Mat(np.concatenate([d.view(np.uint8).reshape(N, 1, 2), qs], 2).reshape(-1, 18), N, K, "cuda")
    xq = torch.randint(-127, 128, (T, K), device=cuda, dtype=torch.int32, generator=torch.Generator(cuda).manual_seed(1)).to(torch.int8)
    xds = torch.full((T, 1, 2), 0.01, dtype=torch.float16, device=cuda)
    bias = torch.zeros(N, device=cuda)
    cos, sin = torch.ones(64, 64, device=cuda), torch.zeros(64, 64, device=cuda)
    pos = torch.zeros(T, dtype=torch.int32, device=cuda)
    table = torch.zeros(1, dtype=torch.int32, device=cuda)
    kc, vc = (torch.zeros(1, nkv, 64, 128, dtype=torch.float16, device=cuda) for _ in range(2))

    def run(first, n):
        q = torch.zeros(n, nh * 128, dtype=torch.float16, device=cuda)
        call("q355_mmq_qkv_rope", ptr(W.qs), ptr(W.d), N, K, ptr(xq[first:]), ptr(xds[first:]), n, ptr(bias), ptr(cos), ptr(sin),
             ptr(pos), ptr(table), 1, 0, ptr(kc), ptr(vc), ptr(q), None, nh, nkv)
        return q

    q = run(0, T)
    assert torch.equal(q[-100:], run(T - 100, 100)) and torch.equal(q[:600], run(0, 600)) and bool((q[-100:] != 0).any())
