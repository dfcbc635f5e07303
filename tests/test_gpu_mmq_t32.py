"""The prefill products on 32 x 32 x 32 int8 tiles (k_mmq_t32, k_mmq_s32) at the sizes where they can go wrong: K shorter than a
staged chunk of 4 or 8 blocks, K that ends inside one, token counts around a tile, every tile form, activations of -128
and subnormal scales.

Reference: the exact block dots with their scales, summed in float64. The kernel adds the nb exact terms of an output in
fp32 (possibly as four chains, joined in f64), so |error| <= (nb + 1) 2^-24 sum |terms| to first order; 2^-23 covers the rest."""
import numpy as np
import pytest

from lab import qwen_model as QM
from lab.hip import call, ptr
from oracle import quant as OQ
from test_gpu_prefill import test_mmq_qkv_rope_equals_finish as qkv_rope_equals_finish

pytestmark = pytest.mark.gpu


def problem(N, K, T, seed):
    rng = np.random.default_rng(seed)
    nb = K // 32
    qs = rng.integers(0, 256, (N, nb, 16), dtype=np.uint8)
    dw = (rng.standard_normal((N, nb)) * 0.01).astype(np.float16)
    dw[rng.random((N, nb)) < 0.1] = np.float16(3e-6)                    # subnormal in fp16
    xq = rng.integers(-128, 128, (T, K), dtype=np.int8)
    dx = (rng.random((T, nb)) * 0.02).astype(np.float16)
    dx[rng.random((T, nb)) < 0.1] = np.float16(1e-5)
    wb = np.concatenate([dw.view(np.uint8).reshape(N, nb, 2), qs], axis=2).reshape(-1, 18)
    return wb, dw, xq, dx


def reference(wb, dw, xq, dx, N, K, T):
    nb = K // 32
    qw = OQ.q4_0_blocks(wb)[1].reshape(N, K)
    sq = xq.reshape(T, nb, 32).astype(np.int64).sum(axis=2)
    y, mag = np.zeros((T, N)), np.zeros((T, N))
    for b in range(nb):
        dot = OQ.block_dots(qw[:, 32 * b:32 * b + 32], xq[:, 32 * b:32 * b + 32])[:, :, 0] - 8 * sq[:, b:b + 1]
        term = dot * dw[:, b].astype(np.float64)[None] * dx[:, b].astype(np.float64)[:, None]
        y += term
        mag += np.abs(term)
    return y, (nb + 1) * 2.0 ** -23 * mag


# dispatch: 49 to 255 tokens over a short K: RESID_FIX slices of one tile per workgroup (k_mmq_s32, f64 up to 64 tokens; one
# to three slices a wave), STORE from 65 tokens eight K waves; then up to 4096 rows one 32 x 32 tile per wave, with four K
# waves from 256 to 511 tokens (64 x 64 workgroups from 512, 128 x 32 past two per CU), the residual at every width; wider
# STORE 256 x 32 (77 and 200 tokens of 17920 rows), 128 x 64 or 128 x 128 (333 and 1100)
@pytest.mark.parametrize("N,K,T", [(64, 32, 49), (128, 224, 64), (1536, 1536, 50), (64, 32, 65), (128, 288, 97),
                                   (1536, 1536, 97), (1024, 2048, 100), (512, 4096, 250), (2048, 128, 255),
                                   (1536, 160, 200), (192, 8960, 70), (4096, 96, 255),
                                   (64, 32, 256), (128, 288, 257), (1536, 160, 333), (192, 96, 511), (4096, 64, 300),
                                   (128, 32, 512), (64, 96, 545), (192, 128, 513), (128, 160, 575),
                                   (128, 288, 576), (4096, 96, 513), (2048, 32, 1100), (4096, 288, 700),
                                   (4224, 32, 512), (4224, 160, 513), (4224, 416, 640), (4160, 96, 300),
                                   (17920, 96, 65), (17920, 32, 333), (17920, 288, 77), (17920, 416, 200), (17920, 288, 333),
                                   (17920, 160, 1100), (17920, 416, 400)])
def test_mmq_t32_store_and_resid(cuda, N, K, T):
    import torch
    wb, dw, xq, dx = problem(N, K, T, N + K + T)
    W = QM.Q4Mat(wb, N, K, "cuda")
    xq_d = torch.from_numpy(xq).cuda()
    xds_d = torch.from_numpy(np.stack([dx, np.zeros_like(dx)], -1)).cuda()
    ref, bound = reference(wb, dw, xq, dx, N, K, T)
    y = torch.full((T, N), float("nan"), device=cuda)
    call("q355_mmq_q4_0_q8_1", ptr(W.qs), ptr(W.d), N, K, ptr(xq_d), ptr(xds_d), T, 0, ptr(y), None, None, None, None, None)
    h0 = torch.from_numpy(np.random.default_rng(T).integers(-2 ** 40, 2 ** 40, (T, N))).cuda()
    h = h0.clone()
    call("q355_mmq_q4_0_q8_1", ptr(W.qs), ptr(W.d), N, K, ptr(xq_d), ptr(xds_d), T, 6, None, ptr(h), None, None, None, None)
    torch.cuda.synchronize()
    assert (np.abs(y.cpu().numpy() - ref) <= bound).all()
    got = (h - h0).cpu().numpy() / QM.FIX_SCALE                          # 2^-49: the fixed-point rounding
    assert (np.abs(got - ref) <= bound + 2.0 ** -48).all()


def chains(wb, dw, xq, dx, N, K, T, n):
    """The sum as n fp32 chains (block b in chain b % n, one rounding a step), joined in float64 in order: [T, N]."""
    nb = K // 32
    qw = OQ.q4_0_blocks(wb)[1].reshape(N, K)
    sq = xq.reshape(T, nb, 32).astype(np.int64).sum(axis=2)
    acc = np.zeros((n, T, N), np.float32)
    for b in range(nb):
        dot = OQ.block_dots(qw[:, 32 * b:32 * b + 32], xq[:, 32 * b:32 * b + 32])[:, :, 0] - 8 * sq[:, b:b + 1]
        s = dw[:, b].astype(np.float32)[None] * dx[:, b].astype(np.float32)[:, None]         # exact
        acc[b % n] = (s.astype(np.longdouble) * dot + acc[b % n].astype(np.longdouble)).astype(np.float32)
    y = np.zeros((T, N))
    for c in acc:
        y += c
    return y


# 256 to 511 tokens of fewer than 256 tiles of 128 x 64, and rows an odd multiple of 64 from 256 tokens on
@pytest.mark.parametrize("N,K,T", [(4224, 384, 256), (4608, 256, 448), (1536, 384, 333), (192, 1280, 513),
                                   (4160, 384, 520), (64, 256, 1030)])
def test_sums_of_four_chains(cuda, N, K, T):
    """These sizes add K as four chains, bit for bit: one chain would double the error of a long K."""
    import torch
    wb, dw, xq, dx = problem(N, K, T, N + K + T)
    W = QM.Q4Mat(wb, N, K, "cuda")
    xq_d = torch.from_numpy(xq).cuda()
    xds_d = torch.from_numpy(np.stack([dx, np.zeros_like(dx)], -1)).cuda()
    want = chains(wb, dw, xq, dx, N, K, T, 4)
    y = torch.full((T, N), float("nan"), device=cuda)
    call("q355_mmq_q4_0_q8_1", ptr(W.qs), ptr(W.d), N, K, ptr(xq_d), ptr(xds_d), T, 0, ptr(y), None, None, None, None, None)
    h = torch.zeros(T, N, dtype=torch.int64, device=cuda)
    call("q355_mmq_q4_0_q8_1", ptr(W.qs), ptr(W.d), N, K, ptr(xq_d), ptr(xds_d), T, 6, None, ptr(h), None, None, None, None)
    torch.cuda.synchronize()
    np.testing.assert_array_equal(y.cpu().numpy(), want.astype(np.float32))
    np.testing.assert_array_equal(h.cpu().numpy(), np.rint(want * QM.FIX_SCALE).astype(np.int64))


# the tied head of a batch: 16-token tiles up to 16 tokens, 64 x 32 (up to 65536 rows) or 128 x 32 up to 32, 128 x 64 up to 64
@pytest.mark.parametrize("N,K,T", [(32896, 32, 1), (32896, 160, 16), (32896, 32, 17), (32896, 160, 31), (32896, 288, 32),
                                   (65536, 544, 32), (65664, 32, 17), (65664, 160, 31), (65664, 288, 32), (32896, 96, 33),
                                   (32896, 1536, 63), (32896, 128, 64)])
def test_logits_and_their_partials(cuda, N, K, T):
    """Logits within the bound; every (max, lowest row) over 64 rows is that of the stored logits, also without them."""
    import torch
    wb, dw, xq, dx = problem(N, K, T, K + T)
    W = QM.Q4Mat(wb, N, K, "cuda")
    xq_d = torch.from_numpy(xq).cuda()
    xds_d = torch.from_numpy(np.stack([dx, np.zeros_like(dx)], -1)).cuda()
    ref, bound = reference(wb, dw, xq, dx, N, K, T)
    y = torch.full((T, N), float("nan"), device=cuda)
    for out in (ptr(y), None):
        pmax = torch.full((T, N // 64), float("nan"), device=cuda)
        pidx = torch.full((T, N // 64), -1, dtype=torch.int32, device=cuda)
        call("q355_mmq_q4_0_q8_1", ptr(W.qs), ptr(W.d), N, K, ptr(xq_d), ptr(xds_d), T, 5, out, None, None, None, ptr(pmax),
             ptr(pidx))
        torch.cuda.synchronize()
        got = y.cpu().numpy()
        tiles = got.reshape(T, N // 64, 64)
        np.testing.assert_array_equal(pmax.cpu().numpy(), tiles.max(axis=2))
        np.testing.assert_array_equal(pidx.cpu().numpy(), tiles.argmax(axis=2) + 64 * np.arange(N // 64))
    assert (np.abs(got - ref) <= bound).all()


@pytest.mark.parametrize("T", [256, 300, 448, 512, 577, 1100])
def test_mmq_t32_swiglu_is_the_quantized_store(cuda, T):
    """SWIGLU_Q8 gives the Q8_1 rule of silu(g) u: codes within one step of those of the STORE sums, and d equal to the
    fp16 of their block maximum / 127 within the error of the hardware exp2 and reciprocal (about 2e-6 relative)."""
    import torch
    N, K = 4224, 160
    wb, dw, xq, dx = problem(N, K, T, T)
    W = QM.Q4Mat(wb, N, K, "cuda")
    xq_d = torch.from_numpy(xq).cuda()
    xds_d = torch.from_numpy(np.stack([dx, np.zeros_like(dx)], -1)).cuda()
    y = torch.zeros(T, N, device=cuda)
    oq = torch.zeros(T, N // 2, dtype=torch.int8, device=cuda)
    ods = torch.zeros(T, N // 64, 2, dtype=torch.float16, device=cuda)
    args = ptr(W.qs), ptr(W.d), N, K, ptr(xq_d), ptr(xds_d), T
    call("q355_mmq_q4_0_q8_1", *args, 0, ptr(y), None, None, None, None, None)
    call("q355_mmq_q4_0_q8_1", *args, 7, None, None, ptr(oq), ptr(ods), None, None)
    torch.cuda.synchronize()
    g, u = y.double()[:, 0::2], y.double()[:, 1::2]
    m = (g / (1 + torch.exp(-g)) * u).cpu().numpy()
    q, d, s = OQ.quantize_q8_1(m.astype(np.float32))
    dq = np.abs(oq.cpu().numpy().astype(int) - q)
    assert dq.max() <= 1 and (dq > 0).mean() < 1e-3
    ds = ods.cpu().numpy().astype(np.float64)
    assert (np.abs(ds[..., 0] - d) <= 2.0 ** -10 * np.abs(d) + 2.0 ** -24).all()
    assert np.allclose(ds[..., 1], ds[..., 0] * oq.cpu().numpy().reshape(T, -1, 32).sum(2), rtol=2e-3, atol=1e-3)


# 64 x 32 with four K waves, 128 x 64; of 17920 rows 256 x 32 (77 and 200 tokens), 128 x 128 (333 and 1100), 128 x 64 (400)
@pytest.mark.parametrize("N,K,T", [(4224, 416, 300), (4224, 288, 448), (4224, 416, 577), (17920, 288, 77), (17920, 416, 200), (17920, 288, 333),
                                   (17920, 416, 1100), (17920, 288, 400)])
def test_mmq_t32_swiglu_is_the_quantized_product(cuda, N, K, T):
    """SWIGLU_Q8 gives the Q8_1 rule of silu(g) u of the float64 sums: codes within one step, few of them off, and d equal
    to the fp16 of their block maximum / 127 within the error of the hardware exp2 and reciprocal (about 2e-6 relative) and
    the sums (below 1e-5 of a block's largest value)."""
    import torch
    wb, dw, xq, dx = problem(N, K, T, T)
    W = QM.Q4Mat(wb, N, K, "cuda")
    xq_d = torch.from_numpy(xq).cuda()
    xds_d = torch.from_numpy(np.stack([dx, np.zeros_like(dx)], -1)).cuda()
    oq = torch.zeros(T, N // 2, dtype=torch.int8, device=cuda)
    ods = torch.zeros(T, N // 64, 2, dtype=torch.float16, device=cuda)
    call("q355_mmq_q4_0_q8_1", ptr(W.qs), ptr(W.d), N, K, ptr(xq_d), ptr(xds_d), T, 7, None, None, ptr(oq), ptr(ods), None, None)
    torch.cuda.synchronize()
    # whole Q8_1 blocks (64 rows): every wave's place in the widest workgroup, and the last
    blocks = np.r_[0:4, 65, N // 64 - 1]
    rows = (blocks[:, None] * 64 + np.arange(64)).reshape(-1)
    y, _ = reference(wb.reshape(N, -1, 18)[rows].reshape(-1, 18), dw[rows], xq, dx, len(rows), K, T)
    g, u = y[:, 0::2], y[:, 1::2]
    with np.errstate(over="ignore"):
        m = g / (1 + np.exp(-g)) * u
    q, d, _ = OQ.quantize_q8_1(m.astype(np.float32))
    got = oq.cpu().numpy().reshape(T, -1, 32)[:, blocks].reshape(T, -1)
    dq = np.abs(got.astype(int) - q)
    assert dq.max() <= 1 and (dq > 0).mean() < 1e-3
    ds = ods.cpu().numpy().astype(np.float64)[:, blocks]
    assert (np.abs(ds[..., 0] - d) <= 2.0 ** -10 * np.abs(d) + 2.0 ** -24).all()
    assert np.allclose(ds[..., 1], ds[..., 0] * got.reshape(T, -1, 32).sum(2), rtol=2e-3, atol=1e-3)


@pytest.mark.parametrize("T,seq_stride", [(33, 0), (64, 1), (65, 0), (255, 0), (256, 0), (511, 0), (512, 0)])
def test_qkv_rope_forms(cuda, T, seq_stride):
    """The fused QKV finish of every form (k_mmq_s32 in f64 and fp32, four K waves, one) against the split product."""
    qkv_rope_equals_finish(cuda, T, seq_stride)


# register-resident; k_mmq_s32 in f64 and fp32 (4, 12 and 16 slices); 64 x 64 below 256 tiles and from 512 tokens; four K
# waves; 128 x 32; wide: 128 x 64, 128 x 128, 256 x 32
@pytest.mark.parametrize("nh,nkv,K,T", [(12, 2, 512, 20), (12, 2, 512, 50), (12, 2, 1536, 40), (2, 1, 2048, 64),
                                        (12, 2, 512, 255), (2, 1, 2048, 100), (12, 2, 480, 100), (28, 4, 288, 77),
                                        (12, 2, 544, 300), (28, 4, 416, 300), (12, 2, 288, 520), (12, 2, 416, 1100),
                                        (28, 4, 160, 600), (40, 8, 160, 1100), (50, 4, 160, 544)])
def test_qkv_forms_against_float64(cuda, nh, nkv, K, T):
    """q, K and V of every form of the fused QKV: the float64 product, bias and RoPE rounded to fp16 once, within the
    products' fp32 bound."""
    import torch
    N, nq, nk = (nh + 2 * nkv) * 128, nh * 128, nkv * 128
    wb, dw, xq, dx = problem(N, K, T, N + K + T)
    W = QM.Q4Mat(wb, N, K, "cuda")
    rng = np.random.default_rng(T)
    bias = rng.standard_normal(N).astype(np.float32)
    pages = (T + 63) // 64
    table, pos = rng.permutation(pages).astype(np.int32), np.arange(T, dtype=np.int32)
    cos, sin = QM.rope_tables(64 * pages)
    t = lambda a: torch.from_numpy(a).cuda()  # noqa: E731
    kc = torch.zeros(pages, nkv, 64, 128, dtype=torch.float16, device=cuda)
    vc = torch.zeros_like(kc)
    q = torch.zeros(T, nq, dtype=torch.float16, device=cuda)
    q64 = torch.zeros(T, nq, dtype=torch.float64, device=cuda)
    args = [t(xq), t(np.stack([dx, np.zeros_like(dx)], -1)), t(bias), t(cos), t(sin), t(pos), t(table)]
    p = [ptr(a) for a in args]
    call("q355_mmq_qkv_rope", ptr(W.qs), ptr(W.d), N, K, p[0], p[1], T, *p[2:], pages, 0, ptr(kc), ptr(vc), ptr(q), ptr(q64),
         nh, nkv)
    torch.cuda.synchronize()
    y, bound = reference(wb, dw, xq, dx, N, K, T)
    y += bias.astype(np.float64)
    a, b = (y[:, :nq + nk].reshape(T, nh + nkv, 64, 2)[..., i] for i in (0, 1))         # device rows: pairs (d, d + 64)
    ea, eb = (bound[:, :nq + nk].reshape(T, nh + nkv, 64, 2)[..., i] for i in (0, 1))
    c, s = (f[pos][:, None].astype(np.float64) for f in (cos, sin))
    rot = np.concatenate([a * c - b * s, b * c + a * s], -1).reshape(T, -1)
    tol = np.concatenate([ea * np.abs(c) + eb * np.abs(s), eb * np.abs(c) + ea * np.abs(s)], -1).reshape(T, -1)
    rows = lambda x: x[table.astype(np.int64)].permute(0, 2, 1, 3).reshape(64 * pages, nk)[:T].cpu().numpy()  # noqa: E731
    got = np.concatenate([q.cpu().numpy(), rows(kc), rows(vc)], 1).astype(np.float64)
    want, tol = np.concatenate([rot, y[:, nq + nk:]], 1), np.concatenate([tol, bound[:, nq + nk:]], 1)
    assert (np.abs(got - want) <= tol + 2.0 ** -11 * (np.abs(want) + tol) + 2.0 ** -25).all()
    assert np.array_equal(q64.cpu().numpy(), got[:, :nq])
