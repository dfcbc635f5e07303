// Q6_K x Q8_1 LM head for decode batches on int8 MFMA (v_mfma_i32_16x16x32_i8), gfx950.
//
// Replaces the reference's batched Q6_K head (head_v2_source, lab/qwen_batched.py:681-833): logits of up to 32
// tokens over llama.cpp's Q6_K output.weight and the argmax partials of every 64 rows, read once from HBM.
//
// Weights come in the library's Q6_K planes (lab/gguf.py:tile_q6_k): per 16-row tile and 32-weight block, lo
// (16 B per row: low 4 bits of v_i and v_{i+16}), hi (8 B per row: bits 4-5 of v_{b+8j} at bits 2j of byte b),
// sc (2 int8 sub-block scales per row) and, per 256-weight super-block, d (fp16 per row); weight i of a block is
// d * sc[i / 16] * (v_i - 32).
//
// A wave takes one 16-row tile, four consecutive blocks at a time: lane l loads the whole row l % 16 of block l / 16, so
// the four blocks' planes are three contiguous loads (1 KB, 512 B and 128 B). The weight rows are the MFMA's columns, so
// a lane holds one row's scales and four tokens' products.
// Up to 8 tokens the weights stay where they are: k-group l / 16 is the lane's block, and row 4 u + t of the activation
// operand holds token t in k-group u alone (the others zero), so that lane l receives the products of ITS block with
// four tokens: per sub-block two MFMAs of 8 weights a lane. One fp32 chain per block index mod 4, added at the end.
// More tokens would repeat those MFMAs per four of them, so there a 4 x 4 transpose of the lane groups (eight lane
// swaps) spreads each block over its k-groups, and a block against 16 tokens is two MFMAs, the weights of the other
// sub-block zeroed. It keeps the same four chains, so that a sequence's logits have the same bits whatever the batch.
// Either way a sub-block is an exact int32 sum of (v - 32) q_x, and sc0 C0 + sc1 C1 (exact int32, |.| < 2^24) is scaled by
// d d_x (exact fp32 product) into fp32 accumulators.
//
// Workgroup: 8 or 4 waves, one tile each; every 4 waves are the 64 rows of one argmax partial. Activations of all
// tokens in LDS. Weights stay four groups ahead in registers.
// What bounds it: up to 8 tokens HBM (151936 x 1536: 191 MB, 37 us at the 5.15 TB/s of a large copy), more tokens VALU
// issue (five instructions per output and block). Three 2- to 8-byte loads a lane and BLOCK had kept the address unit
// busy, whatever the VALU did (us with logits at 8 / 16 / 32 tokens: 63 / 64 / 113; now 45 / 57 / 107).
#include "common.h"
#include "q355_kernels.h"

namespace q355 {

// bytes after each activation row: 32 zero ones for the lanes outside a token's k-group (up to 8 tokens), else 16, which
// put the 16 tokens of an operand read on different banks
__host__ __device__ constexpr int q6m_pad(bool own) { return own ? 32 : 16; }

struct Q6Group {                 // this lane's row of one of four consecutive blocks
  u32x4 lo;
  uint2 hi;
  int sc;                        // both int8 sub-block scales
  float d;
};

__device__ __forceinline__ void q6m_load(Q6Group& G, const GemvArgs& a, int tile, int grp, int nb, int lane) {
  const size_t r = ((size_t)tile * nb + 4 * grp) * 16 + lane;
  G.lo = __builtin_nontemporal_load((const u32x4*)a.qs + r);
  G.hi = ld_stream8((const uint2*)a.qhi + r);
  G.sc = ((const short*)a.qsc)[r];
  G.d = __half2float(a.d[((size_t)tile * (nb / 8) + grp / 2) * 16 + (lane & 15)]);
}

// 4 bytes v = l | h (l in 0..15, h in {0, 16, 32, 48}) -> v - 32 in two's complement, with no carry between bytes
__device__ __forceinline__ unsigned q6m_signed(unsigned l, unsigned h) {
  return (((l & 0x0F0F0F0Fu) | (h & 0x30303030u)) + 0x60606060u) ^ 0x80808080u;
}
__device__ __forceinline__ long pack64(unsigned x, unsigned y) { return (long)(((unsigned long)y << 32) | x); }

// weights 8 m .. 8 m + 7 of this lane's row (bits 2 m .. 2 m + 1 of the hi bytes)
__device__ __forceinline__ void q6m_weights(const Q6Group& G, long (&w)[4]) {
  const u32x4 L = G.lo;
  const uint2 h = G.hi;
  w[0] = pack64(q6m_signed(L.x, h.x << 4), q6m_signed(L.y, h.y << 4));
  w[1] = pack64(q6m_signed(L.z, h.x << 2), q6m_signed(L.w, h.y << 2));
  w[2] = pack64(q6m_signed(L.x >> 4, h.x), q6m_signed(L.y >> 4, h.y));
  w[3] = pack64(q6m_signed(L.z >> 4, h.x >> 2), q6m_signed(L.w >> 4, h.y >> 2));
}

// x of lanes 32 .. 63 <-> y of lanes 0 .. 31, and within each half x of rows 16 .. 31 <-> y of rows 0 .. 15
__device__ __forceinline__ void swap32(unsigned& x, unsigned& y) {
  const auto r = __builtin_amdgcn_permlane32_swap(x, y, false, false);
  x = r[0];
  y = r[1];
}
__device__ __forceinline__ void swap16(unsigned& x, unsigned& y) {
  const auto r = __builtin_amdgcn_permlane16_swap(x, y, false, false);
  x = r[0];
  y = r[1];
}
// w[m] of lane group u <-> w[u] of lane group m
__device__ __forceinline__ void transpose4(unsigned (&w)[4]) {
  swap32(w[0], w[2]);
  swap32(w[1], w[3]);
  swap16(w[0], w[1]);
  swap16(w[2], w[3]);
}

// Four blocks against TG groups of 16 tokens: xl = this lane's token and k-group, xd = its accumulators' tokens; block u
// adds to the chain acc[u]
template <int TG>
__device__ __forceinline__ void q6m_group_t(const Q6Group& G, const int8_t* xl, int xstride, const float* xd, bool sub0,
                                            float (&acc)[4][TG][4]) {
  constexpr int TT = 16 * TG;
  long w[4];
  q6m_weights(G, w);
  unsigned x[4], y[4], sc[4];
#pragma unroll
  for (int m = 0; m < 4; ++m) {
    x[m] = (unsigned)w[m];
    y[m] = (unsigned)((unsigned long)w[m] >> 32);
    sc[m] = (unsigned)G.sc;                                         // after the transpose: lane group m's
  }
  transpose4(x);
  transpose4(y);
  transpose4(sc);
  const v4i zero = {0, 0, 0, 0};
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    const long b0 = sub0 ? pack64(x[u], y[u]) : 0l, b1 = sub0 ? 0l : pack64(x[u], y[u]);
    const int sc0 = (int)(signed char)sc[u], sc1 = (int)sc[u] >> 8;
#pragma unroll
    for (int g = 0; g < TG; ++g) {
      const long xa = *(const long*)(xl + 16 * g * xstride + 32 * u);
      const float4 dx = *(const float4*)(xd + u * TT + 16 * g);
      const v4i c0 = __builtin_amdgcn_mfma_i32_16x16x32_i8(xa, b0, zero, 0, 0, 0);
      const v4i c1 = __builtin_amdgcn_mfma_i32_16x16x32_i8(xa, b1, zero, 0, 0, 0);
      const float s[4] = {G.d * dx.x, G.d * dx.y, G.d * dx.z, G.d * dx.w};
#pragma unroll
      for (int v = 0; v < 4; ++v)
        acc[u][g][v] = fmaf(s[v], (float)(__mul24(sc0, c0[v]) + __mul24(sc1, c1[v])), acc[u][g][v]);
    }
  }
}

// Four blocks against TQ quads of tokens, each lane its own block
template <int TQ>
__device__ __forceinline__ void q6m_group(const Q6Group& G, const int8_t* xl, int xstride, const float* xd, float (&acc)[TQ][4]) {
  long w[4];
  q6m_weights(G, w);
  const int sc0 = (int)(signed char)G.sc, sc1 = G.sc >> 8;
  const v4i zero = {0, 0, 0, 0};
#pragma unroll
  for (int q = 0; q < TQ; ++q) {
    const u32x4 x0 = *(const u32x4*)(xl + 4 * q * xstride), x1 = *(const u32x4*)(xl + 4 * q * xstride + 16);
    const float4 dx = *(const float4*)(xd + 4 * q);
    v4i c0 = __builtin_amdgcn_mfma_i32_16x16x32_i8(pack64(x0.x, x0.y), w[0], zero, 0, 0, 0);
    v4i c1 = __builtin_amdgcn_mfma_i32_16x16x32_i8(pack64(x1.x, x1.y), w[2], zero, 0, 0, 0);
    c0 = __builtin_amdgcn_mfma_i32_16x16x32_i8(pack64(x0.z, x0.w), w[1], c0, 0, 0, 0);
    c1 = __builtin_amdgcn_mfma_i32_16x16x32_i8(pack64(x1.z, x1.w), w[3], c1, 0, 0, 0);
    const float s[4] = {G.d * dx.x, G.d * dx.y, G.d * dx.z, G.d * dx.w};
#pragma unroll
    for (int v = 0; v < 4; ++v)
      acc[q][v] = fmaf(s[v], (float)(__mul24(sc0, c0[v]) + __mul24(sc1, c1[v])), acc[q][v]);
  }
}

// TG groups of 16 tokens, or (0) up to 8 tokens in the first form; NW waves
template <int TG, int NW>
__global__ void __launch_bounds__(NW * 64) k_mmq_q6k_logits(const GemvArgs a) {
  extern __shared__ __align__(16) char q6m_lds[];
  constexpr bool OWN = TG == 0;
  constexpr int AHEAD = 4;                                         // groups of four blocks in flight per wave
  constexpr int TT = OWN ? 8 : 16 * TG, TQ = OWN ? 2 : TG;         // TQ accumulator quads a lane
  const int K = a.K, nb = K / 32, ng = nb / 4, xstride = K + q6m_pad(OWN);
  int8_t* xs = (int8_t*)q6m_lds;                                   // [TT][K + 32]
  float* xd = (float*)(q6m_lds + (size_t)TT * xstride);            // [nb][TT]
  __shared__ float pv[NW][TT];
  __shared__ int pi[NW][TT];
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, li = lane & 15, lg = lane >> 4;
  const int tile = blockIdx.x * NW + wv;
  Q6Group G[AHEAD];
#pragma unroll
  for (int i = 0; i < AHEAD; ++i) q6m_load(G[i], a, tile, min(i, ng - 1), nb, lane);
  // stage the activations (tokens past T are zero)
  const int pieces = xstride / 16;
  for (int e = threadIdx.x; e < TT * pieces; e += NW * 64) {
    const int j = e / pieces, c = e % pieces;
    const uint4 v = j < a.T && c < K / 16 ? *(const uint4*)(a.xq + (size_t)j * K + 16 * c) : make_uint4(0, 0, 0, 0);
    *(uint4*)(xs + (size_t)j * xstride + 16 * c) = v;
  }
  for (int e = threadIdx.x; e < TT * nb; e += NW * 64) {
    const int j = e / nb, b = e % nb;
    xd[b * TT + j] = j < a.T ? __low2float(a.xds[(size_t)j * nb + b]) : 0.f;
  }
  __syncthreads();
  // OWN: operand row li = token li % 4 in k-group li / 4; the other lanes of the row read its zero bytes, at every group.
  // Else operand row li = token li, k-group lg.
  const bool own = (li >> 2) == lg;
  const int8_t* xl = OWN ? xs + (size_t)(li & 3) * xstride + (own ? 32 * lg : K) : xs + (size_t)li * xstride + 8 * lg;
  const int step = !OWN || own ? 128 : 0;
  const float* xdl = OWN ? xd + lg * TT : xd + 4 * lg;
  constexpr int NC = OWN ? 1 : 4;                                  // chains in this lane's registers
  float acc[NC][TQ][4];
#pragma unroll
  for (int c = 0; c < NC; ++c)
#pragma unroll
    for (int q = 0; q < TQ; ++q)
#pragma unroll
      for (int v = 0; v < 4; ++v) acc[c][q][v] = 0.f;
  for (int g = 0; g < ng; g += AHEAD)
#pragma unroll
    for (int i = 0; i < AHEAD; ++i)
      if (g + i < ng) {                                             // uniform
        if constexpr (OWN) q6m_group<TQ>(G[i], xl, xstride, xdl, acc[0]);
        else q6m_group_t<TG>(G[i], xl, xstride, xdl, lg < 2, acc);
        if (g + i + AHEAD < ng) q6m_load(G[i], a, tile, g + i + AHEAD, nb, lane);
        xl += step;
        xdl += 4 * TT;
      }
  // logits (optional) and the (max, lowest row) of this wave's 16 rows
  const int row = tile * 16 + li;
  const auto finish = [&](int tok, float bv) {
    int bi = row;
    if (a.y && tok < a.T) a.y[(size_t)tok * a.N + row] = bv;
    amax_dpp<DPP_XOR1>(bv, bi);
    amax_dpp<DPP_XOR2>(bv, bi);
    amax_dpp<DPP_HALF_MIRROR>(bv, bi);
    amax_dpp<DPP_MIRROR>(bv, bi);
    if (li == 0) { pv[wv][tok] = bv; pi[wv][tok] = bi; }
  };
#pragma unroll
  for (int q = 0; q < TQ; ++q) {
    if constexpr (OWN) {                                            // the sum of the four chains; lane group lg takes token lg
      float s[4];
#pragma unroll
      for (int v = 0; v < 4; ++v) s[v] = xsum32(xsum16(acc[0][q][v]));
      finish(4 * q + lg, lg == 0 ? s[0] : lg == 1 ? s[1] : lg == 2 ? s[2] : s[3]);
    } else {
#pragma unroll
      for (int v = 0; v < 4; ++v)
        finish(16 * q + 4 * lg + v, (acc[0][q][v] + acc[1][q][v]) + (acc[2][q][v] + acc[3][q][v]));
    }
  }
  __syncthreads();
  if (threadIdx.x < TT * (NW / 4)) {
    const int tok = threadIdx.x % TT, q = threadIdx.x / TT;
    if (tok < a.T) {
      float bv = pv[4 * q][tok];
      int bi = pi[4 * q][tok];
#pragma unroll
      for (int w = 1; w < 4; ++w)                                  // rows increase with w: '>' keeps the lowest
        if (pv[4 * q + w][tok] > bv) { bv = pv[4 * q + w][tok]; bi = pi[4 * q + w][tok]; }
      const int np = a.N / 64;
      a.pmax[(size_t)tok * np + blockIdx.x * (NW / 4) + q] = bv;
      a.pidx[(size_t)tok * np + blockIdx.x * (NW / 4) + q] = bi;
    }
  }
}

}  // namespace q355
