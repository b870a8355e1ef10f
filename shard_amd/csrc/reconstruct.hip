// Full fp16 reconstruction of the compressed cache for unfused consumers
// (_ensure_dequant, cache.py:87-124) and the stream dequantizer
// (_dequant_stream, cache.py:243-279).  Off the decode hot path: used on the
// first decode step (compression happens inside it), for q_len > 1 extends and
// for callers that read layer.keys / layer.values.
#include <algorithm>

#include "common.h"

namespace shard {

constexpr int kRcTok = 32;   // tokens per tile

// The rebuilt rows of one call: K and V go to rows row0 + t, t < n_comp, of
// (B, G, T, D) buffers.
struct RebuildOut {
  uint16_t *k, *v;
  int64_t T;
  int32_t row0;
};

// ---- K on MFMA (ranks that are multiples of 32 up to 256).
// One 512-thread workgroup holds the basis of 8 / (HD / 64) kv heads in
// registers (a wave: rows [32 j, 32 j + 32) and HD/2 + the same of its head,
// the two halves of 32 RoPE pairs, all ranks) and walks units of 32 tokens x
// one batch row, the batch rows of a token tile in turn.  Per unit:
//   stage   the packed coefficients become fp16(nib * cs) rows in LDS (once
//           per workgroup, the next unit's loads in flight during this one);
//           the phases (cos, sin)(fl(pos theta)) of a new token tile too.
//   MFMA    2 x KS 32x32x16 f16 per wave, B = the staged rows (columns =
//           tokens): element i of lane half hh is pair 32 j + 8 (i / 4) +
//           4 hh + i % 4 of token col = lane % 32, both halves in one lane.
//   store   rounding, mean and rotation in registers; the lane halves swap so
//           that each lane stores 8 consecutive dims (16 bytes).
// Every value is rounded as in the general kernel below; only the order of
// the fp32 sums over the ranks differs.  Bound by the 2 x 256 bytes written
// per token and head.  8,124 tokens x 8 heads of 128 dims, rank 192: the
// scalar kernel's dot products from LDS took 242 us; a whole layer with V and
// the segments (one torch.cat pass over each of K and V before) went from 290
// to 27 us, batch 4 x 2,933 x 8 heads of 64 from 202 to 22.8 us.  Not kept: the
// basis rows turned into operand order through LDS (30.2 us).
template <int HD, int KS>
struct RebuildLds {
  static constexpr int kRow = 16 * KS + 8;     // halves per coefficient row: 16 bytes of padding
  uint16_t cf[2][kRcTok * kRow];
  float4 ph[2][2][HD / 8][kRcTok];             // [buffer][cos, sin][pair / 4][token]
  uint16_t cs[16 * KS];
};

// 8 packed nibbles -> fp16(nib - 8) * cs, rounded to fp16 (rank order)
__device__ __forceinline__ uint4 nib8_times(uint32_t x, const uint4 cs) {
  const uint32_t c[4] = {cs.x, cs.y, cs.z, cs.w};
  uint32_t r[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    // 1024 + n in both halves (exact), less 1032
    const uint32_t n2 = ((x >> (8 * e)) & 15u) | (((x >> (8 * e + 4)) & 15u) << 16) | 0x64006400u;
    const half2v off = {(half_t)1032.f, (half_t)1032.f};
    const half2v v = (__builtin_bit_cast(half2v, n2) - off) * __builtin_bit_cast(half2v, c[e]);
    r[e] = __builtin_bit_cast(uint32_t, v);
  }
  return make_uint4(r[0], r[1], r[2], r[3]);
}

template <int HD, int KS>
__global__ __launch_bounds__(512, 1)
void k_rebuild_k(const uint8_t* __restrict__ coef, const uint16_t* __restrict__ cs,
                 const uint16_t* __restrict__ basis, const uint16_t* __restrict__ mean,
                 const float* __restrict__ inv_freq, int B, int G, int n_comp, int cstart,
                 int units_per_wg, RebuildOut out) {
  constexpr int NJ = HD / 64;       // waves per head
  constexpr int HPW = 8 / NJ;       // heads per workgroup
  constexpr int rank = 16 * KS;
  constexpr int kDw = 2 * KS;       // packed dwords per row
  constexpr int kPer = (kRcTok * kDw + 511) / 512;
  __shared__ __align__(16) RebuildLds<HD, KS> L;
  const int tid = threadIdx.x, lane = tid & 63, col = lane & 31, hh = lane >> 5;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int g0 = (int)blockIdx.y * HPW + w / NJ, j = w % NJ;
  const int g = min(g0, G - 1);     // waves past the last head compute and do not store
  const int n_tiles = (n_comp + kRcTok - 1) / kRcTok;
  const int n_units = n_tiles * B;  // unit = token tile * B + batch row
  const int u0 = (int)blockIdx.x * units_per_wg, u1 = min(u0 + units_per_wg, n_units);

  half8 a0[KS], a1[KS];
  uint2 mc[4], md[4];
  {
    const uint16_t* r0 = basis + ((int64_t)g * HD + 32 * j + col) * rank + 8 * hh;
#pragma unroll
    for (int s = 0; s < KS; ++s) {
      a0[s] = __builtin_bit_cast(half8, *(const uint4*)(r0 + 16 * s));
      a1[s] = __builtin_bit_cast(half8, *(const uint4*)(r0 + (HD / 2) * rank + 16 * s));
    }
    const uint16_t* m0 = mean + g * HD + 32 * j + 4 * hh;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      mc[q] = *(const uint2*)(m0 + 8 * q);
      md[q] = *(const uint2*)(m0 + HD / 2 + 8 * q);
    }
  }
  if (tid < rank / 2) ((uint32_t*)L.cs)[tid] = ((const uint32_t*)cs)[tid];

  uint32_t pk[kPer];
  auto load_unit = [&](int u) {
    const int t0 = (u / B) * kRcTok, b = u % B;
#pragma unroll
    for (int m = 0; m < kPer; ++m) {
      const int i = tid + 512 * m, t = t0 + i / kDw;
      pk[m] = 0x88888888u;          // nibble 8: coefficient 0
      if (i < kRcTok * kDw && t < n_comp)
        pk[m] = ((const uint32_t*)coef)[((int64_t)b * n_comp + t) * kDw + i % kDw];
    }
  };
  auto stage_unit = [&](uint16_t* cf) {
#pragma unroll
    for (int m = 0; m < kPer; ++m) {
      const int i = tid + 512 * m, dw = i % kDw;
      if (i < kRcTok * kDw)
        *(uint4*)(cf + (i / kDw) * RebuildLds<HD, KS>::kRow + 8 * dw) =
            nib8_times(pk[m], *(const uint4*)(L.cs + 8 * dw));
    }
  };
  auto phases = [&](int tile, int buf) {
#pragma unroll 1
    for (int e = tid; e < kRcTok * HD / 2; e += 512) {
      const int t = e % kRcTok, i = e / kRcTok;
      float sn, cn;
      sincosf(__fmul_rn((float)(cstart + tile * kRcTok + t), inv_freq[i]), &sn, &cn);
      ((float*)&L.ph[buf][0][i >> 2][t])[i & 3] = cn;
      ((float*)&L.ph[buf][1][i >> 2][t])[i & 3] = sn;
    }
  };

  if (u0 < u1) load_unit(u0);
  __syncthreads();                  // L.cs
  if (u0 < u1) {
    stage_unit(L.cf[0]);
    phases(u0 / B, 0);
  }
  __syncthreads();
  int cur = 0, pc = 0;
  for (int u = u0; u < u1; ++u) {
    const int tile = u / B, b = u % B, t = tile * kRcTok + col;
    if (u + 1 < u1) load_unit(u + 1);
    float16v c = {}, d = {};
    const uint16_t* cf = L.cf[cur] + col * RebuildLds<HD, KS>::kRow + 8 * hh;
#pragma unroll
    for (int s = 0; s < KS; ++s) {
      const half8 bv = *(const half8*)(cf + 16 * s);
      c = __builtin_amdgcn_mfma_f32_32x32x16_f16(a0[s], bv, c, 0, 0, 0);
      d = __builtin_amdgcn_mfma_f32_32x32x16_f16(a1[s], bv, d, 0, 0, 0);
    }
    uint2 oc[4], od[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const float4 c4 = L.ph[pc][0][8 * j + 2 * q + hh][col];
      const float4 s4 = L.ph[pc][1][8 * j + 2 * q + hh][col];
      const float cn[4] = {c4.x, c4.y, c4.z, c4.w}, sn[4] = {s4.x, s4.y, s4.z, s4.w};
      const uint32_t mcw[2] = {mc[q].x, mc[q].y}, mdw[2] = {md[q].x, md[q].y};
      uint32_t ow[2], pw[2];
#pragma unroll
      for (int e2 = 0; e2 < 2; ++e2) {
        uint32_t lo_hi[2] = {0, 0}, lo_hi_d[2] = {0, 0};
#pragma unroll
        for (int e1 = 0; e1 < 2; ++e1) {
          const int e = 2 * e2 + e1;
          // recon = fp16(coeffs @ basis^T) + mean, both fp16
          const float cm = h2f(f2h(h2f(f2h(c[4 * q + e])) + h2f((uint16_t)(mcw[e2] >> (16 * e1)))));
          const float dm = h2f(f2h(h2f(f2h(d[4 * q + e])) + h2f((uint16_t)(mdw[e2] >> (16 * e1)))));
          // reapply_rope: k*cos + rotate_half(k)*sin with fp32 phase fl(pos*theta)
          lo_hi[e1] = f2h(__fsub_rn(__fmul_rn(cm, cn[e]), __fmul_rn(dm, sn[e])));
          lo_hi_d[e1] = f2h(__fadd_rn(__fmul_rn(dm, cn[e]), __fmul_rn(cm, sn[e])));
        }
        ow[e2] = lo_hi[0] | (lo_hi[1] << 16);
        pw[e2] = lo_hi_d[0] | (lo_hi_d[1] << 16);
      }
      oc[q] = make_uint2(ow[0], ow[1]);
      od[q] = make_uint2(pw[0], pw[1]);
    }
    if (g0 < G && t < n_comp) {
      uint16_t* o = out.k + (((int64_t)b * G + g) * out.T + out.row0 + t) * HD + 32 * j + 8 * hh;
#pragma unroll
      for (int q = 0; q < 4; q += 2) {
        // lane half 0 collects dims 8 q .. 8 q + 7, half 1 dims 8 q + 8 .. 8 q + 15
        const auto x0 = __builtin_amdgcn_permlane32_swap(oc[q].x, oc[q + 1].x, false, false);
        const auto y0 = __builtin_amdgcn_permlane32_swap(oc[q].y, oc[q + 1].y, false, false);
        const auto x1 = __builtin_amdgcn_permlane32_swap(od[q].x, od[q + 1].x, false, false);
        const auto y1 = __builtin_amdgcn_permlane32_swap(od[q].y, od[q + 1].y, false, false);
        *(uint4*)(o + 8 * q) = make_uint4(x0[0], y0[0], x0[1], y0[1]);
        *(uint4*)(o + HD / 2 + 8 * q) = make_uint4(x1[0], y1[0], x1[1], y1[1]);
      }
    }
    if (u + 1 < u1) {
      stage_unit(L.cf[cur ^ 1]);
      if ((u + 1) / B != tile) phases((u + 1) / B, pc ^ 1);
    }
    __syncthreads();
    cur ^= 1;
    if (u + 1 < u1 && (u + 1) / B != tile) pc ^= 1;
  }
}

// K of other ranks, or unaligned operands: block = (b, 32-token tile, kv head
// g); 256 threads = 32 tokens x 8 lanes, each lane owns HD / 16 RoPE pairs of
// its token.  The head's basis rows and the tile's coefficients are staged in
// LDS.
template <int HD>
__global__ __launch_bounds__(256)
void k_reconstruct_k(const uint8_t* __restrict__ coef, const uint16_t* __restrict__ cs,
                     const uint16_t* __restrict__ basis, const uint16_t* __restrict__ mean,
                     const float* __restrict__ inv_freq, int B, int G, int rank, int n_comp,
                     int cstart, RebuildOut out) {
  constexpr int kRcHD = HD;
  extern __shared__ __align__(16) unsigned char smem[];
  uint16_t* cf = (uint16_t*)smem;                  // [kRcTok][rank] fp16(nib*cs)
  uint16_t* bb = cf + kRcTok * rank;               // [HD][rank] basis rows of head g
  const int tid = threadIdx.x;
  const int g = blockIdx.y, b = blockIdx.z;
  const int t0 = blockIdx.x * kRcTok;
  const int row_bytes = rank / 2;
  for (int i = tid; i < kRcTok * rank; i += 256) {
    const int tt = i / rank, r = i - tt * rank;
    const int t = t0 + tt;
    uint16_t v = 0;
    if (t < n_comp) {
      const uint8_t byte = coef[((int64_t)b * n_comp + t) * row_bytes + (r >> 1)];
      const int nib = (r & 1) ? (byte >> 4) : (byte & 15);
      // fp16(nib - 8) * fp16(cs) rounded to fp16, as the reference's fp16 multiply
      v = f2h((float)(nib - 8) * h2f(cs[r]));
    }
    cf[i] = v;
  }
  for (int i = tid; i < kRcHD * rank; i += 256)
    bb[i] = basis[(int64_t)g * kRcHD * rank + i];
  __syncthreads();
  const int tt = tid >> 3, part = tid & 7;
  const int t = t0 + tt;
  if (t >= n_comp) return;
  const uint16_t* cr = cf + tt * rank;
  const int pos = cstart + t;
  constexpr int PL = HD / 16;  // pairs per lane
#pragma unroll 1
  for (int u = 0; u < PL; ++u) {
    const int i = part * PL + u;  // pair index 0 .. HD/2 - 1
    float c = 0.f, d = 0.f;
    const uint16_t* b0 = bb + i * rank;
    const uint16_t* b1 = bb + (i + HD / 2) * rank;
    for (int r = 0; r < rank; ++r) {
      const float cv = h2f(cr[r]);
      c += cv * h2f(b0[r]);
      d += cv * h2f(b1[r]);
    }
    // recon = fp16(coeffs @ basis^T) + mean, both fp16
    const float cm = h2f(f2h(h2f(f2h(c)) + h2f(mean[g * kRcHD + i])));
    const float dm = h2f(f2h(h2f(f2h(d)) + h2f(mean[g * kRcHD + i + HD / 2])));
    // reapply_rope: k*cos + rotate_half(k)*sin with fp32 phase fl(pos*theta)
    float sn, csn;
    sincosf(__fmul_rn((float)pos, inv_freq[i]), &sn, &csn);
    uint16_t* o = out.k + (((int64_t)b * G + g) * out.T + out.row0 + t) * kRcHD;
    o[i] = f2h(__fsub_rn(__fmul_rn(cm, csn), __fmul_rn(dm, sn)));
    o[i + HD / 2] = f2h(__fadd_rn(__fmul_rn(dm, csn), __fmul_rn(cm, sn)));
  }
}

// The fp16 rows around the compressed span, in output order: sink, then (after
// the span) window, stream, decode tokens.  Stream rows are (tokens, B, G, D).
struct RebuildSegs {
  const uint16_t *k[4], *v[4];
  int32_t n[4], dec_stride, total, vec;  // vec: every pointer is 16-byte aligned
};

template <int HD>
__device__ __forceinline__ void rebuild_copy(const RebuildSegs& sg, const RebuildOut& out, int B,
                                             int G, int n_comp, int64_t bg, int blk) {
  constexpr int CH = HD / 8;        // 8-value chunks per row
  const int i = blk * 256 + (int)threadIdx.x;
  int x = i / CH;
  const int c = 8 * (i % CH);
  if (x >= sg.total) return;
  const int64_t orow = x < sg.n[0] ? x : x + n_comp;
  int seg = 0;
  while (seg < 3 && x >= sg.n[seg]) x -= sg.n[seg++];
  const int64_t row = seg == 2 ? (int64_t)x * B * G + bg
                               : bg * (seg == 3 ? sg.dec_stride : sg.n[seg]) + x;
  const uint16_t *ks = sg.k[seg] + row * HD + c, *vs = sg.v[seg] + row * HD + c;
  uint16_t* ko = out.k + (bg * out.T + orow) * HD + c;
  uint16_t* vo = out.v + (bg * out.T + orow) * HD + c;
  if (sg.vec) {
    *(uint4*)ko = *(const uint4*)ks;
    *(uint4*)vo = *(const uint4*)vs;
  } else {
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      ko[e] = ks[e];
      vo[e] = vs[e];
    }
  }
}

// V: fp16(hadamard(cb[idx] * ch)), fp32 math; subvectors of gs = 2^LG values
// (D / gs indices per token), a codebook of cbn rows (an index past it reads
// its last row).  A lane holds 16 consecutive dims, HD / 16 lanes a row:
// 16 >> LG index bytes in one load, the codebook from LDS, four butterfly
// stages in registers and log2(HD / 16) across lanes, 32 bytes stored.
// Division by sqrt(HD) through its reciprocal (exact for finite values, see
// div_by_rcp); a wave that holds a non-finite value divides instead.  Blocks
// past the rows' copy the fp16 segments.  vec: indices and output are aligned
// for the wide accesses (otherwise element by element).  Bound by the 256 bytes written per
// row; one wave per row with a 2-byte store per lane took 18.7 us at
// 8,124 x 8 rows of 128.
constexpr int kRvSteps = 1;  // row groups per wave: a whole 8K layer 27.0 us, with 4 29.3, with 8 31.7
template <int HD, int LG>
__global__ __launch_bounds__(256)
void k_rebuild_v(const uint8_t* __restrict__ vidx, const uint16_t* __restrict__ vcb,
                 const uint16_t* __restrict__ vch, int64_t BG, int B, int G, int n_comp, int cbn,
                 int row_blocks, int vec, RebuildSegs sg, RebuildOut out) {
  constexpr int LR = HD / 16, RW = 64 / LR, NI = 16 >> LG, GS = 1 << LG;
  __shared__ __align__(16) uint16_t cb[256 * GS];
  const int tid = threadIdx.x, lane = tid & 63;
  if ((int)blockIdx.x >= row_blocks) {
    for (int64_t bg = blockIdx.y; bg < BG; bg += gridDim.y)
      rebuild_copy<HD>(sg, out, B, G, n_comp, bg, (int)blockIdx.x - row_blocks);
    return;
  }
  for (int i = tid; i < 256 * GS; i += 256) cb[i] = vcb[min(i >> LG, cbn - 1) * GS + (i & (GS - 1))];
  __syncthreads();
  const int lr = lane % LR;
  const float root = (float)sqrt((double)HD), rcp = div_rn(1.f, root);
  const int rbase = ((int)blockIdx.x * 4 + (tid >> 6)) * (RW * kRvSteps) + lane / LR;
  for (int64_t bg = blockIdx.y; bg < BG; bg += gridDim.y) {
    float ch[16];
#pragma unroll
    for (int e = 0; e < 16; ++e) ch[e] = h2f(vch[bg * HD + 16 * lr + e]);
    uint32_t iw[kRvSteps][(NI + 3) / 4];
#pragma unroll
    for (int m = 0; m < kRvSteps; ++m) {   // every index load of the wave in flight at once
      const int t = min(rbase + RW * m, n_comp - 1);
      const uint8_t* ix = vidx + (bg * n_comp + t) * (int64_t)(HD >> LG) + NI * lr;
      if (!vec) {
#pragma unroll
        for (int i = 0; i < NI; ++i)
          iw[m][i >> 2] = (i & 3 ? iw[m][i >> 2] : 0u) | ((uint32_t)ix[i] << (8 * (i & 3)));
      } else if constexpr (NI == 16) {
        const uint4 q = *(const uint4*)ix;
        iw[m][0] = q.x; iw[m][1] = q.y; iw[m][2] = q.z; iw[m][3] = q.w;
      } else if constexpr (NI == 8) {
        const uint2 q = *(const uint2*)ix;
        iw[m][0] = q.x; iw[m][1] = q.y;
      } else if constexpr (NI == 4) {
        iw[m][0] = *(const uint32_t*)ix;
      } else {
        iw[m][0] = *(const uint16_t*)ix;
      }
    }
#pragma unroll
    for (int m = 0; m < kRvSteps; ++m) {
      const int t = rbase + RW * m;
      float x[16];
#pragma unroll
      for (int i = 0; i < NI; ++i) {
        const int e = (int)((iw[m][i >> 2] >> (8 * (i & 3))) & 255u);
        uint32_t cw[4] = {0u, 0u, 0u, 0u};
        if constexpr (GS == 8) {
          const uint4 q = *(const uint4*)(cb + 8 * e);
          cw[0] = q.x; cw[1] = q.y; cw[2] = q.z; cw[3] = q.w;
        } else if constexpr (GS == 4) {
          const uint2 q = *(const uint2*)(cb + 4 * e);
          cw[0] = q.x; cw[1] = q.y;
        } else if constexpr (GS == 2) {
          cw[0] = *(const uint32_t*)(cb + 2 * e);
        } else {
          cw[0] = cb[e];
        }
#pragma unroll
        for (int k = 0; k < GS; ++k)
          x[GS * i + k] = __fmul_rn(h2f((uint16_t)(cw[k >> 1] >> (16 * (k & 1)))), ch[GS * i + k]);
      }
#pragma unroll
      for (int h = 1; h < 16; h <<= 1) {
#pragma unroll
        for (int e = 0; e < 16; ++e) {
          if ((e & h) == 0) {
            const float a = x[e], b = x[e | h];
            x[e] = add_rn(a, b);
            x[e | h] = sub_rn(a, b);
          }
        }
      }
      fwht_lane_stage<1>(x, lane);
      fwht_lane_stage<2>(x, lane);
      if constexpr (HD >= 128) fwht_lane_stage<4>(x, lane);
      if constexpr (HD >= 256) fwht_lane_stage<8>(x, lane);
      bool odd = false;
#pragma unroll
      for (int e = 0; e < 16; ++e) odd |= !(fabsf(x[e]) < INFINITY);
      uint32_t ow[8];
      if (__builtin_amdgcn_ballot_w64(odd) == 0) {
#pragma unroll
        for (int e = 0; e < 8; ++e)
          ow[e] = (uint32_t)f2h_opaque(div_by_rcp(x[2 * e], root, rcp)) |
                  ((uint32_t)f2h_opaque(div_by_rcp(x[2 * e + 1], root, rcp)) << 16);
      } else {
#pragma unroll
        for (int e = 0; e < 8; ++e)
          ow[e] = (uint32_t)f2h_opaque(div_rn(x[2 * e], root)) |
                  ((uint32_t)f2h_opaque(div_rn(x[2 * e + 1], root)) << 16);
      }
      if (t < n_comp) {
        uint16_t* o = out.v + (bg * out.T + out.row0 + t) * HD + 16 * lr;
        if (vec) {
          *(uint4*)o = make_uint4(ow[0], ow[1], ow[2], ow[3]);
          *(uint4*)(o + 8) = make_uint4(ow[4], ow[5], ow[6], ow[7]);
        } else {
#pragma unroll
          for (int e = 0; e < 16; ++e) o[e] = (uint16_t)(ow[e >> 1] >> (16 * (e & 1)));
        }
      }
    }
  }
}

// Stream rows: fp16(fp16(hadamard(cb[idx] (+ QJL term)) * signs) * norm), one
// wave per row of D = 64 E elements (element i = lane + 64 k).
template <int E>
__global__ void k_stream_dequant(const uint8_t* __restrict__ idx, const uint16_t* __restrict__ norm,
                                 const uint8_t* __restrict__ qsign,
                                 const uint16_t* __restrict__ qscale, int64_t rows,
                                 const float* __restrict__ signs, const float* __restrict__ cb,
                                 uint16_t* __restrict__ y) {
  constexpr int D = 64 * E;
  const int l = (int)lane_id();
  int64_t wave = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) >> 6;
  int64_t nw = ((int64_t)gridDim.x * blockDim.x) >> 6;
  for (int64_t r = wave; r < rows; r += nw) {
    float x[E];
#pragma unroll
    for (int k = 0; k < E; ++k) x[k] = cb[idx[r * D + l + 64 * k]];
    if (qsign) {  // QJL: cb[idx] + (2 s - 1) * scale (streaming.py:76-77)
      const float sc = h2f(qscale[r]);
#pragma unroll
      for (int k = 0; k < E; ++k) x[k] = __fadd_rn(x[k], qsign[r * D + l + 64 * k] ? sc : -sc);
    }
    wave_fwht<E>(x, D);
    const float n = h2f(norm[r]);
    // fp16(fp16(x * sign) * norm): the sign flip is exact, the product of two
    // fp16 values is exact in fp32, so each line rounds exactly twice like torch
#pragma unroll
    for (int k = 0; k < E; ++k)
      y[r * D + l + 64 * k] = f2h_opaque(h2f(f2h(mul_sign(x[k], signs[l + 64 * k]))) * n);
  }
}

}  // namespace shard

namespace shard {
namespace {

bool aligned(const void* p, size_t n) { return ((uintptr_t)p & (n - 1)) == 0; }

// Workgroups of one K launch: two per CU would not fit (8 waves of up to 256
// registers), so the units (32-token tiles x batch rows) are dealt to about
// one workgroup per CU, each keeping its basis rows in registers.
template <int HD, int KS>
void launch_rebuild_k(const shard_decode_args* a, const RebuildOut& out, hipStream_t s) {
  constexpr int HPW = 8 / (HD / 64);
  const int gy = (a->n_kv_heads + HPW - 1) / HPW;
  const int64_t units = (int64_t)((a->n_comp + kRcTok - 1) / kRcTok) * a->batch;
  const int want = std::max(1, 256 / gy);
  const int per = (int)((units + want - 1) / want);
  hipLaunchKernelGGL((k_rebuild_k<HD, KS>), dim3((unsigned)((units + per - 1) / per), (unsigned)gy),
                     dim3(512), 0, s, a->k_coeffs, a->k_coeff_scale, a->k_basis, a->k_mean,
                     a->inv_freq, a->batch, a->n_kv_heads, a->n_comp, a->compress_start, per, out);
}

template <int HD>
int launch_k(const shard_decode_args* a, const RebuildOut& out, hipStream_t s) {
  // the MFMA kernel reads 4- and 16-byte vectors of these and stores 16 bytes
  const bool fit = a->rank % 32 == 0 && a->rank <= 256 && aligned(a->k_coeffs, 4) &&
                   aligned(a->k_coeff_scale, 4) && aligned(a->k_basis, 16) &&
                   aligned(a->k_mean, 8) && aligned(out.k, 16) &&
                   (int64_t)((a->n_comp + kRcTok - 1) / kRcTok) * a->batch < INT32_MAX;
  if (fit) {
    switch (a->rank / 32) {
      case 1: launch_rebuild_k<HD, 2>(a, out, s); return SHARD_OK;
      case 2: launch_rebuild_k<HD, 4>(a, out, s); return SHARD_OK;
      case 3: launch_rebuild_k<HD, 6>(a, out, s); return SHARD_OK;
      case 4: launch_rebuild_k<HD, 8>(a, out, s); return SHARD_OK;
      case 5: launch_rebuild_k<HD, 10>(a, out, s); return SHARD_OK;
      case 6: launch_rebuild_k<HD, 12>(a, out, s); return SHARD_OK;
      case 7: launch_rebuild_k<HD, 14>(a, out, s); return SHARD_OK;
      default: launch_rebuild_k<HD, 16>(a, out, s); return SHARD_OK;
    }
  }
  // the tile's fp16 coefficients and the head's basis rows in LDS: up to
  // 160 KB (rank 512 at head_dim 128, 284 at 256)
  const size_t lds = (size_t)(kRcTok + HD) * a->rank * sizeof(uint16_t);
  if (lds > 64 * 1024) {  // LDS beyond the default dynamic limit (160 KB per CU on gfx950)
    const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(&k_reconstruct_k<HD>),
                                             hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (e != hipSuccess) {
      set_last_error("shard_kv_reconstruct LDS attribute", e);
      return SHARD_ERR_HIP;
    }
  }
  dim3 grid((unsigned)((a->n_comp + kRcTok - 1) / kRcTok), (unsigned)a->n_kv_heads,
            (unsigned)a->batch);
  hipLaunchKernelGGL(k_reconstruct_k<HD>, grid, dim3(256), lds, s, a->k_coeffs, a->k_coeff_scale,
                     a->k_basis, a->k_mean, a->inv_freq, a->batch, a->n_kv_heads, a->rank,
                     a->n_comp, a->compress_start, out);
  return SHARD_OK;
}

template <int HD>
void launch_v(const shard_decode_args* a, const RebuildOut& out, const RebuildSegs& sg, int lg,
              int cbn, hipStream_t s) {
  const int64_t bg = (int64_t)a->batch * a->n_kv_heads;
  const int rows_wg = 4 * kRvSteps * (64 / (HD / 16));
  const int rb = (a->n_comp + rows_wg - 1) / rows_wg;
  const int xb = (int)(((int64_t)sg.total * (HD / 8) + 255) / 256);
  const dim3 grid((unsigned)(rb + xb), (unsigned)std::min<int64_t>(bg, 65535));
  const int vec = aligned(a->v_idx, 16 >> lg) && aligned(out.v, 16);
  auto go = [&](auto kern) {
    hipLaunchKernelGGL(kern, grid, dim3(256), 0, s, a->v_idx, a->v_codebook, a->v_ch, bg, a->batch,
                       a->n_kv_heads, a->n_comp, cbn, rb, vec, sg, out);
  };
  switch (lg) {
    case 0: go(k_rebuild_v<HD, 0>); break;
    case 1: go(k_rebuild_v<HD, 1>); break;
    case 2: go(k_rebuild_v<HD, 2>); break;
    default: go(k_rebuild_v<HD, 3>); break;
  }
}

int kv_rebuild(const shard_decode_args* a, uint16_t* k_out, uint16_t* v_out, bool segments,
               hipStream_t s) {
  if (!a || !a->k_coeffs || !a->k_coeff_scale || !a->k_basis || !a->k_mean || !a->v_idx ||
      !a->v_codebook || !a->v_ch || !a->inv_freq || !k_out || !v_out)
    return SHARD_ERR_ARG;
  if (a->batch <= 0 || a->n_comp <= 0 || a->n_kv_heads <= 0) return SHARD_ERR_ARG;
  const int hd = a->head_dim;
  const size_t lds = (size_t)(kRcTok + hd) * (a->rank > 0 ? a->rank : 0) * sizeof(uint16_t);
  if ((hd != 64 && hd != 128 && hd != 256) || a->rank <= 0 || (a->rank & 1) || lds > 160 * 1024)
    return SHARD_ERR_SHAPE;
  const int gs = a->v_group ? a->v_group : 4, cbn = a->v_codebook_n ? a->v_codebook_n : 256;
  const int lg = gs == 1 ? 0 : gs == 2 ? 1 : gs == 4 ? 2 : gs == 8 ? 3 : -1;
  if (lg < 0 || cbn < 1 || cbn > 256) return SHARD_ERR_SHAPE;
  RebuildOut out = {k_out, v_out, a->n_comp, 0};
  RebuildSegs sg = {};
  if (segments) {
    if (a->n_sink < 0 || a->n_win < 0 || a->n_dec < 0 || a->n_stream < 0) return SHARD_ERR_ARG;
    if ((a->n_sink && (!a->sink_k || !a->sink_v)) || (a->n_win && (!a->win_k || !a->win_v)) ||
        (a->n_dec && (!a->dec_k || !a->dec_v || a->dec_stride < a->n_dec)) ||
        (a->n_stream && (!a->s_k || !a->s_v)))
      return SHARD_ERR_ARG;
    const int64_t total = (int64_t)a->n_sink + a->n_win + a->n_dec + a->n_stream;
    if (total + a->n_comp > INT32_MAX / 32) return SHARD_ERR_SHAPE;
    sg = {{a->sink_k, a->win_k, a->s_k, a->dec_k}, {a->sink_v, a->win_v, a->s_v, a->dec_v},
          {a->n_sink, a->n_win, a->n_stream, a->n_dec}, a->dec_stride, (int32_t)total, 1};
    for (int i = 0; i < 4; ++i)
      if (sg.n[i] && (!aligned(sg.k[i], 16) || !aligned(sg.v[i], 16))) sg.vec = 0;
    if (!aligned(k_out, 16) || !aligned(v_out, 16)) sg.vec = 0;
    out.T = total + a->n_comp;
    out.row0 = a->n_sink;
  }
  const int rc = hd == 64 ? launch_k<64>(a, out, s) : hd == 128 ? launch_k<128>(a, out, s)
                                                                : launch_k<256>(a, out, s);
  if (rc != SHARD_OK) return rc;
  if (hd == 64) launch_v<64>(a, out, sg, lg, cbn, s);
  else if (hd == 128) launch_v<128>(a, out, sg, lg, cbn, s);
  else launch_v<256>(a, out, sg, lg, cbn, s);
  SHARD_LAUNCH_CHECK("shard_kv_reconstruct");
  return SHARD_OK;
}

}  // namespace
}  // namespace shard

using namespace shard;

extern "C" {

int shard_kv_reconstruct(const shard_decode_args* a, uint16_t* k_out, uint16_t* v_out,
                         void* stream) {
  return kv_rebuild(a, k_out, v_out, false, (hipStream_t)stream);
}

int shard_kv_rebuild(const shard_decode_args* a, uint16_t* k_out, uint16_t* v_out, void* stream) {
  return kv_rebuild(a, k_out, v_out, true, (hipStream_t)stream);
}

int shard_stream_dequant_qjl(const uint8_t* idx, const uint16_t* norm, const uint8_t* qsign,
                             const uint16_t* qscale, int64_t rows, int32_t hd, const float* signs,
                             const float* codebook, uint16_t* y, void* stream) {
  if (!idx || !norm || !signs || !codebook || !y || rows <= 0) return SHARD_ERR_ARG;
  if ((qsign == nullptr) != (qscale == nullptr)) return SHARD_ERR_ARG;
  hipStream_t s = (hipStream_t)stream;
  const dim3 grid(grid_cap((rows + 3) / 4, 16384)), block(256);
  switch (hd) {
    case 64: hipLaunchKernelGGL(k_stream_dequant<1>, grid, block, 0, s, idx, norm, qsign, qscale, rows, signs, codebook, y); break;
    case 128: hipLaunchKernelGGL(k_stream_dequant<2>, grid, block, 0, s, idx, norm, qsign, qscale, rows, signs, codebook, y); break;
    case 256: hipLaunchKernelGGL(k_stream_dequant<4>, grid, block, 0, s, idx, norm, qsign, qscale, rows, signs, codebook, y); break;
    default: return SHARD_ERR_SHAPE;
  }
  SHARD_LAUNCH_CHECK("shard_stream_dequant");
  return SHARD_OK;
}

int shard_stream_dequant(const uint8_t* idx, const uint16_t* norm, int64_t rows, int32_t hd,
                         const float* signs, const float* codebook, uint16_t* y, void* stream) {
  return shard_stream_dequant_qjl(idx, norm, nullptr, nullptr, rows, hd, signs, codebook, y, stream);
}

}  // extern "C"
