// Fused causal BASED attention, parallel form, bf16, for the head dims the packed d = 16 kernel does
// not take (d <= 64 with d % 8 == 0, dv <= 128 with dv % 8 == 0, 16-byte aligned tensors) and for that
// kernel's own where the grid is small.  Same function, precision and range as based_parallel.hip
// (see there: u = (q.k + 1/c)^2 - 1/c^2 in fp16, V^T in fp16 with exponents, the 1 of p kept exact),
// other data paths:
//
//   wide_pack_kernel  one work-group per 64-key block: V as an fp16 V^T block in the main kernel's
//                     LDS layout with an exponent of its own, and its fp32 column sums;
//   wide_kernel       K rows (from the caller's tensor) and V^T blocks copied global -> LDS with
//                     buffer_load ... lds into a ring; S^T = K Q^T on bf16 MFMAs, u in registers,
//                     O^T += V^T u^T on fp16 MFMAs, row sums of u with v_dot2.
//
// There is no scan between them: a work-group adds the column sums of the blocks before its own
// queries itself (DV floats per block, against 2 (d + dv) 64 bytes of K and V that it reads of each),
// and a wave takes the largest exponent of the blocks it attends to; a block with a smaller one
// takes u with that power of two if it is one step (2^-8), else (rare) multiplies into cleared
// accumulators that are added in fp32 with it.
//
// What bounds it: matrix cores and LDS reads.  A wave owns 64 queries (two 32-wide tiles), so a K
// or V^T fragment read (1 KB, 16 bytes a lane) feeds two MFMAs: d = dv = 64 reads 16 KB per 32 MFMAs
// and wave, 64 of 128 bytes a clock at full MFMA rate; with one tile (32 queries) it would be all of
// them.  256-query work-groups (four waves) where they fill the CUs twice; else 128-query ones, whose
// wave pairs share queries and take one 32-key half of every block each (their accumulators meet
// in LDS at the end), so that the grid is twice as large at the same reads per MFMA.
//
// Chunked calls of the same shapes take these kernels too (chunked_general.hip), with scores and V of
// any size, and no less exact than the segment path that they replace (fp16 prefixes and features;
// inside a 512-token segment p in 16 bits against exact V): ANY.  A work-group takes the blocks before
// its own queries as above where that loses nothing: from row kExactRows on, |u| inside fp16 by
// sum |q| max |k| (the pre-pass then also reads K), V exponents at most a step apart and the values of
// every block held in fp16 to 2^-14 of their column's largest.  All other blocks, its own always, run
// `precise`: p in fp32, as bf16 hi and lo parts against the V rows themselves.  So what a row gets
// depends on no later key or value.  Relative error of fp32 outputs, rows before / from 512, against
// the segment path's: B1 H4 N4096 d64 dv64, q and k of the benchmark 2.6e-6 / 3.2e-6 (2.6e-6 / 1.9e-4),
// four times as large 2.5e-6 / 4.9e-5 (2.5e-6 / 1.9e-4), sixteen times 2.4e-6 / 2.0e-4 (2.4e-6 / 2.7e-4).
// The blocks that run `precise` cost B2 H16 N8192 d64 dv64 3 % (265 -> 273 us); all of them, for
// scores out of range, 432 us (the segment path 423).
//
// Measured (pre-pass + kernel, us; the register-staged kernel and its max pass before): B2 H16 d64 dv64
// N2048 7 + 29 (5 + 62), N8192 14 + 252 (8 + 445): 1.04 PFLOP/s, matrix cores busy 57 % of the
// cycles at the 1.9 GHz that the card holds under this load.  At N2048 20 of the 29 us are the loop
// of the longest work-groups (16 steps), the rest launch, queries, column sums and the epilogue.
#include <type_traits>

#include "../../include/based_la.h"
#include "la_common.hpp"
#include "la_internal.hpp"
#include "la_pack.hpp"

namespace la {
namespace {

struct WideParams {
  const uint16_t* q;
  const uint16_t* k;
  const uint16_t* v;
  uint16_t* vt;          // [BH][nb][32 MT rows][64] fp16
  float* sums;           // [BH][nb][32 MT] column sums of V
  int* eb;               // [BH][nb] V exponents
  u32* kmx;              // ANY: [BH][nb]: largest finite |k| (bf16 bits), kCoarse where fp16 V^T will not do
  void* out;
  float* den;
  int BH, H, N, d, dv, nqb, nb;
  // element strides {batch, head, token} of q and k, of v and of the output
  long long ks[3], vs[3], os[3];
  float inv_c, inv_c2, fscale, eps, qscale;
  u32 ones_hi, ones_lo;
  int normalize, out_f32, xcd_cus;
};

// V^T rows: 64 keys = eight 16-byte units; unit 2 m + h of a row holds keys 16 m + 4 h + {0..3, 8..11}
// (the order of a score accumulator's registers, so a unit is a whole A operand of the P.V MFMA),
// stored at unit ^ swz64(row).  K rows of 2 KS 16-byte chunks: chunk c at c ^ kwz(key).  Both make
// the 16 lanes of a ds_read_b128 pass touch all 64 banks once.
template <int KS>
__device__ __forceinline__ int kwz(int key) {
  return KS == 1 ? ((key >> 2) ^ (key >> 3)) & 1 : KS == 2 ? (key >> 2) & 3 : swz64(key);
}

constexpr u32 kCoarse = 0x80000000u;
constexpr int kExactRows = 512;   // the first segment of the path that chunked calls took before

__device__ __forceinline__ size_t head_offset(const WideParams& p, const long long (&s)[3], int bh) {
  if (p.H == p.BH) return (size_t)bh * s[1];   // one batch: no division
  const int b = bh / p.H;
  return (size_t)(b * s[0] + (bh - b * p.H) * s[1]);
}

// ---------------------------------------------------------------- V^T blocks
// Thread -> keys 2 kp, 2 kp + 1 and eight columns; column sums through LDS.  Any dv: rows past dv
// and keys past N are zero.
template <int MT, bool ANY>
__global__ __launch_bounds__(256) void wide_pack_kernel(const WideParams p) {
  constexpr int DV = 32 * MT, CPR = DV / 8, IT = (32 * CPR + 255) / 256;
  __shared__ __attribute__((aligned(16))) uint16_t img[DV * BN];
  __shared__ float csum[32][DV + 1];
  __shared__ u32 vmx[4], kmxl[4];
  __shared__ u32 lost[ANY ? DV : 1];   // a value of this column is not exact in fp16
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const int bh = blockIdx.x / p.nb, blk = blockIdx.x - bh * p.nb, dv = p.dv;
  const int vrow = (int)p.vs[2];   // elements per token
  const __amdgpu_buffer_rsrc_t rv =
      make_rsrc(p.v + head_offset(p, p.vs, bh), ((u32)(p.N - 1) * (u32)vrow + (u32)dv) * 2u);
  u32x4 a[IT], b[IT];
  u32 m = 0u;
#pragma unroll
  for (int x = 0; x < IT; ++x) {
    const int t = tid + 256 * x, kp = t / CPR, col = 8 * (t % CPR);
    const int off = kp < 32 && col < dv ? ((blk * BN + 2 * kp) * vrow + col) * 2 : kOffOutOfRange;
    a[x] = buf_load_b128(rv, off);
    b[x] = buf_load_b128(rv, off == kOffOutOfRange ? off : off + 2 * vrow);
  }
#pragma unroll
  for (int x = 0; x < IT; ++x)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const u32 y = a[x][i] & 0x7fff7fffu, z = b[x][i] & 0x7fff7fffu;
      m = max(m, max(max(y & 0xffffu, y >> 16), max(z & 0xffffu, z >> 16)));
    }
  m = wave_max_u32(m);
  if (lane == 0) vmx[w] = m;
  if (ANY && tid < DV) lost[tid] = 0u;
  if constexpr (ANY) {   // contiguous k rows, d % 8 == 0
    const __amdgpu_buffer_rsrc_t rk = make_rsrc(p.k + (size_t)bh * p.N * p.d, (u32)p.N * (u32)p.d * 2u);
    u32 mk = 0u;
    for (int x = tid; x < BN * p.d / 8; x += 256) {
      const u32x4 y = buf_load_b128(rk, (blk * BN * p.d + 8 * x) * 2);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const u32 lo = y[i] & 0x7fffu, hi = (y[i] >> 16) & 0x7fffu;
        mk = max(mk, max(lo < 0x7f80u ? lo : 0u, hi < 0x7f80u ? hi : 0u));
      }
    }
    mk = wave_max_u32(mk);
    if (lane == 0) kmxl[w] = mk;
  }
  __syncthreads();
  const int eb = vexp_step(max(max(vmx[0], vmx[1]), max(vmx[2], vmx[3])) << 16);
#pragma unroll
  for (int x = 0; x < IT; ++x) {
    const int t = tid + 256 * x, kp = t / CPR, col = 8 * (t % CPR);
    if (kp >= 32) continue;
    // keys 2 kp, 2 kp + 1 = 16 m + 8 (e / 4) + 4 h + e % 4
    const int r = (2 * kp) & 15, unit = 2 * (kp >> 3) + ((r >> 2) & 1), e = ((r >> 3) << 2) | (r & 3);
#pragma unroll
    for (int c = 0; c < 8; ++c) {
      const float f0 = (c & 1) ? bf16_hi_to_f32(a[x][c >> 1]) : bf16_lo_to_f32(a[x][c >> 1]);
      const float f1 = (c & 1) ? bf16_hi_to_f32(b[x][c >> 1]) : bf16_lo_to_f32(b[x][c >> 1]);
      const int row = col + c;
      csum[kp][row] = f0 + f1;
      const float g0 = __builtin_ldexpf(f0, -eb), g1 = __builtin_ldexpf(f1, -eb);
      const u32 y = pack_f16x2(g0, g1);
      if (ANY && (f16_lo_to_f32(y) != g0 || f16_hi_to_f32(y) != g1)) lost[row] = 1u;
      *reinterpret_cast<u32*>(&img[row * BN + ((unit ^ swz64(row)) << 3) + e]) = y;
    }
  }
  __syncthreads();
  const size_t rec = (size_t)bh * p.nb + blk;
  u32x4* dst = reinterpret_cast<u32x4*>(p.vt + rec * (DV * BN));
  int coarse = eb == 128;   // infinities and NaN
  for (int i = tid; i < DV * BN / 8; i += 256) {
    const u32x4 x = reinterpret_cast<const u32x4*>(img)[i];
    dst[i] = x;
    if constexpr (ANY) {
      // eight lanes hold a column: what fp16 drops of it, at most 2^-25, stays below 2^-14 of its largest value
      u32 mc = 0u;
#pragma unroll
      for (int e = 0; e < 4; ++e) mc = max(mc, max(x[e] & 0x7fffu, (x[e] >> 16) & 0x7fffu));
#pragma unroll
      for (int y = 1; y < 8; y <<= 1) mc = max(mc, (u32)__shfl_xor((int)mc, y));
      coarse |= lost[i >> 3] != 0u && mc < 0x1000u;   // fp16 2^-11
    }
  }
  if constexpr (ANY) {
    coarse = __syncthreads_or(coarse);
    if (tid == 0) p.kmx[rec] = max(max(kmxl[0], kmxl[1]), max(kmxl[2], kmxl[3])) | (coarse ? kCoarse : 0u);
  }
  if (tid < DV) {
    float s = 0.f;
#pragma unroll
    for (int i = 0; i < 32; ++i) s += csum[i][tid];
    p.sums[rec * DV + tid] = s;
  }
  if (tid == 0) p.eb[rec] = eb;
}

// ---------------------------------------------------------------- attention
// KS: 16-wide steps of d; MT: 32-wide tiles of dv; QT: 32-query tiles per wave; NKH: waves sharing a
// query group (2: each takes one 32-key half of every block).  UNIT: 1/c scales to exactly 1/2.  ROWS:
// calls of the packed kernel's shapes that return denominators, which that kernel takes from fp32
// statistics: row sums of u in fp32 beside those of its fp16 form, which divide the output as in calls
// without (B2 H4 N2048 d16 dv64, q and k four times the benchmark's, denominators of rows 64 to 512:
// 1.0e-5 off from the fp16 sums, 3.6e-8 so, packed 3.3e-6).
template <int KS, int MT, int QT, int NKH, bool UNIT, bool ANY, bool ROWS>
__global__ __launch_bounds__(256, KS == 1 && MT == 1 && !ROWS ? 3 : 2) void wide_kernel(const WideParams p) {
  constexpr int DV = 32 * MT, NQW = 4 / NKH, BM = 32 * QT * NQW;
  constexpr int UB = NKH;                           // blocks per step (two 32-key units per wave either way)
  constexpr int UK = 2 * KS, UV = 4 * MT;           // 1 KB copy units of a block
  constexpr int CW = (UK + UV + 3) / 4;             // copies per wave and block
  constexpr int BLK = 4 * CW * 512;                 // halves per block in LDS
  constexpr int NSR = NKH == 2 ? 2 : CW <= 4 ? 4 : 3;   // steps in the ring
  __shared__ __attribute__((aligned(16))) uint16_t ring[NSR * UB][BLK];
  __shared__ float vsl[NQW][DV];
  __shared__ u32 wst[ANY ? 4 : 1][5];

  const int tid = threadIdx.x, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6), h = lane >> 5, n = lane & 31;
  const int qg = NKH == 2 ? wv >> 1 : wv, kh = NKH == 2 ? wv & 1 : 0;
  const int N = p.N, d = p.d, dv = p.dv;
  int bh, qb;
  map_causal_block(blockIdx.x, p.BH, p.nqb, bh, qb, p.xcd_cus);
  const int q0 = qb * BM, jb0 = q0 / BN;
  const int nblk = min(p.nb, (q0 + BM + BN - 1) / BN), nstep = (nblk + UB - 1) / UB;
  const int wq0 = q0 + 32 * QT * qg, jd = wq0 / BN;
  const bool live = wq0 < N;
  const size_t hrow = (size_t)bh * N;

  // ---- ring copies: unit u < UK of a block are K rows, then V^T rows (then padding, never read)
  const int krow = (int)p.ks[2] * 2, vrow = (int)p.vs[2] * 2;   // bytes per token
  const size_t kbase = head_offset(p, p.ks, bh);
  const u32x4 rk = buffer_rsrc(p.k + kbase, (u32)(N - 1) * (u32)krow + (u32)d * 2u);
  const u32x4 rv = buffer_rsrc(p.vt + (size_t)bh * p.nb * (DV * BN), (u32)p.nb * (u32)(DV * BN * 2));
  // ANY: blocks from jraw on come as rows of V (of DV columns in LDS) in place of the V^T block; at
  // first on the assumption that the others may be taken as such
  static_assert(kExactRows % 256 == 0, "whole work-groups");
  int jraw = q0 >= kExactRows ? jb0 : 0;
  const u32x4 rw = buffer_rsrc(p.v + head_offset(p, p.vs, bh), (u32)(N - 1) * (u32)vrow + (u32)dv * 2u);
  int uoff[CW], woff[CW];
#pragma unroll
  for (int x = 0; x < CW; ++x) {
    const int u = 4 * x + wv;
    if (u < UK) {
      const int sl = 64 * u + lane, key = sl / (2 * KS), c = (sl % (2 * KS)) ^ kwz<KS>(key);
      uoff[x] = 8 * c < d ? key * krow + 16 * c : kOffOutOfRange;
    } else {
      uoff[x] = u < UK + UV ? 1024 * (u - UK) + 16 * lane : kOffOutOfRange;
    }
    const int sl = 64 * (u - UK) + lane, key = sl / (4 * MT), c = sl % (4 * MT);
    woff[x] = u >= UK && u < UK + UV && 8 * c < dv ? key * vrow + 16 * c : kOffOutOfRange;
  }
  auto issue = [&](int s) {   // steps and blocks past the last read nothing: the counts stay equal
#pragma unroll
    for (int t = 0; t < UB; ++t) {
      const int j = UB * s + t;
      const u32 lds = lds_addr(&ring[(s % NSR) * UB + t][0]);
      // one branch per block: a choice of resource per copy made one each, and 5 % of the chunked loop
      auto copies = [&](const u32x4& r, const int (&off)[CW], int step) {
#pragma unroll
        for (int x = 0; x < CW; ++x) {
          const int u = 4 * x + wv;
          const bool isk = u < UK;
          const int o = isk ? uoff[x] : off[x];
          lds_copy16(isk ? rk : r, lds + 1024 * u,
                     j < nblk && o != kOffOutOfRange ? o + j * (isk ? BN * krow : step) : kOffOutOfRange);
        }
      };
      if (ANY && j >= jraw)
        copies(rw, woff, BN * vrow);
      else
        copies(rv, uoff, DV * BN * 2);
    }
  };
#pragma unroll
  for (int s = 0; s < NSR - 1; ++s) issue(s);

  // ---- queries (B operand of S^T = K Q^T): q[query][16 kk + 8 h .. + 7], scaled by a power of two
  u32x4 qf[QT][KS];
#pragma unroll
  for (int qt = 0; qt < QT; ++qt) {
    const int query = wq0 + 32 * qt + n;
#pragma unroll
    for (int kk = 0; kk < KS; ++kk) {
      const int col = 16 * kk + 8 * h;
      u32x4 x = {0u, 0u, 0u, 0u};
      if (query < N && col < d) x = *reinterpret_cast<const u32x4*>(p.q + kbase + (size_t)query * p.ks[2] + col);
      qf[qt][kk] = scale_bf16x8(x, p.qscale);
    }
  }
  // ---- exponents of the blocks that this wave attends to (ANY: of those before the work-group's
  // queries); all-zero blocks (-128) go with any
  const int* __restrict__ ebs = p.eb + (size_t)bh * p.nb;
  int emax = -128, emin = 1 << 20;
  // near: two exponents a step of 8 apart, whose lower blocks take u by 2^-8 (V near the edge of a step has
  // both in most heads); mixed: more.  ANY: fast: blocks before jb0 as u and V^T
  bool near = false, mixed = false, fast = true;
  if constexpr (ANY) {
    fast = jraw > 0;
    if (fast) {
      u32 km = 0u, bad = 0u;
      for (int j = tid; j < jb0; j += 256) {
        const int e = ebs[j];
        const u32 m = p.kmx[(size_t)bh * p.nb + j];
        emax = max(emax, e);
        emin = min(emin, e == -128 ? emin : e);
        km = max(km, m & ~kCoarse);
        bad |= m & kCoarse;
      }
      float l1 = 0.f;   // the largest sum of |q| of the wave's queries (NaN: above every number)
#pragma unroll
      for (int qt = 0; qt < QT; ++qt) {
        float y = 0.f;
#pragma unroll
        for (int kk = 0; kk < KS; ++kk)
#pragma unroll
          for (int e = 0; e < 4; ++e)
            y += __builtin_fabsf(bf16_lo_to_f32(qf[qt][kk][e])) + __builtin_fabsf(bf16_hi_to_f32(qf[qt][kk][e]));
        y += __shfl_xor(y, 32);
        l1 = __builtin_bit_cast(float, max(__builtin_bit_cast(u32, l1), __builtin_bit_cast(u32, y)));
      }
      const u32 st[5] = {wave_max_u32((u32)(emax + 1024)), wave_max_u32((u32)((1 << 21) - emin)), wave_max_u32(km),
                         wave_max_u32(__builtin_bit_cast(u32, l1)), wave_max_u32(bad)};
      if (lane == 0)
#pragma unroll
        for (int i = 0; i < 5; ++i) wst[wv][i] = st[i];
      __syncthreads();
      u32 all[5];
#pragma unroll
      for (int i = 0; i < 5; ++i)
        all[i] = (u32)__builtin_amdgcn_readfirstlane((int)max(max(wst[0][i], wst[1][i]), max(wst[2][i], wst[3][i])));
      emax = (int)all[0] - 1024;
      emin = (1 << 21) - (int)all[1];
      // u in fp16: |b| = |q~ k + 1/c| <= 240 keeps b^2 - 1/c^2 below 57600
      const float bound = __builtin_bit_cast(float, all[3]) * __builtin_bit_cast(float, all[2] << 16) + p.inv_c;
      fast = __builtin_amdgcn_readfirstlane(emin >= emax - 8 && all[4] == 0u && bound <= 240.f);
      near = emin < emax;
      if (!fast) {   // the copies under way are of the wrong kind
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
        jraw = 0;
#pragma unroll
        for (int s = 0; s < NSR - 1; ++s) issue(s);
      }
    }
  } else {
    if (live)
      for (int j = lane; j <= jd; j += 64) {
        const int e = ebs[j];
        emax = max(emax, e);
        emin = min(emin, e == -128 ? emin : e);
      }
    emax = (int)wave_max_u32((u32)(emax + 1024)) - 1024;
    emin = (1 << 21) - (int)wave_max_u32((u32)((1 << 21) - emin));
    near = emin < emax;
    mixed = live && emin < emax - 8;
  }
  // ---- column sums of V over the blocks before each query group's diagonal block (`precise` counts the 1 of
  // p itself)
  if (fast) {
    constexpr int PARTS = 256 / DV, PF = 8;
    float* psum = reinterpret_cast<float*>(&ring[(NSR - 1) * UB][0]);   // the last step's place, still free
    const float* __restrict__ sm = p.sums + (size_t)bh * p.nb * DV + tid % DV;
    float s = 0.f;
    for (int j = tid / DV; j < jb0; j += PARTS * PF) {
      float y[PF];
#pragma unroll
      for (int t = 0; t < PF; ++t) y[t] = j + PARTS * t < jb0 ? sm[(size_t)(j + PARTS * t) * DV] : 0.f;
#pragma unroll
      for (int t = 0; t < PF; ++t) s += y[t];
    }
    psum[tid] = s;
    __syncthreads();
    if (kh == 0)
      for (int c = lane; c < DV; c += 64) {
        float t = 0.f;
#pragma unroll
        for (int x = 0; x < PARTS; ++x) t += psum[x * DV + c];
        if (!ANY)
          for (int j = jb0; j < min(jd, p.nb); ++j) t += p.sums[((size_t)bh * p.nb + j) * DV + c];
        vsl[qg][c] = t;
      }
    __syncthreads();   // psum read before the ring takes its place
  } else {
    for (int c = tid; c < NQW * DV; c += 256) vsl[c / DV][c % DV] = 0.f;   // read after the loops' barriers
  }

  f32x16 acc[QT][MT];
  float rsum[QT], rsx[QT];
#pragma unroll
  for (int qt = 0; qt < QT; ++qt) {
    rsum[qt] = rsx[qt] = 0.f;
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) acc[qt][mt] = splat16(0.f);
  }
  const float inv_c = UNIT ? 0.5f : p.inv_c, inv_c2 = UNIT ? 0.25f : p.inv_c2;
  constexpr u32 kOnes = 0x3c003c00u, kOnesBf = 0x3f803f80u;   // packed (1, 1) in fp16, bf16

  auto kfrag = [&](const uint16_t* st, int ks, int kk) {
    const int key = 32 * ks + n;
    return *reinterpret_cast<const u32x4*>(st + key * (16 * KS) + (((2 * kk + h) ^ kwz<KS>(key)) << 3));
  };
  auto vfrag = [&](const uint16_t* st, int ks, int m, int mt) {
    const int row = 32 * mt + n;
    return *reinterpret_cast<const u32x4*>(st + UK * 512 + row * BN + (((4 * ks + 2 * m + h) ^ swz64(row)) << 3));
  };
  // pieces of a full 32-key unit: scores b = K Q^T + 1/c; u = b b - 1/c^2 in fp16 and its row sums;
  // acc += V^T u^T
  auto S = [&](const uint16_t* st, int ks, f32x16 (&b)[QT]) {
    u32x4 kf[KS];
#pragma unroll
    for (int kk = 0; kk < KS; ++kk) kf[kk] = kfrag(st, ks, kk);
#pragma unroll
    for (int qt = 0; qt < QT; ++qt) {
      b[qt] = splat16(inv_c);
#pragma unroll
      for (int kk = 0; kk < KS; ++kk) b[qt] = mfma32x32x16(kf[kk], qf[qt][kk], b[qt]);
    }
  };
  // NEAR: low blocks (an exponent 8 below the wave's) take u 2^-8, whose rounding at 2^-25 is 2^-16 of the 1 of p
  auto E = [&](auto near_tag, bool low, const f32x16 (&b)[QT], u32x4 (&pf)[QT][2]) {
    constexpr bool NEAR = decltype(near_tag)::value;
    const float f = low ? 0.0625f : 1.0f, cc = low ? -0.00390625f * inv_c2 : -inv_c2;
    const u32 ones = low ? 0x5c005c00u : kOnes;   // fp16 2^8
#pragma unroll
    for (int qt = 0; qt < QT; ++qt)
#pragma unroll
      for (int m = 0; m < 2; ++m)
#pragma unroll
        for (int c = 0; c < 4; ++c) {
          const float b0 = b[qt][8 * m + 2 * c], b1 = b[qt][8 * m + 2 * c + 1];
          pf[qt][m][c] = NEAR ? sq_plus_f16x2(b0 * f, b1 * f, cc) : sq_plus_f16x2(b0, b1, -inv_c2);
          rsum[qt] = dot2_f16(pf[qt][m][c], NEAR ? ones : kOnes, rsum[qt]);
          if (ROWS) rsx[qt] += __builtin_fmaf(b0, b0, -inv_c2) + __builtin_fmaf(b1, b1, -inv_c2);
        }
  };
  auto P = [&](const uint16_t* st, int ks, const u32x4 (&pf)[QT][2]) {
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
      for (int m = 0; m < 2; ++m) {
        const u32x4 vf = vfrag(st, ks, m, mt);
#pragma unroll
        for (int qt = 0; qt < QT; ++qt) acc[qt][mt] = mfma32x32x16_f16(vf, pf[qt][m], acc[qt][mt]);
      }
  };
  // acc += 2^e V^T x^T for operands x[nx][QT][2], through cleared accumulators
  auto Pscaled = [&](const uint16_t* st, int ks, const u32x4 (*x)[QT][2], int nx, const bool (&act)[QT], int e) {
    const float f = __builtin_ldexpf(1.0f, e);
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
      const u32x4 v0 = vfrag(st, ks, 0, mt), v1 = vfrag(st, ks, 1, mt);
#pragma unroll
      for (int qt = 0; qt < QT; ++qt) {
        if (!act[qt]) continue;
        f32x16 t = splat16(0.f);
#pragma unroll
        for (int y = 0; y < 3; ++y) {
          if (y >= nx) continue;
          t = mfma32x32x16_f16(v0, x[y][qt][0], t);
          t = mfma32x32x16_f16(v1, x[y][qt][1], t);
        }
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[qt][mt][r] = __builtin_fmaf(f, t[r], acc[qt][mt][r]);
      }
    }
  };
  // a unit of the wave's diagonal block, or a full unit of a block with a smaller V exponent
  auto general = [&](const uint16_t* st, int j, int ks) {
    const int kb = BN * j + 32 * ks, e = near ? max(ebs[j] - emax, -126) : 0;
    u32x4 x[3][QT][2];   // u, then the mask times W's hi and lo parts (the exact 1 of p)
    bool act[QT];
    u32x4 kf[KS];
#pragma unroll
    for (int kk = 0; kk < KS; ++kk) kf[kk] = kfrag(st, ks, kk);
    const bool diag = j == jd;
#pragma unroll
    for (int qt = 0; qt < QT; ++qt) {
      const int qbase = wq0 + 32 * qt, query = qbase + n;
      act[qt] = kb <= qbase + 31 && qbase < N;
      const u32 whi = p.ones_hi, wlo = p.ones_lo;
      f32x16 b = splat16(inv_c);
#pragma unroll
      for (int kk = 0; kk < KS; ++kk) b = mfma32x32x16(kf[kk], qf[qt][kk], b);
#pragma unroll
      for (int m = 0; m < 2; ++m)
#pragma unroll
        for (int c = 0; c < 4; ++c) {
          const int i = 8 * m + 2 * c, k0 = kb + c32_row(i, h);   // keys k0, k0 + 1
          const float u0 = __builtin_fmaf(b[i], b[i], -inv_c2), u1 = __builtin_fmaf(b[i + 1], b[i + 1], -inv_c2);
          const bool in0 = k0 <= query, in1 = k0 + 1 <= query;
          x[0][qt][m][c] = pack_f16x2(in0 ? u0 : 0.f, in1 ? u1 : 0.f);
          x[1][qt][m][c] = (in0 ? whi & 0xffffu : 0u) | (in1 ? whi & 0xffff0000u : 0u);
          x[2][qt][m][c] = (in0 ? wlo & 0xffffu : 0u) | (in1 ? wlo & 0xffff0000u : 0u);
          if (!act[qt]) continue;
          rsum[qt] = dot2_f16(x[0][qt][m][c], kOnes, rsum[qt]);
          if (ROWS) rsx[qt] += (in0 ? u0 : 0.f) + (in1 ? u1 : 0.f);
        }
    }
    Pscaled(st, ks, x, !diag ? 1 : p.ones_lo != 0u ? 3 : 2, act, e);
  };
  // ANY: W p = b^2 + 1/c^2 in fp32, carried as bf16 hi + lo (16 bits) against the rows of V (exact) that
  // the stage holds; the row sums take the same two parts, so that a row's rounding cancels in the quotient
  auto weights = [&](const f32x16& b, int kb, int query, bool masked, float& sum, u32x4 (&hi)[2], u32x4 (&lo)[2]) {
#pragma unroll
    for (int m = 0; m < 2; ++m)
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        const int i = 8 * m + 2 * c, k0 = kb + c32_row(i, h);   // keys k0, k0 + 1
        float w0 = __builtin_fmaf(b[i], b[i], inv_c2), w1 = __builtin_fmaf(b[i + 1], b[i + 1], inv_c2);
        if (masked) {
          w0 = k0 <= query ? w0 : 0.f;
          w1 = k0 + 1 <= query ? w1 : 0.f;
        }
        hi[m][c] = pack_bf16x2(w0, w1);
        lo[m][c] = pack_bf16x2(w0 - bf16_lo_to_f32(hi[m][c]), w1 - bf16_hi_to_f32(hi[m][c]));
        sum = dot2_bf16(lo[m][c], kOnesBf, dot2_bf16(hi[m][c], kOnesBf, sum));
      }
  };
  // A operand of P.V from the rows of V: column 32 mt + n, keys 16 m + 4 h + {0..3, 8..11}
  auto vrows = [&](const uint16_t* st, int ks, int m, int mt) {
    const uint16_t* x = st + UK * 512 + (32 * ks + 4 * h + 16 * m) * DV + n + 32 * mt;
    return (u32x4){(u32)x[0] | ((u32)x[DV] << 16), (u32)x[2 * DV] | ((u32)x[3 * DV] << 16),
                   (u32)x[8 * DV] | ((u32)x[9 * DV] << 16), (u32)x[10 * DV] | ((u32)x[11 * DV] << 16)};
  };
  auto precise = [&](const uint16_t* st, int kb, int ks, auto masked_tag) {
    constexpr bool MASKED = decltype(masked_tag)::value;
    u32x4 kf[KS], vf[MT][2];
#pragma unroll
    for (int kk = 0; kk < KS; ++kk) kf[kk] = kfrag(st, ks, kk);
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
      for (int m = 0; m < 2; ++m) vf[mt][m] = vrows(st, ks, m, mt);
#pragma unroll
    for (int qt = 0; qt < QT; ++qt) {
      const int qbase = wq0 + 32 * qt;
      if (MASKED && kb > qbase + 31) continue;   // no weight for any query (an infinite V there would count)
      f32x16 b = splat16(inv_c);
#pragma unroll
      for (int kk = 0; kk < KS; ++kk) b = mfma32x32x16(kf[kk], qf[qt][kk], b);
      u32x4 hi[2], lo[2];
      weights(b, kb, qbase + n, MASKED && kb + 31 > qbase, rsum[qt], hi, lo);
#pragma unroll
      for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int m = 0; m < 2; ++m) {
          acc[qt][mt] = mfma32x32x16(vf[mt][m], hi[m], acc[qt][mt]);
          acc[qt][mt] = mfma32x32x16(vf[mt][m], lo[m], acc[qt][mt]);
        }
    }
  };

  // step s of this wave landed (NSR - 2 later ones may be in flight), then every wave's; every wave is
  // past step s - 1, whose place the next copies take
  auto begin = [&](int s) {
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"i"((NSR - 2) * UB * CW) : "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    issue(s + NSR - 1);
  };
  // The step's two units: the halves of block s (NKH = 1), or this wave's half of blocks 2 s, 2 s + 1.
  // Steps before the wave's diagonal block in a loop of their own: as one branch of a common loop the
  // accumulators were copied at its end (32 v_mov_b64 per step).  The waves leave it at different steps
  // and meet at the same count of barriers.
  const int nfull = ANY ? jraw / UB : !live || mixed ? 0 : min(jd / UB, nstep);
  unsigned long long low = 0ull;
  auto full = [&](auto near_tag, int s) {
    constexpr bool NEAR = decltype(near_tag)::value;
    begin(s);
    // the low blocks of 64 at a time: a load per block would wait for the copies in flight
    if (NEAR && (UB * s & 63) == 0) low = __ballot(ebs[min(UB * s + lane, p.nb - 1)] < emax);
    const bool l0 = NEAR && (low >> (UB * s & 63) & 1), l1 = NEAR && (low >> ((UB * s & 63) + UB - 1) & 1);
    const uint16_t* s0 = &ring[(s % NSR) * UB][0];
    const uint16_t* s1 = NKH == 2 ? &ring[(s % NSR) * UB + 1][0] : s0;
    const int k0 = NKH == 2 ? kh : 0, k1 = NKH == 2 ? kh : 1;
    f32x16 b0[QT], b1[QT];
    u32x4 p0[QT][2], p1[QT][2];
    S(s0, k0, b0);
    S(s1, k1, b1);
    E(near_tag, l0, b0, p0);
    P(s0, k0, p0);
    E(near_tag, l1, b1, p1);
    P(s1, k1, p1);
  };
  if (near)
    for (int s = 0; s < nfull; ++s) full(std::true_type{}, s);
  else
    for (int s = 0; s < nfull; ++s) full(std::false_type{}, s);
  if (ANY && jraw > 0) {   // acc in units of 1 from here on
#pragma unroll
    for (int qt = 0; qt < QT; ++qt)
#pragma unroll
      for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[qt][mt][r] = __builtin_ldexpf(acc[qt][mt][r], emax);
  }
  const int npre = ANY && live ? max(nfull, min(jd / UB, nstep)) : nfull;
  if constexpr (ANY) {
#pragma unroll 1
    for (int s = nfull; s < npre; ++s) {
      begin(s);
#pragma unroll
      for (int t = 0; t < 2; ++t)
        precise(&ring[(s % NSR) * UB + (NKH == 2 ? t : 0)][0], 0, NKH == 2 ? kh : t, std::false_type{});
    }
  }
#pragma unroll 1
  for (int s = npre; s < nstep; ++s) {
    begin(s);
#pragma unroll 1
    for (int t = 0; t < 2; ++t) {
      const int j = UB * s + (NKH == 2 ? t : 0), ks = NKH == 2 ? kh : t;
      const uint16_t* st = &ring[(s % NSR) * UB + (NKH == 2 ? t : 0)][0];
      if (live && j <= jd && BN * j + 32 * ks <= wq0 + 32 * QT - 1) {
        if constexpr (ANY)
          precise(st, BN * j + 32 * ks, ks, std::true_type{});
        else
          general(st, j, ks);
      }
    }
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // no copy in flight into the ring
  __syncthreads();

  // ---- the halves' sums: the wave pair splits its two query tiles, each adds the other's part
  constexpr int QE = QT / NKH;   // query tiles a wave finishes, from tile e0
  static_assert(NKH == 1 || QT == 2, "a wave pair finishes one tile each");
  const int e0 = NKH == 2 ? kh : 0;
  f32x16 fin[QE][MT];
  float rs[QE], rx[QE];
  if constexpr (NKH == 2) {
    constexpr int PW = (16 * MT + 2) * 64;   // floats of a wave's part
    static_assert(4 * PW * 4 <= (int)sizeof(ring), "parts fit in the ring");
    float* mine = reinterpret_cast<float*>(&ring[0][0]) + wv * PW + lane;
    float* other = reinterpret_cast<float*>(&ring[0][0]) + (wv ^ 1) * PW + lane;
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
      for (int r = 0; r < 16; ++r) mine[(16 * mt + r) * 64] = kh ? acc[0][mt][r] : acc[1][mt][r];
    mine[16 * MT * 64] = kh ? rsum[0] : rsum[1];
    if (ROWS) mine[16 * MT * 64 + 64] = kh ? rsx[0] : rsx[1];
    __syncthreads();
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
      for (int r = 0; r < 16; ++r) fin[0][mt][r] = (kh ? acc[1][mt][r] : acc[0][mt][r]) + other[(16 * mt + r) * 64];
    rs[0] = (kh ? rsum[1] : rsum[0]) + other[16 * MT * 64];
    rx[0] = ROWS ? (kh ? rsx[1] : rsx[0]) + other[16 * MT * 64 + 64] : 0.f;
    __syncthreads();   // read before the output tiles take their place
  } else {
#pragma unroll
    for (int qt = 0; qt < QT; ++qt) {
      rs[qt] = rsum[qt];
      rx[qt] = rsx[qt];
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) fin[qt][mt] = acc[qt][mt];
    }
  }
  if (!live) return;

  // ---- out = (acc 2^E / W + column sums) / (t + 1 + row sum / W + eps), 32 rows x 64 columns at a
  // time through this wave's own LDS, so that stores write whole lines (ANY: E = 0, and jraw 64 in place
  // of t + 1)
  const float fscale = p.fscale, afs = ANY ? fscale : fscale * __builtin_ldexpf(1.0f, emax);
  auto store = [&](auto f32_tag) {
    constexpr bool F32 = decltype(f32_tag)::value;
    constexpr int CT = MT == 1 ? 1 : 2, EB = F32 ? 4 : 2, RB = 32 * CT * EB, RS = RB + 16, CPR = RB / 16;
    static_assert(4 * 32 * RS <= (int)sizeof(ring), "output tiles fit in the ring");
    char* tile = reinterpret_cast<char*>(&ring[0][0]) + wv * (32 * RS);
    char* obase = static_cast<char*>(p.out) + head_offset(p, p.os, bh) * EB;
    const u32 orow = (u32)p.os[2] * EB;   // bytes per token
#pragma unroll
    for (int qe = 0; qe < QE; ++qe) {
      const int qbase = wq0 + 32 * (e0 + qe), query = qbase + n;
      const float r2 = rs[qe] + __shfl_xor(rs[qe], 32);
      const float den = (float)(ANY ? BN * jraw : query + 1) + fscale * r2;
      const float inv = p.normalize ? 1.0f / (den + p.eps) : 1.0f;
      const float x2 = ROWS ? rx[qe] + __shfl_xor(rx[qe], 32) : 0.f;
      if (p.den != nullptr && h == 0 && query < N) p.den[hrow + query] = ROWS ? (float)(query + 1) + fscale * x2 : den;
#pragma unroll
      for (int ct = 0; ct < MT; ct += CT) {
#pragma unroll
        for (int mt = 0; mt < CT; ++mt)
#pragma unroll
          for (int g = 0; g < 4; ++g) {
            float y[4];
#pragma unroll
            for (int e = 0; e < 4; ++e)
              y[e] = (afs * fin[qe][ct + mt][4 * g + e] + vsl[qg][32 * (ct + mt) + 8 * g + 4 * h + e]) * inv;
            char* dst = tile + n * RS + (32 * mt + 8 * g + 4 * h) * EB;
            if (F32)
              *reinterpret_cast<f32x4*>(dst) = (f32x4){y[0], y[1], y[2], y[3]};
            else
              *reinterpret_cast<u32x2*>(dst) = (u32x2){pack_bf16x2(y[0], y[1]), pack_bf16x2(y[2], y[3])};
          }
        char* out = obase + ((size_t)qbase * p.os[2] + 32 * ct) * EB;
        const int cols = (dv - 32 * ct) * EB;   // bytes of a row from this column on
#pragma unroll
        for (int it = 0; it < CPR / 2; ++it) {
          const int idx = 64 * it + lane, r = idx / CPR, c = idx % CPR;
          const u32x4 y = *reinterpret_cast<const u32x4*>(tile + r * RS + 16 * c);
          if (qbase + r < N && 16 * c < cols) *reinterpret_cast<u32x4*>(out + (u32)r * orow + 16 * c) = y;   // orow < 2^26
        }
      }
    }
  };
  if (p.out_f32)
    store(std::true_type{});
  else
    store(std::false_type{});
}

template <int KS, int MT, int QT, int NKH>
int launch_main(const WideParams& pp, hipStream_t stream) {
  WideParams p = pp;
  constexpr int BM = 128 * QT / NKH;
  p.nqb = (p.N + BM - 1) / BM;
  const dim3 grid((unsigned)(p.nqb * p.BH)), block(256);
  if constexpr (KS == 1 && MT <= 2) {
    if (p.kmx == nullptr && p.d == 16 && p.den != nullptr) {
      hipLaunchKernelGGL((wide_kernel<KS, MT, QT, NKH, false, false, true>), grid, block, 0, stream, p);
      return (int)hipGetLastError();
    }
  }
  if (p.kmx != nullptr)
    hipLaunchKernelGGL((wide_kernel<KS, MT, QT, NKH, false, true, false>), grid, block, 0, stream, p);
  else if (p.inv_c == 0.5f && p.inv_c2 == 0.25f)
    hipLaunchKernelGGL((wide_kernel<KS, MT, QT, NKH, true, false, false>), grid, block, 0, stream, p);
  else
    hipLaunchKernelGGL((wide_kernel<KS, MT, QT, NKH, false, false, false>), grid, block, 0, stream, p);
  return (int)hipGetLastError();
}

template <int KS, int MT>
int launch_wide(const WideParams& p, int stages, hipStream_t stream) {
  if (stages & 1) {
    const dim3 pgrid((unsigned)(p.BH * p.nb));
    if (p.kmx != nullptr)
      hipLaunchKernelGGL((wide_pack_kernel<MT, true>), pgrid, dim3(256), 0, stream, p);
    else
      hipLaunchKernelGGL((wide_pack_kernel<MT, false>), pgrid, dim3(256), 0, stream, p);
    const int e = (int)hipGetLastError();
    if (e != 0) return e;
  }
  if (!(stages & 2)) return 0;
  if constexpr (MT == 4) {
    return launch_main<KS, 4, 1, 1>(p, stream);   // 64-query waves would need 128 accumulators more
  } else {
    const long long wg256 = (long long)((p.N + 255) / 256) * p.BH;
    return wg256 >= 2LL * device_cu_count() ? launch_main<KS, MT, 2, 1>(p, stream) : launch_main<KS, MT, 2, 2>(p, stream);
  }
}

}  // namespace

bool wide_shape(int N, int d, int dv) { return wide_shape(N, d, dv, d, dv); }

bool wide_shape(int N, int d, int dv, long long krow, long long vrow) {   // rows of krow, vrow elements
  const size_t nb = ((size_t)N + BN - 1) / BN;
  return d % 8 == 0 && d <= 64 && dv % 8 == 0 && dv <= 128 && nb * (size_t)(32 * dv_tiles(dv) * BN * 2) < ((size_t)1 << 30) && (unsigned long long)N * krow * 2 < ((size_t)1 << 30) &&
         (unsigned long long)N * vrow * 2 < ((size_t)1 << 30);
}

size_t wide_workspace_bytes(int BH, int N, int dv) {
  const size_t nb = ((size_t)N + BN - 1) / BN, DV = 32 * dv_tiles(dv);
  return up256(BH * nb * DV * BN * 2) + up256(BH * nb * DV * 4) + 2 * up256(BH * nb * 4);
}

int launch_wide_parallel(const ParallelArgs& a, void* workspace, bool any_range, hipStream_t stream, const WideStrides* st) {
  const WideScale s = parallel_scale(a.scale);
  WideParams p{};
  p.q = static_cast<const uint16_t*>(a.q);
  p.k = static_cast<const uint16_t*>(a.k);
  p.v = static_cast<const uint16_t*>(a.v);
  p.out = a.out;
  p.den = a.den;
  p.BH = a.BH;
  p.H = st != nullptr ? st->H : a.BH;
  p.N = a.N;
  p.d = a.d;
  p.dv = a.dv;
  for (int i = 0; i < 3; ++i) {   // contiguous: one batch of BH heads
    const long long n[3] = {0, a.N, 1};
    p.ks[i] = st != nullptr ? st->k[i] : n[i] * a.d;
    p.vs[i] = st != nullptr ? st->v[i] : n[i] * a.dv;
    p.os[i] = st != nullptr ? st->out[i] : n[i] * a.dv;
  }
  p.nb = (a.N + BN - 1) / BN;
  const size_t DV = 32 * dv_tiles(a.dv), blocks = (size_t)a.BH * p.nb;
  char* ws = static_cast<char*>(workspace);
  p.vt = reinterpret_cast<uint16_t*>(ws);
  p.sums = reinterpret_cast<float*>(ws + up256(blocks * DV * BN * 2));
  p.eb = reinterpret_cast<int*>(ws + up256(blocks * DV * BN * 2) + up256(blocks * DV * 4));
  p.kmx = any_range ? reinterpret_cast<u32*>(reinterpret_cast<char*>(p.eb) + up256(blocks * 4)) : nullptr;
  p.inv_c = s.inv_c;
  p.inv_c2 = s.inv_c2;
  p.fscale = s.fscale;
  p.qscale = s.qscale;
  p.ones_hi = s.ones_hi;
  p.ones_lo = s.ones_lo;
  p.eps = a.eps;
  p.normalize = a.normalize ? 1 : 0;
  p.out_f32 = a.out_f32 ? 1 : 0;
  p.xcd_cus = device_cu_count() / 8;
  const int ks = a.d <= 16 ? 1 : a.d <= 32 ? 2 : 4, mt = dv_tiles(a.dv);
#define LA_WIDE(K, M) \
  if (ks == K && mt == M) return launch_wide<K, M>(p, a.stages, stream)
  LA_WIDE(1, 1);
  LA_WIDE(1, 2);
  LA_WIDE(1, 4);
  LA_WIDE(2, 1);
  LA_WIDE(2, 2);
  LA_WIDE(2, 4);
  LA_WIDE(4, 1);
  LA_WIDE(4, 2);
  LA_WIDE(4, 4);
#undef LA_WIDE
  return LA_ERR_UNSUPPORTED_DIM;
}

}  // namespace la
