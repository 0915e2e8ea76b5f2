// State import and export for the segment-state chunked shapes (bf16, d <= 64, dv <= 128), whose
// sequence kernels keep their states in an internal basis: the states here are the caller's fp32
// (BH, F, dv + 1) = [sum phi(k) v^T | sum phi(k)] in the feature order of taylor_feature_map
// (benchmarks/chunked_attention_benchmark.py:34-53), phi taken of a x with a = (scale^2 d)^(1/4).
// phi is never written to memory: the quadratic features factor as x_i x_j, so every contraction
// over them is a product over j (matrix cores) for each i.
//
// Precision.  Both directions stand in for fp32 products of phi with V or with the state, so every
// operand keeps its bits.  Export: a product k_i v has at most 16 significant bits and is carried as
// bf16 hi + lo, exactly and over the whole range of fp32, against the bf16 rows of k: no channel,
// column or token takes bits from another.  Import: a state entry is carried as three bf16 parts
// (24 bits, exactly) against the bf16 rows of q.  Sums are fp32.  Relative error (2-norm) against 64
// bits, against fp32 phi and fp32 GEMMs on the same inputs: quadratic state rows at B1 H4 N3001 d64
// dv64 1.1e-7 (9.0e-7); the first 64 outputs after a state of 500 tokens 6.4e-7 (1.4e-6), of a column
// of v 2^-28 below the others 4.1e-7 (1.2e-6).
//
// Measured at B1 H16 N3001 d64 dv64 (us): prep 8 + export 66, pack 9 + apply 65, where
// phi written to memory and GEMMs took 1210.
//
//   sprep_kernel    64-token chunks of k and v transposed to rows of tokens, once
//   sexport_kernel  state rows from those: work-group = (head, 32 value columns, four i0), the
//                   chunks through an LDS ring; parts of the sequence where heads are few, added
//                   by scombine_kernel in order (no atomics)
//   spack_kernel    a state's rows as bf16 MFMA fragments in three parts, 1 KB each, i-major
//   sapply_kernel   phi(a q) [S | z] added to a numerator and denominator, and the division
#include <type_traits>

#include "../../include/based_la.h"
#include "../../include/based_la_ext.h"
#include "la_common.hpp"
#include "la_internal.hpp"
#include "la_stage.hpp"

namespace la {
namespace {

constexpr int TC = 64;          // tokens per chunk of the export (a transposed row: 128 bytes)
// Rows are swizzled by swz64; the transposing 8-byte writes (rows four apart) are two-way conflicts at most.
__host__ __device__ __forceinline__ long long feat(int d) { return 1 + d + (long long)d * (d + 1) / 2; }
// First off-diagonal feature row of x_i x_j, j > i (row of j = i + 1).
__host__ __device__ __forceinline__ int off_row(int d, int i) { return 1 + 2 * d + i * (2 * d - i - 1) / 2; }

struct ExportParams {
  const uint16_t* k;
  const uint16_t* v;
  const float* state_in;
  float* dst;             // state_out, or the parts [S][BH][F][dv + 1]
  u32* far;               // [BH][chunks]: not 0 where a product k_i v may be infinite
  uint16_t* kv;           // [BH][chunks][32 DT k rows, 32 nct v rows][TC] bf16
  int BH, N, d, dv, nct, ngrp, parts, cpp;   // column tiles, i0 groups, parts of cpp 64-token chunks
  float c_lin, c_diag, c_off;                // a / d^(1/4), a^2 / sqrt(2 d), a^2 / sqrt(d)
};

// One 4-token x 4-column group of a bf16 array [rows][w]: rows row0 .. row0 + 3 (zero past N),
// columns col .. col + 3 (zero past w).
template <bool VEC>
__device__ __forceinline__ void load44(const uint16_t* __restrict__ g, int row0, int col, int N, int w, u32x2 (&x)[4]) {
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    x[i] = (u32x2){0u, 0u};
    if (row0 + i >= N) continue;
    const uint16_t* src = g + (size_t)(row0 + i) * w + col;
    if (VEC) {
      if (col < w) x[i] = *reinterpret_cast<const u32x2*>(src);
    } else {
      u32 e[4];
#pragma unroll
      for (int t = 0; t < 4; ++t) e[t] = col + t < w ? src[t] : 0u;
      x[i] = (u32x2){e[0] | (e[1] << 16), e[2] | (e[3] << 16)};
    }
  }
}
// The group transposed into rows row .. row + 3 at tokens t0 .. t0 + 3.  Returns its largest magnitude (bf16 bits).
__device__ __forceinline__ u32 store44(uint16_t* dst, int row, int t0, const u32x2 (&x)[4]) {
  u32 m = 0u;
#pragma unroll
  for (int c = 0; c < 4; ++c) {
    u32 y[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      y[i] = (c & 1) ? x[i][c >> 1] >> 16 : x[i][c >> 1] & 0xffffu;
      m = max(m, y[i] & 0x7fffu);
    }
    *reinterpret_cast<u32x2*>(dst + (row + c) * TC + (((t0 >> 3) ^ swz64(row + c)) << 3) + (t0 & 4)) =
        (u32x2){y[0] | (y[1] << 16), y[2] | (y[3] << 16)};
  }
  return m;
}

// One work-group per (chunk, head).
template <int DT, bool VEC>
__global__ __launch_bounds__(256) void sprep_kernel(const ExportParams p) {
  __shared__ __attribute__((aligned(16))) uint16_t img[(32 * DT + 128) * TC];
  const int tid = threadIdx.x, N = p.N, d = p.d, dv = p.dv, nch = (N + TC - 1) / TC;
  const int bh = blockIdx.x / nch, c = blockIdx.x - bh * nch;
  const uint16_t* __restrict__ kg = p.k + (size_t)bh * N * d;
  const uint16_t* __restrict__ vg = p.v + (size_t)bh * N * dv;
  u32x2 kx[4], vx[2][4];
  const int kcol = 4 * (tid % (8 * DT)), kt0 = 4 * (tid / (8 * DT));
  const bool kst = DT == 2 || tid < 128;
  if (kst) load44<VEC>(kg, TC * c + kt0, kcol, N, d, kx);
  const int vg4 = 8 * p.nct, ngr = 16 * vg4;   // v: 4-column groups per row, groups of a chunk
#pragma unroll
  for (int x = 0; x < 2; ++x)
    if (tid + 256 * x < ngr) load44<VEC>(vg, TC * c + 4 * ((tid + 256 * x) / vg4), 4 * ((tid + 256 * x) % vg4), N, dv, vx[x]);
  __shared__ u32 wm[2][4];
  u32 mk = 0u, mv = 0u;
  if (kst) mk = store44(img, kcol, kt0, kx);
#pragma unroll
  for (int x = 0; x < 2; ++x)
    if (tid + 256 * x < ngr)
      mv = max(mv, store44(img, 32 * DT + 4 * ((tid + 256 * x) % vg4), 4 * ((tid + 256 * x) / vg4), vx[x]));
  mk = wave_max_u32(mk);
  mv = wave_max_u32(mv);
  if ((tid & 63) == 0) {
    wm[0][tid >> 6] = mk;
    wm[1][tid >> 6] = mv;
  }
  __syncthreads();
  if (tid == 0) {   // exponents of the largest |k| and |v|: their sum bounds the products below 2^128, or does not
    mk = max(max(wm[0][0], wm[0][1]), max(wm[0][2], wm[0][3])) >> 7;
    mv = max(max(wm[1][0], wm[1][1]), max(wm[1][2], wm[1][3])) >> 7;
    p.far[(size_t)bh * nch + c] = mk == 255u || mv == 255u || mk + mv > 2u * 127u + 125u ? 1u : 0u;
  }
  const int units = (32 * DT + 32 * p.nct) * TC / 8;
  u32x4* dst = reinterpret_cast<u32x4*>(p.kv + ((size_t)bh * nch + c) * ((32 * DT + 32 * p.nct) * TC));
  for (int x = tid; x < units; x += 256) dst[x] = reinterpret_cast<const u32x4*>(img)[x];
}

// ---------------------------------------------------------------- export
// DT 32-wide tiles of j (d <= 32 DT).  The quadratic work-groups: wave w takes i0 = 4 g + w and
// i1 = i0 + 16 DT; A = the k rows j over tokens, B = the products k_i v of a value column (formed in
// registers: 44 VALU per fragment for the six MFMAs of two), so C[j][column] is the state row (i, j).
// Only tiles with j >= i are formed: i0 both (DT = 2) or the one, i1 the last.  The last work-group of
// a (head, column tile) takes the linear rows, the constant row and, in column tile 0, the K-sums (the
// Gram matrix of [k | 1]).
// What bounds it: VALU (88 per K step and wave against six MFMAs and five LDS reads).  The products as
// fp16 hi + lo with one exponent of k and of v per head, two packed VALU per pair, took 57 us (and 11
// for maxima and rows against 8) and lost the bits of every channel far below the head's largest.
// 32 columns per work-group rather than dv: at 16 heads, d = 64 that makes 288 work-groups for
// 256 CUs without splitting the sequence, whose parts would cost a pass over fp32 partials; two fit a
// CU (128 VGPRs; with 147 and one per CU the last 32 ran a second round: 90 us for 66).  Eight waves
// share the tokens, for the LDS and MFMA latencies that four leave open: waves 0-3 the even chunks,
// waves 4-7 the odd ones with the same rows, added through LDS at the end.
template <int DT>
__global__ __launch_bounds__(512, 4) void sexport_kernel(const ExportParams p) {
  constexpr int NS = 3, CW = DT + 1;           // ring stages (two chunks each); 1 KB copies per wave and stage
  constexpr int CH = 32 * CW * TC;             // halves per chunk in a stage
  __shared__ __attribute__((aligned(16))) uint16_t ring[NS][2 * CH];
  const int tid = threadIdx.x, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6), h = lane >> 5, n = lane & 31;
  const int w = wv & 3, half = wv >> 2;
  int id = blockIdx.x;
  const int bh = id % p.BH;
  id /= p.BH;
  const int ct = id % p.nct;
  id /= p.nct;
  const int g = id % (p.ngrp + 1), part = id / (p.ngrp + 1);
  const bool linear = g == p.ngrp;
  const int N = p.N, d = p.d, dv = p.dv;
  const int nch = (N + TC - 1) / TC, c0 = part * p.cpp, c1 = min(c0 + p.cpp, nch), nst = (c1 - c0 + 1) / 2;
  const int cbytes = (32 * DT + 32 * p.nct) * TC * 2;
  // chunks c0 .. c1 - 1, a resource for each stage of two; a missing second chunk lies past it and reads
  // as zeros, which add nothing
  const char* kv = reinterpret_cast<const char*>(p.kv) + (size_t)bh * nch * cbytes;
  // wave wv copies 1 KB units wv, wv + 8, ...: per chunk the k rows, then this column tile's v
  // rows; stages past the last read nothing, so that every wave's count of copies is the same
  auto issue = [&](int s) {
    const u32 lds = lds_addr(&ring[s % NS][0]);
    const RecordWindow win = record_window(c0 + 2LL * s, c1, 2, (u32)cbytes);
    const u32x4 rk = buffer_rsrc(kv + win.offset, win.bytes);
#pragma unroll
    for (int x = 0; x < CW; ++x) {
      const int u = 8 * x + wv, sub = u >= 4 * CW ? 1 : 0, r = u - 4 * CW * sub;
      lds_copy16(rk, lds + 1024 * u,
                 sub * cbytes + 1024 * (r < 4 * DT ? r : r + 4 * ct) + 16 * lane);
    }
  };
  const int i0 = 4 * g + w, i1 = i0 + 16 * DT;
  f32x16 acc[3];
#pragma unroll
  for (int x = 0; x < 3; ++x) acc[x] = splat16(0.f);
#pragma unroll
  for (int s = 0; s < NS - 1; ++s) issue(s);
  auto frag = [&](const uint16_t* st, int row, int u) {
    return *reinterpret_cast<const u32x4*>(st + row * TC + ((u ^ swz64(row)) << 3));
  };
  // stage s of this wave landed (NS - 2 later ones may be in flight), then every wave's; every wave
  // is past stage s - 1, whose place the next copies take.  Returns this wave's chunk.
  auto next = [&](int s) {
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"i"((NS - 2) * CW) : "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    issue(s + NS - 1);
    return static_cast<const uint16_t*>(&ring[s % NS][half * CH]);
  };
  // Products of a K step.  FAR: the remainder of an infinite one (inf - inf), or none beside an infinite
  // k_j (0 inf), is a tiny number of the product's sign.
  constexpr float tiny = 0x1p-126f;
  auto step = [&](auto far_tag, const uint16_t* kt, const uint16_t* vt, int u) {
    constexpr bool FAR = decltype(far_tag)::value;
    u32x4 kf[DT];
#pragma unroll
    for (int jt = 0; jt < DT; ++jt) kf[jt] = frag(kt, 32 * jt + n, u);
    const u32x4 vf = frag(vt, n, u);
    // the rows i of this half's eight tokens, the same for its 32 lanes
    const u32x4 ki[2] = {frag(kt, i0, u), frag(kt, i1, u)};
    u32x4 hi[2], lo[2];
#pragma unroll
    for (int x = 0; x < 2; ++x)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        // 16 significant bits: the upper half of the word holds eight of them, its remainder is a bf16 too
        const float p0 = bf16_lo_to_f32(ki[x][e]) * bf16_lo_to_f32(vf[e]), p1 = bf16_hi_to_f32(ki[x][e]) * bf16_hi_to_f32(vf[e]);
        const u32 b0 = __builtin_bit_cast(u32, p0), b1 = __builtin_bit_cast(u32, p1);
        float r0 = p0 - bf16_hi_to_f32(b0), r1 = p1 - bf16_hi_to_f32(b1);
        if (FAR) {
          if (r0 == 0.f || __builtin_isinf(p0)) r0 = p0 == 0.f ? 0.f : __builtin_copysignf(tiny, p0);
          if (r1 == 0.f || __builtin_isinf(p1)) r1 = p1 == 0.f ? 0.f : __builtin_copysignf(tiny, p1);
        }
        hi[x][e] = __builtin_amdgcn_perm(b1, b0, 0x07060302u);
        lo[x][e] = __builtin_amdgcn_perm(__builtin_bit_cast(u32, r1), __builtin_bit_cast(u32, r0), 0x07060302u);
      }
#pragma unroll
    for (int x = 0; x < DT + 1; ++x) acc[x] = mfma32x32x16(kf[x < DT ? x : DT - 1], hi[x < DT ? 0 : 1], acc[x]);
#pragma unroll
    for (int x = 0; x < DT + 1; ++x) acc[x] = mfma32x32x16(kf[x < DT ? x : DT - 1], lo[x < DT ? 0 : 1], acc[x]);
  };
  if (!linear) {
    // one rule for the part: as a branch inside one loop the accumulators were copied between the two
    int far = 0;
    for (int c = c0 + tid; c < c1; c += 512) far |= p.far[(size_t)bh * nch + c] != 0u;
    auto run = [&](auto far_tag) {
      for (int s = 0; s < nst; ++s) {
        const uint16_t* kt = next(s);
#pragma unroll 2
        for (int ks = 0; ks < TC / 16; ++ks) step(far_tag, kt, kt + 32 * DT * TC, 2 * ks + h);
      }
    };
    if (__syncthreads_or(far))
      run(std::true_type{});
    else
      run(std::false_type{});
  } else {
    // A operands a[x], B operands b[x] of this wave's products
    const u32x4 one = {0x3f803f80u, 0x3f803f80u, 0x3f803f80u, 0x3f803f80u};   // bf16 1
    for (int s = 0; s < nst; ++s) {
      const uint16_t* kt = next(s);
      const uint16_t* vt = kt + 32 * DT * TC;
#pragma unroll
      for (int ks = 0; ks < TC / 16; ++ks) {
        const int u = 2 * ks + h;
        const u32x4 kf0 = frag(kt, n, u), kf1 = frag(kt, 32 * (DT - 1) + n, u), vf = frag(vt, n, u);
        const u32x4 a0 = w == 1 ? one : kf0, b0 = w <= 1 ? vf : w == 2 ? kf0 : one;
        const u32x4 a1 = w == 2 ? kf0 : kf1, b1 = w <= 1 ? vf : w == 2 ? kf1 : one;
        acc[0] = mfma32x32x16(a0, b0, acc[0]);
        if (DT == 2) {
          acc[1] = mfma32x32x16(a1, b1, acc[1]);
          acc[2] = mfma32x32x16(kf1, kf1, acc[2]);
        }
      }
    }
  }
  // ---- rows out, through LDS: the odd chunks' sums, then (odd + even) as [tile][row][32 columns];
  // all waves copy them out with short loops (written straight from the accumulators, the unrolled
  // stores alone were 20 KB of code, fetched once per work-group)
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // no copy in flight into the ring
  __syncthreads();
  constexpr int NTILE = DT + 1;
  float* sum = reinterpret_cast<float*>(&ring[0][0]);
  static_assert(sizeof(ring) >= 4 * 3 * 16 * 64 * 4, "sums fit in the ring");
  auto slot = [&](int x, int r) { return ((w * 3 + x) * 32 + c32_row(r, h)) * 32 + n; };
  if (half == 1)
#pragma unroll
    for (int x = 0; x < 3; ++x)
#pragma unroll
      for (int r = 0; r < 16; ++r) sum[slot(x, r)] = acc[x][r];
  __syncthreads();
  if (half == 0)
#pragma unroll
    for (int x = 0; x < 3; ++x)
#pragma unroll
      for (int r = 0; r < 16; ++r) sum[slot(x, r)] += acc[x][r];
  __syncthreads();
  const int ld = dv + 1;
  const size_t hb = (size_t)bh * feat(d) * ld;
  float* dst = p.dst + (size_t)part * p.BH * feat(d) * ld + hb;
  const float* sin = p.parts == 1 && p.state_in != nullptr ? p.state_in + hb : nullptr;
  // Half-waves take the rows of the 12 tiles in turn, four at a time (the loads of the old state
  // before the stores: the caller may update a state in place).  row < 0: nothing there.
  auto copy_out = [&](auto where) {
    const int hw = 2 * wv + h;
    for (int x0 = hw; x0 < 4 * 3 * 32; x0 += 64) {
      int o[4];
      float y[4], old[4];
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        const int x = x0 + 16 * t;   // row x & 31 of tile (x >> 5) % 3 of wave x / 96
        float f = 0.f;
        o[t] = x < 4 * 3 * 32 ? where(x / 96, (x >> 5) % 3, x & 31, f) : -1;
        y[t] = sum[(x < 4 * 3 * 32 ? x : 0) * 32 + n] * f;
        old[t] = sin != nullptr && o[t] >= 0 ? sin[o[t]] : 0.f;
      }
#pragma unroll
      for (int t = 0; t < 4; ++t)
        if (o[t] >= 0) dst[o[t]] = y[t] + old[t];
    }
  };
  const int col = 32 * ct + n;
  auto quad = [&](int i, int j, int c, float& f) {
    f = j == i ? p.c_diag : p.c_off;
    return j < i || j >= d ? -1 : (j == i ? 1 + d + i : off_row(d, i) + j - i - 1) * ld + c;
  };
  if (!linear) {
    copy_out([&](int ww, int x, int r, float& f) {
      if (x >= NTILE || col >= dv) return -1;
      return quad(4 * g + ww + (x < DT ? 0 : 16 * DT), 32 * (x < DT ? x : DT - 1) + r, col, f);
    });
    return;
  }
  // wave 0: k V; wave 1: the sum of V in every row of tile 0; column tile 0, wave 2: the Gram tiles
  // (0, 0), (0, 1), (1, 1); wave 3: the sums of k in every column
  copy_out([&](int ww, int x, int r, float& f) {
    const int j = 32 * x + r;
    if (ww == 0 || (ww == 3 && ct == 0 && n == 0)) {
      f = p.c_lin;
      const int c = ww == 0 ? col : dv;
      return x < DT && j < d && (ww == 3 || c < dv) ? (1 + j) * ld + c : -1;
    }
    if (ww == 1) {
      f = 1.0f;
      return x == 0 && r == 0 && col < dv ? col : -1;
    }
    if (ww == 2 && ct == 0 && (DT == 2 || x == 0)) return quad((x == 2 ? 32 : 0) + r, (x >= 1 ? 32 : 0) + n, dv, f);
    return -1;
  });
  if (ct == 0 && tid == 0)
    dst[dv] = (float)(min(N, TC * c1) - min(N, TC * c0)) + (sin != nullptr ? sin[dv] : 0.f);
}

// state_out = state_in (or 0) + the parts in order.
__global__ __launch_bounds__(256) void scombine_kernel(const float* __restrict__ part, const float* __restrict__ state_in,
                                                       float* __restrict__ out, long long n, int parts) {
  const long long i = (long long)blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  float x = 0.f;
  for (int s = 0; s < parts; ++s) x += part[(size_t)s * n + i];
  out[i] = state_in != nullptr ? state_in[i] + x : x;
}

// ---------------------------------------------------------------- import
// Fragments of a state: for every feature row i (0 .. DP - 1, then the linear row DP) and 16-wide
// block J of j (from block i / 16; all blocks of the linear row), for every 32-column tile the three
// bf16 parts of M_i[column][j] as A operands (lane: column n, j = 16 J + 8 h ..),
// M_i[.][j] = S(i, j) for j > i, S(i, i) / sqrt(2) (so that one factor a^2 / sqrt(d) serves the
// row), zero for j < i.  Then Z(i, j), the K-sums the same way, as DT x DB x 3 fragments with rows i.
template <int DP>
struct SPack {
  static constexpr int DB = DP / 16, DT = (DP + 31) / 32;
  static constexpr int NQ = 8 * DB * (DB + 1);     // quadratic blocks (i, J)
  static constexpr int NBLK = NQ + DB;             // + the linear row's
  static constexpr int ZU = 3 * DT * DB;           // 1 KB units of Z
  static __host__ __device__ constexpr int first(int i) {   // block index of (i, i / 16)
    const int I = i / 16;
    return 16 * (I * DB - I * (I - 1) / 2) + (i - 16 * I) * (DB - I);
  }
};
static_assert(SPack<64>::first(63) + 1 == SPack<64>::NQ && SPack<16>::first(15) + 1 == SPack<16>::NQ &&
                  SPack<48>::first(47) + 1 == SPack<48>::NQ && SPack<48>::first(16) == 48,
              "block order");

struct ApplyParams {
  const uint16_t* q;
  const float* state;
  const float* num;       // (BH, N, dv), without the state's part
  const float* den;       // (BH, N)
  void* out;
  uint16_t* frag;         // [BH][NBLK][MT][3][512], then [BH][ZU][512]
  uint16_t* zfrag;
  int BH, N, d, dv;
  float c_lin, c_off, eps;
  int normalize, out_f32;
};

// Work-group (i, head): i < DP a feature row, DP the linear row; its state rows (j >= i) through
// LDS, once.
template <int DP, int MT>
__global__ __launch_bounds__(256) void spack_kernel(const ApplyParams p) {
  using SP = SPack<DP>;
  constexpr int DB = SP::DB;
  __shared__ float row[DP * (32 * MT + 1)];
  const int tid = threadIdx.x, bh = blockIdx.x / (DP + 1), i = blockIdx.x - bh * (DP + 1), d = p.d, dv = p.dv, ld = dv + 1;
  const float* __restrict__ S = p.state + (size_t)bh * feat(d) * ld;
  const int j0 = i < DP ? i : 0, cnt = i < d || i == DP ? d - j0 : 0;   // rows j0 .. d - 1 (none past d)
  // row j0 of a quadratic i is its square; the others follow each other in memory
  const float* __restrict__ rest = i < DP ? S + (size_t)(off_row(d, i) - 1) * ld : S + ld;
  constexpr int PF = 8;   // loads in flight per thread
  for (int x0 = tid; x0 < cnt * ld; x0 += 256 * PF) {
    float y[PF];
#pragma unroll
    for (int u = 0; u < PF; ++u) {
      const int x = x0 + 256 * u;
      y[u] = x >= cnt * ld ? 0.f : i < DP && x < ld ? S[(size_t)(1 + d + i) * ld + x] * 0.70710678118654752f : rest[x];
    }
#pragma unroll
    for (int u = 0; u < PF; ++u)
      if (x0 + 256 * u < cnt * ld) row[x0 + 256 * u] = y[u];
  }
  __syncthreads();
  // a 16-byte unit: column c, rows j .. j + 7; the second and third parts 512 and 1024 halves later.  A
  // part is the upper half of the word, exactly what it leaves the next one; infinities leave nothing.
  auto put = [&](uint16_t* dst, int j, int c) {
    u32x4 p[3];
#pragma unroll
    for (int x = 0; x < 4; ++x) {
      u32 b[2][3];
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        const int r = j + 2 * x + t - j0;
        float y = r >= 0 && r < cnt && c < ld ? row[r * ld + c] : 0.f;
        const bool fin = __builtin_fabsf(y) < __builtin_inff();
#pragma unroll
        for (int k = 0; k < 3; ++k) {
          b[t][k] = y != y ? 0x7fc00000u : __builtin_bit_cast(u32, y) & 0xffff0000u;
          y = fin ? y - __builtin_bit_cast(float, b[t][k]) : 0.f;
        }
      }
#pragma unroll
      for (int k = 0; k < 3; ++k) p[k][x] = (b[0][k] >> 16) | b[1][k];
    }
#pragma unroll
    for (int k = 0; k < 3; ++k) *reinterpret_cast<u32x4*>(dst + 512 * k) = p[k];
  };
  const int J0 = i < DP ? i / 16 : 0, b0 = i < DP ? SP::first(i) : SP::NQ;
  uint16_t* dst = p.frag + ((size_t)bh * SP::NBLK + b0) * (MT * 1536);
  for (int x = tid; x < (DB - J0) * MT * 64; x += 256) {
    const int l = x & 63, mt = (x >> 6) % MT, J = J0 + (x >> 6) / MT, c = 32 * mt + (l & 31);
    put(dst + ((size_t)(J - J0) * MT + mt) * 1536 + 8 * l, 16 * J + 8 * (l >> 5), c < dv ? c : ld);
  }
  if (i < DP && tid < 2 * DB) {   // Z's row i: lanes i % 32 and i % 32 + 32 of its fragments
    const int J = tid >> 1, h = tid & 1;
    put(p.zfrag + (size_t)bh * SP::ZU * 512 + (size_t)((i >> 5) * DB + J) * 1536 + 8 * ((i & 31) + 32 * h),
        16 * J + 8 * h, dv);
  }
}

// Work-group: 128 QT queries of one head, 4 MT waves: wave w takes 32 QT queries (w % 4) and value
// columns 32 (w / 4) .. + 31.  Per feature row i: Y = M_i q on MFMAs (A the row's fragments from
// an LDS ring, B the wave's queries, resident), then acc += q_i Y: 16 QT fused multiply-adds against
// 3 QT x (blocks of the row) MFMAs.  Matrix-core bound once the ring's copies are hidden: a fragment
// (1 KB) feeds QT MFMAs of four waves.  QT = 1 is taken where 256-query work-groups would leave half of
// the CUs idle, and at MT = 4, whose 16 waves have 128 VGPRs each (QT = 2 spills 27 of them: B2 H16
// N3001 d64 dv128 238 us, 211 so).  (Two fp16 parts with an exponent per feature row took 54 us, and lost the bits of
// columns far below the row's largest.)
template <int DP, int MT, int QT, bool VEC>
__global__ __launch_bounds__(256 * MT, MT) void sapply_kernel(const ApplyParams p) {
  using SP = SPack<DP>;
  constexpr int DB = SP::DB, DT = SP::DT, NBLK = SP::NBLK, TQ = 128 * QT;
  constexpr int GB = 4;                            // blocks per stage
  constexpr int UB = 3 * MT, SU = GB * UB;         // 1 KB units per block and per stage
  constexpr int CW = SU / (4 * MT);                // copies per wave and stage
  constexpr int NST = (NBLK + GB - 1) / GB, NS = MT == 4 ? 2 : 4;
  __shared__ __attribute__((aligned(16))) uint16_t ring[NS][SU * 512];
  __shared__ __attribute__((aligned(16))) uint16_t Aq[DP * TQ];
  const int tid = threadIdx.x, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6), h = lane >> 5, n = lane & 31;
  const int w = wv & 3, mt = wv >> 2;
  const int N = p.N, d = p.d, dv = p.dv, ld = dv + 1;
  const int bh = blockIdx.x % p.BH, t0 = (blockIdx.x / p.BH) * TQ;
  const float* __restrict__ S = p.state + (size_t)bh * feat(d) * ld;

  const u32x4 rf = buffer_rsrc(p.frag + (size_t)bh * NBLK * (MT * 1536), (u32)(NBLK * MT * 3072));
  auto issue = [&](int s) {   // past the last stage nothing is read, so that every wave's counts agree
    const u32 base = lds_addr(&ring[s % NS][0]);
#pragma unroll
    for (int x = 0; x < CW; ++x) {
      const int u = 4 * MT * x + wv;
      lds_copy16(rf, base + 1024 * u, s < NST ? s * (SU * 1024) + 1024 * u + 16 * lane : kOffOutOfRange);
    }
  };

  // the ring's first stages before everything else: loads that follow only make the waits on
  // them stricter (they are counted in order)
#pragma unroll
  for (int s = 0; s < NS - 1; ++s) issue(s);

  // ---- queries: fragments, and a table [dim][query] for the factors q_i
  u32x4 qf[QT][DB];
#pragma unroll
  for (int qt = 0; qt < QT; ++qt) {
    const int tok = t0 + 32 * QT * w + 32 * qt + n;
#pragma unroll
    for (int J = 0; J < DB; ++J) {
      qf[qt][J] = load_row8<VEC>(p.q + ((size_t)bh * N + tok) * d, 16 * J + 8 * h, d, tok < N);
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (mt == 0) {
          uint16_t* a = Aq + (16 * J + 8 * h + 2 * e) * TQ + 32 * QT * w + 32 * qt + n;
          a[0] = (uint16_t)(qf[qt][J][e] & 0xffffu);
          a[TQ] = (uint16_t)(qf[qt][J][e] >> 16);
        }
    }
  }
  const float zlin = lane < d ? S[(size_t)(1 + lane) * ld + dv] : 0.f;   // the linear K-sum of lane i
  const float z0 = S[dv];
  auto from_lane = [](float x, int l) {
    return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, x), l));
  };

  // ---- denominator: q^T Z q and the linear K-sums
  float den[QT];
  {
    const u32x4* __restrict__ zf = reinterpret_cast<const u32x4*>(p.zfrag + (size_t)bh * SP::ZU * 512);
    f32x16 Y[QT][DT];
#pragma unroll
    for (int rt = 0; rt < DT; ++rt) {
#pragma unroll
      for (int qt = 0; qt < QT; ++qt) Y[qt][rt] = splat16(0.f);
#pragma unroll
      for (int J = 0; J < DB; ++J)
#pragma unroll
        for (int x = 0; x < 3; ++x) {
          const u32x4 a = zf[((rt * DB + J) * 3 + x) * 64 + lane];
#pragma unroll
          for (int qt = 0; qt < QT; ++qt) Y[qt][rt] = mfma32x32x16(a, qf[qt][J], Y[qt][rt]);
        }
    }
    __syncthreads();   // the table of q
#pragma unroll
    for (int qt = 0; qt < QT; ++qt) {
      const uint16_t* aq = Aq + 32 * QT * w + 32 * qt + n;
      float dq = 0.f, dl = 0.f;
#pragma unroll
      for (int rt = 0; rt < DT; ++rt)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int i0 = 32 * rt + c32_row(r, 0);   // row i0 + 4 h
          if (i0 >= DP) continue;
          dq = __builtin_fmaf(bf16_bits_to_f32(aq[(i0 + 4 * h) * TQ]), Y[qt][rt][r], dq);
        }
#pragma unroll 4
      for (int i = 0; i < DP / 2; ++i) {   // lane half h sums rows h DP / 2 ..
        const float za = from_lane(zlin, i), zb = from_lane(zlin, i + DP / 2);
        dl = __builtin_fmaf(bf16_bits_to_f32(aq[(i + h * (DP / 2)) * TQ]), h ? zb : za, dl);
      }
      dq += __shfl_xor(dq, 32);
      dl += __shfl_xor(dl, 32);
      const int tok = min(t0 + 32 * QT * w + 32 * qt + n, N - 1);
      den[qt] = p.den[(size_t)bh * N + tok] + z0 + dl * p.c_lin + dq * p.c_off;
    }
  }

  f32x16 acc[QT];
#pragma unroll
  for (int qt = 0; qt < QT; ++qt) acc[qt] = splat16(0.f);
  int b = 0;   // block index, i-major
  // Y of one row: blocks J0 .. DB - 1
  auto row = [&](int J0, f32x16 (&Y)[QT]) {
#pragma unroll
    for (int J = 0; J < DB; ++J) {
      if (J < J0) continue;
      if ((b & (GB - 1)) == 0) {
        // stage b / GB landed (NS - 2 later ones may be in flight); every wave is past the stage
        // before, which the next copies overwrite
        asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"i"((NS - 2) * CW) : "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        issue(b / GB + NS - 1);
      }
      const u32x4* st = reinterpret_cast<const u32x4*>(&ring[(b / GB) % NS][((b & (GB - 1)) * UB + 3 * mt) * 512]);
#pragma unroll
      for (int x = 0; x < 3; ++x) {
        const u32x4 a = st[x * 64 + lane];
#pragma unroll
        for (int qt = 0; qt < QT; ++qt) Y[qt] = mfma32x32x16(a, qf[qt][J], Y[qt]);
      }
      ++b;
    }
  };
#pragma unroll
  for (int I = 0; I < DB; ++I) {
#pragma unroll 1
    for (int i = 16 * I; i < 16 * I + 16; ++i) {
      f32x16 Y[QT];
#pragma unroll
      for (int qt = 0; qt < QT; ++qt) Y[qt] = splat16(0.f);
      row(I, Y);
#pragma unroll
      for (int qt = 0; qt < QT; ++qt) {
        const float a = bf16_bits_to_f32(Aq[i * TQ + 32 * QT * w + 32 * qt + n]);
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[qt][r] = __builtin_fmaf(a, Y[qt][r], acc[qt][r]);
      }
    }
  }
  f32x16 Yl[QT];
#pragma unroll
  for (int qt = 0; qt < QT; ++qt) Yl[qt] = splat16(0.f);
  row(0, Yl);
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // no copy outlives the work-group

  // ---- (num + state's) / (den + state's + eps); all loads together (out may be num)
  f32x4 s0[4], num[QT][4];
#pragma unroll
  for (int q4 = 0; q4 < 4; ++q4) {
    const int c = 32 * mt + 8 * q4 + 4 * h;
#pragma unroll
    for (int e = 0; e < 4; ++e) s0[q4][e] = c + e < dv ? S[c + e] : 0.f;
#pragma unroll
    for (int qt = 0; qt < QT; ++qt) {
      const int tok = min(t0 + 32 * QT * w + 32 * qt + n, N - 1);
      const float* np = p.num + ((size_t)bh * N + tok) * dv + c;
      if (VEC) {
        num[qt][q4] = c < dv ? *reinterpret_cast<const f32x4*>(np) : (f32x4){0.f, 0.f, 0.f, 0.f};
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e) num[qt][q4][e] = c + e < dv ? np[e] : 0.f;
      }
    }
  }
#pragma unroll
  for (int qt = 0; qt < QT; ++qt) {
    const int tok = t0 + 32 * QT * w + 32 * qt + n;
    if (tok >= N) continue;
    const float inv = p.normalize ? 1.0f / (den[qt] + p.eps) : 1.0f;
    const size_t ob = ((size_t)bh * N + tok) * dv;
#pragma unroll
    for (int q4 = 0; q4 < 4; ++q4) {
      float y[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int r = 4 * q4 + e;
        const float x = acc[qt][r] * p.c_off + Yl[qt][r] * p.c_lin;
        y[e] = (num[qt][q4][e] + (x + s0[q4][e])) * inv;
      }
      store_out4<VEC>(p.out, p.out_f32 != 0, ob, 32 * mt + 8 * q4 + 4 * h, dv, y);
    }
  }
}

int dp_of(int d) { return 16 * ((d + 15) / 16); }
// Parts of the sequence of an export: one when the (head, column tile, i0 group) work-groups fill
// the CUs, else enough for two per CU, of at least four 64-token chunks.
void export_plan(int BH, int N, int d, int dv, ExportParams& p) {
  p.nct = (dv + 31) / 32;
  const int span = d <= 32 ? 16 : 32;
  p.ngrp = ((d < span ? d : span) + 3) / 4;
  const long long units = (long long)BH * p.nct * (p.ngrp + 1);
  const int nch = (N + TC - 1) / TC, cus = device_cu_count();
  int parts = units >= cus ? 1 : (int)((2LL * cus + units - 1) / units);
  parts = parts < 1 ? 1 : parts;
  if (parts > nch / 4) parts = nch / 4 > 1 ? nch / 4 : 1;
  p.cpp = (nch + parts - 1) / parts;
  p.parts = p.cpp > 0 ? (nch + p.cpp - 1) / p.cpp : 1;
}

struct ExportLayout {
  size_t kv, parts, total;
};
ExportLayout export_layout(int BH, int N, int d, int dv, const ExportParams& p) {
  ExportLayout L{};
  L.kv = up256((size_t)BH * ((N + TC - 1) / TC) * 4);
  L.parts = L.kv + up256((size_t)BH * ((N + TC - 1) / TC) * (32 * (d <= 32 ? 1 : 2) + 32 * p.nct) * TC * 2);
  L.total = L.parts + (p.parts > 1 ? (size_t)p.parts * BH * feat(d) * (dv + 1) * 4 : 0);
  return L;
}
size_t export_bytes(int BH, int N, int d, int dv) {
  ExportParams p{};
  export_plan(BH, N, d, dv, p);
  return export_layout(BH, N, d, dv, p).total;
}

struct ApplyLayout {
  size_t z, total;
};
ApplyLayout apply_layout(int BH, int d, int dv) {
  const int DP = dp_of(d), DB = DP / 16, DT = (DP + 31) / 32, nblk = 8 * DB * (DB + 1) + DB;
  ApplyLayout L{};
  L.z = up256((size_t)BH * nblk * dv_tiles(dv) * 3072);
  L.total = L.z + up256((size_t)BH * 3 * DT * DB * 1024);
  return L;
}

bool aligned(const void* p, uintptr_t b) { return (reinterpret_cast<uintptr_t>(p) & (b - 1)) == 0; }

template <int DP, int MT>
int launch_apply(const ApplyParams& p, hipStream_t stream) {
  hipLaunchKernelGGL((spack_kernel<DP, MT>), dim3((DP + 1) * (unsigned)p.BH), dim3(256), 0, stream, p);
  const int e = (int)hipGetLastError();
  if (e != 0) return e;
  const bool vec = p.d % 8 == 0 && p.dv % 4 == 0 && aligned(p.q, 16) && aligned(p.out, 16) && aligned(p.num, 16);
  const unsigned wg2 = (unsigned)p.BH * (unsigned)((p.N + 255) / 256), wg1 = (unsigned)p.BH * (unsigned)((p.N + 127) / 128);
  const dim3 block(256 * MT);
  if constexpr (MT < 4) {
    if ((int)wg1 > device_cu_count()) {
      if (vec)
        hipLaunchKernelGGL((sapply_kernel<DP, MT, 2, true>), dim3(wg2), block, 0, stream, p);
      else
        hipLaunchKernelGGL((sapply_kernel<DP, MT, 2, false>), dim3(wg2), block, 0, stream, p);
      return (int)hipGetLastError();
    }
  }
  if (vec)
    hipLaunchKernelGGL((sapply_kernel<DP, MT, 1, true>), dim3(wg1), block, 0, stream, p);
  else
    hipLaunchKernelGGL((sapply_kernel<DP, MT, 1, false>), dim3(wg1), block, 0, stream, p);
  return (int)hipGetLastError();
}

template <int DP>
int launch_apply_mt(const ApplyParams& p, hipStream_t stream) {
  switch (dv_tiles(p.dv)) {
    case 1: return launch_apply<DP, 1>(p, stream);
    case 2: return launch_apply<DP, 2>(p, stream);
    default: return launch_apply<DP, 4>(p, stream);
  }
}

int check_state_args(int in_dtype, int B, int H, int N, int d, int dv, float scale) {
  if (B < 0 || H < 0 || N < 0 || d < 1 || dv < 1) return LA_ERR_BAD_SHAPE;
  if (in_dtype != LA_BF16) return LA_ERR_BAD_DTYPE;
  if (d > 64 || dv > 128) return LA_ERR_UNSUPPORTED_DIM;
  if (!(scale > 0.f) || !(scale < 3.4e38f)) return LA_ERR_BAD_SCALAR;
  if ((long long)B * H > 0x7fffffLL || (long long)N * (d > dv ? d : dv) > 0x7fffffffLL) return LA_ERR_BAD_SHAPE;
  return LA_OK;
}

}  // namespace
}  // namespace la

extern "C" {

size_t la_based_state_workspace_bytes(int B, int H, int N, int d, int dv) {
  if (B < 1 || H < 1 || N < 1 || d < 1 || dv < 1 || d > 64 || dv > 128) return 0;
  const size_t a = la::export_bytes(B * H, N, d, dv), b = la::apply_layout(B * H, d, dv).total;
  return a > b ? a : b;
}

int la_based_state_export(const void* k, const void* v, int in_dtype, const float* state_in_or_null, float* state_out,
                          int B, int H, int N, int d, int dv, float scale, void* workspace, size_t workspace_bytes,
                          void* hip_stream) {
  using namespace la;
  const int rc = check_state_args(in_dtype, B, H, N, d, dv, scale);
  if (rc != LA_OK || (long long)B * H * N == 0) return rc;
  if (k == nullptr || v == nullptr || state_out == nullptr) return LA_ERR_NULL_POINTER;
  if (!aligned(k, 2) || !aligned(v, 2) || !aligned(state_out, 4) || !aligned(state_in_or_null, 4)) return LA_ERR_BAD_ALIGNMENT;
  if (workspace == nullptr || workspace_bytes < export_bytes(B * H, N, d, dv)) return LA_ERR_WORKSPACE;
  if (!aligned(workspace, 16)) return LA_ERR_BAD_ALIGNMENT;
  const hipStream_t stream = static_cast<hipStream_t>(hip_stream);
  ExportParams p{};
  export_plan(B * H, N, d, dv, p);
  const double a2 = (double)scale * __builtin_sqrt((double)d), sd = __builtin_sqrt((double)d);   // a^2, sqrt(d)
  p.k = static_cast<const uint16_t*>(k);
  p.v = static_cast<const uint16_t*>(v);
  p.state_in = state_in_or_null;
  p.far = static_cast<u32*>(workspace);
  const ExportLayout L = export_layout(B * H, N, d, dv, p);
  p.kv = reinterpret_cast<uint16_t*>(static_cast<char*>(workspace) + L.kv);
  float* parts = reinterpret_cast<float*>(static_cast<char*>(workspace) + L.parts);
  p.dst = p.parts > 1 ? parts : state_out;
  p.BH = B * H;
  p.N = N;
  p.d = d;
  p.dv = dv;
  p.c_lin = (float)__builtin_sqrt(a2 / sd);
  p.c_diag = (float)(a2 / (sd * 1.4142135623730951));
  p.c_off = (float)(a2 / sd);
  const dim3 pgrid((unsigned)((N + TC - 1) / TC) * (unsigned)p.BH);
  const dim3 grid((unsigned)((long long)p.BH * p.nct * (p.ngrp + 1) * p.parts));
  const bool vec = d % 4 == 0 && dv % 4 == 0 && aligned(k, 8) && aligned(v, 8);
  if (d <= 32) {
    if (vec)
      hipLaunchKernelGGL((sprep_kernel<1, true>), pgrid, dim3(256), 0, stream, p);
    else
      hipLaunchKernelGGL((sprep_kernel<1, false>), pgrid, dim3(256), 0, stream, p);
    hipLaunchKernelGGL((sexport_kernel<1>), grid, dim3(512), 0, stream, p);
  } else {
    if (vec)
      hipLaunchKernelGGL((sprep_kernel<2, true>), pgrid, dim3(256), 0, stream, p);
    else
      hipLaunchKernelGGL((sprep_kernel<2, false>), pgrid, dim3(256), 0, stream, p);
    hipLaunchKernelGGL((sexport_kernel<2>), grid, dim3(512), 0, stream, p);
  }
  const int e = (int)hipGetLastError();
  if (e != 0 || p.parts == 1) return e;
  const long long n = (long long)p.BH * feat(d) * (dv + 1);
  hipLaunchKernelGGL(scombine_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, stream, parts, state_in_or_null,
                     state_out, n, p.parts);
  return (int)hipGetLastError();
}

int la_based_state_apply(const void* q, int in_dtype, const float* state, const float* num, const float* den, void* out,
                         int out_dtype, int B, int H, int N, int d, int dv, float scale, float eps, int normalize,
                         void* workspace, size_t workspace_bytes, void* hip_stream) {
  using namespace la;
  const int rc = check_state_args(in_dtype, B, H, N, d, dv, scale);
  if (rc != LA_OK) return rc;
  if (out_dtype != LA_F32 && out_dtype != LA_BF16) return LA_ERR_BAD_DTYPE;
  if (!(eps >= 0.f) || !(eps < 3.4e38f)) return LA_ERR_BAD_SCALAR;
  if ((long long)B * H * N == 0) return LA_OK;
  if (q == nullptr || state == nullptr || num == nullptr || den == nullptr || out == nullptr) return LA_ERR_NULL_POINTER;
  if (!aligned(q, 2) || !aligned(state, 4) || !aligned(num, 4) || !aligned(den, 4) ||
      !aligned(out, out_dtype == LA_F32 ? 4 : 2))
    return LA_ERR_BAD_ALIGNMENT;
  const ApplyLayout L = apply_layout(B * H, d, dv);
  if (workspace == nullptr || workspace_bytes < L.total) return LA_ERR_WORKSPACE;
  if (!aligned(workspace, 16)) return LA_ERR_BAD_ALIGNMENT;
  const hipStream_t stream = static_cast<hipStream_t>(hip_stream);
  const double a2 = (double)scale * __builtin_sqrt((double)d), sd = __builtin_sqrt((double)d);
  ApplyParams p{};
  p.q = static_cast<const uint16_t*>(q);
  p.state = state;
  p.num = num;
  p.den = den;
  p.out = out;
  p.frag = static_cast<uint16_t*>(workspace);
  p.zfrag = reinterpret_cast<uint16_t*>(static_cast<char*>(workspace) + L.z);
  p.BH = B * H;
  p.N = N;
  p.d = d;
  p.dv = dv;
  p.c_lin = (float)__builtin_sqrt(a2 / sd);
  p.c_off = (float)(a2 / sd);
  p.eps = eps;
  p.normalize = normalize != 0;
  p.out_f32 = out_dtype == LA_F32;
  switch (dp_of(d)) {
    case 16: return launch_apply_mt<16>(p, stream);
    case 32: return launch_apply_mt<32>(p, stream);
    case 48: return launch_apply_mt<48>(p, stream);
    default: return launch_apply_mt<64>(p, stream);
  }
}

}  // extern "C"
