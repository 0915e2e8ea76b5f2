// One recurrent (decode) step of BASED causal linear attention for gfx950, on the state the
// chunked kernel exports: per head the fp32 (F x (dv + 1)) matrix [S | z] with
// S = sum_u phi(k_u) v_u^T and z = sum_u phi(k_u) over the tokens so far, phi the Taylor
// feature map of benchmarks/chunked_attention_benchmark.py:34-53 in its order
//   phi(x) = [1, x_i / d^(1/4), x_i^2 / (sqrt(d) sqrt(2)), x_i x_j / sqrt(d) (i < j, row-major)],
// F = 1 + d + d(d+1)/2, so that phi(q).phi(k) = 1 + s + s^2/2 with s = q.k / sqrt(d).
// For the new token (q, k, v) of every head the step does
//   [S | z] += phi(k) [v | 1],   num = phi(q)^T [S | z],   y = num[:dv] / (num[dv] + eps)
// which is the chunk recurrence of kernels/nki_attention_chunked.py:65-109 for a chunk of one
// token (its intra-chunk term phi(q).phi(k) v is the contribution of the token's own row of the
// update).  The reference has no decode path; this continues a prefill that exported its state.
//
// A head's F state rows are one work-group's, or R groups of consecutive rows, one work-group
// each, when the heads alone are too few.  A wave takes whole rows, a lane the same column of
// each, so a row is one coalesced load and store, phi(q) and phi(k) of the row are LDS broadcasts,
// the column sums stay in registers and no element needs its row or column worked out.  The loads
// of a work-group's rows (up to 20 per lane) are issued before anything else.  With R = 1 the
// work-group adds its waves' column sums in wave order, normalises and stores the output itself;
// with R > 1 it stores them to a workspace and a combine kernel adds the R partial sums of every
// column in group order (deterministic) and normalises.
//
// HBM-bound in large batches: the state is read and written once (4 F (dv + 1) bytes each way per
// head).  Whole calls, us (a sweep by linear element index, with a division per element, products
// through LDS and one tile of loads at a time / this): B64 H16 d16 dv64 27.0 / 18.2 (4.5 TB/s), dv128
// 41.3 / 30.1, B64 H16 d64 dv64 498 / 260 (4.4 TB/s), B16 H16 d64 136 / 72; B2 H16 d16 dv64 8.4 / 7.1 on
// the device (launch and two memory latencies).
#include <math.h>

#include <algorithm>

#include "la_common.hpp"
#include "la_internal.hpp"

namespace la {

namespace {

struct DecodeParams {
  const void* q;
  const void* k;
  const void* v;
  float* state;
  void* out;
  int BH, d, dv, F;
  float eps, r4, rsq, rd;   // d^(-1/4), 1 / sqrt(2 d), 1 / sqrt(d)
  int normalize, in_f32, out_f32;
};

constexpr int kDecThreads = 256;
constexpr int kDecMaxD = 64;
constexpr int kDecMaxC = 129;   // dv + 1 for dv <= 128
constexpr int kDecMaxF = 1 + kDecMaxD + kDecMaxD * (kDecMaxD + 1) / 2;
constexpr int kDecMinRows = 8;  // fewest state rows per work-group when a head is split
constexpr int kDecLoads = 20;   // state elements of a lane in flight
// States of at most this many floats per head (40 KB; d = 16 with dv <= 65) stay with one
// work-group: the second launch of a split costs as much as it saves.
constexpr int kOneGroupElems = 10240;
#ifndef LA_DECODE_TARGET_WGS
#define LA_DECODE_TARGET_WGS 1024   // split heads until about this many work-groups launch
#endif

__device__ __forceinline__ float load_elem(const void* base, size_t i, bool f32) {
  return f32 ? static_cast<const float*>(base)[i] : bf16_bits_to_f32(static_cast<const uint16_t*>(base)[i]);
}

// Feature f of phi(x) (reference order), x in LDS.
__device__ __forceinline__ float feature(const float* x, int f, int d, float r4, float rsq, float rd) {
  if (f == 0) return 1.f;
  if (f <= d) return x[f - 1] * r4;
  if (f <= 2 * d) {
    const float t = x[f - 1 - d];
    return t * t * rsq;
  }
  // pair t of the strict upper triangle: row i starts at i (2 d - i - 1) / 2
  const int t = f - 1 - 2 * d;
  const float b = (float)(2 * d - 1);
  int i = (int)((b - __builtin_sqrtf(b * b - 8.0f * (float)t)) * 0.5f);
  while (i > 0 && i * (2 * d - i - 1) / 2 > t) --i;
  while ((i + 1) * (2 * d - i - 2) / 2 <= t) ++i;
  return x[i] * x[i + 1 + t - i * (2 * d - i - 1) / 2] * rd;
}

__device__ __forceinline__ float wave_sum(float x) {
#pragma unroll
  for (int m = 1; m < 64; m <<= 1) x += __shfl_xor(x, m);
  return x;
}

// Rows [g RW, min(F, (g + 1) RW)) of head bh = blockIdx.x, g = blockIdx.y.  LPR lanes per row, CPL
// columns per lane (LPR CPL >= dv), NW waves.  PARTIAL: store the group's column sums to
// part[(bh R + g) C + c]; else (R = 1) normalise and store the output.
template <int LPR, int CPL, int NW, bool PARTIAL>
__global__ __launch_bounds__(64 * NW) void based_decode_kernel(const DecodeParams p, int RW, float* part) {
  constexpr int NT = 64 * NW, RPW = 64 / LPR;          // rows per load of a wave
  constexpr int PF = kDecLoads / CPL / 2, WR = PF * RPW, BR = NW * WR;   // rows per wave and block batch
  static_assert(WR <= 64, "a lane per row for the K-sum column");
  __shared__ float xq[kDecMaxD], xk[kDecMaxD];
  __shared__ float phq[kDecMaxF], phk[kDecMaxF];
  __shared__ float red[NW][LPR * CPL], zred[NW];
  const int bh = blockIdx.x, g = blockIdx.y, tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const int d = p.d, dv = p.dv, F = p.F, C = dv + 1;
  const int rb = g * RW, re = min(F, rb + RW), rows = re - rb;
  const int col = lane % LPR, r0 = w * WR;
  float* __restrict__ st = p.state + (size_t)bh * F * C + (size_t)rb * C;

  // A wave takes WR consecutive rows at a time and lane l < WR the K-sum entry of row l, so that the
  // lines between two rows are touched once (the K-sum column in a pass of its own, or rows dealt out
  // one by one, cost HBM a second read and write of those lines).  Two register sets: while one is
  // updated and stored the other's loads are in flight.
  float s[2][PF][CPL], z[2];
  auto load = [&](int set, int first) {
#pragma unroll
    for (int i = 0; i < PF; ++i)
#pragma unroll
      for (int c = 0; c < CPL; ++c) {
        const int r = first + RPW * i + lane / LPR;
        s[set][i][c] = r < rows && col + LPR * c < dv ? st[(size_t)r * C + col + LPR * c] : 0.f;
      }
    z[set] = lane < WR && first + lane < rows ? st[(size_t)(first + lane) * C + dv] : 0.f;
  };
  load(0, r0);
  load(1, r0 + BR);
  float v[CPL];
#pragma unroll
  for (int c = 0; c < CPL; ++c) v[c] = col + LPR * c < dv ? load_elem(p.v, (size_t)bh * dv + col + LPR * c, p.in_f32) : 0.f;
  if (tid < d) xq[tid] = load_elem(p.q, (size_t)bh * d + tid, p.in_f32);
  if (tid >= NT - d) xk[tid - (NT - d)] = load_elem(p.k, (size_t)bh * d + tid - (NT - d), p.in_f32);
  __syncthreads();
  for (int f = tid; f < rows; f += NT) {
    phq[f] = feature(xq, rb + f, d, p.r4, p.rsq, p.rd);
    phk[f] = feature(xk, rb + f, d, p.r4, p.rsq, p.rd);
  }
  __syncthreads();

  float sum[CPL], zsum = 0.f;
#pragma unroll
  for (int c = 0; c < CPL; ++c) sum[c] = 0.f;
  auto update = [&](int set, int first) {
#pragma unroll
    for (int i = 0; i < PF; ++i) {
      const int r = first + RPW * i + lane / LPR;
      if (r >= rows) break;
      const float a = phk[r], b = phq[r];
#pragma unroll
      for (int c = 0; c < CPL; ++c) {
        const float y = __builtin_fmaf(a, v[c], s[set][i][c]);
        if (col + LPR * c < dv) st[(size_t)r * C + col + LPR * c] = y;
        sum[c] = __builtin_fmaf(b, y, sum[c]);
      }
    }
    if (lane < WR && first + lane < rows) {
      const float y = phk[first + lane] + z[set];
      st[(size_t)(first + lane) * C + dv] = y;
      zsum = __builtin_fmaf(phq[first + lane], y, zsum);
    }
  };
  for (int first = r0; first < rows; first += 2 * BR) {
    update(0, first);
    if (first + 2 * BR < rows) load(0, first + 2 * BR);
    update(1, first + BR);
    if (first + 3 * BR < rows) load(1, first + 3 * BR);
  }
  // column sums: the rows of a wave, then the waves in order
#pragma unroll
  for (int c = 0; c < CPL; ++c) {
#pragma unroll
    for (int m = LPR; m < 64; m <<= 1) sum[c] += __shfl_xor(sum[c], m);
    if (lane < LPR) red[w][lane + LPR * c] = sum[c];
  }
  zsum = wave_sum(zsum);
  if (lane == 0) zred[w] = zsum;
  __syncthreads();
  float num = 0.f, den = 0.f;
  if (tid < dv)
#pragma unroll
    for (int x = 0; x < NW; ++x) num += red[x][tid];
#pragma unroll
  for (int x = 0; x < NW; ++x) den += zred[x];
  if (PARTIAL) {
    float* o = part + ((size_t)bh * gridDim.y + g) * C;
    if (tid < dv) o[tid] = num;
    if (tid == dv) o[dv] = den;
    return;
  }
  if (tid < dv) {
    const float y = p.normalize ? num / (den + p.eps) : num;
    const size_t o = (size_t)bh * dv + tid;
    if (p.out_f32)
      static_cast<float*>(p.out)[o] = y;
    else
      static_cast<uint16_t*>(p.out)[o] = f32_to_bf16_bits(y);
  }
}

// Head bh = blockIdx.x: column c = sum over groups g = 0 .. R-1 (in that order) of
// part[(bh R + g) C + c], then the output as in the single-group kernel.
__global__ __launch_bounds__(kDecThreads) void decode_combine_kernel(const DecodeParams p, int R,
                                                                     const float* __restrict__ part) {
  __shared__ float den;
  const int bh = blockIdx.x, tid = threadIdx.x, dv = p.dv, C = dv + 1;
  float colsum = 0.f;
  if (tid < C) {
    // eight loads in flight at a time; the additions keep group order
    const float* src = part + (size_t)bh * R * C + tid;
    int g = 0;
    for (; g + 8 <= R; g += 8) {
      float t[8];
#pragma unroll
      for (int i = 0; i < 8; ++i) t[i] = src[(size_t)(g + i) * C];
#pragma unroll
      for (int i = 0; i < 8; ++i) colsum += t[i];
    }
    for (; g < R; ++g) colsum += src[(size_t)g * C];
  }
  if (tid == dv) den = colsum;
  __syncthreads();
  if (tid < dv) {
    const float y = p.normalize ? colsum / (den + p.eps) : colsum;
    const size_t o = (size_t)bh * dv + tid;
    if (p.out_f32)
      static_cast<float*>(p.out)[o] = y;
    else
      static_cast<uint16_t*>(p.out)[o] = f32_to_bf16_bits(y);
  }
}

}  // namespace

bool decode_shape(int d, int dv) { return d >= 1 && d <= kDecMaxD && dv >= 1 && dv + 1 <= kDecMaxC; }

// Row groups per head: enough work-groups for the chip, at least kDecMinRows rows each; RW =
// rows per group (the last group may have fewer).
static void decode_groups(long long BH, int d, int& R, int& RW) {
  const int F = 1 + d + d * (d + 1) / 2;
  long long r = (LA_DECODE_TARGET_WGS + BH - 1) / BH;
  r = std::max(1LL, std::min(r, (long long)((F + kDecMinRows - 1) / kDecMinRows)));
  RW = (int)((F + r - 1) / r);
  R = (F + RW - 1) / RW;
}

static bool decode_one_group(int d, int dv) { return (1 + d + d * (d + 1) / 2) * (dv + 1) <= kOneGroupElems; }

size_t decode_workspace_bytes(long long BH, int d, int dv) {
  if (decode_one_group(d, dv)) return 0;
  int R, RW;
  decode_groups(BH, d, R, RW);
  return R > 1 ? (size_t)BH * R * (dv + 1) * sizeof(float) : 0;
}

namespace {

template <int NW, bool PARTIAL>
void launch_rows(const DecodeParams& p, int R, int RW, float* part, hipStream_t stream) {
  const dim3 grid((unsigned)p.BH, (unsigned)R), block(64 * NW);
  if (p.dv <= 16)
    hipLaunchKernelGGL((based_decode_kernel<16, 1, NW, PARTIAL>), grid, block, 0, stream, p, RW, part);
  else if (p.dv <= 32)
    hipLaunchKernelGGL((based_decode_kernel<32, 1, NW, PARTIAL>), grid, block, 0, stream, p, RW, part);
  else if (p.dv <= 64)
    hipLaunchKernelGGL((based_decode_kernel<64, 1, NW, PARTIAL>), grid, block, 0, stream, p, RW, part);
  else
    hipLaunchKernelGGL((based_decode_kernel<64, 2, NW, PARTIAL>), grid, block, 0, stream, p, RW, part);
}

}  // namespace

int launch_decode_step(const DecodeArgs& a, hipStream_t stream) {
  DecodeParams p{};
  p.q = a.q;
  p.k = a.k;
  p.v = a.v;
  p.state = a.state;
  p.out = a.out;
  p.BH = a.BH;
  p.d = a.d;
  p.dv = a.dv;
  p.F = 1 + a.d + a.d * (a.d + 1) / 2;
  p.eps = a.eps;
  p.rd = 1.0f / sqrtf((float)a.d);
  p.r4 = sqrtf(p.rd);
  p.rsq = p.rd * 0.70710678118654752f;
  p.normalize = a.normalize ? 1 : 0;
  p.in_f32 = a.in_f32 ? 1 : 0;
  p.out_f32 = a.out_f32 ? 1 : 0;
  int R = 1, RW = p.F;
  if (a.workspace != nullptr && !decode_one_group(a.d, a.dv)) decode_groups(a.BH, a.d, R, RW);
  if (R == 1) {
    // four waves per work-group where heads fill the chip (B64 H16 d16 dv64, with one register set: 20.1
    // us, eight 21.5, sixteen 29.1), eight where their latency counts or rows have 128 columns (B64 H16
    // dv128 32.2 us, 33.0 with four)
    if (a.dv <= 64 && a.BH > device_cu_count())
      launch_rows<4, false>(p, 1, RW, nullptr, stream);
    else
      launch_rows<8, false>(p, 1, RW, nullptr, stream);
  } else {
    float* part = static_cast<float*>(a.workspace);
    launch_rows<4, true>(p, R, RW, part, stream);
    hipLaunchKernelGGL(decode_combine_kernel, dim3((unsigned)a.BH), dim3(kDecThreads), 0, stream, p, R,
                       static_cast<const float*>(part));
  }
  return (int)hipGetLastError();
}

}  // namespace la
