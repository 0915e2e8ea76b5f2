// BASED Taylor feature map for gfx950 (benchmarks/chunked_attention_benchmark.py:23-53):
//   phi(x) = [1, x / d^(1/4), x_i^2 / (sqrt(d) sqrt(2)) (i = 0..d-1),
//             x_i x_j / sqrt(d) (i < j, torch.triu_indices(d, d, 1) row-major order)]
// F = 1 + d + d(d+1)/2 outputs per row.  Products are formed in fp32 and divided by the fp32
// value of each constant, which is how the reference evaluates it for fp32 inputs.
//
// HBM-bound elementwise work on the outputs (F of them for d inputs): a work-group takes RW whole
// rows, whose outputs are one contiguous stretch, and its threads four consecutive outputs at a
// time (16-byte stores; row and feature by increment).  A feature's two factors come from an LDS
// table of index pairs into the row with a 1 appended, worked out once per work-group; a division
// by a power of two (sqrt(d) for d = 16 or 64) is the multiplication with its reciprocal, exactly.
// One thread per output with two integer divisions, a square root and an fp32 division each was
// bound by those: 48016 rows of d = 64 to fp32 (412 MB) 358 -> 125 us (1.15 -> 3.3 TB/s), 262144
// rows of d = 16 160 -> 63 us, 100 rows of d = 64 (eight-row work-groups) 42 -> 16 us.
#include "la_common.hpp"
#include "la_internal.hpp"

namespace la {

namespace {

constexpr int kMaxRows = 32;   // rows per work-group (8 where that leaves CUs idle)
constexpr int kMaxD = 128, kMaxF = 1 + kMaxD + kMaxD * (kMaxD + 1) / 2;

struct FmParams {
  const void* x;
  void* out;
  long long rows;
  int d, F, RW;
  float rrd, rd_r2, rd;
  float inv_rd;   // 1 / rd when rd is a power of two, else 0
  int in_f32, out_f32, vec;
};

__global__ __launch_bounds__(256) void feature_map_kernel(const FmParams p) {
  __shared__ float xs[kMaxRows][kMaxD + 1];
  __shared__ uint16_t pair[kMaxF];   // i | j << 8: the feature is x_i x_j over its divisor, x_d = 1
  const int d = p.d, F = p.F, tid = threadIdx.x;
  const long long r0 = (long long)blockIdx.x * p.RW;
  const int rows = (int)min((long long)p.RW, p.rows - r0);
  for (int t = tid; t < rows * d; t += 256) {
    const int r = t / d, c = t - r * d;
    const size_t idx = (size_t)(r0 + r) * d + c;
    xs[r][c] = p.in_f32 ? static_cast<const float*>(p.x)[idx] : bf16_bits_to_f32(static_cast<const uint16_t*>(p.x)[idx]);
  }
  for (int r = tid; r < rows; r += 256) xs[r][d] = 1.0f;
  for (int f = tid; f < F; f += 256) {
    int i = d, j = d;
    if (f > 2 * d) {
      // off-diagonal pair index q -> (i, j), i < j, row-major over the strict upper triangle:
      // row i starts at off(i) = i*(2d - i - 1)/2
      const int q = f - 2 * d - 1;
      const float b = (float)(2 * d - 1);
      i = (int)((b - __builtin_sqrtf(b * b - 8.0f * (float)q)) * 0.5f);
      i = max(0, min(i, d - 2));
      while (i > 0 && i * (2 * d - i - 1) / 2 > q) --i;
      while ((i + 1) * (2 * d - i - 2) / 2 <= q) ++i;
      j = q - i * (2 * d - i - 1) / 2 + i + 1;
    } else if (f > d) {
      i = j = f - d - 1;
    } else if (f > 0) {
      i = f - 1;
    }
    pair[f] = (uint16_t)(i | (j << 8));
  }
  __syncthreads();
  const int total = rows * F;
  const size_t o0 = (size_t)r0 * F;
  // 1024 outputs per pass: thread t the four from 4 t on
  const int dr = 1024 / F, df = 1024 - dr * F;
  int r = (4 * tid) / F, f = 4 * tid - r * F;
  for (int t = 4 * tid; t < total; t += 1024) {
    float y[4];
    int rr = r, ff = f;
    const bool plain = p.inv_rd != 0.f && f > 2 * d && f + 3 < F;   // four off-diagonal pairs of one row
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      if (t + e < total) {
        const u32 ij = pair[ff];
        const float v = xs[rr][ij & 0xffu] * xs[rr][ij >> 8];
        y[e] = plain ? v * p.inv_rd : ff == 0 ? 1.0f : v / (ff <= d ? p.rrd : ff <= 2 * d ? p.rd_r2 : p.rd);
      }
      if (++ff == F) {
        ff = 0;
        ++rr;
      }
    }
    if (p.vec && t + 4 <= total) {
      if (p.out_f32)
        *reinterpret_cast<f32x4*>(static_cast<float*>(p.out) + o0 + t) = (f32x4){y[0], y[1], y[2], y[3]};
      else
        *reinterpret_cast<u32x2*>(static_cast<uint16_t*>(p.out) + o0 + t) =
            (u32x2){pack_bf16x2(y[0], y[1]), pack_bf16x2(y[2], y[3])};
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        if (t + e >= total) continue;
        if (p.out_f32)
          static_cast<float*>(p.out)[o0 + t + e] = y[e];
        else
          static_cast<uint16_t*>(p.out)[o0 + t + e] = f32_to_bf16_bits(y[e]);
      }
    }
    r += dr;
    f += df;
    if (f >= F) {
      f -= F;
      ++r;
    }
  }
}

}  // namespace

int launch_feature_map(const FeatureMapArgs& a, hipStream_t stream) {
  FmParams p{};
  p.x = a.x;
  p.out = a.out;
  p.rows = a.rows;
  p.d = a.d;
  p.F = 1 + a.d + a.d * (a.d + 1) / 2;
  const double rd = __builtin_sqrt((double)a.d);
  p.rrd = (float)__builtin_sqrt(rd);
  p.rd_r2 = (float)(rd * __builtin_sqrt(2.0));
  p.rd = (float)rd;
  p.in_f32 = a.in_f32 ? 1 : 0;
  p.out_f32 = a.out_f32 ? 1 : 0;
  int ex;
  p.inv_rd = __builtin_frexpf(p.rd, &ex) == 0.5f ? 1.0f / p.rd : 0.f;
  // 32 rows per work-group amortise the table; eight where that would not fill the CUs twice.  Both are
  // multiples of four, so every work-group's stretch of outputs starts 16-byte (bf16: 8-byte) aligned.
  p.RW = a.rows >= 2LL * kMaxRows * device_cu_count() ? kMaxRows : 8;
  p.vec = (reinterpret_cast<uintptr_t>(a.out) & 15) == 0 ? 1 : 0;
  const long long nwg = (a.rows + p.RW - 1) / p.RW;
  if (nwg > 0x7fffffffLL) return -2;
  hipLaunchKernelGGL(feature_map_kernel, dim3((unsigned)nwg), dim3(256), 0, stream, p);
  return (int)hipGetLastError();
}

}  // namespace la
