// Density-field quantization of the SSM state at a chunk boundary (gfx950).
//
// training/df_ssm_mamba2_distill_dfw.py:139-165 (df_ssd_scan) quantizes the running state after
// every block_len tokens, per (sequence, head, state row p) over its d_state values:
//   mean, std (unbiased, clamped to 1e-8); lo = mean - 3 std; range = max(6 std, 1e-8)
//   hs = clamp((h - lo) / range, 0, 1); hc = clamp(hs + e, 0, 1) with sigma-delta error e
//   q  = (number of bank thresholds below hc) / KK              (SprayBank.quantize, :88-91)
//   e  = round(clamp(hc - q, -1, 1) 2^(bits-1)) / 2^(bits-1)     (_quantize_error, :105-110)
//   h  = q range + lo
// Two rows of 128 values per wave (half-wave h: row 2w + h; lane l of the half: values 4l .. 4l+3,
// one 16-byte access, so the access instructions of a workgroup's four waves cover 4 KiB
// contiguous). The two row sums are fp64 sums over the adjacent-pair tree: (v0 + v1) + (v2 + v3) in
// the lane, then a butterfly over the 32 lanes of the half (a + b is the same bits as b + a), so a
// sequential restatement with the same tree reproduces them exactly; every other operation is a
// single correctly rounded fp32 operation (no contraction).
//
// Bound by HBM (16 bytes per value), as long as the arithmetic stays below it: about 280 wave
// instructions per 256 values. So the butterflies run on DPP and lane swaps, the four threshold
// searches of a lane advance together (a fixed number of steps on thresholds padded to a power of
// two: their LDS reads overlap, and up to 64 thresholds fit one row of banks), the quotients count /
// kk come from a table, the row's divisions share one reciprocal, the division by the power of two is
// a product, and a workgroup walks many row groups, the next one's values on their way
// (thresholds and quotients are set up once). 393 216 rows with 64 thresholds, against one row group per
// workgroup and four searches one after the other: 195 -> 137 us with an error (5.9 TB/s; 8192 workgroups
// 145, 2048 158 us), 214 -> 130 us without, which is the arithmetic.
#include "common.h"
#include "dfssm_kernels.h"

namespace dfssm {

constexpr int kDfRows = 8;        // rows per workgroup and turn (4 waves x 2)
constexpr int kDfGrid = 256 * 64;  // workgroups at most: eight rounds of 32 waves per CU
constexpr int kStateDfSteps = 11;  // 2^11 > kStateDfMaxKK
static_assert((1 << kStateDfSteps) > kStateDfMaxKK && (1 << (kStateDfSteps - 1)) <= kStateDfMaxKK, "steps");

// Sum over the 32 lanes of each half-wave, every lane with the total: the butterfly xor 1, 2, 4, 8,
// 16. After two steps the lanes of a quad agree, so the mirror of 8 lanes stands for xor 4 and the
// mirror of 16 for xor 8.
__device__ __forceinline__ double tree_sum32(double v) {
  v += dpp_f64<0xB1>(v);   // quad_perm 1,0,3,2
  v += dpp_f64<0x4E>(v);   // quad_perm 2,3,0,1
  v += dpp_f64<0x141>(v);  // row_half_mirror
  v += dpp_f64<0x140>(v);  // row_mirror
  const uint64_t u = __builtin_bit_cast(uint64_t, v);
  const auto lo = __builtin_amdgcn_permlane16_swap((uint32_t)u, (uint32_t)u, false, false);
  const auto hi = __builtin_amdgcn_permlane16_swap((uint32_t)(u >> 32), (uint32_t)(u >> 32), false, false);
  return __builtin_bit_cast(double, ((uint64_t)hi[0] << 32) | lo[0]) +
         __builtin_bit_cast(double, ((uint64_t)hi[1] << 32) | lo[1]);
}

template <bool ERR>
__global__ __launch_bounds__(32 * kDfRows) void state_df_kernel(StateDfArgs a, int steps) {
  __shared__ float R[2 * kStateDfMaxKK];      // 2^steps - 1 sorted thresholds, +inf past kk
  __shared__ float quot[kStateDfMaxKK + 1];   // n / kk
  const int tid = threadIdx.x, lane = tid & 31;
  for (int i = tid; i < (1 << steps) - 1; i += 32 * kDfRows) R[i] = i < a.kk ? a.thresholds[i] : __builtin_inff();
  for (int i = tid; i <= a.kk; i += 32 * kDfRows) quot[i] = (float)i / (float)a.kk;
  __syncthreads();
  const float scale = a.sd_bits < 32 ? (float)(1 << (a.sd_bits - 1)) : 1.0f;
  const float inv_scale = 1.0f / scale;  // a power of two: e / scale == e inv_scale
  const long long stride = (long long)gridDim.x * kDfRows;
  long long row = (long long)blockIdx.x * kDfRows + (tid >> 5);
  // rows past the end re-read the last one (a half-wave still takes part in the exchanges)
  auto at = [&](float* p, long long r) { return p + (r < a.rows ? r : a.rows - 1) * 128 + 4 * lane; };
  f32x4 hn = ld_nt_f4(at(a.h, row)), en = {0.0f, 0.0f, 0.0f, 0.0f};
  if (ERR) en = ld_nt_f4(at(a.sd_error, row));
  for (long long base = (long long)blockIdx.x * kDfRows; base < a.rows; base += stride, row += stride) {
    const f32x4 hv = hn, ev = en;
    hn = ld_nt_f4(at(a.h, row + stride));  // (past the last turn: unused)
    if (ERR) en = ld_nt_f4(at(a.sd_error, row + stride));
    const double S = tree_sum32(((double)hv.x + (double)hv.y) + ((double)hv.z + (double)hv.w));
    const float mean = (float)(S / 128.0);
    const float d0 = hv.x - mean, d1 = hv.y - mean, d2 = hv.z - mean, d3 = hv.w - mean;
    const double SS = tree_sum32(((double)d0 * (double)d0 + (double)d1 * (double)d1) +
                                 ((double)d2 * (double)d2 + (double)d3 * (double)d3));
    float sd = sqrt_rn((float)(SS / 127.0));
    sd = sd > 1e-8f ? sd : 1e-8f;
    const float t3 = 3.0f * sd, t6 = 6.0f * sd;
    const float lo = mean - t3;
    const float range = t6 > 1e-8f ? t6 : 1e-8f;
    // num / range for all values of the row as one product each: in fp64 num * RN(1 / range) is within
    // 2^-52 of the quotient, and a quotient of two fp32 values is at least 2^-49 (relative) away from
    // any midpoint of neighbouring normal fp32 values, so both round to the same fp32 value. A subnormal
    // quotient can be a tie; it needs lo = 0 (else num is 0 or at least 2^-50 range): that row divides
    const double rinv = 1.0 / (double)range;
    const bool any0 = __builtin_expect(__builtin_amdgcn_ballot_w64(lo == 0.0f) != 0, 0);  // uniform
    float quo[4], hc[4], out[4], err[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) quo[k] = (float)((double)(hv[k] - lo) * rinv);
    if (any0) {
#pragma unroll
      for (int k = 0; k < 4; ++k) quo[k] = lo == 0.0f ? (hv[k] - lo) / range : quo[k];
    }
    uint32_t first[4];  // number of thresholds below hc, times 4
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      float hs = quo[k];
      hs = hs < 0.0f ? 0.0f : (hs > 1.0f ? 1.0f : hs);
      hc[k] = hs;
      if (ERR) {
        const float c = hs + ev[k];
        hc[k] = c < 0.0f ? 0.0f : (c > 1.0f ? 1.0f : c);
      }
      first[k] = 0;
    }
#pragma unroll
    for (int i = kStateDfSteps - 1; i >= 0; --i) {
      if (i < steps) {  // uniform
#pragma unroll
        for (int k = 0; k < 4; ++k)
          first[k] += *(const float*)((const char*)R + first[k] + 4 * ((1 << i) - 1)) < hc[k] ? 4 << i : 0;
      }
    }
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const float q = *(const float*)((const char*)quot + first[k]);
      float e = hc[k] - q;  // (both in [0, 1]: the reference's clamp to [-1, 1] changes nothing)
      if (a.sd_bits < 32) e = __builtin_rintf(e * scale) * inv_scale;
      err[k] = e;
      const float qr = q * range;
      out[k] = qr + lo;
    }
    if (row < a.rows) {
      st_nt_f4(at(a.h, row), f32x4{out[0], out[1], out[2], out[3]});
      if (ERR) st_nt_f4(at(a.sd_error, row), f32x4{err[0], err[1], err[2], err[3]});
    }
  }
}

hipError_t launch_state_df(const StateDfArgs& a, hipStream_t s) {
  if (a.rows <= 0) return hipSuccess;
  const long long groups = (a.rows + kDfRows - 1) / kDfRows;
  const dim3 g((unsigned)(groups < kDfGrid ? groups : kDfGrid));
  int steps = 1;  // 2^steps > kk
  while ((1 << steps) <= a.kk) ++steps;
  if (a.sd_error) hipLaunchKernelGGL(state_df_kernel<true>, g, dim3(32 * kDfRows), 0, s, a, steps);
  else hipLaunchKernelGGL(state_df_kernel<false>, g, dim3(32 * kDfRows), 0, s, a, steps);
  return hipGetLastError();
}

}  // namespace dfssm
