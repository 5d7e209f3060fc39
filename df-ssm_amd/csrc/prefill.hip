// Prompt prefill, layer-major (gfx950): the n prompt tokens of every sequence go through one
// layer together, then the next layer. The projections and their prologues are row-independent,
// so they run on all batch x n rows at once; only the two recurrences walk the tokens, here:
//
//   conv_tokens_kernel  conv + SiLU of every (token, channel) from the raw projection rows:
//                    out = s0 w0 + s1 w1 + s2 w2 + x w3 + b (left to right, fp32), fp16(out sigmoid(out)),
//                    and the head's decay factors softplus dt, exp(dt A). x goes to the rows the scan
//                    overwrites with g, B | C to rows of their own.
//   ssm_scan_kernel  the SSM recurrence and the gate, one workgroup per (sequence, head, 16-row
//                    blocks): the fp32 state stays in registers for all n tokens (read and written
//                    once per layer instead of once per token).
//
// Every rounding here and the order of the scan's readout are the decode step's (ssm_kernel), so together
// with the row-wise kernels the prefill equals n calls of the decode step bit for bit (Mamba-2
// recurrence of df_ssm_kernels.cu:53-103 / training/df_ssm_mamba2_distill_dfw.py:346-381, evaluated
// token by token as the reference's cpu_inference_driver.py:186-204 ingests a prompt), up to the fp64
// sums that the decode's launches and the prefill add in different orders: sum(x^2) and sum(g^2) (here in
// prep_kernel's order at every row count) and the LoRA sums (above 64 rows on the fp64 matrix cores). Two
// orders are a few units of 2^-53 apart at most, which shows only where an fp32 rounding boundary lies
// between them: about one row in 10^9 for sum(g^2).
#include <type_traits>

#include "common.h"
#include "dfssm_kernels.h"

namespace dfssm {

// The caller's conv tensors carry no alignment beyond their 2-byte elements (the address mode of the
// target takes a vector access at any address).
typedef u32x4 u32x4_a2 __attribute__((aligned(2)));

// ------------------------------------------------------------------------------------------
// conv_tokens_kernel: a thread owns 8 channels and walks tc tokens (16-byte rows in and out), the
// three raw inputs before its first token re-read from the rows (or the conv state). The tokens
// of a sequence are independent once the raw rows are kept, so they spread over the grid: a thread
// that walked the whole sequence with the outputs in place took 208 us for 999 tokens of one
// sequence at the 1.3B shape (17 workgroups on the chip), this one 13 us. The first token range also writes the new
// conv state, the last three raw inputs. The last block of the x grid computes the decay factors of
// its tokens, one (token, head) per thread. VALU issue and the rows' traffic take about the same time (36
// instructions per value, 20 of them the exponential and the reciprocal; 133 us for 16 384 rows of the 2.7B
// shape, 71 us at the rate of a copy).
// ------------------------------------------------------------------------------------------
__global__ __launch_bounds__(256) void conv_tokens_kernel(ConvTokArgs a) {
  const int tid = threadIdx.x, b = blockIdx.z;
  const int t0 = (int)blockIdx.y * a.tc, t1 = t0 + a.tc < a.T ? t0 + a.tc : a.T;
  const size_t row0 = (size_t)b * a.T;
  if (blockIdx.x == gridDim.x - 1) {
    for (int i = tid; i < (t1 - t0) * a.H; i += 256) {
      const int t = t0 + i / a.H, hd = i % a.H;
      const float dt = dev_log1pf(dev_expf(h2f(a.dt[(row0 + t) * a.ld + hd]) + a.dt_bias[hd]));
      a.dec_out[(row0 + t) * a.H + hd] = float2{dt, dev_expf(dt * -dev_expf(a.A_log[hd]))};
    }
    return;
  }
  const int ch = 8 * ((int)blockIdx.x * 256 + tid);
  if (ch >= a.C) return;
  const uint16_t* raw = a.xbc + row0 * a.ld + ch;
  u32x4 wr[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) wr[i] = *(const u32x4_a2*)(a.w + (size_t)ch * 4 + 8 * i);
  const u32x4 br = *(const u32x4_a2*)(a.b + ch);
  uint16_t s[3][8];  // the three inputs before the current token
  u32x4_a2* cs = (u32x4_a2*)(a.state + ((size_t)b * a.C + ch) * 3);  // 8 channels x 3 halves
  if (t0 == 0) {
    const u32x4 st[3] = {cs[0], cs[1], cs[2]};
#pragma unroll
    for (int e = 0; e < 8; ++e)
#pragma unroll
      for (int k = 0; k < 3; ++k) s[k][e] = (uint16_t)(st[(3 * e + k) >> 3][((3 * e + k) & 7) >> 1] >> (16 * ((3 * e + k) & 1)));
  } else {
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      const u32x4 v = *(const u32x4*)(raw + (size_t)(t0 - 3 + k) * a.ld);
#pragma unroll
      for (int e = 0; e < 8; ++e) s[k][e] = (uint16_t)(v[e >> 1] >> (16 * (e & 1)));
    }
  }
  if (t0 == 0) {  // the conv state after the sequence (nobody else reads or writes it)
    uint16_t n[3][8];
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      const int t = a.T - 3 + k;
      const u32x4 v = *(const u32x4*)(raw + (size_t)(t < 0 ? 0 : t) * a.ld);
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const uint16_t keep = a.T + k < 3 ? s[a.T == 1 ? (k + 1 > 2 ? 2 : k + 1) : 2][e] : (uint16_t)0;
        n[k][e] = t < 0 ? keep : (uint16_t)(v[e >> 1] >> (16 * (e & 1)));
      }
    }
    u32x4 o[3] = {};
#pragma unroll
    for (int e = 0; e < 8; ++e)
#pragma unroll
      for (int k = 0; k < 3; ++k) o[(3 * e + k) >> 3][((3 * e + k) & 7) >> 1] |= (uint32_t)n[k][e] << (16 * ((3 * e + k) & 1));
#pragma unroll
    for (int i = 0; i < 3; ++i) cs[i] = o[i];
  }
  const bool is_x = ch < a.DI;  // (DI is a multiple of 8)
  uint16_t* out = is_x ? a.x_out + row0 * a.DI + ch : a.bc_out + row0 * (a.C - a.DI) + (ch - a.DI);
  const int ld_out = is_x ? a.DI : a.C - a.DI;
  // four tokens at a time, the next four on their way (tc is a multiple of four; clamped past the end)
  constexpr int U = 4;
  u32x4 cur[U], nx[U];
  auto load = [&](u32x4 (&v)[U], int t) {
#pragma unroll
    for (int u = 0; u < U; ++u) v[u] = *(const u32x4*)(raw + (size_t)(t + u < t1 ? t + u : t1 - 1) * a.ld);
  };
  load(nx, t0);
  for (int t = t0; t < t1; t += U) {
#pragma unroll
    for (int u = 0; u < U; ++u) cur[u] = nx[u];
    load(nx, t + U);
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const u32x4 v = cur[u];
      u32x4 o = {0u, 0u, 0u, 0u};
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const uint16_t xo = (uint16_t)(v[e >> 1] >> (16 * (e & 1)));
        const uint32_t w01 = wr[e >> 1][2 * (e & 1)], w23 = wr[e >> 1][2 * (e & 1) + 1];
        float f = h2f(s[0][e]) * h2f((uint16_t)w01);
        f = f + h2f(s[1][e]) * h2f((uint16_t)(w01 >> 16));
        f = f + h2f(s[2][e]) * h2f((uint16_t)w23);
        f = f + h2f(xo) * h2f((uint16_t)(w23 >> 16));
        f = f + h2f((uint16_t)(br[e >> 1] >> (16 * (e & 1))));
        const float sig = dev_sigmoid(f);
        o[e >> 1] |= (uint32_t)f2h(f * sig) << (16 * (e & 1));
        s[0][e] = s[1][e];
        s[1][e] = s[2][e];
        s[2][e] = xo;
      }
      if (t + u < t1) *(u32x4*)(out + (size_t)(t + u) * ld_out) = o;
    }
  }
}

// ------------------------------------------------------------------------------------------
// ssm_scan_kernel<W, RB>: RB 16-row blocks of one head per workgroup, W waves per block.
//
// What bounds it is VALU issue: a state element takes four instructions per token (x dt B, the fma
// of the state, the widening of h and the fp64 fma of the readout), and everything else is kept
// off the elements. Lane (g, r) = (lane / 16, lane % 16) of a wave holds row r of the block and
// 32 / W of its 128 state columns; the four lane groups (and the W waves) hold the others. So
// * B and C are the same for the 16 lanes of a group: each lane reads one pair of columns per token
//   from LDS (widened while staging) and the multiply and the fp64 fma take the other lanes' pairs
//   as DPP row broadcasts, at no cost;
// * one row sum per token and lane crosses lanes, and the sums of four tokens together: the lane
//   swaps of gfx950 exchange two tokens' values between lane groups (reduce4), after which lane
//   group g holds token t + g's sums, so the readout, the gate and the store run once per four
//   tokens on full waves.
// Measured per layer, against the map this replaces (ssm_kernel's own, two rows and four columns per
// lane, whose reductions took two thirds of the instructions and which kept a head on one CU):
// 4796 -> 1449 us at the 2.7B shape and 64 x 256 tokens (1.07 ms if the four instructions per
// element issued back to back; a wave-token takes 680 clocks of its SIMD for about 165 instructions),
// 916 -> 147 us at the 1.3B shape and 1 x 999 tokens, 32.6 -> 8.4 us at 1 x 32 (W = 8).
//
// The readout's sum is ssm_kernel's tree: quads A_j of four columns summed in order from zero (the
// product C h is exact in fp64, so an fma rounds as its multiply-then-add), Q_i = (A_4i + A_4i+1) +
// (A_4i+2 + A_4i+3), then ((Q0 + Q3) + (Q2 + Q1)) + ((Q4 + Q7) + (Q6 + Q5)). The columns are dealt
// out so that the tree's levels are, from the inside: the lane, the lane groups 16 lanes apart, 32
// lanes apart, the waves:
//   W = 1: group g holds Q_2g and Q_(2g ^ 3);
//   W = 2: wave w holds Q_4w .. Q_4w+3, group g Q_4w + (-g mod 4);
//   W = 4: wave w holds Q_2w (groups 0, 1: its halves) and Q_(2w ^ 3) (groups 2, 3);
//   W = 8: wave w holds Q_w, group g its quad g.
// More waves per block cost more instructions per element (the per-token work is shared by fewer
// columns) and a partial sum through LDS, but fill the chip when there are few blocks
// (launch_ssm_scan).
//
// Rounds of TT tokens are staged in LDS, double-buffered, their operands loaded one round ahead.
// ------------------------------------------------------------------------------------------
constexpr int scan_tt(int W) { return W <= 2 ? 8 : 16; }  // tokens per round

template <int W, int RB>
struct ScanBuf {
  static constexpr int TT = scan_tt(W);
  float bf[TT][128];       // B of each token, widened
  double cd[TT][128];      // C of each token, widened
  float X[TT][16 * RB];    // x dt of the workgroup's rows
  float abar[TT];          // exp(dt A)
  double part[W > 1 ? W : 1][W > 1 ? TT : 1][16 * RB];  // the waves' row sums
};

// Raw operands of one round, loaded into registers one round ahead. A thread's items are the
// (token, row) pairs it finishes: W = 1: its lane's row and tokens 4 k + g; W > 1: one item per
// thread, token tid / (16 RB), row tid % (16 RB).
template <int W, int RB>
struct ScanRaw {
  static constexpr int NT = 64 * W * RB, TT = scan_tt(W);
  static constexpr int NI = W == 1 ? TT / 4 : 1;      // items per thread (W = 8: of the first half)
  static constexpr int NB = TT * 32 / NT;             // 16-byte vectors of B | C per thread
  static_assert(NB * NT == TT * 32 && (W == 8 ? 2 : 1) * TT * 16 * RB == NI * NT, "whole vectors and items");
  u32x4 bc[NB];
  uint16_t x[NI], z[NI];
  float dt[NI];
  float abar;  // token tid % TT
};

template <int W, int RB>
__device__ __forceinline__ int scan_item_token(int k) {
  return W == 1 ? 4 * k + (((int)threadIdx.x & 63) >> 4) : (int)threadIdx.x / (16 * RB) % scan_tt(W);
}
template <int W, int RB>
__device__ __forceinline__ int scan_item_row() {
  return W == 1 ? 16 * ((int)threadIdx.x >> 6) + ((int)threadIdx.x & 15) : (int)threadIdx.x % (16 * RB);
}
// Vector i of a round's B | C: token and 8-column block of B (below 16) or C; the order keeps a
// wave's vectors all B or all C
template <int TT>
__device__ __forceinline__ void scan_bc_pos(int i, int& t, int& c) {
  t = (i % (16 * TT)) / 16;
  c = (i / (16 * TT)) * 16 + i % 16;
}

template <int W, int RB>
__device__ __forceinline__ ScanRaw<W, RB> scan_load(const ScanArgs& a, int b, int head, int col0, int t0) {
  using Raw = ScanRaw<W, RB>;
  const int tid = threadIdx.x;
  Raw r;
  // clamped token indices: tokens past the end re-read the last one (never consumed). 32-bit element
  // offsets: at most 32768 rows of under 32768 elements.
  auto row = [&](int t) { return (uint32_t)(b * a.T + (t < a.T ? t : a.T - 1)); };
#pragma unroll
  for (int k = 0; k < Raw::NB; ++k) {
    int t, c;
    scan_bc_pos<Raw::TT>(tid + Raw::NT * k, t, c);
    r.bc[k] = *(const u32x4*)(a.bc + (row(t0 + t) * 256u + 8u * c));
  }
  const uint32_t col = col0 + scan_item_row<W, RB>();
#pragma unroll
  for (int k = 0; k < Raw::NI; ++k) {
    const uint32_t m = row(t0 + scan_item_token<W, RB>(k));
    r.x[k] = a.xg[m * (uint32_t)(a.H * a.P) + col];
    r.z[k] = a.z[m * (uint32_t)a.ld_z + col];
    r.dt[k] = a.dec[m * (uint32_t)a.H + head].x;
  }
  r.abar = a.dec[row(t0 + tid % Raw::TT) * (uint32_t)a.H + head].y;
  return r;
}

template <int W, int RB>
__device__ __forceinline__ void scan_stage(ScanBuf<W, RB>& S, const ScanRaw<W, RB>& r) {
  using Raw = ScanRaw<W, RB>;
  const int tid = threadIdx.x;
#pragma unroll
  for (int k = 0; k < Raw::NB; ++k) {
    int t, c;
    scan_bc_pos<Raw::TT>(tid + Raw::NT * k, t, c);
    float f[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) f[e] = h2f((uint16_t)(r.bc[k][e >> 1] >> (16 * (e & 1))));
    if (c < 16) {
      *(f32x4*)&S.bf[t][8 * c] = f32x4{f[0], f[1], f[2], f[3]};
      *(f32x4*)&S.bf[t][8 * c + 4] = f32x4{f[4], f[5], f[6], f[7]};
    } else {
      double* d = &S.cd[t][8 * (c - 16)];
#pragma unroll
      for (int e = 0; e < 8; ++e) d[e] = (double)f[e];
    }
  }
  if (W < 8 || tid < Raw::NT / 2) {
#pragma unroll
    for (int k = 0; k < Raw::NI; ++k) S.X[scan_item_token<W, RB>(k)][scan_item_row<W, RB>()] = h2f(r.x[k]) * r.dt[k];
  }
  if (tid < Raw::TT) S.abar[tid] = r.abar;
}

// Quads 2 I and 2 I + 1 of one token: the state updates (in place) and the quads' fp64 sums. b0, b1 /
// c0, c1: this lane's pair of columns of B / C; lanes 4 I .. 4 I + 3 of its row hold the eight columns.
// In asm because the fp64 fma with a row broadcast has no builtin, and so that the state stays in its
// registers. The first two instructions write none of the registers the DPP reads come from, which
// covers the two wait states between a VALU write and a DPP read, whatever precedes the block; two
// independent chains throughout.
template <int I>
__device__ __forceinline__ void scan_quads(float* h, float abar, float X, float b0, float b1, double c0, double c1,
                                           double& s0, double& s1) {
  float t0, t1, t2, t3;
  double d0, d1, d2, d3;
#define DFSSM_ROW(n) " row_newbcast:" n " row_mask:0xf bank_mask:0xf\n\t"
  asm("v_mov_b64 %0, 0\n\t"
      "v_mov_b64 %1, 0\n\t"
      "v_mul_f32_dpp %10, %20, %19" DFSSM_ROW("%24")
      "v_mul_f32_dpp %11, %20, %19" DFSSM_ROW("%26")
      "v_mul_f32_dpp %12, %21, %19" DFSSM_ROW("%24")
      "v_mul_f32_dpp %13, %21, %19" DFSSM_ROW("%26")
      "v_fma_f32 %2, %18, %2, %10\n\t"
      "v_fma_f32 %6, %18, %6, %11\n\t"
      "v_fma_f32 %3, %18, %3, %12\n\t"
      "v_fma_f32 %7, %18, %7, %13\n\t"
      "v_cvt_f64_f32 %14, %2\n\t"
      "v_cvt_f64_f32 %15, %6\n\t"
      "v_cvt_f64_f32 %16, %3\n\t"
      "v_cvt_f64_f32 %17, %7\n\t"
      "v_mul_f32_dpp %10, %20, %19" DFSSM_ROW("%25")
      "v_mul_f32_dpp %11, %20, %19" DFSSM_ROW("%27")
      "v_fmac_f64_dpp %0, %22, %14" DFSSM_ROW("%24")
      "v_fmac_f64_dpp %1, %22, %15" DFSSM_ROW("%26")
      "v_mul_f32_dpp %12, %21, %19" DFSSM_ROW("%25")
      "v_mul_f32_dpp %13, %21, %19" DFSSM_ROW("%27")
      "v_fma_f32 %4, %18, %4, %10\n\t"
      "v_fma_f32 %8, %18, %8, %11\n\t"
      "v_fmac_f64_dpp %0, %23, %16" DFSSM_ROW("%24")
      "v_fmac_f64_dpp %1, %23, %17" DFSSM_ROW("%26")
      "v_fma_f32 %5, %18, %5, %12\n\t"
      "v_fma_f32 %9, %18, %9, %13\n\t"
      "v_cvt_f64_f32 %14, %4\n\t"
      "v_cvt_f64_f32 %15, %8\n\t"
      "v_cvt_f64_f32 %16, %5\n\t"
      "v_cvt_f64_f32 %17, %9\n\t"
      "v_fmac_f64_dpp %0, %22, %14" DFSSM_ROW("%25")
      "v_fmac_f64_dpp %1, %22, %15" DFSSM_ROW("%27")
      "v_fmac_f64_dpp %0, %23, %16" DFSSM_ROW("%25")
      "v_fmac_f64_dpp %1, %23, %17" DFSSM_ROW("%27")
      : "=&v"(s0), "=&v"(s1), "+v"(h[0]), "+v"(h[1]), "+v"(h[2]), "+v"(h[3]), "+v"(h[4]), "+v"(h[5]), "+v"(h[6]),
        "+v"(h[7]), "=&v"(t0), "=&v"(t1), "=&v"(t2), "=&v"(t3), "=&v"(d0), "=&v"(d1), "=&v"(d2), "=&v"(d3)
      : "v"(abar), "v"(X), "v"(b0), "v"(b1), "v"(c0), "v"(c1), "n"(4 * I), "n"(4 * I + 1), "n"(4 * I + 2), "n"(4 * I + 3));
#undef DFSSM_ROW
}

// One quad (W = 8): columns in lanes 0 and 1 of the row.
__device__ __forceinline__ void scan_quad(float* h, float abar, float X, float b0, float b1, double c0, double c1, double& s0) {
  float t0, t1, t2, t3;
  double d0, d1, d2, d3;
#define DFSSM_ROW(n) " row_newbcast:" n " row_mask:0xf bank_mask:0xf\n\t"
  asm("v_mov_b64 %0, 0\n\t"
      "s_nop 0\n\t"
      "v_mul_f32_dpp %5, %15, %14" DFSSM_ROW("0")
      "v_mul_f32_dpp %6, %16, %14" DFSSM_ROW("0")
      "v_mul_f32_dpp %7, %15, %14" DFSSM_ROW("1")
      "v_mul_f32_dpp %8, %16, %14" DFSSM_ROW("1")
      "v_fma_f32 %1, %13, %1, %5\n\t"
      "v_fma_f32 %2, %13, %2, %6\n\t"
      "v_fma_f32 %3, %13, %3, %7\n\t"
      "v_fma_f32 %4, %13, %4, %8\n\t"
      "v_cvt_f64_f32 %9, %1\n\t"
      "v_cvt_f64_f32 %10, %2\n\t"
      "v_cvt_f64_f32 %11, %3\n\t"
      "v_cvt_f64_f32 %12, %4\n\t"
      "v_fmac_f64_dpp %0, %17, %9" DFSSM_ROW("0")
      "v_fmac_f64_dpp %0, %18, %10" DFSSM_ROW("0")
      "v_fmac_f64_dpp %0, %17, %11" DFSSM_ROW("1")
      "v_fmac_f64_dpp %0, %18, %12" DFSSM_ROW("1")
      : "=&v"(s0), "+v"(h[0]), "+v"(h[1]), "+v"(h[2]), "+v"(h[3]), "=&v"(t0), "=&v"(t1), "=&v"(t2), "=&v"(t3),
        "=&v"(d0), "=&v"(d1), "=&v"(d2), "=&v"(d3)
      : "v"(abar), "v"(X), "v"(b0), "v"(b1), "v"(c0), "v"(c1));
#undef DFSSM_ROW
}

// The lane swaps on fp64 values: a's odd 16-lane rows change places with b's even ones; a's upper
// 32 lanes with b's lower ones.
__device__ __forceinline__ void swap16_f64(double& a, double& b) {
  const uint64_t u = __builtin_bit_cast(uint64_t, a), v = __builtin_bit_cast(uint64_t, b);
  const auto lo = __builtin_amdgcn_permlane16_swap((uint32_t)u, (uint32_t)v, false, false);
  const auto hi = __builtin_amdgcn_permlane16_swap((uint32_t)(u >> 32), (uint32_t)(v >> 32), false, false);
  a = __builtin_bit_cast(double, ((uint64_t)hi[0] << 32) | lo[0]);
  b = __builtin_bit_cast(double, ((uint64_t)hi[1] << 32) | lo[1]);
}
__device__ __forceinline__ void swap32_f64(double& a, double& b) {
  const uint64_t u = __builtin_bit_cast(uint64_t, a), v = __builtin_bit_cast(uint64_t, b);
  const auto lo = __builtin_amdgcn_permlane32_swap((uint32_t)u, (uint32_t)v, false, false);
  const auto hi = __builtin_amdgcn_permlane32_swap((uint32_t)(u >> 32), (uint32_t)(v >> 32), false, false);
  a = __builtin_bit_cast(double, ((uint64_t)hi[0] << 32) | lo[0]);
  b = __builtin_bit_cast(double, ((uint64_t)hi[1] << 32) | lo[1]);
}
// Lane group g's result: (v_g of group 0 + of group 1) + (of group 2 + of group 3), row by row.
__device__ __forceinline__ double reduce4(double v0, double v1, double v2, double v3) {
  swap16_f64(v0, v1);
  swap16_f64(v2, v3);
  double a = v0 + v1, b = v2 + v3;
  swap32_f64(a, b);
  return a + b;
}

template <int W, int RB>
__global__ __launch_bounds__(64 * W * RB, 4) void ssm_scan_kernel(ScanArgs a) {
  using Buf = ScanBuf<W, RB>;
  using Raw = ScanRaw<W, RB>;
  constexpr int TT = Buf::TT, NQ = 8 / W;  // tokens per round; quads per lane
  __shared__ Buf buf[2];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int blk = wave / W, w = wave % W;  // 16-row block within the workgroup; wave of the block
  const int g = lane >> 4, r = lane & 15;
  const int b = blockIdx.y;
  const int wg_per_head = a.P / (16 * RB);
  const int head = (int)blockIdx.x / wg_per_head;
  const int p0 = ((int)blockIdx.x % wg_per_head) * (16 * RB);  // first row of the workgroup in the head
  const int col0 = head * a.P + p0;
  const int rl = 16 * blk + r;
  const float Dh = a.D[head];
  // this lane's columns: quads 4 q .. of Qa and Qb, and its pair of columns for the broadcasts
  const int Qa = W == 1 ? 2 * g : W == 2 ? 4 * w + ((4 - g) & 3) : W == 4 ? (g < 2 ? 2 * w : (2 * w) ^ 3) : w;
  const int Qb = W == 1 ? Qa ^ 3 : Qa;
  const int part = W == 4 ? 8 * (g & 1) : W == 8 ? 4 * g : 0;  // first column within Qa
  const int pair = W == 1 && r >= 8 ? 8 * Qb + r - 8 : 8 * Qa + part / 2 + (r & (W <= 2 ? 7 : W == 4 ? 3 : 1));

  Raw raw = scan_load<W, RB>(a, b, head, col0, 0);
  float* hp = a.h + (((size_t)b * a.H + head) * a.P + p0 + rl) * a.N;
  float h[4 * NQ];
#pragma unroll
  for (int q = 0; q < NQ; ++q) {
    const f32x4 v = ld_nt_f4(hp + 16 * (q < 4 ? Qa : Qb) + part + 4 * (q & 3));
    h[4 * q] = v.x; h[4 * q + 1] = v.y; h[4 * q + 2] = v.z; h[4 * q + 3] = v.w;
  }
  scan_stage<W, RB>(buf[0], raw);
  lds_barrier();

  const int rounds = (a.T + TT - 1) / TT;
  for (int rd = 0; rd < rounds; ++rd) {
    const int t0 = rd * TT;
    Buf& S = buf[rd & 1];
    // this round's items, kept for the gate, and the next round's operands on their way (past the
    // last round a re-read that nobody consumes: a branch would make the loads' users wait)
    const Raw cur = raw;
    raw = scan_load<W, RB>(a, b, head, col0, t0 + TT);
    const int nt = a.T - t0 < TT ? a.T - t0 : TT;
    auto finish = [&](double s, int k) {  // item k of this thread from its row's readout
      const int t = scan_item_token<W, RB>(k);
      const float z = h2f(cur.z[k]);
      const float sz = r16(z * r16(dev_sigmoid(z)));
      const float y = r16((float)s + h2f(cur.x[k]) * Dh);
      if (t < nt) a.xg[((size_t)b * a.T + t0 + t) * (a.H * a.P) + col0 + scan_item_row<W, RB>()] = f2h(y * sz);
    };
#pragma unroll
    for (int k = 0; k < TT / 4; ++k) {
      if (4 * k >= nt) break;
      double acc[4];
      auto tokens = [&](auto full_t) {  // FULL: all four tokens exist (all but a prompt's last ones)
        constexpr bool FULL = decltype(full_t)::value;
        // W > 1: few waves per SIMD, so the four tokens' operands are read before the first is used
        constexpr int PF = W > 1 && FULL ? 4 : 1;
        float2 bp[PF];
        double c0[PF], c1[PF];
        float X[PF], abar[PF];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          if (j % PF == 0) {
#pragma unroll
            for (int u = 0; u < PF; ++u) {
              const int t = 4 * k + j + u;
              bp[u] = *(const float2*)&S.bf[t][2 * pair];
              c0[u] = S.cd[t][2 * pair];
              c1[u] = S.cd[t][2 * pair + 1];
              X[u] = S.X[t][rl];
              abar[u] = S.abar[t];
            }
            if (PF > 1) __builtin_amdgcn_sched_barrier(0);
          }
          acc[j] = 0.0;
          if (!FULL && 4 * k + j >= nt) continue;  // uniform: past the prompt's end
          const int u = j % PF;
          double A[NQ], q;
          if constexpr (NQ == 1) {
            scan_quad(h, abar[u], X[u], bp[u].x, bp[u].y, c0[u], c1[u], q);
          } else {
            scan_quads<0>(h, abar[u], X[u], bp[u].x, bp[u].y, c0[u], c1[u], A[0], A[1]);
            q = A[0] + A[1];
          }
          if constexpr (NQ > 2) {
            scan_quads<1>(h + 8, abar[u], X[u], bp[u].x, bp[u].y, c0[u], c1[u], A[2], A[3]);
            q = q + (A[2] + A[3]);
          }
          if constexpr (NQ > 4) {
            scan_quads<2>(h + 16, abar[u], X[u], bp[u].x, bp[u].y, c0[u], c1[u], A[4], A[5]);
            scan_quads<3>(h + 24, abar[u], X[u], bp[u].x, bp[u].y, c0[u], c1[u], A[6], A[7]);
            q = q + ((A[4] + A[5]) + (A[6] + A[7]));
          }
          acc[j] = q;
        }
      };
      if (W > 1 && 4 * k + 4 <= nt) tokens(std::true_type{});
      else tokens(std::false_type{});
      const double s = reduce4(acc[0], acc[1], acc[2], acc[3]);
      if constexpr (W == 1) finish(s, k);
      else S.part[w][4 * k + g][rl] = s;
    }
    scan_stage<W, RB>(buf[(rd + 1) & 1], raw);
    lds_barrier();
    if constexpr (W > 1) {
      // (the partials of a buffer are rewritten two rounds later, after the next round's barrier)
      const int t = scan_item_token<W, RB>(0), i = scan_item_row<W, RB>();
      double s;
      if constexpr (W == 8)
        s = ((S.part[0][t][i] + S.part[3][t][i]) + (S.part[2][t][i] + S.part[1][t][i])) +
            ((S.part[4][t][i] + S.part[7][t][i]) + (S.part[6][t][i] + S.part[5][t][i]));
      else
        s = S.part[0][t][i] + S.part[1][t][i];
      if constexpr (W == 4) s = s + (S.part[2][t][i] + S.part[3][t][i]);
      if (W < 8 || tid < Raw::NT / 2) finish(s, 0);
    }
  }
#pragma unroll
  for (int q = 0; q < NQ; ++q)
    st_nt_f4(hp + 16 * (q < 4 ? Qa : Qb) + part + 4 * (q & 3), f32x4{h[4 * q], h[4 * q + 1], h[4 * q + 2], h[4 * q + 3]});
}

// dst[b] = src[b * T + T - 1]: the last token's row of every sequence.
__global__ __launch_bounds__(256) void last_rows_kernel(const uint16_t* __restrict__ src, uint16_t* __restrict__ dst,
                                                        int T, int D) {
  const int b = blockIdx.x;
  const uint16_t* s = src + ((size_t)b * T + T - 1) * D;
  for (int k = threadIdx.x; k < D; k += 256) dst[(size_t)b * D + k] = s[k];
}

hipError_t launch_conv_tokens(const ConvTokArgs& args, int batch, hipStream_t s) {
  ConvTokArgs a = args;
  if (a.T < 1 || batch < 1 || a.C % 8 || a.DI % 8 || a.ld % 8) return hipErrorInvalidValue;
  // tokens per thread: 16 (the three re-read rows then cost 3/16 more) while that leaves 64 Ki
  // threads (one wave per SIMD), else fewer, but
  // at least the three tokens before any later range (only the first reads the conv state, which it writes)
  a.tc = 16;
  while (a.tc > 4 && (long long)batch * ((a.T + a.tc - 1) / a.tc) * (a.C / 8) < (1 << 16)) a.tc /= 2;
  const dim3 g((a.C / 8 + 255) / 256 + 1, (a.T + a.tc - 1) / a.tc, batch);
  hipLaunchKernelGGL(conv_tokens_kernel, g, dim3(256), 0, s, a);
  return hipGetLastError();
}

hipError_t launch_ssm_scan(const ScanArgs& a, int batch, hipStream_t s) {
  if (a.T < 1 || a.P % 16 || a.N != 128) return hipErrorInvalidValue;
  // Waves per 16-row block: one where the head has the blocks for a workgroup of four waves and there
  // are enough of them, more where the chip would be idle. Microseconds per 128 tokens with 1 / 2 / 4 / 8
  // waves at the 1.3B shape (256 blocks per sequence): 1 sequence 59 / 35 / 24.6 / 22.4, 2: 60 / 36.7 /
  // 36.0 / 42.3, 4: 63 / 53 / 63 / 79, 12: 134 / 129 / 170 / 227, 16: 170 / 166 / 224 / 303, 64: 589 / 608 /
  // 876 / 1213.
  const int blocks = a.P / 16;
  const long long n = (long long)batch * a.H * blocks;
  if (blocks % 4 == 0 && n >= 4096)
    hipLaunchKernelGGL((ssm_scan_kernel<1, 4>), dim3(a.H * (blocks / 4), batch), dim3(256), 0, s, a);
  else if (blocks % 2 == 0 && n >= 1024)
    hipLaunchKernelGGL((ssm_scan_kernel<2, 2>), dim3(a.H * (blocks / 2), batch), dim3(256), 0, s, a);
  else if (n > 256)
    hipLaunchKernelGGL((ssm_scan_kernel<4, 1>), dim3(a.H * blocks, batch), dim3(256), 0, s, a);
  else
    hipLaunchKernelGGL((ssm_scan_kernel<8, 1>), dim3(a.H * blocks, batch), dim3(512), 0, s, a);
  return hipGetLastError();
}

hipError_t launch_last_rows(const uint16_t* src, uint16_t* dst, int batch, int T, int D, hipStream_t s) {
  hipLaunchKernelGGL(last_rows_kernel, dim3(batch), dim3(256), 0, s, src, dst, T, D);
  return hipGetLastError();
}

}  // namespace dfssm
