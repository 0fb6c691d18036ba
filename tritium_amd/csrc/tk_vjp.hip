// TernaryBackend::mpgemm_projected_vjp on the device (crates/tritium-spec/src/lib.rs:93-117, 217-232):
// the three gradients of one packed ternary mpGEMM, each output element summed by one thread in the
// index order and with the unfused f32 operations of the CPU backend's scalar path
// (crates/tritium-cpu/src/kernel.rs:150-189, 281-317), so the results carry its bits.
//
//   grad_act[m,k] = sum_n upstream[m,n] * (trit[n,k] * scales[n])     n = 0, 1, ...
//   grad_w[n,k]   = sum_m upstream[m,n] * act[m,k]                    m = 0, 1, ...
//   grad_bias[n]  = sum_m upstream[m,n]                               m = 0, 1, ...
//
// Weights are read in the device layout of the forward kernels: the 1-KiB chunk of row tile t and K
// block kb holds, for lane group g = 0..3 and row r = 0..15, the 16 code bytes g*16 .. g*16+15 of that
// row's block at offset g*256 + r*16; byte i of a block holds the elements (i/32)*128 + s*32 + i%32 at
// bit pairs s = 0..3, code = trit + 1.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "tk_internal.h"

#define TKV_GLOBAL __attribute__((address_space(1)))

namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ float ldg(const float *p) { return *(const TKV_GLOBAL float *)p; }
__device__ __forceinline__ f32x4 ldg4(const float *p) { return *(const TKV_GLOBAL f32x4 *)p; }

// XCD-aware order of `total` workgroups: workgroups are dealt to the eight XCDs in turn, so XCD x takes the
// x-th eighth of the index range and its L2 holds one compact part of the operands. Grids are 8 * ceil(total / 8).
__device__ __forceinline__ unsigned xcd_index(unsigned bid, unsigned total) {
  return (bid & 7u) * ((total + 7u) >> 3) + (bid >> 3);
}

// ---- grad_act ----
// The term upstream * (trit * scale) is p * trit with p = upstream * scale rounded once: a trit only negates
// or clears the product. A product with -1, 0 or 1 is exact, so ONE fused multiply-add per term rounds exactly
// as the CPU's separate multiply and add -- and the f32 matrix instructions are chains of such fused multiply-adds:
// v_mfma_f32_16x16x4_f32 adds its four terms in ascending order with one rounding each, denormals kept (compared with
// fmaf chains bit for bit on the device). So the contraction runs on the matrix pipe in the CPU's order.
// Infinities and NaN in the upstream gradient or the scales come out the same either way (an infinite or NaN p times a zero trit is
// NaN, as the CPU's upstream * (0 * scale) is). The one case where p * trit differs from the CPU's term is p overflowing to infinity
// from finite factors under a zero trit (NaN instead of 0). Such a sum can only end as NaN or infinity, so a workgroup whose
// sums do not all end finite looks for such a product among its tokens, and only where it finds one repeats its sums as the
// CPU computes them. M=2048 N=6912 K=2560, all values finite 0.64 ms; an infinity in one token 0.75, NaN in all 0.89; such a
// product in one token 1.8, in all 3.3 (each lane repeating its own sums of a wave: 15.9, 29.5, 16.0, 29.6).
//
// A workgroup owns 16*TT tokens x the 64 columns of one bit pair of a K block; wave g takes piece g of the chunks, of which
// four rows are the 64 contiguous bytes of one wave-wide load, and every decoded operand serves TT matrix instructions.
// The products p of 64 weight rows pass through LDS (two buffers, one barrier per 64 rows); codes and upstream
// values of the next 64 rows are requested before the current ones are used.
// Bound: the f32 matrix pipe (151 TFLOP/s sustained on the device, 157 published). It shares its multipliers with the vector
// ALU, so whatever vector work is left (decoding, the products) adds to its time.
// M=2048 N=6912 K=2560: 0.64 ms = 113 TFLOP/s (2.9 ms as multiply and add per term on the vector ALU); M=64 N=2560
// K=2560: 31 us (1.06 ms).
constexpr int ACT_ROWS = 64;  // weight rows per LDS stage

// The sums of a workgroup term by term: upstream * (trit * scale) and the sum, each rounded. 64 weight rows of upstream values and
// their scales pass through LDS as in the kernel below, whose accumulators this overwrites.
template <int TT>
__device__ __forceinline__ void act_repeat(const uint8_t *__restrict__ codes, int nb, int n, int n_tiles, int kb, int pair,
                                        const float *__restrict__ scales, const float *__restrict__ up_base, int last_token,
                                        float (*s_up)[ACT_ROWS + 4], float *s_sc, f32x4 (&acc)[TT]) {
  int tid = threadIdx.x;
  asm("" : "+v"(tid));  // (what follows is derived anew: the main loop's registers set the occupancy)
  const int g = tid >> 6, lane = tid & 63, c = lane & 15, h = lane >> 4;
#pragma unroll
  for (int t = 0; t < TT; ++t) acc[t] = (f32x4){0.0f, 0.0f, 0.0f, 0.0f};
  for (int r0 = 0; r0 < n; r0 += ACT_ROWS) {
    __syncthreads();
    const int row = r0 + (tid & 63);
    const bool in = row < n;  // rows past the end: 0 * (trit * 0) = +-0 changes nothing
#pragma unroll 8
    for (int i = 0; i < 4 * TT; ++i) {
      const int tok = i * 4 + g;
      s_up[tok][tid & 63] = in ? ldg(up_base + (unsigned)(min(tok, last_token) * n + row)) : 0.0f;
    }
    if (tid < ACT_ROWS) s_sc[tid] = in ? ldg(scales + row) : 0.0f;
    __syncthreads();
    uint32_t w[4];
    auto request = [&](int q) {
      const uint8_t *cp = codes + ((size_t)min((r0 + q) >> 4, n_tiles - 1) * nb + kb) * 1024 + g * 256 + (q & 15) * 16 + c;
#pragma unroll
      for (int x = 0; x < 4; ++x) w[x] = *(const TKV_GLOBAL uint8_t *)(cp + x * 16);
    };
    request(0);
#pragma unroll 1
    for (int q = 0; q < ACT_ROWS; q += 4) {
      const f32x4 sc = *(const f32x4 *)&s_sc[q];
      float proj[4];
#pragma unroll
      for (int x = 0; x < 4; ++x) proj[x] = __fmul_rn((float)((w[x] >> (2 * pair)) & 3u) - 1.0f, sc[x]);
      request(min(q + 4, ACT_ROWS - 4));
#pragma unroll
      for (int t = 0; t < TT; ++t) {
        f32x4 up[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) up[r] = *(const f32x4 *)&s_up[16 * t + h * 4 + r][q];
#pragma unroll
        for (int x = 0; x < 4; ++x)
#pragma unroll
          for (int r = 0; r < 4; ++r) acc[t][r] = __fadd_rn(acc[t][r], __fmul_rn(up[r][x], proj[x]));
        if (t & 1) __builtin_amdgcn_sched_barrier(0);  // (few registers: the kernel's occupancy is that of its main loop)
      }
    }
  }
}

template <int TT>
__global__ __launch_bounds__(256) void tk_vjp_act_kernel(const uint8_t *__restrict__ codes, int nb, int n, int k, int m,
                                                         const float *__restrict__ scales,
                                                         const float *__restrict__ grad_output,
                                                         float *__restrict__ grad_act, int wide) {
  __shared__ float s_p[2][16 * TT][ACT_ROWS + 4];  // [buffer][token][row]; the stride keeps a wave's reads on 64 banks
  __shared__ int s_bad[2];  // a sum is not finite; a product of finite factors is not
  const unsigned cols = (unsigned)nb * 4, total = cols * (unsigned)((m + 16 * TT - 1) / (16 * TT));
  const unsigned idx = xcd_index(blockIdx.x, total);
  if (idx >= total) return;
  const int m0 = (int)(idx / cols) * (16 * TT), kb = (int)(idx % cols) >> 2, pair = (int)(idx & 3);
  const int tid = threadIdx.x, g = tid >> 6, lane = tid & 63, c = lane & 15, h = lane >> 4;
  const int n_tiles = (n + 15) >> 4, stages = (n + ACT_ROWS - 1) / ACT_ROWS;
  if (tid < 2) s_bad[tid] = 0;  // (ordered by the first stage's barrier)
  // staging: a thread takes four rows of UT tokens; addresses are a uniform base per stage and a lane offset, which
  // costs the vector ALU nothing (it shares its lanes with the f32 matrix pipe: their times add up)
  constexpr int QUADS = ACT_ROWS / 4, TPR = 256 / QUADS, UT = 16 * TT / TPR;
  const int ti = tid / QUADS, q = tid % QUADS * 4;
  const float *up_base = grad_output + (size_t)m0 * n;
  unsigned up_off[UT];
#pragma unroll
  for (int t = 0; t < UT; ++t) up_off[t] = (unsigned)(min(ti + TPR * t, m - 1 - m0) * n + q);  // (past the end: not stored)
  const unsigned code_off = (unsigned)(kb * 1024 + g * 256 + lane);

  f32x4 u[UT], sc;
  uint32_t w[ACT_ROWS / 4];
  auto request = [&](int st) {
    const int r = st * ACT_ROWS;
    const float *ub = up_base + r, *sb = scales + r;
    if (wide && r + ACT_ROWS <= n) {  // (uniform)
#pragma unroll
      for (int t = 0; t < UT; ++t) u[t] = ldg4(ub + up_off[t]);
      sc = ldg4(sb + (unsigned)q);
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const bool in = r + q + e < n;
#pragma unroll
        for (int t = 0; t < UT; ++t) u[t][e] = in ? ldg(ub + (up_off[t] + e)) : 0.0f;
        sc[e] = in ? ldg(sb + (unsigned)(q + e)) : 0.0f;  // rows past the end: p = 0, and adding +-0 changes nothing
      }
    }
#pragma unroll
    for (int t = 0; t < ACT_ROWS / 16; ++t) {
      const uint8_t *cp = codes + (size_t)min(st * (ACT_ROWS / 16) + t, n_tiles - 1) * nb * 1024;
#pragma unroll
      for (int x = 0; x < 4; ++x) w[t * 4 + x] = *(const TKV_GLOBAL uint8_t *)(cp + (code_off + x * 64));
    }
  };
  f32x4 acc[TT];
#pragma unroll
  for (int t = 0; t < TT; ++t) acc[t] = (f32x4){0.0f, 0.0f, 0.0f, 0.0f};
  request(0);
  for (int st = 0; st < stages; ++st) {
    float(*buf)[ACT_ROWS + 4] = s_p[st & 1];
#pragma unroll
    for (int t = 0; t < UT; ++t) {
      f32x4 p;
#pragma unroll
      for (int e = 0; e < 4; ++e) p[e] = __fmul_rn(u[t][e], sc[e]);
      *(f32x4 *)&buf[ti + TPR * t][q] = p;
    }
    uint32_t v[ACT_ROWS / 4];
#pragma unroll
    for (int x = 0; x < ACT_ROWS / 4; ++x) v[x] = w[x];
    __syncthreads();
    if (st + 1 < stages) request(st + 1);
#pragma unroll
    for (int x = 0; x < ACT_ROWS / 4; ++x) {
      const float b = (float)((v[x] >> (2 * pair)) & 3u) - 1.0f;
#pragma unroll
      for (int t = 0; t < TT; ++t)
        acc[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(buf[16 * t + c][x * 4 + h], b, acc[t], 0, 0, 0);
    }
  }
  bool finite = true;
#pragma unroll
  for (int t = 0; t < TT; ++t)
#pragma unroll
    for (int r = 0; r < 4; ++r) finite &= fabsf(acc[t][r]) < __builtin_inff();
  if (!finite) s_bad[0] = 1;
  __syncthreads();
  if (s_bad[0]) {
    bool over = false;
    for (int row = tid; row < n; row += 256) {
      const float s = ldg(scales + row);
#pragma unroll 4
      for (int i = 0; i < 16 * TT; ++i) {
        const float up = ldg(up_base + (unsigned)(min(i, m - 1 - m0) * n + row));
        over |= fabsf(__fmul_rn(up, s)) == __builtin_inff() && fabsf(up) < __builtin_inff() && fabsf(s) < __builtin_inff();
      }
    }
    if (over) s_bad[1] = 1;
    __syncthreads();
    if (s_bad[1]) act_repeat<TT>(codes, nb, n, n_tiles, kb, pair, scales, up_base, m - 1 - m0, s_p[0], s_p[1][0], acc);
  }
  // byte c of piece g, bit pair s: element (g/2)*128 + s*32 + (g%2)*16 + c of the K block
  int id = threadIdx.x;
  asm("" : "+v"(id));  // (derived anew: the main loop's registers set the occupancy)
  const int kk = kb * 256 + (id >> 7) * 128 + pair * 32 + ((id >> 6) & 1) * 16 + (id & 15), hh = (id & 63) >> 4;
  if (kk >= k) return;
#pragma unroll
  for (int t = 0; t < TT; ++t)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int mi = m0 + t * 16 + hh * 4 + r;
      if (mi < m) *(TKV_GLOBAL float *)(grad_act + (size_t)mi * k + kk) = acc[t][r];
    }
}

// ---- grad_bias ----
// One thread per column walks the tokens in order, 32 loads in flight per thread.
__device__ __forceinline__ void bias_column(int ni, int n, int m, const float *__restrict__ grad_output,
                                            float *__restrict__ grad_bias) {
  if (ni >= n) return;
  float acc = 0.0f;
  int mi = 0;
  for (; mi + 32 <= m; mi += 32) {
    float v[32];
#pragma unroll
    for (int q = 0; q < 32; ++q) v[q] = ldg(grad_output + (size_t)(mi + q) * n + ni);
#pragma unroll
    for (int q = 0; q < 32; ++q) acc = __fadd_rn(acc, v[q]);
  }
  for (; mi < m; ++mi) acc = __fadd_rn(acc, ldg(grad_output + (size_t)mi * n + ni));
  *(TKV_GLOBAL float *)(grad_bias + ni) = acc;
}

__global__ __launch_bounds__(64) void tk_vjp_bias_kernel(int n, int m, const float *__restrict__ grad_output,
                                                         float *__restrict__ grad_bias) {
  bias_column(blockIdx.x * 64 + threadIdx.x, n, m, grad_output, grad_bias);
}

// ---- grad_w ----
// Here both factors are arbitrary, so a term needs its own rounded product: one multiply and one add on the vector
// ALU (two waves per SIMD issue 69 T lane operations a second on the device; the matrix pipe as the multiplier and the
// vector ALU as the adder measured slower: 22 against 35 T terms). A wave owns TN weight rows x 64*TK columns. Its upstream values are the
// same for every lane: they come through scalar loads and are the multiply's scalar operand, so a token costs a lane one
// load of TK activations for 2*TN*TK operations and nothing passes through LDS (64 x 64 tiles through LDS read two
// 16-byte pieces per 32 operations and were held back by that). Lanes and waves past the end of a row repeat
// the last whole piece: the same values are stored twice.
// The first bias_blocks workgroups sum the columns of grad_bias beside the others (33 us as a launch of its own).
// M=2048 N=6912 K=2560: 1.36 ms with the bias (1.55 + 0.03 ms with 64 x 64 tiles through LDS).
constexpr int W_TOK = 4;  // tokens per step

template <int TN, int TK>
__global__ __launch_bounds__(256) void tk_vjp_weight_kernel(int n, int k, int m, const float *__restrict__ act,
                                                            const float *__restrict__ grad_output,
                                                            float *__restrict__ grad_w, float *__restrict__ grad_bias,
                                                            int bias_blocks) {
  typedef float piece __attribute__((ext_vector_type(TK), aligned(4)));
  if ((int)blockIdx.x < bias_blocks) {
    bias_column(blockIdx.x * 256 + threadIdx.x, n, m, grad_output, grad_bias);
    return;
  }
  const unsigned k_tiles = (unsigned)(k + 64 * TK - 1) / (64 * TK), n_tiles = (unsigned)(n + 4 * TN - 1) / (4 * TN);
  const unsigned idx = xcd_index(blockIdx.x - bias_blocks, k_tiles * n_tiles);
  if (idx >= k_tiles * n_tiles) return;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int nw = (int)(idx / k_tiles) * (4 * TN) + wave * TN;
  if (nw >= n) return;
  const int n0 = min(nw, n - TN), k0 = min((int)(idx % k_tiles) * (64 * TK) + lane * TK, k - TK);
  const float *ap = act + k0, *up = grad_output + n0;
  float acc[TN][TK];
#pragma unroll
  for (int y = 0; y < TN; ++y)
#pragma unroll
    for (int x = 0; x < TK; ++x) acc[y][x] = 0.0f;
  auto fold = [&](const piece &a, const float (&u)[TN]) {
#pragma unroll
    for (int y = 0; y < TN; ++y)
#pragma unroll
      for (int x = 0; x < TK; ++x) acc[y][x] = __fadd_rn(acc[y][x], __fmul_rn(u[y], a[x]));
  };
  auto request = [&](int mi, piece &a, float (&u)[TN]) {
    a = *(const TKV_GLOBAL piece *)(ap + (size_t)mi * k);
#pragma unroll
    for (int y = 0; y < TN; ++y) u[y] = up[(size_t)mi * n + y];
  };
  piece a[W_TOK];
  float u[W_TOK][TN];
#pragma unroll
  for (int i = 0; i < W_TOK; ++i) request(min(i, m - 1), a[i], u[i]);
  int mi = 0;
#pragma unroll 2
  for (; mi + W_TOK <= m; mi += W_TOK) {
    piece an[W_TOK];
    float un[W_TOK][TN];
#pragma unroll
    for (int i = 0; i < W_TOK; ++i) request(min(mi + W_TOK + i, m - 1), an[i], un[i]);
#pragma unroll
    for (int i = 0; i < W_TOK; ++i) fold(a[i], u[i]);
#pragma unroll
    for (int i = 0; i < W_TOK; ++i) {
      a[i] = an[i];
#pragma unroll
      for (int y = 0; y < TN; ++y) u[i][y] = un[i][y];
    }
  }
#pragma unroll
  for (int i = 0; i < W_TOK - 1; ++i)
    if (mi + i < m) fold(a[i], u[i]);
#pragma unroll
  for (int y = 0; y < TN; ++y) {
    piece out;
#pragma unroll
    for (int x = 0; x < TK; ++x) out[x] = acc[y][x];
    *(TKV_GLOBAL piece *)(grad_w + (size_t)(n0 + y) * k + k0) = out;
  }
}

}  // namespace

namespace {

constexpr size_t SIMDS = 1024;  // 256 CUs x 4

template <int TT>
void launch_act(hipStream_t s, const uint8_t *codes, size_t nb, size_t n, size_t k, size_t m, const float *scales,
                const float *grad_output, float *grad_act, int wide) {
  const size_t total = nb * 4 * ((m + 16 * TT - 1) / (16 * TT));
  hipLaunchKernelGGL(tk_vjp_act_kernel<TT>, dim3((unsigned)((total + 7) / 8 * 8)), dim3(256), 0, s, codes, (int)nb,
                     (int)n, (int)k, (int)m, scales, grad_output, grad_act, wide);
}

template <int TN, int TK>
void launch_weight(hipStream_t s, size_t n, size_t k, size_t m, const float *act, const float *grad_output, float *grad_w,
                   float *grad_bias) {
  const size_t tiles = ((k + 64 * TK - 1) / (64 * TK)) * ((n + 4 * TN - 1) / (4 * TN));
  const unsigned bias_blocks = grad_bias ? (unsigned)((n + 255) / 256) : 0;
  hipLaunchKernelGGL((tk_vjp_weight_kernel<TN, TK>), dim3(bias_blocks + (unsigned)((tiles + 7) / 8 * 8)), dim3(256), 0, s,
                     (int)n, (int)k, (int)m, act, grad_output, grad_w, grad_bias, (int)bias_blocks);
}

}  // namespace

// m, n, k > 0 for the matrix kernels (the caller has zero-filled or skipped the degenerate shapes);
// grad_act / grad_w / grad_bias may each be null to skip that output.
hipError_t tk_launch_projected_vjp(hipStream_t s, const uint8_t *codes, size_t nb, size_t n, size_t k, size_t m,
                                   const float *scales, const float *act, const float *grad_output, float *grad_act,
                                   float *grad_w, float *grad_bias) {
  if (grad_act && m && n && k) {
    const int wide = n % 4 == 0 && (uintptr_t)grad_output % 16 == 0 && (uintptr_t)scales % 16 == 0;
    // More tokens per wave share a decoded operand (vector work adds to the matrix time), fewer leave more waves. In
    // 16 x 16 tiles of the output, tiles per wave 1 / 2 / 4, N=2560: 640 tiles 31 / 43 / 62 us, 2560 tiles 60 / 67 / 63,
    // 10240 tiles 168 / 143 / 147; N=6912: 5120 tiles 238 / 241 / 274, 20480 tiles 871 / 732 / 640.
    const size_t tiles = nb * 16 * ((m + 15) / 16);
    if (tiles <= 4 * SIMDS) launch_act<1>(s, codes, nb, n, k, m, scales, grad_output, grad_act, wide);
    else if (tiles <= 12 * SIMDS) launch_act<2>(s, codes, nb, n, k, m, scales, grad_output, grad_act, wide);
    else launch_act<4>(s, codes, nb, n, k, m, scales, grad_output, grad_act, wide);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
  }
  if (grad_w && m && n && k) {
    const size_t outs = n * k;
    // The larger the tile of a wave, the more operations per load; the launch should still have some four waves per SIMD.
    // Rows x columns per lane 4x1 / 8x2 / 8x4: 0.5 M outputs (M=712) 57 / 79 / 108 us, 1.8 M (M=300) 64 / 38 / 50, 6.5 M
    // (M=1024) 591 / 305 / 336, 17.7 M (M=2048) 3014 / 1455 / 1385.
    if (n < 4) launch_weight<1, 1>(s, n, k, m, act, grad_output, grad_w, grad_bias);
    else if (k < 4 || n < 8 || outs < (size_t)1 << 20) launch_weight<4, 1>(s, n, k, m, act, grad_output, grad_w, grad_bias);
    else if (outs < (size_t)1 << 23) launch_weight<8, 2>(s, n, k, m, act, grad_output, grad_w, grad_bias);
    else launch_weight<8, 4>(s, n, k, m, act, grad_output, grad_w, grad_bias);
    return hipGetLastError();
  }
  if (grad_bias && n) {
    hipLaunchKernelGGL(tk_vjp_bias_kernel, dim3((unsigned)((n + 63) / 64)), dim3(64), 0, s, (int)n, (int)m,
                       grad_output, grad_bias);
    return hipGetLastError();
  }
  return hipSuccess;
}
