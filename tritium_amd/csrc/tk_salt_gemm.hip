// Block-scale additive planes (SALT) on many tokens: float activations as four digit rows per token (as in the flow
// form), 64 operand rows (16 tokens) x 32 * PAIRS columns per wave on v_mfma_i32_32x32x32_i8.
//
// A K block of 256 has its own scale per output column, so every block is finished on its own: 16 matrix instructions
// per plane and pair, then 7 vector instructions per output, plane and block. What this form saves over passes of 16 tokens
// through the flow form is the passes: the planes stream once per 64-row tile of a workgroup that shares its L2 with
// the other row tiles of the same columns, and one launch fills the chip where a pass of 16 tokens does not.
// Two planes K=2048 N=8192, 128 tokens, call: 172 us in eight passes -> 26.5 us (kernel 21.5). Bound: the vector work of the
// finishes and expansions beside the matrix pipe for large launches; for small ones the latency of a block's loads (1.7 us
// per block with a single wave per SIMD).
//
// Work split: four waves side by side share the 64 operand rows through LDS (two buffers of one K block, one barrier
// per block; 16 KiB per block are 64 bytes per thread, requested one block ahead). A wave goes through a block in steps of PI
// planes, whose codes and block scales come one step ahead into registers. Accumulators start at minus the block's
// operand-row sums (code = trit + 1), taken as the C operand of the first matrix instruction. The two high and the two low
// digits meet as integers: |x| <= 128 * 256 over a block, so x3 * 256 + x2 stays within 24 bits and its conversion is
// the exact value that the flow form's first two FMAs give. The sum over blocks (ascending) and planes (ascending
// inside a block) is the flow form's: identical bits.
#include "tk_device.h"

typedef int v16i __attribute__((ext_vector_type(16)));

namespace {

// The outputs of column n in the host's order (salt_exact_dot) for the eight tokens of a lane, which of them is asked for or not: one
// pass over the weights, four elements at a time (their codes are four bytes, a token's activations one load), the next four
// requested before these are used. A dot after the other was a pass of dependent loads each: two planes K=8192 N=2048, 8 tokens,
// one / all flagged 3.2 / 12.8 ms -> 1.1 / 1.1; K=2560 N=2560, 16 tokens 0.67 / 5.2 -> 0.31 / 0.31 (in the host's order from the
// start, as tk_salt_seq_kernel runs it, 3.3 and 0.69).
template <bool BF16>
__device__ __forceinline__ void exact_tokens(const TkProblem &pr, int n, const int (&tok)[8], float (&out)[8]) {
  typedef unsigned raw __attribute__((ext_vector_type(BF16 ? 2 : 4), aligned(BF16 ? 2 : 4)));
  const int nb = pr.nb, kdim = pr.k, planes = pr.planes;
  const uint8_t *act = (const uint8_t *)pr.raw_act;
  const size_t tile_base = (size_t)(n >> 4) * nb;
  raw a_next[8];
  unsigned c_next[TK_MAX_PLANES];
  // elements e .. e+3 of a K block: bytes of piece `byte / 16`, bit pair (e & 127) / 32 (code_at)
  auto request = [&](int k) {
    const int e = k & 255, byte = (e >> 7) * 32 + (e & 31);
    const size_t at = ((tile_base + (k >> 8)) * 64 + (byte >> 4) * 16 + (n & 15)) * 16 + (byte & 15);
#pragma unroll
    for (int p = 0; p < TK_MAX_PLANES; ++p)
      if (p < planes) c_next[p] = *(const TK_GLOBAL unsigned *)(pr.codes[p] + at);
    if (k + 4 <= kdim) {
#pragma unroll
      for (int i = 0; i < 8; ++i) a_next[i] = *(const TK_GLOBAL raw *)(act + ((size_t)tok[i] * kdim + k) * (BF16 ? 2 : 4));
    }
  };
  request(0);
#pragma unroll
  for (int i = 0; i < 8; ++i) out[i] = 0.0f;
  for (int kb = 0; kb < nb; ++kb) {
    float sc[TK_MAX_PLANES];
#pragma unroll
    for (int p = 0; p < TK_MAX_PLANES; ++p) sc[p] = p < planes ? gload(pr.bscale[p] + (tile_base + kb) * 16 + (n & 15)) : 0.0f;
    const int kend = min(kdim, (kb + 1) * 256);
#pragma unroll 1
    for (int k = kb * 256; k < kend; k += 4) {
      float a[8][4], w[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
      for (int i = 0; i < 8; ++i)
#pragma unroll
        for (int x = 0; x < 4; ++x) {
          if constexpr (BF16) a[i][x] = __uint_as_float(x & 1 ? a_next[i][x / 2] & 0xFFFF0000u : a_next[i][x / 2] << 16);
          else a[i][x] = __uint_as_float(a_next[i][x]);
        }
      if (k + 4 > kdim) {  // the last elements of a ragged row
#pragma unroll
        for (int i = 0; i < 8; ++i)
#pragma unroll
          for (int x = 0; x < 4; ++x) a[i][x] = load_act(act, BF16 ? TK_BF16 : TK_F32, (size_t)tok[i] * kdim + min(k + x, kdim - 1));
      }
      const int pair = (k & 127) >> 5;
#pragma unroll
      for (int p = 0; p < TK_MAX_PLANES; ++p) {
        if (p >= planes) break;
        const unsigned codes = c_next[p] >> (2 * pair);
#pragma unroll
        for (int x = 0; x < 4; ++x) w[x] = __fadd_rn(w[x], __fmul_rn(sc[p], (float)((int)((codes >> (8 * x)) & 3u) - 1)));
      }
      request(min(k + 4, kdim - 1) & ~3);
#pragma unroll
      for (int x = 0; x < 4; ++x)
        if (k + x < kdim)
#pragma unroll
          for (int i = 0; i < 8; ++i) out[i] = __fadd_rn(out[i], __fmul_rn(a[i][x], w[x]));
    }
  }
}

constexpr int ROWS = 64, SEGS = 16;  // operand rows per workgroup; 1-KiB segments ((j,g) x 64 rows) per K block

// PAIRS: 32-column pairs of tiles per wave; PI: planes per step (divides the layer's planes)
template <int PAIRS, int PI>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2, 2))) void tk_salt_gemm_kernel(const TkProblem single) {
  __shared__ __attribute__((aligned(16))) uint8_t s_a[2][SEGS * ROWS * 16];
  __shared__ __attribute__((aligned(16))) int s_bs[2][ROWS];
  const TkProblem &pr = *single_problem();
  const int nb = pr.nb, R = pr.R, M = pr.M, ncols = pr.n, n_tiles = pr.n_tiles, planes = pr.planes;
  const unsigned grid_m = (unsigned)pr.grid_m, total = grid_m * (unsigned)pr.grid_n;
  // XCD x = id % 8 takes the x-th eighth of the tiles, row tiles of one column block side by side: its L2 keeps the
  // column block's codes while the row tiles pass
  const unsigned idx = (blockIdx.x & 7u) * ((total + 7u) >> 3) + (blockIdx.x >> 3);
  if (idx >= total) return;
  const int row0 = (int)(idx % grid_m) * ROWS;
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  const int r = lane & 15, h = (lane >> 4) & 1, kappa = lane >> 5;
  const int pair0 = ((int)(idx / grid_m) * 4 + wave) * PAIRS;

  // this lane's tile of every pair (tiles past the end re-read the last one; nothing of them is stored)
  unsigned chunk0[PAIRS];
#pragma unroll
  for (int y = 0; y < PAIRS; ++y) chunk0[y] = (unsigned)min((pair0 + y) * 2 + h, n_tiles - 1) * (unsigned)nb;
  const int8_t *ap = pr.ap;
  const int32_t *blocksum = pr.blocksum;

  uint4 a_next[4], w_next[PAIRS][PI][2];
  float s_next[PAIRS][PI];
  int bs_next = 0;
  const int row_in = min(row0 + lane, R - 1);
  auto request_rows = [&](int kb) {
#pragma unroll
    for (int u = 0; u < 4; ++u)
      a_next[u] = gload16(ap + ((size_t)kb * SEGS + u * 4 + wave) * (size_t)R * 16 + (unsigned)row_in * 16u);
    bs_next = gload(blocksum + (size_t)kb * R + row_in);
  };
  auto request_codes = [&](int kb, int p0) {
#pragma unroll
    for (int p = 0; p < PI; ++p) {
      const uint8_t *codes = pr.codes[p0 + p];
      const float *bscale = pr.bscale[p0 + p];
#pragma unroll
      for (int y = 0; y < PAIRS; ++y) {
        const size_t chunk = chunk0[y] + (unsigned)kb;
#pragma unroll
        for (int l = 0; l < 2; ++l) w_next[y][p][l] = gload16(codes + chunk * 1024 + ((2 * l + kappa) * 16 + r) * 16);
        s_next[y][p] = gload(bscale + chunk * 16 + r);
      }
    }
  };
  auto stage = [&](int buf) {
#pragma unroll
    for (int u = 0; u < 4; ++u) *(uint4 *)(s_a[buf] + ((u * 4 + wave) * ROWS + lane) * 16) = a_next[u];
    if (tid < ROWS) s_bs[buf][tid] = -bs_next;
  };

  float facc[2][4][PAIRS];
#pragma unroll
  for (int t = 0; t < 2; ++t)
#pragma unroll
    for (int q = 0; q < 4; ++q)
#pragma unroll
      for (int y = 0; y < PAIRS; ++y) facc[t][q][y] = 0.0f;

  request_rows(0);
  request_codes(0, 0);
  stage(0);
  for (int kb = 0; kb < nb; ++kb) {
    const int buf = kb & 1;
    __syncthreads();  // this block's rows are staged; the other buffer's last readers are past
    if (kb + 1 < nb) request_rows(kb + 1);
    for (int p0 = 0; p0 < planes; p0 += PI) {
      uint4 w[PAIRS][PI][2];
      float sc[PAIRS][PI];
#pragma unroll
      for (int y = 0; y < PAIRS; ++y)
#pragma unroll
        for (int p = 0; p < PI; ++p) {
          w[y][p][0] = w_next[y][p][0];
          w[y][p][1] = w_next[y][p][1];
          sc[y][p] = s_next[y][p];
        }
      {  // (the last step asks for its own codes again)
        const bool same = p0 + PI < planes;
        request_codes(same ? kb : min(kb + 1, nb - 1), same ? p0 + PI : 0);
      }
      v16i acc[2][PAIRS][PI];
#pragma unroll
      for (int l = 0; l < 2; ++l)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          v4i a[2];
#pragma unroll
          for (int t = 0; t < 2; ++t) a[t] = *(const v4i *)(s_a[buf] + ((j * 4 + 2 * l + kappa) * ROWS + t * 32 + (lane & 31)) * 16);
#pragma unroll
          for (int y = 0; y < PAIRS; ++y)
#pragma unroll
            for (int p = 0; p < PI; ++p) {
              const uint4 wl = w[y][p][l];
              const v4i b = expand_codes(j == 0 ? wl.x : (j == 1 ? wl.y : (j == 2 ? wl.z : wl.w)));
#pragma unroll
              for (int t = 0; t < 2; ++t) {
                if (l == 0 && j == 0) {
                  v16i c;
#pragma unroll
                  for (int q = 0; q < 4; ++q) {
                    const v4i bs = *(const v4i *)(s_bs[buf] + t * 32 + q * 8 + kappa * 4);
#pragma unroll
                    for (int e = 0; e < 4; ++e) c[q * 4 + e] = bs[e];
                  }
                  acc[t][y][p] = __builtin_amdgcn_mfma_i32_32x32x32_i8(a[t], b, c, 0, 0, 0);
                } else {
                  acc[t][y][p] = __builtin_amdgcn_mfma_i32_32x32x32_i8(a[t], b, acc[t][y][p], 0, 0, 0);
                }
              }
            }
        }
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int y = 0; y < PAIRS; ++y)
#pragma unroll
          for (int p = 0; p < PI; ++p)
#pragma unroll
            for (int q = 0; q < 4; ++q) {
              const v16i &x = acc[t][y][p];
              const float hi = (float)(x[q * 4 + 3] * 256 + x[q * 4 + 2]), lo = (float)(x[q * 4 + 1] * 256 + x[q * 4]);
              const float v = __builtin_fmaf(hi, 65536.0f, lo);
              facc[t][q][y] = __fadd_rn(facc[t][q][y], __fmul_rn(v, sc[y][p]));
            }
    }
    if (kb + 1 < nb) stage(buf ^ 1);
  }

  // register 4q + e of row tile t is digit e of token 8t + 2q + kappa of the tile
  void *const out = pr.out;
  const int out_dtype = pr.out_dtype;
  int tok[8];
  unsigned mine = 0;
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    tok[i] = min((row0 >> 2) + i * 2 + kappa, M - 1);
    const bool flag = (row0 >> 2) + i * 2 + kappa < M && gload(pr.flags + tok[i]);
    mine |= flag ? 1u << i : 0u;
  }
  const bool any = __ballot(mine != 0) != 0;
#pragma unroll
  for (int y = 0; y < PAIRS; ++y) {
    const int n = ((pair0 + y) * 2 + h) * 16 + r;
    float exact[8];
    if (any && pr.raw_dtype == TK_BF16) exact_tokens<true>(pr, min(n, ncols - 1), tok, exact);
    else if (any) exact_tokens<false>(pr, min(n, ncols - 1), tok, exact);
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      if ((row0 >> 2) + i * 2 + kappa >= M || n >= ncols) continue;
      const float f = (mine >> i) & 1u ? exact[i] : ldexpf(facc[i >> 2][i & 3][y], gload(pr.exps + tok[i]));
      store_out(out, out_dtype, (size_t)tok[i] * ncols + n, f);
    }
  }
}

template <int PAIRS, int PI>
hipError_t launch(hipStream_t s, TkProblem pr) {
  pr.grid_m = (pr.R + ROWS - 1) / ROWS;
  pr.grid_n = ((pr.n_tiles + 1) / 2 + 4 * PAIRS - 1) / (4 * PAIRS);
  const unsigned total = (unsigned)pr.grid_m * (unsigned)pr.grid_n;
  hipLaunchKernelGGL((tk_salt_gemm_kernel<PAIRS, PI>), dim3((total + 7) / 8 * 8), dim3(256), 0, s, pr);
  return hipGetLastError();
}

}  // namespace

hipError_t tk_launch_salt_gemm(hipStream_t s, const TkProblem *single, int compute_units) {
  // 64 columns per wave halve the operand reads per matrix instruction (with 32 columns and one plane per step they keep LDS
  // as busy as the matrix pipe), 32 columns make twice the workgroups. Measured, call, K=2048 N=8192, 32 / 64 columns:
  // 512 tokens (1024 workgroups of the wide form) 67 / 50, 80 / 69, 119 / 88 us for one, two, three planes; 128 tokens
  // (256) 23 / 24, 28 / 30, 34 / 36; K=8192 N=2048 512 tokens (256) 65 / 67, 80 / 93, 116 / 118.
  const long wide = (long)((single->R + ROWS - 1) / ROWS) * ((single->n_tiles + 15) / 16);
  if (wide >= 2l * compute_units) return launch<2, 1>(s, *single);
  // two planes per step: 28 / 28.5 us (128 tokens), 62 / 75 us (K=8192 N=2048 128 tokens) against one
  return single->planes % 2 == 0 ? launch<1, 2>(s, *single) : launch<1, 1>(s, *single);
}
