// Decode of small batches (3 to 64 operand rows): eight waves of a workgroup split the K blocks of 32 output columns.
//
// Launches of such calls are a latency chain: few workgroups, each walking K with its rows staged through LDS behind barriers
// (K-split kernel), or K slices of several workgroups that meet through memory and a counter (prefill kernel with its K split).
// Here a wave takes every eighth K block of a 32-column pair of tiles for all operand rows: rows and codes go from
// memory straight to registers in whole 16-byte pieces (a block's pieces are requested together, one block ahead), 8
// matrix instructions per block, plane and 32 rows, no barrier before the end. Then the eight waves' int32 sums meet in LDS --
// integer adds in any order: the same bits as every other form -- and the epilogue of the decode kernels finishes them.
// The operand rows are read once per workgroup and 32 columns: they come from L2.
// Bound: latency (launch, two or three dependent loads, the meeting in LDS). Registers are held to 128 where that is possible,
// so that two workgroups share a CU: with 160 (two planes) N=13824 K=2560 16 rows took 15.5 us instead of 11.4. Kernel alone
// K=2560 N=2560 32 rows: 15.5 us (prefill kernel with its K split) -> about 6; a decoder layer of hidden 2560 with 32 tokens
// (seven projections, four calls) 75 -> 48 us.
#include "tk_device.h"

typedef int v16i __attribute__((ext_vector_type(16)));

namespace {

constexpr int WAVES = 8;

// RT: 32-row tiles of operand rows (1: up to 32 rows, 2: up to 64)
template <int P, int RT, bool TABLE>
__global__ __launch_bounds__(WAVES * 64) __attribute__((amdgpu_waves_per_eu(RT * P <= 3 ? 4 : 2, RT * P <= 3 ? 4 : 2))) void
tk_waves_kernel(const TkProblem single, const TkProblem *__restrict__ table, const int *__restrict__ wg_prob) {
  __shared__ __attribute__((aligned(16))) v4i part[WAVES][RT][4][64];  // [wave][row tile][register quad][lane]
  const TkProblem &pr = TABLE ? table[wg_prob[blockIdx.x]] : *single_problem();
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int r = lane & 15, h = (lane >> 4) & 1, kappa = lane >> 5;
  const int nb = pr.nb, R = pr.R, n_tiles = pr.n_tiles;
  const int pair = (int)blockIdx.x - (TABLE ? pr.group_begin : 0);
  const size_t chunk0 = (size_t)min(pair * 2 + h, n_tiles - 1) * (unsigned)nb;  // (a tile past the end: not stored)
  const uint8_t *codes[P];
#pragma unroll
  for (int p = 0; p < P; ++p) codes[p] = pr.codes[p] + chunk0 * 1024 + (kappa * 16 + r) * 16;
  const size_t seg = (size_t)pr.rs * 16;  // bytes of one (K block, j, g) segment of operand rows
  const int8_t *rows[RT];
#pragma unroll
  for (int t = 0; t < RT; ++t) rows[t] = pr.ap + kappa * seg + (size_t)min(t * 32 + (lane & 31), R - 1) * 16;

  // a unit of work is a whole K block for one plane and one row tile, else half of one (the registers hold two units)
  constexpr int L = RT * P == 1 ? 2 : 1, PER = 2 / L;
  struct Unit {
    uint4 a[RT][L][4], w[P][L];
  };
  auto request = [&](Unit &b, int u) {
    const int kb = PER == 1 ? u : u >> 1, l0 = PER == 1 ? 0 : u & 1;
#pragma unroll
    for (int p = 0; p < P; ++p)
#pragma unroll
      for (int l = 0; l < L; ++l) b.w[p][l] = gload16(codes[p] + (size_t)kb * 1024 + (l0 + l) * 512);
#pragma unroll
    for (int t = 0; t < RT; ++t)
#pragma unroll
      for (int l = 0; l < L; ++l)
#pragma unroll
        for (int j = 0; j < 4; ++j) b.a[t][l][j] = gload16(rows[t] + ((size_t)kb * 16 + j * 4 + 2 * (l0 + l)) * seg);
  };
  v16i acc[RT][P];
#pragma unroll
  for (int t = 0; t < RT; ++t)
#pragma unroll
    for (int p = 0; p < P; ++p)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[t][p][e] = 0;
  const int units = nb * PER;
  if (wave < units) {
    Unit next;
    request(next, wave);
    for (int u = wave; u < units; u += WAVES) {
      const Unit b = next;
      if (u + WAVES < units) request(next, u + WAVES);
#pragma unroll
      for (int l = 0; l < L; ++l)
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
          for (int p = 0; p < P; ++p) {
            const uint4 wl = b.w[p][l];
            const v4i bw = expand_codes(j == 0 ? wl.x : (j == 1 ? wl.y : (j == 2 ? wl.z : wl.w)));
#pragma unroll
            for (int t = 0; t < RT; ++t) {
              const uint4 q = b.a[t][l][j];
              acc[t][p] = __builtin_amdgcn_mfma_i32_32x32x32_i8(v4i{(int)q.x, (int)q.y, (int)q.z, (int)q.w}, bw, acc[t][p], 0, 0, 0);
            }
          }
    }
  }
  // Thread x of the first RT * 256 finishes quad (x / 64) % 4 of row tile x / 256: four consecutive rows of one column.
  const int et = wave >> 2, eq = wave & 3;
  const bool ends = et < RT;
  v4i sum[P];
#pragma unroll
  for (int p = 0; p < P; ++p) {
    if (p) __syncthreads();
#pragma unroll
    for (int t = 0; t < RT; ++t)
#pragma unroll
      for (int q = 0; q < 4; ++q)
        part[wave][t][q][lane] = v4i{acc[t][p][q * 4], acc[t][p][q * 4 + 1], acc[t][p][q * 4 + 2], acc[t][p][q * 4 + 3]};
    __syncthreads();
    if (ends) {
      sum[p] = part[0][et][eq][lane];
#pragma unroll
      for (int w = 1; w < WAVES; ++w) sum[p] += part[w][et][eq][lane];
    }
  }
  if (!ends) return;
  const int n = (pair * 2 + h) * 16 + r, rowbase = et * 32 + eq * 8 + kappa * 4;
  const TkHot hot = make_hot(pr);
  if (n >= hot.n || rowbase >= R) return;
  float sc[P];
#pragma unroll
  for (int p = 0; p < P; ++p) sc[p] = hot.out_dtype == TK_I32 ? 0.0f : gload(pr.scales[p] + n);
  const RowConst rc = load_row_const(hot, rowbase);
  flow_epilogue<P>(hot, n, rowbase, sum, sc, rc);
  if (rc.flag) exact_rows(pr, n, rowbase, rc.flag);
}

template <int P, int RT>
hipError_t go(hipStream_t s, const TkProblem *single, const TkProblem *table, const int *wg_prob, unsigned grid) {
  const TkProblem dummy = {};
  if (table) hipLaunchKernelGGL((tk_waves_kernel<P, RT, true>), dim3(grid), dim3(WAVES * 64), 0, s, dummy, table, wg_prob);
  else hipLaunchKernelGGL((tk_waves_kernel<P, RT, false>), dim3(grid), dim3(WAVES * 64), 0, s, *single, nullptr, nullptr);
  return hipGetLastError();
}

}  // namespace

hipError_t tk_launch_waves(hipStream_t s, const TkProblem *single, const TkProblem *table, const int *wg_prob, int planes,
                           int rows, unsigned grid) {
  if (rows > 64) return hipErrorInvalidValue;
  const bool two = rows > 32;
  switch (planes) {
    case 1: return two ? go<1, 2>(s, single, table, wg_prob, grid) : go<1, 1>(s, single, table, wg_prob, grid);
    case 2: return two ? go<2, 2>(s, single, table, wg_prob, grid) : go<2, 1>(s, single, table, wg_prob, grid);
    case 3: return two ? hipErrorInvalidValue : go<3, 1>(s, single, table, wg_prob, grid);
    default: return hipErrorInvalidValue;
  }
}
