// gfx950 prefill GEMM, 128 operand rows (96 for three planes) per workgroup: one to three planes under the int8 contract, two and
// three under the float contract.
//
// The 64-row prefill kernel (tk_kernels.hip) is held back by the CU's vector-memory path and by the expansion of the 2-bit
// codes: every wave expands the codes of its own columns, seven vector instructions for an operand that two matrix
// instructions use, and a K block of 64 rows x 384 plane columns brings in 40 KiB. Here a workgroup is four waves side by
// side over 128 rows x 128 plane columns and more: an expanded operand serves four matrix instructions (three for three
// planes: 96 rows, whose 144 accumulators leave room for two waves per SIMD), and a byte that comes in serves a quarter to a
// third more of them. The operand rows come to LDS by DMA in HALF K blocks (128 k: 16 KiB, three slots, two half blocks
// ahead), so that two workgroups still share a CU; the weight codes go straight to registers, one 16-byte piece per lane,
// pair of tiles and half block; one barrier per half block (32 or 36 matrix instructions per wave).
// Lane maps are those of the 64-row kernel (v_mfma_i32_32x32x32_i8): lane L = 32 kappa + 16 h + r takes piece g = 2 l + kappa
// of row r of tile h of a pair, l = the half of the K block; dword j of the piece is the operand of k step j. The codes are
// trit + 1, so the accumulators start at minus the row sums. Same integers, same epilogue arithmetic: identical bits.
// A K whose last block holds at most 128 elements has one half block less (its operand rows are zero there).
//
// One plane has a second form, eight waves of 32 columns in 128 registers: where a CU has one workgroup, four waves leave every
// SIMD a single one to hide its loads behind (gemm128_eight_waves in tk_api.hip).
//
// Bound: in long launches the chip's power -- registers full of gaussian int8 rows and codes, nothing but matrix instructions,
// hold 4.0 to 4.2 POPS of the 5.0 that all-zero operands reach (3.5 with the weights as the first operand: so activations go
// first), and interleaving the expansion with the matrix instructions one by one changed nothing. Otherwise the number of
// workgroups on the CU that has most (gemm128_pays in tk_api.hip). Calls incl. quantization, 64 rows -> 128: 4096 tokens K=5120
// N=17408 three planes 759 -> 738 us, 1024 tokens K=5120 N=5120 79 -> 72, 200 tokens N=17408 73 -> 65; 768 tokens K=6144
// N=20480 one plane 98 -> 83, two planes (N=10240) 87 -> 81; float contract 333 f32 tokens K=2050 N=5003 two planes 43.2 ->
// 41.1 (35.7 with the epilogue and the digit split of now). Counters: the matrix pipes work for 0.77 of a long launch's cycles
// with three planes, 0.72 with two, 0.69 with one; with one workgroup per CU (1024 tokens K=6912 N=6912) for 0.45 on four waves
// and 0.48 on eight.

#include <type_traits>

#include "tk_device.h"

typedef int v16i_g __attribute__((ext_vector_type(16)));

namespace {

constexpr int SLOTS = 3, BAND = 4;

// P planes, W waves, NT tiles of 16 outputs per wave and plane, RT 32-row tiles of operand rows per workgroup
template <int P, int W>
struct Form {
  static constexpr int NT = P == 1 && W == 4 ? 4 : 2, RT = P == 3 ? 3 : 4, ROWS = 32 * RT;
  static constexpr int LOADS = 4 * RT / W;            // wave-wide DMA loads per wave and half block
  static constexpr int SLOT = ROWS * 128;             // bytes of a half block of operand rows
  static constexpr int CST = SLOTS * SLOT;            // float act_scale[128] | int exps[64] | uint flags[128]
  static constexpr int LDS = CST + 512 + 256 + 512;
};

template <int P, int W>
__global__ __launch_bounds__(W * 64) __attribute__((amdgpu_waves_per_eu(W / 2, W / 2))) void tk_gemm128_kernel(const TkProblem single) {
  using F = Form<P, W>;
  constexpr int WAVES = W, LOADS = F::LOADS, NT = F::NT, RT = F::RT, ROWS = F::ROWS, HP = NT / 2, NP = HP * P;
  extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
  const TkProblem &pr = *single_problem();
  const TkHot hot = make_hot(pr);
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r16 = lane & 15, h = (lane >> 4) & 1, r32 = lane & 31, kappa = lane >> 5;
  const int nb = pr.nb, R = pr.R, n_tiles = pr.n_tiles, rs = pr.rs;
  const int H = 2 * nb - (((pr.k - 1) & 255) < 128 ? 1 : 0);  // half blocks that hold elements

  // XCD x = id % 8 owns a compact sub-grid of sub_m x sub_n workgroups and walks it in bands of BAND row blocks, down the
  // band first (as the 64-row kernel does)
  const int xcd = (int)(blockIdx.x & 7u), at = (int)(blockIdx.x >> 3);
  const int sub_m = pr.sub_m, sub_n = pr.sub_n;
  const int band = at / (BAND * sub_n), in_band = at - band * (BAND * sub_n);
  const int band_rows = min(BAND, sub_m - band * BAND);
  if (band_rows <= 0) return;
  const int lm = band * BAND + in_band % band_rows, ln = in_band / band_rows;
  const int bm = (xcd % pr.xr) * sub_m + lm, bn = (xcd / pr.xr) * sub_n + ln;
  if (ln >= sub_n || bm >= pr.grid_m || bn >= pr.grid_n) return;
  const int row0 = bm * ROWS, tile0 = (bn * WAVES + wave) * NT;

  // ---- operand addresses ----
  // weights: lane offset of pair z, the same in every plane (tiles past the end re-read the last one; results dropped)
  unsigned w_off[HP];
#pragma unroll
  for (int z = 0; z < HP; ++z)
    w_off[z] = (unsigned)min(tile0 + 2 * z + h, n_tiles - 1) * (unsigned)nb * 1024u + (unsigned)(kappa * 16 + r16) * 16u;
  // operand rows: a half block is 8 segments (j, kappa) of ROWS pieces, cut into 4 RT wave-wide DMA loads
  unsigned a_off[LOADS];
#pragma unroll
  for (int i = 0; i < LOADS; ++i) {
    const int idx = (wave * LOADS + i) * 64 + lane, seg = idx / ROWS, row = idx - seg * ROWS;
    a_off[i] = (unsigned)((seg >> 1) * 4 + (seg & 1)) * (unsigned)rs * 16u + (unsigned)min(row0 + row, R - 1) * 16u;
  }
  auto load_w = [&](v4i (&w)[NP], int hb) {
#pragma unroll
    for (int p = 0; p < P; ++p) {
      const uint8_t *base = pr.codes[p] + (size_t)(unsigned)hb * 512u;  // wave-uniform
#pragma unroll
      for (int z = 0; z < HP; ++z)
        asm volatile("global_load_dwordx4 %0, %1, %2" : "=v"(w[p * HP + z]) : "v"(w_off[z]), "s"(base));
    }
  };
  auto dma = [&](int hb, int slot) {
    const uint8_t *base = (const uint8_t *)pr.ap + ((size_t)(hb >> 1) * 16 + (hb & 1) * 2) * (size_t)rs * 16;  // wave-uniform
#pragma unroll
    for (int i = 0; i < LOADS; ++i)
      __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void *)(base + a_off[i]),
                                       (__attribute__((address_space(3))) void *)(smem + slot * F::SLOT + (wave * LOADS + i) * 1024), 16, 0, 0);
  };

  // ---- prologue: constants, minus the row sums, the first two half blocks ----
  const bool int8_in = P == 1 || hot.mode == TK_MODE_INT8;  // (one plane: the int8 contract only)
  {
    const void *src = nullptr;
    int last = 0, first = 0, n64 = 0, dst = 0;
    if (wave == 0 && int8_in && hot.act_scale) src = hot.act_scale, first = row0, last = R - 1, n64 = 2, dst = 0;
    if (wave == 1 && !int8_in) src = hot.exps, first = row0 >> 2, last = hot.M - 1, n64 = 1, dst = 512;
    if (wave == 2 && hot.flags) src = hot.flags, first = int8_in ? row0 : row0 >> 2, last = int8_in ? R - 1 : hot.M - 1, n64 = int8_in ? 2 : 1, dst = 768;
    for (int i = 0; i < n64; ++i)
      __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void *)((const uint32_t *)src + min(first + i * 64 + lane, last)),
                                       (__attribute__((address_space(3))) void *)(smem + F::CST + dst + i * 256), 4, 0, 0);
  }
  float sc[HP][P];
#pragma unroll
  for (int z = 0; z < HP; ++z) {
    const int n = (tile0 + 2 * z + h) * 16 + r16;
#pragma unroll
    for (int p = 0; p < P; ++p) sc[z][p] = hot.out_dtype == TK_I32 ? 0.0f : gload(pr.scales[p] + min(n, hot.n - 1));
  }
  // (requested before the row sums are waited for: one trip to memory, not two)
  v4i wset[SLOTS][NP], a[2][RT];
  load_w(wset[0], 0);
  dma(0, 0);
  if (H > 1) {
    load_w(wset[1], 1);
    dma(1, 1);
  }
  v16i_g acc[RT][NP];
  if (row0 + ROWS <= R) {
    v4i rs4[RT][4];
#pragma unroll
    for (int rt = 0; rt < RT; ++rt)
#pragma unroll
      for (int q = 0; q < 4; ++q) rs4[rt][q] = *(const TK_GLOBAL v4i *)(hot.rowsum + row0 + rt * 32 + 8 * q + 4 * kappa);
#pragma unroll
    for (int rt = 0; rt < RT; ++rt)
#pragma unroll
      for (int e = 0; e < 16; ++e)
#pragma unroll
        for (int y = 0; y < NP; ++y) acc[rt][y][e] = -rs4[rt][e >> 2][e & 3];
  } else {
#pragma unroll
    for (int rt = 0; rt < RT; ++rt)
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        const int neg = -gload(hot.rowsum + min(row0 + rt * 32 + 8 * (e >> 2) + 4 * kappa + (e & 3), R - 1));
#pragma unroll
        for (int y = 0; y < NP; ++y) acc[rt][y][e] = neg;
      }
  }

  // wait until at most `ahead` of the youngest half blocks are still in flight
  auto wait_blocks = [&](int ahead) {
    if (ahead <= 0) asm volatile("s_waitcnt vmcnt(0)");
    else asm volatile("s_waitcnt vmcnt(%0)" ::"n"(LOADS + NP));
  };
  auto tie_w = [&](v4i (&w)[NP]) {
#pragma unroll
    for (int y = 0; y < NP; ++y) asm volatile("" : "+v"(w[y]));
  };
  const unsigned lds_lane = (unsigned)(size_t)(__attribute__((address_space(3))) uint8_t *)smem + (unsigned)(kappa * ROWS + r32) * 16u;
  auto lds_read = [&](v4i (&d)[RT], int off) {
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(d[rt]) : "v"(lds_lane), "n"(off + rt * 512));
  };
  // LDS reads return in order: wait until only those of the next k step (or none) are in flight
  auto lds_wait = [&](v4i (&d)[RT], bool ahead) {
    if (ahead) asm volatile("s_waitcnt lgkmcnt(%0)" ::"n"(RT));
    else asm volatile("s_waitcnt lgkmcnt(0)");
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) asm volatile("" : "+v"(d[rt]));
  };
  wait_blocks(0);
#pragma unroll
  for (int s = 0; s < SLOTS; ++s) tie_w(wset[s]);
  __builtin_amdgcn_s_barrier();

  // ---- half block hb in slot `cur`; block hb + 2 goes where block hb - 1 was ----
  auto block = [&](auto cur_c, int hb) {
    constexpr int cur = decltype(cur_c)::value, prev = (cur + 2) % SLOTS, next = (cur + 1) % SLOTS;
    if (hb + 2 < H) {
      load_w(wset[prev], hb + 2);
      dma(hb + 2, prev);
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      if (j < 3) lds_read(a[(j + 1) & 1], cur * F::SLOT + (j + 1) * 2 * ROWS * 16);
      lds_wait(a[j & 1], j < 3);
#pragma unroll
      for (int y = 0; y < NP; ++y) {
        const v4i b = expand_codes((uint32_t)wset[cur][y][j]);
#pragma unroll
        for (int rt = 0; rt < RT; ++rt) acc[rt][y] = __builtin_amdgcn_mfma_i32_32x32x32_i8(a[j & 1][rt], b, acc[rt][y], 0, 0, 0);
      }
    }
    wait_blocks(min(hb + 2, H - 1) - (hb + 1));  // block hb + 1 has landed
    tie_w(wset[next]);
    __builtin_amdgcn_s_barrier();
    lds_read(a[0], next * F::SLOT);  // (behind the last block: stale rows, waited for below)
  };
  lds_read(a[0], 0);
  int hb = 0;
  for (; hb + SLOTS <= H; hb += SLOTS) {  // one exit only: the accumulators keep their registers
    block(std::integral_constant<int, 0>{}, hb);
    block(std::integral_constant<int, 1>{}, hb + 1);
    block(std::integral_constant<int, 2>{}, hb + 2);
  }
  if (hb < H) {
    block(std::integral_constant<int, 0>{}, hb);
    if (hb + 1 < H) block(std::integral_constant<int, 1>{}, hb + 1);
  }
  lds_wait(a[0], false);

  // ---- epilogue ----
  const float *cst_as = (const float *)(smem + F::CST);
  const int *cst_exp = (const int *)(smem + F::CST + 512);
  const uint32_t *cst_flag = (const uint32_t *)(smem + F::CST + 768);
  const int tid = (int)threadIdx.x;
  unsigned my_flag = 0;
  if (hot.flags && tid < ROWS && (int8_in ? row0 + tid < R : (tid < ROWS / 4 && (row0 >> 2) + tid < hot.M))) my_flag = cst_flag[tid] ? 1u : 0u;
  const int wg_flag = __syncthreads_or((int)my_flag);  // (also: every wave is done with the slots)
  const bool has_as = int8_in && hot.act_scale;
  auto consts = [&](int rl) {  // of the 4 rows rl .. rl + 3 of the workgroup
    RowConst rc = {};
    const float4 as4 = *(const float4 *)(cst_as + rl);
    rc.as[0] = as4.x; rc.as[1] = as4.y; rc.as[2] = as4.z; rc.as[3] = as4.w;
    rc.exp = cst_exp[rl >> 2];
    if (wg_flag) {
      if (int8_in) {
#pragma unroll
        for (int r = 0; r < 4; ++r) rc.flag |= cst_flag[rl + r] ? 1u << r : 0u;
      } else {
        rc.flag = cst_flag[rl >> 2] ? 1u : 0u;
      }
    }
    return rc;
  };
  auto quad = [&](int rt, int q, int z, v4i (&av)[P]) {
#pragma unroll
    for (int p = 0; p < P; ++p) {
      const v16i_g &c = acc[rt][p * HP + z];
      av[p] = v4i{c[4 * q], c[4 * q + 1], c[4 * q + 2], c[4 * q + 3]};
    }
  };
  // int8 contract, output rows of whole 16-byte pieces, no residual: a wave stages 32 rows of its columns in its own piece of
  // LDS and writes them as whole segments
  auto staged = [&](auto esz_c) {
    constexpr int ESZ = decltype(esz_c)::value, COLS = NT * 16, STRIDE = COLS * ESZ + 16, PPR = COLS * ESZ / 16, RPI = 64 / PPR;
    static_assert(WAVES * 32 * STRIDE <= F::CST, "the staging areas fit the slots");
    uint8_t *wl = smem + wave * (32 * STRIDE);
    uint8_t *lane_base = wl + (4 * kappa) * STRIDE + (h * 16 + r16) * ESZ;
    const int piece = lane % PPR, srow = lane / PPR, c = tile0 * 16 + piece * (16 / ESZ);
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) {
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const float4 as4 = *(const float4 *)(cst_as + rt * 32 + 8 * q + 4 * kappa);
        RowConst rc = {};
        rc.as[0] = as4.x; rc.as[1] = as4.y; rc.as[2] = as4.z; rc.as[3] = as4.w;
#pragma unroll
        for (int z = 0; z < HP; ++z) {
          v4i av[P];
          quad(rt, q, z, av);
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const float f = int8_value<P>(av, r, sc[z], rc, has_as);
            uint8_t *dst = lane_base + (8 * q + r) * STRIDE + z * 32 * ESZ;
            if (ESZ == 2) *(uint16_t *)dst = f32_to_bf16_hw(f); else *(float *)dst = f;
          }
        }
      }
      __builtin_amdgcn_wave_barrier();
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      if (c < hot.n) {
#pragma unroll
        for (int it = 0; it < 32 / RPI; ++it) {
          const int rl = it * RPI + srow, orow = row0 + rt * 32 + rl;
          if (orow < R && !(wg_flag && cst_flag[rt * 32 + rl]))  // (flagged rows: exact_rows below)
            *(TK_GLOBAL v4u *)((uint8_t *)hot.out + ((size_t)orow * hot.n + c) * ESZ) = *(const v4u *)(wl + rl * STRIDE + piece * 16);
        }
      }
      __builtin_amdgcn_wave_barrier();
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    }
  };
  const int esz = hot.out_dtype == TK_BF16 ? 2 : 4;
  if (int8_in && hot.out_dtype != TK_I32 && (((size_t)hot.n * esz) & 15) == 0 && ((uintptr_t)hot.out & 15) == 0 && !hot.residual) {
    if (esz == 2) staged(std::integral_constant<int, 2>{});
    else staged(std::integral_constant<int, 4>{});
  } else if (!int8_in && !hot.residual && !wg_flag) {
    // float contract: token 8 rt + 2 q + kappa of the workgroup, one output per accumulator quad; a store is 32 adjacent
    // columns of two tokens (straight-line: one address per column, stepped by two tokens, where flow_epilogue decides per
    // output: 333 f32 tokens K=2050 N=5003 two planes, call 37.3 -> 35.7 us)
    auto plain = [&](auto esz_c) {
      constexpr int ESZ = decltype(esz_c)::value;
      const size_t step = (size_t)hot.n * (2 * ESZ);
      const int tok0 = (row0 >> 2) + kappa;
#pragma unroll
      for (int z = 0; z < HP; ++z) {
        const int n = (tile0 + 2 * z + h) * 16 + r16;
        uint8_t *dst = (uint8_t *)hot.out + ((size_t)tok0 * hot.n + n) * ESZ;
        const bool in = n < hot.n;
#pragma unroll
        for (int rt = 0; rt < RT; ++rt)
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            RowConst rc = {};
            rc.exp = cst_exp[rt * 8 + 2 * q + kappa];
            v4i av[P];
            quad(rt, q, z, av);
            const float f = digits_value<P>(av, sc[z], rc);
            if (in && tok0 + rt * 8 + 2 * q < hot.M) {
              if (ESZ == 2) gstore((uint16_t *)dst, f32_to_bf16_hw(f)); else gstore((float *)dst, f);
            }
            dst += step;
          }
      }
    };
    if (esz == 2) plain(std::integral_constant<int, 2>{});
    else plain(std::integral_constant<int, 4>{});
  } else {
#pragma unroll
    for (int rt = 0; rt < RT; ++rt)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int rl = rt * 32 + 8 * q + 4 * kappa;
        const RowConst rc = consts(rl);
#pragma unroll
        for (int z = 0; z < HP; ++z) {
          const int n = (tile0 + 2 * z + h) * 16 + r16;
          if (n >= hot.n) continue;
          v4i av[P];
          quad(rt, q, z, av);
          flow_epilogue<P>(hot, n, row0 + rl, av, sc[z], rc);
        }
      }
  }
  if (wg_flag) {
    for (int z = 0; z < HP; ++z) {
      const int n = (tile0 + 2 * z + h) * 16 + r16;
      if (n >= pr.n) continue;
      for (int rt = 0; rt < RT; ++rt)
        for (int q = 0; q < 4; ++q) {
          const int rowbase = row0 + rt * 32 + 8 * q + 4 * kappa;
          const unsigned fl = row_flags(pr, rowbase);
          if (fl) exact_rows(pr, n, rowbase, fl);
        }
    }
  }
}

template <int P, int W>
hipError_t go(hipStream_t s, const TkProblem *single, unsigned wgs) {
  hipLaunchKernelGGL((tk_gemm128_kernel<P, W>), dim3(wgs), dim3(W * 64), (size_t)(Form<P, W>::LDS), s, *single);
  return hipGetLastError();
}

}  // namespace

int tk_gemm128_rows(int planes) { return planes == 3 ? Form<3, 4>::ROWS : Form<1, 4>::ROWS; }
int tk_gemm128_tiles(int planes) { return 4 * (planes == 1 ? Form<1, 4>::NT : Form<2, 4>::NT); }

hipError_t tk_launch_gemm128(hipStream_t s, const TkProblem *single, bool eight_waves) {
  const unsigned wgs = 8u * (unsigned)single->sub_m * (unsigned)single->sub_n;
  if (!wgs) return hipSuccess;
  switch (single->planes) {
    case 1: return eight_waves ? go<1, 8>(s, single, wgs) : go<1, 4>(s, single, wgs);
    case 2: return go<2, 4>(s, single, wgs);
    case 3: return go<3, 4>(s, single, wgs);
    default: return hipErrorInvalidValue;
  }
}
