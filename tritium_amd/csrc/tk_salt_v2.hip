// SALT V2 on gfx950: the exact forward and the row gather over resident codec payloads.
//
// The reference pins one scalar order per output (crates/tritium-cpu/src/salt_v2.rs:10-23): segments --
// the pieces of a weight row that lie in one 256-coefficient allocation tile and one scale group -- in
// ascending order; within a segment the tile's planes ascending; within a plane one f32 accumulator over
// the columns (add, subtract or skip by the trit), one multiply by the plane's f16 scale, one add into the
// output. Its own device kernel walks all of that with one thread per output
// (crates/tritium-cuda/kernels/salt_v2.cu:133-214). Here the terms of different segments, which do not
// depend on each other, are computed by different lanes: a workgroup takes one weight row and up to eight
// tokens, every lane folds whole segments (decoding each trit once for all tokens) and leaves the products
// in LDS; then one lane per token adds them in the pinned order. Same operations, same order per output,
// so the bits are those of the CPU reference.
//
//
// Rows of whole scale groups (k a multiple of the group, the usual case) take a faster form of the same order on the f32
// matrix pipe: see tk_salt_v2_exact_kernel.
// Compiled with -ffp-contract=off; the sums use explicit round-to-nearest adds and multiplies.

#include <type_traits>

#include "tk_device.h"

namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));

// bytes of one plane of `len` coefficients (crates/tritium-format/src/salt_v2.rs:160-258)
__device__ __forceinline__ unsigned plane_bytes(unsigned codec, unsigned len) {
  if (codec == TK_SALT_V2_D2) return (len + 3u) / 4u;
  if (codec == TK_SALT_V2_B3) return (len + 4u) / 5u;
  return ((len + 3u) / 4u * 5u + 7u) / 8u;
}

// trit `local` of a plane whose payload starts at p (salt_v2.rs:289-322,358-392,454-481)
__device__ __forceinline__ int trit_at(const uint8_t *p, unsigned nbytes, unsigned local, unsigned codec) {
  if (codec == TK_SALT_V2_D2) return (int)((gload(p + (local >> 2)) >> ((local & 3u) * 2u)) & 3u) - 1;
  if (codec == TK_SALT_V2_B3) {
    const unsigned place[5] = {1u, 3u, 9u, 27u, 81u};
    return (int)((gload(p + local / 5u) / place[local % 5u]) % 3u) - 1;
  }
  const unsigned bit = (local >> 2) * 5u, byte = bit >> 3;
  unsigned word = gload(p + byte);
  if (byte + 1u < nbytes) word |= (unsigned)gload(p + byte + 1u) << 8;
  const unsigned code = (word >> (bit & 7u)) & 31u, slot = local & 3u, zero = code & 3u;
  if (slot == zero) return 0;
  const unsigned sign = slot - (slot > zero ? 1u : 0u);
  return (code >> (2u + sign)) & 1u ? 1 : -1;
}

// bytes at .. at+N-1 of a plane in the low bits (N = 4 or 8; whatever lies past the plane's end reads as 0). One load that
// stays inside the plane: planes of whole scale groups have at least 10 bytes.
template <typename T>
__device__ __forceinline__ T plane_word(const uint8_t *p, unsigned nbytes, unsigned at) {
  typedef T loose __attribute__((aligned(1)));
  const unsigned from = min(at, nbytes - (unsigned)sizeof(T));
  return *(const TK_GLOBAL loose *)(p + from) >> (8u * (at - from));
}

// the five digits of a B3 byte (below 243) as 2-bit fields, the first trit lowest ((b * 171) >> 9 is b / 3 exactly)
__device__ __forceinline__ unsigned b3_fields(unsigned b) {
  const unsigned q1 = (b * 171u) >> 9, q2 = (q1 * 171u) >> 9, q3 = (q2 * 171u) >> 9, q4 = (q3 * 171u) >> 9;
  return (b - 3u * q1) | ((q1 - 3u * q2) << 2) | ((q2 - 3u * q3) << 4) | ((q3 - 3u * q4) << 6) | (q4 << 8);
}

// trits local .. local+15 of a plane (local a multiple of 16; all 16 lie inside the plane) as 2-bit codes trit + 1, the
// first in the lowest bits, from the plane's bytes `raw` (the first that holds one of them lowest)
__device__ __forceinline__ unsigned long long raw16(const uint8_t *p, unsigned nbytes, unsigned local, unsigned codec) {
  if (codec == TK_SALT_V2_D2) return plane_word<uint32_t>(p, nbytes, local >> 2);
  if (codec == TK_SALT_V2_B3) return plane_word<unsigned long long>(p, nbytes, local / 5u);
  return plane_word<uint32_t>(p, nbytes, (local >> 2) * 5u >> 3);
}
__device__ __forceinline__ unsigned recode16(unsigned long long raw, unsigned local, unsigned codec, const uint16_t *fields) {
  if (codec == TK_SALT_V2_D2) return (unsigned)raw;
  if (codec == TK_SALT_V2_B3) {  // five bytes hold 25 digits, shifted to the first trit wanted
    unsigned long long digits = 0;
#pragma unroll
    for (int i = 0; i < 5; ++i) digits |= (unsigned long long)fields[(unsigned)(raw >> (8 * i)) & 255u] << (10 * i);
    return (unsigned)(digits >> (2u * (local % 5u)));
  }
  // S34: four groups of five bits (local is a multiple of 16: they start at bit 0 or 4 of the first byte). A group is the
  // slot of its zero and the signs of the other three in order: their codes 2 or 0 as three fields, and code 1 put in between
  const unsigned word = (unsigned)raw >> ((local >> 2) * 5u & 7u);
  unsigned codes = 0;
#pragma unroll
  for (int g = 0; g < 4; ++g) {
    const unsigned code = (word >> (5 * g)) & 31u, at = 2u * (code & 3u), below = (1u << at) - 1u;
    const unsigned signs = ((code >> 1) & 2u) | (code & 8u) | ((code << 1) & 32u);
    codes |= ((signs & below) | (1u << at) | ((signs & ~below) << 2)) << (8 * g);
  }
  return codes;
}

// The 4 x 4 transpose over the four 16-lane rows of a wave: register q of row h becomes register h of row q.
__device__ __forceinline__ void transpose_rows(float (&v)[4]) {
  typedef unsigned u2 __attribute__((ext_vector_type(2)));
  auto bits = [](float f) { return __float_as_uint(f); };
  const u2 a = __builtin_amdgcn_permlane32_swap(bits(v[0]), bits(v[2]), false, false);
  const u2 b = __builtin_amdgcn_permlane32_swap(bits(v[1]), bits(v[3]), false, false);
  const u2 e = __builtin_amdgcn_permlane16_swap(a.x, b.x, false, false);
  const u2 o = __builtin_amdgcn_permlane16_swap(a.y, b.y, false, false);
  v[0] = __uint_as_float(e.x);
  v[1] = __uint_as_float(e.y);
  v[2] = __uint_as_float(o.x);
  v[3] = __uint_as_float(o.y);
}

// the value of every 16-lane row of a wave in all of its lanes
__device__ __forceinline__ void spread_rows(unsigned v, unsigned (&rows)[4]) {
  typedef unsigned u2 __attribute__((ext_vector_type(2)));
  const u2 half = __builtin_amdgcn_permlane32_swap(v, v, false, false);  // rows 0 1 0 1 and 2 3 2 3
  const u2 lo = __builtin_amdgcn_permlane16_swap(half.x, half.x, false, false);
  const u2 hi = __builtin_amdgcn_permlane16_swap(half.y, half.y, false, false);
  rows[0] = lo.x;
  rows[1] = lo.y;
  rows[2] = hi.x;
  rows[3] = hi.y;
}

struct TileView {
  unsigned begin, planes, len;
};
__device__ __forceinline__ TileView tile_view(const TkSaltV2 &t, unsigned tile) {
  TileView v;
  v.begin = gload(t.tile_begin + tile);
  v.planes = gload(t.tile_begin + tile + 1) - v.begin;
  const unsigned long long base = (unsigned long long)tile * 256ull;
  v.len = (unsigned)(t.total - base < 256ull ? t.total - base : 256ull);
  return v;
}

__device__ __forceinline__ float f16_to_f32(uint16_t h) {
  _Float16 x;
  __builtin_memcpy(&x, &h, 2);
  return (float)x;  // exact
}

}  // namespace

// LDS: float term[segments][3 planes][tokens], then one plane count per segment.
// Segment boundaries are the multiples of the scale group (which divides the 256 of a tile).
__global__ __launch_bounds__(64) void tk_salt_v2_forward_kernel(TkSaltV2 t, const float *__restrict__ act, unsigned m,
                                                                float *__restrict__ out, unsigned *__restrict__ flag, unsigned call) {
  extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
  constexpr int MT = TK_SALT_V2_TOKENS;
  const unsigned row = blockIdx.x, tok0 = blockIdx.y * MT;
  const unsigned mt = min((unsigned)MT, m - tok0);
  const unsigned long long row_base = (unsigned long long)row * t.k, row_end = row_base + t.k;
  const unsigned long long first = row_base / t.group;
  const unsigned nseg = (unsigned)((row_end + t.group - 1) / t.group - first);
  float *term = (float *)smem;
  uint8_t *seg_planes = smem + (size_t)nseg * 3 * MT * sizeof(float);
  bool bad = false;

  for (unsigned s = threadIdx.x; s < nseg; s += blockDim.x) {
    const unsigned long long lo = max(row_base, (first + s) * t.group), hi = min(row_end, (first + s + 1) * t.group);
    const unsigned tile = (unsigned)(lo >> 8), local = (unsigned)(lo & 255ull), seg = (unsigned)(hi - lo);
    const TileView tv = tile_view(t, tile);
    const unsigned group = local / t.group;
    const unsigned full_bytes = plane_bytes(t.codec, 256u), cur_bytes = plane_bytes(t.codec, tv.len);
    const unsigned full_groups = 256u / t.group, cur_groups = (tv.len + t.group - 1u) / t.group;
    const unsigned col0 = (unsigned)(lo - row_base);
    seg_planes[s] = (uint8_t)tv.planes;
    for (unsigned j = 0; j < tv.planes; ++j) {
      const uint8_t *p = t.payload + (size_t)tv.begin * full_bytes + (size_t)j * cur_bytes;
      float acc[MT];
#pragma unroll
      for (int x = 0; x < MT; ++x) acc[x] = 0.0f;
      for (unsigned o = 0; o < seg; ++o) {
        const int tr = trit_at(p, cur_bytes, local + o, t.codec);
        if (j == 0) {  // every activation of these tokens passes here once per row: the finiteness check
#pragma unroll
          for (int x = 0; x < MT; ++x)
            if ((unsigned)x < mt) bad |= !(fabsf(gload(act + (size_t)(tok0 + x) * t.k + col0 + o)) <= 3.402823466e38f);
        }
        if (tr == 0) continue;
#pragma unroll
        for (int x = 0; x < MT; ++x) {
          if ((unsigned)x >= mt) continue;
          const float a = gload(act + (size_t)(tok0 + x) * t.k + col0 + o);
          acc[x] = tr > 0 ? __fadd_rn(acc[x], a) : __fsub_rn(acc[x], a);
        }
      }
      const float sc = f16_to_f32(gload(t.scales + (size_t)tv.begin * full_groups + (size_t)j * cur_groups + group));
#pragma unroll
      for (int x = 0; x < MT; ++x) term[((size_t)s * 3 + j) * MT + x] = __fmul_rn(acc[x], sc);
    }
  }
  __syncthreads();
  if (threadIdx.x < mt) {
    float accumulator = 0.0f;
    for (unsigned s = 0; s < nseg; ++s)
      for (unsigned j = 0; j < seg_planes[s]; ++j) accumulator = __fadd_rn(accumulator, term[((size_t)s * 3 + j) * MT + threadIdx.x]);
    // an accumulator that left the finite range never comes back (inf - inf is NaN): the end result tells
    bad |= !(fabsf(accumulator) <= 3.402823466e38f);
    out[(size_t)(tok0 + threadIdx.x) * t.n + row] = accumulator;
  }
  if (bad) gstore(flag, call);  // (whoever stores, stores the same)
}

// ---- rows of whole scale groups (k % group == 0) ----
// The fold of one segment over its columns is a chain of adds of +-activation, i.e. of fused multiply-adds with an exact
// product (a trit times a float), and v_mfma_f32_16x16x4_f32 adds its four terms in ascending order with one rounding each,
// denormals kept. So 16 weight rows x 16 tokens fold on the f32 matrix pipe in the pinned order; a zero trit adds +-0, which
// changes no accumulator that started at +0. (A non-finite activation fails the call, so 0 * inf does not count.)
// A workgroup owns 16 rows x 16 tokens; its 16 waves take every sixteenth segment: each lane recodes a quarter of the segment
// of one row to 2-bit codes (whatever the codec), four lanes exchange them, and a step of four columns is one conversion and
// one matrix instruction. The scaled terms of up to SV2_SLOTS segments meet in LDS (as many as fit, so that the waves drift
// apart and one's loads hide behind another's folds), where one thread per output adds them in the pinned order. Plane counts
// differ by tile: a row without a plane folds its last one again and drops the term.
// Floor: the f32 matrix pipe, 32 cycles per 16 x 16 x 4 (7 us at the size below); the recoding and the latency of the loads add
// to it. 4096 x 4096, two planes, kernels, 8 tokens of B3: 64 us (fold with a lane per row, terms through memory) + 12 us
// (their sum) -> 26 us; call, D2 / B3 / S34: 84 / 98 / 93 -> 35 / 37 / 38 us, one token 57 / 69 / 66 -> 33 / 36 / 37, 64 tokens
// 302 / 389 / 353 -> 99 / 109 / 113 (12 us of the first two from the verdict through pinned memory); up to 16 tokens of
// moderate size, whose results need no launch that commits them, 35 / 37 -> 32 / 34 (D2 / B3, 8 tokens). A segment's codes and
// activations requested ahead of the fold before it: 38.8 against 35.5 for B3. With the activations as 32 four-byte loads per
// lane and the codes as single bytes the kernel took 52 us: the loads of 16 rows a few KiB apart were the bound.
constexpr int SV2_WAVES = 16, SV2_SLOTS = 48, SV2_HEAD = 528;
// out (null: not asked for): a call of one block of tokens writes its results there at once if none of its activations exceeds
// SV2_TAME in magnitude, else to tmp, and says so in *spill. With finite scales (the host's condition) results of such
// activations are below 3 k * SV2_TAME * 2^16, which is finite for every k that is staged, and every workgroup reads all
// activations: none can refuse the call once one has written.
constexpr float SV2_TAME = 18446744073709551616.0f;  // 2^64
template <int G>
__global__ __launch_bounds__(SV2_WAVES * 64) void tk_salt_v2_exact_kernel(TkSaltV2 t, const float *__restrict__ act, unsigned m,
                                                                          float *__restrict__ out, float *__restrict__ tmp,
                                                                          unsigned *__restrict__ flag, unsigned call,
                                                                          unsigned *__restrict__ spill, unsigned slots) {
  constexpr int W = G / 64;  // words of sixteen codes per lane and fold
  extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
  uint16_t *s_fields = (uint16_t *)smem;                                   // [256], B3: the digits of a byte
  int *s_three = (int *)(smem + 512), *s_wild = s_three + 1;               // some tile has three planes; some activation is beyond SV2_TAME
  float *s_term = (float *)(smem + SV2_HEAD);                              // [slot][plane][accumulator register][lane]
  uint8_t *s_planes = smem + SV2_HEAD + (size_t)slots * 3 * 256 * sizeof(float);  // [slot][row]
  const unsigned wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63, c = lane & 15, h = lane >> 4;
  const unsigned row = min(blockIdx.x * 16u + c, t.n - 1u), tok0 = blockIdx.y * 16u;
  const unsigned nseg = t.k / G, codec = t.codec;
  const unsigned full_bytes = plane_bytes(codec, 256u);
  const float *arow = act + (size_t)min(tok0 + c, m - 1u) * t.k + h * 4;
  const unsigned final_row = blockIdx.x * 16u + c, final_tok = tok0 + h * 4 + wave;  // of the thread that adds (waves 0..3)
  const size_t final_at = (size_t)min(final_tok, m - 1u) * t.n + min(final_row, t.n - 1u);
  const bool ends = wave < 4 && final_row < t.n && final_tok < m;
  float sum = 0.0f, top = 0.0f;  // (top: the largest magnitude this lane has seen; NaN stays)
  if (threadIdx.x == 0) *s_three = *s_wild = 0;
  if (codec == TK_SALT_V2_B3 && threadIdx.x < 256) s_fields[threadIdx.x] = (uint16_t)b3_fields(threadIdx.x);
  __syncthreads();
  typedef float quad __attribute__((ext_vector_type(4), aligned(4)));
  struct Codes {
    unsigned long long raw[3][W];
    uint16_t scale[3];
    unsigned planes, most, local;
  };
  float a[W * 4][4];  // [sixteen columns][x]: column 4 x + h of the token, after the transpose
  auto request_act = [&](unsigned s) {
#pragma unroll
    for (int w = 0; w < W * 4; ++w) {
      const quad v = *(const TK_GLOBAL quad *)(arow + (size_t)s * G + w * 16);
#pragma unroll
      for (int x = 0; x < 4; ++x) a[w][x] = v[x];
    }
  };
  auto request_codes = [&](unsigned s, Codes &d) {
    const unsigned long long lo = (unsigned long long)row * t.k + (unsigned long long)s * G;
    const unsigned tile = (unsigned)(lo >> 8);
    d.local = (unsigned)(lo & 255ull);
    const TileView tv = tile_view(t, tile);
    const unsigned cur_bytes = plane_bytes(codec, tv.len), cur_groups = tv.len / G;
    const uint8_t *planes = t.payload + (size_t)tv.begin * full_bytes;
    const uint16_t *scales = t.scales + (size_t)tv.begin * (256u / G) + d.local / G;
    d.planes = tv.planes;
    d.most = __ballot(tv.planes >= 3u) ? 3u : (__ballot(tv.planes >= 2u) ? 2u : 1u);
#pragma unroll
    for (int j = 0; j < 3; ++j) {
      if ((unsigned)j >= d.most) break;
      const unsigned jc = min((unsigned)j, tv.planes - 1u);
#pragma unroll
      for (int i = 0; i < W; ++i) d.raw[j][i] = raw16(planes + (size_t)jc * cur_bytes, cur_bytes, d.local + (h * W + i) * 16u, codec);
      d.scale[j] = gload(scales + (size_t)jc * cur_groups);
    }
  };
  for (unsigned s0 = 0; s0 < nseg; s0 += slots) {
    const unsigned pass = min(slots, nseg - s0);
    for (unsigned slot = wave; slot < pass; slot += SV2_WAVES) {
      Codes cur = {};
      request_act(s0 + slot);
      request_codes(s0 + slot, cur);
      const unsigned local = cur.local, most = cur.most;
      if (h == 0) s_planes[slot * 16 + c] = (uint8_t)cur.planes;
      if (most == 3u && lane == 0) *s_three = 1;
#pragma unroll
      for (int x = 0; x < W * 16; ++x) top = __builtin_elementwise_maximum(top, fabsf(a[x / 4][x % 4]));
#pragma unroll
      for (int w = 0; w < W * 4; ++w) transpose_rows(a[w]);
#pragma unroll
      for (int j = 0; j < 3; ++j) {
        if ((unsigned)j >= most) break;
        unsigned words[4 * W];
#pragma unroll
        for (int i = 0; i < W; ++i) {
          unsigned row_words[4];
          spread_rows(recode16(cur.raw[j][i], local + (h * W + i) * 16u, codec, s_fields), row_words);
#pragma unroll
          for (int q = 0; q < 4; ++q) words[q * W + i] = row_words[q];
        }
        f32x4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int w = 0; w < 4 * W; ++w) {  // sixteen columns: the word of lane group w / W; code = trit + 1 in byte x, field h
          const unsigned word = words[w];
          const unsigned trits = (((word >> (2u * h)) & 0x03030303u) + 0x7F7F7F7Fu) ^ 0x80808080u;  // int8 in every byte
#pragma unroll
          for (int x = 0; x < 4; ++x)
            acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a[w][x], (float)(int8_t)(trits >> (8 * x)), acc, 0, 0, 0);
        }
        const float sc = f16_to_f32(cur.scale[j]);
#pragma unroll
        for (int r = 0; r < 4; ++r) s_term[((slot * 3 + j) * 4 + r) * 64 + lane] = __fmul_rn(acc[r], sc);
      }
    }
    if (!(top <= SV2_TAME)) *s_wild = 1;
    __syncthreads();
    if (wave < 4) {
      auto add = [&](auto np_c) {
        constexpr int NP = decltype(np_c)::value;
#pragma unroll 8
        for (unsigned u = 0; u < pass; ++u) {
          const unsigned planes = s_planes[u * 16 + c];
#pragma unroll
          for (int j = 0; j < NP; ++j) {
            const float next = __fadd_rn(sum, s_term[((u * 3 + j) * 4 + wave) * 64 + lane]);  // (what a plane that is not there left is not taken)
            sum = (unsigned)j < planes ? next : sum;
          }
        }
      };
      if (*s_three) add(std::integral_constant<int, 3>{});
      else add(std::integral_constant<int, 2>{});
    }
    __syncthreads();
  }
  const bool wild = *s_wild;
  bool bad = !(top <= 3.402823466e38f);
  if (ends) {
    // an accumulator that left the finite range never comes back (inf - inf is NaN): the end result tells
    bad |= !(fabsf(sum) <= 3.402823466e38f);
    gstore((out && !wild ? out : tmp) + final_at, sum);
  }
  if (out && wild && threadIdx.x == 0) gstore(spill, 1u);
  if (bad) gstore(flag, call);  // (whoever stores, stores the same)
}

// The results leave the staging buffer only when no activation and no result was found non-finite: the flag then holds the
// number of an earlier call (so it is never cleared). *verdict, in host memory, says which it was. Without a flag (the host has
// looked): always.
__global__ __launch_bounds__(TK_WG) void tk_salt_v2_commit_kernel(const float *__restrict__ tmp, float *__restrict__ out, size_t count,
                                                                  const unsigned *__restrict__ flag, unsigned call,
                                                                  unsigned *__restrict__ verdict) {
  const bool bad = flag && gload(flag) == call;
  const size_t idx = (size_t)blockIdx.x * TK_WG + threadIdx.x;
  if (flag && idx == 0) gstore(verdict, bad ? 1u : 0u);
  if (!bad && idx < count) gstore(out + idx, gload(tmp + idx));
}

// One thread per gathered coefficient (crates/tritium-cuda/kernels/salt_v2.cu:218-304).
__global__ __launch_bounds__(TK_WG) void tk_salt_v2_gather_kernel(TkSaltV2 t, const uint32_t *__restrict__ rows, size_t count,
                                                                  float *__restrict__ out) {
  const size_t idx = (size_t)blockIdx.x * TK_WG + threadIdx.x;
  if (idx >= count * t.k) return;
  const size_t sel = idx / t.k;
  const unsigned col = (unsigned)(idx - sel * t.k);
  const unsigned long long c = (unsigned long long)gload(rows + sel) * t.k + col;
  const unsigned tile = (unsigned)(c >> 8), local = (unsigned)(c & 255ull);
  const TileView tv = tile_view(t, tile);
  const unsigned full_bytes = plane_bytes(t.codec, 256u), cur_bytes = plane_bytes(t.codec, tv.len);
  const unsigned full_groups = 256u / t.group, cur_groups = (tv.len + t.group - 1u) / t.group, group = local / t.group;
  float acc = 0.0f;
  for (unsigned j = 0; j < tv.planes; ++j) {
    const int tr = trit_at(t.payload + (size_t)tv.begin * full_bytes + (size_t)j * cur_bytes, cur_bytes, local, t.codec);
    const float sc = f16_to_f32(gload(t.scales + (size_t)tv.begin * full_groups + (size_t)j * cur_groups + group));
    if (tr > 0) acc = __fadd_rn(acc, sc);
    else if (tr < 0) acc = __fsub_rn(acc, sc);
  }
  out[idx] = acc;
}

size_t tk_salt_v2_lds_bytes(size_t k, size_t group) {
  const size_t nseg = k / group + 2;  // a row that starts and ends inside a group touches two more
  return nseg * 3 * TK_SALT_V2_TOKENS * sizeof(float) + ((nseg + 15) & ~(size_t)15);
}

bool tk_salt_v2_direct(const TkSaltV2 &t, size_t m) { return t.k && t.k % t.group == 0 && m <= 16; }

hipError_t tk_launch_salt_v2_forward(hipStream_t s, const TkSaltV2 &t, const float *act, size_t m, float *out, float *tmp, unsigned *flag,
                                     unsigned call, unsigned *spill) {
  if (!m || !t.n) return hipSuccess;
  if (out && !tk_salt_v2_direct(t, m)) return hipErrorInvalidValue;
  if (t.k && t.k % t.group == 0) {
    const dim3 grid((t.n + 15) / 16, (unsigned)((m + 15) / 16)), block(SV2_WAVES * 64);
    const unsigned nseg = t.k / t.group, slots = nseg < SV2_SLOTS ? nseg : SV2_SLOTS;
    const size_t lds = SV2_HEAD + (size_t)slots * (3 * 256 * sizeof(float) + 16);
    if (lds > 64 * 1024) {
      const hipError_t e = tk_raise_lds_limit(t.group == 128 ? (const void *)tk_salt_v2_exact_kernel<128> : (const void *)tk_salt_v2_exact_kernel<64>, 160 * 1024);
      if (e != hipSuccess) return e;
    }
    if (t.group == 128) hipLaunchKernelGGL(tk_salt_v2_exact_kernel<128>, grid, block, lds, s, t, act, (unsigned)m, out, tmp, flag, call, spill, slots);
    else hipLaunchKernelGGL(tk_salt_v2_exact_kernel<64>, grid, block, lds, s, t, act, (unsigned)m, out, tmp, flag, call, spill, slots);
    return hipGetLastError();
  }
  const size_t lds = tk_salt_v2_lds_bytes(t.k, t.group);
  if (lds > 64 * 1024) {
    const hipError_t e = tk_raise_lds_limit((const void *)tk_salt_v2_forward_kernel, 160 * 1024);
    if (e != hipSuccess) return e;
  }
  const dim3 grid(t.n, (unsigned)((m + TK_SALT_V2_TOKENS - 1) / TK_SALT_V2_TOKENS));
  hipLaunchKernelGGL(tk_salt_v2_forward_kernel, grid, dim3(64), lds, s, t, act, (unsigned)m, tmp, flag, call);
  return hipGetLastError();
}

hipError_t tk_launch_salt_v2_commit(hipStream_t s, const float *tmp, float *out, size_t count, const unsigned *flag, unsigned call,
                                    unsigned *verdict) {
  if (!count) return hipSuccess;
  hipLaunchKernelGGL(tk_salt_v2_commit_kernel, dim3((unsigned)((count + TK_WG - 1) / TK_WG)), dim3(TK_WG), 0, s, tmp, out, count, flag, call, verdict);
  return hipGetLastError();
}

hipError_t tk_launch_salt_v2_gather(hipStream_t s, const TkSaltV2 &t, const uint32_t *rows, size_t count, float *out) {
  const size_t total = count * t.k;
  if (!total) return hipSuccess;
  hipLaunchKernelGGL(tk_salt_v2_gather_kernel, dim3((unsigned)((total + TK_WG - 1) / TK_WG)), dim3(TK_WG), 0, s, t, rows, count, out);
  return hipGetLastError();
}
