// pk_gemm_f32.hip - fused palette-weight GEMM with f32 operands for gfx950:
// the FP32 twin of pk_gemm_f16.hip (reference:
// src/webgpu/kernels/gemm.ts:2356-2599, epilogue :2847-2869).
//
// The f32 matrix units are 16 times slower than the bf16 ones, so every f32
// operand is split into three bf16 terms that add up to it exactly, and six
// of the nine products of terms go through v_mfma_f32_32x32x16_bf16 into one
// f32 accumulator, smallest first; the three left out are below 2^-24 of the
// product. bf16 has the exponents of f32 but not the 16 bits below them that
// the second and third term of an operand under 2^-110 need, so both operands
// are multiplied by 2^24 before the split and the sum by 2^-48 after it:
// every term down to the last bit of the smallest subnormal f32 is then a
// normal bf16. Operands from 2^104 and sums from 2^80 on overflow instead and
// come from the f32 units, output by output. The sums are nearer to 64 bits
// than the f32 units' (norm-wise 4.8e-7 against 5.7e-7 at K = 1024, 9.6e-7
// against 1.1e-6 at K = 4096, 2.4e-7 and 4.8e-7 with K over four waves). The
// unit rounds its sums down, though, and half of that error was one offset for
// all outputs, which attention's average over the keys keeps while it averages
// the rest away (context of 4 x 253 frames 9.1e-7 against 7.3e-7 before); with
// half of the K blocks subtracted the offset is gone (6.2e-7) at 4-6% of the
// time.
//
// Bound: the bf16 matrix units in principle (a sixth of their rate: 417
// TFLOP/s nominal, about 190 at the rate of a large library product), LDS
// reads and the per-step chain in practice. A wave's operands for the next
// 16 k are gathered and read during the products of the current ones, the A
// tile is split once per workgroup on its way into a ring of three LDS
// buffers (32 k each, one barrier per step), and all loads are unconditional
// (a branch around one ends the compiler's scheduling region: 24.3 -> 20.6 us
// at 188 x 1024 -> 4096). The palette lies in LDS as split entries: one 8-byte
// gather per code and three byte permutes per pair.
//
// Against v_mfma_f32_32x32x2_f32 before: 3008 x 1024 -> 4096 (5-bit) 214 ->
// 130 us (194 TFLOP/s), 3008 x 4096 -> 1024 227 -> 143, 3008 x 1024 -> 3072 168
// -> 102, 256 x 1024 -> 4096 (6-bit) 30.5 -> 21.7, 188 x 4096 -> 1024 102 -> 28,
// 16 x 1024 -> 4096 28 -> 10.
//
// Codes in operand order: lane half h owns k = 64 kb + 32 h + u, so MFMA
// sub-step s (0..3) multiplies codes u = 8 s + [0, 8) of both halves.
#include "pk_internal.h"

namespace pk {
namespace {

typedef float float16v __attribute__((ext_vector_type(16)));
typedef float float2v __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

template <int BITS>
__device__ __forceinline__ uint32_t lane_code(const uint32_t* w, int u) {
  constexpr uint32_t mask = (1u << BITS) - 1u;
  const int bit = u * BITS;
  const int word = bit >> 5;
  const int shift = bit & 31;
  if (shift + BITS <= 32) return (w[word] >> shift) & mask;
  return __builtin_amdgcn_alignbit(w[word + 1], w[word], shift) & mask;
}

// SiLU of the reference epilogue, v / (1 + exp(-clamp(v, -20, 20)))
// (gemm.ts:2847-2869 with the activation of :2006-2044): clamp, exp as
// v_exp_f32 of the base-2 argument and v_rcp_f32, each within ~1 ulp.
__device__ __forceinline__ float silu(float v) {
  const float bounded = __builtin_amdgcn_fmed3f(v, -20.0f, 20.0f);
  const float e = __builtin_amdgcn_exp2f(bounded * -1.4426950408889634f);
  return v * __builtin_amdgcn_rcpf(1.0f + e);
}

// Two f32 values rounded to bf16, the first in the low half.
__device__ __forceinline__ uint32_t pack_bf16(float a, float b) {
  const bf16x2 p = __builtin_convertvector((float2v{a, b}), bf16x2);
  return __builtin_bit_cast(uint32_t, p);
}
__device__ __forceinline__ float low_f32(uint32_t p) { return __uint_as_float(p << 16); }
__device__ __forceinline__ float high_f32(uint32_t p) { return __uint_as_float(p & 0xffff0000u); }

constexpr float kOperandScale = 0x1p24f, kSumScale = 0x1p-48f;

// Two scaled f32 values as three bf16 terms each, rounded to nearest one
// after the other: the sum of the three is the value (8 + 8 + 8 significand
// bits, and no term below the smallest normal bf16).
struct Split {
  uint32_t hi, mid, lo;
};
__device__ __forceinline__ Split split2(float a, float b) {
  Split s;
  s.hi = pack_bf16(a, b);
  const float ra = a - low_f32(s.hi), rb = b - high_f32(s.hi);
  s.mid = pack_bf16(ra, rb);
  s.lo = pack_bf16(ra - low_f32(s.mid), rb - high_f32(s.mid));
  return s;
}

template <int BITS, int WN, int MB, int NB, int KS>
__global__ __launch_bounds__(64 * WN * KS, 2) void gemm_f32_kernel(GemmArgs args) {
  static_assert(KS == 1 || (WN == 1 && MB == 1 && NB == 1 && KS == 4), "K over the four waves of one 32 x 32 tile");
  constexpr int T = 64 * WN * KS;  // threads, GT of them share a K block
  constexpr int GT = T / KS;
  constexpr int BM = 32 * MB;
  constexpr int BN = 32 * WN * NB;
  constexpr int E = 1 << BITS;
  constexpr int LUT_CAP = (BN / 16 + 2) * E;
  constexpr int PLANE = BM * 64;  // bytes of one term of a step's A tile: 32 k per row
  constexpr int CH = BM * 8 / GT;  // runs of 4 k per thread
  static_assert(BM * 8 % GT == 0, "the A tile divides evenly");

  __shared__ __align__(16) uint8_t a_lds_all[KS][3][3 * PLANE];
  __shared__ uint2 lut_lds[2 * LUT_CAP];  // {hi | mid << 16, lo}, then the same negated

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = tid >> 6;
  const int wave_n = KS > 1 ? 0 : wave;
  const uint32_t part = KS > 1 ? wave : 0;  // this wave's K blocks: part, part + KS, ...
  const int gtid = KS > 1 ? lane : tid;
  auto& a_lds = a_lds_all[part];
  const int j = lane & 31;
  const int h = lane >> 5;

  const uint32_t M = args.rows;
  const uint32_t K = args.inner;
  const uint32_t N = args.columns;
  const uint32_t k_blocks = (K + 63u) / 64u;
  const uint32_t n_blocks_total = (N + 31u) / 32u;
  const uint32_t n0 = blockIdx.x * BN;
  const uint32_t m0 = blockIdx.y * BM;

  const uint32_t gc = args.palette_group_columns;
  const uint32_t G = args.palette_groups;
  const uint32_t g_lo = min(n0 / gc, G - 1u);
  const uint32_t g_hi = min((min(n0 + BN, N) - 1u) / gc, G - 1u);
  const float* palette = static_cast<const float*>(args.palette);

  const uint32_t nb0 = n0 / 32u + wave_n * NB;
  uint32_t cw[NB][BITS];
  auto load_codes = [&](uint32_t kb, uint32_t (&dst)[NB][BITS]) {
#pragma unroll
    for (int ni = 0; ni < NB; ++ni) {
      const uint32_t nb = min(nb0 + ni, n_blocks_total - 1u);  // past the end: columns never stored
      const uint32_t* blk = args.codes + ((uint64_t)nb * k_blocks + kb) * block_words(BITS);
      const uint4 p0 = reinterpret_cast<const uint4*>(blk)[lane];
      dst[ni][0] = p0.x;
      dst[ni][1] = p0.y;
      dst[ni][2] = p0.z;
      dst[ni][3] = p0.w;
      if constexpr (BITS == 5) {
        dst[ni][4] = blk[256 + lane];
      } else {
        const uint2 p1 = reinterpret_cast<const uint2*>(blk + 256)[lane];
        dst[ni][4] = p1.x;
        dst[ni][5] = p1.y;
      }
    }
  };

  // Step t = 2 kb + half: the k of MFMA sub-steps 2 half and 2 half + 1, i.e.
  // 64 kb + 32 h + 16 half + [0, 16) for both lane halves h, as eight runs of
  // four per row. Loads are unconditional: a row past the end repeats the
  // last one (never stored), a run past K is zeroed.
  const float* a_ptr = static_cast<const float*>(args.a);
  const uint32_t own_blocks = k_blocks > part ? (k_blocks - part + KS - 1u) / KS : 0u;
  const uint32_t steps = 2u * own_blocks;
  float4 a_stage[2][CH];
  auto run_k = [&](uint32_t t, int run) {
    return ((t >> 1) * KS + part) * 64u + (t & 1u) * 16u + ((run >> 2) * 32 + (run & 3) * 4);
  };
  auto load_a = [&](uint32_t t, float4 (&stage)[CH]) {
#pragma unroll
    for (int c = 0; c < CH; ++c) {
      const int idx = gtid + c * GT;
      const uint32_t m = min(m0 + (idx >> 3), M - 1u);
      const uint32_t k = min(run_k(t, idx & 7), K - 4u);
      stage[c] = *reinterpret_cast<const float4*>(a_ptr + (uint64_t)m * K + k);
    }
  };
  auto scale_a = [&](uint32_t t, float4 (&stage)[CH]) {
#pragma unroll
    for (int c = 0; c < CH; ++c) {
      const float scale = run_k(t, (gtid + c * GT) & 7) < K ? kOperandScale : 0.0f;
      stage[c] = make_float4(stage[c].x * scale, stage[c].y * scale, stage[c].z * scale, stage[c].w * scale);
    }
  };
  // A row of a term is 64 bytes, chunk 2 s + h of 16 for sub-step s and lane
  // half h; rows four apart start at the same bank, so the chunk is XORed
  // with bits 2 and 3 of the row.
  auto store_a = [&](uint32_t buf, const float4 (&stage)[CH]) {
#pragma unroll
    for (int c = 0; c < CH; ++c) {
      const int idx = gtid + c * GT;
      const int r = idx >> 3, run = idx & 7;
      const float4 x = stage[c];
      const Split s0 = split2(x.x, x.y);
      const Split s1 = split2(x.z, x.w);
      const int chunk = ((run >> 1) & 1) * 2 + (run >> 2);
      uint8_t* dst = &a_lds[buf][r * 64 + ((chunk ^ ((r >> 2) & 3)) << 4) + (run & 1) * 8];
      *reinterpret_cast<uint2*>(dst) = make_uint2(s0.hi, s1.hi);
      *reinterpret_cast<uint2*>(dst + PLANE) = make_uint2(s0.mid, s1.mid);
      *reinterpret_cast<uint2*>(dst + 2 * PLANE) = make_uint2(s0.lo, s1.lo);
    }
  };

  float16v acc[MB][NB];
#pragma unroll
  for (int mi = 0; mi < MB; ++mi)
#pragma unroll
    for (int ni = 0; ni < NB; ++ni)
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[mi][ni][v] = 0.0f;

  if (steps) {
    load_a(0, a_stage[0]);
    load_codes(part, cw);
    load_a(1, a_stage[1]);
  }
  {
    const uint32_t entries = (g_hi - g_lo + 1u) * E;
    for (uint32_t i = tid; i < entries; i += T) {
      const Split s = split2(palette[(uint64_t)g_lo * E + i] * kOperandScale, 0.0f);
      const uint2 e = make_uint2((s.hi & 0xffffu) | s.mid << 16, s.lo & 0xffffu);
      lut_lds[i] = e;
      lut_lds[LUT_CAP + i] = make_uint2(e.x ^ 0x80008000u, e.y ^ 0x8000u);
    }
  }
  uint32_t lut_base[NB];  // first entry of the lane's column's palette group
#pragma unroll
  for (int ni = 0; ni < NB; ++ni) {
    const uint32_t n = n0 + (wave_n * NB + ni) * 32 + j;
    lut_base[ni] = (min(min(n / gc, G - 1u), g_hi) - g_lo) * E;
  }
  // Weights of a sub-step: the entries of its eight codes per column block,
  // then the three operands.
  auto gather = [&](const uint32_t (&c)[NB][BITS], int sub, uint32_t sign, uint2 (&e)[NB][8]) {
#pragma unroll
    for (int ni = 0; ni < NB; ++ni)
#pragma unroll
      for (int u = 0; u < 8; ++u) e[ni][u] = lut_lds[lut_base[ni] + sign + lane_code<BITS>(c[ni], sub * 8 + u)];
  };
  auto assemble = [&](const uint2 (&e)[NB][8], bf16x8 (&w)[NB][3]) {
#pragma unroll
    for (int ni = 0; ni < NB; ++ni) {
      uint32_t hi[4], mid[4], lo[4];
#pragma unroll
      for (int p = 0; p < 4; ++p) {
        const uint2 e0 = e[ni][2 * p], e1 = e[ni][2 * p + 1];
        hi[p] = __builtin_amdgcn_perm(e1.x, e0.x, 0x05040100u);
        mid[p] = __builtin_amdgcn_perm(e1.x, e0.x, 0x07060302u);
        lo[p] = __builtin_amdgcn_perm(e1.y, e0.y, 0x05040100u);
      }
      w[ni][0] = __builtin_bit_cast(bf16x8, make_uint4(hi[0], hi[1], hi[2], hi[3]));
      w[ni][1] = __builtin_bit_cast(bf16x8, make_uint4(mid[0], mid[1], mid[2], mid[3]));
      w[ni][2] = __builtin_bit_cast(bf16x8, make_uint4(lo[0], lo[1], lo[2], lo[3]));
    }
  };
  auto read_a = [&](uint32_t buf, int s, bf16x8 (&a)[MB][3]) {
#pragma unroll
    for (int mi = 0; mi < MB; ++mi) {
      const int r = mi * 32 + j;
      const uint8_t* src = &a_lds[buf][r * 64 + (((2 * s + h) ^ ((r >> 2) & 3)) << 4)];
#pragma unroll
      for (int q = 0; q < 3; ++q) a[mi][q] = *reinterpret_cast<const bf16x8*>(src + q * PLANE);
    }
  };
  // the smallest products first
  auto multiply = [&](const bf16x8 (&w)[NB][3], const bf16x8 (&a)[MB][3]) {
    constexpr int kTerms[6][2] = {{2, 0}, {0, 2}, {1, 1}, {1, 0}, {0, 1}, {0, 0}};
#pragma unroll
    for (int t = 0; t < 6; ++t)
#pragma unroll
      for (int mi = 0; mi < MB; ++mi)
#pragma unroll
        for (int ni = 0; ni < NB; ++ni)
          acc[mi][ni] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(w[ni][kTerms[t][0]], a[mi][kTerms[t][1]], acc[mi][ni],
                                                               0, 0, 0);
  };

  // A wave that has a K block to itself needs no barrier: its LDS operations
  // complete in order.
  auto sync = [&] {
    if constexpr (KS == 1) {
      __syncthreads();
    } else {
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      __builtin_amdgcn_wave_barrier();
    }
  };
  if constexpr (KS > 1) __syncthreads();  // the palette
  if (steps) {
    scale_a(0, a_stage[0]);
    scale_a(1, a_stage[1]);
    store_a(0, a_stage[0]);
    load_a(min(2u, steps - 1u), a_stage[0]);
    store_a(1, a_stage[1]);
    load_a(min(3u, steps - 1u), a_stage[1]);
    sync();

    // Step t multiplies buffer t % 3 while t + 1 is read for its first
    // sub-step and t + 2 is written; each sub-step's operands are fetched
    // during the products of the one before.
    bf16x8 w[NB][3], a0[MB][3], a1[MB][3];
    uint2 e[NB][8];
    uint32_t buf = 0;
    // The matrix unit rounds its sums down, not to nearest: a bias that the
    // average over many outputs (attention over its keys) would show whole.
    // So half of the runs of blocks (two, or one of a K part or of K <= 128)
    // are subtracted: negated weights into the negated sum, whose roundings
    // then go up. The order + - - + - + + - (the parity of the run's bits)
    // takes out the growth of the sum along K as well, and the K parts begin
    // with signs in that order. Mean offset, in units of the mean magnitude:
    // 1e-8 without (K = 128) -> 1.3e-9, K = 1024 -7e-10 (every second run
    // 4.0e-9, the f32 units -1.0e-9), K = 4096 2.7e-9 (8.1e-9, -2.0e-9). One
    // block (K <= 64) has nothing to alternate with and keeps -9e-9, a tenth of
    // its error; changing sign between its halves left -3.5e-9 and cost 64 x
    // 128 tiles 3% at every K.
    const uint32_t run_shift = KS == 1 && own_blocks > 2u ? 1u : 0u;
    const uint32_t first = KS > 1 ? (uint32_t)__popc(__builtin_amdgcn_readfirstlane((int)part)) : 0u;
    auto sign_of = [&](uint32_t i) { return (((uint32_t)__popc(i >> run_shift) + first) & 1u) * (uint32_t)LUT_CAP; };
    gather(cw, 0, sign_of(0), e);
    read_a(0, 0, a0);
    assemble(e, w);
    auto negate = [&] {
#pragma unroll
      for (int mi = 0; mi < MB; ++mi)
#pragma unroll
        for (int ni = 0; ni < NB; ++ni)
#pragma unroll
          for (int v = 0; v < 16; ++v) acc[mi][ni][v] = -acc[mi][ni][v];
    };
    for (uint32_t i = 0; i < own_blocks; ++i) {
      const uint32_t sign = sign_of(i), next_sign = sign_of(i + 1u);
      uint32_t cn[NB][BITS];
      load_codes(min(i + 1u, own_blocks - 1u) * KS + part, cn);
#pragma unroll
      for (int half = 0; half < 2; ++half) {
        const uint32_t t = 2u * i + half;
        const uint32_t buf1 = buf == 2u ? 0u : buf + 1u, buf2 = buf1 == 2u ? 0u : buf1 + 1u;
        gather(cw, 2 * half + 1, sign, e);
        read_a(buf, 1, a1);
        multiply(w, a0);
        // ahead of the split, whose chain a wave alone on its SIMD waits for
        // (96 x 128, 512 x 4096 -> 1024: 122.7 us, 127.0 inside it), but not
        // with one row block (6-bit 256 x 1024 -> 1024 21.3 us, 20.3 inside)
        const uint32_t next = min(t + 2u, steps - 1u);
        if constexpr (MB > 1) scale_a(next, a_stage[half]);
        assemble(e, w);
        if (half == 0)
          gather(cw, 2, sign, e);
        else
          gather(cn, 0, next_sign, e);
        // three row blocks: the split of the new rows first (3008 x 4096 -> 1024
        // 143 us against 146; 32 x 128 and 64 x 256 lose 2% and 10% that way)
        if constexpr (MB < 3) read_a(buf1, 0, a0);
        if constexpr (MB == 1) scale_a(next, a_stage[half]);
        store_a(buf2, a_stage[half]);
        load_a(min(t + 4u, steps - 1u), a_stage[half]);
        if constexpr (MB >= 3) read_a(buf1, 0, a0);
        multiply(w, a1);
        assemble(e, w);
        sync();
        buf = buf1;
      }
#pragma unroll
      for (int ni = 0; ni < NB; ++ni)
#pragma unroll
        for (int q = 0; q < BITS; ++q) cw[ni][q] = cn[ni][q];
      if (i + 1u < own_blocks ? sign != next_sign : sign != 0u) negate();
    }
  }

  // A value that is infinite, NaN or past the largest bf16 once scaled has no
  // split: its rows or columns come out as NaN or infinity, as a scaled sum
  // that overflows does. A wave that finds one computes its blocks again on
  // the f32 units, one code and one element of A per lane and MFMA, and takes
  // the outputs that are not finite from there: which sum an output gets
  // depends on its own row and column alone.
  auto is_finite = [](float x) { return __builtin_fabsf(x) <= 3.402823466e+38f; };
  bool finite = true;
#pragma unroll
  for (int mi = 0; mi < MB; ++mi)
#pragma unroll
    for (int ni = 0; ni < NB; ++ni)
#pragma unroll
      for (int v = 0; v < 16; ++v) {
        acc[mi][ni][v] *= kSumScale;
        finite &= is_finite(acc[mi][ni][v]);
      }
  if (!__all(finite)) {
#pragma unroll 1
    for (int ni = 0; ni < NB; ++ni) {
      const uint32_t n = n0 + (wave_n * NB + ni) * 32 + j;
      const float* lut = palette + (uint64_t)min(n / gc, G - 1u) * E;
      const uint32_t nb = min(nb0 + ni, n_blocks_total - 1u);
#pragma unroll 1
      for (int mi = 0; mi < MB; ++mi) {
        const uint32_t m = m0 + mi * 32 + j;
        float16v c;
        for (int v = 0; v < 16; ++v) c[v] = 0.0f;
        for (uint32_t kb = part; kb < k_blocks; kb += KS) {
          const uint32_t* blk = args.codes + ((uint64_t)nb * k_blocks + kb) * block_words(BITS);
          uint32_t words[BITS + 1];
          for (int q = 0; q < 4; ++q) words[q] = blk[lane * 4 + q];
          for (int q = 4; q < BITS; ++q) words[q] = blk[256 + lane * (BITS - 4) + q - 4];
          words[BITS] = 0u;
#pragma unroll
          for (int s = 0; s < 32; ++s) {
            const uint32_t k = kb * 64u + h * 32u + s;
            const float x = m < M && k < K ? a_ptr[(uint64_t)m * K + k] : 0.0f;
            c = __builtin_amdgcn_mfma_f32_32x32x2f32(lut[lane_code<BITS>(words, s)], x, c, 0, 0, 0);
          }
        }
#pragma unroll
        for (int i = 0; i < MB; ++i)
#pragma unroll
          for (int o = 0; o < NB; ++o)
#pragma unroll
            for (int v = 0; v < 16; ++v)
              if (i == mi && o == ni && !is_finite(acc[i][o][v])) acc[i][o][v] = c[v];
      }
    }
  }

  if constexpr (KS > 1) {
    // The parts meet in LDS; wave q sums quad q of every column block in part
    // order.
    __syncthreads();
    float4* partial = reinterpret_cast<float4*>(a_lds_all);
#pragma unroll
    for (int q = 0; q < 4; ++q)
      partial[(wave * 4 + q) * 64 + lane] =
          make_float4(acc[0][0][4 * q], acc[0][0][4 * q + 1], acc[0][0][4 * q + 2], acc[0][0][4 * q + 3]);
    __syncthreads();
    float4 sum = partial[wave * 64 + lane];
#pragma unroll
    for (int p = 1; p < KS; ++p) {
      const float4 v = partial[(p * 4 + wave) * 64 + lane];
      sum.x += v.x;
      sum.y += v.y;
      sum.z += v.z;
      sum.w += v.w;
    }
    acc[0][0][0] = sum.x;
    acc[0][0][1] = sum.y;
    acc[0][0][2] = sum.z;
    acc[0][0][3] = sum.w;
  }

  float* out = static_cast<float*>(args.out);
  const float* residual = static_cast<const float*>(args.residual);
#pragma unroll
  for (int mi = 0; mi < MB; ++mi) {
    const uint32_t m = m0 + mi * 32 + j;
    if (m >= M) continue;
#pragma unroll
    for (int ni = 0; ni < NB; ++ni) {
      const uint32_t nbase = n0 + (wave_n * NB + ni) * 32 + h * 4;
#pragma unroll
      for (int q = 0; q < (KS > 1 ? 1 : 4); ++q) {
        const uint32_t n = nbase + (KS > 1 ? wave : q) * 8;
        if (n >= N) continue;
        float v[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = acc[mi][ni][q * 4 + e];
        if (args.bias) {
          const float4 b = *reinterpret_cast<const float4*>(args.bias + n);
          v[0] += b.x;
          v[1] += b.y;
          v[2] += b.z;
          v[3] += b.w;
        }
        if (args.activation == kActSilu) {
#pragma unroll
          for (int e = 0; e < 4; ++e) v[e] = silu(v[e]);
        } else if (args.activation == kActRelu) {
#pragma unroll
          for (int e = 0; e < 4; ++e) v[e] = fmaxf(v[e], 0.0f);
        }
        const uint64_t at = (uint64_t)m * N + n;
        if (residual) {
          const float4 r = *reinterpret_cast<const float4*>(residual + at);
          v[0] = r.x + args.residual_scale * v[0];
          v[1] = r.y + args.residual_scale * v[1];
          v[2] = r.z + args.residual_scale * v[2];
          v[3] = r.w + args.residual_scale * v[3];
        }
        *reinterpret_cast<float4*>(out + at) = make_float4(v[0], v[1], v[2], v[3]);
      }
    }
  }
}

struct Variant {
  TileShape shape;
  const char* name5;
  const char* name6;
  void (*kernel5)(GemmArgs);
  void (*kernel6)(GemmArgs);
};

#define PK_F32_VARIANT(WN, MB, NB, KS)                                                                 \
  Variant {                                                                                            \
    TileShape{1, WN, MB, NB, KS}, "pk_gemm_f32_b5_n" #WN "k" #KS "_m" #MB "n" #NB,                   \
        "pk_gemm_f32_b6_n" #WN "k" #KS "_m" #MB "n" #NB, gemm_f32_kernel<5, WN, MB, NB, KS>, \
        gemm_f32_kernel<6, WN, MB, NB, KS>                                                          \
  }

const Variant kVariants[] = {
    PK_F32_VARIANT(4, 1, 1, 1),  // 32 x 128
    PK_F32_VARIANT(4, 2, 1, 1),  // 64 x 128
    PK_F32_VARIANT(4, 3, 1, 1),  // 96 x 128
    PK_F32_VARIANT(4, 2, 2, 1),  // 64 x 256
    PK_F32_VARIANT(1, 1, 1, 4),  // 32 x 32, K over four waves
};

}  // namespace

int f32_variant_count() { return (int)(sizeof(kVariants) / sizeof(kVariants[0])); }
TileShape f32_variant(int index) { return kVariants[index].shape; }
const char* f32_variant_name(int bits, int index) {
  return bits == 5 ? kVariants[index].name5 : kVariants[index].name6;
}

GemmKernel f32_kernel(int bits, int variant) {
  return bits == 5 ? kVariants[variant].kernel5 : kVariants[variant].kernel6;
}

hipError_t launch_gemm_f32(int bits, int variant, const GemmArgs& args, hipStream_t stream, hipEvent_t start,
                           hipEvent_t stop) {
  const Variant& v = kVariants[variant];
  const uint32_t n_pad = padded_columns(args.columns);
  const dim3 grid((n_pad + v.shape.tile_columns() - 1) / v.shape.tile_columns(),
                  (args.rows + v.shape.tile_rows() - 1) / v.shape.tile_rows());
  if (grid.y == 0) return hipSuccess;
  return launch_timed(f32_kernel(bits, variant), grid, dim3(v.shape.threads()), stream, start, stop, args);
}

}  // namespace pk
