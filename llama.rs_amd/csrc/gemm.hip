// gemm.hip — batched prefill products on int8 MFMA (ops.rs:150-313 with
// RUST_LLAMA_BATCH_INT=1: quantize_q8 of every token, then dot_qk_q8_row per
// (row, token), simd.rs:898-910).
//
// Exactness: for every (token, row) the output is the reference's f32 chain
// `total += term` over the row's terms in index order; each term is formed
// with the reference's expression (simd.rs:581 Q4_K, 663 Q6_K, 863 Q4_0,
// 891 Q8_0). The integer block dots inside the terms come from int8 MFMA and
// are exact. Three identities keep work off the VALU, whose f32 combine is
// what bounds these kernels; none of them changes a rounding:
//   * the MFMA starts from kBase, the bits of an f32 in the middle of its
//     binade, so its i32 result read as f32 is that f32 + dot * 2^-26
//     (|dot| < 2^21), and one f32 subtraction gives dot * 2^-26 exactly; the
//     power of two goes into the row's scale. A v_sub_f32 issues every 2.3
//     cycles per SIMD (two waves or more ready), a v_cvt_f32_i32 every 4.1;
//   * Q6_K and Q4_0 weights enter the MFMA as 4 q and 16 q (the bit field
//     moved to the top of its byte, the sign bit flipped), and their scale is
//     a quarter or a sixteenth: powers of two, exact on both sides;
//   * Q4_K's dmin*m * sum products are a rank-1 product, one f32 MFMA of
//     depth 1 from C = 0 (each result is the product rounded once).
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "gemm.h"
#include "rlh_device.h"

namespace rlh {

namespace {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v16i __attribute__((ext_vector_type(16)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));
typedef float f32x16_t __attribute__((ext_vector_type(16)));
typedef float f32x32_t __attribute__((ext_vector_type(32)));
typedef RLH_LDS uint8_t lbyte;

// The MFMA's C operand: an inline constant of the instruction set, 1 / (2 pi)
// as f32, taken as an integer; kBaseF is its value and 2^-26 its unit.
constexpr int kBase = 0x3e22f983;
constexpr float kBaseF = 0x1.45f306p-3f, kUnit = 67108864.0f;  // 2^26

// Shape of a block. Four waves, 2 token waves x 2 row waves; a wave computes
// a tile of MT tokens x MT rows (MT = the MFMA's edge), tokens in the result
// registers, rows across the lanes.
//   MT 32: 64 tokens x 64 rows per block, stages of half a super-block (128
//          values of the columns), two of them;
//   MT 16: 32 tokens x 32 rows per block, four stages of a super-block (few
//          blocks per CU: the copies run further ahead).
// A stage is copied into LDS by DMA, half by half: the activation tiles'
// quants, scales and sums as they lie in memory (Q8Tiles), the weight rows'
// 16-byte chunks as [chunk][row], and Q6_K's f16 d in its 4-byte word. Half
// super-blocks and at most 128 registers because four MT 32 blocks then fit
// a CU: a SIMD issues f32 adds and multiplies of two waves side by side (2.3
// cycles each, 4.6 when one wave is ready), and with four waves per SIMD two
// are ready most of the time (Q8_0, 24576 x 4096 x 512 tokens: 234 us with
// whole super-blocks and two blocks per CU, 194 with four).
template <uint32_t TY, int MT>
struct Geo {
  static constexpr bool kSums = TY == RLH_TYPE_Q4_K;
  static constexpr uint32_t kActTiles = MT == 32 ? 2 : 1;
  static constexpr uint32_t kTok = 32 * kActTiles;
  static constexpr uint32_t kRows = 2 * MT;
  static constexpr uint32_t kHalves = MT == 32 ? 1 : 2;  // halves of a super-block per stage
  static constexpr uint32_t kStages = MT == 32 ? 2 : 4;
  static constexpr uint32_t kCh = TY == RLH_TYPE_Q8_0 ? 9 : TY == RLH_TYPE_Q6_K ? 7 : 5;  // chunks of a half
  static constexpr uint32_t kActI = 4 * kActTiles + (MT == 32 && kSums ? 2 : 1);          // 1 KB copies
  static constexpr uint32_t kWI = (kCh * kRows * 16 + 1023) / 1024;
  static constexpr uint32_t kTailI = TY == RLH_TYPE_Q6_K ? 1 : 0;  // a 256-byte copy
  static constexpr uint32_t kCopies = kActI + kWI + kTailI;
  static constexpr uint32_t kPerWave = (kCopies + 3) / 4;  // copies of a half per wave
  static constexpr uint32_t kDOff = kActTiles * 4096;      // scales, then sums: 512 bytes per tile
  static constexpr uint32_t kWOff = kActI * 1024, kTailOff = kWOff + kWI * 1024;
  static constexpr uint32_t kHalfBytes = kTailOff + kTailI * 256;
  static constexpr uint32_t kStageBytes = kHalves * kHalfBytes;
  static constexpr uint32_t kLds = kStages * kStageBytes;
  // chunk of the item that staged chunk c of half h holds
  __device__ __forceinline__ static uint32_t chunk(uint32_t c, uint32_t h) {
    if (TY == RLH_TYPE_Q4_K) return c ? c + 4 * h : 0;
    if (TY == RLH_TYPE_Q6_K) return c < 4 ? c + 4 * h : c < 6 ? c + 4 + 2 * h : 12;
    if (TY == RLH_TYPE_Q8_0) return c < 8 ? c + 8 * h : 16;
    return c < 4 ? c + 4 * h : 8;
  }
};

template <int MT>
struct Vec;
template <>
struct Vec<32> {
  typedef v16i I;
  static constexpr int N = 16;
};
template <>
struct Vec<16> {
  typedef v4i I;
  static constexpr int N = 4;
};

__device__ __forceinline__ uint64_t l8(const lbyte* p) { return *(const RLH_LDS uint64_t*)p; }
__device__ __forceinline__ float ub(uint32_t w, int b) { return (float)((w >> (8 * b)) & 0xffu); }

// The steps of a combine over N elements. N = 16: every step over 8 elements
// before the next one, since an f32 add or multiply issues every 4.6 cycles
// from one wave but its result takes 9, and a chain written element by
// element (the order the compiler's scheduler prefers, to save registers)
// runs at half rate. N = 4: left to the scheduler, which has the registers
// to overlap blocks.
template <int N, class... F>
__device__ __forceinline__ void phases(F... f) {
  constexpr int M = N < 8 ? N : 8;
#pragma unroll
  for (int e0 = 0; e0 < N; e0 += M) {
    auto step = [&](auto g) {
#pragma unroll
      for (int e = e0; e < e0 + M; e++) g(e);
      if constexpr (N > 8) __builtin_amdgcn_sched_barrier(0);
    };
    (step(f), ...);
  }
}

// A wave's place in its block and the LDS views of the current stage.
template <uint32_t TY, int MT>
struct Wave {
  using G = Geo<TY, MT>;
  static constexpr int N = Vec<MT>::N;
  uint32_t lane, l, q;  // q: lane group (MT 32: half 0/1; MT 16: 0..3)
  uint32_t tw, rw;
  const lbyte* qs;
  const lbyte* ds;
  const lbyte* w;
  const lbyte* tail;
  __device__ __forceinline__ void view(const lbyte* buf) {
    qs = buf + (MT == 32 ? tw * 4096u : 0u);
    ds = buf + G::kDOff + (MT == 32 ? tw * 512u : 0u);
    w = buf + G::kWOff;
    tail = buf + G::kTailOff;
  }
  // row of the block that the lane holds
  __device__ __forceinline__ uint32_t row() const { return rw * MT + l; }
  // scales of the lane's N tokens for block kb: element e = 4 g + i is token
  // 8 g + 4 q + i (MT 32) or 16 tw + 4 q + i (MT 16)
  __device__ __forceinline__ void scales(float (&d)[N], uint32_t kb) const {
    const RLH_LDS float* b = (const RLH_LDS float*)ds + kb * 32 + 4 * q + (MT == 16 ? 16 * tw : 0u);
#pragma unroll
    for (int g = 0; g < N / 4; g++) {
      const f32x4_t v = *(const RLH_LDS f32x4_t*)(b + 8 * g);
#pragma unroll
      for (int i = 0; i < 4; i++) d[4 * g + i] = v[i];
    }
  }
  // the scales of elements e .. e + 3 (e a multiple of 4) into d[e & 7] ..
  __device__ __forceinline__ void scale8(float (&d)[8], uint32_t kb, int e) const {
    if (e & 3) return;
    const f32x4_t x = *(const RLH_LDS f32x4_t*)((const RLH_LDS float*)ds + kb * 32 + 4 * q +
                                                (MT == 16 ? 16 * tw : 0u) + 2 * e);
#pragma unroll
    for (int i = 0; i < 4; i++) d[(e & 7) + i] = x[i];
  }
  // sum of the quants of block kb of one token per lane: token l (MT 32, its
  // tile) or 16 tw + l (MT 16)
  __device__ __forceinline__ float sum(uint32_t kb) const {
    const RLH_LDS int32_t* b = (const RLH_LDS int32_t*)(ds + 512 * G::kActTiles);
    return (float)b[kb * 32 + (MT == 16 ? 16 * tw : 0u) + l];
  }
  // 16 bytes (MT 32) or 8 (MT 16) of the token operand of block kb; the
  // weight operand (wfrag) takes the same positions in the same order
  __device__ __forceinline__ v4i afrag(uint32_t kb) const {
    if constexpr (MT == 32) {
      return *(const RLH_LDS v4i*)(qs + kb * 1024 + lane * 16);
    } else {
      const uint64_t x = l8(qs + kb * 1024 + (q & 1) * 512 + (16 * tw + l) * 16 + (q >> 1) * 8);
      return v4i{(int)(uint32_t)x, (int)(uint32_t)(x >> 32), 0, 0};
    }
  }
  __device__ __forceinline__ const lbyte* chunk(uint32_t c) const { return w + (c * G::kRows + row()) * 16; }
  // bytes of a 32-value run stored one byte per value in chunks c0, c0 + 1
  __device__ __forceinline__ v4i wfrag(uint32_t c0) const {
    if constexpr (MT == 32) {
      const uint64_t x = l8(chunk(c0) + 8 * q), y = l8(chunk(c0 + 1) + 8 * q);
      return v4i{(int)(uint32_t)x, (int)(uint32_t)(x >> 32), (int)(uint32_t)y, (int)(uint32_t)(y >> 32)};
    } else {
      const uint64_t x = l8(chunk(c0 + (q >> 1)) + 8 * (q & 1));
      return v4i{(int)(uint32_t)x, (int)(uint32_t)(x >> 32), 0, 0};
    }
  }
  __device__ __forceinline__ static typename Vec<MT>::I base() {
    typename Vec<MT>::I m;
#pragma unroll
    for (int i = 0; i < N; i++) m[i] = kBase;
    return m;
  }
  // kBase + the dots of a 32-value block
  __device__ __forceinline__ static typename Vec<MT>::I dot32(v4i a, v4i b) {
    if constexpr (MT == 32)
      return __builtin_amdgcn_mfma_i32_32x32x32_i8(a, b, base(), 0, 0, 0);
    else
      return __builtin_amdgcn_mfma_i32_16x16x32_i8(lo64(a), lo64(b), base(), 0, 0, 0);
  }
  // kBase + the dots of a 16-value half of a block (MT 32: each lane's 8
  // bytes of it; MT 16: lane groups 2s, 2s + 1 hold half s, the others'
  // weights are zero)
  __device__ __forceinline__ static typename Vec<MT>::I dot16(uint64_t a, uint64_t b) {
    if constexpr (MT == 32)
      return __builtin_amdgcn_mfma_i32_32x32x16_i8((long)a, (long)b, base(), 0, 0, 0);
    else
      return __builtin_amdgcn_mfma_i32_16x16x32_i8((long)a, (long)b, base(), 0, 0, 0);
  }
  __device__ __forceinline__ static long lo64(v4i v) { return (long)(((uint64_t)(uint32_t)v.y << 32) | (uint32_t)v.x); }
  // the dot in units of 2^-26
  __device__ __forceinline__ static float dotf(int c) { return __int_as_float(c) - kBaseF; }
};

// ---- half a super-block of a wave, per type ---------------------------------
// acc[e]: the lane's row, its e-th token; h = the half.
template <uint32_t TY, int MT>
struct Step;

// Q4_K: staged chunk 0 = d, dmin, 12 scale bytes; chunks 1 + 2g, 2 + 2g hold
// block 2g of the half in the low and 2g + 1 in the high nibbles.
template <int MT>
struct Step<RLH_TYPE_Q4_K, MT> {
  using W = Wave<RLH_TYPE_Q4_K, MT>;
  static constexpr int N = W::N;
  __device__ __forceinline__ static void run(const W& v, uint32_t h, float (&acc)[N]) {
    const u32x4_t hd = *(const RLH_LDS u32x4_t*)v.chunk(0);
    const float d = kUnit * f16_to_f32(hd.x & 0xffff), dmin = f16_to_f32(hd.x >> 16);
    // get_scale_min_k4 (quant.rs:176-185): the half's four 6-bit values of each kind
    const uint32_t sc = h ? (hd.w & 0x0F0F0F0Fu) | ((hd.y >> 2) & 0x30303030u) : hd.y & 0x3F3F3F3Fu;
    uint32_t mn = h ? ((hd.w >> 4) & 0x0F0F0F0Fu) | ((hd.z >> 2) & 0x30303030u) : hd.z & 0x3F3F3F3Fu;
    mn >>= 8 * v.q;  // the lane group's own block of a rank-1 product in byte 0 (and 2)
    f32x16_t pm;     // MT 16: the half's four rank-1 products
    if constexpr (MT == 16)
      pm = __builtin_amdgcn_mfma_f32_16x16x1f32(v.sum(v.q), dmin * ub(mn, 0), f32x16_t{}, 0, 0, 0);
#pragma unroll
    for (int g = 0; g < 2; g++) {
      const v4i a0 = v.afrag(2 * g), a1 = v.afrag(2 * g + 1), x = v.wfrag(1 + 2 * g);
      v4i b0, b1;
#pragma unroll
      for (int i = 0; i < 4; i++) {
        b0[i] = x[i] & 0x0F0F0F0F;
        b1[i] = (int)(((uint32_t)x[i] >> 4) & 0x0F0F0F0Fu);
      }
      const float d0 = d * ub(sc, 2 * g), d1 = d * ub(sc, 2 * g + 1);
      float p0[N], p1[N];  // dmin*m * sum, each rounded once
      if constexpr (MT == 32) {
        const f32x32_t p =
            __builtin_amdgcn_mfma_f32_32x32x1f32(v.sum(2 * g + v.q), dmin * ub(mn, 2 * g), f32x32_t{}, 0, 0, 0);
#pragma unroll
        for (int e = 0; e < N; e++) p0[e] = p[e], p1[e] = p[N + e];
      } else {
#pragma unroll
        for (int e = 0; e < N; e++) p0[e] = pm[8 * g + e], p1[e] = pm[8 * g + 4 + e];
      }
      // acc + (da * (d0 * dot0 - p0) + db * (d1 * dot1 - p1)) (simd.rs:581),
      // one block after the other and the scales eight at a time: the wave
      // stays within 128 registers
      float f0[N], f1[N], sc8[8];
      const auto c0 = W::dot32(a0, b0);
      phases<N>([&](int e) { v.scale8(sc8, 2 * g, e); }, [&](int e) { f0[e] = W::dotf(c0[e]); },
                [&](int e) { f0[e] = d0 * f0[e]; }, [&](int e) { f0[e] = f0[e] - p0[e]; },
                [&](int e) { f0[e] = sc8[e & 7] * f0[e]; });
      const auto c1 = W::dot32(a1, b1);
      phases<N>([&](int e) { v.scale8(sc8, 2 * g + 1, e); }, [&](int e) { f1[e] = W::dotf(c1[e]); },
                [&](int e) { f1[e] = d1 * f1[e]; }, [&](int e) { f1[e] = f1[e] - p1[e]; },
                [&](int e) { f1[e] = sc8[e & 7] * f1[e]; }, [&](int e) { f0[e] = f0[e] + f1[e]; },
                [&](int e) { acc[e] = acc[e] + f0[e]; });
    }
  }
};

// Q6_K: block c of the half is the nibbles c >> 1 of staged chunks 2 (c & 1)
// .. + 1 and bits 2c, 2c + 1 of chunks 4, 5; chunk 6 = 16 scales.
template <int MT>
struct Step<RLH_TYPE_Q6_K, MT> {
  using W = Wave<RLH_TYPE_Q6_K, MT>;
  static constexpr int N = W::N;
  // the lane's bytes of 16-value half s of chunk pair c0 (MT 16: lane groups
  // 2s, 2s + 1 hold half s, whatever s is asked for)
  __device__ __forceinline__ static uint64_t raw(const W& v, uint32_t c0, int s) {
    return MT == 32 ? l8(v.chunk(c0 + s) + 8 * v.q) : l8(v.chunk(c0 + (v.q >> 1)) + 8 * (v.q & 1));
  }
  // 4 (u - 32) of the four blocks: the six bits at the top of the byte, the
  // sign bit flipped
  __device__ __forceinline__ static void weights(const W& v, int s, uint64_t (&b)[4]) {
    const uint64_t x0 = raw(v, 0, s), x1 = raw(v, 2, s), f = raw(v, 4, s) ^ 0xAAAAAAAAAAAAAAAAull;
    const uint32_t w0[2] = {(uint32_t)x0, (uint32_t)(x0 >> 32)}, w1[2] = {(uint32_t)x1, (uint32_t)(x1 >> 32)};
    const uint32_t wf[2] = {(uint32_t)f, (uint32_t)(f >> 32)};
    uint32_t o[4][2];
#pragma unroll
    for (int i = 0; i < 2; i++) {
      o[0][i] = ((w0[i] << 2) & 0x3C3C3C3Cu) | ((wf[i] << 6) & 0xC0C0C0C0u);
      o[1][i] = ((w1[i] << 2) & 0x3C3C3C3Cu) | ((wf[i] << 4) & 0xC0C0C0C0u);
      o[2][i] = ((w0[i] >> 2) & 0x3C3C3C3Cu) | ((wf[i] << 2) & 0xC0C0C0C0u);
      o[3][i] = ((w1[i] >> 2) & 0x3C3C3C3Cu) | (wf[i] & 0xC0C0C0C0u);
    }
#pragma unroll
    for (int c = 0; c < 4; c++) b[c] = ((uint64_t)o[c][1] << 32) | o[c][0];
  }
  // scale of the row, for weights that enter as 4 q (its f16 sits in a 4-byte
  // word: even rows low, odd rows high)
  __device__ __forceinline__ static float scale(const W& v) {
    const uint32_t r = v.row();
    return 0.25f * kUnit * f16_to_f32((*(const RLH_LDS uint32_t*)(v.tail + 4 * r) >> (16 * (r & 1))) & 0xffff);
  }
  // terms come in the order s = 0 (c = 0..3), then s = 1 (simd.rs:630-665);
  // scales[s + 2c] (simd.rs:626-629)
  //
  // MT 16, with a wave or two per SIMD and little else to hide an LDS read or
  // an MFMA behind: the operands of both halves of a super-block are read
  // first (Half), then four products are issued together and combined (4096
  // x 12288, 61 tokens: 81 -> 77 us; 2560 x 9728, 237 tokens: 132 -> 123.
  // The other types have half the products per value and gained nothing).
  struct Half {
    float dq, da[4][N];
    uint64_t sw, a[4], w[4];
    __device__ __forceinline__ void read(const W& v, uint32_t h) {
      dq = scale(v);
      sw = l8(v.chunk(6) + 8 * h);
#pragma unroll
      for (int c = 0; c < 4; c++) a[c] = (uint64_t)W::lo64(v.afrag(c));
      weights(v, 0, w);
#pragma unroll
      for (int c = 0; c < 4; c++) v.scales(da[c], c);
    }
    __device__ __forceinline__ void combine(const W& v, float (&acc)[N]) const {
#pragma unroll
      for (int s = 0; s < 2; s++) {
        const bool keep = (v.q >> 1) == (uint32_t)s;
        v4i ci[4];
#pragma unroll
        for (int c = 0; c < 4; c++) ci[c] = W::dot16(a[c], keep ? w[c] : 0);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int c = 0; c < 4; c++) {
          const float ds = dq * (float)(int8_t)(sw >> (8 * (s + 2 * c)));
#pragma unroll
          for (int e = 0; e < N; e++) acc[e] = acc[e] + ds * W::dotf(ci[c][e]) * da[c][e];  // simd.rs:663
        }
      }
    }
  };
  __device__ __forceinline__ static void run(const W& v, uint32_t h, float (&acc)[N]) {
    const float dq = scale(v);
    const uint64_t sw = l8(v.chunk(6) + 8 * h);  // the half's 8 scales
#pragma unroll
    for (int s = 0; s < 2; s++) {
      uint64_t b[4];
      weights(v, s, b);
      uint64_t a[2];  // the operand and scales of block c + 1 are read while block c is combined
      float da[2][N];
      auto read = [&](int c) {
        a[c & 1] = l8(v.qs + c * 1024 + v.lane * 16 + 8 * s);
        v.scales(da[c & 1], c);
      };
      read(0);
#pragma unroll
      for (int c = 0; c < 4; c++) {
        if (c < 3) read(c + 1);
        const auto ci = W::dot16(a[c & 1], b[c]);
        const float ds = dq * (float)(int8_t)(sw >> (8 * (s + 2 * c)));
        float f[N];  // acc + (ds * dot) * da (simd.rs:663)
        phases<N>([&](int e) { f[e] = W::dotf(ci[e]); }, [&](int e) { f[e] = ds * f[e]; },
                  [&](int e) { f[e] = f[e] * da[c & 1][e]; }, [&](int e) { acc[e] = acc[e] + f[e]; });
      }
    }
  }
};

// Q8_0: staged chunks 2k, 2k + 1 hold block k of the half, chunk 8 the 8 f16
// scales. Q4_0: chunk k holds block k (positions 0..15 low nibbles, 16..31
// high), chunk 4 the 8 f16 scales; the weights enter as 16 (nibble - 8).
template <uint32_t TY, int MT>
struct Step8 {
  using W = Wave<TY, MT>;
  static constexpr int N = W::N;
  __device__ __forceinline__ static v4i weights(const W& v, uint32_t k) {
    if constexpr (TY == RLH_TYPE_Q8_0) {
      return v.wfrag(2 * k);
    } else {
      const uint64_t x = l8(v.chunk(k) + 8 * (MT == 32 ? v.q : (v.q & 1)));
      const uint32_t w0 = (uint32_t)x, w1 = (uint32_t)(x >> 32), m = 0xF0F0F0F0u, f = 0x80808080u;
      const v4i lo = {(int)(((w0 << 4) & m) ^ f), (int)(((w1 << 4) & m) ^ f), 0, 0};
      const v4i hi = {(int)((w0 & m) ^ f), (int)((w1 & m) ^ f), 0, 0};
      if constexpr (MT == 32) return v4i{lo.x, lo.y, hi.x, hi.y};
      return (v.q >> 1) ? hi : lo;
    }
  }
  __device__ __forceinline__ static void run(const W& v, uint32_t h, float (&acc)[N]) {
    constexpr float kS = TY == RLH_TYPE_Q8_0 ? kUnit : 0.0625f * kUnit;
    const uint64_t dv = l8(v.chunk(TY == RLH_TYPE_Q8_0 ? 8 : 4) + 8 * h);  // the half's four f16 scales
    v4i a[2], b[2];  // the operands and scales of block k + 1 are read while block k is combined
    float da[2][N];
    auto read = [&](int k) {
      a[k & 1] = v.afrag(k);
      b[k & 1] = weights(v, k);
      v.scales(da[k & 1], k);
    };
    read(0);
#pragma unroll
    for (int k = 0; k < 4; k++) {
      if (k < 3) read(k + 1);
      const auto ci = W::dot32(a[k & 1], b[k & 1]);
      const float dk = kS * f16_to_f32((uint32_t)(dv >> (16 * k)) & 0xffff);
      float f[N];  // acc + (dk * dot) * da (simd.rs:891, 863)
      phases<N>([&](int e) { f[e] = W::dotf(ci[e]); }, [&](int e) { f[e] = dk * f[e]; },
                [&](int e) { f[e] = f[e] * da[k & 1][e]; }, [&](int e) { acc[e] = acc[e] + f[e]; });
    }
  }
};
template <int MT>
struct Step<RLH_TYPE_Q8_0, MT> : Step8<RLH_TYPE_Q8_0, MT> {};
template <int MT>
struct Step<RLH_TYPE_Q4_0, MT> : Step8<RLH_TYPE_Q4_0, MT> {};

// Block b runs on XCD b % 8; the blocks of one XCD walk the token tiles of a
// row tile first, so each weight tile is fetched into that XCD's L2 once and
// reused by all token tiles.
template <uint32_t TY, int MT>
__global__ void __launch_bounds__(256, 4) k_gemm(GemmArgs a0) {
  using G = Geo<TY, MT>;
  using V = Wave<TY, MT>;
  constexpr int N = V::N;
  extern __shared__ __attribute__((aligned(16))) uint8_t lds_generic[];
  lbyte* lds = (lbyte*)lds_generic;
  const uint32_t b = blockIdx.x, xcd = b & 7, k = b >> 3;
  const uint32_t tt = k % a0.n_tt, rtg = (k / a0.n_tt) * 8 + xcd;
  if (rtg >= a0.n_rt) return;  // whole block, before any barrier
  // the block's segment (uniform: from the block index)
  DevMat w = a0.w;
  float *y = a0.y, *resid = a0.resid;
  uint32_t rt = rtg;
  if (rtg >= a0.n_rt1) {
    w = a0.w2;
    y = a0.y2;
    resid = nullptr;
    rt = rtg - a0.n_rt1;
  }
  if (rtg >= a0.n_rt2) {
    w = a0.w3;
    y = a0.y3;
    rt = rtg - a0.n_rt2;
  }
  const uint32_t t0 = tt * G::kTok, r0 = rt * G::kRows, nsb = w.cols >> 8;
  const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  V v;
  v.lane = threadIdx.x & 63;
  v.l = v.lane % MT;
  v.q = v.lane / MT;
  v.tw = wave & 1;
  v.rw = wave >> 1;

  // Copies of half i % 2 of super-block i / 2 into a buffer of kHalfBytes.
  // Copy n (1 KB, the tails 256 bytes) belongs to wave n % 4; every wave
  // issues kPerWave of them (the last ones repeat copy kCopies - 1), so its
  // vector-memory count tells which step has landed. Rows past the matrix
  // read its last row, token tiles past the activation its last tile;
  // neither reaches a kept output. Sources are a uniform base plus 32-bit
  // lane offsets (the block's 2 MT rows apart at most).
  // (tile shapes are powers of two: tr = 64 / tj; a division by a value the
  // compiler does not know costs some forty instructions)
  const uint32_t tjb = (uint32_t)__builtin_ctz(w.tj), trb = 6 - tjb, trm = w.tr - 1;
  const uint32_t rt_bytes = w.ntj * 64 * w.ib, rt0 = r0 >> trb;
  const uint8_t* wbase = w.a + (size_t)rt0 * rt_bytes;
  const uint32_t lrow = min(r0 + v.lane % G::kRows, w.rows - 1);  // the lane's row (MT 16: rows 0..31 twice)
  const uint32_t wlane = ((lrow >> trb) - rt0) * rt_bytes + (lrow & trm) * 16;
  const uint32_t tlane = ((lrow >> trb) - rt0) * rt_bytes + (((lrow & trm) * 2) & ~3u);  // (tr is even)
  const uint32_t last_tile = (a0.n - 1) / 32;
  const uint8_t* xbase[2];
#pragma unroll
  for (uint32_t t = 0; t < G::kActTiles; t++)
    xbase[t] = a0.x.p + (size_t)min(t0 / 32 + t, last_tile) * nsb * kQ8TileBytes;
  auto copy = [&](uint32_t i, lbyte* buf) {
    const uint32_t j = i >> 1, h = i & 1, jt = j >> tjb, jr = (j & (w.tj - 1)) << trb;
    const uint8_t* wt = wbase + (size_t)jt * 64 * w.ib + jr * 16;
    const uint32_t xo = j * kQ8TileBytes;
#pragma unroll
    for (uint32_t m = 0; m < G::kPerWave; m++) {
      const uint32_t n = min(wave + 4 * m, G::kCopies - 1);
      const uint8_t* src;
      uint32_t off;
      if (n < 4 * G::kActTiles) {
        src = xbase[n >> 2] + xo + h * 4096 + (n & 3) * 1024;
        off = v.lane * 16;
      } else if (n < G::kActI) {
        const uint32_t l32 = (v.lane & 31) * 16;
        if (MT == 32) {  // scales (then sums) of both tiles
          src = xbase[0] + xo + 8192 + (n - 8) * 1024 + h * 512;
          off = l32 + (v.lane >= 32 ? (uint32_t)(xbase[G::kActTiles - 1] - xbase[0]) : 0u);
        } else {  // scales and sums of the tile
          src = xbase[0] + xo + 8192 + h * 512;
          off = l32 + (v.lane >= 32 ? 1024u : 0u);
        }
      } else if (n < G::kActI + G::kWI) {
        const uint32_t p = n - G::kActI;
        if (MT == 32) {
          src = wt + G::chunk(p, h) * 1024;
          off = wlane;
        } else {  // chunks 2p and 2p + 1 of the 32 rows
          const uint32_t c0 = G::chunk(2 * p, h), c1 = G::chunk(min(2 * p + 1, G::kCh - 1), h);
          src = wt + c0 * 1024;
          off = wlane + (v.lane >= 32 ? (c1 - c0) * 1024 : 0u);
        }
      } else {
        src = wbase + (size_t)jt * 64 * w.ib + (w.ib / 16) * 1024 + jr * 2;
        __builtin_amdgcn_global_load_lds((const RLH_GLOBAL void*)(src + tlane),
                                         (RLH_LDS void*)(buf + G::kTailOff), 4, 0, 0);
        continue;
      }
      __builtin_amdgcn_global_load_lds((const RLH_GLOBAL void*)(src + off), (RLH_LDS void*)(buf + n * 1024), 16, 0, 0);
    }
  };

  float acc[N];
#pragma unroll
  for (int e = 0; e < N; e++) acc[e] = 0.0f;

  // a wave whose tokens all lie past the last one only copies
  const bool live = t0 + MT * v.tw < a0.n;
  const uint32_t steps = 2 * nsb / G::kHalves;
  auto stage = [&](uint32_t i, uint32_t at) {
#pragma unroll
    for (uint32_t h = 0; h < G::kHalves; h++)
      copy(i * G::kHalves + h, lds + at * G::kStageBytes + h * G::kHalfBytes);
  };
#pragma unroll
  for (uint32_t s = 0; s + 1 < G::kStages; s++)
    if (s < steps) stage(s, s);
  uint32_t cur = 0, nxt = G::kStages - 1;  // buffers of step i and of step i + kStages - 1
  for (uint32_t i = 0; i < steps; i++) {
    // step i has landed: this wave's copies by its count (the later steps'
    // copies stay in flight), the others' by the barrier, past which every
    // wave is done with the buffer that step i + kStages - 1 takes
    if (i + G::kStages - 2 < steps)
      wait_vmcnt<(G::kStages - 2) * G::kHalves * G::kPerWave>();
    else
      wait_vmcnt<0>();
    lds_barrier();
    if (i + G::kStages - 1 < steps) stage(i + G::kStages - 1, nxt);
    const lbyte* buf = lds + cur * G::kStageBytes;
    if constexpr (MT == 16 && TY == RLH_TYPE_Q6_K) {
      if (live) {
        typename Step<TY, MT>::Half half[2];
#pragma unroll
        for (uint32_t h = 0; h < 2; h++) {
          v.view(buf + h * G::kHalfBytes);
          half[h].read(v, h);
        }
        __builtin_amdgcn_sched_barrier(0);
        half[0].combine(v, acc);
        half[1].combine(v, acc);
      }
    } else if (live) {
#pragma unroll
      for (uint32_t h = 0; h < G::kHalves; h++) {
        v.view(buf + h * G::kHalfBytes);
        Step<TY, MT>::run(v, G::kHalves == 1 ? i & 1 : h, acc);
      }
    }
    cur = cur + 1 == G::kStages ? 0 : cur + 1;
    nxt = nxt + 1 == G::kStages ? 0 : nxt + 1;
  }
  if (!live) return;  // after the last barrier
  const uint32_t row = r0 + v.row();
  if (row >= w.rows) return;
  const size_t base = (size_t)(t0 + MT * v.tw + 4 * v.q) * w.rows + row;
  const uint32_t left = a0.n - t0 - MT * v.tw;  // tokens of this wave (>= 1)
  if (resid) {  // xs += xb (model.rs:548-552, 569-573)
    float old[N];
#pragma unroll
    for (int e = 0; e < N; e++) {
      const uint32_t o = 8 * (e / 4) + e % 4;
      old[e] = o + 4 * v.q < left ? ld_gf(resid + base + (size_t)o * w.rows) : 0.0f;
    }
#pragma unroll
    for (int e = 0; e < N; e++) {
      const uint32_t o = 8 * (e / 4) + e % 4;
      if (o + 4 * v.q < left) ((RLH_GLOBAL float*)resid)[base + (size_t)o * w.rows] = old[e] + acc[e];
    }
  }
  if (y) {
#pragma unroll
    for (int e = 0; e < N; e++) {
      const uint32_t o = 8 * (e / 4) + e % 4;
      if (o + 4 * v.q < left) ((RLH_GLOBAL float*)y)[base + (size_t)o * w.rows] = acc[e];
    }
  }
}

// ---------------------------------------------------------------------------
// Prefill products for the types with no integer batch path in the reference
// (Q5_K, Q4_1, Q5_0, Q5_1, F16, BF16): matmul_batch's f32 route (ops.rs:237-312)
// dequantizes rows (quant.rs:191-385) and runs dot_multi_rows::<3, 4>
// (simd.rs:779-836) on the f32 activations. Every output of a token group of
// 4 is one 8-lane FMA chain over the row (lane l takes elements 8i + l in
// order) reduced by the AVX2 tree; the last n % 4 tokens take dot_f32_avx2
// (32 chains over 32-value chunks, (a0+a1)+(a2+a3), tree). ys starts at zero
// and gets `+= value`. F32 weights take matmul_batch's F32 fast path
// (ops.rs:165-174): dot(row, x) for every token, stored as is.
//
// The chains run on the f32 MFMA, whose result is the chain of fused
// multiply-adds over k = 0, 1, .. in order, rounded at each (every depth and
// shape; subnormals, infinities and NaN as fmaf), at twice the rate of
// v_fma_f32. A 16 x 16 x 4 product of tokens x rows over elements 32 p + 8 k
// + l (k = 0..3) is four steps of chain l of dot_multi_rows. The same
// weight operand in sixteen 4 x 4 x 1 blocks (4 single tokens; block 4 k + g
// = rows 4 g .. + 3) is one step of the chains (k, l) of dot_f32_avx2. A
// lane's operands of all eight l are 32 consecutive bytes.
//
// Block: 16 RT rows x up to 4 jobs, one wave per job; a job is 16 tokens in
// groups of four, or 4 single tokens (32 RT accumulators either way). 256 /
// RT values of the rows (16 per thread) are dequantized into the second of
// two LDS buffers while the current ones are multiplied; the activations
// come straight from memory (each token's 32 values of a step are one
// 128-byte line), two steps ahead. A 9728 x 2560 Q5_K pair with 131 tokens:
// 658 us with one FMA chain per thread, 191 us; its multiply-adds alone take
// 83 us at the f32 MFMA rate, which no VALU work overlaps (the dequantizing
// adds to it).
// ---------------------------------------------------------------------------
constexpr uint32_t kFT = 16;  // tokens per grouped job

struct GemmF32Args {
  DevMat w;
  DevMat w2, w3;   // further segments of the same type and columns (rows 0: none)
  const float* x;  // [n][cols] f32
  uint32_t n;
  float* y;
  float *y2, *y3;
  float* resid;    // of the first segment
  uint32_t n4;     // tokens handled in groups of 4 (n - n % 4)
  uint32_t n_jb;   // blocks per row tile: jobs / 4, rounded up
  uint32_t n_rt;   // row tiles of all segments
  uint32_t n_rt1;  // row tiles of w
  uint32_t n_rt2;  // row tiles of w and w2
};

__device__ __forceinline__ float tree8(const float* A) {
  return ((A[0] + A[4]) + (A[2] + A[6])) + ((A[1] + A[5]) + (A[3] + A[7]));
}

// Values 16 * dp .. 16 * dp + 15 of super-block j (256 values) of row r,
// dequantized exactly (quant.rs:191-385). The loads come first, the
// conversion second, so that callers can place a barrier between them.
template <uint32_t TY>
struct Dq16 {
  u32x4_t v[4];  // raw bytes
  uint32_t aux0, aux1;
  __device__ __forceinline__ void load(const DevMat& w, uint32_t r, uint32_t j, uint32_t dp) {
    if constexpr (TY == RLH_TYPE_Q5_K) {
      const uint32_t dsub = dp / 2, dl = 16 * (dp % 2);
      v[0] = *(const RLH_GLOBAL u32x4_t*)(w.a + item_offset(w, r, j, 0));
      v[1] = *(const RLH_GLOBAL u32x4_t*)(w.a + item_offset(w, r, j, 48 + 32 * (dsub / 2) + dl));
      v[2] = *(const RLH_GLOBAL u32x4_t*)(w.a + item_offset(w, r, j, 16 + dl));
    } else if constexpr (TY == RLH_TYPE_Q4_1 || TY == RLH_TYPE_Q5_0 || TY == RLH_TYPE_Q5_1) {
      const uint32_t k = dp / 2;  // the 32-value block
      v[0] = *(const RLH_GLOBAL u32x4_t*)(w.a + item_offset(w, r, j, 16 * k));
      const uint32_t sc0 = TY == RLH_TYPE_Q4_1 ? 128 : 160;
      if constexpr (TY != RLH_TYPE_Q4_1) aux1 = *(const RLH_GLOBAL uint32_t*)(w.a + item_offset(w, r, j, 128 + 4 * k));
      if constexpr (TY == RLH_TYPE_Q5_0)
        aux0 = *(const RLH_GLOBAL uint16_t*)(w.a + item_offset(w, r, j, sc0 + 2 * k));
      else
        aux0 = *(const RLH_GLOBAL uint32_t*)(w.a + item_offset(w, r, j, sc0 + 4 * k));
    } else if constexpr (TY == RLH_TYPE_F16 || TY == RLH_TYPE_BF16) {
      const uint8_t* p = w.a + (size_t)r * w.row_bytes + 2 * (256 * (size_t)j + 16 * dp);
      v[0] = *(const RLH_GLOBAL u32x4_t*)p;
      v[1] = *(const RLH_GLOBAL u32x4_t*)(p + 16);
    } else {  // F32
      const uint8_t* p = w.a + (size_t)r * w.row_bytes + 4 * (256 * (size_t)j + 16 * dp);
#pragma unroll
      for (int q = 0; q < 4; q++) v[q] = *(const RLH_GLOBAL u32x4_t*)(p + 16 * q);
    }
  }
  __device__ __forceinline__ void values(uint32_t dp, f32x4_t* o) const {
    if constexpr (TY == RLH_TYPE_Q5_K) {
      const uint32_t dsub = dp / 2;
      const u32x4_t hdr = v[0], qv = v[1], hv = v[2];
      const float d = f16_to_f32(hdr.x & 0xffff), dmin = f16_to_f32(hdr.x >> 16);
      // get_scale_min_k4 (quant.rs:176-185)
      const uint32_t sh = 8 * (dsub & 3), s0 = hdr.y >> sh, s1 = hdr.z >> sh, s2 = hdr.w >> sh;
      const uint32_t sc = dsub < 4 ? s0 & 63 : (s2 & 15) | (s0 >> 2 & 48);
      const uint32_t m = dsub < 4 ? s1 & 63 : (s2 >> 4 & 15) | (s1 >> 2 & 48);
      const float d1 = d * (float)sc, mm1 = dmin * (float)m;
      const uint32_t qw[4] = {qv.x, qv.y, qv.z, qv.w}, hw[4] = {hv.x, hv.y, hv.z, hv.w};
#pragma unroll
      for (int q = 0; q < 4; q++) {
        const uint32_t u = ((qw[q] >> (4 * (dsub & 1))) & 0x0F0F0F0Fu) | (((hw[q] >> dsub) & 0x01010101u) << 4);
        o[q].x = d1 * (float)(u & 0xff) - mm1;
        o[q].y = d1 * (float)((u >> 8) & 0xff) - mm1;
        o[q].z = d1 * (float)((u >> 16) & 0xff) - mm1;
        o[q].w = d1 * (float)(u >> 24) - mm1;
      }
    } else if constexpr (TY == RLH_TYPE_Q4_1 || TY == RLH_TYPE_Q5_0 || TY == RLH_TYPE_Q5_1) {
      const uint32_t half = dp % 2;  // values 16 * half .. + 15 of the block
      const uint32_t qw[4] = {v[0].x, v[0].y, v[0].z, v[0].w};
      float d, m = 0.0f;
      if constexpr (TY == RLH_TYPE_Q5_0) {
        d = f16_to_f32(aux0 & 0xffff);
      } else {
        d = f16_to_f32(aux0 & 0xffff);
        m = f16_to_f32(aux0 >> 16);
      }
#pragma unroll
      for (int q = 0; q < 4; q++) {
        float e[4];
#pragma unroll
        for (int b = 0; b < 4; b++) {
          const uint32_t i = 4 * q + b;  // byte i of the block's quants
          uint32_t x = (qw[q] >> (8 * b + 4 * half)) & 0xF;
          if constexpr (TY != RLH_TYPE_Q4_1) x |= ((aux1 >> (i + 16 * half)) & 1u) << 4;
          if constexpr (TY == RLH_TYPE_Q5_0)
            e[b] = (float)((int)x - 16) * d;
          else
            e[b] = (float)x * d + m;
        }
        o[q] = f32x4_t{e[0], e[1], e[2], e[3]};
      }
    } else if constexpr (TY == RLH_TYPE_F16 || TY == RLH_TYPE_BF16) {
      const uint32_t hw[8] = {v[0].x, v[0].y, v[0].z, v[0].w, v[1].x, v[1].y, v[1].z, v[1].w};
      auto cv = [](uint32_t h) {
        return TY == RLH_TYPE_F16 ? f16_to_f32(h) : __uint_as_float(h << 16);  // quant.rs:115-157, bf16_to_f32
      };
#pragma unroll
      for (int q = 0; q < 4; q++)
        o[q] = f32x4_t{cv(hw[2 * q] & 0xffff), cv(hw[2 * q] >> 16), cv(hw[2 * q + 1] & 0xffff),
                       cv(hw[2 * q + 1] >> 16)};
    } else {
#pragma unroll
      for (int q = 0; q < 4; q++)
        o[q] = f32x4_t{__uint_as_float(v[q].x), __uint_as_float(v[q].y), __uint_as_float(v[q].z),
                       __uint_as_float(v[q].w)};
    }
  }
};

template <uint32_t TY, int RT>
__global__ void __launch_bounds__(256, 3) k_gemm_f32(GemmF32Args a) {
  constexpr uint32_t kFR = 16 * RT, kFV = 256 / RT, kFS = kFV + 4;  // rows, values per stage, LDS row stride
  __shared__ __attribute__((aligned(16))) float ws_g[2][kFR * kFS];
  typedef RLH_LDS float lfloat;
  typedef RLH_LDS f32x4_t lf32x4;
  lfloat* ws = (lfloat*)ws_g;
  // XCD-aware order as in k_gemm
  const uint32_t b = blockIdx.x, k = b >> 3;
  const uint32_t jb = k % a.n_jb, rtg = (k / a.n_jb) * 8 + (b & 7);
  if (rtg >= a.n_rt) return;  // whole block, before any barrier
  DevMat w = a.w;
  float *y = a.y, *resid = a.resid;
  uint32_t r0 = rtg * kFR;
  if (rtg >= a.n_rt1) {
    w = a.w2;
    y = a.y2;
    resid = nullptr;
    r0 = (rtg - a.n_rt1) * kFR;
  }
  if (rtg >= a.n_rt2) {
    w = a.w3;
    y = a.y3;
    r0 = (rtg - a.n_rt2) * kFR;
  }
  const uint32_t tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const uint32_t l = tid & 15, q = (tid >> 4) & 3;
  const uint32_t S = w.cols / 32, nh = w.cols / kFV;
  // the wave's job: the jobs spread evenly over the row tile's blocks, the
  // slots without one over the waves (each wave has a SIMD of its own)
  const uint32_t nm = (a.n4 + kFT - 1) / kFT, jobs = nm + (a.n - a.n4 + 3) / 4;
  const uint32_t per = (jobs + a.n_jb - 1) / a.n_jb, slot = (wave + b / 8 + rtg) & 3, job = per * jb + slot;
  const bool live = slot < per && job < jobs, single = job >= nm;
  const uint32_t tok0 = single ? a.n4 + (job - nm) * 4 : job * kFT, tok_end = single ? a.n : a.n4;
  const float* xp = a.x + (size_t)(live ? min(tok0 + (single ? l & 3 : l), tok_end - 1) : 0u) * w.cols + 8 * q;
  f32x4_t xv[4][2];  // steps p .. p + 2
  auto load_x = [&](uint32_t p) {
    const float* src = xp + 32 * min(p, S - 1);
    xv[p & 3][0] = *(const RLH_GLOBAL f32x4_t*)src;
    xv[p & 3][1] = *(const RLH_GLOBAL f32x4_t*)(src + 4);
  };
  // dequant duty: 16 values (piece dpc) of one of the block's rows
  constexpr uint32_t kPc = kFV / 16;
  const uint32_t drow = min(r0 + tid / kPc, w.rows - 1), dpc = tid % kPc;
  Dq16<TY> dq;
  auto load_w = [&](uint32_t h) { dq.load(w, drow, h / RT, kPc * (h % RT) + dpc); };
  auto store_w = [&](uint32_t h) {
    lfloat* o = ws + (h & 1) * (kFR * kFS) + (tid / kPc) * kFS + 16 * dpc;
    f32x4_t v[4];
    dq.values(kPc * (h % RT) + dpc, v);
#pragma unroll
    for (int i = 0; i < 4; i++) *(lf32x4*)(o + 4 * i) = v[i];
  };
  auto el = [](const f32x4_t (&v)[2], int c) { return v[c >> 2][c & 3]; };

  load_w(0);
#pragma unroll
  for (uint32_t p = 0; p < 2; p++) load_x(p);
  store_w(0);
  if (nh > 1) load_w(1);
  lds_barrier();
  // one loop per kind of job (a condition inside one loop would make the
  // compiler copy the accumulators); all meet the same barriers
  auto sweep = [&](auto mul) {
    for (uint32_t h = 0; h < nh; h++) {
      if (h + 1 < nh) store_w(h + 1);  // that buffer's last readers passed the barrier that ended h - 1
      if (h + 2 < nh) load_w(h + 2);
      const lfloat* wb = ws + (h & 1) * (kFR * kFS) + l * kFS + 8 * q;
      mul(h, wb);
      lds_barrier();
    }
  };
  auto products = [&](auto step) {
    sweep([&](uint32_t h, const lfloat* wb) {
      f32x4_t wv[2][2];  // of product i (step i / RT, rows 16 (i % RT) ..) and of the next one
      auto read_w = [&](int i) {
        const lfloat* wp = wb + 16 * (i % RT) * kFS + 32 * (i / RT);
        wv[i & 1][0] = *(const lf32x4*)wp;
        wv[i & 1][1] = *(const lf32x4*)(wp + 4);
      };
      read_w(0);
#pragma unroll
      for (int i = 0; i < 8; i++) {
        if (i % RT == 0) load_x(kFV / 32 * h + i / RT + 2);
        if (i < 7) read_w(i + 1);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int c = 0; c < 8; c++) step(i % RT, c, el(xv[(i / RT) & 3], c), el(wv[i & 1], c));
        __builtin_amdgcn_sched_barrier(0);
      }
    });
  };
  auto put = [&](uint32_t tok, uint32_t row, float v) {
    if (tok >= tok_end || row >= w.rows) return;
    const size_t idx = (size_t)tok * w.rows + row;
    if (resid) {
      RLH_GLOBAL float* o = (RLH_GLOBAL float*)resid;
      o[idx] = o[idx] + v;
    }
    if (y) ((RLH_GLOBAL float*)y)[idx] = v;
  };
  f32x4_t acc[RT][8];
#pragma unroll
  for (int t = 0; t < RT; t++)
#pragma unroll
    for (int c = 0; c < 8; c++) acc[t][c] = f32x4_t{};
  if (!live) {
    sweep([](uint32_t, const lfloat*) {});
  } else if (!single) {  // element e of a lane: token 4 q + e, row l
    products([&](int t, int c, float xe, float we) {
      acc[t][c] = __builtin_amdgcn_mfma_f32_16x16x4f32(xe, we, acc[t][c], 0, 0, 0);
    });
#pragma unroll
    for (int t = 0; t < RT; t++)
#pragma unroll
      for (int e = 0; e < 4; e++) {
        float c8[8];
#pragma unroll
        for (int c = 0; c < 8; c++) c8[c] = acc[t][c][e];
        // out += hsum(acc) + tail (no tail: cols % 8 == 0)
        put(tok0 + 4 * q + e, r0 + 16 * t + l, 0.0f + (tree8(c8) + 0.0f));
      }
  } else {  // element e of a lane: token e, row l, chains (q, c)
    products([&](int t, int c, float xe, float we) {
      acc[t][c] = __builtin_amdgcn_mfma_f32_4x4x1f32(xe, we, acc[t][c], 0, 0, 0);
    });
#pragma unroll
    for (int t = 0; t < RT; t++)
#pragma unroll
      for (int e = 0; e < 4; e++) {
        float A[8];
#pragma unroll
        for (int c = 0; c < 8; c++) {  // (a0 + a1) + (a2 + a3) over the lane groups
          const float s = acc[t][c][e] + __shfl_xor(acc[t][c][e], 16);
          A[c] = s + __shfl_xor(s, 32);
        }
        // F32 weights store dot(row, x) (ops.rs:169-173); the others add it to
        // the zeroed output (ops.rs:236 ys.fill, then +=)
        const float v = TY == RLH_TYPE_F32 ? tree8(A) : 0.0f + tree8(A);
        if (q == 0) put(tok0 + e, r0 + 16 * t + l, v);
      }
  }
}

}  // namespace

bool gemm_supported(uint32_t ty) {
  return ty == RLH_TYPE_Q4_K || ty == RLH_TYPE_Q6_K || ty == RLH_TYPE_Q8_0 || ty == RLH_TYPE_Q4_0;
}

bool gemm_f32_supported(uint32_t ty) {
  return ty == RLH_TYPE_Q5_K || ty == RLH_TYPE_Q4_1 || ty == RLH_TYPE_Q5_0 || ty == RLH_TYPE_Q5_1 ||
         ty == RLH_TYPE_F16 || ty == RLH_TYPE_BF16 || ty == RLH_TYPE_F32;
}

template <uint32_t TY>
static void launch_f32_type(hipStream_t st, GemmF32Args a) {
  const uint32_t jobs = (a.n4 + kFT - 1) / kFT + (a.n - a.n4 + 3) / 4;
  a.n_jb = (jobs + 3) / 4;
  auto row_tiles = [&](uint32_t fr) {
    a.n_rt1 = (a.w.rows + fr - 1) / fr;
    a.n_rt2 = a.n_rt1 + (a.w2.rows + fr - 1) / fr;
    a.n_rt = a.n_rt2 + (a.w3.rows + fr - 1) / fr;
  };
  // 32-row or 16-row blocks. A block whose every wave multiplies most of the
  // time (four jobs; three for F32 weights, whose jobs are all 4 single
  // tokens) takes about 14 / 23 / 33 us of 1024 columns with one / two / three
  // of 32 rows on a CU and 13 / 20 / 28 / 38 with one to four of 16, so 32
  // rows unless 16 put no more blocks on a CU (an XCD's 32 CUs get every
  // eighth row tile). Both sides, 16 / 32 rows: F32 3072 columns, 131 tokens,
  // 128 blocks of 32 rows 51 / 33, 256 (two on some CUs either way) 51 / 57;
  // 200 tokens, 416 blocks 108 / 57; Q5_K 4096 columns, 200 tokens, 320 blocks
  // 94 / 88.
  // The others overlap up to what is resident. Three jobs, or the types whose
  // dequantizing takes longest: 16 rows until a second round of the three per
  // CU begins (Q5_K 3072 columns, 131 tokens, 384 blocks 55 / 65, 400 77 / 65;
  // Q5_0 4096 columns, 200 tokens, 384 92 / 96, 448 124 / 96). One or two jobs:
  // a little longer (3072 columns, 20 tokens, 512 blocks Q4_1 44 / 61, Q5_K 64
  // / 65; 576 F16 61 / 60, Q5_K 76 / 71).
  const uint32_t per = (jobs + a.n_jb - 1) / a.n_jb;
  auto on_cu = [&] { return (a.n_jb * (uint64_t)((a.n_rt + 7) / 8) + 31) / 32; };
  row_tiles(16);
  const uint64_t on_cu16 = on_cu();
  row_tiles(32);
  const uint64_t blocks32 = (uint64_t)a.n_jb * a.n_rt;
  constexpr bool kSlowDq = TY == RLH_TYPE_Q5_0 || TY == RLH_TYPE_Q5_1;
  const bool busy = (per == 4 && !kSlowDq) || (per == 3 && TY == RLH_TYPE_F32);
  const bool rows32 = busy ? on_cu16 > on_cu() : blocks32 > (per >= 3 ? 384 : 511);
  if (!rows32) row_tiles(16);
  const dim3 grid(a.n_jb * ((a.n_rt + 7) / 8) * 8);
  if (rows32)
    hipLaunchKernelGGL((k_gemm_f32<TY, 2>), grid, dim3(256), 0, st, a);
  else
    hipLaunchKernelGGL((k_gemm_f32<TY, 1>), grid, dim3(256), 0, st, a);
}

static void launch_gemm_f32_args(hipStream_t st, GemmF32Args a) {
  if (a.w.ty == RLH_TYPE_F32) a.n4 = 0;  // every token takes dot_f32_avx2 (ops.rs:165-174)
  switch (a.w.ty) {
    case RLH_TYPE_Q5_K: launch_f32_type<RLH_TYPE_Q5_K>(st, a); break;
    case RLH_TYPE_Q4_1: launch_f32_type<RLH_TYPE_Q4_1>(st, a); break;
    case RLH_TYPE_Q5_0: launch_f32_type<RLH_TYPE_Q5_0>(st, a); break;
    case RLH_TYPE_Q5_1: launch_f32_type<RLH_TYPE_Q5_1>(st, a); break;
    case RLH_TYPE_F16: launch_f32_type<RLH_TYPE_F16>(st, a); break;
    case RLH_TYPE_BF16: launch_f32_type<RLH_TYPE_BF16>(st, a); break;
    case RLH_TYPE_F32: launch_f32_type<RLH_TYPE_F32>(st, a); break;
    default: break;
  }
}

void launch_gemm_f32(hipStream_t st, const DevMat& w, const float* x, uint32_t n, uint32_t n4, float* y,
                     float* resid) {
  GemmF32Args a{};
  a.w = w;
  a.x = x;
  a.n = n;
  a.n4 = n4;
  a.y = y;
  a.resid = resid;
  launch_gemm_f32_args(st, a);
}

bool gemm_f32_pair_supported(const DevMat& w, const DevMat& w2) {
  return gemm_f32_supported(w.ty) && w2.ty == w.ty && w2.cols == w.cols;
}

void launch_gemm_f32_pair(hipStream_t st, const DevMat& w, const DevMat& w2, const float* x, uint32_t n, uint32_t n4,
                          float* y, float* y2, const DevMat* w3, float* y3) {
  GemmF32Args a{};
  if (w3) a.w3 = *w3;
  a.y3 = y3;
  a.w = w;
  a.w2 = w2;
  a.x = x;
  a.n = n;
  a.n4 = n4;
  a.y = y;
  a.y2 = y2;
  launch_gemm_f32_args(st, a);
}

template <uint32_t TY>
static bool set_type_lds() {
  return hipFuncSetAttribute((const void*)k_gemm<TY, 16>, hipFuncAttributeMaxDynamicSharedMemorySize,
                             (int)Geo<TY, 16>::kLds) == hipSuccess &&
         hipFuncSetAttribute((const void*)k_gemm<TY, 32>, hipFuncAttributeMaxDynamicSharedMemorySize,
                             (int)Geo<TY, 32>::kLds) == hipSuccess;
}
bool gemm_set_max_lds() {
  return set_type_lds<RLH_TYPE_Q4_K>() && set_type_lds<RLH_TYPE_Q6_K>() && set_type_lds<RLH_TYPE_Q8_0>() &&
         set_type_lds<RLH_TYPE_Q4_0>();
}

template <uint32_t TY, int MT>
static void launch_variant(hipStream_t st, GemmArgs a) {
  using G = Geo<TY, MT>;
  a.n_tt = (a.n + G::kTok - 1) / G::kTok;
  a.n_rt1 = (a.w.rows + G::kRows - 1) / G::kRows;
  a.n_rt2 = a.n_rt1 + (a.w2.rows + G::kRows - 1) / G::kRows;
  a.n_rt = a.n_rt2 + (a.w3.rows + G::kRows - 1) / G::kRows;
  const uint32_t blocks = a.n_tt * ((a.n_rt + 7) / 8) * 8;
  hipLaunchKernelGGL((k_gemm<TY, MT>), dim3(blocks), dim3(256), G::kLds, st, a);
}

// 32 x 32 tiles one per wave fill the SIMDs once from 1024 tiles on; below,
// 16 x 16 tiles make four times the waves with a quarter of the work each.
// Both sides measured, 16 / 32, us at 512, 1024, 1152 and 2048 tiles (4096
// columns, 237 tokens; the ratios are the same within 4 % from 1024 to 12288
// columns and with 61 and 509 tokens): Q4_K 22 / 45, 42 / 46, 57 / 49, 79 / 51;
// Q6_K 31 / 64, 61 / 65, 77 / 73, 115 / 75; Q8_0 18 / 36, 35 / 37, 45 / 42, 66
// / 44; Q4_0 20 / 36, 39 / 37, 52 / 40, 74 / 41 (equal at 768 already, at most
// 5 % lost in between).
constexpr uint64_t kTiles32 = 1024;

template <uint32_t TY>
static void launch_type(hipStream_t st, const GemmArgs& a) {
  const uint64_t tiles =
      (uint64_t)((a.n + 31) / 32) * ((a.w.rows + 31) / 32 + (a.w2.rows + 31) / 32 + (a.w3.rows + 31) / 32);
  if (tiles < kTiles32)
    launch_variant<TY, 16>(st, a);
  else
    launch_variant<TY, 32>(st, a);
}

static void launch_gemm_args(hipStream_t st, const GemmArgs& a) {
  switch (a.w.ty) {
    case RLH_TYPE_Q4_K: launch_type<RLH_TYPE_Q4_K>(st, a); break;
    case RLH_TYPE_Q6_K: launch_type<RLH_TYPE_Q6_K>(st, a); break;
    case RLH_TYPE_Q8_0: launch_type<RLH_TYPE_Q8_0>(st, a); break;
    case RLH_TYPE_Q4_0: launch_type<RLH_TYPE_Q4_0>(st, a); break;
    default: break;
  }
}

bool gemm_pair_supported(const DevMat& w, const DevMat& w2) {
  return gemm_supported(w.ty) && w2.ty == w.ty && w2.cols == w.cols;
}

void launch_gemm_pair(hipStream_t st, const DevMat& w, const DevMat& w2, const Q8Tiles& x, uint32_t n, float* y,
                      float* y2, const DevMat* w3, float* y3) {
  GemmArgs a{};
  if (w3) a.w3 = *w3;
  a.y3 = y3;
  a.w = w;
  a.w2 = w2;
  a.x = x;
  a.n = n;
  a.y = y;
  a.y2 = y2;
  launch_gemm_args(st, a);
}

void launch_gemm(hipStream_t st, const DevMat& w, const Q8Tiles& x, uint32_t n, float* y, float* resid) {
  GemmArgs a{};
  a.w = w;
  a.x = x;
  a.n = n;
  a.y = y;
  a.resid = resid;
  launch_gemm_args(st, a);
}

}  // namespace rlh
