// fp32 forward on the fp16 matrix cores (included by c6_forward.hip, whose weight rings, first-layer
// loops and board mapping it shares).
//
// Every fp32 operand is two fp16 values: hi = fp16(v), lo = fp16(2^11 (v - hi)), 11 mantissa bits each.  Of a product's four
// the three largest are accumulated in fp32: hi hi in one sum, hi lo and lo hi, which carry 2^11, in another; lo lo is 2^-22
// of the largest.  Three MFMAs per product where the three exact bf16 parts of c6_split.h take six.
//
// What two parts leave of a number is half a unit of its 24th bit or nothing: v - hi has 13 bits, one or two more than lo.
// Against a 64-bit forward the results are no further off than with six products, because what dominates the error is
// another thing, the rounding of a sum of 864 products at each MFMA (twice: the instruction adds 8 of its 16 products at a
// time), and that is less here:
//  * the sum of the hi hi products is taken per kernel row and the three are added up with fused multiply-adds: a third of the
//    squared error;
//  * an activation's lo is what hi leaves of SiLU's quotient and its correction, not of their sum rounded to fp32;
//  * a weight's lo is rounded such that what the nine taps of a channel leave adds up to nothing (half_taps): what is
//    left of a weight is the same in every square, and the mean over them, the value, would keep it;
//  * the first layer takes a third part of its weights: its inputs are 0 and 1, so one product more of 5 % of the work.
// Relative error of logits / of values against a 64-bit forward (24 networks x 12 boards, rms) with the reference's
// initialisation and PyTorch's, and the mean of a network's logit errors:
//     six products                            4.6e-7 / 1.6e-7   6.9e-8 / 3.7e-8   0.8e-8, 0.5e-8
//     three, as they are here                 4.0e-7 / 0.7e-7   3.5e-8 / 2.5e-8   1.3e-8, 0.2e-8
//     fp32 instructions                       1.4e-6 / 3.7e-7   1.8e-7 / 3.6e-8   7.3e-8, 0.3e-8
// (three products with one sum per layer and every lo rounded to nearest are off by 5.6e-7 and, from the last layer on in 64
// bits, 2.2e-7 with the reference's initialisation; half of what the values gained is their sum over the board in 64 bits.)
//
// fp16 ends at 65504 and is exact to 2^-24 of itself in two parts down to 2^-14; all numbers carry factors for that: weights
// 2^4, activations 2^4 (and -log2(e), as in c6_split.h).  So two parts hold what they should while weights are below 2048 (and
// no less than 2e-13, first layer 2e-10, but for zeros), activations below 1400 and the largest activation of each layer's above 5e-6.  A board for which that does not hold, or
// that has an infinity or a NaN anywhere, is seen at its end: every layer keeps the largest of what it stored (half_note), and a
// weight beyond the range is packed as a NaN (with itself in the other two parts).  Such a board goes through c6_split.h.
//
// What bounds it: the matrix cores, 200 k cycles per board (the 1,890 MFMAs of the 3x3 layers and the first layer's 207 three
// times each) of some 310 k; the epilogues, 22 instructions per output of a lane, go in the open.  2,048 boards 2,117 -> 1,382 us (six
// products with the same structure; both sides on one box), 256 boards 271 -> 184, and in teams (c6_team.h) one board 58 -> 49, 53
// boards 117 -> 98, 128 boards 215 -> 142, of which the launch that looks for boards left over is 4.
#pragma once

namespace c6 {

// Parts of a weight that carries kHalfW: two as above, and what they leave of it, in units of the second (first layer) or times
// 2^11 once more (the others, where it is for split_decode alone).  A weight beyond the range, or so small that the parts would hold
// few of its bits, is a NaN, with itself (the fp32 number `raw`) in the other two.
struct HalfParts {
  unsigned short part[3];
};
__device__ __forceinline__ unsigned short half_bits(float v) { return __builtin_bit_cast(unsigned short, (_Float16)v); }
__device__ __forceinline__ float half_value(unsigned short b) { return (float)__builtin_bit_cast(_Float16, b); }
__device__ __forceinline__ HalfParts half_marked(float raw) {
  const unsigned b = __builtin_bit_cast(unsigned, raw);
  return {{(unsigned short)kHalfMark, (unsigned short)b, (unsigned short)(b >> 16)}};
}
__device__ __forceinline__ bool half_fits(float v) { return __builtin_fabsf(v) <= kHalfMost; }   // (no NaN does)
__device__ __forceinline__ HalfParts half_parts(double w) {
  const double v = w * kHalfW;
  if (!half_fits((float)v) || (w != 0.0 && __builtin_fabs(w) < 0x1p-32)) return half_marked((float)w);
  const unsigned short hi = half_bits((float)v);
  const double rest = (v - half_value(hi)) * kHalfLow;
  const unsigned short lo = half_bits((float)rest);
  return {{hi, lo, half_bits((float)(rest - half_value(lo)))}};
}
// The nine taps of one channel of a 3x3 layer.  Where lo lies half-way between two fp16 numbers it takes the one that makes the
// sum of what the taps leave smaller; then the smallest lo, whose steps are the finest, takes that sum in.
__device__ __forceinline__ void half_taps(const float *w, HalfParts (&out)[9]) {
  float rest[9], sum = 0.0f, least = __builtin_inff();
  int fine = -1;
#pragma unroll
  for (int k = 0; k < 9; ++k) {
    const float v = w[k] * kHalfW;
    if (!half_fits(v) || (w[k] != 0.0f && __builtin_fabsf(w[k]) < 0x1p-42f)) {
      out[k] = half_marked(w[k]);
      continue;
    }
    const unsigned short hi = half_bits(v);
    rest[k] = (v - half_value(hi)) * kHalfLow;
    unsigned short lo = half_bits(rest[k]);
    const float left = rest[k] - half_value(lo);
    // (its neighbour on the other side of the number, as far away if that lies half-way)
    const unsigned short other = (unsigned short)(lo + (((lo >> 15) != 0) == (left > 0.0f) ? -1 : 1));
    if (left != 0.0f && (lo & 0x7fff) != 0 && rest[k] - half_value(other) == -left && __builtin_fabsf(sum - left) < __builtin_fabsf(sum + left))
      lo = other;
    out[k].part[0] = hi;
    out[k].part[1] = lo;
    sum += rest[k] - half_value(lo);
    const float size = __builtin_fabsf(half_value(lo));
    if (size < least) {
      least = size;
      fine = k;
    }
  }
#pragma unroll
  for (int k = 0; k < 9; ++k) {
    if (out[k].part[0] == kHalfMark) continue;
    if (k == fine) out[k].part[1] = half_bits(half_value(out[k].part[1]) + sum);
    out[k].part[2] = half_bits((rest[k] - half_value(out[k].part[1])) * kHalfLow);
  }
}

template <> __device__ __forceinline__ void mma<PrecF32S>(const v4i &a, const v4i &b, f32x16 &c) { mma<PrecF16>(a, b, c); }

// LDS as in SplitGeo (the same addresses behind the tile); a position: hi of 96 channels, lo of 96 channels, 16-byte units
// XORed by split_swz.
struct HalfGeo {
  static constexpr int PIXB = SplitGeo::PIXB, PLANEB = 192;
  static constexpr int CHECK = 44;   // words of RED: [0] half_note's, [1] an input is out of range, [2] one is not small
};

// What a sum over a 3x3 layer's products has to be multiplied by to be the pre-activation times kHalfA
constexpr float kHalfUnit = 1.0f / kHalfW;

// ---- range ----
// What a wave's lanes stored of layer l (m: the largest magnitude of a lane's, NaN if there was one), in one word
__device__ __forceinline__ unsigned half_note(int l, float m) {
  unsigned w = __builtin_amdgcn_ballot_w64(!(m <= (l < 7 ? kHalfMost : 3.4e38f))) != 0 ? 1u : 0u;
  if (l < 7) {
    w |= __builtin_amdgcn_ballot_w64(m >= kHalfLeast) != 0 ? 0x100u << l : 0u;
    w |= __builtin_amdgcn_ballot_w64(m != 0.0f) != 0 ? 0x10000u << l : 0u;
  }
  return w;
}
// ... and whether the words of all of a board's squares and layers, put together, say that it needs c6_split.h: something beyond
// the range, or a layer all of whose outputs are small and not all zero
__device__ __forceinline__ bool half_failed(unsigned w) { return (w & 1u) != 0 || ((w >> 16) & ~(w >> 8) & 0x7fu) != 0; }

// ---- activations ----
// SiLU of eight sums (times kHalfA), step by step (a lone wave waits for each result that its next instruction needs):
// u / (1 + 2^u) by the approximate reciprocal r of the denominator: quotient q, and what it leaves, e (the result is
// q + e r).  Where the denominator is infinite, what it leaves is a NaN, which min() drops, and q is 0.
// LAST: without the factor (the heads' sums end where fp32 does).
template <bool LAST> __device__ __forceinline__ void half_silu8(float (&u)[8], float (&q)[8], float (&e)[8], float (&r)[8]) {
#pragma clang fp contract(off)
  float d[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    d[i] = u[i] * (1.0f / kHalfA);
    if constexpr (LAST) u[i] = d[i];
  }
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int i = 0; i < 8; ++i) d[i] = __builtin_amdgcn_exp2f(d[i]);
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int i = 0; i < 8; ++i) d[i] = 1.0f + d[i];
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int i = 0; i < 8; ++i) r[i] = __builtin_amdgcn_rcpf(d[i]);
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int i = 0; i < 8; ++i) q[i] = u[i] * r[i];
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int i = 0; i < 8; ++i) e[i] = fmaf(-d[i], q[i], u[i]);
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int i = 0; i < 8; ++i) e[i] = fminf(e[i], 0x1p100f);
  __builtin_amdgcn_sched_barrier(0);
}
__device__ __forceinline__ float half_larger(float m, float a, float b) {   // (a NaN stays one)
  return __builtin_elementwise_maximum(m, __builtin_elementwise_maximum(__builtin_fabsf(a), __builtin_fabsf(b)));
}
// Both parts of the activations of eight sums; m: the largest so far
__device__ __forceinline__ void half_store8(float (&u)[8], int (&hi)[4], int (&lo)[4], float &m) {
#pragma clang fp contract(off)
  float q[8], e[8], r[8], minus = -1.0f;
  asm volatile("" : "+s"(minus));   // (q - hi as one instruction that takes hi as it is)
  half_silu8<false>(u, q, e, r);
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    hi[i] = pack2<PrecF16>(q[2 * i], q[2 * i + 1]);
    m = half_larger(m, q[2 * i], q[2 * i + 1]);
  }
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int i = 0; i < 8; ++i) q[i] = fmaf((float)__builtin_bit_cast(f16x2, hi[i / 2])[i % 2], minus, q[i]);
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int i = 0; i < 8; ++i) q[i] = fmaf(e[i], r[i], q[i]);
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int i = 0; i < 8; ++i) q[i] *= kHalfLow;
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int i = 0; i < 4; ++i) lo[i] = pack2<PrecF16>(q[2 * i], q[2 * i + 1]);
  __builtin_amdgcn_sched_barrier(0);
}
// ... of the last layer: the activations themselves, for the heads
__device__ __forceinline__ void half_last8(float (&u)[8], float (&v)[8], float &m) {
#pragma clang fp contract(off)
  float q[8], e[8], r[8];
  half_silu8<true>(u, q, e, r);
#pragma unroll
  for (int i = 0; i < 8; ++i) v[i] = fmaf(e[i], r[i], q[i]);
#pragma unroll
  for (int i = 0; i < 4; ++i) m = half_larger(m, v[2 * i], v[2 * i + 1]);
  __builtin_amdgcn_sched_barrier(0);
}

// ---- the 3x3 layers ----
// Weight ring: k-steps of TN cout tiles and two planes in flight.  The loads take some 800 cycles, a k-step 288 TN.
template <int L, int TN> constexpr int half_ring() {
  constexpr int U = 3 * kCinArr[L] / 16;   // k-steps of a kernel row: 6, 12, 18
  return TN == 2 ? 2 : (U % 3 == 0 ? 3 : 2);
}
template <int L, int TN> using HalfWeights = v4i[half_ring<L, TN>()][TN][2];

template <int L, int T0, int TN> __device__ __forceinline__ void half_preload(HalfWeights<L, TN> &ring, const WFrags &wl) {
  constexpr int NT = kCoutArr[L] / 32;
#pragma unroll
  for (int d = 0; d < half_ring<L, TN>(); ++d)
#pragma unroll
    for (int t = 0; t < TN; ++t)
#pragma unroll
      for (int i = 0; i < 2; ++i) ring[d][t][i] = wl[(d * NT + T0 + t) * 3 + i];
  __builtin_amdgcn_sched_barrier(0);
}

// The contraction of 3x3 layer L, TN of its cout tiles from T0 on.  K runs over kernel rows, the three taps of a row, then 16
// channels at a time; each k-step is nine MFMAs per cout tile: three products of each of three pixel tiles.  The sum of a row's hi hi
// products goes to held at its end, the others' sum, low, runs through.
//   ring: the first k-steps on entry
template <int L, int T0, int TN>
__device__ __forceinline__ void half_conv(const unsigned char *smem, const WFrags &wl, HalfWeights<L, TN> &ring, const int (&ci)[3],
                                          int h, f32x16 (&held)[TN][3], f32x16 (&low)[TN][3]) {
  constexpr int NT = kCoutArr[L] / 32, KC = kCinArr[L] / 16, U = 3 * KC, D = half_ring<L, TN>();
  static_assert(U % D == 0 && U % 2 == 0, "double buffers must line up across rows");
  int at[3][4];   // the lane's squares at a tap: where units 32 k (k = 0 ... 3) of a 128-byte block are
  auto set_tap = [&](int ky, int kx) __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < 3; ++j) {
      const int pos = ci[j] + (ky - 1) * kPitch + (kx - 1);
      const int base = pos * HalfGeo::PIXB, x = (h << 4) ^ split_swz(pos);
#pragma unroll
      for (int k = 0; k < 4; ++k) at[j][k] = base + (x ^ (32 * k));
    }
  };
  v4i a[2][3][2];   // [parity][pixel tile][plane]
  auto read = [&](int c, int par, int j, int i) __attribute__((always_inline)) {
    const int o = i * HalfGeo::PLANEB + c * 32;
    a[par][j][i] = *reinterpret_cast<const v4i *>(smem + at[j][o / 32 % 4] + o / 128 * 128);
  };
  f32x16 sum[TN][3];
#pragma unroll
  for (int t = 0; t < TN; ++t)
#pragma unroll
    for (int j = 0; j < 3; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) held[t][j][e] = low[t][j][e] = 0.0f;
  set_tap(0, 0);
#pragma unroll
  for (int j = 0; j < 3; ++j)
#pragma unroll
    for (int i = 0; i < 2; ++i) read(0, 0, j, i);
#pragma unroll 1
  for (int ky = 0; ky < 3; ++ky) {
    const WFrags wn = wl + ((ky * U + D) * NT + T0) * 3;
    static_for<0, U>([&](auto uc) __attribute__((always_inline)) {
      constexpr int u = decltype(uc)::value, par = u & 1, un = u + 1;
      // (behind the last tap this wraps to the first: harmless extra reads)
      if constexpr (un % KC == 0) set_tap(un < U ? ky : (ky == 2 ? 0 : ky + 1), un < U ? un / KC : 0);
      static_for<0, TN * 9>([&](auto gc) __attribute__((always_inline)) {
        constexpr int g = decltype(gc)::value, t = g / 9, m = g % 9 / 3, j = g % 3;
        // lo hi, hi lo, hi hi (weight, activation)
        if constexpr (m == 0) mma<PrecF16>(ring[u % D][t][1], a[par][j][0], low[t][j]);
        if constexpr (m == 1) mma<PrecF16>(ring[u % D][t][0], a[par][j][1], low[t][j]);
        if constexpr (m == 2) {
          if constexpr (u == 0) sum[t][j] = f32x16{};
          mma<PrecF16>(ring[u % D][t][0], a[par][j][0], sum[t][j]);
        }
        if constexpr (g < 6) read(un % KC, par ^ 1, g / 2, g % 2);
        if constexpr (j == 2 && m == 0) ring[u % D][t][1] = wn[(u * NT + t) * 3 + 1];
        if constexpr (j == 2 && m == 2) ring[u % D][t][0] = wn[(u * NT + t) * 3];
        __builtin_amdgcn_sched_barrier(0);
      });
    });
#pragma unroll
    for (int t = 0; t < TN; ++t)
#pragma unroll
      for (int j = 0; j < 3; ++j) {
        // (out of the accumulation registers here, and not all tiles' at once)
        asm volatile("" : "+a"(sum[t][j]));
#pragma unroll
        for (int e = 0; e < 16; ++e) held[t][j][e] = fmaf(sum[t][j][e], kHalfUnit, held[t][j][e]);
        __builtin_amdgcn_sched_barrier(0);
      }
  }
#pragma unroll
  for (int t = 0; t < TN; ++t)
#pragma unroll
    for (int j = 0; j < 3; ++j) asm volatile("" : "+a"(low[t][j]));
}

// First layer, what the inputs' first parts leave: ROWS rows of K, three fragments of 8 columns each, rowb bytes apart in LDS.
template <int ROWS>
__device__ __forceinline__ void half_second(const unsigned char *smem, const WFrags &wl, const int (&at)[3], int rowb, f32x16 (&low)[1][3]) {
#pragma unroll 1
  for (int row = 0; row < ROWS; ++row)
#pragma unroll
    for (int i = 0; i < 3; ++i) {
      const v4i w = wl[(row * 3 + i) * 3];
#pragma unroll
      for (int j = 0; j < 3; ++j) mma<PrecF16>(w, *reinterpret_cast<const v4i *>(smem + at[j] + row * rowb + i * 16), low[0][j]);
    }
}

// the bias of a cout tile as a lane's registers hold its channels, times kHalfA, and what its rounding to fp32 left
struct HalfBias {
  f32x16 high, low;
};
template <int L> __device__ __forceinline__ HalfBias half_bias(const float *tail, int t, int h) {
  f32x16 b[1], l[1];
  load_bias_tiles(b, tail + bias_offset(L) + 32 * t, h);
  load_bias_tiles(l, tail + Geo<PrecF32S>::TAIL_BIAS_LOW + bias_offset(L) + 32 * t, h);
  return {b[0] * kHalfA, l[0] * kHalfA};
}
// eight outputs' pre-activations (times kHalfA) from register e0 on
__device__ __forceinline__ void half_total8(const f32x16 &held, const f32x16 &small, const HalfBias &b, int e0, float (&u)[8]) {
  f32x16 low = small;
  __builtin_amdgcn_sched_barrier(0);
  asm volatile("" : "+a"(low));
#pragma unroll
  for (int i = 0; i < 8; ++i) u[i] = fmaf(low[e0 + i], kHalfUnit / kHalfLow, b.low[e0 + i]);
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int i = 0; i < 8; ++i) u[i] += held[e0 + i] + b.high[e0 + i];
  __builtin_amdgcn_sched_barrier(0);
}

// one tile's activations, both parts of sixteen channels of the lane's square
struct HalfTile {
  int hi[8], lo[8];
};
typedef int v16i __attribute__((ext_vector_type(16)));
__device__ __forceinline__ void half_put(unsigned char *smem, int pos, int h, int t, const HalfTile &v) {
  const int base = pos * HalfGeo::PIXB + 8 * h, sw = split_swz(pos);
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    *reinterpret_cast<v2i *>(smem + base + ((64 * t + 16 * q) ^ sw)) = v2i{v.hi[2 * q], v.hi[2 * q + 1]};
    *reinterpret_cast<v2i *>(smem + base + ((HalfGeo::PLANEB + 64 * t + 16 * q) ^ sw)) = v2i{v.lo[2 * q], v.lo[2 * q + 1]};
  }
}
template <class U> __device__ __forceinline__ HalfTile half_tile(U sums, float &m) {   // sums(e0, u): eight pre-activations
  HalfTile v;
#pragma unroll
  for (int e0 = 0; e0 < 16; e0 += 8) {
    float u[8];
    int hi[4], lo[4];
    sums(e0, u);
    half_store8(u, hi, lo, m);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      v.hi[e0 / 2 + i] = hi[i];
      v.lo[e0 / 2 + i] = lo[i];
    }
  }
  return v;
}

// one 3x3 layer that is not the last.  Three cout tiles go in two passes over K, two and one (the sums of three would fill the
// registers): the first pass's activations wait in registers until every wave has read its last input.
template <int L>
__device__ __forceinline__ void half_layer(unsigned char *smem, const unsigned char *packed, const float *tail, const int (&ci)[3],
                                           int h, int lane, unsigned &note) {
  constexpr int NT = kCoutArr[L] / 32, TN = NT < 2 ? NT : 2;
  const WFrags wl = layer_weights<PrecF32S, L>(packed, lane);
  float m = 0.0f;
  HalfTile wait[TN][3];
  {
    HalfWeights<L, TN> ring;
    half_preload<L, 0, TN>(ring, wl);
    f32x16 held[TN][3], low[TN][3];
    half_conv<L, 0, TN>(smem, wl, ring, ci, h, held, low);
    if constexpr (NT < 3) __syncthreads();   // every wave has finished reading the layer's input
#pragma unroll
    for (int t = 0; t < TN; ++t) {
      const HalfBias b = half_bias<L>(tail, t, h);
#pragma unroll
      for (int j = 0; j < 3; ++j) {
        wait[t][j] = half_tile([&](int e0, float (&u)[8]) __attribute__((always_inline)) { half_total8(held[t][j], low[t][j], b, e0, u); }, m);
        if constexpr (NT < 3) {
          int pos = ci[j];
          asm volatile("" : "+v"(pos));  // (addresses formed here, not kept for the whole kernel)
          half_put(smem, pos, h, t, wait[t][j]);
        }
      }
    }
  }
  if constexpr (NT == 3) {
    // (in accumulation registers, of which this pass leaves some; the vector ones are short)
    v16i kept[2][3];
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int j = 0; j < 3; ++j) {
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          kept[t][j][i] = wait[t][j].hi[i];
          kept[t][j][8 + i] = wait[t][j].lo[i];
        }
        asm volatile("" : "+a"(kept[t][j]));
      }
    HalfWeights<L, 1> ring;
    half_preload<L, 2, 1>(ring, wl);
    f32x16 held[1][3], low[1][3];
    half_conv<L, 2, 1>(smem, wl, ring, ci, h, held, low);
    __syncthreads();
    const HalfBias b = half_bias<L>(tail, 2, h);
#pragma unroll
    for (int j = 0; j < 3; ++j) {
      int pos = ci[j];
      asm volatile("" : "+v"(pos));
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        v16i v = kept[t][j];
        asm volatile("" : "+a"(v));
        HalfTile w;
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          w.hi[i] = v[i];
          w.lo[i] = v[8 + i];
        }
        half_put(smem, pos, h, t, w);
        __builtin_amdgcn_sched_barrier(0);
      }
      half_put(smem, pos, h, 2, half_tile([&](int e0, float (&u)[8]) __attribute__((always_inline)) { half_total8(held[0][j], low[0][j], b, e0, u); }, m));
    }
  }
  note |= half_note(L, m);
  __syncthreads();
}

// A board that this kernel leaves to split_forward_kernel, which follows it on the stream: a word among its outputs that
// nothing else is (or, from a NaN of the caller's with just these bits, means one board more there).
constexpr unsigned kHalfLeft = 0x7fc0c6c6u;
__device__ __forceinline__ void half_leave(const FwdParams &prm, long long b) {
  if (prm.logits != nullptr) static_cast<unsigned *>(prm.logits)[(size_t)b * kPix] = kHalfLeft;
  else if (prm.value != nullptr) reinterpret_cast<unsigned *>(prm.value)[b] = kHalfLeft;
  else if (prm.actions != nullptr) prm.actions[b] = -1;
}
__device__ __forceinline__ bool half_left(const FwdParams &prm, long long b) {
  if (prm.logits != nullptr) return static_cast<const unsigned *>(prm.logits)[(size_t)b * kPix] == kHalfLeft;
  if (prm.value != nullptr) return reinterpret_cast<const unsigned *>(prm.value)[b] == kHalfLeft;
  return prm.actions != nullptr && prm.actions[b] == -1;
}

// The boards that half_forward_kernel left, one workgroup each; there are hardly ever any, and then this takes 4 us.
template <class P> __global__ __launch_bounds__(256) void split_forward_kernel(const FwdParams prm) {
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  // boards dealt out one by one; every wave looks at the same 64, so that all agree
  const long long grid = gridDim.x;
  for (long long first = blockIdx.x; first < prm.total_boards; first += 64 * grid) {
    const long long mine = first + (threadIdx.x & 63) * grid;
    unsigned long long left = __builtin_amdgcn_ballot_w64(mine < prm.total_boards && half_left(prm, mine));
    if (left != 0) __syncthreads();   // (all have looked before an output is written)
    for (; left != 0; left &= left - 1) split_board(prm, smem, first + __builtin_ctzll(left) * grid);
  }
}

// One workgroup (4 waves) per board, persistent over a contiguous run of boards, as
// fused_forward_kernel.
template <class P>
__global__ __launch_bounds__(256) void half_forward_kernel(const FwdParams prm) {
  using G = Geo<P>;
  using S = SplitGeo;
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  constexpr int THREADS = 256, ROUNDS = (kPix + THREADS - 1) / THREADS;
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = tid >> 6;
  const int h = lane >> 5;
  auto tile_pixel = [](int t, int j) __attribute__((always_inline)) {
    const int p = (t >> 6) * kPixPerWave + j * 32 + (t & 31);
    return p < kPix ? p : (kPix - 1);
  };
  int ci[3];
#pragma unroll
  for (int j = 0; j < 3; ++j) {
    const int pc = tile_pixel(tid, j), r = pc / kBoard;
    ci[j] = (r + 1) * kPitch + (pc - r * kBoard + 1);
  }
  unsigned char *occ = smem + S::OCC_OFF;
  float *lgt = reinterpret_cast<float *>(smem + S::LGT_OFF);
  float *red = reinterpret_cast<float *>(smem + S::RED_OFF);
  int *flags = reinterpret_cast<int *>(red) + 40;   // [0]: third plane varies, [1]: an input is not exact in fp16
  unsigned *check = reinterpret_cast<unsigned *>(red) + HalfGeo::CHECK;

  const unsigned per_group = (unsigned)prm.boards_per_group;
  auto packed_of = [&](long long b) { return prm.packed + (size_t)((unsigned)b / per_group) * prm.packed_stride; };
  float xin[ROUNDS][3];
  unsigned char occin[ROUNDS];
  auto fetch_board = [&](long long b) {
    int tid = threadIdx.x;
    asm volatile("" : "+v"(tid));
    if (prm.x_dtype == C6_DT_BOARD_I8) {
      long long src = prm.index ? prm.index[b] : b;
      src = src < 0 ? 0 : (src >= prm.num_states ? prm.num_states - 1 : src);
      const int8_t *board = reinterpret_cast<const int8_t *>(prm.x) + (size_t)src * kPix;
      const int me = prm.player[src];
      const float last = prm.stones_left[src] == 1 ? 1.0f : 0.0f;
#pragma unroll
      for (int r = 0; r < ROUNDS; ++r) {
        const int p = tid + r * THREADS;
        if (p < kPix) {
          const int stone = board[prm.view ? d4_from_view(p, prm.view) : p];
          xin[r][0] = stone == me ? 1.0f : 0.0f;
          xin[r][1] = stone == -me ? 1.0f : 0.0f;
          xin[r][2] = last;
          occin[r] = 0;
        }
      }
      return;
    }
#pragma unroll
    for (int r = 0; r < ROUNDS; ++r) {
      const int p = tid + r * THREADS;
      if (p < kPix) {
#pragma unroll
        for (int ch = 0; ch < 3; ++ch) xin[r][ch] = load_input_raw(prm.x, prm.x_dtype, ((size_t)b * 3 + ch) * kPix + p);
        occin[r] = prm.mask_mode == C6_MASK_LEGAL ? (prm.legal[(size_t)b * kPix + p] == 0) : 0;
      }
    }
  };

  // (board runs dealt out by XCD, as in fused_pipe_kernel)
  const long long per = (prm.total_boards + gridDim.x - 1) / gridDim.x;
  const unsigned xcds = (gridDim.x % 8 == 0) ? 8 : 1;
  const long long run = (long long)(blockIdx.x % xcds) * (gridDim.x / xcds) + blockIdx.x / xcds;
  long long b = run * per;
  const long long b_end = b + per < prm.total_boards ? b + per : prm.total_boards;
  if (b >= b_end) return;
  v4i r1[L1Pipe<P>::D][1];
  fetch_board(b);

  for (; b < b_end; ++b) {
    int tidv = tid;
    asm volatile("" : "+v"(tidv));
    const unsigned char *packed = packed_of(b);
    const float *tail = reinterpret_cast<const float *>(packed + G::TAIL_OFF);
    unsigned note = 0;
    __syncthreads();  // previous board fully written out; LDS is free
    preload_ring<L1Pipe<P>::D, 1>(r1, packed_frags<P>(packed, lane, G::FAST1_OFF));
    // the third plane's share of the first layer, should the plane be constant (see fused_pipe_kernel)
    f32x16 a0[1][3];
    {
      const WFrags tb = packed_frags<P>(packed, lane, G::PLANE2_FRAG_OFF + __builtin_amdgcn_readfirstlane(wave) * 12);
#pragma unroll
      for (int j = 0; j < 3; ++j)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const f32x4 t4 = __builtin_bit_cast(f32x4, tb[j * 4 + q]);
#pragma unroll
          for (int e = 0; e < 4; ++e) a0[0][j][4 * q + e] = t4[e];
        }
      __builtin_amdgcn_sched_barrier(0);
    }
    // ---- stage the input: zero the shifted copies, then scatter the board ----
    // (16-bit elements, and fp32 ones that count as rounded, become values here, when they have arrived)
    if (prm.x_dtype != C6_DT_F32) {
#pragma unroll
      for (int r = 0; r < ROUNDS; ++r)
#pragma unroll
        for (int ch = 0; ch < 3; ++ch) xin[r][ch] = input_value(xin[r][ch], prm.x_dtype);
    }
    if (tid < 2) flags[tid] = 0;
    if (tid < 3) check[tid] = 0;
    if (tid == 0) red[42] = xin[0][2];   // the third plane's value at square 0
    {
      const v4i z = {0, 0, 0, 0};
      for (int i = tidv * 16; i < G::COPIES_BYTES; i += THREADS * 16) *reinterpret_cast<v4i *>(smem + i) = z;
    }
    __syncthreads();
    const float c2 = red[42];
    {
      bool varies = false;
#pragma unroll
      for (int r = 0; r < ROUNDS; ++r)
        if (tidv + r * THREADS < kPix) varies |= __builtin_bit_cast(int, xin[r][2]) != __builtin_bit_cast(int, c2);
      if (varies) flags[0] = 1;
    }
    __syncthreads();
    const bool plane2_varies = flags[0] != 0;
    const int planes_staged = plane2_varies ? 3 : 2;
    int l1base[3];
#pragma unroll
    for (int j = 0; j < 3; ++j) {
      const int pc = tile_pixel(tidv, j), r = pc / kBoard, c = pc - r * kBoard, s = c % G::E;
      l1base[j] = s * G::COPY_BYTES + ((r * 3 + kL1RowsHalf * ((tidv >> 5) & 1)) * kL1RowPitch + (c - s)) * G::EB;
    }
    f32x16 low[1][3];   // small products
    {
      f32x16 b0[1], bl[1];
      load_bias_tiles(b0, tail + bias_offset(0), h);
      load_bias_tiles(bl, tail + G::TAIL_BIAS_LOW + bias_offset(0), h);
#pragma unroll
      for (int j = 0; j < 3; ++j)
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          a0[0][j][i] = kHalfA * (plane2_varies ? b0[0][i] : fmaf(c2, a0[0][j][i], b0[0][i]));
          low[0][j][i] = kHalfA * kHalfLow * bl[0][i];
        }
    }
    static_assert(kHalfA == kHalfW, "the first layer's sums carry the weights' factor alone, and are the others' units");
    // An input that is exact in fp16 (stones, flags) is one part; what is left of any other is staged behind it, for the
    // products with the weights' first parts, which are small ones.
    auto stage = [&](bool first) __attribute__((always_inline)) {
      bool inexact = false, beyond = false, ordinary = false;
#pragma unroll
      for (int r = 0; r < ROUNDS; ++r) {
        const int p = tidv + r * THREADS;
        if (p < kPix) {
          const int row = p / kBoard, c = p - row * kBoard;
          if (first) {
            unsigned char o = occin[r];
            if (prm.mask_mode == C6_MASK_INPUT) o = (xin[r][0] != 0.0f) || (xin[r][1] != 0.0f);
            occ[p] = o;
          }
#pragma unroll
          for (int ch = 0; ch < 3; ++ch) {
            if (ch >= planes_staged) break;
            const unsigned short v16 = half_bits(xin[r][ch]);
            const float rest = xin[r][ch] - half_value(v16);
            inexact |= rest != 0.0f;
            beyond |= !half_fits(xin[r][ch]);
            ordinary |= __builtin_fabsf(xin[r][ch]) >= kHalfLeast;
            const unsigned short staged = first ? v16 : half_bits(rest * kHalfLow);
            const int hrow = (row + kK1 / 2) * 3 + ch;
#pragma unroll
            for (int s = 0; s < G::E; ++s) {
              const int a = s * G::COPY_BYTES + (hrow * kL1RowPitch + (c + kK1 / 2 - s)) * G::EB;
              *reinterpret_cast<unsigned short *>(smem + a) = staged;
            }
          }
        }
      }
      if (first) {
        if (inexact) flags[1] = 1;
        if (beyond) check[1] = 1;
        if (ordinary) check[2] = 1;
      }
      __syncthreads();
    };
    stage(true);
    if (!plane2_varies) {
      int l1fast[3];
#pragma unroll
      for (int j = 0; j < 3; ++j) l1fast[j] = l1base[j] - (kL1RowsHalf - 1) * h * kL1RowPitch * G::EB;
      conv1_fast_pass<P>(smem, packed_frags<P>(packed, lane, G::FAST1_OFF), r1, l1fast, a0, low);
    } else {
      preload_ring<L1Pipe<P>::D, 1>(r1, layer_weights<P, 0>(packed, lane));
      conv1_pass<P>(smem, layer_weights<P, 0>(packed, lane), r1, l1base, a0, low);
    }
#pragma unroll
    for (int j = 0; j < 3; ++j) asm volatile("" : "+a"(a0[0][j]), "+a"(low[0][j]));
    if (flags[1] != 0) {
      if (check[1] != 0 || check[2] == 0) note |= 1;
      __syncthreads();  // everybody has read the first part
      stage(false);
      if (!plane2_varies) {
        int l1fast[3];
#pragma unroll
        for (int j = 0; j < 3; ++j) l1fast[j] = l1base[j] - (kL1RowsHalf - 1) * h * kL1RowPitch * G::EB;
        half_second<kK1>(smem, packed_frags<P>(packed, lane, G::FAST1_OFF), l1fast, 3 * kL1RowPitch * G::EB, low);
      } else {
        half_second<kL1RowsHalf>(smem, layer_weights<P, 0>(packed, lane), l1base, kL1RowPitch * G::EB, low);
      }
    }
    __syncthreads();
    // the copies overlapped the activation tile: restore its zero padding
    for (int i = tidv; i < 60 * (S::PIXB / 16); i += THREADS) {
      const int k = i / (S::PIXB / 16), w16 = i - k * (S::PIXB / 16);
      const int pos = k < 20 ? k : (k < 41 ? 400 + (k - 20) : (k - 40) * kPitch);
      *reinterpret_cast<v4i *>(smem + pos * S::PIXB + w16 * 16) = v4i{0, 0, 0, 0};
    }
    {
      float m = 0.0f;
#pragma unroll
      for (int j = 0; j < 3; ++j) {
        int pos = ci[j];
        asm volatile("" : "+v"(pos));
        half_put(smem, pos, h, 0, half_tile([&](int e0, float (&u)[8]) __attribute__((always_inline)) {
          f32x16 small = low[0][j], large = a0[0][j];
          __builtin_amdgcn_sched_barrier(0);
          asm volatile("" : "+a"(small), "+a"(large));
#pragma unroll
          for (int i = 0; i < 8; ++i) u[i] = fmaf(small[e0 + i], 1.0f / kHalfLow, large[e0 + i]);
          __builtin_amdgcn_sched_barrier(0);
        }, m));
      }
      note |= half_note(0, m);
    }
    __syncthreads();

    half_layer<1>(smem, packed, tail, ci, h, lane, note);
    half_layer<2>(smem, packed, tail, ci, h, lane, note);
    half_layer<3>(smem, packed, tail, ci, h, lane, note);
    half_layer<4>(smem, packed, tail, ci, h, lane, note);
    half_layer<5>(smem, packed, tail, ci, h, lane, note);
    half_layer<6>(smem, packed, tail, ci, h, lane, note);

    // ---- layer 8 + both 1x1 heads straight from the fp32 accumulators ----
    const float *valw = tail + kBiasTotal + kHeadC;
    {
      float m = 0.0f;
      SplitHeads heads(tail, tidv, lane, wave, h, red);
      const WFrags wl = layer_weights<P, 7>(packed, lane);
      auto pass = [&](auto t0c, auto tnc) __attribute__((always_inline)) {
        constexpr int T0 = decltype(t0c)::value, TN = decltype(tnc)::value;
        HalfWeights<7, TN> ring;
        half_preload<7, T0, TN>(ring, wl);
        f32x16 held[TN][3], low8[TN][3];
        half_conv<7, T0, TN>(smem, wl, ring, ci, h, held, low8);
#pragma unroll
        for (int t = 0; t < TN; ++t) {
          const HalfBias bias = half_bias<7>(tail, T0 + t, h);
          heads.tile(T0 + t, [&](int j, int e0, float (&v)[8]) __attribute__((always_inline)) {
            float u[8];
            half_total8(held[t][j], low8[t][j], bias, e0, u);
            half_last8(u, v, m);
          });
        }
      };
      pass(IC<0>{}, IC<2>{});
      if (b + 1 < b_end) fetch_board(b + 1);  // lands while this board is finished
      pass(IC<2>{}, IC<1>{});
      note |= half_note(7, m);
      if (lane == 0) atomicOr(check, note);
      heads.logits(lgt, valw[kHeadC]);
    }
    __syncthreads();
    if (half_failed(__builtin_amdgcn_readfirstlane(*check))) {
      if (tid == 0) half_leave(prm, b);
    } else {
      split_write(prm, b, tidv, lane, wave, occ, lgt, red, valw[kHeadC + 1]);
    }
  }
}

}  // namespace c6
