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
//     three, as they are here                 4.0e-7 / 0.8e-7   3.6e-8 / 2.5e-8   1.3e-8, 0.1e-8
//     fp32 instructions                       1.4e-6 / 3.7e-7   1.8e-7 / 3.6e-8   7.3e-8, 0.3e-8
// (three products with one sum per layer and every lo rounded to nearest are off by 5.6e-7 and, from the last layer on in 64
// bits, 2.2e-7 with the reference's initialisation; half of what the values gained is their sum over the board in 64 bits.)
//
// fp16 ends at 65504, and two parts hold a number to 2^-24 of itself down to 2^-14, below that to 2^-36 (the unit of the second
// part's subnormals).  All numbers carry factors for that.  A layer's weights: the power of two that takes the largest of them to
// [2^14, 2^15) (half_scale_kernel), so that they are held to 2^-50 of the largest.  Activations: 2^4 (and -log2(e), as in
// c6_split.h), so that they are held to 2^-24 of themselves or 6e-13.
// What is not held so goes through c6_split.h, which has packed weights of its own:
//  * a set of weights with an infinity, a NaN, or a layer whose weights are too unequal (half_scale_kernel has the rule): known when
//    the set is packed, so that none of its boards starts here;
//  * a board with activations beyond 1400 or none beyond 3.4e-4 in a layer that has any (but for the last), with an infinity or a
//    NaN, seen at its end: every layer keeps the largest of what it stored (half_note).
// What an output's sum loses to small inputs is then at most 2^-20 of it, and that if its weights for all others are 64 times the
// one for the input that is not small.
//
// What bounds it: the matrix cores, 195 k cycles per board (the 1,890 MFMAs of the 3x3 layers and the first layer's 207 three
// times each) of 330 k at 1.9 GHz; what goes in the open is the epilogue of each layer's last cout tile (5 k), the sums at the ends of kernel rows
// and the first operands of each pass (3 to 5 k), and staging (7 k).  2,048 boards, both sides in turn: 2,117 -> 1,382 us from six
// products to three with the same structure, and 2,260 -> 1,436 on another box with all epilogues but the last tile's behind MFMAs and
// three instructions fewer in each (in cycles 350 k -> 330 k; the clock gives back half of it).  In teams (c6_half_team.h) one board 57 ->
// 45 us, 53 boards 114 -> 82, 128 boards 217 -> 134.
#pragma once

namespace c6 {

// Parts of a weight that carries its layer's factor: two as above, and what they leave of it, in units of the second (first layer) or
// times 2^11 once more (the others, where nothing reads it).
struct HalfParts {
  unsigned short part[3];
};
// What layer l's sums have to be multiplied by to be pre-activations (a scalar load, behind its use in no register of a lane's)
__device__ __forceinline__ float half_unit(const float *tail, int l) {
  typedef const __attribute__((address_space(4))) float scalar;
  return *reinterpret_cast<scalar *>(reinterpret_cast<uintptr_t>(tail + Geo<PrecF32S>::TAIL_SW + l));
}
// A power of two's reciprocal
__device__ __forceinline__ float half_inverse(float p) { return __builtin_bit_cast(float, 0x7f000000 - __builtin_bit_cast(int, p)); }
__device__ __forceinline__ unsigned short half_bits(float v) { return __builtin_bit_cast(unsigned short, (_Float16)v); }
__device__ __forceinline__ float half_value(unsigned short b) { return (float)__builtin_bit_cast(_Float16, b); }
__device__ __forceinline__ bool half_fits(float v) { return __builtin_fabsf(v) <= kHalfMost; }   // (no NaN does)
__device__ __forceinline__ HalfParts half_parts(double v) {
  const unsigned short hi = half_bits((float)v);
  const double rest = (v - half_value(hi)) * kHalfLow;
  const unsigned short lo = half_bits((float)rest);
  return {{hi, lo, half_bits((float)(rest - half_value(lo)))}};
}
// The nine taps of one channel of a 3x3 layer.  Where lo lies half-way between two fp16 numbers it takes the one that makes the
// sum of what the taps leave smaller; then the smallest lo, whose steps are the finest, takes that sum in.
__device__ __forceinline__ void half_taps(const float *w, float factor, HalfParts (&out)[9]) {
  float rest[9], sum = 0.0f, least = __builtin_inff();
  int fine = -1;
#pragma unroll
  for (int k = 0; k < 9; ++k) {
    const float v = w[k] * factor;
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
__device__ __forceinline__ float half_larger(float m, float a, float b) {   // (a NaN stays one)
  return __builtin_elementwise_maximum(m, __builtin_elementwise_maximum(__builtin_fabsf(a), __builtin_fabsf(b)));
}
// The epilogue of one tile, a lane's sixteen pre-activations u, as a list of single instructions: SiLU, eight outputs at a time and
// step by step (a lone wave waits for each result that its next instruction needs): u / (1 + 2^u) by the approximate reciprocal r of
// the denominator, quotient q, and what it leaves, e (the result is q + e r).  Where the denominator is infinite, what it
// leaves is a NaN, which min() drops, and q is 0.  Of q + e r come both parts, times kHalfA (by the denominator); in the last layer (LAST)
// the activations themselves, into the heads' sums.  m: the largest magnitude.
struct HalfTemps {
  float d[8], r[8], q[8], e[8];
};
typedef int v16i __attribute__((ext_vector_type(16)));   // both parts of sixteen channels: hi in pairs, then lo
struct HalfHeads {
  float pol, val;
  f32x16 pw, vw;   // the tile's head weights, as a lane's registers hold its channels
};
template <bool LAST> struct HalfEpi {
  static constexpr int GROUP = LAST ? 76 : 84;
  template <int I, class Out>
  __device__ __forceinline__ static void atom(const f32x16 &u, HalfTemps &t, Out &out, float &m, float minus) {
#pragma clang fp contract(off)
    constexpr int k = I % GROUP, x0 = I / GROUP * 8, i = k % 8, p = k % 4;
    if constexpr (k < 8) t.d[i] = __builtin_amdgcn_exp2f(u[x0 + i]);
    else if constexpr (k < 16) t.d[i] = LAST ? 1.0f + t.d[i] : fmaf(t.d[i], 1.0f / kHalfA, 1.0f / kHalfA);
    else if constexpr (k < 24) t.r[i] = __builtin_amdgcn_rcpf(t.d[i]);
    else if constexpr (k < 32) t.q[i] = u[x0 + i] * t.r[i];
    else if constexpr (k < 40) t.e[i] = fmaf(-t.d[i], t.q[i], u[x0 + i]);
    else if constexpr (k < 48) t.e[i] = fminf(t.e[i], 0x1p100f);
    else if constexpr (LAST) {
      if constexpr (k < 56) t.q[i] = fmaf(t.e[i], t.r[i], t.q[i]);
      else if constexpr (k < 60) m = half_larger(m, t.q[2 * p], t.q[2 * p + 1]);
      else if constexpr (k < 68) out.pol = fmaf(t.q[k - 60], out.pw[x0 + k - 60], out.pol);
      else out.val = fmaf(t.q[k - 68], out.vw[x0 + k - 68], out.val);
    } else {
      if constexpr (k < 52) out[x0 / 2 + p] = pack2<PrecF16>(t.q[2 * p], t.q[2 * p + 1]);
      else if constexpr (k < 56) m = half_larger(m, t.q[2 * p], t.q[2 * p + 1]);
      else if constexpr (k < 64) {
        const int hi = out[x0 / 2 + i / 2];
        t.q[i] = fmaf((float)__builtin_bit_cast(f16x2, hi)[i % 2], minus, t.q[i]);
      } else if constexpr (k < 72) t.q[i] = fmaf(t.e[i], t.r[i], t.q[i]);
      else if constexpr (k < 80) t.q[i] *= kHalfLow;
      else out[8 + x0 / 2 + p] = pack2<PrecF16>(t.q[2 * p], t.q[2 * p + 1]);
    }
  }
  // all at once
  template <class Out> __device__ __forceinline__ static void run(const f32x16 &u, Out &out, float &m) {
    float minus = -1.0f;
    asm volatile("" : "+s"(minus));   // (q - hi as one instruction that takes hi as it is)
    HalfTemps t;
    static_for<0, 2 * GROUP>([&](auto ic) __attribute__((always_inline)) {
      constexpr int i = decltype(ic)::value;
      atom<i>(u, t, out, m, minus);
      if constexpr (i % 4 == 3) __builtin_amdgcn_sched_barrier(0);
    });
  }
};
__device__ __forceinline__ v16i half_activations(const f32x16 &u, float &m) {
  v16i out;
  HalfEpi<false>::run(u, out, m);
  return out;
}
__device__ __forceinline__ void half_put(unsigned char *smem, int pos, int h, int t, const v16i &v) {
  const int base = pos * HalfGeo::PIXB + 8 * h, sw = split_swz(pos);
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    *reinterpret_cast<v2i *>(smem + base + ((64 * t + 16 * q) ^ sw)) = v2i{v[2 * q], v[2 * q + 1]};
    *reinterpret_cast<v2i *>(smem + base + ((HalfGeo::PLANEB + 64 * t + 16 * q) ^ sw)) = v2i{v[8 + 2 * q], v[8 + 2 * q + 1]};
  }
}

// ---- the 3x3 layers ----
// words of the tail as a lane's registers hold a cout tile's channels
__device__ __forceinline__ f32x16 half_tail(const float *words, int h) {
  f32x16 v[1];
  load_bias_tiles(v, words, h);
  return v[0];
}
// What a pass over TN cout tiles of layer L, from T0 on, starts with, asked for in front of the epilogue before it: the weights of
// its first k-steps (two planes; the loads take some 800 cycles, a k-step 288 TN) and its biases.
template <int TN> constexpr int kHalfRing = TN == 2 ? 2 : 3;
template <int TN> struct HalfStart {
  v4i ring[kHalfRing<TN>][TN][2];
  f32x16 bias[TN], low[TN];
};
template <int L, int T0, int TN> __device__ __forceinline__ HalfStart<TN> half_start(const unsigned char *packed, const float *tail, int lane) {
  constexpr int NT = kCoutArr[L] / 32;
  const WFrags wl = layer_weights<PrecF32S, L>(packed, lane);
  HalfStart<TN> v;
#pragma unroll
  for (int t = 0; t < TN; ++t) {
    v.bias[t] = half_tail(tail + bias_offset(L) + 32 * (T0 + t), lane >> 5);
    v.low[t] = half_tail(tail + Geo<PrecF32S>::TAIL_BIAS_LOW + bias_offset(L) + 32 * (T0 + t), lane >> 5);
  }
#pragma unroll
  for (int d = 0; d < kHalfRing<TN>; ++d)
#pragma unroll
    for (int t = 0; t < TN; ++t)
#pragma unroll
      for (int i = 0; i < 2; ++i) v.ring[d][t][i] = wl[(d * NT + T0 + t) * 3 + i];
  __builtin_amdgcn_sched_barrier(0);
  return v;
}

// Pixel tiles whose pre-activations wait for their epilogue while a pass over K runs: UN of them per kernel row, the first in the queue,
// a few instructions behind each MFMA, and then to its end as both parts.
template <int UN> struct HalfQueue {
  f32x16 q[3 * UN];
};
struct HalfIdle {};

// The contraction of 3x3 layer L, TN of its cout tiles from T0 on.  K runs over kernel rows, the three taps of a row, then 16
// channels at a time; each k-step is nine MFMAs per cout tile: three products of each of three pixel tiles.  The sum of a row's hi hi
// products goes to held at its end, the others' sum, low, runs through (from what the bias leaves out); at the end held is the
// pre-activation.
template <int L, int T0, int TN, class Queue>
__device__ __forceinline__ void half_conv(const unsigned char *smem, const unsigned char *packed, const float *tail, HalfStart<TN> &start, const int (&ci)[3],
                                          int lane, f32x16 (&held)[TN][3], Queue &queue, float &m) {
  constexpr int NT = kCoutArr[L] / 32, KC = kCinArr[L] / 16, U = 3 * KC, D = kHalfRing<TN>, SLOTS = U * TN * 9;
  static_assert(U % D == 0 && U % 2 == 0, "double buffers must line up across rows");
  constexpr int UN = std::is_same_v<Queue, HalfIdle> ? 0 : sizeof(Queue) / sizeof(f32x16) / 3;
  const int h = lane >> 5;
  const WFrags wl = layer_weights<PrecF32S, L>(packed, lane);
  const float unit = half_unit(tail, L);
  float minus = -1.0f;
  asm volatile("" : "+s"(minus));   // (q - hi as one instruction that takes hi as it is)
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
  f32x16 sum[TN][3], low[TN][3];
#pragma unroll
  for (int t = 0; t < TN; ++t)
#pragma unroll
    for (int j = 0; j < 3; ++j) {
      held[t][j] = start.bias[t];
      low[t][j] = start.low[t];
    }
  set_tap(0, 0);
#pragma unroll
  for (int j = 0; j < 3; ++j)
#pragma unroll
    for (int i = 0; i < 2; ++i) read(0, 0, j, i);
#pragma unroll 1
  for (int ky = 0; ky < 3; ++ky) {
    const WFrags wn = wl + ((ky * U + D) * NT + T0) * 3;
    HalfTemps temps;
    v16i done[UN > 0 ? UN : 1];
    static_for<0, U>([&](auto uc) __attribute__((always_inline)) {
      constexpr int u = decltype(uc)::value, par = u & 1, un = u + 1;
      // (behind the last tap this wraps to the first: harmless extra reads)
      if constexpr (un % KC == 0) set_tap(un < U ? ky : (ky == 2 ? 0 : ky + 1), un < U ? un / KC : 0);
      static_for<0, TN * 9>([&](auto gc) __attribute__((always_inline)) {
        constexpr int g = decltype(gc)::value, t = g / 9, mm = g % 9 / 3, j = g % 3;
        // lo hi, hi lo, hi hi (weight, activation)
        if constexpr (mm == 0) mma<PrecF16>(start.ring[u % D][t][1], a[par][j][0], low[t][j]);
        if constexpr (mm == 1) mma<PrecF16>(start.ring[u % D][t][0], a[par][j][1], low[t][j]);
        if constexpr (mm == 2) {
          if constexpr (u == 0) sum[t][j] = f32x16{};
          mma<PrecF16>(start.ring[u % D][t][0], a[par][j][0], sum[t][j]);
        }
        if constexpr (g < 6) read(un % KC, par ^ 1, g / 2, g % 2);
        if constexpr (j == 2 && mm == 0) start.ring[u % D][t][1] = wn[(u * NT + t) * 3 + 1];
        if constexpr (j == 2 && mm == 2) start.ring[u % D][t][0] = wn[(u * NT + t) * 3];
        if constexpr (UN > 0) {
          using Epi = HalfEpi<false>;
          constexpr int slot = u * TN * 9 + g, N = UN * 2 * Epi::GROUP;
          static_for<slot * N / SLOTS, (slot + 1) * N / SLOTS>([&](auto ac) __attribute__((always_inline)) {
            constexpr int i = decltype(ac)::value, unit = i / (2 * Epi::GROUP);
            Epi::atom<i % (2 * Epi::GROUP)>(queue.q[unit], temps, done[unit], m, minus);
          });
        }
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
        for (int e = 0; e < 16; ++e) held[t][j][e] = fmaf(sum[t][j][e], unit, held[t][j][e]);
        __builtin_amdgcn_sched_barrier(0);
      }
    if constexpr (UN > 0) {
#pragma unroll
      for (int i = 0; i < 2 * UN; ++i) queue.q[i] = queue.q[i + UN];
#pragma unroll
      for (int i = 0; i < UN; ++i) queue.q[2 * UN + i] = __builtin_bit_cast(f32x16, done[i]);
    }
  }
#pragma unroll
  for (int t = 0; t < TN; ++t)
#pragma unroll
    for (int j = 0; j < 3; ++j) {
      asm volatile("" : "+a"(low[t][j]));
#pragma unroll
      for (int e = 0; e < 16; ++e) held[t][j][e] = fmaf(low[t][j][e], unit * (1.0f / kHalfLow), held[t][j][e]);
      __builtin_amdgcn_sched_barrier(0);
    }
}

// one 3x3 layer that is not the last.  Its cout tiles go in two passes over K, all but the last (two at most: the sums of three would
// fill the registers) and the last: behind the second pass's MFMAs go the first one's epilogues, whose activations wait
// in registers until every wave has read the layer's input.
//   start: of the layer's first pass on entry, of the next layer's on return
template <int L, int TN, int TNN>
__device__ __forceinline__ void half_layer(unsigned char *smem, const unsigned char *packed, const float *tail, const int (&ci)[3],
                                           int lane, HalfStart<TN> &start, HalfStart<TNN> &next, unsigned &note) {
  constexpr int NT = kCoutArr[L] / 32;
  static_assert(TN == (NT == 3 ? 2 : 1), "passes");
  const int h = lane >> 5;
  float m = 0.0f;
  f32x16 held[1][3];
  HalfQueue<TN> queue;
  HalfIdle idle;
  if constexpr (NT == 1) {
    half_conv<L, 0, 1>(smem, packed, tail, start, ci, lane, held, idle, m);
  } else {
    f32x16 first[TN][3];
    half_conv<L, 0, TN>(smem, packed, tail, start, ci, lane, first, idle, m);
    HalfStart<1> second = half_start<L, TN, 1>(packed, tail, lane);
#pragma unroll
    for (int t = 0; t < TN; ++t)
#pragma unroll
      for (int j = 0; j < 3; ++j) queue.q[j * TN + t] = first[t][j];
    half_conv<L, TN, 1>(smem, packed, tail, second, ci, lane, held, queue, m);
  }
  next = half_start<L + 1, 0, TNN>(packed, tail, lane);
  __syncthreads();   // every wave has finished reading the layer's input
#pragma unroll
  for (int j = 0; j < 3; ++j) {
    int pos = ci[j];
    asm volatile("" : "+v"(pos));  // (addresses formed here, not kept for the whole kernel)
    if constexpr (NT > 1) {
#pragma unroll
      for (int t = 0; t < TN; ++t) half_put(smem, pos, h, t, __builtin_bit_cast(v16i, queue.q[j * TN + t]));
    }
    half_put(smem, pos, h, NT - 1, half_activations(held[0][j], m));
  }
  note |= half_note(L, m);
  __syncthreads();
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

// Whether a workgroup of half_forward_kernel does a board that it cannot hold again itself: where that is its only one.  A launch of
// split_forward_kernel, which looks for such boards and hardly ever finds one, takes 4 us: 129 boards 150.5 -> 147 us, 256
// boards 190.2 -> 187.1 us, 384 boards (128 of them in teams) 322 -> 318.5 us.  Behind more boards each the launch stays: up to eight done again where
// they ended gain as much, 512 boards 366.7 -> 363.6 us, 2,048 boards 1,427 -> 1,423 us, but a weight set beyond the range, whose boards
// lie side by side, would go through few workgroups one after the other.
__host__ __device__ inline bool half_redone(long long per_workgroup) { return per_workgroup == 1; }

// The boards that half_forward_kernel left, one workgroup each.  (Teams do without: team_forward_kernel.)
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
  bool again = false;
  // A set of weights that two parts do not hold: none of its boards starts here, but where a run has boards of other sets too.
  // (256 boards of such a set 445 -> 283 us, 2,048 boards 3,660 -> 2,260 us.)
  auto unheld = [&](const unsigned char *packed) __attribute__((always_inline)) {
    bool none = false;
#pragma unroll
    for (int l = 0; l < 8; ++l) none |= half_unit(reinterpret_cast<const float *>(packed + G::TAIL_OFF), l) == 0.0f;
    return none;
  };
  {
    bool all = true;
    for (long long i = b; all && i < b_end; i = ((unsigned)i / per_group + 1ll) * per_group) all = unheld(packed_of(i));
    if (all) {
      again = half_redone(per);
      for (long long i = b + tid; !again && i < b_end; i += THREADS) half_leave(prm, i);
      b = b_end;
    }
  }
  if (b < b_end) fetch_board(b);

  for (; b < b_end; ++b) {
    int tidv = tid;
    asm volatile("" : "+v"(tidv));
    const unsigned char *packed = packed_of(b);
    const float *tail = reinterpret_cast<const float *>(packed + G::TAIL_OFF);
    unsigned note = unheld(packed) ? 1 : 0;
    __syncthreads();  // previous board fully written out; LDS is free
    preload_ring<L1Pipe<P>::D, 1>(r1, packed_frags<P>(packed, lane, G::FAST1_OFF));
    const float unit0 = half_unit(tail, 0);
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
      const float factor = half_inverse(unit0);
#pragma unroll
      for (int j = 0; j < 3; ++j)
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          a0[0][j][i] = factor * (plane2_varies ? b0[0][i] : fmaf(c2, a0[0][j][i], b0[0][i]));
          low[0][j][i] = bl[0][i];
        }
    }
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
    HalfStart<1> one = half_start<1, 0, 1>(packed, tail, lane);
    HalfStart<2> two;
    {
      float m = 0.0f;
#pragma unroll
      for (int j = 0; j < 3; ++j) {
        int pos = ci[j];
        asm volatile("" : "+v"(pos));
        f32x16 small = low[0][j], large = a0[0][j], u;
        __builtin_amdgcn_sched_barrier(0);
        asm volatile("" : "+a"(small), "+a"(large));
#pragma unroll
        for (int i = 0; i < 16; ++i) u[i] = fmaf(small[i], unit0 * (1.0f / kHalfLow), large[i] * unit0);
        half_put(smem, pos, h, 0, half_activations(u, m));
      }
      note |= half_note(0, m);
    }
    __syncthreads();

    half_layer<1>(smem, packed, tail, ci, lane, one, one, note);
    half_layer<2>(smem, packed, tail, ci, lane, one, one, note);
    half_layer<3>(smem, packed, tail, ci, lane, one, one, note);
    half_layer<4>(smem, packed, tail, ci, lane, one, two, note);
    half_layer<5>(smem, packed, tail, ci, lane, two, two, note);
    half_layer<6>(smem, packed, tail, ci, lane, two, two, note);

    // ---- layer 8 + both 1x1 heads ----
    const float *valw = tail + kBiasTotal + kHeadC;
    {
      float m = 0.0f;
      HalfIdle idle;
      SplitHeads heads(tail, tidv, lane, wave, h, red);
      auto head = [&](int t, const f32x16 (&u)[3]) __attribute__((always_inline)) {
        HalfHeads out;
        out.pw = half_tail(tail + kBiasTotal + 32 * t, h);
        out.vw = half_tail(tail + kBiasTotal + kHeadC + 32 * t, h);
        float pol[3], val[3];
#pragma unroll
        for (int j = 0; j < 3; ++j) {
          out.pol = out.val = 0.0f;
          HalfEpi<true>::run(u[j], out, m);
          pol[j] = out.pol;
          val[j] = out.val;
        }
        heads.reduce(t, pol, val);
      };
      {
        f32x16 u[2][3];
        half_conv<7, 0, 2>(smem, packed, tail, two, ci, lane, u, idle, m);
        one = half_start<7, 2, 1>(packed, tail, lane);
        head(0, u[0]);
        head(1, u[1]);
      }
      if (b + 1 < b_end) fetch_board(b + 1);  // lands while this board is finished
      f32x16 u[1][3];
      half_conv<7, 2, 1>(smem, packed, tail, one, ci, lane, u, idle, m);
      head(2, u[0]);
      note |= half_note(7, m);
      if (lane == 0) atomicOr(check, note);
      heads.logits(lgt, valw[kHeadC]);
    }
    __syncthreads();
    if (half_failed(__builtin_amdgcn_readfirstlane(*check))) {
      again = half_redone(per);
      if (!again && tid == 0) half_leave(prm, b);
    } else {
      split_write(prm, b, tidv, lane, wave, occ, lgt, red, valw[kHeadC + 1]);
    }
  }
  if (again) split_board(prm, smem, run);   // (its only board)
}

}  // namespace c6
