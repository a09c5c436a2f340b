// fp32 forward of any board on the bf16 matrix cores (included by c6_forward.hip): the boards and sets of weights whose numbers
// do not fit the two fp16 parts of c6_half.h, which serves all others.
//
// Every fp32 operand is the exact sum of three bf16 values: hi = bf16(v), mid = bf16(v - hi),
// lo = v - hi - mid (8 mantissa bits each, both differences exact).  A product is then nine products
// of bf16 values, each exact in fp32; the six down to 2^-17 of the largest are accumulated in fp32,
// the other three are below 2^-25 of it, less than the rounding of one fp32 addition.
//
// Two sums per output: the products of the two hi in one, the five small products in the other, added
// up at the end.  The matrix instruction drops what lies some eight bits below the last of its sum, towards
// minus infinity: with the small products in the large sum (324 instructions for the 864 products of the
// last layer) that is a bias of 0.77, in units of 2^-24 of the sum's own size, the same in every square,
// which the value head's mean over 361 squares keeps; apart, 0.02, and the scatter is 2.9 in place
// of 7.5 (fp32 instructions: 0.03 and 8.9).
//
// The biases, scaled by -log2(e), are not fp32 numbers any more: the large sum starts with them as fp32, the
// small one with what that leaves.
//
// What bounds it: the matrix cores, 383 k cycles per board with the 1,890 MFMAs of the 3x3 layers
// six times and the first layer's 207 three times (0/1 inputs are exact in one bf16 value); then the
// epilogues, some 25 instructions per output of a lane that one wave per SIMD issues in the open, step by step over eight
// outputs.  The activations of up to 64 channels lie in LDS as their three planes, split once when a layer writes
// them; 96 channels only fit as fp32 (421 positions x 384 bytes are the CU's whole LDS), and the two
// layers that read them split them in registers, 44 instructions for eight values, a few behind each
// MFMA.
//
// An infinity is its own first part; what is left of it is a NaN in the sum of the small products, and the
// large ones alone, which are then infinite or NaN as in fp32 arithmetic, are the result (two_sums).  Parameters and inputs
// have three parts up to the end of fp32;
// a sum or an activation has them up to 2.3e38 (3.39e38, the largest bf16 value, with its factor of 1.44) and
// counts as infinite beyond.
//
// As in the 16-bit modes all activations carry the factor -log2(e), so that SiLU is u / (1 + 2^u); it is
// put in (and taken out behind the heads) with 64 bits, so that nothing is rounded twice for it.
#pragma once

namespace c6 {

template <> __device__ __forceinline__ void mma<PrecF32X>(const v4i &a, const v4i &b, f32x16 &c) { mma<PrecBF16>(a, b, c); }

struct SplitGeo {
  using G = Geo<PrecF32X>;                     // weight stream and first-layer geometry
  static constexpr int PIXB = 384;             // 3 planes x 64 channels x 2 bytes, or 96 x 4
  static constexpr int PLANEB = 128;
  static constexpr int ACT_BYTES = kPos * PIXB;
  static constexpr int OCC_OFF = ACT_BYTES;
  static constexpr int LGT_OFF = OCC_OFF + 384;
  static constexpr int RED_OFF = LGT_OFF + 1456;
  static constexpr int LDS_BYTES = RED_OFF + 48 * 4;
  static_assert(G::COPIES_BYTES <= ACT_BYTES && LDS_BYTES <= 160 * 1024, "LDS map");
};

// 16-byte granule XOR of a position: sixteen consecutive positions read sixteen bank groups
__device__ __forceinline__ int split_swz(int pos) { return ((pos >> 1) & 7) << 4; }

// The heads: sums over the channels, which carry -log2(e), and over all squares.  (In 64 bits, once per square
// and once per board: one rounding each.)
__device__ __forceinline__ float split_logit(float sum, float bias) {
  return (float)((double)sum * (1.0 / kActScale64) + (double)bias);
}
__device__ __forceinline__ float split_value(double sum, float bias) {
  return (float)tanh(sum * (1.0 / kActScale64 / kPix) + (double)bias);
}

// What rounding a pair of values to the bf16 pair `w` leaves out.
__device__ __forceinline__ void split_drop(float &a, float &b, int w) {
#pragma clang fp contract(off)
  a -= __builtin_bit_cast(float, w << 16);
  b -= __builtin_bit_cast(float, w & (int)0xffff0000);
}
// split_drop of four pairs, step by step
__device__ __forceinline__ void split_drop4(float (&v)[8], const int (&w)[4]) {
#pragma clang fp contract(off)
  float r[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) r[e] = __builtin_bit_cast(float, e % 2 ? w[e / 2] & (int)0xffff0000 : w[e / 2] << 16);
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int e = 0; e < 8; ++e) v[e] -= r[e];
}

// Weight ring of a 3x3 layer: two k-steps of all cout tiles and planes.  A k-step of NT cout tiles and N
// pixel tiles is 6 NT N MFMAs, 192 NT N cycles, and a slot is refilled behind its last use.
// (TN of its cout tiles, from T0 on.)
template <int TN> constexpr int kSplitRing = TN == 3 ? 1 : 2;
template <int TN> using SplitWeights = v4i[kSplitRing<TN>][TN][3];

template <int L, int T0, int TN> __device__ __forceinline__ void split_preload(SplitWeights<TN> &ring, const WFrags &wl) {
  constexpr int NT = kCoutArr[L] / 32;
#pragma unroll
  for (int d = 0; d < kSplitRing<TN>; ++d)
#pragma unroll
    for (int t = 0; t < TN; ++t)
#pragma unroll
      for (int i = 0; i < 3; ++i) ring[d][t][i] = wl[(d * NT + T0 + t) * 3 + i];
}

// First layer: ROWS rows of K, three fragments of 8 columns each, rowb bytes apart in LDS; large products to acc, small ones
// to low.  at[j]: where the lane's square of pixel tile j begins.
template <int ROWS>
__device__ __forceinline__ void split_first(const unsigned char *smem, const WFrags &wl, const int (&at)[3], int rowb,
                                            f32x16 (&acc)[1][3], f32x16 (&low)[1][3]) {
  v4i next[3][3];
#pragma unroll
  for (int i = 0; i < 9; ++i) next[i / 3][i % 3] = wl[i];
#pragma unroll 1
  for (int row = 0; row < ROWS; ++row) {
#pragma unroll
    for (int i = 0; i < 3; ++i) {
      v4i w[3];
#pragma unroll
      for (int p = 0; p < 3; ++p) {
        w[p] = next[i][p];
        next[i][p] = wl[((row + 1) * 3 + i) * 3 + p];   // (behind the last row: what follows, unused)
      }
#pragma unroll
      for (int j = 0; j < 3; ++j) {
        const v4i x = *reinterpret_cast<const v4i *>(smem + at[j] + row * rowb + i * 16);
        mma<PrecBF16>(w[0], x, acc[0][j]);
        mma<PrecBF16>(w[1], x, low[0][j]);
        mma<PrecBF16>(w[2], x, low[0][j]);
      }
    }
  }
}

// A product whose sum is in vector registers: the compiler puts every sum of the instruction in accumulation
// registers, and there are 256 of those.  (s_nop: an operand may just have been written by the vector unit.)
// Nothing else may touch such a sum in front of mma_vector_wait: the compiler does not know that it is still being written.
// It has no reason to, since the sums of a layer are written in front of its loop and read behind the wait;
// tests/test_registers.py reads off the built kernel that it did not.
__device__ __forceinline__ void mma_vector(const v4i &a, const v4i &b, f32x16 &c) {
  asm volatile("s_nop 1\n\tv_mfma_f32_32x32x16_bf16 %0, %1, %2, %0" : "+v"(c) : "v"(a), "v"(b));
}
// ... and the wait in front of the first other use of such a sum (the instruction's sixteen passes and what the
// compiler leaves behind them for the sums that it knows of)
__device__ __forceinline__ void mma_vector_wait(f32x16 &a, f32x16 &b) {
  asm volatile("s_nop 15\n\ts_nop 7" : "+v"(a), "+v"(b));
}

// The contraction of 3x3 layer L.  K runs over taps, then 16 channels at a
// time; each k-step is 18 MFMAs per cout tile: six products of each pixel tile.  The five small ones have
// a sum of their own, low, and the large one adds to acc.  Behind each MFMA at most one LDS read of the
// next k-step's activations, one weight load, and (96 input channels) a few instructions of their split.
//   ring: the first k-steps on entry, those behind the layer's last at the end
// The sums of three cout tiles are 288 registers: those of the last pixel tile's last cout tile are vector registers.
// TN of the layer's cout tiles, from T0 on.
template <int L, int T0, int TN>
__device__ __forceinline__ void split_conv(const unsigned char *smem, const WFrags &wl, const float *bias,
                                           SplitWeights<TN> &ring, const int (&ci)[3], int h,
                                           f32x16 (&acc)[TN][3], f32x16 (&low)[TN][3]) {
  constexpr int CIN = kCinArr[L], NT = kCoutArr[L] / 32, KC = CIN / 16, D = kSplitRing<TN>, N = 3;
  constexpr bool WIDE = CIN == 96;   // activations arrive as fp32
  static_assert(KC % 2 == 0 && KC % D == 0, "double buffers must line up across taps");
  int pb[N], xo[N];
  auto set_tap = [&](int tap) __attribute__((always_inline)) {
    const int ky = tap / 3, kx = tap - 3 * ky;
#pragma unroll
    for (int j = 0; j < N; ++j) {
      const int pos = ci[j] + (ky - 1) * kPitch + (kx - 1);
      pb[j] = pos * SplitGeo::PIXB;
      xo[j] = (WIDE ? h << 5 : h << 4) ^ split_swz(pos);
    }
  };
  v4i bq[2][N][3];         // planes of a k-step's activations, [parity][pixel tile][plane]
  f32x4 raw[2][N][2];      // WIDE: the same as fp32, one k-step further ahead
  // part i of pixel tile j of channels 16 c ...: a plane, or (WIDE) four of the eight channels
  auto read = [&](int c, int par, int j, int i) __attribute__((always_inline)) {
    if constexpr (WIDE) {
      if (i < 2)
        raw[par][j][i] = *reinterpret_cast<const f32x4 *>(smem + pb[j] + (c >> 1) * 128 + (xo[j] ^ ((c & 1) * 64 + i * 16)));
    } else {
      bq[par][j][i] = *reinterpret_cast<const v4i *>(smem + pb[j] + (xo[j] ^ (c * 32)) + i * SplitGeo::PLANEB);
    }
  };
  float rest[2];
  auto split_some = [&](int par, auto ac) __attribute__((always_inline)) {  // a quarter of a pair's split
    constexpr int a = decltype(ac)::value, pair = a / 4, j = pair / 4, e = pair % 4;
    if constexpr (a % 4 == 0) {
      rest[0] = raw[par][j][e >> 1][(e & 1) * 2];
      rest[1] = raw[par][j][e >> 1][(e & 1) * 2 + 1];
      bq[par][j][0][e] = pack2<PrecBF16>(rest[0], rest[1]);
    } else if constexpr (a % 4 == 1) {
      split_drop(rest[0], rest[1], bq[par][j][0][e]);
    } else if constexpr (a % 4 == 2) {
      bq[par][j][1][e] = pack2<PrecBF16>(rest[0], rest[1]);
    } else {
      split_drop(rest[0], rest[1], bq[par][j][1][e]);
      bq[par][j][2][e] = pack2<PrecBF16>(rest[0], rest[1]);
    }
  };
  set_tap(0);
#pragma unroll
  for (int j = 0; j < N; ++j)
#pragma unroll
    for (int i = 0; i < 3; ++i) read(0, 0, j, i);
  if constexpr (WIDE) {
#pragma unroll
    for (int j = 0; j < N; ++j)
#pragma unroll
      for (int i = 0; i < 2; ++i) read(1, 1, j, i);
    static_for<0, 16 * N>([&](auto ac) __attribute__((always_inline)) { split_some(0, ac); });
  }
#pragma unroll
  for (int t = 0; t < TN; ++t) {
    f32x16 b[1], bl[1];
    load_bias_tiles(b, bias + 32 * (T0 + t), h);
    load_bias_tiles(bl, bias + Geo<PrecF32X>::TAIL_BIAS_LOW + 32 * (T0 + t), h);
#pragma unroll
    for (int j = 0; j < N; ++j) {
      acc[t][j] = b[0];
      low[t][j] = bl[0];
    }
  }
  constexpr int AHEAD = WIDE ? 2 : 1;
#pragma unroll 1
  for (int tap = 0; tap < 9; ++tap) {
    const WFrags wn = wl + ((tap * KC + D) * NT + T0) * 3;
    static_for<0, KC>([&](auto uc) __attribute__((always_inline)) {
      constexpr int u = decltype(uc)::value, par = u & 1;
      // (after the last tap this wraps to the first: harmless extra reads)
      if constexpr (u + AHEAD == KC) set_tap(tap == 8 ? 0 : tap + 1);
      static_for<0, TN * 6 * N>([&](auto gc) __attribute__((always_inline)) {
        constexpr int g = decltype(gc)::value, t = g / (6 * N), m = (g % (6 * N)) / N, j = g % N;
        constexpr int WP[6] = {0, 1, 2, 0, 1, 0}, AP[6] = {2, 1, 0, 1, 0, 0};
        f32x16 &sum = m < 5 ? low[t][j] : acc[t][j];
        if constexpr (t == 2 && j == 2) mma_vector(ring[u % D][t][WP[m]], bq[par][j][AP[m]], sum);
        else mma<PrecBF16>(ring[u % D][t][WP[m]], bq[par][j][AP[m]], sum);
        if constexpr (WIDE) {
          // raw[par] was split during the k-step before: free for the k-step after next
          if constexpr (g >= 1 && g < 1 + 2 * N) read((u + 2) % KC, par, (g - 1) / 2, (g - 1) % 2);
          constexpr int PER = TN == 1 ? 3 : 1;   // (few MFMAs per k-step: more instructions behind each)
          static_for<PER * g, PER * g + PER>([&](auto ac) __attribute__((always_inline)) {
            if constexpr (decltype(ac)::value < 16 * N) split_some(par ^ 1, ac);
          });
        } else {
          if constexpr (g < 3 * N) read((u + 1) % KC, par ^ 1, g / 3, g % 3);
        }
        // a plane's fragment after its last use in the tile: 2 after product 2, 1 after 4, 0 after 5
        constexpr int done = j == N - 1 ? (m == 2 ? 2 : (m == 4 ? 1 : (m == 5 ? 0 : -1))) : -1;
        if constexpr (done >= 0) {
          ring[u % D][t][done] = wn[(u * NT + t) * 3 + done];
        }
        __builtin_amdgcn_sched_barrier(0);
      });
    });
  }
  if constexpr (TN == 3) {
    mma_vector_wait(acc[2][2], low[2][2]);
#pragma unroll
    for (int k = 0; k < 8; ++k) asm volatile("" : "+a"(acc[k / 3][k % 3]), "+a"(low[k / 3][k % 3]));
  }
}
// The sums of one tile, taken out of the accumulation registers here and not with all the others at once (which is 1,020 bytes of
// scratch a lane, and 3.49 ms for 2,048 boards in place of 2.20)
template <int NT>
__device__ __forceinline__ f32x16 split_total(const f32x16 (&acc)[NT][3], const f32x16 (&low)[NT][3], int t, int j) {
  f32x16 large = acc[t][j], small = low[t][j], sum;
  __builtin_amdgcn_sched_barrier(0);
  if (t == 2 && j == 2) asm volatile("" : "+v"(large), "+v"(small));
  else asm volatile("" : "+a"(large), "+a"(small));
#pragma unroll
  for (int e = 0; e < 16; ++e) sum[e] = large[e] + small[e];
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int e = 0; e < 16; e += 8) {
    bool number[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) number[i] = sum[e + i] == sum[e + i];
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < 8; ++i) sum[e + i] = number[i] ? sum[e + i] : large[e + i];
    __builtin_amdgcn_sched_barrier(0);
  }
  return sum;
}
// SiLU of eight sums from e0 on, step by step (a lone wave waits for each result that its next instruction needs):
// u / (1 + 2^u): the quotient by the approximate reciprocal, then by what it leaves (0.48 ulp rms; by a refined
// reciprocal 0.58).  Where the denominator is infinite, or u is, what it leaves is a NaN, which min() drops: 0 and
// u itself are the results.
__device__ __forceinline__ void split_silu8(const f32x16 &sum, int e0, float (&v)[8]) {
#pragma clang fp contract(off)
  float d[8], r[8], q[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) d[e] = __builtin_amdgcn_exp2f(sum[e0 + e]);
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int e = 0; e < 8; ++e) d[e] = 1.0f + d[e];
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int e = 0; e < 8; ++e) r[e] = __builtin_amdgcn_rcpf(d[e]);
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int e = 0; e < 8; ++e) q[e] = sum[e0 + e] * r[e];
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int e = 0; e < 8; ++e) d[e] = fmaf(-d[e], q[e], sum[e0 + e]);
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int e = 0; e < 8; ++e) d[e] = fminf(d[e], 0x1p100f);
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int e = 0; e < 8; ++e) v[e] = fmaf(d[e], r[e], q[e]);
  __builtin_amdgcn_sched_barrier(0);
}

// The three planes of eight values, step by step
__device__ __forceinline__ void split_planes8(float (&v)[8], int (&w)[3][4]) {
#pragma unroll
  for (int i = 0; i < 3; ++i) {
#pragma unroll
    for (int e = 0; e < 4; ++e) w[i][e] = pack2<PrecBF16>(v[2 * e], v[2 * e + 1]);
    __builtin_amdgcn_sched_barrier(0);
    if (i < 2) {
      split_drop4(v, w[i]);
      __builtin_amdgcn_sched_barrier(0);
    }
  }
}

// SiLU and store of one tile of outputs, in the form the next layer reads.
template <bool PLANES>
__device__ __forceinline__ void split_put(unsigned char *smem, int at, int sw, int h, int t, const f32x16 &sum) {
#pragma unroll
  for (int q = 0; q < 4; q += 2) {
    float v[8];
    split_silu8(sum, 4 * q, v);
    if constexpr (PLANES) {
      int w[3][4];
      split_planes8(v, w);
#pragma unroll
      for (int e = 0; e < 2; ++e) {
        unsigned char *p = smem + at + ((64 * t + 16 * (q + e)) ^ sw) + 8 * h;
#pragma unroll
        for (int i = 0; i < 3; ++i) *reinterpret_cast<v2i *>(p + i * SplitGeo::PLANEB) = v2i{w[i][2 * e], w[i][2 * e + 1]};
      }
    } else {
#pragma unroll
      for (int e = 0; e < 2; ++e)
        *reinterpret_cast<f32x4 *>(smem + at + 128 * t + ((32 * (q + e) + 16 * h) ^ sw)) = f32x4{v[4 * e], v[4 * e + 1], v[4 * e + 2], v[4 * e + 3]};
    }
  }
}
// ... of a layer; sum(t, j): its outputs' sums
template <int NT, bool PLANES, class Sum>
__device__ __forceinline__ void split_store(unsigned char *smem, const int (&ci)[3], int h, Sum sum) {
#pragma unroll
  for (int j = 0; j < 3; ++j) {
    int pos = ci[j];
    asm volatile("" : "+v"(pos));  // (addresses formed here, not kept for the whole kernel)
    const int at = pos * SplitGeo::PIXB, sw = split_swz(pos);
#pragma unroll
    for (int t = 0; t < NT; ++t) split_put<PLANES>(smem, at, sw, h, t, sum(t, j));
  }
}

// one 3x3 layer that is not the last
template <int L>
__device__ __forceinline__ void split_layer(unsigned char *smem, const unsigned char *packed, const float *tail, const int (&ci)[3],
                                            int h, int lane) {
  constexpr int NT = kCoutArr[L] / 32;
  constexpr bool PLANES = kCinArr[L + 1] != 96;
  const WFrags wl = layer_weights<PrecF32X, L>(packed, lane);
  SplitWeights<NT> ring;
  split_preload<L, 0, NT>(ring, wl);
  f32x16 acc[NT][3], low[NT][3];
  split_conv<L, 0, NT>(smem, wl, tail + bias_offset(L), ring, ci, h, acc, low);
  __syncthreads();  // every wave has finished reading the layer's input
  split_store<NT, PLANES>(smem, ci, h, [&](int t, int j) __attribute__((always_inline)) { return split_total<NT>(acc, low, t, j); });
  __syncthreads();
}

// the value head's sum over (cout tile, tile of 32 squares), part(i) of a whole wave's lanes i < 36.  (In 64 bits: 36 additions in
// fp32 were most of the value's error, 2.5e-10 rms of values of 6e-4 with the reference's initialisation.)
template <class Part> __device__ __forceinline__ double split_value_sum(int lane, Part part) {
  return wave_sum_f64(lane < 36 ? (double)part(lane) : 0.0);
}

// ---- what c6_half.h shares ----
// An input value, and whether a square counts as occupied (what the mask of the caller's choice says of it)
__device__ __forceinline__ float board_input(const FwdParams &prm, long long b, int p, int ch) {
  if (prm.x_dtype != C6_DT_BOARD_I8) return load_input(prm.x, prm.x_dtype, ((size_t)b * 3 + ch) * kPix + p);
  long long src = prm.index ? prm.index[b] : b;
  src = src < 0 ? 0 : (src >= prm.num_states ? prm.num_states - 1 : src);
  if (ch == 2) return prm.stones_left[src] == 1 ? 1.0f : 0.0f;
  const int stone = reinterpret_cast<const int8_t *>(prm.x)[(size_t)src * kPix + (prm.view ? d4_from_view(p, prm.view) : p)];
  const int me = prm.player[src];
  return stone == (ch == 0 ? me : -me) ? 1.0f : 0.0f;
}
__device__ __forceinline__ unsigned char board_taken(const FwdParams &prm, long long b, int p, float own, float other) {
  if (prm.mask_mode == C6_MASK_LEGAL) return prm.legal[(size_t)b * kPix + p] == 0;
  return prm.mask_mode == C6_MASK_INPUT && (own != 0.0f || other != 0.0f);
}

// Both heads over a wave's squares.  Partial sums per cout tile and tile of 32 squares, added up in a fixed order: what
// the kernel that shares a board between workgroups can reproduce.
struct SplitHeads {
  int lane, wave, h;
  float *red;
  GlobalF32 pwg;   // the lane's channels of the policy weights: channel 32t + 8q + 4h + e
  int pix[3];
  bool valid[3];
  float tot[3];
  __device__ __forceinline__ SplitHeads(const float *tail, int tid, int lane_, int wave_, int h_, float *red_)
      : lane(lane_), wave(wave_), h(h_), red(red_) {
    const float *pwl = tail + kBiasTotal + 4 * h;
    asm volatile("" : "+v"(pwl));
    pwg = (GlobalF32)pwl;
    int th = tid;
    asm volatile("" : "+v"(th));
#pragma unroll
    for (int j = 0; j < 3; ++j) {
      const int p = (th >> 6) * kPixPerWave + j * 32 + (th & 31);
      valid[j] = p < kPix;
      pix[j] = valid[j] ? p : kPix - 1;
      tot[j] = 0.0f;
    }
  }
  // cout tile t; values(j, e0, v): eight of the activations of the lane's square of pixel tile j, from register e0 on
  template <class V> __device__ __forceinline__ void tile(int t, V values) {
    float pol[3] = {0.0f, 0.0f, 0.0f}, val[3] = {0.0f, 0.0f, 0.0f};
    f32x4 pw[4], vw[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      pw[q] = *(GlobalF32x4)(pwg + 32 * t + 8 * q);
      vw[q] = *(GlobalF32x4)(pwg + kHeadC + 32 * t + 8 * q);
    }
#pragma unroll
    for (int j = 0; j < 3; ++j)
#pragma unroll
      for (int q = 0; q < 4; q += 2) {
        float v[8];
        values(j, 4 * q, v);
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          pol[j] = fmaf(v[e], pw[q + e / 4][e % 4], pol[j]);
          val[j] = fmaf(v[e], vw[q + e / 4][e % 4], val[j]);
        }
      }
    reduce(t, pol, val);
  }
  // ... from a lane's sums over the tile's channels
  __device__ __forceinline__ void reduce(int t, const float (&pol)[3], const float (&val)[3]) {
#pragma unroll
    for (int j = 0; j < 3; ++j) {
      const unsigned bits = __builtin_bit_cast(unsigned, pol[j]);
      const auto r = __builtin_amdgcn_permlane32_swap(bits, bits, false, false);  // the other lane half's channels
      const unsigned r0 = r[0], r1 = r[1];
      const float both = __builtin_bit_cast(float, r0) + __builtin_bit_cast(float, r1);
      tot[j] = t == 0 ? both : tot[j] + both;
      const float vs = wave_sum(valid[j] ? val[j] : 0.0f);
      if (lane == 0) red[t * 12 + 3 * wave + j] = vs;
    }
  }
  __device__ __forceinline__ void logits(float *lgt, float bias) const {
#pragma unroll
    for (int j = 0; j < 3; ++j)
      if (h == 0 && valid[j]) lgt[pix[j]] = split_logit(tot[j], bias);
  }
};

// ---- write out: value, masked logits, optional sampled action ----
__device__ __forceinline__ void split_write(const FwdParams &prm, long long b, int tid, int lane, int wave, const unsigned char *occ,
                                            const float *lgt, const float *red, float value_bias) {
  if (prm.value != nullptr && wave == 3) {   // (beside the draw)
    const double sum = split_value_sum(lane, [&](int i) { return red[i]; });
    if (lane == 0) prm.value[b] = split_value(sum, value_bias);
  }
  if (prm.logits != nullptr) {
    for (int p = tid; p < kPix; p += 256) static_cast<float *>(prm.logits)[(size_t)b * kPix + p] = occ[p] ? prm.fill : lgt[p];
  }
  if (prm.actions != nullptr && wave == 0) {
    float it = prm.inv_temperature;
    asm volatile("" : "+s"(it));
    int a;
    float lp;
    int lane_here = lane;
    asm volatile("" : "+v"(lane_here));
    wave_sample(
        lane_here, prm.u[b], it, [&](int i) { return lgt[i]; }, [&](int i) { return occ[i] == 0; }, a, lp);
    if (lane == 0) {
      prm.actions[b] = a;
      if (prm.logprob != nullptr) prm.logprob[b] = lp;
    }
  }
}

// Board b, by one workgroup of four waves: logits, value and draw, whatever its numbers.
__device__ __forceinline__ void split_board(const FwdParams &prm, unsigned char *smem, long long b) {
  using P = PrecF32X;
  using G = Geo<P>;
  using S = SplitGeo;
  constexpr int THREADS = 256, ROUNDS = (kPix + THREADS - 1) / THREADS;
  int tid = threadIdx.x;
  asm volatile("" : "+v"(tid));   // (nothing of this is formed, or kept, in front of it)
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int h = lane >> 5;
  auto tile_pixel = [](int t, int j, bool &ok) __attribute__((always_inline)) {
    const int p = (t >> 6) * kPixPerWave + j * 32 + (t & 31);
    ok = p < kPix;
    return ok ? p : (kPix - 1);
  };
  int ci[3];
#pragma unroll
  for (int j = 0; j < 3; ++j) {
    bool ok;
    const int pc = tile_pixel(tid, j, ok), r = pc / kBoard;
    ci[j] = (r + 1) * kPitch + (pc - r * kBoard + 1);
  }
  unsigned char *occ = smem + S::OCC_OFF;
  float *lgt = reinterpret_cast<float *>(smem + S::LGT_OFF);
  float *red = reinterpret_cast<float *>(smem + S::RED_OFF);
  int *flags = reinterpret_cast<int *>(red) + 40;   // [0]: third plane varies, [1]: an input is not exact in bf16
  const unsigned char *packed = prm.packed + (size_t)((unsigned)b / (unsigned)prm.boards_per_group) * prm.packed_stride + kSplitOffset;
  const float *tail = reinterpret_cast<const float *>(packed + G::TAIL_OFF);

  float left[ROUNDS][3];   // the input; then what the parts staged so far leave of it
#pragma unroll
  for (int r = 0; r < ROUNDS; ++r) {
    const int p = tid + r * THREADS;
    if (p < kPix)
#pragma unroll
      for (int ch = 0; ch < 3; ++ch) left[r][ch] = board_input(prm, b, p, ch);
  }
  __syncthreads();  // LDS is free
  if (tid < 2) flags[tid] = 0;
  if (tid == 0) red[42] = left[0][2];   // the third plane's value at square 0
  for (int i = tid * 16; i < G::COPIES_BYTES; i += THREADS * 16) *reinterpret_cast<v4i *>(smem + i) = v4i{0, 0, 0, 0};
  __syncthreads();
  const float c2 = red[42];
  bool varies = false;
#pragma unroll
  for (int r = 0; r < ROUNDS; ++r)
    if (tid + r * THREADS < kPix) varies |= __builtin_bit_cast(int, left[r][2]) != __builtin_bit_cast(int, c2);
  if (varies) flags[0] = 1;
  __syncthreads();
  const bool plane2_varies = flags[0] != 0;
  const int planes_staged = plane2_varies ? 3 : 2;
  // An input that is exact in bf16 (stones, flags) is one part; any other goes through the first
  // layer's loop three times, once for each of its bf16 values.
  bool inexact = false;
#pragma unroll
  for (int r = 0; r < ROUNDS; ++r)
    if (tid + r * THREADS < kPix)
#pragma unroll
      for (int ch = 0; ch < 3; ++ch) inexact |= (__builtin_bit_cast(int, left[r][ch]) & 0xffff) != 0 && ch < planes_staged;
  if (inexact) flags[1] = 1;
  __syncthreads();
  const int parts = flags[1] != 0 ? 3 : 1;
  f32x16 a0[1][3], low[1][3], first[1][3];   // large products, small ones; the large ones, once all parts but the first follow
  {
    const WFrags tb = packed_frags<P>(packed, lane, G::PLANE2_FRAG_OFF + wave * 12);
    f32x16 b0[1], bl[1];
    load_bias_tiles(b0, tail + bias_offset(0), h);
    load_bias_tiles(bl, tail + G::TAIL_BIAS_LOW + bias_offset(0), h);
#pragma unroll
    for (int j = 0; j < 3; ++j) {
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const f32x4 t4 = __builtin_bit_cast(f32x4, tb[j * 4 + q]);
#pragma unroll
        for (int e = 0; e < 4; ++e) a0[0][j][4 * q + e] = plane2_varies ? b0[0][4 * q + e] : fmaf(c2, t4[e], b0[0][4 * q + e]);
      }
      low[0][j] = bl[0];
#pragma unroll
      for (int i = 0; i < 16; ++i) first[0][j][i] = 0.0f;
    }
  }
  int l1base[3];
#pragma unroll
  for (int j = 0; j < 3; ++j) {
    bool ok;
    const int pc = tile_pixel(tid, j, ok), r = pc / kBoard, c = pc - r * kBoard, s = c % G::E;
    l1base[j] = s * G::COPY_BYTES + ((r * 3 + (plane2_varies ? kL1RowsHalf : 1) * h) * kL1RowPitch + (c - s)) * G::EB;
  }
#pragma unroll 1
  for (int part = 0; part < parts; ++part) {
    if (part > 0) __syncthreads();  // everybody has read the part before
#pragma unroll
    for (int r = 0; r < ROUNDS; ++r) {
      const int p = tid + r * THREADS;
      if (p < kPix) {
        const int row = p / kBoard, c = p - row * kBoard;
        if (part == 0) occ[p] = board_taken(prm, b, p, left[r][0], left[r][1]);
#pragma unroll
        for (int ch = 0; ch < 3; ++ch) {
          if (ch >= planes_staged) break;
          const unsigned short v16 = bf16_part(left[r][ch]);
          left[r][ch] = bf16_rest(left[r][ch], v16);
          const int hrow = (row + kK1 / 2) * 3 + ch;
#pragma unroll
          for (int s = 0; s < G::E; ++s)
            *reinterpret_cast<unsigned short *>(smem + s * G::COPY_BYTES + (hrow * kL1RowPitch + (c + kK1 / 2 - s)) * G::EB) = v16;
        }
      }
    }
    __syncthreads();
    if (plane2_varies) split_first<kL1RowsHalf>(smem, layer_weights<P, 0>(packed, lane), l1base, kL1RowPitch * G::EB, a0, low);
    else split_first<kK1>(smem, packed_frags<P>(packed, lane, G::FAST1_OFF), l1base, 3 * kL1RowPitch * G::EB, a0, low);
    if (parts > 1 && part == 0) {
#pragma unroll
      for (int j = 0; j < 3; ++j) {
        first[0][j] = a0[0][j];
        a0[0][j] = low[0][j];
#pragma unroll
        for (int i = 0; i < 16; ++i) low[0][j][i] = 0.0f;
      }
    }
  }
  if (parts > 1) {
#pragma unroll
    for (int j = 0; j < 3; ++j)
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        low[0][j][i] += a0[0][j][i];
        a0[0][j][i] = first[0][j][i];
      }
  }
  __syncthreads();
  // the copies overlapped the activation tile: restore its zero padding
  for (int i = tid; i < 60 * (S::PIXB / 16); i += THREADS) {
    const int k = i / (S::PIXB / 16), w16 = i - k * (S::PIXB / 16);
    const int pos = k < 20 ? k : (k < 41 ? 400 + (k - 20) : (k - 40) * kPitch);
    *reinterpret_cast<v4i *>(smem + pos * S::PIXB + w16 * 16) = v4i{0, 0, 0, 0};
  }
  split_store<1, true>(smem, ci, h, [&](int, int j) __attribute__((always_inline)) { return split_total<1>(a0, low, 0, j); });
  __syncthreads();

  split_layer<1>(smem, packed, tail, ci, h, lane);
  split_layer<2>(smem, packed, tail, ci, h, lane);
  split_layer<3>(smem, packed, tail, ci, h, lane);
  split_layer<4>(smem, packed, tail, ci, h, lane);
  split_layer<5>(smem, packed, tail, ci, h, lane);
  split_layer<6>(smem, packed, tail, ci, h, lane);

  // ---- layer 8 + both 1x1 heads straight from the fp32 accumulators ----
  const float *valw = tail + kBiasTotal + kHeadC;
  SplitHeads heads(tail, tid, lane, wave, h, red);
  const WFrags wl = layer_weights<P, 7>(packed, lane);
  SplitWeights<3> ring;
  split_preload<7, 0, 3>(ring, wl);
  f32x16 acc[3][3], low8[3][3];
  split_conv<7, 0, 3>(smem, wl, tail + bias_offset(7), ring, ci, h, acc, low8);
#pragma unroll
  for (int t = 0; t < 3; ++t) {
    f32x16 sum;
    heads.tile(t, [&](int j, int e0, float (&v)[8]) __attribute__((always_inline)) {
      if (e0 == 0) sum = split_total<3>(acc, low8, t, j);
      split_silu8(sum, e0, v);
    });
  }
  heads.logits(lgt, valw[kHeadC]);
  __syncthreads();
  split_write(prm, b, tid, lane, wave, occ, lgt, red, valw[kHeadC + 1]);
}

}  // namespace c6
