// fp32 forward on the bf16 matrix cores (included by c6_forward.hip, whose weight rings, first-layer
// loops and board mapping it shares).
//
// Every fp32 operand is the exact sum of three bf16 values: hi = bf16(v), mid = bf16(v - hi),
// lo = v - hi - mid (8 mantissa bits each, both differences exact).  A product is then nine products
// of bf16 values, each exact in fp32; the six down to 2^-17 of the largest are accumulated in fp32,
// the other three are below 2^-25 of it, less than the rounding of one fp32 addition.  Against the
// fp32 instructions (157 TFLOP/s) six bf16 ones at sixteen times the rate take 3/8 of the time.
//
// Two sums per output: the products of the two hi in one, the five small products in the other, added
// up at the end.  The matrix instruction drops what lies some eight bits below the last of its sum, towards
// minus infinity: with the small products in the large sum (324 instructions for the 864 products of the
// last layer) that is a bias of 0.77, in units of 2^-24 of the sum's own size, the same in every square,
// which the value head's mean over 361 squares keeps; apart, 0.02, and the scatter is 2.9 in place
// of 7.5 (fp32 instructions: 0.03 and 8.9).  Over 64 networks with the reference's initialisation (PyTorch's)
// the value's error against a 64-bit forward is 2.0e-10 (1.5e-9) rms, with fp32 instructions 3.9e-10
// (2.0e-9), its mean per network 5e-11 (3.4e-10) against 2.3e-10 (5.1e-10), and the logits' relative error
// 4.6e-7 (8e-8) against 1.4e-6 (2.0e-7).
//
// The biases, scaled by -log2(e), are not fp32 numbers any more: the large sum starts with them as fp32, the
// small one with what that leaves.  Rounded, they are an error of the same sign in every square: the mean
// of a network's logit errors is then 2.4e-9 of the logits, so 1.1e-9 (fp32 instructions, on parameters as
// they are: 0.7e-9; medians over 256 networks with PyTorch's initialisation).
//
// What bounds it: the matrix cores, 383 k cycles per board with the 1,890 MFMAs of the 3x3 layers
// six times and the first layer's 207 three times (0/1 inputs are exact in one bf16 value); then the epilogues,
// some 25 instructions per output of a lane (two of them at a quarter of the rate) that one wave per SIMD issues in
// the open.  They go step by step over eight outputs, because a lone wave waits wherever an instruction needs the
// one before it (a per cent: 256 boards 281.8 -> 278.6 us, 2,048 boards 2,200 -> 2,184; scratch 200 -> 84 bytes a lane).  The activations of up to 64 channels lie in LDS as their three planes, split once when a layer writes
// them; 96 channels only fit as fp32 (421 positions x 384 bytes are the CU's whole LDS), and the two
// layers that read them split them in registers, 44 instructions for eight values, a few behind each
// MFMA.  2,048 boards take 2.18 ms (2.31 on the same box while the layers of 96 outputs ran in two passes over
// the pixel tiles and read their weights twice, 2.20 in one pass with epilogues output by output; on another 4.35 with
// fp32 instructions).
//
// An infinity is its own first part; what is left of it is a NaN in the sum of the small products, and the
// large ones alone, which are then infinite or NaN as in fp32 arithmetic, are the result (two_sums; 0.4 % of
// the time).  Parameters and inputs have three parts up to the end of fp32;
// a sum or an activation has them up to 2.3e38 (3.39e38, the largest bf16 value, with its factor of 1.44) and
// counts as infinite beyond.
//
// As in the 16-bit modes all activations carry the factor -log2(e), so that SiLU is u / (1 + 2^u); it is
// put in (and taken out behind the heads) with 64 bits, so that nothing is rounded twice for it.
#pragma once

namespace c6 {

template <> __device__ __forceinline__ void mma<PrecF32S>(const v4i &a, const v4i &b, f32x16 &c) {
  mma<PrecBF16>(a, b, c);
}

struct SplitGeo {
  using G = Geo<PrecF32S>;                     // weight stream and first-layer geometry
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
__device__ __forceinline__ float split_value(float sum, float bias) {
  return (float)tanh((double)sum * (1.0 / kActScale64 / kPix) + (double)bias);
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
template <int NT> constexpr int kSplitRing = NT == 3 ? 1 : 2;
template <int L> using SplitWeights = v4i[kSplitRing<kCoutArr[L] / 32>][kCoutArr[L] / 32][3];

template <int NT> __device__ __forceinline__ void split_preload(v4i (&ring)[kSplitRing<NT>][NT][3], const WFrags &wl) {
#pragma unroll
  for (int d = 0; d < kSplitRing<NT>; ++d)
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
      for (int i = 0; i < 3; ++i) ring[d][t][i] = wl[(d * NT + t) * 3 + i];
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
template <int L>
__device__ __forceinline__ void split_conv(const unsigned char *smem, const WFrags &wl, const float *bias,
                                           SplitWeights<L> &ring, const int (&ci)[3], int h,
                                           f32x16 (&acc)[kCoutArr[L] / 32][3], f32x16 (&low)[kCoutArr[L] / 32][3]) {
  constexpr int CIN = kCinArr[L], NT = kCoutArr[L] / 32, KC = CIN / 16, D = kSplitRing<NT>, N = 3;
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
  for (int t = 0; t < NT; ++t) {
    f32x16 b[1], bl[1];
    load_bias_tiles(b, bias + 32 * t, h);
    load_bias_tiles(bl, bias + Geo<PrecF32S>::TAIL_BIAS_LOW + 32 * t, h);
#pragma unroll
    for (int j = 0; j < N; ++j) {
      acc[t][j] = b[0];
      low[t][j] = bl[0];
    }
  }
  constexpr int AHEAD = WIDE ? 2 : 1;
#pragma unroll 1
  for (int tap = 0; tap < 9; ++tap) {
    const WFrags wn = wl + (tap * KC + D) * NT * 3;
    static_for<0, KC>([&](auto uc) __attribute__((always_inline)) {
      constexpr int u = decltype(uc)::value, par = u & 1;
      // (after the last tap this wraps to the first: harmless extra reads)
      if constexpr (u + AHEAD == KC) set_tap(tap == 8 ? 0 : tap + 1);
      static_for<0, NT * 6 * N>([&](auto gc) __attribute__((always_inline)) {
        constexpr int g = decltype(gc)::value, t = g / (6 * N), m = (g % (6 * N)) / N, j = g % N;
        constexpr int WP[6] = {0, 1, 2, 0, 1, 0}, AP[6] = {2, 1, 0, 1, 0, 0};
        f32x16 &sum = m < 5 ? low[t][j] : acc[t][j];
        if constexpr (t == 2 && j == 2) mma_vector(ring[u % D][t][WP[m]], bq[par][j][AP[m]], sum);
        else mma<PrecBF16>(ring[u % D][t][WP[m]], bq[par][j][AP[m]], sum);
        if constexpr (WIDE) {
          // raw[par] was split during the k-step before: free for the k-step after next
          if constexpr (g >= 1 && g < 1 + 2 * N) read((u + 2) % KC, par, (g - 1) / 2, (g - 1) % 2);
          if constexpr (g < 16 * N) split_some(par ^ 1, gc);
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
  if constexpr (NT == 3) {
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

// SiLU and store of one layer's outputs in the form the next one reads.
template <int NT, bool PLANES>
__device__ __forceinline__ void split_store(unsigned char *smem, const int (&ci)[3], int h, const f32x16 (&acc)[NT][3],
                                            const f32x16 (&low)[NT][3]) {
#pragma unroll
  for (int j = 0; j < 3; ++j) {
    int pos = ci[j];
    asm volatile("" : "+v"(pos));  // (addresses formed here, not kept for the whole kernel)
    const int at = pos * SplitGeo::PIXB, sw = split_swz(pos);
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      const f32x16 sum = split_total<NT>(acc, low, t, j);
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
  }
}

// one 3x3 layer that is not the last
template <int L>
__device__ __forceinline__ void split_layer(unsigned char *smem, const unsigned char *packed, const float *tail,
                                            SplitWeights<L> &ring, SplitWeights<L + 1> &next, const int (&ci)[3], int h,
                                            int lane) {
  constexpr int NT = kCoutArr[L] / 32;
  f32x16 acc[NT][3], low[NT][3];
  split_conv<L>(smem, layer_weights<PrecF32S, L>(packed, lane), tail + bias_offset(L), ring, ci, h, acc, low);
  // (with equal widths the over-read has left the next layer's first k-steps in the ring)
  if constexpr (kCoutArr[L + 1] != kCoutArr[L]) split_preload(next, layer_weights<PrecF32S, L + 1>(packed, lane));
  __syncthreads();  // every wave has finished reading the layer's input
  split_store<NT, kCinArr[L + 1] != 96>(smem, ci, h, acc, low);
  __syncthreads();
}

// the value head's sum over (cout tile, tile of 32 squares)
__device__ __forceinline__ float split_value_sum(const float *part) {
  float s = 0.0f;
  for (int i = 0; i < 36; ++i) s += part[i];
  return s;
}

// One workgroup (4 waves) per board, persistent over a contiguous run of boards, as
// fused_forward_kernel.
template <class P>
__global__ __launch_bounds__(256) void split_forward_kernel(const FwdParams prm) {
  using G = Geo<P>;
  using S = SplitGeo;
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  constexpr int THREADS = 256, ROUNDS = (kPix + THREADS - 1) / THREADS;
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = tid >> 6;
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
    if (tid == 0) red[42] = xin[0][2];   // the third plane's value at square 0
    {
      const v4i z = {0, 0, 0, 0};
      for (int i = tidv * 16; i < G::COPIES_BYTES; i += THREADS * 16) *reinterpret_cast<v4i *>(smem + i) = z;
    }
    __syncthreads();
    const float c2 = red[42];
    {
      bool varies = false, inexact = false;
#pragma unroll
      for (int r = 0; r < ROUNDS; ++r)
        if (tidv + r * THREADS < kPix) {
          varies |= __builtin_bit_cast(int, xin[r][2]) != __builtin_bit_cast(int, c2);
#pragma unroll
          for (int ch = 0; ch < 3; ++ch)
            inexact |= (__builtin_bit_cast(int, xin[r][ch]) & 0xffff) != 0 && (ch < 2 || varies);
        }
      if (varies) flags[0] = 1;
      if (inexact) flags[1] = 1;
    }
    __syncthreads();
    const bool plane2_varies = flags[0] != 0;
    const int planes_staged = plane2_varies ? 3 : 2;
    // An input that is exact in bf16 (stones, flags) is one part; any other goes through the first
    // layer's loop three times, once for each of its bf16 values.
    // (a third plane that varies on another thread's squares may be inexact here: look again)
    bool again = false;
    if (plane2_varies) {
#pragma unroll
      for (int r = 0; r < ROUNDS; ++r)
        if (tidv + r * THREADS < kPix) again |= (__builtin_bit_cast(int, xin[r][2]) & 0xffff) != 0;
      if (again) flags[1] = 1;
      __syncthreads();
    }
    const int parts = flags[1] != 0 ? 3 : 1;
    int l1base[3];
#pragma unroll
    for (int j = 0; j < 3; ++j) {
      bool ok;
      const int pc = tile_pixel(tidv, j, ok), r = pc / kBoard, c = pc - r * kBoard, s = c % G::E;
      l1base[j] = s * G::COPY_BYTES + ((r * 3 + kL1RowsHalf * ((tidv >> 5) & 1)) * kL1RowPitch + (c - s)) * G::EB;
    }
    {
      f32x16 b0[1];
      load_bias_tiles(b0, tail + bias_offset(0), h);
#pragma unroll
      for (int j = 0; j < 3; ++j)
#pragma unroll
        for (int i = 0; i < 16; ++i) a0[0][j][i] = plane2_varies ? b0[0][i] : fmaf(c2, a0[0][j][i], b0[0][i]);
    }
    float left[ROUNDS][3];   // what the parts staged so far leave of the input
#pragma unroll
    for (int r = 0; r < ROUNDS; ++r)
#pragma unroll
      for (int ch = 0; ch < 3; ++ch) left[r][ch] = xin[r][ch];
    SplitWeights<1> r2;
    f32x16 low[1][3], first[1][3];   // small products; the large ones, once all parts but the first follow
    {
      f32x16 bl[1];
      load_bias_tiles(bl, tail + G::TAIL_BIAS_LOW + bias_offset(0), h);
#pragma unroll
      for (int j = 0; j < 3; ++j) {
        low[0][j] = bl[0];
#pragma unroll
        for (int i = 0; i < 16; ++i) first[0][j][i] = 0.0f;
      }
    }
#pragma unroll 1
    for (int part = 0; part < parts; ++part) {
      if (part > 0) __syncthreads();  // everybody has read the part before
#pragma unroll
      for (int r = 0; r < ROUNDS; ++r) {
        const int p = tidv + r * THREADS;
        if (p < kPix) {
          const int row = p / kBoard, c = p - row * kBoard;
          if (part == 0) {
            unsigned char o = occin[r];
            if (prm.mask_mode == C6_MASK_INPUT) o = (left[r][0] != 0.0f) || (left[r][1] != 0.0f);
            occ[p] = o;
          }
#pragma unroll
          for (int ch = 0; ch < 3; ++ch) {
            if (ch >= planes_staged) break;
            const unsigned short v16 = bf16_part(left[r][ch]);
            left[r][ch] = bf16_rest(left[r][ch], v16);
            const int hrow = (row + kK1 / 2) * 3 + ch;
#pragma unroll
            for (int s = 0; s < G::E; ++s) {
              const int a = s * G::COPY_BYTES + (hrow * kL1RowPitch + (c + kK1 / 2 - s)) * G::EB;
              *reinterpret_cast<unsigned short *>(smem + a) = v16;
            }
          }
        }
      }
      __syncthreads();
      if (!plane2_varies) {
        int l1fast[3];
#pragma unroll
        for (int j = 0; j < 3; ++j) l1fast[j] = l1base[j] - (kL1RowsHalf - 1) * h * kL1RowPitch * G::EB;
        const WFrags wf = packed_frags<P>(packed, lane, G::FAST1_OFF);
        if (part > 0) preload_ring<L1Pipe<P>::D, 1>(r1, wf);
        conv1_fast_pass<P>(smem, wf, r1, l1fast, a0, low);
      } else {
        preload_ring<L1Pipe<P>::D, 1>(r1, layer_weights<P, 0>(packed, lane));
        conv1_pass<P>(smem, layer_weights<P, 0>(packed, lane), r1, l1base, a0, low);
      }
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
    const long long bn = b + 1;
    if (bn < b_end) fetch_board(bn);  // lands while this board is computed
    split_preload(r2, layer_weights<P, 1>(packed, lane));
    __syncthreads();
    // the copies overlapped the activation tile: restore its zero padding
    for (int i = tidv; i < 60 * (S::PIXB / 16); i += THREADS) {
      const int k = i / (S::PIXB / 16), w16 = i - k * (S::PIXB / 16);
      const int pos = k < 20 ? k : (k < 41 ? 400 + (k - 20) : (k - 40) * kPitch);
      *reinterpret_cast<v4i *>(smem + pos * S::PIXB + w16 * 16) = v4i{0, 0, 0, 0};
    }
    split_store<1, true>(smem, ci, h, a0, low);
    __syncthreads();

    SplitWeights<2> r345;
    SplitWeights<5> r678;
    split_layer<1>(smem, packed, tail, r2, r345, ci, h, lane);
    split_layer<2>(smem, packed, tail, r345, r345, ci, h, lane);
    split_layer<3>(smem, packed, tail, r345, r345, ci, h, lane);
    split_layer<4>(smem, packed, tail, r345, r678, ci, h, lane);
    split_layer<5>(smem, packed, tail, r678, r678, ci, h, lane);
    split_layer<6>(smem, packed, tail, r678, r678, ci, h, lane);

    // ---- layer 8 + both 1x1 heads straight from the fp32 accumulators ----
    {
      f32x16 acc[3][3], low8[3][3];
      split_conv<7>(smem, layer_weights<P, 7>(packed, lane), tail + bias_offset(7), r678, ci, h, acc, low8);
      const float *valw = tail + kBiasTotal + kHeadC;
      const float *pwl = tail + kBiasTotal + 4 * h;  // per-lane base: channel 32t + 8q + 4h + e
      asm volatile("" : "+v"(pwl));
      const GlobalF32 pwg = (GlobalF32)pwl;
      int pix[3];
      bool valid[3];
      int th = tidv;
      asm volatile("" : "+v"(th));
#pragma unroll
      for (int j = 0; j < 3; ++j) pix[j] = tile_pixel(th, j, valid[j]);
      // Partial sums per cout tile and tile of 32 squares, added up in a fixed order: what
      // the kernel that shares a board between workgroups can reproduce.
      float tot[3];
#pragma unroll
      for (int t = 0; t < 3; ++t) {
        float pol[3] = {0.0f, 0.0f, 0.0f}, val[3] = {0.0f, 0.0f, 0.0f};
        f32x4 pw[4], vw[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          pw[q] = *(GlobalF32x4)(pwg + 32 * t + 8 * q);
          vw[q] = *(GlobalF32x4)(pwg + kHeadC + 32 * t + 8 * q);
        }
#pragma unroll
        for (int j = 0; j < 3; ++j) {
          const f32x16 sum = split_total<3>(acc, low8, t, j);
#pragma unroll
          for (int q = 0; q < 4; q += 2) {
            float v[8];
            split_silu8(sum, 4 * q, v);
#pragma unroll
            for (int e = 0; e < 8; ++e) {
              pol[j] = fmaf(v[e], pw[q + e / 4][e % 4], pol[j]);
              val[j] = fmaf(v[e], vw[q + e / 4][e % 4], val[j]);
            }
          }
        }
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
      const float polb = valw[kHeadC], valb = valw[kHeadC + 1];
#pragma unroll
      for (int j = 0; j < 3; ++j)
        if (h == 0 && valid[j]) lgt[pix[j]] = split_logit(tot[j], polb);
      __syncthreads();
      if (tid == 0 && prm.value != nullptr) prm.value[b] = split_value(split_value_sum(red), valb);
    }
    // ---- write out: masked logits, optional sampled action ----
    if (prm.logits != nullptr) {
      for (int p = tidv; p < kPix; p += THREADS)
        static_cast<float *>(prm.logits)[(size_t)b * kPix + p] = occ[p] ? prm.fill : lgt[p];
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
}

}  // namespace c6
