// Many boards in the plain 16-bit modes: TWO workgroups per CU, a board each (included by c6_forward.hip,
// whose first-layer loops it shares).
//
// fused_pipe_kernel has one wave per SIMD and hides a layer's SiLU behind the next layer's MFMAs by hand;
// a lone wave issues an instruction about every five cycles, so a third of its 102 k cycles per board the
// matrix cores still wait (epilogue in the open, staging, heads, barriers).  Here a second board's wave on
// the same SIMD fills those gaps by itself, and the kernel can be plain: contraction, barrier, SiLU and
// store, barrier.  What that takes is half of everything: 256 registers per wave (144 of them the
// accumulators of three cout tiles; rings and queues get the rest) and 80 KB of LDS per board.  The
// activations fit in 78.9 KB without padding because they lie granule-major: the 16-byte granules
// (8 channels) of all 421 positions follow one another, then the next granule's.  Neighbouring squares are
// then neighbouring 16-byte words, which no bank conflict disturbs, and both tap and channel of an operand
// are a constant offset from the square's address.
//
// What it measures (bf16; one workgroup per CU on the left): 257 boards 112 -> 86 us, 512 112 -> 105 us,
// 1,024 221 -> 208 us, 4,096 869 -> 818 us; 111 k cycles for a board that has its CU to itself, 91 k for each
// of two.  What bounds it now is the card's power: the shader clock falls from 1.85 to 1.5-1.7 GHz as the
// matrix cores' share rises, 4,096 boards run at 1.38 PFLOP/s where bare MFMAs with random operands sustain
// 1.5-1.9, and neither deeper rings, biases asked for a layer ahead, nor priorities that even out the two
// boards' turns change the time by more than 1 %.
//
// Every accumulator sees the MFMAs of fused_pipe_kernel in its order, every SiLU and sum its operations:
// the results are the same bit for bit.
#pragma once

namespace c6 {

struct DuoGeo {
  static constexpr int GRAN = kPos * 16;         // one granule of every position
  static constexpr int ACT_BYTES = 12 * GRAN;
  static constexpr int OCC_OFF = ACT_BYTES;
  static constexpr int RED_OFF = OCC_OFF + 384;
  static constexpr int LDS_BYTES = RED_OFF + 64;
  static constexpr int LGT_OFF = 0;              // the logits take the tile's place when it has been read
  static_assert(Geo<PrecBF16>::COPIES_BYTES <= ACT_BYTES && 2 * LDS_BYTES <= 160 * 1024, "LDS map");
};

// modes that have this kernel
template <class P> constexpr bool has_duo() { return P::ID == C6_PREC_BF16 || P::ID == C6_PREC_F16; }

// Workgroups of a forward over `boards` boards, all with one workgroup each.  More boards than CUs: two workgroups per CU, where the mode
// has the kernel for it (257 boards take 86 us so, 112 in two rounds of one).  With a CU per board nothing
// shares the matrix cores, and fused_pipe_kernel's 102 k cycles per board beat this kernel's 111 k.
template <class P> inline long long forward_grid(long long boards, int cus) {
  if (boards <= cus) return boards;
  return has_duo<P>() ? 2 * (long long)cus : cus;
}

// The run of boards of one workgroup: the boards are dealt out to the XCDs in contiguous parts
// (workgroup i runs on XCD i % 8, see fused_pipe_kernel), and an XCD's part to its workgroups, the first
// ones taking one board more where it does not divide: those are the ones that have a CU to themselves
// while the others arrive.
struct DuoRun {
  unsigned run, first, count;
  bool second;   // of the two that share a CU
};
__device__ __forceinline__ DuoRun duo_run(unsigned boards, unsigned grid) {
  const unsigned xcds = (grid % 8 == 0) ? 8 : 1, local = grid / xcds;
  const unsigned x = blockIdx.x % xcds, l = blockIdx.x / xcds;
  const unsigned n0 = boards / xcds, n1 = boards % xcds;
  const unsigned part = x * n0 + (x < n1 ? x : n1), n = n0 + (x < n1 ? 1 : 0);
  const unsigned c0 = n / local, c1 = n % local;
  return {x * local + l, part + l * c0 + (l < c1 ? l : c1), c0 + (l < c1 ? 1 : 0), 2 * l >= local};
}

// Depths, in k-steps: weights in flight (they come from L2 in some 800 cycles; a k-step is 96 cycles per
// cout tile, twice that while the other board's wave has its turn) and activation fragments.
template <int L> struct DuoRing {
  static constexpr int NT = kCoutArr[L] / 32, D = NT == 1 ? 6 : 3, S = NT == 3 ? 2 : 3;
};
template <int L> using DuoWeights = v4i[DuoRing<L>::D][DuoRing<L>::NT];

// fragment (k-step k, cout tile t) in the phase-major stream of a 3x3 layer
template <int L> constexpr int duo_frag(int k, int t) {
  constexpr int NT = kCoutArr[L] / 32, LAST = (kCinArr[L] / 32 - 1) * kPhaseSteps;
  if (NT == 1 || k < LAST) return k * NT + t;
  const int u = k - LAST, base = LAST * NT;   // (the last phase has tile 0 in front)
  return t == 0 ? base + u : base + kPhaseSteps + u * (NT - 1) + t - 1;
}

template <int L> __device__ __forceinline__ void duo_preload(DuoWeights<L> &ring, const WFrags &wl) {
  static_for<0, DuoRing<L>::D>([&](auto dc) __attribute__((always_inline)) {
    constexpr int d = decltype(dc)::value;
#pragma unroll
    for (int t = 0; t < DuoRing<L>::NT; ++t) ring[d][t] = wl[duo_frag<L>(d, t)];
  });
}

// The contraction of 3x3 layer L: k-step k is 16 channels of one tap, phase by phase of 32 channels.
template <class P, int L>
__device__ __forceinline__ void duo_conv(const unsigned char *smem, const WFrags &wl, DuoWeights<L> &ring,
                                         const int (&ci)[3], int h, f32x16 (&acc)[kCoutArr[L] / 32][3]) {
  constexpr int NT = kCoutArr[L] / 32, NTP = kCinArr[L] / 32, KS = NTP * kPhaseSteps;
  constexpr int D = DuoRing<L>::D, S = DuoRing<L>::S, GRAN = DuoGeo::GRAN;
  // (the third phase's granules lie beyond the 64 KB that an LDS read's offset reaches)
  int lo[3], hi[3];
#pragma unroll
  for (int j = 0; j < 3; ++j) {
    lo[j] = (ci[j] - (kPitch + 1)) * 16 + h * GRAN;
    asm volatile("" : "+v"(lo[j]));
    hi[j] = lo[j] + 8 * GRAN;
    if constexpr (NTP == 3) asm volatile("" : "+v"(hi[j]));
  }
  v4i a[S][3];
  auto read = [&](auto kc, int j) __attribute__((always_inline)) {
    constexpr int k = decltype(kc)::value, p = k / kPhaseSteps, u = k % kPhaseSteps, tap = u / 2;
    constexpr int off = (4 * (p % 2) + 2 * (u % 2)) * GRAN + ((tap / 3) * kPitch + tap % 3) * 16;
    a[k % S][j] = *reinterpret_cast<const v4i *>(smem + (p < 2 ? lo[j] : hi[j]) + off);
  };
  static_for<0, S - 1>([&](auto kc) __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < 3; ++j) read(kc, j);
  });
  static_for<0, KS>([&](auto kc) __attribute__((always_inline)) {
    constexpr int k = decltype(kc)::value;
    static_for<0, NT * 3>([&](auto gc) __attribute__((always_inline)) {
      constexpr int g = decltype(gc)::value, t = g / 3, j = g % 3;
      mma<P>(ring[k % D][t], a[k % S][j], acc[t][j]);
      if constexpr (g < 3 && k + S - 1 < KS) read(IC<k + S - 1>{}, g);
      if constexpr (j == 2 && k + D < KS) ring[k % D][t] = wl[duo_frag<L>(k + D, t)];
    });
    interleave_step<3 * NT, 3, NT>();
    __builtin_amdgcn_sched_barrier(0);
  });
}

// SiLU, rounding and store of a layer's outputs
template <class P, int NT>
__device__ __forceinline__ void duo_store(unsigned char *smem, const int (&ci)[3], int h, const f32x16 (&acc)[NT][3]) {
#pragma unroll
  for (int j = 0; j < 3; ++j) {
    int at = ci[j] * 16 + 8 * h;
    asm volatile("" : "+v"(at));
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        float v[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = silu<P>(acc[t][j][4 * q + e]);
        *reinterpret_cast<v2i *>(smem + at + (4 * t + q) * DuoGeo::GRAN) = v2i{pack2<P>(v[0], v[1]), pack2<P>(v[2], v[3])};
      }
  }
}

// one 3x3 layer that is not the last; `next`: the ring of the layer behind it
template <class P, int L>
__device__ __forceinline__ void duo_layer(unsigned char *smem, const unsigned char *packed, const float *tail,
                                          DuoWeights<L> &ring, DuoWeights<L + 1> &next, const int (&ci)[3], int h,
                                          int lane) {
  constexpr int NT = kCoutArr[L] / 32;
  f32x16 acc[NT][3];
  init_acc(acc, tail + bias_offset(L), h);
  duo_conv<P, L>(smem, layer_weights<P, L>(packed, lane), ring, ci, h, acc);
  duo_preload<L + 1>(next, layer_weights<P, L + 1>(packed, lane));
  __syncthreads();  // every wave has finished reading the layer's input
  duo_store<P, NT>(smem, ci, h, acc);
  __syncthreads();
}

// This workgroup's run of the boards, dealt out to the first `grid` workgroups of the launch
template <class P, bool REST = false>
__device__ __forceinline__ void duo_boards(const FwdParams &prm, unsigned char *smem, unsigned grid) {
  using G = Geo<P>;
  using S = DuoGeo;
  constexpr int THREADS = 256, ROUNDS = (kPix + THREADS - 1) / THREADS;
  constexpr bool kCanDetect = P::ID == C6_PREC_BF16;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), h = lane >> 5;
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
  int *flag = reinterpret_cast<int *>(red) + 8;   // the third plane varies

  const unsigned per_group = (unsigned)prm.boards_per_group;
  auto packed_of = [&](unsigned b) { return prm.packed + (size_t)(b / per_group) * prm.packed_stride; };
  float xin[ROUNDS][3];
  unsigned char barred[ROUNDS];   // C6_MASK_LEGAL: the square may not be played
  auto fetch_board = [&](unsigned b) __attribute__((always_inline)) {
    int t = threadIdx.x;
    asm volatile("" : "+v"(t));
    long long src = b;
    int me = 0;
    float last = 0.0f;
    const bool state = prm.x_dtype == C6_DT_BOARD_I8;
    if (state) {
      src = prm.index ? prm.index[b] : (long long)b;
      src = src < 0 ? 0 : (src >= prm.num_states ? prm.num_states - 1 : src);
      me = prm.player[src];
      last = prm.stones_left[src] == 1 ? 1.0f : 0.0f;
    }
#pragma unroll
    for (int r = 0; r < ROUNDS; ++r) {
      const int p = t + r * THREADS;
      if (p < kPix) {
        if (state) {
          const int stone = reinterpret_cast<const int8_t *>(prm.x)[(size_t)src * kPix + (prm.view ? d4_from_view(p, prm.view) : p)];
          xin[r][0] = stone == me ? 1.0f : 0.0f;
          xin[r][1] = stone == -me ? 1.0f : 0.0f;
          xin[r][2] = last;
        } else {
#pragma unroll
          for (int ch = 0; ch < 3; ++ch) xin[r][ch] = load_input_raw(prm.x, prm.x_dtype, ((size_t)b * 3 + ch) * kPix + p);
        }
        barred[r] = prm.mask_mode == C6_MASK_LEGAL ? (prm.legal[(size_t)b * kPix + p] == 0) : 0;
      }
    }
  };

  const DuoRun mine = duo_run((unsigned)prm.total_boards, grid);
  const bool detect = kCanDetect && prm.redo_mode == kRedoDetect;
  int listed = 0;   // cascade: boards of this run listed so far (wave 1 counts)
  if (mine.count > 0) fetch_board(mine.first);
  for (unsigned b = mine.first; b < mine.first + mine.count; ++b) {
    int tidv = tid;
    asm volatile("" : "+v"(tidv));
    // (duo_rest_kernel: its place is wanted)
    if (REST && mine.second && b + 1 == mine.first + mine.count) __builtin_amdgcn_s_setprio(2);
    const unsigned char *packed = packed_of(b);
    const float *tail = reinterpret_cast<const float *>(packed + G::TAIL_OFF);
    __syncthreads();  // previous board fully written out; LDS is free
    v4i r1[L1Pipe<P>::D][1];
    preload_ring<L1Pipe<P>::D, 1>(r1, packed_frags<P>(packed, lane, G::FAST1_OFF));
    // the third plane's share of the first layer, should the plane be constant (see fused_pipe_kernel)
    f32x16 a0[1][3];
    {
      const WFrags tb = packed_frags<P>(packed, lane, G::PLANE2_FRAG_OFF + wave * 12);
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
    if (tid == 0) {
      *flag = 0;
      red[9] = xin[0][2];   // the third plane's value at square 0
    }
    {
      const v4i z = {0, 0, 0, 0};
      constexpr int WHOLE = G::COPIES_BYTES / 16 / THREADS;
      unsigned char *zp = smem + tidv * 16;
#pragma unroll
      for (int u = 0; u < WHOLE; ++u) *reinterpret_cast<v4i *>(zp + u * (THREADS * 16)) = z;
      if (tidv * 16 + WHOLE * (THREADS * 16) < G::COPIES_BYTES)
        *reinterpret_cast<v4i *>(zp + WHOLE * (THREADS * 16)) = z;
    }
    __syncthreads();
    const float c2 = red[9];
    {
      bool varies = false;
#pragma unroll
      for (int r = 0; r < ROUNDS; ++r)
        if (tidv + r * THREADS < kPix)
          varies |= __builtin_bit_cast(int, xin[r][2]) != __builtin_bit_cast(int, c2);
      if (varies) *flag = 1;
    }
    __syncthreads();
    const bool plane2_varies = *flag != 0;
#pragma unroll
    for (int r = 0; r < ROUNDS; ++r) {
      const int p = tidv + r * THREADS;
      if (p < kPix) {
        const int row = p / kBoard, c = p - row * kBoard;
        // bit 0: masked in the output; bit 1: not free when the margin is judged
        const bool taken = prm.mask_mode == C6_MASK_LEGAL ? barred[r] != 0 : (xin[r][0] != 0.0f || xin[r][1] != 0.0f);
        occ[p] = (unsigned char)((taken && prm.mask_mode != C6_MASK_NONE ? 1 : 0) | (taken ? 2 : 0));
#pragma unroll
        for (int ch = 0; ch < 3; ++ch) {
          if (ch == 2 && !plane2_varies) break;
          const int hrow = (row + kK1 / 2) * 3 + ch;
          const unsigned short v16 = bits16<P>(xin[r][ch]);
#pragma unroll
          for (int s = 0; s < G::E; ++s) {
            const int a = s * G::COPY_BYTES + (hrow * kL1RowPitch + (c + kK1 / 2 - s)) * G::EB;
            *reinterpret_cast<unsigned short *>(smem + a) = v16;
          }
        }
      }
    }
    __syncthreads();
    // ---- first layer ----
    {
      int l1base[3];
#pragma unroll
      for (int j = 0; j < 3; ++j) {
        bool ok;
        const int pc = tile_pixel(tidv, j, ok), r = pc / kBoard, c = pc - r * kBoard, s = c % G::E;
        l1base[j] = s * G::COPY_BYTES + ((r * 3 + kL1RowsHalf * ((tidv >> 5) & 1)) * kL1RowPitch + (c - s)) * G::EB;
      }
      f32x16 b0[1];
      load_bias_tiles(b0, tail + bias_offset(0), h);
      if (!plane2_varies) {
#pragma unroll
        for (int j = 0; j < 3; ++j)
#pragma unroll
          for (int i = 0; i < 16; ++i) a0[0][j][i] = fmaf(c2, a0[0][j][i], b0[0][i]);
        int l1fast[3];
#pragma unroll
        for (int j = 0; j < 3; ++j) l1fast[j] = l1base[j] - (kL1RowsHalf - 1) * h * kL1RowPitch * G::EB;
        conv1_fast_pass<P>(smem, packed_frags<P>(packed, lane, G::FAST1_OFF), r1, l1fast, a0, a0);
      } else {
#pragma unroll
        for (int j = 0; j < 3; ++j) a0[0][j] = b0[0];
        preload_ring<L1Pipe<P>::D, 1>(r1, layer_weights<P, 0>(packed, lane));
        conv1_pass<P>(smem, layer_weights<P, 0>(packed, lane), r1, l1base, a0, a0);
      }
    }
    DuoWeights<1> w1;
    DuoWeights<2> w2;
    DuoWeights<3> w3;
    DuoWeights<4> w4;
    DuoWeights<5> w5;
    DuoWeights<6> w6;
    DuoWeights<7> w7;
    duo_preload<1>(w1, layer_weights<P, 1>(packed, lane));
    __syncthreads();
    // the copies overlapped the activation tile: restore its zero padding
    for (int i = tidv; i < 60 * 12; i += THREADS) {
      const int g = i / 60, k = i - g * 60;
      // pad positions: 0..19 (top row), 400..420 (bottom row + tail), 20*R (left column)
      const int pos = k < 20 ? k : (k < 41 ? 400 + (k - 20) : (k - 40) * kPitch);
      *reinterpret_cast<v4i *>(smem + g * S::GRAN + pos * 16) = v4i{0, 0, 0, 0};
    }
    duo_store<P, 1>(smem, ci, h, a0);
    __syncthreads();

    duo_layer<P, 1>(smem, packed, tail, w1, w2, ci, h, lane);
    duo_layer<P, 2>(smem, packed, tail, w2, w3, ci, h, lane);
    duo_layer<P, 3>(smem, packed, tail, w3, w4, ci, h, lane);
    duo_layer<P, 4>(smem, packed, tail, w4, w5, ci, h, lane);
    duo_layer<P, 5>(smem, packed, tail, w5, w6, ci, h, lane);
    duo_layer<P, 6>(smem, packed, tail, w6, w7, ci, h, lane);

    // ---- layer 8 + both 1x1 heads straight from the fp32 accumulators ----
    {
      f32x16 acc[3][3];
      init_acc(acc, tail + bias_offset(7), h);
      duo_conv<P, 7>(smem, layer_weights<P, 7>(packed, lane), w7, ci, h, acc);
      if (b + 1 < mine.first + mine.count) fetch_board(b + 1);   // lands behind the heads and the write-out
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
      // (the sums in fused_pipe_kernel's order: tile 0's value sum is one chain per tile of squares,
      // the others' are added up quad by quad)
      float pol[3] = {0.0f, 0.0f, 0.0f}, val0[3] = {0.0f, 0.0f, 0.0f}, vsum = 0.0f;
#pragma unroll
      for (int t = 0; t < 3; ++t) {
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const f32x4 pw = *(GlobalF32x4)(pwg + 32 * t + 8 * q);
          const f32x4 vw = *(GlobalF32x4)(pwg + kHeadC + 32 * t + 8 * q);
#pragma unroll
          for (int j = 0; j < 3; ++j) {
            float vs = t == 0 ? val0[j] : 0.0f;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              const float a = silu<P>(acc[t][j][4 * q + e]);
              pol[j] = fmaf(a, pw[e], pol[j]);
              vs = fmaf(a, vw[e], vs);
            }
            if (t == 0) val0[j] = vs; else vsum += valid[j] ? vs : 0.0f;
          }
        }
        if (t == 0) {
#pragma unroll
          for (int j = 0; j < 3; ++j) vsum += valid[j] ? val0[j] : 0.0f;
        }
      }
      const float polb = valw[kHeadC], valb = valw[kHeadC + 1];
      vsum = wave_sum(vsum);
      if (lane == 0) red[wave] = vsum;
      __syncthreads();  // every wave has read the last layer's input: the logits may take its place
#pragma unroll
      for (int j = 0; j < 3; ++j) {  // add the other lane half's channels
        const unsigned bits = __builtin_bit_cast(unsigned, pol[j]);
        const auto r = __builtin_amdgcn_permlane32_swap(bits, bits, false, false);
        const unsigned r0 = r[0], r1 = r[1];
        const float tot = __builtin_bit_cast(float, r0) + __builtin_bit_cast(float, r1);
        if (h == 0 && valid[j]) lgt[pix[j]] = tot + polb;
      }
      if (tid == 0 && prm.value != nullptr) {
        float s = 0.0f;
#pragma unroll
        for (int w = 0; w < kWaves; ++w) s += red[w];
        prm.value[b] = tanhf(s * (1.0f / kPix) + valb);
      }
      __syncthreads();
    }
    // ---- write out: masked logits, optional sampled action ----
    if (prm.logits != nullptr) {
      for (int p = tidv; p < kPix; p += THREADS) {
        const float v = (occ[p] & 1) ? prm.fill : lgt[p];
        const size_t at = (size_t)b * kPix + p;
        if (prm.logits_dtype == C6_DT_F32) {
          static_cast<float *>(prm.logits)[at] = v;
        } else if (prm.logits_dtype == C6_DT_BF16) {  // (round to nearest even, as Tensor.to does)
          static_cast<unsigned short *>(prm.logits)[at] = __builtin_bit_cast(unsigned short, (__bf16)v);
        } else {
          static_cast<unsigned short *>(prm.logits)[at] = __builtin_bit_cast(unsigned short, (_Float16)v);
        }
      }
    }
    if (prm.actions != nullptr && wave == 0) {
      int a;
      float lp;
      int lane_here = lane;
      asm volatile("" : "+v"(lane_here));
      wave_sample(
          lane_here, prm.u[b], prm.inv_temperature, [&](int i) { return lgt[i]; },
          [&](int i) { return (occ[i] & 1) == 0; }, a, lp);
      if (lane == 0) {
        prm.actions[b] = a;
        if (prm.logprob != nullptr) prm.logprob[b] = lp;
      }
    }
    if (detect && wave == 1) {   // (see fused_pipe_kernel)
      int lane_here = lane;
      asm volatile("" : "+v"(lane_here));
      const bool again = wave_margin_below(
          lane_here, prm.redo_threshold, [&](int i) { return lgt[i]; }, [&](int i) { return (occ[i] & 2) == 0; });
      if (again) {   // (wave-uniform)
        if (lane == 0) prm.redo_list[(size_t)mine.run * prm.redo_per + listed] = (int)b;
        ++listed;
      }
    }
  }
  if (detect && wave == 1 && lane == 0) prm.redo_counts[mine.run] = listed;
}

template <class P> __global__ __launch_bounds__(256, 2) void duo_forward_kernel(const FwdParams prm) {
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  duo_boards<P>(prm, smem, gridDim.x);
}

}  // namespace c6
