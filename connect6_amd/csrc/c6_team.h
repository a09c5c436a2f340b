// Few boards: a TEAM of workgroups per board (included by c6_forward.hip).
//
// One workgroup per board leaves most of the chip idle when there are fewer boards than CUs, and a
// single board takes as long as 256.  Here 9 (or 3) workgroups share a board: workgroup (s, t) takes
// the third s of the squares (a wave: 32 of them) and, with 9, cout tile t of every layer; with 3 it
// takes all cout tiles.  A layer's outputs go to memory as the next layer reads them, a flag says
// that they are there, and every workgroup loads the rows it needs (its own and one above and below)
// into LDS.  Each accumulator sees the same MFMAs in the same order as in the one-workgroup kernels,
// so the results are the same bit for bit.
//
// The exchange: stores and loads of the activations carry the device-scope cache policy (sc1), the
// flags are relaxed device-scope atomics behind a wait for the stores.  Measured between two
// workgroups: 0.8-0.95 us for a flag, 1.5 us with 4 KB behind it, the same within an XCD and across.
//
// What it costs and gives (fp32, one board, nine workgroups, 76 us against 201 us): per layer 0.6 us
// to see a flag that is already set, 1.8-2.6 us to bring 190 squares from memory into LDS, 1.8 us until
// the stores are acknowledged, and 2-5 us of MFMAs (each wave has one 32 x 32 tile, and its weights
// saturate the L1's 64 bytes a cycle); 53 boards with three workgroups each take 128 us (208 us).
//
// Nothing waits for a workgroup that may not be running: a wait is bounded, and a workgroup whose
// wait runs out does the missing piece of work itself (the earliest one that has no flag; everything
// in front of it has one).  Outputs of every layer have a place of their own, and whoever computes
// a piece writes the same bytes, so doing one twice is harmless; any single workgroup can finish the
// board alone.  The flags of a call are the call's tag: the caller hands a tag that the flag words
// have not held before (or words that are zero).
#pragma once

namespace c6 {

constexpr int kTeamStages = 9;                   // eight layers, then the heads' write-out
constexpr int kSc1 = 16;                         // cache policy: device scope

template <class P> struct TeamGeo {
  using G = Geo<P>;
  static constexpr int NPL = P::ID == C6_PREC_F32S ? 3 : 1;   // planes of an activation
  static constexpr int PXB = NPL * 64;                        // bytes of a square's 32 channels in memory
  static constexpr int BLOCKB = kPix * PXB;                   // one cout tile of one layer
  // memory per board: the outputs of layers 1 .. 7, then the heads' partial sums
  static constexpr int act_off(int l) {
    int s = 0;
    for (int i = 0; i < l; ++i) s += kCoutArr[i] / 32 * BLOCKB;
    return s;
  }
  static constexpr int HEAD_OFF = act_off(7);                 // [3][384] policy, then values
  static constexpr int VAL_OFF = HEAD_OFF + 3 * 384 * 4;
  static constexpr int BOARDB = (VAL_OFF + 1024 * 4 + 255) & ~255;
  // LDS: up to 11 rows of positions (a third of the squares lies in at most 8 board rows)
  static constexpr int RECB = NPL * 192 + 16;
  static constexpr int REGION = (11 * kPitch + 1) * RECB;
  static constexpr int BUF = REGION > G::COPIES_BYTES ? REGION : G::COPIES_BYTES;
  static constexpr int OCC_OFF = (BUF + 15) & ~15;
  static constexpr int LGT_OFF = OCC_OFF + 384;
  static constexpr int RED_OFF = LGT_OFF + 1456;
  static constexpr int LDS_BYTES = RED_OFF + 256;
  static_assert(LDS_BYTES <= 160 * 1024, "LDS map");
};

// fragment (k-step k, cout tile t) of 3x3 layer L in the weight stream of mode P: first of its planes
template <class P, int L> __device__ __forceinline__ int team_frag(int k, int t) {
  constexpr int NT = kCoutArr[L] / 32, NTP = kCinArr[L] / 32;
  if constexpr (P::PIPE) {  // phase-major, the last phase tile 0 first (pipe_frag)
    const int last = (NTP - 1) * kPhaseSteps;
    if (NT > 1 && k >= last) {
      const int u = k - last, base = last * NT;
      return (t == 0 ? base + u : base + kPhaseSteps + u * (NT - 1) + t - 1) * Geo<P>::W;
    }
  }
  return (k * NT + t) * Geo<P>::W;
}

// The contraction of 3x3 layer L for one tile of 32 squares and TT cout tiles from t0 on.  rec: LDS
// address of the lane's square's record one row and one column up, + 16 * lane half.
template <class P, int L, int TT>
__device__ __forceinline__ void team_conv(const unsigned char *smem, const WFrags &wl,
                                          v4i (&ring)[(Geo<P>::W == 3 ? 6 : 18) / TT][TT][Geo<P>::W], int rec, int t0, f32x16 (&acc)[TT]) {
  using T = TeamGeo<P>;
  constexpr int W = Geo<P>::W, NPL = T::NPL, D = (W == 3 ? 6 : 18) / TT;
  constexpr int KC = kCinArr[L] / 16, KS = 9 * KC;
  constexpr int U = P::PIPE ? kPhaseSteps : 3 * KC;     // k-steps of one unrolled round
  static_assert(KS % U == 0 && U % D == 0, "ring");
  // k-step v of round r: (tap, 16 channels)
  auto frag = [&](int r, int v, int pl) __attribute__((always_inline)) {
    const int tap = P::PIPE ? v / 2 : 3 * r + v / KC;
    const int ch = P::PIPE ? 32 * r + 16 * (v % 2) : 16 * (v % KC);
    const int off = P::PIPE ? ((tap / 3) * kPitch + tap % 3) * T::RECB + (v % 2) * 32
                            : (v / KC) * T::RECB + ch * 2;
    const int base = P::PIPE ? r * 64 : r * kPitch * T::RECB;
    return *reinterpret_cast<const v4i *>(smem + rec + base + off + pl * 192);
  };
  v4i a[3][NPL];
#pragma unroll
  for (int v = 0; v < 2; ++v)
#pragma unroll
    for (int i = 0; i < NPL; ++i) a[v][i] = frag(0, v, i);
#pragma unroll 1
  for (int r = 0; r < KS / U; ++r) {
    static_for<0, U>([&](auto vc) __attribute__((always_inline)) {
      constexpr int v = decltype(vc)::value;
      // activations two k-steps ahead (behind the last one: the last round again, unused)
      const int rn = v + 2 < U ? r : (r + 1 < KS / U ? r + 1 : r);
#pragma unroll
      for (int i = 0; i < NPL; ++i) a[(v + 2) % 3][i] = frag(rn, (v + 2) % U, i);
#pragma unroll
      for (int t = 0; t < TT; ++t) {
        if constexpr (NPL == 3) {
          constexpr int WP[6] = {0, 1, 2, 0, 1, 0}, AP[6] = {2, 1, 0, 1, 0, 0};
#pragma unroll
          for (int m = 0; m < 6; ++m) mma<P>(ring[v % D][t][WP[m]], a[v % 3][AP[m]], acc[t]);
        } else {
          mma<P>(ring[v % D][t][0], a[v % 3][0], acc[t]);
        }
        // (behind the last k-steps this reads what follows in the buffer: unused)
        const int kn = r * U + v + D;
        const int f = team_frag<P, L>(kn < KS ? kn : KS - 1, t0 + t);
#pragma unroll
        for (int i = 0; i < W; ++i) ring[v % D][t][i] = wl[f + i];
      }
      __builtin_amdgcn_sched_barrier(0);
    });
  }
}

// TEAM = 9: workgroup = (third of the squares, cout tile); TEAM = 3: all cout tiles
template <class P, int TEAM>
__global__ __launch_bounds__(256) void team_forward_kernel(const TeamParams prm) {
  using G = Geo<P>;
  using T = TeamGeo<P>;
  constexpr int NPL = T::NPL, W = G::W, THREADS = 256;
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, h = lane >> 5;
  const FwdParams &f = prm.f;
  const unsigned b = blockIdx.x / TEAM;
  const int my_role = (int)(blockIdx.x % TEAM);
  unsigned char *occ = smem + T::OCC_OFF;
  float *lgt = reinterpret_cast<float *>(smem + T::LGT_OFF);
  float *red = reinterpret_cast<float *>(smem + T::RED_OFF);
  int *word = reinterpret_cast<int *>(red) + 40;   // what wave 0 found, for the others
  const unsigned char *packed = f.packed + (size_t)(b / (unsigned)f.boards_per_group) * f.packed_stride;
  const float *tail = reinterpret_cast<const float *>(packed + G::TAIL_OFF);
  unsigned char *act = prm.act + (size_t)b * T::BOARDB;
  unsigned *flags = prm.flags + (size_t)b * kTeamFlags;
  const __amdgpu_buffer_rsrc_t mem = __builtin_amdgcn_make_buffer_rsrc(act, 0, T::BOARDB, 0x00020000);

  [[maybe_unused]] const bool trace_on = true;
  C6_MARK(0);
  // does workgroup `role` have a part in stage l?
  auto has_part = [](int l, int role) {
    if (l == 8) return role == 0;
    return TEAM == 3 || role % 3 < kCoutArr[l] / 32;
  };
  auto flag_set = [&](int l, int role) {
    return __hip_atomic_load(&flags[l * 9 + role], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == prm.tag;
  };
  // Are the inputs of stage l there for `role`?  Bounded; the answer is the same in every thread.
  // 1: yes, 0: no, 2: no need, the stage itself has been done.
  auto wait_inputs = [&](int l, int role) {
    if (wave == 0) {
      const int s = TEAM == 9 ? role / 3 : role;
      int need = -1;   // lane < 9: the role of stage l - 1 it watches
      if (l > 0 && lane < TEAM) {
        const int ls = TEAM == 9 ? lane / 3 : lane;
        if (has_part(l - 1, lane) && (l == 8 || (ls >= s - 1 && ls <= s + 1))) need = lane;
      }
      int got = 0;
      for (int k = 0; k < prm.polls && got == 0; ++k) {
        const bool ok = need < 0 || flag_set(l - 1, need);
        const bool done = lane == 63 && flag_set(l, role);
        if (__builtin_amdgcn_ballot_w64(!ok) == 0) got = 1;
        if (__builtin_amdgcn_ballot_w64(done) != 0) got = 2;
      }
      if (lane == 0) *word = got;
    }
    __syncthreads();
    const int got = *word;
    __syncthreads();
    return got;
  };
  auto raise_flag = [&](int l, int role) {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // this wave's stores have arrived
    __syncthreads();
    if (tid == 0) __hip_atomic_store(&flags[l * 9 + role], prm.tag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  };
  // a layer's outputs: SiLU, planes, 64 * NPL consecutive bytes per square
  auto store_tile = [&](const f32x16 &acc, int layer_off, int t, int pix, bool ok) __attribute__((always_inline)) {
    const int at = layer_off + t * T::BLOCKB + pix * T::PXB;
    int pl[4][NPL][2];   // [quad][plane][pair]
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      float v[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        if constexpr (NPL == 3) v[e] = split_silu(acc[4 * q + e]);
        else v[e] = silu<P>(acc[4 * q + e]);
      }
#pragma unroll
      for (int i = 0; i < NPL; ++i) {
        pl[q][i][0] = i + 1 < NPL ? split_take(v[0], v[1]) : pack2<P>(v[0], v[1]);
        pl[q][i][1] = i + 1 < NPL ? split_take(v[2], v[3]) : pack2<P>(v[2], v[3]);
      }
    }
    // lane halves hold alternating groups of four channels: swap so that each lane has eight in a row
#pragma unroll
    for (int qq = 0; qq < 2; ++qq)
#pragma unroll
      for (int i = 0; i < NPL; ++i) {
        v4i o;
#pragma unroll
        for (int d = 0; d < 2; ++d) {
          // lower lane: quad 2 qq of both halves, upper lane: quad 2 qq + 1 of both
          const auto x = __builtin_amdgcn_permlane32_swap((unsigned)pl[2 * qq][i][d], (unsigned)pl[2 * qq + 1][i][d], false, false);
          const unsigned x0 = x[0], x1 = x[1];
          o[d] = (int)x0;
          o[2 + d] = (int)x1;
        }
        if (ok) __builtin_amdgcn_raw_buffer_store_b128(o, mem, at + i * 64 + (2 * qq + h) * 16, 0, kSc1);
      }
  };

  // what the LDS region holds: the rows of third region_s, padding zero
  int region_s = -1;

  auto conv_stage = [&](auto lc, int role) __attribute__((always_inline)) -> bool {
    constexpr int L = decltype(lc)::value;
    constexpr int NT = kCoutArr[L] / 32, NTP = kCinArr[L] / 32, TT = TEAM == 9 ? 1 : NT;
    constexpr int D = (W == 3 ? 6 : 18) / TT;
    const int s = TEAM == 9 ? role / 3 : role, t0 = TEAM == 9 ? role % 3 : 0;
    const WFrags wl = layer_weights<P, L>(packed, lane);
    C6_MARK(6 * L);
    const int got = wait_inputs(L, role);
    if (got != 1) return got == 2;
    C6_MARK(6 * L + 1);
    // ---- rows r0 - 1 .. r1 + 1 into LDS ----
    const int p0 = 128 * s, p1 = p0 + 127 < kPix - 1 ? p0 + 127 : kPix - 1;
    const int r0 = p0 / kBoard, r1 = p1 / kBoard;
    const int base = r0 * kPitch;                       // first position: the row above r0
    if (region_s != s) {
      const v4i z = {0, 0, 0, 0};
      for (int i = tid; i < T::REGION / 16; i += THREADS) reinterpret_cast<v4i *>(smem)[i] = z;
      __syncthreads();
      region_s = s;
    }
    const int ra = r0 > 0 ? r0 - 1 : 0, rb = r1 < kBoard - 1 ? r1 + 1 : kBoard - 1;
    const int first = ra * kBoard, count = (rb - ra + 1) * kBoard;   // squares
    constexpr int UP = 4 * NPL;                                      // 16-byte units per square and tile
    constexpr int ROUNDS = (10 * kBoard * UP + THREADS - 1) / THREADS;
    v4i in[NTP][ROUNDS];
#pragma unroll
    for (int t = 0; t < NTP; ++t)
#pragma unroll
      for (int k = 0; k < ROUNDS; ++k) {
        const int u = tid + k * THREADS;
        if (u < count * UP)
          in[t][k] = __builtin_amdgcn_raw_buffer_load_b128(mem, T::act_off(L - 1) + t * T::BLOCKB + first * T::PXB + u * 16, 0, kSc1);
      }
    // the first weights, behind the activations in the queue: back by the time those are in LDS
    v4i ring[D][TT][W];
    f32x16 acc[TT];
#pragma unroll
    for (int d = 0; d < D; ++d)
#pragma unroll
      for (int t = 0; t < TT; ++t)
#pragma unroll
        for (int i = 0; i < W; ++i) ring[d][t][i] = wl[team_frag<P, L>(d, t0 + t) + i];
    load_bias_tiles(acc, tail + bias_offset(L) + 32 * t0, h);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int t = 0; t < NTP; ++t)
#pragma unroll
      for (int k = 0; k < ROUNDS; ++k) {
        const int u = tid + k * THREADS;
        if (u < count * UP) {
          const int px = first + u / UP, rest = u % UP, r = px / kBoard;
          const int pos = (r + 1) * kPitch + (px - r * kBoard + 1) - base;
          *reinterpret_cast<v4i *>(smem + pos * T::RECB + (rest / 4) * 192 + t * 64 + (rest % 4) * 16) = in[t][k];
        }
      }
    __syncthreads();
    C6_MARK(6 * L + 2);
    // ---- contraction ----
    const int p = (4 * s + wave) * 32 + (lane & 31);
    const bool ok = p < kPix;
    const int pc = ok ? p : kPix - 1, r = pc / kBoard;
    const int rec = (r * kPitch + (pc - r * kBoard) - base) * T::RECB + 16 * h;
    team_conv<P, L, TT>(smem, wl, ring, rec, t0, acc);
    C6_MARK(6 * L + 3);
    if constexpr (L < 7) {
#pragma unroll
      for (int t = 0; t < TT; ++t) store_tile(acc[t], T::act_off(L), t0 + t, pc, ok);
    } else {
      // heads: this wave's share of the policy (per square and cout tile) and of the value
      const float *pw = tail + kBiasTotal + 32 * t0 + 4 * h;
#pragma unroll
      for (int t = 0; t < TT; ++t) {
        float pol = 0.0f, val = 0.0f;
#pragma unroll
        for (int q = 0; q < 4; ++q)
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const float a = split_silu(acc[t][4 * q + e]);
            pol = fmaf(a, pw[32 * t + 8 * q + e], pol);
            val = fmaf(a, pw[kHeadC + 32 * t + 8 * q + e], val);
          }
        const unsigned bits = __builtin_bit_cast(unsigned, pol);
        const auto x = __builtin_amdgcn_permlane32_swap(bits, bits, false, false);
        const unsigned x0 = x[0], x1 = x[1];
        const float tot = __builtin_bit_cast(float, x0) + __builtin_bit_cast(float, x1);
        const float vs = wave_sum(ok ? val : 0.0f);
        if (h == 0 && ok)
          __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(int, tot), mem, T::HEAD_OFF + ((t0 + t) * 384 + pc) * 4, 0, kSc1);
        if (lane == 0)
          __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(int, vs), mem, T::VAL_OFF + ((t0 + t) * 12 + 4 * s + wave) * 4, 0, kSc1);
      }
    }
    raise_flag(L, role);
    C6_MARK(6 * L + 4);
    return true;
  };

  // first layer: every workgroup stages the whole board
  auto first_stage = [&](int role) __attribute__((always_inline)) -> bool {
    const int s = TEAM == 9 ? role / 3 : role;
    int *flag = reinterpret_cast<int *>(red) + 32;   // [0]: third plane varies, [1]: an input is not exact in bf16
    const int p = (4 * s + wave) * 32 + (lane & 31);
    const bool ok = p < kPix;
    const int pc = ok ? p : kPix - 1, r = pc / kBoard, c = pc - r * kBoard;
    region_s = -1;
    f32x16 a0;
    {
      // (the table holds the squares as the one-workgroup kernels' lanes do: wave, pixel tile)
      const WFrags tb = packed_frags<P>(packed, lane, G::PLANE2_FRAG_OFF + __builtin_amdgcn_readfirstlane(4 * s + wave) * 4);
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const f32x4 t4 = __builtin_bit_cast(f32x4, tb[q]);
#pragma unroll
        for (int e = 0; e < 4; ++e) a0[4 * q + e] = t4[e];
      }
    }
    float xin[2][3];
    const bool state = f.x_dtype == C6_DT_BOARD_I8;
    long long src = state && f.index ? f.index[b] : (long long)b;
    if (state) src = src < 0 ? 0 : (src >= f.num_states ? f.num_states - 1 : src);
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      const int sq = tid + k * THREADS;
      if (sq < kPix) {
        if (state) {
          const int stone = reinterpret_cast<const int8_t *>(f.x)[(size_t)src * kPix + (f.view ? d4_from_view(sq, f.view) : sq)];
          const int me = f.player[src];
          xin[k][0] = stone == me ? 1.0f : 0.0f;
          xin[k][1] = stone == -me ? 1.0f : 0.0f;
          xin[k][2] = f.stones_left[src] == 1 ? 1.0f : 0.0f;
        } else {
#pragma unroll
          for (int ch = 0; ch < 3; ++ch) xin[k][ch] = load_x(f.x, f.x_dtype, ((size_t)b * 3 + ch) * kPix + sq);
        }
      }
    }
    if (tid < 2) flag[tid] = 0;
    if (tid == 0) red[34] = xin[0][2];
    {
      const v4i z = {0, 0, 0, 0};
      for (int i = tid * 16; i < G::COPIES_BYTES; i += THREADS * 16) *reinterpret_cast<v4i *>(smem + i) = z;
    }
    __syncthreads();
    const float c2 = red[34];
    bool varies = false;
#pragma unroll
    for (int k = 0; k < 2; ++k)
      if (tid + k * THREADS < kPix) varies |= __builtin_bit_cast(int, xin[k][2]) != __builtin_bit_cast(int, c2);
    if (varies) flag[0] = 1;
    __syncthreads();
    const bool plane2_varies = flag[0] != 0;
    bool inexact = false;
#pragma unroll
    for (int k = 0; k < 2; ++k)
      if (tid + k * THREADS < kPix)
#pragma unroll
        for (int ch = 0; ch < 3; ++ch)
          inexact |= (ch < 2 || plane2_varies) && (__builtin_bit_cast(int, xin[k][ch]) & 0xffff) != 0;
    if (NPL == 3 && inexact) flag[1] = 1;
    __syncthreads();
    const int parts = NPL == 3 && flag[1] != 0 ? 3 : 1;
    const int sh = c % G::E;
    const int l1 = sh * G::COPY_BYTES + (r * 3 * kL1RowPitch + (c - sh)) * G::EB;
    const int steps = plane2_varies ? G::STEPS1 : G::FAST1_STEPS;
    const int row0 = plane2_varies ? l1 + kL1RowsHalf * h * kL1RowPitch * G::EB : l1 + h * kL1RowPitch * G::EB;
    const int rowb = (plane2_varies ? 1 : 3) * kL1RowPitch * G::EB;
    const WFrags wl = plane2_varies ? layer_weights<P, 0>(packed, lane) : packed_frags<P>(packed, lane, G::FAST1_OFF);
    {
      f32x16 b0[1];
      load_bias_tiles(b0, tail + bias_offset(0), h);
#pragma unroll
      for (int i = 0; i < 16; ++i) a0[i] = plane2_varies ? b0[0][i] : fmaf(c2, a0[i], b0[0][i]);
    }
#pragma unroll 1
    for (int part = 0; part < parts; ++part) {
      if (part > 0) __syncthreads();
#pragma unroll
      for (int k = 0; k < 2; ++k) {
        const int sq = tid + k * THREADS;
        if (sq < kPix) {
          const int row = sq / kBoard, col = sq - row * kBoard;
#pragma unroll
          for (int ch = 0; ch < 3; ++ch) {
            if (ch >= (plane2_varies ? 3 : 2)) break;
            const unsigned short v16 = bits16<P>(xin[k][ch]);
            if constexpr (NPL == 3) xin[k][ch] -= __builtin_bit_cast(float, (unsigned)v16 << 16);
            const int hrow = (row + kK1 / 2) * 3 + ch;
#pragma unroll
            for (int q = 0; q < G::E; ++q)
              *reinterpret_cast<unsigned short *>(smem + q * G::COPY_BYTES + (hrow * kL1RowPitch + (col + kK1 / 2 - q)) * G::EB) = v16;
          }
        }
      }
      __syncthreads();
      C6_MARK(1);
      // k-steps in rounds of one kernel row (three fragments); weights two rounds ahead
      v4i w[3][3][W], a[3][3];
      const int rows = steps / 3;
      auto fetch = [&](int row, int slot) __attribute__((always_inline)) {
        const int rr = row < rows ? row : rows - 1;
#pragma unroll
        for (int i = 0; i < 3; ++i) {
#pragma unroll
          for (int j = 0; j < W; ++j) w[slot][i][j] = wl[(rr * 3 + i) * W + j];
          a[slot][i] = *reinterpret_cast<const v4i *>(smem + row0 + rr * rowb + i * 16);
        }
        __builtin_amdgcn_sched_barrier(0);
      };
      auto multiply = [&](int slot) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < 3; ++i)
#pragma unroll
          for (int j = 0; j < W; ++j) mma<P>(w[slot][i][j], a[slot][i], a0);
        __builtin_amdgcn_sched_barrier(0);
      };
      fetch(0, 0);
      fetch(1, 1);
      int row = 0;
#pragma unroll 1
      for (; row + 3 <= rows; row += 3) {
        fetch(row + 2, 2);
        multiply(0);
        fetch(row + 3, 0);
        multiply(1);
        fetch(row + 4, 1);
        multiply(2);
      }
      if (row < rows) multiply(0);
      if (row + 1 < rows) multiply(1);
    }
    C6_MARK(2);
    store_tile(a0, T::act_off(0), 0, pc, ok);
    raise_flag(0, role);
    C6_MARK(3);
    return true;
  };

  // the heads' partial sums into logits, value and draw (one workgroup of the team)
  auto last_stage = [&](int role) __attribute__((always_inline)) -> bool {
    const int got = wait_inputs(8, role);
    if (got != 1) return got == 2;
    const float *valw = tail + kBiasTotal + kHeadC;
    const float polb = valw[kHeadC], valb = valw[kHeadC + 1];
    auto partial = [&](int at) __attribute__((always_inline)) {
      return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(mem, at, 0, kSc1));
    };
    const bool state = f.x_dtype == C6_DT_BOARD_I8;
    long long src = state && f.index ? f.index[b] : (long long)b;
    if (state) src = src < 0 ? 0 : (src >= f.num_states ? f.num_states - 1 : src);
    for (int p = tid; p < kPix; p += THREADS) {
      const float z = ((partial(T::HEAD_OFF + p * 4) + partial(T::HEAD_OFF + (384 + p) * 4)) +
                       partial(T::HEAD_OFF + (768 + p) * 4)) + polb;
      bool o = false;
      if (f.mask_mode == C6_MASK_LEGAL) {
        o = f.legal[(size_t)b * kPix + p] == 0;
      } else if (f.mask_mode == C6_MASK_INPUT) {
        if (state) {
          const int stone = reinterpret_cast<const int8_t *>(f.x)[(size_t)src * kPix + (f.view ? d4_from_view(p, f.view) : p)];
          const int me = f.player[src];
          o = stone == me || stone == -me;
        } else {
          o = load_x(f.x, f.x_dtype, (size_t)b * 3 * kPix + p) != 0.0f || load_x(f.x, f.x_dtype, ((size_t)b * 3 + 1) * kPix + p) != 0.0f;
        }
      }
      lgt[p] = z;
      occ[p] = o;
      if (f.logits != nullptr) static_cast<float *>(f.logits)[(size_t)b * kPix + p] = o ? f.fill : z;
    }
    if (tid < 36) red[tid] = partial(T::VAL_OFF + tid * 4);
    __syncthreads();
    if (tid == 0 && f.value != nullptr) f.value[b] = tanhf(split_value_sum(red) * (1.0f / kPix) + valb);
    if (f.actions != nullptr && wave == 0) {
      int a;
      float lp;
      wave_sample(
          lane, f.u[b], f.inv_temperature, [&](int i) { return lgt[i]; }, [&](int i) { return occ[i] == 0; }, a, lp);
      if (lane == 0) {
        f.actions[b] = a;
        if (f.logprob != nullptr) f.logprob[b] = lp;
      }
    }
    raise_flag(8, role);
    C6_MARK(49);
    return true;
  };

  // Stages in order; `help`: a wait ran out, do the earliest piece that has no flag instead.
  bool help = false;
  for (int l = 0; l < kTeamStages;) {
    if (!help && !has_part(l, my_role)) {
      ++l;
      continue;
    }
    int stage = l, role = my_role;
    if (help) {
      if (wave == 0) {
        int found = l * 16 + my_role;
        for (int k = l - 1; k >= 0; --k) {
          const bool open = lane < TEAM && has_part(k, lane) && !flag_set(k, lane);
          const unsigned long long m = __builtin_amdgcn_ballot_w64(open);
          if (m != 0) found = k * 16 + __builtin_ctzll(m);
        }
        if (lane == 0) *word = found;
      }
      __syncthreads();
      stage = *word >> 4;
      role = *word & 15;
      __syncthreads();
    }
    bool ok = false;
    switch (stage) {
      case 0: ok = first_stage(role); break;
      case 1: ok = conv_stage(IC<1>{}, role); break;
      case 2: ok = conv_stage(IC<2>{}, role); break;
      case 3: ok = conv_stage(IC<3>{}, role); break;
      case 4: ok = conv_stage(IC<4>{}, role); break;
      case 5: ok = conv_stage(IC<5>{}, role); break;
      case 6: ok = conv_stage(IC<6>{}, role); break;
      case 7: ok = conv_stage(IC<7>{}, role); break;
      default: ok = last_stage(role); break;
    }
    if (ok && stage == l && role == my_role) ++l;
    help = !ok;
  }
}

// How many workgroups share a board when there are `boards` of them: nine while that many fit the
// chip at once, then three, then one (the one-workgroup kernels).
inline int team_size(long long boards, int cus) { return boards * 9 <= cus ? 9 : (boards * 3 <= cus ? 3 : 1); }

// modes that have a team kernel
template <class P> constexpr bool has_team() { return P::ID == C6_PREC_F32S; }

}  // namespace c6
