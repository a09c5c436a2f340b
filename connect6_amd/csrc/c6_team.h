// Few boards: a TEAM of workgroups per board (included by c6_forward.hip).
//
// One workgroup per board leaves most of the chip idle when there are fewer boards than CUs, and one
// board takes as long as 256.  Here 12, 6, 3 or 2 workgroups share a board: each takes one, two, four or six
// of the twelve tiles of 32 squares through all layers, its waves dividing tiles and output channels
// between them.  A workgroup's own activations stay in its LDS; what a 3x3 layer reads beyond them,
// twenty squares on either side, goes through memory: the owner stores its squares, waits until the
// stores are acknowledged and raises a flag for the layer.  Each accumulator sees the same MFMAs in
// the same order as in the one-workgroup kernels, and the heads' sums are put together in their
// order, so the results are the same bit for bit.
//
// What it takes (cycles of a 2.4 GHz clock; twelve workgroups, one board): staging the input 7 k, the first layer
// 3 k (fp32 11 k), then per layer 1.2 k (fp32 1.8 k) until the neighbours' flags are seen, 0.5 k (fp32 1 k) until their squares are in LDS,
// the MFMAs (bf16 0.5-2.1 k, fp32 2.8-6.9 k: three per product) and 1.3 k (fp32 2.6-2.9 k: two parts and the range) until the outputs are
// stored and acknowledged, at the end 6 k (fp32 11 k) for the heads' sums: 66 k in bf16, 110 k in fp32 (c6_half_team.h).
//
// The exchange: loads of activations and flags carry the device-scope cache policy (sc1).  So do stores until a
// workgroup has seen that all of its team run on its own XCD (each leaves its XCD's number beside the flags): from
// then on they stay in that XCD's L2, where the loads find them.  Measured between neighbours of a team on one XCD,
// store, wait for the acknowledgement, flag, load: 4 KB a side 2.2 us with the stores going through to memory, 1.1 us
// with stores that stay in L2; 12 KB 3.9 and 1.9 us; 0.3 KB 1.5 and 0.7 us.  (Each word with its tag beside it, no
// flag and no wait, 1.0, 2.0 and 0.5 us: not worth twice the words and memory of its own.)  One board's forward 35.8 ->
// 30.1 us in bf16, with what else changed there: weights asked for in front
// of the wait, addresses of exchanged squares formed once, biases and head weights from LDS.
//
// Nothing waits for a workgroup that may not be running: a wait is bounded, and a workgroup whose
// wait runs out does the missing piece of work itself (the earliest one that has no flag; everything
// in front of it has one).  For that a workgroup also stores the squares that no neighbour reads, behind
// its flag and with a second one.  Outputs of every layer have a place of their own, and whoever computes
// a piece writes the same bytes, so doing one twice is harmless; any single workgroup can finish the
// board alone.  The flags of a launch are its tag: the caller hands a tag that the flag words have
// not held before (or words that are zero).
#pragma once

namespace c6 {

constexpr int kTeamStages = 9;   // eight layers, then the heads' write-out
constexpr int kTeamAll = 128;    // flag words: see team_board
constexpr int kSc1 = 16;         // cache policy: device scope
constexpr int kTeamXcd = kTeamAll + kTeamStages * 12;
constexpr int kTeamListed = kTeamXcd + 12, kTeamDone = kTeamListed + 1;   // see team_cascade_kernel
static_assert(kTeamDone < kTeamFlags && kTeamStages * 12 <= kTeamAll, "flag words");

// modes that have a team kernel
template <class P> constexpr bool has_team() { return P::ID != C6_PREC_F32; }

template <class P> struct TeamGeo {
  using G = Geo<P>;
  static constexpr bool SPLIT = kParts<P> != 0;               // fp32 (two parts: c6_half_team.h)
  static constexpr int NPL = SPLIT ? kParts<P> : 1;           // planes of an activation
  static constexpr int LO_OFF = NPL * 192;                    // fp6 blocks of a record (LO6)
  static constexpr int RECB = NPL * 192 + (P::LO6 ? 96 : 0) + 16;   // an odd number of 16-byte units
  // a square of c channels in memory: 16-byte units of its planes, then of its fp6 blocks
  static constexpr int units(int c) { return NPL * c / 8 + (P::LO6 ? c / 16 : 0); }
  static constexpr int act_off(int l) {
    int s = 0;
    for (int i = 0; i < l; ++i) s += kPix * units(kCoutArr[i]) * 16;
    return s;
  }
  static constexpr int HEAD_OFF = act_off(7);                 // policy sums: SPLIT [3][384], else [384]
  // value sums: SPLIT one per (cout tile, tile of squares), else nine per lane of each tile of squares
  static constexpr int VAL_OFF = HEAD_OFF + 3 * 384 * 4;
  static constexpr int NOTE_OFF = VAL_OFF + 12 * 9 * 64 * 4;   // two parts: a word per (layer, member, wave), half_note
  static constexpr int BOARDB = (NOTE_OFF + (kParts<P> == 2 ? 8 * 12 * 4 * 4 : 0) + 255) & ~255;
  // LDS: up to 11 rows of positions (128 squares lie in at most 8 board rows), 13 for 192 squares (SPLIT; in 11)
  static constexpr int REGION = ((SPLIT ? 13 : 11) * kPitch + 1) * RECB;
  // The first layer's shifted copies hold the halo rows that a workgroup's squares see: three per kernel row of up to
  // twelve rows of squares, and the zero row (an odd number: a copy is then an odd number of 16-byte units long).
  static constexpr int COPY_ROWS = 105, COPY_BYTES = COPY_ROWS * kL1RowPitch * G::EB, COPIES_BYTES = G::E * COPY_BYTES;
  static constexpr int BUF = REGION > COPIES_BYTES ? REGION : COPIES_BYTES;
  static constexpr int OCC_OFF = (BUF + 15) & ~15;
  static constexpr int LGT_OFF = OCC_OFF + 384;
  static constexpr int RED_OFF = LGT_OFF + 1456;
  // a copy of the packed set's biases and head weights: no layer starts behind the latency of their loads
  static constexpr int TAIL_OFF = (RED_OFF + 256 * 4 + 15) & ~15;
  static constexpr int LDS_BYTES = TAIL_OFF + G::TAIL_FLOATS * 4;
  static_assert(RECB / 16 % 2 == 1 && LDS_BYTES <= 160 * 1024, "LDS map");
};

// How a team divides the twelve tiles of squares and a layer's cout tiles: TEAM workgroups with PXT
// tiles of squares each, whose four waves take PT of them and form CG groups of cout tiles.  A wave takes two
// tiles of squares where there are two: with six workgroups each weight is then read by one wave, with three
// by two; with one tile of squares per wave it would be twice as many, 96 and 128 bytes a cycle where the L1
// gives 64 (six workgroups, 22 to 42 boards, bf16 + fp6 62.6 -> 55 us).  (fp32 contracts a weight with three parts, so
// that a tile of squares per wave asks for just those 64, and all four waves have work in layers of two cout tiles.  Counted
// over 53 boards, three workgroups each: of the 263 k cycles of a workgroup 150 k are reads from the L1, 64 bytes each, 128 k
// MFMAs, so the L1 bounds the contractions by a sixth.)
// Three or six tiles of squares go to three waves, all cout tiles in each; the fourth watches the flags.
template <class P, int TEAM> struct TeamShape {
  static constexpr int PXT = 12 / TEAM;
  static constexpr int PT = PXT == 6 ? 2 : (PXT % 2 == 0 && !TeamGeo<P>::SPLIT ? 2 : 1), PG = PXT / PT;
  static constexpr int CG = PG == 3 ? 1 : (PG == 1 ? (PXT == 1 ? 3 : 4) : 4 / PG);   // groups of squares' tiles, of cout tiles
  static constexpr int tiles(int nt) { return (nt + CG - 1) / CG; }   // cout tiles of a wave
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

// k-steps of weights that a wave keeps in flight: the loads take some 800 cycles and a k-step is
// 32 cycles per MFMA
template <class P, int TT, int PT> constexpr int team_ring() {
  return Geo<P>::W == 3 ? (PT > 1 ? 3 : 6) / TT : (Geo<P>::W == 1 ? 18 / TT : (TT == 1 ? 9 : (TT == 2 ? 6 : 3)));
}

// Low-order (fp6) pass of layer L for PT tiles of squares, conv3_lo_pass with TT cout tiles from t0 on.
//   rec: LDS addresses of the lane's squares' records
template <class P, int L, int TT, int PT>
__device__ __forceinline__ void team_lo_pass(const unsigned char *smem, const unsigned char *packed, int lane,
                                             const int (&rec)[PT], int t0, f32x16 (&acc)[PT][TT]) {
  using G = Geo<P>;
  using T = TeamGeo<P>;
  typedef int v8i __attribute__((ext_vector_type(8)));
  constexpr int NT = kCoutArr[L] / 32, PER32 = kCinArr[L] / 32, HC = G::lo_half_chunks(L), NC = G::lo_chunks(L);
  const WFrags wl = packed_frags<P>(packed, lane, G::lo_frag_offset(L));
  const int scale_w = 127 - __builtin_amdgcn_readfirstlane(reinterpret_cast<const int *>(smem + T::TAIL_OFF)[G::TAIL_SW + L]);
  constexpr int D = 4;
  v4i w0[D][TT], w1[D][TT];
  auto load = [&](int c, int d) __attribute__((always_inline)) {
    const int cc = c < NC ? c : NC - 1;
#pragma unroll
    for (int t = 0; t < TT; ++t) {
      const int tile = t0 + t < NT ? t0 + t : NT - 1;
      lo_load_pieces<P>(wl + (cc * NT + tile) * 2, w0[d][t], w1[d][t]);
    }
  };
#pragma unroll
  for (int d = 0; d < D; ++d) load(d, d);
  static_for<0, NC>([&](auto cc) __attribute__((always_inline)) {
    constexpr int c = decltype(cc)::value;
    constexpr int g0 = 2 * c, g1 = 2 * c + 1 < HC ? 2 * c + 1 : HC - 1;
    constexpr int o0 = ((g0 / PER32 / 3 - 1) * kPitch + g0 / PER32 % 3 - 1) * T::RECB + (g0 % PER32) * 32;
    constexpr int o1 = ((g1 / PER32 / 3 - 1) * kPitch + g1 / PER32 % 3 - 1) * T::RECB + (g1 % PER32) * 32;
#pragma unroll
    for (int i = 0; i < PT; ++i) {
      const unsigned char *at = smem + rec[i] + T::LO_OFF + (lane < 32 ? o0 : o1);
      const v4i b0 = *reinterpret_cast<const v4i *>(at);
      const v4i b1 = *reinterpret_cast<const v4i *>(at + 16);
      const v8i b = {b0[0], b0[1], b0[2], b0[3], b1[0], b1[1], b1[2], b1[2]};
#pragma unroll
      for (int t = 0; t < TT; ++t) {
        const v8i a = __builtin_shufflevector(w0[c % D][t], w1[c % D][t], 0, 1, 2, 3, 4, 5, 6, 7);
        acc[i][t] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(a, b, acc[i][t], 2, 2, 0, scale_w, 0, b[6]);
      }
    }
    load(c + D, c % D);
    __builtin_amdgcn_sched_barrier(0);
  });
}

// The contraction of 3x3 layer L for PT tiles of 32 squares and TT cout tiles from t0 on (tiles beyond
// the layer's last repeat it; their results are not used).
//   rec: LDS addresses of the lane's squares' records;  acc: the bias on entry
//   low (fp32): what the bias leaves out, for the small products' sum (split_conv)
template <class P, int L, int TT, int PT>
__device__ __forceinline__ void team_conv(const unsigned char *smem, const unsigned char *packed, const WFrags &wl,
                                          v4i (&ring)[team_ring<P, TT, PT>()][TT][Geo<P>::W], int lane,
                                          const int (&rec)[PT], int t0, f32x16 (&acc)[PT][TT],
                                          f32x16 (&low)[PT][TT]) {
  using T = TeamGeo<P>;
  constexpr int NT = kCoutArr[L] / 32, NTP = kCinArr[L] / 32;
  constexpr int W = Geo<P>::W, NPL = T::NPL, D = team_ring<P, TT, PT>();
  constexpr int KC = kCinArr[L] / 16, KS = 9 * KC;
  constexpr int U = P::PIPE ? kPhaseSteps : 3 * KC;     // k-steps of one unrolled round
  constexpr bool LO = P::LO6 && ((P::LO_MASK >> L) & 1);
  static_assert(KS % U == 0 && U % D == 0, "ring");
  int corner[PT];
#pragma unroll
  for (int p = 0; p < PT; ++p) corner[p] = rec[p] - (kPitch + 1) * T::RECB + 16 * (lane >> 5);
  // k-step v of round r: (tap, 16 channels).  Pipelined modes: a round is a phase, all taps of 32
  // channels; fp32: a round is a kernel row.
  auto frag = [&](int r, int v, int p, int pl) __attribute__((always_inline)) {
    const int tap = v / 2;
    const int off = P::PIPE ? ((tap / 3) * kPitch + tap % 3) * T::RECB + (v % 2) * 32 : (v / KC) * T::RECB + (v % KC) * 32;
    const int base = P::PIPE ? r * 64 : r * kPitch * T::RECB;
    return *reinterpret_cast<const v4i *>(smem + corner[p] + base + off + pl * 192);
  };
  v4i a[3][PT][NPL];
#pragma unroll
  for (int v = 0; v < 2; ++v)
#pragma unroll
    for (int p = 0; p < PT; ++p)
#pragma unroll
      for (int i = 0; i < NPL; ++i) a[v][p][i] = frag(0, v, p, i);
  auto round = [&](int r) __attribute__((always_inline)) {
    // (the low-order pass comes in front of the last phase, as in pipe_layer)
    if constexpr (LO) {
      if (r == NTP - 1) team_lo_pass<P, L, TT, PT>(smem, packed, lane, rec, t0, acc);
    }
    static_for<0, U>([&](auto vc) __attribute__((always_inline)) {
      constexpr int v = decltype(vc)::value;
      // activations two k-steps ahead (behind the last one: the last round again, unused)
      const int rn = v + 2 < U ? r : (r + 1 < KS / U ? r + 1 : r);
#pragma unroll
      for (int p = 0; p < PT; ++p)
#pragma unroll
        for (int i = 0; i < NPL; ++i) a[(v + 2) % 3][p][i] = frag(rn, (v + 2) % U, p, i);
      auto refill = [&](int t) __attribute__((always_inline)) {
        const int kn = r * U + v + D;   // (behind the last k-steps: the last one again, unused)
        const int f = team_frag<P, L>(kn < KS ? kn : KS - 1, t0 + t < NT ? t0 + t : NT - 1);
#pragma unroll
        for (int i = 0; i < W; ++i) ring[v % D][t][i] = wl[f + i];
      };
      if constexpr (NPL == 3) {
        // (An accumulator's next MFMA is eight cycles late if it follows at once, so two tiles take turns: forty boards
        // 102 -> 97 us.  With three the L1's 64 bytes a cycle bound the layer, and loads in a row per tile suit it better:
        // 56 boards 120 us, in turns 123.)
        constexpr int WP[6] = {0, 1, 2, 0, 1, 0}, AP[6] = {2, 1, 0, 1, 0, 0};
        constexpr bool TURNS = TT == 2;
#pragma unroll
        for (int o = 0; o < (TURNS ? 6 : TT); ++o)
#pragma unroll
          for (int n = 0; n < (TURNS ? TT : 6); ++n) {
            const int m = TURNS ? o : n, t = TURNS ? n : o;
#pragma unroll
            for (int p = 0; p < PT; ++p) mma<P>(ring[v % D][t][WP[m]], a[v % 3][p][AP[m]], m < 5 ? low[p][t] : acc[p][t]);
            if (m == 5) refill(t);
          }
      } else {
#pragma unroll
        for (int t = 0; t < TT; ++t) {
#pragma unroll
          for (int i = 0; i < W; ++i)
#pragma unroll
            for (int p = 0; p < PT; ++p) mma<P>(ring[v % D][t][i], a[v % 3][p][0], acc[p][t]);
          refill(t);
        }
      }
      __builtin_amdgcn_sched_barrier(0);
    });
  };
  if constexpr (P::PIPE) {
    // (a k-step is one or two MFMAs: the waits of a loop's back edge would show)
    static_for<0, KS / U>([&](auto rc) __attribute__((always_inline)) { round(decltype(rc)::value); });
  } else {
#pragma unroll 1
    for (int r = 0; r < KS / U; ++r) round(r);
  }
  if constexpr (NPL == 3) {
#pragma unroll
    for (int p = 0; p < PT; ++p)
#pragma unroll
      for (int t = 0; t < TT; ++t)
#pragma unroll
        for (int e = 0; e < 16; ++e) acc[p][t][e] = two_sums(acc[p][t][e], low[p][t][e]);
  }
}

// SiLU of one accumulator tile, step by step: a lone wave waits for each result that its next instruction needs.  Against
// output by output it is worth a per cent, one way or the other: 22 to 40 boards in bf16 and fp16 40.0 -> 39.6 us, 40 boards that
// a cascade lists 117.2 -> 116.2, 86 to 128 fp32 boards 217.2 -> 215.5; but 1 to 16 boards in bf16 30.2 -> 30.6; one and 53 fp32
// boards, and the teams beside whole rounds, the same.
template <class P> __device__ __forceinline__ void silu_tile(const f32x16 &acc, float (&v)[16]) {
  if constexpr (TeamGeo<P>::SPLIT) {
    float half[8];
#pragma unroll
    for (int e0 = 0; e0 < 16; e0 += 8) {
      split_silu8(acc, e0, half);
#pragma unroll
      for (int e = 0; e < 8; ++e) v[e0 + e] = half[e];
    }
  } else {
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int e = 0; e < 16; ++e) v[e] = __builtin_amdgcn_exp2f(acc[e]);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int e = 0; e < 16; ++e) v[e] = 1.0f + v[e];
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int e = 0; e < 16; ++e) v[e] = __builtin_amdgcn_rcpf(v[e]);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int e = 0; e < 16; ++e) v[e] = acc[e] * v[e];
    __builtin_amdgcn_sched_barrier(0);
  }
}

// SiLU of one accumulator tile into the record at `rec` (cout tile t): planes, and the fp6 block.
// UNDER: the one-workgroup kernel takes this tile's low-order parts behind MFMAs (see epi_atom).
template <class P, bool LO, bool UNDER>
__device__ __forceinline__ void team_store(unsigned char *smem, int rec, int h, int t, const f32x16 &acc) {
  using T = TeamGeo<P>;
  unsigned char *at = smem + rec + 64 * t + 8 * h;
  if constexpr (T::SPLIT) {
#pragma unroll
    for (int q = 0; q < 4; q += 2) {
      float v[8];
      int w[3][4];
      split_silu8(acc, 4 * q, v);
      split_planes8(v, w);
#pragma unroll
      for (int i = 0; i < 3; ++i)
#pragma unroll
        for (int e = 0; e < 2; ++e) *reinterpret_cast<v2i *>(at + i * 192 + 16 * (q + e)) = v2i{w[i][2 * e], w[i][2 * e + 1]};
    }
  } else {
    const DropConsts k = drop_consts<P>();
    float v[16], lo[16], m = 0.0f;
    silu_tile<P>(acc, v);
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      int hi[2];
#pragma unroll
      for (int p = 0; p < 2; ++p) {
        const int i = 4 * q + 2 * p;
        const float v0 = v[i], v1 = v[i + 1];
        hi[p] = pack2<P>(v0, v1);
        if constexpr (LO) {
          if constexpr (UNDER) {
            lo[i] = v0 - __builtin_bit_cast(float, hi[p] << 16);
            lo[i + 1] = v1 - __builtin_bit_cast(float, hi[p] & (int)0xffff0000);
          } else {
            lo[i] = dropped_lo(v0, hi[p], k);
            lo[i + 1] = dropped_hi(v1, hi[p], k);
          }
          m = __builtin_amdgcn_fmed3f(__builtin_fabsf(lo[i]), m, __builtin_inff());
          m = __builtin_amdgcn_fmed3f(__builtin_fabsf(lo[i + 1]), m, __builtin_inff());
        }
      }
      *reinterpret_cast<v2i *>(at + 16 * q) = v2i{hi[0], hi[1]};
    }
    if constexpr (LO) {
      const unsigned mb = __builtin_bit_cast(unsigned, m);
      const auto x = __builtin_amdgcn_permlane32_swap(mb, mb, false, false);
      const unsigned x0 = x[0], x1 = x[1];
      int sc = (int)((x0 > x1 ? x0 : x1) >> 23) - 2;
      sc = sc < 1 ? 1 : sc;
      f32x16v even, odd;
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        even[i] = lo[i];
        odd[i] = lo[8 + i];
        even[8 + i] = odd[8 + i] = 0.0f;   // (only slots 0-15 are kept)
      }
      const u32x6 r = to_fp6_block(even, odd, __builtin_bit_cast(float, sc << 23));
      int *d32 = reinterpret_cast<int *>(smem + rec + T::LO_OFF + 32 * t + 12 * h);
      d32[0] = (int)r[0];
      d32[1] = (int)r[1];
      d32[2] = (int)r[2];
      *reinterpret_cast<int *>(smem + rec + T::LO_OFF + 32 * t + 24 + 4 * h) = sc;
    }
  }
}

// Board `b` by the team that this workgroup (its member my_role) belongs to; `slot`: the team's share of
// the exchange memory and of the flags.
template <class P, int TEAM>
__device__ __forceinline__ void team_board(const TeamParams &prm, unsigned char *smem, unsigned b, unsigned slot,
                                           int my_role) {
  using G = Geo<P>;
  using T = TeamGeo<P>;
  using S = TeamShape<P, TEAM>;
  constexpr int NPL = T::NPL, W = G::W, THREADS = 256, PXT = S::PXT, PT = S::PT, CG = S::CG;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), h = lane >> 5;
  const FwdParams &f = prm.f;
  unsigned char *occ = smem + T::OCC_OFF;
  float *lgt = reinterpret_cast<float *>(smem + T::LGT_OFF);
  float *red = reinterpret_cast<float *>(smem + T::RED_OFF);
  int *word = reinterpret_cast<int *>(red) + 255;   // what wave 0 found, for the others
  const unsigned char *packed = f.packed + (size_t)(b / (unsigned)f.boards_per_group) * f.packed_stride;
  const float *tail = reinterpret_cast<const float *>(smem + T::TAIL_OFF);   // (from the first stage on)
  // words of it as a lane's accumulator tile holds its channels
  auto tail_tile = [&](int word) __attribute__((always_inline)) {
    f32x16 v;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const f32x4 b4 = *reinterpret_cast<const f32x4 *>(smem + T::TAIL_OFF + 4 * (word + 8 * q + 4 * h));
#pragma unroll
      for (int e = 0; e < 4; ++e) v[4 * q + e] = b4[e];
    }
    return v;
  };
  unsigned char *act = prm.act + (size_t)slot * T::BOARDB;
  unsigned *flags = prm.flags + (size_t)slot * kTeamFlags;
  const __amdgpu_buffer_rsrc_t mem = __builtin_amdgcn_make_buffer_rsrc(act, 0, T::BOARDB, 0x00020000);
  // Is the whole team known to run on this XCD?  Then what it stores goes to the L2 that they share, where the
  // others' loads find it, and not through it to memory.
  const unsigned xcd = __builtin_amdgcn_s_getreg((2 << 11) | 20);   // (hardware register XCC_ID)
  const unsigned xcd_tag = prm.tag << 4 | 8;   // (no word that is zero looks like one)
  bool local = false;
  auto store16 = [&](const v4i &v, int at) __attribute__((always_inline)) {
    if (local) __builtin_amdgcn_raw_buffer_store_b128(v, mem, at, 0, 0);
    else __builtin_amdgcn_raw_buffer_store_b128(v, mem, at, 0, kSc1);
  };
  auto store4 = [&](float v, int at) __attribute__((always_inline)) {
    if (local) __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(int, v), mem, at, 0, 0);
    else __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(int, v), mem, at, 0, kSc1);
  };
  auto store_flag = [&](int word) __attribute__((always_inline)) {
    if (local) __hip_atomic_store(&flags[word], prm.tag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    else __hip_atomic_store(&flags[word], prm.tag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  };
  [[maybe_unused]] const bool trace_on = true;

  // the wave's first tile of squares within the workgroup's, and its group of cout tiles
  const int wpx = wave % S::PG * PT, cg = wave / S::PG;

  // word l * 12 + role: the squares of stage l that the neighbours read are there; kTeamAll further on:
  // all of them
  auto flag_set = [&](int l, int role) {
    return __hip_atomic_load(&flags[l * 12 + role], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == prm.tag;
  };
  auto has_part = [](int l, int role) { return l < 8 || role == 0; };
  int unfinished = -1;   // word of the piece whose inner squares are still being stored
  // Are the inputs of stage l there for `role` (`own`: its own squares are in LDS)?  Bounded; the answer
  // is the same in every thread.  1: yes, 0: no, 2: no need, the stage itself has been done.
  constexpr int kWatch = S::PG * CG == 3 ? 3 : 0;   // the wave that watches the flags: one that has no weights to wait for
  auto wait_inputs = [&](int l, int role, bool own) {
    if (wave == kWatch) {
      // (Looked at once.  A word that is missing is that of a workgroup that has not come as far as the first layer: then this one
      // stores through to memory to the end, which is correct and slower.  It does not happen where a team lies on one XCD, also
      // not in duo_rest_kernel, whose workgroups start as others end: counted over 257 to 1,616 boards, every one saw all.)
      unsigned about = xcd;
      if (l == 1 && lane < TEAM) about = __hip_atomic_load(&flags[kTeamXcd + lane], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) ^ xcd_tag;
      if (l == 1 && __builtin_amdgcn_ballot_w64(about != xcd) == 0) local = true;
      int need = -1;   // the word of stage l - 1 that this lane watches (less the stage's first)
      if (lane < TEAM && (l == 8 || lane == role - 1 || lane == role + 1)) need = lane;
      if (lane == 62 && !own) need = kTeamAll + role;
      int got = 0;
      for (int k = 0; k < prm.polls && got == 0; ++k) {
        const bool ok = need < 0 || flag_set(l - 1, need);
        const bool done = lane == 63 && flag_set(l, role);
        if (__builtin_amdgcn_ballot_w64(!ok) == 0) got = 1;
        if (__builtin_amdgcn_ballot_w64(done) != 0) got = 2;
      }
      if (lane == 0) *word = got | (local ? 4 : 0);
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // (the inner squares' stores)
    __syncthreads();
    const int got = __builtin_amdgcn_readfirstlane(*word);
    if (tid == 0 && unfinished >= 0) store_flag(kTeamAll + unfinished);
    local = (got & 4) != 0;
    unfinished = -1;
    __syncthreads();
    return got & 3;
  };
  auto raise_flag = [&](int l, int role) {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // this wave's stores have arrived
    __syncthreads();
    if (tid == 0) store_flag(l * 12 + role);
  };

  // The LDS region: positions of the board rows around a role's squares, from the row above the first.
  // region_role's own squares hold the outputs of layer region_layer (0-based), or nothing (-1).
  int region_role = -1, region_layer = -1;
  struct Span {
    int p0, p1, base;   // first and last square, first position
  };
  auto span_of = [](int role) __attribute__((always_inline)) {
    const int p0 = role * PXT * 32, p1 = p0 + PXT * 32 - 1;
    return Span{p0, p1 < kPix ? p1 : kPix - 1, p0 / kBoard * kPitch};
  };
  auto record = [](int p, int base) __attribute__((always_inline)) {
    const int r = p / kBoard;
    return ((r + 1) * kPitch + (p - r * kBoard + 1) - base) * T::RECB;
  };
  auto clear_region = [&](const Span &sp) __attribute__((always_inline)) {   // (its padding stays clear from then on)
    const v4i z = {0, 0, 0, 0};
    const int bytes = ((sp.p1 / kBoard - sp.p0 / kBoard + 3) * kPitch + 1) * T::RECB;
    for (int i = tid; i < bytes / 16; i += THREADS) reinterpret_cast<v4i *>(smem)[i] = z;
    __syncthreads();
  };
  // Squares between LDS and memory, a layer of C channels: a thread has square `sq` of those at hand and 16-byte unit
  // `j` of each plane (then of the fp6 blocks), so that all its addresses are two sums and constants.
  auto unit_of = [&](auto cc, int &sq, int &j) __attribute__((always_inline)) {
    constexpr int J = decltype(cc)::value / 8;
    int t = tid;   // (formed where it is used, not kept for all stages)
    asm volatile("" : "+v"(t));
    sq = t / J;
    j = t - sq * J;
  };
  constexpr int PARTS = NPL + (P::LO6 ? 1 : 0);
  auto part_there = [](auto cc, int k, int j) __attribute__((always_inline)) { return k < NPL || j < decltype(cc)::value / 16; };
  auto part_mem = [](auto cc, int q, int k, int j) __attribute__((always_inline)) {
    constexpr int C = decltype(cc)::value;
    return (q * T::units(C) + k * (C / 8) + j) * 16;
  };
  auto part_lds = [](int k, int j) __attribute__((always_inline)) { return (k < NPL ? k * 192 : T::LO_OFF) + j * 16; };

  // Outputs of layer L (own squares): into the records, and to memory what the neighbours read.
  // acc: N tiles of squares from the workgroup's tile px on
  auto write_out = [&](auto lc, auto nc, int role, const Span &sp, bool active, const auto &acc, int px, int t0) __attribute__((always_inline)) {
    constexpr int L = decltype(lc)::value, N = decltype(nc)::value, C = kCoutArr[L], NT = C / 32;
    constexpr int TT = S::tiles(NT);
    constexpr bool LO = P::LO6 && ((P::LO_MASK >> (L + 1)) & 1);
    if (active) {
#pragma unroll
      for (int i = 0; i < N; ++i) {
        const int p = sp.p0 + (px + i) * 32 + (lane & 31), pc = p < kPix ? p : kPix - 1;
        const int rec = record(pc, sp.base);
#pragma unroll
        for (int t = 0; t < TT; ++t)
          if (t0 + t < NT) team_store<P, LO, (L >= 2)>(smem, rec, h, t0 + t, acc[i][t]);
      }
    }
    __syncthreads();
    int sq, j;
    unit_of(IC<C>{}, sq, j);
    constexpr int PER = THREADS / (C / 8);   // squares at a time
    auto to_memory = [&](int q) __attribute__((always_inline)) {
      const unsigned char *from = smem + record(q, sp.base);
      v4i v[PARTS];
#pragma unroll
      for (int k = 0; k < PARTS; ++k)
        if (part_there(IC<C>{}, k, j)) v[k] = *reinterpret_cast<const v4i *>(from + part_lds(k, j));
#pragma unroll
      for (int k = 0; k < PARTS; ++k)
        if (part_there(IC<C>{}, k, j)) store16(v[k], T::act_off(L) + part_mem(IC<C>{}, q, k, j));
    };
    // twenty squares at either end (all of them where there are no more), then the rest
    const int n = sp.p1 - sp.p0 + 1;
    if (sq < 20 && sq < n) to_memory(sp.p0 + sq);
    if (sq < 20 && sq < n - 20) to_memory(sp.p1 - sq);
    raise_flag(L, role);
    if (sq < PER)
      for (int q = sp.p0 + 20 + sq; q <= sp.p1 - 20; q += PER) to_memory(q);
    unfinished = L * 12 + role;
    region_role = role;
    region_layer = L;
  };

  auto conv_stage = [&](auto lc, int role) __attribute__((always_inline)) -> bool {
    constexpr int L = decltype(lc)::value;
    constexpr int NT = kCoutArr[L] / 32, TT = S::tiles(NT), D = team_ring<P, TT, PT>();
    constexpr int C = kCinArr[L];
    // (opaque per stage: what follows from it is formed here and not, for all stages, in front of the
    // loop over them, in several hundred scalar registers that get spilled)
    int t0 = cg * TT;
    asm volatile("" : "+s"(t0));
    const bool active = cg < CG && t0 < NT;
    const Span sp = span_of(role);
    const WFrags wl = layer_weights<P, L>(packed, lane);
    C6_MARK(6 * L);
    const bool own = region_role == role && region_layer == L - 1;
    v4i ring[D][TT][W];
    f32x16 acc[PT][TT], low[PT][TT];
    auto first_weights = [&]() __attribute__((always_inline)) {
#pragma unroll
      for (int d = 0; d < D; ++d)
#pragma unroll
        for (int t = 0; t < TT; ++t)
#pragma unroll
          for (int i = 0; i < W; ++i) ring[d][t][i] = wl[team_frag<P, L>(d, t0 + t < NT ? t0 + t : NT - 1) + i];
      __builtin_amdgcn_sched_barrier(0);
    };
    // (on their way while the neighbours are waited for; the wave that does the waiting asks for its own behind that)
    if (active && wave != kWatch) first_weights();
    const int got = wait_inputs(L, role, own);
    if (got != 1) return got == 2;
    C6_MARK(6 * L + 1);
    // ---- the neighbours' squares (and, after helping out elsewhere, the own ones) into LDS ----
    if (region_role != role) clear_region(sp);
    const int q0 = sp.p0 - 20 > 0 ? sp.p0 - 20 : 0, q1 = sp.p1 + 20 < kPix ? sp.p1 + 20 : kPix - 1;
    int sq, j;
    unit_of(IC<C>{}, sq, j);
    auto from_memory = [&](int q, v4i (&v)[PARTS]) __attribute__((always_inline)) {
#pragma unroll
      for (int k = 0; k < PARTS; ++k)
        if (part_there(IC<C>{}, k, j))
          v[k] = __builtin_amdgcn_raw_buffer_load_b128(mem, T::act_off(L - 1) + part_mem(IC<C>{}, q, k, j), 0, kSc1);
    };
    auto to_region = [&](int q, const v4i (&v)[PARTS]) __attribute__((always_inline)) {
      unsigned char *at = smem + record(q, sp.base);
#pragma unroll
      for (int k = 0; k < PARTS; ++k)
        if (part_there(IC<C>{}, k, j)) *reinterpret_cast<v4i *>(at + part_lds(k, j)) = v[k];
    };
    v4i left[PARTS], right[PARTS];
    const bool has_left = sq < sp.p0 - q0 && sq < 20, has_right = sq < q1 - sp.p1 && sq < 20;
    if (has_left) from_memory(q0 + sq, left);
    if (has_right) from_memory(sp.p1 + 1 + sq, right);
    if (active && wave == kWatch) first_weights();
    __builtin_amdgcn_sched_barrier(0);
    if (has_left) to_region(q0 + sq, left);
    if (has_right) to_region(sp.p1 + 1 + sq, right);
    if (!own && sq < THREADS / (C / 8))
      for (int q = sp.p0 + sq; q <= sp.p1; q += THREADS / (C / 8)) {
        v4i v[PARTS];
        from_memory(q, v);
        to_region(q, v);
      }
    region_role = -1;   // (until the outputs are in place)
    if (active) {
#pragma unroll
      for (int t = 0; t < TT; ++t) {
        const int word = bias_offset(L) + 32 * (t0 + t < NT ? t0 + t : NT - 1);
#pragma unroll
        for (int i = 0; i < PT; ++i) {
          acc[i][t] = tail_tile(word);
          if constexpr (T::SPLIT) low[i][t] = tail_tile(G::TAIL_BIAS_LOW + word);
        }
      }
    }
    __syncthreads();
    C6_MARK(6 * L + 2);
    // ---- contraction ----
    int p[PT], rec[PT];
    bool ok[PT];
#pragma unroll
    for (int i = 0; i < PT; ++i) {
      p[i] = sp.p0 + (wpx + i) * 32 + (lane & 31);
      ok[i] = p[i] < kPix;
      rec[i] = record(ok[i] ? p[i] : kPix - 1, sp.base);
    }
    if (active) team_conv<P, L, TT, PT>(smem, packed, wl, ring, lane, rec, t0, acc, low);
    C6_MARK(6 * L + 3);
    if constexpr (L < 7) {
      __syncthreads();   // everybody has read this layer's input
      write_out(lc, IC<PT>{}, role, sp, active, acc, wpx, t0);
    } else {
      // heads: this wave's share of the policy (per square) and of the value
      const float *pw = tail + kBiasTotal + 4 * h;
      const int tile = role * PXT + wpx;   // of the twelve
      if constexpr (T::SPLIT) {
        if (active) {
#pragma unroll
          for (int t = 0; t < TT; ++t) {
            if (t0 + t >= NT) continue;
            float pol[PT], val[PT];
#pragma unroll
            for (int i = 0; i < PT; ++i) pol[i] = val[i] = 0.0f;
            float a[PT][16];
#pragma unroll
            for (int i = 0; i < PT; ++i) silu_tile<P>(acc[i][t], a[i]);
#pragma unroll
            for (int q = 0; q < 4; ++q)
#pragma unroll
              for (int e = 0; e < 4; ++e) {
                const float p1 = pw[32 * (t0 + t) + 8 * q + e], v1 = pw[kHeadC + 32 * (t0 + t) + 8 * q + e];
#pragma unroll
                for (int i = 0; i < PT; ++i) {
                  pol[i] = fmaf(a[i][4 * q + e], p1, pol[i]);
                  val[i] = fmaf(a[i][4 * q + e], v1, val[i]);
                }
              }
#pragma unroll
            for (int i = 0; i < PT; ++i) {
              const unsigned bits = __builtin_bit_cast(unsigned, pol[i]);
              const auto x = __builtin_amdgcn_permlane32_swap(bits, bits, false, false);
              const unsigned x0 = x[0], x1 = x[1];
              const float tot = __builtin_bit_cast(float, x0) + __builtin_bit_cast(float, x1);
              const float vs = wave_sum(ok[i] ? val[i] : 0.0f);
              if (h == 0 && ok[i]) store4(tot, T::HEAD_OFF + ((t0 + t) * 384 + p[i]) * 4);
              if (lane == 0) store4(vs, T::VAL_OFF + ((t0 + t) * 12 + tile + i) * 4);
            }
          }
        }
      } else {
        // The one-workgroup kernel runs one chain of multiply-adds over the channels of a lane's
        // square, cout tile after cout tile: the groups of cout tiles take turns and hand it on.
        float *chain = reinterpret_cast<float *>(smem + T::OCC_OFF);   // (not in use before the last stage)
        f32x4 pw4[TT][4];
        if (active) {
#pragma unroll
          for (int t = 0; t < TT; ++t) {
            if (t0 + t >= NT) continue;
            float val0[PT];
#pragma unroll
            for (int i = 0; i < PT; ++i) {
              val0[i] = 0.0f;
              float a[16];
              silu_tile<P>(acc[i][t], a);
#pragma unroll
              for (int e = 0; e < 16; ++e) acc[i][t][e] = a[e];
            }
#pragma unroll
            for (int q = 0; q < 4; ++q) {
              pw4[t][q] = *reinterpret_cast<const f32x4 *>(pw + 32 * (t0 + t) + 8 * q);
              const f32x4 vw4 = *reinterpret_cast<const f32x4 *>(pw + kHeadC + 32 * (t0 + t) + 8 * q);
#pragma unroll
              for (int i = 0; i < PT; ++i) {
                float vs = 0.0f;
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                  const float a = acc[i][t][4 * q + e];
                  val0[i] = fmaf(a, vw4[e], val0[i]);
                  vs = fmaf(a, vw4[e], vs);
                }
                // (tile 0: one chain over its sixteen channels; the others: one sum per four)
                if (t0 + t > 0) store4(vs, T::VAL_OFF + (((tile + i) * 9 + 1 + 4 * (t0 + t - 1) + q) * 64 + lane) * 4);
              }
            }
#pragma unroll
            for (int i = 0; i < PT; ++i)
              if (t0 + t == 0) store4(val0[i], T::VAL_OFF + ((tile + i) * 9 * 64 + lane) * 4);
          }
        }
#pragma unroll
        for (int turn = 0; turn < CG; ++turn) {
          if (turn == cg && active) {
#pragma unroll
            for (int k = 0; k < PT; ++k) {
              float pol = cg > 0 ? chain[(wpx + k) * 64 + lane] : 0.0f;
#pragma unroll
              for (int t = 0; t < TT; ++t) {
                if (t0 + t >= NT) continue;
#pragma unroll
                for (int i = 0; i < 16; ++i) pol = fmaf(acc[k][t][i], pw4[t][i / 4][i % 4], pol);
              }
              chain[(wpx + k) * 64 + lane] = pol;
              if (turn == CG - 1 || t0 + TT >= NT) {
                const unsigned bits = __builtin_bit_cast(unsigned, pol);
                const auto x = __builtin_amdgcn_permlane32_swap(bits, bits, false, false);
                const unsigned x0 = x[0], x1 = x[1];
                const float tot = __builtin_bit_cast(float, x0) + __builtin_bit_cast(float, x1);
                if (h == 0 && ok[k]) store4(tot, T::HEAD_OFF + p[k] * 4);
              }
            }
          }
          if (turn + 1 < CG) __syncthreads();
        }
      }
      raise_flag(L, role);
    }
    C6_MARK(6 * L + 4);
    return true;
  };

  // first layer: every workgroup stages the part of the board that its squares see
  auto first_stage = [&](int role) __attribute__((always_inline)) -> bool {
    const Span sp = span_of(role);
    int *flag = reinterpret_cast<int *>(red) + 64;   // [0]: third plane varies, [1]: an input is not exact in bf16
    constexpr int N1 = PXT > 4 ? 2 : 1;   // (one cout tile: a wave per tile of squares, or per two)
    const int px = wave * N1 < PXT ? wave * N1 : 0;
    const bool active = wave * N1 < PXT;
    region_role = -1;
    f32x16 acc[N1][1];
    if (active) {
      // (the table holds the squares as the one-workgroup kernels' lanes do: by tile of 32)
#pragma unroll
      for (int n = 0; n < N1; ++n) {
        const WFrags tb = packed_frags<P>(packed, lane, G::PLANE2_FRAG_OFF + (role * PXT + px + n) * 4);
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const f32x4 t4 = __builtin_bit_cast(f32x4, tb[q]);
#pragma unroll
          for (int e = 0; e < 4; ++e) acc[n][0][4 * q + e] = t4[e];
        }
      }
    }
    constexpr int TAIL_UNITS = (G::TAIL_FLOATS / 4 + THREADS - 1) / THREADS;
    v4i tl[TAIL_UNITS];
#pragma unroll
    for (int i = 0; i < TAIL_UNITS; ++i)
      if (tid + i * THREADS < G::TAIL_FLOATS / 4) tl[i] = reinterpret_cast<const v4i *>(packed + G::TAIL_OFF)[tid + i * THREADS];
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
          for (int ch = 0; ch < 3; ++ch) xin[k][ch] = load_input(f.x, f.x_dtype, ((size_t)b * 3 + ch) * kPix + sq);
        }
      }
    }
    // halo rows that the squares' 23 kernel rows reach (and the zero row behind the last): those from ha on are staged
    static_assert(((PXT * 32 + kBoard - 2) / kBoard + kK1) * 3 + 1 <= T::COPY_ROWS, "rows of the copies");
    const int ha = sp.p0 / kBoard * 3, hb = (sp.p1 / kBoard + kK1) * 3 + 1;
    {
      const v4i z = {0, 0, 0, 0};
      const int per = (hb - ha) * (kL1RowPitch * G::EB / 16);
#pragma unroll
      for (int s = 0; s < G::E; ++s)
        for (int i = tid; i < per; i += THREADS)
          *reinterpret_cast<v4i *>(smem + s * T::COPY_BYTES + i * 16) = z;
    }
#pragma unroll
    for (int i = 0; i < TAIL_UNITS; ++i)
      if (tid + i * THREADS < G::TAIL_FLOATS / 4) reinterpret_cast<v4i *>(smem + T::TAIL_OFF)[tid + i * THREADS] = tl[i];
    if (tid < 2) flag[tid] = 0;
    if (tid == 0) red[66] = xin[0][2];
    __syncthreads();
    const float c2 = red[66];
    bool varies = false;
#pragma unroll
    for (int k = 0; k < 2; ++k)
      if (tid + k * THREADS < kPix) varies |= __builtin_bit_cast(int, xin[k][2]) != __builtin_bit_cast(int, c2);
    if (varies) flag[0] = 1;
    // (the tag and the XCD in one word, at a place that holds nothing else; behind the input's loads, so that
    // nothing waits for its acknowledgement)
    if (tid == 0 && role == my_role)
      __hip_atomic_store(&flags[kTeamXcd + role], xcd_tag ^ xcd, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __syncthreads();
    const bool plane2_varies = flag[0] != 0;
    int parts = 1;
    if constexpr (T::SPLIT) {
      bool inexact = false;
#pragma unroll
      for (int k = 0; k < 2; ++k)
        if (tid + k * THREADS < kPix)
#pragma unroll
          for (int ch = 0; ch < 3; ++ch)
            inexact |= (ch < 2 || plane2_varies) && (__builtin_bit_cast(int, xin[k][ch]) & 0xffff) != 0;
      if (inexact) flag[1] = 1;
      __syncthreads();
      parts = flag[1] != 0 ? 3 : 1;
    }
    const int rows = (plane2_varies ? G::STEPS1 : G::FAST1_STEPS) / 3;
    int row0[N1];
#pragma unroll
    for (int n = 0; n < N1; ++n) {
      const int p = sp.p0 + (px + n) * 32 + (lane & 31);
      const int pc = p < kPix ? p : kPix - 1, r = pc / kBoard, c = pc - r * kBoard, sh = c % G::E;
      row0[n] = sh * T::COPY_BYTES + ((r * 3 - ha) * kL1RowPitch + (c - sh)) * G::EB + (plane2_varies ? kL1RowsHalf : 1) * h * kL1RowPitch * G::EB;
    }
    const int rowb = (plane2_varies ? 1 : 3) * kL1RowPitch * G::EB;
    const WFrags wl = plane2_varies ? layer_weights<P, 0>(packed, lane) : packed_frags<P>(packed, lane, G::FAST1_OFF);
    if (active) {
      const f32x16 b0 = tail_tile(bias_offset(0));
#pragma unroll
      for (int n = 0; n < N1; ++n)
#pragma unroll
        for (int i = 0; i < 16; ++i) acc[n][0][i] = plane2_varies ? b0[i] : fmaf(c2, acc[n][0][i], b0[i]);
    }
    f32x16 low[N1], large[N1];   // SPLIT: small products; the large ones, once all parts but the first follow
#pragma unroll
    for (int n = 0; n < N1; ++n)
#pragma unroll
      for (int i = 0; i < 16; ++i) low[n][i] = large[n][i] = 0.0f;
    if constexpr (T::SPLIT) {
      if (active) {
#pragma unroll
        for (int n = 0; n < N1; ++n) low[n] = tail_tile(G::TAIL_BIAS_LOW + bias_offset(0));
      }
    }
#pragma unroll 1
    for (int part = 0; part < parts; ++part) {
      if (part > 0) __syncthreads();
#pragma unroll
      for (int k = 0; k < 2; ++k) {
        const int sq = tid + k * THREADS;
        const int row = sq / kBoard, col = sq - row * kBoard;
#pragma unroll
        for (int ch = 0; ch < 3; ++ch) {
          if (ch >= (plane2_varies ? 3 : 2)) break;
          const int hrow = (row + kK1 / 2) * 3 + ch;
          if (sq >= kPix) continue;
          unsigned short v16;
          if constexpr (T::SPLIT) {
            v16 = bf16_part(xin[k][ch]);
            xin[k][ch] = bf16_rest(xin[k][ch], v16);
          } else {
            v16 = bits16<P>(xin[k][ch]);
          }
          if (hrow < ha || hrow >= hb) continue;
#pragma unroll
          for (int q = 0; q < G::E; ++q)
            *reinterpret_cast<unsigned short *>(smem + q * T::COPY_BYTES + ((hrow - ha) * kL1RowPitch + (col + kK1 / 2 - q)) * G::EB) = v16;
        }
      }
      __syncthreads();
      C6_MARK(1);
      if (active) {
        // Kernel rows (three fragments each), the row's activations asked for a row ahead and its weights DW rows, one
        // load behind each MFMA: a lone wave issues an instruction per five cycles, and what it issues between two rows
        // the matrix core waits for (all of a row's loads in front of it: bf16 54 cycles per MFMA, fp32 58).
        constexpr int DW = W == 3 ? (N1 > 1 ? 2 : 4) : 8;
        static_assert(DW % 2 == 0, "activations alternate");
        v4i w[DW][3][W], a[2][3][N1];
        auto weight = [&](int row, int i, int j) __attribute__((always_inline)) {
          return wl[((row < rows ? row : rows - 1) * 3 + i) * W + j];
        };
        auto activation = [&](int row, int i, int n) __attribute__((always_inline)) {
          return *reinterpret_cast<const v4i *>(smem + row0[n] + (row < rows ? row : rows - 1) * rowb + i * 16);
        };
        auto one_row = [&](int row, auto sc) __attribute__((always_inline)) {
          constexpr int s8 = decltype(sc)::value;
#pragma unroll
          for (int i = 0; i < 3; ++i) {
            static_for<0, W>([&](auto jc) __attribute__((always_inline)) {
              constexpr int j = decltype(jc)::value;
#pragma unroll
              for (int n = 0; n < N1; ++n) mma<P>(w[s8][i][j], a[s8 % 2][i][n], T::SPLIT && j > 0 ? low[n] : acc[n][0]);
              w[s8][i][j] = weight(row + DW, i, j);
            });
#pragma unroll
            for (int n = 0; n < N1; ++n) a[(s8 + 1) % 2][i][n] = activation(row + 1, i, n);
          }
#pragma unroll
          for (int i = 0; i < 3 * W; ++i) {
            __builtin_amdgcn_sched_group_barrier(0x008, N1, 0);                    // one MFMA per tile
            __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);                     // one weight
            if (i % W == W - 1) __builtin_amdgcn_sched_group_barrier(0x100, N1, 0);   // one LDS read per tile
          }
          __builtin_amdgcn_sched_barrier(0);
        };
#pragma unroll
        for (int s8 = 0; s8 < DW; ++s8)
#pragma unroll
          for (int i = 0; i < 3; ++i) {
#pragma unroll
            for (int j = 0; j < W; ++j) w[s8][i][j] = weight(s8, i, j);
            if (s8 == 0)
#pragma unroll
              for (int n = 0; n < N1; ++n) a[0][i][n] = activation(0, i, n);
          }
        int row = 0;
#pragma unroll 1
        for (; row + DW <= rows; row += DW) static_for<0, DW>([&](auto sc) __attribute__((always_inline)) { one_row(row + decltype(sc)::value, sc); });
        static_for<0, DW - 1>([&](auto sc) __attribute__((always_inline)) {
          if (row + decltype(sc)::value < rows) one_row(row + decltype(sc)::value, sc);
        });
        if constexpr (T::SPLIT) {
          if (parts > 1 && part == 0) {
#pragma unroll
            for (int n = 0; n < N1; ++n) {
              large[n] = acc[n][0];
              acc[n][0] = low[n];
#pragma unroll
              for (int i = 0; i < 16; ++i) low[n][i] = 0.0f;
            }
          }
        }
      }
    }
    if constexpr (T::SPLIT) {
#pragma unroll
      for (int n = 0; n < N1; ++n)
#pragma unroll
        for (int i = 0; i < 16; ++i)
          acc[n][0][i] = parts > 1 ? two_sums(large[n][i], low[n][i] + acc[n][0][i]) : two_sums(acc[n][0][i], low[n][i]);
    }
    C6_MARK(2);
    __syncthreads();   // the copies give way to the activations
    clear_region(sp);
    write_out(IC<0>{}, IC<N1>{}, role, sp, active, acc, px, 0);
    C6_MARK(3);
    return true;
  };

  // the heads' sums into logits, value, draw and (cascade) the list of close boards: one workgroup
  auto last_stage = [&](int role) __attribute__((always_inline)) -> bool {
    const int got = wait_inputs(8, role, true);
    if (got != 1) return got == 2;
    region_role = -1;
    const float *valw = tail + kBiasTotal + kHeadC;
    const float polb = valw[kHeadC], valb = valw[kHeadC + 1];
    auto partial = [&](int at) __attribute__((always_inline)) {
      return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(mem, at, 0, kSc1));
    };
    const bool state = f.x_dtype == C6_DT_BOARD_I8;
    long long src = state && f.index ? f.index[b] : (long long)b;
    if (state) src = src < 0 ? 0 : (src >= f.num_states ? f.num_states - 1 : src);
    for (int p = tid; p < kPix; p += THREADS) {
      float z = partial(T::HEAD_OFF + p * 4);
      if constexpr (T::SPLIT) z = (z + partial(T::HEAD_OFF + (384 + p) * 4)) + partial(T::HEAD_OFF + (768 + p) * 4);
      if constexpr (T::SPLIT) z = split_logit(z, polb);
      else z += polb;
      bool taken;
      if (f.mask_mode == C6_MASK_LEGAL) {
        taken = f.legal[(size_t)b * kPix + p] == 0;
      } else if (state) {
        const int stone = reinterpret_cast<const int8_t *>(f.x)[(size_t)src * kPix + (f.view ? d4_from_view(p, f.view) : p)];
        const int me = f.player[src];
        taken = stone == me || stone == -me;
      } else {
        taken = load_input(f.x, f.x_dtype, (size_t)b * 3 * kPix + p) != 0.0f || load_input(f.x, f.x_dtype, ((size_t)b * 3 + 1) * kPix + p) != 0.0f;
      }
      const bool masked = taken && f.mask_mode != C6_MASK_NONE;
      lgt[p] = z;
      occ[p] = (unsigned char)((masked ? 1 : 0) | (taken ? 2 : 0));
      if (f.logits != nullptr) {
        const float v = masked ? f.fill : z;
        const size_t at = (size_t)b * kPix + p;
        if (f.logits_dtype == C6_DT_F32) static_cast<float *>(f.logits)[at] = v;
        else if (f.logits_dtype == C6_DT_BF16) static_cast<unsigned short *>(f.logits)[at] = __builtin_bit_cast(unsigned short, (__bf16)v);
        else static_cast<unsigned short *>(f.logits)[at] = __builtin_bit_cast(unsigned short, (_Float16)v);
      }
    }
    if constexpr (T::SPLIT) {
      if (tid < 36) red[tid] = partial(T::VAL_OFF + tid * 4);
    } else {
      // as lane `lane` of wave `wave` of the one-workgroup kernel adds its three squares' sums up
      float part[3][9], vsum = 0.0f;
      bool valid[3];
#pragma unroll
      for (int j = 0; j < 3; ++j) {
        valid[j] = (3 * wave + j) * 32 + (lane & 31) < kPix;
#pragma unroll
        for (int i = 0; i < 9; ++i) part[j][i] = partial(T::VAL_OFF + (((3 * wave + j) * 9 + i) * 64 + lane) * 4);
      }
#pragma unroll
      for (int i = 0; i < 9; ++i)
#pragma unroll
        for (int j = 0; j < 3; ++j) vsum += valid[j] ? part[j][i] : 0.0f;
      vsum = wave_sum(vsum);
      if (lane == 0) red[wave] = vsum;
    }
    __syncthreads();
    if constexpr (T::SPLIT) {
      if (wave == 3 && f.value != nullptr) {   // (beside the draw)
        const double sum = split_value_sum(lane, [&](int i) { return red[i]; });
        if (lane == 0) f.value[b] = split_value(sum, valb);
      }
    } else {
      if (tid == 192 && f.value != nullptr) {   // (beside the draw and the margin)
        float s = 0.0f;
#pragma unroll
        for (int w = 0; w < 4; ++w) s += red[w];
        f.value[b] = tanhf(s * (1.0f / kPix) + valb);
      }
    }
    if (f.actions != nullptr && wave == 0) {
      int a;
      float lp;
      wave_sample(
          lane, f.u[b], f.inv_temperature, [&](int i) { return lgt[i]; }, [&](int i) { return (occ[i] & 1) == 0; }, a, lp);
      if (lane == 0) {
        f.actions[b] = a;
        if (f.logprob != nullptr) f.logprob[b] = lp;
      }
    }
    if constexpr (P::ID == C6_PREC_BF16) {
      if (f.redo_mode == kRedoDetect && wave == 1) {   // (a run of one board: see fused_pipe_kernel)
        const bool again = wave_margin_below(
            lane, f.redo_threshold, [&](int i) { return lgt[i]; }, [&](int i) { return (occ[i] & 2) == 0; });
        if (lane == 0) {
          __hip_atomic_store(&f.redo_counts[(unsigned)f.redo_grid + slot], again ? 1 : 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
          f.redo_list[redo_entry(f.redo_grid + (long long)slot, f.redo_grid, f.redo_per)] = (int)b;
          if (again) store_flag(kTeamListed);   // (in front of the stage's flag)
        }
      }
    }
    raise_flag(8, role);
    C6_MARK(49);
    return true;
  };

  // Stages in order; `help`: a wait ran out, do the earliest piece that has no flag instead.
  C6_MARK(0);
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
          const bool open = lane < TEAM && !flag_set(k, lane);
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
  __syncthreads();
}

// How many workgroups share a board (team_size, below) when there are `boards` of them: as many as fit the chip at once, where
// that beats one workgroup (1: the one-workgroup kernels).  With fewer workgroups per board more waves read
// the same weights, and the L1's 64 bytes a cycle bound the layers; the 16-bit one-workgroup kernel hides its epilogues
// behind its MFMAs, which a team does not.  Measured, us, teams of 12 / 6 / 3 / 2 against one workgroup each, boards:
//   fp32  16: 47 / 62 / 77 / 102   40: 71 / 81 / 108 (without 12)   80: 94 / 113   128: 131   one workgroup each, 129: 147
//   bf16  16: 31 / 41 / 49 / 61 / 45      21: 36 / 41 / - / - / 46   40: 42 / 50 / 61 / 45   42: 48 (teams on two XCDs)
//   bf16 + fp6  21: 44 / 51 / 64 / 81 / 63    42: 57 / 68 / 84 / 64    with low weights  21: 52 / 60 / 78 / 101 / 89
//   42: 67 / 84 / 106 / 89    72: 89 / 110 / 89 (behind a first pass, 53 listed boards, 85 against 110)
// Four workgroups per board are never the best of these by more than 4 %.
//
// The most boards that teams of a size take:
template <class P> __host__ __device__ inline long long team_most(int wgs, int size) {
  if (size == 6 && !TeamGeo<P>::SPLIT && !P::LO6) return wgs * 5 / 32;   // (where all teams have an XCD to themselves)
  if (size == 3 && P::LO6 && P::WLO == 1) return wgs * 2 / 7;
  return wgs / size;
}
template <class P> constexpr int team_least() { return TeamGeo<P>::SPLIT ? 2 : (P::WLO ? 3 : 6); }
template <class P> __host__ __device__ inline int team_size(long long boards, int wgs) {
  const int sizes[4] = {12, 6, 3, 2};
  for (int i = 0; i < 4; ++i)
    if (sizes[i] >= team_least<P>() && boards <= team_most<P>(wgs, sizes[i])) return sizes[i];
  return 1;
}

// exchange memory per board (fp32: of both ways through it, and the second one's flags)
template <class P> constexpr size_t team_board_bytes() {
  if constexpr (kParts<P> == 2) return TeamGeo<P>::BOARDB + TeamGeo<PrecF32X>::BOARDB + kTeamFlags * 4;
  else return TeamGeo<P>::BOARDB;
}
template <class P> inline long long team_most(int wgs) { return team_most<P>(wgs, team_least<P>()); }

// Which team this workgroup belongs to (`items` of them; a slot beyond: to none) and as which member.  A team
// on one XCD (workgroup i runs on XCD i % 8), neighbouring boards on the same one, where that many teams fit: a weight
// set then comes into one L2 and not into eight.  (27 listed boards of 128 weight sets: the cascade 183 -> 179 us; of 16
// sets, 6 boards: 105 -> 96 us; eight fp32 boards of one set 66.5 -> 64.4 us.)
struct TeamPlace {
  unsigned slot;
  int role;
};
__device__ __forceinline__ TeamPlace team_place(unsigned items, int team, unsigned wg, unsigned wgs) {   // (wg of wgs)
  if (wgs % 8 == 0) {
    const unsigned per = (items + 7) / 8, l = wg / 8;
    if (per * (unsigned)team <= wgs / 8)
      return {l / (unsigned)team < per ? wg % 8 * per + l / (unsigned)team : items, (int)(l % (unsigned)team)};
  }
  return {wg / (unsigned)team, (int)(wg % (unsigned)team)};
}
__device__ __forceinline__ TeamPlace team_place(unsigned items, int team) { return team_place(items, team, blockIdx.x, gridDim.x); }

// A workgroup's share of board b, in a team of any size that the mode has.
template <class P>
__device__ __forceinline__ void team_share(const TeamParams &prm, unsigned char *smem, unsigned b, TeamPlace at, int team) {
  if (team == 12) team_board<P, 12>(prm, smem, b, at.slot, at.role);
  if (team == 6) team_board<P, 6>(prm, smem, b, at.slot, at.role);
  if constexpr (team_least<P>() <= 3) {
    if (team == 3) team_board<P, 3>(prm, smem, b, at.slot, at.role);
  }
  if constexpr (team_least<P>() <= 2) {
    if (team == 2) team_board<P, 2>(prm, smem, b, at.slot, at.role);
  }
}

// fp32: c6_half_team.h
template <class P> __device__ __forceinline__ void half_team(const TeamParams &prm, unsigned char *smem, unsigned items, TeamPlace at, int team);
template <class P> __global__ __launch_bounds__(256) void team_forward_kernel(const TeamParams prm) {
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  const unsigned items = (unsigned)prm.f.total_boards;
  const int team = team_size<P>(items, (int)gridDim.x);
  if (team == 1) return;
  const TeamPlace at = team_place(items, team);
  if (at.slot >= items) return;
  if constexpr (kParts<P> == 2) half_team<P>(prm, smem, items, at, team);
  else team_share<P>(prm, smem, prm.first + at.slot, at, team);
}

// The plain 16-bit modes with a few boards beyond whole rounds of one board per CU: teams for them in one launch with the
// two workgroups per CU that serve the others (c6_duo.h).  They start where the first of those end, so the second of the two
// on each CU goes first with its last board (s_setprio): its place is free some 25 us before the other, which had as
// little of the matrix cores as that takes, ends, with an odd number of rounds a board before it; the team's waves, a chain that
// leaves the matrix cores idle most of the time, go in front of the other's.  What it gives stands at team_boards: 777 boards
// in fp16 202 -> 181 us (teams in front without the second workgroup's priority 189; without either, 188 and 71 -> 74 at
// 257 boards).  What bounds it: 512 + 9 boards take 15 us more than 512, of which the other workgroups, alone on their CUs
// in the end, are most.
// Registers: the teams' contractions want more than the 256 that two workgroups per CU leave.  In scratch (80 bytes a lane) is
// what teams of three keep, and with it some addresses of the boards that have a workgroup each: a dozen accesses at the
// head and the end of a board, none between its MFMAs.
// The workgroups per board of a rest (1: none are shared), as many as half of the places hold.  A team lies on one XCD but for
// 17 to 21 boards (of 256 CUs): three teams of twelve do not fit the 32 places that an XCD has, so they are dealt out over all
// XCDs and exchange through memory, as they do without other boards.
template <class P> __host__ __device__ inline int rest_team(long long boards, int cus) {
  if (!has_duo<P>()) return 1;
  if (boards * 12 <= cus) return 12;
  if (boards <= cus * 5 / 32) return 6;
  return boards <= cus * 5 / 16 ? 3 : 1;
}
template <class P> __global__ __launch_bounds__(256, 2) void duo_rest_kernel(const TeamParams prm) {
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  const unsigned cus = gridDim.x / 3, grid = 2 * cus;
  if (blockIdx.x < grid) {
    duo_boards<P, true>(prm.f, smem, grid);
    return;
  }
  const unsigned wg = blockIdx.x - grid;
  const int team = rest_team<P>(prm.rest, (int)cus);
  const TeamPlace at = team_place(prm.rest, team, wg, cus);
  if (at.slot >= prm.rest) return;
  const unsigned b = (unsigned)prm.f.total_boards + at.slot;
  __builtin_amdgcn_s_setprio(3);
  if (team == 12) team_board<P, 12>(prm, smem, b, at.slot, at.role);
  if (team == 6) team_board<P, 6>(prm, smem, b, at.slot, at.role);
  if (team == 3) team_board<P, 3>(prm, smem, b, at.slot, at.role);
}

// The cascade over so few boards that twelve workgroups share each: both passes in one launch.  Where a board's last
// stage is done, its team sees whether the board was listed and goes through it again in the second pass's mode, or ends:
// one board that is not listed 41.4 -> 33.3 us with its mask (the second launch found nothing to do), of which waiting
// for the verdict is 2.
template <class P2> __global__ __launch_bounds__(256) void team_cascade_kernel(const TeamCascadeParams prm) {
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  const unsigned items = (unsigned)prm.first.f.total_boards;   // (at most 64)
  const TeamPlace at = team_place(items, 12);
  if (at.slot >= items) return;
  team_board<PrecBF16, 12>(prm.first, smem, at.slot, at.slot, at.role);
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const unsigned tag = prm.first.tag;
  auto word = [&](unsigned slot, int w) {
    return __hip_atomic_load(&prm.first.flags[(size_t)slot * kTeamFlags + w], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  };
  int *verdict = reinterpret_cast<int *>(smem);
  if (wave == 0) {
    // (bounded as every wait; a team without a member that left here finishes by itself)
    int again = -1;
    for (int k = 0; k < 16 * prm.first.polls && again < 0; ++k)
      if (word(at.slot, 8 * 12) == tag) again = word(at.slot, kTeamListed) == tag ? 1 : 0;
    if (lane == 0) *verdict = again;
    if (at.role == 0) {
      // The caller is told how many boards were listed.  Whoever finds all boards done, its own among them, adds them
      // up: the last one does, and two would write the same.
      if (lane == 0)
        __hip_atomic_store(&prm.first.flags[(size_t)at.slot * kTeamFlags + kTeamDone], tag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      const bool open = (unsigned)lane < items && word(lane, kTeamDone) != tag;
      if (__builtin_amdgcn_ballot_w64(open) == 0) {
        const bool listed = (unsigned)lane < items &&
                            __hip_atomic_load(&prm.first.f.redo_counts[lane], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0;
        const unsigned long long m = __builtin_amdgcn_ballot_w64(listed);
        if (lane == 0) *prm.first.f.redo_count = __builtin_popcountll(m);
      }
    }
  }
  __syncthreads();
  const int again = *verdict;
  __syncthreads();
  if (again != 1) return;
  TeamParams second = prm.first;
  second.f.packed = prm.packed;
  second.f.redo_mode = kRedoNone;
  second.act = prm.act;
  second.flags = prm.flags;
  second.tag = tag + 1;
  team_board<P2, 12>(second, smem, at.slot, at.slot, at.role);
}

// The cascade's second pass: what the listed boards leave beyond whole rounds of the workgroups goes to teams, if
// it is no more than they take, and the others to one workgroup each.  One launch, since nobody knows before it runs how
// many are listed; as a launch each, the one without a board took 4.8 us between the passes (512 boards of 128 sets
// 186.6 -> 184.6 us, 4,096 of 8 sets 944.6 -> 937.2, 1,536 boards 447.9 -> 445.1; the kernel itself takes as long as
// fused_pipe_kernel, 2,540 us on 3,300 listed boards).
template <class P> __global__ __launch_bounds__(256) void second_pass_kernel(const TeamParams prm) {
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  unsigned items = listed_runs<P>(prm.f, smem);
  if (threadIdx.x == 0 && blockIdx.x == 0) *prm.f.redo_count = (int)items;   // for the caller: boards evaluated twice
  const unsigned rest = items % gridDim.x;
  const int team = rest != 0 && prm.act != nullptr ? team_size<P>(rest, (int)gridDim.x) : 1;
  if (team > 1) {
    items -= rest;
    const TeamPlace at = team_place(rest, team);
    if (at.slot < rest) {
      const unsigned b = listed_board<P>(prm.f, smem, items + at.slot);
      __syncthreads();   // (the runs are read; the team's tiles lie on them)
      team_share<P>(prm, smem, b, at, team);
      if (items != 0) listed_runs<P>(prm.f, smem);
    }
  }
  if (items != 0) pipe_boards<P, true>(prm.f, smem, items);
}

}  // namespace c6
