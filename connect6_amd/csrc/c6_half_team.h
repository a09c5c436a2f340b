// Few boards in fp32, two fp16 parts per operand: a team of workgroups per board as in c6_team.h (included by c6_forward.hip behind it),
// whose exchange, flags and order of work this follows; the arithmetic is c6_half.h's, and the results those of half_forward_kernel bit for
// bit.  Apart from the others' teams, since hardly a loop is the same: the waves' shares of squares and cout tiles, the sums per kernel row, the
// epilogues, the range of what is stored.
#pragma once

namespace c6 {

// How a team of TEAM workgroups shares a layer (TeamShape): each takes PXT of the twelve tiles of squares.
// With four or six tiles of squares (RAGGED) a wave takes half of them (PR).  Of two cout tiles it takes one; of three, one for all its
// squares and the middle one for half of them, which balances the waves (nine tiles' MFMAs in each per k-step of four tiles of squares, fifteen of six:
// the fourth group takes one of them a second time, to the same bytes) and has 64 bytes of weights a cycle or less asked for.  One cout
// tile: the tiles of squares are dealt out to the waves.  (All cout tiles of one tile of squares per wave were 85 bytes a cycle, and two of
// squares in three waves left one idle: 53 boards 96 -> 88 us, 85 boards 104 -> 95 us, 100 boards 132 -> 121 us, 128 boards 140 -> 130 us.)
template <int TEAM> struct HalfTeamShape {
  static constexpr int PXT = 12 / TEAM;
  static constexpr bool RAGGED = PXT >= 4;
  static constexpr int PR = RAGGED ? PXT / 2 : 0;
  static constexpr int PT = RAGGED ? PR : 1, PG = PXT / PT;
  static constexpr int CG = PG == 1 ? 3 : 4 / PG;   // groups of squares' tiles, of cout tiles
  static constexpr int tiles(int nt) { return RAGGED ? (nt == 3 ? 2 : 1) : (nt + CG - 1) / CG; }   // cout tiles of a wave
  // ... and of its pairs of a tile of squares and a cout tile, tiles of squares: all cout tiles of each, or (RAGGED) one: team_used()
  static constexpr int squares(int nt) { return !RAGGED ? PT : (nt == 3 ? PR + (PR + 1) / 2 : (nt == 2 ? PR : (PXT + 3) / 4)); }
};
// does a wave have cout tile t of tile of squares p? (PR: of a ragged shape)
template <int PR> constexpr bool team_used(int p, int t) { return PR == 0 || t == (p < PR ? 0 : 1); }

// k-steps of weights that a wave keeps in flight: the loads take some 800 cycles and a k-step 96 per tile, PT of them in a
// ragged shape
template <int TT, int PT> constexpr int half_team_ring() { return PT * TT == 1 ? 9 : (PT >= 5 ? 2 : (PT >= 3 ? 3 : 6)); }
// ... and those of one unrolled round: a kernel row, or all three of them where a k-step is so short that nine are in flight
template <int L, int TT, int PT> constexpr int half_team_round() { return (PT * TT == 1 ? 9 : 3) * kCinArr[L] / 16; }

// The contraction of 3x3 layer L for PT tiles of 32 squares and TT cout tiles, tile(t) of the layer's (beyond
// its last they repeat it; their results are not used), as half_conv.
//   rec: LDS addresses of the lane's squares' records;  unit: the layer's;  acc: the bias on entry, low: what it leaves out
template <int L, int TT, int PT, int PR, class Tile>
__device__ __forceinline__ void half_team_conv(const unsigned char *smem, const unsigned char *packed, const WFrags &wl,
                                               v4i (&ring)[half_team_ring<TT, PT>()][TT][2], int lane,
                                               const int (&rec)[PT], Tile tile, float unit, f32x16 (&acc)[PT][TT],
                                               f32x16 (&low)[PT][TT]) {
  using T = TeamGeo<PrecF32S>;
  constexpr int NT = kCoutArr[L] / 32, W = Geo<PrecF32S>::W, NPL = T::NPL, D = half_team_ring<TT, PT>();
  constexpr int KC = kCinArr[L] / 16, KS = 9 * KC;
  constexpr int U = half_team_round<L, TT, PT>();
  static_assert(KS % U == 0 && U % D == 0, "ring");
  int corner[PT];
#pragma unroll
  for (int p = 0; p < PT; ++p) corner[p] = rec[p] - (kPitch + 1) * T::RECB + 16 * (lane >> 5);
  // k-step v of round r: (tap, 16 channels)
  auto frag = [&](int r, int v, int p, int pl) __attribute__((always_inline)) {
    const int off = ((v / KC / 3) * kPitch + v / KC % 3) * T::RECB + (v % KC) * 32;
    return *reinterpret_cast<const v4i *>(smem + corner[p] + r * kPitch * T::RECB + off + pl * 192);
  };
  // activations two k-steps ahead; one where that is nine MFMAs or more
  constexpr int AHEAD = PT > 2 ? 1 : 2;
  v4i a[AHEAD + 1][PT][NPL];
#pragma unroll
  for (int v = 0; v < AHEAD; ++v)
#pragma unroll
    for (int p = 0; p < PT; ++p)
#pragma unroll
      for (int i = 0; i < NPL; ++i) a[v][p][i] = frag(0, v, p, i);
  f32x16 sum[PT][TT];   // the largest products of a kernel row
#pragma unroll 1
  for (int r = 0; r < KS / U; ++r) {
    static_for<0, U>([&](auto vc) __attribute__((always_inline)) {
      constexpr int v = decltype(vc)::value;
      // (behind the last k-step: the last round again, unused)
      const int rn = v + AHEAD < U ? r : (r + 1 < KS / U ? r + 1 : r);
#pragma unroll
      for (int p = 0; p < PT; ++p)
#pragma unroll
        for (int i = 0; i < NPL; ++i) a[(v + AHEAD) % (AHEAD + 1)][p][i] = frag(rn, (v + AHEAD) % U, p, i);
      auto refill = [&](int t) __attribute__((always_inline)) {
        const int kn = r * U + v + D;   // (behind the last k-steps: the last one again, unused)
        const int f = ((kn < KS ? kn : KS - 1) * NT + (tile(t) < NT ? tile(t) : NT - 1)) * W;
#pragma unroll
        for (int i = 0; i < 2; ++i) ring[v % D][t][i] = wl[f + i];
      };
      // lo hi, hi hi, hi lo (weight, activation).  (An accumulator's next MFMA is eight cycles late if it follows at once: the
      // two sums take turns, and so do two tiles.  With three the L1's 64 bytes a cycle bound the layer, and loads in a row per
      // tile suit it better.)
      constexpr int WP[3] = {1, 0, 0}, AP[3] = {0, 0, 1};
      constexpr bool TURNS = TT == 2;
      if constexpr (v % (3 * KC) == 0) {
#pragma unroll
        for (int p = 0; p < PT; ++p)
#pragma unroll
          for (int t = 0; t < TT; ++t) sum[p][t] = f32x16{};
      }
#pragma unroll
      for (int o = 0; o < (TURNS ? 3 : TT); ++o)
#pragma unroll
        for (int n = 0; n < (TURNS ? TT : 3); ++n) {
          const int m = TURNS ? o : n, t = TURNS ? n : o;
#pragma unroll
          for (int p = 0; p < PT; ++p)
            if (team_used<PR>(p, t)) mma<PrecF32S>(ring[v % D][t][WP[m]], a[v % (AHEAD + 1)][p][AP[m]], m == 1 ? sum[p][t] : low[p][t]);
          if (m == 2) refill(t);
        }
      if constexpr ((v + 1) % (3 * KC) == 0) {
#pragma unroll
        for (int p = 0; p < PT; ++p)
#pragma unroll
          for (int t = 0; t < TT; ++t) {
            if (!team_used<PR>(p, t)) continue;
#pragma unroll
            for (int e = 0; e < 16; ++e) acc[p][t][e] = fmaf(sum[p][t][e], unit, acc[p][t][e]);
          }
      }
      __builtin_amdgcn_sched_barrier(0);
    });
  }
  // (or its products are put off until the sum is used, and their operands kept for that)
#pragma unroll
  for (int p = 0; p < PT; ++p)
#pragma unroll
    for (int t = 0; t < TT; ++t) {
      if (!team_used<PR>(p, t)) continue;
      asm volatile("" : "+a"(low[p][t]));
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[p][t][e] = fmaf(low[p][t][e], unit * (1.0f / kHalfLow), acc[p][t][e]);
    }
}

// SiLU of one accumulator tile into the record at `rec` (cout tile t).  most: the largest so far.
__device__ __forceinline__ void half_team_store(unsigned char *smem, int rec, int h, int t, const f32x16 &acc, float &most) {
  unsigned char *at = smem + rec + 64 * t + 8 * h;
  const v16i v = half_activations(acc, most);
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    *reinterpret_cast<v2i *>(at + 16 * q) = v2i{v[2 * q], v[2 * q + 1]};
    *reinterpret_cast<v2i *>(at + 192 + 16 * q) = v2i{v[8 + 2 * q], v[8 + 2 * q + 1]};
  }
}

// Board `b` by the team that this workgroup (its member my_role) belongs to, as team_board; next: the slot's flags of the second way, cleared
// here.  kHalfAgain, in the workgroup that ends the board (for the others it stands in word kTeamListed): a number on the way was beyond
// what two parts hold, and the board is to be done again.  kHalfUnheld, in every member and before any has raised a flag: two parts do not
// hold the weights.
enum HalfHow { kHalfDone, kHalfAgain, kHalfUnheld };
template <int TEAM>
__device__ __forceinline__ HalfHow half_team_board(const TeamParams &prm, unsigned char *smem, unsigned b, unsigned slot,
                                                int my_role, unsigned *next) {
  using P = PrecF32S;
  using G = Geo<P>;
  using T = TeamGeo<P>;
  using S = HalfTeamShape<TEAM>;
  constexpr int W = G::W, THREADS = 256, PXT = S::PXT, CG = S::CG;
  int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), h = lane >> 5;
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
  // what this wave knows of the numbers in role's squares up to layer l (half_note); a word per layer, so that whoever
  // goes on with another's squares finds it
  bool bad_input = false;
  HalfHow how = kHalfDone;
  unsigned trail = 0;
  auto note_at = [&](int l, int role) { return T::NOTE_OFF + ((l * 12 + role) * 4 + wave) * 4; };
  auto store_note = [&](int l, int role, float most, bool bad) __attribute__((always_inline)) {
    trail = (l > 0 ? trail : 0) | half_note(l, most) | (bad ? 1u : 0u);
    if (lane == 0) store4(__builtin_bit_cast(float, trail), note_at(l, role));
  };

  // the wave's first tile of squares within the workgroup's, and its group of cout tiles
  const int wpx = wave % S::PG * S::PT, cg = wave / S::PG;

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
  // `j` of each plane, so that all its addresses are two sums and constants.
  auto unit_of = [&](auto cc, int &sq, int &j) __attribute__((always_inline)) {
    constexpr int J = decltype(cc)::value / 8;
    int t = tid;   // (formed where it is used, not kept for all stages)
    asm volatile("" : "+v"(t));
    sq = t / J;
    j = t - sq * J;
  };
  constexpr int PARTS = T::NPL;
  auto part_mem = [](auto cc, int q, int k, int j) __attribute__((always_inline)) {
    constexpr int C = decltype(cc)::value;
    return (q * T::units(C) + k * (C / 8) + j) * 16;
  };
  auto part_lds = [](int k, int j) __attribute__((always_inline)) { return k * 192 + j * 16; };

  // Outputs of layer L (own squares): into the records, and to memory what the neighbours read.
  // acc: N tiles of squares, px(i) of the workgroup's, and a wave's cout tiles, tile(t) of the layer's
  auto write_out = [&](auto lc, auto nc, int role, const Span &sp, bool active, const auto &acc, auto px, auto tile) __attribute__((always_inline)) {
    constexpr int L = decltype(lc)::value, N = decltype(nc)::value, C = kCoutArr[L], NT = C / 32;
    constexpr int TT = S::tiles(NT);
    float most = 0.0f;
    if (active) {
#pragma unroll
      for (int i = 0; i < N; ++i) {
        const int p = sp.p0 + px(i) * 32 + (lane & 31), pc = p < kPix ? p : kPix - 1;
        const int rec = record(pc, sp.base);
#pragma unroll
        for (int t = 0; t < TT; ++t) {
          if constexpr (S::RAGGED && L > 0) {
            if (!team_used<S::PR>(i, t)) continue;
          }
          if (tile(t) < NT) half_team_store(smem, rec, h, tile(t), acc[i][t], most);
        }
      }
    }
    store_note(L, role, most, L == 0 && bad_input);
    __syncthreads();
    int sq, j;
    unit_of(IC<C>{}, sq, j);
    constexpr int PER = THREADS / (C / 8);   // squares at a time
    auto to_memory = [&](int q) __attribute__((always_inline)) {
      const unsigned char *from = smem + record(q, sp.base);
      v4i v[PARTS];
#pragma unroll
      for (int k = 0; k < PARTS; ++k)
        v[k] = *reinterpret_cast<const v4i *>(from + part_lds(k, j));
#pragma unroll
      for (int k = 0; k < PARTS; ++k)
        store16(v[k], T::act_off(L) + part_mem(IC<C>{}, q, k, j));
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
    constexpr int NT = kCoutArr[L] / 32, TT = S::tiles(NT), PT = S::squares(NT), D = half_team_ring<TT, PT>();
    constexpr int C = kCinArr[L];
    // (opaque per stage: what follows from it is formed here and not, for all stages, in front of the
    // loop over them, in several hundred scalar registers that get spilled)
    int t0 = S::RAGGED ? cg : cg * TT;
    asm volatile("" : "+s"(t0));
    const bool active = S::RAGGED ? NT > 1 || wave * PT < PXT : cg < CG && t0 < NT;
    // the wave's cout tiles (one beyond the layer's last repeats it, and is not used) and tiles of squares
    auto tile = [&](int t) __attribute__((always_inline)) {
      if constexpr (S::RAGGED) return NT == 3 ? (t == 0 ? 2 * t0 : 1) : (NT == 2 ? t0 : 0);
      else return t0 + t;
    };
    auto tile_or_last = [&](int t) __attribute__((always_inline)) { return tile(t) < NT ? tile(t) : NT - 1; };
    auto px = [&](int i) __attribute__((always_inline)) {
      if constexpr (!S::RAGGED) return wpx + i;
      else if constexpr (NT == 1) return wave * PT + i;
      else return wpx + (i < S::PR ? i : (t0 == 0 ? i - S::PR : 2 * S::PR - 1 - i));
    };
    const Span sp = span_of(role);
    const WFrags wl = layer_weights<P, L>(packed, lane);
    const float unit = __builtin_bit_cast(float, __builtin_amdgcn_readfirstlane(__builtin_bit_cast(int, tail[G::TAIL_SW + L])));
    C6_MARK(6 * L);
    const bool own = region_role == role && region_layer == L - 1;
    v4i ring[D][TT][2];
    f32x16 acc[PT][TT], low[PT][TT];
    auto first_weights = [&]() __attribute__((always_inline)) {
#pragma unroll
      for (int d = 0; d < D; ++d)
#pragma unroll
        for (int t = 0; t < TT; ++t)
#pragma unroll
          for (int i = 0; i < 2; ++i) ring[d][t][i] = wl[(d * NT + tile_or_last(t)) * W + i];
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
        v[k] = __builtin_amdgcn_raw_buffer_load_b128(mem, T::act_off(L - 1) + part_mem(IC<C>{}, q, k, j), 0, kSc1);
    };
    auto to_region = [&](int q, const v4i (&v)[PARTS]) __attribute__((always_inline)) {
      unsigned char *at = smem + record(q, sp.base);
#pragma unroll
      for (int k = 0; k < PARTS; ++k)
        *reinterpret_cast<v4i *>(at + part_lds(k, j)) = v[k];
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
    if (!own) trail = (unsigned)__builtin_amdgcn_raw_buffer_load_b32(mem, note_at(L - 1, role), 0, kSc1);
    if (active) {
#pragma unroll
      for (int t = 0; t < TT; ++t) {
        const int word = bias_offset(L) + 32 * tile_or_last(t);
#pragma unroll
        for (int i = 0; i < PT; ++i) {
          if (!team_used<S::PR>(i, t)) continue;
          acc[i][t] = tail_tile(word);
          low[i][t] = tail_tile(G::TAIL_BIAS_LOW + word);
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
      p[i] = sp.p0 + px(i) * 32 + (lane & 31);
      ok[i] = p[i] < kPix;
      rec[i] = record(ok[i] ? p[i] : kPix - 1, sp.base);
    }
    if (active) half_team_conv<L, TT, PT, S::PR>(smem, packed, wl, ring, lane, rec, tile, unit, acc, low);
    C6_MARK(6 * L + 3);
    if constexpr (L < 7) {
      __syncthreads();   // everybody has read this layer's input
      write_out(lc, IC<PT>{}, role, sp, active, acc, px, tile);
    } else {
      // heads: this wave's share of the policy (per square) and of the value
      float most = 0.0f;
      if (active) {
#pragma unroll
        for (int t = 0; t < TT; ++t) {
          if (tile(t) >= NT) continue;
          HalfHeads out;
          out.pw = tail_tile(kBiasTotal + 32 * tile(t));
          out.vw = tail_tile(kBiasTotal + kHeadC + 32 * tile(t));
#pragma unroll
          for (int i = 0; i < PT; ++i) {
            if (!team_used<S::PR>(i, t)) continue;
            out.pol = out.val = 0.0f;
            HalfEpi<true>::run(acc[i][t], out, most);
            const unsigned bits = __builtin_bit_cast(unsigned, out.pol);
            const auto x = __builtin_amdgcn_permlane32_swap(bits, bits, false, false);
            const unsigned x0 = x[0], x1 = x[1];
            const float tot = __builtin_bit_cast(float, x0) + __builtin_bit_cast(float, x1);
            const float vs = wave_sum(ok[i] ? out.val : 0.0f);
            if (h == 0 && ok[i]) store4(tot, T::HEAD_OFF + (tile(t) * 384 + p[i]) * 4);
            if (lane == 0) store4(vs, T::VAL_OFF + (tile(t) * 12 + role * PXT + px(i)) * 4);
          }
        }
      }
      store_note(L, role, most, false);
      raise_flag(L, role);
    }
    C6_MARK(6 * L + 4);
    return true;
  };

  // first layer: every workgroup stages the part of the board that its squares see
  auto first_stage = [&](int role) __attribute__((always_inline)) -> bool {
    const Span sp = span_of(role);
    int *flag = reinterpret_cast<int *>(red) + 64;   // [0]: third plane varies, [1]: an input is not exact, [3] beyond the range, [4] not small
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
    if (tid < 5 && tid != 2) flag[tid] = 0;
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
    if (tid < 2 * kTeamStages + 1)   // (role's words; acknowledged in front of this stage's flag)
      __hip_atomic_store(&next[tid < kTeamStages ? tid * 12 + role : (tid < 2 * kTeamStages ? kTeamAll + (tid - kTeamStages) * 12 : kTeamXcd) + role], 0u,
                         __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (tid == 0 && role == my_role)
      __hip_atomic_store(&flags[kTeamXcd + role], xcd_tag ^ xcd, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __syncthreads();
    // (the same in every member)
    float held = 1.0f;
#pragma unroll
    for (int l = 0; l < 8; ++l) held = tail[G::TAIL_SW + l] == 0.0f ? 0.0f : held;
    if (__builtin_amdgcn_ballot_w64(held == 0.0f) != 0) {
      how = kHalfUnheld;
      return true;
    }
    const bool plane2_varies = flag[0] != 0;
    bool inexact = false, beyond = false, ordinary = false;   // (as half_forward_kernel)
#pragma unroll
    for (int k = 0; k < 2; ++k)
      if (tid + k * THREADS < kPix)
#pragma unroll
        for (int ch = 0; ch < 3; ++ch) {
          if (ch == 2 && !plane2_varies) continue;
          inexact |= xin[k][ch] - half_value(half_bits(xin[k][ch])) != 0.0f;
          beyond |= !half_fits(xin[k][ch]);
          ordinary |= __builtin_fabsf(xin[k][ch]) >= kHalfLeast;
        }
    if (inexact) flag[1] = 1;
    if (beyond) flag[3] = 1;
    if (ordinary) flag[4] = 1;
    __syncthreads();
    const int parts = flag[1] != 0 ? 2 : 1;
    bad_input = parts > 1 && (flag[3] != 0 || flag[4] == 0);
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
    const float unit = tail[G::TAIL_SW], factor = half_inverse(unit);
    if (active) {
      const f32x16 b0 = tail_tile(bias_offset(0));
#pragma unroll
      for (int n = 0; n < N1; ++n)
#pragma unroll
        for (int i = 0; i < 16; ++i) acc[n][0][i] = factor * (plane2_varies ? b0[i] : fmaf(c2, acc[n][0][i], b0[i]));
    }
    f32x16 low[N1], large[N1];   // small products; the large ones, once a second part follows
    if (active) {
#pragma unroll
      for (int n = 0; n < N1; ++n) low[n] = tail_tile(G::TAIL_BIAS_LOW + bias_offset(0));
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
          const unsigned short v16 = half_bits(xin[k][ch]);
          xin[k][ch] = (xin[k][ch] - half_value(v16)) * kHalfLow;
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
        // the matrix core waits for.
        constexpr int DW = N1 > 1 ? 2 : 4;
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
              for (int n = 0; n < N1; ++n) mma<P>(w[s8][i][j], a[s8 % 2][i][n], j > 0 ? low[n] : acc[n][0]);
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
        if (parts > 1) {   // (the second part's products with the weights' first are small ones, the others are dropped)
#pragma unroll
          for (int n = 0; n < N1; ++n)
#pragma unroll
            for (int i = 0; i < 16; ++i) {
              if (part == 0) {
                large[n][i] = acc[n][0][i];
                acc[n][0][i] = low[n][i];
              } else {
                low[n][i] = acc[n][0][i];
                acc[n][0][i] = large[n][i];
              }
            }
        }
      }
    }
#pragma unroll
    for (int n = 0; n < N1; ++n)
#pragma unroll
      for (int i = 0; i < 16; ++i) acc[n][0][i] = fmaf(low[n][i], unit * (1.0f / kHalfLow), acc[n][0][i] * unit);
    C6_MARK(2);
    __syncthreads();   // the copies give way to the activations
    clear_region(sp);
    write_out(IC<0>{}, IC<N1>{}, role, sp, active, acc, [&](int i) { return px + i; }, [](int t) { return t; });
    C6_MARK(3);
    return true;
  };

  // the heads' sums into logits, value and draw: one workgroup
  auto last_stage = [&](int role) __attribute__((always_inline)) -> bool {
    const int got = wait_inputs(8, role, true);
    if (got != 1) return got == 2;
    region_role = -1;
    const float *valw = tail + kBiasTotal + kHeadC;
    const float polb = valw[kHeadC], valb = valw[kHeadC + 1];
    auto partial = [&](int at) __attribute__((always_inline)) {
      return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(mem, at, 0, kSc1));
    };
    // Everything that is read here is asked for at once, and the value's sum runs beside the logits; a board's squares are
    // known to be in range from the last layer's words alone (store_note).  (Words of all layers, then logits, then the value's
    // 36 sums one after the other in one lane: 21 boards 59.1 -> 56.8 us, 42 boards 79 -> 77 us, one board 48.7 -> 47.8 us.)
    static_assert(TEAM * 4 <= 64, "a wave reads the words");
    float head[2][3], val = 0.0f;
    int note = 0;
#pragma unroll
    for (int k = 0; k < 2; ++k)
#pragma unroll
      for (int t = 0; t < 3; ++t) head[k][t] = partial(T::HEAD_OFF + (t * 384 + (tid + k * THREADS) % 384) * 4);   // (beyond 360: unused)
    if (wave == 3) val = lane < 36 ? partial(T::VAL_OFF + lane * 4) : 0.0f;
    else if (wave == 0 && lane < TEAM * 4) note = __builtin_bit_cast(int, partial(T::NOTE_OFF + (7 * 48 + lane) * 4));
    __builtin_amdgcn_sched_barrier(0);
    if (wave == 0) {   // the verdict, as early as it is known
      const bool again = half_failed((unsigned)wave_allreduce_bits(note, [](int a, int b) { return a | b; }));
      if (again && lane == 0) store_flag(kTeamListed);
      if (again) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      if (lane == 0) {
        store_flag(8 * 12 + role);
        *word = again ? 1 : 0;
      }
    }
    if (wave == 3 && f.value != nullptr) {   // (the sum needs its lanes together)
      const double sum = split_value_sum(lane, [&](int) { return val; });
      if (lane == 0) f.value[b] = split_value(sum, valb);
    }
    const bool state = f.x_dtype == C6_DT_BOARD_I8;
    long long src = state && f.index ? f.index[b] : (long long)b;
    if (state) src = src < 0 ? 0 : (src >= f.num_states ? f.num_states - 1 : src);
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      const int sq = tid + k * THREADS;
      if (sq >= kPix) continue;
      const float z = split_logit((head[k][0] + head[k][1]) + head[k][2], polb);
      bool taken;
      if (f.mask_mode == C6_MASK_LEGAL) {
        taken = f.legal[(size_t)b * kPix + sq] == 0;
      } else if (state) {
        const int stone = reinterpret_cast<const int8_t *>(f.x)[(size_t)src * kPix + (f.view ? d4_from_view(sq, f.view) : sq)];
        const int me = f.player[src];
        taken = stone == me || stone == -me;
      } else {
        taken = load_input(f.x, f.x_dtype, (size_t)b * 3 * kPix + sq) != 0.0f || load_input(f.x, f.x_dtype, ((size_t)b * 3 + 1) * kPix + sq) != 0.0f;
      }
      const bool masked = taken && f.mask_mode != C6_MASK_NONE;
      lgt[sq] = z;
      occ[sq] = masked ? 1 : 0;
      if (f.logits != nullptr) static_cast<float *>(f.logits)[(size_t)b * kPix + sq] = masked ? f.fill : z;
    }
    __syncthreads();
    if (__builtin_amdgcn_readfirstlane(*word) != 0) how = kHalfAgain;
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
    // (opaque: what follows from them is formed in each stage, and not kept for all of them)
    asm volatile("" : "+v"(tid));
    lane = tid & 63;
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
    if (how == kHalfUnheld) break;
    if (ok && stage == l && role == my_role) ++l;
    help = !ok;
  }
  __syncthreads();
  return how;
}

// A workgroup's share of board b, in a team of any size.
__device__ __forceinline__ HalfHow half_team_share(const TeamParams &prm, unsigned char *smem, unsigned b, TeamPlace at, int team, unsigned *next) {
  if (team == 12) return half_team_board<12>(prm, smem, b, at.slot, at.role, next);
  if (team == 6) return half_team_board<6>(prm, smem, b, at.slot, at.role, next);
  if (team == 3) return half_team_board<3>(prm, smem, b, at.slot, at.role, next);
  if (team == 2) return half_team_board<2>(prm, smem, b, at.slot, at.role, next);
  return kHalfDone;
}

// A board that two parts do not hold is done again by its team with three: one board 110 us, 53 boards 196, 128 boards 356 (by the workgroup
// that ends it, alone, 314, 347 and 380); a set of weights that they do not hold, at once: 62, 120, 224.  The members wait for the last stage's verdict, which is given as soon as that stage's loads have
// arrived, so that they end with the workgroup that gives it: boards in range take what they took (given behind the outputs one board 45.2 ->
// 45.7 us, 85 boards 98.5 -> 99.6 us).  The second way has exchange memory and flags of its own, behind the first one's: a member that comes late may
// still be at its part of the first.
template <class P> __device__ __forceinline__ void half_team(const TeamParams &prm, unsigned char *smem, unsigned items, TeamPlace at, int team) {
  TeamParams exact = prm;
  exact.f.packed += kSplitOffset;
  exact.act += (size_t)items * TeamGeo<P>::BOARDB;
  exact.flags = reinterpret_cast<unsigned *>(exact.act + (size_t)items * TeamGeo<PrecF32X>::BOARDB);
  const unsigned b = prm.first + at.slot;
  const HalfHow how = half_team_share(prm, smem, b, at, team, exact.flags + (size_t)at.slot * kTeamFlags);
  bool again = how != kHalfDone;
  if (how == kHalfUnheld) {
    exact.flags = prm.flags;   // (nobody has raised one of them; the others' words may not be clear yet)
  } else if (at.role != 0) {
    const unsigned *flags = prm.flags + (size_t)at.slot * kTeamFlags;
    auto is_set = [&](int w) { return __hip_atomic_load(&flags[w], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == prm.tag; };
    int *verdict = reinterpret_cast<int *>(smem);
    if (threadIdx.x < 64) {
      // (bounded as every wait; a team without a member that left here finishes by itself)
      int found = -1;
      for (int k = 0; k < prm.polls && found < 0; ++k)
        if (is_set(8 * 12)) found = is_set(kTeamListed) ? 1 : 0;
      if (threadIdx.x == 0) *verdict = found;
    }
    __syncthreads();
    again = __builtin_amdgcn_readfirstlane(*verdict) == 1;
  }
  if (!again) return;
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // (behind the other stores of the outputs)
  __syncthreads();
  team_share<PrecF32X>(exact, smem, b, at, team);
}

}  // namespace c6
