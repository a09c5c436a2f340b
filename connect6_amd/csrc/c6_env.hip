// Batched Connect6 rules on device state for gfx950: one environment step (stone placement,
// local win check, turn bookkeeping) and the canonical network input.  Replaces
// VectorConnect6.step / _check_win_local (connect6/vector_env.py:106-193 of the reference) and
// canonical_network_input (connect6/vector_env.py:196-218), each a chain of a dozen small
// PyTorch launches there.  Both kernels are latency / HBM bound: an environment reads at most
// 8 * (win_length - 1) board bytes and a few state bytes and writes one stone and 9 result bytes.
#include "c6_common.h"
#include "c6_device.h"

namespace c6 {

// Eight lanes per game, one for each direction out of the new stone.  A game reads a handful of
// scattered board bytes, so the step is a chain of memory latencies and nothing else: action and
// state, then the neighbours, then the results.  A lane asks for up to eight neighbours of its
// direction at once (five for six in a row) and counts the run of equal stones from the front; the
// two halves of a line meet in one exchange between lanes.  16,384 games: 11.3 us with one thread per
// game walking outward square by square on a quarter of the CUs, 5 us this way.
constexpr int kStepLanes = 8, kStepAhead = 8;
__global__ __launch_bounds__(256) void env_step_kernel(const EnvParams p) {
  const long long i = ((long long)blockIdx.x * blockDim.x + threadIdx.x) / kStepLanes;
  const int d = threadIdx.x % kStepLanes;
  if (i >= p.num) return;   // (whole groups of eight lanes)
  const int n = p.n, cells = n * n;
  long long a = p.actions[i];
  const int8_t actor = p.player[i];
  const int16_t empty = (int16_t)(p.empty_count[i] - 1);
  const int16_t moves = (int16_t)(p.move_count[i] + 1);
  const int8_t left = p.stones_left[i];
  a = a < 0 ? 0 : (a >= cells ? cells - 1 : a);  // never write outside the board
  if (p.view) a = d4_from_view((int)a, p.view, n);  // policy-view square -> board square
  const int row = (int)a / n, col = (int)a - row * n;
  int8_t *board = p.boards + i * cells;

  // lanes d and d + 4 look the two ways along line d: row, column, both diagonals
  const int line = d & 3, s = d < 4 ? 1 : -1;
  const int dr = (line == 0 ? 0 : 1) * s, dc = (line == 1 ? 0 : (line == 3 ? -1 : 1)) * s;
  const int reach = p.win - 1;   // squares each way that can matter
  int run = 0;
  for (int k0 = 0; k0 < reach && run == k0; k0 += kStepAhead) {
    int8_t stone[kStepAhead];
#pragma unroll
    for (int k = 0; k < kStepAhead; ++k) {
      const int r = row + (k0 + k + 1) * dr, c = col + (k0 + k + 1) * dc;
      const bool in = k0 + k < reach && r >= 0 && r < n && c >= 0 && c < n;
      stone[k] = in ? board[r * n + c] : (int8_t)~actor;   // (never equal to actor)
    }
    unsigned other = 1u << kStepAhead;
#pragma unroll
    for (int k = 0; k < kStepAhead; ++k) other |= stone[k] != actor ? 1u << k : 0u;
    run += __builtin_ctz(other);
  }
  const int total = 1 + run + __shfl_xor(run, 4);
  int won = total >= p.win ? 1 : 0;
  won |= __shfl_xor(won, 1);
  won |= __shfl_xor(won, 2);
  if (d != 0) return;
  board[row * n + col] = actor;
  p.empty_count[i] = empty;
  p.move_count[i] = moves;
  const bool done = won || empty == 0;
  p.reward[i] = won ? 1.0f : 0.0f;
  p.done[i] = done ? 1 : 0;
  p.winner[i] = won ? actor : (int8_t)0;
  p.lengths[i] = moves;
  int8_t sign = 0;
  if (!done) {  // a finished game keeps its side to move and its stones_left
    const int8_t remaining = (int8_t)(left - 1);
    if (remaining > 0) {
      p.stones_left[i] = remaining;
      sign = 1;
    } else {
      p.player[i] = (int8_t)-actor;
      p.stones_left[i] = 2;
      sign = -1;
    }
  }
  p.sign[i] = sign;
}

// Plane 0 = stone of the side to move, 1 = of the other side, 2 = this decision is the last
// stone of the turn.  Eight games per workgroup: their int8 boards are staged in LDS with
// coalesced loads, then the 8 x 3 x cells output floats (a whole number of 16-byte units,
// contiguous in memory) are written with 16-byte stores.
// (The 19 x 19 board has canonical_board_kernel.)
constexpr int kCanonGames = 8;
__global__ __launch_bounds__(256) void canonical_input_kernel(const int8_t *__restrict__ boards,
                                                              const int8_t *__restrict__ player,
                                                              const int8_t *__restrict__ stones_left,
                                                              long long num, int cells,
                                                              float *__restrict__ out) {
  extern __shared__ __attribute__((aligned(16))) int8_t s_board[];  // kCanonGames * cells, + 8 so that word reads may run past the end
  __shared__ int s_me[kCanonGames];
  __shared__ float s_last[kCanonGames];
  const long long g0 = (long long)blockIdx.x * kCanonGames;
  const int ng = (int)(num - g0 < kCanonGames ? num - g0 : kCanonGames);
  const int8_t *src = boards + g0 * cells;
  if (ng == kCanonGames && (reinterpret_cast<uintptr_t>(src) & 7u) == 0) {
    // eight boards = 8 * cells bytes: a whole number of 8-byte units
    for (int i = threadIdx.x; i < cells; i += blockDim.x)
      reinterpret_cast<v2i *>(s_board)[i] = reinterpret_cast<const v2i *>(src)[i];
  } else {
    for (int i = threadIdx.x; i < ng * cells; i += blockDim.x) s_board[i] = src[i];
  }
  if ((int)threadIdx.x < ng) {
    s_me[threadIdx.x] = player[g0 + threadIdx.x];
    s_last[threadIdx.x] = stones_left[g0 + threadIdx.x] == 1 ? 1.0f : 0.0f;
  }
  __syncthreads();
  const int per_game = 3 * cells;
  const int total = ng * per_game;
  float *dst = out + g0 * per_game;
  auto value = [&](int o) {
    const int g = o / per_game, rem = o - g * per_game;
    const int plane = rem / cells, cell = rem - plane * cells;
    const int stone = s_board[g * cells + cell], me = s_me[g];
    return plane == 2 ? s_last[g] : ((plane == 0 ? stone == me : stone == -me) ? 1.0f : 0.0f);
  };
  if ((total & 3) == 0 && (reinterpret_cast<uintptr_t>(dst) & 15u) == 0) {
    const unsigned *words = reinterpret_cast<const unsigned *>(s_board);
    // (game, offset inside the game) of the thread's first output, then stepped by 4 * blockDim
    // per iteration: no division in the loop
    int g = (4 * (int)threadIdx.x) / per_game, rem = 4 * (int)threadIdx.x - g * per_game;
    const int step = 4 * (int)blockDim.x, step_g = step / per_game, step_rem = step - step_g * per_game;
    for (int q = threadIdx.x; q < total / 4; q += blockDim.x, g += step_g, rem += step_rem) {
      if (rem >= per_game) {
        rem -= per_game;
        ++g;
      }
      int plane = rem >= 2 * cells ? 2 : (rem >= cells ? 1 : 0);
      int cell = rem - plane * cells;
      const int g_first = g;
      f32x4 o;
      if (cell + 3 < cells) {
        // the four squares sit in one plane: fetch their bytes as one (unaligned) word and
        // compare all four with the wanted stone at once
        if (plane == 2) {
          const float l = s_last[g];
          o = f32x4{l, l, l, l};
        } else {
          const int a = g * cells + cell;
          const unsigned w = __builtin_amdgcn_alignbyte(words[(a >> 2) + 1], words[a >> 2], a & 3);
          const int me = s_me[g];
          const unsigned want = (unsigned)((plane == 0 ? me : -me) & 0xff) * 0x01010101u;
          const unsigned x = w ^ want;  // a zero byte = the wanted stone
#pragma unroll
          for (int e = 0; e < 4; ++e) o[e] = ((x >> (8 * e)) & 0xffu) == 0 ? 1.0f : 0.0f;
        }
      } else {
        int gg = g_first;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int stone = s_board[gg * cells + cell], me = s_me[gg];
          o[e] = plane == 2 ? s_last[gg] : ((plane == 0 ? stone == me : stone == -me) ? 1.0f : 0.0f);
          if (++cell == cells) {
            cell = 0;
            if (++plane == 3) {
              plane = 0;
              gg = gg + 1 < ng ? gg + 1 : gg;
            }
          }
        }
      }
      reinterpret_cast<f32x4 *>(dst)[q] = o;
    }
  } else {
    for (int o = threadIdx.x; o < total; o += blockDim.x) dst[o] = value(o);
  }
}

// The same on the 19 x 19 board: a thread writes QUADS times four consecutive floats, 256 apart, from the four bytes
// they come from and, where they reach into the next plane or game, its first four.  No LDS and no barrier: as many
// workgroups as fit the chip used to read all at once and then write all at once, each behind its loads' latency.
// (1,024 / 4,096 / 16,384 / 65,536 games 6.9 / 8.7 / 15.3 / 68 us, so with two quads 3.2 / 6.2 / 14.0 / 76, with four
// 3.7 / 6.7 / 13.8 / 62; a plain fill of the outputs 2.5 / 4.8 / 11.9 / 41.  Groups of games through LDS with the next
// one's bytes ahead: 5.0 / 7.7 / 16.5 / 78.)
template <int QUADS>
__global__ __launch_bounds__(256) void canonical_board_kernel(const int8_t *__restrict__ boards,
                                                              const int8_t *__restrict__ player,
                                                              const int8_t *__restrict__ stones_left, unsigned num,
                                                              float *__restrict__ out) {
  constexpr unsigned GAME = 3 * kPix;
  const unsigned total = num * GAME, quads = total / 4;   // (below 2^32, see launch_canonical_input)
  const unsigned q0 = blockIdx.x * (256 * QUADS) + threadIdx.x;
  int cell[QUADS], plane[QUADS], me[QUADS], next_me[QUADS], left[QUADS];
  unsigned here[QUADS], next[QUADS];   // four squares of the plane the quad starts in, the first of the one behind it
#pragma unroll
  for (int k = 0; k < QUADS; ++k) {
    const unsigned q = q0 + 256 * k < quads ? q0 + 256 * k : quads - 1;
    const unsigned game = q * 4 / GAME;
    const int rem = (int)(q * 4 - game * GAME);
    plane[k] = rem >= 2 * kPix ? 2 : (rem >= kPix ? 1 : 0);
    cell[k] = rem - plane[k] * kPix;
    const unsigned behind = plane[k] == 2 && game + 1 < num ? game + 1 : game;
    me[k] = player[game];
    next_me[k] = player[behind];
    left[k] = stones_left[game];
    const int at = cell[k] + 3 < kPix ? cell[k] : kPix - 4;   // (not beyond the board)
    __builtin_memcpy(&here[k], boards + (size_t)game * kPix + at, 4);
    here[k] >>= 8 * (cell[k] - at);
    next[k] = 0;
    if (cell[k] + 3 >= kPix) __builtin_memcpy(&next[k], boards + (size_t)behind * kPix, 4);
  }
#pragma unroll
  for (int k = 0; k < QUADS; ++k) {
    const unsigned q = q0 + 256 * k;
    if (q >= quads) break;
    const float last = left[k] == 1 ? 1.0f : 0.0f;
    const unsigned want = (plane[k] == 0 ? me[k] : -me[k]) & 0xff, want_next = (plane[k] == 0 ? -me[k] : next_me[k]) & 0xff;
    f32x4 o;
#pragma unroll
    for (int e = 0; e < 4; ++e) o[e] = plane[k] == 2 ? last : ((here[k] >> (8 * e) & 0xff) == want ? 1.0f : 0.0f);
    if (cell[k] + 3 >= kPix) {
      const int n = kPix - cell[k];   // squares left in the plane, 1 to 3
#pragma unroll
      for (int e = 1; e < 4; ++e)
        if (e >= n) o[e] = plane[k] == 1 ? last : ((next[k] >> (8 * (e - n)) & 0xff) == want_next ? 1.0f : 0.0f);
    }
    reinterpret_cast<f32x4 *>(out)[q] = o;
  }
  // (up to three floats behind the last quad: the last game's third plane)
  if (blockIdx.x == 0 && threadIdx.x < (total & 3u)) out[quads * 4 + threadIdx.x] = stones_left[num - 1] == 1 ? 1.0f : 0.0f;
}

int launch_env_step(const EnvParams &p, hipStream_t st) {
  if (p.num == 0) return C6_OK;
  const long long blocks = (p.num * kStepLanes + 255) / 256;
  if (blocks > 0x7fffffffLL) {
    set_error("c6_env_step: %lld games exceed one launch", p.num);
    return C6_EINVAL;
  }
  hipLaunchKernelGGL(env_step_kernel, dim3((unsigned)blocks), dim3(256), 0, st, p);
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) {
    set_error("env_step_kernel launch failed: %s", hipGetErrorString(e));
    return C6_ELAUNCH;
  }
  return C6_OK;
}

int launch_canonical_input(const int8_t *boards, const int8_t *player, const int8_t *stones_left,
                           long long num, int n, float *out, hipStream_t st) {
  if (num == 0) return C6_OK;
  const int cells = n * n;
  const long long blocks = (num + kCanonGames - 1) / kCanonGames;
  if (n == kBoard && num <= 0xf0000000u / (3 * kPix) && (reinterpret_cast<uintptr_t>(out) & 15u) == 0) {
    const unsigned quads = (unsigned)num * (3 * kPix) / 4;
    if (num < 8192)
      hipLaunchKernelGGL(canonical_board_kernel<2>, dim3((quads + 511) / 512), dim3(256), 0, st, boards, player, stones_left, (unsigned)num, out);
    else
      hipLaunchKernelGGL(canonical_board_kernel<4>, dim3((quads + 1023) / 1024), dim3(256), 0, st, boards, player, stones_left, (unsigned)num, out);
  } else {
    hipLaunchKernelGGL(canonical_input_kernel, dim3((unsigned)blocks), dim3(256),
                       (size_t)kCanonGames * cells + 8, st, boards, player, stones_left, num, cells, out);
  }
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) {
    set_error("canonical_input_kernel launch failed: %s", hipGetErrorString(e));
    return C6_ELAUNCH;
  }
  return C6_OK;
}

}  // namespace c6
