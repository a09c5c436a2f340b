// Whole forward of a small network in ONE launch, for architectures other than the default one
// (connect6/model.py:26-77 of the reference accepts any): every layer an implicit GEMM on the
// matrix cores, activations in LDS from the input planes to the heads.
//
// Replaces one launch of a direct convolution per layer (one thread per output, weights and
// activations re-read from memory for every tap), which ran the 9x9 network with kernels
// [5, 3, 3] and channels [16, 32, 32] on 1024 boards in 913 us; what bounds this kernel is noted at
// small_net_kernel.
//
// fp32 arithmetic on the bf16 matrix cores: every fp32 operand is the exact sum of three bf16
// values (8 + 8 + 8 mantissa bits: hi = bf16(v), mid = bf16(v - hi), lo = v - hi - mid), so a
// product of two is nine products of bf16 values, each exact in fp32.  The six down to 2^-17 of the
// largest are accumulated in fp32; the other three are below 2^-25 of it, under the rounding of one
// fp32 addition.  The five small ones have a sum of their own, which the matrix instruction would
// otherwise cut off towards minus infinity (c6_split.h): over seven architectures the error against a 64-bit
// forward is 0.3 to 0.7 of that of a chain of fp32 multiply-adds in the logits, 0.5 to 1 in the value (with one
// sum up to 1.4, and 2.6 in its mean over a network's boards).  Six bf16 instructions take 3/8 of the time of the fp32 ones (2.5 PFLOP/s / 6
// against 157 TFLOP/s), and the planes need 6 bytes of LDS per value.
#include "c6_common.h"
#include "c6_device.h"

namespace c6 {

constexpr int kSmallMaxLayers = 16;
constexpr int kSmallMaxTiles = 3;      // cout tiles of 16 a wave carries: up to 48 channels
constexpr int kSmallMaxWaves = 8;
constexpr int kSmallTableEntries = 8192;
constexpr int kSmallLds = 160 * 1024;

constexpr int kPlanes = 3;             // of an input board

struct SmallLayer {
  int k, r;              // kernel size and its padding k / 2
  int cin, cb;           // input channels and their blocks of eight
  int cout, tiles;       // output channels and their tiles of sixteen
  int blocks, chunks;    // (tap, channel block) pairs and their groups of four = MFMAs of K 32
  int frag0, bias0;      // first weight fragment; first bias in the tail
  int pitch;             // LDS positions per row of this layer's input: n + r
  unsigned pitch_magic, k_magic, cb_magic;  // ceil(2^32 / d), for the small quotients here
  int positions;         // of one board
  int pixb, planeb;      // bytes of one position, of one precision plane of it
  int boardb;            // bytes of one board
  int table0;            // first entry of the layer's offset table
};

struct SmallParams {
  const void *x;
  int x_dtype;
  long long per_group;
  int wgs_per_group;
  const unsigned char *packed;
  size_t packed_stride, tail;
  int n, nn, layers, nb;       // nb: boards per workgroup
  unsigned n_magic, nn_magic;
  int table_off, pix_off, val_off, tail_off;  // LDS: offset tables, squares, value sums, the packed tail
  int tail_floats;             // of the copy in LDS (0: none)
  int bias_total;
  float *logits, *value;
  int mask_mode;
  const uint8_t *legal;
  float fill;
  SmallLayer layer[kSmallMaxLayers];
  // the parameters as the module holds them (each tensor [groups, ...]), where there is no packed copy
  const float *conv_w[kSmallMaxLayers], *conv_b[kSmallMaxLayers];
  const float *pol_w, *pol_b, *val_w, *val_b;
};

// arithmetic of a mode: bf16 planes of an activation and of a weight, or fp16 operands
template <int NA_, int NW_, bool F16_> struct SmallArith {
  static constexpr int NA = NA_, NW = NW_;
  static constexpr bool F16 = F16_;
};

// ANY: a parameter or an input, which may be infinite or beyond the largest bf16 value
template <class A, bool ANY = false> __device__ __forceinline__ void small_planes(float v, unsigned short (&p)[A::NA]) {
  if constexpr (A::F16) {
    p[0] = __builtin_bit_cast(unsigned short, (_Float16)v);
  } else {
#pragma unroll
    for (int i = 0; i < A::NA; ++i) {
      if constexpr (ANY && A::NA > 1) {
        p[i] = bf16_part(v);
        v = bf16_rest(v, p[i]);
      } else {
        p[i] = __builtin_bit_cast(unsigned short, (__bf16)v);
        v -= __builtin_bit_cast(float, (unsigned)p[i] << 16);
      }
    }
  }
}

__device__ __forceinline__ int small_div(int p, unsigned magic) { return magic == 0 ? p : (int)__umulhi((unsigned)p, magic); }

// Where nothing is rounded to 16 bits, all activations carry the factor -log2(e) / 2, so that SiLU is u / (1 + 2^(2 u));
// it is put in with the first layer's weights and all biases, in 64 bits, and taken out behind the heads.  (The half:
// a factor below 1 leaves fp32 its whole range.)
template <class A> constexpr bool small_scaled() { return A::NA == 3 && A::NW == 3; }
constexpr double kSmallScale = -0.72134752044448170368;
template <class A> __device__ __forceinline__ double small_scale(double v, bool scaled) {
  return small_scaled<A>() && scaled ? v * kSmallScale : v;
}
// a parameter's planes, of its value in 64 bits
template <class A> __device__ __forceinline__ void small_weight_planes64(double v, unsigned short (&p)[A::NW]) {
  if constexpr (small_scaled<A>()) {
#pragma unroll
    for (int i = 0; i < A::NW; ++i) {
      p[i] = bf16_part((float)v);
      v = (p[i] & 0x7f80) == 0x7f80 ? 0.0 : v - (double)__builtin_bit_cast(float, (unsigned)p[i] << 16);
    }
  } else {
    small_planes<SmallArith<A::NW, A::NW, A::F16>, true>((float)v, p);
  }
}
// Two values' next planes in one dword; the values keep what it leaves out.
__device__ __forceinline__ int small_take(float &a, float &b, bool more) {
#pragma clang fp contract(off)
  typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
  const int w = __builtin_bit_cast(int, bf16x2{(__bf16)a, (__bf16)b});
  if (more) {
    a -= __builtin_bit_cast(float, w << 16);
    b -= __builtin_bit_cast(float, w & (int)0xffff0000);
  }
  return w;
}

template <class A> __device__ __forceinline__ f32x4 small_mma(const v4i &w, const v4i &a, const f32x4 &c) {
  if constexpr (A::F16) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, w), __builtin_bit_cast(f16x8, a), c, 0, 0, 0);
  } else {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, w), __builtin_bit_cast(bf16x8, a), c, 0, 0, 0);
  }
}

__device__ __forceinline__ float small_load(const void *x, int dt, size_t i) { return load_input(x, dt, i); }

// Where a wave's weight fragments come from: the packed copy (fragment ((chunk * tiles + tile) *
// planes + plane), see small_pack_kernel) ...
template <class A> struct PackedWeights {
  static constexpr bool kPacked = true;
  const unsigned char *p;
  template <int CT> __device__ __forceinline__ void fetch(int c, v4i (&w)[CT][A::NW]) const {
#pragma unroll
    for (int t = 0; t < CT; ++t)
#pragma unroll
      for (int i = 0; i < A::NW; ++i)
        w[t][i] = *reinterpret_cast<const v4i *>(p + (size_t)((c * CT + t) * A::NW + i) * 1024);
  }
};
// ... or the tensors themselves, for a caller that hands over weights with every call: eight
// gathered loads and the conversion per fragment, the same values.
template <class A, bool FIRST> struct RawWeights {   // FIRST: the first layer's, which are scaled
  static constexpr bool kPacked = false;
  const float *w;  // [cout, cin, k, k] of the weight set
  int cin, cout, kk, cb, cb_magic, blocks, lane;
  template <int CT> __device__ __forceinline__ void fetch(int c, v4i (&out)[CT][A::NW]) const {
    int ln = lane;   // (what follows from it is formed here: registers)
    asm volatile("" : "+v"(ln));
    const int e = 4 * c + (ln >> 4), tap = (e * cb_magic) >> 16, ci0 = 8 * (e - tap * cb);
#pragma unroll
    for (int t = 0; t < CT; ++t) {
      const int co = 16 * t + (ln & 15);
      const bool row = e < blocks && co < cout;
      unsigned short pl[8][A::NW] = {};
#pragma unroll
      for (int i = 0; i < (FIRST ? kPlanes : 8); ++i) {   // (the first layer's other channels are padding)
        const bool in = row && ci0 + i < cin;
        const float v = w[in ? (size_t)(co * cin + ci0 + i) * kk + tap : 0];
        if constexpr (small_scaled<A>() && FIRST) small_weight_planes64<A>(small_scale<A>(in ? v : 0.0f, true), pl[i]);
        else small_planes<SmallArith<A::NW, A::NW, A::F16>, true>(in ? v : 0.0f, pl[i]);
      }
#pragma unroll
      for (int p = 0; p < A::NW; ++p)
#pragma unroll
        for (int d = 0; d < 4; ++d) out[t][p][d] = pl[2 * d][p] | (int)pl[2 * d + 1][p] << 16;
    }
  }
};

// the tail's second part: the biases' low parts
constexpr int small_low(int bias_total) { return bias_total + 2 * 16 * kSmallMaxTiles + 4; }
__device__ __forceinline__ float small_rest(double v, float rounded) {
  return __builtin_fabsf(rounded) < __builtin_inff() ? (float)(v - (double)rounded) : 0.0f;
}

// One layer's contraction for the wave's PT tiles of 16 squares and its CT tiles of 16 channels.
// Operands of the next chunk are fetched while the current one's MFMAs run.
//   NA: planes of its activations that are not zero
template <class A, int NA, int PT, int CT, class Weights>
__device__ __forceinline__ void small_contract(const unsigned char *smem, const unsigned short *table,
                                               const Weights &weights, const SmallLayer &L, int lane,
                                               const int (&base)[PT], f32x4 (&acc)[PT][CT], f32x4 (&low)[PT][CT]) {
  constexpr int NW = A::NW;
  const int q = lane >> 4;
  const unsigned short *tab = table + L.table0 + q;
  const int planeb = L.planeb, chunks = L.chunks;
  v4i w[2][CT][NW], a[2][PT][NA];
  // (a chunk's offset is read a chunk ahead of its operands: no wave waits for one)
  int next = (int)tab[0] * 16;
  auto fetch = [&](int c, int s) __attribute__((always_inline)) {
    weights.template fetch<CT>(c, w[s]);
    const int off = Weights::kPacked ? next : (int)tab[4 * c] * 16;
    if constexpr (Weights::kPacked) next = (int)tab[4 * (c + 1 < chunks ? c + 1 : c)] * 16;
#pragma unroll
    for (int j = 0; j < PT; ++j)
#pragma unroll
      for (int i = 0; i < NA; ++i) a[s][j][i] = *reinterpret_cast<const v4i *>(smem + base[j] + off + i * planeb);
  };
  // Operands in several planes: the small products have a sum of their own (the instruction drops what lies
  // some eight bits below the last of its sum, towards minus infinity; see c6_split.h)
#pragma unroll
  for (int j = 0; j < PT; ++j)
#pragma unroll
    for (int t = 0; t < CT; ++t) low[j][t] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  auto multiply = [&](int s) __attribute__((always_inline)) {
    // smallest products first
#pragma unroll
    for (int d = (A::NA < NW ? A::NA : NW) == 3 ? 2 : A::NA - 1; d >= 0; --d)
#pragma unroll
      for (int i = 0; i <= d; ++i) {  // activation plane d - i, weight plane i
        if (d - i >= NA || i >= NW) continue;
#pragma unroll
        for (int t = 0; t < CT; ++t)
#pragma unroll
          for (int j = 0; j < PT; ++j) {
            f32x4 &sum = d > 0 ? low[j][t] : acc[j][t];
            sum = small_mma<A>(w[s][t][i], a[s][j][d - i], sum);
          }
      }
  };
  fetch(0, 0);
  int c = 0;
#pragma unroll 1
  for (; c + 2 <= chunks; c += 2) {
    fetch(c + 1, 1);
    multiply(0);
    fetch(c + 2 < chunks ? c + 2 : c + 1, 0);
    multiply(1);
  }
  if (c < chunks) multiply(0);
}

// u / (1 + e^-u) to fp32 accuracy with the hardware's exp2 and reciprocal: the product u * log2(e)
// keeps its rounding error, the reciprocal takes one Newton step.
__device__ __forceinline__ float small_silu(float u) {
  constexpr float kLog2e = 1.4426950408889634f, kLog2eLo = 1.925963033e-8f, kLn2 = 0.6931471805599453f;
  const float t = -u * kLog2e;
  const float lo = fmaf(-u, kLog2eLo, fmaf(-u, kLog2e, -t));
  float e = __builtin_amdgcn_exp2f(t);
  e = fabsf(t) < 126.0f ? fmaf(e, lo * kLn2, e) : e;
  const float d = 1.0f + e;
  const float r = __builtin_amdgcn_rcpf(d);
  // (below u = -87 the result is under 2^-119 and the reciprocal on its way to 0)
  return u * (t < 126.0f ? fmaf(r, fmaf(-d, r, 1.0f), r) : 0.0f);
}
// u / (1 + 2^(2 u)), of activations that carry the factor: the quotient by the approximate reciprocal, then by what it
// leaves (0.48 ulp rms; see split_silu8 in c6_split.h)
__device__ __forceinline__ float small_silu2(float u) {
#pragma clang fp contract(off)
  const float d = 1.0f + __builtin_amdgcn_exp2f(u + u);
  const float r = __builtin_amdgcn_rcpf(d);
  const float q = u * r;
  return fmaf(fminf(fmaf(-d, q, u), 0x1p100f), r, q);
}

// A workgroup evaluates `nb` boards of one weight set from input to heads; a wave owns PT tiles of
// 16 squares (of whichever of the boards) and all output channels of them, in every layer.  The
// activation buffer is updated in place: a wave keeps its outputs in accumulators until every wave
// has read its inputs.  Positions are channel-last with the layer's zero padding (rows r apart share
// their padding columns), so that a (tap, block of eight channels) is a constant offset, looked up
// in a table by the lane group that contracts it.
//
// Measured on 1024 boards of the 9x9 network above, fp32, calls in a row: 23 us (914 us layer by layer; 26 with a SiLU that puts the
// factor log2(e) in by itself, planes split value by value, a chunk's offset read in front of its operands, and the
// input loaded board by board behind the tables; 4096 boards of four such networks 96 -> 83 us, twenty 19x19 boards of
// kernels 7,3,3,3,3 and 32 channels 64 -> 53 us).  The MFMAs are 8 us of it at 2.4 GHz, all but the contractions 8 us
// (launch, staging, epilogues); the rest is the two waves per SIMD meeting at two barriers per layer and the reads of
// weights and activations, some 2 and 3 us.
enum : int { kTailInLds, kTailFar, kTailNone };   // (the last: weights read as they are)
template <class A, int PT, int TAIL>
__device__ __forceinline__ void small_net(const SmallParams &prm, unsigned char *smem) {
  constexpr bool RAW = TAIL == kTailNone;
  constexpr int NA = A::NA;
  const int tid = threadIdx.x, threads = blockDim.x;
  const int lane = tid & 63, wave = tid >> 6, q = lane >> 4;
  const int n = prm.n, nn = prm.nn;
  unsigned short *table = reinterpret_cast<unsigned short *>(smem + prm.table_off);
  int *s_pix = reinterpret_cast<int *>(smem + prm.pix_off);
  float *s_val = reinterpret_cast<float *>(smem + prm.val_off);
  int *s_inexact = reinterpret_cast<int *>(s_val);   // (until the heads)

  const long long g = blockIdx.x / prm.wgs_per_group;
  const long long first = (long long)(blockIdx.x % prm.wgs_per_group) * prm.nb;
  const int boards = (int)(prm.per_group - first < prm.nb ? prm.per_group - first : prm.nb);
  const long long b0 = g * prm.per_group + first;
  const unsigned char *weights = prm.packed + (size_t)g * prm.packed_stride;
  // Four words of the packed tail, from `at` on (+ 4 words per lane group): of a copy in LDS, so that no layer starts
  // behind their loads, or (small_full_kernel) from where they lie.
  auto tail4 = [&](int at, int group) __attribute__((always_inline)) {
    return *reinterpret_cast<const f32x4 *>((TAIL == kTailInLds ? smem + prm.tail_off : weights + prm.tail) + 4 * at + 16 * group);
  };
  const int npx = boards * nn;

  // a thread's square (there are as many threads as squares) and its input, asked for before anything else
  const int my_b = small_div(tid, prm.nn_magic), my_s = tid - my_b * nn, my_r = small_div(my_s, prm.n_magic), my_c = my_s - my_r * n;
  const bool has = tid < npx;
  float xin[3];
#pragma unroll
  for (int ch = 0; ch < 3; ++ch)
    xin[ch] = has ? small_load(prm.x, prm.x_dtype, ((size_t)(b0 + my_b) * 3 + ch) * nn + my_s) : 0.0f;
  if (has) s_pix[tid] = my_b << 16 | my_r << 8 | my_c;
  if constexpr (TAIL == kTailInLds)
    for (int i = tid; i < prm.tail_floats / 4; i += threads)
      reinterpret_cast<v4i *>(smem + prm.tail_off)[i] = reinterpret_cast<const v4i *>(weights + prm.tail)[i];
  // every layer's table of offsets (16-byte units)
  for (int l = 0; l < prm.layers; ++l) {
    const SmallLayer &L = prm.layer[l];
    for (int e = tid; e < 4 * L.chunks; e += threads) {
      int off = 0;
      if (e < L.blocks) {
        const int tap = small_div(e, L.cb_magic), cb = e - tap * L.cb, ky = small_div(tap, L.k_magic);
        off = ((ky * L.pitch + tap - ky * L.k) * L.pixb + cb * 16) >> 4;
      }
      table[L.table0 + e] = (unsigned short)off;
    }
  }
  {  // input planes: clear (padding, and the channels that fill a block), then scatter
    const SmallLayer &L = prm.layer[0];
    const v4i z = {0, 0, 0, 0};
    for (int i = tid; i < boards * L.boardb / 16; i += threads) reinterpret_cast<v4i *>(smem)[i] = z;
    if (tid == 0) *s_inexact = 0;
    __syncthreads();
    if (has) {
      bool inexact = false;
#pragma unroll
      for (int ch = 0; ch < 3; ++ch) inexact |= (__builtin_bit_cast(int, xin[ch]) & 0xffff) != 0 || !(__builtin_fabsf(xin[ch]) < __builtin_inff());
      if (inexact) *s_inexact = 1;
      unsigned char *at = smem + my_b * L.boardb + ((my_r + L.r) * L.pitch + my_c + L.r) * L.pixb;
#pragma unroll
      for (int ch = 0; ch < 3; ++ch) {
        unsigned short pl[NA];
        small_planes<A, true>(xin[ch], pl);
#pragma unroll
        for (int i = 0; i < NA; ++i) *reinterpret_cast<unsigned short *>(at + i * L.planeb + 2 * ch) = pl[i];
      }
    }
    __syncthreads();
  }
  const bool one_plane = __builtin_amdgcn_readfirstlane(*s_inexact) == 0;
  if (prm.layers == 1) __syncthreads();   // (no barrier of a layer's between this read and the heads' store to the word)

  int rc[PT];
  bool mine[PT];  // the lane's square exists (the others shadow the last one and store nothing)
#pragma unroll
  for (int j = 0; j < PT; ++j) {
    const int p = (wave * PT + j) * 16 + (lane & 15);
    mine[j] = p < npx;
    rc[j] = s_pix[mine[j] ? p : npx - 1];
  }
  const bool busy = wave * PT * 16 < npx;
  float pol[PT], val[PT];
#pragma unroll
  for (int j = 0; j < PT; ++j) pol[j] = val[j] = 0.0f;

  for (int l = 0; l < prm.layers; ++l) {
    const SmallLayer &L = prm.layer[l];
    const bool last = l + 1 == prm.layers;
    int base[PT];
#pragma unroll
    for (int j = 0; j < PT; ++j)
      base[j] = (rc[j] >> 16) * L.boardb + (((rc[j] >> 8) & 255) * L.pitch + (rc[j] & 255)) * L.pixb;
    auto run = [&](auto ct) __attribute__((always_inline)) {
      constexpr int CT = decltype(ct)::value;
      f32x4 acc[PT][CT], low[PT][CT];
      if (busy) {
#pragma unroll
        for (int t = 0; t < CT; ++t) {
          f32x4 b = {0.0f, 0.0f, 0.0f, 0.0f};
          if constexpr (!RAW) {  // (the tail holds zeros up to the next multiple of sixteen channels)
            b = tail4(L.bias0 + 16 * t, q);
          } else if (prm.conv_b[l] != nullptr) {
#pragma unroll
            for (int i = 0; i < 4; ++i)
              if (16 * t + 4 * q + i < L.cout) b[i] = (float)small_scale<A>(prm.conv_b[l][(size_t)g * L.cout + 16 * t + 4 * q + i], true);
          }
#pragma unroll
          for (int j = 0; j < PT; ++j) acc[j][t] = b;
        }
        if constexpr (RAW) {
          auto raw = [&](auto first) __attribute__((always_inline)) {
            const RawWeights<A, decltype(first)::value> w{prm.conv_w[l] + (size_t)g * L.cout * L.cin * L.k * L.k, L.cin, L.cout,
                                                          L.k * L.k, L.cb, (65536 + L.cb - 1) / L.cb, L.blocks, lane};
            small_contract<A, NA, PT, CT>(smem, table, w, L, lane, base, acc, low);
          };
          if (small_scaled<A>() && l == 0) raw(std::true_type{});
          else raw(std::false_type{});
        } else {
          const PackedWeights<A> w{weights + (size_t)L.frag0 * 1024 + lane * 16};
          // (stones and flags are exact in one plane: half the first layer's products, the others are zeros)
          if (A::NA > 1 && l == 0 && one_plane) small_contract<A, 1, PT, CT>(smem, table, w, L, lane, base, acc, low);
          else small_contract<A, NA, PT, CT>(smem, table, w, L, lane, base, acc, low);
        }
#pragma unroll
        for (int t = 0; t < CT; ++t) {
          f32x4 bl = {0.0f, 0.0f, 0.0f, 0.0f};   // what rounding the scaled biases left out, with the small products
          if constexpr (small_scaled<A>() && !RAW) {
            bl = tail4(small_low(prm.bias_total) + L.bias0 + 16 * t, q);
          } else if constexpr (small_scaled<A>()) {
            if (prm.conv_b[l] != nullptr)
#pragma unroll
              for (int i = 0; i < 4; ++i)
                if (16 * t + 4 * q + i < L.cout) {
                  const double v = small_scale<A>(prm.conv_b[l][(size_t)g * L.cout + 16 * t + 4 * q + i], true);
                  bl[i] = small_rest(v, (float)v);
                }
          }
#pragma unroll
          for (int j = 0; j < PT; ++j)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
              float u = acc[j][t][i];
              if constexpr (A::NA > 1 || A::NW > 1) u = two_sums(u, low[j][t][i] + bl[i]);
              acc[j][t][i] = small_scaled<A>() ? small_silu2(u) : small_silu(u);
            }
        }
      }
      if (last) {
        if (busy) {
          const int pw = prm.bias_total, vw = pw + 16 * kSmallMaxTiles;
#pragma unroll
          for (int t = 0; t < CT; ++t) {
            f32x4 p4 = {0.0f, 0.0f, 0.0f, 0.0f}, v4 = p4;
            if constexpr (RAW) {
#pragma unroll
              for (int i = 0; i < 4; ++i) {
                const int ch = 16 * t + 4 * q + i;
                if (ch >= L.cout) continue;
                p4[i] = prm.pol_w[(size_t)g * L.cout + ch];
                if (prm.val_w != nullptr) v4[i] = prm.val_w[(size_t)g * L.cout + ch];
              }
            } else {
              p4 = tail4(pw + 16 * t, q);
              v4 = tail4(vw + 16 * t, q);
            }
#pragma unroll
            for (int j = 0; j < PT; ++j)
#pragma unroll
              for (int i = 0; i < 4; ++i) {
                pol[j] = fmaf(p4[i], acc[j][t][i], pol[j]);
                val[j] = fmaf(v4[i], acc[j][t][i], val[j]);
              }
          }
        }
        return;
      }
      __syncthreads();  // everybody has read this layer's input
      const SmallLayer &N = prm.layer[l + 1];
      const v4i z = {0, 0, 0, 0};
      if (N.r > 0)
        for (int p = tid; p < N.positions; p += threads) {
          const int row = (int)__umulhi((unsigned)p, N.pitch_magic), col = p - row * N.pitch;
          if (row >= N.r && row < n + N.r && col >= N.r) continue;
          for (int b = 0; b < boards; ++b)
            for (int u = 0; u < N.pixb; u += 16) *reinterpret_cast<v4i *>(smem + b * N.boardb + p * N.pixb + u) = z;
        }
#pragma unroll
      for (int j = 0; j < PT; ++j) {
        if (!mine[j]) continue;
        unsigned char *at = smem + (rc[j] >> 16) * N.boardb +
                            ((((rc[j] >> 8) & 255) + N.r) * N.pitch + (rc[j] & 255) + N.r) * N.pixb;
#pragma unroll
        for (int t = 0; t < CT; ++t) {
          const int ch = 16 * t + 4 * q;
          if (ch >= 8 * N.cb) continue;
          if constexpr (A::F16) {
            unsigned short pl[4][NA];
#pragma unroll
            for (int i = 0; i < 4; ++i) small_planes<A>(acc[j][t][i], pl[i]);
            *reinterpret_cast<v2i *>(at + 2 * ch) = v2i{pl[0][0] | (int)pl[1][0] << 16, pl[2][0] | (int)pl[3][0] << 16};
          } else {
            float v[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) v[i] = acc[j][t][i];
#pragma unroll
            for (int i = 0; i < NA; ++i) {
              const int lo = small_take(v[0], v[1], i + 1 < NA), hi = small_take(v[2], v[3], i + 1 < NA);
              *reinterpret_cast<v2i *>(at + i * N.planeb + 2 * ch) = v2i{lo, hi};
            }
          }
        }
      }
      __syncthreads();
    };
    if (L.tiles == 1) run(std::integral_constant<int, 1>{});
    else if (L.tiles == 2) run(std::integral_constant<int, 2>{});
    else run(std::integral_constant<int, 3>{});
  }

  // heads: the four lane groups hold different channels of the same squares
  float pol_b = 0.0f, val_b = 0.0f;
  if constexpr (RAW) {
    if (prm.pol_b != nullptr) pol_b = prm.pol_b[g];
    if (prm.val_b != nullptr) val_b = prm.val_b[g];
  } else {
    const f32x4 heads = tail4(prm.bias_total + 2 * 16 * kSmallMaxTiles, 0);
    pol_b = heads[0];
    val_b = heads[1];
  }
#pragma unroll
  for (int j = 0; j < PT; ++j) {
    float p = pol[j], v = val[j];
    p += __shfl_xor(p, 16);
    p += __shfl_xor(p, 32);
    v += __shfl_xor(v, 16);
    v += __shfl_xor(v, 32);
    if (q == 0 && mine[j]) {
      const int b = rc[j] >> 16, s = ((rc[j] >> 8) & 255) * n + (rc[j] & 255);
      s_val[b * nn + s] = v;
      if (prm.logits != nullptr) {
        bool occupied = false;
        if (prm.mask_mode == C6_MASK_LEGAL) occupied = prm.legal[(size_t)(b0 + b) * nn + s] == 0;
        if (prm.mask_mode == C6_MASK_INPUT)
          occupied = small_load(prm.x, prm.x_dtype, (size_t)(b0 + b) * 3 * nn + s) != 0.0f ||
                     small_load(prm.x, prm.x_dtype, ((size_t)(b0 + b) * 3 + 1) * nn + s) != 0.0f;
        float z = p + pol_b;
        if constexpr (small_scaled<A>()) z = (float)((double)p * (1.0 / kSmallScale) + (double)pol_b);
        prm.logits[(size_t)(b0 + b) * nn + s] = occupied ? prm.fill : z;
      }
    }
  }
  if (prm.value != nullptr) {
    __syncthreads();
    for (int b = wave; b < boards; b += threads / 64) {
      float v = 0.0f;
      for (int s = lane; s < nn; s += 64) v += s_val[b * nn + s];
      v = wave_sum(v);
      if (lane == 0) prm.value[b0 + b] = (float)tanh((double)v * (small_scaled<A>() ? 1.0 / kSmallScale : 1.0) / nn + (double)val_b);   // (one rounding)
    }
  }
}

template <class A, int PT, bool RAW> __global__ __launch_bounds__(64 * kSmallMaxWaves) void small_net_kernel(const SmallParams prm) {
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  small_net<A, PT, RAW ? kTailNone : kTailInLds>(prm, smem);
}
// Networks whose activations leave no room for the tail's copy (19 x 19, ten layers of kernels 9 and 40 channels): a
// kernel of their own, since a branch at each read of the tail cost the others 1 % (9 x 9, 1,024 boards).
template <class A> __global__ __launch_bounds__(64 * kSmallMaxWaves) void small_full_kernel(const SmallParams prm) {
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  small_net<A, 3, kTailFar>(prm, smem);
}

// ---- weights ---------------------------------------------------------------------------------
// Fragment ((chunk * tiles + tile) * planes + plane) of a layer: lane (q, m) holds output channel
// 16 tile + m, (tap, block of eight input channels) pair 4 chunk + q.  Behind the fragments an fp32
// tail: biases (each layer's up to the next multiple of sixteen), policy and value weights (48
// each), the two head biases.
struct SmallPack {
  const float *conv_w[kSmallMaxLayers], *conv_b[kSmallMaxLayers];
  const float *pol_w, *pol_b, *val_w, *val_b;
  unsigned char *packed;
  size_t packed_stride, tail;
  int layers, frags, bias_total, channels;
  SmallLayer layer[kSmallMaxLayers];
};

template <class A> __global__ void small_pack_kernel(const SmallPack prm) {
  const long long g = blockIdx.y;
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  unsigned char *packed = prm.packed + (size_t)g * prm.packed_stride;
  if (i < (long long)prm.frags * 64) {   // one thread per (group of planes, lane)
    const int lane = (int)(i & 63);
    // (the same in a whole wave: the layer's numbers then come through the scalar cache)
    int f = __builtin_amdgcn_readfirstlane((int)(i >> 6)) * A::NW, l = 0;
    while (l + 1 < prm.layers && f >= prm.layer[l + 1].frag0) ++l;
    const SmallLayer &L = prm.layer[l];
    const int ct = (f - L.frag0) / A::NW, c = ct / L.tiles, t = ct - c * L.tiles;
    const int co = 16 * t + (lane & 15), e = 4 * c + (lane >> 4), tap = e / L.cb, cb = e - tap * L.cb;
    const float *w = prm.conv_w[l] + (size_t)g * L.cout * L.cin * L.k * L.k;
    unsigned short pl[8][A::NW];
    for (int k = 0; k < 8; ++k) {
      const int ci = 8 * cb + k;
      const bool in = e < L.blocks && co < L.cout && ci < L.cin;
      const float v = in ? w[((size_t)co * L.cin + ci) * L.k * L.k + tap] : 0.0f;
      small_weight_planes64<A>(small_scale<A>(v, l == 0), pl[k]);
    }
    for (int p = 0; p < A::NW; ++p) {
      v4i o;
      for (int d = 0; d < 4; ++d) o[d] = pl[2 * d][p] | (int)pl[2 * d + 1][p] << 16;
      *reinterpret_cast<v4i *>(packed + (size_t)(f + p) * 1024 + lane * 16) = o;
    }
    return;
  }
  const int ti = (int)(i - (long long)prm.frags * 64);
  float *tail = reinterpret_cast<float *>(packed + prm.tail);
  constexpr int kHead = 16 * kSmallMaxTiles;
  if (ti >= small_low(prm.bias_total)) return;
  float v = 0.0f;
  if (ti < prm.bias_total) {
    int l = 0;
    while (l + 1 < prm.layers && ti >= prm.layer[l + 1].bias0) ++l;
    const SmallLayer &L = prm.layer[l];
    const int c = ti - L.bias0;
    double b = 0.0;
    if (c < L.cout && prm.conv_b[l] != nullptr) b = small_scale<A>(prm.conv_b[l][(size_t)g * L.cout + c], true);
    v = (float)b;
    tail[small_low(prm.bias_total) + ti] = small_scaled<A>() ? small_rest(b, v) : 0.0f;
  } else {
    const int h = ti - prm.bias_total;
    const int c = h < kHead ? h : h - kHead;
    if (h < kHead) v = c < prm.channels ? prm.pol_w[(size_t)g * prm.channels + c] : 0.0f;
    else if (h < 2 * kHead) v = c < prm.channels && prm.val_w ? prm.val_w[(size_t)g * prm.channels + c] : 0.0f;
    else if (h == 2 * kHead) v = prm.pol_b ? prm.pol_b[g] : 0.0f;
    else if (h == 2 * kHead + 1) v = prm.val_b ? prm.val_b[g] : 0.0f;
  }
  tail[ti] = v;
}

// ---- host side ---------------------------------------------------------------------------------
// Which operands a mode rounds to 16 bits is the layer-by-layer path's contract (c6_generic.hip):
// fp32 and the mode that carries the weights' low part round nothing, the other bf16 modes the
// weights (those that carry the activations' low part) or both, fp16 both.
enum : int { kSmallF32, kSmallW16, kSmallBF16, kSmallF16 };
static int small_arith(int prec) {
  switch (prec) {
    case C6_PREC_F32:
    case C6_PREC_F32S:
    case C6_PREC_BF16F6W: return kSmallF32;
    case C6_PREC_BF16: return kSmallBF16;
    case C6_PREC_F16: return kSmallF16;
    default: return kSmallW16;
  }
}
static int small_weight_planes(int arith) { return arith == kSmallF32 ? 3 : 1; }
static int small_act_planes(int arith) { return arith == kSmallF32 || arith == kSmallW16 ? 3 : 1; }

// p / d as the high half of p * small_magic(d), for p * d < 2^32 (d = 1: p itself, see small_div)
static unsigned small_magic(int d) { return d == 1 ? 0 : (unsigned)((0x100000000ull + d - 1) / d); }

struct SmallPlan {
  SmallLayer layer[kSmallMaxLayers];
  int frags = 0, bias_total = 0, entries = 0, boardb = 0;
  size_t tail = 0, bytes = 0;
};

// copy: with the packed tail behind the rest
static int small_lds(const SmallPlan &pl, int nn, int nb, bool copy, SmallParams *sp = nullptr) {
  const int t = (nb * pl.boardb + 15) & ~15;
  const int p = (t + 2 * pl.entries + 15) & ~15;
  const int v = p + 4 * nb * nn;
  const int w = (v + 4 * nb * nn + 15) & ~15, floats = copy ? (int)((pl.bytes - pl.tail) / 4) : 0;
  if (sp) sp->table_off = t, sp->pix_off = p, sp->val_off = v, sp->tail_off = w, sp->tail_floats = floats;
  return w + 4 * floats;
}

// The layout of a network, or false where one board does not fit: more than 48 channels (a wave
// carries three tiles), more than 8 x 48 squares, or a padded board beyond the LDS of a CU.
static bool small_plan(int n, int layers, const int *kernels, const int *channels, int prec, SmallPlan &pl) {
  if (n < 1 || n > 19 || layers < 1 || layers > kSmallMaxLayers) return false;
  const int arith = small_arith(prec), na = small_act_planes(arith), nw = small_weight_planes(arith);
  int cin = 3;
  for (int l = 0; l < layers; ++l) {
    SmallLayer &L = pl.layer[l];
    if (channels[l] > 16 * kSmallMaxTiles || kernels[l] > 63) return false;
    L.k = kernels[l];
    L.r = L.k / 2;
    L.cin = cin;
    L.cb = (cin + 7) / 8;
    L.cout = channels[l];
    L.tiles = (L.cout + 15) / 16;
    L.blocks = L.k * L.k * L.cb;
    L.chunks = (L.blocks + 3) / 4;
    L.frag0 = pl.frags;
    L.bias0 = pl.bias_total;
    L.pitch = n + L.r;
    L.pitch_magic = small_magic(L.pitch);
    L.k_magic = small_magic(L.k);
    L.cb_magic = small_magic(L.cb);
    L.positions = (n + 2 * L.r) * L.pitch + L.r;
    L.planeb = 16 * L.cb;
    // (an odd number of 16-byte units: sixteen consecutive squares then read sixteen bank groups)
    L.pixb = (na * L.cb) % 2 ? na * L.planeb : na * L.planeb + 16;
    L.boardb = L.positions * L.pixb;
    L.table0 = pl.entries;
    pl.frags += L.chunks * L.tiles * nw;
    pl.bias_total += 16 * L.tiles;
    pl.entries += 4 * L.chunks;
    pl.boardb = L.boardb > pl.boardb ? L.boardb : pl.boardb;
    if (pl.entries > kSmallTableEntries || pl.boardb > kSmallLds) return false;
    cin = L.cout;
  }
  pl.tail = (size_t)pl.frags * 1024;
  pl.bytes = pl.tail + (size_t)(small_low(pl.bias_total) + pl.bias_total) * 4;
  return small_lds(pl, n * n, 1, false) <= kSmallLds;
}

size_t small_packed_bytes(int n, int layers, const int *kernels, const int *channels, int prec) {
  SmallPlan pl;
  return small_plan(n, layers, kernels, channels, prec, pl) ? pl.bytes : 0;
}

static int small_done(const char *what) {
  const hipError_t e = hipGetLastError();
  if (e == hipSuccess) return C6_OK;
  set_error("%s launch failed: %s", what, hipGetErrorString(e));
  return C6_ELAUNCH;
}

int launch_small_pack(long long groups, int n, int layers, const int *kernels, const int *channels,
                      const float *const *conv_w, const float *const *conv_b, const float *pol_w, const float *pol_b,
                      const float *val_w, const float *val_b, int prec, void *packed, size_t packed_stride,
                      hipStream_t st) {
  SmallPlan pl;
  if (!small_plan(n, layers, kernels, channels, prec, pl)) {
    set_error("c6_generic_pack: this architecture has no packed form (c6_generic_packed_bytes is 0)");
    return C6_EINVAL;
  }
  SmallPack pp;
  const int arith = small_arith(prec);
  for (int l = 0; l < layers; ++l) {
    pp.conv_w[l] = conv_w[l];
    pp.conv_b[l] = conv_b ? conv_b[l] : nullptr;
    pp.layer[l] = pl.layer[l];
  }
  pp.pol_w = pol_w;
  pp.pol_b = pol_b;
  pp.val_w = val_w;
  pp.val_b = val_b;
  pp.packed = static_cast<unsigned char *>(packed);
  pp.packed_stride = packed_stride;
  pp.tail = pl.tail;
  pp.layers = layers;
  pp.frags = pl.frags / small_weight_planes(arith);
  pp.bias_total = pl.bias_total;
  pp.channels = channels[layers - 1];
  const long long items = (long long)pp.frags * 64 + small_low(pl.bias_total);
  const dim3 grid((unsigned)((items + 255) / 256), (unsigned)groups);
  switch (arith) {
    case kSmallF32: hipLaunchKernelGGL((small_pack_kernel<SmallArith<3, 3, false>>), grid, dim3(256), 0, st, pp); break;
    case kSmallF16: hipLaunchKernelGGL((small_pack_kernel<SmallArith<1, 1, true>>), grid, dim3(256), 0, st, pp); break;
    default: hipLaunchKernelGGL((small_pack_kernel<SmallArith<1, 1, false>>), grid, dim3(256), 0, st, pp); break;
  }
  return small_done("small_pack_kernel");
}

template <auto KERNEL> static int small_launch(const SmallParams &sp, unsigned grid, int waves, int lds, hipStream_t st) {
  static thread_local int configured = -1;
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e == hipSuccess && configured != dev) {
    e = hipFuncSetAttribute(reinterpret_cast<const void *>(KERNEL), hipFuncAttributeMaxDynamicSharedMemorySize, kSmallLds);
    if (e == hipSuccess) configured = dev;
  }
  if (e != hipSuccess) {
    set_error("small_net_kernel setup failed: %s", hipGetErrorString(e));
    return C6_ELAUNCH;
  }
  hipLaunchKernelGGL(KERNEL, dim3(grid), dim3(64 * waves), lds, st, sp);
  return small_done("small_net_kernel");
}

// packed != nullptr: that copy's weights, else the tensors conv_w ... val_b
int launch_small(const void *x, int x_dtype, long long groups, long long per_group, int n, int layers,
                 const int *kernels, const int *channels, const void *packed, size_t packed_stride,
                 const float *const *conv_w, const float *const *conv_b, const float *pol_w, const float *pol_b,
                 const float *val_w, const float *val_b, int prec, float *logits, float *value, int mask_mode, const uint8_t *legal, float fill, hipStream_t st) {
  SmallPlan pl;
  if (!small_plan(n, layers, kernels, channels, prec, pl)) {
    set_error("c6_forward_generic_packed: this architecture has no packed form (c6_generic_packed_bytes is 0)");
    return C6_EINVAL;
  }
  const int nn = n * n, arith = small_arith(prec);
  // Three tiles of 16 squares per wave read a weight fragment once for three MFMAs (18 in fp32), so
  // that the matrix cores and not the reads from L2 bound the wave; that takes enough squares to
  // give every SIMD of the chip a wave.  Below that one tile per wave: latency counts.
  // (Weights straight from the tensors are converted by every wave: always three tiles.  So where there is no room for
  // the tail's copy: one kernel for those is enough.)
  const bool copy = packed != nullptr && small_lds(pl, nn, 1, true) <= kSmallLds;
  const bool wide = groups * per_group * nn >= 48LL * 1024 || nn > 16 * kSmallMaxWaves || !copy;
  const int span = wide ? 48 : 16;
  // boards per workgroup: four waves' worth of squares (two workgroups and more share a CU), fewer
  // where that would leave CUs without a workgroup, one board at least
  long long nb = 4 * span / nn;
  if (nb > per_group) nb = per_group;
  while (nb > 1 && (groups * ((per_group + nb - 1) / nb) < 256 || small_lds(pl, nn, (int)nb, copy) > kSmallLds / 2))
    --nb;
  if (nb < 1) nb = 1;
  SmallParams sp;
  sp.x = x;
  sp.x_dtype = x_dtype;
  sp.per_group = per_group;
  sp.wgs_per_group = (int)((per_group + nb - 1) / nb);
  sp.packed = static_cast<const unsigned char *>(packed);
  sp.packed_stride = packed_stride;
  sp.tail = pl.tail;
  sp.n = n;
  sp.nn = nn;
  sp.n_magic = small_magic(n);
  sp.nn_magic = small_magic(nn);
  sp.layers = layers;
  sp.nb = (int)nb;
  sp.bias_total = pl.bias_total;
  sp.logits = logits;
  sp.value = value;
  sp.mask_mode = mask_mode;
  sp.legal = legal;
  sp.fill = fill;
  for (int l = 0; l < layers; ++l) {
    sp.layer[l] = pl.layer[l];
    sp.conv_w[l] = conv_w ? conv_w[l] : nullptr;
    sp.conv_b[l] = conv_b ? conv_b[l] : nullptr;
  }
  sp.pol_w = pol_w;
  sp.pol_b = pol_b;
  sp.val_w = val_w;
  sp.val_b = val_b;
  const int lds = small_lds(pl, nn, (int)nb, copy, &sp);
  const int waves = (int)((nb * nn + span - 1) / span);
  const long long grid = groups * sp.wgs_per_group;
  if (grid > 0x7fffffffLL) {
    set_error("c6_forward_generic_packed: %lld workgroups exceed one launch", grid);
    return C6_EINVAL;
  }
#define C6_SMALL(A)                                                           \
  if (packed == nullptr) return small_launch<small_net_kernel<A, 3, true>>(sp, (unsigned)grid, waves, lds, st); \
  if (!copy) return small_launch<small_full_kernel<A>>(sp, (unsigned)grid, waves, lds, st);                      \
  return wide ? small_launch<small_net_kernel<A, 3, false>>(sp, (unsigned)grid, waves, lds, st)                 \
              : small_launch<small_net_kernel<A, 1, false>>(sp, (unsigned)grid, waves, lds, st)
  using F32 = SmallArith<3, 3, false>;
  using W16 = SmallArith<3, 1, false>;
  using B16 = SmallArith<1, 1, false>;
  using H16 = SmallArith<1, 1, true>;
  switch (arith) {
    case kSmallF32: C6_SMALL(F32);
    case kSmallW16: C6_SMALL(W16);
    case kSmallBF16: C6_SMALL(B16);
    default: C6_SMALL(H16);
  }
#undef C6_SMALL
}

}  // namespace c6
