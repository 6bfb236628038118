// Fully connected ("uv") Clebsch-Gordan tensor product in single precision on the half-precision matrix cores:
//
//   out[n, m, w] = sum_t coef_t * y[n, b_t] * sum_u x[n, a_t, u] * W[p_t, u, w]
//
// for the compiled tables; forward, the gradient of x (the same with the rows' roles exchanged and the weight read
// transposed) and the gradient of y.  The order is that of uv_mfma.hip: per weight path and input row two accumulator
// tiles Z = x W, then the coefficients as fp32 multiply-adds between accumulator tiles.
//
// Every fp32 operand a is carried as three bf16 parts, h = bf16(a), m = bf16(a - h), l = a - h - m: 8 bits each, together
// all 24 of a, and bf16 has the exponents of fp32, so no scales (2^-110 <= |a| < 2^60; see below).  Z is h h' + h m' + m h' +
// h l' + l h' + m m', each product exact in fp32, 32 of them summed to a rounding, the five small ones by themselves; what is
// dropped (m l', l m', l l') is about 2^-24 of an element product at most, one rounding of it, and 2^-27 as a rule.  Errors of
// the results against 64 bits, lmax 1 to 3, 32 to 128 channels: 0.5e-7 to 1.7e-7 where fp32 matrix instructions give 0.9e-7 to
// 5.1e-7; with channels and elements spread over thirty binary orders never above them.  The same contraction in fp32
// matrix instructions takes 256 cycles per 16 x 16 tile and 32 channels, this one 96.  (Two half-precision parts and three
// products, 48 cycles, need a common scale per row and path: elements and channels far below the largest lose bits, and
// so do products far from 1.)
//
// What bounds it: a workgroup of four wavefronts owns 16 samples, whose rows (4 or 6 bytes an element) fill most of the LDS at
// 128 channels and lmax = 2 and 3, and every workgroup reads all the weights from L2, 2.3 MB there.  One wavefront per
// SIMD at 128 channels (lmax = 3): matrix pipeline 41 % busy, vector instructions 39 %, waiting for data 18 %.  128 -> 128
// channels, lmax = 3, 32768 samples: forward 1308 -> 677 us, gradient of x 1316 -> 679, of y 1879 -> 649 (fp32 matrix
// instructions, coupling first, against this); 64 -> 64, lmax = 2: 140 / 135 / 188 -> 77 / 76 / 74; 500 samples of 128 channels,
// lmax = 3: 161 / 162 / 228 -> 82 / 82 / 79.  Splitting the rows in every tile that reads them took 800 us there (vector
// instructions 52 %): as many rows as fit are staged as parts (UvsLds), the others split between matrix instructions.
//
// An x or W with an element that is not finite, from 2^60 on (Z could overflow where coupling first does not) or below 2^-110 but
// not zero (its last part could be below the smallest subnormal), a y that is not finite, or a y of 16 and more next to an x or W below 2^-50 (Z could
// underflow where coupling first does not) is not split: the workgroup then forms its samples' results with fp32 matrix
// instructions, the coupling first (UvsPlain), so that such values reach exactly the
// results they couple to.
#include "uv_parts.h"

#include <algorithm>

// accumulator-tile updates are written as o += s * z; let them contract to FMAs in this file
#pragma clang fp contract(fast)

namespace cgtp {

struct UvsTerm {
  float c;
  unsigned char o, a, b, p;      // rows of out, x and y, path
};

#include "generated/uv_split_configs.inc"

constexpr int kUvsSamples = 16;

// Barrier; `m` or'ed over the workgroup's four wavefronts (`words`: four words of LDS).
__device__ __forceinline__ unsigned uvs_all(unsigned m, unsigned* words) {
  unsigned w = 0;
#pragma unroll
  for (unsigned bit = 1; bit <= kUvsLargeY; bit <<= 1) w |= __any((m & bit) != 0) ? bit : 0;
  if ((threadIdx.x & (kWave - 1)) == 0) words[threadIdx.x / kWave] = w;
  __syncthreads();
  return words[0] | words[1] | words[2] | words[3];
}
__device__ __forceinline__ bool uvs_is_plain(unsigned m) {
  return (m & kUvsPlain) || ((m & kUvsSmall) && (m & kUvsLargeY));
}

// The weight as the caller holds it.  With channels on both operands a path has one matrix per channel l of the operand
// that is not contracted; `matrices` is their number (else 1), and a "path" of the packed weight is a (path, l).
struct UvsWeight {
  const float* w;
  int64_t stride_p, stride_k, stride_c, stride_l;
  int matrices;
  __device__ __forceinline__ const float* of(int i) const { return w + (i / matrices) * stride_p + (i % matrices) * stride_l; }
};

// A workgroup per path and block of 32 output channels: the parts of its block in fragment order.  Per path and block 3 (part)
// x 2 (tile) x K / 32 chunks of 1 KB, holding the 16 bytes of every lane; row r of tile t is output channel
// 8 (r / 4) + 4 t + r % 4 of the block.  asks: a word per path and block.
__global__ void __launch_bounds__(256) uvs_pack_kernel(UvsWeight W, __bf16* __restrict__ packed, unsigned* __restrict__ asks, int K,
                                                       int cout) {
  __shared__ unsigned words[4];
  const int p = blockIdx.x, blk = blockIdx.y, ks = K / 32;
  const float* wp = W.of(p);
  unsigned m = 0;
  for (int i = threadIdx.x; i < K * 4; i += 256) {             // fragments of eight k
    const int lane = i & 63, c = i >> 6, k = c % ks, t = c / ks;
    const int r = lane & 15, q = lane >> 4;
    const int row = blk * 32 + 8 * (r >> 2) + 4 * t + (r & 3), col = k * 32 + 8 * q;
    float v[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      v[j] = wp[(col + j) * W.stride_k + row * W.stride_c];
      m |= uvs_asks(v[j]);
    }
    UvsParts<8> part;
#pragma unroll
    for (int j = 0; j < 4; ++j) part.pair(j, v[2 * j], v[2 * j + 1]);
    __bf16* dst = packed + (int64_t)p * K * cout * 3 + ((int64_t)(blk * 6 + t) * ks + k) * 512 + lane * 8;
#pragma unroll
    for (int h = 0; h < 3; ++h) *reinterpret_cast<bf16x8*>(dst + (int64_t)h * 2 * ks * 512) = uvs_frag(part.p[h]);
  }
  m = uvs_all(m, words);
  if (threadIdx.x == 0) asks[p * (cout / 32) + blk] = m;
}

// LDS: per sample DIN rows and 16 bytes of padding, then four words (uvs_all).  The rows from kRaw on hold the three parts of
// CIN elements each, the ones before (those of the low degrees, which fewer tiles read) CIN floats that every tile splits
// anew: as many as the LDS asks for without costing a workgroup per compute unit (two at 32 and 64 channels, one at 128).
constexpr int uvs_raw_rows(int din, int cin) {
  for (int raw = 0; raw < din; ++raw)
    if (kUvsSamples * (cin * (6 * din - 2 * raw) + 16) + 16 <= (cin < 128 ? kLdsBytes / 2 : kLdsBytes)) return raw;
  return din;
}
template <int DIN, int CIN>
struct UvsLds {
  static constexpr int kRaw = uvs_raw_rows(DIN, CIN), kPitch = CIN * (6 * DIN - 2 * kRaw) + 16, kTile = kUvsSamples * kPitch;
  static __device__ __forceinline__ constexpr int row(int r) { return CIN * (6 * r - 2 * (r < kRaw ? r : kRaw)); }
};

// Stages the 16 samples' rows; what this thread's elements ask for.
template <int DIN, int CIN>
__device__ __forceinline__ unsigned uvs_stage(const float* __restrict__ x, int64_t n0, int64_t n_rows, unsigned char* smem) {
  using L = UvsLds<DIN, CIN>;
  constexpr int ROW = CIN / 4, PER = DIN * ROW, TOTAL = kUvsSamples * PER;
  unsigned m = 0;
  constexpr int UNROLL = 8;
  for (int base = 0; base < TOTAL; base += 256 * UNROLL) {
    f32x4 v[UNROLL];
#pragma unroll
    for (int u = 0; u < UNROLL; ++u) {
      const int i = base + u * 256 + (int)threadIdx.x;
      if (i < TOTAL) v[u] = *reinterpret_cast<const f32x4*>(x + min(n0 + i / PER, n_rows - 1) * (DIN * CIN) + i % PER * 4);
    }
#pragma unroll
    for (int u = 0; u < UNROLL; ++u) {
      const int i = base + u * 256 + (int)threadIdx.x;
      if (i < TOTAL) {
        float a[4];                     // a bit cast of the vector's element itself would read element 0
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          a[j] = v[u][j];
          m |= uvs_asks(a[j]);
        }
        unsigned char* row = smem + i / PER * L::kPitch + L::row(i % PER / ROW);
        if (i % PER / ROW >= L::kRaw) {
          UvsParts<4> part;
          part.pair(0, a[0], a[1]);
          part.pair(1, a[2], a[3]);
#pragma unroll
          for (int h = 0; h < 3; ++h)
            *reinterpret_cast<u32x2*>(row + h * CIN * 2 + i % ROW * 8) = u32x2{part.p[h][0], part.p[h][1]};
        } else {
          *reinterpret_cast<f32x4*>(row + i % ROW * 16) = v[u];
        }
      }
    }
  }
  return m;
}

template <int DIN, int CIN>
struct UvsOps {
  using L = UvsLds<DIN, CIN>;
  static constexpr int KS = CIN / 32;
  struct A { bf16x8 f[3][2][KS]; };         // [part][tile][step]
  struct B { u32x4 v[KS][L::kRaw == DIN ? 2 : 3]; bool raw; };
  struct Z { floatx4 z[2], s[2]; };         // sums of the large products and of the small ones
  const __bf16* wp;                         // this lane's fragments of path 0
  int64_t path_stride;
  const unsigned char* xs;                  // its sample's rows
  int q;                                    // its eight elements of a step
  __device__ __forceinline__ void load_a(int p, A& a) const {
#pragma unroll
    for (int h = 0; h < 3; ++h)
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int k = 0; k < KS; ++k)
          a.f[h][t][k] = *reinterpret_cast<const bf16x8*>(wp + p * path_stride + ((h * 2 + t) * KS + k) * 512);
  }
  __device__ __forceinline__ void load_b(int row, B& b) const {
    b.raw = row < L::kRaw;
    const unsigned char* at = xs + L::row(row) + q * (b.raw ? 32 : 16);
#pragma unroll
    for (int k = 0; k < KS; ++k)
#pragma unroll
      for (int h = 0; h < (L::kRaw == DIN ? 2 : 3); ++h)
        if (h < 2 || !b.raw)
          b.v[k][h] = *reinterpret_cast<const u32x4*>(at + k * (b.raw ? 128 : 64) + h * (b.raw ? 16 : CIN * 2));
  }
  // A tile.  A row staged as floats is split here, a step ahead of the matrix instructions that take it: one matrix
  // instruction (16 cycles) and a few vector ones beside it in turn.
  __device__ __forceinline__ void chain(const A& a, const B& b, Z& out) const {
#pragma unroll
    for (int t = 0; t < 2; ++t) out.z[t] = out.s[t] = floatx4{0.f, 0.f, 0.f, 0.f};
    const auto element = [&](int k, int j) __attribute__((always_inline)) {
      const unsigned w = b.v[k][j / 4][j % 4];
      return __builtin_bit_cast(float, w);
    };
    UvsParts<8> part[2];
    if (b.raw) {
#pragma unroll
      for (int j = 0; j < 4; ++j) part[0].pair(j, element(0, 2 * j), element(0, 2 * j + 1));
    }
#pragma unroll
    for (int k = 0; k < KS; ++k) {
      bf16x8 x[3];
#pragma unroll
      for (int h = 0; h < 3; ++h)
        x[h] = b.raw || L::kRaw == DIN ? uvs_frag(part[k & 1].p[h]) : __builtin_bit_cast(bf16x8, b.v[k][L::kRaw == DIN ? 0 : h]);
#pragma unroll
      for (int i = 0; i < 12; ++i) {
        const int t = i & 1, c = i >> 1;          // h h' of the two tiles, then the small products
        const int ha = c == 1 ? 2 : c == 2 || c == 4 ? 1 : 0, hb = c == 3 ? 2 : c == 2 || c == 5 ? 1 : 0;
        floatx4& sum = c == 0 ? out.z[t] : out.s[t];
        sum = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a.f[ha][t][k], x[hb], sum, 0, 0, 0);
        if (b.raw && k + 1 < KS) {
          const int j = i / 3;
          const float v = element(k + 1, 2 * j), w = element(k + 1, 2 * j + 1);
          if (i % 3 == 0) part[(k + 1) & 1].template stage<0>(j, v, w);
          else if (i % 3 == 1) part[(k + 1) & 1].template stage<1>(j, v, w);
          else part[(k + 1) & 1].template stage<2>(j, v, w);
          __builtin_amdgcn_sched_barrier(0);
        }
      }
    }
  }
  static __device__ __forceinline__ void sum(const Z& in, floatx4& z0, floatx4& z1) {
    z0 = in.z[0] + in.s[0];
    z1 = in.z[1] + in.s[1];
  }
};

// ---- workgroups whose operands are not split: fp32 matrix instructions, operands from memory ---------------------
// The coupling comes first, path by path and row by row of the result, so the table is walked in the order of (row, path).
// A lane of the contraction's quarter q holds K / 4 consecutive elements of its sample; any order of k will do where both
// operands agree.  One wavefront per SIMD or two, waiting for memory most of the time.  128 -> 128 channels, lmax 3: a launch
// with one such workgroup 613 us (term by term 2433), 4096 samples that all are 647 (fp32 instructions throughout: 181).
template <int K>
struct UvsPlain {
  static constexpr int N = K / 4;
  float u[N];
  __device__ __forceinline__ void clear() {
#pragma unroll
    for (int i = 0; i < N; ++i) u[i] = 0.f;
  }
  __device__ __forceinline__ void mix(const float* __restrict__ xrow, float s, int q) {
#pragma unroll
    for (int i = 0; i < N; i += 4) {
      const f32x4 v = *reinterpret_cast<const f32x4*>(xrow + q * N + i);
#pragma unroll
      for (int j = 0; j < 4; ++j) u[i + j] += s * v[j];
    }
  }
  // o += u W for the two tiles of block `blk`.
  __device__ __forceinline__ void multiply(const UvsWeight& W, int matrix, int blk, int r, int q, floatx4 (&o)[2]) const {
    const float* wb = W.of(matrix) + (blk * 32 + 8 * (r >> 2) + (r & 3)) * W.stride_c + q * N * W.stride_k;
    floatx4 z[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
    constexpr int STEPS = 8;      // of which the loads are in flight together
#pragma unroll
    for (int i0 = 0; i0 < N; i0 += STEPS) {
      float w[STEPS][2];
#pragma unroll
      for (int i = 0; i < STEPS; ++i)
#pragma unroll
        for (int t = 0; t < 2; ++t) w[i][t] = wb[(i0 + i) * W.stride_k + 4 * t * W.stride_c];
#pragma unroll
      for (int i = 0; i < STEPS; ++i)
#pragma unroll
        for (int t = 0; t < 2; ++t) z[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(w[i][t], u[i0 + i], z[t], 0, 0, 0);
    }
    o[0] += z[0];
    o[1] += z[1];
  }
};
// Rows of the result, of the contracted operand and of the other one; KIND as for the launches with channels on both operands.
template <int KIND>
__device__ __forceinline__ int uvs_row_of(const UvsTerm& e) { return KIND == 0 ? e.o : KIND == 1 ? e.a : e.b; }
template <int KIND>
__device__ __forceinline__ int uvs_in_of(const UvsTerm& e) { return KIND == 0 ? e.a : e.o; }
template <int KIND>
__device__ __forceinline__ int uvs_other_of(const UvsTerm& e) { return KIND == 2 ? e.a : e.b; }
// The terms of (row, path) from t on; `t` moves behind them.
template <class TAB, int KIND, class F>
__device__ __forceinline__ void uvs_segment(int& t, int row, int path, F&& f) {
  for (; t < TAB::N; ++t) {
    const UvsTerm e = TAB::terms(KIND)[t];
    if (uvs_row_of<KIND>(e) != row || e.p != path) break;
    f(e);
  }
}

// DIR 0: forward, 1: gradient of x (terms with the rows of out and x exchanged).
template <class CFG, class TAB, int DIR, int CIN, int WAVES>
__global__ void __launch_bounds__(256, WAVES) uvs_kernel(const float* __restrict__ x, const float* __restrict__ y,
                                                         const __bf16* __restrict__ wp, const unsigned* __restrict__ asks_w,
                                                         float* __restrict__ out, int64_t n_rows, int cout, UvsWeight W) {
  extern __shared__ __align__(16) unsigned char smem[];
  constexpr int DIN = CFG::DIN, DOUT = CFG::DOUT, D2 = CFG::D2;
  using L = UvsLds<DIN, CIN>;
  const int64_t n0 = (int64_t)blockIdx.x * kUvsSamples;
  unsigned m = uvs_stage<DIN, CIN>(x, n0, n_rows, smem);
  const int n_blocks = cout / 32;
  for (int i = threadIdx.x; i < CFG::P * 4; i += blockDim.x) {
    const int blk = blockIdx.y * 4 + (i & 3);
    if (blk < n_blocks) m |= asks_w[(i >> 2) * n_blocks + blk];
  }
  for (int i = threadIdx.x; i < kUvsSamples * D2; i += blockDim.x)
    m |= uvs_asks_y(y[min(n0 + i / D2, n_rows - 1) * D2 + i % D2]);
  const bool plain = uvs_is_plain(uvs_all(m, reinterpret_cast<unsigned*>(smem + L::kTile)));

  const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x / kWave;
  const int n = lane & 15, q = lane >> 4;
  const int64_t row_n = min(n0 + n, n_rows - 1);
  const bool valid = n0 + n < n_rows;
  const int wblk = blockIdx.y * (blockDim.x / kWave) + wave;      // one 32-channel block per wavefront
  if (wblk * 32 >= cout) return;
  float* orow = out + (n0 + n) * DOUT * cout + wblk * 32 + 8 * q;
  auto store = [&](int row, const floatx4& o0, const floatx4& o1) __attribute__((always_inline)) {
    if (valid) {       // written once and not read again by this launch
      __builtin_nontemporal_store(o0, reinterpret_cast<floatx4*>(orow + row * cout));
      __builtin_nontemporal_store(o1, reinterpret_cast<floatx4*>(orow + row * cout + 4));
    }
  };
  if (plain) {
    UvsPlain<CIN> P;
    int t = 0;
    for (int row = 0; row < DOUT; ++row) {
      floatx4 o[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
      while (t < TAB::N && uvs_row_of<DIR>(TAB::terms(DIR)[t]) == row) {
        const int path = TAB::terms(DIR)[t].p;
        P.clear();
        uvs_segment<TAB, DIR>(t, row, path, [&](const UvsTerm& e) __attribute__((always_inline)) {
          P.mix(x + (row_n * DIN + uvs_in_of<DIR>(e)) * CIN, e.c * y[row_n * D2 + e.b], q);
        });
        P.multiply(W, path, wblk, n, q, o);
      }
      store(row, o[0], o[1]);
    }
    return;
  }
  float yv[D2];
#pragma unroll
  for (int j = 0; j < D2; ++j) yv[j] = y[row_n * D2 + j];
  const UvsOps<DIN, CIN> ops{wp + (int64_t)wblk * (6 * (CIN / 32) * 512) + lane * 8, (int64_t)cout * CIN * 3,
                        smem + n * L::kPitch, q};
  CFG::run(ops, yv, store);
}

// gy[n, b] = sum_t coef_t * sum_w g[n, m_t, w] * Z[p_t, a_t][w, n]: the forward's tiles; the lane sums over its channels, the
// four lanes of a sample and the wavefronts (channel blocks, cout <= 128) are then added in a fixed order.
template <class CFG, class TAB, int CIN, int WAVES>
__global__ void __launch_bounds__(256, WAVES) uvs_gy_kernel(const float* __restrict__ x, const float* __restrict__ g,
                                                            const __bf16* __restrict__ wp, const unsigned* __restrict__ asks_w,
                                                            float* __restrict__ gy, int64_t n_rows, int cout, UvsWeight W) {
  extern __shared__ __align__(16) unsigned char smem[];
  constexpr int DIN = CFG::DIN, DOUT = CFG::DOUT, D2 = CFG::D2;
  using L = UvsLds<DIN, CIN>;
  const int64_t n0 = (int64_t)blockIdx.x * kUvsSamples;
  unsigned m = uvs_stage<DIN, CIN>(x, n0, n_rows, smem);
  const int n_blocks = cout / 32;
  for (int i = threadIdx.x; i < CFG::P * 4; i += blockDim.x) {
    const int blk = blockIdx.y * 4 + (i & 3);
    if (blk < n_blocks) m |= asks_w[(i >> 2) * n_blocks + blk];
  }
  const bool plain = uvs_is_plain(uvs_all(m, reinterpret_cast<unsigned*>(smem + L::kTile)));

  const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x / kWave;
  const int n = lane & 15, q = lane >> 4;
  const int64_t row_n = min(n0 + n, n_rows - 1);
  const float* grow = g + row_n * DOUT * cout + min(wave, n_blocks - 1) * 32 + 8 * q;
  float part[D2];
#pragma unroll
  for (int j = 0; j < D2; ++j) part[j] = 0.f;
  auto load_g = [&](int row, floatx4& g0, floatx4& g1) __attribute__((always_inline)) {
    g0 = *reinterpret_cast<const floatx4*>(grow + row * cout);
    g1 = *reinterpret_cast<const floatx4*>(grow + row * cout + 4);
  };
  if (wave < n_blocks) {
    if (plain) {
      UvsPlain<CIN> P;
      for (int t = 0; t < TAB::N;) {      // in the order of (row of x, path), whose terms share Z
        const int row = TAB::terms(1)[t].a, path = TAB::terms(1)[t].p;
        floatx4 z[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
        P.clear();
        P.mix(x + (row_n * DIN + row) * CIN, 1.f, q);
        P.multiply(W, path, wave, n, q, z);
        uvs_segment<TAB, 1>(t, row, path, [&](const UvsTerm& e) __attribute__((always_inline)) {
          floatx4 g0, g1;
          load_g(e.o, g0, g1);
          const float v = e.c * dot8(g0, g1, z[0], z[1]);
#pragma unroll
          for (int j = 0; j < D2; ++j)
            if (j == e.b) part[j] += v;
        });
      }
    } else {
      const UvsOps<DIN, CIN> ops{wp + (int64_t)wave * (6 * (CIN / 32) * 512) + lane * 8, (int64_t)cout * CIN * 3,
                            smem + n * L::kPitch, q};
      CFG::run(ops, part, load_g);
    }
#pragma unroll
    for (int off = 16; off < kWave; off <<= 1) {
      float t[D2];
#pragma unroll
      for (int j = 0; j < D2; ++j) t[j] = lane_exchange(part[j], (lane ^ off) << 2);
#pragma unroll
      for (int j = 0; j < D2; ++j) part[j] += t[j];
    }
  }
  __syncthreads();  // every wavefront is done with the staged rows; reuse the front of LDS for the partial sums
  float* red = reinterpret_cast<float*>(smem);
  if (wave < n_blocks && q == 0) {
#pragma unroll
    for (int j = 0; j < D2; ++j) red[(wave * kUvsSamples + n) * D2 + j] = part[j];
  }
  __syncthreads();
  for (int i = threadIdx.x; i < kUvsSamples * D2; i += blockDim.x) {
    float s = 0.f;
    for (int w = 0; w < n_blocks; ++w) s += red[w * kUvsSamples * D2 + i];
    if (n0 + i / D2 < n_rows) gy[n0 * D2 + i] = s;
  }
}

// With channels on both operands ("uvw"), contracted channels x (n, DIN, 32), the other operand z (n, D2, L):
//   out[n, m, w] = sum_l sum_t coef_t * z[n, b_t, l] * sum_u x[n, a_t, u] * W[p_t, u, l, w]
// is the product above summed over l, with z[., ., l] for y and a weight per (path, l).  A workgroup owns 16 samples and a
// block of 32 produced channels; its four wavefronts take every fourth l each, keep all output rows in registers, and are
// added through LDS in a fixed order.  Mixing z and x first, as the fp32 route does, forms 1024 products per (path, row)
// and sample on the vector units; here they are the matrix cores', and the vector units see one multiply-add per
// coefficient and l.  What bounds it: vector and matrix instructions of two wavefronts per SIMD in about equal parts, and
// the weights from L2 (6 bytes an element and workgroup: 2.2 MB at 32 channels, lmax = 2).
// 32 x 32 -> 32, lmax = 2, 32768 samples: 925 -> 386 us, both gradients alike; 500 samples: 178 -> 58 us with packing; lmax = 1,
// 32768 samples 197 -> 103 us.  Error of the results against 64 bits 0.7e-7 to 1.2e-7, of the
// fp32 route 2.0e-7 to 15.8e-7.
template <class CFG, class TAB, int KIND>
__global__ void __launch_bounds__(256, 2) uvsw_kernel(const float* __restrict__ x, const float* __restrict__ z,
                                                      const __bf16* __restrict__ wp, const unsigned* __restrict__ asks_w,
                                                      float* __restrict__ out, int64_t n_rows, int cout, UvsWeight W) {
  extern __shared__ __align__(16) unsigned char smem[];
  constexpr int CIN = 32, DIN = CFG::DIN, DOUT = CFG::DOUT, D2 = CFG::D2;
  using T = UvsLds<DIN, CIN>;
  const int64_t n0 = (int64_t)blockIdx.x * kUvsSamples;
  const int L = W.matrices, n_mat = CFG::P * L;
  unsigned m = uvs_stage<DIN, CIN>(x, n0, n_rows, smem);
  unsigned* words = reinterpret_cast<unsigned*>(smem + T::kTile);
  float* zs = reinterpret_cast<float*>(words + 4);                // [l][row][sample]
  for (int i = threadIdx.x; i < n_mat; i += blockDim.x) m |= asks_w[i * (cout / 32) + blockIdx.y];
  for (int i = threadIdx.x; i < kUvsSamples * D2 * L; i += blockDim.x) {
    const int s = i / (D2 * L), rest = i - s * (D2 * L), b = rest / L, l = rest - b * L;
    const float v = z[min(n0 + s, n_rows - 1) * (D2 * L) + rest];
    zs[(l * D2 + b) * kUvsSamples + s] = v;
    m |= uvs_asks_y(v);
  }
  const bool plain = uvs_is_plain(uvs_all(m, words));

  const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x / kWave;
  const int n = lane & 15, q = lane >> 4;
  const int64_t row_n = min(n0 + n, n_rows - 1);
  const bool valid = n0 + n < n_rows;
  const int wblk = blockIdx.y;
  float* orow = out + (n0 + n) * DOUT * cout + wblk * 32 + 8 * q;
  auto store = [&](int row, const floatx4& o0, const floatx4& o1) __attribute__((always_inline)) {
    if (valid) {
      __builtin_nontemporal_store(o0, reinterpret_cast<floatx4*>(orow + row * cout));
      __builtin_nontemporal_store(o1, reinterpret_cast<floatx4*>(orow + row * cout + 4));
    }
  };
  if (plain) {
    UvsPlain<CIN> P;
    int t = 0;
    for (int row = 0; row < DOUT; ++row) {
      floatx4 o[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
      while (t < TAB::N && uvs_row_of<KIND>(TAB::terms(KIND)[t]) == row) {
        const int path = TAB::terms(KIND)[t].p;
        int end = t;
        uvs_segment<TAB, KIND>(end, row, path, [](const UvsTerm&) {});
        for (int l = 0; l < L && (row & 3) == wave; ++l) {
          P.clear();
          int i = t;
          uvs_segment<TAB, KIND>(i, row, path, [&](const UvsTerm& e) __attribute__((always_inline)) {
            P.mix(x + (row_n * DIN + uvs_in_of<KIND>(e)) * CIN, e.c * z[(row_n * D2 + uvs_other_of<KIND>(e)) * L + l], q);
          });
          P.multiply(W, path * L + l, wblk, n, q, o);
        }
        t = end;
      }
      if ((row & 3) == wave) store(row, o[0], o[1]);
    }
    return;
  }
  floatx4 acc[DOUT][2];
#pragma unroll
  for (int m = 0; m < DOUT; ++m) acc[m][0] = acc[m][1] = floatx4{0.f, 0.f, 0.f, 0.f};
  const int64_t matrix = (int64_t)cout * CIN * 3;
  for (int l = wave; l < L; l += 4) {
    float zv[D2];
#pragma unroll
    for (int j = 0; j < D2; ++j) zv[j] = zs[(l * D2 + j) * kUvsSamples + n];
    const UvsOps<DIN, CIN> ops{wp + l * matrix + (int64_t)wblk * (6 * 512) + lane * 8, L * matrix,
                          smem + n * T::kPitch, q};
    CFG::run(ops, zv, [&](int row, const floatx4& o0, const floatx4& o1) __attribute__((always_inline)) {
      acc[row][0] += o0;
      acc[row][1] += o1;
    });
  }
  // wavefronts 2 and 3 to 0 and 1, then 1 to 0
  floatx4* red = reinterpret_cast<floatx4*>(smem);
#pragma unroll
  for (int half = 2; half >= 1; half >>= 1) {
    __syncthreads();
    if (wave >= half && wave < 2 * half) {
#pragma unroll
      for (int m = 0; m < DOUT; ++m)
#pragma unroll
        for (int t = 0; t < 2; ++t) red[(((wave - half) * DOUT + m) * 2 + t) * kWave + lane] = acc[m][t];
    }
    __syncthreads();
    if (wave < half) {
#pragma unroll
      for (int m = 0; m < DOUT; ++m)
#pragma unroll
        for (int t = 0; t < 2; ++t) acc[m][t] += red[((wave * DOUT + m) * 2 + t) * kWave + lane];
    }
  }
  if (wave == 0) {
#pragma unroll
    for (int m = 0; m < DOUT; ++m) store(m, acc[m][0], acc[m][1]);
  }
}

// ---- host side ------------------------------------------------------------------------------------------------
using UvsFn = void (*)(const float*, const float*, const __bf16*, const unsigned*, float*, int64_t, int, UvsWeight);
struct UvsEntry {
  int cfg;                 // index of the table among the compiled ones (cgtp_uv_find)
  int p;                   // paths
  int64_t lds[3][3];       // bytes, as fn
  int64_t lds_w[3];        // of the staged rows, as fn_w
  UvsFn fn[3][3];          // [forward, gradient of x, gradient of y][32, 64, 128 contracted channels]
  UvsFn fn_w[3];           // channels on both operands, 32 contracted; null where the rows do not fit the registers
  int rows_w[3][2];        // rows of the operand that is not contracted, and of the produced one
};

// wavefronts per SIMD the registers are kept to: two, except at 128 contracted channels, where the two weight fragments in
// flight alone take 192 registers
constexpr int uvs_waves(int cin) { return cin < 128 ? 2 : 1; }

template <class CFG, class TAB, int KIND>
constexpr UvsFn uvsw_fn() {
  if constexpr (CFG::DOUT <= 9) return uvsw_kernel<CFG, TAB, KIND>;
  else return nullptr;
}

template <class D0, class D1, class GY, class DW, class TAB>
static UvsEntry make_uvs_entry(int cfg) {
  UvsEntry e;
  e.cfg = cfg;
  e.p = D0::P;
#define CGTP_UVS_CIN(i, CIN)                               \
  e.fn[0][i] = uvs_kernel<D0, TAB, 0, CIN, uvs_waves(CIN)>;   \
  e.fn[1][i] = uvs_kernel<D1, TAB, 1, CIN, uvs_waves(CIN)>;   \
  e.fn[2][i] = uvs_gy_kernel<GY, TAB, CIN, uvs_waves(CIN)>;   \
  e.lds[0][i] = UvsLds<D0::DIN, CIN>::kTile + 16;             \
  e.lds[1][i] = UvsLds<D1::DIN, CIN>::kTile + 16;             \
  e.lds[2][i] = UvsLds<GY::DIN, CIN>::kTile + 16;
  CGTP_UVS_CIN(0, 32)
  CGTP_UVS_CIN(1, 64)
  CGTP_UVS_CIN(2, 128)
#undef CGTP_UVS_CIN
  e.lds_w[0] = UvsLds<D0::DIN, 32>::kTile; e.lds_w[1] = UvsLds<D1::DIN, 32>::kTile; e.lds_w[2] = UvsLds<DW::DIN, 32>::kTile;
  e.fn_w[0] = uvsw_fn<D0, TAB, 0>(); e.fn_w[1] = uvsw_fn<D1, TAB, 1>(); e.fn_w[2] = uvsw_fn<DW, TAB, 2>();
  const int rows[3][2] = {{D0::D2, D0::DOUT}, {D1::D2, D1::DOUT}, {DW::D2, DW::DOUT}};
  for (int k = 0; k < 6; ++k) e.rows_w[k / 2][k % 2] = rows[k / 2][k % 2];
  return e;
}

static const UvsEntry* uvs_entry(int cfg) {
#define CGTP_X(INDEX, D0, D1, GY, DW, TAB) make_uvs_entry<D0, D1, GY, DW, TAB>(INDEX),
  static const UvsEntry table[] = {CGTP_FOREACH_UVS_CONFIG(CGTP_X)};
#undef CGTP_X
  for (const UvsEntry& e : table)
    if (e.cfg == cfg) return &e;
  return nullptr;
}

// kind 0: forward, 1: gradient of x, 2: gradient of y
static int uvs_check(int cfg, int kind, const void* x, const void* y, const void* packed, const void* w, const void* out,
                     int64_t n_rows, int cin, int cout, const UvsEntry** entry, int* ci, int64_t* lds) {
  const UvsEntry* e = uvs_entry(cfg);
  if (!e) return CGTP_ERR_CONFIG;
  if (kind < 0 || kind > 2) return CGTP_ERR_SHAPE;
  if (!x || !y || !packed || !w || !out) return CGTP_ERR_NULL;
  if (n_rows < 0 || cout <= 0 || cout % 32 || (kind == 2 && cout > 128)) return CGTP_ERR_SHAPE;
  *ci = cin == 32 ? 0 : cin == 64 ? 1 : cin == 128 ? 2 : -1;
  if (*ci < 0) return CGTP_ERR_SHAPE;
  // One block of produced channels keeps one wavefront in four busy, at 128 contracted channels the only one of its compute
  // unit: 128 -> 32, 32768 samples, lmax 1, 2, 3: 62, 213, 612 us where fp32 matrix instructions take 45, 158, 515 (128 -> 64:
  // 67, 219, 645 for 70, 293, 716; 64 -> 32, two workgroups per compute unit: 22, 58, 170 for 29, 93, 208).
  if (cin == 128 && cout == 32) return CGTP_ERR_SHAPE;
  if (((uintptr_t)x | (uintptr_t)packed | (uintptr_t)(kind == 2 ? y : out)) & 15u) return CGTP_ERR_ALIGN;
  *lds = e->lds[kind][*ci];
  if (*lds > kLdsBytes) return CGTP_ERR_LDS;
  if ((n_rows + kUvsSamples - 1) / kUvsSamples >= (int64_t)1 << 31) return CGTP_ERR_SHAPE;
  *entry = e;
  return CGTP_OK;
}

static int uvs_pack(const UvsWeight& W, void* packed, int64_t matrices, int cin, int cout, hipStream_t stream) {
  hipLaunchKernelGGL(uvs_pack_kernel, dim3((unsigned)matrices, (unsigned)(cout / 32)), dim3(256), 0, stream, W,
                     (__bf16*)packed, (unsigned*)((__bf16*)packed + matrices * cin * cout * 3), cin, cout);
  return hipGetLastError() == hipSuccess ? CGTP_OK : CGTP_ERR_LAUNCH;
}

// The weight (P, U, V, W) as kind 0 (contracts U, produces W, runs over V), 1 (W, U, V) or 2 (W, V, U) reads it.
static UvsWeight uvsw_weight(const float* w, int kind, int u, int v, int c) {
  const int64_t sp = (int64_t)u * v * c, su = (int64_t)v * c, sv = c;
  if (kind == 0) return {w, sp, su, 1, sv, v};
  if (kind == 1) return {w, sp, 1, su, sv, v};
  return {w, sp, 1, sv, su, u};
}

static int uvsw_check(int cfg, int kind, const void* x, const void* z, const void* packed, const void* w, const void* out,
                      int64_t n_rows, int u, int v, int c, const UvsEntry** entry, int64_t* lds) {
  const UvsEntry* e = uvs_entry(cfg);
  if (!e) return CGTP_ERR_CONFIG;
  if (kind < 0 || kind > 2 || !e->fn_w[kind]) return CGTP_ERR_SHAPE;
  if (!x || !z || !packed || !w || !out) return CGTP_ERR_NULL;
  const int cin = kind == 0 ? u : c, cout = kind == 0 ? c : kind == 1 ? u : v, L = kind == 2 ? u : v;
  if (n_rows < 0 || cin != 32 || cout <= 0 || cout % 32 || L <= 0) return CGTP_ERR_SHAPE;
  if (((uintptr_t)x | (uintptr_t)packed | (uintptr_t)out) & 15u) return CGTP_ERR_ALIGN;
  const int d2 = e->rows_w[kind][0], dout = e->rows_w[kind][1];
  const int64_t staged = e->lds_w[kind] + 16 + (int64_t)kUvsSamples * d2 * L * 4;
  const int64_t sums = (int64_t)2 * dout * 2 * kWave * 16;
  *lds = staged > sums ? staged : sums;
  if (2 * *lds > kLdsBytes) return CGTP_ERR_LDS;                  // two workgroups per compute unit, as the registers allow
  if ((n_rows + kUvsSamples - 1) / kUvsSamples >= (int64_t)1 << 31) return CGTP_ERR_SHAPE;
  *entry = e;
  return CGTP_OK;
}

}  // namespace cgtp

using namespace cgtp;

extern "C" {

int64_t cgtp_uvs_packed_bytes(int32_t n_paths, int32_t cin, int32_t cout) {
  if (n_paths <= 0 || cin <= 0 || cout <= 0 || cin % 32 || cout % 32) return 0;
  return (int64_t)n_paths * cin * cout * 6 + ((int64_t)n_paths * (cout / 32) * 4 + 15) / 16 * 16;
}

int cgtp_uvs_pack_weights(const float* w, void* packed, int32_t n_paths, int32_t cin, int32_t cout, int32_t transposed,
                          void* stream) {
  if (!w || !packed) return CGTP_ERR_NULL;
  if (n_paths <= 0 || cin <= 0 || cout <= 0 || cin % 32 || cout % 32) return CGTP_ERR_SHAPE;
  if ((uintptr_t)packed & 15u) return CGTP_ERR_ALIGN;
  const int64_t sp = (int64_t)cin * cout;
  const UvsWeight W = {w, sp, transposed ? 1 : (int64_t)cout, transposed ? (int64_t)cin : 1, 0, 1};
  return uvs_pack(W, packed, n_paths, cin, cout, (hipStream_t)stream);
}

int cgtp_uvs_validate(int cfg, int kind, const void* x, const void* y, const void* packed, const void* w, const void* out,
                      int64_t n_rows, int32_t cin, int32_t cout) {
  const UvsEntry* e = nullptr;
  int ci = 0;
  int64_t lds = 0;
  return uvs_check(cfg, kind, x, y, packed, w, out, n_rows, cin, cout, &e, &ci, &lds);
}

int cgtp_uvs_apply(int cfg, int kind, const void* x, const void* y, const void* packed, const void* w, void* out,
                   int64_t n_rows, int32_t cin, int32_t cout, void* stream) {
  const UvsEntry* e = nullptr;
  int ci = 0;
  int64_t lds = 0;
  const int st = uvs_check(cfg, kind, x, y, packed, w, out, n_rows, cin, cout, &e, &ci, &lds);
  if (st != CGTP_OK || n_rows == 0) return st;
  const UvsFn fn = e->fn[kind][ci];
  if (hipFuncSetAttribute((const void*)fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds) != hipSuccess)
    return CGTP_ERR_LDS;
  const int64_t sp = (int64_t)cin * cout;
  const UvsWeight W = {(const float*)w, sp, kind == 1 ? 1 : (int64_t)cout, kind == 1 ? (int64_t)cin : 1, 0, 1};
  hipLaunchKernelGGL(fn, dim3((unsigned)((n_rows + kUvsSamples - 1) / kUvsSamples), (unsigned)(kind == 2 ? 1 : (cout + 127) / 128)),
                     dim3(256), (size_t)lds, (hipStream_t)stream, (const float*)x, (const float*)y, (const __bf16*)packed,
                     (const unsigned*)((const __bf16*)packed + e->p * sp * 3), (float*)out, n_rows, (int)cout, W);
  return hipGetLastError() == hipSuccess ? CGTP_OK : CGTP_ERR_LAUNCH;
}

int64_t cgtp_uvsw_packed_bytes(int32_t n_paths, int32_t u, int32_t v, int32_t w) {
  if (n_paths <= 0 || u <= 0 || v <= 0 || w <= 0) return 0;
  // any kind: the matrices of a path run over one of the operands' channels, the blocks of 32 over another's
  const int64_t most = std::max({(int64_t)v * w, (int64_t)v * u, (int64_t)u * v}) / 32;
  return (int64_t)n_paths * u * v * w * 6 + (n_paths * most * 4 + 15) / 16 * 16;
}

int cgtp_uvsw_validate(int cfg, int kind, const void* x, const void* z, const void* packed, const void* w, const void* out,
                       int64_t n_rows, int32_t u, int32_t v, int32_t c) {
  const UvsEntry* e = nullptr;
  int64_t lds = 0;
  return uvsw_check(cfg, kind, x, z, packed, w, out, n_rows, u, v, c, &e, &lds);
}

int cgtp_uvsw_apply(int cfg, int kind, const void* x, const void* z, void* packed, const void* w, void* out, int64_t n_rows,
                    int32_t u, int32_t v, int32_t c, void* stream) {
  const UvsEntry* e = nullptr;
  int64_t lds = 0;
  int st = uvsw_check(cfg, kind, x, z, packed, w, out, n_rows, u, v, c, &e, &lds);
  if (st != CGTP_OK || n_rows == 0) return st;
  const int cin = kind == 0 ? u : c, cout = kind == 0 ? c : kind == 1 ? u : v;
  const UvsWeight W = uvsw_weight((const float*)w, kind, u, v, c);
  const int64_t matrices = (int64_t)e->p * W.matrices;
  st = uvs_pack(W, packed, matrices, cin, cout, (hipStream_t)stream);
  if (st != CGTP_OK) return st;
  const UvsFn fn = e->fn_w[kind];
  if (hipFuncSetAttribute((const void*)fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds) != hipSuccess)
    return CGTP_ERR_LDS;
  hipLaunchKernelGGL(fn, dim3((unsigned)((n_rows + kUvsSamples - 1) / kUvsSamples), (unsigned)(cout / 32)), dim3(256),
                     (size_t)lds, (hipStream_t)stream, (const float*)x, (const float*)z, (const __bf16*)packed,
                     (const unsigned*)((const __bf16*)packed + matrices * cin * cout * 3), (float*)out, n_rows, cout, W);
  return hipGetLastError() == hipSuccess ? CGTP_OK : CGTP_ERR_LAUNCH;
}

}  // extern "C"
