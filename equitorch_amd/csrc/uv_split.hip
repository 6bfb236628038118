// Fully connected ("uv") Clebsch-Gordan tensor product in single precision on the half-precision matrix cores:
//
//   out[n, m, w] = sum_t coef_t * y[n, b_t] * sum_u x[n, a_t, u] * W[p_t, u, w]
//
// for the compiled tables; forward, the gradient of x (the same with the rows' roles exchanged and the weight read
// transposed) and the gradient of y.  The order is that of uv_mfma.hip: per weight path and input row two accumulator
// tiles Z = x W, then the coefficients as fp32 multiply-adds between accumulator tiles.
//
// Every fp32 operand a is carried as two halves: with a scaled by a power of two (the largest element of its row of x,
// or of its path of W, lies in [2^13, 2^14)), h = half(a), l = half(a - h).  h + l is a to 2^-24 of it — as near as the
// rounding of a itself — for elements down to 2^-16 of the largest, and to 2^-39 of the largest below.  Z is h h' + h l' +
// l h' (the product l l' is below 2^-24 of the element products), each product exact in fp32 and summed in fp32, 32
// of them to a rounding; the factor that undoes the scales joins the coefficient.  Relative error of Z against 64 bits at
// 128 channels: 0.8e-7, of a chain of fp32 multiply-adds 2.0e-7; of the results over the range of sizes:
// 1.2e-7 to 1.7e-7 where fp32 matrix instructions give 1.6e-7 to 5.1e-7 (lmax 1 to 3, 32 to 128 channels).
// The same contraction in fp32 matrix instructions takes 256 cycles per 16 x 16 tile and 32 channels, this one 48.
//
// What bounds it: a workgroup of four wavefronts owns 16 samples, whose rows (4 bytes an element, both halves) fill most
// of the LDS at 128 channels and lmax = 3, and every workgroup reads all the weights from L2, 1.5 MB there.
// One wavefront per SIMD at 128 channels: matrix pipeline 34 % busy, LDS reads 35 % (bank conflicts another 16 %), vector
// instructions 30 %.  128 -> 128 channels, lmax = 3, 32768 samples: forward 1312 -> 426 us, gradient of x 1314 -> 410, of y
// 1868 -> 422 (fp32 matrix instructions, coupling first, against this); 64 -> 64, lmax = 2: 138 / 134 / 188 -> 62 / 63 / 62;
// 512 samples of 128 channels, lmax = 3: 161 / 161 / 228 -> 51 / 52 / 53.
//
// Rows of x or paths of W that hold an infinity, a NaN or a magnitude past 2^64 are not split, nor is anything multiplied
// by a y that is not finite: the workgroup then forms its samples' results with fp32 matrix instructions, term by term
// of the table and the coupling first (uvs_plain_tile), so that such values reach exactly the results they couple to.
#include "uv_common.h"

// accumulator-tile updates are written as o += s * z; let them contract to FMAs in this file
#pragma clang fp contract(fast)

namespace cgtp {

typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x4 __attribute__((ext_vector_type(4)));

struct UvsTerm {
  float c;
  unsigned char o, a, b, p;      // rows of out, x and y, path
};

#include "generated/uv_split_configs.inc"

constexpr int kUvsSamples = 16;
constexpr unsigned kUvsMaxExp = 127 + 64;      // biased exponent from which an operand is not split

// Power of two that takes a value with biased exponent e (below kUvsMaxExp; 0 counts as the smallest normal range handled)
// into [2^13, 2^14), and its inverse.
__device__ __forceinline__ unsigned uvs_exp(unsigned abs_bits) { return max(abs_bits >> 23, 14u); }
__device__ __forceinline__ float uvs_scale(unsigned e) { return __builtin_bit_cast(float, (267u - e) << 23); }
__device__ __forceinline__ float uvs_unscale(unsigned e) { return __builtin_bit_cast(float, (e - 13u) << 23); }

// The weight as the caller holds it.  With channels on both operands a path has one matrix per channel l of the operand
// that is not contracted; `matrices` is their number (else 1), and a "path" of the packed weight is a (path, l).
struct UvsWeight {
  const float* w;
  int64_t stride_p, stride_k, stride_c, stride_l;
  int matrices;
  __device__ __forceinline__ const float* of(int i) const { return w + (i / matrices) * stride_p + (i % matrices) * stride_l; }
};

// A workgroup per path and block of 32 output channels: the path's largest magnitude (every workgroup of a path reads all of
// it: 64 KB at 128 channels, from L2), then both halves of its block in fragment order.  Per path and block 2 (half) x 2
// (tile) x K / 32 chunks of 1 KB, holding the 16 bytes of every lane; row r of tile t is output channel
// 8 (r / 4) + 4 t + r % 4 of the block.  inv[p]: what undoes the scale, a NaN for a path that is not split.
__global__ void __launch_bounds__(256) uvs_pack_kernel(UvsWeight W, _Float16* __restrict__ packed, float* __restrict__ inv, int K,
                                                       int cout) {
  __shared__ unsigned waves_max[4];
  const int p = blockIdx.x, blk = blockIdx.y, ks = K / 32;
  const float* wp = W.of(p);
  const int64_t stride_k = W.stride_k, stride_c = W.stride_c;
  unsigned m = 0;
  // lanes along the axis of consecutive elements; K and cout are multiples of 32
  const bool k_inner = stride_k == 1;
  const int inner = k_inner ? K : cout;
  const int64_t si = k_inner ? stride_k : stride_c, so = k_inner ? stride_c : stride_k;
#pragma unroll 4
  for (int i = threadIdx.x; i < K * cout; i += 256) {
    const float v = wp[(i / inner) * so + (i % inner) * si];
    m = max(m, __builtin_bit_cast(unsigned, v) & 0x7fffffffu);
  }
  for (int off = 1; off < kWave; off <<= 1) m = max(m, (unsigned)__shfl_xor((int)m, off, kWave));
  if ((threadIdx.x & (kWave - 1)) == 0) waves_max[threadIdx.x / kWave] = m;
  __syncthreads();
  for (int i = 0; i < 4; ++i) m = max(m, waves_max[i]);
  const bool plain = (m >> 23) >= kUvsMaxExp;
  const unsigned e = plain ? 127u : uvs_exp(m);
  if (threadIdx.x == 0 && blk == 0) inv[p] = plain ? __builtin_nanf("") : uvs_unscale(e);
  const float s = uvs_scale(e);
  for (int i = threadIdx.x; i < K * 4; i += 256) {             // fragments of eight k
    const int lane = i & 63, c = i >> 6, k = c % ks, t = c / ks;
    const int r = lane & 15, q = lane >> 4;
    const int row = blk * 32 + 8 * (r >> 2) + 4 * t + (r & 3), col = k * 32 + 8 * q;
    f16x8 h, l;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const float v = wp[(col + j) * stride_k + row * stride_c] * s;
      h[j] = (_Float16)v;
      l[j] = (_Float16)(v - (float)h[j]);
    }
    _Float16* dst = packed + (int64_t)p * K * cout * 2 + ((int64_t)(blk * 4 + t) * ks + k) * 512 + lane * 8;
    *reinterpret_cast<f16x8*>(dst) = h;
    *reinterpret_cast<f16x8*>(dst + (int64_t)2 * ks * 512) = l;
  }
}

// LDS: per sample DIN rows of (CIN high halves, CIN low halves) and 16 bytes of padding; then what undoes the scale of every
// row, [sample][DIN]; then that of every path, and four words (uvs_any).
template <int DIN, int CIN>
struct UvsLds {
  static constexpr int kRow = CIN * 4, kPitch = DIN * kRow + 16, kTile = kUvsSamples * kPitch;
};

// Stages the 16 samples' rows; true if none of this thread's rows has to be left unsplit.
template <int DIN, int CIN>
__device__ __forceinline__ bool uvs_stage(const float* __restrict__ x, int64_t n0, int64_t n_rows, unsigned char* smem) {
  using L = UvsLds<DIN, CIN>;
  constexpr int PIECES = CIN / 4, TOTAL = kUvsSamples * DIN * PIECES;
  float* inv = reinterpret_cast<float*>(smem + L::kTile);
  bool ok = true;
  constexpr int UNROLL = 8;
  static_assert(TOTAL % kWave == 0, "whole wavefronts: the lanes of a row exchange their maxima");
  for (int base = 0; base < TOTAL; base += 256 * UNROLL) {
    f32x4 v[UNROLL];
#pragma unroll
    for (int u = 0; u < UNROLL; ++u) {
      const int i = base + u * 256 + (int)threadIdx.x;
      if (i < TOTAL) {
        const int s = i / (DIN * PIECES), c = i % (DIN * PIECES);
        v[u] = *reinterpret_cast<const f32x4*>(x + min(n0 + s, n_rows - 1) * (DIN * CIN) + c * 4);
      }
    }
#pragma unroll
    for (int u = 0; u < UNROLL; ++u) {
      const int i = base + u * 256 + (int)threadIdx.x;
      if (i < TOTAL) {
        const int s = i / (DIN * PIECES), c = i % (DIN * PIECES), row = c / PIECES, piece = c % PIECES;
        unsigned m = 0;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const float a = v[u][j];      // a bit cast of the vector's element itself would read element 0
          m = max(m, __builtin_bit_cast(unsigned, a) & 0x7fffffffu);
        }
#pragma unroll
        for (int off = 1; off < PIECES; off <<= 1) m = max(m, (unsigned)__shfl_xor((int)m, off, kWave));
        ok = ok && (m >> 23) < kUvsMaxExp;
        const unsigned e = min(uvs_exp(m), kUvsMaxExp);
        const float sc = uvs_scale(e);
        f16x4 h, l;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const float a = v[u][j] * sc;
          h[j] = (_Float16)a;
          l[j] = (_Float16)(a - (float)h[j]);
        }
        unsigned char* dst = smem + s * L::kPitch + row * L::kRow + piece * 8;
        *reinterpret_cast<f16x4*>(dst) = h;
        *reinterpret_cast<f16x4*>(dst + CIN * 2) = l;
        if (piece == 0) inv[s * DIN + row] = uvs_unscale(e);
      }
    }
  }
  return ok;
}

// Barrier; whether `v` holds in any thread of the workgroup's four wavefronts (`words`: four words of LDS).
__device__ __forceinline__ bool uvs_any(bool v, int* words) {
  const bool any = __any(v);
  if ((threadIdx.x & (kWave - 1)) == 0) words[threadIdx.x / kWave] = any;
  __syncthreads();
  return words[0] | words[1] | words[2] | words[3];
}

template <int DIN, int CIN>
struct UvsOps {
  static constexpr int KS = CIN / 32;
  struct A { f16x8 f[2][2][KS]; };          // [half][tile][step]
  struct B { f16x8 f[2][KS]; };
  const _Float16* wp;                       // this lane's fragments of path 0
  int64_t path_stride;
  const unsigned char* xs;                  // this lane's base in its sample's rows
  const float* inv_x;                       // its sample's rows
  const float* inv_w;
  int inv_stride = 1;                       // between the paths of inv_w
  __device__ __forceinline__ void load_a(int p, A& a) const {
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int k = 0; k < KS; ++k)
          a.f[h][t][k] = *reinterpret_cast<const f16x8*>(wp + p * path_stride + ((h * 2 + t) * KS + k) * 512);
  }
  __device__ __forceinline__ void load_b(int row, B& b) const {
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int k = 0; k < KS; ++k)
        b.f[h][k] = *reinterpret_cast<const f16x8*>(xs + row * (CIN * 4) + h * (CIN * 2) + k * 64);
  }
  // the small products first
  __device__ __forceinline__ void chain(const A& a, const B& b, floatx4& z0, floatx4& z1) const {
    z0 = floatx4{0.f, 0.f, 0.f, 0.f};
    z1 = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int part = 0; part < 3; ++part) {
      const int ha = part == 0 ? 1 : 0, hb = part == 1 ? 1 : 0;
#pragma unroll
      for (int k = 0; k < KS; ++k) {
        z0 = __builtin_amdgcn_mfma_f32_16x16x32_f16(a.f[ha][0][k], b.f[hb][k], z0, 0, 0, 0);
        z1 = __builtin_amdgcn_mfma_f32_16x16x32_f16(a.f[ha][1][k], b.f[hb][k], z1, 0, 0, 0);
      }
    }
  }
  __device__ __forceinline__ float scale(int p, int row) const { return inv_x[row] * inv_w[p * inv_stride]; }
};

// (s x) W of one path and row for the two tiles of block `blk`, from memory, in fp32 matrix instructions.
__device__ __forceinline__ void uvs_plain_tile(const UvsWeight& W, int p, int blk, const float* __restrict__ xrow, float s,
                                               int K, int r, int q, floatx4 (&z)[2]) {
  z[0] = z[1] = floatx4{0.f, 0.f, 0.f, 0.f};
  const float* wb = W.of(p) + (blk * 32 + 8 * (r >> 2) + (r & 3)) * W.stride_c;
  for (int k = q; k < K; k += 4) {
    const float b = s * xrow[k];
#pragma unroll
    for (int t = 0; t < 2; ++t)
      z[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(wb[k * W.stride_k + 4 * t * W.stride_c], b, z[t], 0, 0, 0);
  }
}

// DIR 0: forward, 1: gradient of x (terms with the rows of out and x exchanged).
template <class CFG, class TAB, int DIR, int CIN, int WAVES>
__global__ void __launch_bounds__(256, WAVES) uvs_kernel(const float* __restrict__ x, const float* __restrict__ y,
                                                         const _Float16* __restrict__ wp, const float* __restrict__ inv_w,
                                                         float* __restrict__ out, int64_t n_rows, int cout, UvsWeight W) {
  extern __shared__ __align__(16) unsigned char smem[];
  constexpr int DIN = CFG::DIN, DOUT = CFG::DOUT, D2 = CFG::D2;
  using L = UvsLds<DIN, CIN>;
  const int64_t n0 = (int64_t)blockIdx.x * kUvsSamples;
  bool ok = uvs_stage<DIN, CIN>(x, n0, n_rows, smem);
  float* inv_x = reinterpret_cast<float*>(smem + L::kTile);
  float* inv_p = inv_x + kUvsSamples * DIN;
  for (int i = threadIdx.x; i < CFG::P; i += blockDim.x) {
    const float v = inv_w[i];
    inv_p[i] = v;
    ok = ok && v == v;
  }
  for (int i = threadIdx.x; i < kUvsSamples * D2; i += blockDim.x) {
    const float v = y[min(n0 + i / D2, n_rows - 1) * D2 + i % D2];
    ok = ok && v - v == 0.f;
  }
  const bool plain = uvs_any(!ok, reinterpret_cast<int*>(inv_p + CFG::P));

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
    for (int m = 0; m < DOUT; ++m) {
      floatx4 o[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
      for (int t = 0; t < TAB::N; ++t) {
        const UvsTerm e = TAB::terms()[t];
        if ((DIR == 0 ? e.o : e.a) != m) continue;
        floatx4 z[2];
        uvs_plain_tile(W, e.p, wblk, x + (row_n * DIN + (DIR == 0 ? e.a : e.o)) * CIN, e.c * y[row_n * D2 + e.b], CIN, n, q, z);
        o[0] += z[0];
        o[1] += z[1];
      }
      store(m, o[0], o[1]);
    }
    return;
  }
  float yv[D2];
#pragma unroll
  for (int j = 0; j < D2; ++j) yv[j] = y[row_n * D2 + j];
  const UvsOps<DIN, CIN> ops{wp + (int64_t)wblk * (4 * (CIN / 32) * 512) + lane * 8, (int64_t)cout * CIN * 2,
                             smem + n * L::kPitch + q * 16, inv_x + n * DIN, inv_p};
  CFG::run(ops, yv, store);
}

// gy[n, b] = sum_t coef_t * sum_w g[n, m_t, w] * Z[p_t, a_t][w, n]: the forward's tiles; the lane sums over its channels, the
// four lanes of a sample and the wavefronts (channel blocks, cout <= 128) are then added in a fixed order.
template <class CFG, class TAB, int CIN, int WAVES>
__global__ void __launch_bounds__(256, WAVES) uvs_gy_kernel(const float* __restrict__ x, const float* __restrict__ g,
                                                            const _Float16* __restrict__ wp, const float* __restrict__ inv_w,
                                                            float* __restrict__ gy, int64_t n_rows, int cout, UvsWeight W) {
  extern __shared__ __align__(16) unsigned char smem[];
  constexpr int DIN = CFG::DIN, DOUT = CFG::DOUT, D2 = CFG::D2;
  using L = UvsLds<DIN, CIN>;
  const int64_t n0 = (int64_t)blockIdx.x * kUvsSamples;
  bool ok = uvs_stage<DIN, CIN>(x, n0, n_rows, smem);
  float* inv_x = reinterpret_cast<float*>(smem + L::kTile);
  float* inv_p = inv_x + kUvsSamples * DIN;
  for (int i = threadIdx.x; i < CFG::P; i += blockDim.x) {
    const float v = inv_w[i];
    inv_p[i] = v;
    ok = ok && v == v;
  }
  const bool plain = uvs_any(!ok, reinterpret_cast<int*>(inv_p + CFG::P));

  const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x / kWave;
  const int n = lane & 15, q = lane >> 4, n_blk = cout / 32;
  const int64_t row_n = min(n0 + n, n_rows - 1);
  const float* grow = g + row_n * DOUT * cout + min(wave, n_blk - 1) * 32 + 8 * q;
  float part[D2];
#pragma unroll
  for (int j = 0; j < D2; ++j) part[j] = 0.f;
  auto load_g = [&](int row, floatx4& g0, floatx4& g1) __attribute__((always_inline)) {
    g0 = *reinterpret_cast<const floatx4*>(grow + row * cout);
    g1 = *reinterpret_cast<const floatx4*>(grow + row * cout + 4);
  };
  if (wave < n_blk) {
    if (plain) {
      for (int t = 0; t < TAB::N; ++t) {
        const UvsTerm e = TAB::terms()[t];
        floatx4 z[2], g0, g1;
        uvs_plain_tile(W, e.p, wave, x + (row_n * DIN + e.a) * CIN, 1.f, CIN, n, q, z);
        load_g(e.o, g0, g1);
        const float v = e.c * dot8(g0, g1, z[0], z[1]);
#pragma unroll
        for (int j = 0; j < D2; ++j)
          if (j == e.b) part[j] += v;
      }
    } else {
      const UvsOps<DIN, CIN> ops{wp + (int64_t)wave * (4 * (CIN / 32) * 512) + lane * 8, (int64_t)cout * CIN * 2,
                                 smem + n * L::kPitch + q * 16, inv_x + n * DIN, inv_p};
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
  if (wave < n_blk && q == 0) {
#pragma unroll
    for (int j = 0; j < D2; ++j) red[(wave * kUvsSamples + n) * D2 + j] = part[j];
  }
  __syncthreads();
  for (int i = threadIdx.x; i < kUvsSamples * D2; i += blockDim.x) {
    float s = 0.f;
    for (int w = 0; w < n_blk; ++w) s += red[w * kUvsSamples * D2 + i];
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
// the weights from L2 (4 bytes an element and workgroup: 1.4 MB at 32 channels, lmax = 2).
// 32 x 32 -> 32, lmax = 2, 32768 samples: 943 -> 268 us, both gradients alike; 500 samples: 179 -> 44 us with packing; lmax = 1,
// 32768 samples 205 -> 73 us.  Error of the results against 64 bits 1.1e-7 to 1.4e-7, of the fp32 route 2.0e-7 to 1.4e-6.
template <class CFG, class TAB, int KIND>
__global__ void __launch_bounds__(256, 2) uvsw_kernel(const float* __restrict__ x, const float* __restrict__ z,
                                                      const _Float16* __restrict__ wp, const float* __restrict__ inv_w,
                                                      float* __restrict__ out, int64_t n_rows, int cout, UvsWeight W) {
  extern __shared__ __align__(16) unsigned char smem[];
  constexpr int CIN = 32, DIN = CFG::DIN, DOUT = CFG::DOUT, D2 = CFG::D2;
  using T = UvsLds<DIN, CIN>;
  const int64_t n0 = (int64_t)blockIdx.x * kUvsSamples;
  const int L = W.matrices, n_mat = CFG::P * L;
  bool ok = uvs_stage<DIN, CIN>(x, n0, n_rows, smem);
  float* inv_x = reinterpret_cast<float*>(smem + T::kTile);
  float* inv_p = inv_x + kUvsSamples * DIN;
  int* words = reinterpret_cast<int*>(inv_p + n_mat);
  float* zs = reinterpret_cast<float*>(words + 4);                // [l][row][sample]
  for (int i = threadIdx.x; i < n_mat; i += blockDim.x) {
    const float v = inv_w[i];
    inv_p[i] = v;
    ok = ok && v == v;
  }
  for (int i = threadIdx.x; i < kUvsSamples * D2 * L; i += blockDim.x) {
    const int s = i / (D2 * L), rest = i - s * (D2 * L), b = rest / L, l = rest - b * L;
    const float v = z[min(n0 + s, n_rows - 1) * (D2 * L) + rest];
    zs[(l * D2 + b) * kUvsSamples + s] = v;
    ok = ok && v - v == 0.f;
  }
  const bool plain = uvs_any(!ok, words);

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
    for (int m = wave; m < DOUT; m += 4) {
      floatx4 o[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
      for (int t = 0; t < TAB::N; ++t) {
        const UvsTerm e = TAB::terms()[t];
        const int mt = KIND == 0 ? e.o : KIND == 1 ? e.a : e.b, at = KIND == 0 ? e.a : e.o, bt = KIND == 2 ? e.a : e.b;
        if (mt != m) continue;
        for (int l = 0; l < L; ++l) {
          floatx4 v[2];
          uvs_plain_tile(W, e.p * L + l, wblk, x + (row_n * DIN + at) * CIN, e.c * z[(row_n * D2 + bt) * L + l], CIN, n, q, v);
          o[0] += v[0];
          o[1] += v[1];
        }
      }
      store(m, o[0], o[1]);
    }
    return;
  }
  floatx4 acc[DOUT][2];
#pragma unroll
  for (int m = 0; m < DOUT; ++m) acc[m][0] = acc[m][1] = floatx4{0.f, 0.f, 0.f, 0.f};
  const int64_t matrix = (int64_t)cout * CIN * 2;
  for (int l = wave; l < L; l += 4) {
    float zv[D2];
#pragma unroll
    for (int j = 0; j < D2; ++j) zv[j] = zs[(l * D2 + j) * kUvsSamples + n];
    const UvsOps<DIN, CIN> ops{wp + l * matrix + (int64_t)wblk * (4 * 512) + lane * 8, L * matrix,
                               smem + n * T::kPitch + q * 16, inv_x + n * DIN, inv_p + l, L};
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
using UvsFn = void (*)(const float*, const float*, const _Float16*, const float*, float*, int64_t, int, UvsWeight);
struct UvsEntry {
  int cfg;                 // index of the table among the compiled ones (cgtp_uv_find)
  int din[2], p;           // rows of the contracted operand in the forward and in the gradient of x; paths
  UvsFn fn[3][3];          // [forward, gradient of x, gradient of y][32, 64, 128 contracted channels]
  UvsFn fn_w[3];           // channels on both operands, 32 contracted; null where the rows do not fit the registers
  int rows_w[3][3];        // rows of the contracted, the other and the produced operand
};

// wavefronts per SIMD the registers are kept to: two, except at 128 contracted channels, where the three weight fragments in
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
  e.din[0] = D0::DIN; e.din[1] = D1::DIN; e.p = D0::P;
#define CGTP_UVS_CIN(i, CIN)                               \
  e.fn[0][i] = uvs_kernel<D0, TAB, 0, CIN, uvs_waves(CIN)>;   \
  e.fn[1][i] = uvs_kernel<D1, TAB, 1, CIN, uvs_waves(CIN)>;   \
  e.fn[2][i] = uvs_gy_kernel<GY, TAB, CIN, uvs_waves(CIN)>;
  CGTP_UVS_CIN(0, 32)
  CGTP_UVS_CIN(1, 64)
  CGTP_UVS_CIN(2, 128)
#undef CGTP_UVS_CIN
  e.fn_w[0] = uvsw_fn<D0, TAB, 0>(); e.fn_w[1] = uvsw_fn<D1, TAB, 1>(); e.fn_w[2] = uvsw_fn<DW, TAB, 2>();
  const int rows[3][3] = {{D0::DIN, D0::D2, D0::DOUT}, {D1::DIN, D1::D2, D1::DOUT}, {DW::DIN, DW::D2, DW::DOUT}};
  for (int k = 0; k < 9; ++k) e.rows_w[k / 3][k % 3] = rows[k / 3][k % 3];
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
  if (((uintptr_t)x | (uintptr_t)packed | (uintptr_t)(kind == 2 ? y : out)) & 15u) return CGTP_ERR_ALIGN;
  const int din = e->din[kind == 1];
  *lds = (int64_t)kUvsSamples * (din * cin * 4 + 16) + kUvsSamples * din * 4 + e->p * 4 + 16;
  if (*lds > kLdsBytes) return CGTP_ERR_LDS;
  if ((n_rows + kUvsSamples - 1) / kUvsSamples >= (int64_t)1 << 31) return CGTP_ERR_SHAPE;
  *entry = e;
  return CGTP_OK;
}

static int uvs_pack(const UvsWeight& W, void* packed, int64_t matrices, int cin, int cout, hipStream_t stream) {
  hipLaunchKernelGGL(uvs_pack_kernel, dim3((unsigned)matrices, (unsigned)(cout / 32)), dim3(256), 0, stream, W,
                     (_Float16*)packed, (float*)((_Float16*)packed + matrices * cin * cout * 2), cin, cout);
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
  const int din = e->rows_w[kind][0], d2 = e->rows_w[kind][1], dout = e->rows_w[kind][2];
  const int64_t staged = (int64_t)kUvsSamples * (din * cin * 4 + 16) + kUvsSamples * din * 4 + (int64_t)e->p * L * 4 + 16 +
                         (int64_t)kUvsSamples * d2 * L * 4;
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
  return (int64_t)n_paths * cin * cout * 4 + ((int64_t)n_paths * 4 + 15) / 16 * 16;
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
                     dim3(256), (size_t)lds, (hipStream_t)stream, (const float*)x, (const float*)y, (const _Float16*)packed,
                     (const float*)((const _Float16*)packed + e->p * sp * 2), (float*)out, n_rows, (int)cout, W);
  return hipGetLastError() == hipSuccess ? CGTP_OK : CGTP_ERR_LAUNCH;
}

int64_t cgtp_uvsw_packed_bytes(int32_t n_paths, int32_t u, int32_t v, int32_t w) {
  if (n_paths <= 0 || u <= 0 || v <= 0 || w <= 0) return 0;
  // any kind: the matrices of a path run over one of the operands' channels
  return (int64_t)n_paths * u * v * w * 4 + ((int64_t)n_paths * (u > v ? u : v) * 4 + 15) / 16 * 16;
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
                     (size_t)lds, (hipStream_t)stream, (const float*)x, (const float*)z, (const _Float16*)packed,
                     (const float*)((const _Float16*)packed + matrices * cin * cout * 2), (float*)out, n_rows, cout, W);
  return hipGetLastError() == hipSuccess ? CGTP_OK : CGTP_ERR_LAUNCH;
}

}  // extern "C"
