// Channel-wise ("uvu") tensor product over an edge list for a small table handed over as data, on the matrix cores:
// gather at one end, product and segment sum at the other in one launch, fp32 in and accumulated.
//
//   out[v, M, c] = sum_{e in segment v} sum_{(p, M1)} A_e[M, (p, M1)] * (w[e, p, c] * x[other(e), M1, c])
//   A_e[M, (p, M1)] = sum_{M2} coef * y[e, M2]
//
// The coupling matrix A_e of an edge does not depend on the channel, so what interprets the table is done once per edge
// with lanes over its entries (a few instructions for 64 entries), and the rest is a dense contraction over (p, M1) of a
// 16-row matrix with 16 channels per tile: v_mfma_f32_16x16x4_f32, four rows of a path per step ("entry").  The
// sums of the open segment stay in registers over its edges and are stored once.
//
// The backward walks the list sorted by the other end (segments are rows of x) and needs three contractions per edge:
//   grad_x[M1, c] += sum_{(p, M)} A[M, (p, M1)] * (w[p, c] * g[M, c])               accumulators as above
//   grad_y[b]      = sum_t coef_t * G[(p_t, M_t), M1_t],  G[(p, M), M1] = sum_c (w[p, c] * g[M, c]) * x[M1, c]
//   grad_w[p, c]   = sum_M1 x[M1, c] * D[(p, M1), c],     D[(p, M1), c] = sum_M A[M, (p, M1)] * g[M, c]
// In the tiles of D the four rows a group of lanes holds belong to one path, so that its sum over M1 stays in the lane.
//
// What bounds it: LDS reads of the operands and the matrix pipeline (about 90 resp. 240 matrix instructions of 32 cycles
// per edge at 206 coefficients and 64 channels), two wavefronts per SIMD in the backward.  The walk over the table entry
// by entry that this replaces (uvu_tab.hip) ran four wavefronts per compute unit and a dozen instructions per entry:
// 65 536 edges, 4096 nodes, 206 coefficients, 64 channels: forward 411 -> 175 us, backward 1303 -> 453 us (matrix
// pipeline busy 48 resp. 39 % of the time).
//
// The dense form multiplies the zeros of A too, so an infinity or NaN in one operand row would reach rows that do not
// couple to it.  Every result a wavefront writes is checked; a wavefront that sees one not finite raises the flag of
// its range, and the entry-by-entry kernel, launched behind over the same ranges, leaves at once unless a flag of its
// ranges is set and writes those ranges anew.
#include "uvu_common.h"

namespace cgtp {

typedef float mx4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ void mx_sync() {     // LDS operations of a wavefront complete in order: only the compiler
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

constexpr int kMxMaxPaths = 32;
// Words of the device tables (built by the host, see cgtp_uvu_mx in cgtp.h), copied to LDS by every workgroup.
struct MxDev {
  const uint32_t* words;
  int n_words, n_rec, n_ent, n_rowtiles, n_rounds, lanes_log2, n_tiles, n_chunks;
  int D1, D2, DO, P;
  int32_t* flags;      // one word per range: 1 = a result was not finite
};
// Offsets of the parts of the table copy, in words.
struct MxParts {
  int rec, ent, row, term, tile, words;
  __host__ __device__ MxParts(int n_rec, int n_ent, int n_rowtiles, int n_rounds, int n_tiles) {
    rec = 0;                                // n_rec x (coef, coef, b | b << 8 | element of A << 16)
    ent = rec + 3 * n_rec;                  // n_ent x (path | first row << 8)
    row = ent + n_ent;                      // n_rowtiles x 16 x (path | row of grad_out << 8)
    term = row + 16 * n_rowtiles;           // n_rounds x 64 x (coef, element of G)
    tile = term + 128 * n_rounds;           // n_tiles x (first row | steps << 8, 4 x chunk)
    words = (tile + 5 * n_tiles + 3) & ~3;
  }
};
// Per-wavefront LDS, in floats.  Rows of NJ * 16 channels at a pitch of 4 more, so that 16 lanes reading 16 rows at the
// same channels hit distinct banks.
struct MxLayout {
  int pitch, a, w, r1, r2, y, floats;
  __host__ __device__ MxLayout(int nj, int D1, int D2, int DO, int P, int n_ent, int n_rowtiles, bool backward) {
    pitch = 16 * nj + 4;
    int at = 0;
    const auto take = [&](int n) { const int r = at; at += (n + 3) & ~3; return r; };
    a = take(64 * n_ent + 4);
    // the weight rows; in the backward this region holds G and then the weight gradient once they are consumed
    const int g_floats = 256 * n_rowtiles;
    w = take(backward && g_floats > P * pitch ? g_floats : P * pitch);
    r1 = take((backward ? DO + 3 : D1 + 3) * pitch);   // gathered rows; a step of four may reach three rows past the end
    r2 = take(backward ? (D1 + 1) * pitch : 0);        // rows of x, and a zero row
    y = take(D2);
    floats = at;
  }
};

template <int NJ>
struct MxVec {
  using type = typename VecOf<float, NJ>::type;
};

// Segment id, edge and gathered row of up to 64 positions of a range, one per lane.
struct MxIndex {
  int sid, edge, other;
  __device__ __forceinline__ void load(const UvuDev<float>& a, int64_t p, int64_t p1, int lane) {
    const int64_t q = p + lane < p1 ? p + lane : p1 - 1;
    sid = (int)a.seg_ids[q];
    edge = a.perm ? (int)a.perm[q] : (int)q;
    other = (int)a.gather[q];
  }
  static __device__ __forceinline__ int at(int v, int k) { return __builtin_amdgcn_readlane(v, k); }
};

// Rows of `rows` (NJ channels per lane, lane (r, g) takes rows 4 i + g) from memory into registers, and from there to LDS.
template <int NJ, int R>
__device__ __forceinline__ void mx_fetch(float (&v)[R][NJ], const float* __restrict__ src, int64_t C, int rows, int g,
                                         int c0, bool c_ok, bool stream) {
#pragma unroll
  for (int i = 0; i < R; ++i) {
    if (4 * i < rows) {
      const float* p = src + (int64_t)min(4 * i + g, rows - 1) * C + (c_ok ? c0 : 0);
      if (stream) load_vec_stream<float, NJ>(v[i], p);
      else load_vec<float, NJ>(v[i], p);
      if (!c_ok) {
#pragma unroll
        for (int j = 0; j < NJ; ++j) v[i][j] = 0.f;
      }
    }
  }
}
template <int NJ>
__device__ __forceinline__ void mx_put(float* p, const float (&v)[NJ]) {
  typename MxVec<NJ>::type t;
  float* e = reinterpret_cast<float*>(&t);
#pragma unroll
  for (int j = 0; j < NJ; ++j) e[j] = v[j];
  *reinterpret_cast<typename MxVec<NJ>::type*>(p) = t;
}
template <int NJ>
__device__ __forceinline__ void mx_get(float (&v)[NJ], const float* p) {
  const typename MxVec<NJ>::type t = *reinterpret_cast<const typename MxVec<NJ>::type*>(p);
  const float* e = reinterpret_cast<const float*>(&t);
#pragma unroll
  for (int j = 0; j < NJ; ++j) v[j] = e[j];
}
template <int NJ, int R>
__device__ __forceinline__ void mx_stage(float* dst, int pitch, const float (&v)[R][NJ], int rows, int g, int c0) {
#pragma unroll
  for (int i = 0; i < R; ++i)
    if (4 * i + g < rows) mx_put<NJ>(dst + (4 * i + g) * pitch + c0, v[i]);
}

// A_e: the element of every record, at most two terms each (the elements without a record stay zero).
__device__ __forceinline__ void mx_couple(const uint32_t* rec, int n_rec, const float* ys, float* A, int lane) {
  for (int t = lane; t < n_rec; t += kWave) {
    const float c0 = __builtin_bit_cast(float, rec[3 * t]), c1 = __builtin_bit_cast(float, rec[3 * t + 1]);
    const uint32_t k = rec[3 * t + 2];
    A[k >> 16] = fmaf(c1, ys[(k >> 8) & 255], c0 * ys[k & 255]);
  }
}

// acc[j] += A * (w * rows) over the entries.  The operands of the next entry are requested before this one is multiplied.
// An edge's products are summed by themselves before they join the segment's sum: a chain of 16 rounded additions to a
// sum over the edges so far would lose more than the entry-by-entry kernels do.
template <int NJ>
__device__ __forceinline__ void mx_contract(mx4 (&acc)[NJ], const uint32_t* ent, int n_ent, const float* A, const float* ws,
                                            const float* rows, int pitch, int lane) {
  const int g = lane >> 4, c0 = (lane & 15) * NJ;
  const float* wl = ws + c0;
  const float* rl = rows + g * pitch + c0;
  const uint32_t mine = ent[min(lane, n_ent - 1)];      // one entry word per lane (n_ent <= 64)
  float an = A[lane], wn[NJ], rn[NJ];
  const auto request = [&](int e) __attribute__((always_inline)) {
    const uint32_t k = (uint32_t)__builtin_amdgcn_readlane((int)mine, e);
    an = A[e * 64 + lane];
    mx_get<NJ>(wn, wl + (k & 255) * pitch);
    mx_get<NJ>(rn, rl + (k >> 8) * pitch);
  };
  mx4 z[NJ];
#pragma unroll
  for (int j = 0; j < NJ; ++j) z[j] = mx4{0.f, 0.f, 0.f, 0.f};
  request(0);
  for (int e = 0; e < n_ent; ++e) {
    const float a = an;
    float b[NJ];
#pragma unroll
    for (int j = 0; j < NJ; ++j) b[j] = wn[j] * rn[j];
    request(min(e + 1, n_ent - 1));
#pragma unroll
    for (int j = 0; j < NJ; ++j) z[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(a, b[j], z[j], 0, 0, 0);
  }
#pragma unroll
  for (int j = 0; j < NJ; ++j) acc[j] += z[j];
}

// The accumulators hold rows 4 g + i: store those below D as the row of the segment (or a partial row) and clear them.
// `bad` becomes not-a-number when a value is not finite.
template <int NJ>
__device__ __forceinline__ void mx_flush(mx4 (&acc)[NJ], float* dst, int D, int64_t C, int g, int c0, bool c_ok, float& bad) {
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    float v[NJ];
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
      v[j] = acc[j][i];
      bad = fmaf(v[j], 0.f, bad);
      acc[j][i] = 0.f;
    }
    if (4 * g + i < D && c_ok) store_vec<float, NJ>(dst + (4 * g + i) * C + c0, v);
  }
}

// One tile of G: sum over the channels of (w g)[row of this lane] x[.]; wr, gr: the lane's rows at channel 4 g.
template <int NJ>
__device__ __forceinline__ mx4 mx_channels(const float* wr, const float* gr, const float (&xt)[NJ][4]) {
  mx4 z = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int q = 0; q < NJ; ++q) {
    float wq[4], gq[4];
    mx_get<4>(wq, wr + 16 * q);
    mx_get<4>(gq, gr + 16 * q);
#pragma unroll
    for (int i = 0; i < 4; ++i) z = __builtin_amdgcn_mfma_f32_16x16x4f32(wq[i] * gq[i], xt[q][i], z, 0, 0, 0);
  }
  return z;
}
// grad_y of edge e from G in LDS; 1 << lanes_log2 lanes share a component.
__device__ __forceinline__ void mx_grad_y(const UvuDev<float>& a, const MxDev& t, const uint32_t* terms, const float* G, int64_t e,
                                          int lane, float& bad) {
  float sum = 0.f;
  for (int u = 0; u < t.n_rounds; ++u) {
    const uint32_t* term = terms + 2 * (u * kWave + lane);
    sum = fmaf(__builtin_bit_cast(float, term[0]), G[term[1]], sum);
  }
  for (int off = 1; off < (1 << t.lanes_log2); off <<= 1) sum += shfl_xor(sum, off);
  const int b = lane >> t.lanes_log2;
  bad = fmaf(sum, 0.f, bad);
  if ((lane & ((1 << t.lanes_log2) - 1)) == 0 && b < t.D2) a.gy[e * t.D2 + b] = sum;
}
// The weight gradient of edge e from its rows in LDS.
template <int NJ, int WR>
__device__ __forceinline__ void mx_store_grad_w(const UvuDev<float>& a, const MxDev& t, const float* rows, int pitch, int64_t e,
                                                int g, int c0, bool c_ok, float& bad) {
#pragma unroll
  for (int i = 0; i < WR; ++i) {
    if (4 * i + g < t.P) {
      float v[NJ];
      mx_get<NJ>(v, rows + (4 * i + g) * pitch + c0);
#pragma unroll
      for (int j = 0; j < NJ; ++j) bad = fmaf(v[j], 0.f, bad);
      if (c_ok) store_vec_stream<float, NJ>(a.gw + (e * t.P + 4 * i + g) * a.C + c0, v);
    }
  }
}

// First position past the range, and whether its first / last segment lie wholly inside it.
struct MxRange {
  int64_t p0, p1;
  bool first_complete, last_complete;
  __device__ __forceinline__ MxRange(const UvuDev<float>& a, int64_t range) {
    p0 = range * a.pos_per_wave;
    p1 = min(p0 + a.pos_per_wave, a.n_rows);
    first_complete = p0 == 0 || a.seg_ids[p0 - 1] != a.seg_ids[p0];
    last_complete = p1 == a.n_rows || a.seg_ids[p1 - 1] != a.seg_ids[p1];
  }
};

// NJ channels per lane (16 NJ >= C), WR: registers rows of weights (4 WR >= P).
template <int NJ, int WR>
__global__ void __launch_bounds__(256, 2) uvu_mx_fwd_kernel(const UvuDev<float> a, const MxDev t) {
  extern __shared__ __align__(16) float mx_lds[];
  const MxParts parts(t.n_rec, t.n_ent, 0, 0, 0);
  uint32_t* tab = reinterpret_cast<uint32_t*>(mx_lds);
  for (int i = threadIdx.x; i < t.n_words; i += blockDim.x) tab[i] = t.words[i];
  const MxLayout Y(NJ, t.D1, t.D2, t.DO, t.P, t.n_ent, 0, false);
  const int lane = threadIdx.x & (kWave - 1), g = lane >> 4, c0 = (lane & 15) * NJ;
  float* mine = mx_lds + parts.words + (threadIdx.x / kWave) * Y.floats;
  for (int i = lane; i < Y.floats; i += kWave) mine[i] = 0.f;
  __syncthreads();
  const int64_t range = seg_wave_index(a.n_waves);
  if (range < 0) return;
  const MxRange R(a, range);
  const int64_t C = a.C;
  const bool c_ok = c0 < a.C;
  mx4 acc[NJ];
#pragma unroll
  for (int j = 0; j < NJ; ++j) acc[j] = mx4{0.f, 0.f, 0.f, 0.f};
  MxIndex I;
  I.load(a, R.p0, R.p1, lane);
  float xv[4][NJ], wv[WR][NJ], yv, bad = 0.f;
  const auto fetch = [&](int edge, int other) __attribute__((always_inline)) {
    yv = a.y[(int64_t)edge * t.D2 + min(lane, t.D2 - 1)];
    mx_fetch<NJ, 4>(xv, a.x + (int64_t)other * t.D1 * C, C, t.D1, g, c0, c_ok, false);
    mx_fetch<NJ, WR>(wv, a.w + (a.w_shared ? 0 : (int64_t)edge * t.P * C), C, t.P, g, c0, c_ok, !a.w_shared);
  };
  fetch(MxIndex::at(I.edge, 0), MxIndex::at(I.other, 0));
  const int n = (int)(R.p1 - R.p0);
  int cur = -1;
  bool first = true;
  const auto row_of = [&](bool complete) __attribute__((always_inline)) {
    return complete ? a.out + (int64_t)cur * t.DO * C : a.ws + (range * 2 + (first ? 0 : 1)) * t.DO * C;
  };
  for (int k = 0; k < n; ++k) {
    const int sid = MxIndex::at(I.sid, k & 63);
    if (lane < t.D2) mine[Y.y + lane] = yv;
    mx_stage<NJ, WR>(mine + Y.w, Y.pitch, wv, t.P, g, c0);
    mx_stage<NJ, 4>(mine + Y.r1, Y.pitch, xv, t.D1, g, c0);
    mx_sync();
    if (k + 1 < n) {
      if (((k + 1) & 63) == 0) I.load(a, R.p0 + k + 1, R.p1, lane);
      fetch(MxIndex::at(I.edge, (k + 1) & 63), MxIndex::at(I.other, (k + 1) & 63));
    }
    if (sid != cur) {
      if (cur >= 0) {
        mx_flush<NJ>(acc, row_of(first ? R.first_complete : true), t.DO, C, g, c0, c_ok, bad);
        first = false;
      }
      cur = sid;
    }
    mx_couple(tab + parts.rec, t.n_rec, mine + Y.y, mine + Y.a, lane);
    mx_sync();
    mx_contract<NJ>(acc, tab + parts.ent, t.n_ent, mine + Y.a, mine + Y.w, mine + Y.r1, Y.pitch, lane);
    mx_sync();
  }
  mx_flush<NJ>(acc, row_of((first ? R.first_complete : true) && R.last_complete), t.DO, C, g, c0, c_ok, bad);
  const bool any_bad = __any(!(bad == 0.f));
  if (lane == 0) t.flags[range] = any_bad;
}

template <int NJ, int WR>
__global__ void __launch_bounds__(512) uvu_mx_bwd_kernel(const UvuDev<float> a, const MxDev t) {
  extern __shared__ __align__(16) float mx_lds[];
  const MxParts parts(t.n_rec, t.n_ent, t.n_rowtiles, t.n_rounds, t.n_tiles);
  uint32_t* tab = reinterpret_cast<uint32_t*>(mx_lds);
  for (int i = threadIdx.x; i < t.n_words; i += blockDim.x) tab[i] = t.words[i];
  const MxLayout Y(NJ, t.D1, t.D2, t.DO, t.P, t.n_ent, t.n_rowtiles, true);
  const int lane = threadIdx.x & (kWave - 1), g = lane >> 4, r = lane & 15, c0 = r * NJ;
  float* mine = mx_lds + parts.words + (threadIdx.x / kWave) * Y.floats;
  for (int i = lane; i < Y.floats; i += kWave) mine[i] = 0.f;
  __syncthreads();
  const int64_t range = seg_wave_index(a.n_waves);
  if (range < 0) return;
  const MxRange R(a, range);
  const int64_t C = a.C;
  const bool c_ok = c0 < a.C;
  const bool want_gx = a.gx != nullptr, want_gy = a.gy != nullptr, want_gw = a.gw != nullptr;
  float *A = mine + Y.a, *ws = mine + Y.w, *gs = mine + Y.r1, *xs = mine + Y.r2;
  const int pitch = Y.pitch;
  mx4 acc[NJ];
#pragma unroll
  for (int j = 0; j < NJ; ++j) acc[j] = mx4{0.f, 0.f, 0.f, 0.f};
  MxIndex I;
  I.load(a, R.p0, R.p1, lane);
  float gv[4][NJ], wv[WR][NJ], yv, bad = 0.f;
  const auto fetch = [&](int edge, int other) __attribute__((always_inline)) {
    yv = a.y[(int64_t)edge * t.D2 + min(lane, t.D2 - 1)];
    mx_fetch<NJ, 4>(gv, a.g + (int64_t)other * t.DO * C, C, t.DO, g, c0, c_ok, false);
    mx_fetch<NJ, WR>(wv, a.w + (a.w_shared ? 0 : (int64_t)edge * t.P * C), C, t.P, g, c0, c_ok, !a.w_shared);
  };
  fetch(MxIndex::at(I.edge, 0), MxIndex::at(I.other, 0));
  const int n = (int)(R.p1 - R.p0);
  int cur = -1;
  bool first = true;
  float xt[NJ][4];         // x[row r][16 q + 4 g + i]: the second operand of G for the open segment
  const auto row_of = [&](bool complete) __attribute__((always_inline)) {
    return complete ? a.gx + (int64_t)cur * t.D1 * C : a.ws + (range * 2 + (first ? 0 : 1)) * t.D1 * C;
  };
  for (int k = 0; k < n; ++k) {
    const int sid = MxIndex::at(I.sid, k & 63);
    const int64_t e = MxIndex::at(I.edge, k & 63);
    if (lane < t.D2) mine[Y.y + lane] = yv;
    mx_stage<NJ, WR>(ws, pitch, wv, t.P, g, c0);
    mx_stage<NJ, 4>(gs, pitch, gv, t.DO, g, c0);
    if (sid != cur) {
      float xv[4][NJ];
      mx_fetch<NJ, 4>(xv, a.x + (int64_t)sid * t.D1 * C, C, t.D1, g, c0, c_ok, false);
      mx_stage<NJ, 4>(xs, pitch, xv, t.D1, g, c0);
      mx_sync();
      const float* xr = xs + min(r, t.D1) * pitch + 4 * g;
#pragma unroll
      for (int q = 0; q < NJ; ++q) mx_get<4>(xt[q], xr + 16 * q);
      if (cur >= 0) {
        if (want_gx) mx_flush<NJ>(acc, row_of(first ? R.first_complete : true), t.D1, C, g, c0, c_ok, bad);
        first = false;
      }
      cur = sid;
    }
    mx_sync();
    if (k + 1 < n) {
      if (((k + 1) & 63) == 0) I.load(a, R.p0 + k + 1, R.p1, lane);
      fetch(MxIndex::at(I.edge, (k + 1) & 63), MxIndex::at(I.other, (k + 1) & 63));
    }
    mx_couple(tab + parts.rec, t.n_rec, mine + Y.y, A, lane);
    mx_sync();
    if (want_gx) mx_contract<NJ>(acc, tab + parts.ent, t.n_ent, A, ws, gs, pitch, lane);
    if (want_gy) {
      mx4 G[kMxMaxPaths / 4];
#pragma unroll
      for (int s = 0; s < kMxMaxPaths / 4; ++s) {
        if (s < t.n_rowtiles) {
          const uint32_t rw = tab[parts.row + 16 * s + r];
          G[s] = mx_channels<NJ>(ws + (rw & 255) * pitch + 4 * g, gs + (rw >> 8) * pitch + 4 * g, xt);
        }
      }
      mx_sync();            // the weight rows are consumed: G takes their place
#pragma unroll
      for (int s = 0; s < kMxMaxPaths / 4; ++s) {
        if (s < t.n_rowtiles) {
#pragma unroll
          for (int i = 0; i < 4; ++i) ws[(16 * s + 4 * g + i) * 16 + r] = G[s][i];
        }
      }
      mx_sync();
      mx_grad_y(a, t, tab + parts.term, ws, e, lane, bad);
      mx_sync();
    }
    if (want_gw) {          // the weight gradient is gathered in the weight rows' place
      for (int u = 0; u < t.n_tiles; ++u) {
        const uint32_t* tile = tab + parts.tile + 5 * u;
        const uint32_t head = (uint32_t)__builtin_amdgcn_readfirstlane((int)tile[0]);
        const uint32_t mya = tile[1 + (r >> 2)], myc = tile[1 + g];
        const float* Ar = A + (mya & 0xffff) + g * 16 + (r & 3);
        const float* gr = gs + ((head & 255) + g) * pitch + c0;
        mx4 D[NJ];
#pragma unroll
        for (int j = 0; j < NJ; ++j) D[j] = mx4{0.f, 0.f, 0.f, 0.f};
        const int steps = (int)(head >> 8);
        for (int s = 0; s < steps; ++s) {
          const float av = Ar[64 * s];
          float gq[NJ];
          mx_get<NJ>(gq, gr + 4 * s * pitch);
#pragma unroll
          for (int j = 0; j < NJ; ++j) D[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(av, gq[j], D[j], 0, 0, 0);
        }
        // chunk: element of A | path << 16 | (adds to an earlier chunk) << 24 | rows << 25
        const int row0 = (int)(myc & 15), rows = (int)(myc >> 25);
        float v[NJ];
#pragma unroll
        for (int j = 0; j < NJ; ++j) v[j] = 0.f;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          float xr[NJ];
          mx_get<NJ>(xr, xs + (i < rows ? row0 + i : t.D1) * pitch + c0);
#pragma unroll
          for (int j = 0; j < NJ; ++j) v[j] = fmaf(xr[j], D[j][i], v[j]);
        }
        if (rows > 0) {
          float* at = ws + ((myc >> 16) & 255) * pitch + c0;
          if (myc & (1u << 24)) {
            float o[NJ];
            mx_get<NJ>(o, at);
#pragma unroll
            for (int j = 0; j < NJ; ++j) v[j] += o[j];
          }
          mx_put<NJ>(at, v);
        }
      }
      mx_sync();
      mx_store_grad_w<NJ, WR>(a, t, ws, pitch, e, g, c0, c_ok, bad);
      mx_sync();
    }
  }
  if (want_gx) mx_flush<NJ>(acc, row_of((first ? R.first_complete : true) && R.last_complete), t.D1, C, g, c0, c_ok, bad);
  const bool any_bad = __any(!(bad == 0.f));
  if (lane == 0) t.flags[range] = any_bad;
}

// ---- backward, one channel per lane (33 to 64 channels) ----------------------------------------------------------
// A path couples 2 l + 1 of up to 16 rows, so three quarters of a 16-row tile multiply zeros.  v_mfma_f32_4x4x1_16b_f32 takes
// 16 blocks of four channels times four rows and one contracted row in 8 cycles, with A broadcast from one block to
// all: no padding of the contracted rows, none of the tile beyond the multiple of four, and a lane keeps one channel
// throughout.  The rows of x are cut into chunks of up to four rows of one irrep; an item is a path's share of a chunk, up
// to seven rows of grad_out; a register of A holds the eight slots of two items.  D = A^T g of an item gives both
// gradients: grad_x += w D and grad_w = sum over the rows of x D.  At 206 coefficients about 115 such instructions
// replace 136 of 32 cycles per edge; G, whose contraction runs over the channels, stays on 16 x 16 x 4.  65 536 edges, 64
// channels, 206 coefficients: 453 -> 371 us; 32 768 edges, forward and backward: 350 -> 307 us, 58 coefficients 169 -> 158
// us.  The forward gains nothing this way (175 -> 180 us; 58 coefficients 47 -> 61): its single contraction waits for
// two LDS reads per contracted row instead of three per four, so it stays on 16-row tiles.
constexpr int kMxChunks = 8;
struct Mx4Parts {
  int rec, item, chunk, row, term, words;
  __host__ __device__ Mx4Parts(int n_rec, int n_items, int n_rowtiles, int n_rounds) {
    rec = 0;
    item = rec + 3 * n_rec;                 // n_items (even) x (path | first row << 8 | rows << 16 | adds << 20)
    chunk = item + n_items;                 // kMxChunks x (first row | rows << 8 | end of its pairs of items << 16)
    row = chunk + kMxChunks;                // as MxParts
    term = row + 16 * n_rowtiles;
    words = (term + 128 * n_rounds + 3) & ~3;
  }
};
constexpr int kMx4Pitch = 68;               // LDS row: 64 channels, and 4 for the row-wise reads of G
struct Mx4Layout {
  int a, w, r1, e, y, floats;
  __host__ __device__ Mx4Layout(int D2, int DO, int P, int n_items, int n_rowtiles) {
    int at = 0;
    const auto take = [&](int n) { const int r = at; at += (n + 3) & ~3; return r; };
    a = take(32 * n_items);
    w = take(P * kMx4Pitch);
    r1 = take((DO + 6) * kMx4Pitch);                  // an item's seven rows may reach six past the end
    const int g_floats = 256 * n_rowtiles, gw_floats = P * kMx4Pitch;
    e = take(g_floats > gw_floats ? g_floats : gw_floats);      // G, then the weight gradient
    y = take(D2);
    floats = at;
  }
};

// Operands of a pair of items, requested one pair ahead.
struct Mx4Pair {
  uint32_t k[2];
  float a, w[2], r[2][7];
  __device__ __forceinline__ void request(uint32_t items, int pair, const float* A, const float* ws, const float* rows, int lane) {
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      k[h] = (uint32_t)__builtin_amdgcn_readlane((int)items, 2 * pair + h);
      w[h] = ws[(k[h] & 255) * kMx4Pitch + lane];
      const float* at = rows + ((k[h] >> 8) & 255) * kMx4Pitch + lane;
#pragma unroll
      for (int j = 0; j < 7; ++j) r[h][j] = at[j * kMx4Pitch];
    }
    a = A[pair * 64 + lane];
  }
  __device__ __forceinline__ int rows() const { return max((int)(k[0] >> 16) & 15, (int)(k[1] >> 16) & 15); }
};
// z[h] += the slot's four rows times b (A of block 8 h + J broadcast to all blocks)
template <int J>
__device__ __forceinline__ void mx4_step(mx4 (&z)[2], float a, float b0, float b1) {
  z[0] = __builtin_amdgcn_mfma_f32_4x4x1f32(a, b0, z[0], 4, J, 0);
  z[1] = __builtin_amdgcn_mfma_f32_4x4x1f32(a, b1, z[1], 4, 8 + J, 0);
}
// b(h, j): the operand of row j of item h
template <class B>
__device__ __forceinline__ void mx4_multiply(mx4 (&z)[2], float a, int rows, B&& b) {
  mx4_step<0>(z, a, b(0, 0), b(1, 0));
  if (rows > 1) {
    mx4_step<1>(z, a, b(0, 1), b(1, 1));
    mx4_step<2>(z, a, b(0, 2), b(1, 2));
  }
  if (rows > 3) {
    mx4_step<3>(z, a, b(0, 3), b(1, 3));
    mx4_step<4>(z, a, b(0, 4), b(1, 4));
  }
  if (rows > 5) {
    mx4_step<5>(z, a, b(0, 5), b(1, 5));
    mx4_step<6>(z, a, b(0, 6), b(1, 6));
  }
}

__device__ __forceinline__ void mx4_flush(mx4 (&acc)[kMxChunks], uint32_t chunks, int n_chunks, float* dst, int64_t C, int lane,
                                          float& bad) {
#pragma unroll
  for (int c = 0; c < kMxChunks; ++c) {
    if (c < n_chunks) {
      const uint32_t k = (uint32_t)__builtin_amdgcn_readlane((int)chunks, c);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        bad = fmaf(acc[c][i], 0.f, bad);
        if (i < (int)((k >> 8) & 255) && lane < C) dst[((k & 255) + i) * C + lane] = acc[c][i];
      }
      acc[c] = mx4{0.f, 0.f, 0.f, 0.f};
    }
  }
}

template <int WR>
__global__ void __launch_bounds__(512) uvu_mx4_bwd_kernel(const UvuDev<float> a, const MxDev t) {
  extern __shared__ __align__(16) float mx_lds[];
  const Mx4Parts parts(t.n_rec, t.n_ent, t.n_rowtiles, t.n_rounds);
  uint32_t* tab = reinterpret_cast<uint32_t*>(mx_lds);
  for (int i = threadIdx.x; i < t.n_words; i += blockDim.x) tab[i] = t.words[i];
  const Mx4Layout Y(t.D2, t.DO, t.P, t.n_ent, t.n_rowtiles);
  const int lane = threadIdx.x & (kWave - 1), g = lane >> 4, r = lane & 15, c0 = r * 4;
  float* mine = mx_lds + parts.words + (threadIdx.x / kWave) * Y.floats;
  for (int i = lane; i < Y.floats; i += kWave) mine[i] = 0.f;
  __syncthreads();
  const int64_t range = seg_wave_index(a.n_waves);
  if (range < 0) return;
  const MxRange R(a, range);
  const int64_t C = a.C;
  const bool c_ok = c0 < a.C;
  const bool want_gx = a.gx != nullptr, want_gy = a.gy != nullptr, want_gw = a.gw != nullptr;
  float *A = mine + Y.a, *ws = mine + Y.w, *gs = mine + Y.r1, *E = mine + Y.e;
  const uint32_t items = tab[parts.item + min(lane, t.n_ent - 1)], chunks = tab[parts.chunk + min(lane, kMxChunks - 1)];
  mx4 acc[kMxChunks];
#pragma unroll
  for (int c = 0; c < kMxChunks; ++c) acc[c] = mx4{0.f, 0.f, 0.f, 0.f};
  MxIndex I;
  I.load(a, R.p0, R.p1, lane);
  float gv[4][4], wv[WR][4], yv, bad = 0.f;
  const auto fetch = [&](int edge, int other) __attribute__((always_inline)) {
    yv = a.y[(int64_t)edge * t.D2 + min(lane, t.D2 - 1)];
    mx_fetch<4, 4>(gv, a.g + (int64_t)other * t.DO * C, C, t.DO, g, c0, c_ok, false);
    mx_fetch<4, WR>(wv, a.w + (a.w_shared ? 0 : (int64_t)edge * t.P * C), C, t.P, g, c0, c_ok, !a.w_shared);
  };
  fetch(MxIndex::at(I.edge, 0), MxIndex::at(I.other, 0));
  const int n = (int)(R.p1 - R.p0);
  int cur = -1;
  bool first = true;
  float xt[4][4];          // x[row r][16 q + 4 g + i]: the second operand of G for the open segment
  mx4 xr[kMxChunks];       // the open segment's rows of x, this lane's channel
  const auto row_of = [&](bool complete) __attribute__((always_inline)) {
    return complete ? a.gx + (int64_t)cur * t.D1 * C : a.ws + (range * 2 + (first ? 0 : 1)) * t.D1 * C;
  };
  for (int k = 0; k < n; ++k) {
    const int sid = MxIndex::at(I.sid, k & 63);
    const int64_t e = MxIndex::at(I.edge, k & 63);
    if (lane < t.D2) mine[Y.y + lane] = yv;
    mx_stage<4, WR>(ws, kMx4Pitch, wv, t.P, g, c0);
    mx_stage<4, 4>(gs, kMx4Pitch, gv, t.DO, g, c0);
    if (sid != cur) {
      const float* xrow = a.x + (int64_t)sid * t.D1 * C;
      const int cl = lane < C ? lane : 0;
#pragma unroll
      for (int c = 0; c < kMxChunks; ++c) {
        xr[c] = mx4{0.f, 0.f, 0.f, 0.f};
        if (c < t.n_chunks) {
          const uint32_t ck = (uint32_t)__builtin_amdgcn_readlane((int)chunks, c);
#pragma unroll
          for (int i = 0; i < 4; ++i)
            if (i < (int)((ck >> 8) & 255)) {
              const float v = xrow[((ck & 255) + i) * C + cl];
              xr[c][i] = lane < C ? v : 0.f;
            }
        }
      }
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const bool in = r < t.D1 && 16 * q + 4 * g < C;        // C is a multiple of 4
        load_vec<float, 4>(xt[q], xrow + (in ? r * C + 16 * q + 4 * g : 0));
#pragma unroll
        for (int i = 0; i < 4; ++i) xt[q][i] = in ? xt[q][i] : 0.f;
      }
      if (cur >= 0) {
        if (want_gx) mx4_flush(acc, chunks, t.n_chunks, row_of(first ? R.first_complete : true), C, lane, bad);
        first = false;
      }
      cur = sid;
    }
    mx_sync();
    if (k + 1 < n) {
      if (((k + 1) & 63) == 0) I.load(a, R.p0 + k + 1, R.p1, lane);
      fetch(MxIndex::at(I.edge, (k + 1) & 63), MxIndex::at(I.other, (k + 1) & 63));
    }
    mx_couple(tab + parts.rec, t.n_rec, mine + Y.y, A, lane);
    mx_sync();
    if (want_gy) {
      for (int s = 0; s < t.n_rowtiles; ++s) {
        const uint32_t rw = tab[parts.row + 16 * s + r];
        const mx4 G = mx_channels<4>(ws + (rw & 255) * kMx4Pitch + 4 * g, gs + (rw >> 8) * kMx4Pitch + 4 * g, xt);
#pragma unroll
        for (int i = 0; i < 4; ++i) E[(16 * s + 4 * g + i) * 16 + r] = G[i];
      }
      mx_sync();
      mx_grad_y(a, t, tab + parts.term, E, e, lane, bad);
      mx_sync();
    }
    if (want_gx || want_gw) {
      const int last = t.n_ent / 2 - 1;
      int pair = 0;
      Mx4Pair N;
      N.request(items, 0, A, ws, gs, lane);
#pragma unroll
      for (int c = 0; c < kMxChunks; ++c) {
        if (c < t.n_chunks) {
          const int end = (int)((uint32_t)__builtin_amdgcn_readlane((int)chunks, c) >> 16);
          for (; pair < end; ++pair) {
            const Mx4Pair P = N;
            N.request(items, min(pair + 1, last), A, ws, gs, lane);
            mx4 D[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
            mx4_multiply(D, P.a, P.rows(), [&](int h, int j) __attribute__((always_inline)) { return P.r[h][j]; });
            acc[c] += P.w[0] * D[0] + P.w[1] * D[1];
#pragma unroll
            for (int h = 0; h < 2; ++h) {
              float* at = E + (P.k[h] & 255) * kMx4Pitch + lane;
              float v = (P.k[h] >> 20) & 1 ? *at : 0.f;       // an earlier chunk of the path
#pragma unroll
              for (int i = 0; i < 4; ++i) v = fmaf(xr[c][i], D[h][i], v);
              *at = v;
            }
          }
        }
      }
      mx_sync();
      if (want_gw) mx_store_grad_w<4, WR>(a, t, E, kMx4Pitch, e, g, c0, c_ok, bad);
      mx_sync();
    }
  }
  if (want_gx) mx4_flush(acc, chunks, t.n_chunks, row_of((first ? R.first_complete : true) && R.last_complete), C, lane, bad);
  const bool any_bad = __any(!(bad == 0.f));
  if (lane == 0) t.flags[range] = any_bad;
}

// ---- host side ------------------------------------------------------------------------------------------------
struct MxPlan {
  int nj, wr, per, waves_per_group;
  bool wide;             // one channel per lane
  int64_t n_ranges, n_flags, ws_elems;
  size_t lds_bytes;
  int n_words;
};

static int mx_plan(const cgtp_uvu_args* a, const cgtp_uvu_tab* t, const cgtp_uvu_mx* m, int backward, MxPlan* plan) {
  if (!a || !t || !m || !m->fwd || !m->bwd) return CGTP_ERR_NULL;
  const int rc = cgtp_uvu_tab_validate(a, t, backward);      // everything the entry-by-entry kernel asks for holds here too
  if (rc != CGTP_OK) return rc;
  if (t->D1 > 16 || t->D2 > 32 || t->DO > 16 || t->P > kMxMaxPaths) return CGTP_ERR_SHAPE;
  const int n_ent = backward ? m->bwd_entries : m->fwd_entries, n_rec = backward ? m->bwd_records : m->fwd_records;
  if (n_ent <= 0 || n_ent > 64 || n_rec <= 0 || m->row_tiles <= 0 || m->row_tiles > kMxMaxPaths / 4 || m->rounds <= 0 ||
      m->tiles <= 0 || m->lanes_log2 < 0 || (t->D2 << m->lanes_log2) > kWave)
    return CGTP_ERR_SHAPE;
  if (a->C > 64) return CGTP_ERR_SHAPE;
  plan->nj = a->C <= 16 ? 1 : a->C <= 32 ? 2 : 4;
  if (a->C % plan->nj) return CGTP_ERR_SHAPE;
  const uintptr_t bytes = (uintptr_t)a->x | (uintptr_t)a->w | (uintptr_t)a->workspace |
                          (backward ? (uintptr_t)a->grad_out | (uintptr_t)a->grad_x | (uintptr_t)a->grad_w : (uintptr_t)a->out);
  if (bytes & (4 * plan->nj - 1)) return CGTP_ERR_SHAPE;
  plan->wr = t->P <= 16 ? 4 : 8;
  // Few coefficients and few channels leave little to contract: up to 64 coefficients and 32 channels the backward is quicker
  // entry by entry (58 coefficients, 32 768 edges, 32 channels: 97 against 108 us; 206 coefficients: 425 against 203).
  if (backward && plan->nj < 4 && t->nnz <= 64) return CGTP_ERR_SHAPE;
  // one channel per lane past 32 channels, where the rows fit eight chunks (they do unless there are many scalars)
  plan->wide = backward && plan->nj == 4 && m->bwd4 && m->bwd4_chunks > 0 && m->bwd4_chunks <= kMxChunks && m->bwd4_items > 0 &&
               m->bwd4_items <= 64 && m->bwd4_items % 2 == 0;
  const MxParts parts16(n_rec, n_ent, backward ? m->row_tiles : 0, backward ? m->rounds : 0, backward ? m->tiles : 0);
  const Mx4Parts parts4(n_rec, m->bwd4_items, m->row_tiles, m->rounds);
  const MxLayout Y16(plan->nj, t->D1, t->D2, t->DO, t->P, n_ent, m->row_tiles, backward != 0);
  const Mx4Layout Y4(t->D2, t->DO, t->P, m->bwd4_items, m->row_tiles);
  const int wave_floats = plan->wide ? Y4.floats : Y16.floats, words = plan->wide ? parts4.words : parts16.words;
  plan->n_words = words;
  // as many wavefronts per compute unit as the LDS holds, at most two per SIMD in the backward (registers); workgroups
  // of up to eight wavefronts there and four in the forward, sharing one copy of the tables
  const int64_t wave_bytes = 4 * (int64_t)wave_floats, tab_bytes = 4 * (int64_t)words;
  int best = 0;
  for (int w = backward ? 8 : 4; w >= 1; --w) {
    const int64_t group = w * wave_bytes + tab_bytes;
    if (group > kLdsBytes) continue;
    int per_cu = (int)(kLdsBytes / group) * w;
    if (per_cu > 8) per_cu = 8 / w * w;
    if (per_cu > best) {
      best = per_cu;
      plan->waves_per_group = w;
      plan->lds_bytes = (size_t)group;
    }
  }
  if (!best) return CGTP_ERR_LDS;
  // one range per resident wavefront, of at least four positions
  const int64_t resident = 256 * (int64_t)best;
  int64_t per = a->pos_per_wave > 0 ? a->pos_per_wave : (a->n_rows + resident - 1) / resident;
  if (a->pos_per_wave <= 0 && per < 4) per = 4;
  if (per >= (int64_t)1 << 30) return CGTP_ERR_SHAPE;
  plan->per = (int)per;
  plan->n_ranges = (a->n_rows + per - 1) / per;
  plan->n_flags = plan->n_ranges;
  // partial rows, laid out for the padded number of ranges the entry-by-entry kernel may touch, then the flags
  const int64_t rows = (plan->n_ranges + kWave) * 2 * (backward ? t->D1 : t->DO) * a->C;
  plan->ws_elems = !backward || a->grad_x ? (rows + 3) & ~(int64_t)3 : 0;
  return CGTP_OK;
}

template <int NJ>
static const void* mx_kernel(bool backward, int wr) {
  if (backward) return wr == 4 ? (const void*)uvu_mx_bwd_kernel<NJ, 4> : (const void*)uvu_mx_bwd_kernel<NJ, 8>;
  return wr == 4 ? (const void*)uvu_mx_fwd_kernel<NJ, 4> : (const void*)uvu_mx_fwd_kernel<NJ, 8>;
}

static int mx_launch(const cgtp_uvu_args* a, const cgtp_uvu_tab* t, const cgtp_uvu_mx* m, int backward, hipStream_t stream) {
  MxPlan plan;
  const int rc = mx_plan(a, t, m, backward, &plan);
  if (rc != CGTP_OK) return rc;
  float* rows = backward ? (float*)a->grad_x : (float*)a->out;
  if (plan.n_ranges > 0) {
    if (!a->workspace) return CGTP_ERR_WORKSPACE;
    UvuDev<float> d = {};
    d.x = (const float*)a->x; d.y = (const float*)a->y; d.w = (const float*)a->w; d.out = (float*)a->out;
    d.g = (const float*)a->grad_out; d.gx = (float*)a->grad_x; d.gy = (float*)a->grad_y; d.gw = (float*)a->grad_w;
    d.ws = (float*)a->workspace;
    d.ptr = a->ptr; d.perm = a->perm; d.gather = a->gather; d.seg_ids = a->seg_ids;
    d.n_rows = a->n_rows; d.n_seg = a->n_seg; d.n_waves = plan.n_ranges;
    d.C = a->C; d.w_shared = a->w_shared; d.pos_per_wave = plan.per;
    MxDev dev = {};
    dev.words = plan.wide ? m->bwd4 : backward ? m->bwd : m->fwd;
    dev.n_rec = backward ? m->bwd_records : m->fwd_records;
    dev.n_ent = plan.wide ? m->bwd4_items : backward ? m->bwd_entries : m->fwd_entries;
    dev.n_chunks = m->bwd4_chunks;
    dev.n_rowtiles = m->row_tiles; dev.n_rounds = m->rounds; dev.lanes_log2 = m->lanes_log2; dev.n_tiles = m->tiles;
    dev.n_words = plan.n_words;
    dev.D1 = t->D1; dev.D2 = t->D2; dev.DO = t->DO; dev.P = t->P;
    dev.flags = reinterpret_cast<int32_t*>((float*)a->workspace + plan.ws_elems);
    const void* fn = plan.wide ? (plan.wr == 4 ? (const void*)uvu_mx4_bwd_kernel<4> : (const void*)uvu_mx4_bwd_kernel<8>)
                     : plan.nj == 1 ? mx_kernel<1>(backward, plan.wr)
                                  : plan.nj == 2 ? mx_kernel<2>(backward, plan.wr) : mx_kernel<4>(backward, plan.wr);
    if (plan.lds_bytes > 48 * 1024 &&
        hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)plan.lds_bytes) != hipSuccess)
      return CGTP_ERR_LDS;
    const int64_t blocks = (plan.n_ranges + plan.waves_per_group - 1) / plan.waves_per_group;
    const int64_t groups = (blocks + 7) / 8 * 8;       // seg_wave_index deals them to the XCDs
    void* args[] = {&d, &dev};
    if (hipLaunchKernel(fn, dim3((unsigned)groups), dim3((unsigned)(plan.waves_per_group * kWave)), args, plan.lds_bytes,
                        stream) != hipSuccess)
      return CGTP_ERR_LAUNCH;
    const int redo = uvu_tab_redo_flagged(a, t, backward, plan.per, dev.flags, plan.n_flags, stream);
    if (redo != CGTP_OK) return redo;
  }
  if (!rows) return CGTP_OK;
  return uvu_fixup_rows_f32(rows, (const float*)a->workspace, a->ptr, a->n_seg, (backward ? t->D1 : t->DO) * (int64_t)a->C,
                            plan.per, plan.n_ranges, a->n_rows, stream);
}

}  // namespace cgtp

using namespace cgtp;

extern "C" {

int64_t cgtp_uvu_mx_workspace_bytes(const cgtp_uvu_args* a, const cgtp_uvu_tab* t, const cgtp_uvu_mx* m, int backward) {
  MxPlan plan;
  if (mx_plan(a, t, m, backward, &plan) != CGTP_OK) return -1;
  return plan.n_ranges > 0 ? (plan.ws_elems + plan.n_flags) * (int64_t)sizeof(float) : 0;
}

int cgtp_uvu_mx_validate(const cgtp_uvu_args* a, const cgtp_uvu_tab* t, const cgtp_uvu_mx* m, int backward) {
  MxPlan plan;
  return mx_plan(a, t, m, backward, &plan);
}

int cgtp_uvu_mx_fwd(const cgtp_uvu_args* a, const cgtp_uvu_tab* t, const cgtp_uvu_mx* m, void* stream) {
  return mx_launch(a, t, m, 0, (hipStream_t)stream);
}

int cgtp_uvu_mx_bwd(const cgtp_uvu_args* a, const cgtp_uvu_tab* t, const cgtp_uvu_mx* m, void* stream) {
  return mx_launch(a, t, m, 1, (hipStream_t)stream);
}

}  // extern "C"
