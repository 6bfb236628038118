// Channel mixing in single precision on the half-precision matrix cores (IrrepsLinear, SO2Linear('uv'), any table):
//
//   out[n, m, w] = sum_{entries e of row m} coef_e * sum_u x[n, a_e, u] * W[p_e, u, w]
//
// forward, and the gradient of x with the rows' roles exchanged and the weight read transposed.  Operands are three bf16
// parts each and a product is six matrix instructions (uv_parts.h); the coefficient goes into the packed weight.
//
// A workgroup owns 64 NT samples and a group of rows of the result, one or two at a time (two where the same rows of x reach both, the
// +m and -m rows of an SO(2) layer: read and split once); a wavefront 16 NT of the samples, 16 TW channels.  A unit of work is
// 32 contracted channels of one row of x: the wavefront's part comes through LDS of its own in whole lines, is split, and is multiplied
// with the unit's weight fragments, which the four wavefronts share through LDS (the vector L1 delivers 64 bytes a cycle, and
// fragments loaded by each wavefront would take all of it).  Both are requested two units ahead.  The workgroups of one block of
// samples are neighbours on one XCD: rows of x are read again for every group of rows they reach, from its L2.
//
// What bounds it: matrix instructions, at the clock of 1.6 to 1.8 GHz that the card keeps under them (SO2Linear, lmax = 4, 64
// channels, 32768 samples: 134 us of the 270 at 1.7 GHz; without them the launch takes 155, L2 and stores).
// Measured there, one call at a time with the packing (the kernel alone: 252): 571 us on fp32 matrix instructions (uvt_apply_kernel)
// -> 273; lmax 2: 32 channels, 4096 samples 12.9 -> 11.0; IrrepsLinear 64 -> 64, lmax 2, 65536 samples 126 -> 75, 128 -> 128, lmax 3,
// 32768 samples 308 -> 170.  One workgroup per pair of rows, 325 us: a third of its time went into starting; half lines of x from
// memory straight into the operands, 300; three wavefronts per SIMD (spills), eight in a workgroup, matrix and vector instructions in
// turn by hand: no change.  Errors of the results against 64 bits: 0.4e-7 to 3.8e-7, of fp32 matrix instructions 0.9e-7 to 4.5e-7
// (BY_UNIT below).
//
// Values: elements that are not finite or overflow as parts show in the results, and elements below 2^-110 (but not zero; their
// last part could be below the smallest subnormal) are looked for; a wavefront that sees either forms its results
// again with fp32 matrix instructions from memory.
#include "uv_parts.h"

#pragma clang fp contract(fast)

namespace cgtp {

struct UvlDev {
  const float* x;
  const u32x4* packed;
  const unsigned* asks;               // a word per (block, block of produced channels)
  const float* w;
  float* out;
  const cgtp_uvl_step* steps;
  const cgtp_uvl_task* tasks;
  const cgtp_uvl_group* groups;
  const cgtp_uvl_block* blocks;
  int64_t n_rows, stride_p, stride_k, stride_c;
  int dx, dout, cx, cout, n_groups;
  int kc;                             // units of 32 contracted channels
  int cblocks, sblocks;               // blocks of 16 TW produced channels, of samples
};

// A workgroup per (block, block of produced channels): parts of coef * W in fragment order, [unit][part][tile][lane] of 16 bytes.
template <int TW>
__global__ void __launch_bounds__(256) uvl_pack_kernel(const cgtp_uvl_block* __restrict__ blocks, const float* __restrict__ w,
                                                       u32x4* __restrict__ packed, unsigned* __restrict__ asks, int kc, int cx,
                                                       int cout, int64_t stride_p, int64_t stride_k, int64_t stride_c) {
  __shared__ unsigned plain;
  if (threadIdx.x == 0) plain = 0;
  __syncthreads();
  const cgtp_uvl_block b = blocks[blockIdx.x];
  const float* wp = w + b.path * stride_p;
  u32x4* dst = packed + (int64_t)(blockIdx.x * gridDim.y + blockIdx.y) * kc * (TW * 192);
  unsigned m = 0;
  const float lift = b.coef != 0.f ? 0x1p+60f : 0.f;
  for (int i = threadIdx.x; i < kc * TW * 64; i += 256) {
    const int lane = i & 63, t = (i >> 6) % TW, k = (i >> 6) / TW;
    // the columns a lane of uvl_kernel holds for unit k; those of the unit before get zeros
    const int ch = blockIdx.y * 16 * TW + 16 * t + (lane & 15), first = max(min(k * 32, cx - 32), 0) + 8 * (lane >> 4);
    float v[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const int col = first + j;
      const bool in = col >= k * 32 && col < cx && ch < cout;
      const float e = wp[(in ? col : 0) * stride_k + (in ? ch : 0) * stride_c], u = in ? e : 0.f;
      v[j] = b.coef * u;
      // what the coefficient left of a subnormal weight, but not of a large x (no branch: that would sink the loads, 11 -> 15 us
      // a launch of 128 -> 128 channels)
      m |= (uvs_asks(v[j]) & kUvsPlain) | ((unsigned)(v[j] == 0.f) & (unsigned)(u * lift != 0.f));
    }
    UvsParts<8> part;
#pragma unroll
    for (int j = 0; j < 4; ++j) part.pair(j, v[2 * j], v[2 * j + 1]);
#pragma unroll
    for (int h = 0; h < 3; ++h) dst[((k * 3 + h) * TW + t) * 64 + lane] = u32x4{part.p[h][0], part.p[h][1], part.p[h][2], part.p[h][3]};
  }
  if (m) plain = 1;          // whoever writes, writes the same
  __syncthreads();
  if (threadIdx.x == 0) asks[blockIdx.x * gridDim.y + blockIdx.y] = plain;
}

// RW rows of the result at a time.  Per unit of 32 channels a wavefront issues 24 NT RW matrix instructions (TW = 4).
//
// BY_UNIT: the matrix instruction rounds downwards, six times a unit at the size of the row's sum where all six products are added to
// it: 0.75 to 0.85 of the error of fp32 matrix instructions, and so for the tables those take (1 to 24 units of 32 channels, random
// operands or of one sign: 0.4e-7 to 3.8e-7, 0.9e-7 to 4.5e-7).  The larger tables were products of the library, which sums in
// blocks: for them a unit's six are summed by themselves (24 units 3.2e-7 -> 1.0e-7, 96 units 7.7e-7 -> 1.8e-7, of one sign 4.9e-7 ->
// 1.4e-7; a sum of the five small products beside the one of the large ones: 2.7e-7).  It takes 1 to 6 % more time: SO2Linear, lmax 4,
// 64 channels, 32768 samples 259 -> 269 us.
template <int TW, int NT, int RW, bool BY_UNIT>
__global__ void __launch_bounds__(256, NT * RW == 4 ? 2 : 3) uvl_kernel(const UvlDev a) {
  constexpr int CHUNK = TW * 192;                   // 16-byte words of a block's fragments of a unit
  __shared__ u32x4 lds[2][RW][CHUNK];
  __shared__ f32x4 xlds[4][NT * 128];
  // workgroups b, b + 8, ... run on one XCD: the groups of one block of samples there one after the other
  const int parts = a.n_groups * a.cblocks, j = blockIdx.x >> 3, at_part = j % parts;
  const int sb = j / parts * 8 + (blockIdx.x & 7);
  if (sb >= a.sblocks) return;
  const cgtp_uvl_group group = a.groups[at_part / a.cblocks];
  const int cb = at_part % a.cblocks;
  const int tid = threadIdx.x, lane = tid & (kWave - 1), wave = __builtin_amdgcn_readfirstlane(tid / kWave);
  const int r = lane & 15, q = lane >> 4;
  const int64_t first = (int64_t)sb * (64 * NT) + wave * (16 * NT);
  const int64_t n0 = min(first, a.n_rows - 1);      // past the end: the last row again
  const int row_elems = a.dx * a.cx, left = (int)min(a.n_rows - n0, (int64_t)(16 * NT));
  const float* xw = a.x + n0 * row_elems;
  // A wavefront's rows go through LDS of its own: a load takes whole lines of eight samples (16 bytes a lane), where the lanes'
  // matrix operands are 32 bytes of each of 16 samples, half lines whichever way they are loaded.  Piece p of a sample lies at
  // place p ^ (sample % 8), so that neither side has bank conflicts.  A unit's channels start 32 before the last one at most (the weight
  // has zeros where they overlap the unit before); with fewer than 32, the pieces past them are others (and the weight has zeros).
  unsigned at[2 * NT];
#pragma unroll
  for (int i = 0; i < 2 * NT; ++i)
    at[i] = 4u * (min(8 * i + (lane >> 3), left - 1) * row_elems + min(4 * ((lane & 7) ^ (lane >> 3)), a.cx - 4));
  f32x4* mine_x = xlds[wave];

  // lane l holds step l of the group (64 at most)
  const int steps = group.step_end - group.step_begin, units = steps * a.kc;
  const cgtp_uvl_step mine = a.steps[group.step_begin + min(lane, steps - 1)];
  unsigned plain_w = 0;
#pragma unroll
  for (int w = 0; w < RW; ++w) plain_w |= mine.block[w] >= 0 ? a.asks[mine.block[w] * a.cblocks + cb] : 0;
  floatx4 acc[RW][TW][NT];
  auto clear = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int w = 0; w < RW; ++w)
#pragma unroll
      for (int t = 0; t < TW; ++t)
#pragma unroll
        for (int i = 0; i < NT; ++i) acc[w][t][i] = floatx4{0.f, 0.f, 0.f, 0.f};
  };
  // Steps begin .. end again in fp32 matrix instructions, operands from memory.
  auto form_plain = [&](int begin, int end) __attribute__((always_inline)) {
    clear();
    for (int s = begin; s <= end; ++s) {
      const float* xr = xw + __builtin_amdgcn_readlane(mine.row, s) * a.cx;
#pragma unroll
      for (int w = 0; w < RW; ++w) {
        const int b = __builtin_amdgcn_readlane(mine.block[w], s);
        if (b < 0) continue;
        const cgtp_uvl_block of = a.blocks[b];
        const float* wp = a.w + of.path * a.stride_p;
        for (int k = q; k < a.cx; k += 4) {          // cx is a multiple of 4: the same count in every lane
          float xv[NT];
#pragma unroll
          for (int i = 0; i < NT; ++i) xv[i] = of.coef * xr[min(16 * i + r, left - 1) * row_elems + k];
#pragma unroll
          for (int t = 0; t < TW; ++t) {
            const int ch = min(cb * 16 * TW + 16 * t + r, a.cout - 1);
            const float wv = wp[k * a.stride_k + ch * a.stride_c];
#pragma unroll
            for (int i = 0; i < NT; ++i) acc[w][t][i] = __builtin_amdgcn_mfma_f32_16x16x4f32(wv, xv[i], acc[w][t][i], 0, 0, 0);
          }
        }
      }
    }
  };
  struct Cursor { int s, k; };
  auto advance = [&](Cursor& c) __attribute__((always_inline)) {
    if (++c.k == a.kc) {
      c.k = 0;
      c.s = min(c.s + 1, steps - 1);                 // past the last unit: anything that is there
    }
  };
  f32x4 raw[2 * NT];
  auto load_x = [&](const Cursor& c) __attribute__((always_inline)) {
    const char* xr = reinterpret_cast<const char*>(xw + __builtin_amdgcn_readlane(mine.row, c.s) * a.cx + max(min(c.k * 32, a.cx - 32), 0));
#pragma unroll
    for (int i = 0; i < 2 * NT; ++i) raw[i] = *reinterpret_cast<const f32x4*>(xr + at[i]);
  };
  auto put_x = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < 2 * NT; ++i) mine_x[i * 64 + lane] = raw[i];
  };
  constexpr int PER = (CHUNK + 255) / 256;
  u32x4 wreg[RW][PER];
#pragma unroll
  for (int w = 0; w < RW; ++w)
#pragma unroll
    for (int i = 0; i < PER; ++i) wreg[w][i] = u32x4{0, 0, 0, 0};
  auto load_w = [&](const Cursor& c) __attribute__((always_inline)) {
#pragma unroll
    for (int w = 0; w < RW; ++w) {
      const int b = __builtin_amdgcn_readlane(mine.block[w], c.s);
      if (b >= 0) {
        const u32x4* src = a.packed + ((int64_t)(b * a.cblocks + cb) * a.kc + c.k) * CHUNK;
#pragma unroll
        for (int i = 0; i < PER; ++i)
          if (PER * 256 == CHUNK || tid + i * 256 < CHUNK) wreg[w][i] = src[(unsigned)(tid + i * 256)];
      }
    }
  };
  auto put_w = [&](int buf) __attribute__((always_inline)) {
#pragma unroll
    for (int w = 0; w < RW; ++w)
#pragma unroll
      for (int i = 0; i < PER; ++i)
        if (PER * 256 == CHUNK || tid + i * 256 < CHUNK) lds[buf][w][tid + i * 256] = wreg[w][i];
  };

  clear();
  unsigned plain = plain_w;
  int s_first = 0;                                   // of the rows in work
  Cursor cx{0, 0}, cw{0, 0}, now{0, 0};
  load_w(cw);
  advance(cw);
  load_x(cx);
  advance(cx);
  put_w(0);
  put_x();
  load_x(cx);
  advance(cx);
  load_w(cw);
  advance(cw);
  __syncthreads();
  for (int u = 0; u < units; ++u) {
    UvsParts<8> part[NT];
    float low = 1.f;
    f32x4 v[NT][2];
#pragma unroll
    for (int i = 0; i < NT; ++i)
#pragma unroll
      for (int h = 0; h < 2; ++h) v[i][h] = mine_x[(16 * i + r) * 8 + ((2 * q + h) ^ (r & 7))];
    put_x();
    load_x(cx);
    advance(cx);
#pragma unroll
    for (int i = 0; i < NT; ++i)
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int k = 0; k < 4; k += 2) {
          const float v0 = v[i][h][k], v1 = v[i][h][k + 1];
          part[i].pair(2 * h + k / 2, v0, v1);
          low = uvs_least(v0, v1, low);
        }
    if (__any(low < 0x1p-110f)) {                    // a zero, as a rule
#pragma unroll
      for (int i = 0; i < NT; ++i)
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
          for (int k = 0; k < 4; ++k) {
            const float e = v[i][h][k];
            plain |= uvs_asks(e) & kUvsPlain;
          }
    }
    put_w((u + 1) & 1);
    load_w(cw);
    advance(cw);
#pragma unroll
    for (int w = 0; w < RW; ++w) {
      if (__builtin_amdgcn_readlane(mine.block[w], now.s) >= 0) {
        const u32x4* frag = lds[u & 1][w] + lane;
#pragma unroll
        for (int t = 0; t < TW; ++t) {
          bf16x8 f[3];
#pragma unroll
          for (int h = 0; h < 3; ++h) f[h] = __builtin_bit_cast(bf16x8, frag[(h * TW + t) * 64]);
          floatx4 sum[NT];
          if constexpr (BY_UNIT) {
#pragma unroll
            for (int i = 0; i < NT; ++i) sum[i] = floatx4{0.f, 0.f, 0.f, 0.f};
          }
#pragma unroll
          for (int c = 0; c < 6; ++c) {              // the small products first
            constexpr int ha[6] = {2, 1, 0, 1, 0, 0}, hb[6] = {0, 1, 2, 0, 1, 0};
#pragma unroll
            for (int i = 0; i < NT; ++i) {
              floatx4& to = BY_UNIT ? sum[i] : acc[w][t][i];
              to = __builtin_amdgcn_mfma_f32_16x16x32_bf16(f[ha[c]], uvs_frag(part[i].p[hb[c]]), to, 0, 0, 0);
            }
          }
          if constexpr (BY_UNIT) {
#pragma unroll
            for (int i = 0; i < NT; ++i) acc[w][t][i] += sum[i];
          }
        }
      }
    }
    const int end = __builtin_amdgcn_readlane(mine.task, now.s);
    if (end >= 0 && now.k == a.kc - 1) {             // the last unit of these rows
      const cgtp_uvl_task task = a.tasks[end];
#pragma unroll
      for (int w = 0; w < RW; ++w)
#pragma unroll
        for (int t = 0; t < TW; ++t)
#pragma unroll
          for (int i = 0; i < NT; ++i)
#pragma unroll
            for (int k = 0; k < 4; ++k) {
              const float v = acc[w][t][i][k];
              plain |= v - v != 0.f;
            }
      if (__any(plain)) form_plain(s_first, now.s);
#pragma unroll
      for (int w = 0; w < RW; ++w) {
        if (task.row[w] < 0 || first >= a.n_rows) continue;
#pragma unroll
        for (int i = 0; i < NT; ++i) {
          if (16 * i + r < left) {
            float* o = a.out + ((n0 + 16 * i + r) * a.dout + task.row[w]) * a.cout;
#pragma unroll
            for (int t = 0; t < TW; ++t) {
              const int ch = cb * 16 * TW + 16 * t + 4 * q;
              if (ch < a.cout) *reinterpret_cast<floatx4*>(o + ch) = acc[w][t][i];
            }
          }
        }
      }
      clear();
      plain = plain_w;
      s_first = now.s + 1;
    }
    advance(now);
    __syncthreads();
  }
}

// ---- gradient of the weight: gW[p, k, w] = sum_n sum_{entries e of p} coef_e * x[n, a_e, k] * g[n, m_e, w] ---------------------
struct UvlGwDev {
  const float* x;
  const float* g;
  float* part;                        // (n_chunks, n_paths, cx, cout)
  const cgtp_uvl_pair* pairs;
  const int32_t* path_ptr;
  int64_t n_rows;
  int n_paths, dx, dg, cx, cout, chunk, n_chunks, kblocks, wblocks;
};

// A wavefront owns a block of 16 TI x 16 TJ of a path's gradient and a chunk of samples by itself, as uvt_grad_w_small_kernel does: what
// it loads of 32 samples (TI or TJ consecutive channels of eight samples a lane) is the layout of the matrix operands, so nothing is
// exchanged and there is no barrier.  The four wavefronts of a workgroup have four paths in a row: the (w_+, w_-) pairs of an
// SO(2) layer read the same rows, the second time from the L1; the paths of a chunk run on one XCD.
// What bounds it: splitting both operands (64 elements a lane and 32 samples: 390 vector instructions next to 96 matrix ones of 16
// cycles) and the rows from L2.  SO2Linear, lmax 4, 64 channels, 32768 samples 548 -> 346 us, 1000 samples 36 -> 30; IrrepsLinear 64 -> 64,
// lmax 2, 65536 samples 118 -> 84, 128 -> 128, lmax 3, 32768 samples 241 -> 219.
template <int TI, int TJ>
__global__ void __launch_bounds__(256, 2) uvl_gw_kernel(const UvlGwDev a) {
  typedef typename VecOf<float, TI>::type VI;
  typedef typename VecOf<float, TJ>::type VJ;
  const int lane = threadIdx.x & (kWave - 1), wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave), r = lane & 15, q = lane >> 4;
  const int groups = (a.n_paths + 3) / 4, parts = groups * a.kblocks * a.wblocks, j = blockIdx.x >> 3;
  const int at = j % parts, chunk = j / parts * 8 + (blockIdx.x & 7), p = at % groups * 4 + wave;
  if (chunk >= a.n_chunks || p >= a.n_paths) return;
  const int k0 = at / groups % a.kblocks * (16 * TI), w0 = at / groups / a.kblocks * (16 * TJ);
  const int64_t n_begin = (int64_t)chunk * a.chunk, n_end = min(n_begin + a.chunk, a.n_rows);
  const int kc = min(k0 + TI * r, a.cx - TI), wc = min(w0 + TJ * r, a.cout - TJ);      // channels past the last are not stored
  const int xs = a.dx * a.cx, gs = a.dg * a.cout, e0 = a.path_ptr[p], entries = a.path_ptr[p + 1] - e0;
  const int steps = (int)((n_end - n_begin + 31) / 32), units = steps * entries;
  floatx4 acc[TI][TJ];
  auto clear = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < TI; ++i)
#pragma unroll
      for (int t = 0; t < TJ; ++t) acc[i][t] = floatx4{0.f, 0.f, 0.f, 0.f};
  };
  clear();
  unsigned plain = 0;
  if (units > 0) {
    // lane l holds entry l of the path (64 at most)
    const cgtp_uvl_pair mine = a.pairs[e0 + min(lane, entries - 1)];
    auto coef_of = [&](int e) __attribute__((always_inline)) {
      return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, mine.coef), e));
    };
    const unsigned xat = 4u * (unsigned)(8 * q * xs + kc), gat = 4u * (unsigned)(8 * q * gs + wc);
    VI xr[8];
    VJ gr[8];
    auto load = [&](int step, int e) __attribute__((always_inline)) {
      const int64_t n0 = n_begin + (int64_t)step * 32;
      const char* xrow = reinterpret_cast<const char*>(a.x + n0 * xs + __builtin_amdgcn_readlane(mine.row_x, e) * a.cx);
      const char* grow = reinterpret_cast<const char*>(a.g + n0 * gs + __builtin_amdgcn_readlane(mine.row_g, e) * a.cout);
      if (n0 + 32 <= n_end) {
#pragma unroll
        for (int i = 0; i < 8; ++i) xr[i] = *reinterpret_cast<const VI*>(xrow + (int64_t)i * xs * 4 + xat);
#pragma unroll
        for (int i = 0; i < 8; ++i) gr[i] = *reinterpret_cast<const VJ*>(grow + (int64_t)i * gs * 4 + gat);
      } else {
        int left = (int)(n_end - n0);
        asm volatile("" : "+v"(left));                 // its addresses are not kept around the loop
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          const int n = 8 * q + i, nc = min(n, left - 1);
          const VI u = *reinterpret_cast<const VI*>(xrow + 4u * (unsigned)(nc * xs + kc));
          const VJ v = *reinterpret_cast<const VJ*>(grow + 4u * (unsigned)(nc * gs + wc));
#pragma unroll
          for (int k = 0; k < TI; ++k) xr[i][k] = n < left ? u[k] : 0.f;
#pragma unroll
          for (int k = 0; k < TJ; ++k) gr[i][k] = n < left ? v[k] : 0.f;
        }
      }
    };
    int step = 0, e = 0;
    load(0, 0);
    for (int u = 0; u < units; ++u) {
      const float sign = u & 1 ? -1.f : 1.f, c = sign * coef_of(e);
      UvsParts<8> xp[TI];
      VJ gv[8];
      float low = 1.f;
#pragma unroll
      for (int i = 0; i < TI; ++i)
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          const float v0 = c * xr[2 * k][i], v1 = c * xr[2 * k + 1][i];
          xp[i].pair(k, v0, v1);
          low = uvs_least(v0, v1, low);
        }
#pragma unroll
      for (int k = 0; k < 8; ++k) gv[k] = gr[k];
#pragma unroll
      for (int k = 0; k < 8; k += 2)
#pragma unroll
        for (int t = 0; t < TJ; ++t) {
          const float v0 = gv[k][t], v1 = gv[k + 1][t];
          low = uvs_least(v0, v1, low);
        }
      if (__any(low < 0x1p-110f)) {                    // a zero, as a rule
#pragma unroll
        for (int k = 0; k < 8; ++k) {
#pragma unroll
          for (int i = 0; i < TI; ++i) {
            const float v = c * xr[k][i];
            plain |= uvs_asks(v) & kUvsPlain;
          }
#pragma unroll
          for (int t = 0; t < TJ; ++t) {
            const float v = gv[k][t];
            plain |= uvs_asks(v) & kUvsPlain;
          }
        }
      }
      if (++e == entries) {
        e = 0;
        ++step;
      }
      if (u + 1 < units) load(step, e);
#pragma unroll
      for (int t = 0; t < TJ; ++t) {
        UvsParts<8> gp;
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          const float v0 = gv[2 * k][t], v1 = gv[2 * k + 1][t];
          gp.pair(k, v0, v1);
        }
        // The products of 32 samples are summed by themselves, every other time with the sign turned: the matrix instruction rounds
        // downwards, which in a sum over many samples is no small part of the error (IrrepsLinear 64 -> 64, 65536 samples: all
        // parts added to the chunk's sums 7.2e-7, by themselves 6.0e-7, with alternating signs 2.3e-7; fp32 instructions 4.5e-7).
        floatx4 sum[TI];
#pragma unroll
        for (int i = 0; i < TI; ++i) sum[i] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int h = 0; h < 6; ++h) {                  // the small products first
          constexpr int ha[6] = {2, 1, 0, 1, 0, 0}, hb[6] = {0, 1, 2, 0, 1, 0};
#pragma unroll
          for (int i = 0; i < TI; ++i)
            sum[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(uvs_frag(xp[i].p[ha[h]]), uvs_frag(gp.p[hb[h]]), sum[i], 0, 0, 0);
        }
#pragma unroll
        for (int i = 0; i < TI; ++i) acc[i][t] += sign * sum[i];
      }
    }
#pragma unroll
    for (int i = 0; i < TI; ++i)
#pragma unroll
      for (int t = 0; t < TJ; ++t)
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          const float v = acc[i][t][k];
          plain |= v - v != 0.f;
        }
    if (__any(plain)) {                                // fp32 matrix instructions, operands from memory
      clear();
      for (int s = 0; s < entries; ++s) {
        const float c = coef_of(s);
        const float* xrow = a.x + __builtin_amdgcn_readlane(mine.row_x, s) * a.cx + kc;
        const float* grow = a.g + __builtin_amdgcn_readlane(mine.row_g, s) * a.cout + wc;
        for (int64_t n0 = n_begin; n0 < n_end; n0 += 4) {
          const int64_t n = min(n0 + q, n_end - 1);
          const float f = n0 + q < n_end ? 1.f : 0.f;
          const VI u = *reinterpret_cast<const VI*>(xrow + n * xs);
          const VJ v = *reinterpret_cast<const VJ*>(grow + n * gs);
#pragma unroll
          for (int i = 0; i < TI; ++i) {
            const float ui = f != 0.f ? c * u[i] : 0.f;
#pragma unroll
            for (int t = 0; t < TJ; ++t) {
              const float vt = f != 0.f ? v[t] : 0.f;
              acc[i][t] = __builtin_amdgcn_mfma_f32_16x16x4f32(ui, vt, acc[i][t], 0, 0, 0);
            }
          }
        }
      }
    }
  }
  // element e of tile (i, t): channel TI (4 q + e) + i of the contracted axis's block, TJ r + t of the other's
  float* out = a.part + ((int64_t)chunk * a.n_paths + p) * a.cx * a.cout;
  if (w0 + TJ * r < a.cout) {
#pragma unroll
    for (int i = 0; i < TI; ++i)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int k = k0 + TI * (4 * q + e) + i;
        if (k < a.cx) {
          VJ v;
#pragma unroll
          for (int t = 0; t < TJ; ++t) v[t] = acc[i][t][e];
          *reinterpret_cast<VJ*>(out + (int64_t)k * a.cout + w0 + TJ * r) = v;
        }
      }
  }
}

// Samples per wavefront: 32 or more, at most 8192 wavefronts and as many partial results as the fp32 kernels have: 512 up to 64
// channels, 128 past 64 on both sides (128 x 128, lmax 1, 16000 samples 53 us with 512, 42 with 256, 36 with 128; 65536: 129, 119, 111),
// with 64 on one side 256 (64 x 128: 37, 28 and 34 us; 65536: 73, 64, 103).
static int64_t uvl_gw_chunk(const cgtp_uvl_gw_args* a) {
  const int64_t blocks = (int64_t)((a->cx + 63) / 64) * ((a->cout + 63) / 64) * a->n_paths;
  const int64_t partials = (a->cx > 64 ? 1 : 2) * (a->cout > 64 ? 1 : 2) * 128;
  int64_t chunk = 32;
  while ((a->n_rows + chunk - 1) / chunk > partials || (a->n_rows + chunk - 1) / chunk * blocks > 8192) {
    chunk *= 2;
    if (chunk >= a->n_rows) break;
  }
  return chunk;
}

static int uvl_gw_check(const cgtp_uvl_gw_args* a) {
  if (!a || !a->x || !a->g || !a->gw || !a->pairs || !a->path_ptr) return CGTP_ERR_NULL;
  if (a->n_rows <= 0 || a->n_paths <= 0 || a->dx <= 0 || a->dg <= 0 || a->cx <= 0 || a->cout <= 0 || a->cx % 4 || a->cout % 4 ||
      (int64_t)a->dx * a->cx > 1 << 22 || (int64_t)a->dg * a->cout > 1 << 22 || a->max_pairs > kWave)
    return CGTP_ERR_SHAPE;
  if (((uintptr_t)a->x | (uintptr_t)a->g | (uintptr_t)a->gw | (uintptr_t)a->workspace) & 15u) return CGTP_ERR_ALIGN;
  const int64_t blocks = (int64_t)((a->cx + 63) / 64) * ((a->cout + 63) / 64) * ((a->n_paths + 3) / 4);
  const int64_t chunks = (a->n_rows + uvl_gw_chunk(a) - 1) / uvl_gw_chunk(a);
  return (chunks + 7) / 8 * 8 * blocks < (int64_t)1 << 31 ? CGTP_OK : CGTP_ERR_SHAPE;
}

struct UvlPlan {
  UvlDev dev;
  int tw, nt;
  int64_t grid;
};

static int uvl_tiles(int cout) { return cout % 64 == 0 || cout % 64 > 32 ? 4 : 2; }

static int uvl_plan(const cgtp_uvl_args* a, UvlPlan* p) {
  if (!a || !a->x || !a->packed || !a->w || !a->out || !a->steps || !a->tasks || !a->groups || !a->blocks) return CGTP_ERR_NULL;
  if (a->n_rows < 0 || a->n_blocks <= 0 || a->n_groups <= 0 || a->dx <= 0 || a->dout <= 0 || a->cx <= 0 || a->cout <= 0 || a->cx % 4 ||
      a->cout % 4 || (int64_t)a->dx * a->cx > 1 << 22 || a->rows_per_task < 1 || a->rows_per_task > 2 || a->max_steps > kWave || a->by_unit < 0 ||
      a->by_unit > 1)
    return CGTP_ERR_SHAPE;
  if (((uintptr_t)a->x | (uintptr_t)a->packed | (uintptr_t)a->out) & 15u) return CGTP_ERR_ALIGN;
  p->tw = uvl_tiles(a->cout);
  UvlDev& d = p->dev;
  d.kc = (a->cx + 31) / 32;
  d.cblocks = (a->cout + 16 * p->tw - 1) / (16 * p->tw);
  const int64_t parts = (int64_t)a->n_groups * d.cblocks;
  // samples per workgroup: 256 over the rows, fewer while the launch would have less than two workgroups per compute unit
  p->nt = 4 / a->rows_per_task;
  while (p->nt > 1 && (a->n_rows + 64 * p->nt - 1) / (64 * p->nt) * parts < 512) p->nt /= 2;
  const int64_t samples = 64 * p->nt, sblocks = (a->n_rows + samples - 1) / samples;
  p->grid = (sblocks + 7) / 8 * 8 * parts;
  if (p->grid >= (int64_t)1 << 31 || a->n_blocks > 65535 || d.cblocks > 65535) return CGTP_ERR_SHAPE;
  d.sblocks = (int)sblocks;
  d.x = (const float*)a->x; d.packed = (const u32x4*)a->packed; d.w = (const float*)a->w; d.out = (float*)a->out;
  d.asks = (const unsigned*)(d.packed + (int64_t)a->n_blocks * d.cblocks * d.kc * (p->tw * 192));
  d.steps = a->steps; d.tasks = a->tasks; d.groups = a->groups; d.blocks = a->blocks; d.n_groups = a->n_groups;
  d.n_rows = a->n_rows; d.stride_p = a->stride_p; d.stride_k = a->stride_k; d.stride_c = a->stride_c;
  d.dx = a->dx; d.dout = a->dout; d.cx = a->cx; d.cout = a->cout;
  return CGTP_OK;
}

template <int TW, bool BY_UNIT>
static auto uvl_fn(int nt, int rw) {
  return rw == 2 ? (nt == 2 ? uvl_kernel<TW, 2, 2, BY_UNIT> : uvl_kernel<TW, 1, 2, BY_UNIT>)
                 : nt == 4 ? uvl_kernel<TW, 4, 1, BY_UNIT> : nt == 2 ? uvl_kernel<TW, 2, 1, BY_UNIT> : uvl_kernel<TW, 1, 1, BY_UNIT>;
}

}  // namespace cgtp

using namespace cgtp;

extern "C" {

int64_t cgtp_uvl_packed_bytes(int32_t n_blocks, int32_t cx, int32_t cout) {
  if (n_blocks <= 0 || cx <= 0 || cout <= 0) return 0;
  const int64_t tw = uvl_tiles(cout), cblocks = (cout + 16 * tw - 1) / (16 * tw);
  return n_blocks * cblocks * ((cx + 31) / 32 * (tw * 192 * 16) + 4);
}

int cgtp_uvl_validate(const cgtp_uvl_args* a) {
  UvlPlan p;
  return uvl_plan(a, &p);
}

int cgtp_uvl_apply(const cgtp_uvl_args* a, void* stream) {
  UvlPlan p;
  const int st = uvl_plan(a, &p);
  if (st != CGTP_OK || a->n_rows == 0) return st;
  const UvlDev& d = p.dev;
  hipLaunchKernelGGL(p.tw == 4 ? uvl_pack_kernel<4> : uvl_pack_kernel<2>, dim3((unsigned)a->n_blocks, (unsigned)d.cblocks), dim3(256), 0,
                     (hipStream_t)stream, a->blocks, d.w, (u32x4*)a->packed, (unsigned*)d.asks, d.kc, d.cx, d.cout, d.stride_p,
                     d.stride_k, d.stride_c);
  if (hipGetLastError() != hipSuccess) return CGTP_ERR_LAUNCH;
  void (*fn)(const UvlDev) = p.tw == 4 ? (a->by_unit ? uvl_fn<4, true>(p.nt, a->rows_per_task) : uvl_fn<4, false>(p.nt, a->rows_per_task))
                                       : a->by_unit ? uvl_fn<2, true>(p.nt, a->rows_per_task) : uvl_fn<2, false>(p.nt, a->rows_per_task);
  hipLaunchKernelGGL(fn, dim3((unsigned)p.grid), dim3(256), 0, (hipStream_t)stream, d);
  return hipGetLastError() == hipSuccess ? CGTP_OK : CGTP_ERR_LAUNCH;
}

int64_t cgtp_uvl_grad_w_workspace_bytes(const cgtp_uvl_gw_args* a) {
  if (uvl_gw_check(a) != CGTP_OK) return 0;
  const int64_t chunk = uvl_gw_chunk(a);
  return (a->n_rows + chunk - 1) / chunk * a->n_paths * a->cx * a->cout * 4;
}

int cgtp_uvl_grad_w(const cgtp_uvl_gw_args* a, void* stream) {
  const int st = uvl_gw_check(a);
  if (st != CGTP_OK) return st;
  if (!a->workspace) return CGTP_ERR_WORKSPACE;
  UvlGwDev d;
  d.x = (const float*)a->x; d.g = (const float*)a->g; d.part = (float*)a->workspace;
  d.pairs = a->pairs; d.path_ptr = a->path_ptr;
  d.n_rows = a->n_rows; d.n_paths = a->n_paths; d.dx = a->dx; d.dg = a->dg; d.cx = a->cx; d.cout = a->cout;
  const int64_t chunk = uvl_gw_chunk(a), n_chunks = (a->n_rows + chunk - 1) / chunk;
  d.chunk = (int)chunk;
  d.n_chunks = (int)n_chunks;
  const bool ki = a->cx <= 32, wj = a->cout <= 32;     // two channels a lane where 32 cover the axis
  d.kblocks = ki ? 1 : (a->cx + 63) / 64;
  d.wblocks = wj ? 1 : (a->cout + 63) / 64;
  const int64_t grid = (n_chunks + 7) / 8 * 8 * ((a->n_paths + 3) / 4) * d.kblocks * d.wblocks;
  void (*fn)(const UvlGwDev) = ki ? (wj ? uvl_gw_kernel<2, 2> : uvl_gw_kernel<2, 4>) : wj ? uvl_gw_kernel<4, 2> : uvl_gw_kernel<4, 4>;
  hipLaunchKernelGGL(fn, dim3((unsigned)grid), dim3(256), 0, (hipStream_t)stream, d);
  if (hipGetLastError() != hipSuccess) return CGTP_ERR_LAUNCH;
  return uvt_reduce_chunks((const float*)a->workspace, (float*)a->gw, n_chunks, (int64_t)a->n_paths * a->cx * a->cout, (hipStream_t)stream);
}

}  // extern "C"
