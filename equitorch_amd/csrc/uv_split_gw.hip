// Gradient of a shared weight of the fully connected products in single precision on the half-precision matrix cores:
//
//   gW[p, k, (l,) w] = sum_n sum_{terms t of path p} coef_t * x[n, a_t, k] * y[n, b_t(, l)] * g[n, m_t, w]
//
// for the compiled tables, "uv" (y without channels) and "uvw" (a matrix per channel l of y), as many channels of g as of x.
// Operands are three bf16 parts each, a product six matrix instructions (uv_parts.h).
//
// One of x and g is mixed with y, path by path, into as many rows as the other (plain) one has; of two ways the one with fewer
// products (lmax = 3: 75 products of 128 x 128 per sample instead of 99).  The contraction runs over the samples, 16 per
// matrix instruction: a lane holds eight samples of a channel.
//
// A workgroup owns a path (with "uvw" all its l, up to eight a wavefront), all channels and every so many steps of 16 samples.  A
// wavefront owns 32 mixed channels: it keeps the path's rows of the step in registers (a load takes whole lines), forms
// a mixed row from them, splits it and multiplies it with the plain row, whose parts the wavefronts make together and exchange
// through LDS in fragment order.  So each element is read once per path and step and split once per product.
//
// The steps are cut into ranges, one per XCD at a time, and the workgroups of a range (two wavefronts per SIMD) share the work of its
// paths evenly: path p has 64 shares of its steps (step mod 64), dealt to workgroups by cost.  They walk the range side by
// side, so that its rows come from memory once and then from the XCD's L2.  The sums of some products at a time (24 or 64) are added
// to a slot of the workspace (chains as short as those of the fp32 kernel); the slots are added in their order.
//
// What bounds it: waiting (43 % of the wavefronts' time at two per SIMD: rows from the last-level cache, three quarters of the requests
// that miss the L1 at lmax = 3; barriers), then vector and matrix instructions in about equal parts (250 vector ones to 24 matrix
// ones of 32 cycles per product and wavefront).  One call at a time with its reduction (the kernel alone, lmax 3 1218 -> 744 us, "uvw"
// 1336 -> 846), 128 channels, 32768 samples: lmax 3 1253 -> 855 us, lmax 2 444 -> 318; 4096 samples
// 196 -> 130 and 80 -> 60; "uvw" 32 x 32 -> 32, lmax 2, 32768 samples 1280 -> 855 us, 4096 235 -> 162.  With all sums of one sign, 32 products
// each: lmax 3 5.4e-7 in 935 us, 64: 7.2e-7.  Tables walked at run time
// instead of generated: 1390; one wavefront per l with "uvw": 1300.
//
// Values: as in uv_mix.hip; where a workgroup sees an element that is not to be split, a zero that may be what y left of g (paths
// whose g is mixed), or a sum that is not finite, it forms those sums again with fp32 matrix instructions.  Looking at zeros costs
// nothing where there are none and 2 to 8 % with every other element or sample zero.
#include "uv_parts.h"

#pragma clang fp contract(fast)

namespace cgtp {
namespace {

#include "generated/uv_split_gw_configs.inc"

constexpr int kStep = 16;              // samples of a matrix instruction
constexpr unsigned kLeastY = (127u - 30) << 24;        // 2^-30 as by_magnitude() has it

typedef float floatx16 __attribute__((ext_vector_type(16)));
typedef float floatx8 __attribute__((ext_vector_type(8)));

// A value the compiler takes as new each time: addresses formed from it are not kept in registers around the loops.
__device__ __forceinline__ int opaque(int v) {
  asm volatile("" : "+v"(v));
  return v;
}

// Orders by magnitude, a zero as the largest.
__device__ __forceinline__ unsigned by_magnitude(float v) { return (__builtin_bit_cast(unsigned, v) << 1) - 1u; }

struct UvgDev {
  const float* x;
  const float* y;
  const float* g;
  float* slots;
  const cgtp_uvg_job* jobs;
  const int32_t* job_ptr;              // of the workgroups of a range
  int64_t n_rows, slot_elems;
  int C, L;                            // channels of x and g, of y
  int window;                          // products of one sum
  int n_ranges, n_wgs, n_slots;   // workgroups per range
};

// A sample's terms one by one: the mixed side as it is, times the plain side with the coupling.
template <int TB>
struct MixTerm {
  const float* ys;
  int64_t stride;
  const float* row;
  int C;
  bool live;
  const float (&plain)[TB];
  floatx16 (&acc)[TB];
  __device__ __forceinline__ float y(int b) const { return ys[b * stride]; }
  __device__ __forceinline__ void add(int o, float s) const {
    const float v = live ? row[o * C] : 0.f;
#pragma unroll
    for (int tb = 0; tb < TB; ++tb) {
      const float w = live ? s * plain[tb] : 0.f;
      acc[tb] = __builtin_amdgcn_mfma_f32_32x32x2f32(v, w, acc[tb], 0, 0, 0);
    }
  }
  __device__ __forceinline__ void fence() const {}
};

template <int I, int N, class F>
__device__ __forceinline__ void uvg_each(F&& f) {
  if constexpr (I < N) {
    f(std::integral_constant<int, I>{});
    uvg_each<I + 1, N>(f);
  }
}

// TB: tiles of 32 plain channels, at most one per wavefront (NW).  LN > 0 ("uvw"): the wavefront has LN channels l of y, whose
// sums share the rows and the plain row's parts.
template <class CFG, int TB, int NW, int LN>
__global__ void __launch_bounds__(64 * NW, 2) uvg_kernel(const UvgDev a) {
  static_assert(LN == 0 || TB == 1, "channels on y: one tile");
  constexpr bool LV = LN > 0;
  constexpr int CHUNK = TB * 192;                        // 16-byte words of a plain row's parts: [part][tile][lane]
  constexpr int THREADS = 64 * NW, LW = LV ? NW * LN : 1, YN = kStep * CFG::D2, YWORDS = (YN + THREADS - 1) / THREADS;
  constexpr int SETS = LV ? LN : 1;
  __shared__ u32x4 bl[2 * CHUNK];
  __shared__ __align__(16) float yl[LV ? YN * LW : 2 * YN];        // [2: step][row of y][sample], with LV [row][l][sample]
  __shared__ unsigned redo_all;
  // of the y so far, zeros aside; 2^-30 where none is below.  Without channels on y by turns of the steps: the next step's y is noted
  // while some wavefronts still read this one's.
  __shared__ unsigned least_y[LV ? 1 : 2];
  const int tid = threadIdx.x, lane = tid & (kWave - 1), wave = __builtin_amdgcn_readfirstlane(tid / kWave);
  const int r = lane & 31, q = lane >> 5, C = a.C;

  const int range = blockIdx.x % a.n_ranges, wg = blockIdx.x / a.n_ranges;
  const int total = (int)((a.n_rows + kStep - 1) / kStep);
  const int s_begin = (int)((int64_t)total * range / a.n_ranges), s_end = (int)((int64_t)total * (range + 1) / a.n_ranges);
  // this wavefront's 32 mixed channels; channels past the last are others and are not stored
  const int m0 = LV ? 0 : wave * 32, mch = min(m0 + r, C - 1);
  // a thread's channel and eight samples of a plain row
  const bool makes = TB == NW || tid < TB * 64;
  const int pc = tid % (32 * TB), oct = tid / (32 * TB), pcol = min(pc, C - 1);
  u32x4* const plain_to = bl + (pc >> 5) * 64 + oct * 32 + (pc & 31);

  if (tid < (LV ? 1 : 2)) least_y[tid] = kLeastY;        // the first window's barrier is behind it

  for (int job = a.job_ptr[wg]; job < a.job_ptr[wg + 1]; ++job) {
    const cgtp_uvg_job J = a.jobs[job];
    const uint64_t mask = (uint64_t)(unsigned)J.mask_low | (uint64_t)(unsigned)J.mask_high << 32;
    auto next_step = [&](int s) __attribute__((always_inline)) {         // the first of this job's after s
      const int at = (s + 1 - s_begin) & 63;
      const uint64_t ahead = mask >> at | (at ? mask << (64 - at) : 0);
      return min(s + 1 + __builtin_ctzll(ahead), s_end);
    };
    CFG::path(J.path, [&](auto path) __attribute__((always_inline)) {
      using PATH = decltype(path);
      constexpr int NO = PATH::NO, NR = PATH::NR, DM = PATH::SWAPPED ? CFG::DO : CFG::D1, DP = PATH::SWAPPED ? CFG::D1 : CFG::DO;
      const float* mx = (PATH::SWAPPED ? a.g : a.x) + PATH::O0 * C;
      const float* pl = (PATH::SWAPPED ? a.x : a.g) + PATH::R0 * C;
      const unsigned mixed_at = 4u * (unsigned)(8 * q * DM * C + mch), plain_at = 4u * (unsigned)(8 * oct * DP * C + pcol);
      floatx16 acc[SETS][TB];
      floatx8 raw[NO], praw;
      unsigned redo = 0;
      auto clear = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < SETS; ++i)
#pragma unroll
          for (int t = 0; t < TB; ++t)
#pragma unroll
            for (int e = 0; e < 16; ++e) acc[i][t][e] = 0.f;
      };
      auto load_mixed = [&](int s) __attribute__((always_inline)) {
        const int64_t n0 = (int64_t)s * kStep;
        const char* row = reinterpret_cast<const char*>(mx + n0 * DM * C);
        if (n0 + kStep <= a.n_rows) {
#pragma unroll
          for (int o = 0; o < NO; ++o)
#pragma unroll
            for (int j = 0; j < 8; ++j) raw[o][j] = *reinterpret_cast<const float*>(row + (int64_t)(j * DM + o) * C * 4 + mixed_at);
        } else {
          const int left = opaque((int)(a.n_rows - n0));
#pragma unroll
          for (int o = 0; o < NO; ++o)
#pragma unroll
            for (int j = 0; j < 8; ++j) {
              const float e = *reinterpret_cast<const float*>(row + 4u * (unsigned)((min(8 * q + j, left - 1) * DM + o) * C + mch));
              raw[o][j] = 8 * q + j < left ? e : 0.f;
            }
        }
      };
      auto load_plain = [&](int s, int rr) __attribute__((always_inline)) {
        if (!makes) return;
        const int64_t n0 = (int64_t)s * kStep;
        const char* row = reinterpret_cast<const char*>(pl + (n0 * DP + rr) * C);
        if (n0 + kStep <= a.n_rows) {
#pragma unroll
          for (int j = 0; j < 8; ++j) praw[j] = *reinterpret_cast<const float*>(row + (int64_t)j * DP * C * 4 + plain_at);
        } else {
          const int left = opaque((int)(a.n_rows - n0));
#pragma unroll
          for (int j = 0; j < 8; ++j) {
            const float e = *reinterpret_cast<const float*>(row + 4u * (unsigned)(min(8 * oct + j, left - 1) * DP * C + pcol));
            praw[j] = 8 * oct + j < left ? e : 0.f;
          }
        }
      };
      // `zeros` looks at a v with elements of next to nothing, zeros as a rule.
      auto split = [&](const floatx8& v, UvsParts<8>& part, auto&& zeros) __attribute__((always_inline)) {
        float low = 1.f;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const float v0 = v[2 * j], v1 = v[2 * j + 1];
          part.pair(j, v0, v1);
          low = uvs_least(v0, v1, low);
        }
        if (__any(low < 0x1p-110f)) {
#pragma unroll
          for (int j = 0; j < 8; ++j) {
            const float e = v[j];
            redo |= uvs_asks(e) & kUvsPlain;
          }
          zeros(v);
        }
      };
      // Coupled to g first, y may take a product below the smallest number where x would have kept it above.  A zero is that only
      // next to a g and a y of a product below 2^-110 (a sum of terms in y cancels to no less than 2^-35 of them).
      auto look_at_zero = [&](unsigned zero, int ybuf) __attribute__((always_inline)) {
        if (!PATH::SWAPPED || !__any(zero)) return;
        unsigned least = ~0u;
#pragma unroll
        for (int o = 0; o < NO; ++o)
#pragma unroll
          for (int j = 0; j < 8; ++j) {
            const float e = raw[o][j];
            least = min(least, by_magnitude(__builtin_bit_cast(float, opaque(__builtin_bit_cast(int, e)))));
          }
        const float g = __builtin_bit_cast(float, least >> 1), y = __builtin_bit_cast(float, least_y[LV ? 0 : ybuf] >> 1);
        redo |= zero && g * y < 0x1p-110f;               // no g but zeros: not a number, and not below
      };
      auto put_plain = [&](int buf) __attribute__((always_inline)) {
        if (!makes) return;
        UvsParts<8> part;
        split(praw, part, [](const floatx8&) {});
#pragma unroll
        for (int h = 0; h < 3; ++h)
          plain_to[buf * CHUNK + h * TB * 64] = u32x4{part.p[h][0], part.p[h][1], part.p[h][2], part.p[h][3]};
      };
      // The rows of y of a step.  Without channels i = (sample, row) and a step ahead; with them sample by sample, when the step
      // begins (it lasts several thousand cycles).
      float yreg[YWORDS];
      auto note_y = [&](unsigned least, int buf) __attribute__((always_inline)) {       // read past the barrier behind it
        if (PATH::SWAPPED && least < kLeastY) atomicMin(&least_y[buf], least);
      };
      auto load_y = [&](int s) __attribute__((always_inline)) {
        const int64_t n0 = (int64_t)s * kStep, last = min(a.n_rows - n0, (int64_t)kStep) * CFG::D2;
        if constexpr (LV) {
          const int per = a.L / 4, total = YN * per;
          unsigned least = ~0u;
          for (int i = tid; i < total; i += THREADS) {
            const int e = i / per, l4 = i - e * per;
            const f32x4 v = *reinterpret_cast<const f32x4*>(a.y + (n0 * CFG::D2 + (e < last ? e : 0)) * a.L + l4 * 4);
#pragma unroll
            for (int k = 0; k < 4; ++k) yl[(e % CFG::D2 * LW + l4 * 4 + k) * kStep + e / CFG::D2] = v[k];
            least = min(min(least, by_magnitude(v[0])), min(by_magnitude(v[1]), min(by_magnitude(v[2]), by_magnitude(v[3]))));
          }
          note_y(least, 0);
        } else {
#pragma unroll
          for (int k = 0; k < YWORDS; ++k) {
            const int i = opaque(k * THREADS + tid);
            if (i < YN) yreg[k] = a.y[n0 * CFG::D2 + (i < last ? i : 0)];
          }
        }
      };
      auto put_y = [&](int buf) __attribute__((always_inline)) {
        unsigned least = ~0u;
#pragma unroll
        for (int k = 0; k < YWORDS; ++k) {
          const int i = opaque(k * THREADS + tid);
          if (i < YN) yl[buf * YN + i % CFG::D2 * kStep + i / CFG::D2] = yreg[k];
          if (i < YN) least = min(least, by_magnitude(yreg[k]));
        }
        note_y(least, buf);
      };
      struct Mix {
        const float* ys;
        const floatx8* raw;
        floatx8 v;
        __device__ __forceinline__ floatx8 y(int b) const {
          const f32x4 y0 = *reinterpret_cast<const f32x4*>(ys + b * LW * kStep), y1 = *reinterpret_cast<const f32x4*>(ys + b * LW * kStep + 4);
          return __builtin_shufflevector(y0, y1, 0, 1, 2, 3, 4, 5, 6, 7);
        }
        __device__ __forceinline__ void add(int o, const floatx8& s) { v += s * raw[o]; }
        // Between every two terms: with all rows of y of a product read ahead the registers do not hold them.
        __device__ __forceinline__ void fence() const {
          asm volatile("" ::: "memory");
          __builtin_amdgcn_sched_barrier(0);
        }
      };
      struct MixOne {                                    // of one sample, from memory
        const float* ys;
        int64_t stride;
        const float* row;
        int C;
        float v;
        __device__ __forceinline__ float y(int b) const { return ys[b * stride]; }
        __device__ __forceinline__ void add(int o, float s) { v += s * row[o * C]; }
        __device__ __forceinline__ void fence() const {}
      };

      float* out = a.slots + ((int64_t)range * a.n_slots + J.slot) * a.slot_elems;
      bool first = true;
      // The matrix instruction rounds downwards: sums turn their sign from one to the next, of a job and over the workgroups and ranges.
      float sign = (range + wg) & 1 ? -1.f : 1.f;
      int s = next_step(s_begin - 1);
      do {
        // a window: a few steps of the job
        const int STEPS = max(a.window / NR, 1);
        const int s_window = s;
        clear();
        __syncthreads();                                 // LDS and redo_all of the window before
        if (tid == 0) redo_all = 0;
        if (s < s_end) {
          int buf = 0, ybuf = 0, sn = next_step(s);
          load_y(s);
          load_plain(s, 0);
          load_mixed(s);
          if (!LV) put_y(0);
          put_plain(0);
          if (NR > 1) load_plain(s, 1 % NR);
          else if (sn < s_end) load_plain(sn, 0);
          __syncthreads();
          for (int k = 0;; ++k) {
            const bool more = k + 1 < STEPS && sn < s_end;
            const int s2 = NR == 1 ? next_step(sn) : 0;
            uvg_each<0, NR>([&](auto index) __attribute__((always_inline)) {
              constexpr int R = decltype(index)::value;
              bf16x8 f[3];
              auto fragments = [&](int tb) __attribute__((always_inline)) {
                const u32x4* frag = bl + buf * CHUNK + lane;
#pragma unroll
                for (int h = 0; h < 3; ++h) f[h] = __builtin_bit_cast(bf16x8, frag[(h * TB + tb) * 64]);
              };
              if (LV) fragments(0);
              unsigned zero = 0;                         // a mixed element is zero
#pragma unroll
              for (int i = 0; i < SETS; ++i) {
                if (LV && wave * LN + i >= a.L) continue;
                Mix m{yl + (LV ? (wave * LN + i) * kStep : ybuf * YN) + 8 * q, raw, floatx8{0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f}};
                PATH::template mix<R>(m);
                UvsParts<8> part;
                split(sign * m.v, part, [&](const floatx8& v) __attribute__((always_inline)) {
#pragma unroll
                  for (int j = 0; j < 8; ++j) zero |= v[j] == 0.f;
                });
                if (!LV) look_at_zero(zero, ybuf);
                __builtin_amdgcn_sched_barrier(0);
                if (i == SETS - 1) {
                  if (!LV && R == 0 && more) load_y(sn);
                  if (!LV && R == NR - 1 && more) load_mixed(sn);
                }
#pragma unroll
                for (int tb = 0; tb < TB; ++tb) {
                  if (!LV) fragments(tb);
#pragma unroll
                  for (int c = 0; c < 6; ++c) {          // the small products first
                    constexpr int ha[6] = {2, 1, 0, 1, 0, 0}, hb[6] = {0, 1, 2, 0, 1, 0};
                    acc[i][tb] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(uvs_frag(part.p[ha[c]]), f[hb[c]], acc[i][tb], 0, 0, 0);
                  }
                }
              }
              if (LV) look_at_zero(zero, 0);
              if (LV && R == NR - 1 && more) load_mixed(sn);
              __builtin_amdgcn_sched_barrier(0);
              // the plain row of the next product, and the request for the one after
              if (R + 1 < NR || more) put_plain(buf ^ 1);
              if (R + 2 < NR) load_plain(s, (R + 2) % NR);
              else if (NR > 1 ? more : s2 < s_end) load_plain(NR > 1 ? sn : s2, NR > 1 ? (R + 2) % NR : 0);
              if (!LV && R == 0 && more) put_y(ybuf ^ 1);
              buf ^= 1;
              __syncthreads();
            });
            s = sn;
            if (!more) break;
            sn = NR == 1 ? s2 : next_step(s);
            ybuf ^= 1;
            if (LV) {
              load_y(s);                                 // every wavefront is past the barrier behind its reads
              __syncthreads();
            }
          }
        } else {
          __syncthreads();
        }
#pragma unroll
        for (int i = 0; i < SETS; ++i)
#pragma unroll
          for (int t = 0; t < TB; ++t)
#pragma unroll
            for (int e = 0; e < 16; ++e) {
              const float v = acc[i][t][e];
              redo |= v - v != 0.f;
            }
        if (__any(redo) && lane == 0) atomicOr(&redo_all, 1u);
        redo = 0;
        __syncthreads();
        const bool again = redo_all;
        if (again) {                                     // fp32 matrix instructions, operands from memory
          clear();
          int sp = s_window;
          for (int k = 0; k < STEPS && sp < s_end; ++k, sp = next_step(sp)) {
            uvg_each<0, NR>([&](auto index) __attribute__((always_inline)) {
              constexpr int R = decltype(index)::value;
#pragma nounroll
              for (int j = 0; j < 8; ++j) {
                const int64_t n = (int64_t)sp * kStep + 8 * opaque(q) + j, nc = min(n, a.n_rows - 1);
                const float* row = pl + (nc * DP + R) * C;
                float e[TB];
#pragma unroll
                for (int tb = 0; tb < TB; ++tb) e[tb] = n < a.n_rows ? row[min(tb * 32 + r, C - 1)] : 0.f;
#pragma unroll
                for (int i = 0; i < SETS; ++i) {
                  const int l = LV ? min(wave * LN + i, a.L - 1) : 0;
                  const float* ys = a.y + nc * CFG::D2 * a.L + l;
                  if constexpr (PATH::SWAPPED) {
                    // the coupling goes to x here as well, term by term: what overflows is what does in the fp32 kernel
                    PATH::template mix<R>(MixTerm<TB>{ys, a.L, mx + nc * DM * C + mch, C, n < a.n_rows, e, acc[i]});
                  } else {
                    MixOne m{ys, a.L, mx + nc * DM * C + mch, C, 0.f};
                    PATH::template mix<R>(m);
                    const float v = n < a.n_rows ? m.v : 0.f;
#pragma unroll
                    for (int tb = 0; tb < TB; ++tb) acc[i][tb] = __builtin_amdgcn_mfma_f32_32x32x2f32(v, e[tb], acc[i][tb], 0, 0, 0);
                  }
                }
              }
            });
          }
        }
        // element e of a tile: mixed channel 8 (e / 4) + 4 q + e % 4 of the wavefront's 32, plain channel r of the tile's
        // A slot is [mixed channel][l][plain channel] whichever side is mixed: whole lines here, turned by the reduction.
        const int r_now = opaque(r), q_now = opaque(q);
        const float turn = again ? 1.f : sign;
#pragma unroll
        for (int i = 0; i < SETS; ++i) {
          const int l = LV ? wave * LN + i : 0;
          if (LV && l >= a.L) continue;
#pragma unroll
          for (int tb = 0; tb < TB; ++tb) {
            const int c = tb * 32 + r_now;
            if (c < C) {
#pragma unroll
              for (int e = 0; e < 16; ++e) {
                const int mc = m0 + 8 * (e >> 2) + 4 * q_now + (e & 3);
                if (mc < C) {
                  float* at = out + (mc * a.L + l) * C + c;
                  *at = first ? turn * acc[i][tb][e] : *at + turn * acc[i][tb][e];
                }
              }
            }
          }
        }
        first = false;
        sign = -sign;
      } while (s < s_end);
    });
  }
}

// gw[p] = sum over the ranges and slots of path p, in their order: a thread owns four elements of the slots, a wavefront every
// fourth range.  swapped: a bit per path, whose slots are turned.
__global__ void __launch_bounds__(256) uvg_reduce_kernel(const float* __restrict__ slots, const int32_t* __restrict__ slot_ptr,
                                                         float* __restrict__ gw, int n_ranges, int n_slots, int C, int L, uint32_t swapped) {
  __shared__ f32x4 sums[4][kWave];
  const int64_t elems4 = (int64_t)C * L * C / 4;
  const int lane = threadIdx.x & (kWave - 1), slice = threadIdx.x / kWave;
  const int64_t i = min((int64_t)blockIdx.x * kWave + lane, elems4 - 1);
  const int p = blockIdx.y, begin = slot_ptr[p], count = slot_ptr[p + 1] - begin;
  f32x4 sum = {0.f, 0.f, 0.f, 0.f};
  for (int g = slice; g < n_ranges; g += 4) {
    const f32x4* src = reinterpret_cast<const f32x4*>(slots) + ((int64_t)g * n_slots + begin) * elems4 + i;
    int s = 0;
    for (; s + 4 <= count; s += 4) {
      const f32x4 v0 = src[0], v1 = src[elems4], v2 = src[2 * elems4], v3 = src[3 * elems4];
      src += 4 * elems4;
      sum += v0; sum += v1; sum += v2; sum += v3;
    }
    for (; s < count; ++s, src += elems4) sum += *src;
  }
  sums[slice][lane] = sum;
  __syncthreads();
  if (slice == 0 && (int64_t)blockIdx.x * kWave + lane < elems4) {
    for (int k = 1; k < 4; ++k) sum += sums[k][lane];
    float* out = gw + p * elems4 * 4;
    if (swapped >> p & 1) {
      const int e = (int)i * 4, plain = e % C, row = e / C, l = row % L, mixed = row / L;
      for (int k = 0; k < 4; ++k) out[((plain + k) * L + l) * C + mixed] = sum[k];
    } else {
      reinterpret_cast<f32x4*>(out)[i] = sum;
    }
  }
}

using UvgFn = void (*)(const UvgDev);
struct UvgEntry {
  int cfg, p;
  uint32_t swapped;
  UvgFn fn, fn_l;                      // without, with channels on y
};

template <class CFG>
UvgEntry uvg_make(int cfg) {
  UvgEntry e = {cfg, CFG::P, CFG::SWAPPED, nullptr, nullptr};
  if constexpr (CFG::D1 > 4) e.fn = uvg_kernel<CFG, 4, 4, 0>;
  if constexpr (CFG::D1 <= 9) e.fn_l = uvg_kernel<CFG, 1, 4, 8>;
  return e;
}

const UvgEntry* uvg_entry(int cfg) {
#define CGTP_X(INDEX, CFG) uvg_make<CFG>(INDEX),
  static const UvgEntry table[] = {CGTP_FOREACH_UVG_CONFIG(CGTP_X)};
#undef CGTP_X
  for (const UvgEntry& e : table)
    if (e.cfg == cfg) return &e;
  return nullptr;
}

struct UvgPlan {
  UvgDev dev;
  UvgFn fn;
  int paths;
  uint32_t swapped;
  int64_t grid;
};

int uvg_plan(const cgtp_uvg_args* a, UvgPlan* p) {
  if (!a || !a->x || !a->y || !a->g || !a->gw || !a->workspace || !a->jobs || !a->job_ptr || !a->slot_ptr) return CGTP_ERR_NULL;
  const UvgEntry* e = uvg_entry(a->cfg);
  const bool lv = a->cy > 0;
  if (!e || !(lv ? e->fn_l : e->fn)) return CGTP_ERR_CONFIG;
  if (a->n_rows < 0 || a->n_rows > (int64_t)1 << 34 || a->n_wgs <= 0 || a->n_slots <= 0 || a->c <= 0 || a->c % 4 || a->cy < 0 || a->cy % 4 ||
      a->cy > 32 || a->c > (lv ? 32 : 128))
    return CGTP_ERR_SHAPE;
  if (((uintptr_t)a->x | (uintptr_t)a->g | (uintptr_t)a->gw | (uintptr_t)a->workspace | (lv ? (uintptr_t)a->y : 0)) & 15u)
    return CGTP_ERR_ALIGN;
  UvgDev& d = p->dev;
  p->fn = lv ? e->fn_l : e->fn;
  p->paths = e->p;
  p->swapped = e->swapped;
  d.L = lv ? a->cy : 1;
  d.C = a->c;
  const int64_t steps = (a->n_rows + kStep - 1) / kStep;
  // Sums as short as keep the errors at those of the fp32 kernel, whose chunks shrink with the batch and with the table (128
  // channels, relative to 64 bits: lmax 3, 32768 samples 4.6e-7 with 64 products, 7.0e-7 with 256, fp32 6.7e-7; lmax 2, 32768
  // samples 4.5e-7 and 5.8e-7, 8192 samples 3.1e-7 with 32 and fp32; with channels on y 4.5e-7 and 5.8e-7).  Adding a sum to its
  // slot takes as long as several products: lmax 3, 32768 samples 940 us with 32, 855 with 64, 797 with 256.
  d.window = lv || e->p > 11 || a->n_rows >= 16384 ? 64 : 24;
  d.n_ranges = a->n_ranges;
  d.n_wgs = a->n_wgs;
  d.n_slots = a->n_slots;
  p->grid = (int64_t)d.n_ranges * a->n_wgs;
  if (d.n_ranges <= 0 || d.n_ranges > 65535 || p->grid >= (int64_t)1 << 31 || steps >= (int64_t)1 << 30) return CGTP_ERR_SHAPE;
  d.slot_elems = (int64_t)a->c * d.L * a->c;
  d.x = (const float*)a->x; d.g = (const float*)a->g; d.y = (const float*)a->y; d.slots = (float*)a->workspace;
  d.jobs = a->jobs; d.job_ptr = a->job_ptr;
  d.n_rows = a->n_rows;
  return CGTP_OK;
}

}  // namespace
}  // namespace cgtp

using namespace cgtp;

extern "C" {

int cgtp_uvg_validate(const cgtp_uvg_args* a) {
  UvgPlan p;
  return uvg_plan(a, &p);
}

int cgtp_uvg_apply(const cgtp_uvg_args* a, void* stream) {
  UvgPlan p;
  const int st = uvg_plan(a, &p);
  if (st != CGTP_OK) return st;
  hipLaunchKernelGGL(p.fn, dim3((unsigned)p.grid), dim3(256), 0, (hipStream_t)stream, p.dev);
  if (hipGetLastError() != hipSuccess) return CGTP_ERR_LAUNCH;
  const int64_t elems4 = p.dev.slot_elems / 4;
  hipLaunchKernelGGL(uvg_reduce_kernel, dim3((unsigned)((elems4 + kWave - 1) / kWave), (unsigned)p.paths), dim3(256), 0, (hipStream_t)stream,
                     p.dev.slots, a->slot_ptr, (float*)a->gw, p.dev.n_ranges, a->n_slots, p.dev.C, p.dev.L, p.swapped);
  return hipGetLastError() == hipSuccess ? CGTP_OK : CGTP_ERR_LAUNCH;
}

}  // extern "C"
