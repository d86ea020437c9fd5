/*
 * One stage of the apply on the vector units: one right-hand side and a few
 * (from 5 to 8 on, by type and stage size, the matrix cores take over,
 * k_applyN_mfma).
 *
 * Bound: HBM, every stored factor entry is read once (16 B in FP64) and
 * meets NR right-hand sides in registers; what the shape of the kernel is
 * about is keeping enough of those reads in flight.
 *
 *  - A lane owns two adjacent rows and every G-th column: R = ceil(m/2)
 *    lanes across the rows, G = 64/R column groups.  Segments are mostly
 *    11-35 rows high; at 17 rows 63 of 64 lanes work and 17 of 18 row slots
 *    are used, where one row a lane used 51 lanes.  The blocks of a row of a
 *    factor are adjacent in memory and their inputs are too, so the plan
 *    merges them into one term and the G columns of a step are one
 *    contiguous piece of up to 2 KiB.
 *    One right-hand side in FP64 at 2^20 points: 12.1 ms, 6.2 TB/s of
 *    factors and vectors, what a plain read reaches here, in processes where
 *    the kernel before this one took 12.7 ms, and 13.7 ms in those where it
 *    took 14.5; FP32 at 2^19: 4.5 -> 3.4 ms; four right-hand sides at 100003
 *    points, before one lane a right-hand side: 37 -> 1.53 ms.
 *  - The columns of all terms are one sequence of steps, kept in a ring of
 *    RING steps in registers: the loads of the next RING - 1 steps are in
 *    flight while a step is multiplied, across term boundaries.  The terms
 *    sit one per lane and are read with readlane, so moving on to the next
 *    term waits for no memory.
 *  - Where a stage has few segments with many columns (the last one, whose
 *    segments sum the blocks of every butterfly over their rows), a
 *    segment's steps are split evenly over the W waves of a block and meet
 *    in LDS, in wave order: the result does not depend on scheduling.
 */
#include "bf_apply.h"

#include <type_traits>

namespace {

typedef float f4u __attribute__((ext_vector_type(4), aligned(8)));

template <bool F64> struct AccT { typedef double2 T; };
template <> struct AccT<false> { typedef float2 T; };

template <typename T> __device__ __forceinline__ T zero2() {
  T z;
  z.x = z.y = 0;
  return z;
}
__device__ __forceinline__ void fma2(double2 &c, double2 a, double2 b) {
  c.x = fma(a.x, b.x, fma(-a.y, b.y, c.x));
  c.y = fma(a.x, b.y, fma(a.y, b.x, c.y));
}
__device__ __forceinline__ void fma2(float2 &c, float2 a, float2 b) {
  c.x = fmaf(a.x, b.x, fmaf(-a.y, b.y, c.x));
  c.y = fmaf(a.x, b.y, fmaf(a.y, b.x, c.y));
}
template <typename A, typename V> __device__ __forceinline__ A widen(V v) {
  A a;
  a.x = v.x;
  a.y = v.y;
  return a;
}
__device__ __forceinline__ int64_t readlane64(int64_t v, int l) {
  const uint32_t lo = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)v, l);
  const uint32_t hi = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)((uint64_t)v >> 32), l);
  return (int64_t)((uint64_t)hi << 32 | lo);
}

/* Workgroups go to the 8 XCDs round-robin by id; here XCD_GROUP adjacent
 * segments' blocks get ids with equal id % 8, so neighbours, which read the
 * same inputs, share an L2 (12.30 -> 12.11 ms at 2^20 points in FP64; groups
 * of 4 or 64 and whole eighths of the grid were slower).  The last ids, short
 * of a whole group per XCD, keep their order. */
constexpr unsigned XCD_GROUP = 16;
__device__ __forceinline__ int64_t xcd_block(unsigned id, unsigned blocks) {
  constexpr unsigned per = 8 * XCD_GROUP;
  if (id >= blocks / per * per) return id;
  const unsigned g = id / per, w = id - g * per;
  return (int64_t)(g * per + (w & 7) * XCD_GROUP + (w >> 3));
}

/* most rows of a segment per pass where its steps are split over waves (the
 * partial sums of W waves share the LDS) */
constexpr int SPLIT_ROWS = 64;

/* waves a segment may be split over: their partial sums fit in 32 KiB */
constexpr int split_max(int nr) { return nr <= 2 ? 16 : nr <= 4 ? 8 : 4; }

template <typename V, bool LO, bool SUM64, int NR, bool SPLIT, int RING>
__global__ __launch_bounds__(SPLIT ? 64 * split_max(NR) : 256) void k_apply_few(const BfkSeg *__restrict__ segs, int64_t numSegs,
                                                                  const BfkTerm *__restrict__ terms,
                                                                  const V *__restrict__ hi, const V *__restrict__ lo,
                                                                  typename BufsOf<V>::T bufs, int nrhs) {
  constexpr bool F32 = std::is_same<V, float2>::value;
  typedef typename AccT<!F32 || SUM64>::T A;
  extern __shared__ double lds[];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), waves = blockDim.x >> 6;
  const int64_t bid = xcd_block(blockIdx.x, gridDim.x);
  const int64_t si = SPLIT ? bid : bid * waves + wave;
  if (si >= numSegs) return; /* the whole block where it has barriers */
  const BfkSeg S = segs[si];
  const int m = S.m;
  if (m <= 0) return;
  const int R = min((m + 1) >> 1, SPLIT ? SPLIT_ROWS / 2 : 64), G = 64 / R;
  const int gl = lane / R, rl = lane - gl * R;
  V *y = bufs.out[S.ybuf] + S.yOff * nrhs;
  for (int cb = 0; cb < nrhs; cb += NR) {
    /* NR <= nrhs: the last chunk moves back over columns already done */
    const int c0 = min(cb, nrhs - NR);
    for (int rb = 0; rb < m; rb += 2 * R) {
      /* the lane's rows.  FP32: two adjacent ones, one 16-byte load of a pair
       * that lies inside the column (a one-row segment loads its row twice);
       * FP64: R rows apart, so that each of the two loads of a column reads
       * one run of 16 R bytes */
      const int i0 = F32 ? rb + 2 * rl : rb + rl, i1 = F32 ? i0 + 1 : i0 + R;
      const int ia = F32 && m > 1 ? min(i0, m - 2) : min(i0, m - 1);
      const int second = min(i1, m - 1) - ia;
      A acc[2][NR];
#pragma unroll
      for (int c = 0; c < NR; ++c) acc[0][c] = acc[1][c] = zero2<A>();
      for (int tb = S.t0; tb < S.t1; tb += 64) {
        /* this chunk's terms, one per lane */
        const int nT = min(64, S.t1 - tb);
        const BfkTerm T = terms[tb + min(lane, nT - 1)];
        const bool block = lane < nT && T.aOff >= 0 && T.n > 0;
        const int64_t tA = T.aOff + T.rowOff;
        const int its = block ? (T.n + G - 1) / G : 0; /* steps of this term */
        int sum = its;                                 /* steps up to and including it */
        /* the sums over the lanes, as far as there are terms: most segments
         * have one or two, and each of the six steps of a whole wave's scan
         * costs an LDS round trip (3 right-hand sides on 30000 points 401 ->
         * 386 us, box of 16384 points 123 -> 120 us) */
        for (int d = 1; d < nT; d <<= 1) {
          const int o = __shfl_up(sum, d, 64);
          if (lane >= d) sum += o;
        }
        sum = lane < nT ? sum : __builtin_amdgcn_readlane(sum, nT - 1);
        const int total = __builtin_amdgcn_readlane(sum, 63);
        const int first = SPLIT ? (int)((int64_t)total * wave / waves) : 0;
        const int count = (SPLIT ? (int)((int64_t)total * (wave + 1) / waves) : total) - first;
        if (count > 0) {
          const uint64_t some = __ballot(its > 0);
          /* the load cursor: term ct, its column cj (uniform) */
          int ct = __ffsll((unsigned long long)__ballot(sum > first)) - 1;
          int cn = __builtin_amdgcn_readlane(T.n, ct), clda = __builtin_amdgcn_readlane(T.lda, ct);
          const V *cA = hi + readlane64(tA, ct), *cL = LO ? lo + readlane64(tA, ct) : nullptr;
          const V *cX = bufs.in[__builtin_amdgcn_readlane(T.xbuf, ct)] + readlane64(T.xOff, ct) * nrhs + c0;
          int cj = (first - (__builtin_amdgcn_readlane(sum, ct) - __builtin_amdgcn_readlane(its, ct))) * G;
          int issued = 0;
          V xa[RING][NR];
          V a64[RING][2], l64[RING][2];
          f4u a32[RING], l32[RING];
          int sj[RING], sn[RING];
          auto issue = [&](int s) {
            const int j = min(cj + gl, cn - 1);
            const int64_t e = (int64_t)j * clda + ia;
            if constexpr (F32) {
              if (m > 1) { /* uniform */
                a32[s] = *(const f4u *)(cA + e);
                if (LO) l32[s] = *(const f4u *)(cL + e);
              } else {
                const V v = cA[e];
                a32[s] = f4u{v.x, v.y, v.x, v.y};
                if (LO) {
                  const V w = cL[e];
                  l32[s] = f4u{w.x, w.y, w.x, w.y};
                }
              }
            } else {
              a64[s][0] = cA[e];
              a64[s][1] = cA[e + second];
            }
            const V *px = cX + (int64_t)j * nrhs;
#pragma unroll
            for (int c = 0; c < NR; ++c) xa[s][c] = px[c];
            sj[s] = cj;
            sn[s] = cn;
            if (++issued < count) { /* past the last step the cursor stays put */
              cj += G;
              if (cj >= cn) {
                ct = __ffsll((unsigned long long)(some & ~((2ull << ct) - 1))) - 1;
                cn = __builtin_amdgcn_readlane(T.n, ct);
                clda = __builtin_amdgcn_readlane(T.lda, ct);
                cA = hi + readlane64(tA, ct);
                if (LO) cL = lo + readlane64(tA, ct);
                cX = bufs.in[__builtin_amdgcn_readlane(T.xbuf, ct)] + readlane64(T.xOff, ct) * nrhs + c0;
                cj = 0;
              }
            }
          };
          auto multiply = [&](int s) {
            A a0, a1;
            if constexpr (F32) {
              float2 h0 = make_float2(a32[s].x, a32[s].y), h1 = make_float2(a32[s].z, a32[s].w);
              if (ia != i0) h0 = h1;
              if constexpr (LO && SUM64) { /* the pair hi + lo in FP64 */
                float2 w0 = make_float2(l32[s].x, l32[s].y), w1 = make_float2(l32[s].z, l32[s].w);
                if (ia != i0) w0 = w1;
                a0.x = (double)h0.x + (double)w0.x;
                a0.y = (double)h0.y + (double)w0.y;
                a1.x = (double)h1.x + (double)w1.x;
                a1.y = (double)h1.y + (double)w1.y;
              } else {
                a0 = widen<A>(h0);
                a1 = widen<A>(h1);
              }
            } else {
              a0 = a64[s][0];
              a1 = a64[s][1];
            }
#pragma unroll
            for (int c = 0; c < NR; ++c) {
              const A x = widen<A>(xa[s][c]);
              if constexpr (LO && !SUM64) { /* plain FP32 sums: the low part first */
                float2 w0 = make_float2(l32[s].x, l32[s].y), w1 = make_float2(l32[s].z, l32[s].w);
                if (ia != i0) w0 = w1;
                fma2(acc[0][c], w0, x);
                fma2(acc[1][c], w1, x);
              }
              fma2(acc[0][c], a0, x);
              fma2(acc[1][c], a1, x);
            }
          };
          auto compute = [&](int s) {
            if (sj[s] + G <= sn[s]) /* uniform: every group has a column */
              multiply(s);
            else if (sj[s] + gl < sn[s])
              multiply(s);
          };
#pragma unroll
          for (int s = 0; s < RING - 1; ++s) issue(s);
          /* whole turns of the ring, then the last steps, already in flight */
          const int turns = count / RING, tail = count - turns * RING;
          for (int u = 0; u < turns; ++u) {
#pragma unroll
            for (int s = 0; s < RING; ++s) {
              issue((s + RING - 1) % RING);
              compute(s);
            }
          }
#pragma unroll
          for (int s = 0; s < RING - 1; ++s)
            if (s < tail) compute(s);
        }
        /* identity terms: the rows of x themselves, once per segment */
        uint64_t id = __ballot(lane < nT && T.aOff < 0);
        if (!SPLIT || wave == 0)
          while (id) {
            const int t = __ffsll((unsigned long long)id) - 1;
            id &= id - 1;
            const V *x = bufs.in[__builtin_amdgcn_readlane(T.xbuf, t)] + readlane64(T.xOff, t) * nrhs + c0;
            if (gl == 0)
#pragma unroll
              for (int c = 0; c < NR; ++c) {
                const V v0 = x[(int64_t)min(i0, m - 1) * nrhs + c], v1 = x[(int64_t)min(i1, m - 1) * nrhs + c];
                acc[0][c].x += v0.x;
                acc[0][c].y += v0.y;
                acc[1][c].x += v1.x;
                acc[1][c].y += v1.y;
              }
          }
      }
      /* the column groups meet: halving the groups, lane (g, r) takes (g + k, r) */
      for (int gs = G; gs > 1;) {
        const int k = (gs + 1) >> 1;
        const int from = (lane + k * R) & 63;
        const bool add = gl + k < gs;
#pragma unroll
        for (int r = 0; r < 2; ++r)
#pragma unroll
          for (int c = 0; c < NR; ++c) {
            const auto ox = __shfl(acc[r][c].x, from, 64);
            const auto oy = __shfl(acc[r][c].y, from, 64);
            if (add) {
              acc[r][c].x += ox;
              acc[r][c].y += oy;
            }
          }
        gs = k;
      }
      if constexpr (SPLIT) {
        A *part = (A *)lds; /* [wave][row of the pass][column] */
        if (gl == 0)
#pragma unroll
          for (int r = 0; r < 2; ++r)
#pragma unroll
            for (int c = 0; c < NR; ++c) part[(wave * 2 * R + (r ? i1 : i0) - rb) * NR + c] = acc[r][c];
        __syncthreads();
        const int outs = min(2 * R, m - rb) * NR;
        for (int e = threadIdx.x; e < outs; e += blockDim.x) {
          A s = part[e];
          for (int w = 1; w < waves; ++w) {
            const A o = part[w * 2 * R * NR + e];
            s.x += o.x;
            s.y += o.y;
          }
          V out;
          out.x = (decltype(out.x))s.x;
          out.y = (decltype(out.y))s.y;
          y[(int64_t)(rb + e / NR) * nrhs + c0 + e % NR] = out;
        }
        __syncthreads(); /* the next pass writes part again */
      } else if (gl == 0) {
#pragma unroll
        for (int r = 0; r < 2; ++r)
          if ((r ? i1 : i0) < m)
#pragma unroll
            for (int c = 0; c < NR; ++c) {
              V out;
              out.x = (decltype(out.x))acc[r][c].x;
              out.y = (decltype(out.y))acc[r][c].y;
              y[(int64_t)(r ? i1 : i0) * nrhs + c0 + c] = out;
            }
      }
    }
  }
}

/* Waves per segment: doubled as long as every wave keeps 128 columns, or 16
 * while the stage has too few waves to fill the chip's 8192 slots (256 CUs x
 * 32).  The last stage of the 65536-point boundary operator (1951 segments
 * of about 2000 columns) took 833 us at one wave each and 160 us split; the
 * last stage at 4096 points (124 segments) 81 and 17 us.  Halving or
 * doubling any of the three numbers changes the applies by under 2%. */
int split_of(int64_t numSegs, const BfkStageShape &sh, int nrCols) {
  const int64_t mean = numSegs > 0 ? sh.cols / numSegs : 0;
  int w = 1;
  while (w < split_max(nrCols)) {
    const int64_t least = numSegs * w < 8192 ? 16 : 128; /* columns a wave keeps */
    if (mean < 2 * w * least) break;
    w *= 2;
  }
  return w;
}

template <typename V, bool LO, bool SUM64, int NR>
hipError_t launch_nr(hipStream_t st, const BfkSeg *segs, int64_t n, const BfkStageShape &sh, const BfkTerm *terms,
                     const V *hi, const V *lo, const typename BufsOf<V>::T &b, int nrhs, int waves) {
  constexpr int RING = NR <= 4 ? 3 : 2; /* one more step in flight costs more waves than it gives */
  const int w = split_of(n, sh, NR);
  if (w > 1) {
    const size_t elem = std::is_same<V, float2>::value && !SUM64 ? 8 : 16;
    const int rows = sh.maxRows < SPLIT_ROWS ? (sh.maxRows + 1) & ~1 : SPLIT_ROWS;
    hipLaunchKernelGGL((k_apply_few<V, LO, SUM64, NR, true, RING>), dim3((unsigned)n), dim3(64 * w),
                       (size_t)w * rows * NR * elem, st, segs, n, terms, hi, lo, b, nrhs);
  } else {
    const int wv = waves > 0 ? waves : 1;
    hipLaunchKernelGGL((k_apply_few<V, LO, SUM64, NR, false, RING>), dim3((unsigned)((n + wv - 1) / wv)),
                       dim3(64 * wv), 0, st, segs, n, terms, hi, lo, b, nrhs);
  }
  return hipGetLastError();
}

/* columns per pass: all of them up to 8, then equal chunks of at most 8 */
template <typename V, bool LO, bool SUM64>
hipError_t launch_v(hipStream_t st, const BfkSeg *segs, int64_t n, const BfkStageShape &sh, const BfkTerm *terms,
                    const V *hi, const V *lo, const typename BufsOf<V>::T &b, int nrhs, int waves) {
  const int chunks = (nrhs + 7) / 8, nr = (nrhs + chunks - 1) / chunks;
#define FEW(N) \
  case N: return launch_nr<V, LO, SUM64, N>(st, segs, n, sh, terms, hi, lo, b, nrhs, waves)
  switch (nr) {
    FEW(1);
    FEW(2);
    FEW(3);
    FEW(4);
    FEW(5);
    FEW(6);
    FEW(7);
    default: return launch_nr<V, LO, SUM64, 8>(st, segs, n, sh, terms, hi, lo, b, nrhs, waves);
  }
#undef FEW
}

/* plain FP32 sums (an option that trades accuracy away, not the default):
 * fewer widths */
template <bool LO>
hipError_t launch_plain(hipStream_t st, const BfkSeg *segs, int64_t n, const BfkStageShape &sh, const BfkTerm *terms,
                        const float2 *hi, const float2 *lo, const BfkBufsF &b, int nrhs, int waves) {
  if (nrhs < 4) return launch_nr<float2, LO, false, 1>(st, segs, n, sh, terms, hi, lo, b, nrhs, waves);
  return launch_nr<float2, LO, false, 4>(st, segs, n, sh, terms, hi, lo, b, nrhs, waves);
}

} // namespace

hipError_t bfk_launch_few(hipStream_t st, const BfkSeg *segs, int64_t numSegs, const BfkStageShape &shape,
                          const BfkTerm *terms, const double2 *arena, const BfkBufs &b, int nrhs, int waves) {
  return launch_v<double2, false, true>(st, segs, numSegs, shape, terms, arena, nullptr, b, nrhs, waves);
}

hipError_t bfk_launch_few_f32(hipStream_t st, const BfkSeg *segs, int64_t numSegs, const BfkStageShape &shape,
                              const BfkTerm *terms, const float2 *hi, const float2 *lo, const BfkBufsF &b, int nrhs,
                              int waves, int sum64) {
  if (!sum64)
    return lo ? launch_plain<true>(st, segs, numSegs, shape, terms, hi, lo, b, nrhs, waves)
              : launch_plain<false>(st, segs, numSegs, shape, terms, hi, nullptr, b, nrhs, waves);
  return lo ? launch_v<float2, true, true>(st, segs, numSegs, shape, terms, hi, lo, b, nrhs, waves)
            : launch_v<float2, false, true>(st, segs, numSegs, shape, terms, hi, nullptr, b, nrhs, waves);
}
