// k_iir.hip — Triggs-Sdika IIR filtering along one axis in FP64 (gfx950).
//
// Follows _imfilter_dim! (src/imfilter.jl:964-1024) with leftborder!
// (:1027-1048) and rightborder! (:1051-1092): forward recursion with the
// steady-state left initialisation, right-edge initialisation by the 3x3
// matrix M (Triggs & Sdika Eqs. 14-15), backward recursion and scaling.
// Lines of up to 8192 elements run k_iir_line (contiguous axis, through an
// LDS transpose) or k_iir_seg (strided axes): whole lines in registers, the
// axis split into segments of one lane each; short strided lines run
// k_iir_short, one lane per line.  Longer lines run k_iir_rows (contiguous
// axis, LDS-staged chunks) or k_iir_strided (one thread per line).  Lanes sit
// on adjacent lines, which are adjacent in memory for the strided axes
// (coalesced).
#include <type_traits>

#include "ifm_internal.h"

namespace ifm {

#define IFM_GLOBAL __attribute__((address_space(1)))

struct IirArgs {
  const void *src;
  double *dst;        // stage result (the longer lines' kernels also keep forward values there)
  int dt_src;
  int es_src;         // bytes of a source element
  int dt_dst;         // F64, or (register-resident lines only) any floating-point eltype
  int n[MAXD];
  int axis;
  int64_t stride;     // element stride of the filtered axis
  int64_t lines;
  double a[3], b[3], scale, M[9];
  int isfill;
  double fill;
};

// The recursions are sequential along a line, so the inputs of the next
// IC steps are loaded into registers before those steps run (a step never
// waits for its own load).  Reading ahead is safe in place: the forward pass
// only writes positions it has already read, the backward pass likewise.
constexpr int IC = 16;

// Source element as FP64; DT < 0: element type read at run time.
template <int DT>
__device__ __forceinline__ double iir_ld(const IirArgs &p, int64_t i) {
  if constexpr (DT == IFM_F32) return (double)((const float *)p.src)[i];
  else if constexpr (DT == IFM_F64) return ((const double *)p.src)[i];
  else return load_d(p.src, i, (int)p.dt_src);
}

// Line accessor: element i of line `base` with stride `st` (ST1: st == 1, so
// a chunk is contiguous and the loads vectorise).
template <bool ST1, int DT>
__global__ void __launch_bounds__(256) k_iir_strided(IirArgs p) {
  const int64_t line = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (line >= p.lines) return;
  const int n = p.n[p.axis];
  const int64_t st = ST1 ? 1 : p.stride;
  const int64_t pre = line % st, post = line / st;
  const int64_t base = pre + post * st * n;
  const double a1 = p.a[0], a2 = p.a[1], a3 = p.a[2];
  const double b1 = p.b[0], b2 = p.b[1], b3 = p.b[2];
  const double asum = a1 + a2 + a3, bsum = b1 + b2 + b3;
  const double iminus = p.isfill ? p.fill : iir_ld<DT>(p, base);
  const double iplus = p.isfill ? p.fill : iir_ld<DT>(p, base + (int64_t)(n - 1) * st);
  // leftborder!
  const double uminus = iminus / (1 - asum);
  double y0 = iir_ld<DT>(p, base) + a1 * uminus + a2 * uminus + a3 * uminus;
  p.dst[base] = y0;
  double y1 = iir_ld<DT>(p, base + st) + a1 * y0 + a2 * uminus + a3 * uminus;
  p.dst[base + st] = y1;
  double y2 = iir_ld<DT>(p, base + 2 * st) + a1 * y1 + a2 * y0 + a3 * uminus;
  p.dst[base + 2 * st] = y2;
  // forward, omitting the final point
  double ym3 = y0, ym2 = y1, ym1 = y2;
  int i = 3;
  for (; i + IC - 1 <= n - 2; i += IC) {
    double x[IC];
#pragma unroll
    for (int j = 0; j < IC; ++j) x[j] = iir_ld<DT>(p, base + (int64_t)(i + j) * st);
#pragma unroll
    for (int j = 0; j < IC; ++j) {
      const double y = x[j] + a1 * ym1 + a2 * ym2 + a3 * ym3;
      p.dst[base + (int64_t)(i + j) * st] = y;
      ym3 = ym2;
      ym2 = ym1;
      ym1 = y;
    }
  }
  for (; i <= n - 2; ++i) {
    double y = iir_ld<DT>(p, base + (int64_t)i * st) + a1 * ym1 + a2 * ym2 + a3 * ym3;
    p.dst[base + (int64_t)i * st] = y;
    ym3 = ym2;
    ym2 = ym1;
    ym1 = y;
  }
  // rightborder!: the last forward value, then v at and beyond the edge
  const double ylast = iir_ld<DT>(p, base + (int64_t)(n - 1) * st) + a1 * ym1 + a2 * ym2 + a3 * ym3;
  const double uplus = iplus / (1 - asum);
  const double vplus = uplus / (1 - bsum);
  const double d0 = ylast - uplus, d1 = ym1 - uplus, d2 = ym2 - uplus;
  const double v0 = p.M[0] * d0 + p.M[1] * d1 + p.M[2] * d2 + vplus;
  const double v1 = p.M[3] * d0 + p.M[4] * d1 + p.M[5] * d2 + vplus;
  const double v2 = p.M[6] * d0 + p.M[7] * d1 + p.M[8] * d2 + vplus;
  // out[n-1] = v0; out[n-2] = y[n-2] + b1*out[n-1] + b2*v1 + b3*v2;
  // out[n-3] = y[n-3] + b1*out[n-2] + b2*out[n-1] + b3*v1
  const double z2 = v0;
  const double z1 = ym1 + b1 * z2 + b2 * v1 + b3 * v2;
  const double z0 = ym2 + b1 * z1 + b2 * z2 + b3 * v1;
  const double sc = p.scale;
  p.dst[base + (int64_t)(n - 1) * st] = z2 * sc;
  p.dst[base + (int64_t)(n - 2) * st] = z1 * sc;
  p.dst[base + (int64_t)(n - 3) * st] = z0 * sc;
  // backward
  double zp1 = z0, zp2 = z1, zp3 = z2;
  int k = n - 4;
  for (; k - (IC - 1) >= 0; k -= IC) {
    double y[IC];
#pragma unroll
    for (int j = 0; j < IC; ++j) y[j] = p.dst[base + (int64_t)(k - j) * st];
#pragma unroll
    for (int j = 0; j < IC; ++j) {
      const double z = y[j] + b1 * zp1 + b2 * zp2 + b3 * zp3;
      p.dst[base + (int64_t)(k - j) * st] = z * sc;
      zp3 = zp2;
      zp2 = zp1;
      zp1 = z;
    }
  }
  for (; k >= 0; --k) {
    double z = p.dst[base + (int64_t)k * st] + b1 * zp1 + b2 * zp2 + b3 * zp3;
    p.dst[base + (int64_t)k * st] = z * sc;
    zp3 = zp2;
    zp2 = zp1;
    zp1 = z;
  }
}

// Lines along the contiguous axis.  One thread per line would read 64 lines
// per wave instruction, n elements apart; instead a workgroup owns 256 lines
// and walks them in chunks of IR_C elements staged through LDS: the chunk is
// loaded and stored with consecutive lanes on consecutive elements
// (coalesced), and each thread runs its line's recursion over the chunk from
// LDS.  The next chunk's loads are issued before the current chunk is
// filtered.  The arithmetic per element is that of k_iir_strided.
constexpr int IR_C = 16;                   // chunk length
constexpr int IR_L = 256;                  // lines per workgroup
constexpr int IR_P = IR_C + 1;             // LDS pitch (doubles)
constexpr int IR_E = IR_L * IR_C / 256;    // staged elements per thread

template <int DT>
__global__ void __launch_bounds__(256, 2) k_iir_rows(IirArgs p) {
  extern __shared__ double tile[];  // IR_L x IR_P
  const int t = threadIdx.x;
  const int64_t line0 = (int64_t)blockIdx.x * IR_L;
  const int n = p.n[0];
  const int nl = (int)min((int64_t)IR_L, p.lines - line0);
  const int nch = (n + IR_C - 1) / IR_C;
  const double a1 = p.a[0], a2 = p.a[1], a3 = p.a[2];
  const double b1 = p.b[0], b2 = p.b[1], b3 = p.b[2];
  const double asum = a1 + a2 + a3, bsum = b1 + b2 + b3;
  double reg[IR_E];
  // staged element j of the thread: line (t + 256 j) / IR_C, offset (t + 256 j) % IR_C
  auto fetch = [&](const void *src, int dtsrc, int c0, bool typed) {
#pragma unroll
    for (int j = 0; j < IR_E; ++j) {
      const int q = t + 256 * j, l = q / IR_C, e = q % IR_C;
      const int i = c0 + e;
      if (l < nl && i < n) {
        const int64_t g = (line0 + l) * n + i;
        reg[j] = typed ? iir_ld<DT>(p, g) : ((const double *)src)[g];
      }
    }
    (void)dtsrc;
  };
  auto put = [&]() {
#pragma unroll
    for (int j = 0; j < IR_E; ++j) {
      const int q = t + 256 * j;
      tile[(q / IR_C) * IR_P + q % IR_C] = reg[j];
    }
  };
  auto store = [&](int c0) {
#pragma unroll
    for (int j = 0; j < IR_E; ++j) {
      const int q = t + 256 * j, l = q / IR_C, e = q % IR_C;
      const int i = c0 + e;
      if (l < nl && i < n) p.dst[(line0 + l) * n + i] = tile[l * IR_P + e];
    }
  };
  double *row = tile + t * IR_P;
  // forward: y[i] = x[i] + a1 y[i-1] + a2 y[i-2] + a3 y[i-3], with y[-k] = u-
  double um = 0.0, ym1 = 0.0, ym2 = 0.0, ym3 = 0.0, iplus = p.fill;
  fetch(nullptr, 0, 0, true);
  for (int c = 0; c < nch; ++c) {
    const int c0 = c * IR_C;
    put();
    __syncthreads();
    if (c + 1 < nch) fetch(nullptr, 0, c0 + IR_C, true);
    if (t < nl) {
      const int e1 = min(IR_C, n - c0);
      if (c == 0) {
        const double iminus = p.isfill ? p.fill : row[0];
        um = iminus / (1 - asum);
      }
      if (c0 + e1 == n && !p.isfill) iplus = row[e1 - 1];
      for (int e = 0; e < e1; ++e) {
        const int i = c0 + e;  // wave-uniform
        const double x = row[e];
        double y;
        if (i == 0) y = x + a1 * um + a2 * um + a3 * um;
        else if (i == 1) y = x + a1 * ym1 + a2 * um + a3 * um;
        else if (i == 2) y = x + a1 * ym1 + a2 * ym2 + a3 * um;
        else y = x + a1 * ym1 + a2 * ym2 + a3 * ym3;
        row[e] = y;
        ym3 = ym2;
        ym2 = ym1;
        ym1 = y;
      }
    }
    __syncthreads();
    store(c0);
    __syncthreads();
  }
  // right edge (ym1 = y[n-1], ym2 = y[n-2], ym3 = y[n-3]), then backward:
  // z[k] = y[k] + b1 z[k+1] + b2 z[k+2] + b3 z[k+3], the last three from M
  const double sc = p.scale;
  const double uplus = iplus / (1 - asum);
  const double vplus = uplus / (1 - bsum);
  const double d0 = ym1 - uplus, d1 = ym2 - uplus, d2 = ym3 - uplus;
  const double v0 = p.M[0] * d0 + p.M[1] * d1 + p.M[2] * d2 + vplus;
  const double v1 = p.M[3] * d0 + p.M[4] * d1 + p.M[5] * d2 + vplus;
  const double v2 = p.M[6] * d0 + p.M[7] * d1 + p.M[8] * d2 + vplus;
  const double z2 = v0;
  const double z1 = ym2 + b1 * z2 + b2 * v1 + b3 * v2;
  const double z0 = ym3 + b1 * z1 + b2 * z2 + b3 * v1;
  double zp1 = 0.0, zp2 = 0.0, zp3 = 0.0;
  fetch(p.dst, IFM_F64, (nch - 1) * IR_C, false);
  for (int c = nch - 1; c >= 0; --c) {
    const int c0 = c * IR_C;
    put();
    __syncthreads();
    if (c > 0) fetch(p.dst, IFM_F64, c0 - IR_C, false);
    if (t < nl) {
      const int e1 = min(IR_C, n - c0);
      for (int e = e1 - 1; e >= 0; --e) {
        const int k = c0 + e;  // wave-uniform
        double z;
        if (k == n - 1) z = z2;
        else if (k == n - 2) z = z1;
        else if (k == n - 3) z = z0;
        else z = row[e] + b1 * zp1 + b2 * zp2 + b3 * zp3;
        row[e] = z * sc;
        zp3 = zp2;
        zp2 = zp1;
        zp1 = z;
      }
    }
    __syncthreads();
    store(c0);
    __syncthreads();
  }
}

// Lines of up to 8192 elements, held in registers.  The axis is cut into
// segments of IS_S elements, each run by one lane, so every element is read
// once and written once (the one-thread-per-line form writes the forward pass
// out and reads it back, and leaves the chip idle when there are few lines:
// 3840 x 2160 F32 took 1960 + 292 + 20 us for the two axes and the copy into
// an F32 output, and takes 71 us this way, of which the bytes are 40).  The
// recursions are linear: a
// segment's values are its recursion from zero state plus the homogeneous
// response to the state entering it.  Each lane runs its segment from zero
// state; the states are then composed along the line (a shuffle scan within
// the wave, wave totals through LDS), and each lane adds the response to the
// state entering its segment.  The first segment's forward pass and the last
// segment's backward pass start from the reference's border initialisation
// directly (the um / M start of k_iir_strided).
//
// A line that does not fill the workgroup's segments is continued before its
// first element by copies of the value the left border is initialised from
// (that element, or the Fill value): they keep the recursion in the state it
// starts in, the steady state of that value, and nothing is stored for them.
// So every segment has IS_S elements and every loop bound is a constant
// (bounds per element cost 766 against 652 us on 512 x 512 x 256; a second
// body for short segments spilled registers: 604 us on 500 x 300 x 200 F64
// against 275 this way).  What bounds it is HBM on large volumes (512 x 512 x
// 256 F32 -> F64, three axes: 565 us for 2.95 GB, 5.2 TB/s) and the one
// load - recursion - store sequence per workgroup on small images.  Lines above
// 4096 elements run four to a workgroup: 8192 x 8192 F32 -> F64 204 us along the
// contiguous axis and 556 along the other (4700 and 1209 through HBM); 300 lines
// of 8192 23 and 24 us (3879 and 901).
constexpr int IS_S = 32;     // elements per segment (doubles in registers per lane)
constexpr int IS_MAXW = 16;  // most waves per workgroup
constexpr int IS_MINL = 4;   // fewest lines per workgroup: n <= 64 / 4 * 16 * 32 = 8192

struct IirSegTables {
  double pf[5][9];  // forward transfer of a state's differences over 1, 2, 4, 8, 16 segments (row-major 3 x 3)
  double pb[5][9];  // backward
};

// A workgroup owns LN adjacent lines (32, 16, 8 or 4); lane l of wave w runs
// segment w SPW + l / LN of line l mod LN, SPW = 64 / LN.  Segments of 32
// elements keep a lane's share of the line in 64 registers, so four waves
// share each SIMD and one's loads and stores overlap the others' recursions;
// 64-element segments (two waves per SIMD) measured 942 against 767 us on
// 512 x 512 x 256.
//  * k_iir_seg   strided lines: lanes of equal segment read LN adjacent
//                elements.
//  * k_iir_line  contiguous lines: a wave's segments are one run of SPW * 32
//                elements of a line, loaded and stored by its lanes; they
//                pass through a per-wave LDS transpose (rows = (line,
//                segment) pairs): 32 rows per round for inputs staged as FP32
//                values, 16 for FP64 input and for the output.  The buffer is
//                the wave's own, so its rounds need no workgroup barrier.
constexpr int IS_TP = IS_S + 1;           // transpose buffer pitch (elements): conflict-free both ways
constexpr int IS_TB = 16 * IS_TP;         // transpose buffer per wave (doubles)
__host__ __device__ inline size_t iir_seg_lds_doubles(int waves, int ln, bool rows) {
  return 6 * (size_t)waves * ln + (rows ? (size_t)waves * IS_TB : 0);
}

struct Seg {
  int ln, pos, w;  // line and segment of the lane within the wave, wave
  int at0;         // element of the line the lane's segment starts at (negative: before the line)
  bool first, last;
};

template <int LN>
__device__ __forceinline__ Seg seg_lane(int n) {
  Seg g;
  const int lane = threadIdx.x & 63, waves = blockDim.x >> 6;
  constexpr int SPW = 64 / LN;
  g.w = (int)__builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  g.ln = lane % LN;
  g.pos = lane / LN;
  g.at0 = (SPW * g.w + g.pos) * IS_S - (waves * SPW * IS_S - n);
  g.first = g.w == 0 && g.pos == 0;
  g.last = g.w == waves - 1 && g.pos == SPW - 1;
  return g;
}

struct State3 {
  double a, b, c;
};

// s + M t for a 3 x 3 row-major M
__device__ __forceinline__ State3 st_fma(const double *M, const State3 &t, const State3 &s) {
  State3 r;
  r.a = M[0] * t.a + M[1] * t.b + M[2] * t.c + s.a;
  r.b = M[3] * t.a + M[4] * t.b + M[5] * t.c + s.b;
  r.c = M[6] * t.a + M[7] * t.b + M[8] * t.c + s.c;
  return r;
}

__device__ __forceinline__ State3 st_shfl(const State3 &s, int from) {
  State3 r;
  r.a = __shfl(s.a, from);
  r.b = __shfl(s.b, from);
  r.c = __shfl(s.c, from);
  return r;
}

// A state (y, y', y'') as its value and first two differences, and back (the
// map is its own inverse).  The three values are nearly equal for a wide
// Gaussian and the transfer matrices between them have large entries of
// alternating sign, so states composed as values lose digits.  One axis,
// sigma 20, random lines of 200 to 1000 elements, 2-norm of the error against
// extended precision over that of the result: 1.1e-11 to 1.3e-11 as values,
// 4e-14 to 9e-14 this way, 8e-14 to 1e-13 element by element in Float64.
__device__ __forceinline__ State3 st_diff(const State3 &s) {
  return State3{s.a, s.a - s.b, (s.a - s.b) - (s.b - s.c)};
}
__device__ __forceinline__ State3 st_values(const State3 &s) {
  return State3{s.a, s.a - s.b, s.a - (2 * s.b - s.c)};
}

// The state entering the lane's segment, from the zero-state end states `own`
// of every segment (the segment the recursion starts in holds its true end
// state).  REV: the recursion runs from the last segment to the first.  ex:
// waves x 3 x LN doubles of LDS.  One barrier.
template <int LN, bool REV>
__device__ __forceinline__ State3 seg_enter(const double (&pw)[5][9], const Seg &g, State3 own, double *ex) {
  constexpr int SPW = 64 / LN, KW = SPW == 16 ? 4 : SPW == 8 ? 3 : SPW == 4 ? 2 : 1;
  const int lane = threadIdx.x & 63, waves = blockDim.x >> 6;
  const int at = REV ? SPW - 1 - g.pos : g.pos;    // place in the wave's order
  const int w = REV ? waves - 1 - g.w : g.w;       // place of the wave
  const State3 zero = {0.0, 0.0, 0.0};
  own = st_diff(own);
#pragma unroll
  for (int k = 0; k < KW; ++k) {  // inclusive scan within the wave
    const int d = 1 << k;
    const State3 o = st_shfl(own, REV ? lane + d * LN : lane - d * LN);
    if (at >= d) own = st_fma(pw[k], o, own);
  }
  if (at == SPW - 1) {
    ex[(w * 3 + 0) * LN + g.ln] = own.a;
    ex[(w * 3 + 1) * LN + g.ln] = own.b;
    ex[(w * 3 + 2) * LN + g.ln] = own.c;
  }
  State3 t = st_shfl(own, REV ? lane + LN : lane - LN);
  if (at == 0) t = zero;
  __syncthreads();
  State3 c = zero;                        // state entering the wave
#pragma unroll 2
  for (int u = 0; u < w; ++u) {
    const State3 q = {ex[(u * 3 + 0) * LN + g.ln], ex[(u * 3 + 1) * LN + g.ln], ex[(u * 3 + 2) * LN + g.ln]};
    c = st_fma(pw[KW], c, q);
  }
#pragma unroll
  for (int k = 0; k < KW; ++k)            // carried over `at` segments
    if ((at >> k) & 1) c = st_fma(pw[k], c, zero);
  t.a += c.a;
  t.b += c.b;
  t.c += c.c;
  return st_values(t);
}

// End of one step of a recursion: the steps are not interleaved (the response
// does not depend on v, and computed ahead it would take 64 more registers).
__device__ __forceinline__ void step_done(double &v) {
  asm volatile("" : "+v"(v));
  __builtin_amdgcn_sched_barrier(0);
}

// The segmented recursion on v of every lane: forward from zero state (the
// first segment from leftborder!), the homogeneous response of the state
// entering the segment added; the same backward (the last segment from
// rightborder!).  Leaves v scaled by nothing; contains two barriers.
template <int LN>
__device__ __forceinline__ void seg_filter(const IirArgs &p, const IirSegTables &tb, const Seg &g, double *sm,
                                           double (&v)[IS_S]) {
  double *stf = sm, *stb = sm + 3 * LN * (blockDim.x >> 6);
  const double a1 = p.a[0], a2 = p.a[1], a3 = p.a[2];
  const double b1 = p.b[0], b2 = p.b[1], b3 = p.b[2];
  const double asum = a1 + a2 + a3, bsum = b1 + b2 + b3;
  double ym1 = 0.0, ym2 = 0.0, ym3 = 0.0;
  if (g.first) {  // v[0]: the line's first element, or a copy of what the border starts from
    const double iminus = p.isfill ? p.fill : v[0];
    ym1 = ym2 = ym3 = iminus / (1 - asum);
  }
  const double xlast = v[IS_S - 1];
#pragma unroll
  for (int j = 0; j < IS_S; ++j) {
    const double y = v[j] + a1 * ym1 + a2 * ym2 + a3 * ym3;
    v[j] = y;
    ym3 = ym2;
    ym2 = ym1;
    ym1 = y;
    step_done(v[j]);
  }
  State3 r = seg_enter<LN, false>(tb.pf, g, State3{ym1, ym2, ym3}, stf);
#pragma unroll
  for (int j = 0; j < IS_S; ++j) {
    const double y = a1 * r.a + (a2 * r.b + a3 * r.c);
    v[j] += y;
    r = State3{y, r.a, r.b};
    step_done(v[j]);
  }
  double z0 = 0.0, z1 = 0.0, z2 = 0.0;
  if (g.last) {
    const double e0 = v[IS_S - 1], e1 = v[IS_S - 2], e2 = v[IS_S - 3];
    const double iplus = p.isfill ? p.fill : xlast;
    const double uplus = iplus / (1 - asum);
    const double vplus = uplus / (1 - bsum);
    const double d0 = e0 - uplus, d1 = e1 - uplus, d2 = e2 - uplus;
    const double m0 = p.M[0] * d0 + p.M[1] * d1 + p.M[2] * d2 + vplus;
    const double m1 = p.M[3] * d0 + p.M[4] * d1 + p.M[5] * d2 + vplus;
    const double m2 = p.M[6] * d0 + p.M[7] * d1 + p.M[8] * d2 + vplus;
    z2 = m0;
    z1 = e1 + b1 * z2 + b2 * m1 + b3 * m2;
    z0 = e2 + b1 * z1 + b2 * z2 + b3 * m1;
  }
  double zp1 = 0.0, zp2 = 0.0, zp3 = 0.0;
#pragma unroll
  for (int j = IS_S - 1; j >= 0; --j) {
    double z = v[j] + b1 * zp1 + b2 * zp2 + b3 * zp3;
    if (j == IS_S - 1) z = g.last ? z2 : z;
    if (j == IS_S - 2) z = g.last ? z1 : z;
    if (j == IS_S - 3) z = g.last ? z0 : z;
    v[j] = z;
    zp3 = zp2;
    zp2 = zp1;
    zp1 = z;
    step_done(v[j]);
  }
  r = seg_enter<LN, true>(tb.pb, g, State3{zp1, zp2, zp3}, stb);
#pragma unroll
  for (int j = IS_S - 1; j >= 0; --j) {
    const double z = b1 * r.a + (b2 * r.b + b3 * r.c);
    v[j] += z;
    r = State3{z, r.a, r.b};
    step_done(v[j]);
  }
}

// The elements before the line under a Fill border.
__device__ __forceinline__ void seg_lead(const IirArgs &p, const Seg &g, double (&v)[IS_S]) {
  if (!p.isfill || g.at0 >= 0) return;
#pragma unroll
  for (int j = 0; j < IS_S; ++j)
    if (g.at0 + j < 0) v[j] = p.fill;
}

// Stage result in the destination eltype: FP64 between the stages, at the
// last stage whatever the output holds (rounded through FP32 for the 16-bit
// floats, -0 to +0 as the converting copy rounds).
template <int DD>  // IFM_F64, IFM_F32, or -1: one of the 16-bit floats
__device__ __forceinline__ void iir_put(IFM_GLOBAL char *at, int dt, double v) {
  if constexpr (DD == IFM_F64) *(IFM_GLOBAL double *)at = v;
  else if constexpr (DD == IFM_F32) *(IFM_GLOBAL float *)at = (float)v + 0.f;
  else store_f((void *)at, 0, dt, (float)v + 0.f);
}

// Workgroups of neighbouring lines run on one XCD: with LN < 32 they share
// cache lines.
__device__ __forceinline__ int64_t seg_line0(int ln) { return (int64_t)xcd_tile(blockIdx.x, gridDim.x) * ln; }

// Address of element j of a strided line, stepped from element to element:
// left alone the compiler keeps all 31 multiples of the stride in scalar
// registers, which spill.
struct Walk {
  IFM_GLOBAL char *at;
  int64_t step;
  __device__ __forceinline__ Walk(const void *p, int64_t i, int64_t st, int es)
      : at((IFM_GLOBAL char *)((char *)p + i * es)), step(st * es) {}
  __device__ __forceinline__ void next(bool more = true) {
    at += more ? step : 0;
    asm volatile("" : "+v"(at));
  }
};

// FRONT: the wave holds elements before the line.
template <int DT, bool FRONT>
__device__ __forceinline__ void seg_load(const IirArgs &p, const Seg &g, int64_t base, double (&v)[IS_S]) {
  using T = typename std::conditional<DT == IFM_F64, double, float>::type;
  const int64_t i0 = FRONT ? max(g.at0, 0) : g.at0;
  Walk q(p.src, base + i0 * p.stride, p.stride, DT == IFM_F32 || DT == IFM_F64 ? (int)sizeof(T) : p.es_src);
#pragma unroll
  for (int j = 0; j < IS_S; ++j) {
    if constexpr (DT == IFM_F32 || DT == IFM_F64) v[j] = (double)*(const IFM_GLOBAL T *)q.at;
    else v[j] = load_d((const void *)q.at, 0, p.dt_src);
    q.next(!FRONT || g.at0 + j >= 0);
  }
}

template <int DD, bool FRONT>
__device__ __forceinline__ void seg_store(const IirArgs &p, const Seg &g, int64_t base, const double (&v)[IS_S]) {
  const double sc = p.scale;
  const int es = DD == IFM_F64 ? 8 : DD == IFM_F32 ? 4 : 2;
  Walk q(p.dst, base + (int64_t)g.at0 * p.stride, p.stride, es);
#pragma unroll
  for (int j = 0; j < IS_S; ++j) {
    if (!FRONT || g.at0 + j >= 0) iir_put<DD>(q.at, p.dt_dst, v[j] * sc);
    q.next();
  }
}

template <int DT, int LN>
__global__ void __launch_bounds__(64 * IS_MAXW) __attribute__((amdgpu_waves_per_eu(4))) k_iir_seg(IirArgs p, IirSegTables tb) {
  extern __shared__ double sm[];
  const int n = p.n[p.axis];
  const Seg g = seg_lane<LN>(n);
  const int64_t ln = seg_line0(LN) + g.ln;
  const int64_t line = min(ln, p.lines - 1);  // lanes past the last line repeat it and store nothing
  const int64_t base = (line % p.stride) + (line / p.stride) * p.stride * n;
  const bool front = __builtin_amdgcn_readfirstlane(g.at0) < 0;  // lane 0 has the wave's first segment
  double v[IS_S];
  if (front) seg_load<DT, true>(p, g, base, v);
  else seg_load<DT, false>(p, g, base, v);
  seg_lead(p, g, v);
  seg_filter<LN>(p, tb, g, sm, v);
  if (ln >= p.lines) return;
  if (p.dt_dst == IFM_F64) {
    if (front) seg_store<IFM_F64, true>(p, g, base, v);
    else seg_store<IFM_F64, false>(p, g, base, v);
  } else if (p.dt_dst == IFM_F32) {
    seg_store<IFM_F32, true>(p, g, base, v);
  } else {
    seg_store<-1, true>(p, g, base, v);
  }
}

// Element as staged: F64 as it is, every other type as FP32 (exact), N0f8 as
// its code.
template <int DT>
__device__ __forceinline__ typename std::conditional<DT == IFM_F64, double, float>::type line_ld(const void *src,
                                                                                               int64_t i) {
  if constexpr (DT == IFM_F64) return ((const double *)src)[i];
  else if constexpr (DT == IFM_F32) return ((const float *)src)[i];
  else if constexpr (DT == IFM_BF16) return bf16_to_f32(((const uint16_t *)src)[i]);
  else if constexpr (DT == IFM_F16) return __half2float(((const __half *)src)[i]);
  else return (float)((const uint8_t *)src)[i];
}

// Store rounds of the transposed results: RO lines per round.
template <int DD, int LN>
__device__ __forceinline__ void line_store(const IirArgs &p, const Seg &g, double *tr, int64_t line0, int w0,
                                           const double (&v)[IS_S]) {
  constexpr int SPW = 64 / LN, NC = SPW / 2, RO = 16 / SPW;
  const int n = p.n[p.axis], lane = threadIdx.x & 63;
  const int es = DD == IFM_F64 ? 8 : DD == IFM_F32 ? 4 : 2;
  const double sc = p.scale;
#pragma unroll 1
  for (int r = 0; r < LN / RO; ++r) {
    if ((g.ln / RO) == r) {
      const int row = (g.ln - r * RO) * SPW + g.pos;
#pragma unroll
      for (int j = 0; j < IS_S; ++j) tr[row * IS_TP + j] = v[j] * sc;
    }
    wave_lds_fence();
#pragma unroll
    for (int i = 0; i < RO; ++i) {
      const int64_t ln = line0 + r * RO + i;
#pragma unroll
      for (int c = 0; c < NC; ++c) {
        const int e = 64 * c + lane;
        if (w0 + e >= 0 && ln < p.lines)
          iir_put<DD>((IFM_GLOBAL char *)((char *)p.dst + (ln * n + w0 + e) * es), p.dt_dst,
                      tr[(SPW * i + e / IS_S) * IS_TP + e % IS_S]);
      }
    }
    wave_lds_fence();
  }
}

template <int DT, int LN>
__global__ void __launch_bounds__(64 * IS_MAXW) __attribute__((amdgpu_waves_per_eu(4))) k_iir_line(IirArgs p, IirSegTables tb) {
  extern __shared__ double sm[];
  using TE = typename std::conditional<DT == IFM_F64, double, float>::type;
  constexpr int SPW = 64 / LN, NC = SPW / 2;           // NC: 64-element loads covering a wave's run of one line
  constexpr int RI = (DT == IFM_F64 ? 16 : 32) / SPW;  // lines per load round
  const int n = p.n[p.axis], lane = threadIdx.x & 63;
  const Seg g = seg_lane<LN>(n);
  const int w0 = __builtin_amdgcn_readfirstlane(g.at0);  // first element of the wave's run
  const int64_t line0 = seg_line0(LN);
  double *tr = sm + iir_seg_lds_doubles(blockDim.x >> 6, LN, false) + g.w * IS_TB;
  TE *tri = (TE *)tr;
  double v[IS_S];
#pragma unroll 1
  for (int r = 0; r < LN / RI; ++r) {
    TE x[RI][NC];
#pragma unroll
    for (int i = 0; i < RI; ++i) {
      const int64_t ln = min(line0 + r * RI + i, p.lines - 1);
#pragma unroll
      for (int c = 0; c < NC; ++c) x[i][c] = line_ld<DT>(p.src, ln * n + max(w0 + 64 * c + lane, 0));
    }
#pragma unroll
    for (int i = 0; i < RI; ++i)
#pragma unroll
      for (int c = 0; c < NC; ++c) {
        const int e = 64 * c + lane;
        tri[(SPW * i + e / IS_S) * IS_TP + e % IS_S] = x[i][c];
      }
    wave_lds_fence();
    if ((g.ln / RI) == r) {
      const int row = (g.ln - r * RI) * SPW + g.pos;
#pragma unroll
      for (int j = 0; j < IS_S; ++j)
        v[j] = DT == IFM_N0F8 ? (double)tri[row * IS_TP + j] / 255.0 : (double)tri[row * IS_TP + j];
    }
    wave_lds_fence();
  }
  seg_lead(p, g, v);
  seg_filter<LN>(p, tb, g, sm, v);
  if (p.dt_dst == IFM_F64) line_store<IFM_F64, LN>(p, g, tr, line0, w0, v);
  else if (p.dt_dst == IFM_F32) line_store<IFM_F32, LN>(p, g, tr, line0, w0, v);
  else line_store<-1, LN>(p, g, tr, line0, w0, v);
}

// Strided lines of up to IK_MAX elements, one lane per line: no segments to
// compose and, with S the next of a few lengths, few places of a lane's
// registers unused.  The segmented form runs 64 elements for any of these
// lines, and reads the 1- and 2-byte eltypes by a choice per element.  1 M lines
// of 4 / 8 / 16 / 32 elements F64: 57 / 59 / 74 / 106 us segmented, 11 / 20 / 50 /
// 101 this way; N0f8 -> F64 112 / 121 / 141 / 191 and 14 / 16 / 31 / 64.  Bound by
// HBM from a million lines on.  Longer F32 and F64 lines fill segments well
// enough (20000 of 40 F32: 6.3 us segmented, 7.2 this way); the smaller eltypes
// gain up to 48 elements (1 M of 40 N0f8: 206 and 85).
constexpr int IK_MAX = 32, IK_MAX_SMALL = 48;

template <int DT, int S>
__global__ void __launch_bounds__(256) k_iir_short(IirArgs p) {
  const int64_t line = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (line >= p.lines) return;
  const int n = p.n[p.axis], lead = S - n;  // v[lead ..]: the line
  const int64_t base = (line % p.stride) + (line / p.stride) * p.stride * n;
  using TE = decltype(line_ld<DT>(nullptr, 0));
  constexpr int es = DT == IFM_F64 ? 8 : DT == IFM_F32 ? 4 : DT == IFM_U8 || DT == IFM_N0F8 ? 1 : 2;
  TE x[S];
  Walk q(p.src, base, p.stride, es);
#pragma unroll
  for (int j = 0; j < S; ++j) {  // every load unconditional, so that they are in flight together
    x[j] = line_ld<DT>((const void *)q.at, 0);
    q.next(j >= lead);
  }
  double v[S];
#pragma unroll
  for (int j = 0; j < S; ++j) v[j] = DT == IFM_N0F8 ? (double)x[j] / 255.0 : (double)x[j];
  const double a1 = p.a[0], a2 = p.a[1], a3 = p.a[2];
  const double b1 = p.b[0], b2 = p.b[1], b3 = p.b[2];
  const double asum = a1 + a2 + a3, bsum = b1 + b2 + b3;
  const double uminus = (p.isfill ? p.fill : v[0]) / (1 - asum);  // v[0]: the first element, or a copy of it
  const double uplus = (p.isfill ? p.fill : v[S - 1]) / (1 - asum);
  double y1 = uminus, y2 = uminus, y3 = uminus;
#pragma unroll
  for (int j = 0; j < S; ++j) {
    if (j < lead) continue;  // uniform over the grid
    v[j] = v[j] + a1 * y1 + a2 * y2 + a3 * y3;
    y3 = y2;
    y2 = y1;
    y1 = v[j];
  }
  const double vplus = uplus / (1 - bsum);
  const double d0 = y1 - uplus, d1 = y2 - uplus, d2 = y3 - uplus;
  double z1 = p.M[0] * d0 + p.M[1] * d1 + p.M[2] * d2 + vplus;
  double z2 = p.M[3] * d0 + p.M[4] * d1 + p.M[5] * d2 + vplus;  // beyond the edge
  double z3 = p.M[6] * d0 + p.M[7] * d1 + p.M[8] * d2 + vplus;
  v[S - 1] = z1;
#pragma unroll
  for (int j = S - 2; j >= 0; --j) {
    if (j < lead) continue;
    v[j] = v[j] + b1 * z1 + b2 * z2 + b3 * z3;
    z3 = z2;
    z2 = z1;
    z1 = v[j];
  }
  const double sc = p.scale;
  const auto store = [&](auto type) {
    constexpr int DD = decltype(type)::value;
    Walk w(p.dst, base, p.stride, DD == IFM_F64 ? 8 : DD == IFM_F32 ? 4 : 2);
#pragma unroll
    for (int j = 0; j < S; ++j) {
      if (j < lead) continue;
      iir_put<DD>(w.at, p.dt_dst, v[j] * sc);
      w.next();
    }
  };
  if (p.dt_dst == IFM_F64) store(std::integral_constant<int, IFM_F64>());
  else if (p.dt_dst == IFM_F32) store(std::integral_constant<int, IFM_F32>());
  else store(std::integral_constant<int, -1>());
}

template <int DT>
static void short_go(const IirArgs &p, hipStream_t st) {
  const int n = p.n[p.axis];
  const dim3 grid((unsigned)((p.lines + 255) / 256)), blk(256);
  if (n <= 8) hipLaunchKernelGGL((k_iir_short<DT, 8>), grid, blk, 0, st, p);
  else if (n <= 16) hipLaunchKernelGGL((k_iir_short<DT, 16>), grid, blk, 0, st, p);
  else if (n <= 32) hipLaunchKernelGGL((k_iir_short<DT, 32>), grid, blk, 0, st, p);
  else hipLaunchKernelGGL((k_iir_short<DT, 48>), grid, blk, 0, st, p);
}

static int iir_waves(int n, int ln) { return (n + (64 / ln) * IS_S - 1) / ((64 / ln) * IS_S); }

// Lines per workgroup: 32 (the longest runs of adjacent lines) when the
// segments fit 8 waves, so that two workgroups share a CU, and there are
// workgroups for every CU; fewer otherwise, but no fewer than 8 while the
// segments fit 16 waves (200 x 150: 16.9 us with 8, 18.0 with 4; 3840 x 2160:
// 71 with either), and no fewer than put the line into one wave, or a strided
// one into three full ones (4000 strided lines F64, 64 / 128 / 192 elements:
// 5.6 / 5.8 / 6.3 us, 7.3 / 7.5 / 7.8 with 8 lines and more elements before them).
static int iir_lines(int n, int64_t lines, bool strided) {
  int ln = 32;
  while (ln > IS_MINL) {
    const int waves = iir_waves(n, ln);
    if (waves <= IS_MAXW / 2 && (lines + ln - 1) / ln >= 256) break;
    if (waves <= IS_MAXW && ln == 8) break;
    if (waves == 1) break;
    if (strided && waves == 3 && n % (64 / ln * IS_S) == 0) break;
    ln /= 2;
  }
  return ln;
}

template <int DT, int LN>
static void seg_go(const IirArgs &p, const IirSegTables &tb, hipStream_t st) {
  const int waves = iir_waves(p.n[p.axis], LN);
  const dim3 grid((unsigned)((p.lines + LN - 1) / LN)), blk(64 * waves);
  const bool rows = p.stride == 1;
  const size_t lds = sizeof(double) * iir_seg_lds_doubles(waves, LN, rows);
  if (rows) {
    hipLaunchKernelGGL((k_iir_line<DT, LN>), grid, blk, lds, st, p, tb);
  } else {
    constexpr int DS = DT == IFM_F32 || DT == IFM_F64 ? DT : -1;  // strided loads of the other types: run-time type
    hipLaunchKernelGGL((k_iir_seg<DS, LN>), grid, blk, lds, st, p, tb);
  }
}

template <int DT>
static void seg_lines(const IirArgs &p, const IirSegTables &tb, hipStream_t st) {
  switch (iir_lines(p.n[p.axis], p.lines, p.stride != 1)) {
  case 32: seg_go<DT, 32>(p, tb, st); break;
  case 16: seg_go<DT, 16>(p, tb, st); break;
  case 8: seg_go<DT, 8>(p, tb, st); break;
  default: seg_go<DT, 4>(p, tb, st); break;
  }
}

bool iir_in_registers(int64_t n) { return n >= 4 && n <= (64 / IS_MINL) * IS_MAXW * IS_S; }

hipError_t launch_iir(const Dense4 &in, Dense4 &out, int axis, const IirCoef &c, int isfill, double fill,
                      hipStream_t st) {
  IirArgs p;
  p.src = in.data;
  p.dst = (double *)out.data;
  p.dt_src = in.dtype;
  p.es_src = (int)dtype_size(in.dtype);
  p.dt_dst = out.dtype;
  int64_t stride = 1;
  for (int d = 0; d < MAXD; ++d) {
    p.n[d] = (int)in.n[d];
    if (d < axis) stride *= in.n[d];
  }
  p.axis = axis;
  p.stride = stride;
  p.lines = in.count() / in.n[axis];
  for (int i = 0; i < 3; ++i) {
    p.a[i] = c.a[i];
    p.b[i] = c.b[i];
  }
  p.scale = c.scale;
  for (int i = 0; i < 9; ++i) p.M[i] = c.M[i];
  p.isfill = isfill;
  p.fill = fill;
  if (p.lines == 0) return hipSuccess;
  if (stride != 1 && in.n[axis] >= 4 && in.n[axis] <= (dtype_size(in.dtype) >= 4 ? IK_MAX : IK_MAX_SMALL)) {
    switch (in.dtype) {
    case IFM_F32: short_go<IFM_F32>(p, st); break;
    case IFM_F64: short_go<IFM_F64>(p, st); break;
    case IFM_BF16: short_go<IFM_BF16>(p, st); break;
    case IFM_F16: short_go<IFM_F16>(p, st); break;
    case IFM_N0F8: short_go<IFM_N0F8>(p, st); break;
    default: short_go<IFM_U8>(p, st); break;
    }
    return hipGetLastError();
  }
  if (iir_in_registers(in.n[axis])) {  // whole lines held in registers
    IirSegTables tb;
    // Built in extended precision and rounded once.
    long double pf[9], pb[9];
    for (int k = 0; k < 3; ++k) {
      // responses to the state whose differences (st_diff) are the unit e_k:
      // y[-1], y[-2], y[-3] = column k of the map back to values
      const long double e[3][3] = {{1, 1, 1}, {0, -1, -2}, {0, 0, 1}};
      long double hm[3] = {e[k][0], e[k][1], e[k][2]}, gm[3] = {e[k][0], e[k][1], e[k][2]};
      for (int j = 0; j < IS_S; ++j) {
        const long double h = c.a[0] * hm[0] + c.a[1] * hm[1] + c.a[2] * hm[2];
        const long double g = c.b[0] * gm[0] + c.b[1] * gm[1] + c.b[2] * gm[2];
        hm[2] = hm[1];
        hm[1] = hm[0];
        hm[0] = h;
        gm[2] = gm[1];
        gm[1] = gm[0];
        gm[0] = g;
      }
      // the differences after one full segment
      pf[k] = hm[0], pf[3 + k] = hm[0] - hm[1], pf[6 + k] = (hm[0] - hm[1]) - (hm[1] - hm[2]);
      pb[k] = gm[0], pb[3 + k] = gm[0] - gm[1], pb[6 + k] = (gm[0] - gm[1]) - (gm[1] - gm[2]);
    }
    for (int q = 0; q < 5; ++q) {
      long double f[9] = {}, g[9] = {};
      for (int r = 0; r < 3; ++r)
        for (int k = 0; k < 3; ++k) {
          tb.pf[q][3 * r + k] = (double)pf[3 * r + k];
          tb.pb[q][3 * r + k] = (double)pb[3 * r + k];
          for (int i = 0; i < 3; ++i) {
            f[3 * r + k] += pf[3 * r + i] * pf[3 * i + k];
            g[3 * r + k] += pb[3 * r + i] * pb[3 * i + k];
          }
        }
      for (int i = 0; i < 9; ++i) pf[i] = f[i], pb[i] = g[i];
    }
    switch (in.dtype) {
    case IFM_F32: seg_lines<IFM_F32>(p, tb, st); break;
    case IFM_F64: seg_lines<IFM_F64>(p, tb, st); break;
    case IFM_BF16: seg_lines<IFM_BF16>(p, tb, st); break;
    case IFM_F16: seg_lines<IFM_F16>(p, tb, st); break;
    case IFM_N0F8: seg_lines<IFM_N0F8>(p, tb, st); break;
    default: seg_lines<IFM_U8>(p, tb, st); break;
    }
    return hipGetLastError();
  }
  if (out.dtype != IFM_F64) return hipErrorInvalidValue;  // the longer lines' kernels keep forward values in dst
  if (stride == 1) {  // lines along the contiguous axis: LDS-staged chunks
    const unsigned nb = (unsigned)((p.lines + IR_L - 1) / IR_L);
    const size_t lds = sizeof(double) * IR_L * IR_P;
    if (in.dtype == IFM_F32) hipLaunchKernelGGL(k_iir_rows<IFM_F32>, dim3(nb), dim3(256), lds, st, p);
    else if (in.dtype == IFM_F64) hipLaunchKernelGGL(k_iir_rows<IFM_F64>, dim3(nb), dim3(256), lds, st, p);
    else hipLaunchKernelGGL(k_iir_rows<-1>, dim3(nb), dim3(256), lds, st, p);
    return hipGetLastError();
  }
  int64_t blocks = (p.lines + 255) / 256;
  const bool s1 = stride == 1;
  if (in.dtype == IFM_F32) {
    if (s1) hipLaunchKernelGGL((k_iir_strided<true, IFM_F32>), dim3((unsigned)blocks), dim3(256), 0, st, p);
    else hipLaunchKernelGGL((k_iir_strided<false, IFM_F32>), dim3((unsigned)blocks), dim3(256), 0, st, p);
  } else if (in.dtype == IFM_F64) {
    if (s1) hipLaunchKernelGGL((k_iir_strided<true, IFM_F64>), dim3((unsigned)blocks), dim3(256), 0, st, p);
    else hipLaunchKernelGGL((k_iir_strided<false, IFM_F64>), dim3((unsigned)blocks), dim3(256), 0, st, p);
  } else {
    if (s1) hipLaunchKernelGGL((k_iir_strided<true, -1>), dim3((unsigned)blocks), dim3(256), 0, st, p);
    else hipLaunchKernelGGL((k_iir_strided<false, -1>), dim3((unsigned)blocks), dim3(256), 0, st, p);
  }
  return hipGetLastError();
}

}  // namespace ifm
