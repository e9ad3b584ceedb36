// hmv_matmat.hip -- multi-right-hand-side H-matmat Y = H X + beta*Y on MFMA.
//
// X and Y hold k right-hand sides interleaved (row i's k values contiguous,
// N x k row-major); t likewise (slot s's k values at t[s*k]).  The apply runs
// over the same arena and work lists as the single-vector kernel, one wave
// (64 threads) per unit: a work item and a group of up to TW of its 16-row
// tiles.  Launches of few units give each NW waves, which take the unit's
// column groups in turn and add their accumulators in wave order at the end.
//
// The wave walks the item's columns four at a time.  Per column quad, one
// 16-byte (or 8/4-byte) load per lane and two tiles gives two 16 x 4 A
// fragments (lane l: rows 2 (l%16) and 2 (l%16) + 1 of column l/16 of the
// column-major block; a tile on its own: one entry, row l%16), and one load
// per lane and two RHS tiles gives two 4 x 16 B fragments (bcol) straight
// from the interleaved inputs: phase 1 from its item's x run, phase 2
// through a per-wave LDS table of the columns' input addresses (L2-resident
// inputs: the units of an XCD are neighbouring items, so they share
// columns).  Each (tile, RHS tile) pair then takes one
// MFMA (16x16x4; FP64, or FP32 for FP32/BF16 arenas) into its 16 x 16
// accumulator; the B fragment is shared by the group's tiles.  Loads run
// one group of U quads ahead of the MFMAs.  Columns past the block load
// A = 0 through the buffer range check and B = 0 from a zero row.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <algorithm>
#include <mutex>
#include <string>

#include "hmv_engine.h"
#include "hmv_inputs.h"
#include "hmv_internal.h"

namespace {

typedef double d4 __attribute__((ext_vector_type(4)));
typedef float f4 __attribute__((ext_vector_type(4)));
typedef double gd2 __attribute__((ext_vector_type(2)));
typedef float gf2 __attribute__((ext_vector_type(2)));

constexpr int kNT = 2;                  // nontemporal cache policy

__device__ inline __amdgpu_buffer_rsrc_t rsrc(const char *base, uint32_t nbytes) {
  return __builtin_amdgcn_make_buffer_rsrc((void *)base, (short)0, (int)nbytes, 0x00020000);
}

template <typename Acc>
struct Mfma;
// A fragment: lane l holds A[l%16][l/16]; B fragment: lane l holds
// B[l/16][l%16]; result register i of lane l is D[row(l, i)][l%16] (the two
// types order their result rows differently; measured on gfx950).
template <>
struct Mfma<double> {
  using acc = d4;
  __device__ static d4 op(double a, double b, d4 c) {
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
  }
  __device__ static int row(int lane, int i) { return (lane >> 4) + 4 * i; }
};
template <>
struct Mfma<float> {
  using acc = f4;
  __device__ static f4 op(float a, float b, f4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
  }
  __device__ static int row(int lane, int i) { return 4 * (lane >> 4) + i; }
};

// One A entry of a part as loaded (0 when off), widened to the accumulation
// type at its MFMA (so the load's wait sits at the MFMA).
template <int DT>
struct Entry;
template <>
struct Entry<HMV_DT_F64> {
  static constexpr int es = 8;
  using raw = double;
  __device__ static double load_raw(__amdgpu_buffer_rsrc_t r, uint32_t off) {
    return __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(r, off, 0, kNT));
  }
  __device__ static void load_pair(__amdgpu_buffer_rsrc_t r, uint32_t off, double &a, double &b) {
    const gd2 v = __builtin_bit_cast(gd2, __builtin_amdgcn_raw_buffer_load_b128(r, off, 0, kNT));
    a = v.x;
    b = v.y;
  }
  __device__ static double widen(double v) { return v; }
};
template <>
struct Entry<HMV_DT_F32> {
  static constexpr int es = 4;
  using raw = float;
  __device__ static float load_raw(__amdgpu_buffer_rsrc_t r, uint32_t off) {
    return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, off, 0, kNT));
  }
  __device__ static void load_pair(__amdgpu_buffer_rsrc_t r, uint32_t off, float &a, float &b) {
    const gf2 v = __builtin_bit_cast(gf2, __builtin_amdgcn_raw_buffer_load_b64(r, off, 0, kNT));
    a = v.x;
    b = v.y;
  }
  __device__ static float widen(float v) { return v; }
};
template <>
struct Entry<HMV_DT_BF16> {
  static constexpr int es = 2;
  using raw = uint32_t;
  __device__ static uint32_t load_raw(__amdgpu_buffer_rsrc_t r, uint32_t off) {
    return __builtin_amdgcn_raw_buffer_load_b16(r, off, 0, kNT);
  }
  __device__ static void load_pair(__amdgpu_buffer_rsrc_t r, uint32_t off, uint32_t &a,
                                   uint32_t &b) {
    a = __builtin_amdgcn_raw_buffer_load_b32(r, off, 0, kNT);
    b = a >> 16;  // widen() drops a's upper half
  }
  __device__ static float widen(uint32_t v) { return __uint_as_float(v << 16); }
};

// Tile-group width (tiles sharing one B fragment) by RHS tiles, and column
// quads per prefetch group by RHS tiles and active tiles (two groups of
// U * (NT + KT) loads per lane are live; measured on MI355X, deeper or
// wider groups do not gain).
// At KT = 8 (k > 64) two 16-row tiles share each B fragment with FP32
// MFMAs (k = 128: 4.14 against 4.52 ms at 327,680 unknowns), while FP64
// accumulators (twice the registers) are faster one tile per wave (5.2
// against 5.9 ms).
template <int KT, typename Acc>
struct Shape {  // default tiles per unit (TW) by RHS tile count and accumulator type
  static constexpr int TW = KT <= 1 ? 4 : KT <= 4 ? 2 : sizeof(Acc) == 4 ? 2 : 1;
  static constexpr int LOG_TW = TW == 4 ? 2 : TW == 2 ? 1 : 0;
};
template <int KT, int NT>
constexpr int group_quads() {
  return KT + NT <= 6 ? 4 : 2;
}

// Global-address-space inputs: loads through these are global loads, which
// count on vmcnt only (a generic pointer read from LDS would give flat
// loads, which also count on lgkmcnt and so serialise the LDS reads with
// the inputs in flight).
typedef const double __attribute__((address_space(1))) gdouble;

constexpr int kWin = 1024;  // input pointers tabled per window (LDS, per wave)
constexpr int kPad = 32;    // zero-input entries past a window (one group of columns)
// B source of columns past a window or part (never written)
__device__ __attribute__((aligned(16))) double g_zero_inputs[128];

// Right-hand side held by column j0 of RHS tile tt: 16 tt + j0 for one tile;
// from two on the tiles go in pairs, tile 2s + b holding 32 s + 2 j0 + b, so
// that a lane's inputs of the two tiles of a pair are adjacent and one
// 16-byte load brings both (for k = 128 five loads per column quad instead
// of nine: one for A, four for B; 4.62 against 4.96 ms at 327,680 unknowns,
// 2.53 against 2.72 at k = 64, products bit-equal; at k = 32 1.65 against
// 1.69 ms, at k = 50 2.52 against 2.70, at k = 96 4.52 against 4.77).
template <int KT>
constexpr bool bpaired() {
  return KT >= 2;
}
template <int KT>
__device__ inline int bcol(int tt, int j0) {
  return bpaired<KT>() ? 32 * (tt >> 1) + 2 * j0 + (tt & 1) : 16 * tt + j0;
}

// Per-wave constants of the B loads.  Lane l (j0 = l%16) points at its
// column's inputs + jl (jl = bcol(0, j0)); tile tt's input is jd[tt] =
// bcol(tt, j0) - jl past it.  EXACT (k == 16 KT, inputs 16-byte aligned):
// read at 16 tt, or paired tiles as aligned 16-byte loads; otherwise each
// input (KT = 1) is read at min(bcol, k - 1), each pair as a 16-byte load of
// 8-byte alignment at min(bcol, k - 2), where the pair that starts with the
// column's last input takes it from the second half (inputs j >= k only feed
// accumulator columns that are not stored; the clamps keep the reads inside
// the column's k values; k > 16 where there are pairs).
template <int KT>
struct BLane {
  int j0;  // l % 16: the A row of the lane and its accumulator column
  int jl;
  int jd[KT];
  int last;  // pair whose first input is the column's last one (k odd), or -1
};
typedef const gd2 __attribute__((address_space(1))) ggd2;
typedef gd2 gd2u __attribute__((aligned(8)));
typedef const gd2u __attribute__((address_space(1))) ggd2u;

// One prefetch group: U column quads of A (NT tiles) and B (KT RHS tiles),
// as loaded (widened to Acc at the MFMA).
template <int DT, int KT, int NT, int U>
struct Group {
  typename Entry<DT>::raw a[U][NT];
  double b[U][KT];
};

// Where the B loads of a column come from: the window's pointer table
// (tbl[col - tbase]), or, for a part whose inputs are one x run (phase 1),
// straight from that run (xr + col k) with zeros past column hi.
struct BSrc {
  gdouble *const *tbl;
  int tbase;
  gdouble *xr, *zr;
  int hi;
};

// Loads the group of part columns [q0, q0 + 4U): lane l takes column
// q0 + 4u + l/16.  A: row 16 (tile0 + m) + l%16 at byte offset
// col * cs + r_es + 16 m es of a tile on its own, rows 2 (l%16) and one past
// it of the 32 of a pair of tiles in one load (tile_row; its address is
// 4-byte aligned, all that a buffer load needs, since blocks of BF16 have an
// even number of padded rows; with an odd number of FP64 or FP32 rows the
// pair of the last row of the last column ends past the range, which is
// checked dword by dword: the row loads, what follows it is 0); a column past the part lies past the buffer
// range and loads 0, and rows past the block only feed accumulator rows
// that are not stored.  B: from the column's inputs as src gives them
// (zeros past the window or the part).

// Item row of accumulator row r of tile m of a unit of nt tiles: the tiles go
// in pairs, the first of a pair holding the even and the second the odd rows
// of its 32, so that a lane's entries of both are adjacent and one load brings
// them (163,840 unknowns, k = 16 695 -> 663 us, k = 17 797 -> 768, k = 32
// 877 -> 847, k = 64 1,351 -> 1,322; products bit-equal).
__device__ inline int tile_row(int tile0, int m, int nt, int r) {
  return m < (nt & ~1) ? (tile0 + (m & ~1)) * 16 + 2 * r + (m & 1) : (tile0 + m) * 16 + r;
}

template <bool EXACT, bool RUN, int DT, int KT, int NT, int U>
__device__ inline void load_group(Group<DT, KT, NT, U> &g, __amdgpu_buffer_rsrc_t rs, uint32_t cs,
                                 uint32_t r_es, int q0, const BSrc &src, int k,
                                 const BLane<KT> &bl) {
  using E = Entry<DT>;
  const int cq = (threadIdx.x & 63) >> 4;
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const int col = q0 + 4 * u + cq;
    const uint32_t cb = (uint32_t)col * cs + r_es;
#pragma unroll
    for (int m = 0; m + 1 < NT; m += 2)
      E::load_pair(rs, cb + (uint32_t)((m * 16 + bl.j0) * E::es), g.a[u][m], g.a[u][m + 1]);
    if constexpr (NT % 2 != 0)
      g.a[u][NT - 1] = E::load_raw(rs, cb + (uint32_t)((NT - 1) * 16 * E::es));
    gdouble *p;
    if constexpr (RUN)
      p = col < src.hi ? src.xr + (size_t)col * k : src.zr;
    else
      p = src.tbl[col - src.tbase] + bl.jl;
    if constexpr (EXACT && bpaired<KT>()) {
#pragma unroll
      for (int tt = 0; tt < KT; tt += 2) {
        const gd2 v = *(ggd2 *)(p + 32 * (tt >> 1));
        g.b[u][tt] = v.x;
        g.b[u][tt + 1] = v.y;
      }
    } else if constexpr (bpaired<KT>()) {
#pragma unroll
      for (int tt = 0; tt < KT; tt += 2) {
        const gd2u v = *(ggd2u *)(p + bl.jd[tt]);
        g.b[u][tt] = bl.last == (tt >> 1) ? v.y : v.x;
        g.b[u][tt + 1] = v.y;
      }
    } else {
#pragma unroll
      for (int tt = 0; tt < KT; ++tt) g.b[u][tt] = EXACT ? p[16 * tt] : p[bl.jd[tt]];
    }
  }
}

template <typename Acc, int DT, int KT, int TW, int NT, int U>
__device__ inline void mma_group(typename Mfma<Acc>::acc (&acc)[TW][KT],
                                 const Group<DT, KT, NT, U> &g) {
#pragma unroll
  for (int u = 0; u < U; ++u)
#pragma unroll
    for (int m = 0; m < NT; ++m) {
      const Acc a = (Acc)Entry<DT>::widen(g.a[u][m]);
#pragma unroll
      for (int tt = 0; tt < KT; ++tt)
        acc[m][tt] = Mfma<Acc>::op(a, (Acc)g.b[u][tt], acc[m][tt]);
    }
}

// Tables the input pointers of part columns [w0, w1) (item columns cbase +
// ...) at tbl[0 ..), and zeros for the kPad entries that follow.
template <int NW>
__device__ inline void fill_window(gdouble **__restrict__ tbl, const Inputs &in,
                                   const int *__restrict__ codes, int cbase, int w0, int w1,
                                   const double *__restrict__ x, const double *__restrict__ t,
                                   int k) {
  for (int i = (int)threadIdx.x; i < w1 - w0 + kPad; i += 64 * NW) {
    const double *p = g_zero_inputs;
    if (i < w1 - w0) {
      const int code = input_code(in, codes, cbase + w0 + i);
      p = code >= 0 ? x + (size_t)code * k : t + (size_t)(-1 - code) * k;
    }
    tbl[i] = (gdouble *)p;
  }
}

// Multiplies this wave's groups of part columns [lo, hi) into the
// accumulators (U quads a group, every NW-th group of the workgroup's NW
// waves), the next group's loads in flight while the current one multiplies.
template <typename Acc, bool EXACT, bool RUN, int DT, int KT, int TW, int NT, int NW>
__device__ inline void run_columns(typename Mfma<Acc>::acc (&acc)[TW][KT],
                                   __amdgpu_buffer_rsrc_t rs, uint32_t cs, uint32_t r_es, int lo,
                                   int hi, const BSrc &src, int k, const BLane<KT> &bl) {
  constexpr int U = group_quads<KT, NT>();
  constexpr int SG = 4 * U;   // columns per group
  constexpr int S = SG * NW;  // columns between a wave's groups
  static_assert(SG <= kPad, "a group past the window reads zero entries");
  Group<DT, KT, NT, U> g0, g1;
  if constexpr (NW > 1) {
    lo += SG * (int)(threadIdx.x >> 6);
    if (lo >= hi) return;
  }
  load_group<EXACT, RUN>(g0, rs, cs, r_es, lo, src, k, bl);
  int q0 = lo;
  for (; q0 + 2 * S < hi; q0 += 2 * S) {  // g0 holds group q0; two more follow
    load_group<EXACT, RUN>(g1, rs, cs, r_es, q0 + S, src, k, bl);
    mma_group<Acc>(acc, g0);
    load_group<EXACT, RUN>(g0, rs, cs, r_es, q0 + 2 * S, src, k, bl);
    mma_group<Acc>(acc, g1);
  }
  const bool last2 = q0 + S < hi;  // one or two groups left
  if (last2) load_group<EXACT, RUN>(g1, rs, cs, r_es, q0 + S, src, k, bl);
  mma_group<Acc>(acc, g0);
  if (last2) mma_group<Acc>(acc, g1);
}

// Accumulates the product of NT tiles over one part (ncolp columns stored
// with DT at rs, item columns cbase + [0, ncolp)).  Inputs of one x run
// (phase 1) are addressed directly; otherwise kWin columns at a time, the
// window's input pointers tabled in LDS first.
template <typename Acc, bool EXACT, bool RUN, int DT, int KT, int TW, int NT, int NW>
__device__ inline void part_mma(typename Mfma<Acc>::acc (&acc)[TW][KT], __amdgpu_buffer_rsrc_t rs,
                                int rows_p, int tile0, int ncolp, int cbase, const Inputs &in,
                                const int *__restrict__ codes, gdouble **__restrict__ tbl,
                                const double *__restrict__ x, const double *__restrict__ t, int k,
                                const BLane<KT> &bl) {
  if (ncolp <= 0) return;
  const uint32_t cs = (uint32_t)rows_p * Entry<DT>::es;
  const uint32_t r_es = (uint32_t)(tile0 * 16 + bl.j0) * Entry<DT>::es;
  if constexpr (RUN) {
    const BSrc src{nullptr, 0, (gdouble *)(x + (size_t)(in.z0.src + cbase) * k) + bl.jl,
                   (gdouble *)g_zero_inputs + bl.jl, ncolp};
    run_columns<Acc, EXACT, true, DT, KT, TW, NT, NW>(acc, rs, cs, r_es, 0, ncolp, src, k, bl);
  } else {
    for (int w0 = 0; w0 < ncolp; w0 += kWin) {
      const int w1 = min(ncolp, w0 + kWin);
      __syncthreads();  // the table's previous contents are read
      fill_window<NW>(tbl, in, codes, cbase, w0, w1, x, t, k);
      __syncthreads();
      const BSrc src{tbl, w0, nullptr, nullptr, w1};
      run_columns<Acc, EXACT, false, DT, KT, TW, NT, NW>(acc, rs, cs, r_es, w0, w1, src, k, bl);
    }
  }
}

// Both parts of the item for NT tiles (the unit's tile count, fixed at
// compile time so that the accumulators stay in place); an item stored
// with one type has one part.
template <typename Acc, bool EXACT, bool RUN, int DT0, int DT1, int KT, int TW, int NT, int NW>
__device__ inline void unit_mma(typename Mfma<Acc>::acc (&acc)[TW][KT], const HmvWork &w,
                                __amdgpu_buffer_rsrc_t rs0, __amdgpu_buffer_rsrc_t rs1, int tile0,
                                const Inputs &in, const int *__restrict__ codes,
                                gdouble **__restrict__ tbl, const double *__restrict__ x,
                                const double *__restrict__ t, int k, const BLane<KT> &bl) {
  part_mma<Acc, EXACT, RUN, DT0, KT, TW, NT, NW>(acc, rs0, w.rows_p, tile0, w.ncol0, 0, in, codes,
                                             tbl, x, t, k, bl);
  if constexpr (DT0 != DT1)
    part_mma<Acc, EXACT, RUN, DT1, KT, TW, NT, NW>(acc, rs1, w.rows_p, tile0, w.ncol1, w.ncol0, in,
                                               codes, tbl, x, t, k, bl);
}

// NW waves per unit {item, tile0 << 8 | nt}: tiles tile0 .. tile0+nt-1 of
// the item.  PHASE 1: t[outidx[out_base + row] * k + j];  PHASE 2:
// y[(out_base + row) * k + j].
template <typename Acc, int PHASE, int DT0, int DT1, int KT, int TW, bool EXACT, int NW>
__global__ __launch_bounds__(64 * NW) void hmv_matmat_kernel(
    const char *__restrict__ arena, const HmvWork *__restrict__ works, const int2 *__restrict__ units,
    const HmvZSeg *__restrict__ zsegs, const double *__restrict__ x, const int *__restrict__ codes,
    const double *__restrict__ t_in, const int *__restrict__ outidx, double *__restrict__ t_out,
    double *__restrict__ yp, double *__restrict__ y, int k, double beta,
    const int *__restrict__ skip) {
  if (skip && *skip) return;
  static_assert(TW == 1 || TW == 2 || TW == 4, "tiles per unit");
  __shared__ int runs[2 * HMV_RUN_MAX];
  __shared__ gdouble *tbl[PHASE == 1 ? 1 : kWin + kPad];  // phase 1 reads its x run directly
  const int2 unit = units[blockIdx.x];
  const HmvWork w = works[unit.x];
  const int tile0 = unit.y >> 8, nt = unit.y & 255;
  const int lane = threadIdx.x & 63;
  BLane<KT> bl;
  bl.j0 = lane & 15;
  bl.jl = bcol<KT>(0, bl.j0);
#pragma unroll
  for (int tt = 0; tt < KT; ++tt)
    bl.jd[tt] = min(bcol<KT>(tt, bl.j0), k - (bpaired<KT>() ? 2 : 1)) - bl.jl;
  bl.last = (k & 1) && bl.j0 == ((k - 1) & 31) >> 1 ? (k - 1) >> 5 : -1;
  const Inputs in = load_inputs<64 * NW>(w, zsegs, runs);
  const __amdgpu_buffer_rsrc_t rs0 =
      rsrc(arena + w.off0, (uint32_t)((size_t)w.rows_p * w.ncol0 * Entry<DT0>::es));
  const __amdgpu_buffer_rsrc_t rs1 =
      rsrc(arena + (w.ncol1 > 0 ? w.off1 : w.off0),
           (uint32_t)((size_t)w.rows_p * w.ncol1 * Entry<DT1>::es));
  typename Mfma<Acc>::acc acc[TW][KT];
#pragma unroll
  for (int m = 0; m < TW; ++m)
#pragma unroll
    for (int tt = 0; tt < KT; ++tt) acc[m][tt] = typename Mfma<Acc>::acc{0, 0, 0, 0};
  if (nt >= TW)
    unit_mma<Acc, EXACT, PHASE == 1, DT0, DT1, KT, TW, TW, NW>(acc, w, rs0, rs1, tile0, in, codes, tbl, x, t_in, k,
                                               bl);
  else if constexpr (TW == 2)
    unit_mma<Acc, EXACT, PHASE == 1, DT0, DT1, KT, TW, 1, NW>(acc, w, rs0, rs1, tile0, in, codes, tbl, x, t_in, k,
                                              bl);
  else if constexpr (TW == 4) {
    if (nt == 1)
      unit_mma<Acc, EXACT, PHASE == 1, DT0, DT1, KT, TW, 1, NW>(acc, w, rs0, rs1, tile0, in, codes, tbl, x, t_in,
                                                k, bl);
    else if (nt == 2)
      unit_mma<Acc, EXACT, PHASE == 1, DT0, DT1, KT, TW, 2, NW>(acc, w, rs0, rs1, tile0, in, codes, tbl, x, t_in,
                                                k, bl);
    else
      unit_mma<Acc, EXACT, PHASE == 1, DT0, DT1, KT, TW, 3, NW>(acc, w, rs0, rs1, tile0, in, codes, tbl, x, t_in,
                                                k, bl);
  }
  if constexpr (NW > 1) {
    // the waves' accumulators, summed in wave order by wave 0
    __shared__ typename Mfma<Acc>::acc sums[NW - 1][64];
    const int wv = threadIdx.x >> 6;
#pragma unroll
    for (int m = 0; m < TW; ++m) {
      if (m >= nt) continue;
#pragma unroll
      for (int tt = 0; tt < KT; ++tt) {
        __syncthreads();  // the previous tile's sums are read
        if (wv > 0) sums[wv - 1][lane] = acc[m][tt];
        __syncthreads();
        if (wv == 0)
          for (int q = 0; q < NW - 1; ++q) acc[m][tt] += sums[q][lane];
      }
    }
    if (wv > 0) return;
  }
  // lane holds rows Mfma::row(lane, i), column lane%16 of each 16 x 16 tile
  const int j0 = lane & 15;
#pragma unroll
  for (int m = 0; m < TW; ++m) {
    if (m >= nt) continue;
#pragma unroll
    for (int tt = 0; tt < KT; ++tt) {
      const int j = bcol<KT>(tt, j0);
      if (j >= k) continue;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int row = tile_row(tile0, m, min(nt, TW), Mfma<Acc>::row(lane, i));
        if (row >= w.rows) continue;
        const double v = (double)acc[m][tt][i];
        if constexpr (PHASE == 1) {
          t_out[(size_t)outidx[w.out_base + row] * k + j] = v;
        } else {
          if (w.out_base < 0) {  // a piece of a wide item
            yp[(size_t)(row - 1 - w.out_base) * k + j] = v;
            continue;
          }
          double *py = y + (size_t)(w.out_base + row) * k + j;
          *py = beta == 0.0 ? v : __builtin_fma(beta, *py, v);
        }
      }
    }
  }
}

// t[slot*k + j] = sum over p of t[(base+p)*k + j], in chunk order.
__global__ __launch_bounds__(256) void hmv_tfinal_block_kernel(const HmvTFin *__restrict__ fin,
                                                               int nfin, int k,
                                                               double *__restrict__ t,
                                                               const int *__restrict__ skip) {
  if (skip && *skip) return;
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= (int64_t)nfin * k) return;
  const HmvTFin f = fin[i / k];
  const int j = (int)(i % k);
  double s = t[(size_t)f.base * k + j];
  for (int p = 1; p < f.np; ++p) s += t[(size_t)(f.base + p) * k + j];
  t[(size_t)f.slot * k + j] = s;
}

// Rows of the wide items: y = sum of the pieces' partial rows in piece order
// + beta y (k columns interleaved; a workgroup per item and kYRhs of its
// right-hand sides' worth of elements).
constexpr int kYRhs = 4;
__global__ __launch_bounds__(256) void hmv_yfinal_block_kernel(const HmvYFin *__restrict__ fin, int k,
                                                               const double *__restrict__ yp,
                                                               double *__restrict__ y, double beta,
                                                               const int *__restrict__ skip) {
  if (skip && *skip) return;
  const HmvYFin f = fin[blockIdx.x];
  const size_t n = (size_t)f.rows * k;
  double *py = y + (size_t)f.row * k;
  for (size_t e = blockIdx.y * 256 + threadIdx.x; e < n; e += 256 * gridDim.y) {
    const double s = sum_pieces(yp + (size_t)f.base * k + e, n, f.np);
    py[e] = beta == 0.0 ? s : __builtin_fma(beta, py[e], s);
  }
}

// Up to this many units (two fills of the chip at four waves per SIMD), a
// unit's columns are shared by several waves: one wave per unit leaves SIMDs
// idle or with a lone last unit, and a unit's time is its column groups' round
// trips.  Phase 2 (some 1,000 columns an item): four waves; 5,120 unknowns (356
// units), k = 16 / 32 / 128: 29 / 34 / 65 -> 16 / 22 / 38 us; 42,235 (3,113),
// k = 19 / 40: 136 / 232 -> 116 / 200 us; 81,920 (5,674), k = 32: 266 -> 230 us.
// At 327,680 (22,855 units) k = 16 loses 10% and k = 32 gains 1%: one wave.
// Phase 1 (median 50 to 80 columns): two; 42,235 unknowns (7,876 units) 101 ->
// 90 and 189 -> 161 us; from 12,756 units on 3% faster to 19% slower.
constexpr int kFewUnits = 8192;
template <int PHASE>
constexpr int few_waves() {
  return PHASE == 1 ? 2 : 4;
}

template <typename Acc, int PHASE, int DT0, int DT1>
void launch_units(int kt, const HmvLaunch &L, const HmvUnits &U, const HmvWork *works,
                  const double *x, double *t, double *yp, double *y, int k, double beta,
                  const int *skip, hipStream_t s) {
  const double *t_in = PHASE == 2 ? t : nullptr;
  double *t_out = PHASE == 1 ? t : nullptr;
  // EXACT reads the inputs in 16-byte pairs: x and t must be 16-byte aligned
  // (a caller's x may start anywhere; t is allocated by the engine)
  const bool exact = ((uintptr_t)x % 16 == 0) && ((uintptr_t)t % 16 == 0);
#define HMV_MM_GO(KT, TW, EX, NW)                                                              \
  hipLaunchKernelGGL((hmv_matmat_kernel<Acc, PHASE, DT0, DT1, KT, TW, EX, NW>), dim3(n),       \
                     dim3(64 * NW), 0, s, L.arena, works, U.u[PHASE - 1][w], L.zseg, x, L.codes, \
                     t_in, L.outidx, t_out, yp, y, k, beta, skip)
#define HMV_MM_LAUNCH(KT, TW)                                      \
  do {                                                             \
    const int w = TW == 4 ? 2 : TW == 2 ? 1 : 0, n = U.n[PHASE - 1][w]; \
    const bool few = n <= kFewUnits, ex = exact && k == 16 * KT;   \
    if (n > 0) {                                                   \
      if (few && ex)                                               \
        HMV_MM_GO(KT, TW, true, few_waves<PHASE>());               \
      else if (few)                                                \
        HMV_MM_GO(KT, TW, false, few_waves<PHASE>());              \
      else if (ex)                                                 \
        HMV_MM_GO(KT, TW, true, 1);                                \
      else                                                         \
        HMV_MM_GO(KT, TW, false, 1);                               \
    }                                                              \
  } while (0)
  // tiles per unit: the tuned choice of the KT class when it is one of the
  // two instantiated for it, else the default (Shape)
  const int lt = U.log_tw[kt == 1 ? 0 : kt == 2 ? 1 : kt <= 4 ? 2 : 3];
  if (kt == 1) {
    if (lt == 1 || (lt < 0 && Shape<1, Acc>::TW == 2))
      HMV_MM_LAUNCH(1, 2);
    else
      HMV_MM_LAUNCH(1, 4);
  } else if (kt == 2) {
    if (lt == 0 || (lt < 0 && Shape<2, Acc>::TW == 1))
      HMV_MM_LAUNCH(2, 1);
    else
      HMV_MM_LAUNCH(2, 2);
  } else if (kt <= 4) {
    if (lt == 0 || (lt < 0 && Shape<4, Acc>::TW == 1))
      HMV_MM_LAUNCH(4, 1);
    else
      HMV_MM_LAUNCH(4, 2);
  } else {
    if (lt == 1 || (lt < 0 && Shape<8, Acc>::TW == 2))
      HMV_MM_LAUNCH(8, 2);
    else
      HMV_MM_LAUNCH(8, 1);
  }
#undef HMV_MM_LAUNCH
#undef HMV_MM_GO
}

template <typename Acc, int DT0, int DT1>
void launch_block(const HmvLaunch &L, const HmvUnits &U, int k, const double *x, double *t,
                  double *yp, double *y, double beta, const int *skip, hipStream_t s) {
  const int kt = (k + 15) / 16;
  // few right-hand sides stream on the vector units (hmv_kstream.hip) unless
  // the arena's tuning sends their class to MFMA
  const bool vec = k <= (L.mode == 0 ? HMV_KSTREAM_MAX_F64 : HMV_KSTREAM_MAX_NARROW) &&
                   U.vec[k <= 1 ? 0 : k <= 2 ? 1 : k <= 4 ? 2 : 3];
  if (vec)
    (void)hmv_launch_kstream(&L, 1, k, x, t, nullptr, nullptr, 0.0, skip, s);
  else
    launch_units<Acc, 1, DT1, DT1>(kt, L, U, L.work1, x, t, nullptr, nullptr, k, 0.0, skip, s);
  if (L.ntfin > 0) {
    const int64_t n = (int64_t)L.ntfin * k;
    hipLaunchKernelGGL(hmv_tfinal_block_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s,
                       L.tfin, L.ntfin, k, t, skip);
  }
  if (vec)
    (void)hmv_launch_kstream(&L, 2, k, x, t, yp, y, beta, skip, s);
  else
    launch_units<Acc, 2, DT0, DT1>(kt, L, U, L.work2, x, t, yp, y, k, beta, skip, s);
  if (L.nyfin > 0)
    hipLaunchKernelGGL(hmv_yfinal_block_kernel, dim3(L.nyfin, (k + kYRhs - 1) / kYRhs), dim3(256),
                       0, s, L.yfin, k, yp, y, beta, skip);
}

}  // namespace

// Y = H X + beta*Y for k (1..128) interleaved right-hand sides; t holds
// tpart_size * k doubles, yp the partial rows * k.
extern "C" hipError_t hmv_launch_block(const HmvLaunch *L, const HmvUnits *units, int k,
                                       const double *x, double *t, double *yp, double *y,
                                       double beta, const int *skip, hipStream_t stream) {
  if (L->mode == 0)
    launch_block<double, HMV_DT_F64, HMV_DT_F64>(*L, *units, k, x, t, yp, y, beta, skip, stream);
  else if (L->mode == 1)
    launch_block<float, HMV_DT_F32, HMV_DT_F32>(*L, *units, k, x, t, yp, y, beta, skip, stream);
  else if (L->mode == 2)
    launch_block<float, HMV_DT_F32, HMV_DT_BF16>(*L, *units, k, x, t, yp, y, beta, skip, stream);
  else
    launch_block<float, HMV_DT_BF16, HMV_DT_BF16>(*L, *units, k, x, t, yp, y, beta, skip, stream);
  return hipGetLastError();
}

// ---------------------------------------------------------------------------
// Static workspace of hmv_apply_block_static: the H-matmat's t buffer
// (tpart_size * k doubles) in a file-scope device array instead of memory
// allocated on first use.  Every device the library runs on holds its own
// copy until the process ends; host code never passes `scratch` itself (on
// the host it names a stand-in, not device memory): the device address of
// each device's copy comes from hipGetSymbolAddress, taken once per device
// with that device current, and only that address reaches the kernels.
// Nothing in it needs clearing between calls: phase 1 writes every t slot
// and chunk partial that the finalize and phase 2 read.  Calls that overlap
// on one device share the array and race.  The partial rows of wide items
// are in memory of their arena (d_yp), made with it.
static __device__ __align__(256) double scratch[HMV_STATIC_SCRATCH_BYTES / sizeof(double)];

namespace {
constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
double *g_scratch[kMaxDevices] = {};
}  // namespace

namespace hmv {
// Device address of the current device's copy of `scratch`, looked up on
// the first call per device.
int static_scratch(double **out) {
  *out = nullptr;
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return hip_fail(e, "static scratch: hipGetDevice");
  if (dev < 0 || dev >= kMaxDevices) {
    set_error("static scratch: device index " + std::to_string(dev) + " out of range");
    return HMV_ERR_DEVICE;
  }
  std::lock_guard<std::mutex> lk(g_scratch_mu);
  if (!g_scratch[dev]) {
    void *p = nullptr;
    e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess) return hip_fail(e, "static scratch: hipGetSymbolAddress");
    if (!p) {
      set_error("static scratch: no device address");
      return HMV_ERR_DEVICE;
    }
    g_scratch[dev] = static_cast<double *>(p);
  }
  *out = g_scratch[dev];
  return HMV_OK;
}
}  // namespace hmv

extern "C" int hmv_apply_block_static(hmv_arena a, int k, const double *x, double *y, double beta,
                                      void *stream) {
  if (!a || !x || !y || k < 1 || k > HMV_MAX_RHS) {
    hmv::set_error("hmv_apply_block_static: invalid argument (k must be 1..128)");
    return HMV_ERR_ARG;
  }
  const int64_t need = std::max<int64_t>(1, a->tpart_size) * k * (int64_t)sizeof(double);
  if (k > hmv::static_max_rhs(a->tpart_size)) {
    hmv::set_error("hmv_apply_block_static: the product needs " + std::to_string(need) +
                   " bytes of t buffer (k = " + std::to_string(k) +
                   "), the static scratch holds " + std::to_string(HMV_STATIC_SCRATCH_BYTES));
    return HMV_ERR_ARG;
  }
  int dev = -1;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return hmv::hip_fail(e, "hmv_apply_block_static");
  if (dev != a->device) {
    hmv::set_error("hmv_apply_block_static: the arena lives on device " +
                   std::to_string(a->device) + ", the current device is " + std::to_string(dev));
    return HMV_ERR_ARG;
  }
  double *t = nullptr;
  int rc = hmv::static_scratch(&t);
  if (rc) return rc;
  HmvUnits u;
  hmv::fill_units(a, u);
  e = hmv_launch_block(&a->launch, &u, k, x, t, a->d_yp + a->launch.nyp, y, beta, nullptr,
                       (hipStream_t)stream);
  if (e != hipSuccess) return hmv::hip_fail(e, "hmv_apply_block_static: launch");
  return HMV_OK;
}
