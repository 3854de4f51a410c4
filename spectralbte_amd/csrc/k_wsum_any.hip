// k_wsum_any.hip -- folded weighted sum on grids without streaming tiles (FP64).
//
// The sum of k_wsum_stream.hip over the kept rows and columns (see k_fold_w
// there), for any N up to 24: the reference's own N = 8, odd grids, 10, 12, 18,
// 20.  These sums are short (N = 10: 2.8e5 pairs a cell), so what bounds them is
// latency and how much of the chip a batch fills, then LDS: a 16-byte read of F per
// step, product and cell feeds 4 or 5 FP64 instructions a row.
//  * A workgroup owns an x-plane of output rows, TR consecutive ones a lane, for TB
//    cells and a slice of the summed z-lines; c is the same in all lanes, so G is
//    read by scalar loads.
//  * Per summed plane the shifted F x-plane of every cell and product is staged
//    in LDS with every z-line twice in a row: the operand of step cz is at a fixed
//    offset -cz from the lane's base and never wraps; a lane's TR operands slide by
//    one entry a step, so they cost one read (N = 18, 160 cells maxPreserve: 1376 us an
//    evaluation with 3 rows a lane, 2357 with one; N = 10, 75 cells: 76 and 83).
//  * W is column-major over the rows of a plane, padded to whole waves: a wave
//    reads 64 TR contiguous doubles per column, each value feeding TB cells.  With
//    N known at compile time a z-line's weights are all loaded before the first is
//    used, and where registers allow (NT TR <= 40) a line ahead.
// Measured on an MI355X, the sum alone, against one thread per (row, cell) over the
// whole table (k_wsum_generic, which still serves operands that are not
// transforms of real cells, and N > 24, whose staged planes outgrow LDS):
//   N = 8, 250 cells ComputeQ     209 -> 25 us     N = 12, 300 cells maxPr.   8055 -> 381 us
//   N = 10, 75 cells maxPreserve  539 -> 36 us     N = 18, 160 cells maxPr.  101.4 -> 1.27 ms
//   N = 10, one cell maxPreserve  355 -> 12 us     N = 20, 120 cells maxPr.  126.4 -> 2.41 ms
// (even N under 16 sum all rows, see build_mirror: N = 12 252 and N = 10 27 us with half of them).
// N = 18 and 160 cells is 21 TFLOP/s of FP64 (64 measured on FMA chains).
#include <hip/hip_runtime.h>
#include "spbte_internal.h"

namespace {

constexpr int kMaxThreads = 512;

// Rows per lane, consecutive in z: they share every LDS read of F.  As many as
// cost no more (or little more) instructions for the lanes that stay idle in the
// last wave of a plane: N = 10 takes one wave of 50 lanes instead of 100 rows in two.
__host__ __device__ constexpr int rows_per_lane(int N) {
  return N == 12 || N == 18 ? 3 : (N == 20 ? 4 : (N == 10 || N == 14 || N == 22 ? 2 : 1));
}
// Lanes of an x-plane of rows, in whole waves.
__host__ __device__ inline int lane_pad(int N) { return (N * N / rows_per_lane(N) + 63) / 64 * 64; }
// Line slot -> cy: from the outermost to the middle (the large terms last).
__host__ __device__ inline int line_cy(int N, int cl) { return (cl & 1) ? N - 1 - cl / 2 : cl / 2; }

// NT: N at compile time, 0: Nrt; TR rows per lane.
template <int NT, int TR, int NP, int TB>
__global__ void __launch_bounds__(kMaxThreads)
k_wsum_any(int Nrt, int npl, int cfold, const double *__restrict__ Wf, const double2 *__restrict__ F0,
           const double2 *__restrict__ G0, const double2 *__restrict__ F1, const double2 *__restrict__ G1,
           double2 *__restrict__ Qh, int ncell, int csplit, int chunks, double2 *__restrict__ Qp) {
  extern __shared__ __attribute__((aligned(16))) char smem_any[];
  double2 *sF = (double2 *)smem_any;  // [p][b][sy][LE]
  const int N = NT ? NT : Nrt, n2 = N * N, h = N / 2, LP = lane_pad(N), NL = n2 / TR;
  const int LE = 2 * N + TR - 1;  // a staged line: entry q is F[q mod N]
  const size_t n3 = (size_t)n2 * N;
  // XCD x takes the x-th contiguous slice of the list with cell groups innermost,
  // so that the workgroups sharing a piece of W share an L2
  const int ncg = (ncell + TB - 1) / TB, total = npl * chunks * csplit * ncg, per = (total + 7) >> 3;
  const int vid = (blockIdx.x & 7) * per + (blockIdx.x >> 3);
  if ((int)(blockIdx.x >> 3) >= per || vid >= total) return;
  const int cg = vid % ncg, r1 = vid / ncg, cs = r1 % csplit, r2 = r1 / csplit, ch = r2 % chunks, rx = r2 / chunks;
  int first;
  const int ncx = spbte_fold_planes(N, rx, npl < N, cfold, &first);
  first += ncx - 1;  // the outermost plane first
  const int ncols = (cfold ? N / 2 + 1 : N) * n2;
  // this slice's z-lines of the kept summed planes: whole planes where there are
  // enough of them (each plane is then staged once; N = 8, 250 cells: 23.0 us against 25.3)
  const int un = csplit <= ncx ? N : 1, nu = ncx * N / un;
  const int l0 = cs * nu / csplit * un, l1 = (cs + 1) * nu / csplit * un;
  const int lane = ch * blockDim.x + threadIdx.x;
  const int row = (lane < NL ? lane : NL - 1) * TR;
  const int ry = row / N, rz = row - ry * N;
  const double *Wr = Wf + ((size_t)rx * ncols * LP + (lane < LP ? lane : LP - 1)) * TR;
  const size_t ws = (size_t)LP * TR;  // column stride
  const double2 *Fp[2] = {F0, F1}, *Gp[2] = {G0, G1};
  size_t cells[TB];
#pragma unroll
  for (int b = 0; b < TB; ++b) cells[b] = (size_t)(cg * TB + b < ncell ? cg * TB + b : ncell - 1) * n3;
  double2 tot[TB][TR];
#pragma unroll
  for (int b = 0; b < TB; ++b)
#pragma unroll
    for (int t = 0; t < TR; ++t) tot[b][t] = make_double2(0.0, 0.0);

  for (int ln0 = l0; ln0 < l1; ln0 = (ln0 / N + 1) * N) {
    const int cx = cfold ? (first - ln0 / N) % N : ln0 / N;
    const int cl0 = ln0 % N, cl1 = l1 - ln0 < N - cl0 ? cl0 + l1 - ln0 : N;
    const int sx = (rx + h - cx + N) % N;
    __syncthreads();
    for (int e = threadIdx.x; e < NP * TB * n2; e += blockDim.x) {
      const int q = e / n2, yz = e - q * n2, y = yz / N, z = yz - y * N;
      const int p = q / TB, b = q - p * TB;
      size_t co = cells[0];
#pragma unroll
      for (int i = 1; i < TB; ++i) co = b == i ? cells[i] : co;
      const double2 v = Fp[p][co + (size_t)sx * n2 + yz];
      double2 *o = sF + (q * N + y) * LE + z;
      o[0] = v;
      o[N] = v;
      if (z < TR - 1) o[2 * N] = v;
    }
    __syncthreads();
    double2 acc[TB][TR];
#pragma unroll
    for (int b = 0; b < TB; ++b)
#pragma unroll
      for (int t = 0; t < TR; ++t) acc[b][t] = make_double2(0.0, 0.0);
    // one step: w[t] for the lane's rows; f[p][b][t] their operands
    const auto step = [&](const double *w, size_t c, const double2 (&f)[NP][TB][TR]) __attribute__((always_inline)) {
#pragma unroll
      for (int b = 0; b < TB; ++b) {
        const double2 g0 = Gp[0][cells[b] + c];
        double2 g1 = g0;
        if constexpr (NP == 2) g1 = Gp[1][cells[b] + c];
#pragma unroll
        for (int t = 0; t < TR; ++t) {
          const double2 f0 = f[0][b][t];
          double pr = g0.x * f0.x, pi = g0.x * f0.y;
          pr = fma(-g0.y, f0.y, pr);
          pi = fma(g0.y, f0.x, pi);
          if constexpr (NP == 2) {
            const double2 f1 = f[1][b][t];
            pr = fma(g1.x, f1.x, pr);
            pi = fma(g1.x, f1.y, pi);
            pr = fma(-g1.y, f1.y, pr);
            pi = fma(g1.y, f1.x, pi);
          }
          acc[b][t].x = fma(w[t], pr, acc[b][t].x);
          acc[b][t].y = fma(w[t], pi, acc[b][t].y);
        }
      }
    };
    const double *Wl = Wr + (size_t)(ln0 - cl0) * N * ws;  // the plane's columns
    constexpr bool PF = NT != 0 && NT * TR <= 40;  // the next line's weights ahead, in registers
    double wn[PF ? NT : 1][TR];
    if constexpr (PF)
#pragma unroll
      for (int cz = 0; cz < NT; ++cz)
#pragma unroll
        for (int t = 0; t < TR; ++t) wn[cz][t] = Wl[(cl0 * NT + cz) * ws + t];
    constexpr int kLines = NT == 8 ? 2 : 1;  // z-lines a loop body (more than N = 8's spill)
#pragma unroll kLines
    for (int cl = cl0; cl < cl1; ++cl) {
      const int cy = line_cy(N, cl);
      int sy = ry + h - cy;
      sy = sy < 0 ? sy + N : (sy > N - 1 ? sy - N : sy);
      const double2 *line = sF + sy * LE + (rz + h) % N + N;
      const size_t c0 = (size_t)(cx * N + cy) * N;
      // window: f[t] of step cz is line[t - cz]; each step reads one element
      double2 f[NP][TB][TR];
#pragma unroll
      for (int p = 0; p < NP; ++p)
#pragma unroll
        for (int b = 0; b < TB; ++b)
#pragma unroll
          for (int t = 0; t < TR; ++t) f[p][b][t] = line[(p * TB + b) * N * LE + t];
      const auto slide = [&](int cz) __attribute__((always_inline)) {
#pragma unroll
        for (int p = 0; p < NP; ++p)
#pragma unroll
          for (int b = 0; b < TB; ++b) {
#pragma unroll
            for (int t = TR - 1; t > 0; --t) f[p][b][t] = f[p][b][t - 1];
            f[p][b][0] = line[(p * TB + b) * N * LE - cz];
          }
      };
      if constexpr (NT != 0) {
        double w[NT][TR];
        [[maybe_unused]] const int nx = cl + 1 < cl1 ? cl + 1 : cl;  // the last line again, not past the slice
#pragma unroll
        for (int cz = 0; cz < NT; ++cz)
#pragma unroll
          for (int t = 0; t < TR; ++t) {
            if constexpr (PF) {
              w[cz][t] = wn[cz][t];
              wn[cz][t] = Wl[(nx * NT + cz) * ws + t];
            } else {
              w[cz][t] = Wl[(cl * NT + cz) * ws + t];
            }
          }
#pragma unroll
        for (int cz = 0; cz < NT; ++cz) {
          if (cz) slide(cz);
          step(w[cz], c0 + cz, f);
        }
      } else {
#pragma unroll 2
        for (int cz = 0; cz < N; ++cz) {
          if (cz) slide(cz);
          double w[TR];
#pragma unroll
          for (int t = 0; t < TR; ++t) w[t] = Wl[(cl * N + cz) * ws + t];
          step(w, c0 + cz, f);
        }
      }
    }
#pragma unroll
    for (int b = 0; b < TB; ++b)
#pragma unroll
      for (int t = 0; t < TR; ++t) {
        tot[b][t].x += acc[b][t].x;
        tot[b][t].y += acc[b][t].y;
      }
  }
  if (lane >= NL) return;
#pragma unroll
  for (int b = 0; b < TB; ++b) {
    const int cell = cg * TB + b;
    if (cell >= ncell) continue;
    double2 *o = (csplit > 1 ? Qp + ((size_t)cs * ncell + cell) * n3 : Qh + (size_t)cell * n3) + (size_t)rx * n2 + row;
#pragma unroll
    for (int t = 0; t < TR; ++t) o[t] = tot[b][t];
  }
}

// Natural FP64 table -> folded, [rx][column slot][lane of the plane, padded][row].
__global__ void __launch_bounds__(256) k_fold_any(const double *__restrict__ W, double *__restrict__ out, int N, int npl,
                                                  int cfold, spbte_mirror mr) {
  const int n2 = N * N, h = N / 2, RP = lane_pad(N) * rows_per_lane(N), ncp = cfold ? N / 2 + 1 : N;
  const size_t n3 = (size_t)n2 * N, ncols = (size_t)ncp * n2, total = npl * ncols * RP;
  const int a2 = 2 * h;
  for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < total; i += (size_t)gridDim.x * blockDim.x) {
    const int row = (int)(i % RP);
    const size_t q = i / RP;
    const int col = (int)(q % ncols), rx = (int)(q / ncols);
    const int j = col / n2, cl = col / N % N, cz = col % N, cy = line_cy(N, cl);
    int first;
    const int ncx = spbte_fold_planes(N, rx, npl < N, cfold, &first);
    double x = 0.0;
    if (row < n2 && j < ncx) {
      const int ry = row / N, rz = row % N;
      const int cx = cfold ? (first + ncx - 1 - j) % N : j;
      const int sx = (rx + h - cx + N) % N, sy = (ry + h - cy + N) % N, sz = (rz + h - cz + N) % N;
      const bool pair = cfold && sx != cx;
      const double *Wr = W + ((size_t)rx * n2 + row) * n3;
      x = Wr[((size_t)cx * N + cy) * N + cz];
      if (pair) x += Wr[((size_t)sx * N + sy) * N + sz];
      if (npl < N && spbte_fold_image(N, rx, cx, cfold)) {
        const int mx = (a2 - rx + N) % N, my = (a2 - ry + N) % N, mz = (a2 - rz + N) % N;
        const double *Wm = W + (((size_t)mx * N + my) * N + mz) * n3;
        double y = Wm[((size_t)((a2 - cx + N) % N) * N + (a2 - cy + N) % N) * N + (a2 - cz + N) % N];
        if (pair) y += Wm[((size_t)((a2 - sx + N) % N) * N + (a2 - sy + N) % N) * N + (a2 - sz + N) % N];
        x += mr.r[rx] * mr.r[ry] * mr.r[rz] * mr.s[cx] * mr.s[cy] * mr.s[cz] * mr.s[sx] * mr.s[sy] * mr.s[sz] * y;
      }
    }
    out[i] = x;
  }
}

size_t lds_bytes(int N, int nprod, int tb) { return (size_t)nprod * tb * N * (2 * N + rows_per_lane(N) - 1) * sizeof(double2); }

// Cells per workgroup: two share each weight where one a workgroup would give a folded
// table two waves on every SIMD already, with one product one (N = 8, 250 cells: 42 us an
// evaluation against 47; fewer, and the slices that make up for it cost more in staging
// and in the inverse transform's sum), and both cells' planes fit 64 KiB of LDS.
int any_tb(int N, int nprod, int ncell) {
  return ncell >= 2 && (long)(N / 2 + 1) * (lane_pad(N) / 64) * ncell >= (nprod == 1 ? 1024 : 2048) && lds_bytes(N, nprod, 2) <= 65536 ? 2 : 1;
}

template <int NT, int TR, int NP>
void launch_any(int N, int npl, int cfold, int tb, const spbte_wsum_args *a, const void *Wf, int csplit, void *Qp,
                hipStream_t s) {
  const int LP = lane_pad(N), chunks = (LP + kMaxThreads - 1) / kMaxThreads;
  const int T = ((LP / 64 + chunks - 1) / chunks) * 64;
  const size_t lds = lds_bytes(N, NP, tb);
  const int total = npl * chunks * csplit * ((a->ncell + tb - 1) / tb), per = (total + 7) / 8;
  if (tb == 2)
    hipLaunchKernelGGL((k_wsum_any<NT, TR, NP, 2>), dim3(8 * per), dim3(T), lds, s, N, npl, cfold, (const double *)Wf,
                       (const double2 *)a->F0, (const double2 *)a->G0, (const double2 *)a->F1, (const double2 *)a->G1,
                       (double2 *)a->Qh, a->ncell, csplit, chunks, (double2 *)Qp);
  else
    hipLaunchKernelGGL((k_wsum_any<NT, TR, NP, 1>), dim3(8 * per), dim3(T), lds, s, N, npl, cfold, (const double *)Wf,
                       (const double2 *)a->F0, (const double2 *)a->G0, (const double2 *)a->F1, (const double2 *)a->G1,
                       (double2 *)a->Qh, a->ncell, csplit, chunks, (double2 *)Qp);
}

template <int NT, int TR>
void launch_np(int N, int npl, int cfold, int tb, const spbte_wsum_args *a, const void *Wf, int csplit, void *Qp,
               hipStream_t s) {
  if (a->nprod == 2) launch_any<NT, TR, 2>(N, npl, cfold, tb, a, Wf, csplit, Qp, s);
  else launch_any<NT, TR, 1>(N, npl, cfold, tb, a, Wf, csplit, Qp, s);
}

}  // namespace

extern "C" int spbte_any_supported(int N) { return N >= 2 && N <= 24; }

// Bytes of a folded table.
extern "C" size_t spbte_any_table_bytes(int N, int npl, int cfold) {
  return (size_t)npl * (cfold ? N / 2 + 1 : N) * N * N * lane_pad(N) * rows_per_lane(N) * 8;
}

// Slices of the summed z-lines: as many as give 4096 waves (four on every SIMD),
// each of two lines or more, and at most 48 (the inverse transform adds them).
// Waves wanted 1024, 2048, 4096, 8192: N = 18, 160 cells maxPreserve 1997, 1550, 1376,
// 1253 us an evaluation; N = 10, 75 cells 98, 86, 76, 77; N = 8, 250 cells 48, 43, 42, 46.
extern "C" int spbte_any_slices(int N, int npl, int cfold, int nprod, int ncell) {
  const int tb = any_tb(N, nprod, ncell);
  const long waves = (long)npl * (lane_pad(N) / 64) * ((ncell + tb - 1) / tb);
  const long lines = (cfold ? (N + 1) / 2 : N) * (long)N, most = lines >= 96 ? 48 : (lines >= 4 ? lines / 2 : 1);
  const long want = (4096 + waves - 1) / waves;
  return (int)(want > most ? most : want);
}

extern "C" int spbte_launch_fold_any(const double *W64, void *dst, int N, int npl, int cfold, const spbte_mirror *mr,
                                     hipStream_t s) {
  hipLaunchKernelGGL(k_fold_any, dim3(4096), dim3(256), 0, s, W64, (double *)dst, N, npl, cfold, *mr);
  return (int)hipGetLastError();
}

// csplit > 1 needs Qp with room for csplit * ncell * N^3 double2.
extern "C" int spbte_launch_wsum_any(int N, const spbte_wsum_args *a, const void *Wf, int csplit, void *Qp,
                                     hipStream_t s) {
  if (!spbte_any_supported(N) || csplit < 1 || (csplit > 1 && !Qp)) return (int)hipErrorInvalidValue;
  const int npl = a->npl, cf = a->cfold, tb = any_tb(N, a->nprod, a->ncell);
  switch (N) {
    case 6: launch_np<6, rows_per_lane(6)>(N, npl, cf, tb, a, Wf, csplit, Qp, s); break;
    case 8: launch_np<8, rows_per_lane(8)>(N, npl, cf, tb, a, Wf, csplit, Qp, s); break;
    case 9: launch_np<9, rows_per_lane(9)>(N, npl, cf, tb, a, Wf, csplit, Qp, s); break;
    case 10: launch_np<10, rows_per_lane(10)>(N, npl, cf, tb, a, Wf, csplit, Qp, s); break;
    case 12: launch_np<12, rows_per_lane(12)>(N, npl, cf, tb, a, Wf, csplit, Qp, s); break;
    case 18: launch_np<18, rows_per_lane(18)>(N, npl, cf, tb, a, Wf, csplit, Qp, s); break;
    case 20: launch_np<20, rows_per_lane(20)>(N, npl, cf, tb, a, Wf, csplit, Qp, s); break;
    default:
      if (rows_per_lane(N) == 2) launch_np<0, 2>(N, npl, cf, tb, a, Wf, csplit, Qp, s);
      else launch_np<0, 1>(N, npl, cf, tb, a, Wf, csplit, Qp, s);
      break;
  }
  if (csplit > 1 && !a->keep_slices) return spbte_launch_slice_sum(N, npl, a->ncell, csplit, Qp, a->Qh, s);
  return (int)hipGetLastError();
}
