// k_wsum_any.hip -- folded weighted sum on grids without streaming tiles (FP64).
//
// The sum of k_wsum_stream.hip over the kept rows and columns (see k_fold_w
// there), for any N up to 24: the reference's own N = 8, odd grids, 10, 12, 18,
// 20.  These sums are short (N = 10: 2.8e5 pairs a cell), so what bounds them is
// latency and how much of the chip a batch fills, then LDS: one 16-byte read of F
// per pair, product and cell feeds 4 or 5 FP64 instructions.
//  * A workgroup owns an x-plane of output rows (one row per lane) for TB cells
//    and a slice of the summed x-planes; c is the same in all lanes, so G is read
//    by scalar loads.
//  * Per summed plane the shifted F x-plane of every cell and product is staged
//    in LDS with every z-line twice in a row: the operand of step cz is at a fixed
//    offset -cz from the lane's base and never wraps, and the lanes of a z-line
//    read consecutive 16-byte slots.
//  * W is column-major over the rows of a plane, padded to whole waves: a wave
//    reads 512 contiguous bytes per column, each value feeding TB cells.  With N
//    known at compile time the next z-line's N weights are loaded while one is
//    consumed.
// Measured on an MI355X, the sum alone, against one thread per (row, cell) over the
// whole table (k_wsum_generic, which still serves operands that are not
// transforms of real cells, and N > 24, whose staged planes outgrow LDS):
//   N = 8, 250 cells ComputeQ     209 -> 23 us     N = 12, 300 cells ComputeQ  4631 -> 210 us
//   N = 10, 75 cells maxPreserve  539 -> 49 us     N = 18, 160 cells maxPr.  101.4 -> 3.14 ms
//   N = 10, one cell maxPreserve  355 -> 28 us     N = 20, 120 cells maxPr.  126.4 -> 2.93 ms
// N = 20 and 120 cells is 12.6 TFLOP/s of FP64 (64 measured on FMA chains): two LDS
// reads of 16 bytes for 10 FP64 instructions at 2 cells a weight.
#include <hip/hip_runtime.h>
#include "spbte_internal.h"

namespace {

constexpr int kMaxThreads = 512;

__host__ __device__ inline int row_pad(int N) { return (N * N + 63) / 64 * 64; }
// Summed planes of row plane rx under the column fold: m = (rx + h) mod N, cx + s
// = m (mod N); the kept ones are first, first + 1, ... (count of them), mod N.
__host__ __device__ inline int fold_count(int N, int m) { return N % 2 ? (N + 1) / 2 : N / 2 + 1 - (m & 1); }
__host__ __device__ inline int fold_first(int N, int m) {
  return N % 2 ? ((m & 1) ? (m + N) / 2 : m / 2) : (m + 1) / 2;
}
// Line slot -> cy: from the outermost to the middle (the large terms last).
__host__ __device__ inline int line_cy(int N, int cl) { return (cl & 1) ? N - 1 - cl / 2 : cl / 2; }

// NT: N at compile time, 0: Nrt.
template <int NT, int NP, int TB>
__global__ void __launch_bounds__(kMaxThreads)
k_wsum_any(int Nrt, int npl, int cfold, const double *__restrict__ Wf, const double2 *__restrict__ F0,
           const double2 *__restrict__ G0, const double2 *__restrict__ F1, const double2 *__restrict__ G1,
           double2 *__restrict__ Qh, int ncell, int csplit, int chunks, double2 *__restrict__ Qp) {
  extern __shared__ __attribute__((aligned(16))) char smem_any[];
  double2 *sF = (double2 *)smem_any;  // [p][b][sy][2N]
  const int N = NT ? NT : Nrt, n2 = N * N, h = N / 2, RP = row_pad(N);
  const size_t n3 = (size_t)n2 * N;
  // XCD x takes the x-th contiguous slice of the list with cell groups innermost,
  // so that the workgroups sharing a piece of W share an L2
  const int ncg = (ncell + TB - 1) / TB, total = npl * chunks * csplit * ncg, per = (total + 7) >> 3;
  const int vid = (blockIdx.x & 7) * per + (blockIdx.x >> 3);
  if ((int)(blockIdx.x >> 3) >= per || vid >= total) return;
  const int cg = vid % ncg, r1 = vid / ncg, cs = r1 % csplit, r2 = r1 / csplit, ch = r2 % chunks, rx = r2 / chunks;
  const int m = (rx + h) % N;
  const int ncx = cfold ? fold_count(N, m) : N, first = cfold ? fold_first(N, m) + ncx - 1 : 0;
  const int ncols = (cfold ? N / 2 + 1 : N) * n2;
  const int row = ch * blockDim.x + threadIdx.x;
  const int rc = row < n2 ? row : n2 - 1;
  const int ry = rc / N, rz = rc - ry * N;
  const double *Wr = Wf + (size_t)rx * ncols * RP + (row < RP ? row : RP - 1);
  const double2 *Fp[2] = {F0, F1}, *Gp[2] = {G0, G1};
  size_t cells[TB];
#pragma unroll
  for (int b = 0; b < TB; ++b) cells[b] = (size_t)(cg * TB + b < ncell ? cg * TB + b : ncell - 1) * n3;
  double2 tot[TB];
#pragma unroll
  for (int b = 0; b < TB; ++b) tot[b] = make_double2(0.0, 0.0);

  for (int j = cs * ncx / csplit; j < (cs + 1) * ncx / csplit; ++j) {
    const int cx = cfold ? (first - j) % N : j;
    const int sx = (rx + h - cx + N) % N;
    __syncthreads();
    for (int e = threadIdx.x; e < NP * TB * n2; e += blockDim.x) {
      const int q = e / n2, yz = e - q * n2, y = yz / N, z = yz - y * N;
      const int p = q / TB, b = q - p * TB;
      size_t co = cells[0];
#pragma unroll
      for (int i = 1; i < TB; ++i) co = b == i ? cells[i] : co;
      const double2 v = Fp[p][co + (size_t)sx * n2 + yz];
      sF[(q * N + y) * 2 * N + z] = v;
      sF[(q * N + y) * 2 * N + z + N] = v;
    }
    __syncthreads();
    double2 acc[TB];
#pragma unroll
    for (int b = 0; b < TB; ++b) acc[b] = make_double2(0.0, 0.0);
    const double *Wj = Wr + (size_t)j * n2 * RP;
    const auto step = [&](double w, int cy, int cz, const double2 *line) __attribute__((always_inline)) {
      const size_t c = (size_t)(cx * N + cy) * N + cz;
#pragma unroll
      for (int b = 0; b < TB; ++b) {
        const double2 g0 = Gp[0][cells[b] + c], f0 = line[b * N * 2 * N - cz];
        double pr = g0.x * f0.x, pi = g0.x * f0.y;
        pr = fma(-g0.y, f0.y, pr);
        pi = fma(g0.y, f0.x, pi);
        if constexpr (NP == 2) {
          const double2 g1 = Gp[1][cells[b] + c], f1 = line[(TB + b) * N * 2 * N - cz];
          pr = fma(g1.x, f1.x, pr);
          pi = fma(g1.x, f1.y, pi);
          pr = fma(-g1.y, f1.y, pr);
          pi = fma(g1.y, f1.x, pi);
        }
        acc[b].x = fma(w, pr, acc[b].x);
        acc[b].y = fma(w, pi, acc[b].y);
      }
    };
    if constexpr (NT != 0) {
      double w[NT], wn[NT];
#pragma unroll
      for (int cz = 0; cz < NT; ++cz) wn[cz] = Wj[cz * RP];
      for (int cl = 0; cl < NT; ++cl) {
        const int cy = line_cy(NT, cl);
        int sy = ry + h - cy;
        sy = sy < 0 ? sy + NT : (sy > NT - 1 ? sy - NT : sy);
        const double2 *line = sF + sy * 2 * NT + (rz + h) % NT + NT;
        const int nx = cl + 1 < NT ? cl + 1 : cl;  // the last line again, not past the table
#pragma unroll
        for (int cz = 0; cz < NT; ++cz) {
          w[cz] = wn[cz];
          wn[cz] = Wj[(nx * NT + cz) * RP];
        }
#pragma unroll
        for (int cz = 0; cz < NT; ++cz) step(w[cz], cy, cz, line);
      }
    } else {
      for (int cl = 0; cl < N; ++cl) {
        const int cy = line_cy(N, cl);
        int sy = ry + h - cy;
        sy = sy < 0 ? sy + N : (sy > N - 1 ? sy - N : sy);
        const double2 *line = sF + sy * 2 * N + (rz + h) % N + N;
#pragma unroll 4
        for (int cz = 0; cz < N; ++cz) step(Wj[(cl * N + cz) * RP], cy, cz, line);
      }
    }
#pragma unroll
    for (int b = 0; b < TB; ++b) {
      tot[b].x += acc[b].x;
      tot[b].y += acc[b].y;
    }
  }
  if (row >= n2) return;
#pragma unroll
  for (int b = 0; b < TB; ++b) {
    const int cell = cg * TB + b;
    if (cell >= ncell) continue;
    double2 *o = csplit > 1 ? Qp + ((size_t)cs * ncell + cell) * n3 : Qh + (size_t)cell * n3;
    o[(size_t)rx * n2 + row] = tot[b];
  }
}

// Natural FP64 table -> folded, [rx][column slot][row of the plane, padded].
__global__ void __launch_bounds__(256) k_fold_any(const double *__restrict__ W, double *__restrict__ out, int N, int npl,
                                                  int cfold, spbte_mirror mr) {
  const int n2 = N * N, h = N / 2, RP = row_pad(N), ncp = cfold ? N / 2 + 1 : N;
  const size_t n3 = (size_t)n2 * N, ncols = (size_t)ncp * n2, total = npl * ncols * RP;
  const int a2 = 2 * h;
  for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < total; i += (size_t)gridDim.x * blockDim.x) {
    const int row = (int)(i % RP);
    const size_t q = i / RP;
    const int col = (int)(q % ncols), rx = (int)(q / ncols);
    const int j = col / n2, cl = col / N % N, cz = col % N, cy = line_cy(N, cl);
    const int m = (rx + h) % N, ncx = cfold ? fold_count(N, m) : N;
    double x = 0.0;
    if (row < n2 && j < ncx) {
      const int ry = row / N, rz = row % N;
      const int cx = cfold ? (fold_first(N, m) + ncx - 1 - j) % N : j;
      const int sx = (rx + h - cx + N) % N, sy = (ry + h - cy + N) % N, sz = (rz + h - cz + N) % N;
      const bool pair = cfold && sx != cx;
      const double *Wr = W + ((size_t)rx * n2 + row) * n3;
      x = Wr[((size_t)cx * N + cy) * N + cz];
      if (pair) x += Wr[((size_t)sx * N + sy) * N + sz];
      const int mx = (a2 - rx + N) % N;
      if (mr.on && mx != rx) {
        const int my = (a2 - ry + N) % N, mz = (a2 - rz + N) % N;
        const double *Wm = W + (((size_t)mx * N + my) * N + mz) * n3;
        double y = Wm[((size_t)((a2 - cx + N) % N) * N + (a2 - cy + N) % N) * N + (a2 - cz + N) % N];
        if (pair) y += Wm[((size_t)((a2 - sx + N) % N) * N + (a2 - sy + N) % N) * N + (a2 - sz + N) % N];
        x += mr.r[rx] * mr.r[ry] * mr.r[rz] * mr.s[cx] * mr.s[cy] * mr.s[cz] * mr.s[sx] * mr.s[sy] * mr.s[sz] * y;
      }
    }
    out[i] = x;
  }
}

template <int NT, int NP>
void launch_any(int N, int npl, int cfold, int tb, const spbte_wsum_args *a, const void *Wf, int csplit, void *Qp,
                hipStream_t s) {
  const int RP = row_pad(N), chunks = (RP + kMaxThreads - 1) / kMaxThreads;
  const int T = ((RP / 64 + chunks - 1) / chunks) * 64;
  const size_t lds = (size_t)NP * tb * N * 2 * N * sizeof(double2);
  const int total = npl * chunks * csplit * ((a->ncell + tb - 1) / tb), per = (total + 7) / 8;
  if (tb == 2)
    hipLaunchKernelGGL((k_wsum_any<NT, NP, 2>), dim3(8 * per), dim3(T), lds, s, N, npl, cfold, (const double *)Wf,
                       (const double2 *)a->F0, (const double2 *)a->G0, (const double2 *)a->F1, (const double2 *)a->G1,
                       (double2 *)a->Qh, a->ncell, csplit, chunks, (double2 *)Qp);
  else
    hipLaunchKernelGGL((k_wsum_any<NT, NP, 1>), dim3(8 * per), dim3(T), lds, s, N, npl, cfold, (const double *)Wf,
                       (const double2 *)a->F0, (const double2 *)a->G0, (const double2 *)a->F1, (const double2 *)a->G1,
                       (double2 *)a->Qh, a->ncell, csplit, chunks, (double2 *)Qp);
}

template <int NT>
void launch_np(int N, int npl, int cfold, int tb, const spbte_wsum_args *a, const void *Wf, int csplit, void *Qp,
               hipStream_t s) {
  if (a->nprod == 2) launch_any<NT, 2>(N, npl, cfold, tb, a, Wf, csplit, Qp, s);
  else launch_any<NT, 1>(N, npl, cfold, tb, a, Wf, csplit, Qp, s);
}

// Cells per workgroup: two share each weight where one a workgroup gives two waves
// on every SIMD already (fewer, and the slices that make up for it cost more in
// staging and in the inverse transform's sum) and both cells' planes fit 64 KiB of LDS.
int any_tb(int N, int npl, int nprod, int ncell) {
  const int waves = row_pad(N) / 64;
  return ncell >= 2 && (long)npl * waves * ncell >= 2048 && (size_t)nprod * 2 * N * 2 * N * 16 <= 65536 ? 2 : 1;
}

}  // namespace

extern "C" int spbte_any_supported(int N) { return N >= 2 && N <= 24; }

// Bytes of a folded table.
extern "C" size_t spbte_any_table_bytes(int N, int npl, int cfold) {
  return (size_t)npl * (cfold ? N / 2 + 1 : N) * N * N * row_pad(N) * 8;
}

// Slices of the summed planes: as many as give 4096 waves (4 on every SIMD).
extern "C" int spbte_any_slices(int N, int npl, int cfold, int nprod, int ncell) {
  const int tb = any_tb(N, npl, nprod, ncell);
  const long waves = (long)npl * (row_pad(N) / 64) * ((ncell + tb - 1) / tb);
  const long want = (4096 + waves - 1) / waves, most = cfold ? (N + 1) / 2 : N;
  return (int)(want < 1 ? 1 : (want > most ? most : want));
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
  const int npl = a->npl, cf = a->cfold, tb = any_tb(N, npl, a->nprod, a->ncell);
  switch (N) {
    case 6: launch_np<6>(N, npl, cf, tb, a, Wf, csplit, Qp, s); break;
    case 8: launch_np<8>(N, npl, cf, tb, a, Wf, csplit, Qp, s); break;
    case 9: launch_np<9>(N, npl, cf, tb, a, Wf, csplit, Qp, s); break;
    case 10: launch_np<10>(N, npl, cf, tb, a, Wf, csplit, Qp, s); break;
    case 12: launch_np<12>(N, npl, cf, tb, a, Wf, csplit, Qp, s); break;
    case 18: launch_np<18>(N, npl, cf, tb, a, Wf, csplit, Qp, s); break;
    case 20: launch_np<20>(N, npl, cf, tb, a, Wf, csplit, Qp, s); break;
    default: launch_np<0>(N, npl, cf, tb, a, Wf, csplit, Qp, s); break;
  }
  if (csplit > 1 && !a->keep_slices) return spbte_launch_slice_sum(N, a->ncell, csplit, Qp, a->Qh, s);
  return (int)hipGetLastError();
}
