// Image-level kernels of the subset-correlation library and the dispatch of
// the correlation passes (the solver kernels live in dice_k_*.hip).
#include "dice_device.h"

#include <algorithm>

namespace dice_hip {

typedef hipError_t (*PassLauncher)(int, int, int, const Launch &, const KParams &, const DImage &, const DImage &,
                                   const DSubsets &, double *, const PassArgs &, hipStream_t);
hipError_t launch_gn_plain(int, int, int, const Launch &, const KParams &, const DImage &, const DImage &,
                           const DSubsets &, double *, const PassArgs &, hipStream_t);
hipError_t launch_gn_batched(int, int, int, const Launch &, const KParams &, const DImage &, const DImage &,
                             const DSubsets &, double *, const PassArgs &, hipStream_t);
hipError_t launch_simplex_plain(int, int, int, const Launch &, const KParams &, const DImage &, const DImage &,
                                const DSubsets &, double *, const PassArgs &, hipStream_t);
hipError_t launch_gn_lean(int, int, const Launch &, const KParams &, const DImage &, const DImage &, const DSubsets &,
                          double *, const PassArgs &, hipStream_t);
hipError_t launch_simplex_batched(int, int, int, const Launch &, const KParams &, const DImage &, const DImage &,
                                  const DSubsets &, double *, const PassArgs &, hipStream_t);
hipError_t launch_gn_trans(int, int, const Launch &, const KParams &, const DImage &, const DImage &, const DSubsets &,
                           double *, const PassArgs &, hipStream_t);
hipError_t launch_gn_crew(int, int, int, const Launch &, const KParams &, const DImage &, const DImage &,
                          const DSubsets &, double *, const PassArgs &, hipStream_t);
hipError_t launch_gn_wide(int, int, const Launch &, const KParams &, const DImage &, const DImage &, const DSubsets &,
                          double *, const PassArgs &, hipStream_t);
hipError_t launch_simplex_wide(int, int, const Launch &, const KParams &, const DImage &, const DImage &,
                               const DSubsets &, double *, const PassArgs &, hipStream_t);

namespace {
using dev::ldpix;

// FD gradients (Image_::compute_gradients_finite_difference, DICe_Image.cpp:1064-1094):
// 4th-order central differences, first-order one-sided within 2 px of the edge.
template <typename T>
__global__ void gradients_kernel(const void *pix, int w, int h, float *gx, float *gy) {
  const int x = blockIdx.x * blockDim.x + threadIdx.x;
  const int y = blockIdx.y * blockDim.y + threadIdx.y;
  if (x >= w || y >= h) return;
  const int o = y * w + x;
  const float c1 = 1.0f / 12.0f, c2 = -8.0f / 12.0f;
  float vx, vy;
  if (x < 2) vx = ldpix<T>(pix, o + 1) - ldpix<T>(pix, o);
  else if (x >= w - 2) vx = ldpix<T>(pix, o) - ldpix<T>(pix, o - 1);
  else vx = c1 * ldpix<T>(pix, o - 2) + c2 * ldpix<T>(pix, o - 1) - c2 * ldpix<T>(pix, o + 1) - c1 * ldpix<T>(pix, o + 2);
  if (y < 2) vy = ldpix<T>(pix, o + w) - ldpix<T>(pix, o);
  else if (y >= h - 2) vy = ldpix<T>(pix, o) - ldpix<T>(pix, o - w);
  else vy = c1 * ldpix<T>(pix, o - 2 * w) + c2 * ldpix<T>(pix, o - w) - c2 * ldpix<T>(pix, o + w) - c1 * ldpix<T>(pix, o + 2 * w);
  gx[o] = vx;
  gy[o] = vy;
}

// 5x5 binomial smoothing of the gradients (DICe_Image.cpp:1032-1062), interior only.
__global__ void smooth_kernel(const float *inx, const float *iny, int w, int h, float *gx, float *gy) {
  const int x = blockIdx.x * blockDim.x + threadIdx.x;
  const int y = blockIdx.y * blockDim.y + threadIdx.y;
  if (x >= w || y >= h) return;
  const int o = y * w + x;
  if (x < 2 || x >= w - 2 || y < 2 || y >= h - 2) { gx[o] = inx[o]; gy[o] = iny[o]; return; }
  const float k1[5] = {0.0625f, 0.25f, 0.375f, 0.25f, 0.0625f};
  float vx = 0.0f, vy = 0.0f;
  for (int i = 0; i < 5; ++i)
    for (int j = 0; j < 5; ++j) {
      const float c = k1[i] * k1[j];
      vx += c * inx[o + (i - 2) * w + (j - 2)];
      vy += c * iny[o + (i - 2) * w + (j - 2)];
    }
  gx[o] = vx;
  gy[o] = vy;
}

// Gauss filter masks of Image_::gauss_filter (DICe_Image.cpp:54-126, 1194-1240).
// The 2-D masks are the outer products c_i c_j of these 1-D factors (listed
// from the edge to the centre; the 5-point one sums to 0.9458, so its mask is
// not normalised).  gauss_coefficients forms each product in float from the
// float factors: that reproduces the reference's filtered-image goldens
// (tests/component/images/outFilter*.rawi) bit for bit, where its source
// tables, the same products written to nine digits, move a few pixels by an
// ulp.
static const double kGauss5[3] = {0.0014, 0.1574, 0.62825};
static const double kGauss7[4] = {0.006, 0.0606, 0.2418, 0.3831};
static const double kGauss9[5] = {0.0007, 0.0108, 0.0748, 0.2384, 0.3505};
static const double kGauss11[6] = {0.0001, 0.0017, 0.0168, 0.087, 0.2328, 0.3231};
static const double kGauss13[7] = {0.0001, 0.0012, 0.0085, 0.038, 0.1109, 0.2108, 0.2611};

constexpr int kGfMaxMask = 13;
struct GaussCoef {
  float c[kGfMaxMask * kGfMaxMask];  // c[i * M + j]: i the x offset, j the y offset
};

static bool gauss_coefficients(int M, GaussCoef &g) {
  const double *f = M == 5 ? kGauss5 : M == 7 ? kGauss7 : M == 9 ? kGauss9 : M == 11 ? kGauss11 : M == 13 ? kGauss13 : nullptr;
  if (!f) return false;
  for (int i = 0; i < M; ++i)
    for (int j = 0; j < M; ++j)
      g.c[i * M + j] = (float)f[i <= M / 2 ? i : M - 1 - i] * (float)f[j <= M / 2 ? j : M - 1 - j];
  return true;
}

// One 32 x 32 output tile per 32 x 8 block, each thread four rows; the tile
// and its halo are staged in LDS (reads clamped to the image: clamped values
// only reach the copied border band).  Pixels at least M / 2 + 1 from every
// edge get sum_i sum_j c_ij I(x + i - M/2, y + j - M/2), accumulated in float
// with a separate multiply and add per tap (no fused multiply-add) in the
// reference's order, x offset outer; the others are copied.
constexpr int kGfTile = 32;
template <typename T, int M>
__global__ __launch_bounds__(256) void gauss_filter_kernel(const void *in, void *out, int w, int h, GaussCoef g) {
#pragma clang fp contract(off)
  constexpr int R = M / 2, P = kGfTile + 2 * R;
  __shared__ float tile[P * P];
  const T *src = (const T *)in;
  T *dst = (T *)out;
  const int tx = threadIdx.x, ty = threadIdx.y, tid = ty * 32 + tx;
  const int x0 = blockIdx.x * kGfTile, y0 = blockIdx.y * kGfTile;
  for (int k = tid; k < P * P; k += 256) {
    const int ly = k / P, lx = k - ly * P;
    const int gx = min(max(x0 + lx - R, 0), w - 1), gy = min(max(y0 + ly - R, 0), h - 1);
    tile[k] = (float)src[(size_t)gy * w + gx];
  }
  __syncthreads();
  const int hm = R + 1;  // gauss_filter_half_mask_
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int lx = tx, ly = ty + 8 * r;
    const int x = x0 + lx, y = y0 + ly;
    if (x >= w || y >= h) continue;
    const size_t o = (size_t)y * w + x;
    if (x >= hm && x < w - hm && y >= hm && y < h - hm) {
      float value = 0.0f;
#pragma unroll
      for (int i = 0; i < M; ++i)
#pragma unroll
        for (int j = 0; j < M; ++j) value += g.c[i * M + j] * tile[(ly + j) * P + lx + i];
      // cast to the storage type as the reference does (truncating for uint16; the
      // 13-point mask sums to 1.0002, so a saturated 16-bit pixel is clamped)
      if constexpr (std::is_same<T, float>::value) dst[o] = value;
      else dst[o] = (T)fminf(value, 65535.0f);
    } else {
      dst[o] = src[o];
    }
  }
}

template <typename T>
hipError_t launch_gauss_t(const void *in, void *out, int w, int h, int mask, hipStream_t stream) {
  GaussCoef g;
  if (!gauss_coefficients(mask, g)) return hipErrorInvalidValue;
  const dim3 block(32, 8), grid((w + kGfTile - 1) / kGfTile, (h + kGfTile - 1) / kGfTile);
  switch (mask) {
    case 5: hipLaunchKernelGGL((gauss_filter_kernel<T, 5>), grid, block, 0, stream, in, out, w, h, g); break;
    case 7: hipLaunchKernelGGL((gauss_filter_kernel<T, 7>), grid, block, 0, stream, in, out, w, h, g); break;
    case 9: hipLaunchKernelGGL((gauss_filter_kernel<T, 9>), grid, block, 0, stream, in, out, w, h, g); break;
    case 11: hipLaunchKernelGGL((gauss_filter_kernel<T, 11>), grid, block, 0, stream, in, out, w, h, g); break;
    case 13: hipLaunchKernelGGL((gauss_filter_kernel<T, 13>), grid, block, 0, stream, in, out, w, h, g); break;
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

__global__ void zero_ints_kernel(int *p, int count) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < count) p[i] = 0;
}

__global__ void copy_doubles_kernel(double *dst, const double *src, size_t count) {
  for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < count; i += (size_t)gridDim.x * blockDim.x)
    dst[i] = src[i];
}

// One subset per thread: gather the initial guess of subset i from its
// neighbour's fields (see launch_neighbor_guess).
__global__ void neighbor_guess_kernel(const double *start, const double *cur, double *guess, const double *prev,
                                      double tol, int *list, int *count, int n) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const int nb = (int)start[(size_t)F_NEIGHBOR_ID * n + i];
  const bool self = nb < 0 || nb == i;  // the host has checked nb < n
  const int j = self ? i : nb;
  const double *src = (!self && nb < i) ? cur : start;
  const int slots[7] = {F_DISP_X, F_DISP_Y, F_ROT_Z, F_NS_XX, F_NS_YY, F_SS_XY, F_SIGMA};
  double g[kGuessSlots];
#pragma unroll
  for (int k = 0; k < 7; ++k) g[k] = src[(size_t)slots[k] * n + j];
  g[7] = self ? 1.0 : 3.0;  // INITIALIZE_USING_PREVIOUS_FRAME / _NEIGHBOR_VALUE_SUCCESSFUL
  bool redo = prev == nullptr;
  if (!redo) {
#pragma unroll
    for (int k = 0; k < 6; ++k) redo |= tol > 0.0 ? fabs(g[k] - prev[(size_t)k * n + i]) > tol : g[k] != prev[(size_t)k * n + i];
    const double ps = prev[(size_t)6 * n + i];
    redo |= tol > 0.0 ? (g[6] == -1.0) != (ps == -1.0) : g[6] != ps;
    redo |= g[7] != prev[(size_t)7 * n + i];
  }
#pragma unroll
  for (int k = 0; k < kGuessSlots; ++k) guess[(size_t)k * n + i] = redo ? g[k] : prev[(size_t)k * n + i];
  if (redo) list[atomicAdd(count, 1)] = i;
}

__global__ void reset_listed_kernel(const int *list, const int *count, const double *start, double *fields, int n) {
  const int k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= *count) return;
  const int i = list[k];
#pragma unroll
  for (int s = 0; s < kNumFields; ++s) fields[(size_t)s * n + i] = start[(size_t)s * n + i];
}

// 3 x 3 LU with partial pivoting and the inverse from its factors, in double
// (GETRF + GETRI).  Returns false if a pivot is zero.
__device__ bool inverse3(const double (&a_in)[3][3], double (&inv)[3][3]) {
  double a[3][3];
  int piv[3] = {0, 1, 2};
  for (int i = 0; i < 3; ++i)
    for (int j = 0; j < 3; ++j) a[i][j] = a_in[i][j];
  for (int k = 0; k < 3; ++k) {
    int p = k;
    for (int i = k + 1; i < 3; ++i)
      if (fabs(a[i][k]) > fabs(a[p][k])) p = i;
    if (a[p][k] == 0.0) return false;
    if (p != k) {
      for (int j = 0; j < 3; ++j) {
        const double t = a[k][j];
        a[k][j] = a[p][j];
        a[p][j] = t;
      }
      const int t = piv[k];
      piv[k] = piv[p];
      piv[p] = t;
    }
    for (int i = k + 1; i < 3; ++i) {
      a[i][k] /= a[k][k];
      for (int j = k + 1; j < 3; ++j) a[i][j] -= a[i][k] * a[k][j];
    }
  }
  // solve L U x = P e_c for each column c
  for (int c = 0; c < 3; ++c) {
    double x[3];
    for (int i = 0; i < 3; ++i) {
      double v = piv[i] == c ? 1.0 : 0.0;
      for (int j = 0; j < i; ++j) v -= a[i][j] * x[j];
      x[i] = v;
    }
    for (int i = 2; i >= 0; --i) {
      double v = x[i];
      for (int j = i + 1; j < 3; ++j) v -= a[i][j] * x[j];
      x[i] = v / a[i][i];
    }
    for (int i = 0; i < 3; ++i) inv[i][c] = x[i];
  }
  return true;
}

__device__ double norm1_3(const double (&a)[3][3]) {
  double m = 0.0;
  for (int j = 0; j < 3; ++j) {
    const double c = fabs(a[0][j]) + fabs(a[1][j]) + fabs(a[2][j]);
    m = c > m ? c : m;
  }
  return m;
}

// Bounds of the subset centres for the VSG grid, in two launches: each of up
// to kVsgBoundBlocks workgroups reduces a grid-stride share into 5 partials
// (min x, min y, max x, max y over the finite centres, count of non-finite
// ones), then one workgroup folds the partials into out[0..4].
constexpr int kVsgBoundBlocks = 256;

__device__ void vsg_bounds_fold(double (&red)[5][256], double x0, double y0, double x1, double y1, double bad,
                                double *out) {
  const int t = threadIdx.x;
  red[0][t] = x0;
  red[1][t] = y0;
  red[2][t] = x1;
  red[3][t] = y1;
  red[4][t] = bad;
  __syncthreads();
  for (int s = 128; s > 0; s >>= 1) {
    if (t < s) {
      red[0][t] = fmin(red[0][t], red[0][t + s]);
      red[1][t] = fmin(red[1][t], red[1][t + s]);
      red[2][t] = fmax(red[2][t], red[2][t + s]);
      red[3][t] = fmax(red[3][t], red[3][t + s]);
      red[4][t] += red[4][t + s];
    }
    __syncthreads();
  }
  if (t < 5) out[t] = red[t][0];
}

__global__ __launch_bounds__(256) void vsg_bounds_partial_kernel(const double *fields, int n, double *partial) {
  __shared__ double red[5][256];
  const double *X = fields + (size_t)F_COORD_X * n, *Y = fields + (size_t)F_COORD_Y * n;
  double x0 = INFINITY, y0 = INFINITY, x1 = -INFINITY, y1 = -INFINITY, bad = 0.0;
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
    const double x = X[i], y = Y[i];
    if (!isfinite(x) || !isfinite(y)) {
      bad += 1.0;
      continue;
    }
    x0 = fmin(x0, x);
    y0 = fmin(y0, y);
    x1 = fmax(x1, x);
    y1 = fmax(y1, y);
  }
  vsg_bounds_fold(red, x0, y0, x1, y1, bad, partial + 5 * blockIdx.x);
}

__global__ __launch_bounds__(256) void vsg_bounds_final_kernel(const double *partial, int blocks, double *out) {
  __shared__ double red[5][256];
  const int t = threadIdx.x;
  double x0 = INFINITY, y0 = INFINITY, x1 = -INFINITY, y1 = -INFINITY, bad = 0.0;
  if (t < blocks) {
    const double *q = partial + 5 * t;
    x0 = q[0];
    y0 = q[1];
    x1 = q[2];
    y1 = q[3];
    bad = q[4];
  }
  vsg_bounds_fold(red, x0, y0, x1, y1, bad, out);
}

// The cell-ordered list by counting: every subset's cell and its turn to arrive
// there (an atomic per subset), the cells' first entries by a scan of the counts,
// the ids at those places, and last each entry's rank by id among its cell's, so
// that ids ascend within a cell whatever the order of arrival.  That rank reads
// the entries of one cell per entry, never more than the strain's own scan of a
// valid subset does after it.  Five launches of a few us: 155,236 subsets in 18,225 cells 27 us, a
// library radix sort of (cell, id) and the cells' ranges from it 72 us.
//
// Cell of subset i (the same arithmetic as vsg_subset's own cell).
__global__ void vsg_cells_kernel(const double *fields, int n, VsgGrid g, int *count, int *cells, int *turn) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const double xi = fields[(size_t)F_COORD_X * n + i], yi = fields[(size_t)F_COORD_Y * n + i];
  const int ci = min(max((int)floor((xi - g.x0) / g.cell), 0), g.ncx - 1);
  const int cj = min(max((int)floor((yi - g.y0) / g.cell), 0), g.ncy - 1);
  const int c = cj * g.ncx + ci;
  cells[i] = c;
  turn[i] = atomicAdd(count + c, 1);
}

// Exclusive scan of the counts in two launches: the sum of each group of
// kVsgScan cells, then each workgroup adds up the groups before its own and
// scans its cells.  start[ncells] = n.
constexpr int kVsgScan = 1024;
__device__ int vsg_block_sum(int v, int *red) {  // over 256 threads; every thread gets it
  for (int o = 32; o >= 1; o >>= 1) v += __shfl_xor(v, o);
  __syncthreads();
  if (threadIdx.x % 64 == 0) red[threadIdx.x / 64] = v;
  __syncthreads();
  return (red[0] + red[1]) + (red[2] + red[3]);
}
__global__ __launch_bounds__(256) void vsg_sums_kernel(const int *count, int ncells, int *sums) {
  __shared__ int red[4];
  int v = 0;
  for (int t = 0; t < kVsgScan / 256; ++t) {
    const int c = blockIdx.x * kVsgScan + t * 256 + threadIdx.x;
    if (c < ncells) v += count[c];
  }
  v = vsg_block_sum(v, red);
  if (threadIdx.x == 0) sums[blockIdx.x] = v;
}
__global__ __launch_bounds__(256) void vsg_starts_kernel(const int *count, int ncells, int n, const int *sums,
                                                         int *start) {
  __shared__ int red[4];
  __shared__ int scan[256];
  int before = 0;
  for (int t = threadIdx.x; t < (int)blockIdx.x; t += 256) before += sums[t];
  before = vsg_block_sum(before, red);
  // four consecutive cells per thread
  const int c0 = blockIdx.x * kVsgScan + threadIdx.x * 4;
  int v[4], own = 0;
  for (int k = 0; k < 4; ++k) {
    v[k] = c0 + k < ncells ? count[c0 + k] : 0;
    own += v[k];
  }
  scan[threadIdx.x] = own;
  __syncthreads();
  for (int o = 1; o < 256; o <<= 1) {
    const int add = (int)threadIdx.x >= o ? scan[threadIdx.x - o] : 0;
    __syncthreads();
    scan[threadIdx.x] += add;
    __syncthreads();
  }
  int at = before + scan[threadIdx.x] - own;
  for (int k = 0; k < 4; ++k) {
    if (c0 + k < ncells) start[c0 + k] = at;
    at += v[k];
  }
  if (blockIdx.x == 0 && threadIdx.x == 0) start[ncells] = n;
}
__global__ void vsg_place_kernel(const int *cells, const int *turn, const int *start, int n, int *arrived) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) arrived[start[cells[i]] + turn[i]] = i;
}

// Entry of subset i in the cell-ordered list: its cell, its id, ~id when it
// failed (SIGMA < 0), and its centre and displacement as float (the precision
// the strain uses).  hide: the centre of a failed subset as NaN, which fails
// every distance test, so that a radius scan reads one 16-byte record per
// candidate and nothing else.
__global__ void vsg_pack_kernel(const double *fields, const int *cells, const int *start, const int *arrived, int n,
                                int hide, int *keys, int *ids, float4 *rec) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const int c = cells[i];
  const int lo = start[c], hi = start[c + 1];
  int k = lo;
  // (eight loads in flight: a crowded cell is read at its latency otherwise)
#pragma unroll 8
  for (int t = lo; t < hi; ++t) k += arrived[t] < i ? 1 : 0;
  auto F = [&](int s) { return fields[(size_t)s * n + i]; };
  const bool failed = !(F(F_SIGMA) >= 0.0);
  const float x = failed && hide ? __int_as_float(0x7fc00000) : (float)F(F_COORD_X);
  rec[k] = make_float4(x, (float)F(F_COORD_Y), (float)F(F_DISP_X), (float)F(F_DISP_Y));
  keys[k] = c;
  ids[k] = failed ? ~i : i;
}

// Candidate records of the radius scan: straight from the cell-ordered list,
// or from a workgroup's LDS copy of the ranges it needs, one per cell row.
constexpr int kVsgMaxRows = 2 * kVsgRings + 1;
struct VsgGlobalReader {
  const float4 *rec;
  __device__ const float4 *row(int) const { return rec; }
};
struct VsgTileReader {
  const float4 *rec;  // LDS
  const int *shift;   // LDS: where entry 0 would be, per row
  int row0;           // cell row of range 0
  __device__ const float4 *row(int cy) const { return rec + shift[cy - row0]; }
};

// Strain of subset i (see launch_vsg_strain); radius candidates through R.
// L lanes of one wave per subset (L = 1, 2, 4, ...; lane `part` of them): the
// radius scan deals the cell rows out round-robin, or the candidates of a row
// when there are fewer than about five rows (8,000 subsets in 60 x 60 px and three far
// away, window 61: 1.10 ms by rows, 0.52 ms by candidates), and the lanes' sums
// are folded by butterfly shuffles; part 0 finishes.  Every lane of a group must
// reach the fold.  The candidates of a cell row are the cells within the circle's extent
// there (plus g.slack for the rounding of the float distances): with cells of
// a quarter of the radius three in four lie in the circle, against one in three
// of the 3 x 3 cells of the radius.  The kernel is bound by the 11 FP64 sums per
// neighbour and the LDS reads; 155,236 subsets at a step of 5 px, a window of
// 121 px (460 neighbours each): 236 us with cells of the radius, 147 us with these.
template <int L, class Reader>
__device__ void vsg_subset(const VsgGrid &g, float radius, int knn, double *fields, double *vsg, int n, int i,
                           int part, const Reader &R) {
  auto F = [&](int s, int k) -> double & { return fields[(size_t)s * n + k]; };
  const double xi = F(F_COORD_X, i), yi = F(F_COORD_Y, i);
  const float xf = (float)xi, yf = (float)yi;
  const float r2 = radius * radius + 1.0e-5f;  // the reference's rad^2 + tiny in scalar_t
  double sx = 0, sy = 0, sxx = 0, sxy = 0, syy = 0, su = 0, sxu = 0, syu = 0, sv = 0, sxv = 0, syv = 0;
  int valid = 0;
  // the reference keeps the neighbour offsets and the displacements as scalar_t (float)
  auto add = [&](float uf, float vf, float ddx, float ddy) {
    const double dx = ddx, dy = ddy;
    const double u = uf, v = vf;
    ++valid;
    sx += dx; sy += dy;
    sxx += dx * dx; sxy += dx * dy; syy += dy * dy;
    su += u; sxu += dx * u; syu += dy * u;
    sv += v; sxv += dx * v; syv += dy * v;
  };
  const int ci = min(max((int)floor((xi - g.x0) / g.cell), 0), g.ncx - 1);
  const int cj = min(max((int)floor((yi - g.y0) / g.cell), 0), g.ncy - 1);
  if (F(F_SIGMA, i) >= 0.0 && knn == 0) {
    const double rr = sqrt((double)r2) + g.slack;
    const bool rows = 2.0 * g.cell <= (double)radius;  // (the same in every lane)
    const int rings = rows ? kVsgRings : min(kVsgRings, (int)(rr / g.cell) + 1);
    const int row0 = rows ? part : 0, row_step = rows ? L : 1, first = rows ? 0 : part, step = rows ? 1 : L;
    for (int cy = cj - rings + row0; cy <= min(cj + rings, g.ncy - 1); cy += row_step) {
      if (cy < 0) continue;
      const double ya = g.y0 + cy * g.cell, yb = ya + g.cell;
      const double away = fmax(fmax(ya - yi, yi - yb) - g.slack, 0.0);
      if (away > rr) continue;
      const double half = sqrt(rr * rr - away * away) + g.slack;
      const int ca = min(max((int)floor((xi - half - g.x0) / g.cell), 0), g.ncx - 1);
      const int cb = min(max((int)floor((xi + half - g.x0) / g.cell), 0), g.ncx - 1);
      const float4 *q = R.row(cy);
      const int e = g.cell_begin[cy * g.ncx + cb + 1];
      for (int k = g.cell_begin[cy * g.ncx + ca] + first; k < e; k += step) {
        const float4 c = q[k];
        const float ddx = c.x - xf, ddy = c.y - yf;
        if (ddx * ddx + ddy * ddy < r2) add(c.z, c.w, ddx, ddy);
      }
    }
  } else if (F(F_SIGMA, i) >= 0.0) {
    // the knn nearest subsets (this one included) by squared float distance, then id: rings of
    // cells around this one until no unvisited cell can hold a closer subset
    float bd[kVsgMaxK];
    int bj[kVsgMaxK];
    int have = 0;
    const int rings = max(g.ncx, g.ncy);
    for (int r = 0; r <= rings; ++r) {
      for (int cy = cj - r; cy <= cj + r; ++cy) {
        if (cy < 0 || cy >= g.ncy) continue;
        const int step = (cy == cj - r || cy == cj + r) ? 1 : 2 * r;
        for (int cx = ci - r; cx <= ci + r; cx += max(step, 1)) {
          if (cx < 0 || cx >= g.ncx) continue;
          const int c = cy * g.ncx + cx;
          for (int k = g.cell_begin[c]; k < g.cell_begin[c + 1]; ++k) {
            const int j = g.cell_ids[k] < 0 ? ~g.cell_ids[k] : g.cell_ids[k];
            const float4 q = g.rec[k];
            const float ddx = q.x - xf, ddy = q.y - yf;
            const float d2 = ddx * ddx + ddy * ddy;
            if (have == knn && !(d2 < bd[knn - 1] || (d2 == bd[knn - 1] && j < bj[knn - 1]))) continue;
            int pos = have < knn ? have++ : knn - 1;
            while (pos > 0 && (d2 < bd[pos - 1] || (d2 == bd[pos - 1] && j < bj[pos - 1]))) {
              bd[pos] = bd[pos - 1];
              bj[pos] = bj[pos - 1];
              --pos;
            }
            bd[pos] = d2;
            bj[pos] = j;
          }
        }
      }
      const float reach = (float)(r * g.cell);
      if (have == knn && bd[knn - 1] < reach * reach) break;
    }
    if (have > 0 && !(F(F_SIGMA, bj[0]) >= 0.0)) have = 0;  // the nearest must be valid
    for (int k = 0; k < have; ++k) {
      const int j = bj[k];
      if (F(F_SIGMA, j) >= 0.0)
        add((float)F(F_DISP_X, j), (float)F(F_DISP_Y, j), (float)F(F_COORD_X, j) - xf, (float)F(F_COORD_Y, j) - yf);
    }
  }
  if constexpr (L > 1) {
    auto fold = [](double &v) {
#pragma unroll
      for (int o = L / 2; o >= 1; o >>= 1) v += __shfl_xor(v, o);
    };
    fold(sx); fold(sy); fold(sxx); fold(sxy); fold(syy);
    fold(su); fold(sxu); fold(syu); fold(sv); fold(sxv); fold(syv);
#pragma unroll
    for (int o = L / 2; o >= 1; o >>= 1) valid += __shfl_xor(valid, o);
    if (part != 0) return;
  }
  double out[kVsgFields] = {0, 0, 0, 0, 0, 0, 0};
  bool ok = valid >= 3;
  if (ok) {
    const double s1 = valid;
    const double a[3][3] = {{s1, sx, sy}, {sx, sxx, sxy}, {sy, sxy, syy}};
    double inv[3][3];
    ok = inverse3(a, inv);
    // the reciprocal 1-norm condition number (the reference estimates it with GECON)
    if (ok) ok = 1.0 / (norm1_3(a) * norm1_3(inv)) >= 1.0e-12;
    if (ok) {
      const double bu[3] = {su, sxu, syu}, bv[3] = {sv, sxv, syv};
      double cu[3] = {0, 0, 0}, cv[3] = {0, 0, 0};
      for (int r = 0; r < 3; ++r)
        for (int c = 0; c < 3; ++c) {
          cu[r] += inv[r][c] * bu[c];
          cv[r] += inv[r][c] * bv[c];
        }
      const double dudx = cu[1], dudy = cu[2], dvdx = cv[1], dvdy = cv[2];
      out[0] = (float)(0.5 * (2.0 * dudx + dudx * dudx + dvdx * dvdx));
      out[1] = (float)(0.5 * (2.0 * dvdy + dudy * dudy + dvdy * dvdy));
      out[2] = (float)(0.5 * (dudy + dvdx + dudx * dudy + dvdx * dvdy));
      out[3] = (float)dudx;  // stored in scalar_t fields
      out[4] = (float)dudy;
      out[5] = (float)dvdx;
      out[6] = (float)dvdy;
    }
  }
  for (int k = 0; k < kVsgFields; ++k) vsg[(size_t)k * n + i] = out[k];
  if (!ok) F(F_MATCH, i) = -1.0;
}

// k-nearest windows: one subset per thread, in subset order.
__global__ void vsg_strain_kernel(VsgGrid g, float radius, int knn, double *fields, double *vsg, int n) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  vsg_subset<1>(g, radius, knn, fields, vsg, n, i, 0, VsgGlobalReader{g.rec});
}

// Radius windows: kVsgLanes lanes per subset; workgroup b takes entries
// [64 b, 64 b + 64) of the cell-ordered list.  When they lie in one row of cells,
// the candidates they need lie in one contiguous range of the list per cell row
// (from kVsgRings columns left of the first cell to kVsgRings right of the last),
// which the workgroup copies to LDS once; otherwise, or when the ranges exceed
// kVsgTileEntries, its threads read the list directly.  Both give the same
// sums in the same order.
constexpr int kVsgTileEntries = 2048;
constexpr int kVsgLanes = 4;
constexpr int kVsgGroupSubsets = 256 / kVsgLanes;
__global__ __launch_bounds__(256) void vsg_strain_tiled_kernel(VsgGrid g, float radius, double *fields, double *vsg,
                                                               int n) {
  __shared__ float4 srec[kVsgTileEntries];
  __shared__ int lo[kVsgMaxRows], len[kVsgMaxRows], shift[kVsgMaxRows];
  __shared__ int total;
  const int k0 = blockIdx.x * kVsgGroupSubsets;
  const int k1 = min(k0 + kVsgGroupSubsets, n);
  const int cfirst = g.cell_keys[k0], clast = g.cell_keys[k1 - 1];
  const int cj = cfirst / g.ncx;
  bool tiled = false;
  if (clast / g.ncx == cj) {  // uniform over the workgroup
    if (threadIdx.x < kVsgMaxRows) {
      const int r = (int)threadIdx.x, cy = cj - kVsgRings + r;
      int a = 0, b = 0;
      if (cy >= 0 && cy < g.ncy) {
        a = g.cell_begin[cy * g.ncx + max(cfirst - cj * g.ncx - kVsgRings, 0)];
        b = g.cell_begin[cy * g.ncx + min(clast - cj * g.ncx + kVsgRings, g.ncx - 1) + 1];
      }
      lo[r] = a;
      len[r] = b - a;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
      int off = 0;
      for (int r = 0; r < kVsgMaxRows; ++r) {
        shift[r] = off - lo[r];
        off += len[r];
      }
      total = off;
    }
    __syncthreads();
    tiled = total <= kVsgTileEntries;
    if (tiled)
      for (int r = 0; r < kVsgMaxRows; ++r)
        for (int t = threadIdx.x; t < len[r]; t += blockDim.x) srec[shift[r] + lo[r] + t] = g.rec[lo[r] + t];
    __syncthreads();
  }
  const int k = k0 + (int)threadIdx.x / kVsgLanes, part = (int)threadIdx.x % kVsgLanes;
  if (k >= n) return;  // whole groups of lanes
  const int e = g.cell_ids[k];
  const int i = e < 0 ? ~e : e;
  if (tiled)
    vsg_subset<kVsgLanes>(g, radius, 0, fields, vsg, n, i, part, VsgTileReader{srec, shift, cj - kVsgRings});
  else
    vsg_subset<kVsgLanes>(g, radius, 0, fields, vsg, n, i, part, VsgGlobalReader{g.rec});
}

__global__ void uncertainty_kernel(const double *fields, double *out, int n) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const float angle = (float)fields[(size_t)F_FIELD_1 * n + i];
  const float sig = (float)fields[(size_t)F_SIGMA * n + i];
  // 1.0 / angle * sig with the double literal of the reference, stored as scalar_t
  out[i] = sig < 0.0f ? 0.0f : angle == 0.0f ? 0.0f : (float)(1.0 / (double)angle * (double)sig);
  out[(size_t)n + i] = angle;
}

}  // namespace

hipError_t launch_uncertainty(const double *fields, double *out, int n, hipStream_t stream) {
  if (n <= 0) return hipSuccess;
  hipLaunchKernelGGL(uncertainty_kernel, dim3((n + 255) / 256), dim3(256), 0, stream, fields, out, n);
  return hipGetLastError();
}

hipError_t launch_vsg_bounds(const double *fields, int n, double *bounds, hipStream_t stream) {
  if (n <= 0) return hipErrorInvalidValue;
  // bounds holds 5 results, then 5 partials per workgroup
  const int blocks = std::min(kVsgBoundBlocks, (n + 255) / 256);
  hipLaunchKernelGGL(vsg_bounds_partial_kernel, dim3(blocks), dim3(256), 0, stream, fields, n, bounds + 5);
  hipLaunchKernelGGL(vsg_bounds_final_kernel, dim3(1), dim3(256), 0, stream, bounds + 5, blocks, bounds);
  return hipGetLastError();
}

hipError_t launch_vsg_grid(const double *fields, int n, bool radius_window, VsgGrid &g, const VsgWork &w,
                           hipStream_t stream) {
  if (n <= 0) return hipErrorInvalidValue;
  const int ncells = g.ncx * g.ncy, groups = (ncells + kVsgScan - 1) / kVsgScan;
  const dim3 per_subset((n + 255) / 256), block(256);
  hipError_t e = launch_zero_ints(w.count, ncells, stream);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(vsg_cells_kernel, per_subset, block, 0, stream, fields, n, g, w.count, w.cells, w.turn);
  hipLaunchKernelGGL(vsg_sums_kernel, dim3(groups), block, 0, stream, w.count, ncells, w.sums);
  hipLaunchKernelGGL(vsg_starts_kernel, dim3(groups), block, 0, stream, w.count, ncells, n, w.sums, w.cell_start);
  hipLaunchKernelGGL(vsg_place_kernel, per_subset, block, 0, stream, w.cells, w.turn, w.cell_start, n, w.arrived);
  hipLaunchKernelGGL(vsg_pack_kernel, per_subset, block, 0, stream, fields, w.cells, w.cell_start, w.arrived, n,
                     radius_window ? 1 : 0, w.keys, w.ids, w.rec);
  g.cell_begin = w.cell_start;
  g.cell_ids = w.ids;
  g.cell_keys = w.keys;
  g.rec = w.rec;
  return hipGetLastError();
}

hipError_t launch_vsg_strain(const VsgGrid &g, float radius, int knn, double *fields, double *vsg, int n,
                             hipStream_t stream) {
  if (n <= 0) return hipSuccess;
  if (knn < 0 || knn > kVsgMaxK) return hipErrorInvalidValue;
  if (knn == 0)
    hipLaunchKernelGGL(vsg_strain_tiled_kernel, dim3((n + kVsgGroupSubsets - 1) / kVsgGroupSubsets), dim3(256), 0,
                       stream, g, radius, fields, vsg, n);
  else
    hipLaunchKernelGGL(vsg_strain_kernel, dim3((n + 127) / 128), dim3(128), 0, stream, g, radius, knn, fields, vsg,
                       n);
  return hipGetLastError();
}

hipError_t launch_neighbor_guess(const double *start, const double *cur, double *guess, const double *prev_guess,
                                 double tol, int *list, int *count, int n, hipStream_t stream) {
  if (n <= 0) return hipSuccess;
  hipLaunchKernelGGL(neighbor_guess_kernel, dim3((n + 255) / 256), dim3(256), 0, stream, start, cur, guess, prev_guess,
                     tol, list, count, n);
  return hipGetLastError();
}

hipError_t launch_reset_listed(const int *list, const int *count, const double *start, double *fields, int n,
                               hipStream_t stream) {
  if (n <= 0) return hipSuccess;
  hipLaunchKernelGGL(reset_listed_kernel, dim3((n + 255) / 256), dim3(256), 0, stream, list, count, start, fields, n);
  return hipGetLastError();
}

// One optimizer pass over `items` (nullptr: all subsets).  BATCHED mode runs the
// persistent kernel, then correlate_wide_kernel over the subsets whose window
// outgrew a wave's slot, then (Gauss-Newton) the PLAIN kernel over what that one
// leaves.  A Nelder-Mead pass with L.lane_simplex first runs the iterations in
// rows of 8 or 16 lanes per subset (results in nm); the persistent kernel then
// does the checks and the epilogue of each subset around them, and hands any
// subset that kernel left with kNmNoResult to correlate_wide_kernel, which runs
// its simplex.  When no subset's window can fit a wave's slot (L.wide_only),
// correlate_wide_kernel takes every item at once.
// work: the header, then the fallback list and the overflow lists of pass 0 and
// pass 1 (n each); the caller has cleared the header.
static hipError_t launch_pass(bool simplex, int storage, const Launch &L, const KParams &kp, const DImage &ref,
                              const DImage &def, const DSubsets &subs, double *fields, PassArgs pa, int *work,
                              hipStream_t stream) {
  const int defgrad = simplex ? 0 : kp.def_grads;
  const size_t n = (size_t)subs.n;
  PassLauncher plain = simplex ? launch_simplex_plain : launch_gn_plain;
  pa.nm_result = nullptr;
  pa.count_all = nullptr;
  if (L.mode == 0) {
    pa.ov_list = pa.ov_count = nullptr;
    return plain(storage, kp.interp, defgrad, L, kp, ref, def, subs, fields, pa, stream);
  }
  int *const ov0 = work + kWorkHeader + n, *const ov1 = ov0 + n;
  int *const ov_list = pa.pass == 0 ? ov0 : ov1, *const ov_count = work + kWorkOv0Count + pa.pass;
  int *const other = pa.pass == 0 ? ov1 : ov0;  // free once the lean hand-overs have been worked off
  auto set = [&](int which) { return work + (which + 2 * pa.pass) * kWorkCounterInts; };
  PassLauncher batched = simplex ? launch_simplex_batched : launch_gn_batched;
  hipError_t e;
  const bool wide_only = L.wide_only && !defgrad;
  if (!wide_only) {
    // Gauss-Newton pass 0 of square subsets with none of the options that the
    // common-case kernels leave out: they take every subset first and hand the
    // others (and those that leave the common case) to the general kernel
    // (common_kernel says which of them).
    const int np = (kp.en_rot != 0) + (kp.en_normal != 0) + (kp.en_shear != 0);
    if (!simplex && pa.pass == 0 && subs.S > 0 && !subs.mbox && !kp.def_grads && kp.momentum == 0.0f &&
        kp.init_gamma_thr == -1.0 && !kp.has_forced && kp.lm_alpha <= 0.0f && (np == 3 || np == 0)) {
      PassArgs pl = pa;
      pl.counter = work + kWorkSetLean * kWorkCounterInts;
      pl.ov_list = other;
      pl.ov_count = work + kWorkLeanCount;
      const CommonKernel common = common_kernel(
          CommonPass{subs.n, subs.S, np == 3, L.lds_floats_per_wave, kp.interp != 0, kp.uncertainty != 0,
                     pa.items != nullptr, L.border, L.num_cus});
      e = hipSuccess;
      if (common == CommonKernel::kCrew)
        e = launch_gn_crew(storage, kp.interp, np == 0, L, kp, ref, def, subs, fields, pl, stream);
      else if (common == CommonKernel::kLean)
        e = launch_gn_lean(storage, kp.interp, L, kp, ref, def, subs, fields, pl, stream);
      else if (common == CommonKernel::kTrans)
        e = launch_gn_trans(storage, kp.interp, L, kp, ref, def, subs, fields, pl, stream);
      if (e != hipSuccess) return e;
      if (common != CommonKernel::kNone) {
        pa.items = pl.ov_list;
        pa.item_count = pl.ov_count;
      }
    }
    if (simplex && L.lane_simplex) {
      float *nm = reinterpret_cast<float *>(work + kWorkHeader + 3 * n);
      e = launch_simplex_lanes(storage, kp.interp, L.lane_simplex, kp, ref, def, subs, fields, pa, nm,
                               work + kWorkLaneCount + pa.pass, stream);
      if (e != hipSuccess) return e;
      pa.nm_result = nm;
    }
    pa.counter = set(kWorkSetBatched);
    pa.ov_list = ov_list;
    pa.ov_count = ov_count;
    e = batched(storage, kp.interp, defgrad, L, kp, ref, def, subs, fields, pa, stream);
    if (e != hipSuccess) return e;
    pa.items = ov_list;
    pa.item_count = ov_count;
  }
  if (!defgrad) {
    pa.counter = set(kWorkSetWide);
    pa.ov_list = other;
    pa.ov_count = work + kWorkWideCount + pa.pass;
    pa.count_all = wide_only ? ov_count : nullptr;
    e = (simplex ? launch_simplex_wide : launch_gn_wide)(storage, kp.interp, L, kp, ref, def, subs, fields, pa,
                                                         stream);
    if (e != hipSuccess || simplex) return e;
    pa.items = pa.ov_list;
    pa.item_count = pa.ov_count;
  }
  pa.ov_list = pa.ov_count = pa.count_all = nullptr;
  return plain(storage, kp.interp, defgrad, L, kp, ref, def, subs, fields, pa, stream);
}

hipError_t launch_correlate(const Launch &L, int storage, const KParams &kp, const DImage &ref, const DImage &def,
                            const DSubsets &subs, double *fields, int *work, hipStream_t stream, const int *items,
                            const int *item_count) {
  if (subs.n <= 0) return hipSuccess;
  int *fb_list = work + kWorkHeader;
  hipError_t e = launch_zero_ints(work, kWorkHeader, stream);
  if (e != hipSuccess) return e;
  const bool simplex_first = kp.opt == 0 || kp.opt == 3;
  PassArgs pa{0, items, items ? item_count : nullptr, fb_list, work + kWorkFbCount, nullptr, nullptr, work, nullptr,
              nullptr};
  e = launch_pass(simplex_first, storage, L, kp, ref, def, subs, fields, pa, work, stream);
  // the second pass: the fallback optimizer, or Nelder-Mead for the forced subsets of a Gauss-Newton pass
  if (e != hipSuccess || !(kp.opt == 3 || kp.opt == 4 || (kp.has_forced && !simplex_first))) return e;
  PassArgs pb{1, fb_list, work + kWorkFbCount, nullptr, nullptr, nullptr, nullptr, work, nullptr, nullptr};
  return launch_pass(!simplex_first, storage, L, kp, ref, def, subs, fields, pb, work, stream);
}

hipError_t launch_gradients(int storage, const void *pix, int w, int h, float *gx, float *gy, int smooth,
                            float *tmpx, float *tmpy, hipStream_t stream) {
  dim3 block(64, 4), grid((w + 63) / 64, (h + 3) / 4);
  float *ox = smooth ? tmpx : gx, *oy = smooth ? tmpy : gy;
  if (storage == 0)
    hipLaunchKernelGGL(gradients_kernel<float>, grid, block, 0, stream, pix, w, h, ox, oy);
  else
    hipLaunchKernelGGL(gradients_kernel<uint16_t>, grid, block, 0, stream, pix, w, h, ox, oy);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess || !smooth) return e;
  hipLaunchKernelGGL(smooth_kernel, grid, block, 0, stream, tmpx, tmpy, w, h, gx, gy);
  return hipGetLastError();
}

hipError_t launch_gauss_filter(int storage, const void *in, void *out, int w, int h, int mask_size,
                               hipStream_t stream) {
  if (w < mask_size || h < mask_size) return hipErrorInvalidValue;
  return storage == 0 ? launch_gauss_t<float>(in, out, w, h, mask_size, stream)
                      : launch_gauss_t<uint16_t>(in, out, w, h, mask_size, stream);
}

hipError_t launch_zero_ints(int *p, int count, hipStream_t stream) {
  hipLaunchKernelGGL(zero_ints_kernel, dim3((count + 255) / 256), dim3(256), 0, stream, p, count);
  return hipGetLastError();
}

hipError_t launch_copy_doubles(double *dst, const double *src, size_t count, hipStream_t stream) {
  size_t blocks = (count + 255) / 256;
  if (blocks > 4096) blocks = 4096;
  if (blocks == 0) return hipSuccess;
  hipLaunchKernelGGL(copy_doubles_kernel, dim3((unsigned)blocks), dim3(256), 0, stream, dst, src, count);
  return hipGetLastError();
}

}  // namespace dice_hip
