// Pipe density compensation on the device: RECON::dcf_calc
// (recon_lib.cpp:854-917) over DCFgridFFT's real-valued polynomial-kernel
// gridder (DCFgridFFT.cpp:96-440).
//
// Two forms.  With dcf_acc = 1 and half widths below 3 (the defaults) every
// kernel has one width and the scatter is a matrix product per tile (k_dm_*).
// Other settings, one or two iterations of few samples, samples too scattered
// for the tiles, and calls without the memory for the tiles' lists take the
// general form: the samples sorted by 8x8x8-cell brick
// of the grid and 4x4x4 sub-brick, so that a wavefront's samples touch
// neighbouring cells, and scattered with float atomics.  Both sort once; the
// iterations run on the sorted copy and the weights are put back in the
// caller's order at the end.
//
// The trajectory stays resident; one call runs every iteration on the stream:
//   kw = 1; repeat iters: X = 0; X += A^T kw (scatter); kw2 = A X (gather);
//   kw = |kw2| < 1e-3 ? 0 : kw / kw2;   then kw = |kw * scale^3|.
// The gather and the ratio update are one kernel; no per-iteration host sync.
//
// HBM layout: X is the real grid [Sz][Sy][Sx] (x fastest) with the reference's
// extents trunc(os*N + 16), the kx extent taken from Nz (recon_lib.cpp:873).
// The sample order is the caller's (radial spokes run outward, so neighbours
// in a wavefront touch neighbouring cells).
//
// Arithmetic follows the reference expression by expression: float where it
// is float and double where it promotes (the table interpolation and the
// forward scale), with the *_rn intrinsics so that no multiply-add is fused
// where the reference rounds twice.  The general scatter adds with float
// atomics, as the reference's OpenMP atomics do, so the order of the additions
// into a cell differs from run to run; the matrix product sums in FP64, in a
// fixed order, and rounds once.  The gather sums in the reference's tap order.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <climits>
#include <cmath>
#include <cstdint>
#include <cstdio>
#include <cstring>
#include <string>

#include <hipcub/hipcub.hpp>

#include "mrn.h"
#include "mrn_internal.hpp"

namespace mrn {

thread_local std::string g_free_err;  // message of the last failed call without an op

const char *free_error() { return g_free_err.c_str(); }
void free_err_clear() { g_free_err.clear(); }
int free_fail(int status, const char *msg) {
  g_free_err = msg ? msg : "";
  return status;
}

namespace {

constexpr int DCF_MOD = 600;          // table points per cell (DCFgridFFT.cpp:101-103)
constexpr int DCF_MAX_TABLE = 12288;  // table floats held in LDS (48 KB)
// sort brick edge in cells (5.12 M radial samples, 553^3, 20 iterations,
// plain brick order: 8^3 bricks 104.6 ms, 4^3 106.7, 2^3 119, 16^3 155; 8^3
// with a 4096-cell box 115; 8^3 with 4^3 sub-bricks 100.4 against 102.1)
constexpr int DCF_BRICK = 8;
static_assert(DCF_BRICK >= 2 && DCF_BRICK % 2 == 0, "the sort key splits each brick into 8 sub-bricks");

struct DcfGeom {
  int S[3];
  float c[3];   // grid centre Sx/2 (integer division), as float
  float gx;     // grid_x = overgrid
  float dwin;
  float scale;  // dcf_scale applied to k
  float acc;
  int len;
};

int dcf_fail(int status, const char *msg) {
  g_free_err = msg;
  return status;
}

#define DCF_HIP(call)                                                       \
  do {                                                                      \
    hipError_t e_ = (call);                                                 \
    if (e_ != hipSuccess) {                                                 \
      g_free_err = std::string(#call ": ") + hipGetErrorString(e_);         \
      return MRN_EHIP;                                                      \
    }                                                                       \
  } while (0)

// Polynomial table (DCFgridFFT.cpp:56-90, 160-164), on the host in double.
int dcf_table(float dwin, int kernel, float *tab) {
  static const double P1[6] = {1., 0.04522831, -3.36020304, 1.12417012, 2.82448025, -1.63447764};
  static const double P2[6] = {1., 0.03056504, -3.01961845, 0.6679865, 2.77924058, -1.45923643};
  const double *c = kernel == 1 ? P2 : P1;
  const int len = (int)(dwin * (float)DCF_MOD) + 100;
  if (!tab) return len;
  double sum = 0.0;
  for (int i = 0; i < len; i++) {
    const double x = (double)i / (double)len;
    const double x2 = x * x, x4 = x2 * x2, x3 = x * x2, x5 = x * x4;
    tab[i] = (float)(c[0] + c[1] * x + c[2] * x2 + c[3] * x3 + c[4] * x4 + c[5] * x5);
  }
  for (int i = 0; i < len; i++) sum += tab[i];  // float entries summed in double
  const double f = 0.5 * (double)DCF_MOD / sum;
  for (int i = 0; i < len; i++) tab[i] = (float)(tab[i] * f);
  return len;
}

void grid_size(const mrn_dcf_params *p, int S[3]) {
  S[0] = (int)(p->overgrid * (float)p->N[2] + 16.0f);
  S[1] = (int)(p->overgrid * (float)p->N[1] + 16.0f);
  S[2] = (int)(p->overgrid * (float)p->N[0] + 16.0f);
}

__device__ __forceinline__ float kr_of(const DcfGeom &g, float kx, float ky, float kz, float k[3]) {
  k[0] = __fmul_rn(kx, g.scale);
  k[1] = __fmul_rn(ky, g.scale);
  k[2] = __fmul_rn(kz, g.scale);
  return __fsqrt_rn(__fadd_rn(__fadd_rn(__fmul_rn(k[0], k[0]), __fmul_rn(k[1], k[1])), __fmul_rn(k[2], k[2])));
}

// forward / scale_kw: kr / 128.0 * (acc - 1) + 1 in double
__device__ __forceinline__ float scale_fwd(const DcfGeom &g, float kr) {
  return (float)__dadd_rn(__dmul_rn(__ddiv_rn((double)kr, 128.0), (double)(g.acc - 1.0f)), 1.0);
}
// backward: kr / 128 * (acc - 1) + 1 in float
__device__ __forceinline__ float scale_bwd(const DcfGeom &g, float kr) {
  return __fadd_rn(__fmul_rn(__fdiv_rn(kr, 128.0f), __fsub_rn(g.acc, 1.0f)), 1.0f);
}

__device__ __forceinline__ bool axis(const DcfGeom &g, int a, float k, float scale, float &dk, int &s, int &e) {
  dk = __fadd_rn(__fmul_rn(k, g.gx), g.c[a]);
  const float r = __fmul_rn(scale, g.dwin);
  s = max((int)ceilf(__fsub_rn(dk, r)), 0);
  e = min((int)floorf(__fadd_rn(dk, r)), g.S[a] - 1);
  return !(s >= g.S[a] || e < 0);
}

// t[(int)del] * (1.0 - d) + t[(int)del + 1] * d, the first product in double
// and the second in float, as the reference's expression promotes
__device__ __forceinline__ double lerp(const float *tab, float dk, int l, float scale) {
  const float del = __fdiv_rn(fabsf(__fmul_rn((float)DCF_MOD, __fsub_rn(dk, (float)l))), scale);
  const int i = (int)del;
  const float d = __fsub_rn(del, (float)i);
  return __dadd_rn(__dmul_rn((double)tab[i], __dsub_rn(1.0, (double)d)), (double)__fmul_rn(tab[i + 1], d));
}

// Geometry of sample i for the forward gridder (DCFgridFFT.cpp:171-240): its
// kw, kernel scale, window centre dk and tap range [s, e] per axis.  False
// when the sample has no taps (i >= M, kw = 0, scale <= 0, or off the grid).
__device__ __forceinline__ bool fwd_taps(const DcfGeom &g, const float *__restrict__ kw,
                                         const float *__restrict__ kx, const float *__restrict__ ky,
                                         const float *__restrict__ kz, int64_t i, int64_t M, float &temp,
                                         float &scale, float dk[3], int s[3], int e[3]) {
  if (i >= M) return false;
  float k[3];
  scale = scale_fwd(g, kr_of(g, kx[i], ky[i], kz[i], k));
  temp = kw[i];
  bool live = temp != 0.0f && scale > 0.0f;  // a scale <= 0 (acc < 1, large |k|) has no taps
  live = live && axis(g, 0, k[0], scale, dk[0], s[0], e[0]);
  live = live && axis(g, 1, k[1], scale, dk[1], s[1], e[1]);
  live = live && axis(g, 2, k[2], scale, dk[2], s[2], e[2]);
  return live;
}

__device__ __forceinline__ void load_table(float *s_tab, const float *tab, int len) {
  for (int i = threadIdx.x; i < len; i += blockDim.x) s_tab[i] = tab[i];
  __syncthreads();
}

__global__ void k_dcf_fill(float *v, int64_t n, float value) {
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
    v[i] = value;
}

// DCFgridFFT::forward (DCFgridFFT.cpp:171-289): kernel weights with the
// reference's float/double promotions, grid += w * kw.  The samples run in
// DCF_BRICK^3-brick order, so in the dense centre of k-space a workgroup's
// 256 samples reach a box of a few thousand cells.  When the box (the
// bounding box of the taps of the workgroup's samples) holds at most DCF_BOX
// cells, the taps are summed there with FP64 LDS atomics (ds_add_f64; FP32
// LDS atomics are ~20x slower on gfx950) and each touched cell gets one
// float atomic in the grid, instead of one per tap.  Larger boxes (sparse
// regions) take the direct path, DCF_XL lanes per sample.  Launched with 256
// threads per workgroup.  The grid sums were already unordered (float
// atomics); a box only sums its part in double before rounding once.
// FP64 LDS box cells (64 KB).  20 iterations at 5.12 M radial samples, 553^3,
// 4^3 bricks: 105 ms; 4096 cells 113, 2048 120, no box 153 (the dense centre
// contends)
constexpr int DCF_BOX = 8192;
// Lanes per sample on the direct path.  The L2 serves float atomics per
// 64-byte line request: about 21 G requests/s on gfx950 when every lane of a
// wave has its own line, while lanes that share a line share its request
// (16 lanes on one line: 333 G atomics/s).  With one lane per x tap of a
// row, a row's 4-5 taps cost about one request instead of one each.
constexpr int DCF_XL = 8;

// float atomics the scatters of the last mrn_dcf_calc on this device issued
// to the grid (diagnostic: one 64-bit atomic per wavefront and launch)
static __device__ unsigned long long g_dcf_atomics;
__global__ void k_dcf_count_reset() { g_dcf_atomics = 0ull; }
__device__ __forceinline__ void count_atomics(unsigned long long n) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) n += __shfl_xor(n, o);
  if ((threadIdx.x & 63) == 0 && n) atomicAdd(&g_dcf_atomics, n);
}
__global__ __launch_bounds__(256) void k_dcf_scatter_box(float *__restrict__ X, const float *__restrict__ kw,
                                                         const float *__restrict__ kx, const float *__restrict__ ky,
                                                         const float *__restrict__ kz, int64_t M, DcfGeom g,
                                                         const float *__restrict__ tab) {
  extern __shared__ double dsh[];
  double *s_acc = dsh;
  float *s_tab = reinterpret_cast<float *>(dsh + DCF_BOX);
  __shared__ int s_red[6][256 / 64];
  load_table(s_tab, tab, g.len);
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  float temp = 0.0f, scale = 0.0f, dk[3] = {0.f, 0.f, 0.f};
  int s[3] = {0, 0, 0}, e[3] = {-1, -1, -1};
  const bool live = fwd_taps(g, kw, kx, ky, kz, i, M, temp, scale, dk, s, e);
  // bounding box of the workgroup's taps
  int r6[6];
#pragma unroll
  for (int a = 0; a < 3; a++) {
    r6[a] = live ? s[a] : INT_MAX;
    r6[3 + a] = live ? e[a] : INT_MIN;
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1)
#pragma unroll
    for (int a = 0; a < 3; a++) {
      r6[a] = min(r6[a], __shfl_xor(r6[a], o));
      r6[3 + a] = max(r6[3 + a], __shfl_xor(r6[3 + a], o));
    }
  if ((threadIdx.x & 63) == 0)
#pragma unroll
    for (int a = 0; a < 6; a++) s_red[a][threadIdx.x >> 6] = r6[a];
  __syncthreads();
  int lo[3], ext[3];
#pragma unroll
  for (int a = 0; a < 3; a++) {
    int mn = INT_MAX, mx = INT_MIN;
    for (int w = 0; w < 256 / 64; w++) {
      mn = min(mn, s_red[a][w]);
      mx = max(mx, s_red[3 + a][w]);
    }
    lo[a] = mn;
    ext[a] = mx >= mn ? mx - mn + 1 : 0;
  }
  const int64_t vol = (int64_t)ext[0] * ext[1] * ext[2];  // 0: no live sample
  if (vol == 0) return;                                     // (uniform)
  unsigned long long nat = 0;  // grid atomics of this thread
  if (vol > DCF_BOX) {  // (uniform) direct path: DCF_XL lanes per sample, one per x tap
    const int j = (int)(threadIdx.x % DCF_XL);
    const int64_t base = (int64_t)blockIdx.x * blockDim.x + threadIdx.x / DCF_XL;
    for (int r = 0; r < DCF_XL; r++) {  // the workgroup's samples, 256 / DCF_XL at a time
      float t2 = 0.0f, sc2 = 0.0f, dk2[3] = {0.f, 0.f, 0.f};
      int s2[3] = {0, 0, 0}, e2[3] = {-1, -1, -1};
      if (!fwd_taps(g, kw, kx, ky, kz, base + r * (256 / DCF_XL), M, t2, sc2, dk2, s2, e2)) continue;
      for (int lz = s2[2]; lz <= e2[2]; lz++) {
        const float wtz = (float)lerp(s_tab, dk2[2], lz, sc2);
        for (int ly = s2[1]; ly <= e2[1]; ly++) {
          const float wty = (float)__dmul_rn((double)wtz, lerp(s_tab, dk2[1], ly, sc2));
          float *row = X + ((int64_t)lz * g.S[1] + ly) * g.S[0];
          for (int lx = s2[0] + j; lx <= e2[0]; lx += DCF_XL) {
            const float wtx = (float)__dmul_rn((double)wty, lerp(s_tab, dk2[0], lx, sc2));
            atomicAdd(row + lx, __fmul_rn(wtx, t2));
            nat++;
          }
        }
      }
    }
    count_atomics(nat);
    return;
  }
  for (int q = threadIdx.x; q < vol; q += blockDim.x) s_acc[q] = 0.0;
  __syncthreads();
  if (live) {
    for (int lz = s[2]; lz <= e[2]; lz++) {
      const float wtz = (float)lerp(s_tab, dk[2], lz, scale);
      for (int ly = s[1]; ly <= e[1]; ly++) {
        const float wty = (float)__dmul_rn((double)wtz, lerp(s_tab, dk[1], ly, scale));
        double *brow = s_acc + ((lz - lo[2]) * ext[1] + (ly - lo[1])) * ext[0] - lo[0];
        for (int lx = s[0]; lx <= e[0]; lx++) {
          const float wtx = (float)__dmul_rn((double)wty, lerp(s_tab, dk[0], lx, scale));
          atomicAdd(brow + lx, (double)__fmul_rn(wtx, temp));
        }
      }
    }
  }
  __syncthreads();
  // one float atomic per touched cell; consecutive lanes take consecutive x
  for (int q = threadIdx.x; q < vol; q += blockDim.x) {
    const double v = s_acc[q];
    if (v == 0.0) continue;
    const int x = q % ext[0], yz = q / ext[0];
    const int y = yz % ext[1], z = yz / ext[1];
    atomicAdd(X + ((int64_t)(lo[2] + z) * g.S[1] + (lo[1] + y)) * g.S[0] + lo[0] + x, (float)v);
    nat++;
  }
  count_atomics(nat);
}

// DCFgridFFT::backward (DCFgridFFT.cpp:314-440) and the ratio update of
// dcf_calc (recon_lib.cpp:895-905), one thread per sample.  sum (optional)
// collects the iteration's sum of |kw| (the reference prints it).
__global__ __launch_bounds__(256) void k_dcf_gather_update(const float *__restrict__ X, float *__restrict__ kw,
                                                           const float *__restrict__ kx,
                                                           const float *__restrict__ ky,
                                                           const float *__restrict__ kz, int64_t M, DcfGeom g,
                                                           const float *__restrict__ tab, double *sum) {
  extern __shared__ float s_tab[];
  __shared__ double s_part[256 / 64];
  load_table(s_tab, tab, g.len);
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  double mine = 0.0;
  if (i < M) {
    float k[3];
    const float kr = kr_of(g, kx[i], ky[i], kz[i], k);
    const float scale = scale_bwd(g, kr);
    float temp = 0.0f;
    float dk[3];
    int s[3], e[3];
    if (scale > 0.0f && axis(g, 0, k[0], scale, dk[0], s[0], e[0]) && axis(g, 1, k[1], scale, dk[1], s[1], e[1]) &&
        axis(g, 2, k[2], scale, dk[2], s[2], e[2])) {
      for (int lz = s[2]; lz <= e[2]; lz++) {
        const float wtz = (float)lerp(s_tab, dk[2], lz, scale);
        for (int ly = s[1]; ly <= e[1]; ly++) {
          const float wty = (float)__dmul_rn((double)wtz, lerp(s_tab, dk[1], ly, scale));
          const float *row = X + ((int64_t)lz * g.S[1] + ly) * g.S[0];
          const int nx = e[0] - s[0] + 1;
          if (nx <= 8 && s[0] + 8 <= g.S[0]) {
            // the row's taps as two 16-byte loads (4-byte aligned; the 8
            // cells stay inside the row), summed in the same tap order
            float v[8];
            __builtin_memcpy(v, row + s[0], sizeof(v));
#pragma unroll
            for (int q = 0; q < 8; q++)
              if (q < nx) {
                const float wtx = (float)__dmul_rn((double)wty, lerp(s_tab, dk[0], s[0] + q, scale));
                temp = __fadd_rn(temp, __fmul_rn(wtx, v[q]));
              }
          } else {
            for (int lx = s[0]; lx <= e[0]; lx++) {
              const float wtx = (float)__dmul_rn((double)wty, lerp(s_tab, dk[0], lx, scale));
              temp = __fadd_rn(temp, __fmul_rn(wtx, row[lx]));
            }
          }
        }
      }
    }
    float w = kw[i];
    if ((double)fabsf(temp) < 1e-3) {
      w = 0.0f;
    } else {
      w = __fdiv_rn(w, temp);
      mine = (double)fabsf(w);
    }
    kw[i] = w;
  }
  if (sum) {
    for (int o = 32; o > 0; o >>= 1) mine += __shfl_down(mine, o);
    if ((threadIdx.x & 63) == 0) s_part[threadIdx.x >> 6] = mine;
    __syncthreads();
    if (threadIdx.x == 0) {
      double t = 0.0;
      for (int w = 0; w < (int)(blockDim.x >> 6); w++) t += s_part[w];
      atomicAdd(sum, t);
    }
  }
}

// ------------------------------------------- one kernel width (dcf_acc = 1)
// The scatter is a matrix product.  A tile of 4 (z) x 4 (y) x 16 (x) cells is
//   T[zy][x] = sum over samples of (kw wz wy)[zy] wx[x],
// 16 x 16 sums in FP64, by v_mfma_f64_16x16x4_f64, four samples each.  One
// wavefront owns a tile and walks the samples that can reach it (its visits);
// nothing is added with atomics and no cell is zeroed: the cells that a sample
// reads are cells some sample reaches, and those tiles are written whole.
// Samples are sorted by the 4^3-cell bin of their first tap; a tile's visits
// are the bins one bin row below and beside it, contiguous runs along x.
// The box scatter above was bound by the L2's float atomic requests.  5.12 M
// radial samples, 553^3 grid: 3.78 + 0.09 ms per iteration for scatter and
// zeroing before, 0.78 now (20 iterations 91 -> 28 ms); the FP64 LDS sums of
// 16^3-cell bricks with their halos added afterwards took 0.82 + 0.87 ms (random
// LDS banks, 3 times the cells).  What remains is the FP64 weights: 5 visits per
// sample, each evaluating 13 of them; without branches 0.84 ms.
constexpr int DM_BIN = 4;      // bin edge (cells); tiles are DM_X x 4 x 4
constexpr int DM_NB = 1;       // 16-cell blocks of a tile along x (2: 1.1 ms against 0.78)
constexpr int DM_X = 16 * DM_NB;
constexpr int DM_CELLS = DM_X * 16;
constexpr int DM_REACH = 5;    // last minus first tap on an axis, at most
constexpr int DM_XT = DM_REACH + 1;
constexpr int DM_BATCH = 32;   // visits weighted at a time
constexpr int DM_ITEM = 2048;  // visits per work item, at most
constexpr int DM_RUNS = 9;     // bin rows (z, y) of a tile
// consecutive workgroups per XCD: neighbouring samples read the same cells, and
// neighbouring tiles the same samples, through one L2
constexpr int DM_XRUN = 16;

struct DmGeom {
  int nb[3], nt[3];  // bins and tiles per axis
  int reach;         // last minus first tap
  int item;          // visits per work item
};

typedef double dm_v4d __attribute__((ext_vector_type(4)));

// lerp() with a kernel scale of 1, where the reference's division changes nothing
__device__ __forceinline__ double lerp1(const float *tab, float dk, int l) {
  const float del = fabsf(__fmul_rn((float)DCF_MOD, __fsub_rn(dk, (float)l)));
  const int i = (int)del;
  const float d = __fsub_rn(del, (float)i);
  return __dadd_rn(__dmul_rn((double)tab[i], __dsub_rn(1.0, (double)d)), (double)__fmul_rn(tab[i + 1], d));
}

// taps [s, e] of a grid coordinate (axis() with a kernel scale of 1; none: e < s
// or outside [0, S))
__device__ __forceinline__ void taps1(const DcfGeom &g, int a, float dk, int &s, int &e) {
  s = max((int)ceilf(__fsub_rn(dk, g.dwin)), 0);
  e = min((int)floorf(__fadd_rn(dk, g.dwin)), g.S[a] - 1);
}

// coordinates of one sample; false when it has no taps (off the grid, or a
// |k| that is not finite: the reference's scale kr / 128 * 0 + 1 is then NaN)
__device__ __forceinline__ bool coords1(const DcfGeom &g, float kx, float ky, float kz, float dk[3], int s[3]) {
  const float k[3] = {__fmul_rn(kx, g.scale), __fmul_rn(ky, g.scale), __fmul_rn(kz, g.scale)};
  const float r2 = __fadd_rn(__fadd_rn(__fmul_rn(k[0], k[0]), __fmul_rn(k[1], k[1])), __fmul_rn(k[2], k[2]));
  bool live = r2 < INFINITY;
#pragma unroll
  for (int a = 0; a < 3; a++) {
    int e;
    live = live && axis(g, a, k[a], 1.0f, dk[a], s[a], e);
  }
  return live;
}

// sort key: the bin of the first tap; samples without taps last
__global__ void k_dm_keys(const float *__restrict__ kx, const float *__restrict__ ky, const float *__restrict__ kz,
                          int64_t M, DcfGeom g, DmGeom m, uint32_t *__restrict__ keys, uint32_t *__restrict__ idx) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= M) return;
  float dk[3];
  int s[3];
  keys[i] = coords1(g, kx[i], ky[i], kz[i], dk, s)
                ? (uint32_t)(((s[2] / DM_BIN) * m.nb[1] + s[1] / DM_BIN) * m.nb[0] + s[0] / DM_BIN)
                : (uint32_t)(m.nb[0] * m.nb[1] * m.nb[2]);
  idx[i] = (uint32_t)i;
}

// {grid coordinates, kw = 1} in sorted order; a sample without taps lies far
// off the grid
__global__ void k_dm_coords(const uint32_t *__restrict__ perm, const float *__restrict__ kx,
                            const float *__restrict__ ky, const float *__restrict__ kz, int64_t M, DcfGeom g,
                            float4 *__restrict__ c) {
  const int64_t j = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (j >= M) return;
  const uint32_t i = perm[j];
  float dk[3];
  int s[3];
  c[j] = coords1(g, kx[i], ky[i], kz[i], dk, s) ? make_float4(dk[0], dk[1], dk[2], 1.0f)
                                                : make_float4(-1e6f, -1e6f, -1e6f, 1.0f);
}

// first sample of every bin (sorted keys; entry nbins: the samples with taps)
__global__ void k_dm_bins(const uint32_t *__restrict__ keys, int64_t M, int nbins, int32_t *__restrict__ start) {
  const int b = blockIdx.x * blockDim.x + threadIdx.x;
  if (b > nbins) return;
  int64_t lo = 0, hi = M;
  while (lo < hi) {
    const int64_t mid = (lo + hi) >> 1;
    if (keys[mid] < (uint32_t)b) lo = mid + 1;
    else hi = mid;
  }
  start[b] = (int32_t)lo;
}

// bins [b0, b1] on one axis whose samples can reach cells [c0, c0 + n)
__device__ __forceinline__ void dm_reach(const DmGeom &m, int a, int c0, int n, int &b0, int &b1) {
  b0 = max(c0 - m.reach, 0) / DM_BIN;
  b1 = min((c0 + n - 1) / DM_BIN, m.nb[a] - 1);
}

// work items and partial-sum slots of every tile
__global__ void k_dm_count(const int32_t *__restrict__ start, DmGeom m, int ntiles, int32_t *__restrict__ items,
                           int32_t *__restrict__ slots) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t > ntiles) return;
  int n = 0;
  if (t < ntiles) {
    int x0, x1, y0, y1, z0, z1;
    dm_reach(m, 0, (t % m.nt[0]) * DM_X, DM_X, x0, x1);
    dm_reach(m, 1, ((t / m.nt[0]) % m.nt[1]) * DM_BIN, DM_BIN, y0, y1);
    dm_reach(m, 2, (t / (m.nt[0] * m.nt[1])) * DM_BIN, DM_BIN, z0, z1);
    int64_t v = 0;
    for (int z = z0; z <= z1; z++)
      for (int y = y0; y <= y1; y++) {
        const int64_t b = ((int64_t)z * m.nb[1] + y) * m.nb[0];
        v += start[b + x1 + 1] - start[b + x0];
      }
    n = (int)((v + m.item - 1) / m.item);
  }
  items[t] = n;
  slots[t] = n > 1 ? n : 0;
}

// work items {tile, item of the tile, slot + 1 or 0, 0}; the split tiles' list
__global__ void k_dm_items(const int32_t *__restrict__ items, const int32_t *__restrict__ ofs,
                           const int32_t *__restrict__ slot0, int ntiles, int4 *__restrict__ list) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= ntiles) return;
  const int n = items[t], o = ofs[t];
  for (int q = 0; q < n; q++) list[o + q] = make_int4(t, q, n > 1 ? slot0[t] + q + 1 : 0, n);
}

__device__ __forceinline__ void dm_wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

__global__ __launch_bounds__(256, 4) void k_dm_scatter(float *__restrict__ X, double *__restrict__ part,
                                                       const float4 *__restrict__ coords,
                                                       const int32_t *__restrict__ start,
                                                       const int4 *__restrict__ list, int nitems, DcfGeom g, DmGeom m,
                                                       const float *__restrict__ tab) {
  extern __shared__ float s_tab[];
  // per wavefront and visit: 4 z weights (times kw), 4 y weights, DM_XT x weights
  constexpr int W = 8 + DM_XT;
  __shared__ double s_w[4][DM_BATCH * W];
  __shared__ int s_x0[4][DM_BATCH];  // first x tap relative to the tile
  load_table(s_tab, tab, g.len);     // before any wavefront can leave
  // (scalar: the item, its runs and their offsets are the wavefront's)
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int item = xcd_block(blockIdx.x, gridDim.x, DM_XRUN) * 4 + wave;
  if (item >= nitems) return;
  const int4 it = list[item];
  const int t0[3] = {(it.x % m.nt[0]) * DM_X, ((it.x / m.nt[0]) % m.nt[1]) * DM_BIN,
                     (it.x / (m.nt[0] * m.nt[1])) * DM_BIN};
  // the tile's runs: visit v of run r is sample v + add[r] for v >= first[r]
  int x0, x1, y0, y1, z0, z1;
  dm_reach(m, 0, t0[0], DM_X, x0, x1);
  dm_reach(m, 1, t0[1], DM_BIN, y0, y1);
  dm_reach(m, 2, t0[2], DM_BIN, z0, z1);
  int first[DM_RUNS], add[DM_RUNS], total = 0;
  const int ny = y1 - y0 + 1, nruns = ny * (z1 - z0 + 1);
#pragma unroll
  for (int r = 0; r < DM_RUNS; r++) {
    first[r] = INT_MAX;
    add[r] = 0;
    if (r < nruns) {
      const int64_t b = ((int64_t)(z0 + r / ny) * m.nb[1] + y0 + r % ny) * m.nb[0];
      const int s = start[b + x0], n = start[b + x1 + 1] - s;
      first[r] = total;
      add[r] = s - total;
      total += n;
    }
  }
  const int vbeg = it.y * m.item, vend = min(vbeg + m.item, total);
  auto load = [&](int v) -> float4 {  // visit v (the last one past the end)
    v = min(v, vend - 1);
    int q = add[0];
#pragma unroll
    for (int r = 1; r < DM_RUNS; r++) q = v >= first[r] ? add[r] : q;
    return coords[v + q];
  };
  dm_v4d acc[DM_NB];
#pragma unroll
  for (int nb = 0; nb < DM_NB; nb++) acc[nb] = dm_v4d{0.0, 0.0, 0.0, 0.0};
  const int sl = lane >> 1, h = lane & 1;    // weights: visit, half of them
  const int ci = lane & 15, kq = lane >> 4;  // product: zy cell / x cell, sample of the group
  float4 c = load(vbeg + sl);
  for (int base = vbeg; base < vend; base += DM_BATCH) {
    const bool ok = base + sl < vend;
    const float4 cn = load(base + DM_BATCH + sl);
    const float dk[3] = {c.x, c.y, c.z};
    int s[3], e[3];
#pragma unroll
    for (int a = 0; a < 3; a++) taps1(g, a, dk[a], s[a], e[a]);
    const bool any = ok && e[0] >= t0[0] && s[0] < t0[0] + DM_X && s[0] <= e[0] && e[1] >= t0[1] &&
                     s[1] < t0[1] + DM_BIN && e[2] >= t0[2] && s[2] < t0[2] + DM_BIN;
    double *w = &s_w[wave][sl * W];
#pragma unroll
    for (int u = 0; u < 2; u++) {
      const int q = 2 * h + u, lz = t0[2] + q, ly = t0[1] + q;
      w[q] = any && lz >= s[2] && lz <= e[2] ? __dmul_rn(lerp1(s_tab, dk[2], lz), (double)c.w) : 0.0;
      w[4 + q] = any && ly >= s[1] && ly <= e[1] ? lerp1(s_tab, dk[1], ly) : 0.0;
    }
#pragma unroll
    for (int u = 0; u < DM_XT / 2; u++) {
      const int q = h * (DM_XT / 2) + u;
      w[8 + q] = any && s[0] + q <= e[0] ? lerp1(s_tab, dk[0], s[0] + q) : 0.0;
    }
    if (h == 0) s_x0[wave][sl] = s[0] - t0[0];
    unsigned long long hit[DM_NB];  // bits 2 s, 2 s + 1: visit s reaches the block
#pragma unroll
    for (int nb = 0; nb < DM_NB; nb++)
      hit[nb] = __ballot(any && e[0] >= t0[0] + 16 * nb && s[0] < t0[0] + 16 * nb + 16);
    c = cn;
    dm_wave_sync();
#pragma unroll
    for (int q = 0; q < DM_BATCH / 4; q++) {
      const double *v = &s_w[wave][(4 * q + kq) * W];
      const double a = v[ci >> 2] * v[4 + (ci & 3)];
      const int d0 = ci - s_x0[wave][4 * q + kq];
#pragma unroll
      for (int nb = 0; nb < DM_NB; nb++) {
        if (!((hit[nb] >> (8 * q)) & 0xFFull)) continue;  // (uniform)
        const int d = d0 + 16 * nb;
        const double b = (unsigned)d < (unsigned)DM_XT ? v[8 + d] : 0.0;
        acc[nb] = __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, acc[nb], 0, 0, 0);
      }
    }
    dm_wave_sync();
  }
  // register r of lane l: zy cell 4 r + l / 16 (z plane r, y l / 16), x cell l % 16
  const int y = t0[1] + kq;
#pragma unroll
  for (int nb = 0; nb < DM_NB; nb++) {
    const int x = t0[0] + 16 * nb + ci;
#pragma unroll
    for (int r = 0; r < 4; r++) {
      if (it.z) {
        part[(int64_t)(it.z - 1) * DM_CELLS + (nb * 4 + r) * 64 + lane] = acc[nb][r];
      } else if (x < g.S[0] && y < g.S[1] && t0[2] + r < g.S[2]) {
        X[((int64_t)(t0[2] + r) * g.S[1] + y) * g.S[0] + x] = (float)acc[nb][r];
      }
    }
  }
}

// the split tiles: their items' sums added in order
__global__ __launch_bounds__(DM_CELLS) void k_dm_sum(float *__restrict__ X, const double *__restrict__ part,
                                                const int4 *__restrict__ heavy, DcfGeom g, DmGeom m) {
  const int4 it = heavy[blockIdx.x];
  const int lane = threadIdx.x & 63, r = (threadIdx.x >> 6) & 3, nb = threadIdx.x >> 8;
  const int x = (it.x % m.nt[0]) * DM_X + 16 * nb + (lane & 15), y = ((it.x / m.nt[0]) % m.nt[1]) * DM_BIN + (lane >> 4),
            z = (it.x / (m.nt[0] * m.nt[1])) * DM_BIN + r;
  const double *p = part + (int64_t)(it.z - 1) * DM_CELLS + threadIdx.x;
  double a = 0.0;
#pragma unroll 8
  for (int q = 0; q < it.w; q++) a += p[(int64_t)q * DM_CELLS];
  if (x < g.S[0] && y < g.S[1] && z < g.S[2]) X[((int64_t)z * g.S[1] + y) * g.S[0] + x] = (float)a;
}

// the first work item of every split tile
__global__ void k_dm_heavy(const int4 *__restrict__ list, int nitems, int4 *__restrict__ heavy, int *__restrict__ n) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < nitems && list[i].z && list[i].y == 0) heavy[atomicAdd(n, 1)] = list[i];
}

// k_dcf_gather_update with one kernel width: a sample's x weights are
// evaluated once, not once per (z, y) row.  5.12 M samples: 0.58 ms with the
// weights per row, 0.51 now (its row loads' lines in the L1).
__global__ __launch_bounds__(256) void k_dm_gather_update(const float *__restrict__ X, float4 *__restrict__ coords,
                                                          int64_t M, DcfGeom g, const float *__restrict__ tab,
                                                          double *sum) {
  extern __shared__ float s_tab[];
  __shared__ double s_part[256 / 64];
  load_table(s_tab, tab, g.len);
  const int64_t i = (int64_t)xcd_block(blockIdx.x, gridDim.x, DM_XRUN) * blockDim.x + threadIdx.x;
  double mine = 0.0;
  if (i < M) {
    const float4 c = coords[i];
    const float dk[3] = {c.x, c.y, c.z};
    int s[3], e[3];
#pragma unroll
    for (int a = 0; a < 3; a++) taps1(g, a, dk[a], s[a], e[a]);
    const int nx = e[0] - s[0] + 1, ny = e[1] - s[1] + 1;
    double wx[DM_XT], wy[DM_XT];
#pragma unroll
    for (int q = 0; q < DM_XT; q++) {
      wx[q] = q < nx ? lerp1(s_tab, dk[0], s[0] + q) : 0.0;
      wy[q] = q < ny ? lerp1(s_tab, dk[1], s[1] + q) : 0.0;
    }
    float temp = 0.0f;
    if (nx > 0 && ny > 0) {
      const bool whole = s[0] + DM_XT <= g.S[0];  // DM_XT cells from the first tap stay in the row
      for (int lz = s[2]; lz <= e[2]; lz++) {
        const float wtz = (float)lerp1(s_tab, dk[2], lz);
        const float *plane = X + ((int64_t)lz * g.S[1] + s[1]) * g.S[0] + s[0];
        float v[DM_XT][DM_XT];
#pragma unroll
        for (int y = 0; y < DM_XT; y++)
          if (y < ny) {
            if (whole) {
              __builtin_memcpy(v[y], plane + (int64_t)y * g.S[0], sizeof(v[y]));
            } else {
#pragma unroll
              for (int q = 0; q < DM_XT; q++) v[y][q] = q < nx ? plane[(int64_t)y * g.S[0] + q] : 0.0f;
            }
          }
#pragma unroll
        for (int y = 0; y < DM_XT; y++)
          if (y < ny) {
            const float wty = (float)__dmul_rn((double)wtz, wy[y]);
#pragma unroll
            for (int q = 0; q < DM_XT; q++)
              if (q < nx) temp = __fadd_rn(temp, __fmul_rn((float)__dmul_rn((double)wty, wx[q]), v[y][q]));
          }
      }
    }
    float w = c.w;
    if ((double)fabsf(temp) < 1e-3) {
      w = 0.0f;
    } else {
      w = __fdiv_rn(w, temp);
      mine = (double)fabsf(w);
    }
    coords[i].w = w;
  }
  if (sum) {
    for (int o = 32; o > 0; o >>= 1) mine += __shfl_down(mine, o);
    if ((threadIdx.x & 63) == 0) s_part[threadIdx.x >> 6] = mine;
    __syncthreads();
    if (threadIdx.x == 0) {
      double t = 0.0;
      for (int w = 0; w < (int)(blockDim.x >> 6); w++) t += s_part[w];
      atomicAdd(sum, t);
    }
  }
}

// scale_kw (DCFgridFFT.cpp:291-312) and kw = |kw| (recon_lib.cpp:910)
__global__ void k_dcf_finish(float *__restrict__ kw, const float *__restrict__ kx, const float *__restrict__ ky,
                             const float *__restrict__ kz, int64_t M, DcfGeom g) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= M) return;
  float k[3];
  const double s = (double)scale_fwd(g, kr_of(g, kx[i], ky[i], kz[i], k));
  kw[i] = fabsf((float)__dmul_rn((double)kw[i], __dmul_rn(__dmul_rn(s, s), s)));
}

// sort key: the DCF_BRICK^3-cell brick of the sample's nearest grid cell,
// then its (DCF_BRICK / 2)^3 sub-brick: the scatter's workgroups take whole
// bricks (their LDS boxes), the gather's wavefronts sub-bricks (their loads
// stay closer together)
__global__ void k_dcf_keys(const float *__restrict__ kx, const float *__restrict__ ky,
                           const float *__restrict__ kz, int64_t M, DcfGeom g, uint32_t *__restrict__ keys,
                           uint32_t *__restrict__ idx) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= M) return;
  float k[3];
  kr_of(g, kx[i], ky[i], kz[i], k);
  uint32_t key = 0, sub = 0;
  for (int a = 2; a >= 0; a--) {
    const float dk = __fadd_rn(__fmul_rn(k[a], g.gx), g.c[a]);
    int c = (int)floorf(dk);
    c = c < 0 ? 0 : (c > g.S[a] - 1 ? g.S[a] - 1 : c);
    key = key * (uint32_t)((g.S[a] + DCF_BRICK - 1) / DCF_BRICK) + (uint32_t)(c / DCF_BRICK);
    sub = sub * 2u + (uint32_t)((c % DCF_BRICK) / (DCF_BRICK / 2));
  }
  keys[i] = key * 8u + sub;
  idx[i] = (uint32_t)i;
}

__global__ void k_dcf_gather3(const uint32_t *__restrict__ perm, const float *__restrict__ kx,
                              const float *__restrict__ ky, const float *__restrict__ kz, int64_t M,
                              float *__restrict__ sx, float *__restrict__ sy, float *__restrict__ sz) {
  const int64_t j = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (j >= M) return;
  const uint32_t i = perm[j];
  sx[j] = kx[i];
  sy[j] = ky[i];
  sz[j] = kz[i];
}

__global__ void k_dm_unsort(const uint32_t *__restrict__ perm, const float4 *__restrict__ c, int64_t M,
                            float *__restrict__ kw) {
  const int64_t j = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (j < M) kw[perm[j]] = c[j].w;
}

__global__ void k_dcf_unsort(const uint32_t *__restrict__ perm, const float *__restrict__ ws, int64_t M,
                             float *__restrict__ kw) {
  const int64_t j = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (j < M) kw[perm[j]] = ws[j];
}

int64_t nblocks(int64_t n, int b) { return (n + b - 1) / b; }

// Device memory of one call, freed with it: arrays wanted together are one
// allocation (a hipMalloc and hipFree of some MB take 40 us between them).
struct Scratch {
  struct Want {
    void **q;
    size_t at;
  };
  void *p[3];
  Want w[16];
  int n = 0, nw = 0;
  size_t bytes = 0;
  hipStream_t st;
  explicit Scratch(hipStream_t s) : st(s) {}
  Scratch(const Scratch &) = delete;
  template <class T>
  void want(T *&q, int64_t count) {
    q = nullptr;
    w[nw++] = Want{(void **)&q, bytes};
    bytes += (sizeof(T) * (size_t)(count > 0 ? count : 1) + 255) & ~(size_t)255;
  }
  hipError_t take() {  // the arrays wanted since the last one
    void *v = nullptr;
    const hipError_t e = dev_malloc(&v, bytes);
    if (e == hipSuccess) {
      p[n++] = v;
      for (int i = 0; i < nw; i++) *w[i].q = (uint8_t *)v + w[i].at;
    }
    nw = 0;
    bytes = 0;
    return e;
  }
  ~Scratch() {
    if (n > 0) (void)hipStreamSynchronize(st);
    for (int i = 0; i < n; i++) hipFree(p[i]);
  }
};

// Whether the one-width form above covers these settings: one scale, at most
// DM_XT taps per axis (the 1e-3 cells cover the coordinates' float rounding on
// grids below 8192), bins and tiles within 32 bits.
bool dm_fits(const DcfGeom &g, DmGeom &m) {
  if (g.acc != 1.0f) return false;
  m.reach = (int)floorf(2.0f * g.dwin + 1e-3f);
  int64_t bins = 1, tiles = 1;
  for (int a = 0; a < 3; a++) {
    if (g.S[a] > 8192) return false;
    m.nb[a] = (g.S[a] + DM_BIN - 1) / DM_BIN;
    m.nt[a] = a == 0 ? (g.S[a] + DM_X - 1) / DM_X : m.nb[a];
    bins *= m.nb[a];
    tiles *= m.nt[a];
  }
  return m.reach <= DM_REACH && bins < (1 << 30) && tiles < (1 << 30);
}

// Visits per work item.  An item is one wavefront's serial walk, so a dense
// tile's must not outlast the rest of the launch: about 5 visits per sample over
// the chip's 4096 wavefronts, in whole batches.  us per iteration at 128 / 512 /
// 2048 visits per item and by this rule: 32^3, 10000 radial samples 31 / 47 / 107
// / 31, 200000 78 / 72 / 141 / 70; 64^3, 50000 41 / 54 / 124 / 41; 128^3, 500000
// 171 / 164 / 255 / 164; 256^3, 5 M 1450 / 1283 / 1264 / 1264.
int dm_item(int64_t M) {
  return (int)std::min<int64_t>(std::max<int64_t>(5 * M / 4096 / DM_BATCH * DM_BATCH, 128), DM_ITEM);
}

// Whether a call of so many iterations takes the one-width form: it spends 50 to
// 200 us more on its lists than the general form on its sort, and wins 50 us per
// iteration on the smallest calls.  The call in us, general / one-width: 32^3,
// 1000 samples 0 / 1 / 20 iterations 117 / 173, 200 / 219, 1784 / 715; 64^3, 50000
// radial samples, 1 iteration 246 / 363; 2 M 1502 / 1398.
bool dm_iters(int iters, int64_t M) { return iters >= 3 || iters * M >= (1 << 20); }

// Whether its work items are too empty: an item costs a batch of 32 visits even
// where scattered samples leave it with one or two.  Fitted to both forms' times
// per iteration, general / one-width: 256^3, random samples 50000 253 / 288 us
// (206193 items), 200000 507 / 662 (499762), 500000 905 / 896 (621276), 2 M 2850 /
// 1268; 256^3 radial 200000 446 / 194 (108247); 384^3 random 50000 447 / 319
// (235967), 200000 715 / 1016 (793909), 500000 1179 / 1807 (1455385), 2 M 3283 / 3096
// (2090240).  By now the lists are built and the general form starts from its
// own sort: the iterations have to save 600 us.
bool dm_sparse(const DcfGeom &g, int64_t M, int64_t items, int iters) {
  const int64_t cells = (int64_t)g.S[0] * g.S[1] * g.S[2];
  const int64_t over = items - (M + cells / 1740 + 60000);  // at 1.2 ns
  return over * iters > 500000;
}

// A status that is none of the interface's: the call goes on in the general form.
constexpr int DM_GENERAL = -1;
#define DM_MEM(call)                                  \
  do {                                                \
    const hipError_t m_ = (call);                     \
    if (m_ == hipErrorOutOfMemory) {                  \
      (void)hipGetLastError();                        \
      return DM_GENERAL;                              \
    }                                                 \
    DCF_HIP(m_);                                      \
  } while (0)

int dm_calc(const mrn_dcf_params *p, const DcfGeom &g, const DmGeom &m, int64_t M, const float *kx, const float *ky,
            const float *kz, float *kw, double *sums, const float *tab_h, hipStream_t st) {
  Scratch mem(st);
  const int nbins = m.nb[0] * m.nb[1] * m.nb[2], ntiles = m.nt[0] * m.nt[1] * m.nt[2];
  float *X, *tab;
  float4 *coords;
  uint32_t *keys, *perm;  // [2][M] each
  int32_t *start, *items, *ofs, *slots, *slot0;
  int4 *list, *heavy;
  int *nheavy_d;
  double *dsum, *part;
  uint8_t *tmp;
  mem.want(tab, g.len);
  mem.want(dsum, p->iters);
  mem.want(coords, M);
  mem.want(keys, 2 * M);
  mem.want(perm, 2 * M);
  mem.want(start, (int64_t)nbins + 1);
  mem.want(items, (int64_t)ntiles + 1);
  mem.want(ofs, (int64_t)ntiles + 1);
  mem.want(slots, (int64_t)ntiles + 1);
  mem.want(slot0, (int64_t)ntiles + 1);
  mem.want(nheavy_d, 1);
  int bits = 1;
  while ((1ll << bits) <= nbins) bits++;  // keys 0 .. nbins
  size_t tb = 0, sb = 0;
  DCF_HIP(hipcub::DeviceRadixSort::SortPairs(nullptr, tb, keys, keys, perm, perm, (int)M, 0, bits, st));
  DCF_HIP(hipcub::DeviceScan::ExclusiveSum(nullptr, sb, items, ofs, ntiles + 1, st));
  tb = tb > sb ? tb : sb;
  mem.want(tmp, (int64_t)tb);
  DM_MEM(mem.take());
  DCF_HIP(hipMemcpyAsync(tab, tab_h, sizeof(float) * g.len, hipMemcpyHostToDevice, st));
  const size_t lds = sizeof(float) * g.len;
  const dim3 gs((unsigned)nblocks(M, 256));
  hipLaunchKernelGGL(k_dm_keys, gs, dim3(256), 0, st, kx, ky, kz, M, g, m, keys, perm);
  DCF_HIP(hipGetLastError());
  DCF_HIP(hipcub::DeviceRadixSort::SortPairs(tmp, tb, keys, keys + M, perm, perm + M, (int)M, 0, bits, st));
  const uint32_t *order = perm + M;
  hipLaunchKernelGGL(k_dm_coords, gs, dim3(256), 0, st, order, kx, ky, kz, M, g, coords);
  hipLaunchKernelGGL(k_dm_bins, dim3((unsigned)nblocks(nbins + 1, 256)), dim3(256), 0, st, keys + M, M, nbins, start);
  hipLaunchKernelGGL(k_dm_count, dim3((unsigned)nblocks(ntiles + 1, 256)), dim3(256), 0, st, start, m, ntiles, items,
                     slots);
  DCF_HIP(hipGetLastError());
  DCF_HIP(hipcub::DeviceScan::ExclusiveSum(tmp, tb, items, ofs, ntiles + 1, st));
  DCF_HIP(hipcub::DeviceScan::ExclusiveSum(tmp, tb, slots, slot0, ntiles + 1, st));
  int32_t nitems = 0, nslots = 0;
  DCF_HIP(hipMemcpyAsync(&nitems, ofs + ntiles, sizeof(int32_t), hipMemcpyDeviceToHost, st));
  DCF_HIP(hipMemcpyAsync(&nslots, slot0 + ntiles, sizeof(int32_t), hipMemcpyDeviceToHost, st));
  DCF_HIP(hipStreamSynchronize(st));
  if (dm_sparse(g, M, nitems, p->iters)) return DM_GENERAL;
  mem.want(X, (int64_t)g.S[0] * g.S[1] * g.S[2]);
  mem.want(list, nitems);
  mem.want(heavy, nslots);  // at least two slots per split tile
  mem.want(part, (int64_t)nslots * DM_CELLS);
  DM_MEM(mem.take());
  hipLaunchKernelGGL(k_dm_items, dim3((unsigned)nblocks(ntiles, 256)), dim3(256), 0, st, items, ofs, slot0, ntiles, list);
  hipLaunchKernelGGL(k_dcf_fill, dim3(1), dim3(1), 0, st, reinterpret_cast<float *>(nheavy_d), (int64_t)1, 0.0f);
  int nheavy = 0;
  if (nslots > 0) {
    hipLaunchKernelGGL(k_dm_heavy, dim3((unsigned)nblocks(nitems, 256)), dim3(256), 0, st, list, nitems, heavy, nheavy_d);
    DCF_HIP(hipMemcpyAsync(&nheavy, nheavy_d, sizeof(int), hipMemcpyDeviceToHost, st));
    DCF_HIP(hipStreamSynchronize(st));
  }
  DCF_HIP(hipGetLastError());
  hipLaunchKernelGGL(k_dcf_count_reset, dim3(1), dim3(1), 0, st);
  if (p->iters > 0)  // zero the per-iteration sums (a double 0 is two float 0s)
    hipLaunchKernelGGL(k_dcf_fill, dim3(1), dim3(256), 0, st, reinterpret_cast<float *>(dsum), (int64_t)2 * p->iters, 0.0f);
  for (int it = 0; it < p->iters; it++) {
    if (nitems > 0)
      hipLaunchKernelGGL(k_dm_scatter, dim3((unsigned)nblocks(nitems, 4)), dim3(256), lds, st, X, part, coords, start,
                         list, nitems, g, m, tab);
    if (nheavy > 0) hipLaunchKernelGGL(k_dm_sum, dim3(nheavy), dim3(DM_CELLS), 0, st, X, part, heavy, g, m);
    hipLaunchKernelGGL(k_dm_gather_update, gs, dim3(256), lds, st, X, coords, M, g, tab, sums ? dsum + it : nullptr);
    DCF_HIP(hipGetLastError());
  }
  hipLaunchKernelGGL(k_dm_unsort, gs, dim3(256), 0, st, order, coords, M, kw);
  hipLaunchKernelGGL(k_dcf_finish, gs, dim3(256), 0, st, kw, kx, ky, kz, M, g);
  DCF_HIP(hipGetLastError());
  if (sums && p->iters > 0)
    DCF_HIP(hipMemcpyAsync(sums, dsum, sizeof(double) * p->iters, hipMemcpyDeviceToHost, st));
  DCF_HIP(hipStreamSynchronize(st));  // the scratch is freed on return
  return MRN_OK;
}

}  // namespace
}  // namespace mrn

using namespace mrn;

extern "C" {

void mrn_dcf_params_default(mrn_dcf_params *p) {
  if (!p) return;
  std::memset(p, 0, sizeof(*p));
  p->iters = 20;
  p->dwin = 2.1f;
  p->scale = 1.0f;
  p->overgrid = 2.1f;
  p->acc = 1.0f;
  p->kernel = MRN_DCF_POLY;
}

int mrn_dcf_parse_args(mrn_dcf_params *p, int argc, const char **argv) {
  if (!p || (argc > 0 && !argv)) return MRN_EINVAL;
  for (int i = 0; i < argc; i++) {
    const char *s = argv[i];
    const bool has = i + 1 < argc;
    if (!strcmp(s, "-dcf_iter")) {
      if (!has) return MRN_EINVAL;
      p->iters = atoi(argv[++i]);
    } else if (!strcmp(s, "-dcf_dwin") || !strcmp(s, "-dcf_scale") || !strcmp(s, "-dcf_overgrid") ||
               !strcmp(s, "-dcf_acc")) {
      if (!has) return MRN_EINVAL;
      const float v = (float)atof(argv[++i]);
      if (!strcmp(s, "-dcf_dwin")) p->dwin = v;
      else if (!strcmp(s, "-dcf_scale")) p->scale = v;
      else if (!strcmp(s, "-dcf_overgrid")) p->overgrid = v;
      else p->acc = v;
    }
  }
  return MRN_OK;
}

int mrn_dcf_grid_size(const mrn_dcf_params *p, int32_t S[3]) {
  if (!p || !S) return MRN_EINVAL;
  int s[3];
  grid_size(p, s);
  for (int a = 0; a < 3; a++) S[a] = s[a];
  return MRN_OK;
}

int mrn_dcf_last_atomics(int64_t *count) {
  if (!count) return MRN_EINVAL;
  unsigned long long v = 0;
  const hipError_t e = hipMemcpyFromSymbol(&v, HIP_SYMBOL(g_dcf_atomics), sizeof(v), 0, hipMemcpyDeviceToHost);
  if (e != hipSuccess) return dcf_fail(MRN_EHIP, hipGetErrorString(e));
  *count = (int64_t)v;
  return MRN_OK;
}

int mrn_dcf_calc(const mrn_dcf_params *p, int64_t M, const float *kx, const float *ky, const float *kz,
                 float *kw, double *sums, void *stream) {
  g_free_err.clear();
  if (!p) return dcf_fail(MRN_EINVAL, "null parameters");
  if (M < 0 || (M > 0 && (!kx || !ky || !kz || !kw))) return dcf_fail(MRN_EINVAL, "sample arrays");
  if (p->N[0] < 1 || p->N[1] < 1 || p->N[2] < 1) return dcf_fail(MRN_EINVAL, "image size");
  if (p->iters < 0) return dcf_fail(MRN_EINVAL, "dcf_iter < 0");
  if (!(p->dwin > 0.0f) || !(p->overgrid > 0.0f) || !std::isfinite(p->scale) || !std::isfinite(p->acc))
    return dcf_fail(MRN_EINVAL, "dcf_dwin and dcf_overgrid must be positive, dcf_scale and dcf_acc finite");
  if (p->kernel != MRN_DCF_POLY && p->kernel != MRN_DCF_POLY2) return dcf_fail(MRN_EINVAL, "dcf kernel");
  const int len = dcf_table(p->dwin, p->kernel, nullptr);
  if (len > DCF_MAX_TABLE) return dcf_fail(MRN_EUNSUPPORTED, "dcf_dwin too large for the kernel table");
  DcfGeom g;
  grid_size(p, g.S);
  for (int a = 0; a < 3; a++) {
    if (g.S[a] < 1) return dcf_fail(MRN_EINVAL, "grid size");
    g.c[a] = (float)(g.S[a] / 2);
  }
  g.gx = p->overgrid;
  g.dwin = p->dwin;
  g.scale = p->scale;
  g.acc = p->acc;
  g.len = len;
  if (M == 0) return MRN_OK;
  if (M > 0x7fffffffll) return dcf_fail(MRN_EUNSUPPORTED, "more than 2^31 - 1 samples");
  hipStream_t st = (hipStream_t)stream;
  const int64_t nS = (int64_t)g.S[0] * g.S[1] * g.S[2];
  float *tab_h = new float[len];
  dcf_table(p->dwin, p->kernel, tab_h);
  DmGeom m;
  if (dm_iters(p->iters, M) && dm_fits(g, m)) {
    m.item = dm_item(M);
    const int rc = dm_calc(p, g, m, M, kx, ky, kz, kw, sums, tab_h, st);
    if (rc != DM_GENERAL) {
      delete[] tab_h;
      return rc;
    }
  }
  float *X = nullptr, *tab = nullptr, *srt = nullptr;  // srt: sorted kx, ky, kz, kw
  uint32_t *keys = nullptr, *perm = nullptr;           // [2][M] each
  void *tmp = nullptr;
  size_t tb = 0;
  double *dsum = nullptr;
  int rc = MRN_OK;
  auto run = [&]() -> int {
    DCF_HIP(hipMalloc(&X, sizeof(float) * nS));
    DCF_HIP(hipMalloc(&tab, sizeof(float) * len));
    DCF_HIP(hipMalloc(&dsum, sizeof(double) * (p->iters > 0 ? p->iters : 1)));
    DCF_HIP(hipMemcpyAsync(tab, tab_h, sizeof(float) * len, hipMemcpyHostToDevice, st));
    const size_t lds = sizeof(float) * len;
    const size_t lds_box = sizeof(double) * DCF_BOX + lds;
    static const hipError_t box_attr = hipFuncSetAttribute((const void *)k_dcf_scatter_box,
                                                           hipFuncAttributeMaxDynamicSharedMemorySize,
                                                           (int)(sizeof(double) * DCF_BOX + sizeof(float) * DCF_MAX_TABLE));
    DCF_HIP(box_attr);
    const int fillb = 4096;
    const dim3 gs((unsigned)nblocks(M, 256));
    // brick order
    DCF_HIP(hipMalloc(&keys, sizeof(uint32_t) * 2 * M));
    DCF_HIP(hipMalloc(&perm, sizeof(uint32_t) * 2 * M));
    DCF_HIP(hipMalloc(&srt, sizeof(float) * 4 * M));
    hipLaunchKernelGGL(k_dcf_keys, gs, dim3(256), 0, st, kx, ky, kz, M, g, keys, perm);
    DCF_HIP(hipGetLastError());
    const uint64_t nkeys = 8ull * (uint64_t)((g.S[0] + DCF_BRICK - 1) / DCF_BRICK) * ((g.S[1] + DCF_BRICK - 1) / DCF_BRICK) *
                           ((g.S[2] + DCF_BRICK - 1) / DCF_BRICK);
    int bits = 1;
    while (bits < 32 && (1ull << bits) < nkeys) bits++;
    DCF_HIP(hipcub::DeviceRadixSort::SortPairs(nullptr, tb, keys, keys + M, perm, perm + M, (int)M, 0, bits, st));
    DCF_HIP(hipMalloc(&tmp, tb));
    DCF_HIP(hipcub::DeviceRadixSort::SortPairs(tmp, tb, keys, keys + M, perm, perm + M, (int)M, 0, bits, st));
    const uint32_t *order = perm + M;
    float *sx = srt, *sy = srt + M, *sz = srt + 2 * M, *sw = srt + 3 * M;
    hipLaunchKernelGGL(k_dcf_gather3, gs, dim3(256), 0, st, order, kx, ky, kz, M, sx, sy, sz);
    hipLaunchKernelGGL(k_dcf_fill, dim3(fillb), dim3(256), 0, st, sw, M, 1.0f);
    DCF_HIP(hipGetLastError());
    hipLaunchKernelGGL(k_dcf_count_reset, dim3(1), dim3(1), 0, st);
    if (p->iters > 0) {
      // zero the per-iteration sums (a double 0 is two float 0s)
      hipLaunchKernelGGL(k_dcf_fill, dim3(1), dim3(256), 0, st, reinterpret_cast<float *>(dsum),
                         (int64_t)2 * p->iters, 0.0f);
      DCF_HIP(hipGetLastError());
    }
    for (int it = 0; it < p->iters; it++) {
      hipLaunchKernelGGL(k_dcf_fill, dim3(fillb), dim3(256), 0, st, X, nS, 0.0f);
      hipLaunchKernelGGL(k_dcf_scatter_box, gs, dim3(256), lds_box, st, X, sw, sx, sy, sz, M, g, tab);
      hipLaunchKernelGGL(k_dcf_gather_update, gs, dim3(256), lds, st, X, sw, sx, sy, sz, M, g, tab,
                         sums ? dsum + it : nullptr);
      DCF_HIP(hipGetLastError());
    }
    hipLaunchKernelGGL(k_dcf_finish, gs, dim3(256), 0, st, sw, sx, sy, sz, M, g);
    hipLaunchKernelGGL(k_dcf_unsort, gs, dim3(256), 0, st, order, sw, M, kw);
    DCF_HIP(hipGetLastError());
    if (sums && p->iters > 0)
      DCF_HIP(hipMemcpyAsync(sums, dsum, sizeof(double) * p->iters, hipMemcpyDeviceToHost, st));
    DCF_HIP(hipStreamSynchronize(st));  // the scratch grid is freed below
    return MRN_OK;
  };
  rc = run();
  if (rc != MRN_OK) hipStreamSynchronize(st);
  hipFree(X);
  hipFree(tab);
  hipFree(dsum);
  hipFree(keys);
  hipFree(perm);
  hipFree(srt);
  hipFree(tmp);
  delete[] tab_h;
  return rc;
}

}  // extern "C"
