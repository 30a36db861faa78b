// L1 wavelet proximal step of the FISTA loop, on the device.
//
// Follows RECON::L1_threshold (recon_lib.cpp:2416-2527) with its default
// spatial wavelet and fraction threshold, without phase rotation or temporal
// transforms: for each cycle spin, a 3-D periodic wavelet transform of every
// frame (WAVELET3D::forward3D, wavelet3D.cpp:563-594), the fraction threshold
// over all frames on the first spin, scaled by 1/spins
// (THRESHOLD::update_threshold / get_threshold, threshold.cpp:193-380), the
// complex soft threshold (thresholding, threshold.cpp:766-800), and the
// inverse transform (backward3D, wavelet3D.cpp:596-631).
//
// The wavelet is the 4-tap Daubechies pair of the reference's default
// (wavelet3D.cpp:143-190), computed from its closed form.  A line transform
// stages FL lines in LDS and writes the result back in place; the inverse is
// evaluated in gather form (each output sums its two contributing taps).
// The fraction threshold runs entirely on the device: a min/max pass, then 11
// rounds, each of which counts below the bisection's next 63 candidate values
// and replays up to 6 bisection steps, a no-op once the bracket has converged,
// so the whole step can be captured in a hipGraph.  |c| is evaluated as sqrt in
// double rounded to float, so the counts and the threshold do not depend on the
// order of operations.
#include <algorithm>
#include <cmath>
#include <cstring>

#include "mrn_internal.hpp"

namespace mrn {

#define WL_LINES 16

struct D4 {
  float lpf[4], hpf[4], slpf[4], shpf[4];
};

static D4 d4_filters() {
  const double r3 = std::sqrt(3.0), n = 4.0 * std::sqrt(2.0);
  const double h0 = (1 + r3) / n, h1 = (3 + r3) / n, h2 = (3 - r3) / n, h3 = (1 - r3) / n;
  const double lp[4] = {h3, h2, h1, h0}, hp[4] = {-h0, h1, -h2, h3};
  const double sl[4] = {h0, h1, h2, h3}, shp[4] = {h3, -h2, h1, -h0};
  D4 f;
  for (int q = 0; q < 4; q++) {
    f.lpf[q] = (float)lp[q];
    f.hpf[q] = (float)hp[q];
    f.slpf[q] = (float)sl[q];
    f.shpf[q] = (float)shp[q];
  }
  return f;
}

__device__ __forceinline__ int wmod(int i, int n) {
  const int r = i % n;
  return r < 0 ? r + n : r;
}

// In-place one-level transform (INV = 0 analysis, 1 synthesis) of the lines
// along `axis` of the sub-block [0,s0) x [0,s1) x [0,s2) of frame blockIdx.y.
// The shift of the axis is read from sh[axis] (device memory; 0..3).  No
// integer division per element: the workgroup's 16 line bases are computed
// once, the x-axis walk steps by a precomputed quotient and remainder, and
// the periodic index wraps with one add or subtract for lines of 4 or more
// points (the indices reach [-3, pts + 2]).  Launched with 256 threads.
template <int INV>
__global__ __launch_bounds__(256) void k_wave_lines(float2 *X, int N0, int N1, int s0, int s1, int s2,
                                                    int axis, const int *__restrict__ sh, D4 f,
                                                    int64_t frame_stride) {
  extern __shared__ float2 wbuf[];  // [WL_LINES][pts]
  __shared__ int64_t s_base[WL_LINES];
  const int sz[3] = {s0, s1, s2};
  const int pts = sz[axis], h = pts >> 1;
  const int b = axis == 0 ? 1 : 0, c = axis == 2 ? 1 : 2;
  const int64_t st[3] = {1, N0, (int64_t)N0 * N1};
  const int64_t sa = st[axis];
  const int nlines = sz[b] * sz[c];
  const int l0 = blockIdx.x * WL_LINES;
  float2 *Xf = X + (int64_t)blockIdx.y * frame_stride;
  const int shift = sh[axis];
  const int tot = WL_LINES * pts;
  if (threadIdx.x < WL_LINES) {
    const int L = l0 + (int)threadIdx.x, u = L % sz[b], v = L / sz[b];
    s_base[threadIdx.x] = (int64_t)u * st[b] + (int64_t)v * st[c];
  }
  // element e = threadIdx.x + k * blockDim.x as (line, point): an x line is
  // contiguous (ln = e / pts, p = e % pts); along y and z the 16 lines of a
  // point are neighbouring x (or y) cells (p = e / 16, ln = e % 16)
  const int dq = (int)blockDim.x / pts, dr = (int)blockDim.x - dq * pts;
  const int q0 = (int)threadIdx.x / pts, r0 = (int)threadIdx.x - q0 * pts;
  auto walk = [&](auto &&fn) {
    if (axis == 0) {
      int ln = q0, p = r0;
      for (int e = threadIdx.x; e < tot; e += blockDim.x) {
        fn(ln, p);
        p += dr;
        ln += dq;
        if (p >= pts) {
          p -= pts;
          ln++;
        }
      }
    } else {
      const int ln = (int)threadIdx.x % WL_LINES;
      for (int p = (int)threadIdx.x / WL_LINES; p < pts; p += (int)blockDim.x / WL_LINES) fn(ln, p);
    }
  };
  const bool near = pts >= 4;
  auto wrap = [&](int i) { return near ? (i < 0 ? i + pts : (i >= pts ? i - pts : i)) : wmod(i, pts); };
  __syncthreads();
  walk([&](int ln, int p) {
    if (l0 + ln < nlines) wbuf[ln * pts + p] = Xf[s_base[ln] + p * sa];
  });
  __syncthreads();
  walk([&](int ln, int p) {
    if (l0 + ln >= nlines) return;
    const float2 *in = wbuf + ln * pts;
    float2 o = make_float2(0.f, 0.f);
    if (!INV) {  // wave1D: out[pos] = sum lpf * in, out[pos + h] = sum hpf * in
      const bool lo = p < h;
      const int pos = lo ? p : p - h;
#pragma unroll
      for (int fp = 0; fp < 4; fp++) {
        const float2 v = in[wrap(2 * pos - fp + shift)];
        const float w = lo ? f.lpf[fp] : f.hpf[fp];
        o.x += w * v.x;
        o.y += w * v.y;
      }
    } else {  // iwave1D: in[pos] and in[pos + h] reach out[2 pos + fp - 3 + shift]
#pragma unroll
      for (int fp = 0; fp < 4; fp++) {
        const int t = p - fp + 3 - shift;
        if (t & 1) continue;
        const int pos = wrap(t) >> 1;
        const float2 a = in[pos], d = in[pos + h];
        o.x += a.x * f.slpf[fp];
        o.y += a.y * f.slpf[fp];
        o.x += d.x * f.shpf[fp];
        o.y += d.y * f.shpf[fp];
      }
    }
    Xf[s_base[ln] + p * sa] = o;
  });
}

// ------------------------------------------------------- one level, 3 axes
// A level of a 3-D transform, all three axes in one pass from one image to
// another: 7/8 of a transform's traffic is in the first level, which as three
// line passes reads and writes the image three times, and a deeper level's line
// passes are short launches that wait for each other.  A workgroup loads the
// region that its outputs reach into LDS and transforms it along x, y, z
// (synthesis: z, y, x) in place, each thread holding its outputs in registers
// across the barrier; the products and their order are those of k_wave_lines,
// so the results are the same bits.  The detail octants live in the second
// image, the low-pass octant goes to a compact image of its own that the next
// level reads.  The synthesis applies the soft threshold as it loads the seven
// detail octants (the deepest level: all eight).
// 256 x 256 x 192, 4 levels, 4 spins, ms for the step: 3.10 with line passes only,
// 2.01 with the first level here, 1.00 with all levels and the counting below.
// us at the first / second level: analysis 58 / 13, synthesis 72 / 17 (copying the
// image at the card's rate: 42).
#define W3_THREADS 512
#define W3_PX 16  // analysis: output positions of a workgroup (a low- and a high-pass value each per axis)
#define W3_PY 8
#define W3_PZ 4

// (float)sqrt(d), d = x^2 + y^2 in double.  The double square root is some 40
// instructions; here one Newton step on the FP32 root c, c + (d - c^2) / 2c with
// the difference in double, is within 2^-43 of it, which rounds to the same
// float unless it lies within 2^-40 of a point half way between two: those, and
// d outside [2^-80, 2^120], take the double root.
__device__ __forceinline__ float cabs_rn(float2 v) {
  const double d = (double)v.x * v.x + (double)v.y * v.y;
  const float a = (float)d, c = __builtin_amdgcn_sqrtf(a);
  const float r = (float)fma(-(double)c, (double)c, d);
  double s = (double)c + (double)(r * (0.5f * __builtin_amdgcn_rcpf(c)));
  const unsigned low = (unsigned)__double_as_longlong(s) & 0x1fffffffu;  // below the float's last place
  if (!(a >= 0x1p-80f && a <= 0x1p120f) || low - (0x10000000u - 4096u) < 8192u) s = sqrt(d);
  return (float)s;
}
__device__ __forceinline__ float2 soft(float2 v, float thr) {
  const float cc = cabs_rn(v);
  if (cc <= thr) return make_float2(0.f, 0.f);
  const float f = 1.0f - thr / cc;
  return make_float2(v.x * f, v.y * f);
}

// out[(line, pos)] = the filter pair at `pos` over in[base + (2 pos + 3 - fp) st], fp = 0..3
__device__ __forceinline__ void wave_pair(const float2 *in, int at, int st, const D4 &f, float2 &lo, float2 &hi) {
  lo = hi = make_float2(0.f, 0.f);
#pragma unroll
  for (int fp = 0; fp < 4; fp++) {
    const float2 v = in[at + (3 - fp) * st];
    lo.x += f.lpf[fp] * v.x;
    lo.y += f.lpf[fp] * v.y;
    hi.x += f.hpf[fp] * v.x;
    hi.y += f.hpf[fp] * v.y;
  }
}

// An image of the transform: point (x, y, z) of frame fr at p[fr * frame + z * plane + y * row + x]
struct WImg {
  float2 *p;
  int row;
  int64_t plane, frame;
};

// One analysis level of the s0 x s1 x s2 block of X: details to T, low-pass
// octant to L (may be T).
__global__ __launch_bounds__(W3_THREADS) void k_wave3_fwd(WImg T, WImg L, WImg X, int s0, int s1, int s2, int nz,
                                                          const int *__restrict__ sh, D4 f) {
  constexpr int RX = 2 * W3_PX + 2, RY = 2 * W3_PY + 2, RZ = 2 * W3_PZ + 2;
  __shared__ float2 A[RX * RY * RZ];
  __shared__ int s_at[RX + RY + RZ];
  const int fr = blockIdx.z / nz;
  const int p0[3] = {(int)blockIdx.x * W3_PX, (int)blockIdx.y * W3_PY, (int)(blockIdx.z - fr * nz) * W3_PZ};
  const float2 *__restrict__ Xf = X.p + fr * X.frame;
  float2 *__restrict__ Tf = T.p + fr * T.frame;
  float2 *__restrict__ Lf = L.p + fr * L.frame;
  // cell (x, y, z) of the region: image point 2 p0 + shift - 3 + (x, y, z)
  const int ox = 2 * p0[0] + sh[0] - 3, oy = 2 * p0[1] + sh[1] - 3, oz = 2 * p0[2] + sh[2] - 3;
  // (the periodic index once per row, column and plane)
  const int a = threadIdx.x;
  if (a < RX) s_at[a] = wmod(ox + a, s0);
  else if (a < RX + RY) s_at[a] = wmod(oy + a - RX, s1);
  else if (a < RX + RY + RZ) s_at[a] = wmod(oz + a - RX - RY, s2);
  __syncthreads();
  for (int q = threadIdx.x; q < RX * RY * RZ; q += W3_THREADS) {
    const int x = q % RX, yz = q / RX, y = yz % RY, z = yz / RY;
    A[q] = Xf[s_at[RX + RY + z] * X.plane + (int64_t)s_at[RX + y] * X.row + s_at[x]];
  }
  __syncthreads();
  {  // x: RY * RZ lines of W3_PX positions
    constexpr int TOT = RY * RZ * W3_PX, PER = (TOT + W3_THREADS - 1) / W3_THREADS;
    float2 lo[PER], hi[PER];
#pragma unroll
    for (int k = 0; k < PER; k++) {
      const int q = threadIdx.x + k * W3_THREADS, p = q % W3_PX, ln = q / W3_PX;
      if (q < TOT) wave_pair(A, ln * RX + 2 * p, 1, f, lo[k], hi[k]);
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < PER; k++) {
      const int q = threadIdx.x + k * W3_THREADS, p = q % W3_PX, ln = q / W3_PX;
      if (q < TOT) {
        A[ln * RX + p] = lo[k];
        A[ln * RX + W3_PX + p] = hi[k];
      }
    }
    __syncthreads();
  }
  {  // y: 2 W3_PX x RZ lines of W3_PY positions, x fastest
    constexpr int NX = 2 * W3_PX, TOT = NX * RZ * W3_PY, PER = (TOT + W3_THREADS - 1) / W3_THREADS;
    float2 lo[PER], hi[PER];
#pragma unroll
    for (int k = 0; k < PER; k++) {
      const int q = threadIdx.x + k * W3_THREADS, x = q % NX, p = (q / NX) % W3_PY, z = q / (NX * W3_PY);
      if (q < TOT) wave_pair(A, (z * RY + 2 * p) * RX + x, RX, f, lo[k], hi[k]);
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < PER; k++) {
      const int q = threadIdx.x + k * W3_THREADS, x = q % NX, p = (q / NX) % W3_PY, z = q / (NX * W3_PY);
      if (q < TOT) {
        A[(z * RY + p) * RX + x] = lo[k];
        A[(z * RY + W3_PY + p) * RX + x] = hi[k];
      }
    }
    __syncthreads();
  }
  // z, straight to the images
  constexpr int NX = 2 * W3_PX, NY = 2 * W3_PY, TOT = NX * NY * W3_PZ;
  const int h0 = s0 >> 1, h1 = s1 >> 1, h2 = s2 >> 1;
  for (int q = threadIdx.x; q < TOT; q += W3_THREADS) {
    const int x = q % NX, y = (q / NX) % NY, p = q / (NX * NY);
    const int px = p0[0] + x % W3_PX, py = p0[1] + y % W3_PY, pz = p0[2] + p;
    if (px >= h0 || py >= h1 || pz >= h2) continue;
    float2 lo, hi;
    wave_pair(A, (2 * p * RY + y) * RX + x, RY * RX, f, lo, hi);
    float2 *dst = Tf + (int64_t)(py + (y < W3_PY ? 0 : h1)) * T.row + px + (x < W3_PX ? 0 : h0);
    if (x < W3_PX && y < W3_PY)
      Lf[pz * L.plane + (int64_t)py * L.row + px] = lo;
    else
      dst[pz * T.plane] = lo;
    dst[(pz + h2) * T.plane] = hi;
  }
}

// Synthesis.  Points p and p + 1, p - shift odd, are sums over the same two
// positions P = (p + 3 - shift) / 2 and P - 1, so a thread makes both from one
// load of the four values.  A workgroup makes W3_IX x W3_IY x W3_IZ points
// beginning at such a p on each axis (wrapping at the end), from n / 2 + 1
// positions per axis, low-pass then high-pass values.
#define W3_IX 32
#define W3_IY 16
#define W3_IZ 8
template <int H>  // distance of the high-pass value
__device__ __forceinline__ void wave_points(const float2 *in, int st, const D4 &f, float2 &o0, float2 &o1) {
  const float2 a1 = in[0], d1 = in[H], a0 = in[st], d0 = in[st + H];  // positions P - 1, P
  o0 = o1 = make_float2(0.f, 0.f);
  o0.x += a0.x * f.slpf[0];
  o0.y += a0.y * f.slpf[0];
  o0.x += d0.x * f.shpf[0];
  o0.y += d0.y * f.shpf[0];
  o0.x += a1.x * f.slpf[2];
  o0.y += a1.y * f.slpf[2];
  o0.x += d1.x * f.shpf[2];
  o0.y += d1.y * f.shpf[2];
  o1.x += a0.x * f.slpf[1];
  o1.y += a0.y * f.slpf[1];
  o1.x += d0.x * f.shpf[1];
  o1.y += d0.y * f.shpf[1];
  o1.x += a1.x * f.slpf[3];
  o1.y += a1.y * f.slpf[3];
  o1.x += d1.x * f.shpf[3];
  o1.y += d1.y * f.shpf[3];
}

// One synthesis level, T's details and L's low-pass octant to the s0 x s1 x s2
// block of X; all: threshold the low-pass octant too.
__global__ __launch_bounds__(W3_THREADS) void k_wave3_inv(WImg X, WImg T, WImg L, int s0, int s1, int s2, int nz,
                                                          const int *__restrict__ sh, D4 f,
                                                          const float *__restrict__ thr_p, int all) {
  constexpr int CX = W3_IX / 2 + 1, CY = W3_IY / 2 + 1, CZ = W3_IZ / 2 + 1;  // positions
  constexpr int RX = 2 * CX, RY = 2 * CY, RZ = 2 * CZ;
  __shared__ float2 A[RX * RY * RZ];  // [RZ][RY][RX]
  __shared__ int s_at[RX + RY + RZ];
  const int fr = blockIdx.z / nz;
  const int p0[3] = {(int)blockIdx.x * W3_IX, (int)blockIdx.y * W3_IY, (int)(blockIdx.z - fr * nz) * W3_IZ};
  const float2 *__restrict__ Tf = T.p + fr * T.frame;
  const float2 *__restrict__ Lf = L.p + fr * L.frame;
  float2 *__restrict__ Xf = X.p + fr * X.frame;
  const int h0 = s0 >> 1, h1 = s1 >> 1, h2 = s2 >> 1;
  // first point p0 + o, first position P - 1 of it
  const int o0 = (sh[0] + 1) & 1, o1 = (sh[1] + 1) & 1, o2 = (sh[2] + 1) & 1;
  const int b0 = ((p0[0] + o0 + 3 - sh[0]) >> 1) - 1, b1 = ((p0[1] + o1 + 3 - sh[1]) >> 1) - 1,
            b2 = ((p0[2] + o2 + 3 - sh[2]) >> 1) - 1;
  const float thr = *thr_p;
  const int a = threadIdx.x;
  if (a < RX) s_at[a] = a < CX ? wmod(b0 + a, h0) : h0 + wmod(b0 + a - CX, h0);
  else if (a < RX + RY) s_at[a] = a - RX < CY ? wmod(b1 + a - RX, h1) : h1 + wmod(b1 + a - RX - CY, h1);
  else if (a < RX + RY + RZ)
    s_at[a] = a - RX - RY < CZ ? wmod(b2 + a - RX - RY, h2) : h2 + wmod(b2 + a - RX - RY - CZ, h2);
  __syncthreads();
  for (int q = threadIdx.x; q < RX * RY * RZ; q += W3_THREADS) {
    const int x = q % RX, yz = q / RX, y = yz % RY, z = yz / RY;
    const bool det = x >= CX || y >= CY || z >= CZ;
    const int px = s_at[x], py = s_at[RX + y], pz = s_at[RX + RY + z];
    const float2 v = det ? Tf[pz * T.plane + (int64_t)py * T.row + px] : Lf[pz * L.plane + (int64_t)py * L.row + px];
    A[q] = det || all ? soft(v, thr) : v;
  }
  __syncthreads();
  {  // z: [RZ][RY][RX] -> [W3_IZ][RY][RX]
    constexpr int TOT = RX * RY * W3_IZ / 2, PER = (TOT + W3_THREADS - 1) / W3_THREADS;
    float2 u[PER], v[PER];
#pragma unroll
    for (int k = 0; k < PER; k++) {
      const int q = threadIdx.x + k * W3_THREADS, p = q / (RX * RY), xy = q % (RX * RY);
      if (q < TOT) wave_points<CZ * RX * RY>(A + p * RX * RY + xy, RX * RY, f, u[k], v[k]);
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < PER; k++) {
      const int q = threadIdx.x + k * W3_THREADS, p = q / (RX * RY), xy = q % (RX * RY);
      if (q < TOT) {
        A[2 * p * RX * RY + xy] = u[k];
        A[(2 * p + 1) * RX * RY + xy] = v[k];
      }
    }
    __syncthreads();
  }
  {  // y: -> [W3_IZ][W3_IY][RX]
    constexpr int TOT = RX * W3_IY / 2 * W3_IZ, PER = (TOT + W3_THREADS - 1) / W3_THREADS;
    float2 u[PER], v[PER];
#pragma unroll
    for (int k = 0; k < PER; k++) {
      const int q = threadIdx.x + k * W3_THREADS, x = q % RX, p = (q / RX) % (W3_IY / 2), z = q / (RX * W3_IY / 2);
      if (q < TOT) wave_points<CY * RX>(A + (z * RY + p) * RX + x, RX, f, u[k], v[k]);
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < PER; k++) {
      const int q = threadIdx.x + k * W3_THREADS, x = q % RX, p = (q / RX) % (W3_IY / 2), z = q / (RX * W3_IY / 2);
      if (q < TOT) {
        A[(z * W3_IY + 2 * p) * RX + x] = u[k];
        A[(z * W3_IY + 2 * p + 1) * RX + x] = v[k];
      }
    }
    __syncthreads();
  }
  // x, straight to the image
  constexpr int HX = W3_IX / 2;
  for (int q = threadIdx.x; q < HX * W3_IY * W3_IZ; q += W3_THREADS) {
    const int p = q % HX, y = (q / HX) % W3_IY, z = q / (HX * W3_IY);
    if (p0[0] + 2 * p >= s0 || p0[1] + y >= s1 || p0[2] + z >= s2) continue;
    float2 u, v;
    wave_points<CX>(A + (z * W3_IY + y) * RX + p, 1, f, u, v);
    const int x0 = p0[0] + o0 + 2 * p, x1 = x0 + 1;  // s0 is even: only x1 can reach it
    const int py = p0[1] + o1 + y, pz = p0[2] + o2 + z;
    float2 *dst = Xf + (pz < s2 ? pz : pz - s2) * X.plane + (int64_t)(py < s1 ? py : py - s1) * X.row;
    dst[x0] = u;
    dst[x1 < s0 ? x1 : x1 - s0] = v;
  }
}

// ------------------------------------------------------------ threshold
#define THR_DEPTH 6                         // bisection steps per counting pass
#define THR_NODES ((1 << THR_DEPTH) - 1)    // candidate values per pass
#define THR_THREADS 512
struct ThrBracket {
  float value, max_t, min_t;
};
struct ThrState {
  unsigned int umin, umax;  // bit patterns of min / max |c| (non-negative floats)
  float thr;
  ThrBracket b;
  int iter, done;
  long long target, accuracy;
  unsigned int ticket;            // workgroups of this pass that have added their counts
  int rank[THR_NODES];            // node k's candidate is sorted[rank[k]]
  float sorted[THR_NODES];        // ascending; a NaN stands first, as -inf
  unsigned long long hist[THR_NODES + 1];  // hist[q]: sorted[q - 1] <= |c| < sorted[q]
};

// |c| of the counting passes: kept by the min/max pass, or from the coefficients
__device__ __forceinline__ float mag_of(const float *m, int64_t i) { return m[i]; }
__device__ __forceinline__ float mag_of(const float2 *x, int64_t i) { return cabs_rn(x[i]); }

// The next THR_DEPTH values the bisection can query, breadth first: node k
// (value v, bracket [lo, hi]) has children 2k + 1 (count > target: max = v)
// and 2k + 2 (min = v), each at 0.5 * (max + min) as the sequential step
// computes it, so that a pass counts exactly the values the sequence visits.
// They need not ascend from left to right: the first value may lie above the
// first bracket.
__device__ __forceinline__ float thr_node(const ThrBracket &s, int k) {
  float lo = s.min_t, hi = s.max_t, v = s.value;
  const int path = k + 1;
  for (int b = 30 - __builtin_clz(path); b >= 0; b--) {
    if (path >> b & 1)
      lo = v;
    else
      hi = v;
    v = 0.5f * (hi + lo);
  }
  return v;
}

// The last workgroup of a pass, all of its threads: candidates of the next pass
// in ascending order (equal ones by node), counts cleared.
__device__ __forceinline__ void thr_next(ThrState *s, const ThrBracket &b) {
  __shared__ float s_v[THR_NODES];
  const int k = threadIdx.x;
  float v = 0.f;
  if (k < THR_NODES) {
    v = thr_node(b, k);
    if (v != v) v = -INFINITY;  // counts nothing either way
    s_v[k] = v;
  }
  __syncthreads();
  if (k < THR_NODES) {
    int r = 0;
    for (int j = 0; j < THR_NODES; j++) r += s_v[j] < v || (s_v[j] == v && j < k) ? 1 : 0;
    s->rank[k] = r;
    s->sorted[r] = v;
  }
  if (k <= THR_NODES) s->hist[k] = 0ull;
  if (k == 0) s->ticket = 0u;
}

// threshold = scale * value; optionally logged per FISTA iteration
__device__ __forceinline__ void thr_finish(ThrState *s, float value, float scale, double *log, const int *counter, int cap) {
  const float thr = scale * value;
  s->thr = thr;
  if (log) {
    const int it = counter ? *counter - 1 : 0;
    if (it >= 0 && it < cap) log[it] = (double)thr;
  }
}

// True in the workgroup that is the last of the grid to come here.  `wait` is
// false and computed from what the thread's device-scope atomics returned, so
// they have been performed before the ticket is drawn; the last workgroup reads
// their targets with device-scope loads.  (A fence here would write back the L2,
// once per workgroup.)
__device__ __forceinline__ bool thr_last(ThrState *s, bool wait) {
  __shared__ int s_last;
  const int w = __syncthreads_or(wait ? 1 : 0);
  if (threadIdx.x == 0)
    s_last = __hip_atomic_fetch_add(&s->ticket, w ? 0u : 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == gridDim.x - 1;
  __syncthreads();
  return s_last != 0;
}

__global__ void k_thr_reset(ThrState *s) {
  s->umin = 0x7f800000u;  // +inf
  s->umax = 0u;
  s->ticket = 0u;
}

// Smallest and largest |c|; mag (if given) keeps |c| for the counting passes.
// The last workgroup sets the bisection up (get_threshold, threshold.cpp:250-336).
__global__ __launch_bounds__(THR_THREADS) void k_thr_minmax(const float2 *__restrict__ X, float *__restrict__ mag,
                                                            int64_t n, ThrState *s, float fraction, float scale,
                                                            double *log, const int *counter, int cap) {
  float mn = INFINITY, mx = 0.0f;
  for (int64_t i = (int64_t)blockIdx.x * THR_THREADS + threadIdx.x; i < n; i += (int64_t)gridDim.x * THR_THREADS) {
    const float v = cabs_rn(X[i]);
    if (mag) mag[i] = v;
    mn = fminf(mn, v);
    mx = fmaxf(mx, v);
  }
  for (int o = 32; o > 0; o >>= 1) {
    mn = fminf(mn, __shfl_xor(mn, o));
    mx = fmaxf(mx, __shfl_xor(mx, o));
  }
  // one atomic pair per workgroup: atomics on one address serialise in L2
  __shared__ float s_mn[THR_THREADS / 64], s_mx[THR_THREADS / 64];
  if ((threadIdx.x & 63) == 0) {
    s_mn[threadIdx.x >> 6] = mn;
    s_mx[threadIdx.x >> 6] = mx;
  }
  __syncthreads();
  bool wait = false;
  if (threadIdx.x == 0) {
    for (int w = 1; w < THR_THREADS / 64; w++) {
      mn = fminf(mn, s_mn[w]);
      mx = fmaxf(mx, s_mx[w]);
    }
    const unsigned o0 = atomicMin(&s->umin, __float_as_uint(mn)), o1 = atomicMax(&s->umax, __float_as_uint(mx));
    wait = (o0 & o1) == 0xffffffffu;  // (no non-negative float)
  }
  if (!thr_last(s, wait)) return;
  __shared__ ThrBracket s_b;
  if (threadIdx.x == 0) {
    mx = __uint_as_float(__hip_atomic_load(&s->umax, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
    mn = __uint_as_float(__hip_atomic_load(&s->umin, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
    s->target = (long long)(fraction * (double)n);
    s->accuracy = (long long)(0.001 * (double)n);
    s_b.value = 0.5f * (mx - mn);
    s_b.max_t = fraction * mx;
    s_b.min_t = mn;
    s->iter = 0;
    int done = 0;
    if (s->target < 2) {
      s_b.value = 0.0f;
      done = 1;
    } else if (!(llabs(n - s->target) > s->accuracy)) {
      done = 1;
    }
    s->done = done;
    s->b = s_b;
    if (done) thr_finish(s, s_b.value, scale, log, counter, cap);
  }
  __syncthreads();
  thr_next(s, s_b);
}

// One counting pass and up to THR_DEPTH steps of threshold.cpp:250-380's
// bisection: the same values, counts and stopping rule as one step per pass.
// A thread looks its value up among the sorted candidates (LDS, 6 steps) and
// adds to its lane's column of a histogram, so no two lanes of a wave meet on an
// address; the last workgroup sums up and steps.  Against 15 candidates, each
// compared with every value, and |c| computed anew on each pass (its root in double):
// 12.6 M values, 82 us per pass of 4 steps before, 25 to 40 per pass of 6 now.
template <typename V>
__global__ __launch_bounds__(THR_THREADS) void k_thr_count(const V *__restrict__ X, int64_t n, ThrState *s, float scale,
                                                           double *log, const int *counter, int cap) {
  __shared__ unsigned int s_hist[(THR_NODES + 1) * 64];
  __shared__ float s_t[THR_NODES + 1];
  if (s->done) return;  // (uniform)
  for (int q = threadIdx.x; q < (THR_NODES + 1) * 64; q += THR_THREADS) s_hist[q] = 0u;
  if (threadIdx.x < THR_NODES) s_t[threadIdx.x] = s->sorted[threadIdx.x];
  __syncthreads();
  const int lane = threadIdx.x & 63;
  const int64_t step = (int64_t)gridDim.x * THR_THREADS;
  for (int64_t i0 = (int64_t)blockIdx.x * THR_THREADS + threadIdx.x; i0 < n; i0 += 4 * step) {
    float a[4];
    int q[4] = {0, 0, 0, 0};
#pragma unroll
    for (int u = 0; u < 4; u++) a[u] = i0 + u * step < n ? mag_of(X, i0 + u * step) : 0.f;
#pragma unroll
    for (int h = (THR_NODES + 1) / 2; h > 0; h >>= 1)
#pragma unroll
      for (int u = 0; u < 4; u++) q[u] += a[u] < s_t[q[u] + h - 1] ? 0 : h;  // q candidates are not above a (NaN: all)
#pragma unroll
    for (int u = 0; u < 4; u++)
      if (i0 + u * step < n) atomicAdd(&s_hist[q[u] * 64 + lane], 1u);
  }
  __syncthreads();
  bool wait = false;
  {  // 8 threads to a bin
    const int bin = threadIdx.x >> 3, g = threadIdx.x & 7;
    unsigned int c = 0u;
    for (int j = 0; j < 8; j++) c += s_hist[bin * 64 + ((g + bin) & 7) * 8 + j];
    for (int o = 4; o > 0; o >>= 1) c += __shfl_xor(c, o);
    if (g == 0 && c) wait = atomicAdd(&s->hist[bin], (unsigned long long)c) == ~0ull;
  }
  if (!thr_last(s, wait)) return;
  __shared__ long long s_c[THR_NODES + 1];
  __shared__ int s_rank[THR_NODES];
  __shared__ ThrBracket s_b;
  if (threadIdx.x < THR_NODES) s_rank[threadIdx.x] = s->rank[threadIdx.x];
  if (threadIdx.x <= THR_NODES) {  // one wave: s_c[q] = count(|c| < sorted[q])
    long long c = (long long)__hip_atomic_load(&s->hist[threadIdx.x], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    for (int o = 1; o < 64; o <<= 1) {
      const long long up = __shfl_up(c, o);
      if (lane >= o) c += up;
    }
    s_c[threadIdx.x] = c;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    ThrBracket b = s->b;
    const long long target = s->target, accuracy = s->accuracy;
    int iter = s->iter, done = 0, node = 0;
    for (int lvl = 0; lvl < THR_DEPTH; lvl++) {
      const long long found = s_c[s_rank[node]];
      iter++;
      if (!(llabs(found - target) > accuracy && iter < 64)) {
        done = 1;
        break;
      }
      if (found > target) {
        b.max_t = b.value;
        node = 2 * node + 1;
      } else {
        b.min_t = b.value;
        node = 2 * node + 2;
      }
      b.value = 0.5f * (b.max_t + b.min_t);
    }
    s->iter = iter;
    s->done = done;
    s->b = b;
    s_b = b;
    if (done) thr_finish(s, b.value, scale, log, counter, cap);
  }
  __syncthreads();
  thr_next(s, s_b);
}

// soft threshold of the sub-block [0, s0) x [0, s1) x [0, s2) of each frame
__global__ __launch_bounds__(256) void k_soft(float2 *X, int N0, int N1, int s0, int s1, int s2, int64_t frame_stride,
                                              int frames, const ThrState *__restrict__ s) {
  const float thr = s->thr;
  const int64_t n = (int64_t)s0 * s1 * s2;
  for (int fr = blockIdx.y; fr < frames; fr += gridDim.y) {  // (a grid holds 65535 of them)
    float2 *Xf = X + (int64_t)fr * frame_stride;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
      const int64_t yz = i / s0;
      float2 *v = Xf + ((yz / s1) * N1 + yz % s1) * N0 + i % s0;
      *v = soft(*v, thr);
    }
  }
}

// Cycle-spin shifts of FISTA iteration (*counter - 1): entries
// 3*spins*it .. 3*spins*(it+1) of the splitmix64 stream from `seed`, each
// (z >> 33) % 4 (the reference draws rand() % wN, wavelet3D.cpp:443-449).
__global__ void k_spin_shifts(int *sh, int count, unsigned long long seed, const int *counter) {
  const int q = threadIdx.x;
  if (q >= count) return;
  const long long it = counter ? (long long)(*counter - 1) : 0;
  unsigned long long z = seed + (unsigned long long)(it * count + q + 1) * 0x9E3779B97F4A7C15ull;
  z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
  z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
  z ^= z >> 31;
  sh[q] = (int)((z >> 33) % 4ull);
}

// ------------------------------------------------------------ host side
void wavelet_levels(const int N[3], const int req[3], int L[3]) {
  for (int a = 0; a < 3; a++) {
    int l = req[a] < 0 ? 0 : req[a];
    while (l > 0 && (N[a] % (1 << l)) != 0) l--;
    L[a] = l;
  }
}

int ensure_l1_state(mrn_op *op) {
  if (!op->dthr) MRN_HIP(op, hipMalloc(&op->dthr, sizeof(ThrState)));
  if (!op->dsh) MRN_HIP(op, hipMalloc(&op->dsh, sizeof(int) * 3 * MRN_MAX_SPINS));
  if (!op->dthr_log) MRN_HIP(op, hipMalloc(&op->dthr_log, sizeof(double) * MRN_TRACE_CAP));
  return MRN_OK;
}

static int wave_axis(mrn_op *op, float2 *X, int frames, const int s[3], int axis, const int *sh, bool inv,
                     hipStream_t st) {
  static const D4 f = d4_filters();
  const int *N = op->g.N;
  const int pts = s[axis];
  const int b = axis == 0 ? 1 : 0, c = axis == 2 ? 1 : 2;
  const int nlines = s[b] * s[c];
  dim3 g3((unsigned)((nlines + WL_LINES - 1) / WL_LINES), (unsigned)frames);
  const size_t shm = sizeof(float2) * WL_LINES * (size_t)pts;
  if (shm + sizeof(int64_t) * WL_LINES > 160 * 1024)  // + the kernel's line bases
    return fail(op, MRN_EUNSUPPORTED, "wavelet line too long");
  if (inv)
    hipLaunchKernelGGL(k_wave_lines<1>, g3, dim3(256), shm, st, X, N[0], N[1], s[0], s[1], s[2], axis, sh, f,
                       op->nvox);
  else
    hipLaunchKernelGGL(k_wave_lines<0>, g3, dim3(256), shm, st, X, N[0], N[1], s[0], s[1], s[2], axis, sh, f,
                       op->nvox);
  MRN_HIP(op, hipGetLastError());
  return MRN_OK;
}

// forward3D / backward3D of `frames` images, shifts sh[0..2] in device memory;
// levels l0 and deeper (l0 > 0: every axis has l0 levels, done elsewhere)
int wavelet3d(mrn_op *op, float2 *X, int frames, const int req[3], const int *sh, bool inv, hipStream_t st,
              int l0 = 0) {
  const int *N = op->g.N;
  int L[3];
  wavelet_levels(N, req, L);
  int maxl = 0;
  for (int a = 0; a < 3; a++) maxl = L[a] > maxl ? L[a] : maxl;
  if (!inv) {
    int s[3] = {N[0] >> l0, N[1] >> l0, N[2] >> l0};
    for (int l = l0; l < maxl; l++) {
      for (int a = 0; a < 3; a++)
        if (l < L[a]) MRN_TRY(wave_axis(op, X, frames, s, a, sh, false, st));
      for (int a = 0; a < 3; a++)
        if (l < L[a]) s[a] = N[a] >> (l + 1);
    }
  } else {
    int s[3];
    for (int a = 0; a < 3; a++) s[a] = N[a] >> L[a];
    for (int l = maxl - 1; l >= l0; l--) {
      for (int a = 0; a < 3; a++)
        if (l < L[a]) s[a] = N[a] >> l;
      for (int a = 2; a >= 0; a--)
        if (l < L[a]) MRN_TRY(wave_axis(op, X, frames, s, a, sh, true, st));
    }
  }
  return MRN_OK;
}

static unsigned grid_for(int64_t n) {
  int64_t b = (n + 255) / 256;
  if (b > 4096) b = 4096;
  return (unsigned)(b > 0 ? b : 1);
}

// fraction threshold of n coefficients into ThrState.thr (scaled), device only;
// mag: room for n floats (|c| is then computed once), or null
static int fraction_threshold(mrn_op *op, const float2 *X, float *mag, int64_t n, float fraction, float scale,
                              const int *log_counter, hipStream_t st) {
  ThrState *s = (ThrState *)op->dthr;
  double *log = log_counter ? op->dthr_log : nullptr;
  const int64_t nb = (n + 4 * THR_THREADS - 1) / (4 * THR_THREADS);
  const dim3 g3(nb < 512 ? (unsigned)(nb > 0 ? nb : 1) : 512u);
  hipLaunchKernelGGL(k_thr_reset, dim3(1), dim3(1), 0, st, s);
  hipLaunchKernelGGL(k_thr_minmax, g3, dim3(THR_THREADS), 0, st, X, mag, n, s, fraction, scale, log, log_counter,
                     MRN_TRACE_CAP);
  for (int r = 0; r < (64 + THR_DEPTH - 1) / THR_DEPTH; r++) {
    if (mag)
      hipLaunchKernelGGL(k_thr_count<float>, g3, dim3(THR_THREADS), 0, st, mag, n, s, scale, log, log_counter,
                         MRN_TRACE_CAP);
    else
      hipLaunchKernelGGL(k_thr_count<float2>, g3, dim3(THR_THREADS), 0, st, X, n, s, scale, log, log_counter,
                         MRN_TRACE_CAP);
  }
  MRN_HIP(op, hipGetLastError());
  return MRN_OK;
}

static unsigned wave_blocks(int n, int per) { return (unsigned)((n + per - 1) / per); }

// Levels that every axis has (done in one pass each), and the floats2 of the
// second image with the compact low-pass images of all but the last of them.
static int wave_common(const int L[3]) { return std::min(L[0], std::min(L[1], L[2])); }
static int64_t wave_low(const mrn_op *op, int l) { return op->nvox >> (3 * l); }
static int64_t wave_T_size(const mrn_op *op, int frames) {
  int64_t n = op->nvox;
  for (int l = 1; wave_low(op, l) > 0; l++) n += wave_low(op, l);
  return n * frames;
}

// image of level l's input (l = 0) or low-pass values: X, a compact image behind T, or T itself for the last
static WImg wave_img(mrn_op *op, float2 *X, float2 *T, int frames, int l, int last) {
  const int *N = op->g.N;
  const int64_t plane = (int64_t)N[0] * N[1];
  if (l == 0 || l == last) return WImg{l == 0 ? X : T, N[0], plane, op->nvox};
  float2 *p = T + frames * op->nvox;
  for (int q = 1; q < l; q++) p += frames * wave_low(op, q);
  return WImg{p, N[0] >> l, plane >> (2 * l), wave_low(op, l)};
}

// level l of `last` (all axes): from X or level l - 1's low-pass image to T and the next, or back with the threshold
static int wave3_level(mrn_op *op, float2 *X, float2 *T, int frames, int l, int last, const int *sh, bool inv, bool all,
                       hipStream_t st) {
  static const D4 f = d4_filters();
  const int *N = op->g.N;
  const int s[3] = {N[0] >> l, N[1] >> l, N[2] >> l};
  const WImg in = wave_img(op, X, T, frames, l, last), low = wave_img(op, X, T, frames, l + 1, last),
             det{T, N[0], (int64_t)N[0] * N[1], op->nvox};
  if (!inv) {
    const unsigned nz = wave_blocks(s[2] / 2, W3_PZ);
    hipLaunchKernelGGL(k_wave3_fwd, dim3(wave_blocks(s[0] / 2, W3_PX), wave_blocks(s[1] / 2, W3_PY), nz * frames),
                       dim3(W3_THREADS), 0, st, det, low, in, s[0], s[1], s[2], (int)nz, sh, f);
  } else {
    const unsigned nz = wave_blocks(s[2], W3_IZ);
    hipLaunchKernelGGL(k_wave3_inv, dim3(wave_blocks(s[0], W3_IX), wave_blocks(s[1], W3_IY), nz * frames),
                       dim3(W3_THREADS), 0, st, in, det, low, s[0], s[1], s[2], (int)nz, sh, f,
                       &((const ThrState *)op->dthr)->thr, all ? 1 : 0);
  }
  MRN_HIP(op, hipGetLastError());
  return MRN_OK;
}

// Whether the step has a use for the second image: a level on every axis, and a
// launch grid that holds the frames.
static bool wave_two(const mrn_op *op, int frames, const int levels[3]) {
  int L[3];
  wavelet_levels(op->g.N, levels, L);
  return wave_common(L) > 0 && wave_blocks(op->g.N[2], W3_IZ) * (int64_t)frames <= 65535;
}

// The L1 step over `frames` images; shifts of spin q at dsh[3q..3q+2].  With a
// level on every axis and the second image (op->wave_T) the coefficients live
// there; otherwise everything runs in place.
int l1_wavelet_step(mrn_op *op, float2 *X, int frames, float fraction, const int levels[3], int spins,
                    const int *log_counter, hipStream_t st) {
  const int64_t n = (int64_t)frames * op->nvox;
  const int *N = op->g.N;
  int L[3];
  wavelet_levels(N, levels, L);
  const int nf = wave_common(L), maxl = std::max(L[0], std::max(L[1], L[2]));
  const bool two = wave_two(op, frames, levels) && op->wave_T && op->wave_T_cap >= (size_t)wave_T_size(op, frames);
  float2 *T = two ? op->wave_T : X;
  const int s = two ? nf : 0;  // levels from here on in place, in T's (or X's) corner
  const bool rest = !two || maxl > nf;
  for (int q = 0; q < spins; q++) {
    const int *sh = op->dsh + 3 * q;
    for (int l = 0; l < s; l++) MRN_TRY(wave3_level(op, X, T, frames, l, s, sh, false, false, st));
    if (rest) MRN_TRY(wavelet3d(op, T, frames, levels, sh, false, st, s));
    if (q == 0)  // with the second image X is free until the synthesis
      MRN_TRY(fraction_threshold(op, T, two ? (float *)X : nullptr, n, fraction, 1.0f / (float)spins, log_counter, st));
    if (rest) {
      hipLaunchKernelGGL(k_soft, dim3(grid_for((n / frames) >> (3 * s)), std::min(frames, 65535)), dim3(256), 0, st, T,
                         N[0], N[1], N[0] >> s, N[1] >> s, N[2] >> s, op->nvox, frames, (const ThrState *)op->dthr);
      MRN_HIP(op, hipGetLastError());
      MRN_TRY(wavelet3d(op, T, frames, levels, sh, true, st, s));
    }
    for (int l = s - 1; l >= 0; l--) MRN_TRY(wave3_level(op, X, T, frames, l, s, sh, true, !rest && l == s - 1, st));
  }
  return MRN_OK;
}

// The second image of l1_wavelet_step (grow-only; without the memory the step
// runs in place).  Never called while capturing with a larger `frames`.
static void ensure_wave_T(mrn_op *op, int frames, const int levels[3]) {
  const int64_t n = wave_T_size(op, frames);
  if (op->wave_T_cap >= (size_t)n || !wave_two(op, frames, levels)) return;
  if (grow(op->wave_T, op->wave_T_cap, n) != hipSuccess) (void)hipGetLastError();
}

void l1_fista_prepare(mrn_op *op) { ensure_wave_T(op, op->F, op->l1_levels); }

// FISTA's step: shifts for the current iteration from the device counter
int l1_fista_step(mrn_op *op, float2 *X, hipStream_t st) {
  MRN_TRY(ensure_l1_state(op));
  const int count = 3 * op->l1_spins;
  hipLaunchKernelGGL(k_spin_shifts, dim3(1), dim3(3 * MRN_MAX_SPINS), 0, st, op->dsh, count,
                     (unsigned long long)op->l1_seed, op->dcounter);
  MRN_HIP(op, hipGetLastError());
  return l1_wavelet_step(op, X, op->F, op->l1_fraction, op->l1_levels, op->l1_spins, op->dcounter, st);
}

int l1_wavelet_host(mrn_op *op, float2 *X, int frames, float fraction, const int levels[3], int spins,
                    const int32_t *shifts, double *thr, hipStream_t st) {
  MRN_TRY(ensure_l1_state(op));
  ensure_wave_T(op, frames, levels);
  if (shifts) {
    MRN_HIP(op, hipMemcpyAsync(op->dsh, shifts, sizeof(int) * 3 * spins, hipMemcpyHostToDevice, st));
  } else {
    hipLaunchKernelGGL(k_spin_shifts, dim3(1), dim3(3 * MRN_MAX_SPINS), 0, st, op->dsh, 3 * spins,
                       (unsigned long long)op->l1_seed, nullptr);
  }
  MRN_TRY(l1_wavelet_step(op, X, frames, fraction, levels, spins, nullptr, st));
  if (thr) {
    ThrState h;
    MRN_HIP(op, hipMemcpyAsync(&h, op->dthr, sizeof(ThrState), hipMemcpyDeviceToHost, st));
    MRN_HIP(op, hipStreamSynchronize(st));
    *thr = (double)h.thr;
  }
  return MRN_OK;
}

int wavelet_host(mrn_op *op, float2 *X, int frames, const int levels[3], const int32_t shift[3], bool inv,
                 hipStream_t st) {
  MRN_TRY(ensure_l1_state(op));
  MRN_HIP(op, hipMemcpyAsync(op->dsh, shift, sizeof(int) * 3, hipMemcpyHostToDevice, st));
  return wavelet3d(op, X, frames, levels, op->dsh, inv, st);
}

}  // namespace mrn
