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
// The fraction threshold runs entirely on the device: a min/max pass, then 16
// rounds of (count below the bisection's next 15 candidate values, one-thread
// replay of up to 4 bisection steps), each round a no-op once the bracket has
// converged, so the whole step can be captured in a hipGraph.  |c| is evaluated as sqrt in double rounded to float, so the
// counts and the threshold do not depend on the order of operations.
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

// ------------------------------------------------------- first level, 3 axes
// The first level of a 3-D transform, all three axes in one pass from one
// image to another: 7/8 of a transform's traffic is in this level, which as
// three line passes reads and writes the image three times.  A workgroup
// loads the region that its outputs reach into LDS and transforms it along x,
// y, z (synthesis: z, y, x) in place, each thread holding its outputs in
// registers across the barrier; the products and their order are those of
// k_wave_lines, so the results are the same bits.  The synthesis applies the
// soft threshold to the seven detail octants as it loads them (the low-pass
// octant holds the deeper levels' image by then).
// 256 x 256 x 192, 4 levels, 4 spins: the step 3.10 -> 2.05 ms (analysis of the
// first level 63 us, synthesis with the threshold 154 us).
#define W3_THREADS 512
#define W3_PX 16  // analysis: output positions of a workgroup (a low- and a high-pass value each per axis)
#define W3_PY 8
#define W3_PZ 4

__device__ __forceinline__ float cabs_rn(float2 v) {
  return (float)sqrt((double)v.x * v.x + (double)v.y * v.y);
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

__global__ __launch_bounds__(W3_THREADS) void k_wave3_fwd(float2 *__restrict__ T, const float2 *__restrict__ X, int N0,
                                                          int N1, int N2, int nz, const int *__restrict__ sh, D4 f) {
  constexpr int RX = 2 * W3_PX + 2, RY = 2 * W3_PY + 2, RZ = 2 * W3_PZ + 2;
  __shared__ float2 A[RX * RY * RZ];
  const int fr = blockIdx.z / nz;
  const int p0[3] = {(int)blockIdx.x * W3_PX, (int)blockIdx.y * W3_PY, (int)(blockIdx.z - fr * nz) * W3_PZ};
  const int64_t n = (int64_t)N0 * N1 * N2;
  const float2 *Xf = X + fr * n;
  float2 *Tf = T + fr * n;
  // cell (x, y, z) of the region: image point 2 p0 + shift - 3 + (x, y, z)
  const int ox = 2 * p0[0] + sh[0] - 3, oy = 2 * p0[1] + sh[1] - 3, oz = 2 * p0[2] + sh[2] - 3;
  for (int q = threadIdx.x; q < RX * RY * RZ; q += W3_THREADS) {
    const int x = q % RX, yz = q / RX, y = yz % RY, z = yz / RY;
    A[q] = Xf[((int64_t)wmod(oz + z, N2) * N1 + wmod(oy + y, N1)) * N0 + wmod(ox + x, N0)];
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
  // z, straight to the image
  constexpr int NX = 2 * W3_PX, NY = 2 * W3_PY, TOT = NX * NY * W3_PZ;
  const int h0 = N0 >> 1, h1 = N1 >> 1, h2 = N2 >> 1;
  for (int q = threadIdx.x; q < TOT; q += W3_THREADS) {
    const int x = q % NX, y = (q / NX) % NY, p = q / (NX * NY);
    const int px = p0[0] + x % W3_PX, py = p0[1] + y % W3_PY, pz = p0[2] + p;
    if (px >= h0 || py >= h1 || pz >= h2) continue;
    float2 lo, hi;
    wave_pair(A, (2 * p * RY + y) * RX + x, RY * RX, f, lo, hi);
    float2 *dst = Tf + (int64_t)(py + (y < W3_PY ? 0 : h1)) * N0 + px + (x < W3_PX ? 0 : h0);
    dst[(int64_t)pz * N1 * N0] = lo;
    dst[(int64_t)(pz + h2) * N1 * N0] = hi;
  }
}

// Synthesis: a workgroup makes W3_IX x W3_IY x W3_IZ points.  Point p takes the
// positions t / 2 of the even t = p - fp + 3 - shift; the region holds the
// workgroup's n / 2 + 2 positions per axis, low-pass then high-pass values.
#define W3_IX 32
#define W3_IY 16
#define W3_IZ 8
template <int H>  // distance of the high-pass value
__device__ __forceinline__ float2 wave_point(const float2 *in, int p, int shift, int b0, int st, const D4 &f) {
  float2 o = make_float2(0.f, 0.f);
#pragma unroll
  for (int fp = 0; fp < 4; fp++) {
    const int t = p - fp + 3 - shift;
    if (t & 1) continue;
    const int at = ((t >> 1) - b0) * st;
    const float2 a = in[at], d = in[at + H];
    o.x += a.x * f.slpf[fp];
    o.y += a.y * f.slpf[fp];
    o.x += d.x * f.shpf[fp];
    o.y += d.y * f.shpf[fp];
  }
  return o;
}

__global__ __launch_bounds__(W3_THREADS) void k_wave3_inv(float2 *__restrict__ X, const float2 *__restrict__ T, int N0,
                                                          int N1, int N2, int nz, const int *__restrict__ sh, D4 f,
                                                          const float *__restrict__ thr_p) {
  constexpr int CX = W3_IX / 2 + 2, CY = W3_IY / 2 + 2, CZ = W3_IZ / 2 + 2;  // positions
  constexpr int RX = 2 * CX, RY = 2 * CY, RZ = 2 * CZ;
  extern __shared__ float2 A[];  // [RZ][RY][RX]
  const int fr = blockIdx.z / nz;
  const int p0[3] = {(int)blockIdx.x * W3_IX, (int)blockIdx.y * W3_IY, (int)(blockIdx.z - fr * nz) * W3_IZ};
  const int64_t n = (int64_t)N0 * N1 * N2;
  const float2 *Tf = T + fr * n;
  float2 *Xf = X + fr * n;
  const int h0 = N0 >> 1, h1 = N1 >> 1, h2 = N2 >> 1;
  const int s0 = sh[0], s1 = sh[1], s2 = sh[2];
  const int b0 = (p0[0] - s0 + 1) >> 1, b1 = (p0[1] - s1 + 1) >> 1, b2 = (p0[2] - s2 + 1) >> 1;  // first positions
  const float thr = *thr_p;
  for (int q = threadIdx.x; q < RX * RY * RZ; q += W3_THREADS) {
    const int x = q % RX, yz = q / RX, y = yz % RY, z = yz / RY;
    const bool hx = x >= CX, hy = y >= CY, hz = z >= CZ;
    const int px = wmod(b0 + (hx ? x - CX : x), h0) + (hx ? h0 : 0), py = wmod(b1 + (hy ? y - CY : y), h1) + (hy ? h1 : 0),
              pz = wmod(b2 + (hz ? z - CZ : z), h2) + (hz ? h2 : 0);
    const float2 v = Tf[((int64_t)pz * N1 + py) * N0 + px];
    A[q] = hx || hy || hz ? soft(v, thr) : v;
  }
  __syncthreads();
  {  // z
    constexpr int TOT = RX * RY * W3_IZ, PER = (TOT + W3_THREADS - 1) / W3_THREADS;
    float2 o[PER];
#pragma unroll
    for (int k = 0; k < PER; k++) {
      const int q = threadIdx.x + k * W3_THREADS, xy = q % (RX * RY), p = q / (RX * RY);
      if (q < TOT) o[k] = wave_point<CZ * RX * RY>(A + xy, p0[2] + p, s2, b2, RX * RY, f);
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < PER; k++) {
      const int q = threadIdx.x + k * W3_THREADS;
      if (q < TOT) A[q] = o[k];  // [W3_IZ][RY][RX]
    }
    __syncthreads();
  }
  {  // y
    constexpr int TOT = RX * W3_IY * W3_IZ, PER = (TOT + W3_THREADS - 1) / W3_THREADS;
    float2 o[PER];
#pragma unroll
    for (int k = 0; k < PER; k++) {
      const int q = threadIdx.x + k * W3_THREADS, x = q % RX, p = (q / RX) % W3_IY, z = q / (RX * W3_IY);
      if (q < TOT) o[k] = wave_point<CY * RX>(A + z * RY * RX + x, p0[1] + p, s1, b1, RX, f);
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < PER; k++) {
      const int q = threadIdx.x + k * W3_THREADS;
      if (q < TOT) A[q] = o[k];  // [W3_IZ][W3_IY][RX]
    }
    __syncthreads();
  }
  // x, straight to the image
  for (int q = threadIdx.x; q < W3_IX * W3_IY * W3_IZ; q += W3_THREADS) {
    const int p = q % W3_IX, y = (q / W3_IX) % W3_IY, z = q / (W3_IX * W3_IY);
    const int px = p0[0] + p, py = p0[1] + y, pz = p0[2] + z;
    if (px >= N0 || py >= N1 || pz >= N2) continue;
    Xf[((int64_t)pz * N1 + py) * N0 + px] = wave_point<CX>(A + (z * W3_IY + y) * RX, px, s0, b0, 1, f);
  }
}

// ------------------------------------------------------------ threshold
#define THR_DEPTH 4                         // bisection steps per counting pass
#define THR_NODES ((1 << THR_DEPTH) - 1)    // candidate values per pass
struct ThrState {
  unsigned int umin, umax;  // bit patterns of min / max |c| (non-negative floats)
  float value, max_t, min_t, thr;
  int iter, done;
  unsigned long long counter;
  long long found, target, accuracy, total;
  unsigned long long cnt[THR_NODES];  // count(|c| < candidate) of this pass
};

// The next THR_DEPTH values the bisection can query, breadth first: node k
// (value v, bracket [lo, hi]) has children 2k + 1 (count > target: max = v)
// and 2k + 2 (min = v), each at 0.5 * (max + min) as the sequential step
// computes it, so that a pass counts exactly the values the sequence visits.
__device__ __forceinline__ void thr_tree(const ThrState &s, float (&v)[THR_NODES]) {
  float lo[THR_NODES], hi[THR_NODES];
  v[0] = s.value;
  lo[0] = s.min_t;
  hi[0] = s.max_t;
#pragma unroll
  for (int k = 0; 2 * k + 2 < THR_NODES; k++) {
    lo[2 * k + 1] = lo[k];
    hi[2 * k + 1] = v[k];
    v[2 * k + 1] = 0.5f * (hi[2 * k + 1] + lo[2 * k + 1]);
    lo[2 * k + 2] = v[k];
    hi[2 * k + 2] = hi[k];
    v[2 * k + 2] = 0.5f * (hi[2 * k + 2] + lo[2 * k + 2]);
  }
}

__global__ void k_thr_reset(ThrState *s) {
  s->umin = 0x7f800000u;  // +inf
  s->umax = 0u;
  s->counter = 0ull;
}

__global__ __launch_bounds__(256) void k_thr_minmax(const float2 *__restrict__ X, int64_t n, ThrState *s) {
  float mn = INFINITY, mx = 0.0f;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
    const float v = cabs_rn(X[i]);
    mn = fminf(mn, v);
    mx = fmaxf(mx, v);
  }
  for (int o = 32; o > 0; o >>= 1) {
    mn = fminf(mn, __shfl_xor(mn, o));
    mx = fmaxf(mx, __shfl_xor(mx, o));
  }
  // one atomic pair per workgroup: atomics on one address serialise in L2
  __shared__ float s_mn[256 / 64], s_mx[256 / 64];
  if ((threadIdx.x & 63) == 0) {
    s_mn[threadIdx.x >> 6] = mn;
    s_mx[threadIdx.x >> 6] = mx;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int w = 1; w < (int)(blockDim.x >> 6); w++) {
      mn = fminf(mn, s_mn[w]);
      mx = fmaxf(mx, s_mx[w]);
    }
    atomicMin(&s->umin, __float_as_uint(mn));
    atomicMax(&s->umax, __float_as_uint(mx));
  }
}

// get_threshold's set-up (threshold.cpp:250-336)
__global__ void k_thr_init(ThrState *s, long long total, float fraction) {
  const float mx = __uint_as_float(s->umax), mn = __uint_as_float(s->umin);
  s->total = total;
  s->target = (long long)(fraction * (double)total);
  s->accuracy = (long long)(0.001 * (double)total);
  s->value = 0.5f * (mx - mn);
  s->max_t = fraction * mx;
  s->min_t = mn;
  s->iter = 0;
  s->found = total;
  s->counter = 0ull;
  for (int k = 0; k < THR_NODES; k++) s->cnt[k] = 0ull;
  s->done = 0;
  if (s->target < 2) {
    s->value = 0.0f;
    s->done = 1;
  } else if (!(llabs(s->found - s->target) > s->accuracy)) {
    s->done = 1;
  }
}

// One counting pass: count(|c| < v) for every candidate of thr_tree.
__global__ __launch_bounds__(256) void k_thr_count(const float2 *__restrict__ X, int64_t n, ThrState *s) {
  __shared__ unsigned int s_cnt[THR_NODES];
  if (s->done) return;  // (uniform)
  float v[THR_NODES];
  thr_tree(*s, v);
  if (threadIdx.x < THR_NODES) s_cnt[threadIdx.x] = 0u;
  __syncthreads();
  unsigned int cnt[THR_NODES];
#pragma unroll
  for (int k = 0; k < THR_NODES; k++) cnt[k] = 0u;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
    const float a = cabs_rn(X[i]);
#pragma unroll
    for (int k = 0; k < THR_NODES; k++) cnt[k] += a < v[k] ? 1u : 0u;
  }
#pragma unroll
  for (int k = 0; k < THR_NODES; k++) {
    unsigned int c = cnt[k];
    for (int o = 32; o > 0; o >>= 1) c += __shfl_xor(c, o);
    if ((threadIdx.x & 63) == 0 && c) atomicAdd(&s_cnt[k], c);
  }
  __syncthreads();
  if (threadIdx.x < THR_NODES && s_cnt[threadIdx.x])
    atomicAdd(&s->cnt[threadIdx.x], (unsigned long long)s_cnt[threadIdx.x]);
}

// one bisection step after a count (threshold.cpp:337-378)
// Up to THR_DEPTH steps of threshold.cpp:250-380's bisection, from the
// counts of one pass: the same values, counts and stopping rule as one step
// per pass.
__global__ void k_thr_step(ThrState *s) {
  if (s->done) return;
  float v[THR_NODES];
  thr_tree(*s, v);
  int node = 0;
  for (int lvl = 0; lvl < THR_DEPTH; lvl++) {
    s->value = v[node];
    s->found = (long long)s->cnt[node];
    s->iter++;
    if (!(llabs(s->found - s->target) > s->accuracy && s->iter < 64)) {
      s->done = 1;
      break;
    }
    if (s->found > s->target) {
      s->max_t = v[node];
      node = 2 * node + 1;
    } else {
      s->min_t = v[node];
      node = 2 * node + 2;
    }
    if (lvl == THR_DEPTH - 1) s->value = 0.5f * (s->max_t + s->min_t);
  }
  for (int k = 0; k < THR_NODES; k++) s->cnt[k] = 0ull;
}

// global threshold = scale * value; optionally logged per FISTA iteration
__global__ void k_thr_final(ThrState *s, float scale, double *log, const int *counter, int cap) {
  s->thr = scale * s->value;
  if (log) {
    const int it = counter ? *counter - 1 : 0;
    if (it >= 0 && it < cap) log[it] = (double)s->thr;
  }
}

// soft threshold of the sub-block [0, s0) x [0, s1) x [0, s2) of each frame (blockIdx.y)
__global__ __launch_bounds__(256) void k_soft(float2 *X, int N0, int N1, int s0, int s1, int s2, int64_t frame_stride,
                                              const ThrState *__restrict__ s) {
  const float thr = s->thr;
  float2 *Xf = X + (int64_t)blockIdx.y * frame_stride;
  const int64_t n = (int64_t)s0 * s1 * s2;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
    const int64_t yz = i / s0;
    float2 *v = Xf + ((yz / s1) * N1 + yz % s1) * N0 + i % s0;
    *v = soft(*v, thr);
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

// ... and what FISTA's step uses, before any capture
static void ensure_wave_T(mrn_op *op, int frames);
int l1_fista_prepare(mrn_op *op) {
  MRN_TRY(ensure_l1_state(op));
  ensure_wave_T(op, op->F);
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

// fraction threshold of n coefficients into ThrState.thr (scaled), device only
static int fraction_threshold(mrn_op *op, const float2 *X, int64_t n, float fraction, float scale,
                              const int *log_counter, hipStream_t st) {
  ThrState *s = (ThrState *)op->dthr;
  hipLaunchKernelGGL(k_thr_reset, dim3(1), dim3(1), 0, st, s);
  hipLaunchKernelGGL(k_thr_minmax, dim3(grid_for(n) < 1024 ? grid_for(n) : 1024), dim3(256), 0, st, X, n, s);
  hipLaunchKernelGGL(k_thr_init, dim3(1), dim3(1), 0, st, s, (long long)n, fraction);
  for (int r = 0; r < (64 + THR_DEPTH - 1) / THR_DEPTH; r++) {
    hipLaunchKernelGGL(k_thr_count, dim3(grid_for(n)), dim3(256), 0, st, X, n, s);
    hipLaunchKernelGGL(k_thr_step, dim3(1), dim3(1), 0, st, s);
  }
  hipLaunchKernelGGL(k_thr_final, dim3(1), dim3(1), 0, st, s, scale, log_counter ? op->dthr_log : nullptr,
                     log_counter, MRN_TRACE_CAP);
  MRN_HIP(op, hipGetLastError());
  return MRN_OK;
}

static unsigned wave_blocks(int n, int per) { return (unsigned)((n + per - 1) / per); }

// first level of every axis: X -> T, and T (detail octants thresholded) -> X
static int wave3_first(mrn_op *op, float2 *X, float2 *T, int frames, const int *sh, bool inv, hipStream_t st) {
  static const D4 f = d4_filters();
  const int *N = op->g.N;
  if (!inv) {
    const unsigned nz = wave_blocks(N[2] / 2, W3_PZ);
    hipLaunchKernelGGL(k_wave3_fwd, dim3(wave_blocks(N[0] / 2, W3_PX), wave_blocks(N[1] / 2, W3_PY), nz * frames),
                       dim3(W3_THREADS), 0, st, T, X, N[0], N[1], N[2], (int)nz, sh, f);
  } else {
    constexpr size_t lds = sizeof(float2) * (W3_IX + 4) * (W3_IY + 4) * (W3_IZ + 4);
    static const hipError_t attr =
        hipFuncSetAttribute((const void *)k_wave3_inv, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    MRN_HIP(op, attr);
    const unsigned nz = wave_blocks(N[2], W3_IZ);
    hipLaunchKernelGGL(k_wave3_inv, dim3(wave_blocks(N[0], W3_IX), wave_blocks(N[1], W3_IY), nz * frames),
                       dim3(W3_THREADS), lds, st, X, T, N[0], N[1], N[2], (int)nz, sh, f,
                       &((const ThrState *)op->dthr)->thr);
  }
  MRN_HIP(op, hipGetLastError());
  return MRN_OK;
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
  const bool two = L[0] > 0 && L[1] > 0 && L[2] > 0 && op->wave_T && op->wave_T_cap >= (size_t)n &&
                   wave_blocks(N[2], W3_IZ) * (int64_t)frames <= 65535;
  float2 *T = two ? op->wave_T : X;
  const int s = two ? 1 : 0;  // the level in T's (or X's) corner that is left to do in place
  for (int q = 0; q < spins; q++) {
    const int *sh = op->dsh + 3 * q;
    if (two) MRN_TRY(wave3_first(op, X, T, frames, sh, false, st));
    MRN_TRY(wavelet3d(op, T, frames, levels, sh, false, st, s));
    if (q == 0) MRN_TRY(fraction_threshold(op, T, n, fraction, 1.0f / (float)spins, log_counter, st));
    hipLaunchKernelGGL(k_soft, dim3(grid_for((n / frames) >> (3 * s)), frames), dim3(256), 0, st, T, N[0], N[1],
                       N[0] >> s, N[1] >> s, N[2] >> s, op->nvox, (const ThrState *)op->dthr);
    MRN_HIP(op, hipGetLastError());
    MRN_TRY(wavelet3d(op, T, frames, levels, sh, true, st, s));
    if (two) MRN_TRY(wave3_first(op, X, T, frames, sh, true, st));
  }
  return MRN_OK;
}

// The second image of l1_wavelet_step (grow-only; without the memory the step
// runs in place).  Never called while capturing with a larger `frames`.
static void ensure_wave_T(mrn_op *op, int frames) {
  if (op->wave_T_cap >= (size_t)frames * op->nvox) return;
  if (grow(op->wave_T, op->wave_T_cap, (int64_t)frames * op->nvox) != hipSuccess) (void)hipGetLastError();
}

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
  ensure_wave_T(op, frames);
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
