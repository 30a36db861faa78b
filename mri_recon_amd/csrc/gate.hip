// Gated frame selection: GATING::init_time_resolved's scaling of gate times
// (gating.cpp:880-1078, on the host: one value per readout), and on the
// device GATING::weight_data (gating.cpp:1082-1200) with RECON::pregate_data
// (recon_lib.cpp:675-776): for every frame t, keep the samples whose weight is
// positive, in sample order, frame after frame, with kw * 1e6 / count (or 1).
//
// Device side: a stream compaction, HBM-bound.  Pass 1 counts the selected
// samples of each (frame, 256-sample block); one exclusive scan over
// [frame][block] gives every block its output offset in frame-major order;
// pass 2 recomputes the selection and writes each kept sample at its offset
// plus its rank in the block (wavefront ballots), so the order is the input
// order.  A workgroup takes several frames of its block (gate_per), so the
// trajectory and the k-space are read once for those.
#include <algorithm>
#include <cmath>
#include <cstdlib>
#include <cstring>
#include <vector>

#include <hipcub/hipcub.hpp>

#include "mrn_internal.hpp"

namespace mrn {
namespace {

struct GateDev {
  int vs_type, shape, frames, reset;
  int wlo, whi;
  float kmax;
  long long xres, M, nb;  // samples per readout, samples, 256-sample blocks
};

// weight_data(NON_ITERATIVE, TIME_FRAME) > 0 for a sample in frame t: its
// readout's time, the width of the frames it belongs to, and whether its
// weight inside that width is positive -- evaluated once for all frames.
struct Pick {
  double gt, wdth;  // without view sharing: floor(time), unused
  bool pos;
  __device__ __forceinline__ bool in(const GateDev &g, int t) const {
    if (g.vs_type == MRN_VS_TORNADO) return pos && fabs(gt - (0.5 + (double)t)) < wdth;
    return pos && gt == (double)t;
  }
};
__device__ __forceinline__ Pick pick_sample(const GateDev &g, const double *__restrict__ gt,
                                            const float *__restrict__ resp, const float *__restrict__ kx,
                                            const float *__restrict__ ky, const float *__restrict__ kz, long long i) {
  Pick p{0.0, 0.0, false};
  if (i >= g.M) return p;
  const long long j = i / g.xres;
  float w = 1.0f;
  if (resp) w *= resp[j];
  p.gt = gt[j];
  if (g.vs_type == MRN_VS_TORNADO) {
    float kr = 0.0f, pw = 1.0f;
    if (g.shape == MRN_TORNADO_RADIAL) {
      kr = __fsqrt_rn(__fadd_rn(__fmul_rn(kx[i], kx[i]), __fmul_rn(ky[i], ky[i])));
      pw = __fdiv_rn(kr, g.kmax);  // (kr / kmax)^1
    } else if (g.shape == MRN_TORNADO_VIPR) {
      kr = __fsqrt_rn(__fadd_rn(__fadd_rn(__fmul_rn(kx[i], kx[i]), __fmul_rn(ky[i], ky[i])),
                                __fmul_rn(kz[i], kz[i])));
      const float q = __fdiv_rn(kr, g.kmax);
      pw = __fmul_rn(q, q);  // (kr / kmax)^2
    }
    p.wdth = 0.5 * (double)__fadd_rn(__fmul_rn((float)(g.whi - g.wlo), pw), (float)g.wlo);
    // the weight w / wdth inside the width (0 outside: never positive)
    p.pos = (float)((double)w * (1.0 / p.wdth)) > 0.0f;
  } else {
    p.gt = floor(p.gt);
    p.pos = w > 0.0f;
  }
  return p;
}

// Both passes take `per` frames of a 256-sample block in one workgroup: the
// trajectory, the k-space and the weight's arithmetic are read and done once
// for them.  20000 readouts of 256 samples, 8 coils, 12 frames with view
// sharing, a workgroup per frame and block before: counting 185 -> 64 us,
// writing 439 -> 370 us.
__global__ __launch_bounds__(256) void k_gate_count(GateDev g, const double *__restrict__ gt,
                                                    const float *__restrict__ resp, const float *__restrict__ kx,
                                                    const float *__restrict__ ky, const float *__restrict__ kz,
                                                    int per, int64_t *__restrict__ bcnt) {
  const Pick p = pick_sample(g, gt, resp, kx, ky, kz, (long long)blockIdx.x * 256 + threadIdx.x);
  const int t0 = blockIdx.y * per, t1 = min(t0 + per, g.frames);
  for (int t = t0; t < t1; t++) {
    const int n = __syncthreads_count(p.in(g, t));
    if (threadIdx.x == 0) bcnt[(long long)t * g.nb + blockIdx.x] = n;
  }
}

// frame bases and counts from the scanned block offsets: base[t] = boff[t*nb]
__global__ void k_gate_frames(GateDev g, const int64_t *__restrict__ boff, int64_t *__restrict__ fb) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t <= g.frames) fb[t] = boff[(long long)t * g.nb];
}

__global__ __launch_bounds__(256) void k_gate_scatter(GateDev g, const double *__restrict__ gt,
                                                      const float *__restrict__ resp, const float *__restrict__ kx,
                                                      const float *__restrict__ ky, const float *__restrict__ kz,
                                                      const float *__restrict__ kw, int C,
                                                      const float2 *__restrict__ kd, const int64_t *__restrict__ boff,
                                                      const int64_t *__restrict__ fb, float *__restrict__ ox,
                                                      float *__restrict__ oy, float *__restrict__ oz,
                                                      float *__restrict__ ow, float2 *__restrict__ okd, int per) {
  __shared__ int wcount[2][4];
  const long long i = (long long)blockIdx.x * 256 + threadIdx.x;
  const Pick p = pick_sample(g, gt, resp, kx, ky, kz, i);
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int t0 = blockIdx.y * per, t1 = min(t0 + per, g.frames);
  for (int t = t0; t < t1; t++) {
    const bool s = p.in(g, t);
    const unsigned long long m = __ballot(s);
    // two rows in turn: a wavefront writes a row again only after the next
    // frame's barrier, when every wavefront has read it
    int *row = wcount[t & 1];
    if (lane == 0) row[wave] = __popcll(m);
    __syncthreads();
    if (!s) continue;
    int before = __popcll(m & ((1ull << lane) - 1ull));
    for (int w = 0; w < wave; w++) before += row[w];
    const int64_t pos = boff[(long long)t * g.nb + blockIdx.x] + before;
    const int64_t base = fb[t], n = fb[t + 1] - fb[t], o = pos - base;
    ox[pos] = kx[i];
    oy[pos] = ky[i];
    oz[pos] = kz[i];
    const float scale = (float)(1e6 / (double)(float)n);
    ow[pos] = g.reset ? 1.0f : __fmul_rn(scale, kw[i]);
    for (int c = 0; c < C; c++) okd[base * C + (int64_t)c * n + o] = kd[(int64_t)c * g.M + i];
  }
}

// Frames per workgroup.  A workgroup's frames go one after the other, so fewer
// where there are not GATE_GROUPS workgroups of blocks alone.  The call in us
// with 1 frame / this rule / all: 25 blocks x 100 frames 583 / 582 / 658; 125 x
// 12 (16 coils) 156 / 157 / 170; 12 x 1000 5056 / 5088 / 5780; 2000 x 12 221 /
// 195 / 196; 2000 x 100 1021 / 716 / 725; 20000 x 12 999 / 663 / 664.
#define GATE_GROUPS 2048
int gate_per(long long nb, int frames) {
  return (int)std::min<long long>(std::max<long long>(nb * frames / GATE_GROUPS, 1), frames);
}

double median_sorted(const std::vector<double> &v) {
  const size_t n = v.size();
  if (n == 0) return 0.0;
  return (n & 1) ? v[n / 2] : v[n / 2 - 1] + (v[n / 2] - v[n / 2 - 1]) / 2;
}

// Hyndman & Fan method 5 on sorted values (Armadillo's documented quantile)
double quantile5(const std::vector<double> &v, double p) {
  const double n = (double)v.size();
  if (v.empty()) return 0.0;
  const double h = n * p + 0.5;
  if (h <= 1.0) return v.front();
  if (h >= n) return v.back();
  const size_t lo = (size_t)std::floor(h);
  return v[lo - 1] + (h - (double)lo) * (v[lo] - v[lo - 1]);
}

}  // namespace
}  // namespace mrn

using namespace mrn;

extern "C" {

void mrn_gate_params_default(mrn_gate_params *p) {
  if (!p) return;
  std::memset(p, 0, sizeof(*p));
  p->gate_type = MRN_GATE_NONE;
  p->vs_type = MRN_VS_NONE;
  p->frames = 1;
  p->tornado_shape = MRN_TORNADO_VIPR;
  p->wdth_low = 1;
  p->wdth_high = 4;
  p->kmax = 128.0f;
  p->min_quantile = 0.0f;
  p->max_quantile = 1.0f;
  p->ecg_outlier_reject = 1;
}

int mrn_gate_parse_args(mrn_gate_params *p, int argc, const char **argv) {
  if (!p || (argc > 0 && !argv)) return MRN_EINVAL;
  for (int i = 0; i < argc; i++) {
    const char *s = argv[i];
    const bool has = i + 1 < argc;
    auto word = [&](const char *w) { return has && !strcmp(argv[i + 1], w); };
    if (!strcmp(s, "-viewshare_type")) {
      if (word("tornado")) p->vs_type = MRN_VS_TORNADO;
      else if (word("hist")) p->vs_type = MRN_VS_HIST;
      else if (word("none")) p->vs_type = MRN_VS_NONE;
      else return MRN_EINVAL;
      i++;
    } else if (!strcmp(s, "-gating_type")) {
      if (word("retro_ecg")) p->gate_type = MRN_GATE_RETRO_ECG;
      else if (word("resp")) p->gate_type = MRN_GATE_RESP;
      else if (word("ecg")) p->gate_type = MRN_GATE_ECG;
      else if (word("time")) p->gate_type = MRN_GATE_TIME;
      else if (word("prep")) p->gate_type = MRN_GATE_PREP;
      else return MRN_EINVAL;
      i++;
    } else if (!strcmp(s, "-vs_wdth_low") || !strcmp(s, "-vs_wdth_high") || !strcmp(s, "-rcframes")) {
      if (!has) return MRN_EINVAL;
      const int v = atoi(argv[++i]);
      if (!strcmp(s, "-vs_wdth_low")) p->wdth_low = v;
      else if (!strcmp(s, "-vs_wdth_high")) p->wdth_high = v;
      else p->frames = v;
    } else if (!strcmp(s, "-gate_min_quantile") || !strcmp(s, "-gate_max_quantile")) {
      if (!has) return MRN_EINVAL;
      const float v = (float)atof(argv[++i]);
      if (!strcmp(s, "-gate_min_quantile")) p->min_quantile = v;
      else p->max_quantile = v;
    } else if (!strcmp(s, "-ecg_out_reject")) {
      p->ecg_outlier_reject = 1;
    } else if (!strcmp(s, "-wo_ecg_out_reject")) {
      p->ecg_outlier_reject = 0;
    }
  }
  return MRN_OK;
}

int mrn_gate_scale_times(const mrn_gate_params *p, int64_t R, double *t, double info[3]) {
  free_err_clear();
  if (!p || R < 1 || !t) return free_fail(MRN_EINVAL, "gate times");
  if (p->frames < 1) return free_fail(MRN_EINVAL, "frames < 1");
  if (p->vs_type != MRN_VS_TORNADO && p->vs_type != MRN_VS_NONE && p->vs_type != MRN_VS_HIST)
    return free_fail(MRN_EINVAL, "view sharing type");
  std::vector<double> v(t, t + R);
  double mx, mn;
  if (p->gate_type == MRN_GATE_RETRO_ECG) {
    std::sort(v.begin(), v.end());
    mn = 0.0;
    mx = 2.0 * median_sorted(v);
    if (p->ecg_outlier_reject) {
      std::vector<double> w;
      for (int64_t i = 0; i < R; i++)
        if (t[i] < 1.3 * mx) w.push_back(t[i]);
      std::sort(w.begin(), w.end());
      mx = 2.0 * median_sorted(w);
    }
  } else if (p->gate_type == MRN_GATE_RESP) {
    if (p->frames < 2) return free_fail(MRN_EINVAL, "respiratory gating needs 2 or more frames");
    std::sort(v.begin(), v.end());
    const double v0 = quantile5(v, p->min_quantile), v1 = quantile5(v, p->max_quantile);
    const double fw = (v1 - v0) / (p->frames - 1.0);
    mx = v1 + 0.5 * fw;
    mn = v0 - 0.5 * fw;
  } else {
    const auto mm = std::minmax_element(v.begin(), v.end());
    mn = *mm.first;
    mx = *mm.second;
  }
  if (!(mx > mn)) return free_fail(MRN_EINVAL, "gate times span no range");
  const double scale = (float)p->frames / (mx - mn) * (1 - 1e-9);
  const double offset = mn;
  for (int64_t i = 0; i < R; i++) t[i] = (t[i] - offset) * scale;
  if (info) {
    info[0] = offset;
    info[1] = scale;
    info[2] = (mx - mn) / ((float)p->frames);
  }
  if (p->vs_type == MRN_VS_NONE) {
    for (int64_t i = 0; i < R; i++) t[i] = std::floor(t[i]);
  } else if (p->vs_type == MRN_VS_HIST) {
    std::vector<int64_t> idx(R);
    for (int64_t i = 0; i < R; i++) idx[i] = i;
    std::stable_sort(idx.begin(), idx.end(), [&](int64_t a, int64_t b) { return t[a] < t[b]; });
    for (int64_t r = 0; r < R; r++) v[idx[r]] = (double)(int)((double)(r * p->frames) / (double)R);
    std::copy(v.begin(), v.end(), t);
  }
  return MRN_OK;
}

int mrn_pregate(const mrn_gate_params *p, int64_t xres, int64_t R, const double *gt, const float *resp,
                const float *kx, const float *ky, const float *kz, const float *kw, int C, const void *kdata,
                int64_t *counts, float *kx_out, float *ky_out, float *kz_out, float *kw_out, void *kdata_out,
                void *stream) {
  free_err_clear();
  if (!p || !counts || xres < 1 || R < 1 || C < 0) return free_fail(MRN_EINVAL, "sizes");
  if (!gt || !kx || !ky || !kz || !kw || (C > 0 && !kdata)) return free_fail(MRN_EINVAL, "input arrays");
  if (p->frames < 1 || p->frames > 65535) return free_fail(MRN_EINVAL, "frames in 1..65535");
  if (p->vs_type == MRN_VS_TORNADO && !(p->kmax > 0.0f)) return free_fail(MRN_EINVAL, "tornado kmax");
  const bool fill = kx_out != nullptr;
  if (fill && (!ky_out || !kz_out || !kw_out || (C > 0 && !kdata_out)))
    return free_fail(MRN_EINVAL, "output arrays");
  GateDev g;
  g.vs_type = p->vs_type;
  g.shape = p->tornado_shape;
  g.frames = p->frames;
  g.reset = p->reset_dens != 0;
  g.wlo = p->wdth_low;
  g.whi = p->wdth_high;
  g.kmax = p->kmax;
  g.xres = xres;
  g.M = xres * R;
  g.nb = (g.M + 255) / 256;
  if (g.nb > 0x7fffffffll) return free_fail(MRN_EUNSUPPORTED, "too many samples");
  hipStream_t st = (hipStream_t)stream;
  const int64_t nflat = (int64_t)g.frames * g.nb;
  const int per = gate_per(g.nb, g.frames);
  const dim3 grid((unsigned)g.nb, (unsigned)((g.frames + per - 1) / per));
  int64_t *bcnt = nullptr;  // 64-bit: the scan accumulates in its input type
  int64_t *boff = nullptr, *fb = nullptr;
  void *tmp = nullptr;
  size_t tb = 0;
  int rc = MRN_OK;
  std::vector<int64_t> hfb(g.frames + 1);
  auto run = [&]() -> hipError_t {
    hipError_t e;
    if ((e = hipMalloc(&bcnt, sizeof(int64_t) * (nflat + 1))) != hipSuccess) return e;
    if ((e = hipMalloc(&boff, sizeof(int64_t) * (nflat + 1))) != hipSuccess) return e;
    if ((e = hipMalloc(&fb, sizeof(int64_t) * (g.frames + 1))) != hipSuccess) return e;
    if ((e = hipMemsetAsync(bcnt + nflat, 0, sizeof(int64_t), st)) != hipSuccess) return e;
    hipLaunchKernelGGL(k_gate_count, grid, dim3(256), 0, st, g, gt, resp, kx, ky, kz, per, bcnt);
    if ((e = hipGetLastError()) != hipSuccess) return e;
    if ((e = hipcub::DeviceScan::ExclusiveSum(nullptr, tb, bcnt, boff, nflat + 1, st)) != hipSuccess) return e;
    if ((e = hipMalloc(&tmp, tb)) != hipSuccess) return e;
    if ((e = hipcub::DeviceScan::ExclusiveSum(tmp, tb, bcnt, boff, nflat + 1, st)) != hipSuccess) return e;
    hipLaunchKernelGGL(k_gate_frames, dim3((g.frames + 256) / 256), dim3(256), 0, st, g, boff, fb);
    if ((e = hipGetLastError()) != hipSuccess) return e;
    if ((e = hipMemcpyAsync(hfb.data(), fb, sizeof(int64_t) * (g.frames + 1), hipMemcpyDeviceToHost, st)) !=
        hipSuccess)
      return e;
    if (fill) {
      hipLaunchKernelGGL(k_gate_scatter, grid, dim3(256), 0, st, g, gt, resp, kx, ky, kz,
                         kw, C, (const float2 *)kdata, boff, fb, kx_out, ky_out, kz_out, kw_out, (float2 *)kdata_out, per);
      if ((e = hipGetLastError()) != hipSuccess) return e;
    }
    return hipStreamSynchronize(st);
  };
  const hipError_t e = run();
  if (e != hipSuccess) {
    hipStreamSynchronize(st);
    rc = free_fail(MRN_EHIP, hipGetErrorString(e));
  } else {
    for (int t = 0; t < g.frames; t++) counts[t] = hfb[t + 1] - hfb[t];
  }
  hipFree(bcnt);
  hipFree(boff);
  hipFree(fb);
  hipFree(tmp);
  return rc;
}

}  // extern "C"
