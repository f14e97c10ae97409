// Fused 11x11 Gaussian-window SSIM (sigma 1.5, zero padding, "same" output)
// forward with the three partial-derivative maps, and its backward.
//
// Reference: clm_kernels/ssim.cu:187-286 (fusedssimCUDA), :288-366
// (fusedssim_backwardCUDA), clm_kernels/__init__.py:23-61 (autograd wrapper;
// C1 = 0.01^2, C2 = 0.03^2).  Per pixel and channel:
//   mu = G*x, sigma_xx = G*(x^2) - mu^2, sigma_xy = G*(xy) - mu1 mu2
//   C = 2 mu1 mu2 + C1, D = 2 sigma12 + C2, A = mu1^2 + mu2^2 + C1,
//   B = sigma1^2 + sigma2^2 + C2, m = C D / (A B)
//   dm/dmu1, dm/dsigma1^2 (= -C D / (A B^2)), dm/dsigma12 (= 2 C / (A B))
// Backward: dL/dx = G*(g dm/dmu1) + 2 x G*(g dm/dsigma1^2) + y G*(g dm/dsigma12).
//
// Separable passes in the same order as the reference (x first, then y), as
// wavefronts that stream down a strip of columns.  The fused step's loss also
// folds in the L1 term and the clamp(gt/255, 0, 1) target normalisation of
// strategies/base_engine.py:472-488.
#include "tgs_common.cuh"

#include <algorithm>

#define SS_R 5  // window radius

// Normalised Gaussian window, w_i = exp(-(i-5)^2 / 4.5) / sum_j exp(-(j-5)^2 / 4.5).
__constant__ float c_gauss[11] = {
    0.001028380123898387f, 0.0075987582094967365f, 0.036000773310661316f,
    0.10936068743467331f,  0.21300552785396576f,   0.26601171493530273f,
    0.21300552785396576f,  0.10936068743467331f,   0.036000773310661316f,
    0.0075987582094967365f, 0.001028380123898387f};

__device__ __forceinline__ void lr_wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// The window's distinct weights (the taps mirror about the centre) in VGPRs, so
// that every window product takes two VGPR sources (forms that issue in pairs
// on gfx950).
struct Taps {
  float w[6];
  __device__ __forceinline__ Taps() {
#pragma unroll
    for (int t = 0; t < 6; ++t) asm volatile("v_mov_b32 %0, %1" : "=v"(w[t]) : "s"(c_gauss[t]));
  }
  __device__ __forceinline__ float operator()(int t) const { return w[t < 6 ? t : 10 - t]; }
};

#define LR_RING 11  // rows a streaming wavefront keeps in registers: the window's height

// ---------------------------------------------------------------------------
// Drop-in fused SSIM: forward and backward each in one row-streaming pass.
//
// One wavefront per (image, channel, strip of SR_OUT output columns, band of
// rows); lane L holds column x0 - 5 + L.  The wavefront walks the band's input
// rows top to bottom (10 more than its output rows), passes each row through a
// wavefront's LDS row for the horizontal window sums and keeps their last 11
// rows in registers for the vertical ones: no row is filtered twice and no
// workgroup barrier is taken.  The step loop is unrolled by the ring length,
// so every ring index is a constant, and each row is loaded two steps ahead.
// 16x16 tiles with a 26x26 halo in LDS, the form before, filtered 2.6 rows and
// columns per output and idled threads at its barriers: one 1080p image of 3
// channels took 85 us forward and 103 us backward, here 55 and 54 (the mean form 60
// and 48).  What bounds it is a row's chain through LDS and the ring at two
// wavefronts per SIMD: the forward issues its window products at 70% of the rate
// that the fused loss reaches on sixteen such images, the backward at 37%.
// The mean form writes neither the map nor its gradient (a constant): forward
// 20 bytes, backward 24 bytes per value, against 24 + 4 and 28 + 12 with the
// mean's reduction and the gradient's expansion as passes of their own.
//
// The three channel wavefronts of an RGB strip share a workgroup (their reads
// of a channels-last image are the same lines).
// ---------------------------------------------------------------------------
#define SR_OUT (64 - 2 * SS_R)  // output columns per strip

// Band rows for a launch of `planes` planes of H x W: input rows of a band
// (a multiple of the ring) chosen for the least time of the slowest CU, rows
// times the larger of a lone wavefront's time per row and the CU's share.
// `halo`: input rows beyond the output rows; `lone`: the time per row of a
// workgroup that has its CU to itself, in units of a busy CU's time per row and
// workgroup.
static int band_input_rows(int H, int64_t strips_planes, int halo, float lone, int max_periods) {
  int best = LR_RING * 2;
  float best_cost = 0.f;
  for (int k = (halo + LR_RING) / LR_RING; k <= max_periods; ++k) {
    const int rows = k * LR_RING, band = rows - halo;
    if (band <= 0) continue;
    const int64_t wgs = strips_planes * ((H + band - 1) / band);
    const float per_cu = (float)((wgs + 255) / 256);
    const float cost = (float)rows * (per_cu > lone ? per_cu : lone);
    if (best_cost == 0.f || cost < best_cost) {
      best_cost = cost;
      best = rows;
    }
  }
  return best;
}

// Most workgroups that band_input_rows can lead to, for planes and sizes up to
// these: every row a band of its own at the least rows, or what the cost allows (no
// more than the longest bands', whose cost the choice never exceeds).
static int64_t band_workgroups_max(int H, int64_t strips_planes, int halo, float lone,
                                   int max_periods) {
  const int least = (halo + LR_RING) / LR_RING * LR_RING, longest = max_periods * LR_RING;
  const int64_t by_rows = strips_planes * ((H + least - halo - 1) / (least - halo));
  const int64_t wgs = strips_planes * ((H + longest - halo - 1) / (longest - halo));
  const double per_cu = std::max((double)((wgs + 255) / 256), (double)lone);
  // (the slack and the 1: the costs are compared in float)
  return std::min(by_rows, 256 * ((int64_t)(longest * per_cu / least * (1 + 1e-6)) + 1));
}

struct Plane {
  int64_t bs, cs, ys, xs;  // batch, channel, row, column strides (elements)
};

__global__ void __launch_bounds__(192) ssim_fwd_rows_kernel(
    int CH, int H, int W, float C1, float C2, const float* __restrict__ img1, Plane lay,
    const float* __restrict__ img2, float* __restrict__ img1_copy, float* __restrict__ map,
    float* __restrict__ d_mu1, float* __restrict__ d_s11, float* __restrict__ d_s12,
    double* __restrict__ partial, int crop, int rows) {
  __shared__ float2 s_xy[3][64 + 2 * SS_R];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, nw = blockDim.x >> 6;
  const int groups = CH / nw, strips = (W + SR_OUT - 1) / SR_OUT;
  const int pg = blockIdx.x / strips;  // group of nw planes
  const int b = pg / groups, c = (pg % groups) * nw + wave;
  const int band = rows - 2 * SS_R;
  const int x0 = (blockIdx.x % strips) * SR_OUT, y0 = blockIdx.y * band;
  const int xi = x0 - SS_R + lane;
  const bool col_in = xi >= 0 && xi < W;
  const bool col_out = col_in && lane >= SS_R && lane < SS_R + SR_OUT;
  const bool col_sum = col_out && xi >= crop && xi < W - crop;
  const int xc = min(max(xi, 0), W - 1);
  const int64_t plane = ((int64_t)b * CH + c) * H * W;
  const float* p1 = img1 + b * lay.bs + c * lay.cs + xc * lay.xs;
  const float* p2 = img2 + plane + xc;
  float2* xy = s_xy[wave];
  const Taps wgt;
  // values of input row r, loaded from clamped (always valid) addresses
  // without a branch, so that the two-row prefetch really overlaps
  auto load_row = [&](int r, float& u, float& w) {
    const int rc = min(max(r, 0), H - 1);
    u = p1[rc * lay.ys];
    w = p2[(int64_t)rc * W];
  };
  float Hr[5][LR_RING];
#pragma unroll
  for (int k = 0; k < 5; ++k)
#pragma unroll
    for (int t = 0; t < LR_RING; ++t) Hr[k][t] = 0.f;
  const int ys = y0 - SS_R;  // first input row
  float u1, w1, u2, w2;
  load_row(ys, u1, w1);
  load_row(ys + 1, u2, w2);
  float m_acc = 0.f;

#pragma unroll 1
  for (int n0 = 0; n0 < rows; n0 += LR_RING) {
#pragma unroll
    for (int p = 0; p < LR_RING; ++p) {
      const int n = n0 + p;
      const int ri = ys + n;
      const bool ok = col_in && ri >= 0 && ri < H;
      const float u = ok ? u1 : 0.f, w = ok ? w1 : 0.f;
      u1 = u2;
      w1 = w2;
      load_row(ri + 2, u2, w2);
      xy[lane + SS_R] = make_float2(u, w);
      if (img1_copy && col_out && ok && ri >= y0 && ri < y0 + band)
        img1_copy[plane + (int64_t)ri * W + xi] = u;
      lr_wave_sync();
      float h0 = 0.f, h1 = 0.f, h2 = 0.f, h3 = 0.f, h4 = 0.f;
#pragma unroll
      for (int t = 0; t < 11; ++t) {
        const float2 v = xy[lane + t];
        const float wx = wgt(t) * v.x, wy = wgt(t) * v.y;
        h0 += wx;
        h1 += wy;
        h2 = fmaf(wx, v.x, h2);
        h3 = fmaf(wy, v.y, h3);
        h4 = fmaf(wx, v.y, h4);
      }
      Hr[0][p] = h0;
      Hr[1][p] = h1;
      Hr[2][p] = h2;
      Hr[3][p] = h3;
      Hr[4][p] = h4;
      lr_wave_sync();  // every lane has read the row before the next one is written
      if (n >= 2 * SS_R) {
        // output row from input rows ri - 10 .. ri (slots p+1 .. p+11)
        const int ro = ri - SS_R;
        float f[5];
#pragma unroll
        for (int k = 0; k < 5; ++k) {
          float acc = wgt(0) * Hr[k][(p + 1) % LR_RING];
#pragma unroll
          for (int t = 1; t < 11; ++t) acc = fmaf(wgt(t), Hr[k][(p + 1 + t) % LR_RING], acc);
          f[k] = acc;
        }
        if (col_out && ro < H) {
          const float mu1 = f[0], mu2 = f[1];
          const float sigma1_sq = f[2] - mu1 * mu1;
          const float sigma2_sq = f[3] - mu2 * mu2;
          const float sigma12 = f[4] - mu1 * mu2;
          const float Cc = 2.f * mu1 * mu2 + C1;
          const float D = 2.f * sigma12 + C2;
          const float A = mu1 * mu1 + mu2 * mu2 + C1;
          const float Bb = sigma1_sq + sigma2_sq + C2;
          const float r = 1.f / (A * Bb);
          const float CD = Cc * D;
          const float m = CD * r;
          const int64_t o = plane + (int64_t)ro * W + xi;
          if (map) map[o] = m;
          if (d_mu1) {
            const float rA = Bb * r, rB = A * r;  // 1/A, 1/Bb
            d_mu1[o] = 2.f * r * (mu2 * D - mu2 * Cc + mu1 * CD * (rB - rA));
            d_s11[o] = -CD * r * rB;
            d_s12[o] = 2.f * Cc * r;
          }
          if (col_sum && ro >= crop && ro < H - crop) m_acc += m;
        }
      }
    }
  }
  if (partial) {
    const float s = tgs_wave_sum(m_acc);
    if (lane == 0)
      partial[((int64_t)blockIdx.y * gridDim.x + blockIdx.x) * nw + wave] = (double)s;
  }
}

// Mean of the map from the wavefronts' sums, in a fixed order.
__global__ void __launch_bounds__(256) ssim_mean_kernel(const double* __restrict__ partial,
                                                        int64_t n, double count,
                                                        float* __restrict__ mean) {
  __shared__ double s[256];
  double acc = 0.0;
  for (int64_t i = threadIdx.x; i < n; i += 256) acc += partial[i];
  s[threadIdx.x] = acc;
  __syncthreads();
  for (int h = 128; h > 0; h >>= 1) {
    if ((int)threadIdx.x < h) s[threadIdx.x] += s[threadIdx.x + h];
    __syncthreads();
  }
  if (threadIdx.x == 0) *mean = (float)(s[0] / count);
}

// dL/dimg1 = G*(g dm/dmu1) + 2 x G*(g dm/dsigma1^2) + y G*(g dm/dsigma12), with
// g = dL/dmap read from `dmap`, or *g_mean / count inside the crop and 0 outside.
__global__ void __launch_bounds__(192) ssim_bwd_rows_kernel(
    int CH, int H, int W, const float* __restrict__ img1, const float* __restrict__ img2,
    const float* __restrict__ dmap, const float* __restrict__ g_mean, float count, int crop,
    const float* __restrict__ d_mu1, const float* __restrict__ d_s11,
    const float* __restrict__ d_s12, float* __restrict__ grad, Plane lay, int rows) {
  __shared__ float2 s_ab[3][64 + 2 * SS_R];
  __shared__ float s_c[3][64 + 2 * SS_R];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, nw = blockDim.x >> 6;
  const int groups = CH / nw, strips = (W + SR_OUT - 1) / SR_OUT;
  const int pg = blockIdx.x / strips;  // group of nw planes
  const int b = pg / groups, c = (pg % groups) * nw + wave;
  const int band = rows - 2 * SS_R;
  const int x0 = (blockIdx.x % strips) * SR_OUT, y0 = blockIdx.y * band;
  const int xi = x0 - SS_R + lane;
  const bool col_in = xi >= 0 && xi < W;
  const bool col_out = col_in && lane >= SS_R && lane < SS_R + SR_OUT;
  const bool col_g = xi >= crop && xi < W - crop;
  const int xc = min(max(xi, 0), W - 1);
  const int64_t plane = ((int64_t)b * CH + c) * H * W;
  const float g_const = dmap ? 0.f : *g_mean / count;
  const float *pa = d_mu1 + plane + xc, *pb = d_s11 + plane + xc, *pc = d_s12 + plane + xc;
  const float *px = img1 + plane + xc, *py = img2 + plane + xc;
  const float* pd = dmap ? dmap + plane + xc : nullptr;
  float* out = grad + b * lay.bs + c * lay.cs + xc * lay.xs;
  float2* ab = s_ab[wave];
  float* cc = s_c[wave];
  const Taps wgt;
  struct Row {
    float a, b, c, g, x, y;
  };
  // the partial maps (and dL/dmap) of row r, x and y of the output row r - 5
  auto load_row = [&](int r) {
    const int64_t in = (int64_t)min(max(r, 0), H - 1) * W;
    const int64_t o = (int64_t)min(max(r - SS_R, 0), H - 1) * W;
    Row v;
    v.a = pa[in];
    v.b = pb[in];
    v.c = pc[in];
    v.g = pd ? pd[in] : g_const;
    v.x = px[o];
    v.y = py[o];
    return v;
  };
  float Qr[3][LR_RING];
#pragma unroll
  for (int k = 0; k < 3; ++k)
#pragma unroll
    for (int t = 0; t < LR_RING; ++t) Qr[k][t] = 0.f;
  const int ys = y0 - SS_R;
  Row r1 = load_row(ys), r2 = load_row(ys + 1);

#pragma unroll 1
  for (int n0 = 0; n0 < rows; n0 += LR_RING) {
#pragma unroll
    for (int p = 0; p < LR_RING; ++p) {
      const int n = n0 + p;
      const int ri = ys + n;
      const Row cur = r1;
      r1 = r2;
      r2 = load_row(ri + 2);
      const bool ok = col_in && ri >= 0 && ri < H &&
                      (dmap || (col_g && ri >= crop && ri < H - crop));
      ab[lane + SS_R] = ok ? make_float2(cur.g * cur.a, cur.g * cur.b) : make_float2(0.f, 0.f);
      cc[lane + SS_R] = ok ? cur.g * cur.c : 0.f;
      lr_wave_sync();
      float q0 = 0.f, q1 = 0.f, q2 = 0.f;
#pragma unroll
      for (int t = 0; t < 11; ++t) {
        const float2 v = ab[lane + t];
        q0 = fmaf(wgt(t), v.x, q0);
        q1 = fmaf(wgt(t), v.y, q1);
        q2 = fmaf(wgt(t), cc[lane + t], q2);
      }
      Qr[0][p] = q0;
      Qr[1][p] = q1;
      Qr[2][p] = q2;
      lr_wave_sync();
      if (n >= 2 * SS_R) {
        const int ro = ri - SS_R;
        float f[3];
#pragma unroll
        for (int k = 0; k < 3; ++k) {
          float acc = wgt(0) * Qr[k][(p + 1) % LR_RING];
#pragma unroll
          for (int t = 1; t < 11; ++t) acc = fmaf(wgt(t), Qr[k][(p + 1 + t) % LR_RING], acc);
          f[k] = acc;
        }
        if (col_out && ro < H) out[ro * lay.ys] = f[0] + 2.f * cur.x * f[1] + cur.y * f[2];
      }
    }
  }
}

struct SsimGrid {
  dim3 grid, block;
  int rows;
};

// Bands: a lone workgroup's row takes 0.5 us forward and 0.6 us backward, about
// three times a busy CU's with the three wavefronts of an RGB workgroup and six
// times with one (its share of the CU is a third; a CU with several is fuller): one
// plane of 1080p in the bands of 3, 6 and 9 times 39, 24 and 23 us forward and 42,
// 24 and 32 backward (16x16 tiles: 30 and 39), 979x546 of two planes 21, 17, 17
// and 22, 17, 17.  Bands of more than 78 rows gain nothing (sixteen 1080p images,
// 45-, 78- and 133-row bands: forward 780, 758, 766 us, backward 664, 633, 734);
// one 256x256 image in 12-, 23- and 78-row bands: 15, 20, 49 us.
#define SSIM_LONE(nw) ((nw) == 1 ? 6.f : 3.f)
#define SSIM_PERIODS 8
static SsimGrid ssim_grid(int64_t B, int64_t CH, int H, int W) {
  const int nw = CH % 3 == 0 ? 3 : 1;
  const int64_t planes = B * (CH / nw);
  const int strips = (W + SR_OUT - 1) / SR_OUT;
  SsimGrid g;
  g.rows = band_input_rows(H, planes * strips, 2 * SS_R, SSIM_LONE(nw), SSIM_PERIODS);
  const int band = g.rows - 2 * SS_R;
  g.grid = dim3((unsigned)(planes * strips), (H + band - 1) / band);
  g.block = dim3(64 * nw);
  return g;
}

static Plane nchw(int CH, int H, int W) {
  return Plane{(int64_t)CH * H * W, (int64_t)H * W, W, 1};
}
static Plane nhwc(int CH, int H, int W) {
  return Plane{(int64_t)CH * H * W, 1, (int64_t)W * CH, CH};
}

extern "C" int tgs_fused_ssim_fwd(int32_t B, int32_t CH, int32_t H, int32_t W, float C1, float C2,
                                  const float* img1, const float* img2, float* ssim_map,
                                  float* dm_dmu1, float* dm_dsigma1_sq, float* dm_dsigma12,
                                  hipStream_t stream) {
  if ((int64_t)B * CH * H * W == 0) return TGS_OK;
  TGS_CHECK_ARG(img1 && img2 && ssim_map, "fused_ssim_fwd: null pointer");
  TGS_CHECK_ARG((dm_dmu1 && dm_dsigma1_sq && dm_dsigma12) ||
                    (!dm_dmu1 && !dm_dsigma1_sq && !dm_dsigma12),
                "fused_ssim_fwd: partial maps must be all set or all null");
  const SsimGrid g = ssim_grid(B, CH, H, W);
  hipLaunchKernelGGL(ssim_fwd_rows_kernel, g.grid, g.block, 0, stream, CH, H, W, C1, C2, img1,
                     nchw(CH, H, W), img2, (float*)nullptr, ssim_map, dm_dmu1, dm_dsigma1_sq,
                     dm_dsigma12, (double*)nullptr, 0, g.rows);
  TGS_RETURN_LAUNCH("tgs_fused_ssim_fwd");
}

extern "C" int tgs_fused_ssim_bwd(int32_t B, int32_t CH, int32_t H, int32_t W, float C1, float C2,
                                  const float* img1, const float* img2, const float* dL_dmap,
                                  const float* dm_dmu1, const float* dm_dsigma1_sq,
                                  const float* dm_dsigma12, float* dL_dimg1, hipStream_t stream) {
  (void)C1;
  (void)C2;
  if ((int64_t)B * CH * H * W == 0) return TGS_OK;
  TGS_CHECK_ARG(img1 && img2 && dL_dmap && dm_dmu1 && dm_dsigma1_sq && dm_dsigma12 && dL_dimg1,
                "fused_ssim_bwd: null pointer");
  const SsimGrid g = ssim_grid(B, CH, H, W);
  hipLaunchKernelGGL(ssim_bwd_rows_kernel, g.grid, g.block, 0, stream, CH, H, W, img1, img2,
                     dL_dmap, (const float*)nullptr, 1.f, 0, dm_dmu1, dm_dsigma1_sq, dm_dsigma12,
                     dL_dimg1, nchw(CH, H, W), g.rows);
  TGS_RETURN_LAUNCH("tgs_fused_ssim_bwd");
}

// One sum per wavefront of the launch; the buffer's size is no less than any
// smaller image's or batch's (of whatever channel count), so that one sized for the
// largest holds them all.
extern "C" uint64_t tgs_fused_ssim_mean_partials(int32_t B, int32_t CH, int32_t H, int32_t W) {
  if (B <= 0 || CH <= 0 || H <= 0 || W <= 0) return 0;
  const int64_t planes = (int64_t)B * CH, strips = (W + SR_OUT - 1) / SR_OUT;
  const auto most = [&](int64_t n, int nw) {
    return nw * band_workgroups_max(H, n * strips, 2 * SS_R, SSIM_LONE(nw), SSIM_PERIODS);
  };
  return (uint64_t)std::max(most(planes, 1), most((planes + 2) / 3, 3));
}

extern "C" int tgs_fused_ssim_mean_fwd(int32_t B, int32_t CH, int32_t H, int32_t W, float C1,
                                       float C2, const float* img1, int32_t channels_last,
                                       const float* img2, int32_t crop, double* partials,
                                       float* mean, float* img1_copy, float* dm_dmu1,
                                       float* dm_dsigma1_sq, float* dm_dsigma12,
                                       hipStream_t stream) {
  TGS_CHECK_ARG((int64_t)B * CH * H * W > 0 && crop >= 0 && H > 2 * crop && W > 2 * crop,
                "fused_ssim_mean_fwd: empty map");
  TGS_CHECK_ARG(img1 && img2 && partials && mean, "fused_ssim_mean_fwd: null pointer");
  TGS_CHECK_ARG((dm_dmu1 && dm_dsigma1_sq && dm_dsigma12) ||
                    (!dm_dmu1 && !dm_dsigma1_sq && !dm_dsigma12),
                "fused_ssim_mean_fwd: partial maps must be all set or all null");
  const SsimGrid g = ssim_grid(B, CH, H, W);
  hipLaunchKernelGGL(ssim_fwd_rows_kernel, g.grid, g.block, 0, stream, CH, H, W, C1, C2, img1,
                     channels_last ? nhwc(CH, H, W) : nchw(CH, H, W), img2, img1_copy,
                     (float*)nullptr, dm_dmu1, dm_dsigma1_sq, dm_dsigma12, partials, crop, g.rows);
  TGS_LAUNCH_CHECK("tgs_fused_ssim_mean_fwd");
  const double count = (double)B * CH * (H - 2 * crop) * (W - 2 * crop);
  hipLaunchKernelGGL(ssim_mean_kernel, dim3(1), dim3(256), 0, stream, partials,
                     (int64_t)g.grid.x * g.grid.y * (g.block.x / 64), count, mean);
  TGS_RETURN_LAUNCH("tgs_fused_ssim_mean_fwd");
}

extern "C" int tgs_fused_ssim_mean_bwd(int32_t B, int32_t CH, int32_t H, int32_t W,
                                       const float* img1, const float* img2, const float* dL_dmean,
                                       int32_t crop, const float* dm_dmu1,
                                       const float* dm_dsigma1_sq, const float* dm_dsigma12,
                                       float* dL_dimg1, int32_t channels_last,
                                       hipStream_t stream) {
  TGS_CHECK_ARG((int64_t)B * CH * H * W > 0 && crop >= 0 && H > 2 * crop && W > 2 * crop,
                "fused_ssim_mean_bwd: empty map");
  TGS_CHECK_ARG(img1 && img2 && dL_dmean && dm_dmu1 && dm_dsigma1_sq && dm_dsigma12 && dL_dimg1,
                "fused_ssim_mean_bwd: null pointer");
  const SsimGrid g = ssim_grid(B, CH, H, W);
  const float count = (float)((double)B * CH * (H - 2 * crop) * (W - 2 * crop));
  hipLaunchKernelGGL(ssim_bwd_rows_kernel, g.grid, g.block, 0, stream, CH, H, W, img1, img2,
                     (const float*)nullptr, dL_dmean, count, crop, dm_dmu1, dm_dsigma1_sq,
                     dm_dsigma12, dL_dimg1, channels_last ? nhwc(CH, H, W) : nchw(CH, H, W),
                     g.rows);
  TGS_RETURN_LAUNCH("tgs_fused_ssim_mean_bwd");
}

// Fused-step loss of strategies/base_engine.py:464-488 for a batch of B
// rendered images: per image b, L_b = (1-lambda) mean|I_b - gt'_b| +
// lambda (1 - mean SSIM(I_b, gt'_b)), gt' = clamp(gt / gt_div, 0, 1), with
// I [B,H,W,3] (HWC, as rendered) and gt [B,3,H,W] (CHW).  The loss is fixed,
// so dL/dSSIM-map is the constant -lambda/N and the forward and backward run
// in one streaming pass:
//   stats    mu, sigma (separable 11-tap window) giving SSIM and
//            g dm/dmu1, g dm/dsigma1^2, g dm/dsigma12 (zero off the image);
//   gradient G * (g dm): f0 + 2 x f1 + y f2, plus the L1 term.
// sums[2b] += sum|I-gt'|, sums[2b+1] += sum SSIM (double, caller-zeroed).
//
// One wavefront per (image, channel, strip of 44 output columns, band of
// output rows); lane L holds column x0 - 10 + L, so the strip's
// 64 columns cover the outputs and the 10-column halo on each side.  The
// wavefront walks the band's `rows` input rows top to bottom (20 more than it
// outputs: 10 rows of halo above and below) and keeps each stage's last 11 rows in
// registers, so no row is filtered twice:
//   input row r:   x, y into an 11-row LDS ring; horizontal window sums of
//                  x, y, x^2, y^2, xy at the lane's column -> register ring H;
//   stats row r-5: vertical window over H -> SSIM and the scaled partial maps
//                  (zero off the image), through LDS to the lanes' neighbours;
//                  horizontal window of the maps -> register ring Q;
//   output r-10:   vertical window over Q, plus the L1 term -> dL/dI.
// The three channel wavefronts of a strip and band share one workgroup (the
// HWC image rows they read and write are the same lines).  The step loop is
// unrolled by the ring length, so every ring index is a constant.
#define LR_OUT 44  // output columns per strip

__global__ void __launch_bounds__(192) tide_loss_rows_kernel(int H, int W,
                                                             const float* __restrict__ images_hwc,
                                                             const float* __restrict__ gt_chw,
                                                             float gt_div, float C1, float C2,
                                                             float g_ssim, float g_l1,
                                                             float* __restrict__ v_images_hwc,
                                                             double* __restrict__ sums,
                                                             double* __restrict__ partials,
                                                             int rows) {
  // per channel wavefront: ring of (x, y) rows and one row of scaled partial
  // maps, each padded by the window radius on both sides
  __shared__ float2 s_xy[3][LR_RING][64 + 2 * SS_R];
  __shared__ float4 s_dm[3][64 + 2 * SS_R];
  const int c = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int b = blockIdx.z;
  const int x0 = blockIdx.x * LR_OUT, y0 = blockIdx.y * (rows - 4 * SS_R);
  const int xi = x0 - 2 * SS_R + lane;
  const bool col_in = xi >= 0 && xi < W;
  const bool col_out = col_in && lane >= 2 * SS_R && lane < 2 * SS_R + LR_OUT;
  const int HW = H * W;
  const float* img = images_hwc + (int64_t)b * HW * 3 + c;
  const float* gtc = gt_chw + ((int64_t)b * 3 + c) * HW;
  float* vimg = v_images_hwc + (int64_t)b * HW * 3 + c;
  const float rdiv = 1.f / gt_div;
  float2(*xy)[64 + 2 * SS_R] = s_xy[c];
  float4* dm = s_dm[c];
  if (lane < 2 * SS_R) {
    const int e = lane < SS_R ? lane : 64 + lane;  // pads 0..4 and 69..73
#pragma unroll
    for (int k = 0; k < LR_RING; ++k) xy[k][e] = make_float2(0.f, 0.f);
    dm[e] = make_float4(0.f, 0.f, 0.f, 0.f);
  }
  // raw image and target values of input row r at the lane's column, loaded
  // from clamped (always valid) addresses without a branch, so that a fixed
  // number of loads is in flight and the two-row prefetch really overlaps
  const int xc = min(max(xi, 0), W - 1);
  auto load_row = [&](int r, float& u, float& g) {
    const int pix = min(max(r, 0), H - 1) * W + xc;
    u = img[pix * 3];
    g = gtc[pix];
  };
  const Taps wgt;

  float Hr[5][LR_RING];  // horizontal sums of the last 11 input rows
  float Qr[3][LR_RING];  // horizontal sums of the partial maps, last 11 stats rows
#pragma unroll
  for (int k = 0; k < 5; ++k)
#pragma unroll
    for (int t = 0; t < LR_RING; ++t) Hr[k][t] = 0.f;
#pragma unroll
  for (int k = 0; k < 3; ++k)
#pragma unroll
    for (int t = 0; t < LR_RING; ++t) Qr[k][t] = 0.f;
  const int ys = y0 - 2 * SS_R;  // first input row
  float u1, g1, u2, g2;          // raw inputs of the next two rows
  load_row(ys, u1, g1);
  load_row(ys + 1, u2, g2);
  float l1_acc = 0.f, m_acc = 0.f;

#pragma unroll 1
  for (int n0 = 0; n0 < rows; n0 += LR_RING) {
#pragma unroll
    for (int p = 0; p < LR_RING; ++p) {
      const int n = n0 + p;
      const int ri = ys + n;
      // x and clamp(gt / gt_div, 0, 1) of row ri (zero off the image); the
      // division is rounded like a division: product plus one residual correction
      const bool ok = col_in && ri >= 0 && ri < H;
      float q = g1 * rdiv;
      q = fmaf(fmaf(-q, gt_div, g1), rdiv, q);
      const float u = ok ? u1 : 0.f, w = ok ? fminf(fmaxf(q, 0.f), 1.f) : 0.f;
      u1 = u2;
      g1 = g2;
      load_row(ri + 2, u2, g2);
      // input row ri: ring slot p
      xy[p][lane + SS_R] = make_float2(u, w);
      lr_wave_sync();
      {
        float wx[11], wy[11], xv[11], yv[11];
#pragma unroll
        for (int t = 0; t < 11; ++t) {
          const float2 v = xy[p][lane + t];
          xv[t] = v.x;
          yv[t] = v.y;
          wx[t] = wgt(t) * v.x;
          wy[t] = wgt(t) * v.y;
        }
        float h0 = wx[0], h1 = wy[0], h2 = wx[0] * xv[0], h3 = wy[0] * yv[0],
              h4 = wx[0] * yv[0];
#pragma unroll
        for (int t = 1; t < 11; ++t) {
          h0 += wx[t];
          h1 += wy[t];
          h2 = fmaf(wx[t], xv[t], h2);
          h3 = fmaf(wy[t], yv[t], h3);
          h4 = fmaf(wx[t], yv[t], h4);
        }
        Hr[0][p] = h0;
        Hr[1][p] = h1;
        Hr[2][p] = h2;
        Hr[3][p] = h3;
        Hr[4][p] = h4;
      }
      if (n >= 2 * SS_R) {
        // stats row rs = ri - 5 from input rows ri - 10 .. ri (slots p+1 .. p+11)
        const int rs = ri - SS_R;
        float f[5];
#pragma unroll
        for (int k = 0; k < 5; ++k) {
          float acc = wgt(0) * Hr[k][(p + 1) % LR_RING];
#pragma unroll
          for (int t = 1; t < 11; ++t) acc = fmaf(wgt(t), Hr[k][(p + 1 + t) % LR_RING], acc);
          f[k] = acc;
        }
        const float mu1 = f[0], mu2 = f[1];
        const float sigma1_sq = f[2] - mu1 * mu1;
        const float sigma2_sq = f[3] - mu2 * mu2;
        const float sigma12 = f[4] - mu1 * mu2;
        const float Cc = 2.f * mu1 * mu2 + C1;
        const float D = 2.f * sigma12 + C2;
        const float A = mu1 * mu1 + mu2 * mu2 + C1;
        const float Bb = sigma1_sq + sigma2_sq + C2;
        float d0 = 0.f, d1 = 0.f, d2 = 0.f;
        if (col_in && rs >= 0 && rs < H) {
          // the partial maps of clm_kernels/ssim.cu:240-262 from two
          // reciprocals; A >= C1 and Bb >= C2 - (rounding) > 0, so the
          // hardware reciprocal (within 1 ulp) is safe here
          const float rA = __builtin_amdgcn_rcpf(A), rB = __builtin_amdgcn_rcpf(Bb);
          const float rAB = rA * rB;
          const float CD = Cc * D;
          d0 = 2.f * rAB * (mu2 * D - mu2 * Cc + mu1 * CD * (rB - rA));
          d1 = -CD * rAB * rB;
          d2 = 2.f * Cc * rAB;
          if (col_out && rs >= y0 && rs < y0 + rows - 4 * SS_R) m_acc += CD * rAB;
        }
        dm[lane + SS_R] = make_float4(g_ssim * d0, g_ssim * d1, g_ssim * d2, 0.f);
        lr_wave_sync();
        float q0 = 0.f, q1 = 0.f, q2 = 0.f;
#pragma unroll
        for (int t = 0; t < 11; ++t) {
          const float4 v = dm[lane + t];
          q0 = fmaf(wgt(t), v.x, q0);
          q1 = fmaf(wgt(t), v.y, q1);
          q2 = fmaf(wgt(t), v.z, q2);
        }
        Qr[0][p] = q0;
        Qr[1][p] = q1;
        Qr[2][p] = q2;
      }
      if (n >= 4 * SS_R) {
        // output row ro = ri - 10 from stats rows ro - 5 .. ro + 5 (slots p+1 .. p+11)
        const int ro = ri - 2 * SS_R;
        float g3[3];
#pragma unroll
        for (int k = 0; k < 3; ++k) {
          float acc = wgt(0) * Qr[k][(p + 1) % LR_RING];
#pragma unroll
          for (int t = 1; t < 11; ++t) acc = fmaf(wgt(t), Qr[k][(p + 1 + t) % LR_RING], acc);
          g3[k] = acc;
        }
        if (col_out && ro < H) {
          const float2 v = xy[(p + 1) % LR_RING][lane + SS_R];  // x, y of row ro
          const float d = v.x - v.y;
          l1_acc += fabsf(d);
          vimg[(ro * W + xi) * 3] = g3[0] + 2.f * v.x * g3[1] + v.y * g3[2] +
                                    (d > 0.f ? g_l1 : (d < 0.f ? -g_l1 : 0.f));
        }
      }
      // every lane has read this step's rows before the next step writes
      lr_wave_sync();
    }
  }
  const float l1 = tgs_wave_sum(l1_acc);
  const float ms = tgs_wave_sum(m_acc);
  __shared__ float s_red[3][2];
  if (lane == 0) {
    s_red[c][0] = l1;
    s_red[c][1] = ms;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    const double l1_sum = (double)s_red[0][0] + s_red[1][0] + s_red[2][0];
    const double m_sum = (double)s_red[0][1] + s_red[1][1] + s_red[2][1];
    if (partials) {
      double* o = partials + 2 * (((int64_t)b * gridDim.y + blockIdx.y) * gridDim.x + blockIdx.x);
      o[0] = l1_sum;
      o[1] = m_sum;
    } else {
      atomicAdd(&sums[2 * b + 0], l1_sum);
      atomicAdd(&sums[2 * b + 1], m_sum);
    }
  }
}

// sums[2b], sums[2b + 1] from image b's workgroup sums, in a fixed order.
__global__ void __launch_bounds__(128) tide_loss_sums_kernel(const double* __restrict__ partials,
                                                             int per_image,
                                                             double* __restrict__ sums) {
  __shared__ double s[128];
  const double* p = partials + 2 * (int64_t)blockIdx.x * per_image;
  double acc = 0.0;  // even threads L1, odd threads SSIM
  for (int i = threadIdx.x; i < 2 * per_image; i += 128) acc += p[i];
  s[threadIdx.x] = acc;
  __syncthreads();
  for (int h = 64; h >= 2; h >>= 1) {
    if ((int)threadIdx.x < h) s[threadIdx.x] += s[threadIdx.x + h];
    __syncthreads();
  }
  if (threadIdx.x < 2) sums[2 * blockIdx.x + threadIdx.x] = s[threadIdx.x];
}

struct LossGrid {
  dim3 grid;
  int rows;
};

// A lone workgroup takes 0.71 us per row, four on a CU 1.2 us: 2.4 times a busy
// CU's 0.3 us per row and workgroup.  Bands of 123 rows at every size, the rule
// before, left small batches to a few long-running wavefronts: one 256x256 image
// 104 -> 26 us, four 979x546 132 -> 103, one 1080p 133 -> 96; sixteen 1080p images
// keep the 123 rows (1.10 ms; in 13-row bands 1.86).
#define LOSS_LONE 2.4f
#define LOSS_PERIODS 13
static LossGrid loss_grid(int B, int H, int W) {
  LossGrid g;
  const int strips = (W + LR_OUT - 1) / LR_OUT;
  g.rows = band_input_rows(H, (int64_t)strips * B, 4 * SS_R, LOSS_LONE, LOSS_PERIODS);
  const int band = g.rows - 4 * SS_R;
  g.grid = dim3(strips, (H + band - 1) / band, B);
  return g;
}

static int launch_tide_loss(int32_t B, int32_t H, int32_t W, const float* images_hwc,
                            const float* gt_chw, float gt_div, float lambda_dssim, double* sums,
                            double* partials, float* v_images_hwc, hipStream_t stream) {
  TGS_CHECK_ARG(images_hwc && gt_chw && sums && v_images_hwc, "tide_loss: null pointer");
  TGS_CHECK_ARG((int64_t)H * W * 3 < (1ll << 31), "tide_loss: image too large");
  const float inv_n = 1.f / (float)((int64_t)3 * H * W);
  TGS_CHECK_ARG(B <= 65535, "tide_loss: more than 65535 images");
  const LossGrid g = loss_grid(B, H, W);
  hipLaunchKernelGGL(tide_loss_rows_kernel, g.grid, dim3(192), 0, stream, H, W, images_hwc, gt_chw,
                     gt_div, 1e-4f, 9e-4f, -lambda_dssim * inv_n, (1.f - lambda_dssim) * inv_n,
                     v_images_hwc, sums, partials, g.rows);
  if (partials) {
    TGS_LAUNCH_CHECK("tgs_tide_loss");
    hipLaunchKernelGGL(tide_loss_sums_kernel, dim3(B), dim3(128), 0, stream, partials,
                       (int)(g.grid.x * g.grid.y), sums);
  }
  TGS_RETURN_LAUNCH("tgs_tide_loss");
}

extern "C" int tgs_tide_loss(int32_t B, int32_t H, int32_t W, const float* images_hwc,
                             const float* gt_chw, float gt_div, float lambda_dssim, double* sums,
                             float* v_images_hwc, hipStream_t stream) {
  if ((int64_t)B * H * W == 0) return TGS_OK;
  return launch_tide_loss(B, H, W, images_hwc, gt_chw, gt_div, lambda_dssim, sums, nullptr,
                          v_images_hwc, stream);
}

// The same with the sums written (not added to): every workgroup leaves its own
// in `partials` and a small launch adds them in a fixed order.  The atomics of
// the other form queue on one image's two addresses (one 979x546 image in 33-row
// bands: 966 workgroups, 95 us with one atomic per wavefront).
// (Two sums per workgroup; the buffer's size is no less than any smaller image's or
// batch's.)
extern "C" uint64_t tgs_tide_loss_partials(int32_t B, int32_t H, int32_t W) {
  if (B <= 0 || H <= 0 || W <= 0) return 0;
  return 2ull * (uint64_t)band_workgroups_max(H, (int64_t)((W + LR_OUT - 1) / LR_OUT) * B, 4 * SS_R,
                                              LOSS_LONE, LOSS_PERIODS);
}

extern "C" int tgs_tide_loss_summed(int32_t B, int32_t H, int32_t W, const float* images_hwc,
                                    const float* gt_chw, float gt_div, float lambda_dssim,
                                    double* partials, double* sums, float* v_images_hwc,
                                    hipStream_t stream) {
  if ((int64_t)B * H * W == 0) return TGS_OK;
  TGS_CHECK_ARG(partials, "tide_loss_summed: null pointer");
  return launch_tide_loss(B, H, W, images_hwc, gt_chw, gt_div, lambda_dssim, sums, partials,
                          v_images_hwc, stream);
}
