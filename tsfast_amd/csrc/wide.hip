// Weight layouts and gradient sums of the projected scan's wide route (projections by GEMMs around
// the diagonal scan kernels), one launch each way.
//
// The route's GEMMs take the complex weights as real ones with re and im interleaved
// (tsfast/models/_core/scan.py:272-313 writes the same products): w [2N, H] rows 2s, 2s + 1 =
// W_re[s], W_im[s], and c [O, 2N] columns 2s, 2s + 1 = C_re[:, s], -C_im[:, s]; the scan takes lam
// once per batch row. The backward's weight gradients come as split-K partial products in the same
// layouts and grad lam once per batch row. As torch operations (stack, neg, expand, sum over the
// partials, strided copies) these were 14 launches of 3-6 us per forward and backward and most of
// the small calls' host time; both kernels are bound by their own launch.
#include "common.h"
#include "tsfast_hip.h"

using namespace tsf;

namespace {

constexpr int kThreads = 256;

__global__ void __launch_bounds__(kThreads) wide_pack(int64_t B, int64_t H, int64_t N, int64_t O,
                                                      const float* __restrict__ W_re, const float* __restrict__ W_im,
                                                      const float2* __restrict__ lam, const float* __restrict__ C_re,
                                                      const float* __restrict__ C_im, float* __restrict__ w,
                                                      float2* __restrict__ c, float2* __restrict__ rows) {
  const int64_t nw = 2 * N * H, nc = O * N, total = nw + nc + B * N;
  for (int64_t i = blockIdx.x * (int64_t)kThreads + threadIdx.x; i < total; i += gridDim.x * (int64_t)kThreads) {
    if (i < nw) {
      const int64_t r = i / H, h = i - r * H;
      w[i] = ((r & 1) ? W_im : W_re)[(r >> 1) * H + h];
    } else if (i < nw + nc) {
      const int64_t q = i - nw;
      c[q] = make_float2(C_re[q], -C_im[q]);
    } else {
      const int64_t q = i - nw - nc;
      rows[q] = lam[q % N];
    }
  }
}

// Blocks [0, nb): one thread per (s, h) of grad W, then per (o, s) of grad C: the partials added in
// order, in fp64. The other blocks: grad lam, 16 states a block, each state's rows over 16 threads
// (thread j rows j, j + 16, ..), then the 16 sums in order.
__global__ void __launch_bounds__(kThreads) wide_unpack(int64_t B, int64_t H, int64_t N, int64_t O, int64_t parts_w,
                                                        int64_t parts_c, const float* __restrict__ gw,
                                                        const float2* __restrict__ gc, const float2* __restrict__ rows,
                                                        float* __restrict__ gW_re, float* __restrict__ gW_im,
                                                        float2* __restrict__ glam, float* __restrict__ gC_re,
                                                        float* __restrict__ gC_im, unsigned nb) {
  __shared__ double2 red[16][17];
  if (blockIdx.x < nb) {
    const int64_t i = blockIdx.x * (int64_t)kThreads + threadIdx.x, nw = N * H, nc = O * N;
    double re = 0.0, im = 0.0;
    if (i < nw) {
      const int64_t s = i / H, h = i - s * H;
      for (int64_t p = 0; p < parts_w; ++p) {
        const float* q = gw + (p * 2 * N + 2 * s) * H + h;
        re += (double)q[0];
        im += (double)q[H];
      }
      gW_re[i] = (float)re;
      gW_im[i] = (float)im;
    } else if (i < nw + nc) {
      const int64_t q = i - nw;
      for (int64_t p = 0; p < parts_c; ++p) {
        const float2 v = gc[p * nc + q];
        re += (double)v.x;
        im += (double)v.y;
      }
      gC_re[q] = (float)re;
      gC_im[q] = (float)-im;
    }
    return;
  }
  const int js = threadIdx.x & 15, jr = threadIdx.x >> 4;
  const int64_t s = (blockIdx.x - nb) * (int64_t)16 + js;
  double2 acc = make_double2(0.0, 0.0);
  if (s < N)
    for (int64_t b = jr; b < B; b += 16) {
      const float2 v = rows[b * N + s];
      acc.x += (double)v.x;
      acc.y += (double)v.y;
    }
  red[jr][js] = acc;
  __syncthreads();
  if (jr == 0 && s < N) {
    double2 t = red[0][js];
    for (int j = 1; j < 16; ++j) {
      t.x += red[j][js].x;
      t.y += red[j][js].y;
    }
    glam[s] = make_float2((float)t.x, (float)t.y);
  }
}

int args_status(int64_t B, int64_t H, int64_t N, int64_t O) {
  if (B < 0 || H < 0 || N < 0 || O < 0) return TSF_ERR_ARG;
  const int64_t lim = (int64_t)1 << 38;  // the blocks of a launch stay below 2^31
  if (N > 0 && (H > lim / N || O > lim / N)) return TSF_ERR_UNSUPPORTED;
  return TSF_OK;
}

}  // namespace

extern "C" {

int tsfast_hip_wide_pack(int64_t B, int64_t H, int64_t N, int64_t O, const float* W_re, const float* W_im,
                         const void* lam, const float* C_re, const float* C_im, float* w, float* c, void* lam_rows,
                         void* stream) {
  if (const int rc = args_status(B, H, N, O)) return rc;
  const int64_t total = 2 * N * H + O * N + B * N;
  if (total == 0) return TSF_OK;
  if ((N * H > 0 && (!W_re || !W_im || !w)) || (O * N > 0 && (!C_re || !C_im || !c)) ||
      (B * N > 0 && (!lam || !lam_rows)))
    return TSF_ERR_ARG;
  const int64_t blocks = (total + kThreads - 1) / kThreads;
  hipLaunchKernelGGL(wide_pack, dim3((unsigned)(blocks < 4096 ? blocks : 4096)), dim3(kThreads), 0,
                     static_cast<hipStream_t>(stream), B, H, N, O, W_re, W_im, static_cast<const float2*>(lam), C_re,
                     C_im, w, reinterpret_cast<float2*>(c), static_cast<float2*>(lam_rows));
  return tsf_launch_status();
}

int tsfast_hip_wide_unpack(int64_t B, int64_t H, int64_t N, int64_t O, int64_t parts_w, int64_t parts_c,
                           const float* gw, const float* gc, const void* glam_rows, float* gW_re, float* gW_im,
                           void* glam, float* gC_re, float* gC_im, void* stream) {
  if (const int rc = args_status(B, H, N, O)) return rc;
  if (parts_w < 0 || parts_c < 0) return TSF_ERR_ARG;
  if (N == 0) return TSF_OK;
  if ((H > 0 && (!gW_re || !gW_im || (parts_w > 0 && !gw))) || (O > 0 && (!gC_re || !gC_im || (parts_c > 0 && !gc))) ||
      !glam || (B > 0 && !glam_rows))
    return TSF_ERR_ARG;
  const unsigned nb = (unsigned)((N * H + O * N + kThreads - 1) / kThreads), nl = (unsigned)((N + 15) / 16);
  hipLaunchKernelGGL(wide_unpack, dim3(nb + nl), dim3(kThreads), 0, static_cast<hipStream_t>(stream), B, H, N, O, parts_w,
                     parts_c, gw, reinterpret_cast<const float2*>(gc), static_cast<const float2*>(glam_rows), gW_re,
                     gW_im, static_cast<float2*>(glam), gC_re, gC_im, nb);
  return tsf_launch_status();
}

}  // extern "C"
