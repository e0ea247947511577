// Camera staging of one fused-PRoPE forward on gfx950 (skv_prope_stage): the staged frames' cameras
// into the camera store and the forward's tables for every layer's attention, in one launch.
// Reference: causal_model.py:1948-2066 (staging), camera_prope.py:206-231 (P and its inverse).
//
// The work is tiny (a 4x4 product per query frame, key frame and channel group) and was bound by
// launches: as tensor operations it took some 66 kernels a forward, 210 us of GPU time plus the gaps
// between them.  A 30-layer forward (24 heads, 1215 queries over 18 frames, with append and commit)
// went from 5.43 to 4.78 ms with this one launch in their place.  One block a key frame keeps P_k^-1
// uniform; the query frame's P is recomputed by each (frame, group) thread, which is cheaper than an
// exchange.  Everything is float64 until the stored values, as the tensor operations are.
#include <stdint.h>

#include "skv_common.h"

namespace skv {

namespace {

constexpr int kGroups = 11;  // channel groups of 4 that hold temporal RoPE pairs only

struct StageArgs {
  const float* view;    // raw view matrices of the chunk's frames, [B][nb] 4x4 rows
  const float* view_t;  // the same after the translation transform (view itself when linear)
  const float* ks;      // intrinsics, [B][nb] 3x3 rows
  int64_t v_sb, v_sf, t_sb, t_sf, k_sb, k_sf;  // element strides (stream, frame)
  float* store_view;
  float* store_k;
  float* store_inv;
  float* kv_xform;
  float* q_xform_t;
  float* q_xform_s;
  float* out_xform;
  int B, nb, n_keys, n_staged, first;
  int q_pos0, q_step;
  double inv_freq[2 * kGroups];
  int32_t window[SKV_MAX_FRAMES];
  int32_t k_pos[SKV_MAX_FRAMES];
  int32_t staged[SKV_MAX_APPEND_FRAMES];
  int32_t keep[SKV_MAX_APPEND_FRAMES];  // the slot whose camera staged frame i keeps, or -1
};

// P = diag(fx, fy, 1, 1) V and P^-1 = V^-1 diag(1/fx, 1/fy, 1, 1), V^-1 = [R^T  -R^T t; 0 1]
__device__ inline void project(const float* v, const float* k, double (&p)[16], double (&pi)[16]) {
  double m[16];
#pragma unroll
  for (int i = 0; i < 16; ++i) m[i] = (double)v[i];
  const double d[4] = {(double)k[0], (double)k[4], 1.0, 1.0};
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) p[4 * i + j] = d[i] * m[4 * i + j];
#pragma unroll
  for (int i = 0; i < 3; ++i) {
    double t = 0.0;
#pragma unroll
    for (int j = 0; j < 3; ++j) {
      pi[4 * i + j] = m[4 * j + i] / d[j];
      t += m[4 * j + i] * m[4 * j + 3];
    }
    pi[4 * i + 3] = -t / d[3];
  }
  pi[12] = pi[13] = pi[14] = 0.0;
  pi[15] = 1.0;
}

// grid (n_keys + 1, B), block 256.  Block (j, b) builds W = R_k^T (P_q P_k^-1)^T R_q of key frame j
// for every query frame and group; block (n_keys, b) stores the staged frames' cameras and the query
// frames' matrices.  A key frame staged by this launch takes its camera from the inputs (rounded as
// it is stored), not from the store another block is writing.
__global__ __launch_bounds__(256) void prope_stage_kernel(StageArgs a) {
  const int j = blockIdx.x, b = blockIdx.y, tid = threadIdx.x;
  const float* vt = a.view_t + (int64_t)b * a.t_sb;
  const float* vr = a.view + (int64_t)b * a.v_sb;
  const float* kk = a.ks + (int64_t)b * a.k_sb;
  double p[16], pi[16];
  if (j == a.n_keys) {
    for (int i = tid; i < a.n_staged; i += 256) {
      const int64_t dst = (int64_t)a.staged[i] * a.B + b;
      const float *sv, *sk;
      float inv[16];
      if (a.keep[i] >= 0) {
        const int64_t old = (int64_t)a.keep[i] * a.B + b;
        sv = a.store_view + old * 16;
        sk = a.store_k + old * 9;
        for (int e = 0; e < 16; ++e) inv[e] = a.store_inv[old * 16 + e];
      } else {
        const int f = a.first + i;
        sv = vr + (int64_t)f * a.v_sf;
        sk = kk + (int64_t)f * a.k_sf;
        project(vt + (int64_t)f * a.t_sf, sk, p, pi);
        for (int e = 0; e < 16; ++e) inv[e] = (float)pi[e];
      }
      for (int e = 0; e < 16; ++e) {
        a.store_view[dst * 16 + e] = sv[e];
        a.store_inv[dst * 16 + e] = inv[e];
        a.kv_xform[((int64_t)i * a.B + b) * 16 + e] = inv[e];
      }
      for (int e = 0; e < 9; ++e) a.store_k[dst * 9 + e] = sk[e];
    }
    for (int f = tid; f < a.nb; f += 256) {
      project(vt + (int64_t)f * a.t_sf, kk + (int64_t)f * a.k_sf, p, pi);
      const int64_t o = ((int64_t)b * a.nb + f) * 16;
      for (int r = 0; r < 4; ++r)
        for (int c = 0; c < 4; ++c) {
          a.out_xform[o + 4 * r + c] = (float)p[4 * r + c];
          a.q_xform_s[o + 4 * r + c] = (float)p[4 * c + r];
        }
    }
    return;
  }
  const int slot = a.window[j];
  int from = -1;  // the staged frame in this slot
  for (int i = 0; i < a.n_staged; ++i)
    if (a.staged[i] == slot) from = i;
  const int keep = from >= 0 ? a.keep[from] : slot;
  double pk[16];
  if (keep >= 0) {
    const float* s = a.store_inv + ((int64_t)keep * a.B + b) * 16;
#pragma unroll
    for (int e = 0; e < 16; ++e) pk[e] = (double)s[e];
  } else {
    const int f = a.first + from;
    project(vt + (int64_t)f * a.t_sf, kk + (int64_t)f * a.k_sf, p, pi);
#pragma unroll
    for (int e = 0; e < 16; ++e) pk[e] = (double)(float)pi[e];
  }
  for (int i = tid; i < a.nb * kGroups; i += 256) {
    const int f = i / kGroups, g = i - f * kGroups;
    project(vt + (int64_t)f * a.t_sf, kk + (int64_t)f * a.k_sf, p, pi);
    double m[16];  // A = P_q P_k^-1
#pragma unroll
    for (int r = 0; r < 4; ++r)
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        double s = 0.0;
#pragma unroll
        for (int k = 0; k < 4; ++k) s += p[4 * r + k] * pk[4 * k + c];
        m[4 * r + c] = s;
      }
    const double qp = (double)(a.q_pos0 + f * a.q_step), kp = (double)a.k_pos[j];
    double ck[2], sk[2], cq[2], sq[2];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const double w = a.inv_freq[2 * g + h];
      sincos(kp * w, &sk[h], &ck[h]);
      sincos(qp * w, &sq[h], &cq[h]);
    }
    float* o = a.q_xform_t + ((((int64_t)b * a.n_keys + j) * a.nb + f) * kGroups + g) * 16;
    // rows 2h, 2h + 1 of R^T A^T: [c s; -s c] on columns 2h, 2h + 1 of A; R_q likewise on the right
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      double t[2][4];
#pragma unroll
      for (int l = 0; l < 4; ++l) {
        const double x = m[4 * l + 2 * h], y = m[4 * l + 2 * h + 1];
        t[0][l] = ck[h] * x + sk[h] * y;
        t[1][l] = -sk[h] * x + ck[h] * y;
      }
#pragma unroll
      for (int r = 0; r < 2; ++r)
#pragma unroll
        for (int q = 0; q < 2; ++q) {
          const double x = t[r][2 * q], y = t[r][2 * q + 1];
          o[4 * (2 * h + r) + 2 * q] = (float)(x * cq[q] + y * sq[q]);
          o[4 * (2 * h + r) + 2 * q + 1] = (float)(-x * sq[q] + y * cq[q]);
        }
    }
  }
}

}  // namespace

}  // namespace skv

using namespace skv;

extern "C" int skv_prope_stage(const skv_prope_stage_desc* d, skv_stream_t stream) {
  clear_error();
  if (!d || !d->view || !d->view_t || !d->ks || !d->store_view || !d->store_k || !d->store_inv ||
      !d->q_xform_t || !d->q_xform_s || !d->out_xform || !d->window || !d->k_pos || !d->inv_freq) {
    set_error("skv_prope_stage: null descriptor or pointer");
    return SKV_E_ARG;
  }
  if (d->batch <= 0 || d->batch > 65535 || d->n_qframes <= 0 || d->n_keys <= 0 ||
      d->n_keys > SKV_MAX_FRAMES || d->n_staged < 0 || d->n_staged > SKV_MAX_APPEND_FRAMES ||
      d->first < 0 || (int64_t)d->first + d->n_staged > d->n_qframes || d->n_slots <= 0) {
    set_error("skv_prope_stage: bad sizes (batch=%d n_qframes=%d n_keys=%d n_staged=%d first=%d n_slots=%d)",
              d->batch, d->n_qframes, d->n_keys, d->n_staged, d->first, d->n_slots);
    return SKV_E_ARG;
  }
  if (d->n_staged > 0 && (!d->kv_xform || !d->staged || !d->keep)) {
    set_error("skv_prope_stage: staged frames need kv_xform, staged and keep");
    return SKV_E_ARG;
  }
  StageArgs a;
  a.view = d->view, a.view_t = d->view_t, a.ks = d->ks;
  a.v_sb = d->view_sb, a.v_sf = d->view_sf, a.t_sb = d->view_t_sb, a.t_sf = d->view_t_sf;
  a.k_sb = d->ks_sb, a.k_sf = d->ks_sf;
  a.store_view = d->store_view, a.store_k = d->store_k, a.store_inv = d->store_inv;
  a.kv_xform = d->kv_xform, a.q_xform_t = d->q_xform_t, a.q_xform_s = d->q_xform_s;
  a.out_xform = d->out_xform;
  a.B = d->batch, a.nb = d->n_qframes, a.n_keys = d->n_keys, a.n_staged = d->n_staged;
  a.first = d->first, a.q_pos0 = d->q_pos0, a.q_step = d->q_step;
  for (int i = 0; i < 2 * kGroups; ++i) a.inv_freq[i] = d->inv_freq[i];
  for (int i = 0; i < d->n_keys; ++i) {
    if (d->window[i] < 0 || d->window[i] >= d->n_slots) {
      set_error("skv_prope_stage: window[%d]=%d outside [0, %d)", i, d->window[i], d->n_slots);
      return SKV_E_ARG;
    }
    a.window[i] = d->window[i];
    a.k_pos[i] = d->k_pos[i];
  }
  for (int i = 0; i < d->n_staged; ++i) {
    if (d->staged[i] < 0 || d->staged[i] >= d->n_slots || d->keep[i] >= d->n_slots) {
      set_error("skv_prope_stage: staged[%d]=%d / keep=%d outside [0, %d)", i, d->staged[i],
                d->keep[i], d->n_slots);
      return SKV_E_ARG;
    }
    a.staged[i] = d->staged[i];
    a.keep[i] = d->keep[i];
  }
  for (int i = 0; i < d->n_staged; ++i)  // a kept camera must not be overwritten by this launch
    for (int k = 0; k < d->n_staged; ++k)
      if (a.keep[i] == a.staged[k] || (i != k && a.staged[i] == a.staged[k])) {
        set_error("skv_prope_stage: staged slot %d is kept from or staged twice", a.staged[k]);
        return SKV_E_ARG;
      }
  hipLaunchKernelGGL(prope_stage_kernel, dim3(a.n_keys + 1, a.B), dim3(256), 0,
                     static_cast<hipStream_t>(stream), a);
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) {
    set_error("skv_prope_stage: launch failed: %s", hipGetErrorString(e));
    return SKV_E_LAUNCH;
  }
  return SKV_OK;
}
