// ne_wavefront.h -- device functions shared by the staged wavefront pipeline
// (wavefront.hip) and the persistent volume path kernel (paths.hip): path ids
// to pixels, per-sample film slots, and the light sample of a vertex.
#pragma once
#include "ne_launch.h"
#include "ne_trace.h"

namespace ne {

// id / n and id % n for a path id and 0 < n < 2^32 with a quotient below
// 2^32.  The correctly rounded double quotient is within 2^-20 of the true
// one, so its floor is the true quotient or one off, and one correction step
// each way makes it exact (a few instructions instead of a 64-bit integer
// division).
__device__ __forceinline__ void divmod_id(unsigned long long id, uint32_t n, uint32_t& q, uint32_t& r) {
  const double e = floor(double(id) / double(n));
  long long qq = (long long)e;
  long long rr = (long long)id - qq * (long long)n;
  if (rr < 0) { qq -= 1; rr += n; }
  if (rr >= (long long)n) { qq += 1; rr -= n; }
  q = uint32_t(qq);
  r = uint32_t(rr);
}

// path id -> (pixel, sample): one sample index at a time over the rect; full
// 8x8 tiles first (row-major tile order), then the right strip, then the
// bottom strip (row-major): a bijection onto the rect.  (px, py): the pixel's
// coordinates within the rect.  Rects hold at most 2^30 pixels and renders
// fewer than 2^32 samples per pixel.
__device__ __forceinline__ void path_pixel(const WfArgs& a, unsigned long long id, uint32_t& pix, uint32_t& smp,
                                           uint32_t& px, uint32_t& py) {
  const uint32_t rw = uint32_t(a.x1 - a.x0), rh = uint32_t(a.y1 - a.y0);
  uint32_t p;
  divmod_id(id, rw * rh, smp, p);
  const uint32_t full_rows = rh / 8, full_cols = rw / 8;
  const uint32_t tiles_full = full_rows * full_cols;
  if (p < tiles_full * 64) {
    const uint32_t t = p / 64, l = p % 64;
    const uint32_t ty = t / full_cols;
    px = (t - ty * full_cols) * 8 + (l & 7);
    py = ty * 8 + (l >> 3);
  } else {
    uint32_t r = p - tiles_full * 64;
    const uint32_t strip_w = rw - full_cols * 8;
    const uint32_t right = strip_w * full_rows * 8;
    if (r < right) {
      px = full_cols * 8 + r % strip_w;
      py = r / strip_w;
    } else {
      r -= right;
      px = r % rw;
      py = full_rows * 8 + r / rw;
    }
  }
  pix = uint32_t(a.y0 + int(py)) * uint32_t(a.W) + uint32_t(a.x0 + int(px));
}

// Per-sample radiance: with a.sbuf, a path's radiance goes to its own slot
// (sample - sample_offset) * rect pixels + rect pixel, one plain store when
// the path ends; k_wf_flush_samples then sums each pixel's samples in sample
// order in FP64 and adds the fixed-point film, which still takes the final
// vertices' light samples.  Without a.sbuf the fixed-point film takes
// everything.  Both sums are independent of completion order.
__device__ __forceinline__ size_t sample_slot(const WfArgs& a, uint32_t pix, uint32_t smp) {
  const uint32_t px = pix % uint32_t(a.W), py = pix / uint32_t(a.W);
  const size_t rw = size_t(a.x1 - a.x0), rh = size_t(a.y1 - a.y0);
  return (size_t(smp - a.sample_offset) * rh + size_t(py - uint32_t(a.y0))) * rw + size_t(px - uint32_t(a.x0));
}
__device__ __forceinline__ void sample_store(const WfArgs& a, uint32_t pix, uint32_t smp, float r, float g,
                                             float b) {
  float* q = a.sbuf + 3 * sample_slot(a, pix, smp);
  q[0] = r; q[1] = g; q[2] = b;
}

// NEE light sample at x (trace_path's light-selection block).  Returns false
// when no shadow ray is needed.  POINT: the scene has no surfaces, so its
// emitters are point lights.
template <bool MEDIUM, bool POINT = false>
__device__ __forceinline__ bool nee_sample(const DevScene& s, Vec3<float> x, Vec3<float> d, const Glossy<float>& gm,
                                           Vec3<float> wo, Vec3<float> ns, Vec3<float> ss, Vec3<float> ts, float ul,
                                           float ua, float ub, Vec3<float>& wi, float& tmax, Vec3<float>& f,
                                           Vec3<float>& Le, float& wt, float& pl, bool& delta_out) {
  if (s.n_lights <= 0) return false;
  const float nl = float(s.n_lights);
  int li = int(ul * nl);
  li = li < s.n_lights - 1 ? li : s.n_lights - 1;
  Le = v3s(0.0f);
  pl = 0.0f;
  float dist = xinf<float>();
  bool delta = false;
  const int env_slot = s.has_sun ? 1 : 0;
  if (s.has_sun && li == 0) {
    wi = -v3f<float>(s.sun_dir);
    Le = v3f<float>(s.sun_E);
    pl = 1.0f;
    delta = true;
  } else if (s.env_type != 0 && li == env_slot) {
    env_sample<float>(s, ua, ub, wi, pl, Le);
  } else {
    const uint32_t code = s.emitters[li - env_slot - (s.env_type != 0 ? 1 : 0)];
    if constexpr (POINT) {
      sample_point<float>(s, code & 0x3FFFFFFFu, x, wi, dist, pl, Le);
      delta = true;
    } else {
      delta = sample_emitter<float>(s, code, x, ua, ub, wi, dist, pl, Le);
    }
  }
  if (!(pl > 0.0f)) return false;
  float pf;
  if (MEDIUM) {
    const float p = hg_p(s.g, dot(d, wi));
    f = v3s(p);
    pf = p;
  } else {
    const Vec3<float> wol = to_lcs(wo, ns, ss, ts), wil = to_lcs(wi, ns, ss, ts);
    gm.eval_pdf(wol, wil, f, pf);
    f = f * fabsf(wil.z);
  }
  if (is_black(f)) return false;
  tmax = xisinf(dist) ? xinf<float>() : dist * float(1 - 1e-4);
  wt = delta ? 1.0f : power_heuristic(pl, pf);
  delta_out = delta;
  return true;
}

}  // namespace ne
