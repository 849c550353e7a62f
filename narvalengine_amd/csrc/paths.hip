// paths.hip -- persistent volume path kernel for gfx950 (FP32): whole renders
// of volumes lit by the sun, the environment and point lights in one launch.
//
// Without surfaces every stage of the wavefront pipeline (new paths, delta
// tracking, shading with its shadow ray, compaction) only ever touches its
// own chunk of paths, so a resident block can run them in turn on paths it
// holds: no launches per bounce, no plan, and blocks drain without waiting
// for each other.
//
// What binds is VALU issue at the lanes that are live: rays take one to three
// tentative collisions on average but the longest of 64 takes many, so a wave
// that tracks its rays to the end runs most steps with a few lanes (27% in the
// staged stages).  Here a wave tracks a packed group of up to 64 rays only
// until a few of them are left, and puts those back into the block's lists;
// the next iteration packs them with other rays.  A path's shadow ray and its
// continuation are two entries of the lists, so they also run side by side.
//
// Measured against the staged pipeline on one MI355X (both with quads / both with
// bricks): 1920x1080 x 256 spp cloud (512^3, 128 bounces) 177.6 -> 105.0 / 173.3
// -> 112.2 ms, 512x512 x 64 spp fBm volume 8.16 -> 6.63 / 9.32 -> 6.84 ms,
// 960x540 x 16 spp guided cloud 5.75 -> 2.60 / 5.85 -> 2.68 ms; VALU
// instructions of the cloud frame (bricks) 1.0e11 -> 5.6e10, lanes live 28% ->
// 46%.
//
// A 256-thread block owns 256 path slots.  Nothing scans them: every state
// change appends the slot to the list of what comes next.  One iteration:
//   shade    the listed vertices (both rays of the slot are over), packed:
//            light sample, scattering, a shadow ray and a continuation; the
//            paths that ended with a shadow ray out store their radiance
//   track    waves take groups of 64 rays: continuations, then new paths'
//            camera rays (ids from a global counter), then shadow rays
// Draws and arithmetic are those of the staged pipeline, so both give the
// same film.
#include <algorithm>

#include "ne_launch.h"
#include "ne_trace.h"
#include "ne_wavefront.h"

namespace ne {

constexpr int kPathBlock = 256;
// A wave hands its rays back once at most kSuspend of them, or a quarter of
// its group, are left.  Putting a walk away and taking it up again costs about
// one tracking step's instructions per ray.  1920x1080 x 256 spp cloud / 640x360
// x 32 spp cloud / 512x512 x 64 spp fBm / 1280x720 x 64 spp fBm / guided cloud
// frames, ms: 4: 114.0 / 2.68 / 6.66 / 15.9 / 3.17, 6: 111.5 / 2.60 / 6.71 / 16.0
// / 3.12, 8: 109.2 / 2.58 / 6.80 / 16.2 / 3.12, 10: 107.6 / 2.54 / 6.90 / 16.4 /
// 3.10, 12: 106.9 / 2.50 / 6.95 / 16.3 / 3.08, 16: 107.1 / 2.54 / 7.10 / 16.6 /
// 3.08, 20: 107.0 / 2.49 / 7.07 / 16.7 / 3.14.  The fBm volumes, whose walks end
// sooner, gain up to 4% from 4, the cloud loses 7%: 12.
constexpr int kSuspend = 12;

// A slot's depth word: vertices so far, and in the upper half what is over.
// The wave that finds both rays over lists the slot by the end's kind.
constexpr uint32_t kExtOver = 1u << 16, kShdOver = 1u << 17;
constexpr uint32_t kEndMiss = 1u << 18, kEndLimit = 2u << 18, kEndVertex = 3u << 18, kEndMask = 3u << 18;  // 0: collided

// What tracking reads and writes: the block's slots in LDS, structure of arrays.
struct PathSlots {
  float ox[kPathBlock], oy[kPathBlock], oz[kPathBlock], dx[kPathBlock], dy[kPathBlock], dz[kPathBlock];
  float t[kPathBlock], tb[kPathBlock];  // collision distance; suspended: the walk's position and end
  uint32_t cell[kPathBlock];
  uint32_t pix[kPathBlock], smp[kPathBlock], depth[kPathBlock];
  uint32_t rngn[kPathBlock], b0[kPathBlock], b1[kPathBlock], b2[kPathBlock];  // draws consumed, undrawn words
  float wx[kPathBlock], wy[kPathBlock], wz[kPathBlock];  // shadow ray (origin: the path's)
  float tr[kPathBlock], st[kPathBlock], stb[kPathBlock];  // transmittance; position; extent, then the walk's end
  uint32_t scell[kPathBlock], srngn[kPathBlock];
};
constexpr uint32_t kFreshRay = 0xFFFFFFFFu;  // cell word of a ray whose walk has not started

// What only vertices and ends touch: in global memory, one record of
// kColdWords arrays per block (slot index innermost).
enum { kBx = 0, kBy, kBz, kLx, kLy, kLz, kPdf, kFx, kFy, kFz, kWt, kPl, kColdWords };

// New paths of an iteration: n0 ids from base0, then n1 from base1, for the
// `want` free slots that were there.
struct PathIds {
  unsigned long long base0, base1;
  uint32_t n0, n1, want;
};

// Thread 0's cursor into the global work counter: [cur, end) of the batch in
// hand.  take() fills `ids` with up to `want` ids (want <= grab, so two
// segments always suffice).
struct PathCursor {
  unsigned long long cur, end;
  bool dry;
  __device__ __forceinline__ void take(PathIds& ids, uint32_t want, unsigned long long* next, uint32_t grab,
                                       unsigned long long total) {
    const unsigned long long left = end - cur;
    ids.want = want;
    ids.base0 = cur;
    ids.n0 = left < want ? uint32_t(left) : want;
    cur += ids.n0;
    ids.n1 = 0;
    if (ids.n0 < want && !dry) {
      cur = atomicAdd(next, (unsigned long long)grab);
      end = cur + grab < total ? cur + grab : total;
      if (cur >= total) {
        dry = true;
        cur = end = 0;
      } else {
        const uint32_t rest = want - ids.n0;
        ids.base1 = cur;
        ids.n1 = end - cur < rest ? uint32_t(end - cur) : rest;
        cur += ids.n1;
      }
    }
  }
};

// The kernel's arguments, one struct at the start of the kernarg segment.
struct PathArgs {
  WfArgs a;
  DevScene s;
  DevCamera cam;
  GuideUse gu;
  unsigned long long* next;
  float* cold;
  uint32_t grab;
};
typedef const __attribute__((address_space(4))) PathArgs* PathArgsPtr;

// The arguments' address, opaque to the optimiser: what a phase reads through
// it is loaded again by scalar loads there.  Without it the loop's invariants
// (some 250 words of arguments and the floats derived from them) are hoisted
// out of the block's loop and held or spilled across it.
__device__ __forceinline__ const PathArgs& phase_args() {
  PathArgsPtr p = (PathArgsPtr)__builtin_amdgcn_kernarg_segment_ptr();
  asm volatile("" : "+s"(p));
  return *(const PathArgs*)p;
}

// Lists of slots, double-buffered: one phase reads what the one before wrote.
// Vertices and ends share an array, ends from its top (a slot is in one of them).
enum { kListVertex = 0, kListFree, kListExt, kListShadow, kListEnd, kLists };
struct PathLists {
  uint8_t slot[2][kListEnd][kPathBlock];
  uint32_t n[2][kLists];
};
// Appends q where pred holds (in any order: paths are independent).
__device__ __forceinline__ void list_add(PathLists& l, uint32_t buf, int which, bool pred, uint32_t q) {
  const unsigned long long m = __ballot(pred);
  if (m == 0) return;
  const int first = __ffsll((long long)m) - 1, lane = __lane_id();
  uint32_t base = 0;
  if (lane == first) base = atomicAdd(&l.n[buf][which], uint32_t(__popcll(m)));
  base = __builtin_amdgcn_readlane(base, first);
  const uint32_t at = base + uint32_t(__popcll(m & ((1ull << lane) - 1ull)));
  if (pred) {
    if (which == kListEnd) l.slot[buf][kListVertex][uint32_t(kPathBlock) - 1u - at] = uint8_t(q);
    else l.slot[buf][which][at] = uint8_t(q);
  }
}

// Six waves per SIMD: 80 VGPRs without spills, and six blocks' 26.7 KB of LDS
// in a CU's 160 KB (seven waves, with half of the walks' state in memory:
// cloud 123 ms; five waves: 122 ms against 121 ms on an earlier form).
template <bool GUIDED, int GRID>
__global__ __launch_bounds__(kPathBlock, 6) void k_paths(PathArgs args) {
  __shared__ PathSlots P;
  __shared__ PathLists S;
  __shared__ uint32_t group;  // next group to track
  __shared__ PathIds ids;
  const uint32_t t = threadIdx.x;
  const uint32_t lane = uint32_t(__lane_id());
  PathCursor cursor;
  S.slot[0][kListFree][t] = uint8_t(t);
  if (t < 2 * kLists) S.n[t / kLists][t % kLists] = t == kListFree ? uint32_t(kPathBlock) : 0u;
  if (t == 0) {
    const PathArgs& g = phase_args();
    cursor.cur = (unsigned long long)blockIdx.x * g.grab;  // the first batch of each block is its own
    cursor.end = cursor.cur + g.grab < g.a.total_paths ? cursor.cur + g.grab : g.a.total_paths;
    if (cursor.cur > cursor.end) cursor.cur = cursor.end;
    cursor.dry = false;
  }
  Count<false> cnt;
  for (uint32_t p = 0;; p ^= 1u) {
    __syncthreads();
    // ---- shade
    const uint32_t nv = S.n[p][kListVertex], nend = S.n[p][kListEnd], nfree = S.n[p][kListFree];
    if (t == 0) {
      const PathArgs& g = phase_args();
      // (the free list being filled was emptied when it was last read)
      S.n[p ^ 1u][kListVertex] = S.n[p ^ 1u][kListEnd] = S.n[p ^ 1u][kListExt] = S.n[p ^ 1u][kListShadow] = 0;
      group = 0;
      cursor.take(ids, nfree + nend, g.next, g.grab, g.a.total_paths);
    }
    if (t < nv) {
      const PathArgs& g = phase_args();
      const WfArgs& a = g.a;
      const DevScene& s = g.s;
      const GuideUse& gu = g.gu;
      const uint32_t q = S.slot[p][kListVertex][t];
      float* cold = g.cold + size_t(blockIdx.x) * (kColdWords * kPathBlock) + q;
      const Vec3<float> d = v3(P.dx[q], P.dy[q], P.dz[q]);
      const Vec3<float> x = v3(P.ox[q], P.oy[q], P.oz[q]) + P.t[q] * d;
      const uint32_t pix = P.pix[q], smp = P.smp[q], depth = P.depth[q] & 0xFFFFu;
      Vec3<float> beta = v3s(1.0f);
      if (depth != 0) beta = v3(cold[kBx * kPathBlock], cold[kBy * kPathBlock], cold[kBz * kPathBlock]);
      beta = beta * v3(s.albedo[0], s.albedo[1], s.albedo[2]);
      PathRng rng;
      rng.init(a.seed, pix, smp, a.job);
      float u[5];
      rng.five(P.rngn[q], u);
      Vec3<float> wi, f, Le;
      float tmax = 0.0f, wt = 0.0f, pl = 0.0f;
      bool delta = false;
      const Glossy<float> none{};
      const bool shadow = nee_sample<true, true>(s, x, d, none, v3s(0.0f), v3s(0.0f), v3s(0.0f), v3s(0.0f), u[0], u[1],
                                                 u[2], wi, tmax, f, Le, wt, pl, delta);
      const float* mix = nullptr;
      if constexpr (GUIDED) {
        if (int(depth) < gu.max_depth) {
          mix = guide_cache_at(gu.cache, xf_point<float>(s.inv, x) + v3s(0.5f), d);
          if (shadow && !delta)  // the phase-sampling strategy is the mixture
            wt = power_heuristic(pl, (1.0f - gu.prob) * hg_p(s.g, dot(d, wi)) + gu.prob * vmf_mixture_pdf(mix, wi));
        }
      }
      if (shadow) {  // its weight: the throughput before this vertex's scattering weight
        f = beta * f * Le;
        P.wx[q] = wi.x; P.wy[q] = wi.y; P.wz[q] = wi.z;
        P.stb[q] = tmax;
        P.scell[q] = kFreshRay;
        cold[kFx * kPathBlock] = f.x; cold[kFy * kPathBlock] = f.y; cold[kFz * kPathBlock] = f.z;
        cold[kWt * kPathBlock] = wt; cold[kPl * kPathBlock] = pl;
      }
      bool cont = true;
      Vec3<float> nd;
      float ppdf;
      if (GUIDED && mix) {
        const float us = u[3], u0 = u[4], u1 = rng.next(), u2 = rng.next();
        nd = us < gu.prob ? vmf_mixture_sample(mix, u2, u0, u1) : hg_sample(s.g, d, u0, u1);
        const float ph = hg_p(s.g, dot(d, nd));
        ppdf = (1.0f - gu.prob) * ph + gu.prob * vmf_mixture_pdf(mix, nd);
        cont = ppdf > 0.0f;
        if (cont) beta = beta * (ph / ppdf);
      } else {
        nd = hg_sample(s.g, d, u[3], u[4]);
        ppdf = hg_p(s.g, dot(d, nd));
      }
      P.ox[q] = x.x; P.oy[q] = x.y; P.oz[q] = x.z;
      P.dx[q] = nd.x; P.dy[q] = nd.y; P.dz[q] = nd.z;
      P.cell[q] = kFreshRay;
      P.rngn[q] = rng.consumed();
      P.b0[q] = rng.b0; P.b1[q] = rng.b1; P.b2[q] = rng.b2;
      P.depth[q] = (depth + 1u) | (shadow ? 0u : kShdOver) | (cont ? 0u : (kExtOver | kEndVertex));
      cold[kBx * kPathBlock] = beta.x; cold[kBy * kPathBlock] = beta.y; cold[kBz * kPathBlock] = beta.z;
      cold[kPdf * kPathBlock] = ppdf;
      if (depth == 0) cold[kLx * kPathBlock] = cold[kLy * kPathBlock] = cold[kLz * kPathBlock] = 0.0f;
      if (GUIDED && !cont) {  // ended here: its shadow ray still delivers to the film
        const float lx = depth ? cold[kLx * kPathBlock] : 0.0f, ly = depth ? cold[kLy * kPathBlock] : 0.0f,
                    lz = depth ? cold[kLz * kPathBlock] : 0.0f;
        if (a.sbuf) sample_store(a, pix, smp, lx, ly, lz);
        else film_add(a.film_fixed, pix, lx, ly, lz);
      }
      list_add(S, p, kListExt, cont, q);
      list_add(S, p, kListShadow, shadow, q);
      if constexpr (GUIDED) list_add(S, p ^ 1u, kListFree, !cont && !shadow, q);
    } else if (t >= uint32_t(kPathBlock) - nend) {
      // paths that ended before their last shadow ray did
      const PathArgs& g = phase_args();
      const WfArgs& a = g.a;
      const DevScene& s = g.s;
      const uint32_t q = S.slot[p][kListVertex][t];
      const float* cold = g.cold + size_t(blockIdx.x) * (kColdWords * kPathBlock) + q;
      Vec3<float> L = v3(cold[kLx * kPathBlock], cold[kLy * kPathBlock], cold[kLz * kPathBlock]);
      if ((P.depth[q] & kEndMask) == kEndMiss && s.env_type != 0) {
        const Vec3<float> d = v3(P.dx[q], P.dy[q], P.dz[q]);
        const Vec3<float> E = env_le<float>(s, d);
        const float wm = power_heuristic(cold[kPdf * kPathBlock], env_pdf<float>(s, d));
        L.x += cold[kBx * kPathBlock] * E.x * wm;
        L.y += cold[kBy * kPathBlock] * E.y * wm;
        L.z += cold[kBz * kPathBlock] * E.z * wm;
      }
      if (a.sbuf) sample_store(a, P.pix[q], P.smp[q], L.x, L.y, L.z);
      else film_add(a.film_fixed, P.pix[q], L.x, L.y, L.z);
    }
    __syncthreads();
    // ---- track
    const uint32_t nr = S.n[p][kListExt], nshd = S.n[p][kListShadow], nnew = ids.n0 + ids.n1;
    const uint32_t next = nr + nnew;
    if (next + nshd == 0 && ids.want > 0) break;  // free slots, no ids left, nothing in flight
    if (t == 0) S.n[p][kListFree] = 0;            // read by all before the barrier above
    const uint32_t ge = (next + 63) / 64, gs = (nshd + 63) / 64;
    // once no more groups than waves are left and no ids come, to the end
    const bool tail = nnew == 0 && ge + gs <= uint32_t(kPathBlock / 64);
    auto rest = [&](uint32_t n) { return tail ? 0 : min(int(min(64u, n)) / 4, kSuspend); };
    while (true) {
      uint32_t gi = 0;
      if (lane == 0) gi = atomicAdd(&group, 1u);
      gi = __builtin_amdgcn_readfirstlane(gi);
      if (gi >= ge + gs) break;
      const PathArgs& g = phase_args();
      const WfArgs& a = g.a;
      const DevScene& s = g.s;
      Walk w;
      if (gi < ge) {
        // continuations and camera rays
        const int keep = rest(next - gi * 64);
        const bool mine = gi * 64 + lane < next;
        const uint32_t k = mine ? gi * 64 + lane : next - 1u;  // the other lanes read a valid ray and drop it
        const bool fresh = k >= nr;
        uint32_t q, pix, smp, cell = kFreshRay, rngn = 2, w0, w1, w2 = 0;
        Vec3<float> o, d;
        if (fresh) {
          const uint32_t r = k - nr;
          q = r < nfree ? S.slot[p][kListFree][r] : S.slot[p][kListVertex][uint32_t(kPathBlock) - 1u - (r - nfree)];
          uint32_t px, py;
          path_pixel(a, r < ids.n0 ? ids.base0 + r : ids.base1 + (r - ids.n0), pix, smp, px, py);
          smp += a.sample_offset;
          PathRng cam;
          cam.init(a.seed, pix, smp, a.job);
          const float ju = cam.next(), jv = cam.next();
          w0 = cam.b0;
          w1 = cam.b1;
          const float u = (float(uint32_t(a.x0) + px) + ju) / float(a.W);
          const float v = (float(uint32_t(a.y0) + py) + jv) / float(a.H);
          const Vec3<float> pos = v3f<float>(g.cam.pos), ll = v3f<float>(g.cam.lower_left);
          const Vec3<float> hz = v3f<float>(g.cam.horizontal), vt = v3f<float>(g.cam.vertical);
          o = pos;
          d = -normalize(ll + u * hz + v * vt - pos);
          if (mine) {
            P.ox[q] = o.x; P.oy[q] = o.y; P.oz[q] = o.z;
            P.dx[q] = d.x; P.dy[q] = d.y; P.dz[q] = d.z;
            P.pix[q] = pix; P.smp[q] = smp;
            P.depth[q] = kShdOver;
          }
        } else {
          q = S.slot[p][kListExt][k];
          o = v3(P.ox[q], P.oy[q], P.oz[q]);
          d = v3(P.dx[q], P.dy[q], P.dz[q]);
          pix = P.pix[q];
          smp = P.smp[q];
          cell = P.cell[q];
          rngn = P.rngn[q];
          w0 = P.b0[q];
          w1 = P.b1[q];
          w2 = P.b2[q];
        }
        // (the stream is set up here, not in the branches: its key then stays
        // the same for every lane and its schedule in scalar registers)
        PathRng rng;
        rng.init(a.seed, pix, smp, a.job);
        rng.restore(rngn, w0, w1, w2);
        w.ray(s, o, d);
        bool done, in;
        if (cell == kFreshRay) {
          float ta, te;
          done = !w.box(ta, te);
          done = !w.start(s, xmax(ta, 0.0f), te) || done;
          in = true;
        } else {
          w.resume(s, P.t[q], P.tb[q], cell & 0xFFFFFFu);
          done = false;
          in = (cell >> 24) != 0u;
        }
        done = done || !mine;
        in = in && !done && w.look(s);
        bool hit = false;
        asm volatile("" ::: "memory");  // what the ray's slot holds is read again after the loop
        if (int(__popcll(__ballot(!done))) > keep) do {
          if (!done && !in) {
            done = w.leave(s);
            if (!done) in = w.look(s);
          }
          if (in) {
            w.t -= log1m_draw(rng.next_keep1()) * w.imu;
            in = w.t < w.c1;
            if (in) {
              const float sig = sigma_at<float, false, GRID>(s, w.oo, w.dd, w.t, cnt);
              const float ra = rng.next_buffered();
              if (sig * w.imu > ra) {
                hit = true;
                done = true;
                in = false;
              }
            }
          }
        } while (int(__popcll(__ballot(!done))) > keep);
        if (mine) {
          const uint32_t depth = P.depth[q] & 0xFFFFu;
          const bool gone = depth == 0 && done && (!hit || a.max_bounces <= 0);
          bool both = false;  // this ray and the slot's shadow ray are over
          uint32_t kind = 0;
          if (gone) {
            // a camera ray that ends: beta 1, nothing gathered, no MIS
            Vec3<float> E = v3s(0.0f);
            if (!hit && s.env_type != 0) E = env_le<float>(s, v3(P.dx[q], P.dy[q], P.dz[q]));
            if (a.sbuf) sample_store(a, rng.pixel, rng.sample, E.x, E.y, E.z);
            else film_add(a.film_fixed, rng.pixel, E.x, E.y, E.z);
          } else {
            P.t[q] = w.t;
            P.rngn[q] = rng.consumed();
            if (!done) {
              P.tb[q] = w.tb;
              P.cell[q] = w.packed() | (in ? 1u << 24 : 0u);
              P.b0[q] = rng.b0; P.b1[q] = rng.b1; P.b2[q] = rng.b2;
            } else {
              kind = !hit ? kEndMiss : (int(depth) < a.max_bounces ? 0u : kEndLimit);
              both = (atomicOr(&P.depth[q], kExtOver | kind) & kShdOver) != 0u;
            }
          }
          list_add(S, p ^ 1u, kListExt, !done, q);
          list_add(S, p ^ 1u, kListFree, gone, q);
          list_add(S, p ^ 1u, kListVertex, both && kind == 0u, q);
          list_add(S, p ^ 1u, kListEnd, both && kind != 0u, q);
        }
      } else {
        // shadow rays
        const uint32_t i = (gi - ge) * 64 + lane;
        const int keep = rest(nshd - (gi - ge) * 64);
        const bool mine = i < nshd;
        const uint32_t q = S.slot[p][kListShadow][mine ? i : nshd - 1u];
        float tr = 1.0f;
        PathRng rng;
        rng.init(a.seed, P.pix[q], P.smp[q], a.job);
        const uint32_t block0 = kShadowBlockBase + (((P.depth[q] & 0xFFFFu) - 1u) << 20);
        rng.restore(0u, 0u, 0u, 0u, block0);
        w.ray(s, v3(P.ox[q], P.oy[q], P.oz[q]), v3(P.wx[q], P.wy[q], P.wz[q]));
        const uint32_t cell = P.scell[q];
        bool done, in;
        if (cell == kFreshRay) {
          float ta, te;
          done = !w.box(ta, te);
          ta = xmax(ta, 0.0f);
          te = xmin(te, P.stb[q]);
          if (s.homog) {
            if (!done && ta < te) tr = xexp(-s.sigma_bar * (te - ta));
            done = true;
          }
          done = !w.start(s, ta, te) || done;
          in = true;
        } else {
          w.resume(s, P.st[q], P.stb[q], cell & 0xFFFFFFu);
          tr = P.tr[q];
          rng.seek(P.srngn[q], block0);
          done = false;
          in = (cell >> 24) != 0u;
        }
        done = done || !mine;
        in = in && !done && w.look(s);
        if (int(__popcll(__ballot(!done))) > keep) do {
          if (!done && !in) {
            done = w.leave(s);
            if (!done) in = w.look(s);
          }
          if (in) {
            w.t -= log1m_draw(rng.next_keep1()) * w.imu;
            in = w.t < w.c1;
            if (in) {
              const float sig = sigma_at<float, false, GRID>(s, w.oo, w.dd, w.t, cnt);
              tr *= 1.0f - xmax(0.0f, sig * w.imu);
              if (tr < 0.1f) {  // Russian roulette
                const float qq = xmax(0.05f, 1.0f - tr);
                if (rng.next_buffered() < qq) {
                  tr = 0.0f;
                  done = true;
                  in = false;
                } else {
                  tr /= 1.0f - qq;
                }
              }
            }
          }
        } while (int(__popcll(__ballot(!done))) > keep);
        if (mine) {
          uint32_t over = 0;
          if (!done) {
            P.tr[q] = tr;
            P.st[q] = w.t;
            P.stb[q] = w.tb;
            P.scell[q] = w.packed() | (in ? 1u << 24 : 0u);
            P.srngn[q] = rng.consumed() - (block0 << 2);
          } else {
            const bool ended = GUIDED && (P.depth[q] & kEndMask) == kEndVertex;
            if (tr > 0.0f) {
              float* cold = g.cold + size_t(blockIdx.x) * (kColdWords * kPathBlock) + q;
              const float qq = tr * cold[kWt * kPathBlock] * float(s.n_lights) / cold[kPl * kPathBlock];
              const float cx = cold[kFx * kPathBlock] * qq, cy = cold[kFy * kPathBlock] * qq,
                          cz = cold[kFz * kPathBlock] * qq;
              if (ended) {
                film_add(a.film_fixed, P.pix[q], cx, cy, cz);
              } else {
                cold[kLx * kPathBlock] += cx;
                cold[kLy * kPathBlock] += cy;
                cold[kLz * kPathBlock] += cz;
              }
            }
            over = atomicOr(&P.depth[q], kShdOver);
          }
          const bool both = (over & kExtOver) != 0u;
          const uint32_t kind = over & kEndMask;
          list_add(S, p ^ 1u, kListShadow, !done, q);
          list_add(S, p ^ 1u, kListVertex, both && kind == 0u, q);
          list_add(S, p ^ 1u, kListEnd, both && (kind == kEndMiss || kind == kEndLimit), q);
          if constexpr (GUIDED) list_add(S, p ^ 1u, kListFree, both && kind == kEndVertex, q);
        }
      }
    }
  }
}

__global__ void k_paths_init(unsigned long long* next, unsigned long long first) { *next = first; }

// 8 blocks per CU at most (2048 threads), the counter in front.
size_t paths_scratch_bytes(int cus) {
  return 256 + size_t(cus) * (2048 / kPathBlock) * (sizeof(float) * kColdWords * kPathBlock);
}

hipError_t launch_paths(const DevScene& s, const DevCamera& cam, const WfArgs& a, const GuideUse& gu, void* scratch,
                        int cus, hipStream_t st, StageTimer* tm) {
  hipError_t e = hipSuccess;
  const bool guided = gu.cache.mix != nullptr;
  const int form = std::min(s.grid_form, a.grid_max);
  void (*fn)(PathArgs) =
      form == kGridQuad    ? (guided ? &k_paths<true, kGridQuad> : &k_paths<false, kGridQuad>)
      : form == kGridBrick ? (guided ? &k_paths<true, kGridBrick> : &k_paths<false, kGridBrick>)
                           : (guided ? &k_paths<true, kGridWide> : &k_paths<false, kGridWide>);
  int per_cu = 0;
  if ((e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, reinterpret_cast<const void*>(fn), kPathBlock, 0)) !=
      hipSuccess)
    return e;
  const uint64_t resident = uint64_t(cus) * uint64_t(std::min(2048 / kPathBlock, std::max(1, per_cu)));
  const uint32_t blocks = uint32_t(std::min<uint64_t>(resident, (a.total_paths + kPathBlock - 1) / kPathBlock));
  // ids per counter grab: small enough that the blocks' last batches even out
  // (1/8 of a block's share instead of 1/64: fBm frame 6.8 against 6.55 ms),
  // large enough that the counter's same-address atomics (about 11 ns each
  // across the XCDs) do not bind
  const uint64_t grab = std::min<uint64_t>(4096, std::max<uint64_t>(kPathBlock, a.total_paths / (64ull * blocks)));
  unsigned long long* next = static_cast<unsigned long long*>(scratch);
  float* cold = reinterpret_cast<float*>(static_cast<char*>(scratch) + 256);
  if (tm && (e = tm->mark(kStageOther)) != hipSuccess) return e;
  hipLaunchKernelGGL(k_paths_init, dim3(1), dim3(1), 0, st, next, (unsigned long long)(blocks * grab));
  if (tm && (e = tm->mark(kStageMegakernel)) != hipSuccess) return e;
  hipLaunchKernelGGL(fn, dim3(blocks), dim3(kPathBlock), 0, st, PathArgs{a, s, cam, gu, next, cold, uint32_t(grab)});
  if ((e = hipGetLastError()) != hipSuccess) return e;
  if (tm && (e = tm->mark(kStageOther)) != hipSuccess) return e;
  if ((e = wf_flush(a, st)) != hipSuccess) return e;
  if (tm && (e = tm->mark(kStageEnd)) != hipSuccess) return e;
  return hipSuccess;
}

}  // namespace ne
