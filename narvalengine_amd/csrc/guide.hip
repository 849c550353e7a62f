// guide.hip -- learned directional proposal for medium scattering vertices.
//
// Position (unit cube of the volume) -> multiresolution hash-grid encoding
// (16 levels x 2 features, trilinear) ++ incoming direction -> MLP
// 35 -> 64 -> 64 -> 64 -> 64 -> 40 (ReLU) -> mixture of 8 von Mises-Fisher
// lobes (softmax weights, normalised means, kappa = exp).  The MLP runs on
// 16x16x16 BF16 MFMA tiles (BF16 weights and layer inputs, FP32 accumulation
// and biases): a wave evaluates 16 queries per tile, passing activations
// between layers through LDS.
//
// MFMA operand layout (v_mfma_f32_16x16x16_bf16, wave64), lane l:
//   A (16 x 16, rows x k):  row l % 16, k = 4 (l / 16) .. +3
//   B (16 x 16, k x cols):  col l % 16, k = 4 (l / 16) .. +3
//   D (16 x 16):            col l % 16, rows 4 (l / 16) .. +3
//
// Training minimises the Monte-Carlo estimate of KL(target || q) with target
// proportional to Li * phase: loss = -sum_i r_i log q(w_i) / sum_i r_i over a
// batch of (position, direction, sampled direction w_i, weight r_i).  Backward
// runs layer by layer over the whole batch; weight gradients are reduced from
// per-wave partial sums in a fixed order (deterministic), hash-feature
// gradients are summed in LDS, range by range.  Adam updates FP32 masters; BF16
// operand copies (MLP weights and hash features) are re-packed after each step.
#include <algorithm>

#include "ne_guide.h"

namespace ne {

// n queries (position, direction) -> mixture (or raw outputs), 64 per wave tile.
__global__ __launch_bounds__(kGuideBlock) void k_guide_eval(GuideNet g, int n, const float* in6, float* out40,
                                                            int raw) {
  __shared__ __align__(16) unsigned char buf[kWavesPerBlock][kWave64Bytes];
  const int wv = threadIdx.x >> 6, lane = __lane_id();
  const int tiles = (n + 63) / 64;
  for (int t = blockIdx.x * kWavesPerBlock + wv; t < tiles; t += gridDim.x * kWavesPerBlock) {
    wave_sync();
    guide_encode_tile64(g, reinterpret_cast<uint16_t*>(buf[wv]), [&](int i, Vec3<float>& p, Vec3<float>& d, bool& valid) {
      const int q = t * 64 + i;
      valid = q < n;
      const float* s = in6 + 6 * size_t(valid ? q : 0);
      p = v3(s[0], s[1], s[2]);
      d = v3(s[3], s[4], s[5]);
    });
    const float* out = guide_mlp_tile64(g, buf[wv]);
    const int q = t * 64 + lane;
    if (q < n) {
      float* o = out40 + 40 * size_t(q);
      if (raw) {
        for (int c = 0; c < kGuideOutputs; ++c) o[c] = out[lane * kLdOut64 + c];
      } else {
        guide_head(&out[lane * kLdOut64], o);
      }
    }
  }
}

// Tabulated proposal: the mixture at every (cell centre, direction-bin centre)
// of the cache, written to cache.mix (40 floats per entry).
__global__ __launch_bounds__(kGuideBlock) void k_guide_bake(GuideNet g, GuideCache c, float* mix, int n) {
  __shared__ __align__(16) unsigned char buf[kWavesPerBlock][kWave64Bytes];
  const int wv = threadIdx.x >> 6, lane = __lane_id();
  const int nb = c.nd * c.nd;
  const int tiles = (n + 63) / 64;
  for (int t = blockIdx.x * kWavesPerBlock + wv; t < tiles; t += gridDim.x * kWavesPerBlock) {
    wave_sync();
    guide_encode_tile64(g, reinterpret_cast<uint16_t*>(buf[wv]), [&](int i, Vec3<float>& p, Vec3<float>& d, bool& valid) {
      const int q = t * 64 + i;
      valid = q < n;
      const int e = valid ? q : 0;
      const int cell = e / nb, bin = e % nb;
      const int cx = cell % c.nc, cy = (cell / c.nc) % c.nc, cz = cell / (c.nc * c.nc);
      const float inv = 1.0f / float(c.nc);
      p = v3((float(cx) + 0.5f) * inv, (float(cy) + 0.5f) * inv, (float(cz) + 0.5f) * inv);
      const float invd = 1.0f / float(c.nd);
      oct_decode((float(bin % c.nd) + 0.5f) * invd, (float(bin / c.nd) + 0.5f) * invd, d.x, d.y, d.z);
    });
    const float* out = guide_mlp_tile64(g, buf[wv]);
    const int q = t * 64 + lane;
    if (q < n) guide_head(&out[lane * kLdOut64], mix + 40 * size_t(q));
  }
}

// ---- training: forward + loss gradient --------------------------------------------
// Per tile: layer inputs stored for backward (act[l][row][64] BF16), loss
// gradient w.r.t. the 40 raw outputs into dy (BF16, columns 40..47 zero).
// A tile is a chain of gathers, layers and the 16 rows' losses: latency, not
// bandwidth, so every wave takes one tile (65,536 samples in 4096 waves: 75
// us against 218 us with 8 tiles each in 512 waves and a row's 8 lobes on one lane).
__global__ __launch_bounds__(kGuideBlock) void k_guide_train_fwd(GuideNet g, GuideBatch b, GuideTrain t) {
  __shared__ uint16_t xa[kWavesPerBlock][16 * kLdA];
  __shared__ uint16_t xb[kWavesPerBlock][16 * kLdA];
  __shared__ float out[kWavesPerBlock][16 * kLdO];
  const int wv = threadIdx.x >> 6, lane = __lane_id();
  const uint32_t n = min(*b.count, b.cap);
  const uint32_t tiles = (n + 15) / 16;
  const float* S = b.s;
  const uint32_t cap = b.cap;
  float loss = 0.0f, wsum = 0.0f;
  for (uint32_t tt = blockIdx.x * kWavesPerBlock + wv; tt < tiles; tt += gridDim.x * kWavesPerBlock) {
    wave_sync();
    guide_encode_tile(g, xa[wv], [&](int i, Vec3<float>& p, Vec3<float>& d, bool& valid) {
      const uint32_t q = tt * 16 + uint32_t(i);
      valid = q < n;
      const uint32_t k = valid ? q : 0u;
      p = v3(S[k], S[cap + k], S[2 * cap + k]);
      d = v3(S[3 * cap + k], S[4 * cap + k], S[5 * cap + k]);
    });
    // keep every layer input for backward: act[l][row][c]
    uint16_t* bufs[2] = {xa[wv], xb[wv]};
#define NE_STORE_ACT(L, SRC)                                                                 \
    for (int e = lane; e < 16 * 64; e += 64) {                                               \
      const int row = e >> 6, c = e & 63;                                                    \
      const uint32_t q = tt * 16 + uint32_t(row);                                            \
      if (q < n) t.act[(size_t(L) * cap + q) * kGuideWidth + c] = c < guide_in(L) ? (SRC)[row * kLdA + c] : 0; \
    }
    wave_sync();
    NE_STORE_ACT(0, bufs[0]);
    guide_layer<0>(g, xa[wv], xb[wv], out[wv]);
    wave_sync();
    NE_STORE_ACT(1, bufs[1]);
    guide_layer<1>(g, xb[wv], xa[wv], out[wv]);
    wave_sync();
    NE_STORE_ACT(2, bufs[0]);
    guide_layer<2>(g, xa[wv], xb[wv], out[wv]);
    wave_sync();
    NE_STORE_ACT(3, bufs[1]);
    guide_layer<3>(g, xb[wv], xa[wv], out[wv]);
    wave_sync();
    NE_STORE_ACT(4, bufs[0]);
    guide_layer<4>(g, xa[wv], xb[wv], out[wv]);
    wave_sync();
#undef NE_STORE_ACT
    {
      // row r's lobes 2 grp and 2 grp + 1 on lane r + 16 grp; the sums over the
      // lobes run in lobe order on every lane (values by shuffle), so they
      // round as one lane's loop would
      const int row = lane & 15, grp = lane >> 4;
      const uint32_t q = tt * 16 + uint32_t(row);
      const float* y = &out[wv][row * kLdO];
      const float* o = y + 10 * grp;
      auto lobe_sum = [&](float a, float b) {
        float acc = 0.0f;
        for (int k = 0; k < 4; ++k) {
          acc += __shfl(a, row + 16 * k);
          acc += __shfl(b, row + 16 * k);
        }
        return acc;
      };
      const uint32_t qq = q < n ? q : 0u;
      const Vec3<float> w = v3(S[6 * cap + qq], S[7 * cap + qq], S[8 * cap + qq]);
      const float r = S[9 * cap + qq];
      float mx = y[0];
      for (int k = 1; k < kGuideLobes; ++k) mx = xmax(mx, y[5 * k]);
      const float e0 = expf(o[0] - mx), e1 = expf(o[5] - mx);
      const float z = lobe_sum(e0, e1);
      float pi[2] = {e0 / z, e1 / z}, v[2], kap[2], nm[2], cs[2], mu[2][3];
#pragma unroll
      for (int k = 0; k < 2; ++k) {
        const float* p = o + 5 * k;
        nm[k] = xmax(sqrtf(p[1] * p[1] + p[2] * p[2] + p[3] * p[3]), 1e-12f);
        kap[k] = guide_kappa(p[4]);
        v[k] = vmf_pdf(kap[k], (p[1] * w.x + p[2] * w.y + p[3] * w.z) / nm[k]);
#pragma unroll
        for (int a = 0; a < 3; ++a) mu[k][a] = p[1 + a] / nm[k];
        cs[k] = mu[k][0] * w.x + mu[k][1] * w.y + mu[k][2] * w.z;
      }
      const float qsum = xmax(lobe_sum(pi[0] * v[0], pi[1] * v[1]), 1e-30f);
      if (q < n) {
        if (grp == 0) {
          loss += -r * logf(qsum);
          wsum += r;
        }
        const float sc = -r / qsum;  // d(-r log q) / dq
        uint16_t* d = t.dy + size_t(q) * kGuideWidth;
        const float wk[3] = {w.x, w.y, w.z};
#pragma unroll
        for (int k = 0; k < 2; ++k) {
          const float* p = o + 5 * k;
          uint16_t* dk = d + 10 * grp + 5 * k;
          dk[0] = f2bf(sc * pi[k] * (v[k] - qsum));
          const float pv = sc * pi[k] * v[k];
#pragma unroll
          for (int a = 0; a < 3; ++a) dk[1 + a] = f2bf(pv * kap[k] * (wk[a] - cs[k] * mu[k][a]) / nm[k]);
          dk[4] = f2bf((p[4] < 8.0f && p[4] > -10.0f) ? pv * kap[k] * vmf_dlog_dkappa(kap[k], cs[k]) : 0.0f);
        }
        for (int c = 40 + 6 * grp; c < 46 + 6 * grp; ++c) d[c] = 0;
      }
    }
  }
  // loss statistics of the block, summed over the blocks by k_guide_loss
  for (int o = 32; o > 0; o >>= 1) {
    loss += __shfl_down(loss, o);
    wsum += __shfl_down(wsum, o);
  }
  __shared__ float red[2][kWavesPerBlock];
  if (lane == 0) {
    red[0][wv] = loss;
    red[1][wv] = wsum;
  }
  __syncthreads();
  if (threadIdx.x < 2) {
    float v = 0.0f;
    for (int k = 0; k < kWavesPerBlock; ++k) v += red[threadIdx.x][k];
    t.loss_part[2 * blockIdx.x + threadIdx.x] = v;
  }
}

// loss[0..1]: the blocks' sums, in a fixed order.
__global__ __launch_bounds__(256) void k_guide_loss(GuideTrain t, int blocks) {
  __shared__ float red[2][256];
  float a = 0.0f, b = 0.0f;
  for (int k = int(threadIdx.x); k < blocks; k += 256) {
    a += t.loss_part[2 * k];
    b += t.loss_part[2 * k + 1];
  }
  red[0][threadIdx.x] = a;
  red[1][threadIdx.x] = b;
  __syncthreads();
  for (int w = 128; w > 0; w >>= 1) {
    if (int(threadIdx.x) < w) {
      red[0][threadIdx.x] += red[0][threadIdx.x + w];
      red[1][threadIdx.x] += red[1][threadIdx.x + w];
    }
    __syncthreads();
  }
  if (threadIdx.x < 2) t.loss[threadIdx.x] = red[threadIdx.x][0];
}

// ---- training: backward of layer L ------------------------------------------------
// dy: gradient w.r.t. this layer's (pre-ReLU for hidden, raw for the last) output,
// BF16 [n][64].  Writes dx = dy W^T masked by the ReLU of this layer's input
// (which is the previous layer's output) into dx (BF16) or, for L = 0, the
// encoding gradient into denc (FP32, [column][sample], read by level below);
// accumulates dW / db over the wave's tiles, then over the block's waves in
// LDS (in wave order), into the block's partial.  Bound by the latency of a
// tile's loads: 8 waves a block and as many blocks as tiles ask for (65,536
// samples: 4096 waves of one tile staged in LDS, 29 us per 64 x 64 layer; 41 us
// with two-byte reads of its columns from memory, 82 us with 512 waves of 8
// tiles besides).
constexpr int kBwdBlock = 512, kBwdWaves = kBwdBlock / 64;
template <int L>
__global__ __launch_bounds__(kBwdBlock) void k_guide_train_bwd(GuideNet g, GuideBatch b, GuideTrain t,
                                                                 const uint16_t* dy, uint16_t* dx) {
  constexpr int KIN = guide_in(L), NOUT = guide_out(L);
  // the wave's tile of layer inputs and output gradients (rows of 72: 16-byte
  // aligned, columns on different banks); the block's sums use the same space
  // after the tiles
  constexpr int kLdB = 72;
  constexpr int kTiles = kBwdWaves * 2 * 16 * kLdB * 2, kSums = (KIN * NOUT + NOUT) * 4;
  __shared__ __align__(16) unsigned char buf[kTiles > kSums ? kTiles : kSums];
  const int lane = __lane_id(), wv = int(threadIdx.x >> 6);
  uint16_t* sx = reinterpret_cast<uint16_t*>(buf) + wv * (2 * 16 * kLdB);
  uint16_t* sd = sx + 16 * kLdB;
  float* sw = reinterpret_cast<float*>(buf);
  const int r = lane & 15, kq = 4 * (lane >> 4);
  const int wid = int(blockIdx.x) * kBwdWaves + wv;
  const uint32_t n = min(*b.count, b.cap);
  const uint32_t tiles = (n + 15) / 16;
  const uint32_t cap = b.cap;
  const uint16_t* X = t.act + size_t(L) * cap * kGuideWidth;
  const uint16_t* wb = g.wb + guide_w_off(L);
  f32x4 dw[KIN / 16][NOUT / 16];
#pragma unroll
  for (int mt = 0; mt < KIN / 16; ++mt)
#pragma unroll
    for (int nt = 0; nt < NOUT / 16; ++nt) dw[mt][nt] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  float db[NOUT / 16];
#pragma unroll
  for (int nt = 0; nt < NOUT / 16; ++nt) db[nt] = 0.0f;
  for (uint32_t tt = uint32_t(wid); tt < tiles; tt += gridDim.x * uint32_t(kBwdWaves)) {
    const uint32_t row0 = tt * 16;
    // 16 rows of 128 bytes each: lane l holds 16 bytes of rows l / 8 and 8 + l / 8
    wave_sync();
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int row = 8 * h + (lane >> 3), c = 8 * (lane & 7);
      uint4 vx = make_uint4(0, 0, 0, 0), vd = vx;
      if (row0 + uint32_t(row) < n) {
        vx = *reinterpret_cast<const uint4*>(X + size_t(row0 + row) * kGuideWidth + c);
        vd = *reinterpret_cast<const uint4*>(dy + size_t(row0 + row) * kGuideWidth + c);
      }
      *reinterpret_cast<uint4*>(sx + row * kLdB + c) = vx;
      *reinterpret_cast<uint4*>(sd + row * kLdB + c) = vd;
    }
    wave_sync();
    // dx = dy W^T: A = dy rows (k = output index), B = W^T (k = output, n = input)
    f32x4 ax[KIN / 16];
#pragma unroll
    for (int mt = 0; mt < KIN / 16; ++mt) ax[mt] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int ks = 0; ks < NOUT / 16; ++ks) {
      const bf16x4 a = *reinterpret_cast<const bf16x4*>(sd + r * kLdB + 16 * ks + kq);
#pragma unroll
      for (int nt = 0; nt < KIN / 16; ++nt) {
        const bf16x4 bb = *reinterpret_cast<const bf16x4*>(wb + (16 * nt + r) * NOUT + 16 * ks + kq);
        ax[nt] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, bb, ax[nt], 0, 0, 0);
      }
    }
#pragma unroll
    for (int nt = 0; nt < KIN / 16; ++nt) {
      const int col = 16 * nt + r;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const uint32_t row = row0 + uint32_t(kq + j);
        if (row >= n) continue;
        if (L == 0) {
          if (col < kGuideEnc) t.denc[size_t(col) * cap + row] = ax[nt][j];
        } else {
          const float xin = bf2f(sx[(kq + j) * kLdB + col]);  // ReLU output of layer L-1
          dx[size_t(row) * kGuideWidth + col] = f2bf(xin > 0.0f ? ax[nt][j] : 0.0f);
        }
      }
    }
    // dW += X^T dy: A = X^T (m = input, k = row), B = dy (k = row, n = output); rows past n are zero
    bf16x4 bb[NOUT / 16];
#pragma unroll
    for (int nt = 0; nt < NOUT / 16; ++nt)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const uint16_t v = sd[(kq + j) * kLdB + 16 * nt + r];
        bb[nt][j] = short(v);
        db[nt] += bf2f(v);
      }
#pragma unroll
    for (int mt = 0; mt < KIN / 16; ++mt) {
      bf16x4 a;
#pragma unroll
      for (int j = 0; j < 4; ++j) a[j] = short(sx[(kq + j) * kLdB + 16 * mt + r]);
#pragma unroll
      for (int nt = 0; nt < NOUT / 16; ++nt) dw[mt][nt] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, bb[nt], dw[mt][nt], 0, 0, 0);
    }
  }
  __syncthreads();  // the tiles' space becomes the block's sums
  // the block's partial: dW[in][out] (lane: rows kq..kq+3 of each m-tile, column r of each n-tile), db
#pragma unroll
  for (int nt = 0; nt < NOUT / 16; ++nt) {
    db[nt] += __shfl_xor(db[nt], 16);
    db[nt] += __shfl_xor(db[nt], 32);
  }
  for (int k = 0; k < kBwdWaves; ++k) {
    if (wv == k) {
#pragma unroll
      for (int mt = 0; mt < KIN / 16; ++mt)
#pragma unroll
        for (int nt = 0; nt < NOUT / 16; ++nt)
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            float& d = sw[(16 * mt + kq + q) * NOUT + 16 * nt + r];
            d = k == 0 ? dw[mt][nt][q] : d + dw[mt][nt][q];
          }
#pragma unroll
      for (int nt = 0; nt < NOUT / 16; ++nt)
        if (lane < 16) {
          float& d = sw[KIN * NOUT + 16 * nt + r];
          d = k == 0 ? db[nt] : d + db[nt];
        }
    }
    __syncthreads();
  }
  // normalised by sum r here: a sum of all samples' unscaled terms leaves FP32's
  // range where their weights' sum is still in it
  const float scale = t.loss[1] > 0.0f ? 1.0f / t.loss[1] : 0.0f;
  float* part = t.partial + size_t(blockIdx.x) * kGuideParams;
  for (int e = int(threadIdx.x); e < KIN * NOUT; e += kBwdBlock) part[guide_w_off(L) + e] = sw[e] * scale;
  if (threadIdx.x < NOUT) part[guide_b_off(L) + threadIdx.x] = sw[KIN * NOUT + threadIdx.x] * scale;
}

// mlp_grad[p] = sum over the backward blocks of the partials, in a fixed order
// (deterministic): a block takes 64 parameters, its 16 thread groups sum the
// partials w = j mod 16 each, and the group sums are added in order.
__global__ __launch_bounds__(1024) void k_guide_reduce(GuideNet g, GuideTrain t, int parts) {
  __shared__ float part[16][64];
  const int j = int(threadIdx.x >> 6), col = int(threadIdx.x & 63);
  const int p = int(blockIdx.x) * 64 + col;
  float s = 0.0f;
  if (p < kGuideParams)
#pragma unroll 4
    for (int w = j; w < parts; w += 16) s += t.partial[size_t(w) * kGuideParams + p];
  part[j][col] = s;
  __syncthreads();
  if (j == 0 && p < kGuideParams) {
    float v = part[0][col];
    for (int k = 1; k < 16; ++k) v += part[k][col];
    g.mlp_grad[p] = v;
  }
}

// Hash-feature gradients: every sample adds (corner weight x encoding
// gradient) to 8 entries per level.  As global atomics that is 16.8 M adds per
// 65,536 samples, at about 11 G/s across the XCDs (0.9 ms uniform positions,
// 1.5 ms in a cloud).  Instead a block owns kTableRange entries of one level in
// LDS, reads a share of the samples, adds what falls into its range by LDS
// atomics, and writes the range once: no global atomics.  The sums are FP64
// because the LDS adds doubles nine times as fast as floats (64 random adds of
// a wave: ds_add_f64 21 cycles, ds_add_f32 194).  A sample is read by every
// block of its level, but only the blocks that own one of its corners work on
// it: tables of more ranges than the chip has CUs take all samples in every
// block; smaller ones split the samples into `chunks`, each with a copy of the
// ranges (t.table_part, 64 KiB per range and chunk: at most 16 MiB, as chunks x
// ranges fill the chip once: it fits in the weights' partials), and sum the
// copies after (k_guide_table_sum).  The whole training pass with its copies,
// 65,536 samples, this kernel against atomics at every level, us:
// log2_table 15: 488 / 1306, 17: 648 / 1292, 19: 658 / 1301, 21: 971 / 1360,
// 22: 1210 / 1930;
// 8192 samples: 15: 316 / 454, 21: 279 / 333.  Atomics for the large levels
// only lost at every size too (19: 1038).
constexpr uint32_t kTableRange = 8192;   // 128 KiB of LDS: one block per CU
constexpr int kTableBlock = 1024;
// entries that level l addresses (dense levels fewer than the table holds)
__host__ __device__ inline uint32_t guide_level_entries(const GuideNet& g, int l) {
  const uint32_t T = 1u << g.log2T, r1 = uint32_t(g.res[l]) + 1u;
  const uint64_t dense = uint64_t(r1) * r1 * r1;
  return dense <= T ? uint32_t(dense) : T;
}
// Range `unit` of the ranges of all levels: its level, first entry and length.
__device__ inline void guide_table_range(const GuideNet& g, uint32_t unit, int& l, uint32_t& base, uint32_t& len) {
  l = 0;
  uint32_t ent = guide_level_entries(g, 0), nr = (ent + kTableRange - 1) / kTableRange;
  while (unit >= nr) {
    unit -= nr;
    ++l;
    ent = guide_level_entries(g, l);
    nr = (ent + kTableRange - 1) / kTableRange;
  }
  base = unit * kTableRange;
  len = ent - base < kTableRange ? ent - base : kTableRange;
}
__global__ __launch_bounds__(kTableBlock) void k_guide_table_grad(GuideNet g, GuideBatch b, GuideTrain t, int chunks) {
  __shared__ double acc[2 * kTableRange];
  const uint32_t unit = blockIdx.x / uint32_t(chunks), chunk = blockIdx.x % uint32_t(chunks);
  int l;
  uint32_t base, len;
  guide_table_range(g, unit, l, base, len);
  for (uint32_t k = threadIdx.x; k < 2 * len; k += kTableBlock) acc[k] = 0.0;
  __syncthreads();
  const float scale = t.loss[1] > 0.0f ? 1.0f / t.loss[1] : 0.0f;
  const uint32_t n = min(*b.count, b.cap), T = 1u << g.log2T, r1 = uint32_t(g.res[l]) + 1u;
  const uint32_t per = (n + uint32_t(chunks) - 1) / uint32_t(chunks), q1 = min(n, (chunk + 1) * per);
  const bool dense = uint64_t(r1) * r1 * r1 <= T;
  const float rf = float(g.res[l]);
  const float* D0 = t.denc + size_t(2 * l) * b.cap;
  for (uint32_t q = chunk * per + threadIdx.x; q < q1; q += kTableBlock) {
    // the corners of guide_corner, their shared parts computed once
    const float sx = xmin(xmax(b.s[q], 0.0f), 1.0f) * rf, sy = xmin(xmax(b.s[b.cap + q], 0.0f), 1.0f) * rf,
                sz = xmin(xmax(b.s[2 * size_t(b.cap) + q], 0.0f), 1.0f) * rf;
    const float fx = xmin(floorf(sx), rf - 1.0f), fy = xmin(floorf(sy), rf - 1.0f), fz = xmin(floorf(sz), rf - 1.0f);
    const float tx = sx - fx, ty = sy - fy, tz = sz - fz;
    const uint32_t x = uint32_t(fx), y = uint32_t(fy), z = uint32_t(fz);
    const uint32_t my = dense ? r1 : 2654435761u, mz = dense ? r1 * r1 : 805459861u;
    const uint32_t hy0 = y * my, hy1 = hy0 + my, hz0 = z * mz, hz1 = hz0 + mz;
    uint32_t e[8];
    bool any = false;
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      const uint32_t xx = x + (k & 1), yy = (k & 2) ? hy1 : hy0, zz = (k & 4) ? hz1 : hz0;
      e[k] = (dense ? xx + yy + zz : (xx ^ yy ^ zz) & (T - 1u)) - base;
      any = any || e[k] < len;
    }
    if (!any) continue;
    const float d0 = D0[q] * scale, d1 = D0[b.cap + q] * scale;
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      const float w = ((k & 1) ? tx : 1.0f - tx) * ((k & 2) ? ty : 1.0f - ty) * ((k & 4) ? tz : 1.0f - tz);
      if (e[k] < len) {
        atomicAdd(&acc[2 * e[k]], double(w * d0));
        atomicAdd(&acc[2 * e[k] + 1], double(w * d1));
      }
    }
  }
  __syncthreads();
  float2* o = chunks == 1 ? reinterpret_cast<float2*>(g.table_grad) + size_t(l) * T + base
                          : reinterpret_cast<float2*>(t.table_part) + size_t(blockIdx.x) * kTableRange;
  for (uint32_t k = threadIdx.x; k < len; k += kTableBlock) o[k] = make_float2(float(acc[2 * k]), float(acc[2 * k + 1]));
}
// table_grad = the chunks' copies of each range summed in order.
__global__ __launch_bounds__(256) void k_guide_table_sum(GuideNet g, const float* part, int chunks) {
  int l;
  uint32_t base, len;
  constexpr uint32_t kBlocks = kTableRange / 256;  // per range
  const uint32_t unit = blockIdx.x / kBlocks, k = blockIdx.x % kBlocks * 256u + threadIdx.x;
  guide_table_range(g, unit, l, base, len);
  if (k >= len) return;
  const float2* p = reinterpret_cast<const float2*>(part) + size_t(unit) * uint32_t(chunks) * kTableRange + k;
  float2 s = p[0];
  for (int c = 1; c < chunks; ++c) {
    const float2 v = p[size_t(c) * kTableRange];
    s.x += v.x;
    s.y += v.y;
  }
  reinterpret_cast<float2*>(g.table_grad)[(size_t(l) << g.log2T) + base + k] = s;
}

// BF16 copy of the hash features that the encoder reads (after every change
// of the FP32 masters)
__global__ void k_guide_pack_table(GuideNet g, size_t entries) {
  const size_t i = size_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i >= entries) return;
  const float2 v = reinterpret_cast<const float2*>(g.table)[i];
  g.table_bf[i] = uint32_t(f2bf(v.x)) | (uint32_t(f2bf(v.y)) << 16);
}

__global__ void k_guide_adam(float* prm, float* grad, float* m, float* v, size_t n, float lr, float b1, float b2,
                             float eps, float c1, float c2) {
  const size_t i = size_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const float gr = grad[i];
  const float mi = b1 * m[i] + (1.0f - b1) * gr;
  const float vi = b2 * v[i] + (1.0f - b2) * gr * gr;
  m[i] = mi;
  v[i] = vi;
  prm[i] -= lr * (mi / c1) / (sqrtf(vi / c2) + eps);
  grad[i] = 0.0f;
}

__global__ void k_guide_pack(GuideNet g) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= kGuideWeights) return;
  int l = 0;
  while (l + 1 < kGuideLayers && i >= guide_w_off(l + 1)) ++l;
  const int local = i - guide_w_off(l), in = local / guide_out(l), out = local % guide_out(l);
  const uint16_t h = f2bf(g.mlp[i]);
  g.wb[i] = h;                                                   // [in][out]
  g.wf[guide_w_off(l) + out * guide_in(l) + in] = h;             // [out][in]
}

// Initial parameters: hash features U(-1e-4, 1e-4); weights U(-s, s) with
// s = sqrt(6 / fan_in) over the used inputs (He-uniform), padding zero; biases 0.
__device__ __forceinline__ float guide_u01(uint64_t seed, uint32_t stream, uint32_t i) {
  uint32_t c[4] = {i, stream, 0x6775u, 0u};
  philox10(c, uint32_t(seed), uint32_t(seed >> 32));
  return float(c[0] >> 8) * (1.0f / 16777216.0f);
}
__global__ void k_guide_init(GuideNet g, uint64_t seed, size_t table_n) {
  const size_t i = size_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i < table_n) {
    g.table[i] = (2.0f * guide_u01(seed, 1u, uint32_t(i)) - 1.0f) * 1e-4f;
    g.table_grad[i] = 0.0f; g.table_m[i] = 0.0f; g.table_v[i] = 0.0f;
  }
  if (i < size_t(kGuideParams)) {
    float val = 0.0f;
    if (i < size_t(kGuideWeights)) {
      int l = 0;
      while (l + 1 < kGuideLayers && int(i) >= guide_w_off(l + 1)) ++l;
      const int local = int(i) - guide_w_off(l), in = local / guide_out(l), out = local % guide_out(l);
      const int used_in = l == 0 ? kGuideInputs : 64, used_out = l == kGuideLayers - 1 ? kGuideOutputs : 64;
      if (in < used_in && out < used_out) {
        const float s = sqrtf(6.0f / float(used_in));
        val = (2.0f * guide_u01(seed, 2u, uint32_t(i)) - 1.0f) * s;
      }
    }
    g.mlp[i] = val;
    g.mlp_grad[i] = 0.0f; g.mlp_m[i] = 0.0f; g.mlp_v[i] = 0.0f;
  }
}

// ---- launchers ------------------------------------------------------------------------
static size_t table_words(const GuideNet& g) { return size_t(kGuideLevels) * (size_t(1) << g.log2T) * kGuideFeat; }

hipError_t launch_guide_init(const GuideNet& g, uint64_t seed, hipStream_t st) {
  const size_t n = table_words(g);
  hipLaunchKernelGGL(k_guide_init, dim3(uint32_t((n + 255) / 256)), dim3(256), 0, st, g, seed, n);
  return launch_guide_pack(g, st);
}

hipError_t launch_guide_pack(const GuideNet& g, hipStream_t st) {
  hipLaunchKernelGGL(k_guide_pack, dim3((kGuideWeights + 255) / 256), dim3(256), 0, st, g);
  const size_t entries = table_words(g) / kGuideFeat;
  hipLaunchKernelGGL(k_guide_pack_table, dim3(uint32_t((entries + 255) / 256)), dim3(256), 0, st, g, entries);
  return hipGetLastError();
}

hipError_t launch_guide_eval(const GuideNet& g, int n, const float* in6, float* out40, hipStream_t st) {
  const int tiles = (n + 63) / 64;
  const int blocks = std::max(1, std::min(4096, (tiles + kWavesPerBlock - 1) / kWavesPerBlock));
  hipLaunchKernelGGL(k_guide_eval, dim3(blocks), dim3(kGuideBlock), 0, st, g, n, in6, out40, 0);
  return hipGetLastError();
}

hipError_t launch_guide_raw(const GuideNet& g, int n, const float* in6, float* out40, hipStream_t st) {
  const int tiles = (n + 63) / 64;
  const int blocks = std::max(1, std::min(4096, (tiles + kWavesPerBlock - 1) / kWavesPerBlock));
  hipLaunchKernelGGL(k_guide_eval, dim3(blocks), dim3(kGuideBlock), 0, st, g, n, in6, out40, 1);
  return hipGetLastError();
}

hipError_t launch_guide_bake(const GuideNet& g, const GuideCache& c, float* mix, hipStream_t st) {
  const int n = c.nc * c.nc * c.nc * c.nd * c.nd;
  const int tiles = (n + 63) / 64;
  const int blocks = std::max(1, std::min(8192, (tiles + kWavesPerBlock - 1) / kWavesPerBlock));
  hipLaunchKernelGGL(k_guide_bake, dim3(blocks), dim3(kGuideBlock), 0, st, g, c, mix, n);
  return hipGetLastError();
}

// Training samples as the caller gives them (10 floats each) -> the batch's
// arrays, by a block of 256 samples through LDS; *count = n.
__global__ __launch_bounds__(256) void k_guide_set_batch(const float* aos, GuideBatch b, uint32_t n) {
  __shared__ float v[256 * 11];  // a row of 11: conflict-free columns
  const uint32_t q0 = blockIdx.x * 256u, m = n - q0 < 256u ? n - q0 : 256u;
  for (uint32_t e = threadIdx.x; e < 10u * m; e += 256u) v[e / 10u * 11u + e % 10u] = aos[size_t(q0) * 10u + e];
  __syncthreads();
  if (threadIdx.x < m)
    for (uint32_t k = 0; k < 10u; ++k) b.s[size_t(k) * b.cap + q0 + threadIdx.x] = v[threadIdx.x * 11u + k];
  if (blockIdx.x == 0 && threadIdx.x == 0) *b.count = n;
}
hipError_t launch_guide_set_batch(const float* aos, const GuideBatch& b, uint32_t n, hipStream_t st) {
  hipLaunchKernelGGL(k_guide_set_batch, dim3((n + 255) / 256), dim3(256), 0, st, aos, b, n);
  return hipGetLastError();
}

static int table_units(const GuideNet& g) {
  int units = 0;
  for (int l = 0; l < kGuideLevels; ++l) units += int((guide_level_entries(g, l) + kTableRange - 1) / kTableRange);
  return units;
}
// Chunks of the samples in the table gradient: as many as fill the chip once
// (256 CUs, one block each), at most 16.
static int table_chunks(const GuideNet& g) { return std::min(16, std::max(1, 256 / table_units(g))); }
static_assert(256ull * kTableRange * kGuideFeat <= uint64_t(kGuideParts) * kGuideParams, "table_part lies in partial");

// Gradients of the weight-normalised loss -sum r log q / sum r (1 / sum r is
// read on the device after the forward pass).  n: at least the sample count.
hipError_t launch_guide_grad(const GuideNet& g, const GuideBatch& b, const GuideTrain& t, uint32_t n, hipStream_t st) {
  const uint32_t tiles = std::max<uint32_t>(1, (std::min(n, b.cap) + 15) / 16);
  const uint32_t fblocks = std::min<uint32_t>(kGuideFwdBlocks, (tiles + kWavesPerBlock - 1) / kWavesPerBlock);
  const uint32_t blocks = std::min<uint32_t>(kGuideParts, (tiles + kBwdWaves - 1) / kBwdWaves);
  const dim3 blk(kBwdBlock);
  hipLaunchKernelGGL(k_guide_train_fwd, dim3(fblocks), dim3(kGuideBlock), 0, st, g, b, t);
  hipLaunchKernelGGL(k_guide_loss, dim3(1), dim3(256), 0, st, t, int(fblocks));
  hipLaunchKernelGGL((k_guide_train_bwd<4>), dim3(blocks), blk, 0, st, g, b, t, t.dy, t.dy2);
  hipLaunchKernelGGL((k_guide_train_bwd<3>), dim3(blocks), blk, 0, st, g, b, t, t.dy2, t.dy);
  hipLaunchKernelGGL((k_guide_train_bwd<2>), dim3(blocks), blk, 0, st, g, b, t, t.dy, t.dy2);
  hipLaunchKernelGGL((k_guide_train_bwd<1>), dim3(blocks), blk, 0, st, g, b, t, t.dy2, t.dy);
  hipLaunchKernelGGL((k_guide_train_bwd<0>), dim3(blocks), blk, 0, st, g, b, t, t.dy, t.dy2);
  hipLaunchKernelGGL(k_guide_reduce, dim3((kGuideParams + 63) / 64), dim3(1024), 0, st, g, t, int(blocks));
  const uint32_t units = uint32_t(table_units(g));
  const int chunks = table_chunks(g);
  hipLaunchKernelGGL(k_guide_table_grad, dim3(units * uint32_t(chunks)), dim3(kTableBlock), 0, st, g, b, t, chunks);
  if (chunks > 1)
    hipLaunchKernelGGL(k_guide_table_sum, dim3(units * (kTableRange / 256)), dim3(256), 0, st, g, t.table_part, chunks);
  return hipGetLastError();
}

hipError_t launch_guide_adam(const GuideNet& g, float lr_table, float lr_mlp, float beta1, float beta2, float eps,
                             int step, hipStream_t st) {
  const float c1 = 1.0f - powf(beta1, float(step)), c2 = 1.0f - powf(beta2, float(step));
  const size_t nt = table_words(g);
  hipLaunchKernelGGL(k_guide_adam, dim3(uint32_t((nt + 255) / 256)), dim3(256), 0, st, g.table, g.table_grad,
                     g.table_m, g.table_v, nt, lr_table, beta1, beta2, eps, c1, c2);
  hipLaunchKernelGGL(k_guide_adam, dim3((kGuideParams + 255) / 256), dim3(256), 0, st, g.mlp, g.mlp_grad, g.mlp_m,
                     g.mlp_v, size_t(kGuideParams), lr_mlp, beta1, beta2, eps, c1, c2);
  return launch_guide_pack(g, st);
}

}  // namespace ne
