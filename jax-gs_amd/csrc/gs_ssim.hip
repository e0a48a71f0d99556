// L1 and SSIM photometric losses of a rendered image, and their gradient, on gfx950.
//
// Reference: jax_gs/training/losses.py:4-8 (l1_loss) and :16-75 (ssim, d_ssim_loss),
// combined by jax_gs/training/trainer.py:18-26 as (1 - 0.2) l1 + 0.2 d_ssim.
//   taps    w_k = exp(-k^2 / 4.5) / sum, k = -5..5 (window 11, sigma 1.5)
//   blur    correlation with w along H, then along W, 'SAME' zero padding
//   mu1 = blur(x), mu2 = blur(y), s11 = max(0, blur(x^2) - mu1^2),
//   s22 = max(0, blur(y^2) - mu2^2), s12 = blur(x y) - mu1 mu2
//   map = (2 mu1 mu2 + C1)(2 s12 + C2) / ((mu1^2 + mu2^2 + C1)(s11 + s22 + C2)),
//   C1 = 0.01^2, C2 = 0.03^2, clipped to [-1, 1]; ssim = mean over H x W x C.
//
// Forward (one launch + a final sum): a workgroup owns 8 x 116 outputs of every channel.
// The vertical pass runs over 128 columns (116 + the halo): each thread takes one column and
// 4 output rows, reads the 14 input rows it needs once (rows are the wave's, so their
// addresses are scalar) and keeps the five blurred products (x, y, x^2, y^2, x y) in
// registers; they meet in LDS, where the horizontal pass (each thread 4 adjacent outputs of
// one row, 128-bit LDS reads of its 14-column window) completes the blur.  Per output the
// map and, when a gradient is wanted, its derivatives with respect to (mu1, blur(x^2),
// blur(x y)) -- divided by the count and gated by the clip -- are formed; a group of four
// goes to the three planes of the workspace as 16-byte stores.  |x - y| comes from the rows
// that the vertical pass holds.
// What bounds it: the two passes are 2 x 55 of some 170 vector instructions per value, about
// 27 us at 1920x1080 x 3, and reading the images with writing the planes (125 MB) 25 us.  A
// tile of 16 x 54 (halo and idle lanes: 30 % more of both passes, now 10 %) with the planes and
// the gradient staged in LDS took 72 us forward and 52 backward; this takes 47.5 and 32.5.
// Prefetching the next channel's rows beside the horizontal pass costs the forward more
// registers than it hides (53 us, with 3 waves per SIMD 51); the backward's three maps do it.
// Backward: dL/dx = blur(d/dmu1) + 2 x blur(d/dblur(x^2)) + y blur(d/dblur(x y)) (the
// blur is a correlation with a symmetric kernel and zero padding, so it is its own
// adjoint), scaled by the cotangent of the mean SSIM, plus the L1 cotangent times
// sign(x - y) / count.  Same tiling over the three planes.
// Ties follow JAX: max(0, .) and the clip pass half the cotangent at equality.
#include "gs_common.h"

namespace gs {
namespace {

constexpr int kSR = 5;                   // window radius
constexpr int kSTaps = 2 * kSR + 1;      // 11 taps
constexpr int kSTH = 8;                  // output rows per workgroup
constexpr int kSCols = 128;              // columns of the vertical pass
constexpr int kSTW = 116;                // output columns per workgroup: 29 groups of 4, all 14-column windows inside kSCols
constexpr int kSRows = 4 + 2 * kSR;      // input rows of a thread's four output rows
constexpr float kC1 = 0.01f * 0.01f;
constexpr float kC2 = 0.03f * 0.03f;

// A group of four values at any float: 16-byte accesses need only 4-byte alignment, so the rows of
// images whose width is no multiple of four take them as well (value by value, four or twelve floats
// apart from lane to lane, they took 979x546 x 3 from 20 to 23 us forward and 13.6 to 19 backward).
typedef float f4any __attribute__((ext_vector_type(4), aligned(4)));

struct Taps {
  float w[kSTaps];
};

__device__ inline float tie_step(float z) { return z > 0.0f ? 1.0f : (z == 0.0f ? 0.5f : 0.0f); }

// What a thread of the vertical pass reads of one map: rows row0 .. row0 + 13 of its column.  The
// rows are the wave's (scalar addresses); rows and columns outside the image are read at their
// nearest inside one (the caller zeroes them, in the workgroups that have any).
struct Column {
  int off;     // element of (row 0, the thread's column, channel 0), column clamped
  int row0;    // wave-uniform
  int H;
  int stride;  // elements from row to row
};
__device__ inline void load_rows(const float* __restrict__ p, const Column& c, float (&v)[kSRows]) {
#pragma unroll
  for (int i = 0; i < kSRows; ++i) {
    const int r = min(max(c.row0 + i, 0), c.H - 1);
    v[i] = (p + (int64_t)r * c.stride)[c.off];
  }
}
__device__ inline void zero_outside(const Column& c, bool col_in, float (&v)[kSRows]) {
#pragma unroll
  for (int i = 0; i < kSRows; ++i) v[i] = col_in && c.row0 + i >= 0 && c.row0 + i < c.H ? v[i] : 0.0f;
}

// Horizontal pass from LDS row `row` of NM maps: out[m][o] = sum_k w_k V[m][row][c0 + o + k].
template <int NM>
__device__ inline void horizontal4(const Taps& t, const float (*V)[kSTH][kSCols], int row, int c0, float (&out)[NM][4]) {
#pragma unroll
  for (int m = 0; m < NM; ++m) {
    float win[16];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const float4 f = *reinterpret_cast<const float4*>(&V[m][row][c0 + 4 * q]);
      win[4 * q] = f.x;
      win[4 * q + 1] = f.y;
      win[4 * q + 2] = f.z;
      win[4 * q + 3] = f.w;
    }
#pragma unroll
    for (int o = 0; o < 4; ++o) {
      float a = 0.0f;
#pragma unroll
      for (int k = 0; k < kSTaps; ++k) a = fmaf(t.w[k], win[o + k], a);
      out[m][o] = a;
    }
    __asm__ volatile("" ::: "memory");  // one map's window in registers at a time
  }
}

__device__ inline float block_sum256(float v, float* red) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
  __syncthreads();
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
  __syncthreads();
  return (red[0] + red[1]) + (red[2] + red[3]);
}

// XCD-aware tile order: consecutive workgroups go round-robin to the 8 XCDs; workgroup
// b takes tile (b % 8) * per + b / 8, so each XCD's L2 holds a band of tile rows and
// the halo rows two vertically adjacent tiles share are fetched once.
__device__ inline int ssim_tile_of_block(int b, int T) { return (b & 7) * ((T + 7) >> 3) + (b >> 3); }

// Forward, CC channels (1..4), one channel at a time.
template <int CC>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(4))) void l1_ssim_fwd_kernel(
    int H, int W, int TX, int T, const float* __restrict__ x, const float* __restrict__ y, Taps taps,
    float inv_count, float* __restrict__ gmap, float2* __restrict__ partial) {
  __shared__ __align__(16) float V[5][kSTH][kSCols];
  __shared__ float red[4];
  const int tile = ssim_tile_of_block(blockIdx.x, T);
  if (tile >= T) return;
  const int tid = threadIdx.x;
  const int ox = (tile % TX) * kSTW;  // first output column
  const int r0 = (tile / TX) * kSTH;  // first output row
  // vertical pass: column, and the wave's group of 4 rows
  const int vj = tid & 127, vq = __builtin_amdgcn_readfirstlane(tid >> 7);
  const int vcol = ox - kSR + vj;
  const bool vcol_in = vcol >= 0 && vcol < W;
  const Column col{min(max(vcol, 0), W - 1) * CC, r0 + 4 * vq - kSR, H, W * CC};
  const bool border = ox < kSR || ox - kSR + kSCols > W || r0 < kSR || r0 + kSTH + kSR > H;
  const bool vout = vj >= kSR && vj < kSR + kSTW && vcol < W;  // an output column of this tile
  const int hr = tid >> 5, hs = tid & 31;  // horizontal pass: row, group of 4 columns
  const int orow = r0 + hr, ocol = ox + 4 * hs;
  const bool h_on = 4 * hs < kSTW && orow < H && ocol < W;
  const int plane = H * W * CC;  // one gradient map, channel-planar [CC][H][W]
  float l1_acc = 0.0f, ss_acc = 0.0f;
  float xv[kSRows], yv[kSRows];
#pragma unroll 1
  for (int ch = 0; ch < CC; ++ch) {
    load_rows(x + ch, col, xv);
    load_rows(y + ch, col, yv);
    if (border) {
      zero_outside(col, vcol_in, xv);
      zero_outside(col, vcol_in, yv);
    }
    float a[5][4];
#pragma unroll
    for (int m = 0; m < 5; ++m)
#pragma unroll
      for (int o = 0; o < 4; ++o) a[m][o] = 0.0f;
#pragma unroll
    for (int i = 0; i < kSRows; ++i) {
      const float v[5] = {xv[i], yv[i], xv[i] * xv[i], yv[i] * yv[i], xv[i] * yv[i]};
#pragma unroll
      for (int o = 0; o < 4; ++o) {
        const int k = i - o;
        if (k >= 0 && k < kSTaps) {
#pragma unroll
          for (int m = 0; m < 5; ++m) a[m][o] = fmaf(taps.w[k], v[m], a[m][o]);
        }
      }
    }
    // rows outside the image hold zeros in both
    if (vout) {
#pragma unroll
      for (int o = 0; o < 4; ++o) l1_acc += fabsf(xv[kSR + o] - yv[kSR + o]);
    }
    if (ch > 0) __syncthreads();  // the previous channel is done with V
#pragma unroll
    for (int m = 0; m < 5; ++m)
#pragma unroll
      for (int o = 0; o < 4; ++o) V[m][4 * vq + o][vj] = a[m][o];
    __syncthreads();
    if (h_on) {
      float b[5][4];
      horizontal4<5>(taps, V, hr, 4 * hs, b);
      float G0[4], G1[4], G2[4];
#pragma unroll
      for (int o = 0; o < 4; ++o) {
        const float mu1 = b[0][o], mu2 = b[1][o];
        const float m11 = mu1 * mu1, m22 = mu2 * mu2, m12 = mu1 * mu2;
        const float d11 = b[2][o] - m11;
        const float s11 = fmaxf(0.0f, d11), s22 = fmaxf(0.0f, b[3][o] - m22);
        const float s12 = b[4][o] - m12;
        const float A = 2.0f * m12 + kC1, B = 2.0f * s12 + kC2;
        const float Cc = (m11 + m22) + kC1, D = (s11 + s22) + kC2;
        const float num = A * B, den = Cc * D;
        // one reciprocal for the three quotients (den >= C1 C2 > 0; ~1 ulp)
        const float rden = __builtin_amdgcn_rcpf(den);
        const float raw = num * rden;
        if (ocol + o < W) ss_acc += fminf(1.0f, fmaxf(-1.0f, raw));
        // d map / d(mu1, blur(x^2), blur(x y)), times the clip gate and 1 / count
        const float G = inv_count * (tie_step(raw + 1.0f) * tie_step(1.0f - raw));
        const float dnum = G * rden, dden = -(G * raw) * rden;
        const float dA = dnum * B, dB = dnum * A, dCc = dden * D, dD = dden * Cc;
        const float de12 = 2.0f * dB;
        const float dm12 = 2.0f * dA - de12;
        const float de11 = dD * tie_step(d11);
        const float dm11 = dCc - de11;
        G0[o] = 2.0f * mu1 * dm11 + mu2 * dm12;
        G1[o] = de11;
        G2[o] = de12;
      }
      if (gmap != nullptr) {
        float* __restrict__ g = gmap + (ch * H + orow) * W + ocol;
        if (ocol + 4 <= W) {
          *reinterpret_cast<f4any*>(g) = f4any{G0[0], G0[1], G0[2], G0[3]};
          *reinterpret_cast<f4any*>(g + plane) = f4any{G1[0], G1[1], G1[2], G1[3]};
          *reinterpret_cast<f4any*>(g + 2 * (int64_t)plane) = f4any{G2[0], G2[1], G2[2], G2[3]};
        } else {  // the row's last group
#pragma unroll
          for (int o = 0; o < 4; ++o) {
            if (ocol + o >= W) break;
            g[o] = G0[o];
            g[plane + o] = G1[o];
            g[2 * (int64_t)plane + o] = G2[o];
          }
        }
      }
    }
  }
  const float l1s = block_sum256(l1_acc, red);
  const float sss = block_sum256(ss_acc, red);
  if (tid == 0) partial[tile] = make_float2(l1s, sss);
}

// trainer.py:18-26 from the two means; same float32 operations as the host-side formula.
struct LossOut {
  float lam, one_minus_lam;
  float *terms, *total, *l1, *d;  // each may be NULL
};
__device__ inline void loss_terms(float l1, float ssim, const LossOut& o) {
  const float half = (1.0f - ssim) / 2.0f;
  const float d = fmaxf(0.0f, half), total = o.one_minus_lam * l1 + o.lam * d;
  if (o.terms != nullptr) {
    o.terms[0] = d;
    o.terms[1] = total;
    o.terms[2] = o.one_minus_lam;
    const float gate = half > 0.0f ? 1.0f : (half == 0.0f ? 0.5f : 0.0f);
    o.terms[3] = -(o.lam * 0.5f) * gate;
    o.terms[4] = 1.0f - d * 2.0f;
  }
  if (o.total != nullptr) *o.total = total;
  if (o.l1 != nullptr) *o.l1 = l1;
  if (o.d != nullptr) *o.d = d;
}

// out[0] = sum of |x - y| / count, out[1] = sum of the clipped map / count; LOSS: and the
// trainer's loss from them.
template <bool LOSS>
__global__ __launch_bounds__(1024) void l1_ssim_sum_kernel(const float2* __restrict__ partial, int nb,
                                                           float inv_count, float* __restrict__ out,
                                                           const LossOut loss) {
  __shared__ float red[2][16];
  float a = 0.0f, b = 0.0f;
  for (int i = threadIdx.x; i < nb; i += 1024) {
    const float2 v = partial[i];
    a += v.x;
    b += v.y;
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    a += __shfl_xor(a, o, 64);
    b += __shfl_xor(b, o, 64);
  }
  if ((threadIdx.x & 63) == 0) {
    red[0][threadIdx.x >> 6] = a;
    red[1][threadIdx.x >> 6] = b;
  }
  __syncthreads();
  if (threadIdx.x < 2) {
    float s = 0.0f;
    for (int w = 0; w < 16; ++w) s += red[threadIdx.x][w];
    out[threadIdx.x] = s * inv_count;
    const float ssim = __shfl(s * inv_count, 1, 64);
    if (LOSS && threadIdx.x == 0) loss_terms(s * inv_count, ssim, loss);
  }
}

// The cotangents of (l1, ssim) that the backward starts from: an array of two, or formed from
// those of the trainer's loss, of its l1 and of its d_ssim (each a device scalar, NULL for none)
// as autodiff of trainer.py:18-26 forms them (max passes half at a tie).
struct LossCot {
  const float* grad_out;
  const float* l1_ssim;
  const float *total, *l1, *d;
  float lam, one_minus_lam;
};
__device__ inline void loss_cot(const LossCot& c, float& g_l1, float& g_ss) {
  if (c.grad_out != nullptr) {
    g_l1 = c.grad_out[0];
    g_ss = c.grad_out[1];
    return;
  }
  const float half = (1.0f - c.l1_ssim[1]) / 2.0f;
  const float gate = half > 0.0f ? 1.0f : (half == 0.0f ? 0.5f : 0.0f);
  g_l1 = c.l1 != nullptr ? *c.l1 : 0.0f;
  float gd = c.d != nullptr ? *c.d : 0.0f;
  if (c.total != nullptr) {
    g_l1 += *c.total * c.one_minus_lam;
    gd += *c.total * c.lam;
  }
  g_ss = -(gd * gate / 2.0f);
}

// Backward: a thread of the horizontal pass holds its four pixels' values of every channel
// (4 CC contiguous floats) and stores their gradients; the next channel's rows of the maps are
// loaded while the horizontal pass of the current one runs.
template <int CC>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(4))) void l1_ssim_bwd_kernel(
    int H, int W, int TX, int T, const float* __restrict__ x, const float* __restrict__ y, Taps taps,
    float inv_count, const float* __restrict__ gmap, const LossCot cot,
    float* __restrict__ grad) {
  __shared__ __align__(16) float V[3][kSTH][kSCols];
  const int tile = ssim_tile_of_block(blockIdx.x, T);
  if (tile >= T) return;
  const int tid = threadIdx.x;
  const int ox = (tile % TX) * kSTW, r0 = (tile / TX) * kSTH;
  const int vj = tid & 127, vq = __builtin_amdgcn_readfirstlane(tid >> 7);
  const int vcol = ox - kSR + vj;
  const bool vcol_in = vcol >= 0 && vcol < W;
  const Column col{min(max(vcol, 0), W - 1), r0 + 4 * vq - kSR, H, W};
  const bool border = ox < kSR || ox - kSR + kSCols > W || r0 < kSR || r0 + kSTH + kSR > H;
  const int hr = tid >> 5, hs = tid & 31;
  const int orow = r0 + hr, ocol = ox + 4 * hs;
  const bool h_on = 4 * hs < kSTW && orow < H && ocol < W;
  const int64_t plane = (int64_t)H * W * CC;
  float g_l1, g_ss;
  loss_cot(cot, g_l1, g_ss);
  g_l1 *= inv_count;
  const int64_t p = ((int64_t)orow * W + ocol) * CC;  // the thread's first value
  const int nval = h_on ? min(4, W - ocol) * CC : 0;
  float v[3][kSRows];
#pragma unroll
  for (int m = 0; m < 3; ++m) load_rows(gmap + m * plane, col, v[m]);
  float xq[4 * CC], yq[4 * CC];
  if (nval == 4 * CC) {
#pragma unroll
    for (int q = 0; q < CC; ++q) {
      const f4any fx = reinterpret_cast<const f4any*>(x + p)[q], fy = reinterpret_cast<const f4any*>(y + p)[q];
      xq[4 * q] = fx.x, xq[4 * q + 1] = fx.y, xq[4 * q + 2] = fx.z, xq[4 * q + 3] = fx.w;
      yq[4 * q] = fy.x, yq[4 * q + 1] = fy.y, yq[4 * q + 2] = fy.z, yq[4 * q + 3] = fy.w;
    }
  } else {
#pragma unroll
    for (int q = 0; q < 4 * CC; ++q) {
      xq[q] = q < nval ? x[p + q] : 0.0f;
      yq[q] = q < nval ? y[p + q] : 0.0f;
    }
  }
#pragma unroll
  for (int ch = 0; ch < CC; ++ch) {
    if (border) {
#pragma unroll
      for (int m = 0; m < 3; ++m) zero_outside(col, vcol_in, v[m]);
    }
    float a[3][4];
#pragma unroll
    for (int m = 0; m < 3; ++m)
#pragma unroll
      for (int o = 0; o < 4; ++o) {
        a[m][o] = 0.0f;
#pragma unroll
        for (int k = 0; k < kSTaps; ++k) a[m][o] = fmaf(taps.w[k], v[m][o + k], a[m][o]);
      }
    if (ch > 0) __syncthreads();
#pragma unroll
    for (int m = 0; m < 3; ++m)
#pragma unroll
      for (int o = 0; o < 4; ++o) V[m][4 * vq + o][vj] = a[m][o];
    __syncthreads();
    if (ch + 1 < CC) {
#pragma unroll
      for (int m = 0; m < 3; ++m) load_rows(gmap + m * plane + (int64_t)(ch + 1) * H * W, col, v[m]);
    }
    if (h_on) {
      float b[3][4];
      horizontal4<3>(taps, V, hr, 4 * hs, b);
#pragma unroll
      for (int o = 0; o < 4; ++o) {
        const float xv = xq[o * CC + ch], yv = yq[o * CC + ch], d = xv - yv;
        const float sg = d > 0.0f ? 1.0f : (d < 0.0f ? -1.0f : 0.0f);
        const float gs = b[0][o] + 2.0f * xv * b[1][o] + yv * b[2][o];
        xq[o * CC + ch] = g_ss * gs + g_l1 * sg;  // the value is done with
      }
    }
  }
  if (nval == 4 * CC) {
#pragma unroll
    for (int q = 0; q < CC; ++q)
      reinterpret_cast<f4any*>(grad + p)[q] = f4any{xq[4 * q], xq[4 * q + 1], xq[4 * q + 2], xq[4 * q + 3]};
  } else {
#pragma unroll
    for (int q = 0; q < 4 * CC; ++q)
      if (q < nval) grad[p + q] = xq[q];
  }
}

__global__ void l1_ssim_terms_kernel(const float* __restrict__ l1_ssim, const LossOut loss) {
  loss_terms(l1_ssim[0], l1_ssim[1], loss);
}

// ---------------------------------------------------------------------------------
// Any window size (losses.py:16 window_size; the trainer uses 11, served above).  The
// taps are w_j = exp(-(j - L/2)^2 / 4.5) / sum for j < L (x = arange(L) - L//2), and
// XLA's 'SAME' correlation pads (L - 1) / 2 before and L / 2 after, so output i reads
// input i + j - lo with lo = (L - 1) / 2 (for even L the window is not centred).  Planes
// are channel-planar [C][H][W] in the workspace: V (5 vertical blurs), then G (the 3
// gradient maps, as in the 11-tap path); one thread per value, the reads of a pass hit the
// cache.  The backward applies the adjoint correlation, in_s = sum_j w_j out_{s - j + lo},
// to G along W and then H (the two passes act on different axes and commute).
constexpr int kMaxTaps = 63;
struct TapsAny {
  float w[kMaxTaps];
  int L, lo;
};

// vertical blur of x, y, x^2, y^2, x y; x, y interleaved [H][W][C]
__global__ __launch_bounds__(256) void ssim_any_vblur_kernel(int H, int W, int C, const float* __restrict__ x,
                                                             const float* __restrict__ y, TapsAny t,
                                                             float* __restrict__ V) {
  const int64_t n = (int64_t)H * W * C;
  const int64_t q = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (q >= n) return;
  const int col = (int)(q % W), r = (int)((q / W) % H), ch = (int)(q / ((int64_t)W * H));
  float a[5] = {0.0f, 0.0f, 0.0f, 0.0f, 0.0f};
  for (int j = 0; j < t.L; ++j) {
    const int rr = r + j - t.lo;
    if (rr < 0 || rr >= H) continue;
    const int64_t o = ((int64_t)rr * W + col) * C + ch;
    const float xv = x[o], yv = y[o];
    a[0] = fmaf(t.w[j], xv, a[0]);
    a[1] = fmaf(t.w[j], yv, a[1]);
    a[2] = fmaf(t.w[j], xv * xv, a[2]);
    a[3] = fmaf(t.w[j], yv * yv, a[3]);
    a[4] = fmaf(t.w[j], xv * yv, a[4]);
  }
#pragma unroll
  for (int m = 0; m < 5; ++m) V[m * n + q] = a[m];
}

// horizontal blur, the map, |x - y|, per-workgroup sums and (G != NULL) the gradient maps
__global__ __launch_bounds__(256) void ssim_any_map_kernel(int H, int W, int C, const float* __restrict__ x,
                                                           const float* __restrict__ y, TapsAny t,
                                                           const float* __restrict__ V, float inv_count,
                                                           float* __restrict__ G, float2* __restrict__ partial) {
  __shared__ float red[4];
  const int64_t n = (int64_t)H * W * C;
  const int64_t q = (int64_t)blockIdx.x * 256 + threadIdx.x;
  float l1v = 0.0f, ssv = 0.0f;
  if (q < n) {
    const int col = (int)(q % W), r = (int)((q / W) % H), ch = (int)(q / ((int64_t)W * H));
    float b[5] = {0.0f, 0.0f, 0.0f, 0.0f, 0.0f};
    for (int j = 0; j < t.L; ++j) {
      const int cc = col + j - t.lo;
      if (cc < 0 || cc >= W) continue;
#pragma unroll
      for (int m = 0; m < 5; ++m) b[m] = fmaf(t.w[j], V[m * n + q - col + cc], b[m]);
    }
    const float mu1 = b[0], mu2 = b[1];
    const float m11 = mu1 * mu1, m22 = mu2 * mu2, m12 = mu1 * mu2;
    const float d11 = b[2] - m11;
    const float s11 = fmaxf(0.0f, d11), s22 = fmaxf(0.0f, b[3] - m22);
    const float s12 = b[4] - m12;
    const float A = 2.0f * m12 + kC1, B = 2.0f * s12 + kC2;
    const float Cc = (m11 + m22) + kC1, D = (s11 + s22) + kC2;
    const float num = A * B, den = Cc * D;
    const float raw = num / den;
    ssv = fminf(1.0f, fmaxf(-1.0f, raw));
    const int64_t p = ((int64_t)r * W + col) * C + ch;
    l1v = fabsf(x[p] - y[p]);
    if (G != nullptr) {
      const float Gc = inv_count * (tie_step(raw + 1.0f) * tie_step(1.0f - raw));
      const float dnum = Gc / den, dden = -(Gc * raw) / den;
      const float dA = dnum * B, dB = dnum * A, dCc = dden * D, dD = dden * Cc;
      const float de12 = 2.0f * dB;
      const float dm12 = 2.0f * dA - de12;
      const float de11 = dD * tie_step(d11);
      const float dm11 = dCc - de11;
      G[q] = 2.0f * mu1 * dm11 + mu2 * dm12;
      G[n + q] = de11;
      G[2 * n + q] = de12;
    }
  }
  const float l1s = block_sum256(l1v, red);
  const float sss = block_sum256(ssv, red);
  if (threadIdx.x == 0) partial[blockIdx.x] = make_float2(l1s, sss);
}

// adjoint correlation of the 3 gradient maps along W
__global__ __launch_bounds__(256) void ssim_any_hadj_kernel(int H, int W, int C, TapsAny t,
                                                            const float* __restrict__ G, float* __restrict__ U) {
  const int64_t n = (int64_t)H * W * C;
  const int64_t q = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (q >= n) return;
  const int col = (int)(q % W);
  float a[3] = {0.0f, 0.0f, 0.0f};
  for (int j = 0; j < t.L; ++j) {
    const int cc = col - j + t.lo;
    if (cc < 0 || cc >= W) continue;
#pragma unroll
    for (int m = 0; m < 3; ++m) a[m] = fmaf(t.w[j], G[m * n + q - col + cc], a[m]);
  }
#pragma unroll
  for (int m = 0; m < 3; ++m) U[m * n + q] = a[m];
}

// adjoint along H, then dL/dx = g_ssim (B0 + 2 x B1 + y B2) + g_l1 sign(x - y) / count
__global__ __launch_bounds__(256) void ssim_any_grad_kernel(int H, int W, int C, const float* __restrict__ x,
                                                            const float* __restrict__ y, TapsAny t,
                                                            const float* __restrict__ U, float inv_count,
                                                            const float* __restrict__ grad_out,
                                                            float* __restrict__ grad) {
  const int64_t n = (int64_t)H * W * C;
  const int64_t q = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (q >= n) return;
  const int col = (int)(q % W), r = (int)((q / W) % H), ch = (int)(q / ((int64_t)W * H));
  float b[3] = {0.0f, 0.0f, 0.0f};
  for (int j = 0; j < t.L; ++j) {
    const int rr = r - j + t.lo;
    if (rr < 0 || rr >= H) continue;
#pragma unroll
    for (int m = 0; m < 3; ++m) b[m] = fmaf(t.w[j], U[m * n + q + (int64_t)(rr - r) * W], b[m]);
  }
  const int64_t p = ((int64_t)r * W + col) * C + ch;
  const float xv = x[p], yv = y[p], d = xv - yv;
  const float sg = d > 0.0f ? 1.0f : (d < 0.0f ? -1.0f : 0.0f);
  const float gs = b[0] + 2.0f * xv * b[1] + yv * b[2];
  grad[p] = grad_out[1] * gs + (grad_out[0] * inv_count) * sg;
}

TapsAny make_taps_any(int L) {
  TapsAny t;
  double s = 0.0, e[kMaxTaps];
  for (int j = 0; j < L; ++j) {
    const double d = (double)(j - L / 2);
    e[j] = std::exp(-d * d / (2.0 * 1.5 * 1.5));
    s += e[j];
  }
  for (int j = 0; j < kMaxTaps; ++j) t.w[j] = j < L ? (float)(e[j] / s) : 0.0f;
  t.L = L;
  t.lo = (L - 1) / 2;
  return t;
}

struct AnyLayout {
  int64_t count;
  int nblk;
  size_t v_off, g_off, part_off, total;
};

AnyLayout any_layout(int H, int W, int C) {
  AnyLayout A;
  A.count = (int64_t)H * W * C;
  A.nblk = div_up(A.count, 256);
  A.v_off = 0;
  A.g_off = ((size_t)5 * A.count * sizeof(float) + 255) & ~(size_t)255;
  A.part_off = A.g_off + (((size_t)3 * A.count * sizeof(float) + 255) & ~(size_t)255);
  A.total = A.part_off + (size_t)A.nblk * sizeof(float2);
  return A;
}

Taps make_taps() {
  Taps t;
  double s = 0.0, e[kSTaps];
  for (int k = 0; k < kSTaps; ++k) {
    const double d = (double)(k - kSR);
    e[k] = std::exp(-d * d / (2.0 * 1.5 * 1.5));
    s += e[k];
  }
  for (int k = 0; k < kSTaps; ++k) t.w[k] = (float)(e[k] / s);
  return t;
}

struct SsimLayout {
  int64_t count;
  int TX, T;  // tiles per row, tiles
  dim3 grid;
  size_t gmap_off, part_off, total;
};

SsimLayout ssim_layout(int H, int W, int C) {
  SsimLayout L;
  L.count = (int64_t)H * W * C;
  L.TX = div_up(W, kSTW);
  L.T = L.TX * div_up(H, kSTH);
  L.grid = dim3((unsigned)(div_up(L.T, 8) * 8));
  L.gmap_off = 0;
  L.part_off = ((size_t)3 * L.count * sizeof(float) + 255) & ~(size_t)255;
  L.total = L.part_off + (size_t)L.T * sizeof(float2);
  return L;
}

}  // namespace
}  // namespace gs

using namespace gs;

extern "C" size_t gs_l1_ssim_workspace_size(int height, int width, int channels) {
  if (height <= 0 || width <= 0 || channels <= 0 || channels > 4) return 0;
  return ssim_layout(height, width, channels).total;
}

namespace {
int l1_ssim_fwd_run(const char* name, void* stream, int height, int width, int channels, const float* pred,
                    const float* target, float* out, int with_grad, void* workspace, size_t workspace_bytes,
                    const LossOut* loss) {
  GS_REQUIRE(height > 0 && width > 0 && channels > 0 && channels <= 4, "%s: bad image shape %dx%dx%d", name,
             height, width, channels);
  GS_REQUIRE(pred && target && out && workspace, "%s: NULL argument", name);
  GS_REQUIRE(3 * (int64_t)height * width * channels < ((int64_t)1 << 31),
             "%s: image %dx%dx%d too large", name, height, width, channels);
  const SsimLayout L = ssim_layout(height, width, channels);
  GS_REQUIRE(workspace_bytes >= L.total, "%s: workspace of %zu bytes, %zu needed", name, workspace_bytes, L.total);
  hipStream_t s = (hipStream_t)stream;
  char* ws = (char*)workspace;
  const float inv = (float)(1.0 / (double)L.count);
  float2* part = (float2*)(ws + L.part_off);
  float* gmap = with_grad ? (float*)(ws + L.gmap_off) : nullptr;
  const Taps taps = make_taps();
  switch (channels) {
    case 1: hipLaunchKernelGGL(l1_ssim_fwd_kernel<1>, L.grid, dim3(256), 0, s, height, width, L.TX, L.T, pred, target, taps, inv, gmap, part); break;
    case 2: hipLaunchKernelGGL(l1_ssim_fwd_kernel<2>, L.grid, dim3(256), 0, s, height, width, L.TX, L.T, pred, target, taps, inv, gmap, part); break;
    case 3: hipLaunchKernelGGL(l1_ssim_fwd_kernel<3>, L.grid, dim3(256), 0, s, height, width, L.TX, L.T, pred, target, taps, inv, gmap, part); break;
    default: hipLaunchKernelGGL(l1_ssim_fwd_kernel<4>, L.grid, dim3(256), 0, s, height, width, L.TX, L.T, pred, target, taps, inv, gmap, part); break;
  }
  GS_LAUNCH_CHECK("l1_ssim_fwd_kernel");
  if (loss != nullptr)
    hipLaunchKernelGGL(l1_ssim_sum_kernel<true>, dim3(1), dim3(1024), 0, s, (const float2*)part, L.T, inv, out, *loss);
  else
    hipLaunchKernelGGL(l1_ssim_sum_kernel<false>, dim3(1), dim3(1024), 0, s, (const float2*)part, L.T, inv, out,
                       LossOut{});
  GS_LAUNCH_CHECK("l1_ssim_sum_kernel");
  return GS_OK;
}
}  // namespace

extern "C" int gs_l1_ssim(void* stream, int height, int width, int channels, const float* pred,
                          const float* target, float* out, int with_grad, void* workspace, size_t workspace_bytes) {
  return l1_ssim_fwd_run("gs_l1_ssim", stream, height, width, channels, pred, target, out, with_grad, workspace,
                         workspace_bytes, nullptr);
}

extern "C" int gs_l1_ssim_loss(void* stream, int height, int width, int channels, const float* pred,
                               const float* target, double lambda_ssim, float* l1_ssim, float* terms, float* total,
                               float* l1, float* d_ssim, int with_grad, void* workspace, size_t workspace_bytes) {
  GS_REQUIRE(terms == nullptr || (lambda_ssim >= 0.0 && lambda_ssim <= 1.0),
             "gs_l1_ssim_loss: lambda must be in [0, 1] for terms");
  const LossOut loss{(float)lambda_ssim, (float)(1.0 - lambda_ssim), terms, total, l1, d_ssim};
  return l1_ssim_fwd_run("gs_l1_ssim_loss", stream, height, width, channels, pred, target, l1_ssim, with_grad,
                         workspace, workspace_bytes, &loss);
}

namespace {
int l1_ssim_bwd_run(const char* name, void* stream, int height, int width, int channels, const float* pred,
                    const float* target, const LossCot& cot, const void* workspace, size_t workspace_bytes,
                    float* grad_pred) {
  GS_REQUIRE(height > 0 && width > 0 && channels > 0 && channels <= 4,
             "%s: bad image shape %dx%dx%d", name, height, width, channels);
  GS_REQUIRE(pred && target && (cot.grad_out || cot.l1_ssim) && workspace && grad_pred, "%s: NULL argument", name);
  GS_REQUIRE(3 * (int64_t)height * width * channels < ((int64_t)1 << 31),
             "%s: image %dx%dx%d too large", name, height, width, channels);
  const SsimLayout L = ssim_layout(height, width, channels);
  GS_REQUIRE(workspace_bytes >= L.total, "%s: workspace of %zu bytes, %zu needed", name, workspace_bytes,
             L.total);
  hipStream_t s = (hipStream_t)stream;
  const float inv = (float)(1.0 / (double)L.count);
  const float* gmap = (const float*)((const char*)workspace + L.gmap_off);
  const Taps taps = make_taps();
  switch (channels) {
    case 1: hipLaunchKernelGGL(l1_ssim_bwd_kernel<1>, L.grid, dim3(256), 0, s, height, width, L.TX, L.T, pred, target, taps, inv, gmap, cot, grad_pred); break;
    case 2: hipLaunchKernelGGL(l1_ssim_bwd_kernel<2>, L.grid, dim3(256), 0, s, height, width, L.TX, L.T, pred, target, taps, inv, gmap, cot, grad_pred); break;
    case 3: hipLaunchKernelGGL(l1_ssim_bwd_kernel<3>, L.grid, dim3(256), 0, s, height, width, L.TX, L.T, pred, target, taps, inv, gmap, cot, grad_pred); break;
    default: hipLaunchKernelGGL(l1_ssim_bwd_kernel<4>, L.grid, dim3(256), 0, s, height, width, L.TX, L.T, pred, target, taps, inv, gmap, cot, grad_pred); break;
  }
  GS_LAUNCH_CHECK("l1_ssim_bwd_kernel");
  return GS_OK;
}
}  // namespace

extern "C" int gs_l1_ssim_bwd(void* stream, int height, int width, int channels, const float* pred,
                              const float* target, const float* grad_out, const void* workspace,
                              size_t workspace_bytes, float* grad_pred) {
  return l1_ssim_bwd_run("gs_l1_ssim_bwd", stream, height, width, channels, pred, target, LossCot{grad_out}, workspace,
                         workspace_bytes, grad_pred);
}

extern "C" int gs_l1_ssim_loss_bwd(void* stream, int height, int width, int channels, const float* pred,
                                   const float* target, double lambda_ssim, const float* l1_ssim,
                                   const float* g_total, const float* g_l1, const float* g_d_ssim,
                                   const void* workspace, size_t workspace_bytes, float* grad_pred) {
  const LossCot cot{nullptr, l1_ssim, g_total, g_l1, g_d_ssim, (float)lambda_ssim, (float)(1.0 - lambda_ssim)};
  return l1_ssim_bwd_run("gs_l1_ssim_loss_bwd", stream, height, width, channels, pred, target, cot, workspace,
                         workspace_bytes, grad_pred);
}

extern "C" int gs_l1_ssim_terms(void* stream, const float* l1_ssim, double lambda_ssim, float* terms) {
  GS_REQUIRE(l1_ssim && terms, "gs_l1_ssim_terms: NULL argument");
  GS_REQUIRE(lambda_ssim >= 0.0 && lambda_ssim <= 1.0, "gs_l1_ssim_terms: lambda must be in [0, 1]");
  hipLaunchKernelGGL(l1_ssim_terms_kernel, dim3(1), dim3(1), 0, (hipStream_t)stream, l1_ssim,
                     LossOut{(float)lambda_ssim, (float)(1.0 - lambda_ssim), terms, nullptr, nullptr, nullptr});
  GS_LAUNCH_CHECK("l1_ssim_terms_kernel");
  return GS_OK;
}

extern "C" size_t gs_l1_ssim_window_workspace_size(int height, int width, int channels, int window_size) {
  if (height <= 0 || width <= 0 || channels <= 0 || window_size < 1 || window_size > kMaxTaps) return 0;
  return any_layout(height, width, channels).total;
}

extern "C" int gs_l1_ssim_window(void* stream, int height, int width, int channels, int window_size,
                                 const float* pred, const float* target, float* out, int with_grad, void* workspace,
                                 size_t workspace_bytes) {
  GS_REQUIRE(height > 0 && width > 0 && channels > 0, "gs_l1_ssim_window: bad image shape %dx%dx%d", height, width,
             channels);
  GS_REQUIRE(window_size >= 1 && window_size <= kMaxTaps, "gs_l1_ssim_window: window_size must be in [1, %d] (got %d)",
             kMaxTaps, window_size);
  GS_REQUIRE(pred && target && out && workspace, "gs_l1_ssim_window: NULL argument");
  GS_REQUIRE(5 * (int64_t)height * width * channels < ((int64_t)1 << 40), "gs_l1_ssim_window: image too large");
  const AnyLayout A = any_layout(height, width, channels);
  GS_REQUIRE(workspace_bytes >= A.total, "gs_l1_ssim_window: workspace of %zu bytes, %zu needed", workspace_bytes,
             A.total);
  hipStream_t s = (hipStream_t)stream;
  char* ws = (char*)workspace;
  const TapsAny t = make_taps_any(window_size);
  const float inv = (float)(1.0 / (double)A.count);
  float* V = (float*)(ws + A.v_off);
  float* G = with_grad ? (float*)(ws + A.g_off) : nullptr;
  float2* part = (float2*)(ws + A.part_off);
  hipLaunchKernelGGL(ssim_any_vblur_kernel, dim3(A.nblk), dim3(256), 0, s, height, width, channels, pred, target, t,
                     V);
  GS_LAUNCH_CHECK("ssim_any_vblur_kernel");
  hipLaunchKernelGGL(ssim_any_map_kernel, dim3(A.nblk), dim3(256), 0, s, height, width, channels, pred, target, t,
                     (const float*)V, inv, G, part);
  GS_LAUNCH_CHECK("ssim_any_map_kernel");
  hipLaunchKernelGGL(l1_ssim_sum_kernel<false>, dim3(1), dim3(1024), 0, s, (const float2*)part, A.nblk, inv, out,
                     LossOut{});
  GS_LAUNCH_CHECK("l1_ssim_sum_kernel");
  return GS_OK;
}

extern "C" int gs_l1_ssim_window_bwd(void* stream, int height, int width, int channels, int window_size,
                                     const float* pred, const float* target, const float* grad_out, void* workspace,
                                     size_t workspace_bytes, float* grad_pred) {
  GS_REQUIRE(height > 0 && width > 0 && channels > 0, "gs_l1_ssim_window_bwd: bad image shape %dx%dx%d", height,
             width, channels);
  GS_REQUIRE(window_size >= 1 && window_size <= kMaxTaps,
             "gs_l1_ssim_window_bwd: window_size must be in [1, %d] (got %d)", kMaxTaps, window_size);
  GS_REQUIRE(pred && target && grad_out && workspace && grad_pred, "gs_l1_ssim_window_bwd: NULL argument");
  const AnyLayout A = any_layout(height, width, channels);
  GS_REQUIRE(workspace_bytes >= A.total, "gs_l1_ssim_window_bwd: workspace of %zu bytes, %zu needed",
             workspace_bytes, A.total);
  hipStream_t s = (hipStream_t)stream;
  char* ws = (char*)workspace;
  const TapsAny t = make_taps_any(window_size);
  const float inv = (float)(1.0 / (double)A.count);
  const float* G = (const float*)(ws + A.g_off);
  float* U = (float*)(ws + A.v_off);  // the forward's vertical blurs are dead by now
  hipLaunchKernelGGL(ssim_any_hadj_kernel, dim3(A.nblk), dim3(256), 0, s, height, width, channels, t, G, U);
  GS_LAUNCH_CHECK("ssim_any_hadj_kernel");
  hipLaunchKernelGGL(ssim_any_grad_kernel, dim3(A.nblk), dim3(256), 0, s, height, width, channels, pred, target, t,
                     (const float*)U, inv, grad_out, grad_pred);
  GS_LAUNCH_CHECK("ssim_any_grad_kernel");
  return GS_OK;
}
