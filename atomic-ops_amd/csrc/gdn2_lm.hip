// Element-wise and row-wise passes of the language-model block around the operator (e2e_lm.py:
// the causal depthwise convolutions, gates and norms of the reference's benchmark LM) on gfx950.
//
// A block's products are plain library GEMMs; between them stand chains of element-wise steps that
// torch runs as one memory pass each (a convolution alone is four multiply-adds over shifted
// copies).  All of it is bound by HBM, so each chain here is one kernel that reads its GEMM's
// output once and writes what the next product or the operator reads, in that reader's layout:
//   premix   the rows y = x [Wq | Wk | Wv | We | Ww | Wo | Wd] of one wide GEMM -> q, k (conv, SiLU,
//            l2 norm), v (conv, SiLU, clip), the gates b, w and g, all head-major as the operator
//            takes them, and the output gate's logits;
//   rms      RMS norm of rows, optionally of the operator's head-major o and times SiLU(gate);
//   swiglu   SiLU(gate) * up.
// The backward kernels recompute the cheap intermediates from the same rows instead of reading
// stored ones, and leave per-workgroup partial sums of the parameter gradients that lm_reduce adds
// in a fixed order.
// The benchmark LM's forward and backward (B8 L2048, 8 blocks): 73.5 ms with torch's passes, of
// which about 33 were these chains, 38.4 ms with the kernels below (4.5 ms of them).
#include "gdn2_kernels.hpp"

namespace gdn2 {

// e^x to about 1 ulp: x log2(e) in two floats, one hardware 2^y.  Arguments are held to [-103, 88],
// where the result stays a normal float (or 0); NaN is kept.
__device__ __forceinline__ float exp_1ulp(float x) {
  x = clip_nan(x, -103.f, 88.f);
  const float n = x * 1.44269504088896341f;
  const float r = fmaf(x, 1.44269504088896341f, -n) + x * 1.925963033e-8f;
  const float e = __builtin_amdgcn_exp2f(n);
  return fmaf(e, r * 0.693147180559945f, e);
}
// 1 / (1 + e^-x): the hardware reciprocal and one Newton step
__device__ __forceinline__ float sigmoid_1ulp(float x) {
  const float a = 1.f + exp_1ulp(-x);
  const float y = __builtin_amdgcn_rcpf(a);
  return fmaf(fmaf(-a, y, 1.f), y, y);
}
__device__ __forceinline__ float softplus_t(float x) { return x > 20.f ? x : log1pf(expf(x)); }   // torch's softplus
template <int N>
__device__ __forceinline__ float lanes_sum(float x) {
#pragma unroll
  for (int m = N / 2; m >= 1; m >>= 1) x += __shfl_xor(x, m);
  return x;
}
struct F4 {
  float v[4];
};
__device__ __forceinline__ F4 ldf(const float* p) {
  const float4 x = *reinterpret_cast<const float4*>(p);
  return F4{{x.x, x.y, x.z, x.w}};
}
__device__ __forceinline__ void stf(float* p, const F4& x) {
  *reinterpret_cast<float4*>(p) = make_float4(x.v[0], x.v[1], x.v[2], x.v[3]);
}

// ------------------------------------------------------------------------------------
// premix.  A workgroup (256 threads) takes 128 tokens of one (batch, head) and one role
// (blockIdx.y): 0..2 the convolutions of q, k, v; 3, 4 the erase and write gates; 5 the output
// gate's logits (a copy out of the wide rows); 6 the decay.  D / 4 lanes hold one token's head,
// four channels each, so a row is one 512-byte (D = 128) access and the head norm is a reduction
// over those lanes; a lane group walks TR consecutive tokens, so the convolution's window stays in
// registers and a token's row is read once plus 3 / TR for the window's start.  Four tokens' loads
// are issued together.
// B8 L2048 H6 D128: 0.65 GB in 120 us forward (5.5 TB/s), 0.9 GB in 190 us backward (4.8 TB/s).
// ------------------------------------------------------------------------------------
constexpr int LM_TOK = 128;

template <int D>
struct LmTile {
  static constexpr int LPR = D / 4, NG = 256 / LPR, TR = LM_TOK / NG;
  int lane, grp, h, b, tile, t0;
  __device__ LmTile(int L, int H) {
    const int nt = (L + LM_TOK - 1) / LM_TOK;
    lane = threadIdx.x % LPR;
    grp = threadIdx.x / LPR;
    h = blockIdx.x % H;
    tile = (blockIdx.x / H) % nt;
    b = blockIdx.x / (H * nt);
    t0 = tile * LM_TOK + grp * TR;
  }
};

template <int D>
__global__ __launch_bounds__(256) void lm_premix_fwd_kernel(LmPremixArgs a) {
  using Ti = LmTile<D>;
  constexpr int LPR = Ti::LPR, TR = Ti::TR;
  const Ti ti(a.L, a.H);
  const int C = a.H * D, role = blockIdx.y, ch = ti.h * D + 4 * ti.lane, t0 = ti.t0, L = a.L;
  const float* __restrict__ yb = a.y + (size_t)ti.b * L * a.ldy;
  const size_t hb = ((size_t)(ti.b * a.H + ti.h) * L) * D + 4 * ti.lane;
  const F4 zero{{0.f, 0.f, 0.f, 0.f}};
  if (role < 3) {
    const float* __restrict__ yc = yb + role * C + ch;
    auto row = [&](int t) { return t >= 0 && t < L ? ldf(yc + (size_t)t * a.ldy) : zero; };
    F4 wt[4];                                        // channel c's four taps
#pragma unroll
    for (int c = 0; c < 4; ++c) wt[c] = ldf(a.cw[role] + 4 * (ch + c));
    const F4 bias = ldf(a.cb[role] + ch);
    float* __restrict__ out = a.out[role] + hb;
    F4 y1 = row(t0 - 1), y2 = row(t0 - 2), y3 = row(t0 - 3);
    for (int i = 0; i < TR; i += 4) {
      F4 yn[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) yn[j] = row(t0 + i + j);
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int t = t0 + i + j;
        F4 s;
        float ss = 0.f;
#pragma unroll
        for (int c = 0; c < 4; ++c) {
          float u = fmaf(yn[j].v[c], wt[c].v[3], bias.v[c]);
          u = fmaf(y1.v[c], wt[c].v[2], u);
          u = fmaf(y2.v[c], wt[c].v[1], u);
          u = fmaf(y3.v[c], wt[c].v[0], u);
          s.v[c] = u * sigmoid_1ulp(u);
          ss = fmaf(s.v[c], s.v[c], ss);
        }
        if (role < 2) {
          const float r = rsqrtf(lanes_sum<LPR>(ss) + 1e-6f);
#pragma unroll
          for (int c = 0; c < 4; ++c) s.v[c] *= r;
        } else {
#pragma unroll
          for (int c = 0; c < 4; ++c) s.v[c] = clip_nan(s.v[c], -50.f, 50.f);
        }
        if (t < L) stf(out + (size_t)t * D, s);
        y3 = y2;
        y2 = y1;
        y1 = yn[j];
      }
    }
    return;
  }
  if (role < 6) {
    const float* __restrict__ yc = yb + role * C + ch;
    const F4 bias = role < 5 ? ldf(a.gb[role - 3] + ch) : zero;
    // erase -> b (output 4), write -> w (output 3)
    float* __restrict__ out = role < 5 ? a.out[7 - role] + hb : a.og + (size_t)ti.b * L * C + ch;
    const int ldo = role < 5 ? D : C;
    for (int i = 0; i < TR; i += 4) {
      F4 yn[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) yn[j] = t0 + i + j < L ? ldf(yc + (size_t)(t0 + i + j) * a.ldy) : zero;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        if (role < 5) {
#pragma unroll
          for (int c = 0; c < 4; ++c) yn[j].v[c] = sigmoid_1ulp(yn[j].v[c] + bias.v[c]);
        }
        if (t0 + i + j < L) stf(out + (size_t)(t0 + i + j) * ldo, yn[j]);
      }
    }
    return;
  }
  // the head's decay: every lane of the group forms the token's scalar and writes its channels
  const float A = expf(clip_nan(a.decay_a[ti.h], -20.f, 20.f)), db = a.decay_b[ti.h];
  float* __restrict__ out = a.out[5] + hb;
  for (int i = 0; i < TR; ++i) {
    const int t = t0 + i;
    if (t >= L) break;
    const float x = yb[(size_t)t * a.ldy + 6 * C + ti.h] + db;
    const float ldh = -A * softplus_t(x);
    // nan_to_num(nan = 0, +inf = 0, -inf = -20)
    const float ld = ldh != ldh ? 0.f : (ldh == __builtin_inff() ? 0.f : (ldh == -__builtin_inff() ? -20.f : ldh));
    const float g = -fminf(fabsf(ld), a.g_max);
    stf(out + (size_t)t * D, F4{{g, g, g, g}});
  }
}

// Backward: dy (N x ldy, every column written) and per (batch, token tile) partial sums of the
// parameter gradients, row p = b nt + tile of lm_premix_params(H, D) floats:
//   q, k, v: 4 C taps (channel-major) then C biases each; erase and write biases C each; decay
//   bias H; decay_a H.
// dy[t] needs du[t .. t+3] (u the convolution's output): each group walks three tokens past its
// run to form them.
template <int D>
__global__ __launch_bounds__(256) void lm_premix_bwd_kernel(LmPremixBwdArgs a) {
  using Ti = LmTile<D>;
  constexpr int LPR = Ti::LPR, NG = Ti::NG, TR = Ti::TR;
  __shared__ float red[256 * 20];
  const Ti ti(a.f.L, a.f.H);
  const int H = a.f.H, L = a.f.L, ldy = a.f.ldy;
  const int C = H * D, role = blockIdx.y, ch = ti.h * D + 4 * ti.lane, t0 = ti.t0;
  const float* __restrict__ yb = a.f.y + (size_t)ti.b * L * ldy;
  float* __restrict__ dyb = a.dy + (size_t)ti.b * L * ldy;
  const size_t hb = ((size_t)(ti.b * H + ti.h) * L) * D + 4 * ti.lane;
  const int nt = (L + LM_TOK - 1) / LM_TOK;
  float* __restrict__ part = a.part + (size_t)(ti.b * nt + ti.tile) * (17 * C + 2 * H);
  const F4 zero{{0.f, 0.f, 0.f, 0.f}};
  if (role < 3) {
    const float* __restrict__ yc = yb + role * C + ch;
    const float* __restrict__ dc = a.d[role] + hb;
    float* __restrict__ dyc = dyb + role * C + ch;
    auto row = [&](int t) { return t >= 0 && t < L ? ldf(yc + (size_t)t * ldy) : zero; };
    auto grad = [&](int t) { return t < L ? ldf(dc + (size_t)t * D) : zero; };
    F4 wt[4], acc[4];                                // acc[c]: channel c's four taps
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      wt[c] = ldf(a.f.cw[role] + 4 * (ch + c));
      acc[c] = zero;
    }
    const F4 bias = ldf(a.f.cb[role] + ch);
    F4 accb = zero, y1 = row(t0 - 1), y2 = row(t0 - 2), y3 = row(t0 - 3);
    F4 d1 = zero, d2 = zero, d3 = zero;              // du of the three tokens before
    for (int i = 0; i < TR + 3; i += 4) {
      F4 yn[4], dn[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        yn[j] = row(t0 + i + j);
        dn[j] = grad(t0 + i + j);
      }
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int t = t0 + i + j;
        float u[4], sg[4], s[4], S = 0.f, P = 0.f;
#pragma unroll
        for (int c = 0; c < 4; ++c) {
          u[c] = fmaf(yn[j].v[c], wt[c].v[3], bias.v[c]);
          u[c] = fmaf(y1.v[c], wt[c].v[2], u[c]);
          u[c] = fmaf(y2.v[c], wt[c].v[1], u[c]);
          u[c] = fmaf(y3.v[c], wt[c].v[0], u[c]);
          sg[c] = sigmoid_1ulp(u[c]);
          s[c] = u[c] * sg[c];
          S = fmaf(s[c], s[c], S);
          P = fmaf(dn[j].v[c], s[c], P);
        }
        F4 du;
        if (role < 2) {
          // q = s r, r = rsqrt(sum s^2 + eps): ds = r (dq - s r^2 sum(dq s))
          const float r = rsqrtf(lanes_sum<LPR>(S) + 1e-6f), m = r * r * lanes_sum<LPR>(P);
#pragma unroll
          for (int c = 0; c < 4; ++c) du.v[c] = r * fmaf(-s[c], m, dn[j].v[c]);
        } else {
#pragma unroll
          for (int c = 0; c < 4; ++c) du.v[c] = s[c] >= -50.f && s[c] <= 50.f ? dn[j].v[c] : 0.f;
        }
#pragma unroll
        for (int c = 0; c < 4; ++c) du.v[c] = t < L ? du.v[c] * (sg[c] * fmaf(u[c], 1.f - sg[c], 1.f)) : 0.f;
        if (i + j < TR) {
#pragma unroll
          for (int c = 0; c < 4; ++c) {
            acc[c].v[0] = fmaf(du.v[c], y3.v[c], acc[c].v[0]);
            acc[c].v[1] = fmaf(du.v[c], y2.v[c], acc[c].v[1]);
            acc[c].v[2] = fmaf(du.v[c], y1.v[c], acc[c].v[2]);
            acc[c].v[3] = fmaf(du.v[c], yn[j].v[c], acc[c].v[3]);
            accb.v[c] += du.v[c];
          }
        }
        if (i + j >= 3 && i + j < TR + 3 && t - 3 < L) {
          F4 o;
#pragma unroll
          for (int c = 0; c < 4; ++c)
            o.v[c] = fmaf(d3.v[c], wt[c].v[3], fmaf(d2.v[c], wt[c].v[2], fmaf(d1.v[c], wt[c].v[1], du.v[c] * wt[c].v[0])));
          stf(dyc + (size_t)(t - 3) * ldy, o);
        }
        d3 = d2;
        d2 = d1;
        d1 = du;
        y3 = y2;
        y2 = y1;
        y1 = yn[j];
      }
    }
    // [group][lane][20]: four channels' taps, then their biases
    float* my = red + threadIdx.x * 20;
#pragma unroll
    for (int c = 0; c < 4; ++c) {
#pragma unroll
      for (int j = 0; j < 4; ++j) my[4 * c + j] = acc[c].v[j];
      my[16 + c] = accb.v[c];
    }
    __syncthreads();
    for (int x = threadIdx.x; x < LPR * 20; x += 256) {
      float sum = 0.f;
      for (int n = 0; n < NG; ++n) sum += red[n * LPR * 20 + x];
      const int ln = x / 20, k = x % 20, c0 = ti.h * D + 4 * ln;
      part[5 * C * role + (k < 16 ? 4 * c0 + k : 4 * C + c0 + k - 16)] = sum;
    }
    return;
  }
  if (role < 6) {
    float* __restrict__ dyc = dyb + role * C + ch;
    if (role == 5) {
      const float* __restrict__ src = a.dog + (size_t)ti.b * L * C + ch;
      for (int i = 0; i < TR; ++i)
        if (t0 + i < L) stf(dyc + (size_t)(t0 + i) * ldy, ldf(src + (size_t)(t0 + i) * C));
      return;
    }
    const float* __restrict__ dc = a.d[7 - role] + hb;
    const float* __restrict__ sc = a.f.out[7 - role] + hb;
    F4 acc = zero;
    for (int i = 0; i < TR; i += 4) {
      F4 dn[4], sn[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int t = t0 + i + j;
        dn[j] = t < L ? ldf(dc + (size_t)t * D) : zero;
        sn[j] = t < L ? ldf(sc + (size_t)t * D) : zero;
      }
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int t = t0 + i + j;
        F4 o;
#pragma unroll
        for (int c = 0; c < 4; ++c) {
          o.v[c] = dn[j].v[c] * ((1.f - sn[j].v[c]) * sn[j].v[c]);
          acc.v[c] += o.v[c];
        }
        if (t < L) stf(dyc + (size_t)t * ldy, o);
      }
    }
    stf(red + 4 * threadIdx.x, acc);
    __syncthreads();
    for (int x = threadIdx.x; x < LPR * 4; x += 256) {
      float sum = 0.f;
      for (int n = 0; n < NG; ++n) sum += red[n * LPR * 4 + x];
      part[15 * C + (role - 3) * C + ti.h * D + x] = sum;
    }
    return;
  }
  // decay: the channel sum of dg, then the scalar chain on every lane (lane 0 writes)
  const float ca = clip_nan(a.f.decay_a[ti.h], -20.f, 20.f), A = expf(ca), db = a.f.decay_b[ti.h];
  const float* __restrict__ dc = a.d[5] + hb;
  float accx = 0.f, acca = 0.f;
  for (int i = 0; i < TR; ++i) {
    const int t = t0 + i;
    if (t >= L) break;                               // the same for every lane of the group
    const F4 d4 = ldf(dc + (size_t)t * D);
    const float dg = lanes_sum<LPR>((d4.v[0] + d4.v[1]) + (d4.v[2] + d4.v[3]));
    const float x = yb[(size_t)t * ldy + 6 * C + ti.h] + db, sp = softplus_t(x), ldh = -A * sp;
    const bool fin = __builtin_isfinite(ldh);        // nan_to_num passes no gradient elsewhere
    // g = -min(|ld|, g_max): the gradient passes where |ld| <= g_max, with the sign of ld
    const float ad = fabsf(ldh);
    const float dld = fin && ad <= a.f.g_max ? -dg * (ldh > 0.f ? 1.f : (ldh < 0.f ? -1.f : 0.f)) : 0.f;
    const float dsp = -A * dld;
    const float dx = x > 20.f ? dsp : dsp * sigmoid_1ulp(x);
    accx += dx;
    acca = fmaf(-sp, dld, acca);
    if (ti.lane == 0) dyb[(size_t)t * ldy + 6 * C + ti.h] = dx;
    // the columns past the last decay are padding: zero, since the products read them
    if (ti.h == 0)
      for (int c = 6 * C + H + ti.lane; c < ldy; c += LPR) dyb[(size_t)t * ldy + c] = 0.f;
  }
  if (ti.lane == 0) {
    red[2 * ti.grp] = accx;
    red[2 * ti.grp + 1] = acca;
  }
  __syncthreads();
  if (threadIdx.x < 2) {
    float sum = 0.f;
    for (int n = 0; n < NG; ++n) sum += red[2 * n + threadIdx.x];
    const float a0 = a.f.decay_a[ti.h];
    if (threadIdx.x == 0) part[17 * C + ti.h] = sum;
    else part[17 * C + H + ti.h] = a0 >= -20.f && a0 <= 20.f ? sum * A : 0.f;
  }
}

// out[r] = sum_p part[p][r], p ascending within four quarters that are then added in order
__global__ __launch_bounds__(256) void lm_reduce_kernel(const float* part, float* out, int rows, int cols) {
  __shared__ float red[256];
  const int c = blockIdx.x * 64 + (threadIdx.x & 63), seg = threadIdx.x >> 6;
  const int per = (rows + 3) / 4, p0 = seg * per, p1 = min(rows, p0 + per);
  float s = 0.f;
  if (c < cols) {
#pragma unroll 8
    for (int p = p0; p < p1; ++p) s += part[(size_t)p * cols + c];
  }
  red[threadIdx.x] = s;
  __syncthreads();
  if (seg == 0 && c < cols) out[c] = ((red[c & 63] + red[64 + (c & 63)]) + red[128 + (c & 63)]) + red[192 + (c & 63)];
}

// ------------------------------------------------------------------------------------
// rms: y = x rsqrt(mean(x^2) + eps) scale over rows of C floats, one wave per row (NQ float4s per
// lane).  GATED: x is the operator's head-major output (row (b, t) gathered over the heads) and
// y is further multiplied by SiLU(gate).  Backward: dx (GATED: head-major), the gate's gradient,
// dx += res when given (the residual branch's gradient, so that no separate addition reads it
// back), and per-workgroup partial sums of dscale; a wave takes RMS_ROWS rows in turn.
// ------------------------------------------------------------------------------------
constexpr int RMS_ROWS = 8;

template <int NQ, bool GATED>
__device__ __forceinline__ size_t rms_at(const LmRmsArgs& a, int row, int c) {
  if constexpr (!GATED) return (size_t)row * a.C + c;
  const int b = row / a.L, t = row - b * a.L, h = c / a.D, d = c - h * a.D;
  return (((size_t)b * (a.C / a.D) + h) * a.L + t) * a.D + d;
}

template <int NQ, bool GATED>
__global__ __launch_bounds__(256) void lm_rms_fwd_kernel(LmRmsArgs a) {
  const int row = blockIdx.x * 4 + (threadIdx.x >> 6), l = lane_id();
  if (row >= a.rows) return;
  F4 x[NQ], gt[NQ];
  float ss = 0.f;
#pragma unroll
  for (int i = 0; i < NQ; ++i) {
    const int c = 4 * (l + 64 * i);
    x[i] = F4{{0.f, 0.f, 0.f, 0.f}};
    gt[i] = x[i];
    if (c < a.C) {
      x[i] = ldf(a.x + rms_at<NQ, GATED>(a, row, c));
      if constexpr (GATED) gt[i] = ldf(a.gate + (size_t)row * a.C + c);
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) ss = fmaf(x[i].v[e], x[i].v[e], ss);
  }
  const float r = rsqrtf(lanes_sum<64>(ss) * a.inv_c + 1e-6f);
#pragma unroll
  for (int i = 0; i < NQ; ++i) {
    const int c = 4 * (l + 64 * i);
    if (c >= a.C) continue;
    const F4 sc = ldf(a.scale + c);
    F4 y;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      y.v[e] = (x[i].v[e] * r) * sc.v[e];
      if constexpr (GATED) y.v[e] *= gt[i].v[e] * sigmoid_1ulp(gt[i].v[e]);
    }
    stf(a.y + (size_t)row * a.C + c, y);
  }
}

template <int NQ, bool GATED>
__global__ __launch_bounds__(256) void lm_rms_bwd_kernel(LmRmsArgs a) {
  __shared__ float red[4 * 256 * NQ];
  const int wv = threadIdx.x >> 6, l = lane_id(), row0 = (blockIdx.x * 4 + wv) * RMS_ROWS;
  F4 acc[NQ], sc[NQ];
#pragma unroll
  for (int i = 0; i < NQ; ++i) {
    const int c = 4 * (l + 64 * i);
    acc[i] = F4{{0.f, 0.f, 0.f, 0.f}};
    sc[i] = c < a.C ? ldf(a.scale + c) : acc[i];
  }
  for (int k = 0; k < RMS_ROWS; ++k) {
    const int row = row0 + k;
    if (row >= a.rows) break;
    F4 x[NQ], dy[NQ], gt[NQ], rs[NQ];
    float ss = 0.f;
#pragma unroll
    for (int i = 0; i < NQ; ++i) {
      const int c = 4 * (l + 64 * i);
      x[i] = dy[i] = gt[i] = rs[i] = F4{{0.f, 0.f, 0.f, 0.f}};
      if (c < a.C) {
        x[i] = ldf(a.x + rms_at<NQ, GATED>(a, row, c));
        dy[i] = ldf(a.dy + (size_t)row * a.C + c);
        if constexpr (GATED) gt[i] = ldf(a.gate + (size_t)row * a.C + c);
        else if (a.res) rs[i] = ldf(a.res + (size_t)row * a.C + c);
      }
#pragma unroll
      for (int e = 0; e < 4; ++e) ss = fmaf(x[i].v[e], x[i].v[e], ss);
    }
    const float r = rsqrtf(lanes_sum<64>(ss) * a.inv_c + 1e-6f);
    float m = 0.f;
#pragma unroll
    for (int i = 0; i < NQ; ++i) {
      const int c = 4 * (l + 64 * i);
      F4 dgate;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float n = x[i].v[e] * r;
        float d = dy[i].v[e];
        if constexpr (GATED) {
          const float s = sigmoid_1ulp(gt[i].v[e]);
          dgate.v[e] = (d * (n * sc[i].v[e])) * (s * fmaf(gt[i].v[e], 1.f - s, 1.f));
          d *= gt[i].v[e] * s;
        }
        acc[i].v[e] = fmaf(d, n, acc[i].v[e]);
        dy[i].v[e] = d * sc[i].v[e];                 // d of the normalised value
        x[i].v[e] = n;
        m = fmaf(dy[i].v[e], n, m);
      }
      if constexpr (GATED)
        if (c < a.C) stf(a.dgate + (size_t)row * a.C + c, dgate);
    }
    m = lanes_sum<64>(m) * a.inv_c;
#pragma unroll
    for (int i = 0; i < NQ; ++i) {
      const int c = 4 * (l + 64 * i);
      if (c >= a.C) continue;
      F4 dx;
#pragma unroll
      for (int e = 0; e < 4; ++e) dx.v[e] = fmaf(r, fmaf(-x[i].v[e], m, dy[i].v[e]), rs[i].v[e]);
      stf(a.dx + rms_at<NQ, GATED>(a, row, c), dx);
    }
  }
#pragma unroll
  for (int i = 0; i < NQ; ++i) stf(red + wv * 256 * NQ + 256 * i + 4 * l, acc[i]);
  __syncthreads();
  for (int c = threadIdx.x; c < a.C; c += 256)
    a.part[(size_t)blockIdx.x * a.C + c] =
        ((red[c] + red[256 * NQ + c]) + red[512 * NQ + c]) + red[768 * NQ + c];
}

// ------------------------------------------------------------------------------------
// swiglu: gu rows [gate | up] of 2 M floats -> act = SiLU(gate) up (rows of M); backward dgu.
// One float4 of act per thread.
// ------------------------------------------------------------------------------------
template <bool BWD>
__global__ __launch_bounds__(256) void lm_swiglu_kernel(const float* gu, const float* dact, float* out, int rows, int M) {
  const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
  const int q = M / 4;
  const size_t row = i / q;
  const int c = 4 * (int)(i - row * q);
  if (row >= (size_t)rows) return;
  const F4 x = ldf(gu + row * 2 * M + c), u = ldf(gu + row * 2 * M + M + c);
  F4 y, z;
  if constexpr (!BWD) {
#pragma unroll
    for (int e = 0; e < 4; ++e) y.v[e] = (x.v[e] * sigmoid_1ulp(x.v[e])) * u.v[e];
    stf(out + row * M + c, y);
  } else {
    const F4 d = ldf(dact + row * M + c);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const float s = sigmoid_1ulp(x.v[e]);
      y.v[e] = (d.v[e] * u.v[e]) * (s * fmaf(x.v[e], 1.f - s, 1.f));
      z.v[e] = d.v[e] * (x.v[e] * s);
    }
    stf(out + row * 2 * M + c, y);
    stf(out + row * 2 * M + M + c, z);
  }
}

// ------------------------------------------------------------------------------------
// The matrices that share an input as one: n matrices of (rows, width[j]) side by side in rows of
// ld floats (columns past the last one zero), and back into n contiguous matrices.
// ------------------------------------------------------------------------------------
template <bool SPLIT>
__global__ __launch_bounds__(256) void lm_columns_kernel(LmColumnsArgs a) {
  const int row = blockIdx.y, c = blockIdx.x * 256 + threadIdx.x;
  if (c >= a.ld) return;
  int j = 0, c0 = 0;
#pragma unroll
  for (int k = 0; k < LM_MAX_PARTS; ++k)
    if (k < a.n && c >= a.start[k]) {
      j = k;
      c0 = a.start[k];
    }
  const int wd = a.width[j], x = c - c0;
  if constexpr (SPLIT) {
    if (x < wd) a.part[j][(size_t)row * wd + x] = a.wide[(size_t)row * a.ld + c];
  } else {
    a.wide[(size_t)row * a.ld + c] = x < wd ? a.part[j][(size_t)row * wd + x] : 0.f;
  }
}

hipError_t launch_lm_premix_fwd(int D, const LmPremixArgs& a, hipStream_t s) {
  const dim3 grid(a.B * a.H * ((a.L + LM_TOK - 1) / LM_TOK), 7);
  if (D == 128) hipLaunchKernelGGL((lm_premix_fwd_kernel<128>), grid, dim3(256), 0, s, a);
  else hipLaunchKernelGGL((lm_premix_fwd_kernel<64>), grid, dim3(256), 0, s, a);
  return hipGetLastError();
}

int lm_premix_rows(int B, int L) { return B * ((L + LM_TOK - 1) / LM_TOK); }

hipError_t launch_lm_premix_bwd(int D, const LmPremixBwdArgs& a, hipStream_t s) {
  const dim3 grid(a.f.B * a.f.H * ((a.f.L + LM_TOK - 1) / LM_TOK), 7);
  if (D == 128) hipLaunchKernelGGL((lm_premix_bwd_kernel<128>), grid, dim3(256), 0, s, a);
  else hipLaunchKernelGGL((lm_premix_bwd_kernel<64>), grid, dim3(256), 0, s, a);
  const int cols = 17 * a.f.H * D + 2 * a.f.H;
  hipLaunchKernelGGL(lm_reduce_kernel, dim3((cols + 63) / 64), dim3(256), 0, s, a.part, a.dparam,
                     lm_premix_rows(a.f.B, a.f.L), cols);
  return hipGetLastError();
}

template <bool BWD, bool GATED>
static hipError_t rms_launch(const LmRmsArgs& a, hipStream_t s) {
  auto go = [&](auto nq) {
    constexpr int NQ = decltype(nq)::value;
    if constexpr (BWD) {
      const int nb = lm_rms_parts(a.rows);
      hipLaunchKernelGGL((lm_rms_bwd_kernel<NQ, GATED>), dim3(nb), dim3(256), 0, s, a);
      hipLaunchKernelGGL(lm_reduce_kernel, dim3((a.C + 63) / 64), dim3(256), 0, s, a.part, a.dscale, nb, a.C);
    } else {
      hipLaunchKernelGGL((lm_rms_fwd_kernel<NQ, GATED>), dim3((a.rows + 3) / 4), dim3(256), 0, s, a);
    }
  };
  switch ((a.C + 255) / 256) {
    case 1: go(std::integral_constant<int, 1>{}); break;
    case 2: go(std::integral_constant<int, 2>{}); break;
    case 3: go(std::integral_constant<int, 3>{}); break;
    case 4: go(std::integral_constant<int, 4>{}); break;
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}
int lm_rms_parts(int rows) { return (rows + 4 * RMS_ROWS - 1) / (4 * RMS_ROWS); }
hipError_t launch_lm_rms_fwd(const LmRmsArgs& a, hipStream_t s) {
  return a.gate ? rms_launch<false, true>(a, s) : rms_launch<false, false>(a, s);
}
hipError_t launch_lm_rms_bwd(const LmRmsArgs& a, hipStream_t s) {
  return a.gate ? rms_launch<true, true>(a, s) : rms_launch<true, false>(a, s);
}
hipError_t launch_lm_swiglu(const float* gu, const float* dact, float* out, int rows, int M, hipStream_t s) {
  const dim3 grid((unsigned)(((size_t)rows * (M / 4) + 255) / 256));
  if (dact) hipLaunchKernelGGL((lm_swiglu_kernel<true>), grid, dim3(256), 0, s, gu, dact, out, rows, M);
  else hipLaunchKernelGGL((lm_swiglu_kernel<false>), grid, dim3(256), 0, s, gu, dact, out, rows, M);
  return hipGetLastError();
}
hipError_t launch_lm_columns(const LmColumnsArgs& a, bool split, hipStream_t s) {
  const dim3 grid((a.ld + 255) / 256, a.rows);
  if (split) hipLaunchKernelGGL((lm_columns_kernel<true>), grid, dim3(256), 0, s, a);
  else hipLaunchKernelGGL((lm_columns_kernel<false>), grid, dim3(256), 0, s, a);
  return hipGetLastError();
}

}  // namespace gdn2
