// Token recurrence of the GDN-2 operator for serving, on gfx950: the single-token decode step
// and the tail of the forward-only prefill (the tokens after its last full chunk), with the
// semantics of the reference's inference module (notebooks/gdn2_v031_stage2_tpu.ipynb, cell 1,
// INFERENCE_V031: _decode_body and decode_step; the per-token math is reference/ref.py:116-130).
// Per token, for every (batch, head):
//   S = reset ? 0 : state;   h = diag(e^{min(g,0)}) S;   erase_j = sum_d (b k)_d h[d][j];
//   v_new = w v - erase;     h += k v_new^T;              o_j = sum_d h[d][j] (s q)_d;
//   with a cap:  h *= min(1, tau / max(||h||_F, 1e-12))  (per head, NaN propagates);
//   h and o: NaN / +-Inf -> 0;  o stored in the output dtype, the state carried in the state
//   dtype (rounded after every token, as consecutive decode_step calls store it).
// The value columns of the state are independent, so a workgroup takes a slice of columns of one
// (batch, head) -- 32 of them, whole 128-byte lines of a state row; all D with the cap, which needs
// the head's norm -- and keeps it in registers: the state is read and written once per call.
// Element-wise, no MFMA: 2 D^2 state elements per (batch, head), plus 7 D per token.
//   one token (decode_step_kernel): memory-bound at serving batches, so a wave reads whole lines:
//     thread t owns 4 columns (j0 = 4 (t % (CW/4))) of the D/16 key rows of group t / (CW/4); the key
//     vectors go through LDS and the key sums over the 16 groups too.  B64 H16 D128 fp32: 26.6 us,
//     0.81 of the copy rate.
//   several tokens (decode_tail_kernel): bound by a token's dependent chain, so nothing on it goes
//     through memory or a barrier: a lane holds 4 columns of 4 key rows, a key sum is 4 products per
//     lane and a butterfly over the D/4 lanes of its columns, and the next tokens' operands are loaded
//     four tokens ahead.  B2 H16 D128, 56 tokens: 87 -> 40 us, B1 H6 D64, 63 tokens 83 -> 36 us
//     against the one-token form in a loop (three barriers and a round trip per token).  As a
//     one-token kernel it is slower at large batches (37 us at B64 H16 D128: 32-byte pieces of lines).
#include "gdn2_kernels.hpp"

namespace gdn2 {

// jnp.nan_to_num(x, nan=0, posinf=0, neginf=0)
__device__ __forceinline__ float finite_or_zero(float x) { return __builtin_isfinite(x) ? x : 0.f; }
__device__ __forceinline__ float wave_sum(float x) {
#pragma unroll
  for (int m = WAVE / 2; m >= 1; m >>= 1) x += __shfl_xor(x, m);
  return x;
}
// jax.nn.softplus(x) = logaddexp(x, 0) = max(x, 0) + log1p(exp(-|x|)); NaN propagates
__device__ __forceinline__ float softplus(float x) {
  return __builtin_elementwise_maximum(x, 0.f) + log1pf(expf(-fabsf(x)));
}
__device__ __forceinline__ float sigmoid(float x) { return 1.f / (1.f + expf(-x)); }

template <bool BF>
__device__ __forceinline__ float4 ld_quad(const void* p, size_t i) {
  if constexpr (BF) {
    const uint2 u = *reinterpret_cast<const uint2*>(static_cast<const uint16_t*>(p) + i);
    return make_float4(bf16_val(u.x & 0xffffu), bf16_val(u.x >> 16), bf16_val(u.y & 0xffffu), bf16_val(u.y >> 16));
  } else {
    return *reinterpret_cast<const float4*>(static_cast<const float*>(p) + i);
  }
}
template <bool BF>
__device__ __forceinline__ void st_quad(void* p, size_t i, const float4& x) {
  if constexpr (BF) {
    *reinterpret_cast<uint2*>(static_cast<uint16_t*>(p) + i) = make_uint2(bf16_pack(x.x, x.y), bf16_pack(x.z, x.w));
  } else {
    *reinterpret_cast<float4*>(static_cast<float*>(p) + i) = x;
  }
}
template <bool BF>
__device__ __forceinline__ float ld_one(const void* p, size_t i) {
  if constexpr (BF) return bf16_val(static_cast<const uint16_t*>(p)[i]);
  else return static_cast<const float*>(p)[i];
}
__device__ __forceinline__ float4 clean4(const float4& x, bool bf) {
  float4 y = make_float4(finite_or_zero(x.x), finite_or_zero(x.y), finite_or_zero(x.z), finite_or_zero(x.w));
  if (bf) y = make_float4(bf16_round(y.x), bf16_round(y.y), bf16_round(y.z), bf16_round(y.w));
  return y;
}

// A reset flag in the caller's own type (gdn2_decode_flags): no cast launches around a one-token call
__device__ __forceinline__ bool flag_set(const void* p, int type, size_t i) {
  if (type == 1) return static_cast<const int32_t*>(p)[i] > 0;
  if (type == 2) return (int32_t)static_cast<const int64_t*>(p)[i] > 0;
  return static_cast<const uint8_t*>(p)[i] != 0;
}

template <int D, int CW, bool CAP, bool IBF, bool SBF>
__global__ __launch_bounds__(CW / 4 * 16) void decode_step_kernel(DecodeArgs a) {
  constexpr int KG = 16, NQ = CW / 4, NT = NQ * KG, KPK = D / KG, NS = D / CW, NWV = (NT + WAVE - 1) / WAVE;
  static_assert(NT >= D, "the key vectors are formed by one thread per key row");
  __shared__ float4 sVec[D];          // key row d: (s q_d, k_d, b_d k_d, e^{min(g_d,0)})
  __shared__ float4 sEr[KG][NQ];      // key-group partial sums of the erase term, per column quad
  __shared__ float4 sOut[KG][NQ];     // key-group partial sums of the output
  __shared__ float sNrm[NWV];         // per-wave sums of h^2 (cap)
  const int tid = threadIdx.x, cq = tid % NQ, kg = tid / NQ, d0 = kg * KPK;
  const int bh = blockIdx.x / NS, j0 = (blockIdx.x % NS) * CW + 4 * cq;
  const int bi = bh / a.H, hi = bh - bi * a.H;
  const int l = lane_id(), wv = tid / WAVE;
  const size_t sb = (size_t)bh * D * D;

  float4 h[KPK];
#pragma unroll
  for (int i = 0; i < KPK; ++i)
    h[i] = a.state_in ? ld_quad<SBF>(a.state_in, sb + (size_t)(d0 + i) * D + j0) : make_float4(0.f, 0.f, 0.f, 0.f);

  const size_t io = (size_t)bh * a.seq_ld * D;
  // this thread's columns of w and v, issued with the key vectors' loads (one round trip)
  float4 wj = ld_quad<IBF>(a.w, io + j0);
  const float4 vj = ld_quad<IBF>(a.v, io + j0);
  if (a.reset && flag_set(a.reset, a.flag_type, bi)) {
#pragma unroll
    for (int i = 0; i < KPK; ++i) h[i] = make_float4(0.f, 0.f, 0.f, 0.f);
  }
  // the token's key vectors (threads 0 .. D-1, whole waves)
  if (tid < D) {
    float qd = ld_one<IBF>(a.q, io + tid), kd = ld_one<IBF>(a.k, io + tid);
    float bd = ld_one<IBF>(a.b, io + tid), gd = ld_one<IBF>(a.g, io + tid);
    if (a.fuse) {
      // the prologue of _decode_body (fuse_prologue): every wave forms the full l2 sums itself
      float sq = 0.f, sk = 0.f;
#pragma unroll
      for (int m = l; m < D; m += WAVE) {
        const float x = ld_one<IBF>(a.q, io + m), y = ld_one<IBF>(a.k, io + m);
        sq = fmaf(x, x, sq);
        sk = fmaf(y, y, sk);
      }
      sq = wave_sum(sq);
      sk = wave_sum(sk);
      qd *= 1.f / sqrtf(sq + 1e-6f);
      kd *= 1.f / sqrtf(sk + 1e-6f);
      bd = sigmoid(bd);
      gd = -expf(a.a_log[hi]) * softplus(gd + a.dt_bias[tid]);
    }
    sVec[tid] = make_float4(a.scale * qd, kd, bd * kd, exp_nonpos(gd));
  }
  __syncthreads();
  float4 ep = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
  for (int i = 0; i < KPK; ++i) {
    const float4 x = sVec[d0 + i];
    h[i] = scale4(h[i], x.w);
    ep = make_float4(fmaf(x.z, h[i].x, ep.x), fmaf(x.z, h[i].y, ep.y), fmaf(x.z, h[i].z, ep.z), fmaf(x.z, h[i].w, ep.w));
  }
  sEr[kg][cq] = ep;
  __syncthreads();
  float4 er = sEr[0][cq];
#pragma unroll
  for (int m = 1; m < KG; ++m) er = add4(er, sEr[m][cq]);
  if (a.fuse) wj = make_float4(sigmoid(wj.x), sigmoid(wj.y), sigmoid(wj.z), sigmoid(wj.w));
  const float4 vn = make_float4(wj.x * vj.x - er.x, wj.y * vj.y - er.y, wj.z * vj.z - er.z, wj.w * vj.w - er.w);
  float4 op = make_float4(0.f, 0.f, 0.f, 0.f);
  float np = 0.f;
#pragma unroll
  for (int i = 0; i < KPK; ++i) {
    const float4 x = sVec[d0 + i];
    h[i] = make_float4(fmaf(x.y, vn.x, h[i].x), fmaf(x.y, vn.y, h[i].y), fmaf(x.y, vn.z, h[i].z), fmaf(x.y, vn.w, h[i].w));
    op = make_float4(fmaf(h[i].x, x.x, op.x), fmaf(h[i].y, x.x, op.y), fmaf(h[i].z, x.x, op.z), fmaf(h[i].w, x.x, op.w));
    if constexpr (CAP) np = fmaf(h[i].x, h[i].x, fmaf(h[i].y, h[i].y, fmaf(h[i].z, h[i].z, fmaf(h[i].w, h[i].w, np))));
  }
  sOut[kg][cq] = op;
  if constexpr (CAP) {
    np = wave_sum(np);
    if (l == 0) sNrm[wv] = np;
  }
  __syncthreads();
  if (kg == 0) {
    float4 o = sOut[0][cq];
#pragma unroll
    for (int m = 1; m < KG; ++m) o = add4(o, sOut[m][cq]);
    o = clean4(o, false);
    if (a.out_bf16) st_quad<true>(a.o, io + j0, o);
    else st_quad<false>(a.o, io + j0, o);
  }
  if constexpr (CAP) {
    float n2 = 0.f;
#pragma unroll
    for (int m = 0; m < NWV; ++m) n2 += sNrm[m];
    const float nrm = sqrtf(n2);
    const float f = __builtin_elementwise_minimum(1.f, a.tau / __builtin_elementwise_maximum(nrm, 1e-12f));
#pragma unroll
    for (int i = 0; i < KPK; ++i) h[i] = scale4(h[i], f);
  }
#pragma unroll
  for (int i = 0; i < KPK; ++i) h[i] = clean4(h[i], SBF);
#pragma unroll
  for (int i = 0; i < KPK; ++i) st_quad<SBF>(a.state_out, sb + (size_t)(d0 + i) * D + j0, h[i]);
}

// sum over the 16 lanes of a DPP row, the same bits in every lane
template <int ROR>
__device__ __forceinline__ float row_ror(float x) {
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), 0x120 | ROR, 0xf, 0xf, true));
}
// ... or over pairs of rows (KG = 32): the row totals of rows 0 | 1 and of 2 | 3 exchanged
template <int KG>
__device__ __forceinline__ float key_sum(float x) {
  x += row_ror<8>(x);
  x += row_ror<4>(x);
  x += row_ror<2>(x);
  x += row_ror<1>(x);
  if constexpr (KG == 32) {
    // lane ^ 16 within each half of the wave
    x += __builtin_bit_cast(float, __builtin_amdgcn_ds_swizzle(__builtin_bit_cast(int, x), 0x401f));
  }
  return x;
}
template <int KG>
__device__ __forceinline__ float4 key_sum4(const float4& x) {
  return make_float4(key_sum<KG>(x.x), key_sum<KG>(x.y), key_sum<KG>(x.z), key_sum<KG>(x.w));
}

// One token's operands of a lane: its key rows' q, k, b, g (quads) and its columns' w, v
template <int NK>
struct TokenOps {
  float4 q[NK], k[NK], b[NK], g[NK], w, v;
};

// The tokens' operands are loaded PF tokens ahead into a ring of register sets (a token takes less
// than a round trip to HBM).
template <int D, int NWV, bool CAP, bool IBF, bool SBF>
__global__ __launch_bounds__(NWV * WAVE) void decode_tail_kernel(DecodeArgs a) {
  constexpr int KPK = 4, KG = D / KPK, NK = KPK / 4, CWV = 4 * (WAVE / KG), NS = D / (CWV * NWV);
  __shared__ float sNrm[2][NWV];      // per-wave sums of h^2 by token parity (cap)
  const int l = lane_id(), wv = wave_id(), d0 = (l % KG) * KPK;
  const int bh = blockIdx.x / NS, j0 = ((blockIdx.x % NS) * NWV + wv) * CWV + 4 * (l / KG);
  const int bi = bh / a.H, hi = bh - bi * a.H;
  const size_t sb = (size_t)bh * D * D;

  float4 h[KPK];
#pragma unroll
  for (int i = 0; i < KPK; ++i)
    h[i] = a.state_in ? ld_quad<SBF>(a.state_in, sb + (size_t)(d0 + i) * D + j0) : make_float4(0.f, 0.f, 0.f, 0.f);
  float alog = 0.f;
  float4 dtb[NK];
#pragma unroll
  for (int n = 0; n < NK; ++n) dtb[n] = make_float4(0.f, 0.f, 0.f, 0.f);
  if (a.fuse) {
    alog = -expf(a.a_log[hi]);
#pragma unroll
    for (int n = 0; n < NK; ++n)
      dtb[n] = make_float4(a.dt_bias[d0 + 4 * n], a.dt_bias[d0 + 4 * n + 1], a.dt_bias[d0 + 4 * n + 2], a.dt_bias[d0 + 4 * n + 3]);
  }
  auto load = [&](TokenOps<NK>& x, int t) {
    const size_t io = ((size_t)bh * a.seq_ld + t) * D;
#pragma unroll
    for (int n = 0; n < NK; ++n) {
      x.q[n] = ld_quad<IBF>(a.q, io + d0 + 4 * n);
      x.k[n] = ld_quad<IBF>(a.k, io + d0 + 4 * n);
      x.b[n] = ld_quad<IBF>(a.b, io + d0 + 4 * n);
      x.g[n] = ld_quad<IBF>(a.g, io + d0 + 4 * n);
    }
    x.w = ld_quad<IBF>(a.w, io + j0);
    x.v = ld_quad<IBF>(a.v, io + j0);
  };
  auto token = [&](const TokenOps<NK>& op, int t) __attribute__((always_inline)) {
    float sq[KPK], kk[KPK], bk[KPK], eg[KPK];
#pragma unroll
    for (int n = 0; n < NK; ++n) {
      const float4 q = op.q[n], k = op.k[n], b = op.b[n], g = op.g[n];
      const float qa[4] = {q.x, q.y, q.z, q.w}, ka[4] = {k.x, k.y, k.z, k.w}, ba[4] = {b.x, b.y, b.z, b.w};
      const float ga[4] = {g.x, g.y, g.z, g.w};
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        sq[4 * n + e] = qa[e];
        kk[4 * n + e] = ka[e];
        bk[4 * n + e] = ba[e];
        eg[4 * n + e] = ga[e];
      }
    }
    float4 wj = op.w;
    const float4 vj = op.v;
    if (a.fuse) {
      // the prologue of _decode_body (fuse_prologue)
      float nq = 0.f, nk = 0.f;
#pragma unroll
      for (int i = 0; i < KPK; ++i) {
        nq = fmaf(sq[i], sq[i], nq);
        nk = fmaf(kk[i], kk[i], nk);
      }
      const float rq = 1.f / sqrtf(key_sum<KG>(nq) + 1e-6f), rk = 1.f / sqrtf(key_sum<KG>(nk) + 1e-6f);
#pragma unroll
      for (int n = 0; n < NK; ++n) {
        const float da[4] = {dtb[n].x, dtb[n].y, dtb[n].z, dtb[n].w};
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int i = 4 * n + e;
          sq[i] *= rq;
          kk[i] *= rk;
          bk[i] = sigmoid(bk[i]);
          eg[i] = alog * softplus(eg[i] + da[e]);
        }
      }
      wj = make_float4(sigmoid(wj.x), sigmoid(wj.y), sigmoid(wj.z), sigmoid(wj.w));
    }
    if (a.reset && flag_set(a.reset, a.flag_type, (size_t)bi * a.n_tok + t)) {
#pragma unroll
      for (int i = 0; i < KPK; ++i) h[i] = make_float4(0.f, 0.f, 0.f, 0.f);
    }
    float4 ep = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
    for (int i = 0; i < KPK; ++i) {
      sq[i] = a.scale * sq[i];
      const float bkv = bk[i] * kk[i];
      h[i] = scale4(h[i], exp_nonpos(eg[i]));
      ep = make_float4(fmaf(bkv, h[i].x, ep.x), fmaf(bkv, h[i].y, ep.y), fmaf(bkv, h[i].z, ep.z), fmaf(bkv, h[i].w, ep.w));
    }
    const float4 er = key_sum4<KG>(ep);
    const float4 vn = make_float4(wj.x * vj.x - er.x, wj.y * vj.y - er.y, wj.z * vj.z - er.z, wj.w * vj.w - er.w);
    float4 o = make_float4(0.f, 0.f, 0.f, 0.f);
    float np = 0.f;
#pragma unroll
    for (int i = 0; i < KPK; ++i) {
      const float ki = kk[i], qi = sq[i];
      h[i] = make_float4(fmaf(ki, vn.x, h[i].x), fmaf(ki, vn.y, h[i].y), fmaf(ki, vn.z, h[i].z), fmaf(ki, vn.w, h[i].w));
      o = make_float4(fmaf(h[i].x, qi, o.x), fmaf(h[i].y, qi, o.y), fmaf(h[i].z, qi, o.z), fmaf(h[i].w, qi, o.w));
      if constexpr (CAP) np = fmaf(h[i].x, h[i].x, fmaf(h[i].y, h[i].y, fmaf(h[i].z, h[i].z, fmaf(h[i].w, h[i].w, np))));
    }
    o = clean4(key_sum4<KG>(o), false);
    if (l % KG == 0) {
      const size_t oo = ((size_t)bh * a.seq_ld + t) * D + j0;
      if (a.out_bf16) st_quad<true>(a.o, oo, o);
      else st_quad<false>(a.o, oo, o);
    }
    if constexpr (CAP) {
      np = wave_sum(np);
      if (l == 0) sNrm[t & 1][wv] = np;
      __syncthreads();                  // (the other parity's values were read before this barrier)
      float n2 = 0.f;
#pragma unroll
      for (int m = 0; m < NWV; ++m) n2 += sNrm[t & 1][m];
      const float nrm = sqrtf(n2);
      const float f = __builtin_elementwise_minimum(1.f, a.tau / __builtin_elementwise_maximum(nrm, 1e-12f));
#pragma unroll
      for (int i = 0; i < KPK; ++i) h[i] = scale4(h[i], f);
    }
#pragma unroll
    for (int i = 0; i < KPK; ++i) h[i] = clean4(h[i], SBF);
  };
  constexpr int PF = CAP ? 1 : 4;             // (sixteen waves with the cap: no registers for more)
  TokenOps<NK> op[PF];
  const int last = a.n_tok - 1;               // loads past the last token repeat it
#pragma unroll
  for (int i = 0; i < PF; ++i) load(op[i], min(i, last));
  int t = 0;
  for (; t + PF <= a.n_tok; t += PF) {
#pragma unroll
    for (int i = 0; i < PF; ++i) {
      token(op[i], t + i);
      load(op[i], min(t + i + PF, last));
    }
  }
#pragma unroll
  for (int i = 0; i < PF - 1; ++i)
    if (t + i < a.n_tok) token(op[i], t + i);
#pragma unroll
  for (int i = 0; i < KPK; ++i) st_quad<SBF>(a.state_out, sb + (size_t)(d0 + i) * D + j0, h[i]);
}

template <int D, bool CAP, bool IBF, bool SBF>
void launch_decode_t(const DecodeArgs& a, int n_bh, hipStream_t s) {
  if (a.n_tok > 1) {
    constexpr int CWV = 1024 / D, NWV = CAP ? D / CWV : 32 / CWV;       // columns of a wave, waves
    hipLaunchKernelGGL((decode_tail_kernel<D, NWV, CAP, IBF, SBF>), dim3(n_bh * (D / (CWV * NWV))), dim3(NWV * WAVE), 0, s, a);
  } else {
    constexpr int CW = CAP ? D : 32;
    hipLaunchKernelGGL((decode_step_kernel<D, CW, CAP, IBF, SBF>), dim3(n_bh * (D / CW)), dim3(CW / 4 * 16), 0, s, a);
  }
}

template <int D, bool CAP>
void launch_decode_d(const DecodeArgs& a, int n_bh, hipStream_t s) {
  if (a.in_bf16) {
    if (a.state_bf16) launch_decode_t<D, CAP, true, true>(a, n_bh, s);
    else launch_decode_t<D, CAP, true, false>(a, n_bh, s);
  } else {
    if (a.state_bf16) launch_decode_t<D, CAP, false, true>(a, n_bh, s);
    else launch_decode_t<D, CAP, false, false>(a, n_bh, s);
  }
}

hipError_t launch_decode(int D, const DecodeArgs& a, int n_bh, hipStream_t s) {
  if (D == 128) {
    if (a.cap) launch_decode_d<128, true>(a, n_bh, s);
    else launch_decode_d<128, false>(a, n_bh, s);
  } else {
    if (a.cap) launch_decode_d<64, true>(a, n_bh, s);
    else launch_decode_d<64, false>(a, n_bh, s);
  }
  return hipGetLastError();
}

}  // namespace gdn2
