// Backward pass of the GatedDeltaNet layer prefill (omx_gdn_prefill_bwd): the parts
// around the chunked rule's backward (gdn_bwd.hip).
//
// Forward (deltanet.py:243-293, between the projections and out_proj):
//   u = conv(x, w) (causal depthwise, K = 4, bf16), y = silu(u) (bf16), y = [q | k | v];
//   beta = sigmoid(b) (bf16), g = -exp(A_log) softplus(a + dt_bias);
//   o = chunk_gated_delta_rule(q, k, v, g, beta) (fp32);
//   out = w_n * o * rsqrt(mean(o^2) + eps) * silu(z).
// Kernels here, in the order the backward runs them:
//   fwd_pieces_kernel       y from x and w, as the forward's prep computes it, into
//                           separate q, k, v rows for the rule's backward, and g and beta
//                           per (token, value head);
//   norm_bwd_kernel         the gated RMSNorm's adjoint: do, dz and per-workgroup partial
//                           sums of dw_n (o comes from the rule's recompute scan);
//   tail_bwd_kernel         da, db and per-workgroup partial sums of dA_log, d dt_bias;
//                           du = dy silu'(u), dx (the transposed conv) and per-token-block
//                           partial sums of dw;
//   reduce_kernel           all partial sums in a fixed order (deterministic results).
// Dtype casts are differentiated as the identity, as autodiff does.
#include "gdn_chunk.h"
#include "gdn_kernels.h"

namespace omx {

namespace {

constexpr int NT = 256;

// Sequence bounds of token t: packed sequences (cu_seqlens, clamped by seq_range) or batch
// rows of length T.
__device__ __forceinline__ void token_seq(const int32_t* cu, int N, int T, long long t,
                                          long long& s0, long long& s1) {
  if (cu) {
    int lo = 0, hi = N;  // the last n with cu[n] <= t
    while (hi - lo > 1) {
      const int mid = (lo + hi) >> 1;
      if (cu[mid] <= t) lo = mid;
      else hi = mid;
    }
    seq_range(cu, lo, T, s0, s1);
  } else {
    s0 = (t / T) * T;
    s1 = s0 + T;
  }
}

// conv weights of channels c0 .. c0+7 cast to bf16 (deltanet.py:243): wt[e][d] multiplies
// the input d tokens back (tap K-1-d); K = 4
__device__ __forceinline__ void conv_w8(const float* w, int c0, float (*wt)[4]) {
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    const float4 x = *(const float4*)(w + (size_t)(c0 + e) * 4);
    wt[e][0] = round_bf(x.w);
    wt[e][1] = round_bf(x.z);
    wt[e][2] = round_bf(x.y);
    wt[e][3] = round_bf(x.x);
  }
}

__device__ __forceinline__ void load8(const bf16_t* p, float* x) {
  const u32x4 w = *(const u32x4*)p;
  unpack8<false>(&w, x);
}

__device__ __forceinline__ void zero8(float* x) {
#pragma unroll
  for (int e = 0; e < 8; ++e) x[e] = 0.f;
}

// the forward's conv pre-activation, computed and rounded to bf16 as there (the inputs
// and the weights wt are bf16 values, so the pairs pack exactly)
__device__ __forceinline__ float conv_u(const float* wt, float x0, float x1, float x2, float x3) {
  return round_bf(dot4_bf16(pack_bf16(wt[0], wt[1]), pack_bf16(wt[2], wt[3]), pack_bf16(x0, x1),
                            pack_bf16(x2, x3)));
}

// d silu(u) / du
__device__ __forceinline__ float silu_grad(float u) {
  // sigmoid from the hardware exp2 and reciprocal (about 2 ulp in fp32)
  const float s = __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(u * -1.4426950408889634f));
  return s * (1.0f + u * (1.0f - s));
}

// ---------------------------------------------------------------------------- forward pieces

// One thread per (16-token block, 8-channel group): the weights and the last three inputs
// stay in registers while it streams down the block's tokens (every input read once plus a
// 3-token halo).
constexpr int kConvFwdTB = 16;

__device__ __forceinline__ void conv_silu_split(const LayerBwdParams& p, long long idx) {
  const int G = p.conv_dim / 8;
  const long long nblk = (p.tokens + kConvFwdTB - 1) / kConvFwdTB;
  if (idx >= nblk * G) return;
  const long long tb = (idx / G) * kConvFwdTB;
  const long long te = tb + kConvFwdTB < p.tokens ? tb + kConvFwdTB : p.tokens;
  const int c0 = 8 * (int)(idx % G);
  float wt[8][4];
  conv_w8(p.conv_w, c0, wt);
  const int kd = p.Hk * p.dk;
  bf16_t* dst;
  long long ld;
  if (c0 < kd) { dst = p.q + c0; ld = kd; }
  else if (c0 < 2 * kd) { dst = p.k + (c0 - kd); ld = kd; }
  else { dst = p.v + (c0 - 2 * kd); ld = (long long)p.Hv * p.dv; }
  long long s0, s1;
  token_seq(p.cu_seqlens, p.N, p.T, tb, s0, s1);
  float xs[4][8];  // inputs d tokens back
#pragma unroll
  for (int d = 1; d < 4; ++d) {
    if (tb - d >= s0) load8(p.x + (tb - d) * p.conv_dim + c0, xs[d]);
    else zero8(xs[d]);
  }
  // every row of the block is loaded before the first store: one memory round trip per
  // thread.  The loads are unconditional (rows past te reload row te - 1 and are never
  // used), so the compiler can count them and a wait for row m does not also wait for the
  // stores issued before it (the memory counter retires in order).
  u32x4 raw[kConvFwdTB];
#pragma unroll
  for (int m = 0; m < kConvFwdTB; ++m)
    raw[m] = *(const u32x4*)(p.x + (tb + m < te ? tb + m : te - 1) * p.conv_dim + c0);
#pragma unroll
  for (int m = 0; m < kConvFwdTB; ++m) {
    const long long t = tb + m;
    if (t >= te) break;
    if (t >= s1) {  // a new sequence starts at t: no history
      token_seq(p.cu_seqlens, p.N, p.T, t, s0, s1);
#pragma unroll
      for (int d = 1; d < 4; ++d) zero8(xs[d]);
      __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0): the lookup's loads end here
    }
    unpack8<false>(&raw[m], xs[0]);
    float y[8];
#pragma unroll
    for (int e = 0; e < 8; ++e)
      y[e] = round_bf(silu_fast(conv_u(wt[e], xs[0][e], xs[1][e], xs[2][e], xs[3][e])));
    *(u32x4*)(dst + t * ld) = pack8(y);
#pragma unroll
    for (int d = 3; d > 0; --d)
#pragma unroll
      for (int e = 0; e < 8; ++e) xs[d][e] = xs[d - 1][e];
  }
}

// one thread per (token, value head): g and beta as the forward's prep forms them
__device__ __forceinline__ void gates(const LayerBwdParams& p, long long idx) {
  if (idx >= p.tokens * p.Hv) return;
  const int h = (int)(idx % p.Hv);
  p.g[idx] = -expf(p.A_log[h]) * softplusf_(bf2f(p.a[idx]) + p.dt_bias[h]);
  p.beta[idx] = round_bf(sigmoidf_(bf2f(p.b[idx])));
}

// The first gate_blocks workgroups form the gates, the rest the conv: one launch, so the
// gates cost no launch and drain of their own (4.8 us at 3,001 tokens).
__global__ __launch_bounds__(NT) void fwd_pieces_kernel(LayerBwdParams p, unsigned gate_blocks) {
  if (blockIdx.x < gate_blocks) gates(p, (long long)blockIdx.x * NT + threadIdx.x);
  else conv_silu_split(p, (long long)(blockIdx.x - gate_blocks) * NT + threadIdx.x);
}

// ---------------------------------------------------------------------------- gated RMSNorm

// Persistent: each wavefront walks (token, value head) rows of dv <= 128 (lane l: columns
// 2l and 2l + 1, so o and dO move 8 bytes and z, dout, dz 4 bytes per lane).
// n = o r, r = (mean(o^2) + eps)^-1/2, out = w n silu(z):
//   dn = dout w silu(z), dz = dout w n silu'(z), dw = sum dout n silu(z),
//   do = r (dn - n mean(dn n)).
// sigmoid(z) comes from the hardware exp2 and reciprocal (about 2 ulp in fp32).
__global__ __launch_bounds__(NT) void norm_bwd_kernel(LayerBwdParams p) {
  __shared__ float sdw[NT / 64][128];
  const int l = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int dv = p.dv, c = 2 * l;
  const bool in = c < dv;  // dv is even
  const long long rows = p.tokens * p.Hv;
  const long long nw = (long long)gridDim.x * (NT / 64);
  float w[2], dw[2] = {0.f, 0.f};
#pragma unroll
  for (int e = 0; e < 2; ++e) w[e] = in ? p.norm_w[c + e] : 0.f;
  for (long long r = (long long)blockIdx.x * (NT / 64) + wave; r < rows; r += nw) {
    float o[2] = {0.f, 0.f}, z[2] = {0.f, 0.f}, go[2] = {0.f, 0.f};
    if (in) {
      const float2 ov = *(const float2*)(p.o + r * dv + c);
      const uint32_t zv = *(const uint32_t*)(p.z + r * dv + c);
      const uint32_t gv = *(const uint32_t*)(p.dout + r * dv + c);
      o[0] = ov.x; o[1] = ov.y;
      z[0] = __uint_as_float(zv << 16); z[1] = __uint_as_float(zv & 0xffff0000u);
      go[0] = __uint_as_float(gv << 16); go[1] = __uint_as_float(gv & 0xffff0000u);
    }
    float ss = o[0] * o[0] + o[1] * o[1];
#pragma unroll
    for (int s = 1; s < 64; s <<= 1) ss += __shfl_xor(ss, s);
    const float rr = rsqrtf(ss / (float)p.dv_mean + p.eps);
    float n[2], dn[2], dzv[2], dnn = 0.f;
#pragma unroll
    for (int e = 0; e < 2; ++e) {
      n[e] = o[e] * rr;
      const float sg = __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(z[e] * -1.4426950408889634f));
      const float sz = z[e] * sg;                       // silu(z)
      const float sgrad = sg * (1.0f + z[e] * (1.0f - sg));  // silu'(z)
      dn[e] = go[e] * w[e] * sz;
      dnn += dn[e] * n[e];
      dw[e] += go[e] * n[e] * sz;
      dzv[e] = go[e] * w[e] * n[e] * sgrad;
    }
#pragma unroll
    for (int s = 1; s < 64; s <<= 1) dnn += __shfl_xor(dnn, s);
    const float m = dnn / (float)p.dv_mean;
    if (in) {
      *(uint32_t*)(p.dz + r * dv + c) = pack_bf16(dzv[0], dzv[1]);
      *(float2*)(p.dO + r * dv + c) = float2{rr * (dn[0] - n[0] * m), rr * (dn[1] - n[1] * m)};
    }
  }
#pragma unroll
  for (int e = 0; e < 2; ++e)
    if (in) sdw[wave][c + e] = dw[e];
  __syncthreads();
  if (threadIdx.x < dv) {
    float s = 0.f;
#pragma unroll
    for (int v = 0; v < NT / 64; ++v) s += sdw[v][threadIdx.x];
    p.part_norm[(size_t)blockIdx.x * dv + threadIdx.x] = s;
  }
}

// ---------------------------------------------------------------------------- gates

// Workgroup w of the gate part takes a contiguous token range; thread (j, h) = (tid / Hv, tid % Hv) walks its
// tokens j, j + R, ... (R = 256 / Hv) for value head h.
//   da = dg A sigmoid(a + dt_bias), A = -exp(A_log); db = dbeta sigmoid(b)(1 - sigmoid(b));
//   dA_log = sum dg g, d dt_bias = sum da.
__device__ __forceinline__ void gates_bwd(const LayerBwdParams& p, long long blk, long long per,
                                          float (*sacc)[2]) {
  const int Hv = p.Hv, tid = threadIdx.x;
  const int R = NT / Hv;
  const int h = tid % Hv, j = tid / Hv;
  float sA = 0.f, sdt = 0.f;
  if (j < R) {
    const float A = -expf(p.A_log[h]), dtb = p.dt_bias[h];
    const long long t0 = blk * per;
    const long long t1 = t0 + per < p.tokens ? t0 + per : p.tokens;
    for (long long t = t0 + j; t < t1; t += R) {
      const long long i = t * Hv + h;
      const float dgv = p.dg[i];
      const float da = dgv * A * sigmoidf_(bf2f(p.a[i]) + dtb);
      const float sb = sigmoidf_(bf2f(p.b[i]));
      p.da[i] = f2bf(da);
      p.db[i] = f2bf(p.dbeta[i] * sb * (1.f - sb));
      sA += dgv * p.g[i];
      sdt += da;
    }
  }
  sacc[tid][0] = sA;
  sacc[tid][1] = sdt;
  __syncthreads();
  if (tid < Hv) {
    float a0 = 0.f, a1 = 0.f;
    for (int jj = 0; jj < R; ++jj) {
      a0 += sacc[jj * Hv + tid][0];
      a1 += sacc[jj * Hv + tid][1];
    }
    p.part_gates[(size_t)blk * 2 * Hv + tid] = a0;
    p.part_gates[(size_t)blk * 2 * Hv + Hv + tid] = a1;
  }
}

// ---------------------------------------------------------------------------- conv + SiLU

// One workgroup per (64 tokens, 256 channels): wavefront w takes tokens 16w .. 16w + 15 of
// the block, a lane 4 channels.  du = dy silu'(u) with u recomputed;
//   dx[s] = sum_d wt[d] du[s + d], dwt[d] = sum_t du[t] x[t - d],
// both over the pairs (t, d) whose token t - d lies in t's sequence.  Token t's du enters
// dx[t - d], so the wavefront also forms du of the three tokens after its own.
//
// Every row it needs (22 of x, 19 of dy) is loaded before the first use, and the 4 x 256
// channels of a workgroup make 1,500 workgroups of 3,001 tokens x 8,192 channels: with one
// thread walking 64 tokens with a one-row prefetch the kernel waited for one row after the
// other (188 workgroups, 61 us there, and 21 us for the gates in a launch of their own; now
// 40 us for both, 147 MB at 3.7 TB/s).  The four wavefronts' dwt are summed in LDS, so the
// partial sums stay one per 64 tokens.
constexpr int kConvTB = 64;  // tokens per workgroup
constexpr int kConvSB = 16;  // tokens per wavefront

__device__ __forceinline__ void conv_bwd(const LayerBwdParams& p, long long bid, float (*sdw)[64][16]) {
  const int nchg = (p.conv_dim + 255) / 256;
  const long long blk = bid / nchg;
  const int l = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int cg = 256 * (int)(bid % nchg), c0 = cg + 4 * l;
  const bool in = c0 < p.conv_dim;
  const int cc = in ? c0 : p.conv_dim - 4;  // lanes past the channels load the last ones
  const long long tb = blk * kConvTB + wave * kConvSB;
  float dwt[4][4];  // [channel][d]
#pragma unroll
  for (int e = 0; e < 4; ++e)
#pragma unroll
    for (int d = 0; d < 4; ++d) dwt[e][d] = 0.f;
  if (tb < p.tokens) {  // uniform
    const int kd = p.Hk * p.dk;
    const long long vd = (long long)p.Hv * p.dv;
    const bf16_t* dys;
    long long dy_ld;
    if (cc < kd) { dys = p.grad_q + cc; dy_ld = kd; }
    else if (cc < 2 * kd) { dys = p.grad_k + (cc - kd); dy_ld = kd; }
    else { dys = p.grad_v + (cc - 2 * kd); dy_ld = vd; }
    const long long last = p.tokens - 1;
    // rows outside the tokens reload one inside; the masks below leave them out
    u32x2 xr[kConvSB + 6], dyr[kConvSB + 3];
#pragma unroll
    for (int k = 0; k < kConvSB + 6; ++k) {
      long long t = tb - 3 + k;
      t = t < 0 ? 0 : (t > last ? last : t);
      xr[k] = *(const u32x2*)(p.x + t * p.conv_dim + cc);
    }
#pragma unroll
    for (int k = 0; k < kConvSB + 3; ++k) {
      const long long t = tb + k < last ? tb + k : last;
      dyr[k] = *(const u32x2*)(dys + t * dy_ld);
    }
    float wt[4][4];
    uint32_t w01[4], w23[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const float4 w = *(const float4*)(p.conv_w + (size_t)(cc + e) * 4);
      w01[e] = pack_bf16(w.w, w.z);  // the forward's bf16 weights; wt[e][d]: d tokens back
      w23[e] = pack_bf16(w.y, w.x);
      wt[e][0] = __uint_as_float(w01[e] << 16);
      wt[e][1] = __uint_as_float(w01[e] & 0xffff0000u);
      wt[e][2] = __uint_as_float(w23[e] << 16);
      wt[e][3] = __uint_as_float(w23[e] & 0xffff0000u);
    }
    // bit k of back[d]: token tb + k - d lies in token tb + k's sequence.  A sequence that
    // starts at token b clears bits b - tb .. b - tb + d - 1 of back[d].
    unsigned back[4];
#pragma unroll
    for (int d = 0; d < 4; ++d) back[d] = 0xffffffffu;
    auto start_at = [&](long long b) {
      const int k = (int)(b - tb);  // -2 .. kConvSB + 2
#pragma unroll
      for (int d = 1; d < 4; ++d)
#pragma unroll
        for (int m = 0; m < d; ++m)
          if (k + m >= 0) back[d] &= ~(1u << (k + m));
    };
    // (starts at or past the last token cut nothing: rows of offsets are often filled up to a
    // fixed count with empty sequences there)
    const long long t2 = tb > 2 ? tb - 2 : 0;
    const long long tend = tb + kConvSB + 3 < p.tokens ? tb + kConvSB + 3 : p.tokens;
    if (p.cu_seqlens) {
      int lo = 0, hi = p.N;  // the last sequence with cu[n] <= t2
      while (hi - lo > 1) {
        const int mid = (lo + hi) >> 1;
        if (p.cu_seqlens[mid] <= t2) lo = mid;
        else hi = mid;
      }
      for (int n = lo; n < p.N; ++n) {
        const long long b = p.cu_seqlens[n];
        if (b >= tend) break;
        if (b >= t2) start_at(b);
      }
    } else {
      for (long long b = (t2 + p.T - 1) / p.T * p.T; b < tend; b += p.T) start_at(b);
    }
    // the rows this wavefront owns (rows past the tokens and lanes past the channels are
    // outside the range: dropped, no branch)
    const long long rows = p.tokens - tb < kConvSB ? p.tokens - tb : kConvSB;
    const auto dxr = buf_rsrc(p.dx + tb * p.conv_dim, 2u * (unsigned)(rows * p.conv_dim));
    float xf[4][4];  // [d][channel]: x[t - d]
#pragma unroll
    for (int d = 1; d < 4; ++d)
#pragma unroll
      for (int e = 0; e < 4; ++e) xf[d][e] = __uint_as_float(e & 1 ? xr[3 - d][e >> 1] & 0xffff0000u : xr[3 - d][e >> 1] << 16);
    float dx[4][4];  // [d][channel]: dx[t - d] so far
#pragma unroll
    for (int d = 0; d < 4; ++d)
#pragma unroll
      for (int e = 0; e < 4; ++e) dx[d][e] = 0.f;
#pragma unroll
    for (int k = 0; k < kConvSB + 3; ++k) {
      if (tb + k < p.tokens) {  // uniform
        u32x2 x1 = xr[k + 2], x2 = xr[k + 1], x3 = xr[k];
        const u32x2 x0 = xr[k + 3];
        const u32x2 zero = {0u, 0u};
        if (!(back[1] >> k & 1)) x1 = zero;
        if (!(back[2] >> k & 1)) x2 = zero;
        if (!(back[3] >> k & 1)) x3 = zero;
        float du[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const unsigned sel = e & 1 ? 0x07060302u : 0x05040100u;
          const float u = round_bf(dot4_bf16(w01[e], w23[e], __builtin_amdgcn_perm(x1[e >> 1], x0[e >> 1], sel),
                                             __builtin_amdgcn_perm(x3[e >> 1], x2[e >> 1], sel)));
          xf[0][e] = __uint_as_float(e & 1 ? x0[e >> 1] & 0xffff0000u : x0[e >> 1] << 16);
          du[e] = __uint_as_float(e & 1 ? dyr[k][e >> 1] & 0xffff0000u : dyr[k][e >> 1] << 16) * silu_grad(u);
        }
#pragma unroll
        for (int d = 0; d < 4; ++d) {
          if (back[d] >> k & 1) {  // uniform
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              dx[d][e] += wt[e][d] * du[e];
              if (k < kConvSB) dwt[e][d] += du[e] * xf[d][e];
            }
          }
        }
      }
      if (k >= 3)
        __builtin_amdgcn_raw_buffer_store_b64(u32x2{pack_bf16(dx[3][0], dx[3][1]), pack_bf16(dx[3][2], dx[3][3])}, dxr,
                                              in ? 2u * (unsigned)((k - 3) * p.conv_dim + c0) : kDropOffset, 0, 0);
#pragma unroll
      for (int d = 3; d > 0; --d)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          dx[d][e] = dx[d - 1][e];
          xf[d][e] = xf[d - 1][e];
        }
#pragma unroll
      for (int e = 0; e < 4; ++e) dx[0][e] = 0.f;
    }
  }
  // dw in [c][tap] order (tap = 3 - d), the wavefronts' sums in order
#pragma unroll
  for (int e = 0; e < 4; ++e)
    *(float4*)&sdw[wave][l][4 * e] = float4{dwt[e][3], dwt[e][2], dwt[e][1], dwt[e][0]};
  __syncthreads();
  const int c = cg + (int)threadIdx.x;
  if (c < p.conv_dim) {
    float4 t = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int w = 0; w < kConvTB / kConvSB; ++w) {
      const float4 v = *(const float4*)&sdw[w][threadIdx.x >> 2][4 * (threadIdx.x & 3)];
      t = float4{t.x + v.x, t.y + v.y, t.z + v.z, t.w + v.w};
    }
    *(float4*)(p.part_conv + ((size_t)blk * p.conv_dim + c) * 4) = t;
  }
}

// The first gate_blocks workgroups take the gates, the rest the conv (one launch for both)
__global__ __launch_bounds__(NT) void tail_bwd_kernel(LayerBwdParams p, unsigned gate_blocks, long long per) {
  __shared__ __align__(16) float sdw[kConvTB / kConvSB][64][16];
  if (blockIdx.x < gate_blocks) gates_bwd(p, blockIdx.x, per, (float (*)[2])sdw);
  else conv_bwd(p, blockIdx.x - gate_blocks, sdw);
}

// out[c] = sum over rows r of part[r * stride + c], c < ncols: COLS columns per workgroup
// and NT / COLS row groups (rows r = rg mod NT/COLS), each summing its rows into sixteen
// accumulators, so that sixteen loads are in flight (the norm's 4,096 rows bound the launch:
// 20.6 us with four); the partial sums are combined in a fixed order, so the result does not
// depend on timing.
struct ReduceJob {
  const float* part;
  float* out;
  long long nrows;
  int stride, ncols;
  unsigned blocks;  // workgroups of this job
};
struct ReduceJobs {
  ReduceJob j[4];
};

template <int COLS>
__device__ __forceinline__ void col_reduce(const ReduceJob& q, unsigned blk, float* s_part) {
  constexpr int RG = NT / COLS;
  const int cl = threadIdx.x % COLS, rg = threadIdx.x / COLS;
  const int c = (int)blk * COLS + cl;
  constexpr int U = 16;
  float acc[U];
#pragma unroll
  for (int u = 0; u < U; ++u) acc[u] = 0.f;
  if (c < q.ncols) {
    long long r = rg;
    for (; r + (U - 1) * RG < q.nrows; r += U * RG) {
#pragma unroll
      for (int u = 0; u < U; ++u) acc[u] += q.part[(r + u * RG) * q.stride + c];
    }
    for (; r + 3 * RG < q.nrows; r += 4 * RG) {
#pragma unroll
      for (int u = 0; u < 4; ++u) acc[u] += q.part[(r + u * RG) * q.stride + c];
    }
    for (; r < q.nrows; r += RG) acc[0] += q.part[r * q.stride + c];
  }
#pragma unroll
  for (int w = U / 2; w > 0; w >>= 1)
#pragma unroll
    for (int u = 0; u < w; ++u) acc[u] += acc[u + w];
  s_part[threadIdx.x] = acc[0];
  __syncthreads();
  if (rg == 0 && c < q.ncols) {
    float t = 0.f;
    for (int g = 0; g < RG; ++g) t += s_part[g * COLS + cl];
    q.out[c] = t;
  }
}

// narrow column groups (more row groups) for the few-column reductions
constexpr int kReduceNarrow = 2048;

// All four parameter gradients in one launch (each launch and drain of its own cost about
// 4.7 us at 3,001 tokens)
__global__ __launch_bounds__(NT) void reduce_kernel(ReduceJobs jobs) {
  __shared__ float s_part[NT];
  unsigned b = blockIdx.x;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const ReduceJob& q = jobs.j[i];
    if (b < q.blocks) {  // uniform
      if (q.ncols <= kReduceNarrow) col_reduce<8>(q, b, s_part);
      else col_reduce<32>(q, b, s_part);
      return;
    }
    b -= q.blocks;
  }
}

ReduceJob reduce_job(const float* part, long long nrows, int stride, int ncols, float* out) {
  const int cols = ncols <= kReduceNarrow ? 8 : 32;
  return ReduceJob{part, out, nrows, stride, ncols, (unsigned)((ncols + cols - 1) / cols)};
}

}  // namespace

int layer_bwd_norm_blocks() { return 4096; }

long long layer_bwd_conv_blocks(long long tokens) { return (tokens + kConvTB - 1) / kConvTB; }

// about four tokens per thread at 32 value heads; at 256 tokens per workgroup the gates of
// 3,001 tokens ran on 12 workgroups (21 us)
int layer_bwd_gate_blocks(long long tokens) {
  const long long b = (tokens + 31) / 32;
  return (int)(b < 1024 ? (b < 1 ? 1 : b) : 1024);
}

hipError_t launch_layer_fwd_pieces(const LayerBwdParams& p, hipStream_t stream) {
  const long long n1 = (p.tokens + kConvFwdTB - 1) / kConvFwdTB * (p.conv_dim / 8);
  if (n1 > 0) {
    const unsigned gb = (unsigned)((p.tokens * p.Hv + NT - 1) / NT);
    hipLaunchKernelGGL(fwd_pieces_kernel, dim3(gb + (unsigned)((n1 + NT - 1) / NT)), dim3(NT), 0, stream, p, gb);
  }
  return hipGetLastError();
}

hipError_t launch_layer_norm_bwd(const LayerBwdParams& p, hipStream_t stream) {
  hipLaunchKernelGGL(norm_bwd_kernel, dim3(layer_bwd_norm_blocks()), dim3(NT), 0, stream, p);
  return hipGetLastError();
}

hipError_t launch_layer_tail_bwd(const LayerBwdParams& p, hipStream_t stream) {
  const int gb = layer_bwd_gate_blocks(p.tokens);
  const long long per = (p.tokens + gb - 1) / gb;
  const long long nblk = layer_bwd_conv_blocks(p.tokens);
  const unsigned cb = (unsigned)(nblk * ((p.conv_dim + 255) / 256));
  hipLaunchKernelGGL(tail_bwd_kernel, dim3((unsigned)gb + cb), dim3(NT), 0, stream, p, (unsigned)gb, per);
  const ReduceJobs jobs{{reduce_job(p.part_conv, nblk, p.conv_dim * 4, p.conv_dim * 4, p.d_conv_w),
                         reduce_job(p.part_norm, layer_bwd_norm_blocks(), p.dv, p.dv, p.d_norm_w),
                         reduce_job(p.part_gates, gb, 2 * p.Hv, p.Hv, p.dA_log),
                         reduce_job(p.part_gates + p.Hv, gb, 2 * p.Hv, p.Hv, p.d_dt_bias)}};
  const unsigned rb = jobs.j[0].blocks + jobs.j[1].blocks + jobs.j[2].blocks + jobs.j[3].blocks;
  hipLaunchKernelGGL(reduce_kernel, dim3(rb), dim3(NT), 0, stream, jobs);
  return hipGetLastError();
}

}  // namespace omx
