// Backward pass (VJP) of the chunked gated delta rule on gfx950.
//
// The reference trains through chunk_gated_delta_rule (omegalax/models/qwen3_5/
// deltanet.py:53-153) with JAX reverse-mode autodiff (trainers/vlm.py:157-195); this
// file computes that derivative.  Per chunk (G = in-chunk cumsum of g, Gamma_im =
// e^{G_i - G_m} for i >= m, X = (I + L)^-1 with L = diag(beta) Lg, Lg = strict_lower(
// K K^T * Gamma), P = lower(scale Q K^T * Gamma); deltanet.py:98-142):
//     V_new = X diag(beta) (V - diag(e^G) K S)               (:115-116, 133-134)
//     O     = scale diag(e^G) Q S + P V_new                   (:136-137)
//     S'    = e^{G_last} S + K^T diag(e^{G_last - G}) V_new   (:139-142)
// Three kernels, after the forward's preparation and scan have been rerun in their
// backward variants (which leave per chunk X and G, for fp32 inputs Lg and P too, and the
// state entering every chunk plus V_new):
//  1. rscan_kernel walks each sequence's chunks backwards carrying dS, the gradient of
//     the state leaving the chunk, in registers (one workgroup per (sequence, value head,
//     64 columns of dv, or 32 or 16 with bf16 inputs; 16 columns per wavefront):
//         dV_new = P^T dO + diag(e^{G_last - G}) K dS
//         dR     = X^T dV_new
//         dS    <- e^{G_last} dS + scale Q^T diag(e^G) dO - K^T diag(e^G) diag(beta) dR
//     and stores dS per chunk and dR.
//  2. cgrad_kernel forms, for every (chunk, value head) at once, the chunk-local
//     gradients of q, k (per value head), v, g and beta from S, dS, V_new, dR and the
//     chunk's matrices (the test oracle, oracle/gdn_vjp.py, differentiates :100-142 step
//     by step; the products by X it takes drop out, see there).
//  3. qk_final_kernel sums the per-value-head q/k gradients over each key head's value
//     heads (the adjoint of the repeat-interleave, :272-280) and applies the L2-norm
//     backward (:30-32), writing dq, dk at the input precision.
// All products are 16x16x32 bf16 MFMAs on operands split into bf16 hi + lo parts
// (hi*hi + hi*lo + lo*hi, fp32-accurate to ~2^-16); operands known to be exact bf16
// (bf16 q/k rows) skip their lo part.
#include <type_traits>

#include "gdn_chunk.h"
#include "gdn_kernels.h"

namespace omx {

namespace {

constexpr int C = kC;
constexpr int NT = kNT;

struct Op {
  u32x4 h, l;
};

// bf16 hi and lo parts of 8 values (x = hi + lo to ~2^-16 relative)
template <bool LO = true>
__device__ __forceinline__ Op split8(const float* x) {
  Op o;
  o.h = pack8(x);
  if constexpr (LO) o.l = pack8_lo(x);
  else o.l = o.h;
  return o;
}

// acc += A B: hi*hi, plus hi*lo when B has a lo part, plus lo*hi when A has one
template <bool AL, bool BL>
__device__ __forceinline__ f32x4 mm3(f32x4 acc, const Op& a, const Op& b) {
  acc = mma16(a.h, b.h, acc);
  if constexpr (BL) acc = mma16(a.h, b.l, acc);
  if constexpr (AL) acc = mma16(a.l, b.h, acc);
  return acc;
}

// B operand from two C-layout tiles side by side (block-pair contraction order)
__device__ __forceinline__ Op join_op(f32x4 a, f32x4 b) {
  Op o;
  o.h = u32x4{pack_bf16(a[0], a[1]), pack_bf16(a[2], a[3]), pack_bf16(b[0], b[1]),
              pack_bf16(b[2], b[3])};
  const u32x2 la = pack_lo4(a), lb = pack_lo4(b);
  o.l = u32x4{la[0], la[1], lb[0], lb[1]};
  return o;
}

__device__ __forceinline__ float ldx(const float* p) { return *p; }
__device__ __forceinline__ float ldx(const bf16_t* p) { return bf2f(*p); }

// operand row `row` of a row-major M[row][k], slots over k from k0 (slot e of lane group q:
// 8q + e)
template <class T>
__device__ __forceinline__ void frag_row(const T* m, int ld, int row, int k0, float* x) {
  const int q = lane_id() >> 4;
#pragma unroll
  for (int e = 0; e < 8; ++e) x[e] = ldx(m + row * ld + k0 + 8 * q + e);
}
// operand column `col` of a row-major M[k][col], slots over the rows from k0 in the
// block-pair order of two C-layout tiles side by side (4q + e%4, then 16 + 4q + e%4)
template <class T>
__device__ __forceinline__ void frag_col(const T* m, int ld, int col, int k0, float* x) {
  const int q = lane_id() >> 4;
#pragma unroll
  for (int e = 0; e < 8; ++e) x[e] = ldx(m + (k0 + 4 * q + (e & 3) + 16 * (e >> 2)) * ld + col);
}

// K / Q operand fragments from the staged rows: bf16 rows are exact bf16 (one vector or
// two transposed LDS reads, no lo part); fp32 rows are read element-wise and split.
// kq_row: row row0 + lane%16, slots over columns from k0.
__device__ __forceinline__ Op kq_row(const float* m, int ld, int row0, int k0) {
  float x[8];
  frag_row(m, ld, row0 + (lane_id() & 15), k0, x);
  return split8(x);
}
__device__ __forceinline__ Op kq_row(const bf16_t* m, int ld, int row0, int k0) {
  const int l = lane_id(), q = l >> 4;
  Op o;
  o.h = *(const u32x4*)(m + (row0 + (l & 15)) * ld + k0 + 8 * q);
  o.l = o.h;
  return o;
}
// kq_st: column (row lane%16 of state tile t in the scans' order), slots over rows from k0
// in the block-pair order.
__device__ __forceinline__ Op kq_st(const float* m, int ld, int t, int k0) {
  const int r = lane_id() & 15;
  float x[8];
  frag_col(m, ld, 32 * (t >> 1) + 4 * (t & 1) + 8 * (r >> 2) + (r & 3), k0, x);
  return split8(x);
}
__device__ __forceinline__ Op kq_st(const bf16_t* m, int ld, int t, int k0) {
  const int l = lane_id(), q = l >> 4, s = l & 15;
  // source lane s of a 16-lane group points at row s / 4 and the 4 columns of row group s % 4
  const bf16_t* pr = m + (k0 + 4 * q + (s >> 2)) * ld + 32 * (t >> 1) + 4 * (t & 1) + 8 * (s & 3);
  const u32x2 a = ds_read_tr(pr), b = ds_read_tr(pr + 16 * ld);
  Op o;
  o.h = u32x4{a[0], a[1], b[0], b[1]};
  o.l = o.h;
  return o;
}

// Loads whose rows may lie past a sequence's end go through a buffer resource whose range
// ends at the last valid row: the hardware returns zeros beyond it.  So no load sits under
// a branch, which would leave the count of outstanding memory operations unknown and turn
// every later wait for one of them into a wait for all (the previous chunk's stores too).
// Byte offsets are 32-bit.
__device__ __forceinline__ float4 bload4(__amdgpu_buffer_rsrc_t r, unsigned off, const float*, int soff = 0) {
  const u32x4 w = __builtin_amdgcn_raw_buffer_load_b128(r, off, soff, 0);
  return float4{__uint_as_float(w[0]), __uint_as_float(w[1]), __uint_as_float(w[2]),
                __uint_as_float(w[3])};
}
__device__ __forceinline__ u32x2 bload4(__amdgpu_buffer_rsrc_t r, unsigned off, const bf16_t*, int soff = 0) {
  return __builtin_amdgcn_raw_buffer_load_b64(r, off, soff, 0);
}
// 4 elements in registers (4 bf16 in two words, or 4 floats)
template <class T> struct Vec4;
template <> struct Vec4<float> { typedef float4 type; };
template <> struct Vec4<bf16_t> { typedef u32x2 type; };
__device__ __forceinline__ float4 load4(const float* src) { return *(const float4*)src; }
__device__ __forceinline__ void store4(float* dst, float4 x) { *(float4*)dst = x; }
__device__ __forceinline__ float4 to_f4(float4 x) { return x; }
__device__ __forceinline__ float4 to_f4(u32x2 x) {
  return float4{__uint_as_float(x[0] << 16), __uint_as_float(x[0] & 0xffff0000u),
                __uint_as_float(x[1] << 16), __uint_as_float(x[1] & 0xffff0000u)};
}
__device__ __forceinline__ void store4(bf16_t* dst, u32x2 x) { *(u32x2*)dst = x; }
// 8 consecutive elements (16 bytes of bf16, or two 16-byte fp32 loads) as floats
__device__ __forceinline__ void load8v(const bf16_t* p, float* x) {
  const u32x4 w = *(const u32x4*)p;
  unpack8<false>(&w, x);
}
__device__ __forceinline__ void load8v(const float* p, float* x) {
  const float4 a = *(const float4*)p, b = *(const float4*)(p + 4);
  x[0] = a.x; x[1] = a.y; x[2] = a.z; x[3] = a.w; x[4] = b.x; x[5] = b.y; x[6] = b.z; x[7] = b.w;
}

// N consecutive values of one row at a buffer offset (bytes), at the precision T
template <class T, int N>
__device__ __forceinline__ void store_row(__amdgpu_buffer_rsrc_t r, unsigned off, const float* x) {
  if constexpr (std::is_same<T, float>::value) {
#pragma unroll
    for (int e = 0; e < N; e += 4)
      __builtin_amdgcn_raw_buffer_store_b128(u32x4{__float_as_uint(x[e]), __float_as_uint(x[e + 1]),
                                                   __float_as_uint(x[e + 2]), __float_as_uint(x[e + 3])},
                                             r, off + 4u * e, 0, 0);
  } else if constexpr (N == 8) {
    __builtin_amdgcn_raw_buffer_store_b128(pack8(x), r, off, 0, 0);
  } else {
    __builtin_amdgcn_raw_buffer_store_b64(u32x2{pack_bf16(x[0], x[1]), pack_bf16(x[2], x[3])}, r, off, 0, 0);
  }
}

// Row sums of a C-layout tile (lane (q, r) holds rows 16 bi + 4q + v, v = 0..3, of
// column r) into arr[row], without LDS traffic: a reduce-scatter over the 16 lanes of
// each row group with DPP moves.  Lanes r and r ^ 8 split the four rows between them
// (row_ror:8), lanes r and its mirror in the 8-lane half split the pair (row_half_mirror),
// then each quad sums (quad_perm); lane r with r % 4 == 0 ends with row 16 bi + 4q + r / 4.
__device__ __forceinline__ void set_rows(float* arr, int bi, f32x4 x) {
  const int l = lane_id(), r = l & 15;
  const bool up8 = (r & 8) != 0, up4 = (r & 4) != 0;
  const float k0 = up8 ? x[2] : x[0], k1 = up8 ? x[3] : x[1];
  const float g0 = up8 ? x[0] : x[2], g1 = up8 ? x[1] : x[3];
  const float a0 = k0 + dpp_f<0x128>(g0), a1 = k1 + dpp_f<0x128>(g1);
  const float kb = up4 ? a1 : a0, gb = up4 ? a0 : a1;
  float s = kb + dpp_f<0x141>(gb);
  s += dpp_f<0x4E>(s);
  s += dpp_f<0xB1>(s);
  if ((r & 3) == 0) arr[16 * bi + 4 * (l >> 4) + (r >> 2)] = s;
}
// Column sums of a C-layout tile (column 16 bj + r, summed over its 16 rows) into
// arr[col]: the lane's four rows, then across the four row groups with the 16- and 32-lane
// swaps (lanes of row group 0 write).
__device__ __forceinline__ void set_cols(float* arr, int bj, f32x4 x) {
  const int l = lane_id();
  float s = x[0] + x[1] + x[2] + x[3];
  const auto a = __builtin_amdgcn_permlane16_swap(__float_as_uint(s), __float_as_uint(s), false, false);
  s = __uint_as_float(a[0]) + __uint_as_float(a[1]);
  const auto b = __builtin_amdgcn_permlane32_swap(__float_as_uint(s), __float_as_uint(s), false, false);
  s = __uint_as_float(b[0]) + __uint_as_float(b[1]);
  if ((l >> 4) == 0) arr[16 * bj + (l & 15)] = s;
}

// Gamma = e^{a - b}, at most 1, from the hardware exp2 (below 2^-126: zero).  The difference
// comes first: scaled to base 2 one by one, each gate would leave its own rounding in Gamma,
// on its unit diagonal too where a product is contracted into the subtraction.
__device__ __forceinline__ float gate_ratio(float a, float b) {
  return __builtin_amdgcn_exp2f(fminf(a - b, 0.f) * 1.4426950408889634f);
}

// Sum over the 64 lanes, left in every lane (DPP within each row, then the row swaps).
__device__ __forceinline__ float wave_sum(float s) {
  s = group_sum_dpp<16>(s);
  const auto a = __builtin_amdgcn_permlane16_swap(__float_as_uint(s), __float_as_uint(s), false, false);
  s = __uint_as_float(a[0]) + __uint_as_float(a[1]);
  const auto b = __builtin_amdgcn_permlane32_swap(__float_as_uint(s), __float_as_uint(s), false, false);
  return __uint_as_float(b[0]) + __uint_as_float(b[1]);
}

__device__ __forceinline__ int rec_mode(bool f32) { return f32 ? MODE_F32 : MODE_BF16; }

// Split-matrix operands.  A 64-row fp32 matrix the backward kernels read as MFMA operands
// is kept in LDS as bf16 hi and lo planes (hi + lo is the value to ~2^-16 relative), split
// once when it is written, so no fragment read converts.  op_vec: lane (q, r) gets entries
// k0 + 8q .. +7 of storage row r0 + r (one 16-byte read per plane); op_tr: entries
// k0 + 8q .. +7 down storage column c0 + r (two transposed 8-byte reads per plane).
template <bool LO = true>
__device__ __forceinline__ Op op_vec(const bf16_t* h, const bf16_t* lo, int ld, int r0, int k0) {
  const int l = lane_id();
  const int off = (r0 + (l & 15)) * ld + k0 + 8 * (l >> 4);
  Op o;
  o.h = *(const u32x4*)(h + off);
  if constexpr (LO) o.l = *(const u32x4*)(lo + off);
  else o.l = o.h;
  return o;
}
template <bool LO = true>
__device__ __forceinline__ Op op_tr(const bf16_t* h, const bf16_t* lo, int ld, int c0, int k0) {
  Op o;
  o.h = frag_tr(h, ld, k0, c0);
  if constexpr (LO) o.l = frag_tr(lo, ld, k0, c0);
  else o.l = o.h;
  return o;
}
// A C-layout tile (lane (q, r): rows row0 + 4q .. +3 of column col0 + r) into column-major
// planes (storage [col][row]): one 8-byte write per plane.
__device__ __forceinline__ void put_ct(bf16_t* h, bf16_t* lo, int ld, int row0, int col0, f32x4 c) {
  const int l = lane_id();
  const int off = (col0 + (l & 15)) * ld + row0 + 4 * (l >> 4);
  *(u32x2*)(h + off) = pack_hi4(c);
  *(u32x2*)(lo + off) = pack_lo4(c);
}
// Four consecutive entries (one row, 4 columns from col) into row-major planes.
__device__ __forceinline__ void put_row4(bf16_t* h, bf16_t* lo, int off, f32x4 c) {
  *(u32x2*)(h + off) = pack_hi4(c);
  *(u32x2*)(lo + off) = pack_lo4(c);
}

// op_vec in the block-pair contraction order (as frag_col): entries k0 + 4q .. +3 and
// k0 + 16 + 4q .. +3 of storage row r0 + r.
__device__ __forceinline__ Op op_pair(const bf16_t* h, const bf16_t* lo, int ld, int r0, int k0) {
  const int l = lane_id();
  const int off = (r0 + (l & 15)) * ld + k0 + 4 * (l >> 4);
  Op o;
  const u32x2 a = *(const u32x2*)(h + off), b = *(const u32x2*)(h + off + 16);
  const u32x2 c = *(const u32x2*)(lo + off), d = *(const u32x2*)(lo + off + 16);
  o.h = u32x4{a[0], a[1], b[0], b[1]};
  o.l = u32x4{c[0], c[1], d[0], d[1]};
  return o;
}
// op_tr in the block-pair contraction order (as frag_col): entries k0 + 4q .. +3 and
// k0 + 16 + 4q .. +3 down storage column c0 + r
__device__ __forceinline__ Op op_tr_pair(const bf16_t* h, const bf16_t* lo, int ld, int c0, int k0) {
  const int l = lane_id(), q = l >> 4, s = l & 15;
  const int off = (k0 + 4 * q + (s >> 2)) * ld + c0 + 4 * (s & 3);
  const u32x2 a = ds_read_tr(h + off), b = ds_read_tr(h + off + 16 * ld);
  const u32x2 c = ds_read_tr(lo + off), d = ds_read_tr(lo + off + 16 * ld);
  Op o;
  o.h = u32x4{a[0], a[1], b[0], b[1]};
  o.l = u32x4{c[0], c[1], d[0], d[1]};
  return o;
}
// the fp32 values (hi + lo) of an operand's 8 slots
__device__ __forceinline__ void op_values(const Op& o, float* x) {
#pragma unroll
  for (int w = 0; w < 4; ++w) {
    x[2 * w] = __uint_as_float(o.h[w] << 16) + __uint_as_float(o.l[w] << 16);
    x[2 * w + 1] = __uint_as_float(o.h[w] & 0xffff0000u) + __uint_as_float(o.l[w] & 0xffff0000u);
  }
}

// ============================================================================ reverse scan

// index of the lower-triangular 16x16 tile (mb, nb), mb >= nb, of a 64x64 chunk matrix
__device__ __forceinline__ constexpr int ptile_index(int mb, int nb) { return mb * (mb + 1) / 2 + nb; }

// With bf16 inputs (LDR) four loader wavefronts beside the four compute wavefronts move
// each chunk's rows into one of two LDS buffers while the compute wavefronts work on the
// other, and form the chunk's P tiles once for all of them; the compute wavefronts issue
// no loads at all.  Two barriers per chunk: one opens the step (the chunk's rows are
// staged, the other buffer is free), one publishes the P tiles.  fp32 K and Q rows leave
// no room for a second buffer, so with fp32 inputs the compute wavefronts stage the rows
// themselves from a register prefetch two chunks deep.
//
// NWC compute wavefronts of 16 columns each (as the forward scan's workgroups: four, or two
// or one where 64-column workgroups would leave CUs idle; fp32 inputs take four).
template <int DK, bool F32, int NWC>
__global__ __launch_bounds__(F32 ? NT : 64 * NWC + NT) void rscan_kernel(BwdParams p) {
  static_assert(!F32 || NWC == 4, "fp32 inputs: the four compute wavefronts stage the rows");
  constexpr int BV = 16 * NWC;  // columns of dv per workgroup
  using KT = typename std::conditional<F32, float, bf16_t>::type;
  // bf16 rows of 128 lie in the scans' swizzled layout, others padded by 16 bytes.  Padded,
  // half of the LDS's busy cycles were conflicts (the transposed reads four ways, each
  // 16-byte pass one; now 14M of 54M cycles for 40M of 81M): C1 317 -> 307 us, layer rows at
  // B=1 T=3,001 Hv=32 110.5 -> 107.
  constexpr bool SWZ = !F32 && DK == 128;
  constexpr int LDK = SWZ ? DK : DK + (F32 ? 4 : 8);
  constexpr int LDB = C + 8;  // stride (bf16) of a split plane
  constexpr bool LDR = !F32;
  // bf16 inputs form the P operands in registers (PREC) from the staged K and Q rows and G
  constexpr bool PREC = !F32;
  // Buffer 0 and (LDR) buffer 1 are separate objects, so the compiler can tell the
  // loaders' writes to one from the compute wavefronts' reads of the other.
  __shared__ __align__(16) KT sK0[C * LDK], sK1[LDR ? C * LDK : 8];
  __shared__ __align__(16) KT sQ0[C * LDK], sQ1[LDR ? C * LDK : 8];
  // dO (this block's columns), X (fp32 inputs: X^T) and (fp32 inputs) P, row-major, as
  // bf16 hi / lo planes
  __shared__ __align__(16) bf16_t sDO0[2 * C * LDB], sDO1[LDR ? 2 * C * LDB : 8];
  __shared__ __align__(16) bf16_t sX0[2 * C * LDB], sX1[LDR ? 2 * C * LDB : 8];
  __shared__ __align__(16) bf16_t sP[PREC ? 8 : 2 * C * LDB];
  // (LDR) the chunk's ten lower-triangular 16x16 tiles of P, formed once by the loaders:
  // lane l of tile t holds its C-layout values as bf16 hi (2 words) then lo (2 words)
  __shared__ __align__(16) u32x4 sPT[LDR ? 10 : 1][64];
  __shared__ float sGl0[PREC ? C : 1], sGl1[LDR ? C : 1];
  __shared__ __align__(16) float sGate0[4 * C], sGate1[LDR ? 4 * C : 4];
  struct Buf {
    KT* K;
    KT* Q;
    bf16_t* DO;
    bf16_t* X;
    float* Gl;
    float* Gate;
  };
  const Buf B0{sK0, sQ0, sDO0, sX0, sGl0, sGate0};
  const Buf B1{sK1, sQ1, sDO1, sX1, sGl1, sGate1};
  bf16_t* const sPh = sP;
  bf16_t* const sPl = sP + C * LDB;

  const int tid = threadIdx.x, l = tid & 63, lq = l >> 4, lr = l & 15;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const bool loader = LDR && wave >= NWC;      // (LDR) the last four: rows and P tiles only
  const int st = loader ? tid - 64 * NWC : tid;  // index among the NT threads that stage rows
  const ScanItem item = scan_item(p.seq_order, p.N, p.Hk, p.Hv, p.nb, blockIdx.x);
  const int blk = item.blk, h = item.h, n = item.n;
  const int gqa = p.Hv / p.Hk, hk = h / gqa;
  const int DV = p.DV, col0 = BV * blk, c = 16 * wave;
  long long s0, s1;
  seq_range(p.cu_seqlens, n, p.T, s0, s1);
  const int nchunks = (int)((s1 - s0 + C - 1) / C);
  const int cbase = p.chunk_off ? p.chunk_off[n] : n * p.nch;
  const size_t rec_stride = (size_t)rec_bytes(rec_mode(F32), true);
  const long long rs = (long long)p.Hv * DV;  // row stride of dO / dV_new

  // dS[t][v] = dS[st_row(t, v)][col0 + c + lr]: gradient of the state leaving the chunk, its
  // rows in the forward scan's order (two tiles side by side are the B operand over 32
  // consecutive dk, so K's operands are plain rows); dsb: its split operands
  auto st_row = [&](int t, int v) { return 32 * (t >> 1) + 8 * lq + 4 * (t & 1) + v; };
  f32x4 dS[DK / 16];
  Op dsb[DK / 32];
  const size_t st_off = ((size_t)n * p.Hv + h) * DK * DV + col0 + c + lr;
  auto init_dS = [&]() {
#pragma unroll
    for (int t = 0; t < DK / 16; ++t)
#pragma unroll
      for (int v = 0; v < 4; ++v)
        dS[t][v] = p.dht ? p.dht[st_off + (size_t)st_row(t, v) * DV] : 0.f;
#pragma unroll
    for (int s = 0; s < DK / 32; ++s) dsb[s] = join_op(dS[2 * s], dS[2 * s + 1]);
  };
  // gradient of the initial state
  auto write_dh0 = [&]() {
    if (p.dh0) {
#pragma unroll
      for (int t = 0; t < DK / 16; ++t)
#pragma unroll
        for (int v = 0; v < 4; ++v) p.dh0[st_off + (size_t)st_row(t, v) * DV] = dS[t][v];
    }
  };

  // Per-thread register copy of a chunk's inputs: K and Q rows, the chunk's dO columns,
  // X and P, and one gate value, loaded by the NT staging threads (the loaders, or with
  // fp32 inputs the compute wavefronts, two register sets deep) and stored into LDS a
  // chunk step later.
  constexpr int NKQ = 2 * C * (DK / 4) / NT;
  static_assert(NKQ * NT == 2 * C * (DK / 4), "item split");
  constexpr int NXP = (2 * kNPieces * 64 + NT - 1) / NT;  // (PREC) 16-byte items of the record's X
  struct Pf {
    typename Vec4<KT>::type pkq[NKQ];
    float4 pdo[C * BV / 4 / NT], pxp[PREC ? 1 : 2 * C * 16 / NT];
    u32x4 px[PREC ? NXP : 1];
    float pgate, pg;
  };
  // chunk jj into f; every call issues the same loads (a chunk before the sequence's first
  // reloads chunk 0, unused), so the loop's waits stay exact counts
  auto load_chunk = [&](int jj, Pf& f) {
    jj = jj < 0 ? 0 : jj;
    const long long tt = s0 + (long long)jj * C;
    const int nv = (int)((s1 - tt) < C ? (s1 - tt) : C);
    const int sl = cbase + jj < p.n_rec ? cbase + jj : p.n_rec - 1;
    // the chunk's valid rows only (zeros past them)
    const auto kr = buf_rsrc((const KT*)p.ks + tt * p.ks_ld + (long long)hk * DK,
                             (unsigned)(nv * p.ks_ld * (long long)sizeof(KT)));
    const auto qr = buf_rsrc((const KT*)p.qs + tt * p.qs_ld + (long long)hk * DK,
                             (unsigned)(nv * p.qs_ld * (long long)sizeof(KT)));
    const auto dr = buf_rsrc(p.dO + tt * rs + (long long)h * DV + col0, (unsigned)(4 * nv * rs));
    static_assert((C * DK / 4) % NT == 0, "a K / Q item's matrix follows from m alone");
#pragma unroll
    for (int m = 0; m < NKQ; ++m) {
      const int which = m * NT / (C * DK / 4);  // uniform: K items, then Q items
      const int rem = st + m * NT - which * (C * DK / 4);
      const int row = rem / (DK / 4), c4 = 4 * (rem % (DK / 4));
      const long long ld = which ? p.qs_ld : p.ks_ld;
      f.pkq[m] = bload4(which ? qr : kr, (unsigned)((row * ld + c4) * (long long)sizeof(KT)), (const KT*)nullptr);
    }
#pragma unroll
    for (int m = 0; m < C * BV / 4 / NT; ++m) {
      const int it = st + m * NT;
      const int row = it / (BV / 4), c4 = 4 * (it % (BV / 4));
      f.pdo[m] = bload4(dr, (unsigned)(4 * (row * rs + c4)), (const float*)nullptr);
    }
    const float* xb = p.xlpg + ((size_t)sl * p.Hv + h) * xlpg_floats(F32);
    const unsigned char* rec = p.rec + ((size_t)sl * p.Hv + h) * rec_stride;
    if constexpr (PREC) {
#pragma unroll
      for (int m = 0; m < NXP; ++m)
        f.px[m] = *(const u32x4*)(rec + kRecT + 16 * (st + m * NT));  // (past X: P, unused)
      f.pg = xb[kXlpgG + (st & (C - 1))];
    } else {
#pragma unroll
      for (int m = 0; m < 2 * C * 16 / NT; ++m) {
        const int it = st + m * NT;
        const int which = it / (C * 16), rem = it % (C * 16);
        f.pxp[m] = load4(xb + (which ? kXlpgP : kXlpgX) + (rem >> 4) * C + 4 * (rem & 15));
      }
    }
    f.pgate = ((const float*)(rec + kRecG))[st];
  };
  auto store_chunk = [&](const Pf& f, const Buf& bf) {
    bf16_t* const sDOh = bf.DO;
    bf16_t* const sDOl = bf.DO + C * LDB;
    bf16_t* const sXh = bf.X;
    bf16_t* const sXl = bf.X + C * LDB;
#pragma unroll
    for (int m = 0; m < NKQ; ++m) {
      const int it = st + m * NT;
      const int which = it / (C * DK / 4), rem = it % (C * DK / 4);
      const int row = rem / (DK / 4), c4 = 4 * (rem % (DK / 4));
      store4((which ? bf.Q : bf.K) + (SWZ ? swz_off<128>(row, c4) : row * LDK + c4), f.pkq[m]);
    }
#pragma unroll
    for (int m = 0; m < C * BV / 4 / NT; ++m) {
      const int it = st + m * NT;
      put_row4(sDOh, sDOl, (it / (BV / 4)) * LDB + 4 * (it % (BV / 4)), f32x4{f.pdo[m].x, f.pdo[m].y, f.pdo[m].z, f.pdo[m].w});
    }
    if constexpr (PREC) {
      // piece 2x + part of the record's T part, hi (part 0) or lo: lane (q, r) of the pieces
      // x >= 1, pairs (ib, jp) = (1, 0), (2, 0), (3, 0), (3, 1), holds X[16 ib + r][32 jp +
      // 4q .. +3] and [32 jp + 16 + 4q .. +3]; of piece 0 the diagonal tiles (0, 0) and
      // (2, 2), whose right neighbours are zero
#pragma unroll
      for (int m = 0; m < NXP; ++m) {
        const int piece = (st >> 6) + m * (NT / 64), x = piece >> 1;  // uniform per wavefront
        if (x >= kNPieces) break;
        bf16_t* const pl = piece & 1 ? sXl : sXh;
        const u32x2 w0 = {f.px[m][0], f.px[m][1]}, w1 = {f.px[m][2], f.px[m][3]}, z = {0u, 0u};
        const int ib = x < 4 ? x : 3, jp = x == 4;
        bf16_t* d = pl + (16 * ib + lr) * LDB + 32 * jp + 4 * lq;
        *(u32x2*)d = w0;
        *(u32x2*)(d + 16) = x == 0 ? z : w1;
        if (x == 0) {
          bf16_t* e = pl + (32 + lr) * LDB + 32 + 4 * lq;
          *(u32x2*)e = w1;
          *(u32x2*)(e + 16) = z;
        }
      }
    } else {
#pragma unroll
      for (int m = 0; m < 2 * C * 16 / NT; ++m) {
        const int it = st + m * NT;
        const int which = it / (C * 16), rem = it % (C * 16);
        const f32x4 v = f32x4{f.pxp[m].x, f.pxp[m].y, f.pxp[m].z, f.pxp[m].w};
        if (which) put_row4(sPh, sPl, (rem >> 4) * LDB + 4 * (rem & 15), v);
        else put_row4(sXh, sXl, (rem >> 4) * LDB + 4 * (rem & 15), v);
      }
    }
    if constexpr (PREC)
      if (st < C) bf.Gl[st] = f.pg;
    bf.Gate[st] = f.pgate;
  };
  // kq_row and kq_st on the staged K and Q rows
  auto k_row = [&](const auto* m, int r0, int k0) {
    if constexpr (SWZ) {
      Op o;
      o.h = o.l = swz_frag(m, r0, k0);
      return o;
    } else {
      return kq_row(m, LDK, r0, k0);
    }
  };
  auto k_st = [&](const auto* m, int t, int k0) {
    if constexpr (SWZ) {
      Op o;
      o.h = o.l = join(kt_rows4_swz(m, k0, t), kt_rows4_swz(m, k0 + 16, t));
      return o;
    } else {
      return kq_st(m, LDK, t, k0);
    }
  };
  // (LDR) tile (mb, nb) of P = lower(scale Q K^T * Gamma) in the C layout, from the rows
  // staged in bf (with the gates scaled one by one dbeta was 4.9e-5 off at G = -3,800, now 5.6e-6)
  auto form_ptile = [&](int mb, int nb, const Buf& bf) {
    u32x4 qf[DK / 32], kf[DK / 32];
    f32x4 acc = zero4(), w;
    float gm[4];
    const float gn = bf.Gl[16 * nb + lr];
#pragma unroll
    for (int v = 0; v < 4; ++v) gm[v] = bf.Gl[16 * mb + 4 * lq + v];
#pragma unroll
    for (int s2 = 0; s2 < DK / 32; ++s2) {
      qf[s2] = k_row((const bf16_t*)bf.Q, 16 * mb, 32 * s2).h;
      kf[s2] = k_row((const bf16_t*)bf.K, 16 * nb, 32 * s2).h;
    }
    // the factors while the fragments arrive: the compute wavefronts wait for the tiles, so
    // only one product per value follows the MFMAs (B=1 T=3,000 Hv=32 d=128: 141 us, with the
    // factors behind them 144)
#pragma unroll
    for (int v = 0; v < 4; ++v) w[v] = p.scale * gate_ratio(gm[v], gn) * (float)(16 * mb + 4 * lq + v >= 16 * nb + lr);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int s2 = 0; s2 < DK / 32; ++s2) acc = mma16(qf[s2], kf[s2], acc);
    return acc * w;
  };
  // (LDR) the ten tiles, dealt over the four loaders (t = lw, lw + 4, lw + 8), into sPT
  auto form_ptiles = [&](const Buf& bf) {
    const int lw = wave - NWC;
    for (int t = lw; t < 10; t += 4) {  // uniform per wavefront
      const int mb = t < 1 ? 0 : t < 3 ? 1 : t < 6 ? 2 : 3;
      const int nb = t - mb * (mb + 1) / 2;
      const f32x4 x = form_ptile(mb, nb, bf);
      const u32x2 hi = pack_hi4(x), lo = pack_lo4(x);
      sPT[t][l] = u32x4{hi[0], hi[1], lo[0], lo[1]};
    }
  };
  // dR^T of the last computed chunk (tokens dr_t0 .. + dr_n - 1): a lane holds 4 consecutive
  // columns of one token row, one 16-byte store per row block.  It is stored a step later,
  // between the products of the next chunk: stored at once, it met the next chunk's dS stores
  // and the loaders' loads (rscan 334 us; so 320 us; C1).  Rows past the chunk's end lie
  // outside the buffer range and are dropped: no branch.
  f32x4 dr[4];
  long long dr_t0 = 0;
  int dr_n = 0;
#pragma unroll
  for (int i = 0; i < 4; ++i) dr[i] = zero4();
  auto put_dr = [&]() {
    const auto vd = buf_rsrc(p.drows + dr_t0 * rs + (long long)h * DV + col0, 4u * (unsigned)dr_n * (unsigned)rs);
#pragma unroll
    for (int i = 0; i < 4; ++i)
      __builtin_amdgcn_raw_buffer_store_b128(
          u32x4{__float_as_uint(dr[i][0]), __float_as_uint(dr[i][1]), __float_as_uint(dr[i][2]), __float_as_uint(dr[i][3])},
          vd, 4u * ((unsigned)(16 * i + lr) * (unsigned)rs + (unsigned)(c + 4 * lq)), 0, 0);
  };
  // chunk j on the compute wavefronts, from the rows staged in bf
  auto compute = [&](const int j, const Buf& bf) {
    const long long t0 = s0 + (long long)j * C;
    const int nvalid = (int)((s1 - t0) < C ? (s1 - t0) : C);
    const int slot = cbase + j < p.n_rec ? cbase + j : p.n_rec - 1;
    const KT* const sK = bf.K;
    const KT* const sQ = bf.Q;
    const bf16_t* const sDOh = bf.DO;
    const bf16_t* const sDOl = bf.DO + C * LDB;
    const bf16_t* const sXh = bf.X;
    const bf16_t* const sXl = bf.X + C * LDB;
    const float* const sGate = bf.Gate;
    const float* sEG = sGate + kGateEG * C;
    const float* sEGS = sGate + kGateEGS * C;
    const float* sEL = sGate + kGateEL * C;  // e^{G_last - G}; e^{G_last} in the last slot
    const float* sB = sGate + kGateBeta * C;

    // dO of the wavefront's 16 columns over each half of the chunk, in the block-pair order
    // of every product it enters, and scale e^G dO for the state's Q^T term: neither waits
    // for dS, so both are formed beside K dS
    Op dob[2], b1[2];
#pragma unroll
    for (int p2 = 0; p2 < 2; ++p2) dob[p2] = op_tr_pair(sDOh, sDOl, LDB, c, 32 * p2);
    // ---------------------------------------------------------------- K dS
    f32x4 kds[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) kds[i] = zero4();
#pragma unroll
    for (int s = 0; s < DK / 32; ++s)
#pragma unroll
      for (int i = 0; i < 4; ++i) kds[i] = mm3<F32, true>(kds[i], k_row(sK, 16 * i, 32 * s), dsb[s]);
#pragma unroll
    for (int p2 = 0; p2 < 2; ++p2) {
      float x[8];
      op_values(dob[p2], x);
      const float4 ga = *(const float4*)(sEGS + 32 * p2 + 4 * lq), gb = *(const float4*)(sEGS + 32 * p2 + 16 + 4 * lq);
      const float g[8] = {ga.x, ga.y, ga.z, ga.w, gb.x, gb.y, gb.z, gb.w};
#pragma unroll
      for (int e = 0; e < 8; ++e) x[e] *= g[e];
      b1[p2] = split8(x);
    }
    // gradient of the state leaving chunk j, for the chunk-local gradients: column-major per
    // state ([dv][dk]), a lane's 8 rows of a tile pair are contiguous
    {
      float* dd = p.dstates + ((size_t)slot * p.Hv + h) * DK * DV + (size_t)(col0 + c + lr) * DK;
#pragma unroll
      for (int t = 0; t < DK / 16; ++t) *(f32x4*)(dd + st_row(t, 0)) = dS[t];
    }
    // (LDR) the loaders' P tiles of this chunk are in sPT after this barrier
    if constexpr (LDR) lds_barrier();
    // ---------------------------------------------------------------- dV_new = P^T dO + e^{G_last-G} K dS
    f32x4 dvn[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      f32x4 acc = zero4();
#pragma unroll
      for (int p2 = i / 2; p2 < 2; ++p2) {  // P^T is upper triangular
        Op pt;
        if constexpr (PREC) {
          // P^T rows 16i .. +15 over tokens 32 p2 .. +31 from the P tiles (2 p2, i) and
          // (2 p2 + 1, i) side by side ((2 p2, i) is above the diagonal, zero, when
          // 2 p2 < i)
          const u32x4 tb = sPT[ptile_index(2 * p2 + 1, i)][l];
          const u32x4 ta = 2 * p2 >= i ? sPT[ptile_index(2 * p2, i)][l] : u32x4{0u, 0u, 0u, 0u};
          pt.h = u32x4{ta[0], ta[1], tb[0], tb[1]};
          pt.l = u32x4{ta[2], ta[3], tb[2], tb[3]};
        } else {
          pt = op_tr_pair(sPh, sPl, LDB, 16 * i, 32 * p2);
        }
        acc = mm3<true, true>(acc, pt, dob[p2]);
      }
      const float4 el4 = *(const float4*)(sEL + 16 * i + 4 * lq);
      const float el[4] = {el4.x, el4.y, el4.z, i == 3 && lq == 3 ? 1.f : el4.w};  // row C - 1: e^0
#pragma unroll
      for (int v = 0; v < 4; ++v) dvn[i][v] = acc[v] + el[v] * kds[i][v];
    }
    __builtin_amdgcn_sched_barrier(0);
    put_dr();
    __builtin_amdgcn_sched_barrier(0);
    Op dvp[2];
#pragma unroll
    for (int pp = 0; pp < 2; ++pp) dvp[pp] = join_op(dvn[2 * pp], dvn[2 * pp + 1]);
    // ------------------------------------------------ dS <- e^{G_last} dS + scale Q^T diag(e^G) dO
    // (its products fill the matrix cores while the chain's vector work, dV_new and Y, runs)
    const float egl = sEL[C - 1];
#pragma unroll
    for (int t = 0; t < DK / 16; ++t) {
#pragma unroll
      for (int v = 0; v < 4; ++v) dS[t][v] *= egl;
#pragma unroll
      for (int p2 = 0; p2 < 2; ++p2) dS[t] = mm3<F32, true>(dS[t], k_st(sQ, t, 32 * p2), b1[p2]);
    }
    __builtin_amdgcn_sched_barrier(0);
    // ---------------------------------------------------------------- dR = X^T dV_new, Y = diag(beta) dR
    // dR is also formed transposed (dR^T = dV_new^T X, the same operands exchanged), for its
    // stores (put_dr)
    f32x4 y[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      f32x4 acc = zero4();
      dr[i] = zero4();
#pragma unroll
      for (int p2 = i / 2; p2 < 2; ++p2) {  // X^T is upper triangular
        const Op x = PREC ? op_tr_pair(sXh, sXl, LDB, 16 * i, 32 * p2) : op_pair(sXh, sXl, LDB, 16 * i, 32 * p2);
        acc = mm3<true, true>(acc, x, dvp[p2]);
        dr[i] = mm3<true, true>(dr[i], dvp[p2], x);
      }
      const float4 b4 = *(const float4*)(sB + 16 * i + 4 * lq), e4 = *(const float4*)(sEG + 16 * i + 4 * lq);
      y[i] = f32x4{-e4.x * (b4.x * acc[0]), -e4.y * (b4.y * acc[1]), -e4.z * (b4.z * acc[2]), -e4.w * (b4.w * acc[3])};
    }
    __builtin_amdgcn_sched_barrier(0);
    // ---------------------------------------------------------------- dS <- dS - K^T diag(e^G) Y
    Op b2[2];
#pragma unroll
    for (int p2 = 0; p2 < 2; ++p2) b2[p2] = join_op(y[2 * p2], y[2 * p2 + 1]);
    dr_t0 = t0;
    dr_n = nvalid;
#pragma unroll
    for (int t = 0; t < DK / 16; ++t)
#pragma unroll
      for (int p2 = 0; p2 < 2; ++p2) dS[t] = mm3<F32, true>(dS[t], k_st(sK, t, 32 * p2), b2[p2]);
#pragma unroll
    for (int s = 0; s < DK / 32; ++s) dsb[s] = join_op(dS[2 * s], dS[2 * s + 1]);
  };
  // Barriers here order LDS accesses only (lds_barrier): the global stores go to later
  // kernels and the staged rows come from per-thread registers, so neither the loads nor
  // the stores are waited for at a barrier.
  if constexpr (LDR) {
    // Chunk j is computed from one buffer while the loaders store chunk j - 1, loaded
    // during the step before, into the other and load chunk j - 2 (a chunk below the
    // sequence's first reloads chunk 0, unused): the barrier that opens a step finds the
    // next buffer filled and the previous one read.  The two roles run separate loops
    // with the same two barriers per step, so neither holds the other's registers.
    int j = nchunks - 1;
    if (loader) {
      Pf f;
      if (nchunks > 0) {
        load_chunk(nchunks - 1, f);
        store_chunk(f, B0);
        load_chunk(nchunks - 2, f);
      }
      // the P tiles of the chunk the compute wavefronts work on, published by the
      // step's second barrier, then the next chunk's rows
      auto lstep = [&](const Buf& cur, const Buf& nxt, const int jj) {
        lds_barrier();
        form_ptiles(cur);
        lds_barrier();
        store_chunk(f, nxt);
        load_chunk(jj - 2, f);
      };
      for (; j >= 1; j -= 2) {
        lstep(B0, B1, j);
        lstep(B1, B0, j - 1);
      }
      if (j == 0) lstep(B0, B1, 0);
    } else {
      init_dS();
      // the prologue's loads under the uniform p.dht test have landed
      __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0)
      auto cstep = [&](const int jj, const Buf& cur) {
        lds_barrier();
        compute(jj, cur);
      };
      for (; j >= 1; j -= 2) {
        cstep(j, B0);
        cstep(j - 1, B1);
      }
      if (j == 0) cstep(0, B0);
      put_dr();
      write_dh0();
    }
  } else {
    init_dS();
    Pf pfa, pfb;
    if (nchunks > 0) {
      load_chunk(nchunks - 1, pfa);
      load_chunk(nchunks - 2, pfb);
    }
    // the prologue's loads (some under the uniform p.dht test) have landed: the loop's
    // waits then count only the loop's own memory operations
    __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0)
    // chunk j from the registers of cur, which then receive chunk jn (lands during this
    // chunk and the next)
    auto step = [&](const int jj, Pf& cur, const int jn) {
      lds_barrier();  // the previous chunk's readers are done
      store_chunk(cur, B0);
      load_chunk(jn, cur);
      lds_barrier();
      compute(jj, B0);
    };
    // chunks n-1, n-3, ... from pfa and n-2, n-4, ... from pfb, each set reloaded with the
    // chunk two below the one it held
    int j = nchunks - 1;
    for (; j >= 1; j -= 2) {
      step(j, pfa, j - 2);
      step(j - 1, pfb, j - 3);
    }
    if (j == 0) step(0, pfa, -2);
    put_dr();
    write_dh0();
  }
}

// ============================================================================ chunk-local gradients

// One workgroup of four wavefronts per (chunk, value head).  With dR = X^T dV_new (the
// gradient of R = diag(beta) (V - diag(e^G) K S), V_new = X R; stored by the reverse scan)
// the derivative of the solve needs no product with X: dX = dV_new R^T, so
//     dL = -strict_lower(X^T dX X^T) = -strict_lower(dR V_new^T).
// The chunk's gradients are then
//     X1 = diag(e^G) dO S^T          -> dq, G          dP = lower(dO V_new^T)  -> P, G
//     Z  = dR S^T                    -> dk, beta, G    dL                     -> L, beta, G
//     Y  = diag(e^{G_last-G}) V_new dS^T -> dk, G      dv = diag(beta) dR
//     dq = scale (X1 + dPg K),  dk = Y - diag(beta e^G) Z + (Qm + Qm^T) K + scale dPg^T Q,
// dPg = dP * Gamma, Qm = diag(beta) (dL * Gamma).
//
// Bound by memory (328 KiB per workgroup at d = 128, two thirds of it fp32 states and row
// gradients).  So the tile is chosen for loads in flight: 78 KB of LDS and at most 256
// VGPRs leave two workgroups per CU, one of which loads while the other multiplies.  The
// products over dv are formed transposed ([dk][token]: the state's fragments as A operand,
// the rows as B), so a lane ends with consecutive dk of one token: the row sums are
// in-lane, the K and Q rows are read and the gradients written by vectors, and every gate
// is one value per lane.  Wavefront w owns dk rows [CB w, CB w + CB), CB = DK / 4 (16 at
// dk = 32, on two wavefronts), and of the chunk matrices row block w of dP and 3 - w of dL
// (five tiles in all: the lower triangles are dealt evenly).
// C1 (B=4, T=4096, Hk=16, Hv=32, d=128): cgrad 933 -> 553 us, moving 2.9 GB at 5.3 TB/s (the
// build with the products by X: 156 KB of LDS, one workgroup per CU, 336 KiB, 2.9 TB/s);
// the core call 1984 -> 1650 us forward and backward.
constexpr int CW = 4, CNT = 64 * CW;

template <int DK, int DV, bool F32>
__global__ __launch_bounds__(CNT) __attribute__((amdgpu_waves_per_eu(2, 2))) void cgrad_kernel(BwdParams p) {
  using KT = typename std::conditional<F32, float, bf16_t>::type;
  using In = KT;  // v has the input precision too
  constexpr int LDK = DK + (F32 ? 4 : 8);
  constexpr int LDB = C + 8;  // stride (bf16) of a split plane: 64 entries and a pad
  constexpr int NKB = DK >= 128 ? 2 : 1;  // 16-row dk blocks per wavefront
  constexpr int NACT = DK / 16 / NKB;     // wavefronts that own dk rows
  static_assert(NACT <= CW && NACT * NKB * 16 == DK, "dk split");
  __shared__ __align__(16) KT sK[C * LDK];
  __shared__ __align__(16) KT sQ[C * LDK];
  // during the products over dv: the staged 32-column slices of dO, dR and V_new; then the
  // split planes of dPg and Qm, column-major (storage [col][row])
  constexpr int LDR = 40;  // stride (bf16) of a staged 32-column slice plane
  constexpr int SZR = 4 * C * LDB > 6 * C * LDR ? 4 * C * LDB : 6 * C * LDR;
  __shared__ __align__(16) bf16_t sR[SZR];
  bf16_t* const sDOh = sR;
  bf16_t* const sDOl = sR + C * LDR;
  bf16_t* const sDRh = sR + 2 * C * LDR;
  bf16_t* const sDRl = sR + 3 * C * LDR;
  bf16_t* const sVNh = sR + 4 * C * LDR;
  bf16_t* const sVNl = sR + 5 * C * LDR;
  bf16_t* const sDPh = sR;
  bf16_t* const sDPl = sR + C * LDB;
  bf16_t* const sQMh = sR + 2 * C * LDB;
  bf16_t* const sQMl = sR + 3 * C * LDB;
  __shared__ float sG[C], sBt[C];
  // partial sums per wavefront (deterministic: every entry has one writer)
  __shared__ float sX1[CW][C], sZ[CW][C], sY[CW][C];  // rows over the wavefront's dk
  __shared__ float sCol[CW][C];                       // columns of its tiles of P dP and L dL
  __shared__ float sRowP[C], sRowL[C], sRowB[C];      // rows of P dP, of L dL, of Lg dL
  __shared__ float sRV[C];                            // dR . v
  __shared__ float sRed[CW];

  const int tid = threadIdx.x, l = tid & 63, lq = l >> 4, lr = l & 15;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const bool active = NACT == CW || wave < NACT;
  const int Hv = p.Hv, h = blockIdx.x % Hv, ci = blockIdx.x / Hv;
  int n, cc;
  if (p.chunk_off) {
    if (ci >= p.chunk_off[p.N]) return;
    int lo = 0, hi = p.N;
    while (hi - lo > 1) {
      const int mid = (lo + hi) >> 1;
      if (p.chunk_off[mid] <= ci) lo = mid;
      else hi = mid;
    }
    n = lo;
    cc = ci - p.chunk_off[lo];
  } else {
    n = ci / p.nch;
    cc = ci % p.nch;
  }
  long long s0, s1;
  seq_range(p.cu_seqlens, n, p.T, s0, s1);
  const long long t0 = s0 + (long long)cc * C;
  const int nvalid = (int)((s1 - t0) < C ? (s1 - t0) : C);
  if (nvalid <= 0) return;
  const int gqa = Hv / p.Hk, hk = h / gqa;
  const size_t rec_stride = (size_t)rec_bytes(rec_mode(F32), true);
  const float* xb = p.xlpg + ((size_t)ci * Hv + h) * xlpg_floats(F32);
  const long long rs = (long long)Hv * DV;  // row stride of dO, V_new, dR, v
  const float scale = p.scale;

  // dk index of row r of the wavefront's tile t, and of the first of the four consecutive
  // dk a lane holds of that tile: with two tiles, lane group q holds dk 8q .. 8q + 7
  const int dk0 = 16 * NKB * (active ? wave : 0);
  auto dk_row = [&](int t, int r) { return dk0 + (NKB == 2 ? 8 * (r >> 2) + 4 * t + (r & 3) : r); };
  auto dk_own = [&](int t) { return dk0 + (NKB == 2 ? 8 * lq + 4 * t : 4 * lq); };

  // ---------------------------------------------------------------- stage
  // K and Q rows in 16-byte items, every load issued (with the first step's) before any
  // store, so the workgroup waits for one memory round trip rather than one per item.  The
  // chunk's valid rows only (zeros past them, no branch: see bload4).
  const unsigned rows_b = (unsigned)(nvalid * rs);  // elements
  const long long ro = t0 * rs + (long long)h * DV;
  const auto rDO = buf_rsrc(p.dO + ro, 4u * rows_b), rDR = buf_rsrc(p.drows + ro, 4u * rows_b);
  const auto rVN = buf_rsrc(p.vnew + ro, 4u * rows_b);
  const auto rV = buf_rsrc((const In*)p.v + ro, (unsigned)sizeof(In) * rows_b);
  const auto rDV = buf_rsrc((In*)p.dv + ro, (unsigned)sizeof(In) * rows_b);
  constexpr int EPI = 16 / (int)sizeof(KT);  // elements per item
  constexpr int PER = C * DK / EPI;          // items per matrix
  constexpr int NIT = 2 * PER / CNT;
  static_assert(NIT * CNT == 2 * PER && PER % CNT == 0, "staging split");
  u32x4 st[NIT];
  {
    const auto kr = buf_rsrc((const KT*)p.ks + t0 * p.ks_ld + (long long)hk * DK,
                             (unsigned)(nvalid * p.ks_ld * (long long)sizeof(KT)));
    const auto qr = buf_rsrc((const KT*)p.qs + t0 * p.qs_ld + (long long)hk * DK,
                             (unsigned)(nvalid * p.qs_ld * (long long)sizeof(KT)));
#pragma unroll
    for (int m = 0; m < NIT; ++m) {
      const int which = m * CNT / PER;  // uniform: K items, then Q items
      const int rem = tid + m * CNT - which * PER;
      const int row = rem / (DK / EPI), c = EPI * (rem % (DK / EPI));
      const long long ld = which ? p.qs_ld : p.ks_ld;
      st[m] = __builtin_amdgcn_raw_buffer_load_b128(which ? qr : kr,
                                                    (unsigned)((row * ld + c) * (long long)sizeof(KT)), 0, 0);
    }
  }
  // the thread's staged items of a 32-column step: rows srow and srow + 32, 4 columns each
  constexpr int NRI = C * 8 / CNT;
  const int srow = tid >> 3, sc4 = 4 * (tid & 7);
  float4 pf_do[NRI], pf_dr[NRI], pf_vn[NRI];
  typename Vec4<In>::type pf_v[NRI];
  // element offset of the thread's item of row srow; the step's columns go in the scalar
  // offset (a row past the end is past the range without them)
  const unsigned roff = (unsigned)srow * (unsigned)rs + sc4;
  auto load_rows = [&](int u) {
#pragma unroll
    for (int m = 0; m < NRI; ++m) {
      const unsigned off = roff + m * (CNT / 8) * (unsigned)rs;
      pf_do[m] = bload4(rDO, 4u * off, (const float*)nullptr, 4 * 32 * u);
      pf_dr[m] = bload4(rDR, 4u * off, (const float*)nullptr, 4 * 32 * u);
      pf_vn[m] = bload4(rVN, 4u * off, (const float*)nullptr, 4 * 32 * u);
      pf_v[m] = bload4(rV, (unsigned)sizeof(In) * off, (const In*)nullptr, (int)sizeof(In) * 32 * u);
    }
  };
  // state fragments (the states are column-major, [dv][dk]): row dk_row(t, lr), 8
  // consecutive dv
  float sfr[NKB][8], dfr[NKB][8];
  const auto rS = buf_rsrc(p.states + ((size_t)ci * Hv + h) * DK * DV, 4u * DK * DV);
  const auto rDS = buf_rsrc(p.dstates + ((size_t)ci * Hv + h) * DK * DV, 4u * DK * DV);
  const unsigned soff = 4u * (8 * lq * DK + dk_row(0, lr));
  auto load_state = [&](__amdgpu_buffer_rsrc_t r, int u, float (&x)[NKB][8]) {
    // opaque at each use: hoisted out of the loop, every load's offset would hold a register
    // of its own instead of being the instruction's immediate
    unsigned so = soff;
    asm volatile("" : "+v"(so));
#pragma unroll
    for (int t = 0; t < NKB; ++t)
#pragma unroll
      for (int e = 0; e < 8; ++e)
        x[t][e] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(r, so + 4u * (e * DK + 4 * t), 4 * 32 * u * DK, 0));
  };
  load_rows(0);
  load_state(rS, 0, sfr);
  if (tid < C) {
    sG[tid] = xb[kXlpgG + tid];
    sBt[tid] = ((const float*)(p.rec + ((size_t)ci * Hv + h) * rec_stride + kRecG))[kGateBeta * C + tid];
  }
#pragma unroll
  for (int m = 0; m < NIT; ++m) {
    const int it = tid + m * CNT;
    const int which = it / PER, rem = it % PER;
    const int row = rem / (DK / EPI), c = EPI * (rem % (DK / EPI));
    *(u32x4*)((which ? sQ : sK) + row * LDK + c) = st[m];
  }

  // ---------------------------------------------------------------- products over dv
  // accumulators [dk][token]: tile t, token block i; lane (q, r) holds dk_own(t) .. +3 of
  // token 16 i + r
  f32x4 aq[NKB][4], az[NKB][4], ay[NKB][4];  // dO S^T, dR S^T, V_new dS^T, transposed
#pragma unroll
  for (int t = 0; t < NKB; ++t)
#pragma unroll
    for (int i = 0; i < 4; ++i) aq[t][i] = az[t][i] = ay[t][i] = zero4();
  // tiles (rp, j) of dO V_new^T and (rl, j) of dR V_new^T at or below the diagonal: of both
  // for j < 2 (a tile past the diagonal is not formed), of one of them for j >= 2
  const int rp = wave, rl = 3 - wave;
  const bool upper = wave >= 2;  // rp >= 2: the tiles j >= 2 are dP's, else dL's
  f32x4 tp[2], tl[2], tx[2];
#pragma unroll
  for (int j = 0; j < 2; ++j) tp[j] = tl[j] = tx[j] = zero4();
  float sds = 0.f;                     // sum of dS * S in fp32 (each element is loaded once here)
  float rv[NRI];                       // dR . v of the thread's rows, its columns
#pragma unroll
  for (int m = 0; m < NRI; ++m) rv[m] = 0.f;
  auto f4 = [](float4 x) { return f32x4{x.x, x.y, x.z, x.w}; };
  // (the barrier at the top of the first step orders the staging before every read)
#pragma unroll 1
  for (int u = 0; u < DV / 32; ++u) {
    // every barrier in this kernel orders LDS accesses only, as in the reverse scan
    lds_barrier();  // the previous step's readers are done
#pragma unroll
    for (int m = 0; m < NRI; ++m) {
      const int row = srow + m * (CNT / 8), o = row * LDR + sc4;
      put_row4(sDOh, sDOl, o, f4(pf_do[m]));
      put_row4(sDRh, sDRl, o, f4(pf_dr[m]));
      put_row4(sVNh, sVNl, o, f4(pf_vn[m]));
      // dv = diag(beta) dR, written here in whole row pieces (rows past the end dropped)
      const float4 d = pf_dr[m], v4 = to_f4(pf_v[m]);
      rv[m] += d.x * v4.x + d.y * v4.y + d.z * v4.z + d.w * v4.w;
      const float bt = sBt[row];
      const unsigned off = (unsigned)sizeof(In) * (roff + m * (CNT / 8) * (unsigned)rs + 32 * u);
      if constexpr (F32)
        __builtin_amdgcn_raw_buffer_store_b128(
            u32x4{__float_as_uint(bt * d.x), __float_as_uint(bt * d.y), __float_as_uint(bt * d.z),
                  __float_as_uint(bt * d.w)}, rDV, off, 0, 0);
      else
        __builtin_amdgcn_raw_buffer_store_b64(u32x2{pack_bf16(bt * d.x, bt * d.y), pack_bf16(bt * d.z, bt * d.w)},
                                              rDV, off, 0, 0);
    }
    Op bs[NKB];
#pragma unroll
    for (int t = 0; t < NKB; ++t) bs[t] = split8(sfr[t]);
    // The next step's loads, each issued after this step's values are consumed and
    // unconditionally (the last step reloads its own slices, unused): loaded under a branch
    // or hoisted above that use, they would need other registers than the ones the loop
    // carries, and the copies at the end of the step would wait for them.
    __builtin_amdgcn_sched_barrier(0);
    const int un = u + 1 < DV / 32 ? u + 1 : u;
    load_rows(un);
    load_state(rDS, u, dfr);  // this step's, used after the products with S
    lds_barrier();
    // the products with S, then those with dS, then the tiles: few operands live at a time
    // (all of them at once spilled accumulators, whose reloads waited for every load; so, two
    // registers are left spilled at dk = dv = 128, one at dv = 64, none at dk <= 64)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const Op ao = op_vec(sDOh, sDOl, LDR, 16 * i, 0);
      const Op ar = op_vec(sDRh, sDRl, LDR, 16 * i, 0);
      if (active) {
#pragma unroll
        for (int t = 0; t < NKB; ++t) {
          aq[t][i] = mm3<true, true>(aq[t][i], bs[t], ao);
          az[t][i] = mm3<true, true>(az[t][i], bs[t], ar);
        }
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    Op bd[NKB];
#pragma unroll
    for (int t = 0; t < NKB; ++t) {
#pragma unroll
      for (int e = 0; e < 8; ++e) sds += sfr[t][e] * dfr[t][e];
      bd[t] = split8(dfr[t]);
    }
    __builtin_amdgcn_sched_barrier(0);
    load_state(rS, un, sfr);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const Op av = op_vec(sVNh, sVNl, LDR, 16 * j, 0);
      if (active) {
#pragma unroll
        for (int t = 0; t < NKB; ++t) ay[t][j] = mm3<true, true>(ay[t][j], bd[t], av);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    const Op op = op_vec(sDOh, sDOl, LDR, 16 * rp, 0), ol = op_vec(sDRh, sDRl, LDR, 16 * rl, 0);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const Op av = op_vec(sVNh, sVNl, LDR, 16 * j, 0);
      if (j < 2) {
        if (j <= rp) tp[j] = mm3<true, true>(tp[j], op, av);
        if (j <= rl) tl[j] = mm3<true, true>(tl[j], ol, av);
      } else if (upper) {
        if (j <= rp) tx[j - 2] = mm3<true, true>(tx[j - 2], op, av);
      } else {
        if (j <= rl) tx[j - 2] = mm3<true, true>(tx[j - 2], ol, av);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  }
#pragma unroll
  for (int m = 0; m < NRI; ++m) {  // the row's 8 threads
    const float s = group_sum_dpp<8>(rv[m]);
    if ((tid & 7) == 0) sRV[srow + m * (CNT / 8)] = s;
  }
  sds = wave_sum(sds);
  if (l == 0) sRed[wave] = active ? sds : 0.f;
  lds_barrier();  // every read of the staged slices is done: the region now holds dPg and Qm

  // ---------------------------------------------------------------- rows over dk
  auto k4 = [&](const KT* m, int row, int col) { return to_f4(*(const typename Vec4<KT>::type*)(m + row * LDK + col)); };
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int row = 16 * i + lr;
    const float eg = __expf(sG[row]), el = row == C - 1 ? 1.f : __expf(sG[C - 1] - sG[row]);
    float x1 = 0.f, z = 0.f, y = 0.f;
    if (active) {
#pragma unroll
      for (int t = 0; t < NKB; ++t) {
        const float4 q4 = k4(sQ, row, dk_own(t)), kk = k4(sK, row, dk_own(t));
        const float qa[4] = {q4.x, q4.y, q4.z, q4.w}, ka[4] = {kk.x, kk.y, kk.z, kk.w};
        const float bz = sBt[row] * eg;
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          aq[t][i][v] *= eg;
          ay[t][i][v] *= el;
          x1 += qa[v] * aq[t][i][v];
          z += ka[v] * az[t][i][v];
          y += ka[v] * ay[t][i][v];
          ay[t][i][v] -= bz * az[t][i][v];  // dk so far
        }
      }
    }
    // over the lane groups, which hold the same token's other dk
    auto rows4 = [&](float s) {
      const auto a = __builtin_amdgcn_permlane16_swap(__float_as_uint(s), __float_as_uint(s), false, false);
      s = __uint_as_float(a[0]) + __uint_as_float(a[1]);
      const auto b = __builtin_amdgcn_permlane32_swap(__float_as_uint(s), __float_as_uint(s), false, false);
      return __uint_as_float(b[0]) + __uint_as_float(b[1]);
    };
    x1 = rows4(x1);
    z = rows4(z);
    y = rows4(y);
    if (lq == 0) {
      sX1[wave][row] = scale * x1;
      sZ[wave][row] = z;
      sY[wave][row] = y;
    }
  }
  // ---------------------------------------------------------------- dP and dL tiles
  // P = lower(scale Q K^T * Gamma) and Lg = strict_lower(K K^T * Gamma) at this wavefront's
  // tiles: fp32 inputs read them from the preparation kernel's matrices, bf16 inputs form
  // them (the same products summed by the same MFMA over the same dk blocks in the same
  // order).
  {
    f32x4 rowp = zero4(), rowl = zero4(), rowb = zero4();
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      f32x4 cg = zero4();
      const int col = 16 * j + lr;
      const float gc = sG[col];
      if (j <= rp) {  // uniform
        const f32x4 d4 = j < 2 ? tp[j] : tx[j - 2];
        f32x4 pp = zero4(), dpg;
        if constexpr (!F32) {
#pragma unroll
          for (int s2 = 0; s2 < DK / 32; ++s2)
            pp = mma16(frag_bf16((const bf16_t*)sQ, LDK, 16 * rp, 32 * s2),
                       frag_bf16((const bf16_t*)sK, LDK, 16 * j, 32 * s2), pp);
        }
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          const int row = 16 * rp + 4 * lq + v;
          const float e = gate_ratio(sG[row], gc);
          const float d = row >= col ? d4[v] : 0.f;
          const float x = d * (F32 ? xb[kXlpgP + row * C + col] : scale * pp[v] * e);
          rowp[v] += x;
          cg[v] += x;
          dpg[v] = d * e;                                // dPg = dP * Gamma
        }
        put_ct(sDPh, sDPl, LDB, 16 * rp, 16 * j, dpg);
      }
      if (j <= rl) {  // uniform
        const f32x4 d4 = j < 2 ? tl[j] : tx[j - 2];
        f32x4 kk = zero4(), qm;
        if constexpr (!F32) {
#pragma unroll
          for (int s2 = 0; s2 < DK / 32; ++s2)
            kk = mma16(frag_bf16((const bf16_t*)sK, LDK, 16 * rl, 32 * s2),
                       frag_bf16((const bf16_t*)sK, LDK, 16 * j, 32 * s2), kk);
        }
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          const int row = 16 * rl + 4 * lq + v;
          const float e = gate_ratio(sG[row], gc);
          const float d = row > col ? -d4[v] : 0.f;      // dL
          const float x = d * (F32 ? xb[kXlpgLg + row * C + col] : kk[v] * e);
          const float y = sBt[row] * x;                  // dL * L
          rowb[v] += x;
          rowl[v] += y;
          cg[v] += y;
          qm[v] = sBt[row] * d * e;                      // Qm = diag(beta) (dL * Gamma)
        }
        put_ct(sQMh, sQMl, LDB, 16 * rl, 16 * j, qm);
      }
      set_cols(sCol[wave], j, cg);
    }
    set_rows(sRowP, rp, rowp);
    set_rows(sRowL, rl, rowl);
    set_rows(sRowB, rl, rowb);
    // the tiles above the diagonal that complete the block pairs of row blocks 0 and 2
    if (wave < 2) put_ct(sDPh, sDPl, LDB, 32 * wave, 32 * wave + 16, zero4());
    else put_ct(sQMh, sQMl, LDB, 32 * (wave - 2), 32 * (wave - 2) + 16, zero4());
  }
  lds_barrier();

  // ---------------------------------------------------------------- dPg K, (Qm + Qm^T) K, dPg^T Q
  if (active) {
    Op ko[NKB][2], qo[NKB][2];  // K and Q columns dk_row(t, .), slots over 32 tokens
#pragma unroll
    for (int t = 0; t < NKB; ++t)
#pragma unroll
      for (int p2 = 0; p2 < 2; ++p2) {
        if constexpr (F32) {
          float x[8];
#pragma unroll
          for (int e = 0; e < 8; ++e) x[e] = sK[(32 * p2 + 8 * lq + e) * LDK + dk_row(t, lr)];
          ko[t][p2] = split8(x);
#pragma unroll
          for (int e = 0; e < 8; ++e) x[e] = sQ[(32 * p2 + 8 * lq + e) * LDK + dk_row(t, lr)];
          qo[t][p2] = split8(x);
        } else {
          // source lane s of a 16-lane group points at row s / 4 and the 4 columns of row
          // group s % 4 (see ds_read_tr)
          const int o = (32 * p2 + 8 * lq + (lr >> 2)) * LDK + dk_row(t, 4 * (lr & 3));
          const u32x2 a = ds_read_tr((const bf16_t*)sK + o), b = ds_read_tr((const bf16_t*)sK + o + 4 * LDK);
          const u32x2 c = ds_read_tr((const bf16_t*)sQ + o), d = ds_read_tr((const bf16_t*)sQ + o + 4 * LDK);
          ko[t][p2].h = ko[t][p2].l = u32x4{a[0], a[1], b[0], b[1]};
          qo[t][p2].h = qo[t][p2].l = u32x4{c[0], c[1], d[0], d[1]};
        }
      }
    // per value head rows at the input precision: the q/k finalisation sums them and
    // rounds to that precision anyway
    const long long oo = (t0 * Hv + h) * (long long)DK;
    const unsigned ob = (unsigned)(nvalid * (long long)Hv * DK * (long long)sizeof(KT));
    const auto rdq = buf_rsrc((KT*)p.dqh + oo, ob), rdk = buf_rsrc((KT*)p.dkh + oo, ob);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      f32x4 a_t[NKB];
#pragma unroll
      for (int t = 0; t < NKB; ++t) a_t[t] = zero4();
#pragma unroll
      for (int p2 = 0; p2 < 2; ++p2) {
        if (p2 <= i / 2) {  // lower triangular: rows of block i
          const Op b = op_tr(sQMh, sQMl, LDB, 16 * i, 32 * p2), d = op_tr(sDPh, sDPl, LDB, 16 * i, 32 * p2);
#pragma unroll
          for (int t = 0; t < NKB; ++t) {
            ay[t][i] = mm3<F32, true>(ay[t][i], ko[t][p2], b);
            aq[t][i] = mm3<F32, true>(aq[t][i], ko[t][p2], d);
          }
        }
        if (p2 >= i / 2) {  // transposes: upper triangular
          const Op b = op_vec(sQMh, sQMl, LDB, 16 * i, 32 * p2), d = op_vec(sDPh, sDPl, LDB, 16 * i, 32 * p2);
#pragma unroll
          for (int t = 0; t < NKB; ++t) {
            ay[t][i] = mm3<F32, true>(ay[t][i], ko[t][p2], b);
            a_t[t] = mm3<F32, true>(a_t[t], qo[t][p2], d);
          }
        }
      }
      // token 16 i + r, the lane's consecutive dk (rows past the end dropped)
      const unsigned off = (unsigned)(((16 * i + lr) * (long long)Hv * DK + dk_own(0)) * (long long)sizeof(KT));
      float xq[4 * NKB], xk[4 * NKB];
#pragma unroll
      for (int t = 0; t < NKB; ++t)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          xq[4 * t + v] = scale * aq[t][i][v];
          xk[4 * t + v] = ay[t][i][v] + scale * a_t[t][v];
        }
      store_row<KT, 4 * NKB>(rdq, off, xq);
      store_row<KT, 4 * NKB>(rdk, off, xk);
    }
  }

  // ---------------------------------------------------------------- dG, dbeta, dg
  if (wave == 0) {
    const int i = l;
    float rg = sRowP[i] + sRowL[i], rz = 0.f, ry = 0.f;
#pragma unroll
    for (int w = 0; w < CW; ++w) {
      rg += sX1[w][i] - sCol[w][i];
      rz += sZ[w][i];
      ry += sY[w][i];
    }
    const float t = -__expf(sG[i]) * rz;  // of -diag(e^G) K S in R
    float dG = rg - ry + sBt[i] * t;
    const float db = sRV[i] + sRowB[i] + t;
    const float rsum = wave_sum(ry);
    float sds = 0.f;
#pragma unroll
    for (int w = 0; w < CW; ++w) sds += sRed[w];
    if (i == C - 1) dG += rsum + __expf(sG[C - 1]) * sds;
    // dg_t = sum_{i >= t} dG_i (G = cumsum(g), deltanet.py:98)
    float x = dG;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const float y = __shfl_down(x, o);
      if (i + o < 64) x += y;
    }
    if (i < nvalid) {
      p.dg[(t0 + i) * Hv + h] = x;
      p.dbeta[(t0 + i) * Hv + h] = db;
    }
  }
}

// ============================================================================ q/k finalisation

// dk / 8 consecutive threads per (token, key head) row of dq or dk, 8 elements each: the
// sum over the key head's value heads, then (qk_l2norm) the L2-norm backward
// dx = r (dy - y (y . dy)), y = x r, r = rsqrt(sum x^2 + 1e-6) (deltanet.py:30-32; the bf16
// rounding of y is differentiated as the identity, as autodiff does for a dtype cast).
template <bool F32>
__global__ __launch_bounds__(NT) void qk_final_kernel(BwdParams p, long long rows) {
  using In = typename std::conditional<F32, float, bf16_t>::type;
  const int dk = p.dk, tpr = dk / 8, gqa = p.Hv / p.Hk;
  const long long gid = (long long)blockIdx.x * NT + threadIdx.x;
  const long long rid = gid / tpr;
  const int c8 = 8 * (int)(gid % tpr);
  if (rid >= 2 * rows) return;  // whole rows drop out together (tpr divides 64)
  const int which = (int)(rid / rows);
  const long long row = rid % rows;
  const long long token = row / p.Hk;
  const int hk = (int)(row % p.Hk);
  const In* src = (const In*)(which ? p.dkh : p.dqh) + (token * p.Hv + (long long)hk * gqa) * dk + c8;
  float d[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f}, x[8];
  for (int g = 0; g < gqa; ++g) {
    float w[8];
    load8v(src + (long long)g * dk, w);
#pragma unroll
    for (int e = 0; e < 8; ++e) d[e] += w[e];
  }
  load8v((const In*)(which ? p.k : p.q) + row * dk + c8, x);
  if (p.qk_l2norm) {
    float ss = 0.f;
#pragma unroll
    for (int e = 0; e < 8; ++e) ss += x[e] * x[e];
    for (int o = 1; o < tpr; o <<= 1) ss += __shfl_xor(ss, o);
    const float r = rsqrtf(ss + 1e-6f);
    float yd = 0.f;
#pragma unroll
    for (int e = 0; e < 8; ++e) yd += x[e] * r * d[e];
    for (int o = 1; o < tpr; o <<= 1) yd += __shfl_xor(yd, o);
#pragma unroll
    for (int e = 0; e < 8; ++e) d[e] = r * (d[e] - x[e] * r * yd);
  }
  In* out = (In*)(which ? p.dk_out : p.dq) + row * dk + c8;
  if constexpr (F32) {
    *(float4*)out = float4{d[0], d[1], d[2], d[3]};
    *(float4*)(out + 4) = float4{d[4], d[5], d[6], d[7]};
  } else {
    *(u32x4*)out = pack8(d);
  }
}

// p.nb (64-column blocks) is replaced by the scan's own count in a copy of the parameters
template <int DK, bool F32, int NWC>
hipError_t launch_rscan(const BwdParams& p, hipStream_t stream) {
  BwdParams q = p;
  q.nb = p.DV / (16 * NWC);
  hipLaunchKernelGGL((rscan_kernel<DK, F32, NWC>), dim3((unsigned)(q.N * q.Hv * q.nb)),
                     dim3(F32 ? NT : 64 * NWC + NT), 0, stream, q);
  return hipGetLastError();
}

template <int DK, bool F32>
hipError_t launch_bwd_dk(const BwdParams& p, hipStream_t stream) {
  hipError_t e;
  if constexpr (F32) {
    e = launch_rscan<DK, F32, 4>(p, stream);
  } else {
    const int tiles = scan_column_tiles(p.N, p.Hv, p.DV, p.dk, p.cu_seqlens != nullptr, true);
    e = tiles == 1   ? launch_rscan<DK, F32, 1>(p, stream)
        : tiles == 2 ? launch_rscan<DK, F32, 2>(p, stream)
                     : launch_rscan<DK, F32, 4>(p, stream);
  }
  if (e != hipSuccess) return e;
  const unsigned grid = (unsigned)((long long)p.n_rec * p.Hv);
  if (grid > 0) {
    if (p.DV == 128)
      hipLaunchKernelGGL((cgrad_kernel<DK, 128, F32>), dim3(grid), dim3(CNT), 0, stream, p);
    else
      hipLaunchKernelGGL((cgrad_kernel<DK, 64, F32>), dim3(grid), dim3(CNT), 0, stream, p);
    e = hipGetLastError();
    if (e != hipSuccess) return e;
  }
  const long long rows = (long long)p.T * (p.cu_seqlens ? 1 : p.N) * p.Hk;
  if (rows > 0) {
    const long long threads = 2 * rows * (p.dk / 8);
    const unsigned g2 = (unsigned)((threads + NT - 1) / NT);
    hipLaunchKernelGGL((qk_final_kernel<F32>), dim3(g2), dim3(NT), 0, stream, p, rows);
    e = hipGetLastError();
  }
  return e;
}

}  // namespace

bool bwd_dims_supported(int dk, int dv, bool f32_inputs) {
  if (dv != 64 && dv != 128) return false;
  // fp32 inputs at dk = 128 would need 185 KiB of LDS in the gradient kernel
  if (f32_inputs) return dk == 32 || dk == 64;
  return dk == 64 || dk == 128;
}

hipError_t launch_bwd(const BwdParams& p, hipStream_t stream) {
  if (p.in_f32) {
    if (p.dk == 64) return launch_bwd_dk<64, true>(p, stream);
    if (p.dk == 32) return launch_bwd_dk<32, true>(p, stream);
    return hipErrorInvalidValue;
  }
  if (p.dk == 128) return launch_bwd_dk<128, false>(p, stream);
  if (p.dk == 64) return launch_bwd_dk<64, false>(p, stream);
  return hipErrorInvalidValue;
}

}  // namespace omx
