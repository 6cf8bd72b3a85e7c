// Causal flash attention for the GPT block, forward and backward, on CDNA4
// matrix cores (v_mfma_f32_32x32x16_{bf16,f16}).  Any head_dim that is a
// multiple of 8 up to 128 runs on the 64-, 96- or 128-wide kernels with the
// extra head-dim columns loaded as zeros and never stored; any sequence
// length runs on whole 128-row blocks whose rows past the end load as zeros
// (the causal mask already hides keys past every real query) and are never
// stored.
//
// Semantics: O = softmax(Q K^T / sqrt(hn) + causal -inf) V per (batch, head),
// i.e. F.scaled_dot_product_attention(q, k, v, is_causal=True) as called by
// eth/runtime/megatron/model/flex_ops.py:66-96 (ParallelFlashAtten,
// :1401-1426).  Q, K, V, O and their gradients are addressed in place through
// (row, batch, head) strides, so the [s, b, np, 3*hn] output of the QKV GEMM
// is read without the split/permute copies and dQ/dK/dV are written straight
// into the [s, b, np, 3*hn] gradient the QKV backward consumes.
//
// Layout trick.  Scores are computed transposed, S^T = K Q^T, so that each
// lane owns one query (MFMA column) and 32 of the 64 keys of a block sit in
// its registers: row max / row sum need one cross-lane exchange (lane ^ 32),
// and the per-query softmax statistics are per-lane scalars.  K rows are
// read from LDS with bits 2 and 3 of the row index swapped, which makes the
// MFMA result layout of S^T equal to the operand layout of P^T in
// O^T = V^T P^T, so P never leaves registers.  The dK/dV kernel uses the
// mirror image (S = Q K^T, lane = key, query rows swizzled) and computes S
// and P once for both gradients (head dim 128 in pairs of waves that hand P
// over through LDS); dQ has its own kernel (recomputing P), so no atomics are needed and
// results are deterministic.  The dQ kernel runs first and also writes
// delta = rowsum(dO * O), which the dK/dV kernel reads.
//
// Tiles load directly from global memory into swizzled LDS images (fixed
// per-thread offsets, a scalar row advance).  Operands that an MFMA needs
// transposed (V for O^T = V^T P^T, K for dQ^T = K^T dS^T, Q and dO for dK and
// dV) are read from the same images with ds_read_b64_tr_b16.  Softmax runs in
// fp32 base-2 (exp2) with the scale folded.
//
// Forward / backward alone, against kernels that staged the 64- and 96-wide
// tiles through registers into padded copies (us): 4096 x 2 x 16 heads of 64
// 97 / 321 -> 90 / 262, 1500 x 2 x 32 of 80 49 / 175 -> 47 / 142, 2048 x 4 x 16
// of 128 85 / 289 -> 84 / 272, 2048 x 1 x 16 of 128 50 / 124 -> 41 / 114.
// Bound by a wave's own VALU work (5.5 instructions per forward MFMA, one of
// them an exponential), which runs in series with its MFMAs.
#include <type_traits>

#include "common.h"

namespace eth {

typedef __bf16 a_bf16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 a_f16x8 __attribute__((ext_vector_type(8)));
typedef float a_f32x16 __attribute__((ext_vector_type(16)));
typedef uint32_t a_u32x4 __attribute__((ext_vector_type(4)));

template <bool FP16>
__device__ __forceinline__ a_f32x16 mma(const uint4& a, const uint4& b, const a_f32x16& c) {
  if constexpr (FP16)
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(a_f16x8, a), __builtin_bit_cast(a_f16x8, b),
                                                  c, 0, 0, 0);
  else
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(a_bf16x8, a),
                                                   __builtin_bit_cast(a_bf16x8, b), c, 0, 0, 0);
}

template <bool FP16>
__device__ __forceinline__ float to_f(uint16_t v) {
  return FP16 ? h2f_bits(v) : bf2f(v);
}
template <bool FP16>
__device__ __forceinline__ uint16_t from_f(float v) {
  return FP16 ? f2h_bits(v) : f2bf(v);
}
template <bool FP16>
__device__ __forceinline__ uint32_t pack2(float a, float b) {
  if constexpr (FP16)
    return (uint32_t)f2h_bits(a) | ((uint32_t)f2h_bits(b) << 16);
  else
    return f2bf_pair(a, b);
}
__device__ __forceinline__ float fast_exp2(float x) { return __builtin_amdgcn_exp2f(x); }
// s_waitcnt vmcnt(0) (expcnt, lgkmcnt unconstrained) as the builtin, so the
// compiler's own wait-count tracking knows that no vector load is pending
__device__ __forceinline__ void vm_wait_all() { __builtin_amdgcn_s_waitcnt(0x0F70); }
// Between a wave's LDS accesses of one type and its accesses of another to the
// same memory, all of them its own: its LDS operations execute in order, but
// the compiler may take float, 16-bit and 16-byte accesses to be apart and
// move one past the other.  The clobber holds them in place.
__device__ __forceinline__ void wave_lds_fence() { asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); }
// 8 fp32 -> one 16-byte MFMA operand
template <bool FP16>
__device__ __forceinline__ uint4 pack8(const float* v) {
  return make_uint4(pack2<FP16>(v[0], v[1]), pack2<FP16>(v[2], v[3]), pack2<FP16>(v[4], v[5]),
                    pack2<FP16>(v[6], v[7]));
}

__device__ __forceinline__ int swz(int r) {  // swap bits 2 and 3
  return (r & ~12) | ((r & 4) << 1) | ((r & 8) >> 1);
}
// index (within a 32-row MFMA tile) held by accumulator register r of a lane
// in half h, when the operand rows were swizzled
__device__ __forceinline__ int swz_row(int r, int h) { return (r < 8 ? 0 : 16) + h * 8 + (r & 7); }
// natural accumulator row of register r for half h
__device__ __forceinline__ int acc_row(int r, int h) { return (r >> 2) * 8 + h * 4 + (r & 3); }

struct AttnTensor {
  const uint16_t* p;
  int64_t ss, sb, sh;  // strides of sequence, batch, head (elements); dim contiguous
  uint32_t bytes;      // extent from p (buffer-load range)
};
struct AttnOut {
  uint16_t* p;
  int64_t ss, sb, sh;
};

struct AttnArgs {
  AttnTensor q, k, v, o, dout;
  AttnOut out, dq, dk, dv;
  float* lse;    // [B*H, S] log2-domain: m2 + log2(l)
  float* delta;  // [B*H, S] rowsum(dO * O)
  int B, H, S;
  int hd;  // head dim (<= the kernel's D; columns hd..D-1 are zero padding)
  float scale_log2;  // log2(e) / sqrt(hn)
  float scale;       // 1 / sqrt(hn)
};

constexpr int kAttnThreads = 256;
constexpr float kRescaleLog2 = 8.0f;  // forward: tolerated growth of the running max (log2 units)
constexpr int kBQ = 128;   // forward / dQ: queries per workgroup (4 waves x 32)
constexpr int kBKV = 64;   // forward / dQ: keys per step
constexpr int kBKV2 = 128; // dK/dV: keys per workgroup (4 waves x 32)
constexpr int kBQ2 = 64;   // dK/dV: queries per step
constexpr int32_t kAttnOob = (int32_t)0x80000000u;  // buffer offset past any tensor: loads read zeros
// 16 bytes of a row at column `col` of a strided tensor; with PAD, zeros
// past the sequence or the head dim (without, every row and column is real)
template <bool PAD>
__device__ __forceinline__ uint4 load_row16(const uint16_t* row, bool in_seq, int col, int hd) {
  if constexpr (PAD)
    return in_seq && col < hd ? *reinterpret_cast<const uint4*>(row + col) : make_uint4(0u, 0u, 0u, 0u);
  else
    return *reinterpret_cast<const uint4*>(row + col);
}

__device__ __forceinline__ const uint16_t* row_ptr(const AttnTensor& t, int s, int b, int h) {
  return t.p + (int64_t)s * t.ss + (int64_t)b * t.sb + (int64_t)h * t.sh;
}
__device__ __forceinline__ uint16_t* row_ptr(const AttnOut& t, int s, int b, int h) {
  return t.p + (int64_t)s * t.ss + (int64_t)b * t.sb + (int64_t)h * t.sh;
}

typedef __amdgpu_buffer_rsrc_t a_rsrc_t;
typedef short a_s16x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) a_s16x4 a_lds_s16x4;
typedef uint32_t a_u32x2 __attribute__((ext_vector_type(2)));
// ------------------------------------------------------- images in LDS --
// A 64-row block of a tensor lies in LDS as it is in memory, except that chunk
// c (8 columns, 16 bytes) of row r is at c ^ img_swz(r): the row reads of an
// MFMA operand (16 lanes on 16 rows, one chunk) and the transposing
// ds_read_b64_tr_b16 reads (4 rows x 64 bytes per 32 lanes) then both hit
// distinct banks, so one image serves both.  It is filled by direct
// global->LDS loads a whole block ahead: no register staging, no copy phase.
// Each image is an array of its own, so the compiler can tell the loads into
// one from the reads of another and puts no wait between them.
__device__ __forceinline__ int xsw(int r) { return ((r & 3) << 2) | ((r >> 2) & 3); }
template <int D>
__device__ __forceinline__ int img_swz(int r) {
  if constexpr (D == 128)
    return xsw(r);
  else if constexpr (D == 64)  // 128-byte rows: bit 0 of r picks the half of the banks
    return (((r >> 1) & 1) << 2) | (((r >> 3) & 1) << 1) | ((r >> 2) & 1);
  else  // 192-byte rows start 64 bytes apart in the banks: within groups of four chunks
    return (r >> 2) & 3;
}
// the four waves' direct loads: unit u (16 bytes) of the image holds row
// u / CPR, chunk (u % CPR) ^ img_swz(row).  With PAD, rows at or past `seq`
// and columns at or past `hd` read zeros.
template <int D, bool PAD>
struct ImgCopy {
  static constexpr int CPR = D / 8;  // 16-byte chunks per row
  static constexpr int PW = D / 32;  // 1 KB pieces per wave
  int32_t off[PW];
  int row[PW];
  a_rsrc_t rs;
  int32_t row_bytes;
  int w, seq;
  __device__ __forceinline__ void init(const AttnTensor& t, int b, int h, int hd, int s, int wave, int lane) {
    rs = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(t.p), (short)0, (int)t.bytes, 0x00020000);
    row_bytes = (int32_t)(t.ss * 2);
    w = wave;
    seq = s;
#pragma unroll
    for (int j = 0; j < PW; ++j) {
      const int u = (w * PW + j) * 64 + lane;
      const int r = u / CPR, c = (u % CPR) ^ img_swz<D>(r);
      row[j] = r;
      off[j] = !PAD || c * 8 < hd
                   ? (int32_t)(((int64_t)b * t.sb + (int64_t)h * t.sh + (int64_t)r * t.ss + c * 8) * 2)
                   : kAttnOob;
    }
  }
  __device__ __forceinline__ void issue(uint16_t* S, int r0) const {
#pragma unroll
    for (int j = 0; j < PW; ++j) {
      const int32_t o = !PAD || r0 + row[j] < seq ? off[j] : kAttnOob;
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (__attribute__((address_space(3))) void*)(S + (w * PW + j) * 512),
                                               16, o, r0 * row_bytes, 0, 0);
    }
  }
};
// Row reads: row t*32 + swz(lane%32) (the swizzled order that makes the
// result's layout the operand layout of the next product), chunk 2*ks + lane/32:
// element offset of k-step ks within a 32-row tile.
template <int D>
__device__ __forceinline__ int img_row_off(int lane, int ks) {
  const int r = swz(lane & 31);
  return r * D + (((2 * ks + (lane >> 5)) ^ img_swz<D>(r)) << 3);
}
// Transposing reads: rows kk*16 + 8*(l/32) + (l%16)/4 (+4 for the second
// read, hi), columns ct*32 + 16*((l/16)%2) + 4*(l%4): element offset within
// the 16-row group kk.
template <int D>
__device__ __forceinline__ int img_tr_off(int lane, int ct, int hi) {
  const int r = 8 * (lane >> 5) + ((lane & 15) >> 2) + 4 * hi;
  const int c = 4 * ct + 2 * ((lane >> 4) & 1) + ((lane >> 1) & 1);
  return r * D + ((c ^ img_swz<D>(r)) << 3) + (lane & 1) * 4;
}
__device__ __forceinline__ uint4 img_tr(const uint16_t* p, int lo_off, int hi_off) {
  const a_u32x2 lo = __builtin_bit_cast(a_u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((a_lds_s16x4*)(p + lo_off)));
  const a_u32x2 hi = __builtin_bit_cast(a_u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((a_lds_s16x4*)(p + hi_off)));
  return make_uint4(lo.x, lo.y, hi.x, hi.y);
}

// ------------------------------------------------------------------ forward --
// 4 waves x 32 queries; K/V blocks of 64 keys in double-buffered images, one
// barrier per block; two workgroups per CU, so one wave's softmax overlaps
// another's MFMAs.
//
// G = 2: two such groups of waves in a workgroup take alternate key blocks of
// the same queries, each with images of its own, and the first adds the
// second's sums through LDS at the end.  A query block is a chain of up to
// seq / 64 steps, so a grid that leaves half of the CUs' wave slots empty
// takes as long as its longest chain: this halves it (attn_groups).
static_assert(kBQ % (2 * kBKV) == 0, "both groups take the same number of key blocks");
template <int D, bool FP16, bool PAD, int G>
__global__ void __launch_bounds__(G * kAttnThreads, 2) attn_fwd_kernel(AttnArgs a) {
  constexpr int KS = D / 16;  // k-steps over the head dim
  constexpr int DT = D / 32;  // 32-row tiles over the head dim
  constexpr int IMG = kBKV * D;  // elements of one image
  __shared__ __attribute__((aligned(16))) uint16_t K0[G * IMG];
  __shared__ __attribute__((aligned(16))) uint16_t K1[G * IMG];
  __shared__ __attribute__((aligned(16))) uint16_t V0[G * IMG];
  __shared__ __attribute__((aligned(16))) uint16_t V1[G * IMG];

  const int BH = a.B * a.H, nqb = (a.S + kBQ - 1) / kBQ;
  const int bh = blockIdx.x % BH, qb = nqb - 1 - blockIdx.x / BH;
  const int b = bh / a.H, h = bh % a.H;
  const int lane = threadIdx.x & 63, hl = lane >> 5;
  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);  // wave-uniform
  const int w = wid & 3, grp = G == 1 ? 0 : wid >> 2;
  const int q0 = qb * kBQ + w * 32;
  const int q = q0 + (lane & 31);
  const float sl2 = a.scale_log2;

  ImgCopy<D, PAD> kc, vc;
  kc.init(a.k, b, h, a.hd, a.S, w, lane);
  vc.init(a.v, b, h, a.hd, a.S, w, lane);
  const int nkv = (qb * kBQ + kBQ) / kBKV / G;  // a group's blocks up to the diagonal
  kc.issue(K0 + grp * IMG, grp * kBKV);
  vc.issue(V0 + grp * IMG, grp * kBKV);

  uint4 qf[KS];
  {
    const uint16_t* qp = row_ptr(a.q, q, b, h);
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) qf[ks] = load_row16<PAD>(qp, q < a.S, ks * 16 + hl * 8, a.hd);
  }
  a_f32x16 o[DT];
#pragma unroll
  for (int t = 0; t < DT; ++t)
#pragma unroll
    for (int r = 0; r < 16; ++r) o[t][r] = 0.f;
  float m = -1e30f, l = 0.f;  // running max (log2 units) and sum for query q

  int aoff[KS], toff[DT][2];
#pragma unroll
  for (int ks = 0; ks < KS; ++ks) aoff[ks] = img_row_off<D>(lane, ks);
#pragma unroll
  for (int dt = 0; dt < DT; ++dt)
#pragma unroll
    for (int hi = 0; hi < 2; ++hi) toff[dt][hi] = img_tr_off<D>(lane, dt, hi);
  vm_wait_all();
  __syncthreads();

  auto block = [&](int j, auto cur_c) __attribute__((always_inline)) {
    constexpr int cur = decltype(cur_c)::value;
    const int kv0 = (j * G + grp) * kBKV;
    if (j + 1 < nkv) {  // the group's next block, a block ahead
      kc.issue((cur ? K0 : K1) + grp * IMG, kv0 + G * kBKV);
      vc.issue((cur ? V0 : V1) + grp * IMG, kv0 + G * kBKV);
    }
    if (kv0 <= q0 + 31) {  // wave has at least one unmasked key in the block
      const uint16_t* ki = (cur ? K1 : K0) + grp * IMG;
      const uint16_t* vi = (cur ? V1 : V0) + grp * IMG;
      // S^T = K Q^T (raw scores; lane = query, registers = 32 of the keys)
      a_f32x16 sc[2];
      // all K fragments of the first 32-key tile are read before its MFMAs,
      // each register refilled with the second tile's fragment right after
      // its MFMA issues (order pinned: left alone, the compiler reads each
      // fragment one or two MFMAs before its use and waits on the LDS latency)
      {
        uint4 kr[KS];
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) kr[ks] = *reinterpret_cast<const uint4*>(ki + aoff[ks]);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
          sc[0] = mma<FP16>(kr[ks], qf[ks], ks == 0 ? a_f32x16{} : sc[0]);
          __builtin_amdgcn_sched_barrier(0);
          kr[ks] = *reinterpret_cast<const uint4*>(ki + 32 * D + aoff[ks]);
          __builtin_amdgcn_sched_barrier(0);
        }
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) sc[1] = mma<FP16>(kr[ks], qf[ks], ks == 0 ? a_f32x16{} : sc[1]);
      }
      if (kv0 + kBKV - 1 > q0) {  // diagonal block: mask keys after the query
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
          for (int r = 0; r < 16; ++r)
            if (kv0 + t * 32 + swz_row(r, hl) > q) sc[t][r] = -1e30f;
      }
      float mx = sc[0][0];
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int r = 0; r < 16; ++r) mx = fmaxf(mx, sc[t][r]);
      mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
      const float mnew = fmaxf(m, mx * sl2);
      // m is the exponent offset, kept within kRescaleLog2 below the running
      // max: O and l are rescaled only when some row's max grew past that,
      // so p = exp2(s - m) stays <= 2^kRescaleLog2 (exact in fp32, the same
      // relative precision in 16 bits) and most blocks skip the rescale;
      // O / l and lse = m + log2(l) do not depend on the offset
      if (__any(mnew > m + kRescaleLog2)) {
        const float alpha = fast_exp2(m - mnew);
        l *= alpha;
#pragma unroll
        for (int t = 0; t < DT; ++t)
#pragma unroll
          for (int r = 0; r < 16; ++r) o[t][r] *= alpha;
        m = mnew;
      }
      float rs = 0.f;
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const float p = fast_exp2(__builtin_fmaf(sc[t][r], sl2, -m));
          sc[t][r] = p;
          rs += p;
        }
      l += rs;
      // O^T += V^T P^T over the 64 keys (4 k-steps of 16)
#pragma unroll
      for (int kk = 0; kk < 4; ++kk) {
        const int t = kk >> 1, e0 = (kk & 1) * 8;
        const uint4 pb = make_uint4(pack2<FP16>(sc[t][e0 + 0], sc[t][e0 + 1]), pack2<FP16>(sc[t][e0 + 2], sc[t][e0 + 3]),
                                    pack2<FP16>(sc[t][e0 + 4], sc[t][e0 + 5]), pack2<FP16>(sc[t][e0 + 6], sc[t][e0 + 7]));
        const uint16_t* vp = vi + kk * 16 * D;
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) o[dt] = mma<FP16>(img_tr(vp, toff[dt][0], toff[dt][1]), pb, o[dt]);
      }
    }
    vm_wait_all();  // the next block's rows have landed
    __syncthreads();  // this block's images free, the next block's visible
  };
  int j = 0;
  for (; j + 1 < nkv; j += 2) {
    block(j, std::integral_constant<int, 0>{});
    block(j + 1, std::integral_constant<int, 1>{});
  }
  if (j < nkv) block(j, std::integral_constant<int, 0>{});
  l += __shfl_xor(l, 32, 64);
  if constexpr (G == 2) {
    // (the images are free: every group passed the last block's barrier)
    float4* so = reinterpret_cast<float4*>(w < 2 ? K0 : K1) + (w & 1) * (DT * 4 * 64) + lane;
    float2* sml = reinterpret_cast<float2*>(V0) + w * 64 + lane;
    if (grp == 1) {
#pragma unroll
      for (int t = 0; t < DT; ++t)
#pragma unroll
        for (int g = 0; g < 4; ++g)
          so[(t * 4 + g) * 64] = make_float4(o[t][g * 4], o[t][g * 4 + 1], o[t][g * 4 + 2], o[t][g * 4 + 3]);
      *sml = make_float2(m, l);
    }
    __syncthreads();
    if (grp == 1) return;
    const float2 ml = *sml;
    const float mn = fmaxf(m, ml.x), f0 = fast_exp2(m - mn), f1 = fast_exp2(ml.x - mn);
    m = mn;
    l = l * f0 + ml.y * f1;
#pragma unroll
    for (int t = 0; t < DT; ++t)
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const float4 u = so[(t * 4 + g) * 64];
        o[t][g * 4 + 0] = o[t][g * 4 + 0] * f0 + u.x * f1;
        o[t][g * 4 + 1] = o[t][g * 4 + 1] * f0 + u.y * f1;
        o[t][g * 4 + 2] = o[t][g * 4 + 2] * f0 + u.z * f1;
        o[t][g * 4 + 3] = o[t][g * 4 + 3] * f0 + u.w * f1;
      }
  }
  if (PAD && q >= a.S) return;  // a padding row of the last query block
  const float inv = 1.0f / l;
  uint16_t* op = row_ptr(a.out, q, b, h);
#pragma unroll
  for (int t = 0; t < DT; ++t)
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      if (PAD && t * 32 + g * 8 >= a.hd) continue;  // hd % 8 == 0: whole 8-column groups
      uint2 v;
      v.x = pack2<FP16>(o[t][g * 4 + 0] * inv, o[t][g * 4 + 1] * inv);
      v.y = pack2<FP16>(o[t][g * 4 + 2] * inv, o[t][g * 4 + 3] * inv);
      *reinterpret_cast<uint2*>(op + t * 32 + g * 8 + hl * 4) = v;
    }
  if (hl == 0) a.lse[(int64_t)bh * a.S + q] = m + log2f(l);
}

// ------------------------------ backward: dK, dV paired, head_dim 128 --
// Eight waves: wave w < 4 (the dV wave) and wave w + 4 (the dK wave) own the
// same 32 keys and share a SIMD.  In step m (64 queries) the dV wave computes
// S(m) = Q K^T and P(m), hands P (fp32) over through LDS and adds P(m)^T dO(m)
// into dV, while the dK wave first finishes step m-1 -- reads P(m-1), forms
// dS = P (dP - delta) and adds dS^T Q(m-1) into dK -- and then computes
// dP(m) - delta.  S and P are computed once, each step has one barrier, and
// one wave's exponentials or dS arithmetic fall between the other wave's
// MFMAs.  S is computed with lane = key (the mirror image of the forward's
// layout, query rows swizzled), so P and dS are already the A operands of
// dV += P^T dO and dK += dS^T Q.  (At this width the accumulators of both
// gradients and their operands do not fit one wave's registers; narrower
// heads take attn_bwd_dkdv_kernel.)
//
// Step m reads Q(m-1), Q(m) and dO(m), and the rows of step m+1 load directly
// into idle images: three Q images, two dO images and two P buffers (145 KB
// in all).  dP's accumulator starts at -delta.
template <bool FP16, bool PAD>
__global__ void __launch_bounds__(2 * kAttnThreads, 1) attn_bwd_dkdv_x128_kernel(AttnArgs a) {
  constexpr int D = 128, KS = D / 16, DT = D / 32;
  constexpr int IMG = kBQ2 * D;  // elements of one image
  __shared__ __attribute__((aligned(16))) uint16_t Qx[3 * IMG];
  __shared__ __attribute__((aligned(16))) uint16_t O0[IMG];
  __shared__ __attribute__((aligned(16))) uint16_t O1[IMG];
  __shared__ a_u32x4 Ps[2][4][2][4][64];
  __shared__ __attribute__((aligned(16))) float lse_s[2][kBQ2];
  __shared__ __attribute__((aligned(16))) float del_s[2][kBQ2];

  const int BH = a.B * a.H;
  const int bh = blockIdx.x % BH, kb = blockIdx.x / BH;
  const int b = bh / a.H, h = bh % a.H;
  const int lane = threadIdx.x & 63, hl = lane >> 5;
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);  // wave-uniform
  const int w = wv & 3;
  const bool dkw = wv >= 4;  // the dK wave of its pair
  const int rt = threadIdx.x & (kAttnThreads - 1);
  const int k0 = kb * kBKV2 + w * 32;
  const int key = k0 + (lane & 31);

  // B operands of the first product: K rows (S = Q K^T) in the dV wave, V
  // rows (dP = dO V^T) in the dK wave
  uint4 kf[KS];
  {
    const uint16_t* kp = row_ptr(dkw ? a.v : a.k, key, b, h);
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) kf[ks] = load_row16<PAD>(kp, key < a.S, ks * 16 + hl * 8, a.hd);
  }
  a_f32x16 acc[DT];  // dV in the dV wave, dK in the dK wave
#pragma unroll
  for (int t = 0; t < DT; ++t)
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[t][r] = 0.f;

  // direct loads (the dV waves move Q, the dK waves dO): lane l of piece j
  // (4 per wave, 16 per image) fills unit (w*4 + j)*64 + l, i.e. image row
  // u / 16, position u % 16
  const AttnTensor& src = dkw ? a.dout : a.q;
  const a_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(src.p), (short)0, (int)src.bytes,
                                                        0x00020000);
  const int32_t row_bytes = (int32_t)(src.ss * 2);
  int32_t doff[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int u = (w * 4 + j) * 64 + lane;
    const int r = u >> 4, c = (u & 15) ^ xsw(r);
    doff[j] = c * 8 < a.hd ? (int32_t)(((int64_t)b * src.sb + (int64_t)h * src.sh + (int64_t)r * src.ss + c * 8) * 2)
                           : kAttnOob;
  }
  auto issue = [&](uint16_t* img, int r0) __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int32_t o = !PAD || r0 + (w * 4 + j) * 4 + (lane >> 4) < a.S ? doff[j] : kAttnOob;
      __builtin_amdgcn_raw_ptr_buffer_load_lds(
          rs, (__attribute__((address_space(3))) void*)(img + (w * 4 + j) * 512), 16, o,
          r0 * row_bytes, 0, 0);
    }
  };
  int aoff[KS], toff[DT][2];
#pragma unroll
  for (int ks = 0; ks < KS; ++ks) aoff[ks] = img_row_off<D>(lane, ks);
#pragma unroll
  for (int d2 = 0; d2 < DT; ++d2)
#pragma unroll
    for (int hi = 0; hi < 2; ++hi) toff[d2][hi] = img_tr_off<D>(lane, d2, hi);
  auto bfrag = [&](const uint16_t* img, int kk, int d2) __attribute__((always_inline)) {
    return img_tr(img + kk * 16 * D, toff[d2][0], toff[d2][1]);
  };
  // acc += X^T B over a step's 64 queries: X (P or dS, one 32-query tile
  // per t) as the A operand, B from the transposing reads of `img`.  Four
  // B fragments in flight, each refilled with the next k-step's fragment of
  // its head-dim tile right after its MFMA issues (order pinned: the
  // scheduler otherwise hoists every read and runs out of registers)
  // With `pbuf` (the dK wave), tile t's X is first formed as dS = P (dP -
  // delta) from P in `pbuf`, one tile at a time.
  auto second = [&](a_f32x16 (&x)[2], const uint16_t* img, const a_u32x4 (*pbuf)[2][4][64])
                    __attribute__((always_inline)) {
    uint4 fb[DT];
#pragma unroll
    for (int d2 = 0; d2 < DT; ++d2) fb[d2] = bfrag(img, 0, d2);
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      if (pbuf) {
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          const a_u32x4 pv = pbuf[w][t][g][lane];
#pragma unroll
          for (int e = 0; e < 4; ++e) x[t][4 * g + e] = __uint_as_float(pv[e]) * x[t][4 * g + e];
        }
      }
#pragma unroll
      for (int k2 = 0; k2 < 2; ++k2) {
        const int kk = t * 2 + k2, e0 = k2 * 8;
        const uint4 pa = make_uint4(pack2<FP16>(x[t][e0 + 0], x[t][e0 + 1]), pack2<FP16>(x[t][e0 + 2], x[t][e0 + 3]),
                                    pack2<FP16>(x[t][e0 + 4], x[t][e0 + 5]), pack2<FP16>(x[t][e0 + 6], x[t][e0 + 7]));
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int d2 = 0; d2 < DT; ++d2) {
          acc[d2] = mma<FP16>(pa, fb[d2], acc[d2]);
          __builtin_amdgcn_sched_barrier(0);
          if (kk < 3) fb[d2] = bfrag(img, kk + 1, d2);
          __builtin_amdgcn_sched_barrier(0);
        }
      }
    }
  };
  // x = (rows of img) kf^T over the 64 queries of a step: S (dV wave) or
  // dP (dK wave), query index of register r of tile t = t*32 + swz_row(r, hl).
  // A rolling window of four A fragments, pinned like the B fragments
  // x starts at `x0(t)` (zero, or the per-query -delta of the dK wave)
  auto first_product = [&](a_f32x16 (&x)[2], const uint16_t* img, auto x0) __attribute__((always_inline)) {
    auto afrag = [&](int i) __attribute__((always_inline)) {  // fragment i = t*KS + ks
      return *reinterpret_cast<const uint4*>(img + (i / KS) * 32 * D + aoff[i % KS]);
    };
    uint4 fa[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) fa[i] = afrag(i);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) {
        const int i = t * KS + ks;
        x[t] = mma<FP16>(fa[i & 3], kf[ks], ks == 0 ? x0(t) : x[t]);
        __builtin_amdgcn_sched_barrier(0);
        if (i + 4 < 2 * KS) fa[i & 3] = afrag(i + 4);
        __builtin_amdgcn_sched_barrier(0);
      }
  };

  const int first = (kb * kBKV2) / kBQ2, nq = (a.S + kBQ2 - 1) / kBQ2, n = nq - first;
  auto stat = [&](int qs) __attribute__((always_inline)) {
    const bool real = !PAD || qs + rt < a.S;
    const int64_t i = (int64_t)bh * a.S + qs + rt;
    return dkw ? (real ? a.delta[i] : 0.f) : (real ? a.lse[i] : 1e30f);
  };
  // (delta is negated here: at the load, the use would wait for the step's
  // direct loads too)
  auto stat_store = [&](int p, float v) __attribute__((always_inline)) {
    if (dkw)
      del_s[p][rt] = -v;
    else
      lse_s[p][rt] = v;
  };
  float stat_n = 0.f;
  issue(dkw ? O0 : Qx, first * kBQ2);
  if (rt < kBQ2) stat_n = stat(first * kBQ2);
  vm_wait_all();
  if (rt < kBQ2) stat_store(0, stat_n);
  __syncthreads();

  a_f32x16 x[2];  // S then P (dV wave); dP - delta, then dS (dK wave)
  // step j = m - first (Q image j % 3; dO image, P buffer and statistics
  // j % 2 = P, a template constant)
  auto step = [&](int j, int qslot, auto par_c, auto role_c) __attribute__((always_inline)) {
    constexpr int P = decltype(par_c)::value;
    constexpr bool DKW = decltype(role_c)::value;  // the role, a constant here
    const int m = first + j, qs0 = m * kBQ2;
    const int qnext = qslot == 2 ? 0 : qslot + 1, qprev = qslot == 0 ? 2 : qslot - 1;
    // the next step's rows into idle images; the dV waves issue theirs behind
    // their reads of this step's Q (one array holds the three Q images, so
    // the compiler waits for loads in flight to it before a read)
    auto next = [&]() __attribute__((always_inline)) {
      if (j + 1 < n) {
        issue(DKW ? (P ? O0 : O1) : Qx + qnext * IMG, qs0 + kBQ2);
        if (rt < kBQ2) stat_n = stat(qs0 + kBQ2);
      }
    };
    if constexpr (DKW) next();
    // a pair whose keys all follow every query of a step skips its work
    const bool active = qs0 + kBQ2 - 1 >= k0;
    const bool active_prev = j > 0 && qs0 - 1 >= k0;
    // the sub-products are fenced from each other: the scheduler otherwise
    // hoists every fragment read of the next product above the current
    // one and runs out of registers
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (!DKW) {
      if (active) {
        first_product(x, Qx + qslot * IMG, [](int) { return a_f32x16{}; });
      }
      __builtin_amdgcn_sched_barrier(0);
      next();
      __builtin_amdgcn_sched_barrier(0);
      if (active) {
        const bool diag = qs0 < k0 + 31;
#pragma unroll
        for (int t = 0; t < 2; ++t) {
          auto probs = [&](auto masked) __attribute__((always_inline)) {
            // the causal mask: query qs0 + t*32 + swz_row(r, hl) precedes the
            // key when kq > t*32 + swz_row(r, 0) (a constant per register)
            const int kq = key - qs0 - 8 * hl;
#pragma unroll
            for (int g = 0; g < 4; ++g) {
              // lse of the 4 queries of registers 4g..4g+3 (consecutive)
              const float4 l4 = *reinterpret_cast<const float4*>(&lse_s[P][t * 32 + swz_row(4 * g, hl)]);
              const float lv[4] = {l4.x, l4.y, l4.z, l4.w};
#pragma unroll
              for (int e = 0; e < 4; ++e) {
                const int r = 4 * g + e;
                float p = fast_exp2(__builtin_fmaf(x[t][r], a.scale_log2, -lv[e]));
                if (decltype(masked)::value && kq > t * 32 + swz_row(r, 0)) p = 0.f;
                x[t][r] = p;
              }
            }
          };
          if (diag)
            probs(std::true_type{});
          else
            probs(std::false_type{});
#pragma unroll
          for (int g = 0; g < 4; ++g)
            Ps[P][w][t][g][lane] = a_u32x4{__float_as_uint(x[t][4 * g]), __float_as_uint(x[t][4 * g + 1]),
                                           __float_as_uint(x[t][4 * g + 2]), __float_as_uint(x[t][4 * g + 3])};
        }
        __builtin_amdgcn_sched_barrier(0);
        second(x, P ? O1 : O0, nullptr);
      }
    } else {
      if (active_prev)  // finish step m-1: dS = P (dP - delta), dK += dS^T Q
        second(x, Qx + qprev * IMG, Ps[P ^ 1]);
      __builtin_amdgcn_sched_barrier(0);
      if (active) {
        // dP - delta: the accumulator starts at -delta (stored negated)
        first_product(x, P ? O1 : O0, [&](int t) __attribute__((always_inline)) {
          a_f32x16 d;
#pragma unroll
          for (int g = 0; g < 4; ++g) {
            const float4 d4 = *reinterpret_cast<const float4*>(&del_s[P][t * 32 + swz_row(4 * g, hl)]);
            d[4 * g + 0] = d4.x;
            d[4 * g + 1] = d4.y;
            d[4 * g + 2] = d4.z;
            d[4 * g + 3] = d4.w;
          }
          return d;
        });
      }
    }
    __builtin_amdgcn_sched_barrier(0);
    vm_wait_all();  // the next step's rows and statistics have landed
    if (j + 1 < n && rt < kBQ2) stat_store(P ^ 1, stat_n);
    __syncthreads();  // P(m) handed over; images of step m-1 free
  };
  // each role runs its own copy of the step loop (the same barriers in the
  // same order), so neither keeps the other's values alive
  auto run = [&](auto role_c) __attribute__((always_inline)) {
    int j = 0, qslot = 0;
    for (; j + 1 < n; j += 2) {
      step(j, qslot, std::integral_constant<int, 0>{}, role_c);
      qslot = qslot == 2 ? 0 : qslot + 1;
      step(j + 1, qslot, std::integral_constant<int, 1>{}, role_c);
      qslot = qslot == 2 ? 0 : qslot + 1;
    }
    if (j < n) {
      step(j, qslot, std::integral_constant<int, 0>{}, role_c);
      qslot = qslot == 2 ? 0 : qslot + 1;
    }
    // the dK waves finish the last step (its P is in buffer (n - 1) % 2)
    if (decltype(role_c)::value && (nq - 1) * kBQ2 + kBQ2 - 1 >= k0) {
      const int pb = (n - 1) & 1, qlast = qslot == 0 ? 2 : qslot - 1;
      second(x, Qx + qlast * IMG, Ps[pb]);
    }
  };
  if (dkw)
    run(std::true_type{});
  else
    run(std::false_type{});
  // the 32 x 128 tile of each wave (dV or dK, rounded to 16 bits) through
  // LDS, then out in 16-byte row chunks: lane holds d = t*32 + lane%32 for
  // keys acc_row(r, hl); the staging rows are padded by 8 elements
  constexpr int SL = D + 8;
  __syncthreads();  // every image and P buffer read
  // 8.5 KB per wave: the dV waves' in the Q images, the dK waves' in the P buffers
  uint16_t* stage = (dkw ? reinterpret_cast<uint16_t*>(&Ps[0][0][0][0][0]) : Qx) + w * 32 * SL;
  static_assert(4 * 32 * SL <= 3 * IMG && 4 * 32 * SL * 2 <= (int)sizeof(Ps), "staging fits");
#pragma unroll
  for (int t = 0; t < DT; ++t)
#pragma unroll
    for (int r = 0; r < 16; ++r)
      stage[acc_row(r, hl) * SL + t * 32 + (lane & 31)] = from_f<FP16>(dkw ? acc[t][r] * a.scale : acc[t][r]);
  wave_lds_fence();  // the wave reads back only its own rows
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const int c = i * 64 + lane, kr = c >> 4, col = (c & 15) * 8;  // key row, first column of the chunk
    const int key_g = k0 + kr;
    if (PAD && (key_g >= a.S || col >= a.hd)) continue;
    *reinterpret_cast<uint4*>(row_ptr(dkw ? a.dk : a.dv, key_g, b, h) + col) =
        *reinterpret_cast<const uint4*>(stage + kr * SL + col);
  }
}

// ------------------------------------- backward: dK, dV, head dims to 96 --
// dK and dV of 32 keys per wave in one wave, so nothing is handed from wave to
// wave, a workgroup is four independent waves with one barrier per 64 queries,
// and two workgroups share a CU, one computing probabilities while the other's
// MFMAs run.  Both accumulators, the K and V fragments and one 32-query tile
// of S and dP take 208 to 216 VGPRs at a head dim of 64.  At 96 they need more
// than the 256 there are: 10 to 12 are spilled with one group of waves and 22
// to 30 with two, whose reloads between the MFMAs of a step (vector-memory
// loads complete in order) wait for the rows of the next step, so at 96 that
// load is only partly hidden.  It still beats pairs of waves that hand P over
// (backward of 1500 x 2 x 32 heads of 80: 175 us with them, 142 here).  S = Q
// K^T and dP = dO V^T are computed with lane = key (query rows swizzled), so P
// and dS are already the A operands of dV += P^T dO and dK += dS^T Q.
//
// The Q and dO rows of a step load directly into LDS a step ahead, one image
// each, double buffered: chunk c (8 columns) of row r at c ^ img_swz(r), which
// puts both the row reads of the A operands (16 rows, one chunk) and the
// transposing reads of the B operands (4 rows x 64 bytes per 32 lanes) in
// distinct banks.  dP's accumulator starts at -delta.
//
// G = 2 as in the forward: the groups take alternate query blocks.
template <int D, bool FP16, bool PAD, int G>
__global__ void __launch_bounds__(G * kAttnThreads, 2) attn_bwd_dkdv_kernel(AttnArgs a) {
  static_assert(D == 64 || D == 96, "wider heads run on the paired kernel");
  constexpr int KS = D / 16, DT = D / 32, CPR = D / 8;
  constexpr int IMG = kBQ2 * D;             // elements of one image
  // an array per image, so the compiler can tell the direct loads into one
  // from the fragment reads of another
  __shared__ __attribute__((aligned(16))) uint16_t Q0[G * IMG];
  __shared__ __attribute__((aligned(16))) uint16_t Q1[G * IMG];
  __shared__ __attribute__((aligned(16))) uint16_t O0[G * IMG];
  __shared__ __attribute__((aligned(16))) uint16_t O1[G * IMG];
  __shared__ __attribute__((aligned(16))) float lse_s[2][G][kBQ2];
  __shared__ __attribute__((aligned(16))) float del_s[2][G][kBQ2];

  const int BH = a.B * a.H;
  const int bh = blockIdx.x % BH, kb = blockIdx.x / BH;
  const int b = bh / a.H, h = bh % a.H;
  const int lane = threadIdx.x & 63, hl = lane >> 5;
  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);  // wave-uniform
  const int w = wid & 3, grp = G == 1 ? 0 : wid >> 2;
  const int rt = threadIdx.x & (kAttnThreads - 1);  // thread of the group
  const int k0 = kb * kBKV2 + w * 32;
  const int key = k0 + (lane & 31);

  ImgCopy<D, PAD> qc, oc;
  qc.init(a.q, b, h, a.hd, a.S, w, lane);
  oc.init(a.dout, b, h, a.hd, a.S, w, lane);
  // per-query statistics: a group's threads 0-63 lse, 64-127 delta (a padding query gets
  // lse = 1e30, so P = 0); delta is negated when it is stored, not here, where
  // the use would wait for every load in flight
  const float* stats = (rt < 64 ? a.lse : a.delta) + (int64_t)bh * a.S;
  const int si = rt & 63;
  auto stat = [&](int qs) __attribute__((always_inline)) {
    float v = rt < 64 ? 1e30f : 0.f;
    if (!PAD || qs + si < a.S) v = stats[qs + si];
    return v;
  };
  auto stat_store = [&](int p, float v) __attribute__((always_inline)) {
    if (rt < 64)
      lse_s[p][grp][rt] = v;
    else if (rt < 128)
      del_s[p][grp][rt - 64] = -v;
  };
  const int first = (kb * kBKV2) / kBQ2, nq = (a.S + kBQ2 - 1) / kBQ2;
  // steps of a group (an odd count of blocks leaves the second group's last
  // one empty) and its first block
  const int steps = (nq - first + G - 1) / G, mine = first + grp;
  float stat_n = 0.f;
  if (mine < nq) {
    qc.issue(Q0 + grp * IMG, mine * kBQ2);
    oc.issue(O0 + grp * IMG, mine * kBQ2);
    if (rt < 128) stat_n = stat(mine * kBQ2);
  }

  uint4 kf[KS], vf[KS];  // this lane's key: K and V rows, the B operands of S and dP
  {
    const uint16_t* kp = row_ptr(a.k, key, b, h);
    const uint16_t* vp = row_ptr(a.v, key, b, h);
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      kf[ks] = load_row16<PAD>(kp, key < a.S, ks * 16 + hl * 8, a.hd);
      vf[ks] = load_row16<PAD>(vp, key < a.S, ks * 16 + hl * 8, a.hd);
    }
  }
  a_f32x16 dk[DT], dv[DT];
#pragma unroll
  for (int t = 0; t < DT; ++t) dk[t] = dv[t] = a_f32x16{};

  int aoff[KS], toff[DT][2];
#pragma unroll
  for (int ks = 0; ks < KS; ++ks) aoff[ks] = img_row_off<D>(lane, ks);
#pragma unroll
  for (int d2 = 0; d2 < DT; ++d2)
#pragma unroll
    for (int hi = 0; hi < 2; ++hi) toff[d2][hi] = img_tr_off<D>(lane, d2, hi);
  auto bfrag = [&](const uint16_t* img, int kk, int d2) __attribute__((always_inline)) {
    return img_tr(img + kk * 16 * D, toff[d2][0], toff[d2][1]);
  };
  vm_wait_all();
  stat_store(0, stat_n);
  __syncthreads();

  auto step = [&](int i, auto par_c) __attribute__((always_inline)) {
    constexpr int P = decltype(par_c)::value;
    const int m = mine + i * G, qs0 = m * kBQ2;
    const bool more = m + G < nq;
    if (more) {  // the next step's rows into the other images, a step ahead
      qc.issue((P ? Q0 : Q1) + grp * IMG, qs0 + G * kBQ2);
      oc.issue((P ? O0 : O1) + grp * IMG, qs0 + G * kBQ2);
      if (rt < 128) stat_n = stat(qs0 + G * kBQ2);
    }
    const uint16_t* qi = (P ? Q1 : Q0) + grp * IMG;
    const uint16_t* oi = (P ? O1 : O0) + grp * IMG;
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      const int qt = qs0 + t * 32;
      if ((G == 2 && m >= nq) || qt + 31 < k0) continue;  // no block, or every query of the tile precedes the wave's keys
      a_f32x16 s = a_f32x16{}, dp;
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const float4 d4 = *reinterpret_cast<const float4*>(&del_s[P][grp][t * 32 + swz_row(4 * g, hl)]);
        dp[4 * g + 0] = d4.x;
        dp[4 * g + 1] = d4.y;
        dp[4 * g + 2] = d4.z;
        dp[4 * g + 3] = d4.w;
      }
#pragma unroll
      for (int ks = 0; ks < KS; ++ks)
        s = mma<FP16>(*reinterpret_cast<const uint4*>(qi + t * 32 * D + aoff[ks]), kf[ks], s);
#pragma unroll
      for (int ks = 0; ks < KS; ++ks)
        dp = mma<FP16>(*reinterpret_cast<const uint4*>(oi + t * 32 * D + aoff[ks]), vf[ks], dp);
      // P; query of register r = qt + swz_row(r, hl); the causal mask only on
      // the tiles that cross the diagonal
      auto probs = [&](auto masked) __attribute__((always_inline)) {
        const int kq = key - qt - 8 * hl;  // masked when > swz_row(r, 0)
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          const float4 l4 = *reinterpret_cast<const float4*>(&lse_s[P][grp][t * 32 + swz_row(4 * g, hl)]);
          const float lv[4] = {l4.x, l4.y, l4.z, l4.w};
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const int r = 4 * g + e;
            float p = fast_exp2(__builtin_fmaf(s[r], a.scale_log2, -lv[e]));
            if (decltype(masked)::value && kq > swz_row(r, 0)) p = 0.f;
            s[r] = p;
          }
        }
      };
      if (qt < k0 + 31)
        probs(std::true_type{});
      else
        probs(std::false_type{});
#pragma unroll
      for (int k2 = 0; k2 < 2; ++k2) {
        const int kk = t * 2 + k2, e0 = k2 * 8;
        const uint4 pa = make_uint4(pack2<FP16>(s[e0 + 0], s[e0 + 1]), pack2<FP16>(s[e0 + 2], s[e0 + 3]),
                                    pack2<FP16>(s[e0 + 4], s[e0 + 5]), pack2<FP16>(s[e0 + 6], s[e0 + 7]));
#pragma unroll
        for (int d2 = 0; d2 < DT; ++d2) dv[d2] = mma<FP16>(pa, bfrag(oi, kk, d2), dv[d2]);
      }
#pragma unroll
      for (int r = 0; r < 16; ++r) dp[r] = s[r] * dp[r];
#pragma unroll
      for (int k2 = 0; k2 < 2; ++k2) {
        const int kk = t * 2 + k2, e0 = k2 * 8;
        const uint4 sa = make_uint4(pack2<FP16>(dp[e0 + 0], dp[e0 + 1]), pack2<FP16>(dp[e0 + 2], dp[e0 + 3]),
                                    pack2<FP16>(dp[e0 + 4], dp[e0 + 5]), pack2<FP16>(dp[e0 + 6], dp[e0 + 7]));
#pragma unroll
        for (int d2 = 0; d2 < DT; ++d2) dk[d2] = mma<FP16>(sa, bfrag(qi, kk, d2), dk[d2]);
      }
    }
    vm_wait_all();  // the next step's rows and statistics have landed
    if (more) stat_store(P ^ 1, stat_n);
    __syncthreads();  // this step's images free, the next step's visible
  };
  int i = 0;
  for (; i + 1 < steps; i += 2) {
    step(i, std::integral_constant<int, 0>{});
    step(i + 1, std::integral_constant<int, 1>{});
  }
  if (i < steps) step(i, std::integral_constant<int, 0>{});

  if constexpr (G == 2) {
    // (the images are free: every group passed the last step's barrier)
    const int at = (w & 1) * (DT * 4 * 64) + lane;
    float4* mv = reinterpret_cast<float4*>(w < 2 ? O0 : O1) + at;
    float4* mk = reinterpret_cast<float4*>(w < 2 ? Q0 : Q1) + at;
    if (grp == 1) {
#pragma unroll
      for (int t = 0; t < DT; ++t)
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          mv[(t * 4 + g) * 64] = make_float4(dv[t][g * 4], dv[t][g * 4 + 1], dv[t][g * 4 + 2], dv[t][g * 4 + 3]);
          mk[(t * 4 + g) * 64] = make_float4(dk[t][g * 4], dk[t][g * 4 + 1], dk[t][g * 4 + 2], dk[t][g * 4 + 3]);
        }
    }
    __syncthreads();
    if (grp == 1) return;
#pragma unroll
    for (int t = 0; t < DT; ++t)
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const float4 u = mv[(t * 4 + g) * 64], x = mk[(t * 4 + g) * 64];
        dv[t][g * 4 + 0] += u.x;
        dv[t][g * 4 + 1] += u.y;
        dv[t][g * 4 + 2] += u.z;
        dv[t][g * 4 + 3] += u.w;
        dk[t][g * 4 + 0] += x.x;
        dk[t][g * 4 + 1] += x.y;
        dk[t][g * 4 + 2] += x.z;
        dk[t][g * 4 + 3] += x.w;
      }
    wave_lds_fence();  // the rows below go where these sums were
  }

  // out through LDS in 16-byte row chunks: lane holds d = t*32 + lane%32 for
  // keys acc_row(r, hl); dV by way of the dO images, dK of the Q images
  // (with two groups, within the wave's own part of the sums above)
  static_assert(2 * 32 * D <= IMG, "two waves' staging fits an image");
  uint16_t* sv = (w < 2 ? O0 : O1) + (w & 1) * G * 32 * D;
  uint16_t* sk = (w < 2 ? Q0 : Q1) + (w & 1) * G * 32 * D;
#pragma unroll
  for (int t = 0; t < DT; ++t)
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const int o = acc_row(r, hl) * D + t * 32 + (lane & 31);
      sv[o] = from_f<FP16>(dv[t][r]);
      sk[o] = from_f<FP16>(dk[t][r] * a.scale);
    }
  wave_lds_fence();  // a wave reads back only its own rows
#pragma unroll
  for (int i = 0; i < 32 * CPR / 64; ++i) {
    const int c = i * 64 + lane, kr = c / CPR, col = (c % CPR) * 8;
    if (PAD && (k0 + kr >= a.S || col >= a.hd)) continue;
    *reinterpret_cast<uint4*>(row_ptr(a.dv, k0 + kr, b, h) + col) = *reinterpret_cast<const uint4*>(sv + kr * D + col);
    *reinterpret_cast<uint4*>(row_ptr(a.dk, k0 + kr, b, h) + col) = *reinterpret_cast<const uint4*>(sk + kr * D + col);
  }
}

// ------------------------------------------------------------ backward: dQ --
// G = 2 as in the forward (at a head dim of 128 it spills 3 registers, all
// outside the loop, and with PAD 8).
template <int D, bool FP16, bool PAD, int G>
__global__ void __launch_bounds__(G * kAttnThreads, 2) attn_bwd_dq_kernel(AttnArgs a) {
  constexpr int KS = D / 16, DT = D / 32;
  constexpr int IMG = kBKV * D;  // elements of one image
  __shared__ __attribute__((aligned(16))) uint16_t K0[G * IMG];
  __shared__ __attribute__((aligned(16))) uint16_t K1[G * IMG];
  __shared__ __attribute__((aligned(16))) uint16_t V0[G * IMG];
  __shared__ __attribute__((aligned(16))) uint16_t V1[G * IMG];

  const int BH = a.B * a.H, nqb = (a.S + kBQ - 1) / kBQ;
  const int bh = blockIdx.x % BH, qb = nqb - 1 - blockIdx.x / BH;
  const int b = bh / a.H, h = bh % a.H;
  const int lane = threadIdx.x & 63, hl = lane >> 5;
  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);  // wave-uniform
  const int w = wid & 3, grp = G == 1 ? 0 : wid >> 2;
  const int q0 = qb * kBQ + w * 32;
  const int q = q0 + (lane & 31);

  ImgCopy<D, PAD> kc, vc;
  kc.init(a.k, b, h, a.hd, a.S, w, lane);
  vc.init(a.v, b, h, a.hd, a.S, w, lane);
  const int nkv = (qb * kBQ + kBQ) / kBKV / G;
  kc.issue(K0 + grp * IMG, grp * kBKV);
  vc.issue(V0 + grp * IMG, grp * kBKV);

  const bool real = !PAD || q < a.S;  // false on padding rows of the last block
  uint4 qf[KS], of[KS];
  {
    const uint16_t* qp = row_ptr(a.q, q, b, h);
    const uint16_t* op = row_ptr(a.dout, q, b, h);
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      qf[ks] = load_row16<PAD>(qp, real, ks * 16 + hl * 8, a.hd);
      of[ks] = load_row16<PAD>(op, real, ks * 16 + hl * 8, a.hd);
    }
  }
  const float lse = real ? a.lse[(int64_t)bh * a.S + q] : 1e30f;
  // delta = rowsum(dO * O) for this query, from the dO fragments already in
  // registers (the two half-waves hold alternate 8-element chunks of the row);
  // written out for the dK/dV kernel, which runs next
  float del = 0.f;
  {
    const uint16_t* opp = row_ptr(a.o, q, b, h);
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      const uint4 ov = load_row16<PAD>(opp, real, ks * 16 + hl * 8, a.hd);
      const uint32_t ow[4] = {ov.x, ov.y, ov.z, ov.w};
      const uint32_t dw[4] = {of[ks].x, of[ks].y, of[ks].z, of[ks].w};
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        del += to_f<FP16>((uint16_t)(ow[e] & 0xffffu)) * to_f<FP16>((uint16_t)(dw[e] & 0xffffu));
        del += to_f<FP16>((uint16_t)(ow[e] >> 16)) * to_f<FP16>((uint16_t)(dw[e] >> 16));
      }
    }
    del += __shfl_xor(del, 32, 64);
    if (grp == 0 && hl == 0 && real) a.delta[(int64_t)bh * a.S + q] = del;
  }
  a_f32x16 dq[DT];
#pragma unroll
  for (int t = 0; t < DT; ++t)
#pragma unroll
    for (int r = 0; r < 16; ++r) dq[t][r] = 0.f;

  int aoff[KS], toff[DT][2];
#pragma unroll
  for (int ks = 0; ks < KS; ++ks) aoff[ks] = img_row_off<D>(lane, ks);
#pragma unroll
  for (int dt = 0; dt < DT; ++dt)
#pragma unroll
    for (int hi = 0; hi < 2; ++hi) toff[dt][hi] = img_tr_off<D>(lane, dt, hi);
  vm_wait_all();
  __syncthreads();

  auto block = [&](int j, auto cur_c) __attribute__((always_inline)) {
    constexpr int cur = decltype(cur_c)::value;
    const int kv0 = (j * G + grp) * kBKV;
    if (j + 1 < nkv) {  // the group's next block, a block ahead
      kc.issue((cur ? K0 : K1) + grp * IMG, kv0 + G * kBKV);
      vc.issue((cur ? V0 : V1) + grp * IMG, kv0 + G * kBKV);
    }
    const uint16_t* ki = (cur ? K1 : K0) + grp * IMG;
    const uint16_t* vi = (cur ? V1 : V0) + grp * IMG;
    // one 32-key tile at a time: S^T = K Q^T, dP^T = V dO^T (lane = query),
    // dS^T, then dQ^T += K^T dS^T over those 32 keys
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      const int kt0 = kv0 + t * 32;
      if (kt0 > q0 + 31) continue;  // every key of the tile follows the wave's queries
      a_f32x16 s, dp;
#pragma unroll
      for (int r = 0; r < 16; ++r) s[r] = dp[r] = 0.f;
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) {
        s = mma<FP16>(*reinterpret_cast<const uint4*>(ki + t * 32 * D + aoff[ks]), qf[ks], s);
        dp = mma<FP16>(*reinterpret_cast<const uint4*>(vi + t * 32 * D + aoff[ks]), of[ks], dp);
      }
      // causal mask only on the tiles that cross the diagonal
      auto dsoft = [&](auto masked) __attribute__((always_inline)) {
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          float p = fast_exp2(__builtin_fmaf(s[r], a.scale_log2, -lse));
          if (decltype(masked)::value && kt0 + swz_row(r, hl) > q) p = 0.f;
          dp[r] = p * (dp[r] - del);
        }
      };
      if (kt0 + 31 > q0)
        dsoft(std::true_type{});
      else
        dsoft(std::false_type{});
#pragma unroll
      for (int k2 = 0; k2 < 2; ++k2) {
        const int kk = t * 2 + k2, e0 = k2 * 8;
        const uint4 sb = make_uint4(pack2<FP16>(dp[e0 + 0], dp[e0 + 1]), pack2<FP16>(dp[e0 + 2], dp[e0 + 3]),
                                    pack2<FP16>(dp[e0 + 4], dp[e0 + 5]), pack2<FP16>(dp[e0 + 6], dp[e0 + 7]));
#pragma unroll
        for (int dt = 0; dt < DT; ++dt)
          dq[dt] = mma<FP16>(img_tr(ki + kk * 16 * D, toff[dt][0], toff[dt][1]), sb, dq[dt]);
      }
    }
    vm_wait_all();  // the next block's rows have landed
    __syncthreads();  // this block's images free, the next block's visible
  };
  int j = 0;
  for (; j + 1 < nkv; j += 2) {
    block(j, std::integral_constant<int, 0>{});
    block(j + 1, std::integral_constant<int, 1>{});
  }
  if (j < nkv) block(j, std::integral_constant<int, 0>{});
  if constexpr (G == 2) {
    // (the images are free: every group passed the last block's barrier)
    float4* sq = reinterpret_cast<float4*>(w < 2 ? K0 : K1) + (w & 1) * (DT * 4 * 64) + lane;
    if (grp == 1) {
#pragma unroll
      for (int t = 0; t < DT; ++t)
#pragma unroll
        for (int g = 0; g < 4; ++g)
          sq[(t * 4 + g) * 64] = make_float4(dq[t][g * 4], dq[t][g * 4 + 1], dq[t][g * 4 + 2], dq[t][g * 4 + 3]);
    }
    __syncthreads();
    if (grp == 1) return;
#pragma unroll
    for (int t = 0; t < DT; ++t)
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const float4 u = sq[(t * 4 + g) * 64];
        dq[t][g * 4 + 0] += u.x;
        dq[t][g * 4 + 1] += u.y;
        dq[t][g * 4 + 2] += u.z;
        dq[t][g * 4 + 3] += u.w;
      }
  }
  if (PAD && !real) return;
  uint16_t* dqp = row_ptr(a.dq, q, b, h);
#pragma unroll
  for (int t = 0; t < DT; ++t)
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      if (PAD && t * 32 + g * 8 >= a.hd) continue;
      uint2 v;
      v.x = pack2<FP16>(dq[t][g * 4 + 0] * a.scale, dq[t][g * 4 + 1] * a.scale);
      v.y = pack2<FP16>(dq[t][g * 4 + 2] * a.scale, dq[t][g * 4 + 3] * a.scale);
      *reinterpret_cast<uint2*>(dqp + t * 32 + g * 8 + hl * 4) = v;
    }
}

}  // namespace eth

using namespace eth;

static int attn_check(const eth_attn_desc_t* d) {
  ETH_CHECK_ARG(d, "attention: null descriptor");
  ETH_CHECK_ARG(d->dtype == ETH_BF16 || d->dtype == ETH_F16, "attention: dtype must be bf16/fp16");
  ETH_CHECK_ARG(d->head_dim >= 8 && d->head_dim <= 128 && d->head_dim % 8 == 0,
                "attention: head_dim must be a multiple of 8 in [8, 128] (got %d)", d->head_dim);
  ETH_CHECK_ARG(d->seq > 0, "attention: seq must be positive (got %d)", d->seq);
  ETH_CHECK_ARG(d->batch > 0 && d->heads > 0, "attention: bad batch/heads");
  return ETH_OK;
}

static AttnTensor tin(const void* p, const int64_t* st, const eth_attn_desc_t* d) {
  AttnTensor t;
  t.p = (const uint16_t*)p;
  t.ss = st[0];
  t.sb = st[1];
  t.sh = st[2];
  const int64_t extent = ((int64_t)(d->seq - 1) * st[0] + (int64_t)(d->batch - 1) * st[1] +
                          (int64_t)(d->heads - 1) * st[2] + d->head_dim) * 2;
  t.bytes = extent < (1LL << 31) ? (uint32_t)extent : 0u;
  return t;
}
static AttnOut tout(void* p, const int64_t* st) {
  AttnOut t;
  t.p = (uint16_t*)p;
  t.ss = st[0];
  t.sb = st[1];
  t.sh = st[2];
  return t;
}

// Groups of four waves that share a block of the forward, dQ, and dK/dV up to
// a head dim of 96: two where one group per block leaves wave slots empty,
// from the start (up to one workgroup per CU) or once the short chains of a
// grid of up to two have ended, and the chain is long enough to pay for the
// second group's start and the closing addition.  Measured on both sides of
// the lines, forward / backward, one group -> two (us; workgroups, sequence x
// head dim): 256, 2048 x 128 42.1 / 115.8 -> 36.5 / 106.7; 256, 2048 x 64 - /
// 72.3 (dK/dV in one) -> 22.2 / 60.7; 128, 1024 x 64 16.1 / 44.3 -> 13.4 / 36.9;
// 84, 777 x 96 15.9 / 53.1 -> 14.6 / 47.9; 48, 300 x 96 12.3 / 27.4 -> 12.5 /
// 27.7; 512, 4096 x 128 94.3 / 274 -> 87.0 / 256; 512, 4096 x 64 60.5 / 172 ->
// 54.0 / 143; 384, 1500 x 80 31.8 / 104 -> 28.4 / 94.0; 384, 1024 x 128 28.9 /
// 79.8 -> 29.8 / 80.8; 512, 512 x 64 14.1 / 35.8 -> 15.9 / 40.8 (dK/dV in one);
// 768, 1500 x 80 50.7 / 140 -> 54.3 / 149 (dK/dV in one).
static int attn_groups(int grid, int seq) { return seq > (grid <= 256 ? 512 : 1024) && grid <= 512 ? 2 : 1; }

template <int D, bool FP16, bool PAD>
static void launch_fwd(const AttnArgs& a, int grid, hipStream_t s) {
  if (attn_groups(grid, a.S) == 2)
    attn_fwd_kernel<D, FP16, PAD, 2><<<grid, 2 * kAttnThreads, 0, s>>>(a);
  else
    attn_fwd_kernel<D, FP16, PAD, 1><<<grid, kAttnThreads, 0, s>>>(a);
}

// dQ first: it also writes delta, which dK/dV reads
template <int D, bool FP16, bool PAD>
static void launch_bwd(const AttnArgs& a, int g_q, int g_kv, hipStream_t s) {
  if (attn_groups(g_q, a.S) == 2)
    attn_bwd_dq_kernel<D, FP16, PAD, 2><<<g_q, 2 * kAttnThreads, 0, s>>>(a);
  else
    attn_bwd_dq_kernel<D, FP16, PAD, 1><<<g_q, kAttnThreads, 0, s>>>(a);
  if constexpr (D == 128)
    attn_bwd_dkdv_x128_kernel<FP16, PAD><<<g_kv, 2 * kAttnThreads, 0, s>>>(a);
  else if (attn_groups(g_kv, a.S) == 2)
    attn_bwd_dkdv_kernel<D, FP16, PAD, 2><<<g_kv, 2 * kAttnThreads, 0, s>>>(a);
  else
    attn_bwd_dkdv_kernel<D, FP16, PAD, 1><<<g_kv, kAttnThreads, 0, s>>>(a);
}

static bool aligned_rows(const void* p, const int64_t* st) {
  return ((uintptr_t)p & 15) == 0 && st[0] % 8 == 0 && st[1] % 8 == 0 && st[2] % 8 == 0;
}

extern "C" int eth_attn_fwd(const eth_attn_desc_t* d, const void* q, const void* k, const void* v,
                            void* out, float* lse, void* stream) {
  if (int rc = attn_check(d)) return rc;
  ETH_CHECK_ARG(q && k && v && out && lse, "eth_attn_fwd: null pointer");
  ETH_CHECK_ARG(aligned_rows(q, d->q_strides) && aligned_rows(k, d->k_strides) && aligned_rows(v, d->v_strides) &&
                    aligned_rows(out, d->o_strides),
                "eth_attn_fwd: rows must be 16-byte aligned");
  AttnArgs a{};
  a.q = tin(q, d->q_strides, d);
  a.k = tin(k, d->k_strides, d);
  a.v = tin(v, d->v_strides, d);
  a.out = tout(out, d->o_strides);
  ETH_CHECK_ARG(a.q.bytes && a.k.bytes && a.v.bytes, "eth_attn_fwd: tensors above 2 GiB are not supported");
  a.lse = lse;
  a.B = d->batch;
  a.H = d->heads;
  a.S = d->seq;
  a.hd = d->head_dim;
  a.scale = 1.0f / sqrtf((float)d->head_dim);
  a.scale_log2 = a.scale * 1.4426950408889634f;
  const int grid = a.B * a.H * ((a.S + kBQ - 1) / kBQ);
  hipStream_t s = (hipStream_t)stream;
  const bool fp16 = d->dtype == ETH_F16;
  const int width = a.hd > 96 ? 128 : a.hd > 64 ? 96 : 64;
  // full blocks (every row and head-dim column real) take the unguarded kernels
  const bool pad = a.S % kBQ != 0 || a.hd != width;
#define ETH_ATTN_FWD(D, F)                   \
  if (pad)                                   \
    launch_fwd<D, F, true>(a, grid, s);      \
  else                                       \
    launch_fwd<D, F, false>(a, grid, s);
  if (a.hd > 96) {
    if (fp16) { ETH_ATTN_FWD(128, true) } else { ETH_ATTN_FWD(128, false) }
  } else if (a.hd > 64) {
    if (fp16) { ETH_ATTN_FWD(96, true) } else { ETH_ATTN_FWD(96, false) }
  } else {
    if (fp16) { ETH_ATTN_FWD(64, true) } else { ETH_ATTN_FWD(64, false) }
  }
#undef ETH_ATTN_FWD
  ETH_CHECK_LAUNCH("eth_attn_fwd");
  return ETH_OK;
}

extern "C" int eth_attn_bwd(const eth_attn_desc_t* d, const void* q, const void* k, const void* v,
                            const void* out, const void* dout, const float* lse, float* delta, void* dq,
                            void* dk, void* dv, void* stream) {
  if (int rc = attn_check(d)) return rc;
  ETH_CHECK_ARG(q && k && v && out && dout && lse && delta && dq && dk && dv, "eth_attn_bwd: null pointer");
  ETH_CHECK_ARG(aligned_rows(q, d->q_strides) && aligned_rows(k, d->k_strides) && aligned_rows(v, d->v_strides) &&
                    aligned_rows(out, d->o_strides) && aligned_rows(dout, d->do_strides) &&
                    aligned_rows(dq, d->dq_strides) && aligned_rows(dk, d->dk_strides) &&
                    aligned_rows(dv, d->dv_strides),
                "eth_attn_bwd: rows must be 16-byte aligned");
  AttnArgs a{};
  a.q = tin(q, d->q_strides, d);
  a.k = tin(k, d->k_strides, d);
  a.v = tin(v, d->v_strides, d);
  a.o = tin(out, d->o_strides, d);
  a.dout = tin(dout, d->do_strides, d);
  a.dq = tout(dq, d->dq_strides);
  a.dk = tout(dk, d->dk_strides);
  a.dv = tout(dv, d->dv_strides);
  ETH_CHECK_ARG(a.q.bytes && a.k.bytes && a.v.bytes && a.o.bytes && a.dout.bytes,
                "eth_attn_bwd: tensors above 2 GiB are not supported");
  a.lse = (float*)lse;
  a.delta = delta;
  a.B = d->batch;
  a.H = d->heads;
  a.S = d->seq;
  a.hd = d->head_dim;
  a.scale = 1.0f / sqrtf((float)d->head_dim);
  a.scale_log2 = a.scale * 1.4426950408889634f;
  hipStream_t s = (hipStream_t)stream;
  const bool fp16 = d->dtype == ETH_F16;
  const int g_kv = a.B * a.H * ((a.S + kBKV2 - 1) / kBKV2);
  const int g_q = a.B * a.H * ((a.S + kBQ - 1) / kBQ);
  // dQ first: it also writes delta = rowsum(dO * O), which dK/dV reads
  const int width = a.hd > 96 ? 128 : a.hd > 64 ? 96 : 64;
  static_assert(kBKV2 == kBQ, "one padding rule for the three backward kernels");
  const bool pad = a.S % kBKV2 != 0 || a.hd != width;
#define ETH_ATTN_BWD(D, F)                          \
  if (pad)                                          \
    launch_bwd<D, F, true>(a, g_q, g_kv, s);        \
  else                                              \
    launch_bwd<D, F, false>(a, g_q, g_kv, s);
  if (a.hd > 96) {
    if (fp16) { ETH_ATTN_BWD(128, true) } else { ETH_ATTN_BWD(128, false) }
  } else if (a.hd > 64) {
    if (fp16) { ETH_ATTN_BWD(96, true) } else { ETH_ATTN_BWD(96, false) }
  } else {
    if (fp16) { ETH_ATTN_BWD(64, true) } else { ETH_ATTN_BWD(64, false) }
  }
#undef ETH_ATTN_BWD
  ETH_CHECK_LAUNCH("eth_attn_bwd");
  return ETH_OK;
}
