// bf16/fp16 GEMM on CDNA4 matrix cores (v_mfma_f32_32x32x16_{bf16,f16}),
// fp32 accumulation, operands staged through LDS by direct loads.
//
//   C[m, n] (+)= alpha * sum_k A(m, k) * B(k, n)  (+ bias[n])
//
// A(m, k) is read K-contiguous (A[m*lda + k]) or M-contiguous (A[k*lda + m]);
// B(k, n) is read K-contiguous (B[n*ldb + k]) or N-contiguous (B[k*ldb + n]).
// The three GPT linear-layer products are
//   forward  Y = X W^T      : A K-contiguous, B K-contiguous
//   dgrad    dX = dY W      : A K-contiguous, B N-contiguous
//   wgrad    dW += dY^T X   : A M-contiguous, B N-contiguous, fp32 C += (the
//                             Megatron main_grad accumulation, fused)
//
// Kernels:
//  * gemm256_m16_kernel / gemm256_m32_kernel, the main ones: 256x256x64
//    tiles, 4 waves (one per SIMD) of 128x128 each, 256 accumulator
//    registers per lane held in AGPRs.  Operands go global -> LDS with
//    direct loads (buffer_load ... lds) into two stages.  The k loop is
//    software-pipelined by hand: while the MFMAs of k-tile t run, k-tile
//    t+1 streams into the other stage, one 1 KB load per few MFMA gaps,
//    and the next fragments are read from LDS between the MFMAs
//    (sched_barrier fixes the order).  One barrier per k-tile.
//    Row-contiguous operands land as they are in memory and their
//    fragments come out of LDS through ds_read_b64_tr_b16.  The epilogue
//    stages each 32-row slab through LDS and writes whole rows with buffer
//    stores.  m16 (v_mfma_f32_16x16x32, single-buffered fragments) serves
//    the forward, data-gradient and weight-gradient products (for the last,
//    both operands row-contiguous, through asm MFMAs); m32
//    (v_mfma_f32_32x32x16) a row-contiguous A with a K-contiguous B and
//    K % 128 == 0.  Where K is no multiple of 64 (128 in the last layout) m16
//    runs in an instantiation whose last k-tile is short (TAIL), in every
//    layout: forward of [8448, 3648] x 416 took 77 us on 128x128 ring tiles
//    and 68 on the register-staged ones before them, now 41; [12384, 14368] x
//    1496 861, 686, now 485.  C rows must be aligned to four columns.
//  * gemm_ring_kernel: 128x128 or 64x64 tiles with four LDS stages, for the
//    grids that 256x256 tiles leave mostly idle and for every shape and
//    alignment.
// plan_tile() chooses among them by the time each would take.
// Tiles are assigned XCD-aware (consecutive workgroups land on different
// XCDs, so the tile id is remapped to give each XCD a contiguous range) and
// in GROUP_M-row groups so neighbouring workgroups share A and B tiles in L2.
//
// Replaces the F.linear / cuBLAS calls of mpu/layers.py:357-370,452-470 and
// the main_grad.add_ hook of model/distributed.py:116-123.
#include <algorithm>
#include <type_traits>

#include "common.h"

namespace eth {

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8_t __attribute__((ext_vector_type(8)));
typedef float f32x16_t __attribute__((ext_vector_type(16)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2_t __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));

template <bool FP16>
__device__ __forceinline__ f32x16_t mfma32(const uint4& a, const uint4& b, const f32x16_t& c) {
  if constexpr (FP16) {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8_t, a),
                                                  __builtin_bit_cast(f16x8_t, b), c, 0, 0, 0);
  } else {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, a),
                                                   __builtin_bit_cast(bf16x8_t, b), c, 0, 0, 0);
  }
}

// Workgroup barrier after this wave's LDS accesses and direct global->LDS
// loads have completed.  (__syncthreads also fences global memory, which
// makes every wave wait for its outstanding stores.)
__device__ __forceinline__ void dma_barrier() {
  asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
}
// The same with the newest N vector-memory loads of this wave still in
// flight (loads complete in issue order): the prologues start on k-tile 0
// while k-tile 1 is still arriving.
template <int N>
__device__ __forceinline__ void dma_barrier_but() {
  static_assert(N >= 0 && N < 64, "vmcnt is 6 bits");
  asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(N) : "memory");
}

// Map a linear workgroup id to (tile_m, tile_n): XCD-contiguous, then
// GROUP_M-row grouped.
__device__ __forceinline__ void tile_coords(int pid, int tiles_m, int tiles_n, int& tm, int& tn) {
  constexpr int kXcds = 8, kGroupM = 4;
  const int total = tiles_m * tiles_n;
  const int per = (total + kXcds - 1) / kXcds;
  const int tall = total % kXcds == 0 ? kXcds : total % kXcds;
  const int xcd = pid % kXcds, local = pid / kXcds;
  pid = xcd < tall ? xcd * per + local : tall * per + (xcd - tall) * (per - 1) + local;
  const int in_group = kGroupM * tiles_n;
  const int first_m = (pid / in_group) * kGroupM;
  const int gm = min(tiles_m - first_m, kGroupM);
  tm = first_m + (pid % in_group) % gm;
  tn = (pid % in_group) / gm;
}

// Buffer-resource loads: 32-bit byte offsets (one VGPR per chunk, fixed for
// the whole K loop; the k advance goes in the scalar offset) and hardware
// bounds checking -- an offset of kOob reads zeros, which masks rows past
// the matrix and k past K without branches.
typedef __amdgpu_buffer_rsrc_t rsrc_t;
constexpr int32_t kOob = (int32_t)0x80000000u;

__device__ __forceinline__ rsrc_t make_rsrc(const void* p, uint32_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), (short)0, (int)bytes, 0x00020000);
}

// Tile moved by direct global->LDS loads (buffer_load_dwordx4 ... lds):
// lane i of an instruction writes its 16 bytes at the wave's LDS base +
// 16 i, so the tile's LDS image is covered by consecutive 1 KB pieces,
// PER_WAVE of them per wave.
//  * KC (K-contiguous operand): [ROWS][BK] image without padding; the
//    16-byte unit p of row r holds k-chunk p ^ kc_swizzle(r) (the lane that
//    fills unit p loads that chunk), so the fragment reads -- 16 lanes on
//    16 consecutive rows, one chunk -- hit 16 distinct bank groups.
//  * otherwise (row-contiguous operand): [BK][ROWS + 32] image as it is in
//    memory; the padding units get an out-of-range offset (they read zeros).
typedef __attribute__((address_space(3))) void lds_void_t;
__device__ __forceinline__ void dma16(rsrc_t rs, uint16_t* lds, int32_t voff, int32_t soff) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (lds_void_t*)lds, 16, voff, soff, 0, 0);
}
// injective on rows 0-7 and on the even and the odd rows of 0-15 (the rows
// one 128-byte and one 256-byte bank sweep of a fragment read cover), and
// periodic in 16 rows, so every 32-row fragment block shares it
__device__ __forceinline__ int kc_swizzle(int r) { return (r & 7) ^ ((r >> 3) & 1); }
template <int ROWS, int BK, bool KC>
struct DTile {
  static constexpr int UPR = KC ? BK / 8 : ROWS / 8 + 4;  // 16-byte units per LDS row
  static constexpr int DPR = KC ? BK / 8 : ROWS / 8;      // of which data
  static constexpr int NROW = KC ? ROWS : BK;
  static constexpr int PER_WAVE = NROW * UPR / 256;
  static constexpr int IMG = NROW * UPR * 8;  // image size in elements
  static_assert(NROW * UPR % 256 == 0, "tile split");
  static_assert(!KC || BK == 64, "the swizzle covers 8 chunks per row");
  int32_t off[PER_WAVE];
  int wave;
  __device__ __forceinline__ void init(int64_t ld, int r0, int rows) {
    wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int lane = threadIdx.x & 63;
#pragma unroll
    for (int j = 0; j < PER_WAVE; ++j) {
      const int u = (wave * PER_WAVE + j) * 64 + lane;
      const int row = u / UPR, c = u % UPR;
      if (KC)
        off[j] = r0 + row < rows ? (int32_t)((((int64_t)(r0 + row)) * ld + (c ^ kc_swizzle(row)) * 8) * 2) : kOob;
      else if (c >= DPR)
        off[j] = kOob;
      else
        off[j] = r0 + c * 8 < rows ? (int32_t)(((int64_t)row * ld + r0 + c * 8) * 2) : kOob;
    }
  }
  // from here on the pieces' units at k >= left of a k-tile read zeros: set
  // for the last k-tile when K is no multiple of 64, once its turn comes
  __device__ __forceinline__ void limit(int left) {
    const int lane = threadIdx.x & 63;
#pragma unroll
    for (int j = 0; j < PER_WAVE; ++j) {
      const int u = (wave * PER_WAVE + j) * 64 + lane;
      const int row = u / UPR, c = u % UPR;
      if ((KC ? (c ^ kc_swizzle(row)) * 8 : row) >= left) off[j] = kOob;
    }
  }
  // pieces [J0, J1) of k-tile k0 into the LDS image at S
  template <int J0, int J1>
  __device__ __forceinline__ void issue(uint16_t* S, rsrc_t rs, int64_t ld, int k0) {
    const int32_t soff = KC ? k0 * 2 : (int32_t)((int64_t)k0 * ld * 2);
#pragma unroll
    for (int j = J0; j < J1; ++j) dma16(rs, S + (wave * PER_WAVE + j) * 512, off[j], soff);
  }
};

typedef short s16x4_t __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) s16x4_t lds_s16x4_t;
// MFMA operand (8 consecutive k of one row) from a [k][row] LDS tile: two
// transposing reads of 4 k each.  Lane l must pass the address of k-row
// k0 + (l%16)/4 (k0 = 8*(l/32)), element row0 + 16*((l/16)%2) + 4*(l%4);
// it then receives rows row0 + l%32, k = k0 .. k0+7.
__device__ __forceinline__ uint4 tr_frag(const uint16_t* p, int lrow) {
  const u32x2_t lo = __builtin_bit_cast(u32x2_t, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4_t*)p));
  const u32x2_t hi =
      __builtin_bit_cast(u32x2_t, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4_t*)(p + 4 * lrow)));
  return make_uint4(lo.x, lo.y, hi.x, hi.y);
}

// The same for the 16x16x32 layout: lane l passes the address of k-row
// k0 + (l%16)/4 (k0 = 8*(l/16)), element row0 + 4*(l%4); it receives row
// row0 + l%16, k = k0 .. k0+7.
__device__ __forceinline__ uint4 tr_frag16(const uint16_t* p, int lrow) { return tr_frag(p, lrow); }

struct GemmArgs {
  const uint16_t* A;
  const uint16_t* B;
  uint32_t a_bytes, b_bytes;  // extent of A / B for the buffer range checks
  void* C;
  const uint16_t* bias;
  int M, N, K;
  int64_t lda, ldb, ldc;
  int c_dtype;
  int flags;
  float alpha;
  uint32_t c_bytes;  // extent of C (the gemm256 kernels' store range)
  bool c_vec;        // C rows take 4-column vector accesses
  int k_split;              // split-K: k extent per split (0: one split of K)
  int64_t c_split_stride;   // split-K: elements between the splits' C slices
};

// 256x256x64 tiles, 4 waves of 128x128 (one per SIMD).
//
// MFMA v_mfma_f32_16x16x32: a 128x128 wave tile is 8 x 8 blocks of 16x16,
// 4 fp32 accumulators per lane each (256 in all, AGPRs).  A k-tile of 64 is
// two k-steps of 32; a k-step is 64 MFMAs, preceded by the 16 fragment reads
// (8 A row blocks, 8 B column blocks) that feed it.  The 16x16x32 shape
// (twice the MFMA instructions of 32x32x16 for the same work) leaves more
// issue gaps between MFMAs for the fragment reads and direct loads: the same
// tile with 32x32x16 MFMAs ran 6% slower.
template <bool FP16>
__device__ __forceinline__ f32x4_t mfma16(const uint4& a, const uint4& b, const f32x4_t& c) {
  if constexpr (FP16) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8_t, a), __builtin_bit_cast(f16x8_t, b),
                                                  c, 0, 0, 0);
  } else {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, a),
                                                   __builtin_bit_cast(bf16x8_t, b), c, 0, 0, 0);
  }
}

// The same MFMA as inline assembly with the accumulator tied to its AGPRs
// ("+a"), for the kernel whose operands both come through transposing
// reads: through the builtin the register allocator there keeps some 30
// accumulator tuples in VGPRs and copies them around the MFMAs every k-tile.
// The compiler still inserts the LDS waits for the operands (it sees the
// asm's register uses); the only hazard it cannot see, an accumulator read
// right after its MFMA, is covered after the k loop.
template <bool FP16>
__device__ __forceinline__ void mfma16_asm(f32x4_t& c, const uint4& a, const uint4& b) {
  if constexpr (FP16)
    asm volatile("v_mfma_f32_16x16x32_f16 %0, %1, %2, %0"
                 : "+a"(c)
                 : "v"(__builtin_bit_cast(u32x4_t, a)), "v"(__builtin_bit_cast(u32x4_t, b)));
  else
    asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0"
                 : "+a"(c)
                 : "v"(__builtin_bit_cast(u32x4_t, a)), "v"(__builtin_bit_cast(u32x4_t, b)));
}

// The same with the accumulator tied to its VGPRs: for the kernels whose
// accumulators fit there (through the builtin, the allocator rotates them
// through copies around the loop's back edge).
template <bool FP16>
__device__ __forceinline__ void mfma16_tied(f32x4_t& c, const uint4& a, const uint4& b) {
  if constexpr (FP16)
    asm volatile("v_mfma_f32_16x16x32_f16 %0, %1, %2, %0"
                 : "+v"(c)
                 : "v"(__builtin_bit_cast(u32x4_t, a)), "v"(__builtin_bit_cast(u32x4_t, b)));
  else
    asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0"
                 : "+v"(c)
                 : "v"(__builtin_bit_cast(u32x4_t, a)), "v"(__builtin_bit_cast(u32x4_t, b)));
}

template <bool A_K, bool B_K, bool FP16, bool TAIL = false>
__global__ void __launch_bounds__(256, 1) gemm256_m16_kernel(GemmArgs g) {
  constexpr int BM = 256, BN = 256, BK = 64;
  typedef DTile<BM, BK, A_K> ATile;
  typedef DTile<BN, BK, B_K> BTile;
  constexpr int A_IMG = ATile::IMG;           // elements of the A image in a stage
  constexpr int STAGE = A_IMG + BTile::IMG;   // one LDS stage: A image then B image
  constexpr int ER = 128 + 4;                 // epilogue staging row (fp32, padded)
  constexpr int EPI = 4 * 32 * ER * 2;        // epilogue staging in elements
  // the two stages are separate arrays, so the compiler can tell the direct
  // loads into one stage from the fragment reads of the other (it would
  // otherwise wait for the loads before every read); the first also holds
  // the epilogue's staging
  __shared__ __attribute__((aligned(16))) uint16_t smem[STAGE > EPI ? STAGE : EPI];
  __shared__ __attribute__((aligned(16))) uint16_t smem1[STAGE];

  const int tiles_m = (g.M + BM - 1) / BM, tiles_n = (g.N + BN - 1) / BN;
  // split-K launches tiles * splits workgroups: split = blockIdx.x / tiles
  const int tiles = tiles_m * tiles_n;
  const int split = blockIdx.x / tiles;
  const int kb = split * g.k_split;
  int tm, tn;
  tile_coords(blockIdx.x - split * tiles, tiles_m, tiles_n, tm, tn);
  const int m0 = tm * BM, n0 = tn * BN;
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  const int wm = wid >> 1, wn = wid & 1;
  const int l16 = lane & 15, lg = lane >> 4;
  // the 4 output columns this lane writes in the epilogue, and their bias
  // (read now so its latency is hidden behind the k loop)
  const int col = (lane & 31) * 4;
  const int n = n0 + wn * 128 + col;
  float bn[4] = {0.f, 0.f, 0.f, 0.f};
  if ((g.flags & ETH_GEMM_BIAS) && g.bias) {
#pragma unroll
    for (int e = 0; e < 4; ++e)
      if (n + e < g.N) bn[e] = FP16 ? h2f_bits(g.bias[n + e]) : bf2f(g.bias[n + e]);
  }

  // acc[I][J]: C rows I*16 + lane%16, columns J*16 + 4*(lane/16) + 0..3 of
  // the wave's block (B fragment as the MFMA's first operand)
  f32x4_t acc[8][8];
  // pinned to AGPRs where they start, so the register allocator keeps each
  // block in one AGPR tuple and every MFMA accumulates in place (unpinned,
  // it parks some blocks in VGPRs and copies them around the MFMAs)
#define PIN_ACC                                          \
  _Pragma("unroll") for (int i = 0; i < 8; ++i)          \
    _Pragma("unroll") for (int j = 0; j < 8; ++j) asm volatile("" : "+a"(acc[i][j]));
#pragma unroll
  for (int i = 0; i < 8; ++i)
#pragma unroll
    for (int j = 0; j < 8; ++j) acc[i][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  PIN_ACC

  const int span = (g.k_split ? min(g.K, kb + g.k_split) : g.K) - kb;
  const int nk = (span + BK - 1) / BK;
  // TAIL: the last k-tile is short; its loads past K read zeros (left of its
  // k are there; with left == 0 tail stays past it).  An instantiation of its
  // own: the branch in the loop and the scalars it keeps (8 to 18 spilled to
  // vector lanes with a row-contiguous operand) cost 0.5 % of a layer's time.
  // Its MFMAs are asm in every layout: with the builtin ones the branch gets
  // the accumulators copied around ([2048, 8192] x 2048: 77 vs 51 us).
  const int left = span % BK, tail = left ? nk - 1 : nk + 2;
  const rsrc_t ra = make_rsrc(g.A, g.a_bytes), rb = make_rsrc(g.B, g.b_bytes);
  // empty ranges: the loads issued past the last k-tile read zeros
  const rsrc_t ra0 = make_rsrc(g.A, 0), rb0 = make_rsrc(g.B, 0);
  ATile la;
  BTile lb;
  // pieces per half per wave: 8 for a K-contiguous image, 9 for a padded one
  constexpr int NA = ATile::PER_WAVE, NB = BTile::PER_WAVE;
  static_assert((NA == 8 || NA == 9) && (NB == 8 || NB == 9), "the k loop's load slots");
  la.init(g.lda, m0, g.M);
  lb.init(g.ldb, n0, g.N);
#define LIMIT_IF(T)                      \
  if constexpr (TAIL) {                  \
    if ((T) == tail) {                   \
      la.limit(left);                    \
      lb.limit(left);                    \
    }                                    \
  }
  LIMIT_IF(0)
  la.template issue<0, NA>(smem, ra, g.lda, kb);
  lb.template issue<0, NB>(smem + A_IMG, rb, g.ldb, kb);
  LIMIT_IF(1)

  // queue item Q of a k-tile (the A pieces, then the B pieces) into stage S
#define LOAD_Q(Q, S, RSA, RSB, KK)                                      \
  if constexpr ((Q) < NA) {                                             \
    la.template issue<(Q), (Q) + 1>(S, RSA, g.lda, KK);                 \
  } else if constexpr ((Q) < NA + NB) {                                 \
    lb.template issue<(Q) - NA, (Q) - NA + 1>((S) + A_IMG, RSB, g.ldb, KK); \
  }
  // queue items 0-11 of k-tile 1 (the loop's first k-step issues the rest)
  {
    const rsrc_t rsa = nk > 1 ? ra : ra0, rsb = nk > 1 ? rb : rb0;
#define PRO_Q(Q) LOAD_Q(Q, smem1, rsa, rsb, kb + BK)
    PRO_Q(0) PRO_Q(1) PRO_Q(2) PRO_Q(3) PRO_Q(4) PRO_Q(5)
    PRO_Q(6) PRO_Q(7) PRO_Q(8) PRO_Q(9) PRO_Q(10) PRO_Q(11)
#undef PRO_Q
  }
  dma_barrier_but<12>();

  // Fragment of row block I (16 rows) for k-step KS (32 k): lane l holds row
  // l%16, k 8*(l/16) .. +7.
  // K-contiguous images ([row][64], swizzled): one 16-byte read; the unit of
  // k-chunk 4 KS + l/16 depends on KS through the swizzle, so each k-step has
  // its own lane offset, and row block I is a constant 16 rows further (the
  // swizzle has period 16).
  // Row-contiguous images ([64][256 + 32]): two transposing reads of 4 k.
  constexpr int LM = BM + 32;
  int a_frag[2], b_frag[2];
#pragma unroll
  for (int ks = 0; ks < 2; ++ks) {
    const int trl = (32 * ks + 8 * lg + (l16 >> 2)) * LM + (l16 & 3) * 4;
    const int kc = ((4 * ks + lg) ^ kc_swizzle(l16)) * 8;
    a_frag[ks] = A_K ? (wm * 128 + l16) * BK + kc : trl + wm * 128;
    b_frag[ks] = A_IMG + (B_K ? (wn * 128 + l16) * BK + kc : trl + wn * 128);
  }
  // One set of fragments, each re-read as soon as its last MFMA of the
  // k-step has issued.  A k-step's 64 MFMAs run the (row block, column
  // block) pairs column-major, first over row blocks 0-3, then over 4-7:
  //  * A0-A3 die at MFMA 31 and are re-read (next k-step) right after it;
  //  * Bj dies at MFMA 35 + 4j (row block 7) and is re-read right after it,
  //    29 MFMAs before the next k-step's first use (MFMA 4j);
  //  * A4-A7 die at MFMA 63 and are read in the next k-step's first four
  //    gaps, 28 MFMAs before their first use (MFMA 32).
  // The barrier comes 12 MFMAs into the second k-step of a k-tile, after
  // that k-step's own A4-A7 reads from the stage; then direct loads, one
  // every fourth MFMA gap, refill the stage with k-tile t+2 (12 pieces in
  // this k-step, the other 4-6 in the next).
  uint4 fa[8], fb[8];
#define SB __builtin_amdgcn_sched_barrier(0);
#define RD_A(BASE, KS, I)                                                             \
  fa[I] = A_K ? *reinterpret_cast<const uint4*>((BASE) + a_frag[KS] + (I) * 16 * BK) \
              : tr_frag((BASE) + a_frag[KS] + (I) * 16, LM);
#define RD_B(BASE, KS, J)                                                             \
  fb[J] = B_K ? *reinterpret_cast<const uint4*>((BASE) + b_frag[KS] + (J) * 16 * BK) \
              : tr_frag((BASE) + b_frag[KS] + (J) * 16, LM);
#define MM(I, J)                                  \
  if constexpr (A_K && !TAIL)                     \
    acc[I][J] = mfma16<FP16>(fb[J], fa[I], acc[I][J]); \
  else                                            \
    mfma16_asm<FP16>(acc[I][J], fb[J], fa[I]);
  // items 0-11 of k-tile t+2 in the barrier k-step of k-tile t, the rest
  // in the first k-step of k-tile t+1
#define LOAD_CUR(Q) LOAD_Q(Q, cur, rsa2, rsb2, k2)
#define LOAD_NXT(Q) LOAD_Q(Q, nxt, rsa1, rsb1, k1)
#define KSTEP_A(OB, OK, NB, NK)    \
  SB MM(0, 0) SB RD_A(OB, OK, 4) SB MM(1, 0) SB RD_A(OB, OK, 5) SB MM(2, 0) SB RD_A(OB, OK, 6) SB    \
  LOAD_NXT(12) SB MM(3, 0) SB RD_A(OB, OK, 7) SB MM(0, 1) SB MM(1, 1) SB MM(2, 1) SB LOAD_NXT(13) SB \
  MM(3, 1) SB MM(0, 2) SB MM(1, 2) SB MM(2, 2) SB LOAD_NXT(14) SB MM(3, 2) SB MM(0, 3) SB            \
  MM(1, 3) SB MM(2, 3) SB LOAD_NXT(15) SB MM(3, 3) SB MM(0, 4) SB MM(1, 4) SB MM(2, 4) SB            \
  LOAD_NXT(16) SB MM(3, 4) SB MM(0, 5) SB MM(1, 5) SB MM(2, 5) SB LOAD_NXT(17) SB MM(3, 5) SB        \
  MM(0, 6) SB MM(1, 6) SB MM(2, 6) SB MM(3, 6) SB MM(0, 7) SB MM(1, 7) SB MM(2, 7) SB MM(3, 7) SB    \
  MM(4, 0) SB RD_A(NB, NK, 0) SB MM(5, 0) SB RD_A(NB, NK, 1) SB MM(6, 0) SB RD_A(NB, NK, 2) SB       \
  MM(7, 0) SB RD_B(NB, NK, 0) SB MM(4, 1) SB RD_A(NB, NK, 3) SB MM(5, 1) SB MM(6, 1) SB MM(7, 1) SB  \
  RD_B(NB, NK, 1) SB MM(4, 2) SB MM(5, 2) SB MM(6, 2) SB MM(7, 2) SB RD_B(NB, NK, 2) SB MM(4, 3) SB  \
  MM(5, 3) SB MM(6, 3) SB MM(7, 3) SB RD_B(NB, NK, 3) SB MM(4, 4) SB MM(5, 4) SB MM(6, 4) SB         \
  MM(7, 4) SB RD_B(NB, NK, 4) SB MM(4, 5) SB MM(5, 5) SB MM(6, 5) SB MM(7, 5) SB RD_B(NB, NK, 5) SB  \
  MM(4, 6) SB MM(5, 6) SB MM(6, 6) SB MM(7, 6) SB RD_B(NB, NK, 6) SB MM(4, 7) SB MM(5, 7) SB         \
  MM(6, 7) SB MM(7, 7) SB RD_B(NB, NK, 7) SB
#define KSTEP_B(OB, OK, NB, NK)    \
  SB MM(0, 0) SB RD_A(OB, OK, 4) SB MM(1, 0) SB RD_A(OB, OK, 5) SB MM(2, 0) SB RD_A(OB, OK, 6) SB    \
  MM(3, 0) SB RD_A(OB, OK, 7) SB MM(0, 1) SB MM(1, 1) SB MM(2, 1) SB MM(3, 1) SB MM(0, 2) SB         \
  MM(1, 2) SB MM(2, 2) SB MM(3, 2) SB dma_barrier(); SB MM(0, 3) SB LOAD_CUR(0) SB MM(1, 3) SB       \
  MM(2, 3) SB MM(3, 3) SB MM(0, 4) SB LOAD_CUR(1) SB MM(1, 4) SB MM(2, 4) SB MM(3, 4) SB MM(0, 5) SB \
  LOAD_CUR(2) SB MM(1, 5) SB MM(2, 5) SB MM(3, 5) SB MM(0, 6) SB LOAD_CUR(3) SB MM(1, 6) SB          \
  MM(2, 6) SB MM(3, 6) SB MM(0, 7) SB LOAD_CUR(4) SB MM(1, 7) SB MM(2, 7) SB MM(3, 7) SB MM(4, 0) SB \
  LOAD_CUR(5) SB RD_A(NB, NK, 0) SB MM(5, 0) SB RD_A(NB, NK, 1) SB MM(6, 0) SB RD_A(NB, NK, 2) SB    \
  MM(7, 0) SB RD_B(NB, NK, 0) SB MM(4, 1) SB LOAD_CUR(6) SB RD_A(NB, NK, 3) SB MM(5, 1) SB           \
  MM(6, 1) SB MM(7, 1) SB RD_B(NB, NK, 1) SB MM(4, 2) SB LOAD_CUR(7) SB MM(5, 2) SB MM(6, 2) SB      \
  MM(7, 2) SB RD_B(NB, NK, 2) SB MM(4, 3) SB LOAD_CUR(8) SB MM(5, 3) SB MM(6, 3) SB MM(7, 3) SB      \
  RD_B(NB, NK, 3) SB MM(4, 4) SB LOAD_CUR(9) SB MM(5, 4) SB MM(6, 4) SB MM(7, 4) SB                  \
  RD_B(NB, NK, 4) SB MM(4, 5) SB LOAD_CUR(10) SB MM(5, 5) SB MM(6, 5) SB MM(7, 5) SB                 \
  RD_B(NB, NK, 5) SB MM(4, 6) SB LOAD_CUR(11) SB MM(5, 6) SB MM(6, 6) SB MM(7, 6) SB                 \
  RD_B(NB, NK, 6) SB MM(4, 7) SB MM(5, 7) SB MM(6, 7) SB MM(7, 7) SB RD_B(NB, NK, 7) SB

#define ITER(CUR, NXT, KT)                                \
  {                                                       \
    uint16_t* const cur = (CUR);                          \
    uint16_t* const nxt = (NXT);                          \
    const int k1 = kb + ((KT) + 1) * BK;                  \
    const int k2 = kb + ((KT) + 2) * BK;                  \
    const rsrc_t rsa1 = (KT) + 1 < nk ? ra : ra0;         \
    const rsrc_t rsb1 = (KT) + 1 < nk ? rb : rb0;         \
    const rsrc_t rsa2 = (KT) + 2 < nk ? ra : ra0;         \
    const rsrc_t rsb2 = (KT) + 2 < nk ? rb : rb0;         \
    KSTEP_A(cur, 0, cur, 1)                               \
    LIMIT_IF((KT) + 2)                                    \
    KSTEP_B(cur, 1, nxt, 0)                               \
  }
  SB RD_A(smem, 0, 0) SB RD_A(smem, 0, 1) SB RD_A(smem, 0, 2) SB RD_A(smem, 0, 3) SB
#pragma unroll
  for (int j = 0; j < 8; ++j) { RD_B(smem, 0, j) }
  SB
  // two k-tiles per trip, so both LDS stages have fixed addresses (with an
  // odd count the last one is all zeros)
  for (int kt = 0; kt < nk; kt += 2) {
    ITER(smem, smem1, kt)
    ITER(smem1, smem, kt + 1)
  }
  // asm MFMAs: wait states before any instruction reads their accumulators
  if constexpr (!A_K || TAIL) asm volatile("s_nop 7\n\ts_nop 7\n\ts_nop 7" ::: "memory");
#undef PIN_ACC
#undef LIMIT_IF
#undef ITER
#undef KSTEP_A
#undef KSTEP_B
#undef LOAD_Q
#undef LOAD_CUR
#undef LOAD_NXT
#undef MM
#undef RD_A
#undef RD_B
#undef SB

  // Epilogue: each wave stages one 32-row slab of its 128x128 block at a
  // time in its own LDS region (fp32, padded rows) and writes it back as
  // whole rows, two rows per store instruction.  C goes through a buffer
  // resource spanning exactly its extent, so rows past M are dropped by the
  // hardware; lanes whose columns are past N get an out-of-range offset.
  float* stage = reinterpret_cast<float*>(smem) + wid * 32 * ER;
  const int esz = g.c_dtype == ETH_F32 ? 4 : 2;
  const int mode = g.c_dtype == ETH_BF16 ? 0 : g.c_dtype == ETH_F16 ? 1 : (g.flags & ETH_GEMM_ACCUMULATE) ? 3 : 2;
  const rsrc_t rc = make_rsrc(reinterpret_cast<float*>(g.C) + split * g.c_split_stride, g.c_bytes);
  const int32_t row2 = (int32_t)(2 * g.ldc * esz);
  auto write_slab = [&](const int i) __attribute__((always_inline)) {
    // the slab is private to this wave, whose LDS accesses complete in order
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    float4 v[16];
#pragma unroll
    for (int it = 0; it < 16; ++it) {
      v[it] = *reinterpret_cast<const float4*>(stage + (it * 2 + (lane >> 5)) * ER + col);
      v[it].x = v[it].x * g.alpha + bn[0];
      v[it].y = v[it].y * g.alpha + bn[1];
      v[it].z = v[it].z * g.alpha + bn[2];
      v[it].w = v[it].w * g.alpha + bn[3];
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    const int mrow = m0 + wm * 128 + i * 32 + (lane >> 5);
    const int32_t voff = n < g.N ? (int32_t)(((int64_t)mrow * g.ldc + n) * esz) : kOob;
#define OFF(IT) (voff == kOob ? kOob : voff + (IT) * row2)
    if (mode == 0) {
#pragma unroll
      for (int it = 0; it < 16; ++it) {
        u32x2_t o;
        o.x = f2bf_pair(v[it].x, v[it].y);
        o.y = f2bf_pair(v[it].z, v[it].w);
        __builtin_amdgcn_raw_buffer_store_b64(o, rc, OFF(it), 0, 0);
      }
    } else if (mode == 1) {
#pragma unroll
      for (int it = 0; it < 16; ++it) {
        u32x2_t o;
        o.x = f2h_bits(v[it].x) | ((uint32_t)f2h_bits(v[it].y) << 16);
        o.y = f2h_bits(v[it].z) | ((uint32_t)f2h_bits(v[it].w) << 16);
        __builtin_amdgcn_raw_buffer_store_b64(o, rc, OFF(it), 0, 0);
      }
    } else if (mode == 2) {
#pragma unroll
      for (int it = 0; it < 16; ++it)
        __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4_t, v[it]), rc, OFF(it), 0, 0);
    } else {
      // fp32 C += (the main_grad accumulation): all loads first
      u32x4_t old[16];
#pragma unroll
      for (int it = 0; it < 16; ++it) old[it] = __builtin_amdgcn_raw_buffer_load_b128(rc, OFF(it), 0, 0);
#pragma unroll
      for (int it = 0; it < 16; ++it) {
        float4 o = __builtin_bit_cast(float4, old[it]);
        o.x += v[it].x;
        o.y += v[it].y;
        o.z += v[it].z;
        o.w += v[it].w;
        __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4_t, o), rc, OFF(it), 0, 0);
      }
    }
#undef OFF
  };
  dma_barrier();  // every wave is done with the k-loop stages, no load in flight
  // slab S: row blocks 2S, 2S+1 -> staging rows (I % 2) * 16 + lane % 16
#define STAGE_SLAB(S)                                                                     \
  {                                                                                       \
    _Pragma("unroll") for (int h = 0; h < 2; ++h)                                         \
      _Pragma("unroll") for (int j = 0; j < 8; ++j) {                                     \
        const f32x4_t a = acc[2 * (S) + h][j];                                            \
        *reinterpret_cast<float4*>(stage + (h * 16 + l16) * ER + j * 16 + lg * 4) =      \
            make_float4(a[0], a[1], a[2], a[3]);                                          \
      }                                                                                   \
    write_slab(S);                                                                        \
  }
  STAGE_SLAB(0) STAGE_SLAB(1) STAGE_SLAB(2) STAGE_SLAB(3)
#undef STAGE_SLAB
}

// The same tiles with v_mfma_f32_32x32x16 (4 x 4 blocks of 32x32 per wave,
// 16 accumulators per lane each), for a row-contiguous A: with transposing
// reads on both operands the 16x16x32 kernel does not keep its accumulators
// in place in AGPRs (the register allocator moves them around every MFMA).
template <bool A_K, bool B_K, bool FP16>
__global__ void __launch_bounds__(256, 1) gemm256_m32_kernel(GemmArgs g) {
  constexpr int BM = 256, BN = 256, BK = 64;
  typedef DTile<BM, BK, A_K> ATile;
  typedef DTile<BN, BK, B_K> BTile;
  constexpr int A_IMG = ATile::IMG;           // elements of the A image in a stage
  constexpr int STAGE = A_IMG + BTile::IMG;   // one LDS stage: A image then B image
  constexpr int ER = 128 + 4;                 // epilogue staging row (fp32, padded)
  constexpr int EPI = 4 * 32 * ER * 2;        // epilogue staging in elements
  // the two stages are separate arrays, so the compiler can tell the direct
  // loads into one stage from the fragment reads of the other (it would
  // otherwise wait for the loads before every read); the first also holds
  // the epilogue's staging
  __shared__ __attribute__((aligned(16))) uint16_t smem[STAGE > EPI ? STAGE : EPI];
  __shared__ __attribute__((aligned(16))) uint16_t smem1[STAGE];

  const int tiles_m = (g.M + BM - 1) / BM, tiles_n = (g.N + BN - 1) / BN;
  // split-K launches tiles * splits workgroups: split = blockIdx.x / tiles
  const int tiles = tiles_m * tiles_n;
  const int split = blockIdx.x / tiles;
  const int kb = split * g.k_split;
  int tm, tn;
  tile_coords(blockIdx.x - split * tiles, tiles_m, tiles_n, tm, tn);
  const int m0 = tm * BM, n0 = tn * BN;
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  const int wm = wid >> 1, wn = wid & 1;
  const int lr = lane & 31, lk = (lane >> 5) * 8;
  // the 4 output columns this lane writes in the epilogue, and their bias
  // (read now so its latency is hidden behind the k loop)
  const int col = (lane & 31) * 4;
  const int n = n0 + wn * 128 + col;
  float bn[4] = {0.f, 0.f, 0.f, 0.f};
  if ((g.flags & ETH_GEMM_BIAS) && g.bias) {
#pragma unroll
    for (int e = 0; e < 4; ++e)
      if (n + e < g.N) bn[e] = FP16 ? h2f_bits(g.bias[n + e]) : bf2f(g.bias[n + e]);
  }

  f32x16_t acc[4][4];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.f;

  const int nk = (g.k_split ? g.k_split : g.K) / BK;
  const rsrc_t ra = make_rsrc(g.A, g.a_bytes), rb = make_rsrc(g.B, g.b_bytes);
  // empty ranges: the loads issued past the last k-tile read zeros
  const rsrc_t ra0 = make_rsrc(g.A, 0), rb0 = make_rsrc(g.B, 0);
  ATile la;
  BTile lb;
  // pieces per half per wave: 8 for a K-contiguous image, 9 for a padded one
  constexpr int NA = ATile::PER_WAVE, NB = BTile::PER_WAVE;
  static_assert((NA == 8 || NA == 9) && (NB == 8 || NB == 9), "the k loop's load slots");
  la.init(g.lda, m0, g.M);
  lb.init(g.ldb, n0, g.N);
  la.template issue<0, NA>(smem, ra, g.lda, kb);
  lb.template issue<0, NB>(smem + A_IMG, rb, g.ldb, kb);
  // A pieces 0-7 of k-tile 1; the loop's first k-step issues a piece 8
  la.template issue<0, 8>(smem1, nk > 1 ? ra : ra0, g.lda, kb + BK);
  dma_barrier_but<8>();

  // fragment of (row block I, k-step KS): lanes 0-31 hold rows, lanes 32-63
  // the second 8 k of the 16
  // K-contiguous tiles: [row][64] swizzled, one 16-byte read per fragment
  // (the unit of k-chunk 2 KS + lane / 32 depends on KS through the
  // swizzle, so each k-step has its own lane offset; row block I is a
  // constant 32 rows further, with the same swizzle);
  // row-contiguous tiles: [BK][256 + 32], two transposing reads (tr_frag)
  constexpr int LM = BM + 32;
  const int trl = ((lane >> 5) * 8 + ((lane & 15) >> 2)) * LM + ((lane >> 4) & 1) * 16 + (lane & 3) * 4;
  int a_frag[4], b_frag[4];
#pragma unroll
  for (int ks = 0; ks < 4; ++ks) {
    const int ra_ = wm * 128 + lr, rb_ = wn * 128 + lr;
    a_frag[ks] = A_K ? ra_ * BK + ((2 * ks + (lane >> 5)) ^ kc_swizzle(ra_)) * 8 : trl + wm * 128 + ks * 16 * LM;
    b_frag[ks] = A_IMG + (B_K ? rb_ * BK + ((2 * ks + (lane >> 5)) ^ kc_swizzle(rb_)) * 8 : trl + wn * 128 + ks * 16 * LM);
  }
  uint4 fa0[4], fb0[4], fa1[4], fb1[4];
#define SB __builtin_amdgcn_sched_barrier(0);
#define RD_A(FA, BASE, KS, I)                                                         \
  FA[I] = A_K ? *reinterpret_cast<const uint4*>((BASE) + a_frag[KS] + (I) * 32 * BK) \
              : tr_frag((BASE) + a_frag[KS] + (I) * 32, LM);
#define RD_B(FB, BASE, KS, J)                                                         \
  FB[J] = B_K ? *reinterpret_cast<const uint4*>((BASE) + b_frag[KS] + (J) * 32 * BK) \
              : tr_frag((BASE) + b_frag[KS] + (J) * 32, LM);
// B fragment as the MFMA's first operand: the lane then holds 4 consecutive
// output columns (r % 4) of one output row (lane % 32)
#define MMA2(FA, FB, I, J0)                                         \
  acc[I][J0] = mfma32<FP16>(FB[J0], FA[I], acc[I][J0]);             \
  acc[I][J0 + 1] = mfma32<FP16>(FB[J0 + 1], FA[I], acc[I][J0 + 1]);
// next k-step's fragments in the order its MFMA pairs consume them:
// B0 B1 A0 B2 B3 A1 A2 A3
#define RD_SEQ0(GA, GB, RB, RK) RD_B(GB, RB, RK, 0)
#define RD_SEQ1(GA, GB, RB, RK) RD_B(GB, RB, RK, 1)
#define RD_SEQ2(GA, GB, RB, RK) RD_A(GA, RB, RK, 0)
#define RD_SEQ3(GA, GB, RB, RK) RD_B(GB, RB, RK, 2)
#define RD_SEQ4(GA, GB, RB, RK) RD_B(GB, RB, RK, 3)
#define RD_SEQ5(GA, GB, RB, RK) RD_A(GA, RB, RK, 1)
#define RD_SEQ6(GA, GB, RB, RK) RD_A(GA, RB, RK, 2)
#define RD_SEQ7(GA, GB, RB, RK) RD_A(GA, RB, RK, 3)
#define MMA1(FA, FB, I, J) acc[I][J] = mfma32<FP16>(FB[J], FA[I], acc[I][J]);
// one row block of a k-step: 4 MFMAs, with two fragment reads of the next
// k-step into (GA, GB) and two direct-load slots of a tile cycle between them
#define KSTEP_ROW(FA, FB, GA, GB, RB, RK, I, S0, S1, CYC)                                        \
  SB MMA1(FA, FB, I, 0) SB S0(GA, GB, RB, RK) SB MMA1(FA, FB, I, 1) SB CYC(2 * (I)) SB MMA1(FA, FB, I, 2) \
  SB S1(GA, GB, RB, RK) SB MMA1(FA, FB, I, 3) SB CYC(2 * (I) + 1) SB
#define NOCYC(P)
// direct-load slot S (0-7) of a k-step issues one 1 KB piece: pieces 0-7
// of the A half of k-tile t+2 in the k-step after the barrier, then, one
// per slot over the next k-step and a half, the rest of k-tile t+2 (queue
// position Q: A piece 8 first when the A image has 9 pieces, then the B
// pieces) -- one load per slot, so no slot stalls the MFMA issue on a burst
// of loads (measured 3% faster than two bursts of 9)
#define CYC_A(S) la.template issue<(S), (S) + 1>(cur, rsa, g.lda, k2);
#define LOAD_Q(Q)                                                                            \
  if constexpr (NA == 9 && (Q) == 0)                                                         \
    la.template issue<8, 9>(nxt, rsa1, g.lda, k1);                                           \
  else if constexpr ((Q) - (NA - 8) < NB)                                                    \
    lb.template issue<(Q) - (NA - 8), (Q) - (NA - 8) + 1>(nxt + A_IMG, rsb, g.ldb, k1);
#define CYC_AB(S) LOAD_Q(S)
#define CYC_B2(S) LOAD_Q((S) + 8)
#define KSTEP(FA, FB, GA, GB, RB, RK, CYC)                     \
  KSTEP_ROW(FA, FB, GA, GB, RB, RK, 0, RD_SEQ0, RD_SEQ1, CYC) \
  KSTEP_ROW(FA, FB, GA, GB, RB, RK, 1, RD_SEQ2, RD_SEQ3, CYC) \
  KSTEP_ROW(FA, FB, GA, GB, RB, RK, 2, RD_SEQ4, RD_SEQ5, CYC) \
  KSTEP_ROW(FA, FB, GA, GB, RB, RK, 3, RD_SEQ6, RD_SEQ7, CYC) SB
// k-tile KT: k-steps 0-2 from stage CUR while the rest of k-tile KT+1 is
// loaded into NXT (most of its A half was started one k-step earlier); the
// barrier (after this wave's direct loads have landed) means every wave is
// done reading CUR and KT+1 is complete in NXT; k-step 3 then computes from
// registers, reads the first fragments of KT+1 from NXT and starts the A
// half of k-tile KT+2 into CUR
#define ITER(CUR, NXT, KT)                              \
  {                                                     \
    uint16_t* const cur = (CUR);                        \
    uint16_t* const nxt = (NXT);                        \
    const int k1 = kb + ((KT) + 1) * BK;                \
    const int k2 = kb + ((KT) + 2) * BK;                \
    const rsrc_t rsb = (KT) + 1 < nk ? rb : rb0;        \
    const rsrc_t rsa = (KT) + 2 < nk ? ra : ra0;        \
    const rsrc_t rsa1 = (KT) + 1 < nk ? ra : ra0;       \
    KSTEP(fa0, fb0, fa1, fb1, cur, 1, CYC_AB)           \
    KSTEP(fa1, fb1, fa0, fb0, cur, 2, CYC_B2)           \
    KSTEP(fa0, fb0, fa1, fb1, cur, 3, NOCYC)            \
    dma_barrier();                                      \
    KSTEP(fa1, fb1, fa0, fb0, nxt, 0, CYC_A)            \
  }
  SB RD_SEQ0(fa0, fb0, smem, 0) SB RD_SEQ1(fa0, fb0, smem, 0) SB RD_SEQ2(fa0, fb0, smem, 0) SB
  RD_SEQ3(fa0, fb0, smem, 0) SB RD_SEQ4(fa0, fb0, smem, 0) SB RD_SEQ5(fa0, fb0, smem, 0) SB
  RD_SEQ6(fa0, fb0, smem, 0) SB RD_SEQ7(fa0, fb0, smem, 0) SB
  // two k-tiles per trip, so both LDS stages have fixed addresses
  for (int kt = 0; kt < nk; kt += 2) {
    ITER(smem, smem1, kt)
    ITER(smem1, smem, kt + 1)
  }
#undef ITER
#undef KSTEP
#undef CYC_A
#undef CYC_AB
#undef CYC_B2
#undef LOAD_Q
#undef MMA1
#undef NOCYC
#undef KSTEP_ROW
#undef RD_SEQ0
#undef RD_SEQ1
#undef RD_SEQ2
#undef RD_SEQ3
#undef RD_SEQ4
#undef RD_SEQ5
#undef RD_SEQ6
#undef RD_SEQ7
#undef MMA2
#undef RD_A
#undef RD_B
#undef SB

  // Epilogue: each wave stages one 32-row slab of its 128x128 block at a
  // time in its own LDS region (fp32, padded rows) and writes it back as
  // whole rows, two rows per store instruction.  C goes through a buffer
  // resource spanning exactly its extent, so rows past M are dropped by the
  // hardware; lanes whose columns are past N get an out-of-range offset.
  float* stage = reinterpret_cast<float*>(smem) + wid * 32 * ER;
  const int esz = g.c_dtype == ETH_F32 ? 4 : 2;
  const int mode = g.c_dtype == ETH_BF16 ? 0 : g.c_dtype == ETH_F16 ? 1 : (g.flags & ETH_GEMM_ACCUMULATE) ? 3 : 2;
  const rsrc_t rc = make_rsrc(reinterpret_cast<float*>(g.C) + split * g.c_split_stride, g.c_bytes);
  const int32_t row2 = (int32_t)(2 * g.ldc * esz);
  auto write_slab = [&](const int i) __attribute__((always_inline)) {
    // the slab is private to this wave, whose LDS accesses complete in order
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    float4 v[16];
#pragma unroll
    for (int it = 0; it < 16; ++it) {
      v[it] = *reinterpret_cast<const float4*>(stage + (it * 2 + (lane >> 5)) * ER + col);
      v[it].x = v[it].x * g.alpha + bn[0];
      v[it].y = v[it].y * g.alpha + bn[1];
      v[it].z = v[it].z * g.alpha + bn[2];
      v[it].w = v[it].w * g.alpha + bn[3];
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    const int mrow = m0 + wm * 128 + i * 32 + (lane >> 5);
    const int32_t voff = n < g.N ? (int32_t)(((int64_t)mrow * g.ldc + n) * esz) : kOob;
#define OFF(IT) (voff == kOob ? kOob : voff + (IT) * row2)
    if (mode == 0) {
#pragma unroll
      for (int it = 0; it < 16; ++it) {
        u32x2_t o;
        o.x = f2bf_pair(v[it].x, v[it].y);
        o.y = f2bf_pair(v[it].z, v[it].w);
        __builtin_amdgcn_raw_buffer_store_b64(o, rc, OFF(it), 0, 0);
      }
    } else if (mode == 1) {
#pragma unroll
      for (int it = 0; it < 16; ++it) {
        u32x2_t o;
        o.x = f2h_bits(v[it].x) | ((uint32_t)f2h_bits(v[it].y) << 16);
        o.y = f2h_bits(v[it].z) | ((uint32_t)f2h_bits(v[it].w) << 16);
        __builtin_amdgcn_raw_buffer_store_b64(o, rc, OFF(it), 0, 0);
      }
    } else if (mode == 2) {
#pragma unroll
      for (int it = 0; it < 16; ++it)
        __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4_t, v[it]), rc, OFF(it), 0, 0);
    } else {
      // fp32 C += (the main_grad accumulation): all loads first
      u32x4_t old[16];
#pragma unroll
      for (int it = 0; it < 16; ++it) old[it] = __builtin_amdgcn_raw_buffer_load_b128(rc, OFF(it), 0, 0);
#pragma unroll
      for (int it = 0; it < 16; ++it) {
        float4 o = __builtin_bit_cast(float4, old[it]);
        o.x += v[it].x;
        o.y += v[it].y;
        o.z += v[it].z;
        o.w += v[it].w;
        __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4_t, o), rc, OFF(it), 0, 0);
      }
    }
#undef OFF
  };
  dma_barrier();  // every wave is done with the k-loop stages, no load in flight
#define STAGE_SLAB(I)                                                                  \
  {                                                                                    \
    _Pragma("unroll") for (int j = 0; j < 4; ++j)                                      \
      _Pragma("unroll") for (int q = 0; q < 4; ++q) {                                  \
        const float4 o = make_float4(acc[I][j][q * 4 + 0], acc[I][j][q * 4 + 1],       \
                                     acc[I][j][q * 4 + 2], acc[I][j][q * 4 + 3]);      \
        *reinterpret_cast<float4*>(stage + lr * ER + j * 32 + q * 8 + (lane >> 5) * 4) = o; \
      }                                                                                \
    write_slab(I);                                                                     \
  }
  STAGE_SLAB(0) STAGE_SLAB(1) STAGE_SLAB(2) STAGE_SLAB(3)
#undef STAGE_SLAB
}

// TILE x TILE x 64 tiles (128 or 64) on 4 waves in a 2 x 2 grid, four LDS
// stages filled by direct loads up to four k-tiles ahead.  With one or two
// small tiles per CU no other workgroup hides the load latency, so the ring
// does; per k-tile one barrier, set between the two k-steps:
//   k-step 0: the MFMAs of the fragments already in registers run while the
//             fragments of k-step 1 are read;
//   barrier:  this k-tile's LDS reads are done in every wave (its stage is
//             free) and the next k-tile has landed;
//   k-step 1: its MFMAs run while the first fragments of the next k-tile are
//             read, and k-tile t + 4 streams into the freed stage.
// LDS images carry no padding: K-contiguous operands as in DTile,
// row-contiguous ones [64][ROWS] with 16-byte chunk c of k-row k at
// c ^ rc_swizzle(k), so the four k-rows (eight, for two 16-lane groups) that a
// transposing read touches lie in distinct banks.  Any K % 8 == 0 (the last
// k-tile's missing chunks read zeros through an out-of-range offset), any M, N
// and C alignment.  Bound by LDS and L2: a 128x128 k-tile writes 32 KB to LDS
// and reads 64 KB (768 cycles at 128 B/clk) for 512 MFMA cycles, and takes
// about 1000; a 64x64 one has half the work per byte.  The register-staged
// double-buffered tiles it replaced took 57 us for [1024, 1024] x 4096 deep
// (now 17), 33 us for [2048, 2048] x 2048 (24), 139 us for the 8192-deep data
// gradient of the same output (80).
template <int ROWS>
__device__ __forceinline__ int rc_swizzle(int k) {
  return ROWS == 128 ? ((k & 3) << 1) | (((k >> 3) & 1) << 3) : (((k >> 1) & 1) << 1) | (((k >> 3) & 1) << 2);
}
template <int ROWS, bool KC>
struct RingTile {
  static constexpr int UPR = KC ? 8 : ROWS / 8;  // 16-byte units per LDS row
  static constexpr int PER_WAVE = ROWS * 8 / 256;
  static constexpr int IMG = ROWS * 64;
  int32_t off[PER_WAVE];
  int kof[PER_WAVE];  // k of the lane's unit within the k-tile
  int wave;
  __device__ __forceinline__ void init(int64_t ld, int r0, int rows) {
    wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int lane = threadIdx.x & 63;
#pragma unroll
    for (int j = 0; j < PER_WAVE; ++j) {
      const int u = (wave * PER_WAVE + j) * 64 + lane;
      const int line = u / UPR, c = u % UPR;
      const int r = KC ? line : (c ^ rc_swizzle<ROWS>(line)) * 8;
      kof[j] = KC ? (c ^ kc_swizzle(line)) * 8 : line;
      off[j] = r0 + r < rows ? (int32_t)((KC ? (int64_t)(r0 + r) * ld + kof[j] : (int64_t)kof[j] * ld + r0 + r) * 2)
                             : kOob;
    }
  }
  // k-tile [k0, k0 + 64) into the image at S; k at or past kend reads zeros
  // (one compare and select per load, and no second path)
  __device__ __forceinline__ void issue(uint16_t* S, rsrc_t rs, int64_t ld, int k0, int kend) {
    const int32_t soff = k0 < kend ? (KC ? k0 * 2 : (int32_t)((int64_t)k0 * ld * 2)) : 0;
    const int left = kend - k0;
#pragma unroll
    for (int j = 0; j < PER_WAVE; ++j)
      dma16(rs, S + (wave * PER_WAVE + j) * 512, kof[j] < left ? off[j] : kOob, soff);
  }
};

template <int TILE, bool A_K, bool B_K, bool FP16>
__global__ void __launch_bounds__(256, 1) gemm_ring_kernel(GemmArgs g) {
  constexpr int BM = TILE, BN = TILE;
  constexpr int WM = BM / 2, WN = BN / 2;    // a wave's block
  constexpr int TI = WM / 16, TJ = WN / 16;  // of 16 x 16 MFMA blocks
  typedef RingTile<BM, A_K> ATile;
  typedef RingTile<BN, B_K> BTile;
  constexpr int A_IMG = ATile::IMG, STAGE = A_IMG + BTile::IMG;
  constexpr int PPW = ATile::PER_WAVE + BTile::PER_WAVE;  // direct loads of a wave per k-tile
  constexpr int ER = WN + 4;                              // epilogue staging row (fp32, padded)
  static_assert(4 * 16 * ER * 4 <= 2 * STAGE, "the epilogue's staging fits a stage");
  // separate arrays, so the compiler can tell the direct loads into one
  // stage from the fragment reads of another
  __shared__ __attribute__((aligned(16))) uint16_t st0[STAGE];
  __shared__ __attribute__((aligned(16))) uint16_t st1[STAGE];
  __shared__ __attribute__((aligned(16))) uint16_t st2[STAGE];
  __shared__ __attribute__((aligned(16))) uint16_t st3[STAGE];

  const int tiles_m = (g.M + BM - 1) / BM, tiles_n = (g.N + BN - 1) / BN;
  int tm, tn;
  tile_coords(blockIdx.x, tiles_m, tiles_n, tm, tn);
  const int m0 = tm * BM, n0 = tn * BN;
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  const int wm = wid >> 1, wn = wid & 1;
  const int l16 = lane & 15, lg = lane >> 4;
  const int nk = (g.K + 63) / 64;

  const rsrc_t ra = make_rsrc(g.A, g.a_bytes), rb = make_rsrc(g.B, g.b_bytes);
  ATile la;
  BTile lb;
  la.init(g.lda, m0, g.M);
  lb.init(g.ldb, n0, g.N);
#define RING_ISSUE(S, KT)                              \
  {                                                    \
    la.issue(S, ra, g.lda, (KT) * 64, g.K);            \
    lb.issue((S) + A_IMG, rb, g.ldb, (KT) * 64, g.K);  \
  }
  RING_ISSUE(st0, 0)
  RING_ISSUE(st1, 1)
  RING_ISSUE(st2, 2)
  RING_ISSUE(st3, 3)

  f32x4_t acc[TI][TJ];
#pragma unroll
  for (int i = 0; i < TI; ++i)
#pragma unroll
    for (int j = 0; j < TJ; ++j) acc[i][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};

  // lane offsets of the fragments of k-step 0 (k-step 1: see frag): lane l
  // holds row l%16 of the block, k 8*(l/16) .. +7
  int aof[TI], bof[TJ];
#pragma unroll
  for (int i = 0; i < TI; ++i)
    aof[i] = A_K ? (wm * WM + i * 16 + l16) * 64 + ((lg ^ kc_swizzle(l16)) * 8)
                 : (8 * lg + (l16 >> 2)) * BM +
                       ((((wm * WM + i * 16) >> 3) + ((l16 & 3) >> 1)) ^ rc_swizzle<BM>(8 * lg + (l16 >> 2))) * 8 +
                       (l16 & 1) * 4;
#pragma unroll
  for (int j = 0; j < TJ; ++j)
    bof[j] = A_IMG + (B_K ? (wn * WN + j * 16 + l16) * 64 + ((lg ^ kc_swizzle(l16)) * 8)
                          : (8 * lg + (l16 >> 2)) * BN +
                                ((((wn * WN + j * 16) >> 3) + ((l16 & 3) >> 1)) ^
                                 rc_swizzle<BN>(8 * lg + (l16 >> 2))) * 8 +
                                (l16 & 1) * 4);
  uint4 fa[2][TI], fb[2][TJ];
  // k-step 1: chunk 4 + lg is chunk lg with bit 2 flipped (K-contiguous);
  // 32 k-rows further, where rc_swizzle repeats (row-contiguous)
  auto read = [&](auto ks_c, const uint16_t* S) __attribute__((always_inline)) {
    constexpr int ks = decltype(ks_c)::value;
#pragma unroll
    for (int i = 0; i < TI; ++i)
      fa[ks][i] = A_K ? *reinterpret_cast<const uint4*>(S + (aof[i] ^ (ks * 32)))
                      : tr_frag(S + aof[i] + ks * 32 * BM, BM);
#pragma unroll
    for (int j = 0; j < TJ; ++j)
      fb[ks][j] = B_K ? *reinterpret_cast<const uint4*>(S + (bof[j] ^ (ks * 32)))
                      : tr_frag(S + bof[j] + ks * 32 * BN, BN);
  };
  // column blocks [J0, J1) of k-step ks
  auto products = [&](auto ks_c, const int J0, const int J1) __attribute__((always_inline)) {
    constexpr int ks = decltype(ks_c)::value;
#pragma unroll
    for (int j = J0; j < J1; ++j)
#pragma unroll
      for (int i = 0; i < TI; ++i) mfma16_tied<FP16>(acc[i][j], fb[ks][j], fa[ks][i]);
  };
  typedef std::integral_constant<int, 0> K0;
  typedef std::integral_constant<int, 1> K1;
  dma_barrier_but<3 * PPW>();
  read(K0{}, st0);
  __builtin_amdgcn_sched_barrier(0);
#define RING_STEP(S, SN, KT)                \
  {                                         \
    products(K0{}, 0, 1);                   \
    __builtin_amdgcn_sched_barrier(0);      \
    read(K1{}, S);                          \
    products(K0{}, 1, TJ);                  \
    __builtin_amdgcn_sched_barrier(0);      \
    dma_barrier_but<2 * PPW>();             \
    RING_ISSUE(S, (KT) + 4)                 \
    __builtin_amdgcn_sched_barrier(0);      \
    read(K0{}, SN);                         \
    products(K1{}, 0, TJ);                  \
    __builtin_amdgcn_sched_barrier(0);      \
  }
  int kt = 0;
  for (; kt + 4 <= nk; kt += 4) {
    RING_STEP(st0, st1, kt)
    RING_STEP(st1, st2, kt + 1)
    RING_STEP(st2, st3, kt + 2)
    RING_STEP(st3, st0, kt + 3)
  }
  if (kt < nk) RING_STEP(st0, st1, kt)
  if (kt + 1 < nk) RING_STEP(st1, st2, kt + 1)
  if (kt + 2 < nk) RING_STEP(st2, st3, kt + 2)
  // asm MFMAs: wait states before any instruction reads their accumulators
  asm volatile("s_nop 7\n\ts_nop 7\n\ts_nop 7" ::: "memory");
#undef RING_STEP
#undef RING_ISSUE
  dma_barrier();  // every load landed, every wave done with the stages

  // Epilogue: 16-row slabs of the wave's block through its own LDS region,
  // out in whole rows of WN columns
  float* stage = reinterpret_cast<float*>(st0) + wid * 16 * ER;
  constexpr int LPR = WN / 4, RPI = 64 / LPR;  // lanes per row (4 columns each), rows per pass
  const int col = (lane % LPR) * 4, n = n0 + wn * WN + col;
  const bool has_bias = (g.flags & ETH_GEMM_BIAS) && g.bias;
  const bool add = g.flags & ETH_GEMM_ACCUMULATE;
  float bn[4] = {0.f, 0.f, 0.f, 0.f};
  if (has_bias) {
#pragma unroll
    for (int e = 0; e < 4; ++e)
      if (n + e < g.N) bn[e] = FP16 ? h2f_bits(g.bias[n + e]) : bf2f(g.bias[n + e]);
  }
#pragma unroll
  for (int i = 0; i < TI; ++i) {
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // the last slab's reads
#pragma unroll
    for (int j = 0; j < TJ; ++j)
      *reinterpret_cast<f32x4_t*>(stage + l16 * ER + j * 16 + lg * 4) = acc[i][j];
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // private to this wave
#pragma unroll
    for (int p = 0; p < 16 / RPI; ++p) {
      const int r = p * RPI + lane / LPR, m = m0 + wm * WM + i * 16 + r;
      f32x4_t v = *reinterpret_cast<const f32x4_t*>(stage + r * ER + col);
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = v[e] * g.alpha + bn[e];
      if (m >= g.M || n >= g.N) continue;
      const int64_t o = (int64_t)m * g.ldc + n;
      if (g.c_vec) {
        if (g.c_dtype == ETH_F32) {
          f32x4_t* c = reinterpret_cast<f32x4_t*>(reinterpret_cast<float*>(g.C) + o);
          *c = add ? *c + v : v;
        } else {
          u32x2_t w;
          if (g.c_dtype == ETH_BF16) {
            w.x = f2bf_pair(v[0], v[1]);
            w.y = f2bf_pair(v[2], v[3]);
          } else {
            w.x = f2h_bits(v[0]) | ((uint32_t)f2h_bits(v[1]) << 16);
            w.y = f2h_bits(v[2]) | ((uint32_t)f2h_bits(v[3]) << 16);
          }
          *reinterpret_cast<u32x2_t*>(reinterpret_cast<uint16_t*>(g.C) + o) = w;
        }
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          if (n + e >= g.N) break;
          if (g.c_dtype == ETH_F32) {
            float* c = reinterpret_cast<float*>(g.C) + o + e;
            *c = add ? *c + v[e] : v[e];
          } else {
            reinterpret_cast<uint16_t*>(g.C)[o + e] = g.c_dtype == ETH_BF16 ? f2bf(v[e]) : f2h_bits(v[e]);
          }
        }
      }
    }
  }
}

template <int TILE, bool FP16>
static int launch_ring(const GemmArgs& a, int a_k, int b_k, hipStream_t s) {
  const int tiles = ((a.M + TILE - 1) / TILE) * ((a.N + TILE - 1) / TILE);
  if (a_k && b_k)
    gemm_ring_kernel<TILE, true, true, FP16><<<tiles, 256, 0, s>>>(a);
  else if (a_k && !b_k)
    gemm_ring_kernel<TILE, true, false, FP16><<<tiles, 256, 0, s>>>(a);
  else if (!a_k && !b_k)
    gemm_ring_kernel<TILE, false, false, FP16><<<tiles, 256, 0, s>>>(a);
  else
    gemm_ring_kernel<TILE, false, true, FP16><<<tiles, 256, 0, s>>>(a);
  ETH_CHECK_LAUNCH("eth_gemm");
  return ETH_OK;
}

// What a product's time depends on besides its sizes: an fp32 output (the
// accumulating epilogue reads C too), and operands whose rows start off
// 128-byte lines, where every load touches a line more: both K-contiguous
// (skew_k), or one or two row-contiguous (skew_r).  Sizes stand for strides:
// rows are rarely padded.
struct GemmForm {
  bool f32, skew_k;
  int skew_r;
};
static GemmForm gemm_form(int64_t M, int64_t N, int64_t K, int a_kcontig, int b_kcontig, bool f32) {
  return GemmForm{f32, a_kcontig && b_kcontig && K % 64 != 0,
                  (!a_kcontig && M % 64 != 0) + (!b_kcontig && N % 64 != 0)};
}

// Microseconds one launch of TILE x TILE tiles takes, fitted to sweeps (within
// about 15 %): rounds of one workgroup per CU (two for 64x64, whose 64 KB of
// LDS leaves room for a second) times the k-tiles of 64 at the measured pace
// plus the prologue and epilogue.  A 256x256 k-tile runs faster when half the
// CUs idle (more clock and bandwidth for the rest), in a last round too, and
// at full pace with a full one.  Past one round deep products on 64x64 tiles
// lose the L2 (their workgroups drift apart in k), and rows off 128-byte lines
// cost them most.  Measured where an earlier form of this was wrong (us):
// weight gradients on wide tiles / two splits, [3328, 2048] x 3584 tokens 74 /
// 66, [1536, 3200] x 2560 54 / 47; on 64x64 / two splits, [2456, 1544] x 10240
// 209 / 106; 128x128 / wide, [9216, 832] x 2688 60 / 53, [600, 12816] x 1792
// 45 / 38; forward with K off a line, wide / 128x128, [2176, 3072] x 1000
// 30.3 / 32.3, wide / 64x64, [768, 7936] x 2016 45.9 / 48.3, wide / two
// splits, [1008, 6640] x 3928 89 / 69.
static double tile_time(int tile, int64_t M, int64_t N, int64_t K, int splits, GemmForm form) {
  const double tiles = (double)((M + tile - 1) / tile) * (double)((N + tile - 1) / tile) * splits;
  const double nk = (double)(((K + splits - 1) / splits + 63) / 64);
  const double f = form.f32 && splits == 1 ? 1.0 : 0.0, ring = form.skew_k ? 1.1 : 1.0;
  if (tile == 256) {
    const double rounds = floor(tiles / 256), last = tiles - 256 * rounds, edge = 9.0 + 4.8 * f;
    double pace = 0.93 + 0.27 * std::max(0.0, last - 128) / 128;
    if (form.skew_k) pace = std::max(pace, 1.08);
    return 3.0 + rounds * (nk * 1.20 + edge) + (last > 0 ? nk * pace + edge : 0.0);
  }
  if (tile == 128) return 2.0 + ceil(tiles / 256) * (nk * 0.52 * ring + 6.0 + 3.3 * f);
  if (tiles <= 256) return 3.0 + nk * 0.24 * (ring + 0.08 * form.skew_r) + 0.8 * f;
  const double deep = std::min(1.0, std::max(0.0, (nk - 32.0) / 96.0));
  const double lines = form.skew_k ? 0.2 : 0.2 * form.skew_r;
  return 1.0 + ceil(tiles / 512) * (nk * 0.36 * (1.0 + lines + 0.3 * deep) + 2.7 + 1.5 * f);
}

// The tile that finishes first.  Measured on both sides of the lines (us, 256
// / 128 / 64): [2048, 2048] x 2048 deep 39 / 24 / 29, [2048, 6144] x 2048 45 /
// 66 / 76, [1024, 1024] x 4096 69 / 37 / 17, [1024, 4096] x 1024 24 / 16 / 18,
// [3000, 2560] x 2560 48 / 53 / 66.
static int plan_tile(int64_t M, int64_t N, int64_t K, bool wide, GemmForm form) {
  int best = 64;
  double t = tile_time(64, M, N, K, 1, form);
  for (int tile : {128, 256}) {
    if (tile == 256 && !wide) continue;
    const double u = tile_time(tile, M, N, K, 1, form);
    if (u <= t) {
      t = u;
      best = tile;
    }
  }
  return best;
}

template <bool FP16>
static int launch_256(const GemmArgs& a, int a_k, int b_k, hipStream_t s, int splits = 1) {
  const int tiles = ((a.M + 255) / 256) * ((a.N + 255) / 256) * splits;
  const bool tail = a.K % 64;
  if (a_k && b_k)
    tail ? gemm256_m16_kernel<true, true, FP16, true><<<tiles, 256, 0, s>>>(a)
         : gemm256_m16_kernel<true, true, FP16><<<tiles, 256, 0, s>>>(a);
  else if (a_k)
    tail ? gemm256_m16_kernel<true, false, FP16, true><<<tiles, 256, 0, s>>>(a)
         : gemm256_m16_kernel<true, false, FP16><<<tiles, 256, 0, s>>>(a);
  else if (!b_k)
    tail ? gemm256_m16_kernel<false, false, FP16, true><<<tiles, 256, 0, s>>>(a)
         : gemm256_m16_kernel<false, false, FP16><<<tiles, 256, 0, s>>>(a);
  else  // (m32: pairs of whole k-tiles, in every split alike)
    a.K % (a.k_split ? a.k_split : 128) || a.k_split % 128
        ? gemm256_m16_kernel<false, true, FP16, true><<<tiles, 256, 0, s>>>(a)
        : gemm256_m32_kernel<false, true, FP16><<<tiles, 256, 0, s>>>(a);
  ETH_CHECK_LAUNCH("eth_gemm");
  return ETH_OK;
}

// The rows and columns of C to give whole rounds of 256x256 tiles, the rest
// going to a second launch in its own best tile: a grid a little over a whole
// number of rounds otherwise spends a full round on it ([7680, 2560] x 3000:
// 300 tiles, 136 us in two rounds, 125 us as 250 tiles and 200 of 128x128).
// Taken where the model promises 7 %; all of C where not.  Also measured
// (us): [6144, 2816] x 2816 113 -> 80, [4400, 4608] x 1536 70 -> 63,
// [2500, 8192] x 2048 87 -> 77, [1024, 50304] x 1024 107 -> 97.
// From 1024 deep on and where the last round holds 24 to 128 tiles, 2 % will
// do: 68 measured there ran at 0.916 to 1.010 of one launch, 0.964 in the
// mean ([2048, 50304] x 2048 347 -> 329, its weight gradient 407 -> 377,
// [8472, 10176] x 3392 446 -> 424, [14400, 4800] x 1600 216 -> 217).  On the
// other sides a promise of 2 to 7 % was not kept: shallower 0.95 to 1.13
// ([2832, 50304] x 512 201 -> 227), fewer tiles left 0.99 to 1.03 (they start
// on the CUs that end a round early), more 1.00 to 1.03 ([2344, 50304] x 3072
// 592 -> 607).
struct GemmCut {
  int64_t m, n;
};
static GemmCut plan_cut(int64_t M, int64_t N, int64_t K, bool wide, GemmForm form) {
  GemmCut best{M, N};
  if (!wide) return best;
  const int tile = plan_tile(M, N, K, wide, form);
  const int64_t tm = (M + 255) / 256, tn = (N + 255) / 256, rounds = tm * tn / 256;
  if (tile != 256 || rounds < 1 || tm * tn % 256 == 0) return best;
  const int64_t last = tm * tn % 256;
  double t = (K >= 1024 && last >= 24 && last <= 128 ? 0.98 : 0.93) * tile_time(256, M, N, K, 1, form);
  auto rest = [&](int64_t m, int64_t n) { return tile_time(plan_tile(m, n, K, wide, form), m, n, K, 1, form); };
  const int64_t m1 = rounds * 256 / tn * 256, n1 = rounds * 256 / tm * 256;
  if (m1 > 0 && m1 < M) {
    const double u = tile_time(256, m1, N, K, 1, form) + rest(M - m1, N);
    if (u < t) {
      t = u;
      best = GemmCut{m1, N};
    }
  }
  if (n1 > 0 && n1 < N) {
    const double u = tile_time(256, M, n1, K, 1, form) + rest(M, N - n1);
    if (u < t) best = GemmCut{M, n1};
  }
  return best;
}

// The 256x256 kernels take C rows of whole four-column vectors (vector stores)
// and a C extent plus one tile of rows below 2 GiB (their buffer offsets).
static bool wide_takes(int64_t M, int64_t N, int64_t ldc, int esz, bool c_vec) {
  return c_vec && ((M + 255) * ldc + N) * esz < (1LL << 31);
}

static int launch_planned(const GemmArgs& a, int a_k, int b_k, bool fp16, bool wide, GemmForm form, hipStream_t s) {
  switch (plan_tile(a.M, a.N, a.K, wide, form)) {
    case 256:
      return fp16 ? launch_256<true>(a, a_k, b_k, s) : launch_256<false>(a, a_k, b_k, s);
    case 128:
      return fp16 ? launch_ring<128, true>(a, a_k, b_k, s) : launch_ring<128, false>(a, a_k, b_k, s);
    default:
      return fp16 ? launch_ring<64, true>(a, a_k, b_k, s) : launch_ring<64, false>(a, a_k, b_k, s);
  }
}

}  // namespace eth

using namespace eth;

extern "C" int eth_gemm(const void* A, int64_t lda, int a_kcontig, const void* B, int64_t ldb,
                        int b_kcontig, void* C, int64_t ldc, int c_dtype, const void* bias,
                        int64_t M, int64_t N, int64_t K, int in_dtype, int flags, float alpha,
                        void* stream) {
  ETH_CHECK_ARG(in_dtype == ETH_BF16 || in_dtype == ETH_F16, "eth_gemm: inputs must be bf16 or fp16");
  ETH_CHECK_ARG(valid_dtype(c_dtype), "eth_gemm: bad output dtype %d", c_dtype);
  ETH_CHECK_ARG(M > 0 && N > 0 && K > 0 && M < (1LL << 31) && N < (1LL << 31) && K < (1LL << 31),
                "eth_gemm: bad shape %lld x %lld x %lld", (long long)M, (long long)N, (long long)K);
  ETH_CHECK_ARG(A && B && C, "eth_gemm: null operand");
  ETH_CHECK_ARG(K % 8 == 0, "eth_gemm: K (%lld) must be a multiple of 8", (long long)K);
  ETH_CHECK_ARG(lda % 8 == 0 && ldb % 8 == 0, "eth_gemm: lda/ldb must be multiples of 8");
  ETH_CHECK_ARG(((uintptr_t)A & 15) == 0 && ((uintptr_t)B & 15) == 0, "eth_gemm: A/B must be 16-byte aligned");
  ETH_CHECK_ARG(a_kcontig ? lda >= K : (M % 8 == 0 && lda >= M), "eth_gemm: bad A layout");
  ETH_CHECK_ARG(b_kcontig ? ldb >= K : (N % 8 == 0 && ldb >= N), "eth_gemm: bad B layout");
  ETH_CHECK_ARG(ldc >= N, "eth_gemm: ldc < N");
  ETH_CHECK_ARG(!(flags & ETH_GEMM_ACCUMULATE) || c_dtype == ETH_F32, "eth_gemm: accumulate needs fp32 C");
  ETH_CHECK_ARG(!(flags & ETH_GEMM_BIAS) || bias, "eth_gemm: bias flag without bias");
  // extents: A spans M rows of lda (K-contiguous) or K rows of lda; same for B
  const int64_t a_elems = a_kcontig ? (M - 1) * lda + K : (K - 1) * lda + M;
  const int64_t b_elems = b_kcontig ? (N - 1) * ldb + K : (K - 1) * ldb + N;
  ETH_CHECK_ARG(a_elems * 2 < (1LL << 31) && b_elems * 2 < (1LL << 31),
                "eth_gemm: operands above 2 GiB are not supported");
  GemmArgs a;
  a.A = (const uint16_t*)A;
  a.B = (const uint16_t*)B;
  a.a_bytes = (uint32_t)(a_elems * 2);
  a.b_bytes = (uint32_t)(b_elems * 2);
  a.C = C;
  a.bias = (const uint16_t*)bias;
  a.M = (int)M;
  a.N = (int)N;
  a.K = (int)K;
  a.lda = lda;
  a.ldb = ldb;
  a.ldc = ldc;
  a.c_dtype = c_dtype;
  a.flags = flags;
  a.alpha = alpha;
  hipStream_t s = (hipStream_t)stream;
  const int esz = c_dtype == ETH_F32 ? 4 : 2;
  a.c_vec = ldc % 4 == 0 && N % 4 == 0 && ((uintptr_t)C % (4 * esz)) == 0;
  a.k_split = 0;
  a.c_split_stride = 0;
  const bool wide = wide_takes(M, N, ldc, esz, a.c_vec);
  a.c_bytes = wide ? (uint32_t)(((M - 1) * ldc + N) * esz) : 0;
  const bool fp16 = in_dtype == ETH_F16;
  const GemmForm form = gemm_form(M, N, K, a_kcontig, b_kcontig, c_dtype == ETH_F32);
  const GemmCut cut = plan_cut(M, N, K, wide, form);
  if (cut.m == M && cut.n == N) return launch_planned(a, a_kcontig, b_kcontig, fp16, wide, form, s);
  // the part of whole rounds, then the rest (rows or columns of C)
  const int64_t M2 = M - cut.m, N2 = N - cut.n;
  GemmArgs r = a;
  if (M2) {
    a.M = (int)cut.m;
    a.a_bytes = (uint32_t)((a_kcontig ? (cut.m - 1) * lda + K : (K - 1) * lda + cut.m) * 2);
    a.c_bytes = (uint32_t)(((cut.m - 1) * ldc + N) * esz);
    r.M = (int)M2;
    r.A += a_kcontig ? cut.m * lda : cut.m;
    r.a_bytes = (uint32_t)((a_kcontig ? (M2 - 1) * lda + K : (K - 1) * lda + M2) * 2);
    r.C = (char*)C + cut.m * ldc * esz;
    r.c_bytes = (uint32_t)(((M2 - 1) * ldc + N) * esz);
  } else {
    a.N = (int)cut.n;
    a.b_bytes = (uint32_t)((b_kcontig ? (cut.n - 1) * ldb + K : (K - 1) * ldb + cut.n) * 2);
    a.c_bytes = (uint32_t)(((M - 1) * ldc + cut.n) * esz);
    r.N = (int)N2;
    r.B += b_kcontig ? cut.n * ldb : cut.n;
    r.b_bytes = (uint32_t)((b_kcontig ? (N2 - 1) * ldb + K : (K - 1) * ldb + N2) * 2);
    r.C = (char*)C + cut.n * esz;
    if (r.bias) r.bias += cut.n;
    r.c_bytes = (uint32_t)(((M - 1) * ldc + N2) * esz);
  }
  const int rc = launch_planned(a, a_kcontig, b_kcontig, fp16, wide, form, s);
  return rc != ETH_OK ? rc : launch_planned(r, a_kcontig, b_kcontig, fp16, wide, form, s);
}

extern "C" int eth_gemm_plan(int64_t M, int64_t N, int64_t K, int a_kcontig, int b_kcontig, int64_t ldc, int c_dtype,
                             int64_t* plan) {
  ETH_CHECK_ARG(plan, "eth_gemm_plan: null pointer");
  ETH_CHECK_ARG(valid_dtype(c_dtype), "eth_gemm_plan: bad output dtype %d", c_dtype);
  ETH_CHECK_ARG(M > 0 && N > 0 && K > 0 && M < (1LL << 31) && N < (1LL << 31) && K < (1LL << 31) && ldc >= N,
                "eth_gemm_plan: bad shape %lld x %lld x %lld", (long long)M, (long long)N, (long long)K);
  const bool wide = wide_takes(M, N, ldc, c_dtype == ETH_F32 ? 4 : 2, ldc % 4 == 0 && N % 4 == 0);
  const GemmForm form = gemm_form(M, N, K, a_kcontig, b_kcontig, c_dtype == ETH_F32);
  const GemmCut cut = plan_cut(M, N, K, wide, form);
  plan[0] = plan_tile(cut.m, cut.n, K, wide, form);
  plan[1] = cut.m;
  plan[2] = cut.n;
  const int64_t m = cut.m < M ? M - cut.m : M, n = cut.n < N ? N - cut.n : N;
  plan[3] = cut.m == M && cut.n == N ? 0 : plan_tile(m, n, K, wide, form);
  return ETH_OK;
}

namespace eth {
struct SplitSum {
  const float* W;   // [splits][M][N] partial products
  int splits;
  int64_t stride;   // elements between splits
  void* C;
  int64_t ldc;
  const uint16_t* bias;
  int M, N;
  int c_dtype, flags;
  float alpha;
};
// C[m, n] (+)= alpha * sum_s W[s][m*N + n] (+ bias[n]), splits added in order
// (deterministic) and rounded once.  Four columns a thread; the splits' loads
// go out four at a time.
template <bool FP16>
__global__ void __launch_bounds__(256) splitk_sum_kernel(SplitSum g) {
  const int nq = g.N / 4;
  const int64_t total = (int64_t)g.M * nq;
  for (int64_t q = blockIdx.x * 256LL + threadIdx.x; q < total; q += gridDim.x * 256LL) {
    const int m = (int)(q / nq), n = (int)(q - (int64_t)m * nq) * 4;
    const float* w = g.W + (int64_t)m * g.N + n;
    f32x4_t v = *reinterpret_cast<const f32x4_t*>(w);
    int s = 1;
    for (; s + 3 < g.splits; s += 4) {
      f32x4_t u[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) u[e] = *reinterpret_cast<const f32x4_t*>(w + (s + e) * g.stride);
#pragma unroll
      for (int e = 0; e < 4; ++e) v += u[e];
    }
    for (; s < g.splits; ++s) v += *reinterpret_cast<const f32x4_t*>(w + s * g.stride);
    float bn[4] = {0.f, 0.f, 0.f, 0.f};
    if (g.bias) {
#pragma unroll
      for (int e = 0; e < 4; ++e) bn[e] = FP16 ? h2f_bits(g.bias[n + e]) : bf2f(g.bias[n + e]);
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = v[e] * g.alpha + bn[e];
    const int64_t o = (int64_t)m * g.ldc + n;
    if (g.c_dtype == ETH_F32) {
      f32x4_t* c = reinterpret_cast<f32x4_t*>(reinterpret_cast<float*>(g.C) + o);
      *c = (g.flags & ETH_GEMM_ACCUMULATE) ? *c + v : v;
    } else {
      u32x2_t r;
      if (g.c_dtype == ETH_BF16) {
        r.x = f2bf_pair(v[0], v[1]);
        r.y = f2bf_pair(v[2], v[3]);
      } else {
        r.x = f2h_bits(v[0]) | ((uint32_t)f2h_bits(v[1]) << 16);
        r.y = f2h_bits(v[2]) | ((uint32_t)f2h_bits(v[3]) << 16);
      }
      *reinterpret_cast<u32x2_t*>(reinterpret_cast<uint16_t*>(g.C) + o) = r;
    }
  }
}
}  // namespace eth

extern "C" int64_t eth_gemm_splitk_workspace(int64_t M, int64_t N, int splits) {
  return splits > 0 && M > 0 && N > 0 ? (int64_t)splits * M * N * 4 : 0;
}

extern "C" int64_t eth_gemm_splitk_pays(int64_t M, int64_t N, int64_t K, int splits, int a_kcontig, int b_kcontig,
                                        int c_dtype) {
  if (M <= 0 || N <= 0 || K <= 0 || splits < 2) return 0;
  // the second kernel: a launch, and the partials (and an fp32 C) at 4.3 TB/s
  const double sum = 4.5 + 4.0 * (double)M * (double)N * (splits + (c_dtype == ETH_F32 ? 1 : 0)) / 4.3e6;
  const GemmForm form = gemm_form(M, N, K, a_kcontig, b_kcontig, c_dtype == ETH_F32);
  const double one = tile_time(plan_tile(M, N, K, true, form), M, N, K, 1, form);
  return tile_time(256, M, N, K, splits, form) + sum < one;
}

extern "C" int eth_gemm_splitk_out(const void* A, int64_t lda, int a_kcontig, const void* B, int64_t ldb,
                                   int b_kcontig, void* C, int64_t ldc, int c_dtype, const void* bias, int64_t M,
                                   int64_t N, int64_t K, int in_dtype, int flags, float alpha, int splits,
                                   float* workspace, void* stream) {
  ETH_CHECK_ARG(in_dtype == ETH_BF16 || in_dtype == ETH_F16, "eth_gemm_splitk: inputs must be bf16 or fp16");
  ETH_CHECK_ARG(valid_dtype(c_dtype), "eth_gemm_splitk: bad output dtype %d", c_dtype);
  ETH_CHECK_ARG(A && B && C && workspace, "eth_gemm_splitk: null operand");
  ETH_CHECK_ARG(splits >= 1 && splits <= 16, "eth_gemm_splitk: splits must be in [1, 16] (got %d)", splits);
  ETH_CHECK_ARG(M > 0 && N > 0 && K > 0 && M < (1LL << 31) && N < (1LL << 31) && K < (1LL << 31),
                "eth_gemm_splitk: bad shape %lld x %lld x %lld", (long long)M, (long long)N, (long long)K);
  ETH_CHECK_ARG(K % 8 == 0, "eth_gemm_splitk: K (%lld) must be a multiple of 8", (long long)K);
  const int esz = c_dtype == ETH_F32 ? 4 : 2;
  ETH_CHECK_ARG(N % 4 == 0 && ldc % 4 == 0 && ldc >= N && ((uintptr_t)C % (4 * esz)) == 0 &&
                    ((uintptr_t)workspace & 15) == 0,
                "eth_gemm_splitk: C and the workspace need aligned rows of four columns (N %% 4 == 0)");
  ETH_CHECK_ARG(lda % 8 == 0 && ldb % 8 == 0, "eth_gemm_splitk: lda/ldb must be multiples of 8");
  ETH_CHECK_ARG(((uintptr_t)A & 15) == 0 && ((uintptr_t)B & 15) == 0, "eth_gemm_splitk: A/B must be 16-byte aligned");
  ETH_CHECK_ARG(a_kcontig ? lda >= K : (M % 8 == 0 && lda >= M), "eth_gemm_splitk: bad A layout");
  ETH_CHECK_ARG(b_kcontig ? ldb >= K : (N % 8 == 0 && ldb >= N), "eth_gemm_splitk: bad B layout");
  ETH_CHECK_ARG(!(flags & ETH_GEMM_ACCUMULATE) || c_dtype == ETH_F32, "eth_gemm_splitk: accumulate needs fp32 C");
  ETH_CHECK_ARG(!(flags & ETH_GEMM_BIAS) || bias, "eth_gemm_splitk: bias flag without bias");
  const int64_t a_elems = a_kcontig ? (M - 1) * lda + K : (K - 1) * lda + M;
  const int64_t b_elems = b_kcontig ? (N - 1) * ldb + K : (K - 1) * ldb + N;
  const int64_t slice = M * N;
  ETH_CHECK_ARG(a_elems * 2 < (1LL << 31) && b_elems * 2 < (1LL << 31) && (slice + 256 * N) * 4 < (1LL << 31),
                "eth_gemm_splitk: operands above 2 GiB are not supported");
  GemmArgs a{};
  a.A = (const uint16_t*)A;
  a.B = (const uint16_t*)B;
  a.a_bytes = (uint32_t)(a_elems * 2);
  a.b_bytes = (uint32_t)(b_elems * 2);
  a.C = workspace;
  a.bias = nullptr;
  a.M = (int)M;
  a.N = (int)N;
  a.K = (int)K;
  a.lda = lda;
  a.ldb = ldb;
  a.ldc = N;
  a.c_dtype = ETH_F32;
  a.flags = 0;
  a.alpha = 1.0f;
  a.c_bytes = (uint32_t)(slice * 4);
  // whole k-tiles per split, the last split shorter; few k-tiles may leave
  // fewer splits than asked for
  a.k_split = (int)(((K + splits - 1) / splits + 63) / 64 * 64);
  splits = (int)((K + a.k_split - 1) / a.k_split);
  a.c_split_stride = slice;
  hipStream_t s = (hipStream_t)stream;
  const bool fp16 = in_dtype == ETH_F16;
  const int rc = fp16 ? launch_256<true>(a, a_kcontig, b_kcontig, s, splits)
                      : launch_256<false>(a, a_kcontig, b_kcontig, s, splits);
  if (rc != ETH_OK) return rc;
  const SplitSum sum{workspace, splits, slice, C, ldc, (flags & ETH_GEMM_BIAS) ? (const uint16_t*)bias : nullptr,
                     (int)M, (int)N, c_dtype, flags, alpha};
  const int64_t quads = M * (N / 4);
  const int grid = (int)std::min<int64_t>((quads + 255) / 256, 2048);
  if (fp16)
    splitk_sum_kernel<true><<<grid, 256, 0, s>>>(sum);
  else
    splitk_sum_kernel<false><<<grid, 256, 0, s>>>(sum);
  ETH_CHECK_LAUNCH("eth_gemm_splitk");
  return ETH_OK;
}

extern "C" int eth_gemm_splitk(const void* A, int64_t lda, int a_kcontig, const void* B, int64_t ldb, int b_kcontig,
                               float* C, int64_t ldc, int64_t M, int64_t N, int64_t K, int in_dtype, int splits,
                               int accumulate, float* workspace, void* stream) {
  ETH_CHECK_ARG(splits >= 1 && splits <= 16, "eth_gemm_splitk: splits must be in [1, 16] (got %d)", splits);
  ETH_CHECK_ARG(K % (128LL * splits) == 0, "eth_gemm_splitk: K (%lld) must be a multiple of 128 * splits",
                (long long)K);
  return eth_gemm_splitk_out(A, lda, a_kcontig, B, ldb, b_kcontig, C, ldc, ETH_F32, nullptr, M, N, K, in_dtype,
                             accumulate ? ETH_GEMM_ACCUMULATE : 0, 1.0f, splits, workspace, stream);
}
