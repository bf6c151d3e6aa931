// prefill.hip -- batched prefill for gfx950: the MFMA Q4_0 / Q8_0 dequant GEMM
// and the row-wise norm that feeds it.
//
// The reference has no batched prefill: it runs prompt tokens one at a time
// through its decode graph without logits (src/interactive.zig:33-37,
// src/gpu/model_dispatch.zig:144).  Here the T prompt tokens of a layer go
// through each projection as one dense contraction
//     C[T][N] = A[T][K] . deq(W)[N][K]^T
// on the matrix cores, keeping the decode path's accuracy:
//  * weights enter exactly: the MFMA B operand is the integer n - 8 (Q4) or
//    q (Q8), exact in fp16, and each 32-block's f32 scale d is applied to the
//    block's fp32 partial sum (acc += d * block_sum), as the GEMV does;
//  * activations are split a = s (hi + lo) with hi = fp16(a / s),
//    lo = fp16(a / s - hi) and s a power of two per row that puts the row's
//    largest |a| / s in [2^13, 2^14) (no fp16 overflow for any row), and both
//    halves go through the MFMA (22+ significant bits of a).  The split is
//    made once per row (gh_pf_halves_k, or gh_pf_norm_k for normed rows),
//    not in every tile that reads the row, and s is applied in the epilogue
//    (exact: a power of two);
//  * accumulation is fp32.
//
// Three forms, chosen by the host: the weight-streaming GEMM for short batches,
// the wide tile for longer ones (both described at their kernels below), and
// the tiles that follow for what those do not take: K that is no multiple of
// 128, or weights that are not 16-byte aligned.
//
// Tiling (v_mfma_f32_32x32x16_f16): a workgroup of 256 threads (2 x 2
// wavefronts) owns a BM x BN tile
// of C; each wavefront a (BM/2) x (BN/2) sub-tile of 32 x 32 MFMA blocks (the
// _w8 forms of the 128-row tiles: 512 threads, 4 x 2 wavefronts of
// (BM/4) x (BN/2), so a CU's two tiles run four waves per SIMD).  K
// advances one quant block (32) per step: the A slice (as hi and lo) and the
// integer W slice with its scales go to LDS in unpadded, XOR-swizzled rows
// (bank-conflict-free operand reads and stage writes).  Two LDS stages:
// while the MFMAs of step s read one, step s+1's global loads are in flight
// and then stored into the other, one barrier per step.  Workgroups take
// their tiles in an XCD-aware order (the tiles of one XCD share A rows).
//
// MFMA 32x32x16 f16 operand layout (checked on the device): lane l holds
// A[l % 32][8 (l / 32) + e] and B[8 (l / 32) + e][l % 32], e = 0..7; result
// register r of lane l is C[8 (r / 4) + 4 (l / 32) + r % 4][l % 32].
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "../common/load_lds.h"
#include "../common/wide_lds.h"

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

#define PF_NT 256

// Weight words through an explicit global-address-space pointer: the matrix
// is picked at run time (gate or up), which would otherwise degrade to FLAT.
typedef const uint32_t __attribute__((address_space(1)))* gword_ptr;

struct Q4W {  // src/quant.zig:55-90: {f32 d, 4 words of nibbles}
  static constexpr uint32_t kBlockBytes = 20;
  static constexpr int kWords = 3;
  static constexpr bool kBf16 = false;
  // half h (elements 16h .. 16h+15) of a block: scale and its 16 values
  __device__ static void load(const uint8_t* blk, uint32_t h, uint32_t* w) {
    gword_ptr p = (gword_ptr)(blk);
    w[0] = p[0];
    w[1] = p[1 + 2 * h];
    w[2] = p[2 + 2 * h];
  }
  // n - 8 as fp16 pairs, exactly: (w >> 4j) & 0x000F000F | 0x64006400 read as
  // two halves is (1024 + n_j, 1024 + n_{j+4}), and one packed subtract of
  // 1032 leaves (n_j - 8, n_{j+4} - 8).  So the 8 elements of a word come out
  // in the K order (0,4,1,5,2,6,3,7); the A operand is stored in the same
  // order (pf_ax_pos with perm).  out: 8 words = the half-block's 16 halves.
  __device__ static void ints(const uint32_t* w, uint32_t* out) {
    typedef _Float16 h2 __attribute__((ext_vector_type(2)));
    const h2 bias = {(_Float16)-1032.0f, (_Float16)-1032.0f};
#pragma unroll
    for (int k = 0; k < 2; k++)
#pragma unroll
      for (int j = 0; j < 4; j++) {
        const uint32_t pr = ((w[1 + k] >> (4 * j)) & 0x000F000Fu) | 0x64006400u;
        out[4 * k + j] = __builtin_bit_cast(uint32_t, __builtin_bit_cast(h2, pr) + bias);
      }
  }
};

struct Q8W {  // src/quant.zig:20-51: {f32 d, 8 words of int8}
  static constexpr uint32_t kBlockBytes = 36;
  static constexpr int kWords = 5;
  static constexpr bool kBf16 = false;
  __device__ static void load(const uint8_t* blk, uint32_t h, uint32_t* w) {
    gword_ptr p = (gword_ptr)(blk);
    w[0] = p[0];
#pragma unroll
    for (int k = 0; k < 4; k++) w[1 + k] = p[1 + 4 * h + k];
  }
  __device__ static void ints(const uint32_t* w, uint32_t* out) {  // q as fp16, in K order
    typedef _Float16 h2 __attribute__((ext_vector_type(2)));
#pragma unroll
    for (int k = 0; k < 4; k++)
#pragma unroll
      for (int n = 0; n < 4; n += 2) {
        const h2 v = {(_Float16)(int)(int8_t)((w[1 + k] >> (8 * n)) & 0xFFu),
                      (_Float16)(int)(int8_t)((w[1 + k] >> (8 * n + 8)) & 0xFFu)};
        out[2 * k + n / 2] = __builtin_bit_cast(uint32_t, v);
      }
  }
};

typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));
typedef const u32x4_t __attribute__((address_space(1)))* gvec_ptr;

// bf16 rows as stored (mode none, the reference's --gpu weights): 32 bf16 of
// a row per K step go to the stage as they are and feed the bf16 MFMA
// directly; there is no unpacking and no block scale (kBf16).
struct Bf16W {
  static constexpr uint32_t kBlockBytes = 64;
  static constexpr int kWords = 8;
  static constexpr bool kBf16 = true;
  // half h (elements 16h .. 16h+15) of a 32-element segment: 8 words
  __device__ static void load(const uint8_t* blk, uint32_t h, uint32_t* w) {
    gvec_ptr p = (gvec_ptr)(blk + 32 * h);
    const u32x4_t a = p[0], b = p[1];
    w[0] = a.x; w[1] = a.y; w[2] = a.z; w[3] = a.w;
    w[4] = b.x; w[5] = b.y; w[6] = b.z; w[7] = b.w;
  }
  __device__ static void ints(const uint32_t* w, uint32_t* out) {
#pragma unroll
    for (int k = 0; k < 8; k++) out[k] = w[k];
  }
};

__device__ __forceinline__ float gelu_tanh(float x) {
  // kernels.zig:94-97 / fused_mlp_q4.wgsl:15-18
  const float inner = 0.7978845608f * (x + 0.044715f * x * x * x);
  return 0.5f * x * (1.0f + tanhf(inner));
}

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

// The GEMM's A operand layout ("ax"): row t of K elements is 2K halves, the
// hi halves of block b (elements 32b .. 32b+31) at 64b, their lo halves at
// 64b + 32.  With perm (Q4_0 weights) the 8 elements of each group sit in the
// order Q4W::ints unpacks a word: position 2m holds element m, 2m + 1 element
// m + 4.  Offset of element e's hi half within its row:
__device__ __forceinline__ uint32_t pf_ax_pos(uint32_t e, bool perm) {
  const uint32_t j = e & 7;
  return (e >> 5) * 64 + (e & 24) + (perm ? ((j & 3) << 1) | (j >> 2) : j);
}

// NMAT = 1: C = A W^T.  NMAT = 2: C = gelu_tanh(A Wg^T) * (A Wu^T).  A as its
// fp16 hi/lo halves interleaved per 32-element block (pf_ax: a row's K step
// is one contiguous 128-byte segment) and row scales rs; C f32.
// Each step covers KB quant blocks (32 KB elements of K).
// SPLIT (split-K, for few tiles): workgroup z of gridDim.z runs K steps
// [z S / Z, (z + 1) S / Z) and writes its raw sums to C as partial plane
// (z, matrix) of [Z][NMAT][T][N]; gh_pf_splitk_k adds the planes in z order
// and applies the epilogue.
// NW: waves per workgroup, 4 (2 x 2, each (BM/2) x (BN/2)) or 8 (4 x 2, each
// (BM/4) x (BN/2)).
template <class F, int BM, int BN, int NMAT, int KB, bool SPLIT, int NW = 4>
__device__ __forceinline__ void gemm_tile(const _Float16* __restrict__ Ax,
                                          const float* __restrict__ rs,
                                          const uint8_t* __restrict__ W0,
                                          const uint8_t* __restrict__ W1, float* __restrict__ C,
                                          uint32_t T, uint32_t N, uint32_t K) {
  static_assert(KB == 1, "one quant block per K step (the LDS swizzle assumes it)");
  static_assert(NW == 4 || NW == 8, "2 x 2 or 4 x 2 waves");
  constexpr int NT = 64 * NW;
  constexpr int TM = BM / (16 * NW), TN = BN / 64;  // 32x32 blocks per wave in M and N
  static_assert(TM >= 1, "a wave holds at least one 32-row block");
  constexpr int A_CH = 8 * KB;                               // 16-B chunks per row and step
  constexpr int A_PER = BM * A_CH / NT;                      // 16-B chunks per thread
  constexpr int B_ROWS = NMAT * BN;                          // weight rows per step
  constexpr int B_HALVES = 2 * KB * B_ROWS;                  // 16-element half-blocks
  constexpr int B_PER = (B_HALVES + NT - 1) / NT;
  static_assert(A_PER >= 1 && (BM * A_CH) % NT == 0, "A chunks divide the workgroup");
  // Two LDS stages: the MFMAs of step s read one while step s+1 is stored
  // into the other, so a K step needs one barrier.  A row of a stage is 128 B
  // (8 chunks of 8 halves: hi 0-3, lo 4-7), a weight row 64 B (4 chunks), with
  // no padding; chunk k of row r sits at k ^ sa(r) (A) or k ^ sb(r) (weights).
  // The swizzles keep every ds_read_b128 of the MFMA operands (16 rows at one
  // chunk) and every ds_write_b128 of a stage (2 A rows, or 8 weight rows at
  // two chunks) on distinct banks, for 8-lane phases over 32 banks as well as
  // 16-lane phases over 64.  (An 80-byte padded row was conflict-free to read
  // but not to write: write conflicts cost as many LDS cycles as the reads.)
  __shared__ _Float16 SA[2][BM * 64];
  __shared__ _Float16 Bs[2][B_ROWS * 32];
  __shared__ float Ds[2][B_ROWS * KB];
  auto a_at = [](uint32_t r, uint32_t k) { return r * 64 + 8 * (k ^ ((r & 7) ^ ((r >> 3) & 1))); };
  auto b_at = [](uint32_t r, uint32_t k) { return r * 32 + 8 * (k ^ (((r >> 1) ^ (r >> 2)) & 3)); };

  const uint32_t tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  // XCD-aware tile order: workgroups go to the 8 XCDs round-robin (w % 8), so
  // XCD c takes the c-th contiguous eighth of the tiles in (split, m, n)
  // order, n fastest.  The tiles of one XCD then share their A rows (one
  // 128-row block of a 512-token prompt is 2 MB: it stays in the XCD's L2)
  // instead of every XCD cycling through all of A.
  const uint32_t gx = gridDim.x, gy = gridDim.y, gz = SPLIT ? gridDim.z : 1u;
  const uint32_t G = gx * gy * gz;
  uint32_t w = blockIdx.x + gx * (blockIdx.y + gy * (SPLIT ? blockIdx.z : 0u));
  if (G % 8 == 0) w = (w % 8) * (G / 8) + w / 8;
  const uint32_t tn = w % gx, tm = (w / gx) % gy;
  const uint32_t m0 = tm * BM, n0 = tn * BN;
  const uint32_t wm = (wave >> 1) * (BM / (NW / 2)), wn = (wave & 1) * (BN / 2);
  const uint32_t nb = K / 32, nsteps = (nb + KB - 1) / KB;
  const size_t row_bytes = (size_t)nb * F::kBlockBytes;

  // global -> register staging of one K step (blocks past K load block nb - 1
  // and are multiplied by a zero scale)
  u32x4 ra[A_PER];  // a native vector: plain loads and stores, kept in registers
  uint32_t rb[B_PER][F::kWords];
  auto load_step = [&](uint32_t step) {
#pragma unroll
    for (int i = 0; i < A_PER; i++) {
      // chunk c: row c / A_CH; q = c % A_CH -> block q / 8 of the step, plane
      // (q / 4) % 2, 8 halves at (q % 4) * 8
      const uint32_t c = tid + i * NT, q = c % A_CH;
      uint32_t r = m0 + c / A_CH;
      r = r < T ? r : T - 1;
      uint32_t blk = step * KB + q / 8;
      blk = blk < nb ? blk : nb - 1;
      ra[i] = *reinterpret_cast<const u32x4*>(Ax + (size_t)r * 2 * K + (size_t)blk * 64 + 8 * (q % 8));
    }
#pragma unroll
    for (int i = 0; i < B_PER; i++) {
      const uint32_t hb = tid + i * NT;  // ((row * KB) + block) * 2 + half
      if (hb < (uint32_t)B_HALVES) {
        const uint32_t lr = hb / (2 * KB), kq = (hb / 2) % KB, mat = lr / BN;
        uint32_t r = n0 + lr % BN;
        r = r < N ? r : N - 1;
        uint32_t blk = step * KB + kq;
        blk = blk < nb ? blk : nb - 1;
        const uint8_t* W = mat ? W1 : W0;
        F::load(W + (size_t)r * row_bytes + (size_t)blk * F::kBlockBytes, hb % 2, rb[i]);
      }
    }
  };
  auto store_step = [&](int sb, uint32_t step) {
#pragma unroll
    for (int i = 0; i < A_PER; i++) {
      const uint32_t c = tid + i * NT;
      *reinterpret_cast<u32x4*>(&SA[sb][a_at(c / A_CH, c % A_CH)]) = ra[i];
    }
#pragma unroll
    for (int i = 0; i < B_PER; i++) {
      const uint32_t hb = tid + i * NT;
      if (hb < (uint32_t)B_HALVES) {
        const uint32_t lr = hb / (2 * KB), kq = (hb / 2) % KB;
        uint32_t v[8];
        F::ints(rb[i], v);
        *reinterpret_cast<u32x4*>(&Bs[sb][b_at(lr, 2 * (hb % 2))]) = u32x4{v[0], v[1], v[2], v[3]};
        *reinterpret_cast<u32x4*>(&Bs[sb][b_at(lr, 2 * (hb % 2) + 1)]) = u32x4{v[4], v[5], v[6], v[7]};
        if constexpr (!F::kBf16)
          if (hb % 2 == 0) Ds[sb][lr * KB + kq] = step * KB + kq < nb ? __uint_as_float(rb[i][0]) : 0.f;
      }
    }
  };

  f32x16 acc[NMAT][TM][TN];
#pragma unroll
  for (int q = 0; q < NMAT; q++)
#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
      for (int j = 0; j < TN; j++)
#pragma unroll
        for (int r = 0; r < 16; r++) acc[q][i][j][r] = 0.f;

  const uint32_t nz = gz, z = w / (gx * gy);
  const uint32_t s_begin = (uint32_t)((uint64_t)nsteps * z / nz);
  const uint32_t s_end = (uint32_t)((uint64_t)nsteps * (z + 1) / nz);
  if (s_begin < s_end) {
    load_step(s_begin);
    store_step(0, s_begin);
  }
  __syncthreads();
  for (uint32_t step = s_begin; step < s_end; step++) {
    const int cb = (step - s_begin) & 1;
    if (step + 1 < s_end) load_step(step + 1);  // in flight through this step's MFMAs
#pragma unroll
    for (int kq = 0; kq < KB; kq++) {
      half8 ah[2][TM], al[2][TM];
#pragma unroll
      for (int h = 0; h < 2; h++)
#pragma unroll
        for (int i = 0; i < TM; i++) {
          const uint32_t r = wm + 32 * i + lane % 32, k = 2 * h + lane / 32;
          ah[h][i] = *reinterpret_cast<const half8*>(&SA[cb][a_at(r, k)]);
          al[h][i] = *reinterpret_cast<const half8*>(&SA[cb][a_at(r, 4 + k)]);
        }
#pragma unroll
      for (int q = 0; q < NMAT; q++)
#pragma unroll
        for (int j = 0; j < TN; j++) {
          const uint32_t brow = q * BN + wn + 32 * j + lane % 32;
          const half8 b0 = *reinterpret_cast<const half8*>(&Bs[cb][b_at(brow, lane / 32)]);
          const half8 b1 = *reinterpret_cast<const half8*>(&Bs[cb][b_at(brow, 2 + lane / 32)]);
          if constexpr (F::kBf16) {
            // exact bf16 weights and bf16 activation halves: every product
            // accumulates straight into the tile (one block per step, so no
            // step lies past K)
            const bf16x8 c0 = __builtin_bit_cast(bf16x8, b0), c1 = __builtin_bit_cast(bf16x8, b1);
#pragma unroll
            for (int i = 0; i < TM; i++) {
              f32x16 t = acc[q][i][j];
              t = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, ah[0][i]), c0, t, 0, 0, 0);
              t = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, al[0][i]), c0, t, 0, 0, 0);
              t = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, ah[1][i]), c1, t, 0, 0, 0);
              t = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, al[1][i]), c1, t, 0, 0, 0);
              acc[q][i][j] = t;
            }
            continue;
          }
          const float d = Ds[cb][brow * KB + kq];
#pragma unroll
          for (int i = 0; i < TM; i++) {
            f32x16 blk = {};
            blk = __builtin_amdgcn_mfma_f32_32x32x16_f16(ah[0][i], b0, blk, 0, 0, 0);
            blk = __builtin_amdgcn_mfma_f32_32x32x16_f16(al[0][i], b0, blk, 0, 0, 0);
            blk = __builtin_amdgcn_mfma_f32_32x32x16_f16(ah[1][i], b1, blk, 0, 0, 0);
            blk = __builtin_amdgcn_mfma_f32_32x32x16_f16(al[1][i], b1, blk, 0, 0, 0);
#pragma unroll
            for (int r = 0; r < 16; r++) acc[q][i][j][r] += d * blk[r];
          }
        }
    }
    if (step + 1 < s_end) store_step(cb ^ 1, step + 1);
    // the next step reads the stage just stored, and then stores into the
    // stage read here
    __syncthreads();
  }

  // epilogue: result register r of lane l -> row 8 (r/4) + 4 (l/32) + r%4, col l % 32
#pragma unroll
  for (int i = 0; i < TM; i++)
#pragma unroll
    for (int j = 0; j < TN; j++) {
      const uint32_t col = n0 + wn + 32 * j + lane % 32;
#pragma unroll
      for (int r = 0; r < 16; r++) {
        const uint32_t row = m0 + wm + 32 * i + 8 * (r / 4) + 4 * (lane / 32) + r % 4;
        if (row < T && col < N) {
          const float sr = rs[row];
          if constexpr (SPLIT) {
#pragma unroll
            for (int q = 0; q < NMAT; q++)
              C[((size_t)(z * NMAT + q) * T + row) * N + col] = acc[q][i][j][r] * sr;
          } else if constexpr (NMAT == 1) {
            C[(size_t)row * N + col] = acc[0][i][j][r] * sr;
          } else {
            C[(size_t)row * N + col] = gelu_tanh(acc[0][i][j][r] * sr) * (acc[1][i][j][r] * sr);
          }
        }
      }
    }
}

#define GH_GEMM(NAME, F, BM, BN, KB, SPLIT, SUFFIX)                                       \
  extern "C" __global__ __launch_bounds__(PF_NT) GH_PF_OCC_##BM void NAME##_k##KB##SUFFIX( \
      const _Float16* Ax, const float* rs, const uint8_t* W, float* C, uint32_t T,         \
      uint32_t N, uint32_t K) {                                                            \
    gemm_tile<F, BM, BN, 1, KB, SPLIT>(Ax, rs, W, W, C, T, N, K);                          \
  }
#define GH_GEMM_W8(NAME, F, BM, BN, KB, SPLIT, SUFFIX)                                    \
  extern "C" __global__ __launch_bounds__(512) GH_PF_OCC_W8 void NAME##_k##KB##SUFFIX(     \
      const _Float16* Ax, const float* rs, const uint8_t* W, float* C, uint32_t T,         \
      uint32_t N, uint32_t K) {                                                            \
    gemm_tile<F, BM, BN, 1, KB, SPLIT, 8>(Ax, rs, W, W, C, T, N, K);                       \
  }
#define GH_GEMM_PAIR_W8(NAME, F, BM, BN, KB, SPLIT, SUFFIX)                               \
  extern "C" __global__ __launch_bounds__(512) GH_PF_OCC_W8 void NAME##_k##KB##SUFFIX(     \
      const _Float16* Ax, const float* rs, const uint8_t* Wg, const uint8_t* Wu,           \
      float* Act, uint32_t T, uint32_t N, uint32_t K) {                                    \
    gemm_tile<F, BM, BN, 2, KB, SPLIT, 8>(Ax, rs, Wg, Wu, Act, T, N, K);                   \
  }
#define GH_PF_OCC_W8 __attribute__((amdgpu_waves_per_eu(4, 4)))
#define GH_GEMM_PAIR(NAME, F, BM, BN, KB, SPLIT, SUFFIX)                                  \
  extern "C" __global__ __launch_bounds__(PF_NT) GH_PF_OCC_##BM void NAME##_k##KB##SUFFIX( \
      const _Float16* Ax, const float* rs, const uint8_t* Wg, const uint8_t* Wu,           \
      float* Act, uint32_t T, uint32_t N, uint32_t K) {                                    \
    gemm_tile<F, BM, BN, 2, KB, SPLIT>(Ax, rs, Wg, Wu, Act, T, N, K);                      \
  }
// The 128-row tiles are held to 2 waves per SIMD: at 3 (the register count
// allows it) they measured ~2x slower, the third workgroup's tiles evicting
// the first two's operands.
#define GH_PF_OCC_128 __attribute__((amdgpu_waves_per_eu(1, 2)))
#define GH_PF_OCC_64
#define GH_GEMM_ALL                                                       \
  GH_GEMM(gh_pf_gemm_q4_m128_n128, Q4W, 128, 128, 1, false, )             \
  GH_GEMM(gh_pf_gemm_q4_m128_n64, Q4W, 128, 64, 1, false, )               \
  GH_GEMM(gh_pf_gemm_q4_m64_n64, Q4W, 64, 64, 1, false, )                 \
  GH_GEMM(gh_pf_gemm_q8_m128_n128, Q8W, 128, 128, 1, false, )             \
  GH_GEMM(gh_pf_gemm_q8_m128_n64, Q8W, 128, 64, 1, false, )               \
  GH_GEMM(gh_pf_gemm_q8_m64_n64, Q8W, 64, 64, 1, false, )                 \
  GH_GEMM_PAIR(gh_pf_gateup_q4_m128_n64, Q4W, 128, 64, 1, false, )        \
  GH_GEMM_PAIR(gh_pf_gateup_q4_m64_n64, Q4W, 64, 64, 1, false, )          \
  GH_GEMM_PAIR(gh_pf_gateup_q8_m128_n64, Q8W, 128, 64, 1, false, )        \
  GH_GEMM_PAIR(gh_pf_gateup_q8_m64_n64, Q8W, 64, 64, 1, false, )

// One quant block per K step measured fastest (12B prefill 62.7 ms vs 65.9
// and 68.4 ms at 2 and 4 blocks), and loading 2 or 3 steps ahead in a
// register ring slower (72-77 ms vs 64): the step is bound by its barriers
// and MFMA dependency chains, not by load latency.
GH_GEMM_ALL

// Split-K forms, for products whose tiles alone cannot fill the CUs: the
// small tile for a few prompt tokens (without the split each workgroup walks
// all of K one block per step, and that serial chain, not bandwidth, sets the
// time), and the large plain tile for the narrow products of a long prompt
// (o and down, N = 3840), which otherwise fall back to the small tile.
GH_GEMM(gh_pf_gemm_bf16_m128_n128, Bf16W, 128, 128, 1, false, )
GH_GEMM(gh_pf_gemm_bf16_m128_n64, Bf16W, 128, 64, 1, false, )
GH_GEMM(gh_pf_gemm_bf16_m64_n64, Bf16W, 64, 64, 1, false, )
GH_GEMM_PAIR(gh_pf_gateup_bf16_m128_n64, Bf16W, 128, 64, 1, false, )
GH_GEMM_PAIR(gh_pf_gateup_bf16_m64_n64, Bf16W, 64, 64, 1, false, )
GH_GEMM(gh_pf_gemm_bf16_m64_n64, Bf16W, 64, 64, 1, true, _s)
GH_GEMM(gh_pf_gemm_bf16_m128_n128, Bf16W, 128, 128, 1, true, _s)
GH_GEMM_PAIR(gh_pf_gateup_bf16_m64_n64, Bf16W, 64, 64, 1, true, _s)
GH_GEMM(gh_pf_gemm_q4_m64_n64, Q4W, 64, 64, 1, true, _s)
GH_GEMM(gh_pf_gemm_q8_m64_n64, Q8W, 64, 64, 1, true, _s)
GH_GEMM(gh_pf_gemm_q4_m128_n128, Q4W, 128, 128, 1, true, _s)
GH_GEMM(gh_pf_gemm_q8_m128_n128, Q8W, 128, 128, 1, true, _s)
GH_GEMM_PAIR(gh_pf_gateup_q4_m64_n64, Q4W, 64, 64, 1, true, _s)
GH_GEMM_PAIR(gh_pf_gateup_q4_m128_n64, Q4W, 128, 64, 1, true, _s)  // 65-128 tokens
GH_GEMM_PAIR(gh_pf_gateup_q8_m64_n64, Q8W, 64, 64, 1, true, _s)

// 8-wave forms of the 128-row tiles (names end in _w8)
#define GH_GEMM_W8_FMT(FMT, F)                                                  \
  GH_GEMM_W8(gh_pf_gemm_##FMT##_m128_n128, F, 128, 128, 1, false, _w8)          \
  GH_GEMM_W8(gh_pf_gemm_##FMT##_m128_n64, F, 128, 64, 1, false, _w8)            \
  GH_GEMM_W8(gh_pf_gemm_##FMT##_m128_n128, F, 128, 128, 1, true, _s_w8)         \
  GH_GEMM_PAIR_W8(gh_pf_gateup_##FMT##_m128_n64, F, 128, 64, 1, false, _w8)
GH_GEMM_W8_FMT(q4, Q4W)
GH_GEMM_W8_FMT(q8, Q8W)
GH_GEMM_W8_FMT(bf16, Bf16W)
GH_GEMM_PAIR_W8(gh_pf_gateup_q4_m128_n64, Q4W, 128, 64, 1, true, _s_w8)

// ---------------------------------------------------------------------------
// The wide tile GEMM: one 512-thread workgroup per CU owns 64 TM tokens by BR
// (256 or 128) weight rows (for a gate/up pair half of them of each matrix),
// 2 x 4 wavefronts of (32 TM) x (BR / 4) on v_mfma_f32_16x16x32_f16 (or
// _bf16).  Operands as the tile GEMM's above; a block's sum is its hi
// products, then its lo products (the streamed GEMM's order below).
//
// What bounds it: matrix and vector instructions, which overlap only in part, and
// the power they draw.  A step of one block of K is 2048 matrix cycles of a CU at
// TM = 4, BR = 256, and about 1570 vector cycles (a scale FMA per result, the
// weights' unpacking).  Counters of the gate/up of 512 tokens: matrix pipes busy
// 50% of the cycles, vector instructions beside them in 38% of those, waves
// waiting 30%.  Under random data the chip runs these at 1.4-1.8 GHz (a
// register-only loop of the same MFMA: 1.9-2.0 PFLOP/s, 1.65-1.85 for the 32x32x16
// form, which is why this one uses 16x16x32), so whatever else a step does costs
// time as power even where it overlaps:
//  * operands go from memory to LDS directly (16 bytes per lane, no registers
//    and no LDS store instructions).  The A rows are swizzled on the way, by
//    permuting the lanes' source addresses within a row's 128 bytes, so that
//    the operand reads of 16 lanes (one g) meet no bank twice.  The counters
//    still show 4 conflict cycles per LDS instruction, not taken apart yet;
//  * quantized weights stay packed in LDS, four blocks of K (80 or 144 bytes
//    of a row) at a time, and each wavefront unpacks the words of its rows as
//    it reads them: a quarter (Q4) of the LDS bytes of fp16 weights;
//  * one barrier per step, ahead of the last 16 rows, whose MFMAs then cover
//    the next step's first LDS reads; two to four steps of A in flight (one for
//    the largest Q8 tile, whose weights leave LDS for two stages).
// The waits are written out (vmcnt counts the loads issued since), because the
// compiler would wait for every load to LDS before any LDS read.
//
// Sums: an fp32 chain over all of an unsplit K is off by more than the split
// tiles' shorter ones, so runs of blocks (16 for long K) are chains of their own
// whose sums are added up in second registers.  The tiles of 192 and 256 tokens
// by 256 rows have registers for only 3 of 6 and 1 of 8 of their 16-row blocks
// (bf16: for none, but its 16-bit activations are 10 times further off); they
// take the products that were unsplit before.  Against 64 bits, tile GEMM / one
// chain / runs, Q4: gate/up 2 x 15360 x 3840 of 64, 128 and 333 tokens 2.05 / 3.09
// / 1.74e-7, 2.35 / 3.10 / 1.73e-7 and 2.95 / 3.11 / 2.42e-7, down 3840 x 15360 of
// 128 tokens 1.43 / 1.65 / 1.18e-7.  It takes 1.1% in the mean of 165 products: a
// run is a loop of its own, as a branch or selects in one loop over K cost the
// larger tiles registers or 5%.
//
// Measured, 12B gate/up of 512 tokens, tile GEMM -> this (the whole call, its
// activation split included): Q4 281 -> 209 us (1160 TFLOP/s executed), Q8 297 ->
// 219, bf16 269 -> 189.  Within a whole prompt's trace the Q4 kernel alone
// takes 212-221 us, at a lower clock.  Timing-only copies took 11% less without the loads, 22%
// without the LDS reads of A as well.  The gate/up of 128 tokens (TM 2, BR 128,
// which keeps K unsplit) 89 -> 73 us, of 64 tokens 61 -> 52 us.
// ---------------------------------------------------------------------------
#define PF_WIDE_NT 512

template <int N>
__device__ __forceinline__ void wait_loads_barrier() {
  asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(N) : "memory");
}

// The unpacking's constants, held in registers (an instruction takes one
// literal at most).
struct Unpack {
  uint32_t lo = 0x000F000Fu, hi = 0x00F000F0u, magic, sixteenth = 0x2C002C00u, bias = 0xD480D480u;
  __device__ explicit Unpack(bool q8) : magic(q8 ? 0x64646464u : 0x64006400u) {
    asm("" : "+v"(lo), "+v"(hi), "+s"(magic), "+v"(sixteenth), "+s"(bias));
  }
};

// A weight format of the wide tile.  Quantized: kChunks 16-byte pieces of a
// row hold four blocks, and per(rows, j) pieces per thread of a group of four
// blocks are loaded in step j of the four.  bf16: a step's 64 bytes of a row (4 pieces, swizzled), two per thread.
// raw: one block of one row as a lane's operand needs it (elements 8 g ..
// 8 g + 7, g = lane / 16); pair: two of the operand's eight halves.
struct WQ4 {
  static constexpr bool kBf16 = false;
  static constexpr int kChunks = WIDE_CHUNKS_Q4, kRaw = 1;
  static constexpr int per(int rows, int j) { return j == 0 ? rows / 128 : j == 1; }
  __device__ static void raw(const uint8_t* row, uint32_t g, uint32_t* w, float* d) {
    const uint32_t* p = reinterpret_cast<const uint32_t*>(row);
    *d = __uint_as_float(p[0]);
    w[0] = p[1 + g];
  }
  // The operand's pair p, elements p and p + 4 of the word, as n - 8 exactly:
  // nibbles under the exponent of 1024 are 1024 + n in the low position and
  // 1024 + 16 n in the next, and one packed add of -1032, or a multiply-add by
  // 1/16 and -72, leaves n - 8.  So only the upper half of the word is shifted.
  __device__ static uint32_t pair(const uint32_t* w, int p, const Unpack& c) {
    typedef _Float16 h2 __attribute__((ext_vector_type(2)));
    uint32_t pr;
    asm("v_and_or_b32 %0, %1, %2, %3" : "=v"(pr) : "v"(p < 2 ? w[0] : w[0] >> 8), "v"(p % 2 ? c.hi : c.lo), "s"(c.magic));
    const h2 v = __builtin_bit_cast(h2, pr);
    h2 o;
    if (p % 2 == 0)
      o = v + h2{(_Float16)-1032.0f, (_Float16)-1032.0f};
    else
      asm("v_pk_fma_f16 %0, %1, %2, %3" : "=v"(o) : "v"(v), "v"(c.sixteenth), "s"(c.bias));
    return __builtin_bit_cast(uint32_t, o);
  }
};
struct WQ8 {
  static constexpr bool kBf16 = false;
  static constexpr int kChunks = WIDE_CHUNKS_Q8, kRaw = 2;
  static constexpr int per(int rows, int j) { return j < 2 ? (rows == 256 ? 3 : 2) - j : 0; }
  __device__ static void raw(const uint8_t* row, uint32_t g, uint32_t* w, float* d) {
    const uint32_t* p = reinterpret_cast<const uint32_t*>(row);
    *d = __uint_as_float(p[0]);
    w[0] = p[1 + 2 * g];
    w[1] = p[2 + 2 * g];
  }
  // byte q + 128 under the exponent of 1024 is 1024 + (q + 128), exactly; the
  // packed add of -1152 leaves q
  __device__ static uint32_t pair(const uint32_t* w, int p, const Unpack& c) {
    typedef _Float16 h2 __attribute__((ext_vector_type(2)));
    const uint32_t u = __builtin_amdgcn_perm(c.magic, w[p / 2] ^ 0x80808080u, p % 2 ? 0x07030702u : 0x07010700u);
    return __builtin_bit_cast(uint32_t, __builtin_bit_cast(h2, u) + h2{(_Float16)-1152.0f, (_Float16)-1152.0f});
  }
};
struct WBf16 {
  static constexpr bool kBf16 = true;
  static constexpr int kChunks = WIDE_CHUNKS_BF16, kRaw = 4;
  static constexpr int per(int rows, int) { return rows / 128; }
  __device__ static void raw(const uint8_t* chunk, uint32_t, uint32_t* w, float*) {
    const u32x4 v = *reinterpret_cast<const u32x4*>(chunk);
#pragma unroll
    for (int k = 0; k < 4; k++) w[k] = v[k];
  }
  __device__ static uint32_t pair(const uint32_t* w, int p, const Unpack&) { return w[p]; }
};

template <class F, int TM, int NMAT, int BR>
__device__ __forceinline__ void wide_tile(const _Float16* __restrict__ Ax,
                                          const float* __restrict__ rs,
                                          const uint8_t* __restrict__ W0,
                                          const uint8_t* __restrict__ W1, float* __restrict__ C,
                                          uint32_t T, uint32_t N, uint32_t K) {
  constexpr WideLds L = wide_lds(F::kBf16, F::kChunks, TM, BR);
  constexpr int NA = TM;  // A pieces per thread and step (64 TM rows x 8 / 512)
  constexpr int NS = L.stages;
  constexpr int NG = L.groups;
  constexpr uint32_t BN = BR / NMAT;          // columns of C
  constexpr int WN = 4;                       // wavefronts in N (2 in M)
  constexpr int MT = 2 * TM, NT = BR / 64;    // 16 x 16 blocks of a wavefront
  extern __shared__ __attribute__((aligned(16))) uint8_t pf_wide[];
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t*)pf_wide;
  const uint32_t tid = threadIdx.x, lane = tid & 63;
  const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  // XCD-aware tile order, as the tile GEMM's: split, m, n with n fastest
  const uint32_t gx = gridDim.x, gy = gridDim.y, gz = gridDim.z, G = gx * gy * gz;
  uint32_t w = blockIdx.x + gx * (blockIdx.y + gy * blockIdx.z);
  if (G % 8 == 0) w = (w % 8) * (G / 8) + w / 8;
  const uint32_t tn = w % gx, tm = (w / gx) % gy, z = w / (gx * gy);
  const uint32_t m0 = tm * 64 * TM, n0 = tn * BN;
  const uint32_t nq = K / 128;
  const uint32_t q_begin = (uint32_t)((uint64_t)nq * z / gz);
  const uint32_t q_end = (uint32_t)((uint64_t)nq * (z + 1) / gz);
  const uint32_t s_end = 4 * q_end;
  const size_t row_bytes = F::kBf16 ? (size_t)K * 2 : (size_t)nq * (16 * F::kChunks);

  // A: piece c = 512 i + tid of a step is row c / 8, position c % 8, and comes
  // from chunk (c % 8) ^ swizzle(row); rows past T load row T - 1
  auto swz = [](uint32_t r) { return (r & 7) ^ ((r >> 3) & 1); };
  uint32_t a_off[NA];
#pragma unroll
  for (int i = 0; i < NA; i++) {
    const uint32_t r = 64 * i + (tid >> 3);
    a_off[i] = (min(m0 + r, T - 1) - m0) * (4 * K) + 16 * ((tid & 7) ^ swz(r));
  }
  const uint8_t* a_base = reinterpret_cast<const uint8_t*>(Ax) + (size_t)m0 * 4 * K;
  auto load_a = [&](uint32_t step, uint32_t st) {
    const uint8_t* base = a_base + (size_t)min(step, s_end - 1) * 128;
#pragma unroll
    for (int i = 0; i < NA; i++)
      load_lds16(a_off[i], base, lds0 + st * L.a + 8192 * i + 1024 * wave);
  };
  // W: piece c of four blocks is row c / kChunks, part c % kChunks (bf16: of a
  // step, row c / 4, position c % 4 from chunk (c % 4) ^ swizzle)
  constexpr int NB = F::kBf16 ? F::per(BR, 0) : (BR * F::kChunks + PF_WIDE_NT - 1) / PF_WIDE_NT;
  auto bswz = [](uint32_t r) { return ((r >> 1) ^ (r >> 2)) & 3; };
  const uint8_t* b_src[NB];
#pragma unroll
  for (int i = 0; i < NB; i++) {
    const uint32_t c = min(512u * i + tid, (uint32_t)BR * F::kChunks - 1);
    const uint32_t r = c / F::kChunks, part = c % F::kChunks;
    const uint8_t* W = r / BN ? W1 : W0;
    b_src[i] = W + (size_t)min(n0 + r % BN, N - 1) * row_bytes +
               16 * (F::kBf16 ? part ^ bswz(r) : part);
  }
  constexpr uint32_t kB0 = NS * L.a, kPad0 = kB0 + (F::kBf16 ? NS : NG) * L.b;
  auto load_b = [&](int i, uint32_t unit, uint32_t st) {  // unit: a group of four (bf16: a step)
    const uint32_t step_bytes = F::kBf16 ? 64 : 16 * F::kChunks;
    const uint32_t last = (F::kBf16 ? s_end : q_end) - 1;
    // a group's last load may need fewer wavefronts: the others' goes to the pad
    const bool pad = 512u * i + 64u * wave >= (uint32_t)BR * F::kChunks;
    load_lds16(b_src[i] + (size_t)min(unit, last) * step_bytes,
               lds0 + (pad ? kPad0 : kB0 + st * L.b + 8192 * i + 1024 * wave));
  };

  const uint32_t wm = (wave / WN) * (16 * MT), wn = wave % WN, g = lane >> 4, l16 = lane & 15;
  // this lane's bytes of an A row (hi halves: chunk g, lo: 4 + g) and its
  // weight rows (a pair: the first half of the blocks gate, the others the
  // same columns of up)
  const uint32_t a_hi = (wm + l16) * 128 + 16 * (g ^ swz(l16));
  const uint32_t a_lo = (wm + l16) * 128 + 16 * ((4 + g) ^ swz(l16));
  auto b_row = [&](int c) -> uint32_t {
    return NMAT == 2 ? BN * (c / (NT / 2)) + 8 * NT * wn + 16 * (c % (NT / 2)) + l16
                     : 16 * NT * wn + 16 * c + l16;
  };
  auto read_raw = [&](uint32_t (&r)[NT][F::kRaw], float (&d)[NT], uint32_t bst, int j) {
#pragma unroll
    for (int c = 0; c < NT; c++) {
      if constexpr (F::kBf16)
        F::raw(pf_wide + kB0 + bst * L.b + b_row(c) * 64 + 16 * (g ^ bswz(l16)), g, r[c], &d[c]);
      else
        F::raw(pf_wide + kB0 + bst * L.b + b_row(c) * (16 * F::kChunks) + j * (4 * F::kChunks), g, r[c], &d[c]);
    }
  };
  auto read_a = [&](half8 (&a)[2], uint32_t st, int i) {
    a[0] = *reinterpret_cast<const half8*>(pf_wide + st * L.a + a_hi + 2048 * i);
    a[1] = *reinterpret_cast<const half8*>(pf_wide + st * L.a + a_lo + 2048 * i);
  };

  f32x4 acc[MT][NT];
#pragma unroll
  for (int i = 0; i < MT; i++)
#pragma unroll
    for (int c = 0; c < NT; c++) acc[i][c] = f32x4{0.f, 0.f, 0.f, 0.f};
  // the runs' sums: of as many of the 16-row blocks as registers are left for
  constexpr int MR = TM <= 2 || BR == 128 ? MT : F::kBf16 ? 0 : TM == 3 ? 3 : 1;
  f32x4 runs[MR > 0 ? MR : 1][NT];
#pragma unroll
  for (int i = 0; i < MR; i++)
#pragma unroll
    for (int c = 0; c < NT; c++) runs[i][c] = f32x4{0.f, 0.f, 0.f, 0.f};
  const uint32_t nrun = q_end - q_begin;
  const uint32_t run = nrun > 16 ? 4 : nrun > 4 ? 2 : 1;  // groups of a run

  uint32_t step = 4 * q_begin;
  // first loads: the first groups of W and the first NS - 1 steps of A
  constexpr int per_step = NA + (F::kBf16 ? NB : 0);
#pragma unroll
  for (int p = 0; p < NS - 1; p++) {
    if constexpr (F::kBf16) {
#pragma unroll
      for (int i = 0; i < NB; i++) load_b(i, step + p, p);
    } else if (p < NG - 1) {
#pragma unroll
      for (int i = 0; i < NB; i++) load_b(i, q_begin + p, p);
    }
    load_a(step + p, p);
    if constexpr (!F::kBf16 && NS - 1 < NG - 1) {
      if (p == NS - 2) {
#pragma unroll
        for (int i = 0; i < NB; i++) load_b(i, q_begin + p + 1, p + 1);
      }
    }
  }
  wait_loads_barrier<(NS - 2) * per_step>();
  uint32_t st = 0, bq = 0;  // stages of this step's A and of this group's W
  const Unpack uc(F::kChunks == 9);
  half8 a[2][2];
  uint32_t raw[NT][F::kRaw];
  u32x4 b[NT], bn[NT];
  float d[NT], dn[NT], dp[NT];  // this step's scales, the next one's, the previous one's
  f32x4 t[2][NT];               // block sums of 16 rows: this one's, the previous one's
#pragma unroll
  for (int c = 0; c < NT; c++) {
    dp[c] = 0.f;
    t[1][c] = f32x4{0.f, 0.f, 0.f, 0.f};
  }
  static_assert(MT % 2 == 0, "the last 16 rows' sums are in t[1]");
  read_raw(raw, d, 0, 0);
  read_a(a[0], 0, 0);
#pragma unroll
  for (int c = 0; c < NT; c++)
#pragma unroll
    for (int p = 0; p < 4; p++) b[c][p] = F::pair(raw[c], p, uc);

  for (uint32_t q = q_begin; q < q_end;) {
    const uint32_t q_run = MR > 0 ? min(q + run, q_end) : q_end;
    for (; q < q_run; q++) {
      int nload = 0;
#pragma unroll
      for (int j = 0; j < 4; j++) {
        // loads of a later step's operands, into the stage that the previous
        // step read (every wave has passed a barrier since)
        uint32_t nst = st + NS - 1;
        nst = nst >= (uint32_t)NS ? nst - NS : nst;
        if constexpr (F::kBf16) {
#pragma unroll
          for (int i = 0; i < NB; i++) load_b(i, step + NS - 1, nst);
        } else {
          const uint32_t nbq = bq == 0 ? NG - 1 : bq - 1;
#pragma unroll
          for (int p = 0; p < F::per(BR, j); p++) load_b(nload + p, q + NG - 1, nbq);
          nload += F::per(BR, j);
        }
        load_a(step + NS - 1, nst);
        const uint32_t sn = st + 1 == (uint32_t)NS ? 0 : st + 1;
        // quantized: the next step's words are in LDS already (of the next group
        // since the barrier of this group's third step); they are unpacked
        // between the MFMAs
        if constexpr (!F::kBf16) read_raw(raw, dn, j < 3 ? bq : bq + 1 == (uint32_t)NG ? 0 : bq + 1, (j + 1) & 3);
#pragma unroll
        for (int i = 0; i < MT; i++) {
          if (i == MT - 1) {
            // The next step's operands have landed for every wave: of the loads
            // issued since, those of the last NS - 2 steps may be in flight; with
            // two groups of W, in a group's third step only the A of two steps
            // (the next group's last W went out in the second, ahead of that A).
            constexpr int flight = (NS - 2) * per_step;
            if (!F::kBf16 && NG == 2 && j == 2)
              wait_loads_barrier<flight < 2 * NA ? flight : 2 * NA>();
            else
              wait_loads_barrier<flight>();
            if constexpr (F::kBf16) read_raw(raw, dn, sn, 0);
            read_a(a[(i + 1) & 1], sn, 0);
          } else {
            read_a(a[(i + 1) & 1], st, i + 1);
          }
          // (the compiler would sink the reads to just ahead of their use)
          __builtin_amdgcn_sched_barrier(0);
#pragma unroll
          for (int h = 0; h < 2; h++)
#pragma unroll
            for (int c = 0; c < NT; c++) {
              if constexpr (F::kBf16) {
                acc[i][c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                    __builtin_bit_cast(bf16x8, a[i & 1][h]), __builtin_bit_cast(bf16x8, b[c]), acc[i][c], 0, 0, 0);
              } else {
                // one MFMA, then two scale FMAs of the previous 16 rows and a
                // share of the unpacking: an MFMA that finds the matrix pipe
                // busy holds up the SIMD's vector instructions too
                t[i & 1][c] = __builtin_amdgcn_mfma_f32_16x16x32_f16(
                    a[i & 1][h], __builtin_bit_cast(half8, b[c]), h ? t[i & 1][c] : f32x4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
                const int slot = h * NT + c;
#pragma unroll
                for (int e = 2 * slot; e < 2 * slot + 2; e++)
                  acc[(i + MT - 1) % MT][e / 4][e % 4] += (i ? d : dp)[e / 4] * t[(i + 1) & 1][e / 4][e % 4];
                if (i > 0) {
                  constexpr int slots = (MT - 1) * 2 * NT, pairs = 4 * NT;
                  const int u = (i - 1) * 2 * NT + slot;
#pragma unroll
                  for (int p = u * pairs / slots; p < (u + 1) * pairs / slots; p++)
                    bn[p / 4][p % 4] = F::pair(raw[p / 4], p % 4, uc);
                }
              }
            }
        }
#pragma unroll
        for (int c = 0; c < NT; c++) {
          if constexpr (F::kBf16) {
#pragma unroll
            for (int p = 0; p < 4; p++) b[c][p] = raw[c][p];
          } else {
            b[c] = bn[c];
            dp[c] = d[c];
            d[c] = dn[c];
          }
        }
        step++;
        st = sn;
      }
      bq = bq + 1 == (uint32_t)NG ? 0 : bq + 1;
    }
#pragma unroll
    for (int i = 0; i < MR; i++)
#pragma unroll
      for (int c = 0; c < NT; c++) {
        runs[i][c] += acc[i][c];
        acc[i][c] = f32x4{0.f, 0.f, 0.f, 0.f};
      }
  }
  if constexpr (!F::kBf16) {
#pragma unroll
    for (int e = 0; e < 4 * NT; e++) acc[MT - 1][e / 4][e % 4] += dp[e / 4] * t[1][e / 4][e % 4];
  }
#pragma unroll
  for (int i = 0; i < MR; i++)
#pragma unroll
    for (int c = 0; c < NT; c++) acc[i][c] += runs[i][c];
  // no load to LDS may outlive the workgroup
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");

  // epilogue: result register e of lane l -> row 4 (l / 16) + e, column l % 16
#pragma unroll
  for (int i = 0; i < MT; i++) {
#pragma unroll
    for (int e = 0; e < 4; e++) {
      const uint32_t row = m0 + wm + 16 * i + 4 * g + e;
      if (row >= T) continue;
      const float sr = rs[row];
      if constexpr (NMAT == 2) {
#pragma unroll
        for (int c = 0; c < NT / 2; c++) {
          const uint32_t col = n0 + 8 * NT * wn + 16 * c + l16;
          if (col >= N) continue;
          const float x = acc[i][c][e] * sr, y = acc[i][c + NT / 2][e] * sr;
          if (gz > 1) {
            C[((size_t)(2 * z) * T + row) * N + col] = x;
            C[((size_t)(2 * z + 1) * T + row) * N + col] = y;
          } else {
            C[(size_t)row * N + col] = gelu_tanh(x) * y;
          }
        }
      } else {
#pragma unroll
        for (int c = 0; c < NT; c++) {
          const uint32_t col = n0 + 16 * NT * wn + 16 * c + l16;
          if (col < N) C[((size_t)z * T + row) * N + col] = acc[i][c][e] * sr;
        }
      }
    }
  }
}

// (two wavefronts per SIMD at least; the registers and LDS of the 64 x 128 tile,
// but for Q8 weights, let a second workgroup onto a CU)
#define GH_WIDE_TM(FMT, F, TM, BR)                                                            \
  extern "C" __global__ __launch_bounds__(PF_WIDE_NT) __attribute__((amdgpu_waves_per_eu(2)))  \
  void gh_pf_wgemm_##FMT##_m##TM##_n##BR##_k(const _Float16* Ax, const float* rs,              \
                                             const uint8_t* W, float* C, uint32_t T,           \
                                             uint32_t N, uint32_t K) {                         \
    wide_tile<F, TM, 1, BR>(Ax, rs, W, W, C, T, N, K);                                         \
  }                                                                                            \
  extern "C" __global__ __launch_bounds__(PF_WIDE_NT) __attribute__((amdgpu_waves_per_eu(2)))  \
  void gh_pf_wgateup_##FMT##_m##TM##_n##BR##_k(const _Float16* Ax, const float* rs,            \
                                               const uint8_t* Wg, const uint8_t* Wu,           \
                                               float* Act, uint32_t T, uint32_t N,             \
                                               uint32_t K) {                                   \
    wide_tile<F, TM, 2, BR>(Ax, rs, Wg, Wu, Act, T, N, K);                                     \
  }
#define GH_WIDE(FMT, F)                                                            \
  GH_WIDE_TM(FMT, F, 1, 256) GH_WIDE_TM(FMT, F, 2, 256) GH_WIDE_TM(FMT, F, 3, 256) \
  GH_WIDE_TM(FMT, F, 4, 256) GH_WIDE_TM(FMT, F, 1, 128) GH_WIDE_TM(FMT, F, 2, 128) \
  GH_WIDE_TM(FMT, F, 3, 128)
GH_WIDE(q4, WQ4)
GH_WIDE(q8, WQ8)
GH_WIDE(bf16, WBf16)

// The row scale of the GEMM's A operand for a row whose largest |x| is m:
// s = 2^(e - 14) with 2^(e-1) <= m < 2^e (1 for m = 0), so every |x| / s
// < 2^14 fits fp16; returns s and sets *inv = 1 / s (both exact).
__device__ __forceinline__ float row_scale(float m, float* inv) {
  int e = 0;
  if (m > 0.f) frexpf(m, &e);
  const int sh = m > 0.f ? e - 14 : 0;
  *inv = ldexpf(1.f, -sh);
  return ldexpf(1.f, sh);
}

// The MFMA A operand of one f32 row (K <= PF_HALVES_K): hi = fp16(a / s),
// lo = fp16(a / s - hi) with s = row_scale(max|a|), in the ax layout
// (pf_ax_pos).  One workgroup per row; rs[t] = s.
#define PF_HALVES_NT 1024
#define PF_HALVES_G 2  // 8-element groups per thread
#define PF_HALVES_K (8 * PF_HALVES_NT * PF_HALVES_G)

// Round-to-nearest-even bf16 bits of a finite float.
__device__ __forceinline__ uint32_t pf_bf16_bits(float f) {
  const uint32_t b = __float_as_uint(f);
  return (b + 0x7FFFu + ((b >> 16) & 1u)) >> 16;
}

// hi = fp16(x), lo = fp16(x - hi) of one 8-element group, stored in the ax
// layout at dst (16-byte aligned): the group's hi halves, and 32 halves on its
// lo halves, each as one 16-byte store.  fmt 0: fp16 in K order; 1: fp16 in
// the Q4 unpacking's K order; 2: bf16 halves (hi = bf16(x), lo = bf16(x - hi),
// about 16 significant bits) in K order, for the bf16 weights' MFMA.
__device__ __forceinline__ void pf_store_group(const float (&x)[8], uint32_t fmt, _Float16* dst) {
  half8 hi, lo;
  if (fmt == 2u) {
    uint32_t hw[4], lw[4];
#pragma unroll
    for (int k = 0; k < 8; k += 2) {
      const uint32_t h0 = pf_bf16_bits(x[k]), h1 = pf_bf16_bits(x[k + 1]);
      const uint32_t l0 = pf_bf16_bits(x[k] - __uint_as_float(h0 << 16));
      const uint32_t l1 = pf_bf16_bits(x[k + 1] - __uint_as_float(h1 << 16));
      hw[k / 2] = h0 | (h1 << 16);
      lw[k / 2] = l0 | (l1 << 16);
    }
    *reinterpret_cast<u32x4*>(dst) = u32x4{hw[0], hw[1], hw[2], hw[3]};
    *reinterpret_cast<u32x4*>(dst + 32) = u32x4{lw[0], lw[1], lw[2], lw[3]};
    return;
  }
#pragma unroll
  for (int k = 0; k < 8; k++) {
    const int p = fmt == 1u ? ((k & 3) << 1) | (k >> 2) : k;
    const _Float16 h = (_Float16)x[k];
    hi[p] = h;
    lo[p] = (_Float16)(x[k] - (float)h);
  }
  *reinterpret_cast<half8*>(dst) = hi;
  *reinterpret_cast<half8*>(dst + 32) = lo;
}

extern "C" __global__ __launch_bounds__(PF_HALVES_NT) void gh_pf_halves_k(
    const float* __restrict__ A, _Float16* __restrict__ Ax,
    float* __restrict__ rs, uint32_t K, uint32_t perm) {
  __shared__ float red[PF_HALVES_NT / 64];
  const uint32_t t = blockIdx.x, tid = threadIdx.x, n8 = K / 8;
  const float4* a = reinterpret_cast<const float4*>(A + (size_t)t * K);
  float4 v[PF_HALVES_G][2];
  float m = 0.f;
#pragma unroll
  for (int u = 0; u < PF_HALVES_G; u++) {
    const uint32_t g = tid + u * PF_HALVES_NT, gc = g < n8 ? g : n8 - 1;
    v[u][0] = a[2 * gc];
    v[u][1] = a[2 * gc + 1];
#pragma unroll
    for (int h = 0; h < 2; h++)
      if (g < n8)
        m = fmaxf(m, fmaxf(fmaxf(fabsf(v[u][h].x), fabsf(v[u][h].y)), fmaxf(fabsf(v[u][h].z), fabsf(v[u][h].w))));
  }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) m = fmaxf(m, __shfl_xor(m, off, 64));
  if ((tid & 63) == 0) red[tid >> 6] = m;
  __syncthreads();
  m = 0.f;
#pragma unroll
  for (int w = 0; w < PF_HALVES_NT / 64; w++) m = fmaxf(m, red[w]);
  float inv;
  const float sc = row_scale(m, &inv);
#pragma unroll
  for (int u = 0; u < PF_HALVES_G; u++) {
    const uint32_t g = tid + u * PF_HALVES_NT;
    if (g < n8) {
      const float x[8] = {v[u][0].x * inv, v[u][0].y * inv, v[u][0].z * inv, v[u][0].w * inv,
                          v[u][1].x * inv, v[u][1].y * inv, v[u][1].z * inv, v[u][1].w * inv};
      pf_store_group(x, perm, Ax + (size_t)t * 2 * K + pf_ax_pos(8 * g, false));
    }
  }
  if (tid == 0) rs[t] = sc;
}

// C[T][N] from the Z partial planes of a split-K GEMM, added in z order (so
// the result does not depend on scheduling): the plain sum (nmat 1) or
// gelu_tanh(sum of gate planes) * (sum of up planes) (nmat 2).
extern "C" __global__ __launch_bounds__(PF_NT) void gh_pf_splitk_k(const float* __restrict__ P,
                                                                  float* __restrict__ C,
                                                                  uint32_t T, uint32_t N,
                                                                  uint32_t nz, uint32_t nmat) {
  const size_t tn = (size_t)T * N;
  for (size_t i = (size_t)blockIdx.x * PF_NT + threadIdx.x; i < tn; i += (size_t)gridDim.x * PF_NT) {
    float g = 0.f, u = 0.f;
#pragma unroll 4
    for (uint32_t z = 0; z < nz; z++) {
      g += P[(size_t)z * nmat * tn + i];
      if (nmat == 2) u += P[((size_t)z * 2 + 1) * tn + i];
    }
    C[i] = nmat == 2 ? gelu_tanh(g) * u : g;
  }
}

// ---------------------------------------------------------------------------
// Short batches (at most 48 tokens): the weight-streaming GEMM.
//
// With a few tokens a tile is mostly padding, so here every wavefront streams
// its own weight rows, one register set of 16 rows x SB quant blocks in flight
// while the previous set feeds the matrix cores, and the tokens take the MFMA's
// other dimension: v_mfma_f32_16x16x32_f16 (or _bf16) with A = 16 tokens x 32 K
// (the activation halves, as the tile GEMM reads them) and B = 32 K x 16
// weight rows (one quant block of each row, exact integers), so one MFMA
// pair (hi, lo) covers one block of 16 rows and the rows' block scales apply
// to its results.  With TG groups of 16 tokens each group is its own MFMA
// pair on the same weight fragment.
//
// MFMA 16x16x32 operand layout: lane l holds A[l % 16][8 (l / 16) + e] and
// B[8 (l / 16) + e][l % 16], e = 0..7; result register r of lane l is
// D[4 (l / 16) + r][l % 16].  So lane group g = l / 16 takes elements
// 8g .. 8g + 7 of each block (Q4_0: word 1 + g, unpacked in the order the ax
// layout keeps them), and D holds tokens 4g + r of weight row l % 16: one
// block scale per lane.
//
// A set is loaded as the decode streams load: lane l takes PB consecutive
// blocks (16-byte loads) of row l % 16, piece l / 16, so each row's SB
// blocks arrive as one contiguous run.  (Loading each lane's MFMA fragment
// directly, one scale and one word per block from 16 rows 2400 bytes apart,
// reads at about 1.3 TB/s against 5.4-6.0 TB/s for these runs.)  Lane group k
// then holds whole blocks PB k + i of its rows, where the fragments want word
// 1 + g in group g: a 4 x 4 transpose between registers and lane groups, four
// v_permlane swaps for four blocks, in registers (six more spread the four
// scales).  Taking the set through LDS instead (written as loaded, read back
// as fragments) cost a round trip per set and most of the LDS.
//
// Workgroup (x, z) of 8 waves (4 for narrow products) owns RGW row units of 16
// per wave (of each matrix of a gate/up pair, one after the other) and K blocks
// [z KR, z KR + KR) (KR and K / 32 multiples of 4): it stages that slice of the
// T <= 16 TG activation rows in LDS once, and wave w then streams its units with
// no further barrier.  gridDim.z > 1: plane z of [Z][NMAT][T][N] takes the raw
// sums times the row scale, as the tile GEMM's split form writes them;
// gridDim.z = 1: C takes the epilogue.
//
// What bounds it: at a few tokens the weights' bytes and the start (launch,
// first loads, staging), from 16 tokens the vector work per block (unpacking,
// scale FMAs) beside the MFMAs.  Timing-only copies, gate/up of 16 tokens
// (73.7 MB, 13.4 us at 5.5 TB/s): 28 us with its plane sum, 17-18 without the
// arithmetic, 24 without all loads but the first.  Against the form through
// LDS, us with the plane sums (Q4, 3 / 16 / 32 tokens): gate/up 31 / 34 / 46 ->
// 25 / 28 / 39, QKV 13.1 / 15.1 / 18.1 -> 10.7 / 12.2 / 16.1, o 10.0 / 11.4 /
// 13.5 -> 8.1 / 9.5 / 12.4, down 22 / 23 / 30 -> 16.7 / 19.6 / 25.2; Q8 gate/up of 16
// and 32 tokens 51 / 70 -> 38 / 48.
//
// Sums: half a set's blocks are one fp32 chain, these sums of a slice a second and
// the planes a third, so that wide slices cost no precision: against 64 bits the
// Q4 gate/up of 2 x 6144 x 2048, 33 tokens, is off by 1.52e-7, 1.63e-7 in chains of
// a whole set, 1.65e-7 in slices of 16 blocks each one chain; the 12B gate/up of 16
// tokens by 2.34e-7 with one chain per slice of 60.  It takes no measurable time.
// bf16 keeps one chain per slice: its 16-bit activations are 20 times further off,
// and a set's end then waits for its last MFMA (weights from memory, gate/up of 8
// tokens: 52.8 us, 59.5 with a sum per set).
//
// AF (the o and down inputs, and the kernel-level f32 entry points): A comes
// as f32 rows, and the staging splits each token's slice itself, with a
// power-of-two scale of its own (row_scale of the slice's largest |a|); plane z
// then carries that scale instead of the row's.  This saves the separate split
// launch (gh_pf_halves_k).
// ---------------------------------------------------------------------------
// Register r of lane group k <-> register k of lane group r.
__device__ __forceinline__ void transpose4(uint32_t& w0, uint32_t& w1, uint32_t& w2, uint32_t& w3) {
  const auto a = __builtin_amdgcn_permlane32_swap(w0, w2, false, false);
  const auto b = __builtin_amdgcn_permlane32_swap(w1, w3, false, false);
  const auto c = __builtin_amdgcn_permlane16_swap(a[0], b[0], false, false);
  const auto d = __builtin_amdgcn_permlane16_swap(a[1], b[1], false, false);
  w0 = c[0];
  w1 = c[1];
  w2 = d[0];
  w3 = d[1];
}
// d[k] = v of lane group k
__device__ __forceinline__ void spread4(uint32_t v, float (&d)[4]) {
  const auto a = __builtin_amdgcn_permlane32_swap(v, v, false, false);
  const auto b = __builtin_amdgcn_permlane16_swap(a[0], a[0], false, false);
  const auto c = __builtin_amdgcn_permlane16_swap(a[1], a[1], false, false);
  d[0] = __uint_as_float(b[0]);
  d[1] = __uint_as_float(b[1]);
  d[2] = __uint_as_float(c[0]);
  d[3] = __uint_as_float(c[1]);
}

// A streamed format: kPB blocks per lane and set.  take: block i of every lane
// group's piece as the fragments' words (w[k]: block kPB k + i) and scales;
// half: the operand from a fragment's words.
struct SQ4 {  // Q4_0 (src/quant.zig:55-90): {f32 d, 4 words of nibbles}
  static constexpr uint32_t kBlockBytes = 20;
  static constexpr int kPB = 4, kWords = 1;  // 80 bytes
  static constexpr bool kBf16 = false;
  static constexpr uint32_t kFmt = 1;  // pf_store_group format of the A halves
  __device__ static void take(const uint32_t* r, int i, uint32_t (&w)[4][kWords], float (&d)[4]) {
#pragma unroll
    for (int k = 0; k < 4; k++) w[k][0] = r[5 * i + 1 + k];
    transpose4(w[0][0], w[1][0], w[2][0], w[3][0]);
    spread4(r[5 * i], d);
  }
  __device__ static half8 half(const uint32_t* w, const Unpack& c) {
    u32x4 o;
#pragma unroll
    for (int p = 0; p < 4; p++) o[p] = WQ4::pair(w, p, c);
    return __builtin_bit_cast(half8, o);
  }
};

struct SQ8 {  // Q8_0 (src/quant.zig:20-51): {f32 d, 8 words of int8}
  static constexpr uint32_t kBlockBytes = 36;
  static constexpr int kPB = 4, kWords = 2;  // 144 bytes
  static constexpr bool kBf16 = false;
  static constexpr uint32_t kFmt = 0;
  __device__ static void take(const uint32_t* r, int i, uint32_t (&w)[4][kWords], float (&d)[4]) {
#pragma unroll
    for (int h = 0; h < 2; h++) {
#pragma unroll
      for (int k = 0; k < 4; k++) w[k][h] = r[9 * i + 1 + 2 * k + h];
      transpose4(w[0][h], w[1][h], w[2][h], w[3][h]);
    }
    spread4(r[9 * i], d);
  }
  __device__ static half8 half(const uint32_t* w, const Unpack& c) {
    u32x4 o;
#pragma unroll
    for (int p = 0; p < 4; p++) o[p] = WQ8::pair(w, p, c);
    return __builtin_bit_cast(half8, o);
  }
};

struct SBf16 {  // bf16 rows: 32-element segments of 64 bytes, no scale
  static constexpr uint32_t kBlockBytes = 64;
  static constexpr int kPB = 2, kWords = 4;  // 128 bytes
  static constexpr bool kBf16 = true;
  static constexpr uint32_t kFmt = 2;
  __device__ static void take(const uint32_t* r, int i, uint32_t (&w)[4][kWords], float (&d)[4]) {
#pragma unroll
    for (int h = 0; h < 4; h++) {
#pragma unroll
      for (int k = 0; k < 4; k++) w[k][h] = r[16 * i + 4 * k + h];
      transpose4(w[0][h], w[1][h], w[2][h], w[3][h]);
      d[h] = 1.f;
    }
  }
  __device__ static half8 half(const uint32_t* w, const Unpack&) {
    return __builtin_bit_cast(half8, u32x4{w[0], w[1], w[2], w[3]});
  }
};

// 8-element groups a thread holds while it splits f32 rows, for TG groups of
// 16 tokens: a K slice of kr blocks has 4 kr groups per token, over the
// workgroup's threads per token (a power of two)
template <int TG>
struct StreamStage {
  static constexpr int kPer = TG <= 2 ? 10 : 16;
  // threads per token of a workgroup of `waves` waves
  __device__ static uint32_t tpt(uint32_t waves) { return waves * (TG <= 1 ? 4 : TG == 2 ? 2 : 1); }
};

// TG groups of 16 tokens (T <= 16 TG); TG = 0: at most 8 tokens, whose hi and
// lo halves are rows 0-7 and 8-15 of one MFMA.
template <class F, int NMAT, bool AF, int TG>
__device__ __forceinline__ void stream_gemm(const _Float16* __restrict__ Ax,
                                            const float* __restrict__ rs,
                                            const uint8_t* __restrict__ W0,
                                            const uint8_t* __restrict__ W1,
                                            float* __restrict__ C, uint32_t T, uint32_t N,
                                            uint32_t K, uint32_t KR, uint32_t RGW) {
  constexpr int PB = F::kPB, SB = 4 * PB, NV = PB * (int)F::kBlockBytes / 16;
  constexpr bool kPack = TG == 0;
  constexpr int NG = kPack ? 1 : TG, NH = kPack ? 1 : 2;  // token groups, halves apart
  extern __shared__ __attribute__((aligned(16))) uint8_t pf_slice[];
  const uint32_t tid = threadIdx.x, lane = tid & 63;
  const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const uint32_t nthr = blockDim.x, nw = nthr / 64;
  const uint32_t g = lane >> 4, li = lane & 15;
  const uint32_t nb = K / 32, z = blockIdx.z;
  const uint32_t b0 = z * KR, nk = min(nb - b0, KR);  // the host keeps b0 < nb, 4 | nk
  const uint32_t stride = KR * 128 + 16;              // bytes per staged token row
  const size_t row_bytes = (size_t)nb * F::kBlockBytes;
  const uint32_t kchunks = (nk + SB - 1) / SB;  // sets per row unit
  const uint32_t nchunks = RGW * NMAT * kchunks;
  const uint32_t u0 = blockIdx.x * nw * RGW + wave;  // unit j of this wave: u0 + nw j
  // token rows of this lane's A fragments (one per group of 16 tokens):
  // tokens past T read token T - 1 (their D rows are never stored)
  const uint8_t* al_row[NG];
#pragma unroll
  for (int h = 0; h < NG; h++)
    al_row[h] = pf_slice + min(kPack ? li & 7 : 16 * h + li, T - 1) * stride + 16 * g + (kPack && li >= 8 ? 64 : 0);

  // Set c: pass j = c / kchunks over the slice (unit j / NMAT; of a gate/up pair
  // the gate rows, then the up rows), blocks kb0 .. kb0 + SB - 1.  Lane l loads
  // blocks kb0 + PB (l / 16) .. + PB - 1 of row l % 16 (a piece past the slice
  // loads the last one instead and enters as zeros).
  u32x4 ra[NV], rb[NV];
  auto load = [&](uint32_t c, u32x4(&r)[NV]) {
    const uint32_t j = c / kchunks, kb0 = (c % kchunks) * SB;
    const uint32_t kb = min(kb0 + PB * g, nk - PB);
    const uint32_t row = min(16 * (u0 + nw * (j / NMAT)) + li, N - 1);
    const uint8_t* src = (j % NMAT ? W1 : W0) + (size_t)row * row_bytes + (size_t)(b0 + kb) * F::kBlockBytes;
#pragma unroll
    for (int v = 0; v < NV; v++) r[v] = *(gvec_ptr)(src + 16 * v);
  };

  // The slice's loads first, then the first sets' (loads return in order, and
  // the activations come from L2): the staging below runs while those are in
  // flight.  AF: tpt threads per token; thread `sub` takes 8-element groups
  // sub, sub + tpt, ... of the slice (4 nk of them).  Else: 16-byte chunks
  // tid, tid + nthr, ... of the T rows' 8 nk each.
  __shared__ float slice_scale[16 * NG];  // AF: each token's scale for this slice
  constexpr int PER = StreamStage<TG>::kPer;
  const uint32_t tpt = StreamStage<TG>::tpt(nw);
  const uint32_t ngr = nk * 4, at = tid / tpt, sub = tid % tpt, chunks = T * nk * 8;
  float xv[AF ? PER : 1][8];
  u32x4 cv[AF ? 1 : 2 * PER];
  if constexpr (AF) {
    const float* src = reinterpret_cast<const float*>(Ax) + (size_t)min(at, T - 1) * K + (size_t)b0 * 32;
#pragma unroll
    for (int i = 0; i < PER; i++) {
      if (tpt * i >= ngr) continue;  // uniform
      const uint32_t gi = min(sub + tpt * i, ngr - 1);
      const float4 a = *reinterpret_cast<const float4*>(src + 8 * gi);
      const float4 b = *reinterpret_cast<const float4*>(src + 8 * gi + 4);
      xv[i][0] = a.x; xv[i][1] = a.y; xv[i][2] = a.z; xv[i][3] = a.w;
      xv[i][4] = b.x; xv[i][5] = b.y; xv[i][6] = b.z; xv[i][7] = b.w;
    }
  } else {
#pragma unroll
    for (int i = 0; i < 2 * PER; i++) {
      if (nthr * i >= chunks) continue;  // uniform
      const uint32_t c = min(tid + nthr * i, chunks - 1), t = c / (nk * 8), q = c % (nk * 8);
      cv[i] = *reinterpret_cast<const u32x4*>(Ax + (size_t)t * 2 * K + (size_t)b0 * 64 + 8 * q);
    }
  }
  asm volatile("" ::: "memory");
  load(0, ra);
  if (nchunks > 1) load(1, rb);
  asm volatile("" ::: "memory");
  if constexpr (AF) {
    float m = 0.f;
#pragma unroll
    for (int i = 0; i < PER; i++) {
      if (tpt * i >= ngr) continue;
#pragma unroll
      for (int k = 0; k < 8; k++) m = fmaxf(m, fabsf(xv[i][k]));
    }
    for (uint32_t off = tpt / 2; off > 0; off >>= 1) m = fmaxf(m, __shfl_xor(m, off, 64));
    float inv;
    const float sc = row_scale(m, &inv);
    if (at < T) {
#pragma unroll
      for (int i = 0; i < PER; i++) {
        const uint32_t gi = sub + tpt * i;  // group gi: block gi / 4, part gi % 4
        if (gi < ngr) {
          float y[8];
#pragma unroll
          for (int k = 0; k < 8; k++) y[k] = xv[i][k] * inv;
          pf_store_group(y, F::kFmt,
                         reinterpret_cast<_Float16*>(pf_slice + at * stride + (gi >> 2) * 128 + (gi & 3) * 16));
        }
      }
      if (sub == 0) slice_scale[at] = sc;
    }
  } else {
#pragma unroll
    for (int i = 0; i < 2 * PER; i++) {
      const uint32_t c = tid + nthr * i;
      if (c < chunks) *reinterpret_cast<u32x4*>(pf_slice + c / (nk * 8) * stride + 16 * (c % (nk * 8))) = cv[i];
    }
  }
  __syncthreads();

  const Unpack uc(F::kBlockBytes == 36);
  f32x4 total[NG], gate[NG];  // gate: the unit's sums of the first matrix of a pair
#pragma unroll
  for (int h = 0; h < NG; h++) total[h] = f32x4{0.f, 0.f, 0.f, 0.f};

  // the sums of pass j to its unit's plane (or C), or kept; and clear them
  auto epilogue = [&](uint32_t j) {
    const bool keep = NMAT == 2 && j % 2 == 0;
    const uint32_t n = 16 * (u0 + nw * (j / NMAT)) + li;
#pragma unroll
    for (int h = 0; h < NG; h++) {
      const f32x4 sum = total[h];
      total[h] = f32x4{0.f, 0.f, 0.f, 0.f};
      if (keep) {
        gate[h] = sum;
        continue;
      }
#pragma unroll
      for (int r = 0; r < 4; r++) {
        float v[NMAT];
        v[NMAT - 1] = sum[r];
        if constexpr (NMAT == 2) v[0] = gate[h][r];
        if constexpr (kPack) {  // rows 8 apart: lane groups 2 apart
#pragma unroll
          for (int q = 0; q < NMAT; q++) {
            const auto o = __builtin_amdgcn_permlane32_swap(__float_as_uint(v[q]), __float_as_uint(v[q]), false, false);
            v[q] = __uint_as_float(o[0]) + __uint_as_float(o[1]);
          }
        }
        const uint32_t t = 16 * h + 4 * g + r;
        if (t >= T || n >= N) continue;
        const float sr = AF ? slice_scale[t] : rs[t];
        if (NMAT == 2 && gridDim.z == 1) {
          C[(size_t)t * N + n] = gelu_tanh(v[0] * sr) * (v[NMAT - 1] * sr);
        } else {
#pragma unroll
          for (int q = 0; q < NMAT; q++) C[((size_t)(NMAT * z + q) * T + t) * N + n] = v[q] * sr;
        }
      }
    }
  };

  // set c into the sums
  auto compute = [&](uint32_t c, u32x4(&r)[NV]) {
    const uint32_t kb0 = (c % kchunks) * SB;
    if (kb0 + SB > nk) {  // the slice's last set is partial
      if (kb0 + PB * g >= nk) {
#pragma unroll
        for (int i = 0; i < NV; i++) r[i] = u32x4{0, 0, 0, 0};
      }
    }
    // Blocks PB k + i in the order i, then k.  While a block's MFMAs run, the
    // next one's activations are on their way from LDS and its weights are
    // unpacked; its scale FMAs follow.
    uint32_t flat[4 * NV];
#pragma unroll
    for (int e = 0; e < 4 * NV; e++) flat[e] = r[e / 4][e % 4];
    auto read_a = [&](half8(&x)[NH][NG], int p) {
      const uint32_t kb = min(kb0 + PB * (p % 4) + p / 4, nk - 1);
#pragma unroll
      for (int h = 0; h < NG; h++)
#pragma unroll
        for (int s = 0; s < NH; s++)
          x[s][h] = *reinterpret_cast<const half8*>(al_row[h] + kb * 128 + 64 * s);
    };
    half8 x[2][NH][NG], b;
    uint32_t w[4][F::kWords];
    float d[2][4];
    f32x4 acc[NG];
#pragma unroll
    for (int h = 0; h < NG; h++) acc[h] = F::kBf16 ? total[h] : f32x4{0.f, 0.f, 0.f, 0.f};
    read_a(x[0], 0);
    F::take(flat, 0, w, d[0]);
    b = F::half(w[0], uc);
#pragma unroll
    for (int p = 0; p < SB; p++) {
      if (p + 1 < SB) read_a(x[(p + 1) & 1], p + 1);
      // (the compiler would sink the reads to just ahead of their use)
      __builtin_amdgcn_sched_barrier(0);
      f32x4 t[NG];
#pragma unroll
      for (int s = 0; s < NH; s++)
#pragma unroll
        for (int h = 0; h < NG; h++) {
          const half8 v = x[p & 1][s][h];
          if constexpr (F::kBf16)
            acc[h] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, v),
                                                             __builtin_bit_cast(bf16x8, b), acc[h], 0, 0, 0);
          else
            t[h] = __builtin_amdgcn_mfma_f32_16x16x32_f16(v, b, s ? t[h] : f32x4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
        }
      if (p + 1 < SB) {
        if (p % 4 == 3) F::take(flat, p / 4 + 1, w, d[(p / 4 + 1) & 1]);
        b = F::half(w[(p + 1) % 4], uc);
      }
      if constexpr (!F::kBf16) {
#pragma unroll
        for (int h = 0; h < NG; h++) {
#pragma unroll
          for (int e = 0; e < 4; e++) acc[h][e] += d[(p / 4) & 1][p % 4] * t[h][e];
          // (pinned here: put off, the FMAs keep every block's sums in registers)
          asm volatile("" : "+v"(acc[h]));
          if (p == SB / 2 - 1) {
            total[h] += acc[h];
            acc[h] = f32x4{0.f, 0.f, 0.f, 0.f};
          }
        }
      }
    }
#pragma unroll
    for (int h = 0; h < NG; h++) {
      if constexpr (F::kBf16)
        total[h] = acc[h];
      else
        total[h] += acc[h];
    }
  };

  for (uint32_t c = 0; c < nchunks; c += 2) {
    compute(c, ra);
    if (c % kchunks == kchunks - 1) epilogue(c / kchunks);
    if (c + 2 < nchunks) load(c + 2, ra);
    if (c + 1 < nchunks) {
      compute(c + 1, rb);
      if ((c + 1) % kchunks == kchunks - 1) epilogue((c + 1) / kchunks);
      if (c + 3 < nchunks) load(c + 3, rb);
    }
  }
}

// t0: up to 8 tokens, t1 - t3: up to 16, 32, 48
#define GH_SGEMM_TG(NAME, F, NMAT, AF, TG)                                                   \
  extern "C" __global__ __launch_bounds__(512) void NAME##_t##TG##_k(                       \
      const _Float16* Ax, const float* rs, const uint8_t* W0, const uint8_t* W1, float* C,  \
      uint32_t T, uint32_t N, uint32_t K, uint32_t KR, uint32_t RGW) {                      \
    stream_gemm<F, NMAT, AF, TG>(Ax, rs, W0, W1, C, T, N, K, KR, RGW);                      \
  }
#define GH_SGEMM_TG2(FMT, F, TG)                      \
  GH_SGEMM_TG(gh_pf_sgemm_##FMT, F, 1, false, TG)     \
  GH_SGEMM_TG(gh_pf_sgemm_##FMT##_f, F, 1, true, TG)
#define GH_SGATEUP_TG2(FMT, F, TG)                    \
  GH_SGEMM_TG(gh_pf_sgateup_##FMT, F, 2, false, TG)   \
  GH_SGEMM_TG(gh_pf_sgateup_##FMT##_f, F, 2, true, TG)
// (the lengths that the host streams: longer ones take the wide tile)
GH_SGEMM_TG2(q4, SQ4, 0) GH_SGEMM_TG2(q4, SQ4, 1) GH_SGEMM_TG2(q4, SQ4, 2) GH_SGEMM_TG2(q4, SQ4, 3)
GH_SGEMM_TG2(q8, SQ8, 0) GH_SGEMM_TG2(q8, SQ8, 1) GH_SGEMM_TG2(q8, SQ8, 2) GH_SGEMM_TG2(q8, SQ8, 3)
GH_SGEMM_TG2(bf16, SBf16, 0) GH_SGEMM_TG2(bf16, SBf16, 1) GH_SGEMM_TG2(bf16, SBf16, 2)
GH_SGATEUP_TG2(q4, SQ4, 0) GH_SGATEUP_TG2(q4, SQ4, 1) GH_SGATEUP_TG2(q4, SQ4, 2) GH_SGATEUP_TG2(q4, SQ4, 3)
GH_SGATEUP_TG2(q8, SQ8, 0) GH_SGATEUP_TG2(q8, SQ8, 1) GH_SGATEUP_TG2(q8, SQ8, 2) GH_SGATEUP_TG2(q8, SQ8, 3)
GH_SGATEUP_TG2(bf16, SBf16, 0) GH_SGATEUP_TG2(bf16, SBf16, 1)

// ---------------------------------------------------------------------------
// Row-wise x prologue for T tokens (the batched form of the decode GEMVs'
// fused norms, src/gpu/model_dispatch.zig:21,32-34,39-41):
//   mode 1: xn = RMSNorm(x) * w
//   mode 2: x <- (x + RMSNorm(r) * wr) * s  (r as given when wr is null),
//           stored back as the residual stream; xn = RMSNorm(x) * w
// In mode 2, r may arrive as rz unsummed K-split planes of a GEMM ([rz][T][H]);
// they are added in plane order, as gh_pf_splitk_k adds them.
// One workgroup per token row.
// ---------------------------------------------------------------------------
template <int NT>
__device__ __forceinline__ float block_sum(float v, float* red) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
  __syncthreads();
  float t = 0.f;
#pragma unroll
  for (int w = 0; w < NT / 64; w++) t += red[w];
  __syncthreads();
  return t;
}

#define PF_NORM_NT 1024
#define PF_ROW_MAX 8  // elements per thread (one 8-element group): hidden <= 8192

// Every load (x, r, wr, w) is issued before any is used, with clamped
// indices and stand-in pointers for the operands a mode does not read, so
// the row costs one global round trip rather than one per operand.  The
// normed row goes out as the GEMM's A operand: fp16 hi/lo halves in the ax
// layout (pf_ax_pos, [T][2H]) and the row scale rs[t], as gh_pf_halves_k
// makes them.
template <int NT>
__device__ __forceinline__ float block_max(float v, float* red) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v = fmaxf(v, __shfl_xor(v, off, 64));
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
  __syncthreads();
  float t = 0.f;
#pragma unroll
  for (int w = 0; w < NT / 64; w++) t = fmaxf(t, red[w]);
  __syncthreads();
  return t;
}

template <int NT>
__device__ __forceinline__ void pf_norm_row(float* X, const float* R, const float* wr,
                                            const float* w, _Float16* Xa, float* rs, uint32_t H,
                                            float s, float eps, uint32_t mode, uint32_t perm,
                                            uint32_t rz) {
  __shared__ float red[NT / 64];
  // thread t owns the 8-element group t of the row (H <= 8 * NT)
  const uint32_t t = blockIdx.x, tid = threadIdx.x, n8 = H / 8;
  const bool add = mode == 2, has_wr = wr != nullptr, act = tid < n8;
  const uint32_t e0 = 8 * (act ? tid : n8 - 1);
  float* x = X + (size_t)t * H;
  const float* r = add ? R + (size_t)t * H : x;
  const float* wrp = has_wr ? wr : w;
  float v[8], rv[8], wv[8], wrv[8];
  auto load8 = [&](const float* p, float (&o)[8]) {
    const float4 a = *reinterpret_cast<const float4*>(p + e0);
    const float4 b = *reinterpret_cast<const float4*>(p + e0 + 4);
    o[0] = a.x; o[1] = a.y; o[2] = a.z; o[3] = a.w;
    o[4] = b.x; o[5] = b.y; o[6] = b.z; o[7] = b.w;
  };
  load8(x, v);
  load8(r, rv);
  load8(w, wv);
  load8(wrp, wrv);
  if (add) {
    // planes 1 .. rz - 1, 8 in flight at a time (clamped indices), added in
    // plane order
    const size_t plane = (size_t)gridDim.x * H;
    for (uint32_t z = 1; z < rz; z += 8) {
      float pv[8][8];
#pragma unroll
      for (int u = 0; u < 8; u++) load8(r + (size_t)min(z + u, rz - 1) * plane, pv[u]);
#pragma unroll
      for (int u = 0; u < 8; u++)
        if (z + u < rz) {  // uniform
#pragma unroll
          for (int k = 0; k < 8; k++) rv[k] += pv[u][k];
        }
    }
    float ss = 0.f;
#pragma unroll
    for (int k = 0; k < 8; k++) ss += rv[k] * rv[k];
    ss = act ? ss : 0.f;
    const float inv_r = has_wr ? 1.0f / sqrtf(block_sum<NT>(ss, red) / (float)H + eps) : 1.0f;
#pragma unroll
    for (int k = 0; k < 8; k++) {
      const float rr = has_wr ? rv[k] * inv_r * wrv[k] : rv[k];
      v[k] = (v[k] + rr) * s;
    }
    if (act) {
      *reinterpret_cast<float4*>(x + e0) = make_float4(v[0], v[1], v[2], v[3]);
      *reinterpret_cast<float4*>(x + e0 + 4) = make_float4(v[4], v[5], v[6], v[7]);
    }
  }
  float ss = 0.f;
#pragma unroll
  for (int k = 0; k < 8; k++) ss += v[k] * v[k];
  ss = act ? ss : 0.f;
  const float inv = 1.0f / sqrtf(block_sum<NT>(ss, red) / (float)H + eps);
  float m = 0.f;
#pragma unroll
  for (int k = 0; k < 8; k++) {
    v[k] = v[k] * inv * wv[k];
    m = fmaxf(m, fabsf(v[k]));
  }
  float sinv;
  const float sc = row_scale(block_max<NT>(act ? m : 0.f, red), &sinv);
  if (act) {
    float y[8];
#pragma unroll
    for (int k = 0; k < 8; k++) y[k] = v[k] * sinv;
    pf_store_group(y, perm, Xa + (size_t)t * 2 * H + pf_ax_pos(e0, false));
  }
  if (tid == 0) rs[t] = sc;
}

// 1024 threads for rows of up to 8192, 512 for rows of up to 4096 (the 12B
// hidden 3840: 480 groups, so the 1024-thread form idles more than half its
// threads and holds half as many rows per CU)
extern "C" __global__ __launch_bounds__(PF_NORM_NT) void gh_pf_norm_k(
    float* X, const float* R, const float* wr, const float* w, _Float16* Xa,
    float* rs, uint32_t H, float s, float eps, uint32_t mode, uint32_t perm, uint32_t rz) {
  pf_norm_row<PF_NORM_NT>(X, R, wr, w, Xa, rs, H, s, eps, mode, perm, rz);
}
extern "C" __global__ __launch_bounds__(512) void gh_pf_norm_512_k(
    float* X, const float* R, const float* wr, const float* w, _Float16* Xa,
    float* rs, uint32_t H, float s, float eps, uint32_t mode, uint32_t perm, uint32_t rz) {
  pf_norm_row<512>(X, R, wr, w, Xa, rs, H, s, eps, mode, perm, rz);
}
