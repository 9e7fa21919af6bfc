// C[M, N] = A[M, K] * W[N, K]^T for five and more rows of float32 (the 32-bit path) on the bf16 matrix
// cores, with no operand rounded: every float is the sum of three bf16 numbers,
//     x = x0 + x1 + x2,   x0 = x rounded to the nearest bf16 number, x1 = x - x0 rounded likewise, x2 = x - x0 - x1,
// exactly (both differences are exact; with x in [1, 2) x1 is at most 2^-8, x2 at most 2^-17 and a multiple of 2^-23, six
// bits).  A product of two floats is then nine products of bf16 numbers, each exact in float32, of which the six
// x0 w0, x0 w1, x1 w0, x1 w1, x0 w2, x2 w0 are taken: x1 w2 + x2 w1 + x2 w2 is what is left out, at most 2^-24 of the
// product (at 1.0038986 squared; no more than one rounding) and 2^-28 of it on the average of the mantissas, of either sign.
// (Planes cut instead of rounded all have the number's sign and are twice and four times as large: 2^-21 at worst, 2^-24.6 on
// the average, always towards zero.)  Sums are float32, in two levels.  What remains with a sign: the matrix cores cut an
// addend two bits behind the last place of the sum, 2^-26 of a stage's sum where all six products go to one accumulator.
//
// Range: bf16 has the exponents of float32 but no bits below 2^-133, and what the matrix instruction does with numbers
// below 2^-126 is not relied on.  So results that such numbers can have reached are computed again, see redo_limit.
//
// Why: the float32 matrix instruction runs at a sixteenth of the bf16 rate; six bf16 instructions for the same terms
// are 2.7 times as fast where both are at their peak.
#include "common.h"

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float floatx16_t __attribute__((ext_vector_type(16)));
typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));

union Frag8 {
  u32x4_t u;
  bf16x8_t v;
  f32x4_t f;
};

#define SP_BN 128                  // rows of W a workgroup owns
#define SP_WPITCH (SP_BN + 8)      // 16-byte units between the two halves of a stage's columns of W in LDS
// Stages of 16 columns summed in one accumulator before they join the total, out of `n`.  Long inner sizes take more, which
// balances the roundings of the two sums: distance to 64 bits (rms) with 16 / 24 / 32 of them, operands of one sign, K 14336
// 1.02e-7 / 0.90e-7 / 0.85e-7 of the result, of either sign 3.0e-7 / 3.4e-7 / 3.8e-7 (the float32 instruction: 0.95e-7, 4.2e-7).
__device__ __forceinline__ int flush_after(int n) { return n >= 1280 ? 32 : n >= 640 ? 24 : 16; }
#define SP_ROWS_FLUSH 32           // the same in the kernel of few rows, in stages of 64 or 128 columns

typedef __attribute__((address_space(1))) const void* gptr_t;
// All but the newest n of this wave's loads have landed and its LDS operations are done; then the workgroup's barrier
// (which itself waits for nothing: loads for later stages stay in flight across it).
#define SP_STAGE_END(n)                                                                   \
  do {                                                                                    \
    __builtin_amdgcn_sched_barrier(0);                                                    \
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(n) : "memory");      \
    __builtin_amdgcn_sched_barrier(0);                                                    \
  } while (0)
#define SGB(kind, n) __builtin_amdgcn_sched_group_barrier(kind, n, 0)
#define SGB_VALU 0x2
#define SGB_MFMA 0x8
#define SGB_VMEM_READ 0x20
#define SGB_DS_READ 0x100
#define SGB_DS_WRITE 0x200

// Two floats as bf16 numbers, rounded to the nearest (ties to even), side by side, and the first and second of such a pair.
// (The instruction by name: where one of the pair is used again the compiler converts it once more.)
__device__ __forceinline__ uint32_t round2(float lo, float hi) {
  uint32_t u;
  asm("v_cvt_pk_bf16_f32 %0, %1, %2" : "=v"(u) : "v"(lo), "v"(hi));
  return u;
}
__device__ __forceinline__ float first_of(uint32_t u) { return __uint_as_float(u << 16); }
__device__ __forceinline__ float second_of(uint32_t u) { return __uint_as_float(u & 0xffff0000u); }

// Eight floats into the three planes (eight bf16 numbers each, in order).
__device__ __forceinline__ void split8(const f32x4_t& a, const f32x4_t& b, u32x4_t (&p)[3]) {
  const float x[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const uint32_t u0 = round2(x[2 * i], x[2 * i + 1]);
    const float r0 = x[2 * i] - first_of(u0), r1 = x[2 * i + 1] - second_of(u0);
    const uint32_t u1 = round2(r0, r1);
    p[0][i] = u0;
    p[1][i] = u1;
    p[2][i] = round2(r0 - first_of(u1), r1 - second_of(u1));
  }
}

// The largest size among m and eight floats (NaN aside).
__device__ __forceinline__ void max8(float& m, const f32x4_t& a, const f32x4_t& b) {
  asm("v_max3_f32 %0, |%1|, |%2|, %0" : "+v"(m) : "v"(a.x), "v"(a.y));
  asm("v_max3_f32 %0, |%1|, |%2|, %0" : "+v"(m) : "v"(a.z), "v"(a.w));
  asm("v_max3_f32 %0, |%1|, |%2|, %0" : "+v"(m) : "v"(b.x), "v"(b.y));
  asm("v_max3_f32 %0, |%1|, |%2|, %0" : "+v"(m) : "v"(b.z), "v"(b.w));
}

// The rows of A as planes, in the order the product reads them: 16-byte unit ((stage * 3 + plane) * 2 + half) * Mp + row
// holds columns 16 stage + 8 half .. + 7 of a row.  Columns beyond K and rows beyond M are zeros.  A workgroup takes 32
// rows (Mp is a multiple of them) by 64 columns and leaves their largest size in `most` [rows / 32][columns / 64].
__global__ __launch_bounds__(256) void split_rows_kernel(const float* __restrict__ A, u32x4_t* __restrict__ P,
                                                        float* __restrict__ most, int M, int Mp, int K) {
  __shared__ float sizes[4];
  const int k8 = blockIdx.y * 8 + (threadIdx.x & 7);
  const int row = blockIdx.x * 32 + (threadIdx.x >> 3);
  const f32x4_t zero4 = {0.f, 0.f, 0.f, 0.f};
  f32x4_t a = zero4, b = zero4;
  const int k = k8 * 8;
  if (row < M) {
    const float* p = A + (size_t)row * K + k;
    if (k < K) a = *reinterpret_cast<const f32x4_t*>(p);
    if (k + 4 < K) b = *reinterpret_cast<const f32x4_t*>(p + 4);
  }
  u32x4_t q[3];
  split8(a, b, q);
#pragma unroll
  for (int i = 0; i < 3; ++i) P[((size_t)((k8 >> 1) * 3 + i) * 2 + (k8 & 1)) * Mp + row] = q[i];
  float m = 0.f;
  max8(m, a, b);
  m = wave_max(m);
  if ((threadIdx.x & 63) == 0) sizes[threadIdx.x >> 6] = m;
  __syncthreads();
  if (threadIdx.x == 0)
    most[(size_t)blockIdx.x * gridDim.y + blockIdx.y] = fmaxf(fmaxf(sizes[0], sizes[1]), fmaxf(sizes[2], sizes[3]));
}

// Results that are computed again, term by term in 64 bits, if need be.
// * One that is not finite: with an infinite operand, or one that rounds to infinity, the planes' products are not those of
//   the floats (infinity times a zero plane).
// * One that numbers below 2^-126 may have reached.  Taking every plane and every product of planes below that as zero
//   would change a sum of K products by less than 3 K 2^-126 (|a| + |w|) + 6 K 2^-126, with the largest |a| and |w| of the
//   workgroup's rows.  That is nothing (2^-26 of it) to a result above redo_limit.  The others, the zeros among them, are
//   computed again if the operands of the rows they come from are small enough for it: no plane of a number of 2^-103 and
//   more is below 2^-126, and products of planes that are make 2^-29 of the numbers' product where that is 2^-94 and more.
//   Results of rows of zeros, and small ones of ordinary operands, so stay as they are.
__device__ __forceinline__ float redo_limit(float most_a, float most_w, int K) {
  if (most_a == 0.f || most_w == 0.f) return -1.f;                   // (all results are zeros, or not finite)
  const float limit = (float)K * 0x1p-97f * (1.f + most_a + most_w);
  return limit == limit ? limit : INFINITY;
}

// The bits, twice, less one, of the smallest number but zero in rows row0 .. row0 + rows - 1 (below `end`) of X, columns
// k_begin .. k_end - 1; all ones if there is none.  For a whole wave.
__device__ __forceinline__ uint32_t least_key(const float* X, int row0, int rows, int end, int K, int k_begin, int k_end) {
  const int lane = threadIdx.x & 63;
  uint32_t key = 0xffffffffu;
  for (int r = row0; r < row0 + rows; r += 16)
    for (int k = k_begin + lane * 4; k < k_end; k += 256) {
      f32x4_t v[16];
#pragma unroll
      for (int i = 0; i < 16; ++i) v[i] = *reinterpret_cast<const f32x4_t*>(X + (size_t)min(r + i, end - 1) * K + k);
#pragma unroll
      for (int i = 0; i < 16; ++i)
#pragma unroll
        for (int e = 0; e < 4; ++e) key = min(key, (__float_as_uint(v[i][e]) << 1) - 1u);
    }
  for (int o = 32; o > 0; o >>= 1) key = min(key, (uint32_t)__shfl_xor((int)key, o, SA_WAVE));
  return key;
}

// The same of one row.
__device__ __forceinline__ uint32_t least_key(const float* row, int k_begin, int k_end) {
  const int lane = threadIdx.x & 63;
  uint32_t key = 0xffffffffu;
  for (int k = k_begin + lane * 4; k < k_end; k += 16 * 256) {
    f32x4_t v[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) v[i] = *reinterpret_cast<const f32x4_t*>(row + min(k + 256 * i, k_end - 4));
#pragma unroll
    for (int i = 0; i < 16; ++i)
#pragma unroll
      for (int e = 0; e < 4; ++e) key = min(key, (__float_as_uint(v[i][e]) << 1) - 1u);
  }
  for (int o = 32; o > 0; o >>= 1) key = min(key, (uint32_t)__shfl_xor((int)key, o, SA_WAVE));
  return key;
}

// Whether numbers below 2^-126 can have come up in products of operands with these keys.
__device__ __forceinline__ bool small_operands(uint32_t ka, uint32_t kw) {
  if (ka == 0xffffffffu || kw == 0xffffffffu) return false;          // (nothing but zeros)
  const float a = __uint_as_float((ka + 1u) >> 1), w = __uint_as_float((kw + 1u) >> 1);
  return a < 0x1p-103f || w < 0x1p-103f || a * w < 0x1p-94f;
}

// C[m, n], just stored by this lane, once more if it is not finite or at most `limit`.  (Inlined: a call needs a stack, which
// every launch then sets up; 24 rows, 2,048 of W at K 8192 in eight parts 18.5 -> 18.3 us.)
__device__ __forceinline__ void redo(const float* A, const float* W, float* C, int m, int n, int N, int K, int k_begin, int k_end,
                                  float limit) {
  float* cp = C + (size_t)m * N + n;
  const float size = fabsf(*cp);
  if (size > limit && size < INFINITY) return;
  double sum = 0.0;
  for (int k = k_begin; k < k_end; k += 4) {
    const f32x4_t a = *reinterpret_cast<const f32x4_t*>(A + (size_t)m * K + k);
    const f32x4_t w = *reinterpret_cast<const f32x4_t*>(W + (size_t)n * K + k);
#pragma unroll
    for (int e = 0; e < 4; ++e) sum = fma((double)a[e], (double)w[e], sum);
  }
  *cp = (float)sum;
}

// A wave's small results, a bit each in `small`, one at a time by the two rows they come from: sums of ordinary operands that
// cancel to zero, of which large products have one here and there (2,048 x 16,384 of 2,048 columns: one or two in all), and
// those of rows of zeros, which go together.  (512 x 8,192 results, K 2048, one of them zero: 134 us with the wave's rows
// searched as a whole for it, 105 so and without it.  24 rows over 16,384, K 2048, us, with W's row searched too for a row of A of
// zeros / so: none 31.7 / 31.9, one 39.7 / 35.7, twelve 82.9 / 73.3; 100 rows, fifty of zeros 169 / 158.)  True where some are
// left after SP_FEW: the wave's rows are then searched as a whole.  (With twice as many, twelve 49 and fifty 167, but where all
// numbers are small 1,900 us for 1,265 at 24 rows and 3,709 for 3,109 at 100.)  `row_of` and `col_of`
// give a bit's place, `in_row` and `in_col` this lane's bits of a row of A and of one of W.  For a whole wave.
#define SP_FEW 8
template <typename RowOf, typename ColOf, typename InRow, typename InCol>
__device__ __forceinline__ bool settle(const float* A, const float* W, float* C, unsigned long long& small, int N, int K, int k_begin,
                                       int k_end, float limit, RowOf row_of, ColOf col_of, InRow in_row, InCol in_col) {
  const int lane = threadIdx.x & 63;
  for (int turn = 0; turn < SP_FEW; ++turn) {
    const unsigned long long lanes = __ballot(small != 0);
    if (!lanes) return false;
    const int l = __builtin_ctzll(lanes);
    const int x = small ? __builtin_ctzll(small) : 0;
    const int m = __builtin_amdgcn_readlane(row_of(x), l), n = __builtin_amdgcn_readlane(col_of(x), l);
    if (lane == l) small &= small - 1;
    const uint32_t ka = least_key(A + (size_t)m * K, k_begin, k_end);
    if (ka == 0xffffffffu) {                                           // (then W's row is of no account)
      small &= ~in_row(m);
      continue;
    }
    const uint32_t kw = least_key(W + (size_t)n * K, k_begin, k_end);
    if (small_operands(ka, kw) && lane == l) redo(A, W, C, m, n, N, K, k_begin, k_end, limit);
    if (kw == 0xffffffffu) small &= ~in_col(n);
  }
  return __any(small != 0);
}

__device__ __forceinline__ uint32_t lds_offset(const void* p) {
  return (uint32_t)(uintptr_t)(__attribute__((address_space(3))) const void*)p;
}

template <int S>
struct Slot {
  static constexpr int value = S;
};

// A wave's fragments of stage slot S: a[i][plane] and w[j][plane].  One block with its wait: the compiler does not know
// that loads into LDS are stores there, and would otherwise wait for all of them before the reads.
template <int TI, int S>
__device__ __forceinline__ void read_stage(Frag8 (&a)[TI][3], Frag8 (&w)[2][3], uint32_t a_addr, uint32_t w_addr) {
  constexpr int AP = 2 * 64 * TI * 16, WP = 2 * SP_WPITCH * 16;             // bytes from plane to plane
  constexpr int A0 = S * 3 * AP, W0 = (S & 1) * 3 * WP;
  if constexpr (TI == 2) {
    asm volatile(
        "ds_read_b128 %0, %12 offset:%14\n\tds_read_b128 %1, %12 offset:%15\n\t"
        "ds_read_b128 %6, %13 offset:%20\n\tds_read_b128 %9, %13 offset:%23\n\t"
        "ds_read_b128 %2, %12 offset:%16\n\tds_read_b128 %3, %12 offset:%17\n\t"
        "ds_read_b128 %7, %13 offset:%21\n\tds_read_b128 %10, %13 offset:%24\n\t"
        "ds_read_b128 %4, %12 offset:%18\n\tds_read_b128 %5, %12 offset:%19\n\t"
        "ds_read_b128 %8, %13 offset:%22\n\tds_read_b128 %11, %13 offset:%25\n\t"
        "s_waitcnt lgkmcnt(0)"
        : "=&v"(a[0][0].u), "=&v"(a[1][0].u), "=&v"(a[0][1].u), "=&v"(a[1][1].u), "=&v"(a[0][2].u), "=&v"(a[1][2].u),
          "=&v"(w[0][0].u), "=&v"(w[0][1].u), "=&v"(w[0][2].u), "=&v"(w[1][0].u), "=&v"(w[1][1].u), "=&v"(w[1][2].u)
        : "v"(a_addr), "v"(w_addr), "n"(A0), "n"(A0 + 512), "n"(A0 + AP), "n"(A0 + AP + 512), "n"(A0 + 2 * AP),
          "n"(A0 + 2 * AP + 512), "n"(W0), "n"(W0 + WP), "n"(W0 + 2 * WP), "n"(W0 + 512), "n"(W0 + WP + 512),
          "n"(W0 + 2 * WP + 512)
        : "memory");
  } else {
    asm volatile(
        "ds_read_b128 %0, %9 offset:%11\n\tds_read_b128 %3, %10 offset:%14\n\tds_read_b128 %6, %10 offset:%17\n\t"
        "ds_read_b128 %1, %9 offset:%12\n\tds_read_b128 %4, %10 offset:%15\n\tds_read_b128 %7, %10 offset:%18\n\t"
        "ds_read_b128 %2, %9 offset:%13\n\tds_read_b128 %5, %10 offset:%16\n\tds_read_b128 %8, %10 offset:%19\n\t"
        "s_waitcnt lgkmcnt(0)"
        : "=&v"(a[0][0].u), "=&v"(a[0][1].u), "=&v"(a[0][2].u), "=&v"(w[0][0].u), "=&v"(w[0][1].u), "=&v"(w[0][2].u),
          "=&v"(w[1][0].u), "=&v"(w[1][1].u), "=&v"(w[1][2].u)
        : "v"(a_addr), "v"(w_addr), "n"(A0), "n"(A0 + AP), "n"(A0 + 2 * AP), "n"(W0), "n"(W0 + WP), "n"(W0 + 2 * WP),
          "n"(W0 + 512), "n"(W0 + WP + 512), "n"(W0 + 2 * WP + 512)
        : "memory");
  }
}

// A workgroup of four waves owns 64 TI rows of A and 128 rows of W, a wave 32 TI x 64 of them as TI x 2 tiles of
// v_mfma_f32_32x32x16_bf16 (lane l: row l % 32, columns 8 (l / 32) .. + 7 of a stage of 16; result register e is
// C[8 (e / 4) + 4 (l / 32) + e % 4][l % 32]).  A stage of both operands lies in LDS as planes, [plane][half][row], a
// row's eight numbers in 16 bytes, so that the 32 lanes of a fragment read touch consecutive units; two buffers, one
// barrier a stage.  W is split on its way from registers into LDS: its two stages of a 128-byte line are fetched
// together, one stage ahead.  gridDim.z parts of K, each with sums [M, N] of its own.
//
// What bounds it: the matrix cores (24 instructions of 32 cycles a wave and stage, beside 12 16-byte LDS reads and a split
// of eight floats).  Measured, the float32 matrix instruction on 128 x 128 tiles / this kernel with split_rows_kernel, in
// us: 1,050 rows, K 2048, 3,072 rows of W 192 / 110, 16,384 rows 736 / 418; K 8192, 2,048 rows of W 719 / 229 (five parts);
// 2,048 rows, K 2048, 16,384 rows of W 1106 / 712 (193 TFLOP/s).  Distance to 64 bits (rms, of the result's size): normal
// operands, K 2048 4.1e-7 / 2.5e-7, K 8192 4.1e-7 / 2.7e-7, K 14336 4.2e-7 / 3.4e-7; operands in 1 .. 2, 1.7e-7 / 0.8e-7,
// 1.05e-7 / 0.92e-7 and 0.95e-7 / 0.90e-7; all operands the same number (60 pairs of them), K 2048 4.1e-6 / 0.5e-6.
template <int TI>
__global__ __launch_bounds__(256, 2) void gemm_f32_split_kernel(const u32x4_t* __restrict__ P, const float* __restrict__ most,
                                                                const float* __restrict__ A, const float* __restrict__ W,
                                                                float* __restrict__ C, int M, int Mp, int N, int K,
                                                                int mtiles, size_t part_stride) {
  constexpr int BM = 64 * TI;
  constexpr int NA = (6 * BM + 255) / 256;         // kilobytes of A's planes a wave fetches a stage
  __shared__ u32x4_t As[4 * 6 * BM], Ws[2 * 6 * SP_WPITCH];
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave >> 1, wn = wave & 1;
  const int r32 = lane & 31, h = lane >> 5;

  // neighbouring workgroups run on different dies: a die takes a run of tiles, row tiles of one tile of W first, so that
  // the tile of W is read once into its L2
  const int nblk = gridDim.x;
  const int die = blockIdx.x & 7, place = blockIdx.x >> 3;
  const int t = die * (nblk >> 3) + min(die, nblk & 7) + place;
  const int m0 = (t % mtiles) * BM;
  const int n0 = (t / mtiles) * SP_BN;

  const int quads = (K + 63) >> 6;
  const int s_begin = 4 * (int)((long long)blockIdx.z * quads / gridDim.z);
  const int s_end = 4 * (int)((long long)(blockIdx.z + 1) * quads / gridDim.z);
  C += blockIdx.z * part_stride;

  // the largest sizes among this workgroup's rows of A and (this thread's share, as they come by) of W
  float most_a = 0.f, most_w = 0.f;
  for (int i = tid, nq = (s_end - s_begin) >> 2; i < BM / 32 * nq; i += 256)
    most_a = fmaxf(most_a, most[(size_t)(m0 / 32 + i / nq) * quads + (s_begin >> 2) + i % nq]);

  f32x4_t rw0[2][2], rw1[2][2];
  const float* wrow = W + (size_t)min(n0 + (tid >> 1), N - 1) * K;
  const int wk = (tid & 1) * 8;
  // A's planes of a stage straight into LDS, a kilobyte an instruction (of 64 rows: two waves fetch one a second time)
  auto fetch_a = [&](int s, u32x4_t* as) __attribute__((always_inline)) {
    const u32x4_t* p = P + (size_t)min(s, s_end - 1) * 6 * Mp + m0 + lane;
#pragma unroll
    for (int i = 0; i < NA; ++i) {
      const int u = min(wave + 4 * i, 6 * BM / 64 - 1) * 64;
      __builtin_amdgcn_global_load_lds((gptr_t)(p + (size_t)(u / BM) * Mp + (u % BM)),
                                       (__attribute__((address_space(3))) void*)(as + u), 16, 0, 0);
    }
  };
  // (beyond K the planes of A are zeros; W is read from its row's last columns there)
  auto fetch_w = [&](int s, f32x4_t (&rw)[2][2]) __attribute__((always_inline)) {       // stages s and s + 1, s even
    const int k0 = min(s, s_end - 2) * 16 + wk;
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int q = 0; q < 2; ++q) rw[j][q] = *reinterpret_cast<const f32x4_t*>(wrow + min(k0 + 16 * j + 4 * q, K - 4));
  };
  auto stash_w = [&](u32x4_t* ws, f32x4_t (&rw)[2]) __attribute__((always_inline)) {
    u32x4_t q[3];
    split8(rw[0], rw[1], q);
    max8(most_w, rw[0], rw[1]);
#pragma unroll
    for (int i = 0; i < 3; ++i) ws[(i * 2 + (tid & 1)) * SP_WPITCH + (tid >> 1)] = q[i];
  };

  floatx16_t acc[TI][2], total[TI][2];
#pragma unroll
  for (int i = 0; i < TI; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][j][e] = total[i][j][e] = 0.f;

  // Stage s, in slot s % 4 of A's ring and buffer s % 2 of W's; meanwhile stage s + 3 of A is on its way into the slot
  // that the stage before has left, stage s + 1 of W (`next`) is split into the other buffer, and from an even stage the
  // pair of stages s + 4 of W is fetched into `pair`.  The order that the scheduler is asked for: the loads, then the
  // products with the split between them, in the shadow of the matrix instructions.
  const uint32_t a_addr = lds_offset(As) + (h * BM + wm * 32 * TI + r32) * 16;
  const uint32_t w_addr = lds_offset(Ws) + (h * SP_WPITCH + wn * 64 + r32) * 16;
  auto stage = [&](int s, auto slot, f32x4_t (&next)[2], f32x4_t (*pair)[2][2]) __attribute__((always_inline)) {
    constexpr int S = decltype(slot)::value;
    Frag8 a[TI][3], w[2][3];
    read_stage<TI, S>(a, w, a_addr, w_addr);
    stash_w(Ws + ((S + 1) & 1) * 6 * SP_WPITCH, next);
    fetch_a(s + 3, As + ((S + 3) & 3) * 6 * BM);
    if (pair) fetch_w(s + 4, *pair);
    // (the small products first)
    constexpr int PA[6] = {2, 1, 0, 1, 0, 0}, PW[6] = {0, 1, 2, 0, 1, 0};
#pragma unroll
    for (int q = 0; q < 6; ++q)
#pragma unroll
      for (int i = 0; i < TI; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[i][PA[q]].v, w[j][PW[q]].v, acc[i][j], 0, 0, 0);
    SGB(SGB_MFMA, 4 * TI);
#pragma unroll
    for (int q = 0; q < 7 * TI; ++q) {
      SGB(SGB_MFMA, 1);
      SGB(SGB_VALU, 8 / TI);
    }
    SGB(SGB_DS_WRITE, 3);
    SGB(SGB_VMEM_READ, (S & 1) ? NA : NA + 4);
    SGB(SGB_MFMA, TI);
    // this wave's loads of stage s + 1 of A have landed: behind them come those of two stages and four of W
    SP_STAGE_END(2 * NA + 4);
  };

  if (s_begin < s_end) {
    fetch_w(s_begin, rw0);
    fetch_w(s_begin + 2, rw1);
    fetch_a(s_begin, As);
    fetch_a(s_begin + 1, As + 6 * BM);
    fetch_a(s_begin + 2, As + 12 * BM);
    stash_w(Ws, rw0[0]);
    SP_STAGE_END(2 * NA);
    const int flush = flush_after(s_end - s_begin);
    for (int s = s_begin; s < s_end;) {
      const int stop = min(s + flush, s_end);
      for (; s < stop; s += 4) {
        stage(s, Slot<0>(), rw0[1], &rw0);
        stage(s + 1, Slot<1>(), rw1[0], nullptr);
        stage(s + 2, Slot<2>(), rw1[1], &rw1);
        stage(s + 3, Slot<3>(), rw0[0], nullptr);
      }
#pragma unroll
      for (int i = 0; i < TI; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) {
          total[i][j] += acc[i][j];
#pragma unroll
          for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.f;
        }
    }
    SP_STAGE_END(0);                  // (loads into LDS beyond the last stage)
  }

  float* sizes = reinterpret_cast<float*>(As);
  most_a = wave_max(most_a);
  most_w = wave_max(most_w);
  if (lane == 0) {
    sizes[wave] = most_a;
    sizes[4 + wave] = most_w;
  }
  __syncthreads();
  const float limit = redo_limit(fmaxf(fmaxf(sizes[0], sizes[1]), fmaxf(sizes[2], sizes[3])),
                                 fmaxf(fmaxf(sizes[4], sizes[5]), fmaxf(sizes[6], sizes[7])), K);
  unsigned long long small = 0;          // which results of this lane are
  bool odd = false;
#pragma unroll
  for (int i = 0; i < TI; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const int n = n0 + wn * 64 + j * 32 + r32;
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        const int m = m0 + wm * 32 * TI + i * 32 + 8 * (e >> 2) + 4 * h + (e & 3);
        const float v = total[i][j][e];
        if (m < M && n < N) {
          C[(size_t)m * N + n] = v;
          small |= fabsf(v) <= limit ? 1ull << (i * 32 + j * 16 + e) : 0ull;
          odd |= !(fabsf(v) < INFINITY);
        }
      }
    }
  if (!__any(small != 0) && !__any(odd)) return;
  const int k_begin = s_begin * 16, k_end = min(K, s_end * 16);
  const int mw = m0 + wm * 32 * TI, nw = n0 + wn * 64;
  auto row_of = [&](int x) { return mw + (x >> 5) * 32 + 8 * ((x & 15) >> 2) + 4 * h + (x & 3); };
  auto col_of = [&](int x) { return nw + ((x >> 4) & 1) * 32 + r32; };
  auto in_row = [&](int m) {
    const int q = (m - mw) & 31;
    return ((q >> 2) & 1) == h ? 0x10001ull << (((m - mw) & 32) + (q >> 3) * 4 + (q & 3)) : 0ull;
  };
  auto in_col = [&](int n) { return ((n - nw) & 31) == r32 ? 0x0000ffff0000ffffull << (((n - nw) & 32) >> 1) : 0ull; };
  const bool left = settle(A, W, C, small, N, K, k_begin, k_end, limit, row_of, col_of, in_row, in_col);
  const float below = left && small_operands(least_key(A, mw, 32 * TI, M, K, k_begin, k_end),
                                             least_key(W, nw, 64, N, K, k_begin, k_end)) ? limit : -1.f;
  if (!odd && !(small != 0 && below >= 0.f)) return;
  for (int x = 0; x < TI * 32; ++x) {
    const int m = row_of(x), n = col_of(x);
    if (m >= M || n >= N) continue;
    redo(A, W, C, m, n, N, K, k_begin, k_end, below);
  }
}

// ---------------------------------------------------------------------------------------------
// Up to 128 rows (decode steps of the 32-bit path): the work is reading W, once.  A workgroup of eight waves owns 32 NT
// rows of W and MT tiles of 32 rows of A (gridDim.y runs of them; which, see few_rows).  A stage is 128 / NT columns of both (a row of it is 512 / NT bytes),
// loaded straight into LDS, a kilobyte an instruction, in a ring of NB stages: no registers hold what is on its way.
// Wave = (tile of W wt, run of 16 columns kc): it reads its fragments (lane l: row l % 32, eight columns from 8 (l / 32)),
// splits them and multiplies; the sums of a tile's waves are added through LDS at the end, in order.  Segment s (16 bytes)
// of row r lies at slot s ^ (r & 15): a 16-byte LDS read serves 16 lanes a cycle, in the groups 0-3, 12-15, 20-23, 24-27
// and 4-7, 8-11, 16-19, 28-31, and rows of 256 bytes and more then touch every bank once.
// gridDim.z parts of K, each with sums [M, N] of its own.
//
// Measured, the float32 matrix instruction / this kernel in us (weights not in a cache): K 2048, 16,384 rows of W 43 / 33 at
// 24 rows of A, 65 / 41 at 64, 121 / 67 at 128; 3,072 rows of W in four parts 20 / 10, 2,048 in eight 8.7 / 8.3; K 8192, 2,048
// rows in eight parts 24 / 19; 128,256 rows 315 / 219 at 24, 489 / 332 at 64, 965 / 550 at 128.  A step at 24 rows reads
// its 134 MB at 4.1 TB/s; from 64 rows on the splits of A, which every workgroup makes again, weigh as much.  Distance to
// 64 bits (rms, of the result's size), normal operands: K 2048 2.9e-7 / 1.1e-7 at 24 rows and 1.35e-7 at 100, K 8192 3.9e-7 /
// 1.4e-7 at 64 and 100; operands in 1 .. 2: 0.97e-7 / 0.48e-7 and 0.68e-7, 0.88e-7 / 0.56e-7.
// Up to 32 rows of A a workgroup of 64 rows of W stays below half of a compute unit's LDS.  One whose waves take both tiles of W
// (a fragment of A split once for the two, 147 KB of stages) needs a compute unit for itself: 256 of them over 16,384 rows of W
// at K 2048, in decode steps, us a launch: 27.6 on one device, and 27, 34 or 38 by turns (32.2 on the average) on another, as if some had to
// wait there for others to end; this one 29.8 and one mode.
// From five rows, with K in parts: level with the kernel of few rows of csrc/gemm.hip over 3,072 and 2,048 rows of W at K 2048
// (9.3 and 8.2 us there, 9.9 and 8.1 here), 21.3 / 18.6 over 2,048 at K 8192.  Up to 128 rows, which is what a stage has room
// for: at 128 the tiles above take 20, 87 (16,384 rows of W) and 51 us where this takes 15, 64 and 37, and only over
// 128,256 rows of W 366 for 550.
// ---------------------------------------------------------------------------------------------
template <int MT, int NT>
__device__ __forceinline__ void read_rows(Frag8 (&w)[2], Frag8 (&a)[MT][2], uint32_t w0, uint32_t w1, uint32_t a0, uint32_t a1) {
  constexpr int TILE = 32 * 512 / NT;                        // bytes from tile to tile
  // (blocks with their own wait: the compiler does not know that loads into LDS are stores there)
  if constexpr (MT == 1) {
    asm volatile("ds_read_b128 %0, %4\n\tds_read_b128 %1, %5\n\tds_read_b128 %2, %6\n\tds_read_b128 %3, %7\n\t"
                 "s_waitcnt lgkmcnt(0)"
                 : "=&v"(w[0].u), "=&v"(w[1].u), "=&v"(a[0][0].u), "=&v"(a[0][1].u)
                 : "v"(w0), "v"(w1), "v"(a0), "v"(a1)
                 : "memory");
  } else {
    asm volatile("ds_read_b128 %0, %6\n\tds_read_b128 %1, %7\n\tds_read_b128 %2, %8\n\tds_read_b128 %3, %9\n\t"
                 "ds_read_b128 %4, %8 offset:%10\n\tds_read_b128 %5, %9 offset:%10\n\ts_waitcnt lgkmcnt(0)"
                 : "=&v"(w[0].u), "=&v"(w[1].u), "=&v"(a[0][0].u), "=&v"(a[0][1].u), "=&v"(a[1][0].u), "=&v"(a[1][1].u)
                 : "v"(w0), "v"(w1), "v"(a0), "v"(a1), "n"(TILE)
                 : "memory");
    if constexpr (MT == 3)
      asm volatile("ds_read_b128 %0, %2 offset:%4\n\tds_read_b128 %1, %3 offset:%4\n\ts_waitcnt lgkmcnt(0)"
                   : "=&v"(a[2][0].u), "=&v"(a[2][1].u)
                   : "v"(a0), "v"(a1), "n"(2 * TILE)
                   : "memory");
    if constexpr (MT == 4)
      asm volatile("ds_read_b128 %0, %4 offset:%6\n\tds_read_b128 %1, %5 offset:%6\n\t"
                   "ds_read_b128 %2, %4 offset:%7\n\tds_read_b128 %3, %5 offset:%7\n\ts_waitcnt lgkmcnt(0)"
                   : "=&v"(a[2][0].u), "=&v"(a[2][1].u), "=&v"(a[3][0].u), "=&v"(a[3][1].u)
                   : "v"(a0), "v"(a1), "n"(2 * TILE), "n"(3 * TILE)
                   : "memory");
  }
}

template <int MT, int NT, int NB>
__global__ __launch_bounds__(512) void gemm_f32_wide_kernel(const float* __restrict__ A, const float* __restrict__ W,
                                                           float* __restrict__ C, int M, int N, int K, size_t part_stride) {
  constexpr int COLS = 128 / NT;                             // of a stage
  constexpr int ROWB = COLS * 4, SEGS = ROWB / 16;           // bytes and 16-byte segments of a row
  constexpr int ROWS = 32 * (NT + MT);                       // W's, then A's
  constexpr int STAGE = ROWS * ROWB;
  constexpr int RPI = 64 / SEGS;                             // rows an instruction loads
  constexpr int ND = ROWS / RPI / 8;                         // instructions a wave and stage
  static_assert(ROWS % (RPI * 8) == 0, "every wave issues the same number of loads");
  constexpr int KH = 8 / NT;                                 // waves a tile of W
  extern __shared__ __attribute__((aligned(16))) unsigned char ring[];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wt = wave % NT, kc = wave / NT;
  const int r = lane & 31, h = lane >> 5;
  const int n0 = blockIdx.x * 32 * NT, m0 = blockIdx.y * 32 * MT;
  const int all = (K + COLS - 1) / COLS;
  const int s_begin = (int)((long long)blockIdx.z * all / gridDim.z);
  const int n = (int)((long long)(blockIdx.z + 1) * all / gridDim.z) - s_begin;
  C += blockIdx.z * part_stride;

  // what this wave loads of a stage: instruction (wave ND + d), its RPI rows; a lane's row and slot, and so its segment
  const float* src[ND];
  int col[ND];
#pragma unroll
  for (int d = 0; d < ND; ++d) {
    const int row = (wave * ND + d) * RPI + lane / SEGS;
    const int seg = (lane % SEGS) ^ (row & 15);
    src[d] = row < 32 * NT ? W + (size_t)min(n0 + row, N - 1) * K : A + (size_t)min(m0 + row - 32 * NT, M - 1) * K;
    col[d] = seg * 4;
  }
  // Workgroups begin at different stages: neighbours on a die one apart, dies an eighth of the walk.  Where depends on a workgroup's
  // rows of W and on the tiles and parts that the launch has chosen (so on the number of rows of A as far as these do), not on its
  // rows of A.  Rows lie a power of two apart, so that the same columns of many rows are in one channel of a die's L2 and a few
  // of the memory: 24 rows, four steps of the 1B shape 7.80 ms where all begin at the first column, 7.38 so, and 8.35 where a
  // die's workgroups begin eight stages apart (as with the number of the workgroup modulo the stages).  One product, 24 rows, us:
  // 16,384 x 2,048 33.9 -> 32.8, 28,672 x 4,096 107.7 -> 100.1, 128,256 x 2,048 217 -> 201; from 33 rows on within 2 %.
  const int ahead = n > 0 ? (int)(((blockIdx.x >> 3) + (blockIdx.x & 7) * (n >= 8 ? n >> 3 : 1)) % (unsigned)n) : 0;
  auto stage_of = [&](int s) __attribute__((always_inline)) {
    const int t = min(s, n - 1) + ahead;
    return s_begin + (t >= n ? t - n : t);
  };
  auto fetch = [&](int s) __attribute__((always_inline)) {    // (past the last stage it is loaded again, and not read)
    const int k0 = stage_of(s) * COLS;
    unsigned char* at = ring + (s % NB) * STAGE + wave * ND * 1024;
#pragma unroll
    for (int d = 0; d < ND; ++d)
      __builtin_amdgcn_global_load_lds((gptr_t)(src[d] + min(k0 + col[d], K - 4)),
                                       (__attribute__((address_space(3))) void*)(at + d * 1024), 16, 0, 0);
  };
  const int seg0 = kc * 4 + h * 2;
  const uint32_t base = lds_offset(ring);
  const uint32_t w0 = base + (wt * 32 + r) * ROWB + ((seg0 ^ (r & 15)) << 4);
  const uint32_t w1 = base + (wt * 32 + r) * ROWB + (((seg0 + 1) ^ (r & 15)) << 4);
  const uint32_t a0 = base + (32 * NT + r) * ROWB + ((seg0 ^ (r & 15)) << 4);
  const uint32_t a1 = base + (32 * NT + r) * ROWB + (((seg0 + 1) ^ (r & 15)) << 4);

  float most_a = 0.f, most_w = 0.f;                          // the largest sizes of what this wave reads
  // the large products x0 w0 and the small ones in sums of their own: a rounding of the large sum an instruction, not six
  // (the large ones in two levels; with four tiles of A there are no registers for it, and the launch keeps K short)
  constexpr int TOTALS = MT <= 3 ? MT : 0;
  floatx16_t acc[MT], low[MT], total[TOTALS ? TOTALS : 1];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
#pragma unroll
    for (int e = 0; e < 16; ++e) acc[mt][e] = low[mt][e] = 0.f;
#pragma unroll
  for (int mt = 0; mt < TOTALS; ++mt)
#pragma unroll
    for (int e = 0; e < 16; ++e) total[mt][e] = 0.f;

  if (n > 0) {
#pragma unroll
    for (int i = 0; i < NB - 1; ++i) fetch(i);
    for (int s = 0; s < n;) {
      const int stop = min(s + SP_ROWS_FLUSH, n);
      for (; s < stop; ++s) {
        // stage s has landed: behind it come those of NB - 2 stages; everybody has read the one before, whose place is free
        SP_STAGE_END(ND * (NB - 2));
        fetch(s + NB - 1);
        const uint32_t off = (uint32_t)((s % NB) * STAGE);
        Frag8 wf[2], af[MT][2];
        read_rows<MT, NT>(wf, af, w0 + off, w1 + off, a0 + off, a1 + off);
        const int at = stage_of(s), k = at * COLS + kc * 16 + h * 8;
        if ((at + 1) * COLS > K) {                             // the last columns: beyond K the operand of A is zero
          const u32x4_t zero4 = {0u, 0u, 0u, 0u};
#pragma unroll
          for (int mt = 0; mt < MT; ++mt) {
            if (k >= K) af[mt][0].u = zero4;
            if (k + 4 >= K) af[mt][1].u = zero4;
          }
        }
        constexpr int PA[5] = {2, 1, 0, 1, 0}, PW[5] = {0, 1, 2, 0, 1};
        u32x4_t q[3];
        Frag8 w[3], a[MT][3];
        split8(wf[0].f, wf[1].f, q);
        max8(most_w, wf[0].f, wf[1].f);
#pragma unroll
        for (int p = 0; p < 3; ++p) w[p].u = q[p];
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) {
          split8(af[mt][0].f, af[mt][1].f, q);
          max8(most_a, af[mt][0].f, af[mt][1].f);
#pragma unroll
          for (int p = 0; p < 3; ++p) a[mt][p].u = q[p];
          acc[mt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(w[0].v, a[mt][0].v, acc[mt], 0, 0, 0);
#pragma unroll
          for (int p = 0; p < 5; ++p)
            low[mt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(w[PW[p]].v, a[mt][PA[p]].v, low[mt], 0, 0, 0);
        }
      }
#pragma unroll
      for (int mt = 0; mt < TOTALS; ++mt) {
        total[mt] += acc[mt];
#pragma unroll
        for (int e = 0; e < 16; ++e) acc[mt][e] = 0.f;
      }
    }
#pragma unroll
    for (int mt = 0; mt < TOTALS; ++mt) acc[mt] = total[mt];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) acc[mt] += low[mt];
    SP_STAGE_END(0);                                         // (loads beyond the last stage; everybody has read it)
  }

  __shared__ float sizes[16];
  most_a = wave_max(most_a);
  most_w = wave_max(most_w);
  if (lane == 0) {
    sizes[wave] = most_a;
    sizes[8 + wave] = most_w;
  }
  // Every wave hands over its sums, and then adds up those of eight rows of W with all of A's, 16 bytes a lane.  (With a tile
  // of W added and stored by one of its waves, number by number, the others idle, us: 24 rows, K 2048 in four parts,
  // 3,072 rows of W 11.7 / 11.1 so; 100 rows, 16,384 of W 75.5 / 70.6; 128 rows, 128,256 of W 575 / 544.)
  f32x4_t* sums = reinterpret_cast<f32x4_t*>(ring);          // [KH][NT][MT][4][64]
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
#pragma unroll
    for (int q = 0; q < 4; ++q)
      sums[((wave * MT + mt) * 4 + q) * 64 + lane] =
          (f32x4_t){acc[mt][4 * q], acc[mt][4 * q + 1], acc[mt][4 * q + 2], acc[mt][4 * q + 3]};
  __syncthreads();
  if (wave >= 4 * NT) return;
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    most_a = fmaxf(most_a, sizes[i]);
    most_w = fmaxf(most_w, sizes[8 + i]);
  }
  const float limit = redo_limit(most_a, most_w, K);
  const int nw = n0 + wave * 8;                              // (lane l: rows 4 (l / 32) .. + 3 of these)
  bool any_small = false, odd = false;
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) {
    const int m = m0 + mt * 32 + r;
    f32x4_t v = sums[((wave >> 2) * MT + mt) * 256 + (wave & 3) * 64 + lane];
#pragma unroll
    for (int o = 1; o < KH; ++o) v += sums[((o * NT + (wave >> 2)) * MT + mt) * 256 + (wave & 3) * 64 + lane];
    const int cn = nw + h * 4;
    if (m >= M) continue;
    float* cp = C + (size_t)m * N + cn;
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      any_small |= cn + c < N && fabsf(v[c]) <= limit;
      odd |= cn + c < N && !(fabsf(v[c]) < INFINITY);
    }
    if (cn + 3 < N && (((uintptr_t)cp) & 15) == 0) {
      *reinterpret_cast<f32x4_t*>(cp) = v;
    } else {
#pragma unroll
      for (int c = 0; c < 4; ++c)
        if (cn + c < N) cp[c] = v[c];
    }
  }
  if (!__any(any_small) && !__any(odd)) return;
  const int k_begin = s_begin * COLS, k_end = min(K, (s_begin + n) * COLS);
  auto row_of = [&](int x) { return m0 + (x >> 2) * 32 + r; };
  auto col_of = [&](int x) { return nw + h * 4 + (x & 3); };
  auto in_row = [&](int m) { return ((m - m0) & 31) == r ? 0xfull << ((m - m0) >> 5) * 4 : 0ull; };
  auto in_col = [&](int n) { return ((n - nw) >> 2) == h ? 0x1111ull << ((n - nw) & 3) : 0ull; };
  unsigned long long small = 0;                              // which of them, from what this lane has just stored
#pragma unroll 16
  for (int x = 0; x < MT * 4; ++x) {
    const int m = row_of(x), cn = col_of(x);
    const float v = C[(size_t)min(m, M - 1) * N + min(cn, N - 1)];
    small |= m < M && cn < N && fabsf(v) <= limit ? 1ull << x : 0ull;
  }
  const bool left = settle(A, W, C, small, N, K, k_begin, k_end, limit, row_of, col_of, in_row, in_col);
  const float below = left && small_operands(least_key(A, m0, 32 * MT, M, K, k_begin, k_end),
                                             least_key(W, nw, 8, min(nw + 8, N), K, k_begin, k_end)) ? limit : -1.f;
  if (!odd && !(small != 0 && below >= 0.f)) return;
  for (int x = 0; x < MT * 4; ++x) {
    const int m = row_of(x), cn = col_of(x);
    if (m < M && cn < N) redo(A, W, C, m, cn, N, K, k_begin, k_end, below);
  }
}

template <int MT, int NT, int NB>
static int launch_f32_wide(const void* A, const void* W, void* C, int M, int N, int K, int parts, size_t part_stride,
                           hipStream_t stream) {
  constexpr int ring = NB * 32 * (NT + MT) * 512 / NT, sums = 8 * MT * 4096;
  constexpr int lds = ring > sums ? ring : sums;
  static_assert(MT > 1 || NT < 2 || 2 * lds < 160 * 1024, "two workgroups a compute unit");
  static bool sized[64] = {};                      // (per device: more than 64 KB of LDS has to be asked for)
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return (int)e;
  if (dev < 0 || dev >= 64 || !sized[dev]) {
    e = hipFuncSetAttribute(reinterpret_cast<const void*>(&gemm_f32_wide_kernel<MT, NT, NB>),
                            hipFuncAttributeMaxDynamicSharedMemorySize, lds);
    if (e != hipSuccess) return (int)e;
    if (dev >= 0 && dev < 64) sized[dev] = true;
  }
  hipLaunchKernelGGL((gemm_f32_wide_kernel<MT, NT, NB>), dim3((N + 32 * NT - 1) / (32 * NT), (M + 32 * MT - 1) / (32 * MT), parts), dim3(512), lds,
                     stream, (const float*)A, (const float*)W, (float*)C, M, N, K, part_stride);
  SA_LAUNCH_CHECK();
  return 0;
}

// Up to 128 rows.  What a workgroup takes: 32 rows of A and 32 of W where that is one round of the chip at most, 32 and 64
// over slices of up to 1,024 columns, 64 and 32, and only then all rows of A, so that W is read once.  One round costs
// by what a workgroup does alone, so the smallest ones that still are one round win: K 2048, 100 rows, all rows of A a
// workgroup / so, us: 512 rows of W 55.7 / 14.9, 3,072 57 / 22, 512 in eight parts 14.4 / 7.4, 8,192 57 / 37.5 (64 and 64); 64 rows
// over 512 21.4 / 14.8; K 256, 100 rows, 2,048 of W 14.1 / 6.3.  Beyond one round W counts: 16,384 rows of it, 128 of A, 64 with
// all and 78 with 64 a workgroup, in 8,192 in two parts 37 and 43.
static int few_rows(const void* A, const void* W, void* C, int M, int N, int K, int parts, size_t part_stride, hipStream_t stream) {
  const long long cus = compute_units();
  const long long w32 = (long long)((N + 31) / 32) * parts, w64 = (long long)((N + 63) / 64) * parts;
  const int a32 = (M + 31) / 32, a64 = (M + 63) / 64;
  if (w32 * a32 <= cus) return launch_f32_wide<1, 1, 3>(A, W, C, M, N, K, parts, part_stride, stream);
  if (w64 * a32 <= cus && K / parts <= 1024) return launch_f32_wide<1, 2, 3>(A, W, C, M, N, K, parts, part_stride, stream);
  if (w32 * a64 <= cus) return launch_f32_wide<2, 1, 3>(A, W, C, M, N, K, parts, part_stride, stream);
  if (M <= 32) return launch_f32_wide<1, 2, 3>(A, W, C, M, N, K, parts, part_stride, stream);
  // (four tiles of A have no registers for sums in two levels: not over a long inner size)
  if (M <= 64 || w64 * a64 <= cus || (M > 96 && K / parts > 4096))
    return launch_f32_wide<2, 2, 3>(A, W, C, M, N, K, parts, part_stride, stream);
  if (M <= 96) return launch_f32_wide<3, 2, 2>(A, W, C, M, N, K, parts, part_stride, stream);
  return launch_f32_wide<4, 2, 2>(A, W, C, M, N, K, parts, part_stride, stream);
}

// The product of up to 128 rows with K cut into `parts` (1 to 8) over the grid: C fp32 [parts, M, N] takes the partial
// sums, which the consumer adds in order.  Needs K % 4 == 0 and 16-byte aligned A and W.
extern "C" int sa_gemm_f32_mid_parts(const void* A, const void* W, void* C, int M, int N, int K, int parts,
                                     hipStream_t stream) {
  if (M <= 0 || N <= 0) return 0;
  if (K <= 0 || (K & 3) || parts < 1 || parts > 8 || M > 128 || ((((uintptr_t)A | (uintptr_t)W) & 15) != 0))
    return SA_ERR_ARG;
  return few_rows(A, W, C, M, N, K, parts, (size_t)M * N, stream);
}

// Rows of A whose planes are held at a time: whole tiles of 128, at most a quarter of a gigabyte (what the chip's last
// cache holds; a product of more rows goes in runs of so many).  0: not even one tile of rows this long.
static int plane_rows(int M, int K) {
  const long long bytes = ((long long)K + 63) / 64 * 64 * 6;                 // of a row
  const long long run = (256LL << 20) / bytes / 128 * 128;
  const long long all = ((long long)M + 127) / 128 * 128;
  return (int)(run < all ? run : all);
}

// ... and behind them the largest sizes of their pieces of 32 rows by 64 columns.
static long long plane_bytes(int M, int K) { return ((long long)K + 63) / 64 * 64 * 6 * plane_rows(M, K); }

extern "C" long long sa_gemm_f32_split_bytes(int M, int K) {
  return M > 0 && K > 0 ? plane_bytes(M, K) + ((long long)K + 63) / 64 * (plane_rows(M, K) / 32) * 4 : 0;
}

// C fp32 [parts, M, N] (1 to 8 parts of K, which the consumer adds in order); `planes`: sa_gemm_f32_split_bytes of
// scratch memory; the last `tail` rows (0 to 128, fewer than M) go through the kernel of few rows.  Needs K % 4 == 0 and
// 16-byte aligned A, W and planes.  Rows of more than 349,504 columns all go there, 128 at a time, without scratch memory.
extern "C" int sa_gemm_f32_split(const void* A, const void* W, void* C, void* planes, int M, int N, int K, int parts, int tail,
                                 hipStream_t stream) {
  if (M <= 0 || N <= 0) return 0;
  if (K <= 0 || (K & 3) || parts < 1 || parts > 8 || ((((uintptr_t)A | (uintptr_t)W | (uintptr_t)planes) & 15) != 0) ||
      tail < 0 || tail > 128 || tail >= M)
    return SA_ERR_ARG;
  const int quads = (K + 63) / 64;
  const int run = plane_rows(M, K);
  float* most = (float*)((char*)planes + plane_bytes(M, K));
  if (run == 0) {
    for (int row0 = 0; row0 < M; row0 += 128) {
      const int rc = few_rows((const float*)A + (size_t)row0 * K, W, (float*)C + (size_t)row0 * N, M - row0 < 128 ? M - row0 : 128,
                              N, K, parts, (size_t)M * N, stream);
      if (rc != 0) return rc;
    }
    return 0;
  }
  const long long ntiles = ((long long)N + SP_BN - 1) / SP_BN;
  if ((run / 64) * ntiles > 0x7fffffffLL) return SA_ERR_ARG;
  const int tiled = M - tail;
  for (long long row0 = 0; row0 < tiled; row0 += run) {
    const int rows = (int)(tiled - row0 < run ? tiled - row0 : run);
    const int Mp = (rows + 127) / 128 * 128;
    const float* a = (const float*)A + (size_t)row0 * K;
    float* c = (float*)C + (size_t)row0 * N;
    hipLaunchKernelGGL(split_rows_kernel, dim3(Mp / 32, quads), dim3(256), 0, stream, a, (u32x4_t*)planes, most, rows, Mp, K);
    SA_LAUNCH_CHECK();
    // tiles of 128 rows, or of 64 where those would leave compute units without one
    const long long mt128 = (rows + 127) / 128, mt64 = (rows + 63) / 64;
    if (mt128 * ntiles * parts >= compute_units())
      hipLaunchKernelGGL((gemm_f32_split_kernel<2>), dim3(mt128 * ntiles, 1, parts), dim3(256), 0, stream,
                         (const u32x4_t*)planes, most, a, (const float*)W, c, rows, Mp, N, K, (int)mt128, (size_t)M * N);
    else
      hipLaunchKernelGGL((gemm_f32_split_kernel<1>), dim3(mt64 * ntiles, 1, parts), dim3(256), 0, stream,
                         (const u32x4_t*)planes, most, a, (const float*)W, c, rows, Mp, N, K, (int)mt64, (size_t)M * N);
    SA_LAUNCH_CHECK();
  }
  if (tail == 0) return 0;
  return few_rows((const float*)A + (size_t)tiled * K, W, (float*)C + (size_t)tiled * N, tail, N, K, parts, (size_t)M * N, stream);
}
