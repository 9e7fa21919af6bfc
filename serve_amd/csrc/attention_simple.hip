// Paged attention in fp32 arithmetic: one wave per (token, query head) (below), and for prompt
// portions of the float32 path a kernel that shares keys and values across 64 rows (further down).
//
// The first is the general form: any head_dim up to 640, any head counts, any page size, any mix of
// prompt portions and single tokens in one launch.  Formulas as in serve/kernels/attn_prefill.py:56-72,205 and attn_decode.py:99-111,236:
// scores = q.k * scale, key j visible to the query at absolute position p iff j <= p (and
// p - j < window when a window is set; j / chunk == p / chunk when a chunk is: at most one of the two),
// online softmax (m, l, O), O / l at the end.  Query head
// h reads KV head h / (Hq / Hk).  With `sinks` (fp32 [Hq], or null) the softmax of head h has one more
// term exp(sinks[h]) in its denominator (sinks[h] as it is stored: `scale` does not apply to it), which takes
// weight away from the keys and adds nothing to the output: it joins l
// when a row is finished (once per row: in the merge where the key range was cut).
//
// Batch layout: the T tokens of a step are the concatenation of B segments; segment r covers
// tokens cu_q[r] .. cu_q[r+1]-1, which are the last q_len positions of a context of ctx_len[r]
// tokens.  block_table[r, i] is the page of keys i*page_size .. (i+1)*page_size-1.
// k pages [page, Hk, page_size, D]; v pages [page, Hk, D, page_size].
#include "common.h"

#define SA_MAX_D 640

template <typename TA, typename TC>
__global__ __launch_bounds__(64) void paged_attention_simple_kernel(
    const TA* __restrict__ q, int q_stride, TA* __restrict__ out, const TC* __restrict__ k_pages,
    const TC* __restrict__ v_pages, const int* __restrict__ block_table, int max_pages,
    const int* __restrict__ cu_q, const int* __restrict__ ctx_len, const int* __restrict__ seg_of_token,
    int Hq, int Hk, int D, int page_size, float scale, int window, int chunk, int t0, const float* __restrict__ sinks) {
  __shared__ float qs[SA_MAX_D];
  __shared__ float ps[SA_WAVE];
  __shared__ int vbase_page[SA_WAVE];
  __shared__ int vbase_off[SA_WAVE];

  const int t = t0 + blockIdx.y;
  const int h = blockIdx.x;
  const int lane = threadIdx.x;
  const int r = seg_of_token[t];
  const int q_len = cu_q[r + 1] - cu_q[r];
  const int qpos = ctx_len[r] - q_len + (t - cu_q[r]);
  const int g = h / (Hq / Hk);
  const int* bt = block_table + (size_t)r * max_pages;

  const TA* qrow = q + (size_t)t * q_stride + (size_t)h * D;
  for (int i = lane; i < D; i += SA_WAVE) qs[i] = to_float(qrow[i]);
  __syncthreads();

  const int lo = first_seen_key(qpos, window, chunk);
  const int hi = qpos;  // inclusive

  float m = -INFINITY, l = 0.f;
  float acc[SA_MAX_D / SA_WAVE];
#pragma unroll
  for (int a = 0; a < SA_MAX_D / SA_WAVE; ++a) acc[a] = 0.f;

  for (int base = lo; base <= hi; base += SA_WAVE) {
    const int kpos = base + lane;
    const bool valid = kpos <= hi;
    float s = -INFINITY;
    int page = 0, off = 0;
    if (valid) {
      page = bt[kpos / page_size];
      off = kpos % page_size;
      const TC* kp = k_pages + (((size_t)page * Hk + g) * page_size + off) * D;
      float dot = 0.f;
      for (int i = 0; i < D; ++i) dot = fmaf(qs[i], to_float(kp[i]), dot);
      s = dot * scale;
    }
    const float m_new = fmaxf(m, wave_max(s));   // lane 0 is always valid, so m_new is finite
    const float p = valid ? expf(s - m_new) : 0.f;
    const float alpha = expf(m - m_new);         // exp(-inf) = 0 on the first chunk
    l = l * alpha + wave_sum(p);
    m = m_new;
#pragma unroll
    for (int a = 0; a < SA_MAX_D / SA_WAVE; ++a) acc[a] *= alpha;
    ps[lane] = p;
    vbase_page[lane] = page;
    vbase_off[lane] = off;
    __syncthreads();
    const int n = min(SA_WAVE, hi - base + 1);
    for (int j = 0; j < n; ++j) {
      const float pj = ps[j];
      const TC* vp = v_pages + ((size_t)vbase_page[j] * Hk + g) * (size_t)D * page_size + vbase_off[j];
#pragma unroll
      for (int a = 0; a < SA_MAX_D / SA_WAVE; ++a) {
        const int i = lane + a * SA_WAVE;
        if (i < D) acc[a] = fmaf(pj, to_float(vp[(size_t)i * page_size]), acc[a]);
      }
    }
    __syncthreads();
  }
  if (sinks) l += expf(sinks[h] - m);
  const float inv_l = 1.f / l;
  TA* orow = out + (size_t)t * Hq * D + (size_t)h * D;
#pragma unroll
  for (int a = 0; a < SA_MAX_D / SA_WAVE; ++a) {
    const int i = lane + a * SA_WAVE;
    if (i < D) orow[i] = from_float<TA>(acc[a] * inv_l);
  }
}

// ---------------------------------------------------------------------------------------------
// The same attention for prompt portions of the float32 path, tiled, on the matrix cores' float32 instruction
// (v_mfma_f32_16x16x4_f32, fp32 in and out): a workgroup of four waves takes 64 rows (a row = a token of the segment and
// one of the G query heads of a KV head, so the rows of a workgroup share every key and value), a wave 16 of them, and
// walks over the keys in blocks of 64 that are staged in LDS.  S^T = K Q^T: lane (g, c) = (l / 16, l % 16) holds row c's
// scores with keys 16 t + 4 g .. + 3, so row maxima and sums cross two shuffles, and P stays where the second product
// O^T += V^T P^T wants it: instruction e of key tile t contracts keys 16 t + 4 g + e.  The queries stay in registers;
// keys lie in LDS as rows of dims, values as rows of keys (as a page stores them), both read 16 bytes a lane.  A block's
// keys and values are on their way into registers while the block before is used, its page ids one block earlier.
// Needs D % 16 == 0, D <= 128 and a page size that is a multiple of 4 (four consecutive keys then lie in one page).
// Bound by that instruction (128 of 32 cycles a wave and block at heads of 64) beside the exponentials.  The same tile on the
// vector ALU, four by four values a thread, with every operand read from LDS for each of them, / this kernel, 32 heads on
// 8, us: heads of 64, eight ragged prompts up to 256 tokens 67 / 36, one of 512 87 / 34, of 1,500 345 / 149, four portions of
// 333 over 600 keys 288 / 124; heads of 128 205 / 67, 168 / 53, 986 / 259, 875 / 225.  The distance to 64 bits is the same
// (one prompt of 1,500 tokens, rms of the result: 3.6e-7 and 4.2e-7).
// ---------------------------------------------------------------------------------------------
#define TL_ROWS 64
#define TL_KEYS 64
typedef float tl_f4 __attribute__((ext_vector_type(4)));

template <int DV>   // D / 16
__global__ __launch_bounds__(256, 2) void paged_attention_tiled_f32_kernel(
    const float* __restrict__ q, int q_stride, float* __restrict__ out, const float* __restrict__ k_pages,
    const float* __restrict__ v_pages, const int* __restrict__ block_table, int max_pages,
    const int* __restrict__ cu_q, const int* __restrict__ ctx_len, int Hq, int Hk, int page_size, float scale,
    int window, int chunk, int num_splits, float* __restrict__ part_o, float* __restrict__ part_ml,
    const float* __restrict__ sinks) {
  constexpr int D = DV * 16;
  constexpr int LK = D + 4, LV = TL_KEYS + 4;     // row lengths in LDS: 16-byte aligned, spread over the banks
  extern __shared__ __attribute__((aligned(16))) float tl_smem[];
  float* Ks = tl_smem;                            // [64][LK]
  float* Vs = Ks + TL_KEYS * LK;                  // [D][LV]

  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6, g4 = lane >> 4, c = lane & 15;
  const int hk = blockIdx.x % Hk;                 // KV head
  const int item = blockIdx.x / Hk;               // tile of 64 rows within the segment
  const int seg = blockIdx.y / num_splits;
  const int sp = blockIdx.y - seg * num_splits;   // this workgroup's part of the key range
  const int G = Hq / Hk;
  const int q_begin = cu_q[seg];
  const int q_len = cu_q[seg + 1] - q_begin;
  const int rows_total = q_len * G;
  const int r0 = item * TL_ROWS;
  if (r0 >= rows_total) return;
  const int ctx = ctx_len[seg];
  const int ctx_before = ctx - q_len;
  const int* bt = block_table + (size_t)seg * max_pages;

  // this lane's row and its quarter of the query (dims 16 s + 4 g4 .. + 3); a row beyond the segment's is its last once
  // more and is not written
  const int row = r0 + w * 16 + c;
  const bool rvalid = row < rows_total;
  const int j = min(row, rows_total - 1) / G, gi = min(row, rows_total - 1) - j * G;
  const int qpos = ctx_before + j, qlo = first_seen_key(qpos, window, chunk);
  tl_f4 qf[DV];
  {
    const float* qp = q + (size_t)(q_begin + j) * q_stride + (size_t)(hk * G + gi) * D + 4 * g4;
#pragma unroll
    for (int s = 0; s < DV; ++s) qf[s] = *reinterpret_cast<const tl_f4*>(qp + 16 * s);
  }
  const int last_row = min(r0 + TL_ROWS - 1, rows_total - 1);
  const int hi = ctx_before + last_row / G;                                       // last key any row of the tile sees
  const int lo = first_seen_key(ctx_before + r0 / G, window, chunk);              // first key any row sees
  // keys full_lo .. full_hi are visible to every row of the tile
  const int full_hi = ctx_before + r0 / G;
  const int full_lo = first_seen_key(hi, window, chunk);

  float m = -INFINITY, l = 0.f;
  tl_f4 acc[DV];
#pragma unroll
  for (int e = 0; e < DV; ++e) acc[e] = (tl_f4){0.f, 0.f, 0.f, 0.f};

  // the blocks of 64 keys that the tile sees, cut evenly into num_splits parts
  const int b_lo = lo / TL_KEYS, b_hi = hi / TL_KEYS;
  const int per = (b_hi - b_lo + num_splits) / num_splits;
  const int b_first = b_lo + sp * per;
  const int b_last = min(b_hi, b_first + per - 1);

  // Lane l looks up key kb + l; a key outside the tile's range stands for the nearest one of it (the pages before a
  // window may have been given back)
  auto look_up = [&](int kb, int& page, int& place) __attribute__((always_inline)) {
    const int kpos = min(max(kb + lane, lo), hi);
    const int idx = kpos / page_size;
    page = bt[idx];
    place = kpos - idx * page_size;
  };
  // DV pieces of 16 bytes a thread, of the keys and of the values; the values of four consecutive keys of a dim are one
  // piece, from their own place in the page of the nearest key (which is theirs, or they are masked as a whole)
  tl_f4 rk[DV], rv[DV];
  auto fetch = [&](int kb, int page, int place) __attribute__((always_inline)) {
    const int own = (kb + (tid & 15) * 4) % page_size;
#pragma unroll
    for (int n = 0; n < DV; ++n) {
      const int i = tid + 256 * n, key = i / (D / 4), c4 = i - key * (D / 4);
      const int pg = __shfl(page, key, SA_WAVE), pl = __shfl(place, key, SA_WAVE);
      rk[n] = *reinterpret_cast<const tl_f4*>(k_pages + (((size_t)pg * Hk + hk) * page_size + pl) * D + c4 * 4);
    }
    // (keys before the range: the first of the four that lies in it names the page)
    const int quad = (tid & 15) * 4;
    const int named = min(max(kb + quad, lo), hi) - kb;
    const int pv = __shfl(page, min(max(named, quad), quad + 3) & 63, SA_WAVE);
#pragma unroll
    for (int n = 0; n < DV; ++n) {
      const int d = (tid >> 4) + 16 * n;
      rv[n] = *reinterpret_cast<const tl_f4*>(v_pages + (((size_t)pv * Hk + hk) * D + d) * page_size + own);
    }
  };
  int page, place;
  look_up(min(b_first, b_hi) * TL_KEYS, page, place);
  fetch(min(b_first, b_hi) * TL_KEYS, page, place);
  look_up(min(b_first + 1, b_hi) * TL_KEYS, page, place);
  for (int kb = b_first * TL_KEYS; kb <= b_last * TL_KEYS; kb += TL_KEYS) {
    __syncthreads();                              // the block before has been used
#pragma unroll
    for (int n = 0; n < DV; ++n) {
      const int i = tid + 256 * n, key = i / (D / 4), c4 = i - key * (D / 4);
      *reinterpret_cast<tl_f4*>(Ks + key * LK + c4 * 4) = rk[n];
    }
#pragma unroll
    for (int n = 0; n < DV; ++n) {
      // a value beyond what any row sees may be anything (a page that holds another request's data, or none): its weight
      // is 0, and 0 times it must be 0
      const int k0 = kb + (tid & 15) * 4;
      tl_f4 v = rv[n];
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = k0 + e >= lo && k0 + e <= hi ? v[e] : 0.f;
      *reinterpret_cast<tl_f4*>(Vs + ((tid >> 4) + 16 * n) * LV + (tid & 15) * 4) = v;
    }
    __syncthreads();
    const int next = min(kb / TL_KEYS + 1, b_hi) * TL_KEYS;
    fetch(next, page, place);
    look_up(min(kb / TL_KEYS + 2, b_hi) * TL_KEYS, page, place);
    tl_f4 s[4];
#pragma unroll
    for (int t = 0; t < 4; ++t) s[t] = (tl_f4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int d = 0; d < DV; ++d) {
      tl_f4 kf[4];
#pragma unroll
      for (int t = 0; t < 4; ++t) kf[t] = *reinterpret_cast<const tl_f4*>(Ks + (16 * t + c) * LK + 16 * d + 4 * g4);
#pragma unroll
      for (int x = 0; x < 4; ++x)
#pragma unroll
        for (int t = 0; t < 4; ++t) s[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(kf[t][x], qf[d][x], s[t], 0, 0, 0);
    }
#pragma unroll
    for (int t = 0; t < 4; ++t) s[t] *= scale;
    if (kb < full_lo || kb + TL_KEYS - 1 > full_hi) {
#pragma unroll
      for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int key = kb + 16 * t + 4 * g4 + e;
          s[t][e] = key <= qpos && key >= qlo ? s[t][e] : -INFINITY;
        }
    }
    float mx = -INFINITY;
#pragma unroll
    for (int t = 0; t < 4; ++t) mx = fmaxf(mx, fmaxf(fmaxf(s[t][0], s[t][1]), fmaxf(s[t][2], s[t][3])));
    mx = fmaxf(mx, __shfl_xor(mx, 16, SA_WAVE));
    mx = fmaxf(mx, __shfl_xor(mx, 32, SA_WAVE));
    const float m_new = fmaxf(m, mx);
    const float m_safe = m_new == -INFINITY ? 0.f : m_new;        // a row that has seen no key yet
    const float alpha = expf(m - m_safe);                         // exp(-inf) = 0 at the first visible block
    m = m_new;
    float sum = 0.f;
#pragma unroll
    for (int t = 0; t < 4; ++t) {
#pragma unroll
      for (int e = 0; e < 4; ++e) s[t][e] = expf(s[t][e] - m_safe);   // exp(-inf) = 0 for invisible keys
      sum += (s[t][0] + s[t][1]) + (s[t][2] + s[t][3]);
    }
    sum += __shfl_xor(sum, 16, SA_WAVE);
    sum += __shfl_xor(sum, 32, SA_WAVE);
    l = l * alpha + sum;
#pragma unroll
    for (int e = 0; e < DV; ++e) acc[e] *= alpha;
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      tl_f4 vf[DV];
#pragma unroll
      for (int e = 0; e < DV; ++e) vf[e] = *reinterpret_cast<const tl_f4*>(Vs + (16 * e + c) * LV + 16 * t + 4 * g4);
#pragma unroll
      for (int x = 0; x < 4; ++x)
#pragma unroll
        for (int e = 0; e < DV; ++e) acc[e] = __builtin_amdgcn_mfma_f32_16x16x4f32(vf[e][x], s[t][x], acc[e], 0, 0, 0);
    }
  }
  if (!rvalid) return;
  const size_t orow_index = (size_t)(q_begin + j) * Hq + (hk * G + gi);           // (token, head)
  if (num_splits > 1) {
    // unnormalised sums with their maximum and weight: merged by paged_attention_merge_f32_kernel
    float* po = part_o + (orow_index * num_splits + sp) * D + 4 * g4;
#pragma unroll
    for (int e = 0; e < DV; ++e) *reinterpret_cast<tl_f4*>(po + 16 * e) = acc[e];
    if (g4 == 0) {
      part_ml[(orow_index * num_splits + sp) * 2] = m;
      part_ml[(orow_index * num_splits + sp) * 2 + 1] = l;
    }
    return;
  }
  const float inv_l = 1.f / (sinks ? l + expf(sinks[hk * G + gi] - m) : l);
  float* orow = out + orow_index * D + 4 * g4;
#pragma unroll
  for (int e = 0; e < DV; ++e) {
    const tl_f4 v = acc[e] * inv_l;
    if (((uintptr_t)out & 15) == 0) {
      *reinterpret_cast<tl_f4*>(orow + 16 * e) = v;
    } else {
#pragma unroll
      for (int x = 0; x < 4; ++x) orow[16 * e + x] = v[x];
    }
  }
}

// out[row] = sum_s w_s O_s / sum_s w_s l_s with w_s = exp(m_s - max m): the parts of a split key
// range (a part that saw no key has m = -inf and weight 0; at most 64 parts).  One wave per row: the
// lanes first share the parts (weights), then the head dims (weighted sums, whose loads do not wait
// for one another).
__global__ __launch_bounds__(64) void paged_attention_merge_f32_kernel(const float* __restrict__ part_o,
                                                                       const float* __restrict__ part_ml,
                                                                       float* __restrict__ out, int D, int num_splits,
                                                                       const float* __restrict__ sinks, int Hq) {
  __shared__ float wgt[64];
  const size_t row = blockIdx.x;                  // (token, head)
  const int lane = threadIdx.x;
  float ms = -INFINITY, ls = 0.f;
  if (lane < num_splits) {
    ms = part_ml[(row * num_splits + lane) * 2];
    ls = part_ml[(row * num_splits + lane) * 2 + 1];
  }
  const float mx = wave_max(ms);
  const float w = ms == -INFINITY ? 0.f : expf(ms - mx);
  float total = wave_sum(w * ls);
  if (sinks) total += expf(sinks[row % Hq] - mx);
  const float inv = 1.f / total;
  wgt[lane] = w;
  __syncthreads();
  const float* po = part_o + row * num_splits * D;
  for (int d = lane; d < D; d += 64) {
    float o = 0.f;
#pragma unroll 8
    for (int s = 0; s < num_splits; ++s) o = fmaf(wgt[s], po[(size_t)s * D + d], o);
    out[row * D + d] = o * inv;
  }
}

template <int DV>
static int launch_tiled(const void* q, int q_stride, void* out, const void* k_pages, const void* v_pages,
                        const int* block_table, int max_pages, const int* cu_q, const int* ctx_len, int B,
                        int max_q_len, int Hq, int Hk, int page_size, float scale, int window, int chunk, int num_splits,
                        float* part_o, float* part_ml, const float* sinks, hipStream_t stream) {
  constexpr int D = DV * 16;
  const size_t lds = (size_t)(TL_KEYS * (D + 4) + D * (TL_KEYS + 4)) * sizeof(float);
  const long long items = ((long long)max_q_len * (Hq / Hk) + TL_ROWS - 1) / TL_ROWS;
  if (items * Hk > 0x7fffffffLL || (long long)B * num_splits > 65535) return SA_ERR_ARG;
  hipError_t e = hipFuncSetAttribute((const void*)paged_attention_tiled_f32_kernel<DV>,
                                     hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
  if (e != hipSuccess) return (int)e;
  dim3 grid((unsigned)(items * Hk), B * num_splits), block(256);
  hipLaunchKernelGGL((paged_attention_tiled_f32_kernel<DV>), grid, block, lds, stream, (const float*)q, q_stride,
                     (float*)out, (const float*)k_pages, (const float*)v_pages, block_table, max_pages, cu_q,
                     ctx_len, Hq, Hk, page_size, scale, window, chunk, num_splits, part_o, part_ml, sinks);
  SA_LAUNCH_CHECK();
  return 0;
}

// ---------------------------------------------------------------------------------------------
// Single tokens of the float32 path over long contexts: every segment brings one token, so the rows
// that share a KV head's keys and values are only its G query heads, and the tiled kernel above
// would do the arithmetic of 64 rows for them.  Here one wave takes GR query heads of one KV head
// of one segment and one part of the key range, in blocks of 64 keys:
//   scores: four lanes per key, each with a quarter of the dims (the four lanes of a key read 64
//   contiguous bytes at a time), partial sums added across the four lanes;
//   softmax: online, maxima and sums across the wave, p of the block through LDS;
//   values: a lane per dim (V is stored [D, page_size]: the lanes of a wave read whole runs of a
//   page), four keys a load, O += p v for the GR heads.
// Every key and value is read once per GR heads instead of once per head.  Parts as in the kernels
// above: part_o [T Hq num_splits, D], part_ml [T Hq num_splits, 2], merged by
// paged_attention_merge_f32_kernel.  Needs D % 16 == 0, D <= 128, page_size % 4 == 0.
// What bounds it: the chain of one block (table, keys, scores, softmax, values), of which a part has few.  So a lane looks
// up one page (the others ask it by a shuffle), all keys and values of a block are asked for before anything waits, and
// the keys outside the range are masked where the scores are.  Before (the pages looked up by every lane, keys and values
// in two trips of eight) / now, with the merge, 32 heads on 8, us: heads of 64, 24 requests at context 300 23.6 / 19.3, 64
// at 400 29.8 / 26.2, 8 at 4,096 28.6 / 25.0, one at 8,192 21.0 / 17.2; heads of 96 23.9 / 16.4, 28.3 / 20.6, 26.2 / 20.1,
// 21.5 / 17.0 (of 96 over much to read, which wants two waves a SIMD: 8 at 4,096 on 32 heads 46.7 / 35.2, 51 with registers for
// one, 64 at 513 48.1 / 36.3; of 112 49.4 / 39.5); heads of 128 33.9 / 28.4, 54.0 / 47.4, 54.7 / 48.3, 29.9 / 27.0 (64 at 2,000: 1.05 GB in 178 us, 204 before).
// ---------------------------------------------------------------------------------------------
template <int DV, int GR>   // D / 16; query heads per wave
__global__ __launch_bounds__(64, 2) void paged_attention_decode_f32_kernel(
    const float* __restrict__ q, int q_stride, float* __restrict__ out, const float* __restrict__ k_pages,
    const float* __restrict__ v_pages, const int* __restrict__ block_table, int max_pages,
    const int* __restrict__ cu_q, const int* __restrict__ ctx_len, int Hq, int Hk, int page_size, float scale,
    int window, int chunk, int num_splits, float* __restrict__ part_o, float* __restrict__ part_ml,
    const float* __restrict__ sinks) {
  constexpr int D = DV * 16;
  constexpr int NA = (D + 63) / 64;               // dims per lane in the product with V
  __shared__ __attribute__((aligned(16))) float ps[GR][64];
  const int lane = threadIdx.x;
  const int kk = lane >> 2, part = lane & 3;      // key of a group of 16, quarter of the dims
  const int G = Hq / Hk;
  const int chunks = (G + GR - 1) / GR;
  const int g = blockIdx.x / chunks;              // KV head
  const int h0 = (blockIdx.x - g * chunks) * GR;  // first of this wave's query heads within the group
  const int seg = blockIdx.y;
  const int sp = blockIdx.z;
  const int t = cu_q[seg];                        // the segment's one token
  const int qpos = ctx_len[seg] - 1;
  const int* bt = block_table + (size_t)seg * max_pages;
  const int lo = first_seen_key(qpos, window, chunk);
  const int hi = qpos;

  // this lane's quarter of the queries (a head beyond the group repeats the last and is not written)
  float4 qv[GR][DV];
#pragma unroll
  for (int r = 0; r < GR; ++r) {
    const int h = g * G + min(h0 + r, G - 1);
    const float* qp = q + (size_t)t * q_stride + (size_t)h * D;
#pragma unroll
    for (int e = 0; e < DV; ++e) {
      const float4 v = *reinterpret_cast<const float4*>(qp + (part + 4 * e) * 4);
      qv[r][e] = make_float4(v.x * scale, v.y * scale, v.z * scale, v.w * scale);
    }
  }
  float m[GR], l[GR], acc[GR][NA];
#pragma unroll
  for (int r = 0; r < GR; ++r) {
    m[r] = -INFINITY;
    l[r] = 0.f;
#pragma unroll
    for (int a = 0; a < NA; ++a) acc[r][a] = 0.f;
  }

  // the blocks of 64 keys that the token sees, cut evenly into num_splits parts
  const int b_lo = lo >> 6, b_hi = hi >> 6;
  const int per = (b_hi - b_lo + num_splits) / num_splits;
  const int b_first = b_lo + sp * per;
  const int b_last = min(b_hi, b_first + per - 1);
  // Lane l looks up the page of key kb + l, and the others ask it: one division and one trip to the block table a block.
  // A key outside the range stands for the range's nearest key (the pages before a window may have been given back).
  auto look_up = [&](int kb, int& page, int& place) __attribute__((always_inline)) {
    const int kpos = min(max(kb + lane, lo), hi);
    const int idx = kpos / page_size;
    page = bt[idx];
    place = kpos - idx * page_size;
  };
  int page, place;
  look_up(min(b_first, b_hi) * 64, page, place);
  for (int kb = b_first * 64; kb <= b_last * 64; kb += 64) {
    // all loads of the block before anything waits: the time of a short context is this chain's
    constexpr int KN = DV <= 4 ? 4 : GR == 4 && DV >= 6 ? 1 : 2;  // keys of a lane fetched at a time (wide heads: registers are short)
    float4 kv[KN][DV];
    auto fetch_k = [&](int first) __attribute__((always_inline)) {
#pragma unroll
      for (int i = 0; i < KN; ++i) {
        const int pg = __shfl(page, 16 * (first + i) + kk, SA_WAVE);
        const int pl = __shfl(place, 16 * (first + i) + kk, SA_WAVE);
        const float* kp = k_pages + (((size_t)pg * Hk + g) * page_size + pl) * D;
#pragma unroll
        for (int e = 0; e < DV; ++e) kv[i][e] = *reinterpret_cast<const float4*>(kp + (part + 4 * e) * 4);
      }
    };
    fetch_k(0);
    // values: four keys of a dim are one load (they lie in one page, at a multiple of four; keys outside the range are
    // read from the page of its nearest key, at their own place in it)
    constexpr int VN = NA == 1 ? 16 : GR == 4 && DV >= 7 ? 4 : 8;  // groups of four keys fetched at a time
    float4 vv[VN][NA];
    uint32_t voff[NA];
#pragma unroll
    for (int a = 0; a < NA; ++a) voff[a] = (uint32_t)(min(lane + 64 * a, D - 1) * page_size);
    const int own = (kb + lane) % page_size;
    auto fetch_v = [&](int first) __attribute__((always_inline)) {
#pragma unroll
      for (int j = 0; j < VN; ++j) {
        const int pg = __builtin_amdgcn_readlane(page, 4 * (first + j));
        const int pl = __builtin_amdgcn_readlane(own, 4 * (first + j));
        const float* vb = v_pages + ((size_t)pg * Hk + g) * D * page_size + pl;      // (the same for the wave)
#pragma unroll
        for (int a = 0; a < NA; ++a) vv[j][a] = *reinterpret_cast<const float4*>(vb + voff[a]);
      }
    };
    fetch_v(0);
    int next_page = page, next_place = place;
    if (kb < b_last * 64) look_up(kb + 64, next_page, next_place);
    // scores: keys kb + 16 i + kk, the same in the four lanes of a key; keys outside the range are masked
    float s[GR][4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      if (i > 0 && i % KN == 0) {
        __builtin_amdgcn_sched_barrier(0);          // (not earlier: the registers are those of the keys before)
        fetch_k(i);
      }
#pragma unroll
      for (int r = 0; r < GR; ++r) {
        float d = 0.f;
#pragma unroll
        for (int e = 0; e < DV; ++e) {
          d = fmaf(qv[r][e].x, kv[i % KN][e].x, d);
          d = fmaf(qv[r][e].y, kv[i % KN][e].y, d);
          d = fmaf(qv[r][e].z, kv[i % KN][e].z, d);
          d = fmaf(qv[r][e].w, kv[i % KN][e].w, d);
        }
        d += __shfl_xor(d, 1, SA_WAVE);
        d += __shfl_xor(d, 2, SA_WAVE);
        const int key = kb + 16 * i + kk;
        s[r][i] = key >= lo && key <= hi ? d : -INFINITY;
      }
    }
    __syncthreads();                              // the block before has been multiplied
#pragma unroll
    for (int r = 0; r < GR; ++r) {
      float mx = fmaxf(fmaxf(s[r][0], s[r][1]), fmaxf(s[r][2], s[r][3]));
#pragma unroll
      for (int o = 4; o < SA_WAVE; o <<= 1) mx = fmaxf(mx, __shfl_xor(mx, o, SA_WAVE));
      const float m_new = fmaxf(m[r], mx);
      const float m_safe = m_new == -INFINITY ? 0.f : m_new;      // a part that has seen no key yet
      const float alpha = expf(m[r] - m_safe);
      float sum = 0.f;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float pr = expf(s[r][i] - m_safe);                  // exp(-inf) = 0 for invisible keys
        if (part == 0) ps[r][16 * i + kk] = pr;
        sum += pr;
      }
#pragma unroll
      for (int o = 4; o < SA_WAVE; o <<= 1) sum += __shfl_xor(sum, o, SA_WAVE);
      l[r] = l[r] * alpha + sum;
      m[r] = m_new;
#pragma unroll
      for (int a = 0; a < NA; ++a) acc[r][a] *= alpha;
    }
    __syncthreads();
    const bool edge = kb < lo || kb + 63 > hi;
#pragma unroll 1
    for (int first = 0; first < 16; first += VN) {
      if (first > 0) fetch_v(first);
      if (edge) {
        // a value that the token does not see may be anything: its weight is 0, and 0 times it must be 0
#pragma unroll
        for (int j = 0; j < VN; ++j) {
          const int kq = kb + 4 * (first + j);
#pragma unroll
          for (int a = 0; a < NA; ++a) {
            if (kq < lo || kq > hi) vv[j][a].x = 0.f;
            if (kq + 1 < lo || kq + 1 > hi) vv[j][a].y = 0.f;
            if (kq + 2 < lo || kq + 2 > hi) vv[j][a].z = 0.f;
            if (kq + 3 < lo || kq + 3 > hi) vv[j][a].w = 0.f;
          }
        }
      }
#pragma unroll
      for (int j = 0; j < VN; ++j) {
        if (j % 4 == 0) __builtin_amdgcn_sched_barrier(0);     // (the weights of four groups of keys in registers, not of all)
        float4 pv[GR];
#pragma unroll
        for (int r = 0; r < GR; ++r) pv[r] = *reinterpret_cast<const float4*>(&ps[r][4 * (first + j)]);
#pragma unroll
        for (int a = 0; a < NA; ++a) {
#pragma unroll
          for (int r = 0; r < GR; ++r) {
            float o = acc[r][a];
            o = fmaf(pv[r].x, vv[j][a].x, o);
            o = fmaf(pv[r].y, vv[j][a].y, o);
            o = fmaf(pv[r].z, vv[j][a].z, o);
            o = fmaf(pv[r].w, vv[j][a].w, o);
            acc[r][a] = o;
          }
        }
      }
    }
    page = next_page;
    place = next_place;
  }
#pragma unroll
  for (int r = 0; r < GR; ++r) {
    if (h0 + r >= G) continue;
    const size_t row = (size_t)t * Hq + g * G + h0 + r;           // (token, head)
    if (sinks && num_splits == 1) l[r] += expf(sinks[g * G + h0 + r] - m[r]);
#pragma unroll
    for (int a = 0; a < NA; ++a) {
      const int d = lane + 64 * a;
      if (d >= D) continue;
      if (num_splits > 1) part_o[(row * num_splits + sp) * D + d] = acc[r][a];
      else out[row * D + d] = acc[r][a] / l[r];
    }
    if (num_splits > 1 && lane == 0) {
      part_ml[(row * num_splits + sp) * 2] = m[r];
      part_ml[(row * num_splits + sp) * 2 + 1] = l[r];
    }
  }
}

template <int DV>
static int launch_decode_f32(const void* q, int q_stride, void* out, const void* k_pages, const void* v_pages,
                             const int* block_table, int max_pages, const int* cu_q, const int* ctx_len, int B,
                             int Hq, int Hk, int page_size, float scale, int window, int chunk, int num_splits, float* part_o,
                             float* part_ml, const float* sinks, hipStream_t stream) {
  const int G = Hq / Hk;
  const int gr = G >= 3 ? 4 : G;                  // heads per wave: 1, 2 or 4
  const long long gx = (long long)Hk * ((G + gr - 1) / gr);
  if (gx > 0x7fffffffLL || B > 65535 || num_splits > 65535) return SA_ERR_ARG;
  dim3 grid((unsigned)gx, B, num_splits), block(64);
#define GO(GR)                                                                                                    \
  hipLaunchKernelGGL((paged_attention_decode_f32_kernel<DV, GR>), grid, block, 0, stream, (const float*)q,        \
                     q_stride, (float*)out, (const float*)k_pages, (const float*)v_pages, block_table, max_pages, \
                     cu_q, ctx_len, Hq, Hk, page_size, scale, window, chunk, num_splits, part_o, part_ml, sinks)
  if (gr == 1) GO(1);
  else if (gr == 2) GO(2);
  else GO(4);
#undef GO
  SA_LAUNCH_CHECK();
  return 0;
}

// float32 attention of B segments of one token each (token r is the last of a context of ctx_len[r]
// tokens) over their cached keys.  D a multiple of 16 up to 128, page_size a multiple of 4.
// The segments are a run of the step's tokens: segment i is token first_token + i (cu_q[i] must say
// so; the host knows it and the kernels do not check it), which is the row of q, out and the parts it
// uses.  num_splits > 1 cuts every key range into that many parts over the grid; part_o
// [(first_token + B) Hq num_splits, D] and part_ml [(first_token + B) Hq num_splits, 2] (fp32) then
// take the parts, which a second kernel merges for the rows first_token .. first_token + B - 1.
extern "C" int sa_paged_attention_decode_f32(const void* q, int q_stride, void* out, const void* k_pages,
                                             const void* v_pages, const int* block_table, int max_pages,
                                             const int* cu_q, const int* ctx_len, int B, int first_token, int Hq,
                                             int Hk, int D, int page_size, float scale, int window, int chunk,
                                             int num_splits, float* part_o, float* part_ml, const float* sinks, hipStream_t stream) {
  if (B <= 0) return 0;
  if (Hq <= 0 || Hk <= 0 || Hq % Hk || D <= 0 || D > 128 || (D & 15) || page_size <= 0 || (page_size & 3) ||
      max_pages <= 0 || (q_stride & 3) || num_splits < 1 || num_splits > 64 || first_token < 0 ||
      (window > 0 && chunk > 0))
    return SA_ERR_ARG;
  if (num_splits > 1 && (!part_o || !part_ml)) return SA_ERR_ARG;
  int rc = SA_ERR_ARG;
#define GO(DV)                                                                                                   \
  case DV:                                                                                                       \
    rc = launch_decode_f32<DV>(q, q_stride, out, k_pages, v_pages, block_table, max_pages, cu_q, ctx_len, B, Hq, \
                               Hk, page_size, scale, window, chunk, num_splits, part_o, part_ml, sinks, stream); \
    break
  switch (D / 16) {
    GO(1);
    GO(2);
    GO(3);
    GO(4);
    GO(5);
    GO(6);
    GO(7);
    GO(8);
  }
#undef GO
  if (rc != 0 || num_splits == 1) return rc;
  const size_t row0 = (size_t)first_token * Hq;
  hipLaunchKernelGGL(paged_attention_merge_f32_kernel, dim3((unsigned)B * Hq), dim3(64), 0, stream,
                     part_o + row0 * num_splits * D, part_ml + row0 * num_splits * 2, (float*)out + row0 * D, D,
                     num_splits, sinks, Hq);
  SA_LAUNCH_CHECK();
  return 0;
}

// float32 attention of every token of the B segments (T tokens) over their cached keys, 64 rows a
// workgroup.  D a multiple of 16 up to 128, page_size a multiple of 4; max_q_len: the longest
// segment.  num_splits > 1 cuts every tile's key range into that many parts over the grid; part_o
// [T Hq num_splits, D] and part_ml [T Hq num_splits, 2] (fp32) then take the parts, which a second
// kernel merges.
extern "C" int sa_paged_attention_tiled_f32(const void* q, int q_stride, void* out, const void* k_pages,
                                            const void* v_pages, const int* block_table, int max_pages,
                                            const int* cu_q, const int* ctx_len, int B, int T, int max_q_len,
                                            int Hq, int Hk, int D, int page_size, float scale, int window,
                                            int chunk, int num_splits, float* part_o, float* part_ml, const float* sinks,
                                            hipStream_t stream) {
  if (B <= 0 || max_q_len <= 0 || T <= 0) return 0;
  if (Hq <= 0 || Hk <= 0 || Hq % Hk || D <= 0 || D > 128 || (D & 15) || page_size <= 0 || (page_size & 3) ||
      max_pages <= 0 || (q_stride & 3) || num_splits < 1 || num_splits > 64 || (window > 0 && chunk > 0))
    return SA_ERR_ARG;
  if (num_splits > 1 && (!part_o || !part_ml)) return SA_ERR_ARG;
  int rc = SA_ERR_ARG;
#define GO(DV)                                                                                                  \
  case DV:                                                                                                      \
    rc = launch_tiled<DV>(q, q_stride, out, k_pages, v_pages, block_table, max_pages, cu_q, ctx_len, B,         \
                          max_q_len, Hq, Hk, page_size, scale, window, chunk, num_splits, part_o, part_ml, sinks, \
                          stream);                                                                              \
    break
  switch (D / 16) {
    GO(1);
    GO(2);
    GO(3);
    GO(4);
    GO(5);
    GO(6);
    GO(7);
    GO(8);
  }
#undef GO
  if (rc != 0 || num_splits == 1) return rc;
  hipLaunchKernelGGL(paged_attention_merge_f32_kernel, dim3((unsigned)T * Hq), dim3(64), 0, stream, part_o, part_ml,
                     (float*)out, D, num_splits, sinks, Hq);
  SA_LAUNCH_CHECK();
  return 0;
}

extern "C" int sa_paged_attention_simple(const void* q, int q_stride, void* out, int act_dtype,
                                         const void* k_pages, const void* v_pages, int cache_dtype,
                                         const int* block_table, int max_pages, const int* cu_q,
                                         const int* ctx_len, const int* seg_of_token, int T, int Hq,
                                         int Hk, int D, int page_size, float scale, int window, int chunk,
                                         const float* sinks, hipStream_t stream) {
  if (T <= 0) return 0;
  if (Hq <= 0 || Hk <= 0 || Hq % Hk || D <= 0 || D > SA_MAX_D || page_size <= 0 || max_pages <= 0 ||
      (window > 0 && chunk > 0))
    return SA_ERR_ARG;
  if (T > 65535 * 16) return SA_ERR_ARG;
  // grid.y is limited to 65535: long steps are launched in slices of tokens
  const int slice = 32768;
  for (int t0 = 0; t0 < T; t0 += slice) {
    const int n = T - t0 < slice ? T - t0 : slice;
    dim3 grid(Hq, n), block(SA_WAVE);
#define GO(TA, TC)                                                                                   \
  hipLaunchKernelGGL((paged_attention_simple_kernel<TA, TC>), grid, block, 0, stream,                \
                     (const TA*)q, q_stride, (TA*)out, (const TC*)k_pages, (const TC*)v_pages,       \
                     block_table, max_pages, cu_q, ctx_len, seg_of_token, Hq, Hk, D, page_size,     \
                     scale, window, chunk, t0, sinks)
    if (act_dtype == SA_F32 && cache_dtype == SA_F32) GO(float, float);
    else if (act_dtype == SA_BF16 && cache_dtype == SA_BF16) GO(bf16_t, bf16_t);
    else return SA_ERR_UNSUPPORTED;
#undef GO
    SA_LAUNCH_CHECK();
  }
  return 0;
}
