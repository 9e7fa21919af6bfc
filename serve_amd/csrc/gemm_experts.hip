// The two products of routed experts from 65 (token, k) rows on (steps of decoding requests and prompt portions alike), bf16
// with float32 sums, over tiles of one expert's rows from lists that csrc/moe.hip has built on the device.
//
// What bounds them: reading the experts' matrices once (32 experts of 2,048 x 1,024: 403 MB).  So an expert's rows are one
// tile up to 256 of them (beyond that, tiles of equal size), and a workgroup takes 256 weight rows: with 32 experts that is
// one round of the chip for either product, and a row of activations is fetched by 8 workgroups.  Which these are: a die
// takes a run of (tile, weight rows), so the workgroups that read the same activations share an L2, which then holds one
// expert's at a time.
//
// Measured, 1,000 tokens, 4 of 32 experts of 2,048 x 1,024, us: gate/up 88 -> 64 and down 67 -> 41 against tiles of 128 rows
// by 128 weight rows in the order of the grid (an expert with 130 rows read its matrices twice, and every die all of the
// activations).  Of the two, 72 us are the weights' stream (5.6 TB/s; without loads 41 us, without loads and products 23).
#include "common.h"

#include <type_traits>

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float floatx4_t __attribute__((ext_vector_type(4)));
typedef unsigned int u32x4_t __attribute__((ext_vector_type(4)));

union Frag {
  u32x4_t r;
  bf16x8_t v;
};

typedef __attribute__((address_space(3))) u32x4_t* lds_ptr_t;
typedef const __attribute__((address_space(1))) void* gptr_t;

// all but the newest n of this wave's loads have landed
#define SA_WAIT_VMCNT(n) __builtin_amdgcn_s_waitcnt(((n) & 0xf) | (((n) >> 4) << 14) | (0x7 << 4) | (0xf << 8))

#define EX_LDS (160 * 1024)        // of a workgroup, which has a compute unit to itself

// FIRST: act[r] = gate(Wg_e x, Wu_e x) with x = A[perm[r] / top], W [2, E, N, K] (gates, then ups, `up_offset` rows apart).
// else:  C[perm[r]] = W_e A[r], W [E, N, K].  r: grouped rows of this tile.
// SHARED (a template argument): every row in its place; perm, top, the tiles' lists and in_wts are not read.
struct ExpertArgs {
  const bf16_t* A;
  const bf16_t* W;
  void* C;
  int N, K, up_offset, gx, E, top, gate_kind;
  float gate_limit;
  const int* perm;
  const int* tile_expert;
  const int* tile_row0;     // of every tile, and behind the last the number of grouped rows
  const int* num_tiles;
  const float* in_wts;      // FIRST: fp32 [token * top + k], multiplies gate and up sums before the gate (null: not)
};

// Eight waves: two groups of 16 RT rows times four groups of 16 CT weight rows (FIRST: half of a group's are gates, the other
// half their ups, so that a pair meets in a lane).  A stage is 64 columns of both operands, loaded straight into LDS, a
// kilobyte (8 rows of 128 bytes) an instruction; segment s of row r lies at slot s ^ ((r >> 1) & 7), so that the lanes a
// 16-byte LDS read serves together touch every bank once.  Weights come from memory and activations mostly from the die's L2,
// which needs fewer stages ahead: two rings, the weights' filled by waves 0 to 3 and the activations' by waves 4 to 7, since a
// wave's loads land in order and would otherwise wait for each other.
template <int CT, int RT, bool FIRST, bool SHARED = false>
__device__ __forceinline__ void expert_tile(const ExpertArgs& p, u32x4_t* lds, int e, int row0, int M, int col0,
                                            int first) {
  constexpr int BM = 32 * RT, BN = 64 * CT;
  constexpr int COLS = FIRST ? BN / 2 : BN;
  constexpr int A_BYTES = BM * 128, W_BYTES = BN * 128;
  // stages of the rings: of the weights as many as there is room for beside two of the activations
  constexpr int NW = CT == 2 ? 6 : 4 * W_BYTES + 2 * A_BYTES <= EX_LDS ? 4 : 3;
  constexpr int ROOM = (EX_LDS - NW * W_BYTES) / A_BYTES;
  constexpr int NA = ROOM > 4 ? 4 : ROOM;
  static_assert(NA >= 2 && NW >= 3 && NW * W_BYTES + NA * A_BYTES <= EX_LDS, "the LDS of a compute unit");
  constexpr int WI = 2 * CT;                       // instructions a stage and wave: 64 CT weight rows over four waves
  constexpr int NI = WI > RT ? WI : RT;            // (of the activations: 32 RT rows over four waves)
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  const int g = lane >> 4, c = lane & 15;
  const int rg = wave >> 2, cg = wave & 3;
  const int K = p.K, N = p.N;
  const bool loads_w = wave < 4;
  const int lw = wave & 3;

  const bf16_t* src[NI];
  if (loads_w) {
    const bf16_t* W = p.W + (size_t)e * N * K;
#pragma unroll
    for (int d = 0; d < WI; ++d) {
      const int row = (lw * WI + d) * 8 + (lane >> 3);
      const int seg = (lane & 7) ^ ((row >> 1) & 7);
      int n;
      if (FIRST) {
        const int in = row % (16 * CT);
        n = min(col0 + (row / (16 * CT)) * 8 * CT + in % (8 * CT), N - 1) + (in >= 8 * CT ? p.up_offset : 0);
      } else {
        n = min(col0 + row, N - 1);
      }
      src[d] = W + (size_t)n * K + seg * 8;
    }
  } else {
#pragma unroll
    for (int d = 0; d < RT; ++d) {
      const int row = (lw * RT + d) * 8 + (lane >> 3);
      const int seg = (lane & 7) ^ ((row >> 1) & 7);
      const int r = row0 + min(row, M - 1);
      src[d] = p.A + (size_t)(FIRST && !SHARED ? p.perm[r] / p.top : r) * K + seg * 8;
    }
  }
  const lds_ptr_t as = (lds_ptr_t)lds, ws = as + NA * (A_BYTES / 16);
  const uint32_t lds_base = (uint32_t)(uintptr_t)as;
  const uint32_t a_addr = lds_base + (uint32_t)((rg * RT * 16 + c) * 128);
  const uint32_t w_addr = lds_base + NA * A_BYTES + (uint32_t)((cg * CT * 16 + c) * 128);
  const uint32_t slot0 = (uint32_t)((g ^ ((c >> 1) & 7)) * 16), slot1 = (uint32_t)(((4 + g) ^ ((c >> 1) & 7)) * 16);

  const int nstages = K >> 6;
  const int rot = first % nstages;
  auto column = [&](int s) __attribute__((always_inline)) {
    int t = min(s, nstages - 1) + rot;             // past the last stage: the last again (nobody reads it)
    if (t >= nstages) t -= nstages;
    return t * 64;
  };
  auto fetch_w = [&](int s) __attribute__((always_inline)) {
    const int k0 = column(s);
#pragma unroll
    for (int d = 0; d < WI; ++d)
      __builtin_amdgcn_global_load_lds((gptr_t)(src[d] + k0), (__attribute__((address_space(3))) void*)
                                       (ws + (s % NW) * (W_BYTES / 16) + (lw * WI + d) * 64), 16, 0, 0);
  };
  auto fetch_a = [&](int s) __attribute__((always_inline)) {
    const int k0 = column(s);
#pragma unroll
    for (int d = 0; d < RT; ++d)
      __builtin_amdgcn_global_load_lds((gptr_t)(src[d] + k0), (__attribute__((address_space(3))) void*)
                                       (as + (s % NA) * (A_BYTES / 16) + (lw * RT + d) * 64), 16, 0, 0);
  };

  floatx4_t acc[RT][CT];
#pragma unroll
  for (int mt = 0; mt < RT; ++mt)
#pragma unroll
    for (int nt = 0; nt < CT; ++nt) acc[mt][nt] = (floatx4_t){0.f, 0.f, 0.f, 0.f};

  if (loads_w) {
#pragma unroll
    for (int i = 0; i < NW - 1; ++i) fetch_w(i);
  } else {
#pragma unroll
    for (int i = 0; i < NA - 1; ++i) fetch_a(i);
  }
  for (int s = 0; s < nstages; ++s) {
    if (loads_w) SA_WAIT_VMCNT(WI * (NW - 2));     // this wave's part of stage s lies in LDS
    else SA_WAIT_VMCNT(RT * (NA - 2));
    __builtin_amdgcn_s_barrier();                  // everybody's does, and everybody has read the stage before
    if (loads_w) fetch_w(s + NW - 1);
    else fetch_a(s + NA - 1);
    const uint32_t ao = a_addr + (uint32_t)((s % NA) * A_BYTES), wo = w_addr + (uint32_t)((s % NW) * W_BYTES);
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      // (the reads are written as instructions of their own: the compiler does not see the loads into LDS as stores, and
      // would otherwise wait for all of them before every read)
      Frag af[RT], wf[CT];
#pragma unroll
      for (int nt = 0; nt < CT; ++nt)
        asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(wf[nt].r) : "v"(wo + (h ? slot1 : slot0)), "n"(nt * 16 * 128));
#pragma unroll
      for (int mt = 0; mt < RT; ++mt)
        asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(af[mt].r) : "v"(ao + (h ? slot1 : slot0)), "n"(mt * 16 * 128));
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#pragma unroll
      for (int nt = 0; nt < CT; ++nt) asm volatile("" : "+v"(wf[nt].r));
#pragma unroll
      for (int mt = 0; mt < RT; ++mt) asm volatile("" : "+v"(af[mt].r));
#pragma unroll
      for (int mt = 0; mt < RT; ++mt)
#pragma unroll
        for (int nt = 0; nt < CT; ++nt)
          acc[mt][nt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[nt].v, af[mt].v, acc[mt][nt], 0, 0, 0);
    }
  }
  SA_WAIT_VMCNT(0);                                // (loads into LDS beyond the last stage)

  // lane l holds C[m = row tile's row l % 16][n = 4 (l / 16) .. + 3] of every tile pair
  // (the kind of gate is chosen once: a branch at every number is another 4 of 181 us with the whole feed-forward of 1,000 tokens)
  auto store = [&](auto kind) __attribute__((always_inline)) {
#pragma unroll
    for (int mt = 0; mt < RT; ++mt) {
      const int m = (rg * RT + mt) * 16 + c;
      if (m >= M) continue;
      const int r = row0 + m;
      const int at = SHARED ? r : FIRST && !p.in_wts ? 0 : p.perm[r];
      const float in_w = FIRST && !SHARED && p.in_wts ? p.in_wts[at] : 1.f;   // (a weight on the input: gate and up are linear in it)
#pragma unroll
      for (int nt = 0; nt < (FIRST ? CT / 2 : CT); ++nt) {
        const int n = col0 + cg * (COLS / 4) + nt * 16 + 4 * g;
        float o[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          if constexpr (FIRST) {
            const float gt = acc[mt][nt][i] * in_w, up = acc[mt][nt + CT / 2][i] * in_w;
            o[i] = gate_mul_for_bf16<decltype(kind)::value>(gt, up, p.gate_limit);
          } else {
            o[i] = acc[mt][nt][i];
          }
        }
        if (n < N) {                                 // (N is a multiple of 64)
          if constexpr (FIRST) {
            uint2 q;
            q.x = floats_to_bf16_bits(o[0], o[1]);
            q.y = floats_to_bf16_bits(o[2], o[3]);
            *reinterpret_cast<uint2*>(reinterpret_cast<bf16_t*>(p.C) + (size_t)r * N + n) = q;
          } else {
            *reinterpret_cast<float4*>(reinterpret_cast<float*>(p.C) + (size_t)at * N + n) = make_float4(o[0], o[1], o[2], o[3]);
          }
        }
      }
    }
  };
  if (!FIRST || p.gate_kind == SA_GATE_SILU) store(std::integral_constant<int, SA_GATE_SILU>{});
  else if (p.gate_kind == SA_GATE_GELU_TANH) store(std::integral_constant<int, SA_GATE_GELU_TANH>{});
  else store(std::integral_constant<int, SA_GATE_CLAMPED_SWISH>{});
}

// The shared expert's part of a product, in the same launch: of all M rows, tiles of `rows` by 128 weight rows (SHARED_CT), which
// fill what the experts leave of the chip, and save two launches and a pass of the gate where they leave nothing.  Up to SHARED_AHEAD rows they stand before the experts' workgroups in the grid, whose
// stream of weights then begins beside them; of more rows each takes so long that they come behind.  The whole feed-forward, us, the
// shared expert as two products of its own / ahead / behind: 32 experts of 2,048 x 1,024 and a shared one of 2,048 at 129, 256, 400,
// 512, 700, 1,000 and 2,048 tokens 127 / 116 / 132, 142 / 125 / 137, 139 / 125 / 140, 156 / 151 / 153, 168 / 159 / 159, 177 / 170 / 166,
// 259 / 263 / 258; 8 of them and a shared one of 1,024 at 40, 128, 256 and 1,000 53 / 42 / 42, 64 / 52 / 51, 87 / 55 / 54, 122 / 95 / 95.  (Its
// rows in bf16 then; in fp32, as its own products leave them up to 128 rows, up to 1 us more, 2 at the last.)
// What bounds them is the way into a compute unit (a tile reads 1 MB); tiles of 256 weight rows, or of 256 rows, leave half of the chip
// idle: 198 and 228 us at 1,000 tokens.
struct SharedArgs {
  ExpertArgs p;             // (A null: none)
  int M, rows, tiles;       // tiles of rows
  int grid;                 // workgroups (a multiple of 8)
};
#define SHARED_CT 2
#define SHARED_AHEAD 640

template <bool FIRST>
__device__ __forceinline__ void shared_expert_tile(const SharedArgs& s, u32x4_t* lds, int block) {
  const int work = s.tiles * s.p.gx;
  const int die = block & 7, place = block >> 3;           // a die takes a run of weight rows, for all rows each
  const int share = work >> 3, more = work & 7;
  if (place >= share + (die < more ? 1 : 0)) return;
  const int t = die * share + min(die, more) + place;
  const int col = t / s.tiles, row0 = (t - col * s.tiles) * s.rows;
  const int M = min(s.rows, s.M - row0);
  const int eighth = max(1, s.p.K >> 9);
  const int first = col / 8 + eighth * (col % 8);          // (where to begin depends on the weight rows alone, as below)
  const int col0 = col * (FIRST ? 32 : 64) * SHARED_CT;
  if (M <= 32) expert_tile<SHARED_CT, 1, FIRST, true>(s.p, lds, 0, row0, M, col0, first);
  else if (M <= 64) expert_tile<SHARED_CT, 2, FIRST, true>(s.p, lds, 0, row0, M, col0, first);
  else expert_tile<SHARED_CT, 4, FIRST, true>(s.p, lds, 0, row0, M, col0, first);
}

template <int CT, bool FIRST>
__global__ __launch_bounds__(512, 2) void expert_product_kernel(ExpertArgs p, SharedArgs s) {
  extern __shared__ __attribute__((aligned(16))) u32x4_t expert_lds[];
  int block = blockIdx.x;
  if (s.p.A) {
    const int begin = s.M <= SHARED_AHEAD ? 0 : (int)gridDim.x - s.grid;
    if (block >= begin && block < begin + s.grid) {
      shared_expert_tile<FIRST>(s, expert_lds, block - begin);
      return;
    }
    if (begin == 0) block -= s.grid;
  }
  // neighbouring workgroups run on different dies: a die takes a run of the work, the weight rows of one tile together
  const int tiles = *p.num_tiles;
  const int work = tiles * p.gx;
  const int die = block & 7, place = block >> 3;
  const int share = work >> 3, more = work & 7;
  if (place >= share + (die < more ? 1 : 0)) return;       // (the grid is the worst case)
  const int t = die * share + min(die, more) + place;
  const int tile = t / p.gx;
  const int col0 = (t - tile * p.gx) * (FIRST ? 32 * CT : 64 * CT);
  const int e = p.tile_expert[tile], row0 = p.tile_row0[tile];
  const int M = p.tile_row0[tile + 1] - row0;              // the next tile, or the end, follows at once
  // Workgroups begin at different columns, also from die to die: rows of W lie a power of two apart, and the same columns of
  // many rows are in a few channels of the memory (1,000 tokens, both products: 105 us so, 112 with an order that repeats from
  // die to die, 118 with one of eight places, 120 where all begin at the first column).
  const int nstages = p.K >> 6;
  // The place in a list of all experts' weight rows says where, not the one in the grid, so that a row's sums do not depend on
  // what else is in the step.
  const int u = e * p.gx + t - tile * p.gx, part = max(1, p.E * p.gx >> 3);
  const int first = u % part + (nstages >= 8 ? nstages >> 3 : 1) * (u / part);
  // The bodies: a tile's products are made for all rows of its body.  32 experts of 2,048 x 1,024 with the same number of rows each,
  // both products, us: 136 rows 110 with a body for 160 and 121 without, 160 rows 115 and 126.  Bodies for 96 and 224 rows would give
  // less (72 rows 103 -> 101, 96 rows 108 -> 105, 200 rows 143 -> 136, 224 rows 145 -> 140), a third more code: left out.
  if (M <= 32) expert_tile<CT, 1, FIRST>(p, expert_lds, e, row0, M, col0, first);
  else if (M <= 64) expert_tile<CT, 2, FIRST>(p, expert_lds, e, row0, M, col0, first);
  else if (M <= 128) expert_tile<CT, 4, FIRST>(p, expert_lds, e, row0, M, col0, first);
  else if (M <= 160) expert_tile<CT, 5, FIRST>(p, expert_lds, e, row0, M, col0, first);
  else if (M <= 192) expert_tile<CT, 6, FIRST>(p, expert_lds, e, row0, M, col0, first);
  else expert_tile<CT, 8, FIRST>(p, expert_lds, e, row0, M, col0, first);
}

// rows of a tile of the shared expert: equal shares of at most 128, in sixteens
static int shared_rows(int M) {
  const int tiles = (M + 127) / 128;
  return ((M + tiles - 1) / tiles + 15) / 16 * 16;
}

template <int CT, bool FIRST>
static int launch(ExpertArgs p, SharedArgs s, int max_tiles, hipStream_t stream) {
  p.gx = (p.N + (FIRST ? 32 : 64) * CT - 1) / ((FIRST ? 32 : 64) * CT);
  long long grid = ((long long)p.gx * max_tiles + 7) / 8 * 8;
  if (max_tiles < 1 || grid > 0x3fffffffLL) return SA_ERR_ARG;
  if (s.p.A) {
    s.p.gx = (s.p.N + (FIRST ? 32 : 64) * SHARED_CT - 1) / ((FIRST ? 32 : 64) * SHARED_CT);
    s.rows = shared_rows(s.M);
    s.tiles = (s.M + s.rows - 1) / s.rows;
    const long long more = ((long long)s.p.gx * s.tiles + 7) / 8 * 8;
    if (more > 0x3fffffffLL) return SA_ERR_ARG;
    s.grid = (int)more;
    grid += more;
  }
  auto kernel = expert_product_kernel<CT, FIRST>;
  static bool allowed[64] = {};                    // (per device: more than 64 KB of LDS has to be asked for)
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return SA_ERR_ARG;
  if (!allowed[dev]) {
    const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, EX_LDS);
    if (e != hipSuccess) return (int)e;
    allowed[dev] = true;
  }
  hipLaunchKernelGGL(kernel, dim3((unsigned)grid), dim3(512), EX_LDS, stream, p, s);
  SA_LAUNCH_CHECK();
  return 0;
}

// 256 weight rows a workgroup where that still gives most compute units one (every expert chosen), else 128: of E experts with
// `pieces` times 256 weight rows in a product
static bool wide_columns(int E, int pieces) { return (long long)E * pieces * 4 >= 3ll * compute_units(); }

// The most rows of a tile (a multiple of 16), for `rows` (token, k) rows of E experts of width F: 256, so that an expert's matrices
// are read once; 128 where there would be too few tiles for the chip.  Near 256 rows an expert some have one tile and others two, and
// with 192 all have two half as long.  That is better where the second tiles would begin another round of workgroups of 256 rows all
// the same, and worse where the last round has room for them: of the mean 230 about none, of 256 half of the experts have two.  Beyond
// two rounds it is the better one from about 262 rows on.
//
// Both products with tiles of 128 / 192 / 256 rows, us: 32 experts of 2,048 x 1,024 at 3,600 rows 171 / 110 / 109, at 6,000 164 / 191 /
// 138, at 10,000 233 / 194 / 193; 8 of them at 1,400 rows 49 / 69 / 69.  With 192 / 256 at 235, 250, 275 and 295 rows an expert: 16 of
// 2,048 x 1,024 (workgroups of the first product: a round) 101 / 147, 102 / 129, 108 / 131, 115 / 118; 32 of them (a round) 175 / 232, 173 /
// 226, 174 / 210, 187 / 188; 24 (0.75 of a round) 159 / 126, 160 / 187, 162 / 193, 162 / 163; 48 (1.5) 260 / 253, 261 / 310, 267 / 297, 267 /
// 267; 16 of 3,072 x 1,536 (0.75) 236 / 168, 235 / 173, 229 / 236, 230 / 229; 128 of 2,048 x 768 (3) 545 / 519, 554 / 567, 553 / 578, 573 /
// 580; 64 of 4,096 x 1,536 (3) at 250 936 / 887.
extern "C" int sa_expert_tile_rows(int rows, int E, int F) {
  const long long tiles = (rows + 255ll) / 256 > E ? (rows + 255ll) / 256 : E;
  const int cus = compute_units();
  if (tiles * ((F + 63) / 64) * 4 < 3ll * cus) return 128;
  if (rows <= 230ll * E || rows >= 300ll * E) return 256;
  const long long gx = wide_columns(E, (F + 127) / 128) ? (F + 127) / 128 : (F + 63) / 64;
  const long long rounds = (E * gx + cus - 1) / cus, room = (rounds * cus - E * gx) / gx;
  if (rounds > 2) return rows >= 262ll * E ? 192 : 256;
  return room * 56 < rows - 228ll * E ? 192 : 256;
}

// Lists from sa_moe_group with tiles of sa_expert_tile_rows(...) rows at most (max_tiles: the grid's worst case, rows /
// tile rows + E).  bf16; d and F multiples of 64 (whole stages of K).
//   gate/up: h [T, d] gathered by perm / top, Wgu [2, E, F, d] -> act [rows, F] = gate(gate, up)
//            (in_wts, fp32 [T top] or null: both sums times the row's weight first, for weights on the experts' inputs)
//   down:    act [rows, F], Wd [E, d, F] -> yk [T top, d] fp32 at row perm[r]
// Sgu not null: in the same two launches a shared expert for all T rows, its gates and ups Sgu [2 S, d], Sd [d, S], the same kind of
// gate with its own limit: s_act [T, S] bf16, s_out [T, d] fp32 (S a multiple of 64).
extern "C" int sa_expert_products(const void* h, const void* Wgu, const void* Wd, void* act, float* yk, int E, int d, int F,
                                  int max_tiles, const int* perm, const int* tile_expert, const int* tile_row0,
                                  const int* num_tiles, int top, int gate_kind, float gate_limit, const float* in_wts,
                                  const void* Sgu, const void* Sd, void* s_act, void* s_out, int T, int S, float s_limit,
                                  hipStream_t stream) {
  if (E <= 0 || d <= 0 || F <= 0 || (d & 63) || (F & 63) || top <= 0) return SA_ERR_ARG;
  if (gate_kind < 0 || gate_kind >= SA_GATE_KINDS || (long long)E * F > 0x7fffffffLL) return SA_ERR_ARG;
  ExpertArgs p = {(const bf16_t*)h, (const bf16_t*)Wgu, act, F, d, E * F, 0, E, top, gate_kind, gate_limit,
                  perm, tile_expert, tile_row0, num_tiles, in_wts};
  SharedArgs s = {};
  if (Sgu) {
    if (!Sd || !s_act || !s_out || T <= 0 || S <= 0 || (S & 63)) return SA_ERR_ARG;
    s.p = p;
    s.p.W = (const bf16_t*)Sgu;
    s.p.C = s_act;
    s.p.N = s.p.up_offset = S;
    s.p.gate_limit = s_limit;
    s.M = T;
  }
  const int rc = wide_columns(E, (F + 127) / 128) ? launch<4, true>(p, s, max_tiles, stream) : launch<2, true>(p, s, max_tiles, stream);
  if (rc != 0) return rc;
  p.A = (const bf16_t*)act;
  p.W = (const bf16_t*)Wd;
  p.C = yk;
  p.N = d;
  p.K = F;
  p.in_wts = nullptr;
  if (Sgu) {
    s.p.A = (const bf16_t*)s_act;
    s.p.W = (const bf16_t*)Sd;
    s.p.C = s_out;
    s.p.N = d;
    s.p.K = S;
  }
  return wide_columns(E, (d + 255) / 256) ? launch<4, false>(p, s, max_tiles, stream) : launch<2, false>(p, s, max_tiles, stream);
}
