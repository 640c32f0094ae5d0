// Prefill / batched linear layers: y[M, N] = epilogue(x[M, K] W[N, K]^T (+ bias)).
//
// MFMA tiling for CDNA4 (wave64). A block owns a BM x BN output tile (32 x 64
// to 256 x 128) made of 64 x 64 wave tiles (2 x 2 MFMA accumulators of
// 32 x 32; 32 x 64 wave tiles for few rows; 32 x 32 and 64 x 32 ones for
// products of few stages), with WK waves sharing each wave tile's K (one for
// few stages): wave group g takes every WK-th 16-byte substep of a stage and
// the groups' sums are added in group order at the end (a fixed order). Both operands are K-contiguous in memory (x rows
// and W rows), the layout the MFMA fragments want, so nothing is transposed:
//   bf16: v_mfma_f32_32x32x16_bf16 (8 bf16 per lane and operand, k = 8*(lane/32)+i)
//   fp32: 4 x v_mfma_f32_32x32x2f32 per 16 bytes (lane half h holds k 4h .. 4h+3
//         of 8; MFMA i takes element i of both halves)
// W is the MFMA's A operand and x its B operand, so lane l, register r is
// output row l % 32 and column 8*(r/4) + 4*(l/32) + r%4: four consecutive
// columns per register quad, stored as one piece.
//
// K advances in stages of 128 bytes per row, kept in a ring of STAGES LDS
// buffers that global memory is loaded into directly (buffer_load_dwordx4 ...
// lds: no registers, no LDS write instructions); each 16-byte chunk c of row r
// sits at position c ^ (r / 2) % 8, so the lanes reading one fragment column
// spread over all banks. STAGES - 1 stages are in flight: a wave waits for its own share of
// the stage it reads next by count (vmcnt), and one barrier per stage both
// publishes that stage and frees the previous one.
//
// Few output tiles (short prompts, batched decode) split K over blocks as
// well: each split writes fp32 partial sums to a workspace, which
// gemm_reduce_kernel, or the kernel that consumes the product, adds in split
// order (fixed, so results do not depend on timing).
#include <type_traits>

#include "common.h"
#include "kernels.h"

namespace minitp {

namespace {

constexpr int OUT_PARTIAL = 100;  // epilogue: fp32 split-K partials
// epilogue: SwiGLU of a [gate; up] weight (2N rows): per 64 tile columns, 32
// gate rows then the 32 matching up rows, so a wave's two column fragments
// are a gate fragment and its up fragment
constexpr int OUT_SWIGLU = 101;

typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef __bf16 bf16x8_k __attribute__((ext_vector_type(8)));

template <typename T>
__device__ __forceinline__ f32x16 mfma_step(const u32x4& a, const u32x4& b, f32x16 c);
template <>
__device__ __forceinline__ f32x16 mfma_step<bf16>(const u32x4& a, const u32x4& b, f32x16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_k, a), __builtin_bit_cast(bf16x8_k, b), c,
                                                 0, 0, 0);
}
template <>
__device__ __forceinline__ f32x16 mfma_step<float>(const u32x4& a, const u32x4& b, f32x16 c) {
#pragma unroll
  for (int i = 0; i < 4; ++i)
    c = __builtin_amdgcn_mfma_f32_32x32x2f32(__uint_as_float(a[i]), __uint_as_float(b[i]), c, 0, 0, 0);
  return c;
}

// Lane offsets past a resource (the load writes zeros to LDS). ROW_OOB marks a
// row past the matrix, and stays past any resource that ends below it with a
// K offset added; K_OOB, never offset further, is past every resource (their
// spans are multiples of 16 bytes below 4 GiB).
constexpr uint32_t ROW_OOB = 0xF0000000u, K_OOB = 0xFFFFFFF0u;

// 16 bytes per lane from the resource at voff straight into LDS: lane l's
// bytes land at lds_addr + 16 l (wave-uniform, in m0). NT: non-temporal. asm, so that the
// compiler does not wait for these loads at every LDS read: the kernel waits
// for them itself, by count. The s_nop is the wait state that gfx9 hardware
// asks for between the scalar write of m0 and a load to LDS (the compiler
// inserts it for its own loads, but does not look into asm).
template <bool NT>
__device__ __forceinline__ void load16_lds(u32x4 r, uint32_t voff, uint32_t lds_addr) {
  if constexpr (NT)
    asm volatile("s_nop 0\n\tbuffer_load_dwordx4 %0, %1, 0 offen nt lds" ::"v"(voff), "s"(r), "{m0}"(lds_addr) : "memory");
  else
    asm volatile("s_nop 0\n\tbuffer_load_dwordx4 %0, %1, 0 offen lds" ::"v"(voff), "s"(r), "{m0}"(lds_addr) : "memory");
}

__device__ __forceinline__ u32x4 rsrc_span(const void* base, uint32_t bytes) {
  const uint64_t p = (uint64_t)base;
  u32x4 r;
  r.x = (uint32_t)__builtin_amdgcn_readfirstlane((uint32_t)p);
  r.y = (uint32_t)__builtin_amdgcn_readfirstlane((uint32_t)(p >> 32));  // stride 0
  r.z = (uint32_t)__builtin_amdgcn_readfirstlane(bytes);
  r.w = 0x00020000u;
  return r;
}

// this wave's older stage loads have landed (all but the newest N) and its
// LDS reads are done, then the block barrier
template <int N>
__device__ __forceinline__ void stage_barrier() {
  asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(N) : "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

// Tile shape of a launch: BM x BN outputs in wave tiles of FM x FN fragments
// (32 x 32), WK waves per wave tile, a ring of STAGES, non-temporal loads (NT).
// WHOLE: a product of at most STAGES stages, all loaded at once (no ring).
constexpr int KCH = 8;  // 16-byte chunks of K per row and stage
template <int BM_, int BN_, int WK_, int STAGES_, bool NT_ = false, int FM_ = (BM_ >= 64 ? 2 : 1), int FN_ = 2,
          bool WHOLE_ = false>
struct Tile {
  static constexpr bool NT = NT_, WHOLE = WHOLE_;
  static constexpr int BM = BM_, BN = BN_, WK = WK_, STAGES = STAGES_, FM = FM_, FN = FN_;
  static constexpr int WM = BM / (32 * FM), WN = BN / (32 * FN), NW = WM * WN * WK, THREADS = 64 * NW;
  static constexpr int ROWB = KCH * 16;
  static constexpr int STAGE_BYTES = (BM + BN) * ROWB;
  static constexpr int RING_BYTES = STAGES * STAGE_BYTES, XCH_BYTES = WM * WN * (WK - 1) * FM * FN * 4096;
  static constexpr int LDS_BYTES = RING_BYTES > XCH_BYTES ? RING_BYTES : XCH_BYTES;
  static constexpr int PIECE_ROWS = 64 / KCH;                   // rows of one 1 KiB load
  static constexpr int PPW = (BM + BN) / PIECE_ROWS / NW;       // loads per wave and stage
  static_assert((BM + BN) % (PIECE_ROWS * NW) == 0, "a stage splits evenly over the waves");
  static_assert((STAGES - 2) * PPW < 64, "vmcnt counts six bits");
  static_assert((KCH / 2) % WK == 0, "substeps split evenly over the wave groups");
};

// Block b: split b / (tiles), tile b % tiles in XCD-aware order. Blocks go to
// the 8 XCDs round-robin and each XCD has its own L2, so XCD b % 8 takes a
// contiguous range of (split, tile) items, row tiles fastest inside groups of
// 8: the row tiles that share a W panel run on one XCD at the same time.
template <typename T, typename C, int OUT>
__global__ __launch_bounds__(C::THREADS) void gemm_kernel(const T* __restrict__ x, int64_t ldx,
                                                          const T* __restrict__ w, const T* __restrict__ bias, T* y,
                                                          int64_t ldy, const T* aux, float* part, int M, int N, int K,
                                                          int kper, int tiles_m, int tiles_n, int items,
                                                          const StepState* state) {
  constexpr int BM = C::BM, BN = C::BN, WK = C::WK, STAGES = C::STAGES, PPW = C::PPW;
  constexpr int FM = C::FM, FN = C::FN, WN = C::WN, ROWB = C::ROWB, ES = (int)sizeof(T), V = 16 / ES, TK = KCH * V;
  static_assert(OUT != OUT_SWIGLU || FN == 2, "a wave tile holds whole gate and up fragment pairs");
  extern __shared__ __attribute__((aligned(16))) char lds[];
  if (state != nullptr) y = (T*)state->args.logits;
  const int per_xcd = (items + 7) >> 3;
  const int item = (blockIdx.x & 7) * per_xcd + (blockIdx.x >> 3);
  if ((int)(blockIdx.x >> 3) >= per_xcd || item >= items) return;
  const int tiles = tiles_m * tiles_n;
  // (straight-line divisions: branches around those whose quotient is known saved
  // one row tile 70 ns and cost the others up to 0.7 us, 433 x 3584 x 3584 26.9 -> 27.6)
  const int z = item / tiles, t = item - z * tiles;
  const int group = t / (8 * tiles_n), first_m = group * 8, gsz = min(tiles_m - first_m, 8);
  const int in_group = t - group * 8 * tiles_n;
  const int m0 = (first_m + in_group % gsz) * BM, tn = in_group / gsz;
  const int kb = z * kper, ke = min(kb + kper, K);

  const int tid = threadIdx.x, lane = tid & 63, half = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wk = wave / (C::WM * WN), wm = wave / WN % C::WM, wn = wave % WN;

  // the tile's rows of x and of W as buffers; W row r of the tile
  constexpr int BNO = OUT == OUT_SWIGLU ? BN / 2 : BN;  // output columns
  const int n0 = tn * BNO;
  auto w_row = [&](int r) -> int64_t {  // relative to n0, -1: past the matrix
    if (OUT == OUT_SWIGLU) {
      const int c = (r >> 6) * 32 + (r & 31);
      return n0 + c < N ? ((r & 32) ? (int64_t)N + c : c) : -1;
    }
    return n0 + r < N ? r : -1;
  };
  const int x_rows = min(M - m0, BM);
  const int64_t w_rows = OUT == OUT_SWIGLU ? (int64_t)2 * N - n0 : min(N - n0, BN);
  const uint32_t x_bytes = (uint32_t)(((int64_t)(x_rows - 1) * ldx + K) * ES);
  const uint32_t w_bytes = (uint32_t)(w_rows * K * ES);
  const u32x4 xq = rsrc_span(x + (int64_t)m0 * ldx, x_bytes);
  const u32x4 wq = rsrc_span(w + (int64_t)n0 * K, w_bytes);
  // rows past the matrix read zeros; where a tile spans nearly 4 GiB, its
  // last row again (their outputs are not stored either way)
  const uint32_t x_pad = x_bytes <= ROW_OOB ? ROW_OOB : (uint32_t)((int64_t)(x_rows - 1) * ldx * ES);
  const uint32_t w_pad = w_bytes <= ROW_OOB ? ROW_OOB : 0u;
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char*)lds;
  constexpr int A_BYTES = BM * ROWB;
  auto swz = [](int r) { return (r >> 1) & 7; };
  uint32_t voff[PPW];  // byte offset of the lane's chunk at k = 0
  int kc[PPW];         // its first k
#pragma unroll
  for (int j = 0; j < PPW; ++j) {
    const int p = wave * PPW + j;
    const bool is_w = p >= BM / C::PIECE_ROWS;
    const int r = C::PIECE_ROWS * (is_w ? p - BM / C::PIECE_ROWS : p) + lane / KCH;
    const int c = (lane % KCH) ^ swz(r);
    kc[j] = c * V;
    if (!is_w) {
      voff[j] = r < x_rows ? (uint32_t)(((int64_t)r * ldx + c * V) * ES) : x_pad;
    } else {
      const int64_t wr = w_row(r);
      voff[j] = wr >= 0 ? (uint32_t)((wr * K + c * V) * ES) : w_pad;
    }
  }
  const int nk = (ke - kb + TK - 1) / TK;
  // (chunks past the split's end read zeros: steps past the last load nothing,
  // so that every step issues the same number of loads and the waits can
  // count them)
  auto issue = [&](int step, int stage) {
    const int k0 = kb + step * TK;
    const uint32_t base = lds0 + stage * C::STAGE_BYTES + wave * PPW * 1024;
#pragma unroll
    for (int j = 0; j < PPW; ++j)
      load16_lds<C::NT>(wave * PPW + j >= BM / C::PIECE_ROWS ? wq : xq, k0 + kc[j] < ke ? voff[j] + (uint32_t)(k0 * ES) : K_OOB,
                 (uint32_t)__builtin_amdgcn_readfirstlane(base + j * 1024));
  };

  f32x16 acc[FM][FN];  // [x fragment][W fragment]
#pragma unroll
  for (int i = 0; i < FM; ++i)
#pragma unroll
    for (int j = 0; j < FN; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.f;

  const int ar = wm * (32 * FM) + (lane & 31), br = wn * (32 * FN) + (lane & 31);
  // (rows 32 apart share the swizzle)
  const int a_off = ar * ROWB, b_off = A_BYTES + br * ROWB, a_swz = swz(ar), b_swz = swz(br);
  constexpr int KS = KCH / 2 / WK;  // substeps of a stage per wave group
#pragma unroll 1
  for (int s = 0; s < (C::WHOLE ? nk : STAGES - 1); ++s) issue(s, s);
  if constexpr (C::WHOLE) stage_barrier<0>();
  int rd = 0, wr_stage = STAGES - 1;
  for (int kt = 0; kt < nk; ++kt) {
    if constexpr (!C::WHOLE) {
      stage_barrier<(STAGES - 2) * PPW>();
      issue(kt + STAGES - 1, wr_stage);
    }
    const char* st = lds + rd * C::STAGE_BYTES;
    u32x4 av[2][FM], bv[2][FN];
    auto fetch = [&](int s, u32x4(&a)[FM], u32x4(&b)[FN]) {
      const int c = (s * WK + wk) * 2 + half;
#pragma unroll
      for (int i = 0; i < FM; ++i) a[i] = *(const u32x4*)(st + a_off + i * 32 * ROWB + ((c ^ a_swz) << 4));
#pragma unroll
      for (int j = 0; j < FN; ++j) b[j] = *(const u32x4*)(st + b_off + j * 32 * ROWB + ((c ^ b_swz) << 4));
    };
    fetch(0, av[0], bv[0]);
#pragma unroll
    for (int s = 0; s < KS; ++s) {
      if (s + 1 < KS) fetch(s + 1, av[(s + 1) & 1], bv[(s + 1) & 1]);
#pragma unroll
      for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j) acc[i][j] = mfma_step<T>(bv[s & 1][j], av[s & 1][i], acc[i][j]);
    }
    rd = rd + 1 == STAGES ? 0 : rd + 1;
    wr_stage = wr_stage + 1 == STAGES ? 0 : wr_stage + 1;
  }

  // (the steps past the last wrote zeros into the ring: let them land before
  // this block's LDS is reused or given back)
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  // the wave groups' sums of a tile, added in group order: group g finishes
  // the register quads q with q WK / 4 == g of every fragment and hands over
  // the others
  if constexpr (WK > 1) {
    __syncthreads();  // (the ring is free: every wave's last reads and loads are done)
    u32x4* xch = (u32x4*)lds;
    const int wt = wave % (C::WM * WN);
    auto slot = [&](int f, int g, int q) { return (((wt * FM * FN + f) * (WK - 1) + g) * 4 + q) * 64 + lane; };
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int owner = q * WK / 4;
      if (owner == wk) continue;
      const int g = wk < owner ? wk : wk - 1;
#pragma unroll
      for (int f = 0; f < FM * FN; ++f) {
        const f32x16& a = acc[f / FN][f % FN];
        xch[slot(f, g, q)] = u32x4{__float_as_uint(a[4 * q]), __float_as_uint(a[4 * q + 1]),
                                   __float_as_uint(a[4 * q + 2]), __float_as_uint(a[4 * q + 3])};
      }
    }
    __syncthreads();
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      if (q * WK / 4 != wk) continue;
#pragma unroll
      for (int f = 0; f < FM * FN; ++f) {
        float v[4];
#pragma unroll
        for (int g = 0; g < WK; ++g) {
          float p[4];
          if (g == wk) {
#pragma unroll
            for (int e = 0; e < 4; ++e) p[e] = acc[f / FN][f % FN][4 * q + e];
          } else {
            const u32x4 u = xch[slot(f, g < wk ? g : g - 1, q)];
#pragma unroll
            for (int e = 0; e < 4; ++e) p[e] = __uint_as_float(u[e]);
          }
#pragma unroll
          for (int e = 0; e < 4; ++e) v[e] = g == 0 ? p[e] : v[e] + p[e];
        }
#pragma unroll
        for (int e = 0; e < 4; ++e) acc[f / FN][f % FN][4 * q + e] = v[e];
      }
    }
  }

  // outputs of lane l, fragment (i, j), register 4 q + e: row i 32 + l % 32,
  // column j 32 + 8 q + 4 (l / 32) + e. Whole quads go out as one store when
  // rows and base allow it (else element by element).
  using O = typename std::conditional<OUT == OUT_PARTIAL, float, T>::type;
  O* const out = OUT == OUT_PARTIAL ? (O*)(part + (int64_t)z * M * N) : (O*)y;
  const int64_t ldo = OUT == OUT_PARTIAL ? N : ldy;
  const bool quads = N % 4 == 0 && ldo % 4 == 0 && ((uintptr_t)out & (4 * sizeof(O) - 1)) == 0;
  auto finish = [&](int i, int j, int q, int64_t row, int col, float* v) {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const float a = acc[i][j][4 * q + e];
      if constexpr (OUT == OUT_SWIGLU)
        v[e] = swiglu<T>(round_to<T>(a + 0.f), round_to<T>(acc[i][FN - 1][4 * q + e] + 0.f));
      else if constexpr (OUT == MINITP_EPI_RESID)
        v[e] = col + e < N ? add_rn(load_f32<T>(aux, row * ldy + col + e), round_to<T>(a)) : 0.f;
      else if constexpr (OUT == MINITP_EPI_NONE)
        v[e] = a + (bias != nullptr && col + e < N ? load_f32<T>(bias, col + e) : 0.f);
      else
        v[e] = a;
    }
  };
  constexpr int FJ = OUT == OUT_SWIGLU ? 1 : FN;
  const int col0 = n0 + wn * (32 * FJ) + 4 * half;
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    if (WK > 1 && q * WK / 4 != wk) continue;
#pragma unroll
    for (int i = 0; i < FM; ++i) {
      const int64_t row = m0 + wm * (32 * FM) + i * 32 + (lane & 31);
      if (row >= M) continue;
#pragma unroll
      for (int j = 0; j < FJ; ++j) {
        const int col = col0 + j * 32 + 8 * q;
        float v[4];
        if (col >= N) continue;
        finish(i, j, q, row, col, v);
        O* o = out + row * ldo + col;
        if (quads) {
          if constexpr (sizeof(O) == 4)
            *(float4*)o = make_float4(v[0], v[1], v[2], v[3]);
          else
            *(uint2*)o = make_uint2(pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3]));
        } else {
#pragma unroll 1
          for (int e = 0; e < 4 && col + e < N; ++e) store_f32<O>(o, e, e == 0 ? v[0] : e == 1 ? v[1] : e == 2 ? v[2] : v[3]);
        }
      }
    }
  }
}

// The same products as gemm_kernel without a K split or wave groups, for one row
// tile and many column tiles of few stages: a block walks its share of tiles and the ring of stages
// runs on across them, so that a tile's epilogue and the next one's first
// loads overlap (gemm_kernel drains its ring and refills it for every tile:
// 0.5B LM head of 194 rows 107 us, 5 tiles of 14 stages a block; 97 so, bound
// by the stages' MFMAs and LDS reads at two waves a SIMD and a last round two
// thirds full). Loads past the one being waited for include the epilogue's
// stores: the counted wait is then longer than needed, never shorter, since
// vector memory operations retire in issue order. Non-temporal weight loads:
// 4 % slower.
template <typename T, typename C>
__global__ __launch_bounds__(C::THREADS) void gemm_stream_kernel(const T* __restrict__ x, int64_t ldx,
                                                                 const T* __restrict__ w, const T* __restrict__ bias,
                                                                 T* y, int64_t ldy, int M, int N, int K, int items,
                                                                 const StepState* state) {
  constexpr int BM = C::BM, BN = C::BN, STAGES = C::STAGES, PPW = C::PPW;
  constexpr int FM = C::FM, WN = C::WN, ROWB = C::ROWB, ES = (int)sizeof(T), V = 16 / ES, TK = KCH * V;
  static_assert(C::WK == 1, "a wave tile is one wave's");
  extern __shared__ __attribute__((aligned(16))) char lds[];
  if (state != nullptr) y = (T*)state->args.logits;
  // XCD b % 8 takes a contiguous range of tiles, its blocks every stride-th of it
  const int per_xcd = (items + 7) >> 3, stride = gridDim.x >> 3;
  const int first = (blockIdx.x & 7) * per_xcd, mine = min(per_xcd, items - first);
  int li = blockIdx.x >> 3;
  if (li >= mine) return;

  const int tid = threadIdx.x, lane = tid & 63, half = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave / WN % C::WM, wn = wave % WN;
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char*)lds;
  constexpr int A_BYTES = BM * ROWB;
  auto swz = [](int r) { return (r >> 1) & 7; };

  // ---- the load side: the tile whose stages are being issued -----------------
  const uint32_t x_bytes = (uint32_t)(((int64_t)(M - 1) * ldx + K) * ES);
  const uint32_t x_pad = x_bytes <= ROW_OOB ? ROW_OOB : (uint32_t)((int64_t)(M - 1) * ldx * ES);
  const u32x4 xq = rsrc_span(x, x_bytes);
  u32x4 wq;
  uint32_t voff[PPW];
  int kc[PPW];
  auto setup = [&](int t) {
    const int n0 = t * BN;
    const int64_t w_rows = min(N - n0, BN);
    const uint32_t w_bytes = (uint32_t)(w_rows * K * ES);
    wq = rsrc_span(w + (int64_t)n0 * K, w_bytes);
    const uint32_t w_pad = w_bytes <= ROW_OOB ? ROW_OOB : 0u;
#pragma unroll
    for (int j = 0; j < PPW; ++j) {
      const int p = wave * PPW + j;
      const bool is_w = p >= BM / C::PIECE_ROWS;
      const int r = C::PIECE_ROWS * (is_w ? p - BM / C::PIECE_ROWS : p) + lane / KCH;
      const int c = (lane % KCH) ^ swz(r);
      kc[j] = c * V;
      if (!is_w) {
        voff[j] = r < M ? (uint32_t)(((int64_t)r * ldx + c * V) * ES) : x_pad;
      } else {
        voff[j] = n0 + r < N ? (uint32_t)(((int64_t)r * K + c * V) * ES) : w_pad;
      }
    }
  };
  const int nk = (K + TK - 1) / TK;
  int ls = 0, lt = li;  // next stage to issue and its tile
  // (past the last tile the loads read zeros: every step issues the same
  // number, so that the waits can count them)
  auto issue = [&](int stage) {
    if (ls == nk && lt < mine) {
      lt += stride;
      ls = 0;
      if (lt < mine) setup(first + lt);
    }
    const int k0 = lt < mine ? ls * TK : K;
    const uint32_t base = lds0 + stage * C::STAGE_BYTES + wave * PPW * 1024;
#pragma unroll
    for (int j = 0; j < PPW; ++j)
      load16_lds<C::NT>(wave * PPW + j >= BM / C::PIECE_ROWS ? wq : xq, k0 + kc[j] < K ? voff[j] + (uint32_t)(k0 * ES) : K_OOB,
                 (uint32_t)__builtin_amdgcn_readfirstlane(base + j * 1024));
    ++ls;
  };

  const int ar = wm * (32 * FM) + (lane & 31), br = wn * 64 + (lane & 31);
  const int a_off = ar * ROWB, b_off = A_BYTES + br * ROWB, a_swz = swz(ar), b_swz = swz(br);
  constexpr int KS = KCH / 2;
  setup(first + lt);
#pragma unroll 1
  for (int s = 0; s < STAGES - 1; ++s) issue(s);
  int rd = 0, wr_stage = STAGES - 1;
  for (; li < mine; li += stride) {
    f32x16 acc[FM][2];
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.f;
    for (int kt = 0; kt < nk; ++kt) {
      stage_barrier<(STAGES - 2) * PPW>();
      issue(wr_stage);
      const char* st = lds + rd * C::STAGE_BYTES;
      u32x4 av[2][FM], bv[2][2];
      auto fetch = [&](int s, u32x4(&a)[FM], u32x4(&b)[2]) {
        const int c = s * 2 + half;
#pragma unroll
        for (int i = 0; i < FM; ++i) a[i] = *(const u32x4*)(st + a_off + i * 32 * ROWB + ((c ^ a_swz) << 4));
#pragma unroll
        for (int j = 0; j < 2; ++j) b[j] = *(const u32x4*)(st + b_off + j * 32 * ROWB + ((c ^ b_swz) << 4));
      };
      fetch(0, av[0], bv[0]);
#pragma unroll
      for (int s = 0; s < KS; ++s) {
        if (s + 1 < KS) fetch(s + 1, av[(s + 1) & 1], bv[(s + 1) & 1]);
#pragma unroll
        for (int i = 0; i < FM; ++i)
#pragma unroll
          for (int j = 0; j < 2; ++j) acc[i][j] = mfma_step<T>(bv[s & 1][j], av[s & 1][i], acc[i][j]);
      }
      rd = rd + 1 == STAGES ? 0 : rd + 1;
      wr_stage = wr_stage + 1 == STAGES ? 0 : wr_stage + 1;
    }
    const int n0 = (first + li) * BN;
    const bool quads = N % 4 == 0 && ldy % 4 == 0 && ((uintptr_t)y & (4 * sizeof(T) - 1)) == 0;
    const int col0 = n0 + wn * 64 + 4 * half;
#pragma unroll
    for (int i = 0; i < FM; ++i) {
      const int64_t row = wm * (32 * FM) + i * 32 + (lane & 31);
      if (row >= M) continue;
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const int col = col0 + j * 32 + 8 * q;
          if (col >= N) continue;
          float v[4];
#pragma unroll
          for (int e = 0; e < 4; ++e)
            v[e] = acc[i][j][4 * q + e] + (bias != nullptr && col + e < N ? load_f32<T>(bias, col + e) : 0.f);
          T* o = y + row * ldy + col;
          if (quads) {
            store_vec<T, 4>(o, v);
          } else {
#pragma unroll 1
            for (int e = 0; e < 4 && col + e < N; ++e) store_f32<T>(o, e, e == 0 ? v[0] : e == 1 ? v[1] : e == 2 ? v[2] : v[3]);
          }
        }
    }
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // (the last zero stages land before the LDS is given back)
}

// y = epilogue(sum over the S splits of part[s][M][N]), splits added in order;
// PER (4 when N is a multiple of 4) consecutive elements of a row per thread.
template <typename T, int EPI, int PER>
__global__ __launch_bounds__(256) void gemm_reduce_kernel(const float* __restrict__ part, int S, const T* bias, T* y,
                                                          int64_t ldy, const T* aux, int64_t M, int64_t N,
                                                          const StepState* state) {
  if (state != nullptr) y = (T*)state->args.logits;
  const int64_t e0 = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) * PER;
  if (e0 >= M * N) return;
  // (32-bit division where it reaches: a 64-bit one costs more than the loads)
  const int64_t row = e0 < (1LL << 31) ? (int64_t)((uint32_t)e0 / (uint32_t)N) : e0 / N, col = e0 - row * N;
  float v[PER];
  if constexpr (PER == 4) {
    sum_partials<4>(Partials{part, S, M, N}, row, col, v);
  } else {
    v[0] = part[e0];
    for (int s = 1; s < S; ++s) v[0] += part[s * M * N + e0];
  }
#pragma unroll
  for (int u = 0; u < PER; ++u) {
    if constexpr (EPI == MINITP_EPI_RESID)
      v[u] = add_rn(load_f32<T>(aux, row * ldy + col + u), round_to<T>(v[u]));
    else
      v[u] += bias != nullptr ? load_f32<T>(bias, col + u) : 0.f;
  }
  T* o = y + row * ldy + col;
  if (PER == 4 && ((uintptr_t)o & (4 * sizeof(T) - 1)) == 0) {
    store_vec<T, 4>(o, v);
  } else {
#pragma unroll
    for (int u = 0; u < PER; ++u) store_f32<T>(o, u, v[u]);
  }
}

// The tile shapes and what a launch on them costs: measured in a graph between
// other kernels, cold weights, as FIXED_US + rounds x (stages x stage_us +
// round_us), a round being one block per CU (blocks sharing a CU add up their
// times within a few percent) and a stage 128 bytes of K.
//   256 x 128, 16 waves, 144 KiB of LDS: 2000 x 3584 x 3584      53.7 us (957 TFLOP/s)
//   128 x 128,  8 waves, 128 KiB: 433 x 3584 x 3584 in 2 splits  20.7 us
//    64 x 128,  8 waves,  96 KiB: 433 x 4608 x 3584              27.8 us
//    64 x  64,  4 waves,  64 KiB: 1099 x 896 x 4864              19.4 us
//    32 x  64,  4 waves,  72 KiB: 8 x 37888 x 3584               46.7 us (5.8 TB/s)
// against 77.8, 31.0, 32.6, 68.1 and 76.0 us for register-staged 64 x 64 and
// 128 x 128 tiles without the ring. A product of one row tile reads every
// weight once: non-temporal loads (8 x 37888 x 3584: 52.8 us without). Rings: 3 stages of 64 x 64 are 3-10 %
// slower than 4 in bf16, 8 no faster. fp32 (bound by its MFMAs) always takes
// 64 x 64 with 3 stages (32 x 64 up to 32 rows): the fastest or within 3 % at
// every shape measured (999 x 9728 x 896: 153 us against 164-169 and 8 stages
// 204; 30 x 151936 x 896: 114 us against 158 on 64 x 64).
using TileXL = Tile<256, 128, 2, 3>;
using TileL = Tile<128, 128, 2, 4>;
using TileStream = Tile<256, 128, 1, 3>;
using TileN = Tile<64, 128, 4, 4>;
using TileS = Tile<64, 64, 4, 4>;
using TileSnt = Tile<64, 64, 4, 4, true>;
using TileXS = Tile<32, 64, 4, 6, true>;
// Unsplit bf16 products of at most SHORT_STAGES stages: waves with a smaller
// wave tile each instead of wave groups that share K. The groups' exchange and
// the deeper ring cost more than they give there: 64 x 1000 x 520 8.1 us on
// 64 x 64 tiles of groups, 5.7 so; 33 x 64 x 64 4.1, 2.8; 128 x 9728 x 896 (64 x
// 128 tiles) 11.6, 10.7; 256 x 9728 x 896 (128 x 128) 14.4, 13.6; from 24 stages on
// the groups win (600 x 512 x 2048 10.5 against 11.4: a 32 x 32 wave tile reads
// twice the LDS bytes). Many blocks want a short ring, so that more of them share
// a CU: 33 x 151936 x 896 on 64 x 128 53.7 us with 3 stages, 59.0 with 4 (64 on
// groups); 33 x 37888 x 3584, 592 blocks of 64 x 64, 55.7 with 2 stages, 58.1 with 4
// (57.7 on groups and non-temporal loads), so one row tile of many blocks takes them too.
constexpr int64_t SHORT_STAGES = 16;
using TileS2w = Tile<64, 64, 1, 2, false, 1, 1, true>;
using TileS2 = Tile<64, 64, 1, 2, false, 1, 1>;
using TileS4 = Tile<64, 64, 1, 4, false, 1, 1>;
using TileN3 = Tile<64, 128, 1, 3, false, 1, 1>;
using TileN4 = Tile<64, 128, 1, 4, false, 1, 1>;
using TileL3 = Tile<128, 128, 1, 3, false, 2, 1>;
using TileS32 = Tile<64, 64, 4, 3>;
using TileXS32 = Tile<32, 64, 4, 3, true>;

struct TileCost {
  int bm, bn;
  float stage_us, round_us;
};
constexpr TileCost TILE_COST[] = {
    {256, 128, 0.90f, 4.5f}, {128, 128, 0.60f, 3.f}, {64, 128, 0.42f, 2.f}, {64, 64, 0.25f, 0.5f}, {32, 64, 0.22f, 0.5f}};
// fp32: one block alone on a CU leaves its MFMAs idle between stages (0.64 us
// a stage of 64 x 64), blocks that share one fill in for each other (0.53)
constexpr TileCost F32_COST[] = {{64, 64, 0.53f, 1.f}, {32, 64, 0.33f, 0.5f}};
constexpr float F32_ALONE = 1.2f;
enum { KIND_XL = 0, KIND_L = 1, KIND_N = 2, KIND_S = 3, KIND_XS = 4 };
constexpr int64_t XS_ROWS = 32, S_NT_ROWS = 64;
// (REDUCE_US: the reduction launch takes 3 us, and a direct call's host as long
// again for it and its scratch as an unsplit launch: 33 x 4608 x 3584 then
// 33 x 3584 x 3584 and three small kernels, 58.6 us a pass split, host-bound)
constexpr float FIXED_US = 3.3f, REDUCE_US = 12.f;
constexpr float PARTIALS_PER_US = 1e6f;   // fp32 partials written and read back
constexpr int64_t SPLIT_MIN_STAGES = 2;   // stages a split runs at least

struct GemmPlan {
  int kind;
  int64_t S, kper;
  float us;
};

// The cheapest tile shape and number of K splits of an M x N x K product by
// the costs above. ws_bytes: room for the partials (0: no splits); split_us:
// what a split adds (the reduction launch). swiglu: W has 2N rows.
GemmPlan gemm_plan(int dtype, int64_t M, int64_t N, int64_t K, bool swiglu, int64_t ws_bytes, float split_us) {
  const bool f32 = dtype == MINITP_F32;
  const int64_t tk = f32 ? 32 : 64, stages = cdiv(K, tk), cus = device_cus();
  GemmPlan best{-1, 1, stages * tk, 0.f};
  for (int kind = M <= XS_ROWS ? KIND_XS : f32 ? KIND_S : KIND_XL; kind <= (M <= XS_ROWS ? KIND_XS : KIND_S); ++kind) {
    const TileCost& c = f32 ? F32_COST[kind - KIND_S] : TILE_COST[kind];
    const int64_t tiles = cdiv(M, c.bm) * cdiv(swiglu ? 2 * N : N, c.bn);
    for (int64_t s = 1; s <= 16; ++s) {
      if (s > 1 && (s * M * N * 4 > ws_bytes || stages < s * SPLIT_MIN_STAGES || tiles * (s - 1) >= 2 * cus)) break;
      const int64_t per = cdiv(stages, s);
      if (cdiv(stages, per) != s) continue;
      const float alone = f32 && tiles * s <= cus ? F32_ALONE : 1.f;
      const float us = FIXED_US + (float)cdiv(tiles * s, cus) * ((float)per * c.stage_us * alone + c.round_us) +
                       (s > 1 ? split_us + (float)(s * M * N) / PARTIALS_PER_US : 0.f);
      if (best.kind < 0 || us < best.us) best = GemmPlan{kind, s, per * tk, us};
    }
  }
  return best;
}

// Rows of x past 4 GiB from a tile's first row, or a [gate; up] weight past
// it, are out of a buffer resource's reach.
inline bool gemm_operands_fit(int64_t M, int64_t N, int64_t K, int64_t ldx, int64_t es) {
  return N * K * es <= 0xffffffffLL && ((M - 1) * ldx + K) * es <= 0xffffffffLL && M < (1LL << 31) &&
         N < (1LL << 30) && K < (1LL << 26);
}

template <typename T, typename C, int OUT>
int launch_cfg(hipStream_t st, const T* x, int64_t ldx, const T* w, const T* bias, T* y, int64_t ldy, int64_t M,
               int64_t N, int64_t K, const T* aux, const StepState* state, float* part, const GemmPlan& p) {
  if (const int rc = ensure_lds_limit((const void*)gemm_kernel<T, C, OUT>, C::LDS_BYTES)) return rc;
  const int tiles_m = (int)cdiv(M, C::BM), tiles_n = (int)cdiv(OUT == OUT_SWIGLU ? 2 * N : N, C::BN);
  const int64_t items = (int64_t)tiles_m * tiles_n * p.S;
  const dim3 grid((unsigned)(8 * cdiv(items, 8)));
  hipLaunchKernelGGL((gemm_kernel<T, C, OUT>), grid, dim3(C::THREADS), C::LDS_BYTES, st, x, ldx, w, bias, y, ldy, aux,
                     part, (int)M, (int)N, (int)K, (int)p.kper, tiles_m, tiles_n, (int)items, state);
  MINITP_LAUNCH_CHECK();
  return MINITP_OK;
}

// One row tile, two rounds of 256 x 128 tiles and more, of at most 32 stages (more
// row tiles run on the 256 x 256 ones): the running
// ring saves about 4.5 us a tile and its eight waves lose 0.12 a stage against
// gemm_kernel's sixteen (N = 151,936, K = 896, 14 stages: 150 rows 99.5 -> 86.5
// us, 194 rows 107 -> 97, 250 rows 119.6 -> 105; N = 152,064, 200 rows: K = 1,536
// 157 against 152, 2,048 199.5 and 196.9, 2,560 235 and 239, 3,584 307 and 321; N =
// 98,304 crosses between 2,048 and 2,560 too).
inline bool stream_pays(int64_t M, int64_t N, int64_t K) {
  return M <= TileStream::BM && cdiv(N, TileStream::BN) >= 2 * (int64_t)device_cus() && K <= 2048;
}

template <typename T, typename C>
int launch_stream(hipStream_t st, const T* x, int64_t ldx, const T* w, const T* bias, T* y, int64_t ldy, int64_t M,
                  int64_t N, int64_t K, const StepState* state) {
  if (const int rc = ensure_lds_limit((const void*)gemm_stream_kernel<T, C>, C::RING_BYTES)) return rc;
  const int64_t items = cdiv(N, C::BN);
  const dim3 grid((unsigned)(8 * cdiv(std::min<int64_t>(items, device_cus()), 8)));
  hipLaunchKernelGGL((gemm_stream_kernel<T, C>), grid, dim3(C::THREADS), C::RING_BYTES, st, x, ldx, w, bias, y, ldy,
                     (int)M, (int)N, (int)K, (int)items, state);
  MINITP_LAUNCH_CHECK();
  return MINITP_OK;
}

// The tile of an unsplit product (no SwiGLU) of at most SHORT_STAGES stages, or
// of one row tile and many blocks (TileS2w's group above): LONG_TILE for none.
enum ShortTile { LONG_TILE, SHORT_S2W, SHORT_S2, SHORT_S4, SHORT_N3, SHORT_N4, SHORT_L3 };
inline ShortTile short_tile(int kind, int64_t M, int64_t N, int64_t K) {
  const int64_t stages = cdiv(K, 64), cus = device_cus();
  const int64_t blocks = cdiv(M, TILE_COST[kind].bm) * cdiv(N, TILE_COST[kind].bn);
  const bool few = stages <= SHORT_STAGES;
  if (kind == KIND_S && stages <= 2) return SHORT_S2W;
  if (kind == KIND_S && blocks > 2 * cus && (few || M <= S_NT_ROWS)) return SHORT_S2;
  if (kind == KIND_S && few) return SHORT_S4;
  if (kind == KIND_N && few) return blocks > cus ? SHORT_N3 : SHORT_N4;
  if (kind == KIND_L && few) return SHORT_L3;
  return LONG_TILE;
}

// Wave groups that share K in the tiles a plan runs on: with its splits, all
// that the order of a product's sums depends on.
static_assert(TileXL::WK == 2 && TileL::WK == 2 && TileN::WK == 4 && TileS::WK == 4 && TileSnt::WK == 4 &&
                  TileXS::WK == 4 && TileS32::WK == 4 && TileXS32::WK == 4 && TileStream::WK == 1 && TileS4::WK == 1,
              "plan_groups");
inline int plan_groups(int dtype, const GemmPlan& p, int64_t M, int64_t N, int64_t K, bool swiglu) {
  if (dtype == MINITP_F32 || p.kind == KIND_XS) return 4;
  if (!swiglu && p.S == 1 &&
      (p.kind == KIND_XL ? stream_pays(M, N, K) : short_tile(p.kind, M, N, K) != LONG_TILE))
    return 1;
  return p.kind == KIND_XL || p.kind == KIND_L ? 2 : 4;
}

template <typename T, int OUT>
int launch_plan(hipStream_t st, const T* x, int64_t ldx, const T* w, const T* bias, T* y, int64_t ldy, int64_t M,
                int64_t N, int64_t K, const T* aux, const StepState* state, float* part, const GemmPlan& p) {
  auto go = [&](auto cfg) {
    return launch_cfg<T, decltype(cfg), OUT>(st, x, ldx, w, bias, y, ldy, M, N, K, aux, state, part, p);
  };
  if constexpr (sizeof(T) == 2) {
    if constexpr (OUT == MINITP_EPI_NONE)
      if (p.kind == KIND_XL && p.S == 1 && stream_pays(M, N, K))
        return launch_stream<T, TileStream>(st, x, ldx, w, bias, y, ldy, M, N, K, state);
    if constexpr (OUT == MINITP_EPI_NONE || OUT == MINITP_EPI_RESID) {
      switch (short_tile(p.kind, M, N, K)) {
        case SHORT_S2W: return go(TileS2w{});
        case SHORT_S2: return go(TileS2{});
        case SHORT_S4: return go(TileS4{});
        case SHORT_N3: return go(TileN3{});
        case SHORT_N4: return go(TileN4{});
        case SHORT_L3: return go(TileL3{});
        case LONG_TILE: break;
      }
    }
    if (p.kind == KIND_XL) return go(TileXL{});
    if (p.kind == KIND_L) return go(TileL{});
    if (p.kind == KIND_N) return go(TileN{});
    if (p.kind == KIND_XS) return go(TileXS{});
    return M <= S_NT_ROWS ? go(TileSnt{}) : go(TileS{});
  } else {
    return p.kind == KIND_XS ? go(TileXS32{}) : go(TileS32{});
  }
}

template <typename T, int EPI>
int launch_reduce(hipStream_t st, const float* ws, int64_t S, const T* bias, T* y, int64_t ldy, const T* aux,
                  int64_t M, int64_t N, const StepState* state) {
  if (N % 4 == 0 && aligned16(ws)) {
    const unsigned grid = (unsigned)cdiv(M * N / 4, 256);
    hipLaunchKernelGGL((gemm_reduce_kernel<T, EPI, 4>), dim3(grid), dim3(256), 0, st, ws, (int)S, bias, y, ldy, aux, M,
                       N, state);
  } else {
    const unsigned grid = (unsigned)cdiv(M * N, 256);
    hipLaunchKernelGGL((gemm_reduce_kernel<T, EPI, 1>), dim3(grid), dim3(256), 0, st, ws, (int)S, bias, y, ldy, aux, M,
                       N, state);
  }
  MINITP_LAUNCH_CHECK();
  return MINITP_OK;
}

template <typename T>
int gemm_typed(hipStream_t st, const T* x, int64_t ldx, const T* w, const T* bias, T* y, int64_t ldy, int64_t M,
               int64_t N, int64_t K, int epi, const T* aux, const StepState* state, float* ws, int64_t ws_bytes) {
  if (!gemm_operands_fit(M, N, K, ldx, sizeof(T))) {
    set_error("gemm: operands over 4 GiB (M=%lld N=%lld K=%lld)", (long long)M, (long long)N, (long long)K);
    return MINITP_ERR_UNSUPPORTED;
  }
  const GemmPlan p = gemm_plan(sizeof(T) == 4 ? MINITP_F32 : MINITP_BF16, M, N, K, false, ws ? ws_bytes : 0, REDUCE_US);
  const bool resid = epi == MINITP_EPI_RESID;
  if (p.S > 1) {
    const int rc = launch_plan<T, OUT_PARTIAL>(st, x, ldx, w, bias, y, ldy, M, N, K, aux, state, ws, p);
    if (rc) return rc;
    return resid ? launch_reduce<T, MINITP_EPI_RESID>(st, ws, p.S, bias, y, ldy, aux, M, N, state)
                 : launch_reduce<T, MINITP_EPI_NONE>(st, ws, p.S, bias, y, ldy, aux, M, N, state);
  }
  return resid ? launch_plan<T, MINITP_EPI_RESID>(st, x, ldx, w, bias, y, ldy, M, N, K, aux, state, ws, p)
               : launch_plan<T, MINITP_EPI_NONE>(st, x, ldx, w, bias, y, ldy, M, N, K, aux, state, ws, p);
}

// One row block of a packed weight on the splits and wave groups of the whole,
// the larger tile of those groups where it still gives every CU a block.
template <typename T, int OUT>
int launch_block_tile(hipStream_t st, const T* x, int64_t ldx, const T* w, const T* bias, T* y, int64_t ldy, int64_t M,
                      int64_t N, int64_t K, float* part, const GemmPlan& p, int groups) {
  auto go = [&](auto cfg) {
    return launch_cfg<T, decltype(cfg), OUT>(st, x, ldx, w, bias, y, ldy, M, N, K, nullptr, nullptr, part, p);
  };
  if constexpr (sizeof(T) == 4) {
    return M <= XS_ROWS ? go(TileXS32{}) : go(TileS32{});
  } else {
    auto fills = [&](int64_t bm, int64_t bn) { return cdiv(M, bm) * cdiv(N, bn) * p.S >= device_cus(); };
    if constexpr (OUT == MINITP_EPI_NONE)
      if (groups == 1) return fills(128, 128) ? go(TileL3{}) : go(TileS4{});
    if (groups == 2) return fills(256, 128) ? go(TileXL{}) : go(TileL{});
    if (M <= XS_ROWS) return go(TileXS{});
    return fills(64, 128) ? go(TileN{}) : M <= S_NT_ROWS ? go(TileSnt{}) : go(TileS{});
  }
}

template <typename T>
int launch_block(hipStream_t st, const T* x, int64_t ldx, const T* w, const T* bias, T* y, int64_t ldy, int64_t M,
                 int64_t N, int64_t K, const GemmPlan& p, int groups, float* ws) {
  if (p.S == 1)
    return launch_block_tile<T, MINITP_EPI_NONE>(st, x, ldx, w, bias, y, ldy, M, N, K, nullptr, p, groups);
  const int rc = launch_block_tile<T, OUT_PARTIAL>(st, x, ldx, w, bias, y, ldy, M, N, K, ws, p, groups);
  return rc ? rc : launch_reduce<T, MINITP_EPI_NONE>(st, ws, p.S, bias, y, ldy, nullptr, M, N, nullptr);
}

}  // namespace

bool gemm_prefers_tile(int64_t M, int64_t N, int64_t K, int64_t ldx, int64_t ldy, bool swiglu, int64_t ws_bytes,
                       float split_us) {
  if (!gemm_tile_supported(M, N, K, ldx, ldy, swiglu)) return false;
  const int64_t tiles = cdiv(M, 256) * cdiv(swiglu ? 2 * N : N, 256), cus = device_cus(), steps = cdiv(K, 64);
  // (the last round may be split over K when the caller brings the workspace)
  int split;
  const float round = (float)steps * TILE_STAGE_US + TILE_ROUND_US;
  const float last = ws_bytes ? gemm_tile_tail(tiles, steps, cus, &split) : tiles % cus ? round : 0.f;
  const float us = FIXED_US + (float)(tiles / cus) * round + last;
  return us <= gemm_plan(MINITP_BF16, M, N, K, swiglu, swiglu ? 0 : ws_bytes, split_us).us;
}

int64_t gemm_split_bytes(int dtype, int64_t M, int64_t N, int64_t K, bool plain) {
  if (dtype == MINITP_BF16 && plain && gemm_prefers_tile(M, N, K, K, N, false, GEMM_WS_BYTES, REDUCE_US)) return 0;
  const GemmPlan p = gemm_plan(dtype, M, N, K, false, GEMM_WS_BYTES, REDUCE_US);
  return p.S > 1 ? p.S * M * N * 4 : 0;
}

int launch_gemm_swiglu(hipStream_t st, int dtype, const void* x, int64_t ldx, const void* w, void* y, int64_t ldy,
                       int64_t M, int64_t N, int64_t K, TileTail tail) {
  if (M == 0 || N == 0) return MINITP_OK;
  const int64_t es = dtype == MINITP_F32 ? 4 : 2;
  if (dtype == MINITP_BF16 && aligned16(x) && aligned16(w) &&
      gemm_prefers_tile(M, N, K, ldx, ldy, true, tail.part != nullptr ? TILE_TAIL_BYTES : 0, 0.f))
    return launch_gemm_tile(st, x, ldx, w, nullptr, y, ldy, M, N, K, true, tail);
  if (ldy < N || K * es % 16 != 0 || !aligned16(x) || !aligned16(w) || 2 * N * K * es >= (int64_t)ROW_OOB ||
      !gemm_operands_fit(M, 2 * N, K, ldx, es)) {
    set_error("gemm: SwiGLU form M=%lld N=%lld K=%lld not served", (long long)M, (long long)N, (long long)K);
    return MINITP_ERR_UNSUPPORTED;
  }
  const GemmPlan p = gemm_plan(dtype, M, N, K, true, 0, 0.f);
  return dtype == MINITP_F32
             ? launch_plan<float, OUT_SWIGLU>(st, (const float*)x, ldx, (const float*)w, nullptr, (float*)y, ldy, M, N,
                                              K, nullptr, nullptr, nullptr, p)
             : launch_plan<bf16, OUT_SWIGLU>(st, (const bf16*)x, ldx, (const bf16*)w, nullptr, (bf16*)y, ldy, M, N, K,
                                             nullptr, nullptr, nullptr, p);
}

// The 256 x 256 tiles add K in one sequence, as one wave group does.
int launch_gemm_block(hipStream_t st, int dtype, const void* x, int64_t ldx, const void* w, const void* bias, void* y,
                      int64_t ldy, int64_t M, int64_t N, int64_t K, int64_t packed, bool swiglu, void* ws,
                      int64_t ws_bytes) {
  if (M == 0 || N == 0) return MINITP_OK;
  const int64_t es = dtype == MINITP_F32 ? 4 : 2, whole = swiglu ? packed / 2 : packed;
  if (!gemm_operands_fit(M, N, K, ldx, es)) {
    set_error("gemm: operands over 4 GiB (M=%lld N=%lld K=%lld)", (long long)M, (long long)N, (long long)K);
    return MINITP_ERR_UNSUPPORTED;
  }
  const int64_t room = swiglu || ws == nullptr ? 0 : ws_bytes;
  const float split_us = swiglu ? 0.f : REDUCE_US;
  const bool tile = dtype == MINITP_BF16 && gemm_prefers_tile(M, whole, K, ldx, whole, swiglu, room, split_us);
  const GemmPlan p = tile ? GemmPlan{KIND_S, 1, cdiv(K, 64) * 64, 0.f}
                          : gemm_plan(dtype, M, whole, K, swiglu, room, split_us);
  const int groups = tile ? 1 : plan_groups(dtype, p, M, whole, K, swiglu);
  if (groups == 1 && dtype == MINITP_BF16 && aligned16(x) && aligned16(w) &&
      gemm_tile_supported(M, N, K, ldx, ldy, false))
    return launch_gemm_tile(st, x, ldx, w, bias, y, ldy, M, N, K, false);
  return dtype == MINITP_F32
             ? launch_block<float>(st, (const float*)x, ldx, (const float*)w, (const float*)bias, (float*)y, ldy, M, N,
                                   K, p, groups, (float*)ws)
             : launch_block<bf16>(st, (const bf16*)x, ldx, (const bf16*)w, (const bf16*)bias, (bf16*)y, ldy, M, N, K,
                                  p, groups, (float*)ws);
}

int launch_gemm_partials(hipStream_t st, int dtype, const void* x, int64_t ldx, const void* w, int64_t M, int64_t N,
                         int64_t K, void* ws, int64_t ws_bytes, Partials* out) {
  const int64_t es = dtype == MINITP_F32 ? 4 : 2;
  if (M <= 0 || N % 8 != 0 || ws == nullptr || !aligned16(ws) || !aligned16(x) || !aligned16(w) ||
      !gemm_operands_fit(M, N, K, ldx, es) ||
      (dtype == MINITP_BF16 && gemm_prefers_tile(M, N, K, ldx, N, false, ws_bytes, 0.f)))
    return MINITP_ERR_UNSUPPORTED;
  const GemmPlan p = gemm_plan(dtype, M, N, K, false, ws_bytes, 0.f);
  if (p.S < 2) return MINITP_ERR_UNSUPPORTED;
  const int rc =
      dtype == MINITP_F32
          ? launch_plan<float, OUT_PARTIAL>(st, (const float*)x, ldx, (const float*)w, nullptr, nullptr, N, M, N, K,
                                            nullptr, nullptr, (float*)ws, p)
          : launch_plan<bf16, OUT_PARTIAL>(st, (const bf16*)x, ldx, (const bf16*)w, nullptr, nullptr, N, M, N, K,
                                           nullptr, nullptr, (float*)ws, p);
  if (rc) return rc;
  *out = Partials{(const float*)ws, (int)p.S, M, N};
  return MINITP_OK;
}

int launch_gemm(hipStream_t st, int dtype, const void* x, int64_t ldx, const void* w, const void* bias, void* y,
                int64_t ldy, int64_t M, int64_t N, int64_t K, int epi, const void* aux, const StepState* state,
                void* ws, int64_t ws_bytes, TileTail tail) {
  if (M == 0 || N == 0) return MINITP_OK;
  if (epi != MINITP_EPI_NONE && epi != MINITP_EPI_RESID) {
    set_error("gemm: epilogue %d not supported (split SwiGLU runs as its own kernel)", epi);
    return MINITP_ERR_UNSUPPORTED;
  }
  // bf16 products large enough to fill the chip with 256 x 256 tiles
  if (dtype == MINITP_BF16 && epi == MINITP_EPI_NONE && state == nullptr && aligned16(x) && aligned16(w) &&
      gemm_prefers_tile(M, N, K, ldx, ldy, false, ws != nullptr ? ws_bytes : 0, REDUCE_US))
    return launch_gemm_tile(st, x, ldx, w, bias, y, ldy, M, N, K, false, tail);
  return dtype == MINITP_F32
             ? gemm_typed<float>(st, (const float*)x, ldx, (const float*)w, (const float*)bias, (float*)y, ldy, M, N,
                                 K, epi, (const float*)aux, state, (float*)ws, ws_bytes)
             : gemm_typed<bf16>(st, (const bf16*)x, ldx, (const bf16*)w, (const bf16*)bias, (bf16*)y, ldy, M, N, K,
                                epi, (const bf16*)aux, state, (float*)ws, ws_bytes);
}

}  // namespace minitp
