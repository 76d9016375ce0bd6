// Gated-MLP up projection with the SwiGLU epilogue, on the matrix cores:
//
//   out[t, i] = round16(silu(g) * u),  g = x[t, :] . w_gate[i, :],  u = x[t, :] . w_up[i, :]
//
// with g and u accumulated in fp32 and never rounded to 16 bits.  The
// reference runs this as two GEMMs into [T, I] gate and up buffers followed by
// a silu_mul pass over both (vllm_apple/engine/ops/mlp.py:247-330 with
// elementwise.py:114-124); here the epilogue reads g and u from the
// accumulators, so neither intermediate is written or read back.
//
// Tiling (one 4-wave workgroup per CU, 128, 144 or 160 KB of LDS):
//   workgroup = 64 NB tokens (NB = 2, 3 or 4, wide_blocks) x 128 output columns: a
//               64 NB x 256 product of the token rows of x against 256 weight
//               rows (128 gate, then the 128 up rows of the same columns);
//   wave w    = tokens 32 NB*(w/2) .. +32 NB x columns 64*(w%2) .. +64, a 4 x NB
//               grid of 32x32 MFMA tiles (two gate and two up row blocks by
//               NB token blocks), so the gate and up values of one output
//               sit in the same lane, in the same accumulator position;
//   k-step    = 64 hidden elements.  The product is computed transposed,
//               W x^T, with v_mfma_f32_32x32x16: the A operand is 8 weights of
//               one row and the B operand 8 activations of one token, both
//               read from LDS with ds_read_b128.  Lanes 0-31 take the first
//               half of the step's 64 elements and lanes 32-63 the second
//               (the contraction index is a sum, so any assignment that the
//               two operands share is exact).
//
// Memory: both operands are rows contiguous in the hidden dimension.  They
// move from HBM to LDS with direct loads (buffer_load_dwordx4 ... lds: lane i
// of a wave writes LDS bytes [16i, 16i + 16) after the wave-uniform base in
// M0).  The loads are inline asm, so the compiler does not track them (it
// would otherwise wait for every one of them before any LDS read); the
// kernel orders each LDS read behind its own counted vmcnt wait and barrier.
// Weight tiles go through a ring of three 32 KB stages and activation tiles
// through two of 8 NB KB: during step k the wave issues the activation
// loads of step k + 1 and then the weight loads of step k + 2, spread over
// the MFMAs of the step's first half, so the weight stream,
// which comes from HBM, has two steps to land and the activations, which
// come from L2 and the Infinity Cache, one.  The 16-byte chunks of each 128-byte LDS
// row are XOR-swizzled by row & 7,
// so the eight consecutive rows that an operand read spans per 128 bytes hit
// distinct banks.  Token rows past num_tokens read the last token's row
// (always in bounds) and their outputs are not stored.
// What bounds a step is the LDS port beside the MFMAs: the operand reads and
// the direct loads' writes take 1536 of its cycles against 2048 of MFMA at NB = 4
// and 1344 against 1536 at NB = 3.
//
// The same kernel runs 256 rows of a plain product (kPart: the down projection of
// 129 to 1024 tokens) with the k-steps split so that one workgroup runs on every
// CU; the fp32 partials are summed by wide_sum_kernel.
//
// Workgroup order: the 8 XCDs each take a contiguous range of (column tile,
// token tile) pairs, token tile fastest, so all the token tiles that share a
// weight tile run at the same time on one XCD and read it through its L2.
#include "common.h"

#include <algorithm>

namespace vaa {
namespace {

constexpr int kGI = 128;                         // output columns per workgroup
constexpr int kGK = 64;                          // hidden elements per k-step
constexpr int kGWaves = 4;
constexpr int kGThreads = kGWaves * kWave;
constexpr int kGRowB = kGK * 2;                  // bytes per LDS row
constexpr int kGTileB = 256 * kGRowB;            // one operand tile: 256 rows, 32 KB
constexpr int kGLoads = kGTileB / (kGThreads * 16);  // direct loads per wave per operand
constexpr int kGXcds = 8;
#ifndef VAA_GLU_SMALL_TOKENS
#define VAA_GLU_SMALL_TOKENS 128
#endif
constexpr int kSmallTokens = VAA_GLU_SMALL_TOKENS;  // the few-token kernel up to this many tokens
static_assert(kGLoads == 8, "eight 1 KB direct loads per wave and operand");

// Word 3 of a raw buffer resource on gfx9-family parts: 32-bit data format,
// no swizzle, offsets checked against the byte range in word 2.
constexpr int kBufDword3 = 0x00020000;

typedef int i32x4v __attribute__((ext_vector_type(4)));

// Raw buffer resource for [base, base + bytes), in scalar registers.
__device__ __forceinline__ i32x4v buffer_rsrc(const char* base, int bytes) {
  const uint64_t b = reinterpret_cast<uint64_t>(base);
  i32x4v r;
  r[0] = __builtin_amdgcn_readfirstlane(static_cast<int>(b & 0xffffffffu));
  r[1] = __builtin_amdgcn_readfirstlane(static_cast<int>((b >> 32) & 0xffffu));
  r[2] = __builtin_amdgcn_readfirstlane(bytes);
  r[3] = kBufDword3;
  return r;
}
// One direct load of 16 bytes per lane into LDS: lane i writes bytes
// [m0 + 16i, m0 + 16i + 16).  M0 is written here and used by nothing else
// in this kernel.
__device__ __forceinline__ void dma16(const i32x4v& rs, int voff, int soff, uint32_t m0) {
  asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tbuffer_load_dwordx4 %0, %2, %3 offen lds"
               :
               : "v"(voff), "s"(m0), "s"(rs), "s"(soff)
               : "memory", "m0");
}
// The same with the nontemporal hint, for weight tiles that one call reads
// once: with few token tiles (T <= 1024 here, and the small-token kernel) the
// hint speeds the weight stream up (C5 MLP shape: 16 tokens 0.117 -> 0.105
// ms, 6.4 TB/s of weights; 256 tokens 0.181 -> 0.170 ms).  With more token
// tiles the tiles that share a weight tile read it again through L2, and the
// hint stopped helping (2104 tokens: 1.254 against 1.248 ms).
__device__ __forceinline__ void dma16_stream(const i32x4v& rs, int voff, int soff, uint32_t m0) {
  asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tbuffer_load_dwordx4 %0, %2, %3 offen nt lds"
               :
               : "v"(voff), "s"(m0), "s"(rs), "s"(soff)
               : "memory", "m0");
}

struct GluArgs {
  const char* x;
  const char* wg;
  const char* wu;
  char* out;
  int64_t xs, ws, os;  // row strides, bytes
  int num_tokens, ksteps, t_tiles, tiles;
  // Few-token kernel: k-steps per split, byte step of wg and wu between column
  // tiles, and the split's fp32 partials (null: one split, SwiGLU epilogue).
  int k_per;
  int64_t w_tile;
  float* part;
};

// s_waitcnt vmcnt(8) lgkmcnt(0), at the top of step k: every vector memory
// load of this wave but the newest 8 has landed.  Loads complete in issue
// order and the newest 8 are the weights of step k + 1 (issued last in step
// k - 1), so the activations of step k (issued before them) and the weights
// of step k (issued in step k - 2) are in LDS, as far as this wave's loads
// go; the barrier that follows covers the other waves'.
__device__ __forceinline__ void glu_wait_tiles() { __builtin_amdgcn_s_waitcnt(0x0078); }

// NB: 32-token blocks per wave (the workgroup's tile is 64 NB tokens).  kPart:
// the two matrices are 256 rows of one plain product, the k-steps are split and
// the fp32 sums go to a.part.
template <typename T, bool kStreamW, int NB, bool kPart>
__global__ void __launch_bounds__(kGThreads) __attribute__((amdgpu_waves_per_eu(1, 1)))
gate_up_silu_kernel(GluArgs a) {
  constexpr int kTT = 64 * NB;             // tokens per workgroup
  constexpr int kXTile = kTT * kGRowB;     // activation tile, bytes
  constexpr int kXLoads = 2 * NB;          // direct loads per wave per activation tile
  __shared__ __align__(16) char smem[3 * kGTileB + 2 * kXTile];  // W stages 0-2, x stages 0-1
  char* const w0 = smem;
  char* const w1 = smem + kGTileB;
  const uint32_t lds0 = __builtin_amdgcn_readfirstlane(
      static_cast<uint32_t>(reinterpret_cast<uintptr_t>(smem)));

  const int per_xcd = static_cast<int>(gridDim.x) / kGXcds;
  int logical = (static_cast<int>(blockIdx.x) % kGXcds) * per_xcd +
                static_cast<int>(blockIdx.x) / kGXcds;
  // kPart: the tiles of all splits, one split after the other, are dealt over
  // the XCDs together.  (Dealt split by split, a tile count that is no multiple
  // of 8 leaves the same XCDs short in every split and the others with more
  // workgroups than CUs: 18 tiles in 12 splits made 36 on six XCDs of 32 CUs.)
  int split = 0;
  if constexpr (kPart) {
    split = logical / a.tiles;
    if (split * a.k_per >= a.ksteps) return;
    logical -= split * a.tiles;
  } else if (logical >= a.tiles) {
    return;
  }
  const int t0 = (logical % a.t_tiles) * kTT;
  const int i0 = (logical / a.t_tiles) * kGI;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;

  // Direct-load sources, as buffer loads: a wave-uniform resource and k
  // offset, and a per-lane 32-bit offset.  Slot P of a tile is LDS row P / 8,
  // physical chunk P % 8, which holds logical chunk (P % 8) ^ (row & 7).
  // Weight rows 0-127 (waves 0 and 1) are the gate rows i0.., rows 128-255
  // (waves 2 and 3) the up rows of the same columns, so each wave reads one
  // weight matrix; its load q is 8 rows further on.  Every access stays
  // inside its resource's range (rows of x are clamped to num_tokens - 1).
  const char* wbase = (wave < 2 ? a.wg : a.wu) + (logical / a.t_tiles) * a.w_tile;
  const i32x4v wrs = buffer_rsrc(wbase, static_cast<int>(kGI * a.ws));
  const i32x4v xrs = buffer_rsrc(a.x, static_cast<int>(a.num_tokens * a.xs));
  const int rw = 8 * (wave & 1) * kGLoads + (lane >> 3);  // weight row of load 0, mod 128
  const int lc = (lane & 7) ^ (rw & 7);                    // a wave's rows agree mod 8
  const int woff = rw * static_cast<int>(a.ws) + lc * 16;
  const int wstep = 8 * static_cast<int>(a.ws);
  int xoff[kXLoads];
#pragma unroll
  for (int q = 0; q < kXLoads; ++q) {
    const int R = 8 * (wave * kXLoads + q) + (lane >> 3);
    xoff[q] = min(t0 + R, a.num_tokens - 1) * static_cast<int>(a.xs) + lc * 16;
  }
  const int dst0 = 1024 * wave * kGLoads, xdst0 = 1024 * wave * kXLoads;

  // Operand reads: row l % 32 of a 32-row block, logical chunk 4 (l / 32) + s.
  const int l32 = lane & 31, hb = lane >> 5;
  int rd[4];
#pragma unroll
  for (int s = 0; s < 4; ++s) rd[s] = l32 * kGRowB + (((4 * hb + s) ^ (l32 & 7)) << 4);
  const int wi = wave & 1, wt = wave >> 1;
  // Weight row blocks: gate 64wi, 64wi + 32; up 128 + 64wi, 128 + 64wi + 32.
  const int wrow[4] = {64 * wi, 64 * wi + 32, kGI + 64 * wi, kGI + 64 * wi + 32};
  const int xrow0 = 32 * NB * wt;

  f32x16 acc[4][NB];
#pragma unroll
  for (int f = 0; f < 4; ++f)
#pragma unroll
    for (int c = 0; c < NB; ++c)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[f][c][r] = 0.f;

  // Direct load L of a step: the first kXLoads move the activation tile of
  // k-step kx into the LDS address xst, the next eight the weight tile of
  // k-step kw into wst.
  auto load1 = [&](int L, int kbx, int kbw, uint32_t xst, uint32_t wst) {
    if (L < kXLoads)
      dma16(xrs, xoff[L], kbx, xst + xdst0 + 1024 * L);
    else if constexpr (kStreamW)
      dma16_stream(wrs, woff, kbw + (L - kXLoads) * wstep, wst + dst0 + 1024 * (L - kXLoads));
    else
      dma16(wrs, woff, kbw + (L - kXLoads) * wstep, wst + dst0 + 1024 * (L - kXLoads));
  };
  auto frags = [&](const char* wt_, const char* xt_, int s, u32x4 (&A)[4], u32x4 (&B)[NB]) {
#pragma unroll
    for (int f = 0; f < 4; ++f)
      A[f] = *reinterpret_cast<const u32x4*>(wt_ + wrow[f] * kGRowB + rd[s]);
#pragma unroll
    for (int c = 0; c < NB; ++c)
      B[c] = *reinterpret_cast<const u32x4*>(xt_ + (xrow0 + 32 * c) * kGRowB + rd[s]);
  };
  // The 4 NB MFMAs of a sub-step, with nl direct loads from L0 on spread
  // between them.
  auto mfmas = [&](const u32x4 (&A)[4], const u32x4 (&B)[NB], int nl, int L0, int kbx, int kbw,
                   uint32_t xst, uint32_t wst) {
#pragma unroll
    for (int idx = 0; idx < 4 * NB; ++idx) {
      const int f = idx / NB, c = idx % NB;
      acc[f][c] = Elem<T>::mfma32x32x16(__builtin_bit_cast(typename Elem<T>::x8, A[f]),
                                        __builtin_bit_cast(typename Elem<T>::x8, B[c]),
                                        acc[f][c]);
      if ((idx + 1) * nl / (4 * NB) > idx * nl / (4 * NB))
        load1(L0 + idx * nl / (4 * NB), kbx, kbw, xst, wst);
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  // Steps k0 .. k0 + n - 1 of this split.
  const int k0 = kPart ? split * a.k_per : 0;
  const int n = kPart ? min(a.ksteps - k0, a.k_per) : a.ksteps;
  // (Starting the column tiles' steps apart, as the few-token kernel does,
  // measured level here: other tiles' MFMAs spread the loads already.)
  auto kstep = [&](int ks) { return (k0 + min(ks, n - 1)) * kGRowB; };
  // Step ks: weights in W stage ks % 3, activations in x stage ks % 2; it
  // loads the activations of step ks + 1 and then the weights of ks + 2.
  auto step = [&](int ks) {
    glu_wait_tiles();
    __syncthreads();
    const char* cw = smem + (ks % 3) * kGTileB;
    const char* cx = smem + 3 * kGTileB + (ks & 1) * kXTile;
    const uint32_t xst = lds0 + 3 * kGTileB + ((ks + 1) & 1) * kXTile;
    const uint32_t wst = lds0 + ((ks + 2) % 3) * kGTileB;
    const int kbx = kstep(ks + 1);
    const int kbw = kstep(ks + 2);
    u32x4 A0[4], B0[NB], A1[4], B1[NB];
    frags(cw, cx, 0, A0, B0);
    frags(cw, cx, 1, A1, B1);
    __builtin_amdgcn_sched_barrier(0);
    mfmas(A0, B0, kXLoads, 0, kbx, kbw, xst, wst);
    frags(cw, cx, 2, A0, B0);
    __builtin_amdgcn_sched_barrier(0);
    mfmas(A1, B1, kGLoads, kXLoads, kbx, kbw, xst, wst);
    frags(cw, cx, 3, A1, B1);
    __builtin_amdgcn_sched_barrier(0);
    mfmas(A0, B0, 0, 0, 0, 0, 0, 0);
    mfmas(A1, B1, 0, 0, 0, 0, 0, 0);
  };
  // Prologue: weights of steps 0 and 1, activations of step 0, issued so
  // that at the top of every step the newest 8 loads are the only ones that
  // may still be in flight (the weights of the next step).
#pragma unroll
  for (int q = 0; q < kGLoads; ++q)
    dma16(wrs, woff, kstep(0) + q * wstep, lds0 + dst0 + 1024 * q);
#pragma unroll
  for (int q = 0; q < kXLoads; ++q)
    dma16(xrs, xoff[q], kstep(0), lds0 + 3 * kGTileB + xdst0 + 1024 * q);
#pragma unroll
  for (int q = 0; q < kGLoads; ++q)
    dma16(wrs, woff, kstep(1) + q * wstep, lds0 + kGTileB + dst0 + 1024 * q);
  for (int ks = 0; ks < n; ++ks) step(ks);
  // Every load has landed before the workgroup ends and its LDS is released.
  __builtin_amdgcn_s_waitcnt(0x0070);

  if constexpr (kPart) {
    // The sums as the lanes hold them: [split][tile][wave][f][c][r4][lane].
    f32x4* p = reinterpret_cast<f32x4*>(a.part) +
               ((static_cast<int64_t>(split) * a.tiles + logical) * kGWaves + wave) *
                   (4 * NB * 4 * kWave) + lane;
#pragma unroll
    for (int f = 0; f < 4; ++f)
#pragma unroll
      for (int c = 0; c < NB; ++c)
#pragma unroll
        for (int r4 = 0; r4 < 4; ++r4)
          p[((f * NB + c) * 4 + r4) * kWave] =
              f32x4{acc[f][c][4 * r4], acc[f][c][4 * r4 + 1], acc[f][c][4 * r4 + 2],
                    acc[f][c][4 * r4 + 3]};
    return;
  }
  // Epilogue, staged through LDS so that the output leaves in whole rows.
  // The lane holds token xrow0 + 32c + l32 and, for row block f, columns
  // 8 (r / 4) + 4 hb + r % 4 of that block: four runs of four consecutive
  // columns.  silu(g) u is formed in registers and written as 8-byte pieces
  // into a [64 NB tokens][128 columns] tile (the first 32 NB token rows in w0,
  // the others in w1, 256 bytes each, 16-byte chunks XOR-swizzled by row & 15 so the 32
  // token rows of one write hit distinct banks); then each row goes out as
  // sixteen 16-byte stores.
  __syncthreads();  // every wave is done with the operand tiles
  char* stage = wt == 0 ? w0 : w1;
#pragma unroll
  for (int c = 0; c < NB; ++c) {
    const int row = 32 * c + l32;  // within this wave's 32 NB token rows
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int g4 = 0; g4 < 4; ++g4) {
        const int col = 64 * wi + 32 * j + 8 * g4 + 4 * hb;
        T v[4];
#pragma unroll
        for (int e = 0; e < 4; ++e)
          v[e] = Elem<T>::from_f(silu_mul1(acc[j][c][4 * g4 + e], acc[2 + j][c][4 * g4 + e]));
        const int chunk = (col >> 3) ^ (row & 15);
        *reinterpret_cast<u32x2*>(stage + row * 256 + chunk * 16 + (col & 7) * 2) =
            __builtin_bit_cast(u32x2, v);
      }
  }
  __syncthreads();
  const int tid = threadIdx.x;
  const int ch = tid & 15;
#pragma unroll 4
  for (int r0 = 0; r0 < kTT; r0 += kGThreads / 16) {
    const int row = r0 + (tid >> 4);
    const int tok = t0 + row;
    if (tok < a.num_tokens) {
      const int in = row < 32 * NB ? row : row - 32 * NB;
      const char* src = (row < 32 * NB ? w0 : w1) + in * 256 + ((ch ^ (in & 15)) << 4);
      *reinterpret_cast<u32x4*>(a.out + static_cast<int64_t>(tok) * a.os + 2 * (i0 + 8 * ch)) =
          *reinterpret_cast<const u32x4*>(src);
    }
  }
}

// Sums the wide kernel's split partials in a fixed order and rounds: a thread
// owns four consecutive columns of one token, in the partials' order.
template <typename T, int NB>
__global__ void __launch_bounds__(256) wide_sum_kernel(GluArgs a, int splits) {
  constexpr int kPerTile = kGWaves * 4 * NB * 4 * kWave;  // f32x4 of a tile
  const int tile = blockIdx.x, in = blockIdx.y * 256 + threadIdx.x;
  const int lane = in % kWave, r4 = in / kWave % 4, c = in / (4 * kWave) % NB;
  const int f = in / (4 * kWave * NB) % 4, wave = in / (16 * kWave * NB);
  const int tok = (tile % a.t_tiles) * 64 * NB + 32 * NB * (wave >> 1) + 32 * c + (lane & 31);
  if (tok >= a.num_tokens) return;
  const f32x4* p =
      reinterpret_cast<const f32x4*>(a.part) + static_cast<int64_t>(tile) * kPerTile + in;
  const int64_t step = static_cast<int64_t>(a.tiles) * kPerTile;
  f32x4 s = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 8
  for (int z = 0; z < splits; ++z) s += p[z * step];
  T v[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) v[e] = Elem<T>::from_f(s[e]);
  // Row block f of the wave: weight rows 128 (f / 2) + 64 (wave & 1) + 32 (f & 1).
  const int64_t col = static_cast<int64_t>(tile / a.t_tiles) * 2 * kGI + kGI * (f >> 1) +
                      64 * (wave & 1) + 32 * (f & 1) + 8 * r4 + 4 * (lane >> 5);
  *reinterpret_cast<u32x2*>(a.out + tok * a.os + 2 * col) = __builtin_bit_cast(u32x2, v);
}

// ---------------------------------------------------------------------------
// Few tokens (decode-sized batches, T <= 128): the weights are the stream
// (671 MB at hidden 5120 x 2 x intermediate 32768) and the product is small,
// so the 256-token tile above spends most of its MFMAs on padding and runs
// one workgroup per CU.  The same kernel streams the gate and up rows of the
// SwiGLU product or 128 rows of a plain one (the down projection), and where
// the column tiles alone leave CUs idle it splits the contraction: fp32
// partials to a workspace, summed by split_sum_kernel (24 tokens, down
// projection 32768 x 5120: 53 us, 6.3 TB/s, against 160 us for the library's
// GEMM; 14336 x 4096 24 against 32; 8192 x 2048 11.4 against 14; gate/up 2048 x
// 8192 21.7 unsplit -> 17.4).  Here a workgroup owns 64 output columns (64 gate and
// the 64 up rows of the same columns) and all tokens (TB blocks of 32): its
// weight tile is 16 KB per 64-element k-step, so two workgroups share a CU
// and 512 of them cover intermediate 32768.  Tiles move with the same direct
// loads, swizzled 128-byte LDS rows and counted waits as above; weights go
// through a ring of three stages (two steps of lookahead), activations
// through two.  Wave w computes column half c = w & 1 (gate block c and up
// block 2 + c, 32 rows each).  With an even number of token blocks the
// other wave bit picks half of them (every k sub-step, epilogue straight from
// the registers); with one or three, it picks a k half of every step (two of
// the four 16-element sub-steps) for every token block, the k halves are
// summed through LDS and waves 0 and 1 apply the SiLU epilogue.
// Token rows past num_tokens read the last token's row; their outputs are
// not stored.
constexpr int kSCols = 64;                    // output columns per workgroup
constexpr int kSWTile = 2 * kSCols * kGRowB;  // weight tile per k-step: 128 rows, 16 KB
constexpr int kSWStages = 3;
constexpr int kRotStep = 5;  // k-steps between neighbouring tiles' starts

// s_waitcnt vmcnt(4) lgkmcnt(0): all of this wave's loads but the newest 4
// (its weight loads of the next step) have landed.
__device__ __forceinline__ void glu_small_wait() { __builtin_amdgcn_s_waitcnt(0x0074); }

template <typename T, int TB, bool kPart>
__global__ void __launch_bounds__(kGThreads) gate_up_silu_small_kernel(GluArgs a) {
  extern __shared__ __align__(16) char smem[];  // W stages, then x stages
  constexpr int kXTile = TB * 32 * kGRowB;
  constexpr bool kTokSplit = TB % 2 == 0;   // waves split the token blocks, else the k sub-steps
  constexpr int NB = kTokSplit ? TB / 2 : TB;  // token blocks per wave
  constexpr int NS = kTokSplit ? 4 : 2;        // 16-element sub-steps per wave and step
  const uint32_t lds0 = __builtin_amdgcn_readfirstlane(
      static_cast<uint32_t>(reinterpret_cast<uintptr_t>(smem)));
  const int i0 = blockIdx.x * kSCols;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;

  // Loads: weight rows 0-63 are the gate rows i0.., 64-127 the up rows;
  // wave w loads rows 32w .. 32w + 31 (four 1 KB loads of 8 rows) and the
  // activation loads w, w + 4, ... of the TB * 4 in a tile.
  const char* wbase = (wave < 2 ? a.wg : a.wu) + blockIdx.x * a.w_tile;
  const i32x4v wrs = buffer_rsrc(wbase, static_cast<int>(kSCols * a.ws));
  const i32x4v xrs = buffer_rsrc(a.x, static_cast<int>(a.num_tokens * a.xs));
  const int rw = 32 * (wave & 1) + (lane >> 3);  // weight row of load 0 within its matrix
  const int lc = (lane & 7) ^ (rw & 7);
  const int woff = rw * static_cast<int>(a.ws) + lc * 16;
  const int wstep = 8 * static_cast<int>(a.ws);
  int xoff[TB];
#pragma unroll
  for (int j = 0; j < TB; ++j) {
    const int R = 8 * (wave + 4 * j) + (lane >> 3);
    xoff[j] = min(R, a.num_tokens - 1) * static_cast<int>(a.xs) + lc * 16;
  }
  const uint32_t wdst = 1024 * 4 * wave;

  const int l32 = lane & 31, hb = lane >> 5;
  const int c = wave & 1, kh = wave >> 1;
  const int b0 = kTokSplit ? kh * NB : 0;  // first token block of this wave
  int rd[NS];
#pragma unroll
  for (int s = 0; s < NS; ++s)
    rd[s] = l32 * kGRowB + (((4 * hb + (kTokSplit ? s : 2 * kh + s)) ^ (l32 & 7)) << 4);

  f32x16 g[NB], u[NB];
#pragma unroll
  for (int b = 0; b < NB; ++b)
#pragma unroll
    for (int r = 0; r < 16; ++r) g[b][r] = u[b][r] = 0.f;

  // Steps k0 .. k0 + n - 1 of this split.
  const int k0 = kPart ? static_cast<int>(blockIdx.y) * a.k_per : 0;
  const int n = kPart ? min(a.ksteps - k0, a.k_per) : a.ksteps;
  // Row strides that are a multiple of 4 KB put the pieces that every
  // workgroup wants at one step on a few memory channels, so the tiles then
  // walk their steps from different starts (stride 64 KB, K 32768 x 5120, 24
  // tokens: 66.6 -> 53.2 us; stride 8 KB, gate/up 4096 x 14336: 47.8 -> 40.8).
  // Other strides spread by themselves, and one common order keeps the
  // activations in the L1 and L2 (stride 10 KB, gate/up 5120 x 32768: 100.8
  // against 103.1 us).
  const int rot = a.ws % 4096 == 0 ? static_cast<int>((blockIdx.x * kRotStep) % n) : 0;
  auto kstep = [&](int ks) {
    int s = min(ks, n - 1) + rot;
    if (s >= n) s -= n;
    return (k0 + s) * kGRowB;
  };
  auto load_w = [&](int ks, uint32_t dst) {
    const int kb = kstep(ks);
#pragma unroll
    for (int q = 0; q < 4; ++q) dma16_stream(wrs, woff, kb + q * wstep, dst + wdst + 1024 * q);
  };
  auto load_x = [&](int ks, uint32_t dst) {
    const int kb = kstep(ks);
#pragma unroll
    for (int j = 0; j < TB; ++j) dma16(xrs, xoff[j], kb, dst + 1024 * (wave + 4 * j));
  };
  const uint32_t xlds = lds0 + kSWStages * kSWTile;
  load_w(0, lds0);
  load_x(0, xlds);
  load_w(1, lds0 + kSWTile);
  for (int ks = 0; ks < n; ++ks) {
    glu_small_wait();
    __syncthreads();
    const char* cw = smem + (ks % kSWStages) * kSWTile;
    const char* cx = smem + kSWStages * kSWTile + (ks & 1) * kXTile;
    load_x(ks + 1, xlds + ((ks + 1) & 1) * kXTile);
    load_w(ks + 2, lds0 + ((ks + 2) % kSWStages) * kSWTile);
#pragma unroll
    for (int s = 0; s < NS; ++s) {
      const u32x4 ag = *reinterpret_cast<const u32x4*>(cw + (32 * c) * kGRowB + rd[s]);
      const u32x4 au = *reinterpret_cast<const u32x4*>(cw + (kSCols + 32 * c) * kGRowB + rd[s]);
#pragma unroll
      for (int b = 0; b < NB; ++b) {
        const u32x4 bx = *reinterpret_cast<const u32x4*>(cx + (32 * (b0 + b)) * kGRowB + rd[s]);
        g[b] = Elem<T>::mfma32x32x16(__builtin_bit_cast(typename Elem<T>::x8, ag),
                                     __builtin_bit_cast(typename Elem<T>::x8, bx), g[b]);
        u[b] = Elem<T>::mfma32x32x16(__builtin_bit_cast(typename Elem<T>::x8, au),
                                     __builtin_bit_cast(typename Elem<T>::x8, bx), u[b]);
      }
    }
  }
  // Every load has landed and every wave is done with the tiles before the
  // LDS is reused for the k-half sums.
  __builtin_amdgcn_s_waitcnt(0x0070);
  // This lane's four values of matrix m (0: first, 1: second), token block b
  // and column run r4 in the split's partials, laid out as the lanes hold them.
  auto part_at = [&](int m, int b, int r4) {
    const int64_t tile = static_cast<int64_t>(blockIdx.y) * gridDim.x + blockIdx.x;
    return reinterpret_cast<f32x4*>(a.part) +
           ((((tile * 2 + m) * 2 + c) * TB + b) * 4 + r4) * kWave + lane;
  };
  if constexpr (kTokSplit && kPart) {
#pragma unroll
    for (int b = 0; b < NB; ++b)
#pragma unroll
      for (int r4 = 0; r4 < 4; ++r4) {
        *part_at(0, b0 + b, r4) =
            f32x4{g[b][4 * r4], g[b][4 * r4 + 1], g[b][4 * r4 + 2], g[b][4 * r4 + 3]};
        *part_at(1, b0 + b, r4) =
            f32x4{u[b][4 * r4], u[b][4 * r4 + 1], u[b][4 * r4 + 2], u[b][4 * r4 + 3]};
      }
  } else if constexpr (kTokSplit) {
    // Lane holds token 32(b0 + b) + l32 and, of column half c, columns
    // 8 (r / 4) + 4 hb + r % 4.
#pragma unroll
    for (int b = 0; b < NB; ++b) {
      const int tok = 32 * (b0 + b) + l32;
      if (tok >= a.num_tokens) continue;
#pragma unroll
      for (int r4 = 0; r4 < 4; ++r4) {
        T v[4];
#pragma unroll
        for (int e = 0; e < 4; ++e)
          v[e] = Elem<T>::from_f(silu_mul1(g[b][4 * r4 + e], u[b][4 * r4 + e]));
        *reinterpret_cast<u32x2*>(a.out + static_cast<int64_t>(tok) * a.os +
                                  2 * (i0 + 32 * c + 8 * r4 + 4 * hb)) =
            __builtin_bit_cast(u32x2, v);
      }
    }
  } else {
    __syncthreads();
    constexpr int kVals = 2 * TB * 16;
    float* part = reinterpret_cast<float*>(smem) + c * kVals * kWave + lane;
    if (kh == 1) {
#pragma unroll
      for (int b = 0; b < TB; ++b)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          part[(32 * b + r) * kWave] = g[b][r];
          part[(32 * b + 16 + r) * kWave] = u[b][r];
        }
    }
    __syncthreads();
    if (kh == 1) return;
    // Lane holds token 32b + l32 and, of column half c, columns
    // 8 (r / 4) + 4 hb + r % 4.
#pragma unroll
    for (int b = 0; b < TB; ++b) {
      const int tok = 32 * b + l32;
#pragma unroll
      for (int r4 = 0; r4 < 4; ++r4) {
        if constexpr (kPart) {
          f32x4 pg, pu;
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const int r = 4 * r4 + e;
            pg[e] = g[b][r] + part[(32 * b + r) * kWave];
            pu[e] = u[b][r] + part[(32 * b + 16 + r) * kWave];
          }
          *part_at(0, b, r4) = pg;
          *part_at(1, b, r4) = pu;
          continue;
        }
        T v[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int r = 4 * r4 + e;
          v[e] = Elem<T>::from_f(silu_mul1(g[b][r] + part[(32 * b + r) * kWave],
                                           u[b][r] + part[(32 * b + 16 + r) * kWave]));
        }
        if (tok < a.num_tokens)
          *reinterpret_cast<u32x2*>(a.out + static_cast<int64_t>(tok) * a.os +
                                    2 * (i0 + 32 * c + 8 * r4 + 4 * hb)) =
              __builtin_bit_cast(u32x2, v);
      }
    }
  }
}

// Sums the splits' partials in a fixed order and rounds.  kSilu: the first and
// second matrix are the gate and up rows of the same 64 columns; else they are
// 128 columns of one product.  A thread owns four consecutive columns of one
// token, in the partials' own order, so a wave's reads are whole cache lines
// and the splits' loads are independent.
template <typename T, bool kSilu, int TB>
__global__ void __launch_bounds__(256) split_sum_kernel(GluArgs a, int splits) {
  constexpr int kPerM = 2 * TB * 4 * kWave;  // f32x4 of one matrix of a tile
  const int tile = blockIdx.x, in = blockIdx.y * 256 + threadIdx.x;
  const int m = kSilu ? 0 : in / kPerM;
  const int lane = in % kWave, r4 = (in / kWave) % 4;
  const int b = (in / (4 * kWave)) % TB, c = (in / (4 * kWave * TB)) % 2;
  const int tok = 32 * b + (lane & 31);
  if (tok >= a.num_tokens) return;
  const f32x4* p = reinterpret_cast<const f32x4*>(a.part) +
                   static_cast<int64_t>(tile) * 2 * kPerM + in;
  const int64_t step = static_cast<int64_t>(a.tiles) * 2 * kPerM;
  f32x4 s = {0.f, 0.f, 0.f, 0.f}, s2 = s;
#pragma unroll 8
  for (int z = 0; z < splits; ++z) {
    s += p[z * step];
    if constexpr (kSilu) s2 += p[z * step + kPerM];
  }
  T v[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) v[e] = Elem<T>::from_f(kSilu ? silu_mul1(s[e], s2[e]) : s[e]);
  const int64_t col = static_cast<int64_t>(tile) * (kSilu ? kSCols : 2 * kSCols) + kSCols * m +
                      32 * c + 8 * r4 + 4 * (lane >> 5);
  *reinterpret_cast<u32x2*>(a.out + tok * a.os + 2 * col) = __builtin_bit_cast(u32x2, v);
}

// The few-token product over `splits` ranges of a.k_per k-steps.  kSilu: gate
// and up rows with the SwiGLU epilogue (in the product kernel itself without
// partials); else one plain product.
template <typename T, bool kSilu, int TB>
int launch_small_tb(const GluArgs& a, int splits, hipStream_t stream) {
  const size_t lds = static_cast<size_t>(kSWStages) * kSWTile + 2 * TB * 32 * kGRowB;
  if (!a.part) {
    hipLaunchKernelGGL((gate_up_silu_small_kernel<T, TB, false>), dim3(a.tiles), dim3(kGThreads),
                       lds, stream, a);
    return check_launch("gate_up_silu_small_kernel");
  }
  hipLaunchKernelGGL((gate_up_silu_small_kernel<T, TB, true>), dim3(a.tiles, splits),
                     dim3(kGThreads), lds, stream, a);
  const int st = check_launch("gate_up_silu_small_kernel");
  if (st) return st;
  hipLaunchKernelGGL((split_sum_kernel<T, kSilu, TB>), dim3(a.tiles, (kSilu ? 2 : 4) * TB),
                     dim3(256), 0, stream, a, splits);
  return check_launch("split_sum_kernel");
}

template <typename T, bool kSilu>
int launch_small(const GluArgs& a, int splits, hipStream_t stream) {
  switch ((a.num_tokens + 31) / 32) {
    case 1: return launch_small_tb<T, kSilu, 1>(a, splits, stream);
    case 2: return launch_small_tb<T, kSilu, 2>(a, splits, stream);
    case 3: return launch_small_tb<T, kSilu, 3>(a, splits, stream);
    default: return launch_small_tb<T, kSilu, 4>(a, splits, stream);
  }
}

// Splits of the contraction for `tiles` column tiles of `ksteps` k-steps: up to
// one workgroup per CU (256 CUs), each with at least kSplitMinSteps steps; its
// three-stage ring keeps a CU's share of HBM busy, and more splits cost more
// partials than they gain (linear, two workgroups per CU against one: 32768 x
// 5120, 24 tokens 56.2 against 53.2 us, 14336 x 4096, 128 tokens 42.5 against
// 35.7; at least 4 steps against 8: 8192 x 2048, 24 tokens 16.4 against 11.4).
constexpr int kSplitGroups = 256;
constexpr int kSplitMinSteps = 8;

int split_plan(int tiles, int ksteps, int* k_per) {
  const int s = std::max(1, std::min(kSplitGroups / std::max(1, tiles), ksteps / kSplitMinSteps));
  *k_per = (ksteps + s - 1) / s;
  return (ksteps + *k_per - 1) / *k_per;
}

size_t split_bytes(int tiles, int splits, int num_tokens) {
  return static_cast<size_t>(splits) * tiles * 2 * kSCols * ((num_tokens + 31) / 32 * 32) *
         sizeof(float);
}

// 32-token blocks per wave (2, 3 or 4) for a batch over `cols` column tiles: the
// least rounds of one workgroup per CU (256) times a round's time, 17, 21 and 27 for
// NB = 2, 3 and 4: a k-step takes 0.98, 1.22 and 1.57 us where there are several
// rounds.  300 tokens, 4096 x 14336: 104.9 us at NB = 4, 84.8 at 3; 192 tokens 93.4,
// 65.9 at 2; 2104 tokens, 5120 x 32768: 1170, 1151 at 3.  On the other side, which
// rounds costing NB + 1/2 gave to NB = 2: 1024 tokens, 8192 x 28672 809 us at NB = 4,
// 881 at 2; 3584 x 18944 267, 282.
inline int wide_blocks(int num_tokens, int cols) {
  constexpr int kRound[] = {0, 0, 17, 21, 27};
  int best = 4, cost = INT32_MAX;
  for (int nb = 4; nb >= 2; --nb) {
    const int64_t tiles = static_cast<int64_t>((num_tokens + 64 * nb - 1) / (64 * nb)) * cols;
    const int c = static_cast<int>((tiles + 255) / 256) * kRound[nb];
    if (c < cost) {
      cost = c;
      best = nb;
    }
  }
  return best;
}

template <typename T, int NB>
int launch_gate_up_silu_nb(GluArgs a, hipStream_t stream) {
  const int cols = a.tiles;
  a.t_tiles = (a.num_tokens + 64 * NB - 1) / (64 * NB);
  a.tiles = a.t_tiles * cols;
  const int grid = (a.tiles + kGXcds - 1) / kGXcds * kGXcds;
  // Weight tiles read by at most four token tiles stream with the hint.
  if (a.t_tiles <= 4)
    hipLaunchKernelGGL((gate_up_silu_kernel<T, true, NB, false>), dim3(grid), dim3(kGThreads), 0,
                       stream, a);
  else
    hipLaunchKernelGGL((gate_up_silu_kernel<T, false, NB, false>), dim3(grid), dim3(kGThreads), 0,
                       stream, a);
  return check_launch("gate_up_silu_kernel");
}

// a.tiles: column tiles.
template <typename T>
int launch_gate_up_silu(const GluArgs& a, hipStream_t stream) {
  switch (wide_blocks(a.num_tokens, a.tiles)) {
    case 2: return launch_gate_up_silu_nb<T, 2>(a, stream);
    case 3: return launch_gate_up_silu_nb<T, 3>(a, stream);
    default: return launch_gate_up_silu_nb<T, 4>(a, stream);
  }
}

// How vaa_linear runs a product: on the few-token kernel (nb = 0) or the wide
// one with nb blocks of 32 tokens per wave, over `splits` ranges of k_per steps.
struct LinearPlan {
  int nb, splits, k_per;
  size_t bytes;  // workspace; 0: shape not supported
};

// The wide kernel up to kWideTokens tokens: above, the library's GEMM is ahead
// (us, library / this: 512 tokens, 32768 x 5120 289 / 181, 14336 x 4096 91 / 70,
// 8192 x 2048 35 / 31; 1024 tokens 395 / 311, 132 / 117, 53 / 46; 2104
// tokens 553 / 643, 213 / 256, 83 / 88).  Short contractions and wide outputs are
// the library's below that too (kernels.linear_pays).
constexpr int kWideTokens = 1024;

LinearPlan linear_plan(int num_tokens, int ksteps, int out_features) {
  LinearPlan best{0, 1, ksteps, 0};
  if (num_tokens <= kSmallTokens) {
    const int tiles = out_features / (2 * kSCols);
    best.splits = split_plan(tiles, ksteps, &best.k_per);
    best.bytes = split_bytes(tiles, best.splits, num_tokens);
    return best;
  }
  if (num_tokens > kWideTokens || out_features % (2 * kGI) != 0) return best;
  // One workgroup per CU as far as splits of at least kSplitMinSteps steps
  // allow.  Cost in ns: 0.3 us (NB + 1.2) a step and the partials written and
  // read at 6 TB/s, as measured.
  int64_t cost = INT64_MAX;
  for (int nb = 4; nb >= 2; --nb) {
    const int64_t tiles = static_cast<int64_t>((num_tokens + 64 * nb - 1) / (64 * nb)) *
                          (out_features / (2 * kGI));
    const int64_t want = std::max<int64_t>(
        1, std::min<int64_t>(256 / tiles, ksteps / kSplitMinSteps));
    const int k_per = static_cast<int>((ksteps + want - 1) / want);
    const int splits = (ksteps + k_per - 1) / k_per;
    const int64_t bytes = tiles * splits * (64 * nb) * (2 * kGI) * 4;
    const int64_t c = (tiles * splits + 255) / 256 * k_per * (300 * nb + 360) + bytes / 3000;
    if (c < cost) {
      cost = c;
      best = LinearPlan{nb, splits, k_per, static_cast<size_t>(bytes)};
    }
  }
  return best;
}

// Plain product on the wide kernel, split over `splits` ranges of k-steps.
template <typename T, int NB>
int launch_wide_nb(GluArgs a, int splits, hipStream_t stream) {
  const int cols = a.tiles;
  a.t_tiles = (a.num_tokens + 64 * NB - 1) / (64 * NB);
  a.tiles = a.t_tiles * cols;
  const int grid = (a.tiles * splits + kGXcds - 1) / kGXcds * kGXcds;
  hipLaunchKernelGGL((gate_up_silu_kernel<T, false, NB, true>), dim3(grid), dim3(kGThreads), 0,
                     stream, a);
  const int st = check_launch("gate_up_silu_kernel");
  if (st) return st;
  hipLaunchKernelGGL((wide_sum_kernel<T, NB>), dim3(a.tiles, 16 * NB), dim3(256), 0, stream, a,
                     splits);
  return check_launch("wide_sum_kernel");
}

}  // namespace
}  // namespace vaa

using namespace vaa;

namespace vaa {
namespace {

// The body of vaa_gate_up_silu, with the split's workspace (null: none).
int gate_up_silu_impl(const char* what, const uint16_t* x, int64_t x_stride,
                      const uint16_t* w_gate, const uint16_t* w_up, int64_t w_stride,
                      uint16_t* output, int64_t output_stride, int num_tokens, int hidden_size,
                      int intermediate_size, int dtype, void* workspace, size_t workspace_bytes,
                      void* stream) {
  if (!valid_dtype(dtype)) return fail(VAA_ERR_UNSUPPORTED, "%s: dtype=%d", what, dtype);
  if (num_tokens < 0 || hidden_size <= 0 || intermediate_size <= 0)
    return fail(VAA_ERR_INVALID_ARG, "%s: num_tokens=%d hidden_size=%d intermediate_size=%d",
                what, num_tokens, hidden_size, intermediate_size);
  if (hidden_size % kGK != 0 || intermediate_size % kGI != 0)
    return fail(VAA_ERR_UNSUPPORTED,
                "%s: hidden_size=%d must be a multiple of %d and intermediate_size=%d of %d",
                what, hidden_size, kGK, intermediate_size, kGI);
  if (num_tokens == 0) return VAA_OK;
  if (!x || !w_gate || !w_up || !output) return fail(VAA_ERR_INVALID_ARG, "%s: null pointer", what);
  if (x_stride < hidden_size || w_stride < hidden_size || output_stride < intermediate_size ||
      x_stride % 8 != 0 || w_stride % 8 != 0 || output_stride % 8 != 0)
    return fail(VAA_ERR_INVALID_ARG,
                "%s: strides x=%lld w=%lld out=%lld (x, w: multiples of 8 >= hidden_size; out: "
                "a multiple of 8 >= intermediate_size)",
                what, (long long)x_stride, (long long)w_stride, (long long)output_stride);
  if (!aligned16(x) || !aligned16(w_gate) || !aligned16(w_up) || !aligned16(output))
    return fail(VAA_ERR_INVALID_ARG, "%s: x, weights and output must be 16-byte aligned", what);
  GluArgs a;
  a.x = reinterpret_cast<const char*>(x);
  a.wg = reinterpret_cast<const char*>(w_gate);
  a.wu = reinterpret_cast<const char*>(w_up);
  a.out = reinterpret_cast<char*>(output);
  a.xs = 2 * x_stride;
  a.ws = 2 * w_stride;
  a.os = 2 * output_stride;
  a.num_tokens = num_tokens;
  a.ksteps = hidden_size / kGK;
  a.t_tiles = 1;
  const int64_t tiles =
      static_cast<int64_t>((num_tokens + 63) / 64) * (intermediate_size / kGI);
  // Load offsets and buffer ranges are 31-bit: activation rows from x,
  // weight rows from the workgroup's first row.
  if (tiles > (1 << 30) || static_cast<int64_t>(num_tokens) * a.xs >= (int64_t(1) << 31) ||
      static_cast<int64_t>(kGI) * a.ws >= (int64_t(1) << 31))
    return fail(VAA_ERR_UNSUPPORTED, "%s: problem too large", what);
  a.tiles = intermediate_size / kGI;
  a.k_per = a.ksteps;
  a.w_tile = (num_tokens <= kSmallTokens ? kSCols : kGI) * a.ws;
  a.part = nullptr;
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (num_tokens <= kSmallTokens) {
    a.tiles = intermediate_size / kSCols;
    int splits = 1;
    if (workspace) {
      splits = split_plan(a.tiles, a.ksteps, &a.k_per);
      if (splits > 1) {
        const size_t need = split_bytes(a.tiles, splits, num_tokens);
        if (workspace_bytes < need || !aligned16(workspace))
          return fail(VAA_ERR_WORKSPACE,
                      "%s: workspace of %zu bytes (16-byte aligned) needed, got %zu", what, need,
                      workspace_bytes);
        a.part = static_cast<float*>(workspace);
      }
    }
    return dtype == VAA_DTYPE_F16 ? launch_small<f16, true>(a, splits, s)
                                  : launch_small<bf16, true>(a, splits, s);
  }
  return dtype == VAA_DTYPE_F16 ? launch_gate_up_silu<f16>(a, s) : launch_gate_up_silu<bf16>(a, s);
}

}  // namespace
}  // namespace vaa

extern "C" int vaa_gate_up_silu(const uint16_t* x, int64_t x_stride, const uint16_t* w_gate,
                                const uint16_t* w_up, int64_t w_stride, uint16_t* output,
                                int64_t output_stride, int num_tokens, int hidden_size,
                                int intermediate_size, int dtype, void* stream) {
  return gate_up_silu_impl("vaa_gate_up_silu", x, x_stride, w_gate, w_up, w_stride, output,
                           output_stride, num_tokens, hidden_size, intermediate_size, dtype,
                           nullptr, 0, stream);
}

extern "C" size_t vaa_gate_up_silu_workspace_size(int num_tokens, int hidden_size,
                                                  int intermediate_size) {
  if (num_tokens <= 0 || num_tokens > kSmallTokens || hidden_size <= 0 || hidden_size % kGK ||
      intermediate_size <= 0 || intermediate_size % kGI)
    return 0;
  int k_per = 0;
  const int tiles = intermediate_size / kSCols;
  const int splits = split_plan(tiles, hidden_size / kGK, &k_per);
  return splits > 1 ? split_bytes(tiles, splits, num_tokens) : 0;
}

extern "C" int vaa_gate_up_silu_split(const uint16_t* x, int64_t x_stride, const uint16_t* w_gate,
                                      const uint16_t* w_up, int64_t w_stride, uint16_t* output,
                                      int64_t output_stride, int num_tokens, int hidden_size,
                                      int intermediate_size, int dtype, void* workspace,
                                      size_t workspace_bytes, void* stream) {
  const char* what = "vaa_gate_up_silu_split";
  if (!workspace && vaa_gate_up_silu_workspace_size(num_tokens, hidden_size, intermediate_size))
    return fail(VAA_ERR_WORKSPACE, "%s: null workspace", what);
  return gate_up_silu_impl(what, x, x_stride, w_gate, w_up, w_stride, output, output_stride,
                           num_tokens, hidden_size, intermediate_size, dtype, workspace,
                           workspace_bytes, stream);
}

extern "C" size_t vaa_linear_workspace_size(int num_tokens, int in_features, int out_features) {
  if (num_tokens <= 0 || in_features <= 0 || in_features % kGK || out_features <= 0 ||
      out_features % (2 * kSCols))
    return 0;
  return linear_plan(num_tokens, in_features / kGK, out_features).bytes;
}

extern "C" int vaa_linear(const uint16_t* x, int64_t x_stride, const uint16_t* w, int64_t w_stride,
                          uint16_t* output, int64_t output_stride, int num_tokens,
                          int in_features, int out_features, int dtype, void* workspace,
                          size_t workspace_bytes, void* stream) {
  const char* what = "vaa_linear";
  if (!valid_dtype(dtype)) return fail(VAA_ERR_UNSUPPORTED, "%s: dtype=%d", what, dtype);
  if (num_tokens < 0 || in_features <= 0 || out_features <= 0)
    return fail(VAA_ERR_INVALID_ARG, "%s: num_tokens=%d in_features=%d out_features=%d", what,
                num_tokens, in_features, out_features);
  if (num_tokens == 0) return VAA_OK;
  const size_t need = vaa_linear_workspace_size(num_tokens, in_features, out_features);
  if (!need)
    return fail(VAA_ERR_UNSUPPORTED,
                "%s: num_tokens=%d (at most %d), in_features=%d (a multiple of %d), "
                "out_features=%d (a multiple of %d, of %d above %d tokens)",
                what, num_tokens, kWideTokens, in_features, kGK, out_features, 2 * kSCols,
                2 * kGI, kSmallTokens);
  if (!x || !w || !output) return fail(VAA_ERR_INVALID_ARG, "%s: null pointer", what);
  if (x_stride < in_features || w_stride < in_features || output_stride < out_features ||
      x_stride % 8 || w_stride % 8 || output_stride % 8)
    return fail(VAA_ERR_INVALID_ARG, "%s: strides x=%lld w=%lld out=%lld", what,
                (long long)x_stride, (long long)w_stride, (long long)output_stride);
  if (!aligned16(x) || !aligned16(w) || !aligned16(output))
    return fail(VAA_ERR_INVALID_ARG, "%s: x, weights and output must be 16-byte aligned", what);
  const LinearPlan plan = linear_plan(num_tokens, in_features / kGK, out_features);
  const int rows = plan.nb ? kGI : kSCols;  // weight rows of one half of a tile
  GluArgs a;
  a.x = reinterpret_cast<const char*>(x);
  a.wg = reinterpret_cast<const char*>(w);
  a.xs = 2 * x_stride;
  a.ws = 2 * w_stride;
  a.os = 2 * output_stride;
  a.wu = a.wg + rows * a.ws;
  a.w_tile = 2 * rows * a.ws;
  a.out = reinterpret_cast<char*>(output);
  a.num_tokens = num_tokens;
  a.ksteps = in_features / kGK;
  a.k_per = plan.k_per;
  a.t_tiles = 1;
  a.tiles = out_features / (2 * rows);
  if (num_tokens * a.xs >= (int64_t(1) << 31) || rows * a.ws >= (int64_t(1) << 31))
    return fail(VAA_ERR_UNSUPPORTED, "%s: problem too large", what);
  if (!workspace || workspace_bytes < need || !aligned16(workspace))
    return fail(VAA_ERR_WORKSPACE, "%s: workspace of %zu bytes (16-byte aligned) needed, got %zu",
                what, need, workspace ? workspace_bytes : static_cast<size_t>(0));
  a.part = static_cast<float*>(workspace);
  hipStream_t s = static_cast<hipStream_t>(stream);
  const bool f = dtype == VAA_DTYPE_F16;
  switch (plan.nb) {
    case 0:
      return f ? launch_small<f16, false>(a, plan.splits, s)
               : launch_small<bf16, false>(a, plan.splits, s);
    case 2:
      return f ? launch_wide_nb<f16, 2>(a, plan.splits, s)
               : launch_wide_nb<bf16, 2>(a, plan.splits, s);
    case 3:
      return f ? launch_wide_nb<f16, 3>(a, plan.splits, s)
               : launch_wide_nb<bf16, 3>(a, plan.splits, s);
    default:
      return f ? launch_wide_nb<f16, 4>(a, plan.splits, s)
               : launch_wide_nb<bf16, 4>(a, plan.splits, s);
  }
}
