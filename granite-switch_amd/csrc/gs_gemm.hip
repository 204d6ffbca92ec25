// Dense bf16 GEMM C[M,N] = A[M,K] . B[N,K]^T for gfx950 -- the one GEMM of
// the reference's vLLM layer, x_ext = x . w_ext^T, where w_ext stacks the
// base weight and every adapter's lora_A rows, so one pass gives the base
// output and every shrink (src/granite_switch/vllm/core/lora.py:544;
// src/granite_switch/kernels/switch_lora_kernel.py:134-163).
//
// Both operands are K-contiguous rows, the layout MFMA reads directly.  A
// workgroup of 8 waves owns a 256 x 256 tile of C, accumulated in fp32, which
// gives 128 FLOP per byte moved from the L2 into the CU.  Tiles are numbered
// in groups of 8 tile rows (consecutive workgroups share B columns and A rows
// in the L2), and each XCD takes a contiguous range of that order, so the
// tiles running together on one XCD share its L2.  Partial tiles clamp their
// loads to the last row and mask their stores.
//
// Three kernels: for K % 64 == 0 the k-tiles go from global memory
// straight into LDS and the two waves of a SIMD alternate between reading and
// multiplying (gemm_bf16_tn_pingpong_kernel), or, for few tiles, smaller ones
// split K over their waves (gemm_bf16_tn_stream_kernel); otherwise they are loaded into
// registers, zero-filled past K, and written to padded LDS rows
// (gemm_bf16_tn_kernel).
//
// Times in this file: graph replays over buffer sets that together exceed the
// 256 MB MALL, so the operands come from HBM.  One set, its weights in the MALL
// (as bench.py --layer-gemm times it), is faster for few rows: 256 x 7296 x 4096
// 22.5 against 29.3 us, 16 x 7296 x 4096 11.5 against 13.7.
#include <stdarg.h>

#include <algorithm>
#include <set>
#include <type_traits>
#include <utility>
#include <vector>

#include "gs_addr.h"
#include "gs_common.h"

namespace gs {

namespace {

constexpr int kGBM = 256;                       // C rows per workgroup
constexpr int kGBN = 256;                       // C columns per workgroup
constexpr int kGBK = 64;                        // k per tile
constexpr int kGRowBytes = kGBK * 2;            // bytes of one operand row per k-tile
constexpr int kGLd = kGRowBytes + 16;           // padded LDS row stride
constexpr int kGStage = (kGBM + kGBN) * kGLd;   // one k-tile of A and B in LDS
constexpr int kGLds = 2 * kGStage;              // double-buffered
constexpr int kGGroup = 8;                      // tile rows per group of the tile order
static_assert(kGBM == kGBN, "A and B tiles are staged with the same thread mapping");

struct GemmParams {
  const char* a;
  int64_t lda;            // elements
  const char* b;
  int64_t ldb;
  uint16_t* c;
  int64_t ldc;
  int M, N, K;
  int tiles_m, tiles_n;
  int full_rows;          // ping-pong form: tile rows of 256, before
  int half_rows;          // those of 128
};

// C's rows start at 16 bytes: a lane stores 8 consecutive columns at once.
__device__ __forceinline__ bool wide_rows(const GemmParams& p) {
  return p.ldc % 8 == 0 && (reinterpret_cast<uintptr_t>(p.c) & 15) == 0;
}

// WM x WN waves over k-tiles of 64 in two LDS stages (one barrier per k-tile);
// wave (wm, wn) owns rows wm*(256/WM) and columns wn*(256/WN)
// of the tile as MI x NJ blocks of 32 x 32.
template <bool KTAIL, int WM, int WN>
__global__ __launch_bounds__(64 * WM * WN) void gemm_bf16_tn_kernel(GemmParams p) {
  constexpr int kGThreads = 64 * WM * WN;
  constexpr int kGPieces = kGBM * (kGRowBytes / 16) / kGThreads;   // 16-byte pieces per thread and operand
  constexpr int kGRowStep = kGThreads / (kGRowBytes / 16);         // rows between a thread's pieces
  constexpr int MI = kGBM / WM / 32;
  constexpr int NJ = kGBN / WN / 32;
  extern __shared__ __align__(16) char smem[];

  // tile of this workgroup: XCD x = id % 8 takes tiles [x*per, (x+1)*per)
  int tm, tn;
  if (!addr::gemm_tile(static_cast<int>(blockIdx.x), p.tiles_m, p.tiles_n, kGGroup, tm, tn)) return;

  const int tid = threadIdx.x;
  // global -> LDS mapping: 8 consecutive threads move one row's 128 bytes
  const int lrow = tid >> 3;
  const int lpc = (tid & 7) * 16;
  const int kp = (tid & 7) * 8;                 // this thread's k within a tile
  const char* ga[kGPieces];
  const char* gb[kGPieces];
#pragma unroll
  for (int j = 0; j < kGPieces; ++j) {
    const int ra = addr::gemm_row(tm * kGBM + lrow + j * kGRowStep, p.M);
    const int rb = addr::gemm_row(tn * kGBN + lrow + j * kGRowStep, p.N);
    ga[j] = p.a + static_cast<int64_t>(ra) * p.lda * 2;
    gb[j] = p.b + static_cast<int64_t>(rb) * p.ldb * 2;
  }
  u32x4 va[kGPieces], vb[kGPieces];
  // loads from clamped in-bounds addresses, masked afterwards (K % 8 == 0, so
  // a 16-byte piece is entirely inside or entirely past K; a piece past K
  // re-reads the row's first 16 bytes)
  auto gload = [&](int kt) {
    const bool ok = !KTAIL || kt * kGBK + kp < p.K;
    const int64_t off = ok ? static_cast<int64_t>(kt) * kGRowBytes + lpc : 0;
#pragma unroll
    for (int j = 0; j < kGPieces; ++j) {
      va[j] = ld16(ga[j] + off);
      vb[j] = ld16(gb[j] + off);
    }
    if constexpr (KTAIL) {
#pragma unroll
      for (int j = 0; j < kGPieces; ++j) {
        va[j] = sel16(ok, va[j]);
        vb[j] = sel16(ok, vb[j]);
      }
    }
  };
  auto sstore = [&](int buf) {
    char* sa = smem + buf * kGStage;
    char* sb = sa + kGBM * kGLd;
#pragma unroll
    for (int j = 0; j < kGPieces; ++j) {
      st16(sa + (lrow + j * kGRowStep) * kGLd + lpc, va[j]);
      st16(sb + (lrow + j * kGRowStep) * kGLd + lpc, vb[j]);
    }
  };

  const int wave = tid >> 6;
  const int l = tid & 63;
  const int wm = wave / WN;
  const int wn = wave % WN;
  const int i32 = l & 31;
  const int h = l >> 5;
  f32x16 acc[MI][NJ];
#pragma unroll
  for (int i = 0; i < MI; ++i)
#pragma unroll
    for (int j = 0; j < NJ; ++j) acc[i][j] = f32x16{};

  // MFMA operands: lane l reads row (l % 32) of a 32-row block, k 8*(l/32) .. +7
  // of each 16-k step
  auto compute = [&](int buf) {
    const char* sa = smem + buf * kGStage + (wm * MI * 32 + i32) * kGLd + h * 16;
    const char* sb = smem + buf * kGStage + kGBM * kGLd + (wn * NJ * 32 + i32) * kGLd + h * 16;
#pragma unroll
    for (int kk = 0; kk < kGBK / 16; ++kk) {
      u32x4 af[MI], bf[NJ];
#pragma unroll
      for (int i = 0; i < MI; ++i) af[i] = *reinterpret_cast<const u32x4*>(sa + i * 32 * kGLd + kk * 32);
#pragma unroll
      for (int j = 0; j < NJ; ++j) bf[j] = *reinterpret_cast<const u32x4*>(sb + j * 32 * kGLd + kk * 32);
#pragma unroll
      for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int j = 0; j < NJ; ++j) acc[i][j] = mfma32_bf16(af[i], bf[j], acc[i][j]);
    }
  };

  const int nk = (p.K + kGBK - 1) / kGBK;
  gload(0);
  sstore(0);
  lds_barrier();
  for (int kt = 0; kt < nk; ++kt) {
    // the next tile's loads go out before this tile's MFMAs (the scheduling
    // barrier keeps them there); the last iteration re-reads its own tile into
    // the idle buffer
    gload(min(kt + 1, nk - 1));
    __builtin_amdgcn_sched_barrier(0);
    compute(kt & 1);
    sstore((kt + 1) & 1);
    lds_barrier();
  }

  // lane (i32, h) holds column i32 and rows mfma32_row(v, l) of each 32 x 32 block
  const int row0 = tm * kGBM + wm * MI * 32;
  const int col0 = tn * kGBN + wn * NJ * 32 + i32;
#pragma unroll
  for (int i = 0; i < MI; ++i) {
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
      const int col = col0 + j * 32;
      if (col >= p.N) continue;
#pragma unroll
      for (int v = 0; v < 16; ++v) {
        const int row = row0 + i * 32 + mfma32_row(v, l);
        if (row < p.M) p.c[static_cast<int64_t>(row) * p.ldc + col] = f32_to_bf16_bits(acc[i][j][v]);
      }
    }
  }
}

// ---------------------------------------------------------------------------
// The form for K % 64 == 0: the k-tiles travel from global memory
// straight into LDS, and the two waves of a SIMD take turns on its matrix core.
//
// Tile: 256 x 256, wave (wm, wn) of 2 x 4 owns rows half*128 + wm*64 + 0..63
// (half = 0, 1) and columns wn*64 + 0..63, as four quadrants of 64 x 32 (row
// half, column half).  Per k-tile of 64 a wave runs four phases, one quadrant
// each: 16 v_mfma_f32_16x16x32_bf16, 256 matrix-core clocks.  A phase is a
// memory part (LDS reads of the operands that the quadrant newly needs, the
// transfers of one half-operand of k-tile kt+2) and a matrix part, with a
// barrier after each; waves 4-7 run one part behind waves 0-3, so on every
// SIMD one wave multiplies while the other reads.
//
// LDS: two stages of [A half 0, A half 1, B half 0, B half 1], 128 rows of 128
// bytes each.  Schedule of k-tile kt (reads | transfers issued):
//   P1  A0(kt)    | B0(kt+2)      quadrant (0, 0)
//   P2  B1(kt)    | A0(kt+2)      quadrant (0, 1)
//   P3  A1(kt)    | B1(kt+2)      quadrant (1, 0)
//   P4  B0(kt+1)  | A1(kt+2)      quadrant (1, 1)
// A half is overwritten one phase after its last read, by both wave groups'
// barriers (a memory part waits for its own reads before its barrier).  A
// wave has two transfers per phase in flight and waits, at the end of each
// memory part, until those older than six phases have landed: exactly the half
// that the next phase reads.  So a transfer has ~3000 clocks to arrive.
//
// Tile rows of 128 run the two phases of row half 0 only (HALF), at 0.7 of the
// time; those tiles come last in every XCD's range.  As many tile rows are such
// as shorten the last, part-filled round of tiles -- all of them, where 256-row
// tiles would leave most CUs idle (pick_gemm).  A last tile row of at most 128
// rows is a 256-row one where that round is no shorter without it.
//
// Bound by LDS (64 KB of transfers in at 64 bytes per clock, 192 KB of operand
// reads at 128: 2560 clocks per k-tile against 2048 of MFMAs; 1.1 us measured)
// and, with every CU busy, by the clock that the power limit leaves.
//
// A transfer moves 1 KB: 8 LDS rows x 128 bytes, every request one whole cache
// line.  It fills LDS contiguously, so bank spreading comes from an XOR
// swizzle: the 16-byte piece p of row r sits at position p ^ addr::lds_swz(r),
// which puts the operand reads of 16 consecutive rows at one k in distinct
// banks.  B rows are staged in the order (addr::gemm_b_row) that gives a lane
// 8 consecutive columns of its C row, stored as 16 bytes.
//
// Measured: 4144 x 27136 x 4096 890 -> 658 us (1400 TFLOP/s), 8192 x 26368 x
// 4096 1487 -> 1178 (1502), against the form it replaces (one barrier per
// k-tile, all waves reading, then all multiplying; 1 transfer stage in flight).
// Without a pause between calls the power limit takes 5 to 8 % of that.
// ---------------------------------------------------------------------------
constexpr int kPBK = 64;                        // k per tile
constexpr int kPRow = kPBK * 2;                 // bytes of one operand row per tile (one cache line)
constexpr int kPHalf = 128 * kPRow;             // one half-operand of one stage
constexpr int kPStage = 4 * kPHalf;             // A0, A1, B0, B1
constexpr int64_t kPMaxLd = int64_t(1) << 22;   // a tile's rows stay within 32-bit byte offsets
constexpr int kPOutRow = 64 * 2 + 16;           // a wave's 64 x 64 results in LDS (rows 16-byte aligned, banks spread)
constexpr int kPOutWave = 64 * kPOutRow;
static_assert(8 * kPOutWave <= 2 * kPStage, "the results fit the operand stages");

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));

__device__ __forceinline__ f32x4 mfma16_bf16(u32x4 a, u32x4 b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, a), __builtin_bit_cast(bf16x8_t, b), c,
                                                 0, 0, 0);
}

// Transfer of 16 bytes per lane from base + off (a lane's byte offset) to LDS
// at dst + 16 * lane; counts in vmcnt (see dma16).
__device__ __forceinline__ void dma16_at(const char* base, uint32_t off, uint32_t dst) {
  asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(off), "s"(base), "s"(dst)
               : "memory", "m0");
}

// s_waitcnt for "vmcnt <= n and lgkmcnt == 0"
constexpr int wait_vm_lds(int n) { return (n & 15) | (7 << 4) | ((n >> 4) << 14); }

template <bool HALF>
__device__ __forceinline__ void gemm_tile_pingpong(const GemmParams& p, char* smem, int first_row, int tn) {
  constexpr int NA = HALF ? 1 : 2;              // row halves
  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l = tid & 63;
  const int wm = wave >> 2;
  const int wn = wave & 3;
  const int nk = p.K / kPBK;
  const uint32_t lds0 = static_cast<uint32_t>(reinterpret_cast<uintptr_t>((lds_ptr_t)(smem)));

  // transfers j = 0, 1 of this wave and half-operand: LDS rows 8 * (2 * wave + j) on
  uint32_t offa[NA][2], offb[2][2];
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const int r = 8 * (2 * wave + j) + (l >> 3);
    const uint32_t piece = addr::gemm_piece(l, r) * 16;
#pragma unroll
    for (int h = 0; h < NA; ++h)
      offa[h][j] = static_cast<uint32_t>((addr::gemm_row(first_row + h * 128 + r, p.M) - first_row) * p.lda * 2) + piece;
#pragma unroll
    for (int h = 0; h < 2; ++h)
      offb[h][j] = static_cast<uint32_t>((addr::gemm_row(tn * kGBN + addr::gemm_b_row(r, h), p.N) - tn * kGBN) * p.ldb * 2) + piece;
  }
  const char* const basea = p.a + static_cast<int64_t>(first_row) * p.lda * 2;
  const char* const baseb = p.b + static_cast<int64_t>(tn) * kGBN * p.ldb * 2;
  const uint32_t dst0 = lds0 + wave * 2048;
  auto issue_a = [&](int h, int kt) {
    const char* g = basea + static_cast<int64_t>(min(kt, nk - 1)) * kPRow;
    const uint32_t d = dst0 + (kt & 1) * kPStage + h * kPHalf;
    dma16_at(g, offa[HALF ? 0 : h][0], d);
    dma16_at(g, offa[HALF ? 0 : h][1], d + 1024);
  };
  auto issue_b = [&](int h, int kt) {
    const char* g = baseb + static_cast<int64_t>(min(kt, nk - 1)) * kPRow;
    const uint32_t d = dst0 + (kt & 1) * kPStage + (2 + h) * kPHalf;
    dma16_at(g, offb[h][0], d);
    dma16_at(g, offb[h][1], d + 1024);
  };

  f32x4 acc[NA][2][4][2];                       // [row half][column half][16-row block][16-column block]
#pragma unroll
  for (int h = 0; h < NA; ++h)
#pragma unroll
    for (int c = 0; c < 2; ++c)
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) acc[h][c][i][j] = f32x4{0.f, 0.f, 0.f, 0.f};

  // operand reads: lane l reads row l % 16 of a block, k 8 * (l / 16) .. + 7 of each 32
  const int pos = ((l >> 4) ^ addr::lds_swz(l & 15)) * 16;
  const char* const ra = smem + (wm * 64 + (l & 15)) * kPRow;
  const char* const rb = smem + 2 * kPHalf + (wn * 32 + (l & 15)) * kPRow;
  u32x4 fa[4][2], fb[2][2][2];                  // [16-row block][k step], [column half][16-column block][k step]
  auto read_a = [&](int h, int st) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      fa[i][0] = ld16(ra + st * kPStage + h * kPHalf + i * 16 * kPRow + pos);
      fa[i][1] = ld16(ra + st * kPStage + h * kPHalf + i * 16 * kPRow + (pos ^ 64));
    }
  };
  auto read_b = [&](int h, int st) {
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      fb[h][j][0] = ld16(rb + st * kPStage + h * kPHalf + j * 16 * kPRow + pos);
      fb[h][j][1] = ld16(rb + st * kPStage + h * kPHalf + j * 16 * kPRow + (pos ^ 64));
    }
  };
  auto bar = [&]() {
    mem_fence_compiler();
    __builtin_amdgcn_s_barrier();
    mem_fence_compiler();
  };
  // the end of a memory part: own reads done, transfers older than the last n landed
#define GS_GEMM_MEM_END(n)                          \
  do {                                              \
    mem_fence_compiler();                           \
    __builtin_amdgcn_s_waitcnt(wait_vm_lds(n));     \
    bar();                                          \
    __builtin_amdgcn_sched_barrier(0);              \
  } while (0)
  auto mma = [&](int h, int c) {
    __builtin_amdgcn_s_setprio(1);
#pragma unroll
    for (int k = 0; k < 2; ++k)
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
          acc[HALF ? 0 : h][c][i][j] = mfma16_bf16(fb[c][j][k], fa[i][k], acc[HALF ? 0 : h][c][i][j]);
    __builtin_amdgcn_s_setprio(0);
    __builtin_amdgcn_sched_barrier(0);
    bar();
  };

  if constexpr (!HALF) {
#pragma unroll
    for (int kt = 0; kt < 2; ++kt) {
      issue_b(0, kt);
      issue_a(0, kt);
      issue_b(1, kt);
      issue_a(1, kt);
    }
    GS_GEMM_MEM_END(12);                        // B0(0) and A0(0) landed
    read_b(0, 0);
    GS_GEMM_MEM_END(12);                        // every wave holds B0(0)
    if (wm == 1) bar();                         // waves 4-7 start one part behind
    int st = 0;
    for (int kt = 0; kt < nk - 2; ++kt, st ^= 1) {
      read_a(0, st);
      issue_b(0, kt + 2);
      GS_GEMM_MEM_END(12);
      mma(0, 0);
      read_b(1, st);
      issue_a(0, kt + 2);
      GS_GEMM_MEM_END(12);
      mma(0, 1);
      read_a(1, st);
      issue_b(1, kt + 2);
      GS_GEMM_MEM_END(12);
      mma(1, 0);
      // B0(kt+1) replaces the operand that quadrant (1, 0) was the last to use
      read_b(0, st ^ 1);
      issue_a(1, kt + 2);
      GS_GEMM_MEM_END(12);
      mma(1, 1);
    }
    // the last two k-tiles (or the only one, moved into both stages): nothing
    // left to issue, the waits count down.  K = 64: 256 x 7296 6.9 us, 4096 x
    // 27136 75 (register form 11.5 and 86)
    if (nk > 1) {
      read_a(0, st);
      GS_GEMM_MEM_END(10);
      mma(0, 0);
      read_b(1, st);
      GS_GEMM_MEM_END(8);
      mma(0, 1);
      read_a(1, st);
      GS_GEMM_MEM_END(6);
      mma(1, 0);
      read_b(0, st ^ 1);
      GS_GEMM_MEM_END(4);
      mma(1, 1);
      st ^= 1;
    }
    read_a(0, st);
    GS_GEMM_MEM_END(2);
    mma(0, 0);
    read_b(1, st);
    GS_GEMM_MEM_END(0);
    mma(0, 1);
    read_a(1, st);
    GS_GEMM_MEM_END(0);
    mma(1, 0);
    mma(1, 1);
    if (wm == 0) bar();
  } else {
    // two phases per k-tile: P1 reads A0(kt), issues B1(kt+1) and B0(kt+2);
    // P2 reads B1(kt) and B0(kt+1), issues A0(kt+2).  Past the last k-tile
    // the last one is moved again (into a stage nothing reads any more).
    issue_b(0, 0);
    issue_a(0, 0);
    issue_b(1, 0);
    issue_b(0, 1);
    issue_a(0, 1);
    GS_GEMM_MEM_END(6);                         // B0(0) and A0(0) landed
    read_b(0, 0);
    GS_GEMM_MEM_END(6);
    if (wm == 1) bar();
    int st = 0;
    for (int kt = 0; kt < nk; ++kt, st ^= 1) {
      read_a(0, st);
      issue_b(1, kt + 1);
      issue_b(0, kt + 2);
      GS_GEMM_MEM_END(6);
      mma(0, 0);
      read_b(1, st);
      read_b(0, st ^ 1);
      issue_a(0, kt + 2);
      GS_GEMM_MEM_END(6);
      mma(0, 1);
    }
    if (wm == 0) bar();
    __builtin_amdgcn_s_waitcnt(wait_vm(0));     // no transfer may land after the workgroup's LDS is given back
  }
#undef GS_GEMM_MEM_END

  // lane l holds row l % 16 of each 16-row block and columns 8 * (l / 16) .. + 7
  // of each column half
  auto result = [&](int h, int i, int c) {
    const f32x4 lo = acc[h][c][i][0], hi = acc[h][c][i][1];
    return u32x4{pack_bf16x2(lo[0], lo[1]), pack_bf16x2(lo[2], lo[3]), pack_bf16x2(hi[0], hi[1]),
                 pack_bf16x2(hi[2], hi[3])};
  };
  if (wide_rows(p)) {
    const int row0 = first_row + wm * 64 + (l & 15);
    const int col0 = tn * kGBN + wn * 64 + (l >> 4) * 8;
#pragma unroll
    for (int h = 0; h < NA; ++h)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int row = row0 + h * 128 + i * 16;
        if (row >= p.M) continue;
        uint16_t* crow = p.c + static_cast<int64_t>(row) * p.ldc;
#pragma unroll
        for (int c = 0; c < 2; ++c) {
          const int col = col0 + c * 32;
          const u32x4 v = result(h, i, c);
          if (col + 8 <= p.N) {
            st16(crow + col, v);
          } else {
#pragma unroll
            for (int e = 0; e < 8; ++e)
              if (col + e < p.N) crow[col + e] = static_cast<uint16_t>(v[e >> 1] >> (16 * (e & 1)));
          }
        }
      }
    return;
  }
  // rows of C that do not start at 16 bytes: 2-byte stores of a lane's 8 columns
  // would scatter over 16 rows each (497 x 26543 x 128 41 us, 6991 x 11479 x 256
  // 200, 4144 x 4866 x 1024 85), so a wave passes its 64 x 64 results through its
  // part of the operand stages and stores 64 consecutive columns of a row at a
  // time (16, 73 and 50 us)
  lds_barrier();                                // no wave reads the stages, and no transfer lands in them, any more
  char* const mine = smem + wave * kPOutWave;
#pragma unroll
  for (int h = 0; h < NA; ++h) {
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int c = 0; c < 2; ++c) st16(mine + (i * 16 + (l & 15)) * kPOutRow + c * 64 + (l >> 4) * 16, result(h, i, c));
    const int row0 = first_row + h * 128 + wm * 64, col = tn * kGBN + wn * 64 + l;
    uint16_t* crow = p.c + static_cast<int64_t>(row0) * p.ldc + col;
    const int rows = min(64, p.M - row0);
    auto copy = [&](int r, int n) {             // rows r .. r + 15, those below n
      uint16_t v[16];
#pragma unroll
      for (int u = 0; u < 16; ++u) v[u] = *reinterpret_cast<const uint16_t*>(mine + (r + u) * kPOutRow + l * 2);
#pragma unroll
      for (int u = 0; u < 16; ++u)
        if (r + u < n) crow[(r + u) * p.ldc] = v[u];
    };
    if (col >= p.N) continue;
    if (rows == 64) {
#pragma unroll
      for (int r = 0; r < 64; r += 16) copy(r, 64);
    } else {
      for (int r = 0; r < rows; r += 16) copy(r, rows);
    }
  }
}

__global__ __launch_bounds__(512) void gemm_bf16_tn_pingpong_kernel(GemmParams p) {
  __shared__ __align__(16) char smem[2 * kPStage];
  int first, tn;
  bool half;
  if (!addr::gemm_tile_mixed(static_cast<int>(blockIdx.x), p.full_rows, p.half_rows, p.tiles_n, kGGroup, first, tn, half))
    return;
  if (half) gemm_tile_pingpong<true>(p, smem, first, tn);
  else gemm_tile_pingpong<false>(p, smem, first, tn);
}

// ---------------------------------------------------------------------------
// Streaming form (K % 64 == 0), for calls whose 256 x 256 tiles would leave
// most CUs idle: tiles of 16*MB x 16*NB, and the W waves of a workgroup split
// K, each computing the whole tile over its own chunks of 64 k (chunk c
// belongs to wave c % W).  Every byte that a tile needs is then used by one
// wave only, so each wave stages its chunks for itself, with no barrier in
// the loop.
//
// A chunk is MB + NB slots of 2 KB (16 rows x 128 bytes, whole cache lines; a
// load straight into MFMA registers takes 16 rows x 16 bytes per 16 lanes and
// ran at a quarter of the rate): the B blocks, then the A blocks.  A wave's
// LDS ring holds RS slots.  Slots are read LA ahead of their MFMAs (one wave
// per SIMD has nothing else to hide an LDS trip behind), and a slot is
// refilled as soon as its reads have returned.  Waits count transfers (vmcnt);
// the last TC chunks, where refills run out, count down with them.  The W
// partial tiles are summed through LDS at the end, in wave order.
//
// Tiles are numbered down the rows first, in one contiguous range per XCD: the
// row tiles that share weights run together on one XCD, which reads them from
// HBM once.
//
// Bound by LDS (each byte written once and read once) and, for few rows, by
// HBM: 256 x 7296 x 4096 76 -> 29.3 us and 256 x 4480 x 12800 245 -> 79 against
// the 256 x 256 tiles; 16 x 7296 x 4096 47 -> 13.7 us (4.4 TB/s of weights),
// 7 x 4480 x 4096 47 -> 11.2 us (3.3 TB/s).  Deeper rings and longer lookaheads
// measured the same.
// ---------------------------------------------------------------------------
// s_waitcnt for "lgkmcnt <= n"
constexpr int wait_lds(int n) { return 15 | (7 << 4) | (n << 8) | (3 << 14); }
constexpr int kSOutRow = 32 * 2 + 16;           // a unit's 16 x 32 results in LDS
static_assert(16 * kSOutRow <= 2048, "they fit a unit's partial");

template <typename F, int... I>
__device__ __forceinline__ void static_for_impl(F&& f, std::integer_sequence<int, I...>) {
  (f(std::integral_constant<int, I>{}), ...);
}
// f(integral_constant 0) .. f(integral_constant N - 1): steps whose waits are immediates
template <int N, typename F>
__device__ __forceinline__ void static_for(F&& f) {
  static_for_impl(f, std::make_integer_sequence<int, N>{});
}

template <int MB, int NB, int W, int RS, int LA>
struct StreamShape {
  static constexpr int NS = MB + NB;            // slots per chunk
  static constexpr int TC = (RS + NS - 1) / NS; // chunks at the end whose refills run out
  static constexpr int kSlot = 16 * kPRow;
  static constexpr int kRing = RS * kSlot;      // bytes per wave
  static constexpr int NP = NB / 2;                 // column units of a row block: 2 16-column blocks each
  static constexpr int U = MB * NP;
  static constexpr int kSum = W * U * 2048;         // the partial tiles
  static constexpr int kLds = W * kRing > kSum ? W * kRing : kSum;
  static_assert(NB % 2 == 0, "column blocks pair up");
  static_assert(RS >= NS && LA >= 1 && LA < NS && kLds <= 160 * 1024, "the ring holds a chunk, LDS holds the rings");
};

template <int MB, int NB, int W, int RS, int LA>
__global__ __launch_bounds__(64 * W) void gemm_bf16_tn_stream_kernel(GemmParams p) {
  using S = StreamShape<MB, NB, W, RS, LA>;
  constexpr int NS = S::NS, NP = S::NP, U = S::U, TC = S::TC;
  __shared__ __align__(16) char smem[S::kLds];
  int tm, tn;
  if (!addr::gemm_tile(static_cast<int>(blockIdx.x), p.tiles_m, p.tiles_n, p.tiles_m, tm, tn)) return;
  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l = tid & 63;
  const int i16 = l & 15;
  const int q = l >> 4;

  // slot s of a chunk: 16-column block s of B (s < NB), else 16-row block s - NB of A
  uint32_t off[NS][2];
#pragma unroll
  for (int s = 0; s < NS; ++s)
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      const int r = 8 * t + (l >> 3);
      const uint32_t piece = addr::gemm_piece(l, r) * 16;
      off[s][t] = piece + static_cast<uint32_t>(
          s < NB ? (addr::gemm_row(tn * 16 * NB + addr::gemm_s_brow(r, s), p.N) - tn * 16 * NB) * p.ldb * 2
                 : (addr::gemm_row(tm * 16 * MB + 16 * (s - NB) + r, p.M) - tm * 16 * MB) * p.lda * 2);
    }
  const char* const basea = p.a + static_cast<int64_t>(tm) * 16 * MB * p.lda * 2;
  const char* const baseb = p.b + static_cast<int64_t>(tn) * 16 * NB * p.ldb * 2;
  const uint32_t ring0 = static_cast<uint32_t>(reinterpret_cast<uintptr_t>((lds_ptr_t)(smem))) + wave * S::kRing;
  const int mine = addr::gemm_s_chunks(p.K / kPBK, wave, W);   // this wave's chunks
  // slot s of chunk i into the ring at byte `at`
  auto issue = [&](int i, int s, uint32_t at) {
    const char* g = (s < NB ? baseb : basea) + static_cast<int64_t>(wave + W * i) * kPRow;
    dma16_at(g, off[s][0], ring0 + at);
    dma16_at(g, off[s][1], ring0 + at + 1024);
  };
  const char* const rd = smem + wave * S::kRing + i16 * kPRow;
  const int pos = (q ^ addr::lds_swz(i16)) * 16;

  f32x4 acc[MB][NB];
#pragma unroll
  for (int i = 0; i < MB; ++i)
#pragma unroll
    for (int j = 0; j < NB; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  u32x4 fb[NB][2], fa[LA + 1][2];
  auto mma = [&](int i, const u32x4 (&a)[2]) {
#pragma unroll
    for (int k = 0; k < 2; ++k)
#pragma unroll
      for (int j = 0; j < NB; ++j) acc[i][j] = mfma16_bf16(fb[j][k], a[k], acc[i][j]);
  };
  // One chunk, whose slot 0 is at ring byte p0.  Step s reads slot s (once all
  // but the `kYoung` slots issued after it have landed) and completes slot
  // s - LA: its reads are back, its place is refilled, its MFMAs are issued.
  // kTail: -1 while every refill exists, else the chunk's place in the last TC.
  auto chunk = [&](int i, uint32_t p0, auto tail_tag) {
    constexpr int kTail = decltype(tail_tag)::value;
    auto at = [&](int s) {
      const uint32_t x = p0 + s * S::kSlot;
      return x >= S::kRing ? x - S::kRing : x;
    };
    static_for<NS + LA>([&](auto step) {
      constexpr int s = decltype(step)::value;
      if constexpr (s < NS) {
        constexpr int kDone = s > LA ? s - LA : 0;             // slots of this chunk refilled so far
        constexpr int kIssued = kTail < 0 ? RS + kDone
                                          : (RS + kTail * NS + kDone < TC * NS ? RS + kTail * NS + kDone : TC * NS) - kTail * NS;
        constexpr int kYoung = 2 * (kIssued - 1 - s);
        mem_fence_compiler();
        __builtin_amdgcn_s_waitcnt(wait_vm(kYoung < 63 ? kYoung : 63));
        mem_fence_compiler();
        const char* r = rd + at(s);
        if constexpr (s < NB) {
          fb[s][0] = ld16(r + pos);
          fb[s][1] = ld16(r + (pos ^ 64));
        } else {
          fa[s % (LA + 1)][0] = ld16(r + pos);
          fa[s % (LA + 1)][1] = ld16(r + (pos ^ 64));
        }
      }
      if constexpr (s >= LA) {
        constexpr int d = s - LA;                              // the slot completed
        mem_fence_compiler();
        __builtin_amdgcn_s_waitcnt(wait_lds(2 * (s < NS ? LA : NS - 1 - d)));
        mem_fence_compiler();
        if constexpr (kTail < 0 || kTail * NS + d + RS < TC * NS) issue(i + (d + RS) / NS, (d + RS) % NS, at(d));
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (d >= NB) mma(d - NB, fa[d % (LA + 1)]);
      }
    });
  };
  uint32_t p0 = 0;
  auto next = [&]() { p0 = p0 + NS * S::kSlot >= S::kRing ? p0 + NS * S::kSlot - S::kRing : p0 + NS * S::kSlot; };
  static_for<RS>([&](auto g) {
    constexpr int s = decltype(g)::value;
    issue(s / NS, s % NS, s * S::kSlot);
  });
  int i = 0;
  for (; i < mine - TC; ++i) {
    chunk(i, p0, std::integral_constant<int, -1>{});
    next();
  }
  static_for<TC>([&](auto t) {
    chunk(i + decltype(t)::value, p0, t);
    next();
  });
  lds_barrier();                                // every wave is done with its ring

  // sum the waves' partial tiles: unit u (row block u / NP, column unit u % NP)
  // is summed and stored by wave u % W
  f32x4* part = reinterpret_cast<f32x4*>(smem);
#pragma unroll
  for (int i = 0; i < MB; ++i)
#pragma unroll
    for (int j = 0; j < NB; ++j) part[((wave * U + i * NP + j / 2) * 2 + j % 2) * 64 + l] = acc[i][j];
  lds_barrier();
  auto sum = [&](int u) {                       // lane l: row l % 16 of the unit, columns 8 * (l / 16) .. + 7
    f32x4 v[2];
#pragma unroll
    for (int e = 0; e < 2; ++e) v[e] = part[(u * 2 + e) * 64 + l];
#pragma unroll
    for (int w = 1; w < W; ++w)
#pragma unroll
      for (int e = 0; e < 2; ++e) v[e] += part[((w * U + u) * 2 + e) * 64 + l];
    return u32x4{pack_bf16x2(v[0][0], v[0][1]), pack_bf16x2(v[0][2], v[0][3]), pack_bf16x2(v[1][0], v[1][1]),
                 pack_bf16x2(v[1][2], v[1][3])};
  };
  if (wide_rows(p)) {
    for (int u = wave; u < U; u += W) {
      const u32x4 o = sum(u);
      const int row = tm * 16 * MB + (u / NP) * 16 + i16;
      const int col = tn * 16 * NB + (u % NP) * 32 + q * 8;
      if (row >= p.M) continue;
      uint16_t* crow = p.c + static_cast<int64_t>(row) * p.ldc;
      if (col + 8 <= p.N) {
        st16(crow + col, o);
      } else {
#pragma unroll
        for (int e = 0; e < 8; ++e)
          if (col + e < p.N) crow[col + e] = static_cast<uint16_t>(o[e >> 1] >> (16 * (e & 1)));
      }
    }
    return;
  }
  // as in the ping-pong form, through the place of the unit's first partial,
  // which only this wave reads: 32 consecutive columns of 2 rows a store
  for (int u = wave; u < U; u += W) {
    char* const mine = reinterpret_cast<char*>(part + u * 128);
    st16(mine + i16 * kSOutRow + q * 16, sum(u));
    const int row0 = tm * 16 * MB + (u / NP) * 16, col = tn * 16 * NB + (u % NP) * 32 + (l & 31);
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      const int r = 2 * k + (l >> 5);
      const uint16_t x = *reinterpret_cast<const uint16_t*>(mine + r * kSOutRow + (l & 31) * 2);
      if (row0 + r < p.M && col < p.N) p.c[static_cast<int64_t>(row0 + r) * p.ldc + col] = x;
    }
  }
}

// ---- which form a call takes ---------------------------------------------------
// Whole 64-k tiles, and rows within 32-bit offsets of a tile's first.
inline bool pingpong_form(int64_t K, int64_t lda, int64_t ldb) {
  return K % kPBK == 0 && lda <= kPMaxLd && ldb <= kPMaxLd;
}

struct StreamForm {
  int MB, NB, W, RS, LA;
  void (*kernel)(GemmParams);
};
template <int MB, int NB, int W, int RS, int LA>
constexpr StreamForm stream_form() {
  return {MB, NB, W, RS, LA, gemm_bf16_tn_stream_kernel<MB, NB, W, RS, LA>};
}
const StreamForm kStreamForms[] = {
    stream_form<1, 2, 4, 10, 2>(), stream_form<2, 2, 4, 10, 2>(), stream_form<4, 2, 4, 10, 2>(),
    stream_form<4, 4, 4, 10, 3>(), stream_form<8, 4, 4, 16, 3>(),
};

// The form with the fewest clocks per 64 k on the busiest CU: tiles per CU
// times a tile's weight, fitted to the forms' measured times (relative weights:
// 60 for each 2 KB slot of a streaming form, 2400 for the 256 x 256 tile, 1700
// for its 128-row form; their LDS time, transfers in at 64 bytes per clock plus
// operand reads at 128, is 48, 2560 and 1792).  The HBM time of the operands is
// the same for all of them.  Every wave of a streaming form needs TC chunks.
// Measured, M x 7296 x 4096, us, every form (16*MB x 16*NB) that was close:
//   M     16 x 32  32 x 32  64 x 32  64 x 64  128 x 64  128 x 256  256 x 256
//   16      13.2                                                     47
//   32      17.1     14.7                                            48
//   64               21.0     18.2     22.9                49        50
//   128                       26.2     21.4      28.4                55
//   256                                34.8      28.9                76
//   512                                59.2      50.8                75
//   777                                83.3      83.2      55        75
constexpr int64_t kFullClocks = 2400, kHalfClocks = 1700;
// Clocks per 64 k of `full` 256-row tiles followed by `halves` 128-row ones on
// `cus` CUs, each taking the next tile when it is free.
inline int64_t gemm_mixed_clocks(int64_t full, int64_t halves, int64_t cus) {
  const int64_t late = full % cus, early = cus - late;          // CUs that run one full tile more, and the others
  const int64_t t_early = full / cus * kFullClocks, t_late = t_early + kFullClocks;
  const int64_t end = late > 0 ? t_late : t_early;
  if (halves == 0) return end;
  // halves done once the early CUs have run k: early * k + late * (k - 2) at
  // their k-th end, early * k + late * (k - 1) at the late CUs' next one
  static_assert(kFullClocks > kHalfClocks && kFullClocks < 2 * kHalfClocks, "the order of the two groups' ends");
  for (int64_t k = std::max<int64_t>(1, halves / cus - 1);; ++k) {
    if (early * k + late * std::max<int64_t>(0, k - 2) >= halves) return std::max(end, t_early + k * kHalfClocks);
    if (early * k + late * (k - 1) >= halves) return std::max(end, t_late + (k - 1) * kHalfClocks);
  }
}
struct GemmPick {
  const StreamForm* stream;   // nullptr: the ping-pong form
  int full_rows;              // its tile rows of 256
};
// Ping-pong, 4144 x 4864 x 12800 (17 x 19 tiles, the last row of 48): 461 us
// with 16 full tile rows (304 tiles on 256 CUs, 48 in a second round) and one
// half row, 389 us with 13 and 7; 4096 x 4480 x 12800 457 -> 384 us.
inline GemmPick pick_gemm(int64_t M, int64_t N, int64_t K, int64_t cus) {
  auto tiles = [&](int64_t tm, int64_t tn) { return ((M + tm - 1) / tm) * ((N + tn - 1) / tn); };
  auto rounds = [&](int64_t n) { return (n + cus - 1) / cus; };
  const int64_t tiles_m = (M + kGBM - 1) / kGBM, tiles_n = (N + kGBN - 1) / kGBN;
  GemmPick best{nullptr, static_cast<int>(tiles_m)};
  int64_t cost = INT64_MAX;
  // a tile row fewer at a time (16 of them level out any last round)
  for (int64_t f = tiles_m; f >= std::max<int64_t>(0, tiles_m - 16); --f) {
    const int64_t c = gemm_mixed_clocks(f * tiles_n, addr::gemm_half_rows(M, static_cast<int>(f)) * tiles_n, cus);
    if (c < cost) {
      cost = c;
      best.full_rows = static_cast<int>(f);
    }
  }
  for (const StreamForm& f : kStreamForms) {
    const int64_t tc = (f.RS + f.MB + f.NB - 1) / (f.MB + f.NB);
    const int64_t c = 60 * (f.MB + f.NB) * rounds(tiles(16 * f.MB, 16 * f.NB));
    if (K / kPBK / f.W >= tc && c < cost) {
      cost = c;
      best.stream = &f;
    }
  }
  return best;
}

template <bool KTAIL>
void launch_gemm(unsigned grid, const GemmParams& p, hipStream_t st) {
  constexpr int WM = 2, WN = 4;
  auto kern = gemm_bf16_tn_kernel<KTAIL, WM, WN>;
  (void)hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, kGLds);
  hipLaunchKernelGGL(kern, dim3(grid), dim3(64 * WM * WN), kGLds, st, p);
}

// ----------------------------------------------------------------------------
// Address model (test support): replays on the host every global and LDS
// access of both GEMM kernels for one shape -- every workgroup, thread and
// k-tile -- and checks each against its buffer, and that the grid takes
// every tile exactly once.  No HIP call is made.
// ----------------------------------------------------------------------------
struct GemmModel {
  int64_t M, N, K, lda, ldb, ldc;
  int tiles_m, tiles_n;
  int64_t checked = 0, bad = 0;
  char msg[512] = {0};
  void fail(const char* fmt, ...) {
    if (++bad > 1) return;
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(msg, sizeof msg, fmt, ap);
    va_end(ap);
  }
  bool in(const char* what, int64_t lo, int64_t len, int64_t size) {
    ++checked;
    if (lo < 0 || len < 0 || lo + len > size) {
      fail("%s: [%lld, %lld) outside [0, %lld)", what, (long long)lo, (long long)(lo + len), (long long)size);
      return false;
    }
    return true;
  }
  int64_t a_elems() const { return (M - 1) * lda + K; }
  int64_t b_elems() const { return (N - 1) * ldb + K; }
  // the tiles of the grid, each once
  template <typename F>
  void tiles(F&& fn) {
    const int64_t total = int64_t(tiles_m) * tiles_n, grid = 8 * ((total + 7) / 8);
    std::vector<char> seen(total, 0);
    for (int64_t b = 0; b < grid; ++b) {
      int tm, tn;
      if (!addr::gemm_tile(static_cast<int>(b), tiles_m, tiles_n, kGGroup, tm, tn)) continue;
      if (!in("tile row", tm, 1, tiles_m) || !in("tile column", tn, 1, tiles_n)) continue;
      if (seen[int64_t(tm) * tiles_n + tn]++) fail("tile (%d, %d) taken twice", tm, tn);
      fn(tm, tn);
    }
    for (int64_t t = 0; t < total; ++t)
      if (!seen[t]) {
        fail("tile %lld of %lld is never taken", (long long)t, (long long)total);
        break;
      }
  }
  // The layout of one half-operand a writer mapping produces: slot (row,
  // position) must be written exactly once and hold the global piece position
  // ^ lds_swz(row), which is where the operand reads look for it.
  struct HalfLayout {
    std::vector<int> piece = std::vector<int>(128 * 8, -1);
  };
  void put(HalfLayout& st, int row, int pos, int gpiece) {
    ++checked;
    if (row < 0 || row >= 128 || pos < 0 || pos >= 8) return fail("stage slot (%d, %d) outside the half", row, pos);
    int& slot = st.piece[row * 8 + pos];
    if (slot >= 0) return fail("stage slot (%d, %d) written twice", row, pos);
    slot = gpiece;
  }
  void check_layout(const HalfLayout& st) {
    for (int r = 0; r < 128; ++r)
      for (int q = 0; q < 8; ++q) {
        ++checked;
        const int g = st.piece[r * 8 + q];
        if (g != (q ^ addr::lds_swz(r)))
          return fail("stage slot (%d, %d) holds piece %d, the operand reads expect %d", r, q, g, q ^ addr::lds_swz(r));
      }
  }
  void stores(int tm, int tn, int WM, int WN) {
    const int MI = kGBM / WM / 32, NJ = kGBN / WN / 32;
    for (int wave = 0; wave < WM * WN; ++wave)
      for (int l = 0; l < 64; ++l) {
        const int wm = wave / WN, wn = wave % WN;
        const int row0 = tm * kGBM + wm * MI * 32, col0 = tn * kGBN + wn * NJ * 32 + (l & 31);
        for (int i = 0; i < MI; ++i)
          for (int j = 0; j < NJ; ++j) {
            const int col = col0 + j * 32;
            if (col >= N) continue;
            for (int v = 0; v < 16; ++v) {
              const int row = row0 + i * 32 + ((v >> 2) << 3) + ((l >> 5) << 2) + (v & 3);
              if (row < M) in("C", int64_t(row) * ldc + col, 1, (M - 1) * ldc + N);
            }
          }
      }
  }
  // A wave's results of rows x cols passed through LDS rows of out_row bytes
  // (rows of C that do not start at 16 bytes): lane l of the writers gives row
  // l % 16 of each 16-row block 16-byte pieces, the readers take single
  // columns; each must find its own element.
  void out_pass(const char* who, int rows, int cols, int out_row, int64_t lds) {
    std::vector<int> held(lds / 2, -1);
    for (int i = 0; i < rows / 16; ++i)
      for (int c = 0; c < cols / 32; ++c)
        for (int l = 0; l < 64; ++l)
          for (int e = 0; e < 8; ++e) {
            const int64_t at = (i * 16 + (l & 15)) * out_row + c * 64 + (l >> 4) * 16 + 2 * e;
            if (!in(who, at, 2, lds)) continue;
            if (held[at / 2] >= 0) fail("%s: byte %lld written twice", who, (long long)at);
            held[at / 2] = (i * 16 + (l & 15)) * cols + c * 32 + (l >> 4) * 8 + e;
          }
    for (int r = 0; r < rows; ++r)
      for (int col = 0; col < cols; ++col) {
        const int64_t at = r * out_row + col * 2;
        if (in(who, at, 2, lds) && held[at / 2] != r * cols + col) fail("%s: (%d, %d) is another element", who, r, col);
      }
  }
  // gemm_bf16_tn_pingpong_kernel: every workgroup's transfers, operand reads
  // and stores, each tile and each element of C once, and each operand read
  // landing on the rows and columns its result is stored at
  void pingpong(int full) {
    const int nk = static_cast<int>(K / kPBK), halves = addr::gemm_half_rows(M, full);
    const int slots = static_cast<int>((M + 127) / 128);       // tile rows of 128
    HalfLayout st;
    for (int wave = 0; wave < 8; ++wave)
      for (int l = 0; l < 64; ++l)
        for (int j = 0; j < 2; ++j) {
          // a transfer fills 8 rows x 128 bytes of LDS in lane order
          const int64_t lds = (8 * (2 * wave + j)) * kPRow + l * 16;
          put(st, static_cast<int>(lds / kPRow), static_cast<int>((lds % kPRow) / 16),
              addr::gemm_piece(l, 8 * (2 * wave + j) + (l >> 3)));
        }
    check_layout(st);
    for (int wave = 0; wave < 8; ++wave)        // operand reads
      for (int l = 0; l < 64; ++l) {
        const int wm = wave >> 2, wn = wave & 3, pos = ((l >> 4) ^ addr::lds_swz(l & 15)) * 16;
        for (int stage = 0; stage < 2; ++stage)
          for (int h = 0; h < 2; ++h)
            for (int k = 0; k < 2; ++k) {
              for (int i = 0; i < 4; ++i) {
                const int64_t in_half = (wm * 64 + (l & 15) + i * 16) * kPRow + (pos ^ (64 * k));
                in("A operand (LDS)", in_half, 16, kPHalf);
                in("A operand (LDS)", stage * kPStage + h * kPHalf + in_half, 16, 2 * kPStage);
              }
              for (int j = 0; j < 2; ++j) {
                const int r = wn * 32 + (l & 15) + j * 16;
                const int64_t in_half = r * kPRow + (pos ^ (64 * k));
                in("B operand (LDS)", in_half, 16, kPHalf);
                in("B operand (LDS)", stage * kPStage + (2 + h) * kPHalf + in_half, 16, 2 * kPStage);
                // matrix row l % 16 of block j is column 8 * (row / 4) + 4 j + row % 4 of the wave's column half
                if (addr::gemm_b_row(r, h) != wn * 64 + h * 32 + 8 * ((l & 15) >> 2) + 4 * j + (l & 3))
                  fail("B row %d of half %d is staged as tile column %d", r, h, addr::gemm_b_row(r, h));
              }
            }
      }
    out_pass("C through LDS", 64, 64, kPOutRow, kPOutWave);
    const int64_t total = int64_t(slots) * tiles_n, grid = addr::gemm_mixed_grid(full, halves, tiles_n);
    std::vector<char> seen(total, 0);
    for (int64_t b = 0; b < grid; ++b) {
      int first, tn;
      bool half;
      if (!addr::gemm_tile_mixed(static_cast<int>(b), full, halves, tiles_n, kGGroup, first, tn, half)) continue;
      if (!in("tile row", first / 128, 1, slots) || !in("tile column", tn, 1, tiles_n)) continue;
      const int tile_rows = half ? kGBM / 2 : kGBM;
      for (int r = first / 128; r < (first + tile_rows) / 128 && r < slots; ++r)
        if (seen[int64_t(r) * tiles_n + tn]++) fail("rows %d on of tile column %d taken twice", 128 * r, tn);
      std::vector<char> cseen(kGBM * kGBN, 0);
      for (int wave = 0; wave < 8; ++wave)
        for (int l = 0; l < 64; ++l) {
          for (int j = 0; j < 2; ++j) {
            const int r = 8 * (2 * wave + j) + (l >> 3);
            const int piece = addr::gemm_piece(l, r);
            for (int h = 0; h < 2; ++h) {
              const int64_t ra = addr::gemm_row(first + h * 128 + r, static_cast<int>(M));
              const int64_t rb = addr::gemm_row(tn * kGBN + addr::gemm_b_row(r, h), static_cast<int>(N));
              if (h == 0 || !half) in("A offset in 32 bits", (ra - first) * lda * 2 + piece * 16, 16, int64_t(1) << 32);
              in("B offset in 32 bits", (rb - int64_t(tn) * kGBN) * ldb * 2 + piece * 16, 16, int64_t(1) << 32);
              for (int kt = 0; kt < nk; ++kt) {
                if (h == 0 || !half) in("A", ra * lda + int64_t(kt) * kPBK + piece * 8, 8, a_elems());
                in("B", rb * ldb + int64_t(kt) * kPBK + piece * 8, 8, b_elems());
              }
            }
          }
          const int wm = wave >> 2, wn = wave & 3;
          for (int h = 0; h < (half ? 1 : 2); ++h)
            for (int i = 0; i < 4; ++i)
              for (int c = 0; c < 2; ++c)
                for (int e = 0; e < 8; ++e) {
                  const int row = wm * 64 + (l & 15) + h * 128 + i * 16, col = wn * 64 + (l >> 4) * 8 + c * 32 + e;
                  if (first + row >= M || tn * kGBN + col >= N) continue;
                  in("C", int64_t(first + row) * ldc + tn * kGBN + col, 1, (M - 1) * ldc + N);
                  if (cseen[row * kGBN + col]++) fail("C element (%d, %d) of a tile stored twice", row, col);
                }
        }
      for (int r = 0; r < tile_rows; ++r)
        for (int c = 0; c < kGBN; ++c)
          if (first + r < M && tn * kGBN + c < N && !cseen[r * kGBN + c]) {
            fail("C element (%d, %d) of the tile at row %d, tile column %d is never stored", r, c, first, tn);
            r = kGBM;
            break;
          }
    }
    for (int64_t t = 0; t < total; ++t)
      if (!seen[t]) {
        fail("tile %lld of %lld is never taken", (long long)t, (long long)total);
        break;
      }
  }
  // gemm_bf16_tn_stream_kernel: the ring's schedule of every wave (each slot
  // has landed when it is read, and is refilled only after its reads are
  // back), then every workgroup's transfers and stores
  void stream(const StreamForm& f) {
    const int NS = f.MB + f.NB, TC = (f.RS + NS - 1) / NS, nk = static_cast<int>(K / kPBK);
    tiles_m = static_cast<int>((M + 16 * f.MB - 1) / (16 * f.MB));
    tiles_n = static_cast<int>((N + 16 * f.NB - 1) / (16 * f.NB));
    int chunks_seen = 0;
    for (int w = 0; w < f.W; ++w) {
      const int mine = addr::gemm_s_chunks(nk, w, f.W);
      chunks_seen += mine;
      if (mine < TC) return fail("wave %d has %d chunks, its last %d are counted down", w, mine, TC);
      std::vector<int64_t> held(f.RS);                       // the stream slot in each ring place
      int64_t issued = f.RS;
      for (int g = 0; g < f.RS; ++g) held[g] = g;
      for (int i = 0; i < mine; ++i) {
        const int tail = i < mine - TC ? -1 : i - (mine - TC);
        for (int s = 0; s < NS + f.LA; ++s) {
          const int64_t g = int64_t(i) * NS + s;
          if (s < NS) {
            const int done = s > f.LA ? s - f.LA : 0;
            const int iss = tail < 0 ? f.RS + done : std::min(f.RS + tail * NS + done, TC * NS) - tail * NS;
            const int young = std::min(2 * (iss - 1 - s), 63);
            ++checked;
            if (2 * (issued - 1 - g) < young) fail("slot %lld is read before it has landed", (long long)g);
            if (held[g % f.RS] != g) fail("slot %lld is not in its ring place", (long long)g);
          }
          const int d = s - f.LA;
          if (d >= 0 && (tail < 0 || tail * NS + d + f.RS < TC * NS)) {
            const int64_t gd = int64_t(i) * NS + d, nx = gd + f.RS;
            in("chunk", i + (d + f.RS) / NS, 1, mine);
            if (nx != int64_t(i + (d + f.RS) / NS) * NS + (d + f.RS) % NS || nx != issued)
              fail("slot %lld is refilled out of order", (long long)gd);
            held[gd % f.RS] = nx;
            ++issued;
          }
        }
      }
      if (issued != int64_t(mine) * NS) fail("wave %d moved %lld slots of %lld", w, (long long)issued, (long long)mine * NS);
    }
    if (chunks_seen != nk) fail("the waves take %d chunks of %d", chunks_seen, nk);
    for (int l = 0; l < 64; ++l) {                           // LDS: a slot's transfers and operand reads
      const int i16 = l & 15, q = l >> 4, pos = (q ^ addr::lds_swz(i16)) * 16;
      for (int k = 0; k < 2; ++k) {
        in("operand (LDS)", i16 * kPRow + (pos ^ (64 * k)), 16, 16 * kPRow);
        if ((((pos ^ (64 * k)) / 16) ^ addr::lds_swz(i16)) != q + 4 * k) fail("operand reads another piece");
      }
      for (int t = 0; t < 2; ++t) {
        const int r = 8 * t + (l >> 3);
        if ((addr::gemm_piece(l, r) ^ addr::lds_swz(r)) != (l & 7)) fail("transfer lands at another piece");
      }
    }
    out_pass("C unit through LDS", 16, 32, kSOutRow, 2048);
    std::vector<char> cseen(static_cast<size_t>(M) * N, 0);
    const int64_t total = int64_t(tiles_m) * tiles_n;
    for (int64_t b = 0; b < 8 * ((total + 7) / 8); ++b) {
      int tm, tn;
      if (!addr::gemm_tile(static_cast<int>(b), tiles_m, tiles_n, tiles_m, tm, tn)) continue;
      const int row0 = tm * 16 * f.MB, col0 = tn * 16 * f.NB;
      for (int l = 0; l < 64; ++l) {
        for (int s = 0; s < NS; ++s)
          for (int t = 0; t < 2; ++t) {
            const int r = 8 * t + (l >> 3), piece = addr::gemm_piece(l, r);
            const bool isb = s < f.NB;
            const int64_t row = isb ? addr::gemm_row(col0 + addr::gemm_s_brow(r, s), static_cast<int>(N))
                                    : addr::gemm_row(row0 + 16 * (s - f.NB) + r, static_cast<int>(M));
            const int64_t ld = isb ? ldb : lda;
            in("offset in 32 bits", (row - (isb ? col0 : row0)) * ld * 2 + piece * 16, 16, int64_t(1) << 32);
            for (int kt = 0; kt < nk; ++kt)
              in(isb ? "B" : "A", row * ld + int64_t(kt) * kPBK + piece * 8, 8, isb ? b_elems() : a_elems());
          }
        const int NP = f.NB / 2;
        for (int u = 0; u < f.MB * NP; ++u)
          for (int e = 0; e < 8; ++e) {
            const int row = row0 + (u / NP) * 16 + (l & 15), col = col0 + (u % NP) * 32 + (l >> 4) * 8 + e;
            // element e of the lane: matrix row 4 (l / 16) + e % 4 of block 2 (u % NP) + e / 4
            if (addr::gemm_s_brow(4 * (l >> 4) + (e & 3), 2 * (u % NP) + (e >> 2)) != col - col0)
              fail("column %d is stored from another B row", col);
            if (row >= M || col >= N) continue;
            in("C", int64_t(row) * ldc + col, 1, (M - 1) * ldc + N);
            if (cseen[int64_t(row) * N + col]++) fail("C element (%d, %d) stored twice", row, col);
          }
      }
    }
    for (char c : cseen)
      if (!c) return fail("an element of C is never stored");
  }
  // gemm_bf16_tn_kernel<KTAIL, WM, WN>
  void reg(bool KTAIL, int WM, int WN) {
    const int threads = 64 * WM * WN, pieces = kGBM * (kGRowBytes / 16) / threads, step = threads / (kGRowBytes / 16);
    const int MI = kGBM / WM / 32, NJ = kGBN / WN / 32;
    const int nk = static_cast<int>((K + kGBK - 1) / kGBK);
    tiles([&](int tm, int tn) {
      for (int tid = 0; tid < threads; ++tid) {
        const int lrow = tid >> 3, lpc = (tid & 7) * 16, kp = (tid & 7) * 8;
        for (int j = 0; j < pieces; ++j) {
          const int64_t ra = addr::gemm_row(tm * kGBM + lrow + j * step, static_cast<int>(M));
          const int64_t rb = addr::gemm_row(tn * kGBN + lrow + j * step, static_cast<int>(N));
          for (int kt = 0; kt < nk; ++kt) {
            const bool ok = !KTAIL || kt * kGBK + kp < K;
            const int64_t off = ok ? int64_t(kt) * kGBK + lpc / 2 : 0;
            in("A", ra * lda + off, 8, a_elems());
            in("B", rb * ldb + off, 8, b_elems());
          }
          for (int buf = 0; buf < 2; ++buf) {
            in("A stage (LDS)", buf * kGStage + (lrow + j * step) * kGLd + lpc, 16, kGLds);
            in("B stage (LDS)", buf * kGStage + kGBM * kGLd + (lrow + j * step) * kGLd + lpc, 16, kGLds);
          }
        }
      }
      for (int wave = 0; wave < WM * WN; ++wave) {
        const int wm = wave / WN, wn = wave % WN;
        for (int l = 0; l < 64; ++l)
          for (int buf = 0; buf < 2; ++buf)
            for (int kk = 0; kk < kGBK / 16; ++kk) {
              const int64_t sa = buf * kGStage + (wm * MI * 32 + (l & 31)) * kGLd + (l >> 5) * 16 + kk * 32;
              const int64_t sb = buf * kGStage + kGBM * kGLd + (wn * NJ * 32 + (l & 31)) * kGLd + (l >> 5) * 16 + kk * 32;
              for (int i = 0; i < MI; ++i) in("A operand (LDS)", sa + i * 32 * kGLd, 16, kGLds);
              for (int j = 0; j < NJ; ++j) in("B operand (LDS)", sb + j * 32 * kGLd, 16, kGLds);
            }
      }
      stores(tm, tn, WM, WN);
    });
  }
};
}  // namespace

}  // namespace gs

using namespace gs;

extern "C" {

int gs_gemm_bf16_tn(const void* a, int64_t lda, const void* b, int64_t ldb, void* c, int64_t ldc, int64_t M,
                    int64_t N, int64_t K, void* stream) {
  const char* who = "gs_gemm_bf16_tn";
  GS_CHECK_ARG(M >= 0 && N >= 0 && M < (int64_t(1) << 31) && N < (int64_t(1) << 31), "%s: M=%lld N=%lld", who,
               (long long)M, (long long)N);
  GS_CHECK_ARG(K > 0 && K % 8 == 0 && K < (int64_t(1) << 31), "%s: K=%lld must be a positive multiple of 8", who,
               (long long)K);
  GS_CHECK_ARG(lda >= K && ldb >= K && lda % 8 == 0 && ldb % 8 == 0, "%s: lda=%lld ldb=%lld", who, (long long)lda,
               (long long)ldb);
  GS_CHECK_ARG(ldc >= N, "%s: ldc=%lld < N", who, (long long)ldc);
  GS_CHECK_ARG(aligned16(a) && aligned16(b) && (reinterpret_cast<uintptr_t>(c) & 1u) == 0,
               "%s: a and b must be 16-byte aligned, c 2-byte aligned", who);
  if (M == 0 || N == 0) return GS_OK;
  GemmParams p{};
  p.a = static_cast<const char*>(a);
  p.lda = lda;
  p.b = static_cast<const char*>(b);
  p.ldb = ldb;
  p.c = static_cast<uint16_t*>(c);
  p.ldc = ldc;
  p.M = static_cast<int>(M);
  p.N = static_cast<int>(N);
  p.K = static_cast<int>(K);
  p.tiles_m = static_cast<int>((M + kGBM - 1) / kGBM);
  p.tiles_n = static_cast<int>((N + kGBN - 1) / kGBN);
  const int64_t total = static_cast<int64_t>(p.tiles_m) * p.tiles_n;
  GS_CHECK_ARG(total <= (int64_t(1) << 30), "%s: too many tiles", who);
  const unsigned grid = static_cast<unsigned>(8 * ((total + 7) / 8));
  hipStream_t st = static_cast<hipStream_t>(stream);
  if (pingpong_form(K, lda, ldb)) {
    const GemmPick pick = pick_gemm(M, N, K, device_cus());
    if (pick.stream != nullptr) {
      p.tiles_m = static_cast<int>((M + 16 * pick.stream->MB - 1) / (16 * pick.stream->MB));
      p.tiles_n = static_cast<int>((N + 16 * pick.stream->NB - 1) / (16 * pick.stream->NB));
      const int64_t n = 8 * ((static_cast<int64_t>(p.tiles_m) * p.tiles_n + 7) / 8);
      hipLaunchKernelGGL(pick.stream->kernel, dim3(static_cast<unsigned>(n)), dim3(64 * pick.stream->W), 0, st, p);
      GS_CHECK_LAUNCH(who);
      return GS_OK;
    }
    p.full_rows = pick.full_rows;
    p.half_rows = addr::gemm_half_rows(M, p.full_rows);
    const unsigned n = static_cast<unsigned>(addr::gemm_mixed_grid(p.full_rows, p.half_rows, p.tiles_n));
    hipLaunchKernelGGL(gemm_bf16_tn_pingpong_kernel, dim3(n), dim3(512), 0, st, p);
  } else if (K % kGBK == 0) launch_gemm<false>(grid, p, st);
  else launch_gemm<true>(grid, p, st);
  GS_CHECK_LAUNCH(who);
  return GS_OK;
}

int gs_gemm_form(int64_t M, int64_t N, int64_t K, int64_t lda, int64_t ldb, int32_t cus, int32_t* form) {
  const char* who = "gs_gemm_form";
  GS_CHECK_ARG(M > 0 && N > 0 && K > 0 && cus >= 0 && form != nullptr, "%s: sizes", who);
  if (!pingpong_form(K, lda, ldb)) {
    form[0] = GS_GEMM_REGISTER;
    form[1] = form[2] = kGBM;
    return GS_OK;
  }
  const GemmPick pick = pick_gemm(M, N, K, cus > 0 ? cus : device_cus());
  form[0] = pick.stream != nullptr ? GS_GEMM_STREAM : GS_GEMM_PINGPONG;
  form[1] = pick.stream != nullptr ? 16 * pick.stream->MB : pick.full_rows;
  form[2] = pick.stream != nullptr ? 16 * pick.stream->NB : addr::gemm_half_rows(M, pick.full_rows);
  return GS_OK;
}

int64_t gs_check_gemm_addresses(int64_t M, int64_t N, int64_t K, int64_t lda, int64_t ldb, int64_t ldc, char* msg,
                                int64_t msg_len, int64_t* checked) {
  const char* who = "gs_check_gemm_addresses";
  GS_CHECK_ARG(M > 0 && N > 0 && K > 0 && K % 8 == 0 && lda >= K && ldb >= K && ldc >= N, "%s: shape", who);
  GemmModel m{};
  m.M = M;
  m.N = N;
  m.K = K;
  m.lda = lda;
  m.ldb = ldb;
  m.ldc = ldc;
  m.tiles_m = static_cast<int>((M + kGBM - 1) / kGBM);
  m.tiles_n = static_cast<int>((N + kGBN - 1) / kGBN);
  if (pingpong_form(K, lda, ldb)) {
    std::set<int> forms = {m.tiles_m, m.tiles_m - 1, m.tiles_m / 2, 0, pick_gemm(M, N, K, 256).full_rows};
    for (int full : forms) m.pingpong(full);
    for (const StreamForm& f : kStreamForms)
      if (K / kPBK / f.W >= (f.RS + f.MB + f.NB - 1) / (f.MB + f.NB)) m.stream(f);
    m.tiles_m = static_cast<int>((M + kGBM - 1) / kGBM);
    m.tiles_n = static_cast<int>((N + kGBN - 1) / kGBN);
  }
  m.reg(K % kGBK != 0, 2, 4);      // the register-staged form takes any shape
  if (checked) *checked = m.checked;
  if (msg && msg_len > 0) snprintf(msg, static_cast<size_t>(msg_len), "%s", m.msg);
  return m.bad;
}

}  // extern "C"
