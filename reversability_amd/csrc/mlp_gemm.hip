// MFMA GEMMs for the SwiGLU MLP projections on gfx950, with fused epilogues.
//
// The six contractions of one TiledMLP tile (src/reversibility/optimized_v3.py:
// 10-18, 47-63) under fp16 autocast, in the canonical form
//     C[i][j] = sum_k A(i, k) * B(j, k)      (fp16 operands, fp32 accumulate)
//
//   up + SwiGLU   A = x16[m][d]    B = Wup16[g|v][d]    -> o = fp16(silu(fp16 u_g)) * fp16 u_v
//   down          A = o[m][f]      B = Wdown16[d][f]    -> y = fp16(acc)
//   d_o + SwiGLU' A = dy[m][d]     B(f, d) = Wdown16[d][f] -> du = swiglu_bwd(u, fp16(acc))
//   dx            A = du[m][j]     B(d, j) = Wup16[j][d]   -> dx = fp32(fp16(acc))
//   dW_down       A(d, m) = dy[m][d]   B(f, m) = o[m][f]     -> (+)= fp32(fp16(acc))
//   dW_up         A(j, m) = du[m][j]   B(d, m) = x16[m][d]   -> (+)= fp32(fp16(acc))
//
// Every operand is fp16 and is read in its stored layout.  A "KC" source is
// [rows][k] (k contiguous) and is staged in LDS as [row][k]; fragments are one
// ds_read_b128 per lane.  An "RC" source is [k][rows] (rows contiguous) and is
// staged as [k][row]; fragments are two ds_read_b64_tr_b16 per lane, the
// gfx950 LDS transpose read.  Global -> LDS copies are therefore plain 16-byte
// row segments for both kinds, with no scatter.  The fp32 master weights and
// the fp32 normalized activations are cast to fp16 once per call
// (rv_cast_f32_f16) -- the cast autocast's F.linear performs.
//
// Tiling: a workgroup of 4 (2 x 2) or 8 (2 x 4) waves owns a BM x BN tile of
// C; each wave owns TM x TN tiles of 32 x 32 computed with
// v_mfma_f32_32x32x16_f16.  K advances BK (64 or 32) per stage through rings of
// LDS buffers that direct-to-LDS loads fill one to three stages ahead; one
// barrier per stage.  The tile shapes (kShapes) are timed per problem (see
// tune_act); the choice does not change any result bit, because every output
// element sums its k blocks in the same order in every tile shape.  Weight
// gradients over few output tiles may split the token reduction (split-K)
// into fp32 partials summed by a second kernel in a fixed order.
//
// LDS layouts: XOR swizzles of the 16-byte chunk index inside a row, bank
// conflict free for the fragment reads in both a 32- and a 64-bank model
// (f_kc, f_rc).
//
// What bounds the main loop (256 x 256 tile, m = 32768, n = 1024, k = 8192, B an
// RC source; timing copies with one part taken out): MFMA alone 248 us, MFMA
// and fragment reads 302, the loads alone 253, MFMA and loads 337, all three
// 429-437, i.e. 1.26-1.28 PFLOP/s; the same with every load an L2 hit: 423.  The
// LDS carries 64 KB of fragment reads and 32 KB of DMA writes per 32 k (512
// cycles each at 128 and 64 B/clk) against 1024 MFMA cycles, and with one wave
// per SIMD a read or a load that finds its queue full holds up the MFMAs
// behind it.  Before: 64-byte segments of the KC rows per stage, loads and reads
// in bursts, per-load vector address arithmetic and one wait for all of a k
// step's reads: 479-487 us.
//
// MFMA 32x32x16 lane layout (gfx950): lane l supplies A row / B row (l % 32)
// with k = (l/32)*8 + 0..7; accumulator value j of lane l is
// C[(j/4)*8 + (l/32)*4 + j%4][l % 32].  The kernel issues the product as
// B * A^T, so its accumulator holds the transposed tile: lane l owns C row
// l % 32 and four consecutive columns per group of four values.
//
// ds_read_b64_tr_b16 (gfx950): within each 16-lane group, lane i receives
// element (i % 4) of the 8-byte chunks addressed by lanes 4e + i/4, e = 0..3.
// With lanes 4e..4e+3 addressing 16 consecutive halves of LDS row e, lane i
// receives column i of rows 0..3: a 4 (k) x 16 (row) block, transposed.

#include <algorithm>
#include <atomic>
#include <cstdlib>
#include <map>
#include <mutex>
#include <tuple>
#include <type_traits>
#include <utility>

#include "rv_device.h"

namespace {

typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x4 __attribute__((ext_vector_type(4)));
typedef short i16x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));  // 16-byte staging word
#define RV_LDS __attribute__((address_space(3)))

// Tile shapes: BM x BN tile, waves, k per pipeline stage (one or half a
// 128-byte line of a KC row), depth of the two operands' LDS rings, workgroups
// per CU that the rings leave room for.  One workgroup per CU has the least
// LDS and L2 traffic per MFMA; two or three overlap one's epilogue with the
// others' MFMAs, and small problems need the smaller tiles.  Each is the
// fastest of the seven somewhere (us, m x d x f): 256 x 256 dx 32768x1024x4096
// 429 (the others 450-715), with 8 waves up 497 (522-743); 128 x 256 dgate
// 32768x1024x4096 382 (412-497); 128 x 128 with BK 64 dx 16896x256x1024 27.2
// (31.8-42), with BK 32 up + u 33.6 (35-47); 64 x 128 at two per CU dx of 51 rows
// 11.6 (12.6-43), at three proj 16896x256 7.1 (7.5-11).
struct TileShape {
  int bm, bn, waves, bk, ra, rb, per_cu;
};
// The first kRuleShapes are the ones pick_act's rule and the weight-gradient
// plan choose from; the tuner also times the rest.
constexpr int kNumShapes = 7, kRuleShapes = 4;
constexpr TileShape kShapes[kNumShapes] = {
    {256, 256, 4, 64, 3, 2, 1}, {128, 256, 4, 32, 3, 3, 2}, {128, 128, 4, 64, 3, 2, 2},
    {64, 128, 4, 64, 4, 3, 2},  {256, 256, 8, 64, 3, 2, 1}, {128, 128, 4, 32, 3, 3, 3},
    {64, 128, 4, 64, 2, 2, 3}};
constexpr int kCUs = 256;           // MI355X compute units (tile-shape choice only)
constexpr int kRsrcWord3 = 0x00020000;  // raw buffer resource, gfx9 data format

// XOR swizzles of the 16-byte chunk index inside one LDS row (see the layout
// notes at the top of the file).
template <int BK>
__device__ __forceinline__ int f_kc(int row) {
  if constexpr (BK == 64) return (row & 7) ^ ((row >> 3) & 1);
  else return ((row >> 2) & 3) ^ (row & 2);
}
template <int ROWS>
__device__ __forceinline__ int f_rc(int k) {
  return ((ROWS >= 128 ? 0xCA60 : 0x6420) >> ((k & 3) * 4)) & 0xF;
}

// s_waitcnt with vmcnt = N and the other counters left alone (gfx9 encoding).
template <int N>
__device__ __forceinline__ void wait_vmcnt() {
  static_assert(N >= 0 && N < 64, "vmcnt range");
  __builtin_amdgcn_s_waitcnt((N & 15) | (7 << 4) | (15 << 8) | ((N >> 4) << 14));
}

// Workgroup barrier that orders this wave's LDS accesses in program order
// (compiler barriers on both sides) without the release fence of
// __syncthreads, which would wait for every outstanding LDS DMA.
__device__ __forceinline__ void lds_barrier() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

// ---------------------------------------------------------------------------
// Row maps for KC sources: LDS row r of the tile -> source row.
// ---------------------------------------------------------------------------
// Relative to origin, the row the copies' base address is moved to (so that
// offsets stay 32-bit whatever the operand's size).
struct MapDirect {  // row0 + r, clamped to the last valid row (results never stored)
  int64_t row0, rows;
  __device__ __forceinline__ int64_t origin() const { return row0; }
  __device__ __forceinline__ int64_t operator()(int r) const {
    return row0 + r < rows ? r : rows - 1 - row0;
  }
};
// SwiGLU up projection: a BN-row B tile holds BN/2 output columns, as gate
// and value halves per wave column (WCOLS of them, C = BN/WCOLS rows each):
// rows [wn*C, wn*C + C/2) are gate rows col0 + wn*C/2 + w, the next C/2 are
// the value rows f + the same.
template <int BN, int WCOLS>
struct MapGateValue {
  int64_t col0, f;
  __device__ __forceinline__ int64_t origin() const { return 0; }
  __device__ __forceinline__ int64_t operator()(int r) const {
    constexpr int kCol = BN / WCOLS, kHalf = kCol / 2;
    const int wn = r / kCol, w = r % kCol;
    return w < kHalf ? col0 + wn * kHalf + w : f + col0 + wn * kHalf + (w - kHalf);
  }
};

// A wave-uniform 64-bit value in scalar registers: a value that reaches a buffer
// resource through vector registers costs a loop around every load.
__device__ __forceinline__ int64_t uniform(int64_t v) {
  const uint32_t lo = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)v);
  const uint32_t hi = (uint32_t)__builtin_amdgcn_readfirstlane((int)(v >> 32));
  return (int64_t)((uint64_t)hi << 32 | lo);
}

// ---------------------------------------------------------------------------
// Global -> LDS copies: direct-to-LDS buffer loads (buffer_load_dwordx4 ...
// lds).  One wave instruction fills 1 KB of LDS, lane L's 16 bytes at byte
// 16 L; each lane loads the source chunk whose swizzled LDS slot that is.
// A tile of ROWS rows is ROWS * 2 BK bytes per stage (BK halves per row, or
// BK k rows of ROWS halves), i.e. ROWS BK / 512 wave instructions.  A lane's source offsets are fixed for the whole kernel; a
// stage moves the buffer resource's base instead (scalar arithmetic only), and
// the resource ends with the operand, so k rows past the end of an RC source
// read as zero, and a resource of zero bytes (a stage past the end) reads
// nothing and writes zeros.
// ---------------------------------------------------------------------------
template <bool RC, int ROWS, int BK, int WAVES>
struct Dma {
  static constexpr int kPerWave = ROWS * BK / 512 / WAVES;
  static constexpr int kChunks = BK / 8;            // 16-byte chunks per KC row
  static constexpr int kRows = 64 / kChunks;        // KC rows per wave instruction
  uint32_t off[kPerWave];  // byte offset of this lane's chunk at k = 0 of the kernel's range
  int64_t base;            // address of the kernel's first k
  int64_t left;            // bytes from base to the operand's end
  int64_t kstep;           // bytes per stage

  // KC source [rows][ld] (k contiguous), tile rows row0..; rows past `rows`
  // are clamped (their results are never stored); map() gathers B rows.
  template <class Map>
  __device__ __forceinline__ void init_kc(const __half* p, int64_t bytes, int64_t ld,
                                          const Map& map, int64_t kbeg, int wave, int lane) {
    const int64_t first = map.origin() * ld + kbeg;
    base = uniform(reinterpret_cast<int64_t>(p + first));
    left = uniform(bytes - first * 2);
    kstep = BK * 2;
#pragma unroll
    for (int it = 0; it < kPerWave; ++it) {
      const int row = (it * WAVES + wave) * kRows + lane / kChunks;
      off[it] = (uint32_t)((map(row) * ld + ((lane % kChunks) ^ f_kc<BK>(row)) * 8) * 2);
    }
  }
  // RC source [k][ld], tile rows contiguous from row0.
  __device__ __forceinline__ void init_rc(const __half* p, int64_t bytes, int64_t ld,
                                          int64_t row0, int64_t kbeg, int wave, int lane) {
    base = uniform(reinterpret_cast<int64_t>(p + kbeg * ld + row0));
    left = uniform(bytes - (kbeg * ld + row0) * 2);
    kstep = BK * ld * 2;
#pragma unroll
    for (int it = 0; it < kPerWave; ++it) {
      const int b = (it * WAVES + wave) * 1024 + lane * 16;
      const int krow = b / (ROWS * 2), chunk = ((b % (ROWS * 2)) >> 4) ^ f_rc<ROWS>(krow);
      off[it] = (uint32_t)((krow * ld + chunk * 8) * 2);
    }
  }
  // A KC row's last stage holds `valid` < BK values of the reduction: chunks
  // at or past it are sent out of the resource's range and read as zero (stage()
  // gives it at most INT32_MAX bytes, whatever the operand's size).
  __device__ __forceinline__ void cut_kc(int valid, int wave, int lane) {
#pragma unroll
    for (int it = 0; it < kPerWave; ++it) {
      const int row = (it * WAVES + wave) * kRows + lane / kChunks;
      if (((lane % kChunks) ^ f_kc<BK>(row)) * 8 >= valid) off[it] = 0x80000000u;
    }
  }
  __device__ __forceinline__ __amdgpu_buffer_rsrc_t stage(int st, bool live) const {
    const int64_t at = (int64_t)st * kstep, n = left - at;
    return __builtin_amdgcn_make_buffer_rsrc(reinterpret_cast<char*>(base + at), 0,
                                             !live || n <= 0 ? 0 : n < INT32_MAX ? (int)n : INT32_MAX,
                                             kRsrcWord3);
  }
  // Wave instruction `it` of a stage into the tile at `lds`.
  __device__ __forceinline__ void issue(__amdgpu_buffer_rsrc_t rsrc, _Float16* lds, int it,
                                        int wave) const {
    __builtin_amdgcn_raw_ptr_buffer_load_lds(
        rsrc, (RV_LDS void*)(lds + (it * WAVES + wave) * 512), 16, off[it], 0, 0, 0);
  }
};

// ---------------------------------------------------------------------------
// MFMA fragments: lane l -> tile row r0 + l%32, k = ks*16 + (l/32)*8 + 0..7.
// ---------------------------------------------------------------------------
// The LDS reads are inline assembly: through the builtin (and ordinary loads)
// the compiler cannot always tell them from the in-flight LDS DMA writes and
// drains every outstanding DMA (vmcnt(0)) before them.  Their results are
// therefore not tracked by the compiler's LDS counter: the k-step code waits
// for them explicitly (lds_wait) before the MFMAs that use them.
template <int OFF>
__device__ __forceinline__ i16x4 tr_read(uint32_t addr) {
  static_assert(OFF >= 0 && OFF < 65536, "LDS instruction offset");
  i16x4 r;
  asm volatile("ds_read_b64_tr_b16 %0, %1 offset:%2" : "=v"(r) : "v"(addr), "n"(OFF));
  return r;
}
template <int OFF>
__device__ __forceinline__ f16x8 b128_read(uint32_t addr) {
  static_assert(OFF >= 0 && OFF < 65536, "LDS instruction offset");
  f16x8 r;
  asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(r) : "v"(addr), "n"(OFF));
  return r;
}

// A lane's LDS byte addresses of one operand's fragments inside a stage, for
// the wave's rows r0 .. r0 + 32 N - 1: everything but the stage's base and the
// k step.  KC: one address (row r0 + l%32); row block P adds 64 BK P bytes, k
// step ks flips the bits 32 ks (the chunk index is XOR-swizzled).  RC: one
// address per row block (the swizzle reaches the row block's bits); k step ks
// adds 32 ks ROWS bytes, the second half of a fragment (k + 4) 8 ROWS bytes.
template <bool RC, int ROWS, int BK, int N>
struct Frags {
  static constexpr int kReads = RC ? 2 : 1;  // LDS instructions per fragment
  uint32_t at[RC ? N : 1];
  __device__ __forceinline__ void init(int r0, int lane) {
    if constexpr (RC) {
      const int g = lane >> 4, i = lane & 15;
      const int k = (g >> 1) * 8 + (i >> 2);
#pragma unroll
      for (int p = 0; p < N; ++p) {
        const int m = r0 + p * 32 + (g & 1) * 16 + 4 * (i & 3);
        at[p] = (uint32_t)(k * ROWS * 2 + ((f_rc<ROWS>(k) ^ (m >> 3)) << 4) + (m & 7) * 2);
      }
    } else {
      const int row = r0 + (lane & 31);
      at[0] = (uint32_t)(row * BK * 2 + (((lane >> 5) ^ f_kc<BK>(row)) << 4));
    }
  }
  // Fragment P of k step KS from the operand's tile at LDS byte `tile`.
  template <int P, int KS>
  __device__ __forceinline__ f16x8 read(uint32_t tile) const {
    if constexpr (RC) {
      const i16x4 lo = tr_read<KS * 32 * ROWS>(tile + at[P]);
      const i16x4 hi = tr_read<KS * 32 * ROWS + 8 * ROWS>(tile + at[P]);
      const f16x4 a = __builtin_bit_cast(f16x4, lo), b = __builtin_bit_cast(f16x4, hi);
      return f16x8{a[0], a[1], a[2], a[3], b[0], b[1], b[2], b[3]};
    } else {
      return b128_read<P * 64 * BK>((tile + at[0]) ^ (KS * 32));
    }
  }
};

// Wait until at most N of this wave's LDS instructions are outstanding (they
// complete in order); wait for all of them; and pass a fragment through an empty
// asm after that wait so that its users cannot be scheduled before it.
template <int N>
__device__ __forceinline__ void lds_wait() {
  asm volatile("s_waitcnt lgkmcnt(%0)" ::"n"(N < 15 ? N : 15) : "memory");
}
__device__ __forceinline__ void lds_wait_all() { asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); }
__device__ __forceinline__ void after_wait(f16x8& v) { asm volatile("" : "+v"(v)); }

// ---------------------------------------------------------------------------
// The GEMM kernel.
// ---------------------------------------------------------------------------
enum class Epi {
  SwiGLU,         // c = o fp16 [m][n/2... per MapGateValue], optional u = [u_g | u_v]
  StoreF16,       // c fp16 = fp16(acc)
  SwiGLUBwd,      // c = du fp16 [m][2f] from u and d_o = fp16(acc)
  StoreF32OfF16,  // c fp32 = fp32(fp16(acc))
  AccF32OfF16,    // c fp32 (+)= fp32(fp16(acc))
  PartialF32,     // c fp32 partial [split][m][n] = acc
};

constexpr int kSplitStep = 64;  // weight gradients: granularity of a split's token range

struct GemmArgs {
  const __half* a; int64_t lda; int64_t a_bytes;   // source, row stride, bytes addressable
  const __half* b; int64_t ldb; int64_t b_bytes;
  int64_t m, n, k;         // C rows, C columns (B rows), reduction length
  int64_t k_chunk;         // tokens per split (multiple of kSplitStep); == k without split
  int64_t tiles_m, tiles_n;
  void* c; int64_t ldc;
  void* u; int64_t ldu;    // SwiGLU: optional u output; SwiGLUBwd: u input
  int64_t f;               // SwiGLU / SwiGLUBwd: value column offset
  int accumulate;          // AccF32OfF16
  int64_t group = 8;       // M tiles per group of the tile order (tile_of)
  int64_t valid;           // StoreF16: columns valid .. n - 1 are written as zero (0: none)
};

// Workgroups are dispatched to the 8 XCDs round robin.  Tiles are numbered in
// groups of `rows` M-tiles (M fastest inside a group), and each XCD receives a
// contiguous range of tile numbers, so the workgroups sharing one XCD's L2 at
// a time cover a compact block of M x N tiles.
__device__ __forceinline__ void tile_of(int64_t t, int64_t tiles_m, int64_t tiles_n,
                                        int64_t rows, int64_t& tm, int64_t& tn) {
  const int64_t tiles = tiles_m * tiles_n;
  if ((tiles & 7) == 0) t = (t & 7) * (tiles >> 3) + (t >> 3);
  const int64_t group = rows * tiles_n;
  const int64_t g = t / group, r = t % group;
  const int64_t first = g * rows;
  const int64_t gm = tiles_m - first < rows ? tiles_m - first : rows;
  tm = first + r % gm;
  tn = r / gm;
}

// f(integral_constant<int, 0>) .. f(integral_constant<int, N - 1>): loops whose
// index has to be a constant expression.
template <class F, int... I>
__device__ __forceinline__ void static_for_impl(F&& f, std::integer_sequence<int, I...>) {
  (f(std::integral_constant<int, I>{}), ...);
}
template <int N, class F>
__device__ __forceinline__ void static_for(F&& f) {
  static_for_impl(f, std::make_integer_sequence<int, N>{});
}

template <int SHAPE, bool A_RC, bool B_RC, Epi EPI>
__device__ __forceinline__ void gemm_block(const GemmArgs& args, int64_t block) {
  constexpr int BM = kShapes[SHAPE].bm, BN = kShapes[SHAPE].bn, WAVES = kShapes[SHAPE].waves;
  constexpr int BK = kShapes[SHAPE].bk, RA = kShapes[SHAPE].ra, RB = kShapes[SHAPE].rb;
  // waves: 2 rows x WCOLS columns, each owning a WM x WN block of the tile
  constexpr int WCOLS = WAVES / 2, WM = BM / 2, WN = BN / WCOLS;
  constexpr int TM = WM / 32, TN = WN / 32;
  static_assert(RB >= 2 && (RA == RB || RA == RB + 1), "ring depths");
  constexpr int kA = BM * BK, kB = BN * BK;      // halves per stage and operand
  constexpr int kRing = RA * kA + RB * kB;
  constexpr int kStaging = WAVES * WM * (WN + 8);  // fp16 epilogue staging (the fp32 one is less)
  static_assert(WAVES * 32 * (WN + 4) * 2 <= (kRing > kStaging ? kRing : kStaging),
                "fp32 epilogue staging");
  __shared__ __attribute__((aligned(1024))) _Float16 lds[kRing > kStaging ? kRing : kStaging];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm = wave / WCOLS, wn = wave % WCOLS;

  const int64_t tiles = args.tiles_m * args.tiles_n;
  const int64_t split = block / tiles;
  int64_t tm, tn;
  tile_of(block % tiles, args.tiles_m, args.tiles_n, args.group, tm, tn);
  const int64_t m0 = tm * BM;
  const int64_t n0 = (EPI == Epi::SwiGLU) ? tn * (BN / 2) : tn * BN;
  const int64_t kbeg = split * args.k_chunk;
  const int64_t kend = kbeg + args.k_chunk < args.k ? kbeg + args.k_chunk : args.k;
  const int stages =
      __builtin_amdgcn_readfirstlane(kend > kbeg ? (int)((kend - kbeg + BK - 1) / BK) : 0);
  const int ktail = (int)((kend - kbeg) % BK);  // values of a last, partial stage

  Dma<A_RC, BM, BK, WAVES> da;
  Dma<B_RC, BN, BK, WAVES> db;
  if constexpr (A_RC) da.init_rc(args.a, args.a_bytes, args.lda, m0, kbeg, wave, lane);
  else da.init_kc(args.a, args.a_bytes, args.lda, MapDirect{m0, args.m}, kbeg, wave, lane);
  if constexpr (B_RC) db.init_rc(args.b, args.b_bytes, args.ldb, n0, kbeg, wave, lane);
  else if constexpr (EPI == Epi::SwiGLU)
    db.init_kc(args.b, args.b_bytes, args.ldb, MapGateValue<BN, WCOLS>{n0, args.f}, kbeg, wave,
               lane);
  else db.init_kc(args.b, args.b_bytes, args.ldb, MapDirect{n0, args.n}, kbeg, wave, lane);

  f32x16 acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.f;

  // Rings: operand A's stage st lives in buffer st % RA, B's in st % RB (A may
  // be one stage deeper: it is the operand that streams from HBM, B a weight
  // that stays in L2).  A stage is BK / 16 k steps; each k step's fragments
  // are read during the k step before it.  Before its last k step a stage
  //   * waits for its own LDS reads (the last k step's fragments), for its own
  //     DMA of stage st + 1, and joins the workgroup: then all of stage st + 1
  //     has landed and no wave reads stage st any more;
  //   * from then on, until its next wait, issues B's stage st + RB and then A's
  //     stage st + RA into the two buffers just released ("window" st + RB).
  // A stage past the end is still issued, from a resource of zero bytes: it
  // reads nothing from memory and writes zeros into a buffer no later stage
  // uses, and every iteration waits for the same vmcnt.  Fragments prefetched
  // past the last stage are never used.
  //
  // The loop is bound by its waves' issue slots and by the path from L2 to
  // LDS, not by MFMA: with one wave per SIMD an LDS read or a DMA that finds
  // its queue full stalls the MFMAs behind it.  So both are spread evenly over
  // the MFMAs, and each MFMA waits only for its own fragments.
  constexpr int kPA = Dma<A_RC, BM, BK, WAVES>::kPerWave, kPB = Dma<B_RC, BN, BK, WAVES>::kPerWave;
  constexpr int kPerWave = kPA + kPB;
  constexpr int kInFlight = (RB - 2) * kPerWave + (RA - RB) * kPA;  // left at a stage's wait
  // DMA instructions of a window before its k step 0, 1 and 2 (the first ones
  // go into the last k step of the stage that released the buffers); with
  // equal rings of two the whole window has to land within the stage, and its
  // last k step issues none
  constexpr int kSteps = BK / 16 - (kInFlight ? 0 : 1);
  constexpr int kD0 = kPerWave / kSteps, kD1 = kPerWave * 2 / kSteps;
  constexpr int kD2 = BK == 64 ? kPerWave * 3 / kSteps : kPerWave;
  constexpr int kM = TM * TN, kF = TM + TN;
  Frags<A_RC, BM, BK, TM> fra;
  Frags<B_RC, BN, BK, TN> frb;
  fra.init(wm * WM, lane);
  frb.init(wn * WN, lane);
  const uint32_t lds_a = (uint32_t)(size_t)(RV_LDS void*)lds;
  const uint32_t lds_b = lds_a + RA * kA * 2;
  f16x8 fa[2][TM], fb[2][TN];
  __amdgpu_buffer_rsrc_t ra, rb;  // the window being issued
  int ia = 0, ib = 0;             // its buffers

  auto begin_a = [&](int st, int buf) {
    if constexpr (!A_RC)
      if (ktail != 0 && st == stages - 1) da.cut_kc(ktail, wave, lane);
    ra = da.stage(st, st < stages);
    ia = buf;
  };
  auto begin_b = [&](int st, int buf) {
    if constexpr (!B_RC)
      if (ktail != 0 && st == stages - 1) db.cut_kc(ktail, wave, lane);
    rb = db.stage(st, st < stages);
    ib = buf;
  };
  auto dma = [&](int d) {  // instruction d of a window: B's, then A's
    if (d < kPB) db.issue(rb, lds + RA * kA + ib * kB, d, wave);
    else da.issue(ra, lds + ia * kA, d - kPB, wave);
  };
  // Fragment reads go in the order the MFMAs need them: B 0, A 0, B 1 .. , A 1 ..
  auto read = [&](auto slot, auto ks, auto f, uint32_t ta, uint32_t tb) {
    constexpr int S = decltype(slot)::value, K = decltype(ks)::value, P = decltype(f)::value;
    if constexpr (P == 0) fb[S][0] = frb.template read<0, K>(tb);
    else if constexpr (P == 1) fa[S][0] = fra.template read<0, K>(ta);
    else if constexpr (P <= TN) fb[S][P - 1] = frb.template read<P - 1, K>(tb);
    else fa[S][P - TN] = fra.template read<P - TN, K>(ta);
  };
  constexpr auto reads_of = [](int f) {  // LDS instructions of fragment read f
    return f == 0 || (f > 1 && f <= TN) ? Frags<B_RC, BN, BK, TN>::kReads
                                         : Frags<A_RC, BM, BK, TM>::kReads;
  };
  // The MFMAs of fragment slot S, with the reads of k step K of the stage at
  // LDS bytes ta / tb into the other slot, and DMA instructions D0 .. D1 - 1,
  // spread between them at fixed points.  READY: this slot's reads are known
  // to be complete.
  auto kstep = [&](auto slot, auto knext, uint32_t ta, uint32_t tb, auto dfirst, auto dlast,
                   auto ready) {
    constexpr int S = decltype(slot)::value;
    constexpr int D0 = decltype(dfirst)::value, ND = decltype(dlast)::value - D0;
    constexpr bool READY = decltype(ready)::value;
    static_for<kM>([&](auto qc) {
      constexpr int q = decltype(qc)::value, i = q / TN, j = q % TN;
      if constexpr (!READY && (i == 0 || j == 0)) {
        // the last read this MFMA needs, and the LDS instructions after it
        constexpr int need = q == 0 ? 1 : i == 0 ? j + 1 : TN + i;
        constexpr int after = [&] {
          int n = 0;
          for (int f = need + 1; f < kF; ++f) n += reads_of(f);
          for (int f = 0; f < kF; ++f)
            if (f * kM / kF < q) n += reads_of(f);
          return n;
        }();
        lds_wait<after>();
        if constexpr (i == 0) after_wait(fb[S][j]);
        if constexpr (j == 0) after_wait(fa[S][i]);
      }
      acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(fb[S][j], fa[S][i], acc[i][j], 0, 0, 0);
      static_for<kF>([&](auto fc) {
        constexpr int f = decltype(fc)::value;
        if constexpr (f * kM / kF == q)
          read(std::integral_constant<int, S ^ 1>{}, knext, fc, ta, tb);
      });
#pragma unroll
      for (int d = 0; d < ND; ++d)
        if ((2 * d + 1) * kM / (ND ? 2 * ND : 1) == q) dma(D0 + d);
      __builtin_amdgcn_sched_barrier(0);
    });
  };
  using std::integral_constant;
  constexpr integral_constant<int, 0> c0{};
  constexpr integral_constant<int, 1> c1{};
  constexpr integral_constant<int, 2> c2{};
  constexpr integral_constant<int, 3> c3{};
  constexpr integral_constant<int, kD0> d0{};
  constexpr integral_constant<int, kD1> d1{};
  constexpr integral_constant<int, kD2> d2{};
  constexpr integral_constant<int, kPerWave> dn{};
  constexpr integral_constant<bool, false> pending{};
  constexpr integral_constant<bool, true> ready{};

  if (stages > 0) {
    if constexpr (RA > RB) {  // A's extra stage
      begin_a(0, 0);
#pragma unroll
      for (int d = kPB; d < kPerWave; ++d) dma(d);
    }
#pragma unroll
    for (int p = 0; p < RB; ++p) {  // windows 0 .. RB - 1, the last one's first part
      begin_b(p, p);
      begin_a(p + RA - RB, p + RA - RB);
#pragma unroll
      for (int d = 0; d < (p < RB - 1 ? kPerWave : kD0); ++d) dma(d);
    }
    wait_vmcnt<(RA - RB) * kPA + (RB - 2) * kPerWave + kD0>();
    lds_barrier();
    static_for<kF>([&](auto fc) { read(c0, c0, fc, lds_a, lds_b); });
  }
  int ca = 0, cb = 0;  // the stage's buffers
  for (int st = 0; st < stages; ++st) {
    const uint32_t ta = lds_a + ca * (kA * 2), tb = lds_b + cb * (kB * 2);
    kstep(c0, c1, ta, tb, d0, d1, pending);
    if constexpr (BK == 64) {
      kstep(c1, c2, ta, tb, d1, d2, pending);
      kstep(c0, c3, ta, tb, d2, dn, pending);
    }
    lds_wait_all();
#pragma unroll
    for (int i = 0; i < TM; ++i) after_wait(fa[1][i]);
#pragma unroll
    for (int j = 0; j < TN; ++j) after_wait(fb[1][j]);
    wait_vmcnt<kInFlight>();
    lds_barrier();
    begin_b(st + RB, cb);
    begin_a(st + RA, ca);
    ca = ca + 1 == RA ? 0 : ca + 1;
    cb = cb + 1 == RB ? 0 : cb + 1;
    kstep(c1, c0, lds_a + ca * (kA * 2), lds_b + cb * (kB * 2), c0, d0, ready);
  }
  lds_wait_all();  // the last prefetched fragments land before their registers are reused
#pragma unroll
  for (int i = 0; i < TM; ++i) after_wait(fa[0][i]);
#pragma unroll
  for (int j = 0; j < TN; ++j) after_wait(fb[0][j]);
  wait_vmcnt<0>();  // the trailing stages' zero writes land before the ring is reused
  __syncthreads();  // every wave is done with the ring before the epilogue reuses it

  // ---- epilogue ----
  // The MFMA is issued as B * A^T, so each lane holds C row (lane % 32) of
  // its 32x32 tile and, for q = 0..3, the 4 consecutive columns
  // q*8 + (lane/32)*4 + 0..3 (accumulator values 4q..4q+3).
  const int cq = (lane >> 5) * 4;
  if constexpr (EPI == Epi::PartialF32 || EPI == Epi::StoreF32OfF16 ||
                EPI == Epi::AccF32OfF16) {
    // fp32 outputs: each wave passes its block through LDS 32 rows at a time
    // (row stride WN + 4 floats: conflict free both ways), so that a store
    // instruction covers whole rows (512 or 256 contiguous bytes) instead of
    // 32-byte pieces of 32 rows.
    constexpr int S = WN + 4, CPR = WN / 4, RPP = 64 / CPR;
    float* stage = reinterpret_cast<float*>(lds) + wave * (32 * S);
    const int c = lane % CPR * 4;
    float* out = static_cast<float*>(args.c) + n0 + wn * WN + c;
    if constexpr (EPI == Epi::PartialF32) out += split * args.m * args.ldc;
#pragma unroll
    for (int i = 0; i < TM; ++i) {
#pragma unroll
      for (int j = 0; j < TN; ++j)
#pragma unroll
        for (int q = 0; q < 4; ++q)
          *reinterpret_cast<float4*>(stage + (lane & 31) * S + j * 32 + q * 8 + cq) =
              make_float4(acc[i][j][q * 4], acc[i][j][q * 4 + 1], acc[i][j][q * 4 + 2],
                          acc[i][j][q * 4 + 3]);
      lds_wait_all();
      __builtin_amdgcn_wave_barrier();
      const int64_t row0 = m0 + wm * WM + i * 32;
#pragma unroll 8
      for (int r = lane / CPR; r < 32; r += RPP) {
        const int64_t row = row0 + r;
        float4 v = *reinterpret_cast<const float4*>(stage + r * S + c);
        if (row >= args.m) continue;
        float4* dst = reinterpret_cast<float4*>(out + row * args.ldc);
        if constexpr (EPI != Epi::PartialF32) {
          v = make_float4(rv::round_to<__half>(v.x), rv::round_to<__half>(v.y),
                          rv::round_to<__half>(v.z), rv::round_to<__half>(v.w));
          if constexpr (EPI == Epi::AccF32OfF16) {
            if (args.accumulate) {
              const float4 p = *dst;
              v = make_float4(p.x + v.x, p.y + v.y, p.z + v.z, p.w + v.w);
            }
          }
        }
        *dst = v;
      }
      // the next 32 rows' writes follow these reads in the wave's LDS order
      __builtin_amdgcn_wave_barrier();
    }
  } else {
    // fp16 outputs: each wave stages fp16(acc) for its WM x WN block in LDS
    // (row stride WN + 8 halves), then moves whole rows, 16 bytes per lane,
    // so every global access instruction covers full row segments.  The
    // stores are streaming (nt): measured 1-5% faster per GEMM and 0.3-0.5%
    // per training step of the two decoders, consumers included.
    constexpr int S = WN + 8;
    _Float16* stage = lds + wave * (WM * S);
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const __half2 h01 = __floats2half2_rn(acc[i][j][q * 4], acc[i][j][q * 4 + 1]);
          const __half2 h23 = __floats2half2_rn(acc[i][j][q * 4 + 2], acc[i][j][q * 4 + 3]);
          uint2 p;
          p.x = *reinterpret_cast<const uint32_t*>(&h01);
          p.y = *reinterpret_cast<const uint32_t*>(&h23);
          *reinterpret_cast<uint2*>(stage + (i * 32 + (lane & 31)) * S + j * 32 + q * 8 + cq) = p;
        }
    // each wave reads back only its own staged block: a wave-local wait
    // instead of a workgroup barrier, so a wave stores as soon as it has staged
    lds_wait_all();
    __builtin_amdgcn_wave_barrier();
    const int64_t row0 = m0 + wm * WM;
    if constexpr (EPI == Epi::SwiGLU) {
      // gate in staged columns [0, WN/2), value in [WN/2, WN)
      constexpr int CPR = WN / 16, RPP = 64 / CPR;
      const int c = lane % CPR;
      __half* u = static_cast<__half*>(args.u);
      const int64_t col = n0 + wn * (WN / 2) + c * 8;
#pragma unroll 4
      for (int r = lane / CPR; r < WM; r += RPP) {
        const int64_t row = row0 + r;
        if (row >= args.m) break;
        const u32x4 gw = *reinterpret_cast<const u32x4*>(stage + r * S + c * 8);
        const u32x4 vw = *reinterpret_cast<const u32x4*>(stage + r * S + WN / 2 + c * 8);
        const __half* gh = reinterpret_cast<const __half*>(&gw);
        const __half2* vh2 = reinterpret_cast<const __half2*>(&vw);
        // silu rounded to fp16, times v: the exact product of two fp16 values
        // rounded once, so the packed fp16 multiply gives the fp32 expression's
        // bits two values per instruction
        __half2 oh[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float g0 = __half2float(gh[2 * e]), g1 = __half2float(gh[2 * e + 1]);
          const __half2 silu = __floats2half2_rn(g0 * rv::fast_sigmoid(g0),
                                                 g1 * rv::fast_sigmoid(g1));
          oh[e] = __hmul2(silu, vh2[e]);
        }
        __builtin_nontemporal_store(*reinterpret_cast<const u32x4*>(oh), reinterpret_cast<u32x4*>(static_cast<__half*>(args.c) + row * args.ldc + col));
        if (u != nullptr) {
          __builtin_nontemporal_store(gw, reinterpret_cast<u32x4*>(u + row * args.ldu + col));
          __builtin_nontemporal_store(vw, reinterpret_cast<u32x4*>(u + row * args.ldu + args.f + col));
        }
      }
    } else if constexpr (EPI == Epi::StoreF16) {
      constexpr int CPR = WN / 8, RPP = 64 / CPR;
      const int c = lane % CPR;
      const int64_t col = n0 + wn * WN + c * 8;
#pragma unroll 4
      for (int r = lane / CPR; r < WM; r += RPP) {
        const int64_t row = row0 + r;
        if (row >= args.m || col >= args.n) break;
        u32x4 dw = *reinterpret_cast<const u32x4*>(stage + r * S + c * 8);
        if (args.valid != 0 && col + 8 > args.valid) {
#pragma unroll
          for (int e = 0; e < 8; ++e)
            if (col + e >= args.valid)
              dw[e >> 1] = (e & 1) ? dw[e >> 1] & 0xffffu : dw[e >> 1] & 0xffff0000u;
        }
        __builtin_nontemporal_store(dw, reinterpret_cast<u32x4*>(static_cast<__half*>(args.c) + row * args.ldc + col));
      }
    } else {
      // SwiGLUBwd: du from u = [gate | value] and d_o = fp16(acc).  The u
      // reads of up to 16 of a lane's rows are issued together (the
      // accumulators are in LDS by now, their registers free), so the tile's
      // epilogue waits on one memory round trip per 16 rows instead of one
      // per 4; rows past m read the last row and store nothing.
      constexpr int CPR = WN / 8, RPP = 64 / CPR;
      constexpr int ITER = WM / RPP;              // rows per lane
      constexpr int CH = ITER < 16 ? ITER : 16;   // rows whose u reads are in flight together
      static_assert(ITER % CH == 0, "epilogue row chunks");
      const int c = lane % CPR;
      const int64_t col = n0 + wn * WN + c * 8;
      const __half* ubase = static_cast<const __half*>(args.u);
#pragma unroll
      for (int r0 = 0; r0 < ITER; r0 += CH) {
        u32x4 gw[CH], vw[CH];
#pragma unroll
        for (int i = 0; i < CH; ++i) {
          const int64_t rr = row0 + lane / CPR + (r0 + i) * RPP;
          const __half* ur = ubase + (rr < args.m ? rr : args.m - 1) * args.ldu;
          gw[i] = *reinterpret_cast<const u32x4*>(ur + col);
          vw[i] = *reinterpret_cast<const u32x4*>(ur + args.f + col);
        }
#pragma unroll
        for (int i = 0; i < CH; ++i) {
          const int r = lane / CPR + (r0 + i) * RPP;
          const int64_t row = row0 + r;
          if (row < args.m) {
            const u32x4 dw = *reinterpret_cast<const u32x4*>(stage + r * S + c * 8);
            const __half2* dh2 = reinterpret_cast<const __half2*>(&dw);
            const __half* gh = reinterpret_cast<const __half*>(&gw[i]);
            const __half2* vh2 = reinterpret_cast<const __half2*>(&vw[i]);
            // d*v and d*silu are products of two fp16 values rounded to fp16
            // once: packed fp16 multiplies, the same bits as the fp32 forms
            __half2 dgo[4], dvo[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              const float g0 = __half2float(gh[2 * e]), g1 = __half2float(gh[2 * e + 1]);
              const float s0 = rv::fast_sigmoid(g0), s1 = rv::fast_sigmoid(g1);
              const __half2 silu = __floats2half2_rn(g0 * s0, g1 * s1);
              const __half2 dgi = __hmul2(dh2[e], vh2[e]);
              dgo[e] = __floats2half2_rn(__low2float(dgi) * (s0 * (1.0f + g0 * (1.0f - s0))),
                                         __high2float(dgi) * (s1 * (1.0f + g1 * (1.0f - s1))));
              dvo[e] = __hmul2(dh2[e], silu);
            }
            __half* du = static_cast<__half*>(args.c) + row * args.ldc;
            __builtin_nontemporal_store(*reinterpret_cast<const u32x4*>(dgo), reinterpret_cast<u32x4*>(du + col));
            __builtin_nontemporal_store(*reinterpret_cast<const u32x4*>(dvo), reinterpret_cast<u32x4*>(du + args.f + col));
          }
        }
      }
    }
  }
}

template <int SHAPE, bool A_RC, bool B_RC, Epi EPI>
__global__ __launch_bounds__(kShapes[SHAPE].waves * 64,
                             kShapes[SHAPE].per_cu * kShapes[SHAPE].waves / 4)
void gemm_kernel(GemmArgs args) {
  gemm_block<SHAPE, A_RC, B_RC, EPI>(args, blockIdx.x);
}

// Two independent GEMMs in one launch: workgroups [0, first) run g[0], the rest
// g[1].  An MLP's two weight gradients: alone each is one workgroup per CU,
// together they fill the second place that the 128 x 128 and 64 x 128 tiles
// leave, so one's loads and partial sums overlap the other's MFMAs (both
// gradients and their reduce, us, two launches -> one: 51 x 256 x 1024 8.4 -> 4.7,
// 2048 x 256 x 1024 21.3 -> 16.8, 16896 x 256 x 1024 60.8 -> 53.8, 1000 x 768 x 3072
// 34.9 -> 27.7, 3062 x 1024 x 4096 100.7 -> 97.0, 32768 x 1024 x 4096 690 -> 687; tiles in
// groups of 8 on both sides, see wgrad_group).
struct GemmPair {
  GemmArgs g[2];
  int64_t first;
};
template <int SHAPE, Epi EPI>
__global__ __launch_bounds__(kShapes[SHAPE].waves * 64,
                             kShapes[SHAPE].per_cu * kShapes[SHAPE].waves / 4)
void wgrad_pair_kernel(GemmPair pair) {
  const int second = (int64_t)blockIdx.x >= pair.first;
  gemm_block<SHAPE, true, true, EPI>(pair.g[second], blockIdx.x - (second ? pair.first : 0));
}

// Explicit instantiations of every (tile shape, operand layout, epilogue) the
// host dispatch can launch.  Without them this compiler emits the host-side
// launch stubs of only some of the kernels reached through the dispatch
// switch, and the library fails to load with undefined symbols.
#define RV_ACT_KERNELS(SHAPE)                                                        \
  template __global__ void gemm_kernel<SHAPE, false, false, Epi::SwiGLU>(GemmArgs);   \
  template __global__ void gemm_kernel<SHAPE, false, false, Epi::StoreF16>(GemmArgs); \
  template __global__ void gemm_kernel<SHAPE, false, true, Epi::SwiGLUBwd>(GemmArgs); \
  template __global__ void gemm_kernel<SHAPE, false, true, Epi::StoreF16>(GemmArgs);  \
  template __global__ void gemm_kernel<SHAPE, false, true, Epi::StoreF32OfF16>(GemmArgs); \
  template __global__ void gemm_kernel<SHAPE, false, false, Epi::PartialF32>(GemmArgs);  \
  template __global__ void gemm_kernel<SHAPE, false, true, Epi::PartialF32>(GemmArgs);
#define RV_WGRAD_KERNELS(SHAPE)                                                       \
  template __global__ void gemm_kernel<SHAPE, true, true, Epi::AccF32OfF16>(GemmArgs); \
  template __global__ void gemm_kernel<SHAPE, true, true, Epi::StoreF16>(GemmArgs);      \
  template __global__ void gemm_kernel<SHAPE, true, true, Epi::PartialF32>(GemmArgs);    \
  template __global__ void wgrad_pair_kernel<SHAPE, Epi::AccF32OfF16>(GemmPair);         \
  template __global__ void wgrad_pair_kernel<SHAPE, Epi::PartialF32>(GemmPair);
RV_ACT_KERNELS(0) RV_ACT_KERNELS(1) RV_ACT_KERNELS(2) RV_ACT_KERNELS(3)
RV_ACT_KERNELS(4) RV_ACT_KERNELS(5) RV_ACT_KERNELS(6)
RV_WGRAD_KERNELS(0) RV_WGRAD_KERNELS(1) RV_WGRAD_KERNELS(2) RV_WGRAD_KERNELS(3)
static_assert(kNumShapes == 7 && kRuleShapes == 4, "instantiations above");

// acc[i] (+)= fp32(fp16(sum_s part[s][i])), splits summed in order.  This is
// autocast's weight gradient: the fp16 GEMM result, cast to the fp32 weight
// and added to the running per-tile sum.  n % 4 == 0.  One launch finishes up
// to two weight gradients: blocks [0, a.blocks) reduce segment a, the rest b.
struct ReduceSeg {
  const float* part;
  float* out;
  int64_t n;
  int splits;
  int64_t blocks;  // 0: nothing to reduce
};

__global__ __launch_bounds__(256)
void wgrad_reduce(ReduceSeg a, ReduceSeg b, int accumulate) {
  const bool second = (int64_t)blockIdx.x >= a.blocks;
  const float* part = second ? b.part : a.part;
  float* out = second ? b.out : a.out;
  const int64_t n = second ? b.n : a.n;
  const int splits = second ? b.splits : a.splits;
  const int64_t blk = second ? (int64_t)blockIdx.x - a.blocks : (int64_t)blockIdx.x;
  const int64_t i = (blk * 256 + threadIdx.x) * 4;
  if (i >= n) return;
  float4 s = *reinterpret_cast<const float4*>(part + i);
  // the partials of eight splits loaded before the first of their adds (one
  // memory round trip per eight splits instead of per split); same order
  int k = 1;
  for (; k + 8 <= splits; k += 8) {
    float4 t[8];
#pragma unroll
    for (int j = 0; j < 8; ++j)
      t[j] = *reinterpret_cast<const float4*>(part + (int64_t)(k + j) * n + i);
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      s.x = s.x + t[j].x; s.y = s.y + t[j].y; s.z = s.z + t[j].z; s.w = s.w + t[j].w;
    }
  }
  for (; k < splits; ++k) {
    const float4 t = *reinterpret_cast<const float4*>(part + (int64_t)k * n + i);
    s.x = s.x + t.x; s.y = s.y + t.y; s.z = s.z + t.z; s.w = s.w + t.w;
  }
  float4 r = make_float4(rv::round_to<__half>(s.x), rv::round_to<__half>(s.y),
                         rv::round_to<__half>(s.z), rv::round_to<__half>(s.w));
  float4* o = reinterpret_cast<float4*>(out + i);
  if (accumulate) {
    const float4 p = *o;
    r = make_float4(p.x + r.x, p.y + r.y, p.z + r.z, p.w + r.w);
  }
  *o = r;
}

// An activation GEMM's split-K finish: out[i] = fp16(sum_s part[s][i]), splits
// summed in order, stored as fp16 or as that value widened to fp32.  n % 4 == 0.
template <typename T>
__global__ __launch_bounds__(256)
void act_reduce(const float* __restrict__ part, T* __restrict__ out, int64_t n, int splits) {
  const int64_t i = ((int64_t)blockIdx.x * 256 + threadIdx.x) * 4;
  if (i >= n) return;
  float4 s = *reinterpret_cast<const float4*>(part + i);
  int k = 1;
  for (; k + 4 <= splits; k += 4) {  // four splits' loads in flight, added in order
    float4 t[4];
#pragma unroll
    for (int j = 0; j < 4; ++j)
      t[j] = *reinterpret_cast<const float4*>(part + (int64_t)(k + j) * n + i);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      s.x = s.x + t[j].x; s.y = s.y + t[j].y; s.z = s.z + t[j].z; s.w = s.w + t[j].w;
    }
  }
  for (; k < splits; ++k) {
    const float4 t = *reinterpret_cast<const float4*>(part + (int64_t)k * n + i);
    s.x = s.x + t.x; s.y = s.y + t.y; s.z = s.z + t.z; s.w = s.w + t.w;
  }
  const __half2 lo = __floats2half2_rn(s.x, s.y), hi = __floats2half2_rn(s.z, s.w);
  if constexpr (std::is_same<T, float>::value) {
    *reinterpret_cast<float4*>(out + i) =
        make_float4(__low2float(lo), __high2float(lo), __low2float(hi), __high2float(hi));
  } else {
    uint2 v;
    v.x = *reinterpret_cast<const uint32_t*>(&lo);
    v.y = *reinterpret_cast<const uint32_t*>(&hi);
    *reinterpret_cast<uint2*>(out + i) = v;
  }
}

// dst = fp16(src), round to nearest even; 8 elements per thread.
__global__ __launch_bounds__(256)
void cast_f32_f16(const float* __restrict__ src, __half* __restrict__ dst, int64_t n) {
  const int64_t stride = (int64_t)gridDim.x * 256 * 8;
  for (int64_t i = ((int64_t)blockIdx.x * 256 + threadIdx.x) * 8; i < n; i += stride) {
    if (i + 8 <= n) {
      const float4 a = *reinterpret_cast<const float4*>(src + i);
      const float4 b = *reinterpret_cast<const float4*>(src + i + 4);
      const __half2 h0 = __floats2half2_rn(a.x, a.y), h1 = __floats2half2_rn(a.z, a.w);
      const __half2 h2 = __floats2half2_rn(b.x, b.y), h3 = __floats2half2_rn(b.z, b.w);
      uint4 v;
      v.x = *reinterpret_cast<const uint32_t*>(&h0);
      v.y = *reinterpret_cast<const uint32_t*>(&h1);
      v.z = *reinterpret_cast<const uint32_t*>(&h2);
      v.w = *reinterpret_cast<const uint32_t*>(&h3);
      *reinterpret_cast<uint4*>(dst + i) = v;
    } else {
      for (int64_t j = i; j < n; ++j) dst[j] = __float2half_rn(src[j]);
    }
  }
}

// dst[t] = fp16(src[t]) for up to kCastTensors tensors in one launch: the
// pointer table and per-tensor chunk prefix sums travel in the kernel
// arguments; each workgroup casts one chunk of one tensor with cast_f32_f16's
// arithmetic.  A chunk is one pass of the workgroup (2048 elements) as long as
// that gives at most kCastBlocks workgroups, so a decoder's few million
// weights occupy the whole chip (chunks of 32768 elements left half of it
// idle: 28 tensors, 5.2 M elements 10.1 -> 7.9 us; 48 tensors, 151 M elements 233 ->
// 224), and more passes above.
constexpr int kCastTensors = 64;
constexpr int64_t kCastPass = 256 * 8;
constexpr int64_t kCastBlocks = 16384;
struct CastTable {
  const float* src[kCastTensors];
  __half* dst[kCastTensors];
  int64_t n[kCastTensors];
  int chunk_start[kCastTensors + 1];
  int count;
  int64_t chunk;
};

__global__ __launch_bounds__(256)
void cast_multi_k(CastTable tab) {
  int t = 0, above = tab.count;  // last t with chunk_start[t] <= blockIdx.x
  while (above - t > 1) {
    const int mid = (t + above) >> 1;
    if (tab.chunk_start[mid] <= (int)blockIdx.x) t = mid;
    else above = mid;
  }
  const int64_t base = (int64_t)(blockIdx.x - tab.chunk_start[t]) * tab.chunk;
  const int64_t n = tab.n[t];
  const float* src = tab.src[t];
  __half* dst = tab.dst[t];
  const int64_t end = base + tab.chunk < n ? base + tab.chunk : n;
  for (int64_t i = base + threadIdx.x * 8; i < end; i += kCastPass) {
    if (i + 8 <= end) {
      const float4 a = *reinterpret_cast<const float4*>(src + i);
      const float4 b = *reinterpret_cast<const float4*>(src + i + 4);
      const __half2 h0 = __floats2half2_rn(a.x, a.y), h1 = __floats2half2_rn(a.z, a.w);
      const __half2 h2 = __floats2half2_rn(b.x, b.y), h3 = __floats2half2_rn(b.z, b.w);
      uint4 v;
      v.x = *reinterpret_cast<const uint32_t*>(&h0);
      v.y = *reinterpret_cast<const uint32_t*>(&h1);
      v.z = *reinterpret_cast<const uint32_t*>(&h2);
      v.w = *reinterpret_cast<const uint32_t*>(&h3);
      *reinterpret_cast<uint4*>(dst + i) = v;
    } else {
      for (int64_t j = i; j < end; ++j) dst[j] = __float2half_rn(src[j]);
    }
  }
}

// ---------------------------------------------------------------------------
// Host side: tile-shape choice and launches.
// ---------------------------------------------------------------------------
template <bool A_RC, bool B_RC, Epi EPI>
int launch(int shape, const GemmArgs& a, int64_t splits, hipStream_t s) {
  constexpr bool kWgrad = A_RC;  // weight gradients use the rule's shapes only
  const dim3 grid((unsigned)(a.tiles_m * a.tiles_n * splits)), block(kShapes[shape].waves * 64);
#define RV_LAUNCH(SHAPE) \
  hipLaunchKernelGGL((gemm_kernel<SHAPE, A_RC, B_RC, EPI>), grid, block, 0, s, a)
  switch (shape) {
    case 0: RV_LAUNCH(0); break;
    case 1: RV_LAUNCH(1); break;
    case 2: RV_LAUNCH(2); break;
    case 3: RV_LAUNCH(3); break;
    default:
      if constexpr (kWgrad) return RV_ERR_UNSUPPORTED;
      else if (shape == 4) RV_LAUNCH(4);
      else if (shape == 5) RV_LAUNCH(5);
      else RV_LAUNCH(6);
  }
#undef RV_LAUNCH
  return rv_host::check_launch();
}

// Activation GEMMs: C is m x n_out where n_out = n (or n/2 output columns for
// SwiGLU, whose tile covers bn/2 of them).  The largest tile that gives at
// least one workgroup per CU; otherwise the one with the most workgroups.
int pick_act(int64_t m, int64_t n_cols, bool swiglu, int64_t splits) {
  int best = -1;
  int64_t best_blocks = -1;
  for (int i = 0; i < kRuleShapes; ++i) {
    const int64_t cols = swiglu ? kShapes[i].bn / 2 : kShapes[i].bn;
    if (n_cols % cols) continue;
    const int64_t blocks = ((m + kShapes[i].bm - 1) / kShapes[i].bm) * (n_cols / cols) * splits;
    if (blocks >= kCUs) return i;
    if (blocks > best_blocks) best = i, best_blocks = blocks;
  }
  return best;
}

// Measured tile choice.  The fastest tile shape of an activation GEMM depends
// on more than the grid size (how the last round of workgroups fills the
// chip, two workgroups per CU overlapping one's epilogue with the other's
// MFMAs, the k loop's length), and the shape never changes a result bit: every
// output element sums its k blocks in the same order in every shape.  So the
// first call for each (epilogue and its outputs, operand layouts, m, n, k)
// times every shape that fits (one warm-up launch, then two timed ones on the
// caller's stream, which is synchronised after each shape), the three fastest
// of them once more (each shape's faster time counting), and keeps the fastest:
// at most 30 launches.  64-row tiles are left out of products of four rounds of
// 256 x 256 tiles and more, where they take 1.4 times the best shape or longer.
// First forward and backward of an MLP at a new row count, ms (all seven shapes
// twice -> this): 32768 x 1024 x 4096 85.9 -> 51.9, 3062 x 1024 x 4096 13.0 -> 8.9.  The
// epilogues tuned here overwrite their outputs, so the extra launches write the
// same values.  A call made while its stream is being captured into a graph
// never tunes (that would synchronise): it takes the shape already chosen for
// its key, else pick_act's rule.  RV_GEMM_TUNE=0 in the environment turns tuning
// off.
using TuneKey = std::tuple<int, int, int, int64_t, int64_t, int64_t>;
std::atomic<int> g_forced_shape{-1};  // rv_gemm_force_shape; -1: measured / rule choice
std::mutex g_tune_mu;
std::map<TuneKey, int> g_tuned;

bool tuning_enabled() {
  static const bool on = [] {
    const char* v = std::getenv("RV_GEMM_TUNE");
    return !(v && v[0] == '0');
  }();
  return on;
}

bool capturing(hipStream_t s) {
  hipStreamCaptureStatus st = hipStreamCaptureStatusNone;
  if (hipStreamIsCapturing(s, &st) != hipSuccess) return true;  // then do not tune
  return st != hipStreamCaptureStatusNone;
}

// a.k_chunk < a.k: split-K, one partial (Epi::PartialF32) per k_chunk of k.
template <bool A_RC, bool B_RC, Epi EPI>
int launch_shape(int shape, GemmArgs a, int64_t n_cols, hipStream_t s) {
  const bool swiglu = EPI == Epi::SwiGLU;
  const TileShape t = kShapes[shape];
  a.tiles_m = (a.m + t.bm - 1) / t.bm;
  const int64_t cols = swiglu ? t.bn / 2 : t.bn;
  a.tiles_n = (n_cols + cols - 1) / cols;
  return launch<A_RC, B_RC, EPI>(shape, a, (a.k + a.k_chunk - 1) / a.k_chunk, s);
}

template <bool A_RC, bool B_RC, Epi EPI>
int tune_act(const GemmArgs& a, int64_t n_cols, hipStream_t s, int fallback) {
  const bool swiglu = EPI == Epi::SwiGLU;
  hipEvent_t e0, e1;
  if (hipEventCreate(&e0) != hipSuccess) return fallback;
  if (hipEventCreate(&e1) != hipSuccess) {
    (void)hipEventDestroy(e0);
    return fallback;
  }
  // two sweeps over the shapes, each shape keeping its faster one: a clock or
  // cache transient during one sweep does not decide the choice alone
  const int64_t wide = swiglu ? 128 : 256;
  const bool large = (a.m + 255) / 256 * ((n_cols + wide - 1) / wide) >= 4 * kCUs;
  float ms_of[kNumShapes] = {};
  for (int sweep = 0; sweep < 2; ++sweep) {
    float first[kNumShapes];
    std::copy(ms_of, ms_of + kNumShapes, first);
    for (int i = 0; i < kNumShapes; ++i) {
      const int64_t cols = swiglu ? kShapes[i].bn / 2 : kShapes[i].bn;
      if (n_cols % cols || (large && kShapes[i].bm == 64)) continue;
      int faster = 0;  // shapes ahead of this one in the first sweep
      for (int j = 0; j < kNumShapes; ++j)
        faster += first[j] > 0.f && (first[i] == 0.f || first[j] < first[i]);
      if (sweep == 1 && faster >= 3) continue;
      if (launch_shape<A_RC, B_RC, EPI>(i, a, n_cols, s) != RV_OK) continue;
      bool ok = hipEventRecord(e0, s) == hipSuccess;
      ok = ok && launch_shape<A_RC, B_RC, EPI>(i, a, n_cols, s) == RV_OK;
      ok = ok && launch_shape<A_RC, B_RC, EPI>(i, a, n_cols, s) == RV_OK;
      ok = ok && hipEventRecord(e1, s) == hipSuccess && hipEventSynchronize(e1) == hipSuccess;
      float ms = 0.f;
      ok = ok && hipEventElapsedTime(&ms, e0, e1) == hipSuccess;
      if (ok && ms > 0.f && (ms_of[i] == 0.f || ms < ms_of[i])) ms_of[i] = ms;
    }
  }
  int best = fallback;
  float best_ms = 0.f;
  for (int i = 0; i < kNumShapes; ++i)
    if (ms_of[i] > 0.f && (best_ms == 0.f || ms_of[i] < best_ms)) best = i, best_ms = ms_of[i];
  (void)hipEventDestroy(e0);
  (void)hipEventDestroy(e1);
  return best;
}

// fixed >= 0: the tile shape, chosen by the caller (no timing).  ragged: the tile's
// width need not divide n_cols (the epilogue checks columns).
template <bool A_RC, bool B_RC, Epi EPI>
int run_act(GemmArgs a, int64_t n_cols, hipStream_t s, int fixed = -1, bool ragged = false) {
  const bool swiglu = EPI == Epi::SwiGLU;
  if (EPI != Epi::PartialF32) a.k_chunk = a.k;
  const int64_t splits = (a.k + a.k_chunk - 1) / a.k_chunk;
  const int forced = g_forced_shape.load();
  if (forced >= 0) fixed = forced;
  if (fixed >= 0) {
    if (n_cols % (swiglu ? kShapes[fixed].bn / 2 : kShapes[fixed].bn) && !ragged)
      return RV_ERR_UNSUPPORTED;
    return launch_shape<A_RC, B_RC, EPI>(fixed, a, n_cols, s);
  }
  int shape = pick_act(a.m, n_cols, swiglu, splits);
  if (shape < 0) return RV_ERR_UNSUPPORTED;
  if (tuning_enabled()) {
    int device = 0;
    (void)hipGetDevice(&device);
    // the SwiGLU epilogue with and without its u output store different
    // amounts and are tuned apart
    const int variant = (EPI == Epi::SwiGLU && a.u != nullptr) ? 1 : 0;
    const TuneKey key{(int)EPI * 4 + (A_RC ? 2 : 0) + (B_RC ? 1 : 0), device, variant, a.m,
                      n_cols, EPI == Epi::PartialF32 ? a.k * 64 + splits : a.k};
    std::lock_guard<std::mutex> lock(g_tune_mu);
    const auto it = g_tuned.find(key);
    if (it != g_tuned.end()) {
      shape = it->second;
    } else if (!capturing(s)) {
      shape = tune_act<A_RC, B_RC, EPI>(a, n_cols, s, shape);
      g_tuned[key] = shape;
    }
  }
  return launch_shape<A_RC, B_RC, EPI>(shape, a, n_cols, s);
}

// Split count of an activation GEMM without a fused epilogue: the reduction is
// cut into `splits` partials (fp32, summed in order by act_reduce) when few
// output tiles would leave most CUs idle behind a long serial k loop.  Modelled
// on the 64 x 128 tile: 0.33 us per 64 of k for up to one workgroup per CU,
// against 4.5 us for the second launch and the partials' traffic (8 bytes each
// at 5 TB/s); a split has to save a fifth.  Measured (us, unsplit -> best count):
// 51 x 256 x 2048 (m, n, k) 12.9 -> 7.4, 51 x 1024 x 4096 23.0 -> 9.0, 512 x 1024 x
// 4096 23.5 -> 13.9, 1024 x 1024 x 8192 44.9 -> 30.1; not worth it: 51 x 256 x 1024
// 7.9 (6.8), 4096 x 256 x 2048 13.8 (15.8), 2331 x 512 x 1536 11.3 (16.0), 3062 x 1024 x
// 8192 70 (66), 8192 x 1024 x 4096 67 (76).  Depends on the sizes only, so a
// recomputed product has the same bits.
int64_t act_splits(int64_t m, int64_t n, int64_t k) {
  const int64_t tiles = ((m + 63) / 64) * (n / 128);
  if (tiles <= 0 || tiles > kCUs / 2) return 1;
  const double stages = (double)k / kSplitStep * 0.33;
  int64_t best = 1;
  double best_us = 0.8 * stages;
  for (int64_t s = 2; s <= 32 && k / s >= 2 * kSplitStep; ++s) {
    const int64_t wgs = tiles * s;
    const double us = stages / s * (wgs > kCUs ? (double)wgs / kCUs : 1.0) + 4.5 +
                      8.0 * m * n * s / 5e6;
    if (us < best_us) best = s, best_us = us;
  }
  return best;
}
int64_t act_chunk(int64_t m, int64_t n, int64_t k) {
  const int64_t splits = act_splits(m, n, k);
  return ((k + splits - 1) / splits + kSplitStep - 1) / kSplitStep * kSplitStep;
}
// 0 (no split) also for sizes that the split entry points do not take; an unsplit
// one may take them (rv_mlp_down and rv_mlp_dx: reductions of any multiple of 32).
int64_t act_part_bytes(int64_t m, int64_t n, int64_t k) {
  if (n % 128 || k % 128) return 0;
  const int64_t chunk = act_chunk(m, n, k), splits = (k + chunk - 1) / chunk;
  return splits > 1 ? splits * m * n * (int64_t)sizeof(float) : 0;
}

// a.k_chunk set; fp32 partials of each chunk in `part`, summed into out.
template <bool B_RC, typename T>
int run_split(GemmArgs a, T* out, float* part, hipStream_t s, int fixed = -1) {
  a.c = part;
  a.ldc = a.n;
  const int st = run_act<false, B_RC, Epi::PartialF32>(a, a.n, s, fixed);
  if (st != RV_OK) return st;
  const int64_t n = a.m * a.n, splits = (a.k + a.k_chunk - 1) / a.k_chunk;
  hipLaunchKernelGGL(act_reduce<T>, dim3((unsigned)((n / 4 + 255) / 256)), dim3(256), 0, s, part,
                     out, n, (int)splits);
  return rv_host::check_launch();
}

// Weight-gradient plan for an ni x nj output reduced over `rows` tokens: tile
// shape and split count minimising a simple cost (MFMA time at a per-shape
// efficiency, divided by the fraction of the grid's CU rounds that hold a
// workgroup, plus the partial sums' HBM round trip at ~250 flop per byte; at
// 500 the 8192-token tiles' weight gradients kept fewer splits on smaller
// tiles and took 45.3 us (d 256, f 1024) and 267 us (d 1024, f 4096) against
// 42.6 and 261 us).
// A grid past the CU count runs in rounds of all places (CUs times workgroups
// per CU): 540 workgroups of 64 x 128 tiles, priced as three rounds of the CUs, took
// 533 us (30791 rows, 6912 x 640) where 270 of 128 x 128 take 364.
// The split count is the largest that keeps tiles x splits within one round
// of the CUs: a grid a few workgroups past the CU count (C5's qkv weight
// gradient: 96 tiles x 3 splits = 288) leaves those CUs a second turn and
// nearly doubles the kernel.  Depends only on the sizes, so results are
// device-independent.
struct WgradPlan {
  int shape;
  int64_t tiles_m, tiles_n, splits, chunk;
};
bool plan_shape(int i, int64_t rows, int64_t ni, int64_t nj, WgradPlan& plan, double& cost,
                bool ragged = false) {
  // per-shape efficiencies measured on the split-K weight gradients (the
  // 128 x 256 tile's 0.55: at C5's attention-projection shape, 1024 x 1024
  // over 32768 tokens, it took 113 us with 8 splits where 256 x 256 with 16
  // takes 85 us, partial sums and their reduce included; the 64 x 128 tile's
  // 0.42: with half the splits of 128 x 128 it takes 21.4 us against 24.4 for 768
  // x 256 over 16896 tokens, 22.0 against 24.8 for 2048 x 256 over 8192, 13.3
  // against 16.4 for 1536 x 512 over 2331, but 41.2 against 34.7 for 2048 x 256
  // over 16896)
  static const double eff[kRuleShapes] = {0.8, 0.55, 0.5, 0.42};
  const TileShape t = kShapes[i];
  if ((ni % t.bm && !ragged) || nj % t.bn) return false;
  const int64_t tiles_i = (ni + t.bm - 1) / t.bm, tiles = tiles_i * (nj / t.bn);
  int64_t splits = tiles >= kCUs ? 1 : kCUs / tiles;
  const int64_t max_splits = (rows + 2 * kSplitStep - 1) / (2 * kSplitStep);
  if (splits > max_splits) splits = max_splits;
  if (splits > 64) splits = 64;
  if (splits < 1) splits = 1;
  int64_t chunk = (rows + splits - 1) / splits;
  chunk = (chunk + kSplitStep - 1) / kSplitStep * kSplitStep;
  splits = (rows + chunk - 1) / chunk;
  const int64_t wgs = tiles * splits, places = wgs > kCUs ? kCUs * t.per_cu : kCUs;
  const int64_t rounds = (wgs + places - 1) / places;
  const double fill = (double)wgs / (double)(rounds * places);
  const double flops = 2.0 * rows * ni * nj / (eff[i] * fill);
  const double bytes = splits > 1 ? 8.0 * splits * ni * nj : 0.0;
  cost = flops + 250.0 * bytes;
  plan = WgradPlan{i, tiles_i, nj / t.bn, splits, chunk};
  return true;
}
// ragged: ni need not be a multiple of the tile (rows past it are not stored).
WgradPlan plan_wgrad(int64_t rows, int64_t ni, int64_t nj, bool ragged = false) {
  WgradPlan best{-1, 0, 0, 0, 0}, plan;
  double best_cost = 0, cost;
  for (int i = 0; i < kRuleShapes; ++i)
    if (plan_shape(i, rows, ni, nj, plan, cost, ragged)) {
      // alone, 64 x 128 tiles whose number 8 does not divide (tile_of deals them to
      // the XCDs one by one) rate 0.35 once the operands are past the L2s (4 MB an
      // XCD): 384 x 384 over 30844 rows 38 us, 128 x 128 tiles 30; 384 x 768 over 16595
      // 35 and 32, but 896 x 896 over 2093 with qkv's 36 and 41
      if (i == 3 && !ragged && plan.tiles_m * plan.tiles_n % 8 &&
          rows * (ni + nj) * 2 > (int64_t)16 << 20)
        cost *= 0.42 / 0.35;
      if (best.shape >= 0 && cost >= best_cost) continue;
      best = plan;
      best_cost = cost;
    }
  return best;
}

// The plans of two weight gradients over the same rows (a: ai x aj, b: bi x
// bj).  With one tile shape for both they share a launch (launch_pair): the
// shape with the least total cost among those whose two plans are both split
// or both not, as long as that is no more than kPairCost of what the two cost
// with a shape each.  (Each cost is of the product alone: two workgroups per CU
// fill places that each product leaves idle.  256 x 256 tiles run one per CU, and
// share a launch only where they are both products' own shape.)  Measured, us,
// joint / apart, by the ratio of the costs: 1.00 23.9 / 27.8 (3483 rows, d 128, f
// 3584), 1.21 34.3 / 47.2 (2845, 384, 2944), 1.35 32.8 / 45.7 (3000, 768, 1408); 1.44
// 350 / 268 (19018, 768, 2432), 1.93 20.2 / 16.3 (307, 896, 768), 2.36 372 / 287 (32768,
// 768, 1408); 256 x 256 tiles 1.18 78.6 / 64.5 (4325 rows, qkv and proj of 1024).  Over
// 164 pairs, against two launches with a plan each of the fixed 0.35 weighting
// this one replaced: 0.71 on average and none above 1.0 (without a line 0.73, worst
// 1.40).
constexpr double kPairCost = 1.4;
struct PairPlan {
  WgradPlan a, b;
  bool paired;
};
PairPlan plan_pair(int64_t rows, int64_t ai, int64_t aj, int64_t bi, int64_t bj) {
  PairPlan best{plan_wgrad(rows, ai, aj), plan_wgrad(rows, bi, bj), false};
  if (best.a.shape < 0 || best.b.shape < 0) return best;
  double least = 0, ca, cb;
  WgradPlan a, b;
  plan_shape(best.a.shape, rows, ai, aj, a, ca);
  plan_shape(best.b.shape, rows, bi, bj, b, cb);
  const double apart = ca + cb;
  for (int i = 0; i < kRuleShapes; ++i) {
    if (!plan_shape(i, rows, ai, aj, a, ca) || !plan_shape(i, rows, bi, bj, b, cb)) continue;
    if ((a.splits > 1) != (b.splits > 1)) continue;
    if (ca + cb > (kShapes[i].per_cu > 1 ? kPairCost : 1.0) * apart) continue;
    if (!best.paired || ca + cb < least) {
      best = PairPlan{a, b, true};
      least = ca + cb;
    }
  }
  return best;
}

// One weight-gradient GEMM, planned: unsplit it writes (or adds) the result
// itself; split, its fp32 partial sums go to `part` and `seg` describes the
// reduction still to launch (seg.blocks == 0 otherwise).
struct WgradJob {
  WgradPlan plan;
  GemmArgs g;
  ReduceSeg seg;
};
// M tiles per group of a weight gradient's tile order.  Each XCD gets an eighth
// of every split's tiles, a contiguous range of their order: the group makes
// that range as square as the shapes allow, so that its L2 fetches the fewest
// distinct rows of the two operands.  us, groups of 8 -> this rule (an MLP's two
// gradients, rows x d x f): 8192 x 256 x 1024 30.7 -> 27.9, 16896 x 256 x 1024 52.0 -> 48.9,
// 20000 x 384 x 1536 119 -> 109, 32768 x 1024 x 4096 689 -> 676, 8192 x 1024 x 4096 212.2 ->
// 213.8, 51 x 256 x 1024 4.7 either way.  The activation products keep 8 (up, down, dgate
// and dx at 32768 x 1024 x 4096: 8 is the fastest or within 2% of it among 1 .. 32).
int64_t wgrad_group(const WgradPlan& p) {
  const int64_t tiles = p.tiles_m * p.tiles_n, share = tiles / 8;
  if (tiles % 8) return 8;
  int64_t best = 8, least = 0;
  for (int64_t g = 8; g >= 1; g /= 2) {
    int64_t n = (share + g - 1) / g;
    if (n > p.tiles_n) n = p.tiles_n;
    const int64_t rows = (share + n - 1) / n * kShapes[p.shape].bm + n * kShapes[p.shape].bn;
    if (least == 0 || rows < least) best = g, least = rows;
  }
  return best;
}
WgradJob plan_job(const WgradPlan& p, const __half* a, int64_t lda, const __half* b, int64_t ldb,
                  int64_t rows, int64_t ni, int64_t nj, float* out, int accumulate, float* part) {
  WgradJob j{p, {}, {nullptr, nullptr, 0, 0, 0}};
  if (p.shape < 0) return j;
  GemmArgs& g = j.g;
  g.a = a; g.lda = lda; g.a_bytes = rows * lda * 2;
  g.b = b; g.ldb = ldb; g.b_bytes = rows * ldb * 2;
  g.m = ni; g.n = nj; g.k = rows; g.k_chunk = p.chunk;
  g.tiles_m = p.tiles_m; g.tiles_n = p.tiles_n; g.group = wgrad_group(p);
  g.ldc = nj; g.accumulate = accumulate;
  g.c = p.splits == 1 ? out : part;
  if (p.splits > 1) {
    const int64_t n = ni * nj;
    j.seg = ReduceSeg{part, out, n, (int)p.splits, (n / 4 + 255) / 256};
  }
  return j;
}
int launch_job(const WgradJob& j, hipStream_t s) {
  if (j.plan.shape < 0) return RV_ERR_UNSUPPORTED;
  return j.plan.splits == 1 ? launch<true, true, Epi::AccF32OfF16>(j.plan.shape, j.g, 1, s)
                            : launch<true, true, Epi::PartialF32>(j.plan.shape, j.g, j.plan.splits, s);
}

template <Epi EPI>
int launch_pair(const WgradJob& a, const WgradJob& b, hipStream_t s) {
  GemmPair pair{{a.g, b.g}, a.g.tiles_m * a.g.tiles_n * a.plan.splits};
  const dim3 grid((unsigned)(pair.first + b.g.tiles_m * b.g.tiles_n * b.plan.splits));
  const dim3 block(kShapes[a.plan.shape].waves * 64);
#define RV_LAUNCH(SHAPE) \
  hipLaunchKernelGGL((wgrad_pair_kernel<SHAPE, EPI>), grid, block, 0, s, pair)
  switch (a.plan.shape) {
    case 0: RV_LAUNCH(0); break;
    case 1: RV_LAUNCH(1); break;
    case 2: RV_LAUNCH(2); break;
    default: RV_LAUNCH(3); break;
  }
#undef RV_LAUNCH
  return rv_host::check_launch();
}

int launch_reduce(const ReduceSeg& a, const ReduceSeg& b, int accumulate, hipStream_t s) {
  const int64_t blocks = a.blocks + b.blocks;
  if (blocks == 0) return RV_OK;
  hipLaunchKernelGGL(wgrad_reduce, dim3((unsigned)blocks), dim3(256), 0, s, a, b, accumulate);
  return rv_host::check_launch();
}

int run_wgrad(const __half* a, int64_t lda, const __half* b, int64_t ldb, int64_t rows,
              int64_t ni, int64_t nj, float* out, int accumulate, float* part, hipStream_t s) {
  const WgradJob j =
      plan_job(plan_wgrad(rows, ni, nj), a, lda, b, ldb, rows, ni, nj, out, accumulate, part);
  const int st = launch_job(j, s);
  if (st != RV_OK) return st;
  return launch_reduce(j.seg, ReduceSeg{nullptr, nullptr, 0, 0, 0}, accumulate, s);
}

int64_t part_bytes(const WgradPlan& p, int64_t ni, int64_t nj) {
  return p.splits > 1 ? p.splits * ni * nj * (int64_t)sizeof(float) : 0;
}

int64_t align256(int64_t bytes) { return (bytes + 255) & ~(int64_t)255; }

// Both partial sums of a pair side by side (b's first), reduced by one launch.
int64_t pair_bytes(const PairPlan& p, int64_t ai, int64_t aj, int64_t bi, int64_t bj) {
  if (p.a.shape < 0 || p.b.shape < 0) return -(int64_t)RV_ERR_UNSUPPORTED;
  const int64_t a = part_bytes(p.a, ai, aj), b = part_bytes(p.b, bi, bj);
  return (a > 0 ? align256(b) : b) + a;
}

// A weight gradient of a pair: out[ni][nj] (+)= sum_m a[m][ni] b[m][nj].
struct WgradOperands {
  const __half* a;
  int64_t lda;
  const __half* b;
  int64_t ldb;
  int64_t ni, nj;
  float* out;
};
int run_pair(const WgradOperands& x, const WgradOperands& y, int64_t rows, int accumulate,
             float* part, hipStream_t s) {
  const PairPlan p = plan_pair(rows, x.ni, x.nj, y.ni, y.nj);
  float* part_x = part + align256(part_bytes(p.b, y.ni, y.nj)) / (int64_t)sizeof(float);
  const WgradJob jy = plan_job(p.b, y.a, y.lda, y.b, y.ldb, rows, y.ni, y.nj, y.out, accumulate, part);
  const WgradJob jx = plan_job(p.a, x.a, x.lda, x.b, x.ldb, rows, x.ni, x.nj, x.out, accumulate, part_x);
  int st;
  if (p.paired) {
    st = p.a.splits > 1 ? launch_pair<Epi::PartialF32>(jx, jy, s)
                        : launch_pair<Epi::AccF32OfF16>(jx, jy, s);
  } else {
    st = launch_job(jy, s);
    if (st == RV_OK) st = launch_job(jx, s);
  }
  if (st != RV_OK) return st;
  return launch_reduce(jy.seg, jx.seg, accumulate, s);
}

bool ok16(const void* p) { return rv_host::aligned16(p); }

// Splits of the tied head's input gradient (rows x d over the vocabulary): as
// act_splits where even 64 x 128 tiles leave the chip half empty; otherwise the
// largest count that keeps the 256 x 256 tiles within one round of the CUs
// (16896 x 256 over 50304, us by splits: 1 682, 2 531, 3 441, 5 522, 7 444, 8 517).
int64_t head_chunk(int64_t rows, int64_t d, int64_t k) {
  int64_t splits = act_splits(rows, d, k);
  if (splits == 1) {
    const int64_t tiles = ((rows + 255) / 256) * ((d + 255) / 256);
    splits = tiles < kCUs ? kCUs / tiles : 1;
    const int64_t most = k / 2048 > 1 ? k / 2048 : 1;  // partials' traffic below the operand's
    if (splits > most) splits = most;
  }
  return ((k + splits - 1) / splits + kSplitStep - 1) / kSplitStep * kSplitStep;
}
int64_t head_dx_bytes(int64_t rows, int64_t d, int64_t k) {
  const int64_t chunk = head_chunk(rows, d, k), splits = (k + chunk - 1) / chunk;
  return splits > 1 ? splits * rows * d * (int64_t)sizeof(float) : 0;
}

// Tile shapes of the head's logits and input gradient.  They follow from the
// sizes, without the timing sweep of run_act: the products are large, a caller's
// row count may change from call to call, and a sweep of both made the first
// call at a row count 60 ms (16896 x 256 over 50257) where a call takes 2.1.  The
// lines (kShapes' indices) are from all shapes timed at widths 128 .. 2048, 64 .. 32768
// rows and vocabularies 1000 .. 50257, with the operands evicted before each
// product (figures marked c: still cached):
//   logits  4 (eight waves) is the fastest or within 5% of it once its tiles fill
//           the CUs four times (16896 x 256 over 50257: 619 us, the others 670-999);
//           1 at d = 128, where two workgroups per CU hide the epilogues of a
//           short k loop, and below that number of tiles if 8 divides its own
//           (tile_of: c 24000 x 256 over 3000 49 against 57, but 1500 x 512 over 32000
//           87 against 70); 2 and 3 below one and a half rounds, as pick_act
//   dx      where act_splits splits, 3 as long as its workgroups fill one round of
//           the CUs (c 1000 x 512 over 50257: 81 us, 5 takes 116) and 5 past it (c 300
//           x 768: 67, 3 takes 99); 0 (2 at odd multiples of 128) over a long
//           reduction, else as pick_act with 3 below one round
int head_logits_shape(int64_t rows, int64_t d, int64_t padded) {
  const auto tiles = [&](int i) {
    return ((rows + kShapes[i].bm - 1) / kShapes[i].bm) *
           ((padded + kShapes[i].bn - 1) / kShapes[i].bn);
  };
  if (tiles(0) >= 3 * kCUs / 2) {
    if (d <= 128) return 1;
    return tiles(1) % 8 == 0 && tiles(0) < (d <= 256 ? 8 : 4) * kCUs ? 1 : 4;
  }
  if (tiles(2) < kCUs) return 3;
  return tiles(2) % 8 == 0 ? 2 : 4;
}
int head_dx_shape(int64_t rows, int64_t d, int64_t k) {
  const int64_t splits = act_splits(rows, d, k);
  if (splits > 1) return (rows + 63) / 64 * (d / 128) * splits > kCUs ? 5 : 3;
  if (k >= 4096) return d % 256 ? 2 : 0;
  return (rows + 127) / 128 * (d / 128) >= kCUs ? pick_act(rows, d, false, 1) : 3;
}

// A tile's rows of an operand with this row stride stay within 32-bit offsets.
bool span32(int64_t ld) { return ld > 0 && 256 * ld * 2 <= (int64_t)INT32_MAX - (int64_t)(1 << 24); }

int head_check(int64_t rows, int64_t d, int64_t vocab, int64_t padded) {
  if (rows <= 0 || d <= 0 || vocab <= 0 || padded < vocab) return RV_ERR_BAD_SIZE;
  if (d % 128 || padded % 64 || !span32(padded) || !span32(d)) return RV_ERR_UNSUPPORTED;
  return RV_OK;
}

// Buffer loads address an operand with 32-bit byte offsets.
bool fits32(int64_t elems) { return elems > 0 && elems * 2 <= (int64_t)INT32_MAX - (int64_t)(1 << 24); }

}  // namespace

extern "C" {

int rv_gemm_num_shapes(void) { return kNumShapes; }

int rv_gemm_force_shape(int shape) {
  if (shape < -1 || shape >= kNumShapes) return RV_ERR_BAD_SIZE;
  g_forced_shape.store(shape);
  return RV_OK;
}

int rv_cast_f32_f16(const float* src, void* dst, int64_t n, void* stream) {
  if (!src || !dst) return RV_ERR_NULL_POINTER;
  if (n < 0) return RV_ERR_BAD_SIZE;
  if (n == 0) return RV_OK;
  if (!ok16(src) || !ok16(dst)) return RV_ERR_UNSUPPORTED;
  int64_t blocks = (n + 256 * 8 - 1) / (256 * 8);
  if (blocks > 8 * kCUs) blocks = 8 * kCUs;
  hipLaunchKernelGGL(cast_f32_f16, dim3((unsigned)blocks), dim3(256), 0, (hipStream_t)stream, src,
                     static_cast<__half*>(dst), n);
  return rv_host::check_launch();
}

int rv_cast_f32_f16_max_tensors(void) { return kCastTensors; }

int rv_cast_f32_f16_multi(int count, const float* const* src, void* const* dst,
                          const int64_t* numel, void* stream) {
  if (count < 0) return RV_ERR_BAD_SIZE;
  if (count == 0) return RV_OK;
  if (!src || !dst || !numel) return RV_ERR_NULL_POINTER;
  if (count > kCastTensors) return RV_ERR_UNSUPPORTED;
  CastTable tab{};
  int64_t passes = 0;
  for (int i = 0; i < count; ++i) {
    if (!src[i] || !dst[i]) return RV_ERR_NULL_POINTER;
    if (numel[i] < 0) return RV_ERR_BAD_SIZE;
    if (!ok16(src[i]) || !ok16(dst[i])) return RV_ERR_UNSUPPORTED;
    passes += (numel[i] + kCastPass - 1) / kCastPass;
  }
  tab.chunk = kCastPass * ((passes + kCastBlocks - 1) / kCastBlocks);
  if (tab.chunk < kCastPass) tab.chunk = kCastPass;
  int64_t chunks = 0;
  for (int i = 0; i < count; ++i) {
    tab.src[i] = src[i];
    tab.dst[i] = static_cast<__half*>(dst[i]);
    tab.n[i] = numel[i];
    tab.chunk_start[i] = (int)chunks;
    chunks += (numel[i] + tab.chunk - 1) / tab.chunk;
  }
  tab.chunk_start[count] = (int)chunks;
  tab.count = count;
  if (chunks == 0) return RV_OK;
  hipLaunchKernelGGL(cast_multi_k, dim3((unsigned)chunks), dim3(256), 0, (hipStream_t)stream, tab);
  return rv_host::check_launch();
}

int rv_mlp_up_swiglu(const void* x, int64_t ldx, const void* w_up, int64_t rows, int64_t d,
                     int64_t f, void* o, void* u, void* stream) {
  if (!x || !w_up || !o) return RV_ERR_NULL_POINTER;
  if (rows <= 0 || d <= 0 || f <= 0 || ldx < d) return RV_ERR_BAD_SIZE;
  if (d % 32 || f % 64 || ldx % 8) return RV_ERR_UNSUPPORTED;
  if (!ok16(x) || !ok16(w_up) || !ok16(o) || (u && !ok16(u))) return RV_ERR_UNSUPPORTED;
  if (!fits32(rows * ldx) || !fits32(2 * f * d)) return RV_ERR_UNSUPPORTED;
  GemmArgs a{};
  a.a = static_cast<const __half*>(x); a.lda = ldx; a.a_bytes = rows * ldx * 2;
  a.b = static_cast<const __half*>(w_up); a.ldb = d; a.b_bytes = 2 * f * d * 2;
  a.m = rows; a.n = 2 * f; a.k = d;
  a.c = o; a.ldc = f; a.u = u; a.ldu = 2 * f; a.f = f;
  return run_act<false, false, Epi::SwiGLU>(a, f, (hipStream_t)stream);
}

int rv_mlp_down(const void* o, const void* w_down, int64_t rows, int64_t d, int64_t f, void* y,
                void* stream) {
  if (!o || !w_down || !y) return RV_ERR_NULL_POINTER;
  if (rows <= 0 || d <= 0 || f <= 0) return RV_ERR_BAD_SIZE;
  if (f % 32 || d % 128) return RV_ERR_UNSUPPORTED;
  if (!ok16(o) || !ok16(w_down) || !ok16(y)) return RV_ERR_UNSUPPORTED;
  if (!fits32(rows * f) || !fits32(d * f)) return RV_ERR_UNSUPPORTED;
  GemmArgs a{};
  a.a = static_cast<const __half*>(o); a.lda = f; a.a_bytes = rows * f * 2;
  a.b = static_cast<const __half*>(w_down); a.ldb = f; a.b_bytes = d * f * 2;
  a.m = rows; a.n = d; a.k = f;
  a.c = y; a.ldc = d;
  return run_act<false, false, Epi::StoreF16>(a, d, (hipStream_t)stream);
}

int rv_mlp_dgate(const void* dy, const void* w_down, const void* u, int64_t rows, int64_t d,
                 int64_t f, void* du, void* stream) {
  if (!dy || !w_down || !u || !du) return RV_ERR_NULL_POINTER;
  if (rows <= 0 || d <= 0 || f <= 0) return RV_ERR_BAD_SIZE;
  if (d % 32 || f % 128) return RV_ERR_UNSUPPORTED;
  if (!ok16(dy) || !ok16(w_down) || !ok16(u) || !ok16(du)) return RV_ERR_UNSUPPORTED;
  if (!fits32(rows * d) || !fits32(d * f)) return RV_ERR_UNSUPPORTED;
  GemmArgs a{};
  a.a = static_cast<const __half*>(dy); a.lda = d; a.a_bytes = rows * d * 2;
  a.b = static_cast<const __half*>(w_down); a.ldb = f;  // B(f, d) = W_down[d][f]: RC
  a.b_bytes = d * f * 2;
  a.m = rows; a.n = f; a.k = d;
  a.c = du; a.ldc = 2 * f; a.u = const_cast<void*>(u); a.ldu = 2 * f; a.f = f;
  return run_act<false, true, Epi::SwiGLUBwd>(a, f, (hipStream_t)stream);
}

int rv_mlp_dx(const void* du, const void* w_up, int64_t rows, int64_t d, int64_t f, float* dx,
              void* stream) {
  if (!du || !w_up || !dx) return RV_ERR_NULL_POINTER;
  if (rows <= 0 || d <= 0 || f <= 0) return RV_ERR_BAD_SIZE;
  if ((2 * f) % 32 || d % 128) return RV_ERR_UNSUPPORTED;
  if (!ok16(du) || !ok16(w_up) || !ok16(dx)) return RV_ERR_UNSUPPORTED;
  if (!fits32(rows * 2 * f) || !fits32(2 * f * d)) return RV_ERR_UNSUPPORTED;
  GemmArgs a{};
  a.a = static_cast<const __half*>(du); a.lda = 2 * f; a.a_bytes = rows * 2 * f * 2;
  a.b = static_cast<const __half*>(w_up); a.ldb = d;  // B(d, j) = W_up[j][d]: RC
  a.b_bytes = 2 * f * d * 2;
  a.m = rows; a.n = d; a.k = 2 * f;
  a.c = dx; a.ldc = d;
  return run_act<false, true, Epi::StoreF32OfF16>(a, d, (hipStream_t)stream);
}

int rv_linear_fwd(const void* x, int64_t ldx, const void* w, int64_t rows, int64_t in,
                  int64_t out, void* y, void* stream) {
  if (!x || !w || !y) return RV_ERR_NULL_POINTER;
  if (rows <= 0 || in <= 0 || out <= 0 || ldx < in) return RV_ERR_BAD_SIZE;
  if (in % 128 || out % 128 || ldx % 8) return RV_ERR_UNSUPPORTED;
  if (!ok16(x) || !ok16(w) || !ok16(y)) return RV_ERR_UNSUPPORTED;
  if (!fits32(rows * ldx) || !fits32(out * in)) return RV_ERR_UNSUPPORTED;
  GemmArgs a{};
  a.a = static_cast<const __half*>(x); a.lda = ldx; a.a_bytes = rows * ldx * 2;
  a.b = static_cast<const __half*>(w); a.ldb = in; a.b_bytes = out * in * 2;
  a.m = rows; a.n = out; a.k = in;
  a.c = y; a.ldc = out;
  return run_act<false, false, Epi::StoreF16>(a, out, (hipStream_t)stream);
}

int rv_linear_dx(const void* dy, const void* w, int64_t rows, int64_t in, int64_t out, void* dx,
                 int dx_dtype, void* stream) {
  if (!dy || !w || !dx) return RV_ERR_NULL_POINTER;
  if (rows <= 0 || in <= 0 || out <= 0) return RV_ERR_BAD_SIZE;
  if (in % 128 || out % 128) return RV_ERR_UNSUPPORTED;
  if (dx_dtype != RV_F16 && dx_dtype != RV_F32) return RV_ERR_UNSUPPORTED;
  if (!ok16(dy) || !ok16(w) || !ok16(dx)) return RV_ERR_UNSUPPORTED;
  if (!fits32(rows * out) || !fits32(out * in)) return RV_ERR_UNSUPPORTED;
  GemmArgs a{};
  a.a = static_cast<const __half*>(dy); a.lda = out; a.a_bytes = rows * out * 2;
  a.b = static_cast<const __half*>(w); a.ldb = in;  // B(i, o) = W[o][i]: RC
  a.b_bytes = out * in * 2;
  a.m = rows; a.n = in; a.k = out;
  a.c = dx; a.ldc = in;
  const hipStream_t s = (hipStream_t)stream;
  return dx_dtype == RV_F16 ? run_act<false, true, Epi::StoreF16>(a, in, s)
                            : run_act<false, true, Epi::StoreF32OfF16>(a, in, s);
}

int64_t rv_linear_splitk_workspace_bytes(int64_t rows, int64_t n, int64_t k) {
  if (rows <= 0 || n <= 0 || k <= 0) return -(int64_t)RV_ERR_BAD_SIZE;
  return act_part_bytes(rows, n, k);
}

int rv_linear_fwd_ws(const void* x, int64_t ldx, const void* w, int64_t rows, int64_t in,
                     int64_t out, void* y, void* workspace, int64_t workspace_bytes,
                     void* stream) {
  const int64_t need = in > 0 && out > 0 && rows > 0 ? act_part_bytes(rows, out, in) : 0;
  if (need == 0) return rv_linear_fwd(x, ldx, w, rows, in, out, y, stream);
  if (!x || !w || !y) return RV_ERR_NULL_POINTER;
  if (ldx < in) return RV_ERR_BAD_SIZE;
  if (in % 128 || out % 128 || ldx % 8) return RV_ERR_UNSUPPORTED;
  if (!ok16(x) || !ok16(w) || !ok16(y)) return RV_ERR_UNSUPPORTED;
  if (!fits32(rows * ldx) || !fits32(out * in)) return RV_ERR_UNSUPPORTED;
  if (!workspace || workspace_bytes < need || !ok16(workspace)) return RV_ERR_WORKSPACE;
  GemmArgs a{};
  a.a = static_cast<const __half*>(x); a.lda = ldx; a.a_bytes = rows * ldx * 2;
  a.b = static_cast<const __half*>(w); a.ldb = in; a.b_bytes = out * in * 2;
  a.m = rows; a.n = out; a.k = in; a.k_chunk = act_chunk(rows, out, in);
  return run_split<false>(a, static_cast<__half*>(y), static_cast<float*>(workspace),
                          (hipStream_t)stream);
}

int rv_linear_dx_ws(const void* dy, const void* w, int64_t rows, int64_t in, int64_t out, void* dx,
                    int dx_dtype, void* workspace, int64_t workspace_bytes, void* stream) {
  const int64_t need = in > 0 && out > 0 && rows > 0 ? act_part_bytes(rows, in, out) : 0;
  if (need == 0) return rv_linear_dx(dy, w, rows, in, out, dx, dx_dtype, stream);
  if (!dy || !w || !dx) return RV_ERR_NULL_POINTER;
  if (in % 128 || out % 128) return RV_ERR_UNSUPPORTED;
  if (dx_dtype != RV_F16 && dx_dtype != RV_F32) return RV_ERR_UNSUPPORTED;
  if (!ok16(dy) || !ok16(w) || !ok16(dx)) return RV_ERR_UNSUPPORTED;
  if (!fits32(rows * out) || !fits32(out * in)) return RV_ERR_UNSUPPORTED;
  if (!workspace || workspace_bytes < need || !ok16(workspace)) return RV_ERR_WORKSPACE;
  GemmArgs a{};
  a.a = static_cast<const __half*>(dy); a.lda = out; a.a_bytes = rows * out * 2;
  a.b = static_cast<const __half*>(w); a.ldb = in;  // B(i, o) = W[o][i]: RC
  a.b_bytes = out * in * 2;
  a.m = rows; a.n = in; a.k = out; a.k_chunk = act_chunk(rows, in, out);
  const hipStream_t s = (hipStream_t)stream;
  float* part = static_cast<float*>(workspace);
  return dx_dtype == RV_F16 ? run_split<true>(a, static_cast<__half*>(dx), part, s)
                            : run_split<true>(a, static_cast<float*>(dx), part, s);
}

int64_t rv_linear_dw_workspace_bytes(int64_t rows, int64_t in, int64_t out) {
  if (rows <= 0 || in <= 0 || out <= 0) return -(int64_t)RV_ERR_BAD_SIZE;
  const WgradPlan p = plan_wgrad(rows, out, in);
  return p.shape < 0 ? -(int64_t)RV_ERR_UNSUPPORTED : part_bytes(p, out, in);
}

int rv_linear_dw(const void* dy, const void* x, int64_t ldx, int64_t rows, int64_t in,
                 int64_t out, float* dw, int accumulate, void* workspace, int64_t workspace_bytes,
                 void* stream) {
  if (!dy || !x || !dw) return RV_ERR_NULL_POINTER;
  if (rows <= 0 || in <= 0 || out <= 0 || ldx < in) return RV_ERR_BAD_SIZE;
  if (in % 128 || out % 128 || ldx % 8) return RV_ERR_UNSUPPORTED;
  if (!ok16(dy) || !ok16(x) || !ok16(dw)) return RV_ERR_UNSUPPORTED;
  if (!fits32(rows * out) || !fits32(rows * ldx)) return RV_ERR_UNSUPPORTED;
  const int64_t need = rv_linear_dw_workspace_bytes(rows, in, out);
  if (need < 0) return (int)-need;
  if (need > 0 && (workspace == nullptr || workspace_bytes < need || !ok16(workspace)))
    return RV_ERR_WORKSPACE;
  // dW[out][in] = sum_m dy[m][o] x[m][i]
  return run_wgrad(static_cast<const __half*>(dy), out, static_cast<const __half*>(x), ldx, rows,
                   out, in, dw, accumulate, static_cast<float*>(workspace), (hipStream_t)stream);
}

int rv_head_logits(const void* x, const void* head, int64_t rows, int64_t d, int64_t vocab,
                   int64_t padded, void* logits, void* stream) {
  if (!x || !head || !logits) return RV_ERR_NULL_POINTER;
  const int bad = head_check(rows, d, vocab, padded);
  if (bad) return bad;
  if (!ok16(x) || !ok16(head) || !ok16(logits)) return RV_ERR_UNSUPPORTED;
  GemmArgs a{};
  a.a = static_cast<const __half*>(x); a.lda = d; a.a_bytes = rows * d * 2;
  a.b = static_cast<const __half*>(head); a.ldb = d; a.b_bytes = padded * d * 2;
  a.m = rows; a.n = padded; a.k = d;
  a.c = logits; a.ldc = padded; a.valid = vocab;
  return run_act<false, false, Epi::StoreF16>(a, padded, (hipStream_t)stream,
                                              head_logits_shape(rows, d, padded), true);
}

int64_t rv_head_workspace_bytes(int64_t rows, int64_t d, int64_t vocab, int64_t padded) {
  const int bad = head_check(rows, d, vocab, padded);
  if (bad) return -(int64_t)bad;
  const WgradPlan p = plan_wgrad(rows, vocab, d, true);
  if (p.shape < 0) return -(int64_t)RV_ERR_UNSUPPORTED;
  const int64_t dx = head_dx_bytes(rows, d, padded), dw = part_bytes(p, vocab, d);
  return dx > dw ? dx : dw;
}

int rv_head_dx(const void* dlogits, const void* head, int64_t rows, int64_t d, int64_t vocab,
               int64_t padded, void* dx, void* workspace, int64_t workspace_bytes, void* stream) {
  if (!dlogits || !head || !dx) return RV_ERR_NULL_POINTER;
  const int bad = head_check(rows, d, vocab, padded);
  if (bad) return bad;
  if (!ok16(dlogits) || !ok16(head) || !ok16(dx)) return RV_ERR_UNSUPPORTED;
  GemmArgs a{};
  a.a = static_cast<const __half*>(dlogits); a.lda = padded; a.a_bytes = rows * padded * 2;
  a.b = static_cast<const __half*>(head); a.ldb = d;  // B(d, v) = head[v][d]: RC
  a.b_bytes = vocab * d * 2;  // the operand ends here: the pad rows read as zero
  a.m = rows; a.n = d; a.k = padded; a.k_chunk = head_chunk(rows, d, padded);
  const hipStream_t s = (hipStream_t)stream;
  const int64_t need = head_dx_bytes(rows, d, padded);
  const int shape = head_dx_shape(rows, d, padded);
  if (need == 0) {
    a.c = dx; a.ldc = d;
    return run_act<false, true, Epi::StoreF16>(a, d, s, shape);
  }
  if (!workspace || workspace_bytes < need || !ok16(workspace)) return RV_ERR_WORKSPACE;
  return run_split<true>(a, static_cast<__half*>(dx), static_cast<float*>(workspace), s, shape);
}

int rv_head_dw(const void* dlogits, const void* x, int64_t rows, int64_t d, int64_t vocab,
               int64_t padded, void* dw, int dw_dtype, int accumulate, void* workspace,
               int64_t workspace_bytes, void* stream) {
  if (!dlogits || !x || !dw) return RV_ERR_NULL_POINTER;
  const int bad = head_check(rows, d, vocab, padded);
  if (bad) return bad;
  if (dw_dtype != RV_F32 && (dw_dtype != RV_F16 || accumulate)) return RV_ERR_UNSUPPORTED;
  if (!ok16(dlogits) || !ok16(x) || !ok16(dw)) return RV_ERR_UNSUPPORTED;
  const WgradPlan p = plan_wgrad(rows, vocab, d, true);
  if (p.shape < 0) return RV_ERR_UNSUPPORTED;
  const int64_t need = part_bytes(p, vocab, d);
  if (need > 0 && (!workspace || workspace_bytes < need || !ok16(workspace)))
    return RV_ERR_WORKSPACE;
  const hipStream_t s = (hipStream_t)stream;
  float* part = static_cast<float*>(workspace);
  // dW[v][d] = sum_m dlogits[m][v] x[m][d]
  WgradJob j = plan_job(p, static_cast<const __half*>(dlogits), padded,
                        static_cast<const __half*>(x), d, rows, vocab, d,
                        static_cast<float*>(dw), accumulate, part);
  if (dw_dtype == RV_F16 && p.splits == 1)
    return launch<true, true, Epi::StoreF16>(p.shape, j.g, 1, s);
  const int st = launch_job(j, s);
  if (st != RV_OK) return st;
  if (dw_dtype == RV_F32) return launch_reduce(j.seg, ReduceSeg{}, accumulate, s);
  const int64_t n = vocab * d;
  hipLaunchKernelGGL(act_reduce<__half>, dim3((unsigned)((n / 4 + 255) / 256)), dim3(256), 0, s,
                     part, static_cast<__half*>(dw), n, (int)p.splits);
  return rv_host::check_launch();
}

int64_t rv_linear_dw_pair_workspace_bytes(int64_t rows, int64_t in_a, int64_t out_a, int64_t in_b,
                                          int64_t out_b) {
  if (rows <= 0 || in_a <= 0 || out_a <= 0 || in_b <= 0 || out_b <= 0)
    return -(int64_t)RV_ERR_BAD_SIZE;
  return pair_bytes(plan_pair(rows, out_a, in_a, out_b, in_b), out_a, in_a, out_b, in_b);
}

int rv_linear_dw_pair(const void* dy_a, const void* x_a, int64_t in_a, int64_t out_a, float* dw_a,
                      const void* dy_b, const void* x_b, int64_t in_b, int64_t out_b, float* dw_b,
                      int64_t rows, int accumulate, void* workspace, int64_t workspace_bytes,
                      void* stream) {
  if (!dy_a || !x_a || !dw_a || !dy_b || !x_b || !dw_b) return RV_ERR_NULL_POINTER;
  if (rows <= 0 || in_a <= 0 || out_a <= 0 || in_b <= 0 || out_b <= 0) return RV_ERR_BAD_SIZE;
  if (in_a % 128 || out_a % 128 || in_b % 128 || out_b % 128) return RV_ERR_UNSUPPORTED;
  if (!ok16(dy_a) || !ok16(x_a) || !ok16(dw_a) || !ok16(dy_b) || !ok16(x_b) || !ok16(dw_b))
    return RV_ERR_UNSUPPORTED;
  if (!fits32(rows * out_a) || !fits32(rows * in_a) || !fits32(rows * out_b) ||
      !fits32(rows * in_b))
    return RV_ERR_UNSUPPORTED;
  const int64_t need = rv_linear_dw_pair_workspace_bytes(rows, in_a, out_a, in_b, out_b);
  if (need < 0) return (int)-need;
  if (need > 0 && (workspace == nullptr || workspace_bytes < need || !ok16(workspace)))
    return RV_ERR_WORKSPACE;
  return run_pair({static_cast<const __half*>(dy_a), out_a, static_cast<const __half*>(x_a), in_a,
                   out_a, in_a, dw_a},
                  {static_cast<const __half*>(dy_b), out_b, static_cast<const __half*>(x_b), in_b,
                   out_b, in_b, dw_b},
                  rows, accumulate, static_cast<float*>(workspace), (hipStream_t)stream);
}

int64_t rv_mlp_wgrad_workspace_bytes(int64_t rows, int64_t d, int64_t f) {
  if (rows <= 0 || d <= 0 || f <= 0) return -(int64_t)RV_ERR_BAD_SIZE;
  return pair_bytes(plan_pair(rows, 2 * f, d, d, f), 2 * f, d, d, f);
}

int rv_mlp_wgrad(const void* dy, const void* o, const void* du, const void* x, int64_t ldx,
                 int64_t rows, int64_t d, int64_t f, float* ddown, float* dup, int accumulate,
                 void* workspace, int64_t workspace_bytes, void* stream) {
  if (!dy || !o || !du || !x || !ddown || !dup) return RV_ERR_NULL_POINTER;
  if (rows <= 0 || d <= 0 || f <= 0 || ldx < d) return RV_ERR_BAD_SIZE;
  if (d % 128 || f % 128 || ldx % 8) return RV_ERR_UNSUPPORTED;
  if (!ok16(dy) || !ok16(o) || !ok16(du) || !ok16(x) || !ok16(ddown) || !ok16(dup))
    return RV_ERR_UNSUPPORTED;
  if (!fits32(rows * 2 * f) || !fits32(rows * ldx) || !fits32(rows * f)) return RV_ERR_UNSUPPORTED;
  const int64_t need = rv_mlp_wgrad_workspace_bytes(rows, d, f);
  if (need < 0) return (int)-need;
  if (need > 0 && (workspace == nullptr || workspace_bytes < need || !ok16(workspace)))
    return RV_ERR_WORKSPACE;
  const hipStream_t s = (hipStream_t)stream;
  // dW_up[2f][d] = sum_m du[m][j] x16[m][d], dW_down[d][f] = sum_m dy[m][d] o[m][f]
  return run_pair({static_cast<const __half*>(du), 2 * f, static_cast<const __half*>(x), ldx, 2 * f,
                   d, dup},
                  {static_cast<const __half*>(dy), d, static_cast<const __half*>(o), f, d, f, ddown},
                  rows, accumulate, static_cast<float*>(workspace), s);
}

}  // extern "C"
