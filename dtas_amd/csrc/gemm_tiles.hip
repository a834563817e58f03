// Dynamic-M GEMM for gfx950: C[M,N] = A[M,K] . W[N,K]^T (+ bias[N]); fp16 in/out, fp32
// accumulation on the MFMA matrix cores: the entry points, the launch descriptions and the
// instantiations of the tile kernel for a row-major fp16 W.  The fused-epilogue GEMMs and the
// two batched attention matmuls run on the same kernel.
//
// Replaces the kernels DTAS's WMMA rule generates (python/dtas/schedule/tir_wmma.py:20-222:
// pad M to a tile multiple, block tile (i*micro_x*16) x (j*micro_y*16), k tile micro_k*16,
// A/B staged in shared.dyn by cooperative_fetch (python/dtas/schedule/tir_base.py:37-97),
// two-stage software pipeline, accumulators through shared memory to a guarded vector
// store; example output experiment/testIR/GEMM/m_n2560_k10240/wmma/16x16x16/i2j4_x7y2_in8.py).
//
// MFMA kernel (M > 64)
//   tile     : BM x BN x 64 per workgroup; WM x WN wavefronts (8 for 256x256 and, on request, 256x128 /
//              128x256; else 4), each owning (BM/WM) x (BN/WN) as 32x32 blocks of
//              v_mfma_f32_32x32x16_f16 (16x16 blocks of v_mfma_f32_16x16x32_f16 on the 8-wavefront
//              tiles), fp32 accumulators in registers.  Both operands are K-contiguous, so a tile row
//              is one 128-byte line = 8 chunks of 16 bytes.
//   global   : 128-bit buffer loads that write LDS directly (no register staging, no
//              ds_write): one wavefront instruction fills one 1 KiB block = 8 tile rows; which
//              (row, chunk) a lane fetches is the inverse of the LDS swizzle.  Rows past M / N
//              and chunks past K fall outside the buffer's range and arrive as zeros.
//   LDS      : two to four stages of (BM + BN) x 128 B (256x256: a ring of five 32 KiB operand
//              units).  Chunk c of row r sits at a swizzled slot so
//              that the MFMA operand reads (a column of 32 rows per half-wavefront, 128 bit
//              per lane) spread over all 64 banks.
//   pipeline : 4-wavefront tiles: fragments of step s+1 are read from LDS while the MFMAs of step
//              s issue (two register sets); the tile barrier sits before the last step of a k
//              tile, the loads of tile k+2 are issued right after it into the stage just
//              vacated, and the first fragments of tile k+1 are read under the last MFMAs of
//              tile k.  The interleaving is pinned with scheduling barriers.
//              8-wavefront tiles: v_mfma_f32_16x16x32_f16 (more flops per watt than 32x32x16,
//              and the card is power-limited on random operands), a whole k32 step of fragments in
//              registers, one barrier per k tile; wavefronts w and w+4 share a SIMD, the older one
//              wins the MFMA pipe, and each requests its share of the next units while the other
//              multiplies (a wavefront that issues a load stalls until the load path takes it).  What the loads run
//              ahead by decides the smaller of these tiles: with W from memory a k tile of 192x128 takes 0.88 us when
//              it is requested one k tile ahead and 0.67 when two or three are in flight.
//   epilogue : accumulators -> fp16 -> wavefront-private LDS region (xor-swizzled 8-byte
//              slots) -> coalesced stores of whole tile rows (8 bytes per lane, 16 on the
//              8-wavefront tiles) with the bias added on the way out.
//   launch   : workgroup ids are remapped so that each XCD (own L2) works on a compact patch of
//              the tile grid.
//   split K  : few output tiles -> several workgroups share a tile and meet in a workspace.
//   epilogues: bias; bias + two residuals (optionally widened to fp32); bias + erf-GELU; the
//              attention scores' scale / clamp / mask -- every step an fp16 value, as the fused
//              PrimFuncs spell them.
//   batches  : the attention matmuls run all heads in one launch (strides in GemmEpilogue).
//   k-major W: for P.V the V tiles are transposed on their way into the LDS (template flag WT).
// The kernels for few rows of A (SKINNY, STREAM, ROWS) are in gemm_stream.hip, the attention kernels in attention.hip,
// the 8-bit-weight entry point in gemm_q8.hip, the split-K workspace in workspace.hip; the tile kernel itself is the
// template in gemm_tile_kernel.h.
#include <utility>

#include "gemm_tile_kernel.h"

namespace dtas {
namespace {

// threads per workgroup of the MFMA kernel for a tile: 8 wavefronts for 256x256, else 4
inline int mfma_threads(int bm, int bn) { return bm == 256 && bn == 256 ? 512 : 256; }
// LDS stages a launch uses unless told otherwise: 2 for 256x256, 3 for 256x128, 4 below that
inline int mfma_max_stages(int bm, int bn) { return bm + bn >= 512 ? 2 : bm + bn >= 384 ? 3 : 4; }

// The tiles that 8 wavefronts serve with stages of their own, and how many of W (0: none): as many k tiles ahead as the LDS
// holds, at most three.  192x256 and 224x256 have three stages of W and two of A (the kernel's kStagesA): W is what
// comes from memory.
int tile8_stages(int bm, int bn) {
  if (bn == 256) return bm == 96 || bm == 128 || bm == 160 || bm == 192 || bm == 224 ? 3 : 0;
  if (bn == 128) return bm == 224 || bm == 256 ? 3 : bm == 96 || bm == 128 || bm == 160 || bm == 192 ? 4 : 0;
  return bn == 64 && bm == 128 ? 4 : 0;
}
// ... and the ones that also come as a ring of five operand units (cfg.unroll == 2), each the larger operand's rows of a k tile
bool tile8_ring(int bm, int bn) { return (bn == 256 && (bm == 128 || bm == 192)) || (bn == 128 && (bm == 192 || bm == 256)); }
int tile8_lds(int bm, int bn) {
  const int ns = tile8_stages(bm, bn);
  return ((ns * (bm + bn) * kRowBytes <= kLdsBytes ? ns : 2) * bm + ns * bn) * kRowBytes;
}

}  // namespace

// The 8-wavefront 256x256 tile when the library chooses: whole rounds of the chip run one workgroup per tile; the
// tiles of a last, partly filled round are shared by 2..4 workgroups each (as many as still fit the chip at once),
// which split K and meet in the workspace -- a round of half or a third the length instead of a whole one.
// Fewer tiles than CUs in all: every tile is split that way.
void tail_split_256(int64_t M, int64_t N, int64_t K, int* nsplit, unsigned* unsplit) {
  const int64_t tiles = ceil_div(M, 256) * ceil_div(N, 256), ktiles = ceil_div(K, kBK);
  const int64_t rem = tiles % kNumCU;
  *nsplit = 1;
  *unsplit = 0;
  if (rem == 0) return;
  int64_t split = kNumCU / rem;
  if (split > 4) split = 4;
  while (split >= 2 && ktiles / split < 8) --split;  // (a part should still be long against its prologue and the combine)
  // a round that fills only part of the chip runs at a higher clock; against that, parts that fill it again gain
  // only when K is long (measured: 128 tiles in two parts each break even at K = 4096 and win 20 % at K = 11008)
  if (split >= 2 && rem * split > 3 * kNumCU / 4 && ktiles < 128) return;
  if (split < 2) return;
  *nsplit = static_cast<int>(split);
  *unsplit = static_cast<unsigned>(tiles - rem);
}

// launch_args: {grid, 1, 1, block, static LDS bytes, tiles along M, tiles along N}
int describe_gemm(int64_t M, int64_t N, int64_t K, const dtas_config& cfg, int64_t la[7]) {
  for (int i = 0; i < 7; ++i) la[i] = 0;
  la[1] = la[2] = 1;
  if (cfg.variant == DTAS_GEMM_MFMA_ACC16) {  // the reference's fp16 accumulator, rounded once per k step of 16
    if (cfg.tile[0] != 64 || cfg.tile[1] != 64 || cfg.tile[2] != 16) return fail("gemm: the fp16-accumulator kernel takes tile 64x64x16, got %dx%dx%d", cfg.tile[0], cfg.tile[1], cfg.tile[2]);
    if (cfg.block != 256) return fail("gemm: the fp16-accumulator kernel uses 256 threads, got %d", cfg.block);
    if (cfg.vec != 8 && cfg.vec != 1) return fail("gemm: vector width must be 8 (128 bit) or 1, got %d", cfg.vec);
    if (cfg.split_k > 1) return fail("gemm: the fp16 accumulator is rounded step by step along K: K cannot be split (split_k = %d)", cfg.split_k);
    const int64_t tm = ceil_div(M, 64), tn = ceil_div(N, 64);
    if (tm * tn > 0x7fffffff) return fail("gemm: too many tiles");
    la[0] = tm * tn;
    la[3] = 256;
    la[5] = tm;
    la[6] = tn;
    return 0;
  }
  if (cfg.vec == 1) {  // element-access fallback
    int64_t grid = ceil_div(M * N, 256);
    la[0] = grid > 65536 ? 65536 : (grid < 1 ? 1 : grid);
    la[3] = 256;
    return 0;
  }
  if (cfg.vec != 8) return fail("gemm: vector width must be 8 (128 bit) or 1, got %d", cfg.vec);
  if (cfg.variant == DTAS_GEMM_MFMA) {
    const int bm = cfg.tile[0], bn = cfg.tile[1];
    // tiles of 96, 160, 192 and 224 rows (8 wavefronts only): between the others in size, for tile counts that fill the chip
    // better (192 columns: the epilogue's lane map wants wavefront tiles of 32, 64 or 128 columns)
    const bool between = (bm == 96 || bm == 160 || bm == 192 || bm == 224) && (bn == 256 || bn == 128);
    const bool known = (bm == 256 && bn == 256) || (bm == 256 && bn == 128) || (bm == 128 && bn == 256) ||
                       (bm == 128 && bn == 128) || (bm == 64 && bn == 128) || (bm == 128 && bn == 64) ||
                       (bm == 64 && bn == 64) || between;
    if (!known || cfg.tile[2] != kBK) return fail("gemm: no MFMA kernel for tile %dx%dx%d", bm, bn, cfg.tile[2]);
    // 256x256 comes as 8 wavefronts (two per SIMD, 128x64 each) or 4 (one per SIMD, 128x128 each); 256x128, 128x256,
    // 128x128 and 128x64 as 4 wavefronts or 8
    const bool four_waves = bm == 256 && bn == 256 && cfg.block == 256;
    const bool eight_waves = tile8_stages(bm, bn) != 0 && cfg.block == 512;
    if (between && !eight_waves) return fail("gemm: the %dx%d MFMA kernel uses 512 threads, got %d", bm, bn, cfg.block);
    if (cfg.block != mfma_threads(bm, bn) && !four_waves && !eight_waves)
      return fail("gemm: the %dx%d MFMA kernel uses %d threads, got %d", bm, bn, mfma_threads(bm, bn), cfg.block);
    if (K * 2 * (bm > bn ? bm : bn) >= (int64_t{1} << 31)) return fail("gemm: K=%lld too large for 32-bit tile offsets", (long long)K);
    const int64_t tm = ceil_div(M, bm), tn = ceil_div(N, bn);
    if (tm * tn > 0x7fffffff) return fail("gemm: too many tiles");
    // cfg.unroll = LDS stages (the depth of the load pipeline); 0 or 1 = as many as fit
    // (8 wavefronts: 0 or 1 = the stages that tile8_stages says; 2 on 192, 256 or 128 x 256 = the ring of five operand units)
    const int max_stages = bm == 192 ? 2 : eight_waves ? tile8_stages(bm, bn) : mfma_max_stages(bm, bn);
    if (cfg.unroll < 0 || cfg.unroll > max_stages)
      return fail("gemm: the %dx%d tile holds at most %d LDS stages, got %d", bm, bn, max_stages, cfg.unroll);
    int nsplit = cfg.split_k < 1 ? 1 : cfg.split_k;
    if (nsplit > 16) return fail("gemm: split_k must be in [1, 16], got %d", cfg.split_k);
    // split_k = 0 on the 8-wavefront 256x256 tile: only the tiles of a last, partly filled round are split
    unsigned unsplit = 0;
    if (cfg.split_k == 0 && bm == 256 && bn == 256 && !four_waves) tail_split_256(M, N, K, &nsplit, &unsplit);
    if (tm * tn * nsplit > 0x7fffffff) return fail("gemm: too many workgroups");
    la[0] = unsplit + (tm * tn - unsplit) * nsplit;
    la[3] = four_waves ? 256 : eight_waves ? 512 : mfma_threads(bm, bn);
    if ((bm == 256 && bn == 256) || (eight_waves && cfg.unroll == 2 && tile8_ring(bm, bn))) la[4] = 5 * (bm > bn ? bm : bn) * kRowBytes;
    else if (eight_waves) la[4] = tile8_lds(bm, bn);
    else la[4] = (cfg.unroll >= 2 ? cfg.unroll : mfma_max_stages(bm, bn)) * (bm + bn) * kRowBytes;
    la[5] = tm;
    la[6] = tn;
    return 0;
  }
  if (cfg.variant == DTAS_GEMM_ROWS) {
    const int mv = cfg.tile[0], r = cfg.tile[1];
    if ((mv != 2 && mv != 4) || (r != 1 && r != 2 && r != 4))
      return fail("gemm: the row kernel takes tile {2,4} rows of A x {1,2,4} rows of W, got %dx%d", mv, r);
    if (M > mv) return fail("gemm: a row tile of %d rows cannot hold M=%lld", mv, (long long)M);
    if (cfg.block != 64 && cfg.block != 128 && cfg.block != 256) return fail("gemm: the row kernel uses 64, 128 or 256 threads, got %d", cfg.block);
    la[0] = ceil_div(N, static_cast<int64_t>(r) * (cfg.block / 64));
    la[3] = cfg.block;
    la[5] = 1;
    la[6] = la[0];
    if (la[0] > 0x7fffffff) return fail("gemm: too many workgroups");
    return 0;
  }
  if (cfg.variant == DTAS_GEMM_SKINNY) {
    const int mt = cfg.tile[0] / 16;
    if (cfg.tile[0] % 16 != 0 || mt < 1 || mt > 5 || cfg.tile[1] != 16)
      return fail("gemm: skinny tile must be {16,32,48,64,80}x16, got %dx%d", cfg.tile[0], cfg.tile[1]);
    if (M > cfg.tile[0]) return fail("gemm: skinny tile of %d rows cannot hold M=%lld", cfg.tile[0], (long long)M);
    if (cfg.block < 64 || cfg.block > 1024 || cfg.block % 64 != 0)
      return fail("gemm: block must be a multiple of 64 in [64, 1024], got %d", cfg.block);
    la[0] = ceil_div(N, 16);
    la[3] = cfg.block;
    la[4] = 16 * mt * 64 * 16;
    la[5] = 1;
    la[6] = la[0];
    return 0;
  }
  if (cfg.variant == DTAS_GEMM_STREAM && cfg.tile[2] == 256) {  // the looping form: the whole of K per workgroup
    const int stages = stream_loop_stages(cfg.tile[0], cfg.tile[1]);
    if (stages == 0)
      return fail("gemm: the looping W-streaming kernel takes tiles 16x64x256 and 16x16x256, got %dx%dx%d", cfg.tile[0], cfg.tile[1],
                  cfg.tile[2]);
    if (M > cfg.tile[0]) return fail("gemm: a streaming tile of %d rows cannot hold M=%lld", cfg.tile[0], (long long)M);
    if (cfg.block != 4 * cfg.tile[1]) return fail("gemm: the %d-column streaming tile uses %d threads, got %d", cfg.tile[1], 4 * cfg.tile[1], cfg.block);
    if (K * 2 * cfg.tile[1] >= (int64_t{1} << 31)) return fail("gemm: K=%lld too large for 32-bit tile offsets", (long long)K);
    const int64_t tn = ceil_div(N, cfg.tile[1]);
    if (tn > 0x7fffffff) return fail("gemm: too many workgroups");
    la[0] = tn;
    la[3] = cfg.block;
    la[4] = stages * (cfg.tile[0] + cfg.tile[1]) * 512;
    la[5] = 1;
    la[6] = tn;
    return 0;
  }
  if (cfg.variant == DTAS_GEMM_STREAM) {
    const int mt = cfg.tile[0] / 16, waves = cfg.tile[1] / 16, seg = cfg.tile[2] / 512;
    if (!stream_shape_ok(cfg.tile[0], cfg.tile[1], cfg.tile[2]))
      return fail("gemm: the W-streaming kernel takes tiles {16,32,64}x{64,128}x{512,1024} that fit the LDS, got %dx%dx%d", cfg.tile[0],
                  cfg.tile[1], cfg.tile[2]);
    if (M > cfg.tile[0]) return fail("gemm: a streaming tile of %d rows cannot hold M=%lld", cfg.tile[0], (long long)M);
    if (cfg.block != 64 * waves) return fail("gemm: the %d-column streaming tile uses %d threads, got %d", cfg.tile[1], 64 * waves, cfg.block);
    if (K * 2 * cfg.tile[1] >= (int64_t{1} << 31)) return fail("gemm: K=%lld too large for 32-bit tile offsets", (long long)K);
    const int64_t tn = ceil_div(N, cfg.tile[1]), slices = ceil_div(K, cfg.tile[2]);
    if (slices < 1 || tn * slices > 0x7fffffff) return fail("gemm: too many workgroups");
    la[0] = tn * slices;
    la[3] = cfg.block;
    la[4] = (16 * mt + 16 * waves) * seg * 1024;
    la[5] = 1;
    la[6] = tn;
    return 0;
  }
  if (cfg.variant == DTAS_GEMM_SHARE) {
    if (!share_kernel_exists(cfg.tile[0], cfg.tile[1], false))
      return fail("gemm: no share kernel for %d rows of A and %d columns per workgroup", cfg.tile[0], cfg.tile[1]);
    if (M > cfg.tile[0]) return fail("gemm: a share kernel of %d rows cannot hold M=%lld", cfg.tile[0], (long long)M);
    if (cfg.block != 256) return fail("gemm: the share kernel uses 256 threads, got %d", cfg.block);
    if (K < 1 || K * 2 * 128 >= (int64_t{1} << 31)) return fail("gemm: K=%lld does not fit 32-bit offsets", (long long)K);
    if (N > 0x7fffffff) return fail("gemm: too many columns");
    la[0] = share_grid(N, cfg.tile[1]);
    la[3] = 256;
    la[5] = 1;
    la[6] = la[0];
    return 0;
  }
  return fail("gemm: unknown variant %d", cfg.variant);
}

// Every instantiation of the tile kernel for a row-major fp16 W, chosen by cfg (validated by describe_gemm): tile,
// 4 or 8 wavefronts, LDS stages, K split.  `batch` problems in one launch (strides in ep): the attention scores.
int launch_tile_f16(const dtas_config& cfg, hipStream_t s, const half_t* a, const half_t* w, const GemmEpilogue& b, void* c,
                    int64_t M, int64_t N, int64_t K, int batch) {
  const int bm = cfg.tile[0], bn = cfg.tile[1];
  const int ns = cfg.unroll >= 2 ? cfg.unroll : 0;
  const int sk = cfg.split_k < 1 ? 1 : cfg.split_k;
  if (bm == 256 && bn == 256)
  {
    if (cfg.block == 256) return launch_mfma<256, 256, 2, 2, 2>(s, a, w, b, c, M, N, K, sk, batch);
    int split = sk;
    unsigned unsplit = 0;
    if (cfg.split_k == 0 && batch == 1) tail_split_256(M, N, K, &split, &unsplit);  // (split_k >= 1: that split for every tile)
    return launch_mfma<256, 256, 2, 4, 2, false, false, true>(s, a, w, b, c, M, N, K, split, batch, unsplit);
  }
  if (cfg.block == 512) {  // 8 wavefronts on the 16x16x32 loop
#define DTAS_TILE8(BM_, BN_, WM_, WN_, NS_) \
    if (bm == BM_ && bn == BN_ && (NS_ > 2 || (ns == 2 && tile8_ring(bm, bn)))) return launch_mfma<BM_, BN_, WM_, WN_, NS_, false, false, true>(s, a, w, b, c, M, N, K, sk, batch)
    DTAS_TILE8(256, 128, 4, 2, 2);  // the rings of two stages: by a config only, but for 192x256 (kTile8Cost)
    DTAS_TILE8(128, 256, 2, 4, 2);
    DTAS_TILE8(192, 256, 2, 4, 2);
    DTAS_TILE8(192, 128, 4, 2, 2);
    DTAS_TILE8(128, 64, 4, 2, 4);
    DTAS_TILE8(96, 128, 2, 4, 4);
    DTAS_TILE8(128, 128, 4, 2, 4);
    DTAS_TILE8(160, 128, 2, 4, 4);
    DTAS_TILE8(192, 128, 4, 2, 4);
    DTAS_TILE8(224, 128, 2, 4, 3);
    DTAS_TILE8(256, 128, 4, 2, 3);
    DTAS_TILE8(96, 256, 2, 4, 3);
    DTAS_TILE8(128, 256, 2, 4, 3);
    DTAS_TILE8(160, 256, 2, 4, 3);
    DTAS_TILE8(192, 256, 2, 4, 3);
    DTAS_TILE8(224, 256, 2, 4, 3);
#undef DTAS_TILE8
  }
  if (bm == 256 && bn == 128) return ns == 2 ? launch_mfma<256, 128, 2, 2, 2>(s, a, w, b, c, M, N, K, sk, batch)
                                             : launch_mfma<256, 128, 2, 2, 3>(s, a, w, b, c, M, N, K, sk, batch);
  if (bm == 128 && bn == 256) return ns == 2 ? launch_mfma<128, 256, 2, 2, 2>(s, a, w, b, c, M, N, K, sk, batch)
                                             : launch_mfma<128, 256, 2, 2, 3>(s, a, w, b, c, M, N, K, sk, batch);
  if (bm == 128 && bn == 128) return ns == 2   ? launch_mfma<128, 128, 2, 2, 2>(s, a, w, b, c, M, N, K, sk, batch)
                                     : ns == 3 ? launch_mfma<128, 128, 2, 2, 3>(s, a, w, b, c, M, N, K, sk, batch)
                                               : launch_mfma<128, 128, 2, 2, 4>(s, a, w, b, c, M, N, K, sk, batch);
  if (bm == 64 && bn == 128) return ns == 2   ? launch_mfma<64, 128, 2, 2, 2>(s, a, w, b, c, M, N, K, sk, batch)
                                    : ns == 3 ? launch_mfma<64, 128, 2, 2, 3>(s, a, w, b, c, M, N, K, sk, batch)
                                              : launch_mfma<64, 128, 2, 2, 4>(s, a, w, b, c, M, N, K, sk, batch);
  if (bm == 128 && bn == 64) return ns == 2   ? launch_mfma<128, 64, 2, 2, 2>(s, a, w, b, c, M, N, K, sk, batch)
                                    : ns == 3 ? launch_mfma<128, 64, 2, 2, 3>(s, a, w, b, c, M, N, K, sk, batch)
                                              : launch_mfma<128, 64, 2, 2, 4>(s, a, w, b, c, M, N, K, sk, batch);
  if (bm == 64 && bn == 64) return ns == 2    ? launch_mfma<64, 64, 2, 2, 2>(s, a, w, b, c, M, N, K, sk, batch)
                                   : ns == 3  ? launch_mfma<64, 64, 2, 2, 3>(s, a, w, b, c, M, N, K, sk, batch)
                                              : launch_mfma<64, 64, 2, 2, 4>(s, a, w, b, c, M, N, K, sk, batch);
  return fail("gemm: no MFMA kernel for tile %dx%d", bm, bn);
}

// Beyond 128 rows: the tile, and the parts of K.  A candidate's time is
//   rounds of the chip x (a + b x k tiles of a part), a partly filled round at b x (r + (1 - r) x its share of the chip),
//   + w x workgroups per CU + h0 + h1 x parts + h2 x (share of the chip)^4 where K is split (the hand-over of the partial tiles),
// with b growing with 1 / (tile rows of the grid) (fewer workgroups share what W costs to bring in), falling with the rows past M
// in the tiles (nothing is loaded for them), and x pitch or pow2 by K's row_pitch.  (64x64, of which a CU holds
// several, at r + (1 - r) x its share up to one per CU and at 0.75 per workgroup of the fullest CU beyond.)
// Fitted to 537 sizes (M = 129 .. 8192 against 27 W of 512 x 2048 .. 50280 x 2560) x up to 14 configurations each, A, W and C all
// taken from memory: that is what a launch between other kernels costs.  With one A kept for all launches the staged tiles look
// up to 13 % better than in a pass (2048 x 4096 x 11008: 256x128 whole 150 us so and 169 with A from memory, 256x256 with the tiles
// in two parts 155 either way, and a pass of three products 14 us shorter with the latter; 150 x 2560 x 10240: 128x64 in three
// parts 26 / 34, 64x64 in two 29 / 30, a layer 3.6 us shorter).
// In the bucket table (`in_table`): the tiles marked so, K in up to 4 parts of 8 k tiles or more (1.036 of the best configuration's time on
// average).  For a call without a config also the tiles between them, where no more than a fifth of their rows lie past M or
// they make at most three rows of tiles, and up to 6 parts of 6 k tiles: 1.007 (1.026 with the fit to one A).  Up to two rows of tiles
// those take K in parts of fewer than 24 k tiles only if they are ahead by 0.46 us a part: what is nearer is left to the table's
// tile (0.001 of the time; longer parts as they come: 135 .. 192 x 2560 x 10240 on 96x128 in six 28.6 us, on 64x64 in two 30.4, in four 30.5 .. 32.6).
struct Tile8Cost {
  int bm, bn, block, stages;
  bool in_table;
  double a, b, w, r, h0, h1, h2, pitch, pow2, few, pad;
};
constexpr Tile8Cost kTile8Cost[] = {
    {64, 64, 256, 4, true, 3.57, 0.29, 0.478, 0.717, 0.524, 0.734, 0.129, 1.088, 1.009, 0.574, 0.47},
    {128, 64, 512, 0, true, 2.631, 0.403, 1.476, 0.909, 2.034, 0.637, 0.653, 1.108, 0.961, 0.203, 0.153},
    {96, 128, 512, 0, false, 3.519, 0.476, 0.746, 0.809, 1.266, 0.975, 1.735, 1.107, 0.98, 0.614, 0.623},
    {128, 128, 512, 0, true, 3.291, 0.544, 1.551, 0.823, 0.877, 1.463, 2.133, 1.071, 0.951, 0.485, 0.404},
    {160, 128, 512, 0, false, 3.721, 0.611, 0.409, 0.902, 1.024, 1.727, 4.122, 1.08, 0.968, 0.377, 0.217},
    {192, 128, 512, 0, true, 4.008, 0.677, 0.586, 0.909, 1.074, 2.066, 5.196, 1.085, 0.974, 0.301, 0.201},
    {224, 128, 512, 0, false, 4.428, 0.766, 0, 0.849, 2.076, 2.391, 3.818, 1.088, 0.968, 0.232, 0.231},
    {256, 128, 512, 0, true, 5.651, 0.874, 0, 0.737, 1.586, 2.705, 3.646, 1.051, 0.932, 0.223, 0.316},
    {96, 256, 512, 0, false, 3.125, 0.722, 1.919, 0.88, 1.049, 1.981, 2.592, 1.096, 0.96, 0.948, 0.41},
    {128, 256, 512, 0, false, 5.289, 0.846, 0, 0.692, 0.862, 2.651, 2.37, 1.081, 0.954, 0.889, 0.566},
    {160, 256, 512, 0, false, 5.914, 0.99, 0.447, 0.675, -0.599, 3.146, 6.082, 1.054, 0.979, 0.584, 0.593},
    {192, 256, 512, 0, true, 7.283, 1.152, 0.273, 0.69, 0.249, 2.667, 7.583, 1.039, 0.966, 0.497, 0.537},
    {224, 256, 512, 0, false, 7.123, 1.294, 0.808, 0.652, 1.88, 2.796, 4.098, 1.025, 0.983, 0.407, 0.415},
    {256, 256, 512, 2, true, 8.473, 1.449, 0.41, 0.613, -1.316, 4.31, 8.162, 1.011, 0.984, 0.311, 0.395},
    {192, 256, 512, 2, true, 6.715, 1.142, 0.592, 0.663, 2.39, 3.56, 3.96, 1.063, 0.96, 0.508, 0.209},
};
// 192x256 comes twice: W in three stages and A in two, and (stages 2) as a ring, which leads where rows lie a power of two apart
// (2890 x 4096 x 4096: 0.956 of the time, 3001 x 4096 x 8192 0.961, K whole) and is level or behind elsewhere (1024 x 7680 x 2560 1.10, 2561 x 2560 x
// 10240 1.07), so that only those rows look at it.

// One row of the table against M x N x K (instantiated per row: the divisions by its extents are multiplications).
struct Tile8Query {
  int64_t M, N, K, ktiles;
  int64_t steps[7];  // k tiles of the longest of p parts
  bool in_table;
  RowPitch pitch;
  int tail_parts;    // 256x256: parts of the last round's tiles
  int64_t tail_whole;
};
template <int I>
inline void tile8_consider(const Tile8Query& q, double* best, dtas_config* out) {
  constexpr Tile8Cost c = kTile8Cost[I];
  constexpr int64_t kBig = c.bm > c.bn ? c.bm : c.bn, slots = c.bm * c.bn <= 64 * 64 ? 2 * kNumCU : kNumCU;
  constexpr bool whole_rounds = c.bm == 256 && c.bn == 256;  // its split is of the last round's tiles (tail_split_256)
  constexpr bool ring_192 = c.bm == 192 && c.stages == 2;
  if (ring_192 && q.pitch != kPitchPow2) return;
  const int64_t tm = ceil_div(q.M, c.bm), tn = ceil_div(q.N, c.bn), tiles = tm * tn;
  if (!c.in_table && (q.in_table || (tm > 3 && q.M * 5 < tm * c.bm * 4))) return;
  if (q.K * 2 * kBig >= (int64_t{1} << 31)) return;  // (32-bit tile offsets, describe_gemm)
  if (tiles > 0x7fffffff / 8) return;
  const double b = c.b * (q.pitch == kPitchSlow ? c.pitch : q.pitch == kPitchPow2 ? c.pow2 : 1.0) *
                   (1.0 + c.few / static_cast<double>(tm) - c.pad * (1.0 - static_cast<double>(q.M) / static_cast<double>(tm * c.bm)));
  const int most = whole_rounds || ring_192 ? 1 : q.in_table ? 4 : 6;
  for (int parts = 1; parts <= most; ++parts) {
    int last_parts = parts;
    if (whole_rounds) {
      last_parts = q.tail_parts;
      // (inside dtas_gemm_f16_static: only as many partial tiles as there is room for)
      if (!q.in_table && t_fixed_scratch && (tiles - q.tail_whole) * last_parts * c.bm * c.bn * 4 > DTAS_STATIC_SCRATCH_PARTIAL_BYTES) last_parts = 1;
    } else if (parts > 1 && (tiles * parts > slots || q.ktiles < parts * (q.in_table ? 8 : 6) ||
                             tiles * parts * c.bm * c.bn * 4 > DTAS_STATIC_SCRATCH_PARTIAL_BYTES)) {
      break;  // (no more partial tiles than dtas_gemm_f16_static has room for)
    }
    const bool tail = whole_rounds && last_parts > 1;
    const int64_t wgs = whole_rounds ? tiles : tiles * parts, full = wgs / slots, rem = wgs % slots;
    const double steps = static_cast<double>(whole_rounds ? q.ktiles : q.steps[parts]);
    const double share = static_cast<double>(wgs) / kNumCU;
    double us = static_cast<double>(full) * (c.a + b * steps) + c.w * share;
    const double fill = static_cast<double>(whole_rounds ? rem * last_parts : rem) / static_cast<double>(slots);
    if (slots > kNumCU)  // (64x64: two or more workgroups share a CU)
      us = c.a + b * steps * (wgs <= kNumCU ? c.r + (1.0 - c.r) * share : 0.75 * static_cast<double>(ceil_div(wgs, kNumCU))) + c.w * share;
    else if (rem > 0) us += c.a + b * (whole_rounds ? static_cast<double>(q.steps[last_parts]) : steps) * (c.r + (1.0 - c.r) * fill);
    if (last_parts > 1) {
      const double crowd = whole_rounds ? fill : share;
      us += c.h0 + c.h1 * last_parts + c.h2 * crowd * crowd * crowd * crowd;
    }
    if (!c.in_table && tm <= 2 && parts > 1 && q.ktiles < 24 * parts) us += 0.46 * parts;
    if (us < *best) {
      *best = us;
      *out = dtas_config{DTAS_GEMM_MFMA, c.block, 8, c.stages, {c.bm, c.bn, kBK}, tail ? 0 : parts, 0};
    }
  }
}
template <int... I>
inline void tile8_consider_all(const Tile8Query& q, double* best, dtas_config* out, std::integer_sequence<int, I...>) {
  (tile8_consider<I>(q, best, out), ...);
}
bool tile8_policy(int64_t M, int64_t N, int64_t K, bool in_table, dtas_config* out, double* us_out) {
  Tile8Query q{M, N, K, ceil_div(K, kBK), {}, in_table, row_pitch(K), 1, 0};
  q.steps[1] = q.ktiles;
  q.steps[2] = ceil_div(q.ktiles, 2);
  q.steps[3] = ceil_div(q.ktiles, 3);
  q.steps[4] = ceil_div(q.ktiles, 4);
  q.steps[5] = ceil_div(q.ktiles, 5);
  q.steps[6] = ceil_div(q.ktiles, 6);
  unsigned whole = 0;
  tail_split_256(M, N, K, &q.tail_parts, &whole);
  q.tail_whole = whole;
  double best = 1e300;
  tile8_consider_all(q, &best, out, std::make_integer_sequence<int, sizeof(kTile8Cost) / sizeof(kTile8Cost[0])>{});
  if (us_out) *us_out = best;
  return best < 1e300;  // (else nothing was written to *out)
}

// What a call without a config runs: the bucket's row, or ahead of it a kernel chosen by M itself (what A costs it goes
// with M, and the row is sized for the end of its bucket).  vec_ok: 16-byte loads of A and W are possible.
dtas_config builtin_gemm(int64_t M, int64_t N, int64_t K, bool vec_ok) {
  // two rows of A (the first bucket's table row is sized for 16): W streamed in whole rows, as the GEMV does
  if (M == 2 && vec_ok) return dtas_config{DTAS_GEMM_ROWS, 64, 8, 1, {2, N <= 2560 ? 1 : 2, 8}, 1, 0};
  // three or four rows: the row kernel, a row of W per wavefront, against a W too small or too short for the share kernel
  // (3 x 64 x 256, 200 x 520, 255 x 4096, 4096 x 128: 3.1, 3.5, 5.7, 4.0 us against 4.1, 4.6, 7.3, 4.6; with long rows the other
  // way round: 128 x 10240 9.5 / 8.0), and against long rows of W that are few (1024 x 8192 9.2 / 9.8, 2048 x 11008 0.90 of the
  // share kernel's time; level at 2560 rows: 10240 0.99; behind for shorter ones, 1024 x 1024 3.9 / 3.8, 2560 x 2560 1.03)
  const bool few_rows = N < 256 ? K < 8192 : K < 256 ? N <= 4096 : N < 2560 && K >= 6144;
  if ((M == 3 || M == 4) && vec_ok && few_rows) return dtas_config{DTAS_GEMM_ROWS, 64, 8, 1, {4, 1, 8}, 1, 0};
  // up to 128 rows of A: the share kernel where it leads
  int rows = 0, cols = 0;
  if (vec_ok && share_leads(M, N, K, &rows, &cols)) return dtas_config{DTAS_GEMM_SHARE, 256, 8, 1, {rows, cols, 0}, 1, 0};
  dtas_config cfg;
  if (M > 128 && vec_ok && tile8_policy(M, N, K, false, &cfg)) return cfg;
  return builtin_config(DTAS_OP_GEMM_F16, M, N, K).cfg;
}

}  // namespace dtas

extern "C" int dtas_builtin_gemm(int weights_8bit, int64_t M, int64_t N, int64_t K, dtas_launch_info* out) {
  using namespace dtas;
  clear_error();
  if (!out) return fail("dtas_builtin_gemm: out is NULL");
  if (M < 2 || N < 1 || K < 1) return fail("dtas_builtin_gemm: M >= 2, N >= 1 and K >= 1 wanted (one row is the GEMV), got %lld, %lld, %lld", (long long)M, (long long)N, (long long)K);
  memset(out, 0, sizeof(*out));
  out->index = -1;
  out->table_row = -1;
  const char* what = "gemm";
  if (weights_8bit) {
    if (K % 32 != 0) return fail("dtas_builtin_gemm: K must be a multiple of the scale group, 32 (K=%lld)", (long long)K);
    what = "gemm_q8";
    if (builtin_gemm_q8(M, N, K, K % 256 == 0, N <= ((int64_t{1} << 32) - 1) / K, &out->config)) {
      snprintf(out->name, sizeof(out->name), "%s", what);
      return 0;  // (launch_args stay zero: the 8-bit kernels' grids are their launchers')
    }
    what = "decode_q8 + gemm";
  }
  snprintf(out->name, sizeof(out->name), "%s", what);
  out->config = builtin_gemm(M, N, K, K % 8 == 0);
  if (K % 8 != 0) out->config.vec = 1;
  return describe_gemm(M, N, K, out->config, out->launch_args);
}

extern "C" int dtas_gemm_f16(const void* A, const void* W, const void* bias, void* C, int64_t M, int64_t N, int64_t K,
                             const dtas_config* user, void* stream) {
  return dtas_gemm_f16_fused(A, W, bias, nullptr, nullptr, C, M, N, K, DTAS_EPI_BIAS, user, stream);
}

extern "C" int dtas_gemm_f16_static(const void* A, const void* W, const void* bias, void* C, int64_t M, int64_t N, int64_t K,
                                    const dtas_config* user, void* stream) {
  using namespace dtas;
  clear_error();
  void* base = nullptr;
  if (resolve_static_scratch(&base) != 0) return -1;  // (a table lookup after the first call on a device, or after dtas_init)
  const FixedScratch fixed = {reinterpret_cast<float*>(static_cast<unsigned char*>(base) + DTAS_STATIC_SCRATCH_COUNTERS * 4),
                              DTAS_STATIC_SCRATCH_PARTIAL_BYTES, static_cast<unsigned*>(base), DTAS_STATIC_SCRATCH_COUNTERS};
  struct Scope {
    explicit Scope(const FixedScratch* f) { t_fixed_scratch = f; }
    ~Scope() { t_fixed_scratch = nullptr; }
  } scope(&fixed);
  return dtas_gemm_f16_fused(A, W, bias, nullptr, nullptr, C, M, N, K, DTAS_EPI_BIAS, user, stream);
}

extern "C" int dtas_gemm_f16_fused(const void* A, const void* W, const void* bias, const void* res1, const void* res2,
                                   void* C, int64_t M, int64_t N, int64_t K, int32_t epilogue, const dtas_config* user,
                                   void* stream) {
  using namespace dtas;
  clear_error();
  if (epilogue < DTAS_EPI_BIAS || epilogue > DTAS_EPI_BIAS_GELU) return fail("gemm: unknown epilogue %d", epilogue);
  const bool add2 = epilogue == DTAS_EPI_BIAS_ADD2 || epilogue == DTAS_EPI_BIAS_ADD2_CAST_F32;
  const int out_bytes = epilogue == DTAS_EPI_BIAS_ADD2_CAST_F32 ? 4 : 2;
  if (M < 0 || N < 0 || K < 0) return fail("gemm: negative extent M=%lld N=%lld K=%lld", (long long)M, (long long)N, (long long)K);
  if (M == 0 || N == 0) return 0;
  if ((K != 0 && (M > INT64_MAX / 4 / K || N > INT64_MAX / 4 / K)) || M > INT64_MAX / 4 / N) return fail("gemm: extents overflow");
  if (!C || (K > 0 && (!A || !W))) return fail("gemm: NULL buffer");
  if (add2 && (!res1 || !res2)) return fail("gemm: the add-add epilogue needs both residual buffers");
  if (!add2 && (res1 || res2)) return fail("gemm: residual buffers given for an epilogue that takes none");
  if (overlaps(C, M * N * out_bytes, A, M * K * 2) || overlaps(C, M * N * out_bytes, W, N * K * 2) ||
      (add2 && (overlaps(C, M * N * out_bytes, res1, M * N * 2) || overlaps(C, M * N * out_bytes, res2, M * N * 2))))
    return fail("gemm: output overlaps an input");
  // one row of A is the decode GEMV: same PrimFunc shape, dedicated kernel (every epilogue)
  if (!user && M == 1) return dtas_gemv_f16_fused(A, W, bias, res1, res2, C, N, K, epilogue, nullptr, stream);
  const GemmEpilogue ep = {static_cast<const half_t*>(bias), static_cast<const half_t*>(res1),
                           static_cast<const half_t*>(res2), epilogue, out_bytes == 4 ? 1 : 0, 0.f, 0, 0, 0, 0};
  const bool vec_ok = K % 8 == 0 && aligned(A, 16) && aligned(W, 16);
  dtas_config cfg = user ? *user : builtin_gemm(M, N, K, vec_ok);
  if (cfg.vec == 8 && !vec_ok) cfg.vec = 1;  // K % 8 != 0 or odd pointers: element accesses
  int64_t la[7];
  if (describe_gemm(M, N, K, cfg, la) != 0) return -1;
  hipStream_t s = static_cast<hipStream_t>(stream);
  const half_t* a = static_cast<const half_t*>(A);
  const half_t* w = static_cast<const half_t*>(W);
  const GemmEpilogue& b = ep;
  void* c = C;
  if (cfg.variant == DTAS_GEMM_MFMA_ACC16) return launch_gemm_acc16(cfg, s, a, w, b, c, M, N, K);
  if (cfg.vec == 1) return launch_gemm_scalar("gemm", static_cast<unsigned>(la[0]), 1, s, a, w, b, c, M, N, K, false);
  if (cfg.variant == DTAS_GEMM_ROWS) return launch_gemm_rows(cfg, la, s, a, w, b, c, M, N, K);
  if (cfg.variant == DTAS_GEMM_SKINNY) return launch_gemm_skinny(cfg, la, s, a, w, b, c, M, N, K);
  if (cfg.variant == DTAS_GEMM_SHARE) return launch_gemm_share(cfg.tile[0], cfg.tile[1], s, a, w, b, c, M, N, K);
  if (cfg.variant == DTAS_GEMM_STREAM) return launch_gemm_stream(cfg, s, a, w, b, c, M, N, K);
  return launch_tile_f16(cfg, s, a, w, b, c, M, N, K, 1);
}
