// The dynamic-n GEMMs on 8-bit weights (q8f16_1: four bytes to a word, an fp16 scale per 32 elements of a row):
// fused_fused_decode2_fused_NT_matmul6_add4 and its fused-epilogue relatives
// (experiment/ModelIR/dolly-v2-3b-q8f16_1/before_dl.py:371-502), C = epilogue(A . dequant(Wq)^T).
// Few rows: the share kernel (gemm_share.hip) or the W-streaming kernel (gemm_stream.hip) on the bytes.  Otherwise the tile
// kernel with the dequantiser in its W path (template flag WQ, instantiated here), or the dequantiser into a
// library-owned fp16 buffer followed by the fp16 GEMM.
#include <utility>

#include "gemm_tile_kernel.h"

namespace dtas {
namespace {
// The tiles that dequantise in their W path, by the estimate of tile8_policy (the 4-wavefront tiles, of which a CU holds several:
// at r + (1 - r) x share of the chip up to one workgroup per CU, and at 0.75 (64x64) or 0.85 (128x64) per workgroup of the fullest
// CU beyond).  Fitted to 288 sizes (65 .. 2048 rows against 18 W of 1024 x 4096 .. 14336 x 4096) x up to 14 configurations, A, W and C all from
// memory as there: 1.007 of the best one's time (held-out sizes 1.0075); 0.84 of the time of the 4-wavefront tiles that ran before over 121
// sizes outside the fit (with one A for all launches: 203 x 10240 x 2560 34.7 -> 28.0 us, 512 x 7680 x 2560 36.4 -> 30.3, 700 x 2560 x 10240 71.5 -> 55.4).
struct TileQ8Cost {
  int bm, bn, block, stages;
  double a, b, w, r, h0, h1, h2, pitch, pow2, few, pad;
};
constexpr TileQ8Cost kTileQ8Cost[] = {
    {64, 64, 256, 3, 4.639, 0.359, 0, 1.012, 0.992, 0.517, 0.058, 1.025, 0.971, 0.424, 0.194},
    {128, 64, 256, 3, 5.232, 0.483, 0, 0.816, 1.531, 0.623, 0.232, 1.013, 0.959, 0.164, 0.177},
    {96, 128, 512, 0, 2.475, 0.614, 2.37, 0.981, 1.723, 0.886, 0.959, 1.007, 0.964, 0.183, 0.151},
    {128, 128, 512, 0, 2.789, 0.648, 2.086, 0.975, 2.187, 1.157, 1.228, 1.024, 0.966, 0.148, 0.243},
    {160, 128, 512, 0, 4.28, 0.728, 1.15, 0.931, 1.772, 1.527, 1.193, 1.038, 0.987, 0.088, 0.223},
    {192, 128, 512, 0, 5.329, 0.795, 0.105, 0.875, 1.575, 1.905, 2.063, 1.035, 0.983, 0.081, 0.288},
    {256, 128, 512, 0, 6.255, 1.019, 0.056, 0.76, 1.622, 2.452, 1.412, 1.042, 0.972, 0.025, 0.256},
};
// One row of the table against M x N x K (instantiated per row: the divisions by its extents are multiplications).
struct TileQ8Query {
  int64_t M, N, K, ktiles;
  int64_t steps[9];  // k tiles of the longest of p parts
  RowPitch pitch;
};
template <int I>
inline void tile_q8_consider(const TileQ8Query& q, double* best, dtas_config* out) {
  constexpr TileQ8Cost c = kTileQ8Cost[I];
  constexpr int64_t kBig = c.bm > c.bn ? c.bm : c.bn, limit = c.block == 256 ? 2 * kNumCU : kNumCU;
  if (q.K * 2 * kBig >= (int64_t{1} << 31)) return;  // (32-bit tile offsets, describe_gemm)
  const int64_t tm = ceil_div(q.M, c.bm), tn = ceil_div(q.N, c.bn), tiles = tm * tn;
  if (tiles > 0x7fffffff / 8) return;
  const double b = c.b * (q.pitch == kPitchSlow ? c.pitch : q.pitch == kPitchPow2 ? c.pow2 : 1.0) *
                   (1.0 + c.few / static_cast<double>(tm) - c.pad * (1.0 - static_cast<double>(q.M) / static_cast<double>(tm * c.bm)));
  for (int parts = 1; parts <= 8; ++parts) {
    // (K <= 768: a launch is mostly its start, and a hand-over costs what the shorter loop saves: 128 x 2048 x 768 8.6 us whole, 11.3 in three)
    if (parts > 1 && (q.ktiles <= 12 || tiles * parts > limit || q.ktiles < parts * (c.block == 256 ? 4 : 6) ||
                      tiles * parts * c.bm * c.bn * 4 > DTAS_STATIC_SCRATCH_PARTIAL_BYTES)) break;
    const int64_t wgs = tiles * parts, full = wgs / kNumCU, rem = wgs % kNumCU;
    const double steps = static_cast<double>(q.steps[parts]), share = static_cast<double>(wgs) / kNumCU;
    double us = c.w * share;
    if (c.block == 256)
      us += c.a + b * steps * (wgs <= kNumCU ? c.r + (1.0 - c.r) * share : (c.bm == 64 ? 0.75 : 0.85) * static_cast<double>(ceil_div(wgs, kNumCU)));
    else
      us += static_cast<double>(full) * (c.a + b * steps) + (rem > 0 ? c.a + b * steps * (c.r + (1.0 - c.r) * static_cast<double>(rem) / kNumCU) : 0.0);
    if (parts > 1) us += c.h0 + c.h1 * parts + c.h2 * share * share * share * share;
    if (us < *best) {
      *best = us;
      *out = dtas_config{DTAS_GEMM_MFMA, c.block, 8, c.stages, {c.bm, c.bn, kBK}, parts, 0};
    }
  }
}
template <int... I>
inline void tile_q8_consider_all(const TileQ8Query& q, double* best, dtas_config* out, std::integer_sequence<int, I...>) {
  (tile_q8_consider<I>(q, best, out), ...);
}
double tile_q8_policy(int64_t M, int64_t N, int64_t K, dtas_config* out) {
  const int64_t kt = ceil_div(K, kBK);
  const TileQ8Query q{M, N, K, kt, {0, kt, ceil_div(kt, 2), ceil_div(kt, 3), ceil_div(kt, 4), ceil_div(kt, 5), ceil_div(kt, 6), ceil_div(kt, 7), ceil_div(kt, 8)}, row_pitch(K)};
  double best = 1e300;
  tile_q8_consider_all(q, &best, out, std::make_integer_sequence<int, sizeof(kTileQ8Cost) / sizeof(kTileQ8Cost[0])>{});
  return best;
}
}  // namespace

// What a call without a config runs; false: the dequantiser into a library-owned buffer, then the fp16 GEMM.  stream_ok: the
// kernels that stream the bytes of W can take the call (16-byte aligned operands, K % 256 == 0, K < 2^24); vec_ok: the tiles can.
bool builtin_gemm_q8(int64_t M, int64_t N, int64_t K, bool stream_ok, bool vec_ok, dtas_config* out) {
  dtas_config& cfg = *out;
  // Few rows of A: the launch is one read of the bytes of W.
  // up to 96 rows: every CU an equal share of W's rows, nothing handed over (share_leads_q8)
  int rows = 0, cols = 0;
  if (stream_ok && N <= 0x7fffffff && share_leads_q8(M, N, K, &rows, &cols)) {
    cfg = dtas_config{DTAS_GEMM_SHARE, 256, 8, 1, {rows, cols, 0}, 1, 0};
    return true;
  }
  // the W-streaming kernel, which widens the bytes on their way from the LDS into the MFMA
  if (stream_ok && M <= 32) {
    // what the share kernel leaves to it, against the best of the tiles, W from memory: 8 rows against 300 x 14336 8.5 us / 20.3, 16
    // against 1024 x 8192 8.9 / 15.9, 32 against 1024 x 8192 12.3 / 16.1, 768 x 4096 8.6 / 12.1.  512-element slices (three workgroups
    // per CU) unless K is long: from 16 slices on the hand-over of the partial sums costs more than the second
    // workgroup hides (1024-element slices / 512: 16 rows against 512 x 4096 7.5 / 6.8, 2048 x 8192 10.6 / 12.6)
    cfg = dtas_config{DTAS_GEMM_STREAM, 256, 8, 1, {M > 16 ? 32 : 16, 64, M <= 16 && K >= 8192 ? 1024 : 512}, 1, 0};
    return true;
  }
  // up to 64 rows only while its workgroups (64 columns x 512 of K each) run in one round: 48 rows against 512 x 4096 / 1024 x
  // 6144 / 1024 x 8192 10.7 / 13.9 / 15.9 us where the best of the tiles takes 11.7 / 14.5 / 16.2, but 19.5 against 16.3 at 1088 x 8192
  if (stream_ok && M <= 64 && ceil_div(N, 64) * ceil_div(K, 512) <= kNumCU) {
    cfg = dtas_config{DTAS_GEMM_STREAM, 256, 8, 1, {64, 64, 512}, 1, 0};
    return true;
  }
  // Two routes.  (1) Dequantising in the W path of the tile kernel: no intermediate, W read once per row of tiles as bytes.
  // (2) The dequantiser into a library-owned fp16 buffer, then the fp16 GEMM with every tile it has: 3.4 us and 0.49 per million
  // weights more, worth it once the GEMM itself is long (7680 x 2560: from ~1000 rows, 10240 x 2560 ~770, 2560 x 10240 ~1540).  Its time over
  // the fit's sizes: these + the fp16 GEMM's estimate, to 5 %; the lesser of the two estimates is the lesser time to 0.1 %.
  cfg = dtas_config{DTAS_GEMM_MFMA, 256, 8, 3, {128, 128, kBK}, 1, 0};
  const int64_t t128 = ceil_div(M, 128) * ceil_div(N, 128);
  if (!vec_ok) return M <= 512 && t128 <= kNumCU;  // (the element kernel, or the two passes, whose second can run on whole vectors)
  const double us = tile_q8_policy(M, N, K, &cfg);
  dtas_config wide;
  double us16 = 0.;
  return !(M > 128 && tile8_policy(M, N, K, false, &wide, &us16) && 3.445 + 0.486e-6 * static_cast<double>(N) * static_cast<double>(K) + 1.002 * us16 < us);
}
}  // namespace dtas

extern "C" int dtas_gemm_q8_f16_fused(const void* A, const void* Wq, const void* scale, const void* bias, const void* res1,
                                      const void* res2, void* C, int64_t M, int64_t N, int64_t K, int32_t epilogue,
                                      const dtas_config* user, void* stream) {
  using namespace dtas;
  clear_error();
  if (M < 0 || N < 0 || K < 0) return fail("gemm_q8: negative extent M=%lld N=%lld K=%lld", (long long)M, (long long)N, (long long)K);
  if (K % 32 != 0) return fail("gemm_q8: K must be a multiple of the scale group, 32 (K=%lld)", (long long)K);
  if (epilogue < DTAS_EPI_BIAS || epilogue > DTAS_EPI_BIAS_GELU) return fail("gemm_q8: unknown epilogue %d", epilogue);
  if (M == 0 || N == 0) return 0;
  if ((K != 0 && (M > INT64_MAX / 8 / K || N > INT64_MAX / 8 / K)) || M > INT64_MAX / 8 / N) return fail("gemm_q8: extents overflow");
  const bool add2 = epilogue == DTAS_EPI_BIAS_ADD2 || epilogue == DTAS_EPI_BIAS_ADD2_CAST_F32;
  if (!A || !Wq || !scale || !C) {
    if (K > 0 || !C) return fail("gemm_q8: NULL buffer");
  }
  if (add2 && (!res1 || !res2)) return fail("gemm_q8: epilogue %d needs both residuals", epilogue);
  if (!add2 && (res1 || res2)) return fail("gemm_q8: epilogue %d takes no residuals", epilogue);
  const int out_bytes = epilogue == DTAS_EPI_BIAS_ADD2_CAST_F32 ? 4 : 2;
  if (overlaps(C, M * N * out_bytes, A, M * K * 2) || overlaps(C, M * N * out_bytes, Wq, N * K) ||
      overlaps(C, M * N * out_bytes, scale, N * (K / 32) * 2) ||
      (add2 && (overlaps(C, M * N * out_bytes, res1, M * N * 2) || overlaps(C, M * N * out_bytes, res2, M * N * 2))))
    return fail("gemm_q8: output overlaps an input");
  // one row with a plain or GELU epilogue is the dequantising GEMV
  if (!user && M == 1 && (epilogue == DTAS_EPI_BIAS || epilogue == DTAS_EPI_BIAS_GELU))
    return dtas_gemv_q8_f16(A, Wq, scale, bias, C, N, K, epilogue, nullptr, stream);
  GemmEpilogue ep = {static_cast<const half_t*>(bias), static_cast<const half_t*>(res1), static_cast<const half_t*>(res2),
                     epilogue, out_bytes == 4 ? 1 : 0, 0.f, 0, 0, 0, 0, 1, 0, static_cast<const half_t*>(scale)};
  const bool vec_ok = aligned(A, 16) && aligned(Wq, 16) && aligned(scale, 2) && N * K < (int64_t{1} << 32) && K > 0;
  const bool stream_ok = K > 0 && K % 256 == 0 && aligned(A, 16) && aligned(Wq, 16) && aligned(scale, 16) && K < (int64_t{1} << 24);
  dtas_config cfg;
  if (user) {
    cfg = *user;
  } else if (!builtin_gemm_q8(M, N, K, stream_ok, vec_ok, &cfg)) {
    void* wbuf = nullptr;
    std::lock_guard<std::recursive_mutex> ws_lock(g_ws_mutex);  // until both launches are enqueued
    if (operand_workspace(static_cast<hipStream_t>(stream), static_cast<size_t>(N) * K * 2, &wbuf) != 0) return -1;
    if (dtas_decode_q8_f16(Wq, scale, wbuf, N, K, nullptr, stream) != 0) return -1;
    return dtas_gemm_f16_fused(A, wbuf, bias, res1, res2, C, M, N, K, epilogue, nullptr, stream);
  }
  hipStream_t s = static_cast<hipStream_t>(stream);
  const half_t* a = static_cast<const half_t*>(A);
  const half_t* w = static_cast<const half_t*>(Wq);  // (bytes; the kernels take the pointer as they take fp16 W)
  if (cfg.variant == DTAS_GEMM_STREAM) {
    const int bm = cfg.tile[0], bn = cfg.tile[1], bk = cfg.tile[2];
    if (!((bm == 16 && bn == 64 && (bk == 512 || bk == 1024)) || ((bm == 32 || bm == 64) && bn == 64 && bk == 512)))
      return fail("gemm_q8: the W-streaming kernel takes tiles 16x64x512, 16x64x1024, 32x64x512 and 64x64x512 for 8-bit weights, got %dx%dx%d", bm, bn, bk);
    if (cfg.block != 256) return fail("gemm_q8: the 64-column streaming tile uses 256 threads, got %d", cfg.block);
    if (M > bm) return fail("gemm_q8: a streaming tile of %d rows cannot hold M=%lld", bm, (long long)M);
    if (!stream_ok) return fail("gemm_q8: the W-streaming kernel needs K %% 256 == 0 and 16-byte aligned A, W and scales");
    return launch_gemm_stream_q8(bm, bk, s, a, w, ep, C, M, N, K);
  }
  if (cfg.variant == DTAS_GEMM_SHARE) {
    if (!share_kernel_exists(cfg.tile[0], cfg.tile[1], true) || cfg.block != 256)
      return fail("gemm_q8: no share kernel for %d rows of A, %d columns per workgroup and %d threads", cfg.tile[0], cfg.tile[1], cfg.block);
    if (M > cfg.tile[0]) return fail("gemm_q8: a share kernel of %d rows cannot hold M=%lld", cfg.tile[0], (long long)M);
    if (!stream_ok) return fail("gemm_q8: the share kernel needs K %% 256 == 0 and 16-byte aligned A, W and scales");
    return launch_gemm_share_q8(cfg.tile[0], cfg.tile[1], s, a, w, ep, C, M, N, K);
  }
  if (cfg.vec == 8 && !vec_ok) cfg.vec = 1;
  if (cfg.vec == 1) {
    int64_t grid = ceil_div(M * N, 256);
    grid = grid > 65536 ? 65536 : grid;
    return launch_gemm_scalar("gemm_q8", static_cast<unsigned>(grid), 1, s, a, w, ep, C, M, N, K, false);
  }
  if (cfg.vec != 8) return fail("gemm_q8: vector width must be 8 (128 bit) or 1, got %d", cfg.vec);
  if (cfg.variant != DTAS_GEMM_MFMA) return fail("gemm_q8: only the MFMA kernels serve 8-bit weights");
  const int sk = cfg.split_k < 1 ? 1 : cfg.split_k;
  int64_t la[7];
  if (describe_gemm(M, N, K, cfg, la) != 0) return -1;
  const int bm = cfg.tile[0], bn = cfg.tile[1];
  if (cfg.block == 512 && bn == 128 && cfg.unroll == 0) {
    const bool quads = K % 64 == 0 && aligned(scale, 4);  // (a row's scales of four k tiles in one load)
#define DTAS_Q8_CASE(BM_, WM_, WN_)                                                                                        \
  if (bm == BM_)                                                                                                           \
  return quads ? launch_mfma<BM_, 128, WM_, WN_, 4, false, true, true, true>(s, a, w, ep, C, M, N, K, sk)                   \
               : launch_mfma<BM_, 128, WM_, WN_, 4, false, true, true>(s, a, w, ep, C, M, N, K, sk)
    DTAS_Q8_CASE(96, 2, 4);
    DTAS_Q8_CASE(128, 4, 2);
    DTAS_Q8_CASE(160, 2, 4);
    DTAS_Q8_CASE(192, 4, 2);
    DTAS_Q8_CASE(256, 4, 2);
#undef DTAS_Q8_CASE
  }
  if (bm == 128 && bn <= 128 && cfg.block != 256) return fail("gemm_q8: the %dx%d MFMA kernel uses 256 threads, got %d", bm, bn, cfg.block);
  if (bm == 256 && bn == 128 && cfg.unroll == 3) return launch_mfma<256, 128, 2, 2, 3, false, true>(s, a, w, ep, C, M, N, K, sk);
  if (bm == 128 && bn == 128 && cfg.unroll == 3) return launch_mfma<128, 128, 2, 2, 3, false, true>(s, a, w, ep, C, M, N, K, sk);
  if (bm == 64 && bn == 64 && cfg.unroll == 2) return launch_mfma<64, 64, 2, 2, 2, false, true>(s, a, w, ep, C, M, N, K, sk);
  if (bm == 128 && bn == 64 && cfg.unroll == 3) return launch_mfma<128, 64, 2, 2, 3, false, true>(s, a, w, ep, C, M, N, K, sk);
  if (bm == 64 && bn == 64 && cfg.unroll == 3) return launch_mfma<64, 64, 2, 2, 3, false, true>(s, a, w, ep, C, M, N, K, sk);
  if (bm == 64 && bn == 128 && cfg.unroll == 3) return launch_mfma<64, 128, 2, 2, 3, false, true>(s, a, w, ep, C, M, N, K, sk);
  return fail("gemm_q8: 8-bit weights come with tiles 256x128, 128x128, 128x64, 64x128 (three stages) and 64x64 (two or three), and with 512 threads {96, 128, 160, 192, 256} x 128 (unroll 0), got %dx%d with %d", bm, bn, cfg.unroll);
}
