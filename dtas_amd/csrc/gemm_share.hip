// SHARE kernel (DTAS_GEMM_SHARE): C[M,N] = A[M,K] . W[N,K]^T for up to 128 rows of A, fp16 or 8-bit weights: W streamed once,
// every CU an equal share of its rows, nothing handed over between workgroups.  Replaces, for these shapes, the kernels
// DTAS's WMMA rule generates (python/dtas/schedule/tir_wmma.py:20-222), which pad M up to a whole tile.
#include "gemm_common.h"

#include <math.h>

namespace dtas {
namespace {

// With few rows of A the launch is one read of W, and what bounds it is how that read is dealt out.  Tiles of 64 columns
// leave CUs idle (7680 columns: 120 tiles for 256 CUs) unless K is split, and a K split ends in a hand-over through memory
// that costs 3 .. 4 us of a launch of 13; tiles also fetch W as 128 bytes per row (4.5 TB/s over the chip) and pull as many
// bytes of A through each CU's L1 as of W, which takes 45 .. 65 KB/us in all.  Here
//  * a workgroup owns N / (number of CUs) columns -- any whole number up to 16 CB, columns past it cost no traffic -- over
//    the whole of K, so every CU streams the same number of bytes and the sums never leave it; A costs M rows once per CU;
//  * W and A come in as 1 KiB direct-to-LDS loads of 2 .. 4 rows x 256 .. 1024 bytes through a ring of NSTG stages;
//  * the four wavefronts share the k steps of a segment, not its columns: every fragment is read from the LDS (and every
//    8-bit weight widened) once per workgroup; their sums meet in the LDS at the end, added in wavefront order.
// Measured with W from memory, us, before / now: 17 rows against 7680 x 2560, 10240 x 2560, 2560 x 10240, 2560 x 2560 13.1 / 9.8,
// 16.5 / 12.0, 19.3 / 16.3, 8.7 / 6.5; 48 rows against 11008 x 4096, 4096 x 4096 26.0 / 20.5, 13.2 / 12.1; 8-bit weights, 48
// rows against 7680 x 2560, 10240 x 2560 17.1 / 10.8, 17.9 / 12.5 (5.0 TB/s of W at 16 rows against 11008 x 4096, where the
// fp16 GEMV takes 14.7 us and this 17.9).  What bounds it: memory delivers W once (17 rows against 10240 x 2560: 53 MB fetched for 52),
// and a CU pulls A in beside it -- 48 rows against 11008 x 4096: 101 MB of A for 90 of W, 35 KB/us per CU at 890 cycles a request.
// In the LDS the 16-byte chunk c of row r sits in slot c ^ f(r), f(r) = 2 (r & 7) + ((r >> 3) & 1), and lane groups 0..3 of a
// fragment read take chunks 0, 2, 1, 3 of the k step (both operands alike): the 16 rows of a lane group fall into 16 bank groups.
// W is the first MFMA operand: register v of lane l is row l & 15 of C, column 4 (l >> 4) + v of a 16x16 block, so that a
// lane finishes four neighbouring columns at once.
// Q8: W is bytes with an fp16 scale per 32 elements of a row (ep.wscale), widened as the dequantiser rounds them.
__device__ __forceinline__ unsigned share_swizzle(unsigned r) { return ((r & 7u) << 1) | ((r >> 3) & 1u); }

template <int CB, int MT, int SEGK, int NSTG, bool Q8>
struct ShareShape {
  static constexpr int kARow = 2 * SEGK, kWRow = Q8 ? SEGK : 2 * SEGK;                 // bytes of a row in a stage
  static constexpr int kWBytes = 16 * CB * kWRow, kABytes = 16 * MT * kARow, kScaleBytes = Q8 ? 4 * 1024 : 0, kScaleRow = SEGK / 16;
  static constexpr int kStage = kWBytes + kABytes + kScaleBytes;
  static constexpr int kWLoads = CB * kWRow / 256, kALoads = MT * kARow / 256;         // per wavefront and segment
  static constexpr int kLoads = kWLoads + kALoads + (Q8 ? 1 : 0);
  static constexpr int kSteps = SEGK / 32 / 4;  // k steps of a wavefront in a segment
  static_assert(!Q8 || SEGK == 256 || SEGK == 512, "8-bit weights: whole 16-byte pieces of scales");
  static_assert(NSTG >= 2 && NSTG * kStage <= kLdsBytes && (NSTG - 1) * kLoads <= 63, "stages / LDS / vmcnt");
  static_assert(4 * CB * MT * 1024 <= NSTG * kStage, "the wavefronts' sums must fit the stages");
};

__device__ __forceinline__ f16x4 share_load4(const half_t* p, int valid) {
  f16x4 v = {};
  if (valid == 4) v = *reinterpret_cast<const f16x4_a2*>(p);
  else
    for (int e = 0; e < valid; ++e) v[e] = p[e];
  return v;
}

template <int CB, int MT, int SEGK, int NSTG, bool Q8>
__global__ void __launch_bounds__(256) gemm_share_kernel(const half_t* __restrict__ A, const half_t* __restrict__ W, GemmEpilogue ep,
                                                         void* __restrict__ C, int64_t M, int64_t N, int64_t K, unsigned cols,
                                                         unsigned longer) {
  using S = ShareShape<CB, MT, SEGK, NSTG, Q8>;
  __shared__ __attribute__((aligned(1024))) char lds[NSTG * S::kStage];
  const unsigned t = threadIdx.x, l = t & 63u;
  const unsigned wv = __builtin_amdgcn_readfirstlane(t >> 6);
  // this workgroup's columns: `cols`, the first `longer` workgroups one more
  const unsigned wg = __builtin_amdgcn_readfirstlane(xcd_contiguous_id(blockIdx.x, gridDim.x));
  const unsigned n0 = wg * cols + (wg < longer ? wg : longer), mine = cols + (wg < longer ? 1u : 0u);
  const unsigned row_bytes = static_cast<unsigned>(K) * 2u, w_row_bytes = Q8 ? static_cast<unsigned>(K) : row_bytes;
  const __amdgpu_buffer_rsrc_t ra = make_rsrc(A, static_cast<unsigned>(M) * row_bytes);
  const __amdgpu_buffer_rsrc_t rw = make_rsrc(reinterpret_cast<const char*>(W) + static_cast<size_t>(n0) * w_row_bytes, mine * w_row_bytes);
  const unsigned sc_row_bytes = static_cast<unsigned>(K >> 5) * 2u;
  const __amdgpu_buffer_rsrc_t rs = make_rsrc(reinterpret_cast<const char*>(ep.wscale) + static_cast<size_t>(n0) * sc_row_bytes, mine * sc_row_bytes);
  const unsigned nseg = static_cast<unsigned>((K + SEGK - 1) / SEGK);

  // the pieces of C this wavefront finishes: 16x16 blocks wv, wv + 4, ... (block = column block * MT + row block); their
  // bias and residual elements are requested before anything else
  constexpr int kMine = (CB * MT + 3) / 4;
  const unsigned i16 = l & 15u, g = l >> 4;
  const bool add2 = ep.kind == DTAS_EPI_BIAS_ADD2 || ep.kind == DTAS_EPI_BIAS_ADD2_CAST_F32;
  int valid[kMine];
  f16x4 bias[kMine], r1[kMine], r2[kMine];
#pragma unroll
  for (int j = 0; j < kMine; ++j) {
    const unsigned b = wv + 4u * j, c0 = (b / MT) * 16u + 4u * g;
    const int64_t row = (b % MT) * 16u + i16;
    valid[j] = b < CB * MT && row < M && c0 < mine ? static_cast<int>(mine - c0 < 4u ? mine - c0 : 4u) : 0;
    bias[j] = r1[j] = r2[j] = f16x4{};
    if (ep.bias) bias[j] = share_load4(ep.bias + n0 + c0, valid[j]);
    if (add2) {
      r1[j] = share_load4(ep.res1 + row * N + n0 + c0, valid[j]);
      r2[j] = share_load4(ep.res2 + row * N + n0 + c0, valid[j]);
    }
  }

  // a load covers `per` rows; wavefront w takes loads w, w + 4, ...; rows repeat the swizzle every 16
  constexpr unsigned kAChunks = S::kARow / 16, kAPer = 1024 / S::kARow, kAPat = 16 / (4 * kAPer);
  constexpr unsigned kWChunks = S::kWRow / 16, kWPer = 1024 / S::kWRow, kWPat = 16 / (4 * kWPer);
  unsigned off_a[kAPat], off_w[kWPat], chunk_a[kAPat], chunk_w[kWPat];
#pragma unroll
  for (unsigned p = 0; p < kAPat; ++p) {
    const unsigned r = (p * 4u + wv) * kAPer + l / kAChunks;
    chunk_a[p] = (l % kAChunks) ^ share_swizzle(r);
    off_a[p] = r * row_bytes + chunk_a[p] * 16u;
  }
#pragma unroll
  for (unsigned p = 0; p < kWPat; ++p) {
    const unsigned r = (p * 4u + wv) * kWPer + l / kWChunks;
    chunk_w[p] = (l % kWChunks) ^ share_swizzle(r);
    off_w[p] = r * w_row_bytes + chunk_w[p] * 16u;
  }
  constexpr unsigned kPieces = SEGK / 256 > 0 ? SEGK / 256 : 1;  // 16-byte pieces of a row's scales in a segment
  const unsigned off_s = l < 4u * CB * kPieces ? (wv * (4u * CB) + l / kPieces) * sc_row_bytes + (l % kPieces) * 16u : kOob;
  const bool ragged_k = K % SEGK != 0;

  auto request = [&](unsigned seg, char* stage) {
    const bool tail = ragged_k && seg + 1 == nseg;  // (uniform)
    const int64_t k0 = static_cast<int64_t>(seg) * SEGK;
#pragma unroll
    for (unsigned i = 0; i < S::kWLoads; ++i) {
      const unsigned at = tail && k0 + chunk_w[i % kWPat] * (Q8 ? 16 : 8) >= K ? kOob : off_w[i % kWPat];
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rw, (lds_ptr_t)(stage + (i * 4 + wv) * 1024), 16, at,
                                               static_cast<int>((i / kWPat) * 16u * w_row_bytes + seg * S::kWRow), 0, 0);
    }
#pragma unroll
    for (unsigned i = 0; i < S::kALoads; ++i) {
      const unsigned at = tail && k0 + chunk_a[i % kAPat] * 8 >= K ? kOob : off_a[i % kAPat];
      __builtin_amdgcn_raw_ptr_buffer_load_lds(ra, (lds_ptr_t)(stage + S::kWBytes + (i * 4 + wv) * 1024), 16, at,
                                               static_cast<int>((i / kAPat) * 16u * row_bytes + seg * S::kARow), 0, 0);
    }
    if constexpr (Q8) {
      // (a piece past K would be the next row's first scales, which may be anything: inf x the zeros there is NaN)
      const unsigned at = tail && k0 + (l % kPieces) * 256u >= K ? kOob : off_s;
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (lds_ptr_t)(stage + S::kWBytes + S::kABytes + wv * 1024), 16, at, static_cast<int>(seg * S::kScaleRow), 0, 0);
    }
  };
#pragma unroll
  for (int p = 0; p < NSTG - 1; ++p)
    if (static_cast<unsigned>(p) < nseg) request(p, lds + p * S::kStage);

  f32x4v acc[CB][MT];
#pragma unroll
  for (int c = 0; c < CB; ++c)
#pragma unroll
    for (int i = 0; i < MT; ++i) acc[c][i] = f32x4v{0.f, 0.f, 0.f, 0.f};
  const unsigned perm = ((g & 1u) << 1) | (g >> 1);
  const unsigned x16 = (perm ^ share_swizzle(i16)) * 16u, x8 = ((perm >> 1) ^ share_swizzle(i16)) * 16u;
  int cur = 0;
  for (unsigned s = 0; s < nseg; ++s) {
    wait_whole_tiles<S::kLoads, NSTG - 2>(static_cast<int>(nseg - 1 - s));
    __builtin_amdgcn_s_barrier();
    if (s == 0) {
#pragma unroll
      for (int j = 0; j < kMine; ++j) asm volatile("" ::"v"(bias[j]), "v"(r1[j]), "v"(r2[j]));  // (they have arrived: they stay in registers)
    }
    DTAS_SCHED_FENCE();
    const int into = cur == 0 ? NSTG - 1 : cur - 1;  // the stage of the segment before, read by everybody before this barrier
    if (s + NSTG - 1 < nseg) request(s + NSTG - 1, lds + into * S::kStage);
    DTAS_SCHED_FENCE();
    const char* stage = lds + cur * S::kStage;
#pragma unroll
    for (int q = 0; q < S::kSteps; ++q) {
      const unsigned ks = q * 4u + wv;
      f16x8 fw[CB], fa[MT];
#pragma unroll
      for (int c = 0; c < CB; ++c) {
        const unsigned r = c * 16u + i16;
        if constexpr (Q8) {
          const u32x2 raw = *reinterpret_cast<const u32x2*>(stage + r * S::kWRow + (perm & 1u) * 8u + (x8 ^ (ks * 32u)));
          const half_t sc = *reinterpret_cast<const half_t*>(stage + S::kWBytes + S::kABytes + (r / (4u * CB)) * 1024u + (r % (4u * CB)) * S::kScaleRow + ks * 2u);
          const f16x2 s2 = {sc, sc};
          f16x2 d0, d1, d2, d3;
          dequant_q8_word(raw[0], s2, d0, d1);
          dequant_q8_word(raw[1], s2, d2, d3);
          fw[c] = f16x8{d0[0], d0[1], d1[0], d1[1], d2[0], d2[1], d3[0], d3[1]};
        } else {
          fw[c] = *reinterpret_cast<const f16x8*>(stage + r * S::kWRow + (x16 ^ (ks * 64u)));
        }
      }
#pragma unroll
      for (int i = 0; i < MT; ++i)
        fa[i] = *reinterpret_cast<const f16x8*>(stage + S::kWBytes + (i * 16u + i16) * S::kARow + (x16 ^ (ks * 64u)));
#pragma unroll
      for (int c = 0; c < CB; ++c)
#pragma unroll
        for (int i = 0; i < MT; ++i) acc[c][i] = __builtin_amdgcn_mfma_f32_16x16x32_f16(fw[c], fa[i], acc[c][i], 0, 0, 0);
    }
    DTAS_SCHED_FENCE();
    cur = cur + 1 == NSTG ? 0 : cur + 1;
  }

  // the four wavefronts' sums meet in the LDS, added in wavefront order
  __syncthreads();
  f32x4v* sums = reinterpret_cast<f32x4v*>(lds);
#pragma unroll
  for (int c = 0; c < CB; ++c)
#pragma unroll
    for (int i = 0; i < MT; ++i) sums[(wv * (CB * MT) + c * MT + i) * 64 + l] = acc[c][i];
  __syncthreads();
#pragma unroll
  for (int j = 0; j < kMine; ++j) {
    const unsigned b = wv + 4u * j;
    if (valid[j] == 0) continue;
    f32x4v sum = sums[b * 64 + l];
#pragma unroll
    for (int k = 1; k < 4; ++k) sum += sums[(k * (CB * MT) + b) * 64 + l];
    f16x4 o = {static_cast<half_t>(sum[0]), static_cast<half_t>(sum[1]), static_cast<half_t>(sum[2]), static_cast<half_t>(sum[3])};
    const bool hb = ep.bias != nullptr;
    if (ep.kind == DTAS_EPI_BIAS_GELU) o = gelu_erf_f16_steps_vec<f16x4, 4>(o, hb, bias[j]);
    else if (add2) o = add_steps_vec<f16x4, true>(o, hb, bias[j], r1[j], r2[j]);
    else o = add_steps_vec<f16x4, false>(o, hb, bias[j], r1[j], r2[j]);
    const int64_t at = static_cast<int64_t>((b % MT) * 16u + i16) * N + n0 + (b / MT) * 16u + 4u * g;
    if (ep.out_f32) {
      float* c = static_cast<float*>(C) + at;
      if (valid[j] == 4) *reinterpret_cast<f32x4v_a4*>(c) = f32x4v{static_cast<float>(o[0]), static_cast<float>(o[1]), static_cast<float>(o[2]), static_cast<float>(o[3])};
      else
        for (int e = 0; e < valid[j]; ++e) c[e] = static_cast<float>(o[e]);
    } else {
      half_t* c = static_cast<half_t*>(C) + at;
      if (valid[j] == 4) *reinterpret_cast<f16x4_a2*>(c) = o;
      else
        for (int e = 0; e < valid[j]; ++e) c[e] = o[e];
    }
  }
}

template <int CB, int MT, int SEGK, int NSTG, bool Q8>
int launch_share(unsigned grid, hipStream_t s, const half_t* A, const half_t* W, const GemmEpilogue& ep, void* C, int64_t M, int64_t N, int64_t K) {
  hipLaunchKernelGGL((gemm_share_kernel<CB, MT, SEGK, NSTG, Q8>), dim3(grid), dim3(256), 0, s, A, W, ep, C, M, N, K,
                     static_cast<unsigned>(N / grid), static_cast<unsigned>(N % grid));
  return check_launch("gemm");
}

}  // namespace

#define DTAS_SHARE_CASE(ROWS_, COLS_, SEG_, NS_, Q8_) \
  if (rows == ROWS_ && cols == COLS_) return launch_share<COLS_ / 16, ROWS_ / 16, SEG_, NS_, Q8_>(grid, s, a, w, ep, C, M, N, K)
int launch_gemm_share(int rows, int cols, hipStream_t s, const half_t* a, const half_t* w, const GemmEpilogue& ep, void* C, int64_t M,
                      int64_t N, int64_t K) {
  const unsigned grid = static_cast<unsigned>(share_grid(N, cols));
  DTAS_SHARE_CASE(16, 16, 512, 4, false); DTAS_SHARE_CASE(16, 32, 256, 3, false); DTAS_SHARE_CASE(16, 64, 256, 3, false);
  DTAS_SHARE_CASE(16, 128, 128, 3, false);
  DTAS_SHARE_CASE(32, 16, 256, 4, false); DTAS_SHARE_CASE(32, 32, 256, 4, false); DTAS_SHARE_CASE(32, 48, 256, 3, false);
  DTAS_SHARE_CASE(32, 64, 256, 3, false); DTAS_SHARE_CASE(32, 128, 128, 3, false);
  DTAS_SHARE_CASE(48, 16, 256, 4, false); DTAS_SHARE_CASE(48, 32, 256, 3, false); DTAS_SHARE_CASE(48, 48, 256, 3, false);
  DTAS_SHARE_CASE(48, 64, 128, 4, false); DTAS_SHARE_CASE(48, 128, 128, 3, false);
  DTAS_SHARE_CASE(64, 16, 256, 3, false); DTAS_SHARE_CASE(64, 32, 256, 3, false); DTAS_SHARE_CASE(64, 48, 128, 4, false);
  DTAS_SHARE_CASE(64, 64, 128, 4, false); DTAS_SHARE_CASE(64, 128, 128, 3, false);
  DTAS_SHARE_CASE(96, 16, 128, 5, false); DTAS_SHARE_CASE(96, 32, 128, 4, false); DTAS_SHARE_CASE(96, 48, 128, 4, false);
  DTAS_SHARE_CASE(128, 48, 128, 3, false);
  return fail("gemm: no share kernel for %d rows of A and %d columns", rows, cols);
}

int launch_gemm_share_q8(int rows, int cols, hipStream_t s, const half_t* a, const half_t* w, const GemmEpilogue& ep, void* C, int64_t M,
                         int64_t N, int64_t K) {
  const unsigned grid = static_cast<unsigned>(share_grid(N, cols));
  DTAS_SHARE_CASE(16, 16, 512, 4, true); DTAS_SHARE_CASE(16, 32, 512, 3, true); DTAS_SHARE_CASE(16, 48, 512, 3, true);
  DTAS_SHARE_CASE(16, 64, 256, 5, true); DTAS_SHARE_CASE(16, 128, 256, 3, true);
  DTAS_SHARE_CASE(32, 16, 512, 3, true); DTAS_SHARE_CASE(32, 32, 512, 3, true); DTAS_SHARE_CASE(32, 48, 256, 4, true);
  DTAS_SHARE_CASE(32, 64, 256, 4, true); DTAS_SHARE_CASE(32, 128, 256, 3, true);
  DTAS_SHARE_CASE(48, 16, 256, 4, true); DTAS_SHARE_CASE(48, 32, 256, 4, true); DTAS_SHARE_CASE(48, 48, 256, 3, true);
  DTAS_SHARE_CASE(48, 64, 256, 3, true); DTAS_SHARE_CASE(48, 128, 256, 2, true);
  DTAS_SHARE_CASE(64, 16, 256, 3, true); DTAS_SHARE_CASE(64, 32, 256, 3, true); DTAS_SHARE_CASE(64, 48, 256, 3, true);
  DTAS_SHARE_CASE(64, 64, 256, 3, true); DTAS_SHARE_CASE(64, 128, 256, 2, true);
  DTAS_SHARE_CASE(80, 16, 256, 3, true); DTAS_SHARE_CASE(96, 32, 256, 2, true); DTAS_SHARE_CASE(96, 48, 256, 2, true);
  return fail("gemm_q8: no share kernel for %d rows of A and %d columns", rows, cols);
}
#undef DTAS_SHARE_CASE

// Which share kernel serves M rows against an N x K W, if any leads there (false: none).  The rows of A are rounded up to a
// kernel's; the columns are the fewest that give every CU one workgroup (16 rows of A: two, while 32 columns each are
// enough: 11008 x 4096 17.0 us against 17.5 with one of 48), 128 per workgroup beyond.
static bool share_shape(bool q8, int64_t M, int64_t N, int* rows, int* cols) {
  const int64_t per_cu = ceil_div(N, kNumCU);
  *rows = M <= 16 ? 16 : M <= 32 ? 32 : M <= 48 ? 48 : M <= 64 ? 64 : M <= 96 ? 96 : 128;
  if (q8 && M > 64 && M <= 80 && per_cu <= 16) *rows = 80;
  if (!q8 && *rows == 16) *cols = per_cu <= 16 ? 16 : per_cu <= 56 ? 32 : per_cu <= 64 ? 64 : 128;
  else *cols = per_cu <= 16 ? 16 : per_cu <= 32 ? 32 : per_cu <= 48 ? 48 : per_cu <= 64 ? 64 : 128;
  return share_kernel_exists(*rows, *cols, q8);
}

// fp16 weights.  Two estimates in us, fitted to sweeps of 3 .. 128 rows against W of 300 .. 50280 rows and 256 .. 14336
// columns (W from memory).  Share: 3.3 + the root of the squares of what W costs from memory (6.6 TB/s; 5.4 with 128
// columns) and what A and the CU's part of W cost through its L1 (65 KB/us, 55 where the segments are short: 128 columns, or
// more than 64 rows).  The other kernels: 6.5 us + W at 5.5 TB/s + 0.03 per row (wide W: x the rounds of 64-column tiles over
// their exact number), and beyond 64 rows 8.5 us + W at 4.2 TB/s, 8.1 + 4.5 TB/s where their tiles split K evenly (up to 4096
// columns, and long K).  What the line separates, share / others: 64 rows against 4096 x 4096 13.7 / 13.5, 48 rows 12.1 / 13.2; 32
// rows against 4096 x 11008 25.3 / 24.0, 17 rows 22.3 / 23.5; 128 rows against 10240 x 2560 21.7 / 26.7, 7680 x 2560 19.0 / 17.8.
// What the estimates do not see, share / others:
//  * few long rows of W: a workgroup's segments follow one another at 0.8 .. 1.2 us per 1024 of K, while the W-streaming kernel
//    deals K out in slices -- 8 rows against 300 x 14336 14.1 / 8.4, 1024 x 8192 9.5 / 8.6, 17 rows against 512 x 8192 12.3 / 9.3.
//    Its workgroups must fit one round; with 256 of them the share kernel is level (2048 x 8192) and beyond it ahead (0.7);
//  * rows of W 20 or 28 KiB apart (K = 10240, 14336): 33 rows against 5120 x 10240 30.4 / 26.6, 65 against 8192 x 10240 55.3 / 44.6, 5
//    against 8192 x 14336 50.5 / 45.9; not at 12288 (0.82), and not beyond 8192 rows of W (11008: 0.80);
//  * wide W whose rows are short (17 rows against 50280 x 256 12.8 / 11.7), or a power of two long and no fewer than 7/8 of a
//    round of 128-column tiles, which then run as if in whole rounds (48 rows against 28672 x 4096 1.05, x 2560 0.87);
//  * more than 64 rows against short rows of a W beyond 8192 (128 rows against 11008 x 256 8.2 / 6.7,
//    x 1024 13.2 / 12.4, 10240 x 1536 16.3 / 19.4; 80 rows against 11008 x 512 1.03, 10240 x 1024 0.93).
bool share_leads(int64_t M, int64_t N, int64_t K, int* rows, int* cols) {
  if (M < 3 || M > 128 || N < 256 || K < 256 || !share_shape(false, M, N, rows, cols)) return false;
  if (N > 0x7fffffff || K * 2 * 128 >= (int64_t{1} << 31)) return false;  // (describe_gemm refuses these; other kernels hold them)
  const bool wide = *cols == 128;
  if (wide && ((K < 2048 && M > 32) || (K <= 512 && M > 16 && N > 32768))) return false;  // (28672 x 1024: 48 rows 15.6 / 15.5 us, 64 rows 16.7 / 15.9)
  if (*cols == 48 && M > 64 && K < (M > 96 ? 1536 : 1024)) return false;
  if (M <= 32 && ceil_div(N, 64) * ceil_div(K, M <= 16 ? 1024 : 512) <= 240 && (K >= 8192 || (K >= 6144 && N < 1024))) return false;
  const double m = static_cast<double>(M), w_mb = 2e-6 * static_cast<double>(N) * static_cast<double>(K);
  const double a_kb = 2e-3 * m * static_cast<double>(K), w_cu_kb = w_mb * 1e3 / kNumCU;
  const double hbm = w_mb / (wide ? 5.4 : 6.6), l1 = (a_kb + w_cu_kb) / (wide || M > 64 ? 55.0 : 65.0);
  const double pitch = K > 8192 && K % 4096 == 2048 && N > (M < 32 ? 6144 : 4096) && N <= 8192 ? 1.2 : 1.0;
  const double share = 3.3 + pitch * sqrt(hbm * hbm + l1 * l1);
  const int64_t t64 = ceil_div(N, 64), t128 = ceil_div(N, 128);
  const bool whole = (K & (K - 1)) == 0 && t128 <= kNumCU && t128 * 8 >= 7 * kNumCU;
  const double waste = wide && !whole ? static_cast<double>(ceil_div(t64, kNumCU) * kNumCU) / static_cast<double>(t64) : 1.0;
  const bool even = N <= 4096 || (N <= 10240 && K > 5120);
  const double others = M <= 64 ? 6.5 + w_mb / 5.5 * waste + 0.03 * m : (even ? 8.1 + w_mb / 4.5 : 8.5 + w_mb / 4.2) + 0.02 * (m - 64.0);
  return share < others;
}

// 8-bit weights: the other kernels widen every weight once per row of tiles, so the share kernel leads until the rows of A
// that each CU pulls in (2 M K bytes) outgrow both 660 KB and 6.5 times its part of W: 2560 x 10240, 32 rows 18.8 us
// against 19.4, 48 rows 24.5 / 21.2; 4096 x 11008, 48 rows 27.0 / 28.6, 64 rows 33.2 / 29.3; 7680 x 2560, 96 rows 18.2 / 19.7,
// 128 rows (no kernel) 21.2 / 20.8.  And not, from a sweep of 2 .. 96 rows against W of 300 .. 50280 rows and 256 .. 14336 columns
// (W from memory, share / others):
//  * against few long rows of W, which the W-streaming kernel and the tiles take in slices of K while a workgroup here walks
//    them whole: 16 rows against 300 x 14336 18.7 / 8.3, 1024 x 8192 11.8 / 8.7, 1024 x 4096 7.5 / 7.3, 2048 x 2560 0.84, 2560 x 10240
//    0.99; 48 rows against 1024 x 6144 15.7 / 13.5, 2560 x 9216 21.5 / 19.7, 3072 x 10240 0.88; 64 rows against 1536 x 4096 1.07,
//    2048 x 5120 0.95, 6144 x 10240 1.05, 7680 x 10240 0.93.  The fewest rows of W, by the rows of A and K:
//  * more than 64 rows: 80 against 8192 x 8192 1.06, 5120 x 4096 1.05, 2048 x 4096 1.05, but 10240 x 5120 0.95, 4096 x 4096
//    0.92, any W of up to 3328 columns 0.64 .. 1.03, and beyond 10240 rows of W 0.67 .. 0.91;
//  * against a wide W of up to 512 columns (128 columns per workgroup): 8 rows against 50280 x 512 12.8 / 9.9, 17 rows against 28672
//    x 512 1.09, 20480 x 256 0.85, 64 rows against 32000 x 512 11.7 / 9.8; more than 32 rows of A against more than 32768 rows of W
//    are the exception: what is left there writes the weights out in fp16 first (50280 x 512 17.3 / 32.4).
bool share_leads_q8(int64_t M, int64_t N, int64_t K, int* rows, int* cols) {
  if (M > 96 || N < 256 || !share_shape(true, M, N, rows, cols)) return false;
  if (K <= 512 && N > (M <= 16 ? 64 : 80) * kNumCU && (M <= 32 || N <= 32768)) return false;
  if (M > 64) return K < 3584 || N > 10240 || (K < 6144 && N > 5120) || (K < 5120 && N > 2048 && N <= 4096);
  const int64_t least = M <= 32   ? (K >= 8192 ? 2560 : K >= 6144 ? 1536 : K >= 3328 ? 1024 : 0)
                        : M <= 48 ? (K >= 9216 ? 3072 : K >= 6144 ? 1536 : K >= 4096 ? 1024 : 0)
                                  : (K >= 9216 ? 6145 : K >= 3584 ? 2048 : 0);
  if (N < least) return false;
  const double a_kb = 2e-3 * static_cast<double>(M) * static_cast<double>(K);
  const double w_cu_kb = 1.0625e-3 * static_cast<double>(N) * static_cast<double>(K) / kNumCU;
  return a_kb <= 660.0 || a_kb <= 6.5 * w_cu_kb;
}

}  // namespace dtas
