// 16-bit clipped products whose operands the LDS-DMA core cannot read as they
// are: rows that are not 16-byte aligned (odd layer widths), a contraction axis
// that is no multiple of a k-tile in the NN layout, samples beyond a 32-bit
// buffer record.  The same tiles, MFMA code and clipped sum as the streamed
// schedule (wgrad_stream.hpp), fed through registers: 16-byte global loads of any
// alignment (legal on amdhsa targets) two k-tiles ahead, written to the LDS
// slots the DMA would have filled.  Values past an operand's edge are written as
// zeros.
//
// Beside the MFMAs a k-tile costs 6 loads and 6 LDS writes per thread, which is
// why aligned operands keep the DMA.  4 x 512, 768 -> 50257 bf16 (158 GFLOP),
// kernel times: sum 1319 -> 321 us, norms 1099 -> 404 us from the products, 164 us
// in split Gram form; before, 128 x 128 tiles loaded unaligned rows value by value.
#pragma once

#include <type_traits>

#include "wgrad_stream.hpp"

namespace fdp {
namespace wg {

// Eight consecutive 16-bit values from p; `left` values exist (the rest read as
// 0).  (The element loop stays a loop: it runs at an operand's last columns only,
// and unrolled it would hold registers that the accumulators need.)
__device__ __forceinline__ u32x4 load_oct(const uint16_t* p, int64_t left) {
  u32x4 v = {0, 0, 0, 0};
  if (left >= 8) {
    __builtin_memcpy(&v, p, 16);
  } else if (left > 0) {
    uint64_t w[2] = {0, 0};
#pragma unroll 1
    for (int e = 0; e < static_cast<int>(left); ++e) {
      const uint64_t x = static_cast<uint64_t>(p[e]) << (16 * (e & 3));
      w[0] |= e < 4 ? x : 0;
      w[1] |= e < 4 ? 0 : x;
    }
    v = u32x4{static_cast<uint32_t>(w[0]), static_cast<uint32_t>(w[0] >> 32),
              static_cast<uint32_t>(w[1]), static_cast<uint32_t>(w[1] >> 32)};
  }
  return v;
}

// One operand's per-thread part of a k-tile: L chunks of 16 bytes.  KC: k
// contiguous ([R, K] rows), else k-strided ([K, R]).
template <int R, int BK, int L, bool KC>
struct StagedOperand {
  const char* base;      // the next k-tile's first value (uniform)
  uint32_t voff[L];      // byte offsets of this thread's chunks from it

  __device__ __forceinline__ static int slot_row(int j) {  // KC: the tile's row; else its k
    return (((threadIdx.x >> 6) * L + j) * 64 + (threadIdx.x & 63)) / kSlots;
  }
  __device__ __forceinline__ static int slot_col(int j) {  // KC: its first k; else its first column
    const int slot = ((threadIdx.x >> 6) * L + j) * 64 + (threadIdx.x & 63), r = slot / kSlots;
    return 8 * ((slot % kSlots) ^ (KC ? dma::kc_swz<BK>(r) : dma::swz(r)));
  }
  static constexpr int kSlots = KC ? BK / 8 : dma::row_chunks(R);
  static_assert(KC || R % 128 == 0, "no padding slots");

  // left: rows (KC) or columns of the operand from the tile's first on.  Chunks
  // that lie wholly past them load the tile's first row or column instead: no
  // output that counts depends on those.
  __device__ inline void init(int64_t ld, int64_t left) {
#pragma unroll
    for (int j = 0; j < L; ++j) {
      int r = slot_row(j), c = slot_col(j);
      if (KC && r >= left) r = 0;
      if (!KC && c >= left) c = 0;
      voff[j] = static_cast<uint32_t>((r * ld + c) * 2);
    }
  }
  __device__ __forceinline__ void load(u32x4 (&r)[L]) {
#pragma unroll
    for (int j = 0; j < L; ++j) {
      asm volatile("" : "+v"(voff[j]));  // (keeps base + offset a scalar-base access)
      __builtin_memcpy(&r[j], base + voff[j], 16);
    }
  }
  // Values past `rows` rows / `cols` columns from the k-tile's first value are zeros.
  __device__ __forceinline__ void load_checked(u32x4 (&r)[L], int64_t ld, int64_t rows,
                                               int64_t cols) const {
#pragma unroll 1
    for (int j = 0; j < L; ++j) {
      const int row = slot_row(j), col = slot_col(j);
      const u32x4 v = load_oct(reinterpret_cast<const uint16_t*>(base) + row * ld + col,
                               row < rows ? cols - col : 0);
#pragma unroll
      for (int i = 0; i < L; ++i)
        if (i == j) r[i] = v;
    }
  }
  __device__ __forceinline__ void put(const u32x4 (&r)[L], FDP_LDS char* tile) const {
#pragma unroll
    for (int j = 0; j < L; ++j)
      *reinterpret_cast<FDP_LDS u32x4*>(tile + (threadIdx.x >> 6) * L * 1024 + j * 1024 +
                                        (threadIdx.x & 63) * 16) = r[j];
  }
};

// acc over the k-tiles of samples [b0, b0 + nsamp): start(j) before sample j's
// first k-tile returns whether the sample is contracted at all.
//
// A k-tile with another one behind it in its sample is loaded without checks: a
// chunk that straddles the right edge then reads into the next row, which
// exists, and the columns past the edge are ignored.  The last k-tile of a
// sample (past it there may be no memory) is loaded value by value where needed.
template <class DT, class G, class Start>
__device__ __forceinline__ void staged_gemm(const Args& p, int64_t b0, int nsamp, int64_t m0,
                                            int64_t n0, f32x16 (&acc)[G::FI][G::FJ],
                                            FDP_LDS char* ring, const Start& start) {
  constexpr int BK = G::BK;
  const int wave = threadIdx.x >> 6;
  const int64_t nk = (p.K + BK - 1) / BK, nq = nsamp * nk;
  if (nq <= 0) return;
  dma::FragOffsets<G> fo;
  fo.init((wave / G::WGN) * G::WM, (wave % G::WGN) * G::WN);
  StagedOperand<G::BM, BK, G::LOADS_A, G::AKC> oa;
  StagedOperand<G::BN, BK, G::LOADS_B, G::BKC> ob;
  oa.init(p.lda, p.M - m0);
  ob.init(p.ldb, p.N - n0);
  const int64_t step_a = (G::AKC ? BK : BK * p.lda) * 2, step_b = (G::BKC ? BK : BK * p.ldb) * 2;
  oa.base = reinterpret_cast<const char*>(static_cast<const uint16_t*>(p.a) + b0 * p.sab +
                                          (G::AKC ? m0 * p.lda : m0));
  ob.base = reinterpret_cast<const char*>(static_cast<const uint16_t*>(p.b) + b0 * p.sbb +
                                          (G::BKC ? n0 * p.ldb : n0));
  const int64_t wrap_a = p.sab * 2 - nk * step_a, wrap_b = p.sbb * 2 - nk * step_b;
  // k-tiles [0, fast) of a sample need no checks (offsets in a tile below 2^32
  // bytes; a row holds a chunk, so that one more row is enough to read into)
  const bool plain = p.lda < (1 << 21) && p.ldb < (1 << 21) &&
                     (G::AKC || p.lda >= 8) && (G::BKC || p.ldb >= 8);
  const bool whole = p.M - m0 >= G::BM && p.N - n0 >= G::BN && p.K % BK == 0;
  const int64_t fast = !plain ? 0 : whole ? nk : nk - 1;
  int64_t iq = 0, ik = 0;  // the k-tile issued next: overall, and inside its sample
  struct Regs {
    u32x4 a[G::LOADS_A], b[G::LOADS_B];
  } r0, r1;
  auto issue = [&](Regs& r) {
    if (ik < fast && iq < nq) {
      oa.load(r.a);
      ob.load(r.b);
    } else {
      const int64_t kleft = iq < nq ? p.K - ik * BK : 0;
      oa.load_checked(r.a, p.lda, G::AKC ? (iq < nq ? p.M - m0 : 0) : kleft,
                      G::AKC ? kleft : p.M - m0);
      ob.load_checked(r.b, p.ldb, G::BKC ? (iq < nq ? p.N - n0 : 0) : kleft,
                      G::BKC ? kleft : p.N - n0);
      dma::wait_vm<0>();  // (the other path's loads are then the only ones to count)
    }
    oa.base += step_a;
    ob.base += step_b;
    ++iq;
    if (++ik == nk) {
      ik = 0;
      oa.base += wrap_a;
      ob.base += wrap_b;
    }
  };
  auto put = [&](const Regs& r, int s) {
    oa.put(r.a, ring + s * G::STAGE);
    ob.put(r.b, ring + s * G::STAGE + G::TILE_A);
  };
  int64_t ck = 0;  // k-tile being contracted, and its sample
  int cs = 0;
  bool live = false;
  auto step = [&](int s, Regs& next, Regs& fill) {
    issue(fill);
    if (ck == 0) live = start(cs);
    if (live) dma::compute_stage<DT, G>(ring + s * G::STAGE, fo, acc);
    if (++ck == nk) {
      ck = 0;
      ++cs;
    }
    put(next, s ^ 1);
    dma::barrier();
  };
  issue(r0);
  issue(r1);
  put(r0, 0);
  dma::barrier();
  for (int64_t q = 0; q < nq; q += 2) {
    step(0, r1, r0);
    if (q + 1 < nq) step(1, r0, r1);
  }
  __syncthreads();
}

// Per-(tile, sample) squares of the products: grid (tiles, up to kStagedGridY
// samples at a time).
constexpr int kStagedGridY = 32768;
template <class DT, class G>
__global__ __launch_bounds__(NT, 2) void staged_norm_kernel(Args p) {
  __shared__ __attribute__((aligned(16))) char ring[2 * G::STAGE];
  __shared__ float red[NT / kWave];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int tiles = p.tiles_m * p.tiles_n;
  int64_t m0, n0;
  tile_coords_g<G>(p, blockIdx.x, m0, n0);
  for (int64_t b = blockIdx.y; b < p.B; b += gridDim.y) {
    f32x16 acc[G::FI][G::FJ];
    zero_blocks<G>(acc);
    staged_gemm<DT, G>(p, b, 1, m0, n0, acc, (FDP_LDS char*)ring, [](int) { return true; });
    const float s = masked_squares<G>(p, m0, n0, acc);
    if (lane == 0) red[wave] = s;
    __syncthreads();
    if (threadIdx.x == 0)
      p.partials[b * tiles + blockIdx.x] = (red[0] + red[1]) + (red[2] + red[3]);
    __syncthreads();
  }
}

// The clipped sum, as clipsum_kernel (no bias).
template <class DT, class G>
__global__ __launch_bounds__(NT, 2) void staged_sum_kernel(Args p) {
  // (the output staging reuses the ring)
  constexpr int RING = 2 * G::STAGE > G::WM * G::BN * 4 ? 2 * G::STAGE : G::WM * G::BN * 4;
  __shared__ __attribute__((aligned(16))) char ring[RING];
  __shared__ float cfac[kSumFacMax];
  const int tiles = p.tiles_m * p.tiles_n;
  const int lw = logical_wg(blockIdx.x, gridDim.x);
  const int g = lw / tiles, tile = lw % tiles;
  int64_t m0, n0;
  tile_coords_g<G>(p, tile, m0, n0);
  const int64_t b0 = int64_t(g) * p.spg;
  const int64_t b1 = b0 + p.spg < p.B ? b0 + p.spg : p.B;
  const int nsamp = static_cast<int>(b1 - b0);
  f32x16 acc[G::FI][G::FJ];
  zero_blocks<G>(acc);
  if (p.fac_parts > 0) group_factors(p, b0, nsamp, tile, cfac);
  __syncthreads();
  float c_prev = 0.f;
  bool any = false;
  staged_gemm<DT, G>(p, b0, nsamp, m0, n0, acc, (FDP_LDS char*)ring, [&](int j) {
    const float c = p.fac_parts > 0 ? cfac[j] : p.factors[b0 + j];
    if (c != 0.f) start_sample<G>(c, c_prev, any, acc);
    return c != 0.f;  // a zero factor contributes exactly nothing
  });
  __syncthreads();
  const bool single = p.groups == 1;
  const float scale = any ? c_prev * (single ? p.out_scale : 1.f) : 0.f;
  float* lds = reinterpret_cast<float*>(ring);
  float* grows = single ? nullptr : p.group_out + int64_t(g) * p.M * p.N;
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    if (!single) store_half<F32, G>(p, m0, n0, h, acc, scale, lds, grows);
    else if (p.out_dtype == FDP_BF16) store_half<BF16, G>(p, m0, n0, h, acc, scale, lds, nullptr);
    else if (p.out_dtype == FDP_F16) store_half<F16, G>(p, m0, n0, h, acc, scale, lds, nullptr);
    else store_half<F32, G>(p, m0, n0, h, acc, scale, lds, nullptr);
  }
}

// ------------------------------------------------------------ split Gram norm
// ||G_b||^2 = sum (g g^T) .* (x x^T) (see gram_norm_kernel) for unaligned TN
// operands of which one is much wider than the samples are long (a vocabulary
// head): a sample has few 128 x 128 Gram tiles, so the wider operand's are
// contracted in `parts` ranges of its features by a workgroup each
// (gram_part_kernel, fp32 partial tiles in the order of the accumulators), and
// gram_join_kernel adds a tile's parts, forms the other operand's Gram tile and
// sums their product.  4 x 512, 768 -> 50257 bf16: a third of the flops of
// squaring the products.
using GramGeom = dma::Geom<kGramT, kGramT, 64, 2, 2, true, true>;

struct SplitGram {
  const void *wide, *narrow;  // [B] x [T, features]
  int64_t B, T, wide_n, narrow_n;
  int64_t wide_s, wide_ld, narrow_s, narrow_ld;
  int nt, per_sample, parts;
  int64_t span;  // features per part (a multiple of GramGeom::BK)
  float* part;   // [B * per_sample, parts, kGramT * kGramT]
  float* partials;  // [B, per_sample]
};

// The Gram tile of rows t0.. and s0.. over features [f0, f0 + n) of a sample.
template <class DT>
__device__ __forceinline__ void gram_tile(const void* rows, int64_t ld, int64_t T, int64_t t0,
                                          int64_t s0, int64_t f0, int64_t n, f32x16 (&acc)[2][2],
                                          FDP_LDS char* ring) {
  Args q{};
  q.a = static_cast<const uint16_t*>(rows) + t0 * ld + f0;
  q.b = static_cast<const uint16_t*>(rows) + s0 * ld + f0;
  q.lda = q.ldb = ld;
  q.M = T - t0;
  q.N = T - s0;
  q.K = n;
  staged_gemm<DT, GramGeom>(q, 0, 1, 0, 0, acc, ring, [](int) { return true; });
}

template <class DT>
__global__ __launch_bounds__(NT, 2) void gram_part_kernel(SplitGram p) {
  __shared__ __attribute__((aligned(16))) char ring[2 * GramGeom::STAGE];
  // neighbouring workgroups share a sample and a range of features
  const int64_t lw = logical_wg(blockIdx.x, gridDim.x);
  const int64_t r = lw % p.per_sample, bp = lw / p.per_sample;
  const int64_t part = bp % p.parts, b = bp / p.parts;
  int ti, tj;
  gram_item(static_cast<int>(r), p.nt, ti, tj);
  const int64_t f0 = part * p.span, left = p.wide_n - f0;
  f32x16 acc[2][2];
  zero(acc);
  gram_tile<DT>(static_cast<const uint16_t*>(p.wide) + b * p.wide_s, p.wide_ld, p.T,
                int64_t(ti) * kGramT, int64_t(tj) * kGramT, f0, left < p.span ? left : p.span, acc,
                (FDP_LDS char*)ring);
  float* out = p.part + ((b * p.per_sample + r) * p.parts + part) * (kGramT * kGramT);
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) out[((i * 2 + j) * 16 + e) * NT + threadIdx.x] = acc[i][j][e];
}

template <class DT>
__global__ __launch_bounds__(NT, 2) void gram_join_kernel(SplitGram p) {
  __shared__ __attribute__((aligned(16))) char ring[2 * GramGeom::STAGE];
  __shared__ float red[NT / kWave];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int64_t b = blockIdx.x / p.per_sample, r = blockIdx.x % p.per_sample;
  int ti, tj;
  gram_item(static_cast<int>(r), p.nt, ti, tj);
  f32x16 acc[2][2];
  zero(acc);
  gram_tile<DT>(static_cast<const uint16_t*>(p.narrow) + b * p.narrow_s, p.narrow_ld, p.T,
                int64_t(ti) * kGramT, int64_t(tj) * kGramT, 0, p.narrow_n, acc,
                (FDP_LDS char*)ring);
  // rows past the sample's end count for nothing (they repeat other rows)
  const int64_t tl = p.T - int64_t(ti) * kGramT, sl = p.T - int64_t(tj) * kGramT;
  const int wm = (wave >> 1) * 64, wn = (wave & 1) * 64;
  const float* in = p.part + (b * p.per_sample + r) * int64_t(p.parts) * (kGramT * kGramT);
  float sum = 0.f;
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      f32x16 g = {};
      for (int q = 0; q < p.parts; ++q)
#pragma unroll
        for (int e = 0; e < 16; ++e)
          g[e] += in[int64_t(q) * (kGramT * kGramT) + ((i * 2 + j) * 16 + e) * NT + threadIdx.x];
      const bool col = acc_col(wn, j, lane) < sl;
#pragma unroll
      for (int e = 0; e < 16; ++e)
        sum += col && acc_row(wm, i, lane, e) < tl ? g[e] * acc[i][j][e] : 0.f;
    }
  sum = wave_sum(sum);
  if (lane == 0) red[wave] = sum;
  __syncthreads();
  if (threadIdx.x == 0)
    p.partials[blockIdx.x] = (ti == tj ? 1.f : 2.f) * ((red[0] + red[1]) + (red[2] + red[3]));
}

// ------------------------------------------------------------------ host
enum StagedPass { kStagedNorm, kStagedGram, kStagedSum };

// One pass, per type (wgrad_staged_{bf16,f16}.hip).  kStagedGram: a.group_out is
// the partial tiles' buffer.
hipError_t launch_staged_bf16(const Args& a, const StreamPlan& sp, int layout, StagedPass pass,
                              hipStream_t s);
hipError_t launch_staged_f16(const Args& a, const StreamPlan& sp, int layout, StagedPass pass,
                             hipStream_t s);

template <class DT, class G>
void launch_staged_pass(const Args& a, StagedPass pass, hipStream_t s) {
  const unsigned tiles = static_cast<unsigned>(a.tiles_m * a.tiles_n);
  if (pass == kStagedNorm)
    hipLaunchKernelGGL((staged_norm_kernel<DT, G>),
                       dim3(tiles, static_cast<unsigned>(a.B < kStagedGridY ? a.B : kStagedGridY)),
                       dim3(NT), 0, s, a);
  else
    hipLaunchKernelGGL((staged_sum_kernel<DT, G>), dim3(tiles * static_cast<unsigned>(a.groups)),
                       dim3(NT), 0, s, a);
}

template <class DT>
hipError_t launch_staged(Args a, const StreamPlan& sp, int layout, StagedPass pass,
                         hipStream_t s) {
  if (pass == kStagedGram) {
    const bool wa = a.M > a.N;
    SplitGram g{};
    g.wide = wa ? a.a : a.b;
    g.narrow = wa ? a.b : a.a;
    g.B = a.B;
    g.T = a.K;
    g.wide_n = wa ? a.M : a.N;
    g.narrow_n = wa ? a.N : a.M;
    g.wide_s = wa ? a.sab : a.sbb;
    g.wide_ld = wa ? a.lda : a.ldb;
    g.narrow_s = wa ? a.sbb : a.sab;
    g.narrow_ld = wa ? a.ldb : a.lda;
    g.nt = sp.gram_nt;
    g.per_sample = sp.gram_per_sample;
    const int64_t kt = (g.wide_n + GramGeom::BK - 1) / GramGeom::BK;
    const int64_t per = (kt + sp.split_gram - 1) / sp.split_gram;
    g.span = per * GramGeom::BK;
    g.parts = static_cast<int>((kt + per - 1) / per);
    g.part = a.group_out;
    g.partials = a.partials;
    const unsigned items = static_cast<unsigned>(g.B * g.per_sample);
    hipLaunchKernelGGL(gram_part_kernel<DT>, dim3(items * g.parts), dim3(NT), 0, s, g);
    hipLaunchKernelGGL(gram_join_kernel<DT>, dim3(items), dim3(NT), 0, s, g);
    return hipGetLastError();
  }
  (pass == kStagedNorm ? sp.norm : sp.any).set(a);
  const bool small = pass == kStagedNorm ? sp.norm_small : sp.any_small;
  const bool tn = layout == FDP_LAYOUT_TN;
  if (tn && small) launch_staged_pass<DT, SmallGeom>(a, pass, s);
  else if (tn) launch_staged_pass<DT, SumGeom>(a, pass, s);
  else if (small) launch_staged_pass<DT, SmallGeomNN>(a, pass, s);
  else launch_staged_pass<DT, SumGeomNN>(a, pass, s);
  return hipGetLastError();
}

}  // namespace wg
}  // namespace fdp
