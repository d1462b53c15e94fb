// Two-pass clipped weight gradient in full fp32 (v_mfma_f32_32x32x2_f32): the
// schedule of fp32 operands, either layout.
//
//   norm pass   ||G_b||^2 per sample, as partials [B, per_sample]:
//     direct    one workgroup per (output tile, sample) forms the tile product
//               and sums its squares (f32_norm_kernel);
//     row gram  samples of at most kRowGramMax rows (TN): ||G_b||^2 =
//               sum_{t,s} (g_t . g_s)(x_t . x_s) in fp64, one workgroup per
//               sample (f32_rowgram_kernel).  Products of two fp32 values are
//               exact in fp64, so the sum over (t, s) may cancel down to
//               1e-8 of its largest term before it is worse than fp32 squares
//               of the products; an fp32 Gram matrix would lose half the digits.
//   sum pass    out = out_scale sum_b c_b G_b + noise_scale z: ONE contraction
//               over the rows (b, k) of the whole batch, every row of a scaled
//               by its sample's factor while it is staged (f32_sum_kernel).  A
//               k-tile may hold rows of several samples, so samples shorter
//               than a k-tile cost no padding, and the contraction is split
//               anywhere: `splits` workgroups per output tile take equal row
//               ranges and write fp32 partials that wgrad_finalize_kernel adds
//               in order.
//
// Both passes run on square tiles of 128 or 64 outputs, 4 waves of (tile/2)^2.
// v_mfma_f32_32x32x2_f32 takes 64 cycles and reads one float per lane and
// operand, so the matrix pipes, not LDS or the loads, bound a tile that has
// enough workgroups beside it; the 64-wide tiles exist for layers whose 128-wide
// ones are fewer than the CUs.  Global loads are 16 bytes and need only the
// operand's own alignment (global loads of any alignment are legal on amdhsa
// targets), so odd widths and strides take the same code.
//
// Measured against the two passes this replaced (128-wide tiles and one k-tile
// ahead, k-tiles padded per sample, whole samples per split, factors in a launch
// of their own), kernel times:
//   8 x 1024,  768 -> 3072: norms 365 -> 344 us, sum 583 -> 373 us (104 TFLOP/s;
//                           the card's fp32 matrix rate on real data is about 140)
//   4 x 128,   768 ->  768: norms 14 -> 13 us, factors 13 -> 0, sum 67 -> 21 us
//   256 x 1,  1024 -> 4096: norms 419 -> 5 us, sum 406 -> 35 us
#pragma once

#include <type_traits>

#include "wgrad_stream.hpp"

namespace fdp {
namespace wg {

constexpr int kRowGramMax = 16;      // rows of a sample the row-Gram norm takes
constexpr int kF32FacMax = 1024;     // samples per workgroup whose factors it forms itself
constexpr int kF32FacThread = 16;    // partials per sample up to which one thread sums them

// Four consecutive values from p; `left` values exist (the rest read as 0).
__device__ __forceinline__ f32x4 load_quad(const float* p, int64_t left) {
  f32x4 v = {0.f, 0.f, 0.f, 0.f};
  if (left >= 4) {
    __builtin_memcpy(&v, p, 16);
  } else {
    if (left > 0) v[0] = p[0];
    if (left > 1) v[1] = p[1];
    if (left > 2) v[2] = p[2];
  }
  return v;
}

// Factors of the samples a workgroup contracts, as its gemm asks for them.
struct NoFactors {
  static constexpr bool scale = false;
  __device__ __forceinline__ float at(int) const { return 1.f; }
  __device__ __forceinline__ bool zeros() const { return false; }
};

// TM x TM outputs per workgroup; k-tiles of BK rows, double-buffered in LDS.
// An operand tile in LDS is [BK][TM] floats: rows of a multiple of 64 floats, so
// the fragment reads (one float per lane, lanes 32-63 one row on) are
// ds_read2st64_b32 at constant offsets.
//
// What the k-loop must avoid is VALU work: an fp32 MFMA of 64 cycles leaves the
// other pipes idle, but every VALU instruction delays the next MFMA by 2-4
// cycles even with three waves per SIMD (an MFMA loop with 0 / 2 / 4 / 8 VALU
// instructions per MFMA ran at 137 / 132 / 123 / 107 TFLOP/s).  So the loads go
// through scalar bases with constant per-thread offsets where rows lie at one
// stride (always for contiguous operands), and fragments are read one step ahead.
template <int TM_, int BK_>
struct F32Core {
  static constexpr int TM = TM_, BK = BK_;
  static constexpr int BM = TM, BN = TM, WM = TM / 2, WN = TM / 2;
  static constexpr int FI = TM / 64, FJ = TM / 64;
  static constexpr int TILE = BK * TM;               // floats
  static constexpr int NL = TILE / 4 / NT;           // 16-byte loads per thread and operand
  static constexpr int RQ = TM / 4;                  // quads per k-row
  static constexpr int KQ = BK / 4;                  // quads per k-contiguous row
  static constexpr int KCH = FI == 1 ? 4 : 2;        // k-pairs whose fragments are read together
  static constexpr int NC = BK / 2 / KCH;            // steps per k-tile
  static constexpr int WAVES = FI == 1 ? 3 : 2;      // resident waves per SIMD (registers)
  static_assert(NL * NT * 4 == TILE, "whole loads");
  static_assert(WM * TM <= 4 * TILE, "output staging reuses the ring");
  static_assert(NC % 2 == 0, "fragment buffers alternate");

  // One k-tile on its way from memory to LDS: this thread's quads of both
  // operands and the samples (relative to q0's) of their rows.
  struct Regs {
    f32x4 a[NL], b[NL];
    int s[NL];
  };
  // How a k-tile's rows are loaded: checked, or unchecked with (kMany) or
  // without (kOne) several samples in one k-tile.
  enum Load { kChecked, kMany, kOne };
  struct Frags {
    float a[KCH][FI], b[KCH][FJ];
  };

  // acc += sum over contraction rows [q0, q1) of c(row) a[row, m0..] b[row, n0..].
  // TN: row q is (sample q / K, k = q % K).  NN (a is [M, K], k contiguous):
  // K rounded up to BK per sample, so a k-tile never crosses samples.
  // fac.at(j): the factor of the j-th sample from q0's (asked for rows past q1
  // as well, whose quads are zeros).  Rows whose factor is zero are left out
  // entirely (their values may be infinite); fac.zeros(): there may be some.
  //
  // Two k-tiles are in flight: while k-tile kt is contracted, kt + 1 is in
  // registers or on its way there and kt + 2 is issued; kt + 1 goes to the
  // other LDS buffer (scaled) before kt's last step.
  template <int LAYOUT, class Fac>
  __device__ static inline void gemm(const Args& p, int64_t q0, int64_t q1, int64_t m0, int64_t n0,
                                     const Fac& fac, f32x16 (&acc)[FI][FJ], float* smem) {
    constexpr bool TN = LAYOUT == FDP_LAYOUT_TN;
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    const int wm = (wave >> 1) * WM, wn = (wave & 1) * WN;
    const int64_t Kp = TN ? p.K : (p.K + BK - 1) / BK * BK;
    const int64_t nk = (q1 - q0 + BK - 1) / BK;
    if (nk <= 0) return;
    const int64_t sb0 = q0 / Kp, k0 = q0 - sb0 * Kp;
    // k-tiles [0, nfull) are loaded without checks: whole tiles of rows at one
    // stride (TN: over all samples; NN: inside a sample, K a multiple of BK)
    const bool whole = p.M - m0 >= TM && p.N - n0 >= TM;
    const int64_t la = TN && p.K == 1 ? p.sab : p.lda, lb = TN && p.K == 1 ? p.sbb : p.ldb;
    const bool flat = TN ? p.K == 1 || (p.sab == p.K * la && p.sbb == p.K * lb) : p.K == Kp;
    const bool near = la < (1 << 21) && lb < (1 << 21);  // offsets in a tile below 2^31 bytes
    const int64_t nfull = !(whole && flat && near) ? 0 : TN ? (q1 - q0) / BK : nk;
    const bool one = !TN || (p.K % BK == 0 && k0 % BK == 0);  // every k-tile lies in one sample
    const char* fa = reinterpret_cast<const char*>(
        static_cast<const float*>(p.a) + (TN ? q0 * la + m0 : sb0 * p.sab + m0 * la + k0));
    const char* fb = reinterpret_cast<const char*>(
        static_cast<const float*>(p.b) + (TN ? q0 * lb : sb0 * p.sbb + k0 * lb) + n0);
    int va[NL], vb[NL];
#pragma unroll
    for (int i = 0; i < NL; ++i) {
      const int idx = t + NT * i;
      vb[i] = static_cast<int>((idx / RQ) * lb + (idx % RQ) * 4) * 4;
      va[i] = TN ? static_cast<int>((idx / RQ) * la + (idx % RQ) * 4) * 4
                 : static_cast<int>((idx / KQ) * la + (idx % KQ) * 4) * 4;
    }
    // the k-tile issued next: its index, first k and sample (valid where k-tiles
    // lie in one sample), and this thread's rows of it (k: rk, sample: rs; kept up by
    // checked and kMany loads: a step adds adv_b samples and adv_k rows, and a
    // sample more past K)
    int64_t it = 0, ak = k0;
    int as = 0;
    const int adv_b = static_cast<int>(BK / Kp);
    const int64_t adv_k = BK % Kp;
    int64_t rk[NL];
    int rs[NL];
    auto seek = [&] {
#pragma unroll
      for (int i = 0; i < NL; ++i) {
        const int64_t q = q0 + it * BK + (t + NT * i) / RQ, b = q / Kp;
        rk[i] = q - b * Kp;
        rs[i] = static_cast<int>(b - sb0);
      }
    };
    auto issue = [&](Regs& r, auto how) {
      if constexpr (how == kChecked) {
        const int64_t left = q1 - q0 - it * BK;
#pragma unroll
        for (int i = 0; i < NL; ++i) {
          const int idx = t + NT * i;
          const int row = idx / RQ, col = (idx % RQ) * 4;
          const bool in = row < left && rk[i] < p.K;
          const int64_t b = sb0 + rs[i];
          r.b[i] = load_quad(static_cast<const float*>(p.b) + b * p.sbb + rk[i] * p.ldb + n0 + col,
                             in ? p.N - n0 - col : 0);
          if constexpr (TN) {
            r.a[i] = load_quad(static_cast<const float*>(p.a) + b * p.sab + rk[i] * p.lda + m0 + col,
                               in ? p.M - m0 - col : 0);
          } else {
            const int64_t m = m0 + idx / KQ, k = ak + (idx % KQ) * 4;
            r.a[i] = load_quad(static_cast<const float*>(p.a) + (sb0 + as) * p.sab + m * p.lda + k,
                               m < p.M ? p.K - k : 0);
          }
        }
      } else {
        const auto ba = __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(fa), 0, 0x7fffffff,
                                                          kRawBufferWord3);
        const auto bb = __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(fb), 0, 0x7fffffff,
                                                          kRawBufferWord3);
#pragma unroll
        for (int i = 0; i < NL; ++i) {
          r.a[i] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(ba, va[i], 0, 0));
          r.b[i] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(bb, vb[i], 0, 0));
        }
      }
#pragma unroll
      for (int i = 0; i < NL; ++i) {
        r.s[i] = !TN || how == kOne ? as : rs[i];
        if (how != kOne) {
          rk[i] += adv_k;
          rs[i] += adv_b;
          if (rk[i] >= Kp) {
            rk[i] -= Kp;
            ++rs[i];
          }
        }
      }
      fb += BK * lb * 4;
      fa += TN ? BK * la * 4 : BK * 4;
      ++it;
      ak += BK;
      if (ak >= Kp) {
        ak -= Kp;
        ++as;
        if (!TN) {
          fa += (p.sab - Kp) * 4;
          fb += (p.sbb - Kp * lb) * 4;
        }
      }
    };
    auto put = [&](Regs& r, const float (&c)[NL], float* As, float* Bs) {
      if constexpr (Fac::scale) {
#pragma unroll
        for (int i = 0; i < NL; ++i) r.a[i] *= c[i];
        if (__builtin_expect(fac.zeros(), 0)) {
          asm volatile("");  // (a branch, not selects on every call)
#pragma unroll
          for (int i = 0; i < NL; ++i)
            if (c[i] == 0.f) r.a[i] = r.b[i] = f32x4{0.f, 0.f, 0.f, 0.f};
        }
      }
#pragma unroll
      for (int i = 0; i < NL; ++i) {
        const int idx = t + NT * i;
        if constexpr (TN) {
          *reinterpret_cast<f32x4*>(As + idx * 4) = r.a[i];
        } else {
          float* d = As + (idx % KQ) * 4 * TM + idx / KQ;
#pragma unroll
          for (int e = 0; e < 4; ++e) d[e * TM] = r.a[i][e];
        }
        *reinterpret_cast<f32x4*>(Bs + idx * 4) = r.b[i];
      }
    };
    auto factors = [&](const Regs& r, float (&c)[NL]) {
#pragma unroll
      for (int i = 0; i < NL; ++i) c[i] = fac.at(r.s[i]);
    };
    // fragments of step c of the k-tile in LDS buffer s
    const FDP_LDS float *ra[FI], *rb[FJ];
#pragma unroll
    for (int i = 0; i < FI; ++i)
      ra[i] = (const FDP_LDS float*)smem + wm + 32 * i + (lane & 31) + (lane >> 5) * TM;
#pragma unroll
    for (int j = 0; j < FJ; ++j)
      rb[j] = (const FDP_LDS float*)smem + TILE + wn + 32 * j + (lane & 31) + (lane >> 5) * TM;
    // (separate bases: two reads of one base 32 floats apart would be merged
    // into a read of two, whose short offsets cost an address addition each)
#pragma unroll
    for (int i = 0; i < FI; ++i) asm volatile("" : "+v"(ra[i]));
#pragma unroll
    for (int j = 0; j < FJ; ++j) asm volatile("" : "+v"(rb[j]));
    auto read = [&](Frags& f, int s, int c) {
#pragma unroll
      for (int e = 0; e < KCH; ++e) {
#pragma unroll
        for (int i = 0; i < FI; ++i) f.a[e][i] = ra[i][2 * s * TILE + 2 * (c * KCH + e) * TM];
#pragma unroll
        for (int j = 0; j < FJ; ++j) f.b[e][j] = rb[j][2 * s * TILE + 2 * (c * KCH + e) * TM];
      }
    };
    auto mma = [&](const Frags& f) {
#pragma unroll
      for (int e = 0; e < KCH; ++e)
#pragma unroll
        for (int i = 0; i < FI; ++i)
#pragma unroll
          for (int j = 0; j < FJ; ++j)
            acc[i][j] =
                __builtin_amdgcn_mfma_f32_32x32x2f32(f.a[e][i], f.b[e][j], acc[i][j], 0, 0, 0);
    };
    constexpr std::integral_constant<int, kChecked> checked;
    Regs r0, r1;
    Frags f0, f1;
    // the k-tile in buffer s; `next` (k-tile kt + 1) goes to the other buffer,
    // k-tile kt + 2 to `fill`
    auto step = [&](int s, Regs& next, Regs& fill, bool has1, bool has2, auto how) {
      constexpr bool all = how != kChecked;
      if (all || has2) issue(fill, how);
      float c[NL];
      factors(next, c);
#pragma unroll
      for (int ch = 0; ch < NC; ++ch) {
        Frags& cur = ch & 1 ? f1 : f0;
        Frags& nxt = ch & 1 ? f0 : f1;
        if (ch + 1 < NC) {
          read(nxt, s, ch + 1);
        } else if (all || has1) {
          put(next, c, smem + (s ^ 1) * 2 * TILE, smem + (s ^ 1) * 2 * TILE + TILE);
          dma::barrier();
          read(nxt, s ^ 1, 0);
        }
        mma(cur);
        // this step's reads (and writes) ahead of its MFMAs
        __builtin_amdgcn_sched_group_barrier(0x100, KCH * (FI + FJ), 0);
        __builtin_amdgcn_sched_group_barrier(0x008, KCH * FI * FJ, 0);
      }
    };
    // (no branch around a load in this loop, so the compiler counts the loads
    // in flight and waits for the older k-tile's only)
    auto run = [&](int64_t& kt, auto how) {
      for (; kt + 3 < nfull; kt += 2) {
        step(0, r1, r0, true, true, how);
        step(1, r0, r1, true, true, how);
      }
    };
    seek();
    issue(r0, checked);
    if (nk > 1) issue(r1, checked);
    float c0[NL];
    factors(r0, c0);
    put(r0, c0, smem, smem + TILE);
    dma::barrier();
    read(f0, 0, 0);
    int64_t kt = 0;
    if (one) {
      run(kt, std::integral_constant<int, kOne>{});
      seek();
    } else {
      run(kt, std::integral_constant<int, kMany>{});
    }
    for (; kt < nk; kt += 2) {
      step(0, r1, r0, kt + 1 < nk, kt + 2 < nk, checked);
      if (kt + 1 >= nk) break;
      step(1, r0, r1, kt + 2 < nk, kt + 3 < nk, checked);
    }
    __syncthreads();  // the caller reuses the buffers
  }
};

template <class C>
__device__ __forceinline__ void zero_acc(f32x16 (&acc)[C::FI][C::FJ]) {
#pragma unroll
  for (int i = 0; i < C::FI; ++i)
#pragma unroll
    for (int j = 0; j < C::FJ; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.f;
}

// -------------------------------------------------------------- norm pass
// Grid: (tiles, up to kGridY samples at a time).  Rows and columns past M / N
// are staged as zeros and left out of the sum.
constexpr int kGridY = 32768;
template <class C, int LAYOUT>
__global__ __launch_bounds__(NT, C::WAVES) void f32_norm_kernel(Args p) {
  __shared__ __attribute__((aligned(16))) float smem[4 * C::TILE];
  __shared__ float red[NT / kWave];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  int64_t m0, n0;
  tile_coords_g<C>(p, blockIdx.x, m0, n0);
  const int wm = (wave >> 1) * C::WM, wn = (wave & 1) * C::WN;
  const bool whole = p.M - m0 >= C::TM && p.N - n0 >= C::TM;
  const int mleft = static_cast<int>(p.M - m0 < C::TM ? p.M - m0 : C::TM);
  const int nleft = static_cast<int>(p.N - n0 < C::TM ? p.N - n0 : C::TM);
  const int64_t Kp = LAYOUT == FDP_LAYOUT_TN ? p.K : (p.K + C::BK - 1) / C::BK * C::BK;
  for (int64_t b = blockIdx.y; b < p.B; b += gridDim.y) {
    f32x16 acc[C::FI][C::FJ];
    zero_acc<C>(acc);
    C::template gemm<LAYOUT>(p, b * Kp, (b + 1) * Kp, m0, n0, NoFactors{}, acc, smem);
    float s = 0.f;
    if (whole) {
#pragma unroll
      for (int i = 0; i < C::FI; ++i)
#pragma unroll
        for (int j = 0; j < C::FJ; ++j)
#pragma unroll
          for (int r = 0; r < 16; ++r) s += acc[i][j][r] * acc[i][j][r];
    } else {  // (an infinite value times a padding zero is no part of the sum)
#pragma unroll
      for (int i = 0; i < C::FI; ++i)
#pragma unroll
        for (int j = 0; j < C::FJ; ++j) {
          const bool col = acc_col(wn, j, lane) < nleft;
#pragma unroll
          for (int r = 0; r < 16; ++r)
            s += col && acc_row(wm, i, lane, r) < mleft ? acc[i][j][r] * acc[i][j][r] : 0.f;
        }
    }
    s = wave_sum(s);
    if (lane == 0) red[wave] = s;
    __syncthreads();
    if (threadIdx.x == 0)
      p.partials[b * gridDim.x + blockIdx.x] = (red[0] + red[1]) + (red[2] + red[3]);
    __syncthreads();
  }
}

// Sum over a workgroup of one double per thread, in a fixed order; valid in thread 0.
__device__ __forceinline__ double block_sum(double v, double* red) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, kWave);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
  __syncthreads();
  return (red[0] + red[1]) + (red[2] + red[3]);
}

// Samples of one row: ||G_b||^2 = ||a_b||^2 ||b_b||^2, one workgroup per sample.
__device__ __forceinline__ double row_square(const float* p, int64_t n) {
  double s[4] = {};
  for (int64_t i = 4 * int64_t(threadIdx.x); i < n; i += 4 * NT) {
    const f32x4 v = load_quad(p + i, n - i);
#pragma unroll
    for (int j = 0; j < 4; ++j) s[j] += double(v[j]) * v[j];
  }
  return (s[0] + s[1]) + (s[2] + s[3]);
}
template <int = 0>
__global__ __launch_bounds__(NT) void f32_row_kernel(Args p) {
  __shared__ double red[2][NT / kWave];
  for (int64_t b = blockIdx.x; b < p.B; b += gridDim.x) {
    const double a = row_square(static_cast<const float*>(p.a) + b * p.sab, p.M);
    const double x = row_square(static_cast<const float*>(p.b) + b * p.sbb, p.N);
    const double n = block_sum(a, red[0]) * block_sum(x, red[1]);
    if (threadIdx.x == 0) p.partials[b] = static_cast<float>(n);
    __syncthreads();
  }
}

// Samples of 2 .. kRowGramMax rows: both [16, 16] Gram matrices of a sample by
// v_mfma_f64_16x16x4_f64 (lane l holds row l % 16, value l / 16 of 4 for both
// operands: a Gram matrix has one), the waves splitting the features.  The two
// matrices share a layout, so their elementwise product needs no index.
typedef __attribute__((__vector_size__(4 * sizeof(double)))) double f64x4;
__device__ __forceinline__ f64x4 gram_rows(const float* base, int64_t ld, int64_t T, int64_t n) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int t = lane & 15;
  const float* row = base + int64_t(t) * ld;
  f64x4 g = {0., 0., 0., 0.};
  // per wave and step: 64 features, lane group l / 16 takes quads l/16, l/16 + 4, ...
  for (int64_t f0 = 64 * wave; f0 < n; f0 += 64 * (NT / kWave)) {
    f32x4 v[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int64_t f = f0 + 16 * u + 4 * (lane >> 4);
      v[u] = t < T ? load_quad(row + f, n - f) : f32x4{0.f, 0.f, 0.f, 0.f};
    }
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const double e[4] = {v[u][0], v[u][1], v[u][2], v[u][3]};
#pragma unroll
      for (int j = 0; j < 4; ++j) g = __builtin_amdgcn_mfma_f64_16x16x4f64(e[j], e[j], g, 0, 0, 0);
    }
  }
  return g;
}
template <int = 0>
__global__ __launch_bounds__(NT) void f32_rowgram_kernel(Args p) {
  __shared__ double part[2][NT / kWave][4][kWave];
  __shared__ double red[NT / kWave];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  for (int64_t b = blockIdx.x; b < p.B; b += gridDim.x) {
    const f64x4 ga = gram_rows(static_cast<const float*>(p.a) + b * p.sab, p.lda, p.K, p.M);
    const f64x4 gb = gram_rows(static_cast<const float*>(p.b) + b * p.sbb, p.ldb, p.K, p.N);
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      part[0][wave][r][lane] = ga[r];
      part[1][wave][r][lane] = gb[r];
    }
    __syncthreads();
    // wave r takes accumulator register r
    double s[2];
#pragma unroll
    for (int o = 0; o < 2; ++o)
      s[o] = (part[o][0][wave][lane] + part[o][1][wave][lane]) +
             (part[o][2][wave][lane] + part[o][3][wave][lane]);
    const double n = block_sum(s[0] * s[1], red);
    if (threadIdx.x == 0) p.partials[b] = n > 0. ? static_cast<float>(n) : n <= 0. ? 0.f : float(n);
    __syncthreads();
  }
}

// --------------------------------------------------------------- sum pass
// Four consecutive outputs of one row (column n, `left` of them inside the row).
__device__ __forceinline__ void store_quad(const Args& p, const NoiseSrc& nz, int64_t m, int64_t n,
                                           int64_t left, float4 q) {
  float v[4] = {q.x * p.out_scale, q.y * p.out_scale, q.z * p.out_scale, q.w * p.out_scale};
  const int64_t e = m * p.N + n;
  if (nz.draw) {
    float z[4];
    if (p.N % 4 == 0) nz.block(e / 4, z);
    else nz.window(e, z);
#pragma unroll
    for (int j = 0; j < 4; ++j) v[j] += p.noise_scale * z[j];
  } else if (nz.z != nullptr) {
#pragma unroll
    for (int j = 0; j < 4; ++j)
      if (j < left) v[j] += p.noise_scale * load_as_f32(nz.z, e + j, nz.dtype);
  }
  const int64_t o = m * p.ldo + n;
  if (p.out_dtype == FDP_F32 && left >= 4) {
    __builtin_memcpy(static_cast<float*>(p.out) + o, v, 16);
  } else {
#pragma unroll
    for (int j = 0; j < 4; ++j)
      if (j < left) store_from_f32(p.out, o + j, p.out_dtype, v[j]);
  }
}

// The tile's rows of wave-row half h through LDS: out, or fp32 group partial rows.
template <class C>
__device__ inline void store_rows(const Args& p, int64_t m0, int64_t n0, int h,
                                  const f32x16 (&acc)[C::FI][C::FJ], float* lds, float* grows) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  if ((wave >> 1) == h) {
#pragma unroll
    for (int i = 0; i < C::FI; ++i)
#pragma unroll
      for (int j = 0; j < C::FJ; ++j)
#pragma unroll
        for (int r = 0; r < 16; ++r)
          lds[acc_row(0, i, lane, r) * C::TM + acc_col((wave & 1) * C::WN, j, lane)] = acc[i][j][r];
  }
  __syncthreads();
  const NoiseSrc nz = p.noise.resolved();
#pragma unroll 1
  for (int q = threadIdx.x; q < C::WM * C::RQ; q += NT) {
    const int64_t m = m0 + h * C::WM + q / C::RQ, n = n0 + (q % C::RQ) * 4;
    if (m >= p.M || n >= p.N) continue;
    const float4 v = *reinterpret_cast<const float4*>(lds + 4 * q);
    const int64_t left = p.N - n;
    if (grows == nullptr) {
      store_quad(p, nz, m, n, left, v);
    } else {
      float* d = grows + m * p.N + n;
      if (left >= 4) {
        __builtin_memcpy(d, &v, 16);
      } else {
        d[0] = v.x;
        if (left > 1) d[1] = v.y;
        if (left > 2) d[2] = v.z;
      }
    }
  }
  __syncthreads();
}

// The factors of the samples that a gemm of the sum pass contracts, in LDS.
struct SumFactors {
  static constexpr bool scale = true;
  const float* table;
  int last;
  int some_zero;  // uniform
  __device__ __forceinline__ float at(int j) const { return table[j < last ? j : last]; }
  __device__ __forceinline__ bool zeros() const { return some_zero != 0; }
};

// Grid: tiles x splits workgroups (XCD-aware numbering, split-major); split s
// takes contraction rows [s, s + 1) * rows_per_split.
// fac_parts > 0: the clip factors are formed here from partials [B, fac_parts];
// 0: read from `factors`; -1: no clipping (every factor is `clamp`).
template <class C, int LAYOUT>
__global__ __launch_bounds__(NT, C::WAVES) void f32_sum_kernel(Args p, int64_t rows_per_split) {
  __shared__ __attribute__((aligned(16))) float smem[4 * C::TILE];
  __shared__ float cfac[kF32FacMax];
  __shared__ int any_zero;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int tiles = p.tiles_m * p.tiles_n;
  const int lw = logical_wg(blockIdx.x, gridDim.x);
  const int g = lw / tiles, tile = lw % tiles;
  int64_t m0, n0;
  tile_coords_g<C>(p, tile, m0, n0);
  const int64_t Kp = LAYOUT == FDP_LAYOUT_TN ? p.K : (p.K + C::BK - 1) / C::BK * C::BK;
  const int64_t Q = p.B * Kp;
  const int64_t q0 = g * rows_per_split < Q ? g * rows_per_split : Q;
  const int64_t q1 = q0 + rows_per_split < Q ? q0 + rows_per_split : Q;
  float C_ = p.C, clamp = p.clamp;
  if (p.clip_args_dev != nullptr) {
    C_ = p.clip_args_dev[0];
    clamp = p.clip_args_dev[1];
  }
  f32x16 acc[C::FI][C::FJ];
  zero_acc<C>(acc);
  // at most kF32FacMax samples at a time
  for (int64_t qa = q0; qa < q1;) {
    const int64_t b0 = qa / Kp;
    int64_t qe = (b0 + kF32FacMax) * Kp;
    if (qe > q1) qe = q1;
    const int nb = static_cast<int>((qe - 1) / Kp - b0) + 1;
    if (threadIdx.x == 0) any_zero = 0;
    __syncthreads();
    auto put = [&](int j, float c) {
      cfac[j] = c;
      if (c == 0.f) any_zero = 1;
    };
    auto clip = [&](int j, float sq) {
      const float n = sqrtf(sq), c = clip_factor(n, C_, clamp);
      put(j, c);
      if (tile == 0) {
        if (p.norms_out) p.norms_out[b0 + j] = n;
        if (p.factors_out) p.factors_out[b0 + j] = c;
      }
    };
    const int P = p.fac_parts;
    if (P < 0) {  // (one entry serves every sample)
      if (threadIdx.x == 0) put(0, clamp);
      if (tile == 0 && p.factors_out != nullptr)
        for (int j = threadIdx.x; j < nb; j += NT) p.factors_out[b0 + j] = clamp;
    } else if (P == 0) {
      for (int j = threadIdx.x; j < nb; j += NT) put(j, p.factors[b0 + j]);
    } else if (P <= kF32FacThread) {
      for (int j = threadIdx.x; j < nb; j += NT) {
        float s = 0.f;
        for (int i = 0; i < P; ++i) s += p.partials[(b0 + j) * P + i];
        clip(j, s);
      }
    } else {
      for (int j = wave; j < nb; j += NT / kWave) {
        float s = 0.f;
        for (int i = lane; i < P; i += kWave) s += p.partials[(b0 + j) * P + i];
        s = wave_sum(s);
        if (lane == 0) clip(j, s);
      }
    }
    __syncthreads();
    const SumFactors fac{cfac, P < 0 ? 0 : nb - 1, __builtin_amdgcn_readfirstlane(any_zero)};
    C::template gemm<LAYOUT>(p, qa, qe, m0, n0, fac, acc, smem);  // (ends on a barrier)
    qa = qe;
  }
  const bool single = p.groups == 1;
  float* grows = single ? nullptr : p.group_out + int64_t(g) * p.M * p.N;
#pragma unroll
  for (int h = 0; h < 2; ++h) store_rows<C>(p, m0, n0, h, acc, smem, grows);
}

// ------------------------------------------------------------------ host
using F32Big = F32Core<128, 16>;
using F32Small = F32Core<64, 32>;

enum F32Norm { kF32NormDirect = 0, kF32NormRow = 1, kF32NormRowGram = 2 };

struct F32Plan {
  int norm;          // F32Norm
  int norm_small;    // direct norms on 64-wide tiles
  int sum_small;     // sum pass on 64-wide tiles
  int per_sample;    // norm partials per sample
  int splits;
  int64_t rows_per_split;
};

// 64-wide tiles load twice the bytes per flop: at 8 x 1024, 768 -> 3072 the sum
// pass takes 388 us in 4 splits of them, 359 us in 7 splits of 128-wide ones.
constexpr double kF32Small64 = 1.08;

// Workgroups of a pass that the fullest CU runs, side by side or in turn.
inline int64_t f32_rounds(int64_t wgs, int cus) { return (wgs + cus - 1) / cus; }

// The plan of one call.  Times are estimated in matrix cycles per CU: a k-row
// pair of a 128-wide tile takes 256 cycles on each SIMD, of a 64-wide one 64
// (a quarter of the outputs), and the passes run workgroups of one CU side by
// side, so a pass takes ceil(workgroups / CUs) workgroup times.  max_groups:
// most splits the workspace may hold; lean: 128-wide tiles only.
inline F32Plan f32_plan(int64_t B, int64_t K, int64_t M, int64_t N, int layout, int cus,
                        int64_t max_groups, bool lean) {
  F32Plan f{};
  const int64_t t128 = ((M + 127) / 128) * ((N + 127) / 128);
  const int64_t t64 = ((M + 63) / 64) * ((N + 63) / 64);
  const bool tn = layout == FDP_LAYOUT_TN;
  // norm pass
  const double n128 = double(f32_rounds(t128 * B, cus)) * double((K + 15) / 16) * 2048.;
  const double n64 = double(f32_rounds(t64 * B, cus)) * double((K + 31) / 32) * 1024. * kF32Small64;
  f.norm_small = !lean && n64 < n128 ? 1 : 0;
  f.per_sample = static_cast<int>(f.norm_small ? t64 : t128);
  const double direct = f.norm_small ? n64 : n128;
  // the row forms: one workgroup per sample; a 16-row Gram takes 64 cycles per
  // 4 features and wave
  if (tn && K == 1) {
    f.norm = kF32NormRow;
  } else if (tn && K >= 2 && K <= kRowGramMax &&
             double(f32_rounds(B, cus)) * 4. * double(M + N) < direct) {
    f.norm = kF32NormRowGram;
  }
  if (f.norm != kF32NormDirect) f.per_sample = 1;
  // sum pass: the tile and the split with the least estimated time; a split
  // adds its partials' round trip (about 2.5 KB per cycle over the device) and
  // a launch (about 5 us)
  double best = -1.;
  for (int small = 0; small < (lean ? 1 : 2); ++small) {
    const int BK = small ? F32Small::BK : F32Big::BK;
    const int64_t tiles = small ? t64 : t128;
    const int64_t rows = B * (tn ? K : (K + BK - 1) / BK * BK);
    const int64_t kt = (rows + BK - 1) / BK;
    const double cycles = small ? 1024. * kF32Small64 : 2048.;  // per k-tile
    for (int64_t s = 1; s <= 8 && s <= max_groups; ++s) {
      const int64_t per = (kt + s - 1) / s;
      if (s > 1 && per < 4) break;
      const int64_t used = per > 0 ? (kt + per - 1) / per : 1;
      if (used != s && s > 1) continue;
      double t = double(f32_rounds(tiles * s, cus)) * double(per) * cycles;
      // a CU with one or two 4-wave workgroups does not hide its load latency
      if (tiles * s < 2 * int64_t(cus)) t *= 1.3;
      if (s > 1) t += 12000. + 8. * double(s) * double(M) * double(N) / 2500.;
      if (best < 0. || t < best) {
        best = t;
        f.sum_small = small;
        f.splits = static_cast<int>(s);
        f.rows_per_split = per * BK;
      }
    }
  }
  return f;
}

// The two passes of one call (wgrad_f32.hip).  a: operands, outputs, C / clamp,
// partials, factors and group_out set; tiles, groups and factor mode are set here.
hipError_t launch_f32(Args a, const F32Plan& f, int layout, bool noclip, hipStream_t s);
// wgrad_factor_kernel and wgrad_finalize_kernel (wgrad_clip.hip)
void launch_factors(const Args& a, int per_sample, bool noclip, hipStream_t s);
void launch_finalize(const Args& a, hipStream_t s);

}  // namespace wg
}  // namespace fdp
