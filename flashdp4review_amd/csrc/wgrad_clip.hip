// Clipped per-sample weight-gradient sum on CDNA4 MFMA (gfx950).
//
//   out = out_scale * sum_b c_b * G_b + noise_scale * noise,
//   G_b = a_b^T b_b (TN) or a_b b_b (NN),  c_b = min(clamp, C/(||G_b||_F + 1e-10))
//
// Reference math: flashdp/core/linear_clip.py:94-104 (per-sample einsum, norm,
// clamp, mul, sum) and flashdp/core/bmtm_clip_loop.py:137-173 /
// flashdp/core/bmm_clip_loop.py:129-162 (operator layouts).  The reference
// materialises every G_b in HBM and scales it in a second kernel; here no
// per-sample gradient ever leaves the register file.
//
// Four schedules, chosen per call:
//   single pass (wgrad_wide.hpp, wgrad_core.hpp): 16-bit TN operands with aligned
//     rows whose output tiles fit the co-resident grid: every per-sample tile
//     product stays in the register file across one grid barrier.
//   streamed two-pass (wgrad_stream.hpp): the other 16-bit problems with aligned
//     rows (layers larger than the resident grid, the NN layout): per-sample norms
//     in Gram form or from the products, then one clipped-sum contraction per
//     output tile.
//   register-fed two-pass (wgrad_staged.hpp): the same for 16-bit operands the
//     LDS-DMA core cannot read (unaligned rows, ragged K in the NN layout, samples
//     past a 32-bit buffer record).
//   fp32 two-pass (wgrad_f32.hpp): fp32 operands of either layout.
// The two-pass schedules form the clip factors in the sum pass; calls without
// clipping and very large batches launch wgrad_factor_kernel between the passes,
// and a split sum ends in wgrad_finalize_kernel.
#include <cstdlib>

#include "wgrad_stream.hpp"
#include <tuple>

#include "wgrad_f32.hpp"
#include "wgrad_staged.hpp"
#include "wgrad_wide.hpp"

namespace fdp {
namespace wg {

// ---------------------------------------------------------------- factors
// One wavefront per sample: ||G_b|| = sqrt(sum over tiles of partials[b, :]),
// summed in a fixed lane/stride order; c_b = min(clamp, C/(||G_b|| + 1e-10)).
__global__ __launch_bounds__(NT) void wgrad_factor_kernel(const float* partials, int64_t B,
                                                           int tiles, float C, float clamp,
                                                           const float* clip_args_dev,
                                                           int noclip, float* fac_ws,
                                                           float* norms, float* factors,
                                                           int* err) {
  (void)err;  // the two-pass schedule has no bounded waits: the status word stays as it is
  if (clip_args_dev != nullptr) {
    C = clip_args_dev[0];
    clamp = clip_args_dev[1];
  }
  const int lane = threadIdx.x & 63;
  const int64_t waves = int64_t(gridDim.x) * (NT / kWave);
  for (int64_t b = int64_t(blockIdx.x) * (NT / kWave) + (threadIdx.x >> 6); b < B; b += waves) {
    float n = 0.f;
    if (!noclip) {
      float s = 0.f;
      for (int t = lane; t < tiles; t += kWave) s += partials[b * tiles + t];
      s = wave_sum(s);
      n = sqrtf(s < 0.f ? 0.f : s);  // (a Gram sum may round below zero)
    }
    if (lane == 0) {
      const float c = noclip ? clamp : clip_factor(n, C, clamp);
      fac_ws[b] = c;
      if (norms) norms[b] = n;
      if (factors) factors[b] = c;
    }
  }
}

// out = out_scale * sum_g group_out[g] + noise_scale * noise, fixed order in g.
// Memory-bound (groups fp32 reads and one write per output): a thread takes 4
// consecutive outputs, one 16-byte load per group and one Philox block.
template <class OT>
__global__ __launch_bounds__(NT) void wgrad_finalize_kernel(Args p) {
  using S = typename OT::storage;
  const int64_t MN = p.M * p.N;
  const NoiseSrc nz = p.noise.resolved();
  S* out = static_cast<S*>(p.out);
  for (int64_t e = 4 * (int64_t(blockIdx.x) * NT + threadIdx.x); e < MN;
       e += 4 * int64_t(gridDim.x) * NT) {
    const int64_t left = MN - e;
    f32x4 v = {0.f, 0.f, 0.f, 0.f};
    for (int g = 0; g < p.groups; ++g) v += load_quad(p.group_out + int64_t(g) * MN + e, left);
    v *= p.out_scale;
    if (nz.draw) {
      float z[4];
      nz.block(e / 4, z);
#pragma unroll
      for (int j = 0; j < 4; ++j) v[j] += p.noise_scale * z[j];
    } else if (nz.z != nullptr) {
#pragma unroll
      for (int j = 0; j < 4; ++j)
        if (j < left) v[j] += p.noise_scale * nz.at(e + j);
    }
    int64_t m = e / p.N, n = e - m * p.N;
    if (left >= 4 && n + 4 <= p.N) {
      const S q[4] = {OT::from_f32(v[0]), OT::from_f32(v[1]), OT::from_f32(v[2]), OT::from_f32(v[3])};
      __builtin_memcpy(out + m * p.ldo + n, q, sizeof(q));
    } else {
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        if (j >= left) break;
        out[m * p.ldo + n] = OT::from_f32(v[j]);
        if (++n == p.N) {
          n = 0;
          ++m;
        }
      }
    }
  }
}

void launch_factors(const Args& a, int per_sample, bool noclip, hipStream_t s) {
  const unsigned fb = static_cast<unsigned>((a.B + (NT / kWave) - 1) / (NT / kWave));
  hipLaunchKernelGGL(wgrad_factor_kernel, dim3(fb < 1024 ? fb : 1024), dim3(NT), 0, s, a.partials,
                     a.B, per_sample, a.C, a.clamp, a.clip_args_dev, noclip ? 1 : 0,
                     const_cast<float*>(a.factors), a.norms_out, a.factors_out, a.err);
}

void launch_finalize(const Args& a, hipStream_t s) {
  int64_t nb = (a.M * a.N + 4 * NT - 1) / (4 * NT);
  if (nb > 4096) nb = 4096;
  const dim3 grid(static_cast<unsigned>(nb));
  if (a.out_dtype == FDP_BF16)
    hipLaunchKernelGGL(wgrad_finalize_kernel<BF16>, grid, dim3(NT), 0, s, a);
  else if (a.out_dtype == FDP_F16)
    hipLaunchKernelGGL(wgrad_finalize_kernel<F16>, grid, dim3(NT), 0, s, a);
  else
    hipLaunchKernelGGL(wgrad_finalize_kernel<F32>, grid, dim3(NT), 0, s, a);
}

}  // namespace wg
}  // namespace fdp

// ====================================================================== host
using namespace fdp;
using namespace fdp::wg;

namespace {

constexpr size_t kAlign = 256;
inline size_t align_up(size_t v) { return (v + kAlign - 1) / kAlign * kAlign; }


// Workspace layout (both schedules):
//   [0, 256)            status word (int), barrier and finished-workgroup
//                       counters (uint); zero between calls, except a status set
//                       by an expired wait (the only words a reused workspace
//                       must carry over: everything after them is rewritten)
//   off_turn            per-tile counters [tiles] (uint)
//   off_partials        partials [B, max(tiles, Gram items per sample)] (fp32)
//   two-pass:  off_factors [B], off_group [groups, M, N] (fp32)
//   one-pass:  off_slots [groups, tiles, BM*BN] (fp32) per-group tile sums,
//              off_chunk [M, N] (fp32) running sum when the batch needs
//              more than one launch
struct Plan {
  int tiles_m, tiles_n, tiles;
  int spg, groups;
  StreamPlan sp;  // streamed two-pass schedule (16-bit TN operands)
  WidePlan wp;    // wide single-pass schedule (wp.wgm == 0: not used)
  size_t off_turn, off_partials, off_factors, off_group, off_slots, off_chunk;
  size_t off_wide_partials, off_wide_slots, off_wide_bias_part, off_wide_bias_sq;
  size_t total_two_pass, total_fused, total_wide, total;
};

// Smallest share of the CUs the wide kernel's products must fill by default.
constexpr double kWideMinFill = 0.7;

// Polls before a grid wait of the single-pass kernel gives up (seconds of
// waiting).  FDP_WGRAD_SPIN_LIMIT overrides it so that tests can exercise the
// expiry path with every kernel still running to completion.
unsigned spin_limit() {
  const char* e = getenv("FDP_WGRAD_SPIN_LIMIT");
  if (e != nullptr && *e != '\0') return static_cast<unsigned>(strtoul(e, nullptr, 10));
  return kSpinLimit;
}

int num_cus() { return host::device_cus(); }

// lda/ldb: the row strides the call will use (the size query assumes
// contiguous operands, lda = M and ldb = N, which the layers pass).
Plan make_plan(int64_t B, int64_t K, int64_t M, int64_t N, int cus, int flags, int64_t lda = 0,
               int64_t ldb = 0) {
  Plan pl{};
  pl.tiles_m = static_cast<int>((M + BM - 1) / BM);
  pl.tiles_n = static_cast<int>((N + BN - 1) / BN);
  pl.tiles = pl.tiles_m * pl.tiles_n;
  // Two-pass clipped sum: split the batch into groups until there are ~2
  // workgroups per CU, keeping the fp32 group partials (groups*M*N*4 bytes) at
  // or below B*M*N bytes.
  int64_t want = (2 * int64_t(cus) + pl.tiles - 1) / pl.tiles;
  const int64_t cap = B / 4 > 1 ? B / 4 : 1;
  if (want > cap) want = cap;
  if (want < 1) want = 1;
  pl.spg = static_cast<int>((B + want - 1) / want);
  pl.groups = static_cast<int>((B + pl.spg - 1) / pl.spg);
  pl.sp = stream_plan(B, K, M, N, cus);
  pl.off_turn = kWsHead;
  pl.off_partials = pl.off_turn + align_up(sizeof(unsigned) * size_t(pl.tiles));
  const size_t per_sample =
      size_t(pl.tiles > pl.sp.gram_per_sample ? pl.tiles : pl.sp.gram_per_sample);
  const size_t after_partials = pl.off_partials + align_up(sizeof(float) * size_t(B) * per_sample);
  pl.off_factors = after_partials;
  pl.off_group = pl.off_factors + align_up(sizeof(float) * size_t(B));
  int max_groups = pl.groups;
  if (pl.sp.sum.groups > max_groups) max_groups = pl.sp.sum.groups;
  if (pl.sp.any.groups > max_groups) max_groups = pl.sp.any.groups;
  pl.total_two_pass =
      pl.off_group + (max_groups > 1 ? align_up(sizeof(float) * size_t(max_groups) * M * N) : 0);
  const GroupPlan gp = group_plan(B, pl.tiles, 2 * cus);
  pl.off_slots = after_partials;
  pl.off_chunk = pl.off_slots;
  pl.total_fused = 0;
  if (gp.chunk > 0) {
    pl.off_chunk += align_up(sizeof(uint16_t) * size_t(gp.max_nwg) * BM * BN);
    pl.total_fused = pl.off_chunk + (gp.chunk < B ? sizeof(float) * size_t(M) * N : 0);
  }
  pl.total = pl.total_two_pass > pl.total_fused ? pl.total_two_pass : pl.total_fused;
  if ((flags & FDP_WGRAD_NARROW) == 0 && K > 0) {
    pl.wp = wide_plan(B, K, M, N, lda > 0 ? lda : M, ldb > 0 ? ldb : N, cus,
                      (flags & FDP_WGRAD_WIDE) ? 0.0 : kWideMinFill);
    if (flags & FDP_WGRAD_UNPAIRED) pl.wp.pair = 0;
    if (pl.wp.any()) {
      pl.off_wide_partials = kWsHead;
      pl.off_wide_slots = pl.off_wide_partials + align_up(pl.wp.partial_bytes);
      pl.off_wide_bias_part = pl.off_wide_slots + align_up(pl.wp.slot_bytes);
      pl.off_wide_bias_sq = pl.off_wide_bias_part + align_up(pl.wp.bias_part_bytes);
      pl.total_wide = pl.off_wide_bias_sq + pl.wp.bias_sq_bytes;
      if (pl.total_wide > pl.total) pl.total = pl.total_wide;
    }
  }
  return pl;
}

bool valid_dtype(int d) { return d == FDP_F32 || d == FDP_F16 || d == FDP_BF16; }

// make_plan depends only on its arguments: computed once per shape.
Plan cached_plan(int64_t B, int64_t K, int64_t M, int64_t N, int cus, int flags, int64_t lda = 0,
                 int64_t ldb = 0) {
  using Key = std::tuple<int64_t, int64_t, int64_t, int64_t, int, int, int64_t, int64_t>;
  static host::ShapeCache<Key, Plan> cache;
  return cache.get(Key{B, K, M, N, cus, flags, lda, ldb},
                   [&] { return make_plan(B, K, M, N, cus, flags, lda, ldb); });
}

// A plan's workspace with the partial tiles of the split Gram norm behind it.
size_t gram_workspace(const Plan& pl, int64_t B) {
  return align_up(pl.total) + size_t(kGramPartBytes) * size_t(B) * size_t(pl.sp.gram_per_sample) *
                                  size_t(pl.sp.split_gram);
}

// Workspace of the fp32 schedules: of the two-pass one, partials [B, per_sample],
// factors [B], group partials [splits, M, N]; of the paired one, as in Plan.
struct F32Layout {
  F32Plan plan;
  size_t off_partials, off_factors, off_group, total;
  WidePlan wp;
  size_t off_slots, off_bias_part, off_bias_sq, total_pair;
};

// Smallest share of the CUs that the paired kernel's fp32 products must fill: it
// forms every product once, the two-pass schedule twice (or once and a Gram
// form), so a half-filled grid breaks even.
constexpr double kPairF32MinFill = 0.45;

// Splits of the fp32 sum pass: their partials stay below one fp32 gradient per
// sample or 32 MB, whichever is more, and below 256 MB.  lean: the plan that
// fits a workspace of make_plan's size (old_groups group partials).
F32Layout f32_layout(int64_t B, int64_t K, int64_t M, int64_t N, int layout, int cus,
                     int old_groups, int flags, bool lean) {
  using Key = std::tuple<int64_t, int64_t, int64_t, int64_t, int, int, int, int, bool>;
  static host::ShapeCache<Key, F32Layout> cache;
  return cache.get(Key{B, K, M, N, layout, cus, old_groups, flags, lean}, [&] {
    F32Layout l{};
    const double mn = 4. * double(M) * double(N);
    int64_t most = old_groups;
    if (!lean) {
      const double bytes = double(B) * mn > 32e6 ? double(B) * mn : 32e6;
      most = static_cast<int64_t>((bytes < 256e6 ? bytes : 256e6) / mn);
      if (most < old_groups) most = old_groups;
    }
    l.plan = f32_plan(B, K, M, N, layout, cus, most, lean);
    l.off_partials = kWsHead;
    l.off_factors =
        l.off_partials + align_up(sizeof(float) * size_t(B) * size_t(l.plan.per_sample));
    l.off_group = l.off_factors + align_up(sizeof(float) * size_t(B));
    l.total = l.off_group;
    if (l.plan.splits > 1)
      l.total += align_up(sizeof(float) * size_t(l.plan.splits) * size_t(M) * size_t(N));
    if (!lean && layout == FDP_LAYOUT_TN && K > 0 && !(flags & (FDP_WGRAD_NARROW |
        FDP_WGRAD_TWO_PASS | FDP_WGRAD_UNPAIRED | FDP_WGRAD_NOCLIP))) {
      l.wp = wide_plan(B, K, M, N, M, N, cus, (flags & FDP_WGRAD_WIDE) ? 0.0 : kPairF32MinFill, true);
      if (l.wp.pair != 0) {
        l.off_slots = kWsHead + align_up(l.wp.partial_bytes);
        l.off_bias_part = l.off_slots + align_up(l.wp.slot_bytes);
        l.off_bias_sq = l.off_bias_part + align_up(l.wp.bias_part_bytes);
        l.total_pair = l.off_bias_sq + l.wp.bias_sq_bytes;
      }
    }
    return l;
  });
}

// Two-pass schedule of 16-bit operands: norms (Gram form, or from the products),
// factors, then one clipped-sum contraction per output tile.  dma: the operands
// can be read by the LDS-DMA core as they are, else they go through registers
// (gram_part: buffer of the split Gram norm, if the plan has one and it fits).
template <class DT>
hipError_t launch_two_pass(Args a, const Plan& pl, int layout, bool dma, float* gram_part,
                           bool noclip, hipStream_t s) {
  constexpr bool bf = DT::code == FDP_BF16;
  int per_sample = pl.sp.norm.tiles();
  const TilePlan& sum = dma && layout == FDP_LAYOUT_TN ? pl.sp.sum : pl.sp.any;
  hipError_t e = hipSuccess;
  if (!noclip) {
    if (dma && layout == FDP_LAYOUT_TN && pl.sp.gram) {
      GramArgs g{};
      g.a = static_cast<const uint16_t*>(a.a);
      g.b = static_cast<const uint16_t*>(a.b);
      g.B = a.B;
      g.T = a.K;
      g.M = a.M;
      g.N = a.N;
      g.sab = a.sab;
      g.lda = a.lda;
      g.sbb = a.sbb;
      g.ldb = a.ldb;
      g.nt = pl.sp.gram_nt;
      g.per_sample = pl.sp.gram_per_sample;
      g.items = a.B * g.per_sample;
      g.partials = a.partials;
      per_sample = g.per_sample;
      e = bf ? launch_gram_norm_bf16(g, s) : launch_gram_norm_f16(g, s);
    } else if (dma) {
      e = bf ? launch_prod_norm_bf16(a, pl.sp, layout, s) : launch_prod_norm_f16(a, pl.sp, layout, s);
    } else {
      StagedPass pass = kStagedNorm;
      Args n = a;
      if (layout == FDP_LAYOUT_TN && gram_part != nullptr) {
        pass = kStagedGram;
        n.group_out = gram_part;
        per_sample = pl.sp.gram_per_sample;
      }
      e = bf ? launch_staged_bf16(n, pl.sp, layout, pass, s)
             : launch_staged_f16(n, pl.sp, layout, pass, s);
    }
    if (e != hipSuccess) return e;
  }
  // The clipped-sum kernels form the factors from the partials themselves (saving
  // a launch between the passes) unless the call has no clipping or its
  // sample groups are larger than they stage.
  a.fac_parts = 0;
  if (!noclip && sum.spg <= kSumFacMax) a.fac_parts = per_sample;
  else launch_factors(a, per_sample, noclip, s);
  if (dma)
    e = bf ? launch_clipsum_bf16(a, pl.sp, layout, s) : launch_clipsum_f16(a, pl.sp, layout, s);
  else
    e = bf ? launch_staged_bf16(a, pl.sp, layout, kStagedSum, s)
           : launch_staged_f16(a, pl.sp, layout, kStagedSum, s);
  if (e != hipSuccess) return e;
  if (sum.groups > 1) {
    a.groups = sum.groups;
    launch_finalize(a, s);
  }
  return hipGetLastError();
}

}  // namespace

extern "C" int fdp_wgrad_clip_workspace_size(int64_t B, int64_t K, int64_t M, int64_t N,
                                             int dtype, int flags, size_t* bytes) {
  (void)flags;
  if (bytes == nullptr) return FDP_ERR_ARG;
  if (!valid_dtype(dtype)) return FDP_ERR_DTYPE;
  if (B < 1 || M < 1 || N < 1 || K < 0) return FDP_ERR_SHAPE;
  const int cus = num_cus();
  const Plan pl = cached_plan(B, K, M, N, cus, flags);
  *bytes = pl.total;
  if (dtype == FDP_F32) {
    for (int layout : {FDP_LAYOUT_TN, FDP_LAYOUT_NN}) {
      const F32Layout l = f32_layout(B, K, M, N, layout, cus, pl.groups, flags, false);
      if (l.total > *bytes) *bytes = l.total;
      if (l.total_pair > *bytes) *bytes = l.total_pair;
    }
  } else if (pl.sp.split_gram > 0) {
    *bytes = gram_workspace(pl, B);
  }
  return FDP_OK;
}

size_t fdp::wgrad_least_workspace(int64_t B, int64_t K, int64_t M, int64_t N, int flags) {
  return cached_plan(B, K, M, N, num_cus(), flags).total;
}

int fdp::wgrad_check_args(const void* a, const void* b, int64_t B, int64_t K, int64_t M,
                          int64_t N, int64_t lda, int64_t ldb, int layout, int dtype,
                          const void* out, int64_t ldo, int out_dtype, const float* norms,
                          int flags) {
  if (!valid_dtype(dtype) || !valid_dtype(out_dtype)) return FDP_ERR_DTYPE;
  if (layout != FDP_LAYOUT_TN && layout != FDP_LAYOUT_NN) return FDP_ERR_ARG;
  if (B < 1 || M < 1 || N < 1 || K < 0) return FDP_ERR_SHAPE;
  if (ldo < N) return FDP_ERR_SHAPE;
  if (layout == FDP_LAYOUT_TN && (lda < M || ldb < N)) return FDP_ERR_SHAPE;
  if (layout == FDP_LAYOUT_NN && (lda < K || ldb < N)) return FDP_ERR_SHAPE;
  if (M * N > (int64_t(1) << 40) || B > (int64_t(1) << 31)) return FDP_ERR_SHAPE;
  if ((K > 0 && (a == nullptr || b == nullptr)) || out == nullptr) return FDP_ERR_ARG;
  if ((flags & ~(FDP_WGRAD_NOCLIP | FDP_WGRAD_TWO_PASS | FDP_WGRAD_PLAIN_LAUNCH |
                 FDP_WGRAD_CLEAN_WORKSPACE | FDP_WGRAD_WIDE | FDP_WGRAD_NARROW |
                 FDP_WGRAD_UNPAIRED)) != 0)
    return FDP_ERR_ARG;  // (FDP_WGRAD_BIAS_OF_B only with fdp_wgrad_bias_clip)
  if ((flags & FDP_WGRAD_WIDE) && (flags & FDP_WGRAD_NARROW)) return FDP_ERR_ARG;
  if ((flags & FDP_WGRAD_NOCLIP) != 0 && norms != nullptr) return FDP_ERR_ARG;
  return FDP_OK;
}

namespace {

// fdp_wgrad_clip; with `bias`, the 16-bit TN kernels (wide, grouped and
// streamed) also form the bias of operand a (bias_op 1) or b (bias_op 2) from
// the fragments they hold, with its partials in bias_part / bias_sq
// (*bias_done = true), as does the fp32 paired one; the others leave it to the caller.
int wgrad_clip_impl(const void* a, const void* b, int64_t B, int64_t K, int64_t M, int64_t N,
                    int64_t stride_ab, int64_t lda, int64_t stride_bb, int64_t ldb, int layout,
                    int dtype, float C, float clamp, const float* clip_args_dev, float out_scale,
                    const void* noise, float noise_scale, const fdp_noise_key* noise_key,
                    void* out, int64_t ldo, int out_dtype, float* norms, float* factors,
                    int flags, void* workspace, size_t workspace_bytes, void* stream,
                    const fdp_bias_out* bias, int bias_op, float* bias_part, float* bias_sq,
                    bool* bias_done) {
  const int bad = fdp::wgrad_check_args(a, b, B, K, M, N, lda, ldb, layout, dtype, out, ldo,
                                        out_dtype, norms, flags);
  if (bad != FDP_OK) return bad;
  const bool noclip = (flags & FDP_WGRAD_NOCLIP) != 0;

  const int cus = num_cus();
  // the workspace was sized for contiguous operands: the wide plan for the
  // actual strides is taken only if it fits that size
  const Plan pl0 = cached_plan(B, K, M, N, cus, flags);
  if (workspace == nullptr || workspace_bytes < pl0.total) return FDP_ERR_WORKSPACE;
  Plan pl = cached_plan(B, K, M, N, cus, flags, lda, ldb);
  if (pl.total > workspace_bytes) pl.wp.wgm = pl.wp.pair = 0;
  if (reinterpret_cast<uintptr_t>(workspace) % 16 != 0) return FDP_ERR_ALIGN;

  char* ws = static_cast<char*>(workspace);
  Args args{};
  args.a = a;
  args.b = b;
  args.B = B;
  args.K = K;
  args.M = M;
  args.N = N;
  args.sab = stride_ab;
  args.lda = lda;
  args.sbb = stride_bb;
  args.ldb = ldb;
  args.tiles_m = pl.tiles_m;
  args.tiles_n = pl.tiles_n;
  args.spg = pl.spg;
  args.groups = pl.groups;
  args.partials = reinterpret_cast<float*>(ws + pl.off_partials);
  float* fac_ws = reinterpret_cast<float*>(ws + pl.off_factors);
  args.factors = fac_ws;
  args.group_out = pl.groups > 1 ? reinterpret_cast<float*>(ws + pl.off_group) : nullptr;
  args.out = out;
  args.ldo = ldo;
  args.out_dtype = out_dtype;
  args.out_scale = out_scale;
  args.noise = make_noise(noise, out_dtype, noise_scale != 0.f ? noise_key : nullptr, 0);
  args.noise_scale = noise_scale;
  args.units = int64_t(pl.tiles) * B;
  args.err = reinterpret_cast<int*>(ws);
  args.bar = reinterpret_cast<unsigned*>(ws) + 1;
  args.epoch = reinterpret_cast<unsigned*>(ws) + 2;
  args.poison = reinterpret_cast<unsigned*>(ws) + 3;
  args.pair_flag = reinterpret_cast<unsigned*>(ws) + kPairFlag0;
  args.spin_limit = spin_limit();
  args.tile_turn = reinterpret_cast<unsigned*>(ws + pl.off_turn);
  args.tile_acc = reinterpret_cast<float*>(ws + pl.off_slots);
  args.chunk_acc = reinterpret_cast<float*>(ws + pl.off_chunk);
  args.C = C;
  args.clamp = clamp;
  args.clip_args_dev = clip_args_dev;
  args.norms_out = norms;
  args.factors_out = factors;
  if (bias != nullptr) {
    args.bias_op = bias_op;
    args.bias_P = bias_op == 1 ? pl.tiles_n : pl.tiles_m;  // the grouped kernel's tiles
    args.bias_len = bias_op == 1 ? M : N;
    args.bias_part = bias_part;
    args.bias_sq = bias_sq;
    args.bias_out = bias->out;
    args.bias_dtype = bias->out_dtype;
    args.bias_scale = bias->out_scale;
    args.bias_noise = make_noise(bias->noise, bias->out_dtype,
                                 bias->noise_scale != 0.f ? bias->noise_key : nullptr, 0);
    args.bias_noise_scale = bias->noise_scale;
    args.bias_norms = bias->norms;
    args.bias_factors = bias->factors;
  }

  // 16-byte vector loads need 16-byte aligned rows of every sample.
  const int esz = dtype == FDP_F32 ? 4 : 2;
  const int64_t vel = 16 / esz;
  const bool vec = (reinterpret_cast<uintptr_t>(a) % 16 == 0) &&
                   (reinterpret_cast<uintptr_t>(b) % 16 == 0) && lda % vel == 0 &&
                   ldb % vel == 0 && stride_ab % vel == 0 && stride_bb % vel == 0;

  hipStream_t s = static_cast<hipStream_t>(stream);
  // The wide kernels' arguments: plan and workspace parts of the call.
  auto wide_args = [&](const WidePlan& wp, bool pair, size_t off_partials, size_t off_slots,
                       size_t off_bias_part, size_t off_bias_sq) {
    WideArgs w{};
    w.a = static_cast<const uint16_t*>(a);
    w.b = static_cast<const uint16_t*>(b);
    w.B = B;
    w.K = K;
    w.M = M;
    w.N = N;
    w.sab = stride_ab;
    w.lda = lda;
    w.sbb = stride_bb;
    w.ldb = ldb;
    w.tiles_m = pair ? wp.pair_tiles_m : wp.tiles_m;
    w.tiles_n = pair ? wp.pair_tiles_n : wp.tiles_n;
    w.tiles = pair ? wp.pair_tiles : wp.tiles;
    w.nwg = pair ? wp.pair_nwg : wp.nwg;
    w.partials = reinterpret_cast<float*>(ws + off_partials);
    w.slots = ws + off_slots;
    w.slot_blocks = pair ? wp.pair_slot_blocks : wp.slot_blocks;
    w.group_cnt = reinterpret_cast<unsigned*>(ws) + kGroupWord0;
    w.tagged = reinterpret_cast<uint64_t*>(ws + off_partials);
    w.out = out;
    w.ldo = ldo;
    w.out_dtype = out_dtype;
    w.out_scale = out_scale;
    w.noise = args.noise;
    w.noise_scale = noise_scale;
    w.bar = args.bar;
    w.epoch = args.epoch;
    w.poison = args.poison;
    w.err = args.err;
    w.spin_limit = args.spin_limit;
    w.C = C;
    w.clamp = clamp;
    w.clip_args_dev = clip_args_dev;
    w.norms_out = norms;
    w.factors_out = factors;
    if (bias != nullptr) {
      w.bias_op = bias_op;
      w.bias_part = reinterpret_cast<float*>(ws + off_bias_part);
      w.bias_sq = reinterpret_cast<float*>(ws + off_bias_sq);
      w.bias_tagged = reinterpret_cast<uint64_t*>(ws + off_bias_part);
      w.bias_sq_tagged = reinterpret_cast<uint64_t*>(ws + off_bias_sq);
      w.bias_out = bias->out;
      w.bias_dtype = bias->out_dtype;
      w.bias_scale = bias->out_scale;
      w.bias_noise = make_noise(bias->noise, bias->out_dtype,
                                bias->noise_scale != 0.f ? bias->noise_key : nullptr, 0);
      w.bias_noise_scale = bias->noise_scale;
      w.bias_norms = bias->norms;
      w.bias_factors = bias->factors;
    }
    {
      const int oes = out_dtype == FDP_F32 ? 4 : 2;
      w.vec_out = (reinterpret_cast<uintptr_t>(out) % (4 * oes) == 0 && ldo % 4 == 0) ? 1 : 0;
    }
    return w;
  };
  auto clear_head = [&] {
    if ((flags & FDP_WGRAD_CLEAN_WORKSPACE) != 0) return;
    const int64_t words = int64_t(kWsHead / sizeof(unsigned));
    hipLaunchKernelGGL(clear_words_kernel<0>, dim3(static_cast<unsigned>((words + NT - 1) / NT)),
                       dim3(NT), 0, s, reinterpret_cast<unsigned*>(ws), words);
  };
  // Wide single pass: 16-bit TN inputs, aligned rows, two samples' products
  // per CU (paired) or one.
  const bool pair = pl.wp.pair != 0 && pair_records_fit(K, lda, stride_ab) &&
                    pair_records_fit(K, ldb, stride_bb);
  if (!noclip && (flags & FDP_WGRAD_TWO_PASS) == 0 && layout == FDP_LAYOUT_TN && vec && K > 0 &&
      dtype != FDP_F32 && (pair || pl.wp.wgm != 0)) {
    const WideArgs w = wide_args(pl.wp, pair, pl.off_wide_partials, pl.off_wide_slots,
                                 pl.off_wide_bias_part, pl.off_wide_bias_sq);
    const bool plain = (flags & FDP_WGRAD_PLAIN_LAUNCH) != 0;
    clear_head();
    const int wgm = pair ? 1 : pl.wp.wgm;
    const hipError_t e = dtype == FDP_BF16 ? launch_wide_bf16(w, wgm, plain, s)
                                           : launch_wide_f16(w, wgm, plain, s);
    if (e == hipSuccess) {
      if (bias_done != nullptr) *bias_done = bias != nullptr;
      return FDP_OK;
    }
    if (e != hipErrorNotSupported && e != hipErrorCooperativeLaunchTooLarge) {
      (void)hipGetLastError();
      return FDP_ERR_HIP;
    }
    (void)hipGetLastError();
  }
  // Single pass: 16-bit inputs, TN layout, aligned rows, a clip to compute, K > 0.
  if (!noclip && (flags & FDP_WGRAD_TWO_PASS) == 0 && layout == FDP_LAYOUT_TN && vec && K > 0 &&
      dtype != FDP_F32 && pl.total_fused > 0) {
    const bool plain = (flags & FDP_WGRAD_PLAIN_LAUNCH) != 0;
    const bool clean = (flags & FDP_WGRAD_CLEAN_WORKSPACE) != 0;
    hipError_t e;
    if (bias != nullptr)
      e = dtype == FDP_BF16 ? launch_grouped_bias_bf16(args, cus, plain, clean, s)
                            : launch_grouped_bias_f16(args, cus, plain, clean, s);
    else
      e = dtype == FDP_BF16 ? launch_grouped_bf16(args, cus, plain, clean, s)
                            : launch_grouped_f16(args, cus, plain, clean, s);
    if (e == hipSuccess) {
      if (bias_done != nullptr) *bias_done = bias != nullptr;
      return FDP_OK;
    }
    if (e != hipErrorNotSupported && e != hipErrorCooperativeLaunchTooLarge) {
      (void)hipGetLastError();
      return FDP_ERR_HIP;
    }
    (void)hipGetLastError();
  }

  hipError_t e;
  if (dtype != FDP_F32) {
    // The LDS-DMA kernels read 16-byte aligned rows through 32-bit buffer
    // records (larger samples are addressed with 64 bits), and k-contiguous
    // rows (NN) in whole k-tiles only.
    const bool tn = layout == FDP_LAYOUT_TN;
    const bool dma = vec && K > 0 && fits_record(tn ? K : M, lda) && fits_record(K, ldb) &&
                     (tn || K % SumGeomNN::BK == 0);
    if (!(tn && dma)) args.bias_op = 0;  // the caller forms the bias
    args.group_out = reinterpret_cast<float*>(ws + pl.off_group);
    // the split Gram norm's partial tiles follow the rest of the workspace; in a
    // smaller one the norms come from the products
    float* gram_part = nullptr;
    if (pl.sp.split_gram > 0 && gram_workspace(pl, B) <= workspace_bytes)
      gram_part = reinterpret_cast<float*>(ws + align_up(pl.total));
    e = dtype == FDP_BF16 ? launch_two_pass<BF16>(args, pl, layout, dma, gram_part, noclip, s)
                          : launch_two_pass<F16>(args, pl, layout, dma, gram_part, noclip, s);
    if (e != hipSuccess) return FDP_ERR_HIP;
    if (bias_done != nullptr) *bias_done = bias != nullptr && args.bias_op != 0;
    return FDP_OK;
  }
  // fp32: the plan that the workspace query sized, or, in a smaller workspace,
  // the one that fits the least accepted size (the caller forms the bias)
  const F32Layout fl = f32_layout(B, K, M, N, layout, cus, pl0.groups, flags, false);
  // Paired single pass: aligned rows, every product once.
  if (!noclip && fl.wp.pair != 0 && fl.total_pair <= workspace_bytes && vec &&
      lda < (int64_t(1) << 29) && ldb < (int64_t(1) << 29) && stride_ab < (int64_t(1) << 29) &&
      stride_bb < (int64_t(1) << 29) && pair_records_fit(K, 2 * lda, 2 * stride_ab) &&
      pair_records_fit(K, 2 * ldb, 2 * stride_bb)) {
    const WideArgs w = wide_args(fl.wp, true, kWsHead, fl.off_slots, fl.off_bias_part, fl.off_bias_sq);
    clear_head();
    e = launch_pair_f32(w, (flags & FDP_WGRAD_PLAIN_LAUNCH) != 0, s);
    if (e == hipSuccess) {
      if (bias_done != nullptr) *bias_done = bias != nullptr;
      return FDP_OK;
    }
    (void)hipGetLastError();
    if (e != hipErrorNotSupported && e != hipErrorCooperativeLaunchTooLarge) return FDP_ERR_HIP;
  }
  const F32Layout f = fl.total <= workspace_bytes
                          ? fl
                          : f32_layout(B, K, M, N, layout, cus, pl0.groups, flags, true);
  args.bias_op = 0;
  args.partials = reinterpret_cast<float*>(ws + f.off_partials);
  args.factors = reinterpret_cast<float*>(ws + f.off_factors);
  args.group_out = reinterpret_cast<float*>(ws + f.off_group);
  e = launch_f32(args, f.plan, layout, noclip, s);
  return e == hipSuccess ? FDP_OK : FDP_ERR_HIP;
}

}  // namespace

extern "C" int fdp_wgrad_clip(const void* a, const void* b, int64_t B, int64_t K, int64_t M,
                              int64_t N, int64_t stride_ab, int64_t lda, int64_t stride_bb,
                              int64_t ldb, int layout, int dtype, float C, float clamp,
                              const float* clip_args_dev, float out_scale, const void* noise,
                              float noise_scale, const fdp_noise_key* noise_key, void* out,
                              int64_t ldo, int out_dtype,
                              float* norms, float* factors, int flags, void* workspace,
                              size_t workspace_bytes, void* stream) {
  return wgrad_clip_impl(a, b, B, K, M, N, stride_ab, lda, stride_bb, ldb, layout, dtype, C, clamp,
                         clip_args_dev, out_scale, noise, noise_scale, noise_key, out, ldo,
                         out_dtype, norms, factors, flags, workspace, workspace_bytes, stream,
                         nullptr, 0, nullptr, nullptr, nullptr);
}

namespace {

// Workspace of fdp_wgrad_bias_clip (every part 256-aligned): the weight
// gradient's workspace, the column-sum kernel's (the bias when a register-fed
// schedule runs), then the bias partials of the grouped and streamed kernels
// (bias_part [B, P, len], bias_sq [B, tiles], sized for both tile grids).
struct BiasLayout {
  size_t wspan, col_off, part_off, sq_off, total;
};
// least: with the smallest weight workspace that is accepted.
int bias_layout(int64_t B, int64_t K, int64_t M, int64_t N, int dtype, int wflags, int bias_op,
                bool least, BiasLayout* l) {
  size_t w = 0, c = 0;
  int st = fdp_wgrad_clip_workspace_size(B, K, M, N, dtype, wflags, &w);
  if (st != FDP_OK) return st;
  if (least) w = fdp::wgrad_least_workspace(B, K, M, N, wflags);
  st = fdp_colsum_clip_workspace_size(B, K, bias_op == 1 ? M : N, dtype, &c);
  if (st != FDP_OK) return st;
  const int gm = static_cast<int>((M + BM - 1) / BM), gn = static_cast<int>((N + BN - 1) / BN);
  const StreamPlan sp = stream_plan(B, K, M, N, num_cus());
  const int64_t P_group = bias_op == 1 ? gn : gm, P_stream = stream_bias_P(sp, bias_op);
  const int64_t tiles_group = int64_t(gm) * gn, tiles_stream = sp.sum.tiles();
  const int64_t P = P_group > P_stream ? P_group : P_stream;
  const int64_t tiles = tiles_group > tiles_stream ? tiles_group : tiles_stream;
  const int64_t len = bias_op == 1 ? M : N;
  l->wspan = align_up(w);
  l->col_off = l->wspan;
  l->part_off = l->col_off + align_up(c);
  l->sq_off = l->part_off + align_up(sizeof(float) * size_t(len) * size_t(B) * size_t(P));
  l->total = l->sq_off + sizeof(float) * size_t(B) * size_t(tiles);
  return FDP_OK;
}

}  // namespace

extern "C" int fdp_wgrad_bias_clip_workspace_size(int64_t B, int64_t K, int64_t M, int64_t N,
                                                  int dtype, int flags, size_t* bytes) {
  if (bytes == nullptr) return FDP_ERR_ARG;
  if (!valid_dtype(dtype)) return FDP_ERR_DTYPE;
  if (B < 1 || M < 1 || N < 1 || K < 0) return FDP_ERR_SHAPE;
  const int bias_op = (flags & FDP_WGRAD_BIAS_OF_B) ? 2 : 1;
  BiasLayout l{};
  const int st = bias_layout(B, K, M, N, dtype, flags & ~FDP_WGRAD_BIAS_OF_B, bias_op, false, &l);
  if (st != FDP_OK) return st;
  *bytes = l.total;
  return FDP_OK;
}

extern "C" int fdp_wgrad_bias_clip(const void* a, const void* b, int64_t B, int64_t K, int64_t M,
                                   int64_t N, int64_t stride_ab, int64_t lda, int64_t stride_bb,
                                   int64_t ldb, int layout, int dtype, float C, float clamp,
                                   const float* clip_args_dev, float out_scale, const void* noise,
                                   float noise_scale, const fdp_noise_key* noise_key, void* out,
                                   int64_t ldo, int out_dtype, float* norms, float* factors,
                                   int flags, const fdp_bias_out* bias, void* workspace,
                                   size_t workspace_bytes, void* stream) {
  const int bias_op = (flags & FDP_WGRAD_BIAS_OF_B) ? 2 : 1;
  flags &= ~FDP_WGRAD_BIAS_OF_B;
  const int bad = fdp::wgrad_check_args(a, b, B, K, M, N, lda, ldb, layout, dtype, out, ldo,
                                        out_dtype, norms, flags);
  if (bad != FDP_OK) return bad;
  if (bias == nullptr || bias->out == nullptr) return FDP_ERR_ARG;
  if (!valid_dtype(bias->out_dtype)) return FDP_ERR_DTYPE;
  // the bias operand is [B, K, len] over K, contiguous (the column-sum kernel
  // reads it that way when a register-fed schedule runs); the clip is not
  // optional
  if (layout != FDP_LAYOUT_TN || (flags & FDP_WGRAD_NOCLIP) != 0) return FDP_ERR_ARG;
  if (bias_op == 1 && (lda != M || stride_ab != K * M)) return FDP_ERR_SHAPE;
  if (bias_op == 2 && (ldb != N || stride_bb != K * N)) return FDP_ERR_SHAPE;
  BiasLayout l{};
  int st = bias_layout(B, K, M, N, dtype, flags, bias_op, false, &l);
  if (st == FDP_OK && workspace_bytes < l.total)
    st = bias_layout(B, K, M, N, dtype, flags, bias_op, true, &l);
  if (st != FDP_OK) return st;
  if (workspace == nullptr || workspace_bytes < l.total) return FDP_ERR_WORKSPACE;
  char* ws = static_cast<char*>(workspace);
  bool done = false;
  st = wgrad_clip_impl(a, b, B, K, M, N, stride_ab, lda, stride_bb, ldb, layout, dtype, C, clamp,
                       clip_args_dev, out_scale, noise, noise_scale, noise_key, out, ldo,
                       out_dtype, norms, factors, flags, workspace, l.wspan, stream, bias, bias_op,
                       reinterpret_cast<float*>(ws + l.part_off),
                       reinterpret_cast<float*>(ws + l.sq_off), &done);
  if (st != FDP_OK || done) return st;
  return fdp_colsum_clip(bias_op == 1 ? a : b, nullptr, B, K, bias_op == 1 ? M : N, dtype,
                         FDP_NORM_FROB, C, clamp, clip_args_dev, bias->out_scale, bias->noise,
                         bias->noise_scale, bias->noise_key, bias->out, bias->out_dtype,
                         bias->norms, bias->factors, ws + l.col_off, l.part_off - l.col_off,
                         stream);
}
