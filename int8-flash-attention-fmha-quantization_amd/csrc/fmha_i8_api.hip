// C ABI of libfmha_i8.so: argument checking, scale folding and the kernel launch.  Stands where the reference has
// FMHAInferI8 / LaunchFMHAInfer_TCU (src/fmha_i8.cu:31-173): the if/else ladder over (head_dim, seq_len) template
// instantiations becomes a run-time seq_len and a two-way switch on head_dim.
#include <hip/hip_runtime.h>
#include <math.h>
#include <stdint.h>
#include <stdio.h>

#include "../../include/fmha_i8.h"
#include "fmha_i8_kernel.hip"
#ifndef FMHA_NO_SPLIT_KERNEL
#include "fmha_i8_split_kernel.hip"
#include "fmha_i8_pair_kernel.hip"
#include "fmha_i8_few_kernel.hip"
#endif

namespace {

using fmha_i8_gfx950::KernelArgs;

// One shape for both entry points: self-attention is the case seq_len_q == seq_len_kv.
FMHACrossAttnDescriptor as_cross(const AttnDataDescriptor& a) {
  return FMHACrossAttnDescriptor{a.batch_num, a.seq_len, a.seq_len, a.head_num, a.head_dim};
}

// inc/fmha_i8.cuh:71-72: row_scale = 1/sqrt(d), scale_qk_out = q_amax*k_amax/127^2; folded with log2(e) because the
// kernel's exponentials are base 2.
float score_scale_log2(const FMHAParamI8& p, int head_dim) {
  constexpr float kLog2e = 1.4426950408889634f;
  const float row_scale = 1.0f / sqrtf((float)head_dim);
  const float scale_qk_out = p.q_amax * p.k_amax / (127.f * 127.f);
  return row_scale * scale_qk_out * kLog2e;
}
float output_scale(const FMHAParamI8& p) { return p.v_amax / (p.o_amax * 128.f); }  // inc/fmha_i8.cuh:318

int check_args(const FMHAParamI8& p, const FMHACrossAttnDescriptor& a, const void* q, const void* k, const void* v,
               const void* mask, const void* o) {
  if (!q || !k || !v || !mask || !o) return FMHA_I8_ERR_NULL_POINTER;
  if (a.head_dim != 64 && a.head_dim != 128) return FMHA_I8_ERR_HEAD_DIM;
  if (a.seq_len_kv <= 0 || a.seq_len_kv > 65536 || a.seq_len_q <= 0 || a.seq_len_q > 65536) return FMHA_I8_ERR_SEQ_LEN;
  if (a.batch_num <= 0 || a.head_num <= 0) return FMHA_I8_ERR_BATCH_HEAD;
  const long long wgs = (long long)a.batch_num * a.head_num * ((a.seq_len_q + fmha_i8_gfx950::kBlockQ - 1) / fmha_i8_gfx950::kBlockQ);
  if (wgs > 0x7fffffffLL) return FMHA_I8_ERR_BATCH_HEAD;
  const uintptr_t bits = (uintptr_t)q | (uintptr_t)k | (uintptr_t)v | (uintptr_t)o;
  if (bits & 15u) return FMHA_I8_ERR_ALIGNMENT;
  if (!isfinite(p.q_amax) || !isfinite(p.k_amax) || !isfinite(p.v_amax) || !isfinite(p.o_amax) || !(p.o_amax > 0.f))
    return FMHA_I8_ERR_SCALE;
  // amax values are maxima of absolute values.  The kernel takes row maxima on the integer scores, which is only the
  // maximum of the scaled scores while the scale is not negative.
  if (p.q_amax * p.k_amax < 0.f) return FMHA_I8_ERR_SCALE;
  // Finite amax values can still overflow in the scales the kernel works with (1e20 * 1e20, 1e30 / 1e-30); an
  // infinite or NaN scale would turn every score or every output into NaN behind a status of "ok".
  if (!isfinite(score_scale_log2(p, a.head_dim)) || !isfinite(output_scale(p))) return FMHA_I8_ERR_SCALE;
  return FMHA_I8_OK;
}

struct Variant {
  bool bias, fast, full_range_p;
};
// Every launch hands back the status of THAT launch (the return value of hipLaunchKernel), never the thread's last
// error: an unrelated earlier failure of the caller must neither be reported as this call's nor be cleared by it.
template <int D, int BK, bool RAGGED, bool FULLP>
hipError_t launch_variant4(Variant var, dim3 grid, dim3 block, hipStream_t stream, const fmha_i8_gfx950::KernelArgs& args) {
  using namespace fmha_i8_gfx950;
  KernelArgs by_value = args;
  void* kernel_args[] = {&by_value};
#ifdef FMHA_FEW_INSTANTIATIONS
  // Test builds that are compiled many times over (tests/Makefile, target `variants`) carry only the instantiations
  // the five benchmark configurations use: blocks of 128 keys, whole blocks, 128-step P, the one-fma merge.
  if constexpr (BK != kBlockK || RAGGED || FULLP) return hipErrorInvalidDeviceFunction;
  else {
    if (!var.fast) return hipErrorInvalidDeviceFunction;
    return var.bias ? hipLaunchKernel(reinterpret_cast<const void*>(&fmha_i8_fwd_kernel<D, BK, true, true, RAGGED, FULLP>), grid, block, kernel_args, 0, stream)
                    : hipLaunchKernel(reinterpret_cast<const void*>(&fmha_i8_fwd_kernel<D, BK, false, true, RAGGED, FULLP>), grid, block, kernel_args, 0, stream);
  }
#else
#define FMHA_LAUNCH(BB, FF) \
  hipLaunchKernel(reinterpret_cast<const void*>(&fmha_i8_fwd_kernel<D, BK, BB, FF, RAGGED, FULLP>), grid, block, kernel_args, 0, stream)
  if (var.bias) return var.fast ? FMHA_LAUNCH(true, true) : FMHA_LAUNCH(true, false);
  return var.fast ? FMHA_LAUNCH(false, true) : FMHA_LAUNCH(false, false);
#undef FMHA_LAUNCH
#endif
}
template <int D, int BK, bool RAGGED>
hipError_t launch_variant3(Variant var, dim3 grid, dim3 block, hipStream_t stream, const fmha_i8_gfx950::KernelArgs& args) {
  if (var.full_range_p) return launch_variant4<D, BK, RAGGED, true>(var, grid, block, stream, args);
  return launch_variant4<D, BK, RAGGED, false>(var, grid, block, stream, args);
}
template <int D, int BK>
hipError_t launch_variant(Variant var, dim3 grid, dim3 block, hipStream_t stream, const fmha_i8_gfx950::KernelArgs& args) {
  if (args.seq_kv % BK != 0) return launch_variant3<D, BK, true>(var, grid, block, stream, args);
  return launch_variant3<D, BK, false>(var, grid, block, stream, args);
}

// The kernel of 256-row workgroups: args.total_wgs of them.
hipError_t launch_wide(int head_dim, int block_keys, Variant var, hipStream_t stream, const fmha_i8_gfx950::KernelArgs& args) {
  using fmha_i8_gfx950::kBlockK, fmha_i8_gfx950::kBlockKSmall;
  const dim3 grid((unsigned)args.total_wgs), block(fmha_i8_gfx950::kThreads);
  if (head_dim == 128)
    return block_keys == kBlockK ? launch_variant<128, kBlockK>(var, grid, block, stream, args) : launch_variant<128, kBlockKSmall>(var, grid, block, stream, args);
  return block_keys == kBlockK ? launch_variant<64, kBlockK>(var, grid, block, stream, args) : launch_variant<64, kBlockKSmall>(var, grid, block, stream, args);
}

#ifndef FMHA_NO_SPLIT_KERNEL
// R, and row_groups below: groups of 32 query rows per workgroup, or kFew for fmha_i8_few_kernel.
constexpr int kFew = 16;
template <int D, int BK, int R>
const void* split_kernel(Variant var) {
  using namespace fmha_i8_gfx950;
#define FMHA_VARIANT(KERNEL, ...)                                                                                    \
  (var.full_range_p ? (var.bias ? (var.fast ? FMHA_KERNEL(KERNEL, true, true, true) : FMHA_KERNEL(KERNEL, true, false, true))        \
                                : (var.fast ? FMHA_KERNEL(KERNEL, false, true, true) : FMHA_KERNEL(KERNEL, false, false, true)))     \
                    : (var.bias ? (var.fast ? FMHA_KERNEL(KERNEL, true, true, false) : FMHA_KERNEL(KERNEL, true, false, false))      \
                                : (var.fast ? FMHA_KERNEL(KERNEL, false, true, false) : FMHA_KERNEL(KERNEL, false, false, false))))
  if constexpr (R == 4) {
#define FMHA_KERNEL(KERNEL, BB, FF, PP) reinterpret_cast<const void*>(&KERNEL<D, BK, BB, FF, PP>)
    return FMHA_VARIANT(fmha_i8_pair_kernel);
#undef FMHA_KERNEL
  } else if constexpr (R == kFew) {
    if constexpr (D == 128 && BK == kBlockK) return nullptr;  // (shared-out key blocks alone)
    else {
#define FMHA_KERNEL(KERNEL, BB, FF, PP) reinterpret_cast<const void*>(&KERNEL<D, BK, BB, FF, PP, false>)
      return FMHA_VARIANT(fmha_i8_few_kernel);
#undef FMHA_KERNEL
    }
  } else {
#define FMHA_KERNEL(KERNEL, BB, FF, PP) reinterpret_cast<const void*>(&KERNEL<D, BK, BB, FF, PP, R>)
    return FMHA_VARIANT(fmha_i8_split_kernel);
#undef FMHA_KERNEL
  }
#undef FMHA_VARIANT
}
// What a call of few query rows needs to share its key blocks out over workgroups (see fmha_i8_merge_kernel).
struct PartPlan {
  int rounds_per_part = 0;  // 0: it does not
  size_t ml_bytes = 0, bytes = 0;
};
template <int D, int BK>
const void* part_kernel(Variant var, int rows) {
  using namespace fmha_i8_gfx950;
  // (what becomes of the accumulators is up to the merge: FASTACC makes no difference here)
#define FMHA_PART(BB, FF, PP) \
  (rows <= kFewRows ? reinterpret_cast<const void*>(&fmha_i8_few_kernel<D, BK, BB, FF, PP, true>) : reinterpret_cast<const void*>(&fmha_i8_split_kernel<D, BK, BB, FF, PP, 1, true>))
  if (var.full_range_p) return var.bias ? FMHA_PART(true, true, true) : FMHA_PART(false, true, true);
  return var.bias ? FMHA_PART(true, true, false) : FMHA_PART(false, true, false);
#undef FMHA_PART
}
template <int D, int BK>
hipError_t launch_parts(const PartPlan& plan, Variant var, hipStream_t stream, const fmha_i8_gfx950::KernelArgs& of_call, void* workspace) {
  using namespace fmha_i8_gfx950;
  SplitKernelArgs args{of_call};
  const int heads = args.total_wgs / args.q_blocks, n_blocks = (args.seq_kv + BK - 1) / BK;
  const int rounds = (n_blocks + kSplitKeys - 1) / kSplitKeys;
  args.rounds_per_part = plan.rounds_per_part;
  args.q_blocks = (rounds + plan.rounds_per_part - 1) / plan.rounds_per_part;  // parts per head in the place of query blocks
  args.total_wgs = heads * args.q_blocks;
  args.q_blocks_divisor = make_divisor(args.q_blocks);
  args.head_num_divisor = make_divisor(args.head_num);
  args.part_ml = static_cast<v2f*>(workspace);
  args.part_o = reinterpret_cast<int*>(static_cast<char*>(workspace) + plan.ml_bytes);
  void* kernel_args[] = {&args};
  const hipError_t err = hipLaunchKernel(part_kernel<D, BK>(var, args.seq_q), dim3((unsigned)args.total_wgs), dim3(256), kernel_args, 0, stream);
  if (err != hipSuccess) return err;
  int row_lanes = D / 2;
  while (64 / row_lanes < args.seq_q) row_lanes /= 2;
  MergeArgs merge{args.part_ml, args.part_o, args.o, n_blocks, args.seq_q, D, row_lanes, args.floor2, args.out_scale, var.fast, var.full_range_p};
  void* merge_args[] = {&merge};
  return hipLaunchKernel(n_blocks <= 16 ? reinterpret_cast<const void*>(&fmha_i8_merge_kernel<16>) : reinterpret_cast<const void*>(&fmha_i8_merge_kernel<32>), dim3((unsigned)(D / (2 * row_lanes)), (unsigned)heads), dim3(64), merge_args, 0, stream);
}
// A part of a call: rows first_row .. end_row - 1 of `heads` heads from first_head on, by one kernel.
struct Piece {
  int row_groups, first_head, heads, first_row, end_row;
};
template <int D, int BK>
hipError_t launch_split(const Piece& piece, Variant var, hipStream_t stream, const fmha_i8_gfx950::KernelArgs& of_call) {
  using namespace fmha_i8_gfx950;
  SplitKernelArgs args{of_call};
  const int row_groups = piece.row_groups, rows = row_groups == kFew ? kFewRows : 32 * row_groups;
  args.q_blocks = (piece.end_row - piece.first_row + rows - 1) / rows;
  args.total_wgs = piece.heads * args.q_blocks;
  args.first_head = piece.first_head;
  args.first_row = piece.first_row;
  args.q_blocks_divisor = make_divisor(args.q_blocks);
  args.head_num_divisor = make_divisor(args.head_num);
  void* kernel_args[] = {&args};
  const void* kernel = row_groups == kFew ? split_kernel<D, BK, kFew>(var) : row_groups == 1 ? split_kernel<D, BK, 1>(var) : row_groups == 2 ? split_kernel<D, BK, 2>(var) : split_kernel<D, BK, 4>(var);
  return hipLaunchKernel(kernel, dim3((unsigned)args.total_wgs), dim3(row_groups == 1 || row_groups == kFew ? 256 : 512), kernel_args, 0, stream);
}
// What a workgroup of each kernel costs: (start + step * rounds), a round being one key block for the first two and four for the
// split kernel, and `again` for each further one on the same CU, whose prologue nothing covers (the first one's is part of the launch).
// Microseconds * 100 beyond the launch (2.8 us), [head_dim 64, 128][blocks of 64, 128 keys], measured on one MI355X with one
// workgroup on half of the CUs (tests/variant_timing.py --kernel-costs), `again` with two to eight on every CU (--shapes); measurements differ
// by 4 %.  With starts measured before Q went through LDS and no `again`, calls of 130 to 256 keys at d64 took the 256-row kernel
// that smaller workgroups serve faster (B5 H8 S256 6.40 -> 5.41 us, B8 H12 S144 6.62 -> 5.01).
// With all CUs at work the first two take up to 36 and 14 % longer per block (the shader clock drops).
constexpr int kComputeUnits = 256, kLaunch = 280;
struct KernelCost {
  int row_groups, keys_per_round;
  struct { int start, step, again; } cost[2][2];
};
constexpr KernelCost kKernelCosts[] = {{0, 1, {{{70, 80, 120}, {105, 129, 120}}, {{160, 99, 220}, {235, 162, 220}}}},
                                       {4, 1, {{{107, 62, 130}, {142, 96, 140}}, {{171, 82, 190}, {252, 117, 200}}}},
                                       {2, 4, {{{0, 186, 150}, {20, 300, 150}}, {{20, 200, 190}, {61, 332, 260}}}},
                                       {1, 4, {{{0, 136, 20}, {6, 211, 150}}, {{25, 153, 180}, {36, 247, 180}}}}};
// At most 32 query rows: every workgroup, one to a head or to a part of one, fetches keys of its own, and calls of more heads than there
// are compute units run into the memory.  So these have prices of their own, the same way for a head by one workgroup as for key blocks
// shared out ([at most sixteen rows, more][head_dim][block]): the workgroups that run at a time take max(start + step * rounds + again,
// their keys at 67 KB in a hundredth of a microsecond), `again` from the second time on; `together` is how many a CU holds, of which the
// second adds half of the first one's time; `slowed`: percent of the memory's time on top (d128, S4096: H16 21.2 us, H64 22.9, H96 23.2).  Fitted to calls of 1 to 1024 heads timed on both routes; see part_plan_of.
struct HeadCost {
  int start, step, again, together, slowed;
};
constexpr HeadCost kHeadCosts[2][2][2] = {{{{-60, 103, 140, 2}, {-25, 145, 150, 1}}, {{-20, 131, 150, 1}, {10, 230, 200, 1, 12}}},
                                          {{{-15, 135, 150, 2}, {0, 213, 240, 1}}, {{20, 152, 230, 1}, {10, 230, 200, 1, 12}}}};
constexpr HeadCost kPartCosts[2][2][2] = {{{{60, 106, 0, 2}, {20, 200, 80, 1}}, {{20, 165, 130, 1}, {70, 210, 130, 1}}},
                                          {{{35, 90, 70, 1}, {20, 187, 120, 1}}, {{25, 155, 70, 1}, {0, 280, 260, 1}}}};
long long cost_of_head_workgroups(const HeadCost& c, long long wgs, int rounds, long long key_bytes) {
  const long long at_a_time = (long long)kComputeUnits * c.together, full = wgs / at_a_time, rest = wgs % at_a_time;
  auto one_time = [&](long long n, bool first) -> long long {
    const long long alone = c.start + c.step * rounds, memory = n * key_bytes / (wgs * 67000);
    const long long work = (n > kComputeUnits ? alone * 3 / 2 : alone) + (first ? 0 : c.again) + memory * c.slowed / 100;
    return work > memory ? work : memory;
  };
  return (full > 0 ? one_time(at_a_time, true) + (full - 1) * one_time(at_a_time, false) : 0) + (rest > 0 ? one_time(rest, full == 0) : 0);
}
// Groups of 32 query rows per workgroup of the kernel that serves `rows` query rows of `heads` heads: 1 or 2 (fmha_i8_split_kernel), 4
// (fmha_i8_pair_kernel), kFew (fmha_i8_few_kernel), or 0 for the kernel of 256-row workgroups.  All write the same bytes.
//
// Each kernel's time beyond the launch is modelled as (workgroups per CU, rounded up) * (cost of one), and `again` for all but the
// first; at most 32 query rows as above.  What the constants order is far apart nearly everywhere - d128, S2048: H4 31.0 us in 256-row
// workgroups, 24.4 in those of four groups, 17.6 of two, 13.4 of one; H8 31.3, 24.6, 17.9, 25.8; H16 31.7, 26.2, 34.5, 50.3; H24 33.9,
// 48.9, 50.7, 74.6 - so that a few percent of error only shift the boundary between equals.
struct Choice {
  int row_groups;
  long long cost;  // hundredths of a microsecond
};
long long cost_of_workgroups(const KernelCost& kernel, long long wgs, int head_dim, int blocks, int block_keys) {
  const auto& c = kernel.cost[head_dim == 128][block_keys == fmha_i8_gfx950::kBlockK];
  const long long per_cu = (wgs + kComputeUnits - 1) / kComputeUnits;
  return per_cu * (c.start + c.step * ((blocks + kernel.keys_per_round - 1) / kernel.keys_per_round)) + (per_cu - 1) * c.again;
}
int rows_of(const KernelCost& kernel) {
  return kernel.row_groups == 0 ? fmha_i8_gfx950::kBlockQ : 32 * kernel.row_groups;
}
// At most sixteen rows, and not the geometry that the split kernel's second group serves better (see fmha_i8_few_kernel).
bool few_takes(int rows, int head_dim, int block_keys) {
  return rows <= fmha_i8_gfx950::kFewRows && !(head_dim == 128 && block_keys == fmha_i8_gfx950::kBlockK);
}
// With one group's worth of rows the second group of the split kernel only helps to fetch the tiles, which pays where a round is 128 KB
// (B8 H16 Sq1 S2048 d128: 15.9 us with one group, 14.1 with two; H96 S2048 14.9 and 13.7, S16384 116 and 99; with 16 heads 13.1 and
// 12.6; at d64 11.7 either way): there it takes one group's place.
bool second_group_fetches(int rows, int head_dim, int block_keys) { return rows <= 32 && head_dim == 128 && block_keys == fmha_i8_gfx950::kBlockK; }
Choice cheapest_kernel(long long heads, int rows, int head_dim, int blocks, int block_keys) {
  if (rows <= 32) {
    const bool few = few_takes(rows, head_dim, block_keys), fetching = second_group_fetches(rows, head_dim, block_keys);
    // (a last round of one or two key blocks: the two-step form stops behind its first step, half a microsecond sooner)
    const int left_out = fetching && (blocks & 3) != 0 && (blocks & 3) <= 2 ? 50 : 0;
    HeadCost price = kHeadCosts[rows > fmha_i8_gfx950::kFewRows][head_dim == 128][block_keys == fmha_i8_gfx950::kBlockK];
    price.start -= left_out;
    return {few ? kFew : fetching ? 2 : 1, cost_of_head_workgroups(price, heads, (blocks + 3) / 4, 2 * heads * blocks * block_keys * head_dim)};
  }
  Choice best{0, -1};
  for (const KernelCost& kernel : kKernelCosts) {
    const long long cost = cost_of_workgroups(kernel, heads * ((rows + rows_of(kernel) - 1) / rows_of(kernel)), head_dim, blocks, block_keys);
    if (best.cost < 0 || cost < best.cost) best = {kernel.row_groups, cost};
  }
  return best;
}
Choice row_groups_of(const FMHACrossAttnDescriptor& a, int block_keys) {
  if (a.seq_len_kv <= block_keys) return {0, -1};
  const int forced = fmha_i8_gfx950::test_build::forced_route();
  if (forced >= 0 && (forced != kFew || few_takes(a.seq_len_q, a.head_dim, block_keys))) return {forced, -1};
  return cheapest_kernel((long long)a.batch_num * a.head_num, a.seq_len_q, a.head_dim, (a.seq_len_kv + block_keys - 1) / block_keys, block_keys);
}
// The launches of a call: one, or two where large workgroups would leave most compute units idle in their last wave, or in the last
// rows of every head.  The first launch then takes as many heads, or as many rows of every head, as make full waves of workgroups of 256
// or 128 rows, the second one the rest in smaller ones.  A second launch costs 2.8 us, and 5 % are left to the model's error.
int pieces_of(const FMHACrossAttnDescriptor& a, int block_keys, Piece (&pieces)[2]) {
  const int heads = a.batch_num * a.head_num, rows = a.seq_len_q, blocks = (a.seq_len_kv + block_keys - 1) / block_keys;
  const Choice whole = row_groups_of(a, block_keys);
  pieces[0] = {whole.row_groups, 0, heads, 0, rows};
  if (whole.cost < 0 || rows <= 32 || fmha_i8_gfx950::test_build::forced_route() == fmha_i8_gfx950::test_build::kOneLaunch) return 1;
  long long least = whole.cost * 19 / 20;
  int count = 1;
  auto consider = [&](const KernelCost& kernel, int first_heads, int first_rows) {
    const bool by_heads = first_rows == rows;
    const int rest_heads = by_heads ? heads - first_heads : heads, rest_rows = by_heads ? rows : rows - first_rows;
    if (first_heads <= 0 || first_rows <= 0 || rest_heads <= 0 || rest_rows <= 0) return;
    const long long wgs = (long long)first_heads * ((first_rows + rows_of(kernel) - 1) / rows_of(kernel));
    const Choice rest = cheapest_kernel(rest_heads, rest_rows, a.head_dim, blocks, block_keys);
    const long long cost = cost_of_workgroups(kernel, wgs, a.head_dim, blocks, block_keys) + kLaunch + rest.cost;
    if (rest.row_groups == 0 || cost >= least) return;
    least = cost;
    count = 2;
    pieces[0] = {kernel.row_groups, 0, first_heads, 0, first_rows};
    pieces[1] = {rest.row_groups, heads - rest_heads, rest_heads, rows - rest_rows, rows};
  };
  for (const KernelCost& kernel : kKernelCosts) {
    if (kernel.row_groups != 0 && kernel.row_groups != 4) continue;
    const long long per_head = (rows + rows_of(kernel) - 1) / rows_of(kernel), full_waves = heads * per_head / kComputeUnits;
    consider(kernel, (int)(full_waves * kComputeUnits / per_head), rows);
    consider(kernel, heads, rows / rows_of(kernel) * rows_of(kernel));
  }
  return count;
}
// What follows the workgroups of shared-out key blocks ([at most sixteen rows, more], hundredths of a microsecond): the merge's launch and its
// first batch of key blocks, more for batches of 32 instead of 16, for a second batch, for each further one (with more than sixteen rows some row
// moves its reference in nearly every block), and the workspace written and read, bytes in a hundredth of a microsecond, those of its first
// 20 MB on top: with one rate for all (42 KB) calls of 17 to 32 rows over more than 8000 keys lost up to 47 % (H32 Sq32 S14400 d128 100.7 us plain,
// 68.4 shared out).
struct MergeCost {
  int launch, wide, second, further, rate, first_rate;
};
constexpr MergeCost kMergeCosts[2] = {{208, 88, 160, 30, 75000, 174000}, {315, 80, 245, 340, 118000, 55500}};
// Whether a call shares its key blocks out, and how: as few rounds per workgroup as there are compute units for (kPartCosts), and what follows
// them.  (One head and up to eight heads are put 0.4 us too low: calls whose two routes are that close stay shared out, as they have been - H1
// Sq8 S1089 d64 7.2 us either way, H6 Sq5 S1030 d64 7.4 and 8.0.)  Within 5 % of each other (the factor 20/21) the plain route is taken, which
// needs no memory and can write a float output besides.
// One call, plain and shared out, us: d128 B1 H16 Sq1 S2048 12.1 and 8.0, H32 S4096 21.6 and 9.6, H16 Sq32 S4096 21.2 and 14.6, B2 H16 Sq32
// S1664 11.6 and 12.8, S2048 12.1 and 13.7, H16 Sq17 S1152 9.3 and 9.8, H264 Sq1 S640 15.4 and 18.1, S1152 22.3 and 20.3, B8 H16 Sq1 S2048,
// which the memory bounds already, 13.8 and 14.7; d64 H64 Sq1 S2048 8.5 and 7.6, H264 Sq1 S1088 9.3 and 14.2.
// Of 2,316 such calls timed on both routes, 1 to 1024 heads and up to 65536 keys, the choice is more than 2 % slower than the other one in 80,
// more than 10 % in 5; of 500 others, drawn where the two are close, in 28 and 8, at most by 17 % (H140 Sq1 S18624 d64, more than the last cache
// holds).  It was in 398 and 141, and 71 and 21, with a table that priced the two sides apart, took each further workgroup on a CU for as dear as
// the first and the memory for a bound on the whole call alone.
PartPlan part_plan_of(const FMHACrossAttnDescriptor& a, int block_keys) {
  using namespace fmha_i8_gfx950;
  PartPlan plan;
  const int blocks = (a.seq_len_kv + block_keys - 1) / block_keys, rounds = (blocks + kSplitKeys - 1) / kSplitKeys;
  const long long heads = (long long)a.batch_num * a.head_num;
  if (a.seq_len_q > kPartRows || rounds < 2 || heads > 65535) return plan;  // (heads: the y extent of the merge's grid)
  if (test_build::forced_route() >= 0) return plan;
  const bool one_group = a.seq_len_q > kFewRows;
  const MergeCost& c = kMergeCosts[one_group];
  const long long bytes = heads * blocks * a.seq_len_q * (8 * a.head_dim + 16), first_bytes = bytes < 20000000 ? bytes : 20000000;
  const long long merge = c.launch - 42 / heads + (blocks <= 16 ? 0 : heads > 8 ? c.wide : c.wide / 2) + (blocks <= 32 ? 0 : c.second + c.further * ((blocks - 33) / 32)) +
                          bytes / c.rate + first_bytes / c.first_rate;
  const HeadCost& price = kPartCosts[one_group][a.head_dim == 128][block_keys == kBlockK];
  const long long plain = cheapest_kernel(heads, a.seq_len_q, a.head_dim, blocks, block_keys).cost * 20 / 21;
  long long work = 0;
  for (int r = 1; r < rounds; ++r) {
    // (without the memory, which makes equals of splits that are not: H32 Sq1 S8192 d128 18.6 us in 256 workgroups, 22.0 in 512)
    const long long of_r = cost_of_head_workgroups(price, heads * ((rounds + r - 1) / r), r, 0);
    if (plan.rounds_per_part > 0 && of_r > work) continue;
    work = of_r;
    plan.rounds_per_part = r;
  }
  const int r = plan.rounds_per_part;
  work = cost_of_head_workgroups(price, heads * ((rounds + r - 1) / r), r, 2 * heads * blocks * block_keys * a.head_dim);
  if (work + merge >= plain && test_build::forced_route() != test_build::kSharedOut) plan.rounds_per_part = 0;
  const size_t rows = (size_t)heads * blocks * a.seq_len_q;
  plan.ml_bytes = (rows * sizeof(v2f) + 255) / 256 * 256;
  plan.bytes = plan.ml_bytes + rows * a.head_dim * sizeof(int);
  return plan;
}
#endif

// Blocks of 128 keys, as the reference uses for its multiples of 128; its other lengths (64, 192, 320, 448:
// src/fmha_i8.cu:41-60) run in blocks of 64 keys, and so does every other odd multiple of 64 here.
// A key count that is not a multiple of 64 is treated as the next multiple of 64 whose last keys are masked out.
int padded_keys(int seq_len_kv) {
  return (seq_len_kv + fmha_i8_gfx950::kBlockKSmall - 1) / fmha_i8_gfx950::kBlockKSmall * fmha_i8_gfx950::kBlockKSmall;
}
int block_keys_of(int seq_len_kv) {
  return padded_keys(seq_len_kv) % fmha_i8_gfx950::kBlockK == 0 ? fmha_i8_gfx950::kBlockK : fmha_i8_gfx950::kBlockKSmall;
}

int launch(hipStream_t stream, const FMHAParamI8& p, const FMHACrossAttnDescriptor& a, const void* q, const void* k,
           const void* v, const void* mask, void* o, bool full_range_p = false, void* workspace = nullptr, size_t workspace_bytes = 0, void* wide = nullptr,
           bool wide_is_bf16 = false) {
  const int st = check_args(p, a, q, k, v, mask, o);
  if (st != FMHA_I8_OK) return st;
  constexpr float kLog2e = 1.4426950408889634f;
  KernelArgs args;
  args.q = static_cast<const int8_t*>(q);
  args.k = static_cast<const int8_t*>(k);
  args.v = static_cast<const int8_t*>(v);
  args.mask = static_cast<const int8_t*>(mask);
  args.o = static_cast<int8_t*>(o);
  args.seq_q = a.seq_len_q;
  args.seq_kv = a.seq_len_kv;
  args.head_num = a.head_num;
  args.q_blocks = (a.seq_len_q + fmha_i8_gfx950::kBlockQ - 1) / fmha_i8_gfx950::kBlockQ;
  args.total_wgs = a.batch_num * a.head_num * args.q_blocks;
  args.c2 = score_scale_log2(p, a.head_dim);
  // A masked score is replaced by -inf before it is scaled (see the kernel): the scale must not be exactly 0.  With
  // 1e-30 every exponent is below 1e-23 in magnitude and the probabilities are the same floats as with 0.
  if (args.c2 < 1e-30f) args.c2 = 1e-30f;
  args.floor2 = -1e6f * kLog2e;
  args.out_scale = output_scale(p);
  args.wide = wide;
  args.wide_amax = p.o_amax;
  args.wide_is_bf16 = wide_is_bf16;
  args.first_head = args.first_row = 0;
  // The accumulators of Q.K^T can be read as floats without a convert when they start at the bit pattern of a float;
  // the price is that the exponent offset (start value*2^26 + S)*c2 is then rounded on a coarser float grid.  Take that
  // path only while the offset stays below 2^12, i.e. while the rounding moves a whole row by less than 2^-13 in log2.
  // (The start value and the bound on |S| depend on the head size: see score_base_bits in the kernel source.)
  const float offset_ulps = a.head_dim == 64
                                ? fmha_i8_gfx950::score_base_ulps<64>() + fmha_i8_gfx950::score_range_ulps<64>()
                                : fmha_i8_gfx950::score_base_ulps<128>() + fmha_i8_gfx950::score_range_ulps<128>();
  const bool bias = offset_ulps * fabsf(args.c2) < fmha_i8_gfx950::kBiasOffsetLimit;
  // Folding the accumulator offset into the running O (see FASTACC in the kernel) costs a rounding of relative size
  // 2^-24 at magnitude kBase * sum(take) per key block; normalised by the row sum (>= sum(take)) and scaled to output
  // LSBs that is at most about 0.0034 * (v_amax/o_amax) * sqrt(key blocks).  Take it while that stays below 0.1 LSB.
  const int kv_padded = padded_keys(a.seq_len_kv), block_keys = block_keys_of(a.seq_len_kv);
  const float lsb_bound = 0.0034f * fabsf(p.v_amax / p.o_amax) * sqrtf((float)(kv_padded / block_keys));
  const bool fast = lsb_bound < 0.1f;
  const Variant var{bias, fast, full_range_p};
  hipError_t err;
#ifndef FMHA_NO_SPLIT_KERNEL
  if (workspace != nullptr) {
    if ((uintptr_t)workspace & 15u) return FMHA_I8_ERR_ALIGNMENT;
    const PartPlan plan = part_plan_of(a, block_keys);
    if (plan.rounds_per_part > 0 && plan.bytes <= workspace_bytes) {
      if (a.head_dim == 128)
        err = block_keys == fmha_i8_gfx950::kBlockK ? launch_parts<128, fmha_i8_gfx950::kBlockK>(plan, var, stream, args, workspace)
                                                    : launch_parts<128, fmha_i8_gfx950::kBlockKSmall>(plan, var, stream, args, workspace);
      else
        err = block_keys == fmha_i8_gfx950::kBlockK ? launch_parts<64, fmha_i8_gfx950::kBlockK>(plan, var, stream, args, workspace)
                                                    : launch_parts<64, fmha_i8_gfx950::kBlockKSmall>(plan, var, stream, args, workspace);
      return err == hipSuccess ? FMHA_I8_OK : FMHA_I8_ERR_HIP_BASE + (int)err;
    }
  }
  Piece pieces[2];
  const int count = pieces_of(a, block_keys, pieces);
  err = hipSuccess;
  for (int i = 0; i < count && err == hipSuccess; ++i) {
    if (pieces[i].row_groups == 0) {
      args.q_blocks = (pieces[i].end_row + fmha_i8_gfx950::kBlockQ - 1) / fmha_i8_gfx950::kBlockQ;
      args.total_wgs = pieces[i].heads * args.q_blocks;
      err = launch_wide(a.head_dim, block_keys, var, stream, args);
    } else if (a.head_dim == 128) {
      err = block_keys == fmha_i8_gfx950::kBlockK ? launch_split<128, fmha_i8_gfx950::kBlockK>(pieces[i], var, stream, args)
                                                  : launch_split<128, fmha_i8_gfx950::kBlockKSmall>(pieces[i], var, stream, args);
    } else {
      err = block_keys == fmha_i8_gfx950::kBlockK ? launch_split<64, fmha_i8_gfx950::kBlockK>(pieces[i], var, stream, args)
                                                  : launch_split<64, fmha_i8_gfx950::kBlockKSmall>(pieces[i], var, stream, args);
    }
  }
#else
  err = launch_wide(a.head_dim, block_keys, var, stream, args);
#endif
  return err == hipSuccess ? FMHA_I8_OK : FMHA_I8_ERR_HIP_BASE + (int)err;
}

}  // namespace

extern "C" {

int FMHAInferI8CheckArgs(FMHAParamI8 fmha_param, AttnDataDescriptor attn_desc, const void* q, const void* k,
                         const void* v, const void* padding_mask, const void* o) {
  return check_args(fmha_param, as_cross(attn_desc), q, k, v, padding_mask, o);
}

int FMHAInferI8Status(hipStream_t stream, FMHAParamI8 fmha_param, AttnDataDescriptor attn_desc, const void* q,
                      const void* k, const void* v, const void* padding_mask, void* o, bool /*use_tcu*/) {
  return launch(stream, fmha_param, as_cross(attn_desc), q, k, v, padding_mask, o);
}

int FMHAInferI8Cross(hipStream_t stream, FMHAParamI8 fmha_param, FMHACrossAttnDescriptor desc, const void* q,
                     const void* k, const void* v, const void* padding_mask, void* o) {
  return launch(stream, fmha_param, desc, q, k, v, padding_mask, o);
}

int FMHAInferI8CrossFullRangeP(hipStream_t stream, FMHAParamI8 fmha_param, FMHACrossAttnDescriptor desc, const void* q,
                               const void* k, const void* v, const void* padding_mask, void* o) {
  return launch(stream, fmha_param, desc, q, k, v, padding_mask, o, true);
}

int FMHAInferI8CrossToFloat(hipStream_t stream, FMHAParamI8 fmha_param, FMHACrossAttnDescriptor desc, const void* q,
                            const void* k, const void* v, const void* padding_mask, void* o, int full_range_p, void* o_float,
                            int o_float_is_bf16) {
  if (o_float == nullptr) return FMHA_I8_ERR_NULL_POINTER;
  if ((uintptr_t)o_float & 15u) return FMHA_I8_ERR_ALIGNMENT;
  return launch(stream, fmha_param, desc, q, k, v, padding_mask, o, full_range_p != 0, nullptr, 0, o_float, o_float_is_bf16 != 0);
}

size_t FMHAInferI8CrossWorkspaceBytes(FMHACrossAttnDescriptor desc) {
#ifndef FMHA_NO_SPLIT_KERNEL
  if ((desc.head_dim != 64 && desc.head_dim != 128) || desc.seq_len_kv <= 0 || desc.seq_len_kv > 65536 || desc.seq_len_q <= 0 ||
      desc.batch_num <= 0 || desc.head_num <= 0)
    return 0;
  const PartPlan plan = part_plan_of(desc, block_keys_of(desc.seq_len_kv));
  return plan.rounds_per_part > 0 ? plan.bytes : 0;
#else
  return 0;
#endif
}

int FMHAInferI8CrossWithWorkspace(hipStream_t stream, FMHAParamI8 fmha_param, FMHACrossAttnDescriptor desc, const void* q,
                                  const void* k, const void* v, const void* padding_mask, void* o, int full_range_p,
                                  void* workspace, size_t workspace_bytes) {
  return launch(stream, fmha_param, desc, q, k, v, padding_mask, o, full_range_p != 0, workspace, workspace_bytes);
}

int FMHAInferI8CrossCheckArgs(FMHAParamI8 fmha_param, FMHACrossAttnDescriptor desc, const void* q, const void* k,
                              const void* v, const void* padding_mask, const void* o) {
  return check_args(fmha_param, desc, q, k, v, padding_mask, o);
}

void FMHAInferI8(hipStream_t stream, FMHAParamI8 fmha_param, AttnDataDescriptor attn_desc, const void* q, const void* k,
                 const void* v, const void* padding_mask, void* o, bool /*use_tcu*/) {
  const int st = launch(stream, fmha_param, as_cross(attn_desc), q, k, v, padding_mask, o);
  if (st != FMHA_I8_OK)
    fprintf(stderr, "FMHAInferI8: nothing launched, o left untouched: %s (B=%d H=%d S=%d d=%d)\n",
            FMHAInferI8StatusString(st), attn_desc.batch_num, attn_desc.head_num, attn_desc.seq_len,
            attn_desc.head_dim);
}

const char* FMHAInferI8StatusString(int status) {
  switch (status) {
    case FMHA_I8_OK: return "ok";
    case FMHA_I8_ERR_NULL_POINTER: return "null pointer argument";
    case FMHA_I8_ERR_HEAD_DIM: return "head_dim must be 64 or 128";
    case FMHA_I8_ERR_SEQ_LEN: return "seq_len must be between 1 and 65536 (queries and keys alike)";
    case FMHA_I8_ERR_BATCH_HEAD: return "batch_num and head_num must be positive (and the grid must fit)";
    case FMHA_I8_ERR_ALIGNMENT: return "q, k, v and o must be 16-byte aligned";
    case FMHA_I8_ERR_SCALE: return "amax values must be finite, o_amax > 0, q_amax * k_amax >= 0, and the scales derived from them finite";
    default: break;
  }
  if (status >= FMHA_I8_ERR_HIP_BASE) return hipGetErrorString((hipError_t)(status - FMHA_I8_ERR_HIP_BASE));
  return "unknown status";
}

#ifdef FMHA_CHECK_BOUNDS
// Test build only: the number of global accesses that would have left their tensor since the last call of this
// function (synchronises the device; see the kernel source).
int FMHAInferI8DebugOutOfBounds(void) {
  int count = -1, zero = 0;
  if (hipDeviceSynchronize() != hipSuccess) return -1;
  if (hipMemcpyFromSymbol(&count, HIP_SYMBOL(fmha_i8_gfx950::g_fmha_oob_count), sizeof(int)) != hipSuccess) return -1;
  if (hipMemcpyToSymbol(HIP_SYMBOL(fmha_i8_gfx950::g_fmha_oob_count), &zero, sizeof(int)) != hipSuccess) return -1;
  return count;
}
#endif

#ifdef FMHA_FORCED_ROUTE
// Test build only: the kernel that serves the calls from here on (see the flag list of the test builds).
void FMHAInferI8DebugRoute(int route) { fmha_i8_gfx950::test_build::g_route = route; }
// Test build only: how many launches serve a call of this shape, and the heads and the rows of the first one.
int FMHAInferI8DebugLaunches(FMHACrossAttnDescriptor desc, int* first_heads, int* first_rows) {
  Piece pieces[2];
  const int count = pieces_of(desc, block_keys_of(desc.seq_len_kv), pieces);
  *first_heads = pieces[0].heads;
  *first_rows = pieces[0].end_row;
  return count;
}
// Test build only: the rounds of a workgroup of a call that shares its key blocks out, 0 for others.
int FMHAInferI8DebugRoundsPerPart(FMHACrossAttnDescriptor desc) { return part_plan_of(desc, block_keys_of(desc.seq_len_kv)).rounds_per_part; }
// Test build only: the kernel of the second launch, as FMHAInferI8DebugRoute names it, or -1.
int FMHAInferI8DebugSecondKernel(FMHACrossAttnDescriptor desc) {
  Piece pieces[2];
  return pieces_of(desc, block_keys_of(desc.seq_len_kv), pieces) == 2 ? pieces[1].row_groups : -1;
}
#endif

#ifdef FMHA_TRACE_TICKS
// Test build only: copies the first `words` time stamps of the last launch (see the kernel source) to host memory.
int FMHAInferI8DebugReadTrace(unsigned* dst, int words) {
  if (hipDeviceSynchronize() != hipSuccess) return -1;
  if (words < 0 || words > fmha_i8_gfx950::kTraceWorkgroups * 8 * 64) return -1;
  return hipMemcpyFromSymbol(dst, HIP_SYMBOL(fmha_i8_gfx950::g_fmha_trace), sizeof(unsigned) * words) == hipSuccess ? 0 : -1;
}
#endif

const char* FMHAInferI8Version(void) { return "fmha_i8 gfx950 mfma32x32x32 direct-to-lds two-phase"; }

}  // extern "C"
