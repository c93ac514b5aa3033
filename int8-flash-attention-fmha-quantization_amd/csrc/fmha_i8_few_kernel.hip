// The attention kernel for calls of at most sixteen query rows per head: one new row per sequence, or the few of a speculative
// step.  The work of fmha_i8_split_kernel for one row group, with the same bytes, on matrix instructions of 16 query rows
// (v_mfma_i32_16x16x64_i8; keys and output columns are the other operand) in place of 32.
//
// What bounds it: the round of that kernel, 512 keys of one row at d128, was arithmetic from end to end - 1100 cycles GEMM 1, 2100
// softmax, 1650 GEMM 2 and merge, no wait for any load - of which 31 rows in 32 were thrown away.  Here a lane has half the scores
// and the MFMAs take half the cycles; of GEMM 2 the transposing reads of V (64 bytes per cycle) remain.  Before and now, us:
// d64 B8 H16 Sq1 S2048 11.7 and 9.2, B8 H16 Sq4 S2000 with masked keys and 255 steps 15.1 and 10.9, B6 H16 S16384 71.8 and 55.2,
// d128 B8 H16 S1984 (blocks of 64 keys) 15.5 and 14.4, B3 H5 Sq16 S777 9.1 and 7.9.
// At d128 in blocks of 128 keys a CU has 128 KB to fetch per round, at some 43 GB/s, and what counts is that the loads hold nobody
// up: there the second row group of the split kernel, which has no rows and only loads, is the faster one (B8 H16 S2048 13.5
// against 14.6 us), and this kernel serves shared-out key blocks alone.
#pragma once

namespace fmha_i8_gfx950 {

constexpr int kFewRows = 16;

// Lanes l and l^16 hold two of a query row's four parts, as l and l^32 do.
__device__ __forceinline__ int row_max16(int x) {
  const auto r = __builtin_amdgcn_permlane16_swap(x, x, false, false);
  return half_max(max((int)r[0], (int)r[1]));
}

// V tiles are read by ds_read_b64_tr_b8.  Thirty-two lanes read one chunk column of keys {0 .. 7, 16 .. 23} (+8): rows that start in the
// same bank get different chunks by bits 1 (at d128), 2 and 4 of the key.  (By bits 0, 1 and 4, which tell the keys of sixteen lanes
// apart: 256 cycles of bank conflicts per round; B8 H16 Sq1 S2048 d64 9.12 -> 8.97 us, H16 S4096 14.5 -> 14.3, H16 Sq16 S1984 d128
// 14.2 -> 14.0.)
template <int D>
__device__ __forceinline__ int few_v_swizzle(int key) {
  return D == 128 ? (((key >> 1) & 3) | ((key >> 2) & 4)) : (((key >> 2) & 1) | ((key >> 3) & 2));
}

template <int D, int BK, bool BIAS, bool FASTACC, bool FULLP, bool PARTS>
__global__ __launch_bounds__(256, 1) void fmha_i8_few_kernel(const SplitKernelArgs args) {
  constexpr int kTileBytes = BK * D;
  constexpr int kRegions = kTileBytes / 1024;
  constexpr int kLoads = kRegions;  // direct-to-LDS loads per wavefront for its own K tile, and for its share of four V tiles
  constexpr int kChunks = D / 16;
  constexpr int kRowsPerRegion = 1024 / D;
  constexpr int kDSteps = D / 64;
  constexpr int kTiles = BK / 16;         // of 16 keys
  constexpr int kSteps = BK / 64;         // of GEMM 2
  constexpr int kColumnTiles = D / 64;    // of 16 columns, per wavefront
  constexpr bool kTwoBuffersV = kTileBytes <= 8192;  // LDS holds 160 KB
  static_assert(kTwoBuffersV || PARTS, "");

  __shared__ __attribute__((aligned(1024))) int8_t lds_k[kSplitKeys][kTileBytes];
  __shared__ __attribute__((aligned(1024))) int8_t lds_v[kTwoBuffersV ? 2 : 1][kSplitKeys][kTileBytes];
  __shared__ __attribute__((aligned(16))) v4i lds_p[kSplitKeys][kSteps][64];  // P^T as the B operand of GEMM 2
  __shared__ __attribute__((aligned(8))) float lds_ml[kSplitKeys][kFewRows][2];
  __shared__ unsigned lds_class4[kMaxKeyBlocks / 4];
  __shared__ unsigned lds_mask[kMaxKeyBlocks * kBlockKSmall / 32];
  __shared__ int lds_scan[4];

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int c = __builtin_amdgcn_readfirstlane(tid >> 6);  // key block of the round, and the output columns D / 4 * c ..
  const int g = lane >> 4;   // keys 16 t + 4 g .. +3 of a tile of scores
  const int row = lane & 15;

  int wg;
  {  // XCD-aware placement, as in the 256-row kernel
    const int L = blockIdx.x, per = args.total_wgs / kXcds, rem = args.total_wgs % kXcds, x = L % kXcds;
    wg = x * per + (x < rem ? x : rem) + L / kXcds;
  }
  const int bh_here = divide(wg, args.q_blocks_divisor), bh = bh_here + args.first_head;
  const int part = wg - bh_here * args.q_blocks;
  const int b = divide(bh, args.head_num_divisor);
  const int S = args.seq_kv, Sq = args.seq_q;
  const int8_t* __restrict__ kg = args.k + (long)bh * S * D;
  const int8_t* __restrict__ vg = args.v + (long)bh * S * D;
  const int8_t* __restrict__ mg = args.mask + (long)b * S;
  const long q_head_off = (long)bh * Sq * D;
  const int n_blocks = (S + BK - 1) / BK;
  const int first_round = PARTS ? part * args.rounds_per_part : 0;
  const int tail_kb = S % BK != 0 ? n_blocks - 1 : -1;

  // ---- tile loads (see fmha_i8_split_kernel) -------------------------------------------------------------------------
  const int row_in = lane / kChunks, chunk = lane % kChunks;
  int ld_k, ld_k_odd, ld_v;
  {
    ld_k = row_in * D + ((chunk ^ k_swizzle<D>(row_in)) << 4);
    ld_k_odd = row_in * D + ((chunk ^ k_swizzle<D>(row_in + kRowsPerRegion)) << 4);
    ld_v = row_in * D + ((chunk ^ few_v_swizzle<D>(row_in + c * kRowsPerRegion)) << 4) + c * 1024;
  }
  const unsigned k_base = (unsigned)(uintptr_t)(__attribute__((address_space(3))) int8_t*)&lds_k[0][0] + c * kTileBytes;
  const unsigned v_base = (unsigned)(uintptr_t)(__attribute__((address_space(3))) int8_t*)&lds_v[0][0][0] + c * 1024;
  auto load = [&](unsigned dst, int src, const int8_t* from) __attribute__((always_inline)) {
    if (!fmha_in_bounds(src >= 0 && src + 16 <= S * D)) src = 0;
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(dst), "v"(src), "s"(from) : "memory");
  };
  auto tile_of = [&](int kb) { return kb == tail_kb ? (S - BK) * D : kb * kTileBytes; };
  auto load_k = [&](int round, int it, int last) __attribute__((always_inline)) {
    load(k_base + it * 1024, tile_of(min(kSplitKeys * round + c, last)) + it * 1024 + (it & 1 ? ld_k_odd : ld_k), kg);
  };
  auto load_v = [&](int round, int it, int last) __attribute__((always_inline)) {
    const int slot = 4 * it / kRegions, region = 4 * it % kRegions;  // besides region c
    load(v_base + ((kTwoBuffersV ? round & 1 : 0) * kSplitKeys + slot) * kTileBytes + region * 1024,
         tile_of(min(kSplitKeys * round + slot, last)) + region * 1024 + ld_v, vg);
  };
  auto barrier = [&]() { asm volatile("s_barrier" ::: "memory"); };
  auto written = [&]() { asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); };
  auto wait_loads = [&](auto outstanding) { asm volatile("s_waitcnt vmcnt(%0)" ::"n"(decltype(outstanding)::value) : "memory"); };

  // ---- prologue: mask bytes, Q rows, K and V of the first round ------------------------------------------------------
  const int keys_from = PARTS && first_round > 0 ? (kSplitKeys * first_round - 1) * BK : 0;
  const int keys_to = PARTS ? min(n_blocks, kSplitKeys * (first_round + args.rounds_per_part)) * BK : n_blocks * BK;
  v4i mask_bytes, tail_bytes;
  {
    const int mine = keys_from + kMaskBytesPerLane * tid;
    int j = mine + kMaskBytesPerLane <= S ? mine : 0, jt = S - kMaskBytesPerLane;
    if (!fmha_in_bounds(j >= 0 && j + kMaskBytesPerLane <= S && jt >= 0)) j = jt = 0;
    asm volatile("global_load_dwordx4 %0, %2, %3\n\tglobal_load_dwordx4 %1, %4, %3"
                 : "=&v"(mask_bytes), "=v"(tail_bytes) : "v"(j), "s"(mg), "v"(jt) : "memory");
  }
  const int row0 = PARTS ? 0 : args.first_row;
  v4i qreg[kDSteps];
  {
    int qrow = min(row0 + row, Sq - 1);  // rows past the end load the last row (unused)
    if (!fmha_in_bounds(qrow >= 0 && qrow < Sq)) qrow = 0;
    const int8_t* qp = args.q + q_head_off;
#pragma unroll
    for (int kk = 0; kk < kDSteps; ++kk)
      asm volatile("global_load_dwordx4 %0, %1, %2" : "=v"(qreg[kk]) : "v"(qrow * D + 64 * kk + 16 * g), "s"(qp) : "memory");
  }
#pragma unroll
  for (int it = 0; it < kLoads; ++it) load_k(first_round, it, n_blocks - 1);
#pragma unroll
  for (int it = 0; it < kLoads; ++it) load_v(first_round, it, n_blocks - 1);

  // operand addresses
  int k_read_off[kDSteps];
#pragma unroll
  for (int kk = 0; kk < kDSteps; ++kk) k_read_off[kk] = row * D + (((4 * kk + g) ^ k_swizzle<D>(row)) << 4);
  int v_read_off[kColumnTiles];
  {
    const int kslot = row >> 1, key = 4 * g + (kslot < 4 ? kslot : kslot + 12);
#pragma unroll
    for (int u = 0; u < kColumnTiles; ++u)
      v_read_off[u] = key * D + (((kColumnTiles * c + u) ^ few_v_swizzle<D>(key)) << 4) + 8 * (row & 1);
  }

  // ---- state -------------------------------------------------------------------------------------------------------
  float o_f[kColumnTiles][4] = {};
  float m_ref = args.floor2 - 2.f * kLazyLog2, t_run = 0.f, l_run = 0.f;
  const float c2 = BIAS ? args.c2 * kBaseScale : args.c2;
  constexpr int kScoreBaseBits = score_base_bits<D>();
  const float bias_c2 = BIAS ? __builtin_bit_cast(float, kScoreBaseBits) * c2 : 0.f;
  constexpr int kStart = BIAS ? kScoreBaseBits : 0, kMaskedStart = BIAS ? (int)0xFF000000 : (int)0xC0000000;  // (see masked_start)

  // ---- classification of the key blocks ------------------------------------------------------------------------------
  asm volatile("s_waitcnt vmcnt(%2)" : "+v"(mask_bytes), "+v"(tail_bytes) : "n"(kDSteps + 2 * kLoads) : "memory");
  const int live_hi = classify_key_blocks<BK, 4>(mask_bytes, tail_bytes, mg, S, tid, lds_mask,
                                                 reinterpret_cast<unsigned char*>(lds_class4), keys_from, keys_to);
  if (lane == 0) lds_scan[c] = live_hi;
  // K of the first round and the Q rows have landed
  asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(kLoads) : "memory");
#pragma unroll
  for (int kk = 0; kk < kDSteps; ++kk) asm volatile("" : "+v"(qreg[kk]));
  barrier();
  int n = -1;
#pragma unroll
  for (int w = 0; w < 4; ++w) n = max(n, lds_scan[w]);
  n = __builtin_amdgcn_readfirstlane(n) + 1;  // one past the last block with an unmasked key
  const int live_rounds = (n + kSplitKeys - 1) / kSplitKeys;
  const int rounds = PARTS ? min(first_round + args.rounds_per_part, live_rounds) : live_rounds;
  const long part_first = (long)bh * n_blocks;
  auto in_workspace = [&](int kb, int r) __attribute__((always_inline)) {  // (see fmha_i8_split_kernel)
    const long heads = args.total_wgs / args.q_blocks;
    return fmha_in_bounds(kb >= 0 && kb < n_blocks && r >= 0 && r < Sq && (part_first + kb) * Sq + r < heads * n_blocks * Sq);
  };
  if constexpr (PARTS) {
    for (int kb = keys_to / BK - 1 - c; kb >= kSplitKeys * first_round; kb -= 4)
      if ((reinterpret_cast<const unsigned char*>(lds_class4)[kb] & 2) && lane < Sq && (!kCheckBounds || in_workspace(kb, lane)))
        args.part_ml[(part_first + kb) * Sq + lane] = v2f{-__builtin_inff(), 0.f};
  }

  // ---- the rounds --------------------------------------------------------------------------------------------------
  const Const<0> none;
  auto merge_blocks = [&](int i, unsigned cls4, auto count_t) __attribute__((always_inline)) {
    constexpr int kCount = decltype(count_t)::value;
    const int8_t* tiles_v = &lds_v[kTwoBuffersV ? i & 1 : 0][0][0];
    typedef v2i __attribute__((address_space(3))) * lds_v2i_ptr;
    v4i oacc[kCount][kColumnTiles];
    float ml[kCount][2];
    if constexpr (!PARTS) {
#pragma unroll
      for (int j = 0; j < kCount; ++j) {
        ml[j][0] = lds_ml[j][row][0];
        ml[j][1] = lds_ml[j][row][1];
      }
    }
#pragma unroll
    for (int j = 0; j < kCount; ++j) {
      v4i va[kColumnTiles][kSteps], p[kSteps];
#pragma unroll
      for (int t = 0; t < kSteps; ++t) {
        p[t] = lds_p[j][t][lane];
#pragma unroll
        for (int u = 0; u < kColumnTiles; ++u) {
          const int8_t* at = tiles_v + j * kTileBytes + v_read_off[u] + 64 * t * D;
          const v2i lo = __builtin_amdgcn_ds_read_tr8_b64_v2i32((lds_v2i_ptr)at);
          const v2i hi = __builtin_amdgcn_ds_read_tr8_b64_v2i32((lds_v2i_ptr)(at + 32 * D));
          va[u][t] = v4i{lo[0], lo[1], hi[0], hi[1]};
        }
      }
#pragma unroll
      for (int u = 0; u < kColumnTiles; ++u) {
        v4i a = FULLP ? v4i{0, 0, 0, 0} : v4i{kBaseBits, kBaseBits, kBaseBits, kBaseBits};
        if (FULLP) {  // (as in fmha_i8_split_kernel)
          const v4i half = {0x40404040, 0x40404040, 0x40404040, 0x40404040};
#pragma unroll
          for (int t = 0; t < kSteps; ++t) a = __builtin_amdgcn_mfma_i32_16x16x64_i8(va[u][t], half, a, 0, 0, 0);
#pragma unroll
          for (int e = 0; e < 4; ++e) a[e] = 2 * a[e] + kBaseBitsFull;
        }
#pragma unroll
        for (int t = 0; t < kSteps; ++t) a = __builtin_amdgcn_mfma_i32_16x16x64_i8(va[u][t], p[t], a, 0, 0, 0);
        oacc[j][u] = a;
      }
    }
    if constexpr (PARTS) {
#pragma unroll
      for (int j = 0; j < kCount; ++j)
        if (!((cls4 >> (8 * j)) & 2) && row < Sq && (!kCheckBounds || in_workspace(kSplitKeys * i + j, row))) {
#pragma unroll
          for (int u = 0; u < kColumnTiles; ++u)
            *reinterpret_cast<v4i*>(args.part_o + (part_first + kSplitKeys * i + j) * Sq * D + ((4 * (kColumnTiles * c + u) + g) * Sq + row) * 4) = oacc[j][u];
        }
    } else {
#pragma unroll
      for (int j = 0; j < kCount; ++j) {
        const bool dead = (cls4 >> (8 * j)) & 2;
        const float mb = dead ? -__builtin_inff() : ml[j][0], lb = dead ? 0.f : ml[j][1];
        const bool moves = __ballot(mb > m_ref + kLazyLog2) != 0;  // (wave-uniform, rare)
        const float m_new = moves ? fmaxf(m_ref, mb) : m_ref;
        const float keep = __builtin_amdgcn_exp2f(m_ref - m_new);  // exactly 1 where nothing moves
        m_ref = m_new;
        const float take = __builtin_amdgcn_exp2f(mb - m_ref);
        l_run = __builtin_fmaf(take, lb, l_run * keep);
        if (FASTACC) t_run = t_run * keep + take;
#pragma unroll
        for (int u = 0; u < kColumnTiles; ++u) {
          if (moves) {
#pragma unroll
            for (int e = 0; e < 4; ++e) o_f[u][e] *= keep;
          }
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const float v = FASTACC ? __int_as_float(oacc[j][u][e]) : __int_as_float(oacc[j][u][e]) - (FULLP ? kBaseFull : kBase);
            o_f[u][e] = __builtin_fmaf(FULLP ? take : -take, v, o_f[u][e]);
          }
        }
      }
    }
  };
  auto do_round = [&](int i, auto more_t) __attribute__((always_inline)) {
    constexpr bool kMore = decltype(more_t)::value != 0;
    const unsigned cls4 = (unsigned)__builtin_amdgcn_readfirstlane((int)lds_class4[i]);
    const int cls = (cls4 >> (8 * c)) & 3, kb = min(kSplitKeys * i + c, n - 1);
    // Behind the MFMAs of GEMM 1 K of the next round, in the softmax V of the next round; with one buffer V of this round, and K.
    auto loads_in_gemm1 = [&](int slot, int slots) __attribute__((always_inline)) {
#pragma unroll
      for (int it = slot * kLoads / slots; it < (slot + 1) * kLoads / slots; ++it) {
        if (kTwoBuffersV && kMore) load_k(i + 1, it, n - 1);
        if (!kTwoBuffersV && i > first_round) load_v(i, it, n - 1);
      }
    };
    auto loads_in_softmax = [&](int slot, int slots) __attribute__((always_inline)) {
#pragma unroll
      for (int it = slot * kLoads / slots; it < (slot + 1) * kLoads / slots; ++it) {
        if (kTwoBuffersV && kMore) load_v(i + 1, it, n - 1);
        if (!kTwoBuffersV && kMore) load_k(i + 1, it, n - 1);
      }
    };
    // S^T
    v4i ka[kTiles][kDSteps], acc[kTiles];
#pragma unroll
    for (int t = 0; t < kTiles; ++t)
#pragma unroll
      for (int kk = 0; kk < kDSteps; ++kk) ka[t][kk] = *reinterpret_cast<const v4i*>(&lds_k[c][k_read_off[kk] + 16 * t * D]);
#pragma unroll
    for (int t = 0; t < kTiles; ++t) acc[t] = v4i{kStart, kStart, kStart, kStart};
    written();  // the K tile has been read: its place is free
    if (cls & 1) {
      unsigned mw[BK / 32];
      mask_words_of<BK>(mw, lds_mask, kb, tail_kb, S);
#pragma unroll
      for (int t = 0; t < kTiles; ++t)
#pragma unroll
        for (int j = 0; j < 4; ++j)
          acc[t][j] = (mw[t / 2] >> (16 * (t & 1) + 4 * g + j)) & 1u ? kMaskedStart : kStart;
    }
    int mx[2] = {(int)0x80000000, (int)0x80000000};
    auto tile_max = [&](int t) __attribute__((always_inline)) {
      mx[0] = max(max(mx[0], acc[t][0]), acc[t][1]);
      mx[1] = max(max(mx[1], acc[t][2]), acc[t][3]);
    };
#pragma unroll
    for (int t = 0; t < kTiles; ++t) {
#pragma unroll
      for (int kk = 0; kk < kDSteps; ++kk) {
        acc[t] = __builtin_amdgcn_mfma_i32_16x16x64_i8(ka[t][kk], qreg[kk], acc[t], 0, 0, 0);
        loads_in_gemm1(t * kDSteps + kk, kTiles * kDSteps);
      }
      if (t >= 2) tile_max(t - 2);
      __builtin_amdgcn_sched_barrier(0);
    }
    tile_max(kTiles - 2);
    tile_max(kTiles - 1);
    int ti = row_max16(max(mx[0], mx[1]));
    if (cls & 1) ti = max(ti, kStart - 1000000);  // the reference's sentinel (inc/fmha_i8.cuh:191-193)
    const float top = BIAS ? __int_as_float(ti) : (float)ti;
    float off = top * c2;
    if (!BIAS) off = __builtin_fmaf(fabsf(off), 2.384185791015625e-07f, off);
    if (!BIAS) off = fmaxf(off, args.floor2);
    const float m_blk = off - bias_c2;
    const float offq = off - (FULLP ? kLog2PscaleFull : kLog2Pscale);
    float quad_sum[kTiles];
    v4i pk[kSteps];
#pragma unroll
    for (int t = 0; t < kTiles; ++t) {
      float x[4];
#pragma unroll
      for (int j = 0; j < 4; ++j)
        x[j] = __builtin_amdgcn_exp2f(__builtin_fmaf(BIAS ? __int_as_float(acc[t][j]) : (float)acc[t][j], c2, -offq));
      float s01 = x[0] + x[1];
      const float s23 = x[2] + x[3];
      s01 += s23;
      quad_sum[t] = s01;
      const v2s lo = FULLP ? __builtin_amdgcn_cvt_pknorm_i16(x[0], x[1]) : __builtin_amdgcn_cvt_pknorm_i16(-x[0], -x[1]);
      const v2s hi = FULLP ? __builtin_amdgcn_cvt_pknorm_i16(x[2], x[3]) : __builtin_amdgcn_cvt_pknorm_i16(-x[2], -x[3]);
      const int four = __builtin_amdgcn_perm(__builtin_bit_cast(int, hi), __builtin_bit_cast(int, lo), 0x06040200);
      pk[t / 4][t % 4] = FULLP ? four ^ (int)0x80808080 : four;
      asm volatile("" : "+v"(quad_sum[t]));
      loads_in_softmax(t, kTiles);
    }
    // The order of additions of the other kernels: the quads of keys 8 k + 4 h one after the other, h = 0 and 1 apart.  A tile of 16
    // keys holds k = 2 t in lanes 0..31 and k = 2 t + 1 in lanes 32..63; h is bit 4 of the lane.
    float l_blk = 0.f;
#pragma unroll
    for (int t = 0; t < kTiles; ++t) {
      const auto both = __builtin_amdgcn_permlane32_swap(__float_as_int(quad_sum[t]), __float_as_int(quad_sum[t]), false, false);
      l_blk += __int_as_float(both[0]);
      l_blk += __int_as_float(both[1]);
    }
    {
      const auto halves = __builtin_amdgcn_permlane16_swap(__float_as_int(l_blk), __float_as_int(l_blk), false, false);
      l_blk = __int_as_float(halves[0]) + __int_as_float(halves[1]);
    }
    if constexpr (PARTS) {
      if (!(cls & 2) && lane < Sq && (!kCheckBounds || in_workspace(kb, lane))) args.part_ml[(part_first + kb) * Sq + lane] = v2f{m_blk, l_blk};
    } else {
      lds_ml[c][row][0] = m_blk;
      lds_ml[c][row][1] = l_blk;
    }
#pragma unroll
    for (int t = 0; t < kSteps; ++t) lds_p[c][t][lane] = pk[t];
    written();
    // V of this round; what has been asked for since may be in flight
    if (kMore) wait_loads(Const<(kTwoBuffersV ? 2 : 1) * kLoads>{});
    else wait_loads(none);
    barrier();
    // GEMM 2 and the merge of the key blocks, in key order; a last round with no more than two live ones stops behind them
    // (d64 B8 H16 S320 4.97 -> 4.82 us, d128 S1088 10.7 -> 10.5)
    if (!kMore && n - kSplitKeys * i <= 2) merge_blocks(i, cls4, Const<2>{});
    else merge_blocks(i, cls4, Const<kSplitKeys>{});
    if (kMore) {
      // this wavefront's K of the next round; with two buffers V may be in flight
      if (kTwoBuffersV) wait_loads(Const<kLoads>{});
      else wait_loads(none);
      barrier();  // P and V of this round are free
    }
  };
  for (int i = first_round; i + 1 < rounds; ++i) do_round(i, Const<1>{});
  if (rounds > first_round) do_round(rounds - 1, Const<0>{});
  wait_loads(none);  // nothing may still be writing LDS when the wavefront ends (only possible when every key is masked)
  if (PARTS) return;

  // ---- epilogue (see the 256-row kernel) -----------------------------------------------------------------------------
  const float fin = (l_run > 0.f) ? args.out_scale * (128.f / kSnorm) * kBaseScale / l_run : 0.f;
  const float corr = FASTACC ? (FULLP ? -kBaseFull * t_run : kBase * t_run) : 0.f;
  if (row0 + row >= Sq) return;
  if (!fmha_in_bounds(q_head_off + (long)(row0 + row + 1) * D <= ((long)args.total_wgs / args.q_blocks + args.first_head) * Sq * D)) return;
#pragma unroll
  for (int u = 0; u < kColumnTiles; ++u) {
    float y[4];
#pragma unroll
    for (int e = 0; e < 4; ++e)
      y[e] = __builtin_amdgcn_fmed3f(__builtin_fmaf(FASTACC ? o_f[u][e] + corr : o_f[u][e], fin, kMagic), kMagic - 127.f, kMagic + 127.f);
    const int lo = __builtin_amdgcn_perm(__float_as_int(y[1]), __float_as_int(y[0]), 0x0c0c0400);
    const int hi = __builtin_amdgcn_perm(__float_as_int(y[3]), __float_as_int(y[2]), 0x0c0c0400);
    const int w[1] = {(int)__builtin_amdgcn_perm(hi, lo, 0x05040100)};
    const long at = q_head_off + (long)(row0 + row) * D + 16 * (kColumnTiles * c + u) + 4 * g;
    *reinterpret_cast<int*>(args.o + at) = w[0];
    store_wide<D>(args, at, w);
  }
}

}  // namespace fmha_i8_gfx950
