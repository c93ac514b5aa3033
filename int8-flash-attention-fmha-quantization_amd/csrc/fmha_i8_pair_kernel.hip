// The attention kernel with workgroups of 128 query rows, half of those of fmha_i8_fwd_kernel (fmha_i8_kernel.hip) in half
// the time: for calls whose 256-row workgroups leave compute units idle, in their only wave or in their last.  Same
// arithmetic, same BYTES for every row.
//
// Wavefronts w and w + 4 share a SIMD, as in the 256-row kernel, and the same 32 query rows: w computes S^T, softmax and P of
// the even key blocks, w + 4 of the odd ones, and each runs GEMM 2 and the merge of ALL key blocks, in key order, for half of
// the output columns.  What they exchange is P, 4 KB of LDS per key block.  The two halves of the workgroup work in
// anti-phase: in tick T (between two barriers) the half that owns block T runs the matrix phase
//     M(T) = publish P(T), GEMM 2 + merge of block T-1 (the other half's P) and of block T, GEMM 1 of block T+2
// and the other half the softmax and packing of block T+1.  An M phase has the 32 MFMAs of the 256-row kernel's: two key blocks times half
// the columns in GEMM 2.  The half in its softmax requests K and V of two ticks later and waits for them one phase on; the rings
// hold three K and four V tiles.
#pragma once

namespace fmha_i8_gfx950 {

constexpr int kPairRows = 128;

template <int D, int BK, bool BIAS, bool FASTACC, bool FULLP>
__global__ __launch_bounds__(512, 2) void fmha_i8_pair_kernel(const SplitKernelArgs args) {
  constexpr int kChunks = D / 16;
  constexpr int kTileBytes = BK * D;
  constexpr int kRegions = kTileBytes / 1024;
  constexpr int kLoads = kRegions / 4;  // direct-to-LDS loads per wavefront of one half for one tile
  constexpr int kDSteps = D / 32;
  constexpr int kColTiles = kDSteps / 2;  // output column tiles per wavefront
  constexpr int kKeyTiles = BK / 32;
  constexpr int kStagesK = 3, kStagesV = 4;

  __shared__ __attribute__((aligned(1024))) int8_t lds_k[kStagesK][kTileBytes];
  __shared__ __attribute__((aligned(1024))) int8_t lds_v[kStagesV][kTileBytes];
  __shared__ __attribute__((aligned(16))) v4i lds_p[2][4][kKeyTiles][64];    // [half][row group]: P^T as the B operand of GEMM 2
  __shared__ __attribute__((aligned(16))) float lds_ml[2][4][32][2];         // block maximum and row sum per query
  __shared__ __attribute__((aligned(4))) unsigned char lds_class[kMaxKeyBlocks];
  __shared__ unsigned lds_mask[kMaxKeyBlocks * kBlockKSmall / 32];
  __shared__ __attribute__((aligned(16))) int lds_scan[4];

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int g = lane >> 5;
  const int i32 = lane & 31;
  const int r = wave & 3;   // row group
  const int h = wave >> 2;  // half: owns the blocks of its parity

  int wg;
  {  // XCD-aware placement, as in the 256-row kernel
    const int L = blockIdx.x, per = args.total_wgs / kXcds, rem = args.total_wgs % kXcds, x = L % kXcds;
    wg = x * per + (x < rem ? x : rem) + L / kXcds;
  }
  const int bh_here = divide(wg, args.q_blocks_divisor), bh = bh_here + args.first_head;
  const int qb = wg - bh_here * args.q_blocks;
  const int b = divide(bh, args.head_num_divisor);
  const int S = args.seq_kv;
  const int Sq = args.seq_q;
  const int8_t* __restrict__ kg = args.k + (long)bh * S * D;
  const int8_t* __restrict__ vg = args.v + (long)bh * S * D;
  const int8_t* __restrict__ mg = args.mask + (long)b * S;
  const long q_head_off = (long)bh * Sq * D;
  const int n_blocks = (S + BK - 1) / BK;
  const int tail_kb = S % BK != 0 ? n_blocks - 1 : -1;  // a partly filled last block: its tile ends with the last key

  // ---- tile loads: the four wavefronts of a half fetch a tile, regions r, r + 4, ... ---------------------------------
  const int ld_row_in = lane / kChunks;
  int ld_goff[2];
  {
    const int p = lane % kChunks;
    const int vrow = (D == 128) ? (ld_row_in | ((r & 1) << 3)) : ld_row_in;
    ld_goff[0] = ld_row_in * D + ((p ^ k_swizzle<D>(vrow)) << 4) + r * 1024;
    ld_goff[1] = ld_row_in * D + ((p ^ v_swizzle<D>(vrow)) << 4) + r * 1024;
  }
  const unsigned lds_k_base = (unsigned)(uintptr_t)(__attribute__((address_space(3))) int8_t*)&lds_k[0][0] + r * 1024;
  const unsigned lds_v_base = (unsigned)(uintptr_t)(__attribute__((address_space(3))) int8_t*)&lds_v[0][0] + r * 1024;
  auto issue_at = [&](int which, int tile, unsigned dst) __attribute__((always_inline)) {  // which: 0 = K, 1 = V
    int src = tile + ld_goff[which];
    if (!fmha_in_bounds(src >= 0 && src + 16 <= S * D)) src = 0;
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(dst), "v"(src), "s"(which ? vg : kg) : "memory");
  };
  auto issue = [&](int which, int kb, int stage, int it) __attribute__((always_inline)) {
    issue_at(which, (kb == tail_kb ? (S - BK) * D : kb * kTileBytes) + it * 4096,
             (which ? lds_v_base : lds_k_base) + (unsigned)(stage * kTileBytes + it * 4096));
  };
  auto barrier = [&]() { asm volatile("s_barrier" ::: "memory"); };
  auto all_loads_landed = [&]() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); };
  auto written = [&]() { asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); };

  // ---- prologue: mask bytes (first half), Q rows, K of the first own block; all in flight before the first wait --------
  const int row0 = args.first_row + (qb * 4 + r) * 32;
  const bool active = row0 < Sq;
  v4i mask_bytes, tail_bytes;
  {
    const int mine = kMaskBytesPerLane * (tid & 255);
    int j = mine + kMaskBytesPerLane <= S ? mine : 0, jt = S - kMaskBytesPerLane;
    if (!fmha_in_bounds(j >= 0 && j + kMaskBytesPerLane <= S && jt >= 0)) j = jt = 0;
    asm volatile("global_load_dwordx4 %0, %2, %3\n\tglobal_load_dwordx4 %1, %4, %3"
                 : "=&v"(mask_bytes), "=v"(tail_bytes) : "v"(j), "s"(mg), "v"(jt) : "memory");
  }
  v4i qreg[kDSteps];
  // Q: at head_dim 128 through LDS, by whole rows (see the 256-row kernel; B1 H16 S2048 25.39 -> 24.82 us); the two wavefronts of a row group
  // fetch half of its rows each, into what holds P from tick 0 on: of the first half in blocks of 128 keys, of both halves and of other row
  // groups in blocks of 64.  So every wavefront has its operands before it arrives at its next barrier, two in front of the first P (q_rows_read).
  constexpr bool kQThroughLds = D == 128;
  constexpr int kQLoads = kQThroughLds ? kDSteps / 2 : kDSteps;
  const int8_t* lds_q = reinterpret_cast<const int8_t*>(&lds_p[0][0][0][0]) + r * (32 * D);
  static_assert(!kQThroughLds || 4 * 32 * D <= (int)sizeof(lds_p), "");
  if constexpr (kQThroughLds) {
    const unsigned dst = (unsigned)(uintptr_t)(__attribute__((address_space(3))) const int8_t*)lds_q;
    const int8_t* qp = args.q + q_head_off;
#pragma unroll
    for (int it = 0; it < kQLoads; ++it) {
      const int region = kQLoads * h + it, row = region * (1024 / D) + ld_row_in;
      int qrow = min(row0 + row, Sq - 1);  // rows past the end load the last row (unused)
      if (!fmha_in_bounds(qrow >= 0 && qrow < Sq)) qrow = 0;
      const int src = qrow * D + (((lane % kChunks) ^ k_swizzle<D>(row)) << 4);
      asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2 ; Q, shared 1" ::"s"(dst + 1024u * region), "v"(src), "s"(qp) : "memory");
    }
  } else {
    int qrow = min(row0 + i32, Sq - 1);  // rows past the end load the last row (unused)
    if (!fmha_in_bounds(qrow >= 0 && qrow < Sq)) qrow = 0;
    const int8_t* qp = args.q + q_head_off;
    const int qoff = qrow * D + 16 * g;
#pragma unroll
    for (int kk = 0; kk < kDSteps; ++kk)
      asm volatile("global_load_dwordx4 %0, %1, %2" : "=v"(qreg[kk]) : "v"(qoff + 32 * kk), "s"(qp) : "memory");
  }
  // The first half fetches K(0), the other one K(1), V(0) and K(2), which it waits for behind the first barrier.
#pragma unroll
  for (int it = 0; it < kLoads; ++it) issue(0, min(h, n_blocks - 1), h, it);
  if (h != 0) {
#pragma unroll
    for (int it = 0; it < kLoads; ++it) {
      issue(1, 0, 0, it);
      issue(0, min(2, n_blocks - 1), 2, it);
    }
  }

  // operand addresses (see the 256-row kernel)
  int k_read_off[kDSteps];
#pragma unroll
  for (int kk = 0; kk < kDSteps; ++kk) k_read_off[kk] = i32 * D + (((2 * kk + g) ^ k_swizzle<D>(i32)) << 4);
  int v_read_off[kColTiles];
  {
    const int jin = lane & 15, hh = (lane >> 4) & 1, kslot = jin >> 1;
    const int key_lane = 4 * g + (kslot < 4 ? kslot : kslot + 4);
#pragma unroll
    for (int u = 0; u < kColTiles; ++u)
      v_read_off[u] = key_lane * D + (((2 * (h * kColTiles + u) + hh) ^ v_swizzle<D>(key_lane)) << 4) + 8 * (jin & 1);
  }

  // ---- state -------------------------------------------------------------------------------------------------------
  float o_f[kColTiles][16];
#pragma unroll
  for (int u = 0; u < kColTiles; ++u)
#pragma unroll
    for (int e = 0; e < 16; ++e) o_f[u][e] = 0.f;
  float m_ref = args.floor2 - 2.f * kLazyLog2, t_run = 0.f, l_run = 0.f;
  const float c2 = BIAS ? args.c2 * kBaseScale : args.c2;
  constexpr int kScoreBaseBits = score_base_bits<D>();
  const float bias_c2 = BIAS ? __builtin_bit_cast(float, kScoreBaseBits) * c2 : 0.f;
  v16i base_c, base_s;
#pragma unroll
  for (int e = 0; e < 16; ++e) {
    base_c[e] = FULLP ? 0 : kBaseBits;
    base_s[e] = BIAS ? kScoreBaseBits : 0;
  }
  asm volatile("" : "+v"(base_c));
  if (BIAS && !FULLP && kScoreBaseBits == kBaseBits) base_s = base_c;
  else if (BIAS) asm volatile("" : "+v"(base_s));

  // (the second half, which has 2 kLoads more in flight, waits for its Q rows here, and for the mask bytes in vain)
  static_assert(kQLoads <= 2 * kLoads, "");
  asm volatile("s_waitcnt vmcnt(%2)" : "+v"(mask_bytes), "+v"(tail_bytes) : "n"(kQLoads + kLoads) : "memory");
  if (h == 0) {
    const int live_hi = classify_key_blocks<BK, 4>(mask_bytes, tail_bytes, mg, S, tid, lds_mask, lds_class, 0, n_blocks * BK);
    if (lane == 0) lds_scan[r] = live_hi;
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
  }
  barrier();
  all_loads_landed();
  if (kQThroughLds) asm volatile("; Q from LDS, place reused" ::: "memory");
#pragma unroll
  for (int kk = 0; kk < kDSteps; ++kk) {
    if constexpr (kQThroughLds) qreg[kk] = *reinterpret_cast<const v4i*>(lds_q + k_read_off[kk]);
    else asm volatile("" : "+v"(qreg[kk]));
  }
  const v4i scan = *reinterpret_cast<const v4i*>(lds_scan);
  const int n = __builtin_amdgcn_readfirstlane(max(max(scan[0], scan[1]), max(scan[2], scan[3]))) + 1;  // one past the last block with an unmasked key

  // ---- phases ------------------------------------------------------------------------------------------------------
  v16i acc[kKeyTiles];  // S^T, then the exponentials, of the own block
  int mx[2];
  float m_blk = 0.f, l_blk = 0.f;
  auto tile_max_piece = [&](const v16i& a, int j) __attribute__((always_inline)) {
    mx[0] = max(max(mx[0], a[2 * j]), a[2 * j + 1]);
    mx[1] = max(max(mx[1], a[8 + 2 * j]), a[9 + 2 * j]);
  };
  // GEMM 1: operand reads run two key tiles ahead of the MFMAs, the first two are issued inside GEMM 2 (read_first); the row
  // maximum of a tile is taken behind the MFMAs of the next one.
  v4i ka[3][kDSteps];
  auto read_k = [&](int stage, int t) __attribute__((always_inline)) {
#pragma unroll
    for (int kk = 0; kk < kDSteps; ++kk) ka[t % 3][kk] = *reinterpret_cast<const v4i*>(&lds_k[stage][0] + k_read_off[kk] + 32 * t * D);
  };
  auto read_first = [&](int stage) __attribute__((always_inline)) {
    read_k(stage, 0);
    read_k(stage, 1);
  };
  auto gemm1 = [&](int kb, int stage, auto masked_t) __attribute__((always_inline)) {
    constexpr bool kMasked = decltype(masked_t)::value;
    unsigned mw[kKeyTiles];
    if constexpr (kMasked) {
      mask_words_of<BK>(mw, lds_mask, kb, tail_kb, S);
      acc[0] = masked_start(mw[0], MaskedUnits<BIAS>(), base_s);
    }
    mx[0] = mx[1] = (int)0x80000000;
#pragma unroll
    for (int t = 0; t < kKeyTiles; ++t) {
      if (t + 2 < kKeyTiles) read_k(stage, t + 2);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int kk = 0; kk < kDSteps; ++kk) {
        acc[t] = __builtin_amdgcn_mfma_i32_32x32x32_i8(ka[t % 3][kk], qreg[kk], (kk == 0 && !kMasked) ? base_s : acc[t], 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (kMasked)
          if (kk == kDSteps - 2 && t + 1 < kKeyTiles) {
            acc[t + 1] = masked_start(mw[t + 1], MaskedUnits<BIAS>(), base_s);
            __builtin_amdgcn_sched_barrier(0);
          }
        if (t >= 1) {
#pragma unroll
          for (int j = kk * 4 / kDSteps; j < (kk + 1) * 4 / kDSteps; ++j) tile_max_piece(acc[t - 1], j);
          asm volatile("" : "+v"(mx[0]), "+v"(mx[1]));  // keeps these in the shadow of the MFMA
          __builtin_amdgcn_sched_barrier(0);
        }
      }
    }
  };
  // The block softmax in three dense runs, the last of them with the packing of P.
  v4i pk[kKeyTiles];  // P^T of the own block
  auto softmax = [&](int cls, auto between) __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < 4; ++j) tile_max_piece(acc[kKeyTiles - 1], j);
    int ti = half_max(max(mx[0], mx[1]));
    if (cls != 0) ti = max(ti, (BIAS ? kScoreBaseBits : 0) - 1000000);  // the reference's sentinel (inc/fmha_i8.cuh:191-193)
    const float top = BIAS ? __int_as_float(ti) : (float)ti;
    float off = top * c2;
    if (!BIAS) off = __builtin_fmaf(fabsf(off), 2.384185791015625e-07f, off);
    if (!BIAS) off = fmaxf(off, args.floor2);
    m_blk = off - bias_c2;
    const float offq = off - (FULLP ? kLog2PscaleFull : kLog2Pscale);
    constexpr int kQuads = 4 * kKeyTiles;
    float x[kQuads][4];
#pragma unroll
    for (int qd = 0; qd < kQuads; ++qd)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int s = acc[qd / 4][4 * (qd % 4) + j];
        x[qd][j] = __builtin_fmaf(BIAS ? __int_as_float(s) : (float)s, c2, -offq);
      }
#pragma unroll
    for (int qd = 0; qd < kQuads; ++qd) asm volatile("" : "+v"(x[qd][0]), "+v"(x[qd][1]), "+v"(x[qd][2]), "+v"(x[qd][3]));
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int qd = 0; qd < kQuads; ++qd) {
#pragma unroll
      for (int j = 0; j < 4; ++j) x[qd][j] = __builtin_amdgcn_exp2f(x[qd][j]);
      asm volatile("" : "+v"(x[qd][0]), "+v"(x[qd][1]), "+v"(x[qd][2]), "+v"(x[qd][3]));
      between(qd, kQuads);
    }
    __builtin_amdgcn_sched_barrier(0);
    l_blk = 0.f;
#pragma unroll
    for (int qd = 0; qd < kQuads; ++qd) {
      const float(&e)[4] = x[qd];
      float s01 = e[0] + e[1];
      const float s23 = e[2] + e[3];
      s01 += s23;
      l_blk += s01;
      const v2s lo = FULLP ? __builtin_amdgcn_cvt_pknorm_i16(e[0], e[1]) : __builtin_amdgcn_cvt_pknorm_i16(-e[0], -e[1]);
      const v2s hi = FULLP ? __builtin_amdgcn_cvt_pknorm_i16(e[2], e[3]) : __builtin_amdgcn_cvt_pknorm_i16(-e[2], -e[3]);
      const int four = __builtin_amdgcn_perm(__builtin_bit_cast(int, hi), __builtin_bit_cast(int, lo), 0x06040200);
      pk[qd / 4][qd % 4] = FULLP ? four ^ (int)0x80808080 : four;
    }
    l_blk = half_sum(l_blk);
    // all of it stays in front of the barrier
#pragma unroll
    for (int t = 0; t < kKeyTiles; ++t) asm volatile("" : "+v"(pk[t]));
    asm volatile("" : "+v"(l_blk), "+v"(m_blk));
  };
  auto publish = [&]() __attribute__((always_inline)) {
    lds_ml[h][r][i32][0] = m_blk;
    lds_ml[h][r][i32][1] = l_blk;
#pragma unroll
    for (int t = 0; t < kKeyTiles; ++t) lds_p[h][r][t][lane] = pk[t];
  };
  int stage_k = h;  // of the next own block, T + 2 in M(T): (T + 2) mod 3
  // GEMM 2 and merge of block T-1 (the other half's P) and T (own P) for this wavefront's columns.  A block that is not there
  // or has no unmasked key enters with weight 0 (its P may be anything: any int8 leaves the accumulators finite).
  constexpr int kSteps = 2 * kColTiles;
  v4i va[2][kKeyTiles];
  auto read_v = [&](int T, int s, int t) __attribute__((always_inline)) {
    typedef v2i __attribute__((address_space(3))) * lds_v2i_ptr;
    const int8_t* tile = &lds_v[(T - 1 + s / kColTiles) & (kStagesV - 1)][0];
    const v2i lo = __builtin_amdgcn_ds_read_tr8_b64_v2i32((lds_v2i_ptr)(tile + v_read_off[s % kColTiles] + 32 * t * D));
    const v2i hi = __builtin_amdgcn_ds_read_tr8_b64_v2i32((lds_v2i_ptr)(tile + v_read_off[s % kColTiles] + 32 * t * D + 16 * D));
    va[s & 1][t] = v4i{lo[0], lo[1], hi[0], hi[1]};
  };
  auto gemm2_merge = [&](int T, bool live0, bool live1) __attribute__((always_inline)) {
    // Products s = 0 .. kSteps-1: block T-1 and block T, column tile by column tile; an operand is replaced by that of the
    // product two further on as soon as its MFMA has been issued, a product is merged behind the MFMAs of the next one.
    v4i other[kKeyTiles];
    v16i oacc[2];
    const float mb0 = lds_ml[1 - h][r][i32][0], lb0 = lds_ml[1 - h][r][i32][1];
#pragma unroll
    for (int t = 0; t < kKeyTiles; ++t) {
      other[t] = lds_p[1 - h][r][t][lane];
      read_v(T, 0, t);
      read_v(T, 1, t);
    }
    __builtin_amdgcn_sched_barrier(0);
    auto start = [&](int s) __attribute__((always_inline)) {
      oacc[s & 1] = base_c;
      if (FULLP) {  // 128 times the column sums of the tile: a product with 64s, doubled (see the split kernel)
        const v4i half = {0x40404040, 0x40404040, 0x40404040, 0x40404040};
#pragma unroll
        for (int t = 0; t < kKeyTiles; ++t) oacc[s & 1] = __builtin_amdgcn_mfma_i32_32x32x32_i8(va[s & 1][t], half, oacc[s & 1], 0, 0, 0);
#pragma unroll
        for (int e = 0; e < 16; ++e) oacc[s & 1][e] = 2 * oacc[s & 1][e] + kBaseBitsFull;
      }
    };
    auto product = [&](int s, int t) __attribute__((always_inline)) {
      oacc[s & 1] = __builtin_amdgcn_mfma_i32_32x32x32_i8(va[s & 1][t], s < kColTiles ? other[t] : pk[t], oacc[s & 1], 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
      if (s + 2 < kSteps) read_v(T, s + 2, t);
    };
    start(0);
#pragma unroll
    for (int t = 0; t < kKeyTiles; ++t) product(0, t);
    float take[2], keep[2];
    bool moves[2];  // some row's reference exponent moves (wave-uniform, rare): O is rescaled in front of that block's merge
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const bool live = j ? live1 : live0;
      const float mb = live ? (j ? m_blk : mb0) : -__builtin_inff(), lb = live ? (j ? l_blk : lb0) : 0.f;
      moves[j] = __ballot(mb > m_ref + kLazyLog2) != 0;
      const float m_new = moves[j] ? fmaxf(m_ref, mb) : m_ref;
      keep[j] = __builtin_amdgcn_exp2f(m_ref - m_new);  // exactly 1 where nothing moves
      m_ref = m_new;
      take[j] = __builtin_amdgcn_exp2f(mb - m_ref);
      l_run = __builtin_fmaf(take[j], lb, l_run * keep[j]);
      if (FASTACC) t_run = t_run * keep[j] + take[j];
      if (!FULLP) take[j] = -take[j];  // P carries the sign
      asm volatile("" : "+v"(take[j]));
    }
    auto rescale = [&](int j) __attribute__((always_inline)) {
      if (moves[j]) {
#pragma unroll
        for (int u = 0; u < kColTiles; ++u)
#pragma unroll
          for (int e = 0; e < 16; ++e) o_f[u][e] *= keep[j];
      }
    };
    auto merge_piece = [&](int s, int piece, int pieces) __attribute__((always_inline)) {
#pragma unroll
      for (int e = 16 * piece / pieces; e < 16 * (piece + 1) / pieces; ++e) {
        const float v = FASTACC ? __int_as_float(oacc[s & 1][e]) : __int_as_float(oacc[s & 1][e]) - (FULLP ? kBaseFull : kBase);
        o_f[s % kColTiles][e] = __builtin_fmaf(take[s / kColTiles], v, o_f[s % kColTiles][e]);
      }
    };
    rescale(0);
#pragma unroll
    for (int s = 1; s < kSteps; ++s) {
      start(s);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int t = 0; t < kKeyTiles; ++t) {
        product(s, t);
        merge_piece(s - 1, t, kKeyTiles);
        __builtin_amdgcn_sched_barrier(0);
      }
      if (s == kColTiles) rescale(1);
      if (s + 1 == kSteps) read_first(stage_k);
      __builtin_amdgcn_sched_barrier(0);
    }
    merge_piece(kSteps - 1, 0, 1);
  };

  // ---- the schedule ------------------------------------------------------------------------------------------------
  auto cls_of = [&](int kb) { return kb < n ? __builtin_amdgcn_readfirstlane((int)lds_class[kb]) : 2; };
  auto raise_priority = [&]() { asm volatile("s_setprio 3" ::: "memory"); };
  auto drop_priority = [&]() { asm volatile("s_setprio 0" ::: "memory"); };
  auto forget_scores = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int t = 0; t < kKeyTiles; ++t) asm volatile("" : "=v"(acc[t]));
    asm volatile("" : "=v"(mx[0]), "=v"(mx[1]));
  };
  auto gemm1_of = [&](int kb, int cls) __attribute__((always_inline)) {
    if (cls & 2) forget_scores();
    else if (cls & 1) gemm1(kb, stage_k, Const<1>{});
    else gemm1(kb, stage_k, Const<0>{});
    return cls;
  };
  // What the softmax of block T asks for in tick T-1: K(T+3) and V(T+1), the other half's in tick T+1; waited for at the end of
  // M(T).  Their stages held K(T), read in tick T-2, and V(T-3), read last in tick T-2.
  int next_tile[2];    // offsets in K and V
  unsigned next_lds[2];
  bool next_wanted[2];
  auto next_loads = [&](int T) __attribute__((always_inline)) {
#pragma unroll
    for (int which = 0; which < 2; ++which) {
      const int kb = which ? T + 1 : T + 3;
      next_wanted[which] = kb < n;
      next_tile[which] = kb == tail_kb ? (S - BK) * D : kb * kTileBytes;
      next_lds[which] = which ? lds_v_base + ((T + 1) & (kStagesV - 1)) * kTileBytes : lds_k_base + stage_k * kTileBytes;  // (stage_k = T mod 3)
    }
  };
  auto some_loads = [&](int slot, int slots) __attribute__((always_inline)) {  // in pairs where a wavefront has several
    constexpr int kGroup = kLoads >= 2 ? 2 : 1, kGroups = kLoads / kGroup;
#pragma unroll
    for (int group = slot * 2 * kGroups / slots; group < (slot + 1) * 2 * kGroups / slots; ++group) {
      const int which = group / kGroups;
      if (next_wanted[which]) {
#pragma unroll
        for (int it = group % kGroups * kGroup; it < (group % kGroups + 1) * kGroup; ++it)
          issue_at(which, next_tile[which] + it * 4096, next_lds[which] + it * 4096);
      }
    }
  };
  // (the compiler puts the reads of Q behind the one of the scan: nothing else waits for them in front of these barriers)
  auto q_rows_read = [&]() { if (kQThroughLds) asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); };
  if (n > 0) {
    if (h != 0) {
      q_rows_read();
      barrier();  // tick -2 is the first half's: GEMM 1 of block 0
    }
    read_first(stage_k);
    int cls = active ? cls_of(h) : 2;  // of the own block whose scores are in acc
    q_rows_read();
    gemm1_of(h, cls);
    int T = h;
    for (; T <= n; T += 2) {
      barrier();  // tick T-1
      const bool own = !(cls & 2);
      next_loads(T);
      if (own) softmax(cls, some_loads);
      else some_loads(0, 1);
      barrier();  // tick T
      raise_priority();
      const bool before_live = T > 0 && !(cls_of(T - 1) & 2);
      const int cls_next = active ? cls_of(T + 2) : 2;
      if (own) publish();
      stage_k = stage_k == 0 ? 2 : stage_k - 1;  // (T + 2) mod 3
      if (active) gemm2_merge(T, before_live, own);
      cls = gemm1_of(T + 2, cls_next);
      written();
      all_loads_landed();
      drop_priority();
    }
    if (T - 2 < n) barrier();  // the other half's last tick
  }
  all_loads_landed();  // nothing may still be writing LDS when the wavefront ends
  if (!active) return;

  // ---- epilogue (see the 256-row kernel) -----------------------------------------------------------------------------
  const float fin = (l_run > 0.f) ? args.out_scale * (128.f / kSnorm) * kBaseScale / l_run : 0.f;
  const float corr = FASTACC ? (FULLP ? -kBaseFull * t_run : kBase * t_run) : 0.f;
  int w[kColTiles][4];
#pragma unroll
  for (int u = 0; u < kColTiles; ++u)
#pragma unroll
    for (int a = 0; a < 4; ++a) {
      float y[4];
#pragma unroll
      for (int bb = 0; bb < 4; ++bb)
        y[bb] = __builtin_amdgcn_fmed3f(__builtin_fmaf(FASTACC ? o_f[u][4 * a + bb] + corr : o_f[u][4 * a + bb], fin, kMagic),
                                        kMagic - 127.f, kMagic + 127.f);
      const int lo = __builtin_amdgcn_perm(__float_as_int(y[1]), __float_as_int(y[0]), 0x0c0c0400);
      const int hi = __builtin_amdgcn_perm(__float_as_int(y[3]), __float_as_int(y[2]), 0x0c0c0400);
      w[u][a] = __builtin_amdgcn_perm(hi, lo, 0x05040100);
    }
  const bool mine = row0 + i32 < Sq && fmha_in_bounds(row0 + i32 >= 0 && q_head_off + (long)(row0 + i32 + 1) * D <= ((long)args.total_wgs / args.q_blocks + args.first_head) * Sq * D);
  if (kColTiles == 1 && !mine) return;
  int8_t* op = args.o + q_head_off + (long)(row0 + i32) * D + 32 * kColTiles * h;
  if constexpr (kColTiles == 2) {  // 32 contiguous bytes per lane
    op += 32 * g;
    int g0[4], g1[4];
#pragma unroll
    for (int a = 0; a < 4; ++a) {
      const auto s = __builtin_amdgcn_permlane32_swap(w[0][a], w[1][a], false, false);
      g0[a] = s[0];
      g1[a] = s[1];
    }
    if (mine) {
      *reinterpret_cast<v4i*>(op) = v4i{g0[0], g1[0], g0[1], g1[1]};
      *reinterpret_cast<v4i*>(op + 16) = v4i{g0[2], g1[2], g0[3], g1[3]};
    }
    if (args.wide == nullptr) return;
    barrier();  // (as in the 256-row kernel; both halves have passed as many)
    const int both[8] = {g0[0], g1[0], g0[1], g1[1], g0[2], g1[2], g0[3], g1[3]};
    store_wide_rows<D>(args, &lds_v[0][0] + wave * 4096, q_head_off + (long)row0 * D + 64 * h, Sq - row0, both);
  } else {
    op += 16 * g;  // (one store of sixteen bytes per lane, as in the split kernel)
    const auto s0 = __builtin_amdgcn_permlane32_swap(w[0][0], w[0][2], false, false), s1 = __builtin_amdgcn_permlane32_swap(w[0][1], w[0][3], false, false);
    const int both[4] = {(int)s0[0], (int)s0[1], (int)s1[0], (int)s1[1]};
    *reinterpret_cast<v4i*>(op) = v4i{both[0], both[1], both[2], both[3]};
    store_wide<D>(args, op - args.o, both);
  }
}

}  // namespace fmha_i8_gfx950
