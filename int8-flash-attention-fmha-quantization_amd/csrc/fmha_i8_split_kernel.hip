// The attention kernel for calls that fill too few compute units with workgroups of 256 query rows: a handful of heads, a
// chunk of a prefill, one new row per sequence.  Same arithmetic as fmha_i8_fwd_kernel (fmha_i8_kernel.hip) and the same
// BYTES for every row: which kernel serves a call (row_groups_of, part_plan_of) is a question of speed alone.
//
// A workgroup owns R groups of 32 query rows (R = 1 or 2) of one head and works on FOUR key blocks at a time, a "round":
//   * wavefront (r, c) computes S^T, the block softmax and the quantised P^T of row group r and key block 4 i + c, so the
//     part that bounds the attention kernel - the vector instructions of the softmax - is spread over four times as many
//     wavefronts as there are row groups;
//   * P^T goes through LDS to the four wavefronts of the row group, a quarter of what exchanging O would take, and each
//     of them runs GEMM 2 and the online merge of all four key blocks, in key order, for ITS 32 output columns.  Every
//     output element is thus merged by one wavefront, block after block, with the operations of the 256-row kernel in the
//     same order - which no scheme that merges partial results of separate key ranges can do, since float addition is not
//     associative.  (At head_dim 64 there are two column tiles: two wavefronts do each.)
// K and V tiles go HBM -> LDS directly, as in the 256-row kernel and with the same swizzles.  A call has more than one key
// block (the host sees to it): a single one leaves three quarters of the wavefronts without a softmax.
#pragma once

namespace fmha_i8_gfx950 {

typedef float v2f __attribute__((ext_vector_type(2)));

constexpr int kSplitKeys = 4;  // key blocks of a round

template <int N>
struct Const {  // a constant as a function argument
  static constexpr int value = N;
};

// Division of a non-negative int by a divisor known on the host: a multiplication and two shifts where the division takes
// some thirty instructions that everything in the prologue waits for (Granlund and Montgomery, 1994).
struct Divisor {
  unsigned factor;
  int shift;  // of a divisor d > 1: ceil(log2 d) - 1; -1 for d = 1
};
inline Divisor make_divisor(int d) {
  int bits = 0;
  while ((1ll << bits) < d) ++bits;
  if (bits == 0) return {0u, -1};
  return {(unsigned)((((1ull << bits) - (unsigned)d) << 32) / (unsigned)d + 1), bits - 1};
}
__device__ __forceinline__ int divide(int n, Divisor d) {
  if (d.shift < 0) return n;
  const unsigned t = __umulhi(d.factor, (unsigned)n);
  return (int)((t + (((unsigned)n - t) >> 1)) >> d.shift);
}

struct SplitKernelArgs : KernelArgs {
  Divisor q_blocks_divisor, head_num_divisor;
  // Calls of few query rows whose key blocks are shared out (PARTS): rounds per workgroup, and where its results go.
  int rounds_per_part;
  v2f* part_ml;  // [head][key block][row]: block maximum and row sum
  int* part_o;   // [head][key block][head_dim / 4][row][4]: the accumulators of GEMM 2
};

// Classification of the key blocks of a batch entry by the first WAVES wavefronts of a workgroup, sixteen mask bytes per lane
// (the bits are those of fmha_i8_fwd_kernel): mask bits to `words`, per block bit0 = some key masked, bit1 = all keys masked to
// `cls` (blocks that fill up the last four count as the latter).  mask_bytes: the lane's first sixteen bytes, tail_bytes: the
// row's last sixteen (for the one lane that straddles the end); both have landed.  S >= 16.  Returns this wavefront's last
// block with an unmasked key, -1 if there is none.  Only keys from .. to-1 are looked at (multiples of BK).
// What bounds it is a chain of latencies in front of the first barrier: wavefronts whose sixteen bytes per lane lie behind the last key
// have nothing to do here, the neighbour's bits come by a lane permutation of the vector unit and the last live block from a ballot.
// With LDS permutations (seven in a row) and all wavefronts at it: B2 H8 S300 d128 6.76 -> 7.20 us, H16 Sq512 S640 8.92 -> 9.33, d64 B2 H12
// S1024 (pair kernel) 13.14 -> 13.44, B8 H16 Sq1 S2048 (sixteen rows) 8.99 -> 9.34.
constexpr int kMaskBytesPerLane = 16;
template <int BK, int WAVES>
__device__ __forceinline__ int classify_key_blocks(const v4i& mask_bytes, const v4i& tail_bytes, const int8_t* __restrict__ mg, int S,
                                                   int tid, unsigned* words, unsigned char* cls, int from, int to) {
  constexpr int kLanesPerBlock = BK / kMaskBytesPerLane;
  const int lane = tid & 63, n_blocks = (S + BK - 1) / BK;
  auto nonzero_bytes = [](unsigned w) -> unsigned {
    const unsigned t = (((w & 0x7f7f7f7fu) + 0x7f7f7f7fu) | w) & 0x80808080u;
    return (((t >> 7) * 0x00204081u) >> 21) & 15u;
  };
  auto nonzero16 = [&](const v4i& w) -> unsigned {
    return nonzero_bytes((unsigned)w[0]) | (nonzero_bytes((unsigned)w[1]) << 4) | (nonzero_bytes((unsigned)w[2]) << 8) |
           (nonzero_bytes((unsigned)w[3]) << 12);
  };
  const int first_lane = __builtin_amdgcn_readfirstlane(tid - lane);
  int live_hi = -1;
  auto pass = [&](int base, const v4i& w) __attribute__((always_inline)) {
    const int j = base + kMaskBytesPerLane * tid;
    unsigned bits = 0xffffu;  // keys past the end count as masked
    if (j + kMaskBytesPerLane <= S)
      bits = nonzero16(w);
    else if (j < S)  // the one lane that straddles the end of the row
      bits = ((nonzero16(tail_bytes) >> (kMaskBytesPerLane - (S - j))) | (0xffffu << (S - j))) & 0xffffu;
    // (the neighbour's sixteen bits by a lane permutation of the vector unit)
    const unsigned word = bits | ((unsigned)__builtin_amdgcn_mov_dpp((int)bits, 0xB1, 0xf, 0xf, true) << 16);
    if ((lane & 1) == 0 && j < to) words[j >> 5] = word;
    const unsigned long long some = __ballot(bits != 0), all = __ballot(bits == 0xffffu);
    bool lives = false;
    if (lane % kLanesPerBlock == 0 && j < to) {
      constexpr unsigned long long kBlockBits = (1ull << kLanesPerBlock) - 1;
      const bool blk_some = ((some >> lane) & kBlockBits) != 0, blk_all = ((all >> lane) & kBlockBits) == kBlockBits;
      cls[j / BK] = (unsigned char)((blk_some ? 1 : 0) | (blk_all ? 2 : 0));
      lives = !blk_all;
    }
    const unsigned long long live = __ballot(lives);
    if (live != 0) live_hi = (base + kMaskBytesPerLane * (first_lane + 63 - __builtin_clzll(live))) / BK;
  };
  if (from + kMaskBytesPerLane * first_lane < to) pass(from, mask_bytes);
  // Longer rows, out of the way of the others (B8 H16 Sq1 S2048 d128 14.10 -> 14.00 us, H16 Sq512 S512 5.90 -> 5.82 against one loop for
  // all, elsewhere within 1 % either way): two passes at a time, two loads behind one wait (H4 Sq512 S16300 scattered 114.8 -> 113.8).
  constexpr int kKeysPerPass = kMaskBytesPerLane * 64 * WAVES;
  for (int base = from + kKeysPerPass; base + kMaskBytesPerLane * first_lane < to; base += 2 * kKeysPerPass) {
    const int j = base + kMaskBytesPerLane * tid;
    int j0 = j + kMaskBytesPerLane <= S ? j : 0, j1 = j + kKeysPerPass + kMaskBytesPerLane <= S ? j + kKeysPerPass : 0;
    if (!fmha_in_bounds(j0 >= 0 && j0 + kMaskBytesPerLane <= S && j1 >= 0 && j1 + kMaskBytesPerLane <= S)) j0 = j1 = 0;
    v4i w0, w1;
    asm volatile("global_load_dwordx4 %0, %2, %4\n\tglobal_load_dwordx4 %1, %3, %4\n\ts_waitcnt vmcnt(0)"
                 : "=&v"(w0), "=&v"(w1) : "v"(j0), "v"(j1), "s"(mg) : "memory");
    pass(base, w0);
    if (base + kKeysPerPass + kMaskBytesPerLane * first_lane < to) pass(base + kKeysPerPass, w1);
  }
  if (tid < kSplitKeys && n_blocks + tid < (n_blocks + kSplitKeys - 1) / kSplitKeys * kSplitKeys) cls[n_blocks + tid] = 3;
  return live_hi;
}

// The mask bits of block kb; tail_kb: the partly filled last block, whose tile ends with the last key - bit j of word t is key
// S - BK + 32 t + j, the keys it repeats count as masked.
template <int BK>
__device__ __forceinline__ void mask_words_of(unsigned (&mw)[BK / 32], const unsigned* words, int kb, int tail_kb, int S) {
#pragma unroll
  for (int t = 0; t < BK / 32; ++t) mw[t] = (unsigned)__builtin_amdgcn_readfirstlane((int)words[kb * (BK / 32) + t]);
  if (kb != tail_kb) return;
  const int repeated = (tail_kb + 1) * BK - S;
#pragma unroll
  for (int t = 0; t < BK / 32; ++t) {
    const int start = S - BK + 32 * t, w = start >> 5, sh = start & 31;
    const unsigned lo = (unsigned)__builtin_amdgcn_readfirstlane((int)words[w]);
    const unsigned hi = (unsigned)__builtin_amdgcn_readfirstlane((int)words[w + (sh ? 1 : 0)]);
    unsigned word = sh ? (lo >> sh) | (hi << (32 - sh)) : lo;
    const int forced = repeated - 32 * t;
    if (forced >= 32) word = 0xffffffffu;
    else if (forced > 0) word |= (1u << forced) - 1u;
    mw[t] = word;
  }
}

template <int D, int BK, bool BIAS, bool FASTACC, bool FULLP, int R, bool PARTS = false>
__global__ __launch_bounds__(256 * R, R) void fmha_i8_split_kernel(const SplitKernelArgs args) {
  constexpr int kChunks = D / 16;
  constexpr int kTileBytes = BK * D;
  constexpr int kRowWaves = 4 * R;
  constexpr int kRegions = kTileBytes / 1024;
  constexpr int kLoads = kSplitKeys * kRegions / kRowWaves;  // direct-to-LDS loads per wavefront for four K (or V) tiles
  constexpr int kRowsPerRegion = 1024 / D;
  constexpr int kDSteps = D / 32;
  constexpr int kKeyTiles = BK / 32;
  // LDS holds 160 KB: tiles of 8 KB and less are double buffered, unless own K tiles (below) do better: with one row group and
  // blocks of 64 keys H16 Sq512 S576 d128 8.56 -> 8.37 us, H32 Sq200 S960 10.15 -> 10.02, H16 Sq400 S320 d64 5.96 -> 5.90, and at d64 three
  // workgroups fit a CU (H16 Sq777 S777 in 400 of them 16.9 -> 10.9); with blocks of 128 keys, d64, H16 Sq256 S1024 7.54 -> 7.70.
  // Beside 128 KB of tiles there is room for 16 KB of P: all of a round, or, for two row groups and blocks of 128 keys, half of it,
  // which then goes through in two steps.
  constexpr int kBuffers = kTileBytes <= 8192 && !(R == 1 && BK == 64 && !PARTS) ? 2 : 1;
  constexpr bool kTwoSteps = BK == 128 && R == 2;
  constexpr int kPSlots = kTwoSteps ? 2 : 4;
  // With one row group a K tile has one reader: the wavefront fetches it itself, waits for it itself, and asks for the next
  // one as soon as it has read this one's operands, without any barrier.
  constexpr bool kOwnK = kBuffers == 1 && R == 1;
  // PARTS: a workgroup does some rounds of a head and leaves what the merge needs of every key block (see the end of the
  // file).  With one round or two per workgroup the time is that of the first loads, so V is asked for beside K.
  static_assert(!PARTS || R == 1, "");
  constexpr bool kEarlyV = PARTS && kOwnK;
  // P of a wavefront's own key block, an operand of its own GEMM 2 too, need not come back from LDS: H16 Sq512 S960 d64 8.50 -> 8.39 us, B2 H16
  // Sq100 S576 d128 7.86 -> 7.65, with 255 steps H16 Sq512 S960 d64 9.68 -> 9.38, Sq256 S1984 16.6 -> 16.1, short ones level.  The other forms lose more by the branch in the middle of their operand reads than the reads cost (H16 S777 d128
  // 11.30 -> 11.50, H32 Sq512 S4096 31.3 -> 31.8, d64 S2048 11.47 -> 11.79).
  constexpr bool kOwnP = R == 1 && BK == 64 && !PARTS;
  // Q: the operands of GEMM 1 straight from memory touch 32 rows with every load, and the four wavefronts of a row group load the same
  // ones: the first barrier waits for the CU's address path.  Through LDS eight lanes fetch a row's 128 contiguous bytes: with two
  // buffers a quarter of the rows per wavefront, into what holds V of round 1 from the second barrier on; otherwise each wavefront all
  // of them, into a place that it has read again before the first barrier.  d128 H16 S777 12.12 -> 11.50 us (11.71 with each wavefront
  // fetching all of its rows), H32 Sq512 S1152 13.34 -> 12.82, S4096 32.1 -> 31.5, B2 H16 Sq32 S2048 12.6 -> 12.3; with one row group and
  // blocks of 64 keys B2 H8 S300 6.41 -> 6.47, at d64, where 128 bytes hold two rows, 8.46 -> 8.49 (H16 Sq512 S960): those stay.
  constexpr bool kQInRegs = D == 64 || (R == 1 && BK == 64), kQShared = !kQInRegs && kBuffers == 2;
  constexpr int kQLoads = kQShared ? 1 : D / 32;

  __shared__ __attribute__((aligned(1024))) int8_t lds[kBuffers][2][kSplitKeys][kTileBytes];  // [buffer][K|V][slot][tile]
  __shared__ __attribute__((aligned(16))) v4i lds_p[R][kPSlots][kKeyTiles][64];  // P^T as the B operand of GEMM 2
  __shared__ __attribute__((aligned(16))) float lds_ml[R][kSplitKeys][32][2];    // block maximum and row sum per query
  __shared__ unsigned lds_class4[kMaxKeyBlocks / 4];  // byte j: bit0 = block has a masked key, bit1 = all its keys are
  __shared__ unsigned lds_mask[kMaxKeyBlocks * kBlockKSmall / 32];
  __shared__ int lds_scan[kRowWaves];

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int g = lane >> 5;
  const int i32 = lane & 31;
  const int c = wave & 3;   // key block of the round
  const int r = wave >> 2;  // row group
  const int u_out = c & (kDSteps - 1);  // output column tile of this wavefront

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
  const int first_round = PARTS ? qb * args.rounds_per_part : 0;
  // A partly filled last block: the tile is fetched so that it ends with the last key (see the 256-row kernel).
  const int tail_kb = S % BK != 0 ? n_blocks - 1 : -1;

  // ---- tile loads --------------------------------------------------------------------------------------------------
  // A load moves 1 KiB: lane l lands at byte 16 l of a region of the tile and fetches the chunk that the swizzle assigns to
  // that place.  Addresses are 32-bit offsets inside the head.
  const int ld_row_in = lane / kChunks;
  const int region_of_wave = kRegions >= kRowWaves ? wave : wave % kRegions;  // of the loads that the wavefronts share
  int ld_k, ld_k_odd = 0, ld_v;
  {
    const int p = lane % kChunks;
    const int vrow = (D == 128) ? (ld_row_in | ((wave & 1) << 3)) : ld_row_in;
    ld_k = ld_row_in * D + ((p ^ k_swizzle<D>(kOwnK ? ld_row_in : vrow)) << 4) + (kOwnK ? 0 : region_of_wave * 1024);
    if (kOwnK) ld_k_odd = ld_row_in * D + ((p ^ k_swizzle<D>(ld_row_in + kRowsPerRegion)) << 4);
    ld_v = ld_row_in * D + ((p ^ v_swizzle<D>(vrow)) << 4) + region_of_wave * 1024;
  }
  const unsigned lds_base = (unsigned)(uintptr_t)(__attribute__((address_space(3))) int8_t*)&lds[0][0][0][0];
  const unsigned lds_of_wave = lds_base + (unsigned)(region_of_wave * 1024);
  // Load number `it` of this wavefront's kLoads for the four K (which = 0) or V (which = 1) tiles of a round.  A block past
  // the last one (`last`) is replaced by it: the wait counts below are constants.
  auto issue = [&](int round, int which, int it, int last) __attribute__((always_inline)) {
    const bool own = kOwnK && which == 0;
    const int slot = own ? c : kRegions >= kRowWaves ? it * kRowWaves / kRegions : (it * kRowWaves + wave) / kRegions;
    const int region = own ? it : kRegions >= kRowWaves ? it * kRowWaves % kRegions : 0;  // besides region_of_wave
    const int kb = min(kSplitKeys * round + slot, last);
    const int tile = (kb == tail_kb ? (S - BK) * D : kb * kTileBytes) + region * 1024;
    const unsigned dst = (own ? lds_base : lds_of_wave) +
                         (unsigned)((((round & (kBuffers - 1)) * 2 + which) * kSplitKeys + slot) * kTileBytes + region * 1024);
    int src = tile + (which ? ld_v : own && (it & 1) ? ld_k_odd : ld_k);
    if (!fmha_in_bounds(src >= 0 && src + 16 <= S * D)) src = 0;
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(dst), "v"(src), "s"(which ? vg : kg) : "memory");
  };
  auto barrier = [&]() { asm volatile("s_barrier" ::: "memory"); };
  auto wait_loads = [&](auto outstanding) { asm volatile("s_waitcnt vmcnt(%0)" ::"n"(decltype(outstanding)::value) : "memory"); };

  const Const<0> none;
  const Const<kLoads> one_kind;
  const Const<kLoads / 2> half_kind;

  // ---- prologue: mask bytes, Q rows and K of round 0, in this order; every load in flight before the first wait ---------
  const int row0 = PARTS ? 0 : args.first_row + (qb * R + r) * 32;
  const bool active = row0 < Sq;
  // Keys to classify: all, or those of the rounds of this workgroup and the block in front of them (part of which a partly
  // filled last block's tile repeats).
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
  v4i qreg[kDSteps];
  const int8_t* qp = args.q + q_head_off;
  const int8_t* lds_q = nullptr;
  if constexpr (kQInRegs) {
    int qrow = min(row0 + i32, Sq - 1);  // rows past the end load the last row (unused)
    if (!fmha_in_bounds(qrow >= 0 && qrow < Sq)) qrow = 0;
    const int qoff = qrow * D + 16 * g;
#pragma unroll
    for (int kk = 0; kk < kDSteps; ++kk)
      asm volatile("global_load_dwordx4 %0, %1, %2" : "=v"(qreg[kk]) : "v"(qoff + 32 * kk), "s"(qp) : "memory");
  } else {
    lds_q = kQShared ? &lds[kBuffers - 1][1][0][0] + r * (32 * D) : kEarlyV ? reinterpret_cast<const int8_t*>(&lds_p[r][c][0][0]) : &lds[0][1][0][0] + wave * (32 * D);
    static_assert(kEarlyV ? 32 * D <= kKeyTiles * 1024 : kRowWaves * 32 * D <= kSplitKeys * kTileBytes, "");
    const unsigned dst = (unsigned)(uintptr_t)(__attribute__((address_space(3))) const int8_t*)lds_q;
#pragma unroll
    for (int it = 0; it < kQLoads; ++it) {
      const int region = kQShared ? c : it, row = region * kRowsPerRegion + ld_row_in;
      int qrow = min(row0 + row, Sq - 1);
      if (!fmha_in_bounds(qrow >= 0 && qrow < Sq)) qrow = 0;
      const int src = qrow * D + (((lane % kChunks) ^ k_swizzle<D>(row)) << 4);
      asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2 ; Q, shared %3"
                   ::"s"(dst + 1024u * region), "v"(src), "s"(qp), "n"(kQShared) : "memory");
    }
  }
#pragma unroll
  for (int it = 0; it < kLoads; ++it) issue(first_round, 0, it, n_blocks - 1);
  if (kEarlyV) {
#pragma unroll
    for (int it = 0; it < kLoads; ++it) issue(first_round, 1, it, n_blocks - 1);
  }

  // operand addresses (see the 256-row kernel)
  int k_read_off[kDSteps];
#pragma unroll
  for (int kk = 0; kk < kDSteps; ++kk) k_read_off[kk] = i32 * D + (((2 * kk + g) ^ k_swizzle<D>(i32)) << 4);
  int v_read_off;
  {
    const int jin = lane & 15, hh = (lane >> 4) & 1, kslot = jin >> 1;
    const int key_lane = 4 * g + (kslot < 4 ? kslot : kslot + 4);
    v_read_off = key_lane * D + (((2 * u_out + hh) ^ v_swizzle<D>(key_lane)) << 4) + 8 * (jin & 1);
  }

  // ---- state -------------------------------------------------------------------------------------------------------
  float o_f[16];
#pragma unroll
  for (int e = 0; e < 16; ++e) o_f[e] = 0.f;
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
  if (BIAS) asm volatile("" : "+v"(base_s));

  // ---- classification of the key blocks, by all wavefronts (the bits are those of the 256-row kernel) -----------------
  asm volatile("s_waitcnt vmcnt(%2)" : "+v"(mask_bytes), "+v"(tail_bytes) : "n"(kQLoads + (kEarlyV ? 2 : 1) * kLoads) : "memory");
  const int live_hi = classify_key_blocks<BK, kRowWaves>(mask_bytes, tail_bytes, mg, S, tid, lds_mask,
                                                         reinterpret_cast<unsigned char*>(lds_class4), keys_from, keys_to);
  if (lane == 0) lds_scan[wave] = live_hi;
  auto read_q = [&]() __attribute__((always_inline)) {
    asm volatile("; Q from LDS, place reused" ::: "memory");
#pragma unroll
    for (int kk = 0; kk < kDSteps; ++kk) qreg[kk] = *reinterpret_cast<const v4i*>(lds_q + k_read_off[kk]);
  };
  if constexpr (!kQInRegs && !kQShared) {
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"((kEarlyV ? 2 : 1) * kLoads) : "memory");
    read_q();
  }
  // K of round 0 and the Q rows have landed
  asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(kEarlyV ? kLoads : 0) : "memory");
  if constexpr (!kQShared) {
#pragma unroll
    for (int kk = 0; kk < kDSteps; ++kk) asm volatile("" : "+v"(qreg[kk]));
  }
  barrier();
  if constexpr (kQShared) read_q();
  int n = -1;
#pragma unroll
  for (int w = 0; w < kRowWaves; ++w) n = max(n, lds_scan[w]);
  n = __builtin_amdgcn_readfirstlane(n) + 1;  // one past the last block with an unmasked key
  const int rounds = PARTS ? min(first_round + args.rounds_per_part, (n + kSplitKeys - 1) / kSplitKeys) : (n + kSplitKeys - 1) / kSplitKeys;
  const long part_first = (long)bh * n_blocks;  // PARTS: the head's first key block in part_ml and part_o
  auto in_workspace = [&](int kb, int row) __attribute__((always_inline)) {  // block kb of this head, and what the host made room for
    const long heads = args.total_wgs / args.q_blocks;
    return fmha_in_bounds(kb >= 0 && kb < n_blocks && row >= 0 && row < Sq && (part_first + kb) * Sq + row < heads * n_blocks * Sq);
  };
  if constexpr (PARTS) {  // blocks without an unmasked key: a maximum that the merge takes for "nothing here"
    for (int kb = keys_to / BK - 1 - wave; kb >= kSplitKeys * first_round; kb -= kRowWaves)
      if ((reinterpret_cast<const unsigned char*>(lds_class4)[kb] & 2) && lane < Sq && (!kCheckBounds || in_workspace(kb, lane)))
        args.part_ml[(part_first + kb) * Sq + lane] = v2f{-__builtin_inff(), 0.f};
  }

  // ---- one key block of one row group: S^T, softmax, P^T --------------------------------------------------------------
  float m_blk = 0.f, l_blk = 0.f;
  v4i pk[kKeyTiles];
  auto scores_and_softmax = [&](int buf, int kb, int cls, auto between, auto in_softmax) __attribute__((always_inline)) {
    const int8_t* lds_k = &lds[buf][0][c][0];
    v16i acc[kKeyTiles];
    int mx[2] = {(int)0x80000000, (int)0x80000000};
    auto tile_max = [&](const v16i& a, int kk) __attribute__((always_inline)) {
#pragma unroll
      for (int e = 8 * kk / kDSteps; e < 8 * (kk + 1) / kDSteps; e += 2) {
        mx[0] = max(max(mx[0], a[e]), a[e + 1]);
        mx[1] = max(max(mx[1], a[8 + e]), a[9 + e]);
      }
    };
    auto gemm1 = [&](auto masked_t) __attribute__((always_inline)) {
      constexpr bool kMasked = decltype(masked_t)::value;
      unsigned mw[kKeyTiles];
      if constexpr (kMasked) {
        mask_words_of<BK>(mw, lds_mask, kb, tail_kb, S);
        acc[0] = masked_start(mw[0], MaskedUnits<BIAS>(), base_s);
      }
      // Operand reads run two key tiles ahead of the MFMAs, held there by the fences: left alone, the compiler reads each
      // operand right in front of its MFMA and the wavefront waits out the LDS latency sixteen times.
      v4i ka[3][kDSteps];
      auto read_k = [&](int t) __attribute__((always_inline)) {
#pragma unroll
        for (int kk = 0; kk < kDSteps; ++kk) ka[t % 3][kk] = *reinterpret_cast<const v4i*>(lds_k + k_read_off[kk] + 32 * t * D);
      };
      read_k(0);
      if (kKeyTiles > 1) read_k(1);
#pragma unroll
      for (int t = 0; t < kKeyTiles; ++t) {
        if (t + 2 < kKeyTiles) read_k(t + 2);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int kk = 0; kk < kDSteps; ++kk) {
          acc[t] = __builtin_amdgcn_mfma_i32_32x32x32_i8(ka[t % 3][kk], qreg[kk], (kk == 0 && !kMasked) ? base_s : acc[t], 0, 0, 0);
          __builtin_amdgcn_sched_barrier(0);
          if constexpr (kMasked)
            if (kk == kDSteps - 2 && t + 1 < kKeyTiles) acc[t + 1] = masked_start(mw[t + 1], MaskedUnits<BIAS>(), base_s);
          between(t * kDSteps + kk, kKeyTiles * kDSteps);
          if (t >= 1) tile_max(acc[t - 1], kk);
          __builtin_amdgcn_sched_barrier(0);
        }
      }
    };
    if (cls & 1) gemm1(Const<1>{});
    else gemm1(Const<0>{});
#pragma unroll
    for (int kk = 0; kk < kDSteps; ++kk) tile_max(acc[kKeyTiles - 1], kk);
    int ti = max(mx[0], mx[1]);
    ti = half_max(ti);
    if (cls & 1) ti = max(ti, (BIAS ? kScoreBaseBits : 0) - 1000000);  // the reference's sentinel (inc/fmha_i8.cuh:191-193)
    const float top = BIAS ? __int_as_float(ti) : (float)ti;
    float off = top * c2;
    if (!BIAS) off = __builtin_fmaf(fabsf(off), 2.384185791015625e-07f, off);
    if (!BIAS) off = fmaxf(off, args.floor2);
    m_blk = off - bias_c2;
    const float offq = off - (FULLP ? kLog2PscaleFull : kLog2Pscale);
    // Step q: the exponentials of quad q, the scaling of quad q+1 and the sum of quad q-1 (in the order of additions of the
    // other kernel), and a place for a tile load.
    constexpr int kQuads = 4 * kKeyTiles;
    float x[kQuads][4];
    auto scale = [&](int qd) __attribute__((always_inline)) {
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int s = acc[qd / 4][4 * (qd % 4) + j];
        x[qd][j] = __builtin_fmaf(BIAS ? __int_as_float(s) : (float)s, c2, -offq);
      }
    };
    auto sum = [&](int qd) __attribute__((always_inline)) {
      float s01 = x[qd][0] + x[qd][1];
      const float s23 = x[qd][2] + x[qd][3];
      s01 += s23;
      l_blk += s01;
    };
    l_blk = 0.f;
    scale(0);
#pragma unroll
    for (int qd = 0; qd < kQuads; ++qd) {
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int j = 0; j < 4; ++j) x[qd][j] = __builtin_amdgcn_exp2f(x[qd][j]);
      if (qd + 1 < kQuads) scale(qd + 1);
      if (qd >= 1) sum(qd - 1);
      if (kOwnK) {  // (keeps the step in front of the load)
        asm volatile("" : "+v"(x[qd][0]), "+v"(x[qd][1]), "+v"(x[qd][2]), "+v"(x[qd][3]));
        in_softmax(qd, kQuads);
      }
    }
    sum(kQuads - 1);
    l_blk = half_sum(l_blk);
#pragma unroll
    for (int qd = 0; qd < 4 * kKeyTiles; ++qd) {
      const float(&e)[4] = x[qd];
      const v2s lo = FULLP ? __builtin_amdgcn_cvt_pknorm_i16(e[0], e[1]) : __builtin_amdgcn_cvt_pknorm_i16(-e[0], -e[1]);
      const v2s hi = FULLP ? __builtin_amdgcn_cvt_pknorm_i16(e[2], e[3]) : __builtin_amdgcn_cvt_pknorm_i16(-e[2], -e[3]);
      const int four = __builtin_amdgcn_perm(__builtin_bit_cast(int, hi), __builtin_bit_cast(int, lo), 0x06040200);
      pk[qd / 4][qd % 4] = FULLP ? four ^ (int)0x80808080 : four;
    }
  };
  auto publish_p = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int t = 0; t < kKeyTiles; ++t) lds_p[r][c & (kPSlots - 1)][t][lane] = pk[t];
  };
  auto publish_ml = [&](int kb) __attribute__((always_inline)) {
    if constexpr (PARTS) {
      if (lane < Sq && (!kCheckBounds || in_workspace(kb, lane))) args.part_ml[(part_first + kb) * Sq + lane] = v2f{m_blk, l_blk};
      return;
    }
    lds_ml[r][c][i32][0] = m_blk;
    lds_ml[r][c][i32][1] = l_blk;
  };

  // ---- GEMM 2 and the merge of key blocks first .. first+COUNT-1 of the round, for this wavefront's columns -----------
  // A block without an unmasked key enters with weight 0 (its P may be anything: any int8 leaves the accumulators finite).
  int part_kb = 0;  // PARTS: the first key block of the round
  auto gemm2_merge = [&](int buf, int first, auto count_t, unsigned cls4, auto between) __attribute__((always_inline)) {
    constexpr int kCount = decltype(count_t)::value;
    typedef v2i __attribute__((address_space(3))) * lds_v2i_ptr;
    // The operands of all key blocks of a round in registers, or of two.  With all of them the weights of the blocks are computed in front of
    // the first product, over the latency of the reads; with two behind it: H32 Sq512 S4096 d128 31.1 us (31.6 with the weights in front),
    // B2 H16 Sq32 S2048 12.20 (12.31), B8 H16 Sq1 S2048 13.88 (13.99), d64 H16 Sq512 S896 7.11 (7.23), H24 S640 8.42 (8.31).
    constexpr bool kAllHeld = kOwnP && !FULLP;
    constexpr int kHeld = kAllHeld ? kCount : 2;
    v4i va[kHeld][kKeyTiles], p[kHeld][kKeyTiles];
    v16i oacc[2];
    auto read = [&](int j) __attribute__((always_inline)) {
      const int8_t* lds_v = &lds[buf][1][first + j][0];
#pragma unroll
      for (int t = 0; t < kKeyTiles; ++t) {
        const v2i lo = __builtin_amdgcn_ds_read_tr8_b64_v2i32((lds_v2i_ptr)(lds_v + v_read_off + 32 * t * D));
        const v2i hi = __builtin_amdgcn_ds_read_tr8_b64_v2i32((lds_v2i_ptr)(lds_v + v_read_off + 32 * t * D + 16 * D));
        va[j % kHeld][t] = v4i{lo[0], lo[1], hi[0], hi[1]};
      }
      if (kOwnP && c == first + j) {
#pragma unroll
        for (int t = 0; t < kKeyTiles; ++t) p[j % kHeld][t] = pk[t];
      } else {
#pragma unroll
        for (int t = 0; t < kKeyTiles; ++t) p[j % kHeld][t] = lds_p[r][(first + j) & (kPSlots - 1)][t][lane];
      }
    };
    if constexpr (PARTS) {  // the accumulators of every block to memory
      read(0);
#pragma unroll
      for (int j = 0; j < kCount; ++j) {
        if (j + 1 < kCount) read(j + 1);
        __builtin_amdgcn_sched_barrier(0);
        oacc[0] = base_c;
        if (FULLP) {  // (as in start() below)
          const v4i half = {0x40404040, 0x40404040, 0x40404040, 0x40404040};
#pragma unroll
          for (int t = 0; t < kKeyTiles; ++t) oacc[0] = __builtin_amdgcn_mfma_i32_32x32x32_i8(va[j % kHeld][t], half, oacc[0], 0, 0, 0);
#pragma unroll
          for (int e = 0; e < 16; ++e) oacc[0][e] = 2 * oacc[0][e] + kBaseBitsFull;
        }
#pragma unroll
        for (int t = 0; t < kKeyTiles; ++t) {
          oacc[0] = __builtin_amdgcn_mfma_i32_32x32x32_i8(va[j % kHeld][t], p[j % kHeld][t], oacc[0], 0, 0, 0);
          between(j * kKeyTiles + t, kCount * kKeyTiles);
        }
        if (!((cls4 >> (8 * (first + j))) & 2) && c < kDSteps && i32 < Sq &&
            (!kCheckBounds || (in_workspace(part_kb + first + j, i32) && fmha_in_bounds((8 * u_out + g) * 4 + 8 * 3 + 4 <= D)))) {
          int* at = args.part_o + (part_first + part_kb + first + j) * Sq * D + ((8 * u_out + g) * Sq + i32) * 4;
#pragma unroll
          for (int a = 0; a < 4; ++a)
            *reinterpret_cast<v4i*>(at + 8 * a * Sq) = v4i{oacc[0][4 * a], oacc[0][4 * a + 1], oacc[0][4 * a + 2], oacc[0][4 * a + 3]};
        }
      }
      return;
    }
    float take[kCount], keep[kCount];
    auto merge_piece = [&](int j, int piece, int pieces) __attribute__((always_inline)) {
#pragma unroll
      for (int e = 16 * piece / pieces; e < 16 * (piece + 1) / pieces; ++e) {
        const float v = FASTACC ? __int_as_float(oacc[j & 1][e]) : __int_as_float(oacc[j & 1][e]) - (FULLP ? kBaseFull : kBase);
        o_f[e] = __builtin_fmaf(FULLP ? take[j] : -take[j], v, o_f[e]);
      }
    };
    auto start = [&](int j) __attribute__((always_inline)) {
      oacc[j & 1] = base_c;
      if (FULLP) {
        // 128 times the column sums of the tile, in the accumulators' own layout: a product with 64s, doubled
        const v4i half = {0x40404040, 0x40404040, 0x40404040, 0x40404040};
#pragma unroll
        for (int t = 0; t < kKeyTiles; ++t)
          oacc[j & 1] = __builtin_amdgcn_mfma_i32_32x32x32_i8(va[j % kHeld][t], half, oacc[j & 1], 0, 0, 0);
#pragma unroll
        for (int e = 0; e < 16; ++e) oacc[j & 1][e] = 2 * oacc[j & 1][e] + kBaseBitsFull;
      }
    };
    auto product = [&](int j, int t) __attribute__((always_inline)) {
      oacc[j & 1] = __builtin_amdgcn_mfma_i32_32x32x32_i8(va[j % kHeld][t], p[j % kHeld][t], oacc[j & 1], 0, 0, 0);
    };
    // Operand reads one block ahead; the merge of a block stands behind the MFMAs of the next one.
    float ml[kCount][2];
#pragma unroll
    for (int j = 0; j < kCount; ++j) {
      ml[j][0] = lds_ml[r][first + j][i32][0];
      ml[j][1] = lds_ml[r][first + j][i32][1];
    }
#pragma unroll
    for (int j = 0; j < kHeld; ++j) read(j);
    __builtin_amdgcn_sched_barrier(0);
    auto first_products = [&]() __attribute__((always_inline)) {
      start(0);
#pragma unroll
      for (int t = 0; t < kKeyTiles; ++t) {
        product(0, t);
        between(t, kCount * kKeyTiles);
      }
    };
    if constexpr (!kAllHeld) first_products();
    bool moves[kCount];  // some row's reference exponent moves (wave-uniform, rare): O is rescaled in front of that block's merge
#pragma unroll
    for (int j = 0; j < kCount; ++j) {
      const bool dead = (cls4 >> (8 * (first + j))) & 2;
      const float mb = dead ? -__builtin_inff() : ml[j][0], lb = dead ? 0.f : ml[j][1];
      moves[j] = __ballot(mb > m_ref + kLazyLog2) != 0;
      const float m_new = moves[j] ? fmaxf(m_ref, mb) : m_ref;
      keep[j] = __builtin_amdgcn_exp2f(m_ref - m_new);  // exactly 1 where nothing moves
      m_ref = m_new;
      take[j] = __builtin_amdgcn_exp2f(mb - m_ref);
      l_run = __builtin_fmaf(take[j], lb, l_run * keep[j]);
      if (FASTACC) t_run = t_run * keep[j] + take[j];
    }
    auto rescale = [&](int j) __attribute__((always_inline)) {
      if (moves[j]) {
#pragma unroll
        for (int e = 0; e < 16; ++e) o_f[e] *= keep[j];
      }
    };
    if constexpr (kAllHeld) {
      __builtin_amdgcn_sched_barrier(0);
      first_products();
    }
    rescale(0);
#pragma unroll
    for (int j = 1; j < kCount; ++j) {
      start(j);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int t = 0; t < kKeyTiles; ++t) {
        product(j, t);
        __builtin_amdgcn_sched_barrier(0);
        between(j * kKeyTiles + t, kCount * kKeyTiles);
        merge_piece(j - 1, t, kKeyTiles);
        __builtin_amdgcn_sched_barrier(0);
      }
      if (!kAllHeld && j + 1 < kCount) read(j + 1);
      rescale(j);
      __builtin_amdgcn_sched_barrier(0);
    }
    merge_piece(kCount - 1, 0, 1);
  };

  // ---- the rounds --------------------------------------------------------------------------------------------------
  // S: GEMM 1 and softmax of block 4i+c; G: GEMM 2 and merge.  Barrier b1 publishes P and V of the round, b4 frees them and
  // publishes K of the next round.  The tile loads of a round stand behind the MFMAs, one after each: the CU's vector
  // memory path takes 64 bytes per cycle, a wavefront that issues its share in one go is held for 1000 cycles per kind.
  //   two buffers:              S(i) with K(i+1) | b1 | G(i) with V(i+1) | b4
  //   one buffer, R = 1:        S(i) with V(i) behind GEMM 1 and K(i+1) in the softmax | b1 | G(i) | b4
  //   one buffer, two steps:    S(i) with V of blocks 2, 3 of i, P of blocks 0, 1 | b1 | G of blocks 0, 1 with K(i+1) | b2 |
  //                             P of blocks 2, 3 | b3 | G of blocks 2, 3 with V of blocks 0, 1 of i+1 | b4
  auto written = [&]() { asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); };
  // V of round 0, or the half of it that the rounds themselves do not ask for
  if (!kOwnK && rounds > first_round) {
#pragma unroll
    for (int it = 0; it < (kBuffers == 2 ? kLoads : kLoads / 2); ++it) issue(first_round, 1, it, n - 1);
  }
  for (int i = first_round; i < rounds; ++i) {
    part_kb = kSplitKeys * i;
    const int buf = i & (kBuffers - 1);
    const bool more = i + 1 < rounds;
    const unsigned cls4 = (unsigned)__builtin_amdgcn_readfirstlane((int)lds_class4[i]);
    const int cls = (cls4 >> (8 * c)) & 3;
    const bool work = active && !(cls & 2);
    // `loads` tile loads from number `first` on, spread over `slots` places
    auto spread = [&](bool wanted, int round, int which, int first, int loads, int slot, int slots) __attribute__((always_inline)) {
#pragma unroll
      for (int it = slot * loads / slots; it < (slot + 1) * loads / slots; ++it)
        if (wanted) issue(round, which, first + it, n - 1);
    };
    constexpr bool kTwoBuffers = kBuffers == 2;
    constexpr int kHalf = kLoads / 2;
    auto loads_in_gemm1 = [&](int slot, int slots) __attribute__((always_inline)) {
      if (kTwoBuffers) spread(more, i + 1, 0, 0, kLoads, slot, slots);
      else if (kOwnK) spread(!kEarlyV || i > first_round, i, 1, 0, kLoads, slot, slots);
      else spread(true, i, 1, kHalf, kHalf, slot, slots);
    };
    auto loads_in_softmax = [&](int slot, int slots) __attribute__((always_inline)) {
      if (kOwnK) spread(more, i + 1, 0, 0, kLoads, slot, slots);
    };
    auto loads_in_gemm2 = [&](int slot, int slots) __attribute__((always_inline)) {
      if (kTwoBuffers) spread(more, i + 1, 1, 0, kTwoSteps ? kHalf : kLoads, slot, slots);
      else if (!kOwnK) spread(more, i + 1, 0, 0, kLoads, slot, slots);
    };
    auto loads_in_second_step = [&](int slot, int slots) __attribute__((always_inline)) {
      if (kTwoBuffers) spread(more, i + 1, 1, kHalf, kHalf, slot, slots);
      else spread(more, i + 1, 1, 0, kHalf, slot, slots);
    };
    if (work) {
      scores_and_softmax(buf, kSplitKeys * i + c, cls, loads_in_gemm1, loads_in_softmax);
      publish_ml(kSplitKeys * i + c);
      if (!kTwoSteps || c < 2) publish_p();
    } else {
      loads_in_gemm1(0, 1);
      loads_in_softmax(0, 1);
    }
    written();
    // V of this round (of its blocks 0, 1 in the last form); what has been asked for since may be in flight
    if (!kTwoBuffers && !kOwnK) wait_loads(half_kind);
    else if (more) wait_loads(one_kind);
    else wait_loads(none);
    barrier();  // b1
    if (active) gemm2_merge(buf, 0, Const<kTwoSteps ? 2 : 4>{}, cls4, loads_in_gemm2);
    else loads_in_gemm2(0, 1);
    // A last round with no more than two live blocks stops behind them: H32 Sq512 S1152 d128 14.8 -> 13.8 us, B2 H16 Sq512 S1152 d64
    // 12.8 -> 12.1, whole rounds as before.  (In the forms of one step the merge of two blocks beside that of four cost the whole rounds
    // 4 to 8 % and gave the others nothing.)
    if constexpr (kTwoSteps) if (n - kSplitKeys * i > 2) {
      barrier();  // b2
      if (work && c >= 2) publish_p();
      written();
      if (!kTwoBuffers && more) wait_loads(one_kind);  // V of blocks 2, 3
      else if (!kTwoBuffers) wait_loads(none);
      barrier();  // b3
      if (active) gemm2_merge(buf, 2, Const<2>{}, cls4, loads_in_second_step);
      else loads_in_second_step(0, 1);
    }
    // K of the next round
    if (kTwoBuffers && more) wait_loads(one_kind);
    else if (!kTwoBuffers && !kOwnK && more) wait_loads(half_kind);
    else wait_loads(none);
    barrier();  // b4
  }
  wait_loads(none);  // nothing may still be writing LDS when the wavefront ends (only possible when every key is masked)
  if (PARTS || !active || c >= kDSteps) return;

  // ---- epilogue (see the 256-row kernel) -----------------------------------------------------------------------------
  const float fin = (l_run > 0.f) ? args.out_scale * (128.f / kSnorm) * kBaseScale / l_run : 0.f;
  const float corr = FASTACC ? (FULLP ? -kBaseFull * t_run : kBase * t_run) : 0.f;
  int w[4];  // w[a]: output dims 32 u_out + 8a + 4g .. +3 of query row i32
#pragma unroll
  for (int a = 0; a < 4; ++a) {
    float y[4];
#pragma unroll
    for (int bb = 0; bb < 4; ++bb)
      y[bb] = __builtin_amdgcn_fmed3f(__builtin_fmaf(FASTACC ? o_f[4 * a + bb] + corr : o_f[4 * a + bb], fin, kMagic), kMagic - 127.f, kMagic + 127.f);
    const int lo = __builtin_amdgcn_perm(__float_as_int(y[1]), __float_as_int(y[0]), 0x0c0c0400);
    const int hi = __builtin_amdgcn_perm(__float_as_int(y[3]), __float_as_int(y[2]), 0x0c0c0400);
    w[a] = __builtin_amdgcn_perm(hi, lo, 0x05040100);
  }
  if (row0 + i32 >= Sq) return;
  if (!fmha_in_bounds(row0 + i32 >= 0 && q_head_off + (long)(row0 + i32 + 1) * D <= ((long)args.total_wgs / args.q_blocks + args.first_head) * Sq * D)) return;
  // (one store of sixteen bytes per lane, not two of eight: H16 S777 d128 11.51 -> 11.30 us, H32 Sq512 S1152 12.80 -> 12.56, H4 S512 d64 5.08 -> 4.99)
  // words a of lanes l and l+32 are neighbours: the exchanges hand lane l words 0, 1 of both and lane l+32 words 2, 3
  int8_t* op = args.o + q_head_off + (long)(row0 + i32) * D + 32 * u_out + 16 * g;
  const auto s0 = __builtin_amdgcn_permlane32_swap(w[0], w[2], false, false), s1 = __builtin_amdgcn_permlane32_swap(w[1], w[3], false, false);
  const int both[4] = {(int)s0[0], (int)s0[1], (int)s1[0], (int)s1[1]};
  *reinterpret_cast<v4i*>(op) = v4i{both[0], both[1], both[2], both[3]};
  store_wide<D>(args, op - args.o, both);
}

// ---- calls of few query rows: key blocks shared out over workgroups ------------------------------------------------------
// A call of at most kPartRows rows per head has one workgroup per head, which does all of its key blocks: with less than 256
// heads compute units idle, with a long sequence the time is that of one CU (2.4 us per 512 keys at d128).  Up to sixteen rows
// the workgroups are those of fmha_i8_few_kernel.
// Partial results of separate key ranges cannot be merged with the same bytes, but those of single key blocks can: PARTS leaves
// the accumulators of GEMM 2 (whole numbers) and the row's maximum and sum per block, 4 head_dim + 8 bytes per row where the
// block itself has 2 BK head_dim, and this kernel does the online merge of all blocks in key order.
constexpr int kPartRows = 32;

struct MergeArgs {
  const v2f* part_ml;
  const int* part_o;
  int8_t* o;
  int n_blocks, seq_q, head_dim, row_lanes;  // row_lanes: lanes of a wavefront per row, a power of two
  float floor2, out_scale;
  bool fast, full_range_p;
};
// What bounds it is latency, of its loads and of the chain over the blocks: BATCH blocks are loaded together, all of a short
// sequence, 32 of a long one, and where no reference exponent moves in a batch (nearly all behind the first) the weights of all
// of its blocks are independent of each other (B1 H8 Sq1 S65536 d128, 512 blocks: 77 -> 61 us for the call).
// One wavefront per workgroup: 64 / row_lanes rows (the last repeated) by 2 * row_lanes columns of a head, two columns per lane.
// All rows of a head are in one wavefront, because a reference exponent that moves in one row moves in all.
template <int BATCH>
__global__ __launch_bounds__(64, 1) void fmha_i8_merge_kernel(const MergeArgs args) {
  const int lane = threadIdx.x;
  const int Sq = args.seq_q, D = args.head_dim;
  const long bh = blockIdx.y;
  const int row = min(lane / args.row_lanes, Sq - 1);
  const int col = 2 * (blockIdx.x * args.row_lanes + lane % args.row_lanes);
  if (kCheckBounds && !fmha_in_bounds(row >= 0 && row < Sq && col >= 0 && col + 2 <= D)) return;
  const v2f* ml = args.part_ml + bh * args.n_blocks * Sq + row;
  const int* po = args.part_o + bh * args.n_blocks * Sq * D + (col / 4 * Sq + row) * 4 + col % 4;
  const float kGone = -__builtin_inff();
  const float base = args.fast ? 0.f : args.full_range_p ? kBaseFull : kBase;  // (x - 0 is x)
  const float sign = args.full_range_p ? 1.f : -1.f;
  float m_ref = args.floor2 - 2.f * kLazyLog2, t_run = 0.f, l_run = 0.f, o[2] = {0.f, 0.f};
  for (int kb0 = 0; kb0 < args.n_blocks; kb0 += BATCH) {
    v2f s[BATCH];
    v2i x[BATCH];
#pragma unroll
    for (int j = 0; j < BATCH; ++j) {
      long kb = min(kb0 + j, args.n_blocks - 1);
      if (kCheckBounds && !fmha_in_bounds(kb >= 0 && kb < args.n_blocks)) kb = 0;
      s[j] = ml[kb * Sq];
      x[j] = *reinterpret_cast<const v2i*>(po + kb * Sq * D);
    }
    __builtin_amdgcn_sched_barrier(0);
    float top = kGone;
#pragma unroll
    for (int j = 0; j < BATCH; ++j) {  // blocks past the end and those without an unmasked key (their accumulators were not written): weight 0
      if (kb0 + j >= args.n_blocks) s[j] = v2f{kGone, 0.f};
      if (s[j][0] == kGone) x[j] = v2i{0, 0};
      top = fmaxf(top, s[j][0]);
    }
    if (__ballot(top > m_ref + kLazyLog2) == 0) {
#pragma unroll
      for (int j = 0; j < BATCH; ++j) {
        const float take = __builtin_amdgcn_exp2f(s[j][0] - m_ref);
        l_run = __builtin_fmaf(take, s[j][1], l_run);
        t_run += take;
#pragma unroll
        for (int e = 0; e < 2; ++e) o[e] = __builtin_fmaf(sign * take, __int_as_float(x[j][e]) - base, o[e]);
      }
      continue;
    }
#pragma unroll
    for (int j = 0; j < BATCH; ++j) {
      const float mb = s[j][0];
      if (__ballot(mb > m_ref + kLazyLog2) != 0) {
        const float m_new = fmaxf(m_ref, mb), keep = __builtin_amdgcn_exp2f(m_ref - m_new);
        m_ref = m_new;
        l_run *= keep;
        t_run *= keep;
        o[0] *= keep;
        o[1] *= keep;
      }
      const float take = __builtin_amdgcn_exp2f(mb - m_ref);
      l_run = __builtin_fmaf(take, s[j][1], l_run);
      t_run += take;
#pragma unroll
      for (int e = 0; e < 2; ++e) o[e] = __builtin_fmaf(sign * take, __int_as_float(x[j][e]) - base, o[e]);
    }
  }
  const float fin = (l_run > 0.f) ? args.out_scale * (128.f / kSnorm) * kBaseScale / l_run : 0.f;
  const float corr = args.fast ? (args.full_range_p ? -kBaseFull * t_run : kBase * t_run) : 0.f;
  if (lane / args.row_lanes >= Sq) return;
  int y[2];
#pragma unroll
  for (int e = 0; e < 2; ++e)
    y[e] = __float_as_int(__builtin_amdgcn_fmed3f(__builtin_fmaf(args.fast ? o[e] + corr : o[e], fin, kMagic), kMagic - 127.f, kMagic + 127.f)) & 0xff;
  *reinterpret_cast<unsigned short*>(args.o + (bh * Sq + row) * D + col) = (unsigned short)(y[0] | (y[1] << 8));
}

}  // namespace fmha_i8_gfx950
