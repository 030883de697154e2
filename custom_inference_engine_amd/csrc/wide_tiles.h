// Wide query tiles: the key stream of a prefill work item whose columns fill a
// workgroup.
//
// A wide item is up to 8 column tiles of 16 (row, head) columns, two to each of
// the workgroup's four waves (4 and one, in some launches of few columns:
// wide_rule); every wave streams all of the item's keys against its own columns,
// so nothing is folded across waves, and the keys are read once per workgroup and
// staged in LDS.  A narrow item (attn_engine.h) gives every wave all columns and a
// quarter of the keys: short loops that suit few, latency-bound tiles, but at D =
// 64 each 64 columns (D = 128: each 16) read their whole prefix from L2, and each
// item pays its start and its fold.
//
// What bounds it: a wave's 32-key step is a serial chain (operands from LDS, S
// MFMAs, maximum, exponentials, P.V MFMAs, a barrier a stage).  So registers and
// LDS are kept small enough for three workgroups a CU (two at D = 128), whose
// waves fill each other's gaps; the MFMA pipes are then busy 23 % of a launch (4 x
// 2,048 new tokens, 14 / 2 heads, D = 64) to 39 % (1 x 8,192, 16 / 4 heads, D = 128),
// and a third of the LDS cycles at D = 64, half at D = 128, are bank conflicts; K/V
// reads hit L2 at 83-95 %.  Measured, us a launch with narrow items / wide
// (kernel times, profiles/mixed_wide_tiles.md): 4 x 2,048 new tokens (14 / 2 heads,
// D = 64) 86 / 63; 1 x 8,192 305 / 189; 8 x 1,024 (8 / 8 heads) 95 / 30; chunks of
// 1,024, 700 and 450 over 4,096, 2,000 and 1,000 keys with 13 decode rows (32 / 8
// heads, D = 128) 649 / 170; 1 x 8,192 (16 / 4 heads, D = 128) 1,596 / 330 (an S.P.V
// rate of 830 TFLOP/s).
//
// Staging: loads that write LDS (no registers), a stage ahead of its use, into
// the last of three buffers (D = 128: two stages ahead, four), so one barrier a
// stage suffices.  K rows keep their 16-byte chunks XORed with the row's low 3
// bits, so that an operand read (16 rows, one chunk column) spreads over the banks.
// V is read transposed (ds_read_b64_tr_b16: a lane gets 4 keys of its dim, the P.V
// operand, with no VALU), 4 rows of 32 bytes a 16-lane group: its chunk pairs
// are XORed with the row's low 2 bits.
#pragma once

#include "attn_engine.h"

namespace cie {

// Keys a stage (D = 128: half as many, so that four stages leave room in LDS for two
// workgroups a CU).
template <int D>
constexpr int stage_keys() {
  return D <= 64 ? 64 : 32;
}
constexpr int kWideWaves = 4;
constexpr int kWideColTiles = 8;  // column tiles an item holds at most: two a wave

// Waves a SIMD holds (and workgroups a CU, and registers: 512 / this a lane).
template <int D>
constexpr int wide_waves_per_simd() {
  return D <= 64 ? 3 : 2;
}

// LDS buffers of a stage: the published one, the one before it (its last step's
// V), and the others' loads in flight.
template <int D>
constexpr int stage_buffers() {
  return D <= 64 ? 3 : 4;
}

template <int D>
struct WideLds {
  static constexpr int tile = stage_keys<D>() * D;  // f16 of K (or V) a stage
  static constexpr size_t bytes = 2 * stage_buffers<D>() * tile * sizeof(f16);  // K and V
};

// Copies 16 bytes a lane from base + off (bytes, per lane) to the wave's 1 KiB
// at dst (LDS, lane order), without passing through registers.  Written as
// assembly because the compiler, not knowing which LDS the copy fills, would
// make every later LDS read wait for all copies in flight; wait_loads and a
// barrier publish them instead.  base and dst must be wave-uniform.
__device__ __forceinline__ void lds_copy16(f16* dst, const f16* base, uint32_t off) {
  typedef __attribute__((address_space(3))) f16 lds_f16;
  const uint32_t to = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)(lds_f16*)dst);
  const uint64_t b = reinterpret_cast<uint64_t>(base);
  const uint64_t sb = (uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((uint32_t)b) |
                      (uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((uint32_t)(b >> 32)) << 32;
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2"
               :
               : "s"(to), "v"(off), "s"(sb)
               : "memory", "m0");
}
// At most N vector-memory accesses of this wave, its latest, are in flight.
template <int N>
__device__ __forceinline__ void wait_loads() {
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

// V^T operand half: keys 4 * grp + e (e < 4) of a 16-key tile at dim r16 of a
// d-tile, from the wave's 16 rows of 32 bytes.
__device__ __forceinline__ f16x4 lds_read_tr(const f16* p) {
  typedef __fp16 h4 __attribute__((__vector_size__(8)));
  typedef __attribute__((address_space(3))) h4 lds_h4;
  return __builtin_bit_cast(f16x4, __builtin_amdgcn_ds_read_tr16_b64_v4f16((lds_h4*)(p)));
}

// Scores of keys at or past each lane's column limit become -inf.
template <int NCT>
__device__ __forceinline__ void mask_wide(f32x4 (&s)[NCT][2], int key0, const int (&lim)[NCT], int grp) {
  const int k0 = key0 + 4 * grp;
#pragma unroll
  for (int c = 0; c < NCT; ++c)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      s[c][0][r] = k0 + r < lim[c] ? s[c][0][r] : kNegInf;
      s[c][1][r] = k0 + 16 + r < lim[c] ? s[c][1][r] : kNegInf;
    }
}

// P.V operands of the two key tiles at key0: rows of keys at or past lim
// (wave-uniform) become zeros.  va[nt][e] is key key0 + 16 * (e / 4) + 4 * grp +
// e % 4.
template <int NT>
__device__ __forceinline__ void zero_keys(f16x8 (&va)[NT], int key0, int lim, int grp) {
  const int n = lim - key0 - 4 * grp;  // keys of the lane's first four that stay; 16 less: of the others
  uint32_t keep[4];                    // a mask per pair of keys
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int m = n - (i & 1) * 2 - (i >> 1) * 16;
    keep[i] = m <= 0 ? 0u : m == 1 ? 0xffffu : 0xffffffffu;
  }
  typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
#pragma unroll
  for (int nt = 0; nt < NT; ++nt) {
    u32x4 w = __builtin_bit_cast(u32x4, va[nt]);
#pragma unroll
    for (int i = 0; i < 4; ++i) w[i] &= keep[i];
    va[nt] = __builtin_bit_cast(f16x8, w);
  }
}

template <bool B>
struct Bool {
  static constexpr bool value = B;
};

// Streams key tiles [t_begin, t_end) (t_begin even) of the workgroup's item
// through every wave's NCT column tiles.  All waves call it with the same
// bounds; a wave without columns attends with zero queries.  Columns attend keys
// below lim[c], which grows with the column from first_lim, the item's first
// row's; keys at or past key_end do not exist.
// sm: WideLds<D>::bytes, free for the workgroup to write when it is called;
// it is free again when it returns.
template <int D, int NCT>
__device__ __forceinline__ void stream_wide(SoftmaxAcc<D, NCT>& st, const f16x8 (&q)[NCT][Geo<D>::KS],
                                            const int (&lim)[NCT], int first_lim, int t_begin,
                                            int t_end, int key_end, const PagedSrc& src,
                                            float scale_log2, f16* sm) {
  constexpr int KS = Geo<D>::KS;
  constexpr int NT = Geo<D>::NT;
  constexpr int CH = D / 8;            // 16-byte chunks a row
  constexpr int RPW = kWave / CH;      // rows a wave moves a pass
  constexpr int RPP = kWideWaves * RPW;  // rows a pass
  constexpr int kKeys = stage_keys<D>();
  constexpr int kTiles = kKeys / 16, kSub = kKeys / 32;  // key tiles and steps a stage
  constexpr int NP = kKeys / RPP;
  constexpr int kBufs = stage_buffers<D>();
  constexpr int kAhead = kBufs - 2;  // stages whose loads are in flight past the published one
  static_assert(RPP % 8 == 0 && 16 % RPW == 0, "a pass keeps the swizzles, a wave stays in a tile");
  constexpr int kTile = WideLds<D>::tile;
  t_begin = uniform(t_begin);
  t_end = uniform(t_end);
  key_end = uniform(key_end);
  const int n_stages = (t_end - t_begin + kTiles - 1) / kTiles;
  const int lane = opaque((int)threadIdx.x) & (kWave - 1);
  const int wave = uniform((int)threadIdx.x / kWave);
  const int r16 = lane & 15, grp = lane >> 4;
  first_lim = uniform(first_lim);
  // each column tile's largest limit (its last column's).  P is 0 past a column's
  // limit, but 0 times an Inf or NaN in V is NaN, so V rows that no column of a
  // tile attends are zeros for that tile: such a value reaches no row of an
  // earlier 16-row block, as in a narrow launch (16 * G columns are whole tiles).
  int v_end[NCT];
#pragma unroll
  for (int c = 0; c < NCT; ++c) v_end[c] = __builtin_amdgcn_readlane(lim[c], 15);

  // staging: a lane moves the 16 bytes that its slot of the wave's RPW rows
  // holds (byte offsets inside a 16-key tile of the pool)
  const int srow = wave * RPW + lane / CH, sch = lane % CH;
  const uint32_t kgo = (uint32_t)((srow & 15) * D + (sch ^ (srow & 7)) * 8) * 2;
  const uint32_t vgo = (uint32_t)((srow & 15) * D + (sch ^ (2 * (srow & 3))) * 8) * 2;
  // operand reads: K row r16, chunks 4 * ks + grp (XOR flips chunk bit 2 for
  // odd ks); V row 4 * grp + r16 / 4, its 8 bytes of d-tile nt
  int kaddr[2], vaddr[4];
#pragma unroll
  for (int i = 0; i < 2; ++i) kaddr[i] = r16 * D + ((4 * i + grp) ^ (r16 & 7)) * 8;
#pragma unroll
  for (int i = 0; i < 4; ++i)
    vaddr[i] = (4 * grp + (r16 >> 2)) * D + (2 * (i ^ (r16 >> 2)) + ((r16 >> 1) & 1)) * 8 + (r16 & 1) * 4;

  const int tpp = src.page_size >> 4;
  auto offsets = [&](int c0, int page) {  // pool element offset of tile c0 + lane
    const int t = c0 + lane;
    const int in_page = t - magic_div(t, src.tpp_magic) * tpp;
    return (int64_t)page * src.page_stride + src.head_off + (int64_t)(in_page * 16) * D;
  };
  int page = lane_page_id(src, t_begin, t_end, lane);
  int64_t toff = offsets(t_begin, page);
  auto load = [&](int stg) {
    f16* const kb = sm + stg % kBufs * 2 * kTile + wave * RPW * D;
#pragma unroll
    for (int i = 0; i < NP; ++i) {
      // (past the last tile: the last again, its rows never attended or zeroed)
      const int t = min(kTiles * stg + (i * RPP + wave * RPW) / 16, t_end - t_begin - 1);
      const int64_t base = readlane64(toff, t & (kWave - 1));
      lds_copy16(kb + i * RPP * D, src.k_pool + base, kgo);
      lds_copy16(kb + kTile + i * RPP * D, src.v_pool + base, vgo);
    }
  };
  // The stage's loads have landed, in every wave; from then on nothing reads
  // the buffer of stage stg - 2, which stage stg + kAhead goes to.
  auto publish = [&](int stg) {
    if (stg + kAhead <= n_stages)  // loads of the kAhead - 1 stages after it may be in flight
      wait_loads<(kAhead - 1) * 2 * NP>();
    else
      wait_loads<0>();
    __syncthreads();
    const int key0 = (t_begin + kTiles * stg) * 16;
    if (key0 + kKeys > key_end) {  // V rows past the sequence: the pool may hold anything
      f16* const vb = sm + stg % kBufs * 2 * kTile + kTile;
#pragma unroll
      for (int i = 0; i < NP; ++i)
        if (key0 + i * RPP + srow >= key_end)
          *reinterpret_cast<f16x8*>(vb + (i * RPP + srow) * D + sch * 8) = f16x8{};
      __syncthreads();
    }
  };
  // K(step) operands; V(step) operands
  auto buffer = [&](int step) { return sm + (step / kSub) % kBufs * 2 * kTile + (step % kSub) * 32 * D; };
  auto read_k = [&](f16x8 (&kf)[2][KS], int step) {
    const f16* const kb = buffer(step);
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int ks = 0; ks < KS; ++ks)
        kf[t][ks] = *reinterpret_cast<const f16x8*>(kb + kaddr[ks & 1] + (ks >> 1) * 64 + t * 16 * D);
  };
  auto read_v = [&](f16x8 (&va)[NT], int step) {
    const f16* const vb = buffer(step) + kTile;
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
      const f16* const v = vb + vaddr[nt & 3] + (nt >> 2) * 64;
      const f16x4 lo = lds_read_tr(v), hi = lds_read_tr(v + 16 * D);
      va[nt] = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
    }
  };
  const int n_steps = (t_end - t_begin + 1) >> 1;
  for (int i = 0; i < kAhead && i < n_stages; ++i) load(i);
  publish(0);
  if (kAhead < n_stages) load(kAhead);
  float x[NCT][8];  // the step's 2^x arguments: s * scale - m
  auto arguments = [&](const f32x4 (&s)[NCT][2]) {
#pragma unroll
    for (int c = 0; c < NCT; ++c)
#pragma unroll
      for (int e = 0; e < 8; ++e) x[c][e] = __builtin_fmaf(s[c][e / 4][e % 4], scale_log2, -st.m[c]);
  };
  {
    f16x8 kf[2][KS];
    f32x4 s[NCT][2];
    read_k(kf, 0);
#pragma unroll
    for (int c = 0; c < NCT; ++c)
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        s[c][t] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) s[c][t] = mfma16x16x32(kf[t][ks], q[c][ks], s[c][t]);
      }
    if (t_begin * 16 + 32 > first_lim) mask_wide<NCT>(s, t_begin * 16, lim, grp);
    update_max<D, NCT>(st, s, scale_log2);
    arguments(s);
  }
  // (no branch around a step's MFMAs: the compiler would keep two copies of
  // the accumulators)
  auto do_step = [&](int step, auto masked) {
    // the next step's stage, if it is a new one, and the loads of the one after
    const int stg = (step + 1) / kSub;
    if ((step + 1) % kSub == 0 && stg < n_stages) {
      publish(stg);
      const int next = stg + kAhead;
      if (next < n_stages) {
        // page ids of the next 64 tiles half their stages ahead
        constexpr int kPer = kWave / kTiles;  // stages a load of page ids covers
        if (next % kPer == kPer / 2)
          page = lane_page_id(src, t_begin + kTiles * (next + kPer / 2), t_end, lane);
        if (next % kPer == 0) toff = offsets(t_begin + kTiles * next, page);
        load(next);
      }
    }
    // (past the last step: stale LDS, its scores unused)
    f16x8 kf[2][KS], va[NT];
    read_k(kf, step + 1);
    // the step's exponentials among the next step's S MFMAs: a wave keeps
    // issuing while its MFMA runs
    f32x4 s[NCT][2];
    float e[NCT][8];
    constexpr int kMfma = 2 * KS * NCT, kExp = 8 * NCT;
#pragma unroll
    for (int i = 0; i < kMfma; ++i) {
      const int ks = i / (2 * NCT), t = i % 2, c = i / 2 % NCT;
      __builtin_amdgcn_sched_barrier(0);
      s[c][t] = mfma16x16x32(kf[t][ks], q[c][ks], ks == 0 ? f32x4{0.f, 0.f, 0.f, 0.f} : s[c][t]);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int j = i * kExp / kMfma; j < (i + 1) * kExp / kMfma; ++j) e[j / 8][j % 8] = fast_exp2(x[j / 8][j % 8]);
    }
    __builtin_amdgcn_sched_barrier(0);
    read_v(va, step);  // (here: its registers are free of K and x)
    f16x8 pop[NCT];
#pragma unroll
    for (int c = 0; c < NCT; ++c) {
#pragma unroll
      for (int j = 0; j < 8; ++j) pop[c][j] = (f16)e[c][j];
      // (needed here: the exponentials would sink below the branch otherwise)
      asm volatile("" : "+v"(pop[c]));
    }
    const int key0 = (t_begin + 2 * (step + 1)) * 16;
    if constexpr (masked.value) mask_wide<NCT>(s, key0, lim, grp);
    // (the later tile first: what is past its end is past the earlier one's)
#pragma unroll
    for (int c = NCT - 1; c >= 0; --c) {
      if constexpr (masked.value) zero_keys<NT>(va, key0 - 32, v_end[c], grp);
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) st.acc[c][nt] = mfma16x16x32(va[nt], pop[c], st.acc[c][nt]);
      add_row_sums(st.lpart[c], pop[c]);
    }
    if (step + 1 < n_steps) update_max<D, NCT>(st, s, scale_log2);
    arguments(s);
  };
  // A loop for the steps whose next one lies below every limit of the item (the
  // same for all waves, which meet at a stage's barrier), and one for the others:
  // tests for masking and for the V rows in every step cost 3-6 % at D = 64.
  const int open = first_lim - 16 * t_begin - 32;
  const int n_open = open < 32 ? 0 : min(n_steps, open / 32);
  int step = 0;
#pragma unroll 1
  for (; step < n_open; ++step) do_step(step, Bool<false>());
#pragma unroll 1
  for (; step < n_steps; ++step) do_step(step, Bool<true>());
  __syncthreads();  // (the caller may write sm)
}

}  // namespace cie
