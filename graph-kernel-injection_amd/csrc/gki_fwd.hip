// Block-sparse StreamingLLM attention: prefill forward kernel for gfx950.
//
// Replaces the reference's Triton `_fwd_kernel` (sparse_triton_kernel.py:231-352)
// and its launch (sparse_triton_kernel.py:662-682). Semantics follow the
// reference: S = (Q K^T) * scale in fp32, token mask (causal & (sink | window))
// inside visited tiles, online softmax, P cast to V's dtype before P V,
// O = acc / l, LSE = m + log(l) with the (O = 0, LSE = 0) sentinel for rows that
// saw no key (sparse_triton_kernel.py:341-352). The running max m and sum l
// are kept in base 2 (scores times log2 e, for v_exp_f32); the stored LSE is
// the natural m + ln(l) of the reference, converted once per row.
//
// 16-bit design (one workgroup = 4 waves = one 128-row q tile; wave w owns rows
// 32w .. 32w+31):
//  * S^T = K Q^T on v_mfma_f32_32x32x16_{bf16,f16}: a lane holds one query row
//    (and half of the keys), so the running max and sum are per-lane scalars
//    and a row reduction is one exchange between lanes l and l ^ 32.
//  * The S^T accumulators are, register for register, the B operand of
//    O^T += V^T P^T; V^T operands come from the gfx950 LDS transpose read
//    (ds_read_b64_tr_b16) in the same key order (Lane32).
//  * 32x32x16 instead of 16x16x32 (the same flops per cycle): one instruction
//    keeps the matrix core busy for 32 cycles, in which the SIMD issues the
//    softmax of its waves. 8 MFMAs beside 64 VALU operations take 139-149 ns
//    per wave (110 ns alone) against 173 ns for 16 of the smaller ones.
//  * K and V tiles are staged row-major (XOR-swizzled chunks) by LDS-DMA through
//    a buffer resource that covers the rows that exist, double-buffered: one
//    barrier per tile, the next tile's loads in flight during the MFMAs.
//  * Only kept tiles are visited (GPU-resident CSR list); the O^T rescale is
//    skipped, exactly, when no row max of a block moved.
//  * head_dim 128 runs the loop skewed by one kv tile (fwd_kernel_16's PIPE),
//    so that one wave's MFMAs of the next tile overlap its own softmax.
//  * The running max is kept on unscaled scores, so Q is read through the
//    Geom::q_and / q_xor transform that makes the effective scale positive.
// What bounds it: on long rows the matrix cores are 70% busy in cycles and the
// card lowers its clock under them (1.6-1.8 GHz against 2.4), so what is left
// out or not moved counts, not what is overlapped. 64 query rows per wave (half
// the LDS reads per flop, two waves per SIMD, every product slotted between
// softmax operations by hand) ran 6% (head_dim 64) and 28% (128) slower.
// The fp32 path uses v_mfma_f32_16x16x4f32 on 64-row tiles (16 rows per wave).
#include "gki_common.cuh"

namespace gki {
namespace {

// Online-softmax reference max moves only when a tile's row max exceeds it by
// more than this many log2 units, so p = exp2(s - m) stays below 2^8 and the O
// rescale is almost never needed. O = acc / l and LSE = m + ln(l) are exact for
// any reference max.
constexpr float kRescaleSlack = 8.f;
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
// Issue order of the skewed (PIPE) loop, imposed with sched_group_barrier
// (masks: 0x008 MFMA, 0x100 LDS read, 0x002 VALU). S_{j+1}: kPipeAheadS K
// reads first, then per MFMA one more read and kPipeValuS VALU ops of the exp
// work. O += V P: kPipeAheadO V^T reads first, then two reads and kPipeValuO
// VALU ops (the maxima of S_{j+1}) per MFMA. On a B1 H32 N16384 W2048 bf16
// forward: 3 VALU ops 0.542 ms, 5 or 6 0.552-0.557, reads 2 / 4 ahead 0.546,
// 8 / 12 0.557, no imposed order 0.560.
constexpr int kPipeAheadS = 4, kPipeAheadO = 8, kPipeValuS = 3, kPipeValuO = 1;
constexpr int kFwdThreads = 256;
// Waves per SIMD the compiler must fit in registers (HIP's second launch
// bound): 4 (up to 128 VGPRs) for head_dim <= 64, whose 32 KB of K / V buffers
// allow four workgroups per CU; 2 for head_dim 128 (64 KB of buffers, two
// workgroups per CU).
//
// PIPE selects the tile schedule. Without it every kv tile runs S = K Q^T,
// then mask / max / exp, then O += V P in turn, and the matrix cores idle
// through the softmax unless another wave of the SIMD has MFMAs to issue. With
// it the loop is skewed by one tile: iteration j runs S_{j+1} = K_{j+1} Q^T
// while it exponentiates S_j (MFMA and VALU of one wave in one straight-line
// block, interleaved in the order kPipe* describes), then O += V_j P_j while
// it takes the row maxima of S_{j+1}. K is therefore read one tile ahead of V:
// at iteration j the LDS holds K_{j+1} and V_j while K_{j+2} and V_{j+1} land
// in the other halves of the two double buffers (the same 2 x 2 tiles of LDS).
// Either loop is unrolled by two: the buffers are then constants of the LDS
// instructions, and the two score tiles of PIPE swap roles without copies.
// P_j is pinned (an empty asm that takes it) inside the S_{j+1} block:
// otherwise the compiler sinks the exp work past the mask branch into the
// O += V P block and no MFMA of S_{j+1} overlaps it.
//
// Against four waves of 16x16x32 MFMAs on the same tiles (ms, same card, three
// interleaved rounds): B1 H32 N16384 D128 W2048 bf16 0.530 -> 0.523, B4 H16
// N8192 D64 W1024 fp16 0.174 -> 0.168, B1 H16 N131072 D64 W4096 bf16 2.20 ->
// 2.16, 500 queries behind 8500 keys D128 0.0525 -> 0.0467, B4 H8 N2000 D32
// 0.0177 -> 0.0150.
template <typename T, int D, bool PIPE>
__global__ __launch_bounds__(kFwdThreads, D <= 64 ? 4 : 2) void fwd_kernel_16(
    Geom g, const uint16_t* __restrict__ Q, const uint16_t* __restrict__ K,
    const uint16_t* __restrict__ V, uint16_t* __restrict__ O, float* __restrict__ LSE,
    const int32_t* __restrict__ row_ptr, const int32_t* __restrict__ row_idx, int n_qt,
    const int32_t* __restrict__ wg_order) {
  constexpr int KS = D / 16;                   // k-steps of the QK^T contraction
  constexpr int DT = D >= 32 ? D / 32 : 1;     // 32-row tiles of O^T
  constexpr int NW = 4;
  __shared__ __align__(16) uint16_t sk[2][kTileN * D];
  __shared__ __align__(16) uint16_t sv[2][kTileN * D];

  const int n_wg = n_qt * g.B * g.H;
  const int wg = work_of(blockIdx.x, n_wg, wg_order);
  if (wg < 0) return;
  const int bh = wg / n_qt, qt = wg - bh * n_qt;
  const size_t qb = (size_t)bh * g.n_q * D;
  const size_t kb = (size_t)kv_bh(g, bh) * g.n_kv * D;
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lane = tid & 63, hi = lane >> 5, col = lane & 31;
  const Lane32<D> at(lane);
  const int qw = qt * kTileMF + wave * 32;     // first row of this wave

  uint4 qf[KS];
#pragma unroll
  for (int ks = 0; ks < KS; ++ks) {
    const uint4 v = q_words(g, row16_or_zero<D>(Q + qb, qw + col, g.n_q, 16 * ks + 8 * hi));
    qf[ks] = qw + col < g.n_q ? v : make_uint4(0, 0, 0, 0);
  }

  floatx16 o[DT];
#pragma unroll
  for (int i = 0; i < DT; ++i) o[i] = splat16(0.f);
  // Row sums on the MFMA pipe: 16x16x32 reads the P operand of a 32x32x16 as
  // (lane groups 0 and 2: rows 0-15, groups 1 and 3: rows 16-31), so a selector
  // of ones that pairs result row group g with the operand groups of g's parity
  // leaves lane l the sum of row l & 31 (over the same 16-bit P that
  // multiplies V) in every component.
  floatx4 lsum = floatx4{0.f, 0.f, 0.f, 0.f};
  const uint4 ones = ((lane >> 2) & 1) == ((lane >> 4) & 1) ? T::ones8() : make_uint4(0, 0, 0, 0);
  // nm: minus the row's reference max (scaled, log2 units), so P = exp2(S c + nm); thr: the unscaled score
  // above which it must move, (max + slack) / c, -inf until the row has seen a visible key.
  const float slack = kRescaleSlack * __builtin_amdgcn_rcpf(g.qk_scale_log2);   // a trigger: approximate is fine
  float nm = 0.f, thr = kNegInf;

  DmaTile<D, NW, true> dma;
  dma.init(tid);
  auto stage = [&](const uint16_t* src, int k0, uint16_t* dst) { dma.load(src + kb, k0, g.n_kv, dst); };
  auto tile_k0 = [&](int ent) { return (ent & kIdxMask) * kTileN; };

  // S^T of one kv tile: the 32 query rows of the wave against its 64 keys.
  auto scores = [&](const uint16_t* ck, floatx16 (&s)[2]) {
#pragma unroll
    for (int t = 0; t < 2; ++t) {
#pragma unroll
      for (int ks = 0; ks < KS; ++ks)
        s[t] = T::mfma32(at.rows(ck, t, ks), qf[ks], ks == 0 ? splat16(0.f) : s[t]);
    }
  };
  // Token mask of a tile (only where some element of it can be hidden).
  auto apply_mask = [&](int ent, floatx16 (&s)[2]) {
    const int k0 = tile_k0(ent);
    const bool partial = (ent >> kPartialBit) & 1;
    const bool need_mask = partial || (qw + 31 >= g.n_q) || (k0 + kTileN > g.n_kv) ||
                           !tile_all_visible(g, qw, min(qw + 31, g.n_q - 1), k0, k0 + kTileN - 1);
    if (need_mask) {
      const uint64_t bits = row_valid_bits(g, qw + col, k0, partial);
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        const LaneBits32 vis((uint32_t)(bits >> (32 * t)), hi);
#pragma unroll
        for (int r = 0; r < 16; ++r) s[t][r] = vis.pick(r, s[t][r], kNegInf);
      }
    }
  };
  auto lane_max = [&](const floatx16 (&s)[2]) {
    float mx = kNegInf;
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int r = 0; r < 16; ++r) mx = fmaxf(mx, s[t][r]);
    return mx;
  };
  // The reference moves (to the row's max) only when some score exceeds it by
  // the slack: p stays below 2^8 and the rescale of O and the row sums almost
  // never runs. Each lane tests its own half of the row; the cross-lane max
  // runs only then. Runs after every product of the tiles before.
  auto move_max = [&](float mx) {
    if (__any(mx > thr)) {
      const float mr = half_max(mx);
      const bool grow = mr > thr;
      const float nm1 = grow ? -mr * g.qk_scale_log2 : nm;
      // a first reference below zero scales nothing yet (o = lsum = 0)
      const float alpha = __builtin_amdgcn_exp2f(fminf(nm1 - nm, 0.f));
      nm = nm1;
      thr = grow ? mr + slack : thr;
      lsum[0] *= alpha;
#pragma unroll
      for (int dt = 0; dt < DT; ++dt) o[dt] *= alpha;
    }
  };
  // P = exp2(S c + nm) packed to 16-bit MFMA operands (16 keys each).
  auto probs = [&](floatx16 (&s)[2], uint4 (&p)[4]) {
#pragma unroll
    for (int t = 0; t < 2; ++t) {
#pragma unroll
      for (int r = 0; r < 16; ++r) s[t][r] = __builtin_amdgcn_exp2f(__builtin_fmaf(s[t][r], g.qk_scale_log2, nm));
      p[2 * t] = pack8<T>(s[t], 0);
      p[2 * t + 1] = pack8<T>(s[t], 1);
    }
  };
  // O^T += V^T P^T and the row sums.
  auto accumulate = [&](const uint16_t* cv, const uint4 (&p)[4]) {
#pragma unroll
    for (int st = 0; st < 4; ++st) {
#pragma unroll
      for (int dt = 0; dt < DT; ++dt) o[dt] = T::mfma32(at.cols(cv, st, dt), p[st], o[dt]);
      lsum = T::mfma(ones, p[st], lsum);
    }
  };
  const int e_beg = row_ptr[qt], e_end = row_ptr[qt + 1];
  if constexpr (!PIPE) {
    if (e_beg < e_end) {
      stage(K, tile_k0(row_idx[e_beg]), sk[0]);
      stage(V, tile_k0(row_idx[e_beg]), sv[0]);
    }
    dma_wait();
    __syncthreads();

    // unrolled by two so that the buffers are constants of the instructions
    auto step = [&](int e, int buf) {
      const int ent = row_idx[e];
      if (e + 1 < e_end) {
        const int k1 = tile_k0(row_idx[e + 1]);
        stage(K, k1, sk[buf ^ 1]);
        stage(V, k1, sv[buf ^ 1]);
      }
      // Left out where no row of this wave sees a key of the tile (a listed tile
      // is one that some of the workgroup's 128 rows sees): 2.5% of a forward
      // over 18-tile rows, 0.7% over 67 (head_dim 64).
      if (!tile_unseen(g, qw, qw + 31, tile_k0(ent), kTileN)) {
        floatx16 s[2];
        uint4 p[4];
        mfma_priority_hi<true>();
        scores(sk[buf], s);
        mfma_priority_lo<true>();
        apply_mask(ent, s);
        move_max(lane_max(s));
        probs(s, p);
        mfma_priority_hi<true>();
        accumulate(sv[buf], p);
        mfma_priority_lo<true>();
      }
      dma_wait();        // the next tile's LDS-DMA has landed before the barrier
      __syncthreads();
    };
    int e = e_beg;
    for (; e + 1 < e_end; e += 2) {
      step(e, 0);
      step(e + 1, 1);
    }
    if (e < e_end) step(e, 0);
  } else {
    const int n = e_end - e_beg;
    floatx16 sa[2], sb[2];
    // Prologue: K_0, V_0 and K_1 in LDS, S_0 with its maxima.
    if (n > 0) {
      const int k0 = tile_k0(row_idx[e_beg]);
      stage(K, k0, sk[0]);
      stage(V, k0, sv[0]);
      if (n > 1) stage(K, tile_k0(row_idx[e_beg + 1]), sk[1]);
    }
    dma_wait();
    __syncthreads();
    if (n > 0) {
      scores(sk[0], sa);
      apply_mask(row_idx[e_beg], sa);
      move_max(lane_max(sa));
    }
    __syncthreads();   // every wave is done with K_0 before iteration 0 refills its buffer

    // Iteration j (j + 1 < n): S_{j+1} from K_{j+1} into sn while s = S_j
    // becomes P_j; O += V_j P_j while sn's maxima are taken.
    auto step = [&](int j, int par, floatx16 (&s)[2], floatx16 (&sn)[2]) {   // par = j & 1
      const int e = e_beg + j;
      const int ent1 = row_idx[e + 1];
      // LDS: K_{j+1} in sk[(j+1)&1], V_j in sv[j&1]; refill the other halves
      if (j + 2 < n) stage(K, tile_k0(row_idx[e + 2]), sk[par]);
      stage(V, tile_k0(ent1), sv[par ^ 1]);

      uint4 p[4];
      scores(sk[par ^ 1], sn);   // MFMA ...
      probs(s, p);                   // ... under VALU
      // P is formed here, not sunk past the mask branch into the next block
#pragma unroll
      for (int st = 0; st < 4; ++st) {
        u32x4 w = __builtin_bit_cast(u32x4, p[st]);
        asm volatile("" : "+v"(w));
        p[st] = __builtin_bit_cast(uint4, w);
      }
      // issue order: the 2 KS MFMAs of S_{j+1} between the exp work
      __builtin_amdgcn_sched_group_barrier(0x100, kPipeAheadS, 0);
#pragma unroll
      for (int i = 0; i < 2 * KS; ++i) {
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
        if (i + kPipeAheadS < 2 * KS) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
        __builtin_amdgcn_sched_group_barrier(0x002, kPipeValuS, 0);
      }
      apply_mask(ent1, sn);
      accumulate(sv[par], p);           // MFMA ...
      const float mx = lane_max(sn);      // ... under VALU
      // issue order: the 4 DT MFMAs of O += V P (two V^T reads each) with the
      // maxima of S_{j+1} between them
      __builtin_amdgcn_sched_group_barrier(0x100, kPipeAheadO, 1);
#pragma unroll
      for (int i = 0; i < 4 * DT; ++i) {
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 1);
        if (2 * i + kPipeAheadO < 8 * DT) __builtin_amdgcn_sched_group_barrier(0x100, 2, 1);
        __builtin_amdgcn_sched_group_barrier(0x002, kPipeValuO, 1);
      }
      move_max(mx);
      dma_wait();
      __syncthreads();
    };
    auto last = [&](floatx16 (&s)[2], int par) {
      uint4 p[4];
      probs(s, p);
      accumulate(sv[par], p);
    };
    // Unrolled by two so that the score buffers swap roles without copies.
    int j = 0;
    for (; j + 2 < n; j += 2) {
      step(j, 0, sa, sb);
      step(j + 1, 1, sb, sa);
    }
    if (j + 1 < n) {
      step(j, 0, sa, sb);
      last(sb, 1);
    } else if (n > 0) {
      last(sa, 0);
    }
  }

  // The epilogue's row offsets from the lane index afresh (mbcnt: not provably
  // the one above), not the prologue's Q offsets held across the loop.
  const int lane_e = (int)__builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u));
  const int hi_e = lane_e >> 5;
  const int my_q = qw + (lane_e & 31);
  const float l_tot = lsum[0];
  const bool valid = l_tot > 0.f;
  const float inv = valid ? 1.f / l_tot : 1.f;
  if (my_q < g.n_q) {
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
      for (int r = 0; r < (D >= 32 ? 4 : 2); ++r) {     // D = 16: rows past 15 do not exist
        uint2 w;
        w.x = pack2<T>(o[dt][4 * r] * inv, o[dt][4 * r + 1] * inv);
        w.y = pack2<T>(o[dt][4 * r + 2] * inv, o[dt][4 * r + 3] * inv);
        *(uint2*)(O + qb + (size_t)my_q * D + 32 * dt + 8 * r + 4 * hi_e) = w;
      }
    if (hi_e == 0) LSE[(size_t)bh * g.n_q + my_q] = valid ? lse_natural(-nm, l_tot) : 0.f;
  }
}

// ---------------------------------------------------------------------------
// The same for grids too short for the card (fwd_shares_keys): the 128-row q tile of
// the schedule is two workgroups of 64 rows, and a workgroup's eight waves are
// two blocks of 32 rows x 4 shares of the keys. A step stages two kv tiles of
// the list (double-buffered) and share x takes 32 keys of them: tile x >> 1, half
// x & 1. Each share keeps a softmax state; they merge through LDS at the end, in
// order (share x the 32-element slice x of O). Bound by the latency of a wave's
// chain (products, softmax, products, barrier) per step: the split makes it a
// quarter as long per tile and puts twice the workgroups on the card. Kernel
// times, us: 500 queries behind 8500 keys, B1 H32, D128 (128 tiles) 46.8 -> 30.6;
// B1 H8 N1000 D64 (64) 20.7 -> 12.9; B1 H4 N1000 D128 (32) 18.2 -> 13.6.
// ---------------------------------------------------------------------------
template <typename T, int D>
__global__ __launch_bounds__(512, 2) void fwd_split_16(
    Geom g, const uint16_t* __restrict__ Q, const uint16_t* __restrict__ K,
    const uint16_t* __restrict__ V, uint16_t* __restrict__ O, float* __restrict__ LSE,
    const int32_t* __restrict__ row_ptr, const int32_t* __restrict__ row_idx, int n_qt,
    const int32_t* __restrict__ wg_order) {
  constexpr int KS = D / 16;
  constexpr int DT = D >= 32 ? D / 32 : 1;
  constexpr int QB = 2, KB = 4, NW = QB * KB;  // row blocks, key shares, waves
  constexpr int TPS = KB / 2;                  // kv tiles per step
  constexpr int kAhead = 4;                    // operands read ahead
  constexpr int TILE = kTileN * D;
  // K, V of the steps' tiles; at the end every wave's O (fp32)
  constexpr int OF = DT * 16 * 64;             // floats of a wave's O
  constexpr int LDS16 = 2 * TPS * 2 * TILE > NW * OF * 2 ? 2 * TPS * 2 * TILE : NW * OF * 2;
  __shared__ __align__(16) uint16_t stile[LDS16];
  __shared__ float sm[NW][32], sl[NW][32];

  int part;
  const int wg = work_part_of(blockIdx.x, n_qt * g.B * g.H, 4 / QB, wg_order, part);
  if (wg < 0) return;
  const int bh = wg / n_qt, qt = wg - bh * n_qt;
  const size_t qb = (size_t)bh * g.n_q * D;
  const size_t kb = (size_t)kv_bh(g, bh) * g.n_kv * D;
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lane = tid & 63, hi = lane >> 5, col = lane & 31;
  const Lane32<D> at(lane);
  const int blk = wave % QB, share = wave / QB;
  const int qw = qt * kTileMF + 32 * (part * QB + blk);   // first row of this wave
  if (qt * kTileMF + 32 * QB * part >= g.n_q) return;     // a part past the last row

  const int e_beg = row_ptr[qt], n = row_ptr[qt + 1] - e_beg;
  const int32_t* const ents = row_idx + e_beg;
  DmaTile<D, NW, true> dma;
  dma.init(tid);
  auto tile_k0 = [&](int ent) { return (ent & kIdxMask) * kTileN; };
  // the tiles of step s into buffer s & 1: K, V, K, V
  auto stage = [&](int s) {
#pragma unroll
    for (int j = 0; j < TPS; ++j)
      if (TPS * s + j < n) {
        const int k0 = tile_k0(ents[TPS * s + j]);
        uint16_t* const dst = stile + (2 * TPS * (s & 1) + 2 * j) * TILE;
        dma.load(K + kb, k0, g.n_kv, dst);
        dma.load(V + kb, k0, g.n_kv, dst + TILE);
      }
  };
  uint4 qf[KS];
#pragma unroll
  for (int ks = 0; ks < KS; ++ks) {
    const uint4 v = q_words(g, row16_or_zero<D>(Q + qb, qw + col, g.n_q, 16 * ks + 8 * hi));
    qf[ks] = qw + col < g.n_q ? v : make_uint4(0, 0, 0, 0);
  }
  floatx16 o[DT];
#pragma unroll
  for (int i = 0; i < DT; ++i) o[i] = splat16(0.f);
  // the row sum of the fp32 P over the lane's keys; the lazy reference max as in
  // fwd_kernel_16
  float lsum = 0.f;
  const float slack = kRescaleSlack * __builtin_amdgcn_rcpf(g.qk_scale_log2);
  float nm = 0.f, thr = kNegInf;

  const int steps = (n + TPS - 1) / TPS;
  dma_wait();          // the Q loads, before any LDS-DMA is in flight
  if (steps > 0) stage(0);
  const int tj = share >> 1, th = share & 1;
  for (int st = 0; st < steps; ++st) {
    dma_wait();
    __syncthreads();   // step st is in LDS, and every wave is done with the step before
    if (st + 1 < steps) stage(st + 1);
    const int e = TPS * st + tj;
    if (e < n) {
      const int ent = ents[e];
      const int k0 = tile_k0(ent), kw = k0 + 32 * th;
      const bool partial = (ent >> kPartialBit) & 1;
      const uint16_t* ck = stile + (2 * TPS * (st & 1) + 2 * tj) * TILE + 32 * D * th;
      const uint16_t* cv = ck + TILE;
      if (!tile_unseen(g, qw, qw + 31, kw, 32)) {
        // operands read kAhead products ahead, in a pinned order
        floatx16 s = splat16(0.f);
        uint4 op[kAhead];
#pragma unroll
        for (int i = 0; i < kAhead && i < KS; ++i) op[i] = at.rows(ck, 0, i);
#pragma unroll
        for (int i = 0; i < KS; ++i) {
          s = T::mfma32(op[i % kAhead], qf[i], s);
          if (i + kAhead < KS) op[i % kAhead] = at.rows(ck, 0, i + kAhead);
          __builtin_amdgcn_sched_barrier(0);
        }
        // V^T operands of the first products, in flight through the softmax
        uint4 ov[kAhead];
#pragma unroll
        for (int i = 0; i < kAhead && i < 2 * DT; ++i) ov[i] = at.cols(cv, i / DT, i % DT);
        if (partial || qw + 31 >= g.n_q || kw + 32 > g.n_kv || !tile_all_visible(g, qw, qw + 31, kw, kw + 31)) {
          const uint64_t bits = row_valid_bits(opaque_blocks(g), qw + (lane_now() & 31), k0, partial);
          const LaneBits32 vis(th ? (uint32_t)(bits >> 32) : (uint32_t)bits, lane_now() >> 5);
#pragma unroll
          for (int r = 0; r < 16; ++r) s[r] = vis.pick(r, s[r], kNegInf);
        }
        float mx = kNegInf;
#pragma unroll
        for (int r = 0; r < 16; ++r) mx = fmaxf(mx, s[r]);
        if (__any(mx > thr)) {
          const float mr = half_max(mx);
          const bool grow = mr > thr;
          const float nm1 = grow ? -mr * g.qk_scale_log2 : nm;
          const float alpha = __builtin_amdgcn_exp2f(fminf(nm1 - nm, 0.f));
          nm = nm1;
          thr = grow ? mr + slack : thr;
          lsum *= alpha;
#pragma unroll
          for (int dt = 0; dt < DT; ++dt) o[dt] *= alpha;
        }
#pragma unroll
        for (int r = 0; r < 16; ++r) s[r] = __builtin_amdgcn_exp2f(__builtin_fmaf(s[r], g.qk_scale_log2, nm));
#pragma unroll
        for (int r = 0; r < 16; r += 4) lsum += (s[r] + s[r + 1]) + (s[r + 2] + s[r + 3]);
        const uint4 p[2] = {pack8<T>(s, 0), pack8<T>(s, 1)};
#pragma unroll
        for (int i = 0; i < 2 * DT; ++i) {
          o[i % DT] = T::mfma32(ov[i % kAhead], p[i / DT], o[i % DT]);
          if (i + kAhead < 2 * DT) ov[i % kAhead] = at.cols(cv, (i + kAhead) / DT, (i + kAhead) % DT);
          __builtin_amdgcn_sched_barrier(0);
        }
      }
    }
  }
  __syncthreads();

  // Merge (every wave is done with the staging buffers, nothing is in flight). A
  // share that saw no key of a row has lsum = 0 there and weighs nothing.
  float* red = (float*)stile + (size_t)wave * OF;
#pragma unroll
  for (int dt = 0; dt < DT; ++dt)
#pragma unroll
    for (int q = 0; q < 4; ++q)
      *(floatx4*)(red + ((dt * 4 + q) * 64 + lane) * 4) =
          floatx4{o[dt][4 * q], o[dt][4 * q + 1], o[dt][4 * q + 2], o[dt][4 * q + 3]};
  lsum = half_sum(lsum);
  if (hi == 0) {
    sm[wave][col] = lsum > 0.f ? -nm : kNegInf;
    sl[wave][col] = lsum;
  }
  __syncthreads();
  float M = kNegInf, L = 0.f, f[KB];
#pragma unroll
  for (int x = 0; x < KB; ++x) M = fmaxf(M, sm[x * QB + blk][col]);
#pragma unroll
  for (int x = 0; x < KB; ++x) {
    f[x] = M == kNegInf ? 0.f : __builtin_amdgcn_exp2f(sm[x * QB + blk][col] - M);
    L += sl[x * QB + blk][col] * f[x];
  }
  const bool valid = L > 0.f;
  const float inv = valid ? 1.f / L : 1.f;
  const int my_q = qw + col;
  if (my_q >= g.n_q) return;
  for (int dt = share; dt < DT; dt += KB)
#pragma unroll
    for (int q = 0; q < (D >= 32 ? 4 : 2); ++q) {       // D = 16: rows past 15 do not exist
      floatx4 a = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int x = 0; x < KB; ++x)
        a += *(const floatx4*)((const float*)stile + (size_t)(x * QB + blk) * OF + ((dt * 4 + q) * 64 + lane) * 4) * f[x];
      *(uint2*)(O + qb + (size_t)my_q * D + 32 * dt + 8 * q + 4 * hi) =
          make_uint2(pack2<T>(a[0] * inv, a[1] * inv), pack2<T>(a[2] * inv, a[3] * inv));
    }
  if (share == 0 && hi == 0) LSE[(size_t)bh * g.n_q + my_q] = valid ? lse_natural(M, L) : 0.f;
}

// ---------------------------------------------------------------------------
// fp32 path (v_mfma_f32_16x16x4f32, 64-row tiles): K and V row-major in LDS
// (swz_f32), staged by LDS-DMA, double-buffered, one barrier per 32 or 64 keys.
// Bound by the fp32 matrix cores (154 TFLOP/s reached by a large product): B1
// H16 N8192 D64 W1024 428 -> 334 us, N4096 D128 550 -> 319 us against 4-byte LDS
// reads and tiles staged through registers behind two barriers.
// The softmax runs in natural units: the running max m is that of the scaled
// scores S * scale and each exponent is exp2(fma(S, scale, -m) * log2 e), so
// the scale is applied exactly and only the (small) difference is rounded;
// the backward forms P = exp(S * scale - LSE) the same way from the stored
// LSE = m + ln(l), which therefore matches these scores to within its own
// rounding.
// ---------------------------------------------------------------------------
//
// A workgroup's four waves are QB blocks of 16 query rows x 4 / QB shares of
// the keys of each staged step (16 keys each; two such subtiles when QB = 4), so
// a 64-row q tile of the schedule is 4 / QB workgroups. With several shares the
// waves keep a softmax state each and merge through LDS at the end: a grid too
// short for the card (B1 H4 N1024: 64 tiles, 29 us) then runs on four times the
// workgroups, each a quarter of the serial chain (11.6 us).
template <int D, int QB>
__global__ __launch_bounds__(256, D * (QB == 1 ? 4 : 2) >= 512 ? 1 : D * (QB == 1 ? 4 : 2) >= 256 ? 2 : 3) void fwd_kernel_32(
    Geom g, const float* __restrict__ Q, const float* __restrict__ K, const float* __restrict__ V,
    float* __restrict__ O, float* __restrict__ LSE, const int32_t* __restrict__ row_ptr,
    const int32_t* __restrict__ row_idx, int n_qt, const int32_t* __restrict__ wg_order) {
  constexpr int DJ = D / 16;                 // 16-byte chunks of a row per lane; output tiles
  constexpr int KB = 4 / QB;                 // key shares
  constexpr int TR = KB == 4 ? 64 : 32;      // keys per staged step
  constexpr int SUBS = TR / (16 * KB);       // 16-key subtiles per wave and step
  constexpr int HALVES = kTileN / TR;
  constexpr int DV = D >= 64 ? D / 64 : 1;   // 16-byte reads of a V row per lane (64 columns each)
  constexpr int DE = D / (16 * DV);          // output tiles per such read
  __shared__ __align__(16) float sk[2][TR * D];
  __shared__ __align__(16) float sv[2][TR * D];

  int part;
  const int wg = work_part_of(blockIdx.x, n_qt * g.B * g.H, KB, wg_order, part);
  if (wg < 0) return;
  const int bh = wg / n_qt, qt = wg - bh * n_qt;
  const size_t qb = (size_t)bh * g.n_q * D;
  const size_t kb = (size_t)kv_bh(g, bh) * g.n_kv * D;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int grp = lane >> 4, col = lane & 15;
  const int share = wave / QB;
  const int q0 = qt * kTileM + 16 * (part * QB + wave % QB);
  const int my_q = q0 + col;

  floatx4 qf[DJ];
#pragma unroll
  for (int j = 0; j < DJ; ++j)
    qf[j] = my_q < g.n_q ? *(const floatx4*)(Q + qb + (size_t)my_q * D + 16 * j + 4 * grp)
                         : floatx4{0.f, 0.f, 0.f, 0.f};

  // o[v][e]: row x of the tile is element 64 v + DE x + e
  floatx4 o[DV][DE];
#pragma unroll
  for (int v = 0; v < DV; ++v)
#pragma unroll
    for (int e = 0; e < DE; ++e) o[v][e] = floatx4{0.f, 0.f, 0.f, 0.f};
  // the row sum with its rounding error kept apart: an addition per 32 keys left
  // the LSE of a 1024-key row 9% above one rounding (8% per 64 keys, now 6%)
  float m = kNegInf, l = 0.f, lc = 0.f;

  const int e_beg = row_ptr[qt], n_step = (row_ptr[qt + 1] - e_beg) * HALVES;
  DmaTileF32<D, TR> dma;
  dma.init(tid);
  auto step_k0 = [&](int s) {
    return (row_idx[e_beg + s / HALVES] & kIdxMask) * kTileN + (s % HALVES) * TR;
  };
  auto stage = [&](int s, int buf) {
    const int k0 = step_k0(s);
    dma.load(K + kb, k0, g.n_kv, sk[buf]);
    dma.load(V + kb, k0, g.n_kv, sv[buf]);
  };
  dma_wait();          // the Q loads, before any LDS-DMA is in flight
  if (n_step > 0) stage(0, 0);
  dma_wait();
  __syncthreads();
  const int q_hi = min(q0 + 15, g.n_q - 1);
  for (int s = 0; s < n_step; ++s) {
    const int buf = s & 1;
    const bool partial = (row_idx[e_beg + s / HALVES] >> kPartialBit) & 1;
    if (s + 1 < n_step) stage(s + 1, buf ^ 1);
    const float *ck = sk[buf], *cv = sv[buf];
    const int k0 = step_k0(s) + 16 * SUBS * share;       // the wave's first key
    const bool need_mask = partial || (q0 + 15 >= g.n_q) || (k0 + 16 * SUBS > g.n_kv) ||
                           !tile_all_visible(g, q0, q_hi, k0, k0 + 16 * SUBS - 1);
    floatx4 p[SUBS];
#pragma unroll
    for (int t = 0; t < SUBS; ++t) {
      const int r = 16 * (SUBS * share + t) + col;
      p[t] = mfma_f32_dot<4 * DJ>([&](int j) { return *(const floatx4*)(ck + off_f32<D>(r, 4 * j + grp)); }, qf);
    }
    // the largest scaled score: rounding is monotone, so the largest (smallest,
    // for a negative scale) score, scaled
    float mx;
    uint64_t bits = ~0ull;
    if (need_mask) {
      bits = row_valid_bits(g, my_q, k0, partial);
      const LaneBits16 vis(bits, grp);
      mx = kNegInf;
#pragma unroll
      for (int t = 0; t < SUBS; ++t)
#pragma unroll
        for (int i = 0; i < 4; ++i) mx = fmaxf(mx, vis.mask(t, i) ? p[t][i] * g.scale : kNegInf);
    } else if (g.scale >= 0.f) {
      mx = p[0][0];
#pragma unroll
      for (int t = 0; t < SUBS; ++t)
#pragma unroll
        for (int i = 0; i < 4; ++i) mx = fmaxf(mx, p[t][i]);
      mx *= g.scale;
    } else {
      mx = p[0][0];
#pragma unroll
      for (int t = 0; t < SUBS; ++t)
#pragma unroll
        for (int i = 0; i < 4; ++i) mx = fminf(mx, p[t][i]);
      mx *= g.scale;
    }
    if (__any(mx > m)) {               // some row's max moves
      const float m_new = fmaxf(m, wave_max16x4(mx));
      const float alpha = m_new == kNegInf ? 1.f : __builtin_amdgcn_exp2f((m - m_new) * kLog2e);
      m = m_new;
      l *= alpha;
      lc *= alpha;
#pragma unroll
      for (int v = 0; v < DV; ++v)
#pragma unroll
        for (int e = 0; e < DE; ++e) o[v][e] *= alpha;
    }
    const float m_use = m == kNegInf ? 0.f : m;
#pragma unroll
    for (int t = 0; t < SUBS; ++t)
#pragma unroll
      for (int i = 0; i < 4; ++i)
        p[t][i] = __builtin_amdgcn_exp2f(__builtin_fmaf(p[t][i], g.scale, -m_use) * kLog2e);
    if (need_mask) {
      const LaneBits16 vis(bits, grp);
#pragma unroll
      for (int t = 0; t < SUBS; ++t)
#pragma unroll
        for (int i = 0; i < 4; ++i) p[t][i] = vis.keep(t, i, p[t][i]);
    }
    float rs = 0.f;
#pragma unroll
    for (int t = 0; t < SUBS; ++t) rs += (p[t][0] + p[t][1]) + (p[t][2] + p[t][3]);
    const float l_new = l + rs;
    lc += rs - (l_new - l);
    l = l_new;
#pragma unroll
    for (int t = 0; t < SUBS; ++t)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int r = 16 * (SUBS * share + t) + 4 * grp + i;
#pragma unroll
        for (int v = 0; v < DV; ++v) {
          const auto x = cols_f32<D, DE>(cv, r, v, col);
#pragma unroll
          for (int e = 0; e < DE; ++e) o[v][e] = mfma_f32(x[e], p[t][i], o[v][e]);
        }
      }
    dma_wait();        // the next step's LDS-DMA has landed before the barrier
    __syncthreads();
  }

  l = wave_sum16x4(l + lc);
  double l_tot = l;
  if constexpr (KB > 1) {
    // shares 1 .. KB - 1 hand (o, m, l) over through LDS (free: every wave
    // passed the last barrier); share 0 merges them in order, by one factor each
    static_assert((KB - 1) * QB * (D + 2) * 16 <= 2 * TR * D, "the shares' sums fit one staging array");
    float* red = &sk[0][0];
    const int blk = wave % QB;
    auto part_of = [&](int w) { return red + ((size_t)(w - 1) * QB + blk) * (D + 2) * 16; };
    if (share > 0) {
      float* dst = part_of(share) + lane;
#pragma unroll
      for (int v = 0; v < DV; ++v)
#pragma unroll
        for (int e = 0; e < DE; ++e)
#pragma unroll
          for (int i = 0; i < 4; ++i) dst[64 * ((v * DE + e) * 4 + i)] = o[v][e][i];
      if (grp == 0) {
        dst[16 * D] = m;
        dst[16 * D + 16] = l;
      }
    }
    __syncthreads();
    if (share > 0) return;
    float f[KB];
    const float m_own = m;
#pragma unroll
    for (int w = 1; w < KB; ++w) m = fmaxf(m, part_of(w)[16 * D + col]);
    const float m_use = m == kNegInf ? 0.f : m;
    f[0] = __builtin_amdgcn_exp2f((m_own - m_use) * kLog2e);
#pragma unroll
    for (int w = 1; w < KB; ++w) f[w] = __builtin_amdgcn_exp2f((part_of(w)[16 * D + col] - m_use) * kLog2e);
    // the row sum in 64 bits, a lane group per share: 32-bit factors would round it
    // by as much as the stored LSE is rounded
    const int ws = grp % KB;
    const float* of = part_of(ws ? ws : 1) + 16 * D + col;
    l_tot = (double)(ws ? of[16] : l) * exp((double)(ws ? of[0] : m_own) - (double)m_use);
    l_tot += __shfl_xor(l_tot, 16);
    if constexpr (KB == 4) l_tot += __shfl_xor(l_tot, 32);
    l = (float)l_tot;
#pragma unroll
    for (int v = 0; v < DV; ++v)
#pragma unroll
      for (int e = 0; e < DE; ++e)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          float a = o[v][e][i] * f[0];
#pragma unroll
          for (int w = 1; w < KB; ++w)
            a += part_of(w)[64 * ((v * DE + e) * 4 + i) + lane] * f[w];
          o[v][e][i] = a;
        }
  }
  const bool valid = l > 0.f;
  if (my_q < g.n_q) {
    const float den = valid ? l : 1.f;
#pragma unroll
    for (int v = 0; v < DV; ++v)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        float* dst = O + qb + (size_t)my_q * D + 64 * v + DE * (4 * grp + i);
        if constexpr (DE == 4) {
          *(floatx4*)dst = floatx4{o[v][0][i] / den, o[v][1][i] / den, o[v][2][i] / den, o[v][3][i] / den};
        } else {
#pragma unroll
          for (int e = 0; e < DE; ++e) dst[e] = o[v][e][i] / den;
        }
      }
    if (grp == 0) LSE[(size_t)bh * g.n_q + my_q] = valid ? (float)((double)m + log(l_tot)) : 0.f;
  }
}

// The skewed schedule holds two score tiles (32 more VGPRs): head_dim 128
// has them within its 256 (without it 2% slower); at head_dim 64 it would cost
// the fourth workgroup per CU.
template <int D>
constexpr bool kFwdPipe = D >= 128;

template <typename T, int D>
void launch_fwd16(const Geom& g, const void* q, const void* k, const void* v, void* o, float* lse,
                  const int32_t* row_ptr, const int32_t* row_idx, int n_qt, const int32_t* wg_order,
                  hipStream_t stream) {
  const int grid = n_qt * g.B * g.H;
#define GKI_FWD16(KERNEL, GRID, THREADS)                                                           \
  hipLaunchKernelGGL(KERNEL, dim3(GRID), dim3(THREADS), 0, stream, g, (const uint16_t*)q,          \
                     (const uint16_t*)k, (const uint16_t*)v, (uint16_t*)o, lse, row_ptr, row_idx,  \
                     n_qt, wg_order)
  if (fwd_shares_keys(D, grid, row_kv_tiles(g, kTileMF)))
    GKI_FWD16((fwd_split_16<T, D>), work_parts_grid(grid, 2), 512);
  else
    GKI_FWD16((fwd_kernel_16<T, D, kFwdPipe<D>>), grid, kFwdThreads);
#undef GKI_FWD16
}

template <int D>
int launch_fwd(int dtype, const Geom& g, const void* q, const void* k, const void* v, void* o,
               float* lse, const int32_t* row_ptr, const int32_t* row_idx, int n_qt,
               const int32_t* wg_order, hipStream_t stream) {
  const int grid = n_qt * g.B * g.H;
  if (dtype == kF32) {
#define GKI_FWD32(QB)                                                                               \
  hipLaunchKernelGGL((fwd_kernel_32<D, QB>), dim3(work_parts_grid(grid, 4 / QB)), dim3(256), 0,     \
                     stream, g, (const float*)q, (const float*)k, (const float*)v, (float*)o, lse,  \
                     row_ptr, row_idx, n_qt, wg_order)
    const int blocks = f32_row_blocks(D, grid, row_kv_tiles(g, kTileM));
    if (blocks == 1) GKI_FWD32(1);
    else if (blocks == 2) GKI_FWD32(2);
    else GKI_FWD32(4);
#undef GKI_FWD32
  } else if (dtype == kF16) {
    launch_fwd16<F16, D>(g, q, k, v, o, lse, row_ptr, row_idx, n_qt, wg_order, stream);
  } else {
    launch_fwd16<BF16, D>(g, q, k, v, o, lse, row_ptr, row_idx, n_qt, wg_order, stream);
  }
  return check_launch("gki_bsa_fwd");
}

}  // namespace

int fwd_tile_m(int dtype) { return dtype == kF32 ? kTileM : kTileMF; }

int fwd_dispatch(int dtype, int head_dim, const Geom& g, const void* q, const void* k, const void* v,
                 void* o, float* lse, const int32_t* row_ptr, const int32_t* row_idx, int n_qt,
                 const int32_t* wg_order, hipStream_t stream) {
  switch (head_dim) {
    case 16: return launch_fwd<16>(dtype, g, q, k, v, o, lse, row_ptr, row_idx, n_qt, wg_order, stream);
    case 32: return launch_fwd<32>(dtype, g, q, k, v, o, lse, row_ptr, row_idx, n_qt, wg_order, stream);
    case 64: return launch_fwd<64>(dtype, g, q, k, v, o, lse, row_ptr, row_idx, n_qt, wg_order, stream);
    case 128: return launch_fwd<128>(dtype, g, q, k, v, o, lse, row_ptr, row_idx, n_qt, wg_order, stream);
    default: return fail(2, "unsupported head_dim " + std::to_string(head_dim));
  }
}

}  // namespace gki
