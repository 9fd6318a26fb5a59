// Block-sparse StreamingLLM attention: backward kernels for gfx950.
//
// Replaces the reference's three Triton launches in
// `_BlockSparseFlashAttention.backward` (sparse_triton_kernel.py:719-777):
//   * `_bwd_preprocess_kernel` (sparse_triton_kernel.py:354-392),
//       Delta[q] = sum_d fp32(O) * fp32(dO) over the stored O, inside the dQ
//       kernel, which runs first and stores it (negated for 16-bit inputs) for
//       dK/dV. For 16-bit inputs it also stores, once per row, the LSE as the
//       16-bit kernels take it (second half of the row-term workspace): in base 2
//       at head_dim 64, P = exp2 of one fma of the score; elsewhere -LSE / scale,
//       from which the score accumulates, P = exp2 of one product. The fp32
//       kernels form P as exp2(fma(S, scale, -LSE) log2 e) from the stored LSE, as
//       the fp32 forward computed its exponents.
//   * dkdv_kernel   <- `_bwd_dkdv_kernel` (sparse_triton_kernel.py:394-509):
//       one workgroup per 64-row KV tile, loop over the kept q tiles of its
//       column (CSC list), P = exp(S - LSE), dV += P^T dO,
//       dS = P (dP - Delta) * scale, dK += dS^T Q. No atomics; one store per
//       tile.
//   * dq_kernel     <- `_bwd_dq_kernel` (sparse_triton_kernel.py:511-601):
//       one workgroup per 64-row q tile, loop over its kept kv tiles (CSR),
//       dQ += dS K.
// Casts follow the reference: P^T -> dO dtype for dV, dS -> Q/K dtype for
// dK/dQ, results stored in the input dtype.
//
// MI355X specifics: the dK/dV grid runs a work list in which long column walks
// (the sink column, kept by every q tile; the columns of a large grouped-query
// group) are cut into items of bounded length whose fp32 partials a reduce
// pass sums in a fixed order; items are XCD-remapped so neighbouring tiles of
// one head share L2.
#include "gki_common.cuh"

namespace gki {
namespace {

// fp32 gradients accumulate 16 rows at a time in a fresh accumulator, which is
// then added to the running sum with its rounding error kept in a compensation
// term: a long walk (the sink keys of a long sequence, |dV| ~ 10 over thousands of
// rows) then rounds like a short one. The result is sum + compensation. Within a
// walk the error is formed as for |sum| >= |x| (three operations less; a step
// that finds the sum smaller than 16 rows' worth keeps it to the rounding of x):
// per 16 rows at the time that the exact form takes per 32, whose plain sums left
// dQ, dK and dV 3-4.5% further from 64 bits. The exact form (TwoSum) joins whole sums.
__device__ inline void fold(floatx4& sum, floatx4& comp, const floatx4& x) {
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const float s = sum[i] + x[i];
    comp[i] += x[i] - (s - sum[i]);
    sum[i] = s;
  }
}
__device__ inline void two_sum_fold(floatx4& sum, floatx4& comp, const floatx4& x) {
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const float s = sum[i] + x[i];
    const float bp = s - sum[i];
    const float ap = s - bp;
    comp[i] += (sum[i] - ap) + (x[i] - bp);
    sum[i] = s;
  }
}

__device__ inline uint4 and4(const uint4& v, uint32_t m) {
  return make_uint4(v.x & m, v.y & m, v.z & m, v.w & m);
}

// Work item of workgroup b in the dK / dV grid: the items of one (b, kv head)
// are consecutive, XCD-remapped so that neighbouring kv tiles of a head (which
// share most q tiles) run on one XCD and meet in its L2.
struct KvItem {
  int kt, it0, it1, pslot;
};
__device__ inline KvItem kv_item_of(int b, int BH, const KvWork& w, int& bh) {
  const int wg = xcd_remap(b, w.n_items * BH);
  bh = wg / w.n_items;
  const int4 t = ((const int4*)w.items)[wg - bh * w.n_items];
  return {t.x, t.y, t.z, t.w};
}

// The same for items cut into `parts` workgroups each (work_parts_grid); bh < 0
// for a workgroup past the last.
__device__ inline KvItem kv_item_part_of(int b, int BH, int parts, const KvWork& w, int& bh, int& part) {
  const int wg = work_part_of(b, w.n_items * BH, parts, nullptr, part);
  bh = wg < 0 ? -1 : wg / w.n_items;
  if (wg < 0) return {0, 0, 0, -1};
  const int4 t = ((const int4*)w.items)[wg - bh * w.n_items];
  return {t.x, t.y, t.z, t.w};
}

// Sum of a split column's fp32 partials, in item order, cast to the storage
// type. A split column's 2 x 64 x D partial floats (dK then dV) are spread
// over D / 8 workgroups, one float4 per thread; the loads of four partials are
// issued together and added in item order (the sum is deterministic).
template <int D>
constexpr int kReduceWgPerTile = 2 * kTileN * D / (256 * 4);

template <typename T, int D>
__global__ __launch_bounds__(256) void dkdv_reduce_kernel(Geom g, KvWork w,
                                                          typename T::storage* __restrict__ dK,
                                                          typename T::storage* __restrict__ dV) {
  constexpr int TILE = kTileN * D;                     // floats of one dK (or dV) tile
  constexpr int STRIDE = 2 * TILE / 4;                 // float4s between two partials
  constexpr int WGT = kReduceWgPerTile<D>;
  const int rest = blockIdx.x / WGT, part = blockIdx.x - rest * WGT;
  const int bh = rest / w.n_split, s = rest - bh * w.n_split;
  const int kt = w.split[3 * s], p0 = w.split[3 * s + 1], np = w.split[3 * s + 2];
  const int idx = (part * 256 + threadIdx.x) * 4;      // first float of this thread
  const float4* src = (const float4*)(w.partials + ((size_t)bh * w.n_pslots + p0) * 2 * TILE + idx);
  float4 acc = make_float4(0.f, 0.f, 0.f, 0.f);
  int c = 0;
  if constexpr (T::is_f32) {           // compensated (Kahan) sum of the fp32 partials
    float4 comp = make_float4(0.f, 0.f, 0.f, 0.f);
    for (; c < np; ++c) {
      const float4 a = src[(size_t)c * STRIDE];
      const float ya = a.x - comp.x, yb = a.y - comp.y, yc = a.z - comp.z, yd = a.w - comp.w;
      const float ta = acc.x + ya, tb = acc.y + yb, tc = acc.z + yc, td = acc.w + yd;
      comp = make_float4((ta - acc.x) - ya, (tb - acc.y) - yb, (tc - acc.z) - yc, (td - acc.w) - yd);
      acc = make_float4(ta, tb, tc, td);
    }
  }
  for (; c + 4 <= np; c += 4) {
    const float4 a0 = src[(size_t)c * STRIDE], a1 = src[(size_t)(c + 1) * STRIDE];
    const float4 a2 = src[(size_t)(c + 2) * STRIDE], a3 = src[(size_t)(c + 3) * STRIDE];
    acc.x = (((acc.x + a0.x) + a1.x) + a2.x) + a3.x;
    acc.y = (((acc.y + a0.y) + a1.y) + a2.y) + a3.y;
    acc.z = (((acc.z + a0.z) + a1.z) + a2.z) + a3.z;
    acc.w = (((acc.w + a0.w) + a1.w) + a2.w) + a3.w;
  }
  for (; c < np; ++c) {
    const float4 a = src[(size_t)c * STRIDE];
    acc.x += a.x, acc.y += a.y, acc.z += a.z, acc.w += a.w;
  }
  const int which = idx / TILE, rem = idx - which * TILE;   // 4 floats of one row (D % 4 == 0)
  const int row = kt * kTileN + rem / D;
  if (row >= g.n_kv) return;
  typename T::storage* dst = (which ? dV : dK) + (size_t)bh * g.n_kv * D + (size_t)row * D + rem % D;
  dst[0] = T::from_float(acc.x);
  dst[1] = T::from_float(acc.y);
  dst[2] = T::from_float(acc.z);
  dst[3] = T::from_float(acc.w);
}

// ---------------------------------------------------------------------------
// dK / dV, 16-bit, in quadrants: wave w owns kv rows 32 (w & 1) .. +31 of the
// 64-row kv tile (K / V in registers as B operands) against q rows
// 32 (w >> 1) .. +31 of each q tile: one 32x32 block of S and of dP per wave and
// tile, whose accumulators (v_mfma_f32_32x32x16) are the operands of
// dV^T += dO^T P and dK^T += Q^T dS. Q and dO tiles row-major in LDS
// (double-buffered, staged by LDS-DMA), transposed operands by Lane32::cols.
// The two q halves' fp32 sums meet once, through LDS, at the end of the item
// (the qh = 0 wave adds the qh = 1 wave's, a fixed order).
// ---------------------------------------------------------------------------
// Head dims other than 64. At 128 the LDS was the bound (96 reads per 64 small
// MFMAs with 16 kv rows per wave; 48 per 32 large ones now), then the latency of
// operands read one at a time: B2 H32 on 8 kv heads N4096 D128 W1024 bf16, cycles
// per workgroup and tile 5147 -> 4370 with this layout; backward 0.607 -> 0.569 ms
// with it and 0.549 with the reads pinned ahead (B4 H8 N2000 D32 0.071 -> 0.055).
// At head_dim 64 the card's power is the bound (1.9-2.1 GHz under the backward)
// and this form, 7% fewer cycles at a 10% lower clock, ran 2-3% slower than the
// 16x16x32 quadrants below.
// FORM: Geom::bwd_form. A template parameter, so no form carries a branch.
template <typename T, int D, int FORM>
__global__ __launch_bounds__(256, D <= 32 ? 4 : FORM != kBwdPlain ? 2 : 1) void dkdv_kernel_16(
    Geom g, const uint16_t* __restrict__ Q, const uint16_t* __restrict__ K,
    const uint16_t* __restrict__ V, const uint16_t* __restrict__ dO, uint16_t* __restrict__ dK,
    uint16_t* __restrict__ dV, const float* __restrict__ LSE2, const float* __restrict__ Delta,
    const int32_t* __restrict__ col_ptr, const int32_t* __restrict__ col_idx, KvWork w) {
  // LSE2: -LSE / row_scale rows when ROW, else base-2 LSE rows; Delta: -Delta rows
  // (times the scale when PRE); both written by the dQ kernel, which runs first
  constexpr bool ROW = FORM != kBwdPlain, PRE = FORM == kBwdPre;
  constexpr int kAhead = 3;                    // operands read ahead (255 VGPRs at head_dim 128)
  constexpr int KS = D / 16;                   // k-steps of the contractions over d
  constexpr int DT = D >= 32 ? D / 32 : 1;     // 32-row tiles of dK^T / dV^T
  constexpr int TILE = 64 * D;
  // Q, Q, dO, dO; the waves' sums at the end
  constexpr int LDS16 = 4 * TILE > 2 * 2 * DT * 16 * 64 * 2 ? 4 * TILE : 2 * 2 * DT * 16 * 64 * 2;
  __shared__ __align__(16) uint16_t stile[LDS16];
  __shared__ __align__(16) float slse[2][64];
  __shared__ __align__(16) float sdlt[2][64];

  // one workgroup per (b, kv head, work item): a range of the kv tile's walk
  // over (q head of the group, CSC list entry), accumulated in registers
  const int BH = g.B * g.H_kv;
  int bh;
  const KvItem item = kv_item_of(blockIdx.x, BH, w, bh);
  // an empty column (no kept q tile) only writes zeros: its K / V rows are not read
  const bool has_work = item.it1 > item.it0;
  const int kt = item.kt;
  const size_t kb = (size_t)bh * g.n_kv * D;
  const int bhq0 = (bh / g.H_kv) * g.H + (bh % g.H_kv) * g.group;   // first q head
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lane = tid & 63, hi = lane >> 5, col = lane & 31;
  const Lane32<D> at0(lane);
  const int kh = wave & 1, qh = wave >> 1;
  const int k_w = kt * kTileN + 32 * kh;       // the wave's first kv row

  uint4 kf[KS], vf[KS];
  {
    const int my_kv = k_w + col;
    const bool ok = has_work && my_kv < g.n_kv;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      const size_t o = kb + (size_t)my_kv * D + 16 * ks + 8 * hi;
      kf[ks] = ok ? *(const uint4*)(K + o) : make_uint4(0, 0, 0, 0);
      vf[ks] = ok ? *(const uint4*)(V + o) : make_uint4(0, 0, 0, 0);
      if constexpr (FORM == kBwdRow) kf[ks] = and4(kf[ks], g.q_and);
      if constexpr (PRE) vf[ks] = scale8<T>(vf[ks], g.scale);
    }
  }
  floatx16 dk[DT], dv[DT];
#pragma unroll
  for (int i = 0; i < DT; ++i) dk[i] = dv[i] = splat16(0.f);

  const int e_beg = col_ptr[kt], e_end = col_ptr[kt + 1];
  DmaTile<D, 4, true> dma;
  dma.init(tid);
  // Rows past n_q are zeros in Q and dO (the DMA's range check); LSE / Delta
  // rows by a 4-byte LDS-DMA (waves 0 / 1, one lane per row; rows past n_q
  // re-read row n_q - 1, which only masked elements see).
  auto load_tile = [&](int q0, int bhq, int buf) {
    const size_t qb = (size_t)bhq * g.n_q * D;
    dma.load(Q + qb, q0, g.n_q, stile + buf * TILE);
    dma.load(dO + qb, q0, g.n_q, stile + (2 + buf) * TILE);
    if (wave < 2) {
      const float* src = (wave == 0 ? LSE2 : Delta) + (size_t)bhq * g.n_q + min(q0 + lane, g.n_q - 1);
      dma_load4(src, lds_addr(wave == 0 ? slse[buf] : sdlt[buf]));
    }
  };
  // iterations [it0, it1): iteration i visits list entry e_beg + i % L of q
  // head bhq0 + i / L; (e, bhq) advance together
  const int L = e_end - e_beg;
  const int n_it = item.it1 - item.it0;
  const int h0 = L > 0 ? item.it0 / L : 0;
  int e_nx = e_beg + (item.it0 - h0 * L), q_nx = bhq0 + h0;
  if (n_it > 0) load_tile((col_idx[e_nx] & kIdxMask) * kTileM, q_nx, 0);
  dma_wait();
  __syncthreads();

  const int kv_hi_wave = min(k_w + 31, g.n_kv - 1);
  for (int it = 0; it < n_it; ++it) {
    const int buf = it & 1;
    const int ent = col_idx[e_nx];
    if (++e_nx == e_end) {
      e_nx = e_beg;
      ++q_nx;
    }
    const int q0 = (ent & kIdxMask) * kTileM;
    const bool partial = (ent >> kPartialBit) & 1;
    if (it + 1 < n_it) load_tile((col_idx[e_nx] & kIdxMask) * kTileM, q_nx, buf ^ 1);
    const uint16_t* cq = stile + buf * TILE;
    const uint16_t* cdo = stile + (2 + buf) * TILE;
    const int qw0 = q0 + 32 * qh;              // the wave's first q row
    Lane32<D> at = at0;
    if constexpr (D >= 128) at.pin();          // its offsets' XORs per tile, not held in 14 registers
    // left out where none of the wave's rows sees one of its keys
    if (!tile_unseen(g, qw0, qw0 + 31, k_w, 32)) {
      const bool need_mask = partial || (qw0 + 32 > g.n_q) || (k_w + 31 >= g.n_kv) ||
                             !tile_all_visible(g, qw0, qw0 + 31, k_w, kv_hi_wave);
      // register r of lane (hi, col): q row qw0 + acc32_row(r, hi), kv row k_w + col.
      // The accumulators start at the row terms of their q rows: dP at -Delta, so
      // that it ends as dP - Delta (times the scale when PRE), and with ROW S at
      // -LSE / scale, so that P = exp2(S scale log2 e).
      floatx16 s, dp;
      const float* rd = &sdlt[buf][32 * qh + 4 * hi];
      const float* rl = &slse[buf][32 * qh + 4 * hi];
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const float4 l = *(const float4*)(rl + 8 * q), v = *(const float4*)(rd + 8 * q);
        s[4 * q] = ROW ? l.x : 0.f, s[4 * q + 1] = ROW ? l.y : 0.f;
        s[4 * q + 2] = ROW ? l.z : 0.f, s[4 * q + 3] = ROW ? l.w : 0.f;
        dp[4 * q] = v.x, dp[4 * q + 1] = v.y, dp[4 * q + 2] = v.z, dp[4 * q + 3] = v.w;
      }
      // S and dP in turn, each operand read kAhead products ahead (the order is
      // pinned: left alone the compiler has each product wait for its own read)
      auto row_op = [&](int i) { return at.rows(i & 1 ? cdo : cq, qh, i >> 1); };
      uint4 op[kAhead];
#pragma unroll
      for (int i = 0; i < kAhead && i < 2 * KS; ++i) op[i] = row_op(i);
#pragma unroll
      for (int i = 0; i < 2 * KS; ++i) {
        if (i & 1) dp = T::mfma32(op[i % kAhead], vf[i >> 1], dp);
        else s = T::mfma32(op[i % kAhead], kf[i >> 1], s);
        if (i + kAhead < 2 * KS) op[i % kAhead] = row_op(i + kAhead);
        __builtin_amdgcn_sched_barrier(0);
      }
      if constexpr (ROW) {
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          s[r] = __builtin_amdgcn_exp2f(s[r] * g.row_scale_log2);
          dp[r] = PRE ? s[r] * dp[r] : s[r] * (dp[r] * g.scale);
        }
      } else {
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const float4 l = *(const float4*)(rl + 8 * q);             // base-2 LSE
          const float lv[4] = {l.x, l.y, l.z, l.w};
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const int r = 4 * q + i;
            s[r] = __builtin_amdgcn_exp2f(__builtin_fmaf(s[r], g.scale_log2, -lv[i]));
            dp[r] = s[r] * (dp[r] * g.scale);
          }
        }
      }
      // Masked elements: P = dS = 0 (a bit select, so an exp that overflowed on
      // an invisible element cannot leak). One uniform branch per tile keeps the
      // selects off the tiles that need no mask.
      if (need_mask) {
        const uint64_t bits = col_valid_bits(opaque_blocks(g), k_w + (lane_now() & 31), q0, partial);
        const LaneBits32 vis(qh ? (uint32_t)(bits >> 32) : (uint32_t)bits, lane_now() >> 5);
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int m = vis.mask(r);
          s[r] = __int_as_float(__float_as_int(s[r]) & m);
          dp[r] = __int_as_float(__float_as_int(dp[r]) & m);
        }
      }
      uint4 pk[2][2];                          // P and dS, 16 q rows each
#pragma unroll
      for (int st = 0; st < 2; ++st) pk[st][0] = pack8<T>(s, st), pk[st][1] = pack8<T>(dp, st);
      auto col_op = [&](int i) { return at.cols(i & 1 ? cq : cdo, 2 * qh + i / (2 * DT), (i >> 1) % DT); };
      uint4 ot[kAhead];
#pragma unroll
      for (int i = 0; i < kAhead && i < 4 * DT; ++i) ot[i] = col_op(i);
#pragma unroll
      for (int i = 0; i < 4 * DT; ++i) {
        const int st = i / (2 * DT), dt = (i >> 1) % DT;
        if (i & 1) dk[dt] = T::mfma32(ot[i % kAhead], pk[st][1], dk[dt]);
        else dv[dt] = T::mfma32(ot[i % kAhead], pk[st][0], dv[dt]);
        if (i + kAhead < 4 * DT) ot[i % kAhead] = col_op(i + kAhead);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    dma_wait();        // the next tile's LDS-DMA has landed before the barrier
    __syncthreads();
  }

  // the q halves' sums meet in LDS (the Q / dO buffers are free: every wave
  // passed the loop's last barrier): qh = 1 waves store, qh = 0 waves add theirs
  floatx4* red = (floatx4*)stile + kh * (2 * DT * 4 * 64);
  const int lane_e = lane_now(), hi_e = lane_e >> 5;
  if (qh == 1) {
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        red[((2 * dt) * 4 + q) * 64 + lane_e] = floatx4{dk[dt][4 * q], dk[dt][4 * q + 1], dk[dt][4 * q + 2], dk[dt][4 * q + 3]};
        red[((2 * dt + 1) * 4 + q) * 64 + lane_e] = floatx4{dv[dt][4 * q], dv[dt][4 * q + 1], dv[dt][4 * q + 2], dv[dt][4 * q + 3]};
      }
  }
  __syncthreads();
  if (qh == 1) return;
  const bool split = item.pslot >= 0;          // a split column: fp32 partials for the reduce
  const int row = 32 * kh + (lane_e & 31);     // of the kv tile
  if (!split && kt * kTileN + row >= g.n_kv) return;
  float* part = w.partials + ((size_t)bh * w.n_pslots + (split ? item.pslot : 0)) * 2 * TILE + (size_t)row * D;
  const size_t out = kb + (size_t)(kt * kTileN + row) * D;
#pragma unroll
  for (int dt = 0; dt < DT; ++dt)
#pragma unroll
    for (int q = 0; q < (D >= 32 ? 4 : 2); ++q) {      // D = 16: elements past 15 do not exist
      const floatx4 rk = red[((2 * dt) * 4 + q) * 64 + lane_e], rv = red[((2 * dt + 1) * 4 + q) * 64 + lane_e];
      floatx4 a, b;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        a[i] = dk[dt][4 * q + i] + rk[i];
        b[i] = dv[dt][4 * q + i] + rv[i];
      }
      const int d0 = 32 * dt + 8 * q + 4 * hi_e;
      if (split) {
        *(floatx4*)(part + d0) = a;
        *(floatx4*)(part + TILE + d0) = b;
      } else {
        *(uint2*)(dK + out + d0) = make_uint2(pack2<T>(a[0], a[1]), pack2<T>(a[2], a[3]));
        *(uint2*)(dV + out + d0) = make_uint2(pack2<T>(b[0], b[1]), pack2<T>(b[2], b[3]));
      }
    }
}

// ---------------------------------------------------------------------------
// dK / dV, 16-bit, head_dim 64, in quadrants: wave w owns kv rows
// 32 (w & 1) .. +31 of the 64-row kv tile (two 16-row blocks, K / V in
// registers as the B operands) against q rows 32 (w >> 1) .. +31 of each q
// tile (rho subtiles 2 qh, 2 qh + 1). Every Q / dO row read, LSE / Delta read
// and transposed Q / dO read from LDS then feeds the MFMAs of both kv blocks:
// 28 LDS reads per 32 MFMAs per wave and tile instead of 56. The two q
// halves' fp32 dK / dV sums meet once, through LDS, at the end of the item
// (the qh = 0 wave adds the qh = 1 wave's, a fixed order). Waves leave out the
// 32 x 32 blocks they cannot see: B4 H16 N8192 W1024 fp16 backward 0.586 ->
// 0.577 ms (level on walks of 65, B1 H16 N131072 W4096).
// ---------------------------------------------------------------------------
template <typename T, bool PRE>
__global__ __launch_bounds__(256, 3) void dkdv_kernel_q64(
    Geom g, const uint16_t* __restrict__ Q, const uint16_t* __restrict__ K,
    const uint16_t* __restrict__ V, const uint16_t* __restrict__ dO, uint16_t* __restrict__ dK,
    uint16_t* __restrict__ dV, const float* __restrict__ LSE2, const float* __restrict__ Delta,
    const int32_t* __restrict__ col_ptr, const int32_t* __restrict__ col_idx, KvWork w) {
  // LSE2: base-2 LSE rows; Delta: -Delta rows (times the scale when PRE),
  // both written by the dQ kernel, which runs first
  constexpr int D = 64, KS = 2, DT = 4;
  __shared__ __align__(16) uint16_t sq[2][64 * D];
  __shared__ __align__(16) uint16_t sdo[2][64 * D];
  __shared__ __align__(16) float slse[2][64];
  __shared__ __align__(16) float sdlt[2][64];

  const int BH = g.B * g.H_kv;
  int bh;
  const KvItem item = kv_item_of(blockIdx.x, BH, w, bh);
  // an empty column (no kept q tile) only writes zeros: its K / V rows are not read
  const bool has_work = item.it1 > item.it0;
  const int kt = item.kt;
  const size_t kb = (size_t)bh * g.n_kv * D;
  const int bhq0 = (bh / g.H_kv) * g.H + (bh % g.H_kv) * g.group;   // first q head
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  const int grp = lane >> 4, col = lane & 15;
  const int kh = __builtin_amdgcn_readfirstlane(wave & 1), qh = __builtin_amdgcn_readfirstlane(wave >> 1);
  const int k_w = kt * kTileN + 32 * kh;       // the wave's first kv row

  uint4 kf[2][KS], vf[2][KS];
#pragma unroll
  for (int b = 0; b < 2; ++b) {
    const int my_kv = k_w + 16 * b + col;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      const int d0 = 32 * ks + 8 * grp;
      const bool ok = has_work && my_kv < g.n_kv;
      kf[b][ks] = ok ? *(const uint4*)(K + kb + (size_t)my_kv * D + d0) : make_uint4(0, 0, 0, 0);
      vf[b][ks] = ok ? *(const uint4*)(V + kb + (size_t)my_kv * D + d0) : make_uint4(0, 0, 0, 0);
      if constexpr (PRE) vf[b][ks] = scale8<T>(vf[b][ks], g.scale);
    }
  }
  floatx4 dk[2][DT], dv[2][DT];
#pragma unroll
  for (int b = 0; b < 2; ++b)
#pragma unroll
    for (int i = 0; i < DT; ++i) dk[b][i] = dv[b][i] = floatx4{0.f, 0.f, 0.f, 0.f};

  const int e_beg = col_ptr[kt], e_end = col_ptr[kt + 1];
  DmaTile<D> dma;
  dma.init(tid);
  const int wave_u = __builtin_amdgcn_readfirstlane(wave);
  auto load_tile = [&](int q0, int bhq, int buf) {
    const size_t qb = (size_t)bhq * g.n_q * D;
    dma.load(Q + qb, q0, g.n_q, sq[buf]);      // rows past n_q: zeros
    dma.load(dO + qb, q0, g.n_q, sdo[buf]);
    if (wave_u < 2) {
      const float* src = (wave_u == 0 ? LSE2 : Delta) + (size_t)bhq * g.n_q + min(q0 + lane, g.n_q - 1);
      dma_load4(src, lds_addr(wave_u == 0 ? slse[buf] : sdlt[buf]));
    }
  };
  const int L = e_end - e_beg;
  const int n_it = item.it1 - item.it0;
  const int h0 = L > 0 ? item.it0 / L : 0;
  int e_nx = e_beg + (item.it0 - h0 * L), q_nx = bhq0 + h0;
  if (n_it > 0) load_tile((col_idx[e_nx] & kIdxMask) * kTileM, q_nx, 0);
  dma_wait();
  __syncthreads();

  const int kv_hi_wave = min(k_w + 31, g.n_kv - 1);
  for (int it = 0; it < n_it; ++it) {
    const int buf = it & 1;
    const int ent = col_idx[e_nx];
    if (++e_nx == e_end) {
      e_nx = e_beg;
      ++q_nx;
    }
    const int q0 = (ent & kIdxMask) * kTileM;
    const bool partial = (ent >> kPartialBit) & 1;
    if (it + 1 < n_it) load_tile((col_idx[e_nx] & kIdxMask) * kTileM, q_nx, buf ^ 1);
    const uint16_t* cq = sq[buf];
    const uint16_t* cdo = sdo[buf];
    const int qw0 = q0 + 32 * qh;              // the wave's first q row
    // left out where none of the wave's rows sees one of its keys
    if (!tile_unseen(g, qw0, qw0 + 31, k_w, 32)) {
      const bool need_mask = partial || (qw0 + 32 > g.n_q) || (k_w + 31 >= g.n_kv) ||
                             !tile_all_visible(g, qw0, min(qw0 + 31, g.n_q - 1), k_w, kv_hi_wave);
      floatx4 p[2][2], ds[2][2];                 // [subtile 2 qh + u][kv block]
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        const int t = 2 * qh + u;
        const int qr0 = rho(t, 4 * grp);
        const float4 lse4 = *(const float4*)(&slse[buf][qr0]);
        const float4 ndl4 = *(const float4*)(&sdlt[buf][qr0]);
        floatx4 sc[2], dp[2];
#pragma unroll
        for (int b = 0; b < 2; ++b) {
          sc[b] = floatx4{0.f, 0.f, 0.f, 0.f};
          dp[b] = floatx4{ndl4.x, ndl4.y, ndl4.z, ndl4.w};
        }
        const int r = rho(t, col);
        mfma_priority_hi<true>();
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
          const int d0 = 32 * ks + 8 * grp;
          const uint4 aq = lds_row8<D>(cq, r, d0);
          const uint4 ad = lds_row8<D>(cdo, r, d0);
#pragma unroll
          for (int b = 0; b < 2; ++b) {
            sc[b] = T::mfma(aq, kf[b][ks], sc[b]);
            dp[b] = T::mfma(ad, vf[b][ks], dp[b]);
          }
        }
        mfma_priority_lo<true>();
        const float lv[4] = {lse4.x, lse4.y, lse4.z, lse4.w};
#pragma unroll
        for (int b = 0; b < 2; ++b)
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const float pv = __builtin_amdgcn_exp2f(__builtin_fmaf(sc[b][i], g.scale_log2, -lv[i]));
            p[u][b][i] = pv;
            ds[u][b][i] = PRE ? pv * dp[b][i] : pv * (dp[b][i] * g.scale);
          }
      }
      if (need_mask) {     // masked elements: P = dS = 0 (bit select)
#pragma unroll
        for (int b = 0; b < 2; ++b) {
          const LaneBits vis(col_valid_bits(g, k_w + 16 * b + col, q0, partial), grp);
          const uint32_t wq = qh ? vis.w[1] : vis.w[0];   // uniform select, not an index
#pragma unroll
          for (int u = 0; u < 2; ++u)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
              const int m = __builtin_amdgcn_sbfe((int)wq, 4 * u + i, 1);   // 0 or -1
              p[u][b][i] = __int_as_float(__float_as_int(p[u][b][i]) & m);
              ds[u][b][i] = __int_as_float(__float_as_int(ds[u][b][i]) & m);
            }
        }
      }
      uint4 ap[2], as[2];
#pragma unroll
      for (int b = 0; b < 2; ++b) {
        ap[b] = pack8<T>(p[0][b], p[1][b]);
        as[b] = pack8<T>(ds[0][b], ds[1][b]);
      }
      mfma_priority_hi<true>();
#pragma unroll
      for (int dt = 0; dt < DT; ++dt) {
        const uint4 bo = lds_tr8<D>(cdo, 32 * qh, 16 * dt, lane);
        const uint4 bq = lds_tr8<D>(cq, 32 * qh, 16 * dt, lane);
#pragma unroll
        for (int b = 0; b < 2; ++b) {
          dv[b][dt] = T::mfma(ap[b], bo, dv[b][dt]);
          dk[b][dt] = T::mfma(as[b], bq, dk[b][dt]);
        }
      }
      mfma_priority_lo<true>();
    }
    dma_wait();        // the next tile's LDS-DMA has landed before the barrier
    __syncthreads();
  }

  // the q-half sums meet in LDS (the Q / dO buffers are free: every wave passed
  // the loop's last barrier): qh = 1 waves store, qh = 0 waves add theirs first
  floatx4* red = (floatx4*)&sq[0][0] + kh * (4 * DT * 64);
  if (qh == 1) {
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
      for (int dt = 0; dt < DT; ++dt) {
        red[((2 * b + 0) * DT + dt) * 64 + lane] = dk[b][dt];
        red[((2 * b + 1) * DT + dt) * 64 + lane] = dv[b][dt];
      }
  }
  __syncthreads();
  if (qh == 1) return;
#pragma unroll
  for (int b = 0; b < 2; ++b)
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) {
      dk[b][dt] += red[((2 * b + 0) * DT + dt) * 64 + lane];
      dv[b][dt] += red[((2 * b + 1) * DT + dt) * 64 + lane];
    }
  // accumulators: lane holds kv rows k_w + 16 b + 4 grp + i, column 16 dt + col
  if (item.pslot >= 0) {             // a split column: fp32 partials for the reduce
    float* pk = w.partials + ((size_t)bh * w.n_pslots + item.pslot) * 2 * (kTileN * D);
    float* pv = pk + kTileN * D;
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int r = 32 * kh + 16 * b + 4 * grp + i;
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) {
          pk[r * D + 16 * dt + col] = dk[b][dt][i];
          pv[r * D + 16 * dt + col] = dv[b][dt][i];
        }
      }
    return;
  }
#pragma unroll
  for (int b = 0; b < 2; ++b)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int row = k_w + 16 * b + 4 * grp + i;
      if (row < g.n_kv) {
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) {
          dK[kb + (size_t)row * D + 16 * dt + col] = T::from_float(dk[b][dt][i]);
          dV[kb + (size_t)row * D + 16 * dt + col] = T::from_float(dv[b][dt][i]);
        }
      }
    }
}

// ---------------------------------------------------------------------------
// dK / dV, fp32
// ---------------------------------------------------------------------------
// Bound by the fp32 matrix cores and, beside them, the VALU (exponents, the
// compensated folds): B1 H16 N8192 D64 W1024 backward 1.97 -> 1.30 ms (dK/dV and dQ
// 803 us at the nominal MFMA rate), D128 N4096 2.08 -> 1.41, against 4-byte LDS
// reads, tiles staged through registers behind two barriers and a separate Delta
// launch. Three waves per SIMD ran 12% slower than two (head_dim 64).
// As the forward, a workgroup's four waves are KB blocks of 16 kv rows x 4 / KB
// shares of the q rows of each staged step (16 rows each; two subtiles when
// KB = 4), and an item of the work list is 4 / KB workgroups. The shares' sums
// meet through LDS at the end, in order.
template <int D, int KB>
__global__ __launch_bounds__(256, D >= 128 || (D == 64 && KB == 1) ? 1 : 2) void dkdv_kernel_32(
    Geom g, const float* __restrict__ Q, const float* __restrict__ K, const float* __restrict__ V,
    const float* __restrict__ dO, float* __restrict__ dK, float* __restrict__ dV,
    const float* __restrict__ LSE, const float* __restrict__ Delta,
    const int32_t* __restrict__ col_ptr, const int32_t* __restrict__ col_idx, KvWork w) {
  // LSE: the forward's natural LSE; Delta: rowsum(O dO) from the dQ kernel, which runs first
  constexpr int DJ = D / 16;
  constexpr int QS = 4 / KB;                 // q-row shares
  constexpr int TR = QS == 4 ? 64 : 32;      // q rows per staged step
  constexpr int SUBS = TR / (16 * QS);
  constexpr int HALVES = kTileM / TR;
  constexpr int DV = D >= 64 ? D / 64 : 1;
  constexpr int DE = D / (16 * DV);
  __shared__ __align__(16) float sq[2][TR * D];
  __shared__ __align__(16) float sdo[2][TR * D];
  __shared__ __align__(16) float slse[2][64];
  __shared__ __align__(16) float sdlt[2][64];

  const int BH = g.B * g.H_kv;
  int bh, part;
  const KvItem item = kv_item_part_of(blockIdx.x, BH, QS, w, bh, part);
  if (bh < 0) return;
  // an empty column (no kept q tile) only writes zeros: its K / V rows are not read
  const bool has_work = item.it1 > item.it0;
  const int kt = item.kt;
  const size_t kb = (size_t)bh * g.n_kv * D;
  const int bhq0 = (bh / g.H_kv) * g.H + (bh % g.H_kv) * g.group;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int grp = lane >> 4, col = lane & 15;
  const int share = wave / KB;
  const int kr0 = 16 * (part * KB + wave % KB);          // the wave's rows of the kv tile
  const int k_w = kt * kTileN + kr0;
  const int my_kv = k_w + col;

  floatx4 kf[DJ], vf[DJ];
#pragma unroll
  for (int j = 0; j < DJ; ++j) {
    const bool ok = has_work && my_kv < g.n_kv;
    const size_t at = kb + (size_t)my_kv * D + 16 * j + 4 * grp;
    kf[j] = ok ? *(const floatx4*)(K + at) : floatx4{0.f, 0.f, 0.f, 0.f};
    vf[j] = ok ? *(const floatx4*)(V + at) : floatx4{0.f, 0.f, 0.f, 0.f};
  }
  // running sums and their compensation; tile (v, e) column x is element 64 v + DE x + e
  floatx4 dk[DV][DE], dv[DV][DE], ck[DV][DE], cv[DV][DE];
#pragma unroll
  for (int v = 0; v < DV; ++v)
#pragma unroll
    for (int e = 0; e < DE; ++e) dk[v][e] = dv[v][e] = ck[v][e] = cv[v][e] = floatx4{0.f, 0.f, 0.f, 0.f};

  const int e_beg = col_ptr[kt], e_end = col_ptr[kt + 1];
  DmaTileF32<D, TR> dma;
  dma.init(tid);
  const int L = e_end - e_beg;
  const int n_step = (item.it1 - item.it0) * HALVES;
  const int h0 = L > 0 ? item.it0 / L : 0;
  int e_nx = e_beg + (item.it0 - h0 * L), q_nx = bhq0 + h0;
  auto stage = [&](int s, int buf) {
    const int q0 = (col_idx[e_nx] & kIdxMask) * kTileM + (s % HALVES) * TR;
    const size_t qb = (size_t)q_nx * g.n_q * D;
    dma.load(Q + qb, q0, g.n_q, sq[buf]);
    dma.load(dO + qb, q0, g.n_q, sdo[buf]);
    if (wave < 2) {      // rows past n_q re-read the last one, which only masked elements see
      const float* src = (wave == 0 ? LSE : Delta) + (size_t)q_nx * g.n_q + min(q0 + lane, g.n_q - 1);
      dma_load4(src, lds_addr(wave == 0 ? slse[buf] : sdlt[buf]));
    }
  };
  dma_wait();          // the K / V loads, before any LDS-DMA is in flight
  if (n_step > 0) stage(0, 0);
  dma_wait();
  __syncthreads();

  const int kv_hi = min(k_w + 15, g.n_kv - 1);
  for (int s = 0; s < n_step; ++s) {
    const int buf = s & 1;
    const int ent = col_idx[e_nx];
    if (s % HALVES == HALVES - 1 && ++e_nx == e_end) {
      e_nx = e_beg;
      ++q_nx;
    }
    if (s + 1 < n_step) stage(s + 1, buf ^ 1);
    const float *cq = sq[buf], *cdo = sdo[buf];
    const int r0 = 16 * SUBS * share;                    // the wave's first q row of the step
    const int q0 = (ent & kIdxMask) * kTileM + (s % HALVES) * TR + r0;
    const bool partial = (ent >> kPartialBit) & 1;
    const bool need_mask = partial || (q0 + 16 * SUBS > g.n_q) || (k_w + 15 >= g.n_kv) ||
                           !tile_all_visible(g, q0, q0 + 16 * SUBS - 1, k_w, kv_hi);
    uint64_t bits = ~0ull;
    if (need_mask) bits = col_valid_bits(g, my_kv, q0, partial);
    const LaneBits16 vis(bits, grp);
#pragma unroll
    for (int t = 0; t < SUBS; ++t) {
      const int r = r0 + 16 * t;
      floatx4 fk[DV][DE], fv[DV][DE];  // these 16 rows, folded in compensated
#pragma unroll
      for (int v = 0; v < DV; ++v)
#pragma unroll
        for (int e = 0; e < DE; ++e) fk[v][e] = fv[v][e] = floatx4{0.f, 0.f, 0.f, 0.f};
      const floatx4 sc = mfma_f32_dot<4 * DJ>(
          [&](int j) { return *(const floatx4*)(cq + off_f32<D>(r + col, 4 * j + grp)); }, kf);
      const floatx4 dp = mfma_f32_dot<4 * DJ>(
          [&](int j) { return *(const floatx4*)(cdo + off_f32<D>(r + col, 4 * j + grp)); }, vf);
      const floatx4 lse4 = *(const floatx4*)(&slse[buf][r + 4 * grp]);
      const floatx4 dlt4 = *(const floatx4*)(&sdlt[buf][r + 4 * grp]);
      floatx4 pv, ds;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        pv[i] = __builtin_amdgcn_exp2f(__builtin_fmaf(sc[i], g.scale, -lse4[i]) * kLog2e);
        if (need_mask) pv[i] = vis.keep(t, i, pv[i]);
        ds[i] = pv[i] * (dp[i] - dlt4[i]) * g.scale;
      }
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int v = 0; v < DV; ++v) {
          const floatx4 xo = cols_f32<D, DE>(cdo, r + 4 * grp + i, v, col);
          const floatx4 xq = cols_f32<D, DE>(cq, r + 4 * grp + i, v, col);
#pragma unroll
          for (int e = 0; e < DE; ++e) {
            fv[v][e] = mfma_f32(pv[i], xo[e], fv[v][e]);
            fk[v][e] = mfma_f32(ds[i], xq[e], fk[v][e]);
          }
        }
#pragma unroll
      for (int v = 0; v < DV; ++v)
#pragma unroll
        for (int e = 0; e < DE; ++e) {
          fold(dk[v][e], ck[v][e], fk[v][e]);
          fold(dv[v][e], cv[v][e], fv[v][e]);
        }
    }
    dma_wait();        // the next step's LDS-DMA has landed before the barrier
    __syncthreads();
  }
  if constexpr (QS > 1) {
    // shares 1 .. QS - 1 hand their sums over through LDS (free: every wave
    // passed the last barrier); share 0 folds them in, in order
    constexpr int SZ = 2 * 2 * 16 * D;                   // dk, ck, dv, cv of a wave
    static_assert((QS - 1) * KB * SZ / 2 <= 2 * TR * D, "half of the sums fits each staging array");
    float* red = &sq[0][0];
    float* red2 = &sdo[0][0];
    const int blk = wave % KB;
    // dk / ck through sq, dv / cv through sdo
    const size_t at = ((size_t)(share - 1) * KB + blk) * (SZ / 2) + lane;
    if (share > 0) {
#pragma unroll
      for (int v = 0; v < DV; ++v)
#pragma unroll
        for (int e = 0; e < DE; ++e)
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const size_t o = at + 128 * ((v * DE + e) * 4 + i);
            red[o] = dk[v][e][i];
            red[o + 64] = ck[v][e][i];
            red2[o] = dv[v][e][i];
            red2[o + 64] = cv[v][e][i];
          }
    }
    __syncthreads();
    if (share > 0) return;
#pragma unroll
    for (int x = 1; x < QS; ++x) {
      const size_t from = ((size_t)(x - 1) * KB + blk) * (SZ / 2) + lane;
#pragma unroll
      for (int v = 0; v < DV; ++v)
#pragma unroll
        for (int e = 0; e < DE; ++e) {
          floatx4 a, b;
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const size_t o = from + 128 * ((v * DE + e) * 4 + i);
            a[i] = red[o];
            b[i] = red2[o];
            ck[v][e][i] += red[o + 64];
            cv[v][e][i] += red2[o + 64];
          }
          two_sum_fold(dk[v][e], ck[v][e], a);
          two_sum_fold(dv[v][e], cv[v][e], b);
        }
    }
  }
#pragma unroll
  for (int v = 0; v < DV; ++v)
#pragma unroll
    for (int e = 0; e < DE; ++e) {
      dk[v][e] += ck[v][e];
      dv[v][e] += cv[v][e];
    }
  // lane: kv rows 4 grp + i of the wave's 16, elements 64 v + DE col + e
  const bool split = item.pslot >= 0;                    // a split column: partials for the reduce
  float* pk = split ? w.partials + ((size_t)bh * w.n_pslots + item.pslot) * 2 * (kTileN * D) + kr0 * D
                    : dK + kb + (size_t)k_w * D;
  float* pv = split ? w.partials + ((size_t)bh * w.n_pslots + item.pslot) * 2 * (kTileN * D) + (kTileN + kr0) * D
                    : dV + kb + (size_t)k_w * D;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int row = 4 * grp + i;
    if (!split && k_w + row >= g.n_kv) continue;
#pragma unroll
    for (int v = 0; v < DV; ++v) {
      const int c = row * D + 64 * v + DE * col;
      if constexpr (DE == 4) {
        *(floatx4*)(pk + c) = floatx4{dk[v][0][i], dk[v][1][i], dk[v][2][i], dk[v][3][i]};
        *(floatx4*)(pv + c) = floatx4{dv[v][0][i], dv[v][1][i], dv[v][2][i], dv[v][3][i]};
      } else {
#pragma unroll
        for (int e = 0; e < DE; ++e) {
          pk[c + e] = dk[v][e][i];
          pv[c + e] = dv[v][e][i];
        }
      }
    }
  }
}

// ---------------------------------------------------------------------------
// dQ, 16-bit, in quadrants: wave w owns q rows 32 (w >> 1) .. +31 of the 64-row
// q tile (Q / dO in registers as B operands) against kv rows 32 (w & 1) .. +31 of
// each kv tile; the 32x32 block of dS^T is the operand of dQ^T += K^T dS^T. K
// and V tiles row-major in LDS (double-buffered, staged by LDS-DMA). The two kv
// halves' fp32 sums meet once, through LDS, at the end (the kh = 0 wave adds
// the kh = 1 wave's, a fixed order).
// ---------------------------------------------------------------------------
template <typename T, int D, int FORM>
__global__ __launch_bounds__(256, D > 64 ? 2 : 4) void dq_kernel_16(
    Geom g, const uint16_t* __restrict__ Q, const uint16_t* __restrict__ K,
    const uint16_t* __restrict__ V, const uint16_t* __restrict__ O, const uint16_t* __restrict__ dO,
    uint16_t* __restrict__ dQ, const float* __restrict__ LSE, float* __restrict__ Delta,
    const int32_t* __restrict__ row_ptr, const int32_t* __restrict__ row_idx, int n_qt,
    const int32_t* __restrict__ dq_order) {
  constexpr bool ROW = FORM != kBwdPlain, PRE = FORM == kBwdPre;
  constexpr int kAhead = 4;                    // operands read ahead
  constexpr int KS = D / 16;
  constexpr int DT = D >= 32 ? D / 32 : 1;
  constexpr int TILE = 64 * D;
  constexpr int LDS16 = 4 * TILE > 2 * DT * 16 * 64 * 2 ? 4 * TILE : 2 * DT * 16 * 64 * 2;
  __shared__ __align__(16) uint16_t stile[LDS16];      // K, K, V, V; the waves' sums at the end

  const int n_wg = n_qt * g.B * g.H;
  const int wg = work_of(blockIdx.x, n_wg, dq_order);
  if (wg < 0) return;
  const int bh = wg / n_qt, qt = wg - bh * n_qt;
  const size_t qb = (size_t)bh * g.n_q * D;
  const size_t kb = (size_t)kv_bh(g, bh) * g.n_kv * D;
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lane = tid & 63, hi = lane >> 5, col = lane & 31;
  const Lane32<D> at(lane);
  const int qh = wave >> 1, kh = wave & 1;
  const int q0w = qt * kTileM + 32 * qh;       // the wave's first q row

  uint4 qf[KS], df[KS];
  float lse2, ndlt;
  {
    const int my_q = q0w + col;
    const bool ok = my_q < g.n_q;
    float part = 0.f;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      const size_t o = qb + (size_t)my_q * D + 16 * ks + 8 * hi;
      qf[ks] = ok ? *(const uint4*)(Q + o) : make_uint4(0, 0, 0, 0);
      df[ks] = ok ? *(const uint4*)(dO + o) : make_uint4(0, 0, 0, 0);
      // Delta = rowsum(O * dO) in fp32 over the stored O (the preprocessing pass,
      // sparse_triton_kernel.py:354-392, fused here): the lane already holds its
      // half of the row's dO, the two halves are summed across. Every q row has
      // exactly one dQ workgroup, which writes it (and the LSE's form) for the
      // dK/dV kernel that runs next.
      if (ok) {
        const uint4 o4 = *(const uint4*)(O + o);
        const uint16_t* ho = (const uint16_t*)&o4;
        const uint16_t* hd = (const uint16_t*)&df[ks];
#pragma unroll
        for (int i = 0; i < 8; ++i) part += T::to_float(ho[i]) * T::to_float(hd[i]);
      }
    }
    // the row's start of S: -LSE / row_scale with ROW, else (added after) the LSE in
    // base 2; one rounding, once per row
    const float lse = ok ? LSE[(size_t)bh * g.n_q + my_q] : 0.f;
    lse2 = ROW ? (float)(-(double)lse / (double)g.row_scale) : lse_base2(lse);
    // Stored negated: both kernels start their dP accumulators at -Delta, so
    // they end as dP - Delta. With PRE the dO operand and -Delta carry the scale.
    ndlt = PRE ? -half_sum(part) * g.scale : -half_sum(part);
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      if constexpr (FORM == kBwdRow) qf[ks] = and4(qf[ks], g.q_and);
      if constexpr (PRE) df[ks] = scale8<T>(df[ks], g.scale);
    }
    if (ok && hi == 0 && kh == 0) {            // the two kv-half waves hold the same rows
      Delta[(size_t)bh * g.n_q + my_q] = ndlt;
      Delta[(size_t)g.B * g.H * g.n_q + (size_t)bh * g.n_q + my_q] = lse2;
    }
  }
  floatx16 dq[DT];
#pragma unroll
  for (int i = 0; i < DT; ++i) dq[i] = splat16(0.f);

  const int e_beg = row_ptr[qt], e_end = row_ptr[qt + 1];
  DmaTile<D, 4, true> dma;
  dma.init(tid);
  auto stage = [&](int k0, int buf) {
    dma.load(K + kb, k0, g.n_kv, stile + buf * TILE);
    dma.load(V + kb, k0, g.n_kv, stile + (2 + buf) * TILE);
  };
  if (e_beg < e_end) stage((row_idx[e_beg] & kIdxMask) * kTileN, 0);
  dma_wait();
  __syncthreads();
  for (int e = e_beg; e < e_end; ++e) {
    const int buf = (e - e_beg) & 1;
    const int ent = row_idx[e];
    const int k0 = (ent & kIdxMask) * kTileN;
    const bool partial = (ent >> kPartialBit) & 1;
    if (e + 1 < e_end) stage((row_idx[e + 1] & kIdxMask) * kTileN, buf ^ 1);
    const uint16_t* ck = stile + buf * TILE;
    const uint16_t* cv = stile + (2 + buf) * TILE;
    const int kw0 = k0 + 32 * kh;              // the wave's first kv row
    // left out where none of the wave's rows sees one of its keys
    if (!tile_unseen(g, q0w, q0w + 31, kw0, 32)) {
      const bool need_mask = partial || (q0w + 31 >= g.n_q) || (kw0 + 32 > g.n_kv) ||
                             !tile_all_visible(g, q0w, q0w + 31, kw0, kw0 + 31);
      floatx16 s = splat16(ROW ? lse2 : 0.f), dp = splat16(ndlt);
      // operands read kAhead products ahead, in a pinned order (as in dK/dV)
      auto row_op = [&](int i) { return at.rows(i & 1 ? cv : ck, kh, i >> 1); };
      uint4 op[kAhead];
#pragma unroll
      for (int i = 0; i < kAhead && i < 2 * KS; ++i) op[i] = row_op(i);
#pragma unroll
      for (int i = 0; i < 2 * KS; ++i) {
        if (i & 1) dp = T::mfma32(op[i % kAhead], df[i >> 1], dp);
        else s = T::mfma32(op[i % kAhead], qf[i >> 1], s);
        if (i + kAhead < 2 * KS) op[i % kAhead] = row_op(i + kAhead);
        __builtin_amdgcn_sched_barrier(0);
      }
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const float p = __builtin_amdgcn_exp2f(ROW ? s[r] * g.row_scale_log2 : __builtin_fmaf(s[r], g.scale_log2, -lse2));
        dp[r] = PRE ? p * dp[r] : p * (dp[r] * g.scale);
      }
      if (need_mask) {     // masked elements: dS = 0 (bit select, as in the dK/dV kernel)
        const uint64_t bits = row_valid_bits(opaque_blocks(g), q0w + (lane_now() & 31), k0, partial);
        const LaneBits32 vis(kh ? (uint32_t)(bits >> 32) : (uint32_t)bits, lane_now() >> 5);
#pragma unroll
        for (int r = 0; r < 16; ++r) dp[r] = __int_as_float(__float_as_int(dp[r]) & vis.mask(r));
      }
      const uint4 pk[2] = {pack8<T>(dp, 0), pack8<T>(dp, 1)};
      auto col_op = [&](int i) { return at.cols(ck, 2 * kh + i / DT, i % DT); };
      uint4 ot[kAhead];
#pragma unroll
      for (int i = 0; i < kAhead && i < 2 * DT; ++i) ot[i] = col_op(i);
#pragma unroll
      for (int i = 0; i < 2 * DT; ++i) {
        dq[i % DT] = T::mfma32(ot[i % kAhead], pk[i / DT], dq[i % DT]);
        if (i + kAhead < 2 * DT) ot[i % kAhead] = col_op(i + kAhead);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    dma_wait();        // the next tile's LDS-DMA has landed before the barrier
    __syncthreads();
  }
  // the kv halves' sums meet in LDS (the K buffers are free: every wave passed
  // the loop's last barrier): kh = 1 waves store, kh = 0 waves add theirs
  floatx4* red = (floatx4*)stile + qh * (DT * 4 * 64);
  const int lane_e = lane_now(), hi_e = lane_e >> 5;
  if (kh == 1) {
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
      for (int q = 0; q < 4; ++q)
        red[(dt * 4 + q) * 64 + lane_e] = floatx4{dq[dt][4 * q], dq[dt][4 * q + 1], dq[dt][4 * q + 2], dq[dt][4 * q + 3]};
  }
  __syncthreads();
  if (kh == 1) return;
  const int my_q = q0w + (lane_e & 31);
  if (my_q >= g.n_q) return;
#pragma unroll
  for (int dt = 0; dt < DT; ++dt)
#pragma unroll
    for (int q = 0; q < (D >= 32 ? 4 : 2); ++q) {      // D = 16: elements past 15 do not exist
      const floatx4 r = red[(dt * 4 + q) * 64 + lane_e];
      float v[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) v[i] = dq[dt][4 * q + i] + r[i];
      *(uint2*)(dQ + qb + (size_t)my_q * D + 32 * dt + 8 * q + 4 * hi_e) =
          make_uint2(pack2<T>(v[0], v[1]), pack2<T>(v[2], v[3]));
    }
}

// ---------------------------------------------------------------------------
// dQ, 16-bit, head_dim 64, in quadrants: wave w owns q rows 32 (w >> 1) ..
// +31 of the 64-row q tile (two 16-row blocks, the MFMAs' B-operand columns)
// against kv rows 32 (w & 1) .. +31 of each kv tile (rho subtiles 2 kh,
// 2 kh + 1). Every K / V row read and every K^T transposed read from LDS then
// feeds the MFMAs of both q blocks: 16 LDS reads per 24 MFMAs per wave and
// tile instead of 32. The two kv halves' fp32 dQ sums meet once, through LDS,
// at the end (the kh = 0 wave adds the kh = 1 wave's, a fixed order).
// ---------------------------------------------------------------------------
template <typename T, bool PRE>
__global__ __launch_bounds__(256, 4) void dq_kernel_q64(
    Geom g, const uint16_t* __restrict__ Q, const uint16_t* __restrict__ K,
    const uint16_t* __restrict__ V, const uint16_t* __restrict__ O, const uint16_t* __restrict__ dO,
    uint16_t* __restrict__ dQ, const float* __restrict__ LSE, float* __restrict__ Delta,
    const int32_t* __restrict__ row_ptr, const int32_t* __restrict__ row_idx, int n_qt,
    const int32_t* __restrict__ dq_order) {
  constexpr int D = 64, KS = 2, DT = 4;
  __shared__ __align__(16) uint16_t sk[2][64 * D];
  __shared__ __align__(16) uint16_t sv[2][64 * D];

  const int n_wg = n_qt * g.B * g.H;
  const int wg = work_of(blockIdx.x, n_wg, dq_order);
  if (wg < 0) return;
  const int bh = wg / n_qt, qt = wg - bh * n_qt;
  const size_t qb = (size_t)bh * g.n_q * D;
  const size_t kb = (size_t)kv_bh(g, bh) * g.n_kv * D;
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  const int grp = lane >> 4, col = lane & 15;
  const int qh = __builtin_amdgcn_readfirstlane(wave >> 1), kh = __builtin_amdgcn_readfirstlane(wave & 1);
  const int q0w = qt * kTileM + 32 * qh;       // the wave's first q row

  uint4 qf[2][KS], df[2][KS];
  float lse2[2], ndlt[2];
#pragma unroll
  for (int b = 0; b < 2; ++b) {
    const int my_q = q0w + 16 * b + col;
    const bool ok = my_q < g.n_q;
    float part = 0.f;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      const int d0 = 32 * ks + 8 * grp;
      qf[b][ks] = ok ? *(const uint4*)(Q + qb + (size_t)my_q * D + d0) : make_uint4(0, 0, 0, 0);
      df[b][ks] = ok ? *(const uint4*)(dO + qb + (size_t)my_q * D + d0) : make_uint4(0, 0, 0, 0);
      // Delta = rowsum(O * dO) over the stored O (sparse_triton_kernel.py:354-392)
      if (ok) {
        const uint4 o4 = *(const uint4*)(O + qb + (size_t)my_q * D + d0);
        const uint16_t* ho = (const uint16_t*)&o4;
        const uint16_t* hd = (const uint16_t*)&df[b][ks];
#pragma unroll
        for (int i = 0; i < 8; ++i) part += T::to_float(ho[i]) * T::to_float(hd[i]);
      }
    }
    lse2[b] = ok ? lse_base2(LSE[(size_t)bh * g.n_q + my_q]) : 0.f;
    // stored negated (and scaled with PRE), as in dq_kernel_16
    ndlt[b] = PRE ? -wave_sum16x4(part) * g.scale : -wave_sum16x4(part);
    if constexpr (PRE) {
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) df[b][ks] = scale8<T>(df[b][ks], g.scale);
    }
    if (ok && grp == 0 && kh == 0) {     // the two kv-half waves hold the same rows
      Delta[(size_t)bh * g.n_q + my_q] = ndlt[b];
      Delta[(size_t)g.B * g.H * g.n_q + (size_t)bh * g.n_q + my_q] = lse2[b];
    }
  }

  floatx4 dq[2][DT];
#pragma unroll
  for (int b = 0; b < 2; ++b)
#pragma unroll
    for (int i = 0; i < DT; ++i) dq[b][i] = floatx4{0.f, 0.f, 0.f, 0.f};

  const int e_beg = row_ptr[qt], e_end = row_ptr[qt + 1];
  DmaTile<D> dma;
  dma.init(tid);
  auto stage = [&](int k0, int buf) {
    dma.load(K + kb, k0, g.n_kv, sk[buf]);
    dma.load(V + kb, k0, g.n_kv, sv[buf]);
  };
  if (e_beg < e_end) stage((row_idx[e_beg] & kIdxMask) * kTileN, 0);
  dma_wait();
  __syncthreads();
  const int q_hi_wave = min(q0w + 31, g.n_q - 1);
  for (int e = e_beg; e < e_end; ++e) {
    const int buf = (e - e_beg) & 1;
    const int ent = row_idx[e];
    const int k0 = (ent & kIdxMask) * kTileN;
    const bool partial = (ent >> kPartialBit) & 1;
    if (e + 1 < e_end) stage((row_idx[e + 1] & kIdxMask) * kTileN, buf ^ 1);
    const uint16_t* ck = sk[buf];
    const uint16_t* cv = sv[buf];
    const int kw0 = k0 + 32 * kh;              // the wave's first kv row
    // left out where none of the wave's rows sees one of its keys
    if (!tile_unseen(g, q0w, q0w + 31, kw0, 32)) {
      const bool need_mask = partial || (q0w + 31 >= g.n_q) || (kw0 + 32 > g.n_kv) ||
                             !tile_all_visible(g, q0w, q_hi_wave, kw0, kw0 + 31);
      floatx4 ds[2][2];                          // [subtile 2 kh + u][q block]
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        const int r = rho(2 * kh + u, col);
        floatx4 sc[2], dp[2];
#pragma unroll
        for (int b = 0; b < 2; ++b) {
          sc[b] = floatx4{0.f, 0.f, 0.f, 0.f};
          dp[b] = floatx4{ndlt[b], ndlt[b], ndlt[b], ndlt[b]};
        }
        mfma_priority_hi<true>();
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
          const int d0 = 32 * ks + 8 * grp;
          const uint4 ak = lds_row8<D>(ck, r, d0);
          const uint4 av = lds_row8<D>(cv, r, d0);
#pragma unroll
          for (int b = 0; b < 2; ++b) {
            sc[b] = T::mfma(ak, qf[b][ks], sc[b]);
            dp[b] = T::mfma(av, df[b][ks], dp[b]);
          }
        }
        mfma_priority_lo<true>();
#pragma unroll
        for (int b = 0; b < 2; ++b)
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const float pv = __builtin_amdgcn_exp2f(__builtin_fmaf(sc[b][i], g.scale_log2, -lse2[b]));
            ds[u][b][i] = PRE ? pv * dp[b][i] : pv * (dp[b][i] * g.scale);
          }
      }
      if (need_mask) {     // masked elements: dS = 0 (bit select)
#pragma unroll
        for (int b = 0; b < 2; ++b) {
          const LaneBits vis(row_valid_bits(g, q0w + 16 * b + col, k0, partial), grp);
          // the word of subtiles 2 kh, 2 kh + 1, chosen by a uniform select (an
          // index by kh would put the pair in scratch)
          const uint32_t wk = kh ? vis.w[1] : vis.w[0];
#pragma unroll
          for (int u = 0; u < 2; ++u)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
              const int m = __builtin_amdgcn_sbfe((int)wk, 4 * u + i, 1);   // 0 or -1
              ds[u][b][i] = __int_as_float(__float_as_int(ds[u][b][i]) & m);
            }
        }
      }
      uint4 pb[2];
#pragma unroll
      for (int b = 0; b < 2; ++b) pb[b] = pack8<T>(ds[0][b], ds[1][b]);
      mfma_priority_hi<true>();
#pragma unroll
      for (int dt = 0; dt < DT; ++dt) {
        const uint4 a = lds_tr8<D>(ck, 32 * kh, 16 * dt, lane);
#pragma unroll
        for (int b = 0; b < 2; ++b) dq[b][dt] = T::mfma(a, pb[b], dq[b][dt]);
      }
      mfma_priority_lo<true>();
    }
    dma_wait();        // the next tile's LDS-DMA has landed before the barrier
    __syncthreads();
  }
  // the kv-half sums meet in LDS (the K buffers are free: every wave passed the
  // loop's last barrier): kh = 1 waves store, kh = 0 waves add theirs first.
  // Row offsets from the lane index afresh (mbcnt: not provably the one
  // above), not the prologue's held (spilled) across the loop.
  const int lane_e = (int)__builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u));
  const int grp_e = lane_e >> 4, col_e = lane_e & 15;
  floatx4* red = (floatx4*)&sk[0][0] + qh * (2 * DT * 64);
  if (kh == 1) {
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
      for (int dt = 0; dt < DT; ++dt) red[(b * DT + dt) * 64 + lane_e] = dq[b][dt];
  }
  __syncthreads();
  if (kh == 1) return;
#pragma unroll
  for (int b = 0; b < 2; ++b) {
    const int my_q = q0w + 16 * b + col_e;
    if (my_q >= g.n_q) continue;
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) {
      const floatx4 o = dq[b][dt] + red[(b * DT + dt) * 64 + lane_e];
      const uint2 w = make_uint2(pack2<T>(o[0], o[1]), pack2<T>(o[2], o[3]));
      *(uint2*)(dQ + qb + (size_t)my_q * D + 16 * dt + 4 * grp_e) = w;
    }
  }
}

// ---------------------------------------------------------------------------
// dQ, fp32
// ---------------------------------------------------------------------------
// Blocks and shares as in the forward (QB blocks of 16 q rows x 4 / QB shares
// of the keys). Also Delta = rowsum(O dO) of its rows, for itself and for the
// dK/dV kernel, which runs next.
template <int D, int QB>
__global__ __launch_bounds__(256, D * (QB == 1 ? 4 : 2) >= 512 ? 1 : 2) void dq_kernel_32(
    Geom g, const float* __restrict__ Q, const float* __restrict__ K, const float* __restrict__ V,
    const float* __restrict__ O, const float* __restrict__ dO, float* __restrict__ dQ,
    const float* __restrict__ LSE, float* __restrict__ Delta, const int32_t* __restrict__ row_ptr,
    const int32_t* __restrict__ row_idx, int n_qt, const int32_t* __restrict__ dq_order) {
  constexpr int DJ = D / 16;
  constexpr int KB = 4 / QB;
  constexpr int TR = KB == 4 ? 64 : 32;
  constexpr int SUBS = TR / (16 * KB);
  constexpr int HALVES = kTileN / TR;
  constexpr int DV = D >= 64 ? D / 64 : 1;
  constexpr int DE = D / (16 * DV);
  __shared__ __align__(16) float sk[2][TR * D];
  __shared__ __align__(16) float sv[2][TR * D];

  int part;
  const int wg = work_part_of(blockIdx.x, n_qt * g.B * g.H, KB, dq_order, part);
  if (wg < 0) return;
  const int bh = wg / n_qt, qt = wg - bh * n_qt;
  const size_t qb = (size_t)bh * g.n_q * D;
  const size_t kb = (size_t)kv_bh(g, bh) * g.n_kv * D;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int grp = lane >> 4, col = lane & 15;
  const int share = wave / QB;
  const int q0 = qt * kTileM + 16 * (part * QB + wave % QB);
  const int my_q = q0 + col;

  floatx4 qf[DJ], df[DJ];
  float part_d[DJ];
#pragma unroll
  for (int j = 0; j < DJ; ++j) {
    const bool ok = my_q < g.n_q;
    const size_t at = qb + (size_t)my_q * D + 16 * j + 4 * grp;
    qf[j] = ok ? *(const floatx4*)(Q + at) : floatx4{0.f, 0.f, 0.f, 0.f};
    df[j] = ok ? *(const floatx4*)(dO + at) : floatx4{0.f, 0.f, 0.f, 0.f};
    const floatx4 ov = ok ? *(const floatx4*)(O + at) : floatx4{0.f, 0.f, 0.f, 0.f};
    part_d[j] = __builtin_fmaf(ov[3], df[j][3], __builtin_fmaf(ov[2], df[j][2],
                               __builtin_fmaf(ov[1], df[j][1], ov[0] * df[j][0])));
  }
  // pairwise: the rounding of one chain of D / 4 terms showed in dP - Delta
#pragma unroll
  for (int n = DJ / 2; n > 0; n /= 2)
#pragma unroll
    for (int j = 0; j < n; ++j) part_d[j] += part_d[j + n];
  const float dlt = wave_sum16x4(part_d[0]);
  const float lse = my_q < g.n_q ? LSE[(size_t)bh * g.n_q + my_q] : 0.f;   // natural
  if (my_q < g.n_q && grp == 0 && share == 0) Delta[(size_t)bh * g.n_q + my_q] = dlt;
  floatx4 dq[DV][DE], cq[DV][DE];      // running sum and its compensation (two_sum_fold)
#pragma unroll
  for (int v = 0; v < DV; ++v)
#pragma unroll
    for (int e = 0; e < DE; ++e) dq[v][e] = cq[v][e] = floatx4{0.f, 0.f, 0.f, 0.f};

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
  dma_wait();          // the row loads, before any LDS-DMA is in flight
  if (n_step > 0) stage(0, 0);
  dma_wait();
  __syncthreads();
  const int q_hi = min(q0 + 15, g.n_q - 1);
  for (int s = 0; s < n_step; ++s) {
    const int buf = s & 1;
    const bool partial = (row_idx[e_beg + s / HALVES] >> kPartialBit) & 1;
    if (s + 1 < n_step) stage(s + 1, buf ^ 1);
    const float *ck = sk[buf], *cv = sv[buf];
    const int r0 = 16 * SUBS * share;
    const int k0 = step_k0(s) + r0;                      // the wave's first key
    const bool need_mask = partial || (q0 + 15 >= g.n_q) || (k0 + 16 * SUBS > g.n_kv) ||
                           !tile_all_visible(g, q0, q_hi, k0, k0 + 16 * SUBS - 1);
    uint64_t bits = ~0ull;
    if (need_mask) bits = row_valid_bits(g, my_q, k0, partial);
    const LaneBits16 vis(bits, grp);
#pragma unroll
    for (int t = 0; t < SUBS; ++t) {
      const int r = r0 + 16 * t;
      floatx4 fq[DV][DE];              // these 16 keys, folded in compensated
#pragma unroll
      for (int v = 0; v < DV; ++v)
#pragma unroll
        for (int e = 0; e < DE; ++e) fq[v][e] = floatx4{0.f, 0.f, 0.f, 0.f};
      const floatx4 sc = mfma_f32_dot<4 * DJ>(
          [&](int j) { return *(const floatx4*)(ck + off_f32<D>(r + col, 4 * j + grp)); }, qf);
      const floatx4 dp = mfma_f32_dot<4 * DJ>(
          [&](int j) { return *(const floatx4*)(cv + off_f32<D>(r + col, 4 * j + grp)); }, df);
      floatx4 ds;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        float pv = __builtin_amdgcn_exp2f(__builtin_fmaf(sc[i], g.scale, -lse) * kLog2e);
        if (need_mask) pv = vis.keep(t, i, pv);
        ds[i] = pv * (dp[i] - dlt) * g.scale;
      }
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int v = 0; v < DV; ++v) {
          const floatx4 x = cols_f32<D, DE>(ck, r + 4 * grp + i, v, col);
#pragma unroll
          for (int e = 0; e < DE; ++e) fq[v][e] = mfma_f32(x[e], ds[i], fq[v][e]);
        }
#pragma unroll
      for (int v = 0; v < DV; ++v)
#pragma unroll
        for (int e = 0; e < DE; ++e) fold(dq[v][e], cq[v][e], fq[v][e]);
    }
    dma_wait();        // the next step's LDS-DMA has landed before the barrier
    __syncthreads();
  }
  if constexpr (KB > 1) {              // the shares' sums, through LDS, in order
    constexpr int SZ = 2 * 16 * D;                       // dq, cq of a wave
    static_assert((KB - 1) * QB * SZ <= 2 * TR * D, "the sums fit one staging array");
    float* red = &sk[0][0];
    const int blk = wave % QB;
    if (share > 0) {
      float* dst = red + ((size_t)(share - 1) * QB + blk) * SZ + lane;
#pragma unroll
      for (int v = 0; v < DV; ++v)
#pragma unroll
        for (int e = 0; e < DE; ++e)
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            dst[128 * ((v * DE + e) * 4 + i)] = dq[v][e][i];
            dst[128 * ((v * DE + e) * 4 + i) + 64] = cq[v][e][i];
          }
    }
    __syncthreads();
    if (share > 0) return;
#pragma unroll
    for (int x = 1; x < KB; ++x) {
      const float* src = red + ((size_t)(x - 1) * QB + blk) * SZ + lane;
#pragma unroll
      for (int v = 0; v < DV; ++v)
#pragma unroll
        for (int e = 0; e < DE; ++e) {
          floatx4 a;
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            a[i] = src[128 * ((v * DE + e) * 4 + i)];
            cq[v][e][i] += src[128 * ((v * DE + e) * 4 + i) + 64];
          }
          two_sum_fold(dq[v][e], cq[v][e], a);
        }
    }
  }
#pragma unroll
  for (int v = 0; v < DV; ++v)
#pragma unroll
    for (int e = 0; e < DE; ++e) dq[v][e] += cq[v][e];
  if (my_q < g.n_q) {
#pragma unroll
    for (int v = 0; v < DV; ++v)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        float* dst = dQ + qb + (size_t)my_q * D + 64 * v + DE * (4 * grp + i);
        if constexpr (DE == 4) {
          *(floatx4*)dst = floatx4{dq[v][0][i], dq[v][1][i], dq[v][2][i], dq[v][3][i]};
        } else {
#pragma unroll
          for (int e = 0; e < DE; ++e) dst[e] = dq[v][e][i];
        }
      }
  }
}

// dQ first: it also produces the -Delta and LSE rows, which dK/dV reads
// from the two halves of the row-term workspace
template <typename T, int D, int FORM>
void launch_bwd16_as(const Geom& g, const void* q, const void* k, const void* v, const void* o,
                     const void* dout, const float* lse, void* dq, void* dk, void* dv, float* delta,
                     const int32_t* row_ptr, const int32_t* row_idx, int n_qt, const int32_t* dq_order,
                     const int32_t* col_ptr, const int32_t* col_idx, const KvWork& w, hipStream_t stream) {
  const int BH = g.B * g.H, BHkv = g.B * g.H_kv;
  const float* lse2 = delta + (size_t)BH * g.n_q;
  if constexpr (D == 64) {
    constexpr bool PRE = FORM == kBwdPre;
    hipLaunchKernelGGL((dq_kernel_q64<T, PRE>), dim3(n_qt * BH), dim3(256), 0, stream, g,
                       (const uint16_t*)q, (const uint16_t*)k, (const uint16_t*)v, (const uint16_t*)o,
                       (const uint16_t*)dout, (uint16_t*)dq, lse, delta, row_ptr, row_idx, n_qt, dq_order);
    hipLaunchKernelGGL((dkdv_kernel_q64<T, PRE>), dim3(w.n_items * BHkv), dim3(256), 0, stream, g,
                       (const uint16_t*)q, (const uint16_t*)k, (const uint16_t*)v, (const uint16_t*)dout,
                       (uint16_t*)dk, (uint16_t*)dv, lse2, delta, col_ptr, col_idx, w);
  } else {
    hipLaunchKernelGGL((dq_kernel_16<T, D, FORM>), dim3(n_qt * BH), dim3(256), 0, stream, g,
                       (const uint16_t*)q, (const uint16_t*)k, (const uint16_t*)v, (const uint16_t*)o,
                       (const uint16_t*)dout, (uint16_t*)dq, lse, delta, row_ptr, row_idx, n_qt, dq_order);
    hipLaunchKernelGGL((dkdv_kernel_16<T, D, FORM>), dim3(w.n_items * BHkv), dim3(256), 0, stream, g,
                       (const uint16_t*)q, (const uint16_t*)k, (const uint16_t*)v, (const uint16_t*)dout,
                       (uint16_t*)dk, (uint16_t*)dv, lse2, delta, col_ptr, col_idx, w);
  }
}

template <typename T, int D>
void launch_bwd16(const Geom& g, const void* q, const void* k, const void* v, const void* o,
                  const void* dout, const float* lse, void* dq, void* dk, void* dv, float* delta,
                  const int32_t* row_ptr, const int32_t* row_idx, int n_qt, const int32_t* dq_order,
                  const int32_t* col_ptr, const int32_t* col_idx, const KvWork& w, hipStream_t stream) {
#define GKI_BWD16(FORM)                                                                             \
  launch_bwd16_as<T, D, FORM>(g, q, k, v, o, dout, lse, dq, dk, dv, delta, row_ptr, row_idx, n_qt,  \
                              dq_order, col_ptr, col_idx, w, stream)
  // head_dim 64 forms P by an fma of the base-2 LSE, so its first two forms are one
  if (g.bwd_form == kBwdPre) GKI_BWD16(kBwdPre);
  else if (g.bwd_form == kBwdRow && D != 64) GKI_BWD16((D != 64 ? kBwdRow : kBwdPlain));
  else GKI_BWD16(kBwdPlain);
#undef GKI_BWD16
}

template <int D>
int launch_bwd(int dtype, const Geom& g, const void* q, const void* k, const void* v, const void* o,
               const void* dout, const float* lse, void* dq, void* dk, void* dv, float* delta,
               const int32_t* row_ptr, const int32_t* row_idx, int n_qt, const int32_t* dq_order,
               const int32_t* col_ptr, const int32_t* col_idx, const KvWork& w, hipStream_t stream) {
  const int BH = g.B * g.H, BHkv = g.B * g.H_kv;
  const dim3 red_grid(w.n_split * BHkv * kReduceWgPerTile<D>);
  if (dtype == kF32) {
    // dQ first: it also writes Delta, which dK/dV reads
    const int qgrid = n_qt * BH, kgrid = w.n_items * BHkv;
#define GKI_DQ32(QB)                                                                                \
  hipLaunchKernelGGL((dq_kernel_32<D, QB>), dim3(work_parts_grid(qgrid, 4 / QB)), dim3(256), 0,     \
                     stream, g, (const float*)q, (const float*)k, (const float*)v, (const float*)o, \
                     (const float*)dout, (float*)dq, lse, delta, row_ptr, row_idx, n_qt, dq_order)
#define GKI_DKDV32(KB)                                                                              \
  hipLaunchKernelGGL((dkdv_kernel_32<D, KB>), dim3(work_parts_grid(kgrid, 4 / KB)), dim3(256), 0,   \
                     stream, g, (const float*)q, (const float*)k, (const float*)v,                  \
                     (const float*)dout, (float*)dk, (float*)dv, lse, delta, col_ptr, col_idx, w)
    const int qblocks = f32_row_blocks(D, qgrid, row_kv_tiles(g, kTileM));
    if (qblocks == 1) GKI_DQ32(1);
    else if (qblocks == 2) GKI_DQ32(2);
    else GKI_DQ32(4);
    const int kblocks = f32_kv_blocks(D, kgrid);
    if (D <= 64 && kblocks == 1) GKI_DKDV32((D <= 64 ? 1 : 2));
    else if (kblocks <= 2) GKI_DKDV32(2);
    else GKI_DKDV32(4);
#undef GKI_DQ32
#undef GKI_DKDV32
    if (w.n_split > 0)
      hipLaunchKernelGGL((dkdv_reduce_kernel<F32, D>), red_grid, dim3(256), 0, stream, g, w,
                         (float*)dk, (float*)dv);
  } else if (dtype == kF16) {
    launch_bwd16<F16, D>(g, q, k, v, o, dout, lse, dq, dk, dv, delta, row_ptr, row_idx, n_qt,
                         dq_order, col_ptr, col_idx, w, stream);
    if (w.n_split > 0)
      hipLaunchKernelGGL((dkdv_reduce_kernel<F16, D>), red_grid, dim3(256), 0, stream, g, w,
                         (uint16_t*)dk, (uint16_t*)dv);
  } else {
    launch_bwd16<BF16, D>(g, q, k, v, o, dout, lse, dq, dk, dv, delta, row_ptr, row_idx, n_qt,
                          dq_order, col_ptr, col_idx, w, stream);
    if (w.n_split > 0)
      hipLaunchKernelGGL((dkdv_reduce_kernel<BF16, D>), red_grid, dim3(256), 0, stream, g, w,
                         (uint16_t*)dk, (uint16_t*)dv);
  }
  return check_launch("gki_bsa_bwd");
}

}  // namespace

int bwd_dispatch(int dtype, int head_dim, const Geom& g, const void* q, const void* k, const void* v,
                 const void* o, const void* dout, const float* lse, void* dq, void* dk, void* dv,
                 float* delta, const int32_t* row_ptr, const int32_t* row_idx, int n_qt,
                 const int32_t* dq_order, const int32_t* col_ptr, const int32_t* col_idx, const KvWork& w,
                 hipStream_t stream) {
#define GKI_BWD_CASE(DD)                                                                          \
  case DD:                                                                                        \
    return launch_bwd<DD>(dtype, g, q, k, v, o, dout, lse, dq, dk, dv, delta, row_ptr, row_idx,   \
                          n_qt, dq_order, col_ptr, col_idx, w, stream);
  switch (head_dim) {
    GKI_BWD_CASE(16)
    GKI_BWD_CASE(32)
    GKI_BWD_CASE(64)
    GKI_BWD_CASE(128)
    default: return fail(2, "unsupported head_dim " + std::to_string(head_dim));
  }
#undef GKI_BWD_CASE
}

}  // namespace gki
