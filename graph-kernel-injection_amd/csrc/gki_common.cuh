// Shared device/host helpers for the gfx950 block-sparse attention kernels.
//
// Everything here is CDNA4-specific: wave64, v_mfma_f32_16x16x32_{bf16,f16}
// and v_mfma_f32_16x16x4f32 fragments, LDS staging helpers.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <algorithm>
#include <cmath>

#include <string>

namespace gki {

// ---------------------------------------------------------------------------
// Element types. Storage is always the raw 16/32-bit pattern; conversions go
// through __bf16 / _Float16 so the compiler emits v_cvt_pk_bf16_f32 (RNE) and
// v_cvt_f16_f32 (RNE), matching torch's .to(dtype) rounding.
// ---------------------------------------------------------------------------
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef float floatx16 __attribute__((ext_vector_type(16)));

enum DType : int { kF32 = 0, kF16 = 1, kBF16 = 2 };

struct F32 {
  using storage = float;
  static constexpr bool is_f32 = true;
  __device__ static inline float to_float(float x) { return x; }
  __device__ static inline float from_float(float x) { return x; }
};
struct F16 {
  using storage = uint16_t;
  using vec8 = f16x8;
  static constexpr bool is_f32 = false;
  __device__ static inline float to_float(uint16_t x) {
    return (float)__builtin_bit_cast(_Float16, x);
  }
  __device__ static inline uint16_t from_float(float x) {
    return __builtin_bit_cast(uint16_t, (_Float16)x);
  }
  __device__ static inline floatx4 mfma(const uint4& a, const uint4& b, floatx4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a),
                                                   __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
  }
  __device__ static inline floatx16 mfma32(const uint4& a, const uint4& b, floatx16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, a),
                                                   __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
  }
  // eight 1.0 elements: an all-ones MFMA operand (row sums on the matrix pipe)
  __device__ static inline uint4 ones8() { return make_uint4(0x3C003C00u, 0x3C003C00u, 0x3C003C00u, 0x3C003C00u); }
  // a.lo * b.lo + a.hi * b.hi + c in fp32 on packed pairs (v_dot2_f32_f16)
  __device__ static inline float dot2(uint32_t a, uint32_t b, float c) {
    typedef _Float16 h2 __attribute__((ext_vector_type(2)));
    return __builtin_amdgcn_fdot2(__builtin_bit_cast(h2, a), __builtin_bit_cast(h2, b), c, false);
  }
};
struct BF16 {
  using storage = uint16_t;
  using vec8 = bf16x8;
  static constexpr bool is_f32 = false;
  __device__ static inline float to_float(uint16_t x) {
    return __builtin_bit_cast(float, ((uint32_t)x) << 16);
  }
  __device__ static inline uint16_t from_float(float x) {
    return __builtin_bit_cast(uint16_t, (__bf16)x);
  }
  __device__ static inline floatx4 mfma(const uint4& a, const uint4& b, floatx4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a),
                                                    __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
  }
  __device__ static inline floatx16 mfma32(const uint4& a, const uint4& b, floatx16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a),
                                                    __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
  }
  __device__ static inline uint4 ones8() { return make_uint4(0x3F803F80u, 0x3F803F80u, 0x3F803F80u, 0x3F803F80u); }
  // a.lo * b.lo + a.hi * b.hi + c in fp32 on packed pairs (v_dot2_f32_bf16)
  __device__ static inline float dot2(uint32_t a, uint32_t b, float c) {
    typedef __bf16 b2 __attribute__((ext_vector_type(2)));
    return __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(b2, a), __builtin_bit_cast(b2, b), c, false);
  }
};

__device__ inline floatx4 mfma_f32(float a, float b, floatx4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

// fp32 dot products over the head dimension on v_mfma_f32_16x16x4f32, KS
// k-steps of 4: the steps go round-robin into NC independent accumulators,
// summed pairwise at the end, so a long contraction (D = 64: 16 steps, 2 per
// accumulator; D = 128: 32 steps, 4 per accumulator) rounds like a short one.
// With 4 accumulators at D = 64 the scores' and dP's rounding was the largest
// error of the fp32 gradients at large logits (2x the eager path's on some
// inputs); 8 halve it. a(j) / b[j] hold the operands of steps 4 j .. 4 j + 3.
template <int KS, typename FA>
__device__ inline floatx4 mfma_f32_dot(FA a, const floatx4 (&b)[KS / 4]) {
  constexpr int NC = KS >= 16 ? 8 : (KS >= 8 ? 4 : 2);
  floatx4 c[NC];
#pragma unroll
  for (int j = 0; j < NC; ++j) c[j] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int j = 0; j < KS / 4; ++j) {
    const floatx4 x = a(j);
#pragma unroll
    for (int i = 0; i < 4; ++i) c[(4 * j + i) % NC] = mfma_f32(x[i], b[j][i], c[(4 * j + i) % NC]);
  }
  if constexpr (NC == 8) return ((c[0] + c[1]) + (c[2] + c[3])) + ((c[4] + c[5]) + (c[6] + c[7]));
  else if constexpr (NC == 4) return (c[0] + c[1]) + (c[2] + c[3]);
  else return c[0] + c[1];
}

// 16-byte streaming (non-temporal) global load.
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
__device__ inline uint4 ld_nt16(const void* p) {
  const u32x4 v = __builtin_nontemporal_load((const u32x4*)p);
  return make_uint4(v.x, v.y, v.z, v.w);
}

// Two fp32 -> two 16-bit elements in one v_cvt_pk_{bf16,f16}_f32 (RNE).
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
template <typename T>
__device__ inline uint32_t pack2(float a, float b);
template <>
__device__ inline uint32_t pack2<BF16>(float a, float b) {
  return __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2{a, b}, bf16x2));
}
template <>
__device__ inline uint32_t pack2<F16>(float a, float b) {
  return __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2{a, b}, f16x2));
}

// Eight 16-bit elements times a power-of-two scale, rounded back (exact
// unless a result falls below the format's smallest normal).
template <typename T>
__device__ inline uint4 scale8(const uint4& v, float s) {
  const uint16_t* h = (const uint16_t*)&v;
  float f[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) f[i] = T::to_float(h[i]) * s;
  return make_uint4(pack2<T>(f[0], f[1]), pack2<T>(f[2], f[3]), pack2<T>(f[4], f[5]),
                    pack2<T>(f[6], f[7]));
}

// Accumulators of two 16x16 subtiles (rows 0-3 then 4-7) packed to eight 16-bit
// elements: one 16x16x32 MFMA operand.
template <typename T>
__device__ inline uint4 pack8(const floatx4& lo, const floatx4& hi) {
  return make_uint4(pack2<T>(lo[0], lo[1]), pack2<T>(lo[2], lo[3]), pack2<T>(hi[0], hi[1]),
                    pack2<T>(hi[2], hi[3]));
}

// Registers 8 s .. 8 s + 7 of a 32x32 accumulator: one 32x32x16 MFMA operand.
template <typename T>
__device__ inline uint4 pack8(const floatx16& x, int s) {
  return make_uint4(pack2<T>(x[8 * s], x[8 * s + 1]), pack2<T>(x[8 * s + 2], x[8 * s + 3]),
                    pack2<T>(x[8 * s + 4], x[8 * s + 5]), pack2<T>(x[8 * s + 6], x[8 * s + 7]));
}

// LDS tile layout for 16-bit [64][D] tiles: row-major, no padding, 16-byte
// chunks XOR-swizzled per row. gfx950 LDS has 64 banks of 4 bytes (one
// 256-byte "bank row" per clock), so a read is conflict-free when the 16-byte
// chunks that one clock serves land on 16 distinct positions of a bank row.
// With a = row & 3, b = (row >> 3) & 3 the swizzle is a bijection of the
// (a, b) pairs the two read patterns touch at once:
//  * 16-byte reads of rows {b..b+3, b+8..b+11, b+16.., b+24..} at one chunk
//    (the rho() row order; 16 lanes per clock),
//  * ds_read_b64_tr_b16 over rows {r..r+3, r+8..r+11} x 2 adjacent chunks
//    (32 lanes per clock),
// and the tile fill (consecutive lanes, consecutive chunks of one bank row).
// Tiles narrower than 256 bytes share a bank row between 256/(2D) rows; the
// row bits that select the slice take the place of a. D = 16 keeps a 2-way
// conflict (only 2 chunks per row).
// ROW32 (tiles read by v_mfma_f32_32x32x16): row reads take 32 consecutive rows
// at one chunk, so the swizzle is a bijection of row & 15 (any 16 of them that
// one clock serves land on distinct positions), and its low row bits sit above
// the two chunk bits that a transposed read of 4 consecutive rows x 4
// adjacent chunks covers.
template <int D, bool ROW32 = false>
__device__ inline int lds_swz(int row) {
  if constexpr (ROW32) {
    const int lo = (row >> 2) & 3;
    if constexpr (D >= 128) return 4 * (row & 3) + lo;
    else if constexpr (D == 64) return 4 * ((row >> 1) & 1) + lo;
    else if constexpr (D == 32) return lo;
    else return (row >> 3) & 1;
  }
  const int b = (row >> 3) & 3;
  const int bb = 2 * (b & 1) + (b >> 1);
  if constexpr (D >= 128) return (4 * (row & 3) + bb) & (D / 8 - 1);
  else if constexpr (D == 64) return 4 * ((row >> 1) & 1) + bb;
  else if constexpr (D == 32) return bb;
  else return 0;
}
template <int D, bool ROW32 = false>
__device__ inline int lds_off(int row, int col) {
  return row * D + ((((col >> 3) ^ lds_swz<D, ROW32>(row))) << 3) + (col & 7);
}

// Transposed MFMA operand from a swizzled 16-bit LDS tile via
// ds_read_b64_tr_b16: within each 16-lane group, lane l points at row
// k0 + l/4, columns n0 + 4*(l%4) .. +3, and the instruction hands lane i column
// n0 + i of those four rows. Two reads give lane (g, c) = (lane/16, lane%16)
// the 8 elements tile[k0 + 8g + e][n0 + c], e = 0..7: the K-operand layout of
// v_mfma_f32_16x16x32_{bf16,f16} for a matrix stored K-major. (k0 is a
// multiple of 32, so rows r and r+4 share a swizzle.)
typedef short v4i16 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) v4i16 lds_v4i16;
template <int D>
__device__ inline uint4 lds_tr8(const uint16_t* tile, int k0, int n0, int lane) {
  const int g = lane >> 4, l = lane & 15;
  const uint16_t* p = tile + lds_off<D>(k0 + 8 * g + (l >> 2), n0 + 4 * (l & 3));
  const v4i16 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4i16*)p);
  const v4i16 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4i16*)(p + 4 * D));
  const uint2 a = __builtin_bit_cast(uint2, lo), b = __builtin_bit_cast(uint2, hi);
  return make_uint4(a.x, a.y, b.x, b.y);
}
// 16-byte row read (8 elements starting at a multiple-of-8 column).
template <int D>
__device__ inline uint4 lds_row8(const uint16_t* tile, int row, int col) {
  return *(const uint4*)(tile + lds_off<D>(row, col));
}

// Operands of v_mfma_f32_32x32x16 (lane l: row or column l & 31, elements
// 8 (l >> 5) .. +7 of the 16-long contraction) and its accumulator (lane l:
// column l & 31, register r: row 8 (r >> 2) + 4 (l >> 5) + (r & 3)). Registers
// 8 s .. 8 s + 7 of lane half hi therefore hold rows 16 s + 4 hi + (j & 3) +
// 8 (j >> 2), j = 0 .. 7, and serve as an operand of a contraction over rows
// 16 s .. 16 s + 15 whose other operand lists the same rows in the same order:
// Lane32::cols gives lane l a column of exactly those rows, by two transposed
// reads. (A tile of D = 16 columns has none past 15: lanes
// 16 .. 31 of a half repeat columns 0 .. 15.)
// The lane's byte offsets are computed once; rows 32 t / 16 s and the buffer are
// constants of the instruction, chunks an XOR.
template <int D>
struct Lane32 {
  int row;        // row l & 31, columns 8 (l >> 5) ..
  int tr[2];      // rows 4 (l >> 5) + ((l & 15) >> 2) and that + 8, columns 16 ((l >> 4) & 1) + 4 (l & 3) ..
  __device__ inline Lane32(int lane) {
    const int hi = lane >> 5, i = lane & 15;
    row = 2 * lds_off<D, true>(lane & 31, 8 * hi);
    const int r = 4 * hi + (i >> 2), c = (D >= 32 ? 16 * ((lane >> 4) & 1) : 0) + 4 * (i & 3);
    tr[0] = 2 * lds_off<D, true>(r, c);
    tr[1] = 2 * lds_off<D, true>(r + 8, c);
  }
  // From here on the compiler takes the offsets for new values.
  __device__ inline void pin() { asm volatile("" : "+v"(row), "+v"(tr[0]), "+v"(tr[1])); }
  // Row operand: rows 32 t + (l & 31), columns 16 ks + 8 (l >> 5) .. +7.
  __device__ inline uint4 rows(const uint16_t* tile, int t, int ks) const {
    return *(const uint4*)((const char*)tile + 64 * D * t + (row ^ (32 * ks)));
  }
  // Transposed operand: column 32 dt + (l & 31) of rows 16 st .. +15 in accumulator order.
  __device__ inline uint4 cols(const uint16_t* tile, int st, int dt) const {
    const char* p = (const char*)tile + 32 * D * st;
    const v4i16 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4i16*)(p + (tr[0] ^ (64 * dt))));
    const v4i16 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4i16*)(p + (tr[1] ^ (64 * dt))));
    const uint2 a = __builtin_bit_cast(uint2, lo), b = __builtin_bit_cast(uint2, hi);
    return make_uint4(a.x, a.y, b.x, b.y);
  }
};
__device__ inline floatx16 splat16(float x) {
  return floatx16{x, x, x, x, x, x, x, x, x, x, x, x, x, x, x, x};
}
// The lane index afresh (mbcnt): not provably the one derived from threadIdx,
// so that values derived from it late are not kept from the kernel's start.
__device__ inline int lane_now() {
  return (int)__builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u));
}
// Row (of 32) of register r in lane half hi of a 32x32 accumulator.
__device__ inline int acc32_row(int r, int hi) { return 8 * (r >> 2) + 4 * hi + (r & 3); }

// 16 bytes at (row, d0) of a row-major [n_rows, D] 16-bit matrix, zero when
// row >= n_rows or d0 >= D (n_rows >= 1). The load is unconditional, from a
// clamped in-bounds address, and the zero a select: as a predicated load each
// would sit in its own branch with its own wait, so that a kernel prologue's
// row loads would land one after another instead of together.
template <int D>
__device__ inline uint4 row16_or_zero(const uint16_t* base, int row, int n_rows, int d0) {
  const bool ok = row < n_rows && d0 < D;
  const uint4 v = *(const uint4*)(base + (size_t)min(row, n_rows - 1) * D + (d0 < D ? d0 : 0));
  return ok ? v : make_uint4(0, 0, 0, 0);
}

// LDS byte address of a pointer into __shared__ memory.
__device__ inline uint32_t lds_addr(const void* p) {
  return (uint32_t)(uintptr_t)(__attribute__((address_space(3))) const void*)p;
}

// One gfx950 LDS-DMA load: every lane fetches 16 bytes from its global address
// `src` and the wave writes them to LDS bytes [lds, lds + 1024), lane i at
// lds + 16 i. Issued as inline asm so that the compiler does not guard every
// later LDS read with a wait on it (it cannot tell which buffer the DMA
// targets); callers wait explicitly with dma_wait() before the barrier that
// publishes the buffer. Only M0 and memory are touched.
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
__device__ inline void dma_load16(const void* src, uint32_t lds) {
  asm volatile("s_mov_b32 m0, %1\n\tglobal_load_lds_dwordx4 %0, off" ::"v"(src), "s"(lds)
               : "memory", "m0");
}
// Buffer-resource variant: lane i fetches 16 bytes at the resource base +
// voff[i] (same LDS placement), so the per-tile address arithmetic is scalar
// (the base) and the lane offsets stay in registers unchanged; offsets at or
// past `bytes` read zero instead of faulting. Measured faster than the global
// form for the forward's K / V tiles.
typedef int i32x4 __attribute__((ext_vector_type(4)));
__device__ inline i32x4 buffer_rsrc(const void* base, uint32_t bytes) {
  const uint64_t a = (uint64_t)(uintptr_t)base;
  i32x4 r;
  r.x = __builtin_amdgcn_readfirstlane((int)(uint32_t)a);
  r.y = __builtin_amdgcn_readfirstlane((int)(uint32_t)(a >> 32));   // stride 0
  r.z = __builtin_amdgcn_readfirstlane((int)bytes);                   // num_records
  r.w = 0x00020000;                                                   // DATA_FORMAT 32
  return r;
}
// Rows of a TR-row tile that exist when `left` rows remain from its first on
// (uniform). In two steps the compiler cannot join: joined they are a vector
// median and a readfirstlane, which made the D = 128 forward 4% slower.
template <int TR>
__device__ inline int rows_left(int left) {
  left = left < TR ? left : TR;
  asm volatile("" : "+s"(left));
  return left > 0 ? left : 0;
}
__device__ inline void dma_buf16(i32x4 rsrc, int voff, uint32_t lds) {
  asm volatile("s_mov_b32 m0, %2\n\tbuffer_load_dwordx4 %0, %1, 0 offen lds" ::"v"(voff), "s"(rsrc),
               "s"(lds)
               : "memory", "m0");
}
// 4-byte variant: lane i writes lds + 4 i.
__device__ inline void dma_load4(const void* src, uint32_t lds) {
  asm volatile("s_mov_b32 m0, %1\n\tglobal_load_lds_dword %0, off" ::"v"(src), "s"(lds)
               : "memory", "m0");
}
#pragma clang diagnostic pop
// Wait until this wave's vector-memory operations (LDS-DMA included) are done:
// s_waitcnt vmcnt(0) (gfx9 encoding: vmcnt 0, expcnt 7, lgkmcnt 15). Issued via
// the builtin so the compiler's own wait tracking also sees every earlier load
// as complete and inserts no further vmcnt waits for them.
__device__ inline void dma_wait() { __builtin_amdgcn_s_waitcnt(0x0F70); }

// Stage a full 64-row tile of a row-major [n, D] 16-bit matrix straight into
// the swizzled LDS layout with LDS-DMA loads: no VGPR staging and no ds_write.
// One wave instruction fills 1 KB of LDS, lane i writing bytes 16i..16i+15,
// so the swizzle is applied on the global side: lane i fetches the chunk that
// belongs at its LDS position. The workgroup's NW waves cover the tile's D/8
// blocks of 1 KB (block NW p + wave for p = 0, 1, ...); `off` is the lane's
// element offset inside the tile for each block it moves (computed once).
template <int D, int NW = 4, bool ROW32 = false>
struct DmaTile {
  static constexpr int NB = D / 8;                     // 1 KB blocks per tile
  static constexpr int NP = (NB + NW - 1) / NW;        // blocks per wave
  int off[NP];
  int wave;
  __device__ inline void init(int tid) {
    wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int lane = tid & 63;
#pragma unroll
    for (int p = 0; p < NP; ++p) {
      const int e = (NW * p + wave) * 512 + 8 * lane;  // LDS element offset
      const int row = e / D, pch = (e % D) >> 3;
      off[p] = row * D + ((pch ^ lds_swz<D, ROW32>(row)) << 3);
    }
  }
  // Rows r0 .. r0+63 of a matrix of n_rows rows through a buffer resource over
  // those that exist: the tile base is uniform, so a tile costs no per-lane
  // address arithmetic, and the resource's range check makes the rows past the
  // last one zeros in LDS (no separate path for a ragged tile).
  __device__ inline void load(const uint16_t* base, int r0, int n_rows, const uint16_t* lds) const {
    const i32x4 rsrc = buffer_rsrc(base + (size_t)r0 * D, rows_left<64>(n_rows - r0) * D * 2);
    const uint32_t l0 = lds_addr(lds);
#pragma unroll
    for (int p = 0; p < NP; ++p) {
      const int blk = NW * p + wave;
      if (NB % NW == 0 || blk < NB) dma_buf16(rsrc, 2 * off[p], l0 + blk * 1024);
    }
  }
};

// ---------------------------------------------------------------------------
// fp32 tiles: row-major in LDS, 16-byte chunks XOR-swizzled per row, staged by
// LDS-DMA. Two kinds of 16-byte reads feed v_mfma_f32_16x16x4f32, each four
// MFMAs (a 4-byte read per MFMA kept the LDS as busy as the matrix cores):
//  * a lane's four consecutive elements d = 16 j + 4 grp + i of a row: step i of
//    a contraction over d takes {16 j + 4 grp + i, grp = 0 .. 3} (the register
//    operand lists its elements in the same order);
//  * four consecutive columns 4 col + e of row 4 grp + i: step i of a contraction
//    over rows, result column (or row) col of output tile e standing for
//    element 4 col + e.
// The swizzle of 256-byte rows is free of conflicts for both, whether 16
// consecutive lanes or {0-3, 12-15, 20-23, 24-27} are served per clock.
// ---------------------------------------------------------------------------
template <int D>
__device__ inline int swz_f32(int row) {
  if constexpr (D >= 64) return 4 * (row & 3) + ((-(row >> 2)) & 3);
  else if constexpr (D == 32) return (row >> 1) & 7;
  else return (row >> 2) & 3;
}
template <int D>
__device__ inline int off_f32(int row, int chunk) { return row * D + ((chunk ^ swz_f32<D>(row)) << 2); }

// Columns 64 v + DE col + e, e = 0 .. DE - 1, of a row.
template <int D, int DE>
__device__ inline floatx4 cols_f32(const float* tile, int row, int v, int col) {
  if constexpr (DE == 4) {
    return *(const floatx4*)(tile + off_f32<D>(row, 16 * v + col));
  } else {
    floatx4 x = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int e = 0; e < DE; ++e) {
      const int c = DE * col + e;
      x[e] = tile[off_f32<D>(row, c >> 2) + (c & 3)];
    }
    return x;
  }
}

// Stage TR rows of a row-major [n, D] fp32 matrix; rows past the last are zeros.
template <int D, int TR, int NW = 4>
struct DmaTileF32 {
  static constexpr int NB = TR * D / 256;              // 1 KB blocks per tile
  static constexpr int NP = (NB + NW - 1) / NW;        // blocks per wave
  int off[NP];
  int wave;
  __device__ inline void init(int tid) {
    wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int lane = tid & 63;
#pragma unroll
    for (int p = 0; p < NP; ++p) {
      const int e = (NW * p + wave) * 256 + 4 * lane;  // LDS float offset
      const int row = e / D, ch = (e % D) >> 2;
      off[p] = 4 * (row * D + ((ch ^ swz_f32<D>(row)) << 2));
    }
  }
  __device__ inline void load(const float* base, int r0, int n_rows, const float* lds) const {
    const i32x4 rsrc = buffer_rsrc(base + (size_t)r0 * D, rows_left<TR>(n_rows - r0) * D * 4);
    const uint32_t l0 = lds_addr(lds);
#pragma unroll
    for (int p = 0; p < NP; ++p) {
      const int blk = NW * p + wave;
      if (NB % NW == 0 || blk < NB) dma_buf16(rsrc, off[p], l0 + blk * 1024);
    }
  }
};

// ---------------------------------------------------------------------------
// Kernel tiling. The 16-bit forward uses 128x64 (q x kv) tiles, four waves of 32
// query rows each (on short grids two workgroups of eight waves, fwd_split_16);
// the backward kernels use 64x64 tiles, a 32x32 quadrant per wave; the fp32
// kernels 64x64 tiles in blocks of 16 rows. The decode kernel (n_q <=
// kDecodeMaxQ) uses a single 16-row q tile.
// ---------------------------------------------------------------------------
constexpr int kTileM = 64;       // q rows of the dQ / dK-dV tiles
constexpr int kTileN = 64;       // kv rows of every tile
constexpr int kTileMF = 128;     // q rows of the forward tile (4 waves x 32 rows)
constexpr int kDecodeTileM = 16;
constexpr int kDecodeMaxQ = 4;
// dK/dV work items: at least kDkdvMinChunk iterations each, and about
// kDkdvTargetItems items over the whole grid when the column walks are long.
constexpr int kDkdvMinChunk = 32;
constexpr int kDkdvTargetItems = 8192;

// q heads one decode workgroup serves: a whole group of grouped-query heads
// when its group * n_q rows fit the kernel's row limit (K / V read once per
// group), else one head.
inline int decode_heads_per_workgroup(int group, int n_q) {
  return group > 1 && group * n_q <= kDecodeMaxQ ? group : 1;
}

constexpr int kPartialBit = 30;       // schedule entry flag: needs per-element mask lookup
constexpr int kIdxMask = (1 << kPartialBit) - 1;

// Row permutation rho(t, j) of a 64-row tile into four 16-row MFMA subtiles.
// Subtile t = 2s+h, lane-row j = 4a+i holds tile row 32s + 8a + 4h + i. With
// this order the fp32 accumulator of subtiles (2s, 2s+1) held by lane group a
// covers rows 32s+8a .. 32s+8a+7 contiguously, i.e. it already IS the 8-element
// K-operand of a 16x16x32 MFMA over those rows: no register transpose needed.
__device__ inline int rho(int t, int j) {
  return ((t >> 1) << 5) + ((j >> 2) << 3) + ((t & 1) << 2) + (j & 3);
}

// Geometry + masking parameters shared by all attention kernels.
// Forms of the 16-bit backward (Geom::bwd_form).
enum BwdForm : int { kBwdPlain = 0, kBwdRow = 1, kBwdPre = 2 };

// The form a scale takes: dS is cast to 16 bits after the scale, as in the
// reference, so an operand can carry it only where it is a power of two (head_dim
// 16 and 64 by default). Taking a power of two out of other scales (dS / post cast,
// post in [1, 2) multiplied into the sums) saved 0-1% of a bf16 backward at
// head_dim 128, 0-5% at 32 (B8 H16/4 N4096 W1024 316 against 330 us), and cost fp16
// gradients accuracy, as operand and dS / post sink among the subnormal numbers: for
// a dO of 1e-4, ordinary without loss scaling, dQ of N512 W64 was 1.02e-2 (D32) and
// 1.62e-2 (D64, scale 0.1) from 64 bits against 7.1e-3 and 1.02e-2.
__host__ inline int bwd_form_of(int dtype, float scale) {
  int e2 = 0;
  const float mant = std::frexp(scale, &e2);           // |scale| in [2^(e2-1), 2^e2)
  if (dtype != kF32 && mant == 0.f) return kBwdRow;
  if (dtype == kF32 || e2 < -29 || e2 > 30) return kBwdPlain;
  return (mant == 0.5f || mant == -0.5f) && e2 >= -3 && e2 <= 1 ? kBwdPre : kBwdRow;
}

struct Geom {
  int B, H;
  int H_kv, group;    // K/V heads and q heads per K/V head (grouped-query attention; 1 = MHA)
  int n_q, n_kv, q_off;
  float scale;        // natural-log softmax scale (any finite value)
  float scale_log2;   // scale * log2(e)
  // The 16-bit prefill and matrix-core decode kernels track the running max
  // on unscaled scores, which needs a positive scale. They read each 32-bit
  // word w of Q as (w & q_and) ^ q_xor and scale by qk_scale_log2 instead:
  // scale < 0 flips the sign of Q (exact: (-Q) K^T * |scale| equals
  // Q K^T * scale bit for bit), scale == 0 zeroes Q (every score 0, as
  // Q K^T * 0) with qk_scale_log2 = log2(e); scale > 0 leaves Q as it is.
  float qk_scale_log2;
  uint32_t q_and, q_xor;
  // 16-bit backward: dS = P (dP - Delta) scale, cast to 16 bits before the
  // dK / dQ products (bwd_form):
  //  kBwdPre   scale +-2^-4 .. 1: the kernels multiply the V (dK/dV) or dO (dQ)
  //    operand and -Delta by it once; every product and partial sum of the dP
  //    accumulator is then the same value times it (exact in fp32), so it ends
  //    as (dP - Delta) scale and dS costs one multiply. Only a 16-bit operand
  //    that the scale takes below the smallest normal rounds (by at most half
  //    its subnormal spacing, 2^-25 for fp16).
  //  kBwdRow   dS is scaled per element; the row terms still start the
  //    accumulators (-LSE / scale, -Delta). Scale 0: the operand of S is zeroed
  //    (q_and) and row_scale 1 divides the LSE.
  //  kBwdPlain for scales too small or large to divide the LSE (|scale| outside
  //    [2^-30, 2^30)): as kBwdRow with the LSE subtracted in the exponent.
  int bwd_form;
  float row_scale, row_scale_log2;
  int causal, sink, window;
  // original block mask (used only for tiles flagged partial)
  const int32_t* mask;
  int n_qb, n_kb, bm, bn;
};

// Work list of the dK / dV grid (built on the host by gki_dkdv_items). A kv
// tile's walk -- group x (its kept q tiles) iterations, iteration i visiting
// list entry i % L of q head i / L -- is cut into items of at most a chunk of
// iterations, so no workgroup carries a long column (the sink column, the
// columns of a large grouped-query group) alone. A column with one item stores
// dK / dV itself; the items of a split column store fp32 partials, which a
// reduce pass sums in item order (deterministic).
struct KvWork {
  const int32_t* items;   // [n_items][4]: kv tile, first iteration, end iteration, partial slot (-1: none)
  int n_items;
  const int32_t* split;   // [n_split][3]: kv tile, its first partial slot, number of slots
  int n_split;
  int n_pslots;           // partial slots per (b, kv head)
  float* partials;        // [B * H_kv][n_pslots][2 (dK, dV)][64][D] fp32
};

// A 16-byte Q fragment as the unscaled-max kernels read it (see Geom::q_and).
__device__ inline uint4 q_words(const Geom& g, uint4 w) {
  return make_uint4((w.x & g.q_and) ^ g.q_xor, (w.y & g.q_and) ^ g.q_xor, (w.z & g.q_and) ^ g.q_xor,
                    (w.w & g.q_and) ^ g.q_xor);
}

// (b, q head) -> (b, kv head) row index of K / V (and dK / dV).
__device__ inline int kv_bh(const Geom& g, int bh) {
  return g.group == 1 ? bh : (bh / g.H) * g.H_kv + (bh % g.H) / g.group;
}

// Bounds + token predicate for (q row, kv column), branch-free.
__host__ __device__ inline bool elem_tok(const Geom& g, int q_row, int kv) {
  const int qa = q_row + g.q_off;
  const bool in = (q_row < g.n_q) & (kv < g.n_kv);
  const bool vis = (kv <= qa) & ((kv < g.sink) | (kv >= qa - g.window + 1));
  return in & ((g.causal == 0) | vis);
}

// Full element predicate for (q row, kv column) of a tile flagged "needs mask":
// tiles flagged partial also consult the lifted block mask.
__host__ __device__ inline bool elem_valid(const Geom& g, int q_row, int kv, bool partial) {
  bool ok = elem_tok(g, q_row, kv);
  if (partial && ok) ok = g.mask[(size_t)(q_row / g.bm) * g.n_kb + kv / g.bn] != 0;
  return ok;
}

// ---------------------------------------------------------------------------
// The same predicate for 64 elements at once: one query row against the 64
// keys of a tile (or one key against the 64 query rows of a tile) as a 64-bit
// word, bit j = element j. The token rule is an interval condition along
// either axis, so the word costs a few shifts per lane and tile instead of a
// compare chain per element.
// ---------------------------------------------------------------------------

// Bits lo .. hi of a 64-bit word (clamped to 0 .. 63; empty when hi < lo).
__host__ __device__ inline uint64_t bit_range(int lo, int hi) {
  lo = lo < 0 ? 0 : lo;
  hi = hi > 63 ? 63 : hi;
  return hi < lo ? 0 : (~0ull >> (63 - hi)) & (~0ull << lo);
}

// Window length for the visibility words: any window of at least n_kv keys
// reaches key 0 from every row, so clamping there is exact and keeps the
// window-edge arithmetic inside int for n_q, n_kv < 2^30.
__host__ __device__ inline int word_window(const Geom& g) {
  return g.window < g.n_kv ? g.window : g.n_kv;
}

// elem_valid(g, q_row, k0 + j, partial) for j = 0 .. 63, as bits.
__host__ __device__ inline uint64_t row_valid_bits(const Geom& g, int q_row, int k0, bool partial) {
  if (q_row >= g.n_q) return 0;
  uint64_t b = bit_range(0, g.n_kv - 1 - k0);
  if (g.causal) {
    const int qa = q_row + g.q_off - k0;           // key j visible iff j <= qa and
    b &= bit_range(0, qa) &                        // (j >= qa - W + 1 or k0 + j < S)
         (bit_range(qa - word_window(g) + 1, 63) | bit_range(0, g.sink - 1 - k0));
  }
  if (partial) {                                 // kept blocks of the row's block row
    const int mrow = (q_row / g.bm) * g.n_kb;     // 32-bit: the mask has < 2^31 blocks
    uint64_t kept = 0;
    for (int kb = k0 / g.bn; kb < g.n_kb && kb * g.bn < k0 + 64; ++kb)
      if (g.mask[mrow + kb]) kept |= bit_range(kb * g.bn - k0, (kb + 1) * g.bn - 1 - k0);
    b &= kept;
  }
  return b;
}

// elem_valid(g, q0 + j, kv, partial) for j = 0 .. 63, as bits.
__host__ __device__ inline uint64_t col_valid_bits(const Geom& g, int kv, int q0, bool partial) {
  if (kv >= g.n_kv) return 0;
  uint64_t b = bit_range(0, g.n_q - 1 - q0);
  if (g.causal) {
    const int a = kv - g.q_off - q0;               // row j visible iff j >= a and
    b &= bit_range(a, 63) &                        // (kv < S or j <= a + W - 1)
         (kv < g.sink ? ~0ull : bit_range(0, a + word_window(g) - 1));
  }
  if (partial) {                                 // kept blocks of the key's block column
    const int kb = kv / g.bn;
    uint64_t kept = 0;
    for (int qb = q0 / g.bm; qb < g.n_qb && qb * g.bm < q0 + 64; ++qb)
      if (g.mask[qb * g.n_kb + kb]) kept |= bit_range(qb * g.bm - q0, (qb + 1) * g.bm - 1 - q0);
    b &= kept;
  }
  return b;
}

// The 16 elements that lane group `grp` holds in the rho() layout: element
// (t, i) is tile row / key rho(t, 4 grp + i) = 32 (t >> 1) + 8 grp + 4 (t & 1) + i,
// i.e. bit 4 (t & 1) + i of byte `grp` of word half t >> 1. Returned as two
// words whose low 8 bits are those bytes.
struct LaneBits {
  uint32_t w[2];
  __device__ inline LaneBits(uint64_t bits, int grp) {
    w[0] = (uint32_t)bits >> (8 * grp);
    w[1] = (uint32_t)(bits >> 32) >> (8 * grp);
  }
  // x where element (t, i) is set, `other` where it is not (bit-select, no compare)
  __device__ inline float pick(int t, int i, float x, float other) const {
    const int m = __builtin_amdgcn_sbfe((int)w[t >> 1], 4 * (t & 1) + i, 1);   // 0 or -1
    return __int_as_float((__float_as_int(x) & m) | (__float_as_int(other) & ~m));
  }
};

// The same for a 32x32 accumulator: register r of lane half hi is bit
// acc32_row(r, hi) of the 32-bit half of the word that belongs to its subtile.
struct LaneBits32 {
  uint32_t w;
  __device__ inline LaneBits32(uint32_t half, int hi) : w(half >> (4 * hi)) {}
  // 0 or -1: register r visible
  __device__ inline int mask(int r) const {
    return __builtin_amdgcn_sbfe((int)w, 8 * (r >> 2) + (r & 3), 1);
  }
  __device__ inline float pick(int r, float x, float other) const {
    const int m = mask(r);
    return __int_as_float((__float_as_int(x) & m) | (__float_as_int(other) & ~m));
  }
};

// The same for 16x16 subtiles in natural order (fp32): element i of subtile t in
// lane group grp is bit 16 t + 4 grp + i. 0 or -1: element visible.
struct LaneBits16 {
  uint32_t w;
  __device__ inline LaneBits16(uint64_t bits, int grp) : w((uint32_t)(bits >> (4 * grp))) {}
  __device__ inline int mask(int t, int i) const { return __builtin_amdgcn_sbfe((int)w, 16 * t + i, 1); }
  __device__ inline float keep(int t, int i, float x) const { return __int_as_float(__float_as_int(x) & mask(t, i)); }
};

// Is some (q, k) with q in [q_lo, q_hi], k in [k_lo, k_hi] (inclusive, absolute
// positions, non-empty) visible under the token rule (k <= q) & (k < S | k >= q-W+1)?
__device__ inline bool any_visible(long q_lo, long q_hi, long k_lo, long k_hi, long sink, long window) {
  const bool sink_part = k_lo < sink && k_lo <= q_hi;
  // window: some q with max(k_lo, q-W+1) <= min(k_hi, q)
  const long qa = q_lo > k_lo ? q_lo : k_lo;
  const long qb = q_hi < k_hi + window - 1 ? q_hi : k_hi + window - 1;
  const bool window_part = window >= 1 && qa <= qb;
  return sink_part || window_part;
}

// True when every (q, kv) with q in [q_lo, q_hi], kv in [k_lo, k_hi] (inclusive,
// already in bounds) is visible under the StreamingLLM token rule.
__device__ inline bool tile_all_visible(const Geom& g, int q_lo, int q_hi, int k_lo, int k_hi) {
  if (!g.causal) return true;
  const int qa = q_lo + g.q_off, qb = q_hi + g.q_off;
  if (k_hi > qa) return false;
  return (k_hi < g.sink) || (k_lo >= qb - g.window + 1);
}

// The geometry with block sizes the compiler cannot follow back: the divisions
// of a rarely taken mask branch are then not hoisted into registers held
// through a kernel's tile loop.
__device__ inline Geom opaque_blocks(Geom g) {
  asm volatile("" : "+s"(g.bm), "+s"(g.bn));
  return g;
}

// True when no row of [q_lo, q_hi] sees one of the n_k keys from k0 on under the
// token rule (never where the rule does not apply).
__host__ __device__ inline bool tile_unseen(const Geom& g, int q_lo, int q_hi, int k0, int n_k) {
  return g.causal != 0 && (k0 > q_hi + g.q_off ||
                           (k0 >= g.sink && k0 + n_k <= q_lo + g.q_off - word_window(g) + 1));
}

// ---------------------------------------------------------------------------
// Rules of the launches (host).
// ---------------------------------------------------------------------------
// About the kv tiles that a tile of `rows` q rows visits: the window's and the
// sinks' under the token rule, half of them under a block mask (not known here).
inline int row_kv_tiles(const Geom& g, int rows) {
  const int64_t n_kt = (g.n_kv + kTileN - 1) / kTileN;
  if (!g.causal) return (int)((n_kt + 1) / 2);
  const int64_t keys = std::min<int64_t>((int64_t)g.window + rows - 1, g.n_kv);
  return (int)std::min(n_kt, (keys + kTileN - 2) / kTileN + 1 + ((int64_t)g.sink + kTileN - 1) / kTileN);
}

// Does a 16-bit forward grid of `tiles` 128-row q tiles share each tile's keys
// among the waves of two workgroups (fwd_split_16)? Where these all run at once,
// one per CU (its 128 KB of LDS at head_dim 128 hold one), whatever the lists; at
// head_dim <= 64, whose CU holds two, up to twice that if the chain that is cut
// into four is long (8 kv tiles). us, one workgroup per tile against two:
//   D128  128 tiles of 1 / 19 kv tiles  8.86, 27.7 -> 8.87, 22.0
//         160                           8.99, 27.8 -> 15.3, 38.1
//   D64   128                           6.80, 22.3 -> 6.55, 14.5
//         256 tiles of 1 / 3 / 7        7.40, 9.59, 12.6 -> 8.94, 10.0, 12.6
//         256 of 9 / 15, of 1 to 8      16.1, 21.2, 12.3 -> 14.9, 19.1, 10.9
//         288 of 3 / 19                 11.1, 29.3 -> 14.4, 29.7
//   D16   256 of 3 / 7 / 9 / 19         7.04, 9.40, 11.7, 17.9 -> 7.59, 9.57, 10.9, 16.3
inline bool fwd_shares_keys(int head_dim, int tiles, int kv_tiles) {
  return tiles <= 128 || (head_dim <= 64 && tiles <= 256 && kv_tiles >= 8);
}

// fp32: 16-row blocks per workgroup (1, 2 or 4 of a 64-row tile's four; the waves
// share out the keys in fours, in twos, not at all) of a forward or dQ grid of
// `tiles` tiles. One or two where these workgroups (16 KB x head_dim / 16 of LDS
// each for one block, half of it for two) run at once; no shares of one or two kv
// tiles. Forward us with 1 / 2 / 4 blocks, 3 and 19 kv tiles a row:
//   D128   64 tiles  13.1 / 15.7 / 22.0, 46.7 / 62.8 / 101
//         128        24.3 / 17.0 / 23.5, 87.1 / 64.5 / 102
//         256, 512   46.3 / 25.8 / 26.1, 89.1 / 46.2 / 40.2 (3 kv tiles)
//   D64   128        11.3 / 11.5 / 15.1, 34.8 / 41.7 / 61.9
//         192        18.2 / 15.7 / 15.7, 61.0 / 56.9 / 62.0
//         384, 512   29.4 / 21.8 / 23.3, 38.3 / 27.0 / 25.2 (3 kv tiles)
//   D32   256        12.4 / 12.0 / 11.7, 38.2 / 42.2 / 44.0
//         256 tiles of one kv tile: 7.68 / 7.24 / 6.59 (D128 27.7 / 14.5 / 13.6)
// dQ (backward, dK/dV the same): D128 64, 128, 256 tiles 69.9 / 79.3 / 103, 122 /
// 109 / 133, 188 / 157 / 161; D64 128, 256, 512 61.0 / 62.0 / 74.7, 86.9 / 84.8 /
// 88.1, 195 / 187 / 184.
inline int f32_row_blocks(int head_dim, int tiles, int kv_tiles) {
  if (tiles > 128 && kv_tiles <= 2) return 4;
  return tiles <= (head_dim <= 32 ? 256 : head_dim == 64 ? 128 : 64) ? 1 : tiles <= 384 ? 2 : 4;
}

// The same for the kv blocks of a dK/dV grid of `items` work items (one block would
// spill at head_dim 128). Backward us with 1 / 2 / 4 blocks:
//   D128  94, 188, 504 items     - / 54.7 / 64.1, 77.8 / 69.9, 154 / 138
//   D64   36, 94, 188, 376, 504  25.1 / 27.0 / 32.8, 39.6 / 33.5 / 39.2, 51.0 / 41.7 /
//                                41.7, 82.5 / 62.7 / 60.7, 105 / 72.1 / 68.5
//   D32   36, 94, 188, 376, 504  17.7 / 19.4 / 22.6, 23.4 / 23.2 / 26.2, 27.1 / 27.0 /
//                                27.4, 40.1 / 36.4 / 37.7, 49.6 / 44.0 / 42.3
inline int f32_kv_blocks(int head_dim, int items) {
  if (head_dim >= 128) return items <= 128 ? 2 : 4;
  return items <= (head_dim == 64 ? 64 : 128) ? 1 : items <= (head_dim == 64 ? 256 : 384) ? 2 : 4;
}

// XCD-aware remap: hardware dispatches workgroup b to XCD b % 8. Give each XCD
// one contiguous range of logical ids so neighbouring q tiles of one head (which
// share most K/V tiles) run on the same XCD and hit in its L2.
constexpr int kXcd = 8;
// First logical id of XCD x's range (of n); the range holds n / 8 ids, one more
// for the first n % 8 XCDs (as many as the hardware hands that XCD).
__host__ __device__ inline int xcd_start(int x, int n) {
  const int per = n / kXcd, rem = n % kXcd;
  return x < rem ? x * (per + 1) : rem * (per + 1) + (x - rem) * per;
}
__host__ __device__ inline int xcd_remap(int b, int n) { return xcd_start(b % kXcd, n) + b / kXcd; }

// Wave issue priority around a cluster of MFMAs (ON: the D <= 64 kernels).
// While a wave issues its products it wins the SIMD's issue arbitration over
// the waves in their softmax / dS VALU phase, so the matrix pipe is fed more
// evenly: at D = 64 (four waves per SIMD) the forward ran 2% and the
// backward 0.5-1.3% faster on long StreamingLLM sequences; at D = 128 (two
// waves per SIMD) it made the forward 3% slower, so it is off there.
template <bool ON>
__device__ inline void mfma_priority_hi() {
  if constexpr (ON) __builtin_amdgcn_s_setprio(1);
}
template <bool ON>
__device__ inline void mfma_priority_lo() {
  if constexpr (ON) __builtin_amdgcn_s_setprio(0);
}

// Work unit of workgroup b in a launch over n units: its XCD-remapped logical
// id, or, with an order table (gki_fwd_order), the unit that table lists at
// that id (each XCD's range sorted heaviest first, so the units dispatched last
// are the short ones and the launch ends with less idle tail). -1 (the
// workgroup exits) for a table entry outside 0 .. n-1.
__device__ inline int work_of(int b, int n, const int32_t* order) {
  const int l = xcd_remap(b, n);
  if (order == nullptr) return l;
  const int w = __builtin_amdgcn_readfirstlane(order[l]);
  return (unsigned)w < (unsigned)n ? w : -1;
}

// The same for units cut into `parts` workgroups each (grid work_parts_grid):
// the parts of a unit run on one XCD, one after the other.
inline int work_parts_grid(int n, int parts) { return parts == 1 ? n : kXcd * parts * ((n + kXcd - 1) / kXcd); }
__device__ inline int work_part_of(int b, int n, int parts, const int32_t* order, int& part) {
  const int x = b % kXcd, k = b / kXcd, slot = x + kXcd * (k / parts);
  part = k % parts;
  return slot < n ? work_of(slot, n, order) : -1;
}

// Reductions across the 4 lane groups (lanes l, l^16, l^32, l^48) with the
// gfx950 VALU row swaps, no LDS trip. v_permlane32_swap a, b exchanges the
// upper 32 lanes of a with the lower 32 lanes of b; with a = b = x, lane l then
// holds {x[l], x[l^32]} in (a, b). v_permlane16_swap does the same for odd /
// even 16-lane rows ({x[l], x[l^16]}). Inline asm because the compiler's
// builtin returns the first register for both results (checked on gfx950);
// the s_nop pairs keep the VALU -> permlane -> VALU wait states.
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
__device__ inline void swap32(float& a, float& b) {
  asm("s_nop 1\n\tv_permlane32_swap_b32 %0, %1\n\ts_nop 1" : "+v"(a), "+v"(b));
}
__device__ inline void swap16(float& a, float& b) {
  asm("s_nop 1\n\tv_permlane16_swap_b32 %0, %1\n\ts_nop 1" : "+v"(a), "+v"(b));
}
#pragma clang diagnostic pop
// DPP row permute of a float (VALU rate, no LDS): CTRL is a gfx9 dpp_ctrl
// code; all rows / banks enabled, every source lane lies in the same 16-lane row.
template <int CTRL>
__device__ inline float dpp_perm(float x) {
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), CTRL,
                                                               0xF, 0xF, false));
}
constexpr int kDppXor1 = 0xB1;        // quad_perm [1,0,3,2]
constexpr int kDppXor2 = 0x4E;        // quad_perm [2,3,0,1]
constexpr int kDppHalfMirror = 0x141; // lane i of each 8 reads lane 7-i
constexpr int kDppMirror = 0x140;     // lane i of each 16 reads lane 15-i

// Sum over aligned groups of N lanes (N a power of two, 1..64); every lane gets
// its group's sum. Once the lanes of each quad (8, 16-lane half) hold equal
// values, the mirrors pair each with the other quad (half): no LDS traffic.
template <int N>
__device__ inline float group_sum(float x) {
  if constexpr (N >= 2) x += dpp_perm<kDppXor1>(x);
  if constexpr (N >= 4) x += dpp_perm<kDppXor2>(x);
  if constexpr (N >= 8) x += dpp_perm<kDppHalfMirror>(x);
  if constexpr (N >= 16) x += dpp_perm<kDppMirror>(x);
  if constexpr (N >= 32) {
    float a = x, b = x;
    swap16(a, b);
    x = a + b;
  }
  if constexpr (N >= 64) {
    float a = x, b = x;
    swap32(a, b);
    x = a + b;
  }
  return x;
}

// Max across the 64/N aligned groups of N lanes, for values that are uniform
// within each group (so any pairing of whole groups is a valid exchange).
template <int N>
__device__ inline float cross_group_max(float x) {
  if constexpr (N <= 1) x = fmaxf(x, dpp_perm<kDppXor1>(x));
  if constexpr (N <= 2) x = fmaxf(x, dpp_perm<kDppXor2>(x));
  if constexpr (N <= 4) x = fmaxf(x, dpp_perm<kDppHalfMirror>(x));
  if constexpr (N <= 8) x = fmaxf(x, dpp_perm<kDppMirror>(x));
  if constexpr (N <= 16) {
    float a = x, b = x;
    swap16(a, b);
    x = fmaxf(a, b);
  }
  if constexpr (N <= 32) {
    float a = x, b = x;
    swap32(a, b);
    x = fmaxf(a, b);
  }
  return x;
}

// Swaps and maxes in one asm block: through fmaxf the compiler canonicalises
// both asm outputs (v_max x, x, x) before every max.
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
__device__ inline float wave_max16x4(float x) {
  float a = x, b = x;
  asm("s_nop 1\n\tv_permlane32_swap_b32 %0, %1\n\ts_nop 1\n\tv_max_f32 %0, %0, %1\n\t"
      "v_mov_b32 %1, %0\n\ts_nop 1\n\tv_permlane16_swap_b32 %0, %1\n\ts_nop 1\n\t"
      "v_max_f32 %0, %0, %1"
      : "+v"(a), "+v"(b));
  return a;
}
#pragma clang diagnostic pop
// Max / sum of lanes l and l ^ 32 (a column's two halves in a 32x32 accumulator).
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
__device__ inline float half_max(float x) {
  float a = x, b = x;
  asm("s_nop 1\n\tv_permlane32_swap_b32 %0, %1\n\ts_nop 1\n\tv_max_f32 %0, %0, %1" : "+v"(a), "+v"(b));
  return a;
}
#pragma clang diagnostic pop
__device__ inline float half_sum(float x) {
  float a = x, b = x;
  swap32(a, b);
  return a + b;
}
__device__ inline float wave_sum16x4(float x) {
  float a = x, b = x;
  swap32(a, b);
  x = a + b;
  a = x;
  b = x;
  swap16(a, b);
  return a + b;
}

constexpr float kLog2e = 1.4426950408889634f;
constexpr float kNegInf = -__builtin_huge_valf();

// The kernels keep each row's running max m2 and sum l in base 2 (scores
// times log2 e); the stored LSE is the natural log-sum-exp m + ln(l)
// (sparse_triton_kernel.py:351). Both conversions run once per row in double,
// so each is a single fp32 rounding of the exact value.
__device__ inline float lse_natural(float m2, float l) {
  return (float)(((double)m2 + (double)log2f(l)) * 0.6931471805599453);
}
__device__ inline float lse_base2(float lse) { return (float)((double)lse * 1.4426950408889634); }

}  // namespace gki

// ---------------------------------------------------------------------------
// Host-side error plumbing for the C ABI.
// ---------------------------------------------------------------------------
namespace gki {
void set_error(const std::string& msg);
int fail(int code, const std::string& msg);
int check_launch(const char* what);
}  // namespace gki

#define GKI_REQUIRE(cond, code, msg)          \
  do {                                        \
    if (!(cond)) return ::gki::fail(code, msg); \
  } while (0)
