// gnf4_device.h -- device code and launch arguments shared by the HIP sources
// of the grouped 4-bit expert GEMM (gfx950): weight decode, LDS tables,
// buffer resources, waits, kernel arguments.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

#include "../../include/gnf4_hip.h"

namespace gnf4 {

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8_t;
typedef __attribute__((ext_vector_type(2))) __bf16 bf16x2_t;
typedef __attribute__((ext_vector_type(4))) float f32x4_t;
typedef __attribute__((ext_vector_type(4))) unsigned u32x4_t;
typedef __attribute__((ext_vector_type(2))) unsigned u32x2_t;
typedef __attribute__((ext_vector_type(2))) int v2i32_t;

constexpr int kNF4 = GNF4_FMT_NF4;
constexpr int kMX = GNF4_FMT_MXFP4;

// NF4 codebook, reference kernel/nf4_grouped.py:53-70 (code 7 is exactly 0).
static __constant__ float c_nf4[16] = {
    -1.0f, -0.6961928009986877f, -0.5250730514526367f, -0.39491748809814453f,
    -0.28444138169288635f, -0.18477343022823334f, -0.09105003625154495f, 0.0f,
    0.07958029955625534f, 0.16093020141124725f, 0.24611230194568634f,
    0.33791524171829224f, 0.44070982933044434f, 0.5626170039176941f,
    0.7229568362236023f, 1.0f,
};

// ---------------------------------------------------------------- decode --

// The NF4 pair table: 256 bytes x 32 lane columns x float2 = 64 KiB. Entry
// (byte, column) holds the fp32 pair (NF4[byte >> 4], NF4[byte & 15]) in the
// column of lane % 32, so the lanes one LDS pass serves read distinct banks.
// Declared first so it sits at LDS offset 0: one v_perm_b32 then forms the
// full address byte << 8 | (lane % 32) * 8.
constexpr int kPairEntries = 256 * 32;

// Codebook entry `lane % 16` in one register per lane. Kernels load it before
// any weight load: vector loads complete in order, so a codebook read issued
// after the weights would hold the table build until every weight landed.
__device__ __forceinline__ int nf4_lut_lane() {
  return __float_as_int(c_nf4[threadIdx.x & 15]);
}

__device__ __forceinline__ void init_pair_table(float2* tab, int lut) {
  // Thread t fills the columns of byte t % 256 (all 32 of them with 256
  // threads, half of them with 512), rotating the column order by byte so one store instruction
  // touches distinct banks. Entries come from the codebook register of lanes
  // 0..15 through ds_bpermute.
  const unsigned b = threadIdx.x & 255;
  const float hi = __int_as_float(__builtin_amdgcn_ds_bpermute((int)((b >> 4) << 2), lut));
  const float lo = __int_as_float(__builtin_amdgcn_ds_bpermute((int)((b & 15) << 2), lut));
  const float2 e = make_float2(hi, lo);
  // with 512 threads the second 256 fill the other half of the columns
  const int j0 = threadIdx.x < 256 ? 0 : 16;
  const int nj = blockDim.x > 256 ? 16 : 32;
  for (int j = 0; j < nj; ++j) tab[b * 32 + ((j0 + j + b) & 31)] = e;
}

// Codebook value c (0..15) from immediate constants (a select chain): no
// memory load, so a table built from it need not wait for any.
__device__ __forceinline__ float nf4_code_imm(unsigned c) {
  float r = -1.0f;
  r = c == 1 ? -0.6961928009986877f : r;
  r = c == 2 ? -0.5250730514526367f : r;
  r = c == 3 ? -0.39491748809814453f : r;
  r = c == 4 ? -0.28444138169288635f : r;
  r = c == 5 ? -0.18477343022823334f : r;
  r = c == 6 ? -0.09105003625154495f : r;
  r = c == 7 ? 0.0f : r;
  r = c == 8 ? 0.07958029955625534f : r;
  r = c == 9 ? 0.16093020141124725f : r;
  r = c == 10 ? 0.24611230194568634f : r;
  r = c == 11 ? 0.33791524171829224f : r;
  r = c == 12 ? 0.44070982933044434f : r;
  r = c == 13 ? 0.5626170039176941f : r;
  r = c == 14 ? 0.7229568362236023f : r;
  r = c == 15 ? 1.0f : r;
  return r;
}

// The pair table of init_pair_table (64 KiB at LDS offset 0, 32 lane
// columns) filled by 512 threads from nf4_code_imm: thread t fills 16
// columns of byte t % 256.
__device__ __forceinline__ void init_pair_table_imm(char* smem) {
  const unsigned b = threadIdx.x & 255;
  const float2 e = make_float2(nf4_code_imm(b >> 4), nf4_code_imm(b & 15));
  const int j0 = threadIdx.x < 256 ? 0 : 16;
  float2* tab = reinterpret_cast<float2*>(smem);
#pragma unroll
  for (int j = 0; j < 16; ++j) tab[b * 32 + ((j0 + j + b) & 31)] = e;
}

// The same with 16 columns (32 KiB: entry (byte b, column c) at b * 128 + c * 8).
__device__ __forceinline__ void init_pair_table16_imm(char* smem) {
  const unsigned b = threadIdx.x & 255;
  const float2 e = make_float2(nf4_code_imm(b >> 4), nf4_code_imm(b & 15));
  const int j0 = threadIdx.x < 256 ? 0 : 8;
  float2* tab = reinterpret_cast<float2*>(smem);
#pragma unroll
  for (int j = 0; j < 8; ++j) tab[b * 16 + ((j0 + j + b) & 15)] = e;
}

__device__ __forceinline__ unsigned bf16x2_bits(float lo, float hi) {
  bf16x2_t r = {(__bf16)lo, (__bf16)hi};  // v_cvt_pk_bf16_f32, RNE
  return __builtin_bit_cast(unsigned, r);
}

// 8 NF4 elements of one packed dword -> 4 dwords of bf16 pairs in k order.
// lane_off = (lane % 32) * 8: the lane's private column in the pair table.
__device__ __forceinline__ u32x4_t nf4_dword_to_bf16(const float2* tab, unsigned x,
                                                     unsigned lane_off, float s) {
  u32x4_t r;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const unsigned addr = __builtin_amdgcn_perm(x, lane_off, 0x0C0C0000u | ((4u + i) << 8));
    const float2 p = *reinterpret_cast<const float2*>(reinterpret_cast<const char*>(tab) + addr);
    r[i] = bf16x2_bits(p.x * s, p.y * s);
  }
  return r;
}

// ---- exact three-part NF4 codebook (decode kernels) ----
//
// Every fp32 codebook value v splits exactly into three bf16 values,
// v = hi + mid + lo: hi keeps the top 16 bits of v's pattern (sign, exponent,
// 7 mantissa bits), the remainder r = v - hi is exact with at most 16
// significant bits, mid keeps r's top 16 bits and lo = r - mid is exact with
// at most 8 significant bits. Three bf16 MFMAs over the parts therefore sum
// codebook values at full fp32 precision (each product of a bf16 activation
// and a bf16 part is exact in fp32), and absmax multiplies the 64-element
// block sum once, in fp32, as the reference's GEMV does
// (kernel/nf4_grouped.py:508-511).
//
// The split table: 256 bytes x 16 lane columns x 16 B = 64 KiB. Entry (byte,
// column) holds the bf16 pairs (part[byte >> 4], part[byte & 15]) of hi, mid
// and lo in dwords 0..2 (element 2j, the high nibble, in the low half), so
// one 16-byte LDS read decodes a byte into the three MFMA operand dwords.
// Column = lane % 16: the 16 lanes of one LDS pass read distinct banks.
constexpr int kSplitCols = 16;
constexpr int kSplitTabBytes = 256 * kSplitCols * 16;
static_assert(kSplitTabBytes == 8 * kPairEntries, "split and pair tables take the same LDS");

__device__ __forceinline__ void nf4_split_parts(int lut, unsigned& himid, unsigned& lo) {
  const unsigned u = (unsigned)lut;
  const unsigned h = u & 0xFFFF0000u;
  const float r = __uint_as_float(u) - __uint_as_float(h);          // exact
  const unsigned rm = __float_as_uint(r) & 0xFFFF0000u;
  const float l = r - __uint_as_float(rm);                           // exact
  himid = (h >> 16) | rm;                  // hi in the low half, mid in the high half
  lo = __float_as_uint(l) >> 16;
}

// Fill the split table from the codebook register of lanes 0..15 (see
// nf4_lut_lane). Thread t fills byte t % 256; with 512 threads each byte's
// 16 columns are split over two threads. Columns rotate with the byte so one
// store instruction touches distinct banks.
__device__ __forceinline__ void init_split_table(char* tab, int lut) {
  unsigned hm, lo;
  nf4_split_parts(lut, hm, lo);
  const unsigned b = threadIdx.x & 255;
  const unsigned hmh = __builtin_amdgcn_ds_bpermute((int)((b >> 4) << 2), (int)hm);
  const unsigned hml = __builtin_amdgcn_ds_bpermute((int)((b & 15) << 2), (int)hm);
  const unsigned loh = __builtin_amdgcn_ds_bpermute((int)((b >> 4) << 2), (int)lo);
  const unsigned lol = __builtin_amdgcn_ds_bpermute((int)((b & 15) << 2), (int)lo);
  const u32x4_t e = {(hmh & 0xFFFFu) | (hml << 16), (hmh >> 16) | (hml & 0xFFFF0000u),
                     loh | (lol << 16), 0u};
  const int nj = blockDim.x > 256 ? 8 : 16;
  const int j0 = threadIdx.x < 256 ? 0 : 8;
  for (int j = 0; j < nj; ++j)
    *reinterpret_cast<u32x4_t*>(tab + b * (kSplitCols * 16) + (((j0 + j + b) & 15) * 16)) = e;
}

// 16-byte LDS read at a byte address: no base pointer arithmetic around it.
typedef __attribute__((address_space(3))) const u32x4_t lds_u32x4_t;
__device__ __forceinline__ u32x4_t lds_read16(unsigned addr) {
  return *(lds_u32x4_t*)(size_t)addr;
}
// The three bf16 parts of the four bytes of w (lane column lane_off), as the
// hi, mid and lo MFMA operands. One 16-byte read per byte: three separate
// 4-byte reads per byte into the operand registers measured 1.85x slower
// (three times the LDS instructions, four lanes per bank), 12-byte reads
// 2-10 % slower.
__device__ __forceinline__ void split_lookup(unsigned w, unsigned lane_off, u32x4_t& hi,
                                             u32x4_t& mid, u32x4_t& lo) {
  u32x4_t d[4];
#pragma unroll
  for (int b = 0; b < 4; ++b)
    d[b] = lds_read16(__builtin_amdgcn_perm(w, lane_off, 0x0C0C0000u | ((4u + b) << 8)));
  hi = u32x4_t{d[0][0], d[1][0], d[2][0], d[3][0]};
  mid = u32x4_t{d[0][1], d[1][1], d[2][1], d[3][1]};
  lo = u32x4_t{d[0][2], d[1][2], d[2][2], d[3][2]};
}
typedef __attribute__((ext_vector_type(2))) float f32x2_t;
typedef __attribute__((address_space(3))) const f32x2_t lds_f32x2_t;
__device__ __forceinline__ f32x2_t lds_read8f(unsigned addr) {
  return *(lds_f32x2_t*)(size_t)addr;
}

// 8 MXFP4 elements of one packed dword (low nibble first) -> 4 bf16 pairs.
__device__ __forceinline__ u32x4_t mx_dword_to_bf16(unsigned x, float s) {
  u32x4_t r;
  r[0] = __builtin_bit_cast(unsigned, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(x, s, 0));
  r[1] = __builtin_bit_cast(unsigned, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(x, s, 1));
  r[2] = __builtin_bit_cast(unsigned, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(x, s, 2));
  r[3] = __builtin_bit_cast(unsigned, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(x, s, 3));
  return r;
}

// e8m0 byte -> fp32 2^(e - 127): e = 0 is the subnormal 2^-127, e = 255 is
// +inf (so a 0xFF block decodes to +-inf, and zero codes to NaN, like an
// exp2-multiply decode; reference kernel/mxfp4_grouped.py:13-15).
__device__ __forceinline__ float e8m0_to_f32(unsigned e) {
  return __uint_as_float(e == 0 ? 0x00400000u : (e << 23));
}

// Calls fn(integral_constant<I>) for I = 0 .. S - 1 while it returns true.
template <int I, int S>
struct StepUnroll {
  template <class Fn>
  __device__ __forceinline__ static bool run(Fn& fn) {
    if (!fn(std::integral_constant<int, I>{})) return false;
    return StepUnroll<I + 1, S>::run(fn);
  }
};
template <int S>
struct StepUnroll<S, S> {
  template <class Fn>
  __device__ __forceinline__ static bool run(Fn&) { return true; }
};

__device__ __forceinline__ bf16x8_t as_bf16x8(u32x4_t v) {
  return __builtin_bit_cast(bf16x8_t, v);
}

__device__ __forceinline__ f32x4_t mfma(u32x4_t a, u32x4_t b, f32x4_t c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf16x8(a), as_bf16x8(b), c, 0, 0, 0);
}

// Activation chunk (8 consecutive elements) as bf16 bits. fp16 inputs are
// rejected on the host before launch; the kernels take bf16.
__device__ __forceinline__ u32x4_t load_a8(const uint16_t* p) {
  return *reinterpret_cast<const u32x4_t*>(p);
}

__device__ __forceinline__ uint16_t f32_to_bf16_bits(float f) {
  __bf16 b = (__bf16)f;
  return __builtin_bit_cast(uint16_t, b);
}

// ============================================================ decode fwd ==

struct FwdArgs {
  const uint16_t* a;        // [T, lda] bf16
  int64_t lda;
  const uint8_t* B;         // [E, N, K/2]
  int64_t sbe, sbn;         // bytes
  const void* S;            // absmax f32 [E, N, K/64] or e8m0 u8 [E, N, K/32]
  int64_t sse, ssn;         // elements
  const int32_t* eids;      // [G]
  const int32_t* row_off;   // [G + 1] (ro_shift 0), [2 G] (ro_shift 1), or
                            // null: group g is the single row g
  const int32_t* t_row0;    // [n_mtiles] (gemm path)
  const int32_t* t_rows;
  const int32_t* t_group;
  int n_mtiles;
  int G;
  int max_m;                // largest group (decode path)
  // decode path: group g's rows are [row_off[g << ro_shift],
  // row_off[(g << ro_shift) + 1]): ro_shift 0 reads the G + 1 prefix offsets,
  // 1 a (first, end) pair per group, so the groups may come in any order
  int ro_shift;
  int64_t N, K;
  uint16_t* out;            // [T, ldo] bf16
  int64_t ldo;
  // host only: group ids and row offsets to pass in the GEMV kernels'
  // arguments (GemvIds), or null (the kernels read eids / row_off)
  const struct GemvIds* ids_inline;
  // host only: the groups come from device routing and any of them may be
  // empty (the launch covers a bound of the active groups)
  int sparse_groups;
};

// The groups of a decode launch of at most kGemvIdsMax groups, in the GEMV
// kernels' arguments (n > 0): the kernel reads them from the kernarg
// segment it loads anyway, instead of a table in memory behind it (one
// dependent round trip before the first weight load). Entry y (grid row y)
// is a group: its expert id e[y] and rows[y] = first row << 8 | row count.
// The host lists the groups largest first, so the workgroups of the groups
// that take the most passes are dispatched first (every output row is
// computed on its own: the order changes no bits). has_ro: the caller gave
// row offsets (the multi-row GEMV needs them).
constexpr int kGemvIdsMax = 384;
constexpr int kGemvRowsMax = 1 << 23;   // first rows must fit in rows[y] >> 8
struct GemvIds {
  int32_t e[kGemvIdsMax];
  int32_t rows[kGemvIdsMax];
  int32_t n;
  int32_t has_ro;
};

constexpr int kOOB = (int)0x80000000;  // buffer offset past every resource: loads 0

// Buffer resources: raw loads through them are bounds-checked by the
// hardware, so a masked lane gets zeros without a branch (and the compiler
// keeps exact vmcnt counts for the prefetched loads). The check covers the
// lane's offset plus the scalar one: the tile kernels' loads rely on it for
// rows past a tile and behind an expert, their stores for rows past a tile.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t make_rsrc(const void* base, int64_t bytes) {
  const int n = bytes < 0x7FFFFFFF ? (int)bytes : 0x7FFFFFFF;
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), 0, n, 0x00020000);
}

__device__ __forceinline__ u32x4_t buf_load16(__amdgpu_buffer_rsrc_t r, int off) {
  return __builtin_bit_cast(u32x4_t, __builtin_amdgcn_raw_buffer_load_b128(r, off, 0, 0));
}

// Cache-policy bits of a buffer access: kScopeDevice (sc1) makes the access
// coherent at device scope, across the XCDs' separate L2 caches, without any
// cache writeback or invalidate.
constexpr int kScopeDevice = 16;

template <int kAux>
__device__ __forceinline__ u32x4_t buf_load16_aux(__amdgpu_buffer_rsrc_t r, int off) {
  return __builtin_bit_cast(u32x4_t, __builtin_amdgcn_raw_buffer_load_b128(r, off, 0, kAux));
}

__device__ __forceinline__ unsigned buf_load1(__amdgpu_buffer_rsrc_t r, int off) {
  return __builtin_amdgcn_raw_buffer_load_b8(r, off, 0, 0);
}

// off | 0x80000000 when !ok, through an opaque VALU op so the compiler cannot
// turn the masked load back into a branch around two loads.
__device__ __forceinline__ int oob_unless(bool ok, int off) {
  const int mask = ok ? 0 : kOOB;
  int r;
  asm volatile("v_or_b32 %0, %1, %2" : "=v"(r) : "v"(off), "v"(mask));
  return r;
}

template <int FMT>
__device__ __forceinline__ float load_scale(const FwdArgs& p, int64_t e, int64_t n, int64_t k) {
  if constexpr (FMT == kNF4) {
    const float* s = static_cast<const float*>(p.S);
    return s[e * p.sse + n * p.ssn + (k >> 6)];
  } else {
    const uint8_t* s = static_cast<const uint8_t*>(p.S);
    return e8m0_to_f32(s[e * p.sse + n * p.ssn + (k >> 5)]);
  }
}

// ------------------------------------------------------------- tiles --

// cache-policy operand of a buffer store: nt (non-temporal) on gfx950
constexpr int kNonTemporal = 2;

// A 16-byte non-temporal buffer store. The offset is the lane's alone: the
// store reads its data registers after it issues, and behind a store with a
// scalar offset as well the compiler allows a VALU write to one of them in the
// very next instruction, which replaced that dword of the stored data.
__device__ __forceinline__ void store_b128(u32x4_t v, __amdgpu_buffer_rsrc_t r, int voff) {
  __builtin_amdgcn_raw_buffer_store_b128(v, r, voff, 0, kNonTemporal);
}

// s_waitcnt with vmcnt(n) and lgkmcnt(0), expcnt untouched (gfx9 encoding).
template <int n>
__device__ __forceinline__ void wait_vm_lgkm0() {
  static_assert(n >= 0 && n < 64, "vmcnt range");
  __builtin_amdgcn_s_waitcnt((n & 15) | (7 << 4) | (0 << 8) | ((n >> 4) << 14));
}

// Between LDS writes and reads of one wave that hand data from lane to lane
// without a workgroup barrier. The LDS serves a wave's accesses in order, so
// nothing waits; but to the compiler each lane is a thread of its own, and it
// may keep the value of an earlier read on the path of the lanes that did not
// write since.
__device__ __forceinline__ void wave_lds_fence() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

typedef __attribute__((address_space(3))) void* lds_ptr_t;

// Values the kernel knows to be wave-uniform but the compiler may not (it
// would otherwise keep buffer descriptors in VGPRs and loop over lanes).
__device__ __forceinline__ int uniform(int v) { return __builtin_amdgcn_readfirstlane(v); }
template <class T>
__device__ __forceinline__ void* uniform_ptr(const T* ptr) {
  const uint64_t v = reinterpret_cast<uint64_t>(ptr);
  const uint64_t lo = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)v);
  const uint64_t hi = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(v >> 32));
  return reinterpret_cast<void*>(lo | (hi << 32));
}
typedef float f32x16_t __attribute__((ext_vector_type(16)));

// LDS slot swizzle of a staged activation row: 16-byte slot s of row m lives
// at slot s ^ pf_swz(m % 16). Over the 16 rows one operand read touches this
// spreads the 16-byte pieces across all 64 banks.
__device__ __forceinline__ int pf_swz(int m16) { return (m16 ^ (m16 >> 3)) & 7; }

struct PfTile {
  int row0, rows, e, n0;
};

// A tile table small enough to travel in the kernel arguments (n > 0): no
// upload, so a call needs no copy ahead of its launch (and a captured graph
// no copy node). grp holds the group index, or the expert id itself where
// the caller knows the ids on the host (grp_is_expert). 3 KiB, inside the
// kernel-argument limit with FwdArgs.
constexpr int kPwMaxTiles = 256;
struct PwTiles {
  int32_t row0[kPwMaxTiles];
  int32_t rows[kPwMaxTiles];
  int32_t grp[kPwMaxTiles];
  int32_t n;
  int32_t grp_is_expert;
};

}  // namespace gnf4
