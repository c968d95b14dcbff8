// gnf4_tile.hip -- the eight-wave tile kernels of the grouped 4-bit expert
// GEMM on gfx950: the forward (up to 256 token rows of one group x 256 weight
// rows per tile) and the dgrad of groups of up to 160 rows (k_tile_dgrad).
//
// k_tile_fwd: eight waves (two per SIMD) on a persistent grid of one workgroup
// per CU. Wave w owns 32 weight rows for all of the tile's token rows, so no
// weight is decoded twice; a tile runs its own 32-row subtiles only (kM = 1..8,
// one instantiation each). k advances in steps of 64:
//   * activations: a ring of LDS stages filled by direct-to-LDS loads, one
//     barrier per step; each 16-byte operand read feeds one 32x32x16 MFMA;
//   * packed weights: 16 bytes per lane and step straight into a register
//     ring, asked for two or four steps at a time, because the 32-byte pieces
//     of a row share cache lines (4.5 M L2 requests per launch at 32 rows per
//     group, 128 experts, N = 1536, K = 2048; 13.1 M one step at a time),
//     scales four steps at a time;
//   * decode: NF4 through the 32-column pair table (64 KiB of LDS; with 16
//     columns two lanes share a bank pair and a wave pair reads 128 B per
//     clock instead of 256), MXFP4 by the convert instruction; spread between
//     the MFMAs ("rolling") or a step at a time ("phase", short tiles);
//   * the loads run on into the workgroup's next tile, so a tile starts with
//     its first stages and weights in LDS and registers.
// Why eight waves of 32 rows and not four of 64 (half the operand reads): one
// wave per SIMD issues one instruction in four clocks and waits out every LDS
// round trip: 3100 clocks per step at 256 rows and 2500 at 32, where the MFMAs
// need 2048 and 256; this form takes 2330 and 1270 (MXFP4 2310 and 780; clock
// stamps in a measuring build).
// What bounds it: at 256 rows the power limit (283 k clocks per CU in 184 us,
// 1.5 GHz, where 32 rows run at 2.0; the matrix cores are busy 70 % of all
// clocks, 88 % within the steps), below 100 rows the LDS lookups and the VALU
// that follow each other in the step. NF4 takes all 256 registers and spills
// 24 of them (52 bytes of scratch a lane), none within a tile's step loop.
// Measured (MI355X, 128 experts, N = 1536, K = 2048, NF4; 32 / 64 / 128 / 256
// rows per group): 75 / 90 / 118 / 187 us; the four-wave kernel before it 111
// / 122 / 143 / 215 us. N = 2048, K = 768, 256 rows: 104-107 against 126 us.
// MXFP4, 32 experts, N = 5760, K = 2880, 32 / 128 / 256 rows: 84 / 133 / 226
// against 144 / 166 / 239 us.

#include "gnf4_device.h"
#include "gnf4_tile.h"

using namespace gnf4;

namespace {

constexpr int kTlWaves = 8;
constexpr int kTlBN = 256;            // weight rows (output columns) per tile
constexpr int kTlBK = 64;             // k per step
constexpr int kTlLds = 160 * 1024;

// an 8-byte load from any address (e8m0 rows start anywhere)
typedef u32x2_t u32x2_a1_t __attribute__((aligned(1)));
typedef __attribute__((address_space(1))) const u32x2_a1_t* global_u32x2_a1_ptr;
typedef __attribute__((address_space(1))) const uint8_t* global_u8_ptr;

template <int n>
__device__ __forceinline__ void wait_vm() {
  static_assert(n >= 0 && n < 64, "vmcnt range");
  __builtin_amdgcn_s_waitcnt((n & 15) | (7 << 4) | (15 << 8) | ((n >> 4) << 14));
}

// LDS: the NF4 pair table at address 0 (64 KiB), the activation ring behind
// it, the output staging area. Where the ring's three 32 KiB stages leave no
// room (NF4, tall tiles) the output is staged in the one stage that is free
// between two tiles.
template <int FMT>
constexpr int kTlBase = FMT == kNF4 ? 64 * 1024 : 0;
constexpr int kTlOut = 32 * 1024;      // two 32-row subtiles of bf16 output

// Tiles of 1..2, 3..4 and 5..8 subtiles stage 64, 128 and 256 rows per step
// (kP pieces of 8 rows x 128 B per wave).
constexpr int pieces_of(int subtiles) { return subtiles <= 2 ? 1 : subtiles <= 4 ? 2 : 4; }

template <int FMT, int kP>
struct Ring {
  static constexpr int kStage = kP * kTlWaves * 1024;
  static constexpr int kRoom = kTlLds - kTlBase<FMT> - kTlOut;
  static constexpr bool kOwnOut = kRoom >= 3 * kStage;      // a staging area of its own
  static constexpr int kFit = kOwnOut ? kRoom / kStage : 3;
  static constexpr int kS = kFit < 8 ? kFit : 8;            // stages
};

// v, as a value the compiler cannot share with other uses of v: what is
// computed from it is neither hoisted out of the tile loop nor kept in
// registers across a tile's step loop (both spilled).
__device__ __forceinline__ int opaque(int v) {
  asm volatile("" : "+v"(v));
  return v;
}

template <int FMT>
using ScaleVec = std::conditional_t<FMT == kNF4, u32x4_t, u32x2_t>;

// The packed weights a tile starts with, loaded during the previous one.
template <int FMT>
struct TileRegs {
  u32x4_t wr[4];          // packed bytes of steps 0..3: lane half h of row n holds k [32 h, +32)
  ScaleVec<FMT> sc;       // scales of steps 0..3
};

// A tile's loads, all uniform: per lane and per step only fixed offsets are
// added. Rows past the tile (activations) or past N (weights) lie past the
// end of their resource and load zeros; resources of no tile have size 0.
template <int FMT>
struct TileSrc {
  const char* a;
  const char* b;
  const char* s;
  int a_bytes, b_bytes, s_bytes, s_rows;
  __device__ __forceinline__ TileSrc(const FwdArgs& p, const PfTile& t) {
    constexpr int kB = FMT == kNF4 ? 4 : 1;
    const bool live = t.rows > 0;
    a = static_cast<const char*>(uniform_ptr(p.a + (int64_t)t.row0 * p.lda));
    b = static_cast<const char*>(uniform_ptr(p.B + (int64_t)t.e * p.sbe + (int64_t)t.n0 * p.sbn));
    s = static_cast<const char*>(uniform_ptr(static_cast<const char*>(p.S) +
                                             ((int64_t)t.e * p.sse + (int64_t)t.n0 * p.ssn) * kB));
    const int n = (int)(p.N - t.n0 < kTlBN ? p.N - t.n0 : kTlBN);
    a_bytes = uniform(live ? (int)((int64_t)t.rows * p.lda * 2) : 0);
    b_bytes = uniform(live ? (int)(n * p.sbn) : 0);
    s_bytes = uniform(live ? (int)(n * p.ssn * kB) : 0);
    s_rows = n;
  }
};

__device__ __forceinline__ __amdgpu_buffer_rsrc_t rsrc_of(const char* base, int bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(base), 0, bytes, 0x00020000);
}

// Lane constants of the weight loads: row wave * 32 + lane % 32 of the tile.
template <int FMT>
struct WeightLoads {
  int b_voff, s_voff, s_row, s_step;
  __device__ __forceinline__ WeightLoads(const FwdArgs& p, int wave, int lane) {
    s_row = wave * 32 + (lane & 31);
    b_voff = (int)(s_row * p.sbn) + (lane >> 5) * 16;
    s_step = (int)p.ssn;
    s_voff = (int)(s_row * p.ssn * 4);
  }
  // packed bytes of step g
  __device__ __forceinline__ u32x4_t bytes(const char* b, int b_bytes, int g) const {
    return __builtin_bit_cast(
        u32x4_t, __builtin_amdgcn_raw_buffer_load_b128(rsrc_of(b, b_bytes), b_voff, g * 32, 0));
  }
  // Scales of steps 4T .. 4T + 3 of F >= 4: a window that ends inside the
  // row (the resource spans all of the tile's rows, so it does not keep a
  // window from running into the next one). MXFP4: rows past N read the last
  // row's.
  __device__ __forceinline__ ScaleVec<FMT> window(const char* s, int s_bytes, int s_rows,
                                                  int s0) const {
    if constexpr (FMT == kNF4) {
      return __builtin_bit_cast(u32x4_t, __builtin_amdgcn_raw_buffer_load_b128(
                                             rsrc_of(s, s_bytes), s_voff, s0 * 4, 0));
    } else {
      const int row = s_row < s_rows ? s_row : s_rows - 1;
      return *(global_u32x2_a1_ptr)(uintptr_t)(s + s0 * 2 + (int64_t)row * s_step);
    }
  }
  __device__ __forceinline__ ScaleVec<FMT> scales(const TileSrc<FMT>& x, int T, int F) const {
    return window(x.s, x.s_bytes, x.s_rows, uniform(4 * T + 4 <= F ? 4 * T : F - 4));
  }
  __device__ __forceinline__ ScaleVec<FMT> first_scales(const TileSrc<FMT>& x, int F) const {
    if (F >= 4) return scales(x, 0, F);
    if constexpr (FMT == kNF4) {
      const __amdgpu_buffer_rsrc_t r = rsrc_of(x.s, x.s_bytes);
      u32x4_t v{};
      v[0] = __builtin_amdgcn_raw_buffer_load_b32(r, s_voff, 0, 0);
      if (F > 1) v[1] = __builtin_amdgcn_raw_buffer_load_b32(r, s_voff, 4, 0);
      if (F > 2) v[2] = __builtin_amdgcn_raw_buffer_load_b32(r, s_voff, 8, 0);
      return v;
    } else {
      const int row = s_row < x.s_rows ? s_row : x.s_rows - 1;
      uint64_t w = 0;
      for (int j = 0; j < 2 * F; ++j)
        w |= (uint64_t)(*(global_u8_ptr)(uintptr_t)(x.s + (int64_t)row * s_step + j)) << (8 * j);
      return u32x2_t{(unsigned)w, (unsigned)(w >> 32)};
    }
  }
};

// Lane constants of the activation loads: piece i of a wave is rows
// (wave * kP + i) * 8 + lane / 8, 16-byte slot lane % 8 (swizzled) of 128 B.
template <int FMT, int kP>
struct ActLoads {
  int voff[kP];
  __device__ __forceinline__ ActLoads(const FwdArgs& p, int wave, int lane) {
#pragma unroll
    for (int i = 0; i < kP; ++i) {
      const int row = (wave * kP + i) * 8 + (lane >> 3);
      voff[i] = (int)(row * p.lda * 2) + ((lane & 7) ^ pf_swz(row & 15)) * 16;
    }
  }
  // piece i of step g into the stage at byte offset `slot` of the ring
  __device__ __forceinline__ void issue(char* smem, int wave, const char* a, int a_bytes, int g,
                                        int slot, int i) const {
    char* dst = smem + kTlBase<FMT> + slot + (wave * kP + i) * 1024;
    __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc_of(a, a_bytes), (lds_ptr_t)dst, 16, voff[i],
                                             g * (kTlBK * 2), 0, 0);
  }
};

template <int FMT>
__device__ __forceinline__ void first_weights(const FwdArgs& p, const TileSrc<FMT>& x, int F,
                                              TileRegs<FMT>& r) {
  const int lane = opaque(threadIdx.x) & 63, wave = uniform(threadIdx.x >> 6);
  const WeightLoads<FMT> w(p, wave, lane);
#pragma unroll
  for (int g = 0; g < 4; ++g) r.wr[g] = w.bytes(x.b, g < F ? x.b_bytes : 0, g);
  r.sc = w.first_scales(x, F);
}
// A tile's first kS - 1 stages, into ring slots 0.. (the low 64 KiB of the
// ring, so never into the staging area).
template <int FMT, int kP>
__device__ __forceinline__ void first_stages(const FwdArgs& p, const TileSrc<FMT>& x, int F,
                                             char* smem) {
  const int lane = opaque(threadIdx.x) & 63, wave = uniform(threadIdx.x >> 6);
  const ActLoads<FMT, kP> a(p, wave, lane);
#pragma unroll
  for (int g = 0; g < Ring<FMT, kP>::kS - 1; ++g)
#pragma unroll
    for (int i = 0; i < kP; ++i)
      a.issue(smem, wave, x.a, g < F ? x.a_bytes : 0, g, g * Ring<FMT, kP>::kStage, i);
}
template <int FMT>
__device__ __forceinline__ void first_stages_of(const FwdArgs& p, const TileSrc<FMT>& x, int rows,
                                                int F, char* smem) {
  switch (pieces_of((rows + 31) >> 5)) {
    case 4: first_stages<FMT, 4>(p, x, F, smem); break;
    case 2: first_stages<FMT, 2>(p, x, F, smem); break;
    default: first_stages<FMT, 1>(p, x, F, smem); break;
  }
}
// fewest loads that first_stages issues after a tile's stage 0
template <int FMT>
constexpr int kFirstAfter0 = [] {
  const int n1 = Ring<FMT, 1>::kS - 2, n2 = 2 * (Ring<FMT, 2>::kS - 2),
            n4 = 4 * (Ring<FMT, 4>::kS - 2);
  return n1 < n2 ? (n1 < n4 ? n1 : n4) : (n2 < n4 ? n2 : n4);
}();

// One tile, t, whose first weights (regs) and stages are loading, stage 0
// published; ring slot `slot0` holds stage 0. On return tn's are (where there
// is a tn), and the slot of its stage 0 is returned.
//
// The loads run on from one tile into the next: where a step's load would be
// past the end of t, it is tn's instead (weights: when the register ring
// comes out even, F % 4 == 0; activations: when tn stages as many rows and the
// ring is no longer than the tile). The
// others of tn's first loads go out at the end of the steps, ahead of the
// output's stores.
template <int FMT, int kM>
__device__ __forceinline__ int tile_fwd(const FwdArgs& p, const PfTile t, const PfTile tn,
                                        char* smem, uint16_t* __restrict__ out,
                                        TileRegs<FMT>& regs, const int slot0) {
  constexpr int kP = pieces_of(kM), kBase = kTlBase<FMT>;
  using Rg = Ring<FMT, kP>;
  constexpr int kS = Rg::kS, kStage = Rg::kStage;
  constexpr int kAhead = kM >= 5 ? 1 : kM >= 3 ? 2 : 4;   // operand reads ahead, in slices
  constexpr int kBar = 4 - kAhead;          // slice whose start publishes the next stage
  static_assert(kS >= 3, "ring depth");
  const int lane = opaque(threadIdx.x) & 63, wave = uniform(threadIdx.x >> 6);
  const int l32 = lane & 31, h = lane >> 5;
  const int F = uniform((int)(p.K / kTlBK));

  // activation operand of slice kk, subtile i: k [32 h + 8 kk, +8) of row
  // i * 32 + l32, at stage + (a_off ^ (kk * 16)) + i * 4096
  const int a_off = l32 * 128 + ((4 * h) ^ pf_swz(l32 & 15)) * 16;
  const unsigned lds0 = (unsigned)(uintptr_t)(lds_ptr_t)smem + kBase;
  auto act_addr = [&](int stage, int kk) {
    unsigned addr = lds0 + stage + (a_off ^ (kk * 16));
    asm("" : "+v"(addr));   // one base per slice: the subtiles are offsets from it
    return addr;
  };
  const unsigned tab_lane = (unsigned)l32 * 8u;

  const TileSrc<FMT> x(p, t), xn(p, tn);
  const bool next = tn.rows > 0;
  // packed weights: a register ring of kU steps, refilled half (kPhase) or two
  // steps at a time, so that the 32-byte pieces of a row that share a cache
  // line are asked for together; the steps are unrolled kU times
  constexpr bool kPhase = kM <= 2;
  constexpr int kU = kPhase ? 8 : 4;
  const bool run_w = next && F % kU == 0;
  const bool run_a = next && F >= kS - 1 && pieces_of((tn.rows + 31) >> 5) == kP;
  const WeightLoads<FMT> wl(p, wave, lane);
  const ActLoads<FMT, kP> al(p, wave, lane);
  // the stream of stages: step g's next, into the ring byte offset a_slot
  const bool a_past = kS - 1 >= F;
  const char* a_ptr = a_past ? xn.a : x.a;
  int a_size = a_past ? (run_a ? xn.a_bytes : 0) : x.a_bytes;
  int a_g = a_past ? kS - 1 - F : kS - 1, a_slot = (slot0 + kS - 1) % kS * kStage;
  auto issue_a = [&](int i) { al.issue(smem, wave, a_ptr, a_size, a_g, a_slot, i); };
  auto next_a = [&](int f) {
    const bool sw = f + kS == F;   // the next stage is the next tile's first
    a_ptr = sw ? xn.a : a_ptr;
    a_size = sw ? (run_a ? xn.a_bytes : 0) : a_size;
    a_g = sw ? 0 : a_g + 1;
    a_slot = a_slot == (kS - 1) * kStage ? 0 : a_slot + kStage;
  };
  int r_slot = slot0 * kStage;   // ring byte offset of the step's stage
  u32x4_t wr[kU];
  ScaleVec<FMT> scn = regs.sc;
#pragma unroll
  for (int j = 0; j < 4; ++j) wr[j] = regs.wr[j];
  // packed bytes of steps g .. g + n - 1 (n divides kU: they are this tile's
  // or, run_w, the next one's)
  auto issue_w = [&](int g, auto NI, auto SI) {
    const bool cur = g < F;
    const char* w = cur ? x.b : xn.b;
    const int sz = cur ? x.b_bytes : run_w ? xn.b_bytes : 0;
    const int g0 = uniform(cur ? g : g - F);
#pragma unroll
    for (int j = 0; j < decltype(NI)::value; ++j)
      wr[(decltype(SI)::value + j) & (kU - 1)] =
          wl.bytes(w, g0 + j < F ? sz : 0, g0 + j);
  };
  if constexpr (kPhase)
#pragma unroll
    for (int j = 4; j < kU; ++j) wr[j] = wl.bytes(x.b, j < F ? x.b_bytes : 0, j);
  using SVec = ScaleVec<FMT>;
  // the next four steps' scale window (the next tile's first one behind the
  // last; a window ends inside the row)
  auto next_scales = [&](int T) -> SVec {
    const bool nt = run_w && 4 * T >= F;
    return wl.window(nt ? xn.s : x.s, nt ? xn.s_bytes : x.s_bytes, nt ? xn.s_rows : x.s_rows,
                     uniform(nt ? 0 : 4 * T + 4 <= F ? 4 * T : F - 4));
  };
  // element j of a scale window
  auto scale_of = [&](const SVec& v, int j) -> float {
    if constexpr (FMT == kNF4) {
      return __uint_as_float(v[j]);
    } else {
      const unsigned b = v[j >> 1] >> ((j & 1) * 16 + 8 * h);
      return e8m0_to_f32(b & 0xFFu);
    }
  };
  // shift a window by d elements towards 0
  auto shift_scales = [&](SVec& v, int d) {
    if constexpr (FMT == kNF4) {
      if (d & 1) { v[0] = v[1]; v[1] = v[2]; v[2] = v[3]; }
      if (d & 2) { v[0] = v[2]; v[1] = v[3]; }
    } else {
      const uint64_t w = ((uint64_t)v[0] | ((uint64_t)v[1] << 32)) >> (16 * d);
      v[0] = (unsigned)w;
      v[1] = (unsigned)(w >> 32);
    }
  };

  // ---- decode, in pieces of one packed byte: a table lookup (NF4), then the
  // scale multiply and bf16 pack. Two forms:
  //   kPhase (short tiles): a step looks up all of the next step's weights at
  //     its start and packs them at its end, one LDS round trip per step (the
  //     two waves of a SIMD taking the halves in opposite order: no faster);
  //   rolling (tall tiles, whose accumulators leave few registers): half a
  //     slice of MFMAs apart; slice kk packs the target of slice kk - 1 and
  //     looks up its last two bytes and the first two of its own target.
  // The target of slice kk is the next step's slice kk.
  u32x4_t wf[kPhase ? 8 : 4];           // MFMA operands
  f32x2_t tp[kPhase ? 16 : 4];          // NF4: looked-up pairs
  auto look = [&](int e, unsigned x, int pc) {
    if constexpr (FMT == kNF4)
      tp[e] = lds_read8f(__builtin_amdgcn_perm(x, tab_lane, 0x0C0C0000u | ((4u + pc) << 8)));
  };
  auto pack = [&](int d, int pc, int e, unsigned x, float sc) {
    if constexpr (FMT == kNF4) {
      wf[d][pc] = bf16x2_bits(tp[e].x * sc, tp[e].y * sc);
    } else {
      bf16x2_t v;
      if (pc == 0) v = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(x, sc, 0);
      else if (pc == 1) v = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(x, sc, 1);
      else if (pc == 2) v = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(x, sc, 2);
      else v = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(x, sc, 3);
      wf[d][pc] = __builtin_bit_cast(unsigned, v);
    }
  };
  using I0 = std::integral_constant<int, 0>;
  using I1 = std::integral_constant<int, 1>;
  using I2 = std::integral_constant<int, 2>;
  using I3 = std::integral_constant<int, 3>;

  // ---- prologue: step 0's operands
  float sc[4];   // sc[j]: scale of step 4T + j
#pragma unroll
  for (int j = 0; j < 4; ++j) sc[j] = scale_of(scn, j);
#pragma unroll
  for (int kk = 0; kk < 4; ++kk) {
    const int e = kPhase ? kk * 4 : 0;
#pragma unroll
    for (int pc = 0; pc < (kPhase || kk < 3 ? 4 : 2); ++pc) look(e + pc, wr[0][kk], pc);
    if (kPhase || kk < 3)
#pragma unroll
      for (int pc = 0; pc < 4; ++pc) pack(kk, pc, e + pc, wr[0][kk], sc[0]);
  }
  u32x4_t av[kAhead][kM];
#pragma unroll
  for (int s = 0; s < kAhead; ++s)
#pragma unroll
    for (int i = 0; i < kM; ++i) av[s][i] = lds_read16(act_addr(slot0 * kStage, s) + i * 4096);
  f32x16_t acc[kM];
#pragma unroll
  for (int i = 0; i < kM; ++i) acc[i] = f32x16_t{};

  // ---- steps. u: f % 4 (compile time)
  auto step = [&](auto UI, auto TL, int f) {
    constexpr bool kTail = decltype(TL)::value;   // no further turn
    constexpr int u = decltype(UI)::value;
    constexpr int un = (u + 1) & (kU - 1);   // ring slot of the next step
    constexpr int us = u & 3;                 // scale
    constexpr int usn = (u + 1) & 3;
    const int st0 = r_slot, st1 = r_slot == (kS - 1) * kStage ? 0 : r_slot + kStage;
    r_slot = st1;
    auto slice = [&](auto KI) {
      constexpr int kk = decltype(KI)::value;
      __builtin_amdgcn_sched_barrier(0);
      if constexpr (kk == kBar) {
        // stage f + 1 has landed: the loads behind it are the weights and
        // scale windows issued in steps f - kS + 3 .. f and the stages
        // f + 2 .. f + kS - 2 (fewer weights in the first steps)
        // (kBar == 0: a step's weights and scales go out behind its barrier)
        constexpr int kD0 = kBar == 0 ? 1 : 0;
        constexpr int nws = [] {
          int n = 0;
          for (int d = kD0; d <= kS - 3 + kD0; ++d) {
            if (kTail && d <= u) continue;   // (what a last, partial turn loads is not counted)
            n += ((u - d) & 3) == 0;
            n += kPhase ? (((u - d) & 3) == 3 ? 4 : 0) : ((u - d) & 1 ? 2 : 0);
          }
          return n;
        }();
        if (kTail && f + 1 == F) {
          // the last step: nothing of this tile is left to publish
        } else if (kS == 3 || f >= kS - 3 + kD0) {
          wait_vm<(kS - 3) * kP + nws>();
        } else {
          wait_vm<(kS - 3) * kP>();
        }
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_sched_barrier(0);
      }
      if constexpr (kPhase && kk < 2) {
#pragma unroll
        for (int j = 2 * kk; j < 2 * kk + 2; ++j)
#pragma unroll
          for (int pc = 0; pc < 4; ++pc) look((j * 4 + pc) & (kPhase ? 15 : 3), wr[un][j], pc);
      }
      // rolling: the targets being packed (tq) and started (wr[un][kk])
      const unsigned tq = kk == 0 ? wr[u][3] : wr[un][(kk + 3) & 3];
      const float tqs = kk == 0 ? sc[us] : sc[usn];
      constexpr int kn = (kk + kAhead) & 3;
      const unsigned src = act_addr((kk + kAhead < 4) ? st0 : st1, kn);
#pragma unroll
      for (int i = 0; i < kM; ++i) {
        acc[i] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
            as_bf16x8(wf[kPhase ? (u & 1) * 4 + kk : kk]), as_bf16x8(av[kk % kAhead][i]), acc[i], 0, 0, 0);
        av[kk % kAhead][i] = lds_read16(src + i * 4096);
        if constexpr (kk == 1 && !kTail && (kPhase ? us == 3 : u % 2 == 1))
          if (i == 0) {
            constexpr int n = kPhase ? 4 : 2;
            issue_w(f + kU + 1 - n, std::integral_constant<int, n>{},
                    std::integral_constant<int, u + kU + 1 - n>{});
          }
        if constexpr (kk == 1 && us == 0 && (!kTail || u + 4 < kU))
          if (i == 0 && (!kTail || f + 4 < F)) scn = next_scales((f >> 2) + 1);
        // a last, partial turn: the next tile's weights
        if constexpr (kk == 1 && kTail)
          if (i == 0 && next && f + 1 == F) {
#pragma unroll
            for (int j = 0; j < 4; ++j) wr[j] = wl.bytes(xn.b, j < F ? xn.b_bytes : 0, j);
            scn = wl.first_scales(xn, F);
          }
        if constexpr (kk == kBar) {
#pragma unroll
          for (int j = 0; j < kP; ++j)
            if ((j * kM) / kP == i) issue_a(j);
          if (i == kM - 1) next_a(f);
        }
        if constexpr (!kPhase) {
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            if ((q * kM) / 4 != i) continue;
            pack((kk + 3) & 3, q, q, tq, tqs);
            if (q < 2) look(q + 2, tq, q + 2);
            else look(q - 2, wr[un][kk], q - 2);
          }
          __builtin_amdgcn_sched_barrier(0);
        }
      }
      if constexpr (kPhase && kk >= 2) {
#pragma unroll
        for (int j = 2 * kk - 4; j < 2 * kk - 2; ++j)
#pragma unroll
          for (int pc = 0; pc < 4; ++pc)
            pack((((u + 1) & 1) * 4 + j) & (kPhase ? 7 : 3), pc, (j * 4 + pc) & (kPhase ? 15 : 3),
                 wr[un][j], sc[usn]);
      }
    };
    if constexpr (us == 3) {
      // the next four steps' scales (fewer than four: the window ends at the
      // row's end)
      const int d = f + 5 - F;
      if (d > 0 && d < 4) shift_scales(scn, d);
      sc[0] = scale_of(scn, 0);
    }
    slice(I0{});
    slice(I1{});
    slice(I2{});
    slice(I3{});
    if constexpr (us == 3) {
#pragma unroll
      for (int j = 1; j < 4; ++j) sc[j] = scale_of(scn, j);
    }
  };
  int f = 0;
  for (; f + kU <= F; f += kU) {
    step(I0{}, std::false_type{}, f);
    step(I1{}, std::false_type{}, f + 1);
    step(I2{}, std::false_type{}, f + 2);
    step(I3{}, std::false_type{}, f + 3);
    if constexpr (kU == 8) {
      step(std::integral_constant<int, kU / 2>{}, std::false_type{}, f + 4);
      step(std::integral_constant<int, kU / 2 + 1>{}, std::false_type{}, f + 5);
      step(std::integral_constant<int, kU - 2>{}, std::false_type{}, f + 6);
      step(std::integral_constant<int, kU - 1>{}, std::false_type{}, f + 7);
    }
  }
  auto tail = [&](auto UI) {
    if (f < F) step(UI, std::true_type{}, f);
    return ++f < F;
  };
  if (f < F) (void)StepUnroll<0, kU - 1>::run(tail);
#pragma unroll
  for (int j = 0; j < 4; ++j) regs.wr[j] = wr[j];
  regs.sc = scn;

  // ---- epilogue: the bf16 tile goes through LDS, two subtiles at a time, so
  // the global stores write whole rows.
  // LDS tile: row r at r * 512 bytes, 16-byte chunk c at (c ^ (r % 32)) * 16.
  __builtin_amdgcn_sched_barrier(0);
  if (run_a) {
    // the ring runs on; every wave is past its last read of step F - 1's slot
    __builtin_amdgcn_s_waitcnt(0xC07F);   // lgkmcnt(0)
    __builtin_amdgcn_s_barrier();
  } else {
    // past-the-end loads write zeros to their slots: let them land
    wait_vm_lgkm0<0>();
    __builtin_amdgcn_s_barrier();
    if (next) first_stages_of<FMT>(p, xn, tn.rows, F, smem);
  }
  char* ob = smem + kBase + (Rg::kOwnOut ? Rg::kRoom
                             : run_a     ? (slot0 + F - 1) % kS * kStage
                                         : (kS - 1) * kStage);
  constexpr int kRound = kM < 2 ? kM : 2;   // subtiles staged at once
  const __amdgpu_buffer_rsrc_t ro = __builtin_amdgcn_make_buffer_rsrc(
      uniform_ptr(out + (int64_t)t.row0 * p.ldo), 0, uniform((int)((int64_t)t.rows * p.ldo * 2)),
      0x00020000);
  const int ldo2 = (int)(p.ldo * 2);
  const int ln = opaque(threadIdx.x) & 63, r32 = ln & 31, hh = ln >> 5;
  const int col = t.n0 + r32 * 8;   // this lane's 16-byte chunk (chunk r32) of a stored row
  const int coff16 = col + 8 <= p.N ? col * 2 + hh * ldo2 : kOOB;
  const int coff8 = col < p.N && col + 8 > p.N ? col * 2 + hh * ldo2 : kOOB;
  const bool straddle = p.N % 8 != 0;
#pragma unroll
  for (int r0 = 0; r0 < kM; r0 += kRound) {
    if (r0 > 0) {
      __builtin_amdgcn_s_waitcnt(0xC07F);   // lgkmcnt(0)
      __builtin_amdgcn_s_barrier();
    }
#pragma unroll
    for (int i = r0; i < (r0 + kRound < kM ? r0 + kRound : kM); ++i)
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const int row = (i - r0) * 32 + r32;
        const int c = wave * 32 + 8 * g + 4 * hh;   // 4 columns
        u32x2_t v;
        v.x = bf16x2_bits(acc[i][4 * g + 0], acc[i][4 * g + 1]);
        v.y = bf16x2_bits(acc[i][4 * g + 2], acc[i][4 * g + 3]);
        *reinterpret_cast<u32x2_t*>(ob + row * 512 + (((c >> 3) ^ r32) << 4) + (c & 7) * 2) = v;
      }
    __builtin_amdgcn_s_waitcnt(0xC07F);   // lgkmcnt(0)
    __builtin_amdgcn_s_barrier();
    const int nsub = (r0 + kRound < kM ? kRound : kM - r0);
    // wave w stores rows 2 (8 j + w) + lane / 32
#pragma unroll
    for (int j = 0; j < nsub * 2; ++j) {
      const int row = (j * 8 + wave) * 2 + hh;
      const u32x4_t v =
          *reinterpret_cast<const u32x4_t*>(ob + row * 512 + ((r32 ^ (row & 31)) << 4));
      const int so = uniform((r0 * 32 + (j * 8 + wave) * 2) * ldo2);
      store_b128(v, ro, coff16 + so);
      if (straddle) {
        u32x2_t v2;
        v2.x = v[0];
        v2.y = v[1];
        __builtin_amdgcn_raw_buffer_store_b64(v2, ro, coff8, so, kNonTemporal);
      }
    }
  }
  // The next tile's stage 0 has landed: behind it are its other first stages
  // and this wave's stores (2 kM, or twice that with straddling columns).
  // Every wave is past its LDS reads.
  if (run_a) {
    if (straddle) wait_vm_lgkm0<(kS - 2) * kP + 4 * kM>();
    else wait_vm_lgkm0<(kS - 2) * kP + 2 * kM>();
  } else {
    if (straddle) wait_vm_lgkm0<kFirstAfter0<FMT> + 4 * kM>();
    else wait_vm_lgkm0<kFirstAfter0<FMT> + 2 * kM>();
  }
  __builtin_amdgcn_s_barrier();
  return run_a ? (slot0 + F) % kS : 0;
}

// A workgroup's share of the tile list: XCD x = blockIdx % 8 takes the x-th
// contiguous eighth of it (m-tile major), its workgroups every stride-th tile
// (tiles come largest first, so each gets one of every size band).
struct TileWalk {
  int width, n_tiles, idx, stride;
  int64_t lo, hi;
  __device__ __forceinline__ TileWalk(const FwdArgs& p, int cols, int col_tiles)
      : width(cols), n_tiles(col_tiles) {
    const int64_t total = (int64_t)p.n_mtiles * n_tiles;
    const int nx = gridDim.x >= 8 ? 8 : 1;
    const int x = (int)(blockIdx.x % nx);
    idx = (int)(blockIdx.x / nx);
    stride = (int)(gridDim.x / nx);
    lo = total * x / nx;
    hi = total * (x + 1) / nx;
  }
  // The workgroup's first tile with rows from tg on; tg advances to it. A
  // device table may hold empty tiles anywhere (a kernel-argument table does
  // not): they are stepped over. Rows 0: the list has ended.
  __device__ __forceinline__ PfTile next(int64_t& tg, const int32_t* __restrict__ t_row0,
                                         const int32_t* __restrict__ t_rows,
                                         const int32_t* __restrict__ t_group,
                                         const int32_t* __restrict__ eids, const PwTiles& tt) const {
    PfTile t{0, 0, 0, 0};
    int mt = (int)(tg / n_tiles);
    if (tt.n == 0)
      while (tg < hi && t_rows[mt] <= 0) {
        tg += stride;
        mt = (int)(tg / n_tiles);
      }
    if (tg >= hi) return t;
    t.n0 = uniform((int)(tg - (int64_t)mt * n_tiles) * width);
    if (tt.n > 0) {
      t.row0 = uniform(tt.row0[mt]);
      t.rows = uniform(tt.rows[mt]);
      t.e = uniform(tt.grp_is_expert ? tt.grp[mt] : eids[tt.grp[mt]]);
    } else {
      t.row0 = uniform(t_row0[mt]);
      t.rows = uniform(t_rows[mt]);
      t.e = uniform(eids[t_group[mt]]);
    }
    return t;
  }
};

template <int FMT>
__global__ void __launch_bounds__(512, 2)
    k_tile_fwd(const FwdArgs p, const int32_t* __restrict__ t_row0,
               const int32_t* __restrict__ t_rows, const int32_t* __restrict__ t_group,
               const int32_t* __restrict__ eids, uint16_t* __restrict__ out, const PwTiles tt) {
  __shared__ __attribute__((aligned(16))) char smem[kTlLds];
  const TileWalk tw(p, kTlBN, (int)((p.N + kTlBN - 1) / kTlBN));
  int64_t tg = tw.lo + tw.idx;
  PfTile t = tw.next(tg, t_row0, t_rows, t_group, eids, tt);
  if (t.rows <= 0) return;
  const int F = uniform((int)(p.K / kTlBK));
  TileRegs<FMT> regs;
  {
    const TileSrc<FMT> x(p, t);
    first_weights<FMT>(p, x, F, regs);
    first_stages_of<FMT>(p, x, t.rows, F, smem);
  }
  if constexpr (FMT == kNF4) init_pair_table_imm(smem);
  wait_vm_lgkm0<kFirstAfter0<FMT>>();
  __builtin_amdgcn_s_barrier();
  int slot = 0;
  while (t.rows > 0) {
    tg += tw.stride;
    const PfTile tn = tw.next(tg, t_row0, t_rows, t_group, eids, tt);
    switch ((t.rows + 31) >> 5) {
      case 8: slot = tile_fwd<FMT, 8>(p, t, tn, smem, out, regs, slot); break;
      case 7: slot = tile_fwd<FMT, 7>(p, t, tn, smem, out, regs, slot); break;
      case 6: slot = tile_fwd<FMT, 6>(p, t, tn, smem, out, regs, slot); break;
      case 5: slot = tile_fwd<FMT, 5>(p, t, tn, smem, out, regs, slot); break;
      case 4: slot = tile_fwd<FMT, 4>(p, t, tn, smem, out, regs, slot); break;
      case 3: slot = tile_fwd<FMT, 3>(p, t, tn, smem, out, regs, slot); break;
      case 2: slot = tile_fwd<FMT, 2>(p, t, tn, smem, out, regs, slot); break;
      default: slot = tile_fwd<FMT, 1>(p, t, tn, smem, out, regs, slot); break;
    }
    slot = uniform(slot);
    t = tn;
  }
  // no load may write this workgroup's LDS after it ends
  wait_vm_lgkm0<0>();
}

// ================================================================ dgrad ==
//
// k_tile_dgrad: out[t, k] = sum_n grad[t, n] W[e][n, k], tiles of up to 160
// gradient rows of one group x 512 output columns (k), the contraction over n
// in ascending steps of 64 packed rows. Eight waves, two per SIMD, of 64
// columns each: no weight is decoded twice, and one wave's lookups run while
// the other's MFMAs do. (One wave per SIMD, the 256-row kernel's form, waits
// out every LDS round trip when a tile has few rows to hide it behind.)
//   * gradient rows (two-deep) and packed rows and scales (three-deep) come
//     through LDS rings by direct-to-LDS loads: one barrier per step both
//     publishes the next step and frees the last;
//   * one ds_read_b64_tr_b8 per 16-row slice hands each lane one byte column
//     of 8 packed rows. Byte c holds k = 2 c (first nibble) and 2 c + 1, which
//     feed the MFMA blocks 0 and 1: block b, MFMA row i is the wave's column
//     2 i + b. The rows of the tr8 read come in the order 0,2,4,6,1,3,5,7, so
//     dword 0 holds the even rows, dword 1 the odd ones, and the bf16 pair
//     (row 2 m, row 2 m + 1) comes from byte m of each;
//   * slice kk looks up the next slice's weights in its first half and packs
//     them, each row by its own scale, in its second;
//   * the loads run on into the workgroup's next tile.
// The products of an output are added in the 256-row kernel's order: both
// give the same bits. 160 rows are what fits: the accumulators take 160 of a
// wave's 256 registers, the rings and the table 148 KiB of LDS.
// What bounds it: at 128 rows the MFMAs (1024 clocks per wave and step, 2048
// per SIMD) and the LDS (lookups, operand reads and stage writes, about 2400
// clocks) half hide each other, a step takes 3800-4500; at 32 rows the chain
// of lookup, pack and MFMA.
// Measured (MI355X, 32 / 64 / 128 / 160 rows per group; before: the 256-row
// kernel): NF4, 128 experts, N = 2048, K = 768: 45 / 54 / 73 / 83 us (67 / 69 /
// 89 / 92); N = 1536, K = 2048: 74 / 88 / 118 / 135 (105 / 110 / 147 / 160);
// MXFP4, 32 experts, N = 5760, K = 2880: 102 / 117 / 164 / 189 us (177 / 177 /
// 201 / 222). Two waves per 64 columns, each with every second step: 49 / 59 /
// 80 us at 32 / 64 / 128 rows of the first shape, and other bits.
// A wave loading its own 32 bytes of every row: 133 us for MXFP4 at 32 rows.
constexpr int kDtBM = kDgradWideRows;
constexpr int kDtBN = 512;
constexpr int kDtAct = kDtBM * kTlBK * 2;                   // a step's gradient rows
constexpr int kDtRows = 64 * 128;                           // half a step's packed rows
constexpr int kDtHalf = kDtRows + 2048;                     // and scales, a dword each
constexpr int kDtWts = 2 * kDtHalf;                         // 20 KiB
constexpr int kDtTab = 32 * 1024;                           // 16-column pair table
constexpr int kDtW0 = kDtTab + 2 * kDtAct;                  // weight ring, three deep
constexpr int kDtActLoads = (kDtAct / 1024 + kTlWaves - 1) / kTlWaves;
constexpr int kDtOut = kDtW0 + 3 * kDtWts;                  // per wave 16 rows x 64 columns
static_assert(kDtOut + kTlWaves * 2048 <= kTlLds, "dgrad LDS");

template <int FMT>
struct DgradSrc {
  const char* a;
  const char* b;
  const char* s;
  int rows, a_bytes, b_bytes, s_bytes;
  // columns [n0 + 256 half, +256), up to the last byte of the last row:
  // columns past K read what follows their row (never stored), and zeros
  // behind the expert's rows
  __device__ __forceinline__ DgradSrc(const FwdArgs& p, const PfTile& t, int half) {
    constexpr int kB = FMT == kNF4 ? 4 : 1, kBlk = FMT == kNF4 ? 64 : 32;
    const int k0 = t.n0 + half * 256;
    const bool live = t.rows > 0, in = live && k0 < p.K;
    const int64_t k = in ? k0 : 0;
    a = static_cast<const char*>(uniform_ptr(p.a + (int64_t)t.row0 * p.lda));
    b = static_cast<const char*>(uniform_ptr(p.B + (int64_t)t.e * p.sbe + k / 2));
    s = static_cast<const char*>(uniform_ptr(static_cast<const char*>(p.S) +
                                             ((int64_t)t.e * p.sse + k / kBlk) * kB));
    rows = t.rows;
    a_bytes = uniform(live ? (int)((int64_t)t.rows * p.lda * 2) : 0);
    b_bytes = uniform(in ? (int)((p.N - 1) * p.sbn + (p.K - k) / 2) : 0);
    s_bytes = uniform(in ? (int)(((p.N - 1) * p.ssn + (p.K - k) / kBlk) * kB) : 0);
  }
};

template <int FMT>
struct DgradLoads {
  static constexpr int kW = 2 + (FMT == kNF4 ? 1 : 2);   // weight loads per step
  int a_voff, a_piece, b_voff, s_voff, b_step, s_step, b_next, s_next;
  __device__ __forceinline__ DgradLoads(const FwdArgs& p, int wave, int lane) {
    // piece j of a wave: rows (8 j + wave) 8 + lane / 8
    const int row = wave * 8 + (lane >> 3);
    a_voff = (int)(row * p.lda * 2) + ((lane & 7) ^ pf_swz(row & 15)) * 16;
    a_piece = (int)(kTlWaves * 8 * p.lda * 2);
    // the four waves of a half share its loads, so that neighbouring lanes
    // read one row: 8 lanes its 128 packed bytes (16-byte chunk c of row r at
    // c ^ (r % 8) in LDS), 4 lanes its absmax values, 8 its e8m0 bytes
    const int w = wave & 3, l8 = lane >> 3;
    b_voff = (int)((w * 16 + l8) * p.sbn) + ((lane & 7) ^ l8) * 16;
    b_next = (int)(8 * p.sbn);
    b_step = (int)(64 * p.sbn);
    s_voff = FMT == kNF4 ? (int)((w * 16 + (lane >> 2)) * p.ssn + (lane & 3)) * 4
                         : (int)((w * 16 + l8) * p.ssn) + (lane & 7);
    s_next = (int)(8 * p.ssn);
    s_step = (int)(64 * p.ssn * (FMT == kNF4 ? 4 : 1));
  }
  // gradient piece j (of kDtActLoads) of step g (of F); zeros for a step past the end,
  // nothing for rows past the tile
  __device__ __forceinline__ void act(char* smem, const DgradSrc<FMT>& x, int wave, int g, int F,
                                      int slot, int j) const {
    if ((j * kTlWaves + wave) * 8 >= x.rows) return;
    char* dst = smem + kDtTab + slot * kDtAct + (j * kTlWaves + wave) * 1024;
    __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc_of(x.a, g < F ? x.a_bytes : 0), (lds_ptr_t)dst,
                                             16, a_voff, uniform(j * a_piece + g * (kTlBK * 2)), 0, 0);
  }
  // weight load j (0..kW - 1) of step g: packed rows, then scales
  __device__ __forceinline__ void wts(char* smem, const DgradSrc<FMT>& x, int wave, int g, int F,
                                      int slot, int j) const {
    char* w = smem + kDtW0 + slot * kDtWts + (wave >> 2) * kDtHalf;
    const int q = wave & 3;
    if (j < 2) {
      __builtin_amdgcn_raw_ptr_buffer_load_lds(
          rsrc_of(x.b, g < F ? x.b_bytes : 0), (lds_ptr_t)(w + (q * 2 + j) * 1024), 16, b_voff,
          uniform(g < F ? g * b_step + j * b_next : 0), 0, 0);
      return;
    }
    const __amdgpu_buffer_rsrc_t rs = rsrc_of(x.s, g < F ? x.s_bytes : 0);
    if constexpr (FMT == kNF4)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (lds_ptr_t)(w + kDtRows + q * 256), 4, s_voff,
                                               uniform(g < F ? g * s_step : 0), 0, 0);
    else
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (lds_ptr_t)(w + kDtRows + (q * 2 + j - 2) * 256), 1,
                                               s_voff, uniform(g < F ? g * s_step + (j - 2) * s_next : 0), 0, 0);
  }
};

// Ring positions: gradient slot 0..1, weight slot 0..2
struct DgradPos {
  int a, w;
};

// One tile. On entry its step 0 is at `at`, landed and published, and the
// weights of its step 1 are on their way. Returns where tn's step 0 is, in
// the same state.
template <int FMT, int kM>
__device__ __forceinline__ DgradPos tile_dgrad(const FwdArgs& p, const PfTile t, const PfTile tn,
                                          char* smem, uint16_t* __restrict__ out, const DgradPos at) {
  const int lane = opaque(threadIdx.x) & 63, wave = uniform(threadIdx.x >> 6);
  const int l32 = lane & 31, h = lane >> 5;
  const int half = wave >> 2, w = wave & 3;
  const int F = uniform((int)(p.N / kTlBK));
  using L = DgradLoads<FMT>;
  const DgradSrc<FMT> x(p, t, half), xn(p, tn, half);
  const L ld(p, wave, lane);

  const unsigned lds0 = (unsigned)(uintptr_t)(lds_ptr_t)smem;
  const int a_off = kDtTab + l32 * 128 + ((4 * h) ^ pf_swz(l32 & 15)) * 16;
  auto act_addr = [&](int slot, int kk) {
    unsigned addr = lds0 + slot * kDtAct + (a_off ^ (kk * 16));
    asm("" : "+v"(addr));
    return addr;
  };
  // the tr8 read of slice kk: lane i of its 16-lane group supplies 8 bytes of
  // row pi(i / 2), half i % 2 of the group's 16
  const int w_off = kDtW0 + half * kDtHalf;
  const int tr_row = ((lane >> 1) & 3) * 2 + ((lane >> 3) & 1);
  const int tr_off = w_off + (32 * h + tr_row) * 128 +
                     ((w * 2 + ((lane >> 4) & 1)) ^ tr_row) * 16 + (lane & 1) * 8;
  // the scales of row 32 h (MXFP4: of the lane's 32-column block)
  constexpr int kSRow = FMT == kNF4 ? 16 : 32;
  const int s_off = w_off + kDtRows + 32 * h * kSRow +
                    (FMT == kNF4 ? w : w * 2 + (l32 >> 4)) * 4;
  // pair-table address << 1 | column * 16 (nf4_dword_to_bf16_t16's form)
  const unsigned reg2 = (unsigned)(lane & 15) * 16u;

  unsigned pw[2][4];      // packed dwords of a step's slices
  auto read_w = [&](int slot) {
    typedef __attribute__((address_space(3))) v2i32_t lds_v2i32;
#pragma unroll
    for (int kk = 0; kk < 4; ++kk) {
      const v2i32_t r = __builtin_amdgcn_ds_read_tr8_b64_v2i32(
          (lds_v2i32*)(lds_ptr_t)(smem + slot * kDtWts + tr_off + kk * 8 * 128));
      pw[0][kk] = (unsigned)r.x;
      pw[1][kk] = (unsigned)r.y;
    }
  };
  u32x4_t wf[2][2];       // [slice parity][block]
  f32x2_t tp[2][4];       // NF4: looked-up pairs of the target
  unsigned tw[2];         // MXFP4: its dwords
  unsigned ts[8];         // its rows' scales, as read
  // half m2 (bytes 2 m2, 2 m2 + 1) of the target (slot, slice kk)
  auto look = [&](int slot, int kk, int m2) {
    if (m2 == 0) {
      typedef __attribute__((address_space(3))) unsigned lds_u32;
      lds_u32* sp = (lds_u32*)(lds_ptr_t)(smem + slot * kDtWts + s_off + kk * 8 * kSRow);
#pragma unroll
      for (int r = 0; r < 8; ++r) ts[r] = sp[r * kSRow / 4];
      if constexpr (FMT != kNF4) {
        tw[0] = pw[0][kk];
        tw[1] = pw[1][kk];
      }
    }
    if constexpr (FMT == kNF4)
#pragma unroll
      for (int d = 0; d < 2; ++d)
#pragma unroll
        for (int m = 2 * m2; m < 2 * m2 + 2; ++m)
          tp[d][m] = lds_read8f(
              __builtin_amdgcn_perm(pw[d][kk], reg2, 0x0C0C0000u | ((4u + m) << 8)) >> 1);
  };
  auto scale = [&](int r) -> float {
    const unsigned v = ts[r];
    if constexpr (FMT == kNF4) return __uint_as_float(v);
    else return e8m0_to_f32(v & 0xFFu);
  };
  auto pack = [&](int par, int m2) {
#pragma unroll
    for (int m = 2 * m2; m < 2 * m2 + 2; ++m) {
      const float s0 = scale(2 * m), s1 = scale(2 * m + 1);
      if constexpr (FMT == kNF4) {
        wf[par][0][m] = bf16x2_bits(tp[0][m].x * s0, tp[1][m].x * s1);
        wf[par][1][m] = bf16x2_bits(tp[0][m].y * s0, tp[1][m].y * s1);
      } else {
        auto cvt = [&](unsigned v, float sc) {
          bf16x2_t r;
          if (m == 0) r = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(v, sc, 0);
          else if (m == 1) r = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(v, sc, 1);
          else if (m == 2) r = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(v, sc, 2);
          else r = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(v, sc, 3);
          return __builtin_bit_cast(unsigned, r);
        };
        const unsigned c0 = cvt(tw[0], s0), c1 = cvt(tw[1], s1);
        wf[par][0][m] = __builtin_amdgcn_perm(c1, c0, 0x05040100u);
        wf[par][1][m] = __builtin_amdgcn_perm(c1, c0, 0x07060302u);
      }
    }
  };

  // ---- prologue: gradients of step 1, weights of step 2 (of the next tile's
  // step 0 where this one has two), and slice 0 of step 0
  int sa = at.a, sw = at.w;
  auto next_w = [](int v) { return v == 2 ? 0 : v + 1; };
  {
    const int w2 = next_w(next_w(sw));
    const bool cur = F != 2;
    const DgradSrc<FMT>& y = cur ? x : xn;
#pragma unroll
    for (int j = 0; j < kDtActLoads; ++j) ld.act(smem, x, wave, 1, F, sa ^ 1, j);
#pragma unroll
    for (int j = 0; j < L::kW; ++j) ld.wts(smem, y, wave, uniform(cur ? 2 : 0), F, w2, j);
  }
  read_w(sw);
  look(sw, 0, 0);
  look(sw, 0, 1);
  pack(0, 0);
  pack(0, 1);
  u32x4_t av[kM];
#pragma unroll
  for (int i = 0; i < kM; ++i) av[i] = lds_read16(act_addr(sa, 0) + i * 4096);
  f32x16_t acc[2][kM];
#pragma unroll
  for (int b = 0; b < 2; ++b)
#pragma unroll
    for (int i = 0; i < kM; ++i) acc[b][i] = f32x16_t{};

  for (int f = 0; f < F; ++f) {
    const bool last = f + 1 >= F;
    auto slice = [&](auto KI) {
      constexpr int kk = decltype(KI)::value;
      __builtin_amdgcn_sched_barrier(0);
      if constexpr (kk == 3) {
        // step f + 1 has landed (newer: the weights of step f + 2), and every
        // wave has read all of step f's slots
        wait_vm_lgkm0<L::kW>();
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_sched_barrier(0);
        read_w(next_w(sw));
      }
      const int ts_slot = kk == 3 ? next_w(sw) : sw;
      const unsigned src = act_addr(kk == 3 ? sa ^ 1 : sa, (kk + 1) & 3);
      constexpr int n = 2 * kM;
#pragma unroll
      for (int i = 0; i < kM; ++i)
#pragma unroll
        for (int b = 0; b < 2; ++b) {
          acc[b][i] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
              as_bf16x8(wf[kk & 1][b]), as_bf16x8(av[i]), acc[b][i], 0, 0, 0);
          const int pos = 2 * i + b;
          if (b == 1) av[i] = lds_read16(src + i * 4096);
          // the gradients of step f + 2, then the weights of step f + 3 (past
          // the end: the next tile's step 0, steps 0 and 1), into the slots
          // that the barrier freed
          if constexpr (kk == 3) {
            if (!last) {
              constexpr int kAct = kDtActLoads, kAll = kAct + L::kW;
#pragma unroll
              for (int j = 0; j < kAll; ++j) {
                if ((j * n) / kAll != pos) continue;
                const int g = f + (j < kAct ? 2 : 3);
                const bool cur = g < F;
                const DgradSrc<FMT>& y = cur ? x : xn;
                if (j < kAct) ld.act(smem, y, wave, uniform(cur ? g : g - F), F, sa, j);
                else ld.wts(smem, y, wave, uniform(cur ? g : g - F), F, sw, j - kAct);
              }
            }
          }
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            if ((q * n) / 4 != pos) continue;
            if (q < 2) look(ts_slot, (kk + 1) & 3, q);
            else pack((kk + 1) & 1, q - 2);
          }
          __builtin_amdgcn_sched_barrier(0);
        }
    };
    slice(std::integral_constant<int, 0>{});
    slice(std::integral_constant<int, 1>{});
    slice(std::integral_constant<int, 2>{});
    slice(std::integral_constant<int, 3>{});
    sa ^= 1;
    sw = next_w(sw);
  }
  // ---- epilogue. sa and sw (of step F) hold the next tile's step 0, landed
  // and published, unless the tile had a single step. Each wave turns its own
  // 32 x 64 subtiles through its own LDS, and stores whole 128-byte pieces.
  __builtin_amdgcn_sched_barrier(0);
  if (F == 1) {
#pragma unroll
    for (int j = 0; j < kDtActLoads; ++j) ld.act(smem, xn, wave, 0, F, sa, j);
#pragma unroll
    for (int g = 0; g < 2; ++g)
#pragma unroll
      for (int j = 0; j < L::kW; ++j) ld.wts(smem, xn, wave, g, F, g ? next_w(sw) : sw, j);
  }
  char* ob = smem + kDtOut + wave * 2048;
  const __amdgpu_buffer_rsrc_t ro = __builtin_amdgcn_make_buffer_rsrc(
      uniform_ptr(out + (int64_t)t.row0 * p.ldo), 0, uniform((int)((int64_t)t.rows * p.ldo * 2)),
      0x00020000);
  const int ldo2 = (int)(p.ldo * 2);
  const int col = t.n0 + wave * 64 + (lane & 7) * 8;
  const int coff = col < p.K ? col * 2 + (lane >> 3) * ldo2 : kOOB;   // K % 64 == 0
#pragma unroll
  for (int i = 0; i < kM; ++i) {
    // MFMA row 8 g + 4 h + q of block b is column 16 g + 8 h + 2 q + b
    u32x4_t v[4];
#pragma unroll
    for (int g = 0; g < 4; ++g)
#pragma unroll
      for (int q = 0; q < 4; ++q) v[g][q] = bf16x2_bits(acc[0][i][4 * g + q], acc[1][i][4 * g + q]);
#pragma unroll
    for (int r16 = 0; r16 < 2; ++r16) {
      if ((l32 >> 4) == r16)
#pragma unroll
        for (int g = 0; g < 4; ++g)
          *reinterpret_cast<u32x4_t*>(ob + (l32 & 15) * 128 + (((2 * g + h) ^ (l32 & 7)) << 4)) =
              v[g];
      wave_lds_fence();
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        const int row = j * 8 + (lane >> 3);
        const u32x4_t o =
            *reinterpret_cast<const u32x4_t*>(ob + row * 128 + (((lane & 7) ^ (row & 7)) << 4));
        store_b128(o, ro, coff + (i * 32 + r16 * 16 + j * 8) * ldo2);
      }
      wave_lds_fence();
    }
  }
  if (F == 1) {
    wait_vm_lgkm0<0>();
    __builtin_amdgcn_s_barrier();
  }
  return {sa, sw};
}

template <int FMT>
__global__ void __launch_bounds__(512, 2)
    k_tile_dgrad(const FwdArgs p, const int32_t* __restrict__ t_row0,
                 const int32_t* __restrict__ t_rows, const int32_t* __restrict__ t_group,
                 const int32_t* __restrict__ eids, uint16_t* __restrict__ out, const PwTiles tt) {
  __shared__ __attribute__((aligned(16))) char smem[kTlLds];
  const TileWalk tw(p, kDtBN, (int)((p.K + kDtBN - 1) / kDtBN));
  int64_t tg = tw.lo + tw.idx;
  PfTile t = tw.next(tg, t_row0, t_rows, t_group, eids, tt);
  if (t.rows <= 0) return;
  {
    const int lane = opaque(threadIdx.x) & 63, wave = uniform(threadIdx.x >> 6);
    const DgradSrc<FMT> x(p, t, wave >> 2);
    const DgradLoads<FMT> ld(p, wave, lane);
    const int F = uniform((int)(p.N / kTlBK));
#pragma unroll
    for (int j = 0; j < kDtActLoads; ++j) ld.act(smem, x, wave, 0, F, 0, j);
#pragma unroll
    for (int g = 0; g < 2; ++g)
#pragma unroll
      for (int j = 0; j < DgradLoads<FMT>::kW; ++j) ld.wts(smem, x, wave, g, F, g, j);
  }
  if constexpr (FMT == kNF4) init_pair_table16_imm(smem);
  wait_vm_lgkm0<0>();
  __builtin_amdgcn_s_barrier();
  DgradPos at{0, 0};
  while (t.rows > 0) {
    tg += tw.stride;
    const PfTile tn = tw.next(tg, t_row0, t_rows, t_group, eids, tt);
    switch ((t.rows + 31) >> 5) {
      case 5: at = tile_dgrad<FMT, 5>(p, t, tn, smem, out, at); break;
      case 4: at = tile_dgrad<FMT, 4>(p, t, tn, smem, out, at); break;
      case 3: at = tile_dgrad<FMT, 3>(p, t, tn, smem, out, at); break;
      case 2: at = tile_dgrad<FMT, 2>(p, t, tn, smem, out, at); break;
      default: at = tile_dgrad<FMT, 1>(p, t, tn, smem, out, at); break;
    }
    at.a = uniform(at.a);
    at.w = uniform(at.w);
    t = tn;
  }
  // no load may write this workgroup's LDS after it ends
  wait_vm_lgkm0<0>();
}

}  // namespace

namespace gnf4 {

int launch_tile_fwd(int fmt, const FwdArgs& p, const PwTiles& tt, int64_t per_x,
                    hipStream_t stream) {
  const dim3 grid((unsigned)(per_x * 8)), block(64 * kTlWaves);
  if (fmt == kNF4)
    hipLaunchKernelGGL((k_tile_fwd<kNF4>), grid, block, 0, stream, p, p.t_row0, p.t_rows,
                       p.t_group, p.eids, p.out, tt);
  else
    hipLaunchKernelGGL((k_tile_fwd<kMX>), grid, block, 0, stream, p, p.t_row0, p.t_rows,
                       p.t_group, p.eids, p.out, tt);
  return hipGetLastError() == hipSuccess ? 0 : -2;
}

int launch_tile_dgrad(int fmt, const FwdArgs& p, uint16_t* out, const PwTiles& tt, int64_t per_x,
                      hipStream_t stream) {
  const dim3 grid((unsigned)(per_x * 8)), block(64 * kTlWaves);
  if (fmt == kNF4)
    hipLaunchKernelGGL((k_tile_dgrad<kNF4>), grid, block, 0, stream, p, p.t_row0, p.t_rows,
                       p.t_group, p.eids, out, tt);
  else
    hipLaunchKernelGGL((k_tile_dgrad<kMX>), grid, block, 0, stream, p, p.t_row0, p.t_rows,
                       p.t_group, p.eids, out, tt);
  return hipGetLastError() == hipSuccess ? 0 : -2;
}

}  // namespace gnf4
