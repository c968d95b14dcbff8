// gnf4_lora.hip -- the low-rank (LoRA) half of a fine-tuned grouped projection
// on gfx950, over ragged groups, in fp32:
//
//   forward    u = x A[e]^T,  out = base + bf16(s u B[e]^T)
//   backward   gu = s g B[e],  gx = gu A[e],  gA[e] = gu^T x,  gB[e] = s g^T u
//
// x, g, base, out bf16; A [E, r, K], B [E, N, r], u and gu [T, r], gA and gB
// fp32; r % 4 == 0 and r <= 64. Three kernels serve the six products; each
// reads its rows where they lie, in 16-row tiles of one group, so nothing
// is gathered or padded to the widest group.
//
// All of them use v_mfma_f32_16x16x4_f32 (fp32 operands and sums). What they
// contract is small (2 T K r flops); they are bound by reading and writing the
// bf16 rows once. The lanes' k, row and column assignments are chosen so that
// each lane's global accesses are 16 contiguous bytes.
//
// Measured (MI355X, 8192 rows, 128 experts, K = 2048, N = 1536, r = 16): u
// and gu 23 and 18 us (34 and 25 MB of rows: 1.4 TB/s, from the latency of few
// loads per wave), out and gx 24 us each (50 and 34 MB, 2.1 and 1.4 TB/s), gA
// and gB 17 and 14 us (2.0 and 1.8 TB/s). With gathers, padding to the widest
// group, batched fp32 products and index scatters the same parts took about
// 900 us; the whole training pass through the projection went from 1151 to
// 524 us (358 us of kernels, 26 of them the copies its backward reads).

#include "gnf4_device.h"

using namespace gnf4;

namespace {

__device__ __forceinline__ f32x4_t mfma4(float a, float b, f32x4_t c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

__device__ __forceinline__ float bf16_lo(unsigned w) { return __uint_as_float(w << 16); }
__device__ __forceinline__ float bf16_hi(unsigned w) { return __uint_as_float(w & 0xFFFF0000u); }
__device__ __forceinline__ float bf16_elem(u32x4_t v, int i) {
  return i & 1 ? bf16_hi(v[i >> 1]) : bf16_lo(v[i >> 1]);
}

struct LoraGroups {
  const int32_t* tile_off;   // [G + 1] tiles before a group
  const int32_t* row_off;    // [G + 1] rows before it
  const int32_t* ids;        // [G] its expert
  int G;
};

// Tile b of the groups' tiles of kRows rows: one pass over the groups' tile
// ends, 64 at a time.
template <int kRows>
struct LoraTile {
  int row0, rows;
  int64_t e;
  __device__ __forceinline__ LoraTile(const LoraGroups& t, int b) {
    const int lane = threadIdx.x & 63;
    int g = 0;
    for (int c = 0; c < t.G; c += 64) {
      const int end = c + lane < t.G ? t.tile_off[c + lane + 1] : 0x7FFFFFFF;
      g += __popcll(__ballot(end <= b));
    }
    g = uniform(g);
    row0 = t.row_off[g] + kRows * (b - t.tile_off[g]);
    const int left = t.row_off[g + 1] - row0;
    rows = left < kRows ? left : kRows;
    e = t.ids[g];
  }
};

// Y[t, j] = s sum_c X[t, c] M(c, j): M = A[e]^T ([r, C] rows) or, kT, B[e]
// ([C, r] rows). One 16-row tile per workgroup; its four waves take every
// fourth 32-wide chunk of C. Lane (m, q): row m (X) and column m (M) of a
// 16 x 16 block, c [32 chunk + 8 q, +8), one c per MFMA.
template <int RB, bool kT>
__global__ void __launch_bounds__(256) k_lora_down(const uint16_t* __restrict__ X, int64_t ldx,
                                                   const float* __restrict__ M, int64_t C, int r,
                                                   int64_t E, const LoraGroups gr, float s,
                                                   float* __restrict__ Y) {
  __shared__ f32x4_t red[4][RB][64];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int m = lane & 15, q = lane >> 4;
  const LoraTile<16> t(gr, blockIdx.x);
  const int row0 = t.row0, rows = t.rows;
  const int64_t e = t.e;
  const bool known = e >= 0 && e < E;
  f32x4_t acc[RB];
#pragma unroll
  for (int b = 0; b < RB; ++b) acc[b] = f32x4_t{};
  const uint16_t* xr = X + (int64_t)(row0 + (m < rows ? m : 0)) * ldx;
  const float* me = M + (known ? e : 0) * C * r;
  if (known) {
    // two chunks' loads at a time
    for (int64_t c0 = wave * 32; c0 < C; c0 += 256) {
      u32x4_t xv[2];
      float w[2][RB][8];
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        const int64_t c = c0 + 128 * u + 8 * q;
        const bool in = c < C;   // C % 8 == 0: all eight or none
        xv[u] = in && m < rows ? load_a8(xr + c) : u32x4_t{};
#pragma unroll
        for (int b = 0; b < RB; ++b) {
          const int j = 16 * b + m;
          const bool ok = in && j < r;
          if constexpr (kT) {
#pragma unroll
            for (int i = 0; i < 8; ++i) w[u][b][i] = ok ? me[(c + i) * r + j] : 0.f;
          } else {
            const f32x4_t z{};
            const f32x4_t* src = reinterpret_cast<const f32x4_t*>(me + (int64_t)j * C + c);
            const f32x4_t w0 = ok ? src[0] : z, w1 = ok ? src[1] : z;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
              w[u][b][i] = w0[i];
              w[u][b][4 + i] = w1[i];
            }
          }
        }
      }
#pragma unroll
      for (int u = 0; u < 2; ++u)
#pragma unroll
        for (int i = 0; i < 8; ++i)
#pragma unroll
          for (int b = 0; b < RB; ++b) acc[b] = mfma4(bf16_elem(xv[u], i), w[u][b][i], acc[b]);
    }
  }
#pragma unroll
  for (int b = 0; b < RB; ++b) red[wave][b][lane] = acc[b];
  __syncthreads();
  for (int b = wave; b < RB; b += 4) {
    const f32x4_t v = (red[0][b][lane] + red[1][b][lane]) + (red[2][b][lane] + red[3][b][lane]);
    const int j = 16 * b + m;
    if (j < r)
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if (4 * q + i < rows) Y[(int64_t)(row0 + 4 * q + i) * r + j] = s * v[i];
  }
}

// out[t, n] = (base[t, n] +) bf16(s sum_j U[t, j] M(n, j)): M = B[e] ([C, r]
// rows) or, kT, A[e]^T ([r, C] rows); C columns. A wave: 16 rows x 64 columns;
// MFMA row m of block b is column 16 (m / 4) + 4 b + m % 4, so lane (t, q)
// ends with the 16 consecutive columns 16 q of row t.
template <int RB, bool kT, bool kBase>
__global__ void __launch_bounds__(256) k_lora_up(const float* __restrict__ U,
                                                 const float* __restrict__ M, int64_t C, int r,
                                                 int64_t E, const LoraGroups gr, float s,
                                                 const uint16_t* __restrict__ base, int64_t ldb,
                                                 uint16_t* __restrict__ out, int64_t ldo) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int m = lane & 15, q = lane >> 4;
  const LoraTile<16> t(gr, blockIdx.x);
  const int row0 = t.row0, rows = t.rows;
  const int64_t e = t.e;
  const bool known = e >= 0 && e < E;
  const int64_t n0 = ((int64_t)blockIdx.y * 4 + wave) * 64;
  if (n0 >= C) return;
  const float* me = M + (known ? e : 0) * C * r;
  const f32x4_t z{};
  f32x4_t acc[4];
#pragma unroll
  for (int b = 0; b < 4; ++b) acc[b] = z;
#pragma unroll
  for (int rb = 0; rb < RB; ++rb) {
    const int j = 16 * rb + 4 * q;
    const bool jn = known && j < r;   // r % 4 == 0: all four or none
    const f32x4_t uv = jn && m < rows
                           ? *reinterpret_cast<const f32x4_t*>(U + (int64_t)(row0 + m) * r + j) : z;
#pragma unroll
    for (int b = 0; b < 4; ++b) {
      const int64_t n = n0 + 16 * (m >> 2) + 4 * b + (m & 3);
      f32x4_t w = z;
      if (jn && n < C) {
        if constexpr (kT) {
#pragma unroll
          for (int i = 0; i < 4; ++i) w[i] = me[(int64_t)(j + i) * C + n];
        } else {
          w = *reinterpret_cast<const f32x4_t*>(me + n * r + j);
        }
      }
#pragma unroll
      for (int i = 0; i < 4; ++i) acc[b] = mfma4(w[i], uv[i], acc[b]);
    }
  }
  if (m >= rows) return;
  const int64_t n = n0 + 16 * q;
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    if (n + 8 * h >= C) break;   // C % 8 == 0
    u32x4_t v;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const f32x4_t a = acc[2 * h + (i >> 1)];
      v[i] = bf16x2_bits(s * a[(i & 1) * 2], s * a[(i & 1) * 2 + 1]);
    }
    if constexpr (kBase) {
      const u32x4_t bv = load_a8(base + (int64_t)(row0 + m) * ldb + n + 8 * h);
#pragma unroll
      for (int i = 0; i < 4; ++i)
        v[i] = bf16x2_bits(bf16_lo(bv[i]) + bf16_lo(v[i]), bf16_hi(bv[i]) + bf16_hi(v[i]));
    }
    *reinterpret_cast<u32x4_t*>(out + (int64_t)(row0 + m) * ldo + n + 8 * h) = v;
  }
}

// Weight gradients: s sum over rows of P[t, :] Q[t, :], a [C, r] matrix or,
// kT, [r, C]. A wave: 128 columns of P, all r; MFMA row m of block i is column
// 8 m + i, contraction over four rows t (lane quarter q).
template <int RB>
struct WgradAcc {
  f32x4_t acc[8][RB];
  __device__ __forceinline__ WgradAcc() {
#pragma unroll
    for (int i = 0; i < 8; ++i)
#pragma unroll
      for (int b = 0; b < RB; ++b) acc[i][b] = f32x4_t{};
  }
  // adds rows [begin, end); 16 rows' loads at a time
  __device__ __forceinline__ void add(const uint16_t* __restrict__ P, int64_t ldp,
                                      const float* __restrict__ Q, int64_t C, int64_t c, int r,
                                      int begin, int end, int m, int q) {
    for (int t0 = begin; t0 < end; t0 += 16) {
      u32x4_t pv[4];
      float w[4][RB];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int t = t0 + 4 * u + q;
        const bool in = t < end;
        pv[u] = in && c < C ? load_a8(P + (int64_t)t * ldp + c) : u32x4_t{};
#pragma unroll
        for (int b = 0; b < RB; ++b)
          w[u][b] = in && 16 * b + m < r ? Q[(int64_t)t * r + 16 * b + m] : 0.f;
      }
#pragma unroll
      for (int u = 0; u < 4; ++u)
#pragma unroll
        for (int i = 0; i < 8; ++i)
#pragma unroll
          for (int b = 0; b < RB; ++b)
            acc[i][b] = mfma4(bf16_elem(pv[u], i), w[u][b], acc[i][b]);
    }
  }
  template <bool kT>
  __device__ __forceinline__ void store(float* me, int64_t C, int64_t c0, int r, float s, int m,
                                        int q) const {
#pragma unroll
    for (int b = 0; b < RB; ++b) {
      const int j = 16 * b + m;
      if (j >= r) continue;
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const int64_t n = c0 + 8 * (4 * q + k);
        if (n >= C) continue;   // C % 8 == 0
        if constexpr (kT) {
          f32x4_t v0, v1;
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            v0[i] = s * acc[i][b][k];
            v1[i] = s * acc[4 + i][b][k];
          }
          f32x4_t* dst = reinterpret_cast<f32x4_t*>(me + (int64_t)j * C + n);
          dst[0] = v0;
          dst[1] = v1;
        } else {
#pragma unroll
          for (int i = 0; i < 8; ++i) me[(n + i) * r + j] = s * acc[i][b][k];
        }
      }
    }
  }
};

// Calls fn(g) for the groups g of expert e, in order.
template <class Fn>
__device__ __forceinline__ void for_groups_of(int e, const int32_t* __restrict__ ids, int G,
                                              Fn&& fn) {
  const int lane = threadIdx.x & 63;
  for (int g0 = 0; g0 < G; g0 += 64) {
    const int mine = g0 + lane < G ? ids[g0 + lane] : -1;
    uint64_t hit = __ballot(mine == e);
    while (hit) {
      fn(g0 + __ffsll((unsigned long long)hit) - 1);
      hit &= hit - 1;
    }
  }
}

// One wave per expert and 128 columns: dM[e] over all of the expert's rows.
// Every expert of the stack is written (zeros where no group has it); groups
// of one expert are added in group order.
template <int RB, bool kT>
__global__ void __launch_bounds__(256) k_lora_wgrad(const uint16_t* __restrict__ P, int64_t ldp,
                                                    const float* __restrict__ Q, int64_t C, int r,
                                                    const int32_t* __restrict__ ids,
                                                    const int32_t* __restrict__ row_off, int G,
                                                    float s, float* __restrict__ dM) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int m = lane & 15, q = lane >> 4;
  const int e = blockIdx.y;
  const int64_t c0 = ((int64_t)blockIdx.x * 4 + wave) * 128;
  if (c0 >= C) return;
  WgradAcc<RB> acc;
  for_groups_of(e, ids, G, [&](int g) {
    acc.add(P, ldp, Q, C, c0 + 8 * m, r, row_off[g], row_off[g + 1], m, q);
  });
  acc.template store<kT>(dM + (int64_t)e * C * r, C, c0, r, s, m, q);
}

// The same in two launches for experts of many rows: one wave per 256-row
// chunk of a group and 128 columns writes the chunk's sum to part[chunk], and
// k_lora_wgrad_sum adds an expert's chunks in order. A wave needs about 1.3
// (r = 16) to 2.8 us (r = 64) for 16 rows, one after the other, so with a wave
// per expert the largest expert decides: one of 8192 rows, C = 2048, r = 16 /
// 64: 650 / 1416 us in k_lora_wgrad, 35 / 66 us here; 8 experts of 512 rows 38
// / 90 and 24 / 55 us. It is bound by MFMA latency below a round of waves,
// then by the partial sums' traffic (128 experts of 512 rows: 73 / 228 us in
// k_lora_wgrad, 79 / 285 us here).
constexpr int kWgradChunk = 256;

template <int RB, bool kT>
__global__ void __launch_bounds__(256) k_lora_wgrad_part(const uint16_t* __restrict__ P,
                                                         int64_t ldp, const float* __restrict__ Q,
                                                         int64_t C, int r, const LoraGroups gr,
                                                         float s, float* __restrict__ part) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int m = lane & 15, q = lane >> 4;
  const int chunk = blockIdx.x;
  const LoraTile<kWgradChunk> t(gr, chunk);
  const int64_t c0 = ((int64_t)blockIdx.y * 4 + wave) * 128;
  if (c0 >= C) return;
  WgradAcc<RB> acc;
  acc.add(P, ldp, Q, C, c0 + 8 * m, r, t.row0, t.row0 + t.rows, m, q);
  acc.template store<kT>(part + (int64_t)chunk * C * r, C, c0, r, s, m, q);
}

__global__ void __launch_bounds__(256) k_lora_wgrad_sum(const float* __restrict__ part,
                                                        int64_t n, const LoraGroups gr,
                                                        float* __restrict__ dM) {
  const int e = blockIdx.y;
  const int64_t i = ((int64_t)blockIdx.x * 256 + threadIdx.x) * 4;   // n % 4 == 0
  f32x4_t sum{};
  for_groups_of(e, gr.ids, gr.G, [&](int g) {
    if (i < n)
      for (int64_t k = gr.tile_off[g]; k < gr.tile_off[g + 1]; ++k)
        sum += *reinterpret_cast<const f32x4_t*>(part + k * n + i);
  });
  if (i < n) *reinterpret_cast<f32x4_t*>(dM + (int64_t)e * n + i) = sum;
}

template <class Fn>
int by_rank(int r, Fn&& fn) {
  switch ((r + 15) / 16) {
    case 1: fn(std::integral_constant<int, 1>{}); break;
    case 2: fn(std::integral_constant<int, 2>{}); break;
    case 3: fn(std::integral_constant<int, 3>{}); break;
    default: fn(std::integral_constant<int, 4>{}); break;
  }
  return hipGetLastError() == hipSuccess ? 0 : -2;
}

bool rank_ok(int r) { return r >= 4 && r <= 64 && r % 4 == 0; }
bool al16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; }

}  // namespace

extern "C" {

int gnf4_hip_lora_down(const void* x, int64_t ldx, const float* w, int transposed, int64_t E,
                       int64_t C, int r, const int32_t* tile_off, const int32_t* row_off,
                       const int32_t* expert_ids, int G, int n_tiles, float scale, float* y, void* stream) {
  if (n_tiles < 0 || E <= 0 || C <= 0 || C % 8 || !rank_ok(r) || ldx < C || ldx % 8) return -1;
  if (n_tiles == 0) return 0;
  if (!x || !w || !y || !tile_off || !row_off || !expert_ids || G <= 0 || !al16(x) ||
      !al16(w))
    return -1;
  const LoraGroups gr{tile_off, row_off, expert_ids, G};
  hipStream_t s = static_cast<hipStream_t>(stream);
  return by_rank(r, [&](auto RB) {
    constexpr int rb = decltype(RB)::value;
    if (transposed)
      hipLaunchKernelGGL((k_lora_down<rb, true>), dim3((unsigned)n_tiles), dim3(256), 0, s,
                         static_cast<const uint16_t*>(x), ldx, w, C, r, E, gr, scale, y);
    else
      hipLaunchKernelGGL((k_lora_down<rb, false>), dim3((unsigned)n_tiles), dim3(256), 0, s,
                         static_cast<const uint16_t*>(x), ldx, w, C, r, E, gr, scale, y);
  });
}

int gnf4_hip_lora_up(const float* u, const float* w, int transposed, int64_t E, int64_t C, int r,
                     const int32_t* tile_off, const int32_t* row_off, const int32_t* expert_ids,
                     int G, int n_tiles, float scale, const void* base, int64_t ldb, void* out, int64_t ldo,
                     void* stream) {
  if (n_tiles < 0 || E <= 0 || C <= 0 || C % 8 || !rank_ok(r) || ldo < C || ldo % 8) return -1;
  if (base && (ldb < C || ldb % 8 || !al16(base))) return -1;
  if (n_tiles == 0) return 0;
  if (!u || !w || !out || !tile_off || !row_off || !expert_ids || G <= 0 || !al16(u) ||
      !al16(w) || !al16(out))
    return -1;
  const int64_t gy = (C + 255) / 256;
  if (gy > 65535) return -1;
  const LoraGroups gr{tile_off, row_off, expert_ids, G};
  hipStream_t s = static_cast<hipStream_t>(stream);
  const dim3 grid((unsigned)n_tiles, (unsigned)gy);
  const uint16_t* b = static_cast<const uint16_t*>(base);
  uint16_t* o = static_cast<uint16_t*>(out);
  return by_rank(r, [&](auto RB) {
    constexpr int rb = decltype(RB)::value;
    if (transposed && b)
      hipLaunchKernelGGL((k_lora_up<rb, true, true>), grid, dim3(256), 0, s, u, w, C, r, E, gr, scale, b, ldb, o, ldo);
    else if (transposed)
      hipLaunchKernelGGL((k_lora_up<rb, true, false>), grid, dim3(256), 0, s, u, w, C, r, E, gr, scale, b, ldb, o, ldo);
    else if (b)
      hipLaunchKernelGGL((k_lora_up<rb, false, true>), grid, dim3(256), 0, s, u, w, C, r, E, gr, scale, b, ldb, o, ldo);
    else
      hipLaunchKernelGGL((k_lora_up<rb, false, false>), grid, dim3(256), 0, s, u, w, C, r, E, gr, scale, b, ldb, o, ldo);
  });
}

int gnf4_hip_lora_wgrad(const void* p, int64_t ldp, const float* q, int transposed, int64_t E,
                        int64_t C, int r, const int32_t* expert_ids, const int32_t* row_off,
                        int G, float scale, float* dw, void* stream) {
  if (G < 0 || E <= 0 || E > 65535 || C <= 0 || C % 8 || !rank_ok(r) || ldp < C || ldp % 8)
    return -1;
  if (!dw || !al16(dw) || (G > 0 && (!p || !q || !expert_ids || !row_off || !al16(p)))) return -1;
  const int64_t gx = (C + 511) / 512;
  if (gx > 0x7FFFFFFF) return -1;
  hipStream_t s = static_cast<hipStream_t>(stream);
  const dim3 grid((unsigned)gx, (unsigned)E);
  return by_rank(r, [&](auto RB) {
    constexpr int rb = decltype(RB)::value;
    if (transposed)
      hipLaunchKernelGGL((k_lora_wgrad<rb, true>), grid, dim3(256), 0, s,
                         static_cast<const uint16_t*>(p), ldp, q, C, r, expert_ids, row_off, G, scale, dw);
    else
      hipLaunchKernelGGL((k_lora_wgrad<rb, false>), grid, dim3(256), 0, s,
                         static_cast<const uint16_t*>(p), ldp, q, C, r, expert_ids, row_off, G, scale, dw);
  });
}

int gnf4_hip_lora_wgrad_split(const void* p, int64_t ldp, const float* q, int transposed,
                              int64_t E, int64_t C, int r, const int32_t* chunk_off,
                              const int32_t* row_off, const int32_t* expert_ids, int G,
                              int n_chunks, float scale, float* part, float* dw, void* stream) {
  if (G <= 0 || n_chunks <= 0 || E <= 0 || E > 65535 || C <= 0 || C % 8 || !rank_ok(r) ||
      ldp < C || ldp % 8)
    return -1;
  if (!p || !q || !chunk_off || !row_off || !expert_ids || !part || !dw || !al16(p) ||
      !al16(part) || !al16(dw))
    return -1;
  const int64_t gy = (C + 511) / 512, n = C * r, gx = (n / 4 + 255) / 256;
  if (gy > 65535 || gx > 0x7FFFFFFF) return -1;
  const LoraGroups gr{chunk_off, row_off, expert_ids, G};
  hipStream_t s = static_cast<hipStream_t>(stream);
  const dim3 grid((unsigned)n_chunks, (unsigned)gy);
  return by_rank(r, [&](auto RB) {
    constexpr int rb = decltype(RB)::value;
    if (transposed)
      hipLaunchKernelGGL((k_lora_wgrad_part<rb, true>), grid, dim3(256), 0, s,
                         static_cast<const uint16_t*>(p), ldp, q, C, r, gr, scale, part);
    else
      hipLaunchKernelGGL((k_lora_wgrad_part<rb, false>), grid, dim3(256), 0, s,
                         static_cast<const uint16_t*>(p), ldp, q, C, r, gr, scale, part);
    hipLaunchKernelGGL(k_lora_wgrad_sum, dim3((unsigned)gx, (unsigned)E), dim3(256), 0, s, part,
                       n, gr, dw);
  });
}

}  // extern "C"
