// Batched independent streams on gfx950: B streams share the weights and each keeps its own
// K/V ring, hidden state and position. One step advances every stream by one event. The
// projections become skinny GEMMs [B x K] . W^T on MFMA, split over K across the waves of a
// workgroup and summed in LDS in a fixed order, with the phase's epilogue (RoPE and ring write,
// residual, SwiGLU) fused. Storage modes:
//  - FP32 and bfloat16 weights: FP32 activations, K/V and reductions; RMSNorm folded into the
//    projection prologue;
//  - mixed (the reference's FP16 mode): FP16 weights and K/V ring, every value rounded to FP16
//    at the reference's cast points, so each GEMM input is exactly FP16 and runs on
//    v_mfma_f32_16x16x32_f16 with FP32 accumulation; the norms, whose output is cast before the
//    projection, are folded into it too, or kernels of their own for large batches.
// Each stream follows the single-stream runtime's arithmetic up to summation order.
#pragma once

#include "step_device.hpp"

#include <type_traits>

namespace stamd {

constexpr int kBatchMax = 256;   // streams per batch (16 batch tiles of 16 in the GEMM)
constexpr int kBatchTile = 16;   // MFMA rows

typedef float f4v __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));

struct BatchArgs {
  int streams, streams_p;  // B and the padded batch (16, 32 or a multiple of 64)
  int layers, width, heads, dim, ffn, window, features;
  int width_p, ffn_p, features_p;  // padded row lengths
  float epsilon;
  const char* weights;
  uint32_t w_input, w_final_norm, w_score;
  LayerWeights layer[kMaxLayers];
  const float* rope_freq;          // [dim / 2]
  void* keys;                      // [L][B][H][W][dh], FP32 (FP16 in mixed mode): layer-major, so
                                   // that one layer's attention reads one contiguous region
  void* values;
  float* hidden;                   // [B][L][d]
  unsigned long long* position;    // [B]
  // Activations, Bp rows of the padded lengths, in the tiled layouts (act_index, half_index):
  float* in;                       // events (features_p)
  float* x;                        // residual stream (width_p); mixed mode: kSquares floats before it
  float* xn;                       // normalized x (mixed mode, FP16; width_p)
  float* attn;                     // attention output (FP16 in mixed mode; width_p)
  float* act;                      // SwiGLU output (FP16 in mixed mode; ffn_p)
  float* q;                        // [Bp][width] rotated queries
  float* score;                    // [B], host memory mapped into the device
  float2* rope;                    // [Bp][dim / 2] cos, sin of this step's position (batch_proj, kEpInput)
  int* slot;                       // [Bp] ring slot of this step's position
};

constexpr int kSlices = 8;       // K-slices of a projection, K / 8 columns each

// Mixed mode: the squares of x summed over four columns, kept right before x (so that a kernel
// with x's address needs no other argument): column quad n / 4 of row b at squares_index.
constexpr int kSquares = kBatchMax * kMaxDim / 4;
__host__ __device__ __forceinline__ int squares_index(int b, int quad) {
  return ((b >> 4) * (kMaxDim / 4) + quad) * 16 + (b & 15);
}
// Sum of v * v over each aligned quad of lanes. No contraction: every kernel must round alike.
__device__ __forceinline__ float quad_squares(float v) {
#pragma clang fp contract(off)
  const float s = v * v;
  return dpp_add<0x4E>(dpp_add<0xB1>(s));
}
constexpr size_t kInfinityCacheBytes = (size_t)256 << 20;  // MI355X's memory-side cache (MALL)

// Loads from the weight arena through the global address space. The arena's base arrives in
// the arguments block as a generic pointer, and a load through a generic (flat) pointer also
// counts on the LDS counter, so the compiler would wait for every outstanding load, the
// prefetched ones included, before a block's first MFMA.
typedef unsigned u32x2_t __attribute__((ext_vector_type(2)));
typedef unsigned u32x4_t __attribute__((ext_vector_type(4)));
__device__ __forceinline__ u32x4_t gload16(const void* p) {
  return *(const __attribute__((address_space(1))) u32x4_t*)p;
}
__device__ __forceinline__ f4v gload16f(const void* p) {
  return *(const __attribute__((address_space(1))) f4v*)p;
}
__device__ __forceinline__ uint2 gload8(const void* p) {
  return __builtin_bit_cast(uint2, *(const __attribute__((address_space(1))) u32x2_t*)p);
}

// Any pointer read from the arguments block, in the global address space.
template <typename T>
__device__ __forceinline__ __attribute__((address_space(1))) T* in_global(T* p) {
  return (__attribute__((address_space(1))) T*)p;
}

// Activation layouts. The projections' operands (in, x, xn, attn, act) are stored the way the
// weights are (the tiled arena): 16-row tiles of streams, then blocks of KB columns, then the
// 64 lanes of the MFMA operand (stream b mod 16 + 16 x column group), so that a wave loads a
// block as contiguous 16-byte runs in lane order. `cols` is the buffer's padded row length
// (a multiple of 32).
//  - FP32 buffers for the FP32 MFMA (FP32 storage; mixed mode's x and events): KB = 16, four
//    floats per lane.
//  - FP32 buffers for the bfloat16 MFMA (bfloat16 weights): KB = 32, eight floats per lane,
//    stored as two planes of four (the lane's low and high halves), each plane 64 x 16 bytes.
//  - FP16 buffers (mixed mode's xn, attn, act): KB = 32, eight halves per lane.
// Four consecutive columns from a multiple of 4 are consecutive in every layout.
template <int P>
__host__ __device__ __forceinline__ size_t act_index(int b, int n, int cols) {
  if constexpr (P == kBf16w) {
    const int kk = n & 31;
    return ((((size_t)(b >> 4) * (cols >> 5) + (n >> 5)) * 2 + ((kk >> 2) & 1)) * 64 + (b & 15) + 16 * (kk >> 3)) * 4 +
           (kk & 3);
  } else {
    const int kk = n & 15;
    return (((size_t)(b >> 4) * (cols >> 4) + (n >> 4)) * 64 + (b & 15) + 16 * (kk >> 2)) * 4 + (kk & 3);
  }
}
__host__ __device__ __forceinline__ size_t half_index(int b, int n, int cols) {
  const int kk = n & 31;
  return (((size_t)(b >> 4) * (cols >> 5) + (n >> 5)) * 64 + (b & 15) + 16 * (kk >> 3)) * 8 + (kk & 7);
}

enum BatchEpilogue : int { kEpInput = 0, kEpQkv, kEpOut, kEpGateUp, kEpDown };

// The exact three-term bfloat16 split of FP32 values, x = hi + mid + lo: truncations, hi keeps
// the top 8 significand bits, mid the next 8 of the remainder, lo the rest (at most 8 bits).
// Each term times a bfloat16 weight is exact in an FP32 accumulator.
__device__ __forceinline__ void split3(const float (&x)[8], unsigned (&ph)[4], unsigned (&pm)[4], unsigned (&pl)[4]) {
#pragma unroll
  for (int i = 0; i < 4; i++) {
    unsigned h2[2], m2[2], l2[2];
#pragma unroll
    for (int j = 0; j < 2; j++) {
      const float v = x[2 * i + j];
      const unsigned hb = __builtin_bit_cast(unsigned, v) & 0xffff0000u;
      const float r1 = v - __builtin_bit_cast(float, hb);
      const unsigned mb = __builtin_bit_cast(unsigned, r1) & 0xffff0000u;
      const float r2 = r1 - __builtin_bit_cast(float, mb);
      h2[j] = hb;
      m2[j] = mb;
      l2[j] = __builtin_bit_cast(unsigned, r2) & 0xffff0000u;
    }
    ph[i] = h2[1] | (h2[0] >> 16);
    pm[i] = m2[1] | (m2[0] >> 16);
    pl[i] = l2[1] | (l2[0] >> 16);
  }
}

// The K loop of one wave over its slice, columns k0 .. k0 + slice - 1, in blocks of KB columns: a
// ring of R blocks, unrolled so that no fragment is copied: block j + R is loaded into the
// fragments of block j as soon as block j's MFMAs are issued, so R blocks are in flight while one
// computes. The host picks R = 4 for workgroups of at most two tiles when the slice holds a
// multiple of 4 blocks (it always holds an even number), else 2.
// Three things hold the schedule: an empty asm after each block's loads (the compiler would otherwise
// see that a prefetch only feeds the next round and move it next to its use, and group the first
// blocks' loads by operand, so that the first block waits for the last one's); `pin`, which
// passes a fragment's registers through an asm right before its MFMAs (the compiler would
// otherwise hoist the operand arithmetic of every fragment to the top of the round, which waits
// for all loads in flight); and that the fragments are whole 4-register vectors in the pins too
// (pinned as scalars, the loop carried a register copy per element, which waited for every
// load at the end of each round: Large with bfloat16 weights at 32 streams 645 -> 595 us per step).
// `early` runs once, when the first R steps' loads are in flight: the epilogue's own operands
// are fetched there, so that their round trips overlap the loop's. Every form issues the
// MFMAs in block order.
template <int R, int KB, typename Frag, typename Load, typename Pin, typename Mma, typename Early>
__device__ __forceinline__ void k_ring(int k0, int slice, Load&& load, Pin&& pin, Mma&& mma, Early&& early) {
  const int nb = slice / KB;
  Frag f[R];
#pragma unroll
  for (int r = 0; r < R; r++) {
    load(k0 + r * KB, f[r]);
    asm volatile("" ::: "memory");
  }
  early();
  int j = 0;
  for (; j + R < nb; j += R) {
#pragma unroll
    for (int r = 0; r < R; r++) {
      pin(f[r]);
      mma(f[r]);
      load(k0 + (j + R + r) * KB, f[r]);
      asm volatile("" ::: "memory");
    }
  }
#pragma unroll
  for (int r = 0; r < R; r++) {
    pin(f[r]);
    mma(f[r]);
  }
}

__device__ __forceinline__ void pin4(u32x4_t& v) { asm volatile("" : "+v"(v)); }
__device__ __forceinline__ void pin4(f4v& v) { asm volatile("" : "+v"(v)); }
__device__ __forceinline__ void pin4(u32x2_t& v) { asm volatile("" : "+v"(v)); }

// One projection Y = X . W^T over the batch, with its phase's epilogue. Workgroup: CT column
// tiles of 16 outputs and NT batch tiles of 16 streams. K is cut into 8 slices; each of the 8 waves
// accumulates one for every tile pair with MFMA, reusing each X fragment for the CT column tiles
// and each weight fragment for the NT batch tiles. The slice partials are added in one fixed
// pairwise tree, ((s0 + s1) + (s2 + s3)) + ((s4 + s5) + (s6 + s7)), whatever NT and CT are, so a
// stream's outputs depend only on its own row and are bit-identical for every batch size. The
// padded batch is a multiple of NT tiles, so the loops have no branches. X and W are in the tiled operand layout (act_index and the tiled
// arena): one 16 x KB block of either is 64 lanes' contiguous 16-byte pieces in lane order.
// X is the padded buffer of K columns; W the N x K matrix at offset `woff` of the arena
// `weights`; `out` the phase's output buffer (row length out_ld): x, or the SwiGLU output.
// FP32 weights: v_mfma_f32_16x16x4_f32, k block of 16; lane l supplies A[l % 16][l / 16] and
// B[l / 16][l % 16], register r of lane l holds D[4 (l / 16) + r][l % 16]; the four MFMA
// steps use k = kb + 4 (l / 16) + c for step c, the same index for A and B.
// bfloat16 weights: v_mfma_f32_16x16x32_bf16, k block of 32, on the exact split of the FP32
// activation (3 MFMAs), so the product is the FP32 path's up to accumulation order. Lane
// (r16, g) holds k = kb + 8 g .. + 7 for both operands; the sum over k does not depend on how
// the hardware orders the lane groups.
// kNorm: X is the residual stream x and the projection consumes RMSNorm(x) . g
// (src/cuda/Primitives.cuh:122-135). The waves feed x * g to the MFMAs, accumulate the row's
// sum of squares from the same loads, and the epilogue scales the row by
// 1 / sqrt(sum / d + eps). Mixed mode casts the norm's output, so the scale has to be known before
// the MFMAs: the kernels that write x also write its squares summed over four columns
// (kSquares), and each wave adds those of its slice while its first K blocks are in flight. This
// saves the two norm kernels of a layer (about 2.5 us each) where the conversions that every
// column tile's workgroup then repeats cost less (Batch::folds_norm).
//
// Everything a kernel needs before its first load comes in the kernel arguments (the first 16
// dwords are preloaded into SGPRs). What only the epilogue needs (the residual, the RoPE table,
// the ring geometry) is fetched while the K loop's first loads are in flight: read after the
// loop, each of those was a dependent memory round trip on a kernel of 3-5 us (Main with
// bfloat16 weights at 16 streams 195 -> 188 us per step, Large at 32 streams 595 -> 576 us).
template <int P, int E, bool kNorm, int NT, int CT, int R>
__global__ __launch_bounds__(64 * kSlices) void batch_proj(const char* __restrict__ weights,
                                                           const void* __restrict__ X, void* out,
                                                           const BatchArgs* __restrict__ ap, uint32_t woff, int K,
                                                           uint32_t w_norm, int width, int streams, int out_ld,
                                                           int layer) {
  constexpr int kWaves = kSlices, kBlock = 64 * kWaves;
  constexpr bool kCastNorm = kNorm && P == kMixed;  // the norm's output is cast before the MFMAs
  constexpr bool kScale = kNorm && P != kMixed;     // the epilogue applies the norm's scale
  const BatchArgs& a = *ap;
  __shared__ float red[kWaves][NT][CT][16][17];
  __shared__ float sq[kWaves][NT][16];
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int n0 = blockIdx.x * kBatchTile * CT;
  const int t0 = blockIdx.y * NT;
  const int r16 = lane & 15, g = lane >> 4;
  const int slice = K / kSlices, k0 = wave * slice;

  // Epilogue units of this thread: a column, or the column pair of a RoPE or gate-up pair, of
  // one stream. Unit u of the workgroup's tiles is, for the phases that write an activation
  // buffer, in the buffer's own order (four columns of a row, then the 16 rows), so that a wave
  // stores (and loads the residual as) contiguous 256-byte runs; for QKV, whose outputs are
  // row-major, a row's pairs are consecutive.
  constexpr int unit = (E == kEpQkv || E == kEpGateUp) ? 2 : 1;
  constexpr int per_row = kBatchTile * CT / unit;
  constexpr int kUnits = NT * kBatchTile * per_row;
  constexpr int kOwn = (kUnits + kBlock - 1) / kBlock;
  struct Unit {
    int t, row, cc;  // batch tile, row in it, first column in the workgroup's
  };
  auto unit_of = [&](int u) {
    int o = (int)threadIdx.x + u * kBlock;
    if (kUnits % kBlock != 0 && o >= kUnits) o = kUnits - 1;
    if constexpr (E == kEpQkv) return Unit{o / (kBatchTile * per_row), (o / per_row) % kBatchTile, (o % per_row) * unit};
    else return Unit{o / (kBatchTile * per_row), (o >> 2) % kBatchTile, ((o / 64) % (per_row / 4) * 4 + (o & 3)) * unit};
  };
  auto owned = [&](int u) { return kUnits % kBlock == 0 || (int)threadIdx.x + u * kBlock < kUnits; };

  // Epilogue operands, fetched while the K loop's first loads are in flight. No branch around
  // the loads: threads without a unit load the last unit's operands, and rows past the last
  // stream are padding inside the buffers.
  float res[kOwn];           // OUT, down: the residual x
  v2f cs[kOwn];              // QKV: RoPE cos and sin of the pair
  int slot[kOwn];            // QKV: the stream's ring slot
  float epsilon = 0.f;
  float *hidden = nullptr, *qkv_q = nullptr, *qkv_k = nullptr, *qkv_v = nullptr;
  int layers = 0, dim = 1, heads = 1, window = 1;
  auto early = [&] {
    if constexpr (E == kEpInput) {
      // This step's RoPE table and ring slots (src/cuda/Primitives.cuh:148-166), once per step
      // instead of once per layer and unit: the workgroups of a batch tile group share its rows.
      const int half = a.dim / 2, rows = NT * kBatchTile;
      for (int i = (int)(blockIdx.x * kBlock + threadIdx.x); i < rows * half; i += (int)gridDim.x * kBlock) {
        const int b = t0 * kBatchTile + i / half, j = i % half;
        if (b >= streams) break;
        const unsigned long long pos = a.position[b];
        const float angle = (float)pos * a.rope_freq[j];
        a.rope[(size_t)b * half + j] = make_float2(cosf(angle), sinf(angle));
        if (j == 0) a.slot[b] = (int)(pos % (unsigned long long)a.window);
      }
    } else if constexpr (E == kEpQkv) {
      epsilon = a.epsilon;
      qkv_q = a.q;
      qkv_k = reinterpret_cast<float*>(a.keys);
      qkv_v = reinterpret_cast<float*>(a.values);
      dim = a.dim;
      heads = a.heads;
      window = a.window;
      const float2* rope = a.rope;
      const int* slots = a.slot;
      asm volatile("" ::"s"(epsilon), "s"(qkv_q), "s"(qkv_k), "s"(qkv_v), "s"(dim), "s"(heads), "s"(window), "s"(rope),
                   "s"(slots), "s"(layer));
#pragma unroll
      for (int u = 0; u < kOwn; u++) {
        const Unit o = unit_of(u);
        const int b = (t0 + o.t) * kBatchTile + o.row;
        cs[u] = __builtin_bit_cast(v2f, gload8(rope + (size_t)b * (dim / 2) + (n0 + o.cc) % dim / 2));
        slot[u] = in_global(slots)[b];
      }
    } else if constexpr (E == kEpGateUp) {
      if constexpr (kScale) {
        epsilon = a.epsilon;
        asm volatile("" ::"s"(epsilon));
      }
    } else {
      if constexpr (E == kEpDown) {
        hidden = a.hidden;
        layers = a.layers;
        asm volatile("" ::"s"(hidden), "s"(layers), "s"(layer));
      }
#pragma unroll
      for (int u = 0; u < kOwn; u++) {
        const Unit o = unit_of(u);
        res[u] = reinterpret_cast<const float*>(out)[act_index<P>((t0 + o.t) * kBatchTile + o.row, n0 + o.cc, out_ld)];
      }
    }
  };
  f4v acc[NT][CT];
  float ss[NT];
#pragma unroll
  for (int t = 0; t < NT; t++) {
    ss[t] = 0.f;
#pragma unroll
    for (int c = 0; c < CT; c++) acc[t][c] = f4v{0.f, 0.f, 0.f, 0.f};
  }
  // The slices' fixed tree over the waves' partials.
  auto tree = [&](auto at) {
    float p[4];
#pragma unroll
    for (int k = 0; k < 4; k++) p[k] = at(2 * k) + at(2 * k + 1);
    return (p[0] + p[1]) + (p[2] + p[3]);
  };
  // The arena pads a layer norm's gains with zeros to the K columns, so that their load has no
  // branch around it (one in the K loop's rounds drained every load in flight) and a padding
  // column's product is zero whatever the gains are.
  if constexpr (P == kFp32 || (P == kMixed && E == kEpInput)) {
    // FP32 MFMA. Mixed mode takes this path for the input projection only: its operand is
    // the raw FP32 event, and its FP16 weights widen exactly.
    // Tiled operands: block (tile, k / 16) holds 64 lanes x 4 values.
    const int nkb = K / 16;
    const float* xr = reinterpret_cast<const float*>(X) + ((size_t)t0 * nkb * 64 + lane) * 4;
    const char* wr = weights + woff + ((size_t)(n0 / kBatchTile) * nkb * 64 + lane) * 4 * (P == kFp32 ? 4 : 2);
    const float* gr = reinterpret_cast<const float*>(weights + w_norm);
    struct Frag {
      f4v w[CT], gn, x[NT];
    };
    auto load = [&](int k, Frag& f) {
#pragma unroll
      for (int c = 0; c < CT; c++) {
        const size_t blk = ((size_t)c * nkb + k / 16) * 256;
        if constexpr (P == kFp32) {
          f.w[c] = gload16f(reinterpret_cast<const float*>(wr) + blk);
        } else {
          const uint2 h = gload8(reinterpret_cast<const uint16_t*>(wr) + blk);
          f.w[c] = f4v{half_to_float((unsigned short)(h.x & 0xffffu)), half_to_float((unsigned short)(h.x >> 16)),
                       half_to_float((unsigned short)(h.y & 0xffffu)), half_to_float((unsigned short)(h.y >> 16))};
        }
      }
      if constexpr (kNorm) f.gn = gload16f(gr + k + 4 * g);
#pragma unroll
      for (int t = 0; t < NT; t++) f.x[t] = gload16f(xr + ((size_t)t * nkb + k / 16) * 256);
    };
    auto mma = [&](const Frag& f) {
#pragma unroll
      for (int t = 0; t < NT; t++) {
        f4v x = f.x[t];
        if constexpr (kNorm) {
          ss[t] += x.x * x.x;
          ss[t] += x.y * x.y;
          ss[t] += x.z * x.z;
          ss[t] += x.w * x.w;
          x.x *= f.gn.x;
          x.y *= f.gn.y;
          x.z *= f.gn.z;
          x.w *= f.gn.w;
        }
#pragma unroll
        for (int c = 0; c < CT; c++) {
          f4v& d = acc[t][c];
          d = __builtin_amdgcn_mfma_f32_16x16x4f32(x.x, f.w[c].x, d, 0, 0, 0);
          d = __builtin_amdgcn_mfma_f32_16x16x4f32(x.y, f.w[c].y, d, 0, 0, 0);
          d = __builtin_amdgcn_mfma_f32_16x16x4f32(x.z, f.w[c].z, d, 0, 0, 0);
          d = __builtin_amdgcn_mfma_f32_16x16x4f32(x.w, f.w[c].w, d, 0, 0, 0);
        }
      }
    };
    auto pin = [&](Frag& f) {
#pragma unroll
      for (int c = 0; c < CT; c++) pin4(f.w[c]);
#pragma unroll
      for (int t = 0; t < NT; t++) pin4(f.x[t]);
      if constexpr (kNorm) pin4(f.gn);
    };
    k_ring<R, 16, Frag>(k0, slice, load, pin, mma, early);
  } else if constexpr (P == kBf16w) {
    // Tiled operands: weight block (tile, k / 32) holds 64 lanes x 8 values, activation block
    // two planes of 64 lanes x 4 floats.
    const int nkb = K / 32;
    const float* xr = reinterpret_cast<const float*>(X) + ((size_t)t0 * nkb * 128 + lane) * 4;
    const uint16_t* wr = reinterpret_cast<const uint16_t*>(weights + woff) + ((size_t)(n0 / kBatchTile) * nkb * 64 + lane) * 8;
    const uint16_t* gr = reinterpret_cast<const uint16_t*>(weights + w_norm);
    struct Frag {
      u32x4_t w[CT], gn;
      f4v xlo[NT], xhi[NT];
    };
    auto load = [&](int k, Frag& f) {
#pragma unroll
      for (int c = 0; c < CT; c++) f.w[c] = gload16(wr + ((size_t)c * nkb + k / 32) * 512);
      if constexpr (kNorm) f.gn = gload16(gr + k + 8 * g);
#pragma unroll
      for (int t = 0; t < NT; t++) {
        const float* p = xr + ((size_t)t * nkb + k / 32) * 512;
        f.xlo[t] = gload16f(p);
        f.xhi[t] = gload16f(p + 256);
      }
    };
    auto mma = [&](const Frag& f) {
      float gv[8];
      if constexpr (kNorm) {
        const unsigned gu[4] = {f.gn.x, f.gn.y, f.gn.z, f.gn.w};
#pragma unroll
        for (int j = 0; j < 4; j++) {
          gv[2 * j] = __builtin_bit_cast(float, gu[j] << 16);
          gv[2 * j + 1] = __builtin_bit_cast(float, gu[j] & 0xffff0000u);
        }
      }
#pragma unroll
      for (int t = 0; t < NT; t++) {
        float x[8] = {f.xlo[t].x, f.xlo[t].y, f.xlo[t].z, f.xlo[t].w, f.xhi[t].x, f.xhi[t].y, f.xhi[t].z, f.xhi[t].w};
        if constexpr (kNorm) {
#pragma unroll
          for (int j = 0; j < 8; j++) {
            ss[t] += x[j] * x[j];
            x[j] *= gv[j];
          }
        }
        unsigned ph[4], pm[4], pl[4];
        split3(x, ph, pm, pl);
        const bf16x8 h = __builtin_bit_cast(bf16x8, ph), m = __builtin_bit_cast(bf16x8, pm),
                     l = __builtin_bit_cast(bf16x8, pl);
#pragma unroll
        for (int c = 0; c < CT; c++) {
          const bf16x8 wb = __builtin_bit_cast(bf16x8, f.w[c]);
          f4v& d = acc[t][c];
          d = __builtin_amdgcn_mfma_f32_16x16x32_bf16(h, wb, d, 0, 0, 0);
          d = __builtin_amdgcn_mfma_f32_16x16x32_bf16(m, wb, d, 0, 0, 0);
          d = __builtin_amdgcn_mfma_f32_16x16x32_bf16(l, wb, d, 0, 0, 0);
        }
      }
    };
    auto pin = [&](Frag& f) {
#pragma unroll
      for (int c = 0; c < CT; c++) pin4(f.w[c]);
#pragma unroll
      for (int t = 0; t < NT; t++) {
        pin4(f.xlo[t]);
        pin4(f.xhi[t]);
      }
      if constexpr (kNorm) pin4(f.gn);
    };
    k_ring<R, 32, Frag>(k0, slice, load, pin, mma, early);
  } else {
    // Mixed mode: the operand is an FP16 buffer (its values are cast points) and the weights
    // are FP16; one v_mfma_f32_16x16x32_f16 per 32-k block, lane (r16, g) holding
    // k = kb + 8 g .. + 7 of both, 16 bytes each.
    // Tiled operands: block (tile, k / 32) holds 64 lanes x 8 values.
    const int nkb = K / 32;
    const uint16_t* xr = reinterpret_cast<const uint16_t*>(X) + ((size_t)t0 * nkb * 64 + lane) * 8;
    const uint16_t* wr = reinterpret_cast<const uint16_t*>(weights + woff) + ((size_t)(n0 / kBatchTile) * nkb * 64 + lane) * 8;
    if constexpr (kCastNorm) {
      // X is x in FP32 (16-column blocks): lane (r16, g) takes its eight columns as two 16-byte
      // pieces and forms the FP16 operand (x . scale) . g, each value as batch_norm_mixed has it.
      const float* xs = reinterpret_cast<const float*>(X) +
                        (((size_t)t0 * 2 * nkb + (g >> 1)) * 64 + r16 + 32 * (g & 1)) * 4;
      const uint16_t* gr = reinterpret_cast<const uint16_t*>(weights + w_norm);
      // The slice's sums of squares: lane l loads rows 4 (l % 4) .. + 3 of column quad l / 4.
      const float* sr = reinterpret_cast<const float*>(X) - kSquares + squares_index(t0 * kBatchTile, 0) + 4 * lane;
      f4v part[NT];
#pragma unroll
      for (int t = 0; t < NT; t++) {
        const float* p = sr + squares_index(t * kBatchTile, k0 / 4);
        part[t] = gload16f(p);
        // Slices are 64 or 128 columns: 16 or 32 quads.
        if (slice > 64) part[t] += gload16f(p + 256);
      }
      asm volatile("" ::: "memory");
      float scale[NT];
      auto scales = [&] {
        epsilon = ap->epsilon;
#pragma unroll
        for (int t = 0; t < NT; t++)
#pragma unroll
          for (int k = 0; k < 4; k++) {
            const float v = column_sum(part[t][k], 4);
            if (lane < 4) sq[wave][t][4 * lane + k] = v;
          }
        __syncthreads();
#pragma unroll
        for (int t = 0; t < NT; t++) scale[t] = 1.0f / sqrtf(tree([&](int k) { return sq[k][t][r16]; }) / (float)width + epsilon);
      };
      struct Frag {
        u32x4_t w[CT], gn;
        f4v xlo[NT], xhi[NT];
      };
      auto load = [&](int k, Frag& f) {
#pragma unroll
        for (int c = 0; c < CT; c++) f.w[c] = gload16(wr + ((size_t)c * nkb + k / 32) * 512);
        f.gn = gload16(gr + k + 8 * g);
#pragma unroll
        for (int t = 0; t < NT; t++) {
          const float* p = xs + ((size_t)t * nkb + k / 32) * 512;
          f.xlo[t] = gload16f(p);
          f.xhi[t] = gload16f(p + 64);
        }
      };
      auto mma = [&](const Frag& f) {
        const f16x8 gh = __builtin_bit_cast(f16x8, f.gn);
#pragma unroll
        for (int t = 0; t < NT; t++) {
          f16x8 xh;
#pragma unroll
          for (int j = 0; j < 8; j++) xh[j] = (_Float16)((j < 4 ? f.xlo[t][j & 3] : f.xhi[t][j & 3]) * scale[t] * (float)gh[j]);
#pragma unroll
          for (int c = 0; c < CT; c++)
            acc[t][c] = __builtin_amdgcn_mfma_f32_16x16x32_f16(xh, __builtin_bit_cast(f16x8, f.w[c]), acc[t][c], 0, 0, 0);
        }
      };
      auto pin = [&](Frag& f) {
#pragma unroll
        for (int c = 0; c < CT; c++) pin4(f.w[c]);
#pragma unroll
        for (int t = 0; t < NT; t++) {
          pin4(f.xlo[t]);
          pin4(f.xhi[t]);
        }
        pin4(f.gn);
      };
      k_ring<R, 32, Frag>(k0, slice, load, pin, mma, [&] {
        early();
        scales();
      });
    } else {
      struct Frag {
        u32x4_t w[CT], x[NT];
      };
      auto load = [&](int k, Frag& f) {
#pragma unroll
        for (int c = 0; c < CT; c++) f.w[c] = gload16(wr + ((size_t)c * nkb + k / 32) * 512);
#pragma unroll
        for (int t = 0; t < NT; t++) f.x[t] = gload16(xr + ((size_t)t * nkb + k / 32) * 512);
      };
      auto mma = [&](const Frag& f) {
#pragma unroll
        for (int t = 0; t < NT; t++)
#pragma unroll
          for (int c = 0; c < CT; c++)
            acc[t][c] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, f.x[t]),
                                                                  __builtin_bit_cast(f16x8, f.w[c]), acc[t][c], 0, 0, 0);
      };
      auto pin = [&](Frag& f) {
#pragma unroll
        for (int c = 0; c < CT; c++) pin4(f.w[c]);
#pragma unroll
        for (int t = 0; t < NT; t++) pin4(f.x[t]);
      };
      k_ring<R, 32, Frag>(k0, slice, load, pin, mma, early);
    }
  }
#pragma unroll
  for (int t = 0; t < NT; t++) {
#pragma unroll
    for (int c = 0; c < CT; c++)
#pragma unroll
      for (int r = 0; r < 4; r++) red[wave][t][c][4 * g + r][r16] = acc[t][c][r];
    if constexpr (kScale) {
      const float v = column_sum(ss[t], 16);
      if (g == 0) sq[wave][t][r16] = v;
    }
  }
  __syncthreads();
#pragma unroll
  for (int u = 0; u < kOwn; u++) {
    if (!owned(u)) break;
    const Unit o = unit_of(u);
    const int b = (t0 + o.t) * kBatchTile + o.row;
    if (b >= streams) continue;
    const int c = o.cc / kBatchTile, col = o.cc % kBatchTile;
    float s0 = tree([&](int k) { return red[k][o.t][c][o.row][col]; });
    float s1 = unit == 2 ? tree([&](int k) { return red[k][o.t][c][o.row][col + 1]; }) : 0.f;
    if constexpr (kScale) {
      const float sum = tree([&](int k) { return sq[k][o.t][o.row]; });
      const float scale = 1.0f / sqrtf(sum / (float)width + epsilon);
      s0 *= scale;
      s1 *= scale;
    }
    // Projection outputs are cast (mixed mode), then each epilogue casts where the reference
    // does (src/cuda/Primitives.cuh:148-239); cast<P> is the identity for FP32 storage.
    s0 = cast<P>(s0);
    s1 = cast<P>(s1);
    const int n = n0 + o.cc;
    // Mixed mode: the squares of the four columns that a quad of lanes writes to x.
    auto squares = [&](float v) {
      if constexpr (P == kMixed) {
        const float v2 = quad_squares(v);
        if ((lane & 3) == 0) in_global(reinterpret_cast<float*>(out))[squares_index(b, n >> 2) - kSquares] = v2;
      }
    };
    if constexpr (E == kEpInput) {
      reinterpret_cast<float*>(out)[act_index<P>(b, n, out_ld)] = s0;
      squares(s0);
    } else if constexpr (E == kEpQkv) {
      // src/cuda/Primitives.cuh:148-166: RoPE on adjacent pairs of q and k, then the ring write.
      const int sec = (n >= width) + (n >= 2 * width);
      const int i = n - sec * width;
      float va = s0, vb = s1;
      if (sec < 2) {
        // No FMA contraction here: left to the compiler, it fuses one product or the other
        // depending on the kernel variant, and a stream's bits would then depend on the
        // workgroup shape chosen for its batch size.
#pragma clang fp contract(off)
        const float ra = va * cs[u].x - vb * cs[u].y, rb = va * cs[u].y + vb * cs[u].x;
        va = cast<P>(ra);
        vb = cast<P>(rb);
      }
      const int h = i / dim, d = i - h * dim;
      const size_t dst = sec == 0 ? (size_t)b * width + i
                                  : ((((size_t)layer * streams + b) * heads + h) * window + slot[u]) * dim + d;
      float* base = sec == 0 ? qkv_q : sec == 1 ? qkv_k : qkv_v;
      if (P == kMixed && sec != 0) {
        *in_global(reinterpret_cast<unsigned*>(reinterpret_cast<uint16_t*>(base) + dst)) =
            (unsigned)float_to_half(va) | ((unsigned)float_to_half(vb) << 16);
      } else {
        *in_global(reinterpret_cast<v2f*>(base + dst)) = v2f{va, vb};
      }
    } else if constexpr (E == kEpOut) {
      const float v = cast<P>(res[u] + s0);
      reinterpret_cast<float*>(out)[act_index<P>(b, n, out_ld)] = v;
      squares(v);
    } else if constexpr (E == kEpGateUp) {
      const float v = cast<P>((s0 / (1.0f + expf(-s0))) * s1);
      if constexpr (P == kMixed) reinterpret_cast<uint16_t*>(out)[half_index(b, n >> 1, out_ld)] = float_to_half(v);
      else reinterpret_cast<float*>(out)[act_index<P>(b, n >> 1, out_ld)] = v;
    } else {
      const float v = cast<P>(res[u] + s0);
      reinterpret_cast<float*>(out)[act_index<P>(b, n, out_ld)] = v;
      squares(v);
      in_global(hidden)[((size_t)b * layers + layer) * width + n] = v;
    }
  }
}

// Four consecutive ring elements of K or V (FP32, or FP16 in mixed mode) as floats.
// Global (not flat) loads, so that they count on the vector memory counter only; kNT marks
// them non-temporal, for rings larger than the Infinity Cache (see batch_attention).
template <int P, bool kNT>
__device__ __forceinline__ float4 ring4(const void* ring, size_t i) {
  typedef const __attribute__((address_space(1))) u32x2_t g2;
  typedef const __attribute__((address_space(1))) u32x4_t g4;
  if constexpr (P == kMixed) {
    const void* p = reinterpret_cast<const uint16_t*>(ring) + i;
    const uint2 h = __builtin_bit_cast(uint2, kNT ? __builtin_nontemporal_load((g2*)p) : *(g2*)p);
    return make_float4(half_to_float((unsigned short)(h.x & 0xffffu)), half_to_float((unsigned short)(h.x >> 16)),
                       half_to_float((unsigned short)(h.y & 0xffffu)), half_to_float((unsigned short)(h.y >> 16)));
  } else {
    const void* p = reinterpret_cast<const float*>(ring) + i;
    return __builtin_bit_cast(float4, kNT ? __builtin_nontemporal_load((g4*)p) : *(g4*)p);
  }
}

// Four consecutive ring elements as loaded (FP16 pairs in mixed mode), and their FP32 values.
// The chunked attention keeps the loaded form in registers and widens at each use, so that the
// FP16 values feed mixed-precision FMAs directly (widening is exact, the results unchanged).
template <int P>
using RingRaw = std::conditional_t<P == kMixed, u32x2_t, f4v>;
template <int P, bool kNT>
__device__ __forceinline__ RingRaw<P> ring_raw(const void* ring, size_t i) {
  typedef const __attribute__((address_space(1))) u32x2_t g2;
  typedef const __attribute__((address_space(1))) u32x4_t g4;
  if constexpr (P == kMixed) {
    const void* p = reinterpret_cast<const uint16_t*>(ring) + i;
    return kNT ? __builtin_nontemporal_load((g2*)p) : *(g2*)p;
  } else {
    return __builtin_bit_cast(f4v, ring4<P, kNT>(ring, i));
  }
}
__device__ __forceinline__ f4v widen(f4v v) { return v; }
__device__ __forceinline__ f4v widen(u32x2_t h) {
  return f4v{half_to_float((unsigned short)(h.x & 0xffffu)), half_to_float((unsigned short)(h.x >> 16)),
             half_to_float((unsigned short)(h.y & 0xffffu)), half_to_float((unsigned short)(h.y >> 16))};
}

constexpr int kAttnThreads = 256;  // batch_attention's workgroup: four waves, 16 groups of 16 lanes
constexpr int kAttnWaves = kAttnThreads / 64;
constexpr int kBatchChunk = 128;    // ring slots per attention chunk

// The values of lanes 0 .. N - 1 of each row of 16 lanes, in every lane of the row.
template <int N, int K = 0>
__device__ __forceinline__ void row_values(float v, float (&out)[N]) {
  out[K] = dpp_get<0x150 + K>(v);  // row_newbcast:K
  if constexpr (K + 1 < N) row_values<N, K + 1>(v, out);
}

// Weight of a softmax partial with maximum m beside the overall maximum `top`. A partial without
// finite logits (m = -inf) carries zeros and gets weight zero; if every logit is -inf the sum is
// zero and the output 0 / 0, as a softmax over them has it.
__device__ __forceinline__ float partial_weight(float m, float top) { return m == -INFINITY ? 0.f : expf(m - top); }

// One element of the attention output, [b][n] of the padded rows.
template <int P>
__device__ __forceinline__ void put_attn(void* attn, int b, int n, int width_p, float v) {
  if constexpr (P == kMixed) in_global(reinterpret_cast<uint16_t*>(attn))[half_index(b, n, width_p)] = float_to_half(v);
  else in_global(reinterpret_cast<float*>(attn))[act_index<P>(b, n, width_p)] = v;
}

// Attention of one (stream, head) over the stream's valid ring slots [0, valid)
// (src/cuda/Primitives.cuh:167-219): logits q.K/sqrt(dh), softmax, weighted V, cast. Slot order
// does not change the result beyond summation order. Head dims up to 64 DV (DV 1 or 2), a
// multiple of 4.
//
// The window is cut into chunks of kBatchChunk slots. 16 lanes share a K (or V) row, 4 DV elements
// each, so a wave's load covers 4 rows; a wave owns 4 rows of each of the NP passes of 16 rows,
// and the chunk's K and V loads are all issued before the first dot product (NP = 8; windows of
// at most 64 slots take NP = 4). Each wave forms its own softmax partial of a chunk: its rows'
// maximum m, s = sum exp(l - m), o = sum exp(l - m) V, in registers. One barrier, then the
// four waves' partials of each chunk are merged, and the chunks in order. So the critical path of a
// one-chunk window is: position, K and V in one round trip, one barrier. (Before: the arguments
// block, then the position, then K; a maximum, a sum and an output through LDS with five
// barriers. Main with bfloat16 weights at 16 streams 188.7 -> 178.4 us per step, at 256 430.6 ->
// 425.5; mixed mode at 64 streams 243.2 -> 239.3.)
//
// From a few hundred (stream, head) pairs of small heads or short rows on, the instructions bound
// the kernel and not the loads: a row's division and exponential are computed by one of its 16
// lanes and broadcast, chunks before the last test no slot, and empty half chunks are skipped (one
// in each lane, every slot tested, no skip: mixed mode with 35 heads of 16, W = 282, 115 streams
// 44.2 -> 30.3 us per layer; a step of three layers with 112 heads of 4, W = 409, 50 streams
// 286 -> 205 us; Main at 16 streams 152.6 -> 150.7, bit-identical).
//
// Workgroups: gridDim.z == 1: one walks all chunks of its (stream, head), its partials in LDS (at most
// 32 chunks: 34 KB for head dims up to 64, else 67 KB, where registers hold a CU to two to four
// workgroups anyway).
// Otherwise workgroup z takes chunk z, writes the chunk's partial through to memory and counts
// itself; the last to arrive merges the chunks (it finds every partial there: nothing waits).
// Both run the same arithmetic in the same order, so a stream's bits do not depend on the form,
// which the host picks by how many workgroups the (stream, head) pairs alone would give.
//
// kAny: the first loads clamp rows to the window instead of to the valid slots, so that they do
// not wait for the position (slots not yet written hold the zeros of the reset and are dropped).
// kNT: the K and V loads are non-temporal, for rings that do not fit in the Infinity Cache
// beside the weights: a step streams them through once, and cached they would evict the
// weights the projections re-read (Main, bfloat16 weights: 454 -> 436 us per step at 256
// streams, 249 -> 241 at 64; mixed mode 400 -> 382 at 256). Rings that fit stay cached from
// step to step instead (mixed mode at 64 streams: 253 against 270 us).
template <int P, int DV, int NP, bool kAny, bool kNT>
__global__ __launch_bounds__(kAttnThreads) void batch_attention(const unsigned long long* __restrict__ position,
                                                                const float* __restrict__ q, const void* keys,
                                                                const void* values, void* attn, int window, int dim,
                                                                int heads, int width_p, float* partial,
                                                                unsigned* arrived) {
  extern __shared__ float part[];  // [chunk][wave][64 DV + 2]: o, then m and s
  constexpr int kRow = 64 * DV + 2;
  const int h = blockIdx.x, b = blockIdx.y;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, r = tid & 15, grp = tid >> 4;
  const int d = 4 * r;
  const size_t base = ((size_t)b * heads + h) * (size_t)window * dim;
  const bool split = gridDim.z > 1;
  const int first = split ? (int)blockIdx.z : 0;
  const float div = sqrtf((float)dim);
  // K and V stay in their loaded form (RingRaw: FP16 pairs in mixed mode) until used. Lanes past
  // the head dim load the row's last elements and drop them.
  RingRaw<P> kv[NP][DV], vv[NP][DV];
  int dd[DV];
  f4v qv[DV];
#pragma unroll
  for (int j = 0; j < DV; j++) {
    dd[j] = d + 64 * j < dim ? d + 64 * j : dim - 4;
    qv[j] = gload16f(q + ((size_t)b * heads + h) * dim + dd[j]);
  }
  auto load = [&](const void* ring, RingRaw<P> (&f)[NP][DV], int c0, int limit) {
#pragma unroll
    for (int p = 0; p < NP; p++) {
      const int s = c0 + 16 * p + grp;
      const size_t row = base + (size_t)(s < limit ? s : limit - 1) * dim;
#pragma unroll
      for (int j = 0; j < DV; j++) f[p][j] = ring_raw<P, kNT>(ring, row + dd[j]);
    }
    asm volatile("" ::: "memory");  // the loads stay here, ahead of the arithmetic
  };
  int valid = window;
  if constexpr (!kAny) {
    const unsigned long long t = position[b];
    valid = t + 1 < (unsigned long long)window ? (int)(t + 1) : window;
    if (first * kBatchChunk >= valid) return;
  }
  load(keys, kv, first * kBatchChunk, valid);
  load(values, vv, first * kBatchChunk, valid);
  if constexpr (kAny) {
    const unsigned long long t = position[b];
    valid = t + 1 < (unsigned long long)window ? (int)(t + 1) : window;
  }
  const int active = (valid + kBatchChunk - 1) / kBatchChunk;  // chunks with valid slots
  const int last = split ? first + 1 : active;
  // One chunk; with `more` its registers are reloaded with the next chunk's rows as soon as they are
  // used, without a condition (a conditional load came out as a register copy per element at the
  // end of the round, which waited for every load). The pins keep each row's arithmetic after
  // its own load.
  auto chunk = [&](int c, auto more) {
    const int c0 = c * kBatchChunk;
    // Chunks before the last hold valid slots only.
    auto live = [&](int pass) { return more.value || c0 + 16 * pass + grp < valid; };
    // No valid slot in the last chunk's second half: its passes are skipped.
    const bool both = more.value || c0 + 8 * NP < valid;
    // Lane r keeps the logit of pass r mod NP, for one division and one exponential per row.
    float lg = 0.f;
#pragma unroll
    for (int p = 0; p < NP; p++) {
      if (p >= NP / 2 && !both) break;
      float dot = 0.f;
#pragma unroll
      for (int j = 0; j < DV; j++) {
        pin4(kv[p][j]);
        const f4v k = widen(kv[p][j]);
        float part_dot = __builtin_fmaf(qv[j].x, k.x, dot);
        part_dot = __builtin_fmaf(qv[j].y, k.y, part_dot);
        part_dot = __builtin_fmaf(qv[j].z, k.z, part_dot);
        part_dot = __builtin_fmaf(qv[j].w, k.w, part_dot);
        dot = d + 64 * j < dim ? part_dot : dot;
      }
      dot = group_sum(dot, 16);
      lg = r % NP == p ? dot : lg;
    }
    if constexpr (more.value) load(keys, kv, c0 + kBatchChunk, valid);
    lg = live(r % NP) ? lg / div : -INFINITY;
    const float mx = wave_top(lg);
    const float ref = mx == -INFINITY ? 0.f : mx;
    float e[NP];
    row_values<NP>(expf(lg - ref), e);
    float sum = 0.f;
    f4v o[DV];
#pragma unroll
    for (int j = 0; j < DV; j++) o[j] = f4v{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int p = 0; p < NP; p++) {
      if (p >= NP / 2 && !both) break;
      sum += e[p];
#pragma unroll
      for (int j = 0; j < DV; j++) {
        pin4(vv[p][j]);
        const f4v v = widen(vv[p][j]);
        o[j].x = live(p) ? __builtin_fmaf(e[p], v.x, o[j].x) : o[j].x;
        o[j].y = live(p) ? __builtin_fmaf(e[p], v.y, o[j].y) : o[j].y;
        o[j].z = live(p) ? __builtin_fmaf(e[p], v.z, o[j].z) : o[j].z;
        o[j].w = live(p) ? __builtin_fmaf(e[p], v.w, o[j].w) : o[j].w;
      }
    }
    if constexpr (more.value) load(values, vv, c0 + kBatchChunk, valid);
    sum = column_sum(sum, 16);
    float* mine = part + ((c - first) * kAttnWaves + wave) * kRow;
#pragma unroll
    for (int j = 0; j < DV; j++) {
      o[j].x = column_sum(o[j].x, 16);
      o[j].y = column_sum(o[j].y, 16);
      o[j].z = column_sum(o[j].z, 16);
      o[j].w = column_sum(o[j].w, 16);
      if (lane < 16) {
        mine[64 * j + d] = o[j].x;
        mine[64 * j + d + 1] = o[j].y;
        mine[64 * j + d + 2] = o[j].z;
        mine[64 * j + d + 3] = o[j].w;
      }
    }
    if (lane == 0) {
      mine[64 * DV] = mx;
      mine[64 * DV + 1] = sum;
    }
  };
  int c = first;
  for (; c + 1 < last; c++) chunk(c, std::true_type{});
  chunk(c, std::false_type{});
  __syncthreads();
  // The merges, each lane for its own columns lane + 64 j. No FMA contraction: both forms must
  // round alike.
  auto merge_waves = [&](int c, float& m, float& s, float (&o)[DV]) {
    const float* w = part + c * kAttnWaves * kRow;
    float mw[4], e[4];
#pragma unroll
    for (int k = 0; k < 4; k++) mw[k] = w[k * kRow + 64 * DV];
    m = fmaxf(fmaxf(mw[0], mw[1]), fmaxf(mw[2], mw[3]));
#pragma unroll
    for (int k = 0; k < 4; k++) e[k] = partial_weight(mw[k], m);
    auto sum4 = [&](int i) {
#pragma clang fp contract(off)
      return (w[i] * e[0] + w[kRow + i] * e[1]) + (w[2 * kRow + i] * e[2] + w[3 * kRow + i] * e[3]);
    };
    s = sum4(64 * DV + 1);
#pragma unroll
    for (int j = 0; j < DV; j++) o[j] = sum4(lane + 64 * j);
  };
  auto put = [&](const float (&num)[DV], float den) {
#pragma unroll
    for (int j = 0; j < DV; j++)
      if (lane + 64 * j < dim) put_attn<P>(attn, b, h * dim + lane + 64 * j, width_p, num[j] / den);
  };
  float m, s, o[DV];
  float num[DV], den = 0.f, top = -INFINITY;
#pragma unroll
  for (int j = 0; j < DV; j++) num[j] = 0.f;
  auto add_chunk = [&](float mc, float sc, const float (&oc)[DV]) {
#pragma clang fp contract(off)
    const float e = partial_weight(mc, top);
    den = den + sc * e;
#pragma unroll
    for (int j = 0; j < DV; j++) num[j] = num[j] + oc[j] * e;
  };
  if (!split && active > 1) {
    // A wave merges every fourth chunk, into the place of the chunk's first partial; wave 0 adds the
    // chunks in order. (One wave merging all: 512 pairs of 32 chunks 363.8 -> 358.7 us per step of
    // two layers, of 16 FP16 chunks at 1024 pairs 210.6 -> 204.3.)
    auto row = [&](int c) { return part + c * kAttnWaves * kRow; };
    for (int c = wave; c < active; c += kAttnWaves) {
      merge_waves(c, m, s, o);
      float* to = row(c);
#pragma unroll
      for (int j = 0; j < DV; j++) to[lane + 64 * j] = o[j];
      if (lane == 0) {
        to[64 * DV] = m;
        to[64 * DV + 1] = s;
      }
    }
    __syncthreads();
    if (wave != 0) return;
    for (int c = lane; c < active; c += 64) top = fmaxf(top, row(c)[64 * DV]);
    top = wave_top(top);
#pragma unroll 4
    for (int c = 0; c < active; c++) {
#pragma unroll
      for (int j = 0; j < DV; j++) o[j] = row(c)[lane + 64 * j];
      add_chunk(row(c)[64 * DV], row(c)[64 * DV + 1], o);
    }
    put(num, den);
    return;
  }
  if (wave != 0) return;
  if (active == 1) {
    merge_waves(0, m, s, o);
    put(o, s);
    return;
  }
  // This chunk's partial, written through to memory (agent scope) and complete before the count.
  merge_waves(0, m, s, o);
  const int chunks = (int)gridDim.z, pair = b * heads + h;
  float* mine = partial + ((size_t)pair * chunks) * kRow;
  auto at = [&](int c, int i) { return in_global(mine + (size_t)c * kRow + i); };
#pragma unroll
  for (int j = 0; j < DV; j++)
    __hip_atomic_store(at(first, lane + 64 * j), o[j], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  if (lane == 0) {
    __hip_atomic_store(at(first, 64 * DV), m, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __hip_atomic_store(at(first, 64 * DV + 1), s, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  unsigned before = 0;
  if (lane == 0) before = __hip_atomic_fetch_add(arrived + pair, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  before = __builtin_amdgcn_readfirstlane(before);
  if (before + 1 != (unsigned)active) return;
  asm volatile("" ::: "memory");
  if (lane == 0) __hip_atomic_store(arrived + pair, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  auto get = [&](int c, int i) { return __hip_atomic_load(at(c, i), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); };
  // Up to kAhead chunks in one round trip, any others (windows over 1024 slots) after it.
  constexpr int kAhead = 8;
  float mc[kAhead], sc[kAhead], oc[kAhead][DV];
#pragma unroll
  for (int c = 0; c < kAhead; c++) {
    const int cc = c < active ? c : active - 1;
    mc[c] = get(cc, 64 * DV);
    sc[c] = get(cc, 64 * DV + 1);
#pragma unroll
    for (int j = 0; j < DV; j++) oc[c][j] = get(cc, lane + 64 * j);
  }
#pragma unroll
  for (int c = 0; c < kAhead; c++) top = fmaxf(top, mc[c]);
  for (int c = kAhead; c < active; c++) top = fmaxf(top, get(c, 64 * DV));
#pragma unroll
  for (int c = 0; c < kAhead; c++)
    if (c < active) add_chunk(mc[c], sc[c], oc[c]);
  for (int c = kAhead; c < active; c++) {
#pragma unroll
    for (int j = 0; j < DV; j++) o[j] = get(c, lane + 64 * j);
    add_chunk(get(c, 64 * DV), get(c, 64 * DV + 1), o);
  }
  put(num, den);
}

// The same attention for head dims above 128: four waves walk the rows pass by pass, 16 lanes
// per row in pieces of 64 elements, the softmax maximum and sum through LDS, and the 16 lane groups'
// V sums added in group order. Dynamic LDS holds `window` floats of probabilities.
template <int P, bool kNT>
__global__ __launch_bounds__(kAttnThreads) void batch_attention_wide(const unsigned long long* __restrict__ position,
                                                                     const float* __restrict__ qs, const void* keys,
                                                                     const void* values, void* attn, int window, int dim,
                                                                     int heads, int width_p) {
  extern __shared__ float pr[];
  __shared__ float wred[kAttnThreads / 64];
  __shared__ float4 vred[16][17];
  const int h = blockIdx.x, b = blockIdx.y;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int r = tid & 15, grp = tid >> 4;  // 16 groups of 16 lanes
  const unsigned long long t = position[b];
  const int valid = t + 1 < (unsigned long long)window ? (int)(t + 1) : window;
  const size_t base = ((size_t)b * heads + h) * (size_t)window * dim;
  const float* q = qs + ((size_t)b * heads + h) * dim;
  const float div = sqrtf((float)dim);
  float mx = -INFINITY;
  // Rows past `valid` load row valid - 1 and are dropped, so the loop body has no branch
  // around its loads and several passes of loads stay in flight.
#pragma unroll 4
  for (int s0 = 0; s0 < valid; s0 += kAttnThreads / 16) {
    const int s = s0 + grp;
    const size_t row = base + (size_t)(s < valid ? s : valid - 1) * dim;
    float dot = 0.f;
    for (int d = 4 * r; d < dim; d += 64) {
      const float4 kv = ring4<P, kNT>(keys, row + d);
      const float4 qv = *reinterpret_cast<const float4*>(q + d);
      dot += qv.x * kv.x;
      dot += qv.y * kv.y;
      dot += qv.z * kv.z;
      dot += qv.w * kv.w;
    }
    dot = group_sum(dot, 16);
    if (s < valid) {
      const float lg = dot / div;
      if (r == 0) pr[s] = lg;
      mx = fmaxf(mx, lg);
    }
  }
  mx = wave_top(mx);
  if (lane == 0) wred[wave] = mx;
  __syncthreads();
  mx = fmaxf(fmaxf(wred[0], wred[1]), fmaxf(wred[2], wred[3]));
  float sum = 0.f;
  for (int s = tid; s < valid; s += kAttnThreads) {
    const float e = expf(pr[s] - mx);
    pr[s] = e;
    sum += e;
  }
  sum = wave_total(sum);
  __syncthreads();  // every wave has read wred (max) and written its probabilities
  if (lane == 0) wred[wave] = sum;
  __syncthreads();
  sum = (wred[0] + wred[1]) + (wred[2] + wred[3]);
  for (int d0 = 0; d0 < dim; d0 += 64) {
    const int d = d0 + 4 * r;
    float4 o = make_float4(0.f, 0.f, 0.f, 0.f);
    if (d < dim) {
#pragma unroll 4
      for (int s = grp; s < valid; s += 16) {
        const float p = pr[s];
        const float4 vv = ring4<P, kNT>(values, base + (size_t)s * dim + d);
        o.x += p * vv.x;
        o.y += p * vv.y;
        o.z += p * vv.z;
        o.w += p * vv.w;
      }
    }
    vred[grp][r] = o;
    __syncthreads();
    if (tid < 16 && d0 + 4 * tid < dim) {
      float4 acc = vred[0][tid];
      for (int k = 1; k < 16; k++) {
        const float4 v = vred[k][tid];
        acc.x += v.x;
        acc.y += v.y;
        acc.z += v.z;
        acc.w += v.w;
      }
      const float o4[4] = {acc.x / sum, acc.y / sum, acc.z / sum, acc.w / sum};
      const int n = h * dim + d0 + 4 * tid;
#pragma unroll
      for (int j = 0; j < 4; j++) put_attn<P>(attn, b, n + j, width_p, o4[j]);
    }
    __syncthreads();
  }
}

// One element of a norm or score vector in the arena, decoded to FP32.
template <int P>
__device__ __forceinline__ float batch_weight(const char* w, uint32_t off, int i) {
  if constexpr (P == kFp32) return reinterpret_cast<const float*>(w + off)[i];
  if constexpr (P == kMixed) return half_to_float(reinterpret_cast<const uint16_t*>(w + off)[i]);
  return bf16_to_float(reinterpret_cast<const uint16_t*>(w + off)[i]);
}

// Mixed mode, batches whose projections do not fold the norm: RMSNorm of every stream's x into xn
// with the output cast to FP16 (src/cuda/Primitives.cuh:122-135); padding columns and padding
// streams are zero. One workgroup of 256 threads per row of the padded batch; a wave takes two of
// the eight K-slices. The sum of squares is added as the writers of x and the folding projections
// add it (column quads, a slice's 64-column pieces, slices), so that a stream's bits do not depend
// on which of the two ran. Every load (x and the norm vector, at most 4 columns per thread) is
// issued before the reduction: one memory round trip.
static __global__ __launch_bounds__(256) void batch_norm_mixed(const BatchArgs* __restrict__ ap, uint32_t w_norm) {
  const BatchArgs& a = *ap;
  __shared__ float red[4];
  const int b = blockIdx.x, wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const float* x = a.x;
  uint16_t* out = reinterpret_cast<uint16_t*>(a.xn);
  if (b >= a.streams) {
    for (int i = threadIdx.x; i < a.width_p; i += blockDim.x) out[half_index(b, i, a.width_p)] = 0;
    return;
  }
  constexpr int kPer = kMaxDim / 256;
  const int per = a.width_p / 256;  // 64-column pieces of the wave: 2 (one per slice) or 4
  float xv[kPer], gv[kPer], sq[kPer];
#pragma unroll
  for (int j = 0; j < kPer; j++) {
    const int i = (wave * per + j) * 64 + lane;
    const bool in = j < per && i < a.width;
    xv[j] = in ? x[act_index<kMixed>(b, i, a.width_p)] : 0.f;
    gv[j] = in ? batch_weight<kMixed>(a.weights, w_norm, i) : 0.f;
  }
#pragma unroll
  for (int j = 0; j < kPer; j++) sq[j] = quad_squares(xv[j]);
  const float s0 = per > 2 ? sq[0] + sq[1] : sq[0], s1 = per > 2 ? sq[2] + sq[3] : sq[1];
  const float s = column_sum(s0, 4) + column_sum(s1, 4);
  if (lane == 0) red[wave] = s;
  __syncthreads();
  const float scale = 1.0f / sqrtf(((red[0] + red[1]) + (red[2] + red[3])) / (float)a.width + a.epsilon);
#pragma unroll
  for (int j = 0; j < kPer; j++) {
    const int i = (wave * per + j) * 64 + lane;
    if (j < per) out[half_index(b, i, a.width_p)] = i < a.width ? float_to_half(xv[j] * scale * gv[j]) : 0;
  }
}

// Final RMSNorm (cast in mixed mode) and score of every stream (src/cuda/Runtime.cu:380-383;
// the score itself is not cast), then the position advance. One wave per stream.
template <int P>
__global__ __launch_bounds__(64) void batch_final(const BatchArgs* __restrict__ ap) {
  const BatchArgs& a = *ap;
  const int b = blockIdx.x, lane = threadIdx.x;
  const float* x = a.x;
  auto xb = [&](int i) { return x[act_index<P>(b, i, a.width_p)]; };
  // Unrolled so that the loads of several iterations are in flight together (the sums keep
  // their order).
  float s = 0.f;
#pragma unroll 8
  for (int i = lane; i < a.width; i += 64) s += xb(i) * xb(i);
  const float scale = 1.0f / sqrtf(wave_total(s) / (float)a.width + a.epsilon);
  float acc = 0.f;
#pragma unroll 8
  for (int i = lane; i < a.width; i += 64) {
    const float wn = batch_weight<P>(a.weights, a.w_final_norm, i), ws = batch_weight<P>(a.weights, a.w_score, i);
    acc += ws * cast<P>(xb(i) * scale * wn);
  }
  acc = wave_total(acc);
  if (lane == 0) {
    a.score[b] = acc;
    a.position[b] = a.position[b] + 1;
  }
}

// Rows row0 .. row0 + rows - 1 of a step's events, [streams][features] in host memory mapped into
// the device, into the padded input block in the projections' operand layout. A thread per four
// columns: a wave reads up to 1 KB contiguous across PCIe, every piece in one round trip.
// Padding columns stay zero.
template <int P>
__global__ __launch_bounds__(256) void batch_stage(const float* __restrict__ events, float* __restrict__ in, int row0,
                                                   int rows, int features, int features_p) {
  const int per_row = (features + 3) / 4, i = (int)(blockIdx.x * 256 + threadIdx.x);
  if (i >= rows * per_row) return;
  const int b = row0 + i / per_row, k = i % per_row * 4;
  const float* src = events + (size_t)b * features + k;
  f4v v = {0.f, 0.f, 0.f, 0.f};
  if (features % 4 == 0) {
    v = gload16f(src);
  } else {
#pragma unroll
    for (int j = 0; j < 4; j++)
      if (k + j < features) v[j] = src[j];
  }
  *in_global(reinterpret_cast<f4v*>(in + act_index<P>(b, k, features_p))) = v;
}

// Zero the state of stream `stream` (every stream when negative): K/V rows, hidden, position.
// `block_words` is one (layer, stream) block of the K (or V) ring, [H][W][dh], in 4-byte words;
// a stream's K/V is one such block in each layer (the rings are layer-major).
static __global__ void batch_reset(const BatchArgs* __restrict__ ap, int stream, size_t block_words) {
  const BatchArgs& a = *ap;
  const int b0 = stream < 0 ? 0 : stream, b1 = stream < 0 ? a.streams : stream + 1;
  const size_t tid = (size_t)blockIdx.x * blockDim.x + threadIdx.x, step = (size_t)gridDim.x * blockDim.x;
  unsigned* k = reinterpret_cast<unsigned*>(a.keys);
  unsigned* v = reinterpret_cast<unsigned*>(a.values);
  const size_t span = (size_t)(b1 - b0) * block_words;  // the streams' words in one layer
  for (size_t i = tid; i < (size_t)a.layers * span; i += step) {
    const size_t l = i / span, j = ((size_t)l * a.streams + b0) * block_words + i % span;
    k[j] = 0u;
    v[j] = 0u;
  }
  const size_t hper = (size_t)a.layers * a.width;
  for (size_t i = (size_t)b0 * hper + tid; i < (size_t)b1 * hper; i += step) a.hidden[i] = 0.f;
  if (tid == 0)
    for (int b = b0; b < b1; b++) a.position[b] = 0;
}

}  // namespace stamd
