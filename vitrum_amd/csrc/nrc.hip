// nrc.hip -- fused BF16 MFMA kernels of the neural radiance cache.
//
// Network (Mueller et al. 2021, Real-time Neural Radiance Caching): encoded
// input x (64) -> H1..H4 = ReLU(W_l H_{l-1}) (64 wide) -> y = W4 H4 (RGB).
// Input encoding (walkaround-hybrid src/neural/nrc/nrcEncoding.ts): a
// multiresolution hash grid of the position with trainable feature tables
// (Instant-NGP), one-blob bins of the octahedral direction, raw surface
// features.  The tables receive d loss / d input through W0^T, scattered with
// the trilinear weights.
// Loss: relative L2 of walkaround-hybrid/src/neural/nrc/wgsl/fusedMlp.wgsl.ts
// :65-120 (luminance of the prediction as a stop-gradient denominator,
// epsilon 1e-2); Adam as in walkaround-hybrid/src/neural/nrc/
// fusedMlpTrainer.ts:30-84 (FP32 master weights, bf16 copies for the MFMAs).
//
// MFMA formulation.  Every layer is computed transposed, H_out^T = W H_in^T,
// with v_mfma_f32_16x16x32_bf16: A = 16 output neurons x 32 inputs of W,
// B = 32 inputs x 16 samples of H_in^T, C = 16 neurons x 16 samples.  A lane
// (g = lane / 16, r = lane % 16) of C holds neurons 4g..4g+3 of sample r.  The
// 32-wide K of each MFMA step kb is permuted so that lane (g, r) supplies
// inputs {32kb + 4g + j} and {32kb + 16 + 4g + j}, j < 4 -- exactly the values
// the same lane holds in the C tiles of neuron blocks 2kb and 2kb + 1 of the
// previous layer.  Activations therefore pass from layer to layer in
// registers (ReLU, bf16 rounding), with no LDS round trip; the weight
// fragments are packed in the same permuted order.  Backward uses W^T the same
// way.  Weight gradients dW = dH^T H need the sample dimension as K; those
// operands are staged transposed ([neuron][sample]) in LDS.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>

#include "fast_div.h"
#include "nrc.h"

namespace vtn {

typedef __bf16 bf16x8 __attribute__((__vector_size__(8 * sizeof(__bf16))));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef float f32x4 __attribute__((__vector_size__(4 * sizeof(float))));

__device__ __forceinline__ f32x4 mfma(bf16x8 a, bf16x8 b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

__device__ __forceinline__ bf16x8 frag_of(uint4 q) { return __builtin_bit_cast(bf16x8, q); }

// Eight values in bf16, rounded to nearest even two at a time by the
// conversion instruction (the rounding written out in integers took 6
// instructions a value, a third of the inference kernel).
__device__ __forceinline__ uint32_t pack2(float a, float b) {
  return __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2{a, b}, bf16x2));
}
__device__ __forceinline__ uint4 pack8(const float* v) {
  return make_uint4(pack2(v[0], v[1]), pack2(v[2], v[3]), pack2(v[4], v[5]), pack2(v[6], v[7]));
}

// max(x, 0); 0 for a NaN.
__device__ __forceinline__ float relu(float x) { return fmaxf(x, 0.0f); }

// Input neuron of element t (0..7) of lane group g in K step kb.
__host__ __device__ __forceinline__ uint32_t nmap(uint32_t kb, uint32_t g, uint32_t t) {
  return (2u * kb + (t >> 2)) * 16u + g * 4u + (t & 3u);
}

// ---- input encoding (nrcEncoding.ts) --------------------------------------

// The encoding's binary32 operations are those of its definition, in its order
// and each rounded once, so that a cached radiance does not depend on how the
// work is laid out.

// a / b, correctly rounded, from the refined reciprocal y of b: div_by
// (fast_div.h) without the step for operands at the ends of the range.
__device__ __forceinline__ float quotient(float a, float b, float y) {
  float q = a * y;
  q = __builtin_fmaf(__builtin_fmaf(-b, q, a), y, q);
  return __builtin_fmaf(__builtin_fmaf(-b, q, a), y, q);
}

// Instant-NGP spatial hash (nrcEncoding.ts:spatialHash3D): XOR of the corner
// coordinates times 1, 2654435761 and 805459861 (32-bit wraparound), modulo
// the row count (a power of two).  `at` are byte offsets of the rows in the
// level's table (the products are taken eight times as large, a row is 8
// bytes).
struct Corners {
  uint32_t at[8];
  float w[8];
};
constexpr uint32_t kRowBytes = kLevelFeat * 4u, kLevelBytes = kRows * kRowBytes;

// Trilinear corners of level l for a normalised position.
__device__ __forceinline__ void grid_corners(uint32_t l, float nx, float ny, float nz, Corners& c) {
  const float res = (float)(kMinRes << l);
  const float px = nx * res, py = ny * res, pz = nz * res;
  const float x0 = floorf(px), y0 = floorf(py), z0 = floorf(pz);
  const float fx = px - x0, fy = py - y0, fz = pz - z0;
  const uint32_t hx = (uint32_t)x0 * kRowBytes, hy = (uint32_t)y0 * (2654435761u * kRowBytes),
                 hz = (uint32_t)z0 * (805459861u * kRowBytes);
#pragma unroll
  for (uint32_t k = 0; k < 8; ++k) {
    const uint32_t cx = k & 1u, cy = (k >> 1) & 1u, cz = (k >> 2) & 1u;
    const float wx = cx ? fx : 1.0f - fx, wy = cy ? fy : 1.0f - fy, wz = cz ? fz : 1.0f - fz;
    c.w[k] = (wx * wy) * wz;
    c.at[k] = ((hx + cx * kRowBytes) ^ (hy + cy * (2654435761u * kRowBytes)) ^ (hz + cz * (805459861u * kRowBytes))) &
              (kLevelBytes - kRowBytes);
  }
}

// octEncodeDir (nrcEncoding.ts): octahedral map of a direction to [0,1]^2.
__device__ __forceinline__ void oct_encode(float dx, float dy, float dz, float& u, float& v) {
  const float sc = fmaxf(fabsf(dx), fmaxf(fabsf(dy), fabsf(dz)));
  if (!(sc > 0.0f) || !(sc <= 3.402823e38f)) {
    u = v = 0.5f;
    return;
  }
  float sx, sy, sz;
  const uint32_t key = min(min(vtd::div_key(dx), vtd::div_key(dy)), vtd::div_key(dz));
  if (__builtin_expect(vtd::div_den(sc) && key >= vtd::kDivNum, 1)) {
    const float y = vtd::recip_of(sc);
    sx = quotient(dx, sc, y), sy = quotient(dy, sc, y), sz = quotient(dz, sc, y);
  } else {
    sx = dx / sc, sy = dy / sc, sz = dz / sc;
  }
  const float s = (fabsf(sx) + fabsf(sy)) + fabsf(sz);  // in [1, 3]
  const float inv = quotient(1.0f, s, vtd::recip_of(s));
  float px = sx * inv, py = sy * inv;
  if (sz < 0.0f) {
    const float ox = 1.0f - fabsf(py), oy = 1.0f - fabsf(px);
    px = px >= 0.0f ? ox : -ox;
    py = py >= 0.0f ? oy : -oy;
  }
  u = px * 0.5f + 0.5f;
  v = py * 0.5f + 0.5f;
}

// Four of the eight one-blob bins of a scalar (oneBlobEncodeScalar: Gaussian
// kernels at (i + 0.5) / k, sigma 1/k, normalised to unit L1 over the k
// bins): the lower or the upper four.  Lane groups 0 and 1 hold the halves of
// u and 2 and 3 those of v, for the same samples, and exchange them.
__device__ __forceinline__ void one_blob4(float x, uint32_t upper, float* out) {
  const float uc = fminf(fmaxf(x, 0.0f), 1.0f);
  const float c0 = upper ? 4.5f : 0.5f;
  float lower[4], higher[4];
#pragma unroll
  for (uint32_t i = 0; i < 4; ++i) {
    const float d = __builtin_fmaf(uc, (float)kBlobBins, -(c0 + (float)i));  // (uc - centre) * k
    out[i] = expf(-0.5f * (d * d));
    // rows of 16 lanes 0 <-> 1 and 2 <-> 3
    const uint32_t w = __float_as_uint(out[i]);
    const auto rows = __builtin_amdgcn_permlane16_swap(w, w, false, false);
    lower[i] = __uint_as_float(rows[0]), higher[i] = __uint_as_float(rows[1]);
  }
  float sum = 0.0f;
#pragma unroll
  for (uint32_t i = 0; i < 4; ++i) sum += lower[i];
#pragma unroll
  for (uint32_t i = 0; i < 4; ++i) sum += higher[i];
  // From 1.25 (x = 0 or 1, where half of the Gaussian is cut off) to 2.51, and
  // a bin is at least e^-28.2: every quotient is in the normal range.
  const float y = vtd::recip_of(sum);
#pragma unroll
  for (uint32_t i = 0; i < 4; ++i) out[i] = quotient(out[i], sum, y);
}

// The 16 encoded inputs a lane of group g supplies for one sample, in the
// K order of nmap: kb 0 -> dims {4g..4g+3, 16+4g..16+4g+3}, kb 1 -> dims
// {32+4g..32+4g+3, 48+4g..48+4g+3}.  Lane group g owns hash-grid levels 2g
// and 2g + 1.  All four lanes of a sample take part.
// Levels kLdsFirstLevel.. of the tables are read from a workgroup copy in LDS
// when `lds` is given (the inference kernel stages them: their rows are hit
// at random, while the coarse levels' few rows stay in the caches).
constexpr uint32_t kLdsFirstLevel = 3;
constexpr uint32_t kInferBlock = 1024;
constexpr uint32_t kLdsRows = (kLevels - kLdsFirstLevel) * kRows;  // 20,480 float2 = 160 KiB

// A row of the copy, through an LDS pointer: with a generic one the compiler
// folds the two kinds of gather into flat loads.
typedef const __attribute__((address_space(3))) char* lds_bytes;
__device__ __forceinline__ float2 lds_row(const float2* lds, uint32_t at) {
  const auto q = reinterpret_cast<const __attribute__((address_space(3))) f32x2*>((lds_bytes)lds + at);
  const f32x2 v = *q;
  return make_float2(v[0], v[1]);
}

__device__ __forceinline__ void add_row(float2 t, float w, float& f0, float& f1) {
  f0 += w * t.x;
  f1 += w * t.y;
}

__device__ __forceinline__ void encode_lane(uint32_t g, const float* f, const float* __restrict__ tables,
                                            float (&v)[2][8], const float2* lds = nullptr) {
  // hash grid, levels 2g, 2g + 1
#pragma unroll
  for (uint32_t j = 0; j < 2; ++j) {
    Corners c;
    const uint32_t level = 2u * g + j;
    grid_corners(level, f[0], f[1], f[2], c);
    float f0 = 0.0f, f1 = 0.0f;
    if (lds && level >= kLdsFirstLevel) {
      const uint32_t first = (level - kLdsFirstLevel) * kLevelBytes;
#pragma unroll
      for (uint32_t k = 0; k < 8; ++k) add_row(lds_row(lds, c.at[k] | first), c.w[k], f0, f1);
    } else {
      const char* rows = reinterpret_cast<const char*>(tables);
      const uint32_t first = level * kLevelBytes;
#pragma unroll
      for (uint32_t k = 0; k < 8; ++k)
        add_row(*reinterpret_cast<const float2*>(rows + (c.at[k] | first)), c.w[k], f0, f1);
    }
    v[0][2 * j] = f0;
    v[0][2 * j + 1] = f1;
  }
  // one-blob of the direction: groups 0, 1 -> u bins 0-3, 4-7; groups 2, 3 -> v
  float ou, ov;
  oct_encode(f[3], f[4], f[5], ou, ov);
  one_blob4(g < 2u ? ou : ov, g & 1u, &v[0][4]);
  // raw features: dims 32-34 normal, 35 roughness, 36-38 albedo
#pragma unroll
  for (uint32_t t = 0; t < 8; ++t) v[1][t] = 0.0f;
  v[1][0] = g == 0u ? f[6] : (g == 1u ? f[10] : 0.0f);
  v[1][1] = g == 0u ? f[7] : (g == 1u ? f[11] : 0.0f);
  v[1][2] = g == 0u ? f[8] : (g == 1u ? f[12] : 0.0f);
  v[1][3] = g == 0u ? f[9] : 0.0f;
}

// ---- packing: FP32 master weights -> permuted bf16 fragments --------------

__global__ void pack_kernel(const float* __restrict__ w, uint4* __restrict__ frags) {
  const uint32_t id = blockIdx.x * blockDim.x + threadIdx.x;  // one fragment (lane) each
  if (id >= kFrags) return;
  const uint32_t lane = id & 63u, g = lane >> 4, r = lane & 15u;
  float v[8];
  if (id < kHidden * kFragsHidden) {
    // forward, hidden layer l: A = W_l, row o = ob*16 + r, k = nmap(kb, g, t)
    const uint32_t l = id / kFragsHidden, rem = id % kFragsHidden;
    const uint32_t ob = rem / 128u, kb = (rem / 64u) & 1u;
    for (uint32_t t = 0; t < 8; ++t) v[t] = w[l * 4096u + (ob * 16u + r) * 64u + nmap(kb, g, t)];
  } else if (id < kFragsFwd) {
    // forward, output layer: rows 0..2 of W4, zero padding to 16 rows
    const uint32_t kb = ((id - kHidden * kFragsHidden) / 64u) & 1u;
    for (uint32_t t = 0; t < 8; ++t) v[t] = r < kOut ? w[16384u + r * 64u + nmap(kb, g, t)] : 0.0f;
  } else if (id >= kFragsFwd + kFragsBwd) {
    // input gradient of dims 0..15: A = W0^T, row i = r, k = output neuron
    const uint32_t kb = ((id - kFragsFwd - kFragsBwd) / 64u) & 1u;
    for (uint32_t t = 0; t < 8; ++t) v[t] = w[nmap(kb, g, t) * 64u + r];
  } else {
    // backward through W_m (m = 1..4): A = W_m^T, row i = ib*16 + r, k = output neuron
    const uint32_t b = id - kFragsFwd;
    const uint32_t m = 1u + b / kFragsHidden, rem = b % kFragsHidden;
    const uint32_t ib = rem / 128u, kb = (rem / 64u) & 1u;
    const uint32_t i = ib * 16u + r;
    for (uint32_t t = 0; t < 8; ++t) {
      const uint32_t o = nmap(kb, g, t);
      if (m < 4u)
        v[t] = w[m * 4096u + o * 64u + i];
      else
        v[t] = (kb == 0u && o < kOut) ? w[16384u + o * 64u + i] : 0.0f;
    }
  }
  frags[id] = pack8(v);
}

// ---- shared forward ------------------------------------------------------------

// Builds the B fragments of the encoded inputs of 4 sample blocks.
__device__ __forceinline__ void encode_tile(const float* __restrict__ feats, const float* __restrict__ tables,
                                            uint32_t n, uint32_t base, uint32_t g, uint32_t r, uint4 (&B)[4][2],
                                            const float2* lds = nullptr) {
#pragma unroll
  for (uint32_t sb = 0; sb < 4; ++sb) {
    uint32_t s = min(base + sb * 16u + r, n - 1u);  // past the end: the last sample again
    float v[2][8], f[kFeat];
    const float4* fp = reinterpret_cast<const float4*>(feats + (size_t)s * kFeat);
#pragma unroll
    for (uint32_t q = 0; q < 4; ++q) {
      const float4 x = fp[q];
      f[4 * q] = x.x, f[4 * q + 1] = x.y, f[4 * q + 2] = x.z, f[4 * q + 3] = x.w;
    }
    encode_lane(g, f, tables, v, lds);
    B[sb][0] = pack8(v[0]);
    B[sb][1] = pack8(v[1]);
    // packed here: sunk past the branches of the next block's encoding, the
    // sixteen unpacked values would wait in registers that then spill
#pragma unroll
    for (uint32_t kb = 0; kb < 2; ++kb)
      asm volatile("" : "+v"(B[sb][kb].x), "+v"(B[sb][kb].y), "+v"(B[sb][kb].z), "+v"(B[sb][kb].w));
  }
}

// One hidden layer: B (inputs) -> B (ReLU outputs, bf16).
__device__ __forceinline__ void hidden_layer(const uint4* __restrict__ frags, uint32_t lane,
                                             uint4 (&B)[4][2]) {
  f32x4 C[4][4];
#pragma unroll
  for (uint32_t ob = 0; ob < 4; ++ob)
#pragma unroll
    for (uint32_t sb = 0; sb < 4; ++sb) C[ob][sb] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
  for (uint32_t ob = 0; ob < 4; ++ob)
#pragma unroll
    for (uint32_t kb = 0; kb < 2; ++kb) {
      const bf16x8 a = frag_of(frags[(ob * 2u + kb) * 64u + lane]);
#pragma unroll
      for (uint32_t sb = 0; sb < 4; ++sb) C[ob][sb] = mfma(a, frag_of(B[sb][kb]), C[ob][sb]);
    }
#pragma unroll
  for (uint32_t sb = 0; sb < 4; ++sb)
#pragma unroll
    for (uint32_t kb = 0; kb < 2; ++kb) {
      float v[8];
#pragma unroll
      for (uint32_t t = 0; t < 8; ++t) {
        v[t] = relu(C[2u * kb + (t >> 2)][sb][t & 3u]);
      }
      B[sb][kb] = pack8(v);
    }
}

__device__ __forceinline__ void output_layer(const uint4* __restrict__ frags, uint32_t lane,
                                             const uint4 (&B)[4][2], f32x4 (&Y)[4]) {
#pragma unroll
  for (uint32_t sb = 0; sb < 4; ++sb) Y[sb] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
  for (uint32_t kb = 0; kb < 2; ++kb) {
    const bf16x8 a = frag_of(frags[kHidden * kFragsHidden + kb * 64u + lane]);
#pragma unroll
    for (uint32_t sb = 0; sb < 4; ++sb) Y[sb] = mfma(a, frag_of(B[sb][kb]), Y[sb]);
  }
}

// ---- inference: one wave = 64 samples -------------------------------------------
//
// Persistent: one 1024-thread workgroup per CU copies levels 3-7 of the
// tables (160 KiB) into LDS once, then each of its 16 waves takes tiles of 64
// samples, grid-strided.  The encoding reads the same f32 table values as from
// memory, so the outputs are those of a direct gather.
//
// Bound by VALU issue, with the LDS gathers and MFMAs behind it: a tile takes
// 2,370 vector instructions beside 136 MFMAs (4,550 with the bf16 rounding
// written out, eight exponentials a lane and flat gathers; 2,080 and 3 to 5%
// less time with fused grid sums, a quotient corrected once and a shorter
// exponential, which changed the last bits of what the cache answers).
// 2,073,600 samples: 286 -> 185 us.  Blocks of 512 threads (twice the
// registers, two waves per SIMD) took 217 us where these took 180.

__global__ __launch_bounds__(kInferBlock) void infer_kernel(const float* __restrict__ feats, uint32_t cap,
                                                     const uint32_t* __restrict__ n_ptr,
                                                     const uint4* __restrict__ frags,
                                                     const float* __restrict__ tables, float* __restrict__ rgb) {
  __shared__ __align__(16) float2 tab[kLdsRows];
  {
    // all of a thread's loads in flight at once
    constexpr uint32_t kLoads = kLdsRows / 2u / kInferBlock;
    const float4* src = reinterpret_cast<const float4*>(tables + 2u * kLdsFirstLevel * kRows) + threadIdx.x;
    float4 q[kLoads];
#pragma unroll
    for (uint32_t i = 0; i < kLoads; ++i) q[i] = src[i * kInferBlock];
#pragma unroll
    for (uint32_t i = 0; i < kLoads; ++i) reinterpret_cast<float4*>(tab)[threadIdx.x + i * kInferBlock] = q[i];
  }
  __syncthreads();
  const uint32_t n = n_ptr ? min(*n_ptr, cap) : cap;
  const uint32_t lane = threadIdx.x & 63u, g = lane >> 4, r = lane & 15u;
  const uint32_t tiles = (n + 63u) / 64u, waves = gridDim.x * (kInferBlock / 64u);
  for (uint32_t tile = blockIdx.x * (kInferBlock / 64u) + (threadIdx.x >> 6); tile < tiles; tile += waves) {
    const uint32_t base = tile * 64u;
    // re-read the fragments every tile (an opaque offset keeps them from
    // being hoisted out of the loop into spilled registers; an opaque pointer
    // would make the loads flat ones)
    uint32_t zero = 0;
    asm volatile("" : "+s"(zero));
    const uint4* fw = frags + zero;
    uint4 B[4][2];
    encode_tile(feats, tables, n, base, g, r, B, tab);
#pragma unroll
    for (uint32_t l = 0; l < kHidden; ++l) {
      hidden_layer(fw + l * kFragsHidden, lane, B);
    }
    f32x4 Y[4];
    output_layer(fw, lane, B, Y);
    if (g == 0u) {
#pragma unroll
      for (uint32_t sb = 0; sb < 4; ++sb) {
        const uint32_t s = base + sb * 16u + r;
        if (s < n) {
          rgb[3 * (size_t)s] = Y[sb][0];
          rgb[3 * (size_t)s + 1] = Y[sb][1];
          rgb[3 * (size_t)s + 2] = Y[sb][2];
        }
      }
    }
  }
}

// ---- training: forward, relative-L2 gradient, backward, dW ------------------------
//
// A workgroup of four waves trains on tiles of 64 samples; wave w owns the
// samples w*16 .. w*16+15 of a tile (one 16-column block of every MFMA), so a
// wave's activations are 2 fragments per layer.  The layer inputs are staged
// transposed ([neuron][sample], bf16) in the workgroup's LDS for the weight
// gradients, dW = D^T H over the tile's 64 samples, which wave w computes for
// output rows w*16 .. w*16+15 into accumulators that stay in registers across
// all of the workgroup's tiles; they are written to the workgroup's slot once.
//
// Bound by the latency of the chain of layers (fragments from L2, MFMA, bf16,
// LDS, barrier): two workgroups per CU with 256 registers a lane, so that the
// compiler fetches the next layer's fragments early, beat three with 168 by a
// third; 262,144 samples 149 -> 99 us.  A second copy of the deltas in LDS,
// which saves four of the ten barriers, gives nothing more.

constexpr uint32_t kTile = 64u * 64u;  // one transposed [neuron][sample] bf16 tile

// Encoded inputs of sample s for lane group g (zero past n).
__device__ __forceinline__ void encode_block(const float* __restrict__ feats, const float* __restrict__ tables,
                                             uint32_t n, uint32_t s, uint32_t g, uint4 (&B)[2]) {
  float v[2][8];
  if (s < n) {
    float f[kFeat];
    const float4* fp = reinterpret_cast<const float4*>(feats + (size_t)s * kFeat);
#pragma unroll
    for (uint32_t q = 0; q < 4; ++q) {
      const float4 x = fp[q];
      f[4 * q] = x.x, f[4 * q + 1] = x.y, f[4 * q + 2] = x.z, f[4 * q + 3] = x.w;
    }
    encode_lane(g, f, tables, v);
  } else {
#pragma unroll
    for (uint32_t t = 0; t < 8; ++t) v[0][t] = v[1][t] = 0.0f;
  }
  B[0] = pack8(v[0]);
  B[1] = pack8(v[1]);
}

// One hidden layer of one 16-sample block: B -> ReLU(W B) in bf16; returns
// the positive-output mask (bit kb*8 + t).
__device__ __forceinline__ uint32_t hidden_block(const uint4* __restrict__ frags, uint32_t lane, uint4 (&B)[2]) {
  f32x4 C[4];
#pragma unroll
  for (uint32_t ob = 0; ob < 4; ++ob) C[ob] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
  for (uint32_t ob = 0; ob < 4; ++ob)
#pragma unroll
    for (uint32_t kb = 0; kb < 2; ++kb) C[ob] = mfma(frag_of(frags[(ob * 2u + kb) * 64u + lane]), frag_of(B[kb]), C[ob]);
  uint32_t mask = 0;
#pragma unroll
  for (uint32_t kb = 0; kb < 2; ++kb) {
    float v[8];
#pragma unroll
    for (uint32_t t = 0; t < 8; ++t) {
      v[t] = relu(C[2u * kb + (t >> 2)][t & 3u]);
      // positive: the bits as an integer, clamped to [0, 1]
      mask |= (uint32_t)min(max((int)__float_as_uint(v[t]), 0), 1) << (kb * 8u + t);
    }
    B[kb] = pack8(v);
  }
  return mask;
}

// Inference of a few samples: one wave takes one block of 16 and gathers from
// memory, without the copy of the tables: bound by the latency of one wave's
// chain, where the copy and 16 tiles on one CU took 31 us (see kFewSamples).
__global__ __launch_bounds__(64) void infer_few_kernel(const float* __restrict__ feats, uint32_t cap,
                                                       const uint32_t* __restrict__ n_ptr,
                                                       const uint4* __restrict__ frags,
                                                       const float* __restrict__ tables, float* __restrict__ rgb) {
  const uint32_t n = n_ptr ? min(*n_ptr, cap) : cap;
  const uint32_t lane = threadIdx.x, g = lane >> 4, s = blockIdx.x * 16u + (lane & 15u);
  if (blockIdx.x * 16u >= n) return;
  uint4 B[2];
  encode_block(feats, tables, n, s, g, B);
#pragma unroll
  for (uint32_t l = 0; l < kHidden; ++l) (void)hidden_block(frags + l * kFragsHidden, lane, B);
  f32x4 Y = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
  for (uint32_t kb = 0; kb < 2; ++kb)
    Y = mfma(frag_of(frags[kHidden * kFragsHidden + kb * 64u + lane]), frag_of(B[kb]), Y);
  if (g == 0u && s < n) {
    rgb[3 * (size_t)s] = Y[0];
    rgb[3 * (size_t)s + 1] = Y[1];
    rgb[3 * (size_t)s + 2] = Y[2];
  }
}

// Backward through W_m^T for one block: dH = (W_m^T dNext) masked by ReLU'.
__device__ __forceinline__ void backward_block(const uint4* __restrict__ fr, uint32_t lane, uint32_t kbs,
                                               uint32_t mask, uint4 (&B)[2]) {
  f32x4 C[4];
#pragma unroll
  for (uint32_t ib = 0; ib < 4; ++ib) C[ib] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
  for (uint32_t ib = 0; ib < 4; ++ib)
    for (uint32_t kb = 0; kb < kbs; ++kb) C[ib] = mfma(frag_of(fr[(ib * 2u + kb) * 64u + lane]), frag_of(B[kb]), C[ib]);
#pragma unroll
  for (uint32_t kb = 0; kb < 2; ++kb) {
    float v[8];
#pragma unroll
    for (uint32_t t = 0; t < 8; ++t) {
      const uint32_t keep = (uint32_t)((int)(mask << (31u - (kb * 8u + t))) >> 31);
      v[t] = __uint_as_float(__float_as_uint(C[2u * kb + (t >> 2)][t & 3u]) & keep);
    }
    B[kb] = pack8(v);
  }
}

// Where a lane reads and writes a transposed tile.  A row (64 samples, 16-byte
// chunks of 8) is half of the LDS banks long, so a row's chunks are permuted
// by bits 1..3 of its number: the 16 rows that one fragment read takes from a
// chunk, and the four rows that a store's lane groups write, then fall on
// different banks (in order they took 8 and 4 turns).  Two neighbouring
// samples share a dword: the even lane writes the pair's dword of one neuron
// and the odd lane that of the next.
struct TileAt {
  uint32_t write[2];  // rows 4g + (r & 1) and 4g + 2 + (r & 1), this wave's columns
  uint32_t read;      // row r, samples 8g..; samples 32 + 8g.. at read ^ 32
  uint32_t sel;
};
__device__ __forceinline__ uint32_t chunk_at(uint32_t n, uint32_t c) {
  return (c ^ ((((n >> 2) & 3u) << 1) | ((n >> 1) & 1u))) * 8u;
}
__device__ __forceinline__ TileAt tile_at(uint32_t w, uint32_t g, uint32_t r) {
  const uint32_t c = 2u * w + (r >> 3), n = 4u * g;
  return TileAt{{(n + (r & 1u)) * 64u + chunk_at(n, c) + (r & 6u),
                 (n + 2u + (r & 1u)) * 64u + chunk_at(n + 2u, c) + (r & 6u)},
                r * 64u + chunk_at(r, g),
                r & 1u ? 0x03020706u : 0x05040100u};
}

// Stores a block's fragments transposed into the wave's columns.
__device__ __forceinline__ void store_block(uint16_t* T, const TileAt& at, const uint4 (&B)[2]) {
#pragma unroll
  for (uint32_t kb = 0; kb < 2; ++kb) {
    const uint32_t q[4] = {B[kb].x, B[kb].y, B[kb].z, B[kb].w};
#pragma unroll
    for (uint32_t p = 0; p < 4; ++p) {
      const uint32_t other = (uint32_t)__builtin_amdgcn_mov_dpp((int)q[p], 0xB1, 0xF, 0xF, true);  // lane ^ 1
      *reinterpret_cast<uint32_t*>(T + at.write[p & 1u] + (2u * kb + (p >> 1)) * 1024u) =
          __builtin_amdgcn_perm(other, q[p], at.sel);
    }
  }
}

// Row n16 * 16 + r, the lane's eight samples of K step ks.
__device__ __forceinline__ bf16x8 tile_frag(const uint16_t* T, const TileAt& at, uint32_t n16, uint32_t ks) {
  return frag_of(*reinterpret_cast<const uint4*>(T + (at.read ^ (ks * 32u)) + n16 * 1024u));
}

// acc[ib] += D^T H for output rows ob*16.. (A from DT) and input columns
// ib*16.. (B from HT), K = the tile's 64 samples.
__device__ __forceinline__ void weight_grad_rows(const uint16_t* DT, const uint16_t* HT, const TileAt& at, uint32_t ob,
                                                 f32x4 (&acc)[4]) {
#pragma unroll
  for (uint32_t ks = 0; ks < 2; ++ks) {
    const bf16x8 a = tile_frag(DT, at, ob, ks);
#pragma unroll
    for (uint32_t ib = 0; ib < 4; ++ib) acc[ib] = mfma(a, tile_frag(HT, at, ib, ks), acc[ib]);
  }
}

__global__ __launch_bounds__(256, 2) void train_kernel(const float* __restrict__ feats, const float* __restrict__ targets,
                                                    uint32_t cap, const uint32_t* __restrict__ n_ptr,
                                                    const uint4* __restrict__ frags, const float* __restrict__ tables,
                                                    float* __restrict__ partials, float* __restrict__ dx,
                                                    float* __restrict__ loss) {
  const uint32_t n = n_ptr ? min(*n_ptr, cap) : cap;
  const uint32_t tiles = (n + 63u) / 64u;
  __shared__ __align__(16) uint16_t HT[5 * kTile];  // inputs of W0..W4, transposed
  __shared__ __align__(16) uint16_t DT[kTile];      // deltas, transposed
  const uint32_t lane = threadIdx.x & 63u, w = threadIdx.x >> 6, g = lane >> 4, r = lane & 15u;
  const TileAt at = tile_at(w, g, r);
  f32x4 acc[kHidden][4];  // dW_0..dW_3, rows w*16.., all 64 inputs
  f32x4 acc_out;          // dW_4 (rows 0..2 of a 16-row block), inputs w*16..
#pragma unroll
  for (uint32_t m = 0; m < kHidden; ++m)
#pragma unroll
    for (uint32_t ib = 0; ib < 4; ++ib) acc[m][ib] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  acc_out = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  float part = 0.0f;
  // Tiles of 64 samples, strided over the workgroups (uniform loop bounds).
  for (uint32_t tile = blockIdx.x; tile < tiles; tile += gridDim.x) {
    const uint32_t s = tile * 64u + w * 16u + r;
    // The fragments are re-read from the cache every tile: an opaque offset
    // keeps the compiler from hoisting all 68 KB of them out of the loop into
    // (spilled) registers.
    uint32_t zero = 0;
    asm volatile("" : "+s"(zero));
    const uint4* fw = frags + zero;
    const uint4* bw = fw + kFragsFwd;
    __syncthreads();  // the previous tile's last reads of HT/DT
    uint4 B[2];
    uint32_t mask[kHidden];
    encode_block(feats, tables, n, s, g, B);
    store_block(HT, at, B);
#pragma unroll
    for (uint32_t l = 0; l < kHidden; ++l) {
      mask[l] = hidden_block(fw + l * kFragsHidden, lane, B);
      store_block(HT + (l + 1u) * kTile, at, B);
    }
    f32x4 Y = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (uint32_t kb = 0; kb < 2; ++kb)
      Y = mfma(frag_of(fw[kHidden * kFragsHidden + kb * 64u + lane]), frag_of(B[kb]), Y);

    // Relative L2 (fusedMlp.wgsl.ts:65-120): d/dy = 2 (y - t) / (3 n (L^2 + eps)),
    // L = luminance of the prediction, normalised by its largest component.
    // Lanes of group 0 hold outputs 0..2 of their sample.
    float d[8] = {0, 0, 0, 0, 0, 0, 0, 0};
    if (g == 0u && s < n) {
      const float p0 = Y[0], p1 = Y[1], p2 = Y[2];
      const float t0 = targets[3 * (size_t)s], t1 = targets[3 * (size_t)s + 1], t2 = targets[3 * (size_t)s + 2];
      const float sc = fmaxf(fabsf(p0), fmaxf(fabsf(p1), fabsf(p2)));
      float lum = 0.0f;
      if (sc > 0.0f) {
        const float nl = (0.299f * (p0 / sc) + 0.587f * (p1 / sc)) + 0.114f * (p2 / sc);
        lum = fminf(fmaxf(nl, -1.0f), 1.0f) * sc;
      }
      const float bl = fminf(fabsf(lum), 1e19f);
      const float den = bl * bl + 1e-2f;
      const float inv = 2.0f / (float)n / 3.0f / den;
      const float p[3] = {p0, p1, p2}, tg[3] = {t0, t1, t2};
#pragma unroll
      for (uint32_t c = 0; c < 3; ++c) {
        const float e = p[c] - tg[c];
        float x = e * inv;
        x = x != x ? 0.0f : fminf(fmaxf(x, -65504.0f), 65504.0f);
        d[c] = x;
        if (e == e && den == den) part += e * e / den;
      }
    }
    B[0] = pack8(d);
    B[1] = make_uint4(0u, 0u, 0u, 0u);
    // dY^T rows 0..15 of this wave's columns: lane (g, r) writes rows 4g..4g+3
    // (the outputs it holds; rows 3..15 are zero padding).
    {
      const uint32_t q0 = B[0].x, q1 = B[0].y;
#pragma unroll
      for (uint32_t j = 0; j < 4; ++j) {
        const uint32_t bits = g == 0u ? ((j < 2u ? q0 : q1) >> ((j & 1u) * 16u)) & 0xFFFFu : 0u;
        DT[(4u * g + j) * 64u + chunk_at(4u * g + j, 2u * w + (r >> 3)) + (r & 7u)] = (uint16_t)(j < 3u ? bits : 0u);
      }
    }
    __syncthreads();
    // dW4 (rows 0..2 padded to 16) for inputs w*16..: one 16x16 block per wave
#pragma unroll
    for (uint32_t ks = 0; ks < 2; ++ks) {
      acc_out = mfma(tile_frag(DT, at, 0u, ks), tile_frag(HT + 4u * kTile, at, w, ks), acc_out);
    }
    // dH4 through W4^T
    backward_block(bw + 3u * kFragsHidden, lane, 1u, mask[3], B);
#pragma unroll
    for (uint32_t m = 3; m >= 1; --m) {
      __syncthreads();  // every wave's reads of DT are done
      store_block(DT, at, B);  // dH_{m+1} (pre-activation delta of layer m's output)
      __syncthreads();
      weight_grad_rows(DT, HT + m * kTile, at, w, acc[m]);
      backward_block(bw + (m - 1u) * kFragsHidden, lane, 2u, mask[m - 1u], B);
    }
    __syncthreads();
    store_block(DT, at, B);  // dH1
    __syncthreads();
    weight_grad_rows(DT, HT, at, w, acc[0]);
    // d loss / d x of the hash-grid inputs (dims 0..15) = W0^T dH1: lane
    // (g, r) receives dims 4g..4g+3 -- the features of levels 2g, 2g + 1 that
    // it encoded -- of its sample; table_grad_kernel scatters them into the
    // tables with the trilinear weights (hashGridBackward).
    f32x4 X = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (uint32_t kb = 0; kb < 2; ++kb) X = mfma(frag_of(fw[kFragsFwd + kFragsBwd + kb * 64u + lane]), frag_of(B[kb]), X);
    if (s < n) *reinterpret_cast<float4*>(dx + (size_t)s * 16u + 4u * g) = make_float4(X[0], X[1], X[2], X[3]);
  }
  // loss: wave sum, one atomic per wave
  for (uint32_t off = 32; off > 0; off >>= 1) part += __shfl_xor(part, (int)off);
  if (lane == 0 && part != 0.0f) unsafeAtomicAdd(loss, part / (3.0f * (float)n));
  // The workgroup's slot: every element is written by exactly one lane.
  float* __restrict__ slot = partials + (size_t)blockIdx.x * kMlpParams;
#pragma unroll
  for (uint32_t m = 0; m < kHidden; ++m)
#pragma unroll
    for (uint32_t ib = 0; ib < 4; ++ib)
#pragma unroll
      for (uint32_t j = 0; j < 4; ++j) slot[m * 4096u + (w * 16u + g * 4u + j) * 64u + ib * 16u + r] = acc[m][ib][j];
#pragma unroll
  for (uint32_t j = 0; j < 4; ++j)
    if (g * 4u + j < kOut) slot[16384u + (g * 4u + j) * 64u + w * 16u + r] = acc_out[j];
}

// Hash-grid table gradient (hashGridBackward): each input gradient of a
// level's two features, times the trilinear weight of each of the 8 corners,
// accumulates into that corner's row.  One workgroup per (level, chunk of
// samples) sums its chunk into a private copy of the level's 4096 x 2
// gradient in LDS and stores the copy whole into its own partial slice
// (part[(chunk * kLevels + level) * 8192 ..]); table_reduce_kernel then sums
// the chunks' slices.  The LDS copy holds fixed-point integers (2^46 per
// unit): LDS integer atomics run about four times faster than float ones
// here, and integer sums do not depend on the order of the additions.  A
// contribution is clamped to +-4 (far beyond any gradient of a training
// step; 16,384 contributions per element per chunk then stay below 2^63); a
// non-finite one makes the chunk's whole slice NaN, as a float sum would
// carry it, so Adam skips that step for the level.
constexpr float kGradFixClamp = 4.0f;

// v clamped, times 2^46, as a two's complement integer rounded to nearest
// even: the sum with 1.5 * 2^52 has it in its low 52 bits, and taking that
// constant's bits away leaves its sign.
__device__ __forceinline__ unsigned long long grad_fixed(float v) {
  const double x = (double)fminf(fmaxf(v, -kGradFixClamp), kGradFixClamp);
  const double s = __builtin_fma(x, 0x1p46, 0x1.8p52);
  return (unsigned long long)__double_as_longlong(s) - 0x4338000000000000ull;
}

__global__ __launch_bounds__(256) void table_grad_kernel(const float* __restrict__ feats, const float* __restrict__ dx,
                                                         uint32_t cap, const uint32_t* __restrict__ n_ptr,
                                                         uint32_t per_chunk, float* __restrict__ part) {
  __shared__ unsigned long long acc[kRows * kLevelFeat];  // two's complement fixed point
  __shared__ uint32_t nonfinite;
  const uint32_t l = blockIdx.x, tid = threadIdx.x;
  for (uint32_t i = tid; i < kRows * kLevelFeat; i += 256u) acc[i] = 0ull;
  if (tid == 0) nonfinite = 0u;
  __syncthreads();
  const uint32_t n = n_ptr ? min(*n_ptr, cap) : cap;
  const uint32_t lo = blockIdx.y * per_chunk, hi = min(n, lo + per_chunk);
  bool bad = false;
#pragma unroll 2
  for (uint32_t s = lo + tid; s < hi; s += 256u) {
    const float* fp = feats + (size_t)s * kFeat;
    Corners c;
    grid_corners(l, fp[0], fp[1], fp[2], c);
    const float d0 = dx[(size_t)s * 16u + 2u * l], d1 = dx[(size_t)s * 16u + 2u * l + 1u];
    // a weight is not finite only if the position is not, and then none is
    bad = bad || !(fabsf(d0) <= 3.402823e38f) || !(fabsf(d1) <= 3.402823e38f) || c.w[0] != c.w[0];
#pragma unroll
    for (uint32_t k = 0; k < 8; ++k) {
      atomicAdd(&acc[c.at[k] / 4u], grad_fixed(c.w[k] * d0));
      atomicAdd(&acc[c.at[k] / 4u + 1u], grad_fixed(c.w[k] * d1));
    }
  }
  if (bad) nonfinite = 1u;
  __syncthreads();
  float* __restrict__ out = part + ((size_t)blockIdx.y * kLevels + l) * (kRows * kLevelFeat);
  const bool poisoned = nonfinite != 0u;
  for (uint32_t i = tid; i < kRows * kLevelFeat; i += 256u)
    out[i] = poisoned ? __builtin_nanf("") : (float)((double)(long long)acc[i] * (1.0 / 70368744177664.0));
}

// grad[kMlpParams + e] += the sum over the chunks of element e of the
// partial table gradients (one thread per element).
__global__ __launch_bounds__(256) void table_reduce_kernel(const float* __restrict__ part, uint32_t chunks,
                                                           float* __restrict__ tgrad) {
  const uint32_t e = blockIdx.x * 256u + threadIdx.x;
  if (e >= kTableParams) return;
  const uint32_t l = e / (kRows * kLevelFeat), i = e % (kRows * kLevelFeat);
  float sum = 0.0f;
#pragma unroll 8
  for (uint32_t c = 0; c < chunks; ++c) sum += part[((size_t)c * kLevels + l) * (kRows * kLevelFeat) + i];
  tgrad[e] += sum;
}

// grad[i] += sum of the partial MLP weight gradients of the workgroups that
// processed at least one tile; blockIdx.y picks every gridDim.y-th slot.
__global__ __launch_bounds__(256) void reduce_slots_kernel(const float* __restrict__ part, uint32_t slots,
                                                           uint32_t cap, const uint32_t* __restrict__ n_ptr,
                                                           float* __restrict__ grad) {
  const uint32_t i = blockIdx.x * 256u + threadIdx.x;
  const uint32_t n = n_ptr ? min(*n_ptr, cap) : cap;
  const uint32_t used = min(slots, (n + 63u) / 64u);
  if (i >= kMlpParams) return;
  float acc = 0.0f;
#pragma unroll 8
  for (uint32_t k = blockIdx.y; k < used; k += gridDim.y) acc += part[(size_t)k * kMlpParams + i];
  if (acc != 0.0f) unsafeAtomicAdd(grad + i, acc);
}

// ---- Adam (fusedMlpTrainer.ts:30-84) -------------------------------------------

__device__ __forceinline__ bool finite_(float x) { return x == x && fabsf(x) <= 3.402823e38f; }

__global__ void adam_kernel(float* __restrict__ w, float* __restrict__ grad, float* __restrict__ m,
                            float* __restrict__ v, AdamParams p) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= kParams) return;
  const float cur = w[i], om = m[i], ov = v[i], gr = grad[i];
  grad[i] = 0.0f;
  if (!finite_(cur) || !finite_(om) || !finite_(ov) || ov < 0.0f) {
    w[i] = finite_(cur) ? cur : 0.0f;
    m[i] = 0.0f;
    v[i] = 0.0f;
    return;
  }
  if (!finite_(gr)) return;
  const float mi = p.beta1 * om + (1.0f - p.beta1) * gr;
  const float vi = p.beta2 * ov + (1.0f - p.beta2) * gr * gr;
  const float mhat = mi / p.bc1, vhat = vi / p.bc2;
  if (!finite_(mi) || !finite_(vi) || !finite_(mhat) || !finite_(vhat) || vi < 0.0f || vhat < 0.0f) return;
  const float lr = i < kMlpParams ? p.lr : p.lr_table;
  const float upd = cur - lr * mhat / (sqrtf(vhat) + p.eps);
  if (!finite_(upd)) return;
  m[i] = mi;
  v[i] = vi;
  w[i] = fminf(fmaxf(upd, -65504.0f), 65504.0f);
}

__global__ void fill_kernel(float* p, uint32_t n, float value) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = value;
}

// ---- launchers ----------------------------------------------------------------

hipError_t launch_pack(const float* master, uint4* frags, hipStream_t s) {
  hipLaunchKernelGGL(pack_kernel, dim3((kFrags + 255) / 256), dim3(256), 0, s, master, frags);
  return hipGetLastError();
}

// Up to here infer_few_kernel is the faster one (12.1, 15.2, 30.5 and 51.4 us
// for 4,099, 32,768, 131,072 and 262,144 samples with the host's call, against
// 31.2, 31.6, 32.4 and 34.5 us): its time grows with the samples, the staged
// kernel's hardly before every CU has its sixteen tiles.
constexpr uint32_t kFewSamples = 131072;

hipError_t launch_infer(const float* feats, uint32_t n, const uint32_t* n_ptr, const uint4* frags,
                        const float* tables, float* rgb, hipStream_t s) {
  if (n == 0) return hipSuccess;
  // one workgroup per CU (each holds 160 KiB of LDS), fewer for small batches
  static uint32_t cus = 0;
  if (cus == 0) {
    int dev = 0, c = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e == hipSuccess) e = hipDeviceGetAttribute(&c, hipDeviceAttributeMultiprocessorCount, dev);
    if (e != hipSuccess) return e;
    cus = (uint32_t)std::max(1, c);
  }
  if (n <= kFewSamples) {
    hipLaunchKernelGGL(infer_few_kernel, dim3((n + 15u) / 16u), dim3(64), 0, s, feats, n, n_ptr, frags, tables, rgb);
    return hipGetLastError();
  }
  const uint32_t tiles = (n + 63u) / 64u;
  const uint32_t blocks = std::min(cus, (tiles + kInferBlock / 64u - 1u) / (kInferBlock / 64u));
  hipLaunchKernelGGL(infer_kernel, dim3(blocks), dim3(kInferBlock), 0, s, feats, n, n_ptr, frags, tables, rgb);
  return hipGetLastError();
}

hipError_t launch_train(const float* feats, const float* targets, uint32_t n, const uint32_t* n_ptr,
                        const uint4* frags, const float* tables, float* grad, float* part, float* dx, float* loss,
                        hipStream_t s) {
  if (n == 0) return hipSuccess;
  // As many workgroups as are resident at once (bounded by the slots), each
  // looping over tiles, so no workgroup waits for a second wave of launches.
  static uint32_t resident = 0;
  if (resident == 0) {
    int dev = 0, cus = 0, per_cu = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e == hipSuccess) e = hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev);
    if (e == hipSuccess) e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, train_kernel, 256, 0);
    if (e != hipSuccess) return e;
    resident = (uint32_t)std::max(1, cus * std::max(per_cu, 1));
  }
  const uint32_t tiles = (n + 63u) / 64u;
  const uint32_t most = std::min(resident, kGradSlots), rounds = (tiles + most - 1u) / most;
  const uint32_t blocks = (tiles + rounds - 1u) / rounds;  // no more than finish in as many rounds
  hipLaunchKernelGGL(train_kernel, dim3(blocks), dim3(256), 0, s, feats, targets, n, n_ptr, frags, tables, part, dx,
                     loss);
  if (hipError_t e = hipGetLastError()) return e;
  hipLaunchKernelGGL(reduce_slots_kernel, dim3((kMlpParams + 255u) / 256u, 32u), dim3(256), 0, s, part, blocks, n,
                     n_ptr, grad);
  if (hipError_t e = hipGetLastError()) return e;
  // About 4096 samples per workgroup, at most 64 chunks per level; the
  // chunks' partial tables go to `part` (free again once reduce_slots_kernel
  // has read the MLP slots: 64 x 65,536 floats <= kGradSlots x kMlpParams).
  static_assert((size_t)64 * kTableParams <= (size_t)kGradSlots * kMlpParams, "table partials fit the slots");
  const uint32_t chunks = std::min(64u, (n + 4095u) / 4096u);
  const uint32_t per_chunk = (n + chunks - 1u) / chunks;
  hipLaunchKernelGGL(table_grad_kernel, dim3(kLevels, chunks), dim3(256), 0, s, feats, dx, n, n_ptr, per_chunk,
                     part);
  if (hipError_t e = hipGetLastError()) return e;
  hipLaunchKernelGGL(table_reduce_kernel, dim3((kTableParams + 255u) / 256u), dim3(256), 0, s, part, chunks,
                     grad + kMlpParams);
  return hipGetLastError();
}

hipError_t launch_adam(float* master, float* grad, float* m, float* v, AdamParams p, hipStream_t s) {
  hipLaunchKernelGGL(adam_kernel, dim3((kParams + 255) / 256), dim3(256), 0, s, master, grad, m, v, p);
  return hipGetLastError();
}

hipError_t launch_fill(float* p, uint32_t n, float value, hipStream_t s) {
  if (n == 0) return hipSuccess;
  hipLaunchKernelGGL(fill_kernel, dim3((n + 255) / 256), dim3(256), 0, s, p, n, value);
  return hipGetLastError();
}

}  // namespace vtn
