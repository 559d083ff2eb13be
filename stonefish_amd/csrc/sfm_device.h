// Device code of the surrogate network's fused inference, shared by the
// network library (sfh_mlp.hip: sfm_forward) and the hydrodynamics library
// (sfh_hydro.hip: the one-launch surrogate step).  gfx950 only.
//
// A workgroup of eight wavefronts runs TR rows (samples) of one network
// through all five layers.  The hidden activations stay in LDS (two TR x 256
// BF16 buffers, row-major [sample][feature], row stride kActStride).  Each
// layer is computed transposed, H'^T = W H^T: the weights are the MFMA's A
// operand (16-byte loads of W[feature][k..k+7] from global memory; 405 KB of
// BF16 per network, L2-resident) and the activations its B operand (16-byte
// LDS reads of H[sample][k..k+7]), so an accumulator lane holds four
// consecutive output features of one sample and stores them with one 8-byte
// LDS write.  Wavefront w owns output features [32 w, 32 w + 32) of each
// hidden layer (one 32-row tile of W, 64 registers of weights), so two
// wavefronts share each SIMD, and with two workgroups on a CU four: one's
// MFMAs run while the others' GELUs keep the VALU busy.  (Four wavefronts of 64
// features each need 280 registers: one wavefront per SIMD, whose MFMA and GELU
// phases only follow one another.)  The output layer is one 32-feature tile per
// 32-sample tile.
//
// v_mfma_f32_32x32x16_bf16 operand layout (checked on the device by
// sfm_probe_mfma): lane l holds A[l % 32][8 (l / 32) + 0..7] and
// B[8 (l / 32) + 0..7][l % 32]; accumulator register r of lane l is
// C[8 (r / 4) + 4 (l / 32) + r % 4][l % 32].
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

#include "../../include/sfmlp.h"
#include "sfm_gelu.h"

namespace sfm {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

static constexpr int kActStride = SFM_HIDDEN + 8;   // LDS row stride (elements): spreads rows over banks

__device__ __forceinline__ bf16x8 ld8(const uint16_t* p) { return *reinterpret_cast<const bf16x8*>(p); }

// Loads through a global-address-space pointer (global_load, not flat_load:
// a flat load also counts as an LDS access, and waiting for one waits for
// every memory access issued after it).
typedef const __attribute__((address_space(1))) bf16x8 gbf16x8;
__device__ __forceinline__ bf16x8 ld8g(const uint16_t* p) { return *(gbf16x8*)(p); }

// FP32 -> BF16 bits, round to nearest even (v_cvt_pk_bf16_f32).
__device__ __forceinline__ uint16_t f2bf(float f)
{
    const __bf16 h = (__bf16)f;
    return *reinterpret_cast<const uint16_t*>(&h);
}

// Two FP32 -> packed BF16 pair (low half = a).
__device__ __forceinline__ uint32_t f2bf2(float a, float b)
{
    bf16x2 v;
    v[0] = (__bf16)a;
    v[1] = (__bf16)b;
    return *reinterpret_cast<const uint32_t*>(&v);
}

// Row of the 32x32 accumulator tile held by register r of lane `lane`.
__device__ __forceinline__ int acc_row(int r, int lane) { return 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3); }

// Fragment order of a layer's BF16 weights W [out x K] (row-major indices r,
// c) for the fused kernels: the 8 consecutive columns 16 s + 8 h .. + 7 of
// row r = 64 w + 32 m + i are the 16 bytes that lane i + 32 h feeds to k-step s
// of the 32-row tile 2 w + m, and each (tile, s) owns 1 KB of
// contiguous memory, read by one fully coalesced load instruction.  (Row-major
// rows are 512 bytes apart, so the same fragments would touch 32 cache lines
// per instruction.)
__host__ __device__ __forceinline__ size_t frag_index(int r, int c, int K)
{
    const int w = r >> 6, m = (r >> 5) & 1, i = r & 31, s = c >> 4, h = (c >> 3) & 1, e = c & 7;
    return ((((size_t)(2 * w + m) * (K / 16) + s) * 64) + i + 32 * h) * 8 + e;
}

static constexpr int kWaves = SFM_HIDDEN / 32;   // wavefronts of a workgroup: one per 32 features

// Weight fragments of one 32-row tile of W [rows x K]: rows 32 tile + l % 32,
// columns 8 (l / 32) + 16 s.
template <int K>
struct TileW {
    bf16x8 a[K / 16];
};

// Requests a tile's weight fragments (fragment order, frag_index; K / 16
// 16-byte loads per lane, all issued at once: one L2 round trip per layer
// instead of one per k-step).  The weights do not depend on the activations,
// so a caller issues them one layer ahead, before the previous layer's epilogue.
template <int K>
__device__ __forceinline__ void load_tile(const uint16_t* __restrict__ w, int tile, TileW<K>& T)
{
    const uint16_t* p = w + ((size_t)tile * (K / 16) * 64 + (threadIdx.x & 63)) * 8;
#pragma unroll
    for (int s = 0; s < K / 16; ++s) T.a[s] = ld8g(p + 512 * s);
}

// acc[nt] = W-tile products of rows 32 nt .. + 31: input rows at `in` with row
// stride `stride` (LDS, or global memory for the network input), K inputs.
template <int RT, int K>
__device__ __forceinline__ void tile_mma(const TileW<K>& T, const uint16_t* in, int stride, f32x16 (&acc)[RT])
{
    const int lane = threadIdx.x & 63;
    const uint16_t* bp = in + (lane & 31) * stride + (lane >> 5) * 8;
    bf16x8 b[RT], n[RT];
#pragma unroll
    for (int nt = 0; nt < RT; ++nt) {
        acc[nt] = f32x16{};
        b[nt] = ld8(bp + 32 * nt * stride);
    }
    // the operands of the next k-step are read while the current one
    // multiplies; scheduled as written, since reads hoisted further cost
    // registers the occupancy needs
#pragma unroll
    for (int s = 0; s < K / 16; ++s) {
        if (s + 1 < K / 16) {
#pragma unroll
            for (int nt = 0; nt < RT; ++nt) n[nt] = ld8(bp + 32 * nt * stride + 16 * (s + 1));
        }
#pragma unroll
        for (int nt = 0; nt < RT; ++nt) {
            acc[nt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(T.a[s], b[nt], acc[nt], 0, 0, 0);
            b[nt] = n[nt];
        }
        if (s & 1) __builtin_amdgcn_sched_barrier(0);
    }
}

// out = gelu(acc + b) in BF16 (LDS rows, stride kActStride), then a barrier.
// The bias is read from LDS: a global load here would have to wait for the
// next layer's weight loads issued before it (loads complete in order).
template <int RT>
__device__ __forceinline__ void layer_store(const f32x16 (&acc)[RT], const float* bias, uint16_t* out)
{
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int lr = lane & 31, lq = (lane >> 5) * 4;
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const int f0 = 32 * wave + 8 * q + lq;   // four consecutive output features
        const float4 bq = *reinterpret_cast<const float4*>(bias + f0);
#pragma unroll
        for (int nt = 0; nt < RT; ++nt) {
            const f32x16& A = acc[nt];
            uint2 pk;
            pk.x = f2bf2(gelu(A[4 * q] + bq.x), gelu(A[4 * q + 1] + bq.y));
            pk.y = f2bf2(gelu(A[4 * q + 2] + bq.z), gelu(A[4 * q + 3] + bq.w));
            *reinterpret_cast<uint2*>(out + (32 * nt + lr) * kActStride + f0) = pk;
        }
    }
    __syncthreads();
}

// Hidden-layer biases of one network into LDS (bias[l][f], l < 4); the
// caller puts a barrier between this and mlp_hidden.
__device__ __forceinline__ void load_bias(const float* const* B, float (*bias)[SFM_HIDDEN])
{
    const int t = threadIdx.x;
    for (int i = t; i < (SFM_LAYERS - 1) * SFM_HIDDEN; i += blockDim.x)
        bias[i / SFM_HIDDEN][i % SFM_HIDDEN] = B[i / SFM_HIDDEN][i % SFM_HIDDEN];
}

// The four hidden layers of one TR-row tile, given layer 0's weight fragments
// (requested by the caller, possibly long before) and the hidden biases in
// LDS (load_bias).  Layer 0 reads its input
// rows from global memory (xg, row-major [row][32], rows xg .. xg + TR) when
// xg is not null, else from act[1] (row stride kActStride, columns 0..31).
// On return act[1] holds the last hidden layer and wavefronts w < TR / 32
// hold the output layer's fragments in ow.
template <int TR>
__device__ __forceinline__ void mlp_hidden(const uint16_t* const* W, const float (*B)[SFM_HIDDEN],
                                           uint16_t (*act)[TR * kActStride], const uint16_t* __restrict__ xg,
                                           const TileW<SFM_IN_PAD>& w0, TileW<SFM_HIDDEN>& ow)
{
    constexpr int RT = TR / 32;
    const int wave = threadIdx.x >> 6;
    f32x16 acc[RT];
    TileW<SFM_HIDDEN> wn;
    if (xg)
        tile_mma<RT, SFM_IN_PAD>(w0, xg, SFM_IN_PAD, acc);
    else
        tile_mma<RT, SFM_IN_PAD>(w0, act[1], kActStride, acc);
    load_tile<SFM_HIDDEN>(W[1], wave, wn);
    layer_store<RT>(acc, B[0], act[0]);
    tile_mma<RT, SFM_HIDDEN>(wn, act[0], kActStride, acc);
    load_tile<SFM_HIDDEN>(W[2], wave, wn);
    layer_store<RT>(acc, B[1], act[1]);
    tile_mma<RT, SFM_HIDDEN>(wn, act[1], kActStride, acc);
    load_tile<SFM_HIDDEN>(W[3], wave, wn);
    layer_store<RT>(acc, B[2], act[0]);
    tile_mma<RT, SFM_HIDDEN>(wn, act[0], kActStride, acc);
    if (wave < RT) load_tile<SFM_HIDDEN>(W[SFM_LAYERS - 1], 0, ow);   // one tile of outputs
    layer_store<RT>(acc, B[3], act[1]);
}

// Output layer of sample tile `wave` (< TR / 32) from act[1]: on return,
// registers 0..3 of lane l hold outputs 4 (l / 32) + 0..3 (bias included) of
// sample 32 wave + l % 32.
__device__ __forceinline__ void mlp_output(const TileW<SFM_HIDDEN>& L, const float* __restrict__ bias,
                                           const uint16_t* __restrict__ in, float o[4])
{
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int lr = lane & 31, lk = (lane >> 5) * 8, lq = (lane >> 5) * 4;
    f32x16 acc = {};
#pragma unroll
    for (int s = 0; s < SFM_HIDDEN / 16; ++s)
        acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(L.a[s], ld8(in + (32 * wave + lr) * kActStride + 16 * s + lk),
                                                      acc, 0, 0, 0);
#pragma unroll
    for (int i = 0; i < 4; ++i) o[i] = acc[i] + (lq + i < SFM_OUT_PAD ? bias[lq + i] : 0.f);
}

// Workgroup b of a grid of n in XCD-major order: the hardware deals
// workgroups to the eight XCDs round-robin (b % 8), so the workgroups that
// share an XCD (and its L2) get consecutive tiles, which mostly share one
// network's weights.
__device__ __forceinline__ uint32_t xcd_tile(uint32_t b, uint32_t n)
{
    const uint32_t q = n / 8, r = n % 8, x = b % 8, s = b / 8;
    return x * q + (x < r ? x : r) + s;
}

}  // namespace sfm
