// sfmlp: hand-written gfx950 BF16 MFMA kernels of the hydrodynamics surrogate
// (forward, backward, Adam).  No counterpart in the reference.
//
// A training step is three launches:
//   k_train   a workgroup takes 64 rows of the batch through the forward pass,
//             the loss and the backward products: the activations stay in LDS
//             and the pre-activations in registers, and only the transposed
//             layer inputs H^T and output gradients dZ^T (BF16) go to memory;
//   k_wgrad   dW = dZ^T H of all five layers, split over the batch, with the
//             bias gradients (row sums of dZ^T);
//   k_adam    sums the splits' partials in a fixed order and steps Adam.
// Matrix products outside k_train are C = A * Bt^T with A [rows x K] and Bt
// [cols x K] both row-major and contiguous in K, so each lane's MFMA operands
// are one 16-byte load.  Tiles are 32x32 v_mfma_f32_32x32x16_bf16
// accumulators: the products of the 256-wide layers run 64x64 per workgroup
// with the operands staged in LDS, the 32-wide ones one tile per wavefront.
#include <hip/hip_runtime.h>

#include <cmath>
#include <cstdarg>
#include <cstdio>
#include <cstring>
#include <vector>

#include "../../include/sfmlp.h"
#include "sfm_device.h"

using sfm::acc_row;
using sfm::bf16x8;
using sfm::f2bf;
using sfm::f2bf2;
using sfm::ld8g;
using sfm::f32x16;
using sfm::gelu;
using sfm::gelu_grad;
using sfm::kActStride;
using sfm::ld8;
using sfm::load_tile;
using sfm::tile_mma;
using sfm::TileW;

static thread_local char g_err[512] = "";

static int fail(int code, const char* fmt, ...)
{
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(g_err, sizeof(g_err), fmt, ap);
    va_end(ap);
    return code;
}

#define HIPCHK(expr)                                                                    \
    do {                                                                                \
        hipError_t e_ = (expr);                                                         \
        if (e_ != hipSuccess)                                                           \
            return fail(SFM_ERR_HIP, "%s failed: %s", #expr, hipGetErrorString(e_));    \
    } while (0)

extern "C" const char* sfm_last_error(void) { return g_err; }

static constexpr int kDims[SFM_LAYERS + 1] = {SFM_IN_PAD, SFM_HIDDEN, SFM_HIDDEN, SFM_HIDDEN, SFM_HIDDEN, SFM_OUT_PAD};
static constexpr int kReal[SFM_LAYERS + 1] = {SFM_IN, SFM_HIDDEN, SFM_HIDDEN, SFM_HIDDEN, SFM_HIDDEN, SFM_OUT};
static constexpr int kSplitK = 256;   // batch rows per weight-gradient split
static constexpr int kMaxSplits = 64; // batch splits of a weight-gradient product
static constexpr int kTrainRows = 64; // batch rows per workgroup of k_train

// Batch splits of layer l's weight-gradient product at most: the 256 x 256
// products run 16 workgroups per split, the 32-wide ones 2, so the latter
// take more splits to fill the chip; every split's partial sum is read again
// by the Adam launch.
static constexpr int max_splits(int l) { return kDims[l] == SFM_HIDDEN && kDims[l + 1] == SFM_HIDDEN ? 32 : kMaxSplits; }

// ---------------------------------------------------------------------------
// numerics
// ---------------------------------------------------------------------------



// ---------------------------------------------------------------------------
// GEMM tile kernel
// ---------------------------------------------------------------------------

enum { EPI_HIDDEN = 0, EPI_OUT = 1, EPI_WGRAD = 2 };

struct GemmArgs {
    const uint16_t* A;      // [rows x K], lda
    const uint16_t* Bt;     // [cols x K], ldb
    int lda, ldb;
    int rows, cols, K, ksplit;
    const float* bias;      // [cols]                      (HIDDEN, OUT)
    uint16_t* H;            // [rows x cols] BF16          (HIDDEN)
    float* y;               // [rows x SFM_OUT]            (OUT)
    float* part;            // [ksplit][rows x cols] FP32  (WGRAD)
    float* bpart;           // [ksplit][rows] FP32 row sums of A over each split (WGRAD: bias gradient)
};

__device__ __forceinline__ float sum8(const bf16x8& v)
{
    return (((float)v[0] + (float)v[1]) + ((float)v[2] + (float)v[3])) +
           (((float)v[4] + (float)v[5]) + ((float)v[6] + (float)v[7]));
}


// The epilogue of a wavefront's 32x32 tile of C at rows 32 rt and columns 32 ct.
template <int EPI>
__device__ __forceinline__ void gemm_store(const GemmArgs& g, const f32x16& A, int rt, int ct, int split, int lane)
{
    const int n = ct * 32 + (lane & 31), mb = rt * 32;
    if (EPI == EPI_WGRAD) {
        float* out = g.part + (size_t)split * g.rows * g.cols;
#pragma unroll
        for (int r = 0; r < 16; ++r) out[(size_t)(mb + acc_row(r, lane)) * g.cols + n] = A[r];
        return;
    }
    const float b = g.bias[n];
#pragma unroll
    for (int r = 0; r < 16; ++r) {
        const int m = mb + acc_row(r, lane);
        const float z = A[r] + b;
        if (EPI == EPI_HIDDEN) g.H[(size_t)m * g.cols + n] = f2bf(gelu(z));
        else if (n < SFM_OUT) g.y[(size_t)m * SFM_OUT + n] = z;
    }
}

// One wavefront computes a 32 x 32 tile of C: per k-step two 16-byte operand
// loads feed an MFMA.  wave: the tile; split: the part of K.
template <int EPI>
__device__ __forceinline__ void gemm_wave(const GemmArgs& g, int wave, int split)
{
    const int lane = threadIdx.x & 63;
    const int blocks_n = g.cols / 32;
    const int bm = wave / blocks_n, bn = wave - bm * blocks_n;
    if (bm * 32 >= g.rows) return;
    const int kper = g.K / g.ksplit;
    const int kk = split * kper + (lane >> 5) * 8;
    const uint16_t* ap = g.A + (size_t)(bm * 32 + (lane & 31)) * g.lda + kk;
    const uint16_t* bp = g.Bt + (size_t)(bn * 32 + (lane & 31)) * g.ldb + kk;
    f32x16 acc = {};
    // The operands of the next kPF k-steps are in flight while the current
    // one multiplies (a ring of kPF register stages, refilled right after use):
    // a k-step waits for a load issued kPF steps earlier, not for the last one.
    constexpr int kPF = 4;
    bf16x8 ra[kPF], rb[kPF];
#pragma unroll
    for (int s = 0; s < kPF; ++s)
        if (16 * s < kper) {
            ra[s] = ld8g(ap + 16 * s);
            rb[s] = ld8g(bp + 16 * s);
        }
    // the bias gradient rides along the weight gradient: the wavefronts of the
    // first column of tiles also sum their rows of A (each lane 8 of the 16 k
    // of a k-step, the two half-waves combined at the end)
    const bool rsum = EPI == EPI_WGRAD && bn == 0;
    float rs = 0.f;
    for (int k0 = 0; k0 < kper; k0 += 16 * kPF) {
#pragma unroll
        for (int s = 0; s < kPF; ++s) {
            const int k = k0 + 16 * s;
            if (k < kper) {
                if (rsum) rs += sum8(ra[s]);
                acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ra[s], rb[s], acc, 0, 0, 0);
                if (k + 16 * kPF < kper) {
                    ra[s] = ld8g(ap + k + 16 * kPF);
                    rb[s] = ld8g(bp + k + 16 * kPF);
                }
            }
        }
    }
    if (rsum) {
        const float v = rs + __shfl_xor(rs, 32, 64);
        if (lane < 32) g.bpart[(size_t)split * g.rows + bm * 32 + lane] = v;
    }
    gemm_store<EPI>(g, acc, bm, bn, split, lane);
}

// Workgroup-tiled product for the 256-wide layers: the four wavefronts of a
// workgroup, in a 2 x 2 arrangement, cover (64 T) x (64 T) of C, each T x T
// tiles of 32 x 32.  K advances in chunks of kKC: the workgroup copies the
// chunk's rows of A and of Bt into LDS once (the next chunk's global loads in
// flight while the current one multiplies; two LDS buffers) and the wavefronts
// read their MFMA operands from there, so an operand row comes from L2 once per
// workgroup instead of once per wavefront that uses it.
static constexpr int kKC = 64;            // K per chunk
static constexpr int kLdsRow = kKC + 8;   // bf16 per LDS row: 16 bytes of padding against bank conflicts

template <int T>
struct GemmLds {
    uint16_t A[2][64 * T * kLdsRow];
    uint16_t B[2][64 * T * kLdsRow];
};

template <int EPI, int T>
__device__ __forceinline__ void gemm_group(const GemmArgs& g, GemmLds<T>& L, int tile, int split)
{
    constexpr int BT = 64 * T;
    constexpr int SEG = kKC / 8;                 // 16-byte segments per row and chunk
    constexpr int SA = BT * SEG / 256;
    const int t = threadIdx.x, lane = t & 63, w = t >> 6, wm = w >> 1, wn = w & 1;
    const int blocks_n = g.cols / BT;
    const int bm = tile / blocks_n, bn = tile - bm * blocks_n;
    const int kper = g.K / g.ksplit;
    const int kbase = split * kper;
    const int nch = kper / kKC;
    bf16x8 ra[SA], rb[SA];
    auto gload = [&](int c) {
        const int k0 = kbase + c * kKC;
#pragma unroll
        for (int i = 0; i < SA; ++i) {
            const int idx = t + 256 * i, row = idx / SEG, seg = idx % SEG;
            ra[i] = ld8g(g.A + (size_t)(bm * BT + row) * g.lda + k0 + seg * 8);
            rb[i] = ld8g(g.Bt + (size_t)(bn * BT + row) * g.ldb + k0 + seg * 8);
        }
    };
    // bias gradient (see gemm_wave): the workgroups of the first column of
    // tiles sum the rows of A they copy, each thread its 8-value segments
    const bool rsum = EPI == EPI_WGRAD && bn == 0;
    float rs[SA] = {};
    auto lstore = [&](int buf) {
#pragma unroll
        for (int i = 0; i < SA; ++i) {
            const int idx = t + 256 * i, row = idx / SEG, seg = idx % SEG;
            *reinterpret_cast<bf16x8*>(&L.A[buf][row * kLdsRow + seg * 8]) = ra[i];
            *reinterpret_cast<bf16x8*>(&L.B[buf][row * kLdsRow + seg * 8]) = rb[i];
            if (rsum) rs[i] += sum8(ra[i]);
        }
    };
    f32x16 acc[T][T];
#pragma unroll
    for (int i = 0; i < T; ++i)
#pragma unroll
        for (int j = 0; j < T; ++j) acc[i][j] = f32x16{};
    gload(0);
    lstore(0);
    __syncthreads();
    for (int c = 0; c < nch; ++c) {
        const int buf = c & 1;
        if (c + 1 < nch) gload(c + 1);
#pragma unroll
        for (int s = 0; s < kKC / 16; ++s) {
            const int kk = 16 * s + (lane >> 5) * 8;
            bf16x8 fa[T], fb[T];
#pragma unroll
            for (int i = 0; i < T; ++i) {
                fa[i] = ld8(&L.A[buf][((wm * T + i) * 32 + (lane & 31)) * kLdsRow + kk]);
                fb[i] = ld8(&L.B[buf][((wn * T + i) * 32 + (lane & 31)) * kLdsRow + kk]);
            }
#pragma unroll
            for (int i = 0; i < T; ++i)
#pragma unroll
                for (int j = 0; j < T; ++j)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa[i], fb[j], acc[i][j], 0, 0, 0);
        }
        if (c + 1 < nch) lstore(buf ^ 1);
        __syncthreads();
    }
    if (rsum) {   // the SEG threads of a row are consecutive lanes
        static_assert(SEG == 8, "row segments per chunk");
#pragma unroll
        for (int i = 0; i < SA; ++i) {
            float v = rs[i];
            v += __shfl_xor(v, 1, 64);
            v += __shfl_xor(v, 2, 64);
            v += __shfl_xor(v, 4, 64);
            const int idx = t + 256 * i;
            if (idx % SEG == 0) g.bpart[(size_t)split * g.rows + bm * BT + idx / SEG] = v;
        }
    }
#pragma unroll
    for (int i = 0; i < T; ++i)
#pragma unroll
        for (int j = 0; j < T; ++j)
            gemm_store<EPI>(g, acc[i][j], (bm * 2 + wm) * T + i, (bn * 2 + wn) * T + j, split, lane);
}

template <int EPI>
__global__ __launch_bounds__(256) void k_gemm(GemmArgs g)
{
    gemm_wave<EPI>(g, blockIdx.x * 4 + (threadIdx.x >> 6), blockIdx.y);
}

template <int EPI>
__global__ __launch_bounds__(256) void k_gemm_lds(GemmArgs g)
{
    __shared__ __attribute__((aligned(16))) GemmLds<1> L;
    gemm_group<EPI, 1>(g, L, blockIdx.x, blockIdx.y);
}

// The weight- and bias-gradient products of all layers in one launch: 22 us for
// a batch of 16,384 (one launch per layer with 64 x 64 tiles: 43 us; 64 x 64
// tiles in one launch: 30).  Each operand column is read by two workgroups, from
// memory the training kernel has just written (Infinity Cache).
// Workgroups from block0 of a layer on are its: the 256 x 256 layers' by
// (split, 128 x 128 tile), the 32-wide ones' by (split, four 32 x 32 tiles).
static constexpr int kWgradTile = 128;

struct WgradSet {
    GemmArgs g[SFM_LAYERS];
    int block0[SFM_LAYERS];
};

__global__ __launch_bounds__(256) void k_wgrad(WgradSet W)
{
    __shared__ __attribute__((aligned(16))) GemmLds<kWgradTile / 64> L;
    int i = 0;
    while (i + 1 < SFM_LAYERS && (int)blockIdx.x >= W.block0[i + 1]) ++i;
    const GemmArgs& g = W.g[i];
    const int b = (int)blockIdx.x - W.block0[i];
    if (g.rows % kWgradTile == 0 && g.cols % kWgradTile == 0) {
        const int tiles = (g.rows / kWgradTile) * (g.cols / kWgradTile);
        gemm_group<EPI_WGRAD, kWgradTile / 64>(g, L, b % tiles, b / tiles);
    } else {
        const int groups = g.rows * g.cols / (4 * 32 * 32);
        gemm_wave<EPI_WGRAD>(g, (b % groups) * 4 + (threadIdx.x >> 6), b / groups);
    }
}

// ---------------------------------------------------------------------------
// forward, loss and backward of a training step
// ---------------------------------------------------------------------------

struct TrainArgs {
    const uint16_t* x;              // [M x 32] BF16
    const float* target;            // [M x SFM_OUT]
    const uint16_t* W[SFM_LAYERS];  // weights in fragment order
    const uint16_t* Wt[SFM_LAYERS]; // transposed weights [in x out] in fragment order (layers 1..4)
    const float* b[SFM_LAYERS];
    uint16_t* Ht[SFM_LAYERS];       // layer inputs, transposed [in x ldt]
    uint16_t* dZt[SFM_LAYERS];      // layer output gradients, transposed [out x ldt]
    float* loss_part;               // per workgroup
    float scale;                    // 1 / (M * SFM_OUT)
    int ldt;
};

// Transposes 4 x 4 BF16 values over each four lanes: lane i brings four
// features of row i and takes four rows of feature quad_feature(i), so the
// transposed tile goes to memory in 8-byte stores (in 2-byte ones k_train took
// 46 us instead of 40 on 16,384 rows).
__device__ __forceinline__ uint32_t quad_feature(int lane) { return ((lane & 1) << 1) | ((lane >> 1) & 1); }

__device__ __forceinline__ uint2 quad_transpose(uint2 v, int lane)
{
    const bool odd = lane & 1, up = lane & 2;
    const uint32_t r1 = (uint32_t)__builtin_amdgcn_mov_dpp((int)(odd ? v.x : v.y), 0xB1, 0xf, 0xf, true);   // lane ^ 1
    const uint32_t a = odd ? r1 : v.x, b = odd ? v.y : r1;   // rows i & ~1 and i | 1, two features
    const uint32_t lo = __builtin_amdgcn_perm(b, a, 0x05040100u), hi = __builtin_amdgcn_perm(b, a, 0x07060302u);
    const uint32_t r2 = (uint32_t)__builtin_amdgcn_mov_dpp((int)(up ? lo : hi), 0x4E, 0xf, 0xf, true);      // lane ^ 2
    return up ? make_uint2(r2, hi) : make_uint2(lo, r2);
}

// A wavefront's tile of BF16 values to the LDS activations ([row][feature])
// and, transposed, to memory: f(acc value, index) gives the value.
template <typename F>
__device__ __forceinline__ void tile_store(uint16_t* act, uint16_t* __restrict__ outt, uint32_t ldt, int f0, F f)
{
    const int lane = threadIdx.x & 63, lr = lane & 31, lq = (lane >> 5) * 4;
    const uint32_t fi = quad_feature(lane);
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const int fq = f0 + 8 * q + lq;   // four consecutive features
#pragma unroll
        for (int nt = 0; nt < 2; ++nt) {
            uint2 pk;
            pk.x = f2bf2(f(nt, 4 * q), f(nt, 4 * q + 1));
            pk.y = f2bf2(f(nt, 4 * q + 2), f(nt, 4 * q + 3));
            *reinterpret_cast<uint2*>(act + (32 * nt + lr) * kActStride + fq) = pk;
            const uint2 tr = quad_transpose(pk, lane);
            const uint32_t o = ((uint32_t)fq + fi) * ldt + 32u * nt + (uint32_t)(lr & ~3);   // below 2^31: ldt <= 2^22
            *reinterpret_cast<uint2*>(outt + o) = tr;
        }
        __builtin_amdgcn_sched_barrier(0);
    }
}

// One workgroup of eight wavefronts: 64 rows of the batch forward and back.
// Wavefront w owns features 32 w .. + 31 of every hidden layer in both
// directions, so the pre-activations Z that gelu' needs on the way back stay
// where the forward pass left them: 32 registers a layer (layer 0's in LDS)
// beside 64 for the weights requested one layer ahead, which leaves two
// wavefronts per SIMD.  Products are W H^T and W^T dZ^T (the weights the MFMA's
// A operand, in fragment order); the sums over K run in the order of the
// per-layer kernels, so the gradients are theirs bit for bit.  16,384 rows
// (one workgroup per CU): 40 us, where the launches it replaces (a transpose,
// five forward and four backward products through Z, H, H^T, dZ and dZ^T in
// memory) took 155.  About 6 us of it wait on the 70 MB of transposed stores,
// 13 are the GELUs and their derivatives (VALU and transcendentals), the rest
// the products at one workgroup's latency per layer.
__global__ __launch_bounds__(512, 2) void k_train(TrainArgs P)
{
    __shared__ __attribute__((aligned(16))) uint16_t act[2][kTrainRows * kActStride];
    __shared__ __attribute__((aligned(16))) float bias[SFM_LAYERS - 1][SFM_HIDDEN];
    __shared__ float4 z0[8][512];   // layer 0's Z, each thread its own
    __shared__ float lsum[2];
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6, lq = (lane >> 5) * 4, f0 = 32 * wave;
    const size_t row0 = (size_t)blockIdx.x * kTrainRows;
    const uint16_t* xg = P.x + row0 * SFM_IN_PAD;
    TileW<SFM_IN_PAD> w0;
    load_tile<SFM_IN_PAD>(P.W[0], wave, w0);
    sfm::load_bias(P.b, bias);
    {   // x^T: thread t takes row t % 64, inputs 4 (t / 64) .. + 3
        const int r = t & 63, c = 4 * (t >> 6);
        const uint2 v = *reinterpret_cast<const uint2*>(xg + (size_t)r * SFM_IN_PAD + c);
        uint16_t* o = P.Ht[0] + (size_t)c * P.ldt + row0 + r;
        o[0] = (uint16_t)v.x;
        o[P.ldt] = (uint16_t)(v.x >> 16);
        o[2 * (size_t)P.ldt] = (uint16_t)v.y;
        o[3 * (size_t)P.ldt] = (uint16_t)(v.y >> 16);
    }
    __syncthreads();
    f32x16 Z[SFM_LAYERS - 1][2];
    TileW<SFM_HIDDEN> wn;
    tile_mma<2, SFM_IN_PAD>(w0, xg, SFM_IN_PAD, Z[0]);
#pragma unroll
    for (int l = 0; l < SFM_LAYERS - 1; ++l) {
        if (l > 0) tile_mma<2, SFM_HIDDEN>(wn, act[(l - 1) & 1], kActStride, Z[l]);
        if (l < SFM_LAYERS - 2) load_tile<SFM_HIDDEN>(P.W[l + 1], wave, wn);
        else if (wave < 2) load_tile<SFM_HIDDEN>(P.W[l + 1], 0, wn);   // the output layer: one tile of features
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const float4 b = *reinterpret_cast<const float4*>(&bias[l][f0 + 8 * q + lq]);
#pragma unroll
            for (int nt = 0; nt < 2; ++nt) {
                Z[l][nt][4 * q] += b.x;
                Z[l][nt][4 * q + 1] += b.y;
                Z[l][nt][4 * q + 2] += b.z;
                Z[l][nt][4 * q + 3] += b.w;
            }
        }
        if (l == 0) {
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const f32x16& z = Z[0][i >> 2];
                const int r = 4 * (i & 3);
                z0[i][t] = make_float4(z[r], z[r + 1], z[r + 2], z[r + 3]);
            }
        }
        tile_store(act[l & 1], P.Ht[l + 1] + row0, P.ldt, f0, [&](int nt, int r) { return gelu(Z[l][nt][r]); });
        __syncthreads();
    }
    // output layer, loss and its gradient: wavefronts 0 and 1 a row tile each;
    // dZ of the 32 padded outputs goes to act[0] (columns 0..31), whose last
    // reader is behind the barrier above
    TileW<SFM_OUT_PAD> wo;
    load_tile<SFM_OUT_PAD>(P.Wt[SFM_LAYERS - 1], wave, wo);
    if (wave < 2) {
        const int lr = lane & 31, row = 32 * wave + lr;
        const uint16_t* bp = act[1] + row * kActStride + (lane >> 5) * 8;
        f32x16 acc = {};
#pragma unroll
        for (int s = 0; s < SFM_HIDDEN / 16; ++s)
            acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(wn.a[s], ld8(bp + 16 * s), acc, 0, 0, 0);
        const float* tg = P.target + (row0 + row) * SFM_OUT;
        float sq = 0.f, dz[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {   // registers 0..3 of lane l: outputs 4 (l / 32) + 0..3
            dz[i] = 0.f;
            if (lq + i < SFM_OUT) {
                const float z = acc[i] + P.b[SFM_LAYERS - 1][lq + i];
                const float d = z - tg[lq + i];
                sq += d * d;
                dz[i] = 2.0f * d * P.scale;   // dLoss/dz
            }
        }
        uint2 pk;
        pk.x = f2bf2(dz[0], dz[1]);
        pk.y = f2bf2(dz[2], dz[3]);
        uint16_t* a = act[0] + row * kActStride;
        *reinterpret_cast<uint2*>(a + lq) = pk;
#pragma unroll
        for (int c = 8; c < SFM_OUT_PAD; c += 8) *reinterpret_cast<uint2*>(a + c + lq) = make_uint2(0u, 0u);
        uint16_t* o = P.dZt[SFM_LAYERS - 1] + row0 + row;
        const uint32_t pw[2] = {pk.x, pk.y};
#pragma unroll
        for (int c = 0; c < SFM_OUT_PAD; c += 8)   // the padded outputs' rows are zero
#pragma unroll
            for (int i = 0; i < 4; ++i)
                o[(size_t)(c + lq + i) * P.ldt] = c == 0 ? (uint16_t)(pw[i >> 1] >> (16 * (i & 1))) : (uint16_t)0;
#pragma unroll
        for (int off = 32; off >= 1; off >>= 1) sq += __shfl_xor(sq, off, 64);
        if (lane == 0) lsum[wave] = sq * P.scale;
    }
    __syncthreads();
    if (t == 0) P.loss_part[blockIdx.x] = lsum[0] + lsum[1];
    // back: dZ of hidden layer l = (W^T of the layer above dZ) * gelu'(Z)
    f32x16 acc[2];
    tile_mma<2, SFM_OUT_PAD>(wo, act[0], kActStride, acc);
#pragma unroll
    for (int l = SFM_LAYERS - 2; l >= 0; --l) {
        // the gradients alternate between the LDS buffers from act[1] on
        const int buf = (SFM_LAYERS - 1 - l) & 1;
        if (l < SFM_LAYERS - 2) tile_mma<2, SFM_HIDDEN>(wn, act[buf ^ 1], kActStride, acc);
        if (l > 0) load_tile<SFM_HIDDEN>(P.Wt[l], wave, wn);
        __builtin_amdgcn_sched_barrier(0);
        // gelu' shares its erf and exponential with the forward pass's gelu:
        // hidden from the compiler, which would keep two more values per
        // activation alive across the whole kernel
        if (l == 0) {
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const float4 z = z0[i][t];
                const int r = 4 * (i & 3);
                Z[0][i >> 2][r] = z.x; Z[0][i >> 2][r + 1] = z.y; Z[0][i >> 2][r + 2] = z.z; Z[0][i >> 2][r + 3] = z.w;
            }
        }
#pragma unroll
        for (int nt = 0; nt < 2; ++nt) asm volatile("" : "+v"(Z[l][nt]));
        tile_store(act[buf], P.dZt[l] + row0, P.ldt, f0,
                   [&](int nt, int r) { return acc[nt][r] * gelu_grad(Z[l][nt][r]); });
        if (l > 0) __syncthreads();
    }
}

// ---------------------------------------------------------------------------
// fused inference: all five layers of a tile of rows in one workgroup
// ---------------------------------------------------------------------------

struct NetSet {
    int nnets;
    uint32_t row_end[SFM_MAX_GROUP];   // exclusive end row of each network's rows
    const uint16_t* W[SFM_MAX_GROUP][SFM_LAYERS];
    const float* b[SFM_MAX_GROUP][SFM_LAYERS];
};

// Inference of TR consecutive rows of one network per workgroup (the fused
// network of sfm_device.h).
template <int TR>
__global__ __launch_bounds__(64 * sfm::kWaves, 4) void k_mlp_fused(NetSet ns, const uint16_t* __restrict__ x, uint32_t rows,
                                                   float* __restrict__ y)
{
    __shared__ __attribute__((aligned(16))) uint16_t act[2][TR * kActStride];
    __shared__ __attribute__((aligned(16))) float bias[SFM_LAYERS - 1][SFM_HIDDEN];
    const uint32_t row0 = sfm::xcd_tile(blockIdx.x, gridDim.x) * TR;
    if (row0 >= rows) return;
    int k = 0;
    while (k + 1 < ns.nnets && row0 >= ns.row_end[k]) ++k;
    TileW<SFM_IN_PAD> w0;
    load_tile<SFM_IN_PAD>(ns.W[k][0], threadIdx.x >> 6, w0);
    sfm::load_bias(ns.b[k], bias);
    __syncthreads();
    TileW<SFM_HIDDEN> ow;
    sfm::mlp_hidden<TR>(ns.W[k], bias, act, x + (size_t)row0 * SFM_IN_PAD, w0, ow);
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    if (wave < TR / 32) {
        float o[4];
        sfm::mlp_output(ow, ns.b[k][SFM_LAYERS - 1], act[1], o);
        const int lq = (lane >> 5) * 4;
        float* yo = y + (size_t)(row0 + 32 * wave + (lane & 31)) * SFM_OUT;
#pragma unroll
        for (int i = 0; i < 4; ++i)
            if (lq + i < SFM_OUT) yo[lq + i] = o[i];
    }
}

// ---------------------------------------------------------------------------
// small kernels
// ---------------------------------------------------------------------------

// Adam on n parameters of a [rows x cols] matrix (cols = 1 for biases): the
// gradient is the sum of nsplit partials (fixed order); keeps the FP32 master
// copy and refreshes the BF16 copy and its transpose.
// One parameter tensor of an Adam step: its FP32 weights and moments, the
// gradient partials of the batch splits (summed in a fixed order), where the
// summed gradient is kept, and (weights only) the BF16 copies to refresh.
struct AdamSeg {
    float *w, *mo, *ve;
    const float* part;
    float* gsave;
    uint16_t *wb, *wtp, *wp;          // row-major; transposed and plain in fragment order
    int nsplit, rows, cols, block0;   // block0: first workgroup of this tensor in the launch
};

struct AdamSet {
    AdamSeg seg[2 * SFM_LAYERS];
    int nseg;
    int nblk;                 // workgroups of the tensors; one more sums the loss
    const float* loss_part;   // k_train's, one per workgroup
    int nloss;
    float* loss;
};

// Adam with bias correction for every weight and bias tensor of the network
// in one launch (each workgroup finds its tensor from the block offsets).
__global__ __launch_bounds__(256) void k_adam(AdamSet S, float lr, float b1, float b2, float eps, float bc1,
                                              float bc2)
{
    if ((int)blockIdx.x >= S.nblk) {   // the loss: fixed order
        __shared__ float red[4];
        float v = 0.f;
        for (int i = threadIdx.x; i < S.nloss; i += 256) v += S.loss_part[i];
#pragma unroll
        for (int off = 32; off >= 1; off >>= 1) v += __shfl_xor(v, off, 64);
        if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
        __syncthreads();
        if (threadIdx.x == 0) *S.loss = (red[0] + red[1]) + (red[2] + red[3]);
        return;
    }
    int si = 0;
    while (si + 1 < S.nseg && (int)blockIdx.x >= S.seg[si + 1].block0) ++si;
    const AdamSeg& g = S.seg[si];
    const int n = g.rows * g.cols;
    const int i = ((int)blockIdx.x - g.block0) * (int)blockDim.x + (int)threadIdx.x;
    if (i >= n) return;
    float gr = 0.f;
    int s = 0;
    for (; s + 32 <= g.nsplit; s += 32) {   // 32 loads in flight, summed in order
        float v[32];
#pragma unroll
        for (int k = 0; k < 32; ++k) v[k] = g.part[(size_t)(s + k) * n + i];
#pragma unroll
        for (int k = 0; k < 32; ++k) gr += v[k];
    }
    for (; s < g.nsplit; ++s) gr += g.part[(size_t)s * n + i];
    g.gsave[i] = gr;
    const float m = b1 * g.mo[i] + (1.f - b1) * gr;
    const float v = b2 * g.ve[i] + (1.f - b2) * gr * gr;
    g.mo[i] = m;
    g.ve[i] = v;
    const float wn = g.w[i] - lr * (m / bc1) / (sqrtf(v / bc2) + eps);
    g.w[i] = wn;
    if (g.wb) {
        const uint16_t h = f2bf(wn);
        g.wb[i] = h;
        const int r = i / g.cols, c = i - r * g.cols;
        g.wtp[sfm::frag_index(c, r, g.rows)] = h;
        g.wp[sfm::frag_index(r, c, g.cols)] = h;
    }
}

// The summed gradients of one layer: n weights, then nb biases.
__global__ __launch_bounds__(256) void k_gradients(const float* __restrict__ gw, const float* __restrict__ gb, int n,
                                                   int nb, float* __restrict__ dw, float* __restrict__ db)
{
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i < n) dw[i] = gw[i];
    else if (i < n + nb) db[i - n] = gb[i - n];
}

__global__ void k_to_bf16(const float* __restrict__ x, uint16_t* __restrict__ y, uint64_t n)
{
    uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) y[i] = f2bf(x[i]);
}

// One 32x32x16 product with the operand mapping of k_gemm: a [32 x 16],
// b [16 x 32] row-major; c [32 x 32] row-major.
__global__ void k_probe(const uint16_t* __restrict__ a, const uint16_t* __restrict__ b, float* __restrict__ c)
{
    const int lane = threadIdx.x;
    const int kk = (lane >> 5) * 8;
    bf16x8 av, bv;
    for (int i = 0; i < 8; ++i) {
        uint16_t x = a[(lane & 31) * 16 + kk + i];
        uint16_t y = b[(kk + i) * 32 + (lane & 31)];
        av[i] = *reinterpret_cast<const __bf16*>(&x);
        bv[i] = *reinterpret_cast<const __bf16*>(&y);
    }
    f32x16 acc = {};
    acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(av, bv, acc, 0, 0, 0);
    for (int r = 0; r < 16; ++r) c[acc_row(r, lane) * 32 + (lane & 31)] = acc[r];
}

// ---------------------------------------------------------------------------
// host
// ---------------------------------------------------------------------------

struct Layer {
    float *W = nullptr, *b = nullptr, *mW = nullptr, *vW = nullptr, *mb = nullptr, *vb = nullptr;
    float *gW = nullptr, *gb = nullptr;
    uint16_t* Wb = nullptr;
    uint16_t* Wp = nullptr;   // BF16 in fragment order (sfm::frag_index) for the fused kernels
    uint16_t* Wtp = nullptr;  // the transpose [in x out] in fragment order, for the backward products
};

struct sfm_net_t {
    uint32_t maxb = 0;
    uint32_t cus = 256;              // compute units of the device the network was created on
    Layer L[SFM_LAYERS];
    uint16_t* H[SFM_LAYERS] = {};    // H[l] = input of layer l (H[0] unused: the caller's x), per-layer inference
    uint16_t* Ht[SFM_LAYERS] = {};   // training: layer inputs, transposed
    uint16_t* dZt[SFM_LAYERS] = {};  // training: layer output gradients, transposed
    float* loss_part = nullptr;      // per workgroup of k_train
    float* part[SFM_LAYERS] = {};    // per layer: weight-gradient partials of the batch splits (<= max_splits)
    float* dbias[SFM_LAYERS] = {};   // per layer: bias-gradient partials of the same splits
    uint64_t step = 0;
    bool timing = false;
    hipEvent_t ev[2] = {nullptr, nullptr};
    bool pending = false;
    double pending_flops = 0, ms_sum = 0, flops_sum = 0;
    uint32_t timed = 0;
};

static uint64_t splitmix(uint64_t& s)
{
    uint64_t z = (s += 0x9E3779B97F4A7C15ull);
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
    return z ^ (z >> 31);
}

static void net_free(sfm_net_t* n)
{
    for (Layer& l : n->L) {
        for (float* p : {l.W, l.b, l.mW, l.vW, l.mb, l.vb, l.gW, l.gb}) hipFree(p);
        hipFree(l.Wb);
        hipFree(l.Wtp);
        hipFree(l.Wp);
    }
    for (int i = 0; i < SFM_LAYERS; ++i) { hipFree(n->H[i]); hipFree(n->Ht[i]); hipFree(n->dZt[i]); }
    hipFree(n->loss_part);
    for (int i = 0; i < SFM_LAYERS; ++i) { hipFree(n->part[i]); hipFree(n->dbias[i]); }
    for (int i = 0; i < 2; ++i)
        if (n->ev[i]) hipEventDestroy(n->ev[i]);
}

static int upload_layer(sfm_net_t* n, int l, const float* w, const float* b)
{
    const int rows = kDims[l + 1], cols = kDims[l];
    std::vector<uint16_t> wb((size_t)rows * cols), wtp((size_t)rows * cols), wp((size_t)rows * cols);
    for (int r = 0; r < rows; ++r)
        for (int c = 0; c < cols; ++c) {
            float f = w[(size_t)r * cols + c];
            uint32_t u;
            memcpy(&u, &f, 4);
            u += 0x7fffu + ((u >> 16) & 1u);
            uint16_t h = (uint16_t)(u >> 16);
            wb[(size_t)r * cols + c] = h;
            wtp[sfm::frag_index(c, r, rows)] = h;
            wp[sfm::frag_index(r, c, cols)] = h;
        }
    Layer& L = n->L[l];
    HIPCHK(hipMemcpy(L.W, w, sizeof(float) * rows * cols, hipMemcpyHostToDevice));
    HIPCHK(hipMemcpy(L.b, b, sizeof(float) * rows, hipMemcpyHostToDevice));
    HIPCHK(hipMemcpy(L.Wb, wb.data(), 2 * wb.size(), hipMemcpyHostToDevice));
    HIPCHK(hipMemcpy(L.Wtp, wtp.data(), 2 * wtp.size(), hipMemcpyHostToDevice));
    HIPCHK(hipMemcpy(L.Wp, wp.data(), 2 * wp.size(), hipMemcpyHostToDevice));
    return SFM_OK;
}

extern "C" int sfm_create(uint32_t max_batch, uint64_t seed, sfm_net* out)
{
    if (!out) return fail(SFM_ERR_INVALID, "null argument");
    if (max_batch == 0 || max_batch % kSplitK || max_batch > (1u << 22))
        return fail(SFM_ERR_SIZE, "max_batch must be a positive multiple of %d", kSplitK);
    sfm_net_t* n = new sfm_net_t();
    n->maxb = max_batch;
    int dev = 0, cus = 0;
    if (hipGetDevice(&dev) == hipSuccess &&
        hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) == hipSuccess && cus > 0)
        n->cus = (uint32_t)cus;
    auto alloc = [&](void** p, size_t bytes) -> bool {
        if (hipMalloc(p, bytes) != hipSuccess) return false;
        return hipMemset(*p, 0, bytes) == hipSuccess;
    };
    bool ok = true;
    for (int l = 0; l < SFM_LAYERS && ok; ++l) {
        const size_t nw = (size_t)kDims[l + 1] * kDims[l], nb = kDims[l + 1];
        Layer& L = n->L[l];
        ok = alloc((void**)&L.W, 4 * nw) && alloc((void**)&L.b, 4 * nb) && alloc((void**)&L.mW, 4 * nw) &&
             alloc((void**)&L.vW, 4 * nw) && alloc((void**)&L.mb, 4 * nb) && alloc((void**)&L.vb, 4 * nb) &&
             alloc((void**)&L.gW, 4 * nw) && alloc((void**)&L.gb, 4 * nb) && alloc((void**)&L.Wb, 2 * nw) &&
             alloc((void**)&L.Wtp, 2 * nw) && alloc((void**)&L.Wp, 2 * nw);
        if (ok && l > 0) ok = alloc((void**)&n->H[l], 2 * (size_t)max_batch * kDims[l]);
        if (ok) ok = alloc((void**)&n->Ht[l], 2 * (size_t)max_batch * kDims[l]) &&
                     alloc((void**)&n->dZt[l], 2 * (size_t)max_batch * kDims[l + 1]);
    }
    if (ok) ok = alloc((void**)&n->loss_part, 4 * (size_t)(max_batch / kTrainRows));
    for (int l = 0; l < SFM_LAYERS && ok; ++l)
        ok = alloc((void**)&n->part[l], 4 * (size_t)max_splits(l) * kDims[l + 1] * kDims[l]) &&
             alloc((void**)&n->dbias[l], 4 * (size_t)max_splits(l) * kDims[l + 1]);
    if (!ok) { net_free(n); delete n; return fail(SFM_ERR_HIP, "allocation failed"); }
    // Kaiming-uniform weights on the real fan-in, zero biases, padding zero
    uint64_t s = seed;
    for (int l = 0; l < SFM_LAYERS; ++l) {
        const int rows = kDims[l + 1], cols = kDims[l];
        std::vector<float> w((size_t)rows * cols, 0.f), b(rows, 0.f);
        const float bound = 1.0f / std::sqrt((float)kReal[l]);
        for (int r = 0; r < kReal[l + 1]; ++r)
            for (int c = 0; c < kReal[l]; ++c) {
                double u = (double)(splitmix(s) >> 11) * (1.0 / 9007199254740992.0);
                w[(size_t)r * cols + c] = (float)((2.0 * u - 1.0) * bound);
            }
        int rc = upload_layer(n, l, w.data(), b.data());
        if (rc != SFM_OK) { net_free(n); delete n; return rc; }
    }
    *out = n;
    return SFM_OK;
}

extern "C" int sfm_destroy(sfm_net n)
{
    if (!n) return fail(SFM_ERR_INVALID, "null network");
    hipDeviceSynchronize();
    net_free(n);
    delete n;
    return SFM_OK;
}

extern "C" int sfm_param_count(sfm_net n, uint64_t* real_params)
{
    if (!n || !real_params) return fail(SFM_ERR_INVALID, "null argument");
    uint64_t c = 0;
    for (int l = 0; l < SFM_LAYERS; ++l) c += (uint64_t)kReal[l + 1] * kReal[l] + kReal[l + 1];
    *real_params = c;
    return SFM_OK;
}

extern "C" int sfm_layer_io(sfm_net n, int l, float* w, float* b, int set)
{
    if (!n || l < 0 || l >= SFM_LAYERS || !w || !b) return fail(SFM_ERR_INVALID, "bad argument");
    HIPCHK(hipDeviceSynchronize());
    if (set) return upload_layer(n, l, w, b);
    const int rows = kDims[l + 1], cols = kDims[l];
    HIPCHK(hipMemcpy(w, n->L[l].W, sizeof(float) * rows * cols, hipMemcpyDeviceToHost));
    HIPCHK(hipMemcpy(b, n->L[l].b, sizeof(float) * rows, hipMemcpyDeviceToHost));
    return SFM_OK;
}

// Products whose rows and columns are multiples of 64 and whose K is a multiple
// of kKC run workgroup-tiled through LDS, 64 x 64 per workgroup, the 32-wide
// ones (the first layer's K, the output layer) one 32 x 32 tile per wavefront.
template <int EPI>
static void launch_gemm(const GemmArgs& g, hipStream_t s)
{
    if (g.K % kKC == 0 && g.rows % 64 == 0 && g.cols % 64 == 0)
        hipLaunchKernelGGL(k_gemm_lds<EPI>, dim3((g.rows / 64) * (g.cols / 64)), dim3(256), 0, s, g);
    else
        hipLaunchKernelGGL(k_gemm<EPI>, dim3((g.rows / 32 * (g.cols / 32) + 3) / 4), dim3(256), 0, s, g);
}

static GemmArgs gemm(const uint16_t* A, int lda, const uint16_t* Bt, int ldb, int rows, int cols, int K)
{
    GemmArgs g;
    memset(&g, 0, sizeof(g));
    g.A = A; g.lda = lda; g.Bt = Bt; g.ldb = ldb;
    g.rows = rows; g.cols = cols; g.K = K; g.ksplit = 1;
    return g;
}

static double forward_flops(uint32_t batch)
{
    double f = 0;
    for (int l = 0; l < SFM_LAYERS; ++l) f += 2.0 * kReal[l] * kReal[l + 1];
    return f * batch;
}

static void time_begin(sfm_net_t* n, hipStream_t s)
{
    if (!n->timing) return;
    if (n->pending) {
        float ms = 0.f;
        if (hipEventSynchronize(n->ev[1]) == hipSuccess && hipEventElapsedTime(&ms, n->ev[0], n->ev[1]) == hipSuccess) {
            n->ms_sum += ms;
            n->flops_sum += n->pending_flops;
            n->timed++;
        }
        n->pending = false;
    }
    hipEventRecord(n->ev[0], s);
}

static void time_end(sfm_net_t* n, hipStream_t s, double flops)
{
    if (!n->timing) return;
    hipEventRecord(n->ev[1], s);
    n->pending = true;
    n->pending_flops = flops;
}

// Forward through the hidden layers: x -> H[1..4].
static void forward_hidden(sfm_net_t* n, const uint16_t* x, uint32_t M, hipStream_t s)
{
    for (int l = 0; l < SFM_LAYERS - 1; ++l) {
        const uint16_t* A = (l == 0) ? x : n->H[l];
        GemmArgs g = gemm(A, kDims[l], n->L[l].Wb, kDims[l], (int)M, kDims[l + 1], kDims[l]);
        g.bias = n->L[l].b;
        g.H = n->H[l + 1];
        launch_gemm<EPI_HIDDEN>(g, s);
    }
}

// Inference through the fused kernel, in tiles of 32 or 64 rows.  A workgroup
// runs its tile's layers one after the other, so while every CU has at most a
// few workgroups the shorter tile is the faster (half the MFMAs and GELUs per
// wavefront); once the CUs are full the longer one is, which reads the weights
// (405 KB per tile, from L2) half as often.  Measured (tiles of 64 / 32 rows):
// 4,096 rows 15.5 / 10.4 us, 8,192 15.5 / 10.7, 16,384 15.7 / 15.7, 24,576
// 24.8 / 22.7, 32,768 26.1 / 29.6, 65,536 47.7 / 55.3 (554 TFLOP/s; 68.4 us
// with four wavefronts per workgroup).  64-row tiles only where every
// network's row count allows them.
static int forward_group(const sfm_net* nets, uint32_t nnets, const uint32_t* counts, const uint16_t* x, float* y,
                         hipStream_t s)
{
    if (!nets || !counts || !x || !y || nnets == 0) return fail(SFM_ERR_INVALID, "null argument");
    if (nnets > SFM_MAX_GROUP) return fail(SFM_ERR_SIZE, "at most %d networks per call", SFM_MAX_GROUP);
    if ((uintptr_t)x % 16) return fail(SFM_ERR_INVALID, "x must be 16-byte aligned");
    NetSet ns;
    memset(&ns, 0, sizeof(ns));
    ns.nnets = (int)nnets;
    uint64_t total = 0;
    bool even64 = true;
    for (uint32_t i = 0; i < nnets; ++i) {
        if (!nets[i]) return fail(SFM_ERR_INVALID, "null network");
        if (counts[i] % 32) return fail(SFM_ERR_SIZE, "row counts must be multiples of 32");
        even64 = even64 && counts[i] % 64 == 0;
        total += counts[i];
        if (total > (1ull << 31)) return fail(SFM_ERR_SIZE, "too many rows");
        ns.row_end[i] = (uint32_t)total;
        for (int l = 0; l < SFM_LAYERS; ++l) {
            ns.W[i][l] = nets[i]->L[l].Wp;
            ns.b[i][l] = nets[i]->L[l].b;
        }
    }
    if (total == 0) return SFM_OK;
    sfm_net_t* t = nets[0];
    const bool tiles64 = even64 && total > 3 * 32 * (uint64_t)t->cus;
    time_begin(t, s);
    if (tiles64)
        hipLaunchKernelGGL(k_mlp_fused<64>, dim3((unsigned)(total / 64)), dim3(64 * sfm::kWaves), 0, s, ns, x, (uint32_t)total, y);
    else
        hipLaunchKernelGGL(k_mlp_fused<32>, dim3((unsigned)(total / 32)), dim3(64 * sfm::kWaves), 0, s, ns, x, (uint32_t)total, y);
    time_end(t, s, forward_flops((uint32_t)total));
    HIPCHK(hipGetLastError());
    return SFM_OK;
}

extern "C" int sfm_forward(sfm_net n, const uint16_t* x, uint32_t batch, float* y, void* stream)
{
    if (!n || !x || !y) return fail(SFM_ERR_INVALID, "null argument");
    if (batch == 0 || batch % 32) return fail(SFM_ERR_SIZE, "batch must be a positive multiple of 32");
    return forward_group(&n, 1, &batch, x, y, (hipStream_t)stream);
}

extern "C" int sfm_forward_group(const sfm_net* nets, uint32_t nnets, const uint32_t* counts, const uint16_t* x,
                                 float* y, void* stream)
{
    return forward_group(nets, nnets, counts, x, y, (hipStream_t)stream);
}

// Inference through per-layer kernels (kept for checking the fused kernel
// against them).
extern "C" int sfm_forward_layers(sfm_net n, const uint16_t* x, uint32_t batch, float* y, void* stream)
{
    if (!n || !x || !y) return fail(SFM_ERR_INVALID, "null argument");
    if (batch == 0 || batch % 32 || batch > n->maxb) return fail(SFM_ERR_SIZE, "batch must be a multiple of 32 <= %u", n->maxb);
    if ((uintptr_t)x % 16) return fail(SFM_ERR_INVALID, "x must be 16-byte aligned");
    hipStream_t s = (hipStream_t)stream;
    time_begin(n, s);
    forward_hidden(n, x, batch, s);
    GemmArgs g = gemm(n->H[SFM_LAYERS - 1], SFM_HIDDEN, n->L[SFM_LAYERS - 1].Wb, SFM_HIDDEN, (int)batch, SFM_OUT_PAD,
                      SFM_HIDDEN);
    g.bias = n->L[SFM_LAYERS - 1].b;
    g.y = y;
    launch_gemm<EPI_OUT>(g, s);
    time_end(n, s, forward_flops(batch));
    HIPCHK(hipGetLastError());
    return SFM_OK;
}

extern "C" int sfm_train_step(sfm_net n, const uint16_t* x, const float* target, uint32_t batch, float lr, float beta1,
                              float beta2, float eps, float* loss, void* stream)
{
    if (!n || !x || !target || !loss) return fail(SFM_ERR_INVALID, "null argument");
    if (batch == 0 || batch % kSplitK || batch > n->maxb)
        return fail(SFM_ERR_SIZE, "batch must be a multiple of %d <= %u", kSplitK, n->maxb);
    if ((uintptr_t)x % 16) return fail(SFM_ERR_INVALID, "x must be 16-byte aligned");
    hipStream_t s = (hipStream_t)stream;
    const int M = (int)batch;
    time_begin(n, s);
    TrainArgs ta;
    memset(&ta, 0, sizeof(ta));
    ta.x = x;
    ta.target = target;
    ta.loss_part = n->loss_part;
    ta.scale = 1.0f / ((float)M * SFM_OUT);
    ta.ldt = M;
    for (int l = 0; l < SFM_LAYERS; ++l) {
        ta.W[l] = n->L[l].Wp;
        ta.Wt[l] = n->L[l].Wtp;
        ta.b[l] = n->L[l].b;
        ta.Ht[l] = n->Ht[l];
        ta.dZt[l] = n->dZt[l];
    }
    hipLaunchKernelGGL(k_train, dim3(M / kTrainRows), dim3(512), 0, s, ta);
    n->step++;
    const float bc1 = 1.0f - std::pow(beta1, (float)n->step), bc2 = 1.0f - std::pow(beta2, (float)n->step);
    // dW = dZ^T H, split over the batch: at most max_splits(l) splits, each a
    // multiple of 256 rows; their partial sums (weights and biases) are summed
    // in a fixed order by k_adam
    WgradSet wg;
    AdamSet adam;
    adam.nseg = 0;
    int nblk = 0, wblk = 0;
    for (int l = SFM_LAYERS - 1; l >= 0; --l) {
        const int dout = kDims[l + 1], din = kDims[l];
        Layer& L = n->L[l];
        int splits = 1;
        for (int d = max_splits(l); d >= 1; --d)
            if ((M / kSplitK) % d == 0) { splits = d; break; }
        const int i = SFM_LAYERS - 1 - l;
        GemmArgs& g = wg.g[i];
        g = gemm(n->dZt[l], M, n->Ht[l], M, dout, din, M);
        g.ksplit = splits;
        g.part = n->part[l];
        g.bpart = n->dbias[l];
        wg.block0[i] = wblk;
        wblk += splits * (dout % kWgradTile == 0 && din % kWgradTile == 0 ? (dout / kWgradTile) * (din / kWgradTile)
                                                                           : dout * din / (4 * 32 * 32));
        AdamSeg& sw = adam.seg[adam.nseg++];
        sw = AdamSeg{L.W, L.mW, L.vW, n->part[l], L.gW, L.Wb, L.Wtp, L.Wp, splits, dout, din, nblk};
        nblk += (dout * din + 255) / 256;
        AdamSeg& sb = adam.seg[adam.nseg++];
        sb = AdamSeg{L.b, L.mb, L.vb, n->dbias[l], L.gb, nullptr, nullptr, nullptr, splits, dout, 1, nblk};
        nblk += (dout + 255) / 256;
    }
    hipLaunchKernelGGL(k_wgrad, dim3(wblk), dim3(256), 0, s, wg);
    adam.nblk = nblk;
    adam.loss_part = n->loss_part;
    adam.nloss = M / kTrainRows;
    adam.loss = loss;
    hipLaunchKernelGGL(k_adam, dim3(nblk + 1), dim3(256), 0, s, adam, lr, beta1, beta2, eps, bc1, bc2);
    time_end(n, s, 3.0 * forward_flops(batch));
    HIPCHK(hipGetLastError());
    return SFM_OK;
}

extern "C" int sfm_gradients(sfm_net n, int l, float* dw, float* db, void* stream)
{
    if (!n || l < 0 || l >= SFM_LAYERS || !dw || !db) return fail(SFM_ERR_INVALID, "bad argument");
    hipStream_t s = (hipStream_t)stream;
    const int nw = kDims[l + 1] * kDims[l], nb = kDims[l + 1];
    hipLaunchKernelGGL(k_gradients, dim3((nw + nb + 255) / 256), dim3(256), 0, s, n->L[l].gW, n->L[l].gb, nw, nb, dw, db);
    HIPCHK(hipGetLastError());
    return SFM_OK;
}

extern "C" int sfm_to_bf16(const float* x, uint16_t* y, uint64_t n, void* stream)
{
    if ((!x || !y) && n) return fail(SFM_ERR_INVALID, "null argument");
    if (n == 0) return SFM_OK;
    hipLaunchKernelGGL(k_to_bf16, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, (hipStream_t)stream, x, y, n);
    HIPCHK(hipGetLastError());
    return SFM_OK;
}

extern "C" int sfm_probe_mfma(const uint16_t* a, const uint16_t* b, float* c, void* stream)
{
    if (!a || !b || !c) return fail(SFM_ERR_INVALID, "null argument");
    hipLaunchKernelGGL(k_probe, dim3(1), dim3(64), 0, (hipStream_t)stream, a, b, c);
    HIPCHK(hipGetLastError());
    return SFM_OK;
}

extern "C" int sfm_weights(sfm_net n, const uint16_t** w, const float** b)
{
    if (!n || !w || !b) return fail(SFM_ERR_INVALID, "null argument");
    for (int l = 0; l < SFM_LAYERS; ++l) {
        w[l] = n->L[l].Wp;
        b[l] = n->L[l].b;
    }
    return SFM_OK;
}

extern "C" int sfm_timing(sfm_net n, int enable)
{
    if (!n) return fail(SFM_ERR_INVALID, "null network");
    if (enable && !n->ev[0])
        for (int i = 0; i < 2; ++i) HIPCHK(hipEventCreate(&n->ev[i]));
    n->timing = enable != 0;
    n->pending = false;
    n->ms_sum = n->flops_sum = 0;
    n->timed = 0;
    return SFM_OK;
}

extern "C" int sfm_kernel_ms(sfm_net n, double* ms, double* flops, uint32_t* count)
{
    if (!n) return fail(SFM_ERR_INVALID, "null network");
    if (n->pending) {
        float t = 0.f;
        if (hipEventSynchronize(n->ev[1]) == hipSuccess && hipEventElapsedTime(&t, n->ev[0], n->ev[1]) == hipSuccess) {
            n->ms_sum += t;
            n->flops_sum += n->pending_flops;
            n->timed++;
        }
        n->pending = false;
    }
    if (count) *count = n->timed;
    if (ms) *ms = n->timed ? n->ms_sum / n->timed : 0.0;
    if (flops) *flops = n->timed ? n->flops_sum / n->timed : 0.0;
    return SFM_OK;
}
