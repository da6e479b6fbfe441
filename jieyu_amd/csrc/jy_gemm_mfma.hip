// jy_gemm_mfma.hip — prompt (m > 1) GEMMs of Q8_0 matrices on the matrix cores, the
// tolerance mode's form of the generic matmul path (libs/matmul_libs/matmul_q.h:145-161:
// C[i][n] = sum_k A[i][k] * q[n][k] * d[n][k/32]).
//
// Numbers.  The int8 weights are exact in fp16.  Each activation row is scaled by a power
// of two that puts its largest magnitude in [2^13, 2^14) and split into an fp16 high part
// and an fp16 low part (the rounding remainder), 22 significant bits together.  Two
// v_mfma_f32_32x32x16_f16 per part give a 32-weight block's sum sum_k a[k] q[k] in fp32
// (every product exact, fp32 additions); the block's fp16 scale multiplies that sum in an
// fp32 fma into the running result, and the epilogue undoes the row's power of two.  So
// the differences from the reference's fp32 loop are the order of the fp32 additions and
// the 2^-22 relative split of the activations.
//
// Layout.  The matrix is kept a second time for these kernels (built when the mode is
// enabled): for every tile of 16 rows and every block 512 bytes, slot c + 16 g (row c of the
// tile) holding the 16 bytes k = 8 g .. 8 g + 7 and 16 + 8 g .. 16 + 8 g + 7 of the block, which
// one lane of the B operand takes at once; and the block scales as fp32, four blocks of a row
// together (zero past the last block).  v_mfma_f32_32x32x16_f16 takes 16 k from two lane
// groups of 8; lane group g of the h-th of a block's two instructions has k = 16 h + 8 g .. + 7
// in both operands, and the two in turn give bit for bit the sum that one
// v_mfma_f32_16x16x32_f16 over the block gives.
//
// Tiling.  A workgroup of 4 waves computes 32 MT rows (tokens) x 128 NT columns (matrix
// rows), each wave all the rows of its 32 NT columns.  So a wave alone uses its weights and
// takes them straight into registers (16 bytes per lane, reloaded for the next step as each
// block is used up), and only the activations, which all four share, go through LDS, by
// global -> LDS DMA, four blocks a step and two steps deep, with one barrier per step.
//
// What bounds it: at many rows, instruction issue and the vector memory path together; at few,
// the latency of a wave's chain and the weights' bytes.  Measured on the way (gate/up of
// Llama-3-8B, 28672 x 4096, 1024 rows):
//   16x16x32 tiles, everything through LDS, a barrier per block      545-565 us
//   the same with 32x32x16 tiles (16x16x32 takes 4 passes and leaves the vector unit no
//   slot beside it; 32x32x16 takes 8 and hides ~5 ns of vector work) 554
//   weights to registers, a barrier per 4 blocks                     559
//   DMA by whole 128-byte lines and 16-byte weight loads             497
// (the number of cache lines a load instruction touches was the limit: with the loads left out
// the second form took 393 us, the matrix instructions alone 328, 1.47 PFLOP/s.)
// (The kernel alone, in a loop over one matrix.  In a prompt pass it takes 513-520 us; with the
// activation split, both builds in turn, 562 -> 519, and at 61 rows 98 -> 53.)
#include <algorithm>
#include <cstddef>

#include "jy_gemm_offsets.h"
#include "jy_layout.h"
#include "jy_mfma.h"

namespace jy {

static constexpr int GM_TILE = 64;  // activation rows are padded to a multiple of this
static constexpr int GM_KB = 4;     // 32-weight blocks per step of the GEMM

typedef _Float16 h4_t __attribute__((ext_vector_type(4)));

// ---------------------------------------------------------------- the matrix copy

// one thread per (16-row tile t, block b, l): the 8 weights of row 16t + (l % 16),
// k = 32b + 8(l/16) .. +7, into half l/32 of slot (l % 16) + 16 ((l/16) % 2), from the lane-pair layout (slot r*16 + g of chunk b/8 holds
// weights 2g, 2g+1 of each of its 8 blocks at bytes 2j, 2j+1); the scales of blocks
// 4*b4 .. 4*b4+3 of each row by the threads with l < 16 and b % 4 == 0
__global__ void mfma_repack_kernel(Q8Dev W, Q8MfmaDev M) {
    const size_t id = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    const size_t total = (size_t)M.tiles * M.nb * 64;
    if (id >= total) return;
    const int l = (int)(id % 64);
    const size_t tb = id / 64;
    const int b = (int)(tb % M.nb), t = (int)(tb / M.nb);
    const int n = 16 * t + (l % 16), G = l / 16;
    uint32_t w0 = 0, w1 = 0;
    if (n < W.rows) {
        const int rg = n >> 2, r = n & 3, ch = b >> 3, j = b & 7;
        const uint8_t* chunk = W.qs + ((size_t)rg * W.nchp + ch) * 1024;
        uint32_t v[4];
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const uint8_t* s = chunk + (size_t)(r * 16 + 4 * G + i) * 16 + 2 * j;
            v[i] = (uint32_t)s[0] | ((uint32_t)s[1] << 8);
        }
        w0 = v[0] | (v[1] << 16);
        w1 = v[2] | (v[3] << 16);
    }
    uint2* dst = reinterpret_cast<uint2*>(M.q + tb * 512 + (((G & 1) * 16 + (l % 16)) * 2 + (G >> 1)) * 8);
    *dst = make_uint2(w0, w1);
    if (l < 16 && (b & 3) == 0) {
        float4 dv = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        if (n < W.rows) {
            const int rg = n >> 2, r = n & 3;
            float t4[4];
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const int bb = b + i;
                float s = 0.0f;
                if (bb < W.nb) {
                    const uint16_t h = W.d[((size_t)rg * W.nchp + (bb >> 3)) * 32 + r * 8 + (bb & 7)];
                    s = (float)__builtin_bit_cast(_Float16, h);
                }
                t4[i] = s;
            }
            dv = make_float4(t4[0], t4[1], t4[2], t4[3]);
        }
        reinterpret_cast<float4*>(M.d)[((size_t)t * M.nb4 + (b >> 2)) * 16 + l] = dv;
    }
}

void launch_mfma_repack(const Q8Dev& W, const Q8MfmaDev& M, hipStream_t st) {
    const size_t total = (size_t)M.tiles * M.nb * 64;
    hipLaunchKernelGGL(mfma_repack_kernel, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, st, W, M);
}

// ---------------------------------------------------------------- the activation split

// one row of the padded activations (LDS or global, K values; `live` false: the row past m,
// zero) into its fp16 high / low parts and its unscale, by a workgroup of 256 threads
__device__ __forceinline__ void split_row(const float* a, bool live, int K, int row, _Float16* __restrict__ hi,
                                          _Float16* __restrict__ lo, float* __restrict__ unscale, float* red) {
    const int tid = threadIdx.x;
    float amax = 0.0f;
    if (live)
        for (int k = tid; k < K; k += 256) amax = fmaxf(amax, fabsf(a[k]));
    amax = wave_max64(amax);
    if ((tid & 63) == 0) red[tid >> 6] = amax;
    __syncthreads();
    amax = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
    // 2^s with amax * 2^s in [2^13, 2^14); s kept within float's normal exponents
    int ex = 0;
    if (amax > 0.0f) frexpf(amax, &ex);
    const int s = amax > 0.0f ? min(max(14 - ex, -100), 100) : 0;
    const float up = ldexpf(1.0f, s);
    if (tid == 0) unscale[row] = ldexpf(1.0f, -s);
    _Float16* h = hi + (size_t)row * K;
    _Float16* w = lo + (size_t)row * K;
    for (int k = tid; k < K; k += 256) {
        const float v = live ? a[k] * up : 0.0f;
        const _Float16 vh = (_Float16)v;
        h[k] = vh;
        w[k] = (_Float16)(v - (float)vh);
    }
}

// one workgroup per row of the padded activations [mp][K]: rows past m are zero
__global__ __launch_bounds__(256) void mfma_split_kernel(const float* __restrict__ A, int m, int K,
                                                         _Float16* __restrict__ hi, _Float16* __restrict__ lo,
                                                         float* __restrict__ unscale) {
    __shared__ float red[4];
    split_row(A + (size_t)blockIdx.x * K, (int)blockIdx.x < m, K, blockIdx.x, hi, lo, unscale, red);
}

// the same after the row's RMSNorm (block_rmsnorm, as rmsnorm_kernel computes it, in place in
// LDS): one kernel and one pass over the row instead of two
__global__ __launch_bounds__(256) void mfma_norm_split_kernel(const float* __restrict__ X, int m, int K,
                                                              const float* __restrict__ nw, _Float16* __restrict__ hi,
                                                              _Float16* __restrict__ lo,
                                                              float* __restrict__ unscale) {
    extern __shared__ __align__(16) float xr[];
    __shared__ float red[18];
    const bool live = (int)blockIdx.x < m;
    if (live) {
        const float* x = X + (size_t)blockIdx.x * K;
        for (int i = threadIdx.x; i < K; i += 256) xr[i] = x[i];
        __syncthreads();
        block_rmsnorm(xr, K, nw, xr, red);
        __syncthreads();
    }
    split_row(xr, live, K, blockIdx.x, hi, lo, unscale, red);
}

// The same two kernels with the row in registers: NV float4s per thread (element
// 4 (tid + TH j) .. +3 in v[j], TH threads), one read of the row, 16-byte loads and 8-byte stores of
// four halves; the same arithmetic element by element (K a multiple of 4, K <= 4 TH NV).
template <int NV, int TH = 256>
__device__ __forceinline__ void split_row4(const float4 (&v)[NV], int K, int row, _Float16* __restrict__ hi,
                                           _Float16* __restrict__ lo, float* __restrict__ unscale, float* red) {
    const int tid = threadIdx.x;
    float amax = 0.0f;
#pragma unroll
    for (int j = 0; j < NV; j++)
        amax = fmaxf(amax, fmaxf(fmaxf(fabsf(v[j].x), fabsf(v[j].y)), fmaxf(fabsf(v[j].z), fabsf(v[j].w))));
    amax = wave_max64(amax);
    if ((tid & 63) == 0) red[tid >> 6] = amax;
    __syncthreads();
    amax = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
#pragma unroll
    for (int w = 4; w < TH / 64; w++) amax = fmaxf(amax, red[w]);
    int ex = 0;
    if (amax > 0.0f) frexpf(amax, &ex);
    const int s = amax > 0.0f ? min(max(14 - ex, -100), 100) : 0;
    const float up = ldexpf(1.0f, s);
    if (tid == 0) unscale[row] = ldexpf(1.0f, -s);
    _Float16* h = hi + (size_t)row * K;
    _Float16* w = lo + (size_t)row * K;
#pragma unroll
    for (int j = 0; j < NV; j++) {
        const int k4 = tid + TH * j;
        if (4 * k4 >= K) break;
        const float e[4] = {v[j].x * up, v[j].y * up, v[j].z * up, v[j].w * up};
        h4_t vh, vl;
#pragma unroll
        for (int i = 0; i < 4; i++) {
            vh[i] = (_Float16)e[i];
            vl[i] = (_Float16)(e[i] - (float)vh[i]);
        }
        *reinterpret_cast<h4_t*>(h + 4 * k4) = vh;
        *reinterpret_cast<h4_t*>(w + 4 * k4) = vl;
    }
}

template <int NV, int TH = 256>
__global__ __launch_bounds__(TH) void mfma_split4_kernel(const float* __restrict__ A, int m, int K,
                                                          _Float16* __restrict__ hi, _Float16* __restrict__ lo,
                                                          float* __restrict__ unscale) {
    __shared__ float red[TH / 64];
    const int row = blockIdx.x;
    const bool live = row < m;
    const float4* a4 = reinterpret_cast<const float4*>(A + (size_t)row * K);
    float4 v[NV];
#pragma unroll
    for (int j = 0; j < NV; j++) {
        const int k4 = threadIdx.x + TH * j;
        v[j] = live && 4 * k4 < K ? a4[k4] : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    }
    split_row4<NV, TH>(v, K, row, hi, lo, unscale, red);
}

// (kz > 1: X's rows first take the residual add of a GEMM split over K whose sum was
// deferred, X += sum of the kz partials [kz][m][K] in slice order, written back to X: the
// sum kernel's arithmetic)
template <int NV>
__global__ __launch_bounds__(256) void mfma_norm_split4_kernel(float* __restrict__ X, int m, int K,
                                                               const float* __restrict__ nw, _Float16* __restrict__ hi,
                                                               _Float16* __restrict__ lo, float* __restrict__ unscale,
                                                               const float* __restrict__ kp, int kz) {
    extern __shared__ __align__(16) float xr[];
    __shared__ float red[18];
    const int row = blockIdx.x;
    const bool live = row < m;
    float4* x4 = reinterpret_cast<float4*>(xr);
    const float4 z4 = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    // the norm weights go out first (they do not wait for the row), the row to registers
    // and to LDS for the sum of squares in the reference's lane order
    float4 w4[NV], v[NV];
    const float4* n4 = reinterpret_cast<const float4*>(nw);
    const float4* g4 = reinterpret_cast<const float4*>(X + (size_t)row * K);
#pragma unroll
    for (int j = 0; j < NV; j++) {
        const int k4 = threadIdx.x + 256 * j;
        w4[j] = live && 4 * k4 < K ? n4[k4] : z4;
        v[j] = live && 4 * k4 < K ? g4[k4] : z4;
    }
    if (kz > 1 && live) {
        const size_t mk4 = (size_t)m * K / 4;
        const float4* p4 = reinterpret_cast<const float4*>(kp) + (size_t)row * K / 4;
        float4* xw4 = reinterpret_cast<float4*>(X + (size_t)row * K);
#pragma unroll
        for (int j = 0; j < NV; j++) {
            const int k4 = threadIdx.x + 256 * j;
            if (4 * k4 >= K) break;
            float4 y = p4[k4];
            for (int z = 1; z < kz; z++) {
                const float4 t = p4[(size_t)z * mk4 + k4];
                y = make_float4(y.x + t.x, y.y + t.y, y.z + t.z, y.w + t.w);
            }
            v[j] = make_float4(v[j].x + y.x, v[j].y + y.y, v[j].z + y.z, v[j].w + y.w);
            xw4[k4] = v[j];
        }
    }
#pragma unroll
    for (int j = 0; j < NV; j++) {
        const int k4 = threadIdx.x + 256 * j;
        if (live && 4 * k4 < K) x4[k4] = v[j];
    }
    if (live) {
        __syncthreads();
        block_rms_scale(xr, K, red);
        // y = (x * scale) * w, as block_rmsnorm computes it
        const float scale = red[16];
        const bool zero = red[17] != 0.0f;
#pragma unroll
        for (int j = 0; j < NV; j++) {
            v[j].x = zero ? 0.0f : (v[j].x * scale) * w4[j].x;
            v[j].y = zero ? 0.0f : (v[j].y * scale) * w4[j].y;
            v[j].z = zero ? 0.0f : (v[j].z * scale) * w4[j].z;
            v[j].w = zero ? 0.0f : (v[j].w * scale) * w4[j].w;
        }
        __syncthreads();  // (red is reused below)
    }
    split_row4<NV>(v, K, row, hi, lo, unscale, red);
}

// float4s per thread (of 256) for a row of K (0: the scalar kernels, K not a multiple of 4 or
// past 16384; 32: 16 for each of 512 threads, up to 32768, where the caller has that form)
static int split_nv(int K, bool wide = false) {
    if (wide && K % 4 == 0 && K > 16384 && K <= 32768) return 32;
    if (K % 4 || K > 16384) return 0;
    const int n = (K + 1023) / 1024;
    return n <= 1 ? 1 : n <= 2 ? 2 : n <= 4 ? 4 : n <= 8 ? 8 : 16;
}

bool mfma_norm_split_takes_parts(int K) { return split_nv(K) != 0; }

void launch_mfma_norm_split(float* X, int m, int mp, int K, const float* nw, _Float16* hi, _Float16* lo,
                            float* unscale, hipStream_t st, const float* kp, int kz) {
    const size_t lds = (size_t)K * sizeof(float);
    switch (split_nv(K)) {
        case 1: hipLaunchKernelGGL(mfma_norm_split4_kernel<1>, dim3(mp), dim3(256), lds, st, X, m, K, nw, hi, lo, unscale, kp, kz); break;
        case 2: hipLaunchKernelGGL(mfma_norm_split4_kernel<2>, dim3(mp), dim3(256), lds, st, X, m, K, nw, hi, lo, unscale, kp, kz); break;
        case 4: hipLaunchKernelGGL(mfma_norm_split4_kernel<4>, dim3(mp), dim3(256), lds, st, X, m, K, nw, hi, lo, unscale, kp, kz); break;
        case 8: hipLaunchKernelGGL(mfma_norm_split4_kernel<8>, dim3(mp), dim3(256), lds, st, X, m, K, nw, hi, lo, unscale, kp, kz); break;
        case 16: hipLaunchKernelGGL(mfma_norm_split4_kernel<16>, dim3(mp), dim3(256), lds, st, X, m, K, nw, hi, lo, unscale, kp, kz); break;
        default:  // (callers pass no partials here: mfma_norm_split_takes_parts)
            hipLaunchKernelGGL(mfma_norm_split_kernel, dim3(mp), dim3(256), lds, st, X, m, K, nw, hi, lo, unscale);
            break;
    }
}

void launch_mfma_split(const float* A, int m, int mp, int K, _Float16* hi, _Float16* lo, float* unscale,
                       hipStream_t st) {
    switch (split_nv(K, true)) {
        case 1: hipLaunchKernelGGL(mfma_split4_kernel<1>, dim3(mp), dim3(256), 0, st, A, m, K, hi, lo, unscale); break;
        case 2: hipLaunchKernelGGL(mfma_split4_kernel<2>, dim3(mp), dim3(256), 0, st, A, m, K, hi, lo, unscale); break;
        case 4: hipLaunchKernelGGL(mfma_split4_kernel<4>, dim3(mp), dim3(256), 0, st, A, m, K, hi, lo, unscale); break;
        case 8: hipLaunchKernelGGL(mfma_split4_kernel<8>, dim3(mp), dim3(256), 0, st, A, m, K, hi, lo, unscale); break;
        case 16: hipLaunchKernelGGL(mfma_split4_kernel<16>, dim3(mp), dim3(256), 0, st, A, m, K, hi, lo, unscale); break;
        // (18944 wide, 61 rows: 33 us by the scalar kernel)
        case 32: hipLaunchKernelGGL((mfma_split4_kernel<16, 512>), dim3(mp), dim3(512), 0, st, A, m, K, hi, lo, unscale); break;
        default: hipLaunchKernelGGL(mfma_split_kernel, dim3(mp), dim3(256), 0, st, A, m, K, hi, lo, unscale); break;
    }
}

// ---------------------------------------------------------------- the GEMM

// global -> LDS DMA (16 bytes per lane: lane l writes at the M0 base + 16 l),
// issued as inline assembly: the compiler cannot tell a DMA's LDS destination from the LDS
// the waves read and would wait for every DMA before each LDS access; the kernel instead
// waits for its own DMAs explicitly before the barrier that publishes a stage.  The asm sets
// M0 itself; nothing else in these kernels uses M0 (checked in the generated code).
// (M0 is a reserved register: the compiler warns that naming it as clobbered may not be
// honoured, which is harmless here since no compiler-generated code in these kernels uses it)
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
__device__ __forceinline__ void dma_b128(const void* g, uint32_t lds) {
    asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off" ::"v"(g), "s"(lds) : "memory", "m0");
}
#pragma clang diagnostic pop
__device__ __forceinline__ uint32_t lds_byte_addr(const void* p) {
    return (uint32_t)(uintptr_t)(__attribute__((address_space(3))) const unsigned char*)p;
}

// s_waitcnt with only vmcnt <= n (n < 64)
template <int N>
__device__ __forceinline__ void wait_vm() {
    static_assert(N >= 0 && N < 64, "vmcnt");
    __builtin_amdgcn_s_waitcnt((N & 0xF) | ((N >> 4) << 14) | (0x7 << 4) | (0xF << 8));
}

template <int EPI, int MT, int NT>
__global__ __launch_bounds__(256, 2) void gemm_q8_mfma_kernel(
    Q8MfmaDev W, int m, int K, int mtiles, int total, int nbz, const _Float16* __restrict__ ahi,
    const _Float16* __restrict__ alo, const float* __restrict__ unscale, float* __restrict__ C, int ldc,
    const float* __restrict__ aux) {
    constexpr int KB = GM_KB, NW = 4, R = 32 * MT, CC = 32 * NT * NW, RT = R / 16;
    constexpr int NA = 2 * KB * RT / NW;  // DMA instructions per wave and step
    extern __shared__ __align__(16) unsigned char gsmem[];
    h8_t(*As)[2][RT][KB][64] = reinterpret_cast<h8_t(*)[2][RT][KB][64]>(gsmem);  // [buffer][part][row tile][block][lane]
    constexpr uint32_t ABUF = 2u * RT * KB * 1024;
    const int tid = threadIdx.x, l = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int tile = xcd_tile(blockIdx.x, total);
    const int ct = tile / mtiles;
    const int rowt = (tile - ct * mtiles) * R;  // the workgroup's first token row
    const int tilet = ct * (CC / 16) + wave * 2 * NT;  // the wave's first 16-column tile
    const int nb = W.nb;
    // the workgroup's K slice: blocks [b0, b1), its sums into C's slice y ([z][m][ldc]: the
    // partials a sum kernel adds); in steps of KB blocks from the multiple of KB at or before b0
    const int b0 = (int)blockIdx.y * nbz, b1 = min(nb, b0 + nbz);
    C += (size_t)blockIdx.y * m * ldc;
    const uint32_t base = __builtin_amdgcn_readfirstlane(lds_byte_addr(gsmem));

    // One DMA instruction brings 8 rows x 128 bytes (two blocks): row l / 8, and of its eight
    // 16-byte pieces the one of slot l % 8, slots being pieces exchanged by the row's low bits
    // (piece = slot ^ row % 8), so that the fragment reads spread over the banks.
    static_assert(KB == 4 && NA % 4 == 0, "whole 16-row tiles per wave: 8-row halves x block pairs");
    const _Float16* asrc[NA / 4];
#pragma unroll
    for (int j = 0; j < NA / 4; j++) {
        const int i = wave * (NA / 4) + j, part = i / RT, rt = i % RT;
        asrc[j] = (part ? alo : ahi) + (size_t)(rowt + 16 * rt + (l >> 3)) * K;
    }
    const int apc = 8 * ((l & 7) ^ (l >> 3));
    auto issue_a = [&](int b, int buf) {
#pragma unroll
        for (int j = 0; j < NA / 4; j++)
#pragma unroll
            for (int i = 0; i < 4; i++)  // i & 1: rows + 8; i >> 1: blocks + 2
                dma_b128(asrc[j] + (size_t)(i & 1) * 8 * K + min(32 * (b + 2 * (i >> 1)) + apc, K - 8),
                         base + buf * ABUF + (uint32_t)((wave * (NA / 4) + j) * 4 + 2 * (i >> 1) + (i & 1)) * 1024);
    };
    // this lane's column: tile (l & 31) / 16 of a pair, row l % 16 of it; its k: 8 (l / 32) + 16 h .. +7, h = 0, 1.
    // Every load is inside the copy by its own offsets (jy_gemm_offsets.h)
    const int t0 = gm_base_tile(tilet, W.tiles);
    const __amdgpu_buffer_rsrc_t qr = __builtin_amdgcn_make_buffer_rsrc(
        W.q + (size_t)t0 * nb * 512, 0, (int)min((size_t)(W.tiles - t0) * nb * 512, (size_t)0x7fffffff), 0x00020000);
    const __amdgpu_buffer_rsrc_t dr = __builtin_amdgcn_make_buffer_rsrc(
        W.d + (size_t)t0 * W.nb4 * 64, 0, (int)min((size_t)(W.tiles - t0) * W.nb4 * 256, (size_t)0x7fffffff), 0x00020000);
    int qo[NT], dof[NT];
#pragma unroll
    for (int nt = 0; nt < NT; nt++) {
        qo[nt] = gm_q_lane(tilet, nt, l, W.tiles, nb);
        dof[nt] = gm_d_lane(tilet, nt, l, W.tiles, W.nb4);
    }
    uint4 q[KB][NT];
    float4 dcur[NT], dnxt[NT];
    auto load_b = [&](int b, int kb) {
#pragma unroll
        for (int nt = 0; nt < NT; nt++)
            q[kb][nt] = __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(qr, qo[nt], gm_q_block(b + kb, nb), 0));
    };
    auto load_d = [&](int b, float4(&d)[NT]) {
#pragma unroll
        for (int nt = 0; nt < NT; nt++)
            d[nt] = __builtin_bit_cast(float4, __builtin_amdgcn_raw_buffer_load_b128(dr, dof[nt], gm_d_block(b, W.nb4), 0));
    };
    // the scales of the step at b, zero outside the slice (where they are first used: at the load the
    // step would wait for it)
    auto take_d = [&](int b) {
#pragma unroll
        for (int nt = 0; nt < NT; nt++) {
            const float4 v = dnxt[nt];
            dcur[nt] = make_float4(b >= b0 && b < b1 ? v.x : 0.0f, b + 1 >= b0 && b + 1 < b1 ? v.y : 0.0f,
                                   b + 2 >= b0 && b + 2 < b1 ? v.z : 0.0f, b + 3 >= b0 && b + 3 < b1 ? v.w : 0.0f);
        }
    };

    auto mm = [](h8_t a, h8_t b, f16_t c) { return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0); };
    f16_t acc[MT][NT];
#pragma unroll
    for (int mt = 0; mt < MT; mt++)
#pragma unroll
        for (int nt = 0; nt < NT; nt++) acc[mt][nt] = f16_t(0.0f);
    // fragment address: 16-row tile (l & 31) / 16, row l % 16 in it, piece 4 (kb % 2) + 2 h + l / 32
    const int fr = ((l & 31) >> 4) * 4 * 64 + ((l >> 3) & 1) * 64 + (l & 7) * 8;
    auto block = [&](int buf, int kb) {
        h8_t ah[MT][2], al[MT][2];
#pragma unroll
        for (int mt = 0; mt < MT; mt++)
#pragma unroll
            for (int h = 0; h < 2; h++) {
                const int sl = fr + ((4 * (kb & 1) + 2 * h + (l >> 5)) ^ (l & 7)) + (kb >> 1) * 128;
                ah[mt][h] = (&As[buf][0][mt * 2][0][0])[sl];
                al[mt][h] = (&As[buf][1][mt * 2][0][0])[sl];
            }
#pragma unroll
        for (int nt = 0; nt < NT; nt++) {
            const h8_t bq[2] = {q8_to_h8(q[kb][nt].x, q[kb][nt].y), q8_to_h8(q[kb][nt].z, q[kb][nt].w)};
            const float dv = f4_get(dcur[nt], kb);
            f16_t t[MT];
            // (high parts first; the low parts ahead of them: error against 64 bits 1-3 % larger)
#pragma unroll
            for (int mt = 0; mt < MT; mt++) t[mt] = mm(ah[mt][0], bq[0], f16_t(0.0f));
#pragma unroll
            for (int mt = 0; mt < MT; mt++) t[mt] = mm(ah[mt][1], bq[1], t[mt]);
#pragma unroll
            for (int mt = 0; mt < MT; mt++) t[mt] = mm(al[mt][0], bq[0], t[mt]);
#pragma unroll
            for (int mt = 0; mt < MT; mt++) t[mt] = mm(al[mt][1], bq[1], t[mt]);
#pragma unroll
            for (int mt = 0; mt < MT; mt++)
#pragma unroll
                for (int i = 0; i < 16; i++) acc[mt][nt][i] = __builtin_fmaf(dv, t[mt][i], acc[mt][nt][i]);
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    // (a step's blocks outside the slice: their scales are zero, their activations and weights
    // the neighbours' or, past the matrix, repeated)
    if (b0 < b1) {
        const int s0 = b0 / KB * KB;
        issue_a(s0, 0);
#pragma unroll
        for (int kb = 0; kb < KB; kb++) load_b(s0, kb);
        load_d(s0, dnxt);
        take_d(s0);
        int buf = 0;
        for (int b = s0; b < b1; b += KB, buf ^= 1) {
            wait_vm<0>();
            __syncthreads();  // this step's activations are in LDS; the other buffer is read
            if (b + KB < b1) issue_a(b + KB, buf ^ 1);
            load_d(b + KB, dnxt);
#pragma unroll
            for (int kb = 0; kb < KB; kb++) {
                block(buf, kb);
                load_b(b + KB, kb);
                __builtin_amdgcn_sched_barrier(0);
            }
            take_d(b + KB);
        }
    }

    // epilogue: acc[mt][nt][i] is C[row][col] before the row's unscale (row 8 (i / 4) + 4 (l / 32) + i % 4 and
    // column l % 32 of the tile)
    const int N = W.rows;
#pragma unroll
    for (int mt = 0; mt < MT; mt++) {
        const int r0 = rowt + mt * 32 + 4 * (l >> 5);
        float us[16];
#pragma unroll
        for (int i = 0; i < 16; i++) us[i] = unscale[r0 + 8 * (i >> 2) + (i & 3)];
#pragma unroll
        for (int nt = 0; nt < NT; nt++) {
            const int col = 16 * tilet + nt * 32 + (l & 31);
            if (EPI == EPI_SWIGLU) {
                // the gate/up matrix's rows 2j, 2j+1 are gate_j, up_j: columns 2j and 2j+1 of C lie in
                // lanes c and c + 1 of a tile; the even lane writes h[row][j] = silu(gate) * up with
                // the reference's SiLU of element row * F + j of the m x F array (silu_mul_kernel)
                const int F = N >> 1;
#pragma unroll
                for (int i = 0; i < 16; i++) {
                    const int row = r0 + 8 * (i >> 2) + (i & 3);
                    const float y = acc[mt][nt][i] * us[i];
                    const float up = __shfl_xor(y, 1);
                    if (!(l & 1) && col + 1 < N && row < m) {
                        const int j = col >> 1;
                        C[(size_t)row * ldc + j] = silu_at(y, (size_t)row * F + j, (size_t)m * F) * up;
                    }
                }
                continue;
            }
            if (col >= N) continue;
            const float bias = EPI == EPI_BIAS ? aux[col] : 0.0f;
            float old[16];
            if (EPI == EPI_RESID) {
#pragma unroll
                for (int i = 0; i < 16; i++) {
                    const int row = r0 + 8 * (i >> 2) + (i & 3);
                    old[i] = row < m ? C[(size_t)row * ldc + col] : 0.0f;
                }
            }
#pragma unroll
            for (int i = 0; i < 16; i++) {
                const int row = r0 + 8 * (i >> 2) + (i & 3);
                if (row >= m) continue;
                const float y = acc[mt][nt][i] * us[i];
                C[(size_t)row * ldc + col] = EPI == EPI_RESID ? old[i] + y : y + bias;
            }
        }
    }
}

int mfma_rows_padded(int m) { return (m + GM_TILE - 1) / GM_TILE * GM_TILE; }

// ---------------------------------------------------------------- split over K
//
// A small grid that leaves CUs idle, each wave walking a long chain of blocks alone,
// runs as Z slices of K (gridDim.y), each writing its partial sums [z][m][N] (plain stores),
// then gemm_ksum_kernel adds the partials in slice order and applies the epilogue: the same
// result for every run, whatever order the slices finish in.

static constexpr int KSPLIT_MAX = 8;         // slices
static constexpr int KSPLIT_MIN_BLOCKS = 8;  // 32-weight blocks per slice, at least

template <int EPI>
__global__ __launch_bounds__(256) void gemm_ksum_kernel(const float* __restrict__ P, int Z, int m, int N,
                                                        float* __restrict__ C, int ldc, const float* __restrict__ aux) {
    const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
    const size_t mn = (size_t)m * N;
    if (i >= mn) return;
    const int row = (int)(i / N), col = (int)(i - (size_t)row * N);
    float v[KSPLIT_MAX];
#pragma unroll
    for (int z = 0; z < KSPLIT_MAX; z++) v[z] = z < Z ? P[(size_t)z * mn + i] : 0.0f;
    float y = v[0];
#pragma unroll
    for (int z = 1; z < KSPLIT_MAX; z++)
        if (z < Z) y += v[z];
    float* c = C + (size_t)row * ldc + col;
    if (EPI == EPI_RESID)
        *c = *c + y;
    else if (EPI == EPI_BIAS)
        *c = y + aux[col];
    else
        *c = y;
}

template <int MT>
static constexpr size_t gm_lds() {
    return (size_t)2 * 2 * (2 * MT) * GM_KB * 1024;  // two steps of both parts
}

template <int MT, int NT>
static void gemm_launch(const Q8MfmaDev& W, int m, const _Float16* hi, const _Float16* lo, const float* unscale,
                        float* C, int ldc, const float* aux, Epi epi, hipStream_t st, int nbz) {
    const int mtiles = (m + 32 * MT - 1) / (32 * MT), total = mtiles * ((W.tiles + 8 * NT - 1) / (8 * NT));
    const dim3 grid((unsigned)total, (unsigned)((W.nb + nbz - 1) / nbz));
    const int K = W.nb * 32;
#define JY_GM(E)                                                                                                     \
    hipLaunchKernelGGL((gemm_q8_mfma_kernel<E, MT, NT>), grid, dim3(256), gm_lds<MT>(), st, W, m, K, mtiles, total, \
                       nbz, hi, lo, unscale, C, ldc, aux)
    switch (epi) {
        case EPI_BIAS: JY_GM(EPI_BIAS); break;
        case EPI_RESID: JY_GM(EPI_RESID); break;
        case EPI_SWIGLU: JY_GM(EPI_SWIGLU); break;
        default: JY_GM(EPI_STORE); break;
    }
#undef JY_GM
}

template <int MT, int NT>
static hipError_t gemm_attr() {
    hipError_t e = hipSuccess;
    for (const void* f : {reinterpret_cast<const void*>(&gemm_q8_mfma_kernel<EPI_STORE, MT, NT>),
                          reinterpret_cast<const void*>(&gemm_q8_mfma_kernel<EPI_BIAS, MT, NT>),
                          reinterpret_cast<const void*>(&gemm_q8_mfma_kernel<EPI_RESID, MT, NT>),
                          reinterpret_cast<const void*>(&gemm_q8_mfma_kernel<EPI_SWIGLU, MT, NT>)})
        if (e == hipSuccess) e = hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, (int)gm_lds<MT>());
    return e;
}

hipError_t gemm_mfma_init() {
    hipError_t e = gemm_attr<1, 1>();
    if (e == hipSuccess) e = gemm_attr<1, 2>();
    if (e == hipSuccess) e = gemm_attr<2, 1>();
    if (e == hipSuccess) e = gemm_attr<2, 2>();
    return e;
}

static int g_gemm_cus = 0;

static int gemm_cus() {
    if (!g_gemm_cus) {
        int dev = 0, cus = 0;
        if (hipGetDevice(&dev) == hipSuccess &&
            hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) == hipSuccess && cus > 0)
            g_gemm_cus = cus;
        else
            g_gemm_cus = 256;
    }
    return g_gemm_cus;
}

// K slices for C = A W^T over m rows: 1 unless 64 x 128 tiles (rows padded to 128) are fewer
// than the CUs; then up to two such tiles per CU, at most KSPLIT_MAX slices of at least
// KSPLIT_MIN_BLOCKS blocks, none of them empty.  The count does not follow the tile chosen
// below: it decides the rounding (4096 x 4096: error against 64 bits 2.1e-7 unsplit, 1.3e-7
// with 4), and the partial sums' room, which callers with a small fixed workspace count on.
// (The SwiGLU epilogue pairs columns and is not split.)
int gemm_q8_mfma_ksplit(const Q8MfmaDev& W, int m, Epi epi) {
    const int cus = gemm_cus();
    const long wgs = (long)((m + 127) / 128 * 2) * ((W.tiles + 7) / 8);
    if (epi == EPI_SWIGLU || wgs >= cus) return 1;
    const int z = (int)std::min<long>(std::min<long>(KSPLIT_MAX, 2L * cus / std::max(1L, wgs)),
                                      W.nb / KSPLIT_MIN_BLOCKS);
    if (z < 2) return 1;
    const int nbz = (W.nb + z - 1) / z;
    return (W.nb + nbz - 1) / nbz;
}

// The tile (32 MT rows x 128 NT columns per workgroup) of a launch with z slices: the least
// max(lat, thr x the busiest CU's workgroups + off), where lat is a lone workgroup's ns per
// block and thr the ns per block and workgroup of a full CU (32 x 256 gains on 64 x 128 from
// three workgroups: 6144 x 4096 at 1024 rows 120 us against 133; at two, 4096 x 14336, 285
// against 272).  Measured at 28672 x 4096, 6144 x
// 4096, 4096 x 4096, 4096 x 14336, 37888 x 3584, 9728 x 896, 1152 x 896 and 896 x 4864, 61 to
// 1024 rows.
struct GmTile {
    int mt, nt;
    float lat, thr, off;
};
static GmTile gemm_tile(const Q8MfmaDev& W, int m, int z) {
    static constexpr GmTile tiles[] = {{2, 2, 640.0f, 550.0f, 0.0f}, {2, 1, 400.0f, 312.0f, 0.0f},
                                       {1, 2, 400.0f, 290.0f, 60.0f}, {1, 1, 275.0f, 170.0f, 0.0f}};
    const int cus = gemm_cus();
    GmTile best{};
    float cost = 0.0f;
    for (const GmTile& t : tiles) {
        const long wgs = (long)((m + 32 * t.mt - 1) / (32 * t.mt)) * ((W.tiles + 8 * t.nt - 1) / (8 * t.nt)) * z;
        const float c = std::max(t.lat, t.thr * (float)((wgs + cus - 1) / cus) + t.off);
        if (!best.mt || c < cost) {
            cost = c;
            best = t;
        }
    }
    return best;
}

size_t gemm_q8_mfma_kpart_floats(const Q8MfmaDev& W, int m, Epi epi) {
    const int z = gemm_q8_mfma_ksplit(W, m, epi);
    return z > 1 ? (size_t)z * m * W.rows : 0;
}

int launch_gemm_q8_mfma(const Q8MfmaDev& W, int m, const _Float16* hi, const _Float16* lo, const float* unscale,
                        float* C, int ldc, const float* aux, Epi epi, hipStream_t st, float* kpart, size_t kpart_n,
                        bool defer) {
    int Z = gemm_q8_mfma_ksplit(W, m, epi);
    if (Z > 1 && (!kpart || (size_t)Z * m * W.rows > kpart_n)) Z = 1;
    const GmTile g = gemm_tile(W, m, Z);
    const int nbz = (W.nb + Z - 1) / Z;
    auto run = [&](float* out, int ld, const float* ax, Epi e) {
        if (g.mt == 2 && g.nt == 2)
            gemm_launch<2, 2>(W, m, hi, lo, unscale, out, ld, ax, e, st, nbz);
        else if (g.mt == 2)
            gemm_launch<2, 1>(W, m, hi, lo, unscale, out, ld, ax, e, st, nbz);
        else if (g.nt == 2)
            gemm_launch<1, 2>(W, m, hi, lo, unscale, out, ld, ax, e, st, nbz);
        else
            gemm_launch<1, 1>(W, m, hi, lo, unscale, out, ld, ax, e, st, nbz);
    };
    if (Z < 2) {
        run(C, ldc, aux, epi);
        return 0;
    }
    run(kpart, W.rows, nullptr, EPI_STORE);
    if (defer) return Z;
    const size_t n = (size_t)m * W.rows;
    const dim3 grid((unsigned)((n + 255) / 256));
    switch (epi) {
        case EPI_BIAS:
            hipLaunchKernelGGL(gemm_ksum_kernel<EPI_BIAS>, grid, dim3(256), 0, st, kpart, Z, m, W.rows, C, ldc, aux);
            break;
        case EPI_RESID:
            hipLaunchKernelGGL(gemm_ksum_kernel<EPI_RESID>, grid, dim3(256), 0, st, kpart, Z, m, W.rows, C, ldc, aux);
            break;
        default:
            hipLaunchKernelGGL(gemm_ksum_kernel<EPI_STORE>, grid, dim3(256), 0, st, kpart, Z, m, W.rows, C, ldc, aux);
            break;
    }
    return 0;
}

void launch_gemm_ksum(const float* kpart, int Z, int m, int N, float* C, int ldc, const float* aux, Epi epi,
                      hipStream_t st) {
    const dim3 grid((unsigned)(((size_t)m * N + 255) / 256));
    if (epi == EPI_RESID)
        hipLaunchKernelGGL(gemm_ksum_kernel<EPI_RESID>, grid, dim3(256), 0, st, kpart, Z, m, N, C, ldc, aux);
    else if (epi == EPI_BIAS)
        hipLaunchKernelGGL(gemm_ksum_kernel<EPI_BIAS>, grid, dim3(256), 0, st, kpart, Z, m, N, C, ldc, aux);
    else
        hipLaunchKernelGGL(gemm_ksum_kernel<EPI_STORE>, grid, dim3(256), 0, st, kpart, Z, m, N, C, ldc, aux);
}

}  // namespace jy
