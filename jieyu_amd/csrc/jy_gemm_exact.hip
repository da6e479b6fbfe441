// jy_gemm_exact.hip — prompt (m > 1) GEMMs in the reference's order, bit for bit.
//
// Quantized weights: C[i][n] = ((0 + x[i][0] w[n][0]) + x[i][1] w[n][1]) + ..., product and
// sum rounded apart, k ascending (the generic path of matmul_q, libs/matmul_libs/
// matmul_q.h:145-161), each weight dequantized as dequant_block does.  Dense [K][N] weights
// (f32, or f16 converted exactly): C = fma(x[i][k], w[k][n], C), k ascending
// (libs/matmul_libs/x86/x86_classic.txt:2-16, matmul_f16.h:19-41).
//
// The order leaves one chain per output, so the bound is VALU issue: two instructions per
// weight and token for quantized weights, one for dense.  A wave therefore computes 64
// columns (one per lane) x T tokens: the weight is a vector register, the activation is the
// same for all lanes and comes through the scalar unit (s_load), so a multiply and an add are
// all that is spent per product, with no LDS read of activations.  T is chosen per launch
// (gemm_tokens): many tokens per wave amortise the weights' dequantisation and loads, few
// give a short prompt enough waves to fill the chip.
#include <algorithm>
#include <type_traits>

#include "jy_layout.h"

namespace jy {

typedef const __attribute__((address_space(4))) float* sfloat_p;  // (uniform reads: s_load)

// k values per batch of scalar loads: the next batch's loads are issued ahead of a batch's
// arithmetic, so two batches of T x XB activations are in scalar registers
template <int T> struct XBatch { static constexpr int N = T >= 4 ? 4 : 16; };

// acc (+)= over the epilogue; the lane's column n of rows i0 .. i0 + T - 1
template <int T>
__device__ __forceinline__ void gemm_store(const float (&acc)[T], int i0, int m, int n, float* __restrict__ C, int ldc,
                                           const float* __restrict__ aux, int epi) {
    const float b = epi == EPI_BIAS ? aux[n] : 0.0f;
#pragma unroll
    for (int t = 0; t < T; t++) {
        if (i0 + t >= m) break;
        float* c = C + (size_t)(i0 + t) * ldc + n;
        if (epi == EPI_RESID)
            *c = *c + acc[t];
        else
            *c = epi == EPI_BIAS ? acc[t] + b : acc[t];
    }
}

// blocks in launch order go round the 8 XCDs: give each XCD a contiguous run of tiles, so
// that the row groups of one column tile share its L2
__device__ __forceinline__ int xcd_tile(int id, int total) {
    const int x = id & 7, q = total >> 3, r = total & 7;
    return x * q + min(x, r) + (id >> 3);
}

// ---------------------------------------------------------------- quantized weights

// One workgroup: 64 weight rows, 4 waves of T tokens.  Per 256 weights of a row (a chunk of 8
// Q8_0 blocks or one super-block) thread (slot r*16 + g of row groups 4w .. 4w + 3) holds its
// packed pieces in registers, the next chunk's loading meanwhile; per step of 64 it writes its
// 16 weights as floats to LDS, [k / 4][row][k % 4], which the four waves then read (16 bytes
// per lane per 4 k).  Two LDS buffers, one barrier per step.
static constexpr int GX_STRIDE = 64 * 16 + 64;  // bytes per 4 k (the pad spreads the writes over the banks)
static constexpr int GX_BUF = 16 * GX_STRIDE;

struct Q8Pieces {
    static constexpr int TYPE = JY_Q8_0;
    uint4 q[4], d[4];
    __device__ __forceinline__ void load(const Q8Dev& W, int rg0, int ch, int lane) {
        const int groups = W.rows_pad >> 2;
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const size_t c = (size_t)min(rg0 + i, groups - 1) * W.nchp + ch;
            q[i] = *reinterpret_cast<const uint4*>(W.qs + c * 1024 + lane * 16);
            d[i] = *reinterpret_cast<const uint4*>(W.d + c * 32 + (lane >> 4) * 8);
        }
    }
    // the weights (32-weight steps 2 jp, 2 jp + 1) x (2g, 2g + 1) of row group i, as dequant_block
    template <int JP>
    __device__ __forceinline__ void get(int i, int, float (&w)[4]) const {
        const uint32_t qw = JP == 0 ? q[i].x : JP == 1 ? q[i].y : JP == 2 ? q[i].z : q[i].w;
        const uint32_t dw = JP == 0 ? d[i].x : JP == 1 ? d[i].y : JP == 2 ? d[i].z : d[i].w;
        const float d0 = half_to_float((uint16_t)(dw & 0xffffu)), d1 = half_to_float((uint16_t)(dw >> 16));
        w[0] = (float)(int8_t)qw * d0;
        w[1] = (float)(int8_t)(qw >> 8) * d0;
        w[2] = (float)(int8_t)(qw >> 16) * d1;
        w[3] = (float)(int8_t)(qw >> 24) * d1;
    }
};

template <int TY>
struct KQPieces {
    static constexpr int TYPE = TY;
    uint2 nb[4];
    uint32_t hb[4], dm[4];
    uint4 h[4];
    __device__ __forceinline__ void load(const KQDev& W, int rg0, int ch, int lane) {
        const int r = lane >> 4;
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const size_t c = (size_t)min(rg0 + i, W.groups - 1) * W.nsb + ch;
            nb[i] = *reinterpret_cast<const uint2*>(W.nib + c * 512 + lane * 8);
            hb[i] = TY == JY_Q5_K   ? *reinterpret_cast<const uint16_t*>(W.hi + c * 128 + lane * 2)
                    : TY == JY_Q6_K ? *reinterpret_cast<const uint32_t*>(W.hi + c * 256 + lane * 4)
                                    : 0u;
            h[i] = *reinterpret_cast<const uint4*>(W.hdr + c * 64 + r * 16);
            dm[i] = W.dm[c * 4 + r];
        }
    }
    template <int JP>
    __device__ __forceinline__ void get(int i, int g, float (&w)[4]) const {
        const uint32_t nib = JP < 2 ? nb[i].x : nb[i].y;
        uint32_t wt[2] = {nib & 0x0F0F0F0Fu, (nib >> 4) & 0x0F0F0F0Fu};  // targets T = 2 (JP / 2) + u
        const float d = half_to_float((uint16_t)(dm[i] & 0xffffu));
#pragma unroll
        for (int u = 0; u < 2; u++) {
            constexpr int T0 = 2 * (JP >> 1);
            if (TY == JY_Q6_K) {
                const int sh = 2 * (T0 + u) - 4;
                wt[u] |= (sh < 0 ? hb[i] << -sh : hb[i] >> sh) & 0x30303030u;
            }
            if (TY == JY_Q5_K) wt[u] |= ((((hb[i] >> (4 * (T0 + u))) & 15u) * 0x00204081u) << 4) & 0x10101010u;
        }
#pragma unroll
        for (int e = 0; e < 2; e++) {
            const int c = 2 * JP + e, sh = 8 * (c & 3);
            if (TY == JY_Q6_K) {
                const uint32_t s = c < 4 ? (g < 8 ? h[i].x : h[i].z) : (g < 8 ? h[i].y : h[i].w);
                const float ds = d * (float)(int8_t)(s >> sh);
#pragma unroll
                for (int u = 0; u < 2; u++) w[2 * e + u] = ds * ((float)((wt[u] >> sh) & 255u) - 32.0f);
            } else {
                const float dmin = half_to_float((uint16_t)(dm[i] >> 16));
                const float d1 = d * (float)(((c < 4 ? h[i].x : h[i].y) >> sh) & 255u);
                const float n1 = dmin * (float)(((c < 4 ? h[i].z : h[i].w) >> sh) & 255u);
#pragma unroll
                for (int u = 0; u < 2; u++) w[2 * e + u] = __builtin_fmaf((float)((wt[u] >> sh) & 255u), d1, -n1);
            }
        }
    }
};

__device__ __forceinline__ int gx_rows(const Q8Dev& W) { return W.rows; }
__device__ __forceinline__ int gx_rows(const KQDev& W) { return W.rows; }

template <class Pieces, class Dev, int T>
__global__ __launch_bounds__(256) void gemm_exact_kernel(Dev W, int m, int mt, int total, const float* __restrict__ A,
                                                         float* __restrict__ C, int ldc, const float* __restrict__ aux,
                                                         int epi) {
    __shared__ __align__(16) unsigned char wsm[2 * GX_BUF];
    const int lane = threadIdx.x & 63, g = lane & 15, r = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int tile = xcd_tile(blockIdx.x, total);
    const int nt = tile / mt, i0 = (tile - nt * mt) * 4 * T + wave * T;
    const int K = W.cols, nchunk = (K + 255) / 256, rg0 = nt * 16 + wave * 4;
    // (a wave past m repeats the last row: it still stages weights; a row past m within a
    // wave likewise; neither is stored)
    sfloat_p xr[T];
#pragma unroll
    for (int t = 0; t < T; t++) xr[t] = (sfloat_p)(uintptr_t)(A + (size_t)min(i0 + t, m - 1) * K);
    float acc[T];
#pragma unroll
    for (int t = 0; t < T; t++) acc[t] = 0.0f;

    // this thread's LDS place: rows (4 wave + i) * 4 + r, k = 32 e + 2g + u of the step
    unsigned char* wp = wsm + (g >> 1) * GX_STRIDE + (wave * 16 + r) * 16 + (g & 1) * 8;
    const unsigned char* rp = wsm + lane * 16;

    constexpr int XB = XBatch<T>::N, NB = 64 / XB;
    auto compute = [&](const unsigned char* buf, int k0, int steps) {
        float4 wa[XB / 4], wb[XB / 4];
        float xa[T][XB], xb[T][XB];
        auto rd = [&](int b, float4(&w)[XB / 4], float(&x)[T][XB]) {
#pragma unroll
            for (int q = 0; q < XB / 4; q++) w[q] = *reinterpret_cast<const float4*>(buf + (b * (XB / 4) + q) * GX_STRIDE);
#pragma unroll
            for (int t = 0; t < T; t++)
#pragma unroll
                for (int e = 0; e < XB; e++) x[t][e] = xr[t][k0 + b * XB + e];
        };
        auto fm = [&](const float4(&w)[XB / 4], const float(&x)[T][XB]) {
#pragma unroll
            for (int e = 0; e < XB; e++) {
                const float4 v = w[e / 4];
                const float we = (e & 3) == 0 ? v.x : (e & 3) == 1 ? v.y : (e & 3) == 2 ? v.z : v.w;
#pragma unroll
                for (int t = 0; t < T; t++) acc[t] = __fadd_rn(acc[t], __fmul_rn(x[t][e], we));
            }
        };
        rd(0, wa, xa);
        for (int b = 0; b < steps; b += 2) {
            rd(b + 1, wb, xb);
            __builtin_amdgcn_sched_barrier(0);
            fm(wa, xa);
            rd(min(b + 2, steps - 1), wa, xa);
            __builtin_amdgcn_sched_barrier(0);
            fm(wb, xb);
        }
    };
    Pieces cur, nxt;
    cur.load(W, rg0, 0, lane);
    for (int ch = 0; ch < nchunk; ch++) {
        nxt.load(W, rg0, min(ch + 1, nchunk - 1), lane);
        const int left = K - ch * 256;  // a multiple of 32
        auto step = [&](auto jp) {
            constexpr int JP = decltype(jp)::value;
            if (JP * 64 >= left) return;  // (uniform)
            constexpr int B = (JP & 1) * GX_BUF;
#pragma unroll
            for (int i = 0; i < 4; i++) {
                float w[4];
                cur.template get<JP>(i, g, w);
                *reinterpret_cast<float2*>(wp + B + i * 64) = make_float2(w[0], w[1]);
                *reinterpret_cast<float2*>(wp + B + 8 * GX_STRIDE + i * 64) = make_float2(w[2], w[3]);
            }
            lds_barrier();
            compute(rp + B, ch * 256 + JP * 64, min(left - JP * 64, 64) / XB);
        };
        step(std::integral_constant<int, 0>());
        step(std::integral_constant<int, 1>());
        step(std::integral_constant<int, 2>());
        step(std::integral_constant<int, 3>());
        // (a chunk cut short after an odd number of steps is the last one)
        cur = nxt;
    }
    const int n = nt * 64 + lane;
    if (n < gx_rows(W)) gemm_store<T>(acc, i0, m, n, C, ldc, aux, epi);
}

// ---------------------------------------------------------------- dense weights

// One wave: the 64 columns of a panel x T tokens, weights straight from the panel (16-byte
// pieces [ceil(K / PER)][64][PER], consecutive lanes on consecutive pieces), PF pieces per
// register buffer and two buffers.  The four waves of a workgroup take the same panel.
template <typename E, int T>
__global__ __launch_bounds__(256) void gemm_dense_exact_kernel(const E* __restrict__ B, int K, int N, int m, int mt,
                                                               int total, const float* __restrict__ A,
                                                               float* __restrict__ C, int ldc,
                                                               const float* __restrict__ aux, int epi) {
    constexpr int PER = 16 / (int)sizeof(E);
    constexpr int PF = T <= 2 ? 8 : 16 / PER;     // pieces per register buffer
    constexpr int XK = T <= 2 ? 8 : 4;         // k per batch of scalar loads
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int tile = xcd_tile(blockIdx.x, total);
    const int nt = tile / mt, i0 = (tile - nt * mt) * 4 * T + wave * T;
    if (i0 >= m) return;
    const int nkb = (K + PER - 1) / PER, full = K / PER;  // pieces; whole ones
    const uint4* P = reinterpret_cast<const uint4*>(B) + (size_t)nt * nkb * 64 + lane;
    sfloat_p xr[T];
#pragma unroll
    for (int t = 0; t < T; t++) xr[t] = (sfloat_p)(uintptr_t)(A + (size_t)min(i0 + t, m - 1) * K);
    float acc[T];
#pragma unroll
    for (int t = 0; t < T; t++) acc[t] = 0.0f;
    auto elem = [](const uint4& v, int e) -> float {
        if constexpr (PER == 4) {
            return __builtin_bit_cast(float, e == 0 ? v.x : e == 1 ? v.y : e == 2 ? v.z : v.w);
        } else {
            const uint32_t w = e < 2 ? v.x : e < 4 ? v.y : e < 6 ? v.z : v.w;
            return half_to_float((uint16_t)((e & 1) ? w >> 16 : w & 0xffffu));
        }
    };
    uint4 va[PF], vb[PF];
    auto load = [&](uint4(&v)[PF], int p0) {
#pragma unroll
        for (int i = 0; i < PF; i++) v[i] = P[(size_t)min(p0 + i, nkb - 1) * 64];
    };
    // pieces p0 .. p0 + PF - 1, all whole
    auto block = [&](const uint4(&v)[PF], int p0) {
        constexpr int NX = PF * PER / XK;
        float xa[T][XK], xb[T][XK];
        auto rd = [&](int b, float(&x)[T][XK]) {
#pragma unroll
            for (int t = 0; t < T; t++)
#pragma unroll
                for (int e = 0; e < XK; e++) x[t][e] = xr[t][p0 * PER + b * XK + e];
        };
        auto fm = [&](int b, const float(&x)[T][XK]) {
#pragma unroll
            for (int e = 0; e < XK; e++) {
                const int k = b * XK + e;
                const float w = elem(v[k / PER], k % PER);
#pragma unroll
                for (int t = 0; t < T; t++) acc[t] = __builtin_fmaf(x[t][e], w, acc[t]);
            }
        };
        rd(0, xa);
#pragma unroll
        for (int b = 0; b < NX; b += 2) {
            rd(b + 1, xb);
            __builtin_amdgcn_sched_barrier(0);
            fm(b, xa);
            if (b + 2 < NX) rd(b + 2, xa);
            __builtin_amdgcn_sched_barrier(0);
            fm(b + 1, xb);
        }
    };
    load(va, 0);
    load(vb, PF);
    int p = 0;
    for (; p + 2 * PF <= full; p += 2 * PF) {
        block(va, p);
        load(va, p + 2 * PF);
        block(vb, p + PF);
        load(vb, p + 3 * PF);
    }
    // the rest, one k at a time (va, vb hold pieces p .. p + 2 PF - 1)
#pragma unroll
    for (int i = 0; i < 2 * PF; i++) {
        const uint4& v = i < PF ? va[i] : vb[i - PF];
#pragma unroll
        for (int e = 0; e < PER; e++) {
            const int k = (p + i) * PER + e;
            if (k < K) {  // (uniform)
                const float w = elem(v, e);
#pragma unroll
                for (int t = 0; t < T; t++) acc[t] = __builtin_fmaf(xr[t][k], w, acc[t]);
            }
        }
    }
    const int n = nt * 64 + lane;
    if (n < N) gemm_store<T>(acc, i0, m, n, C, ldc, aux, epi);
}

// ---------------------------------------------------------------- launches

static int g_gx_cus = 256;

hipError_t gemm_exact_init() {
    int dev = 0, cus = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e == hipSuccess) e = hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev);
    if (e == hipSuccess && cus > 0) g_gx_cus = cus;
    return e;
}

// Tokens per wave: the T of tmax, tmax / 2, ... 1 with the least time of the busiest CU, in units of one
// token's arithmetic over a workgroup (4 T tokens cost T units, staging and loads about
// `over` more).  A CU runs several workgroups at a time, so its load is the ceiling of its
// share of the grid.
static int gemm_tokens(int m, int ntiles, int tmax, float over) {
    int best = 1;
    float cost = 0.0f;
    for (int T = tmax; T >= 1; T /= 2) {
        const long wgs = (long)ntiles * ((m + 4 * T - 1) / (4 * T));
        const float c = (float)((wgs + g_gx_cus - 1) / g_gx_cus) * ((float)T + over);
        if (T == tmax || c < cost) {
            best = T;
            cost = c;
        }
    }
    return best;
}

template <class Pieces, class Dev>
static void gemm_exact(const Dev& W, int m, const float* A, float* C, int ldc, const float* aux, Epi epi,
                       hipStream_t st) {
    const int ntiles = (W.rows + 63) / 64, T = gemm_tokens(m, ntiles, 8, 1.0f);
    const int mt = (m + 4 * T - 1) / (4 * T), total = ntiles * mt;
#define JY_GX(TT)                                                                                                  \
    hipLaunchKernelGGL((gemm_exact_kernel<Pieces, Dev, TT>), dim3((unsigned)total), dim3(256), 0, st, W, m, mt, total, \
                       A, C, ldc, aux, (int)epi)
    switch (T) {
        case 8: JY_GX(8); break;
        case 4: JY_GX(4); break;
        case 2: JY_GX(2); break;
        default: JY_GX(1); break;
    }
#undef JY_GX
}

template <typename E>
static void gemm_dense(const E* B, int K, int N, int m, const float* A, float* C, int ldc, const float* aux, Epi epi,
                       hipStream_t st) {
    // (8 tokens do not fit the scalar registers: the straight-line block spills them)
    const int ntiles = (N + 63) / 64, T = gemm_tokens(m, ntiles, 4, 1.0f);
    const int mt = (m + 4 * T - 1) / (4 * T), total = ntiles * mt;
#define JY_GD(TT)                                                                                                   \
    hipLaunchKernelGGL((gemm_dense_exact_kernel<E, TT>), dim3((unsigned)total), dim3(256), 0, st, B, K, N, m, mt, total, \
                       A, C, ldc, aux, (int)epi)
    switch (T) {
        case 4: JY_GD(4); break;
        case 2: JY_GD(2); break;
        default: JY_GD(1); break;
    }
#undef JY_GD
}

void launch_gemm_q8(const Q8Dev& W, int m, const float* A, float* C, const float* aux, Epi epi, hipStream_t st) {
    gemm_exact<Q8Pieces>(W, m, A, C, W.rows, aux, epi, st);
}

void launch_gemm_f32(const float* B, int K, int N, int m, const float* A, float* C, const float* aux, Epi epi,
                     hipStream_t st) {
    gemm_dense<float>(B, K, N, m, A, C, N, aux, epi, st);
}

void launch_gemm(const DevW& W, int m, const float* A, float* C, int ldc, const float* aux, Epi epi,
                 hipStream_t st) {
    switch (W.type) {
        case JY_F32: gemm_dense(static_cast<const float*>(W.dense), W.in, W.out, m, A, C, ldc, aux, epi, st); break;
        case JY_F16: gemm_dense(static_cast<const uint16_t*>(W.dense), W.in, W.out, m, A, C, ldc, aux, epi, st); break;
        case JY_Q8_0: gemm_exact<Q8Pieces>(W.q8, m, A, C, ldc, aux, epi, st); break;
        case JY_Q4_K: gemm_exact<KQPieces<JY_Q4_K>>(W.kq, m, A, C, ldc, aux, epi, st); break;
        case JY_Q5_K: gemm_exact<KQPieces<JY_Q5_K>>(W.kq, m, A, C, ldc, aux, epi, st); break;
        default: gemm_exact<KQPieces<JY_Q6_K>>(W.kq, m, A, C, ldc, aux, epi, st); break;
    }
}

}  // namespace jy
