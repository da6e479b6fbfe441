// jy_gemm_exact.hip — prompt (m > 1) GEMMs in the reference's order, bit for bit.
//
// Quantized weights: C[i][n] = ((0 + x[i][0] w[n][0]) + x[i][1] w[n][1]) + ..., product and
// sum rounded apart, k ascending (the generic path of matmul_q, libs/matmul_libs/
// matmul_q.h:145-161), each weight dequantized as dequant_block does.  Dense [K][N] weights
// (f32, or f16 converted exactly): C = fma(x[i][k], w[k][n], C), k ascending
// (libs/matmul_libs/x86/x86_classic.txt:2-16, matmul_f16.h:19-41).
//
// The order leaves one chain per output, so the bound is instruction issue: a multiply and an
// add per weight and token for quantized weights, a fused multiply-add for dense.  A lane keeps
// a column and a wave T tokens of 64 columns, in two forms:
//   vector unit   the activation is the same for all lanes and comes through the scalar unit;
//   matrix unit   v_mfma_f32_{16x16x1_4b, 4x4x1_16b}: each value is one product, rounded as a
//                 multiply rounds it, or with the sum as addend the fused multiply-add
//                 (compared bit for bit over 50 M operand pairs, subnormals and infinities
//                 among them).  The activations come 16 bytes per lane, and nothing waits on
//                 scalar loads, which return out of order and so can only be waited for all.
// The single-precision matrix instructions take the vector unit's time (16 x 64 products
// 14 ns per SIMD, their 16 adds 17 ns, both together 30; 16 multiplies and adds 29 with two
// waves per SIMD), so the gain is the loads', not the arithmetic's.  T and the form are chosen
// per launch (gemm_form) from times measured per k.
// Llama-3-8B Q8_0, 200 rows, 64 x 64 tiles through LDS -> now (both builds in turn): gate/up 28672 x
// 4096 1423 -> 1072 us, QKV 6144 x 4096 577 -> 302, O 4096 x 4096 560 -> 226, down 4096 x 14336 1912 -> 765.
#include <algorithm>
#include <type_traits>

#include "jy_layout.h"
#include "jy_mfma.h"

namespace jy {

typedef const __attribute__((address_space(4))) float* sfloat_p;  // (uniform reads: s_load)

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

// this thread's 16 weights of step JP of a chunk, dequantized into LDS
template <int JP, class Pieces>
__device__ __forceinline__ void gx_stage(const Pieces& p, int g, unsigned char* wp) {
#pragma unroll
    for (int i = 0; i < 4; i++) {
        float w[4];
        p.template get<JP>(i, g, w);
        *reinterpret_cast<float2*>(wp + i * 64) = make_float2(w[0], w[1]);
        *reinterpret_cast<float2*>(wp + 8 * GX_STRIDE + i * 64) = make_float2(w[2], w[3]);
    }
}

// One or two tokens per wave: multiply and add in the vector unit.
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

    constexpr int XB = 16, NB = 64 / XB;
    static_assert(T <= 2 && NB == 4, "two batches of T x XB activations are in scalar registers");
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
            gx_stage<JP>(cur, g, wp + B);
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

// ---- the products on the matrix cores
//
// v_mfma_f32_{16x16x1_4b, 4x4x1_16b} with a zero addend is an outer product whose values are
// each rounded once, as a multiply's are (subnormals, infinities and all): TT tokens x 64
// columns (one per lane of B) of one k per instruction, and the vector unit adds it to the
// sums.  The product takes the vector unit's time all the same (at the top); what is gained are the
// activations, 16 bytes per lane instead of scalar loads.  One register of A holds 64 / TT k of the TT
// tokens (lane TT j + t: token t), of which the instruction's broadcast picks one (ABID j).

template <int TT> struct Outer;
template <> struct Outer<16> {
    typedef f16_t vec;
    template <int J> static __device__ __forceinline__ vec mm(float a, float b, vec c) {
        return __builtin_amdgcn_mfma_f32_16x16x1f32(a, b, c, 2, J, 0);
    }
    // register i of the product in lane l
    static __device__ __forceinline__ int token(int i, int l) { return 4 * (l >> 4) + (i & 3); }
    static __device__ __forceinline__ int col(int i, int l) { return 16 * (i >> 2) + (l & 15); }
};
template <> struct Outer<4> {
    typedef f4_t vec;
    template <int J> static __device__ __forceinline__ vec mm(float a, float b, vec c) {
        return __builtin_amdgcn_mfma_f32_4x4x1f32(a, b, c, 4, J, 0);
    }
    static __device__ __forceinline__ int token(int i, int) { return i; }
    static __device__ __forceinline__ int col(int, int l) { return l; }
};

template <int I, int N, class F>
__device__ __forceinline__ void static_for(F&& f) {
    if constexpr (I < N) {
        f(std::integral_constant<int, I>());
        static_for<I + 1, N>(f);
    }
}

// the epilogue of MT tiles of TT tokens x 64 columns
template <int TT, int MT>
__device__ __forceinline__ void outer_store(const typename Outer<TT>::vec (&acc)[MT], int i0, int m, int n0, int N,
                                            float* __restrict__ C, int ldc, const float* __restrict__ aux, int epi) {
    const int l = threadIdx.x & 63;
#pragma unroll
    for (int mt = 0; mt < MT; mt++)
#pragma unroll
        for (int i = 0; i < TT; i++) {
            const int row = i0 + TT * mt + Outer<TT>::token(i, l), n = n0 + Outer<TT>::col(i, l);
            if (row >= m || n >= N) continue;
            float* c = C + (size_t)row * ldc + n;
            const float v = acc[mt][i];
            if (epi == EPI_RESID)
                *c = *c + v;
            else
                *c = epi == EPI_BIAS ? v + aux[n] : v;
        }
}

// (registers for three or four workgroups per CU: a lone wave issues a vector instruction per
// 2.05 ns, two or more waves of a SIMD together one per 0.94.  The packed pieces of the next chunk
// replace this one's once its last step is staged, and the activations are reloaded piece by piece
// as they are used up.  Within those registers the 16-token form spills 2 (Q8_0), 6 (Q4_K), 25
// (Q5_K) and 23 (Q6_K), the 8-token form 4 (Q5_K) and 6 (Q6_K) registers.)
template <class Pieces, class Dev, int TT, int MT>
__global__ __launch_bounds__(256, TT == 16 ? 3 : 4) void gemm_exact_mm_kernel(
    Dev W, int m, int mt, int total, const float* __restrict__ A, float* __restrict__ C, int ldc,
    const float* __restrict__ aux, int epi) {
    typedef Outer<TT> O;
    typedef typename O::vec vec;
    constexpr int T = TT * MT, KA = 4 * 64 / TT, NL = 64 / KA;  // k per 16-byte load of A; loads per step of 64 k
    __shared__ __align__(16) unsigned char wsm[2 * GX_BUF];
    const int lane = threadIdx.x & 63, g = lane & 15, r = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int tile = xcd_tile(blockIdx.x, total);
    const int nt = tile / mt, mi = tile - nt * mt;
    // the tile's token groups are dealt to the mt workgroups in turn, and within one to the
    // waves from a rotating first, so that waves without tokens (they only stage weights) are
    // spread over workgroups and SIMDs
    const int i0 = (mi + mt * ((wave + tile) & 3)) * T;
    const int K = W.cols, nchunk = (K + 255) / 256, rg0 = nt * 16 + wave * 4;
    const bool live = i0 < m;
    const float* ar[MT];
#pragma unroll
    for (int t = 0; t < MT; t++) ar[t] = A + (size_t)min(i0 + TT * t + (lane & (TT - 1)), m - 1) * K;
    const int ak = 4 * (lane / TT);
    vec acc[MT];
#pragma unroll
    for (int t = 0; t < MT; t++) acc[t] = vec(0.0f);

    unsigned char* wp = wsm + (g >> 1) * GX_STRIDE + (wave * 16 + r) * 16 + (g & 1) * 8;
    const unsigned char* rp = wsm + lane * 16;

    // activations k0 + KA i .. of a step, 16 bytes per lane and tile; past the row (a last
    // step of 32 k, the step after the last): its last 4 values, unused
    float4 a[MT][NL];
    auto load_a = [&](int k0, int i) {
#pragma unroll
        for (int t = 0; t < MT; t++) a[t][i] = *reinterpret_cast<const float4*>(ar[t] + min(k0 + KA * i + ak, K - 4));
    };
    // a step's first N / MT k from LDS: the product of the next (k, tile) is issued ahead of
    // the adds of this one, two ahead for the short 4 x 4 instruction
    auto compute = [&](auto kc, const unsigned char* buf, int k0) {
        constexpr int KS = decltype(kc)::value, N = KS * MT, D = TT == 4 ? 2 : 1;
        float4 w[2];
        vec p[D + 1];
        w[0] = *reinterpret_cast<const float4*>(buf);
        auto prod = [&](auto ic) {
            constexpr int I = decltype(ic)::value, k = I / MT, t = I % MT;
            if constexpr (t == 0 && k % 4 == 0 && k + 4 < KS)
                w[(k / 4 + 1) & 1] = *reinterpret_cast<const float4*>(buf + (k / 4 + 1) * GX_STRIDE);
            p[I % (D + 1)] = O::template mm<(k % KA) / 4>(f4_get(a[t][k / KA], k % 4), f4_get(w[(k / 4) & 1], k % 4),
                                                          vec(0.0f));
            if constexpr (t == MT - 1 && (k + 1) % KA == 0) load_a(k0 + 64, k / KA);
        };
        static_for<0, D>(prod);
        static_for<0, N>([&](auto ic) {
            constexpr int I = decltype(ic)::value;
            if constexpr (I + D < N) prod(std::integral_constant<int, I + D>());
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int e = 0; e < TT; e++) acc[I % MT][e] = __fadd_rn(acc[I % MT][e], p[I % (D + 1)][e]);
            __builtin_amdgcn_sched_barrier(0);
        });
    };
    Pieces cur;
    cur.load(W, rg0, 0, lane);
#pragma unroll
    for (int i = 0; i < NL; i++) load_a(0, i);
    for (int ch = 0; ch < nchunk; ch++) {
        const int steps = (min(K - ch * 256, 256) + 63) / 64;
        for (int jp = 0; jp < steps; jp++) {
            const int B = (jp & 1) * GX_BUF, k0 = ch * 256 + jp * 64;
            switch (jp) {  // (uniform)
                case 0: gx_stage<0>(cur, g, wp + B); break;
                case 1: gx_stage<1>(cur, g, wp + B); break;
                case 2: gx_stage<2>(cur, g, wp + B); break;
                default: gx_stage<3>(cur, g, wp + B); break;
            }
            if (jp == steps - 1) cur.load(W, rg0, min(ch + 1, nchunk - 1), lane);
            lds_barrier();
            if (!live) continue;
            if (k0 + 64 <= K)
                compute(std::integral_constant<int, 64>(), rp + B, k0);
            else
                compute(std::integral_constant<int, 32>(), rp + B, k0);
        }
    }
    if (live) outer_store<TT, MT>(acc, i0, m, nt * 64, gx_rows(W), C, ldc, aux, epi);
}

// ---------------------------------------------------------------- dense weights

// f16, one or two tokens per wave: 64 columns of a panel, weights straight from the panel (16-byte
// pieces [ceil(K / PER)][64][PER], consecutive lanes on consecutive pieces), PF pieces per
// register buffer and two buffers.  The four waves of a workgroup take the same panel.
template <int T>
__global__ __launch_bounds__(256) void gemm_f16_exact_kernel(const uint16_t* __restrict__ B, int K, int N, int m, int mt,
                                                             int total, const float* __restrict__ A,
                                                             float* __restrict__ C, int ldc,
                                                             const float* __restrict__ aux, int epi) {
    constexpr int PER = 8;
    constexpr int PF = 8;  // pieces per register buffer
    constexpr int XK = 8;  // k per batch of scalar loads
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
        const uint32_t w = e < 2 ? v.x : e < 4 ? v.y : e < 6 ? v.z : v.w;
        return half_to_float((uint16_t)((e & 1) ? w >> 16 : w & 0xffffu));
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

// f32 and f16 on the matrix unit: with the sum as addend the instruction is the fused
// multiply-add of every (token, column) of one k, and the chain is the instruction's own.  The
// four waves of a workgroup take the same panel.  64 k at a time, the next 64 loading; the
// last K % 16 one by one.
template <typename E, int TT, int MT>
__global__ __launch_bounds__(256, 2) void gemm_dense_mm_kernel(const E* __restrict__ B, int K, int N, int m, int mt,
                                                               int total, const float* __restrict__ A,
                                                               float* __restrict__ C, int ldc,
                                                               const float* __restrict__ aux, int epi) {
    typedef Outer<TT> O;
    typedef typename O::vec vec;
    constexpr int T = TT * MT, KA = 4 * 64 / TT, NL = 64 / KA;
    constexpr int PER = 16 / (int)sizeof(E), PF = 64 / PER;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int tile = xcd_tile(blockIdx.x, total);
    const int nt = tile / mt, i0 = (tile - nt * mt) * 4 * T + wave * T;
    if (i0 >= m) return;
    const int nkb = (K + PER - 1) / PER;
    const uint4* P = reinterpret_cast<const uint4*>(B) + (size_t)nt * nkb * 64 + lane;
    const float* ar[MT];
#pragma unroll
    for (int t = 0; t < MT; t++) ar[t] = A + (size_t)min(i0 + TT * t + (lane & (TT - 1)), m - 1) * K;
    const int ak = 4 * (lane / TT);
    vec acc[MT];
#pragma unroll
    for (int t = 0; t < MT; t++) acc[t] = vec(0.0f);
    auto elem = [](const uint4& v, int e) -> float {
        if constexpr (PER == 4) {
            return __builtin_bit_cast(float, e == 0 ? v.x : e == 1 ? v.y : e == 2 ? v.z : v.w);
        } else {
            const uint32_t w = e < 2 ? v.x : e < 4 ? v.y : e < 6 ? v.z : v.w;
            return half_to_float((uint16_t)((e & 1) ? w >> 16 : w & 0xffffu));
        }
    };
    const int kf = K & ~15;
    const bool vec4 = (K & 3) == 0;
    // (loads past the last whole 16 k repeat values in range; they are not used)
    auto load = [&](int k0, uint4(&v)[PF], float4(&a)[MT][NL]) {
#pragma unroll
        for (int i = 0; i < PF; i++) v[i] = P[(size_t)min(k0 / PER + i, nkb - 1) * 64];
#pragma unroll
        for (int i = 0; i < NL; i++)
#pragma unroll
            for (int t = 0; t < MT; t++) {
                const float* x = ar[t] + min(k0 + KA * i + ak, kf - 4);
                a[t][i] = vec4 ? *reinterpret_cast<const float4*>(x) : make_float4(x[0], x[1], x[2], x[3]);
            }
    };
    auto block = [&](int k0, const uint4(&v)[PF], const float4(&a)[MT][NL]) {
        static_for<0, 4>([&](auto sc) {
            constexpr int K0 = 16 * decltype(sc)::value;
            if (k0 + K0 < kf)  // (uniform)
                static_for<0, 16>([&](auto ic) {
                    constexpr int k = K0 + decltype(ic)::value;
                    const float w = elem(v[k / PER], k % PER);
#pragma unroll
                    for (int t = 0; t < MT; t++)
                        acc[t] = O::template mm<(k % KA) / 4>(f4_get(a[t][k / KA], k % 4), w, acc[t]);
                });
        });
    };
    uint4 va[PF], vb[PF];
    float4 aa[MT][NL], ab[MT][NL];
    if (kf) load(0, va, aa);
    for (int k0 = 0; k0 < kf; k0 += 128) {
        load(k0 + 64, vb, ab);
        block(k0, va, aa);
        load(k0 + 128, va, aa);
        block(k0 + 64, vb, ab);
    }
    for (int k = kf; k < K; k++) {
        const E* we = reinterpret_cast<const E*>(P + (size_t)(k / PER) * 64) + k % PER;
        float w;
        if constexpr (PER == 4)
            w = *we;
        else
            w = half_to_float(*we);
#pragma unroll
        for (int t = 0; t < MT; t++) acc[t] = O::template mm<0>(ar[t][k], w, acc[t]);
    }
    outer_store<TT, MT>(acc, i0, m, nt * 64, N, C, ldc, aux, epi);
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

// A form's time per k in ns when the busiest CU has c workgroups of its grid: `one` at least,
// else slope c + off.  Measured with 4096 x 4096, 4096 x 14336, 6144 x 4096 and 28672 x 4096
// weights at 61, 130 and 200 rows (quantized: Q8_0), and with K x N of 512 x 1376, 2048 x 5632,
// 5632 x 2048, 896 x 4864 and others at 8 to 200 rows (dense); the fit is within 15 %.  The k-quants
// take Q8_0's table: their own times, with more unpacking and the spills above, were not fitted.
struct GemmForm {
    int T;
    float one, slope, off;
};
// (T <= 2 on the vector unit, above on the matrix unit)
static constexpr GemmForm GX_FORMS[] = {{1, 13.0f, 6.5f, 4.0f}, {2, 15.0f, 9.2f, 5.0f}, {4, 25.0f, 12.0f, 7.0f},
                                        {8, 39.0f, 20.0f, 12.0f}, {16, 55.0f, 33.0f, 11.0f}};
static constexpr GemmForm F32_FORMS[] = {{4, 9.9f, 9.5f, 0.0f}, {8, 11.3f, 13.0f, 0.0f}, {16, 17.7f, 27.0f, 0.0f}};
static constexpr GemmForm F16_FORMS[] = {{1, 8.5f, 4.5f, 3.0f}, {2, 10.0f, 5.0f, 4.0f}, {4, 14.0f, 7.0f, 5.0f},
                                         {8, 17.0f, 9.5f, 7.0f}, {16, 23.5f, 17.0f, 7.0f}};

template <int N>
static int gemm_form(const GemmForm (&forms)[N], int m, int ntiles) {
    int best = 0;
    float cost = 0.0f;
    for (const GemmForm& f : forms) {
        const long wgs = (long)ntiles * ((m + 4 * f.T - 1) / (4 * f.T));
        const float c = std::max(f.one, f.slope * (float)((wgs + g_gx_cus - 1) / g_gx_cus) + f.off);
        if (!best || c < cost) {
            best = f.T;
            cost = c;
        }
    }
    return best;
}

template <class Pieces, class Dev>
static void gemm_exact(const Dev& W, int m, const float* A, float* C, int ldc, const float* aux, Epi epi,
                       hipStream_t st) {
    const int ntiles = (W.rows + 63) / 64, T = gemm_form(GX_FORMS, m, ntiles);
    const int mt = (m + 4 * T - 1) / (4 * T), total = ntiles * mt;
#define JY_GX(KERNEL) \
    hipLaunchKernelGGL(KERNEL, dim3((unsigned)total), dim3(256), 0, st, W, m, mt, total, A, C, ldc, aux, (int)plain_epi(epi))
    switch (T) {
        case 16: JY_GX((gemm_exact_mm_kernel<Pieces, Dev, 16, 1>)); break;
        case 8: JY_GX((gemm_exact_mm_kernel<Pieces, Dev, 4, 2>)); break;
        case 4: JY_GX((gemm_exact_mm_kernel<Pieces, Dev, 4, 1>)); break;
        case 2: JY_GX((gemm_exact_kernel<Pieces, Dev, 2>)); break;
        default: JY_GX((gemm_exact_kernel<Pieces, Dev, 1>)); break;
    }
#undef JY_GX
}

template <typename E>
static void gemm_dense(const E* B, int K, int N, int m, const float* A, float* C, int ldc, const float* aux, Epi epi,
                       hipStream_t st) {
    const int ntiles = (N + 63) / 64;
    const int T = sizeof(E) == 4 ? gemm_form(F32_FORMS, m, ntiles) : gemm_form(F16_FORMS, m, ntiles);
    const int mt = (m + 4 * T - 1) / (4 * T), total = ntiles * mt;
#define JY_GD(KERNEL) \
    hipLaunchKernelGGL(KERNEL, dim3((unsigned)total), dim3(256), 0, st, B, K, N, m, mt, total, A, C, ldc, aux, (int)plain_epi(epi))
    if constexpr (sizeof(E) == 2) {
        if (T == 1) {
            JY_GD((gemm_f16_exact_kernel<1>));
            return;
        }
        if (T == 2) {
            JY_GD((gemm_f16_exact_kernel<2>));
            return;
        }
    }
    switch (T) {
        case 16: JY_GD((gemm_dense_mm_kernel<E, 16, 1>)); break;
        case 8: JY_GD((gemm_dense_mm_kernel<E, 4, 2>)); break;
        default: JY_GD((gemm_dense_mm_kernel<E, 4, 1>)); break;
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
