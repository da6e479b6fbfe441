// jy_quant.hip — weights of every type jieyu binds besides the Q8_0 fast path:
// k-quant (Q4_K / Q5_K / Q6_K) matrices in HBM, their decode matvec, and the
// per-type dispatch of matvec / GEMM that models of mixed weight types run.
//
// Decode matvec of a k-quant row = dot_row_avx2 (libs/matmul_libs/matmul_q.h:111-132):
// 32 virtual FMA lanes, lane L accumulates x[k] * w[k] for k = L mod 32 ascending,
// each 256-weight block dequantized as dequant_block does (:47-100), then the fixed
// tree s[i] = (a[i]+a[8+i]) + (a[16+i]+a[24+i]), r[i] = s[i]+s[4+i],
// y = (r0+r1)+(r2+r3).  The thread layout is the Q8_0 kernel's: 16 threads per row
// (two lanes each), 4 rows per wave, the activation vector lane-pair major in LDS.
#include <algorithm>

#include "jy_matvec.h"

namespace jy {

// ---------------------------------------------------------------- layout

KQDev kq_shape(int type, int rows, int cols) {
    KQDev w;
    w.type = type;
    w.rows = rows;
    w.cols = cols;
    w.nsb = cols / 256;
    w.groups = (rows + 3) / 4;
    return w;
}

size_t kq_bytes(const KQDev& w, int part) {
    const size_t chunks = (size_t)w.groups * w.nsb;
    switch (part) {
        case 0: return chunks * 512;
        case 1: return w.type == JY_Q5_K ? chunks * 128 : w.type == JY_Q6_K ? chunks * 256 : 0;
        case 2: return chunks * 64;
        default: return chunks * 16;
    }
}

__host__ __device__ static inline int kq_block_bytes(int type) { return type == JY_Q4_K ? 144 : type == JY_Q5_K ? 176 : 210; }

// get_scale_min_k4 (libs/matmul_libs/matmul_q.h:22-33): the 6-bit scale and min of
// 32-weight step j of a Q4_K / Q5_K super-block
__device__ __forceinline__ void kq_scale_min(int j, const uint8_t* q, int& sc, int& mn) {
    if (j < 4) {
        sc = q[j] & 63;
        mn = q[j + 4] & 63;
    } else {
        sc = (q[j + 4] & 0xF) | ((q[j - 4] >> 6) << 4);
        mn = (q[j + 4] >> 4) | ((q[j] >> 6) << 4);
    }
}

// one thread per (row, super-block): GGML block -> the thread-major pieces.  Weight
// 32c + L (L = 2g + u) of the block goes to thread (row & 3) * 16 + g as weight (c, u).
__global__ void repack_kq_kernel(const uint8_t* __restrict__ src, KQDev W) {
    const size_t id = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (id >= (size_t)W.rows * W.nsb) return;
    const int R = (int)(id / W.nsb), sb = (int)(id % W.nsb), ri = R & 3;
    const uint8_t* b = src + id * kq_block_bytes(W.type);
    const size_t chunk = (size_t)(R >> 2) * W.nsb + sb;
    for (int g = 0; g < 16; g++) {
        uint64_t nib = 0;
        uint32_t hb = 0;
        for (int c = 0; c < 8; c++)
            for (int u = 0; u < 2; u++) {
                const int L = 2 * g + u, T = 2 * (c >> 2) + u, kb = c & 3;
                uint32_t lo;
                if (W.type == JY_Q6_K) {  // matmul_q.h:78-96
                    const int nn = c >> 2, tq = c & 3;
                    const uint8_t qb = b[nn * 64 + L + 32 * (tq & 1)];
                    lo = tq < 2 ? (qb & 15u) : (qb >> 4);
                    hb |= ((b[128 + nn * 32 + L] >> (2 * tq)) & 3u) << (8 * kb + 2 * T);
                } else {  // q4.h:23-33, matmul_q.h:52-76
                    const uint8_t* qs = b + (W.type == JY_Q4_K ? 16 : 48);
                    const uint8_t qb = qs[(c >> 1) * 32 + L];
                    lo = (c & 1) ? (qb >> 4) : (qb & 15u);
                    if (W.type == JY_Q5_K) hb |= ((b[16 + L] >> c) & 1u) << (4 * T + kb);
                }
                nib |= (uint64_t)lo << (4 * (2 * c + u));
            }
        const size_t t = chunk * 64 + ri * 16 + g;
        *reinterpret_cast<uint64_t*>(W.nib + t * 8) = nib;
        if (W.type == JY_Q5_K) *reinterpret_cast<uint16_t*>(W.hi + t * 2) = (uint16_t)hb;
        if (W.type == JY_Q6_K) *reinterpret_cast<uint32_t*>(W.hi + t * 4) = hb;
    }
    uint8_t* h = W.hdr + chunk * 64 + ri * 16;
    if (W.type == JY_Q6_K) {
        // scale of step c for weights L < 16 (bytes 0..7) and L >= 16 (bytes 8..15):
        // sc[(c >> 2) * 8 + L / 16 + 2 * (c & 3)] of the block (matmul_q.h:83-90)
        for (int half = 0; half < 2; half++)
            for (int c = 0; c < 8; c++) h[half * 8 + c] = b[192 + (c >> 2) * 8 + half + 2 * (c & 3)];
        W.dm[chunk * 4 + ri] = (uint32_t)(b[208] | (b[209] << 8));
    } else {
        for (int c = 0; c < 8; c++) {
            int sc, mn;
            kq_scale_min(c, b + 4, sc, mn);
            h[c] = (uint8_t)sc;
            h[8 + c] = (uint8_t)mn;
        }
        W.dm[chunk * 4 + ri] = (uint32_t)(b[0] | (b[1] << 8) | (b[2] << 16) | ((uint32_t)b[3] << 24));
    }
}

void launch_repack_kq(const uint8_t* src, const KQDev& dst, hipStream_t st) {
    const size_t n = (size_t)dst.rows * dst.nsb;
    hipLaunchKernelGGL(repack_kq_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, src, dst);
}

// ---------------------------------------------------------------- decode matvec

// byte j (a compile-time constant after unrolling) of a word, as a float: v_cvt_f32_ubyte
__device__ __forceinline__ float ubyte_f(uint32_t w, int j) { return (float)((w >> (8 * j)) & 255u); }

// the 16 weights of this thread in one chunk, fed to its two FMA lanes in order.
// Target word T (= 2*(c >> 2) + u) holds weight (c, u) in byte c & 3 after the mask,
// with the Q5_K / Q6_K high bits merged in above the nibble.
template <int TYPE>
__device__ __forceinline__ void kq_chunk(const uint2& nb, uint32_t hb, const uint4& h, uint32_t dmw, int g,
                                         const float* xv, float& a0, float& a1) {
    uint32_t wt[4] = {nb.x & 0x0F0F0F0Fu, (nb.x >> 4) & 0x0F0F0F0Fu, nb.y & 0x0F0F0F0Fu, (nb.y >> 4) & 0x0F0F0F0Fu};
    const float d = half_to_float((uint16_t)(dmw & 0xffffu));
    if (TYPE == JY_Q6_K) {
        // bits 8k + 2T of hb -> bits 4, 5 of byte k of word T
#pragma unroll
        for (int T = 0; T < 4; T++) wt[T] |= (T < 2 ? hb << (4 - 2 * T) : hb >> (2 * T - 4)) & 0x30303030u;
        const uint32_t s0 = g < 8 ? h.x : h.z, s1 = g < 8 ? h.y : h.w;  // the scales of this lane's half
#pragma unroll
        for (int c = 0; c < 8; c++) {
            const int8_t sc = (int8_t)((c < 4 ? s0 : s1) >> (8 * (c & 3)));
            const float ds = d * (float)sc;
#pragma unroll
            for (int u = 0; u < 2; u++) {
                // (d*sc) * (q - 32), the reference's expression; q - 32 is exact
                const float w = ds * (ubyte_f(wt[2 * (c >> 2) + u], c & 3) - 32.0f);
                if (u == 0)
                    a0 = __builtin_fmaf(xv[2 * c], w, a0);
                else
                    a1 = __builtin_fmaf(xv[2 * c + 1], w, a1);
            }
        }
    } else {
        if (TYPE == JY_Q5_K) {
            // bit 4T + k of hb -> bit 4 of byte k of word T: spread the nibble by a multiply
#pragma unroll
            for (int T = 0; T < 4; T++) wt[T] |= ((((hb >> (4 * T)) & 15u) * 0x00204081u) << 4) & 0x10101010u;
        }
        const float dmin = half_to_float((uint16_t)(dmw >> 16));
#pragma unroll
        for (int c = 0; c < 8; c++) {
            const float d1 = d * ubyte_f(c < 4 ? h.x : h.y, c & 3), n1 = dmin * ubyte_f(c < 4 ? h.z : h.w, c & 3);
#pragma unroll
            for (int u = 0; u < 2; u++) {
                const float w = __builtin_fmaf(ubyte_f(wt[2 * (c >> 2) + u], c & 3), d1, -n1);
                if (u == 0)
                    a0 = __builtin_fmaf(xv[2 * c], w, a0);
                else
                    a1 = __builtin_fmaf(xv[2 * c + 1], w, a1);
            }
        }
    }
}

// The chunk stream of one wave's row groups in registers: U chunks of one matrix.
template <int TYPE, int U>
struct KqBuf {
    uint2 nb[U];
    uint32_t hb[U];
    uint4 h[U];
    uint32_t dm[U];

    // chunks s0 .. s0 + U - 1 of row group rg (indices past the row clamp to its last
    // chunk: read, never used)
    __device__ __forceinline__ void load(const KQDev& W, int rg, int s0, int lane, int r) {
#pragma unroll
        for (int u = 0; u < U; u++) {
            const size_t c = (size_t)rg * W.nsb + min(s0 + u, W.nsb - 1);
            nb[u] = *reinterpret_cast<const uint2*>(W.nib + c * 512 + lane * 8);
            hb[u] = TYPE == JY_Q5_K   ? *reinterpret_cast<const uint16_t*>(W.hi + c * 128 + lane * 2)
                    : TYPE == JY_Q6_K ? *reinterpret_cast<const uint32_t*>(W.hi + c * 256 + lane * 4)
                                      : 0u;
            h[u] = *reinterpret_cast<const uint4*>(W.hdr + c * 64 + r * 16);
            dm[u] = W.dm[c * 4 + r];
        }
    }
};

__device__ __forceinline__ void kq_x(const float* xrow, int s, float* xv) {
    const float4* xp = reinterpret_cast<const float4*>(xrow + 16 * s);
#pragma unroll
    for (int q = 0; q < 4; q++) {
        const float4 v = xp[q];
        xv[4 * q] = v.x;
        xv[4 * q + 1] = v.y;
        xv[4 * q + 2] = v.z;
        xv[4 * q + 3] = v.w;
    }
}

// lanes 2g, 2g+1 -> the reference's reduction tree (as in the Q8_0 matvec)
__device__ __forceinline__ float kq_tree(float a0, float a1) {
    a0 += dpp_f<0x12C>(a0);
    a1 += dpp_f<0x12C>(a1);
    a0 += dpp_f<0x128>(a0);
    a1 += dpp_f<0x128>(a1);
    a0 += dpp_f<0x4E>(a0);
    a1 += dpp_f<0x4E>(a1);
    const float t = a0 + a1;
    return t + dpp_f<0xB1>(t);
}

// x (K floats) into LDS in lane-pair order, `pre()` (the first weight loads) issued once x's
// first loads are out.  With NORM the RMSNorm comes first: x and the norm weights stay in
// registers (NV float4s per thread: K <= 1024 NV; NV = 0: no norm, SB
// float4s per thread at a time), x goes to LDS in its own order for the sum of squares, then
// (x * scale) * w in lane-pair order over it.  Only LDS is ordered by the barriers, so the
// weight loads stay in flight.
static constexpr int KQ_NORM_MAX = 8192;
template <int NV, int SB, class Pre>
__device__ __forceinline__ void kq_stage(const float* __restrict__ x, const float* __restrict__ nw, int K, int XS,
                                         float* xs, float* red, Pre&& pre) {
    const int tid = threadIdx.x, n4 = K / 4;
    const float4* x4 = reinterpret_cast<const float4*>(x);
    auto put = [&](int i, float4 v) {
        xs[xs_index(4 * i, XS)] = v.x;
        xs[xs_index(4 * i + 1, XS)] = v.y;
        xs[xs_index(4 * i + 2, XS)] = v.z;
        xs[xs_index(4 * i + 3, XS)] = v.w;
    };
    if constexpr (NV > 0) {
        const float4* w4 = reinterpret_cast<const float4*>(nw);
        float4 v[NV], wv[NV];
#pragma unroll
        for (int j = 0; j < NV; j++) {
            const int i = tid + 256 * j;
            v[j] = i < n4 ? x4[i] : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
            wv[j] = i < n4 ? w4[i] : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        }
        pre();
#pragma unroll
        for (int j = 0; j < NV; j++) {
            const int i = tid + 256 * j;
            if (i < n4) reinterpret_cast<float4*>(xs)[i] = v[j];
        }
        lds_barrier();
        block_rms_scale(xs, K, red);
        const float scale = red[16];
        const bool zero = red[17] != 0.0f;
#pragma unroll
        for (int j = 0; j < NV; j++) {
            const int i = tid + 256 * j;
            if (i < n4)
                put(i, zero ? make_float4(0.0f, 0.0f, 0.0f, 0.0f)
                            : make_float4((v[j].x * scale) * wv[j].x, (v[j].y * scale) * wv[j].y,
                                          (v[j].z * scale) * wv[j].z, (v[j].w * scale) * wv[j].w));
        }
    } else {
        for (int b0 = 0; b0 < n4; b0 += SB * 256) {
            float4 v[SB];
#pragma unroll
            for (int j = 0; j < SB; j++) {
                const int i = b0 + tid + 256 * j;
                v[j] = i < n4 ? x4[i] : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
            }
            if (b0 == 0) pre();
#pragma unroll
            for (int j = 0; j < SB; j++) {
                const int i = b0 + tid + 256 * j;
                if (i < n4) put(i, v[j]);
            }
        }
    }
    lds_barrier();
}

// Up to three k-quant matrices of the same input in one launch (q, k and v), each with
// workgroups of its own; rows are numbered through them (row0).
struct KqMats {
    KQDev W[3];
    int wg0[4];   // first workgroup of each matrix, then the total
    int row0[3];  // first output row of each matrix
};

// One matrix by `nwg` workgroups of 4 waves.  With the norm (NV > 0) wave w takes row groups w, w +
// 4 nwg, ..., the loads running ahead across them; without, one row group, and with NV = KQ_SHORT
// a row of at most U chunks, one buffer.
static constexpr int KQ_SHORT = -1;
template <int TYPE, int EPI, int NV, int U>
__device__ __forceinline__ void kq_body(const KQDev& W, int wg, int nwg, int row0, const float* __restrict__ x,
                                        const float* __restrict__ nw, float* __restrict__ out, const MvArgs& a,
                                        float* xs, float* red) {
    const int lane = threadIdx.x & 63, r = lane >> 4, g = lane & 15;
    const int wid = wg * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), TW = nwg * 4;
    const int nsb = W.nsb, XS = 16 * nsb + 4;
    // two buffers of U chunks, two ahead of the compute, across row groups
    KqBuf<TYPE, U> A, B;
    int lrg = min(wid, W.groups - 1), lp = 0;  // row group and chunk of the next load
    auto load = [&](KqBuf<TYPE, U>& b) {
        b.load(W, lrg, lp, lane, r);
        lp += U;
        if (lp >= nsb) {
            lp = 0;
            lrg = min(lrg + TW, W.groups - 1);
        }
    };
    kq_stage<NV, U>(x, nw, W.cols, XS, xs, red, [&]() {
        load(A);
    });
    if (NV > 0) load(B);
    const float* xrow = xs + g * XS;
    float bv = 0.0f;
    int bi = 0;
    float a0 = 0.0f, a1 = 0.0f;
    auto compute = [&](const KqBuf<TYPE, U>& b, int s0) {
#pragma unroll
        for (int u = 0; u < U; u++) {
            if (s0 + u < nsb) {
                float xv[16];
                kq_x(xrow, s0 + u, xv);
                kq_chunk<TYPE>(b.nb[u], b.hb[u], b.h[u], b.dm[u], g, xv, a0, a1);
            }
        }
    };
    const int nb = (nsb + U - 1) / U;  // buffers per row group
    if constexpr (NV <= 0) {
        if (wid >= W.groups) return;
        const int lr = wid * 4 + r, row = row0 + lr;
        const bool own = g == 0 && lr < W.rows;
        const MvPre pre = mv_preload<EPI>(row, own, r, a, out);
        if constexpr (NV == KQ_SHORT) {
            compute(A, 0);
        } else {
            for (int s0 = 0; s0 < nsb; s0 += 2 * U) {
                B.load(W, wid, s0 + U, lane, r);
                compute(A, s0);
                if (s0 + 2 * U < nsb) A.load(W, wid, s0 + 2 * U, lane, r);
                compute(B, s0 + U);
            }
        }
        mv_epilogue<EPI>(kq_tree(a0, a1), row, own, r, row0 + W.rows, a, out, bv, bi, &pre);
        return;
    }
    bool cur_b = false;                // whether the next buffer to compute is B
    for (int rg = wid; rg < W.groups; rg += TW) {
        const int lr = rg * 4 + r, row = row0 + lr;
        const bool own = g == 0 && lr < W.rows;
        const MvPre pre = mv_preload<EPI>(row, own, r, a, out);
        a0 = a1 = 0.0f;
        int i = 0;
        if (cur_b) {  // (an odd number of buffers per row group: they swap)
            compute(B, 0);
            load(B);
            i = 1;
        }
        for (; i + 1 < nb; i += 2) {
            compute(A, i * U);
            load(A);
            compute(B, (i + 1) * U);
            load(B);
        }
        if (i < nb) {
            compute(A, i * U);
            load(A);
        }
        cur_b = cur_b != ((nb & 1) != 0);
        mv_epilogue<EPI>(kq_tree(a0, a1), row, own, r, row0 + W.rows, a, out, bv, bi, &pre);
    }
}

// The decode matvec.  What bounds it: at few row groups (1024: one wave per SIMD) the latency of
// the weight stream; past that the dequantisation (about 90 VALU instructions per 256 weights of
// 4 rows).  The vector is staged with its loads ahead of the first weights' (dependent 4-byte loads
// before them: 4096 x 14336 30.5 us).  Without the norm a wave takes one row group: running the loads
// ahead across row groups there cost 0.3 to 0.9 us a launch in buffers read and never used (1024 x 4096
// 7.6 against 6.7).
template <int EPI, int NV, int U>
__global__ __launch_bounds__(256, U == 4 && NV <= 4 ? 4 : 2) void matvec_kq_kernel(KqMats M, const float* __restrict__ x,
                                                        const float* __restrict__ nw, float* __restrict__ out,
                                                        MvArgs a) {
    extern __shared__ __align__(16) float xs[];  // [16][XS]: lane pair g, 16 floats per chunk
    __shared__ float red[18];
    const int b = blockIdx.x;
    const int i = b >= M.wg0[2] ? 2 : b >= M.wg0[1] ? 1 : 0;
    const int wg = b - M.wg0[i], nwg = M.wg0[i + 1] - M.wg0[i];
    switch (M.W[i].type) {  // (uniform over the workgroup)
        case JY_Q4_K: kq_body<JY_Q4_K, EPI, NV, U>(M.W[i], wg, nwg, M.row0[i], x, nw, out, a, xs, red); break;
        case JY_Q5_K: kq_body<JY_Q5_K, EPI, NV, U>(M.W[i], wg, nwg, M.row0[i], x, nw, out, a, xs, red); break;
        default: kq_body<JY_Q6_K, EPI, NV, U>(M.W[i], wg, nwg, M.row0[i], x, nw, out, a, xs, red); break;
    }
}

// gate and up of one type together: RMSNorm, both dots over the same staged vector (each
// chunk's x read from LDS once for the two), out[j] = silu(gate_j) * up_j
template <int TYPE, int NV>
__global__ __launch_bounds__(256, NV <= 4 ? 4 : 2) void matvec_kq_pair_kernel(KQDev W0, KQDev W1, const float* __restrict__ x,
                                                             const float* __restrict__ nw, float* __restrict__ out) {
    extern __shared__ __align__(16) float xs[];
    __shared__ float red[18];
    constexpr int U = 2;
    const int lane = threadIdx.x & 63, r = lane >> 4, g = lane & 15;
    const int wid = blockIdx.x * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), TW = gridDim.x * 4;
    const int nsb = W0.nsb, XS = 16 * nsb + 4, groups = W0.groups;
    KqBuf<TYPE, U> A0, A1, B0, B1;
    int lrg = min(wid, groups - 1), lp = 0;
    auto load = [&](KqBuf<TYPE, U>& p, KqBuf<TYPE, U>& q) {
        p.load(W0, lrg, lp, lane, r);
        q.load(W1, lrg, lp, lane, r);
        lp += U;
        if (lp >= nsb) {
            lp = 0;
            lrg = min(lrg + TW, groups - 1);
        }
    };
    kq_stage<NV, 4>(x, nw, W0.cols, XS, xs, red, [&]() { load(A0, A1); });
    load(B0, B1);
    const float* xrow = xs + g * XS;
    float a0, a1, c0, c1;
    auto compute = [&](const KqBuf<TYPE, U>& p, const KqBuf<TYPE, U>& q, int s0) {
#pragma unroll
        for (int u = 0; u < U; u++) {
            if (s0 + u < nsb) {
                float xv[16];
                kq_x(xrow, s0 + u, xv);
                kq_chunk<TYPE>(p.nb[u], p.hb[u], p.h[u], p.dm[u], g, xv, a0, a1);
                kq_chunk<TYPE>(q.nb[u], q.hb[u], q.h[u], q.dm[u], g, xv, c0, c1);
            }
        }
    };
    const int nb = (nsb + U - 1) / U;
    bool cur_b = false;
    for (int rg = wid; rg < groups; rg += TW) {
        a0 = a1 = c0 = c1 = 0.0f;
        int i = 0;
        if (cur_b) {
            compute(B0, B1, 0);
            load(B0, B1);
            i = 1;
        }
        for (; i + 1 < nb; i += 2) {
            compute(A0, A1, i * U);
            load(A0, A1);
            compute(B0, B1, (i + 1) * U);
            load(B0, B1);
        }
        if (i < nb) {
            compute(A0, A1, i * U);
            load(A0, A1);
        }
        cur_b = cur_b != ((nb & 1) != 0);
        const float yg = kq_tree(a0, a1), yu = kq_tree(c0, c1);
        const int row = rg * 4 + r;
        if (g == 0 && row < W0.rows) out[row] = silu_at(yg, row, W0.rows) * yu;
    }
}

size_t mv_kq_lds_bytes(int cols) { return (size_t)16 * (16 * (cols / 256) + 4) * sizeof(float); }

static int g_kq_cus = 256;

// workgroups of a matrix's launch: one row group per wave up to 4 workgroups per CU, past
// that every workgroup the same number of row groups per wave (the vector is staged and
// normalised once per workgroup)
static int kq_wgs(const KQDev& W) {
    const int max_waves = 16 * g_kq_cus, per = (W.groups + max_waves - 1) / max_waves;
    return (W.groups + 4 * per - 1) / (4 * per);
}

static KqMats kq_mats(const KQDev* const* W, int n) {
    KqMats M;
    int wg = 0, row = 0;
    for (int i = 0; i < 3; i++) {
        M.W[i] = *W[i < n ? i : 0];
        M.wg0[i] = wg;
        M.row0[i] = row;
        if (i < n) {
            wg += kq_wgs(M.W[i]);
            row += M.W[i].rows;
        }
    }
    M.wg0[3] = wg;
    // (matrices past n have no workgroups: their wg0 is the total)
    return M;
}

// Rows of up to 4 chunks (1024 inputs) take one buffer: 64 x 256 2.5 us against 2.9 in the loop.  Eight
// chunks a buffer pay for long rows alone, with at most a workgroup per CU: Q4_K 4096 x 14336 19.5 ->
// 18.7 us, but 2048 x 5632 8.6 -> 9.1, 1024 x 3072 5.7 -> 5.9, 2048 x 2048 4.4 -> 5.5.
template <int EPI, int NV>
static void mv_kq(const KqMats& M, const float* x, const float* nw, float* out, const MvArgs& a, hipStream_t st) {
    const dim3 grid((unsigned)M.wg0[3]), block(256);
    const size_t lds = mv_kq_lds_bytes(M.W[0].cols);
    if constexpr (NV == 0) {
        if (M.W[0].nsb <= 4) {
            hipLaunchKernelGGL((matvec_kq_kernel<EPI, KQ_SHORT, 4>), grid, block, lds, st, M, x, nw, out, a);
            return;
        }
        if (M.wg0[3] <= g_kq_cus && M.W[0].nsb > 32) {
            hipLaunchKernelGGL((matvec_kq_kernel<EPI, 0, 8>), grid, block, lds, st, M, x, nw, out, a);
            return;
        }
    }
    hipLaunchKernelGGL((matvec_kq_kernel<EPI, NV, 4>), grid, block, lds, st, M, x, nw, out, a);
}

static bool is_kq(const DevW& w) { return w.type == JY_Q4_K || w.type == JY_Q5_K || w.type == JY_Q6_K; }

static void mv_kq1(const DevW& W, const float* x, const float* nw, float* out, Epi epi, const float* aux,
                   hipStream_t st) {
    const KQDev* w[1] = {&W.kq};
    KqMats M = kq_mats(w, 1);
    if (!nw) M.wg0[1] = M.wg0[2] = M.wg0[3] = (W.kq.groups + 3) / 4;
    MvArgs a;
    a.aux = aux;
    if (nw) {
        if (W.in <= KQ_NORM_MAX / 2)
            mv_kq<EPI_STORE, 4>(M, x, nw, out, a, st);
        else
            mv_kq<EPI_STORE, 8>(M, x, nw, out, a, st);
        return;
    }
    if (epi == EPI_STORE) mv_kq<EPI_STORE, 0>(M, x, nullptr, out, a, st);
    if (epi == EPI_BIAS) mv_kq<EPI_BIAS, 0>(M, x, nullptr, out, a, st);
    if (epi == EPI_RESID) mv_kq<EPI_RESID, 0>(M, x, nullptr, out, a, st);
}

bool launch_mv_norm(const DevW& W, const float* x, const float* nw, float* out, hipStream_t st) {
    if (!is_kq(W) || W.in > KQ_NORM_MAX) return false;
    mv_kq1(W, x, nw, out, EPI_STORE, nullptr, st);
    return true;
}

bool launch_mv_qkv(const DevW* W, const float* x, const float* nw, float* qkv, const MvArgs& a, hipStream_t st) {
    if (!is_kq(W[0]) || !is_kq(W[1]) || !is_kq(W[2]) || W[0].in > KQ_NORM_MAX) return false;
    const KQDev* w[3] = {&W[0].kq, &W[1].kq, &W[2].kq};
    if (W[0].in <= KQ_NORM_MAX / 2)
        mv_kq<EPI_ROPE, 4>(kq_mats(w, 3), x, nw, qkv, a, st);
    else
        mv_kq<EPI_ROPE, 8>(kq_mats(w, 3), x, nw, qkv, a, st);
    return true;
}

template <int TYPE>
static void mv_kq_pair(const KQDev& gate, const KQDev& up, const float* x, const float* nw, float* h, hipStream_t st) {
    const dim3 grid((unsigned)kq_wgs(gate)), block(256);
    const size_t lds = mv_kq_lds_bytes(gate.cols);
    if (gate.cols <= KQ_NORM_MAX / 2)
        hipLaunchKernelGGL((matvec_kq_pair_kernel<TYPE, 4>), grid, block, lds, st, gate, up, x, nw, h);
    else
        hipLaunchKernelGGL((matvec_kq_pair_kernel<TYPE, 8>), grid, block, lds, st, gate, up, x, nw, h);
}

bool launch_mv_gate_up(const DevW& gate, const DevW& up, const float* x, const float* nw, float* h, hipStream_t st) {
    if (!is_kq(gate) || gate.type != up.type || gate.in > KQ_NORM_MAX) return false;
    switch (gate.type) {
        case JY_Q4_K: mv_kq_pair<JY_Q4_K>(gate.kq, up.kq, x, nw, h, st); break;
        case JY_Q5_K: mv_kq_pair<JY_Q5_K>(gate.kq, up.kq, x, nw, h, st); break;
        default: mv_kq_pair<JY_Q6_K>(gate.kq, up.kq, x, nw, h, st); break;
    }
    return true;
}

void launch_mv(const DevW& W, const float* x, float* out, Epi epi, const float* aux, hipStream_t st) {
    epi = plain_epi(epi);
    switch (W.type) {
        case JY_F32:
            launch_matvec_f32(static_cast<const float*>(W.dense), W.in, W.out, x, out, aux, epi, st);
            break;
        case JY_F16: launch_matvec_f16(static_cast<const uint16_t*>(W.dense), W.in, W.out, x, out, aux, epi, st); break;
        case JY_Q8_0: {
            MvArgs a;
            a.aux = aux;
            launch_matvec_q8(W.q8, x, nullptr, out, epi, a, st);
            break;
        }
        default: mv_kq1(W, x, nullptr, out, epi, aux, st); break;
    }
}

hipError_t quant_init() {
    int dev = 0, cus = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e == hipSuccess) e = hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev);
    if (e == hipSuccess && cus > 0) g_kq_cus = cus;
    for (const void* f : {reinterpret_cast<const void*>(&matvec_kq_kernel<EPI_STORE, 0, 4>),
                          reinterpret_cast<const void*>(&matvec_kq_kernel<EPI_STORE, 0, 8>),
                          reinterpret_cast<const void*>(&matvec_kq_kernel<EPI_STORE, KQ_SHORT, 4>),
                          reinterpret_cast<const void*>(&matvec_kq_kernel<EPI_STORE, 4, 4>),
                          reinterpret_cast<const void*>(&matvec_kq_kernel<EPI_STORE, 8, 4>),
                          reinterpret_cast<const void*>(&matvec_kq_kernel<EPI_BIAS, 0, 4>),
                          reinterpret_cast<const void*>(&matvec_kq_kernel<EPI_BIAS, 0, 8>),
                          reinterpret_cast<const void*>(&matvec_kq_kernel<EPI_BIAS, KQ_SHORT, 4>),
                          reinterpret_cast<const void*>(&matvec_kq_kernel<EPI_RESID, 0, 4>),
                          reinterpret_cast<const void*>(&matvec_kq_kernel<EPI_RESID, 0, 8>),
                          reinterpret_cast<const void*>(&matvec_kq_kernel<EPI_RESID, KQ_SHORT, 4>),
                          reinterpret_cast<const void*>(&matvec_kq_kernel<EPI_ROPE, 4, 4>),
                          reinterpret_cast<const void*>(&matvec_kq_kernel<EPI_ROPE, 8, 4>),
                          reinterpret_cast<const void*>(&matvec_kq_pair_kernel<JY_Q4_K, 4>),
                          reinterpret_cast<const void*>(&matvec_kq_pair_kernel<JY_Q4_K, 8>),
                          reinterpret_cast<const void*>(&matvec_kq_pair_kernel<JY_Q5_K, 4>),
                          reinterpret_cast<const void*>(&matvec_kq_pair_kernel<JY_Q5_K, 8>),
                          reinterpret_cast<const void*>(&matvec_kq_pair_kernel<JY_Q6_K, 4>),
                          reinterpret_cast<const void*>(&matvec_kq_pair_kernel<JY_Q6_K, 8>)})
        if (e == hipSuccess) e = hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024 - 2048);
    return e;
}

}  // namespace jy
