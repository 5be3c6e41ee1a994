// Direct-fragment products: out[M,N] = epilogue(X[M,K] @ W[N,K]^T) whose MFMA
// operands are loaded from global memory straight into registers in the
// operand layout, with no LDS staging (included by gemm.hip).
//
// One load instruction covers 16 rows x 64 bytes (lane l: row l%16, 16 bytes
// at 16*(l/16)): 32 k in bf16 = one v_mfma_f32_16x16x32_bf16 operand, 16 k in
// fp32 = four v_mfma_f32_16x16x4_f32 operands (step e takes element e of every
// lane's four, so the k order within the chunk is permuted the same way for
// both operands).  A wave owns a (16*MT) x (16*NT) tile; KW waves of a block
// split K in contiguous parts and are summed through LDS, so a product with
// few output tiles still fills the chip.
#pragma once

namespace loom {

// Two chunks make a unit, whole 128-byte lines of the rows, whose halves are
// requested back to back.  With SWAP the odd rows of a fragment ask for the
// second half of their line first: the L1 then serves both 64-byte halves at
// a time instead of sixteen times the same one (row strides here are whole
// lines; padding the rows by 64 bytes has the same effect), and the halves are
// exchanged in the registers (999 x 3072 x 768 in bf16 25.8 -> 20.7 us, 128 x
// 768 x 3072 11.3 -> 8.9 us).  fp32 tiles larger than 32 x 16 are bound by
// the matrix cores, where the exchange costs more than it saves (256 x 768 x
// 3072 31 -> 44 us), and take the plain order.
//
// U: units of operands in flight per wave.
template <typename T, int MT, int NT, int KW, int U>
struct FragCfg {
    static constexpr int TM = 16 * MT, TN = 16 * NT;      // wave tile
    static constexpr int THREADS = 64 * KW;
    static constexpr int CK = 64 / (int)sizeof(T);        // k per chunk
    static constexpr bool SWAP = sizeof(T) == 2 || MT * NT <= 2;
};
// k per unit: K (and K1 of a second input) must be a multiple
template <typename T> constexpr int kFragK = 128 / (int)sizeof(T);

template <typename T, int MT, int NT, int KW, int U, bool GATHER, bool DUAL>
__global__ void __launch_bounds__(64 * KW)
gemm_frag_kernel(GemmArgs a) {
    using C = FragCfg<T, MT, NT, KW, U>;
    constexpr int E = (int)sizeof(T);
    const int tid = threadIdx.x, lane = tid & 63;
    const int kw = __builtin_amdgcn_readfirstlane(tid >> 6);
    // the m-tiles of one n-tile are neighbours on one XCD (they share the W
    // rows in its L2; X is the smaller operand in the products this serves)
    const int MTL = (int)ceil_div(a.M, C::TM);
    const int b = xcd_contiguous((int)blockIdx.x, (int)gridDim.x);
    const int64_t n0 = (int64_t)(b / MTL) * C::TN, m0 = (int64_t)(b % MTL) * C::TM;
    const int64_t g = GATHER ? n0 / a.Hq : 0;
    const int64_t ldx = GATHER ? a.Nm : a.ldx;
    const int fr = lane & 15, fq = lane >> 4;
    const bool odd = C::SWAP && (fr & 1) != 0;

    // byte offsets of the lane's rows within the tile (rows past the end read
    // the last row; their results are not stored)
    uint32_t xv[MT], wv[NT], xv2[MT], wv2[NT];
#pragma unroll
    for (int j = 0; j < MT; ++j) {
        const int64_t r = m0 + 16 * j + fr < a.M ? 16 * j + fr : a.M - 1 - m0;
        xv[j] = (uint32_t)(r * ldx * E + 16 * fq);
        xv2[j] = DUAL ? (uint32_t)(r * a.ldx2 * E + 16 * fq) : 0u;
    }
#pragma unroll
    for (int i = 0; i < NT; ++i) {
        const int64_t r = n0 + 16 * i + fr < a.N ? 16 * i + fr : a.N - 1 - n0;
        wv[i] = (uint32_t)(r * a.ldw * E + 16 * fq);
        wv2[i] = DUAL ? (uint32_t)(r * a.ldw2 * E + 16 * fq) : 0u;
    }
    const auto rsrc = [](const void* p) {
        return __builtin_amdgcn_make_buffer_rsrc((void*)p, (short)0, 0x7fffffff, kBufferDword3);
    };
    const auto rw = rsrc((const T*)a.W + n0 * a.ldw);
    const auto rx = rsrc(GATHER ? nullptr : (const T*)a.X + m0 * a.ldx);
    const auto rw2 = rsrc(DUAL ? (const T*)a.W2 + n0 * a.ldw2 : nullptr);
    const auto rx2 = rsrc(DUAL ? (const T*)a.X2 + m0 * a.ldx2 : nullptr);

    struct Frags {
        u32x4 w[NT][2], x[MT][2];
    };
    const int nu = (int)(a.K / (2 * C::CK));
    const uint32_t first = odd ? 64u : 0u;                // byte offset of the half asked for first
    // request unit `unit` (past the end: the last one): register p holds half
    // p of the line, in odd rows of SWAP tiles half 1 - p
    auto load = [&](Frags& f, int unit) {
        const int64_t k = (int64_t)min(unit, nu - 1) * (2 * C::CK);
        const bool second = DUAL && k >= a.K1;            // uniform (K1 is a multiple of the unit)
        const uint32_t sk = (uint32_t)((second ? k - a.K1 : k) * E);
        const auto rwc = second ? rw2 : rw;
#pragma unroll
        for (int i = 0; i < NT; ++i)
#pragma unroll
            for (int p = 0; p < 2; ++p)
                f.w[i][p] = __builtin_amdgcn_raw_buffer_load_b128(
                    rwc, (int)((second ? wv2[i] : wv[i]) + (p == 0 ? first : 64u - first)), (int)sk, 0);
        if constexpr (GATHER) {                           // each half lies in one sector
            const void *s0, *s1;
            int64_t c0, c1;
            gather_half(a, k, g, s0, c0);
            gather_half(a, k + C::CK, g, s1, c1);
            const char* p0 = (const char*)((const T*)s0 + m0 * a.Nm + c0);
            const char* p1 = (const char*)((const T*)s1 + m0 * a.Nm + c1);
            const char* h0 = odd ? p1 : p0;
            const char* h1 = odd ? p0 : p1;
#pragma unroll
            for (int j = 0; j < MT; ++j) {
                f.x[j][0] = *reinterpret_cast<const u32x4*>(h0 + xv[j]);
                f.x[j][1] = *reinterpret_cast<const u32x4*>(h1 + xv[j]);
            }
        } else {
            const auto rxc = second ? rx2 : rx;
#pragma unroll
            for (int j = 0; j < MT; ++j)
#pragma unroll
                for (int p = 0; p < 2; ++p)
                    f.x[j][p] = __builtin_amdgcn_raw_buffer_load_b128(
                        rxc, (int)((second ? xv2[j] : xv[j]) + (p == 0 ? first : 64u - first)), (int)sk, 0);
        }
    };
    f32x4 acc[NT][MT];
#pragma unroll
    for (int i = 0; i < NT; ++i)
#pragma unroll
        for (int j = 0; j < MT; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    auto half = [&](const u32x4 (&r)[2], int p) {         // half p of the line
        if constexpr (!C::SWAP) return r[p];
        u32x4 v;
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = odd ? r[1 - p][e] : r[p][e];
        return v;
    };
    auto mma = [&](const Frags& f) {
#pragma unroll
        for (int p = 0; p < 2; ++p) {
            u32x4 w[NT], x[MT];
#pragma unroll
            for (int i = 0; i < NT; ++i) w[i] = half(f.w[i], p);
#pragma unroll
            for (int j = 0; j < MT; ++j) x[j] = half(f.x[j], p);
            if constexpr (E == 2) {
#pragma unroll
                for (int j = 0; j < MT; ++j)
#pragma unroll
                    for (int i = 0; i < NT; ++i)
                        acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                            __builtin_bit_cast(bf16x8, w[i]), __builtin_bit_cast(bf16x8, x[j]), acc[i][j], 0, 0, 0);
            } else {
#pragma unroll
                for (int e = 0; e < 4; ++e)
#pragma unroll
                    for (int j = 0; j < MT; ++j)
#pragma unroll
                        for (int i = 0; i < NT; ++i)
                            acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(
                                __uint_as_float(w[i][e]), __uint_as_float(x[j][e]), acc[i][j], 0, 0, 0);
            }
        }
    };

    // this wave's units [c0, c1); U of them in flight, every load
    // unconditional, so the loads in flight are the same on every path and each
    // wait is exact
    const int per = (nu + KW - 1) / KW;
    const int c0 = min(kw * per, nu), c1 = min(c0 + per, nu);
    Frags f[U];
#pragma unroll
    for (int u = 0; u < U; ++u) load(f[u], c0 + u);
    int c = c0;
    for (; c + U < c1; c += U) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            mma(f[u]);
            load(f[u], c + u + U);
        }
    }
#pragma unroll
    for (int u = 0; u < U; ++u)
        if (c + u < c1) mma(f[u]);

    // four consecutive columns nb .. nb+3 of row m
    auto store4 = [&](int64_t m, int64_t nb, f32x4 v) {
        if (m >= a.M || nb >= a.N) return;
        if (a.partial != nullptr) {
            float* po = a.partial + m * a.ldp + nb;
            if (nb + 3 < a.N && ((a.ldp | nb) & 3) == 0) {
                *reinterpret_cast<f32x4*>(po) = v;
            } else {
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    if (nb + r < a.N) po[r] = v[r];
            }
            return;
        }
        T* op = (T*)a.out + m * a.ldc + nb;
        if (nb + 3 < a.N && ((uintptr_t)op & (4 * E - 1)) == 0) {
            float o[4];
#pragma unroll
            for (int r = 0; r < 4; ++r) o[r] = epilogue<T>(a, m, nb + r, v[r]);
            if constexpr (E == 2)
                *reinterpret_cast<uint2*>(op) = make_uint2(pack_bf16x2(o[0], o[1]), pack_bf16x2(o[2], o[3]));
            else
                *reinterpret_cast<float4*>(op) = make_float4(o[0], o[1], o[2], o[3]);
        } else {
#pragma unroll
            for (int r = 0; r < 4; ++r)
                if (nb + r < a.N) st(op + r, epilogue<T>(a, m, nb + r, v[r]));
        }
    };
    // partial tiles to LDS: the float4 of lane (fr, fq) of tile (i, j) at
    // slot fr ^ (4*fq + i) of its 16, so that the sum below, which reads
    // row runs (consecutive threads: consecutive columns), spreads over
    // the banks
    __shared__ __attribute__((aligned(16))) f32x4 red[KW][NT * MT * 64];
#pragma unroll
    for (int i = 0; i < NT; ++i)
#pragma unroll
        for (int j = 0; j < MT; ++j)
            red[kw][(i * MT + j) * 64 + fq * 16 + (fr ^ ((4 * fq + i) & 15))] = acc[i][j];
    __syncthreads();
    constexpr int NQ = C::TN / 4;                     // float4 columns of a row
    constexpr int TOT = C::TM * NQ;
#pragma unroll
    for (int it = 0; it < (TOT + C::THREADS - 1) / C::THREADS; ++it) {
        const int q = it * C::THREADS + tid;
        if (TOT % C::THREADS != 0 && q >= TOT) break;
        const int m = q / NQ, n4 = q % NQ, i = n4 >> 2, gq = n4 & 3;
        const int at = (i * MT + (m >> 4)) * 64 + gq * 16 + ((m & 15) ^ ((4 * gq + i) & 15));
        f32x4 s = red[0][at];
#pragma unroll
        for (int w = 1; w < KW; ++w) s += red[w][at];
        store4(m0 + m, n0 + 4 * n4, s);
    }
}

}  // namespace loom
