// Sequence form of the sparse final cross-attention on the matrix cores
// (included by tria.hip): 16 query rows of one batch row per block, so the
// block's keys and values are read once for 16 rows (the one-row kernels read
// them once per row: 8 x 2048 rows over 15 keys of 768 in bf16 253 us, here 14; on
// operands no cache holds yet, launch included, 283 and 38).
//
// Four waves share the D dimensions in slabs of 64: wave w takes slabs w, w+4,
// ... of the scores S = K Q^T (summed over the waves through LDS) and then of
// the output.  S lies with query l%16 and keys 4*(l/16)+r of a 16-key tile in
// lane l, register r; the softmax runs over registers, key tiles and the four
// lane groups.  P stays fp32: O^T = V^T P^T on v_mfma_f32_16x16x4_f32, step r
// taking keys {4g + r}, which is P as it lies; a lane's A operand of step r is
// V[4*(l/16)+r][64s + 4*(l%16) + t], four consecutive values for t = 0..3, and
// its results are 16 consecutive dimensions of its query.
#pragma once

namespace loom {

typedef __bf16 ca_bf16x8 __attribute__((ext_vector_type(8)));
typedef float ca_f32x4 __attribute__((ext_vector_type(4)));

constexpr int kCaTileRows = 16;
constexpr int kCaTileMaxSlabs = 4;     // slabs of 64 dimensions per wave (D <= 1024)

// one row's slab as MFMA operands: C chunks of 64 bytes per 64 elements,
// register c of lane l = bytes 64c + 16*(l/16) of row l%16 (odd rows ask for
// the chunks of a line in the other order, see gemm_frag.h)
template <typename T>
struct CaSlab {
    static constexpr int C = (int)sizeof(T);
    u32x4 r[C];
    __device__ __forceinline__ void load(const T* row, int slab, int fq, bool odd) {
        const char* p = (const char*)(row + 64 * slab) + 16 * fq;
#pragma unroll
        for (int c = 0; c < C; ++c) r[c] = *reinterpret_cast<const u32x4*>(p + 64 * (c ^ (odd ? 1 : 0)));
    }
    __device__ __forceinline__ u32x4 get(int c, bool odd) const {
        u32x4 v;
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = odd ? r[c ^ 1][e] : r[c][e];
        return v;
    }
};

// Independent MFMA chains of a score tile, added pairwise at the end: shorter
// chains issue back to back and round less (fp32: sixteen of 12 products each at
// D = 768, where one chain per wave doubled the error of the one-row kernels).
template <typename T> constexpr int kCaChains = sizeof(T) == 2 ? 2 : 16;

template <typename T>
__device__ __forceinline__ void ca_scores(const CaSlab<T>& k, const CaSlab<T>& q, bool odd,
                                          ca_f32x4 (&s)[kCaChains<T>]) {
#pragma unroll
    for (int c = 0; c < CaSlab<T>::C; ++c) {
        const u32x4 a = k.get(c, odd), b = q.get(c, odd);
        if constexpr (sizeof(T) == 2) {
            s[c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(ca_bf16x8, a),
                                                           __builtin_bit_cast(ca_bf16x8, b), s[c], 0, 0, 0);
        } else {
#pragma unroll
            for (int e = 0; e < 4; ++e)
                s[4 * c + e] = __builtin_amdgcn_mfma_f32_16x16x4f32(__uint_as_float(a[e]), __uint_as_float(b[e]),
                                                                    s[4 * c + e], 0, 0, 0);
        }
    }
}

// four consecutive elements
__device__ __forceinline__ void ca_load4(const bf16_t* p, float v[4]) {
    const uint2 w = *reinterpret_cast<const uint2*>(p);
    v[0] = __uint_as_float(w.x << 16); v[1] = __uint_as_float(w.x & 0xffff0000u);
    v[2] = __uint_as_float(w.y << 16); v[3] = __uint_as_float(w.y & 0xffff0000u);
}
__device__ __forceinline__ void ca_load4(const float* p, float v[4]) {
    const float4 w = *reinterpret_cast<const float4*>(p);
    v[0] = w.x; v[1] = w.y; v[2] = w.z; v[3] = w.w;
}

// NKT: 16-key tiles (K <= 16 * NKT); NS: slabs per wave (D <= 256 * NS)
template <typename T, int NKT, int NS>
__global__ void __launch_bounds__(256)
final_ca_tile_kernel(const T* __restrict__ q, const T* __restrict__ k, const T* __restrict__ v,
                     int64_t kv_stride_b, const uint8_t* __restrict__ allowed, int64_t allowed_stride,
                     const T* __restrict__ residual, float gamma, T* __restrict__ out,
                     float* __restrict__ lse, int64_t T_, int64_t K, const int64_t* __restrict__ k_dev,
                     int D, float scale) {
    __shared__ ca_f32x4 part[4][NKT][64];
    const int64_t Kcap = K;                                   // rows the cache holds (>= 1)
    if (k_dev != nullptr) K = *k_dev < K ? *k_dev : K;        // graph replay: key count on the device
    const int64_t tiles = ceil_div(T_, kCaTileRows);
    const int64_t b = blockIdx.x / tiles, t0 = (blockIdx.x - b * tiles) * kCaTileRows;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int fr = lane & 15, fq = lane >> 4;
    const bool odd = (fr & 1) != 0;
    const int64_t row = b * T_ + min(t0 + fr, T_ - 1);        // this lane's query row
    const bool live = t0 + fr < T_;
    const int slabs = D / 64;
    const T* kb = k + b * kv_stride_b;
    const T* vb = v + b * kv_stride_b;

    // the mask bytes of the lane's keys, requested before anything waits
    uint8_t al[NKT][4];
#pragma unroll
    for (int n = 0; n < NKT; ++n)
#pragma unroll
        for (int r = 0; r < 4; ++r)
            al[n][r] = allowed[row * allowed_stride + min((int64_t)(16 * n + 4 * fq + r), Kcap - 1)];
    CaSlab<T> qs[NS];
#pragma unroll
    for (int i = 0; i < NS; ++i)
        qs[i].load(q + row * D, min(wave + 4 * i, slabs - 1), fq, odd);
    // slabs past D are loaded (the last one again) and not used
    ca_f32x4 s[NKT];
#pragma unroll
    for (int n = 0; n < NKT; ++n) {
        const T* kr = kb + min((int64_t)(16 * n + fr), Kcap - 1) * D;
        CaSlab<T> ks[NS];
#pragma unroll
        for (int i = 0; i < NS; ++i) ks[i].load(kr, min(wave + 4 * i, slabs - 1), fq, odd);
        ca_f32x4 c[kCaChains<T>];
#pragma unroll
        for (int i = 0; i < kCaChains<T>; ++i) c[i] = ca_f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int i = 0; i < NS; ++i)
            if (wave + 4 * i < slabs) ca_scores<T>(ks[i], qs[i], odd, c);
#pragma unroll
        for (int h = kCaChains<T> / 2; h > 0; h >>= 1)
#pragma unroll
            for (int i = 0; i < h; ++i) c[i] += c[i + h];
        part[wave][n][lane] = c[0];
    }
    __syncthreads();
    float mx = -INFINITY;
#pragma unroll
    for (int n = 0; n < NKT; ++n) {
        s[n] = (part[0][n][lane] + part[1][n][lane]) + (part[2][n][lane] + part[3][n][lane]);
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const bool ok = 16 * n + 4 * fq + r < K && al[n][r] != 0;
            s[n][r] = ok ? s[n][r] * scale : -INFINITY;
            mx = fmaxf(mx, s[n][r]);
        }
    }
    mx = fmaxf(mx, __shfl_xor(mx, 16, 64));
    mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
    float sum = 0.0f;
#pragma unroll
    for (int n = 0; n < NKT; ++n)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            s[n][r] = s[n][r] == -INFINITY ? 0.0f : fexp(s[n][r] - mx);
            sum += s[n][r];
        }
    sum += __shfl_xor(sum, 16, 64);
    sum += __shfl_xor(sum, 32, 64);
    const float inv = ca_inv(sum);
#pragma unroll
    for (int n = 0; n < NKT; ++n)
#pragma unroll
        for (int r = 0; r < 4; ++r) s[n][r] *= inv;
    if (lse != nullptr && tid < 16 && live) lse[row] = ca_lse(mx, sum);

    for (int sl = wave; sl < slabs; sl += 4) {
        ca_f32x4 acc[4];
#pragma unroll
        for (int t = 0; t < 4; ++t) acc[t] = ca_f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int n = 0; n < NKT; ++n) {
            float vv[4][4];
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int64_t key = 16 * n + 4 * fq + r;
                ca_load4(vb + min(key, Kcap - 1) * D + 64 * sl + 4 * fr, vv[r]);
#pragma unroll
                for (int t = 0; t < 4; ++t) vv[r][t] = key < K ? vv[r][t] : 0.0f;
            }
#pragma unroll
            for (int r = 0; r < 4; ++r)
#pragma unroll
                for (int t = 0; t < 4; ++t)
                    acc[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(vv[r][t], s[n][r], acc[t], 0, 0, 0);
        }
        if (!live) continue;
        // dimension 64 sl + 16 fq + 4 rr + t of query fr
        const int64_t o = row * D + 64 * sl + 16 * fq;
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            float y[8];
#pragma unroll
            for (int e = 0; e < 8; ++e) y[e] = acc[e & 3][2 * h + (e >> 2)];
            if (residual != nullptr) {
                float rr[8];
                Vec8<T>::load(residual + o + 8 * h, rr);
#pragma unroll
                for (int e = 0; e < 8; ++e) y[e] = rr[e] + gamma * y[e];
            }
            Vec8<T>::store(out + o + 8 * h, y);
        }
    }
}

}  // namespace loom
