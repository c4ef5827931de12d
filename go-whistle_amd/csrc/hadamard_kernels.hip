// gfx950 HadamardMLP: Whistle's Monarch FFN (internal/needle/hadamard.go:
// 12-24, 172-310), float32 throughout as the reference computes it, a
// wavefront per row on the fp32 matrix instruction for factors of 16 and 32
// (hadamard_wave_kernel) or, for all others, a workgroup per row with one
// thread per element of the n = na * nb mix:
//
//   cond = 1 + softmax(x @ cond_v) @ cond_u
//   z1   = kron(d1 * x; w1a, w1b)[p1]
//   z2   = kron(silu(d2 * cond * z1 + b2); w2a, w2b)[p2]
//   out  = d4 * kron(d3 * z2; w3a, w3b)
//
// kron(z; a, b) = a^T Z b with Z = z as na x nb (kronApply, hadamard.go:
// 296-310), as two small products through LDS: Y = Z b (each thread one
// element, a dot of nb), then a^T Y (a dot of na), gathered through the
// stage's permutation. x is zero-padded from the model width dim to n and
// the output cut back to dim. The reference's GEMMs (algo-tensor, absent)
// sum in an order of their own, so the result is held to the reference
// test's bar: within 1e-5 of the float64 form (hadamard_test.go:152-191).
#include "cq_internal.hpp"
#include "cq_device.hpp"

#include <algorithm>

namespace cqhip {
namespace {

constexpr int kHadaMaxN = 1024;
constexpr int kHadaMaxRank = 32;

// out[c] = (a^T Z b)[c] for c = tid < n, Z in zs; ys is scratch of n.
__device__ __forceinline__ float kron_elem(const float *zs, float *ys, const float *a, const float *b, int na,
                                           int nb, int tid, int n) {
    if (tid < n) {
        const int i = tid / nb, l = tid - i * nb;  // Y[i][l] = sum_j Z[i][j] b[j][l]
        float y = 0.0f;
        for (int j = 0; j < nb; ++j) {
            const float p = zs[i * nb + j] * b[j * nb + l];
            y = y + p;
        }
        ys[tid] = y;
    }
    __syncthreads();
    float o = 0.0f;
    if (tid < n) {
        const int k = tid / nb, l = tid - k * nb;  // out[k][l] = sum_i a[i][k] Y[i][l]
        for (int i = 0; i < na; ++i) {
            const float p = a[i * na + k] * ys[i * nb + l];
            o = o + p;
        }
    }
    __syncthreads();
    return o;
}

__global__ __launch_bounds__(kHadaMaxN) void hadamard_mlp_kernel(HadaArgs h) {
    __shared__ float zs[kHadaMaxN], ys[kHadaMaxN], ks[kHadaMaxN];
    __shared__ float part[kHadaMaxN / 64][kHadaMaxRank];
    __shared__ float prob[kHadaMaxRank];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, nw = blockDim.x >> 6;
    const int n = h.na * h.nb, dim = h.dim, rank = h.rank;
    const float *x = h.x + static_cast<long long>(blockIdx.x) * dim;
    float *out = h.out + static_cast<long long>(blockIdx.x) * dim;

    // The conditioning logits x @ cond_v (linear, hadamard.go:176-177): per
    // wavefront partial sums of its 64 inputs, reduced across lanes, then
    // across wavefronts.
    const float xv = tid < dim ? x[tid] : 0.0f;
    for (int r = 0; r < rank; ++r) {
        float v = tid < dim ? xv * h.cond_v[static_cast<long long>(tid) * rank + r] : 0.0f;
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) v = v + __shfl_xor(v, off);
        if (lane == 0) part[wave][r] = v;
    }
    __syncthreads();
    if (tid == 0) {  // softmax over the rank logits (in LDS: no private array)
        float m = -INFINITY;
        for (int r = 0; r < rank; ++r) {
            float s = 0.0f;
            for (int w = 0; w < nw; ++w) s = s + part[w][r];
            prob[r] = s;
            m = go_max(m, s);
        }
        float sum = 0.0f;
        for (int r = 0; r < rank; ++r) {
            prob[r] = expf(prob[r] - m);
            sum = sum + prob[r];
        }
        for (int r = 0; r < rank; ++r) prob[r] = prob[r] / sum;
    }
    __syncthreads();
    float cond = 1.0f;  // 1 + softmax @ cond_u
    if (tid < n) {
        float c = 0.0f;
        for (int r = 0; r < rank; ++r) {
            const float p = prob[r] * h.cond_u[static_cast<long long>(r) * n + tid];
            c = c + p;
        }
        cond = c + 1.0f;
    }

    // z1 = kron(d1 * x; w1)[p1]
    if (tid < n) zs[tid] = tid < dim ? h.d1[tid] * xv : 0.0f;
    __syncthreads();
    float k = kron_elem(zs, ys, h.w1a, h.w1b, h.na, h.nb, tid, n);
    if (tid < n) ks[tid] = k;
    __syncthreads();
    // z2 = kron(silu(d2 * cond * z1 + b2); w2)[p2], sigma as jax.nn.sigmoid
    if (tid < n) {
        const int q = h.p1[tid];
        const float z1 = ks[static_cast<unsigned>(q) < static_cast<unsigned>(n) ? q : 0];  // a permutation of n
        const float t1 = h.d2[tid] * cond;
        const float a = t1 * z1 + h.b2[tid];
        zs[tid] = a * gate_sigmoid(a);
    }
    __syncthreads();
    k = kron_elem(zs, ys, h.w2a, h.w2b, h.na, h.nb, tid, n);
    if (tid < n) ks[tid] = k;
    __syncthreads();
    // out = d4 * kron(d3 * z2; w3)
    if (tid < n) {
        const int q = h.p2[tid];
        zs[tid] = h.d3[tid] * ks[static_cast<unsigned>(q) < static_cast<unsigned>(n) ? q : 0];
    }
    __syncthreads();
    k = kron_elem(zs, ys, h.w3a, h.w3b, h.na, h.nb, tid, n);
    if (tid < dim) out[tid] = h.d4[tid] * k;
}

// A stage's mix of one row on one wavefront, with the fp32 matrix instruction
// v_mfma_f32_16x16x4 (TA x TB tiles of 16; lane = 16 q + c). Z comes in as the
// A operand, lane's rows 16 ta + c, columns 4 TB q + s: Y = Z b runs over its
// columns in that order. A result register r is row 16 ta + 4 q + r of Y, which
// is the B operand of a^T Y as it lies when the sum over Y's rows takes them
// as (ta, r) with row 16 ta + 4 q + r in lane group q: no exchange between the
// two products. out: [k tile][l tile], register r of row 16 tk + 4 q + r,
// column 16 tb + c.
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x4u __attribute__((ext_vector_type(4), aligned(4)));  // loaded from any float's address

template <int TA, int TB>
struct Mix {
    float a[TA][4 * TA];  // a[16 ta + 4 q + r][16 tk + c] at [tk][4 ta + r]
    float b[TB][4 * TB];  // b[4 TB q + s][16 tb + c] at [tb][s]
    __device__ __forceinline__ void load(const float *pa, const float *pb, int q, int c) {
#pragma unroll
        for (int tk = 0; tk < TA; ++tk)
#pragma unroll
            for (int i = 0; i < 4 * TA; ++i) a[tk][i] = pa[((i >> 2) * 16 + 4 * q + (i & 3)) * (16 * TA) + tk * 16 + c];
#pragma unroll
        for (int tb = 0; tb < TB; ++tb)
#pragma unroll
            for (int s = 0; s < 4 * TB; ++s) b[tb][s] = pb[(4 * TB * q + s) * (16 * TB) + tb * 16 + c];
    }
    __device__ __forceinline__ void run(const float (&z)[TA][4 * TB], f32x4 (&out)[TA][TB]) const {
        f32x4 y[TA][TB];
#pragma unroll
        for (int ta = 0; ta < TA; ++ta)
#pragma unroll
            for (int tb = 0; tb < TB; ++tb) y[ta][tb] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int s = 0; s < 4 * TB; ++s)
#pragma unroll
            for (int ta = 0; ta < TA; ++ta)
#pragma unroll
                for (int tb = 0; tb < TB; ++tb)
                    y[ta][tb] = __builtin_amdgcn_mfma_f32_16x16x4f32(z[ta][s], b[tb][s], y[ta][tb], 0, 0, 0);
#pragma unroll
        for (int tk = 0; tk < TA; ++tk)
#pragma unroll
            for (int tb = 0; tb < TB; ++tb) out[tk][tb] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int i = 0; i < 4 * TA; ++i)
#pragma unroll
            for (int tk = 0; tk < TA; ++tk)
#pragma unroll
                for (int tb = 0; tb < TB; ++tb)
                    out[tk][tb] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[tk][i], y[i >> 2][tb][i & 3], out[tk][tb], 0, 0, 0);
    }
};

// HadamardMLP for factors na = 16 TA and nb = 16 TB, a wavefront per row: the
// row's values stay in registers in the A operand's order, the mixes run on the
// matrix cores, and only the permutations go through LDS (the wavefront's
// own, no barrier). A workgroup stages the conditioning weights in LDS once
// (CL, where they fit; in the lanes' order, free of bank conflicts) and its
// four wavefronts run rows in turn with the factors and the element vectors
// in registers, so the weights (60 KiB at 16 x 32 and rank 8) are read once a
// workgroup and behind one load latency instead of one a stage. VEC: dim is a
// multiple of 4, so that a lane's 4 TB columns are whole float4s, loaded from
// any float's address.
// What bounds it: at few rows one row's latency (two load rounds, three pairs
// of products, the float64 sigmoids), then VALU (the sigmoids' float64 and the
// cross-lane sums). Measured on MI355X against the workgroup form (us): 16 x 32
// of 512, rank 8, at 1, 375, 3000 and 12,000 rows 11.5, 15.6, 60, 211 ->
// 8.4, 9.5, 18, 49; of 511 11.5, 15.7, 60, 212 -> 9.2, 10.1, 20, 52; 32 x 32 of
// 1024, rank 16, 23.2, 39.9, 200, 758 -> 21.7, 23.5, 59, 182; 16 x 16 of 256
// 10.8, 12.0, 32.7, 93 -> 5.1, 5.7, 9.5, 26. Its sums are fused (2.4e-7 from the
// float64 form over rows of 512, against 2.5e-7).
template <int TA, int TB, bool VEC, bool CL>
__global__ __launch_bounds__(256) void hadamard_wave_kernel(HadaArgs h, int rows) {
    constexpr int S = 4 * TB, E = TA * S;  // a lane's elements of a row
    extern __shared__ __align__(16) unsigned char smem[];
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6, q = lane >> 4, c = lane & 15;
    constexpr int nb = 16 * TB, n = 16 * TA * nb;
    const int dim = h.dim, rank = h.rank;
    float *zs = reinterpret_cast<float *>(smem) + w * (TA * TB * 256);
    float *cvl = reinterpret_cast<float *>(smem) + 4 * TA * TB * 256;  // [rank / 8][E][2][64][4]
    const int rc = (rank + 7) >> 3;
    float *cul = cvl + static_cast<size_t>(rc) * E * 512;              // [rank][E / 4][64][4]

    // element ta, s of the lane: index (16 ta + c) nb + 4 TB q + s of the mix
    auto index = [&](int ta, int s) { return (16 * ta + c) * nb + S * q + s; };
    // Elements s .. s + 3 of p, zero from lim on. Every load goes out, from inside
    // p: a branch around each would have the next wait for it.
    auto gather4 = [&](const float *p, int ta, int s, int lim) -> float4 {
        const int e = index(ta, s);
        float f[4];
        if constexpr (VEC) {
            const f32x4u v = *reinterpret_cast<const f32x4u *>(p + min(e, lim - 4));
#pragma unroll
            for (int k = 0; k < 4; ++k) f[k] = v[k];
        } else {
#pragma unroll
            for (int k = 0; k < 4; ++k) f[k] = p[min(e + k, lim - 1)];
        }
#pragma unroll
        for (int k = 0; k < 4; ++k) f[k] = e + k < lim ? f[k] : 0.0f;
        return make_float4(f[0], f[1], f[2], f[3]);
    };
    auto gather = [&](float (&d)[TA][S], const float *p, int lim) {
#pragma unroll
        for (int ta = 0; ta < TA; ++ta)
#pragma unroll
            for (int s = 0; s < S; s += 4) {
                const float4 f = gather4(p, ta, s, lim);
                d[ta][s] = f.x;
                d[ta][s + 1] = f.y;
                d[ta][s + 2] = f.z;
                d[ta][s + 3] = f.w;
            }
    };
    // eight conditioning weights of an element, ranks 8 k0 ..
    auto cond8 = [&](int ta, int s, int k0, float4 &f0, float4 &f1) {
        const int e = index(ta, s);
        const float *p = h.cond_v + static_cast<long long>(min(e, dim - 1)) * rank + 8 * k0;
        float v[8];
        if ((rank & 7) == 0) {
            const f32x4u a = *reinterpret_cast<const f32x4u *>(p), b = *reinterpret_cast<const f32x4u *>(p + 4);
#pragma unroll
            for (int k = 0; k < 4; ++k) v[k] = a[k], v[4 + k] = b[k];
        } else {
#pragma unroll
            for (int k = 0; k < 8; ++k) v[k] = p[min(k, rank - 1 - 8 * k0)];
        }
#pragma unroll
        for (int k = 0; k < 8; ++k) v[k] = e < dim && 8 * k0 + k < rank ? v[k] : 0.0f;
        f0 = make_float4(v[0], v[1], v[2], v[3]);
        f1 = make_float4(v[4], v[5], v[6], v[7]);
    };

    int row = blockIdx.x * 4 + w;
    float xv[TA][S], d1[TA][S], d2[TA][S], b2[TA][S], d3[TA][S], d4[TA][TB][4];
    int p1[TA][S], p2[TA][S];
    gather(xv, h.x + static_cast<long long>(min(row, rows - 1)) * dim, dim);
    gather(d1, h.d1, n);
    Mix<TA, TB> m1, m2, m3;
    m1.load(h.w1a, h.w1b, q, c);
    if constexpr (CL) {
        for (int k0 = 0; k0 < rc; ++k0)
            for (int i = w; i < E; i += 4) {
                float4 f0, f1;
                cond8(i / S, i % S, k0, f0, f1);
                float *d = cvl + ((k0 * E + i) * 2 * 64 + lane) * 4;
                *reinterpret_cast<float4 *>(d) = f0;
                *reinterpret_cast<float4 *>(d + 256) = f1;
            }
        for (int i = w; i < rank * (E / 4); i += 4) {
            const int r = i / (E / 4), e4 = i - r * (E / 4);
            *reinterpret_cast<float4 *>(cul + (i * 64 + lane) * 4) =
                gather4(h.cond_u + static_cast<long long>(r) * n, e4 * 4 / S, e4 * 4 % S, n);
        }
    }
    m2.load(h.w2a, h.w2b, q, c);
    m3.load(h.w3a, h.w3b, q, c);
    gather(d2, h.d2, n);
    gather(b2, h.b2, n);
    gather(d3, h.d3, n);
#pragma unroll
    for (int ta = 0; ta < TA; ++ta)
#pragma unroll
        for (int s = 0; s < S; ++s) {
            p1[ta][s] = h.p1[index(ta, s)];
            p2[ta][s] = h.p2[index(ta, s)];
            if (static_cast<unsigned>(p1[ta][s]) >= static_cast<unsigned>(n)) p1[ta][s] = 0;  // a permutation of n
            if (static_cast<unsigned>(p2[ta][s]) >= static_cast<unsigned>(n)) p2[ta][s] = 0;
        }
    auto result = [&](int tk, int tb, int r) { return (16 * tk + 4 * q + r) * nb + 16 * tb + c; };  // register r's index of the mix
#pragma unroll
    for (int tk = 0; tk < TA; ++tk)
#pragma unroll
        for (int tb = 0; tb < TB; ++tb)
#pragma unroll
            for (int r = 0; r < 4; ++r) d4[tk][tb][r] = h.d4[result(tk, tb, r)];
    if constexpr (CL) __syncthreads();  // the only barrier: a wavefront is on its own from here

    for (; row < rows; row += 4 * gridDim.x) {
        const int next = min(row + 4 * static_cast<int>(gridDim.x), rows - 1);
        float z[TA][S], xn[TA][S];
        gather(xn, h.x + static_cast<long long>(next) * dim, dim);  // the next row's values, under this row's work
#pragma unroll
        for (int ta = 0; ta < TA; ++ta)
#pragma unroll
            for (int s = 0; s < S; ++s) z[ta][s] = d1[ta][s] * xv[ta][s];
        f32x4 o[TA][TB];
        m1.run(z, o);
        auto to_lds = [&]() {
#pragma unroll
            for (int tk = 0; tk < TA; ++tk)
#pragma unroll
                for (int tb = 0; tb < TB; ++tb)
#pragma unroll
                    for (int r = 0; r < 4; ++r) zs[result(tk, tb, r)] = o[tk][tb][r];
        };
        to_lds();

        // cond = 1 + softmax(x cond_v) cond_u (hadamard.go:176-190): eight
        // logits at a time, a lane's values then across the lanes; lane r
        // keeps logit r.
        float lg = -INFINITY;
        for (int k0 = 0; k0 < rc; ++k0) {
            float v[8];
#pragma unroll
            for (int k = 0; k < 8; ++k) v[k] = 0.0f;
#pragma unroll
            for (int ta = 0; ta < TA; ++ta)
#pragma unroll
                for (int s = 0; s < S; ++s) {
                    float4 f0, f1;
                    if constexpr (CL) {
                        const float *d = cvl + ((k0 * E + ta * S + s) * 2 * 64 + lane) * 4;
                        f0 = *reinterpret_cast<const float4 *>(d);
                        f1 = *reinterpret_cast<const float4 *>(d + 256);
                    } else {
                        cond8(ta, s, k0, f0, f1);
                    }
                    const float cv[8] = {f0.x, f0.y, f0.z, f0.w, f1.x, f1.y, f1.z, f1.w};
#pragma unroll
                    for (int k = 0; k < 8; ++k) v[k] = fmaf(xv[ta][s], cv[k], v[k]);
                }
#pragma unroll
            for (int hh = 1; hh < 64; hh <<= 1)
#pragma unroll
                for (int k = 0; k < 8; ++k) v[k] = v[k] + xor_lane(v[k], hh);
#pragma unroll
            for (int k = 0; k < 8; ++k)
                if (lane == 8 * k0 + k && lane < rank) lg = v[k];
        }
        float mx = lg;
#pragma unroll
        for (int hh = 32; hh > 0; hh >>= 1) mx = go_max(mx, xor_lane(mx, hh));
        const float ex = lane < rank ? expf(lg - mx) : 0.0f;
        float sum = ex;
#pragma unroll
        for (int hh = 1; hh < 64; hh <<= 1) sum = sum + xor_lane(sum, hh);
        const float prob = ex / sum;
        float cond[TA][S];
#pragma unroll
        for (int ta = 0; ta < TA; ++ta)
#pragma unroll
            for (int s = 0; s < S; ++s) cond[ta][s] = 0.0f;
        for (int r = 0; r < rank; ++r) {
            const float p = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, prob), r));
#pragma unroll
            for (int ta = 0; ta < TA; ++ta)
#pragma unroll
                for (int s = 0; s < S; s += 4) {
                    const float4 f = CL ? *reinterpret_cast<const float4 *>(cul + ((r * (E / 4) + (ta * S + s) / 4) * 64 + lane) * 4)
                                        : gather4(h.cond_u + static_cast<long long>(r) * n, ta, s, n);
                    cond[ta][s] = fmaf(p, f.x, cond[ta][s]);
                    cond[ta][s + 1] = fmaf(p, f.y, cond[ta][s + 1]);
                    cond[ta][s + 2] = fmaf(p, f.z, cond[ta][s + 2]);
                    cond[ta][s + 3] = fmaf(p, f.w, cond[ta][s + 3]);
                }
        }

        // z2's input: silu(d2 cond z1 + b2), z1 through p1
#pragma unroll
        for (int ta = 0; ta < TA; ++ta)
#pragma unroll
            for (int s = 0; s < S; ++s) {
                const float t1 = d2[ta][s] * (cond[ta][s] + 1.0f);
                const float a = t1 * zs[p1[ta][s]] + b2[ta][s];
                z[ta][s] = a * gate_sigmoid(a);
            }
        m2.run(z, o);
        to_lds();
#pragma unroll
        for (int ta = 0; ta < TA; ++ta)
#pragma unroll
            for (int s = 0; s < S; ++s) z[ta][s] = d3[ta][s] * zs[p2[ta][s]];
        m3.run(z, o);
        float *out = h.out + static_cast<long long>(row) * dim;
#pragma unroll
        for (int tk = 0; tk < TA; ++tk)
#pragma unroll
            for (int tb = 0; tb < TB; ++tb)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int e = result(tk, tb, r);
                    if (e < dim) out[e] = d4[tk][tb][r] * o[tk][tb][r];
                }
#pragma unroll
        for (int ta = 0; ta < TA; ++ta)
#pragma unroll
            for (int s = 0; s < S; ++s) xv[ta][s] = xn[ta][s];
    }
}

template <int TA, int TB, bool VEC, bool CL>
hipError_t launch_wave_t(const HadaArgs &h, int rows, size_t lds, int cus, hipStream_t s) {
    static std::atomic<unsigned long long> attr{0};
    if (hipError_t e = lds_limit_once(reinterpret_cast<const void *>(&hadamard_wave_kernel<TA, TB, VEC, CL>), 160 * 1024, attr))
        return e;
    const int wgs = (rows + 3) / 4;  // four wavefronts, each a row at a time; two workgroups a CU at most
    hipLaunchKernelGGL((hadamard_wave_kernel<TA, TB, VEC, CL>), dim3(wgs < 2 * cus ? wgs : 2 * cus), dim3(256), lds, s, h,
                       rows);
    return hipGetLastError();
}

template <int TA, int TB>
hipError_t launch_wave(const HadaArgs &h, int rows, int cus, hipStream_t s) {
    constexpr size_t zs = sizeof(float) * 4 * TA * TB * 256, elems = 4 * TA * TB;
    const size_t lds = zs + sizeof(float) * elems * 64 * ((h.rank + 7) / 8 * 8 + h.rank);
    const bool vec = h.dim % 4 == 0, cl = lds <= 150 * 1024;  // whole float4s a row; the conditioning weights fit
    if (vec) return cl ? launch_wave_t<TA, TB, true, true>(h, rows, lds, cus, s) : launch_wave_t<TA, TB, true, false>(h, rows, zs, cus, s);
    return cl ? launch_wave_t<TA, TB, false, true>(h, rows, lds, cus, s) : launch_wave_t<TA, TB, false, false>(h, rows, zs, cus, s);
}

}  // namespace

hipError_t launch_hadamard_mlp(const HadaArgs &h, int rows, int cus, hipStream_t s) {
    if (rows <= 0) return hipSuccess;
    // By the shape alone, never the rows or the pointers: the two forms sum in
    // different orders, and a row's result is the same in every call. Factors
    // that do not fill their tiles stay on the workgroup form: on the wavefront
    // form, their edges checked, 24 x 32 of 768, rank 8, took 21.5 against 15.2
    // us at one row, 22.5, 23.0 at 375 and 167, 451 at 12,000.
    if ((h.na == 16 || h.na == 32) && (h.nb == 16 || h.nb == 32)) {
        if (h.na == 16) return h.nb == 16 ? launch_wave<1, 1>(h, rows, cus, s) : launch_wave<1, 2>(h, rows, cus, s);
        return h.nb == 16 ? launch_wave<2, 1>(h, rows, cus, s) : launch_wave<2, 2>(h, rows, cus, s);
    }
    const int n = h.na * h.nb;
    const int threads = (n + 63) / 64 * 64;
    const long long most = grid_limit(threads);
    for (long long r0 = 0; r0 < rows; r0 += most) {
        HadaArgs b = h;
        b.x = h.x + r0 * h.dim;
        b.out = h.out + r0 * h.dim;
        hipLaunchKernelGGL(hadamard_mlp_kernel, dim3(static_cast<unsigned>(std::min(most, rows - r0))), dim3(threads), 0, s, b);
        if (hipError_t e = hipGetLastError()) return e;
    }
    return hipSuccess;
}

bool hadamard_shape_ok(int na, int nb, int dim, int rank) {
    const long long n = static_cast<long long>(na) * nb;
    return na > 0 && nb > 0 && n <= kHadaMaxN && dim > 0 && dim <= n && rank > 0 && rank <= kHadaMaxRank;
}

}  // namespace cqhip
