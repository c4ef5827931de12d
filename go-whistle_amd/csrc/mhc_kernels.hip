// gfx950 manifold hyper-connections around a block (internal/needle/mhc.go),
// the pieces on either side of the φ products (which are CQ GEMMs of
// In = lanes * dim): RMSUnit of the lane stream (norm.go:68-81), the heads
// h_pre = sigmoid, h_post = 2 sigmoid and h_res = sinkhorn of their logits
// with the block input u = sum_k h_pre[k] stream[k] (mhc.go:204-219), and
// the mix out[a] = sum_b h_res[a, b] stream[b] + h_post[a] (block(u) - u)
// (mhc.go:229-299). Each is the reference's float32 arithmetic in its
// order; the Sinkhorn runs in float64 in the exp domain (exp_f64, the
// CPU restatement's operations) while the logits' spread allows it, else
// in float32 in the log domain (mhc.go:301-417).
#include "cq_internal.hpp"
#include "cq_device.hpp"

#include <algorithm>

namespace cqhip {
namespace {

constexpr int kMhcMaxLanes = 8;

__global__ __launch_bounds__(64) void rms_unit_kernel(float *dst, const float *x, int dim) {
    const float *row = x + static_cast<long long>(blockIdx.x) * dim;
    float *out = dst + static_cast<long long>(blockIdx.x) * dim;
    const int lane = threadIdx.x;
    const double part = lane < 4 ? zc_partial(row, dim, lane) : 0.0;
    const double p0 = __shfl(part, 0), p1 = __shfl(part, 1), p2 = __shfl(part, 2), p3 = __shfl(part, 3);
    const double s = ((p0 + p1) + p2) + p3;
    const float ms = static_cast<float>(s / static_cast<double>(dim));
    const float e = ms + 1e-6f;
    const float inv = static_cast<float>(1.0 / sqrt(static_cast<double>(e)));
    for (int c = lane; c < dim; c += 64) out[c] = row[c] * inv;
}

// The exp-domain iterations for N lanes a power of two up to 4: the row's
// sum reads its quad's entries by DPP (the entries of a row of 4, or two rows
// of 2, are one quad of lanes), the column's by ds_bpermute, all of them
// issued before the first add; the generic loop waited on each exchange.
// The same operations in the same order. The 40 passes are a chain of an
// exchange, N adds and a float64 divide each: one heads call of one row of 4 x
// 512 took 11.6 us with the generic loop, 4.2 us now, 375 rows 13.8 -> 7.5 us
// (MI355X, kernel trace; u formed beside the Sinkhorn instead of after it).
template <int N>
__device__ __forceinline__ double sinkhorn_exp(double e, int iters, int r, int c) {
    auto quad = [&](int j) -> double {  // entry j of the lane's row
        const long long b = __builtin_bit_cast(long long, e);
        int lo = static_cast<int>(b), hi = static_cast<int>(b >> 32);
        if (N == 4) {
            switch (j) {
                case 0: lo = __builtin_amdgcn_update_dpp(0, lo, 0x00, 0xF, 0xF, true); hi = __builtin_amdgcn_update_dpp(0, hi, 0x00, 0xF, 0xF, true); break;
                case 1: lo = __builtin_amdgcn_update_dpp(0, lo, 0x55, 0xF, 0xF, true); hi = __builtin_amdgcn_update_dpp(0, hi, 0x55, 0xF, 0xF, true); break;
                case 2: lo = __builtin_amdgcn_update_dpp(0, lo, 0xAA, 0xF, 0xF, true); hi = __builtin_amdgcn_update_dpp(0, hi, 0xAA, 0xF, 0xF, true); break;
                default: lo = __builtin_amdgcn_update_dpp(0, lo, 0xFF, 0xF, 0xF, true); hi = __builtin_amdgcn_update_dpp(0, hi, 0xFF, 0xF, 0xF, true); break;
            }
        } else if (j == 0) {  // [0, 0, 2, 2]
            lo = __builtin_amdgcn_update_dpp(0, lo, 0xA0, 0xF, 0xF, true);
            hi = __builtin_amdgcn_update_dpp(0, hi, 0xA0, 0xF, 0xF, true);
        } else {  // [1, 1, 3, 3]
            lo = __builtin_amdgcn_update_dpp(0, lo, 0xF5, 0xF, 0xF, true);
            hi = __builtin_amdgcn_update_dpp(0, hi, 0xF5, 0xF, 0xF, true);
        }
        return __builtin_bit_cast(double, static_cast<long long>(static_cast<unsigned long long>(static_cast<unsigned>(hi)) << 32 |
                                                                 static_cast<unsigned>(lo)));
    };
    for (int it = 0; it < iters; ++it) {
        double v[N];
#pragma unroll
        for (int j = 0; j < N; ++j) v[j] = quad(j);
        double s = 0.0;
#pragma unroll
        for (int j = 0; j < N; ++j) s = s + v[j];
        e = e / s;
#pragma unroll
        for (int j = 0; j < N; ++j) v[j] = __shfl(e, j * N + c);
        s = 0.0;
#pragma unroll
        for (int j = 0; j < N; ++j) s = s + v[j];
        e = e / s;
    }
    return e;
}

// sinkhorn (mhc.go:301-399) of one n x n matrix in k (LDS) by one
// wavefront: lane t < n*n holds entry t = r*n + c. Rows (then columns) are
// independent within a pass, so each lane forms its row's (column's) sum in
// the reference's order from its neighbours' values and divides its own
// entry: the serial routine's operations, n*n of them at a time.
__device__ void sinkhorn_wave(float *k, int n, int iters, int lane) {
    const int nn = n * n;
    const bool act = lane < nn;
    const int r = act ? lane / n : 0, c = act ? lane - r * n : 0;
    float kv = act ? k[lane] : k[0];  // idle lanes repeat entry 0: neutral for min and max
    // slices.Min / slices.Max keep a NaN; min and max are exact in any order
    float lo = kv, hi = kv;
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
        lo = go_min(lo, __shfl_xor(lo, off));
        hi = go_max(hi, __shfl_xor(hi, off));
    }
    const double spread = static_cast<double>(hi) - static_cast<double>(lo);
    if (!(isinf(spread) || isnan(spread) || spread + 2.0 * iters * log(static_cast<double>(n)) > 700.0)) {
        double e = exp_f64(static_cast<double>(kv) - static_cast<double>(hi));
        if (n == 4) {
            e = sinkhorn_exp<4>(e, iters, r, c);
            if (act) k[lane] = static_cast<float>(e);
            return;
        }
        if (n == 2) {
            e = sinkhorn_exp<2>(e, iters, r, c);
            if (act) k[lane] = static_cast<float>(e);
            return;
        }
        for (int it = 0; it < iters; ++it) {
            double s = 0.0;
            for (int j = 0; j < n; ++j) s = s + __shfl(e, r * n + j);
            e = e / s;
            s = 0.0;
            for (int j = 0; j < n; ++j) s = s + __shfl(e, j * n + c);
            e = e / s;
        }
        if (act) k[lane] = static_cast<float>(e);
        return;
    }
    // logSumExp (mhc.go:401-417) of the lane's row (then column), in order
    auto lse = [&](int base, int stride) {
        float m = -INFINITY;
        for (int j = 0; j < n; ++j) m = go_max(m, __shfl(kv, base + j * stride));
        if (isinf(m)) m = 0.0f;
        float s = 0.0f;
        for (int j = 0; j < n; ++j) s = s + static_cast<float>(exp_f64(static_cast<double>(__shfl(kv, base + j * stride) - m)));
        return m + static_cast<float>(log(static_cast<double>(s)));
    };
    for (int it = 0; it < iters; ++it) {
        kv = kv - lse(r * n, 1);
        kv = kv - lse(c, n);
    }
    if (act) k[lane] = static_cast<float>(exp_f64(static_cast<double>(kv)));
}

// One row per workgroup: wavefront 0 runs the Sinkhorn while wavefronts 1-3
// form the block input u, their stream values read before the heads are
// known. u is written in float4s where the lanes are whole ones.
__global__ __launch_bounds__(256) void mhc_heads_kernel(MhcArgs m) {
    __shared__ float hp[kMhcMaxLanes], kr[kMhcMaxLanes * kMhcMaxLanes];
    const int i = blockIdx.x, tid = threadIdx.x, n = m.lanes, dim = m.dim;
    const float *A = m.affine;  // {a_pre, a_post, a_res, b_pre[n], pre_off[n], b_post[n], post_off[n], b_res[n*n]}
    const long long ps = m.logit_stride ? m.logit_stride : n, rs = m.logit_stride ? m.logit_stride : n * n;
    const float *st = m.stream + static_cast<long long>(i) * n * dim;
    float *uo = m.u + static_cast<long long>(i) * dim;
    const bool vec = (dim & 3) == 0 && ((reinterpret_cast<uintptr_t>(m.stream) | reinterpret_cast<uintptr_t>(m.u)) & 15) == 0;
    const int c4 = tid - 64;  // wavefronts 1-3: the thread's first four columns
    float4 sv[kMhcMaxLanes];
    if (vec && c4 >= 0 && c4 < dim / 4) {
#pragma unroll
        for (int k = 0; k < kMhcMaxLanes; ++k)
            if (k < n) sv[k] = *reinterpret_cast<const float4 *>(st + static_cast<long long>(k) * dim + 4 * c4);
    }
    if (tid >= 64 && tid < 64 + n) {  // the pre and post heads on wavefront 1, beside the Sinkhorn's start
        const int t = tid - 64;
        float p = m.pre_logits[i * ps + t], q = m.post_logits[i * ps + t];
        if (A) {
            const float ap = A[0] * p;
            p = ap + A[3 + t] + A[3 + n + t];
            const float aq = A[1] * q;
            q = aq + A[3 + 2 * n + t] + A[3 + 3 * n + t];
        }
        const float h = gate_sigmoid(p);
        hp[t] = h;
        m.h_pre[i * n + t] = h;
        m.h_post[i * n + t] = 2.0f * gate_sigmoid(q);
    }
    if (tid < n * n) {  // n * n <= 64: wavefront 0
        float v = m.res_logits[i * rs + tid];
        if (A) {
            const float av = A[2] * v;
            v = av + A[3 + 4 * n + tid];
        }
        kr[tid] = v;
    }
    __syncthreads();
    if (tid < 64) {
        sinkhorn_wave(kr, n, 20, tid);
        if (tid < n * n) m.h_res[static_cast<long long>(i) * n * n + tid] = kr[tid];  // the lane's own entry
        return;
    }
    if (vec) {  // u = sum_k h_pre[k] stream[k], k in order
        for (int c = c4; c < dim / 4; c += 192) {
            if (c != c4) {
#pragma unroll
                for (int k = 0; k < kMhcMaxLanes; ++k)
                    if (k < n) sv[k] = *reinterpret_cast<const float4 *>(st + static_cast<long long>(k) * dim + 4 * c);
            }
            float4 u = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
#pragma unroll
            for (int k = 0; k < kMhcMaxLanes; ++k)
                if (k < n) {
                    const float h = hp[k];
                    const float px = h * sv[k].x, py = h * sv[k].y, pz = h * sv[k].z, pw = h * sv[k].w;
                    u.x = u.x + px;
                    u.y = u.y + py;
                    u.z = u.z + pz;
                    u.w = u.w + pw;
                }
            *reinterpret_cast<float4 *>(uo + 4 * c) = u;
        }
        return;
    }
    for (int c = tid - 64; c < dim; c += 192) {
        float u = 0.0f;
        for (int k = 0; k < n; ++k) {
            const float pr = hp[k] * st[static_cast<long long>(k) * dim + c];
            u = u + pr;
        }
        uo[c] = u;
    }
}

// The lane mix, a workgroup per row and `per` output lanes (ONE: one): a thread
// reads its columns of every lane once for them. The coefficients come in beside
// the stream's values, into registers for one output lane and into LDS for the
// loop over several, where reading them from memory lane by lane cost a load's
// latency each.
template <int V, bool ONE>
__global__ __launch_bounds__(256) void mhc_mix_kernel(MhcArgs m, int per) {
    __shared__ float hs[ONE ? 1 : kMhcMaxLanes * kMhcMaxLanes], qs[kMhcMaxLanes];
    const int i = blockIdx.x, n = m.lanes, dim = m.dim, tid = threadIdx.x;
    const int a0 = blockIdx.y * per, cnt = ONE ? 1 : min(per, n - a0);
    const float *st = m.stream + static_cast<long long>(i) * n * dim;
    const float *bo = m.block_out + static_cast<long long>(i) * dim, *uo = m.u + static_cast<long long>(i) * dim;
    const float *hr = m.h_res + (static_cast<long long>(i) * n + a0) * n, *hq = m.h_post + static_cast<long long>(i) * n + a0;
    float *o = m.out + (static_cast<long long>(i) * n + a0) * dim;
    float sv[kMhcMaxLanes][V], bv[V], uv[V];
    auto load = [&](float (&d)[V], const float *p) {
        if constexpr (V == 4) {
            const float4 f = *reinterpret_cast<const float4 *>(p);
            d[0] = f.x;
            d[1] = f.y;
            d[2] = f.z;
            d[3] = f.w;
        } else {
            d[0] = *p;
        }
    };
    auto columns = [&](int c) {
        load(bv, bo + c);
        load(uv, uo + c);
#pragma unroll
        for (int b = 0; b < kMhcMaxLanes; ++b)
            if (b < n) load(sv[b], st + static_cast<long long>(b) * dim + c);
    };
    int c = tid * V;
    if (c < dim) columns(c);
    float h1[kMhcMaxLanes], q1 = 0.0f;
    if constexpr (ONE) {
#pragma unroll
        for (int b = 0; b < kMhcMaxLanes; ++b) h1[b] = b < n ? hr[b] : 0.0f;
        q1 = hq[0];
    } else {
        if (tid < cnt * n) hs[tid] = hr[tid];
        if (tid < cnt) qs[tid] = hq[tid];
        __syncthreads();
    }
    while (c < dim) {
        float y[V];
#pragma unroll
        for (int q = 0; q < V; ++q) y[q] = bv[q] - uv[q];
        for (int a = 0; a < cnt; ++a) {
            float v[V];
#pragma unroll
            for (int q = 0; q < V; ++q) v[q] = 0.0f;
#pragma unroll
            for (int b = 0; b < kMhcMaxLanes; ++b)
                if (b < n) {
                    const float h = ONE ? h1[b] : hs[a * n + b];
#pragma unroll
                    for (int q = 0; q < V; ++q) {
                        const float pr = h * sv[b][q];
                        v[q] = v[q] + pr;
                    }
                }
            const float hpost = ONE ? q1 : qs[a];
#pragma unroll
            for (int q = 0; q < V; ++q) {
                const float py = hpost * y[q];
                v[q] = v[q] + py;
            }
            float *op = o + static_cast<long long>(a) * dim + c;
            if constexpr (V == 4)
                *reinterpret_cast<float4 *>(op) = make_float4(v[0], v[1], v[2], v[3]);
            else
                *op = v[0];
        }
        c += blockDim.x * V;
        if (c < dim) columns(c);
    }
}

}  // namespace

bool mhc_shape_ok(int lanes, int dim) { return lanes > 0 && lanes <= kMhcMaxLanes && dim > 0; }

hipError_t launch_rms_unit(float *dst, const float *x, int rows, int dim, hipStream_t s) {
    const long long most = grid_limit(64);
    for (long long r0 = 0; r0 < rows; r0 += most) {
        const dim3 grid(static_cast<unsigned>(std::min(most, rows - r0)));
        hipLaunchKernelGGL(rms_unit_kernel, grid, dim3(64), 0, s, dst + r0 * dim, x + r0 * dim, dim);
        if (hipError_t e = hipGetLastError()) return e;
    }
    return hipSuccess;
}

hipError_t launch_mhc_heads(const MhcArgs &m, int rows, hipStream_t s) {
    if (rows <= 0) return hipSuccess;
    hipLaunchKernelGGL(mhc_heads_kernel, dim3(static_cast<unsigned>(rows)), dim3(256), 0, s, m);
    return hipGetLastError();
}

// Output lanes a workgroup of the mix takes: one while those workgroups are few
// (a row's lanes side by side, bound by a load's latency), all of them once
// reading the stream again for each costs more, two between. Measured on MI355X
// (us, one, two and all): 4 lanes of 512 at 1, 256, 512, 1000 and 12,000 rows
// 2.5, 3.1, 3.9, 5.7, 100 against 2.7, 3.3, 3.7, 4.9, 56 and 3.2, 3.6, 4.2, 4.9,
// 37; 8 of 512 at 37, 375 and 3000 3.0, 12.0, 80 against 3.3, 5.8, 44 and 6.0,
// 7.1, 19; 4 of 64 at 512 and 3000 3.1, 6.2 against 3.2, 5.0 and 3.9, 4.7; 4 of
// 2048 at 128 and 750 4.1, 26 against 4.5, 16 and 5.8, 13. All lanes at every
// size, their coefficients read from memory, took 3.6 us for one row of 4 x 512.
int mix_lanes(int lanes, int dim, int rows) {
    const long long wgs = static_cast<long long>(rows) * lanes, values = wgs * dim;
    if (wgs <= 1024 || (wgs <= 3072 && values <= 1 << 19)) return 1;
    return lanes > 2 && values <= 3 << 19 ? 2 : lanes;
}

hipError_t launch_mhc_mix(const MhcArgs &m, int rows, hipStream_t s) {
    if (rows <= 0) return hipSuccess;
    const uintptr_t all = reinterpret_cast<uintptr_t>(m.stream) | reinterpret_cast<uintptr_t>(m.out) |
                          reinterpret_cast<uintptr_t>(m.block_out) | reinterpret_cast<uintptr_t>(m.u);
    const int v = (m.dim & 3) == 0 && (all & 15) == 0 ? 4 : 1;  // float4s where every row is whole ones
    const int items = (m.dim + v - 1) / v, threads = items >= 256 ? 256 : (items + 63) / 64 * 64;
    const int per = mix_lanes(m.lanes, m.dim, rows);
    const dim3 grid(static_cast<unsigned>(rows), static_cast<unsigned>((m.lanes + per - 1) / per)), block(threads);
    if (v == 4 && per == 1)
        hipLaunchKernelGGL((mhc_mix_kernel<4, true>), grid, block, 0, s, m, per);
    else if (v == 4)
        hipLaunchKernelGGL((mhc_mix_kernel<4, false>), grid, block, 0, s, m, per);
    else if (per == 1)
        hipLaunchKernelGGL((mhc_mix_kernel<1, true>), grid, block, 0, s, m, per);
    else
        hipLaunchKernelGGL((mhc_mix_kernel<1, false>), grid, block, 0, s, m, per);
    return hipGetLastError();
}

}  // namespace cqhip
