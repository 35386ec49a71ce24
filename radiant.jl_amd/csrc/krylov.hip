// krylov.hip -- Arnoldi step, inner products and Anderson step of the single-problem solvers (gfx950).
//
// One step orthogonalises w against the basis V_0..V_(k-1) in two passes over it:
//   dots      a_i = V_i . w, and for the modified Gram-Schmidt form l_i = V_i . V_(k-1)
//   finish    h from a (one block)
//   update    w -= sum_i h_i V_i with |w|^2
//   normalise V_k = w / |w|, and the column to the host
// Modified Gram-Schmidt takes h_i = V_i . (w - sum_(m<i) h_m V_m) = a_i - sum_(m<i) (V_i . V_m) h_m,
// so with the basis' own inner products L_im = V_i . V_m at hand the chain of k dependent
// reductions is a triangular solve, (I + L) h = a (inverse compact WY form; Swirydowicz, Langou,
// Ananthan, Yang, Thomas, "Low synchronization Gram-Schmidt and generalized minimal residual
// algorithms", 2021): the same h up to rounding, at two passes over the basis and four launches
// instead of 2 (k + 1) launches that read and write w k times.  The row l of L is new in every step,
// as V_(k-1) is.
// Bound by the reads of the basis, or by launches and latency where the vectors are short.  With the
// chain a 200-cell slab solve (3 232 values, bases of 1 to 20) took 9.0-10.6 ms, now 4.3; a 40 x 37 x 42
// box with 80 directions (5.1 M values) 15.6 ms, now 13.3 (each vector of the chain 31 us, here 8 + 7);
// errors against a 64-bit reference unchanged (7.4e-12 and 1.5e-12 of the flux, the solver's tolerance).
//
// Every reduction sums a fixed number of block partials in a fixed order, so a result depends on n
// and k only.  The host waits for the column by polling a counter in pinned memory that the last
// kernel's first block writes after the column.
#include "kernels.hpp"

#include <hip/hip_runtime.h>
#include <stdexcept>
#include <string>

namespace rt {

#define RT_HIP(x)                                                                                 \
    do {                                                                                          \
        hipError_t e_ = (x);                                                                      \
        if (e_ != hipSuccess) throw std::runtime_error(std::string("HIP error: ") + hipGetErrorString(e_) + \
                                                       " at " + __FILE__ + ":" + std::to_string(__LINE__)); \
    } while (0)

namespace {

#define RT_GLOBAL __attribute__((address_space(1)))
template <typename T> __device__ inline T gld(const T* p) { return *(const RT_GLOBAL T*)p; }
template <typename T> __device__ inline void gst(T* p, T v) { *(RT_GLOBAL T*)p = v; }

// Sum over the wave in lane 63, by DPP moves (row_shr 1, 2, 4, 8, then the row broadcasts): lanes
// without a source add zero.  Cross-lane reads through the LDS crossbar take several times as long.
template <int CTRL, int ROWS>
__device__ inline double dpp_add(double s) {
    const long long v = __double_as_longlong(s);
    const int lo = __builtin_amdgcn_update_dpp(0, (int)(v & 0xffffffff), CTRL, ROWS, 0xF, false);
    const int hi = __builtin_amdgcn_update_dpp(0, (int)(v >> 32), CTRL, ROWS, 0xF, false);
    return s + __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
}
__device__ inline double wave_sum(double s) {
    s = dpp_add<0x111, 0xF>(s);
    s = dpp_add<0x112, 0xF>(s);
    s = dpp_add<0x114, 0xF>(s);
    s = dpp_add<0x118, 0xF>(s);
    s = dpp_add<0x142, 0xA>(s);
    return dpp_add<0x143, 0xC>(s);
}
__device__ inline double lane_value(double x, int lane) {  // lane uniform
    const long long v = __double_as_longlong(x);
    const int lo = __builtin_amdgcn_readlane((int)(v & 0xffffffff), lane);
    const int hi = __builtin_amdgcn_readlane((int)(v >> 32), lane);
    return __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
}

// The results (n <= 64, by one wave) and then the counter, for a host that polls the counter.  The
// values go out as system-scope stores, past the L2, and have arrived when vmcnt is zero, so the
// counter needs no release: that would write the XCD's whole L2 back, several us in every step.
__device__ inline void to_host(double* host, const double* v, int n, unsigned long long seq) {
    const int lane = threadIdx.x & 63;
    if (lane < n) __hip_atomic_store(host + lane, v[lane], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    if (lane == 0)
        __hip_atomic_store((unsigned long long*)(host + KRY_FLAG), seq, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

// Partial sums of block b: part[b * NV + v].  UE elements per thread and batch, the next batch's
// loads issued before a batch is worked; padding lanes read a clamped element and are masked.
template <int KM, bool MGS>
__global__ __launch_bounds__(256) void arn_dots_kernel(const BasisTab V, const double* __restrict__ w, long n, int k,
                                                       double* __restrict__ part) {
    constexpr int UE = KM <= 4 ? 4 : (KM <= 8 ? 2 : 1);
    constexpr int NV = MGS ? 2 * KM : KM;
    const int tid = threadIdx.x, nb = gridDim.x;
    const long chunk = (n + nb - 1) / nb, lo = (long)blockIdx.x * chunk, hi = lo + chunk < n ? lo + chunk : n;
    const double* __restrict__ Vp[KM];
#pragma unroll
    for (int i = 0; i < KM; ++i) Vp[i] = V.p[i < k ? i : 0];
    const double* __restrict__ vl = V.p[k - 1];
    double a[KM], l[MGS ? KM : 1];
#pragma unroll
    for (int i = 0; i < KM; ++i) a[i] = 0.0;
#pragma unroll
    for (int i = 0; i < (MGS ? KM : 1); ++i) l[i] = 0.0;
    struct Batch { double v[UE][KM], x[UE], y[UE]; };
    auto load = [&](long e0, Batch& B) {
#pragma unroll
        for (int u = 0; u < UE; ++u) {
            const long e = e0 + u * 256 + tid, ec = e < hi ? e : hi - 1;
#pragma unroll
            for (int i = 0; i < KM; ++i) B.v[u][i] = gld(Vp[i] + ec);
            B.x[u] = gld(w + ec);
            if constexpr (MGS) B.y[u] = gld(vl + ec);
        }
    };
    auto work = [&](long e0, const Batch& B) {
#pragma unroll
        for (int u = 0; u < UE; ++u) {
            const double m = e0 + u * 256 + tid < hi ? 1.0 : 0.0;
            const double x = m != 0.0 ? B.x[u] : 0.0;
#pragma unroll
            for (int i = 0; i < KM; ++i) a[i] = fma(B.v[u][i], x, a[i]);
            if constexpr (MGS) {
                const double y = m != 0.0 ? B.y[u] : 0.0;
#pragma unroll
                for (int i = 0; i < KM; ++i) l[i] = fma(B.v[u][i], y, l[i]);
            }
        }
    };
    if (lo < hi) {
        Batch A, B;
        load(lo, A);
        for (long e = lo; e < hi; e += 512 * UE) {
            load(e + 256 * UE, B);
            __builtin_amdgcn_sched_barrier(0);
            work(e, A);
            __builtin_amdgcn_sched_barrier(0);
            load(e + 512 * UE, A);
            __builtin_amdgcn_sched_barrier(0);
            work(e + 256 * UE, B);
        }
    }
    __shared__ double red[4][NV];
    const int lane = tid & 63, wv = tid >> 6;
#pragma unroll
    for (int i = 0; i < KM; ++i) {
        if (i < k) {  // uniform
            const double s = wave_sum(a[i]);
            if (lane == 63) red[wv][i] = s;
            if constexpr (MGS) {
                const double t = wave_sum(l[i]);
                if (lane == 63) red[wv][KM + i] = t;
            }
        }
    }
    __syncthreads();
    double* p = part + (size_t)blockIdx.x * NV;
    for (int i = tid; i < NV; i += 256) {
        const int v = i < KM ? i : i - KM;
        if (v < k) p[i] = ((red[0][i] + red[1][i]) + red[2][i]) + red[3][i];
    }
}

// The triangular solve (I + L) h = a by wave 0, column by column: lane i holds a_i; Ls: the strictly
// lower rows of L in LDS.  Afterwards s_h[0..k-1] = h for the whole block.
__device__ inline void tri_solve(const double* a, const double* Ls, double* s_h, int k) {
    if (threadIdx.x < 64) {
        const int i = threadIdx.x;
        double x = i < k ? a[i] : 0.0;
        for (int m = 0; m + 1 < k; ++m) {
            const double hm = lane_value(x, m);
            if (i > m && i < k) x = fma(-Ls[i * GS_KMAX + m], hm, x);
        }
        if (i < k) s_h[i] = x;
    }
    __syncthreads();
}

template <int KM, bool MGS>
__global__ __launch_bounds__(1024) void arn_finish_kernel(const double* __restrict__ part, int nb, int k,
                                                          double* __restrict__ L, double* __restrict__ h) {
    constexpr int NV = MGS ? 2 * KM : KM;
    __shared__ double s_v[2 * GS_KMAX], s_L[MGS ? GS_KMAX * GS_KMAX : 1], s_h[GS_KMAX];
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    for (int v = wv; v < (MGS ? 2 * k : k); v += 16) {
        const int col = v < k ? v : KM + (v - k);
        double s = 0.0;
        for (int b = lane; b < nb; b += 64) s += part[(size_t)b * NV + col];
        s = wave_sum(s);
        if (lane == 63) s_v[v] = s;
    }
    if constexpr (MGS) {  // the rows of earlier steps
        for (int i = threadIdx.x; i < (k - 1) * GS_KMAX; i += 1024) s_L[i] = L[i];
    }
    __syncthreads();
    if constexpr (MGS) {
        if ((int)threadIdx.x < k - 1) s_L[(k - 1) * GS_KMAX + threadIdx.x] = L[(k - 1) * GS_KMAX + threadIdx.x] = s_v[k + threadIdx.x];
        __syncthreads();
        tri_solve(s_v, s_L, s_h, k);
        if ((int)threadIdx.x < k) h[threadIdx.x] = s_h[threadIdx.x];
    } else if ((int)threadIdx.x < k) {
        h[threadIdx.x] = s_v[threadIdx.x];
    }
}

template <int KM>
__global__ __launch_bounds__(256) void arn_update_kernel(const BasisTab V, double* __restrict__ w, long n, int k,
                                                         const double* __restrict__ h, double* __restrict__ part) {
    constexpr int UE = KM <= 4 ? 4 : (KM <= 8 ? 2 : 1);
    const int tid = threadIdx.x, nb = gridDim.x;
    const long chunk = (n + nb - 1) / nb, lo = (long)blockIdx.x * chunk, hi = lo + chunk < n ? lo + chunk : n;
    const double* __restrict__ Vp[KM];
    double c[KM];
#pragma unroll
    for (int i = 0; i < KM; ++i) {
        Vp[i] = V.p[i < k ? i : 0];
        c[i] = i < k ? h[i] : 0.0;
    }
    double acc = 0.0;
    struct Batch { double v[UE][KM], x[UE]; };
    auto load = [&](long e0, Batch& B) {
#pragma unroll
        for (int u = 0; u < UE; ++u) {
            const long e = e0 + u * 256 + tid, ec = e < hi ? e : hi - 1;
#pragma unroll
            for (int i = 0; i < KM; ++i) B.v[u][i] = gld(Vp[i] + ec);
            B.x[u] = gld(w + ec);
        }
    };
    auto work = [&](long e0, const Batch& B) {
#pragma unroll
        for (int u = 0; u < UE; ++u) {
            const long e = e0 + u * 256 + tid;
            double x = B.x[u];
#pragma unroll
            for (int i = 0; i < KM; ++i) x = fma(-c[i], B.v[u][i], x);
            if (e < hi) {
                gst(w + e, x);
                acc = fma(x, x, acc);
            }
        }
    };
    // a clamped lane may read an element that its owner has already written: it discards it
    if (lo < hi) {
        Batch A, B;
        load(lo, A);
        for (long e = lo; e < hi; e += 512 * UE) {
            load(e + 256 * UE, B);
            __builtin_amdgcn_sched_barrier(0);
            work(e, A);
            __builtin_amdgcn_sched_barrier(0);
            load(e + 512 * UE, A);
            __builtin_amdgcn_sched_barrier(0);
            work(e + 256 * UE, B);
        }
    }
    __shared__ double red[4];
    const double s = wave_sum(acc);
    if ((tid & 63) == 63) red[tid >> 6] = s;
    __syncthreads();
    if (tid == 0) part[blockIdx.x] = ((red[0] + red[1]) + red[2]) + red[3];
}

// Every block sums the nb partials of |w|^2 itself, in the same order.
__global__ __launch_bounds__(256) void arn_normalise_kernel(const double* __restrict__ w, double* __restrict__ vnext, long n,
                                                            const double* __restrict__ part, int nb,
                                                            const double* __restrict__ h, int k, double* host,
                                                            unsigned long long seq) {
    __shared__ double red[4], out[GS_KMAX + 1];
    const int tid = threadIdx.x;
    double s = 0.0;
    for (int b = tid; b < nb; b += 256) s += part[b];
    s = wave_sum(s);
    if ((tid & 63) == 63) red[tid >> 6] = s;
    __syncthreads();
    const double nn = ((red[0] + red[1]) + red[2]) + red[3];
    if (blockIdx.x == 0) {
        if (tid < k) out[tid] = h[tid];
        if (tid == k) out[k] = nn;
        __syncthreads();
        if (tid < 64) to_host(host, out, k + 1, seq);
    }
    if (!(nn > 0.0)) return;
    const double a = 1.0 / sqrt(nn);
    for (long i = blockIdx.x * 256L + tid; i < n; i += gridDim.x * 256L) gst(vnext + i, gld(w + i) * a);
}

// The whole step in one workgroup for short vectors (at most 1024 * ARN_SMALL_E values, ARN_SMALL_READS
// of the basis): w stays in registers and the basis, a few hundred kB, is read from the L2.
constexpr int ARN_SMALL_E = 8;
template <bool MGS>
__global__ __launch_bounds__(1024) void arn_small_kernel(const BasisTab V, double* __restrict__ w, double* __restrict__ vnext,
                                                         int n, int k, double* __restrict__ L, double* host,
                                                         unsigned long long seq) {
    constexpr int E = ARN_SMALL_E, U = 4;
    __shared__ double s_red[16][2 * GS_KMAX], s_v[2 * GS_KMAX], s_L[MGS ? GS_KMAX * GS_KMAX : 1], s_h[GS_KMAX + 1];
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
    double x[E], y[MGS ? E : 1];
#pragma unroll
    for (int e = 0; e < E; ++e) {
        const int i = tid + 1024 * e;
        x[e] = i < n ? gld(w + i) : 0.0;
        if constexpr (MGS) y[e] = i < n ? gld(V.p[k - 1] + i) : 0.0;
    }
    if constexpr (MGS)
        for (int i = tid; i < (k - 1) * GS_KMAX; i += 1024) s_L[i] = L[i];
    for (int i0 = 0; i0 < k; i0 += U) {
        double v[U][E];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const double* p = V.p[i0 + u < k ? i0 + u : k - 1];
#pragma unroll
            for (int e = 0; e < E; ++e) v[u][e] = tid + 1024 * e < n ? gld(p + tid + 1024 * e) : 0.0;
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            if (i0 + u < k) {  // uniform
            double a = 0.0, l = 0.0;
#pragma unroll
            for (int e = 0; e < E; ++e) {
                a = fma(v[u][e], x[e], a);
                if constexpr (MGS) l = fma(v[u][e], y[e], l);
            }
            a = wave_sum(a);
            if (lane == 63) s_red[wv][i0 + u] = a;
            if constexpr (MGS) {
                l = wave_sum(l);
                if (lane == 63) s_red[wv][GS_KMAX + i0 + u] = l;
            }
            }
        }
    }
    __syncthreads();
    if (tid < 2 * GS_KMAX) {
        double s = 0.0;
        const int v = tid < GS_KMAX ? tid : tid - GS_KMAX;
        if (v < k && (MGS || tid < GS_KMAX))
            for (int j = 0; j < 16; ++j) s += s_red[j][tid];
        s_v[tid] = s;
    }
    __syncthreads();
    if constexpr (MGS) {
        if (tid < k - 1) s_L[(k - 1) * GS_KMAX + tid] = L[(k - 1) * GS_KMAX + tid] = s_v[GS_KMAX + tid];
        __syncthreads();
        tri_solve(s_v, s_L, s_h, k);
    } else {
        if (tid < k) s_h[tid] = s_v[tid];
        __syncthreads();
    }
    for (int i0 = 0; i0 < k; i0 += U) {
        double v[U][E], c[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int i = i0 + u < k ? i0 + u : k - 1;
            c[u] = i0 + u < k ? s_h[i] : 0.0;
#pragma unroll
            for (int e = 0; e < E; ++e) v[u][e] = tid + 1024 * e < n ? gld(V.p[i] + tid + 1024 * e) : 0.0;
        }
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
            for (int e = 0; e < E; ++e) x[e] = fma(-c[u], v[u][e], x[e]);
    }
    double s = 0.0;
#pragma unroll
    for (int e = 0; e < E; ++e) s = fma(x[e], x[e], s);
    s = wave_sum(s);
    if (lane == 63) s_red[wv][0] = s;
    __syncthreads();
    double nn = 0.0;
    for (int j = 0; j < 16; ++j) nn += s_red[j][0];
    const double a = nn > 0.0 ? 1.0 / sqrt(nn) : 0.0;
#pragma unroll
    for (int e = 0; e < E; ++e) {
        const int i = tid + 1024 * e;
        if (i < n) {
            gst(w + i, x[e]);
            if (nn > 0.0) gst(vnext + i, x[e] * a);
        }
    }
    if (tid == 0) s_h[k] = nn;
    __syncthreads();
    if (tid < 64) to_host(host, s_h, k + 1, seq);
}

template <int KM>
void arnoldi_km(const BasisTab& V, double* w, double* vnext, long n, int k, bool mgs, const ArnoldiWork& aw, int nb,
                unsigned long long seq, hipStream_t st) {
    double* p2 = aw.part + (size_t)ARN_BLOCKS * 2 * GS_KMAX;  // partials of |w|^2
    if (mgs) {
        hipLaunchKernelGGL((arn_dots_kernel<KM, true>), dim3(nb), dim3(256), 0, st, V, w, n, k, aw.part);
        hipLaunchKernelGGL((arn_finish_kernel<KM, true>), dim3(1), dim3(1024), 0, st, aw.part, nb, k, aw.L, aw.h);
    } else {
        hipLaunchKernelGGL((arn_dots_kernel<KM, false>), dim3(nb), dim3(256), 0, st, V, w, n, k, aw.part);
        hipLaunchKernelGGL((arn_finish_kernel<KM, false>), dim3(1), dim3(1024), 0, st, aw.part, nb, k, aw.L, aw.h);
    }
    hipLaunchKernelGGL((arn_update_kernel<KM>), dim3(nb), dim3(256), 0, st, V, w, n, k, aw.h, p2);
    const long g = (n + 1023) / 1024;
    hipLaunchKernelGGL(arn_normalise_kernel, dim3((unsigned)(g < 1 ? 1 : (g > 2048 ? 2048 : g))), dim3(256), 0, st, w, vnext, n,
                       p2, nb, aw.h, k, aw.host, seq);
}

// ------------------------------------------------------------------------------------------
// Inner products a_i . b_i of up to DOT_MAX pairs in one pass, and the Anderson step.
// ------------------------------------------------------------------------------------------
template <int NV>
__device__ inline void block_partials(double (&v)[NV], int nv, double* __restrict__ part) {
    __shared__ double red[4][NV];
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
#pragma unroll
    for (int i = 0; i < NV; ++i)
        if (i < nv) {  // uniform
            const double s = wave_sum(v[i]);
            if (lane == 63) red[wv][i] = s;
        }
    __syncthreads();
    if ((int)threadIdx.x < nv)
        part[(size_t)blockIdx.x * NV + threadIdx.x] =
            ((red[0][threadIdx.x] + red[1][threadIdx.x]) + red[2][threadIdx.x]) + red[3][threadIdx.x];
}

__global__ __launch_bounds__(256) void dots_kernel(const DotTab t, long n, double* __restrict__ part) {
    double acc[DOT_MAX] = {};
    for (long i = blockIdx.x * 256L + threadIdx.x; i < n; i += gridDim.x * 256L)
#pragma unroll
        for (int j = 0; j < DOT_MAX; ++j)
            if (j < t.n) acc[j] = fma(gld(t.a[j] + i), gld(t.b[j] + i), acc[j]);
    block_partials<DOT_MAX>(acc, t.n, part);
}

// one block: the sums of nv values over nb partials, to the host
template <int NV>
__global__ __launch_bounds__(1024) void sums_to_host_kernel(const double* __restrict__ part, int nb, int nv, double* host,
                                                            unsigned long long seq) {
    __shared__ double out[64];
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    for (int v = wv; v < nv; v += 16) {
        double s = 0.0;
        for (int b = lane; b < nb; b += 64) s += part[(size_t)b * NV + v];
        s = wave_sum(s);
        if (lane == 63) out[v] = s;
    }
    __syncthreads();
    if (threadIdx.x < 64) to_host(host, out, nv, seq);
}

// One pass over the state for one Anderson iteration (anderson.jl:60-99): f = g - z, the new
// differences dF = f - f_old and dG = g - g_old (not in the first iteration), and every inner
// product the host needs: f.f, z.z, g.g, then dF_i . f and dF_new . dF_i of the history, the new
// difference last.
constexpr int AND_NV = 3 + 2 * AND_DEPTH;
__global__ __launch_bounds__(256) void anderson_kernel(const AndersonTab t, long n, double* __restrict__ part) {
    double acc[AND_NV] = {};
    for (long i = blockIdx.x * 256L + threadIdx.x; i < n; i += gridDim.x * 256L) {
        const double g = gld(t.g + i), z = gld(t.z + i), f = g - z;
        gst(t.f + i, f);
        acc[0] = fma(f, f, acc[0]);
        acc[1] = fma(z, z, acc[1]);
        acc[2] = fma(g, g, acc[2]);
        if (t.mk > 0) {  // uniform
            const double dn = f - gld(t.fo + i);
            gst(t.dF[t.mk - 1] + i, dn);
            gst(t.dG[t.mk - 1] + i, g - gld(t.go + i));
#pragma unroll
            for (int j = 0; j < AND_DEPTH; ++j)
                if (j < t.mk) {
                    const double d = j == t.mk - 1 ? dn : gld(t.dF[j] + i);
                    acc[3 + j] = fma(d, f, acc[3 + j]);
                    acc[3 + AND_DEPTH + j] = fma(dn, d, acc[3 + AND_DEPTH + j]);
                }
        }
    }
    block_partials<AND_NV>(acc, AND_NV, part);
}

// z <- z + f - sum_i gamma_i dG_i
__global__ __launch_bounds__(256) void anderson_update_kernel(const AndersonTab t, long n) {
    for (long i = blockIdx.x * 256L + threadIdx.x; i < n; i += gridDim.x * 256L) {
        double z = gld(t.z + i) + gld(t.f + i);
#pragma unroll
        for (int j = 0; j < AND_DEPTH; ++j)
            if (j < t.mk) z = fma(-t.gamma[j], gld(t.dG[j] + i), z);
        gst(t.z + i, z);
    }
}

// r = c - t with |r|^2
__global__ __launch_bounds__(256) void residual_kernel(double* __restrict__ r, const double* __restrict__ c,
                                                       const double* __restrict__ t, long n, double* __restrict__ part) {
    double acc[1] = {0.0};
    for (long i = blockIdx.x * 256L + threadIdx.x; i < n; i += gridDim.x * 256L) {
        const double x = gld(c + i) - gld(t + i);
        gst(r + i, x);
        acc[0] = fma(x, x, acc[0]);
    }
    block_partials<1>(acc, 1, part);
}

__global__ __launch_bounds__(256) void scale_copy_kernel(double* __restrict__ d, const double* __restrict__ s, double a, long n) {
    for (long i = blockIdx.x * 256L + threadIdx.x; i < n; i += gridDim.x * 256L) gst(d + i, gld(s + i) * a);
}

// z = (ADD ? z : 0) + sum_i y_i V_i
template <bool ADD>
__global__ __launch_bounds__(256) void combine_kernel(double* __restrict__ z, const BasisTab V, const Vals32 y, int k, long n) {
    for (long i = blockIdx.x * 256L + threadIdx.x; i < n; i += gridDim.x * 256L) {
        double x = ADD ? gld(z + i) : 0.0;
#pragma unroll 8
        for (int t = 0; t < k; ++t) x = fma(y.v[t], gld(V.p[t] + i), x);
        gst(z + i, x);
    }
}

int red_blocks(long n) {
    const long b = (n + 1023) / 1024;
    return (int)(b < 1 ? 1 : (b > ARN_BLOCKS ? ARN_BLOCKS : b));
}

}  // namespace

void launch_dots(const DotTab& t, long n, const ArnoldiWork& aw, unsigned long long seq, hipStream_t st) {
    if (t.n < 1 || t.n > DOT_MAX) throw std::runtime_error("launch_dots: pairs out of range");
    const int nb = red_blocks(n);
    hipLaunchKernelGGL(dots_kernel, dim3(nb), dim3(256), 0, st, t, n, aw.part);
    hipLaunchKernelGGL((sums_to_host_kernel<DOT_MAX>), dim3(1), dim3(1024), 0, st, aw.part, nb, t.n, aw.host, seq);
    RT_HIP(hipGetLastError());
}

void launch_residual(double* r, const double* c, const double* t, long n, const ArnoldiWork& aw, unsigned long long seq,
                     hipStream_t st) {
    const int nb = red_blocks(n);
    hipLaunchKernelGGL(residual_kernel, dim3(nb), dim3(256), 0, st, r, c, t, n, aw.part);
    hipLaunchKernelGGL((sums_to_host_kernel<1>), dim3(1), dim3(1024), 0, st, aw.part, nb, 1, aw.host, seq);
    RT_HIP(hipGetLastError());
}

void launch_scale_copy(double* d, const double* s, double a, long n, hipStream_t st) {
    hipLaunchKernelGGL(scale_copy_kernel, dim3(2 * red_blocks(n)), dim3(256), 0, st, d, s, a, n);
    RT_HIP(hipGetLastError());
}

void launch_combine(double* z, const BasisTab& V, const Vals32& y, int k, bool add, long n, hipStream_t st) {
    if (k < 0 || k > 32) throw std::runtime_error("launch_combine: vectors out of range");
    if (add) hipLaunchKernelGGL(combine_kernel<true>, dim3(2 * red_blocks(n)), dim3(256), 0, st, z, V, y, k, n);
    else hipLaunchKernelGGL(combine_kernel<false>, dim3(2 * red_blocks(n)), dim3(256), 0, st, z, V, y, k, n);
    RT_HIP(hipGetLastError());
}

void launch_anderson(const AndersonTab& t, long n, const ArnoldiWork& aw, unsigned long long seq, hipStream_t st) {
    if (t.mk < 0 || t.mk > AND_DEPTH) throw std::runtime_error("launch_anderson: depth out of range");
    const int nb = red_blocks(n);
    hipLaunchKernelGGL(anderson_kernel, dim3(nb), dim3(256), 0, st, t, n, aw.part);
    hipLaunchKernelGGL((sums_to_host_kernel<AND_NV>), dim3(1), dim3(1024), 0, st, aw.part, nb, AND_NV, aw.host, seq);
    RT_HIP(hipGetLastError());
}

void launch_anderson_update(const AndersonTab& t, long n, hipStream_t st) {
    hipLaunchKernelGGL(anderson_update_kernel, dim3(red_blocks(n)), dim3(256), 0, st, t, n);
    RT_HIP(hipGetLastError());
}

void launch_arnoldi(const BasisTab& V, double* w, double* vnext, long n, int k, bool mgs, const ArnoldiWork& aw,
                    unsigned long long seq, hipStream_t st) {
    if (k < 1 || k > GS_KMAX || n < 1) throw std::runtime_error("launch_arnoldi: basis size out of range");
    // One workgroup while its own reads of the basis stay under the cost of three more launches
    // (13 us at k = 5 and 17 us at the bound, against 24 us for the four at k = 9 to 16).
    if (n <= 1024 * ARN_SMALL_E && n * k <= ARN_SMALL_READS) {
        if (mgs) hipLaunchKernelGGL(arn_small_kernel<true>, dim3(1), dim3(1024), 0, st, V, w, vnext, (int)n, k, aw.L, aw.host, seq);
        else hipLaunchKernelGGL(arn_small_kernel<false>, dim3(1), dim3(1024), 0, st, V, w, vnext, (int)n, k, aw.L, aw.host, seq);
    } else {
        // a block works 2048 elements or more; few vectors need more blocks to keep loads in flight
        const int top = k <= 4 ? ARN_BLOCKS : (k <= 8 ? ARN_BLOCKS / 2 : ARN_BLOCKS / 4);
        const long b = (n + 2047) / 2048;
        const int nb = (int)(b < top ? b : top);
        if (k <= 2) arnoldi_km<2>(V, w, vnext, n, k, mgs, aw, nb, seq, st);
        else if (k <= 4) arnoldi_km<4>(V, w, vnext, n, k, mgs, aw, nb, seq, st);
        else if (k <= 8) arnoldi_km<8>(V, w, vnext, n, k, mgs, aw, nb, seq, st);
        else if (k <= 16) arnoldi_km<16>(V, w, vnext, n, k, mgs, aw, nb, seq, st);
        else arnoldi_km<GS_KMAX>(V, w, vnext, n, k, mgs, aw, nb, seq, st);
    }
    RT_HIP(hipGetLastError());
}

}  // namespace rt
