// sweep_ho2_pipe.hip -- 2D sweeps of closures with up to 4 moments per cell, pipelined over the
// waves of a workgroup (gfx950).
//
// The same cell system, faces and walk as sweep_2d_ho_kernel (kernels.hip): one workgroup per
// direction, anti-diagonals in sweep order, x-face moments of every row and y-face moments of every
// column in LDS.  There one wave does all of a diagonal's work between two barriers: the loads of
// its cells, their elimination, the faces.  Only the faces depend on the diagonal before.  Here each
// group of waves takes every G-th diagonal and solves its cells ahead of time, for the source and
// for each incoming face moment, so that what is left once the previous diagonal's faces are known is
// psi = x_0 + X f and the outgoing faces: a few fused multiply-adds between two LDS accesses.  The
// diagonals are handed on through a counter in LDS (a wave adds one after its face writes, which the
// LDS performs in order; the next diagonal's waves poll it), as a barrier in every diagonal would
// make each group wait for the others' elimination.
// Bound by the chain of diagonals (LDS read, the multiply-adds, LDS write, counter).  36 x 31 cells of 4
// moments in 128 directions, 66 diagonals: 86 us with the barrier walk, 28 us here; a reflected DG solve
// on them 8.6 -> 5.5 ms.
#include "kernels.hpp"

#include <hip/hip_runtime.h>
#include <hip/hip_ext.h>
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

constexpr int PIPE_WAVES = 8;

template <int KX, int KY, bool FC>
__device__ __forceinline__ constexpr int idx2(int ix, int iy) {
    return FC ? KX * iy + ix : (iy > 0 ? KX - 1 + iy : ix);
}

// wpd: waves per diagonal (a power of two, 64 wpd >= min(Nx, Ny))
template <typename T, int KX, int KY, bool FC>
__global__ __launch_bounds__(64 * PIPE_WAVES) void sweep_2d_ho_pipe_kernel(const PassDesc* __restrict__ pds, int wpd) {
    constexpr int NM = FC ? KX * KY : KX + KY - 1, NF = KY + KX, NR = 1 + NF;
    extern __shared__ __align__(16) unsigned char smem[];
    __shared__ int s_done;  // waves that have finished their part of a diagonal, over all diagonals
    const PassDesc& d = pds[0];
    const int n = blockIdx.x, tid = threadIdx.x, nt = blockDim.x;
    const int Nx = d.Nx, Ny = d.Ny;
    T* FX = (T*)smem;                  // [Ny][KY]
    T* FY = FX + (size_t)Ny * KY;      // [Nx][KX]
    const double mu = d.mu[n], eta = d.eta[n];
    const bool fxs = mu >= 0, fys = eta >= 0;
    const T sx = mu > 0 ? T(1) : (mu < 0 ? T(-1) : T(0)), sy = eta > 0 ? T(1) : (eta < 0 ? T(-1) : T(0));
    T wx[KX + 1], wy[KY + 1], Cx[KX], Cy[KY], px[KX], nx[KX], py[KY], ny[KY];
#pragma unroll
    for (int k = 0; k <= KX; ++k) wx[k] = (T)d.ho_om[k];
#pragma unroll
    for (int k = 0; k <= KY; ++k) wy[k] = (T)d.ho_omy[k];
#pragma unroll
    for (int k = 0; k < KX; ++k) {
        Cx[k] = (T)sqrt(2.0 * k + 1.0);
        px[k] = k == 0 ? T(1) : px[k - 1] * sx;
        nx[k] = k == 0 ? T(1) : -nx[k - 1] * sx;
    }
#pragma unroll
    for (int k = 0; k < KY; ++k) {
        Cy[k] = (T)sqrt(2.0 * k + 1.0);
        py[k] = k == 0 ? T(1) : py[k - 1] * sy;
        ny[k] = k == 0 ? T(1) : -ny[k - 1] * sy;
    }
    T* __restrict__ psi = (T*)d.psi + (size_t)n * d.Nc;
    for (int i = tid; i < Ny * KY; i += nt) FX[i] = d.bin_x ? (T)d.bin_x[(size_t)n * Ny * KY + i] : T(0);
    for (int i = tid; i < Nx * KX; i += nt) FY[i] = d.bin_y ? (T)d.bin_y[(size_t)n * Nx * KX + i] : T(0);
    if (tid == 0) s_done = 0;
    __syncthreads();
    const int ng = PIPE_WAVES / wpd;                     // groups of waves
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), grp = wave / wpd;
    const int li = tid - grp * 64 * wpd;                 // cell of the diagonal
    const int ndiag = Nx + Ny - 1;
    for (int dg = grp; dg < ndiag; dg += ng) {
        const int k0 = dg - (Ny - 1) > 0 ? dg - (Ny - 1) : 0, k1 = dg < Nx - 1 ? dg : Nx - 1;
        const int kx = k0 + li, ky = dg - kx;
        const bool in = kx <= k1;
        const int ix = in ? (fxs ? kx : Nx - 1 - kx) : 0, iy = in ? (fys ? ky : Ny - 1 - ky) : 0;
        const size_t c = (size_t)ix + (size_t)Nx * iy;
        // ---- the cell's moments for its source (column 0) and per unit of each face moment
        T q[NM][NR];
        {
            const T hx = (T)(fabs(mu) / d.dx[ix]), hy = (T)(fabs(eta) / d.dy[iy]);
            const T St = (T)d.sigt[d.mat[c * NM]];
            T S[NM][NM];
#pragma unroll
            for (int i = 0; i < NM; ++i)
#pragma unroll
                for (int j = 0; j < NM; ++j) S[i][j] = i == j ? St : T(0);
#pragma unroll
            for (int ax = 0; ax < KX; ++ax)
#pragma unroll
                for (int ay = 0; ay < KY; ++ay) {
                    if (!FC && ax > 0 && ay > 0) continue;
                    const int i = idx2<KX, KY, FC>(ax, ay);
#pragma unroll
                    for (int bx = 0; bx < KX; ++bx)
#pragma unroll
                        for (int by = 0; by < KY; ++by) {
                            if (!FC && bx > 0 && by > 0) continue;
                            const int j = idx2<KX, KY, FC>(bx, by);
                            if (ay == by) {
                                if (ax > bx && ((ax - bx) & 1)) S[i][j] -= T(2) * Cx[ax] * hx * sx * Cx[bx];
                                S[i][j] += Cx[ax] * hx * px[ax] * Cx[bx] * px[bx] * wx[bx + 1];
                            }
                            if (ax == bx) {
                                if (ay > by && ((ay - by) & 1)) S[i][j] -= T(2) * Cy[ay] * hy * sy * Cy[by];
                                S[i][j] += Cy[ay] * hy * py[ay] * Cy[by] * py[by] * wy[by + 1];
                            }
                        }
                    q[i][0] = psi[(size_t)i + NM * c];
#pragma unroll
                    for (int k = 0; k < KY; ++k) q[i][1 + k] = k == ay ? -(Cx[ax] * hx * (px[ax] * wx[0] - nx[ax])) : T(0);
#pragma unroll
                    for (int k = 0; k < KX; ++k) q[i][1 + KY + k] = k == ax ? -(Cy[ay] * hy * (py[ay] * wy[0] - ny[ay])) : T(0);
                }
            // Gaussian elimination with partial pivoting (row swaps as selects)
#pragma unroll
            for (int p = 0; p < NM; ++p) {
#pragma unroll
                for (int i = p + 1; i < NM; ++i) {
                    const bool sw = fabs(S[i][p]) > fabs(S[p][p]);
#pragma unroll
                    for (int j = p; j < NM; ++j) {
                        const T t = S[p][j];
                        S[p][j] = sw ? S[i][j] : t;
                        S[i][j] = sw ? t : S[i][j];
                    }
#pragma unroll
                    for (int r = 0; r < NR; ++r) {
                        const T t = q[p][r];
                        q[p][r] = sw ? q[i][r] : t;
                        q[i][r] = sw ? t : q[i][r];
                    }
                }
#pragma unroll
                for (int i = p + 1; i < NM; ++i) {
                    const T f = S[i][p] / S[p][p];
#pragma unroll
                    for (int j = p + 1; j < NM; ++j) S[i][j] -= f * S[p][j];
#pragma unroll
                    for (int r = 0; r < NR; ++r) q[i][r] -= f * q[p][r];
                }
            }
#pragma unroll
            for (int i = NM - 1; i >= 0; --i) {
                const T inv = T(1) / S[i][i];
#pragma unroll
                for (int r = 0; r < NR; ++r) {
                    T v = q[i][r];
#pragma unroll
                    for (int j = i + 1; j < NM; ++j) v -= S[i][j] * q[j][r];
                    q[i][r] = v * inv;
                }
            }
        }
        // pinned here: the compiler would otherwise sink the elimination to its use, behind the wait
#pragma unroll
        for (int i = 0; i < NM; ++i)
#pragma unroll
            for (int r = 0; r < NR; ++r) asm volatile("" : "+v"(q[i][r]));
        // ---- wait for the diagonal before: every wave of it has added one
        while (__hip_atomic_load(&s_done, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP) < dg * wpd) {}
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
        T* fx = FX + (size_t)iy * KY;
        T* fy = FY + (size_t)ix * KX;
        T x[NM];
        if (in) {
            T f[NF], o[NF];
#pragma unroll
            for (int k = 0; k < KY; ++k) f[k] = fx[k];
#pragma unroll
            for (int k = 0; k < KX; ++k) f[KY + k] = fy[k];
#pragma unroll
            for (int i = 0; i < NM; ++i) {
                x[i] = q[i][0];
#pragma unroll
                for (int k = 0; k < NF; ++k) x[i] += q[i][1 + k] * f[k];
            }
#pragma unroll
            for (int k = 0; k < KY; ++k) o[k] = wx[0] * f[k];
#pragma unroll
            for (int k = 0; k < KX; ++k) o[KY + k] = wy[0] * f[KY + k];
#pragma unroll
            for (int ax = 0; ax < KX; ++ax)
#pragma unroll
                for (int ay = 0; ay < KY; ++ay) {
                    if (!FC && ax > 0 && ay > 0) continue;
                    const T v = x[idx2<KX, KY, FC>(ax, ay)];
                    o[ay] += Cx[ax] * px[ax] * wx[ax + 1] * v;
                    o[KY + ax] += Cy[ay] * py[ay] * wy[ay + 1] * v;
                }
#pragma unroll
            for (int k = 0; k < KY; ++k) fx[k] = o[k];
#pragma unroll
            for (int k = 0; k < KX; ++k) fy[k] = o[KY + k];
        }
        // ---- hand on
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
        if ((tid & 63) == 0) __hip_atomic_fetch_add(&s_done, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        if (in)
#pragma unroll
            for (int i = 0; i < NM; ++i) psi[(size_t)i + NM * c] = x[i];
    }
    __syncthreads();
    if (d.bx)
        for (int i = tid; i < Ny * KY; i += nt) ((T*)d.bx)[(size_t)n * Ny * KY + i] = FX[i];
    if (d.by)
        for (int i = tid; i < Nx * KX; i += nt) ((T*)d.by)[(size_t)n * Nx * KX + i] = FY[i];
}

template <typename T, int KX, int KY, bool FC>
void pipe_launch(const PassDesc* d_pd, int Nd, int wpd, size_t lds, hipStream_t st) {
    auto fn = sweep_2d_ho_pipe_kernel<T, KX, KY, FC>;
    static const bool attr = [&] {
        RT_HIP(hipFuncSetAttribute((const void*)fn, hipFuncAttributeMaxDynamicSharedMemorySize, PIPE_LDS_MAX));
        return true;
    }();
    (void)attr;
    hipEvent_t a, b;
    take_launch_events(&a, &b);
    if (a) hipExtLaunchKernelGGL(fn, dim3(Nd), dim3(64 * PIPE_WAVES), (uint32_t)lds, st, a, b, 0u, d_pd, wpd);
    else hipLaunchKernelGGL(fn, dim3(Nd), dim3(64 * PIPE_WAVES), (uint32_t)lds, st, d_pd, wpd);
}

template <typename T>
void pipe_dispatch(const PassDesc* d_pd, int Nd, int kx, int ky, bool fc, int wpd, size_t lds, hipStream_t st) {
    if (kx == 1 || ky == 1) fc = true;  // the couplings are the same
    switch (100 * kx + 10 * ky + (fc ? 1 : 0)) {
        case 111: return pipe_launch<T, 1, 1, true>(d_pd, Nd, wpd, lds, st);
        case 121: return pipe_launch<T, 1, 2, true>(d_pd, Nd, wpd, lds, st);
        case 211: return pipe_launch<T, 2, 1, true>(d_pd, Nd, wpd, lds, st);
        case 131: return pipe_launch<T, 1, 3, true>(d_pd, Nd, wpd, lds, st);
        case 311: return pipe_launch<T, 3, 1, true>(d_pd, Nd, wpd, lds, st);
        case 141: return pipe_launch<T, 1, 4, true>(d_pd, Nd, wpd, lds, st);
        case 411: return pipe_launch<T, 4, 1, true>(d_pd, Nd, wpd, lds, st);
        case 221: return pipe_launch<T, 2, 2, true>(d_pd, Nd, wpd, lds, st);
        case 220: return pipe_launch<T, 2, 2, false>(d_pd, Nd, wpd, lds, st);
        case 230: return pipe_launch<T, 2, 3, false>(d_pd, Nd, wpd, lds, st);
        case 320: return pipe_launch<T, 3, 2, false>(d_pd, Nd, wpd, lds, st);
        default: throw std::runtime_error("2D closure orders out of the pipelined sweep's range");
    }
}

}  // namespace

// Up to 4 moments per cell (beyond that the solved columns do not fit the registers of a lane), and
// where the columns solved ahead pay for themselves: every cell is eliminated for 1 + kx + ky right-hand
// sides where the barrier walk has one, by fewer groups the more waves a diagonal takes, and a CU
// holds one or two of these workgroups where it holds four of the walk's.  Against the walk (in us, walk to
// here, 36 to 64, 128 and 200 to 256 cells across at 128 directions unless stated):
//  - One group (more than 256 cells): 693 -> 1317 (FP64, 257 cells of 4 moments), 572 -> 591 (FP32,
//    300 of 2), 1823 -> 1636 (FP64, 512 of 2): the walk.
//  - FP64, up to 3 moments: 78 -> 24, 267 -> 116, 474 -> 369, and still 85 -> 63 and 627 -> 485 at 800
//    directions.
//  - FP64, 4 moments: 93 -> 30, 303 -> 183, but 509 -> 602 with two groups (orders 2, 2; the others
//    612 -> 566 and 581 -> 564, at 288 directions 946 -> 1170), and with the workgroups in rounds of 256 at
//    128 cells 453 -> 410 for 512 directions, 563 -> 616 for 648, at 36 cells 96 -> 85 for 648 and
//    94 -> 109 for 800.
//  - FP32: 77 -> 21, 256 -> 102, 573 -> 423; with 5 face moments 85 -> 23, 285 -> 131, 626 -> 542, with two
//    groups and 288 directions 590 -> 661.
int sweep_2d_pipe_waves(int prec, int Nd, int Nx, int Ny, int kx, int ky, bool fc, size_t lds) {
    const int m = Nx < Ny ? Nx : Ny, nm = fc ? kx * ky : kx + ky - 1, nf = kx + ky;
    if (nm > 4 || m > 64 * PIPE_WAVES / 2 || lds > PIPE_LDS_MAX) return 0;
    int w = 1;
    while (64 * w < m) w *= 2;
    if (prec == P64 && nm == 4) {
        if (Nd > (w == 1 ? 768 : (w == 2 ? 512 : 256)) || (w > 2 && nf < 5)) return 0;
    } else if (w > 2 && nf > 4 && Nd > 256) {
        return 0;
    }
    return w;
}

void launch_sweep_2d_pipe(int prec, const PassDesc* d_pd, int Nd, int kx, int ky, bool fc, int wpd, size_t lds,
                          hipStream_t st) {
    if (Nd <= 0) return;
    if (prec == P64) pipe_dispatch<double>(d_pd, Nd, kx, ky, fc, wpd, lds, st);
    else pipe_dispatch<float>(d_pd, Nd, kx, ky, fc, wpd, lds, st);
    RT_HIP(hipGetLastError());
}

}  // namespace rt
