// kbg_sweep_f32b.hip -- FP32 fused 1D sweep, two distributions, KFVS; the conversions of the FP32
// sweep's stored departures.
#include "kbg_sweep.h"

namespace kbg {

hipError_t launch_sweep_f32_2kfvs(int wg_waves, const Solve1D* d_solves, const WorkItem* d_items, const Pack* d_packs,
                                  int npacks, int par, double* d_rpart, int nstep, hipStream_t st) {
    return launch_sweep_t<float, 2, KFVS>(wg_waves, d_solves, d_items, d_packs, npacks, par, d_rpart, nstep, st);
}

// Conversions of an FP32 swept solve's f buffer between the stored departure d = f - M~(prim) and f
// (kbg_sweep.h maxw_coef / maxw_at): one thread per (storage cell, distribution row).
__global__ __launch_bounds__(256) void k_delta1d(const Solve1D* __restrict__ pS, double* __restrict__ stage, int mode, int buf) {
    const Solve1D& S = *pS;
    const int N = S.nx + 2 * S.ng;
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    const int row = blockIdx.y;  // q nv + v
    if (k >= N) return;
    const int q = row >= S.nv ? 1 : 0, v = row - q * S.nv;
    double p[3];
    conserve_prim<3>(S.w[buf] + (size_t)k * 3, S.gam, p);  // the w buffer paired with f[buf]
    const MaxwCoef mc = maxw_coef(p, S.K);
    const VChunk<float>* vt = (const VChunk<float>*)S.vtab;
    float M = maxw_at(vt[v / kVChunk], mc.A, mc.nl2, mc.U, v % kVChunk);
    if (q == 1) M = maxw_b(M, mc.kb);
    const size_t o = (size_t)row * S.np + k;
    float* f = (float*)S.f[buf];
    if (mode == 0) f[o] = float(stage[o] - double(M));
    else if (mode == 1) f[o] = M + f[o];
    else f[o] = f[o] - M;
}

hipError_t launch_delta1d(const Solve1D& S, const Solve1D* d_S, double* stage, int mode, int buf, hipStream_t st) {
    const int N = S.nx + 2 * S.ng;
    if (!S.delta || N <= 0) return hipSuccess;
    if (mode < 0 || mode > 2 || (mode == 0 && !stage)) return hipErrorInvalidValue;
    hipLaunchKernelGGL(k_delta1d, dim3((N + 255) / 256, S.nf * S.nv), dim3(256), 0, st, d_S, stage, mode, buf);
    return hipGetLastError();
}

// A swept solve's state as the host keeps it: cells k0 .. k0 + n - 1 of buffer `buf`, f [n][nf][nv] as FP64
// (a stored departure as M~ + d, exactly), then w and prim [n][3], written straight into pinned host memory.
// Tiles of 32 cells x 64 velocities turn through LDS: 128-byte reads (FP32) along the cells, 512-byte
// writes along the velocities.  Bound by the host's own copy of the pinned block and the launch and wait per
// solve: 256 ragged tubes (311 MB) 32 ms, 24 of them 3.2 ms.  An FP64 copy in the swept layout, a pageable
// copy of it to the host and one host thread's strided walk took 85 and 10 ms.
template <class T, bool DELTA>
__global__ __launch_bounds__(256) void k_down1d(Solve1D S, int buf, int k0, int n, double* __restrict__ out) {
    __shared__ double tile[64][33];
    const int nv = S.nv, nf = S.nf, q = blockIdx.z, v0 = blockIdx.y * 64;
    if (q == nf) {
        if (blockIdx.y > 0) return;
        double* ow = out + (size_t)n * nf * nv;
        const int e = blockIdx.x * 96 + threadIdx.x;
        if (threadIdx.x < 96 && e < 3 * n) {
            ow[e] = S.w[buf][(size_t)k0 * 3 + e];
            ow[(size_t)3 * n + e] = S.prim[(size_t)k0 * 3 + e];
        }
        return;
    }
    const int c = threadIdx.x & 31, vc = threadIdx.x >> 5, kk = blockIdx.x * 32 + c, k = k0 + kk;
    if (kk < n) {
        const T* f = (const T*)S.f[buf];
        MaxwCoef mc{};
        if constexpr (DELTA) {
            double p[3];
            conserve_prim<3>(S.w[buf] + (size_t)k * 3, S.gam, p);
            mc = maxw_coef(p, S.K);
        }
        for (int j = 0; j < kVChunk; j++) {
            const int v = v0 + vc * kVChunk + j;
            if (v >= nv) break;
            double x = double(f[((size_t)q * nv + v) * S.np + k]);
            if constexpr (DELTA) {
                const VChunk<float>* vt = (const VChunk<float>*)S.vtab;
                float M = maxw_at(vt[v / kVChunk], mc.A, mc.nl2, mc.U, v % kVChunk);
                if (q == 1) M = maxw_b(M, mc.kb);
                x = double(M) + x;
            }
            tile[vc * kVChunk + j][c] = x;
        }
    }
    __syncthreads();
    const int lane = threadIdx.x & 63;
    if (v0 + lane >= nv) return;
    for (int r = threadIdx.x >> 6; r < 32 && blockIdx.x * 32 + r < n; r += 4)
        out[((size_t)(blockIdx.x * 32 + r) * nf + q) * nv + v0 + lane] = tile[lane][r];
}

hipError_t launch_down1d(bool fp64, bool delta, const Solve1D& S, int buf, int k0, int n, double* out, hipStream_t st) {
    if (!S.swept || k0 < 0 || n < 1 || k0 + n > S.nx + 2 * S.ng || (delta && (fp64 || !S.delta))) return hipErrorInvalidValue;
    const dim3 grid((n + 31) / 32, (S.nv + 63) / 64, S.nf + 1);
    if (fp64) hipLaunchKernelGGL((k_down1d<double, false>), grid, dim3(256), 0, st, S, buf, k0, n, out);
    else if (delta) hipLaunchKernelGGL((k_down1d<float, true>), grid, dim3(256), 0, st, S, buf, k0, n, out);
    else hipLaunchKernelGGL((k_down1d<float, false>), grid, dim3(256), 0, st, S, buf, k0, n, out);
    return hipGetLastError();
}

}  // namespace kbg
