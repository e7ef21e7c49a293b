// kbg_fsm.hip -- KitBase's fast spectral Boltzmann collision operator (boltzmann_fft!,
// theory_fsm.jl:271-314) for the 1D1F3V step!(:fsm) (step_1f.jl:122-157), on gfx950.
//
// Per step, for the interior cells c0 .. c0 + ncell - 1 of a solve, with f_spec = fftshift(bfft(f)) / n3,
//   Q = 4 pi^2 / Kn / M^2 Re(sum_d F[f_spec phi_d] F[f_spec psi_d] - F[f_spec phipsi] F[f_spec])
// (d < M(M-1), F the forward 3D transform, sums in FP64).  The kernel modes phi, psi, phipsi
// (kernel_mode, theory_fsm.jl:24-90) come from the host with the descriptor.  Arrays are [w][v][u]
// with u fastest (KitBase's column-major f[i, j, k]); transforms, spectra and modes are FP64 for FP64
// storage and FP32 for FP32 storage (R below).  The update kernel adds dt Q to the transport update.
//
// Cubic grids of side 8, 12, 16, 18 or 24 take the library's own pencil transforms (kbg_fft.h):
//   FP64, modes even in the frequency (KitBase's are): one complex transform per pair of modes
//     k_fsm_spec    f_spec of every cell
//     k_fsm_slab    F of f_spec (a + i b) per (cell, pair), a and b the even parts of the pair's two modes
//     k_fsm_planes  the 2D transforms of the modes' odd parts, which live on the Nyquist planes
//     k_fsm_psum    Q from both
//   FP32: two transforms per pair, all of a pair in LDS
//     k_fsm_load, hipFFT backward, k_fsm_pair, k_fsm_sum
// Other grids and modes go through hipFFT:
//   k_fsm_load    f (storage precision) -> complex spec[cell][n3]
//   hipFFT        batched 3D backward transforms (bfft, unnormalised), one per cell
//   k_fsm_modes   the 2 M(M-1) + 2 products f_spec phi_d, f_spec psi_d, f_spec phipsi, f_spec -> work
//   hipFFT        batched 3D forward transforms of all the products in place
//   k_fsm_q       the sum of the products
#include <hip/hip_runtime.h>
#include <hipfft/hipfft.h>

#include <algorithm>
#include <cmath>
#include <type_traits>

#include "kbg_device.h"
#include "kbg_fft.h"
#include "kbg_types.h"

namespace kbg {

namespace {

template <class R> struct Cx;
template <> struct Cx<double> { using type = double2; };
template <> struct Cx<float> { using type = float2; };
template <class R> using cx_t = typename Cx<R>::type;

template <class T, class R>
__global__ __launch_bounds__(256) void k_fsm_load(const T* __restrict__ f, long fcs, int k0, int ncell, int n3,
                                                  cx_t<R>* __restrict__ spec) {
    const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= (size_t)ncell * n3) return;
    const int ci = int(i / n3), q = int(i % n3);
    cx_t<R> z;
    z.x = R(f[(long)(k0 + ci) * fcs + q]);
    z.y = R(0);
    spec[i] = z;
}

// fftshift: element (i, j, k) of the shifted array is element ((i + nu/2) % nu, ...) of the input
// for even sizes; in general the input index whose shift lands on (i, j, k), as Julia's
// circshift(x, n ÷ 2) and numpy's roll(x, n // 2) place it
template <class R>
__global__ __launch_bounds__(256) void k_fsm_modes(const cx_t<R>* __restrict__ spec, cx_t<R>* __restrict__ work,
                                                   const R* __restrict__ phi, const R* __restrict__ psi,
                                                   const R* __restrict__ phipsi, int nu, int nv, int nw, int nd, int ncell) {
    const int n3 = nu * nv * nw;
    const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= (size_t)ncell * n3) return;
    const int ci = int(i / n3), q = int(i % n3);
    const int iu = q % nu, jv = (q / nu) % nv, kw = q / (nu * nv);
    const int su = (iu - nu / 2 + nu) % nu, sv = (jv - nv / 2 + nv) % nv, sw = (kw - nw / 2 + nw) % nw;
    const cx_t<R> x = spec[(size_t)ci * n3 + su + nu * (sv + nv * sw)];
    const double inv = 1.0 / double(n3);
    const R sr = R(double(x.x) * inv), si = R(double(x.y) * inv);
    cx_t<R>* __restrict__ out = work + (size_t)ci * (2 * nd + 2) * n3 + q;
    cx_t<R> z;
    for (int d = 0; d < nd; d++) {
        const R a = phi[(size_t)d * n3 + q], b = psi[(size_t)d * n3 + q];
        z.x = sr * a;
        z.y = si * a;
        out[(size_t)(2 * d) * n3] = z;
        z.x = sr * b;
        z.y = si * b;
        out[(size_t)(2 * d + 1) * n3] = z;
    }
    const R c = phipsi[q];
    z.x = sr * c;
    z.y = si * c;
    out[(size_t)(2 * nd) * n3] = z;
    z.x = sr;
    z.y = si;
    out[(size_t)(2 * nd + 1) * n3] = z;
}

template <class R>
__global__ __launch_bounds__(256) void k_fsm_q(const cx_t<R>* __restrict__ work, double* __restrict__ Q, int n3, int nd,
                                               int ncell, double scale) {
    const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= (size_t)ncell * n3) return;
    const int ci = int(i / n3), q = int(i % n3);
    const cx_t<R>* __restrict__ in = work + (size_t)ci * (2 * nd + 2) * n3 + q;
    double re = 0.0;
    for (int d = 0; d < nd; d++) {
        const cx_t<R> a = in[(size_t)(2 * d) * n3], b = in[(size_t)(2 * d + 1) * n3];
        re += double(a.x) * double(b.x) - double(a.y) * double(b.y);
    }
    const cx_t<R> a = in[(size_t)(2 * nd) * n3], b = in[(size_t)(2 * nd + 1) * n3];
    re -= double(a.x) * double(b.x) - double(a.y) * double(b.y);
    Q[i] = scale * re;
}

KBG_D int fsm_xcd_item() {
    const int G = gridDim.x, bx = blockIdx.x;
    const int x8 = bx & 7, q8 = G >> 3, r8 = G & 7;
    return x8 * q8 + (x8 < r8 ? x8 : r8) + (bx >> 3);
}

// ---- FP32 storage on a cubic grid of N^3 velocities (N from fsm_cube_size): the forward transforms
// in LDS, no product array.  One workgroup per (cell, pair): pair p < nd transforms f_spec phi_p and
// f_spec psi_p, pair nd transforms f_spec phipsi and f_spec; the product Re(A B) of the two
// transforms is written per pair (part[cell][pair][n3]) and k_fsm_sum adds the pairs in a fixed
// order.  Each transform, with thread t < N^2 at (ta, tb) = (t % N, t / N):
//   1. the thread loads its w-pencil (u, v) = (ta, tb) of f_spec times the mode straight from global
//      memory (f_spec = fftshift(bfft(f)) / N^3), transforms it along w in registers and stores it
//      into an LDS array [w][v][u] whose rows are padded to an odd length (N | 1, so the pencils a
//      wavefront reads fall in different banks);
//   2. transforms the u-pencil (v, w) = (ta, tb) in LDS;
//   3. transforms the v-pencil (u, w) = (ta, tb) and keeps it in registers, where the second
//      transform's pencil meets the first.
template <int N> constexpr int fsm_pair_threads() { return (N * N + 63) / 64 * 64; }
// the first transform's kept v-pencil: its first KEEP values wait in LDS behind the array (registers
// for the rest), which keeps the kernel within the register budget of 576-thread workgroups
constexpr int kFsmKeep = 8;
template <int N> constexpr int fsm_pair_lds() { return N * N * (N | 1) * 8 + kFsmKeep * N * N * 8; }

template <int N>
__global__ __launch_bounds__(fsm_pair_threads<N>()) void k_fsm_pair(const float2* __restrict__ spec, const float* __restrict__ phi,
                                                                  const float* __restrict__ psi, const float* __restrict__ phipsi,
                                                                  const float2* __restrict__ tw, float* __restrict__ part, int nd,
                                                                  int ncell) {
    constexpr int N2 = N * N, N3 = N2 * N, P = N | 1, H = N / 2;
    extern __shared__ float2 lds[];
    const int np = nd + 1;
    const int item = fsm_xcd_item();
    if (item >= ncell * np) return;
    const int ci = item / np, p = item % np;
    const int t = threadIdx.x;
    const bool act = fsm_pair_threads<N>() == N2 || t < N2;  // 24^3: no branch around the pencils, 98 -> 87 us for 48 cells x 21 pairs
    const int ta = t % N, tb = t / N;
    // the thread's column of the unshifted spectrum: fftshift places element (ta, tb, k) at
    // ((ta + N - N/2) % N, (tb + N - N/2) % N, (k + N - N/2) % N)
    const float2* __restrict__ col = spec + (size_t)ci * N3 + (ta + N - H) % N + N * ((tb + N - H) % N);
    const float inv = 1.0f / float(N3);
    float2* keep = lds + N2 * P;  // [kFsmKeep][N2]: the first values of each thread's kept pencil
    float2 A[N];
    for (int h = 0; h < 2; h++) {
        const float* __restrict__ mode = p < nd ? (h ? psi : phi) + (size_t)p * N3 : (h ? nullptr : phipsi);
        if (h) __syncthreads();  // every pencil of the first transform has left the array
        float2 x[N], X[N];
        if (act) {  // 1. along w, from global memory
#pragma unroll
            for (int k = 0; k < N; k++) x[k] = col[N2 * ((k + N - H) % N)];
            const float* __restrict__ mc = mode + ta + N * tb;
#pragma unroll
            for (int k = 0; k < N; k++) {
                const float m = (mode ? mc[N2 * k] : 1.0f) * inv;
                x[k] = make_float2(x[k].x * m, x[k].y * m);
            }
            fft_dit<N, N, 1, float2>(x, X, tw);
            float2* r = lds + ta + P * tb;
#pragma unroll
            for (int k = 0; k < N; k++) r[P * N * k] = X[k];
        }
        __syncthreads();
        if (act) {  // 2. along u: pencil (v, w) = (ta, tb)
            float2* r = lds + P * (ta + N * tb);
#pragma unroll
            for (int k = 0; k < N; k++) x[k] = r[k];
            fft_dit<N, N, 1, float2>(x, X, tw);
#pragma unroll
            for (int k = 0; k < N; k++) r[k] = X[k];
        }
        __syncthreads();
        if (act) {  // 3. along v: pencil (u, w) = (ta, tb), kept in registers
            const float2* r = lds + ta + P * N * tb;
#pragma unroll
            for (int k = 0; k < N; k++) x[k] = r[P * k];
            fft_dit<N, N, 1, float2>(x, X, tw);
            if (h == 0) {
#pragma unroll
                for (int k = 0; k < N; k++) {
                    if (k < kFsmKeep) keep[k * N2 + t] = X[k];  // this thread's slots only
                    else A[k] = X[k];
                }
            } else {
                float* __restrict__ o = part + (size_t)item * N3 + ta + N2 * tb;
#pragma unroll
                for (int k = 0; k < N; k++) {
                    const float2 a = k < kFsmKeep ? keep[k * N2 + t] : A[k];
                    o[N * k] = a.x * X[k].x - a.y * X[k].y;
                }
            }
        }
    }
}

// Q = scale (sum_{p < nd} part_p - part_nd), pairs in order
__global__ __launch_bounds__(256) void k_fsm_sum(const float* __restrict__ part, double* __restrict__ Q, int n3, int nd,
                                                 int ncell, double scale) {
    const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= (size_t)ncell * n3) return;
    const int ci = int(i / n3), q = int(i % n3);
    const float* __restrict__ pp = part + (size_t)ci * (nd + 1) * n3 + q;
    double re = 0.0;
#pragma unroll 10  // ten loads in flight per thread: 10.9 us for the 56 MB of 48 cells of 24^3, 15.7 without
    for (int d = 0; d < nd; d++) re += double(pp[(size_t)d * n3]);
    re -= double(pp[(size_t)nd * n3]);
    Q[i] = scale * re;
}

template <int N> hipError_t launch_pair(const FsmPlan& P, hipStream_t st) {
    const int nd = P.M * (P.M - 1);
    hipLaunchKernelGGL(k_fsm_pair<N>, dim3(P.ncell * (nd + 1)), dim3(fsm_pair_threads<N>()), fsm_pair_lds<N>(), st,
                       (const float2*)P.spec, (const float*)P.phi, (const float*)P.psi, (const float*)P.phipsi,
                       (const float2*)P.tw, (float*)P.part, nd, P.ncell);
    return hipGetLastError();
}

// ---- FP64 storage on a cubic grid of N^3 velocities, even kernel modes ------------------------------
//
// f is real, so f_spec is Hermitian: f_spec(k') = conj f_spec(k), k' the index of the negated frequency
// ((N - i) % N per axis in the shifted layout; index 0, the Nyquist frequency, is its own partner).  A
// mode m splits into m_e(k) = (m(k) + m(k')) / 2 and m_o = m - m_e.  f_spec m_e is Hermitian, its transform
// real; f_spec m_o is anti-Hermitian, its transform imaginary.  For a pair of modes (a, b) the transform
// of f_spec (a_e + i b_e) is then A_r + i B_r -- both real transforms at once -- and that of
// f_spec (a_o + i b_o) is -B_i + i A_i, so with Z and Zo the two transforms
//   Re(F[f_spec a] F[f_spec b]) = A_r B_r - A_i B_i = Re Z Im Z + Re Zo Im Zo.
// KitBase's modes are even functions of the frequency, so m_o vanishes except on the planes where one
// index is 0 (there the partner negates only the other two axes): Zo(x, y, z) = P0(y, z) + P1(x, z) + P2(x, y),
// three 2D transforms.  fsm_pack_modes forms (a_e, b_e) and the planes of (a_o, b_o) on the host,
// scales a and b of a pair to the same size by powers of two (their product is unchanged), and
// reports whether the modes are even off the planes.
//
// Pair p < nd is (phi_p, psi_p).  The loss term takes two transforms, F[f_spec phipsi] and F[f_spec]
// (part[nd] and part[nd + 1] hold their real parts; F[f_spec] is real).  Packed as a pair (phipsi, 1) it
// would lose digits, its two transforms differing by orders of magnitude over the velocity grid (4e-5 of
// Q in FP32 on the 24^3 shock structure, against 3e-6); with F[f_spec] = (-1)^(x+y+z) f, exact, gain and
// loss would no longer come from the same rounded spectrum, and their moments would not cancel.

// w-planes per slab; the N / S slabs of an array take the frequencies congruent r mod N / S
template <int N> constexpr int fsm_slab() { return N % 8 == 0 ? 8 : 6; }
template <int N> constexpr int fsm_slab_threads() { return (fsm_slab<N>() * N + 63) / 64 * 64; }
template <int N> constexpr int fsm_slab_lds() { return fsm_slab<N>() * N * (N | 1) * 16; }

// The S frequencies NS q + r (q < S) of a length-N pencil x: one output of the radix-NS butterfly over
// x[m], x[m + S], .. (decimation in frequency), a twiddle, and a length-S transform.  load(k) returns x[k].
template <int N, int S, int RR, class F> KBG_D void fsm_pencil_part(F&& load, double2 (&X)[S], const double2* __restrict__ tw) {
    constexpr int NS = N / S;
    double2 y[S];
#pragma unroll
    for (int m = 0; m < S; m++) {
        double2 a = load(m);
        if constexpr (NS == 2) {
            const double2 b = load(m + S);
            a = RR ? fft_cx<double2>(a.x - b.x, a.y - b.y) : fft_cx<double2>(a.x + b.x, a.y + b.y);
        } else if constexpr (NS == 3) {
            const double2 b = load(m + S), c = load(m + 2 * S);
            const double2 s = fft_cx<double2>(b.x + c.x, b.y + c.y);
            if constexpr (RR == 0) {
                a = fft_cx<double2>(a.x + s.x, a.y + s.y);
            } else {
                const double h = RR == 1 ? 0.86602540378443864676 : -0.86602540378443864676;
                const double2 d = fft_cx<double2>(b.x - c.x, b.y - c.y);
                a = fft_cx<double2>(a.x - 0.5 * s.x + h * d.y, a.y - 0.5 * s.y - h * d.x);
            }
        }
        y[m] = fft_twiddle<N, double2>(a, m * RR, tw);
    }
    fft_dit<S, N, 1, double2>(y, X, tw);
}

// The slab r of the 3D transform of the array load(pen, k) (pen = u + N v, k the w index): w-pencils in
// registers, the slab's S planes in LDS (rows padded to an odd length, so the pencils a wavefront reads
// fall in different banks), u-pencils in LDS, v-pencils in registers, then store(u, v, q, X) for the
// thread's (u, q) and every v; w frequency NS q + r.  Threads: fsm_slab_threads.
template <int N, class L, class ST>
KBG_D void fsm_slab_transform(int r, double2* __restrict__ slab, const double2* __restrict__ tw, L&& load, ST&& store) {
    constexpr int N2 = N * N, P = N | 1, S = fsm_slab<N>(), NS = N / S, NTH = fsm_slab_threads<N>();
    const int t = threadIdx.x;
    for (int pen = t; pen < N2; pen += NTH) {
        double2 X[S];
        auto ld = [&](int k) { return load(pen, k); };
        if constexpr (NS == 1) {
            fsm_pencil_part<N, S, 0>(ld, X, tw);
        } else {  // r is uniform over the workgroup
            if (r == 0) fsm_pencil_part<N, S, 0>(ld, X, tw);
            else if (r == 1) fsm_pencil_part<N, S, 1>(ld, X, tw);
            else if constexpr (NS == 3) fsm_pencil_part<N, S, 2>(ld, X, tw);
        }
        double2* o = slab + pen % N + P * (pen / N);
#pragma unroll
        for (int q = 0; q < S; q++) o[P * N * q] = X[q];
    }
    __syncthreads();
    const bool act = t < S * N;
    const int ta = t % N, tb = t / N;
    double2 x[N], X[N];
    if (act) {  // u-pencil (v, q) = (ta, tb)
        double2* row = slab + P * (ta + N * tb);
#pragma unroll
        for (int k = 0; k < N; k++) x[k] = row[k];
        fft_dit<N, N, 1, double2>(x, X, tw);
#pragma unroll
        for (int k = 0; k < N; k++) row[k] = X[k];
    }
    __syncthreads();
    if (act) {  // v-pencil (u, q) = (ta, tb)
        const double2* col = slab + ta + P * N * tb;
#pragma unroll
        for (int k = 0; k < N; k++) x[k] = col[P * k];
        fft_dit<N, N, 1, double2>(x, X, tw);
#pragma unroll
        for (int k = 0; k < N; k++) store(ta, k, tb, X[k]);
    }
}

// f_spec = fftshift(bfft(f)) / N^3 of one slab of one cell: f is real, so bfft(f) = conj F[f]
template <int N>
__global__ __launch_bounds__(fsm_slab_threads<N>()) void k_fsm_spec(const double* __restrict__ f, long fcs, int k0, const double2* __restrict__ tw,
                                                                   double2* __restrict__ spec) {
    constexpr int N2 = N * N, N3 = N2 * N, H = N / 2, NS = N / fsm_slab<N>();
    extern __shared__ char smem[];
    const int r = blockIdx.x % NS, ci = blockIdx.x / NS;
    const double* __restrict__ fc = f + (long)(k0 + ci) * fcs;
    double2* __restrict__ o = spec + (size_t)ci * N3;
    const double inv = 1.0 / double(N3);
    fsm_slab_transform<N>(
        r, (double2*)smem, tw, [&](int pen, int k) { return fft_cx<double2>(fc[pen + N2 * k], 0.0); },
        [&](int u, int v, int q, double2 X) {
            o[(u + H) % N + N * ((v + H) % N) + N2 * ((NS * q + r + H) % N)] = fft_cx<double2>(X.x * inv, -X.y * inv);
        });
}

// The order of the slab work: each XCD (workgroup ids congruent mod 8) takes a contiguous run of
// [cell group][pair][cell of the group][slab], groups of ceil(ncell / 8) cells, so a pair's modes are
// read once into an XCD's L2 and reused by the group's cells, whose spectra stay there (FP64 24^3:
// 6 cells x 221 KB + 221 KB of modes against 4.6 MB of modes in cell-major order).
//
// part[cell][pair] = Re Z Im Z, Z the transform of f_spec (a_e + i b_e), and part[cell][nd], [nd + 1] = Re Z for
// the loss; one workgroup per (cell, pair, slab).  A slab keeps S/N of the array in LDS (77 KB of 24^3), so two workgroups share a CU.  For the
// 48 cells x 21 pairs of 24^3: 81 us, and 37 us for k_fsm_psum (two transforms per pair, written and read
// back as 446 MB of complex products, took 167 + 109 us).
template <int N>
__global__ __launch_bounds__(fsm_slab_threads<N>()) void k_fsm_slab(const double2* __restrict__ spec, const double2* __restrict__ ms,
                                                                   const double2* __restrict__ tw, double* __restrict__ part, int np, int ncell,
                                                                   int cg) {
    constexpr int N2 = N * N, N3 = N2 * N, NS = N / fsm_slab<N>();
    extern __shared__ char smem[];
    const int item = fsm_xcd_item(), per = cg * np * NS, g = item / per;
    const int in = item - g * per, ncg = min(cg, ncell - g * cg);
    const int r = in % NS, ci = g * cg + (in / NS) % ncg, p = in / (NS * ncg);
    const double2* __restrict__ sc = spec + (size_t)ci * N3;
    const double2* __restrict__ mp = ms + (size_t)p * N3;
    double* __restrict__ o = part + ((size_t)ci * np + p) * N3;
    fsm_slab_transform<N>(
        r, (double2*)smem, tw,
        [&](int pen, int k) {
            const double2 s = sc[pen + N2 * k], m = mp[pen + N2 * k];
            return fft_cx<double2>(s.x * m.x - s.y * m.y, s.x * m.y + s.y * m.x);
        },
        [&](int u, int v, int q, double2 X) { o[u + N * v + N2 * (NS * q + r)] = p < np - 2 ? X.x * X.y : X.x; });
}

// The 2D transforms of f_spec (a_o + i b_o) on the planes u = 0 ([w][v]), v = 0 ([w][u]) and w = 0
// ([v][u]) of each pair; kFsmPP pairs of one cell per workgroup (at most 64 KB of LDS), one pencil per thread
constexpr int kFsmPP = 2;
template <int N> constexpr int fsm_plane_threads() { return (3 * kFsmPP * N + 63) / 64 * 64; }
template <int N>
__global__ __launch_bounds__(fsm_plane_threads<N>()) void k_fsm_planes(const double2* __restrict__ spec, const double2* __restrict__ mo,
                                                                      const double2* __restrict__ tw, double2* __restrict__ planes,
                                                                      int np) {
    constexpr int N2 = N * N, N3 = N2 * N, P = N | 1, PP = kFsmPP;
    __shared__ double2 lds[3 * PP * N * P];
    const int ng = (np + PP - 1) / PP, ci = blockIdx.x / ng;
    const int t = threadIdx.x, ta = t % N, pl = (t / N) % 3, p = (blockIdx.x % ng) * PP + t / (3 * N);
    const bool act = t < 3 * PP * N && p < np;
    double2* a = lds + (t / N) * N * P;
    double2 x[N], X[N];
    if (act) {  // the pencil along the plane's slow axis at fast index ta
        const double2* __restrict__ sc = spec + (size_t)ci * N3 + (pl == 0 ? N * ta : ta);
        const double2* __restrict__ mp = mo + ((size_t)p * 3 + pl) * N2 + ta;
        const int st = pl == 2 ? N : N2;
#pragma unroll
        for (int k = 0; k < N; k++) {
            const double2 s = sc[st * k], m = mp[N * k];
            x[k] = fft_cx<double2>(s.x * m.x - s.y * m.y, s.x * m.y + s.y * m.x);
        }
        fft_dit<N, N, 1, double2>(x, X, tw);
#pragma unroll
        for (int k = 0; k < N; k++) a[P * k + ta] = X[k];
    }
    __syncthreads();
    if (act) {  // the fast axis at slow index ta
#pragma unroll
        for (int k = 0; k < N; k++) x[k] = a[P * ta + k];
        fft_dit<N, N, 1, double2>(x, X, tw);
        double2* __restrict__ o = planes + (((size_t)ci * np + p) * 3 + pl) * N2 + N * ta;
#pragma unroll
        for (int k = 0; k < N; k++) o[k] = X[k];
    }
}

// Q = scale (sum_{p < nd} (part_p + Re Zo Im Zo) - part_nd part_{nd+1}), pairs in order
template <int N>
__global__ __launch_bounds__(256) void k_fsm_psum(const double* __restrict__ part, const double2* __restrict__ planes, double* __restrict__ Q,
                                                 int nd, int ncell, double scale) {
    constexpr int N2 = N * N, N3 = N2 * N;
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i >= ncell * N3) return;
    const int ci = i / N3, q = i % N3;
    const int x = q % N, y = (q / N) % N, z = q / N2;
    const double* __restrict__ pp = part + (size_t)ci * (nd + 2) * N3 + q;
    const double2* __restrict__ pl = planes + (size_t)ci * nd * 3 * N2;
    double re = 0.0;
#pragma unroll 4
    for (int p = 0; p < nd; p++) {
        const double2* __restrict__ a = pl + (size_t)p * 3 * N2;
        const double2 c0 = a[y + N * z], c1 = a[N2 + x + N * z], c2 = a[2 * N2 + x + N * y];
        const double gr = c0.x + c1.x + c2.x, gi = c0.y + c1.y + c2.y;
        re += pp[(size_t)p * N3] + gr * gi;
    }
    re -= pp[(size_t)nd * N3] * pp[(size_t)(nd + 1) * N3];
    Q[i] = scale * re;
}

template <int N> hipError_t fsm_run_packed(const FsmPlan& P, const double* f, long fcs, int k0, double scale, hipStream_t st) {
    constexpr int NS = N / fsm_slab<N>(), TH = fsm_slab_threads<N>();
    constexpr size_t lds = fsm_slab_lds<N>();
    const int nd = P.M * (P.M - 1), np = nd + 2, cg = (P.ncell + 7) / 8;
    double2* spec = (double2*)P.spec;
    double2* planes = (double2*)P.planes;
    double* part = (double*)P.part;
    const double2* tw = (const double2*)P.tw;
    hipLaunchKernelGGL(k_fsm_spec<N>, dim3(P.ncell * NS), dim3(TH), lds, st, f, fcs, k0, tw, spec);
    hipLaunchKernelGGL(k_fsm_planes<N>, dim3(P.ncell * ((nd + kFsmPP - 1) / kFsmPP)), dim3(fsm_plane_threads<N>()), 0, st, spec,
                       (const double2*)P.mo, tw, planes, nd);
    hipLaunchKernelGGL(k_fsm_slab<N>, dim3(P.ncell * np * NS), dim3(TH), lds, st, spec, (const double2*)P.ms, tw, part, np, P.ncell, cg);
    hipLaunchKernelGGL(k_fsm_psum<N>, dim3((P.ncell * N * N * N + 255) / 256), dim3(256), 0, st, part, planes, P.Q, nd, P.ncell, scale);
    return hipGetLastError();
}

template <int N> hipError_t cube_attr(bool f32) {
    if (f32) return hipFuncSetAttribute((const void*)k_fsm_pair<N>, hipFuncAttributeMaxDynamicSharedMemorySize, fsm_pair_lds<N>());
    const hipError_t e = hipFuncSetAttribute((const void*)k_fsm_spec<N>, hipFuncAttributeMaxDynamicSharedMemorySize, fsm_slab_lds<N>());
    if (e != hipSuccess) return e;
    return hipFuncSetAttribute((const void*)k_fsm_slab<N>, hipFuncAttributeMaxDynamicSharedMemorySize, fsm_slab_lds<N>());
}

// fn(std::integral_constant<int, N>) for the plan's side
template <class F> hipError_t with_cube(int n, F&& fn) {
    switch (n) {
    case 8: return fn(std::integral_constant<int, 8>{});
    case 12: return fn(std::integral_constant<int, 12>{});
    case 16: return fn(std::integral_constant<int, 16>{});
    case 18: return fn(std::integral_constant<int, 18>{});
    case 24: return fn(std::integral_constant<int, 24>{});
    default: return hipErrorInvalidValue;
    }
}

unsigned blocks_of(size_t n) { return unsigned((n + 255) / 256); }

hipfftResult exec(const FsmPlan& P, hipfftHandle_t* plan, void* data, int dir) {
    if (P.f32) return hipfftExecC2C(plan, (hipfftComplex*)data, (hipfftComplex*)data, dir);
    return hipfftExecZ2Z(plan, (hipfftDoubleComplex*)data, (hipfftDoubleComplex*)data, dir);
}

template <class R> hipError_t fsm_run(const FsmPlan& P, bool fp64, const void* f, long fcs, int k0, hipStream_t st) {
    const double scale = 4.0 * kPi * kPi / P.kn / (double(P.M) * P.M);
    const int n3 = P.nu * P.nv * P.nw, nd = P.M * (P.M - 1);
    const size_t cells = (size_t)P.ncell * n3;
    const dim3 g(blocks_of(cells)), b(256);
    if (P.packed)
        return with_cube(P.cube_n, [&](auto n) { return fsm_run_packed<decltype(n)::value>(P, (const double*)f, fcs, k0, scale, st); });
    cx_t<R>* spec = (cx_t<R>*)P.spec;
    cx_t<R>* work = (cx_t<R>*)P.work;
    if (fp64) hipLaunchKernelGGL((k_fsm_load<double, R>), g, b, 0, st, (const double*)f, fcs, k0, P.ncell, n3, spec);
    else hipLaunchKernelGGL((k_fsm_load<float, R>), g, b, 0, st, (const float*)f, fcs, k0, P.ncell, n3, spec);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    if (hipfftSetStream(P.plan_b, st) != HIPFFT_SUCCESS) return hipErrorUnknown;
    if (exec(P, P.plan_b, spec, HIPFFT_BACKWARD) != HIPFFT_SUCCESS) return hipErrorUnknown;
    if (P.cube_n) {  // FP32
        e = with_cube(P.cube_n, [&](auto n) { return launch_pair<decltype(n)::value>(P, st); });
        if (e != hipSuccess) return e;
        hipLaunchKernelGGL(k_fsm_sum, g, b, 0, st, (const float*)P.part, P.Q, n3, nd, P.ncell, scale);
        return hipGetLastError();
    }
    if (hipfftSetStream(P.plan_f, st) != HIPFFT_SUCCESS) return hipErrorUnknown;
    hipLaunchKernelGGL(k_fsm_modes<R>, g, b, 0, st, spec, work, (const R*)P.phi, (const R*)P.psi, (const R*)P.phipsi, P.nu,
                       P.nv, P.nw, nd, P.ncell);
    if ((e = hipGetLastError()) != hipSuccess) return e;
    if (exec(P, P.plan_f, work, HIPFFT_FORWARD) != HIPFFT_SUCCESS) return hipErrorUnknown;
    hipLaunchKernelGGL(k_fsm_q<R>, g, b, 0, st, work, P.Q, n3, nd, P.ncell, scale);
    return hipGetLastError();
}

}  // namespace

int fsm_cube_size(int nu, int nv, int nw, bool f32, int nm, const double* phi, const double* psi, const double* phipsi) {
    if (nu != nv || nu != nw) return 0;
    for (int n : {8, 12, 16, 18, 24})
        if (n == nu) return f32 || !phi || !psi || !phipsi || fsm_pack_modes(n, nm, phi, psi, phipsi, nullptr, nullptr) ? n : 0;
    return 0;
}

bool fsm_pack_modes(int N, int nm, const double* phi, const double* psi, const double* phipsi, double* ms, double* mo) {
    const int nd = nm * (nm - 1), N2 = N * N, N3 = N2 * N;
    if (ms)  // the loss: phipsi as it is, odd part included, and 1
        for (int i = 0; i < N3; i++) {
            ms[((size_t)nd * N3 + i) * 2] = phipsi[i];
            ms[((size_t)(nd + 1) * N3 + i) * 2] = 1.0;
            ms[((size_t)nd * N3 + i) * 2 + 1] = ms[((size_t)(nd + 1) * N3 + i) * 2 + 1] = 0.0;
        }
    for (int p = 0; p < nd; p++) {
        const double* ab[2] = {phi + (size_t)p * N3, psi + (size_t)p * N3};
        double mx[2] = {0.0, 0.0};
        for (int h = 0; h < 2; h++)
            for (int i = 0; i < N3; i++) mx[h] = std::max(mx[h], std::fabs(ab[h][i]));
        if (!std::isfinite(mx[0]) || !std::isfinite(mx[1])) return false;
        // a 2^e and b 2^-e of about the same size: the transforms share one complex array, whose rounding
        // follows the larger of the two
        const int e = mx[0] > 0.0 && mx[1] > 0.0 ? int(std::lround(0.5 * std::log2(mx[1] / mx[0]))) : 0;
        for (int i = 0; i < N3; i++) {
            const int x = i % N, y = (i / N) % N, z = i / N2;
            const int j = (N - x) % N + N * ((N - y) % N) + N2 * ((N - z) % N);
            for (int h = 0; h < 2; h++) {
                const double a = ab[h][i], b = ab[h][j], odd = 0.5 * (a - b), sc = std::ldexp(1.0, h ? -e : e);
                const bool plane = x == 0 || y == 0 || z == 0;
                if (!(std::fabs(odd) <= (plane ? mx[h] : 1e-14 * mx[h]))) return false;  // a NaN, or not even (45 FP64 ulp)
                if (!ms) continue;
                ms[((size_t)p * N3 + i) * 2 + h] = 0.5 * (a + b) * sc;
                if (!plane) continue;
                // one plane per element: u = 0 first, then v = 0, then w = 0
                const int pl = x == 0 ? 0 : (y == 0 ? 1 : 2), at = pl == 0 ? y + N * z : (pl == 1 ? x + N * z : x + N * y);
                mo[(((size_t)p * 3 + pl) * N2 + at) * 2 + h] = odd * sc;
            }
        }
    }
    return true;
}

hipError_t fsm_collision(const FsmPlan& P, bool fp64, const void* f, long fcs, int k0, hipStream_t st) {
    if (P.ncell <= 0) return hipSuccess;
    return P.f32 ? fsm_run<float>(P, fp64, f, fcs, k0, st) : fsm_run<double>(P, fp64, f, fcs, k0, st);
}

hipError_t fsm_plan_create(FsmPlan& P) {
    const int n3 = P.nu * P.nv * P.nw, nd = P.M * (P.M - 1);
    if (P.cube_n) {
        const hipError_t e = with_cube(P.cube_n, [&](auto n) { return cube_attr<decltype(n)::value>(P.f32); });
        if (e != hipSuccess || P.packed) return e;
    }
    int n[3] = {P.nw, P.nv, P.nu};
    const hipfftType t = P.f32 ? HIPFFT_C2C : HIPFFT_Z2Z;
    if (hipfftPlanMany(&P.plan_b, 3, n, nullptr, 1, n3, nullptr, 1, n3, t, P.ncell) != HIPFFT_SUCCESS) return hipErrorUnknown;
    if (!P.cube_n &&
        hipfftPlanMany(&P.plan_f, 3, n, nullptr, 1, n3, nullptr, 1, n3, t, P.ncell * (2 * nd + 2)) != HIPFFT_SUCCESS) {
        hipfftDestroy(P.plan_b);
        return hipErrorUnknown;
    }
    P.planned = true;
    return hipSuccess;
}

void fsm_plan_destroy(FsmPlan& P) {
    if (!P.planned) return;
    hipfftDestroy(P.plan_b);
    if (!P.cube_n) hipfftDestroy(P.plan_f);
    P.planned = false;
}

}  // namespace kbg
