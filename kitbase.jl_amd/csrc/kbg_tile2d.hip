// kbg_tile2d.hip -- the fused 2D time step for van Leer slopes, BGK and Maxwell walls on all sides
// (2D2F2V and 2D1F2V), batched over solves.
//
// One solve!-loop iteration (reconstruct! + evolve! + Maxwell walls + update!) in three launches per
// group of solves of one precision and flux:
//
//   k_tile2d   one thread per velocity, a workgroup of 256 over a tile of kTX cells along x and up to
//              kTile2dRows rows, marching up the rows: every distribution value is loaded once per tile, each
//              cell's slopes are formed once, and the interior face fluxes never go to memory: their
//              places in the flux arrays hold the transport update G = f + sum of face fluxes / ds (g_face).
//              The last step of a call leaves the fluxes there instead, as evolve! does, and k_relax2d
//              forms G from f and them, with the same operations.  The tile's face records sit in
//              LDS: as scalar loads their waits and the spills of scalar registers took a third of the
//              kernel.  Faces between tiles are evaluated by both, with the same operations; the tile to
//              their right (above) adds up their moments in FP64.
//   k_chain2d  16 lanes per cell: the four faces' moments (the workgroups' sums in order) and the FP64 cell
//              chain (w, prim, the relaxation's coefficients).
//   k_relax2d  one workgroup per cell: f = (G + (dt / tau) M) / (1 + dt / tau), and for a cell next to a wall
//              the wall's flux of the next step; workgroups before them form the next step's interface
//              chains (KCU / UGKS: a record of the flux's coefficients in the storage type, FaceRec, and one
//              of its moments, frec), which need only w.
//
// A call's first step takes walls and records from k_pre2d.
//
// k_flux2d / k_cell2d (kbg_step2d.hip) keep every face's flux in memory: seven passes over an array of the
// size of f per step against four here, three loads per face and velocity, and the cell chain between each
// cell's loads and stores.  us per step there / here, h and b: UGKS 64 x 64 cells x 32^2 velocities FP32 91 / 61,
// FP64 151 / 95, 128 x 128 x 48^2 FP32 1140 / 489, 100 x 100 x 40^2 FP64 704 / 426; KFVS 96 x 96 x 32^2 FP32 146 /
// 95.  k_tile2d is bound by the issue of vector instructions (UGKS FP32: 315 us of the 489), k_relax2d by memory
// (4.6 TB/s), k_chain2d by latency; small KFVS meshes, whose walls' latency is
// the step, stay with the other kernels (tiled2d, kbg_api.hip).
//
// The mesh is axis-aligned (x-face normals (n, 0), y-face normals (0, n), n > 0), so a velocity's upwind side
// is the sign of u or v.  Lanes take the velocities in the order of vperm, sorted by the two signs: in most
// wavefronts both are the same for all lanes, and their variants of the flux need no coefficients of the
// other side and no selects.
//
// Reference: the files cited in kbg_step2d.hip.
#include <algorithm>

// Products and sums are contracted to fma within an expression, by the source, and not across expressions by
// the optimizer, which would pick differently in each copy of the flux: a face between two tiles is
// evaluated by both, from different copies, with the same result.
#pragma clang fp contract(on)

#include "kbg_device.h"
#include "kbg_face2d.h"
#include "kbg_types.h"

namespace kbg {

namespace {

constexpr int kTX = kTile2dX;

// An interior face's flux coefficients in the storage type, the length folded in.  With x, y the normal and
// tangential velocity, h, b the upwind face values and sh, sb their slopes, H = exp(nl |c - U|^2):
//   UGKS  fh = x (H (P + x R) + M3 eh), eh = h - rho x sh,  P, R polynomials 1, x, y, x^2 + y^2 (R of the upwind
//         side), rho = M4 / M3; fb = x (H (kb (P + x R) + x2 (P3 + x R3)) + M3 eb)   (flux_ugks.jl:209-245 factored)
//   KCU   fh = x (H P0 + M3 h), fb = x (H kb P0 + M3 b)             (flux_kcu.jl:898-967)
//   KFVS  fh = x M3 eh, fb alike                                    (flux_kfvs.jl:654-697)
// The moment sums run over w x eh, and M3 multiplies them in FP64 (frec).  FP32 carries rho in two parts: a
// coefficient's own rounding is the same for all velocities and does not cancel in the sums as theirs do.
template <class T> struct alignas(16) FaceRec {
    T nl, U, V, kb, M3, rho, x2, r, P[4];  // x2: <xi^4> - <xi^2>^2; r: 1 / centre distance
    struct {
        T q[4], d;  // R, and the signed half width of the side's cell
    } s[2];        // left, right
    T rhol, pad;    // rho + rhol
};
static_assert(sizeof(FaceRec<float>) == kFaceT * 4 && sizeof(FaceRec<double>) == kFaceT * 8, "FaceRec");

template <class T> KBG_D Tile2D bufs(const Solve2D& S) { return tile2d_at(S.tile, S.nx, S.ny, S.nv, sizeof(T)); }

template <class T> KBG_D T nl_of(double lam);
template <> KBG_D float nl_of<float>(double lam) { return float(-lam * 1.4426950408889634074); }
template <> KBG_D double nl_of<double>(double lam) { return -lam; }
// The limiter's quotient.  FP32: the hardware reciprocal, as in every kernel (tdiv).  FP64: a / x by a reciprocal of
// two Newton steps and one correction by the quotient's own remainder (Markstein, IBM J. Res. Dev. 34, 1990): of 4.2 M
// limiter quotients all are the division's to the bit, 18 % are not without the correction; UGKS 100 x 100 cells x
// 40^2 velocities 426 us per step without, 430 with it
KBG_D float quot(float a, float x) { return a * __builtin_amdgcn_rcpf(x); }
KBG_D double quot(double a, double x) {
    double r = __builtin_amdgcn_rcp(x);
    r = __builtin_fma(__builtin_fma(-x, r, 1.0), r, r);
    r = __builtin_fma(__builtin_fma(-x, r, 1.0), r, r);
    const double q = a * r;
    return __builtin_fma(__builtin_fma(-x, q, a), r, q);
}
KBG_D float gauss(float x) { return __builtin_amdgcn_exp2f(x); }
KBG_D double gauss(double x) { return exp(x); }

// the interior face `b` of a solve, x-faces (i = 2..nx) then y-faces (j = 2..ny)
template <class T, int FLUX> KBG_D void face_chain(const Solve2D& S, int b) {
    const int nx = S.nx, ny = S.ny, nxf = (nx - 1) * ny;
    int dir, fi, cL, cR;
    if (b < nxf) {
        dir = 0;
        const int i = b % (nx - 1) + 2, j = b / (nx - 1) + 1;
        fi = (i - 1) + (nx + 1) * (j - 1);
        cL = (i - 2) + nx * (j - 1);
        cR = cL + 1;
    } else {
        b -= nxf;
        dir = 1;
        const int i = b % nx + 1, j = b / nx + 2;
        fi = (i - 1) + nx * (j - 1);
        cL = (i - 1) + nx * (j - 2);
        cR = cL + nx;
    }
    const double* geo = (dir == 0 ? S.xgeo : S.ygeo) + (size_t)fi * 3;
    const double n1 = geo[0], n2 = geo[1], len = geo[2], dt = S.dt;
    const double* d = dir == 0 ? S.dx : S.dy;
    const double dxL = 0.5 * d[cL], dxR = 0.5 * d[cR];
    const Tile2D B = bufs<T>(S);
    FaceRec<T>& o = ((FaceRec<T>*)(dir == 0 ? B.xrec : B.yrec))[fi];
    double* fr = (dir == 0 ? B.xfrec : B.yfrec) + (size_t)fi * 8;
    o.r = T(1.0 / (0.5 * (d[cL] + d[cR])));
    o.s[0].d = T(dxL);
    o.s[1].d = T(-dxR);
    if constexpr (FLUX == KFVS) {
        o.M3 = T(dt * len);
        o.rho = T(0.5 * dt);
        o.rhol = T(0.5 * dt - double(o.rho));
        for (int m = 0; m < 4; m++) fr[m] = 0.0;
        fr[4] = dt * len;
    } else {
        const double* w = S.w;
        double swL[4], swR[4], wl[4], wr[4], WL[4], WR[4];
        wslope(S, w, cL, dir, swL);
        wslope(S, w, cR, dir, swR);
        for (int m = 0; m < 4; m++) {
            wl[m] = w[(size_t)cL * 4 + m] + dxL * swL[m];
            wr[m] = w[(size_t)cR * 4 + m] - dxR * swR[m];
        }
        local_frame4(wl, n1, n2, WL);
        local_frame4(wr, n1, n2, WR);
        if constexpr (FLUX == KCU) {
            KcuFace<4> F;
            kcu_face<4>(WL, WR, S.K, S.gam, S.mu, S.om, dt, F);
            o.nl = nl_of<T>(F.prim[3]);
            o.U = T(F.prim[1]);
            o.V = T(F.prim[2]);
            o.kb = T(S.K / (2.0 * F.prim[3]));
            o.P[0] = T(F.Mt1 * len * (F.prim[0] * (F.prim[3] / kPi)));
            o.M3 = T(F.Mt2 * len);
            for (int m = 0; m < 4; m++) fr[m] = F.fw0[m] * len;
            fr[4] = F.Mt2 * len;
        } else {
            UgksFace2 F;
            ugks_face_2d(WL, WR, S.K, S.gam, S.mu, S.om, dt, dxL, dxR, F);
            const double kb = S.K / (2.0 * F.prim[3]), A = F.prim[0] * (F.prim[3] / kPi) * len;
            const double a0 = A * F.Mt[0], a1 = A * F.Mt[1], a2 = A * F.Mt[2];
            o.nl = nl_of<T>(F.prim[3]);
            o.U = T(F.prim[1]);
            o.V = T(F.prim[2]);
            o.kb = T(kb);
            o.M3 = T(F.Mt[3] * len);
            const double rho = F.Mt[3] != 0.0 ? F.Mt[4] / F.Mt[3] : 0.0;  // both 0 there
            o.rho = T(rho);
            o.rhol = T(rho - double(o.rho));
            o.P[0] = T(a0 + a2 * (F.aT[0] + 0.5 * F.aT[3] * kb));
            o.P[1] = T(a2 * F.aT[1]);
            o.P[2] = T(a2 * F.aT[2]);
            o.P[3] = T(a2 * 0.5 * F.aT[3]);
            o.s[0].q[0] = T(a1 * (F.aL[0] + 0.5 * F.aL[3] * kb));
            o.s[0].q[1] = T(a1 * F.aL[1]);
            o.s[0].q[2] = T(a1 * F.aL[2]);
            o.s[0].q[3] = T(a1 * 0.5 * F.aL[3]);
            o.s[1].q[0] = T(a1 * (F.aR[0] + 0.5 * F.aR[3] * kb));
            o.s[1].q[1] = T(a1 * F.aR[1]);
            o.s[1].q[2] = T(a1 * F.aR[2]);
            o.s[1].q[3] = T(a1 * 0.5 * F.aR[3]);
            o.x2 = T(F.Mxi2 - kb * kb);
            for (int m = 0; m < 4; m++) fr[m] = F.fw0[m] * len;
            fr[4] = F.Mt[3] * len;
        }
    }
    fr[5] = n1;
    fr[6] = n2;
}

// Maxwell wall face fi of direction dir (flux_boundary.jl:190-220) next to cell c, one workgroup: outgoing
// velocities carry the cell's own h, b; incoming ones the wall Maxwellian whose density gives zero mass flux.
// Writes ff, fw and, for departure solves, the face's coefficient of Mr.  The operations of k_flux2d's
// walls (kbg_step2d.hip), with the velocities read twice instead of kept: few registers, so that it can share
// a launch with the relaxation.  red: 36 doubles of LDS.
template <class T> KBG_D void wall2d(const Solve2D& S, int dir, int fi, int side, int c, double* red) {
    const int nv = S.nv, RS = 2 * nv, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const T* h = (const T*)S.f + (size_t)c * RS;  // k_relax2d reads back what each thread stored: no restrict
    T* fo = (T*)(dir == 0 ? S.xff : S.yff) + (size_t)fi * RS;
    double* fwout = (dir == 0 ? S.xfw : S.yfw) + (size_t)fi * 4;
    const T* __restrict__ U = (const T*)S.u;
    const T* __restrict__ V = (const T*)S.v;
    const T* __restrict__ WT = (const T*)S.wt;
    const double* geo = (dir == 0 ? S.xgeo : S.ygeo) + (size_t)fi * 3;
    const double n1 = geo[0], n2 = geo[1], len = geo[2];
    const T n1T = T(n1), n2T = T(n2);
    const double dt = S.dt, K = S.K;
    double bcl[4];
    local_frame4((dir == 0 ? S.xwall : S.ywall) + (size_t)fi * 4, n1, n2, bcl);
    const T Uw = T(bcl[1]), Vw = T(bcl[2]), lw = T(bcl[3]), rotT = (side & 1) ? T(-1) : T(1);
    // FP32 departures: the cell's h, b are Mr + the stored values, and the stored wall flux leaves out
    // Mr's part x Mr len dt
    const bool del = sizeof(T) == 4 && S.delta;
    double r9[9];
#pragma unroll
    for (int m = 0; m < 9; m++) r9[m] = 0.0;
    for (int v0 = tid; v0 < nv; v0 += 1024) {
        T hv[4], bv[4], uv[4], vv[4], wv[4], sm[9];
#pragma unroll
        for (int k = 0; k < 4; k++) {
            const int iv = min(v0 + 256 * k, nv - 1);
            hv[k] = h[iv];
            bv[k] = h[nv + iv];
            uv[k] = U[iv];
            vv[k] = V[iv];
            wv[k] = v0 + 256 * k < nv ? WT[iv] : T(0);
            if constexpr (sizeof(T) == 4) {
                if (del) {
                    hv[k] += S.mref[iv];
                    bv[k] += S.mref[nv + iv];
                }
            }
        }
#pragma unroll
        for (int m = 0; m < 9; m++) sm[m] = T(0);
#pragma unroll
        for (int k = 0; k < 4; k++) {
            const T x = uv[k] * n1T + vv[k] * n2T, y = vv[k] * n1T - uv[k] * n2T, q2 = x * x + y * y, wq = wv[k];
            if (!(x * rotT >= T(0))) {
                sm[0] += wq * x * hv[k];
                sm[1] += wq * (x * x) * hv[k];
                sm[2] += wq * y * (hv[k] * x);
                sm[3] += wq * x * (hv[k] * q2);
                sm[4] += wq * x * bv[k];
            } else {
                const T cu = x - Uw, cv = y - Vw;
                const T e = texp(-lw * (cu * cu + cv * cv));
                sm[5] += wq * x * e;
                sm[6] += wq * (x * x) * e;
                sm[7] += wq * y * (e * x);
                sm[8] += wq * x * (e * q2);
            }
        }
#pragma unroll
        for (int m = 0; m < 9; m++) r9[m] += double(sm[m]);
    }
    double r16[16];
#pragma unroll
    for (int m = 0; m < 16; m++) r16[m] = m < 9 ? r9[m] : 0.0;
    const double t = wave_reduce_scatter<16>(r16);
    if ((lane & 3) == 0 && (lane >> 2) < 9) red[wave * 9 + (lane >> 2)] = t;
    __syncthreads();
    double r[9];
#pragma unroll
    for (int m = 0; m < 9; m++) r[m] = ((red[m] + red[9 + m]) + red[18 + m]) + red[27 + m];
    const double rho = -r[0] / ((bcl[3] / kPi) * r[5]);
    const double Aw = rho * (bcl[3] / kPi), kbw = K / (2.0 * bcl[3]);
    const T AT = T(Aw), kbT = T(kbw), sc = T(len * dt);
#pragma unroll 4
    for (int iv = tid; iv < nv; iv += 256) {
        const T u = U[iv], v = V[iv];
        const T x = u * n1T + v * n2T, y = v * n1T - u * n2T, cu = x - Uw, cv = y - Vw;
        const bool in = x * rotT >= T(0);
        const T H = AT * texp(-lw * (cu * cu + cv * cv)), hk = h[iv], bk = h[nv + iv];
        T hW = in ? H : hk, bW = in ? H * kbT : bk;
        if constexpr (sizeof(T) == 4) {
            if (del) {
                hW = in ? H - S.mref[iv] : hk;
                bW = in ? H * kbT - S.mref[nv + iv] : bk;
            }
        }
        fo[iv] = x * hW * sc;
        fo[nv + iv] = x * bW * sc;
    }
    if (tid == 0) {
        const double m0 = r[0] + Aw * r[5], m1 = r[1] + Aw * r[6], m2 = r[2] + Aw * r[7], m3 = r[3] + Aw * r[8];
        const double m4 = r[4] + Aw * kbw * r[5];
        const double l1 = m1 * len * dt, l2 = m2 * len * dt;
        fwout[0] = m0 * len * dt;
        fwout[1] = l1 * n1 - l2 * n2;
        fwout[2] = l1 * n2 + l2 * n1;
        fwout[3] = (0.5 * m3 + 0.5 * m4) * len * dt;
        if (del) S.cref[(dir == 0 ? 0 : size_t(S.nx + 1) * S.ny) + fi] = len * dt;
    }
}

// the walls of cell c
template <class T> KBG_D void walls2d(const Solve2D& S, int c, double* red) {
    const int nx = S.nx, ny = S.ny, i = c % nx, j = c / nx;
    auto face = [&](int dir, int fi, int side) {
        __syncthreads();
        wall2d<T>(S, dir, fi, side, c, red);
    };
    if (i == 0) face(0, (nx + 1) * j, 0);
    if (i == nx - 1) face(0, (nx + 1) * j + nx, 1);
    if (j == 0) face(1, i, 2);
    if (j == ny - 1) face(1, i + nx * ny, 3);
}

// cells next to a wall come first, then the others
KBG_HD int wall_cells(int nx, int ny) { return nx < 3 || ny < 3 ? nx * ny : 2 * (nx + ny) - 4; }
KBG_D int cell_at(int nx, int ny, int k) {
    if (nx < 3 || ny < 3) return k;
    const int nw = 2 * (nx + ny) - 4;
    if (k >= nw) {
        k -= nw;
        return 1 + k % (nx - 2) + nx * (1 + k / (nx - 2));
    }
    if (k < nx) return k;
    if (k < 2 * nx) return k - nx + nx * (ny - 1);
    k -= 2 * nx;
    return (k & 1 ? nx - 1 : 0) + nx * (1 + k / 2);
}
KBG_HD int interior_faces(int nx, int ny) { return (nx - 1) * ny + nx * (ny - 1); }

// The interior face whose place in the flux arrays holds G of cell (i, j) (from 0): the x-face to its left, in
// the first column the y-face below it, and for the first cell the y-face below cell (1, 1), which no other
// cell takes.
KBG_D int g_face(int nx, int i, int j) { return i > 0 ? i + (nx + 1) * j : j > 0 ? nx * j : nx + 1; }

}  // namespace

// A call's first step: walls and interface chains.  pstart: prefix sums of ceil(interior faces / 256) + cells
// next to a wall
template <class T, int FLUX>
__global__ __launch_bounds__(256) void k_pre2d(const Solve2D* __restrict__ solves, const int* __restrict__ pstart, int nsolves) {
    __shared__ double red[36];
    const int g = blockIdx.x;
    if (g >= pstart[nsolves]) return;
    const int si = owner(pstart, nsolves, g);
    const Solve2D& S = solves[si];
    const int nif = interior_faces(S.nx, S.ny), b = g - pstart[si] - (nif + 255) / 256;
    if (b < 0) {
        const int f = (g - pstart[si]) * 256 + threadIdx.x;
        if (f < nif) face_chain<T, FLUX>(S, f);
    } else {
        walls2d<T>(S, cell_at(S.nx, S.ny, b), red);
    }
}

namespace {

// DPP lane exchanges within 8 (i -> 7 - i), 4 (i -> i ^ 2, i ^ 1) and 16 lanes (i -> i ^ 8)
template <int CTRL> KBG_D float dppx(float x) {
    return __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, x), CTRL, 0xf, 0xf, true));
}
template <int CTRL> KBG_D double dppx(double x) {
    const long long b = __builtin_bit_cast(long long, x);
    const int lo = __builtin_amdgcn_mov_dpp((int)b, CTRL, 0xf, 0xf, true), hi = __builtin_amdgcn_mov_dpp((int)(b >> 32), CTRL, 0xf, 0xf, true);
    return __builtin_bit_cast(double, ((long long)hi << 32) | (long long)(unsigned)lo);
}
// keep + the partner's send, where up lanes keep b and send a, the others keep a and send b
template <int CTRL, class T, class S = T> KBG_D S fold(bool up, T a, T b) {
    // pinned, or the selects become one load through a selected address and the sums go to scratch
    asm volatile("" : "+v"(a), "+v"(b));
    return S(up ? b : a) + S(dppx<CTRL>(up ? a : b));
}
// Sums of 8 values over 8 lanes, in FP64: lane l ends with value l & 7 of its group of 8.  Neighbouring lanes hold
// velocities of one sign, whose terms of the mass flux do not cancel: added in FP32 they left 1.4 to 1.7 times the
// error in rho of k_flux2d, whose lanes each add 8 velocities apart by 64 in FP32 (KFVS, one step of 61 x 60 cells
// x 600 velocities); in FP64 0.6 to 0.8 times.  UGKS FP32 64 x 64 cells x 32^2 velocities 61 us per step either way
// with the rows per tile chosen for each; 45 x 45 x 28^2 46.5 in FP32, 47.7 here.
template <class T> KBG_D double sum8(int lane, T (&v)[8]) {
    double a[4], b[2];
#pragma unroll
    for (int m = 0; m < 4; m++) a[m] = fold<0x141, T, double>((lane & 4) != 0, v[m], v[m + 4]);  // row_half_mirror
#pragma unroll
    for (int m = 0; m < 2; m++) b[m] = fold<0x4e>((lane & 2) != 0, a[m], a[m + 2]);  // quad_perm 2 3 0 1
    return fold<0xb1>((lane & 1) != 0, b[0], b[1]);                                  // quad_perm 1 0 3 2
}

// h and b of one velocity, as a vector: selects between elements of an array of structs would become loads
// through selected addresses, which send the array to scratch memory
template <class T> struct Vec2;
template <> struct Vec2<float> { using type = float __attribute__((ext_vector_type(2))); };
template <> struct Vec2<double> { using type = double __attribute__((ext_vector_type(2))); };
template <class T> using HB = typename Vec2<T>::type;

// SX, SY: the wavefront's velocities have u (v) < 0 (0), >= 0 (1): the flux takes the right or the left state;
// 2: both signs
template <class T, int FLUX, int SX, int SY> struct Tile {
    using Rec = const FaceRec<T>;  // in LDS: every lane reads the same words
    using H2 = HB<T>;
    rsrc_t fin;
    int voff, ohb, RSE;
    T xn[2], xt, xq[2], wq, hw;  // normal velocity (x-faces, y-faces), y-faces' u, n^2 (u^2 + v^2), weight, weight / 2
    T yt;                        // x-faces' v
    bool dx, dy;                 // u >= 0, v >= 0

    KBG_D H2 load(int c) const { return H2{bload((T*)0, fin, voff, c * RSE), bload((T*)0, fin, voff, c * RSE + ohb)}; }
    // difference quotient of two neighbouring cells
    static KBG_D H2 diff(H2 a, H2 c, T r) { return H2{(c.x - a.x) * r, (c.y - a.y) * r}; }
    // van Leer: (sL |sR| + |sL| sR) / (|sL| + |sR| + 1e-7), by reciprocal
    static KBG_D T lim1(T sL, T sR) {
        const T aL = fabs(sL), aR = fabs(sR);
        return quot(sL * aR + aL * sR, aL + aR + T(1e-7));
    }
    static KBG_D H2 lim(H2 l, H2 r) { return H2{lim1(l.x, r.x), lim1(l.y, r.y)}; }
    // one-sided where c
    static KBG_D H2 sel(bool c, H2 a, H2 b) { return H2{c ? a.x : b.x, c ? a.y : b.y}; }
    // flux through the face between cells a and c (DIR 0: x-face, 1: y-face) and, where SUMS, its moment
    // terms.  Mixed signs: both sides' polynomials are evaluated and the upwind one selected (a select of
    // scalar coefficients costs two moves each).
    template <int DIR, bool SUMS> KBG_D H2 flux(Rec* R, H2 fa, H2 sa, H2 fc, H2 sc, T* s) const {
        constexpr int SD = DIR == 0 ? SX : SY;
        const T M3 = R->M3;
        const T x = xn[DIR], q2 = xq[DIR], y = DIR == 0 ? yt : -xt;
        const bool dd = SD == 2 ? (DIR == 0 ? dx : dy) : SD == 1;
        constexpr int sd = SD == 0 ? 1 : 0;
        const T sh = dd ? sa.x : sc.x, sb = dd ? sa.y : sc.y;
        T d = R->s[sd].d;
        if constexpr (SD == 2) {
            const T dr = R->s[1].d;
            d = dd ? d : dr;
        }
        T eh = (dd ? fa.x : fc.x) + sh * d, eb = (dd ? fa.y : fc.y) + sb * d, Fh, Fb;
        if constexpr (FLUX == KCU) {
            const T cu = x - R->U, cv = y - R->V;
            const T g = gauss(R->nl * (cu * cu + cv * cv)) * R->P[0];
            Fh = x * (g + M3 * eh);
            Fb = x * (g * R->kb + M3 * eb);
        } else {
            const T rx = sizeof(T) == 4 ? R->rho * x + R->rhol * x : R->rho * x;
            eh -= rx * sh;
            eb -= rx * sb;
            if constexpr (FLUX == KFVS) {
                Fh = x * (M3 * eh);
                Fb = x * (M3 * eb);
            } else {
                const T cu = x - R->U, cv = y - R->V;
                const T H = gauss(R->nl * (cu * cu + cv * cv));
                T q = R->s[sd].q[0] + x * R->s[sd].q[1] + y * R->s[sd].q[2] + q2 * R->s[sd].q[3];
                T q3 = R->s[sd].q[3];
                if constexpr (SD == 2) {
                    const T qR = R->s[1].q[0] + x * R->s[1].q[1] + y * R->s[1].q[2] + q2 * R->s[1].q[3];
                    const T r3 = R->s[1].q[3];
                    q = dd ? q : qR;
                    q3 = dd ? q3 : r3;
                }
                const T p = R->P[0] + x * R->P[1] + y * R->P[2] + q2 * R->P[3];
                const T g = p + x * q;
                const T t3 = R->P[3] + x * q3;
                const T gb = R->kb * g + R->x2 * t3;
                Fh = x * (H * g + M3 * eh);
                Fb = x * (H * gb + M3 * eb);
            }
        }
        if constexpr (SUMS) {
            const T p = (wq * x) * eh;
            s[0] = p;
            s[1] = x * p;
            s[2] = y * p;
            s[3] = hw * (q2 * (x * eh) + x * eb);
        }
        // the flux is finished here and the next face's record read after this: the operands of several faces'
        // fluxes together would not fit
        asm volatile("" : "+v"(Fh), "+v"(Fb)::"memory");
        __builtin_amdgcn_sched_barrier(0);
        return H2{Fh, Fb};
    }
};

}  // namespace

namespace {

// one wavefront's march: tile columns i0 .. i0 + kTX - 1, rows j0 .. j1 - 1, one velocity per lane; sums:
// [row][pair of faces][8 groups of 8 lanes][8 values]
template <class T, int FLUX, bool KEEP, int SX, int SY>
KBG_D void tile_march(const Solve2D& S, int i0, int j0, int j1, int iv, bool live, T u, T v, int lane, const FaceRec<T>* XR, const FaceRec<T>* YR,
                      const T* RD, double* sums) {
    constexpr int E = sizeof(T);
    using H2 = HB<T>;
    using TL = Tile<T, FLUX, SX, SY>;
    using Rec = typename TL::Rec;
    const int nx = S.nx, ny = S.ny, nv = S.nv;
    const int RSE = 2 * nv * E, ohb = nv * E;
    const T nX = T(S.xgeo[0]), nY = T(S.ygeo[1]), wq = live ? ((const T*)S.wt)[iv] : T(0);  // one normal per direction
    const T xx = u * nX, yx = v * nX, xy = v * nY, yy = u * nY;
    const TL W{make_rsrc(S.f, unsigned(long(nx) * ny * RSE)), iv * E, ohb, RSE, {xx, xy}, yy, {xx * xx + yx * yx, xy * xy + yy * yy}, wq,
               T(0.5) * wq, yx, u >= T(0), v >= T(0)};
    const int voff = iv * E, vst = live ? voff : 0x7fffffff;  // stores of lanes past nv fall outside the buffers
    const rsrc_t xff = make_rsrc(S.xff, unsigned(long(nx + 1) * ny * RSE)), yff = make_rsrc(S.yff, unsigned(long(nx) * (ny + 1) * RSE));
    auto ldf = [&](rsrc_t r, int f) __attribute__((always_inline)) {
        return H2{bload((T*)0, r, voff, f * RSE), bload((T*)0, r, voff, f * RSE + ohb)};
    };
    auto stf = [&](rsrc_t r, int f, H2 x) __attribute__((always_inline)) {
        bstore(x.x, r, vst, f * RSE);
        bstore(x.y, r, vst, f * RSE + ohb);
    };
    // the row's owned faces, two at a time: x-faces to the left of each cell (pairs 0, 1), y-faces below it (2, 3)
    auto put = [&](int row, int pair, T(&s)[8]) __attribute__((always_inline)) { sums[(row * kTX + pair) * 64 + lane] = sum8(lane, s); };
    const bool inL = i0 > 0, inR = i0 + kTX < nx;
    H2 fB[kTX], fC[kTX], fN[kTX], qB[kTX], sB[kTX], FD[kTX];  // rows j, j + 1, j + 2, y-quotient j | j + 1, y-slope j, lower flux
    H2 D[kTX];                                               // a cell's left minus right flux
    T s8[8];                                                 // the moment terms of two faces
    const int c0 = i0 + nx * j0;
    static_for<kTX>([&](auto t) {
        fB[t] = W.load(c0 + t);
        fC[t] = W.load(j0 + 1 < ny ? c0 + t + nx : c0 + t);
    });
    static_for<kTX>([&](auto t) { qB[t] = W.diff(fB[t], fC[t], YR[2 * kTX + t].r); });  // 0 next to a wall
    if (j0 == 0) {
        static_for<kTX>([&](auto t) {
            sB[t] = qB[t];
            FD[t] = ldf(yff, i0 + t);
        });
        sums[2 * 64 + lane] = sums[3 * 64 + lane] = 0.0;
    } else {
        static_for<kTX>([&](auto t) {
            constexpr int o = (t & 1) * 4;
            const int c = c0 + t;
            const H2 fA = W.load(c - nx), fZ = W.load(j0 > 1 ? c - 2 * nx : c - nx);
            const H2 qA = W.diff(fA, fB[t], YR[kTX + t].r), qZ = W.diff(fZ, fA, YR[t].r);
            sB[t] = W.sel(j0 + 1 == ny, qA, W.lim(qA, qB[t]));
            FD[t] = W.template flux<1, true>(YR + kTX + t, fA, W.sel(j0 == 1, qA, W.lim(qZ, qA)), fB[t], sB[t], s8 + o);
            if constexpr (KEEP) stf(yff, i0 + t + nx * j0, FD[t]);
            if constexpr (t & 1) put(0, 2 + t / 2, s8);
        });
    }
    for (int j = j0; j < j1; j++) {
        const int row = j - j0, cj = i0 + nx * j;
        Rec* xj = XR + row * (kTX + 3) + 1;
        const H2 xm2 = W.load(i0 > 1 ? cj - 2 : cj), xm1 = W.load(inL ? cj - 1 : cj);
        const H2 xp0 = W.load(inR ? cj + kTX : cj), xp1 = W.load(i0 + kTX + 1 < nx ? cj + kTX + 1 : cj);
        static_for<kTX>([&](auto t) { fN[t] = W.load(j + 2 < ny ? cj + t + 2 * nx : cj + t); });
        // ---- x: faces 0 .. kTX of the tile; the left cell, its slope and the quotient across the face
        // (records of walls hold zeros)
        H2 qa, sa, F;
        H2 q1 = W.diff(fB[0], fB[1], xj[1].r);
        if (inL) {
            qa = W.diff(xm1, fB[0], xj[0].r);
            sa = W.sel(i0 == 1, qa, W.lim(W.diff(xm2, xm1, xj[i0 == 1 ? 0 : -1].r), qa));
            const H2 sc = W.lim(qa, q1);
            F = W.template flux<0, true>(xj, xm1, sa, fB[0], sc, s8);
            if constexpr (KEEP) stf(xff, i0 + (nx + 1) * j, F);
            sa = sc;
        } else {
            F = ldf(xff, (nx + 1) * j);
            s8[0] = s8[1] = s8[2] = s8[3] = T(0);
            sa = q1;  // the first cell's one-sided slope
        }
        D[0] = F;
        qa = q1;
        static_for<kTX - 1>([&](auto tm) {
            constexpr int t = tm + 1, o = (t & 1) * 4;  // the face between cells t - 1 and t
            H2 fd, qc, sc;
            if constexpr (t + 1 < kTX) fd = fB[t + 1];
            else fd = xp0;
            qc = W.diff(fB[t], fd, xj[t + 1].r);
            sc = W.lim(qa, qc);
            if constexpr (t == kTX - 1) sc = W.sel(!inR, qa, sc);
            F = W.template flux<0, true>(xj + t, fB[t - 1], sa, fB[t], sc, s8 + o);
            if constexpr (KEEP) stf(xff, i0 + t + (nx + 1) * j, F);
            D[t - 1] -= F;
            D[t] = F;
            sa = sc;
            qa = qc;
            if constexpr (t & 1) put(row, t / 2, s8);
        });
        if (inR) {
            const H2 sc = W.sel(i0 + kTX + 1 == nx, qa, W.lim(qa, W.diff(xp0, xp1, xj[i0 + kTX + 1 == nx ? kTX : kTX + 1].r)));
            F = W.template flux<0, false>(xj + kTX, fB[kTX - 1], sa, xp0, sc, s8);
        } else {
            F = ldf(xff, nx + (nx + 1) * j);
        }
        D[kTX - 1] -= F;
        // ---- y: the face above each cell, G, and the roll to the next row
        if (j + 1 < ny) {
            const bool last = j + 2 == ny;
            Rec* yj = YR + (row + 2) * kTX;
            static_for<kTX>([&](auto t) {
                constexpr int o = (t & 1) * 4;
                const H2 qC = W.diff(fC[t], fN[t], yj[kTX + t].r), sC = W.sel(last, qB[t], W.lim(qB[t], qC));
                const H2 FU = W.template flux<1, true>(yj + t, fB[t], sB[t], fC[t], sC, s8 + o);
                if constexpr (KEEP)
                    if (j + 1 < j1) stf(yff, i0 + t + nx * (j + 1), FU);
                D[t] += FD[t] - FU;
                FD[t] = FU;
                qB[t] = qC;
                sB[t] = sC;
                if constexpr (t & 1)
                    if (j + 1 < j1) put(row + 1, 2 + t / 2, s8);
            });
        } else {
            static_for<kTX>([&](auto t) { D[t] += FD[t] - ldf(yff, i0 + t + nx * ny); });
        }
        static_for<kTX>([&](auto t) {
            const T r = RD[row * kTX + t];
            if constexpr (!KEEP) {
                const H2 g{fB[t].x + D[t].x * r, fB[t].y + D[t].y * r};
                if (t == 0 && !inL) stf(yff, g_face(nx, 0, j), g);
                else stf(xff, g_face(nx, i0 + t, j), g);
            }
            fB[t] = fC[t];
            fC[t] = fN[t];
        });
    }
}

}  // namespace

// tstart: prefix sums of the solves' workgroups (tile columns x tile rows of ty cells x chunks of 256
// velocities, tiles fastest: neighbouring tiles share an XCD's L2); KEEP: store the face fluxes.  The last
// tile column ends at the last cell, where nx is no multiple of kTX overlapping its neighbour (both compute
// the shared cells, with the same results).
template <class T, int FLUX, bool KEEP>
__global__ __launch_bounds__(256, sizeof(T) == 4 ? 4 : 2) void k_tile2d(const Solve2D* __restrict__ solves, const int* __restrict__ tstart, int nsolves,
                                                                                int ty) {
    // face records of the tile (x-faces i0 - 1 .. i0 + kTX + 1 of its rows, y-faces of rows j0 - 1 .. j1 + 1), 1 / (dx dy),
    // sums [4 wavefronts][rows][kTX pairs of faces][64]
    extern __shared__ double tile_lds[];
    const int g = xcd_order();
    if (g >= tstart[nsolves]) return;
    const int si = owner(tstart, nsolves, g);
    const Solve2D& S = solves[si];
    const int nx = S.nx, ny = S.ny, nv = S.nv;
    const Tile2D B = bufs<T>(S);
    const int ntx = (nx + kTX - 1) / kTX, nty = (ny + ty - 1) / ty;
    const int b = g - tstart[si], tile = b % (ntx * nty), chunk = b / (ntx * nty);
    const int i0 = min(tile % ntx * kTX, nx - kTX), j0 = tile / ntx * ty, j1 = min(j0 + ty, ny);
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int rows = j1 - j0, nws = rows * kTX * 64;  // sums per wavefront
    FaceRec<T>* XR = reinterpret_cast<FaceRec<T>*>(tile_lds);
    FaceRec<T>* YR = XR + ty * (kTX + 3);
    T* RD = reinterpret_cast<T*>(YR + (ty + 3) * kTX);
    double* sums = reinterpret_cast<double*>(RD + ty * kTX);
    double* ws = sums + (size_t)wave * nws;
    {
        constexpr int P = sizeof(FaceRec<T>) / 16;
        const int nX = rows * (kTX + 3), nR = nX + (rows + 3) * kTX;
        for (int k = tid; k < nR * P; k += 256) {
            const int rec = k / P, part = k % P;
            if (rec < nX) {
                const int r = rec / (kTX + 3), i = min(max(i0 + rec % (kTX + 3) - 1, 0), nx);
                ((uint4*)XR)[k] = ((const uint4*)B.xrec)[((size_t)i + size_t(nx + 1) * (j0 + r)) * P + part];
            } else {
                const int q = rec - nX, j = min(max(j0 - 1 + q / kTX, 0), ny);
                ((uint4*)YR)[q * P + part] = ((const uint4*)B.yrec)[((size_t)(i0 + q % kTX) + size_t(nx) * j) * P + part];
            }
        }
        for (int k = tid; k < rows * kTX; k += 256) RD[k] = ((const T*)B.rds)[i0 + k % kTX + nx * (j0 + k / kTX)];
    }
    __syncthreads();
    if (chunk * 256 + wave * 64 < nv) {
        const int iv0 = chunk * 256 + tid, iv = B.vperm[min(iv0, nv - 1)];
        const T u = ((const T*)S.u)[iv], v = ((const T*)S.v)[iv];
        const unsigned long long bx = __ballot(u >= T(0)), by = __ballot(v >= T(0));
        const bool mixed = (bx != 0ull && ~bx != 0ull) || (by != 0ull && ~by != 0ull), live = iv0 < nv;
#define KBG_M(SX, SY) tile_march<T, FLUX, KEEP, SX, SY>(S, i0, j0, j1, iv, live, u, v, lane, XR, YR, RD, ws)
        if (mixed) KBG_M(2, 2);
        else if (bx == 0ull && by == 0ull) KBG_M(0, 0);
        else if (by == 0ull) KBG_M(1, 0);
        else if (bx == 0ull) KBG_M(0, 1);
        else KBG_M(1, 1);
#undef KBG_M
    } else {
        for (int k = lane; k < nws; k += 64) ws[k] = 0.0;
    }
    __syncthreads();
    const size_t FX = size_t(nx + 1) * ny, F = FX + size_t(nx) * (ny + 1);
    for (int k = tid; k < 2 * kTX * rows * 4; k += 256) {
        // face slots: [row][x-faces | lower y-faces][column]
        const int m = k & 3, sl = k >> 2, t = sl % kTX, ydir = (sl / kTX) & 1, j = j0 + sl / (2 * kTX);
        double q = 0.0;
        for (int w = 0; w < 4; w++) {
            const double* p = sums + (size_t)w * nws + (sl >> 1) * 64 + (sl & 1) * 4 + m;
#pragma unroll
            for (int g8 = 0; g8 < 8; g8++) q += p[g8 * 8];
        }
        const size_t f = ydir ? FX + (i0 + t) + size_t(nx) * j : size_t(i0 + t) + size_t(nx + 1) * j;
        B.psum[(size_t(chunk) * F + f) * 4 + m] = q;
    }
}

// the relaxation's coefficients of a cell as k_chain2d leaves them, in the storage type
namespace {
template <class T> struct alignas(16) CellRec {
    T rT, inv, An, ln, Un, Vn, kbn, Cu, Cv, pad[7];
};
static_assert(sizeof(CellRec<double>) == kCellT * 8 && sizeof(CellRec<float>) == kCellT * 4, "CellRec");
}  // namespace

// update!'s macroscopic part of every cell (all are stepped between Maxwell walls), 16 lanes per cell: lane
// = (face L R D U) 4 + moment.  rows: write the residual rows; keep: store the faces' moments and
// coefficients of Mr (each cell its left and lower face).  Done by each cell's workgroup between its loads and
// stores (k_cell2d) this chain is most of that kernel: 444 us for the 16384 cells x 48^2 velocities of FP32.
template <class T>
__global__ __launch_bounds__(256) void k_chain2d(const Solve2D* __restrict__ solves, const int* __restrict__ wg0, int nsolves, int rows,
                                                 int keep) {
    const int lane = threadIdx.x & 63, g = blockIdx.x * 16 + (threadIdx.x >> 4);
    const bool act = g < wg0[nsolves];  // every lane takes part in the exchanges
    const int gi = act ? g : 0, si = owner(wg0, nsolves, gi), c = gi - wg0[si];
    const Solve2D& S = solves[si];
    const int nx = S.nx, ny = S.ny, i = c % nx, j = c / nx;
    const bool del = sizeof(T) == 4 && S.delta;
    const int fc = (lane >> 2) & 3, m = lane & 3, b0 = lane & 48;
    const size_t FX = size_t(nx + 1) * ny, F = FX + size_t(nx) * (ny + 1);
    const bool xf = fc < 2;
    const int fi = fc == 0 ? i + (nx + 1) * j : fc == 1 ? i + 1 + (nx + 1) * j : fc == 2 ? i + nx * j : i + nx * (j + 1);
    const bool wall = fc == 0 ? i == 0 : fc == 1 ? i == nx - 1 : fc == 2 ? j == 0 : j == ny - 1;
    const Tile2D B = bufs<T>(S);
    const double* fr = (xf ? B.xfrec : B.yfrec) + (size_t)fi * 8;
    const double* geo = (xf ? S.xgeo : S.ygeo) + (size_t)fi * 3;
    const double n1 = geo[0], n2 = geo[1];
    double q = 0.0, cf;
    if (wall) {
        q = (xf ? S.xfw : S.yfw)[(size_t)fi * 4 + m];
        cf = del ? S.cref[(xf ? 0 : FX) + fi] : 0.0;
    } else {
        cf = fr[4];
        const double* ps = B.psum + ((xf ? size_t(fi) : FX + fi)) * 4 + m;
        const int nch = (S.nv + 255) / 256;
#pragma unroll 4
        for (int k = 0; k < nch; k++) q += ps[size_t(k) * F * 4];
        if (del) {
            // the sums ran over departures: the reference Maxwellian's share from its moments
            const double* mm = S.mmom;
            double r;
            if (m == 0) r = n1 * mm[0] + n2 * mm[1];
            else if (m == 1) r = n1 * n1 * mm[2] + 2.0 * n1 * n2 * mm[3] + n2 * n2 * mm[4];
            else if (m == 2) r = (n1 * n1 - n2 * n2) * mm[3] + n1 * n2 * (mm[4] - mm[2]);
            else r = 0.5 * (n1 * (mm[5] + mm[7]) + n2 * (mm[6] + mm[8]) + n1 * mm[9] + n2 * mm[10]);
            q += r;
        }
        q = fr[m] + cf * q;
    }
    const double o = __shfl_xor(q, 3, 64);  // moments 1 and 2 change places
    const double fw = wall ? q : m == 1 ? q * n1 - o * n2 : (m == 2 ? o * n2 + q * n1 : q);
    if (act && keep && !wall && (fc == 0 || fc == 2)) {
        (xf ? S.xfw : S.yfw)[(size_t)fi * 4 + m] = fw;
        if (del && m == 0) S.cref[(xf ? 0 : FX) + fi] = cf;
    }
    const double ds = S.dx[c] * S.dy[c];
    // sum over the faces of a quantity of this lane's moment: L - R + D - U
    auto net = [&](double a) {
        return __shfl(a, b0 + m, 64) - __shfl(a, b0 + 4 + m, 64) + __shfl(a, b0 + 8 + m, 64) - __shfl(a, b0 + 12 + m, 64);
    };
    const double wom = S.w[(size_t)c * 4 + m], wnm = wom + net(fw) / ds;
    // the reference Maxwellian's share of the four fluxes, sum of +-cf (n1 u + n2 v) / ds
    const double cu = net(cf * n1) / ds, cv = net(cf * n2) / ds;
    double wn[4], pn[4];
#pragma unroll
    for (int n = 0; n < 4; n++) wn[n] = __shfl(wnm, b0 + n, 64);
    conserve_prim<4>(wn, S.gam, pn);
    const double r = S.dt / vhs_tau(pn[0], pn[3], S.mu, S.om);
    if (!act) return;
    if ((lane & 15) == 0) {
        flag_health(S.health, prim_health<4>(pn));
        CellRec<T>& k = ((CellRec<T>*)B.crec)[c];
        k.rT = T(r);
        k.inv = T(1.0 / (1.0 + r));
        k.An = T(pn[0] * (pn[3] / kPi));
        k.ln = T(pn[3]);
        k.Un = T(pn[1]);
        k.Vn = T(pn[2]);
        k.kbn = T(S.K / (2.0 * pn[3]));
        k.Cu = T(cu);
        k.Cv = T(cv);
    }
    if (fc == 0) {
        const double p = m == 0 ? pn[0] : m == 1 ? pn[1] : m == 2 ? pn[2] : pn[3];
        S.w[(size_t)c * 4 + m] = wnm;
        S.prim[(size_t)c * 4 + m] = p;
        if (rows && S.rcell) {
            double* rr = S.rcell + (size_t)c * 16;
            const bool inner = i > 0 && i < nx - 1 && j > 0 && j < ny - 1;
            rr[(inner ? 0 : 2) * 4 + m] = (wnm - wom) * (wnm - wom);
            rr[(inner ? 1 : 3) * 4 + m] = fabs(wnm);
            rr[(inner ? 2 : 0) * 4 + m] = 0.0;
            rr[(inner ? 3 : 1) * 4 + m] = 0.0;
        }
    }
}

// update!'s relaxation f = (G + (dt / tau) M) / (1 + dt / tau): a workgroup per cell and 1024 velocities (next
// to a wall: per cell).  NEXT: workgroups before them form the next step's interface chains, and those next
// to a wall its wall fluxes.  KEEP: the flux arrays hold the face fluxes, from which G is formed here.  Bound by
// memory: 604 MB in 124 us at 16384 cells x 48^2 velocities in FP32.
template <class T, int FLUX, bool NEXT, bool KEEP>
__global__ __launch_bounds__(256, NEXT || KEEP ? 4 : 6) void k_relax2d(const Solve2D* __restrict__ solves, const int* __restrict__ rstart, int nsolves) {
    constexpr int VPT = 4;
    __shared__ double red[NEXT ? 36 : 1];
    const int g = KEEP ? xcd_order() : int(blockIdx.x);  // KEEP: neighbouring cells' shared faces from one L2
    if (g >= rstart[nsolves]) return;
    const int si = owner(rstart, nsolves, g);
    const Solve2D& S = solves[si];
    const int nx = S.nx, ny = S.ny, nv = S.nv, per = (nv + 1023) / 1024, tid = threadIdx.x;
    const int nif = interior_faces(nx, ny), nfb = (nif + 255) / 256, nw = wall_cells(nx, ny);
    int b = g - rstart[si] - nfb;
    if (b < 0) {
        if constexpr (NEXT) {
            const int f = (b + nfb) * 256 + tid;
            if (f < nif) face_chain<T, FLUX>(S, f);
        }
        return;
    }
    const bool wall = b < nw;
    const int c = cell_at(nx, ny, wall ? b : nw + (b - nw) / per);
    const bool del = sizeof(T) == 4 && S.delta;
    const int i = c % nx, j = c / nx;
    const T* __restrict__ G = (const T*)(i > 0 ? S.xff : S.yff) + (size_t)g_face(nx, i, j) * 2 * nv;
    const T* __restrict__ xl = (const T*)S.xff + (size_t)(i + (nx + 1) * j) * 2 * nv;
    const T* __restrict__ yd = (const T*)S.yff + (size_t)(i + nx * j) * 2 * nv;
    const Tile2D B = bufs<T>(S);
    const T rds = KEEP ? ((const T*)B.rds)[c] : T(0);
    T* h = (T*)S.f + (size_t)c * 2 * nv;
    auto g_of = [&](int o) {
        if constexpr (KEEP) {
            T d = xl[o] - xl[2 * nv + o];
            d += yd[o] - yd[size_t(nx) * 2 * nv + o];
            return h[o] + d * rds;
        } else {
            return G[o];
        }
    };
    const T* __restrict__ U = (const T*)S.u;
    const T* __restrict__ V = (const T*)S.v;
    const float* __restrict__ R = S.mref;
    const CellRec<T> K = ((const CellRec<T>*)B.crec)[c];
    for (int v0 = wall ? 0 : (b - nw) % per * 1024; v0 < nv; v0 += 1024) {
        T gh[VPT], gb[VPT], u[VPT], v[VPT], rh[VPT], rb[VPT];
#pragma unroll
        for (int k = 0; k < VPT; k++) {
            const int iv = min(v0 + tid + 256 * k, nv - 1);
            gh[k] = g_of(iv);
            gb[k] = g_of(nv + iv);
            u[k] = U[iv];
            v[k] = V[iv];
            if constexpr (sizeof(T) == 4) {
                rh[k] = del ? R[iv] : 0.f;
                rb[k] = del ? R[nv + iv] : 0.f;
            }
        }
#pragma unroll
        for (int k = 0; k < VPT; k++) {
            const int iv = v0 + tid + 256 * k;
            if (iv >= nv) break;
            const T cu = u[k] - K.Un, cv = v[k] - K.Vn;
            T MH = K.An * texp(-K.ln * (cu * cu + cv * cv)), MB = MH * K.kbn;
            if constexpr (sizeof(T) == 4) {
                // departures: they relax toward M - Mr, and Mr's share of the face fluxes is added
                const T jr = K.Cu * u[k] + K.Cv * v[k];
                gh[k] += jr * rh[k];
                gb[k] += jr * rb[k];
                MH -= rh[k];
                MB -= rb[k];
            }
            h[iv] = (gh[k] + K.rT * MH) * K.inv;
            h[nv + iv] = (gb[k] + K.rT * MB) * K.inv;
        }
        if (!wall) return;
    }
    if constexpr (NEXT) walls2d<T>(S, c, red);  // each thread reads back the values it stored
}

int pre2d_wgs(int nx, int ny) { return (interior_faces(nx, ny) + 255) / 256 + wall_cells(nx, ny); }
int relax2d_wgs(int nx, int ny, int nv) { return pre2d_wgs(nx, ny) + (nx * ny - wall_cells(nx, ny)) * ((nv + 1023) / 1024); }
// Fewer rows repeat the two faces' and slopes' work of the rows around a tile more often (about 1.6 rows' work per
// tile), more rows leave too few workgroups to overlap one's waits with another's work.  FP32 holds 4 workgroups per CU
// (LDS, up to 4 rows): the rows whose rounds of 1024 workgroups times their work come out least.  us per step at 1 / 2 /
// 3 / 4 rows: UGKS 24 x 24 cells x 16^2 velocities 28 / 30 / 33 / 36, 45 x 45 x 28^2 53 / 50 / 48 / 51, 64 x 64 x 24^2 59 / 54
// / 58 / 53 (3072 / 1536 / 1056 / 768 workgroups), 64 x 64 x 32^2 69 / 61 / 64 / 61, 100 x 100 x 40^2 247 / 218 / 214 / 218, 128
// x 128 x 48^2 605 / 510 / 496 / 488.  FP64 (2 workgroups per CU) UGKS at 1 / 2 / 3 / 4 / 6 rows: 64 x 64 x 32^2 121 / 102 /
// 103 / 95 / 103, 100 x 100 x 40^2 583 / 500 / 464 / 451 / 435.
int tile2d_rows(bool fp64, const long* wgs) {
    if (fp64) return wgs[1] <= 256 ? 1 : wgs[1] <= 1024 ? 2 : wgs[1] <= 3072 ? 3 : wgs[1] <= 12288 ? 4 : 6;
    int best = 1;
    double least = 0.0;
    for (int k = 1; k <= 4; k++) {
        const double cost = double((wgs[k] + 1023) / 1024) * (k + 1.6);
        if (k == 1 || cost < least) best = k, least = cost;
    }
    return best;
}

// records, 1 / (dx dy) and sums of a tile of ty rows
template <class T> constexpr size_t tile2d_lds(int ty) {
    return (size_t(ty) * (kTX + 3) + size_t(ty + 3) * kTX) * sizeof(FaceRec<T>) + size_t(ty) * kTX * (sizeof(T) + 4 * 64 * sizeof(double));
}
static_assert(tile2d_lds<double>(kTile2dRows) <= 65536, "dynamic LDS a kernel may use without asking");

template <class T, int FLUX>
static hipError_t launch_tile_t(int ty, const Solve2D* d_solves, const int* d_pref, int n, const int* totals, int rows, int first, int last,
                                hipStream_t st) {
    // k_relax2d with the next step's walls and chains holds 4 wavefronts per SIMD, alone 8: sharing the launch
    // pays while the launch is short (us per step, shared / not: 64 x 64 x 32^2 FP32 60 / 66, FP64 95 / 105, 100 x
    // 100 x 40^2 FP64 439 / 451, 128 x 128 x 48^2 FP32 502 / 487)
    const bool share = totals[3] <= 32768;
    if (first || !share) hipLaunchKernelGGL((k_pre2d<T, FLUX>), dim3(totals[0]), dim3(256), 0, st, d_solves, d_pref, n);
    const size_t lds = tile2d_lds<T>(ty);
    if (last) hipLaunchKernelGGL((k_tile2d<T, FLUX, true>), dim3(totals[1]), dim3(256), lds, st, d_solves, d_pref + (n + 1), n, ty);
    else hipLaunchKernelGGL((k_tile2d<T, FLUX, false>), dim3(totals[1]), dim3(256), lds, st, d_solves, d_pref + (n + 1), n, ty);
    hipLaunchKernelGGL(k_chain2d<T>, dim3((totals[2] + 15) / 16), dim3(256), 0, st, d_solves, d_pref + 2 * (n + 1), n, rows, last);
    const dim3 gr(totals[3]), b(256);
    const int* rstart = d_pref + 3 * (n + 1);
    if (last) hipLaunchKernelGGL((k_relax2d<T, KFVS, false, true>), gr, b, 0, st, d_solves, rstart, n);
    else if (share) hipLaunchKernelGGL((k_relax2d<T, FLUX, true, false>), gr, b, 0, st, d_solves, rstart, n);
    else hipLaunchKernelGGL((k_relax2d<T, KFVS, false, false>), gr, b, 0, st, d_solves, rstart, n);
    return hipGetLastError();
}

hipError_t launch_tile2d(bool fp64, int flux, int ty, const Solve2D* d_solves, const int* d_pref, int n, const int* totals, int rows, int first,
                         int last, hipStream_t st) {
    if (ty < 1 || ty > kTile2dRows) return hipErrorInvalidValue;
#define KBG_T(T, FL) return launch_tile_t<T, FL>(ty, d_solves, d_pref, n, totals, rows, first, last, st)
    if (fp64) {
        if (flux == KFVS) KBG_T(double, KFVS);
        if (flux == KCU) KBG_T(double, KCU);
        KBG_T(double, UGKS);
    }
    if (flux == KFVS) KBG_T(float, KFVS);
    if (flux == KCU) KBG_T(float, KCU);
    KBG_T(float, UGKS);
#undef KBG_T
}

}  // namespace kbg
