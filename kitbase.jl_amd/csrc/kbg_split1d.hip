// kbg_split1d.hip -- the fused 1D time step of small FP64 KCU / UGKS launches, velocities split over workgroups.
//
// k_sweep1d keeps a segment of 60 cells in one workgroup, because the cells' FP64 chain needs the face moments
// of all velocities: a solve of a few segments runs on as many CUs, and its step lasts as long as one CU takes
// for a segment's KCU / UGKS fluxes (35.7 us for 400 cells x 101 velocities, h and b).  Here a wavefront holds 8
// velocities of a segment and every step is one launch: a wavefront
//   adds up the moment sums the step before left, runs the cells' chain (w, prim, the relaxation's
//     coefficients) and the faces' chain of its 64 cells, the same in all wavefronts of a segment;
//   relaxes its velocities' transport update G of the step before into f as it loads them, and goes on with
//     slopes, fluxes, moment sums and the next G.
// G takes the f buffers in turn; a last launch (END) relaxes the last one in place.  The 64 lanes of a segment hold
// two halo cells to its left and three to its right (the right face of lane 62 is lane 63's left one).
//
// Every value is formed by k_sweep1d's operations, the sums in its order (chunks of 8 velocities within the
// velocities of one of its wavefronts, then these), so the results are the same, bit for bit, whichever kernel a
// batch takes (kbg_api.hip has the rule).  Bound by the latency of the two chains: 400 cells x 101 velocities,
// h and b, UGKS + Shakhov 35.7 us per step with k_sweep1d, 18.5 here; KCU 23.3 and 16.5.
#include "kbg_sweep.h"

namespace kbg {

namespace {

template <int NF> struct SplitCell {
    double An, nl2, Un, inv, kbn, Ao, nlo2, Uo, lo2, kbo;  // the relaxation of k_sweep1d's pass 2
};

// values per face and parity in psum: every chunk's NR sums, then fw0[3], m3, m4
template <int NF, int FLUX> constexpr int split_rows(int nch) { return nch * SweepCfg<double, NF, FLUX>::NR + 5; }

// w of the lane's cell from the step before (its w and the sums it left), and the cell's relaxation
template <int NF, int FLUX, bool SHAK>
KBG_D void split_cell(const Solve1D& S, const double* __restrict__ P, int kc, int i, double rdx64, bool upd_any, double (&w)[3], double (&pn)[3],
                      SplitCell<NF>& o) {
    using C = SweepCfg<double, NF, FLUX>;
    constexpr int NR = C::NR, NRAW = C::NRAW;
    const int nv = S.nv, nch = (nv + kVChunk - 1) / kVChunk;
    const int gch = sweep_item_vw(nv, sweep_nw(true, NF, nv)) / kVChunk;
    const size_t np = S.np;
    double tot[NR], a[NR];
#pragma unroll
    for (int m = 0; m < NR; m++) tot[m] = a[m] = 0.0;
    // the loads of four chunks before their adds: left to the compiler, BGK's variants waited for each load
    // (2 solves of 1700 cells x 128 velocities UGKS 43.7 us per step, 23.0 here)
    const gptr<const double> Pg = to_global(P);
    int left = gch;
    for (int c0 = 0; c0 < nch; c0 += 4) {
        double v[4][NR];
#pragma unroll
        for (int k = 0; k < 4; k++)
#pragma unroll
            for (int m = 0; m < NR; m++) v[k][m] = Pg[size_t(min(c0 + k, nch - 1) * NR + m) * np + kc];
#pragma unroll
        for (int k = 0; k < 4; k++)
#pragma unroll
            for (int m = 0; m < NR; m++) asm volatile("" : "+v"(v[k][m]));  // not sunk into the branches below
#pragma unroll
        for (int k = 0; k < 4; k++) {
            if (c0 + k >= nch) break;
#pragma unroll
            for (int m = 0; m < NR; m++) a[m] += v[k][m];
            if (--left == 0 || c0 + k == nch - 1) {
#pragma unroll
                for (int m = 0; m < NR; m++) {
                    tot[m] += a[m];
                    a[m] = 0.0;
                }
                left = gch;
            }
        }
    }
    double fw0[3];
#pragma unroll
    for (int m = 0; m < 3; m++) fw0[m] = P[size_t(nch * NR + m) * np + kc];
    const double m3 = P[size_t(nch * NR + 3) * np + kc], m4 = P[size_t(nch * NR + 4) * np + kc];
    double fwl[3];
    if constexpr (FLUX == KCU) {
        fwl[0] = fw0[0] + m3 * tot[0];
        fwl[1] = fw0[1] + m3 * tot[1];
        fwl[2] = fw0[2] + m3 * 0.5 * (NF == 2 ? tot[2] + tot[3] : tot[2]);
    } else {
        fwl[0] = fw0[0] + (m3 * tot[0] - m4 * tot[1]);
        fwl[1] = fw0[1] + (m3 * tot[2] - m4 * tot[3]);
        fwl[2] = fw0[2] + (m3 * 0.5 * tot[4] - m4 * 0.5 * tot[5]);
    }
    double po[3] = {1.0, 0.0, 1.0}, wn[3];
    if (SHAK) conserve_prim<3>(w, S.gam, po);
#pragma unroll
    for (int m = 0; m < 3; m++) wn[m] = w[m] + (fwl[m] - shl1(fwl[m])) * rdx64;
    conserve_prim<3>(wn, S.gam, pn);
    const double rT = relax_ratio<double>(pn[0], pn[2], S.mu, S.om, S.dt);
    o.inv = 1.0 / (1.0 + rT);
    const double A1 = pn[0] * sqrt(pn[2] / kPi), rTi = rT * o.inv;
    o.nl2 = -pn[2] * kLog2e;
    o.Un = pn[1];
    o.kbn = NF == 2 ? S.K / (2.0 * pn[2]) : 0.0;
    o.An = A1 * rTi;
    o.Ao = o.nlo2 = o.Uo = o.lo2 = o.kbo = 0.0;
    if (SHAK && i > 1 && i < S.nx) {  // boundary cells relax with BGK (update_boundary.jl)
        const double q = 0.5 * tot[NRAW];
        const double pre = 0.8 * (1.0 - S.Pr) * (po[2] * po[2]) / po[0] * q * rTi;
        o.Uo = po[1];
        o.lo2 = 2.0 * po[2];
        o.kbo = NF == 2 ? S.K / (2.0 * po[2]) : 0.0;
        o.Ao = po[0] * sqrt(po[2] / kPi) * pre;
        o.nlo2 = -po[2] * kLog2e;
    }
#pragma unroll
    for (int m = 0; m < 3; m++) w[m] = upd_any ? wn[m] : w[m];
}

// f of one velocity from its G
template <int NF, bool SHAK> KBG_D void split_relax(const SplitCell<NF>& o, double K, double u, double (&f)[NF]) {
    const double cn = u - o.Un;
    double MH = o.An * texp2(o.nl2 * (cn * cn));
    double MB = MH * o.kbn;
    if constexpr (SHAK) {
        const double c = u - o.Uo;
        const double Mo = o.Ao * texp2(o.nlo2 * (c * c));
        const double co = u - o.Uo, c2 = co * co;
        const double t = co * Mo;  // Mo carries the prefactor
        if constexpr (NF == 1) {
            MH += t * (o.lo2 * c2 - 5.0);
        } else {
            MH += t * (o.lo2 * c2 + K - 5.0);
            MB += (t * o.kbo) * (o.lo2 * c2 + K - 3.0);
        }
    }
    f[0] = f[0] * o.inv + MH;
    if constexpr (NF == 2) f[1] = f[1] * o.inv + MB;
}

// par: launches of the call so far; END: relax the last G in place
template <int NF, int FLUX, int LIMK, bool SHAK, bool END>
KBG_D void split1d(const Solve1D& S, const WorkItem& wi, int par, int chunk, int lane) {
    using C = SweepCfg<double, NF, FLUX>;
    constexpr int NR = C::NR, CH = kVChunk;
    const int nx = S.nx, ng = S.ng, nv = S.nv, N = nx + 2 * ng, nch = (nv + CH - 1) / CH;
    const size_t np = S.np;
    const int in = (S.cur + par) & 1, vb = chunk * CH, lk = S.limiter;
    const unsigned fbytes = (unsigned)((size_t)NF * nv * np * 8);
    const rsrc_t fin = make_rsrc(S.f[in], fbytes), fout = make_rsrc(S.f[END ? in : in ^ 1], fbytes);
    const int rowb = (int)(np * 8);
    const double dt = S.dt, K = S.K;
    const int k = wi.c0 - 1 + ng - 2 + lane, i = k - ng + 1;
    const int kc = k < 0 ? 0 : (k >= N ? N - 1 : k), voff = k * 8;
    using VC = const __attribute__((address_space(4))) VChunk<double>;
    VC& ch = ((VC*)S.vtab)[chunk];
    // this wavefront's f or G, on its way while the chains run
    double fr[NF][CH];
#pragma unroll
    for (int j = 0; j < CH; j++)
#pragma unroll
        for (int q = 0; q < NF; q++) fr[q][j] = bload((double*)nullptr, fin, voff, (q * nv + vb + j) * rowb);
    const double d0 = S.dx[kc], dm = S.dx[kc > 0 ? kc - 1 : 0], dp = S.dx[kc < N - 1 ? kc + 1 : N - 1];
    const bool slope_on = S.interp2 && i >= S.slope_lo && i <= S.slope_hi && k >= 0 && k < N;
    const double rL = slope_on ? 1.0 / (0.5 * (dm + d0)) : 0.0, rR = slope_on ? 1.0 / (0.5 * (d0 + dp)) : 0.0;
    const double dxh = 0.5 * d0, rdx = 1.0 / d0;
    const bool own = lane >= 2 && lane < 2 + kSplitOut && i >= wi.c0 && i <= wi.c1, upd_any = i >= S.upd_lo && i <= S.upd_hi;
    double w[3], pn[3];
    const double* win = S.w[par > 0 ? in ^ 1 : in];
#pragma unroll
    for (int m = 0; m < 3; m++) w[m] = win[(size_t)kc * 3 + m];
    SplitCell<NF> o{};
    if (par > 0) {
        split_cell<NF, FLUX, SHAK>(S, S.psum + size_t((par - 1) & 1) * split_rows<NF, FLUX>(nch) * np, kc, i, rdx, upd_any, w, pn, o);
        if (chunk == 0 && own) {
            flag_health(S.health, prim_health<3>(pn));
#pragma unroll
            for (int m = 0; m < 3; m++) {
                S.w[in][(size_t)kc * 3 + m] = w[m];
                if constexpr (END) S.prim[(size_t)kc * 3 + m] = pn[m];
            }
        }
        if (upd_any) {
#pragma unroll
            for (int j = 0; j < CH; j++) {
                double f[NF];
#pragma unroll
                for (int q = 0; q < NF; q++) f[q] = fr[q][j];
                split_relax<NF, SHAK>(o, K, ch.u[j], f);
#pragma unroll
                for (int q = 0; q < NF; q++) fr[q][j] = f[q];
            }
        }
    }
    if constexpr (END) {
        if (own) {
#pragma unroll
            for (int j = 0; j < CH; j++)
                if (vb + j < nv) {
#pragma unroll
                    for (int q = 0; q < NF; q++) bstore(fr[q][j], fout, voff, (q * nv + vb + j) * rowb);
                }
        }
        return;
    } else {
        // ---- face coefficients of the lane's left face
        SFace<double> F{};
        double fw0[3], m3, m4 = 0.0, sw[3], wL[3], wR[3];
        const double dxL = shr1(dxh);
#pragma unroll
        for (int m = 0; m < 3; m++) {
            const double wl = shr1(w[m]), wr = shl1(w[m]);
            sw[m] = LIMK == LIM_NONE ? 0.0 : limiter<double>(lk, (w[m] - wl) * rL, (wr - w[m]) * rR);
        }
#pragma unroll
        for (int m = 0; m < 3; m++) {
            wL[m] = shr1(w[m]) + shr1(sw[m]) * dxL;
            wR[m] = w[m] - sw[m] * dxh;
        }
        if constexpr (FLUX == KCU) {
            KcuFace<3> Fk;
            kcu_face<3>(wL, wR, K, S.gam, S.mu, S.om, dt, Fk);
            F.A = Fk.prim[0] * sqrt(Fk.prim[2] / kPi);
            F.nl2 = -Fk.prim[2] * kLog2e;
            F.Ui = Fk.prim[1];
            F.kb = K / (2.0 * Fk.prim[2]);
            F.M0 = Fk.Mt1;
            F.M1 = Fk.Mt2;
            for (int m = 0; m < 3; m++) fw0[m] = Fk.fw0[m];
            m3 = Fk.Mt2;
        } else {
            UgksFace1 Fu;
            ugks_face_1d(wL, wR, K, S.gam, S.mu, S.om, dt, dxL, dxh, Fu);
            F.A = Fu.prim[0] * sqrt(Fu.prim[2] / kPi);
            F.nl2 = -Fu.prim[2] * kLog2e;
            F.Ui = Fu.prim[1];
            F.kb = K / (2.0 * Fu.prim[2]);
            F.Mxi2 = Fu.Mxi2;
            F.M0 = Fu.Mt[0], F.M1 = Fu.Mt[1], F.M2 = Fu.Mt[2], F.M3 = Fu.Mt[3], F.M4 = Fu.Mt[4];
            F.aL0 = Fu.aL[0], F.aL1 = Fu.aL[1], F.aL2 = Fu.aL[2];
            F.aR0 = Fu.aR[0], F.aR1 = Fu.aR[1], F.aR2 = Fu.aR[2];
            F.aT0 = Fu.aT[0], F.aT1 = Fu.aT[1], F.aT2 = Fu.aT[2];
            for (int m = 0; m < 3; m++) fw0[m] = Fu.fw0[m];
            m3 = Fu.Mt[3];
            m4 = Fu.Mt[4];
        }
        // ---- slopes, fluxes, moment sums, transport update (pass 1 of k_sweep1d)
        double part[NR], UoT = 0.0;
        if (SHAK) {
            double pq[3];
            conserve_prim<3>(w, S.gam, pq);
            UoT = pq[1];
        }
#pragma unroll
        for (int m = 0; m < NR; m++) part[m] = 0.0;
        static_for<CH>([&](auto jc) {
            constexpr int j = jc;
            const double u = ch.u[j], uu = ch.uu[j];
            const bool up = (ch.upmask >> j) & 1;  // the same in all lanes
            double fu[NF], su[NF], ff[NF];
#pragma unroll
            for (int q = 0; q < NF; q++) {
                const double f = fr[q][j], d = f - shr1(f);
                const double s = sweep_limit<double, LIMK, false>(lk, d * rL, shl1(d) * rR);
                const double l = shr1(f + s * dxh), r = f - s * dxh, sl = shr1(s);
                fu[q] = up ? l : r;
                su[q] = up ? sl : s;
            }
            if constexpr (FLUX == KCU) {
                const double cI = u - F.Ui;
                const double g = F.A * texp2(F.nl2 * (cI * cI));
                ff[0] = F.M0 * u * g + F.M1 * u * fu[0];
                if constexpr (NF == 2) ff[1] = F.M0 * u * (g * F.kb) + F.M1 * u * fu[1];
                part[0] += ch.wk[1][j] * fu[0];
                part[1] += ch.wk[2][j] * fu[0];
                part[2] += ch.wk[3][j] * fu[0];
                if constexpr (NF == 2) part[3] += ch.wk[1][j] * fu[1];
            } else {
                const double x = u;
                const double cI = x - F.Ui;
                const double H = F.A * texp2(F.nl2 * (cI * cI));
                const double Bq = H * F.kb;
                const double a0 = up ? F.aL0 : F.aR0, a1 = up ? F.aL1 : F.aR1, a2 = up ? F.aL2 : F.aR2;
                const double pH = a0 * H + a1 * x * H + 0.5 * a2 * (uu * H + Bq);
                const double pTH = F.aT0 * H + F.aT1 * x * H + 0.5 * F.aT2 * (uu * H + Bq);
                const double pB = a0 * Bq + a1 * x * Bq + 0.5 * a2 * (uu * Bq + F.Mxi2 * H);
                const double pTB = F.aT0 * Bq + F.aT1 * x * Bq + 0.5 * F.aT2 * (uu * Bq + F.Mxi2 * H);
                ff[0] = F.M0 * x * H + F.M1 * uu * pH + F.M2 * x * pTH + F.M3 * x * fu[0] - F.M4 * uu * su[0];
                ff[NF - 1] = F.M0 * x * Bq + F.M1 * uu * pB + F.M2 * x * pTB + F.M3 * x * fu[NF - 1] - F.M4 * uu * su[NF - 1];
                part[0] += ch.wk[1][j] * fu[0];
                part[1] += ch.wk[2][j] * su[0];
                part[2] += ch.wk[2][j] * fu[0];
                part[3] += ch.wk[3][j] * su[0];
                part[4] += ch.wk[3][j] * fu[0] + ch.wk[1][j] * fu[NF - 1];
                part[5] += ch.wk[4][j] * su[0] + ch.wk[2][j] * su[NF - 1];
            }
            if constexpr (SHAK) {
                const double co = u - UoT;
                const double wc = ch.wk[0][j] * co;
                part[C::NRAW] += (wc * (co * co)) * fr[0][j];
                if constexpr (NF == 2) part[C::NRAW] += wc * fr[1][j];
            }
#pragma unroll
            for (int q = 0; q < NF; q++) {
                const double G = fr[q][j] + (ff[q] - shl1(ff[q])) * rdx;
                if (own && vb + j < nv) bstore(G, fout, voff, (q * nv + vb + j) * rowb);
            }
        });
        // the left faces of the segment's cells, and the last stepped cell's right one
        if (own || (i == S.upd_hi + 1 && wi.c1 == S.upd_hi)) {
            double* P = S.psum + size_t(par & 1) * split_rows<NF, FLUX>(nch) * np + kc;
#pragma unroll
            for (int m = 0; m < NR; m++) P[size_t(chunk * NR + m) * np] = part[m];
            if (chunk == 0) {
#pragma unroll
                for (int m = 0; m < 3; m++) P[size_t(nch * NR + m) * np] = fw0[m];
                P[size_t(nch * NR + 3) * np] = m3;
                P[size_t(nch * NR + 4) * np] = m4;
            }
        }
    }
}

// grid: items x the most chunks of their solves, one wavefront each
template <int NF, int FLUX, bool END>
__global__ __launch_bounds__(64) void k_split1d(const Solve1D* __restrict__ solves, const WorkItem* __restrict__ items, int par) {
    const WorkItem wi = items[blockIdx.x];
    const Solve1D& S = solves[wi.solve];
    const int chunk = blockIdx.y, lane = threadIdx.x;
    if (chunk * kVChunk >= S.nv) return;
#define KBG_L(LIMK, SH) split1d<NF, FLUX, LIMK, SH, END>(S, wi, par, chunk, lane)
    if (S.coll == SHAKHOV) {
        if (!S.interp2) KBG_L(LIM_NONE, true);
        else if (S.limiter == VANLEER) KBG_L(LIM_VANLEER, true);
        else KBG_L(LIM_GENERIC, true);
    } else {
        if (!S.interp2) KBG_L(LIM_NONE, false);
        else if (S.limiter == VANLEER) KBG_L(LIM_VANLEER, false);
        else KBG_L(LIM_GENERIC, false);
    }
#undef KBG_L
}

}  // namespace

size_t split1d_psum(int nf, int flux, int nv, long np) {
    const int nch = (nv + kVChunk - 1) / kVChunk;
    const int rows = flux == UGKS ? split_rows<2, UGKS>(nch) : (nf == 2 ? split_rows<2, KCU>(nch) : split_rows<1, KCU>(nch));
    return size_t(2) * rows * np;
}

hipError_t launch_split1d(int nf, int flux, const Solve1D* d_solves, const WorkItem* d_items, int nitems, int chunks, int par, int end, hipStream_t st) {
    if (nitems <= 0) return hipSuccess;
    if (chunks < 1 || chunks > 65535 || (flux == UGKS && nf != 2) || (flux != UGKS && flux != KCU)) return hipErrorInvalidValue;
    const dim3 grid(nitems, chunks), block(64);
#define KBG_K(NF, FL)                                                                              \
    do {                                                                                           \
        if (end) hipLaunchKernelGGL((k_split1d<NF, FL, true>), grid, block, 0, st, d_solves, d_items, par); \
        else hipLaunchKernelGGL((k_split1d<NF, FL, false>), grid, block, 0, st, d_solves, d_items, par);    \
    } while (0)
    if (flux == UGKS) KBG_K(2, UGKS);
    else if (nf == 2) KBG_K(2, KCU);
    else KBG_K(1, KCU);
#undef KBG_K
    return hipGetLastError();
}

}  // namespace kbg
