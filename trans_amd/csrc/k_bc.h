// Ghost-cell fills: physical BCs (wall, far field, symmetry, inlet, outlet) and the
// block-interface / periodic halo copy, all in one launch over a table of BC patches.
// Patches write disjoint ghost cells and read only interior cells (or ghosts they wrote
// themselves), so the reference's sequential patch order (BC/Boundary.F90:22-47) does not
// change any result.
#pragma once
#include "dev_common.h"

struct DPatch {
    trans_patch p;
    int blk;    // owning block
    int tpatch; // global index of the target patch (interfaces)
    int count;  // face cells of the patch
    int pad;
};

struct BcSeg {
    int patch;
    int base;
};

__device__ __forceinline__ long gidx(const BlkInfo& b, int i, int j, int k)
{
    return cidx(b, i, j, k);
}

// BC/BC_far.F90:135-207
__device__ __forceinline__ void farbond(double XM, double P2, double RR, double Vxi, double Vyi,
                                        double Vzi, double DNx, double DNy, double DNz, double VxF,
                                        double VyF, double VzF, double& PP0, double& RR0, double& VX0,
                                        double& VY0, double& VZ0, double& dir)
{
    const double pGam = 1.4;
    const double AF = 1. / XM;
    const double AE = sqrt(pGam * P2 / RR);
    const double QNE = Vxi * DNx + Vyi * DNy + Vzi * DNz;
    const double QNF = VxF * DNx + VyF * DNy + VzF * DNz;
    const double RF = QNF - 5. * AF;
    const double RE = QNE + 5. * AE;
    const double QN = 0.5 * (RE + RF);
    const double AS = 0.1 * (RE - RF);
    if (QN > -AS && QN < 0.) {
        const double SON = 1. / pGam / (XM * XM);
        VX0 = (VxF - QNF * DNx) + QN * DNx;
        VY0 = (VyF - QNF * DNy) + QN * DNy;
        VZ0 = (VzF - QNF * DNz) + QN * DNz;
        RR0 = pow(AS * AS / SON / pGam, 2.5);
        PP0 = AS * AS * RR0 / pGam;
        dir = -1.;
    }
    if (QN >= 0. && QN < AS) {
        const double SON = P2 / pow(RR, pGam);
        VX0 = (Vxi - QNE * DNx) + QN * DNx;
        VY0 = (Vyi - QNE * DNy) + QN * DNy;
        VZ0 = (Vzi - QNE * DNz) + QN * DNz;
        RR0 = pow(AS * AS / SON / pGam, 2.5);
        PP0 = AS * AS * RR0 / pGam;
        dir = 1.;
    }
    if (QN <= -AS) {
        VX0 = VxF;
        VY0 = VyF;
        VZ0 = VzF;
        RR0 = 1.0;
        PP0 = 1. / pGam / XM / XM;
        dir = -1.;
    }
    if (QN >= AS) {
        VX0 = Vxi;
        VY0 = Vyi;
        VZ0 = Vzi;
        RR0 = RR;
        PP0 = P2;
        dir = 1.;
    }
}

// Geom/startup.F90:1-25
__device__ __forceinline__ void ijk_start_end(int I, int J, int K, const int* tl, const int* tt,
                                              int lcross, int& Is, int& Js, int& Ks)
{
    const int ft1 = tl[0], ft2 = tl[1], ft3 = tl[2];
    const int gt1 = tt[0], gt2 = tt[1], gt3 = tt[2];
    const int lc1 = 1 - lcross;
    const int t1 = ft1 * I + ft2 * J + ft3 * K;
    const int t2 = ft1 * (J * lc1 + K * lcross) + ft2 * (I * lc1 + K * lcross) + ft3 * (I * lc1 + J * lcross);
    const int t3 = ft1 * (J * lcross + K * lc1) + ft2 * (I * lcross + K * lc1) + ft3 * (I * lcross + J * lc1);
    Is = gt1 * t1 + (gt2 + gt3) * t2;
    Js = gt2 * t1 + gt1 * t2 + gt3 * t3;
    Ks = gt3 * t1 + (gt1 + gt2) * t3;
}

__device__ __forceinline__ const int* lay_src(const trans_patch& c, int lay)
{
    return lay == 0 ? c.cijkadd : (lay == 1 ? c.cijkadd1 : c.cijkadd2);
}
__device__ __forceinline__ const int* lay_dst(const trans_patch& c, int lay)
{
    return lay == 0 ? c.ceijkadd : (lay == 1 ? c.ceijkadd1 : c.ceijkadd2);
}

// sine and cosine of an interface's angle, which is zero for all but periodic ones
__device__ __forceinline__ void rotation(double a, double& sint, double& cost)
{
    if (a == 0.0) {
        sint = a;
        cost = 1.0;
    } else {
        sint = sin(a);
        cost = cos(a);
    }
}

// A thread fills the three ghost layers of one face cell.  Bound by the latency of its loads: they
// are all issued before the first store (the compiler keeps a load behind a store that may alias
// it, which made a chain of up to 33 of them).  The third layer's source is interior too, but in a
// block of two cells along k it can be a ghost cell that the first two layers fill: `thin` blocks
// load it after those stores.  Both sweeps of the 0.30M-cell cascade 73 us, now 61 us; of the
// 8.1M-cell sector 554 us, now 490 us.
__global__ void __launch_bounds__(128) k_bc(trans_params p, int if_turb, int sweep, Fields f,
                                            const BlkInfo* __restrict__ blks,
                                            const DPatch* __restrict__ pt, const BcSeg* __restrict__ seg)
{
    const BcSeg sg = seg[blockIdx.x];
    const DPatch& dp = pt[sg.patch];
    const int lin = sg.base + threadIdx.x;
    const trans_patch& c = dp.p;
    const int n0 = c.point_end[0] - c.point_start[0] + 1;
    const int n1 = c.point_end[1] - c.point_start[1] + 1;
    const int n2 = c.point_end[2] - c.point_start[2] + 1;
    if (lin >= n0 * n1 * n2) return;
    const BlkInfo b = blks[dp.blk];
    const long tot = f.tot;
    const int i = c.point_start[0] + lin % n0;
    const int j = c.point_start[1] + (lin / n0) % n1;
    const int k = c.point_start[2] + lin / (n0 * n1);
    const int* ad = c.cijkadd;
    const int* e = c.ceijkadd;

    if (sweep == 0) {
        if (c.bctype == 9) {
            const DPatch& tp = pt[dp.tpatch];
            const BlkInfo br = blks[tp.blk];
            const trans_patch& bc = tp.p;
            const int IIadd = c.point_end[0] - c.point_start[0] + 2;
            const int JJadd = c.point_end[1] - c.point_start[1] + 2;
            const int KKadd = c.point_end[2] - c.point_start[2] + 2;
            int iL = i - c.point_start[0] + 1, jL = j - c.point_start[1] + 1, kL = k - c.point_start[2] + 1;
            iL = c.rev_matrix[0] * IIadd + (1 - 2 * c.rev_matrix[0]) * iL;
            jL = c.rev_matrix[1] * JJadd + (1 - 2 * c.rev_matrix[1]) * jL;
            kL = c.rev_matrix[2] * KKadd + (1 - 2 * c.rev_matrix[2]) * kL;
            int ib, jb, kb;
            ijk_start_end(iL, jL, kL, c.transform, c.transform_t, c.lcross, ib, jb, kb);
            ib += bc.point_start[0] - 1;
            jb += bc.point_start[1] - 1;
            kb += bc.point_start[2] - 1;
            const long src = gidx(br, ib + bc.cijkadd[0], jb + bc.cijkadd[1], kb + bc.cijkadd[2]);
            const long dst = gidx(b, i + e[0], j + e[1], k + e[2]);
            double sint, cost;
            rotation(c.rotate_angle, sint, cost);
            const double cos2t = cost * cost, sin2t = sint * sint, sct = sint * cost;
            double* o = f.DQ;
            double g[18];
#pragma unroll
            for (int L = 0; L < 18; L++) g[L] = o[(long)L * tot + src];
            const double ugx = g[0], ugy = g[1], ugz = g[2];
            const double vgx = g[3], vgy = g[4], vgz = g[5];
            const double wgx = g[6], wgy = g[7], wgz = g[8];
            o[dst] = ugx;
            o[tot + dst] = cost * ugy + sint * ugz;
            o[2 * tot + dst] = -sint * ugy + cost * ugz;
            o[3 * tot + dst] = cost * vgx + sint * wgx;
            o[4 * tot + dst] = cos2t * vgy + sct * (vgz + wgy) + sin2t * wgz;
            o[5 * tot + dst] = cos2t * vgz + sct * (-vgy + wgz) - sin2t * wgy;
            o[6 * tot + dst] = -sint * vgx + cost * wgx;
            o[7 * tot + dst] = -sin2t * vgz + sct * (-vgy + wgz) + cos2t * wgy;
            o[8 * tot + dst] = sin2t * vgy + sct * (vgz + wgy) + cos2t * wgz;
#pragma unroll
            for (int L = 9; L < 18; L += 3) {
                o[(long)L * tot + dst] = g[L];
                o[(long)(L + 1) * tot + dst] = cost * g[L + 1] + sint * g[L + 2];
                o[(long)(L + 2) * tot + dst] = -sint * g[L + 1] + cost * g[L + 2];
            }
        } else if (c.bctype == 1 || c.bctype == 2 || c.bctype == 3 || c.bctype == 5 || c.bctype == 7) {
            const long src = gidx(b, i + ad[0], j + ad[1], k + ad[2]);
            const long dst = gidx(b, i + e[0], j + e[1], k + e[2]);
            double g[18];
#pragma unroll
            for (int L = 0; L < 18; L++) g[L] = f.DQ[(long)L * tot + src];
#pragma unroll
            for (int L = 0; L < 18; L++) f.DQ[(long)L * tot + dst] = g[L];
        }
        return;
    }
    if (sweep != -1) return;
    const bool thin = b.nk < 4;

    switch (c.bctype) {
    case 1: {  // BC/BC_Wall.F90:41-120
        long is = gidx(b, i + ad[0], j + ad[1], k + ad[2]);
        long il = gidx(b, i + e[0], j + e[1], k + e[2]);
        const double ztemp = 0.5 * (f.Zc[is] + f.Zc[il]);
        const double ytemp = 0.5 * (f.Yc[is] + f.Yc[il]);
        const double vibc = 0.0;
        const double vjbc = (double)c.subbctype * p.omega1 * ztemp;
        const double vkbc = -(double)c.subbctype * p.omega1 * ytemp;
        const double dst = if_turb ? f.Dst[il] : 0.0, Rmiuw = if_turb ? f.Rmiu[is] : 0.0;
        const double r0 = f.Rds[is], r1 = f.Rds[tot + is], r2 = f.Rds[2 * tot + is];
        float q0 = 0.f, q1 = 0.f, q2 = 0.f;
        if (f.Rdsf) {
            q0 = f.Rdsf[is];
            q1 = f.Rdsf[tot + is];
            q2 = f.Rdsf[2 * tot + is];
        }
        double pp[3], tt[3];
        auto load = [&](const int lay) {
            const int* sa = lay_src(c, lay);
            const long s2 = gidx(b, i + sa[0], j + sa[1], k + sa[2]);
            pp[lay] = f.PP[s2];
            tt[lay] = f.T[s2];
        };
        double den0 = 0.0;
        auto store = [&](const int lay) {
            const int* ea = lay_dst(c, lay);
            const long d2 = gidx(b, i + ea[0], j + ea[1], k + ea[2]);
            f.PP[d2] = pp[lay];
            f.T[d2] = tt[lay];
            const double den = pp[lay] / (tt[lay] + p.tiny) * p.rxm2;
            if (lay == 0) den0 = den;
            f.V[d2] = den;
            f.V[tot + d2] = vibc * den;
            f.V[2 * tot + d2] = vjbc * den;
            f.V[3 * tot + d2] = vkbc * den;
        };
        load(0);
        load(1);
        if (!thin) load(2);
        store(0);
        f.Rds[il] = r0;
        f.Rds[tot + il] = r1;
        f.Rds[2 * tot + il] = r2;
        if (f.Rdsf) {
            f.Rdsf[il] = q0;
            f.Rdsf[tot + il] = q1;
            f.Rdsf[2 * tot + il] = q2;
        }
        store(1);
        if (thin) load(2);
        store(2);
        if (if_turb) {
            const double Omegaw = 60.0 * sutherland(p, tt[0]) / (den0 * 0.075 * dst * dst * p.ref * p.ref);
#pragma unroll
            for (int lay = 0; lay < 3; lay++) {
                const int* ea = lay_dst(c, lay);
                const long d2 = gidx(b, i + ea[0], j + ea[1], k + ea[2]);
                f.V[5 * tot + d2] = 0.0;
                f.V[6 * tot + d2] = Omegaw;
                f.Rmiu[d2] = Rmiuw;
            }
        }
        break;
    }
    case 2: {  // BC/BC_far.F90:40-118
        const int dn = c.ijkdirect - 1;
        const double out_n = (double)(2 * c.left_or_right - 4);
        long is = gidx(b, i + c.ijkadd[0], j + c.ijkadd[1], k + c.ijkadd[2]);
        const double g = f.Grad[(long)dn * tot + is];
        const double* S = f.SD + (long)dn * tot;
        const double Sout1 = S[is] / g, Sout2 = S[3 * tot + is] / g, Sout3 = S[6 * tot + is] / g;
        const double Dnx = Sout1 * out_n, Dny = Sout2 * out_n, Dnz = Sout3 * out_n;
        is = gidx(b, i + ad[0], j + ad[1], k + ad[2]);
        const double Den = f.V[is];
        const double Vxi = f.V[tot + is] / Den, Vyi = f.V[2 * tot + is] / Den, Vzi = f.V[3 * tot + is] / Den;
        const double P2 = f.PP[is];
        const long il = gidx(b, i + e[0], j + e[1], k + e[2]);
        double vt[2] = {0.0, 0.0}, rmi = 0.0;
        if (if_turb) {
            vt[0] = f.V[5 * tot + is];
            vt[1] = f.V[6 * tot + is];
            rmi = f.Rmiu[is];
        }
        const double ve = f.V[4 * tot + il];  // the energy of the first layer stays as it is
        double PP0 = 0, Den0 = 0, Vx0 = 0, Vy0 = 0, Vz0 = 0, dir = 0;
        farbond(p.xm, P2, Den, Vxi, Vyi, Vzi, Dnx, Dny, Dnz, p.vxf, p.vyf, p.vzf, PP0, Den0, Vx0, Vy0,
                Vz0, dir);
        const double den = 2 * Den0 - Den;
        const double pg = 2.0 * PP0 - P2;
        const double tg = p.rxm2 * pg / den;
        const double vg[5] = {den, 2.0 * Vx0 - Vxi, 2.0 * Vy0 - Vyi, 2.0 * Vz0 - Vzi, ve};
        if (if_turb && !(dir > 0.0)) {
            const double RmiuFar = sutherland(p, tg);
            rmi = 2.0 * p.visratio * RmiuFar - rmi;
            vt[0] = 2.0 * 1.5 * p.fsti * p.fsti * den - vt[0];
            vt[1] = vt[0] / (rmi + p.tiny) * den;
        }
#pragma unroll
        for (int lay = 0; lay < 3; lay++) {
            const int* ea = lay_dst(c, lay);
            const long d2 = gidx(b, i + ea[0], j + ea[1], k + ea[2]);
#pragma unroll
            for (int L = 0; L < 5; L++) f.V[(long)L * tot + d2] = vg[L];
            f.PP[d2] = pg;
            f.T[d2] = tg;
            if (if_turb) {
                f.V[5 * tot + d2] = vt[0];
                f.V[6 * tot + d2] = vt[1];
                f.Rmiu[d2] = rmi;
            }
        }
        break;
    }
    case 3: {  // BC/BC_Symm.F90:42-110 (layer 1 keeps its density)
        const int dn = c.ijkdirect - 1;
        long is = gidx(b, i + c.ijkadd[0], j + c.ijkadd[1], k + c.ijkadd[2]);
        const double g = f.Grad[(long)dn * tot + is];
        const double* S = f.SD + (long)dn * tot;
        const double Sout1 = S[is] / g, Sout2 = S[3 * tot + is] / g, Sout3 = S[6 * tot + is] / g;
        is = gidx(b, i + ad[0], j + ad[1], k + ad[2]);
        const double den = f.V[is];
        const double Vc1 = f.V[tot + is] / den * Sout1 + f.V[2 * tot + is] / den * Sout2 +
                           f.V[3 * tot + is] / den * Sout3;
        double v[3][10];
        auto load = [&](const int lay) {
            const int* sa = lay_src(c, lay);
            const long s2 = gidx(b, i + sa[0], j + sa[1], k + sa[2]);
#pragma unroll
            for (int L = 0; L < 5; L++) v[lay][L] = f.V[(long)L * tot + s2];
            v[lay][5] = f.PP[s2];
            v[lay][6] = f.T[s2];
            if (if_turb) {
                v[lay][7] = f.V[5 * tot + s2];
                v[lay][8] = f.V[6 * tot + s2];
                v[lay][9] = f.Rmiu[s2];
            }
        };
        auto store = [&](const int lay) {
            const int* ea = lay_dst(c, lay);
            const long d2 = gidx(b, i + ea[0], j + ea[1], k + ea[2]);
            const double r1 = v[lay][0];
            if (lay != 1) f.V[d2] = r1;
            f.V[tot + d2] = v[lay][1] - 2 * Sout1 * Vc1 * r1;
            f.V[2 * tot + d2] = v[lay][2] - 2 * Sout2 * Vc1 * r1;
            f.V[3 * tot + d2] = v[lay][3] - 2 * Sout3 * Vc1 * r1;
            f.V[4 * tot + d2] = v[lay][4];
            f.PP[d2] = v[lay][5];
            f.T[d2] = v[lay][6];
            if (if_turb) {
                f.V[5 * tot + d2] = v[lay][7];
                f.V[6 * tot + d2] = v[lay][8];
                f.Rmiu[d2] = v[lay][9];
            }
        };
        load(0);
        load(1);
        if (!thin) load(2);
        store(0);
        store(1);
        if (thin) load(2);
        store(2);
        break;
    }
    case 5: {  // BC/BC_Inlet.F90:38-107
        const long is = gidx(b, i + ad[0], j + ad[1], k + ad[2]);
        const long il = gidx(b, i + e[0], j + e[1], k + e[2]);
        double PsIn = f.PP[is];
        PsIn = fmin(PsIn, 0.999 * p.p0in);
        const double comm = fmax(1.0, pow(p.p0in / PsIn, 1.0 / 3.5));
        const double mach = sqrt((comm - 1.0) * 2 / 0.4);
        const double TsIn = p.t0in / comm;
        const double Roin = p.rxm2 * PsIn / TsIn;
        const double asonic = sqrt(1.4 * PsIn / Roin);
        const double Vabs = mach * asonic;
        const double VxInlet = Vabs;
        const double VyInlet = p.omega1 * (f.Zc[is]);
        const double VzInlet = -p.omega1 * f.Yc[is];
        const double v2 = Roin * VxInlet, v3 = Roin * VyInlet, v4 = Roin * VzInlet;
        double r[3];
#pragma unroll
        for (int d = 0; d < 3; d++) r[d] = f.Rds[(long)d * tot + is];
        const double vg[5] = {Roin, v2, v3, v4,
                              PsIn / 0.4 + 0.5 * (v2 * v2 + v3 * v3 + v4 * v4) / Roin -
                                  0.5 * sqr(p.omega1 * f.rad[il]) * Roin};
        double v6 = 0.0, v7 = 0.0, rm = 0.0;
        if (if_turb) {
            rm = p.visratio * sutherland(p, TsIn);
            v6 = 1.5 * p.fsti * p.fsti * Roin;
            v7 = v6 / (rm + p.tiny) * Roin;
        }
#pragma unroll
        for (int d = 0; d < 3; d++) f.Rds[(long)d * tot + il] = r[d];
        if (f.Rdsf)
            for (int d = 0; d < 3; d++) f.Rdsf[(long)d * tot + il] = f.Rdsf[(long)d * tot + is];
#pragma unroll
        for (int lay = 0; lay < 3; lay++) {
            const int* ea = lay_dst(c, lay);
            const long d2 = gidx(b, i + ea[0], j + ea[1], k + ea[2]);
#pragma unroll
            for (int L = 0; L < 5; L++) f.V[(long)L * tot + d2] = vg[L];
            f.PP[d2] = PsIn;
            f.T[d2] = TsIn;
            if (if_turb) {
                f.V[5 * tot + d2] = v6;
                f.V[6 * tot + d2] = v7;
                f.Rmiu[d2] = rm;
            }
        }
        break;
    }
    case 7: {  // outlet ghosts come from k_bc_outlet; the layer-0 Rds copy is here
        const long is = gidx(b, i + ad[0], j + ad[1], k + ad[2]);
        const long il = gidx(b, i + e[0], j + e[1], k + e[2]);
        double r[3];
#pragma unroll
        for (int d = 0; d < 3; d++) r[d] = f.Rds[(long)d * tot + is];
#pragma unroll
        for (int d = 0; d < 3; d++) f.Rds[(long)d * tot + il] = r[d];
        if (f.Rdsf)
            for (int d = 0; d < 3; d++) f.Rdsf[(long)d * tot + il] = f.Rdsf[(long)d * tot + is];
        break;
    }
    case 9: {  // BC/BC_P2P.F90:76-139
        const DPatch& tp = pt[dp.tpatch];
        const BlkInfo br = blks[tp.blk];
        const trans_patch& bc = tp.p;
        const int IIadd = c.point_end[0] - c.point_start[0] + 2;
        const int JJadd = c.point_end[1] - c.point_start[1] + 2;
        const int KKadd = c.point_end[2] - c.point_start[2] + 2;
        int iL = i - c.point_start[0] + 1, jL = j - c.point_start[1] + 1, kL = k - c.point_start[2] + 1;
        iL = c.rev_matrix[0] * IIadd + (1 - 2 * c.rev_matrix[0]) * iL;
        jL = c.rev_matrix[1] * JJadd + (1 - 2 * c.rev_matrix[1]) * jL;
        kL = c.rev_matrix[2] * KKadd + (1 - 2 * c.rev_matrix[2]) * kL;
        int ib, jb, kb;
        ijk_start_end(iL, jL, kL, c.transform, c.transform_t, c.lcross, ib, jb, kb);
        ib += bc.point_start[0] - 1;
        jb += bc.point_start[1] - 1;
        kb += bc.point_start[2] - 1;
        double sint, cost;
        rotation(c.rotate_angle, sint, cost);
        int pr0, pr1, pr2;
        ijk_start_end(1, 2, 3, c.transform, c.transform_t, c.lcross, pr0, pr1, pr2);
        const bool tthin = br.nk < 4;
        double v[3][11], r[3];
        auto load = [&](const int lay) {
            const int* sa = lay_src(bc, lay);
            const long src = gidx(br, ib + sa[0], jb + sa[1], kb + sa[2]);
#pragma unroll
            for (int L = 0; L < 7; L++) v[lay][L] = f.V[(long)L * tot + src];
            v[lay][7] = f.PP[src];
            v[lay][8] = f.T[src];
            v[lay][9] = f.Rmiu[src];
            v[lay][10] = f.shock[src];
            if (lay == 0)
#pragma unroll
                for (int d = 0; d < 3; d++) r[d] = f.Rds[(long)d * tot + src];
        };
        auto store = [&](const int lay) {
            const int* ea = lay_dst(c, lay);
            const long dst = gidx(b, i + ea[0], j + ea[1], k + ea[2]);
            f.V[dst] = v[lay][0];
            f.V[tot + dst] = v[lay][1];
            f.V[2 * tot + dst] = cost * v[lay][2] + sint * v[lay][3];
            f.V[3 * tot + dst] = -sint * v[lay][2] + cost * v[lay][3];
#pragma unroll
            for (int L = 4; L < 7; L++) f.V[(long)L * tot + dst] = v[lay][L];
            f.PP[dst] = v[lay][7];
            f.T[dst] = v[lay][8];
            f.Rmiu[dst] = v[lay][9];
            f.shock[dst] = v[lay][10];
            if (lay == 0) {
                f.Rds[(long)(pr0 - 1) * tot + dst] = r[0];
                f.Rds[(long)(pr1 - 1) * tot + dst] = r[1];
                f.Rds[(long)(pr2 - 1) * tot + dst] = r[2];
                if (f.Rdsf) {
                    f.Rdsf[(long)(pr0 - 1) * tot + dst] = (float)r[0];
                    f.Rdsf[(long)(pr1 - 1) * tot + dst] = (float)r[1];
                    f.Rdsf[(long)(pr2 - 1) * tot + dst] = (float)r[2];
                }
            }
        };
        load(0);
        load(1);
        if (!tthin) load(2);
        store(0);
        store(1);
        if (tthin) load(2);
        store(2);
        break;
    }
    default:
        break;
    }
}

// ---------------------------------------------------------------------------------------
// BC/BC_Outlet.F90:49-107: static-pressure outlet with the radial-equilibrium march along j
// from the hub.  One workgroup per (i,k) line of an outlet patch: the march inputs are staged
// in LDS by all lanes, lane 0 runs the pressure recurrence, and all lanes write the ghosts
// (the layer-0 Rds copy of the same routine is done by k_bc, after the spectral radius).
// It reads interior cells and geometry only.
//
// Bound by the recurrence: four divisions follow each other in a step.  Three have divisors that
// are known beforehand; the lanes form their reciprocals, and the recurrence corrects the product
// with the reciprocal by two remainders (outlet_div), which is half as long as a division.  The
// next step's inputs are read from LDS a step ahead.  128 steps: 48 us, now 35 us.
constexpr int OUTLET_MAXJ = 512;

struct OutLine {
    int patch;  // index into the device patch table
    int i, k;
};

// a / b, correctly rounded, for y = 1 / b correctly rounded: the second correction of a quotient
// that is within one unit in the last place gives the nearest value (P. Markstein, Computation of
// elementary functions on the IBM RISC System/6000 processor, 1990), as long as nothing over- or
// underflows (outlet_range).
__device__ __forceinline__ double outlet_div(double a, double b, double y)
{
    const double q0 = a * y;
    const double q1 = __builtin_fma(__builtin_fma(-b, q0, a), y, q0);
    return __builtin_fma(__builtin_fma(-b, q1, a), y, q1);
}
__device__ __forceinline__ bool outlet_range(double x) { return fabs(x) > 1e-100 && fabs(x) < 1e100; }

// One j of the march: the state beside the ghost, angle and radii, with the divisors' reciprocals.
struct OutStep {
    double t, rt, v1, rv1, v3, v4, sn, cs;
    double om;     // omega * r
    double dr;     // to the next radius
    double r, rr;  // r + tiny and its reciprocal
};

// The pressure at the next j; DIV: with divisions throughout.  *ok: cleared where a quotient could
// over- or underflow.
template <bool DIV>
__device__ __forceinline__ double outlet_step(const trans_params& p, const OutStep& q, double pp, bool* ok)
{
    // ghost state of this j (density, y/z momentum) as the reference has it
    const double den = (DIV ? pp / q.t : outlet_div(pp, q.t, q.rt)) * p.rxm2;
    const double ratio = DIV ? den / q.v1 : outlet_div(den, q.v1, q.rv1);
    const double gv3 = q.v3 * ratio, gv4 = q.v4 * ratio;
    const double RoVr2 = sqr(gv4 / den * q.cs - q.sn * gv3 / den + q.om);
    const double num = fabs(q.dr * den * RoVr2);
    if (ok) *ok = *ok && outlet_range(pp) && outlet_range(den) && (num == 0.0 || outlet_range(num));
    return pp + (DIV ? num / q.r : outlet_div(num, q.r, q.rr));
}

__global__ void __launch_bounds__(256) k_bc_outlet(trans_params p, int if_turb, Fields f,
                                                   const BlkInfo* __restrict__ blks,
                                                   const DPatch* __restrict__ pt,
                                                   const OutLine* __restrict__ lines)
{
    __shared__ double s_pp[OUTLET_MAXJ];
    __shared__ OutStep s_in[OUTLET_MAXJ];
    const OutLine ln = lines[blockIdx.x];
    const DPatch& dp = pt[ln.patch];
    const trans_patch& c = dp.p;
    const BlkInfo b = blks[dp.blk];
    const long tot = f.tot;
    const int* ad = c.cijkadd;
    const int* e = c.ceijkadd;
    const int j0 = c.point_start[1];
    const int nj = c.point_end[1] - j0 + 1;
    const int i = ln.i, k = ln.k;
    bool ok = true;
    for (int jj = threadIdx.x; jj < nj; jj += blockDim.x) {
        const int j = j0 + jj;
        const long is = gidx(b, i + ad[0], j + ad[1], k + ad[2]);
        const long il = gidx(b, i + e[0], j + e[1], k + e[2]);
        const double t = f.T[is], v1 = f.V[is], r = f.rad[il], th = f.thtc[il];
        const double v3 = f.V[2 * tot + is], v4 = f.V[3 * tot + is];
        const double rnext = jj + 1 < nj ? f.rad[gidx(b, i + e[0], j + 1 + e[1], k + e[2])] : r;
        OutStep q;
        q.t = t;
        q.rt = 1.0 / t;
        q.v1 = v1;
        q.rv1 = 1.0 / v1;
        q.v3 = v3;
        q.v4 = v4;
        q.sn = sin(th);
        q.cs = cos(th);
        q.om = p.omega1 * r;
        q.dr = rnext - r;
        q.r = r + p.tiny;
        q.rr = 1.0 / q.r;
        s_in[jj] = q;
        ok = ok && outlet_range(t) && outlet_range(v1) && outlet_range(q.r);
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        double pp = p.pouthub;
        s_pp[0] = pp;
        OutStep q = s_in[0];
#pragma unroll 2
        for (int jj = 1; jj < nj; jj++) {
            const OutStep n = s_in[jj];
            pp = outlet_step<false>(p, q, pp, nullptr);
            s_pp[jj] = pp;
            q = n;
        }
    }
    __syncthreads();
    for (int jj = threadIdx.x; jj < nj; jj += blockDim.x) (void)outlet_step<false>(p, s_in[jj], s_pp[jj], &ok);
    ok = __syncthreads_and(ok);
    if (!ok) {
        if (threadIdx.x == 0) {
            double pp = p.pouthub;
            for (int jj = 1; jj < nj; jj++) {
                pp = outlet_step<true>(p, s_in[jj - 1], pp, nullptr);
                s_pp[jj] = pp;
            }
        }
        __syncthreads();
    }
    for (int jj = threadIdx.x; jj < nj; jj += blockDim.x) {
        const int j = j0 + jj;
        const long is = gidx(b, i + ad[0], j + ad[1], k + ad[2]);
        const double tt = s_in[jj].t, pp = s_pp[jj];
        const double vx = f.V[tot + is];
        double vk = 0.0, vo = 0.0, rm = 0.0;
        if (if_turb) {
            vk = f.V[5 * tot + is];
            vo = f.V[6 * tot + is];
            rm = f.Rmiu[is];
        }
        const double v1 = pp / tt * p.rxm2;
        const double den_ratio = v1 / s_in[jj].v1;
        const double vg[4] = {v1, vx * den_ratio, s_in[jj].v3 * den_ratio, s_in[jj].v4 * den_ratio};
#pragma unroll
        for (int lay = 0; lay < 3; lay++) {
            const int* ea = lay_dst(c, lay);
            const long d2 = gidx(b, i + ea[0], j + ea[1], k + ea[2]);
#pragma unroll
            for (int L = 0; L < 4; L++) f.V[(long)L * tot + d2] = vg[L];
            f.PP[d2] = pp;
            f.T[d2] = tt;
            if (if_turb) {
                f.V[5 * tot + d2] = vk;
                f.V[6 * tot + d2] = vo;
                f.Rmiu[d2] = rm;
            }
        }
    }
}
