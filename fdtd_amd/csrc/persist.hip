// persist.hip -- many time steps of a small grid in one launch (gfx950).
//
// A grid whose fields fit the chip's LDS (160 KB on each of 256 CUs) is cut
// into one tile per CU, whole x rows of TY x TZ (y, z) columns, and stays
// there for all the steps of a run: a step of the launched sweeps costs two
// launches and a chain of dependent memory round trips however small the
// grid is.  Per step a workgroup exchanges only the rows on its tile's sides
// with its four neighbours: H of the high sides before their E half-step, E
// of the low sides before their H half-step.  A row travels as 64-bit words
// of value and step number, written and read past the L2 of the XCD; a
// reader polls the word itself, so a side costs one trip through memory and
// no fence.  No word is overwritten early: the writer's next value of a row
// depends on what its reader computes from this one.
//
// Every workgroup has to be resident (a cooperative launch, one per CU), and
// every wait ends: a reader gives up after a bounded number of polls, raises
// the launch's flag, and all go on without waiting to the end of their loops
// (the host then reports an error).
//
// What bounds it: the exchange (two trips through memory and two barriers a
// step, 3.2 us where a tile is one row) and, per unit, the vector
// instructions of a half-step at four waves per SIMD (about 1.5 us for each
// unit a wave holds).  64^3 (one unit a wave): 12.2 us a step launched, 3.9
// in one launch; 128x128x64 (four) 19.4 -> 14.5 (27.8 with a launch for each
// region variant).  Units described by scalar
// loads, coefficients and psi read each step: 64^3 5.4, 128x128x64 20.1 (a
// wait for any load also waits for the psi and row stores before it, so
// what can be is kept in registers).
//
// The arithmetic of a cell is that of kernels.hip, in the same order, on
// values rounded to the storage type at every half-step; the stored bits are
// the sweeps'.  psi stays in global memory (only its own lane touches it).
// A probe's sample is stored; the DFT sums are formed from the samples after
// the run, in step order.
#include <hip/hip_runtime.h>
#include <climits>
#include <cstdint>

#include "device_common.h"
#include "internal.h"
#include "persist_common.h"
#include "sweep_common.h"

namespace fdtd {

// A unit is one 64-cell segment of one row of the tile; its six components
// lie side by side in LDS ([unit][6][64]), so one base address and immediate
// offsets reach them.  A wave keeps the same NU units for all steps: their E
// coefficients, x-slab psi and (up to three units) y- and z-slab psi stay in
// registers.  What a half-step needs to know about a unit is the same on
// every lane and every step (PUnit, built by the host, in the order the
// half-step takes the units: those that wait for a neighbour's row last).
template <int NU>
__device__ __forceinline__ PUnit unit_of(const PDesc<NU> &d, int n)
{
    PUnit u;
    u.lds = d.at(n, 0); u.flags = d.at(n, 1); u.i0 = d.at(n, 2); u.j = d.at(n, 3); u.k = d.at(n, 4);
    u.psx = d.at(n, 5); u.psy = d.at(n, 6); u.psz = d.at(n, 7); u.wj = d.at(n, 8); u.wk = d.at(n, 9);
    u.oj = d.at(n, 10); u.ok = d.at(n, 11); u.ev = d.at(n, 12); u.nev = d.at(n, 13);
    return u;
}

// psi of a cell's slabs (two values per axis) and the E coefficients of a unit
struct PPsi {
    float a, b;
};
struct PCoef {
    float xc, xa, xb, yc, ya, yb, zc, za, zb;
};

template <class T, int NU>
__global__ void __launch_bounds__(64 * PW) persist_kernel(const KArgs a, const PArgs p)
{
    extern __shared__ __align__(16) char smem[];
    constexpr int UB = 6 * 64;          // floats of a unit
    constexpr bool YZ = NU <= 3;        // y- and z-slab psi in registers, else read and written where used
    const int nx = a.nx, U = p.units, XS = p.sx * 64;
    const int rowf = p.sx * UB, plnf = p.ty * rowf;   // floats from a row to the next, from a plane to the next
    float *const sf = (float *)smem + 64;             // [unit][ex ey ez hx hy hz][64], 64 floats spare on both sides
    float *const spx = sf + U * UB + 64;              // x profiles b, a, kappa of E, then of H: [6][XS]
    PEvent *const evs = (PEvent *)(spx + 6 * XS);
    const int lane = (int)(threadIdx.x & 63);
    const int w = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const PTile tile = p.tiles[blockIdx.x];
    const int nu = __builtin_amdgcn_readfirstlane(tile.nu);
    PDesc<NU> de, dh;
    de.load(p.units_e + (i64)blockIdx.x * U, w, nu, lane);
    dh.load(p.units_h + (i64)blockIdx.x * U, w, nu, lane);
    float dx = a.d[0], dy = a.d[1], dz = a.d[2];
    const int L0 = a.L[0], L1 = nx - a.L[1];
    auto sx_of = [&](const PUnit &u) { const int i = u.i0 + lane; return u.psx + (i < L0 ? i : i - L1 + L0); };
    auto xs_e = [&](const PUnit &u) {
        const int i = u.i0 + lane;
        return (u.flags & PU_XS) && ((i > 0 && i < L0) || (i >= L1 && i < nx - 1));   // fdtdrav.h:752,777
    };
    auto xs_h = [&](const PUnit &u) {
        const int i = u.i0 + lane;
        return (u.flags & PU_XS) && (i < L0 || (i >= L1 && i < nx - 1));   // fdtdrav.h:402,424
    };

    // ---- load the tile, and post the first H rows
    if (threadIdx.x < 64) {
        sf[(int)threadIdx.x - 64] = 0.f;
        sf[U * UB + (int)threadIdx.x] = 0.f;
    }
    PCoef cf[NU];
    PPsi ex_[NU], hx_[NU];   // psi: E / H half-step, x slab
    constexpr int NP = YZ ? NU : 1;
    PPsi ey_[NP], ez_[NP], hy_[NP], hz_[NP];   // y, z slab
    auto psi_ld = [&](PPsi &q, const void *pa_, const void *pb_, int s) {
        q.a = ld((const T *)pa_ + s);
        q.b = ld((const T *)pb_ + s);
    };
#pragma unroll
    for (int n = 0; n < NU; ++n) {
        const int np = YZ ? n : 0;
        ex_[n] = hx_[n] = ey_[np] = ez_[np] = hy_[np] = hz_[np] = PPsi{0.f, 0.f};
        if (w + n * PW >= nu) continue;
        {
            const PUnit u = unit_of(de, n);
            const int i = u.i0 + lane;
            const i64 c = (i64)u.k * a.plane + (i64)u.j * a.px + i;
            int cl = 0;
            if (a.cls != nullptr && i < nx) cl = p.cls16 ? (int)((const std::uint16_t *)a.cls)[c] : (int)((const u32 *)a.cls)[c];
            if (a.e_uni) cl = 0;
            const float4 *t = a.etab + cl * 3;
            const float4 tx = t[0], ty = t[1], tz = t[2];
            cf[n] = PCoef{tx.x, tx.y, tx.z, ty.x, ty.y, ty.z, tz.x, tz.y, tz.z};
            if (xs_e(u)) psi_ld(ex_[n], a.psi_eyx, a.psi_ezx, sx_of(u));
            if (YZ && (u.flags & PU_YS) && i < nx) psi_ld(ey_[np], a.psi_exy, a.psi_ezy, u.psy + lane);
            if (YZ && (u.flags & PU_ZS) && i < nx) psi_ld(ez_[np], a.psi_exz, a.psi_eyz, u.psz + lane);
        }
        const PUnit u = unit_of(dh, n);
        const int i = u.i0 + lane;
        const i64 c = (i64)u.k * a.plane + (i64)u.j * a.px + i;
        float *o = sf + u.lds + lane;
        const bool in = i < nx;
        float v[6];
        v[0] = in ? ld((const T *)a.ex + c) : 0.f;
        v[1] = in ? ld((const T *)a.ey + c) : 0.f;
        v[2] = in ? ld((const T *)a.ez + c) : 0.f;
        v[3] = in ? ld((const T *)a.hx + c) : 0.f;
        v[4] = in ? ld((const T *)a.hy + c) : 0.f;
        v[5] = in ? ld((const T *)a.hz + c) : 0.f;
        for (int q = 0; q < 6; ++q) o[64 * q] = v[q];
        if (u.flags & PU_GJ) { ll_put(p.ll + u.oj + lane, v[3], p.epoch); ll_put(p.ll + u.oj + XS + lane, v[5], p.epoch); }
        if (u.flags & PU_GK) { ll_put(p.ll + u.ok + lane, v[3], p.epoch); ll_put(p.ll + u.ok + XS + lane, v[4], p.epoch); }
        if (xs_h(u)) psi_ld(hx_[n], a.psi_hyx, a.psi_hzx, sx_of(u));
        if (YZ && (u.flags & PU_YS) && in) psi_ld(hy_[np], a.psi_hxy, a.psi_hzy, u.psy + lane);
        if (YZ && (u.flags & PU_ZS) && in) psi_ld(hz_[np], a.psi_hxz, a.psi_hyz, u.psz + lane);
    }
    for (int i = (int)threadIdx.x; i < XS; i += 64 * PW) {
        const float4 e = i < nx ? a.px_prof[i] : make_float4(0.f, 0.f, 1.f, 0.f);
        const float4 h = i < nx ? a.px_prof[nx + i] : make_float4(0.f, 0.f, 1.f, 0.f);
        spx[i] = e.x; spx[XS + i] = e.y; spx[2 * XS + i] = e.z;
        spx[3 * XS + i] = h.x; spx[4 * XS + i] = h.y; spx[5 * XS + i] = h.z;
    }
    for (int q = (int)threadIdx.x; q < tile.nev; q += 64 * PW) evs[q] = p.events[tile.ev + q];
    __syncthreads();

    bool dead = false;
    const Coef uh{uload(a.htab), uload(a.htab + 1), uload(a.htab + 2)};

    // ---- E half-step of a unit
    auto e_unit = [&](const PCoef &t, PPsi &qx, PPsi &ry, PPsi &rz, const PUnit &u, int m, u32 tag) {
        PPsi qy{0.f, 0.f}, qz{0.f, 0.f};
        if (YZ) {
            qy = ry;
            qz = rz;
        }
        ConstKArgs &ra = rare_args(a);
        const int i = u.i0 + lane, fl = u.flags;
        if (!YZ && (fl & PU_YS) && i < nx) psi_ld(qy, a.psi_exy, a.psi_ezy, u.psy + lane);
        if (!YZ && (fl & PU_ZS) && i < nx) psi_ld(qz, a.psi_exz, a.psi_eyz, u.psz + lane);
        float *const o = sf + u.lds + lane;
        const float *const oj = o - rowf, *const ok = o - plnf;
        const float hx = o[192], hy = o[256], hz = o[320];
        const float ex0 = o[0], ey0 = o[64], ez0 = o[128];
        // H at i-1: the previous lane's; lane 0's from the segment before (unused at i = 0)
        const float *const of = sf + u.lds - ((fl & PU_XL) ? UB : 0) + 63;
        const float hy_im = lane_prev(hy, of[256]), hz_im = lane_prev(hz, of[320]);
        float hx_jm = 0.f, hz_jm = 0.f, hx_km = 0.f, hy_km = 0.f;
        if (fl & (PU_GJ | PU_GK))
            ll_wait(p, (fl & PU_GJ) != 0, p.ll + u.wj + lane, (fl & PU_GK) != 0, p.ll + u.wk + lane, XS, tag, dead, hx_jm,
                    hz_jm, hx_km, hy_km);
        if (fl & PU_IJ) {
            hx_jm = oj[192];
            hz_jm = oj[320];
        }
        if (fl & PU_IK) {
            hx_km = ok[192];
            hy_km = ok[256];
        }
        const bool ilo = i > 0, ihi = i < nx - 1;
        const bool jlo = (fl & PU_JLO) != 0, jhi = (fl & PU_JHI) != 0, klo = (fl & PU_KLO) != 0, khi = (fl & PU_KHI) != 0;
        const bool xs = xs_e(u), ys = (fl & PU_YS) != 0, zs = (fl & PU_ZS) != 0;
        float cbx_hz = t.xa, cbx_hy = t.xb, cby_hx = t.ya, cby_hz = t.yb, cbz_hy = t.za, cbz_hx = t.zb;
        float4 pye = make_float4(0.f, 0.f, 1.f, 0.f), pze = pye;
        if (xs) {
            const float kp = spx[2 * XS + i];
            cby_hz = cby_hz / kp;
            cbz_hy = cbz_hy / kp;
        }
        if (ys) {
            pye = uload(a.py_prof + u.j);
            cbx_hz = cbx_hz / pye.z;
            cbz_hx = cbz_hx / pye.z;
        }
        if (zs) {
            pze = uload(a.pz_prof + u.k);
            cbx_hy = cbx_hy / pze.z;
            cby_hx = cby_hx / pze.z;
        }
        float exn = (t.xc * ex0 + cbx_hz * (hz - hz_jm)) + cbx_hy * (hy - hy_km);
        float eyn = (t.yc * ey0 + cby_hx * (hx - hx_km)) + cby_hz * (hz - hz_im);
        float ezn = (t.zc * ez0 + cbz_hy * (hy - hy_im)) + cbz_hx * (hx - hx_jm);
        const bool upx = ihi && jlo && jhi && klo && khi, upy = ilo && ihi && jhi && klo && khi;
        const bool upz = ilo && ihi && jlo && jhi && khi;
        if (!upx) exn = ex0;
        if (!upy) eyn = ey0;
        if (!upz) ezn = ez0;
        // source edges and probes of the unit (calc_e's source term,
        // fdtdrav.h:726-729, and sampleField, fdtdrav.h:740)
        for (int e = u.ev; e < u.ev + u.nev; ++e) {
            if (evs[e].lane != i) continue;
            if (evs[e].kind == EV_SOURCE) {
                if (upz)
                    ezn = ((evs[e].ceze * ez0 + evs[e].cezhy * (hy - hy_im)) + evs[e].cezhx * (hx - hx_jm)) +
                          evs[e].cezj * ra.vpn[(i64)evs[e].wave * ra.steps_cap + m];
            } else if (ra.rec) {
                const int comp = evs[e].kind - EV_PROBE;
                ra.probe_hist[(i64)evs[e].id * ra.steps_cap + m] =
                    (comp == 0 ? exn : comp == 1 ? eyn : ezn) * pick6(ra.probe_unscale, comp);
            }
        }
        // CPML psi recursions and corrections, fdtdrav.h:750-911
        if (xs && jhi && khi) {
            const float b = spx[i], av = spx[XS + i];
            const float pey = b * qx.a + av * (hz - hz_im);
            const float pez = b * qx.b + av * (hy - hy_im);
            qx.a = rnd(pey, (const T *)nullptr);   // (what a store and a load would give)
            qx.b = rnd(pez, (const T *)nullptr);
            if (klo) eyn = eyn + (t.yb * dx) * pey;
            if (jlo) ezn = ezn + (t.za * dx) * pez;
        }
        if (ys && khi && ihi) {
            const float pex = pye.x * qy.a + pye.y * (hz - hz_jm);
            const float pez = pye.x * qy.b + pye.y * (hx - hx_jm);
            if (YZ) {
                ry.a = rnd(pex, (const T *)nullptr);
                ry.b = rnd(pez, (const T *)nullptr);
            } else {
                st((T *)a.psi_exy + u.psy + lane, pex);
                st((T *)a.psi_ezy + u.psy + lane, pez);
            }
            if (klo) exn = exn + (t.xa * dy) * pex;
            if (ilo) ezn = ezn + (t.zb * dy) * pez;
        }
        if (zs && jhi && ihi) {
            const float pex = pze.x * qz.a + pze.y * (hy - hy_km);
            const float pey = pze.x * qz.b + pze.y * (hx - hx_km);
            if (YZ) {
                rz.a = rnd(pex, (const T *)nullptr);
                rz.b = rnd(pey, (const T *)nullptr);
            } else {
                st((T *)a.psi_exz + u.psz + lane, pex);
                st((T *)a.psi_eyz + u.psz + lane, pey);
            }
            if (jlo) exn = exn + (t.xb * dz) * pex;
            if (ilo) eyn = eyn + (t.ya * dz) * pey;
        }
        exn = rnd(exn, (const T *)nullptr);
        eyn = rnd(eyn, (const T *)nullptr);
        ezn = rnd(ezn, (const T *)nullptr);
        o[0] = exn;
        o[64] = eyn;
        o[128] = ezn;
        // E of the tile's low sides, for the H half-step of the tiles below
        if (fl & PU_GJ) { ll_put(p.ll + u.oj + lane, exn, tag + 1); ll_put(p.ll + u.oj + XS + lane, ezn, tag + 1); }
        if (fl & PU_GK) { ll_put(p.ll + u.ok + lane, exn, tag + 1); ll_put(p.ll + u.ok + XS + lane, eyn, tag + 1); }
        if (a.snap != nullptr && u.j >= a.sb[1] && u.j < a.sb[1] + a.sb[4] && u.k >= a.sb[2] && u.k < a.sb[2] + a.sb[5] &&
            i >= a.sb[0] && i < a.sb[0] + a.sb[3])
            e_snapshot(ra, i, u.j, u.k, m, exn, eyn, ezn);
    };
    // ---- H half-step of a unit
    auto h_unit = [&](PPsi &qx, PPsi &ry, PPsi &rz, const PUnit &u, int m, u32 tag) {
        PPsi qy{0.f, 0.f}, qz{0.f, 0.f};
        if (YZ) {
            qy = ry;
            qz = rz;
        }
        ConstKArgs &ra = rare_args(a);
        const int i = u.i0 + lane, fl = u.flags;
        if (!YZ && (fl & PU_YS) && i < nx) psi_ld(qy, a.psi_hxy, a.psi_hzy, u.psy + lane);
        if (!YZ && (fl & PU_ZS) && i < nx) psi_ld(qz, a.psi_hxz, a.psi_hyz, u.psz + lane);
        float *const o = sf + u.lds + lane;
        const float *const oj = o + rowf, *const ok = o + plnf;
        const float ex = o[0], ey = o[64], ez = o[128];
        const float hx0 = o[192], hy0 = o[256], hz0 = o[320];
        // E at i+1: the next lane's; lane 63's from the segment after (unused at i = nx-1)
        const float *const of = sf + u.lds + ((fl & PU_XL) ? UB : 0);
        const float ey_ip = lane_next(ey, of[64]), ez_ip = lane_next(ez, of[128]);
        float ex_jp = 0.f, ez_jp = 0.f, ex_kp = 0.f, ey_kp = 0.f;
        if (fl & (PU_GJ | PU_GK))
            ll_wait(p, (fl & PU_GJ) != 0, p.ll + u.wj + lane, (fl & PU_GK) != 0, p.ll + u.wk + lane, XS, tag + 1, dead,
                    ex_jp, ez_jp, ex_kp, ey_kp);
        if (fl & PU_IJ) {
            ex_jp = oj[0];
            ez_jp = oj[128];
        }
        if (fl & PU_IK) {
            ex_kp = ok[0];
            ey_kp = ok[64];
        }
        const bool in = i < nx, ihi = i < nx - 1, jhi = (fl & PU_JHI) != 0, khi = (fl & PU_KHI) != 0;
        const bool xs = xs_h(u), ys = (fl & PU_YS) != 0, zs = (fl & PU_ZS) != 0;
        float chx_ey = uh.x.y, chx_ez = uh.x.z, chy_ez = uh.y.y, chy_ex = uh.y.z, chz_ex = uh.z.y, chz_ey = uh.z.z;
        float4 pym = make_float4(0.f, 0.f, 1.f, 0.f), pzm = pym;
        if (xs) {
            const float kp = spx[5 * XS + i];
            chy_ez = chy_ez / kp;
            chz_ey = chz_ey / kp;
        }
        if (ys) {
            pym = uload(a.py_prof + a.ny + u.j);
            chx_ez = chx_ez / pym.z;
            chz_ex = chz_ex / pym.z;
        }
        if (zs) {
            pzm = uload(a.pz_prof + a.nz + u.k);
            chx_ey = chx_ey / pzm.z;
            chy_ex = chy_ex / pzm.z;
        }
        float hxn = (uh.x.x * hx0 + chx_ey * (ey_kp - ey)) + chx_ez * (ez_jp - ez);
        float hyn = (uh.y.x * hy0 + chy_ez * (ez_ip - ez)) + chy_ex * (ex_kp - ex);
        float hzn = (uh.z.x * hz0 + chz_ex * (ex_jp - ex)) + chz_ey * (ey_ip - ey);
        if (!(in && jhi && khi)) hxn = hx0;
        if (!(ihi && khi)) hyn = hy0;
        if (!(ihi && jhi)) hzn = hz0;
        // probes of the unit (sampleField in calc_h, fdtdrav.h:347-391)
        for (int e = u.ev; e < u.ev + u.nev; ++e) {
            if (evs[e].lane != i || !ra.rec) continue;
            const int comp = evs[e].kind - EV_PROBE;
            ra.probe_hist[(i64)evs[e].id * ra.steps_cap + m] =
                (comp == 3 ? hxn : comp == 4 ? hyn : hzn) * pick6(ra.probe_unscale, comp);
        }
        if (xs) {
            const float b = spx[3 * XS + i], av = spx[4 * XS + i];
            const float phy = b * qx.a + av * (ez_ip - ez);
            const float phz = b * qx.b + av * (ey_ip - ey);
            qx.a = rnd(phy, (const T *)nullptr);
            qx.b = rnd(phz, (const T *)nullptr);
            if (khi) hyn = hyn + (uh.y.y * dx) * phy;
            if (jhi) hzn = hzn + (uh.z.z * dx) * phz;
        }
        if (ys && in) {
            const float phx = pym.x * qy.a + pym.y * (ez_jp - ez);
            const float phz = pym.x * qy.b + pym.y * (ex_jp - ex);
            if (YZ) {
                ry.a = rnd(phx, (const T *)nullptr);
                ry.b = rnd(phz, (const T *)nullptr);
            } else {
                st((T *)a.psi_hxy + u.psy + lane, phx);
                st((T *)a.psi_hzy + u.psy + lane, phz);
            }
            if (khi) hxn = hxn + (uh.x.z * dy) * phx;
            if (ihi) hzn = hzn + (uh.z.y * dy) * phz;
        }
        if (zs && in) {
            const float phx = pzm.x * qz.a + pzm.y * (ey_kp - ey);
            const float phy = pzm.x * qz.b + pzm.y * (ex_kp - ex);
            if (YZ) {
                rz.a = rnd(phx, (const T *)nullptr);
                rz.b = rnd(phy, (const T *)nullptr);
            } else {
                st((T *)a.psi_hxz + u.psz + lane, phx);
                st((T *)a.psi_hyz + u.psz + lane, phy);
            }
            if (jhi) hxn = hxn + (uh.x.y * dz) * phx;
            if (ihi) hyn = hyn + (uh.y.z * dz) * phy;
        }
        hxn = rnd(hxn, (const T *)nullptr);
        hyn = rnd(hyn, (const T *)nullptr);
        hzn = rnd(hzn, (const T *)nullptr);
        o[192] = hxn;
        o[256] = hyn;
        o[320] = hzn;
        // H of the tile's high sides, for the E half-step of the tiles above
        if (fl & PU_GJ) { ll_put(p.ll + u.oj + lane, hxn, tag + 1); ll_put(p.ll + u.oj + XS + lane, hzn, tag + 1); }
        if (fl & PU_GK) { ll_put(p.ll + u.ok + lane, hxn, tag + 1); ll_put(p.ll + u.ok + XS + lane, hyn, tag + 1); }
    };

    for (int s = 0; s < p.n; ++s) {
        const int m = p.m0 + s;
        const u32 tag = p.epoch + (u32)s;
        // four units or more: keep coefficient times cell size inside the
        // loop (kept for every unit across it, the products spill)
        if (NU >= 4) asm volatile("" : "+s"(dx), "+s"(dy), "+s"(dz));
#pragma unroll
        for (int n = 0; n < NU; ++n) {
            __builtin_amdgcn_sched_barrier(0);   // one unit's registers at a time
            if (w + n * PW < nu) e_unit(cf[n], ex_[n], ey_[YZ ? n : 0], ez_[YZ ? n : 0], unit_of(de, n), m, tag);
        }
        __syncthreads();
#pragma unroll
        for (int n = 0; n < NU; ++n) {
            __builtin_amdgcn_sched_barrier(0);
            if (w + n * PW < nu) h_unit(hx_[n], hy_[YZ ? n : 0], hz_[YZ ? n : 0], unit_of(dh, n), m, tag);
        }
        __syncthreads();
    }
    // ---- write the tile back
    auto psi_st = [&](const PPsi &q, void *pa_, void *pb_, int s) {
        st((T *)pa_ + s, q.a);
        st((T *)pb_ + s, q.b);
    };
#pragma unroll
    for (int n = 0; n < NU; ++n) {
        if (w + n * PW >= nu) continue;
        const int np = YZ ? n : 0;
        {
            const PUnit u = unit_of(de, n);
            const bool in = u.i0 + lane < nx;
            if (xs_e(u)) psi_st(ex_[n], a.psi_eyx, a.psi_ezx, sx_of(u));
            if (YZ && (u.flags & PU_YS) && in) psi_st(ey_[np], a.psi_exy, a.psi_ezy, u.psy + lane);
            if (YZ && (u.flags & PU_ZS) && in) psi_st(ez_[np], a.psi_exz, a.psi_eyz, u.psz + lane);
        }
        const PUnit u = unit_of(dh, n);
        const int i = u.i0 + lane;
        if (xs_h(u)) psi_st(hx_[n], a.psi_hyx, a.psi_hzx, sx_of(u));
        if (YZ && (u.flags & PU_YS) && i < nx) psi_st(hy_[np], a.psi_hxy, a.psi_hzy, u.psy + lane);
        if (YZ && (u.flags & PU_ZS) && i < nx) psi_st(hz_[np], a.psi_hxz, a.psi_hyz, u.psz + lane);
        const i64 c = (i64)u.k * a.plane + (i64)u.j * a.px + i;
        const float *o = sf + u.lds + lane;
        if (i >= nx) continue;
        st((T *)a.ex + c, o[0]);
        st((T *)a.ey + c, o[64]);
        st((T *)a.ez + c, o[128]);
        st((T *)a.hx + c, o[192]);
        st((T *)a.hy + c, o[256]);
        st((T *)a.hz + c, o[320]);
    }
}

// DFT sums of steps [m0, m0 + n) from the probe samples, in step order
// (record_probe's arithmetic); one thread per probe and frequency.
__global__ void dft_kernel(const KArgs a, int nprobe, int m0, int n)
{
    const int t = (int)(blockIdx.x * blockDim.x + threadIdx.x);
    if (t >= nprobe * a.nfreq) return;
    const int pr = t / a.nfreq, f = t % a.nfreq;
    double2 acc = a.dft[t];
    const float *h = a.probe_hist + (i64)pr * a.steps_cap;
#pragma unroll 8   // (the loads of eight steps together, their sums in order)
    for (int m = m0; m < m0 + n; ++m) {
        const double dv = (double)h[m];
        const double2 ph = a.phasor[(i64)m * a.nfreq + f];
        acc.x = acc.x + dv * ph.x;
        acc.y = acc.y + dv * ph.y;
    }
    a.dft[t] = acc;
}

// ---- launchers --------------------------------------------------------------
size_t persist_lds(int units, int sx)
{
    return (6 * (size_t)units * 64 + 128 + 6 * (size_t)sx * 64) * 4 + P_MAX_EVENTS * sizeof(PEvent);
}
int persist_max_units() { return 5 * PW; }   // the kernel is built for one to five units per wave

template <class T>
static const void *persist_fn_t(int units)
{
    switch ((units + PW - 1) / PW) {
    case 1: return (const void *)persist_kernel<T, 1>;
    case 2: return (const void *)persist_kernel<T, 2>;
    case 3: return (const void *)persist_kernel<T, 3>;
    case 4: return (const void *)persist_kernel<T, 4>;
    case 5: return (const void *)persist_kernel<T, 5>;
    default: return nullptr;
    }
}
static const void *persist_fn(int storage, int units)
{
    switch (storage) {
    case 0: return persist_fn_t<float>(units);
    case 1: return persist_fn_t<_Float16>(units);
    case 2: return persist_fn_t<bf16_t>(units);
    default: return nullptr;
    }
}

bool persist_fits(int storage, int units, int tiles, size_t lds, int device)
{
    return coop_fits(persist_fn(storage, units), tiles, lds, device);
}

hipError_t launch_persist(int storage, const KArgs &a, const PArgs &p, int tiles, size_t lds, hipStream_t s)
{
    const void *fn = persist_fn(storage, p.units);
    if (!fn) return hipErrorInvalidValue;
    void *args[2] = {(void *)&a, (void *)&p};
    return hipLaunchCooperativeKernel(fn, dim3(tiles), dim3(64 * PW), args, (unsigned)lds, s);
}

hipError_t launch_dft(const KArgs &a, int nprobe, int m0, int n, hipStream_t s)
{
    const int t = nprobe * a.nfreq;
    if (t > 0) hipLaunchKernelGGL(dft_kernel, dim3((t + 63) / 64), dim3(64), 0, s, a, nprobe, m0, n);
    return hipGetLastError();
}

}  // namespace fdtd
