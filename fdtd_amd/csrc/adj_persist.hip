// adj_persist.hip -- the reverse steps of a small grid in one launch (gfx950).
//
// The reverse sweeps of adjoint.hip on a grid that persist.hip steps forward
// in one launch: the same tiles, one per CU, and the same exchange of rows
// between them (the transposed H quantities of the high sides before the E
// half-step, the transposed E quantities of the low sides before the H one).
// Launched one by one, a reverse step of 128x128x64 takes 44 us however its
// blocks are cut: launches, and 24 arrays read or written through chains
// of dependent trips to memory.
//
// A wave keeps its units' dJ/dE, dJ/dH, E coefficients and x-slab psi in
// registers for all steps.  LDS holds what other waves gather: of the
// transposed quantities the pairs read at j-+1 and k-+1 (8 values a cell;
// the pair read at i-+1 comes from the adjacent lane).  y- and z-slab psi
// stay in registers up to two units a wave, else in memory, as the design
// gradient's sums do.  E takes a wave's units in order, H in reverse: units
// on a tile's low sides are listed last, those on its high sides first, so
// the units that wait for a neighbour's row come last in both.
//
// What bounds it: as in persist.hip, the exchange and then the vector
// instructions of a half-step at four waves per SIMD.  Reverse step of
// 128x128x64 (four units a wave) 44.0 us launched, 21.1 in one launch; of 64^3
// (one) 18.4, 6.0; of 96^3 (five, which spill 27 registers) 43.2, 26.5.
//
// The arithmetic of a cell is that of adjoint.hip (adj_e_kernel,
// adj_h_kernel), in the same order; the results are the same bits.
#include <hip/hip_runtime.h>
#include <climits>
#include <cstdint>

#include "device_common.h"
#include "internal.h"
#include "persist_common.h"
#include "sweep_common.h"

namespace fdtd {

namespace {

struct RPair {
    float a, b;
};
// a unit's cell on one lane: dJ/dE, dJ/dH, and the transposed pair read at
// i-1 (tz, ry of H) or i+1 (by, az of E), whichever half-step came last
struct RCell {
    float ex, ey, ez, hx, hy, hz, qa, qb;
};
struct RCoef {
    float xc, xa, xb, yc, ya, yb, zc, za, zb;
};
// what a half-step knows of a unit (the same on every lane)
struct RU {
    int fl, i0, j, k;
    __device__ __forceinline__ bool has(int f) const { return (fl & f) != 0; }
};
constexpr int RUB = 8 * 64;   // floats of a unit in LDS

}  // namespace

template <int NU>
__global__ void __launch_bounds__(64 * PW) adj_persist_kernel(const KArgs a, const AArgs b, const RArgs p)
{
    extern __shared__ __align__(16) char smem[];
    constexpr bool YZ = NU <= 2;
    constexpr int NP = YZ ? NU : 1;
    const int nx = a.nx, U = p.units, XS = p.sx * 64;
    const int rowf = p.sx * RUB, plnf = p.ty * rowf;
    float *const sf = (float *)smem;             // [unit][rx sz tx sy ax bz ay bx][64]
    float *const sb = sf + U * RUB;              // [unit][by az of lane 0, tz ry of lane 63]
    float *const spx = sb + U * 4;               // x profiles b, a, kappa of E, then of H: [6][XS]
    REvent *const evs = (REvent *)(spx + 6 * XS);
    const int lane = (int)(threadIdx.x & 63);
    const int w = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const PTile tile = p.tiles[blockIdx.x];
    const int nu = __builtin_amdgcn_readfirstlane(tile.nu);
    PDesc<NU> d;
    d.load(p.u + (i64)blockIdx.x * U, w, nu, lane);
    float dx = a.d[0], dy = a.d[1], dz = a.d[2];
    const int L0 = a.L[0], L1 = nx - a.L[1];
    const Coef uh{uload(a.htab), uload(a.htab + 1), uload(a.htab + 2)};
    auto unit = [&](int n) {
        const int fl = d.at(n, RW_FLAGS), jk = d.at(n, RW_JK);
        return RU{fl, (int)((unsigned)fl >> RU_SEG) * 64, jk & 0xFFFF, (int)((unsigned)jk >> 16)};
    };
    auto xs_e = [&](const RU &u, int i) { return u.has(RU_XS) && ((i > 0 && i < L0) || (i >= L1 && i < nx - 1)); };
    auto xs_h = [&](const RU &u, int i) { return u.has(RU_XS) && (i < L0 || (i >= L1 && i < nx - 1)); };
    auto sx_of = [&](int n, int i) { return d.at(n, RW_PSX) + (i < L0 ? i : i - L1 + L0); };
    auto psi_ld = [&](RPair &q, int pa_, int s) {
        q.a = b.pb[pa_][s];
        q.b = b.pb[pa_ + 1][s];
    };
    auto psi_st = [&](const RPair &q, int pa_, int s) {
        b.pb[pa_][s] = q.a;
        b.pb[pa_ + 1][s] = q.b;
    };

    RCell r[NU];
    RCoef cf[NU];
    RPair exs[NU], hxs[NU];                        // psi of the x slabs
    RPair eys[NP], ezs[NP], hys[NP], hzs[NP];      // of the y, z slabs

    // Transposed H quantities of a cell from its dJ/dH and psi (hq_of): the
    // pairs read at j+1 and k+1 to LDS and, on the tile's high sides, to the
    // neighbours; the pair read at i+1 kept.
    auto put_hq = [&](int n, RCell &c, const RPair &qx, const RPair &qy, const RPair &qz, u32 tag) {
        const RU u = unit(n);
        const int i = u.i0 + lane;
        const bool ihi = i < nx - 1, jhi = u.has(RU_JHI), khi = u.has(RU_KHI);
        const bool ux = jhi && khi, uy = ihi && khi, uz = ihi && jhi;
        const bool xs = xs_h(u, i), ys = u.has(RU_YSH), zs = u.has(RU_ZSH);
        float hxy = uh.x.y, hxz = uh.x.z, hyy = uh.y.y, hyz = uh.y.z, hzy = uh.z.y, hzz = uh.z.z;
        float4 pym = make_float4(0.f, 0.f, 1.f, 0.f), pzm = pym;
        if (zs) {
            pzm = uload(a.pz_prof + a.nz + u.k);
            hxy = hxy / pzm.z;
            hyz = hyz / pzm.z;
        }
        if (ys) {
            pym = uload(a.py_prof + a.ny + u.j);
            hxz = hxz / pym.z;
            hzy = hzy / pym.z;
        }
        if (xs) {
            const float kp = spx[5 * XS + i];
            hyy = hyy / kp;
            hzz = hzz / kp;
        }
        float sy = 0.f, sz = 0.f, tz = 0.f, tx = 0.f, rx = 0.f, ry = 0.f;
        if (ux) {
            sy = hxy * c.hx;
            sz = hxz * c.hx;
        }
        if (uy) {
            tz = hyy * c.hy;
            tx = hyz * c.hy;
        }
        if (uz) {
            rx = hzy * c.hz;
            ry = hzz * c.hz;
        }
        if (xs) {
            const float av = spx[4 * XS + i];
            tz += av * (qx.a + (uy ? (uh.y.y * dx) * c.hy : 0.f));
            ry += av * (qx.b + (uz ? (uh.z.z * dx) * c.hz : 0.f));
        }
        if (ys) {
            sz += pym.y * (qy.a + (ux ? (uh.x.z * dy) * c.hx : 0.f));
            rx += pym.y * (qy.b + (uz ? (uh.z.y * dy) * c.hz : 0.f));
        }
        if (zs) {
            sy += pzm.y * (qz.a + (ux ? (uh.x.y * dz) * c.hx : 0.f));
            tx += pzm.y * (qz.b + (uy ? (uh.y.z * dz) * c.hy : 0.f));
        }
        const int lu = d.at(n, RW_UNIT);
        float *const o = sf + lu * RUB + lane;
        o[0] = rx;
        o[64] = sz;
        o[128] = tx;
        o[192] = sy;
        c.qa = tz;
        c.qb = ry;
        if (u.has(RU_XLH) && lane == 63) {
            sb[lu * 4 + 2] = tz;
            sb[lu * 4 + 3] = ry;
        }
        if (u.has(RU_GJH)) {
            u64 *const q = p.ll + d.at(n, RW_OJH) + lane;
            ll_put(q, rx, tag);
            ll_put(q + XS, sz, tag);
        }
        if (u.has(RU_GKH)) {
            u64 *const q = p.ll + d.at(n, RW_OKH) + lane;
            ll_put(q, tx, tag);
            ll_put(q + XS, sy, tag);
        }
    };

    for (int i = (int)threadIdx.x; i < XS; i += 64 * PW) {
        const float4 e = i < nx ? a.px_prof[i] : make_float4(0.f, 0.f, 1.f, 0.f);
        const float4 h = i < nx ? a.px_prof[nx + i] : make_float4(0.f, 0.f, 1.f, 0.f);
        spx[i] = e.x; spx[XS + i] = e.y; spx[2 * XS + i] = e.z;
        spx[3 * XS + i] = h.x; spx[4 * XS + i] = h.y; spx[5 * XS + i] = h.z;
    }
    for (int q = (int)threadIdx.x; q < tile.nev; q += 64 * PW) evs[q] = p.events[tile.ev + q];
    __syncthreads();

    // ---- load the tile, and post the first H rows
#pragma unroll
    for (int n = 0; n < NU; ++n) {
        const int np = YZ ? n : 0;
        r[n] = RCell{};
        exs[n] = hxs[n] = RPair{0.f, 0.f};
        RPair hy{0.f, 0.f}, hz{0.f, 0.f};
        if (YZ) eys[np] = ezs[np] = hy;
        if (w + n * PW >= nu) continue;
        const RU u = unit(n);
        const int i = u.i0 + lane;
        const i64 c = (i64)u.k * a.plane + (i64)u.j * a.px + i;
        const bool in = i < nx;
        int cl = 0;
        if (a.cls != nullptr && in && !p.euni)
            cl = p.cls16 ? (int)((const std::uint16_t *)a.cls)[c] : (int)((const u32 *)a.cls)[c];
        const float4 *t = a.etab + cl * 3;
        const float4 tx = t[0], ty = t[1], tz = t[2];
        cf[n] = RCoef{tx.x, tx.y, tx.z, ty.x, ty.y, ty.z, tz.x, tz.y, tz.z};
        if (in)
            r[n] = RCell{b.eb[0][c], b.eb[1][c], b.eb[2][c], b.hb[0][c], b.hb[1][c], b.hb[2][c], 0.f, 0.f};
        const int psy = d.at(n, RW_PSY) + lane, psz = d.at(n, RW_PSZ) + lane;
        if (xs_e(u, i)) psi_ld(exs[n], 0, sx_of(n, i));
        if (xs_h(u, i)) psi_ld(hxs[n], 2, sx_of(n, i));
        if (YZ && u.has(RU_YSE) && in) psi_ld(eys[np], 4, psy);
        if (YZ && u.has(RU_ZSE) && in) psi_ld(ezs[np], 8, psz);
        if (u.has(RU_YSH) && in) psi_ld(hy, 6, psy);
        if (u.has(RU_ZSH) && in) psi_ld(hz, 10, psz);
        if (YZ) {
            hys[np] = hy;
            hzs[np] = hz;
        }
        put_hq(n, r[n], hxs[n], hy, hz, p.epoch);
    }
    __syncthreads();

    bool dead = false;

    // The E half-step of step f, pointwise part: psi_e adjoint, the design
    // edges' gradient, dJ/dE <- Ce dJ/dE
    auto finish_e = [&](int n, RCell &c, const RCoef &t, RPair &qx, RPair &qy, RPair &qz, int f) {
        const RU u = unit(n);
        const int i = u.i0 + lane;
        const bool ilo = i > 0, ihi = i < nx - 1;
        const bool jlo = u.has(RU_JLO), jhi = u.has(RU_JHI), klo = u.has(RU_KLO), khi = u.has(RU_KHI);
        const bool ux = ihi && jlo && jhi && klo && khi, uy = ilo && ihi && jhi && klo && khi;
        const bool uz = ilo && ihi && jlo && jhi && khi;
        if (u.j >= b.sb[1] && u.j < b.sb[1] + b.sb[4] && u.k >= b.sb[2] && u.k < b.sb[2] + b.sb[5] && i >= b.sb[0] &&
            i < b.sb[0] + b.sb[3]) {
            const i64 nb = (i64)b.sb[3] * b.sb[4] * b.sb[5];
            const i64 q = (i - b.sb[0]) + (i64)b.sb[3] * ((u.j - b.sb[1]) + (i64)b.sb[4] * (u.k - b.sb[2]));
            const float *h0 = b.hist + (i64)(f - b.hist_base) * 3 * nb;
            const float *h1 = h0 + 3 * nb;
            const float e_[3] = {c.ex, c.ey, c.ez};
            const bool u_[3] = {ux, uy, uz};
            for (int cc = 0; cc < 3; ++cc) {
                const float4 dc = b.dcoef[cc * nb + q];
                const double em = h0[cc * nb + q], ep = h1[cc * nb + q], g = b.gedge[cc * nb + q];
                if (!u_[cc] || (dc.x == 0.f && dc.y == 0.f)) continue;
                const double dE = (double)dc.x * em - (double)dc.y * (ep - (double)dc.z * em);
                b.gedge[cc * nb + q] = g + (double)e_[cc] * dE;
            }
        }
        if (ux || uy || uz) {
            if (xs_e(u, i) && jhi && khi) {
                const float bv = spx[i];
                qx.a = bv * (qx.a + (uy ? (t.yb * dx) * c.ey : 0.f));
                qx.b = bv * (qx.b + (uz ? (t.za * dx) * c.ez : 0.f));
            }
            if (u.has(RU_YSE) && ihi && khi) {
                const float bv = uload(a.py_prof + u.j).x;
                qy.a = bv * (qy.a + (ux ? (t.xa * dy) * c.ex : 0.f));
                qy.b = bv * (qy.b + (uz ? (t.zb * dy) * c.ez : 0.f));
                if (!YZ) psi_st(qy, 4, d.at(n, RW_PSY) + lane);
            }
            if (u.has(RU_ZSE) && ihi && jhi) {
                const float bv = uload(a.pz_prof + u.k).x;
                qz.a = bv * (qz.a + (ux ? (t.xb * dz) * c.ex : 0.f));
                qz.b = bv * (qz.b + (uy ? (t.ya * dz) * c.ey : 0.f));
                if (!YZ) psi_st(qz, 8, d.at(n, RW_PSZ) + lane);
            }
        }
        float ceze = t.zc;   // (a source edge's own, fdtdrav.h:1402-1420)
        for (int e = d.at(n, RW_EVE) & 0xFFFF, e1 = e + (int)((unsigned)d.at(n, RW_EVE) >> 16); e < e1; ++e)
            if (evs[e].kind == EV_SOURCE && evs[e].lane == i) ceze = evs[e].c0;
        if (ux) c.ex = t.xc * c.ex;
        if (uy) c.ey = t.yc * c.ey;
        if (uz) c.ez = ceze * c.ez;
    };

    // ---- E half-step of a unit: finish step m+1's, then gather step m's
    // transposed H half-step
    auto e_unit = [&](int n, RCell &c, const RCoef &t, RPair &qx, RPair &ry_, RPair &rz_, bool fin, int m, u32 tag) {
        const RU u = unit(n);
        const int i = u.i0 + lane;
        const int lu = d.at(n, RW_UNIT);
        const bool ilo = i > 0, ihi = i < nx - 1;
        const bool jlo = u.has(RU_JLO), jhi = u.has(RU_JHI), klo = u.has(RU_KLO), khi = u.has(RU_KHI);
        const bool ys = u.has(RU_YSE), zs = u.has(RU_ZSE);
        RPair ly{0.f, 0.f}, lz{0.f, 0.f};
        if (!YZ && ys && i < nx) psi_ld(ly, 4, d.at(n, RW_PSY) + lane);
        if (!YZ && zs && i < nx) psi_ld(lz, 8, d.at(n, RW_PSZ) + lane);
        RPair &qy = YZ ? ry_ : ly, &qz = YZ ? rz_ : lz;
        if (fin) finish_e(n, c, t, qx, qy, qz, m + 1);
        const float *const o = sf + lu * RUB + lane;
        const float *const oj = o - rowf, *const ok = o - plnf;
        const float rx = o[0], sz = o[64], tx = o[128], sy = o[192];
        const float *const of = sb + (lu - (u.has(RU_XLE) ? 1 : 0)) * 4;
        const float tz_im = lane_prev(c.qa, of[2]), ry_im = lane_prev(c.qb, of[3]);
        float rx_jm = 0.f, sz_jm = 0.f, tx_km = 0.f, sy_km = 0.f;
        if (u.has(RU_GJE | RU_GKE))
            ll_wait(p, u.has(RU_GJE), p.ll + d.at(n, RW_WJE) + lane, u.has(RU_GKE), p.ll + d.at(n, RW_WKE) + lane, XS, tag,
                    dead, rx_jm, sz_jm, tx_km, sy_km);
        if (u.has(RU_IJE)) {
            rx_jm = oj[0];
            sz_jm = oj[64];
        }
        if (u.has(RU_IKE)) {
            tx_km = ok[128];
            sy_km = ok[192];
        }
        const bool ux = ihi && jlo && jhi && klo && khi, uy = ilo && ihi && jhi && klo && khi;
        const bool uz = ilo && ihi && jlo && jhi && khi;
        float ebx = c.ex, eby = c.ey, ebz = c.ez;
        if (ux) {
            ebx += (tx_km - tx) + (rx_jm - rx);
            if (uz) ebz += sz_jm - sz;
        }
        if (uy) eby += (sy_km - sy) + (ry_im - c.qb);
        if (uz) ebz += tz_im - c.qa;
        if (uz && !ux) ebz += sz_jm - sz;
        // dJ/d(probe sample m) of the unit's E probes; the source edges'
        // dJ/dEz for the H half-step's gather
        for (int e = d.at(n, RW_EVE) & 0xFFFF, e1 = e + (int)((unsigned)d.at(n, RW_EVE) >> 16); e < e1; ++e) {
            if (evs[e].lane != i) continue;
            const int kind = evs[e].kind;
            if (kind == EV_SOURCE) continue;
            const float gv = b.g[(i64)evs[e].id * b.gsteps + m];
            if (kind == EV_PROBE) ebx += gv;
            else if (kind == EV_PROBE + 1) eby += gv;
            else ebz += gv;
        }
        if (ux) c.ex = ebx;
        if (uy) c.ey = eby;
        if (uz) c.ez = ebz;
        for (int e = d.at(n, RW_EVE) & 0xFFFF, e1 = e + (int)((unsigned)d.at(n, RW_EVE) >> 16); e < e1; ++e)
            if (evs[e].kind == EV_SOURCE && evs[e].lane == i) evs[e].c1 = c.ez;
        // transposed E quantities (eq_of; of the swept values, as there)
        float ax = 0.f, bx = 0.f, ay = 0.f, by = 0.f, az = 0.f, bz = 0.f;
        if (ihi && jhi && khi) {
            const bool vx = jlo && klo, vy = ilo && klo, vz = ilo && jlo;
            const bool xs = xs_e(u, i);
            float exy = t.xa, exz = t.xb, eyy = t.ya, eyz = t.yb, ezy = t.za, ezz = t.zb;
            float4 pye = make_float4(0.f, 0.f, 1.f, 0.f), pze = pye;
            if (ys) {
                pye = uload(a.py_prof + u.j);
                exy = exy / pye.z;
                ezz = ezz / pye.z;
            }
            if (zs) {
                pze = uload(a.pz_prof + u.k);
                exz = exz / pze.z;
                eyy = eyy / pze.z;
            }
            if (xs) {
                const float kp = spx[2 * XS + i];
                eyz = eyz / kp;
                ezy = ezy / kp;
            }
            if (vx) {
                ax = exy * ebx;
                bx = exz * ebx;
            }
            if (vy) {
                ay = eyy * eby;
                by = eyz * eby;
            }
            if (vz) {
                az = ezy * ebz;
                bz = ezz * ebz;
            }
            if (xs) {
                const float av = spx[XS + i];
                by += av * (qx.a + (vy ? (t.yb * dx) * eby : 0.f));
                az += av * (qx.b + (vz ? (t.za * dx) * ebz : 0.f));
            }
            if (ys) {
                ax += pye.y * (qy.a + (vx ? (t.xa * dy) * ebx : 0.f));
                bz += pye.y * (qy.b + (vz ? (t.zb * dy) * ebz : 0.f));
            }
            if (zs) {
                bx += pze.y * (qz.a + (vx ? (t.xb * dz) * ebx : 0.f));
                ay += pze.y * (qz.b + (vy ? (t.ya * dz) * eby : 0.f));
            }
        }
        float *const q = sf + lu * RUB + lane;
        q[256] = ax;
        q[320] = bz;
        q[384] = ay;
        q[448] = bx;
        c.qa = by;
        c.qb = az;
        if (u.has(RU_XLE) && lane == 0) {
            sb[lu * 4 + 0] = by;
            sb[lu * 4 + 1] = az;
        }
        if (u.has(RU_GJE)) {
            u64 *const l = p.ll + d.at(n, RW_OJE) + lane;
            ll_put(l, ax, tag + 1);
            ll_put(l + XS, bz, tag + 1);
            if (u.has(RU_SRE)) ll_put(l + 2 * XS, c.ez, tag + 1);
        }
        if (u.has(RU_GKE)) {
            u64 *const l = p.ll + d.at(n, RW_OKE) + lane;
            ll_put(l, ay, tag + 1);
            ll_put(l + XS, bx, tag + 1);
        }
    };
    // ---- H half-step of a unit: its pointwise part, then the transposed E
    // half-step gathered
    auto h_unit = [&](int n, RCell &c, RPair &qx, RPair &ry_, RPair &rz_, u32 tag) {
        const RU u = unit(n);
        const int i = u.i0 + lane;
        const int lu = d.at(n, RW_UNIT);
        const bool in = i < nx, ihi = i < nx - 1, jhi = u.has(RU_JHI), khi = u.has(RU_KHI);
        const bool ux = in && jhi && khi, uy = ihi && khi, uz = ihi && jhi;
        const bool ys = u.has(RU_YSH) && in, zs = u.has(RU_ZSH) && in;
        RPair ly{0.f, 0.f}, lz{0.f, 0.f};
        if (!YZ && ys) psi_ld(ly, 6, d.at(n, RW_PSY) + lane);
        if (!YZ && zs) psi_ld(lz, 10, d.at(n, RW_PSZ) + lane);
        RPair &qy = YZ ? ry_ : ly, &qz = YZ ? rz_ : lz;
        const float *const o = sf + lu * RUB + lane;
        const float *const oj = o + rowf, *const ok = o + plnf;
        const float ax = o[256], bz = o[320], ay = o[384], bx = o[448];
        const float *const of = sb + (lu + (u.has(RU_XLH) ? 1 : 0)) * 4;
        const float by_ip = lane_next(c.qa, of[0]), az_ip = lane_next(c.qb, of[1]);
        float ax_jp = 0.f, bz_jp = 0.f, ay_kp = 0.f, bx_kp = 0.f, ez_jp = 0.f;
        if (u.has(RU_GJH | RU_GKH))
            ll_wait(p, u.has(RU_GJH), p.ll + d.at(n, RW_WJH) + lane, u.has(RU_GKH), p.ll + d.at(n, RW_WKH) + lane, XS,
                    tag + 1, dead, ax_jp, bz_jp, ay_kp, bx_kp);
        if (u.has(RU_SRH)) {   // dJ/dEz of the row above, where it holds source edges of another tile
            float t0, t1, t2;
            ll_wait(p, true, p.ll + d.at(n, RW_WJH) + 2 * XS + lane, false, p.ll, 0, tag + 1, dead, ez_jp, t0, t1, t2);
        }
        if (u.has(RU_IJH)) {
            ax_jp = oj[256];
            bz_jp = oj[320];
        }
        if (u.has(RU_IKH)) {
            ay_kp = ok[384];
            bx_kp = ok[448];
        }
        if (xs_h(u, i)) {
            const float bv = spx[3 * XS + i];
            qx.a = bv * (qx.a + (uy ? (uh.y.y * dx) * c.hy : 0.f));
            qx.b = bv * (qx.b + (uz ? (uh.z.z * dx) * c.hz : 0.f));
        }
        if (ys) {
            const float bv = uload(a.py_prof + a.ny + u.j).x;
            qy.a = bv * (qy.a + (ux ? (uh.x.z * dy) * c.hx : 0.f));
            qy.b = bv * (qy.b + (uz ? (uh.z.y * dy) * c.hz : 0.f));
            if (!YZ) psi_st(qy, 6, d.at(n, RW_PSY) + lane);
        }
        if (zs) {
            const float bv = uload(a.pz_prof + a.nz + u.k).x;
            qz.a = bv * (qz.a + (ux ? (uh.x.y * dz) * c.hx : 0.f));
            qz.b = bv * (qz.b + (uy ? (uh.y.z * dz) * c.hy : 0.f));
            if (!YZ) psi_st(qz, 10, d.at(n, RW_PSZ) + lane);
        }
        float hbx = c.hx, hby = c.hy, hbz = c.hz;
        if (ux) hbx = uh.x.x * hbx;
        if (uy) hby = uh.y.x * hby;
        if (uz) hbz = uh.z.x * hbz;
        if (ux) {
            hbx += (ay - ay_kp) + (bz - bz_jp);
            if (uz) hbz += ax - ax_jp;
        }
        if (uy) hby += (bx - bx_kp) + (c.qb - az_ip);
        if (uz) hbz += c.qa - by_ip;
        if (uz && !ux) hbz += ax - ax_jp;
        // the source edges among the Ez gathered (src_terms): of this cell
        // (kind 0), (i+1, j) (1) and (i, j+1) (2)
        for (int e = d.at(n, RW_EVH) & 0xFFFF, e1 = e + (int)((unsigned)d.at(n, RW_EVH) >> 16); e < e1; ++e) {
            if (evs[e].lane != i) continue;
            const int kind = evs[e].kind;
            const float ebz = evs[e].id >= 0 ? evs[evs[e].id].c1 : ez_jp;
            const float tx = evs[e].c0 * ebz - evs[e].c2 * ebz, ty = evs[e].c1 * ebz - evs[e].c3 * ebz;
            if (kind == 0) {
                if (uy) hby += tx;
                if (ux) hbx += ty;
            } else if (kind == 1) {
                if (uy) hby -= tx;
            } else {
                if (ux) hbx -= ty;
            }
        }
        c.hx = hbx;
        c.hy = hby;
        c.hz = hbz;
        put_hq(n, c, qx, qy, qz, tag + 1);
    };

    for (int s = 0; s < p.n; ++s) {
        const int m = p.m1 - s;
        const u32 tag = p.epoch + (u32)s;
        if (NU >= 3) asm volatile("" : "+s"(dx), "+s"(dy), "+s"(dz));   // (as persist.hip)
#pragma unroll
        for (int n = 0; n < NU; ++n) {
            const int np = YZ ? n : 0;
            __builtin_amdgcn_sched_barrier(0);
            if (w + n * PW < nu) e_unit(n, r[n], cf[n], exs[n], eys[np], ezs[np], s > 0, m, tag);
        }
        __syncthreads();
#pragma unroll
        for (int n = NU - 1; n >= 0; --n) {
            const int np = YZ ? n : 0;
            __builtin_amdgcn_sched_barrier(0);
            if (w + n * PW < nu) h_unit(n, r[n], hxs[n], hys[np], hzs[np], tag);
        }
        __syncthreads();
    }
    // ---- finish the first step's E half-step and write the tile back
#pragma unroll
    for (int n = 0; n < NU; ++n) {
        if (w + n * PW >= nu) continue;
        const int np = YZ ? n : 0;
        const RU u = unit(n);
        const int i = u.i0 + lane;
        const bool in = i < nx;
        const int psy = d.at(n, RW_PSY) + lane, psz = d.at(n, RW_PSZ) + lane;
        RPair ly{0.f, 0.f}, lz{0.f, 0.f};
        if (!YZ && u.has(RU_YSE) && in) psi_ld(ly, 4, psy);
        if (!YZ && u.has(RU_ZSE) && in) psi_ld(lz, 8, psz);
        finish_e(n, r[n], cf[n], exs[n], YZ ? eys[np] : ly, YZ ? ezs[np] : lz, p.m1 - p.n + 1);
        if (xs_e(u, i)) psi_st(exs[n], 0, sx_of(n, i));
        if (xs_h(u, i)) psi_st(hxs[n], 2, sx_of(n, i));
        if (YZ && u.has(RU_YSE) && in) psi_st(eys[np], 4, psy);
        if (YZ && u.has(RU_ZSE) && in) psi_st(ezs[np], 8, psz);
        if (YZ && u.has(RU_YSH) && in) psi_st(hys[np], 6, psy);
        if (YZ && u.has(RU_ZSH) && in) psi_st(hzs[np], 10, psz);
        if (!in) continue;
        const i64 c = (i64)u.k * a.plane + (i64)u.j * a.px + i;
        b.eb[0][c] = r[n].ex;
        b.eb[1][c] = r[n].ey;
        b.eb[2][c] = r[n].ez;
        b.hb[0][c] = r[n].hx;
        b.hb[1][c] = r[n].hy;
        b.hb[2][c] = r[n].hz;
    }
}

// ---- launchers --------------------------------------------------------------
size_t adj_persist_lds(int units, int sx, int events)
{
    return ((size_t)units * (RUB + 4) + 6 * (size_t)sx * 64) * 4 + (size_t)events * sizeof(REvent);
}
int adj_persist_max_units() { return 5 * PW; }

static const void *adj_persist_fn(int units)
{
    switch ((units + PW - 1) / PW) {
    case 1: return (const void *)adj_persist_kernel<1>;
    case 2: return (const void *)adj_persist_kernel<2>;
    case 3: return (const void *)adj_persist_kernel<3>;
    case 4: return (const void *)adj_persist_kernel<4>;
    case 5: return (const void *)adj_persist_kernel<5>;
    default: return nullptr;
    }
}

// Whether `tiles` workgroups with `lds` bytes each can be resident at once
// (and the kernel is set up to use them).
bool adj_persist_fits(int units, int tiles, size_t lds, int device)
{
    return coop_fits(adj_persist_fn(units), tiles, lds, device);
}

hipError_t launch_adj_persist(const KArgs &a, const AArgs &b, const RArgs &p, int tiles, size_t lds, hipStream_t s)
{
    const void *fn = adj_persist_fn(p.units);
    if (!fn) return hipErrorInvalidValue;
    void *args[3] = {(void *)&a, (void *)&b, (void *)&p};
    return hipLaunchCooperativeKernel(fn, dim3(tiles), dim3(64 * PW), args, (unsigned)lds, s);
}

}  // namespace fdtd
