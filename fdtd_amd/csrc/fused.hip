// fused.hip -- one FP32 time step (E half-step, then H half-step) in one pass
// over the grid for gfx950 (MI355X).
//
// The two sweeps of kernels.hip move every field value three times a step
// (each sweep reads all six components and writes three).  Here a workgroup
// computes E^{m+1} and H^{m+1} of its tile in one z-march, so a value is read
// once and written once: 12 values per cell and step instead of 18.
//
// A workgroup is FY + 1 wavefronts on a tile of 64 x FY columns.  Wave w < FY
// owns row w: at plane k it computes E(k) from the old H(k), H(k-1), then
// H(k-1), whose z-operands E(k-1), E(k) it holds in registers.  H(k-1) also
// reads E(k-1) at (i+1, j) and (i, j+1): the x-neighbour is the next lane's
// value (a DPP wave shift), the y-neighbour comes from the next row's wave
// through LDS, one barrier per plane.  What lies beyond the tile -- row
// j0 + FY and column i0 + 64 -- is evaluated by the last wave (the row as one
// cell per lane, the column as one row per lane), and the plane above the
// z-block by the rows' own waves; none of these evaluations is stored.  FY +
// 1 = 8 waves put two on each SIMD.
//
// Workgroups evaluate each other's edge cells from old values, so a step
// reads one buffer of each field (and of the E sweep's psi) and writes the
// other.  The arithmetic of every evaluated cell is that of kernels.hip, in
// the same order; the stored bits are the two sweeps'.
//
// What bounds it: HBM.  On 512x512x256 (CPML 16, one H class) the interior
// tiles move 59 B per cell (50 are needed) at 5.2 TB/s, at 8, 16 or 24 waves
// per CU alike; a bare stream of six arrays read and six written in this
// tile order runs at 4.7 TB/s, in linear order at 5.7.  Step 1061 (the
// half-steps of kernels.hip, which win up to 24 M cells) -> 937 us.  Tried and slower: 128 x 7 tiles
// (one workgroup of 16 waves per CU: 992 us), 64 x 3 (1029) and 64 x 15
// tiles (999), z-blocks of 8 and 32 planes (977, 968), ordinary instead of
// non-temporal stores (993), the region variants as branches of one launch
// (984: every tile then has the general variant's registers and spills), and
// 16-bit storage with two cells per thread (1149 us against the pair sweeps'
// 682: its edge variants need 160-215 registers).
//   E: calc_e  fdtdrav.h:665-735, CPML fdtdrav.h:750-911
//   H: calc_h  fdtdrav.h:328-386, CPML fdtdrav.h:398-562
#include <hip/hip_runtime.h>
#include <climits>
#include <cstdint>

#include "device_common.h"
#include "internal.h"
#include "sweep_common.h"

namespace fdtd {

typedef std::uint32_t u32;

constexpr int FY = 7;   // rows of a tile; the eighth wave evaluates the edge cells

// One column of cells (i, j): predicates, slab indices, CPML profiles.
struct FCol {
    int i, j, sx, sy, mycol;
    u32 o0;       // byte offset of (i, j, 0) from the guard-plane base
    u32 cell0;    // class-map index of (i, j, 0)
    bool valid;   // a cell of the grid (off it, loads are clamped to cells that exist)
    bool ilo, ihi, jlo, jhi, xse, yse, xsh, ysh, in_snap;
    float4 pxe, pye, pxm, pym;
};

// OWN: a cell this thread updates (E and H), else one whose E is evaluated.
template <class T, int V, bool OWN>
__device__ __forceinline__ FCol fcol(const KArgs &a, int i, int j)
{
    FCol c;
    const int nx = a.nx, ny = a.ny;
    c.valid = (!(V & V_X) || i < nx) && (!(V & V_Y) || j < ny);
    c.i = (V & V_X) ? min(i, a.px - 1) : i;
    c.j = (V & V_Y) ? min(j, ny - 1) : j;
    const u32 col = (u32)c.j * (u32)a.px + (u32)c.i;
    c.cell0 = col;
    c.o0 = (col + (u32)a.plane) * (u32)sizeof(T);
    c.mycol = c.j * nx + min(c.i, nx - 1);
    c.ilo = !(V & V_X) || i > 0;
    c.ihi = !(V & V_X) || i < nx - 1;
    c.jlo = !(V & V_Y) || j > 0;
    c.jhi = !(V & V_Y) || j < ny - 1;
    c.xse = (V & V_X) && c.valid && ((c.ilo && i < a.L[0]) || (i >= nx - a.L[1] && c.ihi));   // fdtdrav.h:752,777
    c.yse = (V & V_Y) && c.valid && ((c.jlo && j < a.L[2]) || (j >= ny - a.L[3] && c.jhi));   // fdtdrav.h:803,827
    c.xsh = OWN && (V & V_X) && c.valid && (i < a.L[0] || (i >= nx - a.L[1] && c.ihi));       // fdtdrav.h:402,424
    c.ysh = OWN && (V & V_Y) && c.valid && (j < a.L[2] || (j >= ny - a.L[3] && c.jhi));       // fdtdrav.h:447,471
    c.sx = i < a.L[0] ? i : i - (nx - a.L[1]) + a.L[0];
    c.sy = j < a.L[2] ? j : j - (ny - a.L[3]) + a.L[2];
    const float4 none = make_float4(0.f, 0.f, 1.f, 0.f);
    c.pxe = c.xse ? a.px_prof[i] : none;
    c.pye = c.yse ? a.py_prof[j] : none;
    c.pxm = c.xsh ? a.px_prof[nx + i] : none;
    c.pym = c.ysh ? a.py_prof[ny + j] : none;
    c.in_snap = OWN && a.snap != nullptr && c.valid && i >= a.sb[0] && i < a.sb[0] + a.sb[3] && j >= a.sb[1] &&
                j < a.sb[1] + a.sb[4];
    return c;
}

// Values plane k of a column reads.
struct FPlane {
    float hx, hy, hz, hy_im, hz_im, hx_jm, hz_jm, ex, ey, ez;
    float pe_yx, pe_zx, pe_xy, pe_zy, pe_xz, pe_yz;   // old psi_e of the slabs the cell is in
    float ph_yx, ph_zx, ph_xy, ph_zy, ph_xz, ph_yz;   // psi_h (own cells)
    int cln;                                            // class index of plane k+1
};

// Old field bases (guard plane below k = 0).
template <class T>
struct FBase {
    const T *ex, *ey, *ez, *hx, *hy, *hz;
};

// CX, CY, CZ: the E components evaluated.  SHIFT: the columns of a wave are
// adjacent cells (the x-neighbour is the previous lane's value; the load
// fills lane 0, one address for the wave).
template <class T, int CM, int V, bool OWN, bool CX, bool CY, bool CZ, bool SHIFT>
__device__ __forceinline__ void ffetch(FPlane &p, const KArgs &a, const FCol &c, const FBase<T> &f, int k, int k1)
{
    ConstKArgs &ra = rare_args(a);
    constexpr u32 S = sizeof(T);
    const u32 o = c.o0 + (u32)k * ((u32)a.plane * S);
    const u32 ojm = o - (u32)a.px * S;
    const u32 oim = (SHIFT ? (u32)__builtin_amdgcn_readfirstlane((int)o) : o) - S;
    if (CY || CZ) p.hx = ld(at(f.hx, o));
    if (CX || CZ) p.hy = ld(at(f.hy, o));
    if (CX || CY) p.hz = ld(at(f.hz, o));
    if (CZ) p.hy_im = ld(at(f.hy, oim));
    if (CY) p.hz_im = ld(at(f.hz, oim));
    if (CZ) p.hx_jm = ld(at(f.hx, ojm));
    if (CX) p.hz_jm = ld(at(f.hz, ojm));
    if (OWN) {
        p.ex = ldn(at(f.ex, o));
        p.ey = ldn(at(f.ey, o));
        p.ez = ldn(at(f.ez, o));
    } else {
        if (CX) p.ex = ld(at(f.ex, o));
        if (CY) p.ey = ld(at(f.ey, o));
        if (CZ) p.ez = ld(at(f.ez, o));
    }
    // class map (no guard planes): the entry of plane k+1, or the last plane's
    p.cln = CM != CLS_UNIFORM
                ? class_at<CM>(a.cls, (u32)min(k + 1, a.nz - 1) * (u32)a.plane + c.cell0)
                : 0;
    p.pe_yx = p.pe_zx = p.pe_xy = p.pe_zy = p.pe_xz = p.pe_yz = 0.f;
    const bool khi = !(V & V_Z) || k < a.nz - 1;
    if ((V & V_X) && c.xse && c.jhi && khi) {
        const u32 q = (((u32)k * ra.ny + c.j) * ra.Lx + c.sx) * S;
        if (CY) p.pe_yx = ld(at((const T *)ra.psi_eyx, q));
        if (CZ) p.pe_zx = ld(at((const T *)ra.psi_ezx, q));
    }
    if ((V & V_Y) && c.yse && c.ihi && khi) {
        const u32 q = (((u32)k * ra.Ly + c.sy) * ra.px + c.i) * S;
        if (CX) p.pe_xy = ld(at((const T *)ra.psi_exy, q));
        if (CZ) p.pe_zy = ld(at((const T *)ra.psi_ezy, q));
    }
    if (V & V_Z) {
        const int nz = a.nz;
        const int sz = k < a.L[4] ? k : k - (nz - a.L[5]) + a.L[4];
        const u32 q = (((u32)sz * ra.ny + c.j) * ra.px + c.i) * S;
        if ((CX || CY) && ((k > 0 && k < a.L[4]) || (k >= nz - a.L[5] && k < nz - 1)) && c.valid && c.ihi && c.jhi) {
            if (CX) p.pe_xz = ld(at((const T *)ra.psi_exz, q));
            if (CY) p.pe_yz = ld(at((const T *)ra.psi_eyz, q));
        }
        if (OWN) {
            p.ph_xz = p.ph_yz = 0.f;
            if (k < k1 && (k < a.L[4] || (k >= nz - a.L[5] && k < nz - 1)) && c.valid) {
                p.ph_xz = ld(at((const T *)ra.psi_hxz, q));
                p.ph_yz = ld(at((const T *)ra.psi_hyz, q));
            }
        }
    }
    if (OWN) {
        p.ph_yx = p.ph_zx = p.ph_xy = p.ph_zy = 0.f;
        if ((V & V_X) && c.xsh && k < k1) {
            const u32 q = (((u32)k * ra.ny + c.j) * ra.Lx + c.sx) * S;
            p.ph_yx = ld(at((const T *)ra.psi_hyx, q));
            p.ph_zx = ld(at((const T *)ra.psi_hzx, q));
        }
        if ((V & V_Y) && c.ysh && k < k1) {
            const u32 q = (((u32)k * ra.Ly + c.sy) * ra.px + c.i) * S;
            p.ph_xy = ld(at((const T *)ra.psi_hxy, q));
            p.ph_zy = ld(at((const T *)ra.psi_hzy, q));
        }
    }
}

// E^{m+1} at plane k of a column (calc_e and its CPML, as kernels.hip
// e_update).  store: an own cell's plane (psi is written, probes are
// recorded), else the value is only evaluated.
template <class T, int V, bool OWN, bool CX, bool CY, bool CZ, bool SHIFT>
__device__ __forceinline__ void fe_update(const FPlane &p, const Coef &t, const KArgs &a, const FCol &c, int k, int m,
                                          bool store, float hx_km, float hy_km, int &ev, int &ek, float &exn,
                                          float &eyn, float &ezn)
{
    ConstKArgs &ra = rare_args(a);
    const int nz = a.nz;
    constexpr u32 S = sizeof(T);
    const float hx = p.hx, hy = p.hy, hz = p.hz;
    const float hy_im = SHIFT ? lane_prev(hy, p.hy_im) : p.hy_im;
    const float hz_im = SHIFT ? lane_prev(hz, p.hz_im) : p.hz_im;
    const bool klo = !(V & V_Z) || k > 0, khi = !(V & V_Z) || k < nz - 1;
    const bool ux = c.ihi && c.jlo && c.jhi && klo && khi;
    const bool uy = c.ilo && c.ihi && c.jhi && klo && khi;
    const bool uz = c.ilo && c.ihi && c.jlo && c.jhi && khi;
    const bool zs = (V & V_Z) && ((k > 0 && k < a.L[4]) || (k >= nz - a.L[5] && k < nz - 1));   // fdtdrav.h:853,879

    float cbx_hz = t.x.y, cbx_hy = t.x.z, cby_hx = t.y.y, cby_hz = t.y.z, cbz_hy = t.z.y, cbz_hx = t.z.z;
    float4 pze = make_float4(0.f, 0.f, 1.f, 0.f);
    if (c.xse) {
        if (CY) cby_hz = cby_hz / c.pxe.z;
        if (CZ) cbz_hy = cbz_hy / c.pxe.z;
    }
    if (c.yse) {
        if (CX) cbx_hz = cbx_hz / c.pye.z;
        if (CZ) cbz_hx = cbz_hx / c.pye.z;
    }
    if (zs) {
        pze = uload(a.pz_prof + k);
        if (CX) cbx_hy = cbx_hy / pze.z;
        if (CY) cby_hx = cby_hx / pze.z;
    }
    if (CX) { exn = p.ex; if (ux) exn = (t.x.x * p.ex + cbx_hz * (hz - p.hz_jm)) + cbx_hy * (hy - hy_km); }
    if (CY) { eyn = p.ey; if (uy) eyn = (t.y.x * p.ey + cby_hx * (hx - hx_km)) + cby_hz * (hz - hz_im); }
    if (CZ) { ezn = p.ez; if (uz) ezn = (t.z.x * p.ez + cbz_hy * (hy - hy_im)) + cbz_hx * (hx - p.hx_jm); }

    if (CZ && k == ek) {   // source edges; probes of own cells
        while (ev >= 0 && ra.events[ev].k == k && ra.events[ev].col == c.mycol) {
            const Event e = ra.events[ev];
            if (e.kind == EV_SOURCE) {
                if (uz) {
                    const SrcEdge s = ra.srcs[e.id];
                    ezn = ((s.ceze * p.ez + s.cezhy * (hy - hy_im)) + s.cezhx * (hx - p.hx_jm)) +
                          s.cezj * ra.vpn[(i64)s.wave * ra.steps_cap + m];
                }
            } else if (OWN && store && ra.rec) {
                const int comp = e.kind - EV_PROBE;
                record_probe(ra, e.id, comp, comp == 0 ? exn : comp == 1 ? eyn : ezn, m);
            }
            ++ev;
        }
        ek = first_k(ra, ev, c.mycol);
    }

    // CPML psi recursions and corrections, fdtdrav.h:750-911
    const float dx = ra.d[0], dy = ra.d[1], dz = ra.d[2];
    if (c.xse && c.jhi && khi) {
        const u32 q = (((u32)k * ra.ny + c.j) * ra.Lx + c.sx) * S;
        const float pey = c.pxe.x * p.pe_yx + c.pxe.y * (hz - hz_im);
        const float pez = c.pxe.x * p.pe_zx + c.pxe.y * (hy - hy_im);
        if (OWN && store) {
            st(at((T *)ra.npsi_eyx, q), pey);
            st(at((T *)ra.npsi_ezx, q), pez);
        }
        if (CY && klo) eyn = eyn + (t.y.z * dx) * pey;
        if (CZ && c.jlo) ezn = ezn + (t.z.y * dx) * pez;
    }
    if (c.yse && c.ihi && khi) {
        const u32 q = (((u32)k * ra.Ly + c.sy) * ra.px + c.i) * S;
        const float pex = c.pye.x * p.pe_xy + c.pye.y * (hz - p.hz_jm);
        const float pez = c.pye.x * p.pe_zy + c.pye.y * (hx - p.hx_jm);
        if (OWN && store) {
            st(at((T *)ra.npsi_exy, q), pex);
            st(at((T *)ra.npsi_ezy, q), pez);
        }
        if (CX && klo) exn = exn + (t.x.y * dy) * pex;
        if (CZ && c.ilo) ezn = ezn + (t.z.z * dy) * pez;
    }
    if (zs && c.valid && c.ihi && c.jhi) {
        const int sz = k < a.L[4] ? k : k - (nz - a.L[5]) + a.L[4];
        const u32 q = (((u32)sz * ra.ny + c.j) * ra.px + c.i) * S;
        const float pex = pze.x * p.pe_xz + pze.y * (hy - hy_km);
        const float pey = pze.x * p.pe_yz + pze.y * (hx - hx_km);
        if (OWN && store) {
            st(at((T *)ra.npsi_exz, q), pex);
            st(at((T *)ra.npsi_eyz, q), pey);
        }
        if (CX && c.jlo) exn = exn + (t.x.z * dz) * pex;
        if (CY && c.ilo) eyn = eyn + (t.y.y * dz) * pey;
    }
    // the H half-step reads what is stored
    if (CX) exn = rnd(exn, (const T *)nullptr);
    if (CY) eyn = rnd(eyn, (const T *)nullptr);
    if (CZ) ezn = rnd(ezn, (const T *)nullptr);
    if (OWN && store && c.in_snap && k >= a.sb[2] && k < a.sb[2] + a.sb[5])
        e_snapshot(ra, c.i, c.j, k, m, exn, eyn, ezn);
}

// What a row's wave carries from plane k to plane k+1.
struct FCarry {
    float hx, hy, hz;        // old H(k)
    float ex, ey, ez;        // E^{m+1}(k)
    float ez_jp, ex_jp;      // ... at (i, j+1)
    float ez_f, ey_f;        // ... at the column after the tile (lane 63's x-neighbour)
    float ph_yx, ph_zx, ph_xy, ph_zy, ph_xz, ph_yz;
};

// H^{m+1} at plane k (calc_h and its CPML, as kernels.hip h_update); ex_kp,
// ey_kp = E^{m+1}(k+1).
template <class T, int V>
__device__ __forceinline__ void fh_update(const FCarry &q_, const Coef &t, const KArgs &a, const FCol &c, T *hxo,
                                          T *hyo, T *hzo, int k, int m, float ex_kp, float ey_kp, int &ev, int &ek)
{
    ConstKArgs &ra = rare_args(a);
    const int nz = a.nz;
    constexpr u32 S = sizeof(T);
    const u32 o = c.o0 + (u32)k * ((u32)a.plane * S);
    const float ex = q_.ex, ey = q_.ey, ez = q_.ez;
    const float ez_ip = lane_next(ez, q_.ez_f), ey_ip = lane_next(ey, q_.ey_f);
    const float ez_jp = q_.ez_jp, ex_jp = q_.ex_jp;
    const bool khi = !(V & V_Z) || k < nz - 1;
    const bool ux = c.jhi && khi, uy = c.ihi && khi, uz = c.ihi && c.jhi;
    const bool zs = (V & V_Z) && (k < a.L[4] || (k >= nz - a.L[5] && k < nz - 1)) && c.valid;   // fdtdrav.h:500,531

    float chx_ey = t.x.y, chx_ez = t.x.z, chy_ez = t.y.y, chy_ex = t.y.z, chz_ex = t.z.y, chz_ey = t.z.z;
    float4 pzm = make_float4(0.f, 0.f, 1.f, 0.f);
    if (c.xsh) { chy_ez = chy_ez / c.pxm.z; chz_ey = chz_ey / c.pxm.z; }
    if (c.ysh) { chx_ez = chx_ez / c.pym.z; chz_ex = chz_ex / c.pym.z; }
    if (zs) {
        pzm = uload(a.pz_prof + nz + k);
        chx_ey = chx_ey / pzm.z;
        chy_ex = chy_ex / pzm.z;
    }
    float hxn = q_.hx, hyn = q_.hy, hzn = q_.hz;
    if (ux) hxn = (t.x.x * q_.hx + chx_ey * (ey_kp - ey)) + chx_ez * (ez_jp - ez);
    if (uy) hyn = (t.y.x * q_.hy + chy_ez * (ez_ip - ez)) + chy_ex * (ex_kp - ex);
    if (uz) hzn = (t.z.x * q_.hz + chz_ex * (ex_jp - ex)) + chz_ey * (ey_ip - ey);

    if (k == ek) {   // probes on this cell
        const EvH r = h_events(ra, ev, k, c.mycol, m, hxn, hyn, hzn);
        ev = r.ev;
        ek = r.ek;
    }

    const float dx = ra.d[0], dy = ra.d[1], dz = ra.d[2];
    if (c.xsh) {
        const u32 q = (((u32)k * ra.ny + c.j) * ra.Lx + c.sx) * S;
        const float phy = c.pxm.x * q_.ph_yx + c.pxm.y * (ez_ip - ez);
        const float phz = c.pxm.x * q_.ph_zx + c.pxm.y * (ey_ip - ey);
        st(at((T *)ra.psi_hyx, q), phy);
        st(at((T *)ra.psi_hzx, q), phz);
        if (khi) hyn = hyn + (t.y.y * dx) * phy;
        if (c.jhi) hzn = hzn + (t.z.z * dx) * phz;
    }
    if (c.ysh) {
        const u32 q = (((u32)k * ra.Ly + c.sy) * ra.px + c.i) * S;
        const float phx = c.pym.x * q_.ph_xy + c.pym.y * (ez_jp - ez);
        const float phz = c.pym.x * q_.ph_zy + c.pym.y * (ex_jp - ex);
        st(at((T *)ra.psi_hxy, q), phx);
        st(at((T *)ra.psi_hzy, q), phz);
        if (khi) hxn = hxn + (t.x.z * dy) * phx;
        if (c.ihi) hzn = hzn + (t.z.y * dy) * phz;
    }
    if (zs) {
        const int sz = k < a.L[4] ? k : k - (nz - a.L[5]) + a.L[4];
        const u32 q = (((u32)sz * ra.ny + c.j) * ra.px + c.i) * S;
        const float phx = pzm.x * q_.ph_xz + pzm.y * (ey_kp - ey);
        const float phy = pzm.x * q_.ph_yz + pzm.y * (ex_kp - ex);
        st(at((T *)ra.psi_hxz, q), phx);
        st(at((T *)ra.psi_hyz, q), phy);
        if (c.jhi) hxn = hxn + (t.x.y * dz) * phx;
        if (c.ihi) hyn = hyn + (t.y.z * dz) * phy;
    }
    if (c.valid) {
        stn(at(hxo, o), hxn);
        stn(at(hyo, o), hyn);
        stn(at(hzo, o), hzn);
    }
}

// Workgroup barrier ordering LDS only: the loads of the next plane stay in
// flight across it.
__device__ __forceinline__ void lds_barrier()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// E values the rows of a plane share: ex, ez of rows 1 .. FY (row FY: beyond
// the tile) and ey, ez of the column after the tile.  Two buffers, planes in
// turn: a plane's is written again two planes later, after a barrier that
// every wave reaches only with its reads of it done.
struct FShare {
    float ex[2][FY + 1][TX], ez[2][FY + 1][TX];
    float cy[2][TX], cz[2][TX];
};

template <int CM>
__device__ __forceinline__ Coef ucoef(const float4 *tab)
{
    Coef t;
    t.x = uload(tab);
    t.y = uload(tab + 1);
    t.z = uload(tab + 2);
    return t;
}

// CM: class map of the E sweep, CH: of the H sweep.
template <class T, int CM, int CH, int V>
__global__ void __launch_bounds__(TX *(FY + 1))
__attribute__((amdgpu_waves_per_eu(4))) step_kernel(const KArgs a, const int m)
{
    __shared__ FShare sh;
    int tx, ty, tz;
    tile_of_region<V>(a, tx, ty, tz, blockIdx.x);
    const int lane = (int)(threadIdx.x & (TX - 1));
    const int w = __builtin_amdgcn_readfirstlane((int)(threadIdx.x / TX));
    const int i0 = tx * TX, j0 = ty * FY;
    const int k0 = tz * a.kchunk;
    const int k1 = min(a.nz, k0 + a.kchunk);
    constexpr u32 S = sizeof(T);
    const u32 ob = (u32)a.plane * S;
    const FBase<T> f{(const T *)a.ex - a.plane, (const T *)a.ey - a.plane, (const T *)a.ez - a.plane,
                     (const T *)a.hx - a.plane, (const T *)a.hy - a.plane, (const T *)a.hz - a.plane};

    if (w < FY) {
        // ---- a row of own cells: E(k), then H(k-1)
        const FCol c = fcol<T, V, true>(a, i0 + lane, j0 + w);
        T *__restrict__ exo = (T *)a.nex - a.plane;
        T *__restrict__ eyo = (T *)a.ney - a.plane;
        T *__restrict__ ezo = (T *)a.nez - a.plane;
        T *__restrict__ hxo = (T *)a.nhx - a.plane;
        T *__restrict__ hyo = (T *)a.nhy - a.plane;
        T *__restrict__ hzo = (T *)a.nhz - a.plane;
        int ev = c.valid ? first_event(a, a.e_first, c.mycol, k0) : -1;
        int ek = first_k(a, ev, c.mycol);
        int hv = c.valid ? first_event(a, a.h_first, c.mycol, k0) : -1;
        int hk = first_k(a, hv, c.mycol);
        FCarry q{};
        q.hx = ld(at(f.hx, c.o0 + (u32)(k0 - 1) * ob));
        q.hy = ld(at(f.hy, c.o0 + (u32)(k0 - 1) * ob));
        FPlane A, B;
        Coef tA, tB, tH;
        if (CM == CLS_UNIFORM) tA = tB = ucoef<CM>(a.etab);
        if (CH == CLS_UNIFORM) tH = ucoef<CH>(a.htab);
        const int c0 = (CM != CLS_UNIFORM || CH != CLS_UNIFORM)
                           ? class_at<CM != CLS_UNIFORM ? CM : CH>(a.cls, (u32)k0 * (u32)a.plane + c.cell0)
                           : 0;
        int cl = c0;
        constexpr int CF = CM != CLS_UNIFORM ? CM : CH;   // the class map is read when either sweep uses it
        if (CM != CLS_UNIFORM) tA = coef_of<CM>(a.etab, c0);
        ffetch<T, CF, V, true, true, true, true, true>(A, a, c, f, k0, k1);

        // plane k of the march (not the last: H(k) still to come)
        auto plane = [&](const FPlane &p, const Coef &t, int k) {
            float exn, eyn, ezn;
            fe_update<T, V, true, true, true, true, true>(p, t, a, c, k, m, true, q.hx, q.hy, ev, ek, exn, eyn, ezn);
            const u32 o = c.o0 + (u32)k * ob;
            if (c.valid) {
                stn(at(exo, o), exn);
                stn(at(eyo, o), eyn);
                stn(at(ezo, o), ezn);
            }
            const int b = (k - k0) & 1;
            if (w > 0) {
                sh.ex[b][w][lane] = exn;
                sh.ez[b][w][lane] = ezn;
            }
            if (k > k0) fh_update<T, V>(q, tH, a, c, hxo, hyo, hzo, k - 1, m, exn, eyn, hv, hk);
            lds_barrier();
            q.ex_jp = sh.ex[b][w + 1][lane];
            q.ez_jp = sh.ez[b][w + 1][lane];
            q.ey_f = sh.cy[b][w];
            q.ez_f = sh.cz[b][w];
            q.ex = exn;
            q.ey = eyn;
            q.ez = ezn;
            q.hx = carry(p.hx);
            q.hy = carry(p.hy);
            q.hz = carry(p.hz);
            q.ph_yx = p.ph_yx; q.ph_zx = p.ph_zx; q.ph_xy = p.ph_xy;
            q.ph_zy = p.ph_zy; q.ph_xz = p.ph_xz; q.ph_yz = p.ph_yz;
            if (CH != CLS_UNIFORM) {
                tH = coef_of<CH>(a.htab, cl);
                cl = p.cln;
            }
        };
        // the plane above the block: E for H(k1-1), nothing stored
        auto top = [&](const FPlane &p, const Coef &t) {
            float exn, eyn, ezn;
            fe_update<T, V, true, true, true, true, true>(p, t, a, c, k1, m, false, q.hx, q.hy, ev, ek, exn, eyn, ezn);
            fh_update<T, V>(q, tH, a, c, hxo, hyo, hzo, k1 - 1, m, exn, eyn, hv, hk);
        };
        for (int k = k0;; k += 2) {
            ffetch<T, CF, V, true, true, true, true, true>(B, a, c, f, k + 1, k1);
            if (CM != CLS_UNIFORM) tB = coef_of<CM>(a.etab, A.cln);
            plane(A, tA, k);
            if (k + 1 == k1) {
                top(B, tB);
                break;
            }
            ffetch<T, CF, V, true, true, true, true, true>(A, a, c, f, k + 2, k1);
            if (CM != CLS_UNIFORM) tA = coef_of<CM>(a.etab, B.cln);
            plane(B, tB, k + 1);
            if (k + 2 == k1) {
                top(A, tA);
                break;
            }
        }
    } else {
        // ---- the cells beyond the tile: E of row j0 + FY (ex, ez; one cell
        // per lane) and of column i0 + 64 (ey, ez; lane r: row j0 + r)
        const FCol cr = fcol<T, V, false>(a, i0 + lane, j0 + FY);
        const FCol cc = fcol<T, V, false>(a, i0 + TX, j0 + min(lane, FY - 1));
        int rv = cr.valid ? first_event(a, a.e_first, cr.mycol, k0) : -1;
        int rk = first_k(a, rv, cr.mycol);
        int xv = cc.valid ? first_event(a, a.e_first, cc.mycol, k0) : -1;
        int xk = first_k(a, xv, cc.mycol);
        float r_hy = ld(at(f.hy, cr.o0 + (u32)(k0 - 1) * ob));
        float x_hx = ld(at(f.hx, cc.o0 + (u32)(k0 - 1) * ob));
        FPlane RA, XA, RB, XB;
        Coef rA, xA, rB, xB;
        if (CM == CLS_UNIFORM) {
            rA = xA = rB = xB = ucoef<CM>(a.etab);
        } else {
            rA = coef_of<CM>(a.etab, class_at<CM>(a.cls, (u32)k0 * (u32)a.plane + cr.cell0));
            xA = coef_of<CM>(a.etab, class_at<CM>(a.cls, (u32)k0 * (u32)a.plane + cc.cell0));
        }
        auto fetch = [&](FPlane &r, FPlane &x, int k) {
            k = min(k, k1 - 1);
            ffetch<T, CM, V, false, true, false, true, true>(r, a, cr, f, k, k1);
            ffetch<T, CM, V, false, false, true, true, false>(x, a, cc, f, k, k1);
        };
        auto plane = [&](const FPlane &r, const FPlane &x, const Coef &tr, const Coef &tc, int k) {
            float exn = 0.f, eyn = 0.f, ezn = 0.f, exc = 0.f, eyc = 0.f, ezc = 0.f;
            fe_update<T, V, false, true, false, true, true>(r, tr, a, cr, k, m, false, 0.f, r_hy, rv, rk, exn, eyn, ezn);
            fe_update<T, V, false, false, true, true, false>(x, tc, a, cc, k, m, false, x_hx, 0.f, xv, xk, exc, eyc,
                                                             ezc);
            const int b = (k - k0) & 1;
            sh.ex[b][FY][lane] = exn;
            sh.ez[b][FY][lane] = ezn;
            sh.cy[b][lane] = eyc;
            sh.cz[b][lane] = ezc;
            r_hy = carry(r.hy);
            x_hx = carry(x.hx);
            lds_barrier();
        };
        fetch(RA, XA, k0);
        for (int k = k0;; k += 2) {
            fetch(RB, XB, k + 1);
            if (CM != CLS_UNIFORM) {
                rB = coef_of<CM>(a.etab, RA.cln);
                xB = coef_of<CM>(a.etab, XA.cln);
            }
            plane(RA, XA, rA, xA, k);
            if (k + 1 == k1) break;
            fetch(RA, XA, k + 2);
            if (CM != CLS_UNIFORM) {
                rA = coef_of<CM>(a.etab, RB.cln);
                xA = coef_of<CM>(a.etab, XB.cln);
            }
            plane(RB, XB, rB, xB, k + 1);
            if (k + 2 == k1) break;
        }
    }
}

// ---- launchers --------------------------------------------------------------
template <class T, int V>
static void launch_step_v(int em, int hm, const KArgs &a, int m, int nt, hipStream_t s)
{
    dim3 grid(nt), block(TX * (FY + 1));
    if (hm != CLS_UNIFORM) em = hm;   // (the E table has an entry per class either way)
#define GO(E, H) hipLaunchKernelGGL((step_kernel<T, E, H, V>), grid, block, 0, s, a, m)
    if (em == CLS_UNIFORM) GO(CLS_UNIFORM, CLS_UNIFORM);
    else if (em == CLS_U16 && hm == CLS_UNIFORM) GO(CLS_U16, CLS_UNIFORM);
    else if (em == CLS_U16) GO(CLS_U16, CLS_U16);
    else if (hm == CLS_UNIFORM) GO(CLS_U32, CLS_UNIFORM);
    else GO(CLS_U32, CLS_U32);
#undef GO
}

template <class T>
static hipError_t launch_step_t(int em, int hm, const KArgs &a, int m, hipStream_t s)
{
    int nb, nx, nzt, ng;
    region_tiles(a, nb, nx, nzt, ng);
    if (nb > 0) launch_step_v<T, V_IN>(em, hm, a, m, nb, s);
    if (nx > 0) launch_step_v<T, V_X>(em, hm, a, m, nx, s);
    if (ng > 0) launch_step_v<T, V_GEN>(em, hm, a, m, ng, s);
    return hipGetLastError();
}

// One fused step of FP32 fields.  em, hm: ClassMode of the E and the H half-step.
hipError_t launch_step(int em, int hm, const KArgs &a, int m, hipStream_t s)
{
    return launch_step_t<float>(em, hm, a, m, s);
}

int fused_rows() { return FY; }

}  // namespace fdtd
