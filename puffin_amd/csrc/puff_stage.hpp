// Device helpers shared by the forward RK4 stage kernels (puff_push.hip) and
// their adjoints (puff_adjoint.hip): cell location, undulator fields, the
// workgroup's cell box and the weighted scatter onto the mesh.
//
// Reference arithmetic restated (UKFELs/Puffin):
//   getInterps_3D   interaction/system_interpolation.f90:25-98
//   1-D branch      interaction/system_interpolation_1D.f90:24-179
//   getSource_3D    interaction/system_interpolation.f90:150-248
//   b-fields        undulator/bfields.f90:36-881 (per-stage coefficients are
//                   computed on the host, see stage_scalars in puff_ctx.hip)
#pragma once

#include "puff_common.hpp"
#include "puff_kernels.hpp"

namespace puff {

// A value through an empty asm statement: computed here, not later.
template <typename T>
__device__ __forceinline__ void hold(T& v) {
    asm volatile("" : "+v"(v));
}

// Cell of one particle and its interpolation fractions.  ix and iy share a
// register (an FFT line fits a workgroup's LDS, so both are below 2^13).
template <typename R>
struct Cell {
    int ixy, iz0;
    R fx, fy, fz;   // x_in2, y_in2, z2_in2
    __device__ __forceinline__ int ix() const { return ixy & 0xffff; }
    __device__ __forceinline__ int iy() const { return ixy >> 16; }
};

// Node and fractions of a particle (getInterps_3D / _1D).  Returns flag bits;
// 0 means every node index is inside the mesh.
template <typename R>
__device__ __forceinline__ int locate(const MeshGeom& m, R x, R y, double z2,
                                      Cell<R>& c) {
    int flag = 0;
    const double zq = floor(z2 * m.inv_dz2);
    if (m.periodic) {
        if (!(fabs(zq) < 1.0e9)) return FLAG_Z2MESH;
        long long q = (long long)zq;
        long long r = q % m.nzp;
        if (r < 0) r += m.nzp;
        c.iz0 = (int)r;
    } else {
        // temporal mesh: z2node >= NZ2 stops the reference
        // (system_interpolation.f90:70-75); z2 < 0 is refused too.
        if (!(zq >= 0.0 && zq <= (double)(m.nzp - 2))) return FLAG_Z2MESH;
        c.iz0 = (int)zq;
    }
    const double locz2 = z2 - zq * m.dz2;
    c.fz = (R)(locz2 * m.inv_dz2);
    if (m.one_d) {
        c.ixy = 0;
        c.fx = 0;
        c.fy = 0;
        return 0;
    }
    const MeshScale<R>& q = m.template scale<R>();
    const R tx = (x + q.halfx) * q.inv_dx;
    const R ty = (y + q.halfy) * q.inv_dy;
    const R xq = floor(tx), yq = floor(ty);
    // xnode >= nspinDX .or. xnode < 1 (system_interpolation.f90:60-68)
    if (!(xq >= (R)0 && xq <= (R)(m.nx - 2))) flag |= FLAG_TRANSVERSE;
    if (!(yq >= (R)0 && yq <= (R)(m.ny - 2))) flag |= FLAG_TRANSVERSE;
    if (flag) return flag;
    c.ixy = (int)xq | ((int)yq << 16);
    c.fx = (x + q.halfx - xq * q.dx) * q.inv_dx;
    c.fy = (y + q.halfy - yq * q.dy) * q.inv_dy;
    return 0;
}

// 1 / a by the hardware's estimate and two Newton steps: the bits of the correctly
// rounded divide (no difference in 10^9 draws from 1e-30 to 1e30), in half its
// instructions.
__device__ __forceinline__ double reciprocal(double a) {
    double r = __builtin_amdgcn_rcp(a);
    r = fma(r, fma(-a, r, 1.0), r);
    return fma(r, fma(-a, r, 1.0), r);
}

// p2 (gamma_to_p2.f90:84-85) and (1 + eta p2) / Gamma of one macroparticle,
// in FP64.  The difference 1/sqrt(D) - 1 loses a factor 1/eta of its digits,
// so the root and its reciprocal are formed with the bits of the correctly
// rounded sqrt and divide (no difference in 10^9 draws over gamma_r 10 to
// 1e4): the estimate of 1/sqrt(D), one coupled
// Newton step for the root r and h = 1/(2 r), one for the residue of r, one
// for that of 1/r;
// 28 instructions instead of 45.
// Without contraction and with its FMAs written out, as in rates(): a stage
// forms the previous trial state's derivatives of x, y and z2 again, and they
// are the bits that the previous stage checked its successor's trial position
// with.
struct Drift {
    double p2, fac;
};

__device__ __forceinline__ Drift drift_of(const Physics& ph, double pr, double pi, double g) {
#pragma clang fp contract(off)
    const double invg = __builtin_amdgcn_div_fixup(reciprocal(g), g, 1.0);   // as 1/g at 0, infinity and NaN
    const double D = fma(-(ph.inv_gr2 * invg * invg), fma(ph.aw2, fma(pr, pr, pi * pi), 1.0), 1.0);
    const double y = __builtin_amdgcn_rsq(D);
    const double r0 = D * y, h0 = 0.5 * y;
    const double e = fma(-h0, r0, 0.5);
    const double r1 = fma(r0, e, r0), h1 = fma(h0, e, h0);
    const double r = fma(fma(-r1, r1, D), h1, r1);
    const double q = h1 + h1;
    const double um1 = fma(q, fma(-r, q, 1.0), q) - 1.0;
    return {um1 * ph.inv_eta, fma(um1, invg, invg)};
}

// Derivatives of x, y and z2 (puffin_equations.f90:115-117, 144-146, 172):
// zero when the electrons do not evolve (rhs.f90:301-308).  z2's is rounded to
// the type of the stored derivatives, as k_1 to k_3 of the momenta are.
template <typename R>
struct Rates {
    R x, y;
    double z2;
};

template <typename R>
__device__ __forceinline__ Rates<R> rates(const Physics& ph, const Drift& d, R pr, R pi) {
#pragma clang fp contract(off)
    if (!ph.electrons_evolve) return {(R)0, (R)0, 0.0};
    const R v = ph.template scale<R>().c_dx * (R)d.fac;
    return {v * pr, -v * pi, (double)(R)d.p2};
}

// Trial state y0 + c k_{s-1} of one macroparticle (puffin_mpi_RK4.f90:190-195
// etc.): p_r, p_i and Gamma from the stored derivative, x, y and z2 from the
// rates of the previous trial state's momenta, y0 + cprev k_{s-2} (those of
// y0 itself in stage 2).
template <typename R>
struct Trial {
    R x, y, pr, pi;
    double z2, g;
    Rates<R> v;     // rates of the previous trial state
};

template <typename R, int STAGE>
__device__ __forceinline__ Trial<R> trial_state(const Physics& ph, R x0, R y0, double z20, R pr0, R pi0, double g0,
                                                R kr, R ki, R kg, R qr, R qi, R qg, double cin, double cprev, R c,
                                                R cp) {
    Trial<R> t;
    R ppr = pr0, ppi = pi0;
    double pg = g0;
    if (STAGE > 2) {
        ppr = fma(cp, qr, pr0);
        ppi = fma(cp, qi, pi0);
        pg = fma(cprev, (double)qg, g0);
    }
    t.v = rates<R>(ph, drift_of(ph, (double)ppr, (double)ppi, pg), ppr, ppi);
    t.x = fma(c, t.v.x, x0);
    t.y = fma(c, t.v.y, y0);
    t.z2 = fma(cin, t.v.z2, z20);
    t.pr = fma(c, kr, pr0);
    t.pi = fma(c, ki, pi0);
    t.g = fma(cin, (double)kg, g0);
    return t;
}

// Scaled undulator field at one particle from the stage coefficients
// (bfields.f90): see stage_scalars() on the host for the coefficient map.
// POLE = false: compiled without the hyperbolic functions of the plane-pole
// and curved-pole types (15 to 20 registers of a stage kernel).
// Which product of a sum of two is rounded is written out: left to the compiler
// it changes with the code around, and the mixed form's z2 by up to 1.4e-9 over 25
// steps of a focusing curved-pole undulator.
template <typename R, bool POLE = true>
__device__ __forceinline__ void bfield(const StageScalars& s, R x, R y, R& bx,
                                       R& by, R& bz) {
    if (POLE && s.und_type == PUFF_UND_PLANEPOLE) {
        bx = s.template coef<R>(3) * y;
        by = s.template coef<R>(1) + s.template coef<R>(4) * x;
        bz = s.template coef<R>(2) * sinh(s.template coef<R>(7) * y);
    } else if (POLE && s.und_type == PUFF_UND_CURVED) {
        const R kx = s.template coef<R>(5), ky = s.template coef<R>(6);
        bx = fma(s.template coef<R>(3), y, s.template coef<R>(0) * sinh(kx * x) * sinh(ky * y));
        by = fma(s.template coef<R>(4), x, s.template coef<R>(1) * cosh(kx * x) * cosh(ky * y));
        bz = s.template coef<R>(2) * cosh(kx * x) * sinh(ky * y);
    } else {
        bx = s.template coef<R>(0) + s.template coef<R>(3) * y;
        by = s.template coef<R>(1) + s.template coef<R>(4) * x;
        bz = fma(s.template coef<R>(6), y, s.template coef<R>(5) * x);
    }
}

// Transverse derivatives of bfield(): g = {dbx/dx, dbx/dy, dby/dx, dby/dy,
// dbz/dx, dbz/dy}.
__device__ __forceinline__ void bfield_grad(const StageScalars& s, double x, double y,
                                            double g[6]) {
    g[0] = 0.0;
    g[1] = s.c[3];
    g[2] = s.c[4];
    g[3] = 0.0;
    if (s.und_type == PUFF_UND_PLANEPOLE) {
        g[4] = 0.0;
        g[5] = s.c[2] * s.c[7] * cosh(s.c[7] * y);
    } else if (s.und_type == PUFF_UND_CURVED) {
        const double kx = s.c[5], ky = s.c[6];
        const double shx = sinh(kx * x), chx = cosh(kx * x), shy = sinh(ky * y), chy = cosh(ky * y);
        g[0] = s.c[0] * kx * chx * shy;
        g[1] += s.c[0] * ky * shx * chy;
        g[2] += s.c[1] * kx * shx * chy;
        g[3] = s.c[1] * ky * chx * shy;
        g[4] = s.c[2] * kx * shx * shy;
        g[5] = s.c[2] * ky * chx * chy;
    } else {
        g[4] = s.c[5];
        g[5] = s.c[6];
    }
}

template <typename R>
__device__ __forceinline__ void atomic_add(R* p, R v) {
    unsafeAtomicAdd(p, v);
}

// Node box of the cells of one workgroup (origin and extent in nodes, i.e.
// cells + 1), and the step's active box: one atomic per workgroup into one
// of BOX_COPIES spread copies (same-address atomics would serialise).  Must
// be reached by every thread of the workgroup.
struct TileBox {
    int bx0, by0, bz0;
    int tx, ty, tz;
    int hz;        // last cell plane
    bool any;
    int extra;     // block maximum of workgroup_box's `extra` (NX = 7)
};

// Lane's cell bounds over its macroparticles: x, y, z2 as (lo, -hi), so that
// every entry reduces by minimum; and `extra` (negated, a block maximum).
struct LaneBox {
    int v[7];
};

__device__ __forceinline__ LaneBox lane_box() {
    return {{0x7fffffff, 1, 0x7fffffff, 1, 0x7fffffff, 1, 0}};
}

template <typename R>
__device__ __forceinline__ void lane_box_add(LaneBox& b, bool ok, const Cell<R>& c, int extra = 0) {
    if (ok) {
        b.v[0] = min(b.v[0], c.ix());
        b.v[1] = min(b.v[1], -c.ix());
        b.v[2] = min(b.v[2], c.iy());
        b.v[3] = min(b.v[3], -c.iy());
        b.v[4] = min(b.v[4], c.iz0);
        b.v[5] = min(b.v[5], -c.iz0);
    }
    b.v[6] = min(b.v[6], -extra);
}

// Minima of the workgroup's wavefronts (LDS), for workgroup_box.
struct WaveBoxes {
    int v[MAX_BOX_WAVES][8];
};

// Box of a set of minima, all lanes equal (scalar values from here on).
template <int NX>
__device__ __forceinline__ TileBox tile_box(const MeshGeom& m, const int (&r)[NX]) {
    int v[NX];
#pragma unroll
    for (int d = 0; d < NX; ++d) v[d] = __builtin_amdgcn_readfirstlane(r[d]);
    TileBox t;
    t.extra = 0;
    if constexpr (NX > 6) t.extra = -v[6];
    t.any = v[1] <= 0;
    t.bx0 = v[0];
    t.by0 = v[2];
    t.bz0 = v[4];
    t.hz = -v[5];
    t.tx = t.any ? (m.one_d ? 1 : -v[1] - t.bx0 + 2) : 0;
    t.ty = t.any ? (m.one_d ? 1 : -v[3] - t.by0 + 2) : 0;
    t.tz = t.any ? -v[5] - t.bz0 + 2 : 0;
    return t;
}

// NX = 7 also reduces `extra` to its block maximum, returned in
// TileBox::extra.  One barrier: every thread combines the wavefronts' minima
// itself.
template <int NX = 6>
__device__ __forceinline__ TileBox workgroup_box(const MeshGeom& m, const LaneBox& lb, Box* box, WaveBoxes& s_red) {
    const int lane = threadIdx.x & 63;
    const int wv = threadIdx.x >> 6;
    int v[NX];
#pragma unroll
    for (int d = 0; d < NX; ++d) v[d] = wave_min(lb.v[d]);
    if (lane == 0) {
#pragma unroll
        for (int d = 0; d < NX; ++d) s_red.v[wv][d] = v[d];
    }
    __syncthreads();
#pragma unroll
    for (int d = 0; d < NX; ++d) {
        int r = s_red.v[0][d];
#pragma unroll
        for (int k = 1; k < MAX_BOX_WAVES; ++k) r = min(r, s_red.v[k][d]);
        v[d] = r;
    }
    const TileBox t = tile_box<NX>(m, v);
    if (t.any && threadIdx.x < 6) {
        const int d = threadIdx.x >> 1;
        Box* b = box + (blockIdx.x % BOX_COPIES);
        const int lo = d == 0 ? v[0] : (d == 1 ? v[2] : v[4]), hi = d == 0 ? v[1] : (d == 1 ? v[3] : v[5]);
        if (threadIdx.x & 1) atomicMax(&b->hi[d], -hi);
        else atomicMin(&b->lo[d], lo);
    }
    return t;
}

// Box of wavefront k of the workgroup.
__device__ __forceinline__ TileBox wave_box(const MeshGeom& m, const WaveBoxes& s_red, int k) {
    int v[6];
#pragma unroll
    for (int d = 0; d < 6; ++d) v[d] = s_red.v[k][d];
    return tile_box<6>(m, v);
}

// Node q of a box -> (lx, ly, lz), x fastest, without integer division: the
// quotients come from the hardware reciprocal of the box extents (v_rcp_f32,
// within 1 ulp), exact while q < 2^21 (the relative error of
// (q + 1/2) * rcp(t), below 2^-22, keeps it within the distance 1/(2t) of
// (q + 1/2)/t from the next integer); boxes here hold at most a few thousand
// nodes.  (A correctly rounded 1/t is a 12-instruction sequence, twice per
// box: 6 % of a mixed-form stage kernel's VALU instructions.)
struct BoxDiv {
    int tx, ty;
    float inv_tx, inv_ty;
};

__device__ __forceinline__ BoxDiv box_div(const TileBox& t) {
    return BoxDiv{t.tx, t.ty, __builtin_amdgcn_rcpf((float)t.tx), __builtin_amdgcn_rcpf((float)t.ty)};
}

__device__ __forceinline__ void box_coords(const BoxDiv& d, int q, int& lx, int& ly, int& lz) {
    const int r = (int)(((float)q + 0.5f) * d.inv_tx);
    lx = q - r * d.tx;
    lz = (int)(((float)r + 0.5f) * d.inv_ty);
    ly = r - lz * d.ty;
}

// Union of the spread box copies, one copy per lane and six wavefront
// reductions.  Every lane of the wavefront must be active.  (Each thread
// reading all 64 copies in turn is a chain of 384 loads: it held the field
// combination at 24 us on any mesh, however small.)
__device__ __forceinline__ Box merged_box(const Box* box) {
    static_assert(BOX_COPIES == 64, "one copy per lane");
    const Box mine = box[threadIdx.x & 63];
    Box b;
#pragma unroll
    for (int d = 0; d < 3; ++d) {
        b.lo[d] = wave_min(mine.lo[d]);
        b.hi[d] = wave_max(mine.hi[d]);
    }
    return b;
}

// f(ix, iy, iz) for every node that the cells of box b touch (all planes of a
// periodic mesh), x fastest, over the whole grid of workgroups.  The indexes
// are split with 32-bit divisions where they fit (a 64-bit one is some hundred
// instructions).  With the skipped nodes of k_field_combine: 104 -> 97 us on
// 129 x 129 x 1024 with 2^24 macroparticles (FP64), 56 -> 53 us (mixed).
template <typename F>
__device__ __forceinline__ void each_active_node(const Box& b, int nx, int ny, int nzp, int periodic, int one_d, F f) {
    if (b.hi[0] < 0) return;   // no particle deposited
    const int x0 = b.lo[0], x1 = min(b.hi[0] + 1, nx - 1);
    const int y0 = one_d ? 0 : b.lo[1], y1 = one_d ? 0 : min(b.hi[1] + 1, ny - 1);
    const int z0 = periodic ? 0 : b.lo[2];
    const int z1 = periodic ? nzp - 1 : min(b.hi[2] + 1, nzp - 1);
    const uint32_t lx = (uint32_t)(x1 - x0 + 1), ly = (uint32_t)(y1 - y0 + 1);
    const int64_t vol = (int64_t)lx * ly * (z1 - z0 + 1);
    const int64_t first = (int64_t)blockIdx.x * blockDim.x + threadIdx.x, step = (int64_t)gridDim.x * blockDim.x;
    for (int64_t t = first; t < vol; t += step) {
        uint32_t x, r;
        if (vol <= 0xffffffffll) {
            r = (uint32_t)t / lx;
            x = (uint32_t)t - r * lx;
        } else {
            r = (uint32_t)(t / lx);   // a row: fewer than 2^32
            x = (uint32_t)(t - (int64_t)r * lx);
        }
        const uint32_t z = r / ly;
        f(x0 + (int)x, y0 + (int)(r - z * ly), z0 + (int)z);
    }
}

template <typename R>
__device__ __forceinline__ bool all_zero(const cplx<R>& a, const cplx<R>& b) {
    return a.x == (R)0 && a.y == (R)0 && b.x == (R)0 && b.y == (R)0;
}

// Whether the workgroup's node box fits the LDS tile and does not wrap
// around a periodic mesh (block-uniform).
template <int TILE>
__device__ __forceinline__ bool tile_fits(const MeshGeom& m, const TileBox& t) {
    return t.any && (int64_t)t.tx * t.ty * t.tz <= TILE && !(m.periodic && t.hz + 1 >= m.nzp);
}

// Nodes of a lane's cell: first node of its lower (b0) and upper (b1)
// z2 plane, its first node in the workgroup's tile (t0), and its key
// (unique negative key on lanes without a cell).
struct CellRef {
    int b0, b1, t0, key;
};

template <typename R>
__device__ __forceinline__ CellRef cell_ref(const MeshGeom& m, bool ok, const Cell<R>& c,
                                            const TileBox& t, int lane) {
    CellRef r;
    // the upper z2 plane, wrapping on a periodic mesh (on a temporal mesh
    // locate keeps iz0 below nzp - 1)
    const int iz1 = (c.iz0 + 1 == m.nzp) ? 0 : c.iz0 + 1;
    if (m.one_d) {
        r.b0 = ok ? c.iz0 : 0;
        r.b1 = ok ? iz1 : 0;
        r.t0 = ok ? c.iz0 - t.bz0 : 0;
        r.key = ok ? c.iz0 : -1 - lane;
        return r;
    }
    const int ntr = m.nx * m.ny;
    r.b0 = ok ? c.iz0 * ntr + c.iy() * m.nx + c.ix() : 0;
    r.b1 = ok ? iz1 * ntr + c.iy() * m.nx + c.ix() : 0;
    r.t0 = ok ? ((c.iz0 - t.bz0) * t.ty + (c.iy() - t.by0)) * t.tx + (c.ix() - t.bx0) : 0;
    r.key = ok ? r.b0 : -1 - lane;
    return r;
}

// Weight and node of corner k of a lane's cell, in getInterps_3D's order
// (x fastest, then y, then z2): w = (1-fx | fx)(1-fy | fy)(1-fz | fz).
// 1-D: lis_GR(1) = 1 - locz2/dz2, lis_GR(2) = 1 - lis_GR(1) at nodes iz0, iz1.
template <typename R>
__device__ __forceinline__ R corner_weight(const MeshGeom& m, const Cell<R>& c, int k) {
    if (m.one_d) {
        const R w0 = (R)1 - c.fz;
        return k ? (R)1 - w0 : w0;
    }
    const R wx = (k & 1) ? c.fx : (R)1 - c.fx;
    const R wy = (k & 2) ? c.fy : (R)1 - c.fy;
    const R wz = (k & 4) ? c.fz : (R)1 - c.fz;
    return wx * wy * wz;
}

// The eight corners of a lane's 3-D cell at once, for the LDS-tile paths:
// weights w = (wx wy) wz as corner_weight forms them, and tile offsets.
// Corner label q stands for corner k = q ^ rot (rot < 8): visiting the
// labels 0..7 in order with rot = lane mod 8 sends the lanes of one cell to
// different corners at each visit, so that an instruction's LDS atomics do
// not pile onto one word.  rot = 0: getInterps_3D's order.  Formed once per
// lane: the per-corner selects of corner_weight / corner_tile under a
// lane-dependent order cost about 25 VALU instructions per corner.
template <typename R>
struct CornerSet {
    R xy[4];     // wx wy of labels 0..3 (x, then y)
    R z[2];      // wz of the labels' z plane (labels 0-3, 4-7)
    int oxy[4];  // tile offset of labels 0..3 within the z plane
    int oz[2];   // tile offset of the two z planes
};

template <typename R>
__device__ __forceinline__ CornerSet<R> corner_set(const Cell<R>& c, const TileBox& t, int rot) {
    const R ux = (R)1 - c.fx, uy = (R)1 - c.fy, uz = (R)1 - c.fz;
    const bool rx = rot & 1, ry = rot & 2, rz = rot & 4;
    const R ax0 = rx ? c.fx : ux, ax1 = rx ? ux : c.fx;
    const R ay0 = ry ? c.fy : uy, ay1 = ry ? uy : c.fy;
    CornerSet<R> s;
    s.xy[0] = ax0 * ay0;
    s.xy[1] = ax1 * ay0;
    s.xy[2] = ax0 * ay1;
    s.xy[3] = ax1 * ay1;
    s.z[0] = rz ? c.fz : uz;
    s.z[1] = rz ? uz : c.fz;
    const int ox0 = rx ? 1 : 0, ox1 = 1 - ox0;
    const int oy0 = ry ? t.tx : 0, oy1 = t.tx - oy0;
    s.oxy[0] = ox0 + oy0;
    s.oxy[1] = ox1 + oy0;
    s.oxy[2] = ox0 + oy1;
    s.oxy[3] = ox1 + oy1;
    const int txy = t.tx * t.ty;
    s.oz[0] = rz ? txy : 0;
    s.oz[1] = txy - s.oz[0];
    return s;
}

__device__ __forceinline__ int corner_node(const MeshGeom& m, const CellRef& r, int k) {
    if (m.one_d) return k ? r.b1 : r.b0;
    return ((k & 4) ? r.b1 : r.b0) + (k & 1) + ((k & 2) ? m.nx : 0);
}

__device__ __forceinline__ int corner_tile(const MeshGeom& m, const TileBox& t, const CellRef& r, int k) {
    if (m.one_d) return r.t0 + k;
    return r.t0 + (k & 1) + ((k & 2) ? t.tx : 0) + ((k & 4) ? t.tx * t.ty : 0);
}

// The deposit out[node_k] += w_k (sr, si) of a workgroup, in one of three ways:
//   an LDS tile over the workgroup's node box (real parts, then imaginary
//     parts; element type D), cleared (tile_clear), added to by every lane
//     with a cell (tile_add) and flushed with one global atomic per touched
//     node and component (tile_flush), a barrier between each.  Each lane
//     visits the corners in a rotated order so that lanes of one cell do not
//     hit the same LDS address in the same instruction;
//   where the workgroup's box does not fit the tile, the same for one
//     wavefront after the other (tile_deposit): a run of slots that crosses
//     from one row of bricks to the next has a box across the whole beam, but
//     only in the one wavefront that holds the crossing;
//   global_add, for a wavefront whose own box does not fit: lanes of a
//     wavefront that share a cell are summed first (runs of equal keys), then
//     one global atomic per run and corner (sr = si = 0 on lanes without a
//     cell; all lanes call).

template <typename D>
__device__ __forceinline__ void tile_clear(D* tile, int words) {
    for (int q = threadIdx.x; q < words; q += blockDim.x) tile[q] = (D)0;
}

template <typename R, typename D>
__device__ __forceinline__ void tile_add(const MeshGeom& m, const TileBox& t, const Cell<R>& c, const CellRef& cr,
                                         R sr, R si, D* s_tile) {
    const int lane = threadIdx.x & 63;
    const int nt = t.tx * t.ty * t.tz;
    const D dsr = (D)sr, dsi = (D)si;
    if (!m.one_d) {
        const CornerSet<R> cs = corner_set<R>(c, t, lane & 7);
#pragma unroll
        for (int q = 0; q < 8; ++q) {
            const D wk = (D)(cs.xy[q & 3] * cs.z[q >> 2]);
            const int tk = cr.t0 + cs.oxy[q & 3] + cs.oz[q >> 2];
            atomicAdd(&s_tile[tk], wk * dsr);
            atomicAdd(&s_tile[nt + tk], wk * dsi);
        }
    } else {
        for (int q = 0; q < 2; ++q) {
            const int k = (q + lane) & 1;
            const D wk = (D)corner_weight<R>(m, c, k);
            const int tk = corner_tile(m, t, cr, k);
            atomicAdd(&s_tile[tk], wk * dsr);
            atomicAdd(&s_tile[nt + tk], wk * dsi);
        }
    }
}

// Lanes 2j and 2j + 1 take the real and imaginary parts of node j, so that one
// atomic instruction covers both parts of 32 nodes (each device-scope atomic
// is a memory-side request per 32-byte sector and instruction: half the
// requests of one instruction per part).
template <typename R, typename D>
__device__ __forceinline__ void tile_flush(const MeshGeom& m, const TileBox& t, cplx<R>* out, const D* s_tile) {
    const int nt = t.tx * t.ty * t.tz;
    const int ntr = m.nx * m.ny;
    const BoxDiv bd = box_div(t);
    R* outc = reinterpret_cast<R*>(out);
    for (int e = threadIdx.x; e < 2 * nt; e += blockDim.x) {
        const int q = e >> 1, part = e & 1;
        const D v = s_tile[part * nt + q];
        if (v != (D)0) {
            int lx, ly, lz;
            box_coords(bd, q, lx, ly, lz);
            const int node = (t.bz0 + lz) * ntr + (t.by0 + ly) * m.nx + (t.bx0 + lx);
            atomic_add(outc + node_component(node, part), (R)v);
        }
    }
}

template <typename R>
__device__ __forceinline__ void global_add(const MeshGeom& m, bool ok, const Cell<R>& c, const CellRef& cr, R sr,
                                           R si, cplx<R>* out) {
    const int lane = threadIdx.x & 63;
    const int nnb = m.one_d ? 2 : 8;
    const int prev = __shfl_up(cr.key, 1, 64);
    const bool head = (lane == 0) || (prev != cr.key);
    const unsigned long long heads = __ballot(head);
    const unsigned long long after = (lane == 63) ? 0ull : (heads >> (lane + 1));
    const int seg_end = after ? lane + __builtin_ctzll(after) : 63;
    const int maxlen = wave_max(head ? seg_end - lane + 1 : 1);
#pragma unroll
    for (int k = 0; k < 8; ++k) {
        if (k < nnb) {
            const R wk = ok ? corner_weight<R>(m, c, k) : (R)0;
            R vr = wk * sr, vi = wk * si;
            for (int o = 1; o < maxlen; o <<= 1) {
                const R tr = __shfl_down(vr, o, 64);
                const R ti = __shfl_down(vi, o, 64);
                if (lane + o <= seg_end) {
                    vr += tr;
                    vi += ti;
                }
            }
            if (ok && head) {
                const int node = corner_node(m, cr, k);
                atomic_add(&out[node].x, vr);
                atomic_add(&out[node].y, vi);
            }
        }
    }
}

// The tile deposits of a workgroup: add(t) (the lanes of the box t) and
// flush(t), once for the whole workgroup when its box fits the tile (which is
// clear then, a barrier passed), else for one wavefront after the other, with
// clear(t) before and spill() on the lanes of a wavefront whose own box does
// not fit.  One loop for both, so that the code is there once: the two
// together, inlined, took 18 to 40 registers more.
// 2^20 macroparticles on 129 x 129 x 1024 (14 to 23 % of the FP64 workgroups
// do not fit): a stage 200 us with global atomics for the whole workgroup, 97
// wavefront by wavefront; 2 10^5 of them (all workgroups): 147 and 80 us.  With
// 2^24 (0.8 %) no change.  (Mixed form: k_stage.)
template <int TILE, typename C, typename A, typename F, typename S>
__device__ __forceinline__ void tile_deposit(const MeshGeom& m, const TileBox& tb, bool whole,
                                             const WaveBoxes& s_red, C clear, A add, F flush, S spill) {
    const int wv = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int groups = whole ? 1 : MAX_BOX_WAVES;
#pragma unroll 1
    for (int k = 0; k < groups; ++k) {
        TileBox t = tb;
        if (!whole) {
            t = wave_box(m, s_red, k);
            if (!t.any) continue;
            if (!tile_fits<TILE>(m, t)) {
                if (wv == k) spill();
                continue;
            }
            __syncthreads();   // the tile may be in use
            clear(t);
            __syncthreads();
        }
        if (whole || wv == k) add(t);
        __syncthreads();
        flush(t);
    }
}

// The mixed form's deposit wavefront by wavefront: FP64 words, the real parts and
// then the imaginary ones of a box's nodes, both at once where 2 nt words fit
// the tile's WORDS, else one after the other.  Apart from the workgroup's own
// (packed) deposit: in one loop with it, as tile_deposit, a step of 2^24
// macroparticles took 1545 instead of 1470 us.  The corners in a loop: unrolled
// they take the kernel from 78 to 127 registers (1760 us).
template <int WORDS, typename R, typename S>
__device__ __forceinline__ void wave_deposit(const MeshGeom& m, const WaveBoxes& s_red, bool ok, const Cell<R>& c,
                                             R sr, R si, double* tile, cplx<R>* out, S spill) {
    const int wv = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int lane = threadIdx.x & 63;
    const int ntr = m.nx * m.ny;
    R* outc = reinterpret_cast<R*>(out);
#pragma unroll 1
    for (int k = 0; k < MAX_BOX_WAVES; ++k) {
        const TileBox t = wave_box(m, s_red, k);
        if (!t.any) continue;
        if (!tile_fits<WORDS>(m, t)) {
            if (wv == k) spill();
            continue;
        }
        const int nt = t.tx * t.ty * t.tz;
        const bool both = 2 * nt <= WORDS;
        const BoxDiv bd = box_div(t);
#pragma unroll 1
        for (int part = 0; part < (both ? 1 : 2); ++part) {
            __syncthreads();   // the tile may be in use
            tile_clear(tile, both ? 2 * nt : nt);
            __syncthreads();
            if (wv == k && ok) {
                const CellRef cr = cell_ref<R>(m, true, c, t, lane);
                const double s0 = (double)(part ? si : sr), s1 = (double)si;
#pragma unroll 1
                for (int q = 0; q < (m.one_d ? 2 : 8); ++q) {
                    const int e = (q + lane) & (m.one_d ? 1 : 7);   // rotated, as tile_add's
                    const double wk = (double)corner_weight<R>(m, c, e);
                    const int tk = corner_tile(m, t, cr, e);
                    atomicAdd(&tile[tk], wk * s0);
                    if (both) atomicAdd(&tile[nt + tk], wk * s1);
                }
            }
            __syncthreads();
            for (int e = threadIdx.x; e < (both ? 2 * nt : nt); e += blockDim.x) {
                const int q = both ? e >> 1 : e, p = both ? e & 1 : part;
                const double v = tile[both ? p * nt + q : q];
                if (v != 0.0) {
                    int lx, ly, lz;
                    box_coords(bd, q, lx, ly, lz);
                    const int node = (t.bz0 + lz) * ntr + (t.by0 + ly) * m.nx + (t.bx0 + lx);
                    atomic_add(outc + node_component(node, p), (R)v);
                }
            }
        }
    }
}

// ---- packed fixed-point tile of a whole workgroup (mixed form) -----------------

// One LDS atomic per corner for both components: each contribution becomes
// the integers qr = rint(w sr S), qi = rint(w si S) with the workgroup's
// power-of-two scale S, and qr 2^32 + qi is added to one 64-bit word of the
// tile.  S puts the largest |s| at 2^21 .. 2^22 - 4, so a node's sums, of at
// most PACK_MAX contributions of at most the largest |s|, stay below 2^31 in
// magnitude: the low half never carries into the high half beyond what its
// sign extension undoes, the word is sum qr 2^32 + sum qi exactly, and sum qi
// is its low 32 bits read as signed.  Integer sums are exact (and independent
// of the atomics' order); each contribution is rounded once, to 2^-22 of the
// largest |s|.  The flush divides by S and adds in FP32.
//
// In 3-D each contribution (wx wy) (wz s S) is rounded to an integer by one
// FMA with 1.5 2^23 added (|w s S| < 2^22 puts the sum in [2^23, 2^24), where
// FP32 steps by 1, so the FMA's single rounding is rint), whose bit pattern
// is 0x4B400000 + the integer: the two patterns of a contribution, as one
// 64-bit word, minus 0x4B4000004B400000 are qr 2^32 + qi (modulo 2^64).
constexpr float PACK_MAGIC = 12582912.0f;                      // 1.5 2^23
constexpr unsigned long long PACK_MAGIC2 = 0x4B4000004B400000ull;   // its pattern, twice

constexpr int PACK_MAX = 512;   // macroparticles of a workgroup
static_assert(PACK_MAX >= STAGE_THREADS, "node sums below 2^31");

// log2 of S for the workgroup's largest |s| (its bit pattern, max_bits): with
// e taken 2^-20 above it, |s| S < 2^22 (1 - 2^-21), so |q| <= 2^22 - 1.
__device__ __forceinline__ int packed_scale_log2(int max_bits) {
    const float mx = __int_as_float(max_bits);
    if (!(mx > 0.0f)) return 0;
    int e = 0;
    frexpf(mx * 1.00000095367431640625f, &e);
    return 22 - e;
}

__device__ __forceinline__ void packed_add(const MeshGeom& m, const TileBox& t, const Cell<float>& c,
                                           const CellRef& cr, float sr, float si, int log2S,
                                           unsigned long long* s_tile) {
    const int lane = threadIdx.x & 63;
    const float ssr = ldexpf(sr, log2S), ssi = ldexpf(si, log2S);
    if (!m.one_d) {
        const CornerSet<float> cs = corner_set<float>(c, t, lane & 7);
        const float zr[2] = {cs.z[0] * ssr, cs.z[1] * ssr};
        const float zi[2] = {cs.z[0] * ssi, cs.z[1] * ssi};
#pragma unroll
        for (int q = 0; q < 8; ++q) {
            const float vr = fmaf(cs.xy[q & 3], zr[q >> 2], PACK_MAGIC);
            const float vi = fmaf(cs.xy[q & 3], zi[q >> 2], PACK_MAGIC);
            const unsigned long long wq =
                (((unsigned long long)__float_as_uint(vr) << 32) | __float_as_uint(vi)) - PACK_MAGIC2;
            atomicAdd(&s_tile[cr.t0 + cs.oxy[q & 3] + cs.oz[q >> 2]], wq);
        }
    } else {
        for (int q = 0; q < 2; ++q) {
            const int k = (q + lane) & 1;
            const float wk = corner_weight<float>(m, c, k);
            const long long qr = (long long)(int)rintf(wk * ssr);
            const long long qi = (long long)(int)rintf(wk * ssi);
            atomicAdd(&s_tile[corner_tile(m, t, cr, k)], (unsigned long long)(qr * 4294967296LL + qi));
        }
    }
}

__device__ __forceinline__ void packed_flush(const MeshGeom& m, const TileBox& t, int log2S, cplx<float>* out,
                                             const unsigned long long* s_tile) {
    const int nt = t.tx * t.ty * t.tz;
    const int ntr = m.nx * m.ny;
    const BoxDiv bd = box_div(t);
    const float inv = ldexpf(1.0f, -log2S);
    float* outc = reinterpret_cast<float*>(out);
    // lanes 2j and 2j + 1: real and imaginary part of node j (as tile_flush)
    for (int e = threadIdx.x; e < 2 * nt; e += blockDim.x) {
        const int q = e >> 1, part = e & 1;
        const long long w = (long long)s_tile[q];
        const long long lo = (long long)(int)(unsigned int)(w & 0xffffffffLL);
        const long long v = part ? lo : (w - lo) >> 32;   // exact: w - lo is a multiple of 2^32
        if (v != 0) {
            int lx, ly, lz;
            box_coords(bd, q, lx, ly, lz);
            const int node = (t.bz0 + lz) * ntr + (t.by0 + ly) * m.nx + (t.bx0 + lx);
            atomic_add(outc + node_component(node, part), (float)v * inv);
        }
    }
}

// ---- deterministic deposit (FP64 form; see DetState) -------------------------

// Fixed-point pair of one contribution: t = v 2^F is exact (a power-of-two
// scaling) and so is t - rint(t) (Sterbenz: |t - rint(t)| <= 1/2 with
// rint(t) within a factor 2 of t, or rint(t) = 0), so hi + lo 2^-DET_LO_BITS
// is v 2^F rounded once, at 2^-DET_LO_BITS.  Two's-complement words: integer
// atomics add them modulo 2^64, which is exact while the sums stay in range.
__device__ __forceinline__ void det_split(double v, double scale, unsigned long long& hi,
                                          unsigned long long& lo) {
    const double t = v * scale;
    const double r = rint(t);
    hi = (unsigned long long)(long long)r;
    lo = (unsigned long long)(long long)rint((t - r) * (double)(1ull << DET_LO_BITS));
}

// The deposit in fixed point: the same two ways as above (LDS tile over the
// workgroup's node box, or runs of lanes that share a cell), with integer adds
// throughout, so neither the order of the LDS atomics nor that of the global
// ones changes a bit.  s_tile: DET_WORDS x nt words (Re hi | Re lo | Im hi |
// Im lo); out: DET_WORDS words per mesh node.
__device__ __forceinline__ void det_add(const MeshGeom& m, const TileBox& t, const Cell<double>& c,
                                        const CellRef& cr, double sr, double si, double scale,
                                        unsigned long long* s_tile) {
    const int lane = threadIdx.x & 63;
    const int nt = t.tx * t.ty * t.tz;
    auto add = [&](double wk, int tk) {
        unsigned long long h, l;
        det_split(wk * sr, scale, h, l);
        atomicAdd(&s_tile[tk], h);
        atomicAdd(&s_tile[nt + tk], l);
        det_split(wk * si, scale, h, l);
        atomicAdd(&s_tile[2 * nt + tk], h);
        atomicAdd(&s_tile[3 * nt + tk], l);
    };
    if (!m.one_d) {
        const CornerSet<double> cs = corner_set<double>(c, t, lane & 7);
#pragma unroll
        for (int q = 0; q < 8; ++q) add(cs.xy[q & 3] * cs.z[q >> 2], cr.t0 + cs.oxy[q & 3] + cs.oz[q >> 2]);
    } else {
        for (int q = 0; q < 2; ++q) {
            const int k = (q + lane) & 1;
            add(corner_weight<double>(m, c, k), corner_tile(m, t, cr, k));
        }
    }
}

// Lanes DET_WORDS j .. DET_WORDS j + 3 take the words of node j (one 32-byte
// sector): one atomic instruction covers 16 nodes.
__device__ __forceinline__ void det_flush(const MeshGeom& m, const TileBox& t, unsigned long long* out,
                                          const unsigned long long* s_tile) {
    const int nt = t.tx * t.ty * t.tz;
    const int64_t ntr = (int64_t)m.nx * m.ny;
    const BoxDiv bd = box_div(t);
    for (int e = threadIdx.x; e < DET_WORDS * nt; e += blockDim.x) {
        const int q = e / DET_WORDS, j = e % DET_WORDS;
        const unsigned long long w = s_tile[j * nt + q];
        if (w) {
            int lx, ly, lz;
            box_coords(bd, q, lx, ly, lz);
            const int64_t node = (int64_t)(t.bz0 + lz) * ntr + (int64_t)(t.by0 + ly) * m.nx + (t.bx0 + lx);
            atomicAdd(out + DET_WORDS * node + j, w);
        }
    }
}

__device__ __forceinline__ void det_global_add(const MeshGeom& m, bool ok, const Cell<double>& c, const CellRef& cr,
                                               double sr, double si, double scale, unsigned long long* out) {
    const int lane = threadIdx.x & 63;
    const int nnb = m.one_d ? 2 : 8;
    const int prev = __shfl_up(cr.key, 1, 64);
    const bool head = (lane == 0) || (prev != cr.key);
    const unsigned long long heads = __ballot(head);
    const unsigned long long after = (lane == 63) ? 0ull : (heads >> (lane + 1));
    const int seg_end = after ? lane + __builtin_ctzll(after) : 63;
    const int maxlen = wave_max(head ? seg_end - lane + 1 : 1);
#pragma unroll
    for (int k = 0; k < 8; ++k) {
        if (k < nnb) {
            const double wk = ok ? corner_weight<double>(m, c, k) : 0.0;
            unsigned long long w[DET_WORDS];
            det_split(wk * sr, scale, w[0], w[1]);
            det_split(wk * si, scale, w[2], w[3]);
            for (int o = 1; o < maxlen; o <<= 1) {
#pragma unroll
                for (int j = 0; j < DET_WORDS; ++j) {
                    const unsigned long long u = __shfl_down(w[j], o, 64);
                    if (lane + o <= seg_end) w[j] += u;
                }
            }
            if (ok && head) {
                unsigned long long* o = out + DET_WORDS * (int64_t)corner_node(m, cr, k);
#pragma unroll
                for (int j = 0; j < DET_WORDS; ++j)
                    if (w[j]) atomicAdd(o + j, w[j]);
            }
        }
    }
}

}  // namespace puff
