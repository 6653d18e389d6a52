// RK4 stage kernels of the macroparticle push: trial state, p2, tri-linear
// gather of A_perp, current deposit, undulator fields and the six scaled
// equations, fused into one kernel per RK4 stage; plus the field RK4
// combination.
//
// Reference arithmetic restated (UKFELs/Puffin):
//   rk4par          interaction/puffin_mpi_RK4.f90:38-366
//   getrhs          interaction/rhs.f90:60-330
//   getP2           utilities/gamma_to_p2.f90:84-85
//   getInterps_3D   interaction/system_interpolation.f90:25-98
//   getFFelecs_3D   interaction/system_interpolation.f90:110-142
//   getSource_3D    interaction/system_interpolation.f90:150-248
//   1-D branch      interaction/system_interpolation_1D.f90:24-179
//   equations       interaction/puffin_equations.f90:17-176
//   b-fields        undulator/bfields.f90:36-881 (per-stage coefficients are
//                   computed on the host, see puff_ctx.hip)
#include "puff_stage.hpp"

namespace puff {

// One RK4 stage.  STAGE = 1..4 (rk4par's four derivs calls).  DET: the
// deterministic fixed-point deposit (FP64 form only; see DetState).
//
// One macroparticle per thread (P): with two, a workgroup's box, field tile and
// flush serve twice as many, which took 20 % off the mixed stage 1 of 2^24 on
// 129 x 129 x 1024, and added 40 to 120 % to the stages of thin beams, whose
// boxes then grow past the tile.  (Written without the loops over P the
// compiler specialises the gather's branches: 1 to 3 % slower stages.)
template <typename R, int STAGE, bool DET, bool POLE>
__global__ __launch_bounds__(STAGE_THREADS) void k_stage(StageArgs<R> a) {
    constexpr int P = 1;
    static_assert(P == 1 || !DET, "the deterministic range checks take one macroparticle per thread");
    // Deposit tiles: two doubles per node in the FP64 form; DET_WORDS 8-byte
    // integers in its deterministic mode; one 8-byte packed fixed-point word
    // in the mixed form (packed_add: one ds_add_u64 per corner for
    // both components).  Measured on the C1 beam, mixed form: an FP32 tile
    // (ds_add_f32) ran each stage 3.1x slower than the FP64 tile, and a
    // compensated FP32 tile (ds_add_rtn_f32 + TwoSum) 5.7x slower, with the
    // same count of LDS instructions per wave but 6x the LDS-active and 24x
    // the LDS-wait cycles of ds_add_f64; the packed tile cut the LDS-wait
    // cycles per wave from 398 to 6 and the step by 3-4 %.
    // The field tile shares the deposit tile's LDS: it is used only for boxes
    // of at most FIELD_TILE_NODES nodes, whose deposit needs the first
    // WORDS x FIELD_TILE_NODES words, so it sits right after them.
    constexpr bool PACKED = sizeof(R) == 4 && PUFF_MIXED_TILE == 0 && !DET;
    constexpr int TILE = stage_tile_nodes<R>();
    using D = typename std::conditional<
        PACKED, unsigned long long,
        typename std::conditional<sizeof(R) == 4 && PUFF_MIXED_TILE == 2, float, double>::type>::type;
    constexpr int WORDS = DET ? DET_WORDS : (PACKED ? 1 : 2);
    static_assert(WORDS * FIELD_TILE_NODES * sizeof(D) + FIELD_TILE_NODES * sizeof(cplx<R>) <=
                      WORDS * TILE * sizeof(D), "field tile inside the deposit tile");
    __shared__ D s_dep[WORDS * TILE];
    cplx<R>* s_fld = reinterpret_cast<cplx<R>*>(s_dep + WORDS * FIELD_TILE_NODES);

    // Flags raised by an earlier kernel of this step do not stop stages 1-3:
    // they write only the step's scratch (k_s, dA_s), and a particle whose
    // trial position is off the mesh takes no part in the gather and deposit
    // (locate raises the flag again).  Stage 4 writes the state, and only
    // when no flag is set: read here, with the particle loads.  No workgroup of
    // stage 4 raises a flag, or others would have written by then: stage 3
    // checks stage 4's trial positions and, for the deterministic deposit, its
    // sources.
    const int rejected = (STAGE == 4) ? *a.flags : 0;
    // Slots of the workgroup: s0 + t, with s0 scalar and t 32 bits, so that an
    // access is a scalar base and one register of offset (64-bit lane addresses
    // took two registers and three instructions per array).
    const int64_t s0 = (int64_t)blockIdx.x * (STAGE_THREADS * P);
    const unsigned left = (unsigned)min<int64_t>(a.n - s0, STAGE_THREADS * P);
    auto at = [s0](auto* q, unsigned t) -> auto& { return (q + s0)[t]; };
    const MeshGeom& m = a.mesh;
    const Physics& ph = a.phys;

    // ---- trial state y_s = y0 + c k_{s-1} (puffin_mpi_RK4.f90:190-195 etc.)
    bool in[P];
    R x[P], y[P], pr[P], pi[P], chi[P];
    double z2[P], g[P];
    R x0[P], y0[P], pr0[P], pi0[P];
    double z20[P], g0[P];
#pragma unroll
    for (int p = 0; p < P; ++p) {
        const unsigned i = threadIdx.x + p * STAGE_THREADS;
        in[p] = i < left;
        x0[p] = y0[p] = pr0[p] = pi0[p] = chi[p] = 0;
        z20[p] = 0.0;
        g0[p] = 1.0;
        if (in[p]) {
            x0[p] = at(a.y0.x, i);
            y0[p] = at(a.y0.y, i);
            z20[p] = at(a.y0.z2, i);
            pr0[p] = at(a.y0.pr, i);
            pi0[p] = at(a.y0.pi, i);
            g0[p] = at(a.y0.g, i);
            chi[p] = at(a.chi, i);
        }
    }
    if constexpr (STAGE == 1) {
#pragma unroll
        for (int p = 0; p < P; ++p) {
            x[p] = x0[p]; y[p] = y0[p]; z2[p] = z20[p]; pr[p] = pr0[p]; pi[p] = pi0[p]; g[p] = g0[p];
            const unsigned i = threadIdx.x + p * STAGE_THREADS;
            if (in[p] && a.ycap.x) {
                at(a.ycap.x, i) = x0[p];
                at(a.ycap.y, i) = y0[p];
                at(a.ycap.z2, i) = z20[p];
                at(a.ycap.pr, i) = pr0[p];
                at(a.ycap.pi, i) = pi0[p];
                at(a.ycap.g, i) = g0[p];
                at(a.chicap, i) = chi[p];
            }
        }
    } else {
        R kr[P], ki[P], kg[P], qr[P], qi[P], qg[P];
#pragma unroll
        for (int p = 0; p < P; ++p) {
            const unsigned i = threadIdx.x + p * STAGE_THREADS;
            kr[p] = ki[p] = kg[p] = qr[p] = qi[p] = qg[p] = 0;
            if (in[p]) {
                kr[p] = at(a.kin.pr, i);
                ki[p] = at(a.kin.pi, i);
                kg[p] = at(a.kin.g, i);
                if (STAGE > 2) {
                    qr[p] = at(a.kprev.pr, i);
                    qi[p] = at(a.kprev.pi, i);
                    qg[p] = at(a.kprev.g, i);
                }
            }
        }
#pragma unroll
        for (int p = 0; p < P; ++p) {
            const Trial<R> t = trial_state<R, STAGE>(ph, x0[p], y0[p], z20[p], pr0[p], pi0[p], g0[p], kr[p], ki[p],
                                                     kg[p], qr[p], qi[p], qg[p], a.cin, a.cprev, a.cin_r, a.cprev_r);
            x[p] = t.x; y[p] = t.y; z2[p] = t.z2; pr[p] = t.pr; pi[p] = t.pi; g[p] = t.g;
            if (STAGE == 4) {
                // y0 + h/6 (k1 + 2 (k2 + k3)) formed now: the end of the kernel
                // adds h/6 k4 only, and no k array is read after the deposit
                // (puffin_mpi_RK4.f90:274-279).  The rates of y0, y0 + h/2 k1
                // and y0 + h/2 k2 are k1 to k3 of x, y and z2.
                const unsigned i = threadIdx.x + p * STAGE_THREADS;
                const R h6 = a.h6_r, hh = a.cprev_r;
                R k1r = 0, k1i = 0, k1g = 0;
                if (in[p]) {
                    k1r = at(a.k1.pr, i);
                    k1i = at(a.k1.pi, i);
                    k1g = at(a.k1.g, i);
                }
                Rates<R> v1 = rates<R>(ph, drift_of(ph, (double)pr0[p], (double)pi0[p], g0[p]), pr0[p], pi0[p]);
                // one rate after the other: side by side they take 20 registers more
                hold(v1.x);
                hold(v1.y);
                hold(v1.z2);
                hold(k1r);
                const R p2r = fma(hh, k1r, pr0[p]), p2i = fma(hh, k1i, pi0[p]);
                const Rates<R> v2 =
                    rates<R>(ph, drift_of(ph, (double)p2r, (double)p2i, fma(a.cprev, (double)k1g, g0[p])), p2r, p2i);
                x0[p] = fma(h6, v1.x + (R)2 * (v2.x + t.v.x), x0[p]);
                y0[p] = fma(h6, v1.y + (R)2 * (v2.y + t.v.y), y0[p]);
                z20[p] = fma(a.h6, v1.z2 + 2.0 * (v2.z2 + t.v.z2), z20[p]);
                pr0[p] = fma(h6, k1r + (R)2 * (qr[p] + kr[p]), pr0[p]);
                pi0[p] = fma(h6, k1i + (R)2 * (qi[p] + ki[p]), pi0[p]);
                g0[p] = fma(a.h6, (double)k1g + 2.0 * ((double)qg[p] + (double)kg[p]), g0[p]);
                // formed here: left alone, the compiler moves them behind the
                // deposit, with their inputs live across it
                hold(x0[p]);
                hold(y0[p]);
                hold(z20[p]);
                hold(pr0[p]);
                hold(pi0[p]);
                hold(g0[p]);
            }
        }
    }

    // ---- p2 in FP64 and (1 + eta p2) / Gamma; node and weights; sources
    // (getSource): s = chi / dV3 (1 + eta p2) p / Gamma
    double fac[P];
    R ep2k[P], sr[P], si[P];
    Cell<R> c[P];
    bool ok[P];
    bool next_ok = false;   // (DET) the next stage's trial position is on the mesh
    LaneBox lb = lane_box();
#pragma unroll
    for (int p = 0; p < P; ++p) {
        hold(g[p]);
        const double prd = (double)pr[p], pid = (double)pi[p];
        const Drift dr = drift_of(ph, prd, pid, g[p]);
        fac[p] = dr.fac;
        ep2k[p] = (R)(ph.eta_k2 * dr.p2);
        c[p] = Cell<R>{};
        int flag = in[p] ? locate<R>(m, x[p], y[p], z2[p], c[p]) : 0;
        ok[p] = in[p] && flag == 0;
        sr[p] = ok[p] ? (R)((double)chi[p] * ph.inv_dV3 * fac[p] * prd) : (R)0;
        si[p] = ok[p] ? (R)((double)chi[p] * ph.inv_dV3 * fac[p] * pid) : (R)0;
        lane_box_add<R>(lb, ok[p], c[p], PACKED ? __float_as_int(fmaxf(fabsf((float)sr[p]), fabsf((float)si[p]))) : 0);
        const Rates<R> v = rates<R>(ph, dr, pr[p], pi[p]);
        if (STAGE < 4) {
            // next stage's trial state must lie inside the mesh, else the next
            // derivs call would raise the flag (checked here, on the rates the
            // next stage forms again, so that no later kernel writes state when
            // it does)
            const R cn = a.cnext_r;
            Cell<R> cc;
            if (in[p]) {
                const int off = locate<R>(m, fma(cn, v.x, x0[p]), fma(cn, v.y, y0[p]), fma(a.cnext, v.z2, z20[p]), cc);
                next_ok = off == 0;
                flag |= off;
            }
        } else {
            // x, y and z2 of the step's end do not wait for the field
            const unsigned i = threadIdx.x + p * STAGE_THREADS;
            if (in[p] && !rejected) {
                at(a.y0.x, i) = fma(a.h6_r, v.x, x0[p]);
                at(a.y0.y, i) = fma(a.h6_r, v.y, y0[p]);
                at(a.y0.z2, i) = fma(a.h6, ph.electrons_evolve ? dr.p2 : 0.0, z20[p]);   // k_4: as it is
            }
        }
        if (flag) atomicOr(a.flags, flag);
        // kept as they stand across the barriers (see the sums above)
        hold(fac[p]);
        hold(ep2k[p]);
    }

    // ---- node box of this workgroup's cells and the step's active box (and,
    // for the packed fixed-point tile, the workgroup's largest |s|)
    const int lane = threadIdx.x & 63;
    __shared__ WaveBoxes s_red;
    const TileBox tb = workgroup_box<PACKED ? 7 : 6>(m, lb, a.box, s_red);
    const bool use_tile = ph.field_evolve && tile_fits<TILE>(m, tb);
    if (threadIdx.x == 0 && ph.field_evolve && tb.any && !use_tile) atomicAdd(a.flags + FLAG_WORD_FALLBACK, 1);

    // ---- gather F = sum_k w_k (A0 + c dA_{s-1})[node_k]  (getFFelecs).
    // When the workgroup's node box is small (the dense part of the beam),
    // A0 + c dA_{s-1} is formed once per node of the box in LDS and the
    // corners are read from there; else from global memory.  Same arithmetic
    // either way.
    const R cA = a.cin_r;
    const int nt = tb.tx * tb.ty * tb.tz;
    const bool lds_field = use_tile && nt <= FIELD_TILE_NODES;
    if (lds_field) {
        const int ntr = m.nx * m.ny;
        const BoxDiv bd = box_div(tb);
        for (int q = threadIdx.x; q < nt; q += blockDim.x) {
            int lx, ly, lz;
            box_coords(bd, q, lx, ly, lz);
            const int node = (tb.bz0 + lz) * ntr + (tb.by0 + ly) * m.nx + (tb.bx0 + lx);
            cplx<R> v = a.A0[node];
            if (STAGE > 1) {
                const cplx<R> d = a.dAin[node];
                v.x = fma(cA, d.x, v.x);
                v.y = fma(cA, d.y, v.y);
            }
            s_fld[q] = v;
        }
    }
    if (use_tile) {
        tile_clear(s_dep, WORDS * nt);
        __syncthreads();
    }
    const int nnb = m.one_d ? 2 : 8;
    const int log2S = PACKED ? packed_scale_log2(tb.extra) : 0;
    R fr[P], fi[P];
    double det_scale = 0.0, det_lim = 0.0;
    if constexpr (DET) {
        // n |s| 2^F <= 2^62 keeps every node's integer sums in range
        det_scale = ldexp(1.0, *a.det.shift);
        det_lim = ldexp(1.0, 62) / det_scale / (double)a.n;
    }
    // ---- momentum equations (puffin_equations.f90:17-104)
    auto equations = [&](int p) {
        const unsigned i = threadIdx.x + p * STAGE_THREADS;
        R kpr = 0, kpi = 0;
        double kg = 0.0;
        if (ph.electrons_evolve) {
            R bx, by, bz;
            bfield<R, POLE>(a.s, x[p], y[p], bx, by, bz);
            const R facr = (R)fac[p];
            const R n2col = a.s.template strength<R>();
            const R kappa = ph.template scale<R>().kappa, inv2rho = ph.template scale<R>().inv2rho;
            // the roundings written out: a different contraction moves the
            // mixed form's p_r by 2e-6 and z2 by 2e-9 over a lattice
            const R pull_r = inv2rho * fma(n2col, by, -(ep2k[p] * fr[p]));
            kpr = fma(kappa * pi[p] * facr * n2col, bz, pull_r);
            kpi = fma(inv2rho, fma(n2col, bx, -(ep2k[p] * fi[p])), -(kappa * pr[p] * facr * n2col * bz));
            kg = -ph.rho * fac[p] * 2.0 * ((double)pr[p] * (double)fr[p] + (double)pi[p] * (double)fi[p]);
        }
        if (STAGE < 4) {
            if (in[p]) {
                at(a.kout.pr, i) = kpr;
                at(a.kout.pi, i) = kpi;
                at(a.kout.g, i) = (R)kg;   // FP32 in the mixed form (see KPtrs)
            }
            if constexpr (DET && STAGE == 3) {
                // stage 4's sources, as it will form them
                const double r4 = fma(a.cnext, kpr, pr0[p]), i4 = fma(a.cnext, kpi, pi0[p]);
                const double q4 = chi[p] * ph.inv_dV3 * drift_of(ph, r4, i4, fma(a.cnext, kg, g0[p])).fac;
                if (ph.field_evolve && next_ok && (fabs(q4 * r4) > det_lim || fabs(q4 * i4) > det_lim))
                    atomicOr(a.flags, FLAG_DET_RANGE);
            }
        } else if (in[p] && !rejected) {
            // y = (y0 + h/6 (k1 + 2 (k2 + k3))) + h/6 k4 (puffin_mpi_RK4.f90:274-279, 307-312)
            at(a.y0.pr, i) = fma(a.h6_r, kpr, pr0[p]);
            at(a.y0.pi, i) = fma(a.h6_r, kpi, pi0[p]);
            at(a.y0.g, i) = fma(a.h6, kg, g0[p]);
        }
    };
#pragma unroll
    for (int p = 0; p < P; ++p) {
        const CellRef cr = cell_ref<R>(m, ok[p], c[p], tb, lane);
        fr[p] = fi[p] = 0;
        if (ok[p] && lds_field && !m.one_d) {
            // getFFelecs' corner order, the weights formed once per lane
            const CornerSet<R> cs = corner_set<R>(c[p], tb, 0);
#pragma unroll
            for (int q = 0; q < 8; ++q) {
                const cplx<R> v = s_fld[cr.t0 + cs.oxy[q & 3] + cs.oz[q >> 2]];
                const R wk = cs.xy[q & 3] * cs.z[q >> 2];
                fr[p] = fma(wk, v.x, fr[p]);
                fi[p] = fma(wk, v.y, fi[p]);
            }
        } else if (ok[p]) {
#pragma unroll
            for (int q = 0; q < 8; ++q) {
                if (q < nnb) {
                    cplx<R> v;
                    if (lds_field) {
                        v = s_fld[corner_tile(m, tb, cr, q)];
                    } else {
                        const int node = corner_node(m, cr, q);
                        v = a.A0[node];
                        if (STAGE > 1) {
                            const cplx<R> d = a.dAin[node];
                            v.x = fma(cA, d.x, v.x);
                            v.y = fma(cA, d.y, v.y);
                        }
                    }
                    const R wk = corner_weight<R>(m, c[p], q);
                    fr[p] = fma(wk, v.x, fr[p]);
                    fi[p] = fma(wk, v.y, fi[p]);
                }
            }
        }
        if (!ph.coupling) { fr[p] = 0; fi[p] = 0; }   // rhs.f90:221-224

        equations(p);
    }

    // ---- deposit w_k s into dA_s (getSource)
    auto add = [&](const TileBox& t) {
#pragma unroll
        for (int p = 0; p < P; ++p) {
            // the deposit's weights are formed here, not beside the gather's
            hold(c[p].fx);
            hold(c[p].fy);
            hold(c[p].fz);
            if (!ok[p]) continue;
            const CellRef cr = cell_ref<R>(m, true, c[p], t, lane);
            if constexpr (DET)
                det_add(m, t, c[p], cr, (double)sr[p], (double)si[p], det_scale,
                        reinterpret_cast<unsigned long long*>(s_dep));
            else if constexpr (PACKED) packed_add(m, t, c[p], cr, (float)sr[p], (float)si[p], log2S, s_dep);
            else tile_add<R, D>(m, t, c[p], cr, sr[p], si[p], s_dep);
        }
    };
    auto flush = [&](const TileBox& t) {
        if constexpr (DET) det_flush(m, t, a.det.acc, reinterpret_cast<const unsigned long long*>(s_dep));
        else if constexpr (PACKED) packed_flush(m, t, log2S, reinterpret_cast<cplx<float>*>(a.dAout), s_dep);
        else tile_flush<R, D>(m, t, a.dAout, s_dep);
    };
    if constexpr (DET && STAGE < 4) {
        if (ph.field_evolve && ok[0] && (fabs((double)sr[0]) > det_lim || fabs((double)si[0]) > det_lim))
            atomicOr(a.flags, FLAG_DET_RANGE);
    }
    if (!ph.field_evolve) return;
    auto spill = [&]() {
#pragma unroll
        for (int p = 0; p < P; ++p) {
            const CellRef cr = cell_ref<R>(m, ok[p], c[p], tb, lane);
            if constexpr (DET)
                det_global_add(m, ok[p], c[p], cr, (double)sr[p], (double)si[p], det_scale, a.det.acc);
            else global_add<R>(m, ok[p], c[p], cr, sr[p], si[p], a.dAout);
        }
    };
    if constexpr (PACKED) {
        // wavefronts that deposit in turn add in FP64: the packed words round to
        // 2^-22 of the workgroup's largest source, which a workgroup spread over
        // the beam may hold far from its smallest.  A step on 129 x 129 x 1024 of
        // 2^17 (all workgroups overflow), 2^20 (5 %) and 2^24 macroparticles
        // (0.3 %): 258, 347 and 1470 us; packed words for the single wavefronts
        // too, 238, 324 and 1500; global atomics for whole workgroups, 482, 510
        // and 1680.
        static_assert(P == 1, "one macroparticle per thread");
        if (use_tile) {
            add(tb);
            __syncthreads();
            flush(tb);
        } else {
            wave_deposit<TILE, R>(m, s_red, ok[0], c[0], sr[0], si[0], reinterpret_cast<double*>(s_dep), a.dAout, spill);
        }
    } else {
        tile_deposit<TILE>(
            m, tb, use_tile, s_red, [&](const TileBox& t) { tile_clear(s_dep, WORDS * t.tx * t.ty * t.tz); }, add,
            flush, spill);
    }
}

// Start of a step: clear flags and the active box.
__global__ void k_step_begin(int* flags, Box* box) {
    if (threadIdx.x < FLAG_WORD_STICKY) flags[threadIdx.x] = 0;
    for (int k = threadIdx.x; k < BOX_COPIES; k += blockDim.x) {
        for (int d = 0; d < 3; ++d) {
            box[k].lo[d] = 0x7fffffff;
            box[k].hi[d] = -1;
        }
    }
}

// A += h/6 (dA1 + dA4 + 2 (dA2 + dA3)) over the active box
// (puffin_mpi_RK4.f90:281-282, 314-315), then clear the deposits there (all
// four, or only the last when the first three are kept for the adjoint).
// The periodic mesh keeps its aliased last plane equal to plane 0.
// Bound by memory: 160 bytes per node in FP64, of which a node that took no
// deposit (the corners of the box around a round beam) needs only the 64 of
// the reads.
template <typename R>
__global__ __launch_bounds__(256) void k_field_combine(CombineArgs<R> a) {
    if (blockIdx.x == 0 && threadIdx.x == 0 && a.flags[0]) atomicOr(a.flags + FLAG_WORD_STICKY, a.flags[0]);
    const bool update = (*a.flags == 0);
    const R h6 = (R)a.h6;
    const int64_t ntr = (int64_t)a.nx * a.ny;
    each_active_node(merged_box(a.box), a.nx, a.ny, a.nzp, a.periodic, a.one_d, [&](int ix, int iy, int iz) {
        const int64_t j = (int64_t)iz * ntr + (int64_t)iy * a.nx + ix;
        const cplx<R> d0 = a.d[0][j], d1 = a.d[1][j], d2 = a.d[2][j], d3 = a.d[3][j];
        const bool alias = a.periodic && iz == 0;
        if (all_zero(d0, d1) && all_zero(d2, d3) && !alias) return;
        if (update) {
            cplx<R> v = a.A[j];
            const R tx = d1.x + d2.x, ty = d1.y + d2.y;
            v.x = v.x + h6 * (d0.x + d3.x + (R)2 * tx);
            v.y = v.y + h6 * (d0.y + d3.y + (R)2 * ty);
            a.A[j] = v;
            if (alias) a.A[(int64_t)(a.nz2 - 1) * ntr + (int64_t)iy * a.nx + ix] = v;
        }
        const cplx<R> zero = {(R)0, (R)0};
        for (int k = a.clear_from; k < 4; ++k) a.d[k][j] = zero;
    });
}

// ---- deterministic deposit ---------------------------------------------------

// Largest |source| chi / dV3 (1 + eta p2) |p_r|, |p_i| / Gamma of the state y,
// reduced as the bits of a non-negative double: their integer order is the
// value order, so the integer maximum is exact whatever the atomics' order.
__global__ __launch_bounds__(256) void k_det_bound(PartPtrs<double> y, const double* chi, int64_t n,
                                                   Physics ph, unsigned long long* bound) {
    double v = 0.0;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
         i += (int64_t)gridDim.x * blockDim.x) {
        const double pr = y.pr[i], pi = y.pi[i];
        const double invg = 1.0 / y.g[i];
        const double p2 = ((1.0 / sqrt(1.0 - ph.inv_gr2 * invg * invg * (1.0 + ph.aw * ph.aw * (pr * pr + pi * pi)))) -
                           1.0) * ph.inv_eta;
        const double s = chi[i] * ph.inv_dV3 * (1.0 + ph.eta * p2) * invg;
        v = fmax(v, fmax(fabs(s * pr), fabs(s * pi)));
    }
    for (int o = 32; o > 0; o >>= 1) v = fmax(v, __shfl_xor(v, o, 64));
    if ((threadIdx.x & 63) == 0 && v > 0.0) atomicMax(bound, (unsigned long long)__double_as_longlong(v));
}

// F of the step: DET_SAFETY n max|s| < 2^(62 - F), i.e. 62 minus the binary
// exponent e of that bound (frexp: bound < 2^e).  Clears the bound word for
// the next step.
__global__ void k_det_shift(unsigned long long* bound, int* shift, int64_t n) {
    const double m = __longlong_as_double((long long)*bound);
    int F = 0;
    if (m > 0.0) {
        int e = 0;
        frexp((double)DET_SAFETY * (double)n * m, &e);
        F = 62 - e;
        F = F > 1000 ? 1000 : (F < -1000 ? -1000 : F);
    }
    *shift = F;
    *bound = 0ull;
}

// dA = Re hi 2^-F + Re lo 2^-(F + DET_LO_BITS) (and Im) over the step's
// active box so far, clearing the integer sums there.
__global__ __launch_bounds__(256) void k_det_convert(DetState d, cplx<double>* dA, const Box* box, int nx,
                                                     int ny, int nzp, int periodic, int one_d) {
    const int F = *d.shift;
    const double inv_hi = ldexp(1.0, -F), inv_lo = ldexp(1.0, -(F + DET_LO_BITS));
    const int64_t ntr = (int64_t)nx * ny;
    each_active_node(merged_box(box), nx, ny, nzp, periodic, one_d, [&](int ix, int iy, int iz) {
        const int64_t j = (int64_t)iz * ntr + (int64_t)iy * nx + ix;
        unsigned long long* w = d.acc + DET_WORDS * j;
        const long long rh = (long long)w[0], rl = (long long)w[1], ih = (long long)w[2], il = (long long)w[3];
        dA[j] = {(double)rh * inv_hi + (double)rl * inv_lo, (double)ih * inv_hi + (double)il * inv_lo};
        if (rh | rl | ih | il) {
            w[0] = 0ull;
            w[1] = 0ull;
            w[2] = 0ull;
            w[3] = 0ull;
        }
    });
}

// Periodic z2 wrap (para_field.f90:212-215).
__global__ void k_wrap_z2(double* z2, int64_t n, double lenz2) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) z2[i] = z2[i] - (floor(z2[i] / lenz2) * lenz2);
}

// ---- host launchers --------------------------------------------------------

template <typename R, int STAGE>
static void launch_stage_n(const StageArgs<R>& a, hipStream_t s) {
    const int64_t blocks = stage_workgroups(a.n);
    const dim3 grid((unsigned)(blocks > 0 ? blocks : 1)), thr(STAGE_THREADS);
    if constexpr (sizeof(R) == 8) {
        if (a.det.acc) {
            hipLaunchKernelGGL((k_stage<R, STAGE, true, true>), grid, thr, 0, s, a);
            return;
        }
    }
    if (stage_pole(a.s.und_type)) hipLaunchKernelGGL((k_stage<R, STAGE, false, true>), grid, thr, 0, s, a);
    else hipLaunchKernelGGL((k_stage<R, STAGE, false, false>), grid, thr, 0, s, a);
}

template <typename R>
void launch_stage(int stage, const StageArgs<R>& a, hipStream_t s) {
    switch (stage) {
        case 1: return launch_stage_n<R, 1>(a, s);
        case 2: return launch_stage_n<R, 2>(a, s);
        case 3: return launch_stage_n<R, 3>(a, s);
        default: return launch_stage_n<R, 4>(a, s);
    }
}

void launch_det_scale(const PartPtrs<double>& y, const double* chi, int64_t n, const Physics& ph,
                      const DetState& d, hipStream_t s) {
    int64_t blocks = (n + 255) / 256;
    if (blocks > 2048) blocks = 2048;
    if (blocks < 1) blocks = 1;
    hipLaunchKernelGGL(k_det_bound, dim3((unsigned)blocks), dim3(256), 0, s, y, chi, n, ph, d.bound);
    hipLaunchKernelGGL(k_det_shift, dim3(1), dim3(1), 0, s, d.bound, d.shift, n);
}

void launch_det_convert(const DetState& d, cplx<double>* dA, const Box* box, int nx, int ny, int nzp,
                        int periodic, int one_d, hipStream_t s) {
    hipLaunchKernelGGL(k_det_convert, dim3(mesh_grid((int64_t)nx * ny * nzp)), dim3(256), 0, s, d, dA, box, nx, ny,
                       nzp, periodic, one_d);
}

void launch_step_begin(int* flags, Box* box, hipStream_t s) {
    hipLaunchKernelGGL(k_step_begin, dim3(1), dim3(64), 0, s, flags, box);
}

template <typename R>
void launch_combine(const CombineArgs<R>& a, hipStream_t s) {
    hipLaunchKernelGGL((k_field_combine<R>), dim3(mesh_grid((int64_t)a.nx * a.ny * a.nzp)), dim3(256), 0, s, a);
}

void launch_wrap(double* z2, int64_t n, double lenz2, hipStream_t s) {
    if (n <= 0) return;
    hipLaunchKernelGGL(k_wrap_z2, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, z2, n, lenz2);
}

template void launch_stage<double>(int, const StageArgs<double>&, hipStream_t);
template void launch_stage<float>(int, const StageArgs<float>&, hipStream_t);
template void launch_combine<double>(const CombineArgs<double>&, hipStream_t);
template void launch_combine<float>(const CombineArgs<float>&, hipStream_t);

}  // namespace puff
