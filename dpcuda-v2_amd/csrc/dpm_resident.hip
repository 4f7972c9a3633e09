// dpm_resident.hip -- NVE and FIRE loops of a small disk system by one workgroup.
//
// The chunked loops (dpm_core.hip) take one launch a step for NVE and three for FIRE, and a list
// rebuild ends a FIRE chunk; below a few thousand particles a step is all launch gaps.  Here the
// system stays in one CU (dpm_resident.hpp) for hundreds of steps: phases are separated by
// workgroup barriers, lists and cells are rebuilt in place.  Arithmetic, row order, particle
// order and the canonical reduction order are those of the chunked loops, so results are the
// same bits.  A row that outgrows the ELL halts the step, which the rebuild chain then finishes.
// What bounds it: the CU's vector pipe and the chain of a step's phases (2 barriers and two LDS
// round trips for NVE, 4 barriers, a reduction and the decision for FIRE): 1.5 us a step with 128
// particles, where no pipe is busy, 3.3 us with 1,000.  Measured (before, after, ms): 1,024
// disks, 1000 NVE steps 5.9, 3.4; 777 disks, 2000 FIRE steps 38.6, 12.3.
#include "dpm_resident.hpp"

namespace dpm {

template <int T, int NP>
struct ResSystem : ResCore<T, NP> {
    double part[4][16];  // by chunk: F_x v_x, PE, F_y v_y, max F^2
    FireCtl F;
    int lflag, cflag;  // step + 1 of the last step that asked for a list / cell rebuild
    int over, done;
};

// `steps` steps (fewer once FIRE is done).  FIRE: d.fire holds the loop's state, the forces are
// current; NVE: dt.  Needs p.fast && p.fastdiv, N <= NP and, for the cell method, 3 to sqrt(NP)
// cells a side.
template <bool FIRE, int T, int NP>
__global__ __launch_bounds__(T) void k_resident(Dev d, Spare sp, PairParams p, NbrParams nb,
                                                double dt_nve, int steps) {
    __shared__ ResSystem<T, NP> L;
    Ctl* c = d.ctl;
    const int i = threadIdx.x, lane = i % WAVE, ch = i / WAVE;
    if (c->halt) return;
    if (FIRE) {
        static_assert(sizeof(FireCtl) % sizeof(int) == 0, "copied by words");
        for (int w = i; w < (int)(sizeof(FireCtl) / sizeof(int)); w += T)
            ((int*)&L.F)[w] = ((const int*)d.fire)[w];
    }
    if (i == 0) {
        L.lflag = 0;
        L.cflag = 0;
        L.over = 0;
        L.done = 0;
    }
    __syncthreads();
    if (FIRE && L.F.done) return;
    const int n = (int)d.N, nc = (n + WAVE - 1) / WAVE;
    const bool live = i < n;
    const bool cells = nb.method == DPM_NBR_CELL;
    const int ncell = cells ? (int)nb.ncells : 0;
    const double delta2 = 2.0 * sqrt(fmax(nb.thr, 0.0) / 3.0);
    const ResRows R{d.nbr, (long long)d.N, 0, d.cap};
    double4 q = make_double4(0.0, 0.0, 1.0, 1.0);
    double2 v = make_double2(0.0, 0.0), f = v, lref = v, cref = v;
    double pe = 0.0;
    int full = 0, cell = 0, mx = 0, lists = 0, sorts = 0;
    if (live) {
        q = d.P0[i];
        v = d.vel[i];
        f = d.frc[i];
        lref = d.lref[i];
        cref = d.cref[i];
        pe = d.pe[i];
        full = d.nnum[i];
        if (cells) cell = d.cell_of[i];
        L.x[i] = make_double2(q.x, q.y);
        L.r[i] = q.z;
    } else if (i < NP) {  // the rest of the last wave sums the zero pair
        for (int k = 0; k < RES_LC; ++k) L.row[k][i] = (unsigned short)L.MP;
    }
    if (i < ncell) L.cend[i] = d.cell_start[i + 1];
    double dtm = FIRE ? 0.0 : (0.5 * dt_nve) / q.w;
    __syncthreads();
    int len = live ? res_load_row(L, R, d.lref, i, full, delta2, p) : 0;
    len = res_pairs(L, n, len);
    int step = 0, halt = 0;
    double dt_kick = -1.0;  // the time step that dtm was formed for
    for (; step < steps; ++step) {
        // the move: Fire::step's first half (k_fire_move) or the opening kick and drift
        const double dt = FIRE ? uniform_d(L.F.dt) : dt_nve;
        if (ch < nc) {
            bool far = false, cfar = false;
            if (live) {
                if (FIRE) {
                    if (L.F.uphill) {
                        const double bdt = -dt / 2.0;
                        q.x += v.x * bdt;
                        q.y += v.y * bdt;
                        v.x = 0.0;
                        v.y = 0.0;
                    }
                    if (dt != dt_kick) dtm = (dt / 2.0) / q.w;
                }
                v.x += f.x * dtm;
                v.y += f.y * dtm;
                if (FIRE) mix_hot(v, f, uniform_d(L.F.alpha));
                q.x += v.x * dt;
                q.y += v.y * dt;
                L.x[i] = make_double2(q.x, q.y);
                const double dx = q.x - lref.x, dy = q.y - lref.y;
                far = 3.0 * (dx * dx + dy * dy) > nb.thr;
                const double cx = q.x - cref.x, cy = q.y - cref.y;
                cfar = cells && 3.0 * (cx * cx + cy * cy) > nb.cthr;
            }
            if (__builtin_amdgcn_ballot_w64(far) != 0 && lane == 0) L.lflag = step + 1;
            if (__builtin_amdgcn_ballot_w64(cfar) != 0 && lane == 0) L.cflag = step + 1;
        }
        dt_kick = dt;
        __syncthreads();  // every position of the step
        const bool sort = L.cflag == step + 1;
        if (sort || L.lflag == step + 1) {
            int near = 0;
            if (sort) {  // cells formed anew, particles in cell order (k_cell_*, k_reorder_*)
                auto cell_at = [&](double4 x) -> int {
                    const long long k = (long long)cell_coord(x.x, nb.cs, nb.ncd) +
                                        (long long)cell_coord(x.y, nb.cs, nb.ncd) * nb.ncd;
                    if (k >= 0 && k < ncell) return (int)k;
                    c->bad_pos = 1;  // a non-finite position
                    return 0;
                };
                if (live) {
                    sp.P[i] = q;
                    sp.vel[i] = v;
                    sp.sidx[i] = d.sidx[i];
                    if (d.m1) {
                        sp.m1[i] = d.m1[i];
                        sp.m2[i] = d.m2[i];
                    }
                }
                res_sort(L, n, ncell, live ? cell_at(q) : 0);
                if (live) {
                    const int o = L.lst[i];
                    q = sp.P[o];
                    v = sp.vel[o];
                    d.sidx[i] = sp.sidx[o];
                    if (d.m1) {
                        d.m1[i] = sp.m1[o];
                        d.m2[i] = sp.m2[o];
                    }
                    cref = make_double2(q.x, q.y);
                    cell = cell_at(q);
                    L.x[i] = cref;
                    L.r[i] = q.z;
                    d.cref[i] = cref;
                    d.cell_of[i] = cell;
                    dtm = (FIRE ? dt / 2.0 : 0.5 * dt_nve) / q.w;
                }
                sorts++;
                __syncthreads();
            }
            if (cells) {
                if (live)
                    full = res_row_cell(L, R, i, cell, nb.ncd, nb.rc2, delta2, p, near);
            } else {
                const double w = sqrt(nb.rc2) * (1.0 + 1e-9), most = floor(sqrt((double)NP));
                const int nx = (int)fmin(most, floor(nb.Lx / w));
                const int ny = (int)fmin(most, floor(nb.Ly / w));
                const bool grid = nx >= 3 && ny >= 3;
                int cx = 0, cy = 0;
                if (grid) {
                    if (live) {  // (a non-finite position has no neighbours, whatever its cell)
                        cx = min(max(cell_coord(q.x, nb.Lx / nx, nx), 0), nx - 1);
                        cy = min(max(cell_coord(q.y, nb.Ly / ny, ny), 0), ny - 1);
                    }
                    res_sort(L, n, nx * ny, cx + nx * cy);
                }
                if (live)
                    full = res_row_verlet(L, R, i, n, grid, cx, cy, nx, ny, nb.rc2, delta2, p,
                                          near);
            }
            if (live) {
                lref = make_double2(q.x, q.y);
                d.lref[i] = lref;
                mx = max(mx, full);
                if (full > d.cap) L.over = 1;
            }
            len = res_pairs(L, n, near);
            if (L.over) {  // the chain rebuilds (and counts) the list once it has grown
                halt = 1;
                break;
            }
            lists++;
        }
        // forces and the closing kick (k_fire_force, nve_force_body)
        const bool energy = FIRE || step == steps - 1, dense = L.dense != 0;
        if (!dense) {
            if (energy) res_pair_forces<true>(L, p);
            else res_pair_forces<false>(L, p);
        }
        __syncthreads();  // every pair of the step; every position has been read
        if (ch < nc) {
            double ax = 0.0, ay = 0.0, e = 0.0;
            if (dense) {
                if (live) res_sum_full(L, R, p, i, full, ax, ay, e);
            } else if (energy) {
                res_sum<true>(L, i, len, ax, ay, e);
            } else {
                res_sum<false>(L, i, len, ax, ay, e);
            }
            double pxv = 0.0, pyv = 0.0, f2 = 0.0;
            if (live) {
                const double fx = 0.0 + ax, fy = 0.0 + ay;
                f = make_double2(fx, fy);
                if (energy) pe = 0.0 + e;
                v.x += fx * dtm;
                v.y += fy * dtm;
                pxv = fx * v.x;
                pyv = fy * v.y;
                f2 = fx * fx + fy * fy;
            }
            if (FIRE) {
                const double s = wave_reduce4(pxv, pyv, pe, f2);
                if (lane % 16 == 0) L.part[lane / 16][ch] = s;
            }
        }
        // a dense row is read from the positions, which the next step moves
        if (FIRE || dense) __syncthreads();
        if (FIRE) {
            if (ch == 0) {  // k_fire_ctl: up to 16 partials, a row of lanes for each sum
                FireCtl F = L.F;
                const int k = lane % 16;
                const double s = rows_reduce(k < nc ? 0.0 + L.part[lane / 16][k] : 0.0);
                if (fire_advance(F, lane_value(s, 0), lane_value(s, 32), lane_value(s, 16),
                                 lane_value(s, 48), nullptr))
                    L.done = 1;
                L.F = F;
            }
            __syncthreads();  // the state of the next step
            if (L.done) {
                ++step;
                break;
            }
        }
    }
    // what a later launch or the other loops go on from
    __syncthreads();
    if (ch < nc) {
        double nd = 0.0, cd = 0.0;
        if (live) {
            d.P0[i] = q;
            if (sorts) d.P1[i] = q;
            d.vel[i] = v;
            d.frc[i] = f;
            d.pe[i] = pe;
            d.nnum[i] = full;
            const double dx = q.x - lref.x, dy = q.y - lref.y;
            nd = dx * dx + dy * dy;
            const double cx = q.x - cref.x, cy = q.y - cref.y;
            cd = cx * cx + cy * cy;
        }
        nd = wave_max(nd);
        cd = wave_max(cd);
        mx = wave_max_i(mx);
        if (lane == 0) {
            L.part[0][ch] = nd;
            L.part[1][ch] = cd;
            if (mx > 0) atomicMax(&c->max_nnum_all, mx);
        }
    }
    if (sorts) {
        if (i < ncell) d.cell_start[i + 1] = L.cend[i];
        if (i == 0) d.cell_start[0] = 0;
    }
    if (FIRE) {
        for (int w = i; w < (int)(sizeof(FireCtl) / sizeof(int)); w += T)
            ((int*)d.fire)[w] = ((const int*)&L.F)[w];
    }
    __syncthreads();
    // the displacement maxima of the final state by tiles of BLOCK particles (disp_epilogue)
    constexpr int PER = BLOCK / WAVE;
    if (i * PER < nc) {
        double nd = L.part[0][i * PER], cd = L.part[1][i * PER];
        for (int k = i * PER + 1; k < min(nc, (i + 1) * PER); ++k) {
            nd = fmax(nd, L.part[0][k]);
            cd = fmax(cd, L.part[1][k]);
        }
        d.pmax_nd[i] = nd;
        d.pmax_cd[i] = cd;
    }
    if (i == 0) {
        c->n_rebuilds += lists;
        c->n_cell_rebuilds += sorts;
        if (FIRE && L.done) c->done = 1;
        // a halted NVE step counts now (the chain applies its force and closing kick), a
        // halted FIRE step when the chain has finished it
        c->progress = step + (halt && !FIRE ? 1 : 0);
        if (halt) {
            c->halt = 1;
            c->halt_pos = 0;
            c->halt_mode = FIRE ? H_FIRE : H_NVE_FORCE;
            c->halt_kind = 1;
        }
    }
}

template <bool FIRE>
static void launch_resident(dpm_system* s, double dt, int steps) {
    const PairParams p = params_of(s);
    const NbrParams nb = nbr_params(s);
    const int64_t need = std::max(s->N, s->method == DPM_NBR_CELL ? s->ncells : (int64_t)0);
    hipStream_t st = s->stream;
    if (need <= 256)
        hipLaunchKernelGGL((k_resident<FIRE, 512, 256>), dim3(1), dim3(512), 0, st, s->d, s->sp,
                           p, nb, dt, steps);
    else if (need <= 512)
        hipLaunchKernelGGL((k_resident<FIRE, 1024, 512>), dim3(1), dim3(1024), 0, st, s->d, s->sp,
                           p, nb, dt, steps);
    else
        hipLaunchKernelGGL((k_resident<FIRE, 1024, 1024>), dim3(1), dim3(1024), 0, st, s->d,
                           s->sp, p, nb, dt, steps);
}

bool resident_ok(const dpm_system* s) {
    if (s->kind != DPM_DISK || s->N > RESIDENT_MAX_N) return false;
    if (s->method == DPM_NBR_CELL) {
        if (s->ncd < 3 || s->ncells > RESIDENT_MAX_N) return false;
    } else if (s->method != DPM_NBR_VERLET) {
        return false;
    }
    const PairParams p = params_of(s);
    return p.fast && p.fastdiv;
}

void resident_nve(dpm_system* s, double dt, int64_t steps) {
    launch_resident<false>(s, dt, (int)steps);
}

void resident_fire(dpm_system* s, int64_t steps) { launch_resident<true>(s, 0.0, (int)steps); }

}  // namespace dpm
