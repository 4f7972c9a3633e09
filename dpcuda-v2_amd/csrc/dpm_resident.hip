// dpm_resident.hip -- NVE and FIRE loops of a small disk system by one workgroup.
//
// The chunked loops (dpm_core.hip) take one launch a step for NVE and three for FIRE, and a list
// rebuild ends a FIRE chunk; below a few thousand particles a step is all launch gaps.  Here the
// system stays in one CU (dpm_resident.hpp) for hundreds of steps: phases are separated by
// workgroup barriers, lists and cells are rebuilt in place.  Arithmetic, row order, particle
// order and the canonical reduction order are those of the chunked loops, so results are the
// same bits.  A row that outgrows the ELL halts the step, which the rebuild chain then finishes.
// What bounds it: one CU's vector pipe (busy 57 % of the time with 777 disks, LDS 10 %) and the
// chain of a step's phases, in which its waves wait (2 barriers and two LDS round trips for NVE, 4
// barriers, a reduction and the decision for FIRE): 1.5 us a step with 128 particles, where no
// pipe is busy, 3.4 us with 1,000.  Measured (before, after, ms):
// 1,024 disks, 1000 NVE steps 5.9, 3.5; 777 disks, 2000 FIRE steps 38.6, 12.4.
#include "dpm_resident.hpp"

namespace dpm {

template <int T, int NP>
struct ResSystem : ResCore<T, NP> {
    double part[4][NP / WAVE];  // by chunk: F_x v_x, PE, F_y v_y, max F^2
    FireCtl F;
    int lflag, cflag;  // step + 1 of the last step that asked for a list / cell rebuild
    int over, done;
};

// `steps` steps (fewer once FIRE is done).  FIRE: d.fire holds the loop's state, the forces are
// current; NVE: dt.  rows: RES_LC * NP entries (two particles a thread).  Needs p.fast &&
// p.fastdiv, N <= NP and, for the cell method, 3 to sqrt(NP) cells a side.
template <bool FIRE, int T, int NP>
__global__ __launch_bounds__(T) void k_resident(Dev d, Spare sp, PairParams p, NbrParams nb,
                                                double dt_nve, int steps,
                                                unsigned short* rows) {
    using C = ResCore<T, NP>;
    constexpr int PPT = C::PPT;
    __shared__ ResSystem<T, NP> L;
    Ctl* c = d.ctl;
    const int tid = threadIdx.x, lane = tid % WAVE;
    if (c->halt) return;
    if (FIRE) {
        static_assert(sizeof(FireCtl) % sizeof(int) == 0, "copied by words");
        for (int w = tid; w < (int)(sizeof(FireCtl) / sizeof(int)); w += T)
            ((int*)&L.F)[w] = ((const int*)d.fire)[w];
    }
    if (tid == 0) {
        L.lflag = 0;
        L.cflag = 0;
        L.over = 0;
        L.done = 0;
    }
    __syncthreads();
    if (FIRE && L.F.done) return;
    const int n = (int)d.N, nc = (n + WAVE - 1) / WAVE;
    const bool cells = nb.method == DPM_NBR_CELL;
    const int ncell = cells ? (int)nb.ncells : 0;
    const double delta2 = res_reach(nb.thr);
    const ResRows R{d.nbr, (long long)d.N, 0, d.cap};
    ResKept<T, NP> K;
    K.row = rows;
    double mass[PPT], dtm[PPT], pe[PPT];
    double2 v[PPT], f[PPT], own = make_double2(0.0, 0.0);  // (own: one a thread)
    double2 lref[C::BIG ? 1 : PPT], cref[C::BIG ? 1 : PPT];  // (two a thread: read from HBM)
    int full[PPT], len[PPT], cell[PPT], near[PPT], mx = 0, lists = 0, sorts = 0;
#pragma unroll
    for (int m = 0; m < PPT; ++m) {
        const int i = tid + m * T;
        const bool live = i < n;
        const double4 q = live ? d.P0[i] : make_double4(0.0, 0.0, 1.0, 1.0);
        v[m] = live ? d.vel[i] : make_double2(0.0, 0.0);
        f[m] = live ? d.frc[i] : make_double2(0.0, 0.0);
        pe[m] = live ? d.pe[i] : 0.0;
        full[m] = live ? d.nnum[i] : 0;
        cell[m] = live && cells ? d.cell_of[i] : 0;
        if (!C::BIG) {
            lref[m] = live ? d.lref[i] : make_double2(0.0, 0.0);
            cref[m] = live ? d.cref[i] : make_double2(0.0, 0.0);
        }
        mass[m] = q.w;
        if (!C::BIG) own = make_double2(q.x, q.y);
        dtm[m] = FIRE ? 0.0 : (0.5 * dt_nve) / q.w;
        if (i < NP) {
            L.x[i] = make_double2(q.x, q.y);
            L.r[i] = q.z;
        }
    }
    __syncthreads();
#pragma unroll
    for (int m = 0; m < PPT; ++m) {
        const int i = tid + m * T;
        near[m] = i < n ? res_load_row(L, R, d.lref, i, full[m], delta2, p) : 0;
    }
    res_pairs(L, K, n, true, near, len);
    int step = 0, halt = 0;
    double dt_kick = -1.0;  // the time step that dtm was formed for
    for (; step < steps; ++step) {
        // the move: Fire::step's first half (k_fire_move) or the opening kick and drift
        const double dt = FIRE ? uniform_d(L.F.dt) : dt_nve;
        const double alpha = FIRE ? uniform_d(L.F.alpha) : 0.0;
        const int uphill = FIRE ? L.F.uphill : 0;
        bool far = false, cfar = false;
#pragma unroll
        for (int m = 0; m < PPT; ++m) {
            const int i = tid + m * T;
            if (i >= n) continue;
            const double2 ln = C::BIG ? d.lref[i] : lref[C::BIG ? 0 : m];
            double2 lc = ln;
            if (cells) lc = C::BIG ? d.cref[i] : cref[C::BIG ? 0 : m];
            double2 x = C::BIG ? L.x[i] : own;
            if (FIRE) {
                if (uphill) {
                    const double bdt = -dt / 2.0;
                    x.x += v[m].x * bdt;
                    x.y += v[m].y * bdt;
                    v[m].x = 0.0;
                    v[m].y = 0.0;
                }
                if (dt != dt_kick) dtm[m] = (dt / 2.0) / mass[m];
            }
            v[m].x += f[m].x * dtm[m];
            v[m].y += f[m].y * dtm[m];
            if (FIRE) mix_hot(v[m], f[m], alpha);
            x.x += v[m].x * dt;
            x.y += v[m].y * dt;
            L.x[i] = x;
            if (!C::BIG) own = x;
            const double dx = x.x - ln.x, dy = x.y - ln.y;
            far = far || 3.0 * (dx * dx + dy * dy) > nb.thr;
            const double cx = x.x - lc.x, cy = x.y - lc.y;
            cfar = cfar || (cells && 3.0 * (cx * cx + cy * cy) > nb.cthr);
        }
        if (__builtin_amdgcn_ballot_w64(far) != 0 && lane == 0) L.lflag = step + 1;
        if (__builtin_amdgcn_ballot_w64(cfar) != 0 && lane == 0) L.cflag = step + 1;
        dt_kick = dt;
        __syncthreads();  // every position of the step
        const bool sort = L.cflag == step + 1;
        if (__builtin_expect(sort || L.lflag == step + 1, 0)) {
            const int tid = res_tid();
            if (sort) {  // cells formed anew, particles in cell order (k_cell_*, k_reorder_*)
                auto cell_at = [&](double2 x) -> int {
                    const long long k = (long long)cell_coord(x.x, nb.cs, nb.ncd) +
                                        (long long)cell_coord(x.y, nb.cs, nb.ncd) * nb.ncd;
                    if (k >= 0 && k < ncell) return (int)k;
                    c->bad_pos = 1;  // a non-finite position
                    return 0;
                };
#pragma unroll
                for (int m = 0; m < PPT; ++m) {
                    const int i = tid + m * T;
                    if (i >= n) continue;
                    const double2 x = L.x[i];
                    cell[m] = cell_at(x);
                    sp.P[i] = make_double4(x.x, x.y, L.r[i], mass[m]);
                    sp.vel[i] = v[m];
                    sp.sidx[i] = d.sidx[i];
                    if (d.m1) {
                        sp.m1[i] = d.m1[i];
                        sp.m2[i] = d.m2[i];
                    }
                }
                res_sort(L, n, ncell, cell);
                for (int k = tid; k <= ncell; k += T)
                    d.cell_start[k] = k == 0 ? 0 : L.p.b.cend[k - 1];
#pragma unroll
                for (int m = 0; m < PPT; ++m) {
                    const int i = tid + m * T;
                    if (i >= n) continue;
                    const int o = L.p.b.lst[i];
                    const double4 q = sp.P[o];
                    v[m] = sp.vel[o];
                    d.sidx[i] = sp.sidx[o];
                    if (d.m1) {
                        d.m1[i] = sp.m1[o];
                        d.m2[i] = sp.m2[o];
                    }
                    const double2 x = make_double2(q.x, q.y);
                    L.x[i] = x;
                    if (!C::BIG) own = x;
                    L.r[i] = q.z;
                    mass[m] = q.w;
                    cell[m] = cell_at(x);
                    if (!C::BIG) cref[m] = x;
                    d.cref[i] = x;
                    d.cell_of[i] = cell[m];
                    dtm[m] = (FIRE ? dt / 2.0 : 0.5 * dt_nve) / q.w;
                }
                sorts++;
                __syncthreads();
            }
            if (cells) {
                if (!sort) {
                    for (int k = tid; k < ncell; k += T) L.p.b.cend[k] = d.cell_start[k + 1];
                    __syncthreads();
                }
#pragma unroll
                for (int m = 0; m < PPT; ++m) {
                    const int i = tid + m * T;
                    near[m] = 0;
                    if (i < n)
                        full[m] = res_row_cell(L, R, i, cell[m], nb.ncd, nb.rc2, delta2, p,
                                               near[m]);
                }
            } else {
                const double w = sqrt(nb.rc2) * (1.0 + 1e-9), most = floor(sqrt((double)NP));
                const int nx = (int)fmin(most, floor(nb.Lx / w));
                const int ny = (int)fmin(most, floor(nb.Ly / w));
                const bool grid = nx >= 3 && ny >= 3;
#pragma unroll
                for (int m = 0; m < PPT; ++m) {
                    const int i = tid + m * T;
                    if (!grid || i >= n) continue;
                    // (a non-finite position has no neighbours, whatever its cell)
                    const double2 x = L.x[i];
                    cell[m] = min(max(cell_coord(x.x, nb.Lx / nx, nx), 0), nx - 1) +
                              nx * min(max(cell_coord(x.y, nb.Ly / ny, ny), 0), ny - 1);
                }
                if (grid) res_sort(L, n, nx * ny, cell);
#pragma unroll
                for (int m = 0; m < PPT; ++m) {
                    const int i = tid + m * T;
                    near[m] = 0;
                    if (i < n)
                        full[m] = res_row_verlet(L, R, i, n, grid, grid ? cell[m] % nx : 0,
                                                 grid ? cell[m] / nx : 0, nx, ny, nb.rc2, delta2,
                                                 p, near[m]);
                }
            }
#pragma unroll
            for (int m = 0; m < PPT; ++m) {
                const int i = tid + m * T;
                if (i >= n) continue;
                const double2 x = L.x[i];
                if (!C::BIG) lref[m] = x;
                d.lref[i] = x;
                mx = max(mx, full[m]);
                if (full[m] > d.cap) L.over = 1;
            }
            res_pairs(L, K, n, true, near, len);
            if (L.over) {  // the chain rebuilds (and counts) the list once it has grown
                halt = 1;
                break;
            }
            lists++;
        }
        // forces and the closing kick (k_fire_force, nve_force_body)
        const bool energy = FIRE || step == steps - 1, dense = L.dense != 0;
        double ax[PPT], ay[PPT], e[PPT];
        if (__builtin_expect(dense, 0)) {
            const int tid = res_tid();
#pragma unroll
            for (int m = 0; m < PPT; ++m) {
                ax[m] = ay[m] = e[m] = 0.0;
                if (tid + m * T < n)
                    res_sum_full(L, R, p, tid + m * T, full[m], ax[m], ay[m], e[m]);
            }
            __syncthreads();  // every position has been read
        } else if (energy) {
            res_forces<true>(L, K, p, nc, len, ax, ay, e);
        } else {
            res_forces<false>(L, K, p, nc, len, ax, ay, e);
        }
#pragma unroll
        for (int m = 0; m < PPT; ++m) {
            const int i = tid + m * T, ch = i / WAVE;
            if (ch >= nc) continue;  // uniform over the wave
            double pxv = 0.0, pyv = 0.0, f2 = 0.0;
            if (i < n) {
                const double fx = 0.0 + ax[m], fy = 0.0 + ay[m];
                f[m] = make_double2(fx, fy);
                if (energy) pe[m] = 0.0 + e[m];
                v[m].x += fx * dtm[m];
                v[m].y += fy * dtm[m];
                pxv = fx * v[m].x;
                pyv = fy * v[m].y;
                f2 = fx * fx + fy * fy;
            }
            if (FIRE) {
                const double s = wave_reduce4(pxv, pyv, pe[m], f2);
                if (lane % 16 == 0) L.part[lane / 16][ch] = s;
            }
        }
        if (FIRE) {
            __syncthreads();  // every partial of the step
            if (tid < WAVE) {  // k_fire_ctl: a row of lanes for each sum
                FireCtl F = L.F;
                const double s = res_final<NP / WAVE>(L.part, nc);
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
#pragma unroll
    for (int m = 0; m < PPT; ++m) {
        const int i = tid + m * T, ch = i / WAVE;
        if (ch >= nc) continue;
        double nd = 0.0, cd = 0.0;
        if (i < n) {
            const double2 x = L.x[i];
            const double4 q = make_double4(x.x, x.y, L.r[i], mass[m]);
            d.P0[i] = q;
            if (sorts) d.P1[i] = q;
            d.vel[i] = v[m];
            d.frc[i] = f[m];
            d.pe[i] = pe[m];
            d.nnum[i] = full[m];
            disp_of(d, i, x.x, x.y, nd, cd);
        }
        nd = wave_max(nd);
        cd = wave_max(cd);
        if (lane == 0) {
            L.part[0][ch] = nd;
            L.part[1][ch] = cd;
        }
    }
    mx = wave_max_i(mx);
    if (lane == 0 && mx > 0) atomicMax(&c->max_nnum_all, mx);
    if (FIRE) {
        for (int w = tid; w < (int)(sizeof(FireCtl) / sizeof(int)); w += T)
            ((int*)d.fire)[w] = ((const int*)&L.F)[w];
    }
    __syncthreads();
    // the displacement maxima of the final state by tiles of BLOCK particles (disp_epilogue)
    constexpr int PER = BLOCK / WAVE;
    if (tid * PER < nc) {
        double nd = L.part[0][tid * PER], cd = L.part[1][tid * PER];
        for (int k = tid * PER + 1; k < min(nc, (tid + 1) * PER); ++k) {
            nd = fmax(nd, L.part[0][k]);
            cd = fmax(cd, L.part[1][k]);
        }
        d.pmax_nd[tid] = nd;
        d.pmax_cd[tid] = cd;
    }
    if (tid == 0) {
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

// Whether a system is expected to have near rows and pairs that some class holds.
constexpr double RES_MOST_PAIRS = 3.0 * 2048;
static bool resident_sparse(const ResLoad& l) {
    return l.row <= RES_ROW && l.pairs <= RES_MOST_PAIRS;
}

// The size class of a system: its particles, its cells and, unless it is dense in every class, its
// expected pairs must fit (a class that they outgrow costs more than the next).
static int64_t resident_need(const dpm_system* s) {
    const ResLoad l(s->N, s->box[0] * s->box[1], s->rmin, s->rmax, s->thr_sq);
    int64_t need = std::max(s->N, s->method == DPM_NBR_CELL ? s->ncells : (int64_t)0);
    if (resident_sparse(l)) need = std::max(need, (int64_t)std::ceil(l.pairs / 3.0));
    return need;
}

template <bool FIRE>
static int launch_resident(dpm_system* s, double dt, int steps) {
    const PairParams p = params_of(s);
    const NbrParams nb = nbr_params(s);
    const int64_t need = resident_need(s);
    hipStream_t st = s->stream;
    if (need <= 256)
        hipLaunchKernelGGL((k_resident<FIRE, 512, 256>), dim3(1), dim3(512), 0, st, s->d, s->sp,
                           p, nb, dt, steps, nullptr);
    else if (need <= 512)
        hipLaunchKernelGGL((k_resident<FIRE, 1024, 512>), dim3(1), dim3(1024), 0, st, s->d, s->sp,
                           p, nb, dt, steps, nullptr);
    else if (need <= 1024)
        hipLaunchKernelGGL((k_resident<FIRE, 1024, 1024>), dim3(1), dim3(1024), 0, st, s->d,
                           s->sp, p, nb, dt, steps, nullptr);
    else
        hipLaunchKernelGGL((k_resident<FIRE, 1024, 2048>), dim3(1), dim3(1024), 0, st, s->d,
                           s->sp, p, nb, dt, steps, s->res_rows);
    return check_launch();
}

bool resident_ok(const dpm_system* s, bool fire) {
    const int64_t most = fire ? RESIDENT_MAX_FIRE : RESIDENT_MAX_NVE;
    if (s->kind != DPM_DISK || s->N > most) return false;
    if (s->method == DPM_NBR_CELL) {
        if (s->ncd < 3 || s->ncells > most) return false;
    } else if (s->method != DPM_NBR_VERLET) {
        return false;
    }
    const PairParams p = params_of(s);
    if (!p.fast || !p.fastdiv) return false;
    const ResLoad l(s->N, s->box[0] * s->box[1], s->rmin, s->rmax, s->thr_sq);
    return resident_sparse(l) || s->N <= (fire ? RESIDENT_DENSE_FIRE : RESIDENT_DENSE_NVE);
}

int resident_prepare(dpm_system* s) {
    const bool big = resident_need(s) > 1024;
    if (!big || s->res_rows) return 0;
    return dalloc(s, &s->res_rows, (int64_t)RES_LC * 2048);
}

int resident_nve(dpm_system* s, double dt, int64_t steps) {
    return launch_resident<false>(s, dt, (int)steps);
}

int resident_fire(dpm_system* s, int64_t steps) {
    return launch_resident<true>(s, 0.0, (int)steps);
}

}  // namespace dpm
