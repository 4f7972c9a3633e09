// dpm_batch_resident.hpp -- disk systems of the batched engine that one workgroup advances by
// itself (included by dpm_batch.hip, inside namespace dpm).
//
// A disk system of up to RES_MAX_N particles fits a CU: each such system gets a workgroup that
// runs many steps of its jam in one launch -- the phases of the batched step with workgroup
// barriers between them instead of kernel boundaries, in the same arithmetic and the same
// canonical reduction order, so every result bit is that of the per-phase kernels.  Systems need
// nothing from each other, so a small one is not held to the pace of a large one, and a step
// moves no particle data through HBM.
// Up to 2,048 particles LDS holds the pairs that can touch, each evaluated once; beyond, it holds
// positions and radii and the near rows are walked (dpm_resident.hpp).
// What bounds it: the vector pipe of its CU (busy 55 to 58 % of the time from 512 particles up, LDS
// 7 to 10 %) and the chain of a step's phases, in which waves wait 57 to 74 % of their time.
// Measured, 64 systems jammed, ms (full rows walked from both sides, as it is now): up to 256
// particles 48, 35; 512 63, 47; 1,024 95, 64; 2,048 167, 123; 4,096 397, 308.  384 systems of 64
// to 2,048 particles (log-uniform): 708 ms on the per-phase kernels (seven launches a step), 203,
// 157.
constexpr int RES_MAX_N = 4096;

// The size classes: a wave or more per SIMD from 256 particles up; systems of more than 512
// particles have a CU's LDS to themselves.  The first class is for more systems of its size than
// there are CUs (RES_CROWD): its two waves leave room for several systems a CU, where the next
// class's eight take them all.  us a FIRE step (row builds of a thread a row and the per-phase
// kernels, class of 256, of 128): 1,024 systems of 16 disks 35, 16, 6.8; 16,384 of 16 157, 229,
// 66; 8,192 of 64 128, 222, 53.
constexpr int RES_CLASSES = 6;
constexpr int RES_LIMIT[RES_CLASSES] = {128, 256, 512, 1024, 2048, 4096};
constexpr int RES_CROWD = 256;
constexpr int RES_ROWS = 4;  // from this class on, the near rows lie in HBM

// bparams, held in scalar registers (every lane reads the same record)
__device__ __forceinline__ PairParams res_params(const BDev& b, const BSys& S) {
    PairParams p = bparams(b, S);
    p.Lx = uniform_d(p.Lx);
    p.Ly = uniform_d(p.Ly);
    p.invLx = uniform_d(p.invLx);
    p.invLy = uniform_d(p.invLy);
    p.halfLx = uniform_d(p.halfLx);
    p.halfLy = uniform_d(p.halfLy);
    p.e_c = uniform_d(p.e_c);
    p.fast = __builtin_amdgcn_readfirstlane(p.fast);
    return p;
}

// A chunk sum's final stage over at most 64 partials, by one wave (wave_final_sum)
__device__ __forceinline__ double res_final_sum(const double* P, int nc) {
    const int t = threadIdx.x % WAVE;
    return wave_tree_sum(t < nc ? 0.0 + P[t] : 0.0);
}

// b_slot_ops on a particle held in registers
__device__ __forceinline__ double4 res_slot_ops(const BDev& b, const BSys& S, long long i,
                                                double4 q) {
    if (S.snap_op == 2) q = b.snap[i];
    if (S.snap_op == 1) b.snap[i] = q;
    if (S.scale_f != 0.0) {
        q.x *= S.scale_f;
        q.y *= S.scale_f;
    }
    if (S.snap_op == 3) b.snap[i] = q;
    return q;
}

template <int T, int NP>
struct ResBatch : ResCore<T, NP> {
    double part[4][NP / WAVE];  // by chunk: F_x v_x, PE, F_y v_y, max F^2
    double eval[4][NP / WAVE];  // sigma_xx, sigma_yy, r^2, contacts
    BSys S;
    double pe;  // the last step's energy
    int far, apply;
};

// b_fire_decide on the record in LDS: its fields are loaded together (one wave; every lane forms
// the same values)
__device__ __forceinline__ bool res_decide(BSys& S, double px, double py, double pe, double fm) {
    FireCtl F;
    F.alpha = S.alpha;
    F.alpha_init = S.J.alpha0;
    F.dt = S.dt;
    F.dt_max = S.dt_max;
    F.dt_min = S.dt_min;
    F.avg_pe_target = S.J.pe_t;
    F.avg_pe_diff_target = S.J.pe_diff_t;
    F.fmax_target_sq = S.J.fmax2;
    F.dof = (double)S.n;
    F.last_avg_pe = S.last_avg_pe;
    F.power = S.power;
    F.n_good = S.n_good;
    F.n_bad = S.n_bad;
    F.step = S.step;
    F.max_steps = S.J.max_steps;
    F.stopped = S.stopped;
    F.done = S.done;
    F.converged = S.converged;
    F.uphill = S.uphill;
    const bool ended = S.mode == BM_PROLOGUE ? fire_begin(F, px, py, pe, fm, nullptr)
                                             : fire_advance(F, px, py, pe, fm, nullptr);
    S.rebuild = 0;  // the list this step used is current
    S.mode = BM_FIRE;
    S.fmax_sq = F.fmax_sq;
    S.avg_pe = F.avg_pe;
    S.last_avg_pe = F.last_avg_pe;
    S.power = F.power;
    S.alpha = F.alpha;
    S.dt = F.dt;
    S.n_good = F.n_good;
    S.n_bad = F.n_bad;
    S.step = F.step;
    S.stopped = F.stopped;
    S.done = F.done;
    S.converged = F.converged;
    S.uphill = F.uphill;
    return ended;
}

// b_eval_disk on positions in LDS and the full row in HBM
template <int T, int NP>
__device__ __forceinline__ void res_eval_full(const ResBatch<T, NP>& L, const ResRows& R,
                                              const PairParams& p, int i, double mass, int nn,
                                              double& sxx, double& syy, double& z) {
    const double2 x = L.x[i];
    const double r = L.r[i];
    double axx = mass * 0.0 * 0.0, ayy = axx;  // (the kinetic terms, of zero velocity)
    int c = 0;
#pragma unroll 1
    for (int k = 0; k < nn; ++k) {
        const int j = (int)(R.nbr[(long long)k * R.stride + R.base + i] - R.base);
        const double2 xj = L.x[j];
        const double rj = L.r[j];
        const double xd = pbc(x.x, xj.x, p.Lx, p.invLx, p.halfLx, p.fast);
        const double yd = pbc(x.y, xj.y, p.Ly, p.invLy, p.halfLy, p.fast);
        const double4 qi = make_double4(x.x, x.y, r, 0.0);
        const double4 qj = make_double4(xj.x, xj.y, rj, 0.0);
        double fx, fy;
        if (p.fast) pair_hot<false>(qi, qj, true, p, fx, fy);
        else pair_hot<false, true>(qi, qj, true, p, fx, fy);
        axx += xd * fx / 2;
        ayy += yd * fy / 2;
        const double dist = sqrt(xd * xd + yd * yd);
        if (dist < r + rj) c++;
    }
    const double area = L.S.Lx * L.S.Ly;
    sxx = axx / area;
    syy = ayy / area;
    z = (double)c;
}

// `steps` steps of each listed system (fewer once it finishes): ids[blockIdx.x] names the
// workgroup's system, base is the number of batched steps before this launch; rows: RES_LC * NP
// entries a workgroup (more than a particle a thread).  Needs the pair law's short sequences
// (BDev::fastdiv) and n <= NP.
template <int T, int NP>
__global__ __launch_bounds__(T) void k_b_resident(BDev b, const int* ids, long long base, int steps,
                                               unsigned short* rows) {
    using C = ResCore<T, NP>;
    constexpr int PPT = C::PPT;
    __shared__ ResBatch<T, NP> L;
    const int sid = ids[blockIdx.x], tid = threadIdx.x, lane = tid % WAVE;
    static_assert(sizeof(BSys) % sizeof(int) == 0, "the record is copied by words");
    for (int w = tid; w < (int)(sizeof(BSys) / sizeof(int)); w += T)
        ((int*)&L.S)[w] = ((const int*)(b.sys + sid))[w];
    __syncthreads();
    BSys& S = L.S;
    if (S.mode == BM_DONE || S.mode == BM_EMPTY) return;
    const int n = S.n, nc = S.nc;
    const long long off = S.off;
    const ResRows R{b.nbr, b.nslot, off, b.cap};
    ResKept<T, NP> K;
    K.row = rows + (C::BIG ? (long long)blockIdx.x * RES_LC * NP : 0);
    double mass[PPT], dtm[PPT];
    double2 v[PPT], f[PPT];
    double2 lref[C::BIG ? 1 : PPT];  // (two particles a thread: read from HBM)
    int full[PPT], len[PPT], near[PPT], mx = 0;
    if (tid == 0) L.far = S.far;
#pragma unroll
    for (int m = 0; m < PPT; ++m) {
        const int i = tid + m * T;
        const bool live = i < n;
        const double4 q = live ? b.P[off + i] : make_double4(0.0, 0.0, 1.0, 1.0);
        v[m] = live ? b.vel[off + i] : make_double2(0.0, 0.0);
        f[m] = live ? b.frc[off + i] : make_double2(0.0, 0.0);
        full[m] = live ? b.nnum[off + i] : 0;
        if (!C::BIG) lref[m] = live ? b.lref[off + i] : make_double2(0.0, 0.0);
        mass[m] = q.w;
        dtm[m] = 0.0;
        if (i < NP) {
            L.x[i] = make_double2(q.x, q.y);
            L.r[i] = q.z;
        }
    }
    __syncthreads();
    PairParams p = res_params(b, S);
    const double thr2 = uniform_d(S.thr2);
    const double delta2 = res_reach(thr2);
    // the near rows of the list that the last launch left, in the present box
    auto load_near = [&](bool any) {
#pragma unroll
        for (int m = 0; m < PPT; ++m) {
            const int i = res_tid() + m * T;
            near[m] = any && i < n ? res_load_row(L, R, b.lref, i, full[m], delta2, p) : 0;
            res_keep_row(L, K, i, near[m]);
        }
        res_pairs(L, K, n, p.fast != 0, near, len);
    };
    load_near(!S.rebuild);
    double dt_kick = -1.0;  // the time step that dtm was formed for
    for (int step = 0; step < steps; ++step) {
        // the controller's operations, then Fire::step's first half (b_prep_slot, b_move_slot)
        const int mode = S.mode;
        if (mode == BM_DONE) break;
        const bool start = mode == BM_PROLOGUE;
        if (mode != BM_FIRE) p = res_params(b, S);
        if (__builtin_expect(start || S.snap_op != 0, 0)) {
#pragma unroll
            for (int m = 0; m < PPT; ++m) {
                const int i = res_tid() + m * T;
                if (i >= n) continue;
                const double2 x = L.x[i];
                const double4 q = res_slot_ops(b, S, off + i,
                                               make_double4(x.x, x.y, L.r[i], mass[m]));
                L.x[i] = make_double2(q.x, q.y);
                if (start) v[m] = make_double2(0.0, 0.0);
            }
        }
        if (mode == BM_FIRE) {
            const double dt = uniform_d(S.dt), alpha = uniform_d(S.alpha);
            const int uphill = S.uphill;
            bool far = false;
#pragma unroll
            for (int m = 0; m < PPT; ++m) {
                const int i = tid + m * T;
                if (i >= n) continue;
                const double2 l = C::BIG ? b.lref[off + i] : lref[C::BIG ? 0 : m];
                double2 x = L.x[i];
                if (uphill) {
                    const double bdt = -dt / 2.0;
                    x.x += v[m].x * bdt;
                    x.y += v[m].y * bdt;
                    v[m].x = 0.0;
                    v[m].y = 0.0;
                }
                if (dt != dt_kick) dtm[m] = (dt / 2.0) / mass[m];
                v[m].x += f[m].x * dtm[m];
                v[m].y += f[m].y * dtm[m];
                mix_hot(v[m], f[m], alpha);
                x.x += v[m].x * dt;
                x.y += v[m].y * dt;
                L.x[i] = x;
                const double dx = x.x - l.x, dy = x.y - l.y;
                far = far || 3.0 * (dx * dx + dy * dy) > thr2;
            }
            dt_kick = dt;
            if (__builtin_amdgcn_ballot_w64(far) != 0 && lane == 0) L.far = 1;
        }
        __syncthreads();  // every position of the step
        const bool rebuild = S.rebuild || mode == BM_RESTORE || L.far;  // b_rebuild_now
        if (__builtin_expect(rebuild, 0)) {
            const double w = S.rc * (1.0 + 1e-9) * b.cell_scale, rc2 = S.rc2;
            const double most = floor(sqrt((double)NP));
            const int nx = (int)fmin(most, floor(S.Lx / w)), ny = (int)fmin(most, floor(S.Ly / w));
            const bool grid = nx >= 3 && ny >= 3;
            int cell[PPT];
#pragma unroll
            for (int m = 0; m < PPT; ++m) {
                const int i = res_tid() + m * T;
                cell[m] = 0;
                if (!grid || i >= n) continue;
                const double2 x = L.x[i];
                cell[m] = bc_coord(x.x, S.Lx, S.Lx / nx, nx) +
                          nx * bc_coord(x.y, S.Ly, S.Ly / ny, ny);
            }
            if (grid) res_sort(L, n, nx * ny, cell);
#pragma unroll
            for (int m = 0; m < PPT; ++m) {
                const int i = res_tid() + m * T;
                near[m] = 0;
                if (i >= n) continue;
                full[m] = res_row_verlet(L, R, i, n, grid, grid ? cell[m] % nx : 0,
                                         grid ? cell[m] / nx : 0, nx, ny, rc2, delta2, p,
                                         near[m]);
                res_keep_row(L, K, i, near[m]);
                mx = max(mx, full[m]);
                const double2 x = L.x[i];
                b.lref[off + i] = x;
                if (!C::BIG) lref[m] = x;
            }
            res_pairs(L, K, n, p.fast != 0, near, len);
        } else if (start) {
            // the box has changed under the list: this evaluation takes the full rows, as the
            // displacements are not looked at before the first move
            load_near(true);
        }
        if (mode != BM_RESTORE) {  // forces, the closing kick and the chunk partials (k_b_force)
            double ax[PPT], ay[PPT], e[PPT];
            if (__builtin_expect(L.dense != 0 || (start && !rebuild), 0)) {
#pragma unroll
                for (int m = 0; m < PPT; ++m) {
                    const int i = res_tid() + m * T;
                    ax[m] = ay[m] = e[m] = 0.0;
                    if (i < n) res_sum_full(L, R, p, i, full[m], ax[m], ay[m], e[m]);
                }
            } else {
                res_forces<true>(L, K, p, nc, len, ax, ay, e);
            }
#pragma unroll
            for (int m = 0; m < PPT; ++m) {
                const int i = tid + m * T, ch = i / WAVE;
                if (ch >= nc) continue;  // uniform over the wave
                double pxv = 0.0, pyv = 0.0, pe = 0.0, f2 = 0.0;
                if (i < n) {
                    const double fx = 0.0 + ax[m], fy = 0.0 + ay[m];
                    f[m] = make_double2(fx, fy);
                    pe = 0.0 + e[m];
                    if (mode == BM_FIRE) {
                        v[m].x += fx * dtm[m];
                        v[m].y += fy * dtm[m];
                    }
                    pxv = fx * v[m].x;
                    pyv = fy * v[m].y;
                    f2 = fx * fx + fy * fy;
                }
                const double s = wave_reduce4(pxv, pyv, pe, f2);
                if (lane % 16 == 0) L.part[lane / 16][ch] = s;
            }
        }
        __syncthreads();  // every partial of the step
        if (tid < WAVE) {  // k_b_ctl
            if (mode != BM_RESTORE) {
                const double s = res_final<NP / WAVE>(L.part, nc);
                const double pe = lane_value(s, 16);
                b_step_begin(S);
                const bool ended = res_decide(S, lane_value(s, 0), lane_value(s, 32), pe,
                                              lane_value(s, 48));
                L.pe = pe;
                L.far = 0;
                if (ended) S.mode = BM_EVAL;
            } else if (lane == 0) {
                b_step_begin(S);
            }
        }
        __syncthreads();  // the record for the rest of this step and the next
        if (__builtin_expect(S.mode != BM_EVAL, 1)) continue;
        // the end of a minimisation (k_b_eval, k_b_jam)
        bool far = false;
#pragma unroll
        for (int m = 0; m < PPT; ++m) {
            const int i = res_tid() + m * T, ch = i / WAVE;
            if (ch >= nc) continue;
            double sxx = 0.0, syy = 0.0, r2 = 0.0, z = 0.0;
            if (i < n) {
                v[m] = make_double2(0.0, 0.0);
                res_eval_full(L, R, p, i, mass[m], min(full[m], b.cap), sxx, syy, z);
                r2 = L.r[i] * L.r[i];
                const double2 l = b.lref[off + i], x = L.x[i];
                const double dx = x.x - l.x, dy = x.y - l.y;
                far = far || 3.0 * (dx * dx + dy * dy) > thr2;
            }
            const double s0 = wave_tree_sum(sxx), s1 = wave_tree_sum(syy);
            const double s2 = wave_tree_sum(r2), s3 = wave_tree_sum(z);
            if (lane == 0) {
                L.eval[0][ch] = s0;
                L.eval[1][ch] = s1;
                L.eval[2][ch] = s2;
                L.eval[3][ch] = s3;
            }
        }
        if (__builtin_amdgcn_ballot_w64(far) != 0 && lane == 0) L.far = 1;
        __syncthreads();
        if (tid < WAVE) {
            const double sxx = res_final_sum(L.eval[0], nc);
            const double syy = res_final_sum(L.eval[1], nc);
            const double r2 = res_final_sum(L.eval[2], nc);
            const double z = res_final_sum(L.eval[3], nc);  // whole numbers
            if (lane == 0) L.apply = b_jam_step(b, S, sxx, syy, z, L.pe, r2, base + step + 1);
        }
        __syncthreads();
        if (S.mode != BM_DONE) continue;
        if (L.apply) {  // a finished system sees the controller's last operations at once
#pragma unroll
            for (int m = 0; m < PPT; ++m) {
                const int i = res_tid() + m * T;
                if (i >= n) continue;
                const double2 x = L.x[i];
                const double4 q = res_slot_ops(b, S, off + i,
                                               make_double4(x.x, x.y, L.r[i], mass[m]));
                L.x[i] = make_double2(q.x, q.y);
            }
        }
        __syncthreads();
        if (tid == 0) {
            S.snap_op = 0;
            S.scale_f = 0.0;
            const int k = atomicAdd(&b.flags[2], 1);
            b.done_list[k % b.nsys] = sid;
        }
        break;
    }
    // the state a later launch goes on from
    __syncthreads();
#pragma unroll
    for (int m = 0; m < PPT; ++m) {
        const int i = tid + m * T;
        if (i >= n) continue;
        const double2 x = L.x[i];
        b.P[off + i] = make_double4(x.x, x.y, L.r[i], mass[m]);
        b.vel[off + i] = v[m];
        b.frc[off + i] = f[m];
        b.nnum[off + i] = full[m];
    }
    if (tid == 0) S.far = L.far;
    mx = wave_max_i(mx);
    if (lane == 0) {
        atomicMax(&b.flags[1], mx);
        if (mx > b.cap) atomicMax(&b.flags[0], 1);
    }
    __syncthreads();
    for (int w = tid; w < (int)(sizeof(BSys) / sizeof(int)); w += T)
        ((int*)(b.sys + sid))[w] = ((const int*)&L.S)[w];
}
