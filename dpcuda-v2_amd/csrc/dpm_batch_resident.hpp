// dpm_batch_resident.hpp -- disk systems of the batched engine that one workgroup advances by
// itself (included by dpm_batch.hip, inside namespace dpm).
//
// A disk system of up to RES_MAX_N particles fits a CU: each such system gets a workgroup that
// runs many steps of its jam in one launch -- the phases of the batched step with workgroup
// barriers between them instead of kernel boundaries, in the same arithmetic and the same
// canonical reduction order, so every result bit is that of the per-phase kernels.  Systems need
// nothing from each other, so a small one is not held to the pace of a large one, and a step
// moves no particle data through HBM.
// Up to 2,048 particles k_b_pairs holds the pairs that can touch in LDS and evaluates each once
// (dpm_resident.hpp); beyond, LDS holds positions and radii and k_b_resident walks the rows.
// What bounds it: LDS gathers and the vector pipe of its CU, and for small systems the chain of
// a step's phases.
// Measured, 64 systems jammed, ms (rows walked from both sides, pairs once): up to 256 particles
// 48, 35; 512 63, 47; 1,024 95, 64; 2,048 167, 123.  384 systems of 64 to 2,048 particles
// (log-uniform): 708 ms on the per-phase kernels (seven launches a step), 203, 157.
constexpr int RES_MAX_N = 4096;

// The size classes: a wave or more per SIMD from 256 particles up; systems of more than 512
// particles have a CU's LDS to themselves; 4,096 particles leave no room for rows or pairs, which
// stay in the arena's ELL (L2).
constexpr int RES_CLASSES = 5;
constexpr int RES_LIMIT[RES_CLASSES] = {256, 512, 1024, 2048, 4096};
constexpr int RES_PAIRS_BIG = 3;  // the class of two particles a thread

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

template <int T, int PPT, int LC>
struct ResLds {
    static constexpr int NP = T * PPT;
    double2 x[NP];
    double r[NP];
    unsigned short row[LC > 0 ? LC : 1][NP];
    int cend[NP];  // a cell grid of at most NP cells
    unsigned short lst[NP];
    int wsum[T / WAVE];
    double part[BP_COUNT][NP / WAVE];
    BSys S;
    int far, apply;
};

// The rows of every particle of the system from a cell grid (or, in a box under three cells a
// side, from all pairs): the particles within rc in ascending index, as k_b_build and
// k_b_build_cells list them.  Positions are in LDS; nn[k] receives the row lengths of the
// thread's particles.  Ends without a barrier: a row is read by the thread that wrote it.
template <int T, int PPT, int LC>
__device__ __forceinline__ void res_build(const BDev& b, ResLds<T, PPT, LC>& L,
                                          const PairParams& p, int (&nn)[PPT]) {
    constexpr int NP = T * PPT;
    const BSys& S = L.S;
    const int tid = res_tid(), n = S.n;
    const long long off = S.off;
    const double w = S.rc * (1.0 + 1e-9) * b.cell_scale, rc2 = S.rc2;
    const double dmax = floor(sqrt((double)NP));
    const int nx = (int)fmin(dmax, floor(S.Lx / w)), ny = (int)fmin(dmax, floor(S.Ly / w));
    const bool grid = nx >= 3 && ny >= 3;
    const double csx = S.Lx / nx, csy = S.Ly / ny;
    const int ncell = nx * ny;
    auto cell = [&](double2 x) {
        return bc_coord(x.x, S.Lx, csx, nx) + nx * bc_coord(x.y, S.Ly, csy, ny);
    };
    if (grid) {
        for (int c = tid; c < ncell; c += T) L.cend[c] = 0;
        __syncthreads();
        for (int i = tid; i < n; i += T) atomicAdd(&L.cend[cell(L.x[i])], 1);
        __syncthreads();
        // exclusive scan of the counts: each thread owns a run of consecutive cells
        const int per = (ncell + T - 1) / T;
        const int c0 = min(tid * per, ncell), c1 = min(c0 + per, ncell);
        int local = 0;
        for (int c = c0; c < c1; ++c) local += L.cend[c];
        const int lane = tid % WAVE, wv = tid / WAVE;
        int incl = local;
#pragma unroll
        for (int d = 1; d < WAVE; d <<= 1) {
            const int o = __shfl_up(incl, d, WAVE);
            if (lane >= d) incl += o;
        }
        if (lane == WAVE - 1) L.wsum[wv] = incl;
        __syncthreads();
        int run = incl - local;
        for (int k = 0; k < wv; ++k) run += L.wsum[k];
        for (int c = c0; c < c1; ++c) {
            const int t = L.cend[c];
            L.cend[c] = run;
            run += t;
        }
        __syncthreads();
        for (int i = tid; i < n; i += T)
            L.lst[atomicAdd(&L.cend[cell(L.x[i])], 1)] = (unsigned short)i;
        __syncthreads();
        for (int c = tid; c < ncell; c += T) {  // ascending members (a few per cell)
            const int a = c == 0 ? 0 : L.cend[c - 1], e = L.cend[c];
            for (int u = a + 1; u < e; ++u) {
                const unsigned short v = L.lst[u];
                int k = u - 1;
                while (k >= a && L.lst[k] > v) {
                    L.lst[k + 1] = L.lst[k];
                    --k;
                }
                L.lst[k + 1] = v;
            }
        }
        __syncthreads();
    }
#pragma unroll
    for (int m = 0; m < PPT; ++m) {
        const int i = tid + m * T;
        if (i >= n) continue;
        const double2 xi = L.x[i];
        int cnt = 0;
        auto test = [&](int j) {
            const double2 xj = L.x[j];
            double dx, dy;
            if (p.fast) {
                dx = pbc_rint(xi.x, xj.x, p.Lx, p.invLx);
                dy = pbc_rint(xi.y, xj.y, p.Ly, p.invLy);
            } else {
                dx = pbc(xi.x, xj.x, p.Lx, p.invLx, p.halfLx, 0);
                dy = pbc(xi.y, xj.y, p.Ly, p.invLy, p.halfLy, 0);
            }
            if (dx * dx + dy * dy < rc2) {
                if (LC > 0 && cnt < LC) L.row[cnt][i] = (unsigned short)j;
                else if (cnt < b.cap) b.nbr[(long long)cnt * b.nslot + off + i] = (int)(off + j);
                cnt++;
            }
        };
        if (grid) {  // the nine cells' lists, merged in ascending order
            constexpr int NONE = 0x7fffffff;
            const int cx = bc_coord(xi.x, S.Lx, csx, nx), cy = bc_coord(xi.y, S.Ly, csy, ny);
            int pa[9], pe[9], h[9];
#pragma unroll
            for (int t = 0; t < 9; ++t) {
                int x = cx + t % 3 - 1, y = cy + t / 3 - 1;
                x = x < 0 ? x + nx : (x >= nx ? x - nx : x);
                y = y < 0 ? y + ny : (y >= ny ? y - ny : y);
                const int c = x + nx * y;
                pa[t] = c == 0 ? 0 : L.cend[c - 1];
                pe[t] = L.cend[c];
                h[t] = pa[t] < pe[t] ? L.lst[pa[t]] : NONE;
            }
            while (true) {
                int best = h[0], bt = 0;
#pragma unroll
                for (int t = 1; t < 9; ++t)
                    if (h[t] < best) {
                        best = h[t];
                        bt = t;
                    }
                if (best == NONE) break;
#pragma unroll
                for (int t = 0; t < 9; ++t)
                    if (t == bt) {
                        pa[t]++;
                        h[t] = pa[t] < pe[t] ? L.lst[pa[t]] : NONE;
                    }
                if (best != i) test(best);
            }
        } else {
            for (int j = 0; j < n; ++j)
                if (j != i) test(j);
        }
        nn[m] = cnt;
        b.lref[off + i] = xi;
    }
}

// Force and energy sums of particle i over its row (k_b_force's loop on LDS).  EXACT: the
// reference's minimum image, for a box too small for the branch-free one.
template <bool EXACT, int T, int PPT, int LC>
__device__ __forceinline__ void res_row_forces(const BDev& b, const ResLds<T, PPT, LC>& L,
                                               const PairParams& p, long long off, int i,
                                               double4 qi, int nn, double& ax, double& ay,
                                               double& e) {
    // entry k of the row: k is the same in the whole wave; entries past a row's end are some
    // particle of the system (LDS rows hold nothing else) and add +0.0
    auto entry = [&](int k) -> int {
        if (k < LC) return L.row[k][i];
        return k < nn ? (int)(b.nbr[(long long)k * b.nslot + off + i] - off) : 0;
    };
    ax = 0.0;
    ay = 0.0;
    e = 0.0;
    int j0 = entry(0), j1 = entry(1);
    for (int k = 0; __builtin_amdgcn_ballot_w64(k < nn) != 0; k += 2) {
        const double2 x0 = L.x[j0], x1 = L.x[j1];
        const double4 q0 = make_double4(x0.x, x0.y, L.r[j0], 0.0);
        const double4 q1 = make_double4(x1.x, x1.y, L.r[j1], 0.0);
        if (__builtin_amdgcn_ballot_w64(k + 2 < nn) != 0) {
            j0 = entry(k + 2);
            j1 = entry(k + 3);
        }
        double fx, fy, ie;
        ie = pair_hot<true, EXACT>(qi, q0, k < nn, p, fx, fy);
        ax += fx;
        ay += fy;
        e += ie;
        ie = pair_hot<true, EXACT>(qi, q1, k + 1 < nn, p, fx, fy);
        ax += fx;
        ay += fy;
        e += ie;
    }
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

// b_eval_disk on positions in LDS
template <int T, int PPT, int LC>
__device__ __forceinline__ void res_eval(const BDev& b, const ResLds<T, PPT, LC>& L,
                                         const PairParams& p, long long off, int i, double4 qi,
                                         int nn, double& sxx, double& syy, double& z) {
    double axx = qi.w * 0.0 * 0.0, ayy = axx;  // (the kinetic terms, of zero velocity)
    int c = 0;
    for (int k = 0; k < nn; ++k) {
        const int j = k < LC ? (int)L.row[k][i]
                             : (int)(b.nbr[(long long)k * b.nslot + off + i] - off);
        const double2 xj = L.x[j];
        const double rj = L.r[j];
        const double xd = pbc(qi.x, xj.x, p.Lx, p.invLx, p.halfLx, p.fast);
        const double yd = pbc(qi.y, xj.y, p.Ly, p.invLy, p.halfLy, p.fast);
        const double4 qj = make_double4(xj.x, xj.y, rj, 0.0);
        double fx, fy;
        if (p.fast) pair_hot<false>(qi, qj, true, p, fx, fy);
        else pair_hot<false, true>(qi, qj, true, p, fx, fy);
        axx += xd * fx / 2;
        ayy += yd * fy / 2;
        const double dist = sqrt(xd * xd + yd * yd);
        if (dist < qi.z + rj) c++;
    }
    const double area = L.S.Lx * L.S.Ly;
    sxx = axx / area;
    syy = ayy / area;
    z = (double)c;
}

// `steps` steps of each listed system (fewer once it finishes): ids[blockIdx.x] names the
// workgroup's system, base is the number of batched steps before this launch.  Needs the
// pair law's short sequences (BDev::fastdiv) and n <= T * PPT.
template <int T, int PPT, int LC>
__global__ __launch_bounds__(T) void k_b_resident(BDev b, const int* ids, long long base,
                                                  int steps) {
    constexpr int NP = T * PPT;
    __shared__ ResLds<T, PPT, LC> L;
    const int sid = ids[blockIdx.x], tid = threadIdx.x, lane = tid % WAVE;
    static_assert(sizeof(BSys) % sizeof(int) == 0, "the record is copied by words");
    for (int w = tid; w < (int)(sizeof(BSys) / sizeof(int)); w += T)
        ((int*)&L.S)[w] = ((const int*)(b.sys + sid))[w];
    __syncthreads();
    BSys& S = L.S;
    if (S.mode == BM_DONE || S.mode == BM_EMPTY) return;
    const int n = S.n, nc = S.nc;
    const long long off = S.off;
    double4 q[PPT];
    double2 v[PPT], f[PPT];
    double dtm[PPT];
    int nn[PPT], mx = 0;
    if (tid == 0) L.far = S.far;
#pragma unroll
    for (int m = 0; m < PPT; ++m) {
        const int i = tid + m * T;
        const bool live = i < n;
        q[m] = live ? b.P[off + i] : make_double4(0.0, 0.0, 1.0, 1.0);
        v[m] = live ? b.vel[off + i] : make_double2(0.0, 0.0);
        f[m] = live ? b.frc[off + i] : make_double2(0.0, 0.0);
        nn[m] = live ? b.nnum[off + i] : 0;
        dtm[m] = 0.0;
        L.x[i] = make_double2(q[m].x, q[m].y);
        L.r[i] = q[m].z;
        for (int k = 0; k < LC; ++k)
            L.row[k][i] = live && !S.rebuild && k < min(nn[m], b.cap)
                              ? (unsigned short)(b.nbr[(long long)k * b.nslot + off + i] - off)
                              : (unsigned short)0;
    }
    __syncthreads();
    PairParams p = res_params(b, S);
    const double thr2 = S.thr2;
    for (int step = 0; step < steps; ++step) {
        // the controller's operations, then Fire::step's first half (b_prep_slot, b_move_slot)
        const int mode = S.mode;
        if (mode == BM_DONE) break;
        const bool start = mode == BM_PROLOGUE;
        if (mode != BM_FIRE) p = res_params(b, S);
        if (start || S.snap_op != 0) {
#pragma unroll
            for (int m = 0; m < PPT; ++m) {
                const int i = res_tid() + m * T;
                if (i >= n) continue;
                q[m] = res_slot_ops(b, S, off + i, q[m]);
                L.x[i] = make_double2(q[m].x, q[m].y);
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
                const double2 l = b.lref[off + i];
                if (uphill) {
                    const double bdt = -dt / 2.0;
                    q[m].x += v[m].x * bdt;
                    q[m].y += v[m].y * bdt;
                    v[m].x = 0.0;
                    v[m].y = 0.0;
                }
                dtm[m] = (dt / 2.0) / q[m].w;
                v[m].x += f[m].x * dtm[m];
                v[m].y += f[m].y * dtm[m];
                mix_one(v[m], f[m], alpha);
                q[m].x += v[m].x * dt;
                q[m].y += v[m].y * dt;
                L.x[i] = make_double2(q[m].x, q[m].y);
                const double dx = q[m].x - l.x, dy = q[m].y - l.y;
                const double d2 = dx * dx + dy * dy;
                far = far || 3.0 * d2 > thr2;
            }
            if (__builtin_amdgcn_ballot_w64(far) != 0 && lane == 0) L.far = 1;
        }
        __syncthreads();  // every position of the step
        if (S.rebuild || mode == BM_RESTORE || L.far) {  // b_rebuild_now
            res_build<T, PPT, LC>(b, L, p, nn);
#pragma unroll
            for (int m = 0; m < PPT; ++m) mx = max(mx, nn[m]);
        }
        if (mode != BM_RESTORE) {  // forces, the closing kick and the chunk partials (k_b_force)
#pragma unroll
            for (int m = 0; m < PPT; ++m) {
                const int i = tid + m * T, ch = i / WAVE;
                if (ch >= nc) continue;  // uniform over the wave
                const bool live = i < n;
                const int row = live ? min(nn[m], b.cap) : 0;
                double ax, ay, e;
                if (p.fast) res_row_forces<false>(b, L, p, off, i, q[m], row, ax, ay, e);
                else res_row_forces<true>(b, L, p, off, i, q[m], row, ax, ay, e);
                double pxv = 0.0, pyv = 0.0, pe = 0.0, f2 = 0.0;
                if (live) {
                    const double fx = 0.0 + ax, fy = 0.0 + ay;
                    f[m] = make_double2(fx, fy);
                    pe = 0.0 + e;
                    if (mode == BM_FIRE) {
                        v[m].x += fx * dtm[m];
                        v[m].y += fy * dtm[m];
                    }
                    pxv = fx * v[m].x;
                    pyv = fy * v[m].y;
                    f2 = fx * fx + fy * fy;
                }
                const double s0 = wave_tree_sum(pxv), s1 = wave_tree_sum(pyv);
                const double s2 = wave_tree_sum(pe), s3 = wave_max(f2);
                if (lane == 0) {
                    L.part[BP_PX][ch] = s0;
                    L.part[BP_PY][ch] = s1;
                    L.part[BP_PE][ch] = s2;
                    L.part[BP_F2][ch] = s3;
                }
            }
        }
        __syncthreads();  // every partial of the step
        if (tid < WAVE) {  // k_b_ctl
            const double px = res_final_sum(L.part[BP_PX], nc);
            const double py = res_final_sum(L.part[BP_PY], nc);
            const double pe = res_final_sum(L.part[BP_PE], nc);
            const double fm = wave_max(lane < nc ? L.part[BP_F2][lane] : 0.0);
            if (lane == 0) {
                b_step_begin(S);
                if (mode != BM_RESTORE) {
                    L.far = 0;
                    if (b_fire_decide(S, pe, px + py, fm)) S.mode = BM_EVAL;
                }
            }
        }
        __syncthreads();  // the record for the rest of this step and the next
        if (S.mode != BM_EVAL) continue;
        // the end of a minimisation (k_b_eval, k_b_jam)
        bool far = false;
#pragma unroll
        for (int m = 0; m < PPT; ++m) {
            const int i = res_tid() + m * T, ch = i / WAVE;
            if (ch >= nc) continue;
            double sxx = 0.0, syy = 0.0, r2 = 0.0, z = 0.0;
            if (i < n) {
                v[m] = make_double2(0.0, 0.0);
                res_eval<T, PPT, LC>(b, L, p, off, i, q[m], min(nn[m], b.cap), sxx, syy, z);
                r2 = q[m].z * q[m].z;
                const double2 l = b.lref[off + i];
                const double dx = q[m].x - l.x, dy = q[m].y - l.y;
                const double d2 = dx * dx + dy * dy;
                far = far || 3.0 * d2 > thr2;
            }
            const double s0 = wave_tree_sum(sxx), s1 = wave_tree_sum(syy);
            const double s2 = wave_tree_sum(r2), s3 = wave_tree_sum(z);
            if (lane == 0) {
                L.part[BP_SXX][ch] = s0;
                L.part[BP_SYY][ch] = s1;
                L.part[BP_R2][ch] = s2;
                L.part[BP_Z][ch] = s3;
            }
        }
        if (__builtin_amdgcn_ballot_w64(far) != 0 && lane == 0) L.far = 1;
        __syncthreads();
        if (tid < WAVE) {
            const double sxx = res_final_sum(L.part[BP_SXX], nc);
            const double syy = res_final_sum(L.part[BP_SYY], nc);
            const double pe = res_final_sum(L.part[BP_PE], nc);
            const double r2 = res_final_sum(L.part[BP_R2], nc);
            const double z = res_final_sum(L.part[BP_Z], nc);  // whole numbers
            if (lane == 0) L.apply = b_jam_step(b, S, sxx, syy, z, pe, r2, base + step + 1);
        }
        __syncthreads();
        if (S.mode != BM_DONE) continue;
        if (L.apply) {  // a finished system sees the controller's last operations at once
#pragma unroll
            for (int m = 0; m < PPT; ++m) {
                const int i = tid + m * T;
                if (i < n) q[m] = res_slot_ops(b, S, off + i, q[m]);
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
#pragma unroll
    for (int m = 0; m < PPT; ++m) {
        const int i = tid + m * T;
        if (i >= n) continue;
        b.P[off + i] = q[m];
        b.vel[off + i] = v[m];
        b.frc[off + i] = f[m];
        b.nnum[off + i] = nn[m];
        for (int k = 0; k < min(nn[m], LC); ++k)
            b.nbr[(long long)k * b.nslot + off + i] = (int)(off + L.row[k][i]);
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

// ---- systems whose pairs fit LDS (dpm_resident.hpp) ------------------------------------------
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
// entries a workgroup (two particles a thread).  Needs the pair law's short sequences
// (BDev::fastdiv) and n <= NP.
template <int T, int NP>
__global__ __launch_bounds__(T) void k_b_pairs(BDev b, const int* ids, long long base, int steps,
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
    const double delta2 = 2.0 * sqrt(fmax(thr2, 0.0) / 3.0);
    // the near rows of the list that the last launch left, in the present box
    auto load_near = [&](bool any) {
#pragma unroll
        for (int m = 0; m < PPT; ++m) {
            const int i = res_tid() + m * T;
            near[m] = any && i < n ? res_load_row(L, R, b.lref, i, full[m], delta2, p) : 0;
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
