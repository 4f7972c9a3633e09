// dpm_kernels.hpp -- launch helpers shared between the library's .hip sources.
#pragma once
#include <mutex>
#include <vector>

#include "dpm_internal.hpp"

namespace dpm {

inline PairParams pair_params(const dpm_system* s, double e_c, double n_c) {
    PairParams p{};
    p.Lx = s->box[0];
    p.Ly = s->box[1];
    p.invLx = 1.0 / s->box[0];
    p.invLy = 1.0 / s->box[1];
    p.halfLx = 0.5 * s->box[0];
    p.halfLy = 0.5 * s->box[1];
    p.e_c = e_c;
    p.n_c = n_c;
    p.ncm1 = n_c - 1.0;
    p.two_nc = 2.0 * n_c;
    // x/(2 n_c) == x*(1/(2 n_c)) exactly when 2 n_c is a power of two
    int ex;
    double m = frexp(p.two_nc, &ex);
    p.inv2nc = (m == 0.5) ? 1.0 / p.two_nc : 0.0;
    p.fast = 0;
    return p;
}

inline dim3 pgrid(int64_t n) {
    return dim3((unsigned)std::max<int64_t>(1, (n + BLOCK - 1) / BLOCK));
}

// which per-particle quantity a chunk-sum kernel reduces
enum SumWhat {
    S_PE = 0, S_KE, S_FXVX, S_FYVY, S_FX, S_FY, S_SXX, S_SYY, S_SXY, S_SYX, S_VX, S_VY, S_R2,
    S_TQW, S_COUNT, S_VCOUNT
};
enum MaxWhat { M_ND = 0, M_CD, M_F2, M_T2 };

// How a loop kernel decides whether to run: G_NORMAL inside a chunk (skip after a
// halt, halt on a matching rebuild request), G_RESUME in the rebuild chain (run only
// to finish a halted step), G_ALWAYS unconditionally, G_STEP inside a chunk of the rigid NVE
// loop (skip after a halt; the FIRE state is not looked at).
enum Gate { G_NORMAL = 0, G_RESUME = 1, G_ALWAYS = 2, G_STEP = 3 };

// ---- control-block helpers shared by the loop kernels ----
constexpr long long STAMP_STRIDE = 8192;  // > any chunk length
__device__ __forceinline__ long long stamp(long long epoch, int pos) {
    return epoch * STAMP_STRIDE + pos + 1;
}

// The end of a launch unit: copies the control block into slot (pub_seq mod 4) of the
// pinned host mirror and advances pub_seq; the host reads the slot once the event behind
// the unit has completed.  Called by every thread of one block, after the block's last
// write to the control block.
__device__ __forceinline__ void publish_ctl(const Dev& d) {
    Ctl* c = d.ctl;
    const int k = c->pub_seq;
    constexpr int NW = (int)(sizeof(Ctl) / sizeof(int));
    int* dst = (int*)(d.hpub + (k & 3));
    const int* src = (const int*)c;
    for (int w = threadIdx.x; w < NW; w += blockDim.x) dst[w] = src[w];
    __threadfence_system();
    __syncthreads();  // every lane has read the sequence number and copied its words
    if (threadIdx.x == 0) c->pub_seq = k + 1;
}

__device__ __forceinline__ bool resumable(const Dev& d) {
    const Ctl* c = d.ctl;
    return c->max_nnum <= d.cap && (d.vnbr == nullptr || c->max_vnum <= d.vcap);
}


__device__ __forceinline__ int64_t particle_of_thread(int& tile) {
    tile = xcd_tile(blockIdx.x, gridDim.x);
    return (int64_t)tile * BLOCK + threadIdx.x;
}

// Per-block maxima of the two displacement arrays (the reference keeps the full
// arrays, particle.cu:1094-1100; only their maxima are ever read) and the rebuild
// request of Particle::checkFor{Cell,Verlet}ListUpdate (particle.cu:1141-1161):
// 3*max > threshold.  wr < 0: no request.
__device__ __forceinline__ void disp_epilogue(const Dev& d, const NbrParams& nb, int tile,
                                              double nd, double cd, int wr, long long st) {
    double bn = nd, bc = cd;
    block_max2(bn, bc);
    if (threadIdx.x == 0) {
        d.pmax_nd[tile] = bn;
        d.pmax_cd[tile] = bc;
        if (wr >= 0 && (nb.method == DPM_NBR_CELL || nb.method == DPM_NBR_VERLET)) {
            if (nb.method == DPM_NBR_CELL && 3.0 * bc > nb.cthr) d.ctl->cflag[wr] = st;
            if (3.0 * bn > nb.thr) d.ctl->flag[wr] = st;
        }
    }
}

// The rebuild decision of disp_epilogue without the block maxima: 3 max d^2 > thr holds
// exactly when 3 d^2 > thr holds for some particle (3x is monotone under rounding), so a
// wave ballot per test replaces the block reduction.  For the steps inside a chunk, whose
// maxima nothing reads; the partials are written at the end of the chunk.
__device__ __forceinline__ void disp_flags(const Dev& d, const NbrParams& nb, double nd,
                                           double cd, int wr, long long st) {
    if (nb.method != DPM_NBR_CELL && nb.method != DPM_NBR_VERLET) return;
    const bool cf = nb.method == DPM_NBR_CELL && 3.0 * cd > nb.cthr;
    const bool lf = 3.0 * nd > nb.thr;
    const uint64_t bc = __builtin_amdgcn_ballot_w64(cf);
    const uint64_t bl = __builtin_amdgcn_ballot_w64(lf);
    if ((threadIdx.x & (WAVE - 1)) == 0) {
        if (bc) d.ctl->cflag[wr] = st;
        if (bl) d.ctl->flag[wr] = st;
    }
}

__device__ __forceinline__ void disp_of(const Dev& d, int64_t i, double x, double y, double& nd,
                                        double& cd) {
    double2 ln = d.lref[i], lc = d.cref[i];
    double dxn = x - ln.x, dyn = y - ln.y;
    nd = dxn * dxn + dyn * dyn;
    double dxc = x - lc.x, dyc = y - lc.y;
    cd = dxc * dxc + dyc * dyc;
}

// The rebuild a step at (epoch, pos) must perform before its forces:
// 0 none, 1 list, 2 cells + list (the cell test is the reference's first,
// particle.cu:1141-1161), 3 the list of the last in-kernel rebuild again, from its
// stored build positions, with a larger capacity.  ovf holds the stamp of the step
// whose in-kernel rebuild overflowed; that step itself ignores it, so every block of
// a launch reaches the same decision.
__device__ __forceinline__ bool ovf_pending(const Ctl* c, long long st) {
    return c->ovf != 0 && c->ovf != st;
}

__device__ __forceinline__ int pending_rebuild(const Ctl* c, long long epoch, int pos) {
    long long st = stamp(epoch, pos);
    if (c->cflag[pos & 1] == st) return 2;
    bool list = c->flag[pos & 1] == st;
    if (ovf_pending(c, st)) return list ? 1 : 3;
    return list ? 1 : 0;
}

// kernelMixVelocitiesAndForces (src/particles/base/kernels.cu:91-112): per-particle FIRE
// mixing with the 1e-16 force-norm guard
__device__ __forceinline__ void mix_one(double2& v, double2 f, double alpha) {
    double fn = sqrt(f.x * f.x + f.y * f.y);
    double vn = sqrt(v.x * v.x + v.y * v.y);
    double mr = 0.0;
    if (fn > 1e-16) {
        mr = vn / fn * alpha;
    } else {
        v.x = 0.0;
        v.y = 0.0;
        mr = 0.0;
    }
    v.x = v.x * (1 - alpha) + f.x * mr;
    v.y = v.y * (1 - alpha) + f.y * mr;
}

__device__ __forceinline__ int cell_coord(double pos, double cs, int n) {
    // getPBCCellIndex, include/particles/base/kernels.cuh:285-301
    long long idx = (long long)floor(pos / cs);
    return (int)(idx >= 0 ? idx % n : (idx % n + n) % n);
}

// isWithinCutoffSquared, include/particles/base/kernels.cuh:249-260
__device__ __forceinline__ bool within(double ax, double ay, double bx, double by,
                                       const NbrParams& nb, double c2) {
    double dx = pbc(ax, bx, nb.Lx, nb.invLx, nb.halfLx, nb.fast);
    double dy = pbc(ay, by, nb.Ly, nb.invLy, nb.halfLy, nb.fast);
    return dx * dx + dy * dy < c2;
}

// The candidates of a particle in cell (cx, cy) of a grid of nx x ny >= 3 x 3 cells, for lanes
// that test them side by side: the list entries of the 3 x 3 cells around it, rows and cells of
// a row in ascending order, which are one run in each row of cells, or two where the row wraps.
// range(c0, c1, a, e) gives the entries [a, e) of cells c0 to c1.
struct CellRuns {
    int a[6], m[6], count;
    template <class Range>
    __device__ __forceinline__ void set(int cx, int cy, int nx, int ny, bool live, Range range) {
        count = 0;
#pragma unroll
        for (int r = 0; r < 3; ++r) {
            const int y = cy + r - 1 < 0 ? ny - 1 : (cy + r - 1 >= ny ? 0 : cy + r - 1);
            const int c = y * nx;
            int b, e, wb = 0, we = 0;
            range(c + max(cx - 1, 0), c + min(cx + 1, nx - 1), b, e);
            if (cx == 0 || cx == nx - 1) {
                const int w = c + (cx == 0 ? nx - 1 : 0);
                range(w, w, wb, we);
            }
            const bool swap = cx == 0;  // the cell across the boundary comes first
            a[2 * r] = swap ? wb : b;
            m[2 * r] = live ? (swap ? we - wb : e - b) : 0;
            a[2 * r + 1] = swap ? b : wb;
            m[2 * r + 1] = live ? (swap ? e - b : we - wb) : 0;
            count += m[2 * r] + m[2 * r + 1];
        }
    }
    __device__ __forceinline__ int entry(int t) const {  // the list entry of candidate t
        int u = a[0] + t, base = m[0];
#pragma unroll
        for (int r = 1; r < 6; ++r) {
            if (t >= base) u = a[r] + (t - base);
            base += m[r];
        }
        return u;
    }
};

// LDS writes of the wave's lanes before its lanes' later reads
__device__ __forceinline__ void wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// Fire::step's decision for the next iteration (src/integrator/fire.cu:14-33);
// RigidBumpy::getPowerFire adds sum(tau*w) (rigid_bumpy.cu:1181-1191; null for disks).  True
// when the loop has ended.
__device__ __forceinline__ bool fire_decide(FireCtl& F, double px, double py,
                                            const double* spin) {
    double power = px + py;
    if (spin) power = power + *spin;
    F.power = power;
    if (power > 0) {
        F.n_good++;
        F.n_bad = 0;
        if (F.n_good > 5) {
            F.dt = fmin(F.dt * 1.1, F.dt_max);
            F.alpha *= 0.99;
        }
        F.uphill = 0;
    } else {
        F.n_good = 0;
        F.n_bad++;
        if (F.n_bad > 10) {
            F.stopped = 1;
            F.step += 1;  // the stopped step counts as executed
            F.done = 1;
            return true;
        }
        F.dt = fmax(F.dt * 0.5, F.dt_min);
        F.alpha = F.alpha_init;
        F.uphill = 1;
    }
    return false;
}

// minimizeFire's prologue: records the first average energy
__device__ __forceinline__ bool fire_begin(FireCtl& F, double px, double py, double pe,
                                           double fm, const double* spin) {
    F.fmax_sq = fm;
    F.avg_pe = pe / F.dof;
    F.last_avg_pe = F.avg_pe;
    if (F.max_steps <= 0) {
        F.done = 1;
        return true;
    }
    return fire_decide(F, px, py, spin);
}

// The end of a step: minimizeFire's stop test (src/routines/minimization.cu:99-105), then the
// decision for the next step.  One thread calls these.
__device__ __forceinline__ bool fire_advance(FireCtl& F, double px, double py, double pe,
                                             double fm, const double* spin) {
    const double avg = pe / F.dof;
    F.fmax_sq = fm;
    F.avg_pe = avg;
    const double diff = fabs(avg / F.last_avg_pe - 1);
    F.last_avg_pe = avg;
    const bool fok = F.fmax_target_sq > 0.0 && fm < F.fmax_target_sq;
    F.step += 1;
    if (diff < F.avg_pe_diff_target || avg < F.avg_pe_target || fok) {
        F.converged = 1;
        F.done = 1;
        return true;
    }
    if (F.step >= F.max_steps) {
        F.done = 1;
        return true;
    }
    return fire_decide(F, px, py, spin);
}

// mix_one by the short square root and quotient sequences: the same bits, for squared norms in
// the range that they cover; other lanes take the general form.
__device__ __forceinline__ void mix_hot(double2& v, double2 f, double alpha) {
    const double f2 = f.x * f.x + f.y * f.y, v2 = v.x * v.x + v.y * v.y;
    if (f2 > 0x1p-100 && f2 < 0x1p500 && v2 > 0x1p-600 && v2 < 0x1p500) {  // (fn > 1e-16)
        const double fn = sqrt_rn_normal(f2), vn = sqrt_rn_normal(v2);
        const double mr = div_rn_normal(vn, fn) * alpha;
        v.x = v.x * (1 - alpha) + f.x * mr;
        v.y = v.y * (1 - alpha) + f.y * mr;
    } else {
        mix_one(v, f, alpha);
    }
}

// ---- host helpers (dpm_core.hip) ----
std::mutex& capture_mutex();
int dalloc_bytes(dpm_system* s, void** p, size_t bytes);
template <class T>
int dalloc(dpm_system* s, T** p, int64_t n) {
    void* q = nullptr;
    if (dalloc_bytes(s, &q, sizeof(T) * (size_t)std::max<int64_t>(n, 1))) return -1;
    *p = (T*)q;
    return 0;
}
void dfree(dpm_system* s, void* p);
int64_t pow2_at_least(int64_t m);
int check_launch();
int scopy(dpm_system* s, void* dst, const void* src, size_t bytes, hipMemcpyKind kind);
PairParams params_of(const dpm_system* s);
NbrParams nbr_params(const dpm_system* s);
int launch_chunk_sum(dpm_system* s, int what, double* out_dev);
int sum_to_host(dpm_system* s, int what, double* out);
int sums_to_host(dpm_system* s, const int* what, int n, double* out);
int field_get(dpm_system* s, char kind, int comp, const void* plain, void* host);
int field_set(dpm_system* s, char kind, int comp, double* plain, const double* host);
int max_to_host(dpm_system* s, int what, double* out);
int ensure_ell(dpm_system* s, int64_t cap);
int device_rebuild(dpm_system* s, int mode, int* kind_out);
int check_and_rebuild(dpm_system* s, int* kind_out);
int refresh_rmax(dpm_system* s);
void enqueue_list_build(dpm_system* s, int gated);
void reset_ctl(dpm_system* s, int config);
int ensure_cells(dpm_system* s, int64_t nc);
int update_verlet_grid(dpm_system* s);
int bumpy_check_ring(dpm_system* s);
void collect_timing(dpm_system* s);

// Brackets one launch with HIP events on the system stream when timing is on.
struct Timed {
    dpm_system* s;
    int cls;
    hipEvent_t a = nullptr, b = nullptr;
    Timed(dpm_system* s_, int cls_);
    ~Timed();
};

// ---- small disk systems (dpm_resident.hip) ----
// Loops of up to RESIDENT_MAX_* particles run in one workgroup, from RESIDENT_MIN_STEPS steps.
// Measured against the chunked loops, us a step of 1,000 (chunked, resident): NVE 4.5, 1.5 at
// 128 particles; 5.9, 3.4 at 1,000; 6.1, 5.1 at 1,500; 6.1, 6.3 at 2,040; FIRE 14, 3.4 at 128;
// 20, 7.2 at 1,000; 20, 14.4 at 2,040; NVE in runs of 16 steps 7.2, 5.0 at 1,000.  One CU's LDS
// and vector pipe bound it, where the chunked step is launch gaps.
constexpr int64_t RESIDENT_MAX_NVE = 1536, RESIDENT_MAX_FIRE = 2048;
// Systems that are expected to be dense (dpm_resident.hpp: a wide skin) sum full rows, which one CU
// takes long over: us a step with a skin of 1.0 (chunked, resident): NVE 6.1, 5.4 at 256
// particles, 6.4, 8.8 at 384, 7.3, 22 at 1,536; FIRE 14, 9.4 at 384, 14.5, 12 at 700, 15.3, 15.1
// at 1,000 (1.3: 15.5, 16.8), 15, 29 at 2,000.
constexpr int64_t RESIDENT_DENSE_NVE = 256, RESIDENT_DENSE_FIRE = 768;
constexpr int64_t RESIDENT_MIN_STEPS = 16;
bool resident_ok(const dpm_system* s, bool fire);
int resident_prepare(dpm_system* s);
int resident_nve(dpm_system* s, double dt, int64_t steps);
int resident_fire(dpm_system* s, int64_t steps);

// ---- rigid bumpy (dpm_bumpy.hip) ----
int bumpy_alloc(dpm_system* s);
bool bumpy_fused_lists(const dpm_system* s);
int bumpy_forces(dpm_system* s, int mode);
void bumpy_enqueue_vertex_build(dpm_system* s, int gated);
void bumpy_enqueue_vertex_reorder(dpm_system* s, int gated);
int bumpy_ensure_vcap(dpm_system* s, int64_t cap);
int bumpy_kick(dpm_system* s, double dt);
int bumpy_drift(dpm_system* s, double dt);
int bumpy_adam_update(dpm_system* s, double alpha, double b1, double b2, double omb1,
                      double omb2, double eps);
int bumpy_mix(dpm_system* s, double alpha);
int bumpy_stress(dpm_system* s);
int bumpy_contacts(dpm_system* s);
int bumpy_nve_step(dpm_system* s, double dt);
void bumpy_enqueue_nve_steps(dpm_system* s, double dt, int64_t c);
void bumpy_enqueue_nve_resume(dpm_system* s, double dt);
void bumpy_enqueue_fire_forces(dpm_system* s, int kick, int gate, int check_pos = -1);
void bumpy_enqueue_fire_step(dpm_system* s, int pos);
int bumpy_snapshot(dpm_system* s, bool save);
int bumpy_download(dpm_system* s, int field, void* data, int64_t count);
int bumpy_upload(dpm_system* s, int field, const void* data, int64_t count);

}  // namespace dpm
