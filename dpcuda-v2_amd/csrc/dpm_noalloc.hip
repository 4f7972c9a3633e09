// dpm_noalloc.hip -- disk forces, energies and the total potential energy of caller-owned
// device arrays, with no device allocation: the working memory (cell grid, particle lists,
// reduction partials) is the file-scope array `scratch`, resident on every device the
// library runs on until the process ends.
//
// What it computes is what a disk system with the Verlet method (cutoff rc) returns from
// dpm_neighbor_init + dpm_zero_forces + dpm_compute_forces + dpm_reduce(DPM_RED_PE):
// Disk::calculateForces (src/particles/disk/disk.cu:218-221) over the rows of
// kernelUpdateNeighborList (src/particles/base/kernels.cu:256-293, all pairs within rc in
// ascending j), then totalPotentialEnergy (src/particles/base/particle.cu:1078-1080) in the
// library's canonical summation order.  The pairs come from a cell grid (cells at least rc
// wide; each particle's hits are ranked by index), so the order of a particle's sum, and every
// result bit, equal the list-based path.
#include <mutex>
#include <type_traits>

#include "dpm_kernels.hpp"

namespace dpm {

// the rebuild kernels of dpm_core.hip that the grid reuses (counting sort of the cells)
__global__ void k_scan_a(Dev d, long long nc, int gated);
__global__ void k_scan_b(Dev d, long long nb_blocks, int gated);
__global__ void k_scan_c(Dev d, long long nc, int gated);

// ---- scratch layout -----------------------------------------------------------------------
constexpr int64_t NA_MAX_N = 1 << 20;      // particles per call
constexpr int64_t NA_MAX_CELLS = 1 << 20;  // grid cells
constexpr int64_t NA_MAX_ALL_PAIRS = 4096; // particles of a box too small for a grid
constexpr int64_t NA_SCAN_TILE = 1024;     // cells per scan block (k_scan_a/c)
constexpr int64_t NA_MAX_SB = NA_MAX_CELLS / NA_SCAN_TILE + 1;
constexpr size_t na_align(size_t b) { return (b + 255) / 256 * 256; }
constexpr size_t NA_OFF_CNT = 0;
constexpr size_t NA_OFF_START = NA_OFF_CNT + na_align(sizeof(int) * NA_MAX_CELLS);
constexpr size_t NA_OFF_CUR = NA_OFF_START + na_align(sizeof(int) * (NA_MAX_CELLS + 1));
constexpr size_t NA_OFF_BSUM = NA_OFF_CUR + na_align(sizeof(int) * NA_MAX_CELLS);
constexpr size_t NA_OFF_CELL = NA_OFF_BSUM + na_align(sizeof(int) * (NA_MAX_SB + 1));
constexpr size_t NA_OFF_REC = NA_OFF_CELL + na_align(sizeof(int) * NA_MAX_N);
constexpr size_t NA_OFF_PART = NA_OFF_REC + na_align(sizeof(double4) * NA_MAX_N);
constexpr size_t NA_SCRATCH_BYTES = NA_OFF_PART + na_align(sizeof(double) * (NA_MAX_N / 64 + 1));
// 48.1 MiB per device

static __device__ __align__(256) unsigned char scratch[NA_SCRATCH_BYTES];

// The device address of `scratch` on each device, looked up once per device (the name is a
// host-side stand-in: only this address may be handed to kernels or copies).
constexpr int NA_MAX_DEVICES = 64;
static void* g_scratch[NA_MAX_DEVICES];
static std::mutex g_scratch_mu;

static int scratch_of_current_device(unsigned char** out) {
    int dev = 0;
    DPM_HIP(hipGetDevice(&dev));
    if (dev < 0 || dev >= NA_MAX_DEVICES) {
        set_error("dpm_disk_forces_noalloc: device index out of range");
        return -1;
    }
    std::lock_guard<std::mutex> g(g_scratch_mu);
    if (!g_scratch[dev]) {
        void* p = nullptr;
        DPM_HIP(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
        if (!p) {
            set_error("dpm_disk_forces_noalloc: no device address for the scratch array");
            return -1;
        }
        g_scratch[dev] = p;
    }
    *out = (unsigned char*)g_scratch[dev];
    return 0;
}

// ---- kernels --------------------------------------------------------------------------------
struct NaGrid {
    int ncx, ncy;    // cells per side (1 x 1: every particle is a candidate of every other)
    double csx, csy; // cell sides
};

__global__ void k_na_fill(int* a, int64_t n) {
    int64_t i = (int64_t)blockIdx.x * BLOCK + threadIdx.x;
    if (i < n) a[i] = 0;
}

__device__ __forceinline__ int na_coord(double pos, double cs, int n) {
    // getPBCCellIndex, include/particles/base/kernels.cuh:285-301
    long long idx = (long long)floor(pos / cs);
    long long m = idx % n;
    return (int)(m < 0 ? m + n : m);
}

// (non-finite positions go to cell 0)
__device__ __forceinline__ int na_cell(double x, double y, const NaGrid& g) {
    if (!(isfinite(x) && isfinite(y) && fabs(x) < 1e15 * g.csx && fabs(y) < 1e15 * g.csy)) return 0;
    return na_coord(x, g.csx, g.ncx) + g.ncx * na_coord(y, g.csy, g.ncy);
}

// cell of each particle + counting-sort histogram
__global__ void k_na_bin(const double* x, const double* y, int64_t n, NaGrid g, int* cell,
                         int* cnt) {
    int64_t i = (int64_t)blockIdx.x * BLOCK + threadIdx.x;
    if (i >= n) return;
    const int c = na_cell(x[i], y[i], g);
    cell[i] = c;
    atomicAdd(&cnt[c], 1);
}

// The particles in cell order (in no order within a cell): one record each, {x, y, radius, index}
__global__ void k_na_scatter(const double* x, const double* y, const double* rad, int64_t n,
                             const int* cell, int* cur, double4* rec) {
    const int64_t i = (int64_t)blockIdx.x * BLOCK + threadIdx.x;
    if (i >= n) return;
    const double4 q = make_double4(x[i], y[i], rad[i], (double)i);
    rec[atomicAdd(&cur[cell[i]], 1)] = q;
}

// Up to NA_LDS_N particles every workgroup forms the whole cell grid in its own LDS, and the call
// is two launches; beyond, the particles are sorted into records by cell over six launches, so
// that candidates are neighbours in memory.  Measured, us a call (in LDS, sorted): 26, 31 at
// 8,192 particles; 42, 34 at 16,400.
constexpr int NA_LDS_N = 8192;
constexpr int NA_LDS_CELLS = 8192;

constexpr int NA_T = 1024;            // threads: 16 lanes for each of a chunk's particles
constexpr int NA_GROUP = NA_T / CHUNK;
constexpr int NA_HITS = 32;           // pairs of a particle that LDS holds

struct NaForces {
    double2 f[CHUNK][NA_HITS];  // pair forces and energies in the order of the particle's sum
    double e[CHUNK][NA_HITS];
    int hit[CHUNK][NA_HITS];    // partners as they are found, by place
    int key[CHUNK][NA_HITS];    // and their indices
    double pe[CHUNK];
    int wsum[NA_T / WAVE];
};

struct NaGridLds {
    int cend[NA_LDS_CELLS];         // end of each cell's list
    unsigned short lst[NA_LDS_N];   // the lists, in no order within a cell
};

struct NaNone {};

// The counting sort of all particles into the grid's cells, by one workgroup.
__device__ __forceinline__ void na_lds_grid(NaGridLds& G, NaForces& L, const double* x,
                                            const double* y, int n, const NaGrid& g) {
    const int tid = threadIdx.x, lane = tid % WAVE, wv = tid / WAVE, ncell = g.ncx * g.ncy;
    for (int c = tid; c < ncell; c += NA_T) G.cend[c] = 0;
    __syncthreads();
    for (int i = tid; i < n; i += NA_T) atomicAdd(&G.cend[na_cell(x[i], y[i], g)], 1);
    __syncthreads();
    // exclusive scan of the counts: each thread owns a run of consecutive cells
    const int per = (ncell + NA_T - 1) / NA_T;
    const int c0 = min(tid * per, ncell), c1 = min(c0 + per, ncell);
    int local = 0;
    for (int c = c0; c < c1; ++c) local += G.cend[c];
    int incl = local;
#pragma unroll
    for (int s = 1; s < WAVE; s <<= 1) {
        const int o = __shfl_up(incl, s, WAVE);
        if (lane >= s) incl += o;
    }
    if (lane == WAVE - 1) L.wsum[wv] = incl;
    __syncthreads();
    int run = incl - local;
    for (int k = 0; k < wv; ++k) run += L.wsum[k];
    for (int c = c0; c < c1; ++c) {
        const int t = G.cend[c];
        G.cend[c] = run;
        run += t;
    }
    __syncthreads();
    for (int i = tid; i < n; i += NA_T)
        G.lst[atomicAdd(&G.cend[na_cell(x[i], y[i], g)], 1)] = (unsigned short)i;
    __syncthreads();
}

// The total of nc partials in wave_final_sum's order (lane t adds partials t, t + 64, ...): all
// threads bring a stretch of them to LDS, one wave adds it.
constexpr int NA_STRETCH = 4096;

__global__ __launch_bounds__(NA_T) void k_na_total(const double* part, int64_t nc,
                                                   double* total) {
    __shared__ double stretch[NA_STRETCH];
    const int tid = threadIdx.x;
    double s = 0.0;
    for (int64_t base = 0; base < nc; base += NA_STRETCH) {
        const int len = (int)min((int64_t)NA_STRETCH, nc - base);
        __syncthreads();
        for (int k = tid; k < len; k += NA_T) stretch[k] = part[base + k];
        __syncthreads();
        if (tid < WAVE)
            for (int k = tid; k < len; k += WAVE) s = s + stretch[k];
    }
    if (tid >= WAVE) return;
    s = wave_tree_sum(s);
    if (tid == 0) *total = s;
}

// Forces and energies: a workgroup per 64 particles, 16 lanes a particle.  The lanes test the
// candidates of the nine cells side by side, append the hits, rank them by index and evaluate
// one pair each; three lanes then add the components in rank order (the ascending order of the
// Verlet rows).  A serial walk that merged the nine lists in order spent some 60 instructions
// and a dependent load on each of 27 candidates.
// A particle with more hits than LDS holds takes them by windows of the index, each found by all
// lanes again: 2,000 particles at a cutoff of 3.5 (some 30 to 45 pairs) 43 us a call, 2,077 when
// three lanes looked for one pair at a time, 211 by the serial walk; 4,000 particles in a cluster
// (up to 160 pairs) 330, 33,500 and 1,460 us.
// LDS: the grid is the workgroup's own, the particles are the caller's arrays in their order, and
// the workgroup is a chunk of the energy sum.  Otherwise `rec` holds the particles in cell order
// and `start` the cells' first records: reading the caller's arrays at random costs a cache line
// for each coordinate of each candidate (1,010 us at 1,048,576 particles).
// What bounds it: at a thousand particles the host's launches, at a million the records' scatter
// and the candidates.  Measured, us a call (before, now): 1,500 particles 70, 13; 16,400 75, 34;
// 1,048,576 1,013, 537.
template <bool LDS>
__global__ __launch_bounds__(NA_T) void k_na_forces(const double* x, const double* y,
                                                    const double* rad, int64_t n, NaGrid g,
                                                    PairParams p, double rc2, const int* start,
                                                    const double4* rec, double* fx, double* fy,
                                                    double* pe, double* part) {
    __shared__ NaForces L;
    __shared__ typename std::conditional<LDS, NaGridLds, NaNone>::type G;
    const int tid = threadIdx.x, lane = tid % WAVE, sub = lane % NA_GROUP, k = tid / NA_GROUP;
    if constexpr (LDS) na_lds_grid(G, L, x, y, (int)n, g);
    // a particle's place: its index, or its record's
    const int tile = LDS ? (int)blockIdx.x : xcd_tile(blockIdx.x, gridDim.x);
    const int64_t me = (int64_t)tile * CHUNK + k;
    const bool live = me < n;
    auto load = [&](int64_t u) {
        if constexpr (LDS) return make_double4(x[u], y[u], rad[u], 0.0);
        else return rec[u];
    };
    auto key_of = [&](int u, const double4& q) {
        if constexpr (LDS) return u;
        else return (int)q.w;
    };
    const double4 q = load(live ? me : 0);
    // the runs of list entries in the three rows of cells: one each, two where a row wraps
    auto range = [&](int c0, int c1, int& a, int& b) {
        if constexpr (LDS) {
            a = c0 == 0 ? 0 : G.cend[c0 - 1];
            b = G.cend[c1];
        } else {
            a = start[c0];
            b = start[c1 + 1];
        }
    };
    const int cid = na_cell(q.x, q.y, g);
    CellRuns runs;
    runs.set(cid % g.ncx, cid / g.ncx, g.ncx, g.ncy, live, range);
    const int cand = runs.count;
    auto candidate = [&](int t) {  // the place of candidate t
        if constexpr (LDS) return (int)G.lst[runs.entry(t)];
        else return runs.entry(t);
    };
    auto listed = [&](const double4& o) {
        const double dx = pbc(q.x, o.x, p.Lx, p.invLx, p.halfLx, 1);
        const double dy = pbc(q.y, o.y, p.Ly, p.invLy, p.halfLy, 1);
        return dx * dx + dy * dy < rc2;
    };
    const int shift = lane - sub;
    // the hits (with an index in [lo, lo + width)): as many as LDS holds, and their number
    auto collect = [&](auto window, int lo, int width) {
        int cnt = 0;
        for (int t = sub; __builtin_amdgcn_ballot_w64(t < cand) != 0; t += NA_GROUP) {
            int u = -1, key = 0;
            bool hit = false;
            if (t < cand) {
                u = candidate(t);
                const double4 o = load(u);
                key = key_of(u, o);
                hit = u != (int)me && listed(o);
                if constexpr (window.value) hit = hit && key >= lo && key - lo < width;
            }
            const unsigned mask =
                (unsigned)(__builtin_amdgcn_ballot_w64(hit) >> shift) & ((1u << NA_GROUP) - 1);
            const int pos = cnt + __popc(mask & ((1u << sub) - 1));
            if (hit && pos < NA_HITS) {
                L.hit[k][pos] = u;
                L.key[k][pos] = key;
            }
            cnt += __popc(mask);
        }
        wave_sync();
        return cnt;
    };
    auto pair = [&](int u, double& px, double& py) {
        const double4 o = load(u);
        const double rs = q.z + o.z;
        PairParams w = p;  // the short sequences, where they give the same bits
        w.fastdiv = p.fastdiv && rs >= 0x1p-99 && rs <= 0x1p99;
        return pair_law(q.x, q.y, q.z, o.x, o.y, o.z, w, px, py);
    };
    double acc = 0.0;
    auto add = [&](int cnt) {  // the hits in LDS, in ascending order
        for (int h = sub; h < cnt; h += NA_GROUP) {
            const int key = L.key[k][h];
            int rank = 0;
            for (int v = 0; v < cnt; ++v) rank += L.key[k][v] < key ? 1 : 0;
            double px, py;
            const double e = pair(L.hit[k][h], px, py);
            L.f[k][rank] = make_double2(px, py);
            L.e[k][rank] = e;
        }
        wave_sync();
        if (sub < 3) {
            for (int v = 0; v < cnt; ++v)
                acc += sub == 0 ? L.f[k][v].x : (sub == 1 ? L.f[k][v].y : L.e[k][v]);
        }
    };
    const int total = collect(std::false_type{}, 0, 0);
    if (total <= NA_HITS) {
        add(total);
    } else {  // by windows of the index that LDS holds
        int width = max(1, (int)(n * (NA_HITS * 2 / 3) / total));
        for (int lo = 0, done = 0; done < total && lo < n;) {
            const int cnt = collect(std::true_type{}, lo, width);
            if (cnt > NA_HITS) {
                width /= 2;
                continue;
            }
            add(cnt);
            wave_sync();  // the next window's take this one's place
            done += cnt;
            lo += width;
            if (cnt < NA_HITS / 2) width = min(2 * width, (int)n);
        }
    }
    acc = 0.0 + acc;
    const int i = key_of((int)me, q);
    if (live) {
        if (sub == 0) fx[i] = acc;
        if (sub == 1) fy[i] = acc;
        if (sub == 2) pe[i] = acc;
    }
    if constexpr (LDS) {  // the chunk's partial of the energy sum (k_chunk_sum's tree)
        if (sub == 2) L.pe[k] = live ? acc : 0.0;
        __syncthreads();
        if (tid >= WAVE) return;
        const double v = wave_tree_sum(L.pe[tid]);
        if (tid == 0) part[blockIdx.x] = v;
    }
}

// The chunk partials of the energy sum
__global__ __launch_bounds__(BLOCK) void k_na_chunks(const double* pe, int64_t n, double* part) {
    const int64_t i = (int64_t)blockIdx.x * BLOCK + threadIdx.x;
    const double v = wave_tree_sum(i < n ? pe[i] : 0.0);
    if (threadIdx.x % WAVE == 0 && i < n) part[i / CHUNK] = v;
}

// The same for a box under three cutoffs a side: every particle is a candidate, in ascending
// order; a thread per particle, a chunk per workgroup.
__global__ __launch_bounds__(CHUNK) void k_na_forces_all(const double* x, const double* y,
                                                         const double* rad, int64_t n,
                                                         PairParams p, double rc2, double* fx,
                                                         double* fy, double* pe, double* part) {
    const int64_t i = (int64_t)blockIdx.x * CHUNK + threadIdx.x;
    double e = 0.0;
    if (i < n) {
        const double xi = x[i], yi = y[i], ri = rad[i];
        double ax = 0.0, ay = 0.0;
        for (int64_t j = 0; j < n; ++j) {
            if (j == i) continue;
            const double dx = pbc(xi, x[j], p.Lx, p.invLx, p.halfLx, 0);
            const double dy = pbc(yi, y[j], p.Ly, p.invLy, p.halfLy, 0);
            if (dx * dx + dy * dy < rc2) {
                double px, py;
                const double ie = pair_law(xi, yi, ri, x[j], y[j], rad[j], p, px, py);
                ax += px;
                ay += py;
                e += ie;
            }
        }
        fx[i] = 0.0 + ax;
        fy[i] = 0.0 + ay;
        e = 0.0 + e;
        pe[i] = e;
    }
    const double v = wave_tree_sum(e);
    if (threadIdx.x == 0) part[blockIdx.x] = v;
}

}  // namespace dpm

using namespace dpm;

extern "C" {

int dpm_disk_forces_noalloc(const double* x, const double* y, const double* radius, int64_t n,
                            double lx, double ly, double e_c, double n_c, double cutoff,
                            double* fx, double* fy, double* pe, double* pe_total, void* stream) {
    if (n < 1 || n > NA_MAX_N) {
        set_error("dpm_disk_forces_noalloc: particle count must be in [1, 1048576] (the size "
                  "of the library's scratch array)");
        return -1;
    }
    if (!x || !y || !radius || !fx || !fy || !pe || !pe_total) {
        set_error("dpm_disk_forces_noalloc: null array");
        return -1;
    }
    if (!(lx > 0) || !(ly > 0) || !(cutoff > 0) || !(e_c > 0) || !(n_c > 0)) {
        set_error("dpm_disk_forces_noalloc: box sides, cutoff, e_c and n_c must be positive");
        return -1;
    }
    unsigned char* base = nullptr;
    if (scratch_of_current_device(&base)) return -1;
    hipStream_t st = (hipStream_t)stream;
    const bool lds = n <= NA_LDS_N;
    // the grid: cells at least cutoff (1 + 1e-9) wide, at most about two per particle and
    // what the cell arrays hold; under three a side, one cell holds every particle
    const double cw = cutoff * (1.0 + 1e-9);
    double fx_c = std::floor(lx / cw), fy_c = std::floor(ly / cw);
    const double cap = std::min<double>(lds ? (double)NA_LDS_CELLS : (double)NA_MAX_CELLS,
                                        std::max(9.0, 2.0 * (double)n));
    if (fx_c * fy_c > cap) {  // shrunk in proportion, then to the limit
        const double f = std::sqrt(fx_c * fy_c / cap);
        if (std::min(fx_c, fy_c) > 3.0 * f) {
            fx_c = std::floor(fx_c / f) + 1.0;
            fy_c = std::floor(fy_c / f) + 1.0;
        }
    }
    while (fx_c * fy_c > cap) {
        if (fx_c >= fy_c) fx_c -= 1.0;
        else fy_c -= 1.0;
    }
    NaGrid g{1, 1, lx, ly};
    if (fx_c >= 3 && fy_c >= 3) g = NaGrid{(int)fx_c, (int)fy_c, lx / fx_c, ly / fy_c};
    if (g.ncx == 1 && n > NA_MAX_ALL_PAIRS) {
        set_error("dpm_disk_forces_noalloc: a box under three cutoffs a side takes at most "
                  "4096 particles (every pair is tested)");
        return -1;
    }
    const int64_t nc = (int64_t)g.ncx * g.ncy;
    // carve the scratch array
    Dev d{};
    d.N = n;
    d.cell_cnt = (int*)(base + NA_OFF_CNT);
    d.cell_start = (int*)(base + NA_OFF_START);
    d.cell_cur = (int*)(base + NA_OFF_CUR);
    d.scan_bsum = (int*)(base + NA_OFF_BSUM);
    d.cell_tmp = (int*)(base + NA_OFF_CELL);
    double4* rec = (double4*)(base + NA_OFF_REC);
    double* part = (double*)(base + NA_OFF_PART);
    // the pair law's parameters (pair_params without a system)
    PairParams p{};
    p.Lx = lx;
    p.Ly = ly;
    p.invLx = 1.0 / lx;
    p.invLy = 1.0 / ly;
    p.halfLx = 0.5 * lx;
    p.halfLy = 0.5 * ly;
    p.e_c = e_c;
    p.n_c = n_c;
    p.ncm1 = n_c - 1.0;
    p.two_nc = 2.0 * n_c;
    int ex;
    p.inv2nc = (std::frexp(p.two_nc, &ex) == 0.5) ? 1.0 / p.two_nc : 0.0;
    p.fast = 0;
    p.fastdiv = n_c == 2.0 && e_c >= 0x1p-100 && e_c <= 0x1p100;  // (radii: the kernels)
    const int64_t nsb = (nc + NA_SCAN_TILE - 1) / NA_SCAN_TILE;
    const double rc2 = cutoff * cutoff;
    const dim3 chunks((unsigned)((n + CHUNK - 1) / CHUNK)), threads(NA_T);
    if (g.ncx == 1) {
        p.fastdiv = 0;
        hipLaunchKernelGGL(k_na_forces_all, chunks, dim3(CHUNK), 0, st, x, y, radius, n, p, rc2,
                           fx, fy, pe, part);
    } else if (lds) {
        p.fast = 1;  // half a side exceeds the cutoff, and only pairs within it count
        hipLaunchKernelGGL(k_na_forces<true>, chunks, threads, 0, st, x, y, radius, n, g, p, rc2,
                           nullptr, nullptr, fx, fy, pe, part);
    } else {  // counting sort into the cells (cells cleared by a kernel: no memset node, so a
              // captured graph replays correctly)
        p.fast = 1;
        hipLaunchKernelGGL(k_na_fill, pgrid(nc), dim3(BLOCK), 0, st, d.cell_cnt, nc);
        hipLaunchKernelGGL(k_na_bin, pgrid(n), dim3(BLOCK), 0, st, x, y, n, g, d.cell_tmp,
                           d.cell_cnt);
        hipLaunchKernelGGL(k_scan_a, dim3((unsigned)nsb), dim3(BLOCK), 0, st, d, (long long)nc, 0);
        hipLaunchKernelGGL(k_scan_b, dim3(1), dim3(1024), 0, st, d, (long long)nsb, 0);
        hipLaunchKernelGGL(k_scan_c, dim3((unsigned)nsb), dim3(BLOCK), 0, st, d, (long long)nc, 0);
        hipLaunchKernelGGL(k_na_scatter, pgrid(n), dim3(BLOCK), 0, st, x, y, radius, n,
                           d.cell_tmp, d.cell_cur, rec);
        hipLaunchKernelGGL(k_na_forces<false>, chunks, threads, 0, st, x, y, radius, n, g, p, rc2,
                           d.cell_start, rec, fx, fy, pe, part);
        hipLaunchKernelGGL(k_na_chunks, pgrid(n), dim3(BLOCK), 0, st, pe, n, part);
    }
    hipLaunchKernelGGL(k_na_total, dim3(1), threads, 0, st, part, (n + CHUNK - 1) / CHUNK,
                       pe_total);
    return check_launch();
}

}  // extern "C"
