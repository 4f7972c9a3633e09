// dpm_resident.hpp -- a disk system of up to 4,096 particles held in one workgroup: positions,
// radii and (up to 2,048) the list of pairs in LDS, the rest of a particle's state in the
// registers of its thread.  Shared by the single-system loops (dpm_resident.hip) and the batched
// engine (dpm_batch_resident.hpp).
//
// Near pairs.  The full rows (every particle within the list cutoff, what queries and the other
// kernels read) go to the ELL in HBM; LDS holds the pairs that can touch before the list is next
// rebuilt.  Every step tests the displacements from the list's reference positions before it
// sums forces, so each particle is within delta = sqrt(thr / 3) of its reference, and a pair
// whose reference positions are further apart than r_i + r_j + 2 delta cannot touch: its term is
// +0.0 and leaves every sum as it is.  For half and half disks of 1 : 1.4 and a skin of 0.3 that
// drops a fifth of the entries.
//
// Each pair once.  A row walk evaluates a pair from both sides and pads every lane to its wave's
// longest row: some nine rounds of 60 double precision instructions, in one dependent chain
// each, for 2.6 pairs a particle.  Here the threads take the pairs one by one (any thread any
// pair) and leave the force on the lower particle and the energy in LDS; the force on the other
// particle is its exact negative (the minimum image and the contact radius are antisymmetric
// and symmetric to the bit).  Then each particle's thread adds its pairs in the order of its
// row, which gives the row walk's sums.
#pragma once
#include <cmath>

#include "dpm_kernels.hpp"

namespace dpm {

__device__ __forceinline__ double uniform_d(double v) {
    return __hiloint2double(__builtin_amdgcn_readfirstlane(__double2hiint(v)),
                            __builtin_amdgcn_readfirstlane(__double2loint(v)));
}

// The final stage of three chunk sums and a maximum (wave_final_sum), in part's rows 0 to 3:
// lanes 0, 16, 32 and 48 receive them.  Up to 16 partials take the last four stages only; more
// (up to 64) are halved first, lane t adding partial t + 32, then t + 16 (a sum that starts
// from 0.0 has no negative zero, so a missing partial's 0.0 changes nothing).
template <int NC>
__device__ __forceinline__ double res_final(const double (&part)[4][NC], int nc) {
    const int lane = threadIdx.x % WAVE, row = lane / 16, k = lane % 16;
    auto at = [&](int t) { return t < nc ? 0.0 + part[row][t] : 0.0; };
    double v = at(k);
    auto join = [&](double a, double b) { return row < 3 ? a + b : fmax(a, b); };
    if constexpr (NC > 32) v = join(join(v, at(k + 32)), join(at(k + 16), at(k + 48)));
    else if constexpr (NC > 16) v = join(v, at(k + 16));
    return rows_reduce(v);
}

// The thread's number, for the rare parts of a step loop (list builds): addresses formed from
// threadIdx.x there are loop invariants, and the compiler kept some hundred registers of them
// alive through the steps, which spilled.
__device__ __forceinline__ int res_tid() {
    int t = threadIdx.x;
    __asm__ __volatile__("" : "+v"(t));
    return t;
}

// Where the full rows are: entry k of slot i at nbr[k * stride + base + i], holding base + j
struct ResRows {
    int* nbr;
    long long stride, base;
    int cap;
};

// Rows of more than RES_LC near entries or more than 3 NP pairs (a mean of six near entries), and
// boxes too small for the branch-free minimum image, make a system "dense": its forces are then
// summed over the full rows.
constexpr int RES_LC = 16;

// What a system of n particles spread over its box is expected to have (host): the near entries of
// a large particle and the pairs, from the mean density.  A cluster in a large box has more.
// Counted on half and half disks of 1 : 1.4 at phi 0.70 to 0.90, skins of 0.3 to 1.0, relaxed:
// 0.80 to 1.04 of the pairs (above 0.95 only at the narrow end, where every class has room), and
// rows of up to 13 where 10.7 entries are expected, 16 where 12.0 are (longer ones in motion).
constexpr double RES_ROW = 11.0, RES_PAIR_SHARE = 0.93;
struct ResLoad {
    double row, pairs;
    ResLoad(double n, double area, double rmin, double rmax, double thr) {
        const double rho = n / area * 3.141592653589793, mid = 0.5 * (rmin + rmax);
        const double delta2 = 2.0 * std::sqrt(std::max(thr, 0.0) / 3.0);
        row = rho * (rmax + mid + delta2) * (rmax + mid + delta2);
        pairs = RES_PAIR_SHARE * 0.5 * n * rho * (2.0 * mid + delta2) * (2.0 * mid + delta2);
    }
};
constexpr unsigned short RES_FLIP = 0x8000;  // the particle is its pair's upper one

// How a system of NP particles is held by T threads
enum ResForm {
    RES_SMALL,  // a particle a thread: pairs and their results in LDS
    RES_BIG,    // two: LDS holds the build arrays, the pairs' forces or their energies at a time
                // (the energies follow in the forces' place once those are summed); after a build
                // a thread keeps its pairs in registers and the rows lie in HBM (read in order)
    RES_WALK    // four: LDS holds positions and radii, the near rows lie in HBM and are walked
                // from both sides
};

// What a list build works on
template <int NP, int COLS, bool PAIRS>
struct ResBuild {
    unsigned short row[RES_LC][COLS]; // near row: particles, then pair numbers (RES_FLIP), 3 NP
                                      // past its end
    int cend[NP];                     // end of each cell's list
    unsigned short lst[NP];           // the cells' lists
    unsigned short first[PAIRS ? NP : 1];  // the particle's first pair (as the lower one)
    unsigned pij[PAIRS ? 3 * NP : 1];      // lower particle | upper particle << 16
};

// Build arrays and the pairs' results (force on the lower particle, half pair energy; the last
// entry stays zero)
template <int T, int NP, ResForm FORM>
struct ResPairs {
    ResBuild<NP, NP, true> b;
    double2 f[3 * NP + 1];
    double e[3 * NP + 1];
};
template <int T, int NP>
struct ResPairs<T, NP, RES_BIG> {
    union {
        ResBuild<NP, NP, true> b;
        double2 f[3 * NP + 1];
        double e[3 * NP + 1];
    };
};
template <int T, int NP>
struct ResPairs<T, NP, RES_WALK> {
    ResBuild<NP, T, false> b;
};

// T threads, NP particles at most (PPT a thread: tid, tid + T, ...), a cell grid of at most NP
// cells
template <int T_, int NP_>
struct ResCore {
    static constexpr int T = T_, NP = NP_, MP = 3 * NP, PPT = NP > T ? NP / T : 1;
    static constexpr ResForm FORM = PPT == 1 ? RES_SMALL : (PPT == 2 ? RES_BIG : RES_WALK);
    static constexpr bool BIG = PPT > 1;
    static constexpr int PAIRS = (MP + T - 1) / T;  // a thread's pairs
    static_assert(FORM == RES_WALK || MP < RES_FLIP, "15-bit pair numbers");
    double2 x[NP];
    ResPairs<T, NP, FORM> p;
    double r[NP];
    int wsum[T / WAVE];
    int pairs, dense;
    // the column of particle i in p.b.row
    static __device__ __forceinline__ int col(int i) { return FORM == RES_WALK ? i % T : i; }
};

// A thread's pairs and the rows' place in HBM (not RES_SMALL; NP entries a column)
template <int T, int NP>
struct ResKept {
    unsigned ij[ResCore<T, NP>::FORM == RES_BIG ? ResCore<T, NP>::PAIRS : 1];
    unsigned short* row;
};

// Exclusive prefix sum of v over the workgroup's threads; total receives the sum.  Two barriers.
template <int T, int NP>
__device__ __forceinline__ int res_scan(ResCore<T, NP>& L, int v, int& total) {
    const int tid = res_tid(), lane = tid % WAVE, wv = tid / WAVE;
    int incl = v;
#pragma unroll
    for (int d = 1; d < WAVE; d <<= 1) {
        const int o = __shfl_up(incl, d, WAVE);
        if (lane >= d) incl += o;
    }
    __syncthreads();
    if (lane == WAVE - 1) L.wsum[wv] = incl;
    __syncthreads();
    int run = incl - v;
    total = 0;
#pragma unroll
    for (int k = 0; k < T / WAVE; ++k) {
        if (k == wv) run += total;
        total += L.wsum[k];
    }
    return run;
}

// Counting sort of the n particles into ncell <= NP cells, each list in ascending index: the
// lists in b.lst, their ends in b.cend.  mine: the cells of the thread's particles.
template <int T, int NP>
__device__ __forceinline__ void res_sort(ResCore<T, NP>& L, int n, int ncell,
                                         const int (&mine)[ResCore<T, NP>::PPT]) {
    constexpr int PPT = ResCore<T, NP>::PPT;
    auto& B = L.p.b;
    const int tid = res_tid();
    for (int c = tid; c < ncell; c += T) B.cend[c] = 0;
    __syncthreads();
#pragma unroll
    for (int m = 0; m < PPT; ++m)
        if (tid + m * T < n) atomicAdd(&B.cend[mine[m]], 1);
    __syncthreads();
    // each thread owns a run of consecutive cells
    const int per = (ncell + T - 1) / T;
    const int c0 = min(tid * per, ncell), c1 = min(c0 + per, ncell);
    int local = 0, total;
    for (int c = c0; c < c1; ++c) local += B.cend[c];
    int run = res_scan(L, local, total);
    for (int c = c0; c < c1; ++c) {
        const int t = B.cend[c];
        B.cend[c] = run;
        run += t;
    }
    __syncthreads();
#pragma unroll
    for (int m = 0; m < PPT; ++m) {
        const int i = tid + m * T;
        if (i < n) B.lst[atomicAdd(&B.cend[mine[m]], 1)] = (unsigned short)i;
    }
    __syncthreads();
    for (int c = tid; c < ncell; c += T) {  // ascending members (a few per cell)
        const int a = c == 0 ? 0 : B.cend[c - 1], e = B.cend[c];
        for (int u = a + 1; u < e; ++u) {
            const unsigned short v = B.lst[u];
            int k = u - 1;
            while (k >= a && B.lst[k] > v) {
                B.lst[k + 1] = B.lst[k];
                --k;
            }
            B.lst[k + 1] = v;
        }
    }
    __syncthreads();
}

// 2 delta: how much nearer two particles can come before 3 d^2 > thr asks for a rebuild (an
// undefined threshold never does: every listed pair is near)
__device__ __forceinline__ double res_reach(double thr) {
    return 2.0 * sqrt((thr < 0.0 ? 0.0 : thr) / 3.0);
}

// Whether a pair listed at reference positions a, b can touch before the next rebuild.  The
// bound is widened by the rounding of the coordinates; a NaN keeps the entry.  (a, b) and (b, a)
// have the same answer to the bit: near rows are symmetric where the full rows are.
__device__ __forceinline__ bool res_near(double2 a, double2 b, double rs, double delta2,
                                         const PairParams& p) {
    const double dx = pbc_rint(a.x, b.x, p.Lx, p.invLx);
    const double dy = pbc_rint(a.y, b.y, p.Ly, p.invLy);
    const double size = (fabs(a.x) + fabs(a.y)) + (fabs(b.x) + fabs(b.y));
    const double lim = (rs + delta2) * (1.0 + 1e-9) + 1e-14 * size;
    return !(dx * dx + dy * dy > lim * lim);
}

__device__ __forceinline__ bool res_listed(double2 a, double2 b, double rc2,
                                           const PairParams& p) {
    double dx, dy;
    if (p.fast) {
        dx = pbc_rint(a.x, b.x, p.Lx, p.invLx);
        dy = pbc_rint(a.y, b.y, p.Ly, p.invLy);
    } else {
        dx = pbc(a.x, b.x, p.Lx, p.invLx, p.halfLx, 0);
        dy = pbc(a.y, b.y, p.Ly, p.invLy, p.halfLy, 0);
    }
    return dx * dx + dy * dy < rc2;
}

// The runs of list entries in the 3 x 3 cells around (cx, cy), lower row first: the cells of
// a row are neighbours in b.lst, except where it wraps.  visit(a, b) takes entries [a, b).
template <int T, int NP, class Visit>
__device__ __forceinline__ void res_stencil(const ResCore<T, NP>& L, int cx, int cy, int nx,
                                            int ny, Visit visit) {
    const int* cend = L.p.b.cend;
    auto start = [&](int c) { return c == 0 ? 0 : cend[c - 1]; };
    const bool wraps = cx == 0 || cx == nx - 1;
    // (one copy of visit: unrolled, the build took the registers of the step loop around it)
#pragma unroll 1
    for (int t = 0; t < 6; ++t) {  // two parts a row; the second is empty without a wrap
        const int oy = t / 2 - 1;
        const int y = cy + oy < 0 ? cy + oy + ny : (cy + oy >= ny ? cy + oy - ny : cy + oy);
        const bool far = wraps && (t % 2 == 0) == (cx == 0);  // the part across the boundary
        if (t % 2 == 1 && !wraps) continue;
        const int c0 = y * nx + (far ? (cx == 0 ? nx - 1 : 0) : max(cx - 1, 0));
        const int c1 = y * nx + (far ? (cx == 0 ? nx - 1 : 0) : min(cx + 1, nx - 1));
        visit(start(c0), cend[c1]);
    }
}

// The row of particle i under the cell method (stencil_build's order; the particles are in cell
// order, so list entry j is particle j): the full row in HBM, the near row's particles in b.row.
// Returns the full length; near receives the near row's.
template <int T, int NP>
__device__ __forceinline__ int res_row_cell(ResCore<T, NP>& L, const ResRows& R, int i, int cell,
                                            int nc, double rc2, double delta2,
                                            const PairParams& p, int& near) {
    const double2 xi = L.x[i];
    const double ri = L.r[i];
    int cnt = 0, nr = 0;
    res_stencil(L, cell % nc, cell / nc, nc, nc, [&](int a, int b) {
#pragma unroll 1
        for (int j = a; j < b; ++j) {
            const double2 xj = L.x[j];
            if (j == i || !res_listed(xi, xj, rc2, p)) continue;
            if (cnt < R.cap) R.nbr[(long long)cnt * R.stride + R.base + i] = (int)(R.base + j);
            cnt++;
            if (!res_near(xi, xj, ri + L.r[j], delta2, p)) continue;
            if (nr < RES_LC) L.p.b.row[nr][L.col(i)] = (unsigned short)j;
            nr++;
        }
    });
    near = nr;
    return cnt;
}

// The same under the Verlet method: the particles within the cutoff in ascending index, from
// the lists of a cell grid (cells at least the cutoff wide) or, without one, from all pairs.
// Hits are kept sorted in b.row; a row that does not fit there is found by increasing index,
// one pass over the candidates an entry.
template <int T, int NP>
__device__ __forceinline__ int res_row_verlet(ResCore<T, NP>& L, const ResRows& R, int i, int n,
                                              bool grid, int cx, int cy, int nx, int ny,
                                              double rc2, double delta2, const PairParams& p,
                                              int& near) {
    const double2 xi = L.x[i];
    const double ri = L.r[i];
    auto& row = L.p.b.row;
    const unsigned short* lst = L.p.b.lst;
    const int at = L.col(i);
    int cnt = 0, nr = 0;
    auto put = [&](int k, int j) {
        if (k < R.cap) R.nbr[(long long)k * R.stride + R.base + i] = (int)(R.base + j);
    };
    if (!grid) {
#pragma unroll 1
        for (int j = 0; j < n; ++j) {
            const double2 xj = L.x[j];
            if (j == i || !res_listed(xi, xj, rc2, p)) continue;
            put(cnt++, j);
            if (!res_near(xi, xj, ri + L.r[j], delta2, p)) continue;
            if (nr < RES_LC) row[nr][at] = (unsigned short)j;
            nr++;
        }
        near = nr;
        return cnt;
    }
    res_stencil(L, cx, cy, nx, ny, [&](int a, int b) {
#pragma unroll 1
        for (int u = a; u < b; ++u) {
            const int j = lst[u];
            if (j == i || !res_listed(xi, L.x[j], rc2, p)) continue;
            if (cnt < RES_LC) {
                int k = cnt;
                for (; k > 0 && row[k - 1][at] > j; --k) row[k][at] = row[k - 1][at];
                row[k][at] = (unsigned short)j;
            }
            cnt++;
        }
    });
    if (cnt <= RES_LC) {
#pragma unroll 1
        for (int k = 0; k < cnt; ++k) {
            const int j = row[k][at];
            put(k, j);
            if (res_near(xi, L.x[j], ri + L.r[j], delta2, p)) row[nr++][at] = (unsigned short)j;
        }
    } else {
        nr = cnt;  // dense: the forces walk the full rows
#pragma unroll 1
        for (int k = 0, last = -1; k < cnt; ++k) {
            int next = n;
            res_stencil(L, cx, cy, nx, ny, [&](int a, int b) {
#pragma unroll 1
                for (int u = a; u < b; ++u) {
                    const int j = lst[u];
                    if (j > last && j < next && j != i && res_listed(xi, L.x[j], rc2, p)) next = j;
                }
            });
            put(k, next);
            last = next;
        }
    }
    near = nr;
    return cnt;
}

// The near row of a list that was built before (reference positions ref[base + j]), in the
// present box.
template <int T, int NP>
__device__ __forceinline__ int res_load_row(ResCore<T, NP>& L, const ResRows& R,
                                            const double2* ref, int i, int full, double delta2,
                                            const PairParams& p) {
    const double2 xi = ref[R.base + i];
    const double ri = L.r[i];
    const int nn = min(full, R.cap);
    int near = 0;
#pragma unroll 1
    for (int k = 0; k < nn; ++k) {
        const int j = (int)(R.nbr[(long long)k * R.stride + R.base + i] - R.base);
        if (!res_near(xi, ref[R.base + j], ri + L.r[j], delta2, p)) continue;
        if (near < RES_LC) L.p.b.row[near][L.col(i)] = (unsigned short)j;
        near++;
    }
    return near;
}

// RES_WALK: particle i's near row out of b.row, which the thread's next particle takes
template <int T, int NP>
__device__ __forceinline__ void res_keep_row(const ResCore<T, NP>& L, const ResKept<T, NP>& K,
                                             int i, int near) {
    if constexpr (ResCore<T, NP>::FORM == RES_WALK) {
        for (int k = 0; k < min(near, RES_LC); ++k) K.row[k * NP + i] = L.p.b.row[k][L.col(i)];
    }
}

// The pairs of the near rows (particle numbers in b.row; near[m]: their lengths, 0 without a
// particle): numbered by lower particle, then in its row's order; b.row receives the pair
// numbers (BIG: K, which outlives the build arrays).  len[m]: the lengths of the force sums.
// Ends with a barrier.
template <int T, int NP>
__device__ __forceinline__ void res_pairs(ResCore<T, NP>& L, ResKept<T, NP>& K, int n, bool fast,
                                          const int (&near)[ResCore<T, NP>::PPT],
                                          int (&len)[ResCore<T, NP>::PPT]) {
    constexpr int PPT = ResCore<T, NP>::PPT, MP = ResCore<T, NP>::MP;
    auto& B = L.p.b;
    const int tid = res_tid();
    if (tid == 0) L.dense = fast ? 0 : 1;
    if constexpr (ResCore<T, NP>::FORM == RES_WALK) {
        __syncthreads();
#pragma unroll
        for (int m = 0; m < PPT; ++m) {
            len[m] = min(near[m], RES_LC);
            if (near[m] > RES_LC) L.dense = 1;
        }
        __syncthreads();
        return;
    }
    int total = 0, first[PPT];
#pragma unroll
    for (int m = 0; m < PPT; ++m) {
        const int i = tid + m * T, nr = min(near[m], RES_LC);
        int own = 0, sum;
#pragma unroll 1
        for (int k = 0; k < nr; ++k) own += (int)B.row[k][i] > i ? 1 : 0;
        first[m] = total + res_scan(L, own, sum);  // (its barriers order the write above)
        total += sum;
        len[m] = nr;
    }
    bool over = total > MP;
#pragma unroll
    for (int m = 0; m < PPT; ++m) {
        const int i = tid + m * T;
        over = over || near[m] > RES_LC;
        if (i >= n) continue;
        B.first[i] = (unsigned short)min(first[m], MP);
#pragma unroll 1
        for (int k = 0, s = first[m]; k < len[m]; ++k) {
            const int j = B.row[k][i];
            if (j > i && s < MP) B.pij[s++] = (unsigned)i | (unsigned)j << 16;
        }
    }
    if (over) L.dense = 1;
    if (tid == 0) L.pairs = min(total, MP);
    __syncthreads();
    if (!L.dense) {
#pragma unroll
        for (int m = 0; m < PPT; ++m) {
            const int i = tid + m * T;
            if (i >= NP) continue;
#pragma unroll 1
            for (int k = 0, s = first[m]; k < len[m]; ++k) {
                const int j = B.row[k][i];
                unsigned short e;
                if (j > i) {
                    e = (unsigned short)s++;
                } else {  // listed by j, whose pairs are consecutive
                    int t = B.first[j];
                    while (t < L.pairs && (int)(B.pij[t] >> 16) != i) ++t;
                    if (t == L.pairs) L.dense = 1;  // (rows that are not symmetric)
                    e = (unsigned short)t | RES_FLIP;
                }
                B.row[k][i] = e;
            }
            for (int k = len[m]; k < RES_LC; ++k) B.row[k][i] = (unsigned short)MP;
        }
    }
    if constexpr (ResCore<T, NP>::FORM == RES_BIG) {
#pragma unroll
        for (int k = 0; k < ResCore<T, NP>::PAIRS; ++k) {
            const int t = tid + k * T;
            K.ij[k] = t < MP ? B.pij[t] : 0u;
        }
#pragma unroll
        for (int m = 0; m < PPT; ++m)
            for (int k = 0; k < RES_LC; ++k)
                K.row[k * NP + tid + m * T] = B.row[k][tid + m * T];
    }
    __syncthreads();
}

// v with its sign flipped where the entry is the pair's upper particle
__device__ __forceinline__ double res_flip(double v, unsigned e) {
    const unsigned s = (e & RES_FLIP) << 16;
    return __hiloint2double((int)((unsigned)__double2hiint(v) ^ s), __double2loint(v));
}

// RES_WALK: the near rows in row order, the wave to its longest row, two entries at a time with
// the next two loaded ahead (entries past a row's end are any particle and add +0.0).  No
// barrier: the positions must rest until every thread is through.
template <bool ENERGY, int T, int NP>
__device__ __forceinline__ void res_walk(const ResCore<T, NP>& L, const ResKept<T, NP>& K,
                                         const PairParams& p, int nc,
                                         const int (&len)[ResCore<T, NP>::PPT],
                                         double (&ax)[ResCore<T, NP>::PPT],
                                         double (&ay)[ResCore<T, NP>::PPT],
                                         double (&e)[ResCore<T, NP>::PPT]) {
#pragma unroll
    for (int m = 0; m < ResCore<T, NP>::PPT; ++m) {
        ax[m] = ay[m] = e[m] = 0.0;
        const int i = threadIdx.x + m * T, nn = len[m];
        if (i / WAVE >= nc) continue;  // uniform over the wave
        const double4 qi = make_double4(L.x[i].x, L.x[i].y, L.r[i], 0.0);
        auto entry = [&](int k) { return k < nn ? (int)K.row[k * NP + i] : 0; };
        int j0 = entry(0), j1 = entry(1);
#pragma unroll 1
        for (int k = 0; __builtin_amdgcn_ballot_w64(k < nn) != 0; k += 2) {
            const double4 q0 = make_double4(L.x[j0].x, L.x[j0].y, L.r[j0], 0.0);
            const double4 q1 = make_double4(L.x[j1].x, L.x[j1].y, L.r[j1], 0.0);
            j0 = entry(k + 2);
            j1 = entry(k + 3);
            double fx, fy;
            double w = pair_hot<ENERGY>(qi, q0, k < nn, p, fx, fy);
            ax[m] += fx;
            ay[m] += fy;
            if (ENERGY) e[m] += w;
            if (__builtin_amdgcn_ballot_w64(k + 1 < nn) == 0) break;
            w = pair_hot<ENERGY>(qi, q1, k + 1 < nn, p, fx, fy);
            ax[m] += fx;
            ay[m] += fy;
            if (ENERGY) e[m] += w;
        }
        __builtin_amdgcn_sched_barrier(0);
    }
}

// Forces (and energies) of the thread's particles: every pair once, then the sums over the rows
// of len[m] pairs in row order (the wave walks its longest row, four entries at a time; entries
// past the end are the zero pair).  Every position has been written behind a barrier; no thread
// reads a position or writes a pair's result after the last barrier in here (RES_WALK: has none).
template <bool ENERGY, int T, int NP>
__device__ __forceinline__ void res_forces(ResCore<T, NP>& L, const ResKept<T, NP>& K,
                                           const PairParams& p, int nc,
                                           const int (&len)[ResCore<T, NP>::PPT],
                                           double (&ax)[ResCore<T, NP>::PPT],
                                           double (&ay)[ResCore<T, NP>::PPT],
                                           double (&e)[ResCore<T, NP>::PPT]) {
    using C = ResCore<T, NP>;
    constexpr int PPT = C::PPT, MP = C::MP;
    if constexpr (C::FORM == RES_WALK) {
        res_walk<ENERGY>(L, K, p, nc, len, ax, ay, e);
        return;
    } else {
    const int tid = threadIdx.x, np = L.pairs;
    double keep[(C::FORM == RES_BIG) ? C::PAIRS : 1];
    auto pair = [&](int t, unsigned ij) {
        const int i = (int)(ij & 0xffff), j = (int)(ij >> 16);
        const double2 a = L.x[i], b = L.x[j];
        double fx, fy;
        const double w = pair_hot<ENERGY>(make_double4(a.x, a.y, L.r[i], 0.0),
                                          make_double4(b.x, b.y, L.r[j], 0.0), true, p, fx, fy);
        L.p.f[t] = make_double2(fx, fy);
        return w;
    };
    if constexpr ((C::FORM == RES_BIG)) {
#pragma unroll
        for (int k = 0; k < C::PAIRS; ++k) {
            const int t = tid + k * T;
            keep[k] = 0.0;
            if (t < np) keep[k] = pair(t, K.ij[k]);
            if (k % 2 == 1) __builtin_amdgcn_sched_barrier(0);  // (six at once spill)
        }
    } else {
        for (int t = tid; t < np; t += T) {
            const double w = pair(t, L.p.b.pij[t]);
            if (ENERGY) L.p.e[t] = w;
        }
    }
    if (tid == 0) {
        L.p.f[MP] = make_double2(0.0, 0.0);
        if (ENERGY && !(C::FORM == RES_BIG)) L.p.e[MP] = 0.0;
    }
    __syncthreads();
    auto entry = [&](int k, int i) -> unsigned {
        if constexpr ((C::FORM == RES_BIG)) return K.row[k * NP + i];
        else return L.p.b.row[k][i];
    };
#pragma unroll
    for (int m = 0; m < PPT; ++m) {
        ax[m] = ay[m] = e[m] = 0.0;
        const int i = tid + m * T;
        if (i / WAVE >= nc) continue;  // uniform over the wave
#pragma unroll 1
        for (int k = 0; __builtin_amdgcn_ballot_w64(k < len[m]) != 0; k += 4) {
            unsigned s[4];
            double2 f[4];
            double w[4];
#pragma unroll
            for (int t = 0; t < 4; ++t) s[t] = entry(k + t, i);
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                f[t] = L.p.f[s[t] & (RES_FLIP - 1)];
                if (ENERGY && !(C::FORM == RES_BIG)) w[t] = L.p.e[s[t] & (RES_FLIP - 1)];
            }
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                ax[m] += res_flip(f[t].x, s[t]);
                ay[m] += res_flip(f[t].y, s[t]);
                if (ENERGY && !(C::FORM == RES_BIG)) e[m] += w[t];
            }
        }
    }
    if constexpr (ENERGY && (C::FORM == RES_BIG)) {
        __syncthreads();
#pragma unroll
        for (int k = 0; k < C::PAIRS; ++k)
            if (tid + k * T < np) L.p.e[tid + k * T] = keep[k];
        if (tid == 0) L.p.e[MP] = 0.0;
        __syncthreads();
#pragma unroll
        for (int m = 0; m < PPT; ++m) {
            const int i = tid + m * T;
            if (i / WAVE >= nc) continue;
            for (int k = 0; __builtin_amdgcn_ballot_w64(k < len[m]) != 0; k += 4) {
                unsigned s[4];
#pragma unroll
                for (int t = 0; t < 4; ++t) s[t] = entry(k + t, i);
#pragma unroll
                for (int t = 0; t < 4; ++t) e[m] += L.p.e[s[t] & (RES_FLIP - 1)];
            }
        }
    }
    }
}

// The same over the full row in HBM, pair by pair (dense systems).  No barrier: the positions
// must rest until every thread is through.
template <int T, int NP>
__device__ __forceinline__ void res_sum_full(const ResCore<T, NP>& L, const ResRows& R,
                                             const PairParams& p, int i, int full, double& ax,
                                             double& ay, double& e) {
    const double4 qi = make_double4(L.x[i].x, L.x[i].y, L.r[i], 0.0);
    ax = 0.0;
    ay = 0.0;
    e = 0.0;
#pragma unroll 1
    for (int k = 0; k < min(full, R.cap); ++k) {
        const int j = (int)(R.nbr[(long long)k * R.stride + R.base + i] - R.base);
        const double4 qj = make_double4(L.x[j].x, L.x[j].y, L.r[j], 0.0);
        double fx, fy;
        const double ie = p.fast ? pair_hot<true>(qi, qj, true, p, fx, fy)
                                 : pair_hot<true, true>(qi, qj, true, p, fx, fy);
        ax += fx;
        ay += fy;
        e += ie;
    }
}

}  // namespace dpm
