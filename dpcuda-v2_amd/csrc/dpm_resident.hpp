// dpm_resident.hpp -- a disk system of up to 1,024 particles held in one workgroup: positions,
// radii and the list of pairs in LDS, the rest of a particle's state in the registers of its
// thread.  Included by dpm_resident.hip.
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
#include "dpm_kernels.hpp"

namespace dpm {

__device__ __forceinline__ double uniform_d(double v) {
    return __hiloint2double(__builtin_amdgcn_readfirstlane(__double2hiint(v)),
                            __builtin_amdgcn_readfirstlane(__double2loint(v)));
}

// Where the full rows are: entry k of slot i at nbr[k * stride + base + i], holding base + j
struct ResRows {
    int* nbr;
    long long stride, base;
    int cap;
};

// T threads, NP <= T particles at most, a cell grid of at most NP cells.  Rows of more than
// RES_LC near entries or more than MP pairs (a mean of six near entries) make the system
// "dense": its forces are then summed over the full rows.
constexpr int RES_LC = 16;
constexpr unsigned short RES_FLIP = 0x8000;  // the particle is its pair's upper one

template <int T, int NP_>
struct ResCore {
    static constexpr int NP = NP_, MP = 3 * NP_;
    static_assert(NP <= T && MP < RES_FLIP, "a thread per particle, 15-bit pair numbers");
    double2 x[NP];
    double2 pf[MP + 1];  // force on the pair's lower particle; the last one stays zero
    double pe[MP + 1];   // half pair energy
    double r[NP];
    unsigned pij[MP];                 // lower particle | upper particle << 16
    unsigned short row[RES_LC][NP];   // near row: pair number (RES_FLIP), MP past its end
    unsigned short first[NP];         // the particle's first pair (as the lower one)
    int cend[NP];                     // end of each cell's list
    unsigned short lst[NP];           // the cells' lists
    int wsum[T / WAVE];
    int pairs, dense;
};

// Exclusive prefix sum of v over the workgroup's threads; total receives the sum.  Two barriers.
template <int T, int NP>
__device__ __forceinline__ int res_scan(ResCore<T, NP>& L, int v, int& total) {
    const int lane = threadIdx.x % WAVE, wv = threadIdx.x / WAVE;
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
// lists in L.lst, their ends in L.cend.  mine: the cell of the thread's particle.
template <int T, int NP>
__device__ __forceinline__ void res_sort(ResCore<T, NP>& L, int n, int ncell, int mine) {
    const int tid = threadIdx.x;
    if (tid < ncell) L.cend[tid] = 0;
    __syncthreads();
    if (tid < n) atomicAdd(&L.cend[mine], 1);
    __syncthreads();
    int total;
    const int run = res_scan(L, tid < ncell ? L.cend[tid] : 0, total);
    if (tid < ncell) L.cend[tid] = run;
    __syncthreads();
    if (tid < n) L.lst[atomicAdd(&L.cend[mine], 1)] = (unsigned short)tid;
    __syncthreads();
    if (tid < ncell) {  // ascending members (a few per cell)
        const int a = tid == 0 ? 0 : L.cend[tid - 1], e = L.cend[tid];
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
    const double dx = pbc_rint(a.x, b.x, p.Lx, p.invLx);
    const double dy = pbc_rint(a.y, b.y, p.Ly, p.invLy);
    return dx * dx + dy * dy < rc2;
}

// The three runs of particles in the 3 x 3 cells around (cx, cy), lower row first: the cells of
// a row are neighbours in L.lst, except where it wraps.  visit(a, b) takes list entries [a, b).
template <int T, int NP, class Visit>
__device__ __forceinline__ void res_stencil(const ResCore<T, NP>& L, int cx, int cy, int nx,
                                            int ny, Visit visit) {
    auto start = [&](int c) { return c == 0 ? 0 : L.cend[c - 1]; };
    for (int oy = -1; oy <= 1; ++oy) {
        const int y = cy + oy < 0 ? cy + oy + ny : (cy + oy >= ny ? cy + oy - ny : cy + oy);
        const int c = y * nx;
        if (cx == 0) visit(start(c + nx - 1), L.cend[c + nx - 1]);
        visit(start(c + max(cx - 1, 0)), L.cend[c + min(cx + 1, nx - 1)]);
        if (cx == nx - 1) visit(start(c), L.cend[c]);
    }
}

// The row of the thread's particle under the cell method (stencil_build's order; the particles
// are in cell order, so list entry j is particle j): the full row in HBM, the near row's
// particles in L.row.  Returns the full length; near receives the near row's.
template <int T, int NP>
__device__ __forceinline__ int res_row_cell(ResCore<T, NP>& L, const ResRows& R, int i, int cell,
                                            int nc, double rc2, double delta2,
                                            const PairParams& p, int& near) {
    const double2 xi = L.x[i];
    const double ri = L.r[i];
    int cnt = 0, nr = 0;
    res_stencil(L, cell % nc, cell / nc, nc, nc, [&](int a, int b) {
        for (int j = a; j < b; ++j) {
            const double2 xj = L.x[j];
            if (j == i || !res_listed(xi, xj, rc2, p)) continue;
            if (cnt < R.cap) R.nbr[(long long)cnt * R.stride + R.base + i] = (int)(R.base + j);
            cnt++;
            if (!res_near(xi, xj, ri + L.r[j], delta2, p)) continue;
            if (nr < RES_LC) L.row[nr][i] = (unsigned short)j;
            nr++;
        }
    });
    near = nr;
    return cnt;
}

// The same under the Verlet method: the particles within the cutoff in ascending index, from
// the lists of a cell grid (cells at least the cutoff wide) or, without one, from all pairs.
// Hits are kept sorted in L.row; a row that does not fit there is found by increasing index,
// one pass over the candidates an entry.
template <int T, int NP>
__device__ __forceinline__ int res_row_verlet(ResCore<T, NP>& L, const ResRows& R, int i, int n,
                                              bool grid, int cx, int cy, int nx, int ny,
                                              double rc2, double delta2, const PairParams& p,
                                              int& near) {
    const double2 xi = L.x[i];
    const double ri = L.r[i];
    int cnt = 0, nr = 0;
    auto put = [&](int k, int j) {
        if (k < R.cap) R.nbr[(long long)k * R.stride + R.base + i] = (int)(R.base + j);
    };
    if (!grid) {
        for (int j = 0; j < n; ++j) {
            const double2 xj = L.x[j];
            if (j == i || !res_listed(xi, xj, rc2, p)) continue;
            put(cnt++, j);
            if (!res_near(xi, xj, ri + L.r[j], delta2, p)) continue;
            if (nr < RES_LC) L.row[nr][i] = (unsigned short)j;
            nr++;
        }
        near = nr;
        return cnt;
    }
    res_stencil(L, cx, cy, nx, ny, [&](int a, int b) {
        for (int u = a; u < b; ++u) {
            const int j = L.lst[u];
            if (j == i || !res_listed(xi, L.x[j], rc2, p)) continue;
            if (cnt < RES_LC) {
                int k = cnt;
                for (; k > 0 && L.row[k - 1][i] > j; --k) L.row[k][i] = L.row[k - 1][i];
                L.row[k][i] = (unsigned short)j;
            }
            cnt++;
        }
    });
    if (cnt <= RES_LC) {
        for (int k = 0; k < cnt; ++k) {
            const int j = L.row[k][i];
            put(k, j);
            if (res_near(xi, L.x[j], ri + L.r[j], delta2, p)) L.row[nr++][i] = (unsigned short)j;
        }
    } else {
        nr = cnt;  // dense: the forces walk the full rows
        for (int k = 0, last = -1; k < cnt; ++k) {
            int next = n;
            res_stencil(L, cx, cy, nx, ny, [&](int a, int b) {
                for (int u = a; u < b; ++u) {
                    const int j = L.lst[u];
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

// The near row of a list that an earlier launch built (reference positions ref[base + j]).
template <int T, int NP>
__device__ __forceinline__ int res_load_row(ResCore<T, NP>& L, const ResRows& R,
                                            const double2* ref, int i, int full, double delta2,
                                            const PairParams& p) {
    const double2 xi = ref[R.base + i];
    const double ri = L.r[i];
    const int nn = min(full, R.cap);
    int near = 0;
    for (int k = 0; k < nn; ++k) {
        const int j = (int)(R.nbr[(long long)k * R.stride + R.base + i] - R.base);
        if (!res_near(xi, ref[R.base + j], ri + L.r[j], delta2, p)) continue;
        if (near < RES_LC) L.row[near][i] = (unsigned short)j;
        near++;
    }
    return near;
}

// The pairs of the near rows (particle numbers in L.row, `near` of the thread's particle; 0
// without one): numbered by lower particle, then in its row's order; L.row receives the pair
// numbers.  Returns the length of the force sum's row.  Ends with a barrier.
template <int T, int NP>
__device__ __forceinline__ int res_pairs(ResCore<T, NP>& L, int n, int near) {
    const int i = threadIdx.x;
    const int nr = min(near, RES_LC);
    int own = 0;
    for (int k = 0; k < nr; ++k) own += (int)L.row[k][i] > i ? 1 : 0;
    if (i == 0) L.dense = 0;
    int total;
    const int first = res_scan(L, own, total);  // (its barriers order the write above)
    if (near > RES_LC || total > L.MP) L.dense = 1;
    if (i < n) L.first[i] = (unsigned short)min(first, L.MP);
    if (i == 0) {
        L.pairs = min(total, L.MP);
        L.pf[L.MP] = make_double2(0.0, 0.0);
        L.pe[L.MP] = 0.0;
    }
    for (int k = 0, s = first; k < nr; ++k) {
        const int j = L.row[k][i];
        if (j > i && s < L.MP) L.pij[s++] = (unsigned)i | (unsigned)j << 16;
    }
    __syncthreads();
    if (i < n && !L.dense) {
        for (int k = 0, s = first; k < nr; ++k) {
            const int j = L.row[k][i];
            unsigned short e;
            if (j > i) {
                e = (unsigned short)s++;
            } else {  // listed by j, whose pairs are consecutive
                int t = L.first[j];
                while (t < L.pairs && (int)(L.pij[t] >> 16) != i) ++t;
                if (t == L.pairs) L.dense = 1;  // (rows that are not symmetric)
                e = (unsigned short)t | RES_FLIP;
            }
            L.row[k][i] = e;
        }
        for (int k = nr; k < RES_LC; ++k) L.row[k][i] = (unsigned short)L.MP;
    }
    __syncthreads();
    return nr;
}

// Every pair's force and energy (no barrier at either end)
template <bool ENERGY, int T, int NP>
__device__ __forceinline__ void res_pair_forces(ResCore<T, NP>& L, const PairParams& p) {
    const int np = L.pairs;
    for (int t = threadIdx.x; t < np; t += T) {
        const unsigned ij = L.pij[t];
        const int i = (int)(ij & 0xffff), j = (int)(ij >> 16);
        const double2 a = L.x[i], b = L.x[j];
        double fx, fy;
        const double e = pair_hot<ENERGY>(make_double4(a.x, a.y, L.r[i], 0.0),
                                          make_double4(b.x, b.y, L.r[j], 0.0), true, p, fx, fy);
        L.pf[t] = make_double2(fx, fy);
        if (ENERGY) L.pe[t] = e;
    }
}

// v with its sign flipped where the entry is the pair's upper particle
__device__ __forceinline__ double res_flip(double v, unsigned e) {
    const unsigned s = (e & RES_FLIP) << 16;
    return __hiloint2double((int)((unsigned)__double2hiint(v) ^ s), __double2loint(v));
}

// The sums of the thread's particle over its row of nn pairs, in row order; the wave walks its
// longest row, four entries at a time (entries past the end are the zero pair)
template <bool ENERGY, int T, int NP>
__device__ __forceinline__ void res_sum(const ResCore<T, NP>& L, int i, int nn, double& ax,
                                        double& ay, double& e) {
    ax = 0.0;
    ay = 0.0;
    e = 0.0;
    for (int k = 0; __builtin_amdgcn_ballot_w64(k < nn) != 0; k += 4) {
        unsigned s[4];
        double2 f[4];
        double w[4];
#pragma unroll
        for (int t = 0; t < 4; ++t) s[t] = L.row[k + t][i];
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            f[t] = L.pf[s[t] & (RES_FLIP - 1)];
            if (ENERGY) w[t] = L.pe[s[t] & (RES_FLIP - 1)];
        }
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            ax += res_flip(f[t].x, s[t]);
            ay += res_flip(f[t].y, s[t]);
            if (ENERGY) e += w[t];
        }
    }
}

// The same over the full row in HBM, pair by pair (dense systems)
template <int T, int NP>
__device__ __forceinline__ void res_sum_full(const ResCore<T, NP>& L, const ResRows& R,
                                             const PairParams& p, int i, int full, double& ax,
                                             double& ay, double& e) {
    const double4 qi = make_double4(L.x[i].x, L.x[i].y, L.r[i], 0.0);
    ax = 0.0;
    ay = 0.0;
    e = 0.0;
    for (int k = 0; k < min(full, R.cap); ++k) {
        const int j = (int)(R.nbr[(long long)k * R.stride + R.base + i] - R.base);
        double fx, fy;
        const double ie = pair_hot<true>(qi, make_double4(L.x[j].x, L.x[j].y, L.r[j], 0.0), true,
                                         p, fx, fy);
        ax += fx;
        ay += fy;
        e += ie;
    }
}

}  // namespace dpm
