// dpm_rigid.hpp -- per-particle and per-vertex rigid-body arithmetic shared by the
// single-system rigid bumpy kernels (dpm_bumpy.hip) and the batched engine
// (dpm_batch.hip), so that a rigid system carries the same bits on either path.
#pragma once
#include "dpm_kernels.hpp"
#include "dpm_trig.hpp"

namespace dpm {

// kernelMixRigidVelocitiesAndForces, rigid_bumpy/kernels.cu:89-121
__device__ __forceinline__ void rigid_mix_one(double2& v, double2 f, double& w, double t,
                                              double alpha) {
    double fn = sqrt(f.x * f.x + f.y * f.y);
    double vn = sqrt(v.x * v.x + v.y * v.y);
    double mr = 0.0;
    if (fn > 1e-16) {
        mr = vn / fn * alpha;
    } else {
        v.x = 0.0;
        v.y = 0.0;
    }
    double tn = fabs(t), wn = fabs(w), tmr = 0.0;
    if (tn > 1e-16) {
        tmr = wn / tn * alpha;
    } else {
        w = 0.0;
        tmr = 0.0;
    }
    v = make_double2(v.x * (1 - alpha) + f.x * mr, v.y * (1 - alpha) + f.y * mr);
    w = w * (1 - alpha) + t * tmr;
}

// kernelTranslateAndRotateVertices1 (rigid_bumpy/kernels.cu:152-201) for one vertex: the
// back-step rotation by dth0 about the old centre onto the back-stepped one (when
// uphill), then the rotation by dth about that centre onto the new one.  (s0, c0) and
// (s1, c1) are dpm_sincos of dth0 and dth.
__device__ __forceinline__ double2 bfire_vertex_one(double2 x, double2 old, double2 mid,
                                                    double2 now, double s0, double c0,
                                                    double s1, double c1, int uphill) {
    if (uphill) {
        double rx = x.x - old.x, ry = x.y - old.y;
        double rxr = rx * c0 - ry * s0;
        double ryr = rx * s0 + ry * c0;
        x = make_double2(mid.x + rxr, mid.y + ryr);
    }
    double rx = x.x - mid.x, ry = x.y - mid.y;
    double rxr = rx * c1 - ry * s1;
    double ryr = rx * s1 + ry * c1;
    return make_double2(now.x + rxr, now.y + ryr);
}

// Vertex k of a ring particle of centre c, radius r and angle a with nv vertices of
// radius rv (kernelInitializeVerticesOnParticles, rigid_bumpy/kernels.cu:1137-1162):
// on the circle of radius r - rv at angle k * 2 pi / nv + a.
__device__ __forceinline__ double2 ring_vertex(double2 c, double r, double a, int nv, double rv,
                                               int k) {
    double inc = 2 * M_PI / nv;
    double inner = r - rv;
    double va = k * inc + a;
    double sv, cv;
    dpm_sincos(va, &sv, &cv);
    return make_double2(c.x + inner * cv, c.y + inner * sv);
}

// The ring's reach: every vertex of q (radius r_q, vertex radius rv) lies at r_q - rv from its
// centre (to rounding of the rotations, far below the margin), so by the triangle inequality a
// vertex at squared distance d2 from the centre has none of them within vc when d2 >=
// (r_q - rv + vc)^2.  The tests keep a relative margin of 1e-6 and so only skip scans that would
// list nothing.

// The image index k of a minimum image, pbc(a, b) = d - L k with d = a - b, as pbc forms it (0
// when |d| < L/2 on the fast path, where pbc returns d itself).
__device__ __forceinline__ double image_index(double d, double L, double invL, double halfL,
                                              int fast) {
    if (fast) return fabs(d) < halfL ? 0.0 : round(d * invL);
    return round(d / L);
}

// The half box a system needs for the image of two centres whose rings can reach each other
// (their distance is at most two ring radii and vc) to serve every vertex of both: the distance
// of any two of those vertices stays below it.
__device__ __host__ inline double ring_shift_limit(double rmax, double rv, double vc) {
    return (3.0 * rmax - 3.0 * rv + vc) * (1.0 + 1e-6);
}

// The half box from which a ring's window can be taken around its centre's nearest image: a vertex of
// the ring within vc of a point lies on an image of the ring whose centre is within ring radius +
// vc of the point, and two such images are a box side apart.  In smaller boxes (one to three
// particles) another image than the nearest may be the one that reaches the point.
__device__ __host__ inline double ring_window_limit(double rmax, double rv, double vc) {
    return (rmax - rv + vc) * (1.0 + 1e-6);
}

// atan2(y, x) to 1.2e-5 (an odd polynomial on [0, 1], fitted to the least largest error)
__device__ __forceinline__ float atan2_coarse(float y, float x) {
    const float ax = fabsf(x), ay = fabsf(y), hi = fmaxf(ax, ay), lo = fminf(ax, ay);
    const float t = hi > 0.0f ? lo * __builtin_amdgcn_rcpf(hi) : 0.0f, q = t * t;
    float r = t * (0.99986631f + q * (-0.33030444f + q * (0.18015778f +
                  q * (-0.08515398f + q * 0.0208439f))));
    r = ay > ax ? 1.57079633f - r : r;
    r = x < 0.0f ? 3.14159265f - r : r;
    return y < 0.0f ? -r : r;
}

// A neighbouring particle q of a particle row, as the vertex rows need it: centre, the shift
// L k of the minimum image of v - x_q, the squared distance below which a vertex looks at its
// ring (min of the vertex-particle cutoff's square and the ring's reach), vertex 0 from
// the centre, and the window's half width.
//
// The window: which vertices of ring q (n of them, radius R, evenly spaced counterclockwise from
// vertex 0) can lie within vc of a point in the direction (dx, dy) from q's centre: at most
// asin(vc / R) away from that direction, wherever the point is.  Single precision decides only
// the window, which is 0.02 of a spacing and the angle's error wider than it has to be on
// either side (asin(x) < x + x^3/4 up to x = 0.6; the spacing's tolerance of 1e-6 and the
// rotations' rounding stay far below that).
struct RingEntry {
    double cx, cy, sx, sy, lim;
    float x0, y0;    // vertex 0 from the centre
    float per, half; // spacings per radian; the window's half width in spacings (-1: all)
    int first, n;    // vertex range
};

// The vertex rows of one particle (kernelUpdateVertexNeighborList, rigid_bumpy/kernels.cu:
// 870-922: for vertex v, over the particle row in order, the particles q whose centre lies
// within vp of v, then q's vertices in order within vc of v), for vertices on their rings (even:
// evenly spaced ones, in a box of ring_window_limit): a half-wave per particle, lane a0 + lane
// its vertex xv; the return value is the lane's row length, emit(pos, u) stores entry pos.  R: 32
// entries of LDS of the half-wave's own.
//   1. each lane loads one row entry and puts it into R if some vertex of the particle can
//      reach it (in row order);
//   2. every lane tests the entries (vp and the ring's reach) into a bit mask;
//   3. every lane walks its own mask and tests the window of q's vertices (3 or 4 of 20 to 28)
//      that can be within vc, or all of an uneven ring's, four loads at a time.
// SHIFT: the minimum image of x_p - x_q serves every vertex of both rings (ring_shift_limit):
// pbc(v, u) = (v - u) - L k with one k, the same bits.  It is formed once per row entry; a lane
// that formed it for every vertex and entry spent most of its instructions on it.
// Without it (boxes of a few diameters) every vertex is tested by its own image.
// What bounds it: the gathers of the row entries and of their rings' vertices (halving the vector
// instructions, by fields in LDS instead of cross-lane reads, took a build of 65,536 particles of
// 24 vertices from 82 us to 70).
template <bool SHIFT, class Box, class Entry, class Emit>
__device__ __forceinline__ int vertex_row(const Box& bx, const double4* P, const int* vst,
                                          const int* nvt, const double2* vpos, double rv,
                                          double vc, double vc2, double vp2, int lane, int hs,
                                          bool has, double2 xv, double4 cp, int nn, bool even,
                                          RingEntry* R, Entry entry, Emit emit) {
    constexpr int HALF = WAVE / 2;
    int cnt = 0;
    auto image = [&](double a, double b, double s, double L, double invL, double halfL) {
        if constexpr (SHIFT) return (a - b) - s;
        else return pbc(a, b, L, invL, halfL, bx.fast);
    };
    for (int k0 = 0; __builtin_amdgcn_ballot_w64(k0 < nn) != 0; k0 += HALF) {
        RingEntry e;
        bool near = false;
        if (k0 + lane < nn) {
            const int q = entry(k0 + lane);
            const double4 c = P[q];
            e.first = vst[q];
            e.n = nvt[q];
            e.cx = c.x;
            e.cy = c.y;
            e.sx = e.sy = 0.0;
            near = true;
            if constexpr (SHIFT) {  // both rings' radii and vc, with the margin
                e.sx = bx.Lx * image_index(cp.x - c.x, bx.Lx, bx.invLx, bx.halfLx, bx.fast);
                e.sy = bx.Ly * image_index(cp.y - c.y, bx.Ly, bx.invLy, bx.halfLy, bx.fast);
                const double ex = (cp.x - c.x) - e.sx, ey = (cp.y - c.y) - e.sy;
                const double reach = (cp.z - rv) + (c.z - rv) + vc;
                near = ex * ex + ey * ey < reach * reach * (1.0 + 1e-6);
            }
            if (near) {
                const double2 u = vpos[e.first];
                const double reach = c.z - rv + vc;
                e.lim = fmin(vp2, reach * reach * (1.0 + 1e-6));
                e.x0 = (float)(u.x - c.x);
                e.y0 = (float)(u.y - c.y);
                e.per = (float)e.n * 0.15915494f;
                const float x = (float)vc / (float)(c.z - rv);
                e.half = (x + 0.25f * x * x * x) * e.per + 0.02f + 2e-5f * e.per;
                if (!even || !(x < 0.6f && 2.0f * e.half + 2.0f < (float)e.n)) e.half = -1.0f;
            }
        }
        const unsigned nm = (unsigned)(__builtin_amdgcn_ballot_w64(near) >> hs);
        if (near) R[__popc(nm & ((1u << lane) - 1u))] = e;
        wave_sync();
        const int entries = __popc(nm);
        unsigned gm = 0;
        for (int k = 0; k < entries; ++k) {
            const double dx = image(xv.x, R[k].cx, R[k].sx, bx.Lx, bx.invLx, bx.halfLx);
            const double dy = image(xv.y, R[k].cy, R[k].sy, bx.Ly, bx.invLy, bx.halfLy);
            if (has && dx * dx + dy * dy < R[k].lim) gm |= 1u << k;
        }
        while (gm != 0) {
            const RingEntry& q = R[__builtin_ctz(gm)];
            gm &= gm - 1;
            const double sx = q.sx, sy = q.sy;
            int lo = 0, count = q.n, first = q.first, n = q.n;
            if (q.half >= 0.0f) {
                const float dx = (float)image(xv.x, q.cx, sx, bx.Lx, bx.invLx, bx.halfLx);
                const float dy = (float)image(xv.y, q.cy, sy, bx.Ly, bx.invLy, bx.halfLy);
                const float t = q.per * atan2_coarse(q.x0 * dy - q.y0 * dx,
                                                     q.x0 * dx + q.y0 * dy);
                lo = (int)ceilf(t - q.half);
                count = (int)floorf(t + q.half) - lo + 1;
                if (lo < 0) lo += n;
            }
            // the candidates in ascending order: those beyond the ring's last vertex first
            const int wrapped = max(0, lo + count - n);
            constexpr int LOADS = 4;
            for (int c0 = 0; c0 < count; c0 += LOADS) {
                int u[LOADS];
                double2 xu[LOADS];
#pragma unroll
                for (int t = 0; t < LOADS; ++t) {
                    const int c = min(c0 + t, count - 1);
                    u[t] = first + (c < wrapped ? c : lo + c - wrapped);
                    xu[t] = vpos[u[t]];
                }
#pragma unroll
                for (int t = 0; t < LOADS; ++t) {
                    const double ex = image(xv.x, xu[t].x, sx, bx.Lx, bx.invLx, bx.halfLx);
                    const double ey = image(xv.y, xu[t].y, sy, bx.Ly, bx.invLy, bx.halfLy);
                    if (c0 + t < count && ex * ex + ey * ey < vc2) emit(cnt++, u[t]);
                }
            }
        }
        wave_sync();  // the next entries take these ones' place
    }
    return cnt;
}

// The Fire::step moves of one rigid particle (src/integrator/fire.cu:20-40 with the
// rigid overrides, rigid_bumpy/kernels.cu:21-150): [uphill: updatePositions(-dt/2) with
// the decreased dt, zero v and omega] + updateVelocities(dt/2) + mix + updatePositions(dt).
// q, v, a, w are updated in place; old / mid are the centre before and after the
// back-step, dth0 / dth the two rotation angles.
__device__ __forceinline__ void rigid_fire_move(double4& q, double2& v, double& a, double& w,
                                                double2 f, double t, double moi, double dt,
                                                double alpha, int uphill, int rotation,
                                                double2& old, double2& mid, double& dth0,
                                                double& dth) {
    old = make_double2(q.x, q.y);
    dth0 = 0.0;
    if (uphill) {
        double bdt = -dt / 2.0;
        double ddx = v.x * bdt, ddy = v.y * bdt;
        dth0 = w * bdt;
        q.x = q.x + ddx;
        q.y = q.y + ddy;
        a = a + dth0;
        v = make_double2(0.0, 0.0);
        w = 0.0;
    }
    mid = make_double2(q.x, q.y);
    // updateVelocities(dt/2) (kernelUpdateRigidVelocities)
    double hdt = dt / 2.0;
    if (rotation) w += t * hdt / moi;
    else w = 0.0;
    v.x += f.x * hdt / q.w;
    v.y += f.y * hdt / q.w;
    rigid_mix_one(v, f, w, t, alpha);
    // updatePositions(dt) (kernelUpdateRigidPositions)
    double ddx = v.x * dt, ddy = v.y * dt, dda = w * dt;
    dth = dda;
    q.x = q.x + ddx;
    q.y = q.y + ddy;
    a = a + dda;
}

}  // namespace dpm
