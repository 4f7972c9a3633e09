// dpm_rigid.hpp -- per-particle and per-vertex rigid-body arithmetic shared by the
// single-system rigid bumpy kernels (dpm_bumpy.hip) and the batched engine
// (dpm_batch.hip), so that a rigid system carries the same bits on either path.
#pragma once
#include "dpm_device.hpp"
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

// Whether a vertex v at squared distance d2 from the centre of particle q (radius r_q,
// vertex radius rv) can have one of q's vertices within vc: every vertex of q lies at
// r_q - rv from its centre (to rounding of the rotations, far below the margin), so by
// the triangle inequality none can when d2 >= (r_q - rv + vc)^2; the test keeps a
// relative margin of 1e-6 and so only skips vertex scans that would list nothing.
__device__ __forceinline__ bool vertex_ring_near(double d2, double rq, double rv, double vc) {
    const double reach = rq - rv + vc;
    return d2 < reach * reach * (1.0 + 1e-6);
}

// Vertex rows through the centre's image.  For a vertex v and a particle q that passed
// vertex_ring_near, every vertex u of q lies within ring reach + (r_q - r_v) of v; when
// half the box exceeds that bound (vertex_shift_ok), the minimum image of v - u is the
// image of v - x_q: pbc(v, u) = (v - u) - L k with the same k.  image_index gives that k
// as pbc forms it (0 when |d| < L/2 on the fast path, where pbc returns d itself), and
// pbc_known applies it with pbc's own operations, so the bits are pbc's.
__device__ __forceinline__ double image_index(double d, double L, double invL, double halfL,
                                              int fast) {
    if (fast) return fabs(d) < halfL ? 0.0 : round(d * invL);
    return round(d / L);
}

__device__ __forceinline__ double pbc_known(double a, double b, double L, double k, int fast) {
    const double d = a - b;
    if (fast && k == 0.0) return d;
    return d - L * k;
}

// The half box a system needs for the image shortcut: ring reach plus ring radius of the
// largest particle (vertex_ring_near's relative margin included).
__device__ __host__ inline double vertex_shift_limit(double rmax, double rv, double vc) {
    return (2.0 * rmax - 2.0 * rv + vc) * (1.0 + 1e-6);
}

// Which vertices of ring q (nq of them, radius R, evenly spaced counterclockwise from vertex 0
// at r0 from the centre) can lie within vc of a point at (dx, dy) from q's centre: at most
// asin(vc / R) away from the point's direction, wherever the point is.  The candidates in
// ascending order are c < wrapped ? c : first + c - wrapped for c in [0, count).  Single
// precision decides only the window, which is 0.02 of a spacing wider than it has to be on
// either side (asin(x) < x + x^3/4 up to x = 0.6; the rounding of atan2f, the spacing's
// tolerance of 1e-6 and the rotations' rounding stay far below that).
struct RingWindow {
    int first, count, wrapped;
};
__device__ __forceinline__ RingWindow ring_window(double dx, double dy, double2 r0, double R,
                                                  double vc, int nq) {
    const float x = (float)vc / (float)R;
    const float per = (float)nq * 0.15915494f;  // spacings per radian
    const float half = x < 0.6f ? (x + 0.25f * x * x * x) * per + 0.02f : 1e9f;
    if (!(2.0f * half + 2.0f < (float)nq)) return {0, nq, 0};
    const float t = per * atan2f((float)(r0.x * dy - r0.y * dx), (float)(r0.x * dx + r0.y * dy));
    const int lo = (int)ceilf(t - half), hi = (int)floorf(t + half);
    const int first = lo < 0 ? lo + nq : lo;
    return {first, hi - lo + 1, max(0, first + (hi - lo + 1) - nq)};
}

// The vertex rows of one particle (kernelUpdateVertexNeighborList, rigid_bumpy/kernels.cu:
// 870-922: for vertex v, over the particle row in order, the particles q whose centre lies
// within vp of v, then q's vertices in order within vc of v), for evenly spaced rings: a
// half-wave per particle, lane a0 + lane its vertex xv; the return value is the lane's row
// length, emit(pos, u) stores entry pos.
//   1. each lane loads one row entry (q's record, vertex range and first vertex) and drops the
//      q that no vertex of the particle can reach;
//   2. every lane tests the remaining centres (vp and vertex_ring_near) into a bit mask;
//   3. every lane walks its own mask and tests the window of q's vertices (3 or 4 of 20 to 28)
//      that can be within vc.
// A vertex passes the gate of one or two of its particle's neighbours, so the wave takes two
// or three rounds of step 3.  Before, a gated vertex was tested against all of q's vertices by
// the 32 lanes, one after another (some 36 rounds a particle, nine cross-lane reads each).
template <class Box, class Entry, class Emit>
__device__ __forceinline__ int vertex_row(const Box& bx, const double4* P, const int* vst,
                                          const int* nvt, const double2* vpos, double rv,
                                          double vc, double vc2, double vp2, bool shift,
                                          int lane, int hs, bool has, double2 xv, double4 cp,
                                          int nn, Entry entry, Emit emit) {
    constexpr int HALF = WAVE / 2;
    int cnt = 0;
    for (int k0 = 0; k0 < nn; k0 += HALF) {
        int rf = 0, rn = 0;
        double rx = 0.0, ry = 0.0, rr = 0.0;
        double2 r0 = make_double2(0.0, 0.0);
        bool near = false;
        if (k0 + lane < nn) {
            const int q = entry(k0 + lane);
            const double4 c = P[q];
            rx = c.x;
            ry = c.y;
            rr = c.z;
            rf = vst[q];
            rn = nvt[q];
            const double2 u = vpos[rf];
            r0 = make_double2(u.x - c.x, u.y - c.y);
            near = true;
            if (shift) {  // both rings' radii and vc, with vertex_ring_near's margin
                const double ex = pbc(cp.x, c.x, bx.Lx, bx.invLx, bx.halfLx, bx.fast);
                const double ey = pbc(cp.y, c.y, bx.Ly, bx.invLy, bx.halfLy, bx.fast);
                const double reach = (cp.z - rv) + (c.z - rv) + vc;
                near = ex * ex + ey * ey < reach * reach * (1.0 + 1e-6);
            }
        }
        unsigned gm = 0;
        for (unsigned m = (unsigned)(__builtin_amdgcn_ballot_w64(near) >> hs); m; m &= m - 1) {
            const int k = __builtin_ctz(m);
            const double cx = __shfl(rx, k, HALF), cy = __shfl(ry, k, HALF);
            const double cr = __shfl(rr, k, HALF);
            const double kx = image_index(xv.x - cx, bx.Lx, bx.invLx, bx.halfLx, bx.fast);
            const double ky = image_index(xv.y - cy, bx.Ly, bx.invLy, bx.halfLy, bx.fast);
            const double dx = pbc_known(xv.x, cx, bx.Lx, kx, bx.fast);  // = pbc(xv, cq)
            const double dy = pbc_known(xv.y, cy, bx.Ly, ky, bx.fast);
            const double d2 = dx * dx + dy * dy;
            if (has && d2 < vp2 && vertex_ring_near(d2, cr, rv, vc)) gm |= 1u << k;
        }
        while (__builtin_amdgcn_ballot_w64(gm != 0) != 0) {
            const bool on = gm != 0;
            const int k = on ? __builtin_ctz(gm) : 0;
            const double cx = __shfl(rx, k, HALF), cy = __shfl(ry, k, HALF);
            const double cr = __shfl(rr, k, HALF);
            const double2 v0 = make_double2(__shfl(r0.x, k, HALF), __shfl(r0.y, k, HALF));
            const int f0 = __shfl(rf, k, HALF), nq = __shfl(rn, k, HALF);
            if (on) {
                const double kx = image_index(xv.x - cx, bx.Lx, bx.invLx, bx.halfLx, bx.fast);
                const double ky = image_index(xv.y - cy, bx.Ly, bx.invLy, bx.halfLy, bx.fast);
                const double dx = pbc_known(xv.x, cx, bx.Lx, kx, bx.fast);
                const double dy = pbc_known(xv.y, cy, bx.Ly, ky, bx.fast);
                const RingWindow w = ring_window(dx, dy, v0, cr - rv, vc, nq);
                for (int c = 0; c < w.count; ++c) {
                    const int u = f0 + (c < w.wrapped ? c : w.first + c - w.wrapped);
                    const double2 xu = vpos[u];
                    double ex, ey;
                    if (shift) {
                        ex = pbc_known(xv.x, xu.x, bx.Lx, kx, bx.fast);
                        ey = pbc_known(xv.y, xu.y, bx.Ly, ky, bx.fast);
                    } else {
                        ex = pbc(xv.x, xu.x, bx.Lx, bx.invLx, bx.halfLx, bx.fast);
                        ey = pbc(xv.y, xu.y, bx.Ly, bx.invLy, bx.halfLy, bx.fast);
                    }
                    if (ex * ex + ey * ey < vc2) emit(cnt++, u);
                }
            }
            gm &= gm - 1;
        }
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
