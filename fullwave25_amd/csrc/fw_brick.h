// Bricks of a 3D grid: the geometry, and the staging of three components with the arms of the derivative
// along each (fw_kernels_brick3d.hip, fw_kernels_adjoint3d.hip).
#pragma once

#include "fw_quad.h"

namespace fw {

namespace {

constexpr int BX = kBrickX, BY = kBrickY, BZ = kBrickZ;
static_assert(BX == 4 && BY == 8 && BZ == 32, "wavefront = x plane, lane = (row, quad)");

// Where a workgroup's brick and a lane's quad are.
struct Brick {
    int i0, j0, k0;      // first cell
    int wave, row, quad; // the wavefront's x plane, the lane's row and quad within the brick
    uint32_t c;          // element of the quad
    int n;               // its updated cells (0: none)
};
// Workgroup to brick. With `runs` each XCD takes a contiguous run of bricks, so that neighbours' arms share
// an L2 (131 x 117 x 109: 53.5 -> 49.0 us a step; 200 x 180 x 160: 160.5 -> 148.2); on large grids eight
// runs at once read more than the memory-side cache holds (600 x 500 x 200: 1782 -> 1939; 400 x 400 x 360:
// velocity 838 -> 898, pressure 878 -> 857). The caller times both.
__device__ __forceinline__ uint32_t brick_number(bool runs) { return runs ? xcd_order(blockIdx.x, gridDim.x) : blockIdx.x; }
__device__ inline Brick brick_of(const DevSim& s, uint32_t tile, uint32_t ny, uint32_t nz) {
    Brick b;
    const uint32_t t = tile / nz, bz = tile - t * nz, bx = t / ny, by = t - bx * ny;
    b.i0 = kHalo + (int)bx * BX;
    b.j0 = kHalo + (int)by * BY;
    b.k0 = (int)bz * BZ;
    b.wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    b.row = (threadIdx.x >> 3) & 7;
    b.quad = threadIdx.x & 7;
    const int i = b.i0 + b.wave, j = b.j0 + b.row, k = b.k0 + 4 * b.quad;
    b.c = (uint32_t)i * (uint32_t)s.sx + (uint32_t)(j * (int)s.sy + k);
    const int left = (int)s.nz - kHalo - k;
    b.n = i < (int)s.nx - kHalo && j < (int)s.ny - kHalo && k >= kHalo && left > 0 ? min(left, 4) : 0;
    return b;
}
// plane i0 + dx of a field, and a quad's element within a plane; both clamped into the grid
__device__ inline const float* plane(const DevSim& s, const Brick& b, const float* f, int dx) {
    return f + (uint32_t)min(max(b.i0 + dx, 0), (int)s.nx - 1) * (uint64_t)s.sx;
}
__device__ inline uint32_t in_plane(const DevSim& s, const Brick& b, int dy, int z) {
    const int j = min(max(b.j0 + dy, 0), (int)s.ny - 1);
    return (uint32_t)(j * (int)s.sy + min(max(b.k0 + z, 0), (int)s.sy - 4));
}

// LDS. X arms: planes from XLO (a multiple of 4 loads), [plane][row][32 columns], so that load l of
// thread t goes to quad 256 l + t. Row sets: the rows -8 .. 15 of the BX updated planes, then SIDE rows
// from FIRST of the planes -1 and BX, with 4 columns on each side; the z arms' outer quads apart.
constexpr int kArm = BX + 15, kArmLoads = (kArm + 3) / 4, kArmSize = kArm * BY * BZ;
constexpr int R = BZ + 8;  // a row of a row set
template <int LO, int HI, int SIDE, int FIRST = -1>
struct Rows {
    static constexpr int N = HI - LO;
    static constexpr int size = (BX * N + 2 * SIDE) * R;
    __device__ static int at(int dx) {  // row 0, column 0 of a plane
        const int row = dx < 0 ? BX * N - FIRST : dx < BX ? dx * N - LO : BX * N + SIDE - FIRST;
        return row * R + 4;
    }
};
constexpr int kEnds = 8;  // columns -8 .. -5 and BZ + 4 .. BZ + 7 of a row
__device__ __forceinline__ F4 lds4(const float* p) { return *reinterpret_cast<const F4*>(p); }
__device__ __forceinline__ void put4(float* p, const F4& v) { *reinterpret_cast<F4*>(p) = v; }

// columns -8 .. 11 from the quad at q (`centre`), whose row's ends are `ends`
__device__ __forceinline__ void z_arm(const float* q, const float* ends, int quad, const F4& centre, float (&z)[20]) {
    const F4 x[5] = {lds4(quad > 0 ? q - 8 : ends), lds4(q - 4), centre, lds4(q + 4), lds4(quad < BZ / 4 - 1 ? q + 8 : ends + 4)};
#pragma unroll
    for (int i = 0; i < 20; ++i) z[i] = x[i / 4][i % 4];
}
// elements beside a quad: [e + 1] with `right` after the last, [e - 1] with `left` before the first
__device__ __forceinline__ float after(const F4& q, float right, int e) { return e < 3 ? q[e + 1] : right; }
__device__ __forceinline__ float before(const F4& q, float left, int e) { return e > 0 ? q[e - 1] : left; }

// Store a quad of which the first n cells (1 to 4) are updated.
template <bool NT>
__device__ __forceinline__ F4 load_memory(const float* f, uint32_t c) {
    return NT ? ld4nt(f, c) : ld4(f, c);
}
template <bool NT>
__device__ inline void store_quad(float* f, uint32_t c, const F4& v, int n) {
    if (n == 4) {
        if (NT) st4nt(f, c, v);
        else st4(f, c, v);
        return;
    }
#pragma unroll
    for (int e = 0; e < 3; ++e)
        if (e < n) gst32(f, c + e, v[e]);
}

// Three components, each differentiated along its own axis, as the difference between the cells at
// m - 1 + SH and -m + SH (m = 1 .. 8), with the transverse pairs beside SH and SH - 1: SH = 0 backward
// (pressure from velocities; the transpose of the forward one), SH = 1 forward.
// x: the x arm, the rows -1 and BY of the planes SH - 1 .. SH + BX - 1, and the columns beside their rows
template <int SH>
using YRows = Rows<-8, BY + 8, BY + 1, SH - 1>;
using ZRows = Rows<-1, BY + 1, BY + 1>;
constexpr int kXLoads = kArmLoads + 1;
template <int SH>
struct Arms {
    __attribute__((aligned(16))) float X[kArmSize], F[(BX + 1) * 2 * BZ], Y[YRows<SH>::size], Z[ZRows::size], E[BX * BY * kEnds],
        G[(BX + 1) * BY * 2];
};

// the quads of x beside its arm (160), of y beside the planes and arms (88), of z (24, and 128 ends)
struct SideQuad {
    int dx, dy, z;
    bool used;
};
template <int SH>
__device__ inline SideQuad x_side(int t) {
    if (t < 80) return SideQuad{(t >> 4) - 1 + SH, t & 8 ? BY : -1, 4 * (t & 7), true};
    const int q = min(t - 80, 79);
    return SideQuad{(q >> 4) - 1 + SH, (q >> 1) & 7, q & 1 ? BZ : -4, t < 160};
}
template <int SH>
__device__ inline SideQuad y_side(int t) {
    if (t < 16) return SideQuad{t & 8 ? BX : -1, SH ? BY : -1, 4 * (t & 7), true};
    const int q = min(t - 16, 71), row = q >> 1;  // nine rows of the updated planes
    return SideQuad{row / 9, row % 9 - 1 + SH, q & 1 ? BZ : -4, t < 88};
}
template <int SH>
__device__ inline SideQuad z_beside(const Brick& b, int t) {  // rows -1 and BY (wavefront 2), the column beside (3)
    if (b.wave == 2) return SideQuad{b.row >> 1, b.row & 1 ? BY : -1, 4 * b.quad, true};
    const int q = min(t & 63, 23);
    return SideQuad{q < 8 ? -1 : q < 16 ? BX : (q - 16) >> 1, q < 16 ? q & 7 : q & 1 ? BY : -1, SH ? BZ : -4, (t & 63) < 24};
}
__device__ inline SideQuad z_end(int t) {  // beside the rows of the updated planes
    const int q = min(t, 127), h = q & 3;
    return SideQuad{q >> 5, (q >> 2) & 7, h < 2 ? 4 * h - 8 : BZ + 4 * h - 8, t < 128};
}
__device__ __forceinline__ uint64_t plane_at(const DevSim& s, const Brick& b, int dx) {
    return (uint32_t)min(max(b.i0 + dx, 0), (int)s.nx - 1) * (uint64_t)s.sx;
}
__device__ __forceinline__ uint32_t side_element(const DevSim& s, const Brick& b, const SideQuad& w) {
    return (uint32_t)plane_at(s, b, w.dx) + in_plane(s, b, w.dy, w.z);
}

// the quads a lane stages
struct ArmQuads {
    F4 x[kXLoads], y0, y1, y2, y3, z0, z1, z2;
};
// load(component, element the wavefront shares, element of the lane)
template <int SH, class Load>
__device__ __forceinline__ void load_arms(const DevSim& s, const Brick& b, const Load& load, ArmQuads& q) {
    const int t = threadIdx.x;
    const uint32_t mid = in_plane(s, b, b.row, 4 * b.quad);
    const uint32_t arm = in_plane(s, b, (b.wave & 1 ? BY : -8) + b.row, 4 * b.quad);
    // (plane 19 of the x arm isn't used)
#pragma unroll
    for (int l = 0; l < kArmLoads; ++l) q.x[l] = load(0, plane_at(s, b, min(b.wave + 4 * l, kArm - 1) - 8 + SH), mid);
    q.x[kArmLoads] = load(0, 0, side_element(s, b, x_side<SH>(t)));
    q.y0 = load(1, plane_at(s, b, b.wave), mid);
    q.y1 = load(1, plane_at(s, b, b.wave >> 1), arm);
    q.y2 = load(1, plane_at(s, b, 2 + (b.wave >> 1)), arm);
    // wavefronts 0 and 1: the planes -1 and BX of y and z, and z's ends; 2 and 3 what lies beside
    const uint32_t other = (uint32_t)plane_at(s, b, b.wave & 1 ? BX : -1) + mid;
    const uint32_t beside = side_element(s, b, z_beside<SH>(b, t));
    q.y3 = load(1, 0, b.wave < 2 ? other : side_element(s, b, y_side<SH>(max(t - 128, 0))));
    q.z0 = load(2, plane_at(s, b, b.wave), mid);
    q.z1 = load(2, 0, b.wave < 2 ? other : beside);
    q.z2 = load(2, 0, side_element(s, b, z_end(t)));
}
template <int SH>
__device__ __forceinline__ void put_arms(const Brick& b, const ArmQuads& q, Arms<SH>& m) {
    const int t = threadIdx.x, at = b.row * R + 4 * b.quad;
    const F4 side = q.x[kArmLoads], y3 = q.y3, z1 = q.z1, z2 = q.z2;
#pragma unroll
    for (int l = 0; l < kArmLoads; ++l)
        if (l < kArmLoads - 1 || b.wave + 4 * l < kArm) put4(m.X + 4 * (256 * l + t), q.x[l]);
    {
        const SideQuad w = x_side<SH>(t);
        const float lo = side.x, hi = side.w;
        if (t < 80) put4(m.F + 4 * t, side);
        else if (w.used) m.G[t - 80] = w.z < 0 ? hi : lo;
    }
    put4(m.Y + YRows<SH>::at(b.wave) + at, q.y0);
    put4(m.Y + YRows<SH>::at(b.wave >> 1) + (b.wave & 1 ? BY : -8) * R + at, q.y1);
    put4(m.Y + YRows<SH>::at(2 + (b.wave >> 1)) + (b.wave & 1 ? BY : -8) * R + at, q.y2);
    put4(m.Z + ZRows::at(b.wave) + at, q.z0);
    if (b.wave < 2) {
        put4(m.Y + YRows<SH>::at(b.wave ? BX : -1) + at, y3);
        put4(m.Z + ZRows::at(b.wave ? BX : -1) + at, z1);
        const SideQuad w = z_end(t);
        const bool end = w.z < -4 || w.z > BZ;
        put4(end ? m.E + ((w.dx * BY + w.dy) * 2 + (w.z > 0)) * 4 : m.Z + ZRows::at(w.dx) + w.dy * R + w.z, z2);
    } else {
        const SideQuad w = y_side<SH>(t - 128);
        if (w.used) put4(m.Y + YRows<SH>::at(w.dx) + w.dy * R + w.z, y3);
        const SideQuad v = z_beside<SH>(b, t);
        if (v.used) put4(m.Z + ZRows::at(v.dx) + v.dy * R + v.z, z1);
    }
}

// The derivative of component A along its axis at this lane's quad; k.w(e, m) weighs offset m (8: the
// transverse pairs) of cell e.
template <int A, int SH, class Weights>
__device__ __forceinline__ void derivative(const Brick& b, const Arms<SH>& lds, const Weights& k, F4& D) {
    const int at = b.row * R + 4 * b.quad;
    if constexpr (A == 0) {
        const float* X = lds.X + 4 * threadIdx.x + 8 * BY * BZ;  // the plane SH
        const F4 x0 = lds4(X), xm = lds4(X - BY * BZ);
#pragma unroll
        for (int m = 1; m <= 8; ++m) {
            const F4 hi = m == 1 ? x0 : lds4(X + (m - 1) * BY * BZ), lo = m == 1 ? xm : lds4(X - m * BY * BZ);
#pragma unroll
            for (int e = 0; e < 4; ++e) D[e] = tap(D[e], k.w(e, m - 1), hi[e], lo[e]);
        }
        // rows and columns beside: within the arm, or the fringe
        const float *F = lds.F + (b.wave + 1) * 2 * BZ + 4 * b.quad, *G = lds.G + ((b.wave + 1) * BY + b.row) * 2;
        const bool last = b.row == BY - 1, first = b.row == 0, left = b.quad == 0, right = b.quad == BZ / 4 - 1;
        const F4 u0 = lds4(last ? F + BZ : X + BZ), um = lds4(last ? F - BZ : X - BY * BZ + BZ);
        const F4 d0 = lds4(first ? F : X - BZ), dm = lds4(first ? F - 2 * BZ : X - BY * BZ - BZ);
        const float l0 = *(left ? G : X - 1), lm = *(left ? G - 2 * BY : X - BY * BZ - 1);
        const float r0 = *(right ? G + 1 : X + 4), rm = *(right ? G - 2 * BY + 1 : X - BY * BZ + 4);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            float tr = 0.f;
            tr += (u0[e] - um[e]) + (d0[e] - dm[e]);
            tr += (after(x0, r0, e) - after(xm, rm, e)) + (before(x0, l0, e) - before(xm, lm, e));
            D[e] = __builtin_fmaf(k.w(e, 8), tr, D[e]);
        }
    } else if constexpr (A == 1) {
        const float* Y = lds.Y + YRows<SH>::at(b.wave) + at + SH * R;
        const float *Yp = lds.Y + YRows<SH>::at(b.wave + 1) + at + SH * R, *Ym = lds.Y + YRows<SH>::at(b.wave - 1) + at + SH * R;
        const F4 y0 = lds4(Y), ym = lds4(Y - R);
#pragma unroll
        for (int m = 1; m <= 8; ++m) {
            const F4 hi = m == 1 ? y0 : lds4(Y + (m - 1) * R), lo = m == 1 ? ym : lds4(Y - m * R);
#pragma unroll
            for (int e = 0; e < 4; ++e) D[e] = tap(D[e], k.w(e, m - 1), hi[e], lo[e]);
        }
        const F4 u0 = lds4(Yp), um = lds4(Yp - R), d0 = lds4(Ym), dm = lds4(Ym - R);
        const float l0 = Y[-1], r0 = Y[4], lm = Y[-R - 1], rm = Y[-R + 4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            float tr = 0.f;
            tr += (u0[e] - um[e]) + (d0[e] - dm[e]);
            tr += (after(y0, r0, e) - after(ym, rm, e)) + (before(y0, l0, e) - before(ym, lm, e));
            D[e] = __builtin_fmaf(k.w(e, 8), tr, D[e]);
        }
    } else {
        const float *Z = lds.Z + ZRows::at(b.wave) + at, *Zp = lds.Z + ZRows::at(b.wave + 1) + at, *Zm = lds.Z + ZRows::at(b.wave - 1) + at;
        float z[20];
        z_arm(Z, lds.E + (b.wave * BY + b.row) * kEnds, b.quad, lds4(Z), z);
        const F4 xp = lds4(Zp), xm = lds4(Zm), yp = lds4(Z + R), ym = lds4(Z - R);
        constexpr int side = SH ? 4 : -1;
        const float xp_s = Zp[side], xm_s = Zm[side], yp_s = Z[R + side], ym_s = Z[-R + side];
        auto pair = [](const F4& q, float beside, int e) { return SH ? after(q, beside, e) - q[e] : q[e] - before(q, beside, e); };
#pragma unroll
        for (int e = 0; e < 4; ++e) {
#pragma unroll
            for (int m = 1; m <= 8; ++m) D[e] = tap(D[e], k.w(e, m - 1), z[8 + SH + e + m - 1], z[8 + SH + e - m]);
            float tr = 0.f;
            tr += pair(xp, xp_s, e) + pair(xm, xm_s, e);
            tr += pair(yp, yp_s, e) + pair(ym, ym_s, e);
            D[e] = __builtin_fmaf(k.w(e, 8), tr, D[e]);
        }
    }
}

}  // namespace

}  // namespace fw
