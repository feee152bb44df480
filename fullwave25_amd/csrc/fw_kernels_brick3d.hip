// Brick kernels for 3D grids (kernel variant 5): a workgroup of 256 lanes updates a brick of 4 x 8 x 32
// (x, y, z) cells, each lane a quad of 4 consecutive z cells, each wavefront one x plane of 8 rows.
//
// The marching kernels (fw_kernels_pipe3d.hip) stream large grids, but a chunk of planes is a serial
// chain, and small grids have too few of them; the per-cell kernels have enough wavefronts, but read 55
// (velocity) and 72 (pressure) stencil values a cell through the address unit, which is busy 75 % of
// their time (131 x 117 x 109 cells: 1.25 M read instructions in the velocity update). Here a brick's
// arms are staged in LDS with 16-byte loads, 8 (velocity) and 13 (pressure) a lane, all issued before
// the first is waited for, as are the memory variables and the coefficient rows; a quad's stencil reads
// are 16-byte LDS reads. us a step, best of the other families -> bricks (16 read and written fields):
//   88 x 88 x 88      33.9 -> 21.8       131 x 117 x 109   68.0 -> 49.0      200 x 180 x 160   192 -> 148
//   300 x 64 x 300     206 -> 132        600 x 500 x 200   2126 -> 1782
// 400 x 400 x 360: velocity 886 -> 838, pressure 839 (marching) and 857. 64 x 64 x 64: 12.9 (per-cell)
// and 14.9, too few bricks. Exponential model, 131 x 117 x 109: 42.1 -> 37.9; 200 x 180 x 160: 134 -> 103.
// What bounds it: at 131 x 117 x 109 the phases of a brick (load, compute, store) with two rounds of
// three workgroups a CU (166 registers, 39 and 49 KB of LDS); large grids the memory traffic.
// Measured and left out: reading the stencil from the caches with 16-byte loads in place of LDS (131 x
// 117 x 109: 58.7, five dependent load phases); bricks from column 8 (partial cache lines written: 94 ->
// 59 with the former); 128 registers (spills: 82); bands of 2 to 8 bricks in y (51.6 to 52.5).
//
// Needs weights that all axes share, and rows with coefficients and weights (DevSim::rwide_v) or the
// exponential model. A wavefront whose cells share a code (exponential: a weight set) reads its row
// (weights) with scalar loads; the arithmetic order is the other families'.
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
// from -1 of the planes -1 and BX, with 4 columns on each side; the z arms' outer quads apart.
constexpr int kArm = BX + 15, kArmLoads = (kArm + 3) / 4, kArmSize = kArm * BY * BZ;
constexpr int R = BZ + 8;  // a row of a row set
template <int LO, int HI, int SIDE>
struct Rows {
    static constexpr int N = HI - LO;
    static constexpr int size = (BX * N + 2 * SIDE) * R;
    __device__ static int at(int dx) {  // row 0, column 0 of a plane
        const int row = dx < 0 ? BX * N + 1 : dx < BX ? dx * N - LO : BX * N + SIDE + 1;
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

// Coefficients and weights of a quad's cells. Of a wavefront whose cells share a code (SHARED; scalar
// registers), of one whose cells share a weight set, of cells that share neither.
struct SharedCoefs {
    float ik, a1, a2, b1, b2, weight[kNCoef];
    __device__ CodedCoef of(int) const { return CodedCoef{ik, a1, a2, b1, b2, 0}; }
    __device__ float w(int, int m) const { return weight[m]; }
};
struct CellCoefs {
    CodedCoef q[4];
    float weight[kNCoef];
    __device__ const CodedCoef& of(int e) const { return q[e]; }
    __device__ float w(int, int m) const { return weight[m]; }
};
struct MixedCoefs {
    CodedCoef q[4];
    float weight[4][kNCoef];
    __device__ const CodedCoef& of(int e) const { return q[e]; }
    __device__ float w(int e, int m) const { return weight[e][m]; }
};
__device__ inline void shared_weights(const DevSim& s, uint32_t set, float (&w)[kNCoef]) {
    const scalar_ptr p = as_scalar(s.coef) + set * 3 * kNCoef;
#pragma unroll
    for (int m = 0; m < kNCoef; ++m) w[m] = p[m];
}
__device__ inline bool all_are(const I4& q, int x) { return __all(q.x == x && q.y == x && q.z == x && q.w == x); }

// The coefficients of this lane's quad: codes (or sets) first, then, where the wavefront's codes differ,
// the cells' rows; both are loads that the staging hides.
template <bool VEL, bool EXPO>
struct BrickCoef {
    uint2 cw;
    I4 dc;
    uint32_t key;
    bool shared;
    CodedCoef q[4];
    __device__ void head(const DevSim& s, const Brick& b) {
        dc = I4{0, 0, 0, 0};
        if (!EXPO) cw = ldc4(s.rcode, b.c);
        else if (s.ndmap > 1) dc = ldi4(s.dcmap, b.c);
    }
    __device__ void rows(const DevSim& s, const Brick& b) {
        shared = false;
        if (EXPO) return;
        shared = wave_code(cw, &key);
        if (shared) return;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const uint32_t code = ((e < 2 ? cw.x : cw.y) >> (16 * (e & 1))) & 0xffffu;
            q[e] = coded_coef(VEL ? s.rtab_v : s.rtab_p, code != kCodeEscape ? code : 0u);
            if (code == kCodeEscape) q[e] = escape_coef<VEL, false>(s, b.c + e);
        }
    }
    // body(coefficients of the wavefront's active lanes)
    template <class Body>
    __device__ __forceinline__ void with(const DevSim& s, const Body& body) {
        if (shared) {
            const scalar_ptr row = as_scalar(VEL ? s.rwide_v : s.rwide_p) + key * kWideStride;
            SharedCoefs k{row[0], row[1], row[2], row[3], row[4], {}};
#pragma unroll
            for (int m = 0; m < kNCoef; ++m) k.weight[m] = row[5 + m];
            body(k);
            return;
        }
        if (!EXPO) dc = I4{q[0].dc, q[1].dc, q[2].dc, q[3].dc};
        const int set = __builtin_amdgcn_readfirstlane(dc.x);
        if (all_are(dc, set)) {
            CellCoefs k;
#pragma unroll
            for (int e = 0; e < 4; ++e) k.q[e] = q[e];
            shared_weights(s, (uint32_t)set, k.weight);
            body(k);
            return;
        }
        MixedCoefs k;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            k.q[e] = q[e];
            const float* w = s.coef + dc[e] * 3 * kNCoef;
#pragma unroll
            for (int m = 0; m < kNCoef; ++m) k.weight[e][m] = w[m];
        }
        body(k);
    }
};

// ---- velocity ---------------------------------------------------------------------------------

using VelRows = Rows<-8, BY + 8, BY + 2>;
constexpr int kVelLoads = kArmLoads + 3;
struct VelLds {
    __attribute__((aligned(16))) float X[kArmSize], Y[VelRows::size], E[BX * BY * kEnds];
};

// quads beside the rows: 4 of each of the rows 0 .. 7 of the updated planes, 2 of the others
struct VelSide {
    int dx, dy, z;
    __device__ explicit VelSide(int t) {
        const int q = t < 128 ? t >> 2 : 32 + ((t - 128) >> 1), h = t < 128 ? t & 3 : 1 + (t & 1);
        // rows 32 .. 51: the planes -1 and BX; 52 .. 59: rows -1 and BY of the updated planes
        dx = q < 32 ? q >> 3 : q < 42 ? -1 : q < 52 ? BX : (q - 52) >> 1;
        dy = q < 32 ? q & 7 : q < 42 ? q - 33 : q < 52 ? q - 43 : q & 1 ? BY : -1;
        z = h < 2 ? 4 * h - 8 : BZ + 4 * h - 8;
    }
};

__device__ __forceinline__ void vel_load(const DevSim& s, const Brick& b, F4 (&q)[kVelLoads]) {
    const int t = threadIdx.x, z = 4 * b.quad;
    const uint32_t mid = in_plane(s, b, b.row, z);
#pragma unroll
    for (int l = 0; l < kArmLoads; ++l) {  // plane 19: rows -1 and BY of the planes -1 and BX
        const int e = b.wave + 4 * l;
        if (l < kArmLoads - 1 || e < kArm) q[l] = ld4(plane(s, b, s.p, e - 7), mid);
        else q[l] = ld4(s.p, (uint32_t)(plane(s, b, s.p, b.row & 1 ? BX : -1) - s.p) + in_plane(s, b, b.row & 2 ? BY : -1, z));
    }
    const uint32_t arm = in_plane(s, b, (b.wave & 1 ? BY : -8) + b.row, z);
#pragma unroll
    for (int l = 0; l < 2; ++l) q[kArmLoads + l] = ld4(plane(s, b, s.p, 2 * l + (b.wave >> 1)), arm);
    const VelSide w(min(t, 183));
    q[kArmLoads + 2] = ld4(s.p, (uint32_t)(plane(s, b, s.p, w.dx) - s.p) + in_plane(s, b, w.dy, w.z));
}
__device__ __forceinline__ void vel_put(const Brick& b, const F4 (&q)[kVelLoads], VelLds& m) {
    const int t = threadIdx.x, at = b.row * R + 4 * b.quad;
#pragma unroll
    for (int l = 0; l < kArmLoads; ++l) {
        const int e = b.wave + 4 * l, dx = e - 7;
        if (l == kArmLoads - 1 && e >= kArm) {
            if (b.row < 4) put4(m.Y + VelRows::at(b.row & 1 ? BX : -1) + (b.row & 2 ? BY : -1) * R + 4 * b.quad, q[l]);
            continue;
        }
        put4(m.X + 4 * (256 * l + t), q[l]);
        if (dx >= -1 && dx <= BX) put4(m.Y + VelRows::at(dx) + at, q[l]);
    }
#pragma unroll
    for (int l = 0; l < 2; ++l)
        put4(m.Y + VelRows::at(2 * l + (b.wave >> 1)) + (b.wave & 1 ? BY : -8) * R + at, q[kArmLoads + l]);
    const VelSide w(min(t, 183));
    if (t < 184) {
        const bool end = w.z < -4 || w.z > BZ;
        float* e = m.E + ((w.dx * BY + w.dy) * 2 + (w.z > 0)) * 4;
        put4(end ? e : m.Y + VelRows::at(w.dx) + w.dy * R + w.z, q[kArmLoads + 2]);
    }
}

struct VelIn {
    F4 v[3], psi[3][2], decay, rho, rho_x, rho_y;
    float rho_z;
};

template <bool EXPO, bool TAPE, bool NT, class Coefs>
__device__ __forceinline__ void vel_axis(const DevSim& s, const Brick& b, int a, const F4& D, const F4& rn, const Coefs& k, const VelIn& o) {
    F4 tu, v = o.v[a], q1 = o.psi[a][0], q2 = o.psi[a][1];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        if (EXPO) {
            v[e] = o.decay[e] * velocity_step(v[e], s.dt, o.rho[e], rn[e], D[e]);
            tu[e] = o.decay[e] * D[e];
            continue;
        }
        const CodedCoef c = k.of(e);
        q1[e] = memory_step(c.b1, q1[e], c.a1, D[e]);
        q2[e] = memory_step(c.b2, q2[e], c.a2, D[e]);
        tu[e] = corrected(D[e], c.ik, q1[e], q2[e]);
        v[e] = velocity_step(v[e], s.dt, o.rho[e], rn[e], tu[e]);
    }
    if (!EXPO) {
        store_quad<NT>(s.psi[a][0], b.c, q1, b.n);
        store_quad<NT>(s.psi[a][1], b.c, q2, b.n);
    }
    store_quad<false>(s.v[a], b.c, v, b.n);
    if (TAPE) store_quad<false>(s.tape_u[a], b.c, tu, b.n);
}

// X: the X arm, Y: the Y rows, both at this lane's quad
template <bool EXPO, bool TAPE, bool NT, class Coefs>
__device__ __forceinline__ void vel_update(const DevSim& s, const Brick& b, const Coefs& k, const VelIn& o, const VelLds& lds) {
    const int at = b.row * R + 4 * b.quad;
    const float *X = lds.X + 4 * (256 + threadIdx.x) + 3 * BY * BZ, *Y = lds.Y + VelRows::at(b.wave) + at;
    const float *Yp = lds.Y + VelRows::at(b.wave + 1) + at, *Ym = lds.Y + VelRows::at(b.wave - 1) + at;
    auto x4 = [&](int m) { return lds4(X + m * BY * BZ); };
    auto y4 = [&](int dx, int dy, int z) { return lds4((dx > 0 ? Yp : dx < 0 ? Ym : Y) + dy * R + z); };
    auto y1 = [&](int dx, int dy, int z) { return (dx > 0 ? Yp : dx < 0 ? Ym : Y)[dy * R + z]; };
    const F4 c0 = y4(0, 0, 0), xp = y4(1, 0, 0), xm = y4(-1, 0, 0), yp = y4(0, 1, 0), ym = y4(0, -1, 0), xpyp = y4(1, 1, 0);
    const float c_l = y1(0, 0, -1), c_r = y1(0, 0, 4), xp_r = y1(1, 0, 4), yp_r = y1(0, 1, 4);
    {
        F4 D{};
#pragma unroll
        for (int m = 1; m <= 8; ++m) {
            const F4 hi = m == 1 ? xp : x4(m), lo = m == 1 ? c0 : m == 2 ? xm : x4(-(m - 1));
#pragma unroll
            for (int e = 0; e < 4; ++e) D[e] = tap(D[e], k.w(e, m - 1), hi[e], lo[e]);
        }
        const F4 xpym = y4(1, -1, 0);
        const float xp_l = y1(1, 0, -1);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            float tr = 0.f;
            tr += (xpyp[e] - yp[e]) + (xpym[e] - ym[e]);
            tr += (after(xp, xp_r, e) - after(c0, c_r, e)) + (before(xp, xp_l, e) - before(c0, c_l, e));
            D[e] = __builtin_fmaf(k.w(e, 8), tr, D[e]);
        }
        vel_axis<EXPO, TAPE, NT>(s, b, 0, D, o.rho_x, k, o);
    }
    {
        F4 D{};
#pragma unroll
        for (int m = 1; m <= 8; ++m) {
            const F4 hi = m == 1 ? yp : y4(0, m, 0), lo = m == 1 ? c0 : m == 2 ? ym : y4(0, -(m - 1), 0);
#pragma unroll
            for (int e = 0; e < 4; ++e) D[e] = tap(D[e], k.w(e, m - 1), hi[e], lo[e]);
        }
        const F4 xmyp = y4(-1, 1, 0);
        const float yp_l = y1(0, 1, -1);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            float tr = 0.f;
            tr += (xpyp[e] - xp[e]) + (xmyp[e] - xm[e]);
            tr += (after(yp, yp_r, e) - after(c0, c_r, e)) + (before(yp, yp_l, e) - before(c0, c_l, e));
            D[e] = __builtin_fmaf(k.w(e, 8), tr, D[e]);
        }
        vel_axis<EXPO, TAPE, NT>(s, b, 1, D, o.rho_y, k, o);
    }
    {
        float z[20];
        z_arm(Y, lds.E + (b.wave * BY + b.row) * kEnds, b.quad, c0, z);
        const float xm_r = y1(-1, 0, 4), ym_r = y1(0, -1, 4);
        F4 D{}, rn;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
#pragma unroll
            for (int m = 1; m <= 8; ++m) D[e] = tap(D[e], k.w(e, m - 1), z[8 + e + m], z[8 + e - (m - 1)]);
            float tr = 0.f;
            tr += (after(xp, xp_r, e) - xp[e]) + (after(xm, xm_r, e) - xm[e]);
            tr += (after(yp, yp_r, e) - yp[e]) + (after(ym, ym_r, e) - ym[e]);
            D[e] = __builtin_fmaf(k.w(e, 8), tr, D[e]);
            rn[e] = after(o.rho, o.rho_z, e);
        }
        vel_axis<EXPO, TAPE, NT>(s, b, 2, D, rn, k, o);
    }
}

template <bool EXPO, bool TAPE, bool NT>
__global__ __launch_bounds__(256) void k_velocity_brick(DevSim batch, uint32_t nby, uint32_t nbz, bool runs) {
    __shared__ VelLds lds;
    const DevSim s = shot_view(batch, blockIdx.y);
    const Brick b = brick_of(s, brick_number(runs), nby, nbz);
    BrickCoef<true, EXPO> kc;
    if (b.n > 0) kc.head(s, b);
    F4 q[kVelLoads];
    vel_load(s, b, q);
    VelIn o;
    if (b.n > 0) {
#pragma unroll
        for (int a = 0; a < 3; ++a) {
            if (EXPO) continue;
            o.psi[a][0] = load_memory<NT>(s.psi[a][0], b.c);
            o.psi[a][1] = load_memory<NT>(s.psi[a][1], b.c);
        }
        if (EXPO) o.decay = ld4(s.aexp, b.c);
        kc.rows(s, b);
    }
    vel_put(b, q, lds);
    __syncthreads();
    if (b.n <= 0) return;
    o.rho = ld4(s.rho, b.c);
    o.rho_x = ld4(s.rho, b.c + (uint32_t)s.sx);
    o.rho_y = ld4(s.rho, b.c + (uint32_t)s.sy);
    o.rho_z = ld1(s.rho, b.c + 4);  // read by a fourth updated cell only; else within the array all the same
    for (int a = 0; a < 3; ++a) o.v[a] = ld4(s.v[a], b.c);
    kc.with(s, [&](const auto& k) { vel_update<EXPO, TAPE, NT>(s, b, k, o, lds); });
}

// ---- pressure ---------------------------------------------------------------------------------

// v_x: its x arm, the rows -1 and BY of the planes -1 .. BX - 1, and the columns beside the rows between
using PyRows = Rows<-8, BY + 8, BY + 1>;  // v_y
using PzRows = Rows<-1, BY + 1, BY + 1>;  // v_z
constexpr int kPxLoads = kArmLoads + 1;
struct PreLds {
    __attribute__((aligned(16))) float X[kArmSize], F[(BX + 1) * 2 * BZ], Y[PyRows::size], Z[PzRows::size], E[BX * BY * kEnds],
        G[(BX + 1) * BY * 2];
};

// the quads of v_x beside its x arm (160), of v_y beside the planes and arms (88), of v_z (24, and 128 ends)
struct PreSide {
    int dx, dy, z;
    bool used;
};
__device__ inline PreSide px_side(int t) {
    if (t < 80) return PreSide{(t >> 4) - 1, t & 8 ? BY : -1, 4 * (t & 7), true};
    const int q = min(t - 80, 79);
    return PreSide{(q >> 4) - 1, (q >> 1) & 7, q & 1 ? BZ : -4, t < 160};
}
__device__ inline PreSide py_side(int t) {
    if (t < 16) return PreSide{t & 8 ? BX : -1, -1, 4 * (t & 7), true};
    const int q = min(t - 16, 71), row = q >> 1;  // the rows -1 .. 7 of the updated planes
    return PreSide{row / 9, row % 9 - 1, q & 1 ? BZ : -4, t < 88};
}
__device__ inline PreSide pz_beside(const Brick& b, int t) {  // rows -1 and BY (wavefront 2), before the rows (3)
    if (b.wave == 2) return PreSide{b.row >> 1, b.row & 1 ? BY : -1, 4 * b.quad, true};
    const int q = min(t & 63, 23);
    return PreSide{q < 8 ? -1 : q < 16 ? BX : (q - 16) >> 1, q < 16 ? q & 7 : q & 1 ? BY : -1, -4, (t & 63) < 24};
}
__device__ inline PreSide pz_end(int t) {  // beside the rows of the updated planes
    const int q = min(t, 127), h = q & 3;
    return PreSide{q >> 5, (q >> 2) & 7, h < 2 ? 4 * h - 8 : BZ + 4 * h - 8, t < 128};
}
__device__ __forceinline__ uint32_t side_element(const DevSim& s, const Brick& b, const PreSide& w) {
    return (uint32_t)(plane(s, b, s.p, w.dx) - s.p) + in_plane(s, b, w.dy, w.z);
}

// the quads a lane stages
struct PreStage {
    F4 x[kPxLoads], y0, y1, y2, y3, z0, z1, z2;
};
__device__ __forceinline__ void pre_load(const DevSim& s, const Brick& b, PreStage& q) {
    const int t = threadIdx.x;
    const uint32_t mid = in_plane(s, b, b.row, 4 * b.quad);
    const uint32_t arm = in_plane(s, b, (b.wave & 1 ? BY : -8) + b.row, 4 * b.quad);
    // (plane 19 of the x arm isn't used)
#pragma unroll
    for (int l = 0; l < kArmLoads; ++l) q.x[l] = ld4(plane(s, b, s.v[0], min(b.wave + 4 * l, kArm - 1) - 8), mid);
    q.x[kArmLoads] = ld4(s.v[0], side_element(s, b, px_side(t)));
    q.y0 = ld4(plane(s, b, s.v[1], b.wave), mid);
    q.y1 = ld4(plane(s, b, s.v[1], b.wave >> 1), arm);
    q.y2 = ld4(plane(s, b, s.v[1], 2 + (b.wave >> 1)), arm);
    // wavefronts 0 and 1: the planes -1 and BX of v_y and v_z, and v_z's ends; 2 and 3 what lies beside
    const uint32_t other = (uint32_t)(plane(s, b, s.p, b.wave & 1 ? BX : -1) - s.p) + mid;
    const uint32_t beside = side_element(s, b, pz_beside(b, t));
    q.y3 = ld4(s.v[1], b.wave < 2 ? other : side_element(s, b, py_side(max(t - 128, 0))));
    q.z0 = ld4(plane(s, b, s.v[2], b.wave), mid);
    q.z1 = ld4(s.v[2], b.wave < 2 ? other : beside);
    q.z2 = ld4(s.v[2], side_element(s, b, pz_end(t)));
}
__device__ __forceinline__ void pre_put(const Brick& b, const PreStage& q, PreLds& m) {
    const int t = threadIdx.x, at = b.row * R + 4 * b.quad;
    const F4 side = q.x[kArmLoads], y3 = q.y3, z1 = q.z1, z2 = q.z2;
#pragma unroll
    for (int l = 0; l < kArmLoads; ++l)
        if (l < kArmLoads - 1 || b.wave + 4 * l < kArm) put4(m.X + 4 * (256 * l + t), q.x[l]);
    {
        const PreSide w = px_side(t);
        const float lo = side.x, hi = side.w;
        if (t < 80) put4(m.F + 4 * t, side);
        else if (w.used) m.G[t - 80] = w.z < 0 ? hi : lo;
    }
    put4(m.Y + PyRows::at(b.wave) + at, q.y0);
    put4(m.Y + PyRows::at(b.wave >> 1) + (b.wave & 1 ? BY : -8) * R + at, q.y1);
    put4(m.Y + PyRows::at(2 + (b.wave >> 1)) + (b.wave & 1 ? BY : -8) * R + at, q.y2);
    put4(m.Z + PzRows::at(b.wave) + at, q.z0);
    if (b.wave < 2) {
        put4(m.Y + PyRows::at(b.wave ? BX : -1) + at, y3);
        put4(m.Z + PzRows::at(b.wave ? BX : -1) + at, z1);
        const PreSide w = pz_end(t);
        const bool end = w.z < -4 || w.z > BZ;
        put4(end ? m.E + ((w.dx * BY + w.dy) * 2 + (w.z > 0)) * 4 : m.Z + PzRows::at(w.dx) + w.dy * R + w.z, z2);
    } else {
        const PreSide w = py_side(t - 128);
        if (w.used) put4(m.Y + PyRows::at(w.dx) + w.dy * R + w.z, y3);
        const PreSide v = pz_beside(b, t);
        if (v.used) put4(m.Z + PzRows::at(v.dx) + v.dy * R + v.z, z1);
    }
}

struct PreIn {
    F4 phi[3][2], decay;
};

template <bool EXPO, bool NT, class Coefs>
__device__ __forceinline__ void pre_axis(const DevSim& s, const Brick& b, int a, const F4& D, const Coefs& k, const PreIn& o, F4& div) {
    if (EXPO) {
#pragma unroll
        for (int e = 0; e < 4; ++e) div[e] += D[e];
        return;
    }
    F4 q1 = o.phi[a][0], q2 = o.phi[a][1];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        const CodedCoef c = k.of(e);
        q1[e] = memory_step(c.b1, q1[e], c.a1, D[e]);
        q2[e] = memory_step(c.b2, q2[e], c.a2, D[e]);
        div[e] += corrected(D[e], c.ik, q1[e], q2[e]);
    }
    store_quad<NT>(s.phi[a][0], b.c, q1, b.n);
    store_quad<NT>(s.phi[a][1], b.c, q2, b.n);
}

template <bool EXPO, bool TAPE, bool NT, class Coefs>
__device__ __forceinline__ void pre_update(const DevSim& s, const Brick& b, const Coefs& k, const PreIn& o, const PreLds& lds) {
    const int at = b.row * R + 4 * b.quad;
    F4 p = ld4(s.p, b.c), div{};
    const F4 K = ld4(s.K, b.c);
    {
        const float* X = lds.X + 4 * (512 + threadIdx.x);
        F4 D{};
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
        pre_axis<EXPO, NT>(s, b, 0, D, k, o, div);
    }
    {
        const float *Y = lds.Y + PyRows::at(b.wave) + at;
        const float *Yp = lds.Y + PyRows::at(b.wave + 1) + at, *Ym = lds.Y + PyRows::at(b.wave - 1) + at;
        F4 D{};
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
        pre_axis<EXPO, NT>(s, b, 1, D, k, o, div);
    }
    {
        const float *Z = lds.Z + PzRows::at(b.wave) + at;
        const float *Zp = lds.Z + PzRows::at(b.wave + 1) + at, *Zm = lds.Z + PzRows::at(b.wave - 1) + at;
        float z[20];
        z_arm(Z, lds.E + (b.wave * BY + b.row) * kEnds, b.quad, lds4(Z), z);
        const F4 xp = lds4(Zp), xm = lds4(Zm), yp = lds4(Z + R), ym = lds4(Z - R);
        const float xp_l = Zp[-1], xm_l = Zm[-1], yp_l = Z[R - 1], ym_l = Z[-R - 1];
        F4 D{};
#pragma unroll
        for (int e = 0; e < 4; ++e) {
#pragma unroll
            for (int m = 1; m <= 8; ++m) D[e] = tap(D[e], k.w(e, m - 1), z[8 + e + m - 1], z[8 + e - m]);
            float tr = 0.f;
            tr += (xp[e] - before(xp, xp_l, e)) + (xm[e] - before(xm, xm_l, e));
            tr += (yp[e] - before(yp, yp_l, e)) + (ym[e] - before(ym, ym_l, e));
            D[e] = __builtin_fmaf(k.w(e, 8), tr, D[e]);
        }
        pre_axis<EXPO, NT>(s, b, 2, D, k, o, div);
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        const float x = pressure_step(p[e], s.dt, K[e], div[e]);
        p[e] = EXPO ? o.decay[e] * x : x;
    }
    store_quad<false>(s.p, b.c, p, b.n);
    if (TAPE) store_quad<false>(s.tape_div, b.c, div, b.n);
}

// gs.g non-null: each workgroup then also does the step's source, pressure-release and sensor work of
// its brick, for shot blockIdx.y
template <bool EXPO, bool TAPE, bool NT>
__global__ __launch_bounds__(256) void k_pressure_brick(DevSim batch, uint32_t nby, uint32_t nbz, bool runs, GroupStep gs) {
    __shared__ PreLds lds;
    TileWork w{};
    if (gs.g) {
        const GroupBoundary& e = gs.g[blockIdx.y];
        w = tile_work(e, brick_number(runs), e.step0 + gs.it + (gs.base ? *gs.base : 0));
    }
    const DevSim s = shot_view(batch, blockIdx.y);
    const Brick b = brick_of(s, brick_number(runs), nby, nbz);
    BrickCoef<false, EXPO> kc;
    if (b.n > 0) kc.head(s, b);
    PreStage q;
    pre_load(s, b, q);
    PreIn o;
    if (b.n > 0) {
#pragma unroll
        for (int a = 0; a < 3; ++a) {
            if (EXPO) continue;
            o.phi[a][0] = load_memory<NT>(s.phi[a][0], b.c);
            o.phi[a][1] = load_memory<NT>(s.phi[a][1], b.c);
        }
        if (EXPO) o.decay = ld4(s.aexp, b.c);
        kc.rows(s, b);
    }
    pre_put(b, q, lds);
    __syncthreads();
    if (b.n > 0) kc.with(s, [&](const auto& k) { pre_update<EXPO, TAPE, NT>(s, b, k, o, lds); });
    if (!gs.g) return;
    __syncthreads();
    tile_boundary(w);
}

// Memory variables go past the caches (non-temporal) where a step's arrays (about 20 of 4 bytes a cell)
// exceed the memory-side cache of 256 MB anyway. us a step with and without: 131 x 117 x 109 (2.0 M
// elements) 61.8 / 54.4, 160 x 140 x 150 (3.6 M) 98.9 / 95.5, 150 x 160 x 170 (4.6 M) 128.5 / 132.5,
// 190 x 190 x 180 (6.9 M) 192.9 / 203.0.
bool memory_streams(const DevSim& s) { return s.nx * s.sx * (int64_t)s.nshots >= ((int64_t)1 << 22); }

template <bool EXPO, bool TAPE, bool NT>
void launch_bricks(const DevSim& s, bool runs, bool velocity, const GroupStep& gs, hipStream_t st) {
    const BrickGrid g = brick_grid(s);
    const dim3 grid((unsigned)(g.nx * g.ny * g.nz), (unsigned)s.nshots);
    if (velocity) hipLaunchKernelGGL((k_velocity_brick<EXPO, TAPE, NT>), grid, dim3(256), 0, st, s, (uint32_t)g.ny, (uint32_t)g.nz, runs);
    else hipLaunchKernelGGL((k_pressure_brick<EXPO, TAPE, NT>), grid, dim3(256), 0, st, s, (uint32_t)g.ny, (uint32_t)g.nz, runs, gs);
}

}  // namespace

BrickGrid brick_grid(const DevSim& s) {
    // from column 0: the rows of a brick are then whole cache lines
    return BrickGrid{(s.nx - 2 * kHalo + BX - 1) / BX, (s.ny - 2 * kHalo + BY - 1) / BY, (s.nz - kHalo + BZ - 1) / BZ};
}

bool brick_supported(const DevSim& s) {
    if (s.ndim != 3 || !s.coef_axes_same || !(s.aexp || (s.rcode && s.rwide_v))) return false;
    if (s.nx * s.sx >= ((int64_t)1 << 30)) return false;
    const BrickGrid g = brick_grid(s);
    return g.nx * g.ny * g.nz < ((int64_t)1 << 31);
}

hipError_t launch_brick(const DevSim& s, const LaunchCfg& cfg, bool velocity, const GroupStep& gs, hipStream_t st) {
    const bool runs = cfg.chunk == 1;
    const bool nt = memory_streams(s);
    if (s.aexp) {  // no memory variables
        if (s.tape_div) launch_bricks<true, true, false>(s, runs, velocity, gs, st);
        else launch_bricks<true, false, false>(s, runs, velocity, gs, st);
    } else if (s.tape_div) {
        if (nt) launch_bricks<false, true, true>(s, runs, velocity, gs, st);
        else launch_bricks<false, true, false>(s, runs, velocity, gs, st);
    } else {
        if (nt) launch_bricks<false, false, true>(s, runs, velocity, gs, st);
        else launch_bricks<false, false, false>(s, runs, velocity, gs, st);
    }
    return hipGetLastError();
}

}  // namespace fw
