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
//   88 x 88 x 88      27.1 -> 20.2       131 x 117 x 109   53.4 -> 45.7      200 x 180 x 160   192 -> 149
//   300 x 64 x 300     192 -> 130        600 x 500 x 200   2126 -> 1782
// 400 x 400 x 360: velocity 888 -> 831, pressure 846 (marching) and 835. 64 x 64 x 64: 14.0 (per-cell)
// and 14.8, too few bricks. Exponential model, 131 x 117 x 109: 43.0 -> 35.7; 200 x 180 x 160: 138 -> 89.
// What bounds it: at 131 x 117 x 109 the phases of a brick (load, compute, store) with two rounds of
// three workgroups a CU (166 registers, 39 and 49 KB of LDS); large grids the memory traffic.
// Measured and left out: reading the stencil from the caches with 16-byte loads in place of LDS (131 x
// 117 x 109: 58.7, five dependent load phases); bricks from column 8 (partial cache lines written: 94 ->
// 59 with the former); 128 registers (spills: 82); bands of 2 to 8 bricks in y (51.6 to 52.5).
//
// Needs weights that all axes share, and rows with coefficients and weights (DevSim::rwide_v) or the
// exponential model. A wavefront whose cells share a code (exponential: a weight set) reads its row
// (weights) with scalar loads; the arithmetic order is the other families'.
#include "fw_brick.h"

namespace fw {

namespace {

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
            q[e] = coded_coef(VEL ? s.rtab_v : s.rtab_p, code);
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
__device__ __forceinline__ void pre_update(const DevSim& s, const Brick& b, const Coefs& k, const PreIn& o, const Arms<0>& lds) {
    F4 p = ld4(s.p, b.c), div{};
    const F4 K = ld4(s.K, b.c);
    {
        F4 D{};
        derivative<0, 0>(b, lds, k, D);
        pre_axis<EXPO, NT>(s, b, 0, D, k, o, div);
    }
    {
        F4 D{};
        derivative<1, 0>(b, lds, k, D);
        pre_axis<EXPO, NT>(s, b, 1, D, k, o, div);
    }
    {
        F4 D{};
        derivative<2, 0>(b, lds, k, D);
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
    __shared__ Arms<0> lds;
    TileWork w{};
    if (gs.g) {
        const GroupBoundary& e = gs.g[blockIdx.y];
        w = tile_work(e, brick_number(runs), e.step0 + gs.it + (gs.base ? *gs.base : 0));
    }
    const DevSim s = shot_view(batch, blockIdx.y);
    const Brick b = brick_of(s, brick_number(runs), nby, nbz);
    BrickCoef<false, EXPO> kc;
    if (b.n > 0) kc.head(s, b);
    ArmQuads q;
    load_arms<0>(s, b, [&](int a, uint64_t c0, uint32_t c) { return ld4(s.v[a] + c0, c); }, q);
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
    put_arms<0>(b, q, lds);
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

hipError_t load_brick_code() {
    hipFuncAttributes a;
    return hipFuncGetAttributes(&a, reinterpret_cast<const void*>(&k_velocity_brick<true, false, false>));
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
