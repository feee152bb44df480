// Tiled 2D kernels with 4-wide vector access (gfx950).
//
// A workgroup of 256 lanes (4 wavefronts) owns a tile of TX rows x TW columns. It stages the input
// field(s) of the tile plus the stencil halo into LDS with 16-byte loads, then every lane updates
// 4 consecutive cells (one float4 column quad) a pass. All per-cell maps and memory variables
// move as float4, which is what lets the HBM stream approach the copy-kernel rate; the stencil
// operands come from LDS.
//
// What bounds it, and why it is laid out so (us a step, velocity + pressure, 4256 x 2208 / 1152^2 /
// 672^2 cells, coded coefficients):
//   * large grids stream at the rate of a 9-read, 6-write probe (5.8 TB/s); small ones wait for
//     memory: a chain of code -> table row -> arithmetic -> store per workgroup, with too few
//     workgroups to hide it. So the staging loads, the first pass's operands and the table row
//     are all issued before the first of them is waited for, and the tiles are small (1024 or 2048
//     cells): 185 / 42 / 27 -> 183 / 34.4 / 18.0 against 256-column tiles staged by a loop of
//     load, wait and store.
//   * tiles nearer to square stage fewer halo cells: 2.1-3.2 staged cells of p per updated one
//     instead of 2.1-3.1 of tiles four times as wide, at half or a quarter of the cells a
//     workgroup.
//   * a row gather of each cell's coefficients costs 13 % of the velocity kernel. Media are
//     piecewise constant, so most wavefronts hold one code: those read the row and the stencil
//     weights once with scalar loads (WaveCoef): 183 -> 177 at 4256 x 2208.
//
// Requires ny % 4 == 0 (16-byte aligned rows). Arithmetic order is the per-cell kernels'.
#include "fw_quad.h"

namespace fw {

namespace {

constexpr int kLanes = 256;  // threads per workgroup

// A tile shape: TX rows x TW columns, updated in passes of kRows rows (each lane one quad a pass).
template <int TW_, int TX_>
struct Shape {
    static constexpr int TW = TW_, TX = TX_;
    static constexpr int kQuads = TW / 4;           // column quads per tile row
    static constexpr int kRows = kLanes / kQuads;   // tile rows per pass
    static constexpr int kPasses = TX / kRows;
    static_assert(TX % kRows == 0, "whole passes");
};

// the relaxation coefficients and coefficient-set indices of a quad: from the code table
// (CODED: `cw`, the quad's four codes, loaded beforehand) or from the per-cell maps. Each coded
// cell reads its table row as one 16-byte and one 8-byte load (a cell without a code reads row
// 0 first); the rare cells without a code then take their maps in a branch of their own, so
// that the compiler does not turn the row reads into lane-selected 4-byte loads.
template <bool CODED, bool UNIFORM, bool VEL, int NA>
__device__ inline void quad_coef(const DevSim& s, uint32_t c, uint2 cw, F4* ik, F4* b1, F4* b2, F4* a1, F4* a2,
                                 I4& dc) {
    const float* const* ik_m = VEL ? s.ikv : s.ikp;
    const float* const (*a_m)[kNRelax] = VEL ? s.av : s.ap;
    const float* const (*b_m)[kNRelax] = VEL ? s.bv : s.bp;
    if (CODED) {
        const uint32_t cs[4] = {cw.x & 0xffffu, cw.x >> 16, cw.y & 0xffffu, cw.y >> 16};
        int d[4];
        bool esc = false;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const CodedCoef k = coded_coef(VEL ? s.rtab_v : s.rtab_p, cs[e] != kCodeEscape ? cs[e] : 0u);
            ik[0][e] = k.ik;
            a1[0][e] = k.a1;
            a2[0][e] = k.a2;
            b1[0][e] = k.b1;
            b2[0][e] = k.b2;
            d[e] = UNIFORM ? 0 : k.dc;
            esc = esc || cs[e] == kCodeEscape;
        }
        if (esc) {
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                if (cs[e] != kCodeEscape) continue;
                const CodedCoef k = mapped_coef<UNIFORM>(ik_m[0], a_m[0][0], a_m[0][1], b_m[0][0], b_m[0][1],
                                                         s.dcmap, c + e);
                ik[0][e] = k.ik;
                a1[0][e] = k.a1;
                a2[0][e] = k.a2;
                b1[0][e] = k.b1;
                b2[0][e] = k.b2;
                d[e] = UNIFORM ? 0 : k.dc;
            }
        }
        dc = I4{d[0], d[1], d[2], d[3]};
        return;
    }
    dc = UNIFORM ? I4{0, 0, 0, 0} : ldi4(s.dcmap, c);
#pragma unroll
    for (int a = 0; a < NA; ++a) {
        ik[a] = ld4(ik_m[a], c);
        b1[a] = ld4(b_m[a][0], c);
        b2[a] = ld4(b_m[a][1], c);
        a1[a] = ld4(a_m[a][0], c);
        a2[a] = ld4(a_m[a][1], c);
    }
}

// The codes of the quad at row i, column jq of a coded grid, for rows the tile updates (i <
// nx - 8; ny % 4 == 0, so the quad lies in its row); else 0. A tile loads the codes of a lane's
// next row one row ahead: its row gathers then do not wait behind the row's other loads (the
// memory wait counter completes loads in issue order).
template <bool CODED>
__device__ inline uint2 quad_codes(const DevSim& s, int64_t i, int64_t jq) {
    if (!CODED || i >= s.nx - kHalo) return uint2{0u, 0u};
    return ldc4(s.rcode, (uint32_t)(i * s.ny + jq));
}

// LDS tile layout: each staged row of `pitch` floats is split into four planes of pitch / 4
// floats by tile column % 4, each plane holding its columns in order. The lanes of a wavefront
// own consecutive column quads, so when they all read the same element of their quads (at the
// same stencil offset) they touch consecutive words: the LDS serves these single-float reads
// without bank conflicts, where a row-major tile (lanes 4 floats apart) conflicts four ways.
//
// The staged region of one field: NROWS rows x (TW + HL + HR) columns in rows of PITCH floats
// (pitch mod 32 keeps the rows that one half of a wavefront reads on different banks). Each lane owns
// fixed quads of it and issues all of their loads (load) before it stores any (store), so the
// staging takes one memory latency: looping over load-and-store took one per quad, 7 in a row for
// the 23 x 272 tile of a pressure workgroup.
template <int TW, int NROWS_, int HL_, int HR_>
struct Staged {
    static constexpr int NROWS = NROWS_, HL = HL_;
    static constexpr int QPR = (TW + HL_ + HR_) / 4;       // quads per row
    static constexpr int MOD = TW >= 128 ? 0 : TW == 64 ? 16 : 24;
    static constexpr int PITCH = TW >= 128 ? 4 * QPR : (4 * QPR - MOD + 31) / 32 * 32 + MOD;
    static constexpr int PLANE = PITCH / 4;
    static constexpr int NQ = NROWS * QPR;
    static constexpr int NL = (NQ + kLanes - 1) / kLanes;  // quads per lane
    float v[NROWS * PITCH];
};
template <class T>
struct StageRegs {
    F4 q[T::NL];
    // Rows [r0, r0 + NROWS) x columns [j0 - HL, ...) of f; quads outside the grid (no updated cell's
    // stencil reaches one) repeat the nearest one, so that the loads need no branch.
    __device__ inline void load(const float* __restrict__ f, int r0, int j0, int nx, int ny) {
#pragma unroll
        for (int l = 0; l < T::NL; ++l) {
            const int t = min((int)threadIdx.x + l * kLanes, T::NQ - 1);
            const int row = t / T::QPR, qd = t - row * T::QPR;
            const int r = min(max(r0 + row, 0), nx - 1), jj = min(max(j0 - T::HL + 4 * qd, 0), ny - 4);
            q[l] = ld4(f, (uint32_t)(r * ny + jj));
        }
    }
    __device__ inline void store(T& tile) const {
#pragma unroll
        for (int l = 0; l < T::NL; ++l) {
            const int t = threadIdx.x + l * kLanes;
            const int row = t / T::QPR, qd = t - row * T::QPR;
            if (l == T::NL - 1 && t >= T::NQ) continue;
            float* dst = tile.v + row * T::PITCH + qd;
            dst[0] = q[l].x;
            dst[T::PLANE] = q[l].y;
            dst[2 * T::PLANE] = q[l].z;
            dst[3 * T::PLANE] = q[l].w;
        }
    }
};

// Element at row offset dr and column offset dc from tile row `row` of the lane's quad base
// `lb` (= lds + row * pitch + qd): K = hl + e + dc is the column within the quad grid (hl + e
// for the lane's own cell e); every index part is a compile-time constant after unrolling.
template <int PITCH, int HL>
__device__ inline float tl(const float* lb, int dr, int col) {
    const int K = HL + col;  // >= 0 for every offset used
    return lb[dr * PITCH + (K & 3) * (PITCH / 4) + (K >> 2)];
}

// LDS coefficient sets: [set][axis][kCS], or [set][kCS] when both axes share their sets (equal
// spacings; SAME), which halves the table, lets one more workgroup fit on a CU, and lets a cell read
// its weights once for both axes. Each set of 9 weights is padded to 12 floats, so a cell reads
// them as two 16-byte loads and one 4-byte load.
constexpr int kCS = 12;
template <bool UNIFORM, bool SAME>
__device__ inline const float* cset(const float* lds_coef, int dc, int axis) {
    return lds_coef + ((UNIFORM ? 0 : dc) * (SAME ? 1 : 2) + (SAME ? 0 : axis)) * kCS;
}

struct W9 {
    float w[9];
};
__device__ inline W9 weights(const float* c) {
    const F4 a = *reinterpret_cast<const F4*>(c), b = *reinterpret_cast<const F4*>(c + 4);
    return W9{{a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w, c[8]}};
}

// Stage the coefficient sets into LDS (all axes, or axis 0 only when they are the same).
template <bool UNIFORM, bool SAME>
__device__ inline void stage_coef(float* lds_coef, const DevSim& s) {
    constexpr int axes = SAME ? 1 : 2;
    const int n = (UNIFORM ? 1 : s.ndmap) * axes * kNCoef;
    for (int t0 = 0; t0 < n; t0 += 4 * kLanes) {  // four loads in flight a lane
        float v[4];
#pragma unroll
        for (int l = 0; l < 4; ++l) {
            const int t = t0 + l * kLanes + threadIdx.x, set = t / kNCoef, k = t - set * kNCoef;
            v[l] = t < n ? s.coef[(SAME ? set * 2 : set) * kNCoef + k] : 0.f;
        }
#pragma unroll
        for (int l = 0; l < 4; ++l) {
            const int t = t0 + l * kLanes + threadIdx.x, set = t / kNCoef, k = t - set * kNCoef;
            if (t < n) lds_coef[set * kCS + k] = v[l];
        }
    }
}

// The coefficients of one quad as the arithmetic reads them. QuadCoef: each cell its own, in vector
// registers, with its weights from LDS.
template <bool UNIFORM, bool ISO, bool SAME>
struct QuadCoef {
    static constexpr int NA = ISO ? 1 : 2;
    F4 ik_[NA], b1_[NA], b2_[NA], a1_[NA], a2_[NA];
    I4 dc;
    __device__ float ik(int a, int e) const { return ik_[ISO ? 0 : a][e]; }
    __device__ float a1(int a, int e) const { return a1_[ISO ? 0 : a][e]; }
    __device__ float a2(int a, int e) const { return a2_[ISO ? 0 : a][e]; }
    __device__ float b1(int a, int e) const { return b1_[ISO ? 0 : a][e]; }
    __device__ float b2(int a, int e) const { return b2_[ISO ? 0 : a][e]; }
    __device__ W9 w(const DevSim&, const float* lds_coef, int a, int e) const {
        return weights(cset<UNIFORM, SAME>(lds_coef, dc[e], a));
    }
};
// WaveCoef: every cell of the wavefront has the same code, so the row and the weights are read once
// with scalar loads and stay in scalar registers.
template <bool UNIFORM, bool SAME>
struct WaveCoef {
    float ik_, a1_, a2_, b1_, b2_;
    int dc;
    __device__ float ik(int, int) const { return ik_; }
    __device__ float a1(int, int) const { return a1_; }
    __device__ float a2(int, int) const { return a2_; }
    __device__ float b1(int, int) const { return b1_; }
    __device__ float b2(int, int) const { return b2_; }
    __device__ W9 w(const DevSim& s, const float*, int a, int) const {
        const scalar_ptr c = as_scalar(s.coef) + ((UNIFORM ? 0 : dc * 2) + (SAME ? 0 : a)) * kNCoef;
        W9 r;
#pragma unroll
        for (int k = 0; k < kNCoef; ++k) r.w[k] = c[k];
        return r;
    }
    // the values again as the (active) lanes' common ones: across a branch the compiler takes them for
    // per-lane values
    __device__ void rejoin() {
        for (float* f : {&ik_, &a1_, &a2_, &b1_, &b2_}) *f = __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(*f)));
        dc = __builtin_amdgcn_readfirstlane(dc);
    }
    __device__ void load(const float* tab, uint32_t code) {
        const scalar_ptr row = as_scalar(tab) + code * kCodeStride;
        ik_ = row[0];
        a1_ = row[1];
        a2_ = row[2];
        b1_ = row[3];
        b2_ = row[4];
        dc = __float_as_int(row[5]);
    }
};

// velocity: p rows i0-7 .. i0+TX+7, columns j0-8 .. j0+TW+7
template <class S>
struct VelTile {
    using P = Staged<S::TW, S::TX + 15, 8, 8>;
    P p;
};

// operands of one quad of the velocity update
struct VelQuad {
    F4 rho0, rho1, ps1[2], ps2[2], v[2];
    float rho_r;
};

__device__ inline void load_vel_quad(const DevSim& s, VelQuad& o, uint32_t c) {
    o.rho0 = ld4(s.rho, c);
    o.rho1 = ld4(s.rho, c + (uint32_t)s.ny);
    o.rho_r = ld1(s.rho, c + 4);
#pragma unroll
    for (int a = 0; a < 2; ++a) {
        o.ps1[a] = ld4nt(s.psi[a][0], c);
        o.ps2[a] = ld4nt(s.psi[a][1], c);
        o.v[a] = ld4(s.v[a], c);
    }
}

// The velocity update of the quad at element c with coefficients k; lb: its base in the staged p.
template <int PITCH, bool SAME, bool TAPE, class Coef>
__device__ inline void velocity_quad(const DevSim& s, uint32_t c, VelQuad& o, const Coef& k, const float* lb,
                                     const float* lds_coef) {
    const float dt = s.dt;
    auto pa = [&](int e, int dr, int dc_) { return tl<PITCH, 8>(lb, dr, e + dc_); };
    F4 tu[2];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        W9 wv = k.w(s, lds_coef, 0, e);
        {
            float acc = 0.f;
#pragma unroll
            for (int m = 1; m <= 8; ++m) acc = tap(acc, wv.w[m - 1], pa(e, m, 0), pa(e, -(m - 1), 0));
            float tr = 0.f;
            tr += (pa(e, 1, 1) - pa(e, 0, 1)) + (pa(e, 1, -1) - pa(e, 0, -1));
            const float D = __builtin_fmaf(wv.w[8], tr, acc);
            const float q1 = memory_step(k.b1(0, e), o.ps1[0][e], k.a1(0, e), D);
            const float q2 = memory_step(k.b2(0, e), o.ps2[0][e], k.a2(0, e), D);
            o.ps1[0][e] = q1;
            o.ps2[0][e] = q2;
            const float u = corrected(D, k.ik(0, e), q1, q2);
            o.v[0][e] = velocity_step(o.v[0][e], dt, o.rho0[e], o.rho1[e], u);
            if (TAPE) tu[0][e] = u;
        }
        {
            if (!SAME) wv = k.w(s, lds_coef, 1, e);
            float acc = 0.f;
#pragma unroll
            for (int m = 1; m <= 8; ++m) acc = tap(acc, wv.w[m - 1], pa(e, 0, m), pa(e, 0, -(m - 1)));
            float tr = 0.f;
            tr += (pa(e, 1, 1) - pa(e, 1, 0)) + (pa(e, -1, 1) - pa(e, -1, 0));
            const float D = __builtin_fmaf(wv.w[8], tr, acc);
            const float q1 = memory_step(k.b1(1, e), o.ps1[1][e], k.a1(1, e), D);
            const float q2 = memory_step(k.b2(1, e), o.ps2[1][e], k.a2(1, e), D);
            o.ps1[1][e] = q1;
            o.ps2[1][e] = q2;
            const float rho_right = e < 3 ? o.rho0[e + 1] : o.rho_r;
            const float u = corrected(D, k.ik(1, e), q1, q2);
            o.v[1][e] = velocity_step(o.v[1][e], dt, o.rho0[e], rho_right, u);
            if (TAPE) tu[1][e] = u;
        }
    }
#pragma unroll
    for (int a = 0; a < 2; ++a) {
        st4nt(s.psi[a][0], c, o.ps1[a]);
        st4nt(s.psi[a][1], c, o.ps2[a]);
        st4(s.v[a], c, o.v[a]);
        if (TAPE) st4(s.tape_u[a], c, tu[a]);
    }
}

// The velocity update of tile (bx, by) of grid s: columns [bx * TW, bx * TW + TW), rows
// [8 + by * TX, 8 + by * TX + TX). TAPE: also the adjoint tape (DevSim::tape_u). The ghost border is
// two quads wide and ny % 4 == 0, so a quad is updated whole or not at all: its four cells run
// as one straight line of code, which shares the columns that their stencils read (a test per cell
// kept them apart: 144 LDS words a quad and axis pair instead of 93, and no overlap between cells).
template <class S, bool UNIFORM, bool ISO, bool CODED, bool SAME, bool TAPE = false>
__device__ inline void velocity_tile(const DevSim& s, unsigned bx, unsigned by, VelTile<S>& L, float* lds_coef) {
    using T = typename VelTile<S>::P;
    const int64_t nx = s.nx, ny = s.ny;
    const int64_t j0 = (int64_t)bx * S::TW;
    const int64_t i0 = kHalo + (int64_t)by * S::TX;
    const int qd = threadIdx.x % S::kQuads;
    const int ty = threadIdx.x / S::kQuads;
    const int64_t jq = j0 + 4 * qd;  // first column of this lane's quad
    const bool active = jq >= kHalo && jq < ny - kHalo;
    uint2 cw = active ? quad_codes<CODED>(s, i0 + ty, jq) : uint2{0u, 0u};
    StageRegs<T> st;
    st.load(s.p, (int)i0 - 7, (int)j0, (int)nx, (int)ny);
    VelQuad o;
    QuadCoef<UNIFORM, ISO, SAME> kq;
    WaveCoef<UNIFORM, SAME> kw;
    bool wave = false;
    auto load_coef = [&](uint32_t c) {
        uint32_t code = 0;
        wave = CODED && wave_code(cw, &code);
        if (wave) kw.load(s.rtab_v, code);
        else quad_coef<CODED, UNIFORM, true, QuadCoef<UNIFORM, ISO, SAME>::NA>(s, c, cw, kq.ik_, kq.b1_, kq.b2_, kq.a1_, kq.a2_, kq.dc);
    };
    if (active && i0 + ty < nx - kHalo) {
        const uint32_t c = (uint32_t)((i0 + ty) * ny + jq);
        load_vel_quad(s, o, c);
        load_coef(c);
    }
    stage_coef<UNIFORM, SAME>(lds_coef, s);
    st.store(L.p);
    __syncthreads();

    if (!active) return;
#pragma unroll 1
    for (int m = 0; m < S::kPasses; ++m) {
        const int lr = ty + S::kRows * m;  // row within the tile
        const int64_t i = i0 + lr;
        if (i >= nx - kHalo) break;
        const uint32_t c = (uint32_t)(i * ny + jq);
        if (m > 0) {
            load_vel_quad(s, o, c);
            load_coef(c);
        }
        if (m + 1 < S::kPasses) cw = quad_codes<CODED>(s, i + S::kRows, jq);
        // LDS row of tile row lr is lr + 7; column j is tile column j - j0 + 8
        const float* lb = L.p.v + (lr + 7) * T::PITCH + qd;
        if (CODED && __builtin_amdgcn_readfirstlane(wave)) {
            kw.rejoin();
            velocity_quad<T::PITCH, SAME, TAPE>(s, c, o, kw, lb, lds_coef);
        } else {
            velocity_quad<T::PITCH, SAME, TAPE>(s, c, o, kq, lb, lds_coef);
        }
    }
}

// pressure: vx rows i0-8 .. i0+TX+6, columns j0-4 .. j0+TW+3;
//           vy rows i0-1 .. i0+TX, columns j0-8 .. j0+TW+7
template <class S>
struct PreTile {
    using X = Staged<S::TW, S::TX + 15, 4, 4>;
    using Y = Staged<S::TW, S::TX + 2, 8, 8>;
    X x;
    Y y;
};

// operands of one quad of the pressure update
struct PreQuad {
    F4 p, K, ph1[2], ph2[2];
};

__device__ inline void load_pre_quad(const DevSim& s, PreQuad& o, uint32_t c) {
    o.p = ld4(s.p, c);
    o.K = ld4(s.K, c);
#pragma unroll
    for (int a = 0; a < 2; ++a) {
        o.ph1[a] = ld4nt(s.phi[a][0], c);
        o.ph2[a] = ld4nt(s.phi[a][1], c);
    }
}

// The pressure update of the quad at element c; xb, yb: its base in the staged vx and vy.
template <int XP, int YP, bool SAME, bool TAPE, class Coef>
__device__ inline void pressure_quad(const DevSim& s, uint32_t c, PreQuad& o, const Coef& k, const float* xb,
                                     const float* yb, const float* lds_coef) {
    const float dt = s.dt;
    auto xa = [&](int e, int dr, int dc_) { return tl<XP, 4>(xb, dr, e + dc_); };
    auto ya = [&](int e, int dr, int dc_) { return tl<YP, 8>(yb, dr, e + dc_); };
    F4 td;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        float div = 0.f;
        W9 wv = k.w(s, lds_coef, 0, e);
        {
            float acc = 0.f;
#pragma unroll
            for (int m = 1; m <= 8; ++m) acc = tap(acc, wv.w[m - 1], xa(e, m - 1, 0), xa(e, -m, 0));
            float tr = 0.f;
            tr += (xa(e, 0, 1) - xa(e, -1, 1)) + (xa(e, 0, -1) - xa(e, -1, -1));
            const float D = __builtin_fmaf(wv.w[8], tr, acc);
            const float q1 = memory_step(k.b1(0, e), o.ph1[0][e], k.a1(0, e), D);
            const float q2 = memory_step(k.b2(0, e), o.ph2[0][e], k.a2(0, e), D);
            o.ph1[0][e] = q1;
            o.ph2[0][e] = q2;
            div += corrected(D, k.ik(0, e), q1, q2);
        }
        {
            if (!SAME) wv = k.w(s, lds_coef, 1, e);
            float acc = 0.f;
#pragma unroll
            for (int m = 1; m <= 8; ++m) acc = tap(acc, wv.w[m - 1], ya(e, 0, m - 1), ya(e, 0, -m));
            float tr = 0.f;
            tr += (ya(e, 1, 0) - ya(e, 1, -1)) + (ya(e, -1, 0) - ya(e, -1, -1));
            const float D = __builtin_fmaf(wv.w[8], tr, acc);
            const float q1 = memory_step(k.b1(1, e), o.ph1[1][e], k.a1(1, e), D);
            const float q2 = memory_step(k.b2(1, e), o.ph2[1][e], k.a2(1, e), D);
            o.ph1[1][e] = q1;
            o.ph2[1][e] = q2;
            div += corrected(D, k.ik(1, e), q1, q2);
        }
        o.p[e] = pressure_step(o.p[e], dt, o.K[e], div);
        if (TAPE) td[e] = div;
    }
    st4(s.p, c, o.p);
    if (TAPE) st4(s.tape_div, c, td);
#pragma unroll
    for (int a = 0; a < 2; ++a) {
        st4nt(s.phi[a][0], c, o.ph1[a]);
        st4nt(s.phi[a][1], c, o.ph2[a]);
    }
}

// The pressure update of tile (bx, by) of grid s (as velocity_tile; TAPE: DevSim::tape_div).
template <class S, bool UNIFORM, bool ISO, bool CODED, bool SAME, bool TAPE = false>
__device__ inline void pressure_tile(const DevSim& s, unsigned bx, unsigned by, PreTile<S>& L, float* lds_coef) {
    using X = typename PreTile<S>::X;
    using Y = typename PreTile<S>::Y;
    const int64_t nx = s.nx, ny = s.ny;
    const int64_t j0 = (int64_t)bx * S::TW;
    const int64_t i0 = kHalo + (int64_t)by * S::TX;
    const int qd = threadIdx.x % S::kQuads;
    const int ty = threadIdx.x / S::kQuads;
    const int64_t jq = j0 + 4 * qd;
    const bool active = jq >= kHalo && jq < ny - kHalo;
    uint2 cw = active ? quad_codes<CODED>(s, i0 + ty, jq) : uint2{0u, 0u};
    StageRegs<X> sx;
    StageRegs<Y> sy;
    sx.load(s.v[0], (int)i0 - 8, (int)j0, (int)nx, (int)ny);
    sy.load(s.v[1], (int)i0 - 1, (int)j0, (int)nx, (int)ny);
    PreQuad o;
    QuadCoef<UNIFORM, ISO, SAME> kq;
    WaveCoef<UNIFORM, SAME> kw;
    bool wave = false;
    auto load_coef = [&](uint32_t c) {
        uint32_t code = 0;
        wave = CODED && wave_code(cw, &code);
        if (wave) kw.load(s.rtab_p, code);
        else quad_coef<CODED, UNIFORM, false, QuadCoef<UNIFORM, ISO, SAME>::NA>(s, c, cw, kq.ik_, kq.b1_, kq.b2_, kq.a1_, kq.a2_, kq.dc);
    };
    if (active && i0 + ty < nx - kHalo) {
        const uint32_t c = (uint32_t)((i0 + ty) * ny + jq);
        load_pre_quad(s, o, c);
        load_coef(c);
    }
    stage_coef<UNIFORM, SAME>(lds_coef, s);
    sx.store(L.x);
    sy.store(L.y);
    __syncthreads();

    if (!active) return;
#pragma unroll 1
    for (int m = 0; m < S::kPasses; ++m) {
        const int lr = ty + S::kRows * m;
        const int64_t i = i0 + lr;
        if (i >= nx - kHalo) break;
        const uint32_t c = (uint32_t)(i * ny + jq);
        if (m > 0) {
            load_pre_quad(s, o, c);
            load_coef(c);
        }
        if (m + 1 < S::kPasses) cw = quad_codes<CODED>(s, i + S::kRows, jq);
        const float* xb = L.x.v + (lr + 8) * X::PITCH + qd;  // vx(i, .): tile column j - j0 + 4
        const float* yb = L.y.v + (lr + 1) * Y::PITCH + qd;  // vy(i, .): tile column j - j0 + 8
        if (CODED && __builtin_amdgcn_readfirstlane(wave)) {
            kw.rejoin();
            pressure_quad<X::PITCH, Y::PITCH, SAME, TAPE>(s, c, o, kw, xb, yb, lds_coef);
        } else {
            pressure_quad<X::PITCH, Y::PITCH, SAME, TAPE>(s, c, o, kq, xb, yb, lds_coef);
        }
    }
}

// The tile of this workgroup within its shot, in row-major order: each XCD takes a contiguous run of
// them, so that the halo rows that neighbouring tiles stage come from one L2. us a step against the
// launch order: 672^2 cells 17.5 -> 15.0, 1152^2 33.7 -> 32.0, 4256 x 2208 176.5 -> 174.0 (at the
// fastest shape of each).
__device__ inline uint32_t shot_tile() {
    return xcd_order(blockIdx.y * gridDim.x + blockIdx.x, gridDim.x * gridDim.y);
}

template <class S, bool UNIFORM, bool ISO, bool CODED, bool SAME, bool TAPE>
__global__ __launch_bounds__(kLanes) void k_velocity_tile(DevSim batch) {
    __shared__ __attribute__((aligned(16))) VelTile<S> L;
    extern __shared__ __attribute__((aligned(16))) float lds_coef[];
    const uint32_t t = shot_tile();
    velocity_tile<S, UNIFORM, ISO, CODED, SAME, TAPE>(shot_view(batch, blockIdx.z), t % gridDim.x, t / gridDim.x, L, lds_coef);
}

// gs.g non-null: each workgroup then also does the step's source, pressure-release and sensor
// work of its tile (tile shot_tile() of shot blockIdx.z), as the group
// kernels do
template <class S, bool UNIFORM, bool ISO, bool CODED, bool SAME, bool TAPE>
__global__ __launch_bounds__(kLanes) void k_pressure_tile(DevSim batch, GroupStep gs) {
    __shared__ __attribute__((aligned(16))) PreTile<S> L;
    extern __shared__ __attribute__((aligned(16))) float lds_coef[];
    const uint32_t t = shot_tile();
    TileWork w{};
    if (gs.g) {
        const GroupBoundary& e = gs.g[blockIdx.z];
        w = tile_work(e, t, e.step0 + gs.it + (gs.base ? *gs.base : 0));
    }
    pressure_tile<S, UNIFORM, ISO, CODED, SAME, TAPE>(shot_view(batch, blockIdx.z), t % gridDim.x, t / gridDim.x, L, lds_coef);
    if (!gs.g) return;
    __syncthreads();
    tile_boundary(w);
}

// grouped launches: the tiles of several grids (different sizes and media, isotropic
// relaxation) in one 1D launch. FAST: every grid reads coded coefficients and has the same weights on
// both axes; otherwise each grid takes the coded or the per-cell-map path by its own handle, with the
// sets of both axes staged.
template <class S, bool FAST>
__global__ __launch_bounds__(kLanes) void k_velocity_tile_group(const GroupTile* __restrict__ t, int n) {
    __shared__ __attribute__((aligned(16))) VelTile<S> L;
    extern __shared__ __attribute__((aligned(16))) float lds_coef[];
    const uint32_t gid = xcd_order(blockIdx.x, gridDim.x);
    const int m = group_entry(t, n, gid);
    const DevSim s = t[m].s;
    const unsigned local = gid - t[m].start;
    const unsigned bx = local % t[m].gx, by = local / t[m].gx;
    if (FAST) velocity_tile<S, false, true, true, true>(s, bx, by, L, lds_coef);
    else if (s.rcode) velocity_tile<S, false, true, true, false>(s, bx, by, L, lds_coef);
    else velocity_tile<S, false, true, false, false>(s, bx, by, L, lds_coef);
}

// the pressure update of the tile, then its share of the step's boundary work (gs.g non-null)
template <class S, bool FAST>
__global__ __launch_bounds__(kLanes) void k_pressure_tile_group(const GroupTile* __restrict__ t, int n, GroupStep gs) {
    __shared__ __attribute__((aligned(16))) PreTile<S> L;
    extern __shared__ __attribute__((aligned(16))) float lds_coef[];
    const uint32_t gid = xcd_order(blockIdx.x, gridDim.x);
    const int m = group_entry(t, n, gid);
    const DevSim s = t[m].s;
    const unsigned local = gid - t[m].start;
    const unsigned bx = local % t[m].gx, by = local / t[m].gx;
    TileWork w{};
    if (gs.g) w = tile_work(gs.g[m], local, gs.g[m].step0 + gs.it + (gs.base ? *gs.base : 0));
    if (FAST) pressure_tile<S, false, true, true, true>(s, bx, by, L, lds_coef);
    else if (s.rcode) pressure_tile<S, false, true, true, false>(s, bx, by, L, lds_coef);
    else pressure_tile<S, false, true, false, false>(s, bx, by, L, lds_coef);
    if (!gs.g) return;
    __syncthreads();
    tile_boundary(w);
}

template <class S, bool FAST>
hipError_t launch_group_tile(const GroupTile* t, int n, uint32_t blocks, int lds, bool velocity, const GroupStep& gs,
                             hipStream_t st) {
    if (velocity) hipLaunchKernelGGL((k_velocity_tile_group<S, FAST>), dim3(blocks), dim3(kLanes), lds, st, t, n);
    else hipLaunchKernelGGL((k_pressure_tile_group<S, FAST>), dim3(blocks), dim3(kLanes), lds, st, t, n, gs);
    return hipGetLastError();
}

template <class S>
hipError_t launch_group_tile_any(const GroupTile* t, int n, uint32_t blocks, int lds, bool fast, bool velocity,
                                 const GroupStep& gs, hipStream_t st) {
    return fast ? launch_group_tile<S, true>(t, n, blocks, lds, velocity, gs, st)
                : launch_group_tile<S, false>(t, n, blocks, lds, velocity, gs, st);
}

template <class S, bool UNIFORM, bool ISO, bool CODED, bool SAME, bool TAPE>
void launch_tile_kernel(const DevSim& s, bool velocity, const GroupStep& gs, hipStream_t st) {
    const int lds = (UNIFORM ? 1 : s.ndmap) * (SAME ? 1 : 2) * kCS * 4;
    const int64_t rows = s.nx - 2 * kHalo;
    const dim3 g((unsigned)((s.ny + S::TW - 1) / S::TW), (unsigned)((rows + S::TX - 1) / S::TX), (unsigned)s.nshots);
    if (velocity) hipLaunchKernelGGL((k_velocity_tile<S, UNIFORM, ISO, CODED, SAME, TAPE>), g, dim3(kLanes), lds, st, s);
    else hipLaunchKernelGGL((k_pressure_tile<S, UNIFORM, ISO, CODED, SAME, TAPE>), g, dim3(kLanes), lds, st, s, gs);
}

template <class S, bool SAME, bool TAPE>
hipError_t launch_tile_same(const DevSim& s, bool velocity, const GroupStep& gs, hipStream_t st) {
    const bool u = s.ndmap == 1, coded = s.isotropic && s.rcode;
    if (u && coded) launch_tile_kernel<S, true, true, true, SAME, TAPE>(s, velocity, gs, st);
    else if (u && s.isotropic) launch_tile_kernel<S, true, true, false, SAME, TAPE>(s, velocity, gs, st);
    else if (u) launch_tile_kernel<S, true, false, false, SAME, TAPE>(s, velocity, gs, st);
    else if (coded) launch_tile_kernel<S, false, true, true, SAME, TAPE>(s, velocity, gs, st);
    else if (s.isotropic) launch_tile_kernel<S, false, true, false, SAME, TAPE>(s, velocity, gs, st);
    else launch_tile_kernel<S, false, false, false, SAME, TAPE>(s, velocity, gs, st);
    return hipGetLastError();
}

template <class S, bool TAPE = false>
hipError_t launch_tile(const DevSim& s, bool velocity, const GroupStep& gs, hipStream_t st) {
    return s.coef_axes_same ? launch_tile_same<S, true, TAPE>(s, velocity, gs, st)
                            : launch_tile_same<S, false, TAPE>(s, velocity, gs, st);
}

}  // namespace

// The tile shape that each row count stands for.
using Tile8 = Shape<128, 8>;
using Tile16 = Shape<128, 16>;
using Tile32 = Shape<64, 32>;

int tile2d_width(int rows) {
    return rows == 8 ? Tile8::TW : rows == 32 ? Tile32::TW : Tile16::TW;
}

// The most sound speeds (coefficient sets) the tiled kernels stage: two padded sets (one per
// axis, unequal spacings) of every sound speed next to the largest tile must fit in the 160 KiB of
// LDS a workgroup can have on gfx950, for both kernels and for the group kernels (which stage the
// largest member's sets next to the same tiles).
constexpr int kMaxTileSets = 768;
constexpr size_t kLdsPerWorkgroup = size_t(160) << 10;
static_assert(sizeof(PreTile<Tile32>) + size_t(2) * kMaxTileSets * kCS * sizeof(float) <= kLdsPerWorkgroup,
              "tiled pressure kernel: 32-row tile plus the staged sets exceeds the LDS of a workgroup");
static_assert(sizeof(VelTile<Tile32>) + size_t(2) * kMaxTileSets * kCS * sizeof(float) <= kLdsPerWorkgroup,
              "tiled velocity kernel: 32-row tile plus the staged sets exceeds the LDS of a workgroup");

bool tile2d_supported(const DevSim& s) {
    return !s.aexp && s.ndim == 2 && s.ny % 4 == 0 && s.ndmap <= kMaxTileSets && s.nx * s.ny < ((int64_t)1 << 30);
}

unsigned group_tile_rows(int64_t nx, int rows) { return (unsigned)((nx - 2 * kHalo + rows - 1) / rows); }

hipError_t launch_group_tile2d(const GroupTile* t, int n, uint32_t blocks, int rows, int coef_sets, bool fast,
                               bool velocity, const GroupStep& gs, hipStream_t st) {
    if (n <= 0 || blocks == 0) return hipSuccess;
    const int lds = coef_sets * kCS * 4;  // the largest member's staged sets (stage_coef)
    switch (rows) {
        case 8: return launch_group_tile_any<Tile8>(t, n, blocks, lds, fast, velocity, gs, st);
        case 32: return launch_group_tile_any<Tile32>(t, n, blocks, lds, fast, velocity, gs, st);
        default: return launch_group_tile_any<Tile16>(t, n, blocks, lds, fast, velocity, gs, st);
    }
}

hipError_t load_tile2d_code() {
    hipFuncAttributes a;
    return hipFuncGetAttributes(&a, reinterpret_cast<const void*>(&k_velocity_tile_group<Tile8, true>));
}

hipError_t launch_tile2d(const DevSim& s, const LaunchCfg& cfg, bool velocity, const GroupStep& gs, hipStream_t st) {
    if (s.tape_div) return launch_tile<Tile8, true>(s, velocity, gs, st);  // taped steps: 8-row tiles
    switch (cfg.chunk) {
        case 8: return launch_tile<Tile8>(s, velocity, gs, st);
        case 32: return launch_tile<Tile32>(s, velocity, gs, st);
        default: return launch_tile<Tile16>(s, velocity, gs, st);
    }
}

}  // namespace fw
