// The adjoint sweep of a 3D grid on bricks (geometry and staging: fw_brick.h; the recursion:
// fw_kernels_adjoint.hip): the transposed gathers fused with the pointwise steps that follow them.
//   k_adj_velocity_brick  lambda_v_a += (D-_a)^T H_a, then the velocity transposed
//   k_adj_pressure_brick  lambda_p += sum_a (D+_a)^T G_a, then the next (earlier) step's sparse part and
//                         pressure transposed
// Each was two or three per-cell launches, whose gathers read every neighbour's set index and weights from
// memory (55 cells by three components): us a reverse step, per-cell -> bricks, with 13 sound speeds:
//   136 x 120 x 112  203 -> 140      100 x 88 x 90  109 -> 69      64 x 64 x 64  37.0 -> 28.8
// one sound speed 136 -> 116, 71.7 -> 59.2, 27.1 -> 23.7; exponential model 175 -> 111 at the first size.
// What bounds it: the traffic of the pointwise parts (59 fields of 4 bytes a cell read and written: 81 us
// at the first size at 6 TB/s), then the load, compute and store phases of three workgroups a CU.
// Measured and left out: the pointwise operands loaded before the staging is waited for (144); a pass over
// the brick for each set in its arms, the other sets' cells staged as zeros (177; 64 x 64 x 64: 80.7).
//
// A gather weighs each neighbour by the neighbour's own coefficient set. With one set of weights w,
// (D-_a)^T is minus the forward derivative and (D+_a)^T minus the backward one, so the staging and the
// derivative are the forward kernels', with scalar weights. A brick whose arms hold cells of several
// sets (w.sets) looks the weights up in LDS by the cells' sets.
#include "fw_brick.h"

namespace fw {

namespace {

struct SetWeights {
    float weight[kNCoef];
    __device__ float w(int, int m) const { return weight[m]; }
};

constexpr uint32_t kMixedSets = 0xffffffffu;

// The derivative of component A as derivative() computes it, each neighbour weighed by its own set:
// `table` holds the sets' weights in LDS, dc8 the cells' sets.
template <int A, int SH>
__device__ __forceinline__ void mixed_derivative(const DevSim& s, const uint8_t* dc8, const Brick& b, const Arms<SH>& lds,
                                                 const float* table, F4& D) {
    const int at = b.row * R + 4 * b.quad;
    // the sets of the quad at (dx, dy, z) from this lane's
    auto sets = [&](int dx, int dy, int z) {
        return *reinterpret_cast<const uint32_t*>(dc8 + (b.c + (uint32_t)(dx * (int)s.sx + dy * (int)s.sy + z)));
    };
    // D[e] += weight m of set byte qe of q, times v
    auto add = [&](int e, uint32_t q, int qe, int m, float v) {
        D[e] = __builtin_fmaf(table[((q >> (8 * qe)) & 0xffu) * kNCoef + m], v, D[e]);
    };
    auto quad = [&](uint32_t q, int m, const F4& v, float sign) {
#pragma unroll
        for (int e = 0; e < 4; ++e) add(e, q, e, m, sign * v[e]);
    };
    // the cells e + 1 and e - 1 of a quad with neighbours l and r
    auto beside = [&](uint32_t q, uint32_t ql, uint32_t qr, const F4& v, float l, float r, float sign) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            add(e, e < 3 ? q : qr, e < 3 ? e + 1 : 0, 8, sign * after(v, r, e));
            add(e, e > 0 ? q : ql, e > 0 ? e - 1 : 3, 8, sign * before(v, l, e));
        }
    };
    if constexpr (A == 0) {
        const float* X = lds.X + 4 * threadIdx.x + 8 * BY * BZ;  // the plane SH
#pragma unroll
        for (int m = 1; m <= 8; ++m) {
            quad(sets(m - 1 + SH, 0, 0), m - 1, lds4(X + (m - 1) * BY * BZ), 1.f);
            quad(sets(SH - m, 0, 0), m - 1, lds4(X - m * BY * BZ), -1.f);
        }
        const float *F = lds.F + (b.wave + 1) * 2 * BZ + 4 * b.quad, *G = lds.G + ((b.wave + 1) * BY + b.row) * 2;
        const bool last = b.row == BY - 1, first = b.row == 0, left = b.quad == 0, right = b.quad == BZ / 4 - 1;
        quad(sets(SH, 1, 0), 8, lds4(last ? F + BZ : X + BZ), 1.f);
        quad(sets(SH - 1, 1, 0), 8, lds4(last ? F - BZ : X - BY * BZ + BZ), -1.f);
        quad(sets(SH, -1, 0), 8, lds4(first ? F : X - BZ), 1.f);
        quad(sets(SH - 1, -1, 0), 8, lds4(first ? F - 2 * BZ : X - BY * BZ - BZ), -1.f);
        beside(sets(SH, 0, 0), sets(SH, 0, -4), sets(SH, 0, 4), lds4(X), *(left ? G : X - 1), *(right ? G + 1 : X + 4), 1.f);
        beside(sets(SH - 1, 0, 0), sets(SH - 1, 0, -4), sets(SH - 1, 0, 4), lds4(X - BY * BZ),
               *(left ? G - 2 * BY : X - BY * BZ - 1), *(right ? G - 2 * BY + 1 : X - BY * BZ + 4), -1.f);
    } else if constexpr (A == 1) {
        const float* Y = lds.Y + YRows<SH>::at(b.wave) + at + SH * R;
        const float *Yp = lds.Y + YRows<SH>::at(b.wave + 1) + at + SH * R, *Ym = lds.Y + YRows<SH>::at(b.wave - 1) + at + SH * R;
#pragma unroll
        for (int m = 1; m <= 8; ++m) {
            quad(sets(0, m - 1 + SH, 0), m - 1, lds4(Y + (m - 1) * R), 1.f);
            quad(sets(0, SH - m, 0), m - 1, lds4(Y - m * R), -1.f);
        }
        quad(sets(1, SH, 0), 8, lds4(Yp), 1.f);
        quad(sets(1, SH - 1, 0), 8, lds4(Yp - R), -1.f);
        quad(sets(-1, SH, 0), 8, lds4(Ym), 1.f);
        quad(sets(-1, SH - 1, 0), 8, lds4(Ym - R), -1.f);
        beside(sets(0, SH, 0), sets(0, SH, -4), sets(0, SH, 4), lds4(Y), Y[-1], Y[4], 1.f);
        beside(sets(0, SH - 1, 0), sets(0, SH - 1, -4), sets(0, SH - 1, 4), lds4(Y - R), Y[-R - 1], Y[-R + 4], -1.f);
    } else {
        const float *Z = lds.Z + ZRows::at(b.wave) + at, *Zp = lds.Z + ZRows::at(b.wave + 1) + at, *Zm = lds.Z + ZRows::at(b.wave - 1) + at;
        float z[20];
        z_arm(Z, lds.E + (b.wave * BY + b.row) * kEnds, b.quad, lds4(Z), z);
        uint32_t q[5];
#pragma unroll
        for (int i = 0; i < 5; ++i) q[i] = sets(0, 0, 4 * i - 8);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
#pragma unroll
            for (int m = 1; m <= 8; ++m) {
                const int hi = 8 + SH + e + m - 1, lo = 8 + SH + e - m;
                add(e, q[hi / 4], hi % 4, m - 1, z[hi]);
                add(e, q[lo / 4], lo % 4, m - 1, -z[lo]);
            }
        }
        // the cells e + SH and e + SH - 1 of the rows beside
        constexpr int side = SH ? 4 : -1;
        auto row = [&](int dx, int dy, const float* v) {
            const uint32_t r = sets(dx, dy, 0), t = sets(dx, dy, SH ? 4 : -4);
            const F4 c = lds4(v);
            const float x = v[side];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                if (SH) {
                    add(e, e < 3 ? r : t, e < 3 ? e + 1 : 0, 8, after(c, x, e));
                    add(e, r, e, 8, -c[e]);
                } else {
                    add(e, r, e, 8, c[e]);
                    add(e, e > 0 ? r : t, e > 0 ? e - 1 : 3, 8, -before(c, x, e));
                }
            }
        };
        row(1, 0, Zp);
        row(-1, 0, Zm);
        row(0, 1, Z + R);
        row(0, -1, Z - R);
    }
}

// Stages the arms of the components f; D[a * STEP] += minus the gather of component a.
template <int SH, bool UNI, int STEP>
__device__ __forceinline__ void gather(const DevSim& s, const AdjView& w, const Brick& b, uint32_t tile, const float* const (&f)[3],
                                       Arms<SH>& lds, float* table, F4* D) {
    uint32_t set = 0;
    if (!UNI) {
        set = (uint32_t)__builtin_amdgcn_readfirstlane(w.sets[tile]);
        if (set == kMixedSets)
            for (int t = threadIdx.x; t < s.ndmap * kNCoef; t += 256) table[t] = s.coef[t / kNCoef * 3 * kNCoef + t % kNCoef];
    }
    {
        ArmQuads q;
        load_arms<SH>(s, b, [&](int a, uint64_t c0, uint32_t c) { return ld4(f[a] + c0, c); }, q);
        put_arms<SH>(b, q, lds);
    }
    __syncthreads();
    if (b.n <= 0) return;
    if (UNI || set != kMixedSets) {
        SetWeights k;
        const scalar_ptr p = as_scalar(s.coef) + set * 3 * kNCoef;
#pragma unroll
        for (int m = 0; m < kNCoef; ++m) k.weight[m] = p[m];
        derivative<0, SH>(b, lds, k, D[0]);
        derivative<1, SH>(b, lds, k, D[STEP]);
        derivative<2, SH>(b, lds, k, D[2 * STEP]);
    } else {
        mixed_derivative<0, SH>(s, w.dc8, b, lds, table, D[0]);
        mixed_derivative<1, SH>(s, w.dc8, b, lds, table, D[STEP]);
        mixed_derivative<2, SH>(s, w.dc8, b, lds, table, D[2 * STEP]);
    }
}

// The coefficients of the quad's cells; from the codes alone (bricks are coded or exponential).
template <bool VEL>
struct QuadCoefs {
    CodedCoef q[4];
    __device__ QuadCoefs(const DevSim& s, uint32_t c) {
        const uint2 cw = ldc4(s.rcode, c);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const uint32_t code = ((e < 2 ? cw.x : cw.y) >> (16 * (e & 1))) & 0xffffu;
            q[e] = coded_coef(VEL ? s.rtab_v : s.rtab_p, code);
        }
    }
};

// One memory variable's adjoint: lam + t to `tot`, b (lam + t) stored; returns a (lam + t) added to g.
__device__ __forceinline__ float memory_adjoint(float& lam, float t, float a, float b, float g) {
#pragma clang fp contract(off)
    const float tot = lam + t;
    lam = b * tot;
    return __builtin_fmaf(a, tot, g);
}

template <bool UNI, bool EXPO>
__global__ __launch_bounds__(256) void k_adj_velocity_brick(DevSim s, AdjView w, uint32_t nby, uint32_t nbz) {
    __shared__ Arms<1> lds;
    extern __shared__ float table[];
    const uint32_t tile = brick_number(true);
    const Brick b = brick_of(s, tile, nby, nbz);
    const float* const H[3] = {w.H[0], w.H[1], w.H[2]};
    F4 D[3] = {};
    gather<1, UNI, 1>(s, w, b, tile, H, lds, table, D);
    if (b.n <= 0) return;
    const uint32_t c = b.c;
    const F4 rho = ld4(s.rho, c);
    const float rho_z = ld1(s.rho, c + 4);
    F4 A{};
    if (EXPO) A = ld4(s.aexp, c);
    auto body = [&](const CodedCoef* kc) {
#pragma unroll
        for (int a = 0; a < 3; ++a) {
            F4 nu = ld4(w.lv[a], c), g, q1{}, q2{}, rn{};
            const F4 u = ld4(w.tu[a], c);
            F4 grb = ld4(w.gRb[a], c);
            if (a < 2) rn = ld4(s.rho, c + (uint32_t)(a == 0 ? s.sx : s.sy));
            if (!EXPO) {
                q1 = ld4(w.lpsi[a][0], c);
                q2 = ld4(w.lpsi[a][1], c);
            }
#pragma unroll
            for (int e = 0; e < 4; ++e) {
#pragma clang fp contract(off)
                nu[e] = nu[e] - D[a][e];
                const float rb = 0.5f * (rho[e] + (a < 2 ? rn[e] : after(rho, rho_z, e)));
                const float beta = s.dt / rb;
                grb[e] = __builtin_fmaf(nu[e] * u[e], s.dt / (rb * rb), grb[e]);
                if (EXPO) {
                    g[e] = -A[e] * beta * nu[e];
                    nu[e] = A[e] * nu[e];
                    continue;
                }
                const float t = -beta * nu[e];
                g[e] = t * kc[e].ik;
                g[e] = memory_adjoint(q1[e], t, kc[e].a1, kc[e].b1, g[e]);
                g[e] = memory_adjoint(q2[e], t, kc[e].a2, kc[e].b2, g[e]);
            }
            if (!EXPO) {
                store_quad<false>(w.lpsi[a][0], c, q1, b.n);
                store_quad<false>(w.lpsi[a][1], c, q2, b.n);
            }
            store_quad<false>(w.lv[a], c, nu, b.n);
            store_quad<false>(w.G[a], c, g, b.n);
            store_quad<false>(w.gRb[a], c, grb, b.n);
        }
    };
    if constexpr (EXPO) {
        body(nullptr);
    } else {
        const QuadCoefs<true> kc(s, c);
        body(kc.q);
    }
}

// what a launch does: the gather alone, the gather and the next step's start, that start alone (its sparse
// part is then k_adj_sparse's)
enum { kGather = 0, kGatherNext = 1, kStart = 2 };

template <bool UNI, bool EXPO, int DO>
__global__ __launch_bounds__(256, 3) void k_adj_pressure_brick(DevSim s, AdjView w, AdjNext nx, uint32_t nby, uint32_t nbz) {
    __shared__ Arms<0> lds;
    extern __shared__ float table[];
    const uint32_t tile = brick_number(true);
    const Brick b = brick_of(s, tile, nby, nbz);
    F4 D{};
    if constexpr (DO != kStart) {
        const float* const G[3] = {w.G[0], w.G[1], w.G[2]};
        gather<0, UNI, 0>(s, w, b, tile, G, lds, table, &D);
    }
    if (b.n <= 0) return;
    const uint32_t c = b.c;
    F4 mu = ld4(w.lp, c);
#pragma unroll
    for (int e = 0; e < 4; ++e) mu[e] = mu[e] - D[e];
    if constexpr (DO == kGather) {
        store_quad<false>(w.lp, c, mu, b.n);
        return;
    }
    if constexpr (DO == kGatherNext) {
        const uint32_t kind = *reinterpret_cast<const uint32_t*>(nx.kind + c);
        if (kind) {
#pragma unroll
            for (int e = 0; e < 4; ++e) mu[e] = next_mu(nx, (int64_t)c + e, (kind >> (8 * e)) & 0xffu, mu[e]);
        }
    }
    const F4 K = ld4(s.K, c), div = ld4(w.tdiv, c);
    F4 gk = ld4(w.gK, c), t;
    if constexpr (EXPO) {
        const F4 A = ld4(s.aexp, c);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
#pragma clang fp contract(off)
            t[e] = -A[e] * s.dt * K[e] * mu[e];
            gk[e] = __builtin_fmaf(mu[e] * (-A[e] * s.dt), div[e], gk[e]);
            mu[e] = A[e] * mu[e];
        }
#pragma unroll
        for (int a = 0; a < 3; ++a) store_quad<false>(w.H[a], c, t, b.n);
        store_quad<false>(w.lp, c, mu, b.n);
    } else {
        const QuadCoefs<false> kc(s, c);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
#pragma clang fp contract(off)
            t[e] = -s.dt * K[e] * mu[e];
            gk[e] = __builtin_fmaf(mu[e] * (-s.dt), div[e], gk[e]);
        }
#pragma unroll
        for (int a = 0; a < 3; ++a) {
            F4 q1 = ld4(w.lphi[a][0], c), q2 = ld4(w.lphi[a][1], c), h;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                h[e] = t[e] * kc.q[e].ik;
                h[e] = memory_adjoint(q1[e], t[e], kc.q[e].a1, kc.q[e].b1, h[e]);
                h[e] = memory_adjoint(q2[e], t[e], kc.q[e].a2, kc.q[e].b2, h[e]);
            }
            store_quad<false>(w.lphi[a][0], c, q1, b.n);
            store_quad<false>(w.lphi[a][1], c, q2, b.n);
            store_quad<false>(w.H[a], c, h, b.n);
        }
        if (DO == kGatherNext) store_quad<false>(w.lp, c, mu, b.n);
    }
    store_quad<false>(w.gK, c, gk, b.n);
}

// The set of the updated cells in each brick's arms, or kMixedSets.
__global__ __launch_bounds__(256) void k_adj_brick_sets(DevSim s, const uint8_t* dc8, uint32_t nby, uint32_t nbz, uint32_t* sets) {
    __shared__ uint32_t least, most;
    const Brick b = brick_of(s, blockIdx.x, nby, nbz);
    if (threadIdx.x == 0) {
        least = 255;
        most = 0;
    }
    __syncthreads();
    uint32_t lo = 255, hi = 0;
    for (int a = 0; a < 3; ++a) {
        const int ex = a == 0 ? 8 : 1, ey = a == 1 ? 8 : 1, ez = a == 2 ? 8 : 1;
        const int wy = BY + 2 * ey, wz = BZ + 2 * ez, n = (BX + 2 * ex) * wy * wz;
        for (int t = threadIdx.x; t < n; t += 256) {
            const int i = b.i0 - ex + t / (wy * wz), j = b.j0 - ey + t / wz % wy, k = b.k0 - ez + t % wz;
            if (i < kHalo || i >= (int)s.nx - kHalo || j < kHalo || j >= (int)s.ny - kHalo || k < kHalo || k >= (int)s.nz - kHalo)
                continue;
            const uint32_t set = dc8[(uint32_t)i * (uint64_t)s.sx + (uint32_t)(j * (int)s.sy + k)];
            lo = min(lo, set);
            hi = max(hi, set);
        }
    }
    atomicMin(&least, lo);
    atomicMax(&most, hi);
    __syncthreads();
    if (threadIdx.x == 0) sets[blockIdx.x] = least == most ? least : kMixedSets;
}

size_t table_bytes(const DevSim& s) { return s.ndmap == 1 ? 0 : (size_t)s.ndmap * kNCoef * sizeof(float); }

dim3 bricks_of(const BrickGrid& g) { return dim3((unsigned)(g.nx * g.ny * g.nz)); }

template <int DO>
void launch_pressure_bricks(const DevSim& s, const AdjView& w, const AdjNext& nx, hipStream_t st) {
    const BrickGrid g = brick_grid(s);
    const uint32_t ny = (uint32_t)g.ny, nz = (uint32_t)g.nz;
    const dim3 n = bricks_of(g);
    const size_t lds = DO == kStart ? 0 : table_bytes(s);
    if (s.ndmap == 1) {
        if (s.aexp) hipLaunchKernelGGL((k_adj_pressure_brick<true, true, DO>), n, dim3(256), lds, st, s, w, nx, ny, nz);
        else hipLaunchKernelGGL((k_adj_pressure_brick<true, false, DO>), n, dim3(256), lds, st, s, w, nx, ny, nz);
    } else {
        if (s.aexp) hipLaunchKernelGGL((k_adj_pressure_brick<false, true, DO>), n, dim3(256), lds, st, s, w, nx, ny, nz);
        else hipLaunchKernelGGL((k_adj_pressure_brick<false, false, DO>), n, dim3(256), lds, st, s, w, nx, ny, nz);
    }
}

}  // namespace

bool adj_bricks_supported(const DevSim& s) { return brick_supported(s) && s.ndmap <= kAdjBrickSets; }

hipError_t launch_adj_brick_sets(const DevSim& s, const uint8_t* dc8, uint32_t* sets, hipStream_t st) {
    const BrickGrid g = brick_grid(s);
    hipLaunchKernelGGL(k_adj_brick_sets, bricks_of(g), dim3(256), 0, st, s, dc8, (uint32_t)g.ny, (uint32_t)g.nz, sets);
    return hipGetLastError();
}

hipError_t launch_adj_start_bricks(const DevSim& s, const AdjView& w, hipStream_t st) {
    launch_pressure_bricks<kStart>(s, w, AdjNext{}, st);
    return hipGetLastError();
}

hipError_t launch_adj_rest_bricks(const DevSim& s, const AdjView& w, const AdjNext* next, hipStream_t st) {
    const BrickGrid g = brick_grid(s);
    const uint32_t ny = (uint32_t)g.ny, nz = (uint32_t)g.nz;
    const dim3 n = bricks_of(g);
    const size_t lds = table_bytes(s);
    if (s.ndmap == 1) {
        if (s.aexp) hipLaunchKernelGGL((k_adj_velocity_brick<true, true>), n, dim3(256), lds, st, s, w, ny, nz);
        else hipLaunchKernelGGL((k_adj_velocity_brick<true, false>), n, dim3(256), lds, st, s, w, ny, nz);
    } else {
        if (s.aexp) hipLaunchKernelGGL((k_adj_velocity_brick<false, true>), n, dim3(256), lds, st, s, w, ny, nz);
        else hipLaunchKernelGGL((k_adj_velocity_brick<false, false>), n, dim3(256), lds, st, s, w, ny, nz);
    }
    if (!next) {
        launch_pressure_bricks<kGather>(s, w, AdjNext{}, st);
        return hipGetLastError();
    }
    AdjView wn = w;  // the next step's pressure transposed reads its own tape
    wn.tdiv = next->tdiv;
    launch_pressure_bricks<kGatherNext>(s, wn, *next, st);
    return hipGetLastError();
}

}  // namespace fw
