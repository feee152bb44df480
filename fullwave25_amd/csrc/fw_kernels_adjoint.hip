// Adjoint (reverse-mode) kernels: one time step of the update transposed.
//
// The forward step is, per active cell c and axis a (h_a folded into the coefficients):
//   velocity:  g_a = D+_a p,  psi' = b psi + a g_a,  u_a = g_a / kappa + sum psi',
//              v_a' = v_a - beta_a u_a
//   pressure:  h_a = D-_a v_a',  phi' = b phi + a h_a,  div = sum_a (h_a / kappa + sum phi'),
//              p' = p - dt K div
//   then p'[source] = signal, p'[air] = 0, and the sensors record p'
// (the exponential model: u_a = A g_a, v_a' = A v_a - beta_a u_a; div = sum_a h_a,
// p' = A (p - dt K div)), with beta_a = dt / rho_bar_a. The forward kernels write u_a and div
// of every step to a tape (DevSim::tape_u, tape_div): that is all the sweep needs of the forward
// state. Going back through step n with the adjoint state lambda of the state after the step:
//   1. lambda_p[sensor] += dL/d record, then lambda_p[source] = lambda_p[air] = 0 (k_adj_sparse;
//      those values were overwritten)
//   2. pressure transposed (k_adj_pressure): t = -dt K mu, mu = lambda_p;
//        lambda_phi_tot = lambda_phi + t, H_a = t / kappa + sum a lambda_phi_tot,
//        lambda_phi = b lambda_phi_tot, dL/dK += mu * (-dt) * div
//   3. lambda_v_a += (D-_a)^T H_a   (gather form)
//   4. velocity transposed (k_adj_velocity): nu = lambda_v_a;
//        lambda_psi_tot = lambda_psi - beta nu, G_a = -beta nu / kappa + sum a lambda_psi_tot,
//        lambda_psi = b lambda_psi_tot, dL/d rho_bar_a += nu * u_a * dt / rho_bar^2
//   5. lambda_p += sum_a (D+_a)^T G_a   (gather form)
// The coefficient sets (dcmap) are constants. The transposed stencils gather: the value at x
// collects every active cell whose stencil reads x, with that cell's coefficients. In 2D, steps
// 3 and 4 run as one tiled kernel (the gather yields nu of its own cell, which step 4 needs
// alone) and step 5 as another, which also runs steps 1 and 2 of the next (earlier) step for its
// cells when that step's tape is held (they need lambda_p of the cell alone); in 3D the same on bricks
// (fw_kernels_adjoint3d.hip); elsewhere each step is its own per-cell kernel.
#include <algorithm>
#include <cstdlib>
#include <cstring>
#include <type_traits>

#include "fw_internal.h"

namespace fw {

namespace {

template <int ND>
__device__ inline bool adj_cell(const DevSim& s, int64_t& i, int64_t& j, int64_t& k) {
    if (ND == 2) {
        k = 0;
        j = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
        i = (int64_t)blockIdx.y * blockDim.y + threadIdx.y;
        return i >= kHalo && i < s.nx - kHalo && j >= kHalo && j < s.ny - kHalo;
    }
    k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    j = (int64_t)blockIdx.y * blockDim.y + threadIdx.y;
    i = blockIdx.z;
    return i >= kHalo && i < s.nx - kHalo && j >= kHalo && j < s.ny - kHalo && k >= kHalo && k < s.nz - kHalo;
}

// The coefficient set of cell c on axis a. UNI: one sound speed (ndmap == 1), the same set
// everywhere, so the gathers skip the per-neighbour dcmap load.
template <bool UNI>
__device__ inline const float* wts(const DevSim& s, int64_t c, int nd, int a) {
    if (UNI) return s.coef + a * kNCoef;
    return s.coef + ((int64_t)s.dcmap[c] * nd + a) * kNCoef;
}

// Records, then the overwritten points, of one step (see AdjSparse). One thread per distinct
// sensor voxel sums its sensors' weights; a voxel that the same step zeroes keeps no record, so
// no two threads write one address.
__global__ __launch_bounds__(256) void k_adj_sparse(float* lp, const float* grow, AdjSparse sp, int injecting) {
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (grow && t < sp.nvox) {
        const int m = sp.vmask[t];
        if (!(m == 1 || (m == 2 && injecting))) {
            float acc = 0.f;
            for (int32_t q = sp.first[t]; q < sp.first[t + 1]; ++q) acc += grow[sp.order[q]];
            lp[sp.vox[t]] += acc;
        }
    }
    if (injecting && t < sp.nsrc && sp.src_lin[t] >= 0) lp[sp.src_lin[t]] = 0.f;
    if (t < sp.nzero) lp[sp.zero_lin[t]] = 0.f;
}

// The pointwise steps take their operands from a struct loaded ahead of the arithmetic: the tiled
// kernels load a row's operands before the gathers that precede their use, so that the loads are
// in flight during the gathers. The per-cell kernels use the same structs and the same arithmetic.

// operands of the pressure transposed at one cell
template <int ND, bool EXPO, bool CODED>
struct PreOps {
    float lp, K, div, gk, A;
    float phi[ND][kNRelax];
    CodedCoef kc[ND];
    uint32_t code, kind;
};

template <int ND, bool EXPO, bool CODED>
__device__ inline void pre_load(const DevSim& s, const AdjView& w, int64_t c, PreOps<ND, EXPO, CODED>& o) {
    o.lp = w.lp[c];
    o.K = s.K[c];
    o.div = w.tdiv[c];
    o.gk = w.gK[c];
    if (EXPO) {
        o.A = s.aexp[c];
        return;
    }
#pragma unroll
    for (int a = 0; a < ND; ++a) {
#pragma unroll
        for (int nu = 0; nu < kNRelax; ++nu) o.phi[a][nu] = w.lphi[a][nu][c];
        if (!CODED) o.kc[a] = CodedCoef{s.ikp[a][c], s.ap[a][0][c], s.ap[a][1][c], s.bp[a][0][c], s.bp[a][1][c], 0};
    }
    if (CODED) o.code = gld16(s.rcode, (uint32_t)c);
}

template <int ND, bool EXPO, bool CODED>
__device__ inline void pre_decode(const DevSim& s, int64_t c, PreOps<ND, EXPO, CODED>& o) {
    if (!CODED || EXPO) return;
    const CodedCoef k = coef_of_code<false, true>(s, (uint32_t)c, o.code);
#pragma unroll
    for (int a = 0; a < ND; ++a) o.kc[a] = k;
}

// The pressure transposed at active cell c with mu = lambda_p[c] after the step's sparse part;
// leaves lambda_p[c] = mu (STORE_MU; the exponential model always stores A mu).
template <int ND, bool EXPO, bool CODED, bool STORE_MU>
__device__ inline void pre_store(const DevSim& s, const AdjView& w, int64_t c, float mu, const PreOps<ND, EXPO, CODED>& o) {
    if (EXPO) {
        const float t = -o.A * s.dt * o.K * mu;
#pragma unroll
        for (int a = 0; a < ND; ++a) w.H[a][c] = t;
        w.lp[c] = o.A * mu;
        w.gK[c] = o.gk + mu * (-o.A * s.dt) * o.div;
        return;
    }
    const float t = -s.dt * o.K * mu;
#pragma unroll
    for (int a = 0; a < ND; ++a) {
        const CodedCoef& k = o.kc[a];
        float lh = t * k.ik;
#pragma unroll
        for (int nu = 0; nu < kNRelax; ++nu) {
            const float tot = o.phi[a][nu] + t;
            lh += (nu ? k.a2 : k.a1) * tot;
            w.lphi[a][nu][c] = (nu ? k.b2 : k.b1) * tot;
        }
        w.H[a][c] = lh;
    }
    if (STORE_MU) w.lp[c] = mu;
    w.gK[c] = o.gk + mu * (-s.dt) * o.div;
}

// CODED (isotropic relaxation with codes): the relaxation coefficients of the cell come from its
// code's table row (2 bytes a cell) instead of the five per-cell maps
template <int ND, bool EXPO, bool CODED>
__global__ __launch_bounds__(256) void k_adj_pressure(DevSim s, AdjView w) {
    int64_t i, j, k;
    if (!adj_cell<ND>(s, i, j, k)) return;
    const int64_t c = i * s.sx + j * s.sy + k;
    PreOps<ND, EXPO, CODED> o;
    pre_load(s, w, c, o);
    pre_decode(s, c, o);
    pre_store<ND, EXPO, CODED, false>(s, w, c, o.lp, o);
}

// lambda_v_a += (D-_a)^T H_a at active cells
template <int ND, bool UNI>
__global__ __launch_bounds__(256) void k_adj_dminus_t(DevSim s, AdjView w) {
    int64_t i, j, k;
    if (!adj_cell<ND>(s, i, j, k)) return;
    const int64_t x = i * s.sx + j * s.sy + k;
    const int64_t st[3] = {s.sx, s.sy, 1};
#pragma unroll
    for (int a = 0; a < ND; ++a) {
        const float* H = w.H[a];
        const int64_t sa = st[a];
        float acc = 0.f;
#pragma unroll
        for (int m = 1; m <= 8; ++m) {
            const int64_t c1 = x - (m - 1) * sa, c2 = x + m * sa;
            acc += wts<UNI>(s, c1, ND, a)[m - 1] * H[c1] - wts<UNI>(s, c2, ND, a)[m - 1] * H[c2];
        }
#pragma unroll
        for (int b = 0; b < ND; ++b) {
            if (b == a) continue;
            const int64_t sb = st[b];
#pragma unroll
            for (int sg = -1; sg <= 1; sg += 2) {
                const int64_t c1 = x - sg * sb, c2 = x + sa - sg * sb;
                acc += wts<UNI>(s, c1, ND, a)[8] * H[c1] - wts<UNI>(s, c2, ND, a)[8] * H[c2];
            }
        }
        w.lv[a][x] += acc;
    }
}

// operands of the velocity transposed at one cell (nu: lambda_v as loaded)
template <int ND, bool EXPO, bool CODED>
struct VelOps {
    float nu[ND], rc, rn[ND], u[ND], grb[ND], A;
    float psi[ND][kNRelax];
    CodedCoef kc[ND];
    uint32_t code;
};

template <int ND, bool EXPO, bool CODED>
__device__ inline void vel_load(const DevSim& s, const AdjView& w, int64_t c, VelOps<ND, EXPO, CODED>& o) {
    const int64_t st[3] = {s.sx, s.sy, 1};
    o.rc = s.rho[c];
#pragma unroll
    for (int a = 0; a < ND; ++a) {
        o.nu[a] = w.lv[a][c];
        o.rn[a] = s.rho[c + st[a]];
        o.u[a] = w.tu[a][c];
        o.grb[a] = w.gRb[a][c];
    }
    if (EXPO) {
        o.A = s.aexp[c];
        return;
    }
#pragma unroll
    for (int a = 0; a < ND; ++a) {
#pragma unroll
        for (int q = 0; q < kNRelax; ++q) o.psi[a][q] = w.lpsi[a][q][c];
        if (!CODED) o.kc[a] = CodedCoef{s.ikv[a][c], s.av[a][0][c], s.av[a][1][c], s.bv[a][0][c], s.bv[a][1][c], 0};
    }
    if (CODED) o.code = gld16(s.rcode, (uint32_t)c);
}

template <int ND, bool EXPO, bool CODED>
__device__ inline void vel_decode(const DevSim& s, int64_t c, VelOps<ND, EXPO, CODED>& o) {
    if (!CODED || EXPO) return;
    const CodedCoef k = coef_of_code<true, true>(s, (uint32_t)c, o.code);
#pragma unroll
    for (int a = 0; a < ND; ++a) o.kc[a] = k;
}

// The velocity transposed at active cell c with o.nu[a] = nu (lambda_v_a after the gather);
// STORE_NU: also store lambda_v = nu (the exponential model always stores A nu).
template <int ND, bool EXPO, bool CODED, bool STORE_NU>
__device__ inline void vel_store(const DevSim& s, const AdjView& w, int64_t c, const VelOps<ND, EXPO, CODED>& o) {
#pragma unroll
    for (int a = 0; a < ND; ++a) {
        const float nu = o.nu[a];
        const float rb = 0.5f * (o.rc + o.rn[a]);
        const float beta = s.dt / rb;
        float lg;
        if (EXPO) {
            lg = -o.A * beta * nu;
            w.lv[a][c] = o.A * nu;
        } else {
            const CodedCoef& k = o.kc[a];
            lg = -beta * nu * k.ik;
#pragma unroll
            for (int q = 0; q < kNRelax; ++q) {
                const float tot = o.psi[a][q] - beta * nu;
                lg += (q ? k.a2 : k.a1) * tot;
                w.lpsi[a][q][c] = (q ? k.b2 : k.b1) * tot;
            }
            if (STORE_NU) w.lv[a][c] = nu;
        }
        w.G[a][c] = lg;
        w.gRb[a][c] = o.grb[a] + nu * o.u[a] * s.dt / (rb * rb);
    }
}

template <int ND, bool EXPO, bool CODED>
__global__ __launch_bounds__(256) void k_adj_velocity(DevSim s, AdjView w) {
    int64_t i, j, k;
    if (!adj_cell<ND>(s, i, j, k)) return;
    const int64_t c = i * s.sx + j * s.sy + k;
    VelOps<ND, EXPO, CODED> o;
    vel_load(s, w, c, o);
    vel_decode(s, c, o);
    vel_store<ND, EXPO, CODED, false>(s, w, c, o);
}

// lambda_p += sum_a (D+_a)^T G_a at active cells
template <int ND, bool UNI>
__global__ __launch_bounds__(256) void k_adj_dplus_t(DevSim s, AdjView w) {
    int64_t i, j, k;
    if (!adj_cell<ND>(s, i, j, k)) return;
    const int64_t x = i * s.sx + j * s.sy + k;
    const int64_t st[3] = {s.sx, s.sy, 1};
    float acc = 0.f;
#pragma unroll
    for (int a = 0; a < ND; ++a) {
        const float* G = w.G[a];
        const int64_t sa = st[a];
#pragma unroll
        for (int m = 1; m <= 8; ++m) {
            const int64_t c1 = x - m * sa, c2 = x + (m - 1) * sa;
            acc += wts<UNI>(s, c1, ND, a)[m - 1] * G[c1] - wts<UNI>(s, c2, ND, a)[m - 1] * G[c2];
        }
#pragma unroll
        for (int b = 0; b < ND; ++b) {
            if (b == a) continue;
            const int64_t sb = st[b];
#pragma unroll
            for (int sg = -1; sg <= 1; sg += 2) {
                const int64_t c1 = x - sa - sg * sb, c2 = x - sg * sb;
                acc += wts<UNI>(s, c1, ND, a)[8] * G[c1] - wts<UNI>(s, c2, ND, a)[8] * G[c2];
            }
        }
    }
    w.lp[x] += acc;
}

// The transposed gathers of a 2D step on tiles, with the gathered field (H or G) staged in LDS. A
// workgroup of 256 lanes owns a tile of ATX rows (x) by ATY columns (y); lane (r, j) updates
// rows r, r + 4, ... of column j. Axis x's field is staged over rows [i0 - 8, i0 + ATX + 8) and
// columns [j0 - 1, j0 + ATY + 1), axis y's over rows [i0 - 1, i0 + ATX + 1) and columns
// [j0 - 8, j0 + ATY + 8): every offset either gather reads (along its axis -8..+8, across it
// -1..+1). Quads outside the grid stage the ghost border's values (H and G are 0 off the updated
// cells). Every lane issues all of its staging loads before it stores any of them, so one memory
// latency covers the staging. A gather weighs each neighbour by the neighbour's own coefficient
// set: where the arms of a tile hold one set (AdjView::tile_sets) its weights are scalar
// registers; a tile of several sets also stages the cells' set indices and the weights of the handle's sets
// (tall tiles: of its own) in dynamic LDS, two dependent LDS reads a neighbour. The arithmetic and its order are the
// per-cell kernels', so the results are the same bit for bit.
constexpr int ATY = 64, kAdjLanes = 256;
constexpr int kShortTile = 8, kTallTile = 16;  // ATX
constexpr int AXC = ATY + 2, AYC = ATY + 16;   // columns of the staged regions
// How a launch weighs: the grid has one set; tiles of one set and tiles that look theirs up in the whole
// table; tiles that all look up, in a table of their own sets.
enum { kOneSet = 0, kAnySets = 1, kLookUp = 2 };
constexpr int kAdjLdsSets = 256;  // coefficient sets staged (ndmap beyond: per-cell kernels)
// A tile's word in AdjView::tile_sets: the lowest set of its arms, and how many from there.
__device__ __forceinline__ uint32_t lowest_set(uint32_t word) { return word & 0xffu; }
__device__ __forceinline__ uint32_t set_span(uint32_t word) { return word >> 8; }

// Stage R x C cells of `f` from row i, column j, with MIXED their set indices (above `lowest`) too; load
// first, put after.
template <int R, int C, bool MIXED>
struct GatherStage {
    static constexpr int N = (R * C + kAdjLanes - 1) / kAdjLanes;
    float v[N];
    uint8_t d[MIXED ? N : 1];
    __device__ __forceinline__ void load(const DevSim& s, const float* f, const uint8_t* dc8, uint32_t lowest, int i, int j) {
#pragma unroll
        for (int q = 0; q < N; ++q) {
            const int t = min((int)threadIdx.x + q * kAdjLanes, R * C - 1);
            const int r = t / C, cc = t - r * C;
            const uint32_t c = (uint32_t)(min(max(i + r, 0), (int)s.nx - 1) * (int)s.ny + min(max(j + cc, 0), (int)s.ny - 1));
            v[q] = gld32(f, c);
            if (MIXED) d[q] = (uint8_t)(dc8[c] - lowest);
        }
    }
    __device__ __forceinline__ void put(float* F, uint8_t* D) const {
#pragma unroll
        for (int q = 0; q < N; ++q) {
            const int t = threadIdx.x + q * kAdjLanes;
            if (t >= R * C) continue;
            F[t] = v[q];
            if (MIXED) D[t] = d[q];
        }
    }
};
// The weights of `n` sets from `lowest`, as pairs (9 a set), five loads in flight a lane.
__device__ __forceinline__ void stage_weights(const DevSim& s, uint32_t lowest, int sets, float* CT) {
    const int n = sets * kNCoef;
    const float2* from = reinterpret_cast<const float2*>(s.coef) + lowest * kNCoef;
    float2* to = reinterpret_cast<float2*>(CT);
    if (n <= 2 * kAdjLanes) {
        for (int t = threadIdx.x; t < n; t += kAdjLanes) to[t] = from[t];
        return;
    }
    constexpr int K = 5;
    for (int t0 = threadIdx.x; t0 < n; t0 += K * kAdjLanes) {
        float2 v[K];
#pragma unroll
        for (int k = 0; k < K; ++k) v[k] = from[min(t0 + k * kAdjLanes, n - 1)];
#pragma unroll
        for (int k = 0; k < K; ++k)
            if (t0 + k * kAdjLanes < n) to[t0 + k * kAdjLanes] = v[k];
    }
}
// word: the tile's, with OWN table of its sets; else the handle's table.
template <int ATX, bool MIXED, bool OWN>
__device__ __forceinline__ void stage_gather(const DevSim& s, const uint8_t* dc8, uint32_t word, const float* fx, const float* fy,
                                             int i0, int j0, float* FX, float* FY, uint8_t* DX, uint8_t* DY, float* CT) {
    GatherStage<ATX + 16, AXC, MIXED> x;
    GatherStage<ATX + 2, AYC, MIXED> y;
    x.load(s, fx, dc8, OWN ? lowest_set(word) : 0u, i0 - 8, j0 - 1);
    y.load(s, fy, dc8, OWN ? lowest_set(word) : 0u, i0 - 1, j0 - 8);
    if (MIXED && OWN) stage_weights(s, lowest_set(word), (int)set_span(word), CT);
    if (MIXED && !OWN)
        for (int t = threadIdx.x; t < s.ndmap * 2 * kNCoef; t += kAdjLanes) CT[t] = s.coef[t];
    x.put(FX, DX);
    y.put(FY, DY);
}

// Each tile's word: of the updated cells in its arms (the fields are 0 elsewhere); of tall tiles, whose tables
// hold no other sets, every cell of the grid in its arms.
template <int ATX>
__global__ __launch_bounds__(kAdjLanes) void k_adj_tile_sets(DevSim s, const uint8_t* dc8, uint32_t* sets) {
    __shared__ uint32_t least, most;
    constexpr int edge = ATX == kTallTile ? 0 : kHalo;
    const int i0 = kHalo + (int)blockIdx.y * ATX, j0 = kHalo + (int)blockIdx.x * ATY;
    if (threadIdx.x == 0) {
        least = 255;
        most = 0;
    }
    __syncthreads();
    uint32_t lo = 255, hi = 0;
    for (int a = 0; a < 2; ++a) {
        const int ei = a ? 1 : 8, ej = a ? 8 : 1, cols = ATY + 2 * ej, n = (ATX + 2 * ei) * cols;
        for (int t = threadIdx.x; t < n; t += kAdjLanes) {
            const int i = i0 - ei + t / cols, j = j0 - ej + t % cols;
            if (i < edge || i >= (int)s.nx - edge || j < edge || j >= (int)s.ny - edge) continue;
            const uint32_t set = dc8[(uint32_t)(i * (int)s.ny + j)];
            lo = min(lo, set);
            hi = max(hi, set);
        }
    }
    atomicMin(&least, lo);
    atomicMax(&most, hi);
    __syncthreads();
    if (threadIdx.x == 0) sets[blockIdx.x + blockIdx.y * gridDim.x] = (most - least + 1) << 8 | least;
}

// DMINUS: lambda_v_a += (D-_a)^T H_a, then the velocity transposed of the cell (EXPO, CODED as
// k_adj_velocity); else lambda_p += sum_a (D+_a)^T G_a, then with NEXT the next step's sparse
// part and pressure transposed of the cell (EXPO, CODED as k_adj_pressure; w.tdiv is then the
// next step's tape). Each lane loads the operands of its first row before the staging and those
// of row m + 1 before the gathers of row m, so their memory latency overlaps other work.
//
// What bounds it: the latencies of a workgroup's load, gather and store phases (small grids have few
// workgroups a CU), the memory traffic on large ones. us a reverse step with 6 sound speeds, tiles of 16
// rows that always looked weights up -> these with 16 rows -> with 8 rows: 240 x 256 22.6 -> 20.0 -> 14.5;
// 640 x 640 30.9 -> 27.4 -> 26.0; 1184 x 1184 71.4 -> 70.7 -> 65.9; 1700 x 1700 152.6 -> 150.4 -> 147.7.
// One sound speed, 640 x 640: 24.1 -> 23.0 -> 21.3; exponential model 27.6 -> 25.1 -> 23.9. Many sets on large
// grids: tiles of 16 rows that all look up, in a table of the sets that they hold (adj_may_take_tall_tiles).
// Measured and left out: both rows' operands and table rows before the staging (640 x 640: 28.3); in the
// short tiles the tile's own table (640 x 640, 6 sets: 25.8 -> 26.1; 1152 x 1152, 31 sets: 63.2 -> 63.7).
template <int ATX, int SETS, bool DMINUS, bool EXPO, bool CODED, bool NEXT>
__global__ __launch_bounds__(kAdjLanes) void k_adj_gather_tile2d(DevSim s, AdjView w, AdjNext nx) {
    constexpr int AXR = ATX + 16, AYR = ATX + 2;  // rows of the staged regions
    __shared__ float FX[AXR * AXC];
    __shared__ float FY[AYR * AYC];
    __shared__ uint8_t DX[SETS == kOneSet ? 1 : AXR * AXC];
    __shared__ uint8_t DY[SETS == kOneSet ? 1 : AYR * AYC];
    extern __shared__ __attribute__((aligned(8))) float CT[];  // [set][axis][9], the handle's sets or the tile's
    constexpr int NR = ATX / 4;    // rows per lane: rl, rl + 4, ...
    // Each XCD takes a contiguous run of tiles, so that neighbouring tiles, which stage the same halo
    // cells, share an L2: the fetch from memory drops by 40 % and the kernels run 17 % faster than with
    // the tiles in launch order.
    const uint32_t tile = xcd_order(blockIdx.x + blockIdx.y * gridDim.x, gridDim.x * gridDim.y);
    const uint32_t bx = tile % gridDim.x, by = tile / gridDim.x;
    const int64_t i0 = kHalo + (int64_t)by * ATX, j0 = kHalo + (int64_t)bx * ATY;
    const int jl = threadIdx.x % ATY, rl = threadIdx.x / ATY;
    const int64_t j = j0 + jl;
    // this lane's rows that hold updated cells
    const int64_t left = s.nx - kHalo - (i0 + rl);
    const int nrows = j >= s.ny - kHalo || left <= 0 ? 0 : (int)(left >= 4 * NR ? NR : (left + 3) / 4);
    using Ops = std::conditional_t<DMINUS, VelOps<2, EXPO, CODED>, PreOps<2, EXPO, CODED>>;
    Ops ops[2];
    auto load = [&](int m, Ops& o) {
        const int64_t x = (i0 + rl + 4 * m) * s.sx + j;
        if constexpr (DMINUS) {
            vel_load(s, w, x, o);
        } else if constexpr (NEXT) {
            pre_load(s, w, x, o);
            o.kind = nx.kind[x];
        } else {
            o.lp = w.lp[x];
        }
    };
    if (nrows > 0) load(0, ops[0]);
    const uint32_t word = SETS == kOneSet ? 1u << 8 : (uint32_t)__builtin_amdgcn_readfirstlane(w.tile_sets[tile]);
    const bool one = SETS == kOneSet || (SETS == kAnySets && set_span(word) == 1);
    const float *fx = DMINUS ? w.H[0] : w.G[0], *fy = DMINUS ? w.H[1] : w.G[1];
    if (one) stage_gather<ATX, false, false>(s, w.dc8, word, fx, fy, (int)i0, (int)j0, FX, FY, DX, DY, CT);
    else stage_gather<ATX, true, SETS == kLookUp>(s, w.dc8, word, fx, fy, (int)i0, (int)j0, FX, FY, DX, DY, CT);
    __syncthreads();
    // staged element at (di, dj) from cell (il, jl) of the tile, for axis x's and axis y's field
    auto ex = [&](int il, int di, int dj) { return (il + 8 + di) * AXC + (jl + 1 + dj); };
    auto ey = [&](int il, int di, int dj) { return (il + 1 + di) * AYC + (jl + 8 + dj); };
    // wx, wy: weight k of the staged element e, of axis x's and axis y's field
    auto rows = [&](const auto& wx, const auto& wy) {
#pragma unroll
        for (int m = 0; m < NR; ++m) {
            if (m >= nrows) break;
            Ops& o = ops[m & 1];
            const int il = rl + 4 * m;
            const int64_t x = (i0 + il) * s.sx + j;
            if constexpr (DMINUS) vel_decode(s, x, o);
            else if constexpr (NEXT) pre_decode(s, x, o);
            if (m + 1 < nrows) load(m + 1, ops[(m + 1) & 1]);
            if constexpr (DMINUS) {
                // axis x: c1 = x - (m-1) e_x, c2 = x + m e_x; transverse c1 = x -+ e_y, c2 = x + e_x -+ e_y
                float acc = 0.f;
#pragma unroll
                for (int q = 1; q <= 8; ++q) {
                    const int e1 = ex(il, -(q - 1), 0), e2 = ex(il, q, 0);
                    acc += wx(e1, q - 1) * FX[e1] - wx(e2, q - 1) * FX[e2];
                }
#pragma unroll
                for (int sg = -1; sg <= 1; sg += 2) {
                    const int e1 = ex(il, 0, -sg), e2 = ex(il, 1, -sg);
                    acc += wx(e1, 8) * FX[e1] - wx(e2, 8) * FX[e2];
                }
                o.nu[0] = o.nu[0] + acc;
                acc = 0.f;
#pragma unroll
                for (int q = 1; q <= 8; ++q) {
                    const int e1 = ey(il, 0, -(q - 1)), e2 = ey(il, 0, q);
                    acc += wy(e1, q - 1) * FY[e1] - wy(e2, q - 1) * FY[e2];
                }
#pragma unroll
                for (int sg = -1; sg <= 1; sg += 2) {
                    const int e1 = ey(il, -sg, 0), e2 = ey(il, -sg, 1);
                    acc += wy(e1, 8) * FY[e1] - wy(e2, 8) * FY[e2];
                }
                o.nu[1] = o.nu[1] + acc;
                vel_store<2, EXPO, CODED, true>(s, w, x, o);
            } else {
                // axis x: c1 = x - m e_x, c2 = x + (m-1) e_x; transverse c1 = x - e_x -+ e_y, c2 = x -+ e_y
                float acc = 0.f;
#pragma unroll
                for (int q = 1; q <= 8; ++q) {
                    const int e1 = ex(il, -q, 0), e2 = ex(il, q - 1, 0);
                    acc += wx(e1, q - 1) * FX[e1] - wx(e2, q - 1) * FX[e2];
                }
#pragma unroll
                for (int sg = -1; sg <= 1; sg += 2) {
                    const int e1 = ex(il, -1, -sg), e2 = ex(il, 0, -sg);
                    acc += wx(e1, 8) * FX[e1] - wx(e2, 8) * FX[e2];
                }
#pragma unroll
                for (int q = 1; q <= 8; ++q) {
                    const int e1 = ey(il, 0, -q), e2 = ey(il, 0, q - 1);
                    acc += wy(e1, q - 1) * FY[e1] - wy(e2, q - 1) * FY[e2];
                }
#pragma unroll
                for (int sg = -1; sg <= 1; sg += 2) {
                    const int e1 = ey(il, -sg, -1), e2 = ey(il, -sg, 0);
                    acc += wy(e1, 8) * FY[e1] - wy(e2, 8) * FY[e2];
                }
                if constexpr (NEXT) pre_store<2, EXPO, CODED, true>(s, w, x, next_mu(nx, x, o.kind, o.lp + acc), o);
                else w.lp[x] = o.lp + acc;
            }
        }
    };
    if (one) {
        float kx[kNCoef], ky[kNCoef];
        const scalar_ptr c = as_scalar(s.coef) + lowest_set(word) * 2 * kNCoef;
#pragma unroll
        for (int k = 0; k < kNCoef; ++k) {
            kx[k] = c[k];
            ky[k] = c[kNCoef + k];
        }
        rows([&](int, int k) { return kx[k]; }, [&](int, int k) { return ky[k]; });
    } else {
        rows([&](int e, int k) { return CT[(int)DX[e] * 2 * kNCoef + k]; },
             [&](int e, int k) { return CT[((int)DY[e] * 2 + 1) * kNCoef + k]; });
    }
}

__global__ __launch_bounds__(256) void k_adj_set_index(const int32_t* dcmap, uint8_t* dc8, int64_t n) {
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t < n) dc8[t] = (uint8_t)dcmap[t];
}

// d/d rho[x] = sum_a (g_rb_a[x] + g_rb_a[x - e_a]) / 2, over the whole (padded) grid
__global__ __launch_bounds__(256) void k_adj_rho(DevSim s, AdjView w, float* grho) {
    const int64_t x = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int64_t n = s.nx * s.sx;
    if (x >= n) return;
    const int64_t i = x / s.sx, rem = x - (x / s.sx) * s.sx;
    const int64_t j = s.ndim == 3 ? rem / s.sy : rem, k = s.ndim == 3 ? rem - (rem / s.sy) * s.sy : 0;
    if (j >= s.ny || k >= s.nz) {  // row padding
        grho[x] = 0.f;
        return;
    }
    const int64_t coord[3] = {i, j, k};
    const int64_t st[3] = {s.sx, s.sy, 1};
    float acc = 0.f;
    for (int a = 0; a < s.ndim; ++a) {
        acc += w.gRb[a][x];
        if (coord[a] > 0) acc += w.gRb[a][x - st[a]];
    }
    grho[x] = 0.5f * acc;
}

}  // namespace

static dim3 adj_grid(const DevSim& s) {
    if (s.ndim == 2) return dim3((unsigned)((s.ny + 63) / 64), (unsigned)((s.nx + 3) / 4), 1);
    return dim3((unsigned)((s.nz + 63) / 64), (unsigned)((s.ny + 3) / 4), (unsigned)s.nx);
}

hipError_t launch_adj_sparse(float* lp, const float* grow, const AdjSparse& sp, bool injecting, hipStream_t st) {
    int64_t n = sp.nzero;
    if (grow && sp.nvox > n) n = sp.nvox;
    if (injecting && sp.nsrc > n) n = sp.nsrc;
    if (n == 0) return hipSuccess;
    hipLaunchKernelGGL(k_adj_sparse, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, lp, grow, sp,
                       injecting ? 1 : 0);
    return hipGetLastError();
}

// the transposed gathers on LDS tiles: 2D grids of at most kAdjLdsSets coefficient sets (the
// staged set indices are bytes)
bool adj_tiles(const DevSim& s) { return s.ndim == 2 && s.ndmap <= kAdjLdsSets && s.nx * s.ny < ((int64_t)1 << 30) && s.nx < kShortTile * (int64_t)65535; }

// FULLWAVE_HIP_ADJ_GATHERS=percell keeps the per-cell kernels (to compare the two forms)
bool adj_percell_gathers() {
    const char* e = getenv("FULLWAVE_HIP_ADJ_GATHERS");
    return e && !strncmp(e, "percell", 7);
}

bool adj_fuses_next(const DevSim& s, const AdjView& w) { return w.sets || (adj_tiles(s) && !adj_percell_gathers()); }

hipError_t launch_adj_set_index(const int32_t* dcmap, uint8_t* dc8, int64_t n, hipStream_t st) {
    if (n <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_adj_set_index, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, dcmap, dc8, n);
    return hipGetLastError();
}

static dim3 adj_tile_grid(const DevSim& s, bool tall) {
    const int rows = tall ? kTallTile : kShortTile;
    return dim3((unsigned)((s.ny - 2 * kHalo + ATY - 1) / ATY), (unsigned)((s.nx - 2 * kHalo + rows - 1) / rows));
}

size_t adj_tile_count(const DevSim& s, bool tall) {
    const dim3 g = adj_tile_grid(s, tall);
    return (size_t)g.x * g.y;
}

// Tall tiles stage fewer halo cells a cell (3.5 against 4.7); short ones have twice as many workgroups, weigh
// tiles of one set with scalars, and stage the whole table in the others. us a reverse step, short -> tall, of
// media whose tiles mostly hold several sets, smooth / random cells (short tiles in brackets):
//   sets   640 x 640 (780)               900 x 900 (1554)             1152 x 1152 (2556)
//     6    27.5 -> 31.5 / 27.1 -> 30.1   39.8 -> 42.8 / 42.6 -> 43.4   56.3 -> 56.8 / 60.4 -> 58.7
//    30    27.8 -> 30.0 / 29.9 -> 31.6   43.3 -> 42.8 / 45.5 -> 46.3   60.6 -> 56.9 / 64.7 -> 61.5
//   130    29.4 -> 30.2 / 34.9 -> 34.2   46.4 -> 43.1 / 52.5 -> 52.7   64.8 -> 57.7 / 75.1 -> 67.9
// So tall from 32 sets and 1280 short tiles (five workgroups a CU, the most that run at once), where the
// part of the short tiles that hold several sets makes up for the others: at 130 sets on 1152 x 1152 with
// 38 % of them 60.6 -> 57.7, with 13 % left short at 56.4 (tall: 57.5).
bool adj_may_take_tall_tiles(const DevSim& s) { return s.ndmap >= 32 && adj_tile_count(s, false) >= 1280; }

bool adj_takes_tall_tiles(const DevSim& s, const std::vector<uint32_t>& words) {
    size_t several = 0;
    for (uint32_t w : words) several += (w >> 8) > 1;
    return (double)several >= (0.2 + 16.0 / s.ndmap) * (double)words.size();
}

uint32_t adj_tile_span(const std::vector<uint32_t>& words) {
    uint32_t span = 1;
    for (uint32_t w : words) span = std::max(span, w >> 8);
    return span;
}

hipError_t launch_adj_tile_sets(const DevSim& s, const uint8_t* dc8, bool tall, uint32_t* sets, hipStream_t st) {
    const dim3 g = adj_tile_grid(s, tall);
    if (tall) hipLaunchKernelGGL(k_adj_tile_sets<kTallTile>, g, dim3(kAdjLanes), 0, st, s, dc8, sets);
    else hipLaunchKernelGGL(k_adj_tile_sets<kShortTile>, g, dim3(kAdjLanes), 0, st, s, dc8, sets);
    return hipGetLastError();
}

template <bool DMINUS, bool EXPO, bool CODED, bool NEXT>
void launch_gather_tile2d(const DevSim& s, const AdjView& w, const AdjNext& nx, hipStream_t st) {
    const dim3 g = adj_tile_grid(s, w.tall_span != 0), b(kAdjLanes);
    const size_t lds = (size_t)(w.tall_span ? w.tall_span : (uint32_t)s.ndmap) * 2 * kNCoef * sizeof(float);
    if (s.ndmap == 1) hipLaunchKernelGGL((k_adj_gather_tile2d<kShortTile, kOneSet, DMINUS, EXPO, CODED, NEXT>), g, b, 0, st, s, w, nx);
    else if (w.tall_span) hipLaunchKernelGGL((k_adj_gather_tile2d<kTallTile, kLookUp, DMINUS, EXPO, CODED, NEXT>), g, b, lds, st, s, w, nx);
    else hipLaunchKernelGGL((k_adj_gather_tile2d<kShortTile, kAnySets, DMINUS, EXPO, CODED, NEXT>), g, b, lds, st, s, w, nx);
}

static bool adj_coded(const DevSim& s) { return !s.aexp && s.isotropic && s.rcode; }

template <int ND>
void launch_pressure_nd(const DevSim& s, const AdjView& w, dim3 g, dim3 b, hipStream_t st) {
    if (s.aexp) hipLaunchKernelGGL((k_adj_pressure<ND, true, false>), g, b, 0, st, s, w);
    else if (adj_coded(s)) hipLaunchKernelGGL((k_adj_pressure<ND, false, true>), g, b, 0, st, s, w);
    else hipLaunchKernelGGL((k_adj_pressure<ND, false, false>), g, b, 0, st, s, w);
}

template <int ND, bool UNI>
void launch_rest_nd(const DevSim& s, const AdjView& w, dim3 g, dim3 b, hipStream_t st) {
    hipLaunchKernelGGL((k_adj_dminus_t<ND, UNI>), g, b, 0, st, s, w);
    if (s.aexp) hipLaunchKernelGGL((k_adj_velocity<ND, true, false>), g, b, 0, st, s, w);
    else if (adj_coded(s)) hipLaunchKernelGGL((k_adj_velocity<ND, false, true>), g, b, 0, st, s, w);
    else hipLaunchKernelGGL((k_adj_velocity<ND, false, false>), g, b, 0, st, s, w);
    hipLaunchKernelGGL((k_adj_dplus_t<ND, UNI>), g, b, 0, st, s, w);
}

hipError_t launch_adj_pressure(const DevSim& s, const AdjView& w, hipStream_t st) {
    if (w.sets) return launch_adj_start_bricks(s, w, st);
    const dim3 g = adj_grid(s), b(64, 4);
    if (s.ndim == 2) launch_pressure_nd<2>(s, w, g, b, st);
    else launch_pressure_nd<3>(s, w, g, b, st);
    return hipGetLastError();
}

hipError_t launch_adj_rest(const DevSim& s, const AdjView& w, const AdjNext* next, hipStream_t st) {
    if (w.sets) return launch_adj_rest_bricks(s, w, next, st);
    if (adj_fuses_next(s, w)) {
        const AdjNext none{};
        if (s.aexp) launch_gather_tile2d<true, true, false, false>(s, w, none, st);
        else if (adj_coded(s)) launch_gather_tile2d<true, false, true, false>(s, w, none, st);
        else launch_gather_tile2d<true, false, false, false>(s, w, none, st);
        if (!next) {
            launch_gather_tile2d<false, false, false, false>(s, w, none, st);
        } else {
            AdjView wn = w;  // the next step's pressure transposed reads its own tape
            wn.tdiv = next->tdiv;
            if (s.aexp) launch_gather_tile2d<false, true, false, true>(s, wn, *next, st);
            else if (adj_coded(s)) launch_gather_tile2d<false, false, true, true>(s, wn, *next, st);
            else launch_gather_tile2d<false, false, false, true>(s, wn, *next, st);
        }
        return hipGetLastError();
    }
    if (next) return hipErrorInvalidValue;  // the per-cell kernels do not take the next step
    const dim3 g = adj_grid(s), b(64, 4);
    const bool u = s.ndmap == 1;
    if (s.ndim == 2) {
        if (u) launch_rest_nd<2, true>(s, w, g, b, st);
        else launch_rest_nd<2, false>(s, w, g, b, st);
    } else {
        if (u) launch_rest_nd<3, true>(s, w, g, b, st);
        else launch_rest_nd<3, false>(s, w, g, b, st);
    }
    return hipGetLastError();
}

hipError_t launch_adj_rho(const DevSim& s, const AdjView& w, float* grho, hipStream_t st) {
    const int64_t n = s.nx * s.sx;
    hipLaunchKernelGGL(k_adj_rho, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, s, w, grho);
    return hipGetLastError();
}

}  // namespace fw
