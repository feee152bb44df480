// Per-cell kernels: one lane per grid cell, stencil operands straight from global memory (the caches
// serve their overlap). They take every model, size and type, and are the fastest kernels of small
// grids, of grids whose rows are not 16-byte aligned, and of small 3D grids: no staging, no barrier,
// and as many wavefronts as there are cells.
//
// What bounds them is the chain of dependent loads of a wavefront (small grids run few wavefronts a
// SIMD), so every load is issued before the first result is needed, and the chain is short: the cell's
// code, then one 64-byte row that holds its relaxation coefficients and its stencil weights (DevSim::
// rwide_v / rwide_p), or its set index, then its weights. A wavefront whose cells share the code (or the
// set) reads the row (or the weights) with scalar loads. The pressure kernel also does the step's
// sources, pressure release and sensors at the points of its own cells. Before (axis after axis, each
// waiting for the stores of the last, the per-cell maps, a boundary launch of its own), us a step:
// 256 x 224 cells 10.7 -> 9.3 (two launches of the host; the kernels take 3.6 and 4.3); 1003 x 677 35.7 ->
// 22.9; exponential model on 1152 x 1150 32.0 -> 22.3; 131 x 117 x 109 69.5 -> 53.4 (there the 72 stencil
// reads a cell bound it, and the memory variables go through the caches: cell_memory_streams).
//
// A workgroup of 256 lanes takes 4 rows of 64 cells. The arithmetic and its order are the other
// families'.
#include "fw_internal.h"

namespace fw {

namespace {

// What a cell's coefficients are read from.
enum CellModel { kCellMaps, kCellAxes, kCellCoded, kCellExpo };

// The rows of contiguous cells of a grid that hold updated cells: `first` + [0, count), `pitch`
// elements each (2D: a row per x, 3D: a row per (x, y), of which those in the ghost border of y do
// nothing).
struct CellRows {
    int64_t first, count, pitch;
};
__host__ __device__ inline CellRows cell_rows(const DevSim& s) {
    if (s.ndim == 2) return CellRows{kHalo, s.nx - 2 * kHalo, s.sx};
    return CellRows{kHalo * s.ny, (s.nx - 2 * kHalo) * s.ny, s.sy};
}

// The tile of this workgroup (2D: each XCD a contiguous run of them; in 3D, where a run's stencils reach
// over whole planes, the launch order is 3 % faster).
template <int ND>
__device__ inline uint32_t cell_tile() {
    return ND == 2 ? xcd_order(blockIdx.x, gridDim.x) : blockIdx.x;
}

// The cell of this lane: its element, and whether it is updated. Tile `tile` of the grid, tiles
// in row-major order, `gx` across.
template <int ND, class Idx>
__device__ inline bool cell_of_lane(const DevSim& s, unsigned tile, unsigned gx, Idx& c) {
    const unsigned by = tile / gx, bx = tile - by * gx;
    const CellRows rows = cell_rows(s);
    const Idx row = (Idx)__builtin_amdgcn_readfirstlane(by * kCellTileRows + threadIdx.x / kCellTileCols);
    const Idx k = (Idx)(bx * kCellTileCols + threadIdx.x % kCellTileCols);
    const Idx r = (Idx)rows.first + row;
    c = r * (Idx)rows.pitch + k;
    if ((int64_t)row >= rows.count) return false;
    const Idx n = (Idx)(ND == 2 ? s.ny : s.nz);
    bool ok = k >= (Idx)kHalo && k < n - (Idx)kHalo;
    if (ND == 3) {
        const Idx j = r % (Idx)s.ny;
        ok = ok && j >= (Idx)kHalo && j < (Idx)s.ny - (Idx)kHalo;
    }
    return ok;
}

// element c of the array `base` elements further on; the address is a scalar base and a 32-bit lane
// offset where the grid has fewer than 2^30 cells
__device__ __forceinline__ float at(const float* f, int64_t base, uint32_t c) { return gld32(f + base, c); }
__device__ __forceinline__ float at(const float* f, int64_t base, int64_t c) { return f[base + c]; }
template <bool NT>
__device__ __forceinline__ float at_nt(const float* f, uint32_t c) { return NT ? gldnt(f, c) : gld32(f, c); }
template <bool NT>
__device__ __forceinline__ float at_nt(const float* f, int64_t c) { return f[c]; }
__device__ __forceinline__ void put(float* f, uint32_t c, float v) { gst32(f, c, v); }
__device__ __forceinline__ void put(float* f, int64_t c, float v) { f[c] = v; }
template <bool NT>
__device__ __forceinline__ void put_nt(float* f, uint32_t c, float v) {
    if (NT) gstnt(f, c, v);
    else gst32(f, c, v);
}
template <bool NT>
__device__ __forceinline__ void put_nt(float* f, int64_t c, float v) { f[c] = v; }

// The coefficients of a cell: one set for all axes, or (kCellAxes) one per axis; the weights of axis 0.
template <int ND, int MODEL>
struct CellCoef {
    static constexpr int NA = MODEL == kCellAxes ? ND : 1;
    float ik[NA], a[NA][2], b[NA][2], decay;
    float w[kNCoef];
    int32_t dc;
    uint32_t code;
};

__device__ inline void load_weights(float (&w)[kNCoef], const DevSim& s, int32_t dc, int nd, int axis) {
    const int32_t d0 = __builtin_amdgcn_readfirstlane(dc);
    if (__all(dc == d0)) {
        const scalar_ptr c = as_scalar(s.coef) + ((int64_t)d0 * nd + axis) * kNCoef;
#pragma unroll
        for (int k = 0; k < kNCoef; ++k) w[k] = c[k];
    } else {
        const float* c = s.coef + ((int64_t)dc * nd + axis) * kNCoef;
#pragma unroll
        for (int k = 0; k < kNCoef; ++k) w[k] = c[k];
    }
}

// The first load of the chain: the code, or the set index.
template <int ND, int MODEL, class Idx>
__device__ inline void coef_head(CellCoef<ND, MODEL>& k, const DevSim& s, Idx c) {
    if (MODEL == kCellCoded) k.code = gld16(s.rcode, (uint32_t)c);
    else k.dc = s.ndmap == 1 ? 0 : s.dcmap[c];
}

// The per-cell maps (issued with the operands).
template <int ND, int MODEL, bool VEL, class Idx>
__device__ inline void coef_maps(CellCoef<ND, MODEL>& k, const DevSim& s, Idx c) {
    if (MODEL == kCellExpo) k.decay = at(s.aexp, 0, c);
    if (MODEL != kCellMaps && MODEL != kCellAxes) return;
#pragma unroll
    for (int a = 0; a < CellCoef<ND, MODEL>::NA; ++a) {
        k.ik[a] = at(VEL ? s.ikv[a] : s.ikp[a], 0, c);
#pragma unroll
        for (int nu = 0; nu < kNRelax; ++nu) {
            k.a[a][nu] = at(VEL ? s.av[a][nu] : s.ap[a][nu], 0, c);
            k.b[a][nu] = at(VEL ? s.bv[a][nu] : s.bp[a][nu], 0, c);
        }
    }
}

// The rest of the chain: the row of the code, or the weights of the set.
template <int ND, int MODEL, bool VEL>
__device__ inline void coef_tail(CellCoef<ND, MODEL>& k, const DevSim& s) {
    if (MODEL != kCellCoded) {
        load_weights(k.w, s, k.dc, ND, 0);
        return;
    }
    const float* tab = VEL ? s.rwide_v : s.rwide_p;
    const uint32_t c0 = __builtin_amdgcn_readfirstlane(k.code);
    if (__all(k.code == c0)) {
        const scalar_ptr row = as_scalar(tab) + c0 * kWideStride;
        k.ik[0] = row[0];
        k.a[0][0] = row[1];
        k.a[0][1] = row[2];
        k.b[0][0] = row[3];
        k.b[0][1] = row[4];
#pragma unroll
        for (int m = 0; m < kNCoef; ++m) k.w[m] = row[5 + m];
        return;
    }
    const float4* row = reinterpret_cast<const float4*>(tab + k.code * kWideStride);
    const float4 q0 = row[0], q1 = row[1], q2 = row[2], q3 = row[3];
    k.ik[0] = q0.x;
    k.a[0][0] = q0.y;
    k.a[0][1] = q0.z;
    k.b[0][0] = q0.w;
    k.b[0][1] = q1.x;
    const float w[kNCoef] = {q1.y, q1.z, q1.w, q2.x, q2.y, q2.z, q2.w, q3.x, q3.y};
#pragma unroll
    for (int m = 0; m < kNCoef; ++m) k.w[m] = w[m];
}

// TAPE: also write the adjoint tape of the step (DevSim::tape_u, tape_div)
template <int ND, int MODEL, bool TAPE, bool NT, class Idx>
__global__ __launch_bounds__(256) void k_velocity_cell(DevSim batch, unsigned gx) {
    const DevSim s = shot_view(batch, blockIdx.y);
    Idx c;
    if (!cell_of_lane<ND, Idx>(s, cell_tile<ND>(), gx, c)) return;
    CellCoef<ND, MODEL> k;
    coef_head(k, s, c);
    const int64_t st[3] = {s.sx, s.sy, 1};
    // p along each axis (element m: c + (m - 7) e_a) and on the diagonals c + e_a + e_b, c + e_a - e_b
    float ax[ND][16], pp[ND][ND], pm[ND][ND];
    float rho_c, rho_n[ND], psi[ND][2], v[ND];
#pragma unroll
    for (int a = 0; a < ND; ++a) {
        const int64_t sa = ND == 2 && a == 1 ? 1 : st[a];
#pragma unroll
        for (int m = 0; m < 16; ++m)
            if (a == 0 || m != 7) ax[a][m] = at(s.p, (m - 7) * sa, c);
#pragma unroll
        for (int b = 0; b < ND; ++b) {
            const int64_t sb = ND == 2 && b == 1 ? 1 : st[b];
            if (b > a) pp[a][b] = at(s.p, sa + sb, c);
            if (b != a) pm[a][b] = at(s.p, sa - sb, c);
        }
        rho_n[a] = at(s.rho, sa, c);
        v[a] = at(s.v[a], 0, c);
        if (MODEL != kCellExpo) {
            psi[a][0] = at_nt<NT>(s.psi[a][0], c);
            psi[a][1] = at_nt<NT>(s.psi[a][1], c);
        }
    }
    rho_c = at(s.rho, 0, c);
    coef_maps<ND, MODEL, true>(k, s, c);
    coef_tail<ND, MODEL, true>(k, s);
#pragma unroll
    for (int a = 0; a < ND; ++a) {
        if (MODEL != kCellCoded && a > 0 && !s.coef_axes_same) load_weights(k.w, s, k.dc, ND, a);
        auto on = [&](int axis, int m) { return m == 7 ? ax[0][7] : ax[axis][m]; };
        float acc = 0.f;
#pragma unroll
        for (int m = 1; m <= 8; ++m) acc = tap(acc, k.w[m - 1], on(a, 7 + m), on(a, 8 - m));
        float tr = 0.f;
#pragma unroll
        for (int b = 0; b < ND; ++b) {
            if (b == a) continue;
            tr += ((a < b ? pp[a][b] : pp[b][a]) - on(b, 8)) + (pm[a][b] - on(b, 6));
        }
        const float D = __builtin_fmaf(k.w[8], tr, acc);
        if (MODEL == kCellExpo) {
            put(s.v[a], c, k.decay * velocity_step(v[a], s.dt, rho_c, rho_n[a], D));
            if (TAPE) put(s.tape_u[a], c, k.decay * D);
            continue;
        }
        constexpr bool axes = MODEL == kCellAxes;
        const float q1 = memory_step(k.b[axes ? a : 0][0], psi[a][0], k.a[axes ? a : 0][0], D);
        const float q2 = memory_step(k.b[axes ? a : 0][1], psi[a][1], k.a[axes ? a : 0][1], D);
        put_nt<NT>(s.psi[a][0], c, q1);
        put_nt<NT>(s.psi[a][1], c, q2);
        const float u = corrected(D, k.ik[axes ? a : 0], q1, q2);
        put(s.v[a], c, velocity_step(v[a], s.dt, rho_c, rho_n[a], u));
        if (TAPE) put(s.tape_u[a], c, u);
    }
}

template <int ND, int MODEL, bool TAPE, bool NT, class Idx>
__device__ inline void pressure_cell(const DevSim& s, Idx c) {
    CellCoef<ND, MODEL> k;
    coef_head(k, s, c);
    const int64_t st[3] = {s.sx, s.sy, 1};
    // v_a along its axis (element m: c + (m - 8) e_a) and beside it: [b][0..3] at c + e_b, c - e_a + e_b,
    // c - e_b, c - e_a - e_b
    float ax[ND][16], side[ND][ND][4];
    float phi[ND][2];
#pragma unroll
    for (int a = 0; a < ND; ++a) {
        const int64_t sa = ND == 2 && a == 1 ? 1 : st[a];
        const float* va = s.v[a];
#pragma unroll
        for (int m = 0; m < 16; ++m) ax[a][m] = at(va, (m - 8) * sa, c);
#pragma unroll
        for (int b = 0; b < ND; ++b) {
            if (b == a) continue;
            const int64_t sb = ND == 2 && b == 1 ? 1 : st[b];
            side[a][b][0] = at(va, sb, c);
            side[a][b][1] = at(va, sb - sa, c);
            side[a][b][2] = at(va, -sb, c);
            side[a][b][3] = at(va, -sa - sb, c);
        }
        if (MODEL != kCellExpo) {
            phi[a][0] = at_nt<NT>(s.phi[a][0], c);
            phi[a][1] = at_nt<NT>(s.phi[a][1], c);
        }
    }
    const float p = at(s.p, 0, c), K = at(s.K, 0, c);
    coef_maps<ND, MODEL, false>(k, s, c);
    coef_tail<ND, MODEL, false>(k, s);
    float div = 0.f;
#pragma unroll
    for (int a = 0; a < ND; ++a) {
        if (MODEL != kCellCoded && a > 0 && !s.coef_axes_same) load_weights(k.w, s, k.dc, ND, a);
        float acc = 0.f;
#pragma unroll
        for (int m = 1; m <= 8; ++m) acc = tap(acc, k.w[m - 1], ax[a][7 + m], ax[a][8 - m]);
        float tr = 0.f;
#pragma unroll
        for (int b = 0; b < ND; ++b) {
            if (b == a) continue;
            tr += (side[a][b][0] - side[a][b][1]) + (side[a][b][2] - side[a][b][3]);
        }
        const float D = __builtin_fmaf(k.w[8], tr, acc);
        if (MODEL == kCellExpo) {
            div += D;
            continue;
        }
        constexpr bool axes = MODEL == kCellAxes;
        const float q1 = memory_step(k.b[axes ? a : 0][0], phi[a][0], k.a[axes ? a : 0][0], D);
        const float q2 = memory_step(k.b[axes ? a : 0][1], phi[a][1], k.a[axes ? a : 0][1], D);
        put_nt<NT>(s.phi[a][0], c, q1);
        put_nt<NT>(s.phi[a][1], c, q2);
        div += corrected(D, k.ik[axes ? a : 0], q1, q2);
    }
    const float out = pressure_step(p, s.dt, K, div);
    put(s.p, c, MODEL == kCellExpo ? k.decay * out : out);
    if (TAPE) put(s.tape_div, c, div);
}

// gs.g non-null: each workgroup then also does the step's source, pressure-release and sensor work of
// its tile (tile blockIdx.x of shot blockIdx.y)
template <int ND, int MODEL, bool TAPE, bool NT, class Idx>
__global__ __launch_bounds__(256) void k_pressure_cell(DevSim batch, unsigned gx, GroupStep gs) {
    TileWork w{};
    if (gs.g) {
        const GroupBoundary& e = gs.g[blockIdx.y];
        w = tile_work(e, cell_tile<ND>(), e.step0 + gs.it + (gs.base ? *gs.base : 0));
    }
    const DevSim s = shot_view(batch, blockIdx.y);
    Idx c;
    if (cell_of_lane<ND, Idx>(s, cell_tile<ND>(), gx, c)) pressure_cell<ND, MODEL, TAPE, NT, Idx>(s, c);
    if (!gs.g) return;
    __syncthreads();
    tile_boundary(w);
}

// Source injection, then pressure release, then sensor gather, for step `n`. Sources that
// sit on a pressure-release point or repeat a later source are dropped on the host, and
// sensors on such points read the value written there, so no two threads touch one address.
// The shot is blockIdx.y.
__global__ __launch_bounds__(256) void k_boundary(DevSim s, DevBoundary b, int64_t n, int64_t rec_row) {
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int64_t shot = blockIdx.y;
    float* p = s.p + shot * s.shot_stride;
    const float* icmat_t = b.icmat_t + shot * b.icmat_stride;
    const bool inject = n < b.ntic;
    if (inject && t < b.ncoords) {
        const int64_t lin = b.src_lin[t];
        if (lin >= 0) p[lin] = icmat_t[n * b.ncoords + t];
    }
    if (t < b.nzero) p[b.zero_lin[t]] = 0.f;
    if (rec_row >= 0 && t < b.nout) {
        float val;
        if (b.out_air[t]) {
            val = 0.f;
        } else {
            const int32_t src = b.out_src[t];
            val = (inject && src >= 0) ? icmat_t[n * b.ncoords + src] : p[b.out_lin[t]];
        }
        b.rec[shot * b.rec_stride + rec_row * b.nout + t] = val;
    }
}

// The same pass with the step read from device memory (steps replayed from a captured graph).
__global__ __launch_bounds__(256) void k_boundary_dev(DevSim s, DevBoundary b, const int64_t* step, int64_t modt) {
    const int64_t n = *step;
    const int64_t rec_row = (modt > 0 && n % modt == 0) ? n / modt : -1;
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int64_t shot = blockIdx.y;
    float* p = s.p + shot * s.shot_stride;
    const float* icmat_t = b.icmat_t + shot * b.icmat_stride;
    const bool inject = n < b.ntic;
    if (inject && t < b.ncoords) {
        const int64_t lin = b.src_lin[t];
        if (lin >= 0) p[lin] = icmat_t[n * b.ncoords + t];
    }
    if (t < b.nzero) p[b.zero_lin[t]] = 0.f;
    if (rec_row >= 0 && t < b.nout) {
        float val;
        if (b.out_air[t]) {
            val = 0.f;
        } else {
            const int32_t src = b.out_src[t];
            val = (inject && src >= 0) ? icmat_t[n * b.ncoords + src] : p[b.out_lin[t]];
        }
        b.rec[shot * b.rec_stride + rec_row * b.nout + t] = val;
    }
}

// Advance (or set, with set >= 0) the device step counter; one lane writes it.
__global__ void k_tick(int64_t* step, int64_t set) {
    if (threadIdx.x == 0 && blockIdx.x == 0) *step = set >= 0 ? set : *step + 1;
}

// Add k to a device counter; one lane writes it.
__global__ void k_advance(int64_t* counter, int64_t k) {
    if (threadIdx.x == 0 && blockIdx.x == 0) *counter += k;
}

// One 16-byte element per lane: the fastest plain copy measured on the chip (a grid-stride loop
// over the same buffers reached 78 % of its rate).
__global__ __launch_bounds__(256) void k_copy(const float4* __restrict__ src, float4* __restrict__ dst, int64_t n) {
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t < n) dst[t] = src[t];
}

// `nr` read streams and `nw` write streams of one float per lane at the same element index: the
// access pattern of the stencil kernels' per-cell operands without their stencils (the velocity
// kernel of a 3D grid reads 12 such streams and writes 9).
__global__ __launch_bounds__(256) void k_streams(StreamSet a, int nr, int nw, int64_t n) {
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= n) return;
    float v[kMaxStreams];
#pragma unroll
    for (int r = 0; r < kMaxStreams; ++r) v[r] = r < nr ? a.r[r][t] : 0.f;
    float sum = 0.f;
#pragma unroll
    for (int r = 0; r < kMaxStreams; ++r) sum += v[r];
#pragma unroll
    for (int w = 0; w < kMaxStreams; ++w)
        if (w < nw) a.w[w][t] = sum * (float)(w + 1);
}

__global__ __launch_bounds__(256) void k_reciprocal(float* data, int64_t n) {
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t < n) data[t] = data[t] != 0.f ? 1.0f / data[t] : 0.f;  // zero: row padding
}

// Source signals from the file layout [shot][ncoords][ntic] (source-major) to the device
// layout [shot][ntic][ncoords] (one coalesced row per step), in 32 x 32 tiles through LDS:
// both the reads and the writes of a tile are row-contiguous. The grid strides over the tiles
// (every lane of a workgroup runs the same number of iterations, so the barriers are uniform).
__global__ __launch_bounds__(256) void k_transpose_icmat(const float* __restrict__ in, float* __restrict__ out,
                                                         int64_t nq, int64_t nt, int64_t ntiles) {
    __shared__ float tile[32][33];
    const int64_t tq = (nq + 31) / 32, tn = (nt + 31) / 32, per = tq * tn;
    const int tx = threadIdx.x % 32, ty = threadIdx.x / 32;  // ty: 0 .. 7
    for (int64_t t = blockIdx.x; t < ntiles; t += gridDim.x) {
        const int64_t b = t / per, r = t - b * per;
        const int64_t q0 = (r / tn) * 32, n0 = (r % tn) * 32;
        const float* src = in + b * nq * nt;
        float* dst = out + b * nq * nt;
        for (int k = ty; k < 32; k += 8) {
            const int64_t q = q0 + k, n = n0 + tx;
            if (q < nq && n < nt) tile[k][tx] = src[q * nt + n];
        }
        __syncthreads();
        for (int k = ty; k < 32; k += 8) {
            const int64_t n = n0 + k, q = q0 + tx;
            if (q < nq && n < nt) dst[n * nq + q] = tile[tx][k];
        }
        __syncthreads();
    }
}

}  // namespace

unsigned cell_tiles_x(const DevSim& s) {
    const int64_t n = s.ndim == 2 ? s.ny : s.nz;
    return (unsigned)((n + kCellTileCols - 1) / kCellTileCols);
}

int64_t cell_tiles(const DevSim& s) {
    return (cell_rows(s).count + kCellTileRows - 1) / kCellTileRows * cell_tiles_x(s);
}

int64_t cell_first_row(const DevSim& s) { return cell_rows(s).first; }
int64_t cell_row_count(const DevSim& s) { return cell_rows(s).count; }

template <int ND, int MODEL, bool TAPE, bool NT, class Idx>
static hipError_t launch_cell(const DevSim& s, bool velocity, const GroupStep& gs, hipStream_t st) {
    const int64_t tiles = cell_tiles(s);
    if (tiles > 0x7fffffff) return hipErrorInvalidValue;
    const dim3 g((unsigned)tiles, (unsigned)s.nshots), b(kCellTileCols * kCellTileRows);
    if (velocity) hipLaunchKernelGGL((k_velocity_cell<ND, MODEL, TAPE, NT, Idx>), g, b, 0, st, s, cell_tiles_x(s));
    else hipLaunchKernelGGL((k_pressure_cell<ND, MODEL, TAPE, NT, Idx>), g, b, 0, st, s, cell_tiles_x(s), gs);
    return hipGetLastError();
}

// Whether the memory variables go past the caches (non-temporal): in 3D where the arrays of a step (so many
// of 4 bytes a cell) exceed the memory-side cache of 256 MB by a third or more anyway; 2D grids of any
// size. us a step, past the caches / through them:
//   codes  112 x 120 x 100  59 / 47   128 x 136 x 128  77 / 61   180 x 170 x 180  212 / 234
//   maps   112 x 120 x 100  62 / 53   128 x 136 x 128  81 / 71   150 x 140 x 150  134 / 148
//   axes   112 x 120 x 100  64 / 60   128 x 136 x 128  96 / 101  150 x 160 x 170  207 / 217
static bool cell_memory_streams(const DevSim& s, int model) {
    return s.nx * s.sx * (int64_t)s.nshots * (model == kCellCoded ? 20 : model == kCellMaps ? 29 : 49) >= ((int64_t)20 << 22);
}

template <int ND, int MODEL, bool TAPE>
static hipError_t launch_cell_tape(const DevSim& s, bool velocity, const GroupStep& gs, hipStream_t st) {
    // 32-bit offsets where the grid (with the row padding of its last plane) has fewer than 2^30 cells
    if (s.nx * s.sx >= ((int64_t)1 << 30)) return launch_cell<ND, MODEL, TAPE, true, int64_t>(s, velocity, gs, st);
    if constexpr (ND == 3 && MODEL != kCellExpo) {  // (the exponential model has no memory variables)
        if (!cell_memory_streams(s, MODEL)) return launch_cell<ND, MODEL, TAPE, false, uint32_t>(s, velocity, gs, st);
    }
    return launch_cell<ND, MODEL, TAPE, true, uint32_t>(s, velocity, gs, st);
}

template <int ND, int MODEL>
static hipError_t launch_cell_model(const DevSim& s, bool velocity, const GroupStep& gs, hipStream_t st) {
    return s.tape_div ? launch_cell_tape<ND, MODEL, true>(s, velocity, gs, st)
                      : launch_cell_tape<ND, MODEL, false>(s, velocity, gs, st);
}

template <int ND>
static hipError_t launch_cell_nd(const DevSim& s, bool velocity, const GroupStep& gs, hipStream_t st) {
    if (s.aexp) return launch_cell_model<ND, kCellExpo>(s, velocity, gs, st);
    if (!s.isotropic) return launch_cell_model<ND, kCellAxes>(s, velocity, gs, st);
    if (s.rcode && s.rwide_v) return launch_cell_model<ND, kCellCoded>(s, velocity, gs, st);
    return launch_cell_model<ND, kCellMaps>(s, velocity, gs, st);
}

hipError_t launch_simple(const DevSim& s, bool velocity, const GroupStep& gs, hipStream_t st) {
    return s.ndim == 2 ? launch_cell_nd<2>(s, velocity, gs, st) : launch_cell_nd<3>(s, velocity, gs, st);
}

hipError_t load_cell_code() {
    hipFuncAttributes a;
    return hipFuncGetAttributes(&a, reinterpret_cast<const void*>(&k_reciprocal));
}

hipError_t launch_boundary(const DevSim& s, const DevBoundary& b, int64_t step, int64_t modt,
                           hipStream_t st) {
    // lanes for what this step does: a step between two records of the whole domain injects a few
    // points only
    const int64_t rec_row = (modt > 0 && step % modt == 0) ? step / modt : -1;
    int64_t n = b.nzero;
    if (step < b.ntic && b.ncoords > n) n = b.ncoords;
    if (rec_row >= 0 && b.nout > n) n = b.nout;
    if (n == 0) return hipSuccess;
    hipLaunchKernelGGL(k_boundary, dim3((unsigned)((n + 255) / 256), (unsigned)s.nshots), dim3(256), 0, st, s, b,
                       step, rec_row);
    return hipGetLastError();
}

hipError_t launch_boundary_dev(const DevSim& s, const DevBoundary& b, const int64_t* step, int64_t modt,
                               hipStream_t st) {
    int64_t n = b.ncoords;
    if (b.nzero > n) n = b.nzero;
    if (b.nout > n) n = b.nout;
    if (n == 0) return hipSuccess;
    hipLaunchKernelGGL(k_boundary_dev, dim3((unsigned)((n + 255) / 256), (unsigned)s.nshots), dim3(256), 0, st, s, b,
                       step, modt);
    return hipGetLastError();
}

hipError_t launch_streams(const StreamSet& a, int nr, int nw, int64_t n, hipStream_t st) {
    if (n <= 0) return hipSuccess;
    const int64_t blocks = (n + 255) / 256;
    if (blocks > 0x7fffffff) return hipErrorInvalidValue;
    hipLaunchKernelGGL(k_streams, dim3((unsigned)blocks), dim3(256), 0, st, a, nr, nw, n);
    return hipGetLastError();
}

hipError_t launch_tick(int64_t* step, int64_t set, hipStream_t st) {
    hipLaunchKernelGGL(k_tick, dim3(1), dim3(64), 0, st, step, set);
    return hipGetLastError();
}

hipError_t launch_advance(int64_t* counter, int64_t k, hipStream_t st) {
    hipLaunchKernelGGL(k_advance, dim3(1), dim3(64), 0, st, counter, k);
    return hipGetLastError();
}

hipError_t launch_copy(const void* src, void* dst, int64_t n16, hipStream_t st) {
    if (n16 == 0) return hipSuccess;
    const int64_t blocks = (n16 + 255) / 256;
    if (blocks > 0x7fffffff) return hipErrorInvalidValue;  // 2^39 bytes and more: not a probe size
    hipLaunchKernelGGL(k_copy, dim3((unsigned)blocks), dim3(256), 0, st, (const float4*)src, (float4*)dst, n16);
    return hipGetLastError();
}

hipError_t launch_transpose_icmat(const float* in, float* out, int64_t nshots, int64_t ncoords, int64_t ntic,
                                  hipStream_t st) {
    const int64_t ntiles = nshots * ((ncoords + 31) / 32) * ((ntic + 31) / 32);
    if (ntiles == 0) return hipSuccess;
    const int64_t blocks = ntiles < 256 * 64 ? ntiles : 256 * 64;
    hipLaunchKernelGGL(k_transpose_icmat, dim3((unsigned)blocks), dim3(256), 0, st, in, out, ncoords, ntic, ntiles);
    return hipGetLastError();
}

hipError_t launch_reciprocal(float* data, int64_t n, hipStream_t st) {
    if (n == 0) return hipSuccess;
    hipLaunchKernelGGL(k_reciprocal, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, data, n);
    return hipGetLastError();
}

}  // namespace fw
