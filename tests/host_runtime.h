// A host stand-in for the HIP runtime, for checks of the engine's host code under AddressSanitizer
// without a GPU: "device" memory is malloc'ed (so the sanitizer sees every access to it after its free
// or past its end), streams run at once, a captured graph is a list of launches, and time is a counter
// that each launch advances by a cost the check chooses. Kernels are known by their
// names. The stencil kernels compute nothing, but a pressure launch that does its tiles' boundary work
// does it for every tile of its grid, reading the point table as the device code does; the passes that the
// host code reads back (boundary, step counter, source transpose, coding) are carried out.
// Included by one source file, which is linked with the engine's sources compiled for the host only.
#pragma once
#include <cxxabi.h>

#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <functional>
#include <map>
#include <set>
#include <string>
#include <vector>

#include "../include/fullwave_hip.h"
#include "../fullwave25_amd/csrc/fw_sim.h"

namespace rt {

int failures = 0;
#define CHECK(cond)                                                                       \
    do {                                                                                  \
        if (!(cond)) {                                                                    \
            std::fprintf(stderr, "%s:%d: check failed: %s\n", __FILE__, __LINE__, #cond); \
            ++rt::failures;                                                               \
        }                                                                                 \
    } while (0)

// ---- kernels by name --------------------------------------------------------------------------
std::map<const void*, std::string>& names() {  // (filled by constructors of other source files)
    static std::map<const void*, std::string> m;
    return m;
}
// ---- memory -----------------------------------------------------------------------------------
struct Block {
    size_t bytes;
    bool async;
};
std::map<void*, Block> live;
bool async_fails = false;  // hipMallocAsync fails: the engine's fallback to hipMalloc
hipError_t get(void** p, size_t n, bool async) {
    *p = malloc(n ? n : 1);
    if (!*p) return hipErrorOutOfMemory;
    memset(*p, 0xa5, n);
    live[*p] = Block{n, async};
    return hipSuccess;
}
hipError_t put(void* p, bool async) {
    if (!p) return hipSuccess;
    auto it = live.find(p);
    CHECK(it != live.end());  // freed once
    if (it == live.end()) return hipErrorInvalidValue;
    CHECK(it->second.async == async);  // by the matching call
    live.erase(it);
    free(p);
    return hipSuccess;
}

// ---- launches ---------------------------------------------------------------------------------
struct Launch {
    std::string name;
    dim3 grid;
    std::vector<std::vector<char>> args;  // those that the check knows the size of
    template <class T>
    T arg(size_t i) const {
        T v;
        memcpy(&v, args.at(i).data(), sizeof(T));
        return v;
    }
    bool is(const char* prefix) const { return name.compare(0, strlen(prefix), prefix) == 0; }
    fw::DevSim sim() const { return arg<fw::DevSim>(0); }
};
struct Stream {
    bool capturing = false;
    std::vector<Launch> captured;
};
struct Graph {
    std::vector<Launch> l;
};
std::set<Stream*> streams;
std::set<Graph*> graphs;
double clock_us = 0;
std::function<double(const Launch&)> cost = [](const Launch&) { return 1.0; };
std::function<double(const std::string&)> load = [](const std::string&) { return 0.0; };  // of a kernel's code
std::vector<Launch> log;  // every launch carried out
bool keep_log = false;

template <class... T>
std::vector<std::vector<char>> take(void** a) {
    std::vector<std::vector<char>> out;
    size_t i = 0;
    (void)std::initializer_list<int>{(out.emplace_back((const char*)a[i], (const char*)a[i] + sizeof(T)), ++i, 0)...};
    return out;
}
using fw::DevBoundary;
using fw::DevSim;
using fw::GroupStep;
std::vector<std::vector<char>> args_of(const std::string& n, void** a) {
    auto is = [&](const char* p) { return n.compare(0, strlen(p), p) == 0; };
    if (is("k_velocity_cell")) return take<DevSim, unsigned>(a);
    if (is("k_pressure_cell")) return take<DevSim, unsigned, GroupStep>(a);
    if (is("k_velocity_brick")) return take<DevSim, uint32_t, uint32_t, bool>(a);
    if (is("k_pressure_brick")) return take<DevSim, uint32_t, uint32_t, bool, GroupStep>(a);
    if (is("k_velocity_tile_group") || is("k_pressure_tile_group") || is("k_velocity_2d_group") || is("k_pressure_2d_group")) return {};
    if (is("k_velocity_tile")) return take<DevSim>(a);
    if (is("k_pressure_tile")) return take<DevSim, GroupStep>(a);
    if (is("k_pressure_2d")) return take<DevSim, int, GroupStep>(a);
    if (is("k_velocity_2d") || is("k_velocity_3d") || is("k_pressure_3d") || is("k_velocity_pipe3d") || is("k_pressure_pipe3d"))
        return take<DevSim, int>(a);
    if (is("k_boundary_dev")) return take<DevSim, DevBoundary, const int64_t*, int64_t>(a);
    if (is("k_boundary")) return take<DevSim, DevBoundary, int64_t, int64_t>(a);
    if (is("k_tick") || is("k_advance")) return take<int64_t*, int64_t>(a);
    if (is("k_transpose_icmat")) return take<const float*, float*, int64_t, int64_t, int64_t>(a);
    if (is("k_out_of_range")) return take<const int32_t*, int64_t, int32_t, int32_t*>(a);
    if (is("k_maps_differ_tail")) return take<fw::MapPairs, int64_t, int64_t, int32_t*>(a);
    if (is("k_maps_differ")) return take<fw::MapPairs, int64_t, int32_t*>(a);
    if (is("k_code_insert"))
        return take<fw::CodeMaps, int64_t, unsigned long long*, uint32_t, uint32_t*, int32_t*, int32_t*>(a);
    if (is("k_code_compact"))
        return take<const unsigned long long*, const uint32_t*, const int32_t*, uint32_t, uint32_t*, uint32_t*, uint32_t*, int32_t*>(a);
    if (is("k_code_scatter")) return take<const uint32_t*, int32_t, uint16_t*>(a);
    if (is("k_code_assign"))
        return take<fw::CodeMaps, int64_t, const unsigned long long*, uint32_t, const uint16_t*, uint16_t*, int32_t*>(a);
    if (is("k_code_table")) return take<fw::CodeMaps, int32_t, const int32_t*, float*, float*>(a);
    return {};
}

// the boundary work of every tile of a pressure launch, as tile_work and tile_boundary do it
void boundary_of_tiles(const DevSim& s, const GroupStep& gs, size_t tiles) {
    for (int b = 0; b < s.nshots; ++b) {
        const fw::GroupBoundary e = gs.g[b];
        const int64_t n = e.step0 + gs.it + (gs.base ? *gs.base : 0);
        CHECK((size_t)e.ntiles == tiles);
        if ((size_t)e.ntiles != tiles) return;
        const bool inject = n < e.b.ntic;
        const float* icmat = e.b.icmat_t + n * e.b.ncoords;
        float* rec = e.modt > 0 && n % e.modt == 0 ? e.b.rec + (n / e.modt) * e.b.nout : nullptr;
        const size_t t1 = tiles + 1;
        auto lin = [](const int4& q) { return (int64_t)(((uint64_t)(uint32_t)q.w << 32) | (uint32_t)q.z); };
        for (size_t t = 0; t < tiles; ++t) {
            if (inject)
                for (int32_t k = e.off[t]; k < e.off[t + 1]; ++k) e.p[lin(e.src[k])] = icmat[e.src[k].x];
            for (int32_t k = e.off[t1 + t]; k < e.off[t1 + t + 1]; ++k) e.p[e.zero[k]] = 0.f;
            if (!rec) continue;
            for (int32_t k = e.off[2 * t1 + t]; k < e.off[2 * t1 + t + 1]; ++k) {
                const int4 q = e.out[k];
                rec[q.x] = lin(q) < 0 ? 0.f : inject && q.y >= 0 ? icmat[q.y] : e.p[lin(q)];
            }
        }
    }
}
void boundary_pass(const DevSim& s, const DevBoundary& b, int64_t n, int64_t row, int64_t threads) {
    for (int shot = 0; shot < s.nshots; ++shot) {
        float* p = s.p + shot * s.shot_stride;
        const float* ic = b.icmat_t + shot * b.icmat_stride;
        const bool inject = n < b.ntic;
        for (int64_t t = 0; t < threads; ++t)
            if (inject && t < b.ncoords && b.src_lin[t] >= 0) p[b.src_lin[t]] = ic[n * b.ncoords + t];
        for (int64_t t = 0; t < threads; ++t)
            if (t < b.nzero) p[b.zero_lin[t]] = 0.f;
        for (int64_t t = 0; t < threads; ++t)
            if (row >= 0 && t < b.nout)
                b.rec[shot * b.rec_stride + row * b.nout + t] =
                    b.out_air[t] ? 0.f : inject && b.out_src[t] >= 0 ? ic[n * b.ncoords + b.out_src[t]] : p[b.out_lin[t]];
    }
}

void tuple(const fw::CodeMaps& m, int64_t c, uint32_t (&t)[fw::kCodeVals]) {
    for (int k = 0; k < fw::kCodeVals - 1; ++k) memcpy(&t[k], &m.f[k][c], 4);
    t[fw::kCodeVals - 1] = (uint32_t)m.dcmap[c];
}
unsigned long long key_of(const fw::CodeMaps& m, int64_t c) {
    uint32_t t[fw::kCodeVals];
    tuple(m, c, t);
    unsigned long long h = 1469598103934665603ull;
    for (uint32_t v : t) h = (h ^ v) * 1099511628211ull;
    return h | 1;
}

void carry_out(const Launch& l) {
    clock_us += load(l.name) + cost(l);
    if (keep_log) log.push_back(l);
    auto touch = [](const DevSim& s) {  // the launch writes the whole state of a live handle
        volatile float* p = s.p;
        p[0] = p[0];
    };
    if (l.is("k_pressure_cell") || l.is("k_pressure_brick") || (l.is("k_pressure_tile") && !l.args.empty()) ||
        (l.is("k_pressure_2d") && !l.args.empty())) {
        touch(l.sim());
        const GroupStep gs = l.arg<GroupStep>(l.args.size() - 1);
        const bool flat = l.is("k_pressure_cell") || l.is("k_pressure_brick");
        if (gs.g) boundary_of_tiles(l.sim(), gs, flat ? l.grid.x : (size_t)l.grid.x * l.grid.y);
    } else if (l.is("k_boundary_dev")) {
        const int64_t n = *l.arg<const int64_t*>(2), modt = l.arg<int64_t>(3);
        boundary_pass(l.sim(), l.arg<DevBoundary>(1), n, modt > 0 && n % modt == 0 ? n / modt : -1, (int64_t)l.grid.x * 256);
    } else if (l.is("k_boundary")) {
        boundary_pass(l.sim(), l.arg<DevBoundary>(1), l.arg<int64_t>(2), l.arg<int64_t>(3), (int64_t)l.grid.x * 256);
    } else if (l.is("k_tick")) {
        int64_t* s = l.arg<int64_t*>(0);
        const int64_t set = l.arg<int64_t>(1);
        *s = set >= 0 ? set : *s + 1;
    } else if (l.is("k_advance")) {
        *l.arg<int64_t*>(0) += l.arg<int64_t>(1);
    } else if (l.is("k_transpose_icmat")) {
        const float* in = l.arg<const float*>(0);
        float* out = l.arg<float*>(1);
        const int64_t nq = l.arg<int64_t>(2), nt = l.arg<int64_t>(3), per = (nq + 31) / 32 * ((nt + 31) / 32);
        for (int64_t b = 0; b < l.arg<int64_t>(4) / per; ++b)
            for (int64_t q = 0; q < nq; ++q)
                for (int64_t n = 0; n < nt; ++n) out[(b * nt + n) * nq + q] = in[(b * nq + q) * nt + n];
    } else if (l.is("k_out_of_range")) {
        for (int64_t t = 0; t < l.arg<int64_t>(1); ++t) {
            const int32_t v = l.arg<const int32_t*>(0)[t];
            if (v < 0 || v >= l.arg<int32_t>(2)) *l.arg<int32_t*>(3) = 1;
        }
    } else if (l.is("k_maps_differ")) {
        const fw::MapPairs m = l.arg<fw::MapPairs>(0);
        const bool tail = l.is("k_maps_differ_tail");
        const int64_t from = tail ? l.arg<int64_t>(1) : 0, to = tail ? l.arg<int64_t>(2) : 4 * l.arg<int64_t>(1);
        for (int k = 0; k < m.n; ++k)
            if (memcmp(m.a[k] + from, m.b[k] + from, (size_t)(to - from) * 4)) *l.arg<int32_t*>(tail ? 3 : 2) = 1;
    } else if (l.is("k_code_insert")) {
        const fw::CodeMaps m = l.arg<fw::CodeMaps>(0);
        auto* keys = l.arg<unsigned long long*>(2);
        auto* count = l.arg<uint32_t*>(4);
        auto* rep = l.arg<int32_t*>(5);
        const uint32_t mask = l.arg<uint32_t>(3);
        std::map<unsigned long long, uint32_t> slots;
        for (int64_t c = 0; c < l.arg<int64_t>(1); ++c) {
            const unsigned long long h = key_of(m, c);
            auto it = slots.find(h);
            if (it == slots.end()) {
                if (slots.size() > mask / 2) {
                    l.arg<int32_t*>(6)[0] = 1;
                    return;
                }
                uint32_t q = (uint32_t)h & mask;
                while (keys[q]) q = (q + 1) & mask;
                keys[q] = h;
                it = slots.emplace(h, q).first;
                rep[q] = (int32_t)c;
            }
            ++count[it->second];
        }
    } else if (l.is("k_code_compact")) {
        uint32_t* n = l.arg<uint32_t*>(4);
        for (uint32_t q = 0; q < l.arg<uint32_t>(3); ++q) {
            if (!l.arg<const unsigned long long*>(0)[q]) continue;
            l.arg<uint32_t*>(5)[*n] = q;
            l.arg<uint32_t*>(6)[*n] = l.arg<const uint32_t*>(1)[q];
            l.arg<int32_t*>(7)[*n] = l.arg<const int32_t*>(2)[q];
            ++*n;
        }
    } else if (l.is("k_code_scatter")) {
        for (int32_t i = 0; i < l.arg<int32_t>(1); ++i) l.arg<uint16_t*>(2)[l.arg<const uint32_t*>(0)[i]] = (uint16_t)i;
    } else if (l.is("k_code_assign")) {
        const fw::CodeMaps m = l.arg<fw::CodeMaps>(0);
        const uint32_t mask = l.arg<uint32_t>(3);
        for (int64_t c = 0; c < l.arg<int64_t>(1); ++c) {
            const unsigned long long h = key_of(m, c);
            uint32_t q = (uint32_t)h & mask;
            while (l.arg<const unsigned long long*>(2)[q] != h) q = (q + 1) & mask;
            l.arg<uint16_t*>(5)[c] = l.arg<const uint16_t*>(4)[q];
        }
    } else if (l.is("k_code_table")) {
        const fw::CodeMaps m = l.arg<fw::CodeMaps>(0);
        for (int32_t i = 0; i < l.arg<int32_t>(1); ++i) {
            const int64_t c = l.arg<const int32_t*>(2)[i];
            for (int k = 0; k < 5; ++k) {
                l.arg<float*>(3)[i * fw::kCodeStride + k] = m.f[k][c];
                l.arg<float*>(4)[i * fw::kCodeStride + k] = m.f[5 + k][c];
            }
        }
    }
}

Stream* stream_of(hipStream_t s) {
    static Stream other;  // the null and the per-thread stream
    if (s == nullptr || s == hipStreamPerThread) return &other;
    Stream* q = reinterpret_cast<Stream*>(s);
    CHECK(streams.count(q));
    return streams.count(q) ? q : &other;
}

}  // namespace rt

// ---- the runtime's entry points ---------------------------------------------------------------
extern "C" {
void** __hipRegisterFatBinary(const void*) { return reinterpret_cast<void**>(1); }
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterVar(void**, void*, char*, const char*, int, size_t, int, int) {}
void __hipRegisterFunction(void**, const void* fn, char*, const char* name, unsigned, void*, void*, void*, void*, int*) {
    int st = 0;
    char* full = abi::__cxa_demangle(name, nullptr, nullptr, &st);
    std::string n = full ? full : name;
    free(full);
    const size_t k = n.find("k_");
    rt::names()[fn] = n.substr(k, n.find('(', k) - k);
}
static dim3 cfg_g, cfg_b;
static size_t cfg_m;
static hipStream_t cfg_s;
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t m, hipStream_t s) {
    cfg_g = g, cfg_b = b, cfg_m = m, cfg_s = s;
    return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3* g, dim3* b, size_t* m, hipStream_t* s) {
    *g = cfg_g, *b = cfg_b, *m = cfg_m, *s = cfg_s;
    return hipSuccess;
}
hipError_t hipLaunchKernel(const void* fn, dim3 g, dim3 b, void** a, size_t lds, hipStream_t s) {
    auto it = rt::names().find(fn);
    CHECK(it != rt::names().end());
    if (it == rt::names().end()) return hipErrorInvalidDeviceFunction;
    CHECK(g.x > 0 && g.y > 0 && g.z > 0 && b.x * b.y * b.z <= 1024 && lds <= (160u << 10));
    rt::Launch l{it->second, g, rt::args_of(it->second, a)};
    rt::Stream* q = rt::stream_of(s);
    if (q->capturing) q->captured.push_back(l);
    else rt::carry_out(l);
    return hipSuccess;
}
hipError_t hipFuncGetAttributes(hipFuncAttributes*, const void* fn) {
    auto it = rt::names().find(fn);
    CHECK(it != rt::names().end());
    if (it != rt::names().end()) rt::clock_us += rt::load(it->second);
    return hipSuccess;
}
hipError_t hipGetDeviceCount(int* n) { *n = 1; return hipSuccess; }
hipError_t hipGetDevice(int* d) { *d = 0; return hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
const char* hipGetErrorString(hipError_t e) { return e == hipSuccess ? "no error" : e == hipErrorInvalidValue ? "invalid argument" : "error"; }
hipError_t hipGetLastError(void) { return hipSuccess; }
hipError_t hipDeviceGetDefaultMemPool(hipMemPool_t* p, int) { *p = nullptr; return hipSuccess; }
hipError_t hipMemPoolSetAttribute(hipMemPool_t, hipMemPoolAttr, void*) { return hipSuccess; }
hipError_t hipMemGetInfo(size_t* f, size_t* t) { *f = *t = size_t(2) << 30; return hipSuccess; }
hipError_t hipMalloc(void** p, size_t n) { return rt::get(p, n, false); }
hipError_t hipMallocAsync(void** p, size_t n, hipStream_t) { return rt::async_fails ? hipErrorOutOfMemory : rt::get(p, n, true); }
hipError_t hipFree(void* p) { return rt::put(p, false); }
hipError_t hipFreeAsync(void* p, hipStream_t s) { rt::stream_of(s); return rt::put(p, true); }
hipError_t hipHostMalloc(void** p, size_t n, unsigned) { *p = malloc(n); return *p ? hipSuccess : hipErrorOutOfMemory; }
hipError_t hipHostFree(void* p) { free(p); return hipSuccess; }
hipError_t hipMemset(void* p, int v, size_t n) { memset(p, v, n); return hipSuccess; }
hipError_t hipMemsetAsync(void* p, int v, size_t n, hipStream_t s) {
    CHECK(!rt::stream_of(s)->capturing);
    memset(p, v, n);
    return hipSuccess;
}
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t st) {
    CHECK(!rt::stream_of(st)->capturing);
    memcpy(d, s, n);
    return hipSuccess;
}
hipError_t hipMemcpy2DAsync(void* d, size_t dp, const void* s, size_t sp, size_t w, size_t h, hipMemcpyKind, hipStream_t st) {
    CHECK(!rt::stream_of(st)->capturing && w <= dp && w <= sp);
    for (size_t i = 0; i < h; ++i) memcpy((char*)d + i * dp, (const char*)s + i * sp, w);
    return hipSuccess;
}
hipError_t hipGetSymbolAddress(void**, const void*) { return hipErrorInvalidSymbol; }
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) {
    auto* q = new rt::Stream();
    rt::streams.insert(q);
    *s = reinterpret_cast<hipStream_t>(q);
    return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t s) {
    rt::Stream* q = rt::stream_of(s);
    if (rt::streams.erase(q)) delete q;
    return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t s) { rt::stream_of(s); return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t* e) { *e = reinterpret_cast<hipEvent_t>(new double(0)); return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { return hipEventCreate(e); }
hipError_t hipEventDestroy(hipEvent_t e) { delete reinterpret_cast<double*>(e); return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t e, hipStream_t) { *reinterpret_cast<double*>(e) = rt::clock_us; return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float* ms, hipEvent_t a, hipEvent_t b) {
    *ms = (float)((*reinterpret_cast<double*>(b) - *reinterpret_cast<double*>(a)) * 1e-3);
    return hipSuccess;
}
hipError_t hipStreamBeginCapture(hipStream_t s, hipStreamCaptureMode) {
    rt::Stream* q = rt::stream_of(s);
    q->capturing = true;
    q->captured.clear();
    return hipSuccess;
}
hipError_t hipStreamEndCapture(hipStream_t s, hipGraph_t* g) {
    rt::Stream* q = rt::stream_of(s);
    q->capturing = false;
    auto* x = new rt::Graph{q->captured};
    rt::graphs.insert(x);
    *g = reinterpret_cast<hipGraph_t>(x);
    return hipSuccess;
}
hipError_t hipGraphInstantiate(hipGraphExec_t* e, hipGraph_t g, hipGraphNode_t*, char*, size_t) {
    auto* x = new rt::Graph(*reinterpret_cast<rt::Graph*>(g));
    rt::graphs.insert(x);
    *e = reinterpret_cast<hipGraphExec_t>(x);
    return hipSuccess;
}
static hipError_t drop_graph(rt::Graph* x) {
    CHECK(rt::graphs.erase(x) == 1);
    delete x;
    return hipSuccess;
}
hipError_t hipGraphDestroy(hipGraph_t g) { return drop_graph(reinterpret_cast<rt::Graph*>(g)); }
hipError_t hipGraphExecDestroy(hipGraphExec_t e) { return drop_graph(reinterpret_cast<rt::Graph*>(e)); }
hipError_t hipGraphLaunch(hipGraphExec_t e, hipStream_t) {
    for (const rt::Launch& l : reinterpret_cast<rt::Graph*>(e)->l) rt::carry_out(l);
    return hipSuccess;
}
}
