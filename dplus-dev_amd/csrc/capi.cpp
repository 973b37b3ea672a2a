// capi.cpp -- host side of libdplus_mi355x: device management, grid objects,
// the PDB amplitude builder driver, orientation-average drivers and the C ABI
// declared in include/dplus_mi355x.h.

#include <hip/hip_runtime.h>

#include <algorithm>
#include <chrono>
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <memory>
#include <mutex>
#include <random>
#include <tuple>
#include <stdexcept>
#include <string>
#include <vector>

#include "../../include/dplus_mi355x.h"
#include "common.hpp"
#include "device.hpp"

namespace dplus {

// ------------------------------------------------------------------ errors
static thread_local std::string g_last_error = "{\"code\":0,\"message\":\"\"}";

std::string json_escape(const std::string &s) {
    std::string o;
    for (char c : s) {
        if (c == '"' || c == '\\') {
            o += '\\';
            o += c;
        } else if (c == '\n') {
            o += "\\n";
        } else if ((unsigned char)c < 0x20) {
            char b[8];
            snprintf(b, sizeof b, "\\u%04x", c);
            o += b;
        } else {
            o += c;
        }
    }
    return o;
}

int set_error(int code, const std::string &msg) {
    g_last_error = "{\"code\":" + std::to_string(code) + ",\"message\":\"" + json_escape(msg) + "\"}";
    return code;
}

void check_hip(hipError_t e, const char *what) {
    if (e != hipSuccess) throw Error(kErrGeneral, std::string(what) + ": " + hipGetErrorString(e));
}

// ------------------------------------------------------------------ kernel timing
namespace {
struct TimingState {
    std::mutex mu;
    bool on = false;
    std::map<std::string, std::pair<long long, double>> acc;
    std::vector<std::tuple<std::string, hipEvent_t, hipEvent_t>> pending;
};
TimingState &timing() {
    static TimingState t;
    return t;
}
}  // namespace

KTimer::KTimer(const char *n, hipStream_t st) : name(n), s(st) {
    if (!timing().on) return;
    if (hipEventCreate(&e0) != hipSuccess || hipEventCreate(&e1) != hipSuccess) {
        e0 = e1 = nullptr;
        return;
    }
    (void)hipEventRecord(e0, s);
}

KTimer::~KTimer() {
    if (!e0) return;
    (void)hipEventRecord(e1, s);
    std::lock_guard<std::mutex> lk(timing().mu);
    timing().pending.emplace_back(name, e0, e1);
}

void timing_collect() {
    std::lock_guard<std::mutex> lk(timing().mu);
    for (auto &p : timing().pending) {
        float ms = 0.f;
        (void)hipEventSynchronize(std::get<2>(p));
        if (hipEventElapsedTime(&ms, std::get<1>(p), std::get<2>(p)) == hipSuccess) {
            auto &a = timing().acc[std::get<0>(p)];
            a.first++;
            a.second += ms;
        }
        (void)hipEventDestroy(std::get<1>(p));
        (void)hipEventDestroy(std::get<2>(p));
    }
    timing().pending.clear();
}

void timing_set(bool on) { timing().on = on; }
void timing_clear() {
    std::lock_guard<std::mutex> lk(timing().mu);
    timing().acc.clear();
}
void timing_read(const char *name, long long *n, double *ms) {
    std::lock_guard<std::mutex> lk(timing().mu);
    auto it = timing().acc.find(name);
    if (n) *n = it == timing().acc.end() ? 0 : it->second.first;
    if (ms) *ms = it == timing().acc.end() ? 0.0 : it->second.second;
}

// ------------------------------------------------------------------ device
Device &Device::get() {
    static Device d;
    return d;
}

Device::Device() {
    int n = 0;
    if (hipGetDeviceCount(&n) != hipSuccess || n == 0) {
        ok = false;
        return;
    }
    const char *env = getenv("DPLUS_DEVICE");
    id = env ? atoi(env) : 0;
    if (id >= n) id = 0;
    if (hipSetDevice(id) != hipSuccess) {
        ok = false;
        return;
    }
    hipDeviceProp_t p{};
    if (hipGetDeviceProperties(&p, id) == hipSuccess) {
        name = p.gcnArchName;
        cus = p.multiProcessorCount;
        mem = p.totalGlobalMem;
    }
    ok = hipStreamCreate(&stream) == hipSuccess;
    // keep freed pool memory cached for reuse instead of returning it at every sync
    hipMemPool_t pool;
    if (ok && hipDeviceGetDefaultMemPool(&pool, id) == hipSuccess) {
        uint64_t keep = UINT64_MAX;
        (void)hipMemPoolSetAttribute(pool, hipMemPoolAttrReleaseThreshold, &keep);
    }
}

void Device::require() {
    if (!ok) throw Error(kErrNoGpu, "no usable HIP device (libdplus_mi355x runs on the GPU only)");
    check_hip(hipSetDevice(id), "hipSetDevice");
}

static thread_local hipStream_t t_alloc_stream = nullptr;
hipStream_t alloc_stream() { return t_alloc_stream ? t_alloc_stream : Device::get().stream; }
void set_alloc_stream(hipStream_t s) { t_alloc_stream = s; }

CaptureMutex &capture_mutex() {
    static CaptureMutex m;
    return m;
}

static thread_local Arena *t_arena = nullptr;
void set_arena(Arena *a) { t_arena = a; }
static std::atomic<long long> g_device_allocs{0};
long long device_allocations() { return g_device_allocs.load(); }

DevBuf::~DevBuf() { release(); }
static void free_locked(void *&p, size_t &n, hipStream_t s) {
    if (p) (void)hipFreeAsync(p, s);
    p = nullptr;
    n = 0;
}
void DevBuf::release() {
    if (borrowed) {
        p = nullptr;
        n = 0;
        borrowed = false;
        return;
    }
    std::shared_lock<CaptureMutex> lk(capture_mutex());
    free_locked(p, n, s);
}
void DevBuf::ensure(size_t bytes) {
    if (bytes <= n) return;
    if (t_arena) {
        release();
        const size_t off = (t_arena->used + 255) & ~(size_t)255;
        if (off > t_arena->size || bytes > t_arena->size - off)
            throw Error(kErrInvalidArgs, "scratch exhausted: " + std::to_string(off + bytes) + " bytes needed, " +
                                             std::to_string(t_arena->size) + " available");
        p = t_arena->base + off;
        n = bytes;
        borrowed = true;
        t_arena->used = off + bytes;
        return;
    }
    std::shared_lock<CaptureMutex> lk(capture_mutex());
    if (borrowed) {
        p = nullptr;
        n = 0;
        borrowed = false;
    }
    free_locked(p, n, s);
    if (bytes == 0) return;
    g_device_allocs++;
    s = alloc_stream();
    const hipError_t e = hipMallocAsync(&p, bytes, s);
    if (e != hipSuccess) {
        p = nullptr;
        (void)hipGetLastError();
        throw Error(kErrOutOfMemory, "device allocation of " + std::to_string(bytes) + " bytes failed (" +
                                         hipGetErrorName(e) + ")");
    }
    n = bytes;
}
void DevBuf::upload(const void *src, size_t bytes, hipStream_t s) {
    ensure(bytes);
    if (!bytes) return;
    if (borrowed && t_arena && t_arena->stage((size_t)((char *)p - t_arena->base), src, bytes)) return;
    check_hip(hipMemcpyAsync(p, src, bytes, hipMemcpyHostToDevice, s), "hipMemcpyAsync H2D");
}

bool Arena::stage(size_t dev, const void *src, size_t bytes) {
    if (!staging) return false;
    // a run grows over the alignment padding between consecutive uploads (at most
    // 255 bytes, holding no buffer: a buffer carved between two uploads puts at
    // least 256 bytes between them), so staging mirrors the device layout
    size_t pad = 0;
    bool extend = false;
    if (!runs.empty()) {
        const Run &r = runs.back();
        const size_t end = r.dev + r.bytes;
        if (dev >= end && dev - end < 256) {
            pad = dev - end;
            extend = true;
        }
    }
    if (pad + bytes > staging_size - staged) return false;
    memset(staging + staged, 0, pad);
    memcpy(staging + staged + pad, src, bytes);
    if (extend)
        runs.back().bytes += pad + bytes;
    else
        runs.push_back({dev, staged, bytes});
    staged += pad + bytes;
    return true;
}

void Arena::flush(hipStream_t s) {
    for (const Run &r : runs)
        check_hip(hipMemcpyAsync(base + r.dev, staging + r.host, r.bytes, hipMemcpyHostToDevice, s), "H2D");
    runs.clear();
}

// spline multiplier tables, one set per shell count, kept for the process
struct SplineTables {
    DevBuf tab, off;
};
static std::mutex g_tab_mu;
static std::map<int, SplineTables *> g_tabs;

void build_spline_tables(int nshells, std::vector<double> &tab, std::vector<long long> &off);
void launch_splines(bool fp64, void *grid, int nshells, const double *tab, const long long *off,
                    hipStream_t s);

static SplineTables *tables_for(int nshells, hipStream_t s) {
    std::lock_guard<std::mutex> lk(g_tab_mu);
    auto it = g_tabs.find(nshells);
    if (it != g_tabs.end()) return it->second;
    std::vector<double> tab;
    std::vector<long long> off;
    build_spline_tables(nshells, tab, off);
    SplineTables *t = new SplineTables;
    t->tab.upload(tab.data(), tab.size() * sizeof(double), s);
    t->off.upload(off.data(), off.size() * sizeof(long long), s);
    check_hip(hipStreamSynchronize(s), "spline tables");
    g_tabs[nshells] = t;
    return t;
}

// ------------------------------------------------------------------ grid
Grid::Grid(int gs, double qm, int prec, bool zero) {
    if (gs % 2) gs++;
    if (gs < 2 || gs > 4000 || !(qm > 0)) throw Error(kErrInvalidArgs, "invalid grid size or qmax");
    grid_size = gs;
    qmax = qm;
    precision = prec;
    N = actual_size(gs);
    step = qmax / (double)(gs / 2);
    P = total_points(gs);
    Device::get().require();
    dev.ensure((size_t)P * node_bytes());
    if (zero) check_hip(hipMemsetAsync(dev.p, 0, (size_t)P * node_bytes(), alloc_stream()), "hipMemset");
}

void Grid::ensure_host() {
    if (host_data.size() != (size_t)(2 * P)) host_data.assign(2 * P, 0.0);
    if (host_interp.size() != (size_t)(2 * P)) host_interp.assign(2 * P, 0.0);
}

void launch_pack(bool fp64, const void *grid, long long n, double2 *data, double2 *coeffs, hipStream_t s);
void launch_unpack(bool fp64, const double2 *data, long long n, void *grid, hipStream_t s);

void Grid::splines(hipStream_t s, bool timed) {
    const SplineTables *t = spline_tables ? (const SplineTables *)spline_tables : tables_for(N, s);
    std::unique_ptr<KTimer> kt(timed ? new KTimer("splines", s) : nullptr);
    launch_splines(fp64(), dev.p, N, (const double *)t->tab.p, (const long long *)t->off.p, s);
    check_hip(hipGetLastError(), "splines launch");
}

// the tables live for the process, so the grid keeps their address
void Grid::prepare_splines(hipStream_t s) { spline_tables = tables_for(N, s); }

void Grid::download(hipStream_t s) {
    ensure_host();
    DevBuf tmp;
    tmp.ensure((size_t)P * 2 * sizeof(double2));
    double2 *d = (double2 *)tmp.p;
    launch_pack(fp64(), dev.p, P, d, d + P, s);
    check_hip(hipMemcpyAsync(host_data.data(), d, P * sizeof(double2), hipMemcpyDeviceToHost, s), "D2H");
    check_hip(hipMemcpyAsync(host_interp.data(), d + P, P * sizeof(double2), hipMemcpyDeviceToHost, s), "D2H");
    check_hip(hipStreamSynchronize(s), "download");
}

void Grid::upload(hipStream_t s) {
    ensure_host();
    DevBuf tmp;
    tmp.upload(host_data.data(), P * sizeof(double2), s);
    launch_unpack(fp64(), (const double2 *)tmp.p, P, dev.p, s);
    splines(s);
    check_hip(hipStreamSynchronize(s), "upload");
}

// ------------------------------------------------------------------ PDB builder
void launch_build_atoms(bool fp64, bool phase64, bool reduce, const void *atoms, const void *atoms64,
                        const int4 *tiles, int ntiles, const double *ff, int nion, const int4 *bdims,
                        const double *bcon, double vox, double step, long long nhalf, void *grid, double scale,
                        hipStream_t s);
void launch_set_origin(bool fp64, void *grid, double re, hipStream_t s);

// Atomic Form Factor.cpp:11-27 (cube-mean radius), 91-115 (dummy-atom
// solvent), 160-176 (4 Gaussians + c); evaluated in double per shell radius
void form_factor_table(const dplus_pdb_desc *d, const std::vector<int> &counts, int N, double step,
                       std::vector<double> &ff) {
    const int nion = d->nion;
    double rm = 0.0;
    if (d->flags & DPLUS_CALC_DUMMY_SOLVENT) {
        double num = 0.0, den = 0.0;
        for (int i = 0; i < nion; i++) {
            num += d->rad[i] * d->rad[i] * d->rad[i] * counts[i];
            den += counts[i];
        }
        rm = den > 0 ? std::cbrt(num / den) : 0.0;
    }
    ff.assign((size_t)(N + 1) * nion, 0.0);
    for (int s = 0; s <= N; s++) {
        const double q = s * step;
        const double sqq = q * q / (100.0 * 157.913670417429737901351855998);
        for (int i = 0; i < nion; i++) {
            const double *c = d->coef9 + 9 * i;
            double f = 0.0;
            if (d->flags & DPLUS_CALC_ATOMIC_FORMFACTORS) {
                f = c[8];
                for (int k = 0; k < 4; k++) f += c[2 * k] * std::exp(-sqq * c[2 * k + 1]);
            }
            double sv = 0.0;
            if (d->flags & DPLUS_CALC_DUMMY_SOLVENT) {
                const double r = d->rad[i];
                sv = 4.1887902047863909846 * r * r * r * std::exp(-(rm * rm) * (q * q) * 0.2067834969664667) *
                     d->sol_ed;
                sv *= d->c1 * d->c1 * d->c1 *
                      std::exp(-0.6822178052976590 * q * q * rm * rm * (d->c1 * d->c1 - 1.0));
            }
            ff[(size_t)s * nion + i] = f - sv;
        }
    }
}

namespace {
struct BoxSet {
    int n;
    const int *dims;
    const double *com;
    double contrast;
};

// order: the boxes by shape, then centre.  Counting sorts over the edges, which keep the order
// given: the voxelisation emits the boxes of a shape with rising centres, so those are checked and
// sorted only where they are not (118,000 boxes: 10 ms of comparisons -> 1 ms).
void sort_boxes(const BoxSet &B, std::vector<int> &order) {
    order.resize(B.n);
    for (int b = 0; b < B.n; b++) order[b] = b;
    auto centre = [&](int b) { return std::tie(B.com[3 * b], B.com[3 * b + 1], B.com[3 * b + 2]); };
    auto shape = [&](int b) { return std::tie(B.dims[3 * b], B.dims[3 * b + 1], B.dims[3 * b + 2]); };
    int lo = 0, hi = 0;
    for (size_t i = 0; i < 3 * (size_t)B.n; i++) {
        lo = std::min(lo, B.dims[i]);
        hi = std::max(hi, B.dims[i]);
    }
    if (lo < 0 || hi > 4 * B.n + 1024) {
        std::sort(order.begin(), order.end(), [&](int x, int y) {
            return shape(x) < shape(y) || (shape(x) == shape(y) && centre(x) < centre(y));
        });
        return;
    }
    std::vector<int> next(B.n);
    for (int a = 2; a >= 0; a--) {
        std::vector<int> at(hi + 2, 0);
        for (int b = 0; b < B.n; b++) at[B.dims[3 * b + a] + 1]++;
        for (int v = 0; v <= hi; v++) at[v + 1] += at[v];
        for (int b : order) next[at[B.dims[3 * b + a]]++] = b;
        order.swap(next);
    }
    for (int i = 0, e; i < B.n; i = e) {
        bool rising = true;
        for (e = i + 1; e < B.n && shape(order[e]) == shape(order[i]); e++)
            rising = rising && !(centre(order[e]) < centre(order[e - 1]));
        if (!rising)
            std::sort(order.begin() + i, order.begin() + e, [&](int x, int y) { return centre(x) < centre(y); });
    }
}

// Host side of MeshSources: the cell grid over every atom and box piece (cells of
// kMeshCell nm, larger along an axis where kMeshCells of them do not cover it, and where
// the table of cells would outgrow the sources), the atoms' order by (ion, cell) and the
// box pieces by cell.
struct MeshHost {
    bool ok = false;
    double lo[3] = {0, 0, 0}, hi[3] = {0, 0, 0}, cell0[3] = {0, 0, 0}, cell_inv[3] = {0, 0, 0}, half[3] = {0, 0, 0};
    int ncell[3] = {1, 1, 1}, cells = 1;
    long long npieces = 0;
    std::vector<int> fion, start;

    int cell(const double *p) const {
        int c[3];
        for (int a = 0; a < 3; a++)
            c[a] = std::min(ncell[a] - 1, std::max(0, (int)((p[a] - cell0[a]) * cell_inv[a])));
        return (c[0] * ncell[1] + c[1]) * ncell[2] + c[2];
    }

    // device bytes of [classes | cells | box pieces | edges], each 256-byte aligned
    size_t bytes() const {
        auto al = [](size_t b) { return (b + 255) & ~(size_t)255; };
        if (!ok) return 0;
        return al(fion.size() * sizeof(int)) + al(fion.size() * (size_t)(cells + 1) * sizeof(int)) +
               2 * al((size_t)npieces * sizeof(double4));
    }

    // the cuts of a box of edges len along each axis, at most kMeshPiece apart
    static double cut_box(const double len[3], double cut[3]) {
        double k = 1.0;
        for (int a = 0; a < 3; a++) k *= cut[a] = std::max(1.0, std::ceil(len[a] / kMeshPiece - 1e-9));
        return k;
    }

    // measure: extents, classes and the number of pieces alone
    MeshHost(const dplus_pdb_desc *d, bool atoms_on, const BoxSet *sets, bool measure = false) {
        double c_lo[3], c_hi[3];  // of the centres
        for (int a = 0; a < 3; a++) {
            c_lo[a] = 1e300;
            c_hi[a] = -1e300;
        }
        auto see = [&](const double *p) {
            for (int a = 0; a < 3; a++) {
                c_lo[a] = std::min(c_lo[a], p[a]);
                c_hi[a] = std::max(c_hi[a], p[a]);
            }
            return std::isfinite(p[0]) && std::isfinite(p[1]) && std::isfinite(p[2]);
        };
        if (atoms_on) {
            std::vector<char> used(d->nion, 0);
            for (int a = 0; a < d->natoms; a++) {
                if (!see(d->xyz + 3 * a) || d->ion[a] < 0 || d->ion[a] >= d->nion) return;
                used[d->ion[a]] = 1;
            }
            for (int i = 0; i < d->nion; i++)
                if (used[i]) fion.push_back(i);
        }
        // pieces: a piece costs the host about 60 ns and a build about 2 ns, a source 0.7 us
        // (FP64 4.4) of a direct sum at the largest usual grid; boxes of many more pieces than
        // this stay whole
        const size_t boxes = (size_t)sets[0].n + sets[1].n;
        const size_t most = 64 * boxes + 16 * (size_t)(atoms_on ? d->natoms : 0) + 4096;
        for (int si = 0; si < 2; si++)
            for (int b = 0; b < sets[si].n; b++) {
                const int *n = sets[si].dims + 3 * b;
                const double *com = sets[si].com + 3 * b;
                if (n[0] < 0 || n[1] < 0 || n[2] < 0) return;
                if (n[0] == 0 || n[1] == 0 || n[2] == 0) continue;  // no volume
                double cut[3], end[3];
                const double len[3] = {n[0] * d->vox_step, n[1] * d->vox_step, n[2] * d->vox_step};
                const double k = cut_box(len, cut);
                if (!(k + (double)npieces <= (double)most)) return;
                npieces += (long long)k;
                for (int a = 0; a < 3; a++) half[a] = std::max(half[a], 0.5 * len[a] / cut[a]);
                for (int sgn = -1; sgn <= 1; sgn += 2) {  // the outermost pieces' centres
                    for (int a = 0; a < 3; a++) end[a] = com[a] + sgn * 0.5 * (cut[a] - 1.0) * (len[a] / cut[a]);
                    if (!see(end)) return;
                }
            }
        if (npieces > 0) fion.push_back(-1);
        if (fion.empty() || fion.size() > (size_t)kMeshFields) return;
        double size[3];
        for (int a = 0; a < 3; a++) {
            size[a] = std::max(kMeshCell, (c_hi[a] - c_lo[a]) / kMeshCells * (1.0 + 1e-9));
            if (!std::isfinite(size[a])) return;
        }
        const double room = 2.0 * ((double)(atoms_on ? d->natoms : 0) + (double)npieces) + 8192.0;
        for (;;) {
            cells = 1;
            for (int a = 0; a < 3; a++) {
                cell_inv[a] = 1.0 / size[a];
                ncell[a] = std::min(kMeshCells, (int)((c_hi[a] - c_lo[a]) * cell_inv[a]) + 1);
                cells *= ncell[a];
            }
            if (cells == 1 || (double)fion.size() * (cells + 1.0) <= room) break;
            for (int a = 0; a < 3; a++) size[a] *= 1.26;
        }
        for (int a = 0; a < 3; a++) {
            cell0[a] = c_lo[a];
            lo[a] = c_lo[a] - half[a];
            hi[a] = c_hi[a] + half[a];
        }
        ok = true;
        if (measure) return;
        start.assign(fion.size() * (cells + 1), 0);
    }

    // every piece of every box, in order: f(box set, centre, edges)
    template <typename F>
    static void each_piece(const dplus_pdb_desc *d, const BoxSet *sets, F f) {
        for (int si = 0; si < 2; si++)
            for (int b = 0; b < sets[si].n; b++) {
                const int *n = sets[si].dims + 3 * b;
                const double *com = sets[si].com + 3 * b;
                if (n[0] == 0 || n[1] == 0 || n[2] == 0) continue;
                double cut[3], len[3] = {n[0] * d->vox_step, n[1] * d->vox_step, n[2] * d->vox_step};
                cut_box(len, cut);
                for (int a = 0; a < 3; a++) len[a] /= cut[a];
                for (int x = 0; x < (int)cut[0]; x++)
                    for (int y = 0; y < (int)cut[1]; y++)
                        for (int z = 0; z < (int)cut[2]; z++) {
                            const double p[3] = {com[0] + (x - 0.5 * (cut[0] - 1.0)) * len[0],
                                                 com[1] + (y - 0.5 * (cut[1] - 1.0)) * len[1],
                                                 com[2] + (z - 0.5 * (cut[2] - 1.0)) * len[2]};
                            f(si, p, len);
                        }
            }
    }

    // the pieces sorted by cell, written where they are uploaded from, and their cells' starts
    void place_pieces(const dplus_pdb_desc *d, const BoxSet *sets, double4 *pieces, double4 *lens) {
        if (npieces == 0) return;
        int *st = &start[(fion.size() - 1) * (cells + 1)];
        std::vector<int> key;
        key.reserve(npieces);
        each_piece(d, sets, [&](int, const double *p, const double *) {
            key.push_back(cell(p));
            st[key.back() + 1]++;
        });
        for (int c = 0; c < cells; c++) st[c + 1] += st[c];
        std::vector<int> at(st, st + cells);
        size_t i = 0;
        each_piece(d, sets, [&](int si, const double *p, const double *len) {
            const int k = at[key[i++]]++;
            pieces[k] = make_double4(p[0], p[1], p[2], sets[si].contrast);
            lens[k] = make_double4(len[0], len[1], len[2], 0.0);
        });
    }

    MeshSources sources(long long natoms) const {
        MeshSources m;
        m.ok = ok;
        m.nfield = (int)fion.size();
        m.natoms = natoms;
        m.npieces = npieces;
        for (int a = 0; a < 3; a++) {
            m.lo[a] = lo[a];
            m.hi[a] = hi[a];
            m.cell0[a] = cell0[a];
            m.ncell[a] = ncell[a];
            m.cell_inv[a] = cell_inv[a];
            m.piece_half[a] = half[a];
        }
        return m;
    }

    // order: atoms by (ion, cell), stable; start: every used ion's cells
    void sort_atoms(const dplus_pdb_desc *d, std::vector<int> &order) {
        std::vector<int> field(d->nion, 0), key(d->natoms);
        for (size_t f = 0; f < fion.size(); f++)
            if (fion[f] >= 0) field[fion[f]] = (int)f;
        const int n = cells + 1;
        for (int a = 0; a < d->natoms; a++) {
            key[a] = field[d->ion[a]] * n + cell(d->xyz + 3 * a);
            start[key[a] + 1]++;
        }
        int sum = 0;
        for (size_t f = 0; f < fion.size() && fion[f] >= 0; f++) {
            int *st = &start[f * n];
            st[0] = sum;
            for (int c = 0; c < cells; c++) st[c + 1] += st[c];
            sum = st[cells];
        }
        std::vector<int> at(start);
        for (int a = 0; a < d->natoms; a++) order[at[key[a]]++] = a;
    }
};
}  // namespace

Structure::Structure(const dplus_pdb_desc *d, hipStream_t s, bool with_mesh) {
    if (d->natoms < 0 || d->nion <= 0 || d->nion > 255) throw Error(kErrInvalidArgs, "bad atom/ion counts");
    if (d->nbox < 0 || (d->nbox > 0 && (!d->box_dims || !d->box_com || !(d->vox_step > 0))))
        throw Error(kErrInvalidArgs, "bad solvent boxes");
    if (d->nexcl < 0 || (d->nexcl > 0 && (!d->excl_dims || !d->excl_com || !(d->vox_step > 0))))
        throw Error(kErrInvalidArgs, "bad excluded-volume boxes");
    for (int a = 0; a < d->natoms; a++)
        if (d->ion[a] < 0 || d->ion[a] >= d->nion) throw Error(kErrInvalidArgs, "ion index out of range");
    const bool atoms_on = (d->flags & (DPLUS_CALC_ATOMIC_FORMFACTORS | DPLUS_CALC_DUMMY_SOLVENT)) && d->natoms > 0;
    // box sets: the outer-solvent (hydration) layer added with box_contrast and the
    // excluded volume added with excl_contrast (PDBAmplitude.cpp:277-314)
    const BoxSet sets[2] = {{d->box_contrast != 0.0 ? d->nbox : 0, d->box_dims, d->box_com, d->box_contrast},
                            {d->excl_contrast != 0.0 ? d->nexcl : 0, d->excl_dims, d->excl_com, d->excl_contrast}};
    const bool boxes_on = sets[0].n > 0 || sets[1].n > 0;
    // atoms sorted by ion (ExtractRelevantCoeffs, PDBReaderLib.cpp:1443-1509), stably:
    // a counting sort over the ion index; then each box set sorted by shape
    // (SortSolventBoxEntry, PDBAmplitude.cpp:161-188)
    // and, within an ion, by cell of the mesh builder
    MeshHost mh(d, atoms_on, sets);
    std::vector<int> order(d->natoms);
    if (!atoms_on || !mh.ok) {
        std::vector<int> start(d->nion + 1, 0);
        for (int a = 0; a < d->natoms; a++) start[d->ion[a] + 1]++;
        for (int i = 0; i < d->nion; i++) start[i + 1] += start[i];
        for (int a = 0; a < d->natoms; a++) order[start[d->ion[a]]++] = a;
    } else {
        mh.sort_atoms(d, order);
    }
    if (!with_mesh) mh.ok = false;  // (the same order of atoms, so the same bits of a direct build)
    std::vector<int> border[2];
    for (int si = 0; si < 2; si++) {
        const BoxSet &B = sets[si];
        sort_boxes(B, border[si]);
    }
    const size_t nsrc = (atoms_on ? d->natoms : 0) + border[0].size() + border[1].size();
    // one allocation and one upload: [sources float4 | sources double4 | tiles | box shapes | contrasts]
    // and the mesh builder's [classes | cells | box pieces | edges], each section 256-byte aligned and
    // written in place (the staging is reserved for as many tiles and shapes as sources)
    auto al = [](size_t b) { return (b + 255) & ~(size_t)255; };
    const size_t nput = std::max<size_t>(1, nsrc);
    const size_t o64 = al(nput * sizeof(float4)), ot = o64 + al(nput * sizeof(double4));
    const std::unique_ptr<char[]> hostp(
        new char[ot + 2 * al((nput + 1) * sizeof(int4)) + al((nput + 1) * sizeof(double)) + mh.bytes() + 1024]);
    char *const host = hostp.get();
    float4 *const at32 = (float4 *)host;
    double4 *const at64 = (double4 *)(host + o64);
    at32[0] = make_float4(0.f, 0.f, 0.f, 0.f);
    at64[0] = make_double4(0.0, 0.0, 0.0, 0.0);
    std::vector<int> counts(d->nion, 0);
    for (int a = 0; a < d->natoms; a++) counts[d->ion[a]]++;
    std::vector<int4> tiles, bdims;
    std::vector<double> bcon;
    size_t k = 0;
    if (atoms_on) {
        for (int i = 0; i < d->natoms; i++) {
            const double *p = d->xyz + 3 * order[i];
            at32[k] = make_float4((float)p[0], (float)p[1], (float)p[2], 0.f);
            at64[k] = make_double4(p[0], p[1], p[2], 0.0);
            k++;
        }
        int i = 0;
        while (i < d->natoms) {
            const int ion = d->ion[order[i]];
            int e = i;
            while (e < d->natoms && d->ion[order[e]] == ion && e - i < 256) e++;
            tiles.push_back(make_int4(i, e - i, ion, 0));
            i = e;
        }
    }
    double box_origin = 0.0;
    for (int si = 0; si < 2; si++) {
        const BoxSet &B = sets[si];
        const std::vector<int> &bo = border[si];
        if (bo.empty()) continue;
        const size_t base = k;
        double volume = 0.0;
        for (int b : bo) {
            const double *p = B.com + 3 * b;
            at32[k] = make_float4((float)p[0], (float)p[1], (float)p[2], 0.f);
            at64[k] = make_double4(p[0], p[1], p[2], 0.0);
            volume += (double)B.dims[3 * b] * B.dims[3 * b + 1] * B.dims[3 * b + 2];
            k++;
        }
        box_origin += B.contrast * volume * d->vox_step * d->vox_step * d->vox_step;
        size_t i = 0;
        while (i < bo.size()) {
            const int *di = B.dims + 3 * bo[i];
            bdims.push_back(make_int4(di[0], di[1], di[2], si));
            bcon.push_back(B.contrast);
            size_t e = i;
            while (e < bo.size() && e - i < 256) {
                const int *de = B.dims + 3 * bo[e];
                if (de[0] != di[0] || de[1] != di[1] || de[2] != di[2]) break;
                e++;
            }
            tiles.push_back(make_int4((int)(base + i), (int)(e - i), (int)bdims.size() - 1, 1));
            i = e;
        }
    }
    if (bdims.empty()) {
        bdims.push_back(make_int4(0, 0, 0, 0));
        bcon.push_back(0.0);
    }
    desc = *d;
    desc.xyz = nullptr;
    desc.ion = nullptr;
    desc.box_dims = nullptr;
    desc.box_com = nullptr;
    desc.excl_dims = nullptr;
    desc.excl_com = nullptr;
    coef9.assign(d->coef9, d->coef9 + 9 * d->nion);
    rad.assign(d->rad, d->rad + d->nion);
    desc.coef9 = coef9.data();
    desc.rad = rad.data();
    ion_counts = counts;
    this->box_origin = box_origin;
    this->atoms_on = atoms_on;
    this->boxes_on = boxes_on;
    ntiles = (int)tiles.size();
    tile_len.resize(tiles.size());
    for (size_t t = 0; t < tiles.size(); t++) tile_len[t] = tiles[t].y;
    nsources = (long long)nsrc;
    rmax = 0.0;
    for (size_t i = 0; i < nsrc; i++)
        rmax = std::max(rmax, std::sqrt(at64[i].x * at64[i].x + at64[i].y * at64[i].y + at64[i].z * at64[i].z));
    if (tiles.empty()) tiles.push_back(make_int4(0, 0, 0, 0));
    const size_t od = ot + al(tiles.size() * sizeof(int4));
    const size_t oc = od + al(bdims.size() * sizeof(int4));
    const size_t of = al(oc + bcon.size() * sizeof(double));
    const size_t os = al(of + mh.fion.size() * sizeof(int));
    const size_t op = al(os + mh.start.size() * sizeof(int));
    const size_t ol = al(op + mh.npieces * sizeof(double4));
    const size_t total = mh.ok ? ol + mh.npieces * sizeof(double4) : of;
    if (mh.ok) {
        mh.place_pieces(d, sets, (double4 *)(host + op), (double4 *)(host + ol));
        memcpy(host + of, mh.fion.data(), mh.fion.size() * sizeof(int));
        memcpy(host + os, mh.start.data(), mh.start.size() * sizeof(int));
    }
    memcpy(host + ot, tiles.data(), tiles.size() * sizeof(int4));
    memcpy(host + od, bdims.data(), bdims.size() * sizeof(int4));
    memcpy(host + oc, bcon.data(), bcon.size() * sizeof(double));
    blob.upload(host, total, s);
    char *base = (char *)blob.p;
    d32 = (const float4 *)base;
    d64 = (const double4 *)(base + o64);
    dtiles = (const int4 *)(base + ot);
    ddims = (const int4 *)(base + od);
    dcon = (const double *)(base + oc);
    if (mh.ok) {
        mesh = mh.sources(atoms_on ? d->natoms : 0);
        mesh.fion = (const int *)(base + of);
        mesh.cells = (const int *)(base + os);
        mesh.pieces = (const double4 *)(base + op);
        mesh.lens = (const double4 *)(base + ol);
    }
    check_hip(hipStreamSynchronize(s), "structure upload");
}

// ------------------------------------------------------------------ builder shapes
// Shape table of the paired builder's autotuner: the fastest measured launch
// shape per (grid shells, tile-count class); the class is the tile count's
// half-octave, so structures of similar size share an entry.
namespace {
std::mutex shape_mu;
std::map<std::pair<int, int>, BuildShape> shape_table;

int tile_class(int ntiles) { return (int)std::floor(2.0 * std::log2((double)std::max(ntiles, 1))); }
}  // namespace

bool shape_lookup(int nshells, int ntiles, BuildShape *out) {
    std::lock_guard<std::mutex> lk(shape_mu);
    auto it = shape_table.find({nshells, tile_class(ntiles)});
    if (it == shape_table.end()) return false;
    *out = it->second;
    return true;
}

void shape_record(int nshells, int ntiles, BuildShape shape) {
    std::lock_guard<std::mutex> lk(shape_mu);
    shape_table[{nshells, tile_class(ntiles)}] = shape;
}

BuildShape Structure::shape_for(const Grid &g, bool use_table) const {
    BuildShape sh;
    // the shape table holds the mixed builder's tuned shapes; FP64 builds take the model
    if (!g.fp64() && use_table && shape_lookup(g.N, ntiles, &sh)) return sh;
    sh.wg = 256;
    sh.slices = pair_slices(pair_units(half_base(g.N + 1)), ntiles, sh.wg, g.fp64());
    return sh;
}

// The mesh builder where it is the faster one, within kMeshRoom bytes of workspace or what
// the direct builder's slice partials may take.  DPLUS_BUILD_ROUTE in the environment (a
// diagnostic, as DPLUS_PHASE64 is): "direct" keeps every build direct, "mesh" takes the mesh
// wherever it has a plan.
size_t direct_build_bytes(int N) { return (size_t)kMaxSlices * 12 * pair_units(half_base(N + 1)) * sizeof(double); }

static bool mesh_route_of(const MeshSources &S, long long nsources, int N, double step, bool fp64, int nion, MeshPlan &P,
                          MeshSizes &Z) {
    const char *env = getenv("DPLUS_BUILD_ROUTE");
    const std::string route = env ? env : "";
    return route != "direct" &&
           mesh_plan(S, N, step, fp64, nion, std::max(kMeshRoom, direct_build_bytes(N)), P, Z) &&
           (route == "mesh" || mesh_pays(P, Z, N, (double)nsources, fp64));
}

bool Structure::mesh_route(const Grid &g, MeshPlan &P, MeshSizes &Z) const {
    return mesh_route_of(mesh, nsources, g.N, g.step, g.fp64(), desc.nion, P, Z);
}

size_t mesh_build_bytes(const dplus_pdb_desc *d, int grid_size, double qmax, bool fp64, size_t &held) {
    const bool atoms_on = (d->flags & (DPLUS_CALC_ATOMIC_FORMFACTORS | DPLUS_CALC_DUMMY_SOLVENT)) && d->natoms > 0;
    const BoxSet sets[2] = {{d->box_contrast != 0.0 ? d->nbox : 0, d->box_dims, d->box_com, d->box_contrast},
                            {d->excl_contrast != 0.0 ? d->nexcl : 0, d->excl_dims, d->excl_com, d->excl_contrast}};
    if (grid_size % 2) grid_size++;
    const int N = actual_size(grid_size);
    const MeshHost mh(d, atoms_on, sets, true);
    held = mh.bytes();
    MeshPlan P;
    MeshSizes Z;
    return mesh_route_of(mh.sources(atoms_on ? d->natoms : 0), (atoms_on ? d->natoms : 0) + (long long)sets[0].n + sets[1].n,
                         N, qmax / (double)(grid_size / 2), fp64, d->nion, P, Z)
               ? Z.bytes
               : 0;
}

BuildJob Structure::prepare(Grid &g, int slices, Pending &P, hipStream_t s, bool direct) const {
    std::vector<double> ff;
    form_factor_table(&desc, ion_counts, g.N, g.step, ff);
    // origin: sum of f~(0) over atoms + each box set's contrast * total volume
    P.origin = 0.0;
    if (atoms_on)
        for (int i = 0; i < desc.nion; i++) P.origin += ion_counts[i] * ff[i];
    if (boxes_on) P.origin += box_origin;
    MeshJob &M = P.job;
    P.mesh = !direct && mesh_route(g, M.plan, M.z);
    if (P.mesh) {
        try {
            P.part.ensure(M.z.bytes);
        } catch (const Error &) {  // no room for the workspace: the direct sum takes less
            P.mesh = false;
        }
    }
    if (P.mesh) {
        std::vector<MeshBand> bands;
        mesh_bands(M.plan, M.z, g.N, g.fp64(), bands, M.ntiles);
        // one upload: [form factors | tables | bands]
        const size_t nf = ff.size();
        ff.resize(nf + M.z.tab);
        mesh_tables(M.plan, g.fp64(), ff.data() + nf);
        const size_t bytes = ff.size() * sizeof(double);
        ff.resize(ff.size() + (bands.size() * sizeof(MeshBand) + 7) / 8);
        memcpy((char *)ff.data() + bytes, bands.data(), bands.size() * sizeof(MeshBand));
        P.ff.upload(ff.data(), ff.size() * sizeof(double), s);
        M.atoms = d64;
        M.pieces = mesh.pieces;
        M.lens = mesh.lens;
        M.natoms = mesh.natoms;
        M.npieces = mesh.npieces;
        M.cells = mesh.cells;
        M.fion = mesh.fion;
        M.ff = (const double *)P.ff.p;
        M.tab = M.ff + nf;
        M.bands = (const MeshBand *)((const char *)P.ff.p + bytes);
        M.nbands = (int)bands.size();
        M.work = P.part.p;
        M.grid = g.dev.p;
        M.scale = desc.scale;
        return BuildJob{};
    }
    // unreduced hardware sin/cos while every phase stays below 128 revolutions
    const double qtop = (double)(g.N + 1) * g.step;
    P.reduce = !g.fp64() && (qtop * rmax / k2Pi >= 128.0 || getenv("DPLUS_REDUCE_PHASE") != nullptr);
    P.ff.upload(ff.data(), ff.size() * sizeof(double), s);
    const long long nunits = pair_units(half_base(g.N + 1));
    const int S = std::max(1, std::min({slices, kMaxSlices, std::max(ntiles, 1)}));
    P.part.ensure((size_t)S * 12 * nunits * sizeof(double));
    BuildJob J{};
    J.atoms = d32;
    J.atoms64 = d64;
    J.fp64 = g.fp64() ? 1 : 0;
    J.tiles = dtiles;
    J.ff = (const double *)P.ff.p;
    J.bdims = ddims;
    J.bcon = dcon;
    J.partial = (double *)P.part.p;
    J.grid = g.fp64() ? nullptr : (float4 *)g.dev.p;
    J.grid64 = g.fp64() ? (double4 *)g.dev.p : nullptr;
    J.nunits = nunits;
    J.vox = desc.vox_step;
    J.step = g.step;
    J.scale = desc.scale;
    J.nion = desc.nion;
    J.nslices = S;
    // atom slices of roughly equal work (a tile costs its terms + 8 for its fold)
    for (int y = 0; y <= S; y++) J.slice_begin[y] = ntiles;
    J.slice_begin[0] = 0;
    double total = 0.0;
    for (int t = 0; t < ntiles; t++) total += tile_len[t] + 8.0;
    double acc = 0.0;
    for (int t = 0, y = 1; t < ntiles && y < S; t++) {
        acc += tile_len[t] + 8.0;
        while (y < S && acc >= total * y / S) J.slice_begin[y++] = t + 1;
    }
    return J;
}

void Structure::launch(Grid &g, BuildJob &J, int wg, const Pending &P, hipStream_t s) const {
    if (P.mesh)
        launch_mesh(P.job, g.fp64(), s);
    else
        launch_build_batch(P.reduce, wg, &J, 1, s);
    check_hip(hipGetLastError(), "build launch");
}

void Structure::enqueue_finish(Grid &g, const Pending &P, hipStream_t s, bool timed) const {
    launch_set_origin(g.fp64(), g.dev.p, P.origin * desc.scale, s);
    check_hip(hipGetLastError(), "set_origin launch");
    g.splines(s, timed);
}

void Structure::finish(Grid &g, const Pending &P, bool host_copy, hipStream_t s) const {
    enqueue_finish(g, P, s, true);
    // the per-build buffers are released after the stream has drained
    if (host_copy)
        g.download(s);
    else
        check_hip(hipStreamSynchronize(s), "pdb build");
}

void Structure::build(Grid &g, bool host_copy, hipStream_t s, bool use_table, bool direct) {
    const bool phase64 = getenv("DPLUS_PHASE64") != nullptr;
    // paired builder: every mixed grid (but the FP64-phase diagnostic) and, unless
    // the plain form is selected, every FP64 grid
    if (g.fp64() ? !fp64_plain_builder() : !phase64) {
        // per-build buffers (form factors of this grid's shells, slice partials): a
        // structure can be built into several grids at once on different streams
        Pending P;
        const BuildShape sh = shape_for(g, use_table);
        BuildJob J = prepare(g, sh.slices, P, s, direct);
        {
            KTimer kt("build", s);
            launch(g, J, sh.wg, P, s);
        }
        finish(g, P, host_copy, s);
        timing_collect();
        return;
    }
    std::vector<double> ff;
    form_factor_table(&desc, ion_counts, g.N, g.step, ff);
    double origin = 0.0;
    if (atoms_on)
        for (int i = 0; i < desc.nion; i++) origin += ion_counts[i] * ff[i];
    if (boxes_on) origin += box_origin;
    DevBuf bff;
    bff.upload(ff.data(), ff.size() * sizeof(double), s);
    const long long nhalf = half_base(g.N + 1);
    {
        KTimer kt("build", s);
        const double qtop = (double)(g.N + 1) * g.step;
        const bool reduce = qtop * rmax / k2Pi >= 128.0 || getenv("DPLUS_REDUCE_PHASE") != nullptr;
        launch_build_atoms(g.fp64(), phase64, reduce, d32, d64, dtiles, ntiles,
                           (const double *)bff.p, desc.nion, ddims, dcon, desc.vox_step,
                           g.step, nhalf, g.dev.p, desc.scale, s);
        check_hip(hipGetLastError(), "build_atoms launch");
    }
    launch_set_origin(g.fp64(), g.dev.p, origin * desc.scale, s);
    g.splines(s);
    if (host_copy)
        g.download(s);
    else
        check_hip(hipStreamSynchronize(s), "pdb build");
    timing_collect();
}

// Autotuner of the paired builder: every workgroup size (64..512 units) with
// every slice count 1..min(8, tiles) builds grid g once untimed per workgroup
// size and once timed (HIP events on s); the fastest is recorded in the shape
// table and builds the grid a last time, so it holds the bits every later
// build of its class gives (the workgroup size changes no sum; the slice
// count regroups the FP64 partial sums).
BuildShape Structure::autotune(Grid &g, hipStream_t s, double *best_ms, double *model_ms, bool direct) {
    if (g.fp64()) throw Error(kErrInvalidArgs, "the autotuner serves the mixed-precision builder");
    const long long nunits = pair_units(half_base(g.N + 1));
    BuildShape model;
    model.wg = 256;
    model.slices = pair_slices(nunits, ntiles, 256);
    hipEvent_t e0, e1;
    check_hip(hipEventCreate(&e0), "hipEventCreate");
    check_hip(hipEventCreate(&e1), "hipEventCreate");
    BuildShape best = model;
    double tbest = 1e300, tmodel = 0.0;
    try {
        Pending P;
        const int smax = std::min(kMaxSlices, std::max(ntiles, 1));
        for (int wg : {64, 128, 256, 512}) {
            for (int S = 0; S <= smax; S++) {
                // S = 0: the untimed warm-up of this workgroup size
                BuildJob J = prepare(g, std::max(S, 1), P, s, true);
                check_hip(hipEventRecord(e0, s), "hipEventRecord");
                launch_build_batch(P.reduce, wg, &J, 1, s);
                check_hip(hipGetLastError(), "build_atoms launch");
                check_hip(hipEventRecord(e1, s), "hipEventRecord");
                check_hip(hipEventSynchronize(e1), "hipEventSynchronize");
                if (S == 0) continue;
                float ms = 0.f;
                check_hip(hipEventElapsedTime(&ms, e0, e1), "hipEventElapsedTime");
                if (wg == model.wg && S == model.slices) tmodel = ms;
                if (ms < tbest) {
                    tbest = ms;
                    best.wg = wg;
                    best.slices = S;
                }
            }
        }
        BuildJob J = prepare(g, best.slices, P, s, direct);
        launch(g, J, best.wg, P, s);
        finish(g, P, false, s);
    } catch (...) {
        (void)hipEventDestroy(e0);
        (void)hipEventDestroy(e1);
        throw;
    }
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    shape_record(g.N, ntiles, best);
    if (best_ms) *best_ms = tbest;
    if (model_ms) *model_ms = tmodel;
    return best;
}

void pdb_build(Grid &g, const dplus_pdb_desc *d, bool host_copy, hipStream_t s) {
    Structure st(d, s);
    st.build(g, host_copy, s);
}

// ------------------------------------------------------------------ orientation averages
void launch_mc(bool fp64, bool single, const void *const *grids, const RotDev *rots, int nrot, const double4 *trans,
               const ZCopyDev *zc, int nz, const GroupDev *groups, const int *active, int nactive, int mstride, const double *qs,
               double step, uint64_t seed, long long dir0, int nblk, int chunk, double *partial, double *out,
               hipStream_t s);
void launch_vegas_iter(bool fp64, bool single, const void *const *grids, const RotDev *rots, int nrot, const double4 *trans,
                       const GroupDev *groups, const int *active, int nactive, int mstride, const double *qs,
                       double step, uint64_t seed, int iter, int ppb, double *bounds, double *binsum,
                       double *binvar, double *hist, int nq, hipStream_t s);
void launch_docked_cart(bool fp64, const void *const *grids, const LeafGeo *geo, const RotDev *rots, int nrot,
                        const double4 *trans, int n, const double *qxyz, double *out, hipStream_t s);
void launch_azimuthal(bool fp64, const void *const *grids, const LeafGeo *geo, const RotDev *rots, int nrot,
                      const double4 *trans, int npts, const double2 *pts, int nphi, uint64_t seed, double *out,
                      hipStream_t s);

void azimuthal_average(const DockSet &D, int npts, const double *q, const double *theta, int nphi, uint64_t seed,
                       double *out, hipStream_t s) {
    if (npts <= 0) return;
    if (nphi < 1) throw Error(kErrInvalidArgs, "the azimuthal average needs at least one phi sample");
    const double qlim = (D.grid_size / 2 + 1) * D.step;
    std::vector<double2> pts(npts);
    for (int i = 0; i < npts; i++) {
        if (!(q[i] >= 0.0 && q[i] <= qlim) || !(theta[i] >= 0.0 && theta[i] <= kPi))
            throw Error(kErrInvalidArgs, "2-D point outside the grid (q in [0, qmax], theta in [0, pi])");
        pts[i] = make_double2(q[i] * std::sin(theta[i]), q[i] * std::cos(theta[i]));
    }
    DevBuf bp, bo;
    bp.upload(pts.data(), pts.size() * sizeof(double2), s);
    bo.ensure((size_t)npts * sizeof(double));
    {
        KTimer kt("azimuthal", s);
        launch_azimuthal(D.fp64, (const void *const *)D.grids.p, (const LeafGeo *)D.geos.p, (const RotDev *)D.rotb.p,
                         D.nrot, (const double4 *)D.trb.p, npts, (const double2 *)bp.p, nphi, seed, (double *)bo.p, s);
    }
    check_hip(hipGetLastError(), "azimuthal launch");
    check_hip(hipMemcpyAsync(out, bo.p, (size_t)npts * sizeof(double), hipMemcpyDeviceToHost, s), "D2H");
    check_hip(hipStreamSynchronize(s), "azimuthal");
}

// R^T with R = Rx(a) Ry(b) Rz(c) (EulerD, Amplitude.h:557-573; HybridOA.cu:60-63)
void euler_rt(double a, double b, double c, double m[9]) {
    const double s1 = std::sin(a), c1 = std::cos(a), s2 = std::sin(b), c2 = std::cos(b), s3 = std::sin(c),
                 c3 = std::cos(c);
    const double rt[9] = {c2 * c3, c1 * s3 + c3 * s1 * s2, s1 * s3 - c1 * c3 * s2,
                          -(c2 * s3), c1 * c3 - s1 * s2 * s3, c3 * s1 + c1 * s2 * s3,
                          s2, -(c2 * s1), c1 * c2};
    for (int i = 0; i < 9; i++) m[i] = rt[i];
}

bool z_copies(const RotDev *rots, int nrot, const double4 *tr, std::vector<ZCopyDev> &out) {
    // DPLUS_ZCOPY=0 keeps such dockings on the general kernel (for A/B checks)
    const char *env = getenv("DPLUS_ZCOPY");
    if (env && std::strcmp(env, "0") == 0) return false;
    std::vector<ZCopyDev> zc;
    for (int r = 0; r < nrot; r++) {
        const double *m = rots[r].m;
        // R^T = Rz(alpha)^T = [[c, s, 0], [-s, c, 0], [0, 0, 1]]: the z row and
        // column exactly as Euler angles (0, 0, alpha) give them, so the general
        // lookup would take the direction's own polar angle
        if (m[2] != 0.0 || m[5] != 0.0 || m[6] != 0.0 || m[7] != 0.0 || m[8] != 1.0) return false;
        if (std::fabs(m[3] + m[1]) > 1e-12 || std::fabs(m[4] - m[0]) > 1e-12) return false;
        double a = std::atan2(m[1], m[0]);
        if (a < 0.0) a += 2.0 * kPi;
        if (a >= 2.0 * kPi) a = 0.0;
        for (int t = 0; t < rots[r].nt; t++) {
            const double4 v = tr[rots[r].t0 + t];
            zc.push_back(ZCopyDev{a, {v.x, v.y, v.z}, rots[r].scale, rots[r].leaf, 0, 0, 0});
        }
    }
    std::stable_sort(zc.begin(), zc.end(), [](const ZCopyDev &x, const ZCopyDev &y) {
        return x.leaf != y.leaf ? x.leaf < y.leaf : x.alpha < y.alpha;
    });
    // a chunk of 64 copies spanning d alpha covers at most d alpha * 6 l / (2 pi) + 3
    // nodes of a shell-l row (its two ends and the last node's right neighbour):
    // within the 64-node window while l <= 61 * 2 pi / (6 d alpha); one node
    // of margin for rounding.  Chunks spanning two leaves take the direct
    // lookup in the kernel and do not bound it.
    double lfit = 1e9;
    for (size_t c0 = 0; c0 < zc.size(); c0 += 64) {
        const size_t last = std::min(zc.size() - 1, c0 + 63);
        if (zc[c0].leaf != zc[last].leaf) continue;
        const double da = zc[last].alpha - zc[c0].alpha;
        if (da > 0.0) lfit = std::min(lfit, std::floor(60.0 * 2.0 * kPi / (6.0 * da)));
    }
    for (int i = (int)zc.size() - 1; i >= 0; i--)
        zc[i].run = i + 1 < (int)zc.size() && zc[i + 1].leaf == zc[i].leaf ? zc[i + 1].run : i + 1;
    if (!zc.empty()) zc[0].aux = (int)std::min(lfit, 1e9);
    out.swap(zc);
    return true;
}

// GridSymmetry::OrganizeParameters/PreCalculate (DefaultModels/Symmetries.cpp:29-97):
// angles wrapped to [-pi, pi), validated, and the basis a = (da,0,0),
// b = db (cos g, sin g, 0), c = dc (cos b, sin b cat, sin b sin(acos cat)),
// cat = (cos a - cos b cos g) / (sin b sin g)
LatticeDev space_filling_lattice(const double *d, const double *deg, const double *reps) {
    double ang[3];
    for (int k = 0; k < 3; k++) {
        double a = deg[k] * kPi / 180.0;
        while (a < -kPi) a += 2.0 * kPi;
        while (a >= kPi) a -= 2.0 * kPi;
        ang[k] = a;
    }
    const double al = ang[0], be = ang[1], ga = ang[2];
    for (int k = 0; k < 3; k++)
        if (ang[k] == 0.0 || std::fabs(std::fabs(ang[k]) - kPi) < 1e-6)
            throw Error(kErrInvalidArgs, "Angles in a Space-filling Symmetry cannot be zero or 180. The result is a 2D "
                                         "space. To create a 2D space, make the angle 90 degrees and one repetition in "
                                         "that direction.");
    if (std::fabs(al) + std::fabs(be) <= std::fabs(ga) || std::fabs(ga) + std::fabs(be) <= std::fabs(al) ||
        std::fabs(al) + std::fabs(ga) <= std::fabs(be))
        throw Error(kErrInvalidArgs, "In the Space-filling Symmetry, the sum of any two angles must be greater than the third.");
    const double cat = (std::cos(al) - std::cos(be) * std::cos(ga)) / (std::sin(be) * std::sin(ga));
    if (std::fabs(cat) > 1.0) throw Error(kErrInvalidArgs, "In the Space-filling Symmetry, the angles don't form a valid basis.");
    LatticeDev L{};
    L.v[0] = d[0];
    L.v[3] = d[1] * std::cos(ga);
    L.v[4] = d[1] * std::sin(ga);
    L.v[6] = d[2] * std::cos(be);
    L.v[7] = d[2] * std::sin(be) * cat;
    L.v[8] = d[2] * std::sin(be) * std::sin(std::acos(cat));
    for (int k = 0; k < 3; k++) {
        if (!(reps[k] >= 1.0)) throw Error(kErrInvalidArgs, "space-filling repetitions must be at least 1");
        L.n[k] = reps[k];
    }
    L.on = 1;
    return L;
}

// shell groups (OAJacob.cu:234-249): consecutive q with L*step < q <= (L+1)*step
std::vector<GroupDev> make_groups(const double *q, int nq, double step) {
    std::vector<GroupDev> gs;
    int layer = 0, q0 = 0;
    while (q0 < nq) {
        while (q[q0] > (double)(layer + 1) * step) layer++;
        int e = q0 + 1;
        while (e < nq && !(q[e] > (double)(layer + 1) * step)) e++;
        int uniform = 0;
        if (e - q0 > 1) {
            const double dq = (q[e - 1] - q[q0]) / (double)(e - 1 - q0), tol = 1e-12 * std::fabs(q[e - 1]);
            uniform = 1;
            for (int j = q0; j < e; j++)
                if (std::fabs(q[j] - (q[q0] + (double)(j - q0) * dq)) > tol) uniform = 0;
        }
        gs.push_back({layer, q0, e - q0, uniform});
        q0 = e;
        layer++;
    }
    return gs;
}

static bool converged3(const std::vector<double> &hist, int k, int q0, int m, int nq, double eps) {
    if (!(k > 2 && eps > 0.0)) return false;
    for (int j = 0; j < m; j++) {
        const double c = hist[(size_t)k * nq + q0 + j];
        for (int b = 1; b <= 3; b++)
            if (std::fabs(1.0 - c / hist[(size_t)(k - b) * nq + q0 + j]) > eps) return false;
    }
    return true;
}

DockSet::DockSet(int nleaf, const dplus_leaf *leaves, hipStream_t s) {
    if (nleaf <= 0) throw Error(kErrInvalidArgs, "no leaves");
    std::vector<Grid *> gl;
    std::vector<RotDev> rots;
    std::vector<double4> tr;
    for (int l = 0; l < nleaf; l++) {
        const dplus_leaf &L = leaves[l];
        if (!L.grid) throw Error(kErrInvalidArgs, "leaf without grid");
        gl.push_back((Grid *)L.grid);
        int t0 = 0;
        for (int r = 0; r < L.nrot; r++) {
            RotDev rd;
            euler_rt(L.rot[4 * r], L.rot[4 * r + 1], L.rot[4 * r + 2], rd.m);
            rd.scale = L.rot[4 * r + 3];
            rd.leaf = l;
            rd.t0 = (int)tr.size();
            rd.nt = L.ntrans[r];
            rd.pad = 0;
            if (rd.nt < 0) throw Error(kErrInvalidArgs, "negative translation count");
            for (int t = 0; t < rd.nt; t++)
                tr.push_back(make_double4(L.trans[3 * (t0 + t)], L.trans[3 * (t0 + t) + 1], L.trans[3 * (t0 + t) + 2], 0.0));
            t0 += rd.nt;
            rots.push_back(rd);
        }
    }
    finish(gl, rots, tr, s);
}

DockSet::DockSet(const std::vector<Placement> &pl, hipStream_t s) {
    if (pl.empty()) throw Error(kErrInvalidArgs, "no placements");
    std::vector<Grid *> gl;
    std::vector<RotDev> rots;
    std::vector<std::vector<double4>> per_rot;
    for (const Placement &p : pl) {
        if (!p.grid) throw Error(kErrInvalidArgs, "placement without grid");
        int l = (int)(std::find(gl.begin(), gl.end(), p.grid) - gl.begin());
        if (l == (int)gl.size()) gl.push_back(p.grid);
        size_t r = 0;
        for (; r < rots.size(); r++)
            if (rots[r].leaf == l && rots[r].scale == p.scale && std::equal(p.rt, p.rt + 9, rots[r].m)) break;
        if (r == rots.size()) {
            RotDev rd;
            std::copy(p.rt, p.rt + 9, rd.m);
            rd.scale = p.scale;
            rd.leaf = l;
            rd.t0 = rd.nt = rd.pad = 0;
            rots.push_back(rd);
            per_rot.emplace_back();
        }
        per_rot[r].push_back(make_double4(p.t[0], p.t[1], p.t[2], 0.0));
    }
    std::vector<double4> tr;
    for (size_t r = 0; r < rots.size(); r++) {
        rots[r].t0 = (int)tr.size();
        rots[r].nt = (int)per_rot[r].size();
        tr.insert(tr.end(), per_rot[r].begin(), per_rot[r].end());
    }
    finish(gl, rots, tr, s);
}

void DockSet::finish(std::vector<Grid *> &gl, std::vector<RotDev> &rots, std::vector<double4> &tr, hipStream_t s) {
    std::vector<const void *> gp;
    std::vector<LeafGeo> geo;
    for (size_t l = 0; l < gl.size(); l++) {
        const Grid *g = gl[l];
        if (l == 0) {
            grid_size = g->grid_size;
            qmax = g->qmax;
            step = g->step;
            fp64 = g->fp64();
        } else if (g->grid_size != grid_size || g->qmax != qmax || g->fp64() != fp64) {
            throw Error(kErrInvalidArgs, "all leaves of one orientation average must share grid size, qmax and precision");
        }
        gp.push_back(g->dev.p);
        geo.push_back({g->N, g->step});
    }
    if (tr.empty()) tr.push_back(make_double4(0, 0, 0, 0));
    nrot = (int)rots.size();
    static const double eye[9] = {1, 0, 0, 0, 1, 0, 0, 0, 1};
    single = nrot == 1 && rots[0].nt == 1 && rots[0].t0 == 0 && tr.size() == 1 && tr[0].x == 0.0 &&
             tr[0].y == 0.0 && tr[0].z == 0.0 && std::equal(eye, eye + 9, rots[0].m);
    grids.upload(gp.data(), gp.size() * sizeof(void *), s);
    geos.upload(geo.data(), geo.size() * sizeof(LeafGeo), s);
    rotb.upload(rots.data(), std::max<size_t>(1, rots.size()) * sizeof(RotDev), s);
    trb.upload(tr.data(), tr.size() * sizeof(double4), s);
    std::vector<ZCopyDev> zc;
    nz = 0;
    if (!single && z_copies(rots.data(), nrot, tr.data(), zc) && (int)zc.size() >= kZCopyMin) {
        nz = (int)zc.size();
        zcb.upload(zc.data(), zc.size() * sizeof(ZCopyDev), s);
    }
}

void launch_mc_finish(const GroupDev *groups, int ngroups, int mstride, const double *out, double total, double *I,
                      hipStream_t s);
void launch_chi2(const double *I, const double *y, const double *sig, int n, double scale, double constant,
                 double *chi2, hipStream_t s);

void check_q_range(const DockSet &D, int nq, const double *q) {
    for (int i = 1; i < nq; i++)
        if (q[i] < q[i - 1]) throw Error(kErrInvalidArgs, "q must be ascending");
    if (nq <= 0) return;
    if (!(q[0] >= 0)) throw Error(kErrInvalidArgs, "q must be non-negative");
    if (q[nq - 1] > D.qmax * (1.0 + 1e-12) + 0.0) {
        // the reference integrates up to the grid's qmax; beyond it the extra shells are extrapolation
        if (q[nq - 1] > (D.grid_size / 2 + 1) * D.step) throw Error(kErrInvalidArgs, "q beyond the grid");
    }
}

void FixedAverage::prepare(const DockSet &D, int nq_, const double *q, const dplus_oa_params *p,
                           const Chi2Request *c, hipStream_t s) {
    if (!(p->eps <= 0.0) || (p->method != DPLUS_OA_MC && p->method != DPLUS_OA_VEGAS))
        throw Error(kErrInvalidArgs, "a fixed-count average is Monte Carlo or VEGAS with eps <= 0");
    if (nq_ <= 0) throw Error(kErrInvalidArgs, "a fixed-count average needs q values");
    check_q_range(D, nq_, q);
    nq = nq_;
    method = p->method;
    seed = p->seed;
    const std::vector<GroupDev> groups = make_groups(q, nq, D.step);
    ng = (int)groups.size();
    mstride = 1;
    for (auto &g : groups) mstride = std::max(mstride, g.m);
    std::vector<int> act(ng);
    for (int i = 0; i < ng; i++) act[i] = i;
    bq.upload(q, nq * sizeof(double), s);
    bg.upload(groups.data(), ng * sizeof(GroupDev), s);
    bact.upload(act.data(), ng * sizeof(int), s);
    if (method == DPLUS_OA_MC) {
        chunk = p->chunk > 0 ? p->chunk : 8192;
        if (chunk % 256) throw Error(kErrInvalidArgs, "MC chunk must be a multiple of 256");
        const long long nchunks = (std::max<long long>(1, p->max_dirs) + chunk - 1) / chunk;
        // one launch covers every direction of every group
        total = nchunks * chunk;
        if (total / 256 > 2147483647LL) throw Error(kErrInvalidArgs, "too many directions");
        nblk = (int)(total / 256);
        bpart.ensure((size_t)ng * nblk * mstride * sizeof(double));
        bout.ensure((size_t)ng * mstride * sizeof(double));
        bI.ensure((size_t)nq * sizeof(double));
    } else {
        iters = std::max(1, p->vegas_iterations);
        ppb = std::max(1, p->vegas_points_per_bin);
        if (ppb > 256) throw Error(kErrInvalidArgs, "VEGAS points per bin must be <= 256");
        std::vector<double> bounds((size_t)ng * 66);
        for (int g = 0; g < ng; g++)
            for (int i = 0; i <= 32; i++) {
                bounds[(size_t)g * 66 + i] = (double)i / 32;
                bounds[(size_t)g * 66 + 33 + i] = (double)i / 32;
            }
        bb.upload(bounds.data(), bounds.size() * sizeof(double), s);
        bsum.ensure((size_t)ng * mstride * 1024 * sizeof(double));
        bvar.ensure((size_t)ng * 1024 * sizeof(double));
        bh.ensure((size_t)iters * nq * sizeof(double));
    }
    chi = c != nullptr;
    if (chi) {
        by.upload(c->y, nq * sizeof(double), s);
        bsig.upload(c->sigma, nq * sizeof(double), s);
        bchi.ensure(sizeof(double));
        chi_scale = c->scale;
        chi_constant = c->constant;
    }
}

void FixedAverage::enqueue_kernels(const DockSet &D, hipStream_t s, bool timed) const {
    if (method == DPLUS_OA_MC) {
        {
            std::unique_ptr<KTimer> kt(timed ? new KTimer("mc", s) : nullptr);
            launch_mc(D.fp64, D.single, (const void *const *)D.grids.p, (const RotDev *)D.rotb.p, D.nrot,
                      (const double4 *)D.trb.p, (const ZCopyDev *)D.zcb.p, D.nz, (const GroupDev *)bg.p, (const int *)bact.p, ng, mstride,
                      (const double *)bq.p, D.step, seed, 0, nblk, chunk, (double *)bpart.p, (double *)bout.p, s);
        }
        check_hip(hipGetLastError(), "mc launch");
        launch_mc_finish((const GroupDev *)bg.p, ng, mstride, (const double *)bout.p, (double)total, (double *)bI.p, s);
        check_hip(hipGetLastError(), "mc finish launch");
    } else {
        launch_fill_zero((double *)bh.p, (size_t)iters * nq, s);
        check_hip(hipGetLastError(), "fill launch");
        for (int k = 0; k < iters; k++) {
            std::unique_ptr<KTimer> kt(timed ? new KTimer("vegas", s) : nullptr);
            launch_vegas_iter(D.fp64, D.single, (const void *const *)D.grids.p, (const RotDev *)D.rotb.p, D.nrot,
                              (const double4 *)D.trb.p, (const GroupDev *)bg.p, (const int *)bact.p, ng, mstride,
                              (const double *)bq.p, D.step, seed, k, ppb, (double *)bb.p, (double *)bsum.p,
                              (double *)bvar.p, (double *)bh.p, nq, s);
            check_hip(hipGetLastError(), "vegas launch");
        }
        // every group runs every iteration: the result is the last iteration's running mean
    }
    if (chi) {
        launch_chi2(result(), (const double *)by.p, (const double *)bsig.p, nq, chi_scale, chi_constant,
                    (double *)bchi.p, s);
        check_hip(hipGetLastError(), "chi2 launch");
    }
}

void FixedAverage::download(double *I, double *chi2, hipStream_t s) const {
    if (chi) check_hip(hipMemcpyAsync(chi2, bchi.p, sizeof(double), hipMemcpyDeviceToHost, s), "D2H");
    check_hip(hipMemcpyAsync(I, result(), nq * sizeof(double), hipMemcpyDeviceToHost, s), "D2H");
}

void orientation_average(const DockSet &D, int nq, const double *q, const dplus_oa_params *p, double *out,
                         dplus_oa_stats *st, hipStream_t s, Chi2Request *chi) {
    if (chi) chi->on_device = false;
    check_q_range(D, nq, q);
    if (nq <= 0) return;
    if (p->eps <= 0.0 && (p->method == DPLUS_OA_MC || p->method == DPLUS_OA_VEGAS)) {
        // fixed count: every group takes every direction / iteration, no host decisions
        FixedAverage F;
        F.prepare(D, nq, q, p, chi, s);
        F.enqueue(D, out, chi ? &chi->chi2 : nullptr, s, true);
        check_hip(hipStreamSynchronize(s), p->method == DPLUS_OA_MC ? "mc" : "vegas");
        if (chi) chi->on_device = true;
        if (st) {
            if (p->method == DPLUS_OA_MC)
                st->dirs_used = F.total;
            else
                st->iterations_used = F.iters;
        }
        return;
    }
    const std::vector<GroupDev> groups = make_groups(q, nq, D.step);
    const int ng = (int)groups.size();
    int mstride = 1;
    for (auto &g : groups) mstride = std::max(mstride, g.m);
    DevBuf bq, bg, bact;
    bq.upload(q, nq * sizeof(double), s);
    bg.upload(groups.data(), ng * sizeof(GroupDev), s);
    std::vector<int> act(ng);
    for (int i = 0; i < ng; i++) act[i] = i;
    bact.upload(act.data(), ng * sizeof(int), s);
    if (p->method == DPLUS_OA_MC) {
        const int chunk = p->chunk > 0 ? p->chunk : 8192;
        if (chunk % 256) throw Error(kErrInvalidArgs, "MC chunk must be a multiple of 256");
        long long nchunks = (std::max<long long>(1, p->max_dirs) + chunk - 1) / chunk;
        std::vector<double> hist((size_t)nchunks * nq, 0.0), sum(nq, 0.0);
        DevBuf bpart, bout;
        long long used = 0;
        // chunked with the reference's three-back convergence test (GPUHybridCalc.cu:705-720)
        const int nblk = chunk / 256;
        bpart.ensure((size_t)ng * nblk * mstride * sizeof(double));
        bout.ensure((size_t)ng * mstride * sizeof(double));
        std::vector<int> active = act;
        std::vector<int> done_k(ng, -1);
        std::vector<double> r((size_t)ng * mstride);
        for (long long k = 0; k < nchunks && !active.empty(); k++) {
            bact.upload(active.data(), active.size() * sizeof(int), s);
            {
                KTimer kt("mc", s);
                launch_mc(D.fp64, D.single, (const void *const *)D.grids.p, (const RotDev *)D.rotb.p, D.nrot,
                          (const double4 *)D.trb.p, (const ZCopyDev *)D.zcb.p, D.nz, (const GroupDev *)bg.p, (const int *)bact.p,
                          (int)active.size(), mstride, (const double *)bq.p, D.step, p->seed, k * chunk, nblk,
                          chunk, (double *)bpart.p, (double *)bout.p, s);
            }
            check_hip(hipGetLastError(), "mc launch");
            check_hip(hipMemcpyAsync(r.data(), bout.p, active.size() * mstride * sizeof(double),
                                     hipMemcpyDeviceToHost, s), "D2H");
            check_hip(hipStreamSynchronize(s), "mc chunk");
            std::vector<int> next;
            for (size_t ai = 0; ai < active.size(); ai++) {
                const GroupDev &G = groups[active[ai]];
                for (int j = 0; j < G.m; j++) {
                    sum[G.q0 + j] += r[ai * mstride + j];
                    hist[(size_t)k * nq + G.q0 + j] = sum[G.q0 + j] / ((double)(k + 1) * chunk);
                }
                if (converged3(hist, (int)k, G.q0, G.m, nq, p->eps) || k == nchunks - 1)
                    done_k[active[ai]] = (int)k;
                else
                    next.push_back(active[ai]);
            }
            active.swap(next);
        }
        for (int gi = 0; gi < ng; gi++) {
            const int k = done_k[gi];
            used = std::max<long long>(used, (long long)(k + 1) * chunk);
            for (int j = 0; j < groups[gi].m; j++) out[groups[gi].q0 + j] = hist[(size_t)k * nq + groups[gi].q0 + j];
        }
        if (st) st->dirs_used = used;
    } else if (p->method == DPLUS_OA_VEGAS) {
        const int iters = std::max(1, p->vegas_iterations);
        const int ppb = std::max(1, p->vegas_points_per_bin);
        if (ppb > 256) throw Error(kErrInvalidArgs, "VEGAS points per bin must be <= 256");
        std::vector<double> bounds((size_t)ng * 66);
        for (int g = 0; g < ng; g++)
            for (int i = 0; i <= 32; i++) {
                bounds[(size_t)g * 66 + i] = (double)i / 32;
                bounds[(size_t)g * 66 + 33 + i] = (double)i / 32;
            }
        DevBuf bb, bsum, bvar, bh;
        bb.upload(bounds.data(), bounds.size() * sizeof(double), s);
        bsum.ensure((size_t)ng * mstride * 1024 * sizeof(double));
        bvar.ensure((size_t)ng * 1024 * sizeof(double));
        bh.ensure((size_t)iters * nq * sizeof(double));
        launch_fill_zero((double *)bh.p, (size_t)iters * nq, s);
        check_hip(hipGetLastError(), "fill launch");
        std::vector<double> hist((size_t)iters * nq, 0.0);
        std::vector<int> active = act, done_k(ng, iters - 1);
        int used = 0;
        for (int k = 0; k < iters && !active.empty(); k++) {
            if (k > 0) bact.upload(active.data(), active.size() * sizeof(int), s);
            {
                KTimer kt("vegas", s);
                launch_vegas_iter(D.fp64, D.single, (const void *const *)D.grids.p, (const RotDev *)D.rotb.p, D.nrot,
                                  (const double4 *)D.trb.p, (const GroupDev *)bg.p, (const int *)bact.p,
                                  (int)active.size(), mstride, (const double *)bq.p, D.step, p->seed, k, ppb,
                                  (double *)bb.p, (double *)bsum.p, (double *)bvar.p, (double *)bh.p, nq, s);
            }
            check_hip(hipGetLastError(), "vegas launch");
            used = k + 1;
            check_hip(hipMemcpyAsync(hist.data() + (size_t)k * nq, (double *)bh.p + (size_t)k * nq,
                                     nq * sizeof(double), hipMemcpyDeviceToHost, s), "D2H");
            check_hip(hipStreamSynchronize(s), "vegas iter");
            std::vector<int> next;
            for (int g : active) {
                if (converged3(hist, k, groups[g].q0, groups[g].m, nq, p->eps))
                    done_k[g] = k;
                else
                    next.push_back(g);
            }
            active.swap(next);
        }
        check_hip(hipMemcpyAsync(hist.data(), bh.p, hist.size() * sizeof(double), hipMemcpyDeviceToHost, s), "D2H");
        check_hip(hipStreamSynchronize(s), "vegas");
        for (int g = 0; g < ng; g++)
            for (int j = 0; j < groups[g].m; j++) out[groups[g].q0 + j] = hist[(size_t)done_k[g] * nq + groups[g].q0 + j];
        if (st) st->iterations_used = used;
    } else if (p->method == DPLUS_OA_GK) {
        gk_average(D, nq, q, p->eps, p->gk_max_depth > 0 ? p->gk_max_depth : (1LL << 40), out, st, s);
    } else {
        throw Error(kErrInvalidArgs, "unknown orientation method");
    }
    if (chi && !chi->on_device) {
        double c2 = 0.0;
        for (int i = 0; i < nq; i++)
            if (chi->sigma[i] > 0.0) {
                const double r = (chi->scale * out[i] + chi->constant - chi->y[i]) / chi->sigma[i];
                c2 = std::fma(r, r, c2);
            }
        chi->chi2 = c2;
    }
}

// Device bytes the Monte Carlo / VEGAS orientation average takes from a
// scratch arena: every DevBuf of DockSet and of FixedAverage / the
// orientation average's MC and VEGAS branches, in their sizes, each 256-byte
// aligned (and the chi^2 inputs of a fixed-count average); *upload_bytes: the
// aligned sizes of the uploaded ones.
size_t oa_arena_bytes(int nleaf, long long nrot, long long ntr, int nq, const double *q, double step,
                      const dplus_oa_params *p, bool chi, size_t *upload_bytes) {
    auto al = [](size_t b) { return (b + 255) & ~(size_t)255; };
    size_t up = 0;
    auto upl = [&](size_t b) {
        up += al(b);
        return al(b);
    };
    size_t b = upl((size_t)nleaf * sizeof(void *)) + upl((size_t)nleaf * sizeof(LeafGeo)) +
               upl((size_t)std::max<long long>(1, nrot) * sizeof(RotDev)) +
               upl((size_t)std::max<long long>(1, ntr) * sizeof(double4)) +
               upl((size_t)std::max<long long>(1, ntr) * sizeof(ZCopyDev));
    if (nq > 0) {
        const std::vector<GroupDev> groups = make_groups(q, nq, step);
        const size_t ng = groups.size();
        size_t mstride = 1;
        for (auto &g : groups) mstride = std::max<size_t>(mstride, (size_t)g.m);
        b += upl((size_t)nq * 8) + upl(ng * sizeof(GroupDev)) + upl(ng * sizeof(int));
        if (p->method == DPLUS_OA_MC) {
            const long long chunk = p->chunk > 0 ? p->chunk : 8192;
            const long long nchunks = (std::max<long long>(1, p->max_dirs) + chunk - 1) / chunk;
            const size_t nblk = (size_t)(p->eps <= 0.0 ? nchunks * chunk / 256 : chunk / 256);
            b += al(ng * nblk * mstride * 8) + al(ng * mstride * 8) + (p->eps <= 0.0 ? al((size_t)nq * 8) : 0);
        } else {
            const size_t iters = (size_t)std::max(1, p->vegas_iterations);
            b += upl(ng * 66 * 8) + al(ng * mstride * 1024 * 8) + al(ng * 1024 * 8) + al(iters * nq * 8);
        }
        if (chi) b += upl((size_t)nq * 8) + upl((size_t)nq * 8) + al(8);
    }
    if (upload_bytes) *upload_bytes = up;
    return b;
}

}  // namespace dplus

using namespace dplus;

#define API_GUARD(...)                                      \
    try {                                                   \
        __VA_ARGS__;                                        \
        return kOk;                                         \
    } catch (const Error &e) {                              \
        return set_error(e.code, e.what());                 \
    } catch (const std::exception &e) {                     \
        return set_error(kErrGeneral, e.what());            \
    } catch (...) {                                         \
        return set_error(kErrGeneral, "unknown exception"); \
    }

extern "C" {

const char *dplus_last_error(void) { return g_last_error.c_str(); }

int dplus_device_info(char *buf, int len) {
    API_GUARD({
        Device &d = Device::get();
        std::string s = "{\"ok\":" + std::string(d.ok ? "true" : "false") + ",\"device\":" + std::to_string(d.id) +
                        ",\"arch\":\"" + json_escape(d.name) + "\",\"cus\":" + std::to_string(d.cus) +
                        ",\"memory\":" + std::to_string(d.mem) +
                        ",\"device_allocations\":" + std::to_string(device_allocations()) + "}";
        if (buf && len > 0) {
            strncpy(buf, s.c_str(), len - 1);
            buf[len - 1] = 0;
        }
    })
}

int dplus_grid_create(int grid_size, double qmax, int precision, dplus_grid **out) {
    API_GUARD({
        if (!out) throw Error(kErrInvalidArgs, "null output");
        if (precision != DPLUS_PRECISION_FP64 && precision != DPLUS_PRECISION_MIXED)
            throw Error(kErrInvalidArgs, "unknown precision");
        *out = (dplus_grid *)new Grid(grid_size, qmax, precision);
    })
}

void dplus_grid_destroy(dplus_grid *g) { delete (Grid *)g; }

int dplus_grid_info(const dplus_grid *gh, int *grid_size, double *qmax, double *step, int *actual_size,
                    long long *points, int *precision) {
    API_GUARD({
        const Grid *g = (const Grid *)gh;
        if (!g) throw Error(kErrInvalidArgs, "null grid");
        if (grid_size) *grid_size = g->grid_size;
        if (qmax) *qmax = g->qmax;
        if (step) *step = g->step;
        if (actual_size) *actual_size = g->N;
        if (points) *points = g->P;
        if (precision) *precision = g->precision;
    })
}

double *dplus_grid_data(dplus_grid *gh) {
    Grid *g = (Grid *)gh;
    if (!g) return nullptr;
    g->ensure_host();
    return g->host_data.data();
}

double *dplus_grid_interp(dplus_grid *gh) {
    Grid *g = (Grid *)gh;
    if (!g) return nullptr;
    g->ensure_host();
    return g->host_interp.data();
}

long long dplus_grid_index_from_indices(int qi, long long ti, long long pi) { return index_from_indices(qi, ti, pi); }

void dplus_grid_indices_from_index(long long index, int *qi, long long *ti, long long *pi) {
    if (index <= 0) {
        *qi = 0;
        *ti = 0;
        *pi = 0;
        return;
    }
    long long q = (long long)std::cbrt((double)index / 6.0);
    if (q < 1) q = 1;
    while (q > 1 && shell_base(q) > index) q--;
    while (shell_base(q + 1) <= index) q++;
    long long rem = index - shell_base(q);
    *qi = (int)q;
    *ti = rem / (6 * q);
    *pi = rem % (6 * q);
}

int dplus_grid_upload(dplus_grid *gh) {
    API_GUARD({
        Grid *g = (Grid *)gh;
        if (!g) throw Error(kErrInvalidArgs, "null grid");
        Device::get().require();
        g->upload(Device::get().stream);
    })
}

int dplus_grid_calculate_splines(dplus_grid *gh) {
    API_GUARD({
        Grid *g = (Grid *)gh;
        if (!g) throw Error(kErrInvalidArgs, "null grid");
        Device::get().require();
        g->splines(Device::get().stream);
        check_hip(hipStreamSynchronize(Device::get().stream), "splines");
    })
}

int dplus_grid_download(dplus_grid *gh) {
    API_GUARD({
        Grid *g = (Grid *)gh;
        if (!g) throw Error(kErrInvalidArgs, "null grid");
        Device::get().require();
        g->download(Device::get().stream);
    })
}

}  // extern "C"
namespace dplus {
void launch_sphr_batch(bool fp64, const void *g, int N, double step, int n, const double *q, const double *th,
                       const double *ph, double2 *out, hipStream_t s);
void launch_seeded_samples(bool fp64, const void *g, int N, double step, double q, long long n,
                           const double *phi, const double *v2, double *out, hipStream_t s);
void launch_plane_batch(bool fp64, const void *g, int n, const int *ri, const double *th, const double *ph,
                        double2 *out, hipStream_t s);
void launch_gather_probe(const void *grid, int N, const RotDev *rots, int nrot, int layer0, int nlayers, int nblk,
                         uint64_t seed, int chunk, float *sink, hipStream_t s);
}  // namespace dplus
extern "C" {

int dplus_grid_get_sphr(dplus_grid *gh, int n, const double *q, const double *th, const double *ph, double *out) {
    API_GUARD({
        Grid *g = (Grid *)gh;
        if (!g || n < 0) throw Error(kErrInvalidArgs, "bad arguments");
        if (n == 0) return kOk;
        for (int i = 0; i < n; i++)
            if (!(q[i] >= 0 && q[i] <= (g->N - 2) * g->step && th[i] >= 0 && th[i] <= kPi && ph[i] >= 0 &&
                  ph[i] <= k2Pi))
                throw Error(kErrInvalidArgs, "lookup point outside the grid (q in [0, qmax], theta in [0,pi], phi in [0,2pi])");
        hipStream_t s = Device::get().stream;
        DevBuf bq, bt, bp, bo;
        bq.upload(q, n * sizeof(double), s);
        bt.upload(th, n * sizeof(double), s);
        bp.upload(ph, n * sizeof(double), s);
        bo.ensure(n * sizeof(double2));
        launch_sphr_batch(g->fp64(), g->dev.p, g->N, g->step, n, (const double *)bq.p, (const double *)bt.p,
                          (const double *)bp.p, (double2 *)bo.p, s);
        check_hip(hipGetLastError(), "sphr launch");
        check_hip(hipMemcpyAsync(out, bo.p, n * sizeof(double2), hipMemcpyDeviceToHost, s), "D2H");
        check_hip(hipStreamSynchronize(s), "sphr");
    })
}

int dplus_grid_interpolate_theta_phi_plane(dplus_grid *gh, int n, const int *ri, const double *th, const double *ph,
                                           double *out) {
    API_GUARD({
        Grid *g = (Grid *)gh;
        if (!g || n < 0 || (n > 0 && (!ri || !th || !ph || !out))) throw Error(kErrInvalidArgs, "bad arguments");
        if (n == 0) return kOk;
        for (int i = 0; i < n; i++)
            if (!(ri[i] >= 1 && ri[i] <= g->N && th[i] >= 0 && th[i] <= kPi && ph[i] >= 0 && ph[i] <= k2Pi))
                throw Error(kErrInvalidArgs,
                            "plane lookup outside the grid (shell in [1, actual size], theta in [0,pi], phi in [0,2pi])");
        hipStream_t s = Device::get().stream;
        DevBuf br, bt, bp, bo;
        br.upload(ri, n * sizeof(int), s);
        bt.upload(th, n * sizeof(double), s);
        bp.upload(ph, n * sizeof(double), s);
        bo.ensure(n * sizeof(double2));
        launch_plane_batch(g->fp64(), g->dev.p, n, (const int *)br.p, (const double *)bt.p, (const double *)bp.p,
                           (double2 *)bo.p, s);
        check_hip(hipGetLastError(), "plane launch");
        check_hip(hipMemcpyAsync(out, bo.p, n * sizeof(double2), hipMemcpyDeviceToHost, s), "D2H");
        check_hip(hipStreamSynchronize(s), "plane");
    })
}

int dplus_grid_calculate_intensity(dplus_grid *gh, double q, double theta, double eps, unsigned seed,
                                   unsigned long long iterations, double phi_min, double phi_max, double *result) {
    API_GUARD({
        Grid *g = (Grid *)gh;
        if (!g || !result || iterations == 0) throw Error(kErrInvalidArgs, "bad arguments");
        if ((phi_min < 0) || (phi_max > k2Pi) || (phi_min > phi_max))
            throw Error(kErrGeneral, "phi_min or phi_max are invalid");
        if (!(q >= 0 && q <= (g->N - 2) * g->step)) throw Error(kErrInvalidArgs, "q outside the grid");
        hipStream_t s = Device::get().stream;
        if (q == 0.0) {
            double o[2];
            const double z = 0.0;
            DevBuf bz, bo;
            bz.upload(&z, sizeof z, s);
            bo.ensure(sizeof(double2));
            launch_sphr_batch(g->fp64(), g->dev.p, g->N, g->step, 1, (const double *)bz.p, (const double *)bz.p,
                              (const double *)bz.p, (double2 *)bo.p, s);
            check_hip(hipMemcpyAsync(o, bo.p, sizeof o, hipMemcpyDeviceToHost, s), "D2H");
            check_hip(hipStreamSynchronize(s), "intensity");
            *result = o[0] * o[0] + o[1] * o[1];
            return kOk;
        }
        // Grid.cpp:415-425: phi ~ U(phi_min, phi_max), v2 ~ U(0, 2) from std::mt19937(seed)
        if (theta < 0) {
            phi_min = 0.0;
            phi_max = k2Pi;
        }
        const long long n = (long long)iterations;
        std::vector<double> phi(n), v2(n);
        std::mt19937 rng;
        rng.seed(seed);
        std::uniform_real_distribution<double> ranU2(0.0, 2.0);
        std::uniform_real_distribution<double> ranPHI(phi_min, phi_max);
        for (long long i = 0; i < n; i++) {
            phi[i] = ranPHI(rng);
            v2[i] = ranU2(rng);
            if (theta >= 0) v2[i] = std::cos(theta) + 1.0;
        }
        DevBuf bphi, bv2, bo;
        bphi.upload(phi.data(), n * sizeof(double), s);
        bv2.upload(v2.data(), n * sizeof(double), s);
        bo.ensure(n * sizeof(double));
        launch_seeded_samples(g->fp64(), g->dev.p, g->N, g->step, q, n, (const double *)bphi.p,
                              (const double *)bv2.p, (double *)bo.p, s);
        check_hip(hipGetLastError(), "seeded launch");
        std::vector<double> I(n);
        check_hip(hipMemcpyAsync(I.data(), bo.p, n * sizeof(double), hipMemcpyDeviceToHost, s), "D2H");
        check_hip(hipStreamSynchronize(s), "intensity");
        // running mean and the convergence test of Grid.cpp:456-467
        std::vector<double> res(n);
        const unsigned long long minIter = iterations / 20;
        double acc = 0.0;
        for (long long i = 0; i < n; i++) {
            acc += I[i];
            res[i] = acc / (double)(i + 1);
            if ((unsigned long long)i >= minIter && eps > 0.0) {
                if (std::fabs(1.0 - res[i] / res[i >> 1]) < eps && std::fabs(1.0 - res[i] / res[(i << 1) / 3]) < eps &&
                    std::fabs(1.0 - res[i] / res[(3 * i) >> 2]) < eps) {
                    *result = res[i];
                    return kOk;
                }
            }
        }
        *result = res[n - 1];
    })
}

int dplus_pdb_build_grid(dplus_grid *gh, const dplus_pdb_desc *d, int host_copy) {
    API_GUARD({
        Grid *g = (Grid *)gh;
        if (!g || !d) throw Error(kErrInvalidArgs, "null argument");
        Device::get().require();
        pdb_build(*g, d, host_copy != 0, Device::get().stream);
    })
}

int dplus_orientation_average(int nleaf, const dplus_leaf *leaves, int nq, const double *q, const dplus_oa_params *p,
                              double *intensity, dplus_oa_stats *st) {
    API_GUARD({
        if (!leaves || !q || !p || !intensity || nq < 0) throw Error(kErrInvalidArgs, "null argument");
        Device::get().require();
        auto t0 = std::chrono::steady_clock::now();
        hipStream_t s = Device::get().stream;
        DockSet D(nleaf, leaves, s);
        if (st) memset(st, 0, sizeof *st);
        orientation_average(D, nq, q, p, intensity, st, s);
        timing_collect();
        if (st) st->seconds = std::chrono::duration<double>(std::chrono::steady_clock::now() - t0).count();
    })
}

int dplus_orientation_average_noalloc(int nleaf, const dplus_leaf *leaves, int nq, const double *q,
                                      const dplus_oa_params *p, double *intensity, dplus_oa_stats *st) {
    API_GUARD({
        if (!leaves || !q || !p || !intensity || nq < 0 || nleaf <= 0) throw Error(kErrInvalidArgs, "null argument");
        if (p->method != DPLUS_OA_MC && p->method != DPLUS_OA_VEGAS)
            throw Error(kErrInvalidArgs, "the allocation-free orientation average runs Monte Carlo or VEGAS only");
        if (p->method == DPLUS_OA_MC) {
            const int chunk = p->chunk > 0 ? p->chunk : 8192;
            if (chunk % 256) throw Error(kErrInvalidArgs, "MC chunk must be a multiple of 256");
        }
        for (int i = 1; i < nq; i++)
            if (q[i] < q[i - 1]) throw Error(kErrInvalidArgs, "q must be ascending");
        if (nq > 0 && !(q[0] >= 0)) throw Error(kErrInvalidArgs, "q must be non-negative");
        long long nrot = 0, ntr = 0;
        for (int l = 0; l < nleaf; l++) {
            if (!leaves[l].grid) throw Error(kErrInvalidArgs, "leaf without grid");
            nrot += leaves[l].nrot;
            for (int r = 0; r < leaves[l].nrot; r++) ntr += leaves[l].ntrans[r];
        }
        const size_t need = oa_arena_bytes(nleaf, nrot, ntr, nq, q, ((Grid *)leaves[0].grid)->step, p);
        if (need > scratch_capacity())
            throw Error(kErrInvalidArgs, "the allocation-free orientation average needs " + std::to_string(need) +
                                             " bytes of scratch, above its maximum of " +
                                             std::to_string(scratch_capacity()) + " bytes");
        Device &dev = Device::get();
        dev.require();
        std::lock_guard<std::mutex> use(scratch_lock(dev.id));
        Arena arena;
        arena.base = (char *)scratch_address(dev.id);
        arena.size = scratch_capacity();
        struct Install {
            explicit Install(Arena *a) { set_arena(a); }
            ~Install() { set_arena(nullptr); }
        } install(&arena);
        auto t0 = std::chrono::steady_clock::now();
        hipStream_t s = dev.stream;
        DockSet D(nleaf, leaves, s);
        if (st) memset(st, 0, sizeof *st);
        orientation_average(D, nq, q, p, intensity, st, s);
        timing_collect();
        if (st) st->seconds = std::chrono::duration<double>(std::chrono::steady_clock::now() - t0).count();
    })
}

int dplus_azimuthal_average(int nleaf, const dplus_leaf *leaves, int npts, const double *q, const double *theta,
                            int nphi, unsigned long long seed, double *intensity) {
    API_GUARD({
        if (!leaves || npts < 0 || (npts > 0 && (!q || !theta || !intensity)))
            throw Error(kErrInvalidArgs, "null argument");
        Device::get().require();
        hipStream_t s = Device::get().stream;
        DockSet D(nleaf, leaves, s);
        azimuthal_average(D, npts, q, theta, nphi, seed, intensity, s);
        timing_collect();
    })
}

int dplus_dock_grid(dplus_grid *outh, int nleaf, const dplus_leaf *leaves, double scale) {
    API_GUARD({
        Grid *out = (Grid *)outh;
        if (!out || !leaves) throw Error(kErrInvalidArgs, "null argument");
        Device::get().require();
        hipStream_t s = Device::get().stream;
        DockSet D(nleaf, leaves, s);
        if (D.fp64 != out->fp64()) throw Error(kErrInvalidArgs, "output precision differs from the leaves'");
        dock_grid(D, *out, scale, s);
    })
}

int dplus_dock_grid_space_filling(dplus_grid *outh, int nleaf, const dplus_leaf *leaves, double scale,
                                  const double *distances, const double *angles_deg, const double *reps) {
    API_GUARD({
        Grid *out = (Grid *)outh;
        if (!out || !leaves || !distances || !angles_deg || !reps) throw Error(kErrInvalidArgs, "null argument");
        Device::get().require();
        hipStream_t s = Device::get().stream;
        LatticeDev lat = space_filling_lattice(distances, angles_deg, reps);
        DockSet D(nleaf, leaves, s);
        if (D.fp64 != out->fp64()) throw Error(kErrInvalidArgs, "output precision differs from the leaves'");
        dock_grid(D, *out, scale, s, &lat);
    })
}

int dplus_structure_create(const dplus_pdb_desc *d, dplus_structure **out) {
    API_GUARD({
        if (!d || !out) throw Error(kErrInvalidArgs, "null argument");
        Device::get().require();
        *out = (dplus_structure *)new Structure(d, Device::get().stream);
    })
}

void dplus_structure_destroy(dplus_structure *s) { delete (Structure *)s; }

int dplus_structure_build_grid(dplus_structure *sh, dplus_grid *gh, int host_copy) {
    API_GUARD({
        Structure *st = (Structure *)sh;
        Grid *g = (Grid *)gh;
        if (!st || !g) throw Error(kErrInvalidArgs, "null argument");
        Device::get().require();
        st->build(*g, host_copy != 0, Device::get().stream);
    })
}

int dplus_structure_build_grids(int n, dplus_structure *const *sh, dplus_grid *const *gh, int host_copy) {
    API_GUARD({
        if (n < 0 || (n > 0 && (!sh || !gh))) throw Error(kErrInvalidArgs, "null argument");
        for (int i = 0; i < n; i++) {
            if (!sh[i] || !gh[i]) throw Error(kErrInvalidArgs, "null structure or grid");
            for (int k = 0; k < i; k++)
                if (gh[k] == gh[i]) throw Error(kErrInvalidArgs, "a grid appears twice in one grouped build");
        }
        Device::get().require();
        const hipStream_t s = Device::get().stream;
        // mixed grids in grouped launches of up to 16 per phase form; FP64 grids and those of the
        // mesh builder one by one (its workspaces released in stream order as it goes)
        std::vector<int> mixed;
        for (int i = 0; i < n; i++) {
            Grid *g = (Grid *)gh[i];
            Structure *st = (Structure *)sh[i];
            MeshPlan mp;
            MeshSizes mz;
            if (g->fp64() || getenv("DPLUS_PHASE64")) {
                st->build(*g, host_copy != 0, s);
            } else if (st->mesh_route(*g, mp, mz)) {
                Structure::Pending P;
                const BuildShape sh = st->shape_for(*g);
                BuildJob J = st->prepare(*g, sh.slices, P, s);
                {
                    KTimer kt("build", s);
                    st->launch(*g, J, sh.wg, P, s);
                }
                st->enqueue_finish(*g, P, s, true);
                if (host_copy) g->download(s);
            } else {
                mixed.push_back(i);
            }
        }
        std::vector<Structure::Pending> P(mixed.size());
        std::vector<BuildJob> jobs(mixed.size());
        for (size_t k = 0; k < mixed.size(); k++) {
            Structure *st = (Structure *)sh[mixed[k]];
            Grid *g = (Grid *)gh[mixed[k]];
            jobs[k] = st->prepare(*g, st->shape_for(*g).slices, P[k], s);
        }
        {
            KTimer kt("build", s);
            for (int red = 0; red < 2; red++) {
                std::vector<BuildJob> batch;
                for (size_t k = 0; k < mixed.size(); k++) {
                    if ((int)P[k].reduce != red) continue;
                    batch.push_back(jobs[k]);
                    if ((int)batch.size() == kMaxBuildJobs) {
                        launch_build_batch(red != 0, 256, batch.data(), (int)batch.size(), s);
                        batch.clear();
                    }
                }
                if (!batch.empty()) launch_build_batch(red != 0, 256, batch.data(), (int)batch.size(), s);
            }
            check_hip(hipGetLastError(), "grouped build launch");
        }
        for (size_t k = 0; k < mixed.size(); k++)
            ((Structure *)sh[mixed[k]])->finish(*(Grid *)gh[mixed[k]], P[k], host_copy != 0, s);
        check_hip(hipStreamSynchronize(s), "grouped build");
        timing_collect();
    })
}

int dplus_structure_build_shape(dplus_structure *sh, dplus_grid *gh, int *wg, int *slices, int *tuned) {
    API_GUARD({
        Structure *st = (Structure *)sh;
        Grid *g = (Grid *)gh;
        if (!st || !g) throw Error(kErrInvalidArgs, "null argument");
        BuildShape b;
        const bool t = !g->fp64() && shape_lookup(g->N, st->ntiles, &b);
        if (!t) b = st->shape_for(*g);
        if (wg) *wg = b.wg;
        if (slices) *slices = b.slices;
        if (tuned) *tuned = t ? 1 : 0;
    })
}

int dplus_structure_build_route(dplus_structure *sh, dplus_grid *gh, int *mesh) {
    API_GUARD({
        const Structure *st = (const Structure *)sh;
        const Grid *g = (const Grid *)gh;
        if (!st || !g || !mesh) throw Error(kErrInvalidArgs, "null argument");
        MeshPlan P;
        MeshSizes Z;
        const bool paired = g->fp64() ? !fp64_plain_builder() : getenv("DPLUS_PHASE64") == nullptr;
        *mesh = paired && st->mesh_route(*g, P, Z) ? 1 : 0;
    })
}

int dplus_set_fp64_builder(int plain) {
    API_GUARD({
        if (plain != 0 && plain != 1) throw Error(kErrInvalidArgs, "the FP64 builder form is 0 (paired) or 1 (plain)");
        set_fp64_plain_builder(plain != 0);
    })
}

int dplus_build_shapes_clear(void) {
    API_GUARD({
        std::lock_guard<std::mutex> lk(shape_mu);
        shape_table.clear();
    })
}

int dplus_structure_autotune(dplus_structure *sh, dplus_grid *gh, int *wg, int *slices, double *best_ms,
                             double *model_ms) {
    API_GUARD({
        Structure *st = (Structure *)sh;
        Grid *g = (Grid *)gh;
        if (!st || !g) throw Error(kErrInvalidArgs, "null argument");
        Device::get().require();
        double tb = 0.0, tm = 0.0;
        const BuildShape b = st->autotune(*g, Device::get().stream, &tb, &tm);
        if (wg) *wg = b.wg;
        if (slices) *slices = b.slices;
        if (best_ms) *best_ms = tb;
        if (model_ms) *model_ms = tm;
    })
}

int dplus_build_shapes_save(char **text, long long *len) {
    API_GUARD({
        if (!text || !len) throw Error(kErrInvalidArgs, "null argument");
        std::string out;
        {
            std::lock_guard<std::mutex> lk(shape_mu);
            for (auto &kv : shape_table)
                out += std::to_string(kv.first.first) + " " + std::to_string(kv.first.second) + " " +
                       std::to_string(kv.second.wg) + " " + std::to_string(kv.second.slices) + "\n";
        }
        *text = (char *)malloc(out.size() + 1);
        if (!*text) throw Error(kErrOutOfMemory, "out of host memory");
        memcpy(*text, out.data(), out.size());
        (*text)[out.size()] = '\0';
        *len = (long long)out.size();
    })
}

int dplus_build_shapes_load(const char *text) {
    API_GUARD({
        if (!text) throw Error(kErrInvalidArgs, "null argument");
        std::vector<std::pair<std::pair<int, int>, BuildShape>> rows;
        const char *p = text;
        while (*p) {
            while (*p == ' ' || *p == '\n' || *p == '\r' || *p == '\t') p++;
            if (!*p) break;
            if (*p == '#') {  // comment line
                while (*p && *p != '\n') p++;
                continue;
            }
            int n = 0, c = 0, w = 0, sl = 0, used = 0;
            if (sscanf(p, "%d %d %d %d%n", &n, &c, &w, &sl, &used) != 4)
                throw Error(kErrInvalidArgs, "shape table line is not \"grid_shells tile_class wg slices\"");
            if (n < 1 || (w != 64 && w != 128 && w != 256 && w != 512) || sl < 1 || sl > kMaxSlices)
                throw Error(kErrInvalidArgs, "shape table entry out of range");
            BuildShape b;
            b.wg = w;
            b.slices = sl;
            rows.push_back({{n, c}, b});
            p += used;
        }
        std::lock_guard<std::mutex> lk(shape_mu);
        for (auto &r : rows) shape_table[r.first] = r.second;
    })
}

int dplus_timing_enable(int on) {
    API_GUARD({
        timing_collect();
        timing_set(on != 0);
    })
}

int dplus_timing_get(const char *kernel, long long *launches, double *ms) {
    API_GUARD({
        if (!kernel) throw Error(kErrInvalidArgs, "null kernel name");
        timing_collect();
        timing_read(kernel, launches, ms);
    })
}

int dplus_timing_reset(void) {
    API_GUARD({
        timing_collect();
        timing_clear();
    })
}

int dplus_microbench_valu(double *fma32, double *sin32, double *cos32, double *fma64) {
    API_GUARD({
        Device::get().require();
        microbench_valu(Device::get().stream, fma32, sin32, cos32, fma64);
    })
}

int dplus_copy_probe(long long bytes, double *ms) {
    API_GUARD({
        if (bytes <= 0 || bytes % 16) throw Error(kErrInvalidArgs, "bytes must be a positive multiple of 16");
        Device::get().require();
        copy_probe(Device::get().stream, bytes, ms);
    })
}

int dplus_gather_probe(dplus_grid *gh, int nrot, const double *rot, long long directions, int layer0, int nlayers,
                       double *ms, double *lookups) {
    API_GUARD({
        Grid *g = (Grid *)gh;
        if (!g || g->fp64()) throw Error(kErrInvalidArgs, "the gather probe reads a mixed-precision grid");
        if (nrot < 0 || (nrot > 0 && !rot) || directions < 256 || directions % 256 || layer0 < 0 || nlayers < 1 ||
            layer0 + nlayers > g->N - 1)
            throw Error(kErrInvalidArgs, "bad gather-probe arguments");
        if (directions / 256 > 2147483647LL) throw Error(kErrInvalidArgs, "too many directions");
        Device::get().require();
        hipStream_t s = Device::get().stream;
        const int nblk = (int)(directions / 256);
        const int chunk = directions % 8192 == 0 ? 8192 : 256;
        DevBuf brot, bsink;
        std::vector<RotDev> rots((size_t)std::max(1, nrot));
        for (int r = 0; r < nrot; r++) {
            euler_rt(rot[4 * r], rot[4 * r + 1], rot[4 * r + 2], rots[r].m);
            rots[r].scale = rot[4 * r + 3];
            rots[r].leaf = rots[r].t0 = rots[r].pad = 0;
            rots[r].nt = 1;
        }
        brot.upload(rots.data(), rots.size() * sizeof(RotDev), s);
        bsink.ensure((size_t)nblk * nlayers * 4 * sizeof(float));
        hipEvent_t e0, e1;
        check_hip(hipEventCreate(&e0), "event");
        check_hip(hipEventCreate(&e1), "event");
        // one untimed launch brings the grid into the caches, as in an average
        launch_gather_probe(g->dev.p, g->N, nrot ? (const RotDev *)brot.p : nullptr, std::max(1, nrot), layer0,
                            nlayers, nblk, 12345, chunk, (float *)bsink.p, s);
        check_hip(hipEventRecord(e0, s), "record");
        launch_gather_probe(g->dev.p, g->N, nrot ? (const RotDev *)brot.p : nullptr, std::max(1, nrot), layer0,
                            nlayers, nblk, 777, chunk, (float *)bsink.p, s);
        check_hip(hipGetLastError(), "gather probe launch");
        check_hip(hipEventRecord(e1, s), "record");
        check_hip(hipEventSynchronize(e1), "sync");
        float t = 0.f;
        check_hip(hipEventElapsedTime(&t, e0, e1), "elapsed");
        (void)hipEventDestroy(e0);
        (void)hipEventDestroy(e1);
        if (ms) *ms = t;
        if (lookups) *lookups = (double)directions * nlayers * std::max(1, nrot);
    })
}

int dplus_synth_walk(unsigned long long seed, int n, double step, double min_sep, double ax, double ay, double az,
                     double *xyz) {
    API_GUARD({
        if (n < 0 || !xyz || step <= 0 || min_sep < 0 || ax <= 0 || ay <= 0 || az <= 0)
            throw Error(kErrInvalidArgs, "bad walk parameters");
        synth_walk(seed, n, step, min_sep, ax, ay, az, xyz);
    })
}

}  // extern "C"
