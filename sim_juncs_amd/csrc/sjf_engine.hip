// sjf_engine.hip -- host side of the MI355X FDTD engine behind include/sjf.h.
//
// An engine owns the device state of one simulation (fields, materials, PML auxiliaries,
// polarisation state, sources, monitors, DFT accumulators).  Stepping goes through a launch
// set: one engine, or a batch of engines, compiled into small device tables so that each
// time step is a fixed sequence of launches on one stream,
//   [k_monitor when step % save_span == 0] -> k_step -> [k_source] -> [k_dft] (or k_tick),
// the last of which advances the step counters, whatever the number of instances; source and
// DFT share one launch (k_source_dft) when no DFT region holds a source cell.  The per-step
// scalars (step index, pulse value, DFT phase) are computed on the device from each engine's
// step counter, so a run of steps is
// captured once in a hipGraph and replayed.  This is the sequence bound_geom::run performs
// around fields.step() (reference src/disp.cpp:719-741).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <climits>
#include <cmath>
#include <cstdio>
#include <cstring>
#include <mutex>
#include <string>
#include <type_traits>
#include <vector>

#include "../../include/sjf.h"
#include "sjf_kernels.h"

using sjf::kMaxPoles;

namespace {

thread_local std::string g_create_error;

struct Source {
    int comp;
    sjf_pulse p;
    sjf::PulseDev dev;
    std::vector<long> idx;
    std::vector<double> wt;
    std::vector<int> ids[3];  // its cells: the product of these, each ascending
};

struct Monitor {
    int comp;
    long idx[8];
    double w[8];
};

struct Dft {
    int lo[3], hi[3];
    int mask;
    std::vector<double> freqs;
    long ncell;
    int ncomp;
    int comps[6];
    double2* acc = nullptr;
    double2* cmp = nullptr;
    double* d_freq = nullptr;
};

struct LaunchSet;

}  // namespace

struct sjf_engine {
    sjf_grid g{};
    int prec = 4;
    long N = 0;
    double dt = 0;
    hipStream_t stream = nullptr;
    std::string err;
    long version = 0;  // bumped by every change that invalidates compiled launch tables

    void* Fbuf[2] = {};  // field sets [x][Ex Ey Ez Hx Hy Hz][y][z]; step n reads set n&1
    long* d_step = nullptr;  // step counter and its shadow (sjf_kernels.h)
    long step = 0;

    // materials: given* as the caller set them; matw / lut_h / nmat / maxp are what the kernels run
    // (the given map, with Lorentz poles folded out of the PML slabs when pml_fref > 0: twin)
    bool have_mat = false;
    bool mat_ready = true;  // false from the first change a call makes until it has made all of them
    uint32_t* given = nullptr;  // device, [x][y][z]
    std::vector<sjf_material> given_lut;
    double pml_fref = 0;
    std::vector<int> twin;  // per given material its id in the PML slabs, or -1
    std::vector<sjf_material> lut_h;
    uint32_t* matw = nullptr;
    uint32_t* seg = nullptr;  // material segment codes (k_words)
    double pole_bytes = 0;    // pole state the step moves
    double pole_values = 0;   // poles summed over cells and components
    size_t pol_bytes = 0;     // size of Qbuf (and of Pbuf where there is one)
    void* lut = nullptr;
    int nmat = 1;
    int maxp = 0;
    void* Qbuf = nullptr;  // [x][slot * 3 + comp][y][z]
    void* Pbuf = nullptr;  // the same, present when a slot holds a Lorentz pole
    bool uniform = true;
    int dlo[3] = {0, 0, 0}, dhi[3] = {0, 0, 0};
    std::vector<double> deps_h;
    void* dinv = nullptr;
    std::vector<double> emap_h;  // per-cell eps_inf [Ex Ey Ez][x][y][z] as given (sjf_set_eps_maps)
    std::vector<double> emap_eff;  // as run (Lorentz poles folded in inside the PML slabs)
    void* emap = nullptr;          // 1/eps_inf on the device, [x][Ex Ey Ez][y][z]

    // PML
    int pml[6] = {0, 0, 0, 0, 0, 0};
    bool pml_on[3] = {false, false, false};
    bool pml_ready = true;    // as mat_ready
    void* coefbuf = nullptr;  // per axis: bE[n], aE[n], bH[n], aH[n]
    int coff[3] = {0, 0, 0};
    long slab[3] = {0, 0, 0};
    void* psibuf[3] = {};  // per axis [3][slab][2]: E pair, H pairs A and B

    std::vector<Source> src;
    std::vector<Monitor> mon;
    int save_span = 1;
    long nsamp = 0, samp_cap = 0;
    double* d_samples = nullptr;
    std::vector<Dft> dft;

    int form = SJF_TILE_REGISTER_ROWS;  // fused-kernel form
    int ty = 1, xc = 16;                // y rows per thread (register form) or per workgroup
    int zseg = 0;                       // register form: z cells per workgroup pass (0: default)
    bool tile_set = false;
    int graph_chunk = 32;  // steps per captured graph (0: no graphs)

    // fused reverse-step kernel of the last adjoint run: mean duration and launch shape
    double adj_ms = 0;
    int adj_threads = 0, adj_groups = 0;
    // its tile (sjf_set_adjoint_tile): form, owned rows of a row-of-threads tile, x-chunk (0: default)
    int adj_form = SJF_TILE_REGISTER_ROWS;
    int adj_rows = 0, adj_xc = 0;
    bool adj_set = false;  // set by sjf_set_adjoint_tile (else the default of adj_tile_of)

    LaunchSet* own = nullptr;
    sjf_batch* batch = nullptr;
};

namespace {

#define HIPCHK(e, call)                                                                  \
    do {                                                                                 \
        hipError_t _st = (call);                                                         \
        if (_st != hipSuccess) {                                                         \
            (e)->err = std::string(#call) + ": " + hipGetErrorString(_st);               \
            return SJF_E_HIP;                                                            \
        }                                                                                \
    } while (0)

int fail(sjf_engine* e, int code, const std::string& m) {
    e->err = m;
    return code;
}

// A failed allocation is reported by its own call alone: the error it leaves behind would otherwise be
// taken for that of the next launch, and a step that has run be reported as failed.
hipError_t device_malloc(void** p, size_t bytes) {
    const hipError_t st = hipMalloc(p, bytes);
    if (st != hipSuccess) (void)hipGetLastError();
    return st;
}

int dev_alloc(sjf_engine* e, void** p, size_t bytes) {
    if (*p) return SJF_OK;
    hipError_t st = device_malloc(p, bytes ? bytes : 16);
    if (st != hipSuccess) {
        *p = nullptr;
        e->err = std::string("hipMalloc(") + std::to_string(bytes) + "): " + hipGetErrorString(st);
        return SJF_E_NOMEM;
    }
    st = hipMemsetAsync(*p, 0, bytes ? bytes : 16, e->stream);
    if (st == hipSuccess) st = hipStreamSynchronize(e->stream);
    if (st != hipSuccess) return fail(e, SJF_E_HIP, hipGetErrorString(st));
    return SJF_OK;
}

template <typename P>
void dev_free(P*& p) {
    if (p) (void)hipFree((void*)p);
    p = nullptr;
}

// All copies are ordered on the engine's (non-blocking) stream and completed before return.
int h2d(sjf_engine* e, void* dst, const void* src, size_t bytes) {
    if (bytes == 0) return SJF_OK;
    HIPCHK(e, hipMemcpyAsync(dst, src, bytes, hipMemcpyHostToDevice, e->stream));
    HIPCHK(e, hipStreamSynchronize(e->stream));
    return SJF_OK;
}

int d2h(sjf_engine* e, void* dst, const void* src, size_t bytes) {
    if (bytes == 0) return SJF_OK;
    HIPCHK(e, hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, e->stream));
    HIPCHK(e, hipStreamSynchronize(e->stream));
    return SJF_OK;
}

// the field set read by the next step
void* field_set(sjf_engine* e) { return e->Fbuf[e->step & 1]; }

// byte offset of component comp of cell q in a field set
size_t field_offset(const sjf_engine* e, int comp, long q) {
    return (size_t)e->prec * sjf::field_index(q, comp, (long)e->g.ny * e->g.nz);
}

const double kCompOff[6][3] = {{0.5, 0.0, 0.0}, {0.0, 0.5, 0.0}, {0.0, 0.0, 0.5},
                               {0.0, 0.5, 0.5}, {0.5, 0.0, 0.5}, {0.5, 0.5, 0.0}};

long cell_index(const sjf_engine* e, int i, int j, int k) {
    return ((long)i * e->g.ny + j) * e->g.nz + k;
}

int axis_n(const sjf_engine* e, int d) { return d == 0 ? e->g.nx : (d == 1 ? e->g.ny : e->g.nz); }

// Weights of an extent [lo, hi] on the lattice (i + off) dx: delta function (linear / dx) for
// zero extent, cell overlap / dx otherwise.
void axis_weights(int n, double dx, double off, int periodic, double lo, double hi,
                  std::vector<int>& ids, std::vector<double>& w) {
    ids.clear();
    w.clear();
    if (hi < lo) std::swap(lo, hi);
    if (hi - lo < 1e-9 * dx) {
        const double s = lo / dx - off;
        const double fl = std::floor(s);
        const int i0 = (int)fl;
        const double f = s - fl;
        for (int q = 0; q < 2; ++q) {
            int i = i0 + q;
            const double ww = (q == 0 ? 1.0 - f : f) / dx;
            if (ww == 0.0) continue;
            if (periodic) i = ((i % n) + n) % n;
            else if (i < 0 || i >= n) continue;
            if (!ids.empty() && ids.back() == i) {  // a periodic axis of one cell: both images are it
                w.back() += ww;
                continue;
            }
            ids.push_back(i);
            w.push_back(ww);
        }
        return;
    }
    // on a periodic axis the cell of lattice point p also has images p +- n dx
    for (int i = 0; i < n; ++i) {
        double ww = 0;
        for (int m = periodic ? -1 : 0; m <= (periodic ? 1 : 0); ++m) {
            const double p = (i + off) * dx + m * n * dx;
            const double a = std::max(lo, p - 0.5 * dx), b = std::min(hi, p + 0.5 * dx);
            if (b > a) ww += (b - a) / dx;
        }
        if (ww > 0) {
            ids.push_back(i);
            w.push_back(ww);
        }
    }
}

// 1/eps at component c of cell q, whose material word (as the kernels run it) is w
double inv_eps_at(const sjf_engine* e, long q, int c, uint32_t w) {
    if (!e->have_mat) return 1.0;
    const int m = (w >> (8 * c)) & 0xff;
    if (m == e->nmat) {
        const int k = (int)(q % e->g.nz);
        const long r = q / e->g.nz;
        const int j = (int)(r % e->g.ny), i = (int)(r / e->g.ny);
        const long dq = ((long)(i - e->dlo[0]) * (e->dhi[1] - e->dlo[1]) + (j - e->dlo[1])) *
                            (e->dhi[2] - e->dlo[2]) +
                        (k - e->dlo[2]);
        return 1.0 / e->deps_h[dq];
    }
    if (!e->emap_eff.empty()) return 1.0 / e->emap_eff[(size_t)c * e->N + q];
    return 1.0 / e->lut_h[m].eps_inf;
}

// Pinned host memory of the read-outs.  A read-out takes a buffer for its duration and gives it back; at
// most kStageKept bytes are kept for later ones (two large read-outs at a time), whatever the number of
// engines, and none once the last engine is gone.  Allocating one costs as much as a small read-out.
constexpr size_t kReadChunk = 4u << 20;
constexpr size_t kStageKept = 4 * kReadChunk;
struct Stage {
    void* p;
    size_t bytes;
    int device;
};
std::mutex g_stage_mu;
std::vector<Stage> g_stages;  // given back
size_t g_stage_bytes = 0;     // of these
long g_engines = 0;

void stage_engines(int change) {
    std::vector<Stage> last;
    {
        std::lock_guard<std::mutex> lk(g_stage_mu);
        g_engines += change;
        if (g_engines > 0) return;
        last.swap(g_stages);
        g_stage_bytes = 0;
    }
    for (const Stage& s : last) (void)hipHostFree(s.p);
}

// At least `bytes` of pinned memory while it lives.  done(): the device no longer writes to it.
class StageLease {
public:
    StageLease(sjf_engine* e, size_t bytes) : e_(e) {
        {
            std::lock_guard<std::mutex> lk(g_stage_mu);
            int best = -1;  // the smallest that holds it
            for (int q = 0; q < (int)g_stages.size(); ++q)
                if (g_stages[q].device == e->g.device && g_stages[q].bytes >= bytes &&
                    (best < 0 || g_stages[q].bytes < g_stages[best].bytes))
                    best = q;
            if (best >= 0) {
                s_ = g_stages[best];
                g_stages.erase(g_stages.begin() + best);
                g_stage_bytes -= s_.bytes;
                return;
            }
        }
        s_ = {nullptr, std::max<size_t>(bytes, 4096), e->g.device};
        if (hipHostMalloc(&s_.p, s_.bytes, hipHostMallocDefault) != hipSuccess) {
            (void)hipGetLastError();
            s_.p = nullptr;
            e->err = "read-out buffer allocation failed";
        }
    }
    StageLease(const StageLease&) = delete;
    ~StageLease() {
        if (!s_.p) return;
        if (done_) {
            std::lock_guard<std::mutex> lk(g_stage_mu);
            if (g_stage_bytes + s_.bytes <= kStageKept) {
                g_stages.push_back(s_);
                g_stage_bytes += s_.bytes;
                return;
            }
        } else {
            (void)hipStreamSynchronize(e_->stream);  // a call in between failed
        }
        (void)hipHostFree(s_.p);
    }
    void* get() const { return s_.p; }
    void done() { done_ = true; }

private:
    sjf_engine* e_;
    Stage s_{};
    bool done_ = false;
};

// Material words of the listed cells, through the read-out stage
int words_at(sjf_engine* e, const std::vector<long>& cells, std::vector<uint32_t>& w) {
    const long n = (long)cells.size(), most = (long)(kReadChunk / 16);
    w.assign(n, 0u);
    if (!e->matw) return SJF_OK;  // no materials yet, or refused ones
    if (n == 0) return SJF_OK;
    StageLease stage(e, 16 * (size_t)std::min(n, most));
    if (!stage.get()) return SJF_E_NOMEM;
    for (long q = 0; q < n; q += most) {
        const long m = std::min(most, n - q);
        long* in = (long*)stage.get();
        uint32_t* out = (uint32_t*)(in + m);
        std::memcpy(in, cells.data() + q, sizeof(long) * m);
        hipLaunchKernelGGL(sjf::k_read_words, dim3((unsigned)((m + 255) / 256)), dim3(256), 0, e->stream, e->matw, in, m, out);
        HIPCHK(e, hipGetLastError());
        HIPCHK(e, hipStreamSynchronize(e->stream));
        std::memcpy(w.data() + q, out, sizeof(uint32_t) * m);
    }
    stage.done();
    return SJF_OK;
}

// Row-of-threads form: (rows + 1) thread rows of nz threads per workgroup, 32-bit offsets.
bool thread_rows_fit(const sjf_engine* e, int rows) { return rows >= 1 && (long)(rows + 1) * e->g.nz <= 1024; }

double field_bytes(const sjf_engine* e) { return 12.0 * e->prec * (double)e->N; }

// Bytes one step touches above which its stores take the non-temporal hint: below, the 256 MB Infinity
// Cache holds what a step wrote until the next one reads it.  Pole state counts in whole 64-cell
// segments, so the line lies above that size.  Measured on MI355X, us per step without and with the
// hint: FP64 96x96x96 (184 MB) 39.8, 48.9; FP32 150x150x96 (234 MB) 47.2, 50.2; FP32 150x150x160
// periodic (282 MB) 65.9, 63.4; FP32 151x133x117 (285 MB) 53.8, 57.0; FP64 120x120x96 (291 MB) 67.8,
// 70.4; FP64 128x128x100 (350 MB) 87.5, 78.4; FP32 192x192x96 (386 MB) 80.0, 74.6; FP32 200x200x125
// (592 MB) 125.2, 113.9.
constexpr double kStreamBytes = 300e6;
// What one fused step touches: two field sets, pole state, PML auxiliaries, material words, eps maps
double step_set_bytes(const sjf_engine* e) {
    double b = field_bytes(e) + e->pole_bytes + (e->uniform ? 0.0 : 4.0 * (double)e->N);
    if (e->emap) b += 3.0 * e->prec * (double)e->N;
    for (int d = 0; d < 3; ++d) b += 6.0 * e->prec * (double)e->slab[d];
    return b;
}

// Whether a tile's exchange planes (values) and the coefficients of nmat materials fit 64 KiB.  The
// padded table and a second copy of the planes then stay within the CU's 160 KiB.
template <typename T>
bool lds_fits(size_t values, int nmat) {
    return sizeof(T) * values + (14 * sizeof(T) + 8) * (size_t)nmat <= 65536;
}

// z cells per pass of a register-rows workgroup with `rows` rows per thread: the set value, else the
// whole line, but 128-cell passes for one row per thread on a non-periodic z line longer than the
// 1024 threads of a workgroup.  The tile that the library chooses also takes 256-cell passes in FP64
// above 512 cells (a 1024-thread FP64 workgroup spills) and otherwise spans the line (448x224x512
// FP32: one pass 0.731 ms per step, 128-cell passes 0.846 ms: their tile takes 161 registers, 3 waves
// per SIMD, the one-pass tile 109 and 4); a tile set by the caller (given) keeps its documented
// 128-cell passes on lines above 256 cells that are a multiple of 256.
int zseg_of(const sjf_engine* e, int rows, bool given) {
    const int nz = e->g.nz;
    if (e->zseg > 0) return std::min(e->zseg, nz);
    if (rows == 1 && !e->g.periodic[2]) {
        if (nz > 1024 || (given && nz > 256 && nz % 256 == 0)) return 128;
        if (!given && e->prec == 8 && nz > 512) return 256;
    }
    return nz;
}

// Thread rows a row-of-threads tile owns by default: as many as 1024 threads hold (FP64 512: at 1024
// the register budget of 128 per thread spills) with the halo row, spread evenly over the grid's rows.
int default_thread_rows(const sjf_engine* e) {
    const int most = std::max(1, (e->prec == 8 ? 512 : 1024) / e->g.nz - 1);
    const int tiles = (e->g.ny + most - 1) / most;
    return (e->g.ny + tiles - 1) / tiles;
}

int block_threads_for(const sjf_engine* e, int form, int ty, bool given) {
    const int t = form == SJF_TILE_THREAD_ROWS ? (ty + 1) * e->g.nz : zseg_of(e, ty, given);
    return ((t + 63) / 64) * 64;
}

int block_threads(const sjf_engine* e) { return block_threads_for(e, e->form, e->ty, e->tile_set); }

// x-chunk of a tile with nty rows of tiles: a workgroup's time is its chunk and about `extra` planes
// of start-up, and the chip runs `slots` workgroups at once; a launch that needs a little more than
// a whole number of such rounds waits for a last one that is nearly empty (forward step of
// 192x192x96 FP32, 9 thread rows, 256 slots: 242 workgroups of 18 planes 80.6 us, 264 of 16 planes
// 112 us, 484 of 9 planes 83.9 us).  So: the rounds for which rounds * (chunk + extra) is least, with
// chunks of at most 64 planes (a longer march drifts apart) and at most 16 rounds.
int round_chunk(int nx, int nty, long slots, int extra) {
    long best = LONG_MAX;
    int xc = std::min(nx, 64);
    for (int m = 1; m <= 16; ++m) {
        const long nxc = std::min<long>(nx, m * slots / nty);
        if (nxc < 1) continue;
        const int c = (int)((nx + nxc - 1) / nxc);
        if (c > 64) continue;
        if (m * (long)(c + extra) <= best) best = m * (long)(c + extra), xc = c;
    }
    return xc;
}

// Workgroups of w wavefronts that a CU holds at once where the registers leave `waves` per SIMD.  Beyond
// four wavefronts a workgroup is placed only where every SIMD has room for the most that it puts on one: of
// five wavefronts 3, 2 and 1 fit at 5, 4 and 3 per SIMD, not 4, 3 and 2 (43x46x320 FP32 with gold, 4 per
// SIMD: 690 workgroups of 3 planes 30.3 us, 506 of 4 planes 24.9; without poles, 5 per SIMD: 1012 of 2
// planes 26.2, 690 of 3 22.5; 32x35x300 FP64 without poles, 3 per SIMD: 385 of 3 planes 30.6, 245 of 5
// 25.7), of six 2 and 1 at 5 and 3 (40x43x384 FP32: 602 of 3 planes 27.0, 430 of 4 23.4).
int resident(int w, int waves) {
    const int most = (w + 3) / 4;
    if (w <= 4) return std::max(1, 4 * waves / w);
    int n = std::max(1, waves / most);
    if (w % 4 == 1)  // the odd wavefront goes to another SIMD each time
        for (n = 1; (n * w + 3) / 4 + most <= waves;) ++n;
    return n;
}

// x-chunk of a tile whose workgroups have w wavefronts: round_chunk on the places that the registers leave,
// or, where fewer workgroups are resident and that would make a second round, the shortest chunk that runs
// in one if it saves 15 % of the planes (less was as often lost as gained).
int resident_chunk(int nx, int nty, int w, int waves) {
    const long all = 256L * std::max(1, 4 * waves / w), held = 256L * resident(w, waves);
    const int xc = round_chunk(nx, nty, all, 2);
    if (held >= all || nty > held) return xc;
    const int nxc = (int)std::min<long>(nx, held / nty), one = (nx + nxc - 1) / nxc;
    const long rounds = ((long)nty * ((nx + xc - 1) / xc) + held - 1) / held;
    return one <= 64 && 1.15 * (one + 2) < (double)rounds * (xc + 2) ? one : xc;
}

int tiles_of(const sjf_engine* e, int ty, int xc) {
    const int nty = (e->g.ny + ty - 1) / ty;
    const int nxc = (e->g.nx + xc - 1) / xc;
    return nty * nxc;
}

// Pole slots compiled into the step kernel: 0, 1, 3 or 4 (a material with 2 poles runs the
// 3-slot variant; unused slots are predicated off).
int np_variant_of(int maxp, bool uniform) {
    if (uniform || maxp == 0) return 0;
    if (maxp == 1) return 1;
    if (maxp <= 3) return 3;
    return 4;
}

template <typename T>
sjf::StepArgs<T> step_args(const sjf_engine* e, int ty, int xc, bool given = false) {
    sjf::StepArgs<T> a;
    std::memset(&a, 0, sizeof(a));
    a.rt = ty + 1;
    a.zseg = zseg_of(e, ty, given);
    a.nx = e->g.nx;
    a.ny = e->g.ny;
    a.nz = e->g.nz;
    a.px = e->g.periodic[0];
    a.py = e->g.periodic[1];
    a.pz = e->g.periodic[2];
    a.nty = (e->g.ny + ty - 1) / ty;
    a.xc = xc;
    a.N = e->N;
    a.cdt = (T)(e->dt / e->g.dx);
    a.F[0] = (T*)e->Fbuf[0];
    a.F[1] = (T*)e->Fbuf[1];
    a.d_step = e->d_step;
    a.uniform = e->uniform ? 1 : 0;
    a.nmat = e->nmat;
    a.matw = e->matw;
    a.seg = e->seg;
    a.lut = (const sjf::MatLut<T>*)e->lut;
    a.Q = (T*)e->Qbuf;
    // FP32 slots alternate between two arrays; Drude slots alone are updated in place
    a.P = (T*)(e->Pbuf || !sjf::kPolePair<T> ? e->Pbuf : e->Qbuf);
    a.nqp = e->Qbuf ? 3 * e->maxp : 0;
    for (int d = 0; d < 3; ++d) {
        a.pml_on[d] = e->pml_on[d] ? 1 : 0;
        a.plo[d] = e->pml[2 * d];
        a.phi[d] = e->pml[2 * d + 1];
        a.S[d] = e->slab[d];
        a.psi[d] = (T*)e->psibuf[d];
        a.coff[d] = e->coff[d];
        a.dlo[d] = e->dlo[d];
        a.dhi[d] = e->dhi[d];
    }
    a.coef = (const T*)e->coefbuf;
    a.dinv = (const T*)e->dinv;
    a.emap = (const T*)e->emap;
    return a;
}

// ======================================================================== launch sets =====

struct LaunchSet {
    std::vector<sjf_engine*> eng;
    hipStream_t stream = nullptr;
    bool own_stream = false;
    int prec = 4, ty = 1, npv = 0, block = 64;
    int form = SJF_TILE_REGISTER_ROWS;
    int xc = 0;  // x-chunk of every instance of a batch (0: each engine's own)
    bool tile_set = false;  // form and xc of a batch were set by the caller
    bool zpass = false;  // register form with some z line stepped in passes (k_step_z)
    bool nts = false;    // stores with the non-temporal hint (step_set_bytes > kStreamBytes)
    size_t lds = 0;
    std::vector<long> versions;
    bool built = false;
    // step kernel tables
    void* d_args = nullptr;
    int* d_tile_first = nullptr;
    int ntiles = 0;
    // sources
    void* d_src = nullptr;
    int* d_blk_src = nullptr;
    long* d_blk_first = nullptr;
    long* d_blk_end = nullptr;
    long* d_src_idx = nullptr;
    double* d_src_coef = nullptr;
    std::vector<int> src_at;  // first workgroup of each layer (source_layers) and their number
    // magnetic sources (injected into H before the fused update), same table layout
    void* d_hsrc = nullptr;
    int* d_hblk_src = nullptr;
    long* d_hblk_first = nullptr;
    long* d_hblk_end = nullptr;
    long* d_hsrc_idx = nullptr;
    double* d_hsrc_coef = nullptr;
    std::vector<int> hsrc_at;
    // monitors
    void* d_mon = nullptr;
    int nmon = 0;
    // DFT
    void* d_dft = nullptr;
    int ndft = 0;
    long dft_total = 0;
    int dft_blocks = 0;  // workgroups of one frequency
    int dft_maxnf = 0;   // most frequencies of any region (the launch's second dimension)
    bool src_dft_one_launch = false;  // no DFT region holds a source cell: one launch for both
    // step counters, which the last kernel of a step advances
    long** d_counters = nullptr;
    // graph
    hipGraph_t graph = nullptr;
    hipGraphExec_t gexec = nullptr;
    long gK = 0;
};

void set_free_tables(LaunchSet* s) {
    dev_free(s->d_args);
    dev_free(s->d_tile_first);
    dev_free(s->d_src);
    dev_free(s->d_blk_src);
    dev_free(s->d_blk_first);
    dev_free(s->d_blk_end);
    dev_free(s->d_src_idx);
    dev_free(s->d_src_coef);
    dev_free(s->d_hsrc);
    dev_free(s->d_hblk_src);
    dev_free(s->d_hblk_first);
    dev_free(s->d_hblk_end);
    dev_free(s->d_hsrc_idx);
    dev_free(s->d_hsrc_coef);
    s->src_at.clear();
    s->hsrc_at.clear();
    dev_free(s->d_mon);
    dev_free(s->d_dft);
    dev_free(s->d_counters);
    if (s->gexec) (void)hipGraphExecDestroy(s->gexec);
    if (s->graph) (void)hipGraphDestroy(s->graph);
    s->gexec = nullptr;
    s->graph = nullptr;
    s->gK = 0;
    s->built = false;
}

template <typename V>
int upload_vec(sjf_engine* e, hipStream_t st, void** dst, const std::vector<V>& v) {
    const size_t bytes = sizeof(V) * std::max<size_t>(v.size(), 1);
    hipError_t rc = device_malloc(dst, bytes);
    if (rc != hipSuccess) return fail(e, SJF_E_NOMEM, "launch table allocation failed");
    if (!v.empty()) {
        rc = hipMemcpyAsync(*dst, v.data(), sizeof(V) * v.size(), hipMemcpyHostToDevice, st);
        if (rc == hipSuccess) rc = hipStreamSynchronize(st);
        if (rc != hipSuccess) return fail(e, SJF_E_HIP, hipGetErrorString(rc));
    }
    return SJF_OK;
}

// Whether two sources inject into a common value
bool sources_meet(const Source& a, const Source& b) {
    if (a.comp != b.comp) return false;
    for (int d = 0; d < 3; ++d) {
        size_t i = 0, j = 0;
        const std::vector<int>&p = a.ids[d], &q = b.ids[d];
        while (i < p.size() && j < q.size() && p[i] != q[j]) ++(p[i] < q[j] ? i : j);
        if (i == p.size() || j == q.size()) return false;
    }
    return true;
}

// Layer of each source of an engine: sources of a layer share no value, so that one launch adds them
// without a race; sources that meet are added in the order in which they were given.
std::vector<int> source_layers(const std::vector<Source>& src) {
    std::vector<int> layer(src.size(), 0);
    for (size_t b = 1; b < src.size(); ++b)
        for (size_t a = 0; a < b; ++a)
            if (layer[a] >= layer[b] && sources_meet(src[a], src[b])) layer[b] = layer[a] + 1;
    return layer;
}

template <typename T>
int build_set_t(LaunchSet* s) {
    sjf_engine* e0 = s->eng[0];
    set_free_tables(s);
    // step kernel
    std::vector<sjf::StepArgs<T>> args;
    std::vector<int> first;
    int maxp = 0, block = 64;
    bool all_uniform = true;
    int t = 0;
    size_t zh = 0;  // register form with z passes: values of the pass halo in LDS
    for (sjf_engine* e : s->eng) {
        if (!e->mat_ready) return fail(e0, SJF_E_STATE, "the materials are incomplete: the call that last set them failed");
        if (!e->pml_ready) return fail(e0, SJF_E_STATE, "the PML is incomplete: the call that last set it failed");
        // the engine's own set runs its tuned rows; a batch picks rows per engine for its form
        const int rows = (s == e->own) ? e->ty
                                       : (s->form == SJF_TILE_THREAD_ROWS ? default_thread_rows(e) : s->ty);
        const int xc = (s == e->own || s->xc <= 0) ? e->xc : std::min(s->xc, e->g.nx);
        const bool given = s == e->own ? e->tile_set : s->tile_set;
        args.push_back(step_args<T>(e, rows, xc, given));
        first.push_back(t);
        t += tiles_of(e, rows, xc);
        maxp = std::max(maxp, e->maxp);
        all_uniform = all_uniform && e->uniform;
        block = std::max(block, block_threads_for(e, s->form, rows, given));
        if (s->form == SJF_TILE_REGISTER_ROWS && zseg_of(e, rows, given) < e->g.nz) {
            if (rows != 1) return fail(e0, SJF_E_UNSUPPORTED, "z passes run one row per thread");
            zh = std::max<size_t>(zh, 4 * (size_t)xc);
        }
        if (block_threads_for(e, s->form, rows, given) > 1024)
            return fail(e0, SJF_E_UNSUPPORTED, "a z line longer than 1024 cells needs one row per thread (z passes)");
    }
    s->zpass = zh > 0;
    double fb = 0;
    for (sjf_engine* e : s->eng) fb += step_set_bytes(e);
    s->nts = fb > kStreamBytes;
    first.push_back(t);
    s->ntiles = t;
    s->block = block;
    s->npv = np_variant_of(maxp, all_uniform);
    int nmat = 1;
    for (sjf_engine* e : s->eng) nmat = std::max(nmat, e->nmat);
    s->lds = (s->form == SJF_TILE_THREAD_ROWS ? sizeof(T) * 12 * block : sizeof(T) * 4 * s->ty * (block + 1)) +
             sjf::lut_lds_bytes<T>(nmat) + sizeof(T) * zh;
    // (the row-of-threads tile holds its exchange planes twice: 64 KiB bound one copy)
    if (!lds_fits<T>((s->form == SJF_TILE_THREAD_ROWS ? 6 : 4 * s->ty) * (size_t)block + zh, nmat))
        return fail(e0, SJF_E_UNSUPPORTED, "tile needs more than 64 KiB of LDS; use fewer rows");
    int rc = upload_vec(e0, s->stream, &s->d_args, args);
    if (!rc) rc = upload_vec(e0, s->stream, (void**)&s->d_tile_first, first);
    if (rc) return rc;

    // sources: entries of every source of every engine, in blocks of 256 of one source, layer by layer;
    // electric sources (coefficient dt * weight / eps) and magnetic ones (dt * weight, mu = 1) in
    // separate tables
    std::vector<std::vector<int>> layers;
    int nlayer = 0;
    for (sjf_engine* e : s->eng) {
        layers.push_back(source_layers(e->src));
        for (const int l : layers.back()) nlayer = std::max(nlayer, l + 1);
    }
    for (int mag = 0; mag < 2; ++mag) {
        std::vector<sjf::SrcDev<T>> srcs;
        std::vector<int> blk_src, at(1, 0);
        std::vector<long> blk_first, blk_end, idx;
        std::vector<double> coef;
        for (int layer = 0; layer < nlayer; ++layer) {
            for (size_t i = 0; i < s->eng.size(); ++i) {
                sjf_engine* e = s->eng[i];
                for (size_t k = 0; k < e->src.size(); ++k) {
                    const Source& src = e->src[k];
                    if (layers[i][k] != layer || src.idx.empty() || (src.comp >= 3) != (mag == 1)) continue;
                    sjf::SrcDev<T> d;
                    std::memset(&d, 0, sizeof(d));
                    d.p = src.dev;
                    d.p.part = e->g.part;
                    d.p.dt = e->dt;
                    for (int b = 0; b < 2; ++b) d.F[b] = (T*)e->Fbuf[b];
                    d.d_step = e->d_step;
                    const int sid = (int)srcs.size();
                    srcs.push_back(d);
                    const long base = (long)idx.size();
                    std::vector<uint32_t> word;
                    if (!mag && (rc = words_at(e, src.idx, word))) return rc;
                    for (size_t q = 0; q < src.idx.size(); ++q) {
                        idx.push_back(sjf::field_index(src.idx[q], src.comp, (long)e->g.ny * e->g.nz));
                        coef.push_back(e->dt * src.wt[q] * (mag ? 1.0 : inv_eps_at(e, src.idx[q], src.comp, word[q])));
                    }
                    const long n = (long)src.idx.size();
                    for (long b = 0; b < n; b += 256) {
                        blk_src.push_back(sid);
                        blk_first.push_back(base + b);
                        blk_end.push_back(base + std::min(n, b + 256));
                    }
                }
            }
            if ((int)blk_src.size() > at.back()) at.push_back((int)blk_src.size());
        }
        const int nblk = (int)blk_src.size();
        if (!nblk) continue;
        void** tsrc = mag ? &s->d_hsrc : &s->d_src;
        int** tbs = mag ? &s->d_hblk_src : &s->d_blk_src;
        long** tbf = mag ? &s->d_hblk_first : &s->d_blk_first;
        long** tbe = mag ? &s->d_hblk_end : &s->d_blk_end;
        long** tidx = mag ? &s->d_hsrc_idx : &s->d_src_idx;
        double** tcoef = mag ? &s->d_hsrc_coef : &s->d_src_coef;
        (mag ? s->hsrc_at : s->src_at) = at;
        rc = upload_vec(e0, s->stream, tsrc, srcs);
        if (!rc) rc = upload_vec(e0, s->stream, (void**)tbs, blk_src);
        if (!rc) rc = upload_vec(e0, s->stream, (void**)tbf, blk_first);
        if (!rc) rc = upload_vec(e0, s->stream, (void**)tbe, blk_end);
        if (!rc) rc = upload_vec(e0, s->stream, (void**)tidx, idx);
        if (!rc) rc = upload_vec(e0, s->stream, (void**)tcoef, coef);
        if (rc) return rc;
    }

    // monitors
    std::vector<sjf::MonDev<T>> mons;
    for (sjf_engine* e : s->eng) {
        for (size_t p = 0; p < e->mon.size(); ++p) {
            sjf::MonDev<T> m;
            std::memset(&m, 0, sizeof(m));
            const int c = e->mon[p].comp;
            for (int b = 0; b < 2; ++b) m.F[b] = (const T*)e->Fbuf[b];
            m.d_step = e->d_step;
            m.out = e->d_samples;
            m.npt = (int)e->mon.size();
            m.p = (int)p;
            m.span = e->save_span;
            for (int q = 0; q < 8; ++q) {
                const long cq = e->mon[p].idx[q];
                m.idx[q] = cq >= 0 ? sjf::field_index(cq, c, (long)e->g.ny * e->g.nz) : -1;
                m.w[q] = e->mon[p].w[q];
            }
            mons.push_back(m);
        }
    }
    s->nmon = (int)mons.size();
    if (s->nmon) {
        rc = upload_vec(e0, s->stream, &s->d_mon, mons);
        if (rc) return rc;
    }

    // DFT regions
    std::vector<sjf::DftDev<T>> regs;
    long tot = 0;
    for (sjf_engine* e : s->eng) {
        for (const Dft& d : e->dft) {
            sjf::DftDev<T> r;
            std::memset(&r, 0, sizeof(r));
            for (int b = 0; b < 2; ++b) r.F[b] = (const T*)e->Fbuf[b];
            r.d_step = e->d_step;
            r.N = e->N;
            r.nyz = (long)e->g.ny * e->g.nz;
            r.nz = e->g.nz;
            for (int q = 0; q < 3; ++q) {
                r.lo[q] = d.lo[q];
                r.ext[q] = d.hi[q] - d.lo[q];
            }
            r.ncell = d.ncell;
            r.first = tot;
            for (int q = 0; q < 6; ++q) r.comps[q] = d.comps[q];
            r.ncomp = d.ncomp;
            r.nf = (int)d.freqs.size();
            r.freq = d.d_freq;
            r.dt = e->dt;
            r.acc = d.acc;
            r.cmp = d.cmp;
            regs.push_back(r);
            tot += d.ncell * d.ncomp;  // one thread per (component, cell) of each frequency
        }
    }
    s->ndft = (int)regs.size();
    s->dft_total = tot;
    // sources and DFT can share a launch when no DFT region of an engine holds one of its
    // source cells
    s->src_dft_one_launch = !s->src_at.empty() && s->ndft > 0;
    for (sjf_engine* e : s->eng) {
        const long nyz = (long)e->g.ny * e->g.nz;
        for (const Source& src : e->src)
            for (const long q : (src.comp < 3 ? src.idx : std::vector<long>())) {
                const int i = (int)(q / nyz), j = (int)((q % nyz) / e->g.nz), k = (int)(q % e->g.nz);
                for (const Dft& d : e->dft)
                    if (i >= d.lo[0] && i < d.hi[0] && j >= d.lo[1] && j < d.hi[1] && k >= d.lo[2] && k < d.hi[2])
                        s->src_dft_one_launch = false;
            }
    }
    s->dft_maxnf = 0;
    for (const auto& r : regs) s->dft_maxnf = std::max(s->dft_maxnf, r.nf);
    // a grid dimension holds less than 2^32 threads
    constexpr long most = (1L << 24) - 1;  // workgroups of 256 threads
    const long per_freq = (tot + 255) / 256;
    if (per_freq > most) return fail(e0, SJF_E_UNSUPPORTED, "DFT regions exceed 2^32 values per frequency");
    s->dft_blocks = (int)per_freq;
    if (s->src_dft_one_launch && s->src_at.back() + per_freq * s->dft_maxnf > most) s->src_dft_one_launch = false;
    if (s->ndft) {
        rc = upload_vec(e0, s->stream, &s->d_dft, regs);
        if (rc) return rc;
    }

    std::vector<long*> ctr;
    for (sjf_engine* e : s->eng) ctr.push_back(e->d_step);
    rc = upload_vec(e0, s->stream, (void**)&s->d_counters, ctr);
    if (rc) return rc;

    s->versions.clear();
    for (sjf_engine* e : s->eng) s->versions.push_back(e->version);
    s->built = true;
    return SJF_OK;
}

int build_set(LaunchSet* s) { return s->prec == 4 ? build_set_t<float>(s) : build_set_t<double>(s); }

bool set_stale(const LaunchSet* s) {
    if (!s->built) return true;
    for (size_t i = 0; i < s->eng.size(); ++i)
        if (s->eng[i]->version != s->versions[i]) return true;
    return false;
}

#define SETCHK(s, call)                                                                  \
    do {                                                                                 \
        hipError_t _st = (call);                                                         \
        if (_st != hipSuccess) {                                                         \
            (s)->eng[0]->err = std::string(#call) + ": " + hipGetErrorString(_st);       \
            return SJF_E_HIP;                                                            \
        }                                                                                \
    } while (0)

// The fused step of a launch set, by its form and workgroup size.  Kernels whose registers leave room
// for a 1024-thread workgroup (128 per lane: the FP32 one-row tile) are compiled for it alone.
template <typename T, int NP>
int launch_step_np(LaunchSet* s) {
    const dim3 grid(s->ntiles), block(s->block);
    const auto* args = (const sjf::StepArgs<T>*)s->d_args;
    const int n = (int)s->eng.size();
#define SJF_LAUNCH(...) hipLaunchKernelGGL((__VA_ARGS__), grid, block, s->lds, s->stream, args, s->d_tile_first, n)
    if (s->form == SJF_TILE_THREAD_ROWS) {
        if (s->block <= 512) {
            if (s->nts) SJF_LAUNCH(sjf::k_step_rows<T, NP, 512, true>);
            else SJF_LAUNCH(sjf::k_step_rows<T, NP, 512>);
        } else if (s->nts) {
            SJF_LAUNCH(sjf::k_step_rows<T, NP, 1024, true>);
        } else {
            SJF_LAUNCH(sjf::k_step_rows<T, NP, 1024>);
        }
    } else if (s->zpass) {
        if (s->block > 256) SJF_LAUNCH(sjf::k_step_z<T, NP, 1024>);
        else if (s->nts) SJF_LAUNCH(sjf::k_step_z<T, NP, 256, true>);
        else SJF_LAUNCH(sjf::k_step_z<T, NP, 256>);
    } else if (s->ty == 1) {
        constexpr int M = sizeof(T) == 4 ? 1024 : 512;
        if (s->block > M) SJF_LAUNCH(sjf::k_step<T, 1, NP, 1024>);
        else if (s->nts) SJF_LAUNCH(sjf::k_step<T, 1, NP, M, true>);
        else SJF_LAUNCH(sjf::k_step<T, 1, NP, M>);
    } else if (s->ty == 2) {
        constexpr int M = sizeof(T) == 4 ? 512 : 256;  // FP64: 512 registers per lane up to 256 threads, none spilled
        if (s->block <= M) SJF_LAUNCH(sjf::k_step<T, 2, NP, M>);
        else if (s->block <= 512) SJF_LAUNCH(sjf::k_step<T, 2, NP, 512>);
        else SJF_LAUNCH(sjf::k_step<T, 2, NP, 1024>);
    } else if (s->ty == 4) {
        constexpr int M = sizeof(T) == 4 ? 512 : 256;
        if (s->block <= M) SJF_LAUNCH(sjf::k_step<T, 4, NP, M>);
        else if (s->block <= 512) SJF_LAUNCH(sjf::k_step<T, 4, NP, 512>);
        else SJF_LAUNCH(sjf::k_step<T, 4, NP, 1024>);
    } else {
        return fail(s->eng[0], SJF_E_ARG, "tile rows must be 1, 2 or 4");
    }
#undef SJF_LAUNCH
    SETCHK(s, hipGetLastError());
    return SJF_OK;
}

template <typename T>
int launch_step_t(LaunchSet* s) {
    switch (s->npv) {
        case 0: return launch_step_np<T, 0>(s);
        case 1: return launch_step_np<T, 1>(s);
        case 3: return launch_step_np<T, 3>(s);
        default: return launch_step_np<T, 4>(s);
    }
}

// One time step of every engine in the set.  `sample` launches the monitor gather first.
template <typename T>
int launch_one_step_t(LaunchSet* s, bool sample, hipEvent_t ev_a, hipEvent_t ev_b, bool bare = false) {
    if (sample && s->nmon && !bare) {
        hipLaunchKernelGGL((sjf::k_monitor<T>), dim3((s->nmon + 255) / 256), dim3(256), 0, s->stream,
                           (const sjf::MonDev<T>*)s->d_mon, s->nmon);
        SETCHK(s, hipGetLastError());
    }
    for (size_t l = 0; l + 1 < s->hsrc_at.size(); ++l) {
        const int first = s->hsrc_at[l], blocks = s->hsrc_at[l + 1] - first;
        const sjf::SrcTables<T> ht{(const sjf::SrcDev<T>*)s->d_hsrc, s->d_hblk_src + first, s->d_hblk_first + first,
                                   s->d_hblk_end + first, s->d_hsrc_idx, s->d_hsrc_coef};
        hipLaunchKernelGGL((sjf::k_source_h<T>), dim3(blocks), dim3(256), 0, s->stream, ht);
        SETCHK(s, hipGetLastError());
    }
    if (ev_a) SETCHK(s, hipEventRecord(ev_a, s->stream));
    int rc = launch_step_t<T>(s);
    if (rc) return rc;
    if (ev_b) SETCHK(s, hipEventRecord(ev_b, s->stream));
    // the last kernel of the step advances the step counters: the DFT kernel when there is
    // one, else the source kernel, else k_tick
    const int n = (int)s->eng.size();
    const bool dft = s->ndft && !bare;
    const sjf::Tick tick{s->d_counters, n}, none{s->d_counters, 0};
    const size_t nlayer = s->src_at.empty() ? 0 : s->src_at.size() - 1;
    for (size_t l = 0; l < nlayer; ++l) {
        const int first = s->src_at[l], blocks = s->src_at[l + 1] - first;
        const bool last = l + 1 == nlayer;
        const sjf::SrcTables<T> st{(const sjf::SrcDev<T>*)s->d_src, s->d_blk_src + first, s->d_blk_first + first,
                                   s->d_blk_end + first, s->d_src_idx, s->d_src_coef};
        if (last && dft && s->src_dft_one_launch) {
            hipLaunchKernelGGL((sjf::k_source_dft<T>), dim3((unsigned)(blocks + s->dft_blocks * s->dft_maxnf)), dim3(256), 0,
                               s->stream, st, blocks, (const sjf::DftDev<T>*)s->d_dft, s->ndft, s->dft_total,
                               s->dft_blocks, tick);
            SETCHK(s, hipGetLastError());
            return SJF_OK;
        }
        hipLaunchKernelGGL((sjf::k_source<T>), dim3(blocks), dim3(256), 0, s->stream, st, last && !dft ? tick : none);
        SETCHK(s, hipGetLastError());
    }
    if (dft) {
        hipLaunchKernelGGL((sjf::k_dft<T>), dim3((unsigned)s->dft_blocks, (unsigned)s->dft_maxnf), dim3(256), 0, s->stream,
                           (const sjf::DftDev<T>*)s->d_dft, s->ndft, s->dft_total, tick);
        SETCHK(s, hipGetLastError());
    } else if (nlayer == 0) {
        hipLaunchKernelGGL(sjf::k_tick, dim3((n + 63) / 64), dim3(64), 0, s->stream, s->d_counters, n);
        SETCHK(s, hipGetLastError());
    }
    return SJF_OK;
}

int launch_one_step(LaunchSet* s, bool sample, hipEvent_t a = nullptr, hipEvent_t b = nullptr) {
    return s->prec == 4 ? launch_one_step_t<float>(s, sample, a, b) : launch_one_step_t<double>(s, sample, a, b);
}

// step kernel + sources + counter only (forward recomputation inside the adjoint)
int launch_bare_step(LaunchSet* s) {
    return s->prec == 4 ? launch_one_step_t<float>(s, false, nullptr, nullptr, true)
                        : launch_one_step_t<double>(s, false, nullptr, nullptr, true);
}

bool samples_at(const LaunchSet* s, long step) {
    for (const sjf_engine* e : s->eng)
        if (!e->mon.empty() && step % e->save_span == 0) return true;
    return false;
}

int sync_engine(sjf_engine* e);

int ensure_sample_capacity(sjf_engine* e, long need) {
    const int npt = (int)e->mon.size();
    if (npt == 0 || need <= e->samp_cap) return SJF_OK;
    // the old samples may still be in flight on a batch stream
    if (int rc = sync_engine(e)) return rc;
    const long cap = std::max(need, 2 * e->samp_cap);
    double* p = nullptr;
    if (device_malloc((void**)&p, sizeof(double) * cap * npt) != hipSuccess)
        return fail(e, SJF_E_NOMEM, "sample buffer allocation failed");
    if (e->d_samples && e->nsamp > 0)
        HIPCHK(e, hipMemcpyAsync(p, e->d_samples, sizeof(double) * e->nsamp * npt, hipMemcpyDeviceToDevice,
                                 e->stream));
    HIPCHK(e, hipStreamSynchronize(e->stream));
    dev_free(e->d_samples);
    e->d_samples = p;
    e->samp_cap = cap;
    e->version++;
    return SJF_OK;
}

long samples_in(long a, long b, int span) {
    // multiples of span in [a, b)
    if (b <= a) return 0;
    const long first = (a + span - 1) / span, last = (b - 1) / span;
    return std::max(0L, last - first + 1);
}

int prepare_set(LaunchSet* s, long n) {
    for (sjf_engine* e : s->eng) {
        if (e->mon.empty()) continue;
        const long need = (e->step + n + e->save_span - 1) / e->save_span;
        int rc = ensure_sample_capacity(e, need);
        if (rc) return rc;
    }
    if (set_stale(s)) return build_set(s);
    return SJF_OK;
}

void advance_hosts(LaunchSet* s, long n) {
    for (sjf_engine* e : s->eng) {
        if (!e->mon.empty()) e->nsamp += samples_in(e->step, e->step + n, e->save_span);
        e->step += n;
    }
}

long set_span(const LaunchSet* s) {
    long span = 1;
    for (const sjf_engine* e : s->eng)
        if (!e->mon.empty()) span = e->save_span;
    return span;
}

// Steps per captured graph: a multiple of the save span so every replay starts aligned.
long graph_chunk(const LaunchSet* s) {
    const sjf_engine* e0 = s->eng[0];
    if (e0->graph_chunk <= 0) return 0;
    const long span = set_span(s);
    return std::max(1L, (e0->graph_chunk + span - 1) / span) * span;
}

int capture_graph(LaunchSet* s, long K) {
    if (s->gexec) (void)hipGraphExecDestroy(s->gexec);
    if (s->graph) (void)hipGraphDestroy(s->graph);
    s->gexec = nullptr;
    s->graph = nullptr;
    const long s0 = s->eng[0]->step;
    SETCHK(s, hipStreamBeginCapture(s->stream, hipStreamCaptureModeThreadLocal));
    int rc = SJF_OK;
    for (long q = 0; q < K && !rc; ++q) rc = launch_one_step(s, samples_at(s, s0 + q));
    hipGraph_t g = nullptr;
    const hipError_t st = hipStreamEndCapture(s->stream, &g);
    if (rc) {
        if (g) (void)hipGraphDestroy(g);
        return rc;
    }
    SETCHK(s, st);
    s->graph = g;
    SETCHK(s, hipGraphInstantiate(&s->gexec, g, nullptr, nullptr, 0));
    s->gK = K;
    return SJF_OK;
}

int run_set(LaunchSet* s, long n) {
    int rc = prepare_set(s, n);
    if (rc) return rc;
    const long K = graph_chunk(s);
    const long span = set_span(s);
    long done = 0;
    auto eager = [&](long m) -> int {
        for (long q = 0; q < m; ++q) {
            const int r = launch_one_step(s, samples_at(s, s->eng[0]->step));
            if (r) return r;
            advance_hosts(s, 1);
        }
        return SJF_OK;
    };
    const long lead = K > 0 ? (span - s->eng[0]->step % span) % span : 0;
    if (K > 0 && n - lead >= K) {
        // align the first replay to the save span, then replay whole chunks
        rc = eager(lead);
        if (rc) return rc;
        done += lead;
        if (!s->gexec || s->gK != K) {
            rc = capture_graph(s, K);
            if (rc) return rc;
        }
        while (n - done >= K) {
            SETCHK(s, hipGraphLaunch(s->gexec, s->stream));
            advance_hosts(s, K);
            done += K;
        }
    }
    return eager(n - done);
}

LaunchSet* own_set(sjf_engine* e) {
    if (!e->own) {
        e->own = new LaunchSet();
        e->own->eng.push_back(e);
        e->own->stream = e->stream;
        e->own->prec = e->prec;
    }
    if (e->own->ty != e->ty || e->own->form != e->form) {
        e->own->ty = e->ty;
        e->own->form = e->form;
        e->own->built = false;
    }
    return e->own;
}

void destroy_set(LaunchSet* s) {
    if (!s) return;
    set_free_tables(s);
    if (s->own_stream && s->stream) (void)hipStreamDestroy(s->stream);
    delete s;
}

int timed_set(LaunchSet* s, long n, double* ms_total, double* ms_kernel_mean) {
    int rc = prepare_set(s, n);
    if (rc) return rc;
    std::vector<hipEvent_t> evs(2 * n);
    for (auto& ev : evs) SETCHK(s, hipEventCreate(&ev));
    hipEvent_t t0, t1;
    SETCHK(s, hipEventCreate(&t0));
    SETCHK(s, hipEventCreate(&t1));
    SETCHK(s, hipStreamSynchronize(s->stream));
    SETCHK(s, hipEventRecord(t0, s->stream));
    for (long q = 0; q < n; ++q) {
        rc = launch_one_step(s, samples_at(s, s->eng[0]->step), evs[2 * q], evs[2 * q + 1]);
        if (rc) return rc;
        advance_hosts(s, 1);
    }
    SETCHK(s, hipEventRecord(t1, s->stream));
    SETCHK(s, hipEventSynchronize(t1));
    float tot = 0;
    SETCHK(s, hipEventElapsedTime(&tot, t0, t1));
    double ksum = 0;
    for (long q = 0; q < n; ++q) {
        float ms = 0;
        SETCHK(s, hipEventElapsedTime(&ms, evs[2 * q], evs[2 * q + 1]));
        ksum += ms;
    }
    for (auto& ev : evs) (void)hipEventDestroy(ev);
    (void)hipEventDestroy(t0);
    (void)hipEventDestroy(t1);
    *ms_total = tot;
    *ms_kernel_mean = ksum / n;
    return SJF_OK;
}

// ======================================================================== engine helpers ==

// Waves per SIMD that the step kernel of an engine's tile runs (its registers; see the kernels).
template <typename T>
int tile_waves(const sjf_engine* e) {
    auto of = [&](auto np) {
        constexpr int NP = decltype(np)::value;
        if (e->form == SJF_TILE_THREAD_ROWS) return sjf::rows_waves<T, NP>();
        return zseg_of(e, 1, false) < e->g.nz ? sjf::step_waves<T, 1, NP, true>() : sjf::step_waves<T, 1, NP>();
    };
    switch (np_variant_of(e->maxp, e->uniform)) {
        case 0: return of(std::integral_constant<int, 0>{});
        case 1: return of(std::integral_constant<int, 1>{});
        case 3: return of(std::integral_constant<int, 3>{});
        default: return of(std::integral_constant<int, 4>{});
    }
}

// Default tile, after a change of the materials (their pole slots set the kernel's registers).
//
// Form: thread rows where a workgroup holds three owned rows or more, which share one halo row and
// leave few lanes idle on a z line of any length (FP32 below 256 cells, FP64 below 128).  Measured on
// MI355X, us per step of the best x-chunk, thread rows and one register row per workgroup: FP64 41^3
// 13.0, 15.3; 72x64x56 20.4, 21.0; 96^3 36.1, 42.0; 101^3 39.7, 54.0; 128^3 105.7, 105.3; FP32
// 192x192x96 80.4, 93.9; 151x133x117 54.4, 70.2; 256x256x128 191.7, 201.7; 150x150x200 90.0, 112.7;
// 120x160x250 95.9, 120.6; 512x512x256 1061, 1039.
void choose_tile(sjf_engine* e) {
    if (e->tile_set) return;
    const int rows = default_thread_rows(e), full = e->prec == 8 ? 128 : 256;
    const bool thread_rows = e->g.nz < full && zseg_of(e, 1, false) == e->g.nz && thread_rows_fit(e, rows);
    e->form = thread_rows ? SJF_TILE_THREAD_ROWS : SJF_TILE_REGISTER_ROWS;
    e->ty = thread_rows ? rows : 1;
    const int waves = e->prec == 4 ? tile_waves<float>(e) : tile_waves<double>(e);
    e->xc = resident_chunk(e->g.nx, (e->g.ny + e->ty - 1) / e->ty, block_threads(e) / 64, waves);
}

// Default form of a batch: thread rows where some instance would take them alone (choose_tile) and all
// fit.  Measured on MI355X, us per step, thread rows and one register row: 24 grids of 64^3 to
// 192x192x128 (FP32) 915, 1074; six of 192x192x96 467, 487; two 170, 191; FP32 lines of 100 and 500
// cells (1.5 M cells each) 95, 137; of 100 and three of 400 cells 224, 233; FP64 lines of 100 and 200
// cells 187, 216.  The chunk matters little with many rounds of workgroups (24 grids: 4 planes 919, 6
// 915, 8 918, 12 941, 18 955; four grids: 4 planes 139, 6 132, 8 132, 12 130, 18 159).
//
// FP64 workgroups of more than 512 threads spill and cost about 1.6 times as much a thread: there
// thread rows are taken where they leave so many fewer lanes idle (or run half of the threads of a long
// line on its halo row) that this is made up for, or where all of them run at once.  FP64, 1.5 M cells
// each: lines of 60, 60, 60, 300 cells 688, 999; 64, 500 346, 464; 100, 100, 100, 500 730, 749; 100, 500
// 383, 311; 100, 300 393, 287; 120, 300, 400, 500 741, 463; 100, 300 of 0.3 M cells (245 workgroups) 83, 95.
constexpr int kBatchRowsChunk = 8;
int batch_form(sjf_engine* const* engines, int n) {
    bool any = false;
    int rows_block = 64, line_block = 64;
    long groups = 0;
    for (int i = 0; i < n; ++i) {
        const sjf_engine* e = engines[i];
        const int rows = default_thread_rows(e);
        if (!thread_rows_fit(e, rows)) return SJF_TILE_REGISTER_ROWS;
        any = any || e->g.nz < (e->prec == 8 ? 128 : 256);
        rows_block = std::max(rows_block, ((rows + 1) * e->g.nz + 63) / 64 * 64);
        line_block = std::max(line_block, (e->g.nz + 63) / 64 * 64);
        groups += tiles_of(e, rows, std::min(kBatchRowsChunk, e->g.nx));
    }
    if (!any) return SJF_TILE_REGISTER_ROWS;
    if (engines[0]->prec == 4 || rows_block <= 512 || groups <= 256) return SJF_TILE_THREAD_ROWS;
    double by_rows = 0, by_lines = 0;  // threads times planes
    for (int i = 0; i < n; ++i) {
        const sjf_engine* e = engines[i];
        by_rows += (double)e->N * rows_block / (default_thread_rows(e) * e->g.nz);
        by_lines += (double)e->N * line_block / e->g.nz;
    }
    return 1.6 * by_rows < by_lines ? SJF_TILE_THREAD_ROWS : SJF_TILE_REGISTER_ROWS;
}

int free_all(sjf_engine* e) {
    destroy_set(e->own);
    e->own = nullptr;
    for (int b = 0; b < 2; ++b) dev_free(e->Fbuf[b]);
    dev_free(e->d_step);
    dev_free(e->given);
    dev_free(e->matw);
    dev_free(e->seg);
    dev_free(e->lut);
    dev_free(e->dinv);
    dev_free(e->emap);
    dev_free(e->Qbuf);
    dev_free(e->Pbuf);
    dev_free(e->coefbuf);
    for (int d = 0; d < 3; ++d) dev_free(e->psibuf[d]);
    dev_free(e->d_samples);
    for (auto& d : e->dft) {
        dev_free(d.acc);
        dev_free(d.cmp);
        dev_free(d.d_freq);
    }
    return SJF_OK;
}

template <typename T>
int convert_to_device(sjf_engine* e, void* dst, const double* src, long n) {
    if (sizeof(T) == sizeof(double)) return h2d(e, dst, src, sizeof(double) * n);
    std::vector<T> tmp(n);
    for (long q = 0; q < n; ++q) tmp[q] = (T)src[q];
    return h2d(e, dst, tmp.data(), sizeof(T) * n);
}

// One component of the current field set to / from a dense z-fastest host array: the component
// is one plane of ny * nz values in each x plane of six, a pitched copy.
template <typename T>
int write_component(sjf_engine* e, int comp, const double* src) {
    const size_t plane = sizeof(T) * (size_t)e->g.ny * e->g.nz;
    std::vector<T> tmp(e->N);
    for (long q = 0; q < e->N; ++q) tmp[q] = (T)src[q];
    char* dst = (char*)field_set(e) + plane * comp;
    HIPCHK(e, hipMemcpy2DAsync(dst, 6 * plane, tmp.data(), plane, plane, e->g.nx, hipMemcpyHostToDevice, e->stream));
    HIPCHK(e, hipStreamSynchronize(e->stream));
    return SJF_OK;
}

// n values of `size` bytes into dst: launch(first, count, p) has the device write values first ..
// first + count - 1 to p.  More than one chunk: the device fills one half of the stage while the other
// is copied out.
template <typename L>
int read_out(sjf_engine* e, void* dst, long n, size_t size, L launch) {
    const long per = std::min<long>(n, (long)(kReadChunk / size));
    const bool one = per >= n;
    StageLease stage(e, (one ? 1 : 2) * (size_t)per * size);
    if (!stage.get()) return SJF_E_NOMEM;
    char* half[2] = {(char*)stage.get(), (char*)stage.get() + (one ? 0 : (size_t)per * size)};
    long done = 0, have = 0;  // values copied out; values of the chunk the stage holds, not yet copied
    for (long first = 0, c = 0; first < n || have > 0; ++c) {
        const long count = std::min(per, n - first);
        if (count > 0) {
            launch(first, count, (void*)half[c & 1]);
            HIPCHK(e, hipGetLastError());
            first += count;
        }
        if (have > 0) std::memcpy((char*)dst + (size_t)done * size, half[(c & 1) ^ 1], (size_t)have * size);
        done += have;
        have = std::max(count, 0L);
        HIPCHK(e, hipStreamSynchronize(e->stream));
    }
    stage.done();
    return SJF_OK;
}

// The cell box [lo, hi) of one component of the current field set, z-fastest FP64.
template <typename T>
int read_component_box(sjf_engine* e, int comp, const int* lo, const int* hi, double* dst) {
    const long plane = (long)e->g.ny * e->g.nz;
    const int by = hi[1] - lo[1], bz = hi[2] - lo[2];
    const T* base = (const T*)field_set(e) + (6L * lo[0] + comp) * plane + (long)lo[1] * e->g.nz + lo[2];
    return read_out(e, dst, (long)(hi[0] - lo[0]) * by * bz, sizeof(double), [&](long first, long count, void* p) {
        hipLaunchKernelGGL((sjf::k_read_box<T>), dim3((unsigned)std::min(1024L, (count + 255) / 256)), dim3(256), 0,
                           e->stream, base, 6 * plane, e->g.nz, by, bz, first, count, (double*)p);
    });
}

template <typename T>
int read_component(sjf_engine* e, int comp, double* dst) {
    const int lo[3] = {0, 0, 0}, hi[3] = {e->g.nx, e->g.ny, e->g.nz};
    return read_component_box<T>(e, comp, lo, hi, dst);
}

template <typename T>
int upload_lut_t(sjf_engine* e) {
    std::vector<sjf::MatLut<T>> l(e->nmat + 1);  // the last: zeros, for design voxels
    std::memset((void*)l.data(), 0, sizeof(sjf::MatLut<T>) * l.size());
    const double dt = e->dt;
    for (int m = 0; m < e->nmat; ++m) {
        const sjf_material& M = e->lut_h[m];
        sjf::MatLut<T>& L = l[m];
        L.inv_eps = (T)(1.0 / M.eps_inf);
        L.np = M.npoles;
        for (int s = 0; s < M.npoles; ++s) {
            // coefficients formed in FP64 (sigma * w0^2 spans ~1e21 * 1e-22 for Au Drude)
            const double w0 = 2 * M_PI * M.f0[s];
            const double gm = 2 * M_PI * M.gamma[s];
            const double g = gm * dt / 2;
            const double Lf = M.is_drude[s] ? 0.0 : 1.0;
            L.pole[s].alpha = (T)((1 - g) / (1 + g));
            L.pole[s].beta = (T)(-Lf * w0 * w0 * dt * dt / (1 + g));
            L.pole[s].c3 = (T)(M.sigma[s] * (w0 * w0) * dt * dt / (1 + g));
            L.pole[s].lor = (T)Lf;
            if (!M.is_drude[s]) L.lorentz_mask |= 1 << s;
        }
    }
    dev_free(e->lut);
    int rc = dev_alloc(e, &e->lut, sizeof(sjf::MatLut<T>) * l.size());
    if (rc) return rc;
    return h2d(e, e->lut, l.data(), sizeof(sjf::MatLut<T>) * l.size());
}

int upload_lut(sjf_engine* e) { return e->prec == 4 ? upload_lut_t<float>(e) : upload_lut_t<double>(e); }

// The words and segment codes the kernels run (k_words; after a change of the given words, the twins
// or the LUT), and what the step moves of pole state: bytes of whole segments, and poles.
int update_words(sjf_engine* e) {
    const long n = (long)e->g.nx * e->g.ny * ((e->g.nz + 63) / 64);
    int rc = dev_alloc(e, (void**)&e->matw, sizeof(uint32_t) * e->N);
    if (!rc) rc = dev_alloc(e, (void**)&e->seg, sizeof(uint32_t) * (n + 5));
    if (rc) return rc;
    auto* sums = (unsigned long long*)(e->seg + n + (n & 1));
    unsigned long long count[2] = {0, 0};
    HIPCHK(e, hipMemcpyAsync(sums, count, sizeof(count), hipMemcpyHostToDevice, e->stream));
    sjf::WordMap map;
    const int dim[3] = {e->g.nx, e->g.ny, e->g.nz};
    for (int d = 0; d < 3; ++d) {
        map.lo[d] = e->pml_on[d] ? e->pml[2 * d] : 0;
        map.hi[d] = dim[d] - (e->pml_on[d] ? e->pml[2 * d + 1] : 0);
    }
    for (int m = 0; m < 256; ++m)
        map.twin[m] = (unsigned char)(m < (int)e->twin.size() && e->twin[m] >= 0 ? e->twin[m] : m);
    const dim3 grid((unsigned)std::min(512L, (n + 3) / 4)), block(256);
    if (e->prec == 4)
        hipLaunchKernelGGL((sjf::k_words<float>), grid, block, 0, e->stream, e->given, e->matw, e->seg,
                           (const sjf::MatLut<float>*)e->lut, dim[0], dim[1], dim[2], e->nmat, map, sums);
    else
        hipLaunchKernelGGL((sjf::k_words<double>), grid, block, 0, e->stream, e->given, e->matw, e->seg,
                           (const sjf::MatLut<double>*)e->lut, dim[0], dim[1], dim[2], e->nmat, map, sums);
    HIPCHK(e, hipGetLastError());
    HIPCHK(e, hipMemcpyAsync(count, sums, sizeof(count), hipMemcpyDeviceToHost, e->stream));
    HIPCHK(e, hipStreamSynchronize(e->stream));
    e->pole_bytes = 64.0 * 3 * (e->Pbuf ? 2 : 1) * e->prec * (double)count[0];
    e->pole_values = (double)count[1];
    return SJF_OK;
}

// 1/eps_inf of the effective map on the device in the plane layout [x][Ex Ey Ez][y][z]
template <typename T>
int upload_emap_t(sjf_engine* e) {
    const long nyz = (long)e->g.ny * e->g.nz;
    std::vector<T> h((size_t)3 * e->N);
    for (int i = 0; i < e->g.nx; ++i)
        for (int c = 0; c < 3; ++c)
            for (long r = 0; r < nyz; ++r)
                h[((size_t)i * 3 + c) * nyz + r] = (T)(1.0 / e->emap_eff[(size_t)c * e->N + (long)i * nyz + r]);
    int rc = dev_alloc(e, &e->emap, sizeof(T) * 3 * e->N);
    if (rc) return rc;
    return h2d(e, e->emap, h.data(), sizeof(T) * 3 * e->N);
}

int upload_emap(sjf_engine* e) { return e->prec == 4 ? upload_emap_t<float>(e) : upload_emap_t<double>(e); }

// Real part of a Lorentz pole's susceptibility at meep frequency f:
// sigma w0^2 (w0^2 - w^2) / ((w0^2 - w^2)^2 + w^2 gamma'^2), w = 2 pi f, w0 = 2 pi f0, gamma' = 2 pi gamma.
double lorentz_re_chi(const sjf_material& M, int s, double f) {
    const double w = 2 * M_PI * f, w0 = 2 * M_PI * M.f0[s], g = 2 * M_PI * M.gamma[s];
    const double d = w0 * w0 - w * w;
    return M.sigma[s] * w0 * w0 * d / (d * d + w * w * g * g);
}

bool cell_in_pml(const sjf_engine* e, long q) {
    const int n[3] = {e->g.nx, e->g.ny, e->g.nz};
    const long nyz = (long)n[1] * n[2];
    const int ijk[3] = {(int)(q / nyz), (int)((q % nyz) / n[2]), (int)(q % n[2])};
    for (int d = 0; d < 3; ++d)
        if (e->pml_on[d] && (ijk[d] < e->pml[2 * d] || ijk[d] >= n[d] - e->pml[2 * d + 1])) return true;
    return false;
}

// What the kernels run for a LUT: with pml_fref > 0 every cell inside a PML slab whose material has
// Lorentz poles takes a twin of that material with them folded out (their real susceptibility at
// pml_fref added to eps_inf when the sum stays >= 1, else eps_inf kept; Drude poles kept).
struct MatPlan {
    std::vector<sjf_material> lut;  // the given materials and the twins
    std::vector<int> twin;          // per given material its twin, or -1
    std::vector<double> fold_add;   // sum of the folded Lorentz poles' Re chi
};

// The plan for `given`; refuses without changing the engine.
int plan_materials(sjf_engine* e, const std::vector<sjf_material>& given, double fref, bool any_pml, MatPlan* p) {
    const int ng = (int)given.size();
    p->lut = given;
    p->twin.assign(ng, -1);
    p->fold_add.assign(ng, 0.0);
    if (!(fref > 0 && any_pml)) return SJF_OK;
    for (int m = 0; m < ng; ++m) {
        const sjf_material& M = given[m];
        sjf_material T = M;
        T.npoles = 0;
        double eps = M.eps_inf;
        bool has_lor = false;
        for (int s = 0; s < M.npoles; ++s) {
            if (M.is_drude[s]) {
                const int t = T.npoles++;
                T.f0[t] = M.f0[s];
                T.gamma[t] = M.gamma[s];
                T.sigma[t] = M.sigma[s];
                T.is_drude[t] = 1;
            } else {
                has_lor = true;
                eps += lorentz_re_chi(M, s, fref);
            }
        }
        if (!has_lor) continue;
        p->fold_add[m] = eps - M.eps_inf;
        T.eps_inf = eps >= 1.0 ? eps : M.eps_inf;
        for (int s = T.npoles; s < SJF_MAX_POLES; ++s) T.f0[s] = T.gamma[s] = T.sigma[s] = 0, T.is_drude[s] = 0;
        if ((int)p->lut.size() >= SJF_MAX_MATERIALS)
            return fail(e, SJF_E_UNSUPPORTED, "materials and their PML twins exceed 255");
        p->twin[m] = (int)p->lut.size();
        p->lut.push_back(T);
    }
    return SJF_OK;
}

bool any_pml(const sjf_engine* e) { return e->pml_on[0] || e->pml_on[1] || e->pml_on[2]; }

int plan_materials(sjf_engine* e, MatPlan* p) { return plan_materials(e, e->given_lut, e->pml_fref, any_pml(e), p); }

// A call that changes what the kernels read begins: launch tables built before are void, and steps are
// refused until `ready` is set again.  A call that fails half-way so leaves an engine that says so
// instead of one that reads freed memory.
void begin_change(sjf_engine* e, bool& ready) {
    ready = false;
    e->version++;
}

// The default medium as given words and LUT, where a map or a design box comes before any materials.
int default_words(sjf_engine* e) {
    if (e->have_mat) return SJF_OK;
    if (int rc = dev_alloc(e, (void**)&e->given, sizeof(uint32_t) * e->N)) return rc;
    e->given_lut = e->lut_h;
    e->have_mat = true;
    return SJF_OK;
}

// The material map of the plan: uploads the words, the LUT and the eps maps and resets the
// polarisation state.
int apply_materials(sjf_engine* e, const MatPlan& plan) {
    begin_change(e, e->mat_ready);
    const int ng = (int)e->given_lut.size();
    const std::vector<int>& twin = plan.twin;
    const bool fold = plan.lut.size() > (size_t)ng;
    e->lut_h = plan.lut;
    e->twin = twin;
    // per-cell eps_inf map: the given values, with the same fold inside the PML slabs
    if (!e->emap_h.empty()) {
        e->emap_eff = e->emap_h;
        if (fold) {
            std::vector<uint32_t> given(e->N);
            if (int rc = d2h(e, given.data(), e->given, sizeof(uint32_t) * e->N)) return rc;
            for (long q = 0; q < e->N; ++q) {
                if (!cell_in_pml(e, q)) continue;
                for (int c = 0; c < 3; ++c) {
                    const int m = (given[q] >> (8 * c)) & 0xff;
                    if (m >= ng || twin[m] < 0) continue;
                    double& v = e->emap_eff[(size_t)c * e->N + q];
                    if (v + plan.fold_add[m] >= 1.0) v += plan.fold_add[m];
                }
            }
        }
        if (int rc = upload_emap(e)) return rc;
    }
    int maxp = 0;
    bool anylor = false;
    for (const sjf_material& M : e->lut_h) {
        maxp = std::max(maxp, M.npoles);
        for (int s = 0; s < M.npoles; ++s)
            if (!M.is_drude[s]) anylor = true;
    }
    e->nmat = (int)e->lut_h.size();
    e->maxp = maxp;
    e->uniform = (e->nmat == 1 && maxp == 0 && e->deps_h.empty() && e->emap_h.empty());
    // polarisation state, zeroed (the second array where a slot holds a Lorentz pole)
    const size_t pol = maxp > 0 ? (size_t)e->prec * 3 * maxp * e->N : 0;
    const bool pair = pol > 0 && anylor;
    if (pol != e->pol_bytes) dev_free(e->Qbuf), dev_free(e->Pbuf);
    if (!pair) dev_free(e->Pbuf);
    e->pol_bytes = pol;
    for (void** b : {&e->Qbuf, &e->Pbuf}) {
        if (pol == 0 || (b == &e->Pbuf && !pair)) continue;
        if (*b) HIPCHK(e, hipMemsetAsync(*b, 0, pol, e->stream));
        else if (int rc = dev_alloc(e, b, pol)) return rc;
    }
    int rc = upload_lut(e);
    if (!rc) rc = update_words(e);
    if (rc) return rc;
    choose_tile(e);
    e->mat_ready = true;
    return SJF_OK;
}

void trilinear(const sjf_engine* e, int comp, const double* xyz, long* idx, double* w) {
    int i0[3];
    double f[3];
    const int n[3] = {e->g.nx, e->g.ny, e->g.nz};
    for (int d = 0; d < 3; ++d) {
        const double s = xyz[d] / e->g.dx - kCompOff[comp][d];
        const double fl = std::floor(s);
        i0[d] = (int)fl;
        f[d] = s - fl;
    }
    int q = 0;
    for (int a = 0; a < 2; ++a)
        for (int b = 0; b < 2; ++b)
            for (int c = 0; c < 2; ++c, ++q) {
                int ii[3] = {i0[0] + a, i0[1] + b, i0[2] + c};
                const double ww = (a ? f[0] : 1 - f[0]) * (b ? f[1] : 1 - f[1]) * (c ? f[2] : 1 - f[2]);
                bool ok = true;
                for (int d = 0; d < 3; ++d) {
                    if (e->g.periodic[d]) ii[d] = ((ii[d] % n[d]) + n[d]) % n[d];
                    else if (ii[d] < 0 || ii[d] >= n[d]) ok = false;
                }
                idx[q] = ok ? cell_index(e, ii[0], ii[1], ii[2]) : -1;
                w[q] = ok ? ww : 0.0;
            }
}



double engine_step_bytes(const sjf_engine* e) {
    const double p = e->prec;
    double b = e->N * (12 * p + (e->uniform ? 0 : 4));
    // polarisation: per pole and dispersive component 3p, the compulsory state of the textbook
    // recurrence (read P^n and P^{n-1}, write P^{n+1})
    if (e->have_mat && e->maxp > 0) b += 3 * p * e->pole_values;
    if (!e->deps_h.empty()) b += p * (double)e->deps_h.size();
    if (!e->emap_h.empty()) b += 3 * p * (double)e->N;  // per-cell 1/eps_inf of the three E components
    // PML: per cell and PML axis, 2 E + 2 H auxiliaries, each read + written
    const int n[3] = {e->g.nx, e->g.ny, e->g.nz};
    for (int d = 0; d < 3; ++d)
        if (e->pml_on[d]) b += 8 * p * (double)(e->pml[2 * d] + e->pml[2 * d + 1]) * (e->N / n[d]);
    return b;
}

}  // namespace


// ======================================================================== adjoint =========

namespace {

// Everything that evolves with the time step (the current field set, polarisation state and all
// PML auxiliaries), in bytes.
struct StateLayout {
    size_t fields = 0, q = 0, p = 0, psi[3] = {0, 0, 0}, total = 0;
};

StateLayout state_layout(const sjf_engine* e) {
    StateLayout L;
    L.fields = (size_t)e->prec * 6 * e->N;
    L.q = e->Qbuf ? (size_t)e->prec * 3 * e->maxp * e->N : 0;
    L.p = e->Pbuf ? (size_t)e->prec * 3 * e->maxp * e->N : 0;
    L.total = L.fields + L.q + L.p;
    for (int d = 0; d < 3; ++d) {
        L.psi[d] = e->psibuf[d] ? (size_t)e->prec * 6 * e->slab[d] : 0;
        L.total += L.psi[d];
    }
    return L;
}

// (on the engine's stream, or on `st` when given: a batch's stream)
int copy_state(sjf_engine* e, char* ck, const StateLayout& L, bool save, hipStream_t st = nullptr) {
    if (!st) st = e->stream;
    auto cp = [&](void* dev, size_t off, size_t bytes) -> hipError_t {
        if (!bytes) return hipSuccess;
        return save ? hipMemcpyAsync(ck + off, dev, bytes, hipMemcpyDeviceToDevice, st)
                    : hipMemcpyAsync(dev, ck + off, bytes, hipMemcpyDeviceToDevice, st);
    };
    size_t off = 0;
    HIPCHK(e, cp(e->Fbuf[e->step & 1], off, L.fields));
    off += L.fields;
    HIPCHK(e, cp(e->Qbuf, off, L.q));
    off += L.q;
    HIPCHK(e, cp(e->Pbuf, off, L.p));
    off += L.p;
    for (int d = 0; d < 3; ++d) {
        HIPCHK(e, cp(e->psibuf[d], off, L.psi[d]));
        off += L.psi[d];
    }
    return SJF_OK;
}

int set_step(sjf_engine* e, long n) {
    e->step = n;
    HIPCHK(e, hipMemcpyAsync(e->d_step, &e->step, sizeof(long), hipMemcpyHostToDevice, e->stream));
    HIPCHK(e, hipStreamSynchronize(e->stream));
    return SJF_OK;
}

// x-chunk of the fused reverse step (one y row per workgroup) unless sjf_set_adjoint_tile sets
// one: enough chunks for about `target` workgroups over `rows` y rows (the engine's own, or those
// of every engine of a batch), independent of the forward tile.  Measured on MI355X: alone,
// 256x256x128 runs 1.019 ms per gradient step at 4 planes (16384 workgroups), 1.041 at 8 and
// 1.13 at 16; sixteen 192x192x96 engines in one batch run the reverse launch in 1.96 ms at 3
// planes (196608 workgroups), 1.82 ms at 6 and 1.79 ms at 12 on one box, and in 1.61 ms at 18
// planes (33792 workgroups) against 1.64-1.68 ms at 12 and 1.69-1.71 ms at 32 on another.
int adj_xchunk(const sjf_engine* e, long target = 16384, long rows = 0) {
    if (rows <= 0) rows = e->g.ny;
    long nxc = std::max(1L, (target + rows - 1) / rows);
    nxc = std::min<long>(nxc, e->g.nx);
    return std::max(1, (int)((e->g.nx + nxc - 1) / nxc));
}

// workgroups the reverse launch of a batch aims at (x-chunks common to all engines)
constexpr long kBatchAdjGroups = 32768;

// Tile of the reverse step: the one sjf_set_adjoint_tile gave; else thread rows wherever one owned
// row and the halo row fit a workgroup (FP64 512 threads), on grids, or batches, of at least
// kAdjRowsBytes of fields; else one row per workgroup.  Both forms give the same bits.  Measured on
// MI355X, us per reverse step, thread rows and one row: FP32 192x192x96 93, 138; 141x129x95 46, 73;
// 256x256x128 226, 232; 120x120x256 80, 145; 120x100x320 91, 200; 100x100x500 150, 232; FP64
// 72x64x56 22, 33; 100x100x128 80, 107; 100x100x200 140, 223; 52^3 19.1, 23.5.  Below the line a
// launch fills no more than a part of the chip either way and one row per workgroup has the shorter
// chain: FP32 52^3 17.8, 16.7; 32^3 13.9, 13.9.
constexpr double kAdjRowsBytes = 12e6;
struct AdjTile {
    bool rows;
    int nrows, xc;  // nrows 0: each engine's default; xc 0: the default chunks
};
template <typename T>
AdjTile adj_tile_of(const sjf_engine* e, double bytes, int nmat) {
    if (e->adj_set)
        return {e->adj_form == SJF_TILE_THREAD_ROWS, e->adj_form == SJF_TILE_THREAD_ROWS ? e->adj_rows : 1,
                e->adj_xc > 0 ? std::min(e->adj_xc, e->g.nx) : 0};
    const size_t block = sizeof(T) == 8 ? 512 : 1024;
    const bool rows = bytes >= kAdjRowsBytes && (size_t)(default_thread_rows(e) + 1) * e->g.nz <= block &&
                      lds_fits<T>(8 * block + 2 * (size_t)e->g.nz, nmat);
    return {rows, rows ? 0 : 1, 0};
}

// Waves per SIMD of the row-of-threads reverse kernel (its registers)
template <typename T>
int adj_rows_waves(int npv) {
    return sizeof(T) == 4 ? 4 : npv == 0 ? 3 : 2;
}

// Default x-chunk of a batched reverse launch in rows of threads: 12 planes (six 192x192x96 FP32 engines, us
// per reverse launch: 4 planes 584, 6 549, 8 537, 12 526, 18 533, 24 540), or the shorter one for which
// the rounds of resident workgroups times chunk and start-up (round_chunk) are fewer, where the launch does
// not fill the chip twice.  Gold, us per launch at 12 planes, so, and one row per workgroup: FP32 four of
// 48^3 52, 22.5, 30.7; two of 64^3 57, 24, 29; two of 96^3 54, 44, 79; FP64 two of 64^3 55, 34, 38.
template <typename T>
int adj_batch_chunk(const LaunchSet* s) {
    int block = 64, npv = 0;
    for (const sjf_engine* e : s->eng) {
        block = std::max(block, ((default_thread_rows(e) + 1) * e->g.nz + 63) / 64 * 64);
        npv = std::max(npv, np_variant_of(e->maxp, e->uniform));
    }
    const long slots = 256L * std::max(1, 4 * adj_rows_waves<T>(npv) / (block / 64));
    auto groups = [&](int c) {
        long g = 0;
        for (const sjf_engine* e : s->eng) g += tiles_of(e, default_thread_rows(e), std::min(c, e->g.nx));
        return g;
    };
    int best = 12;
    if (groups(best) >= 2 * slots) return best;
    auto cost = [&](int c) { return (groups(c) + slots - 1) / slots * (c + 3); };
    for (int c = 11; c > 0; --c)
        if (cost(c) < cost(best)) best = c;
    return best;
}

template <typename T, int NP, bool NTS>
void launch_adj_one_row(sjf_engine* e, const sjf::AdjArgs<T>& g, int block, unsigned tiles, size_t lds) {
    if (block <= 256) hipLaunchKernelGGL((sjf::k_adj_step<T, NP, 256, NTS>), dim3(tiles), dim3(block), lds, e->stream, g);
    else if (block <= 512) hipLaunchKernelGGL((sjf::k_adj_step<T, NP, 512, NTS>), dim3(tiles), dim3(block), lds, e->stream, g);
    else hipLaunchKernelGGL((sjf::k_adj_step<T, NP, 1024, NTS>), dim3(tiles), dim3(block), lds, e->stream, g);
}

template <typename T, int NP>
void launch_adj_np(sjf_engine* e, const sjf::AdjArgs<T>& g, int block, unsigned tiles, size_t lds) {
    // the reverse step streams the adjoint fields as the forward step streams E and H: the same line, alone
    // and in a batch (FP64 70x70x300, 141 MB of fields: 106 us without the hint, 117 with it)
    if (step_set_bytes(e) > kStreamBytes) launch_adj_one_row<T, NP, true>(e, g, block, tiles, lds);
    else launch_adj_one_row<T, NP, false>(e, g, block, tiles, lds);
}

template <typename T, int NP>
void launch_adj_rows_np(sjf_engine* e, const sjf::AdjArgs<T>& g, int block, unsigned tiles, size_t lds) {
    const bool nts = step_set_bytes(e) > kStreamBytes;  // (192x192x96 FP32: 96.8 us without, 93.0 with the hint)
#define SJF_LAUNCH(...) hipLaunchKernelGGL((__VA_ARGS__), dim3(tiles), dim3(block), lds, e->stream, g)
    if (block <= 512) {
        if (nts) SJF_LAUNCH(sjf::k_adj_rows<T, NP, 512, true>);
        else SJF_LAUNCH(sjf::k_adj_rows<T, NP, 512>);
    } else if (nts) {
        SJF_LAUNCH(sjf::k_adj_rows<T, NP, 1024, true>);
    } else {
        SJF_LAUNCH(sjf::k_adj_rows<T, NP, 1024>);
    }
#undef SJF_LAUNCH
}

template <typename T>
int launch_adj_step(sjf_engine* e, const sjf::AdjArgs<T>& g, int npv, int block, unsigned tiles, size_t lds,
                    bool rows) {
    switch (npv) {
        case 0: rows ? launch_adj_rows_np<T, 0>(e, g, block, tiles, lds) : launch_adj_np<T, 0>(e, g, block, tiles, lds); break;
        case 1: rows ? launch_adj_rows_np<T, 1>(e, g, block, tiles, lds) : launch_adj_np<T, 1>(e, g, block, tiles, lds); break;
        case 3: rows ? launch_adj_rows_np<T, 3>(e, g, block, tiles, lds) : launch_adj_np<T, 3>(e, g, block, tiles, lds); break;
        default: rows ? launch_adj_rows_np<T, 4>(e, g, block, tiles, lds) : launch_adj_np<T, 4>(e, g, block, tiles, lds); break;
    }
    HIPCHK(e, hipGetLastError());
    return SJF_OK;
}

// LDS of the reverse step: E-term and H-term exchange planes (row-of-threads form: twice) and the
// material table
template <typename T>
size_t adj_lds_bytes(bool rows, int block, int nmat) {
    return sizeof(T) * (rows ? 16 : 12) * (size_t)block + sjf::lut_lds_bytes<T>(nmat);
}

template <typename T>
int adjoint_run_t(sjf_engine* e, long nsteps, long K, long gap, double* J_out, double* grad, long nd) {
    LaunchSet* s = own_set(e);
    int rc = prepare_set(s, nsteps);
    if (rc) return rc;
    const StateLayout L = state_layout(e);
    const long slot = 3 * nd + 3;  // E of the design region and of the objective cell
    // Record mode (K == 0 and the record fits a quarter of the free device memory): the forward
    // pass records E of the design region and the objective cell after every step, so the
    // reverse pass needs no recomputation.  Otherwise the forward pass checkpoints the full state
    // every K steps (K == 0: about sqrt(nsteps)) and the reverse pass recomputes each segment.
    bool rec_all = false;
    if (K == 0) {
        size_t fr = 0, tot = 0;
        HIPCHK(e, hipMemGetInfo(&fr, &tot));
        rec_all = (double)sizeof(T) * slot * (nsteps + 1) <= 0.25 * (double)fr;
        if (!rec_all) K = std::max(1L, std::lround(std::sqrt((double)nsteps)));
    }
    K = std::min(K, nsteps);  // a longer interval holds one segment of nsteps all the same
    const long nck = rec_all ? 0 : (nsteps + K - 1) / K;
    const long nslots = rec_all ? nsteps + 1 : K + 1;
    char* cks = nullptr;
    if (!rec_all && device_malloc((void**)&cks, L.total * (nck + 1)) != hipSuccess)
        return fail(e, SJF_E_NOMEM, "checkpoint storage allocation failed (" +
                                        std::to_string((double)L.total * (nck + 1) / 1e9) + " GB)");
    double* dJ = nullptr;
    double* gacc = nullptr;
    T* ring = nullptr;
    T* A = nullptr;
    T* Aq = nullptr;
    T* Ap = nullptr;
    T* Apsi[3] = {nullptr, nullptr, nullptr};
    auto cleanup = [&]() {
        dev_free(cks);
        dev_free(dJ);
        dev_free(gacc);
        dev_free(ring);
        dev_free(A);
        dev_free(Aq);
        dev_free(Ap);
        for (int d = 0; d < 3; ++d) dev_free(Apsi[d]);
    };
    auto bail = [&](int r) {
        cleanup();
        return r;
    };
    // adjoint fields: two sets of six components (read / written per reverse step)
    if (dev_alloc(e, (void**)&dJ, sizeof(double)) || dev_alloc(e, (void**)&gacc, sizeof(double) * nd) ||
        dev_alloc(e, (void**)&ring, sizeof(T) * slot * nslots) || dev_alloc(e, (void**)&A, sizeof(T) * 12 * e->N) ||
        (L.q && dev_alloc(e, (void**)&Aq, L.q)) || (L.p && dev_alloc(e, (void**)&Ap, L.p)))
        return bail(SJF_E_NOMEM);
    // auxiliary bars: per axis 8 slots (E pair, two H pairs, second E pair)
    for (int d = 0; d < 3; ++d) {
        // the reverse step addresses the eight slots of a slab within one 2 GiB buffer range
        if ((double)L.psi[d] / 6 * 8 >= 2147483648.0)
            return bail(fail(e, SJF_E_UNSUPPORTED, "adjoint PML auxiliaries exceed 2 GiB on one axis"));
        if (L.psi[d] && dev_alloc(e, (void**)&Apsi[d], L.psi[d] / 6 * 8)) return bail(SJF_E_NOMEM);
    }

    const double dt = e->dt;
    const unsigned gdes = (unsigned)((nd + 3 + 255) / 256);
    const int de0 = e->dhi[0] - e->dlo[0], de1 = e->dhi[1] - e->dlo[1], de2 = e->dhi[2] - e->dlo[2];
    const long nyz = (long)e->g.ny * e->g.nz;
    auto record = [&](long sl, bool objective = false) -> int {
        const T* E = (const T*)e->Fbuf[e->step & 1];
        hipLaunchKernelGGL((sjf::k_adj_record<T>), dim3(gdes), dim3(256), 0, e->stream, E, nyz, e->g.ny, e->g.nz,
                           e->dlo[0], e->dlo[1], e->dlo[2], de0, de1, de2, gap, ring, sl, dt, objective ? dJ : nullptr);
        HIPCHK(e, hipGetLastError());
        return SJF_OK;
    };
    // ---- forward pass: the objective after every step; checkpoints every K steps or the record
    if (rec_all && (rc = record(0))) return bail(rc);
    for (long n = 0; n < nsteps; ++n) {
        if (!rec_all && n % K == 0) {
            if ((rc = copy_state(e, cks + L.total * (n / K), L, true))) return bail(rc);
        }
        if ((rc = launch_one_step(s, samples_at(s, e->step)))) return bail(rc);
        advance_hosts(s, 1);
        if (rec_all) {
            if ((rc = record(n + 1, true))) return bail(rc);
            continue;
        }
        const T* E = (const T*)e->Fbuf[e->step & 1];
        hipLaunchKernelGGL((sjf::k_adj_objective<T>), dim3(1), dim3(64), 0, e->stream, E, nyz, gap, dt, dJ);
        HIPCHK(e, hipGetLastError());
    }
    if (!rec_all && (rc = copy_state(e, cks + L.total * nck, L, true))) return bail(rc);
    HIPCHK(e, hipStreamSynchronize(e->stream));
    if ((rc = d2h(e, J_out, dJ, sizeof(double)))) return bail(rc);

    // ---- backward pass
    sjf::AdjArgs<T> g;
    std::memset(&g, 0, sizeof(g));
    // register form: one y row per workgroup; row-of-threads form: arows owned rows
    const AdjTile at = adj_tile_of<T>(e, field_bytes(e), e->nmat);
    const bool rows = at.rows;
    const int arows = at.nrows > 0 ? at.nrows : default_thread_rows(e);
    const int npv = np_variant_of(e->maxp, e->uniform);
    int axc = at.xc > 0 ? at.xc : adj_xchunk(e);
    if (rows && at.xc == 0 && at.nrows > 0) {  // about 16384 workgroups over the tile rows
        const long trows = (e->g.ny + arows - 1) / arows;
        const long nxc = std::min<long>(std::max(1L, (16384 + trows - 1) / trows), e->g.nx);
        axc = (int)((e->g.nx + nxc - 1) / nxc);
    } else if (rows && at.xc == 0) {
        const int wg = ((arows + 1) * e->g.nz + 63) / 64;
        axc = round_chunk(e->g.nx, (e->g.ny + arows - 1) / arows, 256L * std::max(1, 4 * adj_rows_waves<T>(npv) / wg), 3);
    }
    g.f = step_args<T>(e, arows, axc);
    g.A[0] = A;
    g.A[1] = A + (size_t)6 * e->N;
    g.rd = 0;
    g.Aq = Aq;
    g.Ap = Ap;
    for (int d = 0; d < 3; ++d) g.Apsi[d] = Apsi[d];
    const int block = (((rows ? arows + 1 : 1) * e->g.nz + 63) / 64) * 64;
    const unsigned tiles = (unsigned)((long)g.f.nty * ((e->g.nx + g.f.xc - 1) / g.f.xc));
    const size_t lds = adj_lds_bytes<T>(rows, block, e->nmat);
    if (!lds_fits<T>(rows ? 8 * (size_t)block + 2 * (size_t)e->g.nz : 12 * (size_t)block, e->nmat))
        return bail(fail(e, SJF_E_UNSUPPORTED, "adjoint tile needs more than 64 KiB of LDS"));
    auto ebar = [&]() { return g.A[g.rd]; };
    std::vector<uint32_t> gw;
    if ((rc = words_at(e, {gap}, gw))) return bail(rc);
    const double ie[3] = {inv_eps_at(e, gap, 0, gw[0]), inv_eps_at(e, gap, 1, gw[0]), inv_eps_at(e, gap, 2, gw[0])};
    auto inject = [&](long sl) -> int {
        hipLaunchKernelGGL((sjf::k_adj_inject<T>), dim3(1), dim3(64), 0, e->stream, ebar(), nyz, ring, nd, sl, gap, dt,
                           ie[0], ie[1], ie[2]);
        HIPCHK(e, hipGetLastError());
        return SJF_OK;
    };
    // HIP events around the fused reverse kernel of the first kTimed reverse steps (its mean
    // duration is reported by sjf_adjoint_kernel_info)
    constexpr int kTimed = 64;
    std::vector<hipEvent_t> evs;
    long ntimed = 0;
    auto free_events = [&]() {
        for (auto& ev : evs) (void)hipEventDestroy(ev);
        evs.clear();
    };
    for (int q = 0; q < 2 * kTimed; ++q) {
        hipEvent_t ev = nullptr;
        if (hipEventCreate(&ev) != hipSuccess) {
            free_events();
            return bail(fail(e, SJF_E_HIP, "hipEventCreate failed"));
        }
        evs.push_back(ev);
    }
    // reverse steps n1 - 1 .. n0 with the record slots of steps n0 .. n1 at slot (n - base)
    auto reverse = [&](long n0, long n1, long base) -> int {
        for (long n = n1 - 1; n >= n0; --n) {
            hipLaunchKernelGGL((sjf::k_adj_grad<T>), dim3((unsigned)((nd + 255) / 256)), dim3(256), 0, e->stream,
                               g.f, ebar(), ring, n + 1 - base, n - base, gacc);
            HIPCHK(e, hipGetLastError());
            g.hr = (n & 1) ? 2 : 4;
            g.hw = (n & 1) ? 4 : 2;
            g.er = (n & 1) ? 0 : 6;
            g.ew = (n & 1) ? 6 : 0;
            const bool timed = ntimed < kTimed;
            if (timed) HIPCHK(e, hipEventRecord(evs[2 * ntimed], e->stream));
            int r = launch_adj_step<T>(e, g, npv, block, tiles, lds, rows);
            if (r) return r;
            if (timed) HIPCHK(e, hipEventRecord(evs[2 * ntimed++ + 1], e->stream));
            g.rd = 1 - g.rd;
            if (n >= 1 && (r = inject(n - base))) return r;
        }
        return SJF_OK;
    };
    auto bail_ev = [&](int r) {
        free_events();
        return bail(r);
    };
    if (rec_all) {
        if ((rc = inject(nsteps))) return bail_ev(rc);
        if ((rc = reverse(0, nsteps, 0))) return bail_ev(rc);
    } else {
        for (long k = nck - 1; k >= 0; --k) {
            const long n0 = k * K, n1 = std::min(n0 + K, nsteps);
            if ((rc = set_step(e, n0))) return bail_ev(rc);
            if ((rc = copy_state(e, cks + L.total * k, L, false))) return bail_ev(rc);
            if ((rc = record(0))) return bail_ev(rc);
            for (long n = n0; n < n1; ++n) {
                if ((rc = launch_bare_step(s))) return bail_ev(rc);
                e->step++;
                if ((rc = record(n + 1 - n0))) return bail_ev(rc);
            }
            if (k == nck - 1 && (rc = inject(n1 - n0))) return bail_ev(rc);
            if ((rc = reverse(n0, n1, n0))) return bail_ev(rc);
        }
    }
    if (hipStreamSynchronize(e->stream) != hipSuccess) return bail_ev(fail(e, SJF_E_HIP, "hipStreamSynchronize failed"));
    double msum = 0;
    for (long q = 0; q < ntimed; ++q) {
        float ms = 0;
        if (hipEventElapsedTime(&ms, evs[2 * q], evs[2 * q + 1]) != hipSuccess)
            return bail_ev(fail(e, SJF_E_HIP, "hipEventElapsedTime failed"));
        msum += ms;
    }
    free_events();
    e->adj_ms = ntimed ? msum / ntimed : 0;
    e->adj_threads = block;
    e->adj_groups = (int)tiles;
    std::vector<double> gh(nd);
    if ((rc = d2h(e, gh.data(), gacc, sizeof(double) * nd))) return bail(rc);
    // the state is Ubar = Ebar / eps, so the accumulated sum already carries the 1/eps_v factor
    for (long v = 0; v < nd; ++v) grad[v] = -gh[v];
    // leave the engine in its final forward state (record mode never left it)
    if (!rec_all) {
        if ((rc = set_step(e, nsteps))) return bail(rc);
        if ((rc = copy_state(e, cks + L.total * nck, L, false))) return bail(rc);
        HIPCHK(e, hipStreamSynchronize(e->stream));
    }
    cleanup();
    return SJF_OK;
}

template <typename T, int NP, bool NTS>
void launch_adj_batch_step(LaunchSet* s, const sjf::AdjArgs<T>* args, const int* first, int n, int block,
                           unsigned tiles, size_t lds) {
    if (block <= 256)
        hipLaunchKernelGGL((sjf::k_adj_step_batch<T, NP, 256, NTS>), dim3(tiles), dim3(block), lds, s->stream, args, first, n);
    else if (block <= 512)
        hipLaunchKernelGGL((sjf::k_adj_step_batch<T, NP, 512, NTS>), dim3(tiles), dim3(block), lds, s->stream, args, first, n);
    else
        hipLaunchKernelGGL((sjf::k_adj_step_batch<T, NP, 1024, NTS>), dim3(tiles), dim3(block), lds, s->stream, args,
                           first, n);
}

template <typename T, int NP>
void launch_adj_batch_np(LaunchSet* s, const sjf::AdjArgs<T>* args, const int* first, int n, int block,
                         unsigned tiles, size_t lds, bool rows) {
    if (rows) {
#define SJF_LAUNCH(...) hipLaunchKernelGGL((__VA_ARGS__), dim3(tiles), dim3(block), lds, s->stream, args, first, n)
        if (block <= 512) {
            if (s->nts) SJF_LAUNCH(sjf::k_adj_rows_batch<T, NP, 512, true>);
            else SJF_LAUNCH(sjf::k_adj_rows_batch<T, NP, 512>);
        } else if (s->nts) {
            SJF_LAUNCH(sjf::k_adj_rows_batch<T, NP, 1024, true>);
        } else {
            SJF_LAUNCH(sjf::k_adj_rows_batch<T, NP, 1024>);
        }
#undef SJF_LAUNCH
        return;
    }
    if (s->nts) launch_adj_batch_step<T, NP, true>(s, args, first, n, block, tiles, lds);
    else launch_adj_batch_step<T, NP, false>(s, args, first, n, block, tiles, lds);
}

// Adjoint gradients of every engine of a launch set in one pass: the forward steps are the set's
// own fused launches; after each of them one launch adds the objectives of all engines (and, in
// record mode, records their design fields); each reverse step is one gradient launch, one fused
// reverse launch over all engines' tiles and one injection launch.  With checkpoints (K > 0, or
// when the record does not fit a quarter of the free memory) every engine's state is saved every
// K steps and each segment is recomputed with bare batch steps, as adjoint_run_t does for one
// engine.  The arithmetic of every cell is that of adjoint_run_t, so each engine's J and gradient
// are those of its own run.  gaps[i]: objective cell index of engine i; nds[i]: its design voxels.
template <typename T>
int batch_adjoint_run_t(LaunchSet* s, long nsteps, long K, const long* gaps, const long* nds, double* J_out,
                        double* const* grads, double* ms_out, int* threads_out, int* groups_out) {
    sjf_engine* e0 = s->eng[0];
    const int n = (int)s->eng.size();
    int rc = prepare_set(s, nsteps);
    if (rc) return rc;
    bool rec_all = K == 0;
    if (rec_all) {
        double rec_bytes = 0;
        for (int i = 0; i < n; ++i) rec_bytes += (double)sizeof(T) * (3 * nds[i] + 3) * (nsteps + 1);
        size_t fr = 0, tot = 0;
        HIPCHK(e0, hipMemGetInfo(&fr, &tot));
        rec_all = rec_bytes <= 0.25 * (double)fr;
        if (!rec_all) K = std::max(1L, std::lround(std::sqrt((double)nsteps)));
    }
    K = std::min(K, nsteps);  // a longer interval holds one segment of nsteps all the same
    const long nck = rec_all ? 0 : (nsteps + K - 1) / K;
    // record slots per engine; with checkpoints slot K + 1 takes the forward pass's writes, which
    // nothing reads (that pass only needs the objectives)
    const long nslots = rec_all ? nsteps + 1 : K + 2;
    std::vector<StateLayout> Ls(n);
    std::vector<char*> cks(n, nullptr);
    std::vector<void*> mem;
    auto cleanup = [&]() {
        for (void*& p : mem) dev_free(p);
        mem.clear();
    };
    auto bail = [&](int r) {
        cleanup();
        return r;
    };
    auto alloc = [&](void** p, size_t bytes) -> int {
        *p = nullptr;
        const int r = dev_alloc(e0, p, bytes);
        if (!r) mem.push_back(*p);
        return r;
    };
    std::vector<sjf::AdjBatchDev<T>> tab(n);
    std::vector<sjf::AdjArgs<T>> args(n);
    std::vector<int> first;
    int t = 0, nmat = 1;
    long maxv = 0, rows = 0;
    // rows of threads where the batch takes them (adj_tile_of), each engine its default rows; else one
    // row per workgroup with x-chunks common to all engines; a tile set on the first engine holds for
    // all (its rows at most each engine's ny, its x-chunk)
    double bytes = 0;
    for (const sjf_engine* e : s->eng) {
        rows += e->g.ny;
        bytes += field_bytes(e);
        nmat = std::max(nmat, e->nmat);
    }
    AdjTile bt = adj_tile_of<T>(e0, bytes, nmat);
    for (const sjf_engine* e : s->eng)
        if (bt.nrows == 0 && (default_thread_rows(e) + 1) * e->g.nz > (sizeof(T) == 8 ? 512 : 1024)) bt = {false, 1, 0};
    const bool brows = bt.rows;
    const int bxc = bt.xc > 0 ? bt.xc : bt.nrows > 0 ? 6 : brows ? adj_batch_chunk<T>(s) : 12;
    int bblock = 64;
    for (int i = 0; i < n; ++i) {
        sjf_engine* e = s->eng[i];
        const StateLayout L = state_layout(e);
        const long nd = nds[i];
        void *A = nullptr, *Aq = nullptr, *Ap = nullptr, *ring = nullptr, *gacc = nullptr, *dJ = nullptr;
        void* Apsi[3] = {nullptr, nullptr, nullptr};
        if (alloc(&A, sizeof(T) * 12 * e->N) || (L.q && alloc(&Aq, L.q)) || (L.p && alloc(&Ap, L.p)) ||
            alloc(&ring, sizeof(T) * (3 * nd + 3) * nslots) || alloc(&gacc, sizeof(double) * nd) ||
            alloc(&dJ, sizeof(double)))
            return bail(SJF_E_NOMEM);
        Ls[i] = L;
        if (!rec_all && alloc((void**)&cks[i], L.total * (nck + 1)))
            return bail(fail(e0, SJF_E_NOMEM, "checkpoint storage allocation failed (" +
                                                  std::to_string((double)L.total * (nck + 1) / 1e9) + " GB)"));
        for (int d = 0; d < 3; ++d) {
            if ((double)L.psi[d] / 6 * 8 >= 2147483648.0)
                return bail(fail(e0, SJF_E_UNSUPPORTED, "adjoint PML auxiliaries exceed 2 GiB on one axis"));
            if (L.psi[d] && alloc(&Apsi[d], L.psi[d] / 6 * 8)) return bail(SJF_E_NOMEM);
        }
        sjf::AdjBatchDev<T>& d = tab[i];
        std::memset(&d, 0, sizeof(d));
        d.F[0] = (const T*)e->Fbuf[0];
        d.F[1] = (const T*)e->Fbuf[1];
        d.A[0] = (T*)A;
        d.A[1] = (T*)A + (size_t)6 * e->N;
        d.ring = (T*)ring;
        d.gacc = (double*)gacc;
        d.J = (double*)dJ;
        d.nyz = (long)e->g.ny * e->g.nz;
        d.ny = e->g.ny;
        d.nz = e->g.nz;
        std::vector<uint32_t> gw;
        if ((rc = words_at(e, {gaps[i]}, gw))) return bail(rc);
        for (int q = 0; q < 3; ++q) {
            d.dlo[q] = e->dlo[q];
            d.de[q] = e->dhi[q] - e->dlo[q];
            d.ie[q] = inv_eps_at(e, gaps[i], q, gw[0]);
        }
        d.nd = nd;
        d.gap = gaps[i];
        d.dt = e->dt;
        sjf::AdjArgs<T>& g = args[i];
        std::memset(&g, 0, sizeof(g));
        // the first engine's tile form for all (they share nz and the precision)
        if (brows) {
            const int r = bt.nrows > 0 ? std::min(bt.nrows, e->g.ny) : default_thread_rows(e);
            g.f = step_args<T>(e, r, std::min(bxc, e->g.nx));
            bblock = std::max(bblock, (((r + 1) * e->g.nz + 63) / 64) * 64);
        } else {
            g.f = step_args<T>(e, 1, adj_xchunk(e, kBatchAdjGroups, rows));  // one y row per workgroup
            g.f.nty = e->g.ny;
        }
        g.A[0] = d.A[0];
        g.A[1] = d.A[1];
        g.Aq = (T*)Aq;
        g.Ap = (T*)Ap;
        for (int q = 0; q < 3; ++q) g.Apsi[q] = (T*)Apsi[q];
        first.push_back(t);
        t += (int)((long)g.f.nty * ((e->g.nx + g.f.xc - 1) / g.f.xc));
        maxv = std::max(maxv, nd + 3);
    }
    first.push_back(t);
    // the reverse step's buffer roles alternate with the parity p of the step index n: read set
    // rd = (nsteps - 1 - n) & 1, H auxiliary pair read 2 / 4 and E pair read 0 / 6
    std::vector<sjf::AdjArgs<T>> argp[2] = {args, args};
    for (int p = 0; p < 2; ++p)
        for (sjf::AdjArgs<T>& g : argp[p]) {
            g.rd = (int)((nsteps - 1 - p) & 1);
            g.hr = p ? 2 : 4;
            g.hw = p ? 4 : 2;
            g.er = p ? 0 : 6;
            g.ew = p ? 6 : 0;
        }
    void *d_tab = nullptr, *d_args0 = nullptr, *d_args1 = nullptr, *d_first = nullptr;
    auto upload = [&](void** dst, auto const& v) -> int {
        *dst = nullptr;
        const int r = upload_vec(e0, s->stream, dst, v);
        if (*dst) mem.push_back(*dst);  // freed with the rest, also when the copy failed
        return r;
    };
    if ((rc = upload(&d_tab, tab)) || (rc = upload(&d_args0, argp[0])) || (rc = upload(&d_args1, argp[1])) ||
        (rc = upload(&d_first, first)))
        return bail(rc);
    const auto* tabp = (const sjf::AdjBatchDev<T>*)d_tab;
    const sjf::AdjArgs<T>* argd[2] = {(const sjf::AdjArgs<T>*)d_args0, (const sjf::AdjArgs<T>*)d_args1};
    const int block = brows ? bblock : ((e0->g.nz + 63) / 64) * 64;
    const size_t lds = adj_lds_bytes<T>(brows, block, nmat);
    if (!lds_fits<T>(brows ? 8 * (size_t)block + 2 * (size_t)e0->g.nz : 12 * (size_t)block, nmat))
        return bail(fail(e0, SJF_E_UNSUPPORTED, "adjoint tile needs more than 64 KiB of LDS"));
    const int npv = np_variant_of(e0->maxp, e0->uniform);
    const dim3 grid_v((unsigned)((maxv + 255) / 256), (unsigned)n);
    auto record = [&](long sl, int objective) -> int {
        hipLaunchKernelGGL((sjf::k_adj_record_batch<T>), grid_v, dim3(256), 0, s->stream, tabp,
                           (int)(e0->step & 1), sl, objective);
        SETCHK(s, hipGetLastError());
        return SJF_OK;
    };
    auto save_all = [&](long k, bool save) -> int {
        for (int i = 0; i < n; ++i) {
            const int r = copy_state(s->eng[i], cks[i] + Ls[i].total * k, Ls[i], save, s->stream);
            if (r) return r;
        }
        return SJF_OK;
    };
    // ---- forward pass: the objectives after every step; the record or checkpoints every K steps
    if (rec_all && (rc = record(0, 0))) return bail(rc);
    for (long q = 0; q < nsteps; ++q) {
        if (!rec_all && q % K == 0 && (rc = save_all(q / K, true))) return bail(rc);
        if ((rc = launch_one_step(s, samples_at(s, e0->step)))) return bail(rc);
        advance_hosts(s, 1);
        if ((rc = record(rec_all ? q + 1 : K + 1, 1))) return bail(rc);
    }
    if (!rec_all && (rc = save_all(nck, true))) return bail(rc);
    // ---- reverse pass
    constexpr int kTimed = 64;
    std::vector<hipEvent_t> evs;
    auto free_events = [&]() {
        for (auto& ev : evs) (void)hipEventDestroy(ev);
        evs.clear();
    };
    auto bail_ev = [&](int r) {
        free_events();
        return bail(r);
    };
    for (int q = 0; q < 2 * kTimed; ++q) {
        hipEvent_t ev = nullptr;
        if (hipEventCreate(&ev) != hipSuccess) return bail_ev(fail(e0, SJF_E_HIP, "hipEventCreate failed"));
        evs.push_back(ev);
    }
    int rd = 0;
    auto inject = [&](long sl) -> int {
        hipLaunchKernelGGL((sjf::k_adj_inject_batch<T>), dim3(1, (unsigned)n), dim3(64), 0, s->stream, tabp, rd, sl);
        SETCHK(s, hipGetLastError());
        return SJF_OK;
    };
    const dim3 grid_g((unsigned)((maxv - 3 + 255) / 256), (unsigned)n);
    long ntimed = 0;
    // one reverse step: gradient term, fused reverse launch (timed for the first kTimed steps)
    auto reverse_step = [&](long q, long base) -> int {
        hipLaunchKernelGGL((sjf::k_adj_grad_batch<T>), grid_g, dim3(256), 0, s->stream, tabp, rd, q + 1 - base,
                           q - base);
        SETCHK(s, hipGetLastError());
        const bool timed = ntimed < kTimed;
        if (timed) SETCHK(s, hipEventRecord(evs[2 * ntimed], s->stream));
        const sjf::AdjArgs<T>* ad = argd[q & 1];
        switch (npv) {
            case 0: launch_adj_batch_np<T, 0>(s, ad, (const int*)d_first, n, block, (unsigned)t, lds, brows); break;
            case 1: launch_adj_batch_np<T, 1>(s, ad, (const int*)d_first, n, block, (unsigned)t, lds, brows); break;
            case 3: launch_adj_batch_np<T, 3>(s, ad, (const int*)d_first, n, block, (unsigned)t, lds, brows); break;
            default: launch_adj_batch_np<T, 4>(s, ad, (const int*)d_first, n, block, (unsigned)t, lds, brows); break;
        }
        SETCHK(s, hipGetLastError());
        if (timed) SETCHK(s, hipEventRecord(evs[2 * ntimed++ + 1], s->stream));
        return SJF_OK;
    };
    // reverse steps q1 - 1 .. q0 with the record slots of steps q0 .. q1 at slot (q - base)
    auto reverse = [&](long q0, long q1, long base) -> int {
        for (long q = q1 - 1; q >= q0; --q) {
            int r = reverse_step(q, base);
            if (r) return r;
            rd = 1 - rd;
            if (q >= 1 && (r = inject(q - base))) return r;
        }
        return SJF_OK;
    };
    auto set_steps = [&](long step) -> int {
        if (hipStreamSynchronize(s->stream) != hipSuccess) return fail(e0, SJF_E_HIP, "hipStreamSynchronize failed");
        for (sjf_engine* e : s->eng) {
            const int r = set_step(e, step);
            if (r) return r;
        }
        return SJF_OK;
    };
    if (rec_all) {
        if ((rc = inject(nsteps)) || (rc = reverse(0, nsteps, 0))) return bail_ev(rc);
    } else {
        for (long k = nck - 1; k >= 0; --k) {
            const long q0 = k * K, q1 = std::min(q0 + K, nsteps);
            if ((rc = set_steps(q0)) || (rc = save_all(k, false)) || (rc = record(0, 0))) return bail_ev(rc);
            for (long q = q0; q < q1; ++q) {
                if ((rc = launch_bare_step(s))) return bail_ev(rc);
                for (sjf_engine* e : s->eng) e->step++;
                if ((rc = record(q + 1 - q0, 0))) return bail_ev(rc);
            }
            if (k == nck - 1 && (rc = inject(q1 - q0))) return bail_ev(rc);
            if ((rc = reverse(q0, q1, q0))) return bail_ev(rc);
        }
    }
    if (hipStreamSynchronize(s->stream) != hipSuccess)
        return bail_ev(fail(e0, SJF_E_HIP, "hipStreamSynchronize failed"));
    double msum = 0;
    for (long q = 0; q < ntimed; ++q) {
        float ms = 0;
        if (hipEventElapsedTime(&ms, evs[2 * q], evs[2 * q + 1]) != hipSuccess)
            return bail_ev(fail(e0, SJF_E_HIP, "hipEventElapsedTime failed"));
        msum += ms;
    }
    free_events();
    *ms_out = ntimed ? msum / ntimed : 0;
    *threads_out = block;
    *groups_out = t;
    for (int i = 0; i < n; ++i) {
        std::vector<double> gh(nds[i]);
        if ((rc = d2h(e0, gh.data(), tab[i].gacc, sizeof(double) * nds[i])) ||
            (rc = d2h(e0, &J_out[i], tab[i].J, sizeof(double))))
            return bail(rc);
        // the state is Ubar = Ebar / eps, so the sums already carry the 1/eps_v factor
        for (long v = 0; v < nds[i]; ++v) grads[i][v] = -gh[v];
    }
    // leave every engine in its final forward state (record mode never left it)
    if (!rec_all) {
        if ((rc = set_steps(nsteps)) || (rc = save_all(nck, false))) return bail(rc);
        if (hipStreamSynchronize(s->stream) != hipSuccess) return bail(fail(e0, SJF_E_HIP, "hipStreamSynchronize failed"));
    }
    cleanup();
    return SJF_OK;
}

}  // namespace

extern "C" int sjf_adjoint_run(sjf_engine* e, long nsteps, int checkpoint_every, const int gap[3], double* J,
                               double* grad, size_t cap) {
    if (!e || nsteps < 1 || checkpoint_every < 0 || !gap || !J || !grad) return SJF_E_ARG;
    if (!e->emap_h.empty()) return fail(e, SJF_E_UNSUPPORTED, "adjoint runs take the LUT's eps_inf (no eps maps)");
    if (e->g.nz > 1024) return fail(e, SJF_E_UNSUPPORTED, "the reverse step spans the z line: nz <= 1024");
    if (e->batch) return fail(e, SJF_E_STATE, "engine is stepped by its batch");
    if (e->step != 0) return fail(e, SJF_E_STATE, "the adjoint run starts from step 0");
    if (e->deps_h.empty()) return fail(e, SJF_E_STATE, "no design region (sjf_set_design_eps)");
    const int n[3] = {e->g.nx, e->g.ny, e->g.nz};
    for (int d = 0; d < 3; ++d)
        if (gap[d] < 0 || gap[d] >= n[d]) return fail(e, SJF_E_ARG, "objective cell outside the grid");
    const long nd = (long)e->deps_h.size();
    if (cap < (size_t)nd) return fail(e, SJF_E_ARG, "gradient buffer smaller than the design region");
    HIPCHK(e, hipSetDevice(e->g.device));
    const long q = cell_index(e, gap[0], gap[1], gap[2]);
    return e->prec == 4 ? adjoint_run_t<float>(e, nsteps, checkpoint_every, q, J, grad, nd)
                        : adjoint_run_t<double>(e, nsteps, checkpoint_every, q, J, grad, nd);
}

extern "C" int sjf_set_adjoint_tile(sjf_engine* e, int form, int rows, int xchunk) {
    if (!e || xchunk < 0) return SJF_E_ARG;
    if (form == SJF_TILE_REGISTER_ROWS) {
        if (rows != 1) return fail(e, SJF_E_ARG, "the register form of the reverse step owns one row per workgroup");
    } else if (form == SJF_TILE_THREAD_ROWS) {
        if (!thread_rows_fit(e, rows))
            return fail(e, SJF_E_ARG, "row-of-threads tile needs (rows + 1) * nz <= 1024");
        const int block = (((rows + 1) * e->g.nz + 63) / 64) * 64;
        // FP64 tiles stop at 512 threads: at 1024 the register budget of 128 per thread spills
        if (e->prec == 8 && block > 512)
            return fail(e, SJF_E_ARG, "FP64 row-of-threads reverse tile needs (rows + 1) * nz <= 512");
        const size_t values = 8 * (size_t)block + 2 * (size_t)e->g.nz;
        if (!(e->prec == 4 ? lds_fits<float>(values, e->nmat) : lds_fits<double>(values, e->nmat)))
            return fail(e, SJF_E_ARG, "adjoint row-of-threads tile needs more than 64 KiB of LDS");
    } else {
        return fail(e, SJF_E_ARG, "unknown tile form");
    }
    e->adj_form = form;
    e->adj_rows = rows;
    e->adj_xc = xchunk;
    e->adj_set = true;
    return SJF_OK;
}

extern "C" int sjf_adjoint_kernel_info(const sjf_engine* e, double* ms_mean, int* threads, int* groups) {
    if (!e || !ms_mean) return SJF_E_ARG;
    if (e->adj_groups == 0) return SJF_E_STATE;
    *ms_mean = e->adj_ms;
    if (threads) *threads = e->adj_threads;
    if (groups) *groups = e->adj_groups;
    return SJF_OK;
}

// ============================================================================ batches ====

namespace {

// ======================================================================== flux read-out ===
// The flux of a DFT plane is reduced on the device in two launches (k_dft_flux_part,
// k_dft_flux_sum) through a buffer of nf * (nb + 1) doubles: nb partial sums per frequency, then
// the nf results that are copied out.  sjf_dft_flux allocates that buffer per call;
// sjf_dft_flux_noalloc uses `scratch`, a static device array of at most 64 frequencies x 65
// doubles (33 KiB) that every device the library runs on holds until the process ends.  Every
// slot a call reads is written earlier in the same call, so nothing needs clearing; calls that
// overlap on one device share the array and race.
constexpr int kFluxMaxBlocks = 64;
constexpr int kFluxScratchDoubles = SJF_MAX_DFT_FREQS * (kFluxMaxBlocks + 1);
static __device__ __align__(256) double scratch[kFluxScratchDoubles];

std::mutex g_scratch_mu;
std::vector<double*> g_scratch_ptr;  // per device: the address of `scratch` there

// Resolves this device's copy of `scratch` (the device must be current).  The array's name in
// host code is only a stand-in; kernels and copies take the address resolved here.
int scratch_setup(int device) {
    std::lock_guard<std::mutex> lk(g_scratch_mu);
    if ((int)g_scratch_ptr.size() <= device) g_scratch_ptr.resize(device + 1, nullptr);
    if (g_scratch_ptr[device]) return SJF_OK;
    void* p = nullptr;
    const hipError_t st = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (st != hipSuccess || !p) {
        g_create_error = std::string("hipGetSymbolAddress(scratch): ") + hipGetErrorString(st);
        return SJF_E_HIP;
    }
    g_scratch_ptr[device] = (double*)p;
    return SJF_OK;
}

double* scratch_on(int device) {
    std::lock_guard<std::mutex> lk(g_scratch_mu);
    return device >= 0 && device < (int)g_scratch_ptr.size() ? g_scratch_ptr[device] : nullptr;
}

struct FluxPlan {
    const Dft* d;
    int slot[4];  // E_a, E_b, H_a, H_b
    int nf, nb;
    long scratch_doubles() const { return (long)nf * (nb + 1); }
};

int flux_plan(sjf_engine* e, int id, int axis, const double* flux, size_t cap, FluxPlan* fp) {
    if (!e || !flux || id < 0 || id >= (int)e->dft.size() || axis < 0 || axis > 2) return SJF_E_ARG;
    const Dft& d = e->dft[id];
    if (d.hi[axis] - d.lo[axis] != 1) return fail(e, SJF_E_ARG, "a flux plane is one cell thick along its normal");
    const int a = (axis + 1) % 3, b = (axis + 2) % 3;
    int slot[6] = {-1, -1, -1, -1, -1, -1};
    for (int q = 0; q < d.ncomp; ++q) slot[d.comps[q]] = q;
    if (slot[a] < 0 || slot[b] < 0 || slot[3 + a] < 0 || slot[3 + b] < 0)
        return fail(e, SJF_E_ARG, "a flux plane needs both tangential E and both tangential H components");
    fp->d = &d;
    fp->slot[0] = slot[a];
    fp->slot[1] = slot[b];
    fp->slot[2] = slot[3 + a];
    fp->slot[3] = slot[3 + b];
    fp->nf = (int)d.freqs.size();
    fp->nb = (int)std::min<long>(kFluxMaxBlocks, std::max<long>(1, (d.ncell + 255) / 256));
    if (cap < (size_t)fp->nf) return fail(e, SJF_E_ARG, "output buffer too small");
    return SJF_OK;
}

// buf: nf * nb partial sums, then the nf results
int flux_run(sjf_engine* e, const FluxPlan& fp, double* buf, double* flux) {
    const Dft& d = *fp.d;
    hipLaunchKernelGGL(sjf::k_dft_flux_part, dim3(fp.nb, fp.nf), dim3(256), 0, e->stream, (const double2*)d.acc,
                       (const double2*)d.cmp, d.ncell, fp.nf, fp.slot[0], fp.slot[1], fp.slot[2], fp.slot[3], fp.nb,
                       buf);
    if (hipGetLastError() != hipSuccess) return fail(e, SJF_E_HIP, "k_dft_flux_part launch failed");
    double* out = buf + (long)fp.nf * fp.nb;
    hipLaunchKernelGGL(sjf::k_dft_flux_sum, dim3(1), dim3(64), 0, e->stream, (const double*)buf, fp.nf, fp.nb,
                       e->g.dx * e->g.dx, out);
    if (hipGetLastError() != hipSuccess) return fail(e, SJF_E_HIP, "k_dft_flux_sum launch failed");
    return d2h(e, flux, out, sizeof(double) * fp.nf);
}

}  // namespace

struct sjf_batch {
    LaunchSet* set = nullptr;
    std::string err;
    double adj_ms = 0;  // fused reverse launch of the last batched adjoint run
    int adj_threads = 0, adj_groups = 0;
};

namespace {
int sync_engine(sjf_engine* e) {
    HIPCHK(e, hipSetDevice(e->g.device));
    if (e->batch) HIPCHK(e, hipStreamSynchronize(e->batch->set->stream));
    HIPCHK(e, hipStreamSynchronize(e->stream));
    return SJF_OK;
}
}  // namespace

// =========================================================================== C ABI ====

extern "C" {

int sjf_create(const sjf_grid* g, sjf_engine** out) {
    if (!g || !out) {
        g_create_error = "null argument";
        return SJF_E_ARG;
    }
    *out = nullptr;
    if (g->nx < 1 || g->ny < 1 || g->nz < 1 || !(g->dx > 0) || !(g->courant > 0)) {
        g_create_error = "grid dimensions, dx and courant must be positive";
        return SJF_E_ARG;
    }
    if (g->nz > 1024 && g->periodic[2]) {
        g_create_error = "a z line longer than 1024 cells is stepped in passes, which needs a non-periodic z axis";
        return SJF_E_UNSUPPORTED;
    }
    if (g->precision != SJF_FP32 && g->precision != SJF_FP64) {
        g_create_error = "precision must be SJF_FP32 (4) or SJF_FP64 (8)";
        return SJF_E_ARG;
    }
    if ((double)g->nx * g->ny * g->nz * 6 >= 4294967296.0) {
        g_create_error = "grid too large for one engine (6 * cells must stay below 2^32)";
        return SJF_E_UNSUPPORTED;
    }
    int ndev = 0;
    hipError_t st = hipGetDeviceCount(&ndev);
    if (st != hipSuccess || ndev == 0) {
        g_create_error = std::string("no HIP device available: ") + hipGetErrorString(st);
        return SJF_E_HIP;
    }
    if (g->device < 0 || g->device >= ndev) {
        g_create_error = "device ordinal out of range";
        return SJF_E_ARG;
    }
    st = hipSetDevice(g->device);
    if (st != hipSuccess) {
        g_create_error = std::string("hipSetDevice: ") + hipGetErrorString(st);
        return SJF_E_HIP;
    }
    if (int rc = scratch_setup(g->device)) return rc;
    stage_engines(1);
    sjf_engine* e = new sjf_engine();
    e->g = *g;
    e->prec = g->precision;
    e->N = (long)g->nx * g->ny * g->nz;
    e->dt = g->courant * g->dx;
    st = hipStreamCreateWithFlags(&e->stream, hipStreamNonBlocking);
    if (st != hipSuccess) {
        g_create_error = std::string("hipStreamCreate: ") + hipGetErrorString(st);
        delete e;
        stage_engines(-1);
        return SJF_E_HIP;
    }
    auto bail = [&](int rc) {
        g_create_error = e->err;
        free_all(e);
        (void)hipStreamDestroy(e->stream);
        delete e;
        stage_engines(-1);
        return rc;
    };
    for (int b = 0; b < 2; ++b) {
        int rc = dev_alloc(e, &e->Fbuf[b], (size_t)e->prec * 6 * e->N);
        if (rc) return bail(rc);
    }
    if (int rc = dev_alloc(e, (void**)&e->d_step, 2 * sizeof(long))) return bail(rc);
    // PML tables for all axes (b = 1, a = 0 until sjf_set_pml fills an axis)
    {
        const int n3[3] = {g->nx, g->ny, g->nz};
        int off = 0;
        for (int d = 0; d < 3; ++d) {
            e->coff[d] = off;
            off += 4 * n3[d];
        }
        std::vector<double> tab(off, 0.0);
        for (int d = 0; d < 3; ++d)
            for (int i = 0; i < n3[d]; ++i) {
                tab[e->coff[d] + i] = 1.0;
                tab[e->coff[d] + 2 * n3[d] + i] = 1.0;
            }
        int rc = dev_alloc(e, &e->coefbuf, (size_t)e->prec * off);
        if (!rc) rc = e->prec == 4 ? convert_to_device<float>(e, e->coefbuf, tab.data(), off)
                                   : convert_to_device<double>(e, e->coefbuf, tab.data(), off);
        if (rc) return bail(rc);
    }
    // default material: vacuum
    e->lut_h.assign(1, sjf_material{});
    e->lut_h[0].eps_inf = 1.0;
    e->nmat = 1;
    if (int rc = upload_lut(e)) return bail(rc);
    choose_tile(e);
    *out = e;
    return SJF_OK;
}

int sjf_destroy(sjf_engine* e) {
    if (!e) return SJF_E_ARG;
    if (e->batch) return fail(e, SJF_E_STATE, "destroy the batch before its engines");
    (void)hipSetDevice(e->g.device);
    (void)hipStreamSynchronize(e->stream);
    free_all(e);
    (void)hipStreamDestroy(e->stream);
    delete e;
    stage_engines(-1);
    return SJF_OK;
}

const char* sjf_last_error(const sjf_engine* e) { return e ? e->err.c_str() : g_create_error.c_str(); }

int sjf_set_materials(sjf_engine* e, const uint32_t* mat_word, const sjf_material* lut, int n_mat) {
    if (!e || !mat_word || !lut) return SJF_E_ARG;
    if (n_mat < 1 || n_mat > SJF_MAX_MATERIALS) return fail(e, SJF_E_ARG, "n_mat must be in [1, 255]");
    if (int rc = sync_engine(e)) return rc;
    for (int m = 0; m < n_mat; ++m) {
        if (lut[m].npoles < 0 || lut[m].npoles > SJF_MAX_POLES)
            return fail(e, SJF_E_ARG, "npoles must be in [0, 4]");
        if (!(lut[m].eps_inf > 0)) return fail(e, SJF_E_ARG, "eps_inf must be positive");
    }
    // the words go to a buffer of their own: a word that is refused leaves the materials as they were
    uint32_t* words = nullptr;
    unsigned long long *d_first = nullptr, first = ~0ull;
    int rc = dev_alloc(e, (void**)&words, sizeof(uint32_t) * e->N);
    if (!rc) rc = dev_alloc(e, (void**)&d_first, sizeof(first));
    if (!rc) rc = h2d(e, words, mat_word, sizeof(uint32_t) * e->N);
    if (!rc) rc = h2d(e, d_first, &first, sizeof(first));
    if (!rc) {
        hipLaunchKernelGGL(sjf::k_check_words, dim3((unsigned)std::min(2048L, (e->N + 255) / 256)), dim3(256), 0,
                           e->stream, words, e->N, n_mat, !e->deps_h.empty(), d_first);
        rc = hipGetLastError() == hipSuccess ? d2h(e, &first, d_first, sizeof(first))
                                             : fail(e, SJF_E_HIP, "k_check_words launch failed");
    }
    dev_free(d_first);
    if (!rc && first != ~0ull)
        rc = first & 1 ? fail(e, SJF_E_STATE, "design id 255 used before sjf_set_design_eps")
                       : fail(e, SJF_E_ARG, "material word references an id >= n_mat");
    MatPlan plan;
    if (!rc) rc = plan_materials(e, std::vector<sjf_material>(lut, lut + n_mat), e->pml_fref, any_pml(e), &plan);
    if (rc) {
        dev_free(words);
        return rc;
    }
    dev_free(e->given);
    e->given = words;
    e->given_lut.assign(lut, lut + n_mat);
    e->have_mat = true;
    return apply_materials(e, plan);
}

int sjf_set_eps_maps(sjf_engine* e, const double* eps) {
    if (!e) return SJF_E_ARG;
    if (int rc = sync_engine(e)) return rc;
    if (!eps) {
        if (!e->have_mat) return SJF_OK;  // there is none
    } else {
        for (long q = 0; q < 3 * e->N; ++q)
            if (!(eps[q] > 0) || !std::isfinite(eps[q])) return fail(e, SJF_E_ARG, "map eps must be positive and finite");
        if (int rc = default_words(e)) return rc;
    }
    MatPlan plan;
    if (int rc = plan_materials(e, &plan)) return rc;
    begin_change(e, e->mat_ready);
    if (eps) {
        e->emap_h.assign(eps, eps + 3 * e->N);
    } else {
        e->emap_h.clear();
        e->emap_eff.clear();
        dev_free(e->emap);
    }
    return apply_materials(e, plan);
}

int sjf_set_pml_dispersion(sjf_engine* e, double f_ref) {
    if (!e) return SJF_E_ARG;
    if (!(f_ref >= 0) || !std::isfinite(f_ref)) return fail(e, SJF_E_ARG, "f_ref must be >= 0");
    if (e->step != 0) return fail(e, SJF_E_STATE, "the PML media must be set before the first step");
    if (int rc = sync_engine(e)) return rc;
    MatPlan plan;
    if (e->have_mat)
        if (int rc = plan_materials(e, e->given_lut, f_ref, any_pml(e), &plan)) return rc;
    e->pml_fref = f_ref;
    return e->have_mat ? apply_materials(e, plan) : SJF_OK;
}

int sjf_set_design_eps(sjf_engine* e, const int lo[3], const int hi[3], const double* eps) {
    if (!e || !lo || !hi || !eps) return SJF_E_ARG;
    const int n[3] = {e->g.nx, e->g.ny, e->g.nz};
    long cnt = 1;
    for (int d = 0; d < 3; ++d) {
        if (lo[d] < 0 || hi[d] > n[d] || hi[d] <= lo[d]) return fail(e, SJF_E_ARG, "design box outside grid");
        cnt *= hi[d] - lo[d];
    }
    if (!e->deps_h.empty())
        for (int d = 0; d < 3; ++d)
            if (lo[d] != e->dlo[d] || hi[d] != e->dhi[d])
                return fail(e, SJF_E_STATE, "design box cannot change once set");
    for (long q = 0; q < cnt; ++q)
        if (!(eps[q] > 0)) return fail(e, SJF_E_ARG, "design eps must be positive");
    if (int rc = sync_engine(e)) return rc;
    const bool first = !e->dinv, whole = !e->mat_ready;  // whole: an earlier call left the materials incomplete
    MatPlan plan;
    if (whole)
        if (int rc = plan_materials(e, &plan)) return rc;
    int rc = dev_alloc(e, &e->dinv, (size_t)e->prec * cnt);
    if (!rc) rc = default_words(e);
    if (rc) {
        if (first) dev_free(e->dinv);
        return rc;
    }
    begin_change(e, e->mat_ready);
    for (int d = 0; d < 3; ++d) {
        e->dlo[d] = lo[d];
        e->dhi[d] = hi[d];
    }
    e->deps_h.assign(eps, eps + cnt);
    std::vector<double> inv(cnt);
    for (long q = 0; q < cnt; ++q) inv[q] = 1.0 / eps[q];
    rc = e->prec == 4 ? convert_to_device<float>(e, e->dinv, inv.data(), cnt)
                      : convert_to_device<double>(e, e->dinv, inv.data(), cnt);
    if (rc) return rc;
    // mark design voxels in the material word (all three E components)
    hipLaunchKernelGGL(sjf::k_mark_design, dim3((unsigned)((cnt + 255) / 256)), dim3(256), 0, e->stream, e->given, n[1],
                       n[2], lo[0], lo[1], lo[2], hi[1] - lo[1], hi[2] - lo[2], cnt);
    HIPCHK(e, hipGetLastError());
    if (whole) return apply_materials(e, plan);
    rc = update_words(e);
    if (rc) return rc;
    e->uniform = false;
    choose_tile(e);
    e->mat_ready = true;
    return SJF_OK;
}

int sjf_set_pml(sjf_engine* e, const int cells[6], double R, double power) {
    if (!e || !cells) return SJF_E_ARG;
    if (!(R > 0 && R < 1) || !(power >= 0)) return fail(e, SJF_E_ARG, "R must be in (0,1), power >= 0");
    if (e->step != 0) return fail(e, SJF_E_STATE, "PML must be set before the first step");
    bool some = false;
    for (int d = 0; d < 3; ++d) {
        const int n = axis_n(e, d);
        const int lo = cells[2 * d], hi = cells[2 * d + 1];
        if (lo < 0 || hi < 0 || lo + hi > n) return fail(e, SJF_E_ARG, "PML thicker than the grid");
        if ((lo > 0 || hi > 0) && e->g.periodic[d]) return fail(e, SJF_E_ARG, "PML on a periodic axis");
        // the step kernels address the six auxiliary slots of a slab within one 2 GiB buffer range
        if ((double)e->prec * 6 * (lo + hi) * (e->N / n) >= 2147483648.0)
            return fail(e, SJF_E_UNSUPPORTED, "PML slab auxiliaries exceed 2 GiB on one axis");
        some = some || lo > 0 || hi > 0;
    }
    MatPlan plan;
    const bool fold = e->have_mat && e->pml_fref > 0;
    if (fold)
        if (int rc = plan_materials(e, e->given_lut, e->pml_fref, some, &plan)) return rc;
    if (int rc = sync_engine(e)) return rc;
    begin_change(e, e->pml_ready);
    int off = 0;
    for (int d = 0; d < 3; ++d) off += 4 * axis_n(e, d);
    std::vector<double> tab(off, 0.0);
    for (int d = 0; d < 3; ++d) {
        const int n = axis_n(e, d);
        const int lo = cells[2 * d], hi = cells[2 * d + 1];
        e->pml[2 * d] = lo;
        e->pml[2 * d + 1] = hi;
        e->pml_on[d] = (lo > 0 || hi > 0);
        dev_free(e->psibuf[d]);
        e->slab[d] = 0;
        const double dx = e->g.dx;
        // sigma(u) = sigma_max (u/d)^p, sigma_max = -(p+1) ln R / (2 d): meep::pml(d) defaults
        auto sigma = [&](double x) {
            double s = 0;
            if (lo > 0) {
                const double L = lo * dx, u = L - x;
                if (u > 0) s += -(power + 1) * std::log(R) / (2 * L) * std::pow(u / L, power);
            }
            if (hi > 0) {
                const double L = hi * dx, u = x - (n - hi) * dx;
                if (u > 0) s += -(power + 1) * std::log(R) / (2 * L) * std::pow(u / L, power);
            }
            return s;
        };
        for (int i = 0; i < n; ++i) {
            const double bE = std::exp(-sigma(i * dx) * e->dt);
            const double bH = std::exp(-sigma((i + 0.5) * dx) * e->dt);
            tab[e->coff[d] + i] = bE;
            tab[e->coff[d] + n + i] = bE - 1.0;
            tab[e->coff[d] + 2 * n + i] = bH;
            tab[e->coff[d] + 3 * n + i] = bH - 1.0;
        }
        if (!e->pml_on[d]) continue;
        e->slab[d] = (long)(lo + hi) * (e->N / n);
        int rc = dev_alloc(e, &e->psibuf[d], (size_t)e->prec * 6 * e->slab[d]);
        if (rc) return rc;
    }
    int rc = e->prec == 4 ? convert_to_device<float>(e, e->coefbuf, tab.data(), off)
                          : convert_to_device<double>(e, e->coefbuf, tab.data(), off);
    if (rc) return rc;
    e->pml_ready = true;
    return fold ? apply_materials(e, plan) : SJF_OK;  // the slabs moved
}

int sjf_add_source(sjf_engine* e, int comp, const double box[6], const sjf_pulse* p, double amp_re,
                   double amp_im) {
    if (!e || !box || !p) return SJF_E_ARG;
    if (comp < 0 || comp > 5) return fail(e, SJF_E_ARG, "source component must be Ex..Hz");
    if (p->kind != SJF_SRC_GAUSSIAN && p->kind != SJF_SRC_CONTINUOUS) return fail(e, SJF_E_ARG, "bad pulse kind");
    if (!(p->freq > 0)) return fail(e, SJF_E_ARG, "pulse frequency must be positive");
    if (p->kind == SJF_SRC_GAUSSIAN && !(p->width > 0)) return fail(e, SJF_E_ARG, "pulse width must be positive");
    Source s;
    s.comp = comp;
    s.p = *p;
    std::memset(&s.dev, 0, sizeof(s.dev));
    s.dev.kind = p->kind;
    s.dev.amp_re = amp_re;
    s.dev.amp_im = amp_im;
    if (p->kind == SJF_SRC_GAUSSIAN) {
        // gaussian_src_time_phase constructor (reference src/disp.cpp:378-393)
        s.dev.omega = 2 * M_PI * p->freq;
        s.dev.width = p->width;
        s.dev.phi = p->phase + M_PI;
        s.dev.peak = 0.5 * (p->t_start + p->t_end);
        double cut = (p->t_end - p->t_start) * 0.5;
        while (std::exp(-cut * cut / (2 * p->width * p->width)) < 1e-100) cut *= 0.9;
        s.dev.cutoff = (double)(float)cut;
    } else {
        s.dev.freq = p->freq;
        s.dev.cw_width = p->width;
        s.dev.t_start = p->t_start;
        s.dev.t_end = p->t_end;
        s.dev.slow = p->slowness;
    }
    std::vector<int> ids[3];
    std::vector<double> ws[3];
    for (int d = 0; d < 3; ++d)
        axis_weights(axis_n(e, d), e->g.dx, kCompOff[comp][d], e->g.periodic[d], box[d], box[3 + d], ids[d], ws[d]);
    for (size_t a = 0; a < ids[0].size(); ++a)
        for (size_t b = 0; b < ids[1].size(); ++b)
            for (size_t c = 0; c < ids[2].size(); ++c) {
                s.idx.push_back(cell_index(e, ids[0][a], ids[1][b], ids[2][c]));
                s.wt.push_back(ws[0][a] * ws[1][b] * ws[2][c]);
            }
    for (int d = 0; d < 3; ++d) {
        s.ids[d] = ids[d];
        std::sort(s.ids[d].begin(), s.ids[d].end());
    }
    e->src.push_back(std::move(s));
    e->version++;
    return SJF_OK;
}

int sjf_last_source_time(const sjf_engine* e, double* t) {
    if (!e || !t) return SJF_E_ARG;
    double m = 0;
    for (const auto& s : e->src) {
        // src_time::last_time rounds to float (gaussian_src_time_phase: src/disp.hpp:119)
        const double lt = s.p.kind == SJF_SRC_GAUSSIAN ? (double)(float)(s.dev.peak + s.dev.cutoff)
                                                       : (double)(float)s.p.t_end;
        m = std::max(m, lt);
    }
    *t = m;
    return SJF_OK;
}

int sjf_dt(const sjf_engine* e, double* dt) {
    if (!e || !dt) return SJF_E_ARG;
    *dt = e->dt;
    return SJF_OK;
}

int sjf_time(const sjf_engine* e, double* t) {
    if (!e || !t) return SJF_E_ARG;
    *t = e->step * e->dt;
    return SJF_OK;
}

int sjf_step_count(const sjf_engine* e, long* n) {
    if (!e || !n) return SJF_E_ARG;
    *n = e->step;
    return SJF_OK;
}

int sjf_add_monitors(sjf_engine* e, int comp, const double* xyz, int n) {
    if (!e || (!xyz && n > 0) || n < 0) return SJF_E_ARG;
    if (comp < 0 || comp > 5) return fail(e, SJF_E_ARG, "bad component");
    if (e->nsamp > 0) return fail(e, SJF_E_STATE, "monitors must be added before sampling starts");
    for (int p = 0; p < n; ++p) {
        Monitor m;
        m.comp = comp;
        trilinear(e, comp, xyz + 3 * p, m.idx, m.w);
        e->mon.push_back(m);
    }
    dev_free(e->d_samples);
    e->samp_cap = 0;
    e->version++;
    return SJF_OK;
}

int sjf_set_save_span(sjf_engine* e, int span) {
    if (!e) return SJF_E_ARG;
    const int s = span > 0 ? span : 1;
    if (e->nsamp > 0 && s != e->save_span) return fail(e, SJF_E_STATE, "save span cannot change once sampling started");
    e->save_span = s;
    e->version++;
    return SJF_OK;
}

int sjf_read_monitors(sjf_engine* e, double* out, size_t cap, long* n_samples) {
    if (!e || !n_samples) return SJF_E_ARG;
    *n_samples = e->nsamp;
    const long npt = (long)e->mon.size();
    const long tot = e->nsamp * npt;
    if (!out || tot == 0) return SJF_OK;
    if ((size_t)(2 * tot) > cap) return fail(e, SJF_E_ARG, "output buffer too small");
    if (int rc = sync_engine(e)) return rc;
    std::vector<double> tmp(tot);
    int rc = d2h(e, tmp.data(), e->d_samples, sizeof(double) * tot);
    if (rc) return rc;
    for (long q = 0; q < tot; ++q) {
        out[2 * q] = tmp[q];
        out[2 * q + 1] = 0.0;
    }
    return SJF_OK;
}

int sjf_get_field(sjf_engine* e, int comp, const double xyz[3], double out[2]) {
    if (!e || !xyz || !out || comp < 0 || comp > 5) return SJF_E_ARG;
    if (int rc = sync_engine(e)) return rc;
    long idx[8];
    double w[8];
    trilinear(e, comp, xyz, idx, w);
    sjf::GatherPoint g;
    for (int q = 0; q < 8; ++q) {
        g.idx[q] = idx[q] < 0 ? -1 : sjf::field_index(idx[q], comp, (long)e->g.ny * e->g.nz);
        g.w[q] = w[q];
    }
    double v = 0;
    const int rc = read_out(e, &v, 1, sizeof(v), [&](long, long, void* p) {
        if (e->prec == 4)
            hipLaunchKernelGGL((sjf::k_read_point<float>), dim3(1), dim3(64), 0, e->stream, (const float*)field_set(e), g,
                               (double*)p);
        else
            hipLaunchKernelGGL((sjf::k_read_point<double>), dim3(1), dim3(64), 0, e->stream, (const double*)field_set(e),
                               g, (double*)p);
    });
    if (rc) return rc;
    out[0] = v;
    out[1] = 0.0;
    return SJF_OK;
}

int sjf_add_dft(sjf_engine* e, const int lo[3], const int hi[3], int comp_mask, const double* freqs, int nf,
                int* id) {
    if (!e || !lo || !hi || !freqs || !id) return SJF_E_ARG;
    if (nf < 1 || nf > SJF_MAX_DFT_FREQS) return fail(e, SJF_E_ARG, "nf must be in [1, 64]");
    if (comp_mask <= 0 || comp_mask >= 64) return fail(e, SJF_E_ARG, "comp_mask must select components 0..5");
    const int n[3] = {e->g.nx, e->g.ny, e->g.nz};
    Dft d;
    d.ncell = 1;
    for (int q = 0; q < 3; ++q) {
        if (lo[q] < 0 || hi[q] > n[q] || hi[q] <= lo[q]) return fail(e, SJF_E_ARG, "DFT box outside grid");
        d.lo[q] = lo[q];
        d.hi[q] = hi[q];
        d.ncell *= hi[q] - lo[q];
    }
    d.mask = comp_mask;
    d.freqs.assign(freqs, freqs + nf);
    d.ncomp = 0;
    for (int c = 0; c < 6; ++c)
        if (comp_mask >> c & 1) d.comps[d.ncomp++] = c;
    if (int rc = sync_engine(e)) return rc;
    const size_t bytes = sizeof(double2) * d.ncomp * nf * d.ncell;
    int rc = dev_alloc(e, (void**)&d.acc, bytes);
    if (!rc) rc = dev_alloc(e, (void**)&d.cmp, bytes);
    if (!rc) rc = dev_alloc(e, (void**)&d.d_freq, sizeof(double) * nf);
    if (!rc) rc = h2d(e, d.d_freq, d.freqs.data(), sizeof(double) * nf);
    if (rc) {
        dev_free(d.acc);
        dev_free(d.cmp);
        dev_free(d.d_freq);
        return rc;
    }
    e->dft.push_back(d);
    *id = (int)e->dft.size() - 1;
    e->version++;
    return SJF_OK;
}

int sjf_read_dft(sjf_engine* e, int id, double* out, size_t cap) {
    if (!e || !out || id < 0 || id >= (int)e->dft.size()) return SJF_E_ARG;
    const Dft& d = e->dft[id];
    const long n = (long)d.ncomp * (long)d.freqs.size() * d.ncell;
    if ((size_t)(2 * n) > cap) return fail(e, SJF_E_ARG, "output buffer too small");
    if (int rc = sync_engine(e)) return rc;
    return read_out(e, out, n, sizeof(double2), [&](long first, long count, void* p) {
        hipLaunchKernelGGL(sjf::k_read_dft, dim3((unsigned)std::min(1024L, (count + 255) / 256)), dim3(256), 0, e->stream,
                           (const double2*)d.acc + first, (const double2*)d.cmp + first, count, (double2*)p);
    });
}

int sjf_dft_flux(sjf_engine* e, int id, int axis, double* flux, size_t cap) {
    FluxPlan fp;
    if (int rc = flux_plan(e, id, axis, flux, cap, &fp)) return rc;
    if (int rc = sync_engine(e)) return rc;
    double* buf = nullptr;
    if (int rc = dev_alloc(e, (void**)&buf, sizeof(double) * fp.scratch_doubles())) return rc;
    int rc = flux_run(e, fp, buf, flux);
    dev_free(buf);
    return rc;
}

int sjf_dft_flux_noalloc(sjf_engine* e, int id, int axis, double* flux, size_t cap) {
    FluxPlan fp;
    if (int rc = flux_plan(e, id, axis, flux, cap, &fp)) return rc;
    if (fp.scratch_doubles() > (long)kFluxScratchDoubles)
        return fail(e, SJF_E_ARG, "flux needs " + std::to_string(fp.scratch_doubles()) +
                                      " doubles of scratch; the allocation-free buffer holds " +
                                      std::to_string(kFluxScratchDoubles));
    double* buf = scratch_on(e->g.device);
    if (!buf) return fail(e, SJF_E_STATE, "no scratch address for this device (sjf_create sets it up)");
    if (int rc = sync_engine(e)) return rc;
    return flux_run(e, fp, buf, flux);
}

int sjf_step(sjf_engine* e, long n) {
    if (!e || n < 0) return SJF_E_ARG;
    if (e->batch) return fail(e, SJF_E_STATE, "engine is stepped by its batch");
    HIPCHK(e, hipSetDevice(e->g.device));
    return run_set(own_set(e), n);
}

int sjf_reserve_steps(sjf_engine* e, long n) {
    if (!e || n < 0) return SJF_E_ARG;
    if (e->batch) return fail(e, SJF_E_STATE, "engine is stepped by its batch");
    HIPCHK(e, hipSetDevice(e->g.device));
    return prepare_set(own_set(e), n);
}

int sjf_synchronize(sjf_engine* e) {
    if (!e) return SJF_E_ARG;
    return sync_engine(e);
}

int sjf_set_graph(sjf_engine* e, int chunk) {
    if (!e || chunk < 0) return SJF_E_ARG;
    e->graph_chunk = chunk;
    e->version++;
    return SJF_OK;
}

int sjf_timed_steps(sjf_engine* e, long n, double* ms_total, double* ms_kernel_mean) {
    if (!e || n < 1 || !ms_total || !ms_kernel_mean) return SJF_E_ARG;
    if (e->batch) return fail(e, SJF_E_STATE, "engine is stepped by its batch");
    HIPCHK(e, hipSetDevice(e->g.device));
    return timed_set(own_set(e), n, ms_total, ms_kernel_mean);
}

int sjf_read_field(sjf_engine* e, int comp, double* out) {
    if (!e || !out || comp < 0 || comp > 5) return SJF_E_ARG;
    if (int rc = sync_engine(e)) return rc;
    return e->prec == 4 ? read_component<float>(e, comp, out) : read_component<double>(e, comp, out);
}

int sjf_read_field_box(sjf_engine* e, int comp, const int lo[3], const int hi[3], double* out) {
    if (!e || !lo || !hi || comp < 0 || comp > 5) return SJF_E_ARG;
    const int n[3] = {e->g.nx, e->g.ny, e->g.nz};
    for (int d = 0; d < 3; ++d)
        if (lo[d] < 0 || hi[d] > n[d] || lo[d] > hi[d]) return fail(e, SJF_E_ARG, "field box outside the grid");
    if (lo[0] == hi[0] || lo[1] == hi[1] || lo[2] == hi[2]) return SJF_OK;  // empty box: nothing to copy
    if (!out) return SJF_E_ARG;
    if (int rc = sync_engine(e)) return rc;
    return e->prec == 4 ? read_component_box<float>(e, comp, lo, hi, out)
                        : read_component_box<double>(e, comp, lo, hi, out);
}

int sjf_write_field(sjf_engine* e, int comp, const double* in) {
    if (!e || !in || comp < 0 || comp > 5) return SJF_E_ARG;
    if (int rc = sync_engine(e)) return rc;
    return e->prec == 4 ? write_component<float>(e, comp, in) : write_component<double>(e, comp, in);
}

int sjf_step_bytes(const sjf_engine* e, double* bytes) {
    if (!e || !bytes) return SJF_E_ARG;
    *bytes = engine_step_bytes(e);
    return SJF_OK;
}

int sjf_launch_info(const sjf_engine* e, int* form, int* ty, int* xchunk, int* threads, int* groups) {
    if (!e) return SJF_E_ARG;
    if (form) *form = e->form;
    if (ty) *ty = e->ty;
    if (xchunk) *xchunk = e->xc;
    if (threads) *threads = block_threads(e);
    if (groups) *groups = tiles_of(e, e->ty, e->xc);
    return SJF_OK;
}

int sjf_set_zsegment(sjf_engine* e, int cells) {
    if (!e) return SJF_E_ARG;
    if (cells != 0 && (cells < 64 || cells > 1024 || cells % 64 != 0))
        return fail(e, SJF_E_ARG, "z segment must be 0 or a multiple of 64 from 64 to 1024");
    if (cells > 0 && cells < e->g.nz && e->g.periodic[2])
        return fail(e, SJF_E_ARG, "z passes need a non-periodic z axis");
    e->zseg = cells;
    choose_tile(e);
    e->version++;
    return SJF_OK;
}

int sjf_set_tile(sjf_engine* e, int form, int ty, int xchunk) {
    if (!e) return SJF_E_ARG;
    if (form == SJF_TILE_REGISTER_ROWS) {
        if (ty != 1 && ty != 2 && ty != 4) return fail(e, SJF_E_ARG, "rows per thread must be 1, 2 or 4");
    } else if (form == SJF_TILE_THREAD_ROWS) {
        if (!thread_rows_fit(e, ty))
            return fail(e, SJF_E_ARG, "row-of-threads tile needs (rows + 1) * nz <= 1024 and 4-byte-addressable arrays");
    } else {
        return fail(e, SJF_E_ARG, "unknown tile form");
    }
    if (xchunk < 1) return fail(e, SJF_E_ARG, "xchunk must be >= 1");
    e->form = form;
    e->ty = ty;
    e->xc = std::min(xchunk, e->g.nx);
    e->tile_set = true;
    e->version++;
    return SJF_OK;
}

// ---- batches --------------------------------------------------------------------------------

int sjf_batch_create(sjf_engine* const* engines, int n, sjf_batch** out) {
    if (!engines || n < 1 || !out) {
        g_create_error = "null argument";
        return SJF_E_ARG;
    }
    *out = nullptr;
    sjf_engine* e0 = engines[0];
    if (!e0) return SJF_E_ARG;
    long span = -1;
    for (int i = 0; i < n; ++i) {
        sjf_engine* e = engines[i];
        if (!e) return SJF_E_ARG;
        std::string why;
        if (e->batch) why = "engine already belongs to a batch";
        else if (e->g.device != e0->g.device) why = "engines of a batch must share a device";
        else if (e->prec != e0->prec) why = "engines of a batch must share a precision";
        else if (e->step != e0->step) why = "engines of a batch must be at the same step";
        else if (!e->mon.empty()) {
            if (span >= 0 && span != e->save_span) why = "engines of a batch must share a save span";
            span = e->save_span;
        }
        for (int j = 0; j < i && why.empty(); ++j)
            if (engines[j] == e) why = "engine listed twice";
        if (!why.empty()) {
            g_create_error = why;
            return SJF_E_ARG;
        }
    }
    if (hipSetDevice(e0->g.device) != hipSuccess) {
        g_create_error = "hipSetDevice failed";
        return SJF_E_HIP;
    }
    for (int i = 0; i < n; ++i)
        if (hipStreamSynchronize(engines[i]->stream) != hipSuccess) {
            g_create_error = "stream synchronisation failed";
            return SJF_E_HIP;
        }
    sjf_batch* b = new sjf_batch();
    LaunchSet* s = new LaunchSet();
    if (hipStreamCreateWithFlags(&s->stream, hipStreamNonBlocking) != hipSuccess) {
        delete s;
        delete b;
        g_create_error = "hipStreamCreate failed";
        return SJF_E_HIP;
    }
    s->own_stream = true;
    s->prec = e0->prec;
    s->ty = 1;
    s->form = batch_form(engines, n);
    s->xc = s->form == SJF_TILE_THREAD_ROWS ? kBatchRowsChunk : 16;
    for (int i = 0; i < n; ++i) {
        s->eng.push_back(engines[i]);
        engines[i]->batch = b;
    }
    b->set = s;
    *out = b;
    return SJF_OK;
}

int sjf_batch_set_tile(sjf_batch* b, int form, int xchunk) {
    if (!b || xchunk < 0) return SJF_E_ARG;
    LaunchSet* s = b->set;
    if (form == SJF_TILE_THREAD_ROWS) {
        for (sjf_engine* e : s->eng)
            if (!thread_rows_fit(e, default_thread_rows(e))) {
                b->err = "an instance does not fit the row-of-threads tile";
                return SJF_E_ARG;
            }
    } else if (form != SJF_TILE_REGISTER_ROWS) {
        b->err = "unknown tile form";
        return SJF_E_ARG;
    }
    s->form = form;
    s->ty = 1;
    s->xc = xchunk;
    s->tile_set = true;
    s->built = false;
    return SJF_OK;
}

int sjf_batch_step(sjf_batch* b, long n) {
    if (!b || n < 0) return SJF_E_ARG;
    LaunchSet* s = b->set;
    if (hipSetDevice(s->eng[0]->g.device) != hipSuccess) return SJF_E_HIP;
    const int rc = run_set(s, n);
    if (rc) b->err = s->eng[0]->err;
    return rc;
}

int sjf_batch_reserve_steps(sjf_batch* b, long n) {
    if (!b || n < 0) return SJF_E_ARG;
    LaunchSet* s = b->set;
    if (hipSetDevice(s->eng[0]->g.device) != hipSuccess) return SJF_E_HIP;
    const int rc = prepare_set(s, n);
    if (rc) b->err = s->eng[0]->err;
    return rc;
}

int sjf_batch_timed_steps(sjf_batch* b, long n, double* ms_total, double* ms_kernel_mean) {
    if (!b || n < 1 || !ms_total || !ms_kernel_mean) return SJF_E_ARG;
    LaunchSet* s = b->set;
    if (hipSetDevice(s->eng[0]->g.device) != hipSuccess) return SJF_E_HIP;
    const int rc = timed_set(s, n, ms_total, ms_kernel_mean);
    if (rc) b->err = s->eng[0]->err;
    return rc;
}

int sjf_batch_synchronize(sjf_batch* b) {
    if (!b) return SJF_E_ARG;
    if (hipStreamSynchronize(b->set->stream) != hipSuccess) return SJF_E_HIP;
    return SJF_OK;
}

int sjf_batch_info(const sjf_batch* b, long* cells, double* bytes_per_step) {
    if (!b) return SJF_E_ARG;
    long c = 0;
    double by = 0;
    for (const sjf_engine* e : b->set->eng) {
        c += e->N;
        by += engine_step_bytes(e);
    }
    if (cells) *cells = c;
    if (bytes_per_step) *bytes_per_step = by;
    return SJF_OK;
}

int sjf_batch_launch_info(const sjf_batch* b, int* threads, int* groups) {
    if (!b) return SJF_E_ARG;
    if (!b->set->built) return SJF_E_STATE;
    if (threads) *threads = b->set->block;
    if (groups) *groups = b->set->ntiles;
    return SJF_OK;
}

int sjf_batch_adjoint_run(sjf_batch* b, long nsteps, int checkpoint_every, const int* gaps, double* J,
                          double* const* grads, const size_t* caps) {
    if (!b || nsteps < 1 || checkpoint_every < 0 || !gaps || !J || !grads || !caps) return SJF_E_ARG;
    for (const sjf_engine* e : b->set->eng)
        if (!e->emap_h.empty()) {
            b->err = "adjoint runs take the LUT's eps_inf (no eps maps)";
            return SJF_E_UNSUPPORTED;
        }
    LaunchSet* s = b->set;
    sjf_engine* e0 = s->eng[0];
    const int n = (int)s->eng.size();
    std::vector<long> q(n, 0), nd(n, 0);
    std::string why;
    for (int i = 0; i < n && why.empty(); ++i) {
        const sjf_engine* e = s->eng[i];
        const int ext[3] = {e->g.nx, e->g.ny, e->g.nz};
        if (e->step != 0) why = "the adjoint run starts from step 0";
        else if (e->deps_h.empty()) why = "an engine has no design region (sjf_set_design_eps)";
        else if (e->g.nz != e0->g.nz) why = "engines of a batched adjoint run must share nz";
        else if (e->g.nz > 1024) why = "the reverse step spans the z line: nz <= 1024";
        else if (np_variant_of(e->maxp, e->uniform) != np_variant_of(e0->maxp, e0->uniform))
            why = "engines of a batched adjoint run must share the pole-slot variant";
        else if (!grads[i]) why = "null gradient buffer";
        for (int d = 0; d < 3 && why.empty(); ++d)
            if (gaps[3 * i + d] < 0 || gaps[3 * i + d] >= ext[d]) why = "objective cell outside the grid";
        if (why.empty()) {
            nd[i] = (long)e->deps_h.size();
            if (caps[i] < (size_t)nd[i]) why = "gradient buffer smaller than the design region";
            q[i] = cell_index(e, gaps[3 * i], gaps[3 * i + 1], gaps[3 * i + 2]);
        }
    }
    if (!why.empty()) {
        b->err = why;
        return SJF_E_ARG;
    }
    if (hipSetDevice(e0->g.device) != hipSuccess) return SJF_E_HIP;
    double ms = 0;
    int th = 0, gr = 0;
    const int rc = s->prec == 4
                       ? batch_adjoint_run_t<float>(s, nsteps, checkpoint_every, q.data(), nd.data(), J, grads, &ms,
                                                    &th, &gr)
                       : batch_adjoint_run_t<double>(s, nsteps, checkpoint_every, q.data(), nd.data(), J, grads, &ms,
                                                     &th, &gr);
    if (rc) {
        b->err = e0->err;
        return rc;
    }
    b->adj_ms = ms;
    b->adj_threads = th;
    b->adj_groups = gr;
    return SJF_OK;
}

int sjf_batch_adjoint_kernel_info(const sjf_batch* b, double* ms_mean, int* threads, int* groups) {
    if (!b || !ms_mean) return SJF_E_ARG;
    if (b->adj_groups == 0) return SJF_E_STATE;
    *ms_mean = b->adj_ms;
    if (threads) *threads = b->adj_threads;
    if (groups) *groups = b->adj_groups;
    return SJF_OK;
}

const char* sjf_batch_last_error(const sjf_batch* b) { return b ? b->err.c_str() : g_create_error.c_str(); }

int sjf_batch_destroy(sjf_batch* b) {
    if (!b) return SJF_E_ARG;
    LaunchSet* s = b->set;
    (void)hipSetDevice(s->eng[0]->g.device);
    (void)hipStreamSynchronize(s->stream);
    for (sjf_engine* e : s->eng) e->batch = nullptr;
    destroy_set(s);
    delete b;
    return SJF_OK;
}

// ---- measurement probe ------------------------------------------------------------------------

int sjf_copy_probe(int device, size_t bytes, int iters, double* gbs) {
    if (!gbs || bytes < 16 || iters < 1) return SJF_E_ARG;
    if (hipSetDevice(device) != hipSuccess) return SJF_E_HIP;
    const long n = (long)(bytes / 16);
    float4 *a = nullptr, *b = nullptr;
    if (device_malloc((void**)&a, n * 16) != hipSuccess) return SJF_E_NOMEM;
    if (device_malloc((void**)&b, n * 16) != hipSuccess) {
        (void)hipFree(a);
        return SJF_E_NOMEM;
    }
    (void)hipMemset(a, 0, n * 16);
    (void)hipMemset(b, 0, n * 16);
    hipEvent_t t0, t1;
    (void)hipEventCreate(&t0);
    (void)hipEventCreate(&t1);
    const unsigned blocks = (unsigned)((n + 255) / 256);
    hipLaunchKernelGGL(sjf::k_copy, dim3(blocks), dim3(256), 0, 0, a, b, n);
    (void)hipEventRecord(t0, 0);
    for (int it = 0; it < iters; ++it) hipLaunchKernelGGL(sjf::k_copy, dim3(blocks), dim3(256), 0, 0, a, b, n);
    (void)hipEventRecord(t1, 0);
    const hipError_t st = hipEventSynchronize(t1);
    float ms = 0;
    (void)hipEventElapsedTime(&ms, t0, t1);
    (void)hipEventDestroy(t0);
    (void)hipEventDestroy(t1);
    (void)hipFree(a);
    (void)hipFree(b);
    if (st != hipSuccess) return SJF_E_HIP;
    *gbs = 2.0 * n * 16 * iters / (ms * 1e-3) / 1e9;
    return SJF_OK;
}

}  // extern "C"
