// sjf_kernels.h -- gfx950 kernels of the FDTD engine (device code only).
//
// Hot path: one fused launch per time step (k_step) that performs, for every cell,
//   H^{n+1/2} = H^{n-1/2} - (dt/dx) (dE + psi_H)                       (Yee curl, CPML)
//   Q_k^{n+1} = alpha_k Q_k^n + beta_k P_k^n + c3_k E^n, P_k^{n+1} = P_k^n + Q_k^{n+1}
//   E^{n+1}   = E^n + inv_eps ((dt/dx) (dH + psi_E) - sum_k Q_k^{n+1})
// This is the E-direct form of meep's D/E split (src/disp.cpp:740 fields.step(): B, H, D,
// polarisation, E): with D = eps_inf E + sum P, D^{n+1} - D^n = dt curl H, and
// Q = P^{n+1} - P^n the textbook Lorentz/Drude recurrence becomes the (P, Q) pair above,
// which needs no D array and, for Drude poles, no P array.  In FP32 a Lorentz pole keeps P^n
// and P^{n-1} (Q^n = P^n - P^{n-1}) in two slots whose roles alternate with the step parity,
// so each step reads both and writes only P^{n+1} over P^{n-1}: 3 values moved per pole and
// component instead of 4 for a stored (P, Q).  FP64 keeps (P, Q): its tile is held to 3
// wavefronts per SIMD by its registers and runs faster without the role selects.  A Drude pole
// keeps Q^n alone (2 values).
//
// Layout in HBM: each component is a dense nx*ny*nz array, z fastest.  E and H and the H
// auxiliaries are double-buffered (read buffer 0, write buffer 1, swapped every step) because
// neighbouring workgroups recompute one halo row of H from the old state; polarisation state
// and the E auxiliaries are only touched by the owning thread and are updated in place.
//
// Work decomposition (MI355X: 64-wide wavefronts, 8 XCDs with private L2):
//   * one workgroup spans the whole z line (blockDim = nz rounded up to 64, <= 1024), so the
//     z neighbours of H come from LDS and the z halo disappears;
//   * each thread owns TY consecutive y rows (register blocking) and recomputes H on one
//     extra row below them (the y halo);
//   * the workgroup marches along x over a chunk of planes, carrying E^n of the next plane
//     and H^{n+1/2} of the previous plane in registers (no x halo except one plane per chunk);
//   * workgroup ids are remapped so that consecutive tiles land on the same XCD and share
//     halo rows in that XCD's L2.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace sjf {

constexpr int kMaxPoles = 4;
// Lorentz poles stored as (P^n, P^{n-1}) with alternating roles (FP32) or as (P, Q) (FP64)
template <typename T>
constexpr bool kPolePair = sizeof(T) == 4;
constexpr int kDesignMat = 255;
constexpr int kMaxDftFreqs = 64;

// recurrence coefficients of one pole; lor: 1 for a Lorentz pole, 0 for a Drude one (and unused slots)
template <typename T>
struct __align__(16) PoleCoef {
    T alpha, beta, c3, lor;
};

// One entry per material and, last, one of zeros that design voxels index.
template <typename T>
struct __align__(16) MatLut {
    int np;
    int lorentz_mask;
    T inv_eps;
    PoleCoef<T> pole[kMaxPoles];
};

// bytes the material table takes in LDS
template <typename T>
__host__ __device__ constexpr size_t lut_lds_bytes(int nmat) { return sizeof(MatLut<T>) * (nmat + 1); }

// Kernel arguments of the fused step.  Few base pointers on purpose: the component, pole-slot
// and PML-segment arrays are addressed as offsets from them, so the whole argument block stays
// in scalar registers (a per-array pointer table overflows the SGPR file and spills into
// vector-register lanes).
template <typename T>
struct StepArgs {
    int nx, ny, nz;
    int px, py, pz;
    int nty, xc;
    int rt;       // row-of-threads form: thread rows per workgroup (owned rows + 1 halo row)
    int zseg;     // register form: z cells per pass of a workgroup (nz: one pass)
    long N;       // cells
    T cdt;        // dt / dx
    T* F[2];              // field sets [x][Ex Ey Ez Hx Hy Hz][y][z]; step n reads F[n&1], writes F[~n&1]
    long* d_step;         // the engine's step counter and its shadow
    int uniform;  // 1: single non-dispersive material, no material word read
    int nmat;     // materials; the id of design voxels in the words
    const uint32_t* matw;
    const uint32_t* seg;  // one code per 64 cells of a z line (k_words), [x][y][(nz + 63) / 64]
    const MatLut<T>* lut;
    T* Q;     // [x][slot * 3 + comp][y][z]
    T* P;     // [x][slot * 3 + comp][y][z] (Lorentz slots)
    int nqp;  // polarisation planes per x plane (3 * slots)
    int pml_on[3], plo[3], phi[3];
    long S[3];      // PML slab sizes (cells) per axis
    T* psi[3];      // per axis [3][S][2]: E auxiliary pair, H pairs A and B (two components each);
                    // step n reads pair A and writes pair B when n is even, the reverse when odd
    const T* coef;  // PML tables: for axis d at coff[d]: bE[n], aE[n], bH[n], aH[n]
    int coff[3];
    int dlo[3], dhi[3];
    const T* dinv;
    const T* emap;  // per-cell 1/eps_inf [x][Ex Ey Ez][y][z] (sjf_set_eps_maps), or null: the LUT's
};

#define GLOBAL __attribute__((address_space(1)))
// memory no kernel writes while it is read: uniform reads go through the scalar cache
#define CONST __attribute__((address_space(4)))

__device__ __forceinline__ int wrap_or_ghost(int c, int n, int periodic) {
    if (c >= 0 && c < n) return c;
    if (!periodic) return -1;
    // any number of periods away: a tile's rows (and the planes ahead of its march) can lie
    // more than one period past the edge of an axis shorter than the tile
    const int m = c % n;
    return m < 0 ? m + n : m;
}

// the same for c in [-1, n]
__device__ __forceinline__ int wrap_one(int c, int n, int periodic) {
    return c < 0 ? (periodic ? n - 1 : -1) : c < n ? c : periodic ? 0 : -1;
}
// c in [0, ...): past the end of a periodic axis of any length back into it, else unchanged
__device__ __forceinline__ int wrap_up(int c, int n, int periodic) { return periodic && c >= n ? 0 : c; }

template <typename T>
__device__ __forceinline__ bool in_pml(const StepArgs<T>& a, int d, int c, int n) {
    return a.pml_on[d] && (c < a.plo[d] || c >= n - a.phi[d]);
}

// The sums of the update, with the fused products spelled out: every kernel form and every place of
// a plane's H (its own, the halo's, a chunk's first plane) then rounds alike, whatever else the
// compiler fuses.
__device__ __forceinline__ float fma_(float a, float b, float c) { return __builtin_fmaf(a, b, c); }
__device__ __forceinline__ double fma_(double a, double b, double c) { return __builtin_fma(a, b, c); }
// the updated CPML auxiliary b psi + c d of a term d, which adds it: along x and z, and along y (one
// product is rounded, the other is not; which one is a choice that later sums must repeat)
template <typename T>
__device__ __forceinline__ T aux_next(T d, T b, T c, T psi) { return fma_(c, d, b * psi); }
template <typename T>
__device__ __forceinline__ T aux_next_y(T d, T b, T c, T psi) { return fma_(b, psi, c * d); }
// H - cdt (x - y)
template <typename T>
__device__ __forceinline__ T h_next(T h, T cdt, T x, T y) { return fma_(-cdt, x - y, h); }
// E + inv (cdt curl - sum of Q^{n+1})
template <typename T>
__device__ __forceinline__ T e_next(T e, T inv, T cdt, T curl, T sq) { return fma_(inv, fma_(cdt, curl, -sq), e); }

// LDS-scoped workgroup barrier: orders only the LDS exchange, so global loads issued before it
// (next-plane prefetch) and global stores stay in flight across it.
__device__ __forceinline__ void lds_barrier() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// ---- raw buffer access ----------------------------------------------------------------------
// A raw buffer descriptor over p (no stride, the gfx9 dword data format) whose range is the first
// 2 GiB from p.  A load or store through it names the descriptor (four scalar registers), a 32-bit
// per-lane offset (one vector register) and a 32-bit wave-uniform offset (one scalar register), so
// an access needs no vector address arithmetic and a loop-invariant lane offset stays a single
// register.  A lane whose offset is kOOB lies outside the range: its load returns 0 and its store
// is dropped without a memory access, which predicates single lanes without branching.  Callers
// keep every in-range access (lane plus uniform offset) below 2 GiB from the descriptor base.
typedef __amdgpu_buffer_rsrc_t Rsrc;
typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));
constexpr uint32_t kOOB = 0x80000000u;
__device__ __forceinline__ Rsrc rsrc(const void* p) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), (short)0, (int)0x80000000u, 0x00020000);
}
// the same over nothing unless `need` (uniform): loads return 0 without a memory access
__device__ __forceinline__ Rsrc rsrc(const void* p, bool need) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), (short)0, need ? (int)0x80000000u : 0, 0x00020000);
}
template <typename T>
__device__ __forceinline__ T bld(Rsrc r, uint32_t v, uint32_t s);
template <>
__device__ __forceinline__ float bld<float>(Rsrc r, uint32_t v, uint32_t s) {
    return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, (int)v, (int)s, 0));
}
template <>
__device__ __forceinline__ double bld<double>(Rsrc r, uint32_t v, uint32_t s) {
    return __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(r, (int)v, (int)s, 0));
}
template <>
__device__ __forceinline__ uint32_t bld<uint32_t>(Rsrc r, uint32_t v, uint32_t s) {
    return __builtin_amdgcn_raw_buffer_load_b32(r, (int)v, (int)s, 0);
}
// NT: the non-temporal cache policy (a hint that the line will not be read again soon).  A step
// over more data than the caches hold cannot find its writes there at the next step, and the
// hint keeps the written lines from displacing the y-halo rows that neighbouring workgroups
// read again.
template <bool NT = false>
__device__ __forceinline__ void bst(Rsrc r, uint32_t v, uint32_t s, float x) {
    __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(uint32_t, x), r, (int)v, (int)s, NT ? 2 : 0);
}
template <bool NT = false>
__device__ __forceinline__ void bst(Rsrc r, uint32_t v, uint32_t s, double x) {
    __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(u32x2, x), r, (int)v, (int)s, NT ? 2 : 0);
}
// two consecutive values
template <typename T>
using Pair2 = T __attribute__((ext_vector_type(2)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
template <typename T>
__device__ __forceinline__ Pair2<T> bld2(Rsrc r, uint32_t v, uint32_t s) {
    if constexpr (sizeof(T) == 4) return __builtin_bit_cast(Pair2<T>, __builtin_amdgcn_raw_buffer_load_b64(r, (int)v, (int)s, 0));
    else return __builtin_bit_cast(Pair2<T>, __builtin_amdgcn_raw_buffer_load_b128(r, (int)v, (int)s, 0));
}
// (FP64: two stores.  One of 16 bytes with a scalar offset stored what the next instruction wrote to
// its data registers: the compiler takes this form to need no wait state there, and on gfx950 pairs
// of the x layers came out wrong under load.)
template <bool NT = false, typename P>
__device__ __forceinline__ void bst2(Rsrc r, uint32_t v, uint32_t s, P x) {
    if constexpr (sizeof(P) == 8) {
        __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(u32x2, x), r, (int)v, (int)s, NT ? 2 : 0);
    } else {
        const u32x4 w = __builtin_bit_cast(u32x4, x);
        __builtin_amdgcn_raw_buffer_store_b64(u32x2{w.x, w.y}, r, (int)v, (int)s, NT ? 2 : 0);
        __builtin_amdgcn_raw_buffer_store_b64(u32x2{w.z, w.w}, r, (int)v, (int)s + 8, NT ? 2 : 0);
    }
}
// the lane offset of a pair from that of a value (kOOB stays out of range)
__device__ __forceinline__ uint32_t two(uint32_t o) { return o == kOOB ? kOOB : 2u * o; }
// true in every lane of the wavefront when p holds in at least one active lane (wave-uniform)
__device__ __forceinline__ bool wave_any(bool p) { return __builtin_amdgcn_ballot_w64(p) != 0; }

// A register copy the compiler does not look through.  Where a value moves on to a register that an
// earlier one leaves (plane i + 1 becoming plane i), it would otherwise rename instead and copy the
// next plane's loads at the end of the loop, waiting for them.
__device__ __forceinline__ float reg_copy(float x) {
    float y;
    asm("v_mov_b32 %0, %1" : "=v"(y) : "v"(x));
    return y;
}
__device__ __forceinline__ uint32_t reg_copy(uint32_t x) {
    uint32_t y;
    asm("v_mov_b32 %0, %1" : "=v"(y) : "v"(x));
    return y;
}
__device__ __forceinline__ double reg_copy(double x) {
    double y;
    asm("v_mov_b64 %0, %1" : "=v"(y) : "v"(x));
    return y;
}

// Computes x here: keeps the compiler from sinking what x is made of past the loads that follow, into
// the registers it still occupies.
__device__ __forceinline__ void pin(float& x) { asm volatile("" : "+v"(x)); }
__device__ __forceinline__ void pin(double& x) { asm volatile("" : "+v"(x)); }

// Field and polarisation layout: x planes of components, [x][comp][y][z] for a field set (six
// components) and [x][slot * 3 + comp][y][z] for Q and P.  One x plane of a set is contiguous,
// so a kernel addresses a plane through one descriptor and a component by a 32-bit offset.
__host__ __device__ __forceinline__ long field_index(long q, int c, long nyz) { return q + (5 * (q / nyz) + c) * nyz; }

// the material table (with its last entry of zeros) into LDS
template <typename T>
__device__ __forceinline__ void copy_lut(const StepArgs<T>& a, MatLut<T>* lds) {
    GLOBAL const u32x4* src = (GLOBAL const u32x4*)a.lut;
    u32x4* dst = reinterpret_cast<u32x4*>(lds);
    const int n = (int)(sizeof(MatLut<T>) / 16) * (a.nmat + 1);
    for (int q = threadIdx.x; q < n; q += blockDim.x) dst[q] = src[q];
}

// ---- material segments ----------------------------------------------------------------------
// What the 64 cells of one z segment run.  Segments of one material for all three E components
// carry its id (bits 0-7) and pole count (8-10); other segments the flag kSegMixed, the largest pole
// count of a cell, and kSegDesign when a design voxel is among them.  kSegSpecial: mixed or with
// poles, so that the material table is needed.
constexpr uint32_t kSegMixed = 0x80000000u, kSegDesign = 0x40000000u, kSegSpecial = 0x20000000u;
// In the words themselves, above the three ids: the largest pole count of the cell's materials, and
// whether a component is a design voxel.
constexpr uint32_t kWordDesign = 0x08000000u;
__device__ __forceinline__ int word_poles(uint32_t w) { return (int)((w >> 24) & 7); }
__device__ __forceinline__ int seg_material(uint32_t code) { return (int)(code & 0xff); }
__device__ __forceinline__ int seg_poles(uint32_t code) { return (int)((code >> 8) & 7); }

// ---- material words ------------------------------------------------------------------------------

// Cells outside [lo, hi) of some axis lie in a PML slab and take material twin[m] for m.
struct WordMap {
    int lo[3], hi[3];
    unsigned char twin[256];
};

// The words and segment codes the kernels run, from the given words: the PML twins, design ids
// (kDesignMat) as nmat (the table's entry of zeros), the marks above.  One wavefront per segment;
// count: pole slots of all segments, and poles over all cells and components.  Bound by memory: 256 x
// 256 x 128 cells 0.03 ms (on the host, three loops over the cells and a second upload: 30 ms).
template <typename T>
__global__ void __launch_bounds__(256) k_words(const uint32_t* __restrict__ given, uint32_t* __restrict__ matw,
                                               uint32_t* __restrict__ seg, const MatLut<T>* __restrict__ lut, int nx,
                                               int ny, int nz, int nmat, const WordMap map,
                                               unsigned long long* __restrict__ count) {
    const int nseg = (nz + 63) >> 6, lane = threadIdx.x & 63;
    const long n = (long)nx * ny * nseg;
    unsigned long long slots = 0, poles = 0;
    for (long q = (long)blockIdx.x * 4 + (threadIdx.x >> 6); q < n; q += (long)gridDim.x * 4) {
        const long row = q / nseg;
        const int k = (int)(q - row * nseg) * 64 + lane, i = (int)(row / ny), j = (int)(row - (long)i * ny);
        const bool in = k < nz;
        const bool slab = i < map.lo[0] || i >= map.hi[0] || j < map.lo[1] || j >= map.hi[1] || k < map.lo[2] ||
                          k >= map.hi[2];
        const uint32_t w = in ? given[row * nz + k] : 0u;
        bool des = false;
        int np = 0;
        uint32_t out = 0u;  // the three ids
        for (int c = 0; c < 3; ++c) {
            int m = (w >> (8 * c)) & 0xff;
            const bool d = in && m == kDesignMat;
            if (slab) m = map.twin[m];
            m = d ? nmat : min(m, nmat);
            des = des || d;
            const int p = in ? lut[m].np : 0;
            np = max(np, p);
            poles += p;
            out |= (uint32_t)m << (8 * c);
        }
        if (in) matw[row * nz + k] = out | (uint32_t)np << 24 | (des ? kWordDesign : 0u);
        const uint32_t first = (uint32_t)__builtin_amdgcn_readfirstlane((int)out);
        const uint32_t id = first & 0xff;
        const bool mixed = first != id * 0x010101u || wave_any(des) || wave_any(in && out != first);
        uint32_t code = mixed ? kSegMixed | kSegSpecial | (wave_any(des) ? kSegDesign : 0u) : id;
        for (int s = kMaxPoles; s > 0; --s)
            if (wave_any(np >= s)) {
                code |= kSegSpecial | (uint32_t)s << 8;
                break;
            }
        if (lane == 0) seg[q] = code;
        slots += seg_poles(code);
    }
    for (int o = 32; o > 0; o >>= 1) poles += __shfl_down(poles, o, 64);
    __shared__ unsigned long long sums[4][2];
    if (lane == 0) sums[threadIdx.x >> 6][0] = slots, sums[threadIdx.x >> 6][1] = poles;
    __syncthreads();
    if (threadIdx.x < 2) {
        unsigned long long t = 0;
        for (int w = 0; w < 4; ++w) t += sums[w][threadIdx.x];
        if (t) atomicAdd(count + threadIdx.x, t);
    }
}

// The first id that is neither below nmat nor an allowed design id, in the order of cells and
// components: *first = 2 * (3 * cell + component), + 1 for a design id.
__global__ void __launch_bounds__(256) k_check_words(const uint32_t* __restrict__ given, long n, int nmat, bool design,
                                                     unsigned long long* __restrict__ first) {
    for (long q = (long)blockIdx.x * blockDim.x + threadIdx.x; q < n; q += (long)gridDim.x * blockDim.x) {
        const uint32_t w = given[q];
        for (int c = 0; c < 3; ++c) {
            const int m = (w >> (8 * c)) & 0xff;
            if (m < nmat || (m == kDesignMat && design)) continue;
            atomicMin(first, 2ull * (3 * q + c) + (m == kDesignMat ? 1 : 0));
            break;
        }
    }
}

// Design ids on the box [lo, lo + ext)
__global__ void __launch_bounds__(256) k_mark_design(uint32_t* __restrict__ given, int ny, int nz, int lx, int ly, int lz,
                                                     int ey, int ez, long n) {
    const long q = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (q >= n) return;
    const long r = q / ez, i = r / ey;
    given[((lx + i) * ny + ly + (r - i * ey)) * nz + lz + (q - r * ez)] = 0x00ffffffu;
}

// Words of listed cells
__global__ void __launch_bounds__(256) k_read_words(const uint32_t* __restrict__ matw, const long* __restrict__ cell,
                                                    long n, uint32_t* __restrict__ out) {
    const long q = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (q < n) out[q] = matw[cell[q]];
}

// Fused H / polarisation / E update of one time step.  TY: y rows per thread; NP: pole slots
// compiled in (>= the largest pole count of any material).
// A workgroup covers one z line (thread k = cell k) of TY consecutive y rows and marches along
// x.  On grids that the caches hold the step is bound by the instructions a plane takes and by the
// latency of what it waits for, on large ones by memory; so:
//   * Every register that a plane's update has read is loaded again for the plane that needs it
//     next as soon as it has been read -- H, the PML auxiliaries, the pole state and the material
//     words for plane i + 1, E for plane i + 2.  No load is waited for in the iteration that issues
//     it, and none is copied from register to register while it is in flight (such a copy waits for
//     the load and, both counting in vmcnt, for the iteration's stores).  The loop starts with the
//     E phase, the first H phase standing before it, and the last H phase runs past the chunk: all
//     ways into the loop then have the same loads and stores in flight in the same order, and the
//     wait counts need not assume the worse of two.  The loads and stores of a plane that is not
//     needed (past the chunk, past a metallic edge) go through a descriptor of length zero: they
//     return 0 or are dropped without a memory access.
//   * One word per 64 cells of a z line (k_words) says whether a wavefront's cells all run one
//     material without poles; then its constant is a scalar and neither the per-cell words nor the
//     material table are read.
//   * A thread's byte offset within a component plane depends only on its row and z cell, so it is
//     fixed for the whole march; each access is a per-plane descriptor, that lane offset and a
//     uniform component offset.  Ghost rows, lanes past the end of the z line and lanes outside a
//     z PML layer, a pole slot or the design region carry the out-of-range offset instead of
//     branching; what holds for a whole wavefront (row, plane, x/y PML, any lane in a z layer,
//     material segment) is a bit of a scalar and a branch.  Registers that a branch alone loads and
//     uses are left unset otherwise.
// Measured on MI355X, us per step before (every register loaded in the iteration that uses it, rotated
// by copies) and now: FP32 512x512x256 1183, 1047 (5.0 TB/s of fields, what a plain copy that marches
// alike reaches); 448x224x512 922, 732; 192x192x96 118, 94; FP64 96^3 51, 42.
template <typename T, int TY, int NP, bool ZP, bool NTS>
__device__ __forceinline__ void step_tile(const StepArgs<T>& a, const int t) {
    constexpr uint32_t TS = sizeof(T);
    constexpr int NS = NP > 0 ? NP : 1;
    // FP64 rows of two or four with poles have no registers for the loads of a plane ahead: they load H, the
    // auxiliaries and the pole state where they use them.  us per step, all of it ahead and with 256 registers
    // per lane, and as now (512 registers up to 256 threads): 100x100x96 two rows 163, 119, four rows 637, 193;
    // 120x120x250 four rows 968, 283; without poles (ahead, 512 registers) four rows 252, 137 and 447, 184
    constexpr bool kAhead = sizeof(T) == 4 || TY == 1 || NP == 0;
    typedef T Pair __attribute__((ext_vector_type(2)));
    typedef T Erows[TY + 2][3];  // E of rows -1..TY (Ey of row TY unused)
    extern __shared__ __align__(16) unsigned char smem_raw[];
    const int B = blockDim.x;
    Pair* sh = reinterpret_cast<Pair*>(smem_raw);  // [2 parity][TY][B + 1] (Hx, Hy); slot B: zero
    MatLut<T>* slut = reinterpret_cast<MatLut<T>*>(sh + 2 * TY * (B + 1));
    copy_lut(a, slut);
    if (threadIdx.x < 2 * TY) sh[threadIdx.x * (B + 1) + B] = Pair{T(0), T(0)};

    const long step = *(CONST const long*)a.d_step;
    if (t == 0 && threadIdx.x == 0) a.d_step[1] = step;  // for the kernels after this one
    const bool odd = (step & 1) != 0;
    const char* F0 = (const char*)a.F[odd ? 1 : 0];
    const long F01 = (const char*)a.F[odd ? 0 : 1] - F0;  // from the set read to the set written
    const int hr = odd ? 2 : 1;  // H auxiliary pair read this step
    const int hw = odd ? 1 : 2;  // and written
    // FP32 pole slots alternate between two arrays: step n reads P^n (Lorentz) or Q^n (Drude) from
    // Q when n is even, from P when it is odd, and writes the new value to the other, where a
    // Lorentz pole has read P^{n-1}.  Without a Lorentz pole both are one array: each slot is read and
    // written by one lane, the read before the write.  FP64 slots hold Q^n and P^n.
    const char* Pcur = (const char*)(kPolePair<T> && odd ? a.P : a.Q);
    const char* Pold = (const char*)(kPolePair<T> && odd ? a.Q : a.P);
    CONST const uint32_t* seg = (CONST const uint32_t*)a.seg;
    CONST const T* coef = (CONST const T*)a.coef;
    CONST const MatLut<T>* clut = (CONST const MatLut<T>*)a.lut;
    const int nx = a.nx, ny = a.ny, nz = a.nz;
    const int xci = t / a.nty, tyi = t - xci * a.nty;
    const int j0 = tyi * TY;
    const int x0 = xci * a.xc;
    const int x1 = min(x0 + a.xc, nx);
    // The z line in passes of zseg cells (one pass when the workgroup spans the whole line).  The
    // last lane of a pass keeps the H it forms in zh, where the first lane of the next pass reads
    // its z neighbour; passes alternate between two halves of zh.
    const int Z = ZP ? a.zseg : nz;  // ZP: compiled for z passes
    const int npass = ZP ? (nz + Z - 1) / Z : 1;
    Pair* zh = reinterpret_cast<Pair*>((unsigned char*)slut + lut_lds_bytes<T>(a.nmat));  // [2 pass parity][xc][TY]
    const int kl = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int nseg = (nz + 63) >> 6;
    const bool uniform = a.uniform != 0;
    const bool emap = a.emap != nullptr;
    const T cdt = a.cdt;
    const uint32_t PB = (uint32_t)ny * (uint32_t)nz * TS;  // bytes of one component plane
    const long FPB = 6L * PB;                             // bytes of one x plane of a field set
    const long QPB = (long)a.nqp * PB;                    // and of the polarisation
    const int Ly = a.plo[1] + a.phi[1], Lz = a.plo[2] + a.phi[2];
    const uint32_t SP0 = (uint32_t)(2 * a.S[0] * TS), SP1 = (uint32_t)(2 * a.S[1] * TS), SP2 = (uint32_t)(2 * a.S[2] * TS);
    const Rsrc rpx = rsrc(a.psi[0]), rpy = rsrc(a.psi[1]), rpz = rsrc(a.psi[2]);
    CONST const T* cx = coef + a.coff[0];
    CONST const T* cy = coef + a.coff[1];
    // planes outside [xlo, xlo + xin) lie in an x layer
    const int xlo = a.pml_on[0] ? a.plo[0] : 0;
    const unsigned xin = a.pml_on[0] ? (unsigned)(nx - a.phi[0] - a.plo[0]) : 0xffffffffu;
    auto in_x = [&](int p) { return (unsigned)(p - xlo) >= xin; };

    int gj[TY + 2];  // global row of local row r-1 (r = 0 is the halo row below the tile), -1 outside
    int sy[TY + 1];  // its row within the y layers
    uint32_t fl = 0; // bits r: row r lies in a y layer; 8 + r: row r is inside the grid; 16 + r: owned row r - 1
#pragma unroll
    for (int r = 0; r < TY + 2; ++r) gj[r] = TY > 1 ? wrap_or_ghost(j0 + r - 1, ny, a.py) : wrap_one(j0 + r - 1, ny, a.py);
#pragma unroll
    for (int r = 0; r < TY + 1; ++r) {
        const bool y = gj[r] >= 0 && in_pml(a, 1, gj[r], ny);
        sy[r] = y ? (gj[r] < a.plo[1] ? gj[r] : gj[r] - (ny - a.phi[1]) + a.plo[1]) : 0;
        fl |= (y ? 1u << r : 0u) | (gj[r] >= 0 ? 0x100u << r : 0u) | (r > 0 && j0 + r - 1 < ny ? 0x10000u << r : 0u);
    }
    fl = __builtin_amdgcn_readfirstlane(fl);
    auto in_y = [&](int r) { return ((fl >> r) & 1) != 0; };
    auto valid = [&](int r) { return ((fl >> (8 + r)) & 1) != 0; };
    auto own = [&](int r) { return TY == 1 || ((fl >> (17 + r)) & 1) != 0; };
    const bool yany = (fl & 0xff) != 0;
    auto xslab = [&](int p) -> uint32_t { return (uint32_t)(p < a.plo[0] ? p : p - (nx - a.phi[0]) + a.plo[0]) * 2u * PB; };
    auto yslab = [&](int p, int r) -> uint32_t { return (uint32_t)((p * Ly + sy[r]) * nz) * 2u * TS; };

    for (int pass = 0; pass < npass; ++pass) {
        const int k = pass * Z + kl;
        const bool kin = kl < Z && k < nz;
        const int kp1 = k + 1 < nz ? k + 1 : a.pz ? 0 : -1;
        uint32_t oR[TY + 2];   // byte offset of (row, k) within a component plane, or kOOB
        uint32_t oK1[TY + 1];  // byte offset of (row, k + 1), or kOOB
#pragma unroll
        for (int r = 0; r < TY + 2; ++r) oR[r] = gj[r] >= 0 && kin ? (uint32_t)(gj[r] * nz + k) * TS : kOOB;
#pragma unroll
        for (int r = 0; r < TY + 1; ++r)
            oK1[r] = (gj[r] >= 0 && kin && kp1 >= 0) ? (uint32_t)(gj[r] * nz + kp1) * TS : kOOB;

        const bool zpml = kin && in_pml(a, 2, k, nz);
        const bool zany = wave_any(zpml);  // some lane of this wavefront lies in a z PML layer
        const uint32_t oK = kin ? (uint32_t)k * 2u * TS : kOOB;  // in a y slab
        const uint32_t oZ = zpml ? (uint32_t)(k < a.plo[2] ? k : k - (nz - a.phi[2]) + a.plo[2]) * 2u * TS : kOOB;
        T bEz = T(0), aEz = T(0), bHz = T(0), aHz = T(0);
        if (zpml) {
            GLOBAL const T* cz = (GLOBAL const T*)a.coef + a.coff[2];
            bEz = cz[k], aEz = cz[nz + k], bHz = cz[2 * nz + k], aHz = cz[3 * nz + k];
        }
        // segment of this wavefront (one past the line, in a batch of longer lines, has no cell)
        const int sg = min((ZP ? pass * (Z >> 6) : 0) + wave, nseg - 1);
        // the z neighbour below: the lane below in this pass, else the periodic image (one pass),
        // else the zero slot; the first lane of a later pass reads zh
        const int kb = kl > 0 ? kl - 1 : (a.pz ? nz - 1 : B);
        lds_barrier();  // the material table; the exchange slots of the previous pass

        // the registers each plane loads anew
        Erows ec, en;                                      // E^n of planes i and i + 1
        T h0[TY + 1][3], ek[TY + 1][2];                    // H^{n-1/2} of plane i; E^n at k + 1
        Pair pHx[TY + 1], pHy[TY + 1], pHz[TY + 1];        // H auxiliaries
        Pair pEx[TY], pEy[TY], pEz[TY];                    // E auxiliaries
        T em[TY][3];                                       // 1/eps of the maps
        T Qv[TY][3][NS], Pv[TY][3][NS];                    // pole state
        uint32_t mw[TY], mwn[TY];                          // material words of planes i, i + 1
        T hp[TY][2];                                       // H^{n+1/2} (Hy, Hz) of plane i - 1
        T h[TY + 1][3], e0[TY][3];                         // H^{n+1/2} and E^n (owned rows) of plane i
        T iv[TY], inv[TY][3], sq[TY][3];                   // 1/eps (of a one-material segment, of each E) and sum of Q^{n+1}
        T dv[TY][3];                                       // 1/eps and material words of design voxels
        uint32_t dw[TY];
        uint32_t cc[TY], cn[TY], cnn[TY];                  // segment codes of planes i, i + 1, i + 2

        auto code_of = [&](int p, int r) -> uint32_t { return seg[(uint32_t)((p * ny + gj[r + 1]) * nseg + sg)]; };
        auto load_e = [&](const char* f, bool need, Erows& e) {
            const Rsrc rn = rsrc(f, need);
#pragma unroll
            for (int r = 0; r < TY + 2; ++r)
#pragma unroll
                for (int c = 0; c < 3; ++c)
                    if (c != 1 || r < TY + 1) e[r][c] = bld<T>(rn, oR[r], c * PB);
        };
        auto load_h = [&](const char* f, bool need) {
            const Rsrc rn = rsrc(f, need);
#pragma unroll
            for (int r = 0; r < TY + 1; ++r) {
#pragma unroll
                for (int c = 0; c < 3; ++c) h0[r][c] = bld<T>(rn, oR[r], (3 + c) * PB);
#pragma unroll
                for (int c = 0; c < 2; ++c) ek[r][c] = bld<T>(rn, oK1[r], c * PB);
            }
        };
        auto zrow = [&](int p, int r) -> uint32_t { return (uint32_t)((p * ny + gj[r]) * Lz) * 2u * TS; };
        auto load_psi_h = [&](int p) {
            if (zany) {
#pragma unroll
                for (int r = 0; r < TY + 1; ++r)
                    if (valid(r)) pHz[r] = bld2<T>(rpz, oZ, hr * SP2 + zrow(p, r));
            }
            if (__builtin_expect(yany, 0)) {
#pragma unroll
                for (int r = 0; r < TY + 1; ++r)
                    if (in_y(r)) pHy[r] = bld2<T>(rpy, oK, hr * SP1 + yslab(p, r));
            }
            if (__builtin_expect(in_x(p), 0)) {
                const uint32_t so = hr * SP0 + xslab(p);
#pragma unroll
                for (int r = 0; r < TY + 1; ++r) pHx[r] = bld2<T>(rpx, two(oR[r]), so);
            }
        };
        auto load_psi_e = [&](int p, int r) {
            if (zany) pEz[r] = bld2<T>(rpz, oZ, zrow(p, r + 1));
            if (__builtin_expect(yany, 0)) {
                if (in_y(r + 1)) pEy[r] = bld2<T>(rpy, oK, yslab(p, r + 1));
            }
            if (__builtin_expect(in_x(p), 0)) pEx[r] = bld2<T>(rpx, two(oR[r + 1]), xslab(p));
            if (__builtin_expect(emap, 0)) {
                const Rsrc re = rsrc((const char*)a.emap + (long)p * 3 * PB);
#pragma unroll
                for (int c = 0; c < 3; ++c) em[r][c] = bld<T>(re, oR[r + 1], c * PB);
            }
        };
        auto load_word = [&](int p, int r, uint32_t code, uint32_t& w) {  // where a segment is mixed
            if (code & kSegMixed) {
                const uint32_t o = oR[r + 1];
                w = bld<uint32_t>(rsrc((const char*)a.matw + (long)p * ny * nz * 4), TS == 4 || o == kOOB ? o : o / 2, 0);
            }
        };
        // material words of a segment of one material are its id three times
        auto words = [&](uint32_t code, uint32_t w) { return code & kSegMixed ? w : (uint32_t)seg_material(code) * 0x010101u; };
        // pole state of plane p, whose segment code is `code` and material words are w
        auto load_poles = [&](int p, int r, uint32_t code, uint32_t w) {
            const int npx = seg_poles(code);
            const Rsrc rc = rsrc(Pcur + (long)p * QPB), ro = rsrc(Pold + (long)p * QPB);
            int np[3], lm[3];
#pragma unroll
            for (int c = 0; c < 3; ++c) {
                const MatLut<T>& L = slut[(w >> (8 * c)) & 0xff];
                np[c] = L.np;
                lm[c] = L.lorentz_mask;
            }
#pragma unroll
            for (int s = 0; s < NP; ++s) {
                if (s >= npx) break;
#pragma unroll
                for (int c = 0; c < 3; ++c) {
                    // (a Drude slot reads one value; the second array may be absent without Lorentz poles)
                    Qv[r][c][s] = bld<T>(rc, s < np[c] ? oR[r + 1] : kOOB, (s * 3 + c) * PB);
                    Pv[r][c][s] = bld<T>(ro, (lm[c] >> s) & 1 ? oR[r + 1] : kOOB, (s * 3 + c) * PB);
                }
            }
        };

        // ---- the chunk's first planes; H (y and z components) of the plane before it
        int pi = x0, pn = wrap_up(x0 + 1, nx, a.px), pnn = wrap_up(pn + 1, nx, a.px);  // nx or more: past the edge
        const char* fW = F0 + (long)pi * FPB;  // plane i, then i + 1 and i + 2, of the set read
        const char* fN = F0 + (long)min(pn, nx - 1) * FPB;
        const char* fNN = F0 + (long)min(pnn, nx - 1) * FPB;
#pragma unroll
        for (int r = 0; r < TY; ++r) {
            cc[r] = uniform || !own(r) ? 0u : code_of(pi, r);
            cn[r] = uniform || !own(r) || x0 + 1 >= x1 ? 0u : code_of(pn, r);
            hp[r][0] = hp[r][1] = T(0);
        }
        load_e(fW, true, ec);
        if (x0 > 0 || a.px) {
            const int p = x0 > 0 ? x0 - 1 : nx - 1;
            const bool xp = in_x(p);
            const Rsrc rn = rsrc(F0 + (long)p * FPB);
            T eh[TY + 1][3], hh[TY][2], ekx[TY];
            Pair qx[TY], qy[TY], qz[TY];
#pragma unroll
            for (int r = 0; r < TY + 1; ++r)  // rows 0..TY; row TY: Ex alone
#pragma unroll
                for (int c = 0; c < 3; ++c)
                    if (c == 0 || r < TY) eh[r][c] = bld<T>(rn, oR[r + 1], c * PB);
#pragma unroll
            for (int r = 0; r < TY; ++r) {
                hh[r][0] = bld<T>(rn, oR[r + 1], 4 * PB);
                hh[r][1] = bld<T>(rn, oR[r + 1], 5 * PB);
                ekx[r] = bld<T>(rn, oK1[r + 1], 0);
                if (!own(r)) continue;
                if (xp) qx[r] = bld2<T>(rpx, two(oR[r + 1]), hr * SP0 + xslab(p));
                if (in_y(r + 1)) qy[r] = bld2<T>(rpy, oK, hr * SP1 + yslab(p, r + 1));
                if (zany) qz[r] = bld2<T>(rpz, oZ, hr * SP2 + zrow(p, r + 1));
            }
#pragma unroll
            for (int r = 0; r < TY; ++r) {
                if (!own(r)) continue;
                T dEx_y = eh[r + 1][0] - eh[r][0];
                T dEx_z = ekx[r] - eh[r][0];
                T dEz_x = ec[r + 1][2] - eh[r][2];
                T dEy_x = ec[r + 1][1] - eh[r][1];
                if (in_y(r + 1)) dEx_y += aux_next_y(dEx_y, cy[2 * ny + gj[r + 1]], cy[3 * ny + gj[r + 1]], qy[r].y);
                if (zany) dEx_z += aux_next(dEx_z, bHz, aHz, qz[r].y);
                if (xp) {
                    const T b = cx[2 * nx + p], c = cx[3 * nx + p];
                    dEz_x += aux_next(dEz_x, b, c, qx[r].x);
                    dEy_x += aux_next(dEy_x, b, c, qx[r].y);
                }
                hp[r][0] = h_next(hh[r][0], cdt, dEx_z, dEz_x);
                hp[r][1] = h_next(hh[r][1], cdt, dEy_x, dEx_y);
            }
        }
        load_e(fN, pn < nx, en);
        if constexpr (kAhead) {
            load_h(fW, true);
            load_psi_h(pi);
        }
#pragma unroll
        for (int r = 0; r < TY; ++r) {
            if (!own(r)) continue;
            if constexpr (kAhead) load_psi_e(pi, r);
            load_word(pi, r, cc[r], mw[r]);
            load_word(pn, r, cn[r], mwn[r]);
            if (cc[r] & kSegSpecial) {
                mw[r] = words(cc[r], mw[r]);
                if constexpr (kAhead)
                    if (NP > 0 && seg_poles(cc[r]) > 0) load_poles(pi, r, cc[r], mw[r]);
            }
        }

        auto h_phase = [&](const int i) __attribute__((always_inline)) {
            const bool live = i < x1, next = i + 1 < x1;
            const bool xpml = live && in_x(pi);
            const Rsrc rW = rsrc(fW + F01, live);
#pragma unroll
            for (int r = 0; r < TY; ++r) {
                cnn[r] = uniform || !own(r) || i + 2 >= x1 ? 0u : code_of(pnn, r);
                iv[r] = clut[seg_material(cc[r])].inv_eps;
            }
            if constexpr (!kAhead) {
                load_h(fW, live);
                if (live) load_psi_h(pi);
            }
            T d[TY + 1][6];  // dEz_y, dEx_y, dEy_z, dEx_z, dEz_x, dEy_x
#pragma unroll
            for (int r = 0; r < TY + 1; ++r) {
                d[r][0] = ec[r + 1][2] - ec[r][2];
                d[r][1] = ec[r + 1][0] - ec[r][0];
                d[r][2] = ek[r][1] - ec[r][1];
                d[r][3] = ek[r][0] - ec[r][0];
                d[r][4] = en[r][2] - ec[r][2];
                d[r][5] = en[r][1] - ec[r][1];
            }
            if (zany) {  // lanes outside the layers: b = a = 0 leaves the term unchanged
#pragma unroll
                for (int r = 0; r < TY + 1; ++r) {
                    if (!valid(r)) continue;
                    const T q0 = aux_next(d[r][2], bHz, aHz, pHz[r].x), q1 = aux_next(d[r][3], bHz, aHz, pHz[r].y);
                    d[r][2] += q0;
                    d[r][3] += q1;
                    if (r > 0 && own(r - 1) && live) bst2<NTS>(rpz, oZ, hw * SP2 + zrow(pi, r), Pair{q0, q1});
                }
            }
            if (__builtin_expect(yany, 0)) {
#pragma unroll
                for (int r = 0; r < TY + 1; ++r) {
                    if (!in_y(r)) continue;
                    const T b = cy[2 * ny + gj[r]], c = cy[3 * ny + gj[r]];
                    const T q0 = aux_next_y(d[r][0], b, c, pHy[r].x), q1 = aux_next_y(d[r][1], b, c, pHy[r].y);
                    d[r][0] += q0;
                    d[r][1] += q1;
                    if (r > 0 && own(r - 1) && live) bst2<NTS>(rpy, oK, hw * SP1 + yslab(pi, r), Pair{q0, q1});
                }
            }
            if (__builtin_expect(xpml, 0)) {
                const T b = cx[2 * nx + pi], c = cx[3 * nx + pi];
                const uint32_t so = hw * SP0 + xslab(pi);
#pragma unroll
                for (int r = 0; r < TY + 1; ++r) {
                    const T q0 = aux_next(d[r][4], b, c, pHx[r].x), q1 = aux_next(d[r][5], b, c, pHx[r].y);
                    d[r][4] += q0;
                    d[r][5] += q1;
                    if (r > 0 && own(r - 1)) bst2<NTS>(rpx, two(oR[r]), so, Pair{q0, q1});
                }
            }
#pragma unroll
            for (int r = 0; r < TY + 1; ++r) {
                h[r][0] = h_next(h0[r][0], cdt, d[r][0], d[r][2]);
                h[r][1] = h_next(h0[r][1], cdt, d[r][3], d[r][4]);
                h[r][2] = h_next(h0[r][2], cdt, d[r][5], d[r][1]);
                // outside a metallic edge H is identically zero (ghost row of the halo)
                if (!valid(r)) h[r][0] = h[r][1] = h[r][2] = T(0);
#pragma unroll
                for (int c = 0; c < 3; ++c) pin(h[r][c]);
                if (r > 0 && own(r - 1)) {
#pragma unroll
                    for (int c = 0; c < 3; ++c) bst<NTS>(rW, oR[r], (3 + c) * PB, h[r][c]);
                }
            }
            Pair* buf = sh + (i & 1) * TY * (B + 1);
#pragma unroll
            for (int r = 0; r < TY; ++r) {
                buf[r * (B + 1) + kl] = Pair{h[r + 1][0], h[r + 1][1]};
#pragma unroll
                for (int c = 0; c < 3; ++c) e0[r][c] = reg_copy(ec[r + 1][c]);
            }
            if (ZP && live && pass + 1 < npass && kl == Z - 1) {
                Pair* zo = zh + ((pass & 1) * a.xc + (i - x0)) * TY;
#pragma unroll
                for (int r = 0; r < TY; ++r) zo[r] = Pair{h[r + 1][0], h[r + 1][1]};
            }
            // ------------------------------- polarisation: sum of Q^{n+1} over the poles; 1/eps
#pragma unroll
            for (int r = 0; r < TY; ++r) {
#pragma unroll
                for (int c = 0; c < 3; ++c) inv[r][c] = iv[r], sq[r][c] = T(0);
                if (!own(r)) continue;
                const uint32_t code = cc[r];
                if (code & kSegSpecial) {
                    const MatLut<T>* L[3];
#pragma unroll
                    for (int c = 0; c < 3; ++c) {
                        L[c] = slut + ((mw[r] >> (8 * c)) & 0xff);
                        inv[r][c] = L[c]->inv_eps;
                    }
                    const int npx = seg_poles(code);
                    if (NP > 0 && npx > 0) {
                        if constexpr (!kAhead) load_poles(pi, r, code, mw[r]);
                        const Rsrc rc = rsrc(Pcur + (long)pi * QPB), ro = rsrc(Pold + (long)pi * QPB);
                        int np[3];
#pragma unroll
                        for (int c = 0; c < 3; ++c) np[c] = L[c]->np;
#pragma unroll
                        for (int s = 0; s < NP; ++s) {
                            if (s >= npx) break;
                            PoleCoef<T> p[3];
#pragma unroll
                            for (int c = 0; c < 3; ++c) p[c] = L[c]->pole[s];
#pragma unroll
                            for (int c = 0; c < 3; ++c) {
                                const uint32_t so = (s * 3 + c) * PB;
                                const bool vq = s < np[c];
                                const T cur = Qv[r][c][s], old = Pv[r][c][s];
                                T qn;
                                if constexpr (kPolePair<T>) {  // Lorentz: P^n, P^{n-1}; Drude (lor = beta = 0): Q^n
                                    qn = fma_(p[c].c3, e0[r][c], fma_(p[c].alpha, fma_(-p[c].lor, old, cur), p[c].beta * cur));
                                    bst<NTS>(ro, vq ? oR[r + 1] : kOOB, so, fma_(p[c].lor, cur, qn));
                                } else {  // Q^n, P^n (zero for a Drude pole)
                                    qn = fma_(p[c].beta, old, fma_(p[c].alpha, cur, p[c].c3 * e0[r][c]));
                                    bst<NTS>(ro, vq && p[c].lor != T(0) ? oR[r + 1] : kOOB, so, old + qn);
                                    bst<NTS>(rc, vq ? oR[r + 1] : kOOB, so, qn);
                                }
                                sq[r][c] += vq ? qn : T(0);
                            }
                        }
                    }
                    if (code & kSegDesign) {
                        // design voxels: 1/eps from the design array [dx][dy][dz]
                        const Rsrc rd = rsrc(a.dinv);
                        const uint32_t dq = (uint32_t)(((pi - a.dlo[0]) * (a.dhi[1] - a.dlo[1]) + (gj[r + 1] - a.dlo[1])) *
                                                           (a.dhi[2] - a.dlo[2]) + (k - a.dlo[2])) * TS;
#pragma unroll
                        for (int c = 0; c < 3; ++c) dv[r][c] = bld<T>(rd, (int)((mw[r] >> (8 * c)) & 0xff) == a.nmat ? dq : kOOB, 0);
                        dw[r] = mw[r];
                    }
                }
                if (cn[r] & kSegSpecial) {
                    const uint32_t w = words(cn[r], mwn[r]);
                    if constexpr (kAhead)
                        if (NP > 0 && seg_poles(cn[r]) > 0) load_poles(pn, r, cn[r], w);
                    mw[r] = reg_copy(w);
                }
                load_word(pnn, r, cnn[r], mwn[r]);
            }
            // ------------------------------- loads for the planes ahead
#pragma unroll
            for (int r = 0; r < TY + 2; ++r)
#pragma unroll
                for (int c = 0; c < 3; ++c)
                    if (c != 1 || r < TY + 1) ec[r][c] = reg_copy(en[r][c]);
            if constexpr (kAhead) load_h(fN, next);
            load_e(fNN, next && pnn < nx, en);
            if constexpr (kAhead)
                if (next) load_psi_h(pn);
        };

        auto e_phase = [&](const int i) __attribute__((always_inline)) {
            const bool next = i + 1 < x1;
            const bool xpml = in_x(pi);
            const Rsrc rW = rsrc(fW + F01);
            const Pair* buf = sh + (i & 1) * TY * (B + 1);
            // ------------------------------- E^{n+1}
            lds_barrier();
#pragma unroll
            for (int r = 0; r < TY; ++r) {
                if (!own(r)) continue;
                if constexpr (!kAhead) load_psi_e(pi, r);
                const uint32_t o = oR[r + 1];
                const Pair* below = buf + r * (B + 1) + kb;
                if (ZP && pass > 0 && kl == 0) below = zh + (((pass - 1) & 1) * a.xc + (i - x0)) * TY + r;
                const Pair hk = *below;
                T dHz_y = h[r + 1][2] - h[r][2];
                T dHx_y = h[r + 1][0] - h[r][0];
                T dHy_z = h[r + 1][1] - hk.y;
                T dHx_z = h[r + 1][0] - hk.x;
                T dHz_x = h[r + 1][2] - hp[r][1];
                T dHy_x = h[r + 1][1] - hp[r][0];
                if (zany) {
                    const T q0 = aux_next(dHy_z, bEz, aEz, pEz[r].x), q1 = aux_next(dHx_z, bEz, aEz, pEz[r].y);
                    dHy_z += q0;
                    dHx_z += q1;
                    bst2<NTS>(rpz, oZ, zrow(pi, r + 1), Pair{q0, q1});
                }
                if (__builtin_expect(yany, 0)) {
                    if (in_y(r + 1)) {
                        const T b = cy[gj[r + 1]], c = cy[ny + gj[r + 1]];
                        const T q0 = aux_next_y(dHz_y, b, c, pEy[r].x), q1 = aux_next_y(dHx_y, b, c, pEy[r].y);
                        dHz_y += q0;
                        dHx_y += q1;
                        bst2<NTS>(rpy, oK, yslab(pi, r + 1), Pair{q0, q1});
                    }
                }
                if (__builtin_expect(xpml, 0)) {
                    const T b = cx[pi], c = cx[nx + pi];
                    const T q0 = aux_next(dHz_x, b, c, pEx[r].x), q1 = aux_next(dHy_x, b, c, pEx[r].y);
                    dHz_x += q0;
                    dHy_x += q1;
                    bst2<NTS>(rpx, two(o), xslab(pi), Pair{q0, q1});
                }
                const T curl[3] = {dHz_y - dHy_z, dHx_z - dHz_x, dHy_x - dHx_y};
                if (__builtin_expect(emap, 0)) {
#pragma unroll
                    for (int c = 0; c < 3; ++c) inv[r][c] = em[r][c];
                }
                if (cc[r] & kSegDesign) {
#pragma unroll
                    for (int c = 0; c < 3; ++c) inv[r][c] = (int)((dw[r] >> (8 * c)) & 0xff) == a.nmat ? dv[r][c] : inv[r][c];
                }
#pragma unroll
                for (int c = 0; c < 3; ++c) bst<NTS>(rW, o, c * PB, e_next(e0[r][c], inv[r][c], cdt, curl[c], sq[r][c]));
                hp[r][0] = reg_copy(h[r + 1][1]);
                hp[r][1] = reg_copy(h[r + 1][2]);
                if constexpr (kAhead)
                    if (next) load_psi_e(pn, r);
                cc[r] = cn[r];
                cn[r] = cnn[r];
            }
            // the next plane
            fW = fN;
            fN = fNN;
            pi = pn;
            pn = pnn;
            ++pnn;
            fNN += FPB;
            if (__builtin_expect(pnn >= nx, 0)) {
                if (a.px) pnn = 0;
                fNN = F0;  // of plane 0, or not read
            }
        };

        h_phase(x0);
        for (int i = x0; i < x1; ++i) {
            e_phase(i);
            h_phase(i + 1);
        }
    }  // pass
}

// Material of a wavefront's cells from their words: kSegSpecial with the most pole slots of a lane
// (bits 8-10), or the id of their one material without poles
template <int NP>
__device__ __forceinline__ uint32_t classify(uint32_t w) {
    const uint32_t first = (uint32_t)__builtin_amdgcn_readfirstlane((int)w), id = first & 0xff;
    if (first == id * 0x010101u && !wave_any(w != first)) return id;
    uint32_t code = kSegSpecial;
    if (wave_any((w & kWordDesign) != 0)) code |= kSegDesign;
    const int np = word_poles(w);
#pragma unroll
    for (int s = NP; s > 0; --s)
        if (wave_any(np >= s)) {
            code |= (uint32_t)s << 8;
            break;
        }
    return code;
}

// Fused step, row-of-threads form.  A workgroup holds a.rt rows of nz threads (one cell of a
// y row per thread); thread row 0 recomputes H on the row below the tile (the y halo) and rows
// 1..rt-1 own rows j0..j0+rt-2.  The y and z neighbours of E (for H) and of H (for E) are
// exchanged through LDS, so each field value is loaded from global memory once per tile and
// the y halo costs one extra row per rt-1 owned rows instead of one per row.  The top thread
// row loads E of the row above the tile (Ex, Ez) itself.  The tile marches along x; loads,
// register copies, loop shape and addressing as in step_tile.  One barrier per plane: E of plane
// i + 1, which H^{n+1/2} of plane i needs anyway, goes to LDS together with that H (both in two
// halves used in turn), so a plane's H phase starts from what the barrier before it published.
// A wavefront can span rows, so row conditions are per lane and the wavefront's material is found
// from its words (k_words marks in them the cells with poles and the design voxels).
// Bound by the latency of a plane's serial part (exchange, barrier, pole recursion) at 4 waves per
// SIMD on grids of up to about 3 M cells, by memory above.  Measured on MI355X, us per step before
// (two barriers, loads waited for in the iteration that issued them) and now: 24 FP32 grids of 64^3
// to 192x192x128 in one launch 1126, 915; FP32 141x129x95 76.6, 40.2; FP32 151x133x117 77.4 (one
// row), 53.6; FP64 101x101x101 58.6 (one row), 41.4; FP64 41x41x41 22.3, 13.0.
template <typename T, int NP, bool NTS>
__device__ __forceinline__ void step_rows(const StepArgs<T>& a, const int t) {
    constexpr uint32_t W = sizeof(T);
    constexpr int NS = NP > 0 ? NP : 1;
    typedef Pair2<T> Pair;
    extern __shared__ __align__(16) unsigned char smem_raw[];
    const int B = blockDim.x;
    Pair* sExz = reinterpret_cast<Pair*>(smem_raw);       // [2][B] (Ex, Ez) of E^n
    Pair* sHxz = sExz + 2 * B;                            // [2][B] (Hx, Hz) of H^{n+1/2}
    T* sEy = reinterpret_cast<T*>(sHxz + 2 * B);          // [2][B] Ey
    T* sHy = sEy + 2 * B;                                 // [2][B] Hy
    MatLut<T>* slut = reinterpret_cast<MatLut<T>*>(sHy + 2 * B);
    copy_lut(a, slut);

    const long step = *(CONST const long*)a.d_step;
    if (t == 0 && threadIdx.x == 0) a.d_step[1] = step;  // for the kernels after this one
    const bool odd = (step & 1) != 0;
    const char* F0 = (const char*)a.F[odd ? 1 : 0];
    const long F01 = (const char*)a.F[odd ? 0 : 1] - F0;  // from the set read to the set written
    const uint32_t hr = odd ? 2 : 1;  // H auxiliary pair read this step
    const uint32_t hw = odd ? 1 : 2;  // and written
    const char* Pcur = (const char*)(kPolePair<T> && odd ? a.P : a.Q);  // pole slots as in step_tile
    const char* Pold = (const char*)(kPolePair<T> && odd ? a.Q : a.P);
    CONST const T* coef = (CONST const T*)a.coef;
    CONST const MatLut<T>* clut = (CONST const MatLut<T>*)a.lut;
    const int nx = a.nx, ny = a.ny, nz = a.nz;
    const int RT = a.rt, R = RT - 1;
    const int tid = threadIdx.x;
    const bool act = tid < RT * nz;
    const int r = act ? tid / nz : 0;
    const int k = act ? tid - r * nz : 0;
    const int xci = t / a.nty, tyi = t - xci * a.nty;
    const int jr = tyi * R + r - 1;  // unwrapped global row of this thread row
    const int j = act ? wrap_or_ghost(jr, ny, a.py) : -1;
    const bool valid = j >= 0;
    const bool owned = act && r >= 1 && jr < ny;  // implies valid
    const bool top = act && r == RT - 1;
    const int ju = act ? wrap_or_ghost(jr + 1, ny, a.py) : -1;  // the row above
    const int kp1 = k + 1 < nz ? k + 1 : a.pz ? 0 : -1;
    const int km1 = k > 0 ? k - 1 : a.pz ? nz - 1 : -1;
    const T cdt = a.cdt;
    const bool uniform = a.uniform != 0;
    const bool emap = a.emap != nullptr;
    const uint32_t PB = (uint32_t)ny * (uint32_t)nz * W;  // bytes of one component plane
    const long FPB = 6L * PB;                            // bytes of one x plane of a field set
    const long QPB = (long)a.nqp * PB;                   // and of the polarisation
    const long PW = (long)ny * nz * 4;                   // and of the material words
    const int Ly = a.plo[1] + a.phi[1], Lz = a.plo[2] + a.phi[2];
    const uint32_t YP = (uint32_t)(Ly * nz) * 2u * W, ZP = (uint32_t)(ny * Lz) * 2u * W;  // bytes of a slab per plane
    const uint32_t SP0 = (uint32_t)(2 * a.S[0] * W), SP1 = (uint32_t)(2 * a.S[1] * W), SP2 = (uint32_t)(2 * a.S[2] * W);
    const Rsrc rpx = rsrc(a.psi[0]), rpy = rsrc(a.psi[1]), rpz = rsrc(a.psi[2]);
    // planes outside [xlo, xlo + xin) lie in an x layer
    const int xlo = a.pml_on[0] ? a.plo[0] : 0;
    const unsigned xin = a.pml_on[0] ? (unsigned)(nx - a.phi[0] - a.plo[0]) : 0xffffffffu;
    auto in_x = [&](int p) { return (unsigned)(p - xlo) >= xin; };
    auto xslab = [&](int p) -> uint32_t { return (uint32_t)(p < a.plo[0] ? p : p - (nx - a.phi[0]) + a.plo[0]) * 2u * PB; };
    CONST const T* cx = coef + a.coff[0];

    // lane offsets; kOOB for lanes that neither read nor write
    const uint32_t oc = valid ? ((uint32_t)j * nz + k) * W : kOOB;          // the cell
    const uint32_t oo = owned ? oc : kOOB;                                  // owned cells
    const uint32_t ot = top && ju >= 0 ? ((uint32_t)ju * nz + k) * W : kOOB;  // the row above the tile
    const uint32_t ow = owned ? ((uint32_t)j * nz + k) * 4u : kOOB;         // material words
    const bool ypml = valid && in_pml(a, 1, j, ny);
    const bool zpml = valid && in_pml(a, 2, k, nz);
    const uint32_t oy = ypml ? (uint32_t)((j < a.plo[1] ? j : j - (ny - a.phi[1]) + a.plo[1]) * nz + k) * 2u * W : kOOB;
    const uint32_t oz = zpml ? (uint32_t)(j * Lz + (k < a.plo[2] ? k : k - (nz - a.phi[2]) + a.plo[2])) * 2u * W : kOOB;
    const uint32_t oyw = owned ? oy : kOOB, ozw = owned ? oz : kOOB;
    // wavefront-uniform summaries of the per-lane conditions
    const bool yany = wave_any(ypml), zany = wave_any(zpml), tany = wave_any(ot != kOOB);
    T bEy = T(0), aEy = T(0), bHy = T(0), aHy = T(0);
    if (ypml) {
        GLOBAL const T* cy = (GLOBAL const T*)a.coef + a.coff[1];
        bEy = cy[j], aEy = cy[ny + j], bHy = cy[2 * ny + j], aHy = cy[3 * ny + j];
    }
    T bEz = T(0), aEz = T(0), bHz = T(0), aHz = T(0);
    if (zpml) {
        GLOBAL const T* cz = (GLOBAL const T*)a.coef + a.coff[2];
        bEz = cz[k], aEz = cz[nz + k], bHz = cz[2 * nz + k], aHz = cz[3 * nz + k];
    }
    // exchange slots of the row above (top row: te), the row below and the z neighbours
    const int up = (top || !act) ? tid : tid + nz, dn = owned ? tid - nz : tid;
    const int kup = kp1 >= 0 ? r * nz + kp1 : tid, kdn = km1 >= 0 ? r * nz + km1 : tid;

    const int x0 = xci * a.xc;
    const int x1 = min(x0 + a.xc, nx);

    // the registers each plane loads anew
    T ec[3], en[3];                    // E^n of planes i and i + 1
    T te[2] = {T(0), T(0)}, ten[2] = {T(0), T(0)};  // (Ex, Ez) of the row above the tile: zero past the edge
    T h0[3];                           // H^{n-1/2} of plane i
    Pair pHx, pHy, pHz, pEx, pEy, pEz; // PML auxiliaries
    T em[3];                           // 1/eps of the maps
    T Qv[3][NS], Pv[3][NS];            // pole state
    uint32_t mw = 0, mwn = 0;          // material words of planes i, i + 1
    T hp[2] = {T(0), T(0)};            // H^{n+1/2} (Hy, Hz) of plane i - 1
    T h[3], e0[3], inv[3], sq[3], dv[3];
    uint32_t dw = 0;
    uint32_t cls = 0;                  // material of the wavefront on plane i (classify)

    auto load_e = [&](const char* f, bool need) {
        const Rsrc rn = rsrc(f, need);
#pragma unroll
        for (int c = 0; c < 3; ++c) en[c] = bld<T>(rn, oc, c * PB);
        if (tany) {
            ten[0] = bld<T>(rn, ot, 0);
            ten[1] = bld<T>(rn, ot, 2 * PB);
        }
    };
    auto load_h = [&](const char* f, bool need) {
        const Rsrc rn = rsrc(f, need);
#pragma unroll
        for (int c = 0; c < 3; ++c) h0[c] = bld<T>(rn, oc, (3 + c) * PB);
    };
    auto load_psi_h = [&](int p) {
        if (zany) pHz = bld2<T>(rpz, oz, hr * SP2 + p * ZP);
        if (yany) pHy = bld2<T>(rpy, oy, hr * SP1 + p * YP);
        if (__builtin_expect(in_x(p), 0)) pHx = bld2<T>(rpx, two(oc), hr * SP0 + xslab(p));
    };
    auto load_psi_e = [&](int p) {
        if (zany) pEz = bld2<T>(rpz, ozw, p * ZP);
        if (yany) pEy = bld2<T>(rpy, oyw, p * YP);
        if (__builtin_expect(in_x(p), 0)) pEx = bld2<T>(rpx, two(oo), xslab(p));
        if (__builtin_expect(emap, 0)) {
            const Rsrc re = rsrc((const char*)a.emap + (long)p * 3 * PB);
#pragma unroll
            for (int c = 0; c < 3; ++c) em[c] = bld<T>(re, oo, c * PB);
        }
    };
    auto load_poles = [&](int p, uint32_t code, uint32_t w) {
        const int npx = seg_poles(code);
        const Rsrc rc = rsrc(Pcur + (long)p * QPB), ro = rsrc(Pold + (long)p * QPB);
        int np[3], lm[3];
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            const MatLut<T>& L = slut[(w >> (8 * c)) & 0xff];
            np[c] = L.np;
            lm[c] = L.lorentz_mask;
        }
#pragma unroll
        for (int s = 0; s < NP; ++s) {
            if (s >= npx) break;
#pragma unroll
            for (int c = 0; c < 3; ++c) {
                // (a Drude slot reads one value; the second array may be absent without Lorentz poles)
                Qv[c][s] = bld<T>(rc, s < np[c] ? oo : kOOB, (s * 3 + c) * PB);
                Pv[c][s] = bld<T>(ro, (lm[c] >> s) & 1 ? oo : kOOB, (s * 3 + c) * PB);
            }
        }
    };

    // ---- the chunk's first planes; H (y and z components) of the plane before it
    int pi = x0, pn = wrap_up(x0 + 1, nx, a.px), pnn = wrap_up(pn + 1, nx, a.px);  // nx or more: past the edge
    const char* fW = F0 + (long)pi * FPB;  // plane i, then i + 1 and i + 2, of the set read
    const char* fN = F0 + (long)min(pn, nx - 1) * FPB;
    const char* fNN = F0 + (long)min(pnn, nx - 1) * FPB;
    load_e(fW, true);
#pragma unroll
    for (int c = 0; c < 3; ++c) ec[c] = en[c];
    te[0] = ten[0];
    te[1] = ten[1];
    load_h(fW, true);
    if (!uniform) {
        mw = bld<uint32_t>(rsrc((const char*)a.matw + (long)pi * PW), ow, 0);
        mwn = bld<uint32_t>(rsrc((const char*)a.matw + (long)min(pn, nx - 1) * PW, x0 + 1 < x1), ow, 0);
    }
    if (x0 > 0 || a.px) {
        const int p = x0 > 0 ? x0 - 1 : nx - 1;
        const bool xp = in_x(p);
        const Rsrc rn = rsrc(F0 + (long)p * FPB);
        const uint32_t ou = owned && ju >= 0 ? ((uint32_t)ju * nz + k) * W : kOOB;
        const uint32_t ok = owned && kp1 >= 0 ? ((uint32_t)j * nz + kp1) * W : kOOB;
        T eh[3], eu, ekx, hh[2];
        Pair qx, qy, qz;
#pragma unroll
        for (int c = 0; c < 3; ++c) eh[c] = bld<T>(rn, oo, c * PB);
        eu = bld<T>(rn, ou, 0);
        ekx = bld<T>(rn, ok, 0);
        hh[0] = bld<T>(rn, oo, 4 * PB);
        hh[1] = bld<T>(rn, oo, 5 * PB);
        if (xp) qx = bld2<T>(rpx, two(oo), hr * SP0 + xslab(p));
        if (yany) qy = bld2<T>(rpy, oyw, hr * SP1 + p * YP);
        if (zany) qz = bld2<T>(rpz, ozw, hr * SP2 + p * ZP);
        T dEx_y = eu - eh[0], dEx_z = ekx - eh[0], dEz_x = ec[2] - eh[2], dEy_x = ec[1] - eh[1];
        if (yany) dEx_y += aux_next_y(dEx_y, bHy, aHy, qy.y);
        if (zany) dEx_z += aux_next(dEx_z, bHz, aHz, qz.y);
        if (xp) {
            const T b = cx[2 * nx + p], c = cx[3 * nx + p];
            dEz_x += aux_next(dEz_x, b, c, qx.x);
            dEy_x += aux_next(dEy_x, b, c, qx.y);
        }
        hp[0] = h_next(hh[0], cdt, dEx_z, dEz_x);
        hp[1] = h_next(hh[1], cdt, dEy_x, dEx_y);
    }
    sExz[(x0 & 1) * B + tid] = Pair{ec[0], ec[2]};
    sEy[(x0 & 1) * B + tid] = ec[1];
    lds_barrier();  // also the material table
    load_e(fN, pn < nx);
    load_psi_h(pi);
    load_psi_e(pi);
    if (!uniform) {
        cls = classify<NP>(mw);
        if (NP > 0 && seg_poles(cls) > 0) load_poles(pi, cls, mw);
    }

    auto h_phase = [&](const int i) __attribute__((always_inline)) {
        const bool live = i < x1, next = i + 1 < x1;
        const bool xpml = live && in_x(pi);
        const Rsrc rW = rsrc(fW + F01, live);
        const int half = (i & 1) * B, other = B - half;
        const T iv = clut[cls & 0xff].inv_eps;
        // ------------------------------- H^{n+1/2}
        {
            const Pair eu = sExz[half + up];
            const T exk = sExz[half + kup].x, eyk = sEy[half + kup];
            T dEz_y = (top ? te[1] : eu.y) - ec[2];
            T dEx_y = (top ? te[0] : eu.x) - ec[0];
            T dEy_z = (kp1 >= 0 ? eyk : T(0)) - ec[1];
            T dEx_z = (kp1 >= 0 ? exk : T(0)) - ec[0];
            T dEz_x = en[2] - ec[2];
            T dEy_x = en[1] - ec[1];
            // lanes outside a PML layer carry zero coefficients: no change
            if (zany) {
                const T q0 = aux_next(dEy_z, bHz, aHz, pHz.x), q1 = aux_next(dEx_z, bHz, aHz, pHz.y);
                dEy_z += q0;
                dEx_z += q1;
                if (live) bst2<NTS>(rpz, ozw, hw * SP2 + pi * ZP, Pair{q0, q1});
            }
            if (yany) {
                const T q0 = aux_next_y(dEz_y, bHy, aHy, pHy.x), q1 = aux_next_y(dEx_y, bHy, aHy, pHy.y);
                dEz_y += q0;
                dEx_y += q1;
                if (live) bst2<NTS>(rpy, oyw, hw * SP1 + pi * YP, Pair{q0, q1});
            }
            if (__builtin_expect(xpml, 0)) {
                const T b = cx[2 * nx + pi], c = cx[3 * nx + pi];
                const T q0 = aux_next(dEz_x, b, c, pHx.x), q1 = aux_next(dEy_x, b, c, pHx.y);
                dEz_x += q0;
                dEy_x += q1;
                bst2<NTS>(rpx, two(oo), hw * SP0 + xslab(pi), Pair{q0, q1});
            }
            // outside a metallic edge H is identically zero (ghost rows)
            h[0] = valid ? h_next(h0[0], cdt, dEz_y, dEy_z) : T(0);
            h[1] = valid ? h_next(h0[1], cdt, dEx_z, dEz_x) : T(0);
            h[2] = valid ? h_next(h0[2], cdt, dEy_x, dEx_y) : T(0);
        }
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            pin(h[c]);
            bst<NTS>(rW, oo, (3 + c) * PB, h[c]);
            e0[c] = reg_copy(ec[c]);
        }
        sHxz[half + tid] = Pair{h[0], h[2]};
        sHy[half + tid] = h[1];
        sExz[other + tid] = Pair{en[0], en[2]};
        sEy[other + tid] = en[1];
        // ------------------------------- polarisation: sum of Q^{n+1} over the poles; 1/eps
#pragma unroll
        for (int c = 0; c < 3; ++c) inv[c] = iv, sq[c] = T(0);
        if (cls & kSegSpecial) {
            const MatLut<T>* L[3];
#pragma unroll
            for (int c = 0; c < 3; ++c) {
                L[c] = slut + ((mw >> (8 * c)) & 0xff);
                inv[c] = L[c]->inv_eps;
            }
            const int npx = seg_poles(cls);
            if (NP > 0 && npx > 0) {
                const Rsrc rc = rsrc(Pcur + (long)pi * QPB), ro = rsrc(Pold + (long)pi * QPB);
                int np[3];
#pragma unroll
                for (int c = 0; c < 3; ++c) np[c] = L[c]->np;
#pragma unroll
                for (int s = 0; s < NP; ++s) {
                    if (s >= npx) break;
                    PoleCoef<T> p[3];
#pragma unroll
                    for (int c = 0; c < 3; ++c) p[c] = L[c]->pole[s];
#pragma unroll
                    for (int c = 0; c < 3; ++c) {
                        const uint32_t so = (s * 3 + c) * PB;
                        const bool vq = s < np[c];
                        const T cur = Qv[c][s], old = Pv[c][s];
                        T qn;
                        if constexpr (kPolePair<T>) {  // Lorentz: P^n, P^{n-1}; Drude (lor = beta = 0): Q^n
                            qn = fma_(p[c].c3, e0[c], fma_(p[c].alpha, fma_(-p[c].lor, old, cur), p[c].beta * cur));
                            bst<NTS>(ro, vq ? oo : kOOB, so, fma_(p[c].lor, cur, qn));
                        } else {  // Q^n, P^n (zero for a Drude pole)
                            qn = fma_(p[c].beta, old, fma_(p[c].alpha, cur, p[c].c3 * e0[c]));
                            bst<NTS>(ro, vq && p[c].lor != T(0) ? oo : kOOB, so, old + qn);
                            bst<NTS>(rc, vq ? oo : kOOB, so, qn);
                        }
                        sq[c] += vq ? qn : T(0);
                    }
                }
            }
            if (cls & kSegDesign) {
                // design voxels: 1/eps from the design array [dx][dy][dz]
                const Rsrc rd = rsrc(a.dinv);
                const uint32_t dq = (uint32_t)(((pi - a.dlo[0]) * (a.dhi[1] - a.dlo[1]) + (j - a.dlo[1])) *
                                                   (a.dhi[2] - a.dlo[2]) + (k - a.dlo[2])) * W;
#pragma unroll
                for (int c = 0; c < 3; ++c)
                    dv[c] = bld<T>(rd, owned && (int)((mw >> (8 * c)) & 0xff) == a.nmat ? dq : kOOB, 0);
                dw = mw;
            }
        }
        // ------------------------------- loads for the planes ahead
        uint32_t cn = 0u;
        if (!uniform && next) {
            cn = classify<NP>(mwn);
            if (NP > 0 && seg_poles(cn) > 0) load_poles(pn, cn, mwn);
        }
        mw = reg_copy(mwn);
#pragma unroll
        for (int c = 0; c < 3; ++c) ec[c] = reg_copy(en[c]);
        if (tany) {
            te[0] = reg_copy(ten[0]);
            te[1] = reg_copy(ten[1]);
        }
        load_h(fN, next);
        load_e(fNN, next && pnn < nx);
        if (!uniform) mwn = bld<uint32_t>(rsrc((const char*)a.matw + (long)(i + 2 < x1 ? pnn : 0) * PW, i + 2 < x1), ow, 0);
        if (next) load_psi_h(pn);
        return cn;
    };

    auto e_phase = [&](const int i) __attribute__((always_inline)) {
        const bool next = i + 1 < x1;
        const bool xpml = in_x(pi);
        const Rsrc rW = rsrc(fW + F01);
        const int half = (i & 1) * B;
        lds_barrier();
        const Pair hd = sHxz[half + dn];
        const T hxk = sHxz[half + kdn].x, hyk = sHy[half + kdn];
        T dHz_y = h[2] - hd.y;
        T dHx_y = h[0] - hd.x;
        T dHy_z = h[1] - (km1 >= 0 ? hyk : T(0));
        T dHx_z = h[0] - (km1 >= 0 ? hxk : T(0));
        T dHz_x = h[2] - hp[1];
        T dHy_x = h[1] - hp[0];
        if (zany) {
            const T q0 = aux_next(dHy_z, bEz, aEz, pEz.x), q1 = aux_next(dHx_z, bEz, aEz, pEz.y);
            dHy_z += q0;
            dHx_z += q1;
            bst2<NTS>(rpz, ozw, pi * ZP, Pair{q0, q1});
        }
        if (yany) {
            const T q0 = aux_next_y(dHz_y, bEy, aEy, pEy.x), q1 = aux_next_y(dHx_y, bEy, aEy, pEy.y);
            dHz_y += q0;
            dHx_y += q1;
            bst2<NTS>(rpy, oyw, pi * YP, Pair{q0, q1});
        }
        if (__builtin_expect(xpml, 0)) {
            const T b = cx[pi], c = cx[nx + pi];
            const T q0 = aux_next(dHz_x, b, c, pEx.x), q1 = aux_next(dHy_x, b, c, pEx.y);
            dHz_x += q0;
            dHy_x += q1;
            bst2<NTS>(rpx, two(oo), xslab(pi), Pair{q0, q1});
        }
        const T curl[3] = {dHz_y - dHy_z, dHx_z - dHz_x, dHy_x - dHx_y};
        if (__builtin_expect(emap, 0)) {
#pragma unroll
            for (int c = 0; c < 3; ++c) inv[c] = em[c];
        }
        if (cls & kSegDesign) {
#pragma unroll
            for (int c = 0; c < 3; ++c) inv[c] = (int)((dw >> (8 * c)) & 0xff) == a.nmat ? dv[c] : inv[c];
        }
#pragma unroll
        for (int c = 0; c < 3; ++c) bst<NTS>(rW, oo, c * PB, e_next(e0[c], inv[c], cdt, curl[c], sq[c]));
        hp[0] = reg_copy(h[1]);
        hp[1] = reg_copy(h[2]);
        if (next) load_psi_e(pn);
        // the next plane
        fW = fN;
        fN = fNN;
        pi = pn;
        pn = pnn;
        ++pnn;
        fNN += FPB;
        if (__builtin_expect(pnn >= nx, 0)) {
            if (a.px) pnn = 0;
            fNN = F0;  // of plane 0, or not read
        }
    };

    uint32_t cn = h_phase(x0);
    for (int i = x0; i < x1; ++i) {
        e_phase(i);
        cls = cn;
        cn = h_phase(i + 1);
    }
}


// XCD-aware tile order: hardware places workgroup w on XCD w % 8; map so that each XCD
// receives a contiguous run of logical tiles (y-tile fastest, then x-chunk), then find the
// instance that owns the tile: instance b owns tile_first[b] <= t < tile_first[b+1].
__device__ __forceinline__ int tile_instance(const int* __restrict__ tile_first, int ninst, int& t) {
    const int w = blockIdx.x, nw = gridDim.x;
    t = (nw % 8 == 0) ? ((w & 7) * (nw >> 3) + (w >> 3)) : w;
    int lo = 0, hi = ninst - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) / 2;
        if (tile_first[mid] <= t) lo = mid;
        else hi = mid - 1;
    }
    t -= tile_first[lo];
    return lo;
}

// Fused step over all instances of a launch set (rows-per-thread form).
// Waves per SIMD the register allocator must leave room for.  FP32 one-row tiles: 4 (109 registers
// with three pole slots, no scratch; at 5 waves, 96 registers, 80-100 bytes of scratch per lane took
// 2.3 times as long), 5 without poles (88 registers), 3 in z passes (161); FP64 one-row tiles: 2
// (178-215 registers; at 3 waves 170-220 bytes of scratch took 1.4 times as long), 3 without poles
// (162); two FP32 rows: 2 (178).
template <typename T, int TY, int NP, bool ZP = false>
constexpr int step_waves() {
    if (TY > 2 || (TY == 2 && sizeof(T) == 8)) return 1;
    if (sizeof(T) == 8) return NP == 0 && !ZP ? 3 : 2;
    return TY == 2 ? 2 : ZP ? 3 : NP == 0 ? 5 : 4;
}

// The same of the row-of-threads tiles: FP32 81-117 registers, FP64 136 without poles, 155 with one,
// 187-199 with more (no scratch up to 512 threads; FP64 at 1024 threads, 128 registers, spills).
template <typename T, int NP>
constexpr int rows_waves() {
    return sizeof(T) == 4 ? 4 : NP <= 1 ? 3 : 2;
}

// NTS: stores with the non-temporal hint (launch sets that stream more than the caches hold).
template <typename T, int TY, int NP, int MAXT, bool NTS = false>
__global__ void __launch_bounds__(MAXT) __attribute__((amdgpu_waves_per_eu(step_waves<T, TY, NP>())))
k_step(const StepArgs<T>* __restrict__ args, const int* __restrict__ tile_first, int ninst) {
    int t;
    const int b = tile_instance(tile_first, ninst, t);
    step_tile<T, TY, NP, false, NTS>(args[b], t);
}

// The same with the z line in passes of StepArgs::zseg cells (one row per thread)
template <typename T, int NP, int MAXT, bool NTS = false>
__global__ void __launch_bounds__(MAXT) __attribute__((amdgpu_waves_per_eu(step_waves<T, 1, NP, true>())))
k_step_z(const StepArgs<T>* __restrict__ args, const int* __restrict__ tile_first, int ninst) {
    int t;
    const int b = tile_instance(tile_first, ninst, t);
    step_tile<T, 1, NP, true, NTS>(args[b], t);
}

// Fused step over all instances of a launch set (row-of-threads form).
template <typename T, int NP, int MAXT, bool NTS = false>
__global__ void __launch_bounds__(MAXT) k_step_rows(const StepArgs<T>* __restrict__ args,
                                                    const int* __restrict__ tile_first, int ninst) {
    int t;
    const int b = tile_instance(tile_first, ninst, t);
    step_rows<T, NP, NTS>(args[b], t);
}

// ---- read-outs ---------------------------------------------------------------------------------
// They write FP64 values into pinned host memory, in the order the caller receives them: one launch
// and one wait per chunk, and the copy into the caller's array is a plain memcpy.  Bound by the
// host link and by that memcpy, not by the kernels.

// Cells first, first + 1, .. of the box at `base` (its first cell of the component) of by x bz cells
// per x plane; planes are `plane` values apart, rows nz.
template <typename T>
__global__ void __launch_bounds__(256) k_read_box(const T* __restrict__ base, long plane, int nz, int by, int bz,
                                                  long first, long count, double* __restrict__ out) {
    const long stride = (long)gridDim.x * blockDim.x;
    for (long q = (long)blockIdx.x * blockDim.x + threadIdx.x; q < count; q += stride) {
        const long row = (first + q) / bz;
        const int k = (int)(first + q - row * bz);
        const long i = row / by;
        out[q] = (double)base[i * plane + (row - i * by) * nz + k];
    }
}

// DFT values: running sum and its compensation
__global__ void __launch_bounds__(256) k_read_dft(const double2* __restrict__ acc, const double2* __restrict__ cmp,
                                                  long count, double2* __restrict__ out) {
    const long stride = (long)gridDim.x * blockDim.x;
    for (long q = (long)blockIdx.x * blockDim.x + threadIdx.x; q < count; q += stride) {
        const double2 a = acc[q], c = cmp[q];
        out[q] = double2{a.x + c.x, a.y + c.y};
    }
}

// A field value between cells: eight cells (element indices, -1: outside) and their weights, summed
// in order with separate products and sums, as the host sums them
struct GatherPoint {
    long idx[8];
    double w[8];
};
template <typename T>
__global__ void k_read_point(const T* __restrict__ F, const GatherPoint g, double* __restrict__ out) {
    T f[8];
#pragma unroll
    for (int q = 0; q < 8; ++q) f[q] = g.idx[q] >= 0 ? F[g.idx[q]] : T(0);
    double v = 0;
#pragma unroll
    for (int q = 0; q < 8; ++q)
        if (g.idx[q] >= 0) v = __dadd_rn(v, __dmul_rn(g.w[q], (double)f[q]));
    if (threadIdx.x == 0) out[0] = v;
}

// ---- per-step scalars live on the device --------------------------------------------------
// Every engine owns a device step counter and its shadow (d_step[0], d_step[1]), so a sequence of steps
// can be captured once in a hipGraph and replayed at any step.  The kernels up to the fused update
// read the counter, which also fixes the read/write field buffer by its parity; the fused update's
// first tile copies it to the shadow, which the source and DFT kernels after it read, and the
// first workgroup of a step's last kernel sets the counter to shadow + 1: no kernel writes a word
// that one of its workgroups reads, and no workgroup has to know that the others are done, or signs off
// on a shared word.

__global__ void k_tick(long* const* counters, int n) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) counters[i][0] += 1;
}

// The same, in the first workgroup of the step's last kernel (n = 0: not the last)
struct Tick {
    long* const* counters;
    int n;
};
__device__ __forceinline__ void advance(const Tick& tk) {
    if (blockIdx.x == 0 && blockIdx.y == 0)
        for (int i = threadIdx.x; i < tk.n; i += blockDim.x) tk.counters[i][0] = tk.counters[i][1] + 1;
}

// ---- source time functions (FP64) ---------------------------------------------------------
// gaussian_src_time_phase::dipole (reference src/disp.cpp:395-400) and meep's
// continuous_src_time::dipole, evaluated in FP64 on the device.
struct PulseDev {
    int kind;  // 0 gaussian, 1 continuous
    int part;  // 0 real part, 1 imaginary part of amp * current
    double omega, width, phi, peak, cutoff;
    double freq, cw_width, t_start, t_end, slow;
    double amp_re, amp_im;
    double dt;
};

__device__ inline void dipole_dev(const PulseDev& s, double t, double* re, double* im) {
    if (s.kind == 0) {
        const double tt = t - s.peak;
        if ((double)(float)fabs(tt) > s.cutoff) {
            *re = *im = 0.0;
            return;
        }
        const double g = exp(-tt * tt / (2 * s.width * s.width));
        double sn, cs;
        sincos(-s.omega * tt - s.phi, &sn, &cs);
        // polar(1, th) / (-i omega) = (cos th + i sin th) (i / omega)
        *re = -g * sn / s.omega;
        *im = g * cs / s.omega;
    } else {
        const float rt = (float)t;
        if (rt < s.t_start || rt > s.t_end) {
            *re = *im = 0.0;
            return;
        }
        const double w = 2 * M_PI * s.freq;
        double env = 1.0;
        if (s.cw_width != 0.0) {
            const double ts = (t - s.t_start) / s.cw_width - s.slow;
            const double te = (s.t_end - t) / s.cw_width - s.slow;
            env = (1.0 + tanh(ts)) * (1.0 + tanh(te)) * 0.25;
        }
        double sn, cs;
        sincos(-w * t, &sn, &cs);
        *re = -env * sn / w;
        *im = env * cs / w;
    }
}

// amp * J^{n+1/2}, J = (dipole(t_{n+1}) - dipole(t_n)) / dt, real or imaginary part
__device__ inline double source_current(const PulseDev& s, long step) {
    double r0, i0, r1, i1;
    dipole_dev(s, step * s.dt, &r0, &i0);
    dipole_dev(s, (step + 1) * s.dt, &r1, &i1);
    const double jr = (r1 - r0) / s.dt, ji = (i1 - i0) / s.dt;
    return s.part ? s.amp_re * ji + s.amp_im * jr : s.amp_re * jr - s.amp_im * ji;
}

// amp * K^n of a magnetic current, K^n = (dipole(t_n + dt/2) - dipole(t_n - dt/2)) / dt: centred on
// t_n, the midpoint of the H update from n - 1/2 to n + 1/2, as J^{n+1/2} is on that of the E update
__device__ inline double source_current_h(const PulseDev& s, long step) {
    double r0, i0, r1, i1;
    dipole_dev(s, (step - 0.5) * s.dt, &r0, &i0);
    dipole_dev(s, (step + 0.5) * s.dt, &r1, &i1);
    const double kr = (r1 - r0) / s.dt, ki = (i1 - i0) / s.dt;
    return s.part ? s.amp_re * ki + s.amp_im * kr : s.amp_re * kr - s.amp_im * ki;
}

// ---- source injection: E -= coef * J on the source's cells (coef = dt * weight * inv_eps)
// One block covers entries of one source; the block's source and entry range come from
// per-block tables, so all sources of all engines in a launch set go in one launch.
template <typename T>
struct SrcDev {
    PulseDev p;
    T* F[2];             // field set 0 / 1 (entries hold layout indices of the source component)
    const long* d_step;  // the owning engine's step counter and its shadow
};

// the tables of the source launch: per workgroup its source and range of entries; per entry
// the layout index and FP64 coefficient
template <typename T>
struct SrcTables {
    const SrcDev<T>* src;
    const int* blk_src;
    const long* blk_first;
    const long* blk_end;
    const long* idx;
    const double* coef;
};

// the cells of source workgroup blk
template <typename T>
__device__ __forceinline__ void source_block(const SrcTables<T>& t, const int blk) {
    __shared__ double J;
    const int sid = t.blk_src[blk];
    const SrcDev<T>& S = t.src[sid];
    const long step = S.d_step[1];
    if (threadIdx.x == 0) J = source_current(S.p, step);
    __syncthreads();
    const long e = t.blk_first[blk] + threadIdx.x;
    if (e >= t.blk_end[blk] || J == 0.0) return;
    T* F = S.F[(step + 1) & 1];  // the step just completed wrote the other buffer
    const long q = t.idx[e];
    F[q] = (T)((double)F[q] - t.coef[e] * J);
}

// Magnetic currents (dB/dt = -curl E - K, mu = 1): H^{n-1/2} -= dt * weight * K^n in the set the
// coming step reads, before the fused update; the update then forms
// H^{n+1/2} = (H^{n-1/2} - dt K^n) - dt curl E^n, so every workgroup that recomputes a halo row of H
// sees the injected value.  Launched after the monitor gather of step n (samples see H^{n-1/2}).
template <typename T>
__global__ void __launch_bounds__(256) k_source_h(const SrcTables<T> t) {
    __shared__ double K;
    const int blk = blockIdx.x;
    const int sid = t.blk_src[blk];
    const SrcDev<T>& S = t.src[sid];
    const long step = *S.d_step;
    if (threadIdx.x == 0) K = source_current_h(S.p, step);
    __syncthreads();
    const long e = t.blk_first[blk] + threadIdx.x;
    if (e >= t.blk_end[blk] || K == 0.0) return;
    T* F = S.F[step & 1];  // the set step n reads
    const long q = t.idx[e];
    F[q] = (T)((double)F[q] - t.coef[e] * K);
}

// A step with sources and no DFT region ends here: the source kernel advances the counters.
template <typename T>
__global__ void __launch_bounds__(256) k_source(const SrcTables<T> t, const Tick tk) {
    source_block(t, blockIdx.x);
    advance(tk);
}

// ---- point monitors: trilinear gather, FP64 result --------------------------------------
template <typename T>
struct MonDev {
    const T* F[2];       // field set 0 / 1 (idx holds layout indices of the sampled component)
    const long* d_step;  // owning engine's counter
    double* out;         // sample buffer of the owning engine: [sample][npt]
    int npt;             // points of the owning engine
    int p;               // index of this point within its engine
    int span;            // save span
    long idx[8];
    double w[8];
};

template <typename T>
__global__ void __launch_bounds__(256) k_monitor(const MonDev<T>* __restrict__ mon, int n) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const MonDev<T>& m = mon[i];
    const long step = *m.d_step;
    if (step % m.span) return;
    const T* f = m.F[step & 1];
    double v = 0.0;
#pragma unroll
    for (int q = 0; q < 8; ++q)
        if (m.idx[q] >= 0) v += m.w[q] * (double)f[m.idx[q]];
    m.out[(step / m.span) * m.npt + m.p] = v;
}

// ---- DFT: Neumaier-compensated FP64 accumulation of F exp(i 2 pi f t) dt ----------------
__device__ __forceinline__ void neumaier(double& s, double& c, double x) {
    const double t = s + x;
    if (fabs(s) >= fabs(x)) c += (s - t) + x;
    else c += (x - t) + s;
    s = t;
}

template <typename T>
struct DftDev {
    const T* F[2];       // field set 0 / 1 base, [x][6][y][z]
    const long* d_step;  // owning engine's counter and its shadow
    long N, nyz, nz;
    int lo[3], ext[3];
    long ncell;
    long first;          // first global index of this region's (component, cell) pairs
    int comps[6];
    int ncomp;
    int nf;
    const double* freq;  // nf frequencies
    double dt;
    double2* acc;        // [slot][f][cell]
    double2* cmp;        // compensation terms, same layout
};

// One thread per (component, cell, frequency): a workgroup takes one frequency and 256 (component,
// cell) pairs.  Bound by the latency of a thread's chain on small regions and by memory (an accumulator
// and its compensation, 32 bytes read and written) on large ones: the loads are issued before the
// phase is formed, the phase is one FP64 sincos (of the component's own time level), and indices
// are split with 32-bit divisions where the launch's pairs allow it.  Several accumulators per thread
// shared the sincos but left too few loads in flight (102 us in the case below).  Measured on MI355X,
// two planes of 150 x 150 cells, 4 components, 20 frequencies (3.6 M accumulators, 230 MB): with two
// sincos each, 64-bit divisions and a sign-off per workgroup 85 us, now 75; 96 x 96 cells, 5 frequencies
// in FP64 7.9, 7.0.
template <typename T, typename I>
__device__ __forceinline__ void dft_cell(const DftDev<T>& a, const long g, const int f) {
    if (f >= a.nf) return;
    const I local = (I)(g - a.first), ncell = (I)a.ncell;
    const int s = (int)(local / ncell);  // component slot
    const I cell = local - (I)s * ncell;
    const I rest = cell / (I)a.ext[2];
    const int kk = (int)(cell - rest * (I)a.ext[2]);
    const int ii = (int)(rest / (I)a.ext[1]);
    const int jj = (int)(rest - (I)ii * (I)a.ext[1]);
    const int c = a.comps[s];
    const long step = a.d_step[1];
    const long o = ((long)s * a.nf + f) * a.ncell + (long)cell;
    double2 sm = a.acc[o], cp = a.cmp[o];
    // component c of cell (lo + (ii, jj, kk)) in the layout [x][6][y][z]
    const double v = (double)a.F[(step + 1) & 1][(6L * (a.lo[0] + ii) + c) * a.nyz + (long)(a.lo[1] + jj) * a.nz +
                                                 (a.lo[2] + kk)] * a.dt;
    // phase at the time level of E, t = (n+1) dt, or of H, (n+1/2) dt
    double co, si;
    sincos(2 * M_PI * a.freq[f] * (c < 3 ? (step + 1) * a.dt : (step + 0.5) * a.dt), &si, &co);
    neumaier(sm.x, cp.x, v * co);
    neumaier(sm.y, cp.y, v * si);
    a.acc[o] = sm;
    a.cmp[o] = cp;
}
// the region of pair g
template <typename T>
__device__ __forceinline__ int dft_region(const DftDev<T>* __restrict__ regs, const int nreg, const long g) {
    int ri = 0;
    for (int hi = nreg - 1; ri < hi;) {  // region with first <= g
        const int mid = (ri + hi + 1) / 2;
        if (regs[mid].first <= g) ri = mid;
        else hi = mid - 1;
    }
    return ri;
}
template <typename T>
__device__ __forceinline__ void dft_block(const DftDev<T>* __restrict__ regs, const int nreg, const long total,
                                          const int bx, const int f) {
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const long g0 = (long)bx * 256 + wave * 64, g = g0 + (threadIdx.x & 63);
    if (g0 >= total) return;
    // a wavefront within one region reads its description as scalars
    const int ri = dft_region(regs, nreg, g0);
    if (g0 + 63 < (ri + 1 < nreg ? regs[ri + 1].first : total)) {
        if (total < 0x7fffffff) dft_cell<T, uint32_t>(regs[ri], g, f);
        else dft_cell<T, long>(regs[ri], g, f);
    } else if (g < total) {
        dft_cell<T, long>(regs[dft_region(regs, nreg, g)], g, f);
    }
}

// (the frequency is the grid's y: regions of many pairs beside one of many frequencies have more threads
// than HIP takes along one dimension)
template <typename T>
__global__ void __launch_bounds__(256) k_dft(const DftDev<T>* __restrict__ regs, int nreg, long total, const Tick tk) {
    dft_block(regs, nreg, total, blockIdx.x, blockIdx.y);
    advance(tk);
}

// Source injection and DFT in one launch, for steps whose DFT regions hold no source cell (so
// neither part reads what the other writes): workgroups [0, nsrc) inject, the rest accumulate (dftx per
// frequency; a launch too large for one grid dimension goes out as two).
template <typename T>
__global__ void __launch_bounds__(256) k_source_dft(const SrcTables<T> t, int nsrc, const DftDev<T>* __restrict__ regs,
                                                    int nreg, long total, int dftx, const Tick tk) {
    const int b = blockIdx.x;
    if (b < nsrc) {
        source_block(t, b);
    } else {
        const int f = (b - nsrc) / dftx;
        dft_block(regs, nreg, total, b - nsrc - f * dftx, f);
    }
    advance(tk);
}

// ---- flux through a DFT plane ------------------------------------------------------------
// out[f] = dA * Re sum_cells (E_a conj(H_b) - E_b conj(H_a)) for each frequency f, with each
// spectrum value acc + cmp of the region's [slot][f][cell] accumulators (sa, sb, ha, hb: the slots
// of E_a, E_b, H_a, H_b).  Two launches, both in a fixed order, so the result does not vary from
// run to run:
//   k_dft_flux_part, grid (nb, nf): workgroup (b, f) sums cells b*256 + t + m*nb*256 in FP64 per
//     thread, the wavefronts reduce by shuffles and the first thread adds the wavefront sums in
//     order into part[f * nb + b];
//   k_dft_flux_sum, one thread per frequency: out[f] = dA * (part[f*nb] + ... + part[f*nb + nb-1]).
__global__ void __launch_bounds__(256) k_dft_flux_part(const double2* __restrict__ acc, const double2* __restrict__ cmp,
                                                       long ncell, int nf, int sa, int sb, int ha, int hb, int nb,
                                                       double* __restrict__ part) {
    const int b = blockIdx.x, f = blockIdx.y;
    auto value = [&](int slot, long c) {
        const long o = ((long)slot * nf + f) * ncell + c;
        const double2 x = acc[o], y = cmp[o];
        return make_double2(x.x + y.x, x.y + y.y);
    };
    double sum = 0;
    const long stride = (long)nb * blockDim.x;
    for (long c = (long)b * blockDim.x + threadIdx.x; c < ncell; c += stride) {
        const double2 ea = value(sa, c), eb = value(sb, c), Ha = value(ha, c), Hb = value(hb, c);
        sum += (ea.x * Hb.x + ea.y * Hb.y) - (eb.x * Ha.x + eb.y * Ha.y);
    }
    for (int off = 32; off > 0; off >>= 1) sum += __shfl_down(sum, off, 64);
    __shared__ double wsum[4];
    if ((threadIdx.x & 63) == 0) wsum[threadIdx.x >> 6] = sum;
    __syncthreads();
    if (threadIdx.x == 0) {
        double t = 0;
        for (int w = 0; w < (int)(blockDim.x + 63) / 64; ++w) t += wsum[w];
        part[(long)f * nb + b] = t;
    }
}

__global__ void __launch_bounds__(64) k_dft_flux_sum(const double* __restrict__ part, int nf, int nb, double dA,
                                                     double* __restrict__ out) {
    const int f = threadIdx.x;
    if (f >= nf) return;
    double t = 0;
    for (int b = 0; b < nb; ++b) t += part[(long)f * nb + b];
    out[f] = t * dA;
}

// ===================================================== adjoint (reverse-mode) kernels ======
// Exact transpose of one k_step update (Yee curls, CPML recursions, (P, Q) pole recursions),
// applied backwards in time to the adjoint state (Ebar, Hbar, Qbar, Pbar, psiEbar, psiHbar).
// With b the CPML decay of a derivative term and a = b - 1, the forward term
//   d~ = b (d + psi),  psi' = b psi + (b - 1) d
// transposes to  dbar = b dbar~ + (b - 1) psibar',  psibar = b (dbar~ + psibar').
// Non-PML terms have b = 1.  The adjoint of a backward difference e(r) = H(r) - H(r-1) adds
// ebar(q) - ebar(q+1) to Hbar(q); the adjoint of a forward difference d(r) = E(r+1) - E(r)
// adds dbar(q-1) - dbar(q) to Ebar(q); positions outside a metallic edge contribute zero.
// One fused launch per reverse step (adj_tile) does both halves:
//   phase 1, Hbar_total(q) = Hbar'(q) + sum over E-terms [ebar(q) - ebar(q + e_d)], and the new
//            H auxiliary bars psiHbar = bH (-s cdt Hbar_total + psiHbar');
//   phase 2, Ebar(q) = Ebar'(q) + sum over H-terms [dbar(q - e_d) - dbar(q)] + the pole
//            recursions, and the new E auxiliary bars psiEbar = bE (s cdt u + psiEbar');
// with u = inv_eps Ebar', ebar = s cdt u (PML: bE s cdt u + (bE - 1) psiEbar'), dbar = -s cdt
// Hbar_total (PML: bH (-s cdt Hbar_total) + (bH - 1) psiHbar').  The terms, as (E comp, axis,
// sign, H comp, aux slot on that axis):
//   E-terms: (Ex, y, +, Hz, 0) (Ex, z, -, Hy, 0) (Ey, z, +, Hx, 1) (Ey, x, -, Hz, 0)
//            (Ez, x, +, Hy, 1) (Ez, y, -, Hx, 1)
//   H-terms: (Hx, y, +, Ez, 0) (Hx, z, -, Ey, 0) (Hy, z, +, Ex, 1) (Hy, x, -, Ez, 0)
//            (Hz, x, +, Ey, 1) (Hz, y, -, Ex, 1)
// This has the dependency pattern of the forward step (phase 1 uses forward differences,
// phase 2 backward ones), so the same tilings apply: rows of threads (adj_rows), or a workgroup that
// spans a z line, each thread one y row plus a halo row below it where phase 1 is recomputed, z
// neighbours through LDS (adj_tile); the tile marches along x carrying u of the next planes.  Adjoint
// fields and E auxiliary bars are double-buffered (neighbouring workgroups read the old values of the
// halo row); Qbar and Pbar are only touched by their owner and are updated in place.

template <typename T>
struct AdjArgs {
    StepArgs<T> f;     // forward description (geometry, materials, PML tables, tiles)
    T* A[2];           // adjoint field sets [x][Ubar x,y,z, Hbar x,y,z][y][z] with Ubar = Ebar / eps:
                       // read A[rd], write A[1 - rd]
    int rd;
    T* Aq;             // Qbar [x][slot * 3 + comp][y][z]
    T* Ap;             // Pbar, the same layout
    T* Apsi[3];        // per axis four pairs of auxiliary bars [S][2]: E at 0 and 6 S, H at 2 S and 4 S
    int er, ew;        // E pair read (0 or 6) / written (6 or 0)
    int hr, hw;        // H pair read (2 or 4) / written (4 or 2)
};

// b dbar + (b - 1) psibar of a term and its auxiliary bar
template <typename T>
__device__ __forceinline__ T adj_term(T b, T t, T psi) { return fma_(b - T(1), psi, b * t); }

// One tile of the fused reverse step: a z line of one y row (j0), marching along x.  Addressing
// and predication as in step_tile: per-plane descriptors, lane offsets fixed for the march, the
// out-of-range offset for ghost rows and for lanes past the z line, outside a z PML layer, a
// pole slot or the design region; whole-wavefront conditions are uniform branches.
template <typename T, int NP, bool NTS>
__device__ __forceinline__ void adj_tile(const AdjArgs<T>& g, const int t) {
#pragma clang fp contract(off)
    typedef Pair2<T> Pair;
    constexpr uint32_t TS = sizeof(T);
    const StepArgs<T>& a = g.f;
    extern __shared__ __align__(16) unsigned char smem_raw[];
    const int B = blockDim.x;
    T* se = reinterpret_cast<T*>(smem_raw);  // [2 parity][4][B]: z E-terms of rows -1 and 0
    T* sd = se + 8 * B;                      // [2 parity][2][B]: z H-terms of row 0
    MatLut<T>* slut = reinterpret_cast<MatLut<T>*>(sd + 4 * B);
    copy_lut(a, slut);
    const char* AR = (const char*)g.A[g.rd];
    const char* AW = (const char*)g.A[1 - g.rd];
    const char* matw = (const char*)a.matw;
    GLOBAL const T* coef = (GLOBAL const T*)a.coef;
    const int nx = a.nx, ny = a.ny, nz = a.nz;
    const int j0 = t % a.nty, xci = t / a.nty;
    const int x0 = xci * a.xc, x1 = min(x0 + a.xc, nx);
    const int k = threadIdx.x;
    const bool kin = k < nz;
    const int kp1 = wrap_or_ghost(k + 1, nz, a.pz), km1 = wrap_or_ghost(k - 1, nz, a.pz);
    const T cdt = a.cdt;
    const bool uniform = a.uniform != 0;
    const uint32_t er = g.er, ew = g.ew, hr = g.hr, hw = g.hw;
    const uint32_t PB = (uint32_t)ny * (uint32_t)nz * TS;  // bytes of one component plane
    const long FPB = 6L * PB, QPB = (long)a.nqp * PB, PW = (long)ny * nz * 4;
    const int Ly = a.plo[1] + a.phi[1], Lz = a.plo[2] + a.phi[2];
    const uint32_t SB0 = (uint32_t)(a.S[0] * TS), SB1 = (uint32_t)(a.S[1] * TS), SB2 = (uint32_t)(a.S[2] * TS);
    const Rsrc rpx = rsrc(g.Apsi[0]), rpy = rsrc(g.Apsi[1]), rpz = rsrc(g.Apsi[2]);
    // rows: 0 = j0 - 1 (halo), 1 = j0 (owned), 2 = j0 + 1 (its +y neighbour); uniform validity
    int gj[3], sy[3];
    bool rv[3], ypml[3];
    uint32_t oR[3], oW[3];
#pragma unroll
    for (int r = 0; r < 3; ++r) {
        gj[r] = wrap_or_ghost(j0 + r - 1, ny, a.py);
        rv[r] = gj[r] >= 0;
        ypml[r] = rv[r] && in_pml(a, 1, gj[r], ny);
        sy[r] = ypml[r] ? (gj[r] < a.plo[1] ? gj[r] : gj[r] - (ny - a.phi[1]) + a.plo[1]) : 0;
        const bool ok = rv[r] && kin;
        oR[r] = ok ? (uint32_t)(gj[r] * nz + k) * TS : kOOB;
        oW[r] = ok ? (uint32_t)(gj[r] * nz + k) * 4u : kOOB;
    }
    const bool zpml = kin && in_pml(a, 2, k, nz);
    const bool zany = wave_any(zpml);
    const uint32_t oK = kin ? (uint32_t)k * 2u * TS : kOOB;  // in a y slab
    const uint32_t oZ = zpml ? (uint32_t)(k < a.plo[2] ? k : k - (nz - a.phi[2]) + a.plo[2]) * 2u * TS : kOOB;
    GLOBAL const T* cy = coef + a.coff[1];
    GLOBAL const T* cz = coef + a.coff[2];
    GLOBAL const T* cx = coef + a.coff[0];
    const T bEz = zpml ? cz[k] : T(1), bHz = zpml ? cz[2 * nz + k] : T(1);
    const Rsrc rd = rsrc(a.dinv);
    const int dey = a.dhi[1] - a.dlo[1], dez = a.dhi[2] - a.dlo[2];

    const int istart = (x0 > 0 || a.px) ? x0 - 1 : x0;
    // u = Ubar' (the state itself) on planes i and i + 1 (rows 0..2; plane i + 1 is loaded with
    // the other loads of iteration i) and the owned row's material word of both planes
    T uc[3][3], un[3][3];
    uint32_t wc1 = 0u, wn1 = 0u;
    auto load_u = [&](int p, T (&u)[3][3], uint32_t& w1) {
        const int pp = wrap_or_ghost(p, nx, a.px);
        const long pc = pp >= 0 ? pp : 0;
        const Rsrc rf = rsrc(AR + pc * FPB);
#pragma unroll
        for (int r = 0; r < 3; ++r) {
            const uint32_t o = pp >= 0 ? oR[r] : kOOB;
#pragma unroll
            for (int c = 0; c < 3; ++c) u[r][c] = bld<T>(rf, o, c * PB);
        }
        w1 = uniform ? 0u : bld<uint32_t>(rsrc(matw + pc * PW), pp >= 0 ? oW[1] : kOOB, 0);
    };
    lds_barrier();  // LUT in LDS
    load_u(istart, uc, wc1);
    T dbx_prev[2] = {T(0), T(0)};  // x H-terms of row 0 on plane i - 1: (Hz -> Ey), (Hy -> Ez)

    for (int i = istart; i < x1; ++i) {
        const bool own_plane = i >= x0;
        const int pi = wrap_or_ghost(i, nx, a.px);
        const int pn = wrap_or_ghost(i + 1, nx, a.px);
        load_u(i + 1, un, wn1);
        const bool xpml = in_pml(a, 0, pi, nx);
        const bool xpmln = pn >= 0 && in_pml(a, 0, pn, nx);
        const uint32_t sxo = xpml ? (uint32_t)(pi < a.plo[0] ? pi : pi - (nx - a.phi[0]) + a.plo[0]) * 2u * PB : 0u;
        const uint32_t sxn = xpmln ? (uint32_t)(pn < a.plo[0] ? pn : pn - (nx - a.phi[0]) + a.plo[0]) * 2u * PB : 0u;
        const T bEx = xpml ? cx[pi] : T(1), bHx = xpml ? cx[2 * nx + pi] : T(1);
        const T bExn = xpmln ? cx[pn] : T(1);
        const Rsrc rA = rsrc(AR + (long)pi * FPB);
        const Rsrc rB = rsrc(AW + (long)pi * FPB);

        // ---- the global loads of plane i, issued together (u of the planes ahead is already in
        // flight): Hbar' of rows -1 and 0, the z auxiliary bars, the owned cell's design 1/eps
        // and pole state; the y and x auxiliary bars (layers of a few tiles) are loaded in place
        T hb[2][3];
#pragma unroll
        for (int r = 0; r < 2; ++r)
#pragma unroll
            for (int c = 0; c < 3; ++c) hb[r][c] = bld<T>(rA, oR[r], (3 + c) * PB);
        Pair pzE[2] = {Pair{T(0), T(0)}, Pair{T(0), T(0)}}, phz = Pair{T(0), T(0)};
        if (zany) {  // lanes outside the layers: b = 1 and a zero auxiliary
#pragma unroll
            for (int r = 0; r < 2; ++r) {
                if (!rv[r]) continue;
                const uint32_t so = (uint32_t)((pi * ny + gj[r]) * Lz) * 2u * TS;
                pzE[r] = bld2<T>(rpz, oZ, er * SB2 + so);
                if (r == 1) phz = bld2<T>(rpz, oZ, hr * SB2 + so);
            }
        }
        const bool wr = own_plane && rv[1];
        // material of the owned cell: pole count per component and the LUT entry (design voxels:
        // 1/eps from the design array, no poles)
        int mm[3] = {0, 0, 0}, npl[3] = {0, 0, 0};
        bool des[3] = {false, false, false};
        T dv[3];
        bool desany = false;
        uint32_t sact = 0u;  // pole slots some lane of the wavefront uses (uniform)
        T qv[NP > 0 ? NP : 1][3], pv[NP > 0 ? NP : 1][3];
        if (wr && !uniform) {
#pragma unroll
            for (int c = 0; c < 3; ++c) {
                const int m = (wc1 >> (8 * c)) & 0xff;
                des[c] = m == a.nmat;
                mm[c] = des[c] ? 0 : m;
                npl[c] = des[c] ? 0 : slut[mm[c]].np;
            }
            desany = wave_any(des[0] || des[1] || des[2]);
            if (desany) {
                const uint32_t dq =
                    (uint32_t)(((pi - a.dlo[0]) * dey + (gj[1] - a.dlo[1])) * dez + (k - a.dlo[2])) * TS;
#pragma unroll
                for (int c = 0; c < 3; ++c) dv[c] = bld<T>(rd, des[c] ? dq : kOOB, 0);
            }
            if (NP > 0) {
                const uint32_t o = oR[1];
                const Rsrc rQ = rsrc((const char*)g.Aq + (long)pi * QPB);
                const Rsrc rP = rsrc((const char*)g.Ap + (long)pi * QPB);
#pragma unroll
                for (int s = 0; s < NP; ++s) {
                    if (!wave_any(s < npl[0] || s < npl[1] || s < npl[2])) continue;
                    sact |= 1u << s;
#pragma unroll
                    for (int c = 0; c < 3; ++c) {
                        const bool vq = s < npl[c];
                        const bool vp = vq && ((slut[mm[c]].lorentz_mask >> s) & 1);
                        const uint32_t so = (s * 3 + c) * PB;
                        pv[s][c] = bld<T>(rP, vp ? o : kOOB, so);
                        qv[s][c] = bld<T>(rQ, vq ? o : kOOB, so);
                    }
                }
            }
        }

        // ---- phase 1: E-terms and Hbar_total on rows -1 and 0 of plane i ----------------
        // E-terms on rows r = 0, 1 (labels: y (Ex->Hz), z (Ex->Hy), z (Ey->Hx), x (Ey->Hz),
        // x (Ez->Hy), y (Ez->Hx)) and the y-terms of row 2
        T eb[3][6];
        // (the new E auxiliary bars of the owned row are stored as soon as its terms are formed)
#pragma unroll
        for (int r = 0; r < 3; ++r) {
            const bool ok = rv[r];
            const int j = gj[r];
            const T ux = uc[r][0], uy = uc[r][1], uz = uc[r][2];
            T t_ex_y = cdt * ux, t_ex_z = -cdt * ux, t_ey_z = cdt * uy, t_ey_x = -cdt * uy, t_ez_x = cdt * uz,
              t_ez_y = -cdt * uz;
            if (ypml[r]) {
                const T b = cy[j];
                const uint32_t so = (uint32_t)((pi * Ly + sy[r]) * nz) * 2u * TS;
                const Pair q = bld2<T>(rpy, oK, er * SB1 + so);
                t_ex_y = adj_term(b, t_ex_y, q.x);
                t_ez_y = adj_term(b, t_ez_y, q.y);
                if (r == 1 && wr)  // (Ex, y, +, slot 0), (Ez, y, -, slot 1)
                    bst2<NTS>(rpy, oK, ew * SB1 + so, Pair{b * (cdt * ux + q.x), b * (-cdt * uz + q.y)});
            }
            if (r < 2) {
                if (ok && zany) {
                    if (r == 1 && wr)  // (Ex, z, -, slot 0), (Ey, z, +, slot 1)
                        bst2<NTS>(rpz, oZ, ew * SB2 + (uint32_t)((pi * ny + j) * Lz) * 2u * TS,
                                  Pair{bEz * (-cdt * ux + pzE[1].x), bEz * (cdt * uy + pzE[1].y)});
                    t_ex_z = adj_term(bEz, t_ex_z, pzE[r].x);
                    t_ey_z = adj_term(bEz, t_ey_z, pzE[r].y);
                }
                if (ok && xpml) {
                    const Pair q = bld2<T>(rpx, two(oR[r]), er * SB0 + sxo);
                    t_ey_x = adj_term(bEx, t_ey_x, q.x);
                    t_ez_x = adj_term(bEx, t_ez_x, q.y);
                    if (r == 1 && wr)  // (Ey, x, -, slot 0), (Ez, x, +, slot 1)
                        bst2<NTS>(rpx, two(oR[1]), ew * SB0 + sxo, Pair{bEx * (-cdt * uy + q.x), bEx * (cdt * uz + q.y)});
                }
            }
            eb[r][0] = t_ex_y;
            eb[r][1] = t_ex_z;
            eb[r][2] = t_ey_z;
            eb[r][3] = t_ey_x;
            eb[r][4] = t_ez_x;
            eb[r][5] = t_ez_y;
        }
        // x-terms of plane i + 1, rows 0 and 1
        T ebn[2][2];
#pragma unroll
        for (int r = 0; r < 2; ++r) {
            T a1 = -cdt * un[r][1], a2 = cdt * un[r][2];  // (Ey -> Hz), (Ez -> Hy)
            if (rv[r] && xpmln) {
                const Pair q = bld2<T>(rpx, two(oR[r]), er * SB0 + sxn);
                a1 = adj_term(bExn, a1, q.x);
                a2 = adj_term(bExn, a2, q.y);
            }
            ebn[r][0] = (rv[r] && pn >= 0) ? a1 : T(0);
            ebn[r][1] = (rv[r] && pn >= 0) ? a2 : T(0);
        }
        // z-terms through LDS
        T* bufe = se + (i & 1) * 4 * B;
#pragma unroll
        for (int r = 0; r < 2; ++r) {
            bufe[(2 * r + 0) * B + k] = eb[r][1];  // (Ex -> Hy)
            bufe[(2 * r + 1) * B + k] = eb[r][2];  // (Ey -> Hx)
        }
        lds_barrier();
        T tot[2][3];
#pragma unroll
        for (int r = 0; r < 2; ++r) {
            const bool ok = rv[r];
            const T exz_k = kp1 >= 0 ? bufe[(2 * r + 0) * B + kp1] : T(0);
            const T eyz_k = kp1 >= 0 ? bufe[(2 * r + 1) * B + kp1] : T(0);
            // Hx: (Ey, z) and (Ez, y); Hy: (Ex, z) and (Ez, x); Hz: (Ex, y) and (Ey, x)
            tot[r][0] = ok ? hb[r][0] + (eb[r][2] - eyz_k) + (eb[r][5] - eb[r + 1][5]) : T(0);
            tot[r][1] = ok ? hb[r][1] + (eb[r][1] - exz_k) + (eb[r][4] - ebn[r][1]) : T(0);
            tot[r][2] = ok ? hb[r][2] + (eb[r][0] - eb[r + 1][0]) + (eb[r][3] - ebn[r][0]) : T(0);
        }
        // H auxiliary bars of the owned row (read by the update below and by phase 2)
        Pair phy = Pair{T(0), T(0)}, phx = Pair{T(0), T(0)};
        if (ypml[1]) {
            const uint32_t so = (uint32_t)((pi * Ly + sy[1]) * nz) * 2u * TS;
            phy = bld2<T>(rpy, oK, hr * SB1 + so);
        }
        if (rv[1] && xpml) phx = bld2<T>(rpx, two(oR[1]), hr * SB0 + sxo);
        // own row: Hbar at the old time and the new H auxiliary bars
        if (wr) {
            const int j = gj[1];
            bst<NTS>(rB, oR[1], 3 * PB, tot[1][0]);
            bst<NTS>(rB, oR[1], 4 * PB, tot[1][1]);
            bst<NTS>(rB, oR[1], 5 * PB, tot[1][2]);
            if (ypml[1]) {  // (Hx, y, +, slot 0), (Hz, y, -, slot 1)
                const T b = cy[2 * ny + j];
                const uint32_t so = (uint32_t)((pi * Ly + sy[1]) * nz) * 2u * TS;
                bst2<NTS>(rpy, oK, hw * SB1 + so, Pair{b * (-cdt * tot[1][0] + phy.x), b * (cdt * tot[1][2] + phy.y)});
            }
            if (zany) {  // (Hx, z, -, slot 0), (Hy, z, +, slot 1)
                const uint32_t so = (uint32_t)((pi * ny + j) * Lz) * 2u * TS;
                bst2<NTS>(rpz, oZ, hw * SB2 + so, Pair{bHz * (cdt * tot[1][0] + phz.x), bHz * (-cdt * tot[1][1] + phz.y)});
            }
            if (xpml) {  // (Hy, x, -, slot 0), (Hz, x, +, slot 1)
                bst2<NTS>(rpx, two(oR[1]), hw * SB0 + sxo, Pair{bHx * (cdt * tot[1][1] + phx.x), bHx * (-cdt * tot[1][2] + phx.y)});
            }
        }

        // ---- phase 2: H-terms and Ebar on row 0 of plane i --------------------------------
        // H-terms of row 0: (Hx, y) (Hx, z) (Hy, z) (Hy, x) (Hz, x) (Hz, y); y-terms of row -1
        T db[6], dbh[2];
        {
            const int j = gj[1];
            T d_hx_y = -cdt * tot[1][0], d_hx_z = cdt * tot[1][0], d_hy_z = -cdt * tot[1][1], d_hy_x = cdt * tot[1][1],
              d_hz_x = -cdt * tot[1][2], d_hz_y = cdt * tot[1][2];
            if (ypml[1]) {
                const T b = cy[2 * ny + j];
                d_hx_y = adj_term(b, d_hx_y, phy.x);
                d_hz_y = adj_term(b, d_hz_y, phy.y);
            }
            if (rv[1] && zany) {
                d_hx_z = adj_term(bHz, d_hx_z, phz.x);
                d_hy_z = adj_term(bHz, d_hy_z, phz.y);
            }
            if (rv[1] && xpml) {
                d_hy_x = adj_term(bHx, d_hy_x, phx.x);
                d_hz_x = adj_term(bHx, d_hz_x, phx.y);
            }
            db[0] = d_hx_y;
            db[1] = d_hx_z;
            db[2] = d_hy_z;
            db[3] = d_hy_x;
            db[4] = d_hz_x;
            db[5] = d_hz_y;
        }
        {
            const int j = gj[0];
            T d_hx_y = -cdt * tot[0][0], d_hz_y = cdt * tot[0][2];
            if (ypml[0]) {
                const T b = cy[2 * ny + j];
                const uint32_t so = (uint32_t)((pi * Ly + sy[0]) * nz) * 2u * TS;
                const Pair q = bld2<T>(rpy, oK, hr * SB1 + so);
                d_hx_y = adj_term(b, d_hx_y, q.x);
                d_hz_y = adj_term(b, d_hz_y, q.y);
            }
            dbh[0] = rv[0] ? d_hx_y : T(0);
            dbh[1] = rv[0] ? d_hz_y : T(0);
        }
        if (own_plane) {
            T* bufd = sd + (i & 1) * 2 * B;
            bufd[0 * B + k] = db[2];  // (Hy -> Ex)
            bufd[1 * B + k] = db[1];  // (Hx -> Ey)
            lds_barrier();
            if (wr) {
                const int j = gj[1];
                const uint32_t o = oR[1];
                const T hyz_k = km1 >= 0 ? bufd[0 * B + km1] : T(0);
                const T hxz_k = km1 >= 0 ? bufd[1 * B + km1] : T(0);
                // Ex: (Hy, z) and (Hz, y); Ey: (Hx, z) and (Hz, x); Ez: (Hx, y) and (Hy, x)
                const T u0[3] = {uc[1][0], uc[1][1], uc[1][2]};
                // the differences of each component; sum of the pole terms
                const T x[3] = {(hyz_k - db[2]) + (dbh[1] - db[5]), (hxz_k - db[1]) + (dbx_prev[0] - db[4]),
                                (dbh[0] - db[0]) + (dbx_prev[1] - db[3])};
                T sq[3] = {T(0), T(0), T(0)};
                if (NP > 0 && !uniform) {
                    const Rsrc rQ = rsrc((const char*)g.Aq + (long)pi * QPB);
                    const Rsrc rP = rsrc((const char*)g.Ap + (long)pi * QPB);
#pragma unroll
                    for (int s = 0; s < NP; ++s) {
                        if (!((sact >> s) & 1u)) continue;
#pragma unroll
                        for (int c = 0; c < 3; ++c) {
                            const MatLut<T>& L = slut[mm[c]];
                            const bool vq = s < npl[c];
                            const bool vp = vq && ((L.lorentz_mask >> s) & 1);
                            const uint32_t so = (s * 3 + c) * PB;
                            const T pb = pv[s][c];
                            const T qb = vq ? qv[s][c] + pb - u0[c] : T(0);
                            bst<NTS>(rQ, vq ? o : kOOB, so, L.pole[s].alpha * qb);
                            bst<NTS>(rP, vp ? o : kOOB, so, fma_(L.pole[s].beta, qb, pb));
                            sq[c] = fma_(L.pole[s].c3, qb, sq[c]);
                        }
                    }
                }
                // the state is Ubar = Ebar / eps: the differences and the pole terms add 1/eps of their sum
#pragma unroll
                for (int c = 0; c < 3; ++c) {
                    T inv = slut[mm[c]].inv_eps;
                    if (desany) inv = des[c] ? dv[c] : inv;
                    bst<NTS>(rB, o, c * PB, fma_(inv, x[c] + sq[c], u0[c]));
                }
            }
        } else {
            lds_barrier();  // keep the barrier count uniform across iterations
        }
        dbx_prev[0] = rv[1] ? db[4] : T(0);
        dbx_prev[1] = rv[1] ? db[3] : T(0);
#pragma unroll
        for (int r = 0; r < 3; ++r)
#pragma unroll
            for (int c = 0; c < 3; ++c) uc[r][c] = un[r][c];
        wc1 = wn1;
    }
}

// One tile of the fused reverse step, row-of-threads form.  A workgroup holds a.rt rows of nz
// threads (one cell of a y row per thread): thread row 0 is the row below the tile, rows
// 1..rt-1 own rows j0..j0+rt-2, and the top thread row also forms the y-terms of the row above
// the tile.  The y and z neighbours' E-terms (for Hbar) and H-terms (for Ebar) pass through LDS,
// so each adjoint value is loaded once per tile and the y halo costs one row per rt-1 owned
// rows.  The arithmetic of every cell is that of adj_tile, bit for bit.
// Pipelined as step_rows is: every register is loaded for the plane that needs it next as soon as it
// has been read, the loop starts with the Ebar phase, and one barrier per plane publishes both the
// H-terms of plane i and the E-terms of plane i + 1 (which Hbar of plane i needs anyway), each in two
// halves used in turn.  The plane before the chunk runs as an iteration whose stores are dropped.
// Bound by latency and by the pole state's four accesses per slot; us per reverse step on MI355X
// before (this form with the loads of a plane waited for in its iteration, and one row per workgroup)
// and now: FP32 192x192x96 138 (one row), 93; 120x120x256 122, 80; FP64 72x64x56 33 (one row), 22.
template <typename T, int NP, bool NTS>
__device__ __forceinline__ void adj_rows(const AdjArgs<T>& g, const int t) {
#pragma clang fp contract(off)
    constexpr uint32_t W = sizeof(T);
    constexpr int NS = NP > 0 ? NP : 1;
    typedef Pair2<T> Pair;
    const StepArgs<T>& a = g.f;
    extern __shared__ __align__(16) unsigned char smem_raw[];
    const int B = blockDim.x;
    Pair* sEz = reinterpret_cast<Pair*>(smem_raw);  // [2][B] E-terms (Ex->Hy, Ey->Hx) along z
    Pair* sEy = sEz + 2 * B;                        // [2][B] E-terms (Ex->Hz, Ez->Hx) along y
    Pair* sDz = sEy + 2 * B;                        // [2][B] H-terms (Hy->Ex, Hx->Ey) along z
    Pair* sDy = sDz + 2 * B;                        // [2][B] H-terms (Hx->Ez, Hz->Ex) along y
    MatLut<T>* slut = reinterpret_cast<MatLut<T>*>(sDy + 2 * B);
    copy_lut(a, slut);

    const char* A0 = (const char*)g.A[g.rd];
    const long A01 = (const char*)g.A[1 - g.rd] - A0;  // from the set read to the set written
    CONST const T* coef = (CONST const T*)a.coef;
    CONST const MatLut<T>* clut = (CONST const MatLut<T>*)a.lut;
    const int nx = a.nx, ny = a.ny, nz = a.nz;
    const int RT = a.rt, R = RT - 1;
    const int tid = threadIdx.x;
    const bool act = tid < RT * nz;
    const int r = act ? tid / nz : 0;
    const int k = act ? tid - r * nz : 0;
    const int xci = t / a.nty, tyi = t - xci * a.nty;
    const int jr = tyi * R + r - 1;  // unwrapped global row of this thread row
    const int j = act ? wrap_or_ghost(jr, ny, a.py) : -1;
    const bool valid = j >= 0;
    const bool owned = act && r >= 1 && jr < ny;  // implies valid
    const bool top = act && r == RT - 1;
    const int ju = act ? wrap_or_ghost(jr + 1, ny, a.py) : -1;  // the row above
    const int kp1 = k + 1 < nz ? k + 1 : a.pz ? 0 : -1;
    const int km1 = k > 0 ? k - 1 : a.pz ? nz - 1 : -1;
    const T cdt = a.cdt;
    const bool uniform = a.uniform != 0;
    const uint32_t PB = (uint32_t)ny * (uint32_t)nz * W;  // bytes of one component plane
    const long FPB = 6L * PB, QPB = (long)a.nqp * PB, PW = (long)ny * nz * 4;
    const int Ly = a.plo[1] + a.phi[1], Lz = a.plo[2] + a.phi[2];
    const uint32_t YP = (uint32_t)(Ly * nz) * 2u * W, ZP = (uint32_t)(ny * Lz) * 2u * W;  // bytes of a slab per plane
    const uint32_t S0 = (uint32_t)(a.S[0] * W), S1 = (uint32_t)(a.S[1] * W), S2 = (uint32_t)(a.S[2] * W);
    const uint32_t er0 = g.er * S0, er1 = g.er * S1, er2 = g.er * S2, ew0 = g.ew * S0, ew1 = g.ew * S1, ew2 = g.ew * S2;
    const uint32_t hr0 = g.hr * S0, hr1 = g.hr * S1, hr2 = g.hr * S2, hw0 = g.hw * S0, hw1 = g.hw * S1, hw2 = g.hw * S2;
    const int xlo = a.pml_on[0] ? a.plo[0] : 0;
    const unsigned xin = a.pml_on[0] ? (unsigned)(nx - a.phi[0] - a.plo[0]) : 0xffffffffu;
    auto in_x = [&](int p) { return p < nx && (unsigned)(p - xlo) >= xin; };
    auto xslab = [&](int p) -> uint32_t { return (uint32_t)(p < a.plo[0] ? p : p - (nx - a.phi[0]) + a.plo[0]) * 2u * PB; };
    CONST const T* cx = coef + a.coff[0];

    // lane offsets; kOOB for lanes that neither read nor write
    const uint32_t oc = valid ? ((uint32_t)j * nz + k) * W : kOOB;            // the cell
    const uint32_t oo = owned ? oc : kOOB;                                    // owned cells
    const uint32_t ot = top && ju >= 0 ? ((uint32_t)ju * nz + k) * W : kOOB;  // the row above the tile
    const uint32_t ow = owned ? ((uint32_t)j * nz + k) * 4u : kOOB;           // material words
    const bool ypml = valid && in_pml(a, 1, j, ny);
    const bool tpml = top && ju >= 0 && in_pml(a, 1, ju, ny);
    const bool zpml = valid && in_pml(a, 2, k, nz);
    auto yrow = [&](int q) { return (uint32_t)((q < a.plo[1] ? q : q - (ny - a.phi[1]) + a.plo[1]) * nz + k) * 2u * W; };
    const uint32_t oy = ypml ? yrow(j) : kOOB, oyt = tpml ? yrow(ju) : kOOB;
    const uint32_t oz = zpml ? (uint32_t)(j * Lz + (k < a.plo[2] ? k : k - (nz - a.phi[2]) + a.plo[2])) * 2u * W : kOOB;
    const uint32_t oyw = owned ? oy : kOOB, ozw = owned ? oz : kOOB;
    // wavefront-uniform summaries of the per-lane conditions
    const bool yany = wave_any(ypml), zany = wave_any(zpml), tany = wave_any(ot != kOOB), tyany = wave_any(tpml);
    GLOBAL const T* cy = (GLOBAL const T*)a.coef + a.coff[1];
    GLOBAL const T* cz = (GLOBAL const T*)a.coef + a.coff[2];
    const T bEz = zpml ? cz[k] : T(1), bHz = zpml ? cz[2 * nz + k] : T(1);
    const T bEy = ypml ? cy[j] : T(1), bHy = ypml ? cy[2 * ny + j] : T(1);
    const T bEt = tpml ? cy[ju] : T(1);
    // exchange slots of the row above (top row: tu), the row below and the z neighbours
    const int up = (top || !act) ? tid : tid + nz, dn = owned ? tid - nz : tid;
    const int kup = kp1 >= 0 ? r * nz + kp1 : tid, kdn = km1 >= 0 ? r * nz + km1 : tid;

    const int x0 = xci * a.xc;
    const int x1 = min(x0 + a.xc, nx);
    const int istart = (x0 > 0 || a.px) ? x0 - 1 : x0;  // the plane before the chunk, where there is one

    // the registers each plane loads anew
    T un[3], ten[2] = {T(0), T(0)};      // u = Ubar' of plane i + 1; (x, z) of the row above the tile
    T hb[3];                             // Hbar' of plane i
    Pair pEx, pEy, pEz, pEt;             // E auxiliary bars of plane i + 1 (pEt: y, the row above the tile)
    Pair pHx, pHy, pHz;                  // H auxiliary bars of plane i
    T Qv[3][NS], Pv[3][NS];              // pole state
    uint32_t mw = 0, mwn = 0;            // material words of planes i, i + 1
    T uc[3];                             // u of plane i
    T tc[6];                             // E-terms of plane i: Ex y, Ex z, Ey z, Ey x, Ez x, Ez y
    T tu[2] = {T(0), T(0)};              // y-terms (Ex, Ez) of the row above the tile, plane i
    T dx[2] = {T(0), T(0)};              // x H-terms (Hz, Hy) of plane i - 1
    T u0[3], inv[3], sq[3], d[6], dv[3];
    uint32_t dw = 0, cls = 0;            // cls: material of the wavefront on plane i (classify)

    auto load_u = [&](const char* f, bool need) {
        const Rsrc rn = rsrc(f, need);
#pragma unroll
        for (int c = 0; c < 3; ++c) un[c] = bld<T>(rn, oc, c * PB);
        if (tany) {
            ten[0] = bld<T>(rn, ot, 0);
            ten[1] = bld<T>(rn, ot, 2 * PB);
        }
    };
    auto load_aux_e = [&](int p, bool yz) {
        if (yz) {
            if (zany) pEz = bld2<T>(rsrc(g.Apsi[2]), oz, er2 + p * ZP);
            if (yany) pEy = bld2<T>(rsrc(g.Apsi[1]), oy, er1 + p * YP);
            if (tyany) pEt = bld2<T>(rsrc(g.Apsi[1]), oyt, er1 + p * YP);
        }
        if (__builtin_expect(in_x(p), 0)) pEx = bld2<T>(rsrc(g.Apsi[0]), two(oc), er0 + xslab(p));
    };
    auto load_h = [&](const char* f, int p, bool need) {
        const Rsrc rn = rsrc(f, need);
#pragma unroll
        for (int c = 0; c < 3; ++c) hb[c] = bld<T>(rn, oc, (3 + c) * PB);
        if (need) {
            if (zany) pHz = bld2<T>(rsrc(g.Apsi[2]), ozw, hr2 + p * ZP);
            if (yany) pHy = bld2<T>(rsrc(g.Apsi[1]), oy, hr1 + p * YP);
            if (__builtin_expect(in_x(p), 0)) pHx = bld2<T>(rsrc(g.Apsi[0]), two(oo), hr0 + xslab(p));
        }
    };
    auto load_poles = [&](int p, uint32_t code, uint32_t w) {
        const int npx = seg_poles(code);
        const Rsrc rq = rsrc((const char*)g.Aq + (long)p * QPB), rp = rsrc((const char*)g.Ap + (long)p * QPB);
        int np[3], lm[3];
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            const MatLut<T>& L = slut[(w >> (8 * c)) & 0xff];
            np[c] = L.np;
            lm[c] = L.lorentz_mask;
        }
#pragma unroll
        for (int s = 0; s < NP; ++s) {
            if (s >= npx) break;
#pragma unroll
            for (int c = 0; c < 3; ++c) {
                Qv[c][s] = bld<T>(rq, s < np[c] ? oo : kOOB, (s * 3 + c) * PB);
                Pv[c][s] = bld<T>(rp, (lm[c] >> s) & 1 ? oo : kOOB, (s * 3 + c) * PB);
            }
        }
    };
    // E-terms te and tt (row above the tile) of plane p from un, ten and the E auxiliary bars, and the new
    // bars (`own`: of a plane of this chunk)
    auto e_terms = [&](int p, bool own, T (&te)[6], T (&tt)[2]) {
        te[0] = cdt * un[0], te[1] = -cdt * un[0], te[2] = cdt * un[1];
        te[3] = -cdt * un[1], te[4] = cdt * un[2], te[5] = -cdt * un[2];
        tt[0] = cdt * ten[0], tt[1] = -cdt * ten[1];
        if (zany) {  // (Ex, z, -, slot 0), (Ey, z, +, slot 1); lanes outside the layers: b = 1
            bst2<NTS>(rsrc(g.Apsi[2], own), ozw, ew2 + p * ZP, Pair{bEz * (te[1] + pEz.x), bEz * (te[2] + pEz.y)});
            te[1] = adj_term(bEz, te[1], pEz.x);
            te[2] = adj_term(bEz, te[2], pEz.y);
        }
        if (yany) {  // (Ex, y, +, slot 0), (Ez, y, -, slot 1)
            bst2<NTS>(rsrc(g.Apsi[1], own), oyw, ew1 + p * YP, Pair{bEy * (te[0] + pEy.x), bEy * (te[5] + pEy.y)});
            te[0] = adj_term(bEy, te[0], pEy.x);
            te[5] = adj_term(bEy, te[5], pEy.y);
        }
        if (tyany) {
            tt[0] = adj_term(bEt, tt[0], pEt.x);
            tt[1] = adj_term(bEt, tt[1], pEt.y);
        }
        if (__builtin_expect(in_x(p), 0)) {  // (Ey, x, -, slot 0), (Ez, x, +, slot 1)
            const T b = cx[p];
            bst2<NTS>(rsrc(g.Apsi[0], own), two(oo), ew0 + xslab(p), Pair{b * (te[3] + pEx.x), b * (te[4] + pEx.y)});
            te[3] = adj_term(b, te[3], pEx.x);
            te[4] = adj_term(b, te[4], pEx.y);
        }
    };

    // ---- the first plane's E-terms
    int pi = istart < 0 ? nx - 1 : istart, pn = wrap_up(pi + 1, nx, a.px), pnn = wrap_up(pn + 1, nx, a.px);
    const char* fW = A0 + (long)pi * FPB;  // plane i, then i + 1 and i + 2, of the set read
    const char* fN = A0 + (long)min(pn, nx - 1) * FPB;
    const char* fNN = A0 + (long)min(pnn, nx - 1) * FPB;
    load_u(fW, true);
    load_aux_e(pi, true);
    load_h(fW, pi, true);
    if (!uniform) {
        mw = bld<uint32_t>(rsrc((const char*)a.matw + (long)pi * PW, istart == x0), ow, 0);
        mwn = bld<uint32_t>(rsrc((const char*)a.matw + (long)min(pn, nx - 1) * PW, istart + 1 < x1), ow, 0);
    }
    e_terms(pi, istart == x0, tc, tu);
#pragma unroll
    for (int c = 0; c < 3; ++c) uc[c] = un[c];
    sEz[(istart & 1) * B + tid] = Pair{tc[1], tc[2]};
    sEy[(istart & 1) * B + tid] = Pair{tc[0], tc[5]};
    lds_barrier();  // also the material table
    load_u(fN, pn < nx);
    load_aux_e(pn, istart + 1 < x1);
    if (!uniform && istart == x0) {
        cls = classify<NP>(mw);
        if (NP > 0 && seg_poles(cls) > 0) load_poles(pi, cls, mw);
    }

    auto h_phase = [&](const int i) __attribute__((always_inline)) {
        const bool own = i >= x0 && i < x1, next = i + 1 < x1;
        const bool xpml = in_x(pi) && i < x1;
        const int half = (i & 1) * B, other = B - half;
        // ------------------------------- E-terms of plane i + 1
        T tn[6], tun[2];
        e_terms(pn, next, tn, tun);
        // ------------------------------- Hbar and the H auxiliary bars of plane i
        {
            const Pair ez = sEz[half + kup], ey = sEy[half + up];
            const T exz = kp1 >= 0 ? ez.x : T(0), eyz = kp1 >= 0 ? ez.y : T(0);
            const T exy = top ? tu[0] : ey.x, ezy = top ? tu[1] : ey.y;
            T tot[3];
            // Hx: (Ey, z) and (Ez, y); Hy: (Ex, z) and (Ez, x); Hz: (Ex, y) and (Ey, x)
            tot[0] = valid ? hb[0] + (tc[2] - eyz) + (tc[5] - ezy) : T(0);
            tot[1] = valid ? hb[1] + (tc[1] - exz) + (tc[4] - tn[4]) : T(0);
            tot[2] = valid ? hb[2] + (tc[0] - exy) + (tc[3] - tn[3]) : T(0);
            const Rsrc rW = rsrc(fW + A01, own);
#pragma unroll
            for (int c = 0; c < 3; ++c) {
                pin(tot[c]);
                bst<NTS>(rW, oo, (3 + c) * PB, tot[c]);
            }
            // H-terms: Hx y, Hx z, Hy z, Hy x, Hz x, Hz y
            d[0] = -cdt * tot[0], d[1] = cdt * tot[0], d[2] = -cdt * tot[1];
            d[3] = cdt * tot[1], d[4] = -cdt * tot[2], d[5] = cdt * tot[2];
            if (yany) {  // (Hx, y, +, slot 0), (Hz, y, -, slot 1)
                bst2<NTS>(rsrc(g.Apsi[1], own), oyw, hw1 + pi * YP, Pair{bHy * (d[0] + pHy.x), bHy * (d[5] + pHy.y)});
                d[0] = adj_term(bHy, d[0], pHy.x);
                d[5] = adj_term(bHy, d[5], pHy.y);
            }
            if (zany) {  // (Hx, z, -, slot 0), (Hy, z, +, slot 1)
                bst2<NTS>(rsrc(g.Apsi[2], own), ozw, hw2 + pi * ZP, Pair{bHz * (d[1] + pHz.x), bHz * (d[2] + pHz.y)});
                d[1] = adj_term(bHz, d[1], pHz.x);
                d[2] = adj_term(bHz, d[2], pHz.y);
            }
            if (__builtin_expect(xpml, 0)) {  // (Hy, x, -, slot 0), (Hz, x, +, slot 1)
                const T b = cx[2 * nx + pi];
                bst2<NTS>(rsrc(g.Apsi[0], own), two(oo), hw0 + xslab(pi), Pair{b * (d[3] + pHx.x), b * (d[4] + pHx.y)});
                d[3] = adj_term(b, d[3], pHx.x);
                d[4] = adj_term(b, d[4], pHx.y);
            }
        }
#pragma unroll
        for (int c = 0; c < 6; ++c) pin(d[c]);
        sDz[half + tid] = Pair{d[2], d[1]};
        sDy[half + tid] = Pair{d[0], d[5]};
        sEz[other + tid] = Pair{tn[1], tn[2]};
        sEy[other + tid] = Pair{tn[0], tn[5]};
#pragma unroll
        for (int c = 0; c < 6; ++c) tc[c] = reg_copy(tn[c]);
        tu[0] = reg_copy(tun[0]);
        tu[1] = reg_copy(tun[1]);
#pragma unroll
        for (int c = 0; c < 3; ++c) u0[c] = reg_copy(uc[c]);
        // ------------------------------- pole recursions of plane i; 1/eps
        const T iv = clut[cls & 0xff].inv_eps;
#pragma unroll
        for (int c = 0; c < 3; ++c) inv[c] = iv, sq[c] = T(0);
        if (cls & kSegSpecial) {
            const MatLut<T>* L[3];
#pragma unroll
            for (int c = 0; c < 3; ++c) {
                L[c] = slut + ((mw >> (8 * c)) & 0xff);
                inv[c] = L[c]->inv_eps;
            }
            const int npx = seg_poles(cls);
            if (NP > 0 && npx > 0) {
                const Rsrc rq = rsrc((const char*)g.Aq + (long)pi * QPB), rp = rsrc((const char*)g.Ap + (long)pi * QPB);
                int np[3];
#pragma unroll
                for (int c = 0; c < 3; ++c) np[c] = L[c]->np;
#pragma unroll
                for (int s = 0; s < NP; ++s) {
                    if (s >= npx) break;
                    PoleCoef<T> p[3];
#pragma unroll
                    for (int c = 0; c < 3; ++c) p[c] = L[c]->pole[s];
#pragma unroll
                    for (int c = 0; c < 3; ++c) {
                        const uint32_t so = (s * 3 + c) * PB;
                        const bool vq = s < np[c];
                        const T pb = Pv[c][s];
                        const T qb = vq ? Qv[c][s] + pb - u0[c] : T(0);
                        bst<NTS>(rq, vq ? oo : kOOB, so, p[c].alpha * qb);
                        bst<NTS>(rp, vq && p[c].lor != T(0) ? oo : kOOB, so, fma_(p[c].beta, qb, pb));
                        sq[c] = fma_(p[c].c3, qb, sq[c]);
                    }
                }
            }
            if (cls & kSegDesign) {
                // design voxels: 1/eps from the design array [dx][dy][dz]
                const Rsrc rd = rsrc(a.dinv);
                const uint32_t dq = (uint32_t)(((pi - a.dlo[0]) * (a.dhi[1] - a.dlo[1]) + (j - a.dlo[1])) *
                                                   (a.dhi[2] - a.dlo[2]) + (k - a.dlo[2])) * W;
#pragma unroll
                for (int c = 0; c < 3; ++c)
                    dv[c] = bld<T>(rd, owned && (int)((mw >> (8 * c)) & 0xff) == a.nmat ? dq : kOOB, 0);
                dw = mw;
            }
        }
        // ------------------------------- loads for the planes ahead
        uint32_t cn = 0u;
        if (!uniform && next) {
            cn = classify<NP>(mwn);
            if (NP > 0 && seg_poles(cn) > 0) load_poles(pn, cn, mwn);
        }
        mw = reg_copy(mwn);
#pragma unroll
        for (int c = 0; c < 3; ++c) uc[c] = reg_copy(un[c]);
        load_u(fNN, next && pnn < nx);
        if (next) load_aux_e(pnn, i + 2 < x1);
        load_h(fN, pn, next);
        if (!uniform) mwn = bld<uint32_t>(rsrc((const char*)a.matw + (long)(i + 2 < x1 ? pnn : 0) * PW, i + 2 < x1), ow, 0);
        return cn;
    };

    auto e_phase = [&](const int i) __attribute__((always_inline)) {
        const Rsrc rW = rsrc(fW + A01, i >= x0);
        const int half = (i & 1) * B;
        lds_barrier();
        const Pair dz = sDz[half + kdn], dy = sDy[half + dn];
        const T hyz = km1 >= 0 ? dz.x : T(0), hxz = km1 >= 0 ? dz.y : T(0);
        if (cls & kSegDesign) {
#pragma unroll
            for (int c = 0; c < 3; ++c) inv[c] = (int)((dw >> (8 * c)) & 0xff) == a.nmat ? dv[c] : inv[c];
        }
        // Ex: (Hy, z) and (Hz, y); Ey: (Hx, z) and (Hz, x); Ez: (Hx, y) and (Hy, x)
        bst<NTS>(rW, oo, 0, fma_(inv[0], ((hyz - d[2]) + (dy.y - d[5])) + sq[0], u0[0]));
        bst<NTS>(rW, oo, PB, fma_(inv[1], ((hxz - d[1]) + (dx[0] - d[4])) + sq[1], u0[1]));
        bst<NTS>(rW, oo, 2 * PB, fma_(inv[2], ((dy.x - d[0]) + (dx[1] - d[3])) + sq[2], u0[2]));
        dx[0] = reg_copy(d[4]);
        dx[1] = reg_copy(d[3]);
        // the next plane
        fW = fN;
        fN = fNN;
        pi = pn;
        pn = pnn;
        ++pnn;
        fNN += FPB;
        if (__builtin_expect(pnn >= nx, 0)) {
            if (a.px) pnn = 0;
            fNN = A0;  // of plane 0, or not read
        }
    };

    uint32_t cn = h_phase(istart);
    for (int i = istart; i < x1; ++i) {
        e_phase(i);
        cls = cn;
        cn = h_phase(i + 1);
    }
}

// Fused reverse step over one engine, row-of-threads form (tile t after the XCD-aware remap).
template <typename T, int NP, int MAXT, bool NTS = false>
__global__ void __launch_bounds__(MAXT) k_adj_rows(const AdjArgs<T> g) {
    const int w = blockIdx.x, nw = gridDim.x;
    const int t = (nw % 8 == 0) ? ((w & 7) * (nw >> 3) + (w >> 3)) : w;
    adj_rows<T, NP, NTS>(g, t);
}

// Fused reverse step over one engine: workgroup w handles tile w after the XCD-aware remap.
// With the loads of a plane issued together, the FP32 reverse step needs 92 registers with three
// pole slots (5 wavefronts per SIMD) and 98 with four (4 wavefronts).
template <typename T>
constexpr int adj_waves() { return sizeof(T) == 4 ? 4 : 1; }

template <typename T, int NP, int MAXT, bool NTS = false>
__global__ void __launch_bounds__(MAXT) __attribute__((amdgpu_waves_per_eu(adj_waves<T>())))
k_adj_step(const AdjArgs<T> g) {
    const int w = blockIdx.x, nw = gridDim.x;
    const int t = (nw % 8 == 0) ? ((w & 7) * (nw >> 3) + (w >> 3)) : w;
    adj_tile<T, NP, NTS>(g, t);
}

// objective J += dt * sum_c E_c(gap)^2 for the state after a step (FP64)
template <typename T>
__device__ __forceinline__ void add_objective(const T* E, long nyz, long gap, double dt, double* J) {
    double s = 0;
    for (int c = 0; c < 3; ++c) {
        const double v = (double)E[field_index(gap, c, nyz)];
        s += v * v;
    }
    *J += s * dt;
}

// record E of the design box and of the objective cell into slot `slot` of a ring buffer; with J, the
// thread of the objective cell's first component adds the objective
template <typename T>
__global__ void __launch_bounds__(256) k_adj_record(const T* E, long nyz, int ny, int nz, int dlo0, int dlo1,
                                                    int dlo2, int de0, int de1, int de2, long gap,
                                                    T* ring, long slot, double dt, double* J) {
    const long nd = (long)de0 * de1 * de2;
    const long v = (long)blockIdx.x * blockDim.x + threadIdx.x;
    T* out = ring + slot * (3 * nd + 3);
    if (v < nd) {
        const int kk = (int)(v % de2);
        const long r = v / de2;
        const int jj = (int)(r % de1), ii = (int)(r / de1);
        const long q = ((long)(dlo0 + ii) * ny + (dlo1 + jj)) * nz + (dlo2 + kk);
#pragma unroll
        for (int c = 0; c < 3; ++c) out[c * nd + v] = E[field_index(q, c, nyz)];
    } else if (v < nd + 3) {
        const int c = (int)(v - nd);
        out[3 * nd + c] = E[field_index(gap, c, nyz)];
        if (J && c == 0) add_objective(E, nyz, gap, dt, J);
    }
}

template <typename T>
__global__ void k_adj_objective(const T* E, long nyz, long gap, double dt, double* J) {
    if (threadIdx.x == 0 && blockIdx.x == 0) add_objective(E, nyz, gap, dt, J);
}

// gradient term of step n:
//   gacc[v] += sum_c Ubar_c^{n+1}(v) (E_c^{n+1}(v) - E_c^n(v))   (before the adjoint step)
// With Ubar = Ebar / eps_v this is (1/eps_v) sum_c Ebar_c^{n+1} (E^{n+1} - E^n): the gradient
// dJ/d eps_v = -(1/eps_v) sum_n sum_c Ebar (E^{n+1} - E^n) is minus the accumulated sum.
// Ebar: the adjoint field set holding Ubar^{n+1} ([x][comp][y][z]).
template <typename T>
__global__ void __launch_bounds__(256) k_adj_grad(const StepArgs<T> a, const T* Ebar, const T* ring, long s_next,
                                                  long s_cur, double* gacc) {
    const long nd = (long)(a.dhi[0] - a.dlo[0]) * (a.dhi[1] - a.dlo[1]) * (a.dhi[2] - a.dlo[2]);
    const long v = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (v >= nd) return;
    const int de1 = a.dhi[1] - a.dlo[1], de2 = a.dhi[2] - a.dlo[2];
    const int kk = (int)(v % de2);
    const long r = v / de2;
    const int jj = (int)(r % de1), ii = (int)(r / de1);
    const long q = ((long)(a.dlo[0] + ii) * a.ny + (a.dlo[1] + jj)) * a.nz + (a.dlo[2] + kk);
    const T* e1 = ring + s_next * (3 * nd + 3);
    const T* e0 = ring + s_cur * (3 * nd + 3);
    double acc = 0;
#pragma unroll
    for (int c = 0; c < 3; ++c)
        acc += (double)Ebar[field_index(q, c, (long)a.ny * a.nz)] * ((double)e1[c * nd + v] - (double)e0[c * nd + v]);
    gacc[v] += acc;
}

// Ebar^n(gap) += dJ/dE^n = 2 dt E^n(gap), on the state Ubar = Ebar / eps: Ubar(gap) gains
// 2 dt E^n(gap) / eps(gap) per component (ie = 1/eps at the gap's three E points)
template <typename T>
__global__ void k_adj_inject(T* Ubar, long nyz, const T* ring, long nd, long slot, long gap, double dt, double ie0,
                             double ie1, double ie2) {
    const int c = threadIdx.x;
    if (blockIdx.x == 0 && c < 3) {
        const double e = (double)ring[slot * (3 * nd + 3) + 3 * nd + c];
        const double ie = c == 0 ? ie0 : (c == 1 ? ie1 : ie2);
        const long o = field_index(gap, c, nyz);
        Ubar[o] = (T)((double)Ubar[o] + 2.0 * dt * e * ie);
    }
}

// ---- adjoint over a batch: the kernels above, one launch for every engine of the set --------
// Per-engine table of the batched record, gradient and injection kernels (blockIdx.y is the
// engine); the fused reverse step maps workgroups to engines as k_step_rows does.
template <typename T>
struct AdjBatchDev {
    const T* F[2];   // forward field sets 0 / 1
    T* A[2];         // adjoint field sets (Ubar, Hbar)
    T* ring;         // record: per step E of the design box (3 nd) and of the objective cell (3)
    double* gacc;    // nd gradient sums
    double* J;       // objective
    long nyz;
    int ny, nz;
    int dlo[3], de[3];
    long nd;
    long gap;        // objective cell
    double dt;
    double ie[3];    // 1/eps at the objective cell's three E points
};

// k_adj_record for every engine (E = field set `par`), and with `objective` set also
// k_adj_objective: the thread of the objective cell's first component adds dt sum_c E_c(gap)^2
template <typename T>
__global__ void __launch_bounds__(256) k_adj_record_batch(const AdjBatchDev<T>* __restrict__ tab, int par,
                                                          long slot, int objective) {
    const AdjBatchDev<T>& a = tab[blockIdx.y];
    const long nd = a.nd;
    const long v = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (v >= nd + 3) return;
    const T* E = a.F[par];
    T* out = a.ring + slot * (3 * nd + 3);
    if (v < nd) {
        const int kk = (int)(v % a.de[2]);
        const long r = v / a.de[2];
        const int jj = (int)(r % a.de[1]), ii = (int)(r / a.de[1]);
        const long q = ((long)(a.dlo[0] + ii) * a.ny + (a.dlo[1] + jj)) * a.nz + (a.dlo[2] + kk);
#pragma unroll
        for (int c = 0; c < 3; ++c) out[c * nd + v] = E[field_index(q, c, a.nyz)];
    } else {
        const int c = (int)(v - nd);
        out[3 * nd + c] = E[field_index(a.gap, c, a.nyz)];
        if (objective && c == 0) add_objective(E, a.nyz, a.gap, a.dt, a.J);
    }
}

// k_adj_grad for every engine (Ubar^{n+1} in adjoint set `rd`)
template <typename T>
__global__ void __launch_bounds__(256) k_adj_grad_batch(const AdjBatchDev<T>* __restrict__ tab, int rd,
                                                        long s_next, long s_cur) {
    const AdjBatchDev<T>& a = tab[blockIdx.y];
    const long nd = a.nd;
    const long v = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (v >= nd) return;
    const int kk = (int)(v % a.de[2]);
    const long r = v / a.de[2];
    const int jj = (int)(r % a.de[1]), ii = (int)(r / a.de[1]);
    const long q = ((long)(a.dlo[0] + ii) * a.ny + (a.dlo[1] + jj)) * a.nz + (a.dlo[2] + kk);
    const T* Ebar = a.A[rd];
    const T* e1 = a.ring + s_next * (3 * nd + 3);
    const T* e0 = a.ring + s_cur * (3 * nd + 3);
    double acc = 0;
#pragma unroll
    for (int c = 0; c < 3; ++c)
        acc += (double)Ebar[field_index(q, c, a.nyz)] * ((double)e1[c * nd + v] - (double)e0[c * nd + v]);
    a.gacc[v] += acc;
}

// k_adj_inject for every engine (into adjoint set `rd`, record slot `slot`)
template <typename T>
__global__ void k_adj_inject_batch(const AdjBatchDev<T>* __restrict__ tab, int rd, long slot) {
    const AdjBatchDev<T>& a = tab[blockIdx.y];
    const int c = threadIdx.x;
    if (blockIdx.x == 0 && c < 3) {
        const double e = (double)a.ring[slot * (3 * a.nd + 3) + 3 * a.nd + c];
        const long o = field_index(a.gap, c, a.nyz);
        T* U = a.A[rd];
        U[o] = (T)((double)U[o] + 2.0 * a.dt * e * a.ie[c]);
    }
}

// Fused reverse step over every engine of a batch (tile t of engine b after the XCD-aware remap)
template <typename T, int NP, int MAXT, bool NTS = false>
__global__ void __launch_bounds__(MAXT) __attribute__((amdgpu_waves_per_eu(adj_waves<T>())))
k_adj_step_batch(const AdjArgs<T>* __restrict__ args, const int* __restrict__ tile_first, int ninst) {
    int t;
    const int b = tile_instance(tile_first, ninst, t);
    adj_tile<T, NP, NTS>(args[b], t);
}

// The same, row-of-threads form
template <typename T, int NP, int MAXT, bool NTS = false>
__global__ void __launch_bounds__(MAXT) k_adj_rows_batch(const AdjArgs<T>* __restrict__ args,
                                                         const int* __restrict__ tile_first, int ninst) {
    int t;
    const int b = tile_instance(tile_first, ninst, t);
    adj_rows<T, NP, NTS>(args[b], t);
}

// ---- plain streaming copy (achievable-bandwidth probe and counter calibration) -----------
// one float4 per thread over the whole array (the fastest plain copy measured on MI355X)
__global__ void __launch_bounds__(256) k_copy(const float4* __restrict__ src, float4* __restrict__ dst,
                                              long n) {
    const long q = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (q < n) dst[q] = src[q];
}

}  // namespace sjf
