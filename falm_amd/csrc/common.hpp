// common.hpp — shared host/device helpers of the gfx950 library.
//
// Layout: the reference's Matrix layout (src/matrix.h:20), one column per
// component, x fastest over the padded local shape.  Kernels receive one
// pointer per column so that no 64-bit column arithmetic happens on device.
#pragma once

#include <hip/hip_runtime.h>

#include <cstddef>
#include <initializer_list>
#include <cstdint>
#include <cstdio>
#include <string>

#include "../../include/falm_amd.h"

namespace falm {

// ------------------------------------------------------------------ errors
void set_error(const char *fmt, ...);
falm_status hip_status(hipError_t e, const char *what);

#define FALM_HIP(expr)                                                      \
    do {                                                                    \
        hipError_t _e = (expr);                                             \
        if (_e != hipSuccess) return ::falm::hip_status(_e, #expr);         \
    } while (0)

#define FALM_TRY(expr)                                                      \
    do {                                                                    \
        falm_status _s = (expr);                                            \
        if (_s != FALM_OK) return _s;                                       \
    } while (0)

#define FALM_CHECK_LAUNCH(name) FALM_HIP(hipGetLastError())

// ----------------------------------------------------------------- domain
// Device-side view of a falm_domain (src/region.h:8-31 + CPM::gc).
struct Geom {
    int nx, ny, nz;     // padded local shape
    int gc;
    int osum;           // sum of pdm.offset: parity term of the RB colour
    int nxy;            // nx*ny
    __host__ __device__ inline int id(int i, int j, int k) const { return i + nx * j + nxy * k; }
};

inline Geom make_geom(const falm_domain *d) {
    Geom g;
    g.nx = d->shape[0];
    g.ny = d->shape[1];
    g.nz = d->shape[2];
    g.gc = d->gc;
    g.osum = d->offset[0] + d->offset[1] + d->offset[2];
    g.nxy = g.nx * g.ny;
    return g;
}

inline size_t ncell_of(const falm_domain *d) {
    return (size_t)d->shape[0] * (size_t)d->shape[1] * (size_t)d->shape[2];
}

falm_status check_domain(const falm_domain *d);
// FALM_ERR_INVALID unless every pointer is hipMalloc'd device memory (the
// adjoint kernels accumulate into such outputs with FP64 atomics)
falm_status vjp_outputs_on_device(std::initializer_list<const void *> outs);

// A box of cells [lo, lo+n) in padded local indices.
struct Box {
    int lo[3];
    int n[3];
    __host__ __device__ inline long long size() const { return (long long)n[0] * n[1] * n[2]; }
};

inline Box interior_box(const Geom &g) {
    return Box{{g.gc, g.gc, g.gc}, {g.nx - 2 * g.gc, g.ny - 2 * g.gc, g.nz - 2 * g.gc}};
}
// Region(pdm.shape, gc) with shape += 1 and offset -= 1 (src/FalmCFD.cpp:119-126).
inline Box face_box(const Geom &g) {
    return Box{{g.gc - 1, g.gc - 1, g.gc - 1},
               {g.nx - 2 * g.gc + 1, g.ny - 2 * g.gc + 1, g.nz - 2 * g.gc + 1}};
}

// ----------------------------------------------------------- launch shape
// Stencil launches use 64x4 threads (one wavefront per x row segment) over a
// 1-D grid.  The 1-D block id is remapped so that each of the 8 XCDs of an
// MI355X (workgroups are dealt to XCDs round-robin) gets one contiguous
// slab of tiles: neighbouring tiles then share that XCD's L2.
constexpr int TX = 64;
constexpr int TY = 4;
constexpr int NXCD = 8;

struct Tiling {
    Box box;
    int tx, ty;          // tiles along x, y
    int tiles;           // tx*ty*box.n[2]
    __host__ __device__ inline int ntiles() const { return tiles; }
};

inline Tiling make_tiling(const Box &b) {
    Tiling t;
    t.box = b;
    t.tx = (b.n[0] + TX - 1) / TX;
    t.ty = (b.n[1] + TY - 1) / TY;
    t.tiles = t.tx * t.ty * b.n[2];
    return t;
}

// physical block id -> logical tile id, XCD-contiguous
__device__ inline int xcd_tile(int bid, int nblocks) {
    int per = (nblocks + NXCD - 1) / NXCD;
    int xcd = bid % NXCD;
    int loc = bid / NXCD;
    int full = nblocks % NXCD;          // XCDs that receive `per` blocks
    // blocks are dealt round robin: XCDs [0, full) get `per` blocks and the
    // rest get per-1 when nblocks is not a multiple of NXCD
    if (full == 0) return xcd * per + loc;
    if (xcd < full) return xcd * per + loc;
    return full * per + (xcd - full) * (per - 1) + loc;
}

// Tile order: x tile fastest, then y, then k, so consecutive workgroups
// stream through contiguous memory (a k-fastest order that keeps stencil
// neighbours in flight together measured slower: every tile then starts a
// new DRAM page).
__host__ __device__ inline void tile_coords(const Tiling &t, int tile, int &bx, int &by, int &kk) {
    const int txy = t.tx * t.ty;
    kk = tile / txy;
    const int r = tile - kk * txy;
    by = r / t.tx;
    bx = r - by * t.tx;
}

// cell coordinates of this thread in tile `tile`; false outside the box.
// A wavefront covers one x row of the tile, so j and k are wave-uniform:
// readfirstlane makes that visible to the compiler, which then keeps them
// (and loads indexed by them alone) in scalar registers.
__device__ inline bool tile_cell_at(const Tiling &t, int tile, int &i, int &j, int &k) {
    int bx, by;
    tile = __builtin_amdgcn_readfirstlane(tile);
    tile_coords(t, tile, bx, by, k);
    i = bx * TX + (int)(threadIdx.x & (TX - 1));
    j = by * TY + __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    if (i >= t.box.n[0] || j >= t.box.n[1]) return false;
    i += t.box.lo[0];
    j += t.box.lo[1];
    k += t.box.lo[2];
    return true;
}

// Reduction kernels run at most RED_BLOCKS workgroups; each walks a
// contiguous run of tiles (of the XCD-contiguous order), so the finalize
// kernel sums at most RED_BLOCKS partials.
constexpr int RED_BLOCKS = 4096;
inline dim3 red_grid(const Tiling &t) { return dim3((unsigned)(t.tiles < RED_BLOCKS ? t.tiles : RED_BLOCKS)); }
inline int red_blocks(const Tiling &t) { return t.tiles < RED_BLOCKS ? t.tiles : RED_BLOCKS; }
__device__ inline void tile_range(int ntiles, int &t0, int &t1) {
    const int L = xcd_tile(blockIdx.x, gridDim.x);
    const int C = (ntiles + (int)gridDim.x - 1) / (int)gridDim.x;
    t0 = L * C;
    t1 = t0 + C < ntiles ? t0 + C : ntiles;
}

// The non-reducing kernels take one tile per workgroup (one_tile_grid):
// measured on MI355X, walking several tiles per workgroup made the stencil
// kernels slower.  f(i, j, k) is called for this thread's cell of the tile
// (return in f ends the thread's work).
template <class F>
__device__ inline void for_each_cell(const Tiling &t, F f) {
    int i, j, k;
    if (tile_cell_at(t, xcd_tile(blockIdx.x, gridDim.x), i, j, k)) f(i, j, k);
}

// cell coordinates of this thread for one tile per workgroup; false outside
// the box
__device__ inline bool tile_cell(const Tiling &t, int &i, int &j, int &k) {
    return tile_cell_at(t, xcd_tile(blockIdx.x, gridDim.x), i, j, k);
}

// one tile per workgroup (for_each_cell, tile_cell)
inline dim3 tiling_grid(const Tiling &t) { return dim3((unsigned)t.tiles); }
inline dim3 one_tile_grid(const Tiling &t) { return dim3((unsigned)t.tiles); }
inline dim3 tiling_block() { return dim3(TX * TY); }

// Access at an unsigned 32-bit byte offset from a wave-uniform base pointer.
// The compiler then emits the SGPR-base form of the global load/store (one
// VGPR offset shared by every array indexed at the same cell, constant
// neighbour offsets folded into the instruction), where a signed element
// index costs a 64-bit address computation per access.  Arrays addressed
// this way must be below 4 GiB (checked by the launchers, by
// falm_solver_create and by falm_case_create).
template <class T>
__device__ __forceinline__ T ld_at(const T *p, unsigned off) {
    return *reinterpret_cast<const T *>(reinterpret_cast<const char *>(p) + off);
}
template <class T>
__device__ __forceinline__ void st_at(T *p, unsigned off, T v) {
    *reinterpret_cast<T *>(reinterpret_cast<char *>(p) + off) = v;
}

// Read of a wave-uniform element of a table the kernel never writes (the
// per-axis coefficient tables), through the constant address space: the
// compiler then issues a scalar load, counted by lgkmcnt.  A plain load of
// such a value is a vector load when the kernel also stores to global
// memory, and waiting for it (vmcnt) also waits for every vector load issued
// before it: in a k-marching loop, for the prefetches of the next planes.
// p and i must be the same in every lane of the wave.
template <class T>
__device__ __forceinline__ T ld_uniform(const T *p, int i) {
    return ((const __attribute__((address_space(4))) T *)p)[i];
}

// the ld_at/st_at kernels address one field column of ncell elements
inline falm_status check_byte_offsets(size_t ncell, size_t elem) {
    if (ncell * elem >= (size_t(1) << 32)) {
        set_error("a field column exceeds 4 GiB (the stencil kernels use 32-bit byte offsets)");
        return FALM_ERR_UNSUPPORTED;
    }
    return FALM_OK;
}

// 1-D element-wise launches
constexpr int EW_BLOCK = 256;
inline dim3 ew_grid(size_t n) {
    size_t b = (n + EW_BLOCK - 1) / EW_BLOCK;
    if (b > 2147483647ull) b = 2147483647ull;
    return dim3((unsigned)b);
}

// ------------------------------------------------------------- reductions
// Wavefront (64 lanes) then block reduction of doubles.  The lanes are added
// through DPP moves (rows of 16 by shifts, then the row totals broadcast to
// the rows above), which stay in the vector unit: a __shfl_down is two LDS
// permutes a step, 12 a sum, and the waves of a reduction share one LDS.
// With the values of a block side by side on its waves (block_sum_n) the
// finalize and the ends of the reducing kernels got shorter: the window
// gradient at 96 x 48 x 48 64.1 -> 59.8 ms.  Every lane gets the sum; all 64 must be active.
template <int CTRL, int ROWS>
__device__ inline double dpp_shifted(double v) {  // 0 where a lane receives none
    const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(v), CTRL, ROWS, 0xf, true);
    const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(v), CTRL, ROWS, 0xf, true);
    return __hiloint2double(hi, lo);
}
__device__ inline double wave_sum(double v) {
    v += dpp_shifted<0x111, 0xf>(v);  // row_shr:1
    v += dpp_shifted<0x112, 0xf>(v);  // row_shr:2
    v += dpp_shifted<0x114, 0xf>(v);  // row_shr:4
    v += dpp_shifted<0x118, 0xf>(v);  // row_shr:8: lane 15 of a row has the row's sum
    v += dpp_shifted<0x142, 0xa>(v);  // row_bcast:15 into rows 1 and 3
    v += dpp_shifted<0x143, 0xc>(v);  // row_bcast:31 into rows 2 and 3
    const int lo = __builtin_amdgcn_readlane(__double2loint(v), 63);
    const int hi = __builtin_amdgcn_readlane(__double2hiint(v), 63);
    return __hiloint2double(hi, lo);
}

// Wavefront minimum / maximum through the same moves (a lane that receives
// nothing keeps its own value); every lane gets it.
template <int CTRL, int ROWS>
__device__ inline int dpp_or_own(int v) {
    return __builtin_amdgcn_update_dpp(v, v, CTRL, ROWS, 0xf, false);
}
template <int CTRL, int ROWS>
__device__ inline double dpp_or_own(double v) {
    return __hiloint2double(dpp_or_own<CTRL, ROWS>(__double2hiint(v)), dpp_or_own<CTRL, ROWS>(__double2loint(v)));
}
__device__ inline int lane63(int v) { return __builtin_amdgcn_readlane(v, 63); }
__device__ inline double lane63(double v) {
    return __hiloint2double(lane63(__double2hiint(v)), lane63(__double2loint(v)));
}
template <class V, class F>
__device__ inline V wave_reduce(V v, F f) {
    v = f(v, dpp_or_own<0x111, 0xf>(v));
    v = f(v, dpp_or_own<0x112, 0xf>(v));
    v = f(v, dpp_or_own<0x114, 0xf>(v));
    v = f(v, dpp_or_own<0x118, 0xf>(v));
    v = f(v, dpp_or_own<0x142, 0xa>(v));
    v = f(v, dpp_or_own<0x143, 0xc>(v));
    return lane63(v);
}

// Multi-value block sum (NV values per thread): every wave's sums go to LDS
// (lds holds NV * NT/64), and wave q sums value q's NT/64 of them, so that the
// values are summed side by side and not one after the other in one thread.
// The result of value q is returned in every lane of wave q < NV (q on the
// waves that have one, -1 on the others).
template <int NT, int NV>
__device__ inline int block_sum_n(double (&v)[NV], double *lds, double &total) {
    constexpr int NW = NT / 64;
    static_assert(NV <= NW && NW <= 64, "a wave per value");
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
#pragma unroll
    for (int q = 0; q < NV; q++) {
        const double x = wave_sum(v[q]);
        if (lane == 0) lds[q * NW + wid] = x;
    }
    __syncthreads();
    total = 0.0;
    if (wid >= NV) return -1;
    total = wave_sum(lane < NW ? lds[wid * NW + lane] : 0.0);
    return wid;
}

// Deterministic two-phase grid reduction.  Phase 1 (in the producing
// kernel): each workgroup reduces its values and writes one partial per
// value with a plain store.  Phase 2 (a separate one-workgroup kernel that
// the stream orders after phase 1): the partials are summed in a fixed
// order.  No device-scope fences or atomics are needed: a per-workgroup
// release fence would write back the XCD's L2 in every one of tens of
// thousands of workgroups.
template <int NT, int NV>
__device__ inline void block_partials(double (&v)[NV], double *partials, double *lds) {
    double t;
    const int q = block_sum_n<NT, NV>(v, lds, t);
    if (q >= 0 && (threadIdx.x & 63) == 0) partials[(size_t)q * gridDim.x + blockIdx.x] = t;
}

// A launch gated on a device flag: the kernel does nothing unless *gate is
// nonzero (gate null: always runs).  The step driver enqueues the kernels
// after the Poisson solve gated on the solver's "finished" flag before it
// knows whether the first batch of iterations finished the solve.
__device__ inline bool gated_off(const int *gate) { return gate && !*gate; }

constexpr int FIN_NT = 1024;  // threads of a finalize workgroup

// Phase 2 helper for an NT-thread workgroup: totals of nb partials per
// value, valid in every thread.  Used by the one-workgroup finalize kernels,
// and by consumer kernels whose every workgroup needs a reduction's result:
// each sums the same partials in the same order, so all get the same bits
// (no finalize launch between producer and consumer).
template <int NV, int NT = FIN_NT>
__device__ inline void sum_partials(const double *partials, int nb, double (&tot)[NV]) {
    __shared__ double lds[NV * (NT / 64)];
    __shared__ double bc[NV];
    double acc[NV];
#pragma unroll
    for (int q = 0; q < NV; q++) {
        double s = 0.0;
        for (int b = threadIdx.x; b < nb; b += NT) s += partials[(size_t)q * nb + b];
        acc[q] = s;
    }
    double t;
    const int q = block_sum_n<NT, NV>(acc, lds, t);
    if (q >= 0 && (threadIdx.x & 63) == 0) bc[q] = t;
    __syncthreads();
#pragma unroll
    for (int q = 0; q < NV; q++) tot[q] = bc[q];
}

// ------------------------------------------------------------ precision
template <class T> struct PrecOf;
template <> struct PrecOf<double> { static constexpr int value = FALM_F64; };
template <> struct PrecOf<float> { static constexpr int value = FALM_F32; };

inline size_t prec_bytes(int prec) { return prec == FALM_F32 ? 4 : 8; }

inline bool overlaps(const void *a, size_t abytes, const void *b, size_t bbytes) {
    const char *x = (const char *)a, *y = (const char *)b;
    return x < y + bbytes && y < x + abytes;
}

// column pointer helper
template <class T> inline T *col(void *p, size_t ncell, int c) { return (T *)p + (size_t)c * ncell; }
template <class T> inline const T *col(const void *p, size_t ncell, int c) {
    return (const T *)p + (size_t)c * ncell;
}

// -------------------------------------------------------------- scratch
// Library-owned device scratch for one-shot reductions (per device).
struct ReduceScratch {
    double *partials = nullptr;  // 8 * max_blocks doubles
    double *host = nullptr;      // 8 doubles of pinned host memory, written by the finalize kernel
    size_t max_blocks = 0;
};
falm_status reduce_scratch(size_t nblocks, ReduceScratch **out);

// compute units of the current device
int cu_count();
// device address of falm_dot_noalloc's workspace on the current device,
// taken on first use (falm_init calls it for its device)
falm_status noalloc_setup(double **out);

// ------------------------------------------------------------ timing
struct TimedLaunch {
    int family;
    hipStream_t stream;
    bool on;
    TimedLaunch(int fam, hipStream_t s);
    void done(double bytes);
    // bytes known only after the launch (e.g. a box the kernels chose);
    // counts toward the family's total when the launch was timed
    void add_bytes(double bytes);
};

}  // namespace falm
