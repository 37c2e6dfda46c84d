// libadfvm: HIP kernels for gfx950 (MI355X) and the C ABI of include/adfvm.h.
//
// Design (one GPU, one context per mesh):
//  * the caller's state and gradient arrays are structure-of-arrays rows of
//    nInternalCells scalars in the context precision (float or double); the
//    library's own are records in tile order (tile_kernels.inc);
//  * every face->cell accumulation is a sum over the cell's six cellFaces
//    slots in order (owned faces in face order, then neighbour faces,
//    cmesh.cpp:9-19).  No atomics: results are bit-identical from run to run;
//  * cyclic ghosts are resolved at set-up to the paired internal cell; the
//    ghost of a non-cyclic boundary face is evaluated where it is used, from
//    its owner cell and the patch's values (a ghost array is filled only for
//    the ghost-value entry point and the adjoint viscosity);
//  * reductions (objective, dtc) write one partial per block and a single
//    block folds the partials in index order, in FP64.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>
#include <cstdio>
#include <cstring>
#include <exception>
#include <future>
#include <initializer_list>
#include <mutex>
#include <string>
#include <vector>

#include "adfvm.h"
#include "fvm_math.hpp"
#include "adjoint_math.hpp"
#include "dual.hpp"
#include "tiles.hpp"

using namespace adfvm;

#define BLOCK 256

// Workgroups of a launch are dealt to the 8 XCDs round-robin (block b runs
// on XCD b % 8), and each XCD has its own L2.  The stencil kernels remap
// block b to a tile so that every XCD works through one contiguous eighth of
// the tiles: those it works on at one time lie near one another in the mesh
// (order_tiles), and a tile's halo is in its L2 as its neighbours' own cells.
// The map is a bijection of [0, gridDim.x).
__device__ __forceinline__ int xcd_block() {
    const unsigned nb = gridDim.x, b = blockIdx.x;
    const unsigned q = nb >> 3, r = nb & 7u, x = b & 7u, k = b >> 3;
    return (int)(x * q + (x < r ? x : r) + k);
}

// ------------------------------------------------------------- tables ----
// slot flags: bit 0 = this cell owns the face; bits 1-2 = slot kind
enum { SLOT_INTERNAL = 0, SLOT_COUPLED = 1, SLOT_CHARACTERISTIC = 2, SLOT_BOUNDARY = 3 };
__host__ __device__ __forceinline__ int slot_kind(int flags) { return (flags >> 1) & 3; }
// face kind bytes (device copy): FACE_* in bits 0-1, bit 2 for a boundary
// face whose ghost's values are the owner's (zeroGradient U, and zeroGradient or
// symmetry T and p: BCs.py:97-104,120-137), so that neither the ghost rule nor its
// adjoint needs the patch
constexpr int FACE_GHOST_COPY = 4;
__host__ __device__ __forceinline__ int face_kind(int k) { return k & 3; }

// the ghost of a non-characteristic patch is its owner's values
inline bool ghost_copies_owner(const adfvm_patch_desc& Pd) {
    auto scalarCopy = [](int bc) { return bc == ADFVM_BC_ZERO_GRADIENT || bc == ADFVM_BC_SYMMETRY; };
    return Pd.fluxKind == ADFVM_FLUX_BOUNDARY && Pd.cbc == ADFVM_CBC_NONE && Pd.bcU == ADFVM_BC_ZERO_GRADIENT &&
           scalarCopy(Pd.bcT) && scalarCopy(Pd.bcp);
}

// face geometry rows (each nFaces long)
enum { G_A = 0, G_NX, G_NY, G_NZ, G_W, G_DELTA, G_DX, G_DY, G_DZ, G_LW0, G_LW1,
       G_Q0X, G_Q0Y, G_Q0Z, G_Q1X, G_Q1Y, G_Q1Z, G_ROWS };

struct DPatch {
    int start, n, fluxKind, bcU, bcT, bcp, cbc, hasDir;
    long valU, valT, valp, valTt, valpt, valDir;   // offsets into the value buffer, -1 if absent
};

template <typename T> struct DMesh {
    int nIC, nIF, nF, nBF;
    const T* geo;           // [G_ROWS][nF]
    const T* vol;           // [nIC]
    const int* sFace;       // [6][nIC]
    const int* sOther;      // [6][nIC]: internal cell, or -1-b for boundary face b
    const unsigned char* sFlags;  // [6][nIC]
    const int* sPair;       // [6][nIC]: paired face of a coupled slot, else -1
    const int* owner;       // [nF]
    const int* fOther;      // [nF]: neighbour, paired internal cell (cyclic) or -1-b (ghost)
    const unsigned char* fKind;  // [nF]: face kind bytes
    const int* bPatch;      // [nBF]
    const DPatch* patches;
    const T* bcval;
};

// Loads of data a launch touches once, in pieces whose cache lines one
// instruction consumes whole (a tile's tables and geometry; ldp the same in 16
// bytes): non-temporal, so that they are first out of L2 and the records that
// neighbouring tiles read again stay in it (128^3 FP32 step 907 -> 802 us).  Not for
// records that straddle lines or that lanes share: there the hint re-fetches
// lines.
// ST selects it per context (adfvm_ctx::stream): on meshes whose stage works on
// less than the 256 MB Infinity Cache the next kernels and stages find the same
// tables there, and plain loads keep them (a 64^3 FP32 step takes 119 us
// streamed, 108 not).
template <bool ST, typename T> __device__ __forceinline__ T ld(const T* p) {
    if constexpr (ST) return __builtin_nontemporal_load(p);
    else return *p;
}

// Geometry of face f.
template <typename T> __device__ __forceinline__ void load_geo(const DMesh<T>& m, int f, FaceGeo<T>& g) {
    auto row = [&](int r) { return m.geo[(long)r * m.nF + f]; };
    g.A = row(G_A);
    g.n[0] = row(G_NX); g.n[1] = row(G_NY); g.n[2] = row(G_NZ);
    g.w = row(G_W);
    g.delta = row(G_DELTA);
    g.D[0] = row(G_DX); g.D[1] = row(G_DY); g.D[2] = row(G_DZ);
    g.lw0 = row(G_LW0); g.lw1 = row(G_LW1);
    g.qw0[0] = row(G_Q0X); g.qw0[1] = row(G_Q0Y); g.qw0[2] = row(G_Q0Z);
    g.qw1[0] = row(G_Q1X); g.qw1[1] = row(G_Q1Y); g.qw1[2] = row(G_Q1Z);
}

// primitive values of a value source: internal cell (from the state) or ghost.
// Branch-free (one strided load from either source, then a per-element
// select) so that w stays in registers: writing the array in two branches
// made the compiler place it in scratch memory.
template <typename T>
__device__ __forceinline__ void load_prim(const Phys<T>& ph, const T* __restrict__ u, long nIC,
                                          const T* __restrict__ ghost, long nBF, int src, T* w) {
    const bool internal = src >= 0;
    const T* base = internal ? u + src : ghost + (-1 - src);
    const long stride = internal ? nIC : nBF;
    T q[5], p[5];
    for (int i = 0; i < 5; i++) q[i] = base[i * stride];
    primitive(ph, q, p);
    for (int i = 0; i < 5; i++) w[i] = internal ? p[i] : q[i];
}

// cell adjoint records: gradient adjoint (15), primitive adjoint (5)
constexpr int AREC = 20;

// N contiguous values from / to a 16-byte aligned address (N a multiple of
// 16/sizeof(T)), as 16-byte memory operations.  The copies go through
// __builtin_memcpy so that no object is read through a pointer of another
// type: the T values are never accessed as a vector type or vice versa.
template <int N, typename T> __device__ __forceinline__ void vload(const T* __restrict__ p, T* out) {
    static_assert((N * sizeof(T)) % 16 == 0, "vector width");
    const T* a = static_cast<const T*>(__builtin_assume_aligned(p, 16));
#pragma unroll
    for (int k = 0; k < (int)(N * sizeof(T) / 16); k++) __builtin_memcpy(out + k * (16 / sizeof(T)), a + k * (16 / sizeof(T)), 16);
}

template <int N, typename T> __device__ __forceinline__ void vstore(T* __restrict__ p, const T* in) {
    static_assert((N * sizeof(T)) % 16 == 0, "vector width");
    T* a = static_cast<T*>(__builtin_assume_aligned(p, 16));
#pragma unroll
    for (int k = 0; k < (int)(N * sizeof(T) / 16); k++) __builtin_memcpy(a + k * (16 / sizeof(T)), in + k * (16 / sizeof(T)), 16);
}

// ------------------------------------------------------------- kernels ---

// Ghost primitive values of non-cyclic boundary face b from its owner's
// primitive values w (Solver.boundary + characteristicBoundary,
// solver.py:106-114, density.py:333-337, BCs.py): every rule reads only the
// owner, the face normal and the patch's values, so the kernels that need a
// ghost evaluate it where they use it.  ghost_rule takes the normal from
// nrm(n) (called only by the rules that use it) and computes in T, S or
// Dual<S>; ghost_value reads the normal from the face geometry.
template <typename T, typename S, typename NormalFn>
__device__ __forceinline__ void ghost_rule(const DMesh<S>& m, const Phys<T>& ph, int b, const T* w,
                                           NormalFn nrm, T* out) {
    const DPatch P = m.patches[m.bPatch[b]];
    const int f = m.nIF + b;
    const int k = f - P.start;
    const S* V = m.bcval;
    if (P.cbc == ADFVM_CBC_UPT) {                    // BCs.py:152-161
        for (int i = 0; i < 3; i++) out[i] = T(V[P.valU + 3 * k + i]);
        out[3] = T(V[P.valT + k]);
        out[4] = T(V[P.valp + k]);
    } else if (P.cbc == ADFVM_CBC_TOTAL_PT) {        // BCs.py:164-184
        T d[3];
        if (P.hasDir) { for (int i = 0; i < 3; i++) d[i] = T(V[P.valDir + 3 * k + i]); }
        else nrm(d);
        T Tt = T(V[P.valTt + k]), pt = T(V[P.valpt + k]);
        T Un = w[0] * d[0] + w[1] * d[1] + w[2] * d[2];
        for (int i = 0; i < 3; i++) out[i] = Un * d[i];
        out[3] = Tt - T(0.5) * Un * Un / ph.Cp;
        out[4] = pt * pow(w[3] / Tt, ph.gamma / (ph.gamma - T(1)));
    } else {
        // U
        if (P.bcU == ADFVM_BC_FIXED_VALUE || P.bcU == ADFVM_BC_CALCULATED) {
            for (int i = 0; i < 3; i++) out[i] = T(V[P.valU + 3 * k + i]);
        } else {
            for (int i = 0; i < 3; i++) out[i] = w[i];
            if (P.bcU == ADFVM_BC_SYMMETRY) {        // BCs.py:125-133
                T n[3];
                nrm(n);
                T un = out[0] * n[0] + out[1] * n[1] + out[2] * n[2];
                out[0] -= un * n[0]; out[1] -= un * n[1]; out[2] -= un * n[2];
            }
        }
        out[3] = (P.bcT == ADFVM_BC_FIXED_VALUE || P.bcT == ADFVM_BC_CALCULATED) ? T(V[P.valT + k]) : w[3];
        out[4] = (P.bcp == ADFVM_BC_FIXED_VALUE || P.bcp == ADFVM_BC_CALCULATED) ? T(V[P.valp + k]) : w[4];
    }
}

template <typename T>
__device__ __forceinline__ void ghost_value(const DMesh<T>& m, const Phys<T>& ph, int b, const T* w, T* out) {
    const int f = m.nIF + b;
    ghost_rule(m, ph, b, w, [&](T* n) {
        const long s = m.nF;
        n[0] = m.geo[G_NX * s + f]; n[1] = m.geo[G_NY * s + f]; n[2] = m.geo[G_NZ * s + f];
    }, out);
}

// The ghost array (ghost primitives [5][nBF]), for the consumers that read
// it as an array: the ghost-value entry point and the adjoint viscosity.
template <typename T>
__global__ void __launch_bounds__(BLOCK) ghost_kernel(DMesh<T> m, Phys<T> ph, const T* __restrict__ u,
                                                      T* __restrict__ ghost) {
    int b = blockIdx.x * blockDim.x + threadIdx.x;
    if (b >= m.nBF) return;
    const DPatch P = m.patches[m.bPatch[b]];
    if (P.bcU == ADFVM_BC_CYCLIC && P.cbc == ADFVM_CBC_NONE) return;   // resolved by the slot tables
    const long nIC = m.nIC, nBF = m.nBF;
    const int c = m.owner[m.nIF + b];
    T q[5], w[5], out[5];
    for (int i = 0; i < 5; i++) q[i] = u[i * nIC + c];
    primitive(ph, q, w);
    ghost_value(m, ph, b, w, out);
    for (int i = 0; i < 5; i++) ghost[i * nBF + b] = out[i];
}

// What the reductions combine two values by: op 0 their sum, 1 the larger of
// them.  A NaN on either side is kept: a comparison alone would drop the one on
// its left, and the time step limit of a diverged state would look finite.
template <int OP> __device__ __forceinline__ double combine(double a, double b) {
    return OP == 0 ? a + b : (a > b || a != a ? a : b);
}

// Block reduction of one double per thread, in thread 0.
template <int OP, int BS = BLOCK>
__device__ double block_reduce(double v) {
    __shared__ double sh[BS];
    sh[threadIdx.x] = v;
    __syncthreads();
    for (int s = BS / 2; s > 0; s >>= 1) {
        if (threadIdx.x < s) sh[threadIdx.x] = combine<OP>(sh[threadIdx.x], sh[threadIdx.x + s]);
        __syncthreads();
    }
    return sh[0];
}

template <int OP, int BS = BLOCK>
__device__ void block_reduce_store(double v, double* out) {
    v = block_reduce<OP, BS>(v);
    if (threadIdx.x == 0) out[blockIdx.x] = v;
}

// A thread's share of n partials, those at its index and every THREADS-th after
// it, folded in order.  Loads in batches of 32: one block waits for each batch,
// and nothing else runs meanwhile (a load at a time, 33k partials took 44 us); one
// partial a thread skips the rest of its batch (a 1000-cell FP64 step 32.9 -> 31.7
// us).
template <int OP, int THREADS>
__device__ __forceinline__ double fold_partials(const double* __restrict__ partials, int n) {
    constexpr int BATCH = 32;
    const double none = OP == 0 ? 0.0 : -1.0e308;
    if (n <= THREADS) return combine<OP>(none, (int)threadIdx.x < n ? partials[threadIdx.x] : none);
    double v = none;
    for (int i = threadIdx.x; i < n; i += BATCH * THREADS) {
        double x[BATCH];
#pragma unroll
        for (int k = 0; k < BATCH; k++) x[k] = i + k * THREADS < n ? partials[i + k * THREADS] : none;
#pragma unroll
        for (int k = 0; k < BATCH; k++) v = combine<OP>(v, x[k]);
    }
    return v;
}

// Folds n partials inside one block: out = op(partials).  Sums by 256 threads,
// whose order they keep; the largest value, which has none, by 1024.
template <int OP> constexpr int FINAL_THREADS = OP == 0 ? BLOCK : 1024;
template <int OP>
__global__ void __launch_bounds__(FINAL_THREADS<OP>) finalize_kernel(const double* __restrict__ partials, int n,
                                                                     double* out) {
    block_reduce_store<OP, FINAL_THREADS<OP>>(fold_partials<OP, FINAL_THREADS<OP>>(partials, n), out);
}

// A step's objective (the sum of nSum values, folded as finalize_kernel folds
// them) and time step limit (the largest of nMax) in one launch, a block each.
__global__ void __launch_bounds__(1024) finalize_step_kernel(const double* __restrict__ sums, int nSum, double* sum,
                                                             const double* __restrict__ largest, int nMax,
                                                             double* max) {
    const bool first = blockIdx.x == 0;
    const double v = first ? block_reduce<0, 1024>(threadIdx.x < BLOCK ? fold_partials<0, BLOCK>(sums, nSum) : 0.0)
                           : block_reduce<1, 1024>(fold_partials<1, 1024>(largest, nMax));
    if (threadIdx.x == 0) *(first ? sum : max) = v;
}

// Kinetic energy 0.5*rho*|U|^2*V of a cell of state q.
template <typename T> __device__ __forceinline__ T kinetic_energy(const T* q, T V) {
    T rho = q[0];
    T Ux = q[1] / rho, Uy = q[2] / rho, Uz = q[3] / rho;
    return T(0.5) * rho * (Ux * Ux + Uy * Uy + Uz * Uz) * V;
}

#include "tile_kernels.inc"

// Objective partial sums (FP64): kinetic energy 0.5*rho*|U|^2*V per cell.
template <typename T>
__global__ void __launch_bounds__(BLOCK) ke_kernel(DMesh<T> m, const T* __restrict__ u, double* partial) {
    int c = blockIdx.x * blockDim.x + threadIdx.x;
    const long nIC = m.nIC;
    double v = 0.0;
    if (c < m.nIC) {
        const T q[4] = {u[c], u[nIC + c], u[2 * nIC + c], u[3 * nIC + c]};
        v = (double)kinetic_energy(q, m.vol[c]);
    }
    block_reduce_store<0>(v, partial);
}

// The same from the cells' kinetic energies.
template <typename T>
__global__ void __launch_bounds__(BLOCK) ke_sum_kernel(long nIC, const T* __restrict__ ke, double* partial) {
    const long c = (long)blockIdx.x * BLOCK + threadIdx.x;
    block_reduce_store<0>(c < nIC ? (double)ke[c] : 0.0, partial);
}

// Kinetic energy per cell segment (an ensemble of meshes in one context):
// block b covers cells segCell[k] + 256*(b - segBlock[k]) .. of segment
// k = blockSeg[b], so each segment's partials group its cells exactly as a
// context holding that segment alone would.
template <typename T>
__global__ void __launch_bounds__(BLOCK) ke_seg_kernel(DMesh<T> m, const T* __restrict__ u,
                                                       const long* __restrict__ segCell,
                                                       const int* __restrict__ segBlock,
                                                       const int* __restrict__ blockSeg, double* partial) {
    const int k = blockSeg[blockIdx.x];
    const long c = segCell[k] + (long)(blockIdx.x - segBlock[k]) * BLOCK + threadIdx.x;
    const long nIC = m.nIC;
    double v = 0.0;
    if (c < segCell[k + 1]) {
        T rho = u[c];
        T Ux = u[nIC + c] / rho, Uy = u[2 * nIC + c] / rho, Uz = u[3 * nIC + c] / rho;
        T ke = T(0.5) * rho * (Ux * Ux + Uy * Uy + Uz * Uz) * m.vol[c];
        v = (double)ke;
    }
    block_reduce_store<0>(v, partial);
}

// One block per segment: out[k] = sum of its partials, folded as
// finalize_kernel folds a whole context's.
__global__ void __launch_bounds__(BLOCK) finalize_seg_kernel(const double* __restrict__ partials,
                                                             const int* __restrict__ segBlock, double* out) {
    const int k = blockIdx.x;
    const int b0 = segBlock[k], n = segBlock[k + 1] - b0;
    const double v = fold_partials<0, BLOCK>(partials + b0, n);
    __shared__ double sh[BLOCK];
    sh[threadIdx.x] = v;
    __syncthreads();
    for (int st = BLOCK / 2; st > 0; st >>= 1) {
        if (threadIdx.x < st) sh[threadIdx.x] = sh[threadIdx.x] + sh[threadIdx.x + st];
        __syncthreads();
    }
    if (threadIdx.x == 0) out[k] = sh[0];
}

// Drag on one patch (templates/cylinder_test.py:9-19): sum (p0 nx - mu(T0)(U0x-Uix)/delta) A.
template <typename T>
__global__ void __launch_bounds__(BLOCK) drag_kernel(DMesh<T> m, Phys<T> ph, const T* __restrict__ u, int start,
                                                     int n, double* partial) {
    int k = blockIdx.x * blockDim.x + threadIdx.x;
    double v = 0.0;
    if (k < n) {
        const int f = start + k;
        const int b = f - m.nIF;
        const long nIC = m.nIC, nF = m.nF;
        T wi[5], wg[5];
        load_prim(ph, u, nIC, u, nIC, m.owner[f], wi);
        ghost_value(m, ph, b, wi, wg);
        T U0 = wg[0], p0 = wg[4], T0 = wg[3];
        T nx = m.geo[G_NX * nF + f];
        T mungUx = viscosity(ph, T0) * (U0 - wi[0]) / m.geo[G_DELTA * nF + f];
        v = (double)((p0 * nx - mungUx) * m.geo[G_A * nF + f]);
    }
    block_reduce_store<0>(v, partial);
}

template <typename T>
__global__ void __launch_bounds__(BLOCK) prim_ghost_kernel(DMesh<T> m, Phys<T> ph, const T* __restrict__ u,
                                                           const T* __restrict__ ghost, T* __restrict__ prim) {
    // prim [5][nC]: internal rows from the state, ghost rows from the ghost
    // array or (cyclic) the paired owner.
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    const long nIC = m.nIC, nBF = m.nBF, nC = (long)m.nIC + m.nBF;
    if (i >= nC) return;
    T w[5];
    if (i < m.nIC) {
        load_prim(ph, u, nIC, ghost, nBF, i, w);
    } else {
        int b = i - m.nIC;
        const DPatch P = m.patches[m.bPatch[b]];
        if (P.bcU == ADFVM_BC_CYCLIC && P.cbc == ADFVM_CBC_NONE) {
            // cyclic ghost: the paired owner, as resolved in the owner's slot
            int f = m.nIF + b;
            int c = m.owner[f];
            int partner = -1;
            for (int j = 0; j < 6; j++)
                if (m.sFace[j * nIC + c] == f) partner = m.sOther[j * nIC + c];
            load_prim(ph, u, nIC, ghost, nBF, partner, w);
        } else {
            for (int r = 0; r < 5; r++) w[r] = ghost[r * nBF + b];
        }
    }
    for (int r = 0; r < 5; r++) prim[r * nC + i] = w[r];
}

// op.gradCell over a caller field given on all nCells (reference cellNeighbours,
// no boundary update), k components.
template <typename T>
__global__ void __launch_bounds__(BLOCK) grad_field_kernel(DMesh<T> m, const int* __restrict__ cellNb,
                                                           const T* __restrict__ phi, int k, long nC,
                                                           T* __restrict__ grad) {
    int c = blockIdx.x * blockDim.x + threadIdx.x;
    if (c >= m.nIC) return;
    const long nIC = m.nIC, nF = m.nF;
    for (int comp = 0; comp < k; comp++) {
        T g0 = 0, g1 = 0, g2 = 0;
        T pc = phi[comp * nC + c];
        for (int j = 0; j < 6; j++) {
            const int f = m.sFace[j * nIC + c];
            const bool own = m.sFlags[j * nIC + c] & 1;
            const int nb = cellNb[j * nIC + c];
            T S = m.geo[G_A * nF + f];
            T N[3] = {m.geo[G_NX * nF + f], m.geo[G_NY * nF + f], m.geo[G_NZ * nF + f]};
            T w = m.geo[G_W * nF + f];
            if (!own) { N[0] = -N[0]; N[1] = -N[1]; N[2] = -N[2]; }
            else w = T(1) - w;
            T phiF = pc * (T(1) - w) + phi[comp * nC + nb] * w;
            g0 += phiF * (S * N[0]); g1 += phiF * (S * N[1]); g2 += phiF * (S * N[2]);
        }
        T V = m.vol[c];
        grad[(3 * comp + 0) * nIC + c] = g0 / V;
        grad[(3 * comp + 1) * nIC + c] = g1 / V;
        grad[(3 * comp + 2) * nIC + c] = g2 / V;
    }
}

// interp.secondOrder on every face: phi [k][nC], grad [3k][nC], out [k][nF].
template <typename T>
__global__ void __launch_bounds__(BLOCK) interp_kernel(DMesh<T> m, const int* __restrict__ nbFull,
                                                       const T* __restrict__ phi, const T* __restrict__ grad,
                                                       int k, long nC, int swap, T* __restrict__ out) {
    int f = blockIdx.x * blockDim.x + threadIdx.x;
    if (f >= m.nF) return;
    const long nF = m.nF;
    int p = m.owner[f], n = nbFull[f];
    if (swap) { int t = p; p = n; n = t; }
    T lw = m.geo[(swap ? G_LW1 : G_LW0) * nF + f];
    T qw[3];
    for (int i = 0; i < 3; i++) qw[i] = m.geo[((swap ? G_Q1X : G_Q0X) + i) * nF + f];
    for (int comp = 0; comp < k; comp++) {
        T pc = phi[comp * nC + p], pd = phi[comp * nC + n];
        T g0 = grad[(3 * comp) * nC + p], g1 = grad[(3 * comp + 1) * nC + p], g2 = grad[(3 * comp + 2) * nC + p];
        out[comp * nF + f] = pc + (pd - pc) * lw + (qw[0] * g0 + qw[1] * g1 + qw[2] * g2);
    }
}

template <typename T>
__global__ void __launch_bounds__(BLOCK) dot_kernel(const T* __restrict__ a, const T* __restrict__ b, long n,
                                                    double* partial) {
    double v = 0.0;
    for (long i = (long)blockIdx.x * BLOCK + threadIdx.x; i < n; i += (long)gridDim.x * BLOCK)
        v += (double)a[i] * (double)b[i];
    block_reduce_store<0>(v, partial);
}

// adjoint energy, cmesh.cpp:342-425 (per-cell entropy-variable quadratic form)
template <typename T>
__global__ void __launch_bounds__(BLOCK) energy_kernel(DMesh<T> m, Phys<T> ph, const T* __restrict__ ua,
                                                       const T* __restrict__ u, double* partial) {
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    const long nIC = m.nIC;
    double e = 0.0;
    if (i < m.nIC) {
        double g = (double)ph.gamma;
        double v = m.vol[i];
        double rho = u[i], rE = u[4 * nIC + i];
        double u1 = u[nIC + i] / rho, u2 = u[2 * nIC + i] / rho, u3 = u[3 * nIC + i] / rho;
        double q2 = u1 * u1 + u2 * u2 + u3 * u3;
        double p = (rE - rho * q2 / 2) * (g - 1);
        double H = g * p / (rho * (g - 1)) + q2 / 2;
        double w1 = ua[i] / v, w2 = ua[nIC + i] / v, w3 = ua[2 * nIC + i] / v, w4 = ua[3 * nIC + i] / v,
               w5 = ua[4 * nIC + i] / v;
        double A11 = rho, A12 = rho * u1, A13 = rho * u2, A14 = rho * u3, A15 = rE;
        double A22 = rho * u1 * u1 + p, A23 = rho * u1 * u2, A24 = rho * u1 * u3, A25 = rho * H * u1;
        double A33 = rho * u2 * u2 + p, A34 = rho * u2 * u3, A35 = rho * H * u2;
        double A44 = rho * u3 * u3 + p, A45 = rho * H * u3;
        double A55 = rho * H * H - g * p * p / (rho * (g - 1));
        e = (A11 * w1 * w1 + A22 * w2 * w2 + A33 * w3 * w3 + A44 * w4 * w4 + A55 * w5 * w5 +
             2 * (A12 * w1 * w2 + A13 * w1 * w3 + A14 * w1 * w4 + A15 * w1 * w5 + A23 * w2 * w3 + A24 * w2 * w4 +
                  A25 * w2 * w5 + A34 * w3 * w4 + A35 * w3 * w5 + A45 * w4 * w5)) * v;
    }
    block_reduce_store<0>(e, partial);
}

template <typename T>
__global__ void __launch_bounds__(BLOCK) pack_kernel(long n, const T* __restrict__ rho, const T* __restrict__ rhoU,
                                                     const T* __restrict__ rhoE, T* __restrict__ u) {
    long c = (long)blockIdx.x * BLOCK + threadIdx.x;
    if (c >= n) return;
    u[c] = rho[c];
    u[n + c] = rhoU[3 * c]; u[2 * n + c] = rhoU[3 * c + 1]; u[3 * n + c] = rhoU[3 * c + 2];
    u[4 * n + c] = rhoE[c];
}

template <typename T>
__global__ void __launch_bounds__(BLOCK) unpack_kernel(long n, const T* __restrict__ u, T* __restrict__ rho,
                                                       T* __restrict__ rhoU, T* __restrict__ rhoE) {
    long c = (long)blockIdx.x * BLOCK + threadIdx.x;
    if (c >= n) return;
    rho[c] = u[c];
    rhoU[3 * c] = u[n + c]; rhoU[3 * c + 1] = u[2 * n + c]; rhoU[3 * c + 2] = u[3 * n + c];
    rhoE[c] = u[4 * n + c];
}

__global__ void fill_kernel(double* p, int n, double v) {
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = v;
}

// ----------------------------------------------------------- context -----

struct adfvm_ctx {
    int prec = 4;
    int nIC = 0, nIF = 0, nF = 0, nBF = 0, nC = 0;
    int nPatches = 0;
    bool hasGhostKernel = false;
    int objective = ADFVM_OBJ_NONE, objectivePatch = -1;
    int objState = ADFVM_OBJSTATE_STAGE1;   // the state the objective is evaluated on
    int integrator = ADFVM_RK_SSPRK3;
    Phys<double> phd;
    std::string err;
    std::vector<DPatch> hpatches;
    std::vector<int> hBPatch;  // boundary face -> patch (host copy)
    // device; the tables are parts of faceTables, meshTables and tileTables
    void *faceTables = nullptr, *meshTables = nullptr, *tileTables = nullptr;
    void* geo = nullptr; void* vol = nullptr; void* bcval = nullptr;
    int* sFace = nullptr; int* sOther = nullptr; unsigned char* sFlags = nullptr; int* sPair = nullptr;
    int* owner = nullptr; int* bPatch = nullptr; DPatch* patches = nullptr;
    int* cellNbFull = nullptr;   // reference cellNeighbours [6][nIC]
    int* nbFull = nullptr;       // ghost-extended neighbour [nF]
    void* ghost = nullptr;
    // adjoint viscosity, from its first call on: [6][nIC] slot coefficients,
    // [nIC] diagonal, [nIC] eigenvalue; from its first call outside a capture on,
    // where they pay, the patches' tables (sweeps at a time, patches) and [nPos][12]
    // slot coefficients, diagonal, right side
    void* visc = nullptr;
    bool ringsTried = false;
    int ringK = 1, ringN = 0;
    RingCell* ringCell = nullptr;
    int* ringCount = nullptr;
    void* ringCoef = nullptr;
    void* st[3] = {nullptr, nullptr, nullptr};    // state records of the step's start and its intermediate stages
    void* rows1 = nullptr;     // [5][nIC] the objective stage's state in the caller's numbering
    void* rec[3] = {nullptr, nullptr, nullptr};   // [nIC][CREC] stage records
    void* adjU = nullptr;      // [nIC][5] adjoint between the stages
    void* adjAcc = nullptr;    // [nIC][5] adjoint of u0 accumulated over the stages
    void* adjG = nullptr;      // [nIC][AREC] cell adjoint records
    double* partial = nullptr; int nPartial = 0;     // [2][nPartial]: block sums; a step's objective
    double tuneMs[6] = {-1, -1, -1, -1, -1, -1};   // measured time of each stencil kernel (adfvm_autotune)
    // cell segments (adfvm_set_segments): objective per segment
    int nSeg = 1, nSegBlocks = 0;
    void* segTables = nullptr;  // the three below
    long* segCell = nullptr; int* segBlock = nullptr; int* blockSeg = nullptr;
    double* scal = nullptr;    // small device scalars
    int* fOther = nullptr; unsigned char* fKind = nullptr;
    // the streaming policy (ld / st): non-temporal single-use rows when one
    // stage's working set exceeds the Infinity Cache (adfvm_set_streaming)
    bool stream = false;
    void* meshGrad = nullptr;  // caller's mesh-geometry gradient array (adfvm_set_mesh_grad), or none
    // cell tiles (tiles.hpp), their face geometry and the cell geometry by position
    int nTiles = 0;
    long nPos() const { return (long)TILE_CELLS * nTiles; }
    long nTileFaces() const { return (long)TILE_FACES * nTiles; }
    TileRing* tileRing = nullptr;   // [nTiles], null: stages in two launches
    int* toUser = nullptr; int* toTile = nullptr; int* tileFaceId = nullptr;
    unsigned long long* tilePairs = nullptr;
    unsigned char* tileBlock = nullptr; void* tileFaceW = nullptr;
    // per-kernel event timing (adfvm_profile)
    bool prof = false;
    std::vector<hipEvent_t> evPool;
    struct Pending { const char* name; hipEvent_t a, b; };
    std::vector<Pending> pending;
    std::vector<std::string> profNames;
    std::vector<double> profMs;
    std::vector<long long> profCount;
};

namespace {

// Records a start/stop event pair around the kernel launched in its scope
// when the context's profiling is on (on the launch stream, so the timing is
// that kernel's execution on that stream).
struct KTimer {
    adfvm_ctx* c; const char* name; hipStream_t s; hipEvent_t a = nullptr, b = nullptr;
    static hipEvent_t take(adfvm_ctx* c) {
        if (!c->evPool.empty()) { hipEvent_t e = c->evPool.back(); c->evPool.pop_back(); return e; }
        hipEvent_t e = nullptr;
        if (hipEventCreate(&e) != hipSuccess) return nullptr;
        return e;
    }
    KTimer(adfvm_ctx* c_, const char* n, hipStream_t s_) : c(c_), name(n), s(s_) {
        if (!c->prof) return;
        a = take(c); b = take(c);
        if (a) (void)hipEventRecord(a, s);
    }
    ~KTimer() {
        if (!c->prof || !a || !b) return;
        (void)hipEventRecord(b, s);
        c->pending.push_back({name, a, b});
    }
};

int set_err(adfvm_ctx* ctx, int code, const std::string& m) {
    if (ctx) ctx->err = m;
    return code;
}

#define HIPCHK(ctx, expr)                                                              \
    do {                                                                               \
        hipError_t e_ = (expr);                                                        \
        if (e_ != hipSuccess)                                                          \
            return set_err(ctx, ADFVM_ERR_HIP, std::string(#expr) + ": " + hipGetErrorString(e_)); \
    } while (0)

int grid_for(long n) { return (int)((n + BLOCK - 1) / BLOCK); }
int grid_bs(long n, int bs) { return (int)((n + bs - 1) / bs); }

// The stencil kernels' names and the block sizes adfvm_set_kernel_block
// takes.  A tile fixes the blocks: TILE_CELLS threads (one per cell) for the
// gradient and its transpose, else TILE_THREADS (one per face); the flux and the
// stage update, and the face adjoint and its gather, are one kernel each.
enum { K_GRAD = 0, K_FLUX, K_STAGE, K_FVJP, K_GATHER, K_GVJP, K_TUNABLE };
const char* const kTunableName[K_TUNABLE] = {"grad_kernel", "face_flux_kernel", "stage_kernel",
                                              "face_vjp_kernel", "vjp_gather_kernel", "grad_vjp_kernel"};
const int kBlockChoices[4] = {64, 128, 256, 512};

// Calls f(std::bool_constant<st>): the streaming policy of the kernels that
// take one (ld / st).
template <typename F> void with_stream(bool st, F&& f) {
    if (st) f(std::bool_constant<true>());
    else f(std::bool_constant<false>());
}

// Calls f(std::bool_constant<gh>): whether the mesh has faces with a ghost
// (the kernels that evaluate ghosts in place are built without that code
// for meshes that have none).
template <typename F> void with_ghosts(bool gh, F&& f) {
    if (gh) f(std::bool_constant<true>());
    else f(std::bool_constant<false>());
}

// The automatic streaming policy: on when what a stage works on exceeds the
// 256 MB Infinity Cache: the tiles' blocks, the stage records and three states
// (the stage's, the step's start and the next).  Off -> on, steps in us: 268 MB (80^3
// FP32) 210 -> 213, with their adjoint steps 495 -> 490; 458 MB (96^3) 366 -> 339 and 850
// -> 803; 228 MB (410k cells of an O-grid) 178 -> 185 and 421 -> 428; FP64 263 MB
// (64^3) 225 -> 232 and 573 -> 569; 375 MB (72^3) 316 -> 304 and 793 -> 771; 215 MB (a
// 60^3 duct) 252 -> 261 and 575 -> 580.
template <typename T> bool stream_auto(const adfvm_ctx* c) {
    const double tile = TileBlock<T>::BYTES + (CREC + 15.0) * TILE_CELLS * sizeof(T);
    return c->nTiles * tile > 256.0 * (1 << 20);
}
bool stream_auto(const adfvm_ctx* c) { return c->prec == 4 ? stream_auto<float>(c) : stream_auto<double>(c); }

template <typename T> Phys<T> phys_cast(const Phys<double>& p) {
    Phys<T> o;
    o.gamma = (T)p.gamma; o.Cp = (T)p.Cp; o.Cv = (T)p.Cv; o.Pr = (T)p.Pr; o.invCv = (T)p.invCv;
    o.small = (T)p.small; o.mu0 = (T)p.mu0; o.muA = (T)p.muA; o.muTs = (T)p.muTs;
    o.muModel = p.muModel; o.riemann = p.riemann; o.boundaryRiemann = p.boundaryRiemann; o.limit = p.limit;
    return o;
}

template <typename T> DMesh<T> dmesh(const adfvm_ctx* c) {
    DMesh<T> m;
    m.nIC = c->nIC; m.nIF = c->nIF; m.nF = c->nF; m.nBF = c->nBF;
    m.geo = (const T*)c->geo; m.vol = (const T*)c->vol;
    m.sFace = c->sFace; m.sOther = c->sOther; m.sFlags = c->sFlags; m.sPair = c->sPair;
    m.owner = c->owner; m.bPatch = c->bPatch; m.patches = c->patches; m.bcval = (const T*)c->bcval;
    m.fOther = c->fOther; m.fKind = c->fKind;
    return m;
}

template <typename T> DTiles<T> dtiles(const adfvm_ctx* c) {
    DTiles<T> t;
    t.n = c->nTiles;
    t.ring = c->tileRing; t.block = c->tileBlock; t.toUser = c->toUser; t.toTile = c->toTile; t.faceId = c->tileFaceId; t.pairs = c->tilePairs;
    t.faceW = (const T*)c->tileFaceW;
    return t;
}

// The most tiles for which a stage takes one launch (20 a compute unit), and one
// whose records are kept: 4, or 1 where a compute unit holds two blocks only
// (FP64 with ghosts: 69 KB of LDS).  Measured at launch_stage.
constexpr int ONE_LAUNCH_TILES = 5120;
int one_launch_rec_tiles(const adfvm_ctx* c) { return c->prec == 8 && c->hasGhostKernel ? 256 : 1024; }

// Host tables that go to the device together, into parts of one allocation.  A
// copy takes 10 us and more whatever its size, so the small ones go as one, from a
// host buffer (a 1000-cell tube's context 0.71 -> 0.35 ms).
struct Table {
    void** part;
    const void* host;
    size_t bytes;
};
template <typename D, typename T, typename A> Table table(D*& part, const std::vector<T, A>& v) {
    return {(void**)&part, v.data(), v.size() * sizeof(T)};
}
int upload(adfvm_ctx* ctx, void** base, std::initializer_list<Table> tables) {
    constexpr size_t ALIGN = 256, SMALL = 128 << 10;
    auto padded = [](size_t bytes) { return (bytes + ALIGN - 1) / ALIGN * ALIGN; };
    size_t all = ALIGN, small = 0, at = 0;
    for (const Table& t : tables) {
        all += padded(t.bytes);
        if (t.bytes <= SMALL) small += padded(t.bytes);
    }
    HIPCHK(ctx, hipMalloc(base, all));
    Buffer<char> host(small);
    for (const Table& t : tables) {
        if (t.bytes > SMALL) continue;
        *t.part = (char*)*base + at;
        if (t.bytes) std::memcpy(host.data() + at, t.host, t.bytes);
        at += padded(t.bytes);
    }
    if (small) HIPCHK(ctx, hipMemcpy(*base, host.data(), small, hipMemcpyHostToDevice));
    for (const Table& t : tables) {
        if (t.bytes <= SMALL) continue;
        *t.part = (char*)*base + at;
        HIPCHK(ctx, hipMemcpy(*t.part, t.host, t.bytes, hipMemcpyHostToDevice));
        at += padded(t.bytes);
    }
    return ADFVM_OK;
}

// The tables by face and by patch.
template <typename T> int create_face_tables(adfvm_ctx* ctx, const adfvm_solver_desc* d) {
    const long nF = ctx->nF, nIC = ctx->nIC;
    Buffer<T> geo((size_t)G_ROWS * nF);
    over_threads((int)nF, 2 * CELL_GRAIN, [&](int a, int b, int) {
        for (long f = a; f < b; f++) {
            geo[G_A * nF + f] = (T)d->areas[f];
            for (int i = 0; i < 3; i++) geo[(G_NX + i) * nF + f] = (T)d->normals[3 * f + i];
            geo[G_W * nF + f] = (T)d->weights[f];
            geo[G_DELTA * nF + f] = (T)d->deltas[f];
            for (int i = 0; i < 3; i++) geo[(G_DX + i) * nF + f] = (T)d->deltasUnit[3 * f + i];
            geo[G_LW0 * nF + f] = (T)d->linearWeights[2 * f];
            geo[G_LW1 * nF + f] = (T)d->linearWeights[2 * f + 1];
            for (int i = 0; i < 3; i++) {
                geo[(G_Q0X + i) * nF + f] = (T)d->quadraticWeights[6 * f + i];
                geo[(G_Q1X + i) * nF + f] = (T)d->quadraticWeights[6 * f + 3 + i];
            }
        }
    });
    std::vector<T> vol(nIC);
    for (long c = 0; c < nIC; c++) vol[c] = (T)d->volumes[c];
    // boundary-condition values
    std::vector<T> vals;
    for (int p = 0; p < d->nPatches; p++) {
        const adfvm_patch_desc& P = d->patches[p];
        DPatch& D = ctx->hpatches[p];
        auto add = [&](const double* src, long cnt) -> long {
            if (!src) return -1;
            long off = (long)vals.size();
            for (long i = 0; i < cnt; i++) vals.push_back((T)src[i]);
            return off;
        };
        D.valU = add(P.valueU, 3L * P.nFaces);
        D.valT = add(P.valueT, P.nFaces);
        D.valp = add(P.valuep, P.nFaces);
        D.valTt = add(P.Tt, P.nFaces);
        D.valpt = add(P.pt, P.nFaces);
        D.valDir = add(P.direction, 3L * P.nFaces);
        D.hasDir = P.direction != nullptr;
    }
    return upload(ctx, &ctx->faceTables,
                  {table(ctx->geo, geo), table(ctx->vol, vol), table(ctx->bcval, vals), table(ctx->patches, ctx->hpatches)});
}

// The tables by tile and the work buffers.
template <typename T> int create_tile_tables(adfvm_ctx* ctx, const adfvm_solver_desc* d, const Tiles& t) {
    const Buffer<int>& toUser = t.toUser;
    const long nF = ctx->nF, nIC = ctx->nIC, nBF = ctx->nBF;
    int rc;
    if ((rc = upload(ctx, &ctx->tileTables, {table(ctx->toUser, t.toUser), table(ctx->toTile, t.toTile),
                                             table(ctx->tileFaceId, t.faceId), table(ctx->tilePairs, t.pairs)})) != ADFVM_OK)
        return rc;
    const long nPos = ctx->nPos();
    // Gauss-gradient geometry per cell slot, by position, computed in FP64 and cast once:
    // the cell's outward S*n and the weight w' of the other side's value
    // (phi_f = phi_c (1 - w') + phi_other w'), streamed by the gradient
    // kernels instead of gathering face rows.
    Buffer<T> sn((size_t)24 * nPos);
    over_threads(ctx->nTiles, TILE_GRAIN, [&](int a, int b, int) {
        for (long p = (long)a * TILE_CELLS; p < (long)b * TILE_CELLS; p++) {
            const long c = toUser[p];
            if (c < 0) {
                std::fill_n(&sn[24 * p], 24, T(0));
                continue;
            }
            for (int j = 0; j < 6; j++) {
                const long f = d->cellFaces[6 * c + j];
                const bool own = d->cellOwner[6 * c + j] != 0;
                const double sgn = own ? 1.0 : -1.0;
                const double w = d->weights[f];
                for (int k = 0; k < 3; k++) sn[24 * p + 4 * j + k] = (T)(sgn * (d->areas[f] * d->normals[3 * f + k]));
                sn[24 * p + 4 * j + 3] = (T)(own ? 1.0 - w : w);
            }
        }
    });
    {
        // the tables the blocks are filled from, freed at the end of the scope
        struct Temp {
            void* p = nullptr;
            ~Temp() { if (p) (void)hipFree(p); }
        } tmp;
        void *dsn, *nbr, *slots, *halo, *face, *over;
        const std::vector<int> none(1, 0);
        if ((rc = upload(ctx, &tmp.p, {table(dsn, sn), table(nbr, t.nbr), table(slots, t.slots), table(halo, t.halo),
                                       table(face, t.face), table(over, none)})) != ADFVM_OK)
            return rc;
        HIPCHK(ctx, hipMalloc((void**)&ctx->tileBlock, (size_t)ctx->nTiles * TileBlock<T>::BYTES));
        HIPCHK(ctx, hipMalloc(&ctx->tileFaceW, ctx->nTileFaces() * sizeof(T)));
        tile_block_kernel<T><<<ctx->nTiles, TILE_FACES>>>(
            (const T*)ctx->geo, nF, (const T*)dsn, (const unsigned long long*)nbr, (const unsigned long long*)slots,
            (const int*)halo, ctx->toUser, (const T*)ctx->vol, (const unsigned*)face, ctx->tileFaceId, ctx->tileBlock,
            (T*)ctx->tileFaceW);
        HIPCHK(ctx, hipGetLastError());
        // the rings around the tiles, where stages are to take one launch
        // (launch_stage): not where one does not fit, or the memory for them is
        // not to be had
        if (ctx->nTiles <= ONE_LAUNCH_TILES &&
            hipMalloc((void**)&ctx->tileRing, (size_t)ctx->nTiles * sizeof(TileRing)) == hipSuccess) {
            int unfit = 0;
            tile_ring_kernel<<<ctx->nTiles, TILE_HALO>>>(nIC, (const int*)halo, ctx->toUser, ctx->toTile, ctx->sOther,
                                                         ctx->sFace, ctx->fKind, ctx->tileRing, (int*)over);
            HIPCHK(ctx, hipGetLastError());
            HIPCHK(ctx, hipMemcpy(&unfit, over, sizeof(int), hipMemcpyDeviceToHost));
            if (unfit) { (void)hipFree(ctx->tileRing); ctx->tileRing = nullptr; }
        } else {
            (void)hipGetLastError();
            ctx->tileRing = nullptr;
        }
        HIPCHK(ctx, hipDeviceSynchronize());
    }
    // work buffers
    const size_t st = 5 * nIC * sizeof(T), sp = 5 * nPos * sizeof(T);
    HIPCHK(ctx, hipMalloc(&ctx->ghost, std::max<size_t>(1, 5 * nBF) * sizeof(T)));
    HIPCHK(ctx, hipMemset(ctx->ghost, 0, std::max<size_t>(1, 5 * nBF) * sizeof(T)));
    for (int i = 0; i < 3; i++) {
        HIPCHK(ctx, hipMalloc(&ctx->st[i], sp));
        HIPCHK(ctx, hipMalloc(&ctx->rec[i], (size_t)CREC * nPos * sizeof(T)));
    }
    HIPCHK(ctx, hipMalloc(&ctx->rows1, st));
    HIPCHK(ctx, hipMalloc(&ctx->adjU, sp));
    HIPCHK(ctx, hipMalloc(&ctx->adjAcc, sp));
    HIPCHK(ctx, hipMalloc(&ctx->adjG, (size_t)AREC * nPos * sizeof(T)));
    return ADFVM_OK;
}

template <typename T> T* P(void* p) { return (T*)p; }

// ghost refresh for state u (no-op for meshes with only cyclic patches)
template <typename T> void launch_ghosts(adfvm_ctx* c, const T* u, hipStream_t s) {
    if (!c->hasGhostKernel) return;
    KTimer kt(c, "ghost_kernel", s);
    ghost_kernel<T><<<grid_for(c->nBF), BLOCK, 0, s>>>(dmesh<T>(c), phys_cast<T>(c->phd), u, P<T>(c->ghost));
}

// Stage records (GONLY: gradients alone) of state u: the caller's rows (user) or
// state records; copy (nullable): u as state records.
template <typename T, bool GONLY = false> void launch_grad(adfvm_ctx* c, const T* u, bool user, T* copy, T* rec, hipStream_t s) {
    KTimer kt(c, "grad_kernel", s);
    with_stream(c->stream, [&](auto SP) {
        with_ghosts(c->hasGhostKernel, [&](auto G) {
            constexpr bool ST = decltype(SP)::value, GH = decltype(G)::value;
            grad_kernel<T, ST, GH, GONLY><<<c->nTiles, TILE_CELLS, 0, s>>>(dmesh<T>(c), dtiles<T>(c),
                                                                      phys_cast<T>(c->phd), u, user, copy, rec);
        });
    });
}

// u_{i+1} = a0*u0 + ai*u_i - beta*(L-S)*dt.  Every stage of the tables
// below with a0 != 0 has a0 + ai = 1, and the stage kernels evaluate it as
// u0 + (ai*(u_i - u0) - beta*(L-S)*dt), so sum(V*u) is kept up to unbiased
// rounding.  (Taken as a0*u0 + ai*u_i with the coefficients rounded apart,
// SSP-RK3's 1/3 and 2/3 both round up in FP32, to a sum of 1 + 2^-25: the
// state would grow by that factor every step.)  The adjoint uses a0 formed
// as 1 - ai in the compute precision, the coefficient the primal applies.
struct Stage {
    double a0, ai, beta;
    template <typename T> T a0_as() const { return a0 == 0.0 ? T(0) : T(1) - (T)ai; }
};

// Fluxes of all faces at the stage of records rec (state records u) and the
// stage update into next (state records) and rows (the caller's), or the
// residual.
template <typename T, int MODE>
void launch_flux_and_stage(adfvm_ctx* c, const T* rec, const T* u, const T* u0, const Stage& st, double dt,
                           const T* S, T* next, T* rows, T* dtcCell, double* dtcPartial, hipStream_t s,
                           T* keCell = nullptr) {
    KTimer kt(c, MODE == 0 ? "flux_stage_kernel" : "residual_kernel", s);
    with_stream(c->stream, [&](auto SP) {
        with_ghosts(c->hasGhostKernel, [&](auto G) {
            constexpr bool ST = decltype(SP)::value, GH = decltype(G)::value;
            flux_stage_kernel<T, MODE, ST, GH><<<c->nTiles, TILE_THREADS, 0, s>>>(
                dmesh<T>(c), dtiles<T>(c), phys_cast<T>(c->phd), rec, u, u0, (T)st.ai, (T)(-st.beta), (T)dt, S, next,
                rows, dtcCell, dtcPartial, keCell);
        });
    });
}

// Gradients, fluxes and the stage update (or the residual): one launch, or two
// through the records work.  u: the caller's rows (user) or state records,
// copy (nullable): its records, which the update reads; rec (nullable): where
// the stage's records are kept.
// One launch saves a launch and, where records are not kept, their way through
// memory; it forms a halo cell's gradients again in every tile beside it (2.5
// times the gradient work, from 2.6 times the slot geometry).  Steps in us,
// two -> one launches: 1000 cells in a tube FP64 44.3 -> 39.7, 32^3 FP64 70.5 ->
// 66.8, 48^3 75.9 -> 71.4 (FP64 129.5 -> 119.2), 64^3 (4.2k tiles) 129.9 -> 126.5
// (FP64 273 -> 245), 80^3 (8k tiles) 248 -> 259, 101x83x67 269 -> 279.  Steps that
// keep records with their adjoint steps: 16^3 63.3 -> 57.8, 48^3 (1.8k tiles) 160.5
// -> 159.8, 64^3 292 -> 296; cells of an O-grid 8.6k 86 -> 79, 33k 104 -> 100 (FP64
// 104 -> 96, 168 -> 168), a duct of 25k FP64 156 -> 159.  Two launches also where a tile's ring does not fit
// and where the rows written are those read.
template <typename T, int MODE>
void launch_stage(adfvm_ctx* c, const T* u, bool user, T* copy, T* rec, T* work, const T* u0, const Stage& st, double dt,
                  const T* S, T* next, T* rows, T* dtcCell, double* dtcPartial, hipStream_t s,
                  T* keCell = nullptr) {
    auto over_u = [&](const T* out, long n) { return user && out && out < u + 5L * c->nIC && u < out + n; };
    const bool overlap = over_u(rows, 5L * c->nIC) || over_u(dtcCell, c->nIC);
    if (!c->tileRing || overlap || (rec && c->nTiles > one_launch_rec_tiles(c))) {
        T* r = rec ? rec : work;
        launch_grad<T>(c, u, user, copy, r, s);
        launch_flux_and_stage<T, MODE>(c, r, user ? copy : u, u0, st, dt, S, next, rows, dtcCell, dtcPartial, s, keCell);
        return;
    }
    KTimer kt(c, MODE == 0 ? "tile_stage_kernel" : "tile_residual_kernel", s);
    with_stream(c->stream, [&](auto SP) {
        with_ghosts(c->hasGhostKernel, [&](auto G) {
            constexpr bool ST = decltype(SP)::value, GH = decltype(G)::value;
            tile_stage_kernel<T, MODE, ST, GH><<<c->nTiles, TILE_THREADS, 0, s>>>(
                dmesh<T>(c), dtiles<T>(c), phys_cast<T>(c->phd), u, user, copy, rec, u0, (T)st.ai, (T)(-st.beta), (T)dt, S,
                next, rows, dtcCell, dtcPartial, keCell);
        });
    });
}

// Whether steps turn the caller's rows into records, and back, in launches of
// their own.  In the tile kernels a tile's cells lie in runs of 3 to 6 in a row,
// of which every line is read or written by several tiles, apart in time: at
// 128^3 FP32 a step's first and last stages took 160 us longer than with records,
// the conversions take 27 each.  A step 940 -> 816 us, with its adjoint step
// 2185 -> 1962; 64^3 (4.2k tiles) 120.5 -> 115 and 279 -> 277, 72^3 382 -> 369; 48^3
// (1.8k tiles) 155 -> 157, cells of an O-grid (longer runs) 131k (2.2k tiles) 193
// -> 202, 410k (6.9k tiles) 439 -> 443.  12 tiles a compute unit:
constexpr int CONVERT_TILES = 3072;
bool converts_rows(const adfvm_ctx* c) { return c->nTiles > CONVERT_TILES; }
template <typename T> void launch_to_records(adfvm_ctx* c, const T* rows, T* rec, hipStream_t s) {
    KTimer kt(c, "to_records_kernel", s);
    to_records_kernel<T><<<grid_for(c->nIC), BLOCK, 0, s>>>(c->nIC, c->toTile, rows, rec);
}
template <typename T> void launch_to_rows(adfvm_ctx* c, const T* rec, T* rows, hipStream_t s) {
    KTimer kt(c, "to_rows_kernel", s);
    to_rows_kernel<T><<<grid_for(c->nIC), BLOCK, 0, s>>>(c->nIC, c->toTile, rec, rows);
}

template <typename T> void launch_objective(adfvm_ctx* c, const T* u, double* out, hipStream_t s) {
    KTimer kt(c, "objective", s);
    if (c->objective == ADFVM_OBJ_KINETIC_ENERGY && c->nSeg > 1) {
        ke_seg_kernel<T><<<c->nSegBlocks, BLOCK, 0, s>>>(dmesh<T>(c), u, c->segCell, c->segBlock, c->blockSeg,
                                                         c->partial);
        finalize_seg_kernel<<<c->nSeg, BLOCK, 0, s>>>(c->partial, c->segBlock, out);
    } else if (c->objective == ADFVM_OBJ_KINETIC_ENERGY) {
        int g = grid_for(c->nIC);
        ke_kernel<T><<<g, BLOCK, 0, s>>>(dmesh<T>(c), u, c->partial);
        finalize_kernel<0><<<1, FINAL_THREADS<0>, 0, s>>>(c->partial, g, out);
    } else if (c->objective == ADFVM_OBJ_DRAG) {
        const DPatch& Pp = c->hpatches[c->objectivePatch];
        int g = grid_for(Pp.n);
        drag_kernel<T><<<g, BLOCK, 0, s>>>(dmesh<T>(c), phys_cast<T>(c->phd), u, Pp.start, Pp.n, c->partial);
        finalize_kernel<0><<<1, FINAL_THREADS<0>, 0, s>>>(c->partial, g, out);
    } else {
        fill_kernel<<<grid_for(c->nSeg), BLOCK, 0, s>>>(out, c->nSeg, 0.0);   // one zero per segment
    }
}

void stages(int integrator, std::vector<Stage>& st) {
    st.clear();
    if (integrator == ADFVM_RK_EULER) { st.push_back({0, 1, 1}); return; }
    st.push_back({0.0, 1.0, 1.0});
    st.push_back({3.0 / 4.0, 1.0 / 4.0, 1.0 / 4.0});
    st.push_back({1.0 / 3.0, 2.0 / 3.0, 2.0 / 3.0});
}

// The stage whose state the step's objective is evaluated on: the first
// intermediate stage (density.py:412-413; the state a tape holds first), or
// the step's start state u_n when the caller asked for it
// (ADFVM_OBJSTATE_START; no counterpart in the reference).  dtc is taken on
// the first intermediate stage either way.
int objective_stage(const adfvm_ctx* c, int ns) {
    return (ns > 1 && c->objState == ADFVM_OBJSTATE_STAGE1) ? 1 : 0;
}

// A step tape holds the first intermediate stage's state in the caller's
// numbering (schemes of several stages; what an objective of that stage
// reads), then every stage's records: [5][nIC], [ns][nPos][CREC] scalars, both
// from 16-byte boundaries of the tape.
long tape_rows_scalars(const adfvm_ctx* c, int ns) { return ns > 1 ? (5L * c->nIC + 3) / 4 * 4 : 0; }
long tape_scalars(const adfvm_ctx* c, int ns) { return tape_rows_scalars(c, ns) + (long)ns * CREC * c->nPos(); }

template <typename T> void tape_slots(const adfvm_ctx* c, int ns, T* tape, T** rec) {
    T* r = tape + tape_rows_scalars(c, ns);
    for (int i = 0; i < ns; i++) rec[i] = r + (long)i * CREC * c->nPos();
}

template <typename T>
int primal_step_t(adfvm_ctx* c, T* u, double dt, const T* S, double* dtc_out, double* obj_out, T* tape,
                  hipStream_t s) {
    std::vector<Stage> st;
    stages(c->integrator, st);
    const int ns = (int)st.size();
    T* rec[3] = {P<T>(c->rec[0]), P<T>(c->rec[1]), P<T>(c->rec[2])};
    if (tape) tape_slots(c, ns, tape, rec);
    const int objStage = objective_stage(c, ns);
    const int dtcStage = ns > 1 ? 1 : 0;    // density.py:412-413
    // the cells' kinetic energies at the first intermediate stage come from the
    // kernel that makes it: five rows less to write, scattered by the caller's
    // numbering, and to read again (128^3 FP32 step without a tape 1005 -> 940 us)
    const bool ke1 = obj_out && objStage == 1 && c->objective == ADFVM_OBJ_KINETIC_ENERGY && c->nSeg <= 1;
    T* keCell = ke1 ? P<T>(c->rows1) : nullptr;
    double* kePartial = c->partial + c->nPartial;
    const int gKe = grid_for(c->nIC);
    // the objective stage's state in the caller's numbering, where one is needed
    T* rows1 = ns == 1 ? nullptr : tape ? tape : (obj_out && objStage == 1 && !ke1) ? P<T>(c->rows1) : nullptr;
    const bool convert = converts_rows(c);
    T* const u0rec = P<T>(c->st[0]);
    if (convert) launch_to_records<T>(c, u, u0rec, s);
    for (int i = 0; i < ns; i++) {
        if (i == objStage && obj_out && !ke1) launch_objective<T>(c, i == 0 ? u : rows1, obj_out, s);
        const bool wantDtc = (i == dtcStage) && dtc_out;
        const T* u0 = (i > 0 && st[i].a0 != 0.0) ? u0rec : nullptr;
        // the last stage writes the caller's state in place: the kernels of
        // this step read it no more (its records are st[0]); st[1] is free then
        const bool last = i == ns - 1, user = i == 0 && !convert;
        T* rows = last ? u : i == 0 ? rows1 : nullptr;
        T* next = !last ? P<T>(c->st[i + 1]) : convert ? P<T>(c->st[1]) : nullptr;
        launch_stage<T, 0>(c, user ? u : P<T>(c->st[i]), user, user ? u0rec : nullptr, tape ? rec[i] : nullptr,
                           P<T>(c->rec[i]), u0, st[i], dt, S, next, convert ? nullptr : rows, nullptr,
                           wantDtc ? c->partial : nullptr, s, i == 0 ? keCell : nullptr);
        if (convert && rows) launch_to_rows<T>(c, next, rows, s);
        if (i != dtcStage) continue;
        if (ke1) {
            KTimer kt(c, "objective", s);
            ke_sum_kernel<T><<<gKe, BLOCK, 0, s>>>(c->nIC, keCell, kePartial);
            if (wantDtc)
                finalize_step_kernel<<<2, 1024, 0, s>>>(kePartial, gKe, obj_out, c->partial, c->nTiles, dtc_out);
            else
                finalize_kernel<0><<<1, FINAL_THREADS<0>, 0, s>>>(kePartial, gKe, obj_out);
        } else if (wantDtc) {
            finalize_kernel<1><<<1, FINAL_THREADS<1>, 0, s>>>(c->partial, c->nTiles, dtc_out);
        }
    }
    HIPCHK(c, hipGetLastError());
    return ADFVM_OK;
}

}  // namespace

// ------------------------------------------------------------- C ABI -----

// Checks the mesh and the patches, and makes c's tables and work buffers.
static int fill_context(adfvm_ctx* c, const adfvm_solver_desc* d, const adfvm_physics* ph) {
    auto bad = [&](const std::string& m) { c->err = m; return ADFVM_ERR_INVALID; };
    if (ph->precision != 4 && ph->precision != 8) return bad("precision must be 4 or 8");
    c->prec = ph->precision;
    c->nIC = d->sizes.nInternalCells; c->nIF = d->sizes.nInternalFaces; c->nF = d->sizes.nFaces;
    c->nBF = d->sizes.nBoundaryFaces; c->nC = d->sizes.nCells;
    c->nPatches = d->nPatches;
    c->integrator = ph->integrator;
    c->objective = ph->objective;
    c->objectivePatch = ph->objectivePatch;
    c->phd.gamma = ph->gamma; c->phd.Cp = ph->Cp; c->phd.Cv = ph->Cp / ph->gamma; c->phd.Pr = ph->Pr;
    c->phd.invCv = 1.0 / c->phd.Cv; c->phd.small = ph->small;
    c->phd.mu0 = ph->mu0; c->phd.muA = ph->muA; c->phd.muTs = ph->muTs; c->phd.muModel = ph->muModel;
    c->phd.riemann = ph->riemann; c->phd.boundaryRiemann = ph->boundaryRiemann;
    c->phd.limit = ph->limiter;
    if (c->nIC <= 0 || c->nF <= 0 || c->nBF < 0) return bad("bad mesh sizes");
    if (c->objective == ADFVM_OBJ_DRAG && (c->objectivePatch < 0 || c->objectivePatch >= c->nPatches))
        return bad("drag objective needs a valid patch index");
    const long nIC = c->nIC, nF = c->nF, nIF = c->nIF, nBF = c->nBF;

    // boundary face -> patch, patch table
    std::vector<int> bPatch(nBF, -1);
    c->hpatches.resize(d->nPatches);
    for (int p = 0; p < d->nPatches; p++) {
        const adfvm_patch_desc& Pd = d->patches[p];
        if (Pd.startFace < nIF || Pd.startFace + Pd.nFaces > nF) return bad("patch outside boundary faces");
        for (int k = 0; k < Pd.nFaces; k++) bPatch[Pd.startFace - nIF + k] = p;
        DPatch& D = c->hpatches[p];
        D.start = Pd.startFace; D.n = Pd.nFaces; D.fluxKind = Pd.fluxKind;
        D.bcU = Pd.bcU; D.bcT = Pd.bcT; D.bcp = Pd.bcp; D.cbc = Pd.cbc;
        const bool cyc = Pd.fluxKind == ADFVM_FLUX_COUPLED;
        if (cyc && (Pd.neighbourPatch < 0 || Pd.neighbourPatch >= d->nPatches ||
                    d->patches[Pd.neighbourPatch].nFaces != Pd.nFaces))
            return bad("coupled patch without a matching neighbour patch");
        if (cyc && (Pd.bcU != ADFVM_BC_CYCLIC || Pd.bcT != ADFVM_BC_CYCLIC || Pd.bcp != ADFVM_BC_CYCLIC))
            return bad("coupled patches need cyclic conditions on U, T and p");
        if (!cyc && (Pd.bcU == ADFVM_BC_CYCLIC || Pd.bcT == ADFVM_BC_CYCLIC || Pd.bcp == ADFVM_BC_CYCLIC))
            return bad("cyclic condition on a non-coupled patch");
        if (Pd.cbc == ADFVM_CBC_UPT && (!Pd.valueU || !Pd.valueT || !Pd.valuep))
            return bad("CBC_UPT needs U0, T0, p0 values");
        if (Pd.cbc == ADFVM_CBC_TOTAL_PT && (!Pd.Tt || !Pd.pt)) return bad("CBC_TOTAL_PT needs Tt and pt");
        auto needs = [](int bc) { return bc == ADFVM_BC_FIXED_VALUE || bc == ADFVM_BC_CALCULATED; };
        if (Pd.cbc == ADFVM_CBC_NONE && ((needs(Pd.bcU) && !Pd.valueU) || (needs(Pd.bcT) && !Pd.valueT) ||
                                         (needs(Pd.bcp) && !Pd.valuep)))
            return bad("fixedValue/calculated condition without values");
        if (!cyc && Pd.nFaces > 0) c->hasGhostKernel = true;
    }
    for (long b = 0; b < nBF; b++)
        if (bPatch[b] < 0) return bad("boundary face not covered by a patch");

    // slot tables
    std::vector<int> sPair(6 * nIC, -1);
    Buffer<int> sFace(6 * nIC), sOther(6 * nIC), cellNb(6 * nIC);
    Buffer<unsigned char> sFlags(6 * nIC);
    auto slots_of = [&](long cc) -> const char* {         // the message where they are not valid
        for (int j = 0; j < 6; j++) {
            int f = d->cellFaces[6 * cc + j];
            if (f < 0 || f >= nF) return "cellFaces out of range";
            int own = d->cellOwner[6 * cc + j];
            int other, kind;
            if (f < nIF) {
                kind = SLOT_INTERNAL;
                other = own ? d->neighbour[f] : d->owner[f];
            } else {
                if (!own) return "boundary face in a neighbour slot";
                int b = f - nIF;
                const adfvm_patch_desc& Pd = d->patches[bPatch[b]];
                if (Pd.fluxKind == ADFVM_FLUX_COUPLED) {
                    kind = SLOT_COUPLED;
                    int nbStart = d->patches[Pd.neighbourPatch].startFace;
                    int pf = nbStart + (f - Pd.startFace);
                    other = d->owner[pf];
                    sPair[j * nIC + cc] = pf;
                } else {
                    kind = Pd.fluxKind == ADFVM_FLUX_CHARACTERISTIC ? SLOT_CHARACTERISTIC : SLOT_BOUNDARY;
                    other = -1 - b;
                }
            }
            sFace[j * nIC + cc] = f;
            sOther[j * nIC + cc] = other;
            sFlags[j * nIC + cc] = (unsigned char)((own ? 1 : 0) | (kind << 1));
            cellNb[j * nIC + cc] = d->cellNeighbours[6 * cc + j];
        }
        return nullptr;
    };
    std::vector<const char*> wrong(thread_parts((int)nIC, CELL_GRAIN), nullptr);
    over_threads((int)nIC, CELL_GRAIN, [&](int first, int end, int part) {
        for (long cc = first; cc < end && !wrong[part]; cc++) wrong[part] = slots_of(cc);
    });
    for (const char* w : wrong)
        if (w) return bad(w);
    // face tables: the neighbour side's value source and the flux kind
    std::vector<int> fOther(nF);
    std::vector<unsigned char> fKind(nF);
    for (long f = 0; f < nF; f++) {
        if (f < nIF) { fOther[f] = d->neighbour[f]; fKind[f] = FACE_INTERIOR; continue; }
        const long b = f - nIF;
        const adfvm_patch_desc& Pd = d->patches[bPatch[b]];
        if (Pd.fluxKind == ADFVM_FLUX_COUPLED) {
            fOther[f] = d->owner[d->patches[Pd.neighbourPatch].startFace + (f - Pd.startFace)];
            fKind[f] = FACE_INTERIOR;
        } else {
            fOther[f] = (int)(-1 - b);
            fKind[f] = Pd.fluxKind == ADFVM_FLUX_CHARACTERISTIC ? FACE_CHARACTERISTIC : FACE_BOUNDARY;
        }
    }
    // every face must have one slot per side; a cyclic face's neighbour side
    // is the paired cell's, which takes it with its own slot (tiles.hpp)
    std::vector<int> posP(nF, -1), posN(nF, -1);
    int maxExtra = 0;
    for (long cc = 0; cc < nIC; cc++) {
        int e = 0;
        for (int j = 0; j < 6; j++) {
            const int fl = sFlags[j * nIC + cc];
            const int f = sFace[j * nIC + cc];
            int& slot = (fl & 1) ? posP[f] : posN[f];
            if (slot != -1) return bad("face in two slots of the same side");
            slot = (int)cc;
            if (slot_kind(fl) == SLOT_COUPLED) e++;
        }
        maxExtra = std::max(maxExtra, e);
    }
    if ((long)(6 + maxExtra) * nIC > 0x7fffffffL) return bad("mesh too large for 32-bit record indices");
    for (long cc = 0; cc < nIC; cc++) {
        for (int j = 0; j < 6; j++) {
            if (slot_kind(sFlags[j * nIC + cc]) != SLOT_COUPLED) continue;
            const int g = sPair[j * nIC + cc];
            if (posN[g] != -1) return bad("face with two neighbour-side slots");
            posN[g] = (int)cc;
        }
    }
    for (long f = 0; f < nF; f++) {
        if (posP[f] < 0) return bad("face without an owner slot");
        if (fKind[f] == FACE_INTERIOR && posN[f] < 0) return bad("face without a neighbour-side slot");
    }
    for (long b = 0; b < nBF; b++)
        if (ghost_copies_owner(d->patches[bPatch[b]])) fKind[nIF + b] |= FACE_GHOST_COPY;
    // the tiles grow on a thread of their own while the other tables go to the
    // device (a 24.7k-cell duct's context 5.4 -> 4.8 ms, 64^3 62 -> 48); on this one,
    // at get(), where a thread is not to be had or would do little (1000 cells)
    const auto policy = nIC < CELL_GRAIN ? std::launch::deferred : std::launch::async | std::launch::deferred;
    std::future<Tiles> tiles = std::async(policy, [&] {
        Tiles t;
        build_tiles(TileMesh{(int)nIC, (int)nIF, (int)nF, sFace.data(), sOther.data(), sPair.data(), sFlags.data(),
                             fKind.data(), FACE_GHOST_COPY}, t);
        return t;
    });
    int rc;
    std::vector<int> owner(d->owner, d->owner + nF), nbFull(d->neighbour, d->neighbour + nF);
    if ((rc = upload(c, &c->meshTables, {table(c->fOther, fOther), table(c->fKind, fKind), table(c->sFace, sFace),
                                         table(c->sOther, sOther), table(c->sFlags, sFlags), table(c->sPair, sPair),
                                         table(c->cellNbFull, cellNb), table(c->owner, owner), table(c->nbFull, nbFull),
                                         table(c->bPatch, bPatch)})) != ADFVM_OK)
        return rc;
    c->hBPatch = bPatch;
    rc = c->prec == 4 ? create_face_tables<float>(c, d) : create_face_tables<double>(c, d);
    if (rc != ADFVM_OK) return rc;
    const Tiles t = tiles.get();
    c->nTiles = t.n;
    rc = c->prec == 4 ? create_tile_tables<float>(c, d, t) : create_tile_tables<double>(c, d, t);
    if (rc != ADFVM_OK) return rc;
    c->stream = stream_auto(c);
    c->nPartial = std::max(grid_bs(std::max<long>(nIC, nF), kBlockChoices[0]) + 1, c->nTiles);   // the smallest block size
    HIPCHK(c, hipMalloc((void**)&c->partial, 2L * c->nPartial * sizeof(double)));
    HIPCHK(c, hipMalloc((void**)&c->scal, 16 * sizeof(double)));
    return ADFVM_OK;
}

extern "C" int adfvm_ctx_create(const adfvm_solver_desc* d, const adfvm_physics* ph, adfvm_ctx** out) {
    if (!d || !ph || !out) return ADFVM_ERR_INVALID;
    *out = nullptr;
    try {
        *out = new adfvm_ctx();
        return fill_context(*out, d, ph);
    } catch (const std::exception& e) {
        if (*out) (*out)->err = std::string("set-up of the mesh tables: ") + e.what();
        return ADFVM_ERR_INVALID;
    }
}

extern "C" void adfvm_ctx_destroy(adfvm_ctx* c) {
    if (!c) return;
    void* ptrs[] = {c->faceTables, c->meshTables, c->tileTables, c->ghost, c->st[0], c->st[1], c->st[2], c->rows1,
                    c->rec[0], c->rec[1], c->rec[2], c->adjU, c->adjAcc, c->adjG, c->partial, c->scal, c->tileBlock,
                    c->tileRing, c->tileFaceW, c->segTables, c->visc, c->ringCell, c->ringCount,
                    c->ringCoef};
    for (void* p : ptrs)
        if (p) (void)hipFree(p);
    for (auto& p : c->pending) { (void)hipEventDestroy(p.a); (void)hipEventDestroy(p.b); }
    for (auto e : c->evPool) (void)hipEventDestroy(e);
    delete c;
}

extern "C" const char* adfvm_last_error(const adfvm_ctx* c) { return c ? c->err.c_str() : "null context"; }

#ifndef ADFVM_SOURCE_HASH
#define ADFVM_SOURCE_HASH "unknown"
#endif
extern "C" const char* adfvm_source_hash(void) { return ADFVM_SOURCE_HASH; }
extern "C" int adfvm_ctx_precision(const adfvm_ctx* c) { return c ? c->prec : 0; }

namespace {
template <typename T> int set_bc_values_t(adfvm_ctx* c, long off, const double* v, long n, hipStream_t s) {
    std::vector<T> h(v, v + n);
    HIPCHK(c, hipMemcpyAsync((T*)c->bcval + off, h.data(), n * sizeof(T), hipMemcpyHostToDevice, s));
    HIPCHK(c, hipStreamSynchronize(s));
    return ADFVM_OK;
}
}  // namespace

extern "C" int adfvm_set_bc_values(adfvm_ctx* c, int32_t patch, int32_t slot, const double* values, int64_t n,
                                   void* stream) {
    if (!c || !values) return ADFVM_ERR_INVALID;
    if (patch < 0 || patch >= c->nPatches) return set_err(c, ADFVM_ERR_INVALID, "patch index out of range");
    const DPatch& D = c->hpatches[patch];
    long off;
    int k = 1;
    switch (slot) {
        case ADFVM_BCV_U: off = D.valU; k = 3; break;
        case ADFVM_BCV_T: off = D.valT; break;
        case ADFVM_BCV_P: off = D.valp; break;
        case ADFVM_BCV_TT: off = D.valTt; break;
        case ADFVM_BCV_PT: off = D.valpt; break;
        case ADFVM_BCV_DIRECTION: off = D.valDir; k = 3; break;
        default: return set_err(c, ADFVM_ERR_INVALID, "unknown boundary-value slot");
    }
    if (off < 0) return set_err(c, ADFVM_ERR_INVALID, "this patch was created without that value array");
    if (n != (int64_t)k * D.n) return set_err(c, ADFVM_ERR_INVALID, "value count is not nFaces x components");
    hipStream_t s = (hipStream_t)stream;
    return c->prec == 4 ? set_bc_values_t<float>(c, off, values, n, s) : set_bc_values_t<double>(c, off, values, n, s);
}

extern "C" int adfvm_set_segments(adfvm_ctx* c, int32_t nSeg, const int64_t* cellStart) {
    if (!c || nSeg < 1 || !cellStart) return ADFVM_ERR_INVALID;
    if (cellStart[0] != 0 || cellStart[nSeg] != c->nIC)
        return set_err(c, ADFVM_ERR_INVALID, "segments must start at cell 0 and end at nInternalCells");
    for (int k = 0; k < nSeg; k++)
        if (cellStart[k + 1] <= cellStart[k]) return set_err(c, ADFVM_ERR_INVALID, "empty or decreasing segment");
    if (nSeg > 1 && c->objective == ADFVM_OBJ_DRAG)
        return set_err(c, ADFVM_ERR_UNSUPPORTED, "segments with the drag objective");
    std::vector<long> cells(cellStart, cellStart + nSeg + 1);
    std::vector<int> first(nSeg + 1), owner;
    first[0] = 0;
    for (int k = 0; k < nSeg; k++) {
        int nb = grid_for(cells[k + 1] - cells[k]);
        first[k + 1] = first[k] + nb;
        for (int b = 0; b < nb; b++) owner.push_back(k);
    }
    if (first[nSeg] > c->nPartial) return set_err(c, ADFVM_ERR_INVALID, "too many segment blocks");
    if (c->segTables) (void)hipFree(c->segTables);
    c->segTables = nullptr; c->segCell = nullptr; c->segBlock = nullptr; c->blockSeg = nullptr;
    const int rc = upload(c, &c->segTables, {table(c->segCell, cells), table(c->segBlock, first), table(c->blockSeg, owner)});
    if (rc != ADFVM_OK) return rc;
    c->nSeg = nSeg;
    c->nSegBlocks = first[nSeg];
    return ADFVM_OK;
}

extern "C" int adfvm_segments(const adfvm_ctx* c) { return c ? c->nSeg : 0; }

extern "C" int adfvm_set_objective_state(adfvm_ctx* c, int32_t which) {
    if (!c) return ADFVM_ERR_INVALID;
    if (which != ADFVM_OBJSTATE_STAGE1 && which != ADFVM_OBJSTATE_START)
        return set_err(c, ADFVM_ERR_INVALID, "objective state must be ADFVM_OBJSTATE_STAGE1 or ADFVM_OBJSTATE_START");
    c->objState = which;
    return ADFVM_OK;
}

extern "C" int adfvm_objective_state(const adfvm_ctx* c) { return c ? c->objState : -1; }

#define DISPATCH(c, CALL_F, CALL_D) ((c)->prec == 4 ? (CALL_F) : (CALL_D))

extern "C" int adfvm_primal_step(adfvm_ctx* c, void* u, double dt, const void* S, double* dtc_out,
                                 double* obj_out, void* tape, void* stream) {
    if (!c || !u) return ADFVM_ERR_INVALID;
    hipStream_t s = (hipStream_t)stream;
    return DISPATCH(c, primal_step_t<float>(c, (float*)u, dt, (const float*)S, dtc_out, obj_out, (float*)tape, s),
                    primal_step_t<double>(c, (double*)u, dt, (const double*)S, dtc_out, obj_out, (double*)tape, s));
}

namespace {
template <typename T> int gradients_t(adfvm_ctx* c, const T* u, T* grad, hipStream_t s) {
    // as steps do, but in a buffer that steps with a tape do not use.  100^3 FP32
    // 88.5 us on the rows, 71 with the conversion; 64^3 24.8 and 23.9 (FP64 41.3 and
    // 41.1); O-grids of longer runs 30 and 32 (410k cells)
    const bool convert = converts_rows(c);
    if (convert) launch_to_records<T>(c, u, P<T>(c->rec[1]), s);
    launch_grad<T, true>(c, convert ? P<T>(c->rec[1]) : u, !convert, nullptr, P<T>(c->rec[0]), s);
    grad_rows_kernel<T><<<grid_for(c->nIC), BLOCK, 0, s>>>(dtiles<T>(c), c->nIC, P<T>(c->rec[0]), grad);
    HIPCHK(c, hipGetLastError());
    return ADFVM_OK;
}
template <typename T> int residual_t(adfvm_ctx* c, const T* u, T* R, T* dtcCell, hipStream_t s) {
    launch_stage<T, 1>(c, u, true, nullptr, nullptr, P<T>(c->rec[0]), nullptr, Stage{0, 0, 0}, 0.0, nullptr, nullptr, R,
                       dtcCell, nullptr, s);
    HIPCHK(c, hipGetLastError());
    return ADFVM_OK;
}
template <typename T> int objective_t(adfvm_ctx* c, const T* u, double* out, hipStream_t s) {
    launch_objective<T>(c, u, out, s);
    HIPCHK(c, hipGetLastError());
    return ADFVM_OK;
}
template <typename T> int prim_t(adfvm_ctx* c, const T* u, T* prim, hipStream_t s) {
    launch_ghosts<T>(c, u, s);
    prim_ghost_kernel<T><<<grid_for((long)c->nIC + c->nBF), BLOCK, 0, s>>>(dmesh<T>(c), phys_cast<T>(c->phd), u,
                                                                           P<T>(c->ghost), prim);
    HIPCHK(c, hipGetLastError());
    return ADFVM_OK;
}
}  // namespace

extern "C" int adfvm_gradients(adfvm_ctx* c, const void* u, void* grad, void* stream) {
    if (!c || !u || !grad) return ADFVM_ERR_INVALID;
    hipStream_t s = (hipStream_t)stream;
    return DISPATCH(c, gradients_t<float>(c, (const float*)u, (float*)grad, s),
                    gradients_t<double>(c, (const double*)u, (double*)grad, s));
}

extern "C" int adfvm_residual(adfvm_ctx* c, const void* u, void* R, void* dtcCell, void* stream) {
    if (!c || !u || !R) return ADFVM_ERR_INVALID;
    hipStream_t s = (hipStream_t)stream;
    return DISPATCH(c, residual_t<float>(c, (const float*)u, (float*)R, (float*)dtcCell, s),
                    residual_t<double>(c, (const double*)u, (double*)R, (double*)dtcCell, s));
}

extern "C" int adfvm_objective(adfvm_ctx* c, const void* u, double* out, void* stream) {
    if (!c || !u || !out) return ADFVM_ERR_INVALID;
    hipStream_t s = (hipStream_t)stream;
    return DISPATCH(c, objective_t<float>(c, (const float*)u, out, s), objective_t<double>(c, (const double*)u, out, s));
}

extern "C" int adfvm_primitive_ghosts(adfvm_ctx* c, const void* u, void* prim, void* stream) {
    if (!c || !u || !prim) return ADFVM_ERR_INVALID;
    hipStream_t s = (hipStream_t)stream;
    return DISPATCH(c, prim_t<float>(c, (const float*)u, (float*)prim, s), prim_t<double>(c, (const double*)u, (double*)prim, s));
}

extern "C" int adfvm_grad_cell(adfvm_ctx* c, const void* phi, int32_t k, void* grad, void* stream) {
    if (!c || !phi || !grad || k <= 0) return ADFVM_ERR_INVALID;
    hipStream_t s = (hipStream_t)stream;
    long nC = (long)c->nIC + c->nBF;
    if (c->prec == 4)
        grad_field_kernel<float><<<grid_for(c->nIC), BLOCK, 0, s>>>(dmesh<float>(c), c->cellNbFull, (const float*)phi, k, nC, (float*)grad);
    else
        grad_field_kernel<double><<<grid_for(c->nIC), BLOCK, 0, s>>>(dmesh<double>(c), c->cellNbFull, (const double*)phi, k, nC, (double*)grad);
    HIPCHK(c, hipGetLastError());
    return ADFVM_OK;
}

extern "C" int adfvm_interp_second_order(adfvm_ctx* c, const void* phi, const void* grad, int32_t k, int32_t swap,
                                         void* out, void* stream) {
    if (!c || !phi || !grad || !out || k <= 0 || (swap != 0 && swap != 1)) return ADFVM_ERR_INVALID;
    hipStream_t s = (hipStream_t)stream;
    long nC = (long)c->nIC + c->nBF;
    if (c->prec == 4)
        interp_kernel<float><<<grid_for(c->nF), BLOCK, 0, s>>>(dmesh<float>(c), c->nbFull, (const float*)phi, (const float*)grad, k, nC, swap, (float*)out);
    else
        interp_kernel<double><<<grid_for(c->nF), BLOCK, 0, s>>>(dmesh<double>(c), c->nbFull, (const double*)phi, (const double*)grad, k, nC, swap, (double*)out);
    HIPCHK(c, hipGetLastError());
    return ADFVM_OK;
}

extern "C" int adfvm_dot(adfvm_ctx* c, const void* a, const void* b, int64_t n, double* out, void* stream) {
    if (!c || !a || !b || !out || n < 0) return ADFVM_ERR_INVALID;
    hipStream_t s = (hipStream_t)stream;
    int g = std::min<long>(std::max<long>(grid_for(n), 1), c->nPartial);
    if (c->prec == 4) dot_kernel<float><<<g, BLOCK, 0, s>>>((const float*)a, (const float*)b, n, c->partial);
    else dot_kernel<double><<<g, BLOCK, 0, s>>>((const double*)a, (const double*)b, n, c->partial);
    finalize_kernel<0><<<1, FINAL_THREADS<0>, 0, s>>>(c->partial, g, out);
    HIPCHK(c, hipGetLastError());
    return ADFVM_OK;
}

// ---- the allocation-free dot product ------------------------------------
// Block partials of adfvm_dot_noalloc live in this file-scope array, one
// copy per GPU, held until the process ends.  In host code its name is not a
// device address: the address each device holds it at is looked up once per
// device (hipGetSymbolAddress with that device current) and only that
// pointer is passed to kernels.
constexpr long kScratchDoubles = 1L << 19;        // 4 MiB: n <= 2^19 * 256 scalars
static __device__ __align__(256) double scratch[kScratchDoubles];

namespace {
constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
double* g_scratch_ptr[kMaxDevices];

// The current device's copy of scratch (nullptr and a message on failure).
double* scratch_on_current_device(std::string& err) {
    int dev = -1;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices) {
        err = "no current HIP device (or device index >= 64)";
        return nullptr;
    }
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    if (!g_scratch_ptr[dev]) {
        void* ptr = nullptr;
        hipError_t e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
        if (e != hipSuccess || !ptr) {
            err = std::string("hipGetSymbolAddress(scratch): ") + hipGetErrorString(e);
            return nullptr;
        }
        g_scratch_ptr[dev] = (double*)ptr;
    }
    return g_scratch_ptr[dev];
}
thread_local std::string g_noalloc_err;
}  // namespace

extern "C" const char* adfvm_noalloc_last_error(void) { return g_noalloc_err.c_str(); }

extern "C" int adfvm_dot_noalloc(int32_t precision, const void* a, const void* b, int64_t n, double* out,
                                 void* stream) {
    g_noalloc_err.clear();
    if ((n > 0 && (!a || !b)) || !out || n < 0 || (precision != 4 && precision != 8)) {
        g_noalloc_err = "adfvm_dot_noalloc: null pointer, negative n or precision not 4/8";
        return ADFVM_ERR_INVALID;
    }
    const long g = std::max<long>(grid_for(n), 1);
    if (g > kScratchDoubles) {
        g_noalloc_err = "adfvm_dot_noalloc: n = " + std::to_string((long long)n) + " exceeds the maximum " +
                        std::to_string((long long)(kScratchDoubles * BLOCK)) + " scalars";
        return ADFVM_ERR_INVALID;
    }
    double* part = scratch_on_current_device(g_noalloc_err);
    if (!part) return ADFVM_ERR_HIP;
    hipStream_t s = (hipStream_t)stream;
    // every one of the g partials is written by dot_kernel before
    // finalize_kernel reads it, so nothing needs clearing
    if (precision == 4) dot_kernel<float><<<(int)g, BLOCK, 0, s>>>((const float*)a, (const float*)b, n, part);
    else dot_kernel<double><<<(int)g, BLOCK, 0, s>>>((const double*)a, (const double*)b, n, part);
    finalize_kernel<0><<<1, FINAL_THREADS<0>, 0, s>>>(part, (int)g, out);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) {
        g_noalloc_err = std::string("adfvm_dot_noalloc: ") + hipGetErrorString(e);
        return ADFVM_ERR_HIP;
    }
    return ADFVM_OK;
}

extern "C" int adfvm_adjoint_energy(adfvm_ctx* c, const void* ua, const void* u, double* out, void* stream) {
    if (!c || !ua || !u || !out) return ADFVM_ERR_INVALID;
    hipStream_t s = (hipStream_t)stream;
    int g = grid_for(c->nIC);
    if (c->prec == 4) energy_kernel<float><<<g, BLOCK, 0, s>>>(dmesh<float>(c), phys_cast<float>(c->phd), (const float*)ua, (const float*)u, c->partial);
    else energy_kernel<double><<<g, BLOCK, 0, s>>>(dmesh<double>(c), phys_cast<double>(c->phd), (const double*)ua, (const double*)u, c->partial);
    finalize_kernel<0><<<1, FINAL_THREADS<0>, 0, s>>>(c->partial, g, out);
    HIPCHK(c, hipGetLastError());
    return ADFVM_OK;
}

extern "C" int adfvm_pack_state(adfvm_ctx* c, const void* rho, const void* rhoU, const void* rhoE, void* u, void* stream) {
    if (!c || !rho || !rhoU || !rhoE || !u) return ADFVM_ERR_INVALID;
    hipStream_t s = (hipStream_t)stream;
    if (c->prec == 4) pack_kernel<float><<<grid_for(c->nIC), BLOCK, 0, s>>>(c->nIC, (const float*)rho, (const float*)rhoU, (const float*)rhoE, (float*)u);
    else pack_kernel<double><<<grid_for(c->nIC), BLOCK, 0, s>>>(c->nIC, (const double*)rho, (const double*)rhoU, (const double*)rhoE, (double*)u);
    HIPCHK(c, hipGetLastError());
    return ADFVM_OK;
}

extern "C" int adfvm_unpack_state(adfvm_ctx* c, const void* u, void* rho, void* rhoU, void* rhoE, void* stream) {
    if (!c || !rho || !rhoU || !rhoE || !u) return ADFVM_ERR_INVALID;
    hipStream_t s = (hipStream_t)stream;
    if (c->prec == 4) unpack_kernel<float><<<grid_for(c->nIC), BLOCK, 0, s>>>(c->nIC, (const float*)u, (float*)rho, (float*)rhoU, (float*)rhoE);
    else unpack_kernel<double><<<grid_for(c->nIC), BLOCK, 0, s>>>(c->nIC, (const double*)u, (double*)rho, (double*)rhoU, (double*)rhoE);
    HIPCHK(c, hipGetLastError());
    return ADFVM_OK;
}

#include "mesh_adjoint.inc"
#include "adjoint_kernels.inc"
#include "viscosity.inc"
