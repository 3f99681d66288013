// On-device solve of the assembled system Lλx·Δx = Lλ for chain topologies, and the
// Newton-Newmark decrement that consumes Δx (the host steps of src/SweepX.jl:205-211 and
// src/SweepX.jl:98-132 for models whose elements join their nodes into paths).
//
// Block layout
//   The X dofs of one node form one block of B (3 or 6) positions; blocks follow the
//   nodes along each path, paths one after another. Lλx is then block tridiagonal:
//     D[i]  rows of block i, columns of block i        (B×B, column-major: entry (r, c)
//     L[i]  rows of block i, columns of block i-1       at i·B² + c·B + r, so that the rows
//     U[i]  rows of block i, columns of block i+1       of one CSC column land contiguously)
//   Two paths meet with zero L/U blocks, so many chains form one system. A node with
//   fewer than B dofs is padded with identity rows (zero solution).
//   At prepare, slot_kernel gives each nz of Lλx its destination (slot) in D|L|U, and the
//   slots no nz covers are listed; a solve zeroes those, then scatters nzval by slot with
//   coalesced reads.
//   The λ dof of a Hold (src/BasicElements.jl:426-438) is coupled to its held dof h only:
//   row λ reads cL·x_h = r_λ (its diagonal is zero), row h holds cU·λ. The λ row fixes x_h;
//   the pack replaces row h of the block system by that equation, saving the original row
//   so that λ = (r_h − Σ_j K_hj x_j)/cU once x is known.
//
// Block cyclic reduction (no pivoting between blocks, partial pivoting inside a block)
//   level s = 1, 2, 4, …: blocks i ≡ s (mod 2s) are eliminated, blocks j ≡ 0 (mod 2s) kept.
//   eliminate: L_i ← D_i⁻¹L_i, U_i ← D_i⁻¹U_i, b_i ← D_i⁻¹b_i by Gauss-Jordan elimination    (in place)
//   update:    D_j −= L_j U_{j−s} + U_j L_{j+s};  b_j −= L_j b_{j−s} + U_j b_{j+s};
//              L_j ← −L_j L_{j−s} (couples j−2s),  U_j ← −U_j U_{j+s} (couples j+2s)
//   top:       x_0 = D_0⁻¹ b_0
//   back:      for s descending, x_i = b_i − L_i x_{i−s} − U_i x_{i+s}     (x overwrites b)
//   Six levels run in a workgroup's LDS at a time (reduce_kernel): the eliminated blocks of a chunk
//   go back in place, its first block to the system of the next phase.
#pragma once
#include <hip/hip_runtime.h>
#include <cmath>
#include <cstdint>

namespace chain {

constexpr int kCB = 256;

enum : unsigned {
    kBadPattern = 1u,    // an entry outside the block-tridiagonal / λ-pair structure
    kSingular = 2u,      // zero or non-finite pivot in a diagonal block
    kBadPair = 4u,       // a λ row with a nonzero diagonal or a zero coupling
};

// The status words of a solve: flag (the k* bits) at word 0, then, as 64-bit values at
// byte 8 and 16, the bad pivot's place (singular_block) and the first bad λ pair (all ones: none).
constexpr int kStatusBytes = 24;
__device__ inline unsigned long long* status_where(unsigned* f) { return reinterpret_cast<unsigned long long*>(f + 2); }
// A diagonal block's place in the order of elimination: its level (block i = s + 2s·t leaves at level
// s, block 0 is the last one), then the block. The least one is kept: a zero pivot makes later levels'
// blocks of other workgroups bad too, whenever those run.
constexpr int kPlaceShift = 48;
__device__ inline void singular_block(unsigned* f, unsigned long long block) {
    atomicOr(f, kSingular);
    const unsigned long long level = block ? (unsigned long long)__builtin_ctzll(block) : 63ull;
    atomicMin(status_where(f), level << kPlaceShift | block);
}
__global__ void clear_flag(unsigned* f) {
    f[0] = 0u;
    status_where(f)[0] = ~0ull;
    status_where(f)[1] = ~0ull;
}

__global__ __launch_bounds__(kCB) void fill_f64(int64_t n, double* __restrict__ p, double v) {
    const int64_t i = (int64_t)blockIdx.x * kCB + threadIdx.x;
    if (i < n) p[i] = v;
}

__global__ __launch_bounds__(kCB) void fill_i32(int64_t n, int32_t* __restrict__ p, int32_t v) {
    const int64_t i = (int64_t)blockIdx.x * kCB + threadIdx.x;
    if (i < n) p[i] = v;
}

// Prepare: one thread per column c of the CSC pattern. slot[k] of each nz k: ≥ 0, its index
// in D|L|U; −(4p + w + 1), coupling w (0: cL, row λ col h; 1: cU, row h col λ; 2: the λ
// diagonal) of λ pair p. unc[q] is cleared for every slot q that an nz covers.
// pos[d] ≥ 0: block position of dof d; pos[d] = −(p+1): the λ dof of pair p.
template <int B>
__global__ __launch_bounds__(kCB) void slot_kernel(int64_t nX, int64_t nb, const int32_t* __restrict__ colptr,
                                                   const int32_t* __restrict__ rowval, const int32_t* __restrict__ pos,
                                                   const int32_t* __restrict__ hpos, int32_t* __restrict__ slot,
                                                   int32_t* __restrict__ unc, unsigned* __restrict__ flag) {
    const int64_t c = (int64_t)blockIdx.x * kCB + threadIdx.x;
    if (c >= nX) return;
    const int64_t BB = (int64_t)B * B;
    const int32_t pcol = pos[c];
    bool bad = false;
    const int32_t k1 = colptr[c + 1];
    for (int32_t k = colptr[c]; k < k1; ++k) {
        const int32_t prow = pos[rowval[k]];
        int64_t q = -1;
        if (pcol >= 0 && prow >= 0) {
            const int64_t br = prow / B, bc = pcol / B;
            const int64_t o = br * BB + (pcol - bc * B) * B + (prow - br * B);
            if (br == bc) q = o;
            else if (br == bc + 1) q = nb * BB + o;
            else if (br + 1 == bc) q = 2 * nb * BB + o;
            else bad = true;
            if (q >= 0) { slot[k] = (int32_t)q; unc[q] = 0; }
        } else if (pcol < 0 && prow < 0) {
            if (pcol == prow) slot[k] = -(4 * (-pcol - 1) + 2 + 1);
            else bad = true;
        } else if (pcol < 0) {
            const int32_t p = -pcol - 1;
            if (prow == hpos[p]) slot[k] = -(4 * p + 1 + 1);
            else bad = true;
        } else {
            const int32_t p = -prow - 1;
            if (pcol == hpos[p]) slot[k] = -(4 * p + 0 + 1);
            else bad = true;
        }
        if (bad) slot[k] = INT32_MIN;
    }
    if (bad) atomicOr(flag, kBadPattern);
}

// Prepare: the list of uncovered slots (positions from an exclusive scan of unc).
__global__ __launch_bounds__(kCB) void compact_kernel(int64_t n, const int32_t* __restrict__ unc,
                                                      const int32_t* __restrict__ at, int32_t* __restrict__ list) {
    const int64_t q = (int64_t)blockIdx.x * kCB + threadIdx.x;
    if (q < n && unc[q]) list[at[q]] = (int32_t)q;
}

__global__ __launch_bounds__(kCB) void zero_slots_kernel(int64_t n, const int32_t* __restrict__ list,
                                                         double* __restrict__ DLU) {
    const int64_t q = (int64_t)blockIdx.x * kCB + threadIdx.x;
    if (q < n) DLU[list[q]] = 0.0;
}

// Prepare: slots as offsets into the whole chain buffer D|L|U|b|pc (a λ coupling −(4p+w+1)
// becomes pcbase + 4p + w), so that one map serves the pack and an assembly that scatters
// straight into the blocks.
__global__ __launch_bounds__(kCB) void absolute_slot_kernel(int64_t nnz, int64_t pcbase, int32_t* __restrict__ slot) {
    const int64_t k = (int64_t)blockIdx.x * kCB + threadIdx.x;
    if (k >= nnz) return;
    const int32_t q = slot[k];
    if (q < 0 && q != INT32_MIN) slot[k] = (int32_t)(pcbase - (int64_t)q - 1);
}

// One thread per nz: nzval into the chain buffer by slot (coalesced reads; the rows of one
// column are contiguous slots of D|L|U; λ couplings go to pc).
__global__ __launch_bounds__(kCB) void pack_kernel(int64_t nnz, const int32_t* __restrict__ slot,
                                                   const double* __restrict__ nzval, double* __restrict__ cbuf) {
    const int64_t k = (int64_t)blockIdx.x * kCB + threadIdx.x;
    if (k >= nnz) return;
    const int32_t q = __builtin_nontemporal_load(slot + k);
    cbuf[q] = __builtin_nontemporal_load(nzval + k);
}

// One thread per dof: Lλ into b, or into the λ pair's r_λ.
__global__ __launch_bounds__(kCB) void pack_rhs_kernel(int64_t nX, const int32_t* __restrict__ pos,
                                                       const double* __restrict__ rhs, double* __restrict__ b,
                                                       double* __restrict__ pc) {
    const int64_t d = (int64_t)blockIdx.x * kCB + threadIdx.x;
    if (d >= nX) return;
    const int32_t p = pos[d];
    if (p >= 0) b[p] = rhs[d];
    else pc[4 * (int64_t)(-p - 1) + 3] = rhs[d];
}

// One thread per λ pair: save row h (L | D | U parts and r_h), replace it by x_h = r_λ/cL. Then one
// per padding position: its identity row (its slots are uncovered, so zeroed before).
template <int B>
__global__ __launch_bounds__(kCB) void pair_kernel(int64_t np, const int32_t* __restrict__ hpos,
                                                   const double* __restrict__ pc, double* __restrict__ D,
                                                   double* __restrict__ L, double* __restrict__ U,
                                                   double* __restrict__ b, double* __restrict__ saved,
                                                   unsigned* __restrict__ flag, int64_t ndum,
                                                   const int32_t* __restrict__ dpos) {
    const int64_t p = (int64_t)blockIdx.x * kCB + threadIdx.x;
    if (p >= np) {
        if (p - np < ndum) {
            const int64_t q = dpos[p - np], blk = q / B, i = q - blk * B;
            D[blk * B * B + i * B + i] = 1.0;
            b[q] = 0.0;
        }
        return;
    }
    const double cL = pc[4 * p], cU = pc[4 * p + 1], dg = pc[4 * p + 2], rl = pc[4 * p + 3];
    if (dg != 0.0 || cL == 0.0 || cU == 0.0) {
        atomicOr(flag, kBadPair);
        atomicMin(status_where(flag) + 1, (unsigned long long)p);
    }
    const int64_t h = hpos[p], blk = h / B, i = h - blk * B;
    double* sv = saved + p * (3 * B + 1);
    const int64_t o = blk * B * B + i;    // row i of the blocks: entries o + j·B
#pragma unroll
    for (int j = 0; j < B; ++j) {
        sv[j] = L[o + j * B];
        sv[B + j] = D[o + j * B];
        sv[2 * B + j] = U[o + j * B];
        L[o + j * B] = 0.0;
        U[o + j * B] = 0.0;
        D[o + j * B] = (j == i) ? 1.0 : 0.0;
    }
    sv[3 * B] = b[h];
    b[h] = rl / cL;
}

// ---- block cyclic reduction, several levels per launch -------------------------------------
// A workgroup takes a chunk of C consecutive blocks into LDS, eliminates all of them but the
// first (log₂ C levels) and leaves a system of the chunks' first blocks, C times smaller, to the
// next phase; the last phase (at most kTopBlocks blocks) is one workgroup, which also
// back-substitutes. The equations are those of the level-by-level reduction above.
// Bound: latency, the pivots of a level one after another at two workgroups per CU (6.37 million blocks:
// 7.0 ms for the 10.3 GB of the first phase, 1.5 TB/s, each block read once and its D⁻¹L, D⁻¹U, D⁻¹b written
// once); for few blocks the chain of levels. One launch per level and kernel before took three launches and a pass over
// the kept blocks each. Measured on whole Newton iterations of SweepX{2}: 225,000 blocks
// 2.29 → 1.93 ms, 102 blocks 247 → 179 µs; the adjoint solve and gradients of 180 risers (23,000
// blocks) 717 → 426 µs.
// kChunk: 65 blocks of 912 B fill 58 KB of LDS, two workgroups per CU, and six levels per launch;
// kTopBlocks: 128 blocks (114 KB) are what one workgroup's LDS holds with its powers of two.
constexpr int kChunk = 64;
constexpr int kTopBlocks = 128;
constexpr int kReduceThreads = 512;
constexpr int kTopThreads = 1024;

// The block system of one phase. A block's diagonal and right-hand side come in two parts from
// phase 1 on: its own chunk's (D, b) and the previous chunk's (D2, b2, which also gives L).
struct System {
    int64_t n = 0;        // blocks
    int64_t stride = 1;   // blocks of the chain per block of this phase (for the status word)
    double *D = nullptr, *D2 = nullptr, *L = nullptr, *U = nullptr, *b = nullptr, *b2 = nullptr;
};

// A block in LDS: its 3B+1 columns L | D | U | b of B entries. One lane per column: kGroups<B>
// blocks side by side in a wave, lane g·(3B+1)+q the column q of the wave's block g.
template <int B> constexpr int kCols = 3 * B + 1;
template <int B> constexpr int kGroups = 64 / kCols<B>;

template <int B>
__device__ inline void load_col(const double* __restrict__ p, double (&v)[B]) {
#pragma unroll
    for (int r = 0; r < B; ++r) v[r] = p[r];
}

// Gauss-Jordan elimination with partial pivoting of the block whose columns the lanes of a group
// hold: the L, U and b lanes end with D⁻¹L, D⁻¹U, D⁻¹b. base: the group's first lane. Every lane
// takes part (the columns of D are exchanged by shuffles).
template <int B>
__device__ inline bool gauss_jordan(double (&v)[B], int base) {
    bool ok = true;
#pragma unroll
    for (int k = 0; k < B; ++k) {
        double p[B];
#pragma unroll
        for (int r = 0; r < B; ++r) p[r] = __shfl(v[r], base + B + k);
        int q = k;
        double m = fabs(p[k]);
#pragma unroll
        for (int r = k + 1; r < B; ++r) {
            const double a = fabs(p[r]);
            if (a > m) { m = a; q = r; }
        }
#pragma unroll
        for (int r = k + 1; r < B; ++r) {
            const bool sw = q == r;
            const double tp = p[k], tv = v[k];
            p[k] = sw ? p[r] : tp; p[r] = sw ? tp : p[r];
            v[k] = sw ? v[r] : tv; v[r] = sw ? tv : v[r];
        }
        ok = ok && p[k] != 0.0 && isfinite(p[k]);
        v[k] = v[k] / p[k];
#pragma unroll
        for (int r = 0; r < B; ++r)
            if (r != k) v[r] -= p[r] * v[k];
    }
    return ok;
}

// All levels s = 1, 2, 4, … < lim of the m blocks in LDS (M[block][column][row]): blocks
// i ≡ s (mod 2s), i < E, are eliminated, blocks j ≡ 0 (mod 2s) kept and updated. Eliminated
// blocks go to global memory (L, U, b at the chunk's first block) unless L is null.
// block0, stride: for the status word of a zero pivot.
template <int B, int NT>
__device__ inline void reduce_levels(double* __restrict__ M, int m, int E, int lim, double* __restrict__ L,
                                     double* __restrict__ U, double* __restrict__ b, int64_t block0, int64_t stride,
                                     unsigned* __restrict__ flag) {
    constexpr int NC = kCols<B>, G = kGroups<B>, NG = NT / 64 * G, BS = NC * B;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int g = lane / NC, q = lane - g * NC;
    const bool in = g < G;
    const int base = in ? g * NC : 0;
    for (int s = 1; s < lim; s *= 2) {
        const int ne = E > s ? (E - s + 2 * s - 1) / (2 * s) : 0;
        for (int t0 = 0; t0 < ne; t0 += NG) {           // uniform over the workgroup
            const int t = t0 + wave * G + g;
            const bool live = in && t < ne;
            const int i = s + 2 * s * t;
            double v[B];
#pragma unroll
            for (int r = 0; r < B; ++r) v[r] = 0.0;
            double* col = M + (live ? i : 0) * BS + q * B;
            if (live) load_col<B>(col, v);
            const bool ok = gauss_jordan<B>(v, base);
            if (live) {
                if (!ok && q == 0) singular_block(flag, (unsigned long long)((block0 + i) * stride));
                if (q < B || q >= 2 * B) {
#pragma unroll
                    for (int r = 0; r < B; ++r) col[r] = v[r];
                    if (L) {
                        double* d = q < B ? L + (int64_t)i * B * B + q * B
                                          : (q < 3 * B ? U + (int64_t)i * B * B + (q - 2 * B) * B : b + (int64_t)i * B);
#pragma unroll
                        for (int r = 0; r < B; ++r) d[r] = v[r];
                    }
                }
            }
        }
        __syncthreads();
        const int nk = (m + 2 * s - 1) / (2 * s);
        for (int t0 = 0; t0 < nk; t0 += NG) {
            const int t = t0 + wave * G + g;
            const int j = 2 * s * t;
            if (in && t < nk) {
                double* blk = M + j * BS;
                double a[B];
                const bool isD = q >= B && q < 2 * B, isL = q < B, isU = q >= 2 * B && q < 3 * B;
#pragma unroll
                for (int r = 0; r < B; ++r) a[r] = (isL || isU) ? 0.0 : blk[q * B + r];
                const bool left = j >= s, right = j + s < E;
                if (left && !isU) {          // − L_j · (U, L or b column of the left neighbour)
                    const double* nb = M + (j - s) * BS + (isD ? q + B : q) * B;
#pragma unroll
                    for (int k = 0; k < B; ++k) {
                        const double f = nb[k];
#pragma unroll
                        for (int r = 0; r < B; ++r) a[r] -= blk[k * B + r] * f;
                    }
                }
                if (right && !isL) {         // − U_j · (L, U or b column of the right neighbour)
                    const double* nb = M + (j + s) * BS + (isD ? q - B : q) * B;
#pragma unroll
                    for (int k = 0; k < B; ++k) {
                        const double f = nb[k];
#pragma unroll
                        for (int r = 0; r < B; ++r) a[r] -= blk[(2 * B + k) * B + r] * f;
                    }
                }
                // the lanes of a block are one wave's: every read above is done
                __builtin_amdgcn_wave_barrier();
#pragma unroll
                for (int r = 0; r < B; ++r) blk[q * B + r] = a[r];
            }
        }
        __syncthreads();
    }
}

// One phase: a workgroup per chunk of kChunk blocks; y: the system of the next phase.
template <int B>
__global__ __launch_bounds__(kReduceThreads) void reduce_kernel(System x, System y, unsigned* __restrict__ flag) {
    constexpr int NC = kCols<B>, BS = NC * B, BB = B * B;
    __shared__ double M[(kChunk + 1) * BS];
    const int64_t ck = blockIdx.x, k0 = ck * kChunk;
    const int cnt = (int)(x.n - k0 < kChunk ? x.n - k0 : kChunk);
    const bool next = k0 + kChunk < x.n;       // the next chunk's first block bounds this one on the right
    for (int f = threadIdx.x; f < cnt * BB; f += kReduceThreads) {
        const int i = f / BB, e = f - i * BB;
        double* blk = M + i * BS;
        blk[e] = x.L[k0 * BB + f];
        blk[BB + e] = x.D2 ? x.D[k0 * BB + f] + x.D2[k0 * BB + f] : x.D[k0 * BB + f];
        blk[2 * BB + e] = x.U[k0 * BB + f];
    }
    for (int f = threadIdx.x; f < cnt * B; f += kReduceThreads) {
        const int i = f / B, e = f - i * B;
        M[i * BS + 3 * BB + e] = x.b2 ? x.b[k0 * B + f] + x.b2[k0 * B + f] : x.b[k0 * B + f];
    }
    if (next)   // only what this chunk's elimination adds to it, and its coupling to the left
        for (int f = threadIdx.x; f < BS; f += kReduceThreads)
            M[kChunk * BS + f] = f < BB ? x.L[(k0 + kChunk) * BB + f] : 0.0;
    __syncthreads();
    reduce_levels<B, kReduceThreads>(M, next ? kChunk + 1 : cnt, cnt, kChunk, x.L + k0 * BB, x.U + k0 * BB, x.b + k0 * B,
                                     k0, x.stride, flag);
    for (int f = threadIdx.x; f < BB; f += kReduceThreads) {
        y.D[ck * BB + f] = M[BB + f];
        y.U[ck * BB + f] = next ? M[2 * BB + f] : 0.0;
        if (next) {
            y.D2[(ck + 1) * BB + f] = M[kChunk * BS + BB + f];
            y.L[(ck + 1) * BB + f] = M[kChunk * BS + f];
        }
        if (ck == 0) { y.D2[f] = 0.0; y.L[f] = 0.0; }
    }
    if (threadIdx.x < B) {
        y.b[ck * B + threadIdx.x] = M[3 * BB + threadIdx.x];
        if (next) y.b2[(ck + 1) * B + threadIdx.x] = M[kChunk * BS + 3 * BB + threadIdx.x];
        if (ck == 0) y.b2[threadIdx.x] = 0.0;
    }
}

// The last phase, one workgroup: x.n ≤ kTopBlocks blocks reduced to one, solved, and
// back-substituted; the solution overwrites x.b.
template <int B>
__global__ __launch_bounds__(kTopThreads) void top_kernel(System x, unsigned* __restrict__ flag) {
    constexpr int NC = kCols<B>, BS = NC * B, BB = B * B;
    __shared__ double M[kTopBlocks * BS];
    const int n = (int)x.n;
    for (int f = threadIdx.x; f < n * BB; f += kTopThreads) {
        const int i = f / BB, e = f - i * BB;
        double* blk = M + i * BS;
        blk[e] = x.L[f];
        blk[BB + e] = x.D2 ? x.D[f] + x.D2[f] : x.D[f];
        blk[2 * BB + e] = x.U[f];
    }
    for (int f = threadIdx.x; f < n * B; f += kTopThreads) {
        const int i = f / B, e = f - i * B;
        M[i * BS + 3 * BB + e] = x.b2 ? x.b[f] + x.b2[f] : x.b[f];
    }
    __syncthreads();
    reduce_levels<B, kTopThreads>(M, n, n, n, nullptr, nullptr, nullptr, 0, x.stride, flag);
    if (threadIdx.x < 64) {                    // the last block: one group of the first wave
        const int q = threadIdx.x;
        double v[B];
#pragma unroll
        for (int r = 0; r < B; ++r) v[r] = 0.0;
        if (q < NC) load_col<B>(M + q * B, v);
        const bool ok = gauss_jordan<B>(v, 0);
        if (q == 0 && !ok) singular_block(flag, 0ull);
        if (q == 3 * B) {
#pragma unroll
            for (int r = 0; r < B; ++r) M[3 * BB + r] = v[r];
        }
    }
    __syncthreads();
    int s = 1;
    while (2 * s < n) s *= 2;
    for (; s >= 1; s /= 2) {
        const int ne = n > s ? (n - s + 2 * s - 1) / (2 * s) : 0;
        for (int w = threadIdx.x; w < ne * B; w += kTopThreads) {
            const int t = w / B, r = w - t * B, i = s + 2 * s * t;
            double* blk = M + i * BS;
            const double* xl = M + (i - s) * BS + 3 * BB;
            double a = blk[3 * BB + r];
#pragma unroll
            for (int k = 0; k < B; ++k) a -= blk[k * B + r] * xl[k];
            if (i + s < n) {
                const double* xr = M + (i + s) * BS + 3 * BB;
#pragma unroll
                for (int k = 0; k < B; ++k) a -= blk[2 * BB + k * B + r] * xr[k];
            }
            blk[3 * BB + r] = a;
        }
        __syncthreads();
    }
    for (int f = threadIdx.x; f < n * B; f += kTopThreads) {
        const int i = f / B, e = f - i * B;
        x.b[f] = M[i * BS + 3 * BB + e];
    }
}

// Back substitution of one phase: a workgroup per chunk, one lane per row of its blocks; the
// lane's row of D⁻¹L, D⁻¹U is loaded before the levels run. xr: the solution of the next
// phase (the chunks' first blocks). The solution overwrites x.b.
template <int B>
__global__ __launch_bounds__(kChunk* B) void back_kernel(System x, const double* __restrict__ xr) {
    constexpr int BB = B * B;
    __shared__ double xs[(kChunk + 1) * B];
    const int64_t ck = blockIdx.x, k0 = ck * kChunk;
    const int cnt = (int)(x.n - k0 < kChunk ? x.n - k0 : kChunk);
    const bool next = k0 + kChunk < x.n;
    const int i = threadIdx.x / B, r = threadIdx.x - i * B;
    const bool live = i > 0 && i < cnt;
    double cl[B], cu[B], a = 0.0;
    if (live) {
        const double* Li = x.L + (k0 + i) * BB + r;
        const double* Ui = x.U + (k0 + i) * BB + r;
#pragma unroll
        for (int k = 0; k < B; ++k) { cl[k] = Li[k * B]; cu[k] = Ui[k * B]; }
        a = x.b[(k0 + i) * B + r];
    }
    if (i == 0) {
        xs[r] = xr[ck * B + r];
        xs[kChunk * B + r] = next ? xr[(ck + 1) * B + r] : 0.0;
    }
    const int lev = i & -i;                    // the level at which block i was eliminated
    __syncthreads();
    for (int s = kChunk / 2; s >= 1; s /= 2) {
        if (live && lev == s) {
            const double* xl = xs + (i - s) * B;
#pragma unroll
            for (int k = 0; k < B; ++k) a -= cl[k] * xl[k];
            if (i + s < cnt || (next && i + s == kChunk)) {
                const double* xq = xs + (i + s) * B;
#pragma unroll
                for (int k = 0; k < B; ++k) a -= cu[k] * xq[k];
            }
            xs[i * B + r] = a;
        }
        __syncthreads();
    }
    if (i < cnt) x.b[(k0 + i) * B + r] = xs[i * B + r];
}

// Δx of dof c: x at the dof's position, or λ from the saved row of its held dof.
struct Unpack {
    int64_t nb = 0;
    const int32_t *pos = nullptr, *hpos = nullptr;
    const double *pc = nullptr, *saved = nullptr, *x = nullptr;
};
template <int B>
__device__ inline double unpack_dof(const Unpack& u, int64_t c) {
    const int32_t pc_ = u.pos[c];
    if (pc_ >= 0) return u.x[pc_];
    const int64_t p = -pc_ - 1;
    const int64_t h = u.hpos[p], blk = h / B;
    const double* sv = u.saved + p * (3 * B + 1);
    double r = sv[3 * B];
    if (blk > 0)
        for (int k = 0; k < B; ++k) r -= sv[k] * u.x[(blk - 1) * B + k];
    for (int k = 0; k < B; ++k) r -= sv[B + k] * u.x[blk * B + k];
    if (blk + 1 < u.nb)
        for (int k = 0; k < B; ++k) r -= sv[2 * B + k] * u.x[(blk + 1) * B + k];
    return r / u.pc[4 * p + 1];
}
template <int B>
__global__ __launch_bounds__(kCB) void unpack_kernel(int64_t nX, Unpack u, double* __restrict__ dx) {
    const int64_t c = (int64_t)blockIdx.x * kCB + threadIdx.x;
    if (c < nX) dx[c] = unpack_dof<B>(u, c);
}

// Newmarkβdecrement!{OX} (src/SweepX.jl:98-132) over all X dofs, in the host's operation
// order and without contraction, so that a given Δx decrements the state bitwise as the
// host loop does; per-block partial sums of Δx² and Lλ².
// k: the Newmark coefficients (a₁,a₂,a₃,b₁,b₂,b₃) in device memory, so that a captured graph
// replays with the current ones. B > 0: Δx is taken from the solve's blocks (and kept in dx).
template <int B>
__global__ __launch_bounds__(kCB) void newmark_kernel(int64_t nX, int OX, int first, const double* __restrict__ k,
                                                      Unpack u, double* __restrict__ dx, const double* __restrict__ rhs,
                                                      const double* __restrict__ scale, double* __restrict__ X0,
                                                      double* __restrict__ X1, double* __restrict__ X2,
                                                      double* __restrict__ part) {
#pragma clang fp contract(off)
    __shared__ double s1[kCB], s2[kCB];
    const double a1 = k[0], a2 = k[1], a3 = k[2], b1 = k[3], b2 = k[4], b3 = k[5];
    const int64_t c = (int64_t)blockIdx.x * kCB + threadIdx.x;
    double q1 = 0.0, q2 = 0.0;
    if (c < nX) {
        double d;
        if constexpr (B > 0) dx[c] = d = unpack_dof<B>(u, c);
        else d = dx[c];
        const double sc = scale[c], r = rhs[c];
        q1 = d * d;
        q2 = r * r;
        if (OX == 2) {
            double d1, d2;
            if (first) {
                const double x1 = X1[c] / sc, x2 = X2[c] / sc;
                const double a = a2 * x1 + a3 * x2, bb = b2 * x1 + b3 * x2;
                d1 = a1 * d + a;
                d2 = b1 * d + bb;
            } else {
                d1 = a1 * d;
                d2 = b1 * d;
            }
            X0[c] -= d * sc;
            X1[c] -= d1 * sc;
            X2[c] -= d2 * sc;
        } else if (OX == 1) {
            double d1;
            if (first) {
                const double a = a2 * (X1[c] / sc);
                d1 = a1 * d + a;
            } else {
                d1 = a1 * d;
            }
            X0[c] -= d * sc;
            X1[c] -= d1 * sc;
        } else {
            X0[c] -= d * sc;
        }
    }
    s1[threadIdx.x] = q1;
    s2[threadIdx.x] = q2;
    __syncthreads();
    for (int w = kCB / 2; w > 0; w >>= 1) {
        if ((int)threadIdx.x < w) { s1[threadIdx.x] += s1[threadIdx.x + w]; s2[threadIdx.x] += s2[threadIdx.x + w]; }
        __syncthreads();
    }
    if (threadIdx.x == 0) { part[2 * blockIdx.x] = s1[0]; part[2 * blockIdx.x + 1] = s2[0]; }
}
// One workgroup: the partial sums in a fixed order (deterministic), and the solve's status words; both
// to pinned host memory.
__global__ __launch_bounds__(kCB) void norm_kernel(int64_t npart, const double* __restrict__ part,
                                                   double* __restrict__ out, const unsigned* __restrict__ status,
                                                   unsigned* __restrict__ hstatus) {
    __shared__ double s1[kCB], s2[kCB];
    double q1 = 0.0, q2 = 0.0;
    for (int64_t k = threadIdx.x; k < npart; k += kCB) { q1 += part[2 * k]; q2 += part[2 * k + 1]; }
    s1[threadIdx.x] = q1;
    s2[threadIdx.x] = q2;
    __syncthreads();
    for (int w = kCB / 2; w > 0; w >>= 1) {
        if ((int)threadIdx.x < w) { s1[threadIdx.x] += s1[threadIdx.x + w]; s2[threadIdx.x] += s2[threadIdx.x + w]; }
        __syncthreads();
    }
    if (threadIdx.x == 0) { out[0] = s1[0]; out[1] = s2[0]; }
    if (threadIdx.x < kStatusBytes / 4) hstatus[threadIdx.x] = status[threadIdx.x];
}

}  // namespace chain
