// emu_state.hip -- the fused RK4 step on a library-owned, cell-sorted SoA
// particle state (the integrator loop of main.cpp:129-213).
//
// Per step (stage s reads the grid deposited from the stage-s state):
//   stage 1..3 kernels (emu_stage.h): gather + Hamiltonian + commutator + RK
//     update of the particle, then deposit of the next stage state into
//     another grid; stage 1 also finds each particle's move over the step and
//     its rank in it;
//   a stable counting sort plan by the new cell (counts beside stage 2, bases
//     beside stage 3);
//   stage 4 kernel: y_{n+1}, positions, periodic shift, Renormalize (FP64),
//     each particle written straight to its slot in the new cell order; and
//     compute_dt's maximum over the stage-4 deposit (main.cpp:193-197);
//   the deposit of y_{n+1} that the next step's stage 1 reads; and the next dt.
// Five launches, the plan riding on two of them, or seven on large grids, with
// the plan's two on a second stream (kInlinePlanCells).  Three grids take turns,
// so that each stage sets to its base the one that a later stage deposits into,
// in the same launch.
//
// The mesh holds, per cell and flavour component c, the combined fields
//   M_c  = N_c - conj(Nbar)_c  (+ rho Ye/Mp dV on 00, the matter term)
//   Phi_d,c = F_d,c - conj(Fbar_d,c),  d = x, y, z
// which is all the Hamiltonian needs (H_SI = sqrt2 GF/dV (M - p.Phi),
// Hbar = conj(H_vac - H_SI - H_matter), generate_code.py:296-357); compute_dt
// additionally needs N_ii, Nbar_ii and Im(Fbar_d) off the diagonal, which the
// stage-3 kernel deposits into an auxiliary grid.
#include "emu_internal.h"
#include "emu_stage.h"

#include <hipcub/hipcub.hpp>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <vector>

namespace emu {
namespace {

// Base value of the deposit grid: zero except the matter term rho Ye/Mp dV
// on M_00 (inside_parentheses of generate_code.py:335-342, moved into the
// field because it enters the gather with the same weights).
__global__ void k_fill_grid(double* g, int64_t ncell, int Q, double m00, double* aux, int naux)
{
    const int64_t n = ncell * Q;
    for (int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; t < n; t += (int64_t)gridDim.x * blockDim.x)
        g[t] = (t % Q) == 0 ? m00 : 0.0;
    if (aux) {
        const int64_t na = ncell * naux;
        for (int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; t < na; t += (int64_t)gridDim.x * blockDim.x)
            aux[t] = 0.0;
    }
}

// The sort plan by itself: its part of stage 2 or of stage 3.
template <int S> __global__ __launch_bounds__(256) void k_plan(SortPlan plan, Geom g, int ncell)
{
    const int wave = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (wave >= plan.waves) return;
    if (S == 2) plan.counts(wave, lane, g, ncell);
    else plan.bases(wave, lane, g, ncell);
}

template <typename T> using Arrays = PArrays<T>;

// compute_dt over the cells (Evolve.cpp:40-56) from the combined fields and
// the auxiliaries.  HSI = N - conj(Nbar) + matter = M; F - Fbar keeps Re and the
// diagonal of Phi and takes Im(F - Fbar) = Im(Phi) - 2 Im(Fbar).  The
// auxiliaries hold S_ii = N_ii + Nbar_ii, so N_ii = (S_ii + M_ii - m00 d_i0) / 2
// and Nbar_ii = (S_ii - M_ii + m00 d_i0) / 2, then Im(Fbar_ab) per direction.
template <int NF>
__global__ void k_dt_reduce(const double* __restrict__ grid, const double* __restrict__ aux, int64_t ncell,
                            double cell_volume, double m00, int adaptive, unsigned long long* red)
{
    constexpr int nh = NH<NF>;
    constexpr int QG = 4 * nh;
    constexpr int NAUX = NF + 3 * (NF * (NF - 1) / 2);
    const int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    double Vad = 0.0, Vst = 0.0;
    if (t < ncell) {
        const double* G = grid + t * QG;
        const double* A = aux + t * NAUX;
        // the adaptive bound (only where max_adaptive_speedup > 1 uses it: the
        // stage kernel then deposits Im(Fbar) as well)
        if (adaptive) {
            double h[nh];
#pragma unroll
            for (int c = 0; c < nh; c++) h[c] = G[c];
            double V2 = su_mag2<NF, double>(h);
#pragma unroll
            for (int d = 0; d < 3; d++) {
#pragma unroll
                for (int c = 0; c < nh; c++) h[c] = G[(d + 1) * nh + c];
                int o = NF;
#pragma unroll
                for (int x = 0; x < NF; x++)
#pragma unroll
                    for (int y = x + 1; y < NF; y++) {
                        h[herm_im<NF>(x, y)] -= 2.0 * A[o + d];
                        o += 3;
                    }
                V2 += su_mag2<NF, double>(h);
            }
            Vad = sqrt(V2) * M_SQRT2 * phys::GF / cell_volume;
        }
#pragma unroll
        for (int x = 0; x < NF; x++) {
            const double Mxx = G[herm_re<NF>(x, x)] - (x == 0 ? m00 : 0.0);
            const double Nxx = 0.5 * (A[x] + Mxx), Nbxx = 0.5 * (A[x] - Mxx);
            Vst = Vst > Nxx ? Vst : Nxx;
            Vst = Vst > Nbxx ? Vst : Nbxx;
        }
        Vst = Vst > m00 ? Vst : m00;
        Vst *= 2.0 * NF * M_SQRT2 * phys::GF / cell_volume;
    }
    for (int off = 32; off > 0; off >>= 1) {
        Vad = fmax(Vad, __shfl_xor(Vad, off));
        Vst = fmax(Vst, __shfl_xor(Vst, off));
    }
    if ((threadIdx.x & 63) == 0) {
        if (adaptive) atomicMax(&red[0], (unsigned long long)__double_as_longlong(Vad > 0 ? Vad : 0.0));
        atomicMax(&red[DtRed::slot(blockIdx.x)], (unsigned long long)__double_as_longlong(Vst > 0 ? Vst : 0.0));
    }
}

// The starting dt, after a load.
__global__ void k_dt_finalize(unsigned long long* red, DtParams p, double* dt, unsigned long long* err)
{
    const double h = next_dt(red, p, err); // one wave
    if (threadIdx.x == 0) *dt = h;
}

__global__ void k_fill_int(int* p, int64_t n, int v)
{
    for (int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; t < n; t += (int64_t)gridDim.x * blockDim.x) p[t] = v;
}

__global__ void k_fill_u64v(unsigned long long* p, int n, unsigned long long v)
{
    if ((int)threadIdx.x < n) p[threadIdx.x] = v;
}

// Load: bin every particle of a caller's SoA view (PIdx order).
__global__ void k_bin_input(PView P, Geom g, int* cellidx, int* counts)
{
    for (int64_t ip = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; ip < P.np; ip += (int64_t)gridDim.x * blockDim.x) {
        int nc[3];
        for (int d = 0; d < 3; d++) nc[d] = bin1(P.pos[d][ip], g.plo[d], g.dxi[d], g.n[d]);
        const int c = (nc[2] * g.n[1] + nc[1]) * g.n[0] + nc[0];
        cellidx[ip] = c;
        atomicAdd(&counts[c], 1);
    }
}

__global__ void k_iota(int* p, int64_t n)
{
    for (int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; t < n; t += (int64_t)gridDim.x * blockDim.x)
        p[t] = (int)t;
}

// Load: cnt[c] = particles binned in c; counts[c] becomes the slots they take
// (rounded up to a multiple of align).  counts[ncell] and cnt[ncell] stay 0.
__global__ void k_pad_counts(int* __restrict__ counts, int* __restrict__ cnt, int64_t ncell, int align)
{
    for (int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; t <= ncell; t += (int64_t)gridDim.x * blockDim.x) {
        const int n = t < ncell ? counts[t] : 0;
        cnt[t] = n;
        counts[t] = (n + align - 1) / align * align;
    }
}

// Load: the j-th particle in (cell, input index) order is input particle
// order[j] of cell key[j]; it takes slot start[key] + (j - ustart[key]), where
// ustart are the cells' first positions back to back and start their slots.
__global__ void k_load_slots(const int* __restrict__ order, const int* __restrict__ key, const int* __restrict__ start,
                             const int* __restrict__ ustart, int64_t np, int* __restrict__ slot)
{
    for (int64_t j = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; j < np; j += (int64_t)gridDim.x * blockDim.x) {
        const int c = key[j];
        slot[order[j]] = start[c] + ((int)j - ustart[c]);
    }
}

// A loaded particle as one record of 8-byte words: position, id, then in T
// pup[4], N, Nbar, L, Lbar and the flavour rows.  A record has exactly the bytes
// that the particle takes in a copy of the state's arrays.
template <int NF, typename T> struct LoadRec {
    static constexpr int nh = NH<NF>, N = 4, L = 6, F = 8; // T entries after the 4 words
    static constexpr int words = 4 + (8 + 2 * nh) * (int)sizeof(T) / 8;
    static constexpr int row = words | 1; // LDS row stride: odd, so that rows spread over the banks
    static constexpr int waves = 2;       // per workgroup, 2 x 64 rows of LDS (32 KB at most)
};

// The load goes through records because the caller's particles come in their
// own order (a run under way has scattered directions): reading every array
// through the sort order fetched a cache line per value (12 ms at 24.1 M
// particles).  Here a wave reads its 64 particles coalesced, transposes them in
// LDS and writes each record in one piece to its slot; k_load_unpack then turns
// the records, in slot order, into the state's arrays (together 5.1 ms in
// FP32-bulk, 8.0 in FP64).
template <int NF, typename T>
__global__ __launch_bounds__((64 * LoadRec<NF, T>::waves)) void k_load_pack(PView P, const int64_t* __restrict__ ids,
                                                                            const int* __restrict__ slot,
                                                                            int64_t* __restrict__ rec, double nscale)
{
    using I = PIdx<NF>;
    using R = LoadRec<NF, T>;
    constexpr int nh = R::nh;
    __shared__ int64_t lds[64 * R::waves * R::row];
    const int lane = threadIdx.x & 63;
    int64_t* wl = lds + (threadIdx.x - lane) * R::row;
    const int64_t ip = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    const bool act = ip < P.np;
    const int64_t ipl = act ? ip : P.np - 1;
    const int k = act ? slot[ipl] : -1;
    {
        int64_t* r = wl + lane * R::row;
        T* t = (T*)(r + 4);
        for (int d = 0; d < 3; d++) r[d] = __double_as_longlong(P.pos[d][ipl]);
        r[3] = ids ? ids[ipl] : ipl;
        for (int d = 0; d < 4; d++) t[d] = T(P.r[I::pupx + d][ipl]);
        t[R::N] = T(P.r[I::N][ipl] * nscale);
        t[R::N + 1] = T(P.r[I::Nbar][ipl] * nscale);
        t[R::L] = T(P.r[I::L][ipl]);
        t[R::L + 1] = T(P.r[I::Lbar][ipl]);
#pragma unroll
        for (int c = 0; c < nh; c++) {
            t[R::F + c] = T(P.r[I::f + c][ipl]);
            t[R::F + nh + c] = T(P.r[I::fbar + c][ipl]);
        }
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
    for (int j = 0; j < R::words; j++) {
        const int e = j * 64 + lane, r = e / R::words, w = e - r * R::words;
        const int dst = __shfl(k, r);
        if (dst >= 0) rec[(int64_t)dst * R::words + w] = wl[r * R::row + w];
    }
}

// The records of all `cap` slots into the state's arrays (slots between the
// cells' runs hold nothing, before and after).
template <int NF, typename T>
__global__ __launch_bounds__((64 * LoadRec<NF, T>::waves)) void k_load_unpack(const int64_t* __restrict__ rec,
                                                                              Arrays<T> dst, int64_t cap)
{
    using R = LoadRec<NF, T>;
    constexpr int nh = R::nh;
    __shared__ int64_t lds[64 * R::waves * R::row];
    const int lane = threadIdx.x & 63;
    int64_t* wl = lds + (threadIdx.x - lane) * R::row;
    const int64_t k0 = blockIdx.x * (int64_t)blockDim.x + (threadIdx.x - lane), k = k0 + lane;
    const int64_t n = (cap - k0 < 64 ? cap - k0 : 64) * R::words; // words of this wave's records
#pragma unroll
    for (int j = 0; j < R::words; j++) {
        const int e = j * 64 + lane, r = e / R::words, w = e - r * R::words;
        if (e < n) wl[r * R::row + w] = rec[k0 * R::words + e];
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    if (k >= cap) return;
    const int64_t* r = wl + lane * R::row;
    const T* t = (const T*)(r + 4);
    for (int d = 0; d < 3; d++) dst.pos[d][k] = __longlong_as_double(r[d]);
    dst.id[k] = r[3];
    for (int d = 0; d < 4; d++) dst.pup[d][k] = t[d];
    for (int d = 0; d < 2; d++) dst.Nn[d][k] = t[R::N + d];
    for (int d = 0; d < 2; d++) dst.Ll[d][k] = t[R::L + d];
#pragma unroll
    for (int c = 0; c < 2 * nh; c++) dst.f[(int64_t)c * cap + k] = t[R::F + c];
}

// Load: the scalars of a fresh state.
__global__ void k_load_scalars(double* scal, const double* time, int64_t* steps, unsigned long long* err,
                               unsigned long long* dtred)
{
    for (int i = threadIdx.x; i < DtRed::words; i += blockDim.x) dtred[i] = 0;
    if (threadIdx.x == 0) {
        scal[0] = time ? *time : 0.0; // all particles share it (main.cpp:101-110)
        scal[1] = 0.0;
        *steps = 0;
        *err = ~0ull;
    }
}

// Store: one wave per cell copies its cnt[c] particles from slots start[c]..
// to the caller's positions ustart[c].. (cell order, no gaps).
template <int NF, typename T>
__global__ void k_store(Arrays<T> src, PView P, int64_t* ids, const double* time, const int* __restrict__ start,
                        const int* __restrict__ cnt, const int* __restrict__ ustart, int64_t ncell, int64_t stride,
                        double nscale)
{
    using I = PIdx<NF>;
    constexpr int nh = NH<NF>;
    const double t = *time;
    const int64_t waves = (int64_t)gridDim.x * (blockDim.x / 64);
    for (int64_t c = blockIdx.x * (int64_t)(blockDim.x / 64) + threadIdx.x / 64; c < ncell; c += waves) {
        const int n = cnt[c];
        for (int i = threadIdx.x % 64; i < n; i += 64) {
            const int64_t k = (int64_t)start[c] + i, ip = (int64_t)ustart[c] + i;
            for (int d = 0; d < 3; d++) {
                P.pos[d][ip] = src.pos[d][k];
                P.r[I::x + d][ip] = src.pos[d][k];
            }
            P.r[I::time][ip] = t;
            for (int d = 0; d < 4; d++) P.r[I::pupx + d][ip] = double(src.pup[d][k]);
            P.r[I::N][ip] = double(src.Nn[0][k]) / nscale;
            P.r[I::Nbar][ip] = double(src.Nn[1][k]) / nscale;
            P.r[I::L][ip] = double(src.Ll[0][k]);
            P.r[I::Lbar][ip] = double(src.Ll[1][k]);
            for (int c2 = 0; c2 < nh; c2++) {
                P.r[I::f + c2][ip] = double(src.f[(int64_t)c2 * stride + k]);
                P.r[I::fbar + c2][ip] = double(src.f[(int64_t)(nh + c2) * stride + k]);
            }
            if (ids) ids[ip] = src.id[k];
        }
    }
}

// Load: red[0] = min pupt and red[1] = max(|N|, |Nbar|) as the bit patterns of
// non-negative doubles (those order like unsigned integers).
__global__ void k_load_ranges(const double* __restrict__ pupt, const double* __restrict__ N,
                              const double* __restrict__ Nbar, int64_t np, unsigned long long* red)
{
    double lo = INFINITY, hi = 0.0;
    for (int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; t < np; t += (int64_t)gridDim.x * blockDim.x) {
        lo = fmin(lo, pupt[t]);
        hi = fmax(hi, fmax(fabs(N[t]), fabs(Nbar[t])));
    }
    for (int off = 32; off > 0; off >>= 1) {
        lo = fmin(lo, __shfl_xor(lo, off));
        hi = fmax(hi, __shfl_xor(hi, off));
    }
    if ((threadIdx.x & 63) == 0) {
        atomicMin(&red[0], (unsigned long long)__double_as_longlong(lo));
        atomicMax(&red[1], (unsigned long long)__double_as_longlong(hi));
    }
}

__global__ void k_load_ranges_init(unsigned long long* red)
{
    if (threadIdx.x == 0) {
        red[0] = ~0ull >> 1;
        red[1] = 0;
    }
}

// Diagnostic: per cell N_01 = sum_p w N f01 and Nbar_01 (Re, Im), deposited
// with the particle shape factors, then the cell sums of |N_01| and |Nbar_01|.
// One wave per source cell takes its particles 64 at a time; for each of the
// 27 target cells the four weighted values are summed across the wave and
// lane 0 adds them to the target (108 atomics per chunk, not per particle).
__device__ __forceinline__ double wave_sum(double v)
{
    for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off);
    return v;
}

template <int NF, typename T>
__global__ __launch_bounds__(64) void k_diag_deposit(Arrays<T> A, const int* __restrict__ cell_start,
                                                     const int* __restrict__ cell_cnt, Geom g, int64_t np, double* out4)
{
    const int cell = blockIdx.x;
    const int lane = threadIdx.x;
    const int beg = cell_start[cell], end = beg + cell_cnt[cell];
    for (int base = beg; base < end; base += 64) {
        const int ip = base + lane;
        const bool act = ip < end;
        const int ipl = act ? ip : beg;
        int idx[3];
        double wd[3][3];
        for (int d = 0; d < 3; d++) shape3((A.pos[d][ipl] - g.plo[d]) * g.dxi[d], g.order[d], idx[d], wd[d]);
        const double N = act ? double(A.Nn[0][ipl]) : 0.0, Nb = act ? double(A.Nn[1][ipl]) : 0.0;
        const double v[4] = {N * (double)A.f[(int64_t)herm_re<NF>(0, 1) * np + ipl],
                             N * (double)A.f[(int64_t)herm_im<NF>(0, 1) * np + ipl],
                             Nb * (double)A.f[(int64_t)(NH<NF> + herm_re<NF>(0, 1)) * np + ipl],
                             Nb * (double)A.f[(int64_t)(NH<NF> + herm_im<NF>(0, 1)) * np + ipl]};
        // every particle of the cell has the same first stencil cell per dimension
        // (the stencil is centred on the particle's own cell)
        const int cx = cell % g.n[0], cy = (cell / g.n[0]) % g.n[1], cz = cell / (g.n[0] * g.n[1]);
        for (int t = 0; t < 27; t++) {
            const int ii = t % 3, jj = (t / 3) % 3, kk = t / 9;
            const double w = wd[0][ii] * wd[1][jj] * wd[2][kk];
            double s4[4];
            for (int q = 0; q < 4; q++) s4[q] = wave_sum(w * v[q]);
            if (lane == 0 && (s4[0] != 0.0 || s4[1] != 0.0 || s4[2] != 0.0 || s4[3] != 0.0)) {
                const int64_t c = ((int64_t)pmod(cz + kk - 1, g.n[2]) * g.n[1] + pmod(cy + jj - 1, g.n[1])) * g.n[0] +
                                  pmod(cx + ii - 1, g.n[0]);
                for (int q = 0; q < 4; q++) unsafeAtomicAdd(&out4[c * 4 + q], s4[q]);
            }
        }
        (void)idx;
    }
}

__global__ void k_diag_reduce(const double* __restrict__ g4, int64_t ncell, double* sums)
{
    double a = 0, b = 0;
    for (int64_t c = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; c < ncell; c += (int64_t)gridDim.x * blockDim.x) {
        a += sqrt(g4[4 * c] * g4[4 * c] + g4[4 * c + 1] * g4[4 * c + 1]);
        b += sqrt(g4[4 * c + 2] * g4[4 * c + 2] + g4[4 * c + 3] * g4[4 * c + 3]);
    }
    for (int off = 32; off > 0; off >>= 1) {
        a += __shfl_xor(a, off);
        b += __shfl_xor(b, off);
    }
    if ((threadIdx.x & 63) == 0) {
        unsafeAtomicAdd(&sums[0], a);
        unsafeAtomicAdd(&sums[1], b);
    }
}

} // namespace
} // namespace emu

using namespace emu;

// ---------------------------------------------------------------------------
// the state object
// ---------------------------------------------------------------------------
struct emu_state {
    emu_ctx* ctx;
    int64_t np;
    int precision; // EMU_PLAIN_FP64 / EMU_FP32_BULK
    int nf, nh, QG, naux;
    int64_t ncell;
    size_t tsize;
    // Slots: cell c's particles sit in slots cell_start[c] .. cell_start[c] +
    // cell_cnt[c] - 1, and every cell's run starts at a multiple of `align`
    // (1: back to back; 128 bytes of T otherwise, so that a wave's loads and
    // stores of a cell's particles cover whole cache lines that no other cell
    // shares).  cap slots (the stride of the per-particle arrays) hold any
    // layout: np + ncell (align - 1).
    int align = 1;
    int64_t cap = 1;
    bool split = false; // several waves per cell (k_stage's MODE 3)
    bool pairs = false; // two cells per wave (MODE 0)
    // persistent arrays, two copies for the sort
    void* block[2] = {nullptr, nullptr};
    // scratch
    void* Y = nullptr;
    void* acc = nullptr;
    int* rank = nullptr;
    int* counts = nullptr;         // ncell + 1: the scan's input (padded counts); a step's block sums
    int* cell_start = nullptr;     // ncell + 1
    int* new_start = nullptr;      // ncell + 1
    int* cell_cnt = nullptr;       // ncell + 1: particles per cell (current order)
    int* new_cnt = nullptr;        // ncell + 1: the same after this step's moves
    int* mcount = nullptr;         // [ncell][27] particles per (old cell, move)
    int* mbase = nullptr;          // [ncell][27] destination of the first of them
    unsigned char* mv = nullptr;   // move index per particle
    double* grid[3] = {nullptr, nullptr, nullptr}; // [0] the current deposit, [1] at its base, [2] free
    double* aux = nullptr;
    double* scal = nullptr;        // [0] time [1] dt
    int64_t* steps = nullptr;
    unsigned long long* red = nullptr;   // [2] error, [3] pupt min, [4] weight maximum, [4..5] amplitude sums
    unsigned long long* dtred = nullptr; // compute_dt's maxima (DtRed)
    void* cub_tmp = nullptr;
    size_t cub_bytes = 0;
    int cur = 0;      // which persistent copy is current
    bool evolved = false; // a step was taken since the last load
    double Vvac_max = 0.0;
    double m00 = 0.0;
    // The particle weights are held as N * nscale, nscale = 2^-k chosen at load
    // so that the largest weight is in [1, 2): FP32 cannot hold N = n dV for
    // large cells (1e54 for a (1e7 cm)^3 cell), and a power of two scales every
    // product and sum exactly.  The deposited fields carry the same factor,
    // which coef, the matter term and the dt estimate take back out.  The FP64
    // state keeps nscale = 1.
    double nscale = 1.0;
    // timing: an event pair around every profiled launch, by kernel class
    int profile = 0;
    struct Mark { int k; hipEvent_t a, b; };
    std::vector<Mark> marks;
    // on grids of more than kInlinePlanCells cells the sort plan runs on a stream
    // of its own, beside stages 2 and 3 (it needs stage 1's moves, and only
    // stage 4 reads it)
    hipStream_t side = nullptr;
    hipEvent_t ev_stage1 = nullptr, ev_plan = nullptr;
};

namespace {

// Up to here the sort plan's waves ride on the launches of stages 2 and 3 (SortPlan).
// Larger grids have the plan beside those stages on a second stream: there the two
// launches and the event pair are small change, and planning waves at the front of
// a stage keep its own from starting.  us per step, two launches (in line up to
// 32^3, beside from 40^3 on) / riding:
//   1 cell x 24 NF=2 FP64 30 / 28, 8^3 x 40 NF=2 FP32 60 / 46, 16^3 x 26 106 / 91,
//   24^3 x 40 271 / 254, 32^3 x 92 892 / 880, NF=3 FP64 32^3 x 92 2467 / 2451;
//   40^3 x 20 NF=2 FP32 958 / 966, 64^3 x 20 3608 / 3657, NF=3 FP32 8593 / 8737.
constexpr int64_t kInlinePlanCells = 32768;
// a planning wave takes a row of 64 cells, and more on grids of 2^17 cells and more,
// so that the sums which each wave adds up stay about a thousand
constexpr int64_t kPlanRowCells = 65536;

// Whether four waves share a cell (k_stage's MODE 3): where the cells hold more
// than one chunk of 64 particles each and are too few to fill the chip one (or,
// in FP32-bulk, half) a wave.  By LDS the chip holds about 1024 such workgroups
// in FP32-bulk and 768 in FP64 at once; up to twice that they still pay where a
// wave alone would walk 3 chunks or more.  us per step, one wave / four waves per
// cell, NF = 3:
//   FP32-bulk  4^3 cells  x 92: 126 / 70    x 378: 367 / 103
//              8^3        x 92: 141 / 94    x 378: 395 / 159
//              1024 (1-D) x 92:  80 / 70    x 378: 196 / 143
//              12^3       x 92: 201 / 216   x 200: 352 / 245
//              16^3       x 92: 281 / 387   x 378: 819 / 822
//   FP64       8^3        x 92: 132 / 113   x 378: 329 / 211
//              1024 (1-D) x 92:  97 / 110   x 200: 164 / 140
//              12^3       x 92: 204 / 309   x 378: 563 / 634
// and NF = 2, on the same side at each of these, which differ by less where they cross:
//   FP32-bulk  4^3        x 66:  56 / 44    x 378: 131 / 62
//              8^3        x 66:  59 / 50    x 378: 144 / 86
//              10^3       x 66:  70 / 60    x 378: 182 / 117
//              12^3       x 92:  82 / 108   x 200: 136 / 124
//   FP64       8^3        x 66:  61 / 55    x 378: 162 / 105
//              1024 (1-D) x 92:  59 / 55    x 200: 104 / 76
//              10^3       x 92:  84 / 87    x 200: 140 / 108
//              12^3       x 92:  96 / 133   x 378: 264 / 262
bool split_cells(int64_t np, int64_t ncell, int precision)
{
    const int64_t at_once = precision == EMU_FP32_BULK ? 1024 : 768;
    return (ncell <= at_once && np > 64 * ncell) || (ncell <= 2 * at_once && np > 160 * ncell);
}

// Whether a wave takes two cells (k_stage's MODE 0, where it is there): fewer
// chunks are partly filled and neighbours' boxes overlap, but half as many waves run
// at once.  From 3072 cells on, one per wave fills the chip (three waves per SIMD),
// and in FP32-bulk the pairs win; FP64's NF = 2 has registers for fewer waves of
// pairs, so there they pay only where two cells fill one chunk.  us per step, one
// cell / two cells per wave, at 12, 26, 64 and 92 particles a cell:
//   FP32-bulk NF = 2   8^3  55/57 57/62 63/78 -       12^3  71/72 78/78 87/100 103/124
//                     16^3  96/95 101/105 114/125 145/155   24^3 245/235 265/253 317/304 419/409
//             NF = 3   8^3  70/74 76/82 87/112 -      12^3 112/113 120/125 137/157 165/197
//                     16^3 192/182 207/195 237/228 293/275  24^3 524/511 557/546 657/632 803/785
//   FP64      NF = 2  12^3  77/79 85/89 98/122 122/159  16^3 120/106 130/115 155/155 207/194
//                     24^3 291/277 314/311 405/448 569/647
// A domain of one column has no pairs to take: a wave's second cell would be empty and
// its box 36 rows instead of 27.  Narrow odd domains, whose last column goes by itself,
// gain less, but lose only where the waves of pairs just miss the last full round:
//   FP64      NF = 2   at 12, 26, 31   1x64x64 152/166 165/176 164/182    3x33x33 93/90 103/103 104/105
//                     3x64x64 242/239 267/262 266/264    5x32x32 123/120 133/140 135/143
//   FP32-bulk NF = 2   at 26, 92   1x64x64 141/142 195/194    3x33x33 88/87 129/148    3x64x64 227/216 363/362
//                     5x32x32 109/109 171/167
//             NF = 3   1x64x64 213/222 310/322    1x160x160 1115/1148 1596/1652    3x33x33 164/166 252/261
//                     3x64x64 476/470 711/701    5x32x32 216/217 319/316
constexpr int64_t kPairCells = 3072;
bool pair_cells(const Geom& g, int64_t np, int64_t ncell, int precision)
{
    return g.n[0] > 1 && ncell > kPairCells && (precision == EMU_FP32_BULK || np <= 32 * ncell);
}

template <typename T> Arrays<T> arrays_of(emu_state* st, int copy)
{
    Arrays<T> A;
    char* b = (char*)st->block[copy];
    const int64_t np = st->cap;
    for (int d = 0; d < 3; d++) { A.pos[d] = (double*)b; b += np * sizeof(double); }
    A.id = (int64_t*)b;
    b += np * sizeof(int64_t);
    for (int d = 0; d < 4; d++) { A.pup[d] = (T*)b; b += np * sizeof(T); }
    for (int d = 0; d < 2; d++) { A.Nn[d] = (T*)b; b += np * sizeof(T); }
    for (int d = 0; d < 2; d++) { A.Ll[d] = (T*)b; b += np * sizeof(T); }
    A.f = (T*)b;
    return A;
}

size_t persistent_bytes(int64_t np, int nh, size_t tsize)
{
    return (size_t)np * (3 * sizeof(double) + sizeof(int64_t) + (8 + 2 * nh) * tsize);
}

unsigned grid_blocks(int64_t n, int bs = 256)
{
    return (unsigned)std::min<int64_t>(65535 * 16, std::max<int64_t>(1, (n + bs - 1) / bs));
}

int ensure_cub(emu_state* st, size_t need)
{
    if (need > st->cub_bytes) {
        if (st->cub_tmp) (void)hipFree(st->cub_tmp);
        st->cub_tmp = nullptr;
        st->cub_bytes = 0;
        if (hipMalloc(&st->cub_tmp, need) != hipSuccess) return EMU_ERR_NOMEM;
        st->cub_bytes = need;
    }
    return EMU_OK;
}

// out = exclusive scan of in (ncell + 1 entries, in[ncell] = 0)
int scan_counts(emu_state* st, const int* in, int* out)
{
    hipStream_t s = st->ctx->stream;
    size_t need = 0;
    (void)hipcub::DeviceScan::ExclusiveSum(nullptr, need, in, out, (int)(st->ncell + 1), s);
    if (ensure_cub(st, need)) return set_error(st->ctx, EMU_ERR_NOMEM, "scan scratch");
    EMU_HIP(st->ctx, hipcub::DeviceScan::ExclusiveSum(st->cub_tmp, st->cub_bytes, in, out, (int)(st->ncell + 1), s));
    return EMU_OK;
}


SortPlan sort_plan(const emu_state* st)
{
    SortPlan p{st->mcount, st->new_start, st->new_cnt, st->counts, st->mbase, st->align, 1, 0};
    p.per = (int)std::max<int64_t>(1, st->ncell / kPlanRowCells);
    p.waves = (int)(st->ncell / (64 * p.per) + 1); // cell ncell too
    return p;
}

template <int NF, typename T, int WX, int WY, int WZ, int S, int AUX, int MODE>
void launch_stage_mode(emu_state* st, StageArgs<T>& a)
{
    constexpr int WPB = stage_waves_per_block<MODE, AUX>(); // waves per workgroup
    using PT = StagePatch<T, WX, WY, WZ, WPB, MODE>;
    const Geom& g = st->ctx->g;
    const int64_t npatch = (int64_t)((g.n[0] + PT::PX - 1) / PT::PX) * ((g.n[1] + PT::PY - 1) / PT::PY) *
                           ((g.n[2] + PT::PZ - 1) / PT::PZ);
    const int64_t nblk = MODE >= 2 ? npatch : (npatch + WPB - 1) / WPB;
    a.blocks_per_xcd = (int)((nblk + 7) / 8);
    const size_t lds = (size_t)stage_lds_doubles_per_block<NF, T, WX, WY, WZ, WPB, S, AUX, MODE>() * sizeof(double);
    a.plan_blocks = S == 2 || S == 3 ? ((a.plan.waves + WPB - 1) / WPB + 7) / 8 * 8 : 0;
    hipLaunchKernelGGL((k_stage<NF, T, WX, WY, WZ, WPB, S, AUX, MODE>), dim3((unsigned)(a.plan_blocks + 8 * a.blocks_per_xcd)),
                       dim3(64 * WPB), lds, st->ctx->stream, a);
}

template <int NF, typename T, int WX, int WY, int WZ, int S, int AUX>
void launch_stage_k(emu_state* st, StageArgs<T>& a)
{
    if (st->split) {
        launch_stage_mode<NF, T, WX, WY, WZ, S, AUX, 3>(st, a);
    } else if constexpr (stage_merges<T, S, AUX>()) {
        launch_stage_mode<NF, T, WX, WY, WZ, S, AUX, 2>(st, a);
    } else {
        if constexpr (stage_has_pairs<NF, T, WX>()) {
            if (st->pairs) {
                launch_stage_mode<NF, T, WX, WY, WZ, S, AUX, 0>(st, a);
                return;
            }
        }
        launch_stage_mode<NF, T, WX, WY, WZ, S, AUX, 1>(st, a);
    }
}

template <int NF, typename T, int WX, int WY, int WZ>
void launch_stage_t(emu_state* st, StageArgs<T>& a)
{
    // the compute_dt auxiliaries ride on the deposit that compute_dt reads
    const int aux = a.stage == 3 || a.stage == 0 ? a.want_aux : 0;
    switch (a.stage) {
    case 0:
        if (aux == 2) launch_stage_k<NF, T, WX, WY, WZ, 0, 2>(st, a);
        else if (aux == 1) launch_stage_k<NF, T, WX, WY, WZ, 0, 1>(st, a);
        else launch_stage_k<NF, T, WX, WY, WZ, 0, 0>(st, a);
        break;
    case 1: launch_stage_k<NF, T, WX, WY, WZ, 1, 0>(st, a); break;
    case 2: launch_stage_k<NF, T, WX, WY, WZ, 2, 0>(st, a); break;
    case 3:
        if (aux == 2) launch_stage_k<NF, T, WX, WY, WZ, 3, 2>(st, a);
        else if (aux == 1) launch_stage_k<NF, T, WX, WY, WZ, 3, 1>(st, a);
        else launch_stage_k<NF, T, WX, WY, WZ, 3, 0>(st, a);
        break;
    default: launch_stage_k<NF, T, WX, WY, WZ, 4, 0>(st, a); break;
    }
}

// Stencil shapes: 3 cells per dimension with shape order 1 or 2, 1 cell with
// order 0 or in a 1-cell dimension.  (3,3,3), (1,1,3) and (1,1,1) have their
// own kernels; other shapes run the (3,3,3) kernel, whose extra entries carry
// zero weight.
template <int NF, typename T> void launch_stage_shape(emu_state* st, StageArgs<T>& a)
{
    const int* o = st->ctx->g.order;
    const int wx = o[0] > 0 ? 3 : 1, wy = o[1] > 0 ? 3 : 1, wz = o[2] > 0 ? 3 : 1;
    if (wx == 1 && wy == 1 && wz == 1) launch_stage_t<NF, T, 1, 1, 1>(st, a);
    else if (wx == 1 && wy == 1) launch_stage_t<NF, T, 1, 1, 3>(st, a);
    else launch_stage_t<NF, T, 3, 3, 3>(st, a);
}

DtParams dt_params(const emu_state* st, double fixed_dt)
{
    const emu_ctx* ctx = st->ctx;
    const emu_params& p = ctx->p;
    DtParams dp;
    dp.dt_translation = p.cfl_factor > 0.0
                            ? std::min(std::min(ctx->g.dx[0], ctx->g.dx[1]), ctx->g.dx[2]) / phys::c * p.cfl_factor
                            : 0.0;
    dp.flavor_cfl = p.flavor_cfl_factor;
    dp.max_adaptive_speedup = p.max_adaptive_speedup;
    dp.Vvac_max = st->Vvac_max;
    dp.fixed_dt = fixed_dt;
    dp.use_flavor = p.flavor_cfl_factor > 0.0;
    dp.vst_scale = 2.0 * st->nf * M_SQRT2 * phys::GF / (ctx->g.cell_volume * st->nscale);
    return dp;
}

// What a launch does besides its stage.
struct StageExtra {
    bool want_aux = false;     // deposit the compute_dt auxiliaries
    double* gclear = nullptr;  // grid to set to its base
    bool clear_aux = false;
    bool want_dt = false;      // stage 4: the conservative flavour bound
    bool step_end = false;     // stage 0: the next dt and the step's end
    double fixed_dt = 0.0;
};

template <typename T>
StageArgs<T> stage_args(emu_state* st, int stage, const double* gin, double* gout, const StageExtra& x)
{
    StageArgs<T> a;
    a.cur = arrays_of<T>(st, st->cur);
    a.dst = arrays_of<T>(st, 1 - st->cur);
    a.Y = (T*)st->Y;
    a.acc = (T*)st->acc;
    a.rank = st->rank;
    a.mv = st->mv;
    a.mcount = st->mcount;
    a.mbase = st->mbase;
    a.cell_start = st->cell_start;
    a.cell_cnt = st->cell_cnt;
    a.gin = gin;
    a.gout = gout;
    a.aux = st->aux;
    a.gclear = x.gclear;
    a.clear_aux = x.clear_aux;
    a.m00 = st->m00 * st->nscale;
    a.want_dt = x.want_dt;
    a.red = st->dtred;
    a.step_end = x.step_end;
    a.dtp = dt_params(st, x.fixed_dt);
    a.scal = st->scal;
    a.steps = st->steps;
    a.dt = st->scal + 1;
    a.err = st->red + 2;
    a.np = st->cap;
    a.ncell = st->ncell;
    a.stage = stage;
    // the diagonal sums for the conservative flavour bound; Im(Fbar) as well
    // where the adaptive bound is used (max_adaptive_speedup > 1).  FP64 deposits
    // the full set either way: measured at 64^3 x 92, its auxiliary stage ran
    // 2% slower with the diagonal sums alone (FP32-bulk's 1% faster).
    a.want_aux = x.want_aux ? (st->ctx->p.max_adaptive_speedup > 1 || sizeof(T) == 8 ? 2 : 1) : 0;
    a.blocks_per_xcd = 0;
    a.plan = st->ncell <= kInlinePlanCells ? sort_plan(st) : SortPlan{};
    a.g = st->ctx->g;
    const emu_ctx* ctx = st->ctx;
    for (int c = 0; c < 9; c++) a.vac[c] = c < st->nh ? ctx->M2[c] * phys::c4 / 2.0 / phys::hbar : 0.0;
    a.coef = M_SQRT2 * phys::GF * ctx->g.inv_cell_volume / phys::hbar / st->nscale;
    a.maxError = ctx->p.maxError;
    return a;
}

void launch_stage(emu_state* st, int stage, const double* gin, double* gout, const StageExtra& x)
{
    if (st->precision == EMU_FP32_BULK) {
        auto a = stage_args<float>(st, stage, gin, gout, x);
        if (st->nf == 2) launch_stage_shape<2, float>(st, a);
        else launch_stage_shape<3, float>(st, a);
    } else {
        auto a = stage_args<double>(st, stage, gin, gout, x);
        if (st->nf == 2) launch_stage_shape<2, double>(st, a);
        else launch_stage_shape<3, double>(st, a);
    }
}

void fill_grid(emu_state* st, double* g, bool with_aux)
{
    hipLaunchKernelGGL(k_fill_grid, dim3(grid_blocks(st->ncell * st->QG)), dim3(256), 0, st->ctx->stream, g,
                       st->ncell, st->QG, st->m00 * st->nscale, with_aux ? st->aux : nullptr, st->naux);
}

// compute_dt's maxima over the cells of grid g and the auxiliaries, both bounds
void dt_reduce(emu_state* st, const double* g)
{
    emu_ctx* ctx = st->ctx;
    const int adaptive = ctx->p.max_adaptive_speedup > 1 ? 1 : 0;
    const double vol = ctx->g.cell_volume * st->nscale, m00 = st->m00 * st->nscale;
    const dim3 grid(grid_blocks(st->ncell)), block(256);
    if (st->nf == 2) hipLaunchKernelGGL(k_dt_reduce<2>, grid, block, 0, ctx->stream, g, st->aux, st->ncell, vol, m00, adaptive, st->dtred);
    else hipLaunchKernelGGL(k_dt_reduce<3>, grid, block, 0, ctx->stream, g, st->aux, st->ncell, vol, m00, adaptive, st->dtred);
}

// the starting dt (main.cpp:206) from grid g, into scal[1]
int starting_dt(emu_state* st, const double* g)
{
    emu_ctx* ctx = st->ctx;
    if (ctx->p.flavor_cfl_factor > 0.0) dt_reduce(st, g);
    hipLaunchKernelGGL(k_dt_finalize, dim3(1), dim3(64), 0, ctx->stream, st->dtred, dt_params(st, 0.0), st->scal + 1,
                       st->red + 2);
    EMU_LAUNCH_CHECK(ctx, "compute_dt");
    return EMU_OK;
}

// Kernel classes: 0 stage kernels, 1 grid fills, 2 sort, 3 dt reduction.
void ev_record(emu_state* st, int k, bool start, hipStream_t stream = nullptr)
{
    if (!st->profile) return;
    hipEvent_t e;
    (void)hipEventCreate(&e);
    (void)hipEventRecord(e, stream ? stream : st->ctx->stream);
    if (start) st->marks.push_back({k, e, nullptr});
    else st->marks.back().b = e;
}

} // namespace

extern "C" int emu_state_destroy(emu_state* st);

extern "C" int emu_state_create(emu_ctx* ctx, int64_t np, int precision, emu_state** out)
{
    const int layout = precision & ~0xff;
    precision &= 0xff;
    if (!ctx || !out || np < 0 || (precision != EMU_PLAIN_FP64 && precision != EMU_FP32_BULK) ||
        (layout != 0 && layout != EMU_STATE_SLOTS_PACKED && layout != EMU_STATE_SLOTS_ALIGNED))
        return EMU_ERR_ARG;
    if (np > (int64_t)INT32_MAX) return set_error(ctx, EMU_ERR_UNSUPPORTED, "more than 2^31-1 particles per state");
    *out = nullptr;
    auto* st = new emu_state();
    st->ctx = ctx;
    st->np = np;
    st->precision = precision;
    st->nf = ctx->p.nf;
    st->nh = st->nf * st->nf;
    st->QG = 4 * st->nh;
    st->naux = st->nf + 3 * (st->nf * (st->nf - 1) / 2);
    st->ncell = (int64_t)ctx->g.n[0] * ctx->g.n[1] * ctx->g.n[2];
    st->tsize = precision == EMU_FP32_BULK ? sizeof(float) : sizeof(double);
    st->m00 = ctx->p.rho * ctx->p.Ye / phys::Mp / ctx->g.inv_cell_volume;
    // slot alignment: 128 bytes of T; by default only where the cells hold on
    // average two alignments' worth of particles (padding <= np / 2)
    const int a128 = (int)(128 / st->tsize);
    bool aligned = layout == EMU_STATE_SLOTS_ALIGNED || (layout == 0 && np >= 2 * a128 * st->ncell);
    if (np == 0 || np + st->ncell * (a128 - 1) > (int64_t)INT32_MAX) aligned = false;
    st->align = aligned ? a128 : 1;
    st->cap = std::max<int64_t>(np + st->ncell * (st->align - 1), 1);
    st->split = split_cells(np, st->ncell, precision);
    st->pairs = pair_cells(ctx->g, np, st->ncell, precision);
    const int64_t npa = st->cap;
    const size_t pb = persistent_bytes(npa, st->nh, st->tsize);
    bool ok = hipMalloc(&st->block[0], pb) == hipSuccess && hipMalloc(&st->block[1], pb) == hipSuccess &&
              hipMalloc(&st->Y, (size_t)npa * 2 * st->nh * st->tsize) == hipSuccess &&
              hipMalloc(&st->acc, (size_t)npa * 2 * st->nh * st->tsize) == hipSuccess &&
              hipMalloc(&st->rank, (size_t)npa * sizeof(int)) == hipSuccess &&
              hipMalloc(&st->counts, (size_t)(st->ncell + 1) * sizeof(int)) == hipSuccess &&
              hipMalloc(&st->cell_start, (size_t)(st->ncell + 1) * sizeof(int)) == hipSuccess &&
              hipMalloc(&st->new_start, (size_t)(st->ncell + 1) * sizeof(int)) == hipSuccess &&
              hipMalloc(&st->cell_cnt, (size_t)(st->ncell + 1) * sizeof(int)) == hipSuccess &&
              hipMalloc(&st->new_cnt, (size_t)(st->ncell + 1) * sizeof(int)) == hipSuccess &&
              hipMalloc(&st->mcount, (size_t)st->ncell * 27 * sizeof(int)) == hipSuccess &&
              hipMalloc(&st->mbase, (size_t)st->ncell * 27 * sizeof(int)) == hipSuccess &&
              hipMalloc(&st->mv, (size_t)npa) == hipSuccess &&
              hipMalloc(&st->grid[0], (size_t)st->ncell * st->QG * sizeof(double)) == hipSuccess &&
              hipMalloc(&st->grid[1], (size_t)st->ncell * st->QG * sizeof(double)) == hipSuccess &&
              hipMalloc(&st->grid[2], (size_t)st->ncell * st->QG * sizeof(double)) == hipSuccess &&
              hipMalloc(&st->aux, (size_t)st->ncell * st->naux * sizeof(double)) == hipSuccess &&
              hipMalloc(&st->scal, 4 * sizeof(double)) == hipSuccess &&
              hipMalloc(&st->steps, sizeof(int64_t)) == hipSuccess &&
              hipMalloc(&st->red, 8 * sizeof(unsigned long long)) == hipSuccess &&
              hipMalloc(&st->dtred, DtRed::words * sizeof(unsigned long long)) == hipSuccess;
    // default priority, and no implicit synchronisation with the legacy stream
    ok = ok && hipStreamCreateWithFlags(&st->side, hipStreamNonBlocking) == hipSuccess &&
         hipEventCreateWithFlags(&st->ev_stage1, hipEventDisableTiming) == hipSuccess &&
         hipEventCreateWithFlags(&st->ev_plan, hipEventDisableTiming) == hipSuccess;
    if (!ok) {
        emu_state_destroy(st);
        return set_error(ctx, EMU_ERR_NOMEM, "state allocation failed");
    }
    *out = st;
    return EMU_OK;
}

extern "C" int emu_state_destroy(emu_state* st)
{
    if (!st) return EMU_OK;
    void* ptrs[] = {st->block[0], st->block[1],   st->Y,         st->acc,      st->rank,    st->counts, st->cell_start,
                    st->new_start, st->cell_cnt,  st->new_cnt,   st->mcount,   st->mbase,   st->mv,     st->grid[0],
                    st->grid[1],  st->grid[2],    st->aux,       st->scal,     st->steps,   st->red,    st->cub_tmp,
                    st->dtred};
    for (void* p : ptrs)
        if (p) (void)hipFree(p);
    for (auto& m : st->marks) {
        (void)hipEventDestroy(m.a);
        if (m.b) (void)hipEventDestroy(m.b);
    }
    if (st->side) {
        (void)hipStreamSynchronize(st->side);
        (void)hipStreamDestroy(st->side);
    }
    for (hipEvent_t ev : {st->ev_stage1, st->ev_plan})
        if (ev) (void)hipEventDestroy(ev);
    delete st;
    return EMU_OK;
}

template <typename T> static int load_t(emu_state* st, const PView& P, const int64_t* ids)
{
    emu_ctx* ctx = st->ctx;
    hipStream_t s = ctx->stream;
    const int64_t np = st->np;
    // scratch: the stage state's and the accumulator's arrays, free until the
    // first step (at least 32 bytes per slot each), and the other copy's block
    int* cells = (int*)st->Y;
    int* keys = cells + st->cap;
    int* iota = keys + st->cap;
    int* order = (int*)st->acc;
    int* slot = order + st->cap;
    hipLaunchKernelGGL(k_fill_int, dim3(grid_blocks(st->ncell + 1)), dim3(256), 0, s, st->counts, st->ncell + 1, 0);
    if (np > 0)
        hipLaunchKernelGGL(k_bin_input, dim3(grid_blocks(np)), dim3(256), 0, s, P, ctx->g, cells, st->counts);
    // the cells' first positions back to back (new_start, scratch here), then
    // their padded slot runs (cell_start)
    int e = scan_counts(st, st->counts, st->new_start);
    if (e) return e;
    hipLaunchKernelGGL(k_pad_counts, dim3(grid_blocks(st->ncell + 1)), dim3(256), 0, s, st->counts, st->cell_cnt,
                       st->ncell, st->align);
    e = scan_counts(st, st->counts, st->cell_start);
    if (e) return e;
    if (np == 0) return EMU_OK;
    // stable radix sort of (cell, input index)
    hipLaunchKernelGGL(k_iota, dim3(grid_blocks(np)), dim3(256), 0, s, iota, np);
    int end_bit = 1;
    while ((1ll << end_bit) < st->ncell) end_bit++;
    size_t need = 0;
    (void)hipcub::DeviceRadixSort::SortPairs(nullptr, need, cells, keys, iota, order, (int)np, 0, end_bit, s);
    if (ensure_cub(st, need)) return set_error(ctx, EMU_ERR_NOMEM, "radix sort scratch");
    if (hipcub::DeviceRadixSort::SortPairs(st->cub_tmp, st->cub_bytes, cells, keys, iota, order, (int)np, 0, end_bit,
                                           s) != hipSuccess)
        return set_error(ctx, EMU_ERR_HIP, "radix sort");
    hipLaunchKernelGGL(k_load_slots, dim3(grid_blocks(np)), dim3(256), 0, s, order, keys, st->cell_start, st->new_start,
                       np, slot);
    const Arrays<T> A = arrays_of<T>(st, st->cur);
    int64_t* rec = (int64_t*)st->block[1 - st->cur];
    const unsigned block = 64 * LoadRec<2, T>::waves;
    const dim3 gp((unsigned)((np + block - 1) / block)), gu((unsigned)((st->cap + block - 1) / block));
    if (st->nf == 2) {
        hipLaunchKernelGGL((k_load_pack<2, T>), gp, dim3(block), 0, s, P, ids, slot, rec, st->nscale);
        hipLaunchKernelGGL((k_load_unpack<2, T>), gu, dim3(block), 0, s, rec, A, st->cap);
    } else {
        hipLaunchKernelGGL((k_load_pack<3, T>), gp, dim3(block), 0, s, P, ids, slot, rec, st->nscale);
        hipLaunchKernelGGL((k_load_unpack<3, T>), gu, dim3(block), 0, s, rec, A, st->cap);
    }
    EMU_LAUNCH_CHECK(ctx, "state_load");
    return EMU_OK;
}

extern "C" int emu_state_load(emu_state* st, const emu_particles* parts, const int64_t* ids)
{
    if (!st || !parts || parts->np != st->np) return EMU_ERR_ARG;
    emu_ctx* ctx = st->ctx;
    hipStream_t s = ctx->stream;
    PView P;
    P.np = parts->np;
    const int na = 12 + 2 * st->nh;
    for (int d = 0; d < 3; d++) P.pos[d] = parts->pos[d];
    for (int k = 0; k < EMU_MAX_ATTRIBS; k++) P.r[k] = k < na ? parts->rdata[k] : nullptr;
    // the least energy and the largest weight
    hipLaunchKernelGGL(k_load_ranges_init, dim3(1), dim3(64), 0, s, st->red + 3);
    if (st->np > 0)
        hipLaunchKernelGGL(k_load_ranges, dim3(std::min(grid_blocks(st->np), 1024u)), dim3(256), 0, s,
                           P.r[PIdx<2>::pupt], P.r[PIdx<2>::N], P.r[st->nf == 2 ? (int)PIdx<2>::Nbar : (int)PIdx<3>::Nbar],
                           st->np, st->red + 3);
    double range[2];
    EMU_HIP(ctx, hipMemcpyAsync(range, st->red + 3, sizeof range, hipMemcpyDeviceToHost, s));
    EMU_HIP(ctx, hipStreamSynchronize(s));
    const double pupt_min = range[0], nmax = range[1];
    st->nscale = 1.0;
    if (st->precision == EMU_FP32_BULK && nmax > 0.0 && std::isfinite(nmax)) st->nscale = std::ldexp(1.0, -std::ilogb(nmax));
    int e = st->precision == EMU_FP32_BULK ? load_t<float>(st, P, ids) : load_t<double>(st, P, ids);
    if (e) return e;
    // Vvac_max from the minimum energy (FlavoredNeutrinoContainerInit.cpp:657-660)
    double d[9] = {0};
    if (st->nf == 2) {
        for (int i = 0; i < 2; i++) d[herm_re<2>(i, i)] = ctx->p.mass[i] * ctx->p.mass[i];
        st->Vvac_max = std::sqrt(su_mag2<2, double>(d)) * phys::c4 / pupt_min;
    } else {
        for (int i = 0; i < 3; i++) d[herm_re<3>(i, i)] = ctx->p.mass[i] * ctx->p.mass[i];
        st->Vvac_max = std::sqrt(su_mag2<3, double>(d)) * phys::c4 / pupt_min;
    }
    hipLaunchKernelGGL(k_load_scalars, dim3(1), dim3(256), 0, s, st->scal, st->np > 0 ? P.r[PIdx<2>::time] : nullptr,
                       st->steps, st->red + 2, st->dtred);
    // initial deposit (main.cpp:118) and starting dt (main.cpp:206)
    fill_grid(st, st->grid[0], true);
    fill_grid(st, st->grid[1], false);
    StageExtra x;
    x.want_aux = true;
    launch_stage(st, 0, nullptr, st->grid[0], x);
    e = starting_dt(st, st->grid[0]);
    if (e) return e;
    EMU_HIP(ctx, hipStreamSynchronize(s));
    st->evolved = false;
    return EMU_OK;
}

extern "C" int emu_state_set_vvac_max(emu_state* st, double vvac_max)
{
    if (!st || !(vvac_max >= 0.0) || !std::isfinite(vvac_max)) return EMU_ERR_ARG;
    emu_ctx* ctx = st->ctx;
    if (st->evolved) return set_error(ctx, EMU_ERR_ARG, "Vvac_max is set between emu_state_load and the first step");
    st->Vvac_max = vvac_max;
    // grid[0] (and aux) still hold the load's deposit: the starting dt again
    // (main.cpp:206) with the new value
    const int e = starting_dt(st, st->grid[0]);
    if (e) return e;
    EMU_HIP(ctx, hipStreamSynchronize(ctx->stream));
    return EMU_OK;
}

extern "C" int emu_state_store(emu_state* st, emu_particles* parts, int64_t* ids)
{
    if (!st || !parts || parts->np != st->np) return EMU_ERR_ARG;
    emu_ctx* ctx = st->ctx;
    PView P;
    P.np = parts->np;
    const int na = 12 + 2 * st->nh;
    for (int d = 0; d < 3; d++) P.pos[d] = parts->pos[d];
    for (int k = 0; k < EMU_MAX_ATTRIBS; k++) P.r[k] = k < na ? parts->rdata[k] : nullptr;
    if (st->np > 0) {
        // the caller's positions of each cell's first particle (new_start is
        // scratch between steps)
        int e = scan_counts(st, st->cell_cnt, st->new_start);
        if (e) return e;
        const dim3 grid(grid_blocks(st->ncell, 4)), block(256); // one wave per cell
        const int* cs = st->cell_start;
        const int* cn = st->cell_cnt;
        const int* us = st->new_start;
        if (st->precision == EMU_FP32_BULK) {
            Arrays<float> A = arrays_of<float>(st, st->cur);
            if (st->nf == 2)
                hipLaunchKernelGGL((k_store<2, float>), grid, block, 0, ctx->stream, A, P, ids, st->scal, cs, cn, us,
                                   st->ncell, st->cap, st->nscale);
            else
                hipLaunchKernelGGL((k_store<3, float>), grid, block, 0, ctx->stream, A, P, ids, st->scal, cs, cn, us,
                                   st->ncell, st->cap, st->nscale);
        } else {
            Arrays<double> A = arrays_of<double>(st, st->cur);
            if (st->nf == 2)
                hipLaunchKernelGGL((k_store<2, double>), grid, block, 0, ctx->stream, A, P, ids, st->scal, cs, cn, us,
                                   st->ncell, st->cap, st->nscale);
            else
                hipLaunchKernelGGL((k_store<3, double>), grid, block, 0, ctx->stream, A, P, ids, st->scal, cs, cn, us,
                                   st->ncell, st->cap, st->nscale);
        }
    }
    EMU_LAUNCH_CHECK(ctx, "state_store");
    EMU_HIP(ctx, hipStreamSynchronize(ctx->stream));
    return EMU_OK;
}

extern "C" int emu_state_evolve(emu_state* st, int nsteps, double fixed_dt)
{
    if (!st || nsteps < 0) return EMU_ERR_ARG;
    emu_ctx* ctx = st->ctx;
    hipStream_t s = ctx->stream;
    const Geom& g = ctx->g;
    // the deterministic sort assumes moves of at most one cell per step
    if (ctx->p.cfl_factor <= 0.0 || ctx->p.cfl_factor >= 1.0)
        if (fixed_dt <= 0 || fixed_dt * phys::c >= std::min(std::min(g.dx[0], g.dx[1]), g.dx[2]))
            return set_error(ctx, EMU_ERR_MOVE, "fused step needs c*dt < dx (0 < cfl_factor < 1)");
    if (fixed_dt > 0) EMU_HIP(ctx, hipMemcpyAsync(st->scal + 1, &fixed_dt, sizeof(double), hipMemcpyHostToDevice, s));
    if (nsteps > 0) st->evolved = true;
    const bool flavor_dt = ctx->p.flavor_cfl_factor > 0.0 && fixed_dt <= 0;
    const bool adaptive = flavor_dt && ctx->p.max_adaptive_speedup > 1;
    const bool beside = st->ncell > kInlinePlanCells;
    for (int step = 0; step < nsteps; step++) {
        // the grids' turns: A holds the deposit of y_n, B is at its base, C free
        double *A = st->grid[0], *B = st->grid[1], *C = st->grid[2];
        auto stage = [&](int k, const double* gin, double* gout, const StageExtra& x) {
            ev_record(st, 0, true);
            launch_stage(st, k, gin, gout, x);
            ev_record(st, 0, false);
        };
        StageExtra x1, x2, x3, x4, x0;
        x1.gclear = C;
        stage(1, A, B, x1); // also the moves over the step
        // the stable counting-sort plan by the new cell
        if (beside) {
            const SortPlan plan = sort_plan(st);
            const dim3 grid((unsigned)((plan.waves + 3) / 4)), block(256);
            EMU_HIP(ctx, hipEventRecord(st->ev_stage1, s));
            EMU_HIP(ctx, hipStreamWaitEvent(st->side, st->ev_stage1, 0));
            ev_record(st, 2, true, st->side);
            hipLaunchKernelGGL(k_plan<2>, grid, block, 0, st->side, plan, g, (int)st->ncell);
            hipLaunchKernelGGL(k_plan<3>, grid, block, 0, st->side, plan, g, (int)st->ncell);
            ev_record(st, 2, false, st->side);
            EMU_HIP(ctx, hipEventRecord(st->ev_plan, st->side));
        }
        x2.gclear = A;
        x2.clear_aux = flavor_dt;
        stage(2, B, C, x2);
        x3.gclear = B;
        x3.want_aux = flavor_dt;
        stage(3, C, A, x3);
        if (adaptive) {
            ev_record(st, 3, true);
            dt_reduce(st, A);
            ev_record(st, 3, false);
        }
        if (beside) EMU_HIP(ctx, hipStreamWaitEvent(s, st->ev_plan, 0));
        x4.gclear = C;
        x4.want_dt = flavor_dt && !adaptive;
        stage(4, A, nullptr, x4); // writes y_{n+1} into the other copy, new order
        st->cur = 1 - st->cur;
        std::swap(st->cell_start, st->new_start);
        std::swap(st->cell_cnt, st->new_cnt);
        // deposit of y_{n+1} for the next step's stage 1, and the next dt
        x0.step_end = true;
        x0.fixed_dt = fixed_dt;
        stage(0, nullptr, B, x0);
        st->grid[0] = B;
        st->grid[1] = C;
        st->grid[2] = A;
        EMU_LAUNCH_CHECK(ctx, "state_evolve");
    }
    return EMU_OK;
}

extern "C" int emu_state_info(emu_state* st, double* time, double* dt, int64_t* steps, int64_t* bad_index)
{
    if (!st) return EMU_ERR_ARG;
    emu_ctx* ctx = st->ctx;
    double sc[4];
    int64_t n = 0;
    unsigned long long e = 0;
    EMU_HIP(ctx, hipMemcpyAsync(sc, st->scal, sizeof sc, hipMemcpyDeviceToHost, ctx->stream));
    EMU_HIP(ctx, hipMemcpyAsync(&n, st->steps, sizeof n, hipMemcpyDeviceToHost, ctx->stream));
    EMU_HIP(ctx, hipMemcpyAsync(&e, st->red + 2, sizeof e, hipMemcpyDeviceToHost, ctx->stream));
    EMU_HIP(ctx, hipStreamSynchronize(ctx->stream));
    if (time) *time = sc[0];
    if (dt) *dt = sc[1];
    if (steps) *steps = n;
    return status_decode(e, bad_index);
}


extern "C" int emu_state_kernel_ms(emu_state* st, int k, double* avg_ms, int64_t* launches)
{
    if (!st || k < 0 || k > 3) return EMU_ERR_ARG;
    emu_ctx* ctx = st->ctx;
    EMU_HIP(ctx, hipStreamSynchronize(ctx->stream));
    double tot = 0.0;
    int64_t n = 0;
    for (auto& m : st->marks) {
        if (m.k != k || !m.b) continue;
        float ms = 0;
        if (hipEventElapsedTime(&ms, m.a, m.b) == hipSuccess) {
            tot += ms;
            n++;
        }
    }
    if (avg_ms) *avg_ms = n ? tot / n : 0.0;
    if (launches) *launches = n;
    return EMU_OK;
}

extern "C" int emu_state_profile(emu_state* st, int enable)
{
    if (!st) return EMU_ERR_ARG;
    (void)hipStreamSynchronize(st->ctx->stream);
    for (auto& m : st->marks) {
        (void)hipEventDestroy(m.a);
        if (m.b) (void)hipEventDestroy(m.b);
    }
    st->marks.clear();
    st->profile = enable;
    return EMU_OK;
}

template <typename T> static void diag_t(emu_state* st, double* g4)
{
    Arrays<T> A = arrays_of<T>(st, st->cur);
    if (st->nf == 2)
        hipLaunchKernelGGL((k_diag_deposit<2, T>), dim3((unsigned)st->ncell), dim3(64), 0, st->ctx->stream, A,
                           st->cell_start, st->cell_cnt, st->ctx->g, st->cap, g4);
    else
        hipLaunchKernelGGL((k_diag_deposit<3, T>), dim3((unsigned)st->ncell), dim3(64), 0, st->ctx->stream, A,
                           st->cell_start, st->cell_cnt, st->ctx->g, st->cap, g4);
}

extern "C" int emu_state_flavor_amplitude(emu_state* st, double* sums)
{
    if (!st || !sums) return EMU_ERR_ARG;
    emu_ctx* ctx = st->ctx;
    hipStream_t s = ctx->stream;
    // the auxiliary grid (>= 4 values per cell) is free between steps
    hipLaunchKernelGGL(k_fill_grid, dim3(grid_blocks(st->ncell * st->naux)), dim3(256), 0, s, st->aux,
                       st->ncell * st->naux, 1, 0.0, nullptr, 0);
    if (st->precision == EMU_FP32_BULK) diag_t<float>(st, st->aux);
    else diag_t<double>(st, st->aux);
    // the two sums in red[4..5] (free between steps), as doubles
    hipLaunchKernelGGL(k_fill_u64v, dim3(1), dim3(64), 0, s, st->red + 4, 2, 0ull);
    hipLaunchKernelGGL(k_diag_reduce, dim3(grid_blocks(st->ncell)), dim3(256), 0, s, st->aux, st->ncell,
                       reinterpret_cast<double*>(st->red + 4));
    EMU_LAUNCH_CHECK(ctx, "flavor_amplitude");
    double h[2];
    EMU_HIP(ctx, hipMemcpyAsync(h, st->red + 4, sizeof h, hipMemcpyDeviceToHost, s));
    EMU_HIP(ctx, hipStreamSynchronize(s));
    sums[0] = h[0] / st->nscale;
    sums[1] = h[1] / st->nscale;
    return EMU_OK;
}
