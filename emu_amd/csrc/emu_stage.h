// emu_stage.h -- the fused stage kernel: gather + Hamiltonian + commutator +
// RK update of every particle of a cell, and the deposit of the next stage
// state as one small matrix product per cell on the FP64 matrix cores.
//
// A wave owns one cell, or two x-adjacent ones on larger grids, or a quarter of the
// chunks of a cell where cells are few and full (MODE), and takes its particles 64
// at a time (lane = particle).
//
// Gather (MFMA): with s(p) = (1, -vx, -vy, -vz) and G_g(t, c) the four field
// groups (M, Phix, Phiy, Phiz) of neighbour t,
//   inside_c(p) = sum_g s_g(p) sum_t w_t(p) G_g(t, c),
// the sum over t a product of the cell's 27 x 4 NH neighbour fields, staged in
// LDS once per cell with coalesced loads, and the particles' weights (WaveGather).
// Deposit (MFMA): the contribution of the cell's particles p to target cell t
// and field column q is D[t][q] = sum_p W[p][t] R[p][q], with W the shape
// weights and R = (1, vx, vy, vz) x q_c(p), q = N f - conj(Nbar fbar).  Over a
// chunk of 64 particles this is a (27 x 64) x (64 x 4NH) product, done with
// v_mfma_f64_16x16x4 (4 particles per instruction), so the sum over particles
// never leaves the matrix unit; the lane-layout transposition goes through LDS
// (9 shape factors and NH + 3 sources per particle).  The wave's accumulators
// are added to the grid once per cell with FP64 atomics.
#pragma once

#include "emu_internal.h"

namespace emu {

typedef double mf_d4 __attribute__((ext_vector_type(4)));
typedef float mf_f4 __attribute__((ext_vector_type(4)));

// Transpose of a 4 x 4 block of 16-lane rows: row i of register k <-> row k of
// register i.
__device__ __forceinline__ void transpose_rows(unsigned& a, unsigned& b, unsigned& c, unsigned& d)
{
    typedef unsigned u2 __attribute__((ext_vector_type(2)));
    auto swap32 = [](unsigned& x, unsigned& y) __attribute__((always_inline)) { // upper half of x <-> lower half of y
        const u2 r = __builtin_amdgcn_permlane32_swap(x, y, false, false);
        x = r[0];
        y = r[1];
    };
    auto swap16 = [](unsigned& x, unsigned& y) __attribute__((always_inline)) { // odd rows of x <-> even rows of y
        const u2 r = __builtin_amdgcn_permlane16_swap(x, y, false, false);
        x = r[0];
        y = r[1];
    };
    swap32(a, c);
    swap32(b, d);
    swap16(a, b);
    swap16(c, d);
}
__device__ __forceinline__ void transpose_rows(float& a, float& b, float& c, float& d)
{
    typedef unsigned u2 __attribute__((ext_vector_type(2)));
    auto swap32 = [](float& x, float& y) { // upper half of x <-> lower half of y
        const u2 r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(y), false, false);
        x = __uint_as_float(r[0]);
        y = __uint_as_float(r[1]);
    };
    auto swap16 = [](float& x, float& y) { // odd rows of x <-> even rows of y
        const u2 r = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(y), false, false);
        x = __uint_as_float(r[0]);
        y = __uint_as_float(r[1]);
    };
    swap32(a, c);
    swap32(b, d);
    swap16(a, b);
    swap16(c, d);
}
__device__ __forceinline__ void transpose_rows(double& a, double& b, double& c, double& d)
{
    double* v[4] = {&a, &b, &c, &d};
    unsigned lo[4], hi[4];
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const unsigned long long u = (unsigned long long)__double_as_longlong(*v[i]);
        lo[i] = (unsigned)u;
        hi[i] = (unsigned)(u >> 32);
    }
    transpose_rows(lo[0], lo[1], lo[2], lo[3]);
    transpose_rows(hi[0], hi[1], hi[2], hi[3]);
#pragma unroll
    for (int i = 0; i < 4; i++) *v[i] = __longlong_as_double((long long)(((unsigned long long)hi[i] << 32) | lo[i]));
}

template <typename T> struct Mfma16x16x4;
template <> struct Mfma16x16x4<double> {
    typedef mf_d4 acc_t;
    static __device__ __forceinline__ acc_t step(double a, double b, acc_t c)
    {
        return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
    }
    // the group and the component (of 4) of row i of A, such that element g of a
    // lane of the result is group g: element r of lane l holds row 4r + l/16
    static __device__ __forceinline__ int group(int i) { return i >> 2; }
    static __device__ __forceinline__ int comp(int i) { return i & 3; }
    // One component's four groups on the four-block form (16 cycles against 64): A's
    // row l%4 is the group, B as above, the four blocks the quarters of the
    // particles.  Lane l holds group l/16 of particle l%16: its term of the contraction.
    typedef double tail_t;
    static __device__ __forceinline__ tail_t tail_zero() { return 0.0; }
    static __device__ __forceinline__ tail_t tail_step(double a, double b, tail_t c)
    {
        return __builtin_amdgcn_mfma_f64_4x4x4f64(a, b, c, 0, 0, 0);
    }
    static __device__ __forceinline__ double tail_term(tail_t d, int lane, double v0, double v1, double v2)
    {
        const int g = lane >> 4;
        return (g == 0 ? 1.0 : (g == 1 ? v0 : (g == 2 ? v1 : v2))) * d;
    }
};
template <> struct Mfma16x16x4<float> {
    typedef mf_f4 acc_t;
    static __device__ __forceinline__ acc_t step(float a, float b, acc_t c)
    {
        return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
    }
    // element r of lane l holds row 4 (l/16) + r
    static __device__ __forceinline__ int group(int i) { return i & 3; }
    static __device__ __forceinline__ int comp(int i) { return i >> 2; }
    // One component's four groups on the sixteen-block form (8 cycles against 32): A's
    // row l%4 is the group, B as above, a block a neighbour (l/16) and a quarter of
    // the particles.  Element g of lane l is group g of particle l%16 over the
    // neighbours l/16, l/16 + 4, ..: a part of the sum.
    typedef mf_f4 tail_t;
    static __device__ __forceinline__ tail_t tail_zero() { return mf_f4{0.0f, 0.0f, 0.0f, 0.0f}; }
    static __device__ __forceinline__ tail_t tail_step(float a, float b, tail_t c)
    {
        return __builtin_amdgcn_mfma_f32_4x4x1f32(a, b, c, 0, 0, 0);
    }
    static __device__ __forceinline__ float tail_term(tail_t d, int, float v0, float v1, float v2)
    {
        return d[0] + v0 * d[1] + v1 * d[2] + v2 * d[3];
    }
};

// The gather of a wave's chunk of up to 64 particles on the matrix cores:
//   out_c(p) = sum_t w_t(p) (G_0c(t) + s v_1(p) G_1c(t) + s v_2(p) G_2c(t) + s v_3(p) G_3c(t)),
// s = SIGN, t the WX x WY x WZ neighbours, rows of 4 NH fields in LDS.  Per tile of 16
// particles the product is G^T W: A's rows are 4 components x the 4 field groups,
// K the neighbours (4 per step), B's columns the particles, so that a lane's four
// results are the four groups of one component of one particle, and contracting
// them with v is 3 FMAs in the lane: ceil(27 / 4) = 7 steps per 4 components.  (A
// tile of 16 particles by NH of 16 columns with the groups as K takes 27 steps
// for any NH.)  The particle's own lane forms its 27 weights once; a transpose of
// 16-lane rows turns four of them into the operands of all four tiles, and
// another returns the results, without LDS.
// LIN: the neighbours' rows follow each other in t, LIN values apart, and a row of
// zeros (or any finite values) follows the last one.
// BYITSELF: NF = 3's ninth component runs on the small blocks instead of a third tile
// that is three quarters padding (per 16 particles 7 x 48 cycles less in FP64, 7 x 24
// in FP32).  At 64^3 x 92, ms of stages 1 to 4: FP64 3.94 4.18 5.55 4.95 -> 3.87 4.04
// 5.46 4.91.  FP32-bulk 2.70 2.61 3.24 3.12 -> 2.76 2.55 3.17 3.21: its offsets
// cost stage 1 registers that it has not got (scratch memory) and stage 4 its fourth
// wave per SIMD (134 registers, 125 without), so those two keep the third tile.
template <int NF, typename T, int WX, int WY, int WZ, bool PACK = false, int LIN = 0, bool BYITSELF = true> struct WaveGather {
    using MF = Mfma16x16x4<T>;
    static constexpr int nh = NH<NF>, NT = WX * WY * WZ, KK = (NT + 3) / 4;
    static constexpr bool TAIL = BYITSELF && nh % 4 == 1;
    static constexpr int MG = TAIL ? nh / 4 : (nh + 3) / 4;
    // this lane's entry of A at step k, row i = l%16, neighbour t = 4k + l/16 (past
    // the last one: any in-range entry, its weight is zero; rows past NH feed
    // results that are dropped)
    // (LIN: step 0 only; PACK: two 16-bit offsets each, taken apart once per chunk)
    unsigned goff[LIN ? 1 : (PACK ? (KK + 1) / 2 : KK)];
    int tail; // from there to the lane's entry of the last component

    // row(t): offset of neighbour t's row of fields
    __device__ __forceinline__ void init(int lane)
    {
        static_assert(LIN > 0, "rows at a constant distance");
        goff[0] = (lane >> 4) * LIN + MF::group(lane & 15) * nh + MF::comp(lane & 15);
        set_tail(lane);
    }
    __device__ __forceinline__ void set_tail(int lane)
    {
        tail = ((lane & 3) - MF::group(lane & 15)) * nh + nh - 1 - MF::comp(lane & 15);
    }
    template <typename F> __device__ __forceinline__ void init(int lane, F&& row)
    {
        static_assert(LIN == 0, "rows anywhere");
        set_tail(lane);
#pragma unroll
        for (int k = 0; k < KK; k++) {
            const int t = 4 * k + (lane >> 4);
            const unsigned o = row(t < NT ? t : NT - 1) + MF::group(lane & 15) * nh + MF::comp(lane & 15);
            if constexpr (PACK) goff[k / 2] = k % 2 ? goff[k / 2] | o << 16 : o;
            else goff[k] = o;
        }
    }

    // wd: the particle's shape factors; rows(m): the fields of tile m's cell; vel(m):
    // v of particle 16 m + l%16, by pointer; ntile: tiles with particles
    template <int SIGN, typename F, typename V>
    __device__ __forceinline__ void run(const double wd[3][3], int ntile, F&& rows, V&& vel, T* out)
    {
        int off[KK];
#pragma unroll
        for (int k = 0; k < KK; k++) {
            if constexpr (LIN > 0) {
                off[k] = goff[0] + 4 * k * LIN;
            } else if constexpr (PACK) {
                if (k % 2 == 0) asm volatile("" : "+v"(goff[k / 2]));
                off[k] = k % 2 ? goff[k / 2] >> 16 : goff[k / 2] & 0xffffu;
            } else {
                off[k] = goff[k];
            }
        }
        T w[4 * KK];
        {
            T fx[3], fyz[3][3];
#pragma unroll
            for (int i = 0; i < 3; i++) fx[i] = T(wd[0][i]);
#pragma unroll
            for (int k = 0; k < 3; k++)
#pragma unroll
                for (int j = 0; j < 3; j++) fyz[k][j] = T(wd[1][j]) * T(wd[2][k]);
#pragma unroll
            for (int t = 0; t < 4 * KK; t++) {
                const int i = WX == 1 ? 1 : t % WX, j = WY == 1 ? 1 : (t / WX) % WY, k = WZ == 1 ? 1 : (t / (WX * WY)) % 3;
                w[t] = t < NT ? fx[i] * fyz[k][j] : T(0);
            }
        }
#pragma unroll
        for (int k = 0; k < KK; k++) transpose_rows(w[4 * k], w[4 * k + 1], w[4 * k + 2], w[4 * k + 3]);
        // w[4 k + m] now holds tile m's operand of step k
        const int lane = threadIdx.x & 63;
        T res[MG][4], last[4];
#pragma unroll
        for (int m = 0; m < 4; m++) {
            last[m] = T(0);
#pragma unroll
            for (int c = 0; c < MG; c++) res[c][m] = T(0);
            if (m < ntile) {
                const T* G = rows(m);
                T v0, v1, v2;
                vel(m, v0, v1, v2);
                typename MF::acc_t acc[MG];
#pragma unroll
                for (int c = 0; c < MG; c++) acc[c] = typename MF::acc_t{T(0), T(0), T(0), T(0)};
                typename MF::tail_t rest = MF::tail_zero();
#pragma unroll
                for (int k = 0; k < KK; k++) {
#pragma unroll
                    for (int c = 0; c < MG; c++) acc[c] = MF::step(G[off[k] + 4 * c], w[4 * k + m], acc[c]);
                    if (TAIL) rest = MF::tail_step(G[off[k] + tail], w[4 * k + m], rest);
                }
                if (TAIL) last[m] = SIGN < 0 ? MF::tail_term(rest, lane, -v0, -v1, -v2) : MF::tail_term(rest, lane, v0, v1, v2);
#pragma unroll
                for (int c = 0; c < MG; c++)
                    res[c][m] = SIGN < 0 ? acc[c][0] - v0 * acc[c][1] - v1 * acc[c][2] - v2 * acc[c][3]
                                         : acc[c][0] + v0 * acc[c][1] + v1 * acc[c][2] + v2 * acc[c][3];
            }
        }
#pragma unroll
        for (int c = 0; c < MG; c++) {
            transpose_rows(res[c][0], res[c][1], res[c][2], res[c][3]);
#pragma unroll
            for (int j = 0; j < 4; j++)
                if (4 * c + j < nh) out[4 * c + j] = res[c][j];
        }
        if (TAIL) { // the rows hold terms of one sum
            transpose_rows(last[0], last[1], last[2], last[3]);
            out[nh - 1] = (last[0] + last[1]) + (last[2] + last[3]);
        }
    }
};

template <typename T> struct PArrays {
    double* pos[3];
    int64_t* id;
    T* pup[4]; // pupx, pupy, pupz, pupt
    T* Nn[2];  // N, Nbar
    T* Ll[2];  // L, Lbar
    T* f;      // [2 NH][np]: nu components then nubar
};

// What the next step's dt follows from, besides the grid's maxima.
struct DtParams {
    double dt_translation, flavor_cfl, max_adaptive_speedup, Vvac_max, fixed_dt;
    int use_flavor;
    double vst_scale; // 2 NF sqrt2 GF / dV of the scaled weights
};

// compute_dt's maxima, as the bit patterns of non-negative doubles: word 0 the
// adaptive speed, then the conservative one in kSlots words, a cache line
// apart, that the maximum is the largest of.  Stage 4's waves spread over the
// slots: all on one word they queued for it (16^3 cells, NF = 2: 40 us a
// launch against 21).
struct DtRed {
    static constexpr int kSlots = 64, kStride = 16, words = (1 + kSlots) * kStride;
    static EMU_HD int slot(int i) { return (1 + i % kSlots) * kStride; }
};

// main.cpp:193-198 and Evolve.cpp:57-88: the next dt from the maxima, which are
// left at zero for the next step's.  All 64 lanes of one wave call it.
__device__ __forceinline__ double next_dt(unsigned long long* red, const DtParams& p, unsigned long long* err)
{
    const int lane = threadIdx.x & 63;
    double vst_max = __longlong_as_double((long long)red[DtRed::slot(lane)]);
    for (int off = 32; off > 0; off >>= 1) vst_max = fmax(vst_max, __shfl_xor(vst_max, off));
    const double vad_max = __longlong_as_double((long long)red[0]);
    double dt_flavor = 0.0;
    if (p.use_flavor) {
        const double vad = vad_max + p.Vvac_max;
        const double vst = vst_max + p.Vvac_max;
        const double dfa = phys::hbar / vad * p.flavor_cfl;
        const double dfs = phys::hbar / vst * p.flavor_cfl;
        dt_flavor = dfs;
        if (p.max_adaptive_speedup > 1) dt_flavor = fmin(dfs * p.max_adaptive_speedup, dfa);
    }
    red[DtRed::slot(lane)] = 0;
    if (lane == 0) red[0] = 0;
    if (p.fixed_dt > 0) return p.fixed_dt;
    if (p.dt_translation != 0.0 && dt_flavor != 0.0) return fmin(p.dt_translation, dt_flavor);
    if (p.dt_translation != 0.0) return p.dt_translation;
    if (dt_flavor == 0.0 && lane == 0) atomicMin(err, status_word_noindex(EMU_ERR_DT));
    return dt_flavor;
}

// The particles' time after a step of length h: the four weighted stages.
__device__ __forceinline__ double advance_time(double t, double h)
{
#pragma clang fp contract(off)
    t = h * (1. / 6.) * 1.0 + t;
    t = h * (1. / 3.) * 1.0 + t;
    t = h * (1. / 3.) * 1.0 + t;
    t = h * (1. / 6.) * 1.0 + t;
    return t;
}

// ---------------------------------------------------------------------------
// Stable counting sort by cell after each step.  A particle moves at most one
// cell per dimension per step (c dt < dx, checked on the host), so its move
// is one of 27 offsets e.  Particles arriving in cell t are ordered by the
// canonical index of e, then by their position in their old cell: every
// particle's destination is base[old cell][e] + (its rank among the particles
// of its old cell with the same e), which makes the order deterministic.
// ---------------------------------------------------------------------------
__device__ __forceinline__ int wrap_cell(int i, int n) { return i < 0 ? i + n : (i >= n ? i - n : i); }

// f(e, source) for every move e that exists on the grid (a 1-cell dimension
// has only move 0, a 2-cell one 0 and +1), with the cell that particles come
// from into cell t by it; canonical order of e.
template <typename F> __device__ __forceinline__ void for_moves(int t, const Geom& g, F&& f)
{
    const int tx = t % g.n[0], ty = (t / g.n[0]) % g.n[1], tz = t / (g.n[0] * g.n[1]);
#pragma unroll
    for (int ez = -1; ez <= 1; ez++)
#pragma unroll
        for (int ey = -1; ey <= 1; ey++)
#pragma unroll
            for (int ex = -1; ex <= 1; ex++) {
                const int ed[3] = {ex, ey, ez};
                bool ok = true;
#pragma unroll
                for (int d = 0; d < 3; d++) ok = ok && !(g.n[d] == 1 && ed[d] != 0) && !(g.n[d] == 2 && ed[d] == -1);
                if (!ok) continue;
                const int sx = wrap_cell(tx - ex, g.n[0]), sy = wrap_cell(ty - ey, g.n[1]), sz = wrap_cell(tz - ez, g.n[2]);
                f((ez + 1) * 9 + (ey + 1) * 3 + (ex + 1), ((int64_t)sz * g.n[1] + sy) * g.n[0] + sx);
            }
}

// base[source][e] for every source of target t, in canonical move order, from
// the target's first slot.
__device__ __forceinline__ void write_bases(int t, int first, const int* __restrict__ m, const Geom& g, int* __restrict__ base)
{
    int run = first;
    for_moves(t, g, [&](int e, int64_t src) {
        base[src * 27 + e] = run;
        run += m[src * 27 + e];
    });
}

// The sort plan, between stage 1 (which counts the moves) and stage 4 (which needs the
// bases), a lane per target cell: either by waves of its own at the front of the
// stage 2 and stage 3 launches, or by two launches on a second stream (k_plan).
struct SortPlan {
    const int* m;  // mcount
    int* start;    // first slot of each cell's run, a multiple of align
    int* cnt;      // particles arriving in each cell; cnt[ncell] = 0 for the store's scan
    int* sums;     // slots of each wave's cells
    int* base;     // [ncell][27]
    int align;
    int per;       // 64-cell rows a wave takes
    int waves;     // planning waves (per rows of 64 cells each cover 0 .. ncell)

    // stage 2: the counts, and the starts counted from the wave's first slot
    __device__ __forceinline__ void counts(int wave, int lane, const Geom& g, int ncell) const
    {
        int total = 0;
        for (int j = 0; j < per; j++) {
            const int t = (wave * per + j) * 64 + lane;
            int n = 0;
            if (t < ncell) for_moves(t, g, [&](int e, int64_t src) { n += m[src * 27 + e]; });
            const int slots = (n + align - 1) / align * align;
            int upto = slots; // inclusive scan over the lanes
#pragma unroll
            for (int off = 1; off < 64; off <<= 1) {
                const int o = __shfl_up(upto, off);
                if (lane >= off) upto += o;
            }
            if (t <= ncell) cnt[t] = n;
            if (t < ncell) start[t] = total + upto - slots;
            total += __shfl(upto, 63);
        }
        if (lane == 0) sums[wave] = total;
    }
    // stage 3: the slots of the waves before complete the starts; the bases
    __device__ __forceinline__ void bases(int wave, int lane, const Geom& g, int ncell) const
    {
        int before = 0;
        for (int w = lane; w < wave; w += 64) before += sums[w];
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) before += __shfl_xor(before, off);
        for (int j = 0; j < per; j++) {
            const int t = (wave * per + j) * 64 + lane;
            if (t >= ncell) return;
            const int first = start[t] + before;
            start[t] = first;
            write_bases(t, first, m, g, base);
        }
    }
};

template <typename T> struct StageArgs {
    PArrays<T> cur; // current copy, sorted by cell_start
    PArrays<T> dst; // stage 4 writes the step's result here, sorted by the new cells
    T* Y;           // stage state
    T* acc;         // RK accumulator
    // the sort plan: stage 1 writes each particle's move (of 27) and its rank
    // among the particles of its cell with that move, and the cells' counts per
    // move; stage 4 reads rank, move and the moves' destinations
    int* rank;
    unsigned char* mv;
    int* mcount;
    const int* mbase;
    const int* cell_start; // first slot of each cell (a multiple of the slot alignment)
    const int* cell_cnt;   // particles of each cell
    const double* gin;  // grid read by the gather
    double* gout;       // grid deposited by this launch
    double* aux;        // compute_dt auxiliaries
    double* gclear;     // grid this launch sets to its base for a later deposit (null: none)
    int clear_aux;      // and the auxiliaries
    double m00;         // the base: the matter term on component 0, zero elsewhere
    int want_dt;        // stage 4: the conservative flavour bound of the grid it gathers, into red
    unsigned long long* red; // compute_dt's maxima (DtRed)
    int step_end;       // stage 0: also finish the step (time, steps and the next dt)
    DtParams dtp;
    double* scal;       // [0] time [1] dt
    int64_t* steps;
    const double* dt;
    unsigned long long* err;
    int64_t np; // slots per array: the stride of the component-major arrays
    int64_t ncell;
    int stage; // 0 = deposit only, 1..4
    int want_aux;
    int blocks_per_xcd;
    SortPlan plan;   // stages 2 and 3: planned by the first workgroups (none: no waves)
    int plan_blocks; // a multiple of 8, so that the stage's own workgroups keep their XCDs
    Geom g;
    double vac[9]; // M2 c^4 / (2 hbar)
    double coef;   // sqrt2 GF / dV / hbar
    double maxError;
};

// Component of the i-th diagonal entry, i at run time.
template <int NF> __device__ __forceinline__ int herm_re_rt(int i)
{
    return i == 0 ? 0 : (i == 1 ? herm_re<NF>(1, 1) : herm_re<NF>(NF - 1, NF - 1));
}

template <int NF> __device__ __forceinline__ constexpr bool is_im_comp(int c)
{
    for (int a = 0; a < NF; a++)
        for (int b = a + 1; b < NF; b++)
            if (c == herm_im<NF>(a, b)) return true;
    return false;
}

__device__ __forceinline__ int bin1(double pos, double plo, double dxi, int n)
{
#pragma clang fp contract(off)
    return pmod(nearest_cell_center_index((pos - plo) * dxi), n);
}

// x += (dt b_i) v for the four RK4 stages, rounded as the reference's saxpy
// sequence (FlavoredNeutrinoContainer.H:43-45) with v = c pup/pupt.
__device__ __forceinline__ double advance_pos(double x, double v, const double a[4])
{
#pragma clang fp contract(off)
    x = a[0] * v + x;
    x = a[1] * v + x;
    x = a[2] * v + x;
    x = a[3] * v + x;
    return x;
}

__device__ __forceinline__ double wrap1(double x, double rlo, double rhi, double L)
{
#pragma clang fp contract(off)
    // one period per step at most; the bound keeps non-finite input from looping
    if (x > rhi) {
        for (int it = 0; it < 8 && x > rhi; it++) x -= L;
        if (x < rlo || x > rhi) x = rlo;
    } else if (x < rlo) {
        for (int it = 0; it < 8 && x < rlo; it++) x += L;
        if (x > rhi || x < rlo) x = rhi;
    }
    return x;
}

template <int NF>
__device__ __forceinline__ int renorm_fp64(double* f, double L, double maxError)
{
#pragma clang fp contract(off)
    double sumP = 0;
#pragma unroll
    for (int i = 0; i < NF; i++) sumP += f[herm_re<NF>(i, i)];
    double error = sumP - 1.0;
    if (fabs(error) > 100. * maxError) return EMU_ERR_TRACE;
    if (fabs(error) > maxError) {
#pragma unroll
        for (int i = 0; i < NF; i++) f[herm_re<NF>(i, i)] -= error / NF;
    }
#pragma unroll
    for (int i = 0; i < NF; i++) {
        double& fii = f[herm_re<NF>(i, i)];
        if (fii < -100. * maxError) return EMU_ERR_NEGDIAG;
        if (fii < -maxError) fii = 0;
    }
    const double length = sqrt(su_mag2<NF, double>(f));
    error = length - L;
    if (fabs(error) > 100. * maxError) return EMU_ERR_LENGTH;
    if (fabs(error) > maxError) {
#pragma unroll
        for (int c = 0; c < NH<NF>; c++) f[c] /= length / L;
    }
    return EMU_OK;
}

// End-of-step position: the four stage saxpys, then the periodic shift.
__device__ __forceinline__ void end_position(const double pos[3], const double v[3], double dt, const Geom& g,
                                             double npos[3])
{
    const double ai[4] = {dt * (1. / 6.), dt * (1. / 3.), dt * (1. / 3.), dt * (1. / 6.)};
#pragma unroll
    for (int d = 0; d < 3; d++) npos[d] = wrap1(advance_pos(pos[d], v[d], ai), g.rlo[d], g.rhi[d], g.L[d]);
}

// The move (-1, 0, 1) from cell index `from` to the cell of x along one
// dimension of n cells; more than one cell sets bad.  With 2 cells both
// neighbours are the same cell, reached by +1.
__device__ __forceinline__ int move1(int from, double x, double plo, double dxi, int n, bool& bad)
{
    int to;
    {
#pragma clang fp contract(off)
        to = nearest_cell_center_index((x - plo) * dxi);
    }
    if (to < 0) to += n; // x = plo exactly belongs to the last cell
    const int d = to - from;
    if (d == 0) return 0;
    if (d == 1 || d == 1 - n) return 1;
    if (d == -1 || d == n - 1) return -1;
    bad = true;
    return 0;
}

// Ways to map waves to cells (MODE).
//  0: every wave is its own patch of two cells (below), stages its own box and
//     flushes its deposit directly: no workgroup barrier.
//  1: as 0 with one cell (box = its 27 neighbours).
//  2: the WPB waves of a workgroup take a patch of WPB cells (2 along x, then
//     2 along y, when the stencil is 3 wide there, else along z); the patch's
//     neighbourhood box (PX + WX - 1) x (PY + WY - 1) x (PZ + WZ - 1) is staged
//     once for all of them, and the deposits are summed over the box in LDS
//     before one set of global atomics (56% fewer for a 2 x 2 patch at the 3-D
//     stencil).
//  3: the WPB waves of a workgroup share one cell, 64 particles each in turn,
//     with the box staged once and the deposits summed in LDS as in 2: for grids
//     with too few cells to fill the chip and several chunks per cell.
// PM (a shared patch) is MODE >= 2.  In MODE 0 a wave takes CPW = 2
// cells, x-adjacent, as one patch: their particles form one list of 16-particle
// tiles (the first cell's, then the second's), so that a cell of 92 particles no
// longer leaves 36 of a chunk's 64 lanes idle, and the wave stages the two
// cells' 4 x 3 x 3 box once.
template <int WX, int WY, int WZ, int CELLS> struct Patch {
    static constexpr int PX = WX == 3 && CELLS >= 2 ? 2 : 1;
    static constexpr int PY = WY == 3 && CELLS >= 2 * PX ? 2 : 1;
    static constexpr int PZ = CELLS / (PX * PY);
    static_assert(PX * PY * PZ == CELLS, "cells of one patch");
    static constexpr int NBX = PX + WX - 1, NBY = PY + WY - 1, NBZ = PZ + WZ - 1;
    static constexpr int NB = NBX * NBY * NBZ;
};

// compute_dt auxiliaries per cell.  AUX = 1: the diagonal sums N_ii + Nbar_ii
// (i < NF), all that the conservative flavour bound needs; AUX = 2: also
// Nbar Im(fbar_ab) v_d per pair a < b and direction d, for the adaptive bound
// (max_adaptive_speedup > 1).  Deposited columns, and sources per particle:
// N f_ii + Nbar fbar_ii, then Nbar Im(fbar_ab).
template <int NF> constexpr int aux_columns(int AUX)
{
    return AUX == 0 ? 0 : (AUX == 1 ? NF : NF + 3 * (NF * (NF - 1) / 2));
}
template <int NF> constexpr int aux_sources(int AUX)
{
    return AUX == 0 ? 0 : (AUX == 1 ? NF : NF + NF * (NF - 1) / 2);
}

// Values of T per particle in the LDS source rows: NH + 4 main sources, the
// auxiliary ones, and one of padding where that count is even.  The deposit
// reads one column of four consecutive rows at once; an odd row length keeps
// those rows off the same LDS banks (16 doubles = 128 bytes would put every
// row on bank 0).
template <int NF> constexpr int stage_source_row(int AUX)
{
    const int n = NF * NF + 4 + aux_sources<NF>(AUX);
    return n % 2 == 0 ? n + 1 : n;
}

// LDS of one wave's own region, in doubles: 9 shape factors per particle
// (double) and the source row (T).
template <int NF, typename T, int AUX> constexpr int stage_lds_doubles_per_wave()
{
    return 64 * 9 + 64 * stage_source_row<NF>(AUX) * (int)sizeof(T) / 8;
}

// cells per wave: MODE 0 takes two, side by side along x (emu_state::pairs says when)
template <int MODE> constexpr int stage_cells_per_wave() { return MODE == 0 ? 2 : 1; }

// whether MODE 0 is there at all: for the 3-D stencil, where the 4 x 3 x 3 box still
// fits the waves per SIMD that the registers allow (three in FP32-bulk and for NF = 2;
// FP64's NF = 3 would not fit two)
template <int NF, typename T, int WX> constexpr bool stage_has_pairs() { return WX == 3 && (sizeof(T) == 4 || NF == 2); }

template <typename T, int WX, int WY, int WZ, int WPB, int MODE>
using StagePatch = Patch<WX, WY, WZ, (MODE == 2 ? WPB : stage_cells_per_wave<MODE>())>;

// LDS of a workgroup, in doubles.  The tables of the box's cell indices (NB ints)
// come first.  PM: then the staged neighbourhood box (gather stages, NB x 4 NH
// values of T) and the waves' regions; the deposit's merge buffer (NB x deposited
// columns, double) reuses that space once every wave is done with it.  Without
// PM: per wave, its own box and its region.  The host sizes the launch with this
// function.
template <int NF, typename T, int WX, int WY, int WZ, int WPB, int S, int AUX, int MODE>
constexpr int stage_lds_doubles_per_block()
{
    constexpr bool PM = MODE >= 2;
    constexpr int nh = NF * NF;
    constexpr int NB = StagePatch<T, WX, WY, WZ, WPB, MODE>::NB;
    constexpr int ct = (PM ? 1 : WPB) * ((NB + 1) / 2);
    constexpr int gsh = S == 0 ? 0 : (NB * 4 * nh * (int)sizeof(T) + 7) / 8;
    if (!PM) return ct + WPB * (gsh + stage_lds_doubles_per_wave<NF, T, AUX>());
    constexpr int work = gsh + WPB * stage_lds_doubles_per_wave<NF, T, AUX>();
    constexpr int merge = S <= 3 ? NB * (4 * nh + aux_columns<NF>(AUX)) : 0;
    return ct + (work > merge ? work : merge);
}

// the mapping of each launch kind (measured per launch kind at 64^3 x 92,
// NF = 3): the deposit-only launch in both precisions and FP32-bulk stage 4
// merge their deposits (MODE 2); the other RK stages run faster with
// independent waves
template <typename T, int S, int AUX> constexpr bool stage_merges()
{
    return S == 0 || (S == 4 && sizeof(T) == 4);
}
// waves per workgroup: 4 (MODE 2 and 3); otherwise 2, or 1 for the launches
// with the compute_dt auxiliaries, whose larger LDS rows would otherwise leave
// a CU a whole 2-wave workgroup short (FP64 at 64^3 x 92: 6 waves per CU with
// 2-wave workgroups, 7 with single waves)
template <int MODE, int AUX> constexpr int stage_waves_per_block() { return MODE >= 2 ? 4 : (AUX != 0 ? 1 : 2); }

// Columns of patches (k_stage); at 64^3 x 92, NF = 3, ms per step of the five
// launches, FP32-bulk and FP64: plain order 13.77 / 22.2, 4 x 4 13.27 / 21.4, 4 x 8
// 13.14 / 21.3, 8 x 8 13.14 / 21.4, 2 x 2 13.33 / 21.5, 4 x 4 rows taken whole 13.41 / 21.8.
constexpr int kTileY = 4, kTileZ = 8;

// S: 0 = deposit only (the step's result, or the initial state), 1..4 = RK
// stage; AUX: also deposit the compute_dt auxiliaries (S = 0 or 3; 1 or 2 as
// for aux_columns).
template <int NF, typename T, int WX, int WY, int WZ, int WPB, int S, int AUX, int MODE>
__global__ __launch_bounds__(64 * WPB) __attribute__((amdgpu_waves_per_eu(sizeof(T) == 4 ? 3 : 2))) void k_stage(StageArgs<T> a)
{
    constexpr bool PM = MODE >= 2;    // the workgroup shares one patch and its staged box, and merges its deposits in LDS
    constexpr bool SPLIT = MODE == 3; // the patch is one cell, whose chunks the waves take in turn
    constexpr int nh = NH<NF>;
    constexpr int QG = 4 * nh;
    constexpr int NT = WX * WY * WZ;        // target cells of a source cell
    constexpr int MT = (NT + 15) / 16;       // MFMA row tiles
    constexpr int QGA = QG + aux_columns<NF>(AUX); // deposited columns
    constexpr int NTL = (QGA + 15) / 16;     // MFMA column tiles
    constexpr int NPAIR = NF * (NF - 1) / 2;
    // compute_dt auxiliaries per cell (aux_columns): N_ii + Nbar_ii, then (AUX = 2)
    // Nbar Im(fbar_ab) v_d.  N_ii and Nbar_ii separately follow from the sum and
    // M_ii = N_ii - Nbar_ii (+ matter on 00).  They are deposited as columns
    // QG .. QGA - 1 of the same product, into rows of NAUX (the full set's
    // count, whichever part is deposited).
    constexpr int NAUX = NF + 3 * NPAIR;
    constexpr int NSRC = nh + 4;             // q_c, vhat and the constant 1 per particle
    constexpr int NSAUX = aux_sources<NF>(AUX);
    constexpr int NSR = stage_source_row<NF>(AUX); // a particle's source row: main, auxiliary, padding
    static_assert(NSR >= NSRC + NSAUX, "source row");
    extern __shared__ double lds[];

    const Geom& g = a.g;
    constexpr int s = S;
    constexpr bool aux = AUX != 0;
    constexpr int CPW = stage_cells_per_wave<MODE>();
    using PT = StagePatch<T, WX, WY, WZ, WPB, MODE>;
    constexpr int NB = PT::NB;
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int lane = threadIdx.x & 63;
    if constexpr (s == 2 || s == 3) {
        if ((int)blockIdx.x < a.plan_blocks) { // the sort plan's waves
            const int w = blockIdx.x * WPB + wave;
            if (w >= a.plan.waves) return;
            if (s == 2) a.plan.counts(w, lane, g, (int)a.ncell);
            else a.plan.bases(w, lane, g, (int)a.ncell);
            return;
        }
    }
    // blocks go round-robin over the 8 XCDs; give each XCD a contiguous run of patches
    const int npx = (g.n[0] + PT::PX - 1) / PT::PX, npy = (g.n[1] + PT::PY - 1) / PT::PY;
    const int npz = (g.n[2] + PT::PZ - 1) / PT::PZ;
    const int b = blockIdx.x - (s == 2 || s == 3 ? a.plan_blocks : 0);
    const int bgroup = (b & 7) * a.blocks_per_xcd + (b >> 3);
    // PM: the block's patch; otherwise this wave's patch of CPW cells, WPB consecutive per block
    const int patch = __builtin_amdgcn_readfirstlane(PM ? bgroup : bgroup * WPB + wave);
    if (patch >= npx * npy * npz) return; // uniform over the workgroup (PM) or the wave
    // Patches are taken in columns of kTileY x kTileZ along x: the waves in flight on
    // an XCD then hold neighbours in all three dimensions, so that what they
    // exchange (stage 4's particles for a neighbour's lines, the deposits on
    // shared cells, the neighbourhood fields) meets in its L2 and in the memory-side
    // cache.  In plain x, y, z order the z neighbours are a plane apart and stage 4's
    // lines were written to memory in parts.
    int bx, by, bz;
    {
        const int slab = npx * npy * kTileZ, tz = patch / slab;
        int r = patch - tz * slab;
        const int hz = min(kTileZ, npz - tz * kTileZ), rows = npx * kTileY * hz, ty = r / rows;
        r -= ty * rows;
        const int hy = min(kTileY, npy - ty * kTileY), x = r / (hy * hz);
        r -= x * hy * hz;
        bx = x * PT::PX;
        by = (ty * kTileY + r % hy) * PT::PY;
        bz = (tz * kTileZ + r / hy) * PT::PZ;
    }
    const int pw = PM && !SPLIT ? wave : 0; // this wave's cell within the patch
    const int ox = pw % PT::PX, oy = (pw / PT::PX) % PT::PY, oz = pw / (PT::PX * PT::PY);
    const int cx = bx + ox, cy = by + oy, cz = bz + oz;
    // a wave whose cell lies outside the domain (a partial patch) or holds no
    // particle has nothing to do, but it stays for the workgroup's barriers
    const bool inside_domain = cx < g.n[0] && cy < g.n[1] && cz < g.n[2];
    const int cell = inside_domain ? (cz * g.n[1] + cy) * g.n[0] + cx : 0;
    // (wave-uniform, so the particle arrays are addressed from scalar bases)
    const int beg = __builtin_amdgcn_readfirstlane(inside_domain ? a.cell_start[cell] : 0);
    const int end = __builtin_amdgcn_readfirstlane(inside_domain ? beg + a.cell_cnt[cell] : 0);
    // CPW = 2: the wave's second cell, x + 1 (none past the domain's last column)
    const bool inside1 = CPW == 2 && inside_domain && cx + 1 < g.n[0];
    const int cell1 = inside1 ? cell + 1 : 0;
    const int beg1 = __builtin_amdgcn_readfirstlane(inside1 ? a.cell_start[cell1] : 0);
    const int end1 = __builtin_amdgcn_readfirstlane(inside1 ? beg1 + a.cell_cnt[cell1] : 0);
    // cell i of the neighbourhood box, box index (i, j, k) <-> the patch base
    // minus one in each 3-wide dimension, plus (i, j, k), periodic
    // (one conditional wrap covers a single cell's box: offsets are -1..+1 and a
    // 3-wide stencil implies at least 2 cells in that dimension)
    auto wrapc = [](int x, int n) {
        return PM || CPW == 2 ? pmod(x, n) : (x < 0 ? x + n : (x >= n ? x - n : x));
    };
    auto box_cell = [&](int e) -> int64_t {
        const int i = e % PT::NBX, j = (e / PT::NBX) % PT::NBY, k = e / (PT::NBX * PT::NBY);
        const int ci = wrapc(bx - (WX == 3 ? 1 : 0) + i, g.n[0]);
        const int cj = wrapc(by - (WY == 3 ? 1 : 0) + j, g.n[1]);
        const int ck = wrapc(bz - (WZ == 3 ? 1 : 0) + k, g.n[2]);
        return ((int64_t)ck * g.n[1] + cj) * g.n[0] + ci;
    };
    // box index of this wave's stencil target t (of its first cell; the second
    // cell's is one further along x)
    auto box_of = [&](int t) __attribute__((always_inline)) -> int {
        const int ii = t % WX, jj = (t / WX) % WY, kk = t / (WX * WY);
        return ((oz + kk) * PT::NBY + (oy + jj)) * PT::NBX + (ox + ii);
    };
    // set this wave's cells of the grid (and the auxiliaries) that a later launch
    // deposits into: the cells partition over the waves, so no fill launches are
    // needed between the stages
    const bool owner = inside_domain && (!SPLIT || wave == 0); // of the cell's own values
    if (a.gclear && owner) {
        const int n = (inside1 ? 2 : 1) * QG;
        double* gc = a.gclear + (int64_t)cell * QG;
        for (int e = lane; e < n; e += 64) gc[e] = e == 0 || e == QG ? a.m00 : 0.0;
    }
    if (s == 2 && a.clear_aux && owner) {
        const int n = (inside1 ? 2 : 1) * NAUX;
        for (int e = lane; e < n; e += 64) a.aux[(int64_t)cell * NAUX + e] = 0.0;
    }
    if constexpr (s == 4) {
        // compute_dt's conservative bound (Evolve.cpp:40-56) of this wave's cell:
        // N_ii and Nbar_ii from the auxiliaries S_ii and M_ii (CPW = 2: the second
        // cell's in the upper lanes)
        if (a.want_dt && owner) {
            const int i = CPW == 2 ? lane & 31 : lane;
            const bool second = CPW == 2 && lane >= 32;
            double v = 0.0;
            if (i < NF && (!second || inside1)) {
                const int64_t c = cell + (second ? 1 : 0);
                const double M = a.gin[c * QG + herm_re_rt<NF>(i)] - (i == 0 ? a.m00 : 0.0);
                const double sum = a.aux[c * NAUX + i];
                v = fmax(fmax(0.5 * (sum + M), 0.5 * (sum - M)), a.m00);
            }
            v = fmax(v, __shfl_xor(v, 1));
            if (NF == 3) v = fmax(v, __shfl_xor(v, 2));
            if (CPW == 2) v = fmax(v, __shfl_xor(v, 32));
            if (lane == 0 && v > 0.0)
                atomicMax(&a.red[DtRed::slot(blockIdx.x)],
                          (unsigned long long)__double_as_longlong(v * a.dtp.vst_scale));
        }
    }
    if constexpr (s == 0) {
        // the end of the step: this launch neither reads the time nor dt, and the
        // maxima are complete (stage 4 has ended)
        if (a.step_end && blockIdx.x == 0 && wave == 0) {
            const double h = next_dt(a.red, a.dtp, a.err);
            if (lane == 0) {
                a.scal[0] = advance_time(a.scal[0], a.scal[1]);
                a.scal[1] = h;
                *a.steps += 1;
            }
        }
    }
    constexpr int GSH = s == 0 ? 0 : (NB * QG * (int)sizeof(T) + 7) / 8; // doubles of the staged box
    constexpr int per_wave = stage_lds_doubles_per_wave<NF, T, AUX>();
    static_assert(per_wave == 64 * 9 + 64 * NSR * (int)sizeof(T) / 8,
                  "LDS layout and its size function disagree");
    constexpr int CT = (NB + 1) / 2;
    // [NB] the box's cell indices: the block's, or this wave's
    int* ctab = (int*)(PM ? lds : lds + wave * CT);
    double* lw = lds + (PM ? CT : WPB * CT);
    // [NB][QG] neighbourhood fields (gather stages): the block's, or this wave's
    T* Gs = (T*)(PM ? lw : lw + wave * (GSH + per_wave));
    double* Wf = PM ? lw + GSH + wave * per_wave : lw + wave * (GSH + per_wave) + GSH; // [64][9] shape factors
    // q_c, vhat (inside_c during the gather): values of the working precision T,
    // so FP32-bulk keeps them as float (lossless) and the LDS per wave shrinks
    T* Src = (T*)(Wf + 64 * 9);             // [64][NSR]
    // the auxiliary sources sit in T in the same rows: in FP32-bulk the products
    // N f are FP32 values already (their sum over particles is accumulated in FP64)
    constexpr int STRIDE = PM ? 64 * WPB : 64;
    const int tid = PM ? (int)threadIdx.x : lane;
    // the box's cell indices, once: the staging loads and the deposit's flush
    // read them instead of redoing the periodic index arithmetic per element
    for (int e = tid; e < NB; e += STRIDE) ctab[e] = (int)box_cell(e);
    if constexpr (PM) {
        __syncthreads();
    } else {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    }
    if constexpr (s != 0) {
        // stage the box's fields, all waves together: NB rows of QG values, in
        // the working precision (FP32-bulk rounds the FP64 deposit here)
        const double* gsrc = a.gin;
        // a compile-time trip count, unrolled, so that every load is in flight at once
#pragma unroll
        for (int e0 = 0; e0 < NB * QG; e0 += STRIDE) {
            const int e = e0 + tid;
            if (e < NB * QG) {
                const int r = e / QG, q = e - r * QG;
                Gs[e] = T(gsrc[(int64_t)ctab[r] * QG + q]);
            }
        }
        if constexpr (PM) {
            __syncthreads();
        } else {
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        }
    }

    const double dt = *a.dt;
    const double bw[4] = {1. / 6., 1. / 3., 1. / 3., 1. / 6.};
    const double cnext[4] = {0.5, 0.5, 1.0, 0.0};

    // lane constants of the deposit's MFMA operands.  A (row t = 16m + l%16):
    // the three shape factors of target t.  B (column q = 16n + l%16): the
    // product of two entries of the particle's source row, the constant 1
    // standing in where a column has one factor.  Row t of the product depends
    // only on row t of A and column q only on column q of B, so the padding
    // rows (t >= NT) and columns (q >= QGA), which are never flushed, read any
    // in-range entries instead of being masked.
    // PACK: in three registers, taken apart once per chunk.  It pays where the
    // twelve crowd the commutators out into scratch memory (FP32-bulk's NF = 3
    // launch with the auxiliaries, 3.33 -> 3.21 ms at 64^3 x 92) or cost a wave per
    // SIMD (its stage 4; FP64's NF = 2 launch with the auxiliaries, 36 -> 33 us at
    // 16^3 x 26); elsewhere the unpacking costs 2 to 4%.
    constexpr bool PACK = sizeof(T) == 4 ? NF == 3 && (AUX != 0 || s == 4) : NF == 2 && AUX != 0 && s != 0;
    unsigned ptdx = 0, pb1 = 0, pb2 = 0; // 4 bits a shape factor, 8 bits a source
    int tdx[MT][3];
    static_assert(3 * MT <= 8, "eight packed factors");
#pragma unroll
    for (int m = 0; m < MT; m++) {
        const int t = 16 * m + (lane & 15);
        const int tc = t < NT ? t : NT - 1;
        const int ii = tc % WX, jj = (tc / WX) % WY, kk = tc / (WX * WY);
        const int f[3] = {WX == 1 ? 1 : ii, 3 + (WY == 1 ? 1 : jj), 6 + (WZ == 1 ? 1 : kk)};
#pragma unroll
        for (int d = 0; d < 3; d++) {
            tdx[m][d] = f[d];
            ptdx |= (unsigned)f[d] << (4 * (3 * m + d));
        }
    }
    WaveGather<NF, T, WX, WY, WZ, PACK, 0, sizeof(T) == 8 || s == 2 || s == 3> gather;
    if constexpr (s != 0) gather.init(lane, [&](int t) __attribute__((always_inline)) { return box_of(t) * QG; });
    // The last columns, when at most 8 remain past the 16-column tiles (NF = 3:
    // 36 = 2 x 16 + 4 without the auxiliaries, 39 = 2 x 16 + 7 with the
    // diagonal ones), run as 4-column tiles on the 4-block 4x4x4 form instead:
    // 16-cycle steps in place of a 64-cycle 16x16x4 step.  With blocks as the
    // row quarters t = 16m + 4b + i, its A operand is lane for lane the 16x16x4
    // one; the B column of small tile k is 16 NTF + 4k + l%4, and its result
    // D[t][q] sits in lane 16i + 4b + j.
    constexpr int QREM = QGA % 16;
    constexpr bool SMALL = QREM != 0 && QREM <= 8;
    constexpr int NTF = QGA / 16 + (SMALL || QREM == 0 ? 0 : 1); // 16-column tiles
    constexpr int NSM = SMALL ? (QREM + 3) / 4 : 0;               // 4-column tiles
    constexpr int NCG = NTF + NSM;                                // column groups of the B operand
    static_assert(NTL == NTF + (SMALL ? 1 : 0), "column tiles");
    static_assert(NCG <= 4, "four packed columns");
    int bi1[NCG], bi2[NCG];
#pragma unroll
    for (int n = 0; n < NCG; n++) {
        int b1 = nh + 3, b2 = nh + 3;
        const int q = n >= NTF ? 16 * NTF + 4 * (n - NTF) + (lane & 3) : 16 * n + (lane & 15);
        if (q < QG) {
            const int f = q / nh, c = q % nh;
            b1 = c;
            b2 = f == 0 ? nh + 3 : nh + f - 1;
        } else if (aux && q < QGA) {
            const int x = q - QG;
            b1 = NSRC + (x < NF ? x : NF + (x - NF) / 3);
            b2 = x < NF ? nh + 3 : nh + (x - NF) % 3;
        }
        bi1[n] = b1;
        bi2[n] = b2;
        pb1 |= (unsigned)b1 << (8 * n);
        pb2 |= (unsigned)b2 << (8 * n);
    }
    mf_d4 acc[MT][NTF];
    double accs[MT][NSM > 0 ? NSM : 1]; // the 4x4x4 tiles
    auto zero_acc = [&]() {
#pragma unroll
        for (int m = 0; m < MT; m++) {
#pragma unroll
            for (int k = 0; k < NSM; k++) accs[m][k] = 0.0;
#pragma unroll
            for (int n = 0; n < NTF; n++) acc[m][n] = mf_d4{0.0, 0.0, 0.0, 0.0};
        }
    };
    zero_acc();
    const bool deposits = s <= 3;
    // The accumulators' deposit to the grid, for the cell whose box offset
    // along x is w (0, or 1 for a wave's second cell).  For the f64 16x16x4
    // product, element r of lane l holds D[16m + 4r + l/16][16n + l%16] (rows
    // interleaved across the four 16-lane groups, unlike the f32 form's
    // 4(l/16) + r).
    auto flush_direct = [&](int w) {
#pragma unroll
        for (int m = 0; m < MT; m++)
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const int t = 16 * m + 4 * r + (lane >> 4);
                if (t >= NT) continue;
                const int64_t tc = ctab[box_of(t) + w];
#pragma unroll
                for (int n = 0; n < NTF; n++) {
                    const int q = 16 * n + (lane & 15);
                    if (q < QG) unsafeAtomicAdd(&a.gout[tc * QG + q], acc[m][n][r]);
                    else if (aux && q < QGA) unsafeAtomicAdd(&a.aux[tc * NAUX + (q - QG)], acc[m][n][r]);
                }
            }
#pragma unroll
        for (int m = 0; m < MT; m++)
#pragma unroll
            for (int k = 0; k < NSM; k++) {
                const int t = 16 * m + 4 * ((lane >> 2) & 3) + (lane >> 4), q = 16 * NTF + 4 * k + (lane & 3);
                if (t >= NT || q >= QGA) continue;
                const int64_t tc = ctab[box_of(t) + w];
                if (q < QG) unsafeAtomicAdd(&a.gout[tc * QG + q], accs[m][k]);
                else unsafeAtomicAdd(&a.aux[tc * NAUX + (q - QG)], accs[m][k]);
            }
    };

    // The wave's particles as a list of slots: the first cell's in 16-particle
    // tiles (its last tile padded), then the second cell's (CPW = 2), so that a
    // tile never mixes cells; 64 slots (four tiles) per chunk.  With one cell
    // this is the cell's run, 64 particles at a time.
    const int n0 = end - beg, n1 = end1 - beg1;
    const int T0 = (n0 + 15) >> 4;        // tiles of the first cell
    const int NSL = 16 * T0 + n1;         // slots in use
    const int bany = n0 > 0 ? beg : beg1; // a particle of the wave, for inactive lanes' loads
    // (one cell: the loop runs over the cell's run itself, base = beg + sbase)
    const int lo = CPW == 1 ? beg : 0, hi = CPW == 1 ? end : NSL;
    int running = 0; // stage 1: lane 27 i + e holds the count of move e from the wave's cell i so far
    int seen = 0;    // (SPLIT: of the workgroup's finished rounds)
    // SPLIT, stage 1: the waves stay together (their ranks follow from each other's
    // counts), so a round runs for all of them; a wave past the end has no active lane
    __shared__ int moves[SPLIT && s == 1 ? WPB * 27 : 1];
    const int first = SPLIT ? 64 * wave : 0;
    for (int base = lo + first; (SPLIT && s == 1 ? base - first : base) < hi; base += SPLIT ? 64 * WPB : 64) {
        const int sbase = base - lo;
        int64_t ip;
        bool act;
        int pcell;
        if constexpr (CPW == 1) {
            ip = base + lane;
            act = ip < end;
            pcell = cell;
        } else {
            const int sl = sbase + lane;
            const bool first = sl < 16 * T0;
            ip = first ? beg + sl : beg1 + (sl - 16 * T0);
            act = first ? sl < n0 : sl < NSL;
            pcell = first ? cell : cell1; // this lane's particle's cell
        }
        const int64_t ipl = act ? ip : (CPW == 1 ? beg : bany); // a valid index for inactive lanes' loads
        double pos[3];
#pragma unroll
        for (int d = 0; d < 3; d++) pos[d] = a.cur.pos[d][ipl];
        const T pupt = a.cur.pup[3][ipl];
        const T pupv[3] = {a.cur.pup[0][ipl], a.cur.pup[1][ipl], a.cur.pup[2][ipl]};
        // the direction and 1/pupt for the fields (within an ulp of the quotients;
        // the position update keeps the exact quotient)
        const T inv_pupt = T(1) / pupt;
        const T vhat[3] = {pupv[0] * inv_pupt, pupv[1] * inv_pupt, pupv[2] * inv_pupt};
        const T N = a.cur.Nn[0][ipl], Nb = a.cur.Nn[1][ipl];
        int idx[3];
        double wd[3][3];
#pragma unroll
        for (int d = 0; d < 3; d++) shape3((pos[d] - g.plo[d]) * g.dxi[d], g.order[d], idx[d], wd[d]);
        // shape factors and directions of the chunk, for the matrix-core operands
        // of the gather and the deposit (positions are frozen within a step)
#pragma unroll
        for (int d = 0; d < 3; d++)
#pragma unroll
            for (int e = 0; e < 3; e++) Wf[lane * 9 + 3 * d + e] = act ? wd[d][e] : 0.0;
#pragma unroll
        for (int d = 0; d < 3; d++) Src[lane * NSR + nh + d] = act ? vhat[d] : T(0);
        Src[lane * NSR + nh + 3] = T(1);
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        // the stage state: y_n (stages 0, 1), Y2 and Y4 in Y, Y3 in the
        // accumulator's array (stage 2 writes it there: see below)
        T Y[2 * nh];
        const T* ysrc = s <= 1 ? a.cur.f : (s == 3 ? a.acc : a.Y);
#pragma unroll
        for (int c = 0; c < 2 * nh; c++) Y[c] = ysrc[(int64_t)c * a.np + ipl];
        T Dep[2 * nh]; // state deposited by this launch
        if constexpr (s == 0) {
#pragma unroll
            for (int c = 0; c < 2 * nh; c++) Dep[c] = Y[c];
        } else {
            // ---- gather on the matrix cores, 16 particles per tile
            T inside[nh];
            const int ntile = CPW == 1 ? (min(64, end - base) + 15) >> 4 : min(4, (NSL + 15 - sbase) >> 4);
            gather.template run<-1>(
                wd, ntile,
                // the tile's cell's neighbourhood: the second cell's box is one column
                // further along x (box rows of QG values)
                [&](int m) __attribute__((always_inline)) { return Gs + (CPW == 2 && (sbase >> 4) + m >= T0 ? QG : 0); },
                [&](int m, T& v0, T& v1, T& v2) __attribute__((always_inline)) {
                    const T* vp = Src + (16 * m + (lane & 15)) * NSR + nh;
                    v0 = vp[0], v1 = vp[1], v2 = vp[2];
                },
                inside);
            // ---- the RK registers this stage reads, as one batch of loads whose
            // latency the Hamiltonian and commutator arithmetic covers
            T yn[2 * nh], ao[2 * nh];
            // The accumulators after stages 1 and 2 are not stored.  With
            // Y2 = y_n + dt/2 k1 and Y3 = y_n + dt/2 k2,
            //   acc1 = y_n + dt/6 k1 = y_n + (Y2 - y_n)/3,
            //   acc2 = acc1 + dt/3 k2 = Y3 + (Y2 - Y3)/3 (y_n cancels; in this
            //   form the rounded 1/3 only scales the small difference, where
            //   Y2/3 + 2 Y3/3 would scale the state by (1/3 + 2/3 rounded) - 1,
            //   3e-8 in FP32, every step),
            // which stages 2 and 3 rebuild from arrays they read: stage 2 keeps
            // Y2 and writes Y3 into the accumulator's array (free until stage 3
            // writes acc3 there), so stage 3 reads y_n, Y2 and Y3.  That saves
            // two writes and a read of the flavour state per step; the change
            // is at rounding level, with multiplies by the rounded 1/3 and 2/3.
            if constexpr (s == 1) {
#pragma unroll
                for (int c = 0; c < 2 * nh; c++) yn[c] = ao[c] = Y[c];
            } else if constexpr (s == 2) {
#pragma unroll
                for (int c = 0; c < 2 * nh; c++) yn[c] = a.cur.f[(int64_t)c * a.np + ipl];
#pragma unroll
                for (int c = 0; c < 2 * nh; c++) ao[c] = yn[c] + (Y[c] - yn[c]) * T(1.0 / 3.0);
            } else if constexpr (s == 3) {
#pragma unroll
                for (int c = 0; c < 2 * nh; c++) yn[c] = a.cur.f[(int64_t)c * a.np + ipl];
#pragma unroll
                for (int c = 0; c < 2 * nh; c++) ao[c] = a.Y[(int64_t)c * a.np + ipl];
#pragma unroll
                for (int c = 0; c < 2 * nh; c++) ao[c] = (ao[c] - Y[c]) * T(1.0 / 3.0) + Y[c];
            } else {
#pragma unroll
                for (int c = 0; c < 2 * nh; c++) yn[c] = s < 4 ? a.cur.f[(int64_t)c * a.np + ipl] : T(0);
#pragma unroll
                for (int c = 0; c < 2 * nh; c++) ao[c] = a.acc[(int64_t)c * a.np + ipl];
            }
            // ---- Hamiltonians / hbar: H = H_vac + coef inside, Hbar = conj(H_vac - coef inside)
            T H[nh], Hb[nh];
#pragma unroll
            for (int c = 0; c < nh; c++) {
                const T hv = T(a.vac[c]) * inv_pupt;
                const T hs = T(a.coef) * inside[c];
                H[c] = hv + hs;
                Hb[c] = is_im_comp<NF>(c) ? hs - hv : hv - hs;
            }
            T k[2 * nh];
            commutator_rhs<NF, T>(H, Y, k, T(1));
            commutator_rhs<NF, T>(Hb, Y + nh, k + nh, T(1));
            const T a_acc = T(dt * bw[s - 1]);
            if constexpr (s < 4) {
                const T a_next = T(dt * cnext[s - 1]);
#pragma unroll
                for (int c = 0; c < 2 * nh; c++) {
                    Dep[c] = a_next * k[c] + yn[c];
                    ao[c] = a_acc * k[c] + ao[c];
                }
                if (act) {
                    // stage 1: Y2 -> Y; stage 2: Y3 -> acc's array; stage 3: acc3 ->
                    // acc, Y4 -> Y (each lane overwrites only the slot it read)
#pragma unroll
                    for (int c = 0; c < 2 * nh; c++) {
                        if (s == 3) a.acc[(int64_t)c * a.np + ip] = ao[c];
                        if (s == 2) a.acc[(int64_t)c * a.np + ip] = Dep[c];
                        else a.Y[(int64_t)c * a.np + ip] = Dep[c];
                    }
                }
                if constexpr (s == 1) {
                    // The sort plan's first part: the particle's move over the step
                    // and its rank among the particles of its cell with that move,
                    // in slot order (lane order within a chunk, chunks in order), so
                    // that the sort is stable.  One pass per move present in the
                    // chunk; most particles stay in their cell, so there are few.
                    int e = 64;
                    if (act) {
                        double v[3], npos[3];
#pragma unroll
                        for (int d = 0; d < 3; d++) v[d] = double(pupv[d]) / double(pupt) * phys::c;
                        end_position(pos, v, dt, g, npos);
                        const int which = CPW == 2 && pcell != cell ? 1 : 0;
                        bool bad = false;
                        const int ex = move1(cx + which, npos[0], g.plo[0], g.dxi[0], g.n[0], bad);
                        const int ey = move1(cy, npos[1], g.plo[1], g.dxi[1], g.n[1], bad);
                        const int ez = move1(cz, npos[2], g.plo[2], g.dxi[2], g.n[2], bad);
                        // only |p| > p_t outruns c dt < dx
                        if (bad) atomicMin(a.err, status_word(a.cur.id[ip], EMU_ERR_MOVE));
                        e = 27 * which + (ez + 1) * 9 + (ey + 1) * 3 + (ex + 1);
                    }
                    int myrank = 0;
                    unsigned long long left = __ballot(act);
                    while (left) {
                        const int q = __builtin_amdgcn_readlane(e, __ffsll((long long)left) - 1);
                        const unsigned long long msk = __ballot(e == q);
                        if (e == q) myrank = __builtin_amdgcn_readlane(running, q) + __popcll(msk & ((1ull << lane) - 1ull));
                        if (lane == q) running += __popcll(msk);
                        left &= ~msk;
                    }
                    if constexpr (SPLIT) {
                        // `running` holds this chunk's counts alone: add those of the
                        // earlier rounds (in `seen`) and of the earlier waves
                        if (lane < 27) moves[27 * wave + lane] = running;
                        __syncthreads();
                        int before = seen;
                        if (lane < 27)
                            for (int w2 = 0; w2 < WPB; w2++) {
                                const int m = moves[27 * w2 + lane];
                                if (w2 < wave) before += m;
                                seen += m;
                            }
                        running = 0;
                        myrank += __shfl(before, e & 31);
                        __syncthreads();
                    }
                    if (act) {
                        a.rank[ip] = myrank;
                        a.mv[ip] = (unsigned char)(e >= 27 ? e - 27 : e);
                    }
                }
            } else if (act) {
                // y_{n+1} = acc + (dt/6) k4, then the post-step hook (main.cpp:155-199):
                // periodic shift, Renormalize in FP64, and the move to the sorted slot
                double y[2 * nh];
#pragma unroll
                for (int c = 0; c < 2 * nh; c++) y[c] = double(a_acc * k[c] + ao[c]);
                const T L = a.cur.Ll[0][ip], Lb = a.cur.Ll[1][ip];
                const int64_t id = a.cur.id[ip];
                int err = renorm_fp64<NF>(y, double(L), a.maxError);
                if (err == EMU_OK) err = renorm_fp64<NF>(y + nh, double(Lb), a.maxError);
                if (err != EMU_OK) atomicMin(a.err, status_word(id, err));
                double v[3], npos[3];
#pragma unroll
                for (int d = 0; d < 3; d++) v[d] = double(pupv[d]) / double(pupt) * phys::c;
                end_position(pos, v, dt, g, npos);
                const int64_t j = (int64_t)a.mbase[(int64_t)pcell * 27 + a.mv[ip]] + a.rank[ip];
                if (j >= 0 && j < a.np) {
#pragma unroll
                    for (int d = 0; d < 3; d++) a.dst.pos[d][j] = npos[d];
#pragma unroll
                    for (int d = 0; d < 3; d++) a.dst.pup[d][j] = pupv[d];
                    a.dst.pup[3][j] = pupt;
                    a.dst.Nn[0][j] = N;
                    a.dst.Nn[1][j] = Nb;
                    a.dst.Ll[0][j] = L;
                    a.dst.Ll[1][j] = Lb;
                    a.dst.id[j] = id;
#pragma unroll
                    for (int c = 0; c < 2 * nh; c++) a.dst.f[(int64_t)c * a.np + j] = T(y[c]);
                } else {
                    atomicMin(a.err, status_word(id, EMU_ERR_MOVE));
                }
            }
        }
        if (!deposits) continue;
        // ---- stage the chunk's deposit sources in LDS (zeros for inactive lanes)
#pragma unroll
        for (int c = 0; c < nh; c++) {
            const T qc = is_im_comp<NF>(c) ? N * Dep[c] + Nb * Dep[nh + c] : N * Dep[c] - Nb * Dep[nh + c];
            Src[lane * NSR + c] = act ? qc : T(0);
        }
        if (aux) {
#pragma unroll
            for (int x = 0; x < NF; x++)
                Src[lane * NSR + NSRC + x] = act ? N * Dep[herm_re<NF>(x, x)] + Nb * Dep[nh + herm_re<NF>(x, x)] : T(0);
            if constexpr (AUX == 2) {
                int o = NF;
#pragma unroll
                for (int x = 0; x < NF; x++)
#pragma unroll
                    for (int y2 = x + 1; y2 < NF; y2++)
                        Src[lane * NSR + NSRC + (o++)] = act ? Nb * Dep[nh + herm_im<NF>(x, y2)] : T(0);
            }
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        // ---- D += W^T R, four particles per MFMA
        // KU k-steps (4 KU particles) per iteration, so the operand reads of one
        // overlap the matrix work of the others: two, and four in FP32-bulk
        // stages 1 to 3 (one tile of 16 slots an iteration, so the second
        // cell's tiles still begin at an iteration; FP64 measured no faster);
        // rows past the chunk's particles hold zero sources (inactive lanes), so
        // rounding the count up is exact.  The deposit-only launch keeps one
        // k-step per iteration: there the registers of the second cost a wave of
        // occupancy, and measured slower.  Each operand has one per-lane LDS
        // pointer that advances by a whole iteration; the later k-steps are
        // immediate offsets.  B is the product in T: in FP32-bulk the flux
        // sources q v are FP32 values like q itself, and the sum over particles
        // stays FP64.
        constexpr int KU = s == 0 ? 1 : (sizeof(T) == 4 ? 4 : 2);
        // (32-bit LDS pointers made opaque once, so that the wave's base is not
        // split off again and re-added to every address in the loop)
        typedef __attribute__((address_space(3))) const double* lds_d;
        typedef __attribute__((address_space(3))) const T* lds_t;
        // k-step iterations (4 KU slots each) up to the chunk's last particle.
        // With two cells, the first cell is complete at the iteration where the
        // second cell's tiles begin (kb, at a tile boundary): its deposit is
        // flushed there and the accumulators start again from zero.
        const int kend = ((CPW == 1 ? min(64, end - base) : min(NSL - sbase, 64)) + 4 * KU - 1) / (4 * KU);
        const int kb = CPW == 2 && n0 > 0 && sbase < n0 && n0 <= sbase + 64 ? (16 * T0 - sbase) / (4 * KU) : -1;
        lds_d wa[MT][3];
        lds_t sb[NCG][2];
        if (PACK) asm volatile("" : "+v"(ptdx), "+v"(pb1), "+v"(pb2)); // taken apart here, not before the loop
#pragma unroll
        for (int m = 0; m < MT; m++)
#pragma unroll
            for (int d = 0; d < 3; d++) {
                wa[m][d] = (lds_d)(Wf + (lane >> 4) * 9 + (PACK ? (int)((ptdx >> (4 * (3 * m + d))) & 15u) : tdx[m][d]));
                asm volatile("" : "+v"(wa[m][d]));
            }
#pragma unroll
        for (int n = 0; n < NCG; n++) {
            sb[n][0] = (lds_t)(Src + (lane >> 4) * NSR + (PACK ? (int)((pb1 >> (8 * n)) & 255u) : bi1[n]));
            sb[n][1] = (lds_t)(Src + (lane >> 4) * NSR + (PACK ? (int)((pb2 >> (8 * n)) & 255u) : bi2[n]));
            asm volatile("" : "+v"(sb[n][0]));
            asm volatile("" : "+v"(sb[n][1]));
        }
#pragma unroll 1
        for (int kp = 0; kp < kend; kp++) {
            if (CPW == 2 && kp == kb) {
                flush_direct(0);
                zero_acc();
            }
#pragma unroll
            for (int h = 0; h < KU; h++) {
                double A[MT];
#pragma unroll
                for (int m = 0; m < MT; m++) A[m] = wa[m][0][36 * h] * wa[m][1][36 * h] * wa[m][2][36 * h];
#pragma unroll
                for (int n = 0; n < NCG; n++) {
                    const double B = double(sb[n][0][4 * NSR * h] * sb[n][1][4 * NSR * h]);
                    if (n >= NTF) {
#pragma unroll
                        for (int m = 0; m < MT; m++)
                            accs[m][n - NTF] = __builtin_amdgcn_mfma_f64_4x4x4f64(A[m], B, accs[m][n - NTF], 0, 0, 0);
                    } else {
#pragma unroll
                        for (int m = 0; m < MT; m++)
                            acc[m][n] = __builtin_amdgcn_mfma_f64_16x16x4f64(A[m], B, acc[m][n], 0, 0, 0);
                    }
                }
            }
#pragma unroll
            for (int m = 0; m < MT; m++)
#pragma unroll
                for (int d = 0; d < 3; d++) wa[m][d] += 36 * KU;
#pragma unroll
            for (int n = 0; n < NCG; n++) {
                sb[n][0] += 4 * NSR * KU;
                sb[n][1] += 4 * NSR * KU;
            }
        }
        if (CPW == 2 && kb == kend) {
            flush_direct(0);
            zero_acc();
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    }
    if constexpr (s == 1) {
        if (owner && lane < (inside1 ? 54 : 27)) a.mcount[(int64_t)cell * 27 + lane] = SPLIT ? seen : running;
    }
    if (!deposits) return;
    if constexpr (!PM) {
        // ---- flush this wave's (last) cell's deposit straight to the grid
        if constexpr (CPW == 2) {
            if (n1 > 0) flush_direct(1);
            return;
        }
        if (end <= beg) return;
        flush_direct(0);
        return;
    }
    // ---- merge the waves' deposits over the box in LDS, then flush
    double* Mb = lw; // [NB][QGA], over the staged box and the waves' regions (not the cell table)
    __syncthreads();
    for (int e = threadIdx.x; e < NB * QGA; e += 64 * WPB) Mb[e] = 0.0;
    __syncthreads();
    if (end > beg) {
#pragma unroll
        for (int m = 0; m < MT; m++)
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const int t = 16 * m + 4 * r + (lane >> 4);
                if (t >= NT) continue;
                const int bi = box_of(t);
#pragma unroll
                for (int n = 0; n < NTF; n++) {
                    const int q = 16 * n + (lane & 15);
                    if (q < QGA) unsafeAtomicAdd(&Mb[bi * QGA + q], acc[m][n][r]);
                }
            }
#pragma unroll
        for (int m = 0; m < MT; m++)
#pragma unroll
            for (int k = 0; k < NSM; k++) {
                const int t = 16 * m + 4 * ((lane >> 2) & 3) + (lane >> 4), q = 16 * NTF + 4 * k + (lane & 3);
                if (t < NT && q < QGA) unsafeAtomicAdd(&Mb[box_of(t) * QGA + q], accs[m][k]);
            }
    }
    __syncthreads();
    for (int e = threadIdx.x; e < NB * QGA; e += 64 * WPB) {
        const double v = Mb[e];
        if (v == 0.0) continue;
        const int bi = e / QGA, q = e - bi * QGA;
        const int64_t tc = ctab[bi];
        if (q < QG) unsafeAtomicAdd(&a.gout[tc * QG + q], v);
        else unsafeAtomicAdd(&a.aux[tc * NAUX + (q - QG)], v);
    }
}

} // namespace emu
