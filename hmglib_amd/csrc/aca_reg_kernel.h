// aca_reg_kernel.h -- the kernels of aca_reg.h, instantiated by one translation unit
// per kernel kind.
#pragma once
#include <utility>

#include "aca_reg.h"

namespace hmg {
namespace {

// wavefronts per SIMD of a team with nt rank terms in registers (64 or 32 registers of
// them and about 85 for the points and the evaluation)
constexpr int reg_waves(int nt) { return nt == 8 ? 4 : 3; }

// rank terms 0 .. NT-1 of one row of U or of one column's row of V (every access at a
// constant index: registers)
template <int NT>
struct RegRow {
    double t[NT];
};

// f(0), f(1), ... f(N - 1) with constant indices, so that arrays indexed by them stay in
// registers
template <int... I, class F>
__device__ __forceinline__ void static_for_impl(std::integer_sequence<int, I...>, F&& f)
{
    (f(std::integral_constant<int, I>{}), ...);
}
template <int N, class F>
__device__ __forceinline__ void static_for(F&& f)
{
    static_for_impl(std::make_integer_sequence<int, N>{}, f);
}

// double through a DPP lane permutation
template <int CTRL>
__device__ __forceinline__ double dpp(double v)
{
    const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(v), CTRL, 0xf, 0xf, false);
    const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(v), CTRL, 0xf, 0xf, false);
    return __hiloint2double(hi, lo);
}
__device__ __forceinline__ double lane_of(double v, int l)
{
    return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(v), l),
                            __builtin_amdgcn_readlane(__double2loint(v), l));
}
// quad permutations (lane ^ 1, lane ^ 2), half mirror and mirror pair up the 16 lanes of
// a row; the four rows' values are read from one lane each
template <class F>
__device__ __forceinline__ double wave_reduce(double v, F f)
{
    v = f(v, dpp<0xB1>(v));
    v = f(v, dpp<0x4E>(v));
    v = f(v, dpp<0x141>(v));
    v = f(v, dpp<0x140>(v));
    return f(f(lane_of(v, 0), lane_of(v, 16)), f(lane_of(v, 32), lane_of(v, 48)));
}
__device__ __forceinline__ double wave_add(double v)
{
    return wave_reduce(v, [](double x, double y) { return x + y; });
}
__device__ __forceinline__ double wave_max(double v)
{
    return wave_reduce(v, [](double x, double y) { return fmax(x, y); });
}
__device__ __forceinline__ double wave_min(double v)
{
    return wave_reduce(v, [](double x, double y) { return fmin(x, y); });
}

template <int KIND>
constexpr bool reg_monotone()
{
    return KIND == HMG_KERNEL_GAUSSIAN || KIND == HMG_KERNEL_EXPONENTIAL || KIND == HMG_KERNEL_GAUSSIAN_REF;
}

// ---- the search for the next acceptable row ------------------------------------------
// kSearchRows rows at a time, one per lane, against all columns, TILE at a time through
// LDS; the NW wavefronts share out the columns of a tile.  A lane holds its row's U terms
// in registers.  An entry is formed exactly as a rank step forms it; only the order of
// the norm's sum differs, so a row is passed over only when its norm is below the
// threshold by more than any order's rounding (2e-9 relative), and the rank step
// evaluates the row that is found once more.  The columns of a tile whose bound
//   sqrt(TILE) (k(d) + sum_l |U(i,l)|),  d the distance to the tile's box, |V| <= 1
// (v_r is scaled by its largest entry) is small against the threshold are not evaluated;
// the bounds of such tiles are added up instead (k decreasing, no regularization).
// Bound by the evaluations (one block of 16900 rows and columns that rejects nearly all
// of them: 2 ms on the whole chip).  A chunk of one block would keep a single compute unit
// busy for 200 us at 3500 columns; in eight column segments it takes 25.
constexpr int kSearchTerms = 32;  // U terms in registers; later ones are read per column
constexpr int kSearchWaves = 8;   // wavefronts and tile of the search over suspended blocks
constexpr int kSearchTile = 64;
static_assert(kSearchRows == kWave, "one row per lane");

template <int DIM, int NW, int TILE>
struct SearchShared {
    double v[TILE][kSearchTerms];
    double x[DIM][TILE];
    double box[2][DIM];
    double acc[NW][kWave];
    int found;
};

// The first row of first .. first + 63 of block b that may be acceptable at rank step r
// (b's row count when there is none), by the columns of segment seg of nseg: a row whose
// norm is at the threshold has at least one segment with its share of it.  found: a row
// that others may lower meanwhile; rows past it are not searched.  Every thread returns the same row.
template <int KIND, int DIM, int NW, int TILE>
__device__ __forceinline__ int search_rows(const AcaArgs& g, const int4 b, const int first, const int r,
                                           const double* __restrict__ Ub, const int64_t lu,
                                           const double* __restrict__ Vb, const int64_t lv,
                                           SearchShared<DIM, NW, TILE>& sh, const int* found, const int seg,
                                           const int nseg)
{
    const int tid = threadIdx.x, lane = tid % kWave;
    const int w = __builtin_amdgcn_readfirstlane(tid / kWave);
    const int l1 = b.x, m1 = b.y - b.x + 1;
    const int l2 = b.z, m2 = b.w - b.z + 1;
    const KernelParams kp = g.kp;
    const int i = min(first + lane, m1 - 1);
    double u[kSearchTerms], su = 0.0, x[DIM];
#pragma unroll
    for (int l = 0; l < kSearchTerms; l++) {
        u[l] = l < r ? Ub[l * lu + i] : 0.0;
        su += fabs(u[l]);
    }
    for (int l = kSearchTerms; l < r; l++) su += fabs(Ub[l * lu + i]);
#pragma unroll
    for (int d = 0; d < DIM; d++) x[d] = g.c1.x[d][l1 + i];
    const bool diag = kp.reg != 0.0 && l1 <= b.w && l2 <= b.y;
    const bool prune = reg_monotone<KIND>() && !diag;
    const double thr2 = 1.0e-26 * (1.0 - 4e-9) / nseg;
    // a tile may be left out when its bound squared is below this share
    const double share = 0.0625e-26 / ((m2 + TILE - 1) / TILE);
    double acc = 0.0;
    bool live = first + lane < m1;  // these three: the same in all wavefronts
    uint64_t hits = 0;
    const int span = ((m2 + TILE - 1) / TILE + nseg - 1) / nseg * TILE;  // columns of a segment
    const int jend = min(m2, (seg + 1) * span);
    for (int j0 = seg * span; j0 < jend; j0 += TILE) {
        const int nc = min(TILE, m2 - j0);
        __syncthreads();
        if (tid == 0) sh.found = __hip_atomic_load(found, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        for (int q = tid; q < TILE * kSearchTerms; q += NW * kWave) {
            const int jj = q / kSearchTerms, l = q % kSearchTerms;
            sh.v[jj][l] = (l < r && jj < nc) ? Vb[(int64_t)(j0 + jj) * lv + l] : 0.0;
        }
        if (w == 0) {
            const int j = l2 + j0 + min(lane, nc - 1);
#pragma unroll
            for (int d = 0; d < DIM; d++) {
                const double y = g.c2.x[d][j];
                if (lane < TILE) sh.x[d][lane] = y;
                const double lo = wave_min(y), hi = wave_max(y);
                if (lane == 0) {
                    sh.box[0][d] = lo;
                    sh.box[1][d] = hi;
                }
            }
        }
        __syncthreads();
        if (i > sh.found) live = false;  // an earlier row was found already
        bool eval = live;
        double part = 0.0;
        if (prune && live) {
            double r2 = 0.0;
#pragma unroll
            for (int d = 0; d < DIM; d++) {
                const double gap = fmax(0.0, fmax(sh.box[0][d] - x[d], x[d] - sh.box[1][d]));
                r2 += gap * gap;
            }
            const double bound = (kernel_of_r2_k<KIND>(kp, r2 * (1.0 - 1e-9)) + su) * (1.0 + 1e-9);
            const double b2 = TILE * bound * bound;
            eval = !(b2 < share);
            if (!eval && w == 0) part = b2;
        }
        if (eval) {
            const int c1 = min(nc, (w + 1) * (TILE / NW));
            for (int jj = w * (TILE / NW); jj < c1; jj++) {
                double r2 = 0.0;
#pragma unroll
                for (int d = 0; d < DIM; d++) {
                    const double t = x[d] - sh.x[d][jj];
                    r2 = __dadd_rn(r2, __dmul_rn(t, t));
                }
                double val = kernel_of_r2_k<KIND>(kp, r2);
                if (diag && l1 + i == l2 + j0 + jj) val += kp.reg;
#pragma unroll
                for (int q0 = 0; q0 < kSearchTerms; q0 += 8) {
                    if (r > q0) {
#pragma unroll
                        for (int l = q0; l < q0 + 8; l++) val = __fma_rn(-u[l], sh.v[jj][l], val);
                    }
                }
                for (int l = kSearchTerms; l < r; l++)
                    val = __fma_rn(-Ub[l * lu + i], Vb[(int64_t)(j0 + jj) * lv + l], val);
                part = __fma_rn(val, val, part);
            }
        }
        sh.acc[w][lane] = part;
        __syncthreads();
        for (int q = 0; q < NW; q++) acc += sh.acc[q][lane];
        // NaN sums are rejected rows (their norm is not at or above the threshold)
        const bool hit = live && acc >= thr2;
        hits |= __ballot(hit);
        // rows past the first hit need no search
        live = live && !hit && (hits == 0 || lane < __builtin_ctzll(hits));
        if (__ballot(live) == 0) break;
    }
    __syncthreads();
    return hits ? first + __builtin_ctzll(hits) : m1;
}

constexpr int kRegAhead = 4;   // rows tried together after a rejected one

template <int NW, int DIM>
struct RegShared {
    double u[kRegRank];      // U terms of the row being evaluated, and its point
    double xu[DIM];
    double v[kRegRank];      // V terms of the pivot column, and its point
    double xv[DIM];
    double red[NW];          // team reductions
    double best[NW], bval[NW];
    int bj[NW];
    double ext[NW];
    // rows tried together after a rejected one: their U terms, points and norms
    double tu[kRegAhead][kRegRank];
    double tx[kRegAhead][DIM];
    double tn[kRegAhead][NW];
    double g[NW][kRegRank];  // v_l . v_r (tolerance stop)
    int item;
};

// Where one side's factor terms past the registers are: LDS (t, one kRegSlots * TS wide
// row per term) for the next kRegTail terms, then the factor's storage: term l of the
// slot's row or column i[c] (past the block's end: its last one) at p + i[c] * si + l * sp.
struct RegTail {
    double* t;
    double* p;
    int i[kRegSlots];
    int64_t si, sp;
    __device__ double* at(int c, int l) const { return p + i[c] * si + l * sp; }
};

// val[c] -= sum_{l < r} s[l] f[c][l] in l order.  Terms are taken eight at a time up to
// the end of the LDS ones; those at or past r are zero on both sides and change nothing.
template <int TS, int NT>
__device__ __forceinline__ void reg_chain(double (&val)[kRegSlots], const RegRow<NT> (&f)[kRegSlots],
                                          const double* s, int r, const RegTail& q)
{
    static_for<NT / 8>([&](auto h) {
        if (r > 8 * h)
            static_for<8>([&](auto e) {
                constexpr int l = 8 * h + e;
                static_for<kRegSlots>([&](auto c) { val[c] = __fma_rn(-s[l], f[c].t[l], val[c]); });
            });
    });
    if (r > NT) {
#pragma unroll
        for (int l = 0; l < kRegTail; l++)
#pragma unroll
            for (int c = 0; c < kRegSlots; c++)
                val[c] = __fma_rn(-s[NT + l], q.t[(l * kRegSlots + c) * TS], val[c]);
        for (int l = NT + kRegTail; l < r; l++)
#pragma unroll
            for (int c = 0; c < kRegSlots; c++) val[c] = __fma_rn(-s[l], *q.at(c, l), val[c]);
    }
}

// term r (uniform) of slot c becomes x (has: the slot's row or column exists)
template <int TS, int NT>
__device__ __forceinline__ void reg_store(RegRow<NT>& f, int c, int r, double x, bool has, const RegTail& q)
{
    static_for<NT / 4>([&](auto h) {
        if ((r >> 2) == h) {
            static_for<4>([&](auto e) {
                constexpr int l = 4 * h + e;
                f.t[l] = l == r ? x : f.t[l];
            });
            // an empty statement that differs from group to group: the compiler would
            // otherwise merge the groups' stores into one at a variable index, and the
            // array would leave the registers
            asm volatile("; terms %0" ::"i"(4 * (int)h));
        }
    });
    if (r >= NT) {
        if (r < NT + kRegTail)
            q.t[((r - NT) * kRegSlots + c) * TS] = x;
        else if (has)
            *q.at(c, r) = x;
    }
}

// term l past the registers of slot c
template <int TS, int NT>
__device__ __forceinline__ double reg_tail(int c, int l, const RegTail& q)
{
    return l < NT + kRegTail ? q.t[((l - NT) * kRegSlots + c) * TS] : *q.at(c, l);
}

// terms 0 .. r-1 of slot c (uniform) to LDS, in whole groups of eight up to the LDS ones
// (zeros past r); the slots are selected by value, not by address, so that they stay in
// registers
template <int TS, int NT>
__device__ __forceinline__ void reg_publish(double* s, const RegRow<NT> (&f)[kRegSlots], int c, int r, const RegTail& q)
{
    static_for<NT / 8>([&](auto h) {
        if (h == 0 || r > 8 * h)
            static_for<8>([&](auto e) {
                const double x = f[0].t[8 * h + e], y = f[kRegSlots - 1].t[8 * h + e];
                s[8 * h + e] = c == 0 ? x : y;
            });
    });
    if (r > NT) {
#pragma unroll
        for (int l = 0; l < kRegTail; l++) s[NT + l] = q.t[(l * kRegSlots + c) * TS];
        for (int l = NT + kRegTail; l < r; l++) s[l] = q.p[(int64_t)(c == 0 ? q.i[0] : q.i[kRegSlots - 1]) * q.si + l * q.sp];
    }
}

// Bound by latency: a rank step is a chain of two evaluations, two residual chains, four
// barriers and two reductions, about 10^4 cycles for a team alone on its compute unit
// (0.36 of the SIMDs' issue slots), so what counts is how many teams a compute unit holds.
// NT = 16: 64 registers of factor terms, three wavefronts per SIMD, ranks up to 24 on
// chip.  NT = 8: four per SIMD (115 registers), ranks up to 16 on chip, later terms from
// cache.  Of N = 262144 points in 3D, leaf 256, k = 24 (exponential): blocks up to 512 take
// 0.25 us each on 8 wavefronts (two teams per compute unit) against 0.42 on 9 (one), up
// to 320 0.21 on 5 with NT = 8 against 0.28 with 16, up to 256 0.11 on 4.  The whole build
// runs 54 ms of these kernels; the memory form took 150.  No variant of this kernel uses
// scratch memory.
template <int KIND, int DIM, bool TOL, int NW, int NT>
__global__ void __launch_bounds__(NW* kWave) __attribute__((amdgpu_waves_per_eu(reg_waves(NT), reg_waves(NT))))
aca_reg_kernel(AcaArgs g)
{
    __shared__ RegShared<NW, DIM> sh;
    extern __shared__ double tails[];
    if (g.resume && (int)blockIdx.x >= *g.count) return;
    const int a = g.list[blockIdx.x];
    constexpr int TS = NW * kWave;
    constexpr int R = kRegSlots;
    constexpr int SPAN = R * TS;
    const int tid = threadIdx.x;
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const int lane = threadIdx.x % kWave;
    const int4 b = g.blk[a];
    const int k = g.kb[a];
    const int l1 = b.x, m1 = b.y - b.x + 1;
    const int l2 = b.z, m2 = b.w - b.z + 1;
    const KernelParams kp = g.kp;
    double* const Ub = g.ublk ? g.ublk[a] : g.U + g.uoff[a];
    double* const Vb = g.vblk ? g.vblk[a] : g.V + g.voff[a];
    const int64_t lu = g.ldu[a], lv = g.ldv[a];

    // this thread's rows and columns; past the block's end: its last ones, which take
    // part in no reduction and are not written
    double xu[R][DIM], xv[R][DIM];
    bool hu[R], hv[R];
    RegTail qu, qv;
    qu.t = tails + tid;
    qv.t = tails + kRegTail * SPAN + tid;
    qu.p = Ub;
    qu.si = 1;
    qu.sp = lu;
    qv.p = Vb;
    qv.si = lv;
    qv.sp = 1;
#pragma unroll
    for (int c = 0; c < R; c++) {
        hu[c] = tid + c * TS < m1;
        hv[c] = tid + c * TS < m2;
        qu.i[c] = hu[c] ? tid + c * TS : m1 - 1;
        qv.i[c] = hv[c] ? tid + c * TS : m2 - 1;
#pragma unroll
        for (int d = 0; d < DIM; d++) {
            xu[c][d] = g.c1.x[d][l1 + qu.i[c]];
            xv[c][d] = g.c2.x[d][l2 + qv.i[c]];
        }
    }
    // team extreme and sum of one value (every thread ends with the same one)
    auto team_extreme = [&](double v, bool mx) {
        v = mx ? wave_max(v) : wave_min(v);
        if (NW == 1) return v;
        if (lane == 0) sh.ext[w] = v;
        __syncthreads();
        double t = sh.ext[0];
#pragma unroll 4
        for (int q = 1; q < NW; q++) t = mx ? fmax(t, sh.ext[q]) : fmin(t, sh.ext[q]);
        __syncthreads();
        return t;
    };
    auto team_sum = [&](double v) {
        v = wave_add(v);
        if (NW == 1) return v;
        if (lane == 0) sh.ext[w] = v;
        __syncthreads();
        double t = 0.0;
#pragma unroll 4
        for (int q = 0; q < NW; q++) t += sh.ext[q];
        __syncthreads();
        return t;
    };
    const bool diag = kp.reg != 0.0 && l1 <= b.w && l2 <= b.y;  // some entry carries the regularization
    auto entry = [&](const double* x, const double* y, int i, int j) {
        double r2 = 0.0;
#pragma unroll
        for (int d = 0; d < DIM; d++) {
            const double t = x[d] - y[d];
            r2 = __dadd_rn(r2, __dmul_rn(t, t));
        }
        double e = kernel_of_r2_k<KIND>(kp, r2);
        if (diag && i == j) e += kp.reg;
        return e;
    };
    // a block whose entries are all too small for any row to pass the search gets rank
    // 0 without evaluation (the rule and its margins: block_negligible, aca.hip)
    if (g.scan && !g.resume && k > 0 && reg_monotone<KIND>() && !diag) {
        const work_item& wi = g.items[a];
        double r2 = 0.0;
#pragma unroll
        for (int d = 0; d < DIM; d++) {
            const double gap = fmax(0.0, fmax(wi.min1[d] - wi.max2[d], wi.min2[d] - wi.max1[d]));
            r2 += gap * gap;
        }
        const double sm2 = sqrt((double)m2);
        if (!(sm2 * kernel_of_r2_k<KIND>(kp, 0.5 * r2) >= 0.5e-13)) {
            r2 = 0.0;
#pragma unroll
            for (int d = 0; d < DIM; d++) {
                double lo1 = fmin(xu[0][d], xu[R - 1][d]), hi1 = fmax(xu[0][d], xu[R - 1][d]);
                double lo2 = fmin(xv[0][d], xv[R - 1][d]), hi2 = fmax(xv[0][d], xv[R - 1][d]);
                lo1 = team_extreme(lo1, false);
                hi1 = team_extreme(hi1, true);
                lo2 = team_extreme(lo2, false);
                hi2 = team_extreme(hi2, true);
                const double gap = fmax(0.0, fmax(lo1 - hi2, lo2 - hi1));
                r2 += gap * gap;
            }
            if (sm2 * kernel_of_r2_k<KIND>(kp, r2 * (1.0 - 1e-9)) < 0.5e-13) {
                if (tid == 0) g.keff[a] = 0;
                return;
            }
        }
    }

    int i_r = -1, r0 = 0;
    double fro2 = 0.0;
    if (g.resume) {
        i_r = g.found[a] - 1;
        if (i_r >= m1 - 1) return;  // no acceptable row was left: the block is complete
        r0 = g.keff[a];
        fro2 = g.fro2[a];
    }
    RegRow<NT> u[R], v[R];
    static_for<R>([&](auto c) {
        static_for<NT>([&](auto l) {
            double x = 0.0, y = 0.0;
            if (l < r0) {
                x = *qu.at(c, l);
                y = *qv.at(c, l);
            }
            u[c].t[l] = x;
            v[c].t[l] = y;
        });
        if (k > NT) {
            for (int l = 0; l < kRegTail; l++) {
                const bool set = NT + l < r0;
                qu.t[(l * R + c) * TS] = set ? *qu.at(c, NT + l) : 0.0;
                qv.t[(l * R + c) * TS] = set ? *qv.at(c, NT + l) : 0.0;
            }
        }
    });
    // row i's U terms and point for everybody (after the barrier)
    auto publish_row = [&](int i, int r) {
        if (tid == i % TS) {
            const int c = i / TS;
            reg_publish<TS, NT>(sh.u, u, c, r, qu);
            static_for<DIM>([&](auto d) {
                const double x = xu[0][d], y = xu[R - 1][d];
                sh.xu[d] = c == 0 ? x : y;
            });
        }
        __syncthreads();
    };
    int ke = r0;
    bool suspended = false;
    bool met = false;  // the tolerance
    for (int r = r0; r < k && !met; r++) {
        double val[R];
        int jr = -1;
        double p = 0.0;
        bool stop = false;
        int tries = 0;
        for (;;) {
            if (i_r >= m1 - 1) {
                stop = true;
                break;
            }
            i_r++;
            publish_row(i_r, r);
#pragma unroll
            for (int c = 0; c < R; c++)
                val[c] = (c == 0 || c * TS + w * kWave < m2) ? entry(sh.xu, xv[c], l1 + i_r, l2 + tid + c * TS) : 0.0;
            reg_chain<TS, NT>(val, v, sh.u, r, qv);
            double nw = 0.0;
#pragma unroll
            for (int c = 0; c < R; c++)
                if (hv[c]) nw = __fma_rn(val[c], val[c], nw);
            // the wavefront's column-pivot candidate: largest |value|, the last (first)
            // of equal ones
            double best = -1.0, bval = 0.0;
            int bj = -1;
#pragma unroll
            for (int c = 0; c < R; c++) {
                const double ax = fabs(val[c]);
                if (hv[c] && (g.tie_last ? ax >= best : ax > best)) {
                    best = ax;
                    bval = val[c];
                    bj = tid + c * TS;
                }
            }
            nw = wave_add(nw);
            const double wb = wave_max(best);
            uint64_t mask = __ballot(best == wb);
            if (mask & (mask - 1)) {  // equal candidates: the last (first) index
                const double cj = best == wb ? (double)bj : g.tie_last ? -1.0 : 1e300;
                const double pick = g.tie_last ? wave_max(cj) : wave_min(cj);  // by every lane
                mask = __ballot(cj == pick);
            }
            const int wl = __builtin_ctzll(mask);
            const int wj = __builtin_amdgcn_readlane(bj, wl);
            const double wv = lane_of(bval, wl);
            double nrm = nw;
            jr = wj;
            p = wv;
            if (NW > 1) {
                if (lane == 0) {
                    sh.red[w] = nw;
                    sh.best[w] = wb;
                    sh.bval[w] = wv;
                    sh.bj[w] = wj;
                }
                __syncthreads();
                nrm = 0.0;
#pragma unroll 4
                for (int q = 0; q < NW; q++) nrm += sh.red[q];
                double bb = sh.best[0];
                jr = sh.bj[0];
                p = sh.bval[0];
#pragma unroll 4
                for (int q = 1; q < NW; q++) {
                    const double ob = sh.best[q];
                    const int oj = sh.bj[q];
                    if (ob > bb || (ob == bb && (g.tie_last ? oj > jr : (oj < jr && oj >= 0)))) {
                        bb = ob;
                        jr = oj;
                        p = sh.bval[q];
                    }
                }
                // the same in every thread: scalars, so that the branches are scalar too
                nrm = lane_of(nrm, 0);
                jr = __builtin_amdgcn_readlane(jr, 0);
                p = lane_of(p, 0);
            }
            if (sqrt(nrm) >= 1.0e-13) break;
            // a search that does not end within a few rows goes to the search over all
            // suspended blocks
            // the norms of the next rows, together: rejected rows come in runs
            const int n = min(kRegAhead, m1 - 1 - i_r);
            for (int q = 0; q < n; q++) {
                if (tid == (i_r + 1 + q) % TS) {
                    reg_publish<TS, NT>(sh.tu[q], u, (i_r + 1 + q) / TS, r, qu);
                    static_for<DIM>([&](auto d) { sh.tx[q][d] = xu[0][d]; });
                }
            }
            __syncthreads();
            for (int q = 0; q < n; q++) {
                double t[R] = {entry(sh.tx[q], xv[0], l1 + i_r + 1 + q, l2 + tid)};
                reg_chain<TS, NT>(t, v, sh.tu[q], r, qv);
                const double t2 = wave_add(hv[0] ? __fma_rn(t[0], t[0], 0.0) : 0.0);
                if (lane == 0) sh.tn[q][w] = t2;
            }
            __syncthreads();
            int skip = 0;
            for (; skip < n; skip++) {
                double t = 0.0;
                if (NW == 1) t = sh.tn[skip][0];
                if (NW > 1)
#pragma unroll 4
                    for (int q = 0; q < NW; q++) t += sh.tn[skip][q];
                if (sqrt(lane_of(t, 0)) >= 1.0e-13) break;
            }
            i_r += skip;
            tries += 1 + skip;
            if (g.suspend && tries >= g.tries && skip == n) {
                suspended = i_r < m1 - 1;
                stop = true;
                break;
            }
        }
        if (stop) break;
        // the pivot column's V terms and point for everybody, v_r = row / pivot
        if (tid == jr % TS) {
            const int c = jr / TS;
            reg_publish<TS, NT>(sh.v, v, c, r, qv);
            static_for<DIM>([&](auto d) {
                const double x = xv[0][d], y = xv[R - 1][d];
                sh.xv[d] = c == 0 ? x : y;
            });
        }
        static_for<R>([&](auto c) {
            val[c] = val[c] / p;
            reg_store<TS, NT>(v[c], c, r, val[c], hv[c], qv);
        });
        double nu = 0.0, nv = 0.0;  // ||u_r||^2, ||v_r||^2 (tolerance stop)
        __syncthreads();
        double uv[R];
#pragma unroll
        for (int c = 0; c < R; c++)
            uv[c] = (c == 0 || c * TS + w * kWave < m1) ? entry(xu[c], sh.xv, l1 + tid + c * TS, l2 + jr) : 0.0;
        reg_chain<TS, NT>(uv, u, sh.v, r, qu);
        static_for<R>([&](auto c) { reg_store<TS, NT>(u[c], c, r, uv[c], hu[c], qu); });
        ke = r + 1;
        if (TOL) {
            // ||U V^T||_F^2 gains 2 u_r . (U (V^T v_r)) + ||u_r||^2 ||v_r||^2: the dot
            // products v_l . v_r (l < r), then one chain over this thread's U terms
#pragma unroll
            for (int c = 0; c < R; c++) {
                if (hu[c]) nu = __fma_rn(uv[c], uv[c], nu);
                if (!hv[c]) val[c] = 0.0;
                nv = __fma_rn(val[c], val[c], nv);
            }
            auto dots = [&](int l0, double (&q)[4]) {
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    q[e] = wave_add(q[e]);
                    if (lane == 0) sh.g[w][l0 + e] = q[e];
                }
            };
            static_for<NT / 4>([&](auto h) {
                if (4 * h < r) {
                    double q[4];
                    static_for<4>([&](auto e) {
                        q[e] = 0.0;
                        static_for<R>([&](auto c) { q[e] = __fma_rn(v[c].t[4 * h + e], val[c], q[e]); });
                    });
                    dots(4 * h, q);
                }
            });
            for (int l0 = NT; l0 < r; l0 += 4) {
                double q[4];
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    q[e] = 0.0;
                    if (l0 + e < r) {
#pragma unroll
                        for (int c = 0; c < R; c++) q[e] = __fma_rn(reg_tail<TS, NT>(c, l0 + e, qv), val[c], q[e]);
                    }
                }
                dots(l0, q);
            }
            __syncthreads();
            double cross = 0.0;
            if (NW > 1) {
                // the team's sums, formed once
                for (int l = tid; l < r; l += TS) {
                    double x = 0.0;
#pragma unroll 4
                    for (int q = 0; q < NW; q++) x += sh.g[q][l];
                    sh.g[0][l] = x;
                }
                __syncthreads();
            }
            double t[R];
#pragma unroll
            for (int c = 0; c < R; c++) t[c] = 0.0;
            static_for<NT / 4>([&](auto h) {
                if (4 * h < r)
                    static_for<4>([&](auto e) {
                        const double gl = 4 * h + e < r ? sh.g[0][4 * h + e] : 0.0;
                        static_for<R>([&](auto c) { t[c] = __fma_rn(u[c].t[4 * h + e], gl, t[c]); });
                    });
            });
            for (int l = NT; l < r; l++)
#pragma unroll
                for (int c = 0; c < R; c++) t[c] = __fma_rn(reg_tail<TS, NT>(c, l, qu), sh.g[0][l], t[c]);
#pragma unroll
            for (int c = 0; c < R; c++)
                if (hu[c]) cross = __fma_rn(t[c], uv[c], cross);
            nu = team_sum(nu);
            nv = team_sum(nv);
            cross = team_sum(cross);
            fro2 = fro2 + 2.0 * cross + nu * nv;
            const bool m = (g.tol.mode == 2 || r % 5 == 0) && sqrt(nu) * sqrt(nv) <= g.tol.c * sqrt(fmax(fro2, 0.0));
            met = __builtin_amdgcn_readfirstlane(m ? 1 : 0) != 0;
        }
    }
    // the factors: U_b column-major (lanes along a column), V_b row-major (a thread
    // writes its columns' contiguous rows); terms past the LDS ones are there already
    static_for<R>([&](auto c) {
        if (hu[c]) {
            static_for<NT>([&](auto l) {
                if (l < ke) *qu.at(c, l) = u[c].t[l];
            });
            for (int l = NT; l < min(ke, NT + kRegTail); l++)
                *qu.at(c, l) = qu.t[((l - NT) * R + c) * TS];
        }
        if (hv[c]) {
            static_for<NT>([&](auto l) {
                if (l < ke) *qv.at(c, l) = v[c].t[l];
            });
            for (int l = NT; l < min(ke, NT + kRegTail); l++)
                *qv.at(c, l) = qv.t[((l - NT) * R + c) * TS];
        }
    });
    if (tid == 0) {
        g.keff[a] = ke;
        if (suspended) {
            g.row[a] = i_r;
            g.found[a] = m1;
            g.fro2[a] = fro2;
            g.queue[atomicAdd(g.queued, 1)] = a;
        }
    }
}

// ---- wide blocks -------------------------------------------------------------------
// Blocks wider than the largest register team: a workgroup of NW wavefronts, U in U_b
// and V column-major in the workgroup's slab (term l of column j at vt[l * m2 + j]), so
// that every factor read is a run of consecutive values, four columns (rows) per
// thread at a time with eight terms of each in flight.  The slab is written to V_b at the end.
// Bound by those reads (ranks^2 / 2 terms per row, past the L2 for many blocks at once):
// about 9 TB/s at N = 262144 in 3D, 22 ms of that build.  At three wavefronts per SIMD (168
// registers) the variants spill 4 to 12 of them (20 to 52 bytes a lane of scratch memory).
// Sums over columns or rows are formed as a team of kWideWaves wavefronts forms them (one
// partial sum per thread of such a team, reduced per wavefront, added in order), whatever
// NW: a smaller team holds several of its threads' sums.  A block's ranks and factors then
// do not depend on the team that the launch chose.
constexpr int kWideCols = 4;
constexpr int kWideWaves = 8;

// val[e] -= sum_{l < r} s[l] p[l * sp + off[e]] in l order
__device__ __forceinline__ void wide_chain(double (&val)[kWideCols], const double* s, int r, const double* p, int64_t sp,
                                           const int (&off)[kWideCols])
{
    constexpr int E = kWideCols;
    int l = 0;
    for (; l + 8 <= r; l += 8) {
        double x[kWideCols][8];
#pragma unroll
        for (int q = 0; q < 8; q++)
#pragma unroll
            for (int e = 0; e < E; e++) x[e][q] = p[(l + q) * sp + off[e]];
#pragma unroll
        for (int q = 0; q < 8; q++)
#pragma unroll
            for (int e = 0; e < E; e++) val[e] = __fma_rn(-s[l + q], x[e][q], val[e]);
    }
    for (; l < r; l++)
#pragma unroll
        for (int e = 0; e < E; e++) val[e] = __fma_rn(-s[l], p[l * sp + off[e]], val[e]);
}

template <int KIND, int DIM, bool TOL, int NW>
__device__ __forceinline__ void wide_block(const AcaArgs& g, const int a, RegShared<kWideWaves, DIM>& sh, double* vt)
{
    constexpr int TS = NW * kWave, E = kWideCols;
    constexpr int H = kWideWaves / NW;  // partial sums per thread: element i belongs to sum i / TS % H
    static_assert(H * NW == kWideWaves && E % H == 0, "whole wavefronts");
    const int tid = threadIdx.x;
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const int lane = threadIdx.x % kWave;
    const int4 b = g.blk[a];
    const int k = g.kb[a];
    const int l1 = b.x, m1 = b.y - b.x + 1;
    const int l2 = b.z, m2 = b.w - b.z + 1;
    const int64_t vs = m2;
    const KernelParams kp = g.kp;
    double* const Ub = g.ublk ? g.ublk[a] : g.U + g.uoff[a];
    double* const Vb = g.vblk ? g.vblk[a] : g.V + g.voff[a];
    const int64_t lu = g.ldu[a], lv = g.ldv[a];
    auto team_extreme = [&](double v, bool mx) {
        v = mx ? wave_max(v) : wave_min(v);
        if (lane == 0) sh.ext[w] = v;
        __syncthreads();
        double t = sh.ext[0];
        for (int q = 1; q < NW; q++) t = mx ? fmax(t, sh.ext[q]) : fmin(t, sh.ext[q]);
        __syncthreads();
        return t;
    };
    auto team_sum = [&](const double (&v)[H]) {
#pragma unroll
        for (int h = 0; h < H; h++) {
            const double x = wave_add(v[h]);
            if (lane == 0) sh.ext[h * NW + w] = x;
        }
        __syncthreads();
        double t = 0.0;
        for (int q = 0; q < kWideWaves; q++) t += sh.ext[q];
        __syncthreads();
        return t;
    };
    const bool diag = kp.reg != 0.0 && l1 <= b.w && l2 <= b.y;  // some entry carries the regularization
    auto entry = [&](const double* x, const double* y, int i, int j) {
        double r2 = 0.0;
#pragma unroll
        for (int d = 0; d < DIM; d++) {
            const double t = x[d] - y[d];
            r2 = __dadd_rn(r2, __dmul_rn(t, t));
        }
        double e = kernel_of_r2_k<KIND>(kp, r2);
        if (diag && i == j) e += kp.reg;
        return e;
    };
    // rank 0 without evaluation, as in the register form
    if (g.scan && !g.resume && k > 0 && reg_monotone<KIND>() && !diag) {
        const work_item& wi = g.items[a];
        double r2 = 0.0;
#pragma unroll
        for (int d = 0; d < DIM; d++) {
            const double gap = fmax(0.0, fmax(wi.min1[d] - wi.max2[d], wi.min2[d] - wi.max1[d]));
            r2 += gap * gap;
        }
        const double sm2 = sqrt((double)m2);
        if (!(sm2 * kernel_of_r2_k<KIND>(kp, 0.5 * r2) >= 0.5e-13)) {
            r2 = 0.0;
#pragma unroll
            for (int d = 0; d < DIM; d++) {
                double lo1 = 1e300, hi1 = -1e300, lo2 = 1e300, hi2 = -1e300;
                for (int i = tid; i < m1; i += TS) {
                    const double x = g.c1.x[d][l1 + i];
                    lo1 = fmin(lo1, x);
                    hi1 = fmax(hi1, x);
                }
                for (int j = tid; j < m2; j += TS) {
                    const double x = g.c2.x[d][l2 + j];
                    lo2 = fmin(lo2, x);
                    hi2 = fmax(hi2, x);
                }
                lo1 = team_extreme(lo1, false);
                hi1 = team_extreme(hi1, true);
                lo2 = team_extreme(lo2, false);
                hi2 = team_extreme(hi2, true);
                const double gap = fmax(0.0, fmax(lo1 - hi2, lo2 - hi1));
                r2 += gap * gap;
            }
            if (sm2 * kernel_of_r2_k<KIND>(kp, r2 * (1.0 - 1e-9)) < 0.5e-13) {
                if (tid == 0) g.keff[a] = 0;
                return;
            }
        }
    }
    int i_r = -1, r0 = 0;
    double fro2 = 0.0;
    if (g.resume) {
        i_r = g.found[a] - 1;
        if (i_r >= m1 - 1) return;  // no acceptable row was left: the block is complete
        r0 = g.keff[a];
        fro2 = g.fro2[a];
        for (int j = tid; j < m2; j += TS)
            for (int l = 0; l < r0; l++) vt[l * vs + j] = Vb[(int64_t)j * lv + l];
    }
    int ke = r0;
    bool suspended = false, met = false;
    for (int r = r0; r < k && !met; r++) {
        int jr = -1;
        double p = 0.0;
        bool stop = false;
        int tries = 0;
        for (;;) {
            if (i_r >= m1 - 1) {
                stop = true;
                break;
            }
            i_r++;
            // row i_r's U terms and point
            __syncthreads();
            if (tid < r) sh.u[tid] = Ub[tid * lu + i_r];
            if (tid >= kRegRank && tid < kRegRank + DIM) sh.xu[tid - kRegRank] = g.c1.x[tid - kRegRank][l1 + i_r];
            __syncthreads();
            double nw[H] = {0.0}, best = -1.0, bval = 0.0;
            int bj = -1;
            for (int j0 = tid; j0 < m2; j0 += E * TS) {
                int off[E];
#pragma unroll
                for (int e = 0; e < E; e++) off[e] = min(j0 + e * TS, m2 - 1);
                double val[E];
#pragma unroll
                for (int e = 0; e < E; e++) {
                    double y[DIM];
#pragma unroll
                    for (int d = 0; d < DIM; d++) y[d] = g.c2.x[d][l2 + off[e]];
                    val[e] = entry(sh.xu, y, l1 + i_r, l2 + off[e]);
                }
                wide_chain(val, sh.u, r, vt, vs, off);
#pragma unroll
                for (int e = 0; e < E; e++) {
                    const int j = j0 + e * TS;
                    if (j < m2) {
                        vt[r * vs + j] = val[e];
                        nw[e % H] = __fma_rn(val[e], val[e], nw[e % H]);
                        const double ax = fabs(val[e]);
                        if (g.tie_last ? ax >= best : ax > best) {
                            best = ax;
                            bval = val[e];
                            bj = j;
                        }
                    }
                }
            }
#pragma unroll
            for (int h = 0; h < H; h++) nw[h] = wave_add(nw[h]);
            const double wb = wave_max(best);
            uint64_t mask = __ballot(best == wb);
            if (mask & (mask - 1)) {  // equal candidates: the last (first) index
                const double cj = best == wb ? (double)bj : g.tie_last ? -1.0 : 1e300;
                const double pick = g.tie_last ? wave_max(cj) : wave_min(cj);  // by every lane
                mask = __ballot(cj == pick);
            }
            const int wl = __builtin_ctzll(mask);
            const int wj = __builtin_amdgcn_readlane(bj, wl);
            const double wv = lane_of(bval, wl);
            if (lane == 0) {
#pragma unroll
                for (int h = 0; h < H; h++) sh.red[h * NW + w] = nw[h];
                sh.best[w] = wb;
                sh.bval[w] = wv;
                sh.bj[w] = wj;
            }
            __syncthreads();
            double nrm = 0.0;
            for (int q = 0; q < kWideWaves; q++) nrm += sh.red[q];
            double bb = sh.best[0];
            jr = sh.bj[0];
            p = sh.bval[0];
            for (int q = 1; q < NW; q++) {
                const double ob = sh.best[q];
                const int oj = sh.bj[q];
                if (ob > bb || (ob == bb && (g.tie_last ? oj > jr : (oj < jr && oj >= 0)))) {
                    bb = ob;
                    jr = oj;
                    p = sh.bval[q];
                }
            }
            nrm = lane_of(nrm, 0);
            jr = __builtin_amdgcn_readlane(jr, 0);
            p = lane_of(p, 0);
            if (sqrt(nrm) >= 1.0e-13) break;
            // the norms of the next rows, together: one read of V for all of them
            const int n = min(kRegAhead, m1 - 1 - i_r);
            for (int q = tid; q < kRegAhead * kRegRank; q += TS) {
                const int e = min(q / kRegRank, n - 1), l = q % kRegRank;
                if (n > 0 && l < r) sh.tu[q / kRegRank][l] = Ub[l * lu + i_r + 1 + e];
            }
            if (n > 0 && tid < kRegAhead * DIM)
                sh.tx[tid / DIM][tid % DIM] = g.c1.x[tid % DIM][l1 + i_r + 1 + min(tid / DIM, n - 1)];
            __syncthreads();
            for (int h = 0; h < H; h++) {
                double tn[kRegAhead];
#pragma unroll
                for (int e = 0; e < kRegAhead; e++) tn[e] = 0.0;
                for (int j = n > 0 ? tid + h * TS : m2; j < m2; j += H * TS) {
                    double y[DIM], t[kRegAhead];
#pragma unroll
                    for (int d = 0; d < DIM; d++) y[d] = g.c2.x[d][l2 + j];
#pragma unroll
                    for (int e = 0; e < kRegAhead; e++) t[e] = entry(sh.tx[e], y, l1 + i_r + 1 + e, l2 + j);
                    int l = 0;
                    for (; l + 8 <= r; l += 8) {
                        double x[8];
#pragma unroll
                        for (int q = 0; q < 8; q++) x[q] = vt[(l + q) * vs + j];
#pragma unroll
                        for (int q = 0; q < 8; q++)
#pragma unroll
                            for (int e = 0; e < kRegAhead; e++) t[e] = __fma_rn(-sh.tu[e][l + q], x[q], t[e]);
                    }
                    for (; l < r; l++) {
                        const double x = vt[l * vs + j];
#pragma unroll
                        for (int e = 0; e < kRegAhead; e++) t[e] = __fma_rn(-sh.tu[e][l], x, t[e]);
                    }
#pragma unroll
                    for (int e = 0; e < kRegAhead; e++) tn[e] = __fma_rn(t[e], t[e], tn[e]);
                }
#pragma unroll
                for (int e = 0; e < kRegAhead; e++) {
                    tn[e] = wave_add(tn[e]);
                    if (lane == 0) sh.tn[e][h * NW + w] = tn[e];
                }
            }
            __syncthreads();
            int skip = 0;
            for (; skip < n; skip++) {
                double t = 0.0;
                for (int q = 0; q < kWideWaves; q++) t += sh.tn[skip][q];
                if (sqrt(lane_of(t, 0)) >= 1.0e-13) break;
            }
            i_r += skip;
            tries += 1 + skip;
            if (g.suspend && tries >= g.tries && skip == n) {
                suspended = i_r < m1 - 1;
                stop = true;
                break;
            }
        }
        if (stop) break;
        // the pivot column's V terms and point; v_r = row / pivot and the residual column
        if (tid < r) sh.v[tid] = vt[tid * vs + jr];
        if (tid >= kRegRank && tid < kRegRank + DIM) sh.xv[tid - kRegRank] = g.c2.x[tid - kRegRank][l2 + jr];
        __syncthreads();
        double nu[H] = {0.0}, nv[H] = {0.0};
        for (int j0 = tid; j0 < m2; j0 += H * TS) {
#pragma unroll
            for (int h = 0; h < H; h++) {
                const int j = j0 + h * TS;
                if (j < m2) {
                    const double x = vt[r * vs + j] / p;
                    vt[r * vs + j] = x;
                    if (TOL) nv[h] = __fma_rn(x, x, nv[h]);
                }
            }
        }
        for (int i0 = tid; i0 < m1; i0 += E * TS) {
            int off[E];
#pragma unroll
            for (int e = 0; e < E; e++) off[e] = min(i0 + e * TS, m1 - 1);
            double val[E];
#pragma unroll
            for (int e = 0; e < E; e++) {
                double x[DIM];
#pragma unroll
                for (int d = 0; d < DIM; d++) x[d] = g.c1.x[d][l1 + off[e]];
                val[e] = entry(x, sh.xv, l1 + off[e], l2 + jr);
            }
            wide_chain(val, sh.v, r, Ub, lu, off);
#pragma unroll
            for (int e = 0; e < E; e++) {
                if (i0 + e * TS < m1) {
                    Ub[r * lu + i0 + e * TS] = val[e];
                    if (TOL) nu[e % H] = __fma_rn(val[e], val[e], nu[e % H]);
                }
            }
        }
        ke = r + 1;
        if (TOL) {
            // ||U V^T||_F^2 gains 2 u_r . (U (V^T v_r)) + ||u_r||^2 ||v_r||^2
            for (int c = 0; c < (r + 7) / 8 * H; c++) {
                const int q0 = c / H * 8, h = c % H;
                double q[8];
#pragma unroll
                for (int e = 0; e < 8; e++) q[e] = 0.0;
                for (int j = tid + h * TS; j < m2; j += H * TS) {
                    const double x = vt[r * vs + j];
#pragma unroll
                    for (int e = 0; e < 8; e++)
                        if (q0 + e < r) q[e] = __fma_rn(vt[(q0 + e) * vs + j], x, q[e]);
                }
#pragma unroll
                for (int e = 0; e < 8; e++) {
                    q[e] = wave_add(q[e]);
                    if (lane == 0) sh.g[h * NW + w][q0 + e] = q[e];
                }
            }
            __syncthreads();
            if (tid < r) {
                double x = 0.0;
                for (int q = 0; q < kWideWaves; q++) x += sh.g[q][tid];
                sh.v[tid] = -x;
            }
            __syncthreads();
            double cross[H] = {0.0};
            for (int i0 = tid; i0 < m1; i0 += E * TS) {
                int off[E];
                double val[E];
#pragma unroll
                for (int e = 0; e < E; e++) {
                    off[e] = min(i0 + e * TS, m1 - 1);
                    val[e] = 0.0;
                }
                wide_chain(val, sh.v, r, Ub, lu, off);
#pragma unroll
                for (int e = 0; e < E; e++)
                    if (i0 + e * TS < m1) cross[e % H] = __fma_rn(val[e], Ub[r * lu + i0 + e * TS], cross[e % H]);
            }
            const double su = team_sum(nu), sv = team_sum(nv);
            fro2 = fro2 + 2.0 * team_sum(cross) + su * sv;
            const bool m = (g.tol.mode == 2 || r % 5 == 0) && sqrt(su) * sqrt(sv) <= g.tol.c * sqrt(fmax(fro2, 0.0));
            met = __builtin_amdgcn_readfirstlane(m ? 1 : 0) != 0;
        }
    }
    for (int j = tid; j < m2; j += TS)
        for (int l = 0; l < ke; l++) Vb[(int64_t)j * lv + l] = vt[l * vs + j];
    if (tid == 0) {
        g.keff[a] = ke;
        if (suspended) {
            g.row[a] = i_r;
            g.found[a] = m1;
            g.fro2[a] = fro2;
            g.queue[atomicAdd(g.queued, 1)] = a;
        }
    }
}

// The wide blocks, taken from list[] in order by the workgroups of the launch, each with
// its slab: a workgroup ends when the list does.
template <int KIND, int DIM, bool TOL, int NW>
__global__ void __launch_bounds__(NW* kWave) __attribute__((amdgpu_waves_per_eu(3, 3)))
aca_wide_kernel(AcaArgs g)
{
    __shared__ RegShared<kWideWaves, DIM> sh;
    const int n = g.resume ? *g.count : g.nlist;
    double* const vt = g.slabs + (int64_t)blockIdx.x * g.slab;
    for (;;) {
        // This barrier keeps the fetch apart from the last block's "thread 0 writes":
        // without it the compiler joins the two conditions across the loop's edge, and
        // the other threads go round again without thread 0 (and without a new item).
        __syncthreads();
        if (threadIdx.x == 0) sh.item = atomicAdd(g.next, 1);
        __syncthreads();
        const int q = __builtin_amdgcn_readfirstlane(sh.item);
        __syncthreads();
        if (q >= n) return;
        wide_block<KIND, DIM, TOL, NW>(g, g.list[q], sh, vt);
    }
}

// ---- search over suspended blocks ------------------------------------------------
// Workgroup (queue position, chunk, column segment): rows row[a] + 1 + 64 chunk ... of block a.  The
// chunks of a block are far apart in the launch order, so that later rows mostly find an
// earlier one there and end.
template <int KIND, int DIM>
__global__ void __launch_bounds__(kSearchWaves* kWave)
aca_search_kernel(AcaArgs g, int chunk0)
{
    __shared__ SearchShared<DIM, kSearchWaves, kSearchTile> sh;
    if ((int)blockIdx.x >= *g.count) return;
    const int a = g.list[blockIdx.x];
    const int4 b = g.blk[a];
    const int m1 = b.y - b.x + 1;
    const int first = g.row[a] + 1 + (chunk0 + (int)blockIdx.y) * kSearchRows;
    if (first >= m1) return;
    const double* Ub = g.ublk ? g.ublk[a] : g.U + g.uoff[a];
    const double* Vb = g.vblk ? g.vblk[a] : g.V + g.voff[a];
    const int hit = search_rows<KIND, DIM>(g, b, first, g.keff[a], Ub, g.ldu[a], Vb, g.ldv[a], sh, g.found + a,
                                          (int)blockIdx.z, (int)gridDim.z);
    if (threadIdx.x == 0 && hit < m1) atomicMin(g.found + a, hit);
}

template <int KIND, int DIM, bool TOL>
hmg_status reg_launch_nw(const AcaArgs& g, int nw, bool wide, int kmax, hipStream_t s)
{
    const unsigned n = (unsigned)g.nlist;
    if (wide) {
        const unsigned m = (unsigned)std::min(g.nlist, g.nslabs);
        // few blocks: eight wavefronts halve a rank step's latency
        if (nw == 4 && 2 * n > (unsigned)g.few)
            aca_wide_kernel<KIND, DIM, TOL, 4><<<m, 4 * kWave, 0, s>>>(g);
        else
            aca_wide_kernel<KIND, DIM, TOL, 8><<<m, 8 * kWave, 0, s>>>(g);
        HMG_HIP(hipGetLastError());
        return HMG_OK;
    }
    // 5 wavefronts: three teams per compute unit with NT = 8, two with 16; the latter keep
    // ranks past 16 on chip, which is what counts when there are few
    const bool many = n > (unsigned)g.few || kmax <= 8 + kRegTail;
    const int nt = nw == 16 || nw == 8 || nw == 4 || (nw == 5 && many) ? 8 : 16;
    const size_t tail = kmax > nt ? (size_t)2 * kRegTail * nw * kWave * sizeof(double) : 0;
    switch (nw) {
    case 1:
        aca_reg_kernel<KIND, DIM, TOL, 1, 16><<<n, 1 * kWave, tail, s>>>(g);
        break;
    case 2:
        aca_reg_kernel<KIND, DIM, TOL, 2, 16><<<n, 2 * kWave, tail, s>>>(g);
        break;
    case 3:
        aca_reg_kernel<KIND, DIM, TOL, 3, 16><<<n, 3 * kWave, tail, s>>>(g);
        break;
    case 4:
        aca_reg_kernel<KIND, DIM, TOL, 4, 8><<<n, 4 * kWave, tail, s>>>(g);
        break;
    case 5:
        if (nt == 8)
            aca_reg_kernel<KIND, DIM, TOL, 5, 8><<<n, 5 * kWave, tail, s>>>(g);
        else
            aca_reg_kernel<KIND, DIM, TOL, 5, 16><<<n, 5 * kWave, tail, s>>>(g);
        break;
    case 8:
        aca_reg_kernel<KIND, DIM, TOL, 8, 8><<<n, 8 * kWave, tail, s>>>(g);
        break;
    case 9:
        aca_reg_kernel<KIND, DIM, TOL, 9, 16><<<n, 9 * kWave, tail, s>>>(g);
        break;
    case 12:
        aca_reg_kernel<KIND, DIM, TOL, 12, 16><<<n, 12 * kWave, tail, s>>>(g);
        break;
    default:
        aca_reg_kernel<KIND, DIM, TOL, 16, 8><<<n, 16 * kWave, tail, s>>>(g);
        break;
    }
    HMG_HIP(hipGetLastError());
    return HMG_OK;
}

}  // namespace

template <int KIND>
hmg_status aca_reg_launch(const AcaArgs& g, int nw, bool wide, int kmax, hipStream_t s)
{
    const bool tol = g.tol.mode != 0;
    if (g.kp.dim == 3)
        return tol ? reg_launch_nw<KIND, 3, true>(g, nw, wide, kmax, s)
                   : reg_launch_nw<KIND, 3, false>(g, nw, wide, kmax, s);
    return tol ? reg_launch_nw<KIND, 2, true>(g, nw, wide, kmax, s)
               : reg_launch_nw<KIND, 2, false>(g, nw, wide, kmax, s);
}

template <int KIND>
hmg_status aca_search_launch(const AcaArgs& g, int maxm1, hipStream_t s)
{
    const unsigned chunks = (unsigned)((maxm1 + kSearchRows - 1) / kSearchRows);
    // few workgroups: the columns in up to eight segments (the share of a pruned tile is
    // set for that many)
    const int64_t wgs = std::max<int64_t>((int64_t)g.nlist * chunks, 1);
    const unsigned nseg = (unsigned)std::clamp<int64_t>(4 * (int64_t)g.few / wgs, 1, 8);
    for (unsigned c0 = 0; c0 < chunks; c0 += 65535) {
        const dim3 grid((unsigned)g.nlist, std::min(chunks - c0, 65535u), nseg);
        if (g.kp.dim == 3)
            aca_search_kernel<KIND, 3><<<grid, kSearchWaves * kWave, 0, s>>>(g, (int)c0);
        else
            aca_search_kernel<KIND, 2><<<grid, kSearchWaves * kWave, 0, s>>>(g, (int)c0);
        HMG_HIP(hipGetLastError());
    }
    return HMG_OK;
}

}  // namespace hmg
