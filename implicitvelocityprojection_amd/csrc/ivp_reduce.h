// ivp_reduce.h -- grid reductions: per-block partials, folded in a fixed order (deterministic) by a
// one-block finalize kernel or by every block of the pass that needs the sum, which also advance the
// device-resident solver state.
#pragma once

#include <type_traits>

#include "ivp_internal.h"
#include "ivp_launch.h"

namespace ivp {

// Per-block partial sums of up to 3 doubles (fixed order inside the block).  The grid totals are
// formed by a later launch on the stream: the kernel boundary publishes the partials,
// so no device-scope fence (an L2 write-back on a multi-XCD part) is issued per block.
template <int NV, int T = BLOCK>
__device__ __forceinline__ void block_partials(const double (&v)[NV], double* partials, int stride) {
    __shared__ double lds[NV][T / WAVE];
    double s[NV];
    block_sums<NV, T>(v, s, lds);
    if (threadIdx.x == 0)
#pragma unroll
        for (int q = 0; q < NV; ++q) partials[q * stride + blockIdx.x] = s[q];
}

enum FinOp {
    FIN_BUILD, FIN_PACK, FIN_RHS, FIN_FIRST, FIN_FIRST_BUILD, FIN_CG_PAP, FIN_CG_UPDATE, FIN_W18_INIT, FIN_W18_PAP, FIN_W18_UPDATE,
    FIN_CG_REPLACE
};

struct FinArgs {
    const double* partials;
    int stride;
    int nblocks;
    SolverState* st;
    double tol;
    int max_iter;
    int gated;   // FIN_PACK queued behind a CG read-back: only once that CG stopped without failing
    SolverState* host;           // pinned copy of the state for the host (nullptr: none)
    const int* flags;            // the build's error flags, reported with it
    unsigned long long* mark;    // device clock after the reduction (nullptr: none)
};

// Report to the host: the state, with the build's error flags, into pinned memory.  The host waits
// for the kernel; no copy command follows it.
__device__ __forceinline__ void report_state(SolverState* st, SolverState* host, const int* flags) {
    st->flags = *flags;
    *host = *st;
}

constexpr int FIN_BLOCK = 1024;
constexpr int FIN_UNROLL = 4;  // the fold below adds exactly four loads per row

// Fixed-order fold of NV rows of n partials by one FIN_BLOCK-thread block (valid in thread 0).
// Each thread issues NV * FIN_UNROLL independent loads before adding, so the fold costs a few
// memory latencies instead of one per loop trip.
template <int NV>
__device__ __forceinline__ void fold_partials(const double* __restrict__ partials, int stride, int n,
                                              double* t) {
    __shared__ double lds[NV][FIN_BLOCK / WAVE];
    double s[NV];
#pragma unroll
    for (int q = 0; q < NV; ++q) s[q] = 0.0;
    for (int base = 0; base < n; base += FIN_UNROLL * FIN_BLOCK) {
        double v[NV][FIN_UNROLL];
#pragma unroll
        for (int q = 0; q < NV; ++q)
#pragma unroll
            for (int u = 0; u < FIN_UNROLL; ++u) {
                int idx = base + u * FIN_BLOCK + (int)threadIdx.x;
                v[q][u] = idx < n ? partials[q * stride + idx] : 0.0;
            }
#pragma unroll
        for (int q = 0; q < NV; ++q) s[q] += (v[q][0] + v[q][1]) + (v[q][2] + v[q][3]);
    }
    int lane = threadIdx.x & (WAVE - 1), w = threadIdx.x / WAVE;
#pragma unroll
    for (int q = 0; q < NV; ++q) {
        double x = wave_sum(s[q]);
        if (lane == 0) lds[q][w] = x;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
#pragma unroll
        for (int q = 0; q < NV; ++q) {
            double x = 0.0;
            for (int k = 0; k < FIN_BLOCK / WAVE; ++k) x += lds[q][k];
            t[q] = x;
        }
    }
}

// Scalar state update after a reduction (the host logic of ip.py:296-327,
// pressure_base.py:405-423, weiler18.py:330-365), applied to one solver state.
template <int OP>
__device__ __forceinline__ void fin_apply(SolverState* st, const double* t, double tol, int max_iter) {
    if (OP == FIN_BUILD) {
        st->total_pairs = (long long)t[0];
        st->win_entries = (long long)t[1];
    } else if (OP == FIN_PACK) {
        st->err_sum = t[0];
        st->n_active_rows = (int)t[1];
        st->active_pairs = (long long)t[2];
    } else if (OP == FIN_FIRST || OP == FIN_FIRST_BUILD) {
        // the constraint pass's sums, the right-hand side's, and the last build's if they are left
        fin_apply<FIN_PACK>(st, t, tol, max_iter);
        fin_apply<FIN_RHS>(st, t + 3, tol, max_iter);
        if (OP == FIN_FIRST_BUILD) fin_apply<FIN_BUILD>(st, t + BUILD_ROW, tol, max_iter);
    } else if (OP == FIN_RHS || OP == FIN_W18_INIT) {
        double rr = t[0];
        if (OP == FIN_RHS) {
            st->n_touched_rows = (int)t[0];
            st->touched_pairs = (long long)t[1];
            rr = t[2];
        }
        // IP: CG runs when r.r > 1e-30 (ip.py:302); Weiler18: when r.z > 1e-12 (weiler18.py:337)
        double floor_ = OP == FIN_RHS ? 1e-30 : 1e-12;
        st->rr_old = rr;
        st->rr_new = rr;
        st->rr_last = rr;
        st->rr0 = rr;
        st->rr_best = rr;
        st->stalls = 0;
        st->tol = tol;
        st->max_iter = max_iter;
        st->iter = 0;
        st->status = 0;
        st->active = (rr > floor_ && max_iter > 0) ? 1 : 0;
    } else if (OP == FIN_CG_PAP) {
        // ip.py:307-311
        st->pAp = t[0];
        if (t[0] < 0.0) {
            st->status = IVP_NOT_PD;
            st->active = 0;
        } else {
            st->alpha = st->rr_old / (t[0] > 1e-30 ? t[0] : 1e-30);
        }
    } else if (OP == FIN_CG_UPDATE) {
        // ip.py:317-327
        int it = st->iter + 1;
        st->iter = it;
        st->rr_new = t[0];
        st->rr_last = t[0];
        bool stop = (t[0] < st->tol && it >= 2) || it >= st->max_iter;
        if (stop) {
            st->active = 0;
        } else {
            double ro = st->rr_old;
            st->beta = t[0] / (ro > 1e-30 ? ro : 1e-30);
            st->rr_old = t[0];
        }
    } else if (OP == FIN_CG_REPLACE) {
        // CG iteration whose recursive residual (t[0] = its r.r) was replaced by the true
        // residual b - A x (t[1] = its r.r).  The stop test reads the true r.r; beta keeps the
        // recursion's ratio, so a true residual far above the recursive one (an operator error
        // floor) turns p into about r instead of amplifying p.  Two replacements in a row that
        // do not lower the smallest true r.r end the solve: that floor has been reached.
        int it = st->iter + 1;
        st->iter = it;
        st->rr_new = t[1];
        st->rr_last = t[1];
        if (t[1] < st->rr_best) {
            st->rr_best = t[1];
            st->stalls = 0;
        } else {
            st->stalls = st->stalls + 1;
        }
        bool stop = (t[1] < st->tol && it >= 2) || it >= st->max_iter || st->stalls >= 2;
        if (stop) {
            st->active = 0;
        } else {
            double ro = st->rr_old;
            st->beta = t[0] / (ro > 1e-30 ? ro : 1e-30);
            st->rr_old = t[1];
        }
    } else if (OP == FIN_W18_UPDATE) {
        // weiler18.py:350-365 (t[0] = r.r, t[1] = r.z)
        int it = st->iter + 1;
        st->iter = it;
        st->rr_last = t[0];
        bool stop = (t[0] < st->tol && it >= 2) || it >= st->max_iter;
        if (stop) {
            st->active = 0;
        } else {
            double ro = st->rr_old;
            st->beta = t[1] / (ro > 1e-12 ? ro : 1e-12);
            st->rr_old = t[1];
        }
    }
}

template <int OP>
constexpr int fin_nv() {
    return OP == FIN_FIRST_BUILD ? 8 : OP == FIN_FIRST ? 6 : OP == FIN_PACK || OP == FIN_RHS ? 3
           : OP == FIN_BUILD || OP == FIN_W18_UPDATE || OP == FIN_CG_REPLACE ? 2 : 1;
}

// One block: fold the partials of the previous kernel in a fixed order and advance the solver
// state.
template <int OP>
__global__ __launch_bounds__(FIN_BLOCK) void k_finalize(FinArgs a) {
    constexpr int NV = fin_nv<OP>();
    SolverState* st = a.st;
    const bool skip = OP == FIN_PACK && a.gated && (st->active != 0 || st->status != 0);
    if (!skip) {
        double t[8] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
        fold_partials<NV>(a.partials, a.stride, a.nblocks, t);
        if (threadIdx.x == 0) {
            fin_apply<OP>(st, t, a.tol, a.max_iter);
            if (a.mark) *a.mark = wall_clock64();
        }
    }
    if (a.host && threadIdx.x == 0) report_state(st, a.host, a.flags);
}

// ---- folds by the pass that needs the sum ---------------------------------------------------
//
// A finalize launch between two passes costs 2 us and the gap before it for a few scalars.  While the
// readers' blocks times the partials stay below FOLD_READS (42 MB a row, from L2) every block of the next
// pass folds them itself, all to the same bits, and one block writes the state; above it the folds take
// longer than the launch that they save, and k_prefold first reduces each row to PREFOLD partials in
// one short launch of many blocks (15 625 partials: 4.6 us, what the one-block finalize took; the pass
// that folds the rest is then no dependent launch of its own).
// p.Ap has nd / 64 partials, an update's sums one per block of vec_grid, and vec_grid's blocks read both (the
// operator pass's where it forms p).  Up to VEC_MAX rows that is 4.2 million reads at most (16 384 partials
// by 256 blocks), so the readers fold; one row more, back at 256-thread blocks, it is 68 million for p.Ap and
// 17 million for the sums, so in the CG k_prefold runs above VEC_MAX only (elsewhere: finalizes of more
// than FIN_MAX partials).  The line between was measured with 256-thread vector blocks throughout, us per
// implicit viscosity solve, prefolded / folded by the readers: p.Ap at 133k rows 420 / 390, 176k
// 506 / 480, 262k (4.2 million reads) 879 / 861, 350k (7.5 million) 1079 / 1108; the sums at 500k (3.8 million)
// 1378 / 1359, 750k (8.6 million) 1908 / 1956, 1M 2371 / 2535.
constexpr long long FOLD_READS = 5ll << 20;
// Partials (all rows) that the one-block finalize folds alone, us: three rows of 4096 4.3 and 6.9 with a
// prefold; three of 15 625 9.1 and 9.7; six of 15 625 9.7 with one
constexpr int FIN_MAX = 1 << 16;

// `meanwhile` runs with the first partials in flight: the caller's own loads, which would otherwise wait
// for the fold (23k rows: update 3.8 -> 3.4 us, p pass 3.9 -> 3.5).
template <int NV, int T, class M>
__device__ __forceinline__ void block_fold(const double* __restrict__ p, int stride, int n, double (&t)[NV], M&& meanwhile) {
    __shared__ double lds[NV][T / WAVE];
    double s[NV];
#pragma unroll
    for (int q = 0; q < NV; ++q) s[q] = 0.0;
    for (int base = 0; base < n; base += 4 * T) {
        double v[NV][4];
#pragma unroll
        for (int q = 0; q < NV; ++q)
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const int k = base + u * T + (int)threadIdx.x;
                v[q][u] = k < n ? p[(size_t)q * stride + k] : 0.0;
            }
        if (base == 0) meanwhile();
#pragma unroll
        for (int q = 0; q < NV; ++q) s[q] += (v[q][0] + v[q][1]) + (v[q][2] + v[q][3]);
    }
#pragma unroll
    for (int q = 0; q < NV; ++q) {
        const double x = wave_sum(s[q]);
        if ((threadIdx.x & (WAVE - 1)) == 0) lds[q][threadIdx.x >> 6] = x;
    }
    __syncthreads();
#pragma unroll
    for (int q = 0; q < NV; ++q) t[q] = waves_total<T>(lds[q]);
}

// Row q of n partials to PREFOLD partials: block b folds the b-th share
template <int NV>
__global__ __launch_bounds__(BLOCK) void k_prefold(const double* __restrict__ p, int stride, int n,
                                                   double* __restrict__ out) {
    const int per = (n + PREFOLD - 1) / PREFOLD;
    const int k0 = (int)blockIdx.x * per < n ? (int)blockIdx.x * per : n;
    double t[NV];
    block_fold<NV, BLOCK>(p + k0, stride, k0 + per < n ? per : n - k0, t, []() {});
    if (threadIdx.x == 0)
#pragma unroll
        for (int q = 0; q < NV; ++q) out[q * PREFOLD + (int)blockIdx.x] = t[q];
}

// Blocks of a CG's vector passes (update, p): 256 threads of one row each, or between VEC_MIN and VEC_MAX rows at
// most 256 blocks -- one per CU -- of 1024 threads with as many rows each as that takes, all in flight:
// then both the partials they write and the blocks that fold the operator pass's are few, and no
// k_prefold is needed (us per implicit viscosity solve, 256-thread blocks / these: 90k rows 294 / 302, 133k
// 377 / 371, 262k 860 / 843, 350k 1071 / 1025, 500k 1351 / 1287, 1M 2374 / 2283; IP solve at 262k 331 / 315).
// VEC_MAX is what VEC_ROWS rows per thread in registers reach, not where 256-thread blocks become better;
// above it a solve has its 256-thread form with k_prefold (1.06M to 4.1M rows: 1.0 to 1.27 times as fast as with
// one-block finalizes between the passes).
constexpr int VEC_THREADS = 1024, VEC_BLOCKS = 256, VEC_ROWS = 4;
constexpr int VEC_MIN = 1 << 17, VEC_MAX = VEC_THREADS * VEC_BLOCKS * VEC_ROWS;
struct VecGrid {
    int threads, rows, blocks;   // per block; per thread; blocks
};
inline VecGrid vec_grid(int nd) {
    if (nd < VEC_MIN || nd > VEC_MAX) return VecGrid{BLOCK, 1, blocks_for(nd)};
    const int rows = (nd + VEC_THREADS * VEC_BLOCKS - 1) / (VEC_THREADS * VEC_BLOCKS);
    return VecGrid{VEC_THREADS, rows, (nd + VEC_THREADS * rows - 1) / (VEC_THREADS * rows)};
}
// f(threads, rows) of a grid, as compile-time constants
template <class F>
inline int vec_dispatch(const VecGrid& g, F&& f) {
    using std::integral_constant;
    if (g.threads == BLOCK) return f(integral_constant<int, BLOCK>{}, integral_constant<int, 1>{});
    integral_constant<int, VEC_THREADS> t;
    switch (g.rows) {
    case 1: return f(t, integral_constant<int, 1>{});
    case 2: return f(t, integral_constant<int, 2>{});
    case 3: return f(t, integral_constant<int, 3>{});
    default: return f(t, integral_constant<int, VEC_ROWS>{});
    }
}

// Partials to fold: rows `stride` apart, n per row
struct Fold {
    const double* p;
    int stride, n;
};

// The partials in rows row0 .. row0 + NV - 1 for `readers` blocks that each fold them, brought down to
// PREFOLD per row if that is less work
template <int NV>
inline int fold_source(ivp_ctx* c, int row0, int n, int readers, Fold* f) {
    const double* p = c->partials + (size_t)row0 * c->max_blocks;
    *f = Fold{p, c->max_blocks, n};
    if ((long long)n * readers <= FOLD_READS) return IVP_OK;
    double* out = c->partials + (size_t)PARTIAL_ROWS * c->max_blocks + row0 * PREFOLD;
    hipLaunchKernelGGL(k_prefold<NV>, dim3(PREFOLD), dim3(BLOCK), 0, c->stream, p, c->max_blocks, n, out);
    IVP_HIP(hipGetLastError());
    *f = Fold{out, PREFOLD, PREFOLD};
    return IVP_OK;
}

// In an iteration's update pass: alpha from the operator pass's p.Ap (OP = FIN_CG_PAP, FIN_W18_PAP).
// Returns false when there is nothing to update.  The state's own fields stay as they are until
// the p pass; ran and prev_* tell it what happened here.
template <int OP, int T, class M>
__device__ __forceinline__ bool fold_alpha(SolverState* st, const Fold& f, float* alpha, M&& meanwhile) {
    const bool lead = blockIdx.x == 0 && threadIdx.x == 0;
    if (st->active == 0) {
        if (lead) st->ran = 0;
        return false;
    }
    const double rr_old = st->rr_old, rr_best = st->rr_best;
    const int iter = st->iter, stalls = st->stalls;
    double t[1];
    block_fold<1, T>(f.p, f.stride, f.n, t, meanwhile);
    // ip.py:307-311 fails on p.Ap < 0; weiler18.py:338-342 ends the iteration on p.Ap <= 0
    const double least = OP == FIN_CG_PAP ? 1e-30 : 1e-12;
    const bool bad = OP == FIN_CG_PAP ? t[0] < 0.0 : t[0] <= 0.0;
    const double al = rr_old / (t[0] > least ? t[0] : least);
    *alpha = (float)al;
    if (lead) {
        st->pAp = t[0];
        st->ran = bad ? 2 : 1;
        if (!bad) {
            st->alpha = al;
            st->prev_iter = iter;
            st->prev_rr_old = rr_old;
            st->prev_rr_best = rr_best;
            st->prev_stalls = stalls;
        }
    }
    return !bad;
}

struct Advance {
    bool ran;        // the iteration updated x and r
    bool active;     // and the solve goes on
    bool stopped;    // no further iteration, and not because p.Ap failed
    float beta;
};

// In the iteration's p pass: the state after the iteration from the update pass's sums (OP =
// FIN_CG_UPDATE, FIN_CG_REPLACE, FIN_W18_UPDATE), formed by every block and written by one, which
// reports it to the host if asked.
template <int OP, int T, class M>
__device__ __forceinline__ Advance fold_advance(SolverState* st, const Fold& f, SolverState* host, const int* flags,
                                                M&& meanwhile) {
    const bool lead = blockIdx.x == 0 && threadIdx.x == 0;
    const int ran = st->ran;
    Advance a = {ran == 1, false, ran == 0 && st->status == 0, 0.0f};
    if (ran == 1) {
        SolverState s;
        s.iter = st->prev_iter;
        s.rr_old = st->prev_rr_old;
        s.rr_best = st->prev_rr_best;
        s.stalls = st->prev_stalls;
        s.tol = st->tol;
        s.max_iter = st->max_iter;
        s.active = 1;
        s.beta = 0.0;
        s.rr_new = 0.0;
        double t[fin_nv<OP>()];
        block_fold<fin_nv<OP>(), T>(f.p, f.stride, f.n, t, meanwhile);
        fin_apply<OP>(&s, t, 0.0, 0);
        a.active = s.active != 0;
        a.stopped = !a.active;
        a.beta = (float)s.beta;
        if (lead) {
            st->iter = s.iter;
            st->rr_old = s.rr_old;
            if (OP != FIN_W18_UPDATE) st->rr_new = s.rr_new;
            st->rr_last = s.rr_last;
            st->rr_best = s.rr_best;
            st->stalls = s.stalls;
            if (a.active) st->beta = s.beta;
            st->active = s.active;
        }
    } else if (ran == 2) {
        if (OP == FIN_W18_UPDATE) a.stopped = true;
        if (lead) {
            if (OP != FIN_W18_UPDATE) st->status = IVP_NOT_PD;
            st->active = 0;
        }
    }
    if (lead && host) report_state(st, host, flags);
    return a;
}

template <int OP>
inline int finalize(ivp_ctx* c, int nblocks, double tol = 0.0, int max_iter = 0, bool gated = false,
                    SolverState* host = nullptr, unsigned long long* mark = nullptr) {
    constexpr int NV = fin_nv<OP>();
    constexpr int row0 = OP == FIN_RHS ? 3 : OP == FIN_BUILD ? BUILD_ROW : 0;
    Fold f{c->partials + row0 * (size_t)c->max_blocks, c->max_blocks, nblocks};
    if (NV > 1 && nblocks * NV > FIN_MAX) IVP_TRY((fold_source<NV>(c, row0, nblocks, 1 << 20, &f)));
    FinArgs fa{f.p, f.stride, f.n, c->state, tol, max_iter, gated ? 1 : 0, host, c->err_flag, mark};
    hipLaunchKernelGGL(k_finalize<OP>, dim3(1), dim3(FIN_BLOCK), 0, c->stream, fa);
    IVP_HIP(hipGetLastError());
    return IVP_OK;
}

// ---- independent scenes ----------------------------------------------------------------------

// Per-block partial sums split by scene.  A block's rows span at most two scenes (every scene
// holds at least MIN_SCENE_DYNAMIC >= rows of a block): seg = 0 for rows of the block's first
// scene, 1 for the second.  Value q of segment g goes to row 2 q + g, column blk (the block's
// row block, so the blocks of one scene are one contiguous range).  `two` is block-uniform.
template <int NV>
__device__ __forceinline__ void block_partials_seg(const double (&v)[NV], int seg, bool two, double* partials,
                                                   int stride, int blk) {
    __shared__ double lds[2][NV][WAVES_PER_BLOCK];
    double x[NV], s[NV];
#pragma unroll
    for (int q = 0; q < NV; ++q) x[q] = seg == 0 ? v[q] : 0.0;
    block_sums<NV>(x, s, lds[0]);
    if (threadIdx.x == 0)
#pragma unroll
        for (int q = 0; q < NV; ++q) partials[(2 * q) * stride + blk] = s[q];
    if (two) {
#pragma unroll
        for (int q = 0; q < NV; ++q) x[q] = seg == 1 ? v[q] : 0.0;
        block_sums<NV>(x, s, lds[1]);
        if (threadIdx.x == 0)
#pragma unroll
            for (int q = 0; q < NV; ++q) partials[(2 * q + 1) * stride + blk] = s[q];
    }
}

struct FinScenesArgs {
    const double* partials;
    int stride;
    const int* sid;
    SceneState* ss;
    const SceneParams* prm;
    double* hist_err;     // [S * SCENE_HIST]
    int* hist_pcg;        // [S * SCENE_HIST]
    int S;
    int rpb;              // rows per block of the kernel that wrote the partials
};

// One wave per scene: fold the scene's block partials in a fixed order and advance its state
// with the single-scene logic (fin_apply), then its outer-loop phase (the host logic of
// ip.py:345-395 for one scene).  Scenes not in the phase this reduction belongs to are skipped.
template <int OP>
__global__ __launch_bounds__(BLOCK) void k_fin_scenes(FinScenesArgs a) {
    constexpr int NV = fin_nv<OP>();
    constexpr int want = OP == FIN_PACK ? PH_PACK : OP == FIN_RHS ? PH_RHS : PH_CG;
    const int s = blockIdx.x * WAVES_PER_BLOCK + (int)(threadIdx.x >> 6);
    const int lane = threadIdx.x & (WAVE - 1);
    if (s >= a.S) return;
    SceneState* sc = a.ss + s;
    if (sc->phase != want) return;
    const int b0 = sc->row0 / a.rpb, b1 = (sc->row0 + sc->nd - 1) / a.rpb;
    double t[3] = {0.0, 0.0, 0.0};
    for (int b = b0 + lane; b <= b1; b += WAVE) {
        const int seg = a.sid[b * a.rpb] == s ? 0 : 1;
#pragma unroll
        for (int q = 0; q < NV; ++q) t[q] += a.partials[(2 * q + seg) * a.stride + b];
    }
#pragma unroll
    for (int q = 0; q < NV; ++q) t[q] = wave_sum(t[q]);
    if (lane != 0) return;
    const SceneParams& p = *a.prm;
    double* herr = a.hist_err + (size_t)s * SCENE_HIST;
    int* hpcg = a.hist_pcg + (size_t)s * SCENE_HIST;
    if (OP == FIN_PACK) {
        fin_apply<OP>(&sc->cg, t, 0.0, 0);
        double err = sc->cg.err_sum / (double)sc->nd;
        if (sc->n_err < SCENE_HIST) herr[sc->n_err] = err;
        sc->n_err = sc->n_err + 1;
        bool converged = err < p.tol_opt && !p.fixed;
        if ((converged && sc->opt_iter >= 1) || sc->opt_iter >= p.max_opt) {
            sc->phase = PH_DONE;
            sc->final_err = err;
            sc->outer_iters = sc->opt_iter;
            if (!p.fixed && err >= p.tol_opt && sc->opt_iter >= p.max_opt) sc->status = IVP_NOT_CONVERGED;
        } else {
            sc->phase = PH_RHS;
        }
    } else if (OP == FIN_RHS) {
        fin_apply<OP>(&sc->cg, t, p.tol_pcg, p.max_pcg);
        if (sc->cg.active) {
            sc->phase = PH_CG;
        } else {
            sc->phase = PH_DUPDATE;
            if (sc->opt_iter < SCENE_HIST) hpcg[sc->opt_iter] = 0;
        }
    } else if (OP == FIN_CG_PAP) {
        fin_apply<OP>(&sc->cg, t, 0.0, 0);
        if (sc->cg.status == IVP_NOT_PD) {
            sc->status = IVP_NOT_PD;
            sc->phase = PH_DONE;
            sc->outer_iters = sc->opt_iter;
            sc->cg_total = sc->cg_total + sc->cg.iter;
            if (sc->opt_iter < SCENE_HIST) hpcg[sc->opt_iter] = sc->cg.iter;
        }
    } else if (OP == FIN_CG_UPDATE) {
        fin_apply<OP>(&sc->cg, t, 0.0, 0);
        if (!sc->cg.active) {
            sc->phase = PH_DUPDATE;
            sc->cg_total = sc->cg_total + sc->cg.iter;
            if (sc->opt_iter < SCENE_HIST) hpcg[sc->opt_iter] = sc->cg.iter;
        }
    }
}

}  // namespace ivp
