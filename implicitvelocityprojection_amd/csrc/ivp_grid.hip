// ivp_grid.hip -- particle store, cell sort, neighbour rows, density and Aii.
//
// Replaces the reference's Warp HashGrid build + neighbour cache (scripts/sim/
// neighbour_search.py:10-155) and PressureBase.compute_density / compute_Aii
// (scripts/sim/forces/pressure/pressure_base.py:12-87).
//
// Sort: a deterministic counting sort over cell keys.  count (atomic; a step's advection runs in
// the same pass), exclusive scan, scatter (atomic slot), then every particle ranks itself inside
// its cell by user id and moves to its place, so the resulting order -- (cell key, user id) -- depends on
// the positions only.  Cell keys are x-fastest linear, so the three cells (cx-1..cx+1, cy, cz) of a stencil
// row are one contiguous particle range: a query visits 9 ranges per population.
#include <cmath>

#include "ivp_internal.h"
#include "ivp_launch.h"
#include "ivp_reduce.h"

using namespace ivp;

namespace {

constexpr int SCAN_PER_THREAD = 8;
constexpr int SCAN_CHUNK = BLOCK * SCAN_PER_THREAD;

__device__ __forceinline__ int wave_incl_scan(int x, int lane) {
#pragma unroll
    for (int o = 1; o < WAVE; o <<= 1) {
        int y = __shfl_up(x, o, WAVE);
        if (lane >= o) x += y;
    }
    return x;
}

// Exclusive scan of one int per thread over the block; returns the exclusive prefix and the
// block total.
__device__ __forceinline__ int block_excl_scan(int v, int* total) {
    __shared__ int wsum[WAVES_PER_BLOCK];
    int lane = threadIdx.x & (WAVE - 1), w = threadIdx.x >> 6;
    int incl = wave_incl_scan(v, lane);
    if (lane == WAVE - 1) wsum[w] = incl;
    __syncthreads();
    int off = 0, tot = 0;
#pragma unroll
    for (int q = 0; q < WAVES_PER_BLOCK; ++q) {
        if (q < w) off += wsum[q];
        tot += wsum[q];
    }
    __syncthreads();
    *total = tot;
    return off + incl - v;
}

// start[i] = sum(cnt[0..i)) within the block's chunk; bsum[block] = chunk total
__global__ __launch_bounds__(BLOCK) void k_scan1(int n, const int* __restrict__ cnt, int* __restrict__ start,
                                                 int* __restrict__ bsum) {
    int base = blockIdx.x * SCAN_CHUNK + threadIdx.x * SCAN_PER_THREAD;
    int v[SCAN_PER_THREAD];
    int sum = 0;
#pragma unroll
    for (int q = 0; q < SCAN_PER_THREAD; ++q) {
        int idx = base + q;
        v[q] = idx < n ? cnt[idx] : 0;
        sum += v[q];
    }
    int tot;
    int run = block_excl_scan(sum, &tot);
#pragma unroll
    for (int q = 0; q < SCAN_PER_THREAD; ++q) {
        int idx = base + q;
        if (idx < n) start[idx] = run;
        run += v[q];
    }
    if (threadIdx.x == 0) bsum[blockIdx.x] = tot;
}

// single block: exclusive scan of the nb chunk totals, bsum[nb] = grand total
__global__ __launch_bounds__(BLOCK) void k_scan2(int nb, int* __restrict__ bsum) {
    __shared__ int carry_s;
    if (threadIdx.x == 0) carry_s = 0;
    __syncthreads();
    for (int base = 0; base < nb; base += BLOCK) {
        int idx = base + threadIdx.x;
        int v = idx < nb ? bsum[idx] : 0;
        int tot;
        int ex = block_excl_scan(v, &tot);
        int carry = carry_s;
        if (idx < nb) bsum[idx] = carry + ex;
        __syncthreads();
        if (threadIdx.x == 0) carry_s = carry + tot;
        __syncthreads();
    }
    if (threadIdx.x == 0) bsum[nb] = carry_s;
}

__global__ __launch_bounds__(BLOCK) void k_scan3(int n, int* __restrict__ start, const int* __restrict__ bsum, int nb) {
    int base = blockIdx.x * SCAN_CHUNK;
    int add = bsum[blockIdx.x];
    for (int q = threadIdx.x; q < SCAN_CHUNK; q += BLOCK) {
        int idx = base + q;
        if (idx < n) start[idx] += add;
    }
    if (blockIdx.x == 0 && threadIdx.x == 0) start[n] = bsum[nb];
}

// Cell starts in one launch: start[i] = sum(cnt[0..i)), given the chunk totals bsum (k_keys counts
// them with the cells).  Every block sums the totals before its chunk itself; with at most
// CELL_SCAN_CHUNKS of them (16 KB, in L2) that costs less than the two launches it saves: three
// launches took 9.2 us at 8k rows and 14 us at 1M (30k and 860k cells), this one 3.0 and 4.3.
constexpr int CELL_SCAN_CHUNKS = 4096;
__global__ __launch_bounds__(BLOCK) void k_cell_starts(int n, int nb, const int* __restrict__ cnt,
                                                       const int* __restrict__ bsum, int* __restrict__ start) {
    __shared__ int psum[WAVES_PER_BLOCK];
    const int base = blockIdx.x * SCAN_CHUNK + threadIdx.x * SCAN_PER_THREAD;
    int v[SCAN_PER_THREAD];
    int sum = 0;
    if (base + SCAN_PER_THREAD <= n) {   // chunks start on 8-word boundaries of a 256-byte aligned table
        const int4 lo = *reinterpret_cast<const int4*>(cnt + base), hi = *reinterpret_cast<const int4*>(cnt + base + 4);
        v[0] = lo.x; v[1] = lo.y; v[2] = lo.z; v[3] = lo.w;
        v[4] = hi.x; v[5] = hi.y; v[6] = hi.z; v[7] = hi.w;
    } else {
#pragma unroll
        for (int q = 0; q < SCAN_PER_THREAD; ++q) v[q] = base + q < n ? cnt[base + q] : 0;
    }
    int before = 0;
    for (int k = threadIdx.x; k < (int)blockIdx.x; k += BLOCK) before += bsum[k];
#pragma unroll
    for (int q = 0; q < SCAN_PER_THREAD; ++q) sum += v[q];
    before = wave_sum(before);
    if ((threadIdx.x & (WAVE - 1)) == 0) psum[threadIdx.x >> 6] = before;
    int tot;
    int run = block_excl_scan(sum, &tot);   // (its barriers also publish psum)
    before = (psum[0] + psum[1]) + (psum[2] + psum[3]);
    run += before;
    if (base + SCAN_PER_THREAD <= n) {
        int w[SCAN_PER_THREAD];
#pragma unroll
        for (int q = 0; q < SCAN_PER_THREAD; ++q) {
            w[q] = run;
            run += v[q];
        }
        *reinterpret_cast<int4*>(start + base) = make_int4(w[0], w[1], w[2], w[3]);
        *reinterpret_cast<int4*>(start + base + 4) = make_int4(w[4], w[5], w[6], w[7]);
    } else {
#pragma unroll
        for (int q = 0; q < SCAN_PER_THREAD; ++q) {
            if (base + q < n) start[base + q] = run;
            run += v[q];
        }
    }
    if ((int)blockIdx.x == nb - 1 && threadIdx.x == 0) start[n] = before + tot;
}

// Runs of equal keys among the valid lanes of a wave (valid lanes form a prefix of the wave).
// Particles arrive in the previous step's cell order, so runs are ~ one cell long and one
// atomic per run replaces one per particle.
struct KeyRun {
    bool head;   // first lane of its run
    int len;     // run length (head lanes)
    int head_lane;
};

__device__ __forceinline__ KeyRun key_run(int k, bool valid) {
    const int lane = threadIdx.x & (WAVE - 1);
    int prev = __shfl_up(k, 1, WAVE);
    bool head = valid && (lane == 0 || prev != k);
    unsigned long long heads = __ballot(head);
    int nvalid = __popcll(__ballot(valid));
    unsigned long long above = lane == WAVE - 1 ? 0ull : (heads & (~0ull << (lane + 1)));
    int next = above ? __ffsll((long long)above) - 1 : WAVE;
    KeyRun r;
    r.head = head;
    r.len = (next < nvalid ? next : nvalid) - lane;
    unsigned long long upto = lane == WAVE - 1 ? heads : (heads & ((2ull << lane) - 1));
    r.head_lane = upto ? WAVE - 1 - __clzll((long long)upto) : lane;
    return r;
}

// Position of a particle after dt and its domain clamp: advect_position (framework.py:117-136) +
// enforce_boundary (boundary.py:27-91); p and the velocity are updated in place.
struct AdvectArgs {
    float dt, L0, L1, L2, pad;
    float* vel;
    const float* sdom;   // independent scenes: domain size of each scene
};
__device__ __forceinline__ void advect(const AdvectArgs& a, int i, int scene, float4& p) {
    float v[3] = {a.vel[3 * i + 0], a.vel[3 * i + 1], a.vel[3 * i + 2]};
    float x[3] = {p.x + a.dt * v[0], p.y + a.dt * v[1], p.z + a.dt * v[2]};
    float L[3] = {a.L0, a.L1, a.L2};
    if (a.sdom) {
        L[0] = a.sdom[3 * scene + 0]; L[1] = a.sdom[3 * scene + 1]; L[2] = a.sdom[3 * scene + 2];
    }
    float nrm[3] = {0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int q = 0; q < 3; ++q) {
        if (x[q] > L[q] - a.pad) { nrm[q] = nrm[q] + 1.0f; x[q] = L[q] - a.pad; }
        if (x[q] <= a.pad) { nrm[q] = nrm[q] + -1.0f; x[q] = a.pad; }
    }
    float len = len3(nrm[0], nrm[1], nrm[2]);
    if (len > 1e-6f) {
        float c0 = nrm[0] / len, c1 = nrm[1] / len, c2 = nrm[2] / len;
        float s = (1.0f + 0.5f) * (v[0] * c0 + v[1] * c1 + v[2] * c2);
        a.vel[3 * i + 0] = v[0] - s * c0;
        a.vel[3 * i + 1] = v[1] - s * c1;
        a.vel[3 * i + 2] = v[2] - s * c2;
    }
    p = make_float4(x[0], x[1], x[2], p.w);
}

__global__ __launch_bounds__(BLOCK) void k_advect_boundary(int nd, AdvectArgs a, float4* __restrict__ pos,
                                                           const int* __restrict__ sid) {
    int i = blockIdx.x * BLOCK + threadIdx.x;
    if (i >= nd) return;
    float4 p = pos[i];
    advect(a, i, a.sdom ? sid[i] : 0, p);
    pos[i] = p;
}

struct KeysArgs {
    int count;
    float4* pos;
    Grid g;
    const Grid* grids;   // independent scenes: particle i uses the grid of its scene, grids[sid[i]]
    const int* sid;
    int* key;
    int* ccount;
    int* bsum;           // particles per SCAN_CHUNK cells (k_cell_starts), or nullptr
    int* clear_flag;     // zeroed if set: the build's overflow flags, set only by passes after this one
    AdvectArgs adv;
};

constexpr int KEY_SLOTS = 32;    // chunks that a block adds up itself
constexpr int KEY_ROUNDS = 8;    // chunks of one wave

// Cell keys and counts; with ADVECT the particle first moves (the step's advection reads and writes
// the position that its key needs).
template <bool SCENES, bool ADVECT>
__global__ __launch_bounds__(BLOCK) void k_keys(KeysArgs a) {
    int i = blockIdx.x * BLOCK + threadIdx.x;
    if (a.clear_flag && i == 0) *a.clear_flag = 0;
    bool valid = i < a.count;
    int k = -1;
    if (valid) {
        const int scene = SCENES ? a.sid[i] : 0;
        const Grid g = SCENES ? a.grids[scene] : a.g;
        float4 p = a.pos[i];
        if (ADVECT) {
            advect(a.adv, i, scene, p);
            a.pos[i] = p;
        }
        k = cell_key(g, cell_coord(g, p.x, 0), cell_coord(g, p.y, 1), cell_coord(g, p.z, 2));
        a.key[i] = k;
    }
    KeyRun r = key_run(k, valid);
    if (r.head) atomicAdd(&a.ccount[k], r.len);
    if (a.bsum) {
        // chunk totals: a block's particles lie in a few chunks, but rarely in runs (every second one of a
        // lattice crosses into the next row of cells at once), so each wave adds up its own, one chunk a
        // round, into the block's table, and a chunk takes one global atomic per block.  1M rows: 6 us without
        // totals, 26 with an atomic per wave for the first particle's chunk; with one per block for that chunk
        // and one per run for the others 19 us on a disordered state, but 35 on average and 153 at most in the
        // dam break's steps; so 16.
        __shared__ int tag[KEY_SLOTS], num[KEY_SLOTS];
        if (threadIdx.x < KEY_SLOTS) {
            tag[threadIdx.x] = -1;
            num[threadIdx.x] = 0;
        }
        __syncthreads();
        const int c = valid ? k / SCAN_CHUNK : -1;
        const int lane = (int)(threadIdx.x & (WAVE - 1));
        unsigned long long rest = __ballot(valid);
        for (int t = 0; rest && t < KEY_ROUNDS; ++t) {
            const int lead = (int)__builtin_ctzll(rest);
            const int c0 = __builtin_amdgcn_readlane(c, lead);
            const unsigned long long m = __ballot(c == c0);
            rest &= ~m;
            if (lane == lead) {
                const int q = c0 % KEY_SLOTS, n = (int)__popcll(m);
                const int old = atomicCAS(&tag[q], -1, c0);
                atomicAdd(old == -1 || old == c0 ? &num[q] : &a.bsum[c0], n);
            }
        }
        if (rest) {   // particles in no order: an atomic per run
            KeyRun t = key_run(c, valid);
            if (t.head && ((rest >> lane) & 1ull)) atomicAdd(&a.bsum[c], t.len);
        }
        __syncthreads();
        if (threadIdx.x < KEY_SLOTS && num[threadIdx.x] > 0) atomicAdd(&a.bsum[tag[threadIdx.x]], num[threadIdx.x]);
    }
}

// slot = start[key] + (remaining count - 1); leaves ccount at zero for the next sort.  A run's
// head takes the run's slots with one atomic and its lanes take them in order.  The slot receives
// the particle's user id (the ranking below compares user ids within a cell).
__global__ __launch_bounds__(BLOCK) void k_scatter(int count, const int* __restrict__ key,
                                                   const int* __restrict__ start, int* __restrict__ ccount,
                                                   const int* __restrict__ uid, int* __restrict__ cell_uid) {
    int i = blockIdx.x * BLOCK + threadIdx.x;
    bool valid = i < count;
    int k = valid ? key[i] : -1;
    KeyRun r = key_run(k, valid);
    int old = 0;
    if (r.head) old = atomicSub(&ccount[k], r.len);
    old = __shfl(old, r.head_lane, WAVE);
    if (valid) {
        int lane = threadIdx.x & (WAVE - 1);
        int slot = start[k] + old - 1 - (lane - r.head_lane);
        cell_uid[slot] = uid[i];
    }
}

struct PlaceArgs {
    int count, offset;
    const int* key;
    const int* start;
    const int* cell_uid;
    int* bsum;   // chunk totals cleared for the next sort (nullptr: not used)
    int nb;
    const float4* pos; float4* pos_b;
    const float* vel; float* vel_b;
    const float* minv; float* minv_b;
    const float* rho0; float* rho0_b;
    const int* mat; int* mat_b;
    const int* uid; int* uid_b;
    int* inv;
    const float* divg; float* divg_b;
};

// Final place of particle i = cell start + number of cell members with a smaller user id, and its
// arrays moved there.  Particles arrive in the previous step's cell order, so the writes of a wave
// stay close together; ranking and a gather by the inverse order took two launches and the order
// array (1M rows: 7 + 27 us against 25; 8k rows 3.2 + 4.0 against 3.7).
template <bool VEL>
__global__ __launch_bounds__(BLOCK) void k_place(PlaceArgs a) {
    int i = blockIdx.x * BLOCK + threadIdx.x;
    if (a.bsum)
        for (int q = i; q < a.nb; q += (int)gridDim.x * BLOCK) a.bsum[q] = 0;
    if (i >= a.count) return;
    const int src = a.offset + i;
    const int u = a.uid[src];
    const int k = a.key[i];
    const float4 p = a.pos[src];
    const float minv = a.minv[src], rho0 = a.rho0[src];
    const int mat = a.mat[src];
    float v0 = 0.0f, v1 = 0.0f, v2 = 0.0f, dv = 0.0f;
    if (VEL) {
        v0 = a.vel[3 * src + 0]; v1 = a.vel[3 * src + 1]; v2 = a.vel[3 * src + 2];
        dv = a.divg[src];
    }
    const int lo = a.start[k], hi = a.start[k + 1];
    int rank = 0;
#pragma unroll 4
    for (int s = lo; s < hi; ++s) rank += a.cell_uid[s] < u ? 1 : 0;
    const int dst = a.offset + lo + rank;
    a.pos_b[dst] = p;
    if (VEL) {
        a.vel_b[3 * dst + 0] = v0;
        a.vel_b[3 * dst + 1] = v1;
        a.vel_b[3 * dst + 2] = v2;
        a.divg_b[dst] = dv;
    }
    a.minv_b[dst] = minv;
    a.rho0_b[dst] = rho0;
    a.mat_b[dst] = mat;
    a.uid_b[dst] = u;
    a.inv[u] = dst;
}

// ---- neighbour enumeration ---------------------------------------------------------------
// Visits, in order, every particle j of one population (dynamic or static) with j != self and
// sqrtf(dx*dx + dy*dy + dz*dz) < h -- the reference predicate, neighbour_search.py:34-44 --
// over the 9 contiguous (cx-1..cx+1) runs of the 3x3 (dz, dy) stencil.  Within a population the
// visit order is ascending (cell key, user id).
template <class F>
__device__ __forceinline__ void visit(const Grid& g, const int* __restrict__ start, const float4* __restrict__ ppos,
                                      int self, float4 pi, float h, F&& f) {
    int cx = cell_coord(g, pi.x, 0), cy = cell_coord(g, pi.y, 1), cz = cell_coord(g, pi.z, 2);
    int x0 = cx > 0 ? cx - 1 : 0;
    int x1 = cx < g.dims[0] - 1 ? cx + 1 : g.dims[0] - 1;
    for (int dz = -1; dz <= 1; ++dz) {
        int zz = cz + dz;
        if (zz < 0 || zz >= g.dims[2]) continue;
        for (int dy = -1; dy <= 1; ++dy) {
            int yy = cy + dy;
            if (yy < 0 || yy >= g.dims[1]) continue;
            int s0 = start[cell_key(g, x0, yy, zz)];
            int s1 = start[cell_key(g, x1, yy, zz) + 1];
            for (int j = s0; j < s1; ++j) {
                if (j == self) continue;
                float4 pj = ppos[j];
                float rx = pi.x - pj.x, ry = pi.y - pj.y, rz = pi.z - pj.z;
                float rn = len3(rx, ry, rz);
                if (rn < h) f(j, pj, rx, ry, rz, rn);
            }
        }
    }
}

// Candidate scan of one population: calls f(j) for every j != self with
// sqrtf(dx*dx + dy*dy + dz*dz) < h, in the order of `visit`.  The predicate is decided without
// the square root outside a few-ulp band around h^2: d^2 < h2_lo = h^2 (1 - 2^-20) implies
// sqrtf(d^2) < h, and d^2 >= h2_hi = h^2 (1 + 2^-20) implies sqrtf(d^2) >= h.  The correctly
// rounded root runs only when some lane of the wave has a candidate inside the band (a uniform
// branch, so the common case carries no root at all).  Candidates are loaded two at a time.
template <class F>
__device__ __forceinline__ void scan_ids(const Grid& g, const int* __restrict__ start, const float4* __restrict__ ppos,
                                         int self, float4 pi, float h, float h2_lo, float h2_hi, F&& f) {
    int cx = cell_coord(g, pi.x, 0), cy = cell_coord(g, pi.y, 1), cz = cell_coord(g, pi.z, 2);
    int x0 = cx > 0 ? cx - 1 : 0;
    int x1 = cx < g.dims[0] - 1 ? cx + 1 : g.dims[0] - 1;
    auto test = [&](int j, float4 pj) {
        float rx = pi.x - pj.x, ry = pi.y - pj.y, rz = pi.z - pj.z;
        float d2 = rx * rx + ry * ry + rz * rz;
        bool in = d2 < h2_lo;
        bool band = !in && d2 < h2_hi;
        if (__ballot(band)) {
            if (band) {
                // the empty volatile asm keeps the root inside this branch (it would otherwise be
                // evaluated speculatively for every candidate)
                float d = d2;
                asm volatile("" : "+v"(d));
                in = sqrtf(d) < h;
            }
        }
        if (in && j != self) f(j);
    };
    for (int dz = -1; dz <= 1; ++dz) {
        int zz = cz + dz;
        if (zz < 0 || zz >= g.dims[2]) continue;
        for (int dy = -1; dy <= 1; ++dy) {
            int yy = cy + dy;
            if (yy < 0 || yy >= g.dims[1]) continue;
            int s0 = start[cell_key(g, x0, yy, zz)];
            int s1 = start[cell_key(g, x1, yy, zz) + 1];
            for (int j = s0; j < s1; j += 2) {
                int j1 = j + 1 < s1 ? j + 1 : j;
                float4 p0 = ppos[j];
                float4 p1 = ppos[j1];
                __builtin_amdgcn_sched_barrier(0);   // both loads in flight before the first test
                test(j, p0);
                if (j + 1 < s1) test(j1, p1);
            }
        }
    }
}

struct BuildArgs {
    int nd, ns, C, Cs;
    float h, h2_lo, h2_hi;
    float h2;       // h^2 rounded to float32 (the matrix-core distances)
    float kc, ks;   // cubic and spiky kernel constants
    float inv_h;    // 1 / h rounded to nearest (div_rn)
    float inv_gs;   // 1 / scale of float16 gradW records (a power of two)
    Grid g;
    const Grid* grids;   // independent scenes: grid of each scene, indexed by sid
    const int* sid;
    const float4* pos;
    const float* minv;
    const int* dstart;
    const int* sstart;
    uint32_t* nb;
    uint32_t* g16;   // float16 format: gradW / scale as two half-pair words at twice each id's word
    int* tile_len;
    int* wave_len;
    int* rowcnt;
    int* rowtot;
    float* density;
    float* kk;
    float* Ss;
    int* err_flag;
    double* partials;
    int stride;
    // tile windows (k_eval4 with PPT > 0)
    int win_cap;   // largest window kept, <= WIN_MAX
    uint32_t* loc;
    int* win_ids;
    int* win_n;
};

// One thread per dynamic row, one wave per 64-row tile, two phases.
//  A: candidate scan; the ids of dynamic neighbours go to slots 0, 1, ... of the row and the
//     ids of static neighbours to slots Cs-1, Cs-2, ... (a row with more than C neighbours sets
//     the error flag).
//  B: the wave walks its slots in lockstep, computing gradW (stored next to the id, coalesced),
//     density (pressure_base.py:12-46), Aii (pressure_base.py:49-87) and S_i, accumulated in the
//     reference row order: dynamic neighbours, then static neighbours.  Dynamic slots from the
//     row's count up to the tile length -- the wave's longest row rounded up to ROW_PAD slots
//     -- are padded with (id = row, gradW = 0).
// FMT is the row format (include/ivp.h): ids only, ids + float32 gradW, or ids + float16 gradW
// scaled by 1/inv_gs, packed as (gx, gy) and (gz, 0) half pairs.
template <int FMT>
constexpr unsigned rec_words() { return FMT == IVP_ROWS_F32 ? 256u : 64u; }

// Phase B of the build for the wave's 64-row tile (one thread per row, lane = row's place in the
// tile); cnt / cs / tot are the row's stored dynamic and static slots and its neighbour total.
template <int FMT>
__device__ __forceinline__ void build_eval(const BuildArgs& a, int i, int lane, int tile, bool valid, float4 pi,
                                           int cnt, int cs, int tot);

template <int FMT, bool SCENES>
__global__ __launch_bounds__(BLOCK) void k_build(BuildArgs a) {
    constexpr unsigned REC = rec_words<FMT>();
    int blk = xcd_block(blockIdx.x, gridDim.x);
    int i = blk * BLOCK + threadIdx.x;
    int lane = threadIdx.x & (WAVE - 1);
    int tile = i >> 6;
    bool valid = i < a.nd;
    const float h = a.h;
    const int C = a.C, Cs = a.Cs;
    uint32_t* tbase = a.nb + (size_t)tile * (size_t)Cs * REC + row_word0<REC>(lane);
    int cnt = 0, cs = 0, tot = 0;
    float4 pi = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    if (valid) {
        pi = a.pos[i];
        const Grid g = SCENES ? a.grids[a.sid[i]] : a.g;
        scan_ids(g, a.dstart, a.pos, i, pi, h, a.h2_lo, a.h2_hi, [&](int j) {
            if (tot < C) tbase[slot_word<REC>(cnt)] = (uint32_t)j;
            if (tot < C) cnt++;
            tot++;
        });
        scan_ids(g, a.sstart, a.pos + a.nd, -1, pi, h, a.h2_lo, a.h2_hi, [&](int j) {
            if (tot < C) tbase[slot_word<REC>(Cs - 1 - cs)] = (uint32_t)j;
            if (tot < C) cs++;
            tot++;
        });
        if (tot > C) atomicOr(a.err_flag, 1);
    }
    build_eval<FMT>(a, i, lane, tile, valid, pi, cnt, cs, tot);
}

// Predicate codes of the wave-mask compare builtins (LLVM's CmpInst numbering)
constexpr int FCMP_OLT = 4, ICMP_NE = 33, ICMP_ULT = 36;

// Candidate scan of one population with G lanes per row: lane g of the row's group tests the
// candidates s0 + g, s0 + g + G, ... of every run, U batches in flight; the group's ballot
// ranks the hits, so slots fill in the order of the one-lane scan (ascending candidate index).
// `put(j, rank_in_batch, hits_before_batch)` stores a hit; returns the number of hits.
// A batch loads its G * U candidates unconditionally: entries past the run's end (at most
// G * U - 1 <= POS_PAD - 1 past the last particle) lie inside the padded position buffer and are
// masked by j < s1.  The predicate is decided as in scan_ids, on d2 formed with fused
// multiply-adds: that d2 is within 5 * 2^-24 (relative) of the unfused d2 of the reference's
// expression, far inside the 2^-20 margins of h2_lo and h2_hi, so outside the band both give
// the same answer; inside the band the unfused d2 is formed again and the correctly rounded root
// decides, exactly as in scan_ids.
template <int G, int U, class P>
__device__ __forceinline__ int scan_group(const Grid& g, const int* __restrict__ start,
                                          const float4* __restrict__ ppos, int self, float4 pi, float h, float h2_lo,
                                          float h2_hi, int gl, P&& put) {
    const int cx = cell_coord(g, pi.x, 0), cy = cell_coord(g, pi.y, 1), cz = cell_coord(g, pi.z, 2);
    const int x0 = cx > 0 ? cx - 1 : 0;
    const int x1 = cx < g.dims[0] - 1 ? cx + 1 : g.dims[0] - 1;
    const int wl = (int)(threadIdx.x & (WAVE - 1));
    const int base = wl & ~(G - 1);
    static_assert(G <= 8 && G * U <= POS_PAD, "16 lanes take scan_row16; a batch stays inside the position buffer's pad");
    const unsigned long long gmask = (1ull << G) - 1ull;
    const unsigned long long below = (1ull << gl) - 1ull;
    int found = 0;
    for (int dz = -1; dz <= 1; ++dz) {
        int zz = cz + dz;
        if (zz < 0 || zz >= g.dims[2]) continue;
        for (int dy = -1; dy <= 1; ++dy) {
            int yy = cy + dy;
            if (yy < 0 || yy >= g.dims[1]) continue;
            const int s0 = start[cell_key(g, x0, yy, zz)];
            const int s1 = start[cell_key(g, x1, yy, zz) + 1];
            for (int b = s0; b < s1; b += G * U) {
                const float4* q = ppos + (b + gl);
                float4 p[U];
#pragma unroll
                for (int u = 0; u < U; ++u) p[u] = q[u * G];
                __builtin_amdgcn_sched_barrier(0);   // every load of the batch in flight before the tests
#pragma unroll
                for (int u = 0; u < U; ++u) {
                    const int j = b + u * G + gl;
                    float rx = pi.x - p[u].x, ry = pi.y - p[u].y, rz = pi.z - p[u].z;
                    float d2 = fmaf(rz, rz, fmaf(ry, ry, rx * rx));
                    // wave masks straight from the compares: valid candidates (inside the run, not
                    // the row itself), those inside h2_lo, and those in the band [h2_lo, h2_hi)
                    const unsigned long long valid = __builtin_amdgcn_uicmp((unsigned)j, (unsigned)s1, ICMP_ULT) &
                                                     __builtin_amdgcn_uicmp((unsigned)j, (unsigned)self, ICMP_NE);
                    unsigned long long hit = __builtin_amdgcn_fcmpf(d2, h2_lo, FCMP_OLT) & valid;
                    const unsigned long long band = (__builtin_amdgcn_fcmpf(d2, h2_hi, FCMP_OLT) & valid) & ~hit;
                    if (band) {
                        bool in = false;
                        if ((band >> wl) & 1ull) {
                            float d = rx * rx + ry * ry + rz * rz;
                            asm volatile("" : "+v"(d));
                            in = sqrtf(d) < h;
                        }
                        hit |= __builtin_amdgcn_ballot_w64(in);
                    }
                    const unsigned long long m = (hit >> base) & gmask;
                    if ((m >> gl) & 1ull) put(j, __popcll(m & below), found);
                    found += __popcll(m);
                }
            }
        }
    }
    return found;
}

// Lane K of each 16-lane row to the whole row
template <int K>
__device__ __forceinline__ int row_bcast(int v) {
    return __builtin_amdgcn_update_dpp(0, v, 0x150 + K, 0xf, 0xf, true);
}

// scan_group with 16 lanes per row (one DPP row), for counts that leave a SIMD a few waves: a run after
// another, the scan waited for two bounds and one or two candidate batches nine times over.  Here
// lanes 0 to 8 load the nine runs' bounds at once, and the runs end to end -- candidate v of run k is
// particle v + rb[k], its run found by eight compares -- go through in batches of 16 with UL of them in
// flight: 4k rows 12.2 -> 8.8 us alone, 8k 13.8 -> 10 (12 or 17 batches in flight: 9.6 and 10 at 4k; more
// registers and code than the few waves hide).  Same order, same decisions, same ranks.
constexpr int SCAN16_BATCHES = 8;   // batches in flight
struct Row16Runs {
    int s0, end;   // lane k < 9 of the row: run k's candidates [s0, end)
};
__device__ __forceinline__ Row16Runs row16_runs(const Grid& g, const int* __restrict__ start, bool on, float4 pi, int gl) {
    const int cx = cell_coord(g, pi.x, 0), cy = cell_coord(g, pi.y, 1), cz = cell_coord(g, pi.z, 2);
    const int x0 = cx > 0 ? cx - 1 : 0;
    const int x1 = cx < g.dims[0] - 1 ? cx + 1 : g.dims[0] - 1;
    // run gl = 3 (dz + 1) + (dy + 1)
    const int yy = cy + gl % 3 - 1, zz = cz + gl / 3 - 1;
    Row16Runs r = {0, 0};
    if (on && gl < 9 && yy >= 0 && yy < g.dims[1] && zz >= 0 && zz < g.dims[2]) {
        r.s0 = start[cell_key(g, x0, yy, zz)];
        r.end = start[cell_key(g, x1, yy, zz) + 1];
    }
    return r;
}

template <int UL, class P>
__device__ __forceinline__ int scan_row16(const float4* __restrict__ ppos, Row16Runs runs, int self, float4 pi, float h,
                                          float h2_lo, float h2_hi, int gl, P&& put) {
    const int wl = (int)(threadIdx.x & (WAVE - 1));
    const int base = wl & ~15;
    const uint32_t below = (1u << gl) - 1u;
    const int s0 = runs.s0, len = runs.end - runs.s0;
    int end = len;   // inclusive prefix over the row
    end += __builtin_amdgcn_update_dpp(0, end, 0x111, 0xf, 0xf, true);
    end += __builtin_amdgcn_update_dpp(0, end, 0x112, 0xf, 0xf, true);
    end += __builtin_amdgcn_update_dpp(0, end, 0x114, 0xf, 0xf, true);
    end += __builtin_amdgcn_update_dpp(0, end, 0x118, 0xf, 0xf, true);
    const int off = s0 - (end - len);
    const int T = row_bcast<8>(end);
    const int e[8] = {row_bcast<0>(end), row_bcast<1>(end), row_bcast<2>(end), row_bcast<3>(end),
                      row_bcast<4>(end), row_bcast<5>(end), row_bcast<6>(end), row_bcast<7>(end)};
    const int rb[9] = {row_bcast<0>(off), row_bcast<1>(off), row_bcast<2>(off), row_bcast<3>(off), row_bcast<4>(off),
                       row_bcast<5>(off), row_bcast<6>(off), row_bcast<7>(off), row_bcast<8>(off)};
    const int most = wave_max(T);   // the wave's four rows go through together
    int found = 0;
    for (int cb = 0; cb < most; cb += 16 * UL) {
        int j[UL];
        float4 p[UL];
#pragma unroll
        for (int u = 0; u < UL; ++u) {
            const int v = cb + 16 * u + gl;
            int o = rb[0];
#pragma unroll
            for (int k = 0; k < 8; ++k) o = v >= e[k] ? rb[k + 1] : o;
            j[u] = v < T ? v + o : -1;
            if (j[u] >= 0) p[u] = ppos[j[u]];
        }
        __builtin_amdgcn_sched_barrier(0);   // every load of the chunk in flight before the tests
#pragma unroll
        for (int u = 0; u < UL; ++u) {
            if (cb + 16 * u >= most) break;
            float rx = pi.x - p[u].x, ry = pi.y - p[u].y, rz = pi.z - p[u].z;
            float d2 = fmaf(rz, rz, fmaf(ry, ry, rx * rx));
            const bool valid = j[u] >= 0 && j[u] != self;
            bool in = valid && d2 < h2_lo;
            const bool band = valid && !in && d2 < h2_hi;
            if (__builtin_amdgcn_ballot_w64(band)) {
                if (band) {
                    float d = rx * rx + ry * ry + rz * rz;
                    asm volatile("" : "+v"(d));
                    in = sqrtf(d) < h;
                }
            }
            const uint32_t m = (uint32_t)(__builtin_amdgcn_ballot_w64(in) >> base) & 0xffffu;
            if (in) put(j[u], __popc(m & below), found);
            found += __popc(m);
        }
    }
    return found;
}

// Phase A alone with G lanes per row (threads = rows x G): ids into the rows' slots exactly as
// k_build's scan stores them, the row's dynamic slot count into rowcnt and its neighbour total
// into rowtot.  For particle counts that leave few waves per SIMD, where the one-lane scan is a
// chain of dependent load rounds.
template <int FMT, bool SCENES, int G>
__global__ __launch_bounds__(BLOCK) void k_scan(BuildArgs a) {
    constexpr unsigned REC = rec_words<FMT>();
    constexpr int U = G == 2 ? 4 : G == 4 ? 2 : 1;   // batches in flight (measured best per G)
    const int blk = xcd_block(blockIdx.x, gridDim.x);
    const int i = blk * (BLOCK / G) + (int)(threadIdx.x / G);
    const int gl = (int)(threadIdx.x % G);
    const bool on = i < a.nd;
    if (G != 16 && !on) return;   // the G lanes of a row leave together (scan_row16 takes whole waves)
    const int C = a.C, Cs = a.Cs;
    // the wave's rows share one 64-row tile (64 / G rows from a multiple of 64 / G); slot k of the
    // row is word row_word0(lane) + slot_word(k) of the tile, a 32-bit index from the tile's
    // (uniform) base
    uint32_t* tnb = a.nb + (size_t)__builtin_amdgcn_readfirstlane(i >> 6) * (size_t)Cs * REC;
    const uint32_t w0 = row_word0<REC>(i & (WAVE - 1));
    const int ic = on ? i : a.nd - 1;
    const float4 pi = a.pos[ic];
    const Grid g = SCENES ? a.grids[a.sid[ic]] : a.g;
    // the k-th neighbour found (dynamic ones first) is stored when k < C
    Row16Runs rd = {0, 0}, rs = {0, 0};
    if constexpr (G == 16) {   // both populations' bounds in flight together
        rd = row16_runs(g, a.dstart, on, pi, gl);
        rs = row16_runs(g, a.sstart, on, pi, gl);
        __builtin_amdgcn_sched_barrier(0);
    }
    auto scan = [&](const int* start, const float4* ppos, int self, auto&& put) {
        if constexpr (G == 16)
            return scan_row16<SCAN16_BATCHES>(ppos, self >= 0 ? rd : rs, self, pi, a.h, a.h2_lo, a.h2_hi, gl, put);
        else
            return scan_group<G, U>(g, start, ppos, self, pi, a.h, a.h2_lo, a.h2_hi, gl, put);
    };
    int nd_found = scan(a.dstart, a.pos, i, [&](int j, int rank, int before) {
        if (before + rank < C) tnb[slot_word<REC>(before + rank) + w0] = (uint32_t)j;
    });
    int ns_found = scan(a.sstart, a.pos + a.nd, -1, [&](int j, int rank, int before) {
        const int k = nd_found + before + rank;
        if (k < C) tnb[slot_word<REC>(Cs - 1 - (before + rank)) + w0] = (uint32_t)j;
    });
    if (on && gl == 0) {
        const int tot = nd_found + ns_found;
        a.rowcnt[i] = nd_found < C ? nd_found : C;
        a.rowtot[i] = tot;
        if (tot > C) atomicOr(a.err_flag, 1);
    }
}

// Candidate scan by cells (ids-only and float16 rows; one grid or a grid per scene).  A wave takes
// SCAN_ROWS consecutive rows of its block's 64-row tile and cuts them into segments: rows of one
// (y, z) cell row (and scene) within SCAN_SPAN + 1 cells along x.  The rows of a segment share nine
// candidate runs (scan_ids' runs of the 3x3 (y, z) neighbour cells, each widened to the cells
// x_first - 1 .. x_last + 1): a candidate outside a row's own 3x3x3 cells lies a cell width > h away,
// so the wider runs add no neighbour, and the runs end to end keep scan_ids' visiting order.
//
// Distances come from the matrix cores: with a = x_row - o and b = x_candidate - o about the
// segment's centre o, e = |x_row - x_cand|^2 - h^2 = |b|^2 - 2 a.b + (|a|^2 - h^2) is one
// 16x16x4 float32 product of candidates (b, |b|^2) and rows (-2 a, 1) with |a|^2 - h^2 as the
// accumulator's start.  Lane (q, n) of the wave then holds e of row n against 16 candidates per
// batch of 64 -- the candidates of its quarter q of the chunk -- and collects the sign bits.  The
// product's rounding is below 2e-5 h^2 (coordinates within 4 h of o; a segment that holds a
// farther one takes the exact test throughout), so outside |e| < 2^-14 h^2 the sign decides
// sqrtf(d^2) < h as scan_ids does; inside the band the candidate's unfused d^2 and its correctly
// rounded root decide.  A row's quarters are ranked by their hit counts, so the slots fill in the
// one-lane order.
//
// What bounds it: vector instruction issue.  One row at a time with a candidate per lane the scan
// took 14 vector instructions per 64 candidate tests (differences, square, two compares, rank,
// store address); here a test is one sixteenth of a matrix instruction, one funnel shift for the
// mask and half a minimum for the band, and only hits cost a store: 112 -> 75 million vector
// instructions per 1M-row build, 196 -> 150 us (102k rows 33 -> 29, 64 scenes of 1.25M rows 235 ->
// 200).
//
// The slots are collected in LDS (per row Cs words and 4 spare against bank conflicts; each wave
// owns its rows, so no block barrier) and written out as whole 8-slot blocks of the paired
// layout, 512 contiguous bytes per wave and block; words of a written block between the row's
// dynamic [0, cnt) and static [Cs - cs, Cs) ranges get the row's own id, as the exact pass pads.
constexpr int SCAN_ROWS = 16;     // rows per wave: a block's four waves cover its tile
constexpr int SCAN_BATCHES = 4;   // candidate batches of 64 held in registers per chunk
constexpr int SCAN_SPAN = 3;      // a segment's last cell lies at most this many cells past its first
// LDS words of one wave: candidate ids of a chunk, then one batch's candidate records
// (x, y, z, |b|^2), 16 per quarter with the quarters 80 words apart: the 64 lanes' reads of one
// component (candidate 4 t + (n & 3) of quarter n >> 2, component q) hit 64 different banks
constexpr int SCAN_IDS = WAVE * SCAN_BATCHES;
constexpr int SCAN_QUARTER = 80;
constexpr int SCAN_WAVE_LDS = SCAN_IDS + 4 * SCAN_QUARTER;

__device__ __forceinline__ void wave_lds_sync() {
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// The candidate runs of a segment's cells (cx0 .. cx1, cy, cz), both populations at once: lane
// 16 p + k (k < 9) loads population p's run k = 3 (dz + 1) + (dy + 1), the cells cx0 - 1 .. cx1 + 1 of
// row y + dy, layer z + dz (empty outside the grid).  Returns, per lane, the exclusive prefix of
// the run lengths within its population (rp) and the run's first particle minus it (rb: candidate
// v of run k is particle v + rb); lane 16 p + 8 also returns the population's total in T.
struct SegRuns {
    int rp, rb, T;
};
__device__ __forceinline__ SegRuns seg_runs(const BuildArgs& a, const Grid& g, int cx0, int cx1, int cy, int cz) {
    const int lane = (int)(threadIdx.x & (WAVE - 1));
    const int pop = lane >> 4, k = lane & 15;
    const int zz = cz + k / 3 - 1, yy = cy + k % 3 - 1;
    const bool live = pop < 2 && k < 9 && zz >= 0 && zz < g.dims[2] && yy >= 0 && yy < g.dims[1];
    const int x0 = cx0 > 0 ? cx0 - 1 : 0;
    const int x1 = cx1 < g.dims[0] - 1 ? cx1 + 1 : g.dims[0] - 1;
    int s0 = 0, n = 0;
    if (live) {
        const int* start = pop == 0 ? a.dstart : a.sstart;
        s0 = start[cell_key(g, x0, yy, zz)];
        n = start[cell_key(g, x1, yy, zz) + 1] - s0;
    }
    // inclusive prefix over the 16 lanes of the population (DPP row shifts stay inside a row of
    // 16 lanes and bring in 0 from outside it)
    int inc = n;
    inc += __builtin_amdgcn_update_dpp(0, inc, 0x111, 0xf, 0xf, false);   // row_shr:1
    inc += __builtin_amdgcn_update_dpp(0, inc, 0x112, 0xf, 0xf, false);   // row_shr:2
    inc += __builtin_amdgcn_update_dpp(0, inc, 0x114, 0xf, 0xf, false);   // row_shr:4
    inc += __builtin_amdgcn_update_dpp(0, inc, 0x118, 0xf, 0xf, false);   // row_shr:8
    return SegRuns{inc - n, s0 - (inc - n), inc};
}

// The hits of one chunk decided from the positions as scan_ids decides them, for a segment with far
// coordinates (particles outside the grid are in its border cells, at any distance).  A batch's positions go
// to the LDS, where a lane reads the 16 of its quarter: gathered through the ids one after another
// they took twice as long as the rest (104k rows, all outside the grid: build 526 -> 229 us; a third of
// them 150 -> 107).
__device__ __forceinline__ void far_chunk(const BuildArgs& a, const float4* __restrict__ ppos, const uint32_t* ids,
                                          float* cand, int left, int nb, bool mine, float px, float py, float pz,
                                          uint32_t (&W)[2]) {
    typedef float f32x4 __attribute__((ext_vector_type(4)));
    const int lane = (int)(threadIdx.x & (WAVE - 1));
    const int q = lane >> 4, n = lane & 15;
    const int base = 16 * nb * q;
    float* cq = cand + SCAN_QUARTER * q;
    unsigned long long hits = 0ull;
#pragma unroll 1
    for (int u = 0; u < nb; ++u) {
        const int c = base + 16 * u + n;
        const float4 p = ppos[ids[c < left ? c : left - 1]];
        *reinterpret_cast<f32x4*>(cq + 4 * n) = f32x4{p.x, p.y, p.z, 0.0f};
        wave_lds_sync();
        uint32_t h = 0u, band = 0u;
#pragma unroll 4
        for (int k = 0; k < 16; ++k) {
            const f32x4 pj = *reinterpret_cast<const f32x4*>(cq + 4 * k);
            const float rx = px - pj.x, ry = py - pj.y, rz = pz - pj.z;
            const float d2 = fmaf(rz, rz, fmaf(ry, ry, rx * rx));
            h = h << 1 | (d2 < a.h2_lo ? 1u : 0u);
            band = band << 1 | (d2 < a.h2_hi ? 1u : 0u);
        }
        const int valid = left - base - 16 * u;   // candidates of this lane's 16
        const uint32_t in = !mine ? 0u : valid >= 16 ? 0xffffu : valid > 0 ? 0xffffu & ~(0xffffu >> valid) : 0u;
        h &= in;
        band &= in & ~h;
        while (__builtin_amdgcn_ballot_w64(band != 0u)) {
            if (band) {
                const int k = __clz((int)band) - 16;
                const uint32_t bit = 0x8000u >> k;
                band &= ~bit;
                const f32x4 pj = *reinterpret_cast<const f32x4*>(cq + 4 * k);
                const float rx = px - pj.x, ry = py - pj.y, rz = pz - pj.z;
                const float dd = rx * rx + ry * ry + rz * rz;
                h = sqrtf(dd) < a.h ? (h | bit) : h;
            }
        }
        wave_lds_sync();
        hits |= (unsigned long long)h << (48 - 16 * u);
    }
    W[0] = (uint32_t)(hits >> 32);
    W[1] = (uint32_t)hits;
}

// One population of a segment: rows rs .. re - 1 of the wave, whose positions lanes (q, n) hold for
// row n.  found (every lane of row n) counts row n's hits of this population; the dynamic
// population stores hit k at slot k while k < C (an overflowing row's hits past C all go to slot C,
// which no reader uses), the static one at slot Cs - 1 - k while ndf + k < C (ndf = the row's dynamic
// total; other hits go to the row's spare words).
template <bool DYN>
__device__ __forceinline__ void seg_pop_scan(const BuildArgs& a, const SegRuns& R, int T, int rs, int re, int row0,
                                             float px, float py, float pz, float3 o, int& found, int ndf,
                                             uint32_t* st, uint32_t* wl, int S) {
    typedef float f32x4 __attribute__((ext_vector_type(4)));
    constexpr int NB = SCAN_BATCHES;
    constexpr int pl = DYN ? 0 : 16;
    const int lane = (int)(threadIdx.x & (WAVE - 1));
    const int q = lane >> 4, n = lane & 15;
    const float4* __restrict__ ppos = DYN ? a.pos : a.pos + a.nd;
    uint32_t* ids = wl;
    float* cand = reinterpret_cast<float*>(wl + SCAN_IDS);
    int rb[9], rp[9];
#pragma unroll
    for (int k = 0; k < 9; ++k) {
        rp[k] = __builtin_amdgcn_readlane(R.rp, pl + k);
        rb[k] = __builtin_amdgcn_readlane(R.rb, pl + k);
    }
    const bool mine = n >= rs && n < re;
    // the row's operand (component q of (-2 a, 1)) and the accumulator's start
    const float ax = px - o.x, ay = py - o.y, az = pz - o.z;
    const float a2 = fmaf(az, az, fmaf(ay, ay, ax * ax));
    const float rowop = q == 0 ? -2.0f * ax : q == 1 ? -2.0f * ay : q == 2 ? -2.0f * az : 1.0f;
    const float c0 = a2 - a.h2;
    const f32x4 acc0 = {c0, c0, c0, c0};
    const float far2 = 16.0f * a.h2, eps = a.h2 * (1.0f / 16384.0f);
    const bool row_far = __builtin_amdgcn_ballot_w64(mine && !(a2 <= far2)) != 0ull;
    // lane (q, n) writes the record of candidate n of quarter q, and reads component q of candidate
    // 4 t + (n & 3) of quarter n >> 2
    float* cw = cand + SCAN_QUARTER * q + 4 * n;
    const float* cr = cand + SCAN_QUARTER * (n >> 2) + 4 * (n & 3) + q;
    const int lim = DYN ? a.C : (a.C - ndf > 0 ? a.C - ndf : 0);
    uint32_t* srow = st + n * S;
    for (int cb = 0; cb < T; cb += WAVE * NB) {
        const int left = T - cb < WAVE * NB ? T - cb : WAVE * NB;
        const int nb = (left + WAVE - 1) / WAVE;
        const int nbm = row_far ? 0 : nb;   // batches for the matrix cores
        // the chunk's candidate ids in visiting order, run by run
#pragma unroll
        for (int k = 0; k < 9; ++k) {
            const int v1 = k < 8 ? rp[k + 1] : T;
            const int hi = v1 < cb + left ? v1 : cb + left;
            for (int v = (rp[k] > cb ? rp[k] : cb) + lane; v < hi; v += WAVE) ids[v - cb] = (uint32_t)(v + rb[k]);
        }
        wave_lds_sync();
        const int base = 16 * nb * q;   // the quarter's first candidate, relative to cb
        float4 p[NB];
        // all batches' loads in flight together (past the end: the last candidate, never a hit)
#pragma unroll
        for (int u = 0; u < NB; ++u) {
            const int c = base + 16 * u + n;
            if (u < nbm) p[u] = ppos[ids[c < left ? c : left - 1]];
        }
        uint32_t W[2] = {0u, 0u};   // hits, first candidate in the highest bit, 32 per word
        bool far = false;           // a candidate of the chunk with far coordinates
#pragma unroll
        for (int u = 0; u < NB; ++u) {
            uint32_t w = W[u >> 1] << 16;
            if (u < nbm) {
                const float bx = p[u].x - o.x, by = p[u].y - o.y, bz = p[u].z - o.z;
                const float b2 = fmaf(bz, bz, fmaf(by, by, bx * bx));
                const f32x4 rec = {bx, by, bz, base + 16 * u + n < left ? b2 : 1e30f};
                *reinterpret_cast<f32x4*>(cw) = rec;
                wave_lds_sync();
                f32x4 d[4];
#pragma unroll
                for (int t = 0; t < 4; ++t)
                    d[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(cr[16 * t], rowop, acc0, 0, 0, 0);
                wave_lds_sync();
                uint32_t h = 0u;
                float nearest = 1e30f;
#pragma unroll
                for (int k = 0; k < 16; ++k) {
                    const float e = d[k >> 2][k & 3];
                    h = __builtin_amdgcn_alignbit(h, __float_as_uint(e), 31);   // h << 1 | sign
                    nearest = fminf(nearest, fabsf(e));
                }
                far = far || !(b2 <= far2);
                if (__builtin_amdgcn_ballot_w64(mine && nearest < eps)) {
                    // candidates in the band by the exact test
                    uint32_t band = 0u;
#pragma unroll
                    for (int k = 0; k < 16; ++k)
                        band = __builtin_amdgcn_alignbit(band, __float_as_uint(fabsf(d[k >> 2][k & 3]) - eps), 31);
                    const int valid = left - base - 16 * u;   // candidates of this lane's 16
                    const uint32_t in = valid >= 16 ? 0xffffu : valid > 0 ? 0xffffu & ~(0xffffu >> valid) : 0u;
                    band = mine ? band & in : 0u;
                    while (__builtin_amdgcn_ballot_w64(band != 0u)) {
                        if (band) {
                            const int k = __clz((int)band) - 16;
                            const uint32_t bit = 0x8000u >> k;
                            band &= ~bit;
                            const float4 pj = ppos[ids[base + 16 * u + k]];
                            const float rx = px - pj.x, ry = py - pj.y, rz = pz - pj.z;
                            const float dd = rx * rx + ry * ry + rz * rz;
                            h = sqrtf(dd) < a.h ? (h | bit) : (h & ~bit);
                        }
                    }
                }
                w |= h;
            }
            W[u >> 1] = w;
        }
        if (__builtin_expect(row_far || __builtin_amdgcn_ballot_w64(far) != 0ull, 0))
            far_chunk(a, ppos, ids, cand, left, nb, mine, px, py, pz, W);
        if (!mine) W[0] = W[1] = 0u;
        if (DYN) {   // the row itself: in run 4
            const int li = row0 + n - rb[4] - cb - base;
            if (li >= 0 && li < 32) W[0] &= ~(0x80000000u >> li);
            if (li >= 32 && li < 64) W[1] &= ~(0x80000000u >> (li - 32));
        }
        // rank the row's quarters
        const int H = __popc(W[0]) + __popc(W[1]);
        const int h0 = __shfl(H, n, WAVE), h1 = __shfl(H, n + 16, WAVE), h2 = __shfl(H, n + 32, WAVE),
                  h3 = __shfl(H, n + 48, WAVE);
        int k = found + (q > 0 ? h0 : 0) + (q > 1 ? h1 : 0) + (q > 2 ? h2 : 0);
        found += h0 + h1 + h2 + h3;
        auto slot = [&](int k) { return DYN ? (k < a.C ? k : a.C) : (k < lim ? a.Cs - 1 - k : a.Cs + 1); };
#pragma unroll
        for (int g = 0; g < 2; ++g) {
            uint32_t w = W[g];
            const uint32_t* src = ids + base + 32 * g;
            while (__builtin_amdgcn_ballot_w64(w != 0u)) {
                if (w) {   // two hits a round, so that their ids' reads overlap
                    const int c = __clz((int)w);
                    w &= ~(0x80000000u >> c);
                    const uint32_t j0 = src[c], j1 = src[w ? __clz((int)w) : c];
                    srow[slot(k)] = j0;
                    k++;
                    if (w) {
                        w &= ~(0x80000000u >> __clz((int)w));
                        srow[slot(k)] = j1;
                        k++;
                    }
                }
            }
        }
        wave_lds_sync();
    }
}

// LDS of one k_scan_cells block: its tile's 64 rows of Cs + 4 words, then each wave's scratch
inline size_t scan_cells_lds(int Cs) {
    return ((size_t)WAVE * (size_t)(Cs + 4) + WAVES_PER_BLOCK * SCAN_WAVE_LDS) * sizeof(uint32_t);
}
constexpr size_t SCAN_CELLS_LDS_MAX = 64 * 1024;
constexpr size_t SCAN_CELLS_LDS_THREE = 160 * 1024 / 3;   // three blocks per CU
constexpr int SCAN_CELLS_TWO = 2 * 256 * WAVE;            // rows whose tiles two blocks per CU hold

// (at least four waves per SIMD: within 128 registers the matrix results stay in vector registers)
template <int FMT, bool SCENES>
__global__ __launch_bounds__(BLOCK) __attribute__((amdgpu_waves_per_eu(4, 8))) void k_scan_cells(BuildArgs a) {
    static_assert(rec_words<FMT>() == 64u, "the cell scan writes the paired ids-only layout");
    extern __shared__ __align__(16) uint32_t scan_stage[];
    const int tile = xcd_block(blockIdx.x, gridDim.x);
    const int wv = __builtin_amdgcn_readfirstlane((int)(threadIdx.x / WAVE)), lane = (int)(threadIdx.x & (WAVE - 1));
    const int row0 = tile * WAVE + wv * SCAN_ROWS;
    if (row0 >= a.nd) return;   // whole waves; the block has no barrier
    const int nrw = a.nd - row0 < SCAN_ROWS ? a.nd - row0 : SCAN_ROWS;
    const int C = a.C, Cs = a.Cs, S = Cs + 4;
    uint32_t* wl = scan_stage + wv * SCAN_WAVE_LDS;
    uint32_t* st = scan_stage + WAVES_PER_BLOCK * SCAN_WAVE_LDS + wv * SCAN_ROWS * S;
    // lane (q, n): row row0 + n (the last row again past the end), its position and cell
    // (independent scenes: in its scene's grid)
    const int n = lane & 15;
    const int row = row0 + (n < nrw ? n : nrw - 1);
    const float4 p = a.pos[row];
    const int sid = SCENES ? a.sid[row] : 0;
    const Grid& g = SCENES ? a.grids[sid] : a.g;
    const int cx = cell_coord(g, p.x, 0), cy = cell_coord(g, p.y, 1), cz = cell_coord(g, p.z, 2);
    int fd = 0, fs = 0;   // row n's dynamic and static hits
    for (int s = 0; s < nrw;) {
        const int scx = __builtin_amdgcn_readlane(cx, s), scy = __builtin_amdgcn_readlane(cy, s),
                  scz = __builtin_amdgcn_readlane(cz, s), ssid = __builtin_amdgcn_readlane(sid, s);
        const bool other = cy != scy || cz != scz || cx > scx + SCAN_SPAN || (SCENES && sid != ssid);
        const unsigned long long diff = __builtin_amdgcn_ballot_w64(lane > s && lane < nrw && other);
        const int e = diff ? (int)__builtin_ctzll(diff) : nrw;
        const int ecx = __builtin_amdgcn_readlane(cx, e - 1);
        const Grid& sg = SCENES ? a.grids[ssid] : a.g;
        const float w = 1.0f / sg.inv_w;
        const float3 o = make_float3(sg.origin[0] + 0.5f * (float)(scx + ecx + 1) * w,
                                     sg.origin[1] + ((float)scy + 0.5f) * w, sg.origin[2] + ((float)scz + 0.5f) * w);
        const SegRuns R = seg_runs(a, sg, scx, ecx, scy, scz);
        const int Td = __builtin_amdgcn_readlane(R.T, 8), Ts = __builtin_amdgcn_readlane(R.T, 24);
        if (Td > 0) seg_pop_scan<true>(a, R, Td, s, e, row0, p.x, p.y, p.z, o, fd, 0, st, wl, S);
        if (Ts > 0) seg_pop_scan<false>(a, R, Ts, s, e, row0, p.x, p.y, p.z, o, fs, fd, st, wl, S);
        s = e;
    }
    int cnt = 0, cs = 0;
    if (lane < nrw) {
        const int tot = fd + fs;
        cnt = fd < C ? fd : C;
        cs = (tot < C ? tot : C) - cnt;
        a.rowcnt[row0 + lane] = cnt;
        a.rowtot[row0 + lane] = tot;
        if (tot > C) atomicOr(a.err_flag, 1);
    }
    wave_lds_sync();
    // write-out: lane (q, sub) writes slots 8 b + sub and 8 b + sub + 4 of row q (words
    // 512 b + 8 (row's place in the tile) + 2 sub), every block of [0, ceil8(cnt)) and of
    // [floor8(Cs - cs), Cs); the slots of those blocks between the two ranges get the row's own id
    // (the exact pass pads them so; until then it gathers them unused)
    typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
    const int q = lane >> 2, sub = lane & 3;
    const int qc = __shfl(cnt, q, WAVE), qs = __shfl(cs, q, WAVE);
    if (q < nrw) {
        const int nbd = (qc + 7) >> 3;
        const int bs0 = qs > 0 ? (Cs - qs) >> 3 : (Cs >> 3);
        const uint32_t* srow = st + q * S;
        u32x2* dst = reinterpret_cast<u32x2*>(a.nb + (size_t)tile * (size_t)Cs * 64u +
                                              8u * (uint32_t)(wv * SCAN_ROWS + q) + 2u * (uint32_t)sub);
        const uint32_t self = (uint32_t)(row0 + q);
        auto word = [&](int k) { return k < qc || k >= Cs - qs ? srow[k] : self; };
        for (int b = 0; b < (Cs >> 3); ++b)
            if (b < nbd || b >= bs0) dst[b * 256] = u32x2{word(8 * b + sub), word(8 * b + sub + 4)};
    }
}

// Phase B after k_scan for float32-gradient rows: one thread per row, the counts from k_scan
__global__ __launch_bounds__(BLOCK) void k_eval(BuildArgs a) {
    int blk = xcd_block(blockIdx.x, gridDim.x);
    int i = blk * BLOCK + threadIdx.x;
    int lane = threadIdx.x & (WAVE - 1);
    bool valid = i < a.nd;
    int cnt = 0, tot = 0;
    float4 pi = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    if (valid) {
        pi = a.pos[i];
        cnt = a.rowcnt[i];
        tot = a.rowtot[i];
    }
    int cs = (tot < a.C ? tot : a.C) - cnt;
    build_eval<IVP_ROWS_F32>(a, i, lane, i >> 6, valid, pi, cnt, cs, tot);
}

template <int FMT>
__device__ __forceinline__ void build_eval(const BuildArgs& a, int i, int lane, int tile, bool valid, float4 pi,
                                           int cnt, int cs, int tot) {
    constexpr unsigned REC = rec_words<FMT>();
    const float h = a.h;
    const int Cs = a.Cs;
    uint32_t* tbase = a.nb + (size_t)tile * (size_t)Cs * REC + row_word0<REC>(lane);
    int tl = wave_max(cnt);
    int ts = wave_max(cs);
    int tlp = (tl + ROW_PAD - 1) / ROW_PAD * ROW_PAD;   // <= Cs: tl <= C <= Cs, Cs a multiple of ROW_PAD
    float rho = 0.0f;
    rho = rho + pi.w * cubic_kernel(0.0f, h, a.kc);
    float aii = 0.0f;
    float jx = 0.0f, jy = 0.0f, jz = 0.0f;
    float sx = 0.0f, sy = 0.0f, sz = 0.0f;
    // one dynamic slot: gradW (stored next to the id in the float32 format; returned as the two
    // float16 side-array words h0, h1 in the float16 format), density, Aii, S
    auto dyn_slot = [&](uint32_t* rec, int j, float4 pj, float minv_j, uint32_t& h0, uint32_t& h1) {
        if ((unsigned)j >= (unsigned)a.nd) {  // never taken: phase A stored a dynamic id here
            atomicOr(a.err_flag, 4);
            return;
        }
        float rx = pi.x - pj.x, ry = pi.y - pj.y, rz = pi.z - pj.z;
        float rn = len3_rn(rx, ry, rz);
        float3 gw = spiky_grad_rn(rx, ry, rz, rn, h, a.ks);
        if (FMT == IVP_ROWS_F32) {
            rec[64] = __float_as_uint(gw.x);
            rec[128] = __float_as_uint(gw.y);
            rec[192] = __float_as_uint(gw.z);
        } else if (FMT == IVP_ROWS_F16) {
            h0 = pack_half2(gw.x * a.inv_gs, gw.y * a.inv_gs);
            h1 = pack_half2(gw.z * a.inv_gs, 0.0f);
        }
        rho += pj.w * cubic_kernel_rn(rn, h, a.inv_h, a.kc);
        float Jx = pj.w * gw.x, Jy = pj.w * gw.y, Jz = pj.w * gw.z;
        aii += (Jx * Jx + Jy * Jy + Jz * Jz) * minv_j;
        jx -= Jx; jy -= Jy; jz -= Jz;
    };
    // Two slots in flight (the cached-gradient formats): both ids, then both neighbours' (x, m)
    // and 1/m, then the two slots in order (the accumulation order of a one-slot loop).  An id
    // past a row's count is read but never used, and the gathers take a clamped index.
    auto dyn_pair = [&](uint32_t* r0, uint32_t* r1, int j0, int j1, int k, uint32_t (&hq)[4]) {
        // the empty asm statements keep each pair of loads together (the compiler would sink the
        // second slot's loads into its conditional use)
        asm volatile("" ::"v"(j0), "v"(j1));
        const int c0 = (unsigned)j0 < (unsigned)a.nd ? j0 : 0;
        const int c1 = (unsigned)j1 < (unsigned)a.nd ? j1 : 0;
        const float4 p0 = a.pos[c0];
        const float4 p1 = a.pos[c1];
        const float m0 = a.minv[c0];
        const float m1 = a.minv[c1];
        asm volatile("" ::"v"(p0.x), "v"(p0.y), "v"(p0.z), "v"(p0.w), "v"(m0), "v"(p1.x), "v"(p1.y), "v"(p1.z),
                     "v"(p1.w), "v"(m1));
        if (valid && k < cnt) dyn_slot(r0, j0, p0, m0, hq[0], hq[1]);
        if (valid && k + 1 < cnt) dyn_slot(r1, j1, p1, m1, hq[2], hq[3]);
    };
    // Four slots in flight the same way (ids-only rows, whose eight ids of a block come from two
    // loads)
    auto dyn_quad = [&](const int* j, int k, uint32_t (&hq)[8]) {
        asm volatile("" ::"v"(j[0]), "v"(j[1]), "v"(j[2]), "v"(j[3]));
        float4 p[4];
        float m[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int c = (unsigned)j[u] < (unsigned)a.nd ? j[u] : 0;
            p[u] = a.pos[c];
            m[u] = a.minv[c];
        }
        asm volatile("" ::"v"(p[0].x), "v"(p[0].y), "v"(p[0].z), "v"(p[0].w), "v"(m[0]), "v"(p[1].x), "v"(p[1].y),
                     "v"(p[1].z), "v"(p[1].w), "v"(m[1]), "v"(p[2].x), "v"(p[2].y), "v"(p[2].z), "v"(p[2].w), "v"(m[2]),
                     "v"(p[3].x), "v"(p[3].y), "v"(p[3].z), "v"(p[3].w), "v"(m[3]));
#pragma unroll
        for (int u = 0; u < 4; ++u)
            if (valid && k + u < cnt) dyn_slot(nullptr, j[u], p[u], m[u], hq[2 * u], hq[2 * u + 1]);
    };
    if constexpr (REC == 64u) {
        // ids-only rows: the row's 8 words of a block (slots 0, 4, 1, 5, 2, 6, 3, 7) with two
        // 16-byte loads; whole blocks stay inside the tile (Cs is a multiple of 8).  The float16
        // format collects the block's gradient words (slot s at word position
        // ((s & 3) << 1) | (s >> 2), zero past the row's count) and writes them as one 64-byte run
        // at twice the block's word index.
        for (int b = 0; b < tl; b += 8) {
            uint32_t* blk = tbase + slot_word<REC>(b);
            const uint4 w0 = *reinterpret_cast<const uint4*>(blk);
            const uint4 w1 = *reinterpret_cast<const uint4*>(blk + 4);
            const int ids[8] = {(int)w0.x, (int)w0.z, (int)w1.x, (int)w1.z,
                                (int)w0.y, (int)w0.w, (int)w1.y, (int)w1.w};
            uint32_t gq[16];
#pragma unroll
            for (int q = 0; q < 16; ++q) gq[q] = 0u;
#pragma unroll
            for (int t = 0; t < 8; t += 4) {
                if (b + t >= tl) break;
                uint32_t hq[8] = {0u, 0u, 0u, 0u, 0u, 0u, 0u, 0u};
                dyn_quad(ids + t, b + t, hq);
#pragma unroll
                for (int u = 0; u < 4; ++u) {
                    const int sl = t + u, pw = ((sl & 3) << 1) | (sl >> 2);
                    gq[2 * pw] = hq[2 * u]; gq[2 * pw + 1] = hq[2 * u + 1];
                }
            }
            if (FMT == IVP_ROWS_F16 && valid) {
                typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
                u32x4* dst = reinterpret_cast<u32x4*>(a.g16 + 2 * (size_t)(blk - a.nb));
#pragma unroll
                for (int q = 0; q < 4; ++q) dst[q] = u32x4{gq[4 * q], gq[4 * q + 1], gq[4 * q + 2], gq[4 * q + 3]};
            }
        }
    } else {
        for (int k = 0; k < tl; k += 2) {
            uint32_t* r0 = tbase + slot_word<REC>(k);
            uint32_t* r1 = tbase + slot_word<REC>(k + 1 < tl ? k + 1 : k);
            uint32_t hq[4];
            dyn_pair(r0, r1, (int)r0[0], (int)r1[0], k, hq);
        }
    }
    // static slots Cs - 1, Cs - 2, ...: two ids, then both positions, in flight at once
    auto st_slot = [&](int j, float4 pj) {
        if ((unsigned)j >= (unsigned)a.ns) {  // never taken: phase A stored a static id here
            atomicOr(a.err_flag, 4);
            return;
        }
        float rx = pi.x - pj.x, ry = pi.y - pj.y, rz = pi.z - pj.z;
        float rn = len3_rn(rx, ry, rz);
        float3 gw = spiky_grad_rn(rx, ry, rz, rn, h, a.ks);
        rho += pj.w * cubic_kernel_rn(rn, h, a.inv_h, a.kc);
        float Jx = pj.w * gw.x, Jy = pj.w * gw.y, Jz = pj.w * gw.z;
        jx -= Jx; jy -= Jy; jz -= Jz;
        sx += Jx; sy += Jy; sz += Jz;
    };
    for (int k = 0; k < ts; k += 2) {
        const int j0 = (int)tbase[slot_word<REC>(Cs - 1 - k)];
        const int j1 = (int)tbase[slot_word<REC>(k + 1 < ts ? Cs - 2 - k : Cs - 1 - k)];
        asm volatile("" ::"v"(j0), "v"(j1));
        const float4 q0 = a.pos[a.nd + ((unsigned)j0 < (unsigned)a.ns ? j0 : 0)];
        const float4 q1 = a.pos[a.nd + ((unsigned)j1 < (unsigned)a.ns ? j1 : 0)];
        asm volatile("" ::"v"(q0.x), "v"(q0.y), "v"(q0.z), "v"(q0.w), "v"(q1.x), "v"(q1.y), "v"(q1.z), "v"(q1.w));
        if (valid && k < cs) st_slot(j0, q0);
        if (valid && k + 1 < cs) st_slot(j1, q1);
    }
    // Pad only after the static ids (slots Cs-cs .. Cs-1) have been consumed: the padded range
    // [cnt, tlp) follows the wave's longest row and can reach into them.
    for (int k = 0; k < tlp; ++k) {
        if (!valid || k < cnt) continue;
        uint32_t* rec = tbase + slot_word<REC>(k);
        rec[0] = (uint32_t)i;
        if (FMT == IVP_ROWS_F32) {
            rec[64] = 0u;
            rec[128] = 0u;
            rec[192] = 0u;
        }   // float16 gradient words past the count were written as zeros with their block
    }
    if (valid) {
        aii += (jx * jx + jy * jy + jz * jz) * a.minv[i];
        a.kk[i] = 1.0f / (aii + 1e-3f);
        a.density[i] = rho;
        a.Ss[3 * i + 0] = sx;
        a.Ss[3 * i + 1] = sy;
        a.Ss[3 * i + 2] = sz;
        a.rowcnt[i] = cnt;
        a.rowtot[i] = tot;
    }
    // row 1 starts at zero: the window pass adds its tiles' window sizes there
    double v[2] = {(double)cnt, 0.0};
    block_partials<2>(v, a.partials, a.stride);
    if (lane == 0) a.tile_len[tile] = tlp;
    const int wl = row16_max(cnt);
    if ((lane & 15) == 0) a.wave_len[4 * tile + (lane >> 4)] = (wl + ROW_PAD - 1) / ROW_PAD * ROW_PAD;
}

// LDS of the window search: the bitmap and the marks before each of its words
struct WinBitmap {
    uint32_t bm[WIN_SPAN_WORDS];
    uint16_t pre[WIN_SPAN_WORDS];
};

// Tile window of a 64-row tile by its 256 threads.  The window is the ascending list of the distinct
// ids in the walked slots [0, tile_len) of the tile's valid rows (padding slots name the row
// itself); v / on are the thread's word pairs of the tile.  The ids are marked in an LDS bitmap over
// [lo, hi] of the tile's ids, and an id's place in the list is the number of marks below it
// (window_index).  Returns the list's length, or -1 for a tile whose range exceeds
// WIN_SPAN_WORDS words or whose window exceeds the cap (at most WIN_MAX ids).  The result is
// block-uniform; every thread of the block calls it.
struct TileWindow {
    int n, lo;
};
__device__ __forceinline__ uint32_t window_index(const WinBitmap& s, int lo, uint32_t j) {
    const uint32_t p = j - (uint32_t)lo;
    return (uint32_t)s.pre[p >> 5] + (uint32_t)__popc(s.bm[p >> 5] & ((1u << (p & 31)) - 1u));
}
// places of a word pair's two ids, 16 bits each
__device__ __forceinline__ uint32_t window_pair(const WinBitmap& s, int lo, uint32_t x, uint32_t y) {
    return window_index(s, lo, x) | (window_index(s, lo, y) << 16);
}
template <int PPT>
__device__ __forceinline__ TileWindow tile_window(const uint32_t (&vx)[PPT], const uint32_t (&vy)[PPT], const bool (&on)[PPT],
                                                  int cap, WinBitmap& s) {
    __shared__ int red[2 * WAVES_PER_BLOCK];
    int lo = 0x7fffffff, hi = -1;
#pragma unroll
    for (int k = 0; k < PPT; ++k)
        if (on[k]) {
            lo = min(lo, (int)min(vx[k], vy[k]));
            hi = max(hi, (int)max(vx[k], vy[k]));
        }
    lo = wave_min(lo);
    hi = wave_max(hi);
    const int w = threadIdx.x >> 6;
    if ((threadIdx.x & (WAVE - 1)) == 0) {
        red[w] = lo;
        red[WAVES_PER_BLOCK + w] = hi;
    }
    __syncthreads();
    lo = min(min(red[0], red[1]), min(red[2], red[3]));
    hi = max(max(red[4], red[5]), max(red[6], red[7]));
    if (hi < 0) return TileWindow{0, 0};   // no walked slot
    const int words = ((hi - lo) >> 5) + 1;
    if (words > WIN_SPAN_WORDS) return TileWindow{-1, 0};
    for (int k = threadIdx.x; k < words; k += BLOCK) s.bm[k] = 0u;
    __syncthreads();
#pragma unroll
    for (int k = 0; k < PPT; ++k)
        if (on[k]) {
            const uint32_t p0 = vx[k] - (uint32_t)lo, p1 = vy[k] - (uint32_t)lo;
            // an id repeats in many rows of a tile, and atomics on one LDS word serialise: mark
            // only what is not yet marked
            const uint32_t m0 = s.bm[p0 >> 5], m1 = s.bm[p1 >> 5];
            if (!(m0 & (1u << (p0 & 31)))) atomicOr(&s.bm[p0 >> 5], 1u << (p0 & 31));
            if (!(m1 & (1u << (p1 & 31)))) atomicOr(&s.bm[p1 >> 5], 1u << (p1 & 31));
        }
    __syncthreads();
    // thread k counts the marks of words [w0, w1); exclusive scan over the block
    const int per = (words + BLOCK - 1) / BLOCK;
    const int w0 = min((int)threadIdx.x * per, words), w1 = min(w0 + per, words);
    int cnt = 0;
    for (int k = w0; k < w1; ++k) cnt += __popc(s.bm[k]);
    int total;
    int off = block_excl_scan(cnt, &total);
    if (total > cap) return TileWindow{-1, 0};
    for (int k = w0; k < w1; ++k) {
        s.pre[k] = (uint16_t)off;
        off += __popc(s.bm[k]);
    }
    __syncthreads();
    return TileWindow{total, lo};
}

// Four lanes of a row, one term each: acc + t0 + t1 + t2 + t3 in that order on every lane (the
// one-thread accumulation order; adding an unused slot's 0 changes no bit).  The quad broadcast is
// a modifier of the add.
template <int K>
__device__ __forceinline__ float quad_bcast(float v) {
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), K * 0x55, 0xf, 0xf, true));
}
__device__ __forceinline__ void quad_add(float& acc, float t) {
    acc = acc + quad_bcast<0>(t);
    acc = acc + quad_bcast<1>(t);
    acc = acc + quad_bcast<2>(t);
    acc = acc + quad_bcast<3>(t);
}
__device__ __forceinline__ void quad_sub(float& acc, float t) {
    acc = acc - quad_bcast<0>(t);
    acc = acc - quad_bcast<1>(t);
    acc = acc - quad_bcast<2>(t);
    acc = acc - quad_bcast<3>(t);
}

// Phase B of the build with four lanes per row (ids-only and float16 rows): lane g takes slots g and
// g + 4 of every 8-slot block (one 8-byte id load), forms their terms with the expressions of
// build_eval, and the row's sums take the four lanes' terms in slot order, so rho, Aii, S and k are
// bitwise those of the one-thread pass.  A block is one 64-row tile; block partials are per tile.
// With PPT > 0 (rows of at most 8 PPT slots) the block also finds its tile's window
// (tile_window): the thread's ids, loaded at once, are the word pairs that the search needs, the
// window's (x, m) and 1/m go to the LDS, where the pairs read them, and the pass writes the list and
// the slots' indices.  As two passes the ids were read twice and every pair gathered 20 B from
// memory: us per build at 1M rows 102 + 63 apart, 138 together; a whole 4k-particle rebuild 67 / 59.
// With PPT = 0 the neighbours of block b + 1 and the ids of block b + 2 are in flight while block b
// is summed.
// Bound by vector instruction issue from about 250k rows (the correctly rounded root, reciprocal
// and quotients; 109 instructions per 64 slots, 20 of them the ordered adds), by the chain of load
// rounds below, where one thread per row leaves most SIMDs idle: us per build with one thread per
// row and with four lanes, ids-only rows: 8k 20.5 / 10, 102k 24 / 18, 262k 34 / 33, 1M 104 / 94;
// float16 rows 1M 235 / 190.
template <int FMT, int PPT>
__global__ __launch_bounds__(BLOCK, 8) void k_eval4(BuildArgs a) {
    static_assert(rec_words<FMT>() == 64u, "four lanes per row read the paired ids-only layout");
    typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
    typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
    __shared__ int wmax[WAVES_PER_BLOCK];
    const int tile = xcd_block(blockIdx.x, gridDim.x);
    const int r = (int)(threadIdx.x >> 2), g = (int)(threadIdx.x & 3), i = tile * WAVE + r;
    const bool valid = i < a.nd;
    int cnt = 0, cs = 0;
    float4 pi = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    const float h = a.h;
    const size_t w_row = (size_t)tile * (size_t)a.Cs * 64u + 8u * (uint32_t)r;
    uint32_t* row = a.nb + w_row;
    if (valid) {
        pi = a.pos[i];
        cnt = a.rowcnt[i];
        const int tot = a.rowtot[i];
        cs = (tot < a.C ? tot : a.C) - cnt;
    }
    const int wl = __builtin_amdgcn_readfirstlane(wave_max(cnt)), ws = __builtin_amdgcn_readfirstlane(wave_max(cs));
    if ((threadIdx.x & (WAVE - 1)) == 0) {
        wmax[threadIdx.x >> 6] = wl;
        a.wave_len[4 * tile + (int)(threadIdx.x >> 6)] = (wl + ROW_PAD - 1) / ROW_PAD * ROW_PAD;
    }
    float rho = 0.0f, aii = 0.0f, jx = 0.0f, jy = 0.0f, jz = 0.0f, sx = 0.0f, sy = 0.0f, sz = 0.0f;
    rho = rho + pi.w * cubic_kernel(0.0f, h, a.kc);
    const float rho_self = rho;
    const int self = valid ? i : 0;
    // An unused slot takes the row itself with mass and 1/m zero: r = 0, and every term is exactly 0
    // (a row whose position is not finite uses no slot at all: its sums are reset below).
    struct Nb {
        float4 p;
        float m;
    };
    uint32_t top = 0u;   // largest id used: below nd, phase A stored dynamic ids
    auto fetch = [&](uint32_t j, bool use) {
        j = use ? j : (uint32_t)self;
        top = j > top ? j : top;
        const uint32_t c = j < (uint32_t)a.nd ? j : (uint32_t)a.nd - 1u;
        Nb q = {a.pos[c], a.minv[c]};
        return q;
    };
    auto slots = [&](Nb q, bool use, uint32_t& h0, uint32_t& h1) {
        q.p.w = use ? q.p.w : 0.0f;
        q.m = use ? q.m : 0.0f;
        const float rx = pi.x - q.p.x, ry = pi.y - q.p.y, rz = pi.z - q.p.z;
        const float rn = len3_rn(rx, ry, rz);
        const float3 gw = spiky_grad_rn(rx, ry, rz, rn, h, a.ks);
        if (FMT == IVP_ROWS_F16) {   // (r = 0 gives gradient words of 0; a negative zero is cleared)
            const uint32_t keep = use ? 0xffffffffu : 0u;
            h0 = pack_half2(gw.x * a.inv_gs, gw.y * a.inv_gs) & keep;
            h1 = pack_half2(gw.z * a.inv_gs, 0.0f) & keep;
        }
        const float Jx = q.p.w * gw.x, Jy = q.p.w * gw.y, Jz = q.p.w * gw.z;
        quad_add(rho, q.p.w * cubic_kernel_rn(rn, h, a.inv_h, a.kc));
        quad_add(aii, (Jx * Jx + Jy * Jy + Jz * Jz) * q.m);
        quad_sub(jx, Jx);
        quad_sub(jy, Jy);
        quad_sub(jz, Jz);
    };
    const u32x2* ids2 = reinterpret_cast<const u32x2*>(row + 2 * g);
    const int nblk = (wl + 7) >> 3;   // <= Cs / 8: wl <= C
    const u32x2 none = {(uint32_t)self, (uint32_t)self};
    auto store_h = [&](int b, uint32_t (&hq)[4]) {
        if (FMT == IVP_ROWS_F16 && valid)
            *reinterpret_cast<u32x4*>(a.g16 + 2 * (w_row + 2 * (size_t)g + 512u * (uint32_t)b)) = u32x4{hq[0], hq[1], hq[2], hq[3]};
    };
    int nwin = -1;
    int tl = 0, tlp = 0;   // the tile's longest row, and that rounded up to ROW_PAD (<= Cs)
    if constexpr (PPT > 0) {
        // the search's bitmap, then in its place the window's records and list
        union Lds {
            WinBitmap s;
            struct {
                float4 x[WIN_MAX];
                float m[WIN_MAX];
                int id[WIN_MAX];
            } w;
        };
        __shared__ Lds lds_w;
        uint32_t vx[PPT], vy[PPT], ix[PPT];
        bool on[PPT];
#pragma unroll
        for (int b = 0; b < PPT; ++b) {
            const u32x2 v = b < nblk && valid ? ids2[b * 256] : none;
            vx[b] = v.x;
            vy[b] = v.y;
        }
        __syncthreads();   // wmax
        tl = max(max(wmax[0], wmax[1]), max(wmax[2], wmax[3]));
        tlp = (tl + ROW_PAD - 1) / ROW_PAD * ROW_PAD;
        const uint32_t last = (uint32_t)a.nd - 1u;
#pragma unroll
        for (int b = 0; b < PPT; ++b) {
            on[b] = valid && 8 * b < tlp;
            vx[b] = 8 * b + g < cnt ? vx[b] : (uint32_t)self;
            vy[b] = 8 * b + g + 4 < cnt ? vy[b] : (uint32_t)self;
            top = max(top, max(vx[b], vy[b]));
            vx[b] = min(vx[b], last);
            vy[b] = min(vy[b], last);
        }
        const TileWindow tw = tile_window<PPT>(vx, vy, on, a.win_cap, lds_w.s);
        nwin = tw.n;
        if (threadIdx.x == 0) a.win_n[tile] = nwin;
        if (nwin >= 0) {
            // (an empty window has no bitmap to look up)
#pragma unroll
            for (int b = 0; b < PPT; ++b) ix[b] = nwin > 0 && on[b] ? window_pair(lds_w.s, tw.lo, vx[b], vy[b]) : 0u;
            __syncthreads();   // the bitmap has been read
            uint32_t* l32 = a.loc + (size_t)tile * (size_t)a.Cs * (WAVE / 2) + threadIdx.x;
#pragma unroll
            for (int b = 0; b < PPT; ++b)
                if (on[b]) {
                    lds_w.w.id[ix[b] & 0xffffu] = (int)vx[b];   // (slots of one id write the same word)
                    lds_w.w.id[ix[b] >> 16] = (int)vy[b];
                    l32[b * 256] = ix[b];
                }
            __syncthreads();
            for (int k = threadIdx.x; k < nwin; k += BLOCK) {
                const int j = lds_w.w.id[k];
                a.win_ids[(size_t)tile * WIN_MAX + k] = j;
                lds_w.w.x[k] = a.pos[j];
                lds_w.w.m[k] = a.minv[j];
            }
            __syncthreads();
#pragma unroll
            for (int b = 0; b < PPT; ++b) {
                if (8 * b >= wl) break;
                const int k = 8 * b + g;
                uint32_t hq[4] = {0u, 0u, 0u, 0u};
                const uint32_t i0 = ix[b] & 0xffffu, i1 = ix[b] >> 16;
                slots(Nb{lds_w.w.x[i0], lds_w.w.m[i0]}, k < cnt, hq[0], hq[1]);
                if (8 * b + 4 < wl) slots(Nb{lds_w.w.x[i1], lds_w.w.m[i1]}, k + 4 < cnt, hq[2], hq[3]);
                store_h(b, hq);
            }
        }
    }
    if (nwin < 0) {
        u32x2 id1 = nblk > 0 && valid ? ids2[0] : none;
        Nb c0 = fetch(id1.x, g < cnt), c1 = fetch(id1.y, g + 4 < cnt);
        id1 = nblk > 1 && valid ? ids2[256] : none;
        for (int b = 0; b < nblk; ++b) {
            const int k = 8 * b + g;
            const Nb n0 = fetch(id1.x, k + 8 < cnt), n1 = fetch(id1.y, k + 12 < cnt);
            id1 = b + 2 < nblk && valid ? ids2[(b + 2) * 256] : none;
            uint32_t hq[4] = {0u, 0u, 0u, 0u};
            slots(c0, k < cnt, hq[0], hq[1]);
            if (8 * b + 4 < wl) slots(c1, k + 4 < cnt, hq[2], hq[3]);
            store_h(b, hq);
            c0 = n0;
            c1 = n1;
        }
    }
    if (cnt == 0) {
        rho = rho_self;
        aii = jx = jy = jz = 0.0f;
    }
    bool bad = top >= (uint32_t)a.nd;   // never
    // static slots Cs - 1, Cs - 2, ...: lane g the (4 s + g)-th
    for (int s = 0; s < ws; s += 4) {
        const bool use = s + g < cs;
        const int j = use ? (int)row[slot_word<64u>(a.Cs - 1 - s - g)] : 0;
        bad = bad || (use && (unsigned)j >= (unsigned)a.ns);   // never: phase A stored a static id
        const float4 q = a.pos[a.nd + ((unsigned)j < (unsigned)a.ns ? j : 0)];
        const float rx = pi.x - q.x, ry = pi.y - q.y, rz = pi.z - q.z;
        const float rn = len3_rn(rx, ry, rz);
        const float3 gw = spiky_grad_rn(rx, ry, rz, rn, h, a.ks);
        const float Jx = use ? q.w * gw.x : 0.0f, Jy = use ? q.w * gw.y : 0.0f, Jz = use ? q.w * gw.z : 0.0f;
        quad_add(rho, use ? q.w * cubic_kernel_rn(rn, h, a.inv_h, a.kc) : 0.0f);
        quad_sub(jx, Jx);
        quad_sub(jy, Jy);
        quad_sub(jz, Jz);
        quad_add(sx, Jx);
        quad_add(sy, Jy);
        quad_add(sz, Jz);
    }
    if (bad) atomicOr(a.err_flag, 4);
    if constexpr (PPT == 0) {
        __syncthreads();
        tl = max(max(wmax[0], wmax[1]), max(wmax[2], wmax[3]));
        tlp = (tl + ROW_PAD - 1) / ROW_PAD * ROW_PAD;
    }
    // pad only after the static ids have been consumed (the padded range can reach into them; the
    // row's four lanes are in one wave)
    if (valid) {
        for (int b = cnt >> 3; b < (tlp >> 3); ++b) {
            const int k = 8 * b + g;
            uint32_t* w = row + 2 * g + 512 * b;
            if (k >= cnt) w[0] = (uint32_t)i;
            if (k + 4 >= cnt) w[1] = (uint32_t)i;
            // (the wave's own blocks were written above; the tile's longest row may have more)
            if (FMT == IVP_ROWS_F16 && b >= nblk)
                *reinterpret_cast<u32x4*>(a.g16 + 2 * (w_row + 2 * (size_t)g + 512u * (uint32_t)b)) = u32x4{0u, 0u, 0u, 0u};
        }
        if (g == 0) {
            aii += (jx * jx + jy * jy + jz * jz) * a.minv[i];
            a.kk[i] = 1.0f / (aii + 1e-3f);
            a.density[i] = rho;
            a.Ss[3 * i + 0] = sx;
            a.Ss[3 * i + 1] = sy;
            a.Ss[3 * i + 2] = sz;
            a.rowcnt[i] = cnt;
        }
    }
    if (threadIdx.x == 0) a.tile_len[tile] = tlp;
    // row 1: the tile's window size (a window pass of its own adds it)
    double v[1] = {valid && g == 0 ? (double)cnt : 0.0}, s[1];
    __shared__ double lds[1][WAVES_PER_BLOCK];
    block_sums<1>(v, s, lds);
    if (threadIdx.x == 0) {
        a.partials[tile] = s[0];
        a.partials[a.stride + tile] = nwin > 0 ? (double)nwin : 0.0;
    }
}

struct WinArgs {
    int nd, Cs;
    int cap;   // largest window kept, <= WIN_MAX
    const uint32_t* nb;
    const int* tile_len;
    uint32_t* loc;
    int* win_ids;
    int* win_n;
    double* partials;   // the build's partials (row 1: window sizes)
    int stride;
    int tiles_per_block;   // of the pass that wrote those partials
};

// Tile windows in a pass of their own (rows of more than 64 slots, and rows that the one-lane build
// wrote), one block per 64-row tile; each walked slot's index goes 16 bits wide to the slot's id
// word (the 8-byte word pair of slots g, g + 4 becomes one 32-bit word).  Each thread keeps its PPT
// word pairs of the tile in registers from one coalesced load; a pair's places are looked up as it
// is written (kept in registers as well, 1M rows of 256 slots took 145 us a build instead of 105).
template <int PPT>
__global__ __launch_bounds__(BLOCK) void k_window(WinArgs a) {
    typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
    __shared__ WinBitmap s;
    const int t = xcd_block(blockIdx.x, gridDim.x);
    const int nrow = min(WAVE, a.nd - t * WAVE);
    const int npair = a.tile_len[t] * (WAVE / 2);
    const size_t base = (size_t)t * (size_t)a.Cs * WAVE;
    const u32x2* ids2 = reinterpret_cast<const u32x2*>(a.nb + base);
    // word pair q of a tile: block q >> 8, row (q >> 2) & 63; thread pairs q = thread + BLOCK k
    uint32_t vx[PPT], vy[PPT];
    bool on[PPT];
#pragma unroll
    for (int k = 0; k < PPT; ++k) {
        const int q = (int)threadIdx.x + BLOCK * k;
        on[k] = q < npair && ((q >> 2) & (WAVE - 1)) < nrow;
        const u32x2 v = on[k] ? ids2[q] : u32x2{0u, 0u};
        vx[k] = v.x;
        vy[k] = v.y;
    }
    const TileWindow tw = tile_window<PPT>(vx, vy, on, a.cap, s);
    const int total = tw.n;
    if (threadIdx.x == 0) a.win_n[t] = total;
    if (total <= 0) return;
    // every window id is named by some walked slot: each slot writes its id at its index (slots
    // of one id write the same word)
    int* wid = a.win_ids + (size_t)t * WIN_MAX;
    uint32_t* l32 = a.loc + base / 2;
#pragma unroll
    for (int k = 0; k < PPT; ++k)
        if (on[k]) {
            const uint32_t ix = window_pair(s, tw.lo, vx[k], vy[k]);
            wid[ix & 0xffffu] = (int)vx[k];
            wid[ix >> 16] = (int)vy[k];
            l32[threadIdx.x + BLOCK * k] = ix;
        }
    // the build's partial row 1 (zeroed by the build's blocks; the sums are integers, exact in
    // any order)
    if (threadIdx.x == 0) atomicAdd(&a.partials[a.stride + t / a.tiles_per_block], (double)total);
}

struct ExportArgs {
    int n, nd, C;
    float h, ks;
    Grid g;
    const Grid* grids;
    const int* sid;
    const float4* pos;
    const int* dstart;
    const int* sstart;
    const int* uid;
    int* count;
    int* ids;
    float* gradW;
};

// The reference cache layout (every row, user ids, count capped at C), same enumeration as
// k_build.
template <bool SCENES>
__global__ __launch_bounds__(BLOCK) void k_export(ExportArgs a) {
    int s = blockIdx.x * BLOCK + threadIdx.x;
    if (s >= a.n) return;
    const Grid g = SCENES ? a.grids[a.sid[s]] : a.g;
    float4 pi = a.pos[s];
    int u = a.uid[s];
    size_t base = (size_t)u * (size_t)a.C;
    int cnt = 0;
    bool is_dyn = s < a.nd;
    auto put = [&](int jint, float rx, float ry, float rz) {
        if (cnt < a.C) {
            float3 gw = spiky_grad(rx, ry, rz, a.h, a.ks);
            a.ids[base + cnt] = a.uid[jint];
            a.gradW[3 * (base + cnt) + 0] = gw.x;
            a.gradW[3 * (base + cnt) + 1] = gw.y;
            a.gradW[3 * (base + cnt) + 2] = gw.z;
        }
        cnt++;
    };
    visit(g, a.dstart, a.pos, is_dyn ? s : -1, pi, a.h,
          [&](int j, float4, float rx, float ry, float rz, float) { put(j, rx, ry, rz); });
    visit(g, a.sstart, a.pos + a.nd, is_dyn ? -1 : s - a.nd, pi, a.h,
          [&](int j, float4, float rx, float ry, float rz, float) { put(a.nd + j, rx, ry, rz); });
    a.count[u] = cnt < a.C ? cnt : a.C;
}

// ---- particle store loading ----------------------------------------------------------------

__global__ __launch_bounds__(BLOCK) void k_dyn_flags(int n, const int* __restrict__ is_dynamic,
                                                     const int* __restrict__ material, int fluid,
                                                     int* __restrict__ flag, int* __restrict__ err) {
    int u = blockIdx.x * BLOCK + threadIdx.x;
    if (u >= n) return;
    int dyn = is_dynamic[u] != 0 ? 1 : 0;
    flag[u] = dyn;
    if (dyn && material[u] != fluid) atomicOr(err, 2);
    if (!dyn && material[u] == fluid) atomicOr(err, 8);
}

struct StageArgs {
    int n, nd;
    int S;                 // independent scenes (0: one scene)
    const int* ustart;     // S + 1 user-order scene starts
    int* sid;
    const int* dpos;
    const int* is_dynamic;
    const float* x; const float* v; const float* m; const float* m_inv;
    const float* density0; const int* material;
    float4* pos; float* vel; float* minv; float* rho0; int* mat; int* uid; int* inv;
    float* density; float* kk; float* divg;
};

__global__ __launch_bounds__(BLOCK) void k_stage(StageArgs a) {
    int u = blockIdx.x * BLOCK + threadIdx.x;
    if (u >= a.n) return;
    bool dyn = a.is_dynamic[u] != 0;
    int s = dyn ? a.dpos[u] : a.nd + (u - a.dpos[u]);
    a.pos[s] = make_float4(a.x[3 * u + 0], a.x[3 * u + 1], a.x[3 * u + 2], a.m[u]);
    float vx = 0.0f, vy = 0.0f, vz = 0.0f;
    if (dyn) { vx = a.v[3 * u + 0]; vy = a.v[3 * u + 1]; vz = a.v[3 * u + 2]; }
    a.vel[3 * s + 0] = vx; a.vel[3 * s + 1] = vy; a.vel[3 * s + 2] = vz;
    a.minv[s] = a.m_inv[u];
    a.rho0[s] = a.density0[u];
    a.mat[s] = a.material[u];
    a.uid[s] = u;
    a.inv[u] = s;
    if (a.S > 0) {
        int lo = 0, hi = a.S;   // scene q with ustart[q] <= u < ustart[q + 1]
        while (hi - lo > 1) {
            int mid = (lo + hi) >> 1;
            if (a.ustart[mid] <= u) lo = mid; else hi = mid;
        }
        a.sid[s] = lo;
    }
    a.density[s] = a.density0[u];
    a.kk[s] = 0.0f;
    a.divg[s] = 0.0f;
}

__global__ __launch_bounds__(BLOCK) void k_write_x(int nd, const float* __restrict__ x, const int* __restrict__ uid,
                                                   float4* __restrict__ pos) {
    int s = blockIdx.x * BLOCK + threadIdx.x;
    if (s >= nd) return;
    int u = uid[s];
    float4 p = pos[s];
    p.x = x[3 * u + 0]; p.y = x[3 * u + 1]; p.z = x[3 * u + 2];
    pos[s] = p;
}

__global__ __launch_bounds__(BLOCK) void k_write_v(int nd, const float* __restrict__ v, const int* __restrict__ uid,
                                                   float* __restrict__ vel) {
    int s = blockIdx.x * BLOCK + threadIdx.x;
    if (s >= nd) return;
    int u = uid[s];
    vel[3 * s + 0] = v[3 * u + 0];
    vel[3 * s + 1] = v[3 * u + 1];
    vel[3 * s + 2] = v[3 * u + 2];
}

__global__ __launch_bounds__(BLOCK) void k_read_x(int n, const float4* __restrict__ pos, const int* __restrict__ uid,
                                                  float* __restrict__ x) {
    int s = blockIdx.x * BLOCK + threadIdx.x;
    if (s >= n) return;
    int u = uid[s];
    float4 p = pos[s];
    x[3 * u + 0] = p.x; x[3 * u + 1] = p.y; x[3 * u + 2] = p.z;
}

__global__ __launch_bounds__(BLOCK) void k_read_v(int n, int nd, const float* __restrict__ vel,
                                                  const int* __restrict__ uid, float* __restrict__ v) {
    int s = blockIdx.x * BLOCK + threadIdx.x;
    if (s >= n) return;
    int u = uid[s];
    bool dyn = s < nd;
    v[3 * u + 0] = dyn ? vel[3 * s + 0] : 0.0f;
    v[3 * u + 1] = dyn ? vel[3 * s + 1] : 0.0f;
    v[3 * u + 2] = dyn ? vel[3 * s + 2] : 0.0f;
}

__global__ __launch_bounds__(BLOCK) void k_read_f(int n, const float* __restrict__ f, const int* __restrict__ uid,
                                                  float* __restrict__ out) {
    int s = blockIdx.x * BLOCK + threadIdx.x;
    if (s >= n) return;
    out[uid[s]] = f[s];
}

int scan(ivp_ctx* c, const int* cnt, int* start, int n) {
    int nb = (n + SCAN_CHUNK - 1) / SCAN_CHUNK;
    if (nb + 1 > c->nscan_blocks) return IVP_ERR_CAPACITY;
    if (nb == 0) {
        IVP_HIP(hipMemsetAsync(start, 0, sizeof(int), c->stream));
        return IVP_OK;
    }
    hipLaunchKernelGGL(k_scan1, dim3(nb), dim3(BLOCK), 0, c->stream, n, cnt, start, c->scan_bsum);
    hipLaunchKernelGGL(k_scan2, dim3(1), dim3(BLOCK), 0, c->stream, nb, c->scan_bsum);
    hipLaunchKernelGGL(k_scan3, dim3(nb), dim3(BLOCK), 0, c->stream, n, start, c->scan_bsum, nb);
    IVP_HIP(hipGetLastError());
    return IVP_OK;
}

AdvectArgs advect_args(ivp_ctx* c, float dt) {
    return AdvectArgs{dt, c->cfg.domain_size[0], c->cfg.domain_size[1], c->cfg.domain_size[2], c->h, c->vel,
                      c->S > 0 ? c->sdomain : nullptr};
}

template <class T>
void swap_ptr(T*& a, T*& b) {
    T* t = a;
    a = b;
    b = t;
}

}  // namespace

namespace ivp {

// Sort one population [offset, offset + count) of the store by (cell key, user id) and fill
// its cell table `start_table` (ncell + 1 entries, relative to offset).  With adv the particles are
// advected first.
int grid_sort_population(ivp_ctx* c, int offset, int count, int* start_table, bool dynamic, const float* adv_dt) {
    if (count <= 0) {
        IVP_HIP(hipMemsetAsync(start_table, 0, sizeof(int) * (size_t)(c->ncell + 1), c->stream));
        return IVP_OK;
    }
    const dim3 nb(blocks_for(count));
    // bytes: keys (read x 16, write key 4; advection: v read, x written), scatter (key 4 + slot 4),
    // placing (key, uid, cell members ~ 3 x 4, and every per-particle array read and written)
    const double per = 20 + (dynamic ? 2 * (16 + 12 + 4 + 4 + 4 + 4 + 4) + 4 : 2 * (16 + 4 + 4 + 4 + 4) + 4);
    const int chunks = (c->ncell + SCAN_CHUNK - 1) / SCAN_CHUNK;
    // Particles in the caller's order (the first sort after a load, and the statics') rarely share a
    // chunk within a wave: counting the totals would cost an atomic each (1M rows: 0.1 ms), so those
    // sorts scan in three launches.
    int* bsum = dynamic && c->dyn_sorted && chunks <= CELL_SCAN_CHUNKS ? c->cell_bsum : nullptr;
    KeysArgs ka{count, c->pos + offset, c->grid, c->grids, c->sid ? c->sid + offset : nullptr, c->key, c->ccount, bsum,
                // the dynamic population's sort starts a rebuild: its first pass clears the overflow flags
                dynamic ? c->err_flag : nullptr, advect_args(c, adv_dt ? *adv_dt : 0.0f)};
    const double kb = (c->S > 0 ? 24.0 : 20.0) * count + (adv_dt ? 28.0 * count : 0.0);
    if (c->S > 0)
        IVP_TRY(adv_dt ? launch(c, KC_SORT, -1, kb, k_keys<true, true>, nb, ka)
                       : launch(c, KC_SORT, -1, kb, k_keys<true, false>, nb, ka));
    else
        IVP_TRY(adv_dt ? launch(c, KC_SORT, -1, kb, k_keys<false, true>, nb, ka)
                       : launch(c, KC_SORT, -1, kb, k_keys<false, false>, nb, ka));
    if (bsum) {
        hipLaunchKernelGGL(k_cell_starts, dim3(chunks), dim3(BLOCK), 0, c->stream, c->ncell, chunks,
                           (const int*)c->ccount, (const int*)bsum, start_table);
        IVP_HIP(hipGetLastError());
    } else {
        IVP_TRY(scan(c, c->ccount, start_table, c->ncell));
    }
    IVP_TRY(launch(c, KC_SORT, -1, 16.0 * count, k_scatter, nb, count, (const int*)c->key, (const int*)start_table,
                   c->ccount, (const int*)(c->uid + offset), c->tmp_src));
    PlaceArgs pa{count, offset, c->key, start_table, c->tmp_src, bsum, chunks, c->pos, c->pos_b, c->vel, c->vel_b,
                 c->minv, c->minv_b, c->rho0, c->rho0_b, c->mat, c->mat_b, c->uid, c->uid_b, c->inv, c->divg, c->divg_b};
    if (dynamic)
        IVP_TRY(launch(c, KC_SORT, -1, per * count, k_place<true>, nb, pa));
    else
        IVP_TRY(launch(c, KC_SORT, -1, per * count, k_place<false>, nb, pa));
    swap_ptr(c->pos, c->pos_b);
    swap_ptr(c->minv, c->minv_b);
    swap_ptr(c->rho0, c->rho0_b);
    swap_ptr(c->mat, c->mat_b);
    swap_ptr(c->uid, c->uid_b);
    if (dynamic) {
        swap_ptr(c->vel, c->vel_b);
        swap_ptr(c->divg, c->divg_b);
        c->dyn_sorted = true;
    }
    return IVP_OK;
}

int grid_load(ivp_ctx* c, int n, const float* x, const float* v, const float* m, const float* m_inv,
              const float* density0, const int* is_dynamic, const int* material) {
    if (n < 0 || n > c->cap) return IVP_ERR_CAPACITY;
    if (n > 0 && (!x || !v || !m || !m_inv || !density0 || !is_dynamic || !material)) return IVP_ERR_ARG;
    c->loaded = false;
    c->built = false;
    c->dyn_sorted = false;
    c->n = n;
    if (n == 0) {
        c->nd = c->ns = 0;
        c->loaded = true;
        return IVP_OK;
    }
    int nb = blocks_for(n);
    IVP_HIP(hipMemsetAsync(c->err_flag, 0, sizeof(int), c->stream));
    // flags -> exclusive prefix = rank of each dynamic particle
    hipLaunchKernelGGL(k_dyn_flags, dim3(nb), dim3(BLOCK), 0, c->stream, n, is_dynamic, material,
                       c->cfg.material_fluid, c->order, c->err_flag);
    int rc = scan(c, c->order, c->tmp_src, n);
    if (rc != IVP_OK) return rc;
    IVP_HIP(hipMemcpyAsync(c->count_host, c->tmp_src + n, sizeof(int), hipMemcpyDeviceToHost, c->stream));
    IVP_HIP(hipMemcpyAsync(c->err_host, c->err_flag, sizeof(int), hipMemcpyDeviceToHost, c->stream));
    IVP_HIP(hipStreamSynchronize(c->stream));
    c->nd = *c->count_host;
    c->ns = n - c->nd;
    c->all_dyn_fluid = (*c->err_host & 2) == 0;
    c->static_fluid = (*c->err_host & 8) != 0;
    int* ustart = nullptr;
    if (c->S > 0) {
        // scene boundaries in user order -> dynamic / static starts in internal order
        int S = c->S;
        std::vector<int> us(S + 1, 0);
        for (int s = 0; s < S; ++s) us[s + 1] = us[s] + c->scenes[s].n_particles;
        if (us[S] != n) return IVP_ERR_ARG;
        std::vector<int> pre(S + 1, 0);
        for (int s = 0; s <= S; ++s)
            IVP_HIP(hipMemcpy(&pre[s], c->tmp_src + us[s], sizeof(int), hipMemcpyDeviceToHost));
        c->scene_row0.assign(S + 1, 0);
        c->scene_srow0.assign(S + 1, 0);
        for (int s = 0; s <= S; ++s) {
            c->scene_row0[s] = pre[s];
            c->scene_srow0[s] = us[s] - pre[s];
        }
        for (int s = 0; s < S; ++s)
            if (c->scene_row0[s + 1] - c->scene_row0[s] < MIN_SCENE_DYNAMIC) return IVP_ERR_ARG;
        ustart = c->key;   // sort scratch, free until the static sort below
        IVP_HIP(hipMemcpy(ustart, us.data(), sizeof(int) * (S + 1), hipMemcpyHostToDevice));
    }
    StageArgs sa{n, c->nd, c->S, ustart, c->sid, c->tmp_src, is_dynamic, x, v, m, m_inv, density0, material,
                 c->pos, c->vel, c->minv, c->rho0, c->mat, c->uid, c->inv, c->density, c->kk, c->divg};
    hipLaunchKernelGGL(k_stage, dim3(nb), dim3(BLOCK), 0, c->stream, sa);
    IVP_HIP(hipGetLastError());
    // static particles: sort once.  The sort gathers [nd, n) into the reorder buffers and swaps,
    // so afterwards the staged dynamic segment [0, nd) lives in the reorder buffers and the
    // sorted static segment in the primary ones: copy each segment across so both copies of
    // every per-particle array are complete and identical.
    rc = grid_sort_population(c, c->nd, c->ns, c->sstart, false, nullptr);
    if (rc != IVP_OK) return rc;
    size_t off = (size_t)c->nd, cnt = (size_t)c->ns;
    if (cnt > 0) {
        size_t nd = off;
        auto mirror = [&](void* prim, void* alt, size_t elem) -> int {
            char* p = (char*)prim;
            char* b = (char*)alt;
            if (nd > 0) IVP_HIP(hipMemcpyAsync(p, b, nd * elem, hipMemcpyDeviceToDevice, c->stream));
            IVP_HIP(hipMemcpyAsync(b + nd * elem, p + nd * elem, cnt * elem, hipMemcpyDeviceToDevice, c->stream));
            return IVP_OK;
        };
        if ((rc = mirror(c->pos, c->pos_b, sizeof(float4))) != IVP_OK) return rc;
        if ((rc = mirror(c->minv, c->minv_b, sizeof(float))) != IVP_OK) return rc;
        if ((rc = mirror(c->rho0, c->rho0_b, sizeof(float))) != IVP_OK) return rc;
        if ((rc = mirror(c->mat, c->mat_b, sizeof(int))) != IVP_OK) return rc;
        if ((rc = mirror(c->uid, c->uid_b, sizeof(int))) != IVP_OK) return rc;
        // vel and divg were not swapped by the static sort: primary holds everything
        IVP_HIP(hipMemcpyAsync(c->vel_b, c->vel, 3 * (nd + cnt) * sizeof(float), hipMemcpyDeviceToDevice, c->stream));
        IVP_HIP(hipMemcpyAsync(c->divg_b, c->divg, (nd + cnt) * sizeof(float), hipMemcpyDeviceToDevice, c->stream));
        // static density stays rho0 (compute_density skips static rows, pressure_base.py:28-29);
        // static k and divergence are 0 in any order
        IVP_HIP(hipMemcpyAsync(c->density + off, c->rho0 + off, cnt * sizeof(float), hipMemcpyDeviceToDevice, c->stream));
    }
    c->loaded = true;
    return IVP_OK;
}

// Lanes per row of the candidate scan: the option's value, or by the dynamic count.  Measured
// (build and sort per call): 8k rows 132 us with one fused lane, 92 with 16 lanes; 102k rows
// 145 -> 115 with 4 lanes; 1M rows 501 -> 404 with 2 lanes and 4 batches in flight.  Fewer rows
// leave fewer waves per SIMD, and the one-lane scan is then a chain of dependent load rounds.
// 64 is the scan by cells (k_scan_cells), for ids-only and float16 rows (one scene or many) whose
// staged rows fit the LDS, from 20k rows: scan alone, lanes per row (best count) against by cells,
// us: 12k rows 12.3 / 14.7, 16k 13.5 / 15.7, 23k 17.5 / 15.2, 32k 21.2 / 16.6, 48k 27.1 / 17.8, 102k 43 /
// 29, 262k 83 / 50, 1M 225 / 149; where it does not apply, the count's lanes per row (16 below 32k rows: 8 lanes
// took 20 us from 1k to 23k rows against 16).  It needs three of its blocks per CU: rows of up to 168 slots
// (lanes / by cells at 168 slots, 102k rows 43 / 36, 262k 79 / 67, 1M 249 / 220, and at 176, where two
// fit, 42 / 46, 79 / 87, 244 / 300), or so few tiles that two per CU hold them all (27k rows of 216 slots
// 20.4 / 17.6).
static int lanes_by_count(int nd) { return nd >= (1 << 18) ? 2 : nd >= (1 << 15) ? 4 : 16; }

int build_lanes_for(const ivp_ctx* c) {
    const int nd = c->nd;
    const size_t lds = scan_cells_lds(c->Cs);
    const bool cells = c->rec_words == 64 && lds <= SCAN_CELLS_LDS_MAX;
    const bool pays = nd >= 20480 && (lds <= SCAN_CELLS_LDS_THREE || nd <= SCAN_CELLS_TWO);
    int G = c->build_lanes > 0 ? c->build_lanes : cells && pays ? 64 : lanes_by_count(nd);
    if (G == 64 && !cells) G = lanes_by_count(nd);
    return G;
}

template <int FMT, bool SCENES>
int launch_scan(ivp_ctx* c, int G, const BuildArgs& ba) {
    if constexpr (rec_words<FMT>() == 64u) {
        if (G == 64)
            return launch_shm(c, KC_SCAN, -1, 0.0, k_scan_cells<FMT, SCENES>, dim3((c->nd + WAVE - 1) / WAVE),
                              (unsigned)scan_cells_lds(c->Cs), ba);
    }
    const dim3 grid(blocks_for(c->nd * G));
    switch (G) {
    case 2: return launch(c, KC_SCAN, -1, 0.0, k_scan<FMT, SCENES, 2>, grid, ba);
    case 4: return launch(c, KC_SCAN, -1, 0.0, k_scan<FMT, SCENES, 4>, grid, ba);
    case 8: return launch(c, KC_SCAN, -1, 0.0, k_scan<FMT, SCENES, 8>, grid, ba);
    case 16: return launch(c, KC_SCAN, -1, 0.0, k_scan<FMT, SCENES, 16>, grid, ba);
    default: return IVP_ERR_ARG;
    }
}

// advect_position + enforce_boundary of the dynamic particles on their own
int glue_advect_boundary(ivp_ctx* c, float dt) {
    if (!c->loaded) return IVP_ERR_STATE;
    if (c->nd == 0) return IVP_OK;
    IVP_TRY(launch(c, KC_GLUE, -1, 0.0, k_advect_boundary, dim3(blocks_for(c->nd)), c->nd, advect_args(c, dt), c->pos,
                   (const int*)c->sid));
    c->built = false;
    return IVP_OK;
}

int build_fold(ivp_ctx* c) {
    if (!c->build_pending || !c->built || c->nd == 0) return IVP_OK;
    c->build_pending = false;
    return finalize<FIN_BUILD>(c, (c->nd + WAVE - 1) / WAVE);
}

int grid_build(ivp_ctx* c, const float* adv_dt, bool report) {
    if (!c->loaded) return IVP_ERR_STATE;
    if (adv_dt && c->nd > 0) c->built = false;
    if (c->nd > 0) {
        int rc = grid_sort_population(c, 0, c->nd, c->dstart, true, adv_dt);
        if (rc != IVP_OK) return rc;
    } else {
        IVP_HIP(hipMemsetAsync(c->dstart, 0, sizeof(int) * (size_t)(c->ncell + 1), c->stream));
        IVP_HIP(hipMemsetAsync(c->err_flag, 0, sizeof(int), c->stream));   // (else cleared by the sort)
    }
    // tile windows, where a tile's walked slots fit the search (Cs * 32 word pairs, PPT per thread).
    // Independent scenes whose passes run four lanes per row have them too: found in a pass of their own
    // they cost more than they saved (256 columns 4.28 -> 4.48 ms per step), found by the exact pass
    // they save more (64 scenes, two builds and a solve: 1788 -> 1744 us)
    const int ppt = (c->Cs * (WAVE / 2) + BLOCK - 1) / BLOCK;
    const bool windows = c->nd > 0 && c->windows && c->rec_words == 64 &&
                         (c->S == 0 ? ppt <= 32 : ppt <= 8 && c->scene_lanes == 4 && build_lanes_for(c) != 1);
    bool fused = false;   // the exact pass finds the windows
    int tiles_per_block = WAVES_PER_BLOCK;   // of the pass that writes the build's partials
    if (c->nd > 0) {
        // float h2_lo <= h^2 (1 - 2^-20) and h2_hi >= h^2 (1 + 2^-20): the predicate bounds of scan_ids
        const double hh = (double)c->h * (double)c->h;
        float h2_lo = std::nextafter((float)(hh * (1.0 - 1.0 / 1048576.0)), 0.0f);
        float h2_hi = std::nextafter((float)(hh * (1.0 + 1.0 / 1048576.0)), 1.0f);
        BuildArgs ba{c->nd, c->ns, c->C, c->Cs, c->h, h2_lo, h2_hi, (float)hh, c->kcubic, c->kspiky, 1.0f / c->h, 1.0f / c->gscale, c->grid,
                     c->grids, c->sid, c->pos, c->minv, c->dstart, c->sstart, c->nb, c->g16, c->tile_len, c->wave_len,
                     c->rowcnt, c->rowtot, c->density, c->kk, c->Ss, c->err_flag,
                     c->partials + (size_t)BUILD_ROW * c->max_blocks, c->max_blocks,
                     c->win_cap, c->loc, c->win_ids, c->win_n};
        // bytes (pair count of the previous build): the pair records written, the ids read back
        // once, x and m of every particle once, the per-row outputs (rho, k, S, counts)
        double pairs = (double)c->state_host->total_pairs;
        double bytes = pairs * (4.0 * c->rec_words / 64 + 4.0 + (c->row_fmt == IVP_ROWS_F16 ? 8.0 : 0.0)) +
                       16.0 * c->n + 32.0 * c->nd;
        const dim3 nb(blocks_for(c->nd));
        const int G = build_lanes_for(c);
        if (G == 1) {
            if (c->S > 0)   // independent scenes use ids-only rows (ivp_set_scenes fixes the format)
                IVP_TRY(launch(c, KC_BUILD, -1, bytes, k_build<IVP_ROWS_IDS, true>, nb, ba));
            else if (c->row_fmt == IVP_ROWS_F32)
                IVP_TRY(launch(c, KC_BUILD, -1, bytes, k_build<IVP_ROWS_F32, false>, nb, ba));
            else if (c->row_fmt == IVP_ROWS_F16)
                IVP_TRY(launch(c, KC_BUILD, -1, bytes, k_build<IVP_ROWS_F16, false>, nb, ba));
            else
                IVP_TRY(launch(c, KC_BUILD, -1, bytes, k_build<IVP_ROWS_IDS, false>, nb, ba));
        } else {
            if (c->S > 0)
                IVP_TRY((launch_scan<IVP_ROWS_IDS, true>(c, G, ba)));
            else if (c->row_fmt == IVP_ROWS_F32)
                IVP_TRY((launch_scan<IVP_ROWS_F32, false>(c, G, ba)));
            else if (c->row_fmt == IVP_ROWS_F16)
                IVP_TRY((launch_scan<IVP_ROWS_F16, false>(c, G, ba)));
            else
                IVP_TRY((launch_scan<IVP_ROWS_IDS, false>(c, G, ba)));
            // exact pass: float32-gradient rows one thread per row, the paired layout four lanes
            if (c->row_fmt == IVP_ROWS_F32) {
                IVP_TRY(launch(c, KC_BUILD, -1, bytes, k_eval, nb, ba));
            } else {
                tiles_per_block = 1;
                const dim3 tiles((c->nd + WAVE - 1) / WAVE);
                fused = windows && ppt <= 8;
                auto k = c->row_fmt == IVP_ROWS_F16 ? (fused ? k_eval4<IVP_ROWS_F16, 8> : k_eval4<IVP_ROWS_F16, 0>)
                                                    : (fused ? k_eval4<IVP_ROWS_IDS, 8> : k_eval4<IVP_ROWS_IDS, 0>);
                IVP_TRY(launch(c, KC_BUILD, -1, bytes, k, tiles, ba));
            }
        }
    }
    if (windows && !fused) {
        WinArgs wa{c->nd, c->Cs, c->win_cap, c->nb, c->tile_len, c->loc, c->win_ids, c->win_n,
                   c->partials + (size_t)BUILD_ROW * c->max_blocks, c->max_blocks, tiles_per_block};
        const dim3 grid((c->nd + WAVE - 1) / WAVE);
        if (ppt <= 8)
            IVP_TRY(launch(c, KC_WINDOW, -1, 0.0, k_window<8>, grid, wa));
        else if (ppt <= 16)
            IVP_TRY(launch(c, KC_WINDOW, -1, 0.0, k_window<16>, grid, wa));
        else
            IVP_TRY(launch(c, KC_WINDOW, -1, 0.0, k_window<32>, grid, wa));
    }
    c->win_built = windows;
    // pair count and window sizes of the build's blocks: folded here when they are reported, else with the
    // first sums of the next pressure solve (a launch less per step: 4 us of a small one)
    c->build_pending = c->nd > 0;
    if (c->nd > 0 && (report || tiles_per_block != 1)) {
        IVP_TRY(finalize<FIN_BUILD>(c, tiles_per_block == 1 ? (c->nd + WAVE - 1) / WAVE : blocks_for(c->nd), 0.0, 0,
                                    false, report ? c->state_host : nullptr));
        c->build_pending = false;
    }
    c->built = true;
    return IVP_OK;
}

int grid_export(ivp_ctx* c, int cache_size, int* count, int* ids, float* gradW) {
    if (!c->built) return IVP_ERR_STATE;
    if (cache_size <= 0 || !count || !ids || !gradW) return IVP_ERR_ARG;
    if (c->n == 0) return IVP_OK;
    ExportArgs ea{c->n, c->nd, cache_size, c->h, c->kspiky, c->grid, c->grids, c->sid, c->pos, c->dstart, c->sstart,
                  c->uid, count, ids, gradW};
    if (c->S > 0)
        hipLaunchKernelGGL(k_export<true>, dim3(blocks_for(c->n)), dim3(BLOCK), 0, c->stream, ea);
    else
        hipLaunchKernelGGL(k_export<false>, dim3(blocks_for(c->n)), dim3(BLOCK), 0, c->stream, ea);
    IVP_HIP(hipGetLastError());
    return IVP_OK;
}

int store_write(ivp_ctx* c, int field, const void* src) {
    if (!c->loaded) return IVP_ERR_STATE;
    if (!src) return IVP_ERR_ARG;
    if (c->nd == 0) return IVP_OK;
    int nb = blocks_for(c->nd);
    if (field == IVP_FIELD_X) {
        hipLaunchKernelGGL(k_write_x, dim3(nb), dim3(BLOCK), 0, c->stream, c->nd, (const float*)src, c->uid, c->pos);
        c->built = false;
    } else if (field == IVP_FIELD_V) {
        hipLaunchKernelGGL(k_write_v, dim3(nb), dim3(BLOCK), 0, c->stream, c->nd, (const float*)src, c->uid, c->vel);
    } else {
        return IVP_ERR_ARG;
    }
    IVP_HIP(hipGetLastError());
    return IVP_OK;
}

int store_read(ivp_ctx* c, int field, void* dst) {
    if (!c->loaded) return IVP_ERR_STATE;
    if (!dst) return IVP_ERR_ARG;
    if (c->n == 0) return IVP_OK;
    int nb = blocks_for(c->n);
    switch (field) {
        case IVP_FIELD_X:
            hipLaunchKernelGGL(k_read_x, dim3(nb), dim3(BLOCK), 0, c->stream, c->n, c->pos, c->uid, (float*)dst);
            break;
        case IVP_FIELD_V:
            hipLaunchKernelGGL(k_read_v, dim3(nb), dim3(BLOCK), 0, c->stream, c->n, c->nd, c->vel, c->uid, (float*)dst);
            break;
        case IVP_FIELD_DENSITY:
            hipLaunchKernelGGL(k_read_f, dim3(nb), dim3(BLOCK), 0, c->stream, c->n, c->density, c->uid, (float*)dst);
            break;
        case IVP_FIELD_K:
            hipLaunchKernelGGL(k_read_f, dim3(nb), dim3(BLOCK), 0, c->stream, c->n, c->kk, c->uid, (float*)dst);
            break;
        case IVP_FIELD_DIVERGENCE:
            hipLaunchKernelGGL(k_read_f, dim3(nb), dim3(BLOCK), 0, c->stream, c->n, c->divg, c->uid, (float*)dst);
            break;
        default:
            return IVP_ERR_ARG;
    }
    IVP_HIP(hipGetLastError());
    return IVP_OK;
}

}  // namespace ivp
