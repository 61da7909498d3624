// resident.h -- what the one-launch ("resident") solvers of small grids share.
//
// A Poisson solve on a small grid is a chain of some ten dependent sweeps per
// iteration whose data fit on a few compute units; launched one by one, each costs a
// launch (4.7 us on a 64x48x48 grid, of which under 1 us is work).  The resident
// solvers run the whole solve in one launch: each of at most ncu / 4 blocks owns a slab
// of consecutive i planes for the whole solve, keeps its cells in registers and LDS, and
// exchanges only the planes its neighbours' stencils read.
//
// Exchange between blocks.  A word travels through a slot in device memory that holds
// kEmpty until its writer stores the value; the reader polls the slot, takes the value
// and stores kEmpty back.  The value is its own arrival flag, so no fence orders it
// against a separate flag, and every access is a relaxed agent-scope atomic, which is
// coherent across the XCDs' L2s.  kEmpty is a signalling NaN: arithmetic never produces
// one (it returns quiet NaNs), so no computed value can look empty (a value that is
// published uncomputed is quieted first).  Measured: 1.0 us per
// exchange of 64 words between neighbours and 1.45 us for 1024 words each way, 1.35 us
// for a value from each of 64 blocks to all of them (a counter barrier costs 1.37 us
// and carries no data).
//
// Four sets of slots alternate.  A set is written again four exchanges later, and by
// then its reader's kEmpty has landed: a thread waits for its earlier stores (xchg_fence)
// when it has taken its words, before it empties them.  So the kEmpty of exchange n has
// landed before the barrier that ends exchange n + 1, which precedes the block's
// publication n + 2, and the writer has seen publication n + 3 when it writes again.
// (Waiting for them at once, ahead of the barrier, cost a store's way to memory in every
// exchange.)  All slots are empty when a launch ends.
//
// Progress.  The blocks wait for each other, so all of them must be on the GPU at
// once: one block fits a compute unit, and no launch has more than a quarter of the
// compute units, so that the kernels of HIP's four hardware queues fit together.  Every
// wait is bounded all the same: a block that has polled kSpinLimit times (seconds;
// reached only if another program keeps the other blocks off the GPU) raises the abort
// flag, all blocks leave, the result is dropped and the context solves with one launch
// per sweep from then on.  (The environment variable DALM_RESIDENT_SPIN sets another
// limit, so that a test can take that way.)
#pragma once
#include "ctx.h"

typedef unsigned long long u64w;
constexpr u64w kEmpty = 0x7FF4DEADBEEF0001ull;
constexpr unsigned kEmptyF = 0x7FA0DEADu;
constexpr int kSpinLimit = 1 << 21;
constexpr int kSlotSets = 4;
// Threads of a block by positions per thread: as many as leave every thread its Krylov or
// SOR values in registers (a spilled variant ran four times slower)
constexpr int kResThreads = 1024;  // most of any variant
DALM_HD constexpr int res_threads(int M) { return M == 1 ? 1024 : M == 2 ? 768 : 512; }
constexpr int kResMaxM = 4;
constexpr int kResMaxBlocks = 64;  // one lane of a wavefront per block in the all-gather

template <typename T>
struct SlotWord;
template <>
struct SlotWord<double> {
    typedef u64w W;
    static constexpr W empty = kEmpty;
    static __device__ __forceinline__ W bits(double v) { return (W)__double_as_longlong(v); }
    static __device__ __forceinline__ double value(W w) { return __longlong_as_double((long long)w); }
};
template <>
struct SlotWord<float> {
    typedef unsigned W;
    static constexpr W empty = kEmptyF;
    static __device__ __forceinline__ W bits(float v) { return __float_as_uint(v); }
    static __device__ __forceinline__ float value(W w) { return __uint_as_float(w); }
};
template <typename W>
__device__ __forceinline__ W slot_load(const W* p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
template <typename W>
__device__ __forceinline__ void slot_store(W* p, W v) {
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// this thread's stores have reached memory
__device__ __forceinline__ void xchg_fence() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }

// a / b for a normal b whose reciprocal rb is known: the product, its exact remainder and
// one correction (Markstein 1990, "Computation of elementary functions on the IBM RISC
// System/6000 processor"), which gives the correctly rounded quotient (4e8 random pairs
// agree with the division to the last bit); v_div_fixup keeps infinite and NaN dividends
// what a division makes of them.  A solve divides by the same diagonal thousands of
// times, so the reciprocal is formed once per cell.
__device__ __forceinline__ double recip(double b) {
    double y = __builtin_amdgcn_rcp(b);
    y = __builtin_fma(y, __builtin_fma(-b, y, 1.0), y);
    return __builtin_fma(y, __builtin_fma(-b, y, 1.0), y);
}
__device__ __forceinline__ double div_by(double a, double b, double rb) {
    const double q = a * rb;
    return __builtin_amdgcn_div_fixup(__builtin_fma(__builtin_fma(-b, q, a), rb, q), b, a);
}

// A launch's split: block b owns planes [b * P, (b + 1) * P) of the interior.  A row of a
// plane is nk lane positions (one cell each, or a pair of cells); a thread owns position
// k of the rows r0 + m * rw, m < M, of its block's P * ny rows.
struct ResShape {
    int blocks, P, nk, rw, M, threads;
    int spin;         // polls of a wait at most
    int pj, pk;       // rows and positions of a slab plane: ny + 2 and nk + 2
    size_t lds;       // bytes of LDS
    u64w* ring;       // [kSlotSets][2][blocks][ny * nk] halo words (FP64)
    unsigned* ringf;  // the same for FP32 words
    u64w* gath;       // [kSlotSets][blocks reading][4][blocks writing]
    int* abort_flag;
};

template <int M>
struct ResThread {
    int k;                // position in the row; -1: idle lane
    int first, planes;    // first interior plane of the block, planes it owns
    bool has_l, has_r;
    // per position: its slab index (slab plane 1 is the block's first), its word in a halo
    // plane, and (bit m) whether it exists and whether the lower / upper neighbour reads it
    int lds[M], e[M];
    unsigned in, to_l, to_r;
    unsigned n_ring, n_gath, phase;
    __device__ __forceinline__ bool has(int m) const { return (in >> m) & 1; }
    // slab plane (0-based) and interior row of position m (set-up and output only)
    __device__ __forceinline__ int row(const ResShape& s, int m) const { return (int)threadIdx.x / s.nk + m * s.rw; }
};

template <int M>
__device__ __forceinline__ ResThread<M> res_thread(const Dims& d, const ResShape& s) {
    ResThread<M> t;
    const int tid = threadIdx.x, b = blockIdx.x;
    t.first = b * s.P;
    t.planes = d.nx - t.first < s.P ? d.nx - t.first : s.P;
    t.has_l = b > 0;
    t.has_r = b + 1 < s.blocks;
    const int r0 = tid / s.nk;
    t.k = r0 < s.rw ? tid % s.nk : -1;
    t.in = t.to_l = t.to_r = 0;
#pragma unroll
    for (int m = 0; m < M; ++m) {
        const int row = r0 + m * s.rw;
        const bool in = t.k >= 0 && row < t.planes * d.ny;
        const int pl = in ? row / d.ny : 0, j = in ? row % d.ny : 0;
        t.lds[m] = ((pl + 1) * s.pj + j + 1) * s.pk + (in ? t.k : 0) + 1;
        t.e[m] = in ? j * s.nk + t.k : 0;
        if (in) t.in |= 1u << m;
        if (in && t.has_l && pl == 0) t.to_l |= 1u << m;
        if (in && t.has_r && pl == t.planes - 1) t.to_r |= 1u << m;
    }
    t.n_ring = t.n_gath = t.phase = 0;
    return t;
}

// Sum over the wavefront in every lane, by data-parallel moves inside the vector unit (a
// shuffle through LDS costs some 100 cycles a step, and the iterations wait for it)
template <int CTRL, int ROWS>
__device__ __forceinline__ double dpp_add(double v) {
    const long long b = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_update_dpp(0, (int)b, CTRL, ROWS, 0xf, true);
    const int hi = __builtin_amdgcn_update_dpp(0, (int)(b >> 32), CTRL, ROWS, 0xf, true);
    return v + __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
}
__device__ __forceinline__ double wave_total(double v) {
    v = dpp_add<0x111, 0xf>(v);  // row_shr:1, 2, 4, 8: the sum of each row of 16 lanes in its last
    v = dpp_add<0x112, 0xf>(v);
    v = dpp_add<0x114, 0xf>(v);
    v = dpp_add<0x118, 0xf>(v);
    v = dpp_add<0x142, 0xa>(v);  // row_bcast:15 into rows 1 and 3
    v = dpp_add<0x143, 0xc>(v);  // row_bcast:31 into rows 2 and 3: the total in lane 63
    const long long b = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_readlane((int)b, 63), hi = __builtin_amdgcn_readlane((int)(b >> 32), 63);
    return __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
}

// LDS of the exchange: the abort marks of two alternating phases, the wavefronts' partial
// sums and the gathered result
struct ResSync {
    int bad[2];
    double red[4][kResThreads / 64];
    double out[4];
};

// Barrier that also agrees on an abort: a wait that failed in the phase that ends here
// marked bad[phase & 1]; every thread reads that mark after the barrier, and the next
// phase's marks go to the other one.  Returns false when the block is to leave.
template <int M>
__device__ __forceinline__ bool res_barrier(ResSync& sh, ResThread<M>& t) {
    // LDS only: the exchange's stores are not waited for here
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    const bool ok = sh.bad[t.phase & 1] == 0;
    ++t.phase;
    return ok;
}
template <int M>
__device__ __forceinline__ void res_fail(ResSync& sh, const ResThread<M>& t, const ResShape& s) {
    sh.bad[t.phase & 1] = 1;
    slot_store(s.abort_flag, 1);
}
// one poll of a waiting thread: false once it is to give up
__device__ __forceinline__ bool res_wait(int& spins, const ResShape& s) {
    ++spins;
    if ((spins & 255) == 0 && slot_load(s.abort_flag) != 0) return false;
    return spins < s.spin;
}

// Halo exchange of one level: res_publish sends a value of this block's first or last
// plane to the neighbour that reads it; res_take fills the slab's planes 0 and planes + 1
// with the neighbours'.  keep(j, i): whether the value of row j on interior plane i
// travels (one colour of a red-black sweep).
template <typename T>
__device__ __forceinline__ typename SlotWord<T>::W* res_slot(const ResShape& s, const Dims& d, unsigned n, int dir,
                                                             int block) {
    typedef typename SlotWord<T>::W W;
    W* base = sizeof(T) == 8 ? (W*)s.ring : (W*)s.ringf;
    return base + (((size_t)(n % kSlotSets) * 2 + dir) * s.blocks + block) * ((size_t)d.ny * s.nk);
}
template <typename T, int M>
__device__ __forceinline__ void res_publish(const Dims& d, const ResShape& s, const ResThread<M>& t, int m, T v) {
    typedef SlotWord<T> S;
    // dir 0: towards higher i (the reader's lower halo plane); dir 1: towards lower i
    if ((t.to_r >> m) & 1) slot_store(res_slot<T>(s, d, t.n_ring, 0, blockIdx.x + 1) + t.e[m], S::bits(v));
    if ((t.to_l >> m) & 1) slot_store(res_slot<T>(s, d, t.n_ring, 1, blockIdx.x - 1) + t.e[m], S::bits(v));
}
template <typename T, int M, typename Keep>
__device__ __forceinline__ void res_take(const Dims& d, const ResShape& s, ResThread<M>& t, ResSync& sh, T* slab,
                                         Keep&& keep) {
    typedef SlotWord<T> S;
    typedef typename S::W W;
    if (t.k >= 0 && (t.has_l || t.has_r)) {
        W* lo = res_slot<T>(s, d, t.n_ring, 0, blockIdx.x);
        W* hi = res_slot<T>(s, d, t.n_ring, 1, blockIdx.x);
        const int r0 = threadIdx.x / s.nk;
        // every row's words are requested before the first is waited for
        W a[M], b[M];
        bool nl[M], nh[M];
#pragma unroll
        for (int m = 0; m < M; ++m) {
            const int j = r0 + m * s.rw;
            nl[m] = j < d.ny && t.has_l && keep(j, t.first - 1);
            nh[m] = j < d.ny && t.has_r && keep(j, t.first + t.planes);
            a[m] = nl[m] ? slot_load(lo + j * s.nk + t.k) : (W)0;
            b[m] = nh[m] ? slot_load(hi + j * s.nk + t.k) : (W)0;
        }
        int spins = 0;
#pragma unroll
        for (int m = 0; m < M; ++m) {
            const int j = r0 + m * s.rw;
            while (a[m] == S::empty || b[m] == S::empty) {
                if (!res_wait(spins, s)) {
                    res_fail(sh, t, s);
                    break;
                }
                if (a[m] == S::empty) a[m] = slot_load(lo + j * s.nk + t.k);
                if (b[m] == S::empty) b[m] = slot_load(hi + j * s.nk + t.k);
            }
            if (m == 0) xchg_fence();  // the stores of this exchange's publication and before
            const int at = (j + 1) * s.pk + t.k + 1;
            if (nl[m]) {
                slot_store(lo + j * s.nk + t.k, S::empty);
                slab[at] = S::value(a[m]);
            }
            if (nh[m]) {
                slot_store(hi + j * s.nk + t.k, S::empty);
                slab[(size_t)(t.planes + 1) * s.pj * s.pk + at] = S::value(b[m]);
            }
        }
    }
    ++t.n_ring;
}

// Sums of NV values over all cells of all blocks, the same bits in every block, in three
// parts so that an iteration can go on in between: res_sum_wave leaves the wavefronts'
// sums in LDS; after a barrier, res_sum_send adds them (wavefront 0) and sends the block's
// sums to every block, one lane per block; res_sum_take waits for all blocks' and adds
// them, and after another barrier the totals are in sh.out.
template <int NV>
__device__ __forceinline__ void res_sum_wave(const double (&v)[NV], ResSync& sh) {
#pragma unroll
    for (int q = 0; q < NV; ++q) {
        const double w = wave_total(v[q]);
        if ((threadIdx.x & 63) == 0) sh.red[q][threadIdx.x >> 6] = w;
    }
}
template <int NV, int M>
__device__ __forceinline__ void res_sum_send(const ResShape& s, ResThread<M>& t, ResSync& sh) {
    if (threadIdx.x >= 64) return;
    const int lane = threadIdx.x, nw = (blockDim.x + 63) >> 6;
    u64w* set = s.gath + (size_t)(t.n_gath % kSlotSets) * s.blocks * 4 * s.blocks;
#pragma unroll
    for (int q = 0; q < NV; ++q) {
        const double v = wave_total(lane < nw ? sh.red[q][lane] : 0.0);
        if (s.blocks == 1) {
            if (lane == 0) sh.out[q] = v;
        } else if (lane < s.blocks) {
            slot_store(set + ((size_t)lane * 4 + q) * s.blocks + blockIdx.x, SlotWord<double>::bits(v));
        }
    }
}
template <int NV, int M>
__device__ __forceinline__ void res_sum_take(const ResShape& s, ResThread<M>& t, ResSync& sh) {
    if (threadIdx.x < 64 && s.blocks > 1) {
        const int lane = threadIdx.x;
        u64w* set = s.gath + ((size_t)(t.n_gath % kSlotSets) * s.blocks + blockIdx.x) * 4 * s.blocks;
        u64w w[NV];
#pragma unroll
        for (int q = 0; q < NV; ++q) w[q] = lane < s.blocks ? slot_load(set + (size_t)q * s.blocks + lane) : 0;
#pragma unroll
        for (int q = 0; q < NV; ++q) {
            int spins = 0;
            while (w[q] == kEmpty) {
                if (!res_wait(spins, s)) {
                    res_fail(sh, t, s);
                    break;
                }
                w[q] = slot_load(set + (size_t)q * s.blocks + lane);
            }
            if (q == 0) xchg_fence();
            if (lane < s.blocks) slot_store(set + (size_t)q * s.blocks + lane, kEmpty);
            const double v = wave_total(SlotWord<double>::value(w[q]));
            if (lane == 0) sh.out[q] = v;
        }
    }
    ++t.n_gath;
}
// the three at once, with their barriers; false: leave
template <int NV, int M>
__device__ __forceinline__ bool res_sum(const double (&v)[NV], const ResShape& s, ResThread<M>& t, ResSync& sh) {
    res_sum_wave<NV>(v, sh);
    if (!res_barrier(sh, t)) return false;
    res_sum_send<NV, M>(s, t, sh);
    res_sum_take<NV, M>(s, t, sh);
    return res_barrier(sh, t);
}

// host side (resident.hip)
// the split of the grid over at most a quarter of the compute units with `lanes`
// positions per row and `bytes` of LDS per slab position; blocks = 0 when the grid does
// not fit one
ResShape res_shape(const dalm_ctx* ctx, int lanes, size_t bytes);
// allocate and empty the exchange slots on first use (sets ctx->res_off without room)
int res_prepare(dalm_ctx* ctx, ResShape& s);
// whether this context may run a resident solve of up to max_it iterations of so many
// exchanges now
bool res_may_run(const dalm_ctx* ctx, long long max_it, long long exchanges);
// wait for the launch, read its SolveState and copy its result, in ctx->r, to the
// interior of x; *ran is false when the launch was aborted (x is then as it was)
int res_finish(dalm_ctx* ctx, double* x, bool* ran);
