// fused_mixed.hip -- the precision form's BiCGStab half-iterations as single kernels
// (three Jacobi sweeps as preconditioner).
//
// One half-iteration of the preconditioned BiCGStab (src/eq.h:355-385) is a
// pointwise vector update followed by the Jacobi preconditioner and the SpMV:
//
//   p-half   p = r + beta (p - omega q);  z1 = p / a_c;  z2 = J(z1; p);  z3 = J(z2; p);
//            q = A z3,  <r0, q>
//   s-half   s = r - alpha q;              z1 = s / a_c;  z2 = J(z1; s);  z3 = J(z2; s);
//            t = A z3,  <t, s>, <t, t>
//
// where J(z; v) = z + (v - A z) / a_c is one sweep (src/eq.h:6-38: the first sweep
// from zero is z1 = v / a_c).  Run as separate kernels these move 148 B per cell
// and iteration (every level is written to HBM and read back); fused, a block keeps
// the intermediate levels on chip and reads r, p, q, r0 and writes p, z3, q once:
// 28 B per cell for the p-half and 20 B for the s-half.
//
// Temporal blocking along i.  A block of R rows x Q quads (one thread per quad, four
// consecutive k of a row) walks a chunk of `ni` planes and computes the levels with a lag
// of one plane each: at step t, level 0 (the update) at plane t, the first stencil sweep
// at t-1, the second at t-2 and the SpMV at t-3.  Each stencil level needs its input on
// the neighbouring rows, so of the R rows the block owns the inner R - 6 (overlapped
// tiling: level 0 on all of them, each level on one row less on either side); a row
// longer than the block is cut into k tiles, whose first and last quad are halo in the
// same way.  The i neighbours are the thread's own registers of the previous and next
// planes, the k neighbours its own four cells or the adjacent quads' through LDS.  Each
// step exchanges the new plane of every stencil input through LDS (two copies alternate):
// read, compute, write, barrier.  A chunk starts 3 planes early and ends 3 planes late (the
// pipeline's fill and drain).
//
// What bounds it: HBM on rows of 256 cells at 512x256x256 (295 and 230 us a half: 4.1 and
// 3.5 TB/s of algorithmic bytes, 4.4 and 3.9 with the halos, where a plain copy reaches
// 4.8); below that the steps' issue and LDS (3.0 and 2.8 us a step of 11 wavefronts at
// 256x128x128, 41 and 38 us a half, where the separate kernels took 52 and 49).
//
// The arithmetic per cell is that of the separate kernels (kg_p4 / kg_s4, kf_jacobi4,
// kg_spmv4), in their order: FP32 sweeps with FP32 coefficients, the SpMV in FP64 with the
// FP64 operator and its result rounded once, dot products in FP64 of the stored values.  So the
// FP32 vectors are theirs up to a rare last bit (BiCGStab doubles a difference every
// iteration: with another order of the stencil sums the pressure after 12 iterations is
// another one of the same quality, up to five times nearer or further).
// Ghost cells of the preconditioner iterates are zero, as in the reference
// (fill_array(pp, 0) before the sweeps, which write the interior only).
//
// p and q are read at halo cells owned by neighbouring blocks, so the p-half reads
// the previous p and q from one buffer of a pair and writes the new ones to the
// other (the host alternates the pair every iteration).
//
// Rows of 256 cells (MODE 2): the end of an iteration, x += alpha z_p + omega z_s and
// r = s - omega t, has no pass of its own.  The s-half also returns <r0, s>, <r0, t> and |s|^2, from which
// the finalize expands |r|^2 and <r0, r> (FIN_MX_OMEGA); both updates are then
// pending (SolveState.pending) and the next p-half applies them: it forms r from s
// and t where it needs r (every row it computes) and stores r on its owned cells.
// Neither half updates the FP64 pressure x: the finalize records each iteration's
// alpha and omega (SolveState.xdef counts the outstanding updates), z_p and z_s rotate
// through kXGroupF buffer pairs with the iteration, and kg_apply_pending4 applies the
// outstanding updates, in turn, once kXGroupF have gathered or ahead of a residual
// replacement; the host applies the rest after the last iteration of a pass
// (kg_flush_pending4).  Each update is the same two roundings in the same order as one
// update per iteration, so x is the same to the bit.  Per iteration this moves 70 B
// per cell (the p-half 36, the s-half 24, the grouped x update (16 + 8 kXGroupF) /
// kXGroupF) instead of 88.  Other rows keep that pass (kg_xr): the <r0, r> of the stored r
// keeps the separate kernels' iterates, and it costs a finalize and 8 B per cell more
// (1.99 against 1.91 ms a step of 12 iterations at 256x128x128).
#include <algorithm>
#include <type_traits>
#include "ctx.h"
#include "stencil.h"

namespace {

constexpr int kLag = 3;             // planes from level 0 to the SpMV
constexpr int kPad = 4;             // zero cells on either side of an LDS row
// threads of a block: 16 wavefronts of 128 VGPRs where the row's coefficients are scalars,
// else 12 of 168 (the general form in 16 spilled 17 and took 1.15 times as long)
constexpr int kHalfThreads = 1024, kHalfThreadsAny = 768;

typedef float f4 __attribute__((ext_vector_type(4), aligned(16)));
typedef float f4u __attribute__((ext_vector_type(4), aligned(4)));

// LDS of a block of R rows x Q quads:
//   lv[2][3][R][4 Q + 2 kPad]  the new plane of each stencil input (z1, z2, z3), in two
//       alternating copies: a step reads the copy the previous step wrote and writes the
//       other, so one barrier per step orders both (101 of the CU's 160 KB at R Q = 1024)
//   k coefficients at, ab, atu, abu [Q][4] each, FP64 (SpMV) and FP32 (sweeps)
//   FP64 j coefficients an, as, anu, asu of each row
__host__ __device__ inline int half_row_len(int Q) { return 4 * Q + 2 * kPad; }
__host__ __device__ inline size_t half_lds(int R, int Q) {
    return sizeof(float) * (6 * (size_t)R * half_row_len(Q)) + (sizeof(double) + sizeof(float)) * 16 * (size_t)Q +
           sizeof(double) * 4 * (size_t)R;
}

// j and k neighbours of one level at this thread's four cells, from LDS
struct Nb {
    f4 n, s;
    float kb, kf;
};
// lv: this thread's four cells in the level's plane; len: row length
__device__ __forceinline__ Nb nbrs(const float* lv, int len) {
    Nb b;
    b.n = *(const f4*)(lv + len);
    b.s = *(const f4*)(lv - len);
    b.kb = lv[-1];
    b.kf = lv[4];
    return b;
}

// block sum over up to 16 wavefronts in a fixed order (result in thread 0)
template <int NV>
__device__ __forceinline__ void block_sum16(double (&v)[NV]) {
    __shared__ double red[NV][kHalfThreads / 64];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, waves = (int)blockDim.x >> 6;
#pragma unroll
    for (int q = 0; q < NV; ++q) v[q] = wave_sum(v[q]);
    if (lane == 0) {
#pragma unroll
        for (int q = 0; q < NV; ++q) red[q][wave] = v[q];
    }
    __syncthreads();
    if (threadIdx.x == 0) {
#pragma unroll
        for (int q = 0; q < NV; ++q) {
            double s = red[q][0];
            for (int w = 1; w < waves; ++w) s += red[q][w];
            v[q] = s;
        }
    }
}

// WHICH 0: the p-half (vin = previous p, qin = previous q; vout = new p, zout = new
//          z_p, yout = new q; r read, or formed from s_in, t_in and stored; dot
//          <r0, q>)
// WHICH 1: the s-half (r, qin = q; vout = s, zout = z_s, yout = t; dots <t, s>,
//          <t, t>, <r0, s>, <r0, t>, |s|^2)
struct HalfArgs {
    float* r;
    const float *s_in, *t_in;  // p-half: the previous iteration's s, t
    const float *vin, *qin;
    float *vout, *zout, *yout;
    const float* r0;
    double* partials;
};

// MODE 0: any row length.  MODE 1: a multiple of 4, so that no quad reaches beyond its
// row.  MODE 2: rows of 256 cells in blocks of 16 rows x 64 quads, a wavefront a row: its
// coefficients live in scalars and every LDS offset is a constant.
//
// Nothing outside the grid is masked.  Loads are clamped to the padded box, whose ghost
// cells are zero in every Krylov vector, and the off-diagonals of ghost planes, rows and
// cells are zero, so those cells' values stay zero by arithmetic (their diagonals are not
// zero: a ghost cell along k gets one).  Cells of a quad beyond its row's end are cleared
// where they are stored, so that a solve whose scalars are no numbers leaves the ghost
// cells zero.
//
// COLS: every cell column of a chunk has its own sums, and the block adds them as the
// separate kernels' units do (col_unit, block_sum: 64 columns of a row by wave_sum, then four
// rows) into their slots.  Chunks and tiles are then whole units.  The dot products are so
// the same to the bit, and with them the iterates: summed in another order, alpha differs in
// its last bit, which turns an FP32 rounding somewhere in four million cells every few
// iterations, and at 256x128x128 3 pressures of 12 were up to four times further off (or nearer).
template <int WHICH, int MODE, bool COLS>
__global__ __launch_bounds__(MODE == 2 ? kHalfThreads : kHalfThreadsAny) void kg_half4(
    Dims d, PCoefF Af, PCoef A, HalfArgs h, HalfGeom geom, const SolveState* st) {
    if (st->done) return;
    constexpr bool UNI = MODE == 2, WHOLE = MODE >= 1;
    HalfGeom G = geom;
    if (UNI) {
        G.R = 16;
        G.Q = 64;
        G.tk = 1;
    }
    extern __shared__ __align__(16) double half_sh[];
    const int len = half_row_len(G.Q), plane = G.R * len, nk = 4 * G.Q;
    double *const atd = half_sh, *const abd = atd + nk, *const atud = abd + nk, *const abud = atud + nk;
    float *const atf = (float*)(abud + nk), *const abf = atf + nk, *const atuf = abf + nk, *const abuf = atuf + nk;
    double* const jd = (double*)(abuf + nk);  // a row's FP64 an, as, anu, asu
    float* const lv = (float*)(jd + 4 * G.R);
    const int row = UNI ? __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)) : (int)threadIdx.x / G.Q;
    const int lane = UNI ? (int)(threadIdx.x & 63) : (int)threadIdx.x % G.Q;
    const int g = d.gc;
    // unit: j tile jt (rows jt*own .. +own), k tile kt, plane chunk ic; the last chunk of
    // a column starts inside its predecessor (it computes ni planes, owns from own0).
    // Units are numbered j tile fastest, then k tile, and each XCD runs a contiguous
    // range of them: the halo rows that neighbouring tiles of a chunk both read are
    // fetched from HBM once and served to the second from the XCD's L2.
    const int u = xcd_unit((int)blockIdx.x, (int)gridDim.x);
    const int jt = u % G.tj, kt = u / G.tj % G.tk, ic = u / (G.tj * G.tk), ni = G.ni;
    const int own0 = g + ic * ni;
    int i1 = own0 + ni;
    if (i1 > g + d.nx) i1 = g + d.nx;
    const int i0 = i1 - ni;
    const int j = g + jt * (G.R - 2 * kLag) + row - kLag;
    // with several k tiles the first and last quad of a block are halo
    const int quad = G.tk > 1 ? kt * (G.Q - 2) - 1 + lane : lane;
    const int left = d.nz - 4 * quad;  // cells of the row from this quad on; the quad's last may lie beyond it
    const bool in_row = quad >= 0 && left > 0;
    const bool owned = row >= kLag && row < G.R - kLag && j < g + d.ny && in_row &&
                       (G.tk == 1 || (lane >= 1 && lane < G.Q - 1));
    // this thread's bytes into a plane: rows clamped to the padded box, quads off the row
    // to the four ghost cells between its end and the next row's start
    const int jc = j < 0 ? 0 : (j < d.n1 ? j : d.n1 - 1);
    const unsigned off = 4u * (unsigned)(jc * d.sj + (in_row ? g + 4 * quad : g + d.nz));
    const bool first = st->it == 0;
    // p-half: the previous iteration's r is still to be formed (its omega is that of
    // st: FIN_ALPHA runs after this kernel); without, r = r - 0 r, and in the first
    // iteration p = r + 0 (r - omega r): no stale vector is read
    const bool pend = UNI && WHICH == 0 && st->pending;
    const double beta = first ? 0.0 : st->beta, om = st->omega, alpha = st->alpha, om_r = pend ? om : 0.0;
    const float* const r_a = pend ? h.s_in : h.r;
    const float* const r_b = pend ? h.t_in : h.r;
    const float* const v_a = first ? r_a : h.vin;
    const float* const q_a = WHICH == 0 && first ? r_a : h.qin;
    // the SpMV's diagonal is divided by max|a_c|: a product with its reciprocal, and one
    // correction where the separate kernels' quotient is to be met (not on rows of 256)
    const double inv_md = 1.0 / A.max_diag;

    const float an = Af.an[jc], as = Af.as[jc], anu = Af.anu[jc], asu = Af.asu[jc];
    // a uniform row's FP64 coefficients are scalars; otherwise they are read from LDS, where
    // registers would spill
    double an_u = 0, as_u = 0, anu_u = 0, asu_u = 0;
    if (UNI) {
        an_u = A.an[jc];
        as_u = A.as[jc];
        anu_u = A.anu[jc];
        asu_u = A.asu[jc];
    } else if (lane == 0 && row < G.R) {
        jd[4 * row] = A.an[jc];
        jd[4 * row + 1] = A.as[jc];
        jd[4 * row + 2] = A.anu[jc];
        jd[4 * row + 3] = A.asu[jc];
    }
    const int kbase = g + (G.tk > 1 ? 4 * (kt * (G.Q - 2) - 1) : 0);
    for (int t = threadIdx.x; t < nk; t += blockDim.x) {
        const int k = kbase + t;
        const bool in = k >= g && k < g + d.nz;
        atd[t] = in ? A.at[k] : 0.0;
        abd[t] = in ? A.ab[k] : 0.0;
        atud[t] = in ? A.atu[k] : 1.0;
        abud[t] = in ? A.abu[k] : 0.0;
        atf[t] = in ? Af.at[k] : 0.f;
        abf[t] = in ? Af.ab[k] : 0.f;
        atuf[t] = in ? Af.atu[k] : 1.f;
        abuf[t] = in ? Af.abu[k] : 0.f;
    }
    for (int t = threadIdx.x; t < 6 * plane; t += blockDim.x) lv[t] = 0.f;
    __syncthreads();

    const f4 zero = {0.f, 0.f, 0.f, 0.f};
    // pipeline registers: z1 at t-1, t-2, z2 at t-2, t-3, z3 at t-3, t-4; v (p or s) at
    // t-1, t-2, and for the s-half's dots t-3
    f4 z1a = zero, z1b = zero, z2a = zero, z2b = zero, z3a = zero, z3b = zero, va = zero, vb = zero, vc = zero;
    constexpr int kDots = WHICH == 0 ? 1 : UNI ? 5 : 2;
    double acc[kDots][COLS ? 4 : 1] = {};

    const auto at_plane = [&](const float* p, int i) {
        i = i < 0 ? 0 : (i < d.n0 ? i : d.n0 - 1);
        return *(const f4u*)((const char*)(p + (size_t)i * (size_t)d.si) + off);
    };
    const auto put = [&](float* p, int i, f4 x) {
        if (!WHOLE) {
#pragma unroll
            for (int q = 0; q < 4; ++q) x[q] = q < left ? x[q] : 0.f;
        }
        // nontemporal: a stored vector is next read a kernel later, past the last-level cache
        __builtin_nontemporal_store((f4u)x, (f4u*)((char*)(p + (size_t)i * (size_t)d.si) + off));
    };
    // level-0 inputs, requested one step ahead
    struct In {
        f4 a, b, v, q;
    };
    const auto load0 = [&](int i) {
        In x;
        x.a = at_plane(r_a, i);
        x.q = at_plane(q_a, i);
        if (WHICH == 0) {
            if (UNI) x.b = at_plane(r_b, i);
            x.v = at_plane(v_a, i);
        }
        return x;
    };
    In nx0 = load0(i0 - kLag);
    constexpr bool NEED_R0 = WHICH == 0 || UNI;
    f4 r0n = NEED_R0 ? at_plane(h.r0, i0) : zero;
    // this thread's place in a plane; its neighbours' reads stay in range (the block's
    // edge rows' stencil values are not used)
    const int rr = row == 0 ? 1 : (row >= G.R - 1 ? G.R - 2 : row);
    const int me = row * len + kPad + 4 * lane, near = rr * len + kPad + 4 * lane;
    const int lk = 4 * lane;

    // one step at plane t with L = 0, 1, 2 stencil levels (the pipeline's fill) or 3 (and
    // the SpMV).  (The loop unrolled by two, to rename the pipeline registers instead of
    // moving them, spilled 17 to 55 registers and took twice as long.)
    int cw = 0;  // the LDS copy this step writes
    const auto step = [&](auto levels, int t) {
        constexpr int L = decltype(levels)::value;
        const f4 r0c = r0n;
        if (L == 3 && NEED_R0) r0n = at_plane(h.r0, t - kLag + 1);
        const float* prev = lv + (cw ^ 1) * 3 * plane + near;
        const auto clampi = [&](int i) { return i < 0 ? 0 : (i < d.n0 ? i : d.n0 - 1); };
        const int p0 = clampi(t), p1 = clampi(t - 1), p2 = clampi(t - 2), iy = t - kLag;
        const f4 atu = *(const f4*)(atuf + lk), abu = *(const f4*)(abuf + lk);
        const f4 at = *(const f4*)(atf + lk), ab = *(const f4*)(abf + lk);
        // one sweep at plane ip: centre xa, the plane before xb, the plane after xn
        const auto sweep = [&](int ip, const f4& xb, const f4& xa, const f4& xn, const float* at_lv, const f4& rhs) {
            const Nb nb = nbrs(at_lv, len);
            const float acj = (Af.acx[ip] - anu) - asu, ae = Af.ae[ip], aw = Af.aw[ip];
            f4 out;
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const float ac = (acj - atu[q]) - abu[q];
                const float tq = q + 1 < 4 ? xa[q + 1] : nb.kf;
                const float bq = q > 0 ? xa[q - 1] : nb.kb;
                float ax = ac * xa[q];
                ax = fmaf(ae, xn[q], ax);
                ax = fmaf(aw, xb[q], ax);
                ax = fmaf(an, nb.n[q], ax);
                ax = fmaf(as, nb.s[q], ax);
                ax = fmaf(at[q], tq, ax);
                ax = fmaf(ab[q], bq, ax);
                out[q] = fmaf(rhs[q] - ax, __builtin_amdgcn_rcpf(ac), xa[q]);
            }
            return out;
        };
        const bool in_lds = UNI || row < G.R;
        float* now = lv + cw * 3 * plane + me;
        // level 0 at plane t
        f4 z1n, vn;
        {
            const float acj = (Af.acx[p0] - anu) - asu;
            const bool mine = owned && t >= own0 && t < i1;
            f4 rv;
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                float vf;
                if (WHICH == 0) {
                    rv[q] = UNI ? (float)((double)nx0.a[q] - om_r * (double)nx0.b[q]) : nx0.a[q];
                    vf = (float)((double)rv[q] + beta * ((double)nx0.v[q] - om * (double)nx0.q[q]));
                } else {
                    vf = (float)((double)nx0.a[q] - alpha * (double)nx0.q[q]);
                }
                vn[q] = vf;
                z1n[q] = vf * __builtin_amdgcn_rcpf((acj - atu[q]) - abu[q]);
            }
            if (mine) {
                if (pend) put(h.r, t, rv);
                put(h.vout, t, vn);
            }
        }
        if (in_lds) *(f4*)now = z1n;
        nx0 = load0(t + 1);
        // levels 1 and 2 at planes t-1, t-2
        if (L >= 1) {
            const f4 z2n = sweep(p1, z1b, z1a, z1n, prev, va);
            if (in_lds) *(f4*)(now + plane) = z2n;
            if (L >= 2) {
                const f4 z3n = sweep(p2, z2b, z2a, z2n, prev + plane, vb);
                if (in_lds) *(f4*)(now + 2 * plane) = z3n;
                // the SpMV at plane t-3 (FP64 operator, FP64 arithmetic, rounded once)
                if (L == 3 && owned && iy >= own0 && iy < i1) {
                    const Nb nb = nbrs(prev + 2 * plane, len);
                    const double and_ = UNI ? an_u : jd[4 * row], asd = UNI ? as_u : jd[4 * row + 1];
                    const double acj = (A.acx[iy] - (UNI ? anu_u : jd[4 * row + 2])) - (UNI ? asu_u : jd[4 * row + 3]);
                    const double aw = A.aw[iy], ae = A.ae[iy];
                    f4 y;
#pragma unroll
                    for (int q = 0; q < 4; ++q) {
                        const double au = (acj - atud[lk + q]) - abud[lk + q];
                        double ac = au * inv_md;
                        if (!UNI) ac = fma(fma(-ac, A.max_diag, au), inv_md, ac);  // rounded as au / max_diag
                        const double tq = q + 1 < 4 ? (double)z3a[q + 1] : (double)nb.kf;
                        const double bq = q > 0 ? (double)z3a[q - 1] : (double)nb.kb;
                        double yv = ac * (double)z3a[q];
                        yv = fma(ae, (double)z3n[q], yv);
                        yv = fma(aw, (double)z3b[q], yv);
                        yv = fma(and_, (double)nb.n[q], yv);
                        yv = fma(asd, (double)nb.s[q], yv);
                        yv = fma(atd[lk + q], tq, yv);
                        yv = fma(abd[lk + q], bq, yv);
                        const float yf = (float)yv;
                        y[q] = yf;
                        const double ys = (double)yf;
                        const int col = COLS ? q : 0;
                        if (WHICH == 0) {
                            acc[0][col] += (double)r0c[q] * ys;
                        } else {
                            const double sv = (double)vc[q], rz = (double)r0c[q];
                            acc[0][col] += ys * sv;
                            acc[1][col] += ys * ys;
                            if (UNI) {
                                acc[2][col] += rz * sv;
                                acc[3][col] += rz * ys;
                                acc[4][col] += sv * sv;
                            }
                        }
                    }
                    put(h.yout, iy, y);
                    put(h.zout, iy, z3a);
                }
                z3b = z3a;
                z3a = z3n;
            }
            z2b = z2a;
            z2a = z2n;
        }
        z1b = z1a;
        z1a = z1n;
        if (WHICH == 1) vc = vb;
        vb = va;
        va = vn;
        __syncthreads();
        cw ^= 1;
    };
    using std::integral_constant;
    int t = i0 - kLag;
    for (; t < i0 - 1; ++t) step(integral_constant<int, 0>(), t);
    for (; t < i0 + 1; ++t) step(integral_constant<int, 1>(), t);
    for (; t < i0 + kLag; ++t) step(integral_constant<int, 2>(), t);
    for (; t < i1 + kLag; ++t) step(integral_constant<int, 3>(), t);
    if (!COLS) {
        double sum[kDots];
#pragma unroll
        for (int q = 0; q < kDots; ++q) sum[q] = acc[q][0];
        block_sum16<kDots>(sum);
        if (threadIdx.x == 0)
            for (int q = 0; q < kDots; ++q) h.partials[q * gridDim.x + blockIdx.x] = sum[q];
        return;
    }
    // the columns' sums [dot][row][cell] and the rows' [dot][group of 64][row] take the
    // planes' place (the last step's barrier is behind every read of them)
    double* const cols = (double*)lv;
    double* const rows = cols + kDots * G.R * nk;
    if (row < G.R)
#pragma unroll
        for (int q = 0; q < kDots; ++q)
#pragma unroll
            for (int m = 0; m < 4; ++m) cols[(q * G.R + row) * nk + lk + m] = acc[q][COLS ? m : 0];
    __syncthreads();
    const int own = G.R - 2 * kLag, kfrom = G.tk > 1 ? 4 : 0, kto = G.tk > 1 ? nk - 4 : nk;
    const int groups = (kto - kfrom + 63) / 64, wl = (int)threadIdx.x & 63;
    for (int w = (int)threadIdx.x >> 6; w < kDots * groups * own; w += (int)blockDim.x >> 6) {
        const int r = w % own, gq = w / own, q = gq / groups, kk = kfrom + 64 * (gq % groups) + wl;
        const double s = wave_sum(kk < kto ? cols[(q * G.R + kLag + r) * nk + kk] : 0.0);
        if (wl == 0) rows[w] = s;
    }
    __syncthreads();
    const int quads = own / TJ;
    for (int w = (int)threadIdx.x; w < kDots * groups * quads; w += (int)blockDim.x) {
        const int jq = w % quads, gq = w / quads, q = gq / groups;
        const double* const rs = rows + gq * own + TJ * jq;
        double s = rs[0];
        for (int m = 1; m < TJ; ++m) s += rs[m];
        const int ujt = jt * quads + jq, ukt = kt * groups + gq % groups;
        if (ujt < d.tj && ukt < d.tk)
            h.partials[q * d.nunits + virtual_block_index(ic + d.nch * (ukt + d.tk * ujt), d.nunits)] = s;
    }
}

}  // namespace

int fused_planes(const dalm_ctx* ctx, int tiles) {
    const int nx = ctx->d.nx;
    int nch = ctx->ncu / (tiles > 0 ? tiles : 1);
    const int most = (nx + 15) / 16;
    if (nch > most) nch = most;
    if (nch < 1) nch = 1;
    return (nx + nch - 1) / nch;
}

// The split of a grid over the compute units (one block each: its wavefronts fill the
// VGPRs).  Rows of 256 cells take blocks of 16 x 64 in one round, with chunks of at least
// 16 planes.  Otherwise every number of k and j tiles is priced: a block takes
// ni + 2 kLag steps of 1.5 us + 0.2 us per wavefront on its compute unit (measured at
// 10 to 16 wavefronts; both sides of the halos' trade: a thinner chunk or tile recomputes
// more).  At 256x128x128 8 j tiles of 22 rows and chunks of 8 planes are chosen (41 and 38 us
// a half); 4 j tiles of 38 rows in two k tiles took 9 and 8 % more, 8 tiles of 22 rows in
// two 25 %.  Small grids are left with
// the steps: chunks of two planes (8 steps) take 57.8 us an iteration at 64x32x32 with
// everything around it, chunks of four 63.7, the separate kernels 59.0 to 66.1.
constexpr long long kTilesFrom = 1LL << 20, kColsFrom = 1LL << 21;

// what block_sum16 keeps in LDS beside half_lds, at most
constexpr size_t kHalfStatic = 5 * (kHalfThreads / 64) * sizeof(double);

static HalfGeom cheapest_half(const dalm_ctx* ctx, bool cols, double* cost_out) {
    const Dims& d = ctx->d;
    const int NQ = (d.nz + 3) / 4;
    HalfGeom best{};
    double cost = 0;
    for (int tk = 1; tk <= 64; ++tk) {
        const int Q = tk == 1 ? NQ : (NQ + tk - 1) / tk + 2;
        const int most = kHalfThreadsAny / Q;
        if (most < 2 * kLag + 4) continue;
        if (tk > 1 && (Q < 16 || ctx->N < kTilesFrom * (d.nz % 64 ? 1 : 2))) break;
        for (int tj = (d.ny + most - 2 * kLag - 1) / (most - 2 * kLag); tj <= d.ny; ++tj) {
            int own = (d.ny + tj - 1) / tj;
            if (cols) own = (own + TJ - 1) / TJ * TJ;
            const int R = own + 2 * kLag;
            if (own < 4) break;
            if (own > most - 2 * kLag || (cols && tk > 1 && (Q - 2) % 16)) continue;
            // short rows: each of a block's many rows costs its pads too (320 B at one quad)
            if (half_lds(R, Q) + kHalfStatic > kLdsBytes) continue;
            const int waves = (R * Q + 63) / 64;
            const int per_cu = waves <= 6 ? 12 / waves : 1;
            const int slots = ctx->ncu * per_cu;
            for (int rounds = 1; rounds <= 2; ++rounds) {
                int nch = rounds * slots / (tj * tk);
                if (nch < 1) continue;
                if (nch > (d.nx + 1) / 2) nch = (d.nx + 1) / 2;
                const int ni = cols ? d.ni : (d.nx + nch - 1) / nch;
                const int blocks = tj * tk * ((d.nx + ni - 1) / ni);
                const int on_cu = std::min(per_cu, (blocks + ctx->ncu - 1) / ctx->ncu);
                const double c = (blocks + slots - 1) / slots * (ni + 2 * kLag) * (1.5 + 0.2 * waves * on_cu);
                if (best.R == 0 || c < cost) {
                    cost = c;
                    best = HalfGeom{R, Q, tj, tk, ni, blocks, waves * 64, d.nz % 4 == 0 ? 1 : 0,
                                    cols ? d.nunits : blocks, cols, half_lds(R, Q)};
                }
            }
        }
    }
    *cost_out = cost;
    return best;
}

HalfGeom split_half(const dalm_ctx* ctx) {
    const Dims& d = ctx->d;
    HalfGeom best{};
    if (d.nz == 256 && d.ny >= 10) {
        const int tj = (d.ny + 9) / 10, ni = fused_planes(ctx, tj), blocks = tj * ((d.nx + ni - 1) / ni);
        best = HalfGeom{16, 64, tj, 1, ni, blocks, kHalfThreads, 2, blocks, false, half_lds(16, 64)};
    } else {
        // from kColsFrom cells on chunks and tiles of whole units of the separate kernels, but
        // where those cost a quarter more (at 192x128x384 264 blocks, eight of them in a second
        // round: 5.27 ms a step and 4.26; the pressure's error against 64 bits is 4e-7 in
        // either); rows that the separate kernels take four cells per lane have others (col_unit4)
        double cost, cost_cols;
        best = cheapest_half(ctx, false, &cost);
        if (ctx->N >= kColsFrom && !vec4_applies(d)) {
            const HalfGeom c = cheapest_half(ctx, true, &cost_cols);
            if (c.R > 0 && cost_cols <= 1.25 * cost) best = c;
        }
    }
    // a plane within 32-bit offsets, and room for the sums of every block
    if ((long long)d.si * 4 >= (1LL << 31) || 5 * (size_t)best.sums > 8 * (size_t)std::max(ctx->grid, ctx->sgrid))
        best.R = 0;
    return best;
}

// The fused path: three Jacobi sweeps on a grid that splits (R > 0).  Of 240 sizes from 200 to
// 5 10^6 cells it is the faster one at all but three (rows of 160 to 290 cells on grids of few
// rows: at most 4 % slower, 661 and 685 us at 11x18x288): a step of 10 iterations with the separate kernels and fused:
// 654 and 569 us at 30x14x16, 678 and 629 at 96x48x48, 806 and 701 at 128x64x64, 939 and 862 at
// 64x96x128, 1295 and 1048 at 173x101x87, 8110 and 6366 at
// 400x200x190, and of 12 iterations 2245 and 2058 at 256x128x128.  Rows too long for a
// block take k tiles, whose halo quads cost more, from kTilesFrom cells on: 639 and 648 at
// 20x16x700, but 815 and 751 at 60x64x300, 1393 and 1364 at 40x100x600; where the separate
// kernels' wavefronts fill (rows of whole wavefronts) from twice that: 766 and 775 at
// 64x48x384, 796 and 824 at 60x64x320, 1763 and 1676 at 96x100x320, 1074 and 1077 at 100x80x384
// and with 12 iterations 5550 and 4212 at 192x128x384.
const HalfGeom* half_geom(dalm_ctx* ctx, int pc_kind, int pc_it) {
    if (pc_kind != DALM_PC_JACOBI || pc_it != 3 || !ctx->may_take(DALM_PATH_HALVES)) return nullptr;
    if (!ctx->have_half) {
        ctx->half = split_half(ctx);
        ctx->have_half = true;
    }
    return ctx->half.R > 0 ? &ctx->half : nullptr;
}

static int launch_half(dalm_ctx* ctx, int which, const HalfArgs& h, const HalfGeom& G) {
    auto go = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, dim3(G.blocks), dim3(G.threads), G.lds, ctx->stream, ctx->d, ctx->pcf, ctx->coef(), h, G,
                           (const SolveState*)ctx->solve);
    };
    auto pick = [&](auto w) {
        constexpr int W = decltype(w)::value;
        if (G.mode == 2) go(kg_half4<W, 2, false>);
        else if (G.mode == 1) G.cols ? go(kg_half4<W, 1, true>) : go(kg_half4<W, 1, false>);
        else G.cols ? go(kg_half4<W, 0, true>) : go(kg_half4<W, 0, false>);
    };
    if (which == 0) pick(std::integral_constant<int, 0>());
    else pick(std::integral_constant<int, 1>());
    return hipGetLastError() == hipSuccess ? DALM_OK : DALM_HIP_ERROR;
}

int launch_half_p(dalm_ctx* ctx, const HalfGeom& G, const float* p_in, const float* q_in, float* p_out, float* q_out,
                  float* zp_out) {
    HalfArgs h{};
    h.r = ctx->fr;
    h.s_in = ctx->fs;
    h.t_in = ctx->ft;
    h.vin = p_in;
    h.qin = q_in;
    h.vout = p_out;
    h.zout = zp_out;
    h.yout = q_out;
    h.r0 = ctx->fr0;
    h.partials = ctx->partials;
    return launch_half(ctx, 0, h, G);
}

int launch_half_s(dalm_ctx* ctx, const HalfGeom& G, const float* q, float* zs_out) {
    HalfArgs h{};
    h.r = ctx->fr;
    h.qin = q;
    h.vout = ctx->fs;
    h.zout = zs_out;
    h.yout = ctx->ft;
    h.r0 = ctx->fr0;
    h.partials = ctx->partials;
    return launch_half(ctx, 1, h, G);
}
