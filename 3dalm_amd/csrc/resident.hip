// resident.hip -- the FP64 Poisson solvers of small grids in one launch per solve:
// red-black SOR (src/eq.h:145-306) and BiCGStab with Jacobi or SOR preconditioning
// (src/eq.h:6-143, 308-473).  resident.h holds the exchange between blocks.
//
// What bounds them is the chain of dependent phases of an iteration (a colour sweep, a
// Jacobi sweep, a product, a sum over the grid), each a store that must reach the
// neighbour and be read: 1.2 to 1.5 us against the 4.7 us of a launch.  The work inside
// a phase is 0.1 to 0.8 us.  Per iteration, in microseconds, one launch per sweep and
// resident: SOR 64x32x32 15.3 and 3.0, 64x48x48 17.5 and 5.2; BiCGStab with three Jacobi
// sweeps 20x12x12 37.7 and 12.5, 64x32x32 42.8 and 16.5, with two SOR sweeps 52.6 and 15.5,
// 60.2 and 20.5.
//
// Per cell the arithmetic is that of the one-launch-per-sweep kernels in poisson.hip
// (the same operands in the same order, division included), so SOR iterates are the
// reference's bit for bit and BiCGStab differs in the summation order of its dot
// products only.  Compiled with -ffp-contract=off.
#include <float.h>
#include <cstdlib>

#include "resident.h"
#include "stencil.h"

namespace {

// the iteration's end as the finalize kernels decide it (FIN_SOR, FIN_BI_XR)
__device__ __forceinline__ bool sor_done(double err, long long it, long long max_it, double tol, int* status) {
    if (!(err == err) || isinf(err)) {
        *status = DALM_NONFINITE;
        return true;
    }
    if (it < max_it && err > tol) return false;
    *status = err > tol ? DALM_NONCONVERGED : DALM_OK;
    return true;
}
__device__ __forceinline__ void store_state(SolveState* st, long long it, double err, int status) {
    st->it = it;
    st->err = err;
    st->status = status;
    st->done = 1;
}

// ---- red-black SOR -----------------------------------------------------------------
// A lane position is a pair of cells (k = 2 kk, 2 kk + 1), one of either colour, so every
// lane works in both sweeps.  The slab holds the two colours apart: the neighbours of a
// row's cells of one colour are then consecutive in the other colour's plane (no bank
// conflicts), and one of the two k neighbours is the pair's other cell, in a register.
//
// The residual of an iteration costs no pass of its own.  At the colour swept last it is
// evaluated in the sweep, from the neighbours that the sweep has read (they have the other
// colour and stay as they are); at the colour swept first, the next iteration's sweep
// forms it as its correction.  The stopping test of iteration n is therefore known at the
// end of iteration n + 1, and the sum over the blocks travels beside that iteration's
// second sweep; each thread keeps the values of iteration n and puts them back if n was
// the last.
template <int M>
__global__ __launch_bounds__(res_threads(M)) void k_res_sor(Dims d, PCoef A, ResShape s, const double* __restrict__ x,
                                                         const double* __restrict__ b, double* __restrict__ out,
                                                         double omega, long long max_it, double tol, double root_n,
                                                         SolveState* st) {
    extern __shared__ __align__(16) double slab[];
    __shared__ ResSync sh;
    if (threadIdx.x < 2) sh.bad[threadIdx.x] = 0;
    ResThread<M> t = res_thread<M>(d, s);
    const int g = d.gc;
    const int plane = s.pj * s.pk, half = (s.P + 2) * plane;
    // the slab with its shell of neighbours and ghost cells, colour by colour
    for (int e = threadIdx.x; e < 2 * (t.planes + 2) * s.pj * s.pk; e += blockDim.x) {
        const int c = e & 1;  // which cell of the pair
        int r = e >> 1;
        const int kk = r % s.pk - 1;
        r /= s.pk;
        const int j = r % s.pj - 1, p = r / s.pj;
        const int i = t.first + p - 1, k = 2 * kk + c;
        double v = 0.0;
        if (k >= -1 && k <= d.nz) v = x[d.at(g + i, g + j, g + k)];
        const int color = (3 * g + i + j + k) & 1;
        slab[color * half + (p * s.pj + j + 1) * s.pk + kk + 1] = v;
    }
    double xv[2][M], bv[2][M], ac[2][M], ra[2][M], an[M], as[M], ae[M], aw[M], old[2][M];
    unsigned has[2] = {0, 0}, odd = 0;  // odd: the colour-0 cell of the pair is the one with odd k
    double at[2], ab[2];
#pragma unroll
    for (int q = 0; q < 2; ++q) {
        const int k = g + (t.k >= 0 && 2 * t.k + q < d.nz ? 2 * t.k + q : 0);
        at[q] = A.at[k];
        ab[q] = A.ab[k];
    }
#pragma unroll
    for (int m = 0; m < M; ++m) {
        const bool in = t.has(m);
        const int row = in ? t.row(s, m) : 0;
        const int i = g + t.first + row / d.ny, j = g + row % d.ny;
        an[m] = A.an[j];
        as[m] = A.as[j];
        ae[m] = A.ae[i];
        aw[m] = A.aw[i];
        const int o = (i + j + g) & 1;
        odd |= (unsigned)o << m;
#pragma unroll
        for (int c = 0; c < 2; ++c) {
            const int k = in ? 2 * t.k + (c ^ o) : 0;
            const bool cell = in && k < d.nz;
            has[c] |= (unsigned)cell << m;
            // the absent partner of an odd row's last cell is the ghost beyond it
            const int at_ = d.at(i, j, g + k);
            xv[c][m] = old[c][m] = x[at_];
            bv[c][m] = cell ? b[at_] : 0.0;
            const int kc = cell ? g + k : g;
            ac[c][m] = ((((A.acx[i] - A.anu[j]) - A.asu[j]) - A.atu[kc]) - A.abu[kc]) / A.max_diag;
            ra[c][m] = recip(ac[c][m]);
        }
    }
    double v[1] = {0.0};  // this thread's part of |r|^2 of the iteration under test
    auto sweep = [&](int c) {
        const double* O = slab + (c ^ 1) * half;
#pragma unroll
        for (int m = 0; m < M; ++m) {
            const int e = t.lds[m];
            const bool hi = (((odd >> m) & 1) != 0) != (c != 0);  // this cell has odd k
            const double side = O[hi ? e + 1 : e - 1], mate = xv[c ^ 1][m];
            const double xt = hi ? side : mate, xb = hi ? mate : side;
            const double xe = O[e + plane], xw = O[e - plane], xn = O[e + s.pk], xs = O[e - s.pk];
            // A x in the reference's order
            auto apply = [&](double x0) {
                return ac[c][m] * x0 + ae[m] * xe + aw[m] * xw + an[m] * xn + as[m] * xs + (hi ? at[1] : at[0]) * xt +
                       (hi ? ab[1] : ab[0]) * xb;
            };
            const double r = bv[c][m] - apply(xv[c][m]);
            const double x1 = xv[c][m] + omega * div_by(r, ac[c][m], ra[c][m]);
            const double rn = c == 0 ? r : bv[c][m] - apply(x1);
            old[c][m] = xv[c][m];
            if ((has[c] >> m) & 1) {
                v[0] += rn * rn;
                xv[c][m] = x1;
            }
        }
        // the stores after the last read: the positions' chains of arithmetic overlap
#pragma unroll
        for (int m = 0; m < M; ++m)
            if ((has[c] >> m) & 1) {
                res_publish<double, M>(d, s, t, m, xv[c][m]);
                slab[c * half + t.lds[m]] = xv[c][m];
            }
    };
    auto take = [&](int c) {
        res_take<double, M>(d, s, t, sh, slab + c * half, [&](int j, int i) {
            return 2 * t.k + (c ^ ((3 * g + i + j) & 1)) < d.nz;
        });
    };
    if (!res_barrier(sh, t)) return;
    double err = 0;
    int status = DALM_OK;
    // it: iterations finished; the test of the last of them runs beside the next one's
    // second sweep
    long long it = 0;
    for (;; ++it) {
        sweep(0);
        res_sum_wave<1>(v, sh);
        v[0] = 0.0;
        take(0);
        if (!res_barrier(sh, t)) return;
        if (it > 0) res_sum_send<1, M>(s, t, sh);
        sweep(1);
        take(1);
        if (it > 0) res_sum_take<1, M>(s, t, sh);
        if (!res_barrier(sh, t)) return;
        if (it > 0) {
            err = sqrt(sh.out[0]) / root_n;
            if (sor_done(err, it, max_it, tol, &status)) break;
        }
    }
#pragma unroll
    for (int m = 0; m < M; ++m) {
        const int row = t.row(s, m);
#pragma unroll
        for (int c = 0; c < 2; ++c)
            if ((has[c] >> m) & 1)
                out[d.at(g + t.first + row / d.ny, g + row % d.ny, g + 2 * t.k + (c ^ (int)((odd >> m) & 1)))] = old[c][m];
    }
    if (blockIdx.x == 0 && threadIdx.x == 0) store_state(st, it, err, status);
}

// ---- BiCGStab ------------------------------------------------------------------------
// A lane position is a cell; every Krylov vector lives in registers, and the slab holds
// the one vector whose neighbours the next sweep or product reads.  Each level writes
// its cells to the slab, sends and takes the halo planes and meets at a barrier; the
// next level's values replace them after another one.
template <int M, bool JAC>
__global__ __launch_bounds__(res_threads(M)) void k_res_bicgstab(Dims d, PCoef A, ResShape s,
                                                              const double* __restrict__ x_in,
                                                              const double* __restrict__ b, double* __restrict__ out,
                                                              double pc_omega, int pc_it, long long max_it, double tol,
                                                              double root_n, SolveState* st) {
    extern __shared__ __align__(16) double slab[];
    __shared__ ResSync sh;
    if (threadIdx.x < 2) sh.bad[threadIdx.x] = 0;
    ResThread<M> t = res_thread<M>(d, s);
    const int g = d.gc, plane = s.pj * s.pk, cells = (t.planes + 2) * plane;
    for (int e = threadIdx.x; e < cells; e += blockDim.x) {
        const int k = e % s.pk - 1, r = e / s.pk;
        slab[e] = x_in[d.at(g + t.first + r / s.pj - 1, g + r % s.pj - 1, g + k)];
    }
    double x[M], r[M], r0[M], p[M], q[M], sv[M], tv[M], zp[M], z[M], ac[M], ra[M];
    double an[M], as[M], ae[M], aw[M];
    int cell[M];
    unsigned color = 0;
    const int kc = g + (t.k >= 0 ? t.k : 0);
    const double at = A.at[kc], ab = A.ab[kc];
#pragma unroll
    for (int m = 0; m < M; ++m) {
        const int row = t.has(m) ? t.row(s, m) : 0;
        const int i = g + t.first + row / d.ny, j = g + row % d.ny;
        cell[m] = d.at(i, j, kc);
        if ((i + j + kc) & 1) color |= 1u << m;  // padded indices, as the reference's colours
        an[m] = A.an[j];
        as[m] = A.as[j];
        ae[m] = A.ae[i];
        aw[m] = A.aw[i];
        ac[m] = ((((A.acx[i] - A.anu[j]) - A.asu[j]) - A.atu[kc]) - A.abu[kc]) / A.max_diag;
        ra[m] = recip(ac[m]);
    }
    auto apply = [&](int m, double c) {
        const double* Z = slab + t.lds[m];
        return ac[m] * c + ae[m] * Z[plane] + aw[m] * Z[-plane] + an[m] * Z[s.pk] + as[m] * Z[-s.pk] + at * Z[1] +
               ab * Z[-1];
    };
    // the halo of the slab's vector y, whose own cells every thread has in registers
    auto spread = [&](const double(&y)[M]) {
#pragma unroll
        for (int m = 0; m < M; ++m) {
            if (!t.has(m)) continue;
            res_publish<double, M>(d, s, t, m, y[m]);
            slab[t.lds[m]] = y[m];
        }
        res_take<double, M>(d, s, t, sh, slab, [](int, int) { return true; });
        return res_barrier(sh, t);
    };
    // y ~ A^-1 w in pc_it sweeps from zero; leaves y in the slab with its halo
    auto precondition = [&](double(&y)[M], const double(&w)[M]) {
        if (JAC) {
#pragma unroll
            for (int m = 0; m < M; ++m) y[m] = div_by(w[m], ac[m], ra[m]);
            if (!spread(y)) return false;
            for (int n = 1; n < pc_it; ++n) {
#pragma unroll
                for (int m = 0; m < M; ++m)
                    y[m] = y[m] + div_by(w[m] - apply(m, y[m]), ac[m], ra[m]);
                if (!res_barrier(sh, t)) return false;
                if (!spread(y)) return false;
            }
            return true;
        }
        for (int e = threadIdx.x; e < cells; e += blockDim.x) slab[e] = 0.0;
#pragma unroll
        for (int m = 0; m < M; ++m) y[m] = 0.0;
        if (!res_barrier(sh, t)) return false;
        for (int n = 0; n < pc_it; ++n)
            for (int c = 0; c < 2; ++c) {
#pragma unroll
                for (int m = 0; m < M; ++m) {
                    const double y1 = y[m] + pc_omega * div_by(w[m] - apply(m, y[m]), ac[m], ra[m]);
                    if (((color >> m) & 1) == (unsigned)c) y[m] = y1;
                }
#pragma unroll
                for (int m = 0; m < M; ++m) {
                    if (!t.has(m) || ((color >> m) & 1) != (unsigned)c) continue;
                    res_publish<double, M>(d, s, t, m, y[m]);
                    slab[t.lds[m]] = y[m];
                }
                res_take<double, M>(d, s, t, sh, slab, [&](int j, int i) { return ((3 * g + i + j + t.k + c) & 1) == 0; });
                if (!res_barrier(sh, t)) return false;
            }
        return true;
    };
    if (!res_barrier(sh, t)) return;
    double v1[1] = {0.0}, v2[2];
#pragma unroll
    for (int m = 0; m < M; ++m) {
        x[m] = r[m] = r0[m] = p[m] = q[m] = sv[m] = tv[m] = zp[m] = z[m] = 0.0;
        if (!t.has(m)) continue;
        x[m] = x_in[cell[m]];
        r[m] = b[cell[m]] - apply(m, x[m]);
        r0[m] = r[m];
        v1[0] += r[m] * r[m];
    }
    if (!res_sum<1, M>(v1, s, t, sh)) return;
    // the iterates' ghost cells are zero (every thread is past its reads of x)
    for (int e = threadIdx.x; e < cells; e += blockDim.x) slab[e] = 0.0;
    if (!res_barrier(sh, t)) return;
    double rho = sh.out[0], beta = 0, alpha = 1, om = 1, err = 0;
    long long it = 0;
    int status = DALM_OK;
    bool done = false;
    if (fabs(rho) < (double)FLT_MIN) {
        err = rho;
        status = DALM_BREAKDOWN;
        done = true;
    }
    while (!done) {
#pragma unroll
        for (int m = 0; m < M; ++m) p[m] = it == 0 ? r[m] : r[m] + beta * (p[m] - om * q[m]);
        if (!precondition(zp, p)) return;
        v1[0] = 0.0;
#pragma unroll
        for (int m = 0; m < M; ++m)
        {
            q[m] = apply(m, zp[m]);
            if (t.has(m)) v1[0] += r0[m] * q[m];
        }
        if (!res_sum<1, M>(v1, s, t, sh)) return;
        alpha = rho / sh.out[0];
#pragma unroll
        for (int m = 0; m < M; ++m) sv[m] = r[m] - alpha * q[m];
        if (!precondition(z, sv)) return;
        v2[0] = v2[1] = 0.0;
#pragma unroll
        for (int m = 0; m < M; ++m)
        {
            tv[m] = apply(m, z[m]);
            if (t.has(m)) {
                v2[0] += tv[m] * sv[m];
                v2[1] += tv[m] * tv[m];
            }
        }
        if (!res_sum<2, M>(v2, s, t, sh)) return;
        om = sh.out[0] / sh.out[1];
        v2[0] = v2[1] = 0.0;
#pragma unroll
        for (int m = 0; m < M; ++m) {
            x[m] = x[m] + alpha * zp[m] + om * z[m];
            r[m] = sv[m] - om * tv[m];
            if (t.has(m)) {
                v2[0] += r[m] * r[m];
                v2[1] += r0[m] * r[m];
            }
        }
        if (!res_sum<2, M>(v2, s, t, sh)) return;
        err = sqrt(sh.out[0]) / root_n;
        const double rho_new = sh.out[1];
        ++it;
        done = sor_done(err, it, max_it, tol, &status);
        if (!done && fabs(rho_new) < (double)FLT_MIN) {
            err = rho_new;
            status = DALM_BREAKDOWN;
            done = true;
        }
        beta = (rho_new / rho) * (alpha / om);
        rho = rho_new;
    }
#pragma unroll
    for (int m = 0; m < M; ++m)
        if (t.has(m)) out[cell[m]] = x[m];
    if (blockIdx.x == 0 && threadIdx.x == 0) store_state(st, it, err, status);
}

__global__ void k_slots_empty(long long n, u64w* __restrict__ a, long long nf, unsigned* __restrict__ f, int* abort_flag) {
    const long long e0 = blockIdx.x * (long long)blockDim.x + threadIdx.x, step = (long long)gridDim.x * blockDim.x;
    for (long long e = e0; e < n; e += step) a[e] = kEmpty;
    for (long long e = e0; e < nf; e += step) f[e] = kEmptyF;
    if (e0 == 0) *abort_flag = 0;
}

__global__ __launch_bounds__(BLOCK) void k_res_commit(Dims d, double* __restrict__ x, const double* __restrict__ from) {
    const TileRange tr = block_tiles(d);
    for (int q = tr.begin; q < tr.end; ++q) {
        const Cell cc = tile_cell(d, q);
        if (!cc.inside) continue;
        const int c = d.at(cc.i, cc.j, cc.k);
        x[c] = from[c];
    }
}

}  // namespace

// LDS of a slab at most: a compute unit's 160 KB less the static part
constexpr size_t kResLds = 150 * 1024;

ResShape res_shape(const dalm_ctx* ctx, int lanes, size_t bytes) {
    const Dims& d = ctx->d;
    ResShape s{};
    s.nk = lanes;
    s.pj = d.ny + 2;
    s.pk = lanes + 2;
    // positions per thread for slabs of P planes (0: does not fit)
    auto positions = [&](int P) {
        if ((size_t)(P + 2) * s.pj * s.pk * bytes > kResLds) return 0;
        for (int M = 1; M <= kResMaxM; ++M)
            if ((long long)(res_threads(M) / lanes) * M >= (long long)P * d.ny) return M;
        return 0;
    };
    // one block needs no exchange: it takes the whole grid where it fits; otherwise the
    // slabs are as thin as a quarter of the compute units allows
    int P = d.nx;
    if (!positions(P)) {
        int most = ctx->ncu / 4;
        if (most > kResMaxBlocks) most = kResMaxBlocks;
        if (most < 1) most = 1;
        P = (d.nx + most - 1) / most;
        if (!positions(P)) return s;
    }
    s.P = P;
    s.blocks = (d.nx + P - 1) / P;
    s.M = positions(P);
    s.rw = (P * d.ny + s.M - 1) / s.M;
    s.threads = (s.rw * lanes + 63) / 64 * 64;
    s.lds = (size_t)(P + 2) * s.pj * s.pk * bytes;
    return s;
}

int res_prepare(dalm_ctx* ctx, ResShape& s) {
    // slots for the largest split of this grid: one word per cell of a plane, direction,
    // block and set
    const Dims& d = ctx->d;
    const size_t most = d.nx < kResMaxBlocks ? d.nx : kResMaxBlocks;
    const size_t ring = (size_t)kSlotSets * 2 * most * d.ny * d.nz;
    const size_t gath = (size_t)kSlotSets * most * 4 * most;
    if (!ctx->res_ring) {
        if (hipMalloc(&ctx->res_ring, (ring + gath) * sizeof(u64w) + ring * sizeof(unsigned) + 64) != hipSuccess) {
            (void)hipGetLastError();  // no room for the slots: the launches per sweep need none
            ctx->res_ring = nullptr;
            ctx->res_off = true;
            return DALM_OK;
        }
        ctx->res_dirty = true;
        const char* spin = getenv("DALM_RESIDENT_SPIN");
        ctx->res_spin = spin ? atoi(spin) : kSpinLimit;
    }
    s.spin = ctx->res_spin;
    s.ring = (u64w*)ctx->res_ring;
    s.gath = s.ring + ring;
    s.ringf = (unsigned*)(s.gath + gath);
    s.abort_flag = (int*)(s.ringf + ring);
    ctx->res_abort = s.abort_flag;
    if (ctx->res_dirty) {
        hipLaunchKernelGGL(k_slots_empty, dim3(1024), dim3(256), 0, ctx->stream, (long long)(ring + gath), s.ring,
                           (long long)ring, s.ringf, s.abort_flag);
        HIP_TRY(hipGetLastError());
        ctx->res_dirty = false;
    }
    return DALM_OK;
}

int res_finish(dalm_ctx* ctx, double* x, bool* ran) {
    int* flag = (int*)(ctx->h_solve + 2);
    HIP_TRY(hipMemcpyAsync(ctx->h_solve, ctx->solve, sizeof(SolveState), hipMemcpyDeviceToHost, ctx->stream));
    HIP_TRY(hipMemcpyAsync(flag, ctx->res_abort, sizeof(int), hipMemcpyDeviceToHost, ctx->stream));
    HIP_TRY(hipStreamSynchronize(ctx->stream));
    if (*flag != 0) {
        // something keeps this context's blocks off the GPU: it does not wait for that again
        ctx->res_off = true;
        ++ctx->taken[DALM_PATH_GIVEN_UP];
        return DALM_OK;
    }
    hipLaunchKernelGGL(k_res_commit, dim3(ctx->grid), dim3(BLOCK), 0, ctx->stream, ctx->d, x, (const double*)ctx->r);
    HIP_TRY(hipGetLastError());
    *ran = true;
    ++ctx->taken[DALM_PATH_ONE_LAUNCH];
    return DALM_OK;
}

// A solve that may take more exchanges than this keeps the launches per sweep (the GPU stays
// available to other programs between them), and so does one whose launches are timed: at
// 1.2 to 2.6 us each a launch ends after about a second at most, whatever its cap of
// iterations and the sweeps of each (20000 iterations with up to five SOR sweeps fit).
constexpr long long kResMaxExchanges = 1LL << 19;
bool res_may_run(const dalm_ctx* ctx, long long max_it, long long exchanges) {
    return !ctx->res_off && ctx->may_take(DALM_PATH_ONE_LAUNCH) && ctx->probe.kernel == 0 &&
           max_it <= kResMaxExchanges / exchanges;
}

int res_sor(dalm_ctx* ctx, double* x, const double* b, double omega, long long max_it, double tol, bool* ran) {
    *ran = false;
    if (!res_may_run(ctx, max_it, 2)) return DALM_OK;
    ResShape s = res_shape(ctx, (ctx->d.nz + 1) / 2, 2 * sizeof(double));
    if (s.blocks == 0) return DALM_OK;
    if (int rc = res_prepare(ctx, s)) return rc;
    if (ctx->res_off) return DALM_OK;
    const double root_n = sqrt((double)ctx->N);
    auto launch = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, dim3(s.blocks), dim3(s.threads), s.lds, ctx->stream, ctx->d, ctx->coef(), s, x, b,
                           ctx->r, omega, max_it, tol, root_n, ctx->solve);
    };
    switch (s.M) {
    case 1: launch(k_res_sor<1>); break;
    case 2: launch(k_res_sor<2>); break;
    case 3: launch(k_res_sor<3>); break;
    default: launch(k_res_sor<4>); break;
    }
    HIP_TRY(hipGetLastError());
    return res_finish(ctx, x, ran);
}

int res_bicgstab(dalm_ctx* ctx, double* x, const double* b, int pc_kind, double pc_omega, int pc_it, long long max_it,
                 double tol, bool* ran) {
    *ran = false;
    // a cap of no iterations (an adjoint solve's) leaves x as it is: this kernel does one at least
    if (pc_it < 1 || max_it < 1) return DALM_OK;
    // each half-iteration's sweeps (two colours in SOR), and three sums
    if (!res_may_run(ctx, max_it, 2LL * pc_it * (pc_kind == DALM_PC_JACOBI ? 1 : 2) + 3)) return DALM_OK;
    ResShape s = res_shape(ctx, ctx->d.nz, sizeof(double));
    if (s.blocks == 0) return DALM_OK;
    if (int rc = res_prepare(ctx, s)) return rc;
    if (ctx->res_off) return DALM_OK;
    const double root_n = sqrt((double)ctx->N);
    auto launch = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, dim3(s.blocks), dim3(s.threads), s.lds, ctx->stream, ctx->d, ctx->coef(), s, x, b,
                           ctx->r, pc_omega, pc_it, max_it, tol, root_n, ctx->solve);
    };
    const bool jac = pc_kind == DALM_PC_JACOBI;
    switch (s.M) {
    case 1: jac ? launch(k_res_bicgstab<1, true>) : launch(k_res_bicgstab<1, false>); break;
    case 2: jac ? launch(k_res_bicgstab<2, true>) : launch(k_res_bicgstab<2, false>); break;
    case 3: jac ? launch(k_res_bicgstab<3, true>) : launch(k_res_bicgstab<3, false>); break;
    default: jac ? launch(k_res_bicgstab<4, true>) : launch(k_res_bicgstab<4, false>); break;
    }
    HIP_TRY(hipGetLastError());
    return res_finish(ctx, x, ran);
}
