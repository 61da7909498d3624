// resident_mixed.hip -- the precision form's SOR (run_sor_mixed in poisson_mixed.hip) of
// small grids in one launch per solve: FP64 residual, kSorInner red-black FP32 iterations
// on the correction, FP64 update, until the reference's test holds on the true residual.
//
// As the FP64 solver of resident.hip, with the FP32 correction's halo words in the sweeps:
// half the bytes an exchange, and no sum to wait for inside a refinement.  What bounds it
// is the 16 sweeps' chain of exchanges: 64x48x48 takes 5.0 us per iteration of two sweeps,
// against 9.2 us with a launch per sweep.
#include "resident.h"
#include "stencil.h"

namespace {

// Whether a ghost cell that a block's residual reads holds a value that is not finite.  Their
// coefficients are zero, so finite ones need no reading (nor registers: with the slab loaded
// whole, 64x48x48 took 5.24 instead of 5.02 ms), but zero times an infinity is no number, and
// the solve ends on it as with a launch per sweep.
template <int M>
__device__ __forceinline__ bool ghosts_not_finite(const Dims& d, const ResThread<M>& t, const double* __restrict__ x) {
    const int g = d.gc;
    bool bad = false;
    const auto see = [&](int i, int j, int k) { bad |= !(fabs(x[d.at(g + i, g + j, g + k)]) < HUGE_VAL); };
    for (int e = threadIdx.x; e < t.planes * d.ny; e += blockDim.x)
        for (int k : {-1, d.nz}) see(t.first + e / d.ny, e % d.ny, k);
    for (int e = threadIdx.x; e < t.planes * d.nz; e += blockDim.x)
        for (int j : {-1, d.ny}) see(t.first + e / d.nz, j, e % d.nz);
    for (int e = threadIdx.x; e < d.ny * d.nz; e += blockDim.x) {
        if (!t.has_l) see(-1, e / d.nz, e % d.nz);
        if (!t.has_r) see(d.nx, e / d.nz, e % d.nz);
    }
    return bad;
}

template <int M>
__global__ __launch_bounds__(res_threads(M)) void k_res_sor_mixed(Dims d, PCoef A, PCoefF Af, ResShape s,
                                                                  const double* __restrict__ x, const double* b,
                                                                  double* __restrict__ out, float omega, int inner,
                                                                  long long max_it, double tol, double root_n,
                                                                  SolveState* st) {
    extern __shared__ __align__(16) double slab[];  // the residual's x, then the sweeps' e (as floats)
    float* const eslab = (float*)slab;
    __shared__ ResSync sh;
    __shared__ int ghost;
    if (threadIdx.x < 2) sh.bad[threadIdx.x] = 0;
    if (threadIdx.x == 0) ghost = 0;
    __syncthreads();
    ResThread<M> t = res_thread<M>(d, s);
    if (ghosts_not_finite(d, t, x)) ghost = 1;
    const int g = d.gc;
    const int plane = s.pj * s.pk, half = (s.P + 2) * plane;
    double xv[2][M];
    float e[2][M], r[2][M], acf[2][M], rcf[2][M], anf[M], asf[M], aef[M], awf[M];
    unsigned has[2] = {0, 0}, odd = 0;  // odd: the colour-0 cell of the pair is the one with odd k
    float atf[2], abf[2];
#pragma unroll
    for (int q = 0; q < 2; ++q) {
        const int k = g + (t.k >= 0 && 2 * t.k + q < d.nz ? 2 * t.k + q : 0);
        atf[q] = Af.at[k];
        abf[q] = Af.ab[k];
    }
#pragma unroll
    for (int m = 0; m < M; ++m) {
        const bool in = t.has(m);
        const int row = in ? t.row(s, m) : 0;
        const int i = g + t.first + row / d.ny, j = g + row % d.ny;
        anf[m] = Af.an[j], asf[m] = Af.as[j], aef[m] = Af.ae[i], awf[m] = Af.aw[i];
        const int o = (i + j + g) & 1;
        odd |= (unsigned)o << m;
#pragma unroll
        for (int c = 0; c < 2; ++c) {
            const int k = in ? 2 * t.k + (c ^ o) : 0;
            const bool cell = in && k < d.nz;
            has[c] |= (unsigned)cell << m;
            // quieted: x is published as it came, and a signalling NaN of the caller's could be
            // the mark of an empty slot
            xv[c][m] = cell ? __builtin_canonicalize(x[d.at(i, j, g + k)]) : 0.0;
            const int kc = cell ? g + k : g;
            acf[c][m] = (((Af.acx[i] - Af.anu[j]) - Af.asu[j]) - Af.atu[kc]) - Af.abu[kc];
            rcf[c][m] = __builtin_amdgcn_rcpf(acf[c][m]);
            e[c][m] = r[c][m] = 0.f;
        }
    }
    auto keep = [&](int c) {
        return [&d, &t, c, g](int j, int i) { return 2 * t.k + (c ^ ((3 * g + i + j) & 1)) < d.nz; };
    };
    auto sweep = [&](int c) {
        const float* O = eslab + (c ^ 1) * half;
        float e1[M];
#pragma unroll
        for (int m = 0; m < M; ++m) {
            const int q = t.lds[m];
            const bool hi = (((odd >> m) & 1) != 0) != (c != 0);  // this cell has odd k
            const float side = O[hi ? q + 1 : q - 1], mate = e[c ^ 1][m];
            const float et = hi ? side : mate, eb = hi ? mate : side;
            const float ax = acf[c][m] * e[c][m] + aef[m] * O[q + plane] + awf[m] * O[q - plane] + anf[m] * O[q + s.pk] +
                             asf[m] * O[q - s.pk] + (hi ? atf[1] : atf[0]) * et + (hi ? abf[1] : abf[0]) * eb;
            e1[m] = e[c][m] + omega * (r[c][m] - ax) * rcf[c][m];
        }
#pragma unroll
        for (int m = 0; m < M; ++m)
            if ((has[c] >> m) & 1) {
                res_publish<float, M>(d, s, t, m, e1[m]);
                e[c][m] = e1[m];
                eslab[c * half + t.lds[m]] = e1[m];
            }
        res_take<float, M>(d, s, t, sh, eslab + c * half, keep(c));
    };
    double err = 0;
    int status = DALM_OK;
    long long it = 0;
    for (;;) {
        // x and its halo; cells off the interior stay zero (their coefficients are)
        for (int q = threadIdx.x; q < 2 * half; q += blockDim.x) slab[q] = 0.0;
        if (!res_barrier(sh, t)) return;
#pragma unroll
        for (int c = 0; c < 2; ++c) {
#pragma unroll
            for (int m = 0; m < M; ++m)
                if ((has[c] >> m) & 1) {
                    res_publish<double, M>(d, s, t, m, xv[c][m]);
                    slab[c * half + t.lds[m]] = xv[c][m];
                }
            res_take<double, M>(d, s, t, sh, slab + c * half, keep(c));
        }
        if (!res_barrier(sh, t)) return;
        double v[1] = {it == 0 && ghost ? (double)NAN : 0.0};
        // once in `inner` iterations the FP64 operator and b are read again instead of held
        // beside the sweeps' values; the empty statement keeps the compiler from doing that
        // ahead of the loop (the registers it took spilled: 7.8 ms a solve)
        int now = 0;
        asm volatile("" : "+v"(now));
#pragma unroll
        for (int c = 0; c < 2; ++c) {
            const double* O = slab + (c ^ 1) * half;
#pragma unroll
            for (int m = 0; m < M; ++m) {
                if (!((has[c] >> m) & 1)) continue;
                const int q = t.lds[m];
                const bool hi = (((odd >> m) & 1) != 0) != (c != 0);
                const int row = t.row(s, m) + now;
                const int i = g + t.first + row / d.ny, j = g + row % d.ny, k = g + 2 * t.k + (hi ? 1 : 0) + now;
                const double ac = ((((A.acx[i] - A.anu[j]) - A.asu[j]) - A.atu[k]) - A.abu[k]) / A.max_diag;
                const double side = O[hi ? q + 1 : q - 1], mate = xv[c ^ 1][m];
                const double xt = hi ? side : mate, xb = hi ? mate : side;
                const double rv = b[d.at(i, j, k)] -
                                  (ac * xv[c][m] + A.ae[i] * O[q + plane] + A.aw[i] * O[q - plane] +
                                   A.an[j] * O[q + s.pk] + A.as[j] * O[q - s.pk] + A.at[k] * xt + A.ab[k] * xb);
                r[c][m] = (float)rv;
                v[0] += rv * rv;
            }
        }
        if (!res_sum<1, M>(v, s, t, sh)) return;
        err = sqrt(sh.out[0]) / root_n;
        if (!(err == err) || isinf(err)) {
            status = DALM_NONFINITE;
            break;
        }
        if (it > 0 && err <= tol) break;
        if (it >= max_it) {
            status = DALM_NONCONVERGED;
            break;
        }
        it += inner;
        for (int q = threadIdx.x; q < 2 * half; q += blockDim.x) eslab[q] = 0.f;
#pragma unroll
        for (int m = 0; m < M; ++m) e[0][m] = e[1][m] = 0.f;
        if (!res_barrier(sh, t)) return;
        for (int n = 0; n < inner; ++n) {
            sweep(0);
            if (!res_barrier(sh, t)) return;
            sweep(1);
            if (!res_barrier(sh, t)) return;
        }
#pragma unroll
        for (int c = 0; c < 2; ++c)
#pragma unroll
            for (int m = 0; m < M; ++m) xv[c][m] += (double)e[c][m];
    }
#pragma unroll
    for (int m = 0; m < M; ++m) {
        const int row = t.row(s, m);
#pragma unroll
        for (int c = 0; c < 2; ++c)
            if ((has[c] >> m) & 1)
                out[d.at(g + t.first + row / d.ny, g + row % d.ny, g + 2 * t.k + (c ^ (int)((odd >> m) & 1)))] = xv[c][m];
    }
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        st->it = it;
        st->err = err;
        st->status = status;
        st->done = 1;
    }
}

}  // namespace

int res_sor_mixed(dalm_ctx* ctx, double omega, int inner, long long max_it, double tol, bool* ran) {
    *ran = false;
    if (!res_may_run(ctx, max_it, 3)) return DALM_OK;  // two colours, and the refinement's three in `inner`
    ResShape s = res_shape(ctx, (ctx->d.nz + 1) / 2, 2 * sizeof(double));
    if (s.blocks == 0) return DALM_OK;
    if (int rc = res_prepare(ctx, s)) return rc;
    if (ctx->res_off) return DALM_OK;
    const double root_n = sqrt((double)ctx->N);
    auto launch = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, dim3(s.blocks), dim3(s.threads), s.lds, ctx->stream, ctx->d, ctx->coef(), ctx->pcf, s,
                           (const double*)ctx->p, (const double*)ctx->b, ctx->r, (float)omega, inner, max_it, tol, root_n,
                           ctx->solve);
    };
    switch (s.M) {
    case 1: launch(k_res_sor_mixed<1>); break;
    case 2: launch(k_res_sor_mixed<2>); break;
    case 3: launch(k_res_sor_mixed<3>); break;
    default: launch(k_res_sor_mixed<4>); break;
    }
    HIP_TRY(hipGetLastError());
    return res_finish(ctx, ctx->p, ran);
}
