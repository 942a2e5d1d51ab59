// Vector kernels for the Krylov solvers (part of edx_kernels.hip).
//
// Every reduction goes through per-block partial sums reduced by one block in
// a fixed order, so results do not depend on scheduling.  Scalars produced by
// one kernel and consumed by the next stay in device memory; kernels can skip
// themselves on a device flag, so a solver iteration is a fixed launch
// sequence with no host round trip.

namespace {

constexpr int VB = 256;   // threads per block for vector kernels

int vec_blocks(int64_t n) {
    int64_t g = (n + VB - 1) / VB;
    int64_t cap = (int64_t)edx::num_cus() * 4;
    if (g > cap) g = cap;
    if (g < 1) g = 1;
    return (int)g;
}

// sum of partials[0, nb) by one block; every thread gets the total.  A kernel that
// calls it twice needs a barrier between the calls.
__device__ double2 reduce_partials(const double2 *partials, int nb) {
    __shared__ double sx[VB], sy[VB];
    double2 s = make_double2(0, 0);
    for (int i = threadIdx.x; i < nb; i += VB) s = cadd(s, partials[i]);
    sx[threadIdx.x] = s.x;
    sy[threadIdx.x] = s.y;
    __syncthreads();
    for (int off = VB / 2; off > 0; off >>= 1) {
        if (threadIdx.x < off) {
            sx[threadIdx.x] += sx[threadIdx.x + off];
            sy[threadIdx.x] += sy[threadIdx.x + off];
        }
        __syncthreads();
    }
    return make_double2(sx[0], sy[0]);
}

// partials[b] = sum over block b's indices of conj(a) * b
__global__ __launch_bounds__(VB) void k_dot(int64_t n, const double2 *a, const double2 *b,
                                            double2 *partials, const int *run) {
    if (run && *run == 0) return;
    double2 s = make_double2(0, 0);
    for (int64_t i = blockIdx.x * (int64_t)VB + threadIdx.x; i < n; i += (int64_t)gridDim.x * VB)
        s = cadd(s, cconjmul(a[i], b[i]));
    s = block_sum_256(s);
    if (threadIdx.x == 0) partials[blockIdx.x] = s;
}

__global__ __launch_bounds__(VB) void k_reduce_to(const double2 *partials, int nb, double2 *out,
                                                  const int *run) {
    if (run && *run == 0) return;
    double2 s = reduce_partials(partials, nb);
    if (threadIdx.x == 0) *out = s;
}

// y = y / s  (s real, read from device)
__global__ __launch_bounds__(VB) void k_div_real(int64_t n, double2 *y, const double *s,
                                                 const int *run) {
    if (run && *run == 0) return;
    const double d = *s;
    for (int64_t i = blockIdx.x * (int64_t)VB + threadIdx.x; i < n; i += (int64_t)gridDim.x * VB)
        y[i] = make_double2(y[i].x / d, y[i].y / d);
}

// y = y - a * x (a real, device) and partials of |y|^2
template <bool TAIL>
__global__ __launch_bounds__(VB) void k_axpy_norm(int64_t n, double2 *y, const double2 *x,
                                                  const double *a, double2 *partials,
                                                  const int *run, StepTail tail) {
    if (run && *run == 0) return;
    const double al = *a;
    double2 s = make_double2(0, 0);
    for (int64_t i = blockIdx.x * (int64_t)VB + threadIdx.x; i < n; i += (int64_t)gridDim.x * VB) {
        double2 v = make_double2(y[i].x - al * x[i].x, y[i].y - al * x[i].y);
        y[i] = v;
        s.x += v.x * v.x + v.y * v.y;
    }
    s = block_sum_256(s);
    if (threadIdx.x == 0) part_put<TAIL>(partials + blockIdx.x, s);
    step_tail<TAIL>(tail, partials);
}

// Launch of the update that ends a step, on nb workgroups; then beta's part of
// the step where the launch had no tail.
int axpy_norm_step(int64_t n, double2 *y, const double2 *x, const double *a, double2 *partials,
                   const int *run, StepTail t, int nb) {
    hipStream_t s = edx::stream();
    t.op = TAIL_BETA;
    if (update_tail(nb, 1, n)) {
        hipLaunchKernelGGL(k_axpy_norm<true>, dim3(nb), dim3(VB), 0, s, n, y, x, a, partials, run, t);
        EDX_LAUNCH_CHECK();
        return EDX_OK;
    }
    hipLaunchKernelGGL(k_axpy_norm<false>, dim3(nb), dim3(VB), 0, s, n, y, x, a, partials, run, t);
    EDX_LAUNCH_CHECK();
    return step_finish_launch(t, partials, nb);
}

// ------------------------------------------------ Krylov (build_krylov_mp)

struct KrylovDev {
    double2 coef[2];   // SpMV epilogue: y = coef0*A x + coef1*z
    double2 sum;       // scratch for a reduced scalar
    double norm;       // <v0|v0>
    double sqrt_norm;
    double scur;       // scale of the current vector when it is kept unnormalized
    double acoef;      // alpha_i / scur
    int neff;
};

__global__ void k_krylov_init(KrylovDev *st, int *run) {
    st->coef[0] = make_double2(1.0, 0.0);
    st->coef[1] = make_double2(-0.0, 0.0);
    st->scur = 1.0;
    st->acoef = 0.0;
    st->neff = 0;
    run[0] = 1;
}

__global__ __launch_bounds__(VB) void k_krylov_norm(const double2 *partials, int nb, KrylovDev *st) {
    double2 s = reduce_partials(partials, nb);
    if (threadIdx.x == 0) {
        st->norm = s.x;
        st->sqrt_norm = sqrt(s.x);
    }
}

// The state of one recurrence as the step tails see it: a batch of one.
inline BKrylov krylov_state(KrylovDev *st, double *alpha, double *beta, int *run) {
    return BKrylov{alpha,        beta,         &st->norm,  &st->neff, run,
                   &st->coef[1], &st->sum,     &st->coef[0], &st->acoef, &st->scur};
}

// -------------------------------------------------------- MINRES (linsys)

struct MinresDev {
    double beta0, beta1;
    double2 sigma0, sigma1, gamma0, gamma1, eta, res;
    double2 alpha, rho1, rho2, rho3, inv_rho1, xcoef;
    double tol;
    int maxit;
    int iters;
};

__device__ __forceinline__ double2 cdiv(double2 a, double2 b) {
    const double den = b.x * b.x + b.y * b.y;
    return make_double2((a.x * b.x + a.y * b.y) / den, (a.y * b.x - a.x * b.y) / den);
}

// principal complex square root
__device__ __forceinline__ double2 csqrt_dev(double2 z) {
    const double r = hypot(z.x, z.y);
    if (r == 0.0) return make_double2(0.0, 0.0);
    double t = sqrt(0.5 * (r + fabs(z.x)));
    if (z.x >= 0.0) return make_double2(t, z.y / (2.0 * t));
    return make_double2(fabs(z.y) / (2.0 * t), z.y >= 0 ? t : -t);
}

__global__ __launch_bounds__(VB) void k_minres_init(const double2 *partials, int nb, MinresDev *st,
                                                    int *run, double tol, int maxit) {
    double2 s = reduce_partials(partials, nb);
    if (threadIdx.x == 0) {
        st->beta0 = sqrt(s.x);
        st->beta1 = 0.0;
        st->sigma0 = st->sigma1 = make_double2(0, 0);
        st->gamma0 = st->gamma1 = make_double2(1, 0);
        st->eta = make_double2(st->beta0, 0);
        st->res = make_double2(st->beta0, 0);
        st->tol = tol;
        st->maxit = maxit;
        st->iters = 0;
        run[0] = (hypot(st->res.x, st->res.y) > tol && 0 < maxit) ? 1 : 0;   // src/linsys.f90:76
    }
}

__global__ void k_minres_divbeta(int64_t n, double2 *v, const MinresDev *st, const int *run, int i) {
    if (!run[i]) return;
    const double d = st->beta0;
    for (int64_t k = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; k < n;
         k += (int64_t)gridDim.x * blockDim.x)
        v[k] = make_double2(v[k].x / d, v[k].y / d);
}

__global__ __launch_bounds__(VB) void k_minres_alpha(const double2 *partials, int nb, MinresDev *st,
                                                     const int *run, int i) {
    if (!run[i]) return;
    double2 s = reduce_partials(partials, nb);
    if (threadIdx.x == 0) st->alpha = s;
}

// v_prev = tmp - alpha v_curr - beta0 v_prev ; partial |v_prev|^2  (src/linsys.f90:87)
__global__ __launch_bounds__(VB) void k_minres_vupdate(int64_t n, const double2 *tmp,
                                                       const double2 *vc, double2 *vp,
                                                       const MinresDev *st, double2 *partials,
                                                       const int *run, int i) {
    if (!run[i]) return;
    const double2 al = st->alpha;
    const double b0 = st->beta0;
    double2 s = make_double2(0, 0);
    for (int64_t k = blockIdx.x * (int64_t)VB + threadIdx.x; k < n; k += (int64_t)gridDim.x * VB) {
        double2 v = csub(csub(tmp[k], cmul(al, vc[k])), cscale(vp[k], b0));
        vp[k] = v;
        s.x += v.x * v.x + v.y * v.y;
    }
    s = block_sum_256(s);
    if (threadIdx.x == 0) partials[blockIdx.x] = s;
}

// Givens update of src/linsys.f90:88-110 (complex-symmetric rotation)
__global__ __launch_bounds__(VB) void k_minres_scalars(const double2 *partials, int nb,
                                                       MinresDev *st, int *run, int i) {
    if (!run[i]) {
        if (threadIdx.x == 0) run[i + 1] = 0;
        return;
    }
    double2 s = reduce_partials(partials, nb);
    if (threadIdx.x == 0) {
        const double beta1 = sqrt(s.x);
        const double beta0 = st->beta0;
        const double2 alpha = st->alpha;
        const double2 delta = csub(cmul(st->gamma0, alpha), cscale(cmul(st->gamma1, st->sigma0), beta0));
        const double2 rho1 = csqrt_dev(cadd(cmul(delta, delta), make_double2(beta1 * beta1, 0.0)));
        const double2 rho2 = cadd(cmul(st->sigma0, alpha), cscale(cmul(st->gamma1, st->gamma0), beta0));
        const double2 rho3 = cscale(st->sigma1, beta0);
        st->gamma1 = st->gamma0;
        st->sigma1 = st->sigma0;
        st->gamma0 = cdiv(delta, rho1);
        st->sigma0 = cdiv(make_double2(beta1, 0.0), rho1);
        st->rho1 = rho1;
        st->rho2 = rho2;
        st->rho3 = rho3;
        st->inv_rho1 = cdiv(make_double2(1.0, 0.0), rho1);
        st->xcoef = cmul(st->gamma0, st->eta);
        const double as0 = hypot(st->sigma0.x, st->sigma0.y);
        st->res = cscale(st->res, as0);
        st->eta = make_double2(-(st->sigma0.x * st->eta.x - st->sigma0.y * st->eta.y),
                               -(st->sigma0.x * st->eta.y + st->sigma0.y * st->eta.x));
        st->beta1 = beta1;
        st->beta0 = beta1;
        st->iters = i + 1;
        run[i + 1] = (hypot(st->res.x, st->res.y) > st->tol && i + 1 < st->maxit) ? 1 : 0;
    }
}

// w_prev = (v_curr - rho3 w_prev - rho2 w_curr) / rho1 ; x += gamma0*eta*w_prev
__global__ __launch_bounds__(VB) void k_minres_wx(int64_t n, const double2 *vc, double2 *wp,
                                                  const double2 *wc, double2 *x,
                                                  const MinresDev *st, const int *run, int i) {
    if (!run[i]) return;
    const double2 r2 = st->rho2, r3 = st->rho3, ir1 = st->inv_rho1, xc = st->xcoef;
    for (int64_t k = blockIdx.x * (int64_t)VB + threadIdx.x; k < n; k += (int64_t)gridDim.x * VB) {
        double2 w = cmul(csub(csub(vc[k], cmul(r3, wp[k])), cmul(r2, wc[k])), ir1);
        wp[k] = w;
        x[k] = cadd(x[k], cmul(xc, w));
    }
}

// ------------------------------------------- Lanczos (full reorthogonalization)

// partials[c * nbx + bx] = sum_{r in block bx} conj(V[r, c]) * w[r], c in [c0, c0+8)
__global__ __launch_bounds__(VB) void k_gemv_ct(int64_t n, const double2 *V, int64_t ld, int k,
                                                const double2 *w, double2 *partials) {
    const int c0 = blockIdx.y * 8;
    double2 acc[8];
#pragma unroll
    for (int c = 0; c < 8; ++c) acc[c] = make_double2(0, 0);
    for (int64_t r = blockIdx.x * (int64_t)VB + threadIdx.x; r < n; r += (int64_t)gridDim.x * VB) {
        const double2 wr = w[r];
#pragma unroll
        for (int c = 0; c < 8; ++c)
            if (c0 + c < k) acc[c] = cadd(acc[c], cconjmul(V[(int64_t)(c0 + c) * ld + r], wr));
    }
#pragma unroll
    for (int c = 0; c < 8; ++c) {
        double2 s = block_sum_256(acc[c]);
        if (threadIdx.x == 0 && c0 + c < k) partials[(int64_t)(c0 + c) * gridDim.x + blockIdx.x] = s;
    }
}

// h[c] = sum_b partials[c * nbx + b] in the order of b, a workgroup per column: the
// partials are fetched by all threads, added by one.  With alpha, the last
// column is v_j and *alpha = dot + its component.
__global__ __launch_bounds__(VB) void k_reduce_cols(const double2 *partials, int nbx, double2 *h,
                                                    const double2 *dot, double *alpha) {
    __shared__ double2 s_p[VB];
    const double2 *p = partials + (int64_t)blockIdx.x * nbx;
    double2 s = make_double2(0, 0);
    for (int b0 = 0; b0 < nbx; b0 += VB) {
        __syncthreads();
        if (b0 + (int)threadIdx.x < nbx) s_p[threadIdx.x] = p[b0 + threadIdx.x];
        __syncthreads();
        if (threadIdx.x == 0) {
            const int e = nbx - b0 < VB ? nbx - b0 : VB;
#pragma unroll 8
            for (int b = 0; b < e; ++b) s = cadd(s, s_p[b]);
        }
    }
    if (threadIdx.x != 0) return;
    h[blockIdx.x] = s;
    if (alpha && blockIdx.x == gridDim.x - 1) *alpha = dot->x + s.x;
}

// ---- one step of fully reorthogonalized Lanczos
//
// w = H v_j - alpha v_j - beta v_{j-1}, made orthogonal to the k basis columns V
// by two classical Gram-Schmidt passes, in three passes over V instead of four
// (a pass reads 16 n k bytes and little else):
//   k_cgs_pass<FIRST>  the three-term part and c = V^H w;
//   k_cgs_pass         w -= V c and c' = V^H w, V's row staying in registers;
//   k_cgs_last         w -= V c' and |w|^2.
// The scalars stay on the device, so the host waits once per cycle.  Every sum
// is taken in the order of the plain kernels (k_dot, k_gemv_ct, k_gemv_n_sub):
// the signs of the Ritz vectors hang on the last bits of the coefficients (an
// off-diagonal entry at the eigensolver's threshold), so that another order
// would turn them around in a few runs of a hundred.
// A step over 705,432 rows and 3 to 22 columns (trlan, three states) takes 175 us,
// with two separate passes of two kernels, one-thread column sums (26 us each)
// and three waits 320.  k_cgs_pass reads 17 to 22 columns in 45 to 49 us (62
// without the next row's loads in flight); more workgroups would be faster
// (35 us) in another order of summation.

constexpr int CGS_MAXK = 32;   // columns a lane holds with their sums (8 registers each)

// FIRST: w -= dot v + b vprev (dot: the sum of nd partials, also stored to *dot).
// Else w -= V h.  Then partials[c * gridDim.x + bx] of V^H w.  A lane takes a row:
// its k <= KP entries in registers, k running sums.
template <int KP, bool FIRST>
__global__ __launch_bounds__(VB, 1) void k_cgs_pass(int64_t n, const double2 *V, int64_t ld, int k,
                                                    const double2 *h, const double2 *dotp, int nd,
                                                    double2 *dot, const double2 *vprev,
                                                    const double *bprev, double2 *w,
                                                    double2 *partials) {
    __shared__ double2 s_h[KP];
    __shared__ double2 s_sum[4][KP];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const double2 *vj = V + (int64_t)(k - 1) * ld;
    double a = 0.0, b = 0.0;
    if (FIRST) {
        const double2 d = reduce_partials(dotp, nd);
        a = d.x;
        if (vprev) b = *bprev;
        if (blockIdx.x == 0 && threadIdx.x == 0) *dot = d;
    } else {
        for (int c = threadIdx.x; c < k; c += VB) s_h[c] = h[c];
        __syncthreads();
    }
    double2 acc[KP];
#pragma unroll
    for (int c = 0; c < KP; ++c) acc[c] = make_double2(0, 0);
    constexpr bool AHEAD = KP <= 24;   // the next row's columns fit in registers too
    const int64_t stride = (int64_t)gridDim.x * VB;
    int64_t r = blockIdx.x * (int64_t)VB + threadIdx.x;
    double2 vn[AHEAD ? KP : 1], xn = make_double2(0, 0);
    auto ahead = [&](int64_t q) {
        if constexpr (AHEAD) {
            const int64_t o = q < n ? q : n - 1;
            xn = w[o];
#pragma unroll
            for (int c = 0; c < KP; ++c) vn[c] = V[(int64_t)(c < k ? c : k - 1) * ld + o];
        }
    };
    if (r < n) ahead(r);
    for (; r < n; r += stride) {
        double2 v[KP], x;
        if constexpr (AHEAD) {
            x = xn;
#pragma unroll
            for (int c = 0; c < KP; ++c) v[c] = vn[c];
            ahead(r + stride);
        } else {
            x = w[r];
#pragma unroll
            for (int c = 0; c < KP; ++c) v[c] = V[(int64_t)(c < k ? c : k - 1) * ld + r];
        }
        if (FIRST) {
            x = csub(x, cscale(vj[r], a));
            if (vprev) x = csub(x, cscale(vprev[r], b));
        } else {
            double2 s = make_double2(0, 0);
#pragma unroll
            for (int c = 0; c < KP; ++c)
                if (c < k) s = cadd(s, cmul(v[c], s_h[c]));
            x = csub(x, s);
        }
        w[r] = x;
#pragma unroll
        for (int c = 0; c < KP; ++c) acc[c] = cadd(acc[c], cconjmul(v[c], x));
    }
#pragma unroll
    for (int c = 0; c < KP; ++c) {
        double2 q = acc[c];
        for (int off = 32; off > 0; off >>= 1) {
            q.x += __shfl_xor(q.x, off, 64);
            q.y += __shfl_xor(q.y, off, 64);
        }
        if (lane == 0) s_sum[wave][c] = q;
    }
    __syncthreads();
    for (int c = threadIdx.x; c < k; c += VB)   // block_sum_256's order
        partials[(int64_t)c * gridDim.x + blockIdx.x] =
            cadd(cadd(s_sum[0][c], s_sum[1][c]), cadd(s_sum[2][c], s_sum[3][c]));
}

// k <= CGS_MAXK columns
template <bool FIRST>
int cgs_pass(int nb, int64_t n, const double2 *V, int64_t ld, int k, const double2 *h,
             const double2 *dotp, int nd, double2 *dot, const double2 *vprev, const double *bprev,
             double2 *w, double2 *partials) {
    hipStream_t s = edx::stream();
#define CGS_PASS(KP)                                                                             \
    hipLaunchKernelGGL((k_cgs_pass<KP, FIRST>), dim3(nb), dim3(VB), 0, s, n, V, ld, k, h, dotp, \
                       nd, dot, vprev, bprev, w, partials)
    if (k <= 8) CGS_PASS(8);
    else if (k <= 16) CGS_PASS(16);
    else if (k <= 24) CGS_PASS(24);
    else CGS_PASS(CGS_MAXK);
#undef CGS_PASS
    EDX_LAUNCH_CHECK();
    return EDX_OK;
}

// w -= dot vj + bprev vprev (more columns than k_cgs_pass takes)
__global__ __launch_bounds__(VB) void k_cgs_three(int64_t n, double2 *w, const double2 *vj,
                                                  const double2 *dot, const double2 *vprev,
                                                  const double *bprev) {
    const double a = dot->x, b = vprev ? *bprev : 0.0;
    for (int64_t r = blockIdx.x * (int64_t)VB + threadIdx.x; r < n; r += (int64_t)gridDim.x * VB) {
        double2 x = csub(w[r], cscale(vj[r], a));
        if (vprev) x = csub(x, cscale(vprev[r], b));
        w[r] = x;
    }
}

// w[r] -= sum_c V[r, c] h[c]
__global__ __launch_bounds__(VB) void k_gemv_n_sub(int64_t n, const double2 *V, int64_t ld, int k,
                                                   const double2 *h, double2 *w) {
    __shared__ double2 hs[1024];
    for (int c = threadIdx.x; c < k && c < 1024; c += VB) hs[c] = h[c];
    __syncthreads();
    for (int64_t r = blockIdx.x * (int64_t)VB + threadIdx.x; r < n; r += (int64_t)gridDim.x * VB) {
        double2 s = make_double2(0, 0);
        for (int c = 0; c < k; ++c) s = cadd(s, cmul(V[(int64_t)c * ld + r], c < 1024 ? hs[c] : h[c]));
        w[r] = csub(w[r], s);
    }
}

// w -= V h and partials of |w|^2
__global__ __launch_bounds__(VB) void k_cgs_last(int64_t n, const double2 *V, int64_t ld, int k,
                                                 const double2 *h, double2 *w, double2 *partials) {
    __shared__ double2 hs[1024];
    for (int c = threadIdx.x; c < k && c < 1024; c += VB) hs[c] = h[c];
    __syncthreads();
    double2 nrm = make_double2(0, 0);
    for (int64_t r = blockIdx.x * (int64_t)VB + threadIdx.x; r < n; r += (int64_t)gridDim.x * VB) {
        double2 s = make_double2(0, 0);
        for (int c = 0; c < k; ++c) s = cadd(s, cmul(V[(int64_t)c * ld + r], c < 1024 ? hs[c] : h[c]));
        const double2 x = csub(w[r], s);
        w[r] = x;
        nrm = cadd(nrm, cconjmul(x, x));
    }
    nrm = block_sum_256(nrm);
    if (threadIdx.x == 0) partials[blockIdx.x] = nrm;
}

// *beta = |w|; with ab, *alpha and it there
__global__ __launch_bounds__(VB) void k_cgs_beta(const double2 *partials, int nb, double *beta,
                                                 const double *alpha, double *ab) {
    const double2 s = reduce_partials(partials, nb);
    if (threadIdx.x != 0) return;
    const double b = sqrt(fabs(s.x));
    *beta = b;
    if (ab) {
        ab[0] = *alpha;
        ab[1] = b;
    }
}

// *beta = |w| from the nd partials of k_cgs_last, out = w / *beta; 0 past an invariant
// subspace
__global__ __launch_bounds__(VB) void k_cgs_next(int64_t n, const double2 *w, const double2 *partials,
                                                 int nd, double *beta, double2 *out) {
    const double b = sqrt(fabs(reduce_partials(partials, nd).x));
    if (blockIdx.x == 0 && threadIdx.x == 0) *beta = b;
    for (int64_t i = blockIdx.x * (int64_t)VB + threadIdx.x; i < n; i += (int64_t)gridDim.x * VB)
        out[i] = b < 1e-10 ? make_double2(0, 0) : make_double2(w[i].x / b, w[i].y / b);
}

// X[:, j] = sum_c V[:, c] S[c + j*k]  (S real, column-major k x nvec).  KC > 0: a
// row of V (k <= KC columns) in registers, read once for all nvec vectors (12 from
// 22 columns of 705,432 rows: 400 us reading it for each vector).
template <int KC>
__global__ __launch_bounds__(VB) void k_combine(int64_t n, const double2 *V, int64_t ld, int k,
                                                const double *S, int nvec, double2 *X, int64_t ldx) {
    for (int64_t r = blockIdx.x * (int64_t)VB + threadIdx.x; r < n; r += (int64_t)gridDim.x * VB) {
        if constexpr (KC > 0) {
            double2 v[KC];
#pragma unroll
            for (int c = 0; c < KC; ++c) v[c] = c < k ? V[(int64_t)c * ld + r] : make_double2(0, 0);
            for (int j = 0; j < nvec; ++j) {
                double2 s = make_double2(0, 0);
#pragma unroll
                for (int c = 0; c < KC; ++c)
                    if (c < k) s = cadd(s, cscale(v[c], S[(int64_t)j * k + c]));
                X[(int64_t)j * ldx + r] = s;
            }
        } else {
            for (int j = 0; j < nvec; ++j) {
                double2 s = make_double2(0, 0);
                for (int c = 0; c < k; ++c)
                    s = cadd(s, cscale(V[(int64_t)c * ld + r], S[(int64_t)j * k + c]));
                X[(int64_t)j * ldx + r] = s;
            }
        }
    }
}

int combine_launch(int nb, int64_t n, const double2 *V, int64_t ld, int k, const double *S, int nvec,
                   double2 *X, int64_t ldx) {
    hipStream_t s = edx::stream();
    if (k <= 16)
        hipLaunchKernelGGL(k_combine<16>, dim3(nb), dim3(VB), 0, s, n, V, ld, k, S, nvec, X, ldx);
    else if (k <= 24)
        hipLaunchKernelGGL(k_combine<24>, dim3(nb), dim3(VB), 0, s, n, V, ld, k, S, nvec, X, ldx);
    else if (k <= 32)
        hipLaunchKernelGGL(k_combine<32>, dim3(nb), dim3(VB), 0, s, n, V, ld, k, S, nvec, X, ldx);
    else
        hipLaunchKernelGGL(k_combine<0>, dim3(nb), dim3(VB), 0, s, n, V, ld, k, S, nvec, X, ldx);
    EDX_LAUNCH_CHECK();
    return EDX_OK;
}

// A step of the two-pass recurrence after its product w = H v (k_dot's partials
// dotp): w -= alpha v + *bprev vprev, *alpha = Re <v|w>, norm partials.
__global__ __launch_bounds__(VB) void k_two_pass_first(int64_t n, double2 *w, const double2 *v,
                                                       const double2 *dotp, int nd, double *alpha,
                                                       const double2 *vprev, const double *bprev,
                                                       double2 *partials) {
    const double a = reduce_partials(dotp, nd).x, b = vprev ? *bprev : 0.0;
    if (blockIdx.x == 0 && threadIdx.x == 0) *alpha = a;
    double2 s = make_double2(0, 0);
    for (int64_t i = blockIdx.x * (int64_t)VB + threadIdx.x; i < n; i += (int64_t)gridDim.x * VB) {
        double2 x = csub(w[i], cscale(v[i], a));
        if (vprev) x = csub(x, cscale(vprev[i], b));
        w[i] = x;
        s = cadd(s, cconjmul(x, x));
    }
    s = block_sum_256(s);
    if (threadIdx.x == 0) partials[blockIdx.x] = s;
}

// The same step run again with its alpha a and betas: X -= c v, and the next
// vector (w - a v - b vprev) / beta over vprev.
__global__ __launch_bounds__(VB) void k_two_pass_again(int64_t n, const double2 *w, const double2 *v,
                                                       double a, double2 *vprev, int tri, double b,
                                                       double beta, double2 *X, double c) {
    for (int64_t i = blockIdx.x * (int64_t)VB + threadIdx.x; i < n; i += (int64_t)gridDim.x * VB) {
        const double2 vi = v[i];
        X[i] = csub(X[i], cscale(vi, c));
        double2 x = csub(w[i], cscale(vi, a));
        if (tri) x = csub(x, cscale(vprev[i], b));
        vprev[i] = make_double2(x.x / beta, x.y / beta);
    }
}

__device__ __forceinline__ uint64_t splitmix64(uint64_t x) {
    x += 0x9e3779b97f4a7c15ull;
    x = (x ^ (x >> 30)) * 0xbf58476d1ce4e5b9ull;
    x = (x ^ (x >> 27)) * 0x94d049bb133111ebull;
    return x ^ (x >> 31);
}

// real uniform start vector in [-0.5, 0.5) as in src/lanczos.f90:60-61, seeded
__global__ void k_random_real(int64_t n, uint64_t seed, double2 *v) {
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n;
         i += (int64_t)gridDim.x * blockDim.x) {
        uint64_t h = splitmix64(seed * 0x100000001b3ull + (uint64_t)i);
        v[i] = make_double2((double)(h >> 11) * (1.0 / 9007199254740992.0) - 0.5, 0.0);
    }
}

__global__ void k_scale_real(int64_t n, double2 *v, double s) {
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n;
         i += (int64_t)gridDim.x * blockDim.x)
        v[i] = cscale(v[i], s);
}

// w = w - a*x - b*y  (a, b real host scalars)
__global__ void k_axpby_sub(int64_t n, double2 *w, const double2 *x, double a, const double2 *y,
                            double b) {
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n;
         i += (int64_t)gridDim.x * blockDim.x) {
        double2 v = w[i];
        v = csub(v, cscale(x[i], a));
        if (y) v = csub(v, cscale(y[i], b));
        w[i] = v;
    }
}

__global__ void k_copy_div(int64_t n, const double2 *in, double s, double2 *out) {
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n;
         i += (int64_t)gridDim.x * blockDim.x)
        out[i] = make_double2(in[i].x / s, in[i].y / s);
}

__global__ void k_sub_vec(int64_t n, double2 *a, const double2 *b) {
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n;
         i += (int64_t)gridDim.x * blockDim.x)
        a[i] = csub(a[i], b[i]);
}

}  // namespace
