// The scalar work between the passes of a Krylov step (part of edx_kernels.hip).
//
// A step is a product with dot partials, alpha from their sum, a vector update
// with norm partials, beta from their sum (and, in the multi-shift solve, the
// shift recurrences).  On matrices of up to a few hundred thousand rows a pass
// takes 5 to 40 us, so separate one-block kernels for the sums and scalars
// (3 us each at the least, launched one after another) would be up to half of
// the step.  Instead the last workgroup of a pass to finish does them: each
// workgroup stores its partials past the L2 of its XCD (agent scope), waits for
// the stores, and counts itself in; whoever completes the count sums the
// partials in a fixed order, so the result does not depend on who that is.
// Arrivals are counted in TAIL_GROUPS counters and then one, because the adds
// to one address follow one another at 12 ns: a launch of 1024 workgroups takes
// 2.9 us without a tail, 14.9 us with one counter, 5.7 us with 8, and 5.9 us
// followed by a reduction kernel.  Launches too wide for that, or with too many
// partials for one workgroup to sum, end without a tail, and k_step_reduce (one
// workgroup per right-hand side, the sum and the scalars in one launch) follows
// them.  Measured: a step of one vector over 10,296 rows 21.5 -> 15.0 us; a step
// of the two-vector multi-shift solve over 1.0M rows 137 -> 128 us.

namespace {

// The recurrence keeps its vectors unnormalized: the stored u_i is the
// residual w_i of the previous step, with v_i = u_i / s_i and s_i = beta_i
// (s_1 = 1 after the start vector is normalized).  The product of a step is
// y = (1/s_i) H u_i - (beta_i / s_{i-1}) u_{i-1} = H v_i - beta_i v_{i-1}, its
// dot <u_i|y> / s_i = alpha_i, and the residual y - (alpha_i / s_i) u_i is the
// next stored vector: no pass divides a vector by beta.
struct BKrylov {
    double *alpha;     // [maxn * K], alpha[(i-1)*K + k]
    double *beta;      // [(maxn+1) * K]
    double *norm;      // [K]
    int *neff;         // [K]
    int *run;          // [(maxn+1) * K]
    double2 *c1;       // [K]  -beta_i / s_{i-1}: coefficient of u_{i-1} in the product
    double2 *sums;     // [K]
    double2 *c0;       // [K]  1 / s_i: scale of H u_i in the product
    double *acoef;     // [K]  alpha_i / s_i: coefficient of u_i in the residual
    double *scur;      // [K]  s_i
};

struct MsShift {
    double2 sigma;
    double2 eta;       // pivot eta_i
    double2 inv_eta;   // 1 / eta_i
    double2 zeta;      // zeta_i
    double res;        // residual estimate of the last finished iterate (absolute)
    int active;        // still iterating
    int iters;         // iterate the stored projection belongs to
};

struct MsCtl {
    double tol_abs;
    int nactive;
};

__device__ __forceinline__ double2 crecip(double2 a) {
    const double d = a.x * a.x + a.y * a.y;
    return make_double2(a.x / d, -a.y / d);
}

__device__ __forceinline__ double cabs2(double2 a) { return sqrt(a.x * a.x + a.y * a.y); }

enum { TAIL_ALPHA = 1, TAIL_BETA = 2 };
constexpr int TAIL_GROUPS = 32;
constexpr int TAIL_STRIDE = 32;   // counters 128 bytes apart
constexpr size_t TAIL_BYTES = (TAIL_GROUPS + 1) * TAIL_STRIDE * sizeof(unsigned);

// What the end of a pass computes for each right-hand side k < K.
struct StepTail {
    unsigned *count;     // zeroed arrival counters; nullptr: the launch has no tail
    int op;              // TAIL_ALPHA, TAIL_BETA
    int i;               // step, 1-based
    int K;
    BKrylov st;
    // multi-shift solve: K right-hand sides of nshift shifts each, else nshift = 0
    int nshift;
    MsShift *sh;         // [K * nshift]
    MsCtl *ctl;          // [K]
    const double *sqn;   // [K] norms of the right-hand sides
};

// Whether a product's launch of nbx workgroups, each with a partial for K right-hand
// sides, ends with a tail.  The four waves of the last one sum a right-hand side each, so
// a fifth waits; a single one they share.  Measured, us a step with the tail and without:
// one vector, 462 to 24,310 rows 13.5 to 15.4, 14.2 to 16.9; two vectors, 174
// partials 17.4, 18.3, 297 18.5, 18.5, 403 19.3, 18.4; four, 108 18.9, 19.6, 174 19.7,
// 19.7, 215 19.8, 19.5; eight, 29 20.0, 19.9, 403 26.9, 22.8.
bool product_tail(int64_t nbx, int K) {
    return K == 1 ? nbx <= 1024 : K <= 4 && nbx * K <= 640;
}

// The same for the update of K interleaved vectors over n rows, whose workgroups have up
// to sixteen waves.  Measured the same way, without tails of the product: twelve vectors,
// 75 partials 25.3, 25.8, 101 24.0, 23.8; four, 161 23.6, 24.1, 256 (18,018 rows) 26.5,
// 26.4; two, 256 22.3, 23.3, but over 38,610 rows 30.8, 30.6; 24 vectors, 8 partials
// 25.9, 25.6, 256 (48,620 rows) 76.5, 67.0.
bool update_tail(int64_t nbx, int K, int64_t n) {
    return K == 1 ? nbx <= 1024 : K <= 16 && nbx * K <= 900 && n <= 32768;
}

// TAIL: the kernel is the instance for launches with a tail.  (The others stay
// free of its registers: the shift recurrences' divisions take more than most
// passes do.)
template <bool TAIL> __device__ __forceinline__ void part_put(double2 *p, double2 v) {
    if constexpr (TAIL) {
        __hip_atomic_store(&p->x, v.x, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __hip_atomic_store(&p->y, v.y, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    } else {
        *p = v;
    }
}

__device__ __forceinline__ double2 part_get(const double2 *p) {
    return make_double2(__hip_atomic_load(&p->x, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT),
                        __hip_atomic_load(&p->y, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
}

// Step i (1-based) of the shift recurrences of right-hand side k, after alpha_i
// = a is known, by one wave (lanes over shifts).  A shift whose iterate i-1
// already meets the tolerance is frozen there.
__device__ __forceinline__ void tail_shifts(const StepTail &t, int k, double a, int lane) {
    MsShift *sh = t.sh + (int64_t)k * t.nshift;
    MsCtl *ctl = t.ctl + k;
    const int64_t o = (int64_t)(t.i - 1) * t.K + k;
    const double tol = ctl->tol_abs, nb = t.sqn[k];
    int c = 0;
    for (int q = lane; q < t.nshift; q += 64) {
        MsShift s = sh[q];
        if (t.i == 1) {
            s.eta = make_double2(s.sigma.x - a, s.sigma.y);
            s.zeta = make_double2(nb, 0.0);
            s.active = 1;
            s.iters = 0;
            s.res = nb;
        } else if (s.active) {
            const double bp = t.st.beta[o];
            const double2 ratio = cmul(s.zeta, s.inv_eta);   // zeta_{i-1} / eta_{i-1}
            s.res = bp * cabs2(ratio);
            if (s.res <= tol) {
                s.active = 0;
            } else {
                s.zeta = cscale(ratio, bp);
                const double2 r = cscale(s.inv_eta, bp * bp);
                s.eta = make_double2(s.sigma.x - a - r.x, s.sigma.y - r.y);
            }
        }
        if (s.active) {
            s.inv_eta = crecip(s.eta);
            s.iters = t.i;
            ++c;
        }
        sh[q] = s;
    }
    for (int off = 32; off > 0; off >>= 1) c += __shfl_xor(c, off, 64);
    if (lane == 0) ctl->nactive = c;
}

// The scalars of right-hand side k from the sum of its partials, by one wave.
__device__ __forceinline__ void step_finish(const StepTail &t, int k, double2 sum, int lane) {
    const BKrylov &s = t.st;
    const int64_t o = (int64_t)(t.i - 1) * t.K + k;
    const bool run = s.run[o] != 0;
    if (t.op == TAIL_ALPHA) {
        if (!run) return;
        const double inv = s.c0[k].x;
        const double a = sum.x * inv;
        if (lane == 0) {
            s.alpha[o] = a;
            s.acoef[k] = a * inv;
            s.neff[k] = t.i;
        }
        if (t.nshift) tail_shifts(t, k, a, lane);
    } else if (lane == 0) {
        const int64_t on = (int64_t)t.i * t.K + k;
        if (!run) {
            s.run[on] = 0;
            return;
        }
        const double b = sqrt(sum.x);
        s.beta[on] = b;
        s.c1[k] = make_double2(-b / s.scur[k], -0.0);
        s.scur[k] = b;
        s.c0[k] = make_double2(b > 0.0 ? 1.0 / b : 0.0, 0.0);
        // src/lanczos.f90:290-293; a right-hand side without an active shift is done
        s.run[on] = fabs(b) < 1e-10 || (t.nshift && t.ctl[k].nactive == 0) ? 0 : 1;
    }
}

// The sum of one right-hand side's partials: quarter q adds those of index
// q * 64 + lane + 256 j per lane, the quarters are joined per lane as (0 + 2) +
// (1 + 3), then the lanes as a tree.  It does not depend on how many
// right-hand sides or waves there are (and is k_breduce's sum, bit for bit).
__device__ __forceinline__ double2 join_quarters(double2 q0, double2 q1, double2 q2, double2 q3) {
    return cadd(cadd(q0, q2), cadd(q1, q3));
}

__device__ __forceinline__ double2 wave_sum_tail(double2 v) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
        v.x += __shfl_xor(v.x, off, 64);
        v.y += __shfl_xor(v.y, off, 64);
    }
    return v;
}

// Counts workgroup id of total in; true for the one that completes the count
// (which leaves the counters zero).  One thread calls it.
__device__ __forceinline__ bool tail_arrive(unsigned *count, unsigned id, unsigned total) {
    const unsigned g = id % TAIL_GROUPS, of = (total + TAIL_GROUPS - 1 - g) / TAIL_GROUPS;
    unsigned *c = count + g * TAIL_STRIDE, *top = count + TAIL_GROUPS * TAIL_STRIDE;
    if (__hip_atomic_fetch_add(c, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != of - 1)
        return false;
    __hip_atomic_store(c, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    const unsigned ng = total < TAIL_GROUPS ? total : TAIL_GROUPS;
    if (__hip_atomic_fetch_add(top, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != ng - 1)
        return false;
    __hip_atomic_store(top, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    return true;
}

// Quarter q of right-hand side k's partials, per lane.
__device__ __forceinline__ double2 tail_quarter(const double2 *partials, int nb, int K, int k, int q,
                                                int lane) {
    double2 s = make_double2(0, 0);
    const double2 *p = partials + k;
#pragma unroll 4
    for (int b = q * 64 + lane; b < nb; b += 256) s = cadd(s, part_get(p + b * K));
    return s;
}

// End of a pass whose workgroups wrote partials[blockIdx.x * K + k] by part_put.
// Every thread of the workgroup calls it; whole waves.  A wave sums a
// right-hand side; a single one is shared by the four waves of a workgroup.
template <bool TAIL>
__device__ __forceinline__ void step_tail(const StepTail &t, const double2 *partials) {
    if constexpr (!TAIL) return;
    __shared__ int s_last;
    __shared__ double2 s_sum[3][64];
    // this wave's partials have left for memory before its workgroup counts itself in
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (threadIdx.x == 0)
        s_last = tail_arrive(t.count, blockIdx.y * gridDim.x + blockIdx.x, gridDim.x * gridDim.y);
    __syncthreads();
    if (!s_last) return;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, nw = (blockDim.x + 63) >> 6;
    const int nb = gridDim.x, K = t.K;
    if (K == 1 && nw == 4) {
        const double2 q = tail_quarter(partials, nb, 1, 0, wave, lane);
        if (wave) s_sum[wave - 1][lane] = q;
        __syncthreads();
        if (wave == 0)
            step_finish(t, 0, wave_sum_tail(join_quarters(q, s_sum[0][lane], s_sum[1][lane],
                                                          s_sum[2][lane])), lane);
        return;
    }
    for (int k = wave; k < K; k += nw) {
        double2 q[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) q[i] = tail_quarter(partials, nb, K, k, i, lane);
        step_finish(t, k, wave_sum_tail(join_quarters(q[0], q[1], q[2], q[3])), lane);
    }
}

// The sum of right-hand side k's partials by one workgroup of 256 threads, in
// its wave 0.
__device__ __forceinline__ double2 block_partials(const double2 *partials, int nb, int K, int k) {
    __shared__ double2 s_sum[4][64];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    double2 s = make_double2(0, 0);
#pragma unroll 4
    for (int b = threadIdx.x; b < nb; b += 256) s = cadd(s, partials[(int64_t)b * K + k]);
    s_sum[wave][lane] = s;   // wave q: quarter q
    __syncthreads();
    if (wave != 0) return s;
    return wave_sum_tail(join_quarters(s, s_sum[1][lane], s_sum[2][lane], s_sum[3][lane]));
}

// The same for a launch without a tail: workgroup k sums nb partials of
// right-hand side k.
__global__ __launch_bounds__(256) void k_step_reduce(StepTail t, const double2 *partials, int nb) {
    const int k = blockIdx.x;
    const double2 s = block_partials(partials, nb, t.K, k);
    if (threadIdx.x < 64) step_finish(t, k, s, threadIdx.x);
}

// After a pass with tail t: nb = 0 if the pass ran it, else its partials per
// right-hand side.
int step_finish_launch(const StepTail &t, const double2 *partials, int nb) {
    if (nb <= 0) return EDX_OK;
    hipLaunchKernelGGL(k_step_reduce, dim3(t.K), dim3(256), 0, edx::stream(), t, partials, nb);
    EDX_LAUNCH_CHECK();
    return EDX_OK;
}

}  // namespace
