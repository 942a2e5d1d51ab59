// Matrix-free Hamiltonian apply (part of edx_kernels.hip).
//
// For spaces too large to keep as CSR (the core-hole space at norb=26, N=13:
// 57,946,200 rows), y = c0 H x + c1 z is computed on the fly: every term is
// tested, signed and ranked as the CSR build does (the core-hole layout of
// src/ham.f90:419-446), so it lands on the column and with the sign the build
// gives it.  The omega diagonal of ham_sign = -1 is added last as in
// src/ham.f90:156-176.  Only the summation order differs from a CSR product,
// so results agree to rounding.
//
// No matrix is read: per row the traffic is the gathers of x and the epilogue
// vectors, and the work is the term tests (integer ALU).  Two kernels:
//   * k_plan_apply, for complete bases: 64 rows per workgroup over the terms
//     grouped by column (termplan.hip), those of equal action merged;
//   * k_mf, for incomplete bases, more than 4096 terms, rows of more than 255
//     entries, and too few rows for their terms (mf_max_groups): one 64-lane wave per
//     row, its lanes testing the terms in parallel and accumulating
//     val * sign * x[col] over the survivors.

namespace {

constexpr int MF_CAP = 128;   // surviving terms of one row compacted in LDS

__device__ __forceinline__ double2 wave_sum64(double2 v) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
        v.x += __shfl_xor(v.x, off, 64);
        v.y += __shfl_xor(v.y, off, 64);
    }
    return v;
}

// A term survives on word w exactly when its annihilated orbitals are
// occupied and its created ones are empty once those are removed:
//   (w & occ) == occ  and  (w & ~occ & emp) == 0,
// the conditions op_ann / op_cre test one operator at a time (a term that
// annihilates or creates the same orbital twice never survives: occ = ~0).
struct MfMask {
    uint64_t occ, emp;
};

__global__ void k_mf_masks(const uint32_t *ops, int T, int nhop, MfMask *masks) {
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= T) return;
    const uint32_t op = ops[t];
    const int a = op & 63, b = (op >> 8) & 63, c = (op >> 16) & 63, d = (op >> 24) & 63;
    MfMask k;
    if (t < nhop) {
        k.occ = 1ull << a;
        k.emp = 1ull << b;
    } else if (a == b || c == d) {
        k.occ = ~0ull;
        k.emp = 0;
    } else {
        k.occ = (1ull << a) | (1ull << b);
        k.emp = (1ull << c) | (1ull << d);
    }
    masks[t] = k;
}

// Pass 1 of a row: lanes test the terms with the masks and ballot-compact the
// survivors numbered [base, base + MF_CAP) into LDS; returns the row's
// survivor count.
__device__ __forceinline__ int mf_compact(const BuildParams &p, const MfMask *__restrict__ masks,
                                          uint64_t w, int base, uint32_t *s_t) {
    const int lane = threadIdx.x;
    int n = 0;
    for (int t0 = 0; t0 < p.T; t0 += 64) {
        const int t = t0 + lane;
        bool ok = false;
        if (t < p.T) {
            const MfMask k = masks[t];
            ok = (w & k.occ) == k.occ && (w & ~k.occ & k.emp) == 0;
        }
        const uint64_t mask = __ballot(ok);
        const int pos = n + lanes_below(mask) - base;
        n += __popcll(mask);
        if (ok && pos >= 0 && pos < MF_CAP) s_t[pos] = (uint32_t)t;
    }
    return n;
}

// Pass 2: lanes take the compacted survivors: the operator steps of the CSR
// build (new word and fermion sign), the column rank and the x gather.
template <int CK>
__device__ __forceinline__ double2 mf_gather(const BuildParams &p, const double2 *__restrict__ x,
                                             uint64_t w, int count, const uint32_t *s_t) {
    double2 acc = make_double2(0, 0);
    for (int q = threadIdx.x; q < count; q += 64) {
        const int t = (int)s_t[q];
        const uint32_t op = p.ops[t];
        uint64_t m = w;
        int par = 0;
        if (t < p.nhop) {
            op_ann(m, op & 63, par);
            op_cre(m, (op >> 8) & 63, par);
        } else {
            op_ann(m, op & 63, par);
            op_ann(m, (op >> 8) & 63, par);
            op_cre(m, (op >> 16) & 63, par);
            op_cre(m, (op >> 24) & 63, par);
        }
        const int64_t c = col_of<CK>(p, m);
        if (c < 0) continue;
        double2 v = p.tv[t];
        if ((par ^ p.negate) & 1) v = make_double2(-v.x, -v.y);
        acc = cadd(acc, cmul(v, x[c]));
    }
    return acc;
}

// One 64-lane workgroup per row: compact the surviving terms, then rank and
// gather them in parallel, so the costly rank runs once per surviving term
// instead of once per wave-wide batch of terms.  Rows with more than MF_CAP
// survivors take further compaction passes.
template <int RK, int CK>
__global__ __launch_bounds__(64) void k_mf(BuildParams p, const MfMask *__restrict__ masks,
                                           const double2 *__restrict__ x, SpmvEpi e) {
    if (e.run && *e.run == 0) return;
    __shared__ uint32_t s_t[MF_CAP];
    const int lane = threadIdx.x;
    const double2 c0 = e.c0 ? *e.c0 : make_double2(1.0, 0.0);
    const double2 c1 = e.c1 ? *e.c1 : make_double2(1.0, 0.0);
    double2 dot = make_double2(0, 0);
    for (int64_t r = blockIdx.x; r < p.M; r += gridDim.x) {
        const uint64_t w = row_word<RK>(p, r);
        const int n = mf_compact(p, masks, w, 0, s_t);
        __syncthreads();
        double2 acc = mf_gather<CK>(p, x, w, n < MF_CAP ? n : MF_CAP, s_t);
        for (int base = MF_CAP; base < n; base += MF_CAP) {
            __syncthreads();
            mf_compact(p, masks, w, base, s_t);
            __syncthreads();
            acc = cadd(acc, mf_gather<CK>(p, x, w, n - base < MF_CAP ? n - base : MF_CAP, s_t));
        }
        __syncthreads();
        acc = wave_sum64(acc);
        if (lane == 0) {
            double2 ax = acc;
            if (p.omega_on) ax = cadd(ax, cmul(p.omega, x[r]));
            double2 out = cmul(c0, ax);
            if (e.z) out = cadd(out, cmul(c1, e.z[r]));
            e.y[r] = out;
            if (e.dvec) dot = cadd(dot, cconjmul(e.dvec[r], out));
        }
    }
    if (e.dvec && lane == 0) e.partials[blockIdx.x] = dot;
}

// The product over a term plan.  A workgroup of NW waves owns 64 rows.  Lane =
// row throughout: the waves find the surviving groups of their chunks and list
// them per row in LDS; each wave sums its share of the diagonal group, whose
// density terms are the same for every lane and come by scalar loads, and takes
// entries q, q + NW, ... of each row (sum of the group's terms, column rank, x
// gather); the partial rows are added as a tree, so the result does not depend on
// timing.  Bound by integer and LDS instructions (136 groups tested,
// 24 columns ranked per row; the vectors take 0.03 ms): H_n norb 20, 1.0M rows,
// 0.35 ms a product, by k_mf 4.38 ms.
template <int NW, int RK, int CK, class W>
__global__ __launch_bounds__(64 * NW) void k_plan_apply(Plan<W> p, int cap, const double2 *__restrict__ x,
                                                    SpmvEpi e) {
    if (e.run && *e.run == 0) return;
    extern __shared__ __attribute__((aligned(16))) char s_mem[];
    int32_t *s_rank = reinterpret_cast<int32_t *>(s_mem);                   // rank_len
    uint16_t *s_grp = reinterpret_cast<uint16_t *>(s_rank + p.rank_len);    // [cap][64]
    __shared__ int s_cnt[NW][PLAN_ROWS];
    __shared__ double2 s_acc[NW][PLAN_ROWS];
    const int lane = threadIdx.x & 63, wave = plan_wave();
    const int64_t r = (int64_t)blockIdx.x * PLAN_ROWS + lane;
    const bool on = r < p.M;
    const W w = on ? plan_row_word<RK, W>(p, r) : W(0);
    plan_stage_rank<W>(p, s_rank);
    const int n = plan_expand<NW, W>(p, w, on, s_cnt, [&](int i, int g) {
        if (i < cap) s_grp[i * PLAN_ROWS + lane] = (uint16_t)g;
    });
    __syncthreads();
    // this wave's share of the diagonal's terms; added after the others, which are smaller
    double2 diag = make_double2(0.0, 0.0), acc = make_double2(0.0, 0.0);
    if (p.big >= 0) {
        const bool omega = wave == 0 && p.big == p.diag;
        bool any = omega;
        double2 v = plan_big<4, W>(p, wave, NW, w, any);
        if (omega) v = cadd(v, p.omega);
        if (any && on) diag = cmul(v, x[plan_col<CK, W>(p, w ^ p.groups[p.big].flip, s_rank)]);
    }
    for (int i = wave; i < n; i += NW) {
        const int gi = s_grp[i * PLAN_ROWS + lane];
        if (gi == p.big) continue;
        const PlanGroup<W> g = p.groups[gi];
        const double2 xv = x[plan_col<CK, W>(p, w ^ g.flip, s_rank)];
        double2 v = plan_sum<W>(p, g.tbeg, g.tend, w);
        if (gi == p.diag) v = cadd(v, p.omega);
        acc = cadd(acc, cmul(v, xv));
    }
    acc = cadd(acc, diag);
    s_acc[wave][lane] = acc;
    __syncthreads();
    if (wave != 0) return;
    double2 dot = make_double2(0, 0);
    if (on) {
        double2 part[NW];
#pragma unroll
        for (int q = 0; q < NW; ++q) part[q] = s_acc[q][lane];
#pragma unroll
        for (int h = NW / 2; h > 0; h /= 2)
#pragma unroll
            for (int q = 0; q < h; ++q) part[q] = cadd(part[q], part[q + h]);
        acc = part[0];
        double2 out = e.c0 ? cmul(*e.c0, acc) : acc;
        if (e.z) out = cadd(out, e.c1 ? cmul(*e.c1, e.z[r]) : e.z[r]);
        e.y[r] = out;
        if (e.dvec) dot = cconjmul(e.dvec[r], out);
    }
    if (e.dvec) {
        dot = wave_sum64(dot);
        if (lane == 0) e.partials[blockIdx.x] = dot;
    }
}

}  // namespace

struct edx_mfop {
    BuildParams p{};
    TermTable tt;
    MfMask *d_masks = nullptr;
    int corehole = 0;   // row/column layout: core-hole space (H_n) or plain (H_i)
    PlanStore<uint32_t> plan32;   // the one in use has terms grouped for k_plan_apply
    PlanStore<uint64_t> plan64;
    int plan = 0;       // its word bits, or 0: k_mf
    int maxrow = 0;     // longest row of the plan
    ~edx_mfop() { edx::dfree(d_masks); }
};

namespace {

// Waves per workgroup of k_plan_apply.  While the workgroups fill less than two
// a CU the time is one workgroup's own, and sixteen waves share its terms and
// entries: 26 us for 30 at 12,870 rows, 39.1 for 40.6 at 18,018; at 24,310 rows
// (380 workgroups) both take 32.5, at 48,620 sixteen waves 39.7 and four 34.6,
// at 705,432 347 and 202.
constexpr int MF_WIDE = 16;

int mf_waves(int64_t rows) {
    return (rows + PLAN_ROWS - 1) / PLAN_ROWS <= (int64_t)edx::num_cus() * 3 / 2 ? MF_WIDE : PLAN_WAVES;
}

// The most groups that T terms on M rows may have for the plan to be the faster product;
// negative: it is the slower one however they group.  A product's time beyond a launch, in
// us: the plan takes 0.05 a group and 3 (its waves test all groups, whatever the rows,
// while the workgroups fill the chip less than twice); k_mf, whose waves take a row each,
// 0.004 a term and, a row, 5e-4 and 2.2e-6 a term.  Measured (k_mf, plan): 370 terms in
// 46 groups 21.0 and 21.9 us on 2,002 rows, 23.4 and 22.2 on 3,432, 27.1 and 22.5 on 8,008; 965
// in 129, 24.2 and 24.5 on 1,320, 31.6 and 25.0 on 2,772, 53.2 and 25.7 on 10,296; 2,500 in
// 160, 27.7 and 37.6 on 120; random terms, 1000 in 500, 37.7 and 46.0 on 6,435, 58.1 and 47.6
// on 12,870.
double mf_max_groups(int64_t M, int T) {
    const double g = (M * (5e-4 + 2.2e-6 * T) + 0.004 * T - 3.0) / 0.05;
    return 16.0 * g < T ? -1.0 : g;
}

int mf_blocks(const edx_mfop *op) {
    if (op->plan) return (int)std::max<int64_t>((op->p.M + PLAN_ROWS - 1) / PLAN_ROWS, 1);
    int64_t b = op->p.M;
    const int64_t cap = (int64_t)edx::num_cus() * 256;
    if (b > cap) b = cap;
    return (int)std::max<int64_t>(b, 1);
}

int64_t mf_partials_len(const edx_mfop *op) { return mf_blocks(op) + FOLD_N + 64; }

template <int RK, int CK, class W>
void mf_launch_plan(const edx_mfop *op, const Plan<W> &p, int nb, const double2 *x,
                    const SpmvEpi &e) {
    const int cap = std::max(op->maxrow, 1);
    const size_t lds = (size_t)p.rank_len * 4 + (size_t)cap * PLAN_ROWS * 2;
    if (mf_waves(op->p.M) == MF_WIDE)
        hipLaunchKernelGGL((k_plan_apply<MF_WIDE, RK, CK, W>), dim3(nb), dim3(64 * MF_WIDE), lds,
                           edx::stream(), p, cap, x, e);
    else
        hipLaunchKernelGGL((k_plan_apply<PLAN_WAVES, RK, CK, W>), dim3(nb), dim3(64 * PLAN_WAVES), lds,
                           edx::stream(), p, cap, x, e);
}

// Groups the operator's terms where the basis allows; the longest row sizes
// the kernel's lists.
template <int RK, int CK, class W>
int mf_plan(edx_mfop *op, const PlanSpaces &sp, const PlanTerms &pt, PlanStore<W> &store) {
    EDX_TRY(plan_make<W>(sp, pt, op->p.omega_on != 0, op->p.omega, mf_waves(op->p.M), false, store));
    store.p.inter = 0;
    DevBuf flag;
    EDX_TRY(flag.alloc(sizeof(int), "longest row"));
    EDX_HIP(hipMemsetAsync(flag.p, 0, sizeof(int), edx::stream()));
    EDX_TRY((plan_count<RK, W>(store.p, nullptr, flag.as<int>())));
    EDX_HIP(edx::copy_sync(&op->maxrow, flag.p, sizeof(int), hipMemcpyDeviceToHost));
    if (op->maxrow <= 255) op->plan = 8 * (int)sizeof(W);
    return EDX_OK;
}

template <int RK, int CK> int mf_try_plan(edx_mfop *op, const edx_basis *fock) {
    const PlanSpaces sp{RK, CK, op->p.nv, op->p.nc, fock, fock};
    const double most = mf_max_groups(op->p.M, op->tt.T);
    PlanTerms pt;
    if (op->p.M == 0 || op->p.M >= ((int64_t)1 << 31) || most < 0.0 ||
        !plan_usable(sp, op->tt.ops.data(), op->tt.nhop, op->tt.T) ||
        !plan_group(sp, op->tt.ops.data(), op->tt.vals.data(), op->tt.nhop, op->tt.T,
                    op->p.omega_on != 0, op->p.negate != 0, true, most, pt))
        return EDX_OK;
    return plan_bits(sp) <= 32 ? mf_plan<RK, CK, uint32_t>(op, sp, pt, op->plan32)
                               : mf_plan<RK, CK, uint64_t>(op, sp, pt, op->plan64);
}

int mf_launch(const edx_mfop *op, const double2 *x, const SpmvEpi &e, int *nblocks_out) {
    const int nb = mf_blocks(op);
    if (nblocks_out) *nblocks_out = nb;
    if (op->p.M == 0) return EDX_OK;
    if (op->plan == 32 && op->corehole)
        mf_launch_plan<ROW_COREHOLE, COL_COREHOLE>(op, op->plan32.p, nb, x, e);
    else if (op->plan == 32)
        mf_launch_plan<ROW_PLAIN, COL_PLAIN>(op, op->plan32.p, nb, x, e);
    else if (op->plan == 64 && op->corehole)
        mf_launch_plan<ROW_COREHOLE, COL_COREHOLE>(op, op->plan64.p, nb, x, e);
    else if (op->plan == 64)
        mf_launch_plan<ROW_PLAIN, COL_PLAIN>(op, op->plan64.p, nb, x, e);
    else if (op->corehole)
        hipLaunchKernelGGL((k_mf<ROW_COREHOLE, COL_COREHOLE>), dim3(nb), dim3(64), 0,
                           edx::stream(), op->p, op->d_masks, x, e);
    else
        hipLaunchKernelGGL((k_mf<ROW_PLAIN, COL_PLAIN>), dim3(nb), dim3(64), 0, edx::stream(),
                           op->p, op->d_masks, x, e);
    EDX_LAUNCH_CHECK();
    if (e.dvec && nb > FOLD_N) {
        hipLaunchKernelGGL(k_fold_partials, dim3(FOLD_N), dim3(256), 0, edx::stream(), e.partials,
                           nb, e.run);
        hipLaunchKernelGGL(k_move_folded, dim3(1), dim3(FOLD_N), 0, edx::stream(), e.partials, nb,
                           e.run);
        EDX_LAUNCH_CHECK();
        if (nblocks_out) *nblocks_out = FOLD_N;
    }
    return EDX_OK;
}

int mf_make(const edx_tensor2 *hop, int64_t nhopp, const edx_tensor4 *coul, int64_t ncoul,
            double omega_re, double omega_im, double ham_sign, edx_mfop **out, edx_mfop **op) {
    EDX_CHECK(out, EDX_ERR_ARG, "null output");
    *out = nullptr;
    EDX_TRY(check_ham_sign(ham_sign));
    EDX_TRY(edx::ensure_binomials());
    edx_mfop *o = new edx_mfop;
    int rc = parse_terms(hop, nhopp, coul, ncoul, o->tt);
    if (!rc) rc = upload_terms(o->tt);
    if (rc) {
        delete o;
        return rc;
    }
    o->p = base_params(o->tt);
    o->p.ops = o->tt.d_ops;
    o->p.tv = o->tt.d_vals;
    const int T = o->tt.T;
    o->d_masks = (MfMask *)edx::dmalloc((size_t)(T ? T : 1) * sizeof(MfMask), "term masks");
    if (!o->d_masks) {
        delete o;
        return EDX_ERR_NOMEM;
    }
    if (T) {
        hipLaunchKernelGGL(k_mf_masks, dim3((T + 255) / 256), dim3(256), 0, edx::stream(),
                           o->tt.d_ops, T, o->tt.nhop, o->d_masks);
        if (hipGetLastError() != hipSuccess) {
            delete o;
            return edx::set_error(EDX_ERR_HIP, "term mask launch failed");
        }
    }
    o->p.omega_on = ham_sign < 0;
    o->p.omega = make_double2(omega_re, omega_im);
    o->p.negate = ham_sign < 0;
    *op = o;
    return EDX_OK;
}

}  // namespace

extern "C" {

int edx_mf_ham_i(const edx_basis *fock, const edx_tensor2 *hop, int64_t nhopp,
                 const edx_tensor4 *coul, int64_t ncoul, double omega_re, double omega_im,
                 double ham_sign, edx_mfop **out) {
    EDX_CHECK(fock, EDX_ERR_ARG, "null basis");
    edx_mfop *o = nullptr;
    EDX_TRY(mf_make(hop, nhopp, coul, ncoul, omega_re, omega_im, ham_sign, out, &o));
    o->p.M = fock->n;
    o->p.left = fock->d_words;
    o->p.nleft = fock->n;
    o->p.right = view_of(fock);
    o->corehole = 0;
    const int rc = mf_try_plan<ROW_PLAIN, COL_PLAIN>(o, fock);
    if (rc) {
        delete o;
        return rc;
    }
    *out = o;
    return EDX_OK;
}

int edx_mf_ham_n(const edx_basis *fock_n, int num_val_orbs, int num_core_orbs,
                 const edx_tensor2 *hop, int64_t nhopp, const edx_tensor4 *coul, int64_t ncoul,
                 double omega_re, double omega_im, double ham_sign, edx_mfop **out) {
    EDX_CHECK(fock_n, EDX_ERR_ARG, "null basis");
    EDX_TRY(check_core(num_val_orbs, num_core_orbs));
    edx_mfop *o = nullptr;
    EDX_TRY(mf_make(hop, nhopp, coul, ncoul, omega_re, omega_im, ham_sign, out, &o));
    o->p.M = fock_n->n * num_core_orbs;
    o->p.left = fock_n->d_words;
    o->p.nleft = fock_n->n;
    o->p.right = view_of(fock_n);
    o->p.nv = num_val_orbs;
    o->p.nc = num_core_orbs;
    o->corehole = 1;
    const int rc = mf_try_plan<ROW_COREHOLE, COL_COREHOLE>(o, fock_n);
    if (rc) {
        delete o;
        return rc;
    }
    *out = o;
    return EDX_OK;
}

int edx_mf_size(const edx_mfop *op, int64_t *n) {
    EDX_CHECK(op && n, EDX_ERR_ARG, "null argument");
    *n = op->p.M;
    return EDX_OK;
}

int edx_mf_apply(const edx_mfop *op, const void *d_x, void *d_y) {
    EDX_CHECK(op && d_x && d_y, EDX_ERR_ARG, "null argument");
    SpmvEpi e{};
    e.y = (double2 *)d_y;
    e.z = (const double2 *)d_y;   // y += H x
    hipEvent_t pe = edx::prof_start(EDX_C128, EDX_KERNEL_MF, edx::mf_bytes(op->p.M, op->p.M));
    EDX_TRY(mf_launch(op, (const double2 *)d_x, e, nullptr));
    edx::prof_stop(pe);
    EDX_HIP(hipStreamSynchronize(edx::stream()));
    return EDX_OK;
}

int edx_build_krylov_mf(const edx_mfop *op, const void *d_v0, int maxn, int *neff, double *alpha,
                        double *beta, double *norm) {
    EDX_CHECK(op && d_v0 && neff && alpha && beta && norm && maxn >= 1, EDX_ERR_ARG,
              "bad argument");
    auto prod = [&](const double2 *x, const SpmvEpi &e, int *nb, const int *run) {
        (void)run;
        hipEvent_t pe = edx::prof_start(EDX_C128, EDX_KERNEL_MF, edx::mf_bytes(op->p.M, op->p.M));
        int rc = mf_launch(op, x, e, nb);
        edx::prof_stop(pe);
        return rc;
    };
    int rc = krylov_loop(op->p.M, prod, mf_partials_len(op), (const double2 *)d_v0, maxn, neff,
                         alpha, beta, norm);
    if (rc) return rc;
    EDX_HIP(hipStreamSynchronize(edx::stream()));
    return EDX_OK;
}

void edx_mf_free(edx_mfop *op) { delete op; }

}  // extern "C"
