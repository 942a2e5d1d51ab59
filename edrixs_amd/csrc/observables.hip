// Density matrix and continued-fraction spectra (part of edx_kernels.hip).
//
//   edx_denmat       <- src/ed_driver.f90:219-248
//   edx_cf_spectrum  <- edrixs/plot_spectrum.py:52-59 (twin: src/lanczos.f90:306-336)

namespace {

// One block per (i <= j) orbital pair and row chunk; partial sums per block are
// reduced in a fixed order afterwards.
__global__ __launch_bounds__(256) void k_denmat_pairs(BasisView b, int norb, const double2 *v,
                                                      const int2 *pairs, int nchunk,
                                                      double2 *partials) {
    const int pid = blockIdx.x;
    const int i = pairs[pid].x, j = pairs[pid].y;
    const int64_t chunk = (b.n + nchunk - 1) / nchunk;
    const int64_t lo = blockIdx.y * chunk;
    const int64_t hi = lo + chunk < b.n ? lo + chunk : b.n;
    double2 sij = make_double2(0, 0), sji = make_double2(0, 0);
    for (int64_t r = lo + threadIdx.x; r < hi; r += 256) {
        const uint64_t w = (uint64_t)b.words[r];
        const double2 vr = v[r];
        if (i == j) {
            if ((w >> j) & 1ull) sij = cadd(sij, cconjmul(vr, vr));
            continue;
        }
        if (hypot(vr.x, vr.y) < 1e-10) continue;   // src/ed_driver.f90:226
        if (!((w >> i) & 1ull)) continue;
        int par = __popcll(w & ((1ull << i) - 1ull));
        uint64_t m = w ^ (1ull << i);
        if ((m >> j) & 1ull) continue;
        par += __popcll(m & ((1ull << j) - 1ull));
        m |= (1ull << j);
        const int64_t c = basis_index(b, m);
        if (c < 0) continue;
        const double sg = (par & 1) ? -1.0 : 1.0;
        const double2 vc = v[c];
        sij = cadd(sij, cscale(cconjmul(vr, vc), sg));
        sji = cadd(sji, cscale(cconjmul(vc, vr), sg));
    }
    double2 a = block_sum_256(sij);
    double2 c2 = block_sum_256(sji);
    if (threadIdx.x == 0) {
        partials[((int64_t)pid * gridDim.y + blockIdx.y) * 2] = a;
        partials[((int64_t)pid * gridDim.y + blockIdx.y) * 2 + 1] = c2;
    }
}

// The fraction without its divisions.  With D_n = 1, D_{n+1} = 0 and
//     D_j = (z - a_{j+1}) D_{j+1} - b_{j+1}^2 D_{j+2}        (j = n-1 .. 0)
// (the determinants of the trailing blocks of z - T) the fraction is D_1 / D_0.
// A step is two dependent multiply-adds where the nested form waits for a complex
// quotient, and that serial chain is all there is: 300 poles on 2000 points
// took 62 us nested (the whole call 154 us, now 42).  The phases of D_1 and D_0
// gather a rounding a step, so far from the poles, where the fraction is almost
// real, the imaginary part of their quotient is a difference of nearly equal
// products (300 poles, 45 to 85 eV from the middle of a band 60 eV wide, broadening
// 0.1 eV: off by 6e-14 of itself, nested 4e-16).  It is taken there from
// P_j = Im(D_{j+1} conj(D_j)),
//     P_j = b_{j+1}^2 P_{j+1} - gamma |D_{j+1}|^2,
// a sum of terms of one sign, as P_0 / |D_0|^2 (4e-16 too).  Where the imaginary
// part is at least half the real one the quotient loses nothing and is the closer of
// the two (broadening 0.5 eV inside the band: 3.4e-16, nested 3.6e-16, P 5.1e-16).
// D, its predecessor and P are rescaled by powers of two every CF_BLOCK steps.
// Between two rescalings nothing overflows while |a|, b, |gamma| and |e_gs| are below
// CF_MAX and |z| below twice that (|D| grows by at most 2^53 a step), and nothing that
// counts underflows while |gamma| is above 1 / CF_MAX: Im(D_{j+2} / D_{j+1}) has the
// sign that makes |D_j| >= |gamma| |D_{j+1}|, whatever a and b.  Grid points outside
// that take the nested form, all of them (nested) if a coefficient is outside.  The
// coefficients are staged in LDS, one grid point per lane.
constexpr int CF_BLOCK = 8;
constexpr int CF_STAGE = 512;
constexpr double CF_MAX = 1125899906842624.0;   // 2^50

// a / b with the squares of b in range (the same bits as cdiv where they are anyway)
__device__ __forceinline__ double2 cdiv_scaled(double2 a, double2 b) {
    const double m = fmax(fabs(b.x), fabs(b.y));
    if (!(m > 0.0 && m < __builtin_inf())) return cdiv(a, b);
    const int e = ilogb(m);
    const double s = ldexp(1.0, e > -1000 ? -e : 1000);
    return cdiv(cscale(a, s), cscale(b, s));
}

__global__ __launch_bounds__(64) void k_cf(int neff, const double *__restrict__ alpha,
                                           const double *__restrict__ beta, double norm, double e_gs,
                                           double weight, int nw, const double *__restrict__ omega,
                                           const double *__restrict__ gamma, const double *spec,
                                           double *out, int nested) {
    __shared__ double s_a[CF_STAGE], s_b2[CF_STAGE];
    const int w = blockIdx.x * 64 + threadIdx.x;
    const bool on = w < nw;
    const double zx = on ? omega[w] + e_gs : 0.0, zy = on ? gamma[w] : 1.0;
    // a_{j+1} and the b^2 that follows it, j = neff-1 .. 0, a stage of n at a time
    auto sweep = [&](auto take) {
        for (int top = neff; top > 0; top -= CF_STAGE) {
            const int n = top < CF_STAGE ? top : CF_STAGE;
            __syncthreads();
            for (int i = threadIdx.x; i < n; i += 64) {
                const int j = top - 1 - i;
                const double b = j + 1 < neff ? beta[j] : 0.0;
                s_a[i] = alpha[j];
                s_b2[i] = b * b;
            }
            __syncthreads();
            take(n);
        }
    };
    double im = 0.0;
    if (!nested) {
        double2 d = make_double2(1.0, 0.0), q = make_double2(0.0, 0.0);   // D_{j+1}, D_{j+2}
        double p = 0.0;                                                   // P_{j+1}
        auto step = [&](int i) {
            const double x = zx - s_a[i], b2 = s_b2[i];
            const double2 t = make_double2(x * d.x - (zy * d.y + b2 * q.x),
                                           x * d.y + (zy * d.x - b2 * q.y));
            p = b2 * p - zy * (d.x * d.x + d.y * d.y);
            q = d;
            d = t;
        };
        sweep([&](int n) {
            int i = 0;
            for (; i + CF_BLOCK <= n; i += CF_BLOCK) {
#pragma unroll
                for (int u = 0; u < CF_BLOCK; ++u) step(i + u);
                const double big = fmax(fmax(fabs(d.x), fabs(d.y)), fmax(fabs(q.x), fabs(q.y)));
                const double sc = ldexp(1.0, -ilogb(big));
                d = cscale(d, sc);
                q = cscale(q, sc);
                p *= sc * sc;
            }
            for (; i < n; ++i) step(i);
        });
        const double2 t = cdiv(q, d);
        im = fabs(t.y) >= 0.5 * fabs(t.x) ? t.y : p / (d.x * d.x + d.y * d.y);
    }
    const bool out_of_range = nested || !(fabs(zx) < 2.0 * CF_MAX && fabs(zy) < CF_MAX &&
                                          fabs(zy) > 1.0 / CF_MAX);
    if (__any(on && out_of_range)) {
        double2 t = make_double2(1.0, 0.0);
        sweep([&](int n) {
            for (int i = 0; i < n; ++i)
                t = csub(make_double2(zx - s_a[i], zy), cdiv_scaled(make_double2(s_b2[i], 0.0), t));
        });
        if (out_of_range) im = cdiv_scaled(make_double2(1.0, 0.0), t).y;
    }
    if (on) out[w] = spec[w] + -1.0 / 3.14159265358979323846 * im * norm * weight;
}

// Whether the division-free recurrence serves these coefficients (k_cf looks at the
// grid points).
bool cf_in_range(int neff, const double *alpha, const double *beta, double e_gs) {
    bool in = fabs(e_gs) < CF_MAX;
    for (int i = 0; i < neff; ++i) in = in && fabs(alpha[i]) < CF_MAX;
    for (int i = 0; i + 1 < neff; ++i) in = in && fabs(beta[i]) < CF_MAX;
    return in;
}

// Page-locked staging of a thread's small transfers, allocated at its first
// call and released with the thread.
struct PinnedStage {
    static constexpr size_t BYTES = 1 << 20;
    void *p = nullptr;
    bool tried = false;
    void *get(size_t bytes) {
        if (bytes > BYTES) return nullptr;
        if (!tried) {
            tried = true;
            if (hipHostMalloc(&p, BYTES, hipHostMallocPortable) != hipSuccess) {
                (void)hipGetLastError();
                p = nullptr;
            }
        }
        return p;
    }
    ~PinnedStage() {
        if (p) (void)hipHostFree(p);
    }
};
thread_local PinnedStage g_stage;

}  // namespace

extern "C" {

int edx_denmat(const edx_basis *fock, int num_val_orbs, const void *d_vec, double *denmat) {
    EDX_CHECK(fock && d_vec && denmat && num_val_orbs >= 1 && num_val_orbs <= 63, EDX_ERR_ARG,
              "bad argument");
    EDX_TRY(edx::ensure_binomials());
    const int no = num_val_orbs;
    std::vector<int2> pairs;
    for (int i = 0; i < no; ++i)
        for (int j = i; j < no; ++j) pairs.push_back(make_int2(i, j));
    const int np = (int)pairs.size();
    int nchunk = (int)std::min<int64_t>(64, std::max<int64_t>(1, fock->n / 4096));
    DevBuf dp, part;
    EDX_TRY(dp.alloc(np * sizeof(int2), "pairs"));
    EDX_TRY(part.alloc((size_t)np * nchunk * 2 * sizeof(double2), "denmat partials"));
    EDX_HIP(edx::copy_sync(dp.p, pairs.data(), np * sizeof(int2), hipMemcpyHostToDevice));
    hipLaunchKernelGGL(k_denmat_pairs, dim3(np, nchunk), dim3(256), 0, edx::stream(), view_of(fock),
                       no, (const double2 *)d_vec, dp.as<int2>(), nchunk, part.as<double2>());
    EDX_LAUNCH_CHECK();
    std::vector<double2> hp((size_t)np * nchunk * 2);
    EDX_HIP(edx::copy_sync(hp.data(), part.p, hp.size() * sizeof(double2), hipMemcpyDeviceToHost));
    double *dm = denmat;
    std::memset(dm, 0, sizeof(double) * 2 * no * no);
    for (int p = 0; p < np; ++p) {
        double2 a = make_double2(0, 0), c = make_double2(0, 0);
        for (int k = 0; k < nchunk; ++k) {
            a.x += hp[((size_t)p * nchunk + k) * 2].x;
            a.y += hp[((size_t)p * nchunk + k) * 2].y;
            c.x += hp[((size_t)p * nchunk + k) * 2 + 1].x;
            c.y += hp[((size_t)p * nchunk + k) * 2 + 1].y;
        }
        const int i = pairs[p].x, j = pairs[p].y;
        dm[2 * (i * no + j)] += a.x;
        dm[2 * (i * no + j) + 1] += a.y;
        if (i != j) {
            dm[2 * (j * no + i)] += c.x;
            dm[2 * (j * no + i) + 1] += c.y;
        }
    }
    return EDX_OK;
}

int edx_cf_spectrum(int neff, const double *alpha, const double *beta, double norm, double e_gs,
                    double weight, int nw, const double *omega, const double *gamma, double *spec) {
    EDX_CHECK(neff >= 1 && nw >= 0 && alpha && beta && (nw == 0 || (omega && gamma && spec)),
              EDX_ERR_ARG, "bad argument");
    if (nw == 0) return EDX_OK;
    // The inputs lie side by side in page-locked memory where they fit, and the
    // kernel writes its result there.  Where the workgroups together read at most
    // CF_DIRECT bytes of coefficients it reads the inputs there too: one launch
    // and one wait (a transfer each way costs another 10 us; 300 poles on 2000
    // points read 150 KB, 3 us over the bus).  Larger inputs are copied first, those
    // larger than the staging memory from where they are (100 poles on a million
    // points: another copy on the host took 1.5 of 3.9 ms).
    constexpr size_t CF_DIRECT = 256 << 10;
    const int nb = (nw + 63) / 64;
    const size_t count = 2 * (size_t)neff + 4 * (size_t)nw, bytes = sizeof(double) * count;
    const size_t o_om = 2 * (size_t)neff, o_sp = o_om + 2 * (size_t)nw, o_out = o_sp + nw;
    double *host = (double *)g_stage.get(bytes);
    const bool direct = host && (size_t)nb * neff * 16 <= CF_DIRECT;
    DevBuf buf;
    double *d = host;
    hipStream_t s = edx::stream();
    if (!direct) {
        EDX_TRY(buf.alloc(bytes, "cf buffers"));
        d = buf.as<double>();
    }
    const struct {
        size_t at;
        const double *from;
        int n;
    } in[] = {{0, alpha, neff}, {(size_t)neff, beta, neff}, {o_om, omega, nw},
              {o_om + nw, gamma, nw}, {o_sp, spec, nw}};
    for (const auto &q : in) {
        if (host) memcpy(host + q.at, q.from, q.n * sizeof(double));
        else EDX_HIP(hipMemcpyAsync(d + q.at, q.from, q.n * sizeof(double), hipMemcpyHostToDevice, s));
    }
    if (host && !direct) EDX_HIP(hipMemcpyAsync(d, host, o_out * sizeof(double), hipMemcpyHostToDevice, s));
    double *out = host ? host + o_out : d + o_out;
    hipLaunchKernelGGL(k_cf, dim3(nb), dim3(64), 0, s, neff, d, d + neff, norm, e_gs, weight, nw,
                       d + o_om, d + o_om + nw, d + o_sp, out, !cf_in_range(neff, alpha, beta, e_gs));
    EDX_LAUNCH_CHECK();
    if (!host) {
        EDX_HIP(edx::copy_sync(spec, out, nw * sizeof(double), hipMemcpyDeviceToHost));
        return EDX_OK;
    }
    EDX_HIP(hipStreamSynchronize(s));
    memcpy(spec, host + o_out, nw * sizeof(double));
    return EDX_OK;
}

}  // extern "C"
