// Term plans: the terms of an operator grouped by the column they lead to
// (part of edx_kernels.hip).  Used by the CSR builds and the matrix-free apply.
//
// Every term is a string of annihilations and creations applied to a row's
// word w (the order of src/ham.f90: ind1 [, ind2] out, then the others in).
// Whether it survives, where it leads and its fermion sign are closed forms of
// w (Jordan-Wigner strings of fixed positions):
//     survives   (w & M) == V      every operator's orbital is filled / empty
//     column     w ^ F             F = the orbitals the string flips
//     sign       (-1)^(popc(w & S) + c)
// where S is the XOR of the "orbitals below" masks of the operators and c the
// constant part of the flips made on the way.  Terms with the same F reach the
// same column from any row, so a row has at most one entry per distinct F: the
// terms (a thousand for an impurity with a core shell) collapse into groups (a
// hundred or two), most of them of two to six terms.  Only the column-deciding
// part of F counts for operators whose columns ignore the core word
// (src/ham.f90:806-808).
//
// For a complete basis on both sides a term either keeps the particle numbers
// the column space asks for or never reaches it, whatever the row, so columns
// need no membership test.  Incomplete bases keep the term-by-term build.

namespace {

enum { ROW_PLAIN = 0, ROW_COREHOLE = 1, ROW_FULLCORE = 2 };
enum { COL_PLAIN = 0, COL_COREHOLE = 1, COL_VALONLY = 2 };

// the words of a plan: 32 bits where valence and core orbitals fit, else 64
template <class W> struct PlanTest {   // two survival tests; bit: the group's in its chunk
    W m[2], v[2];
    uint32_t bit, pad;
};
template <class W> struct PlanDens {   // a term of the big group whose sign is constant
    W m, v;
    double x;
};
template <class W> struct PlanTerm {
    W m, v, s;
    uint32_t neg;     // bit 0: c, and the operator's overall sign; PLAN_FLIP_X, _Y
};
// The sign applies to the real / imaginary part; clear on a part of merged
// terms that is +0 whatever their sign.
constexpr uint32_t PLAN_FLIP_X = 1u << 30, PLAN_FLIP_Y = 1u << 31;
template <class W> struct PlanGroup {
    W flip;
    int32_t tbeg, tend;   // its terms, in term order
    int32_t pad;
};

constexpr int PLAN_ROWS = 64;        // rows per workgroup: lane = row
constexpr int PLAN_WAVES = 4;        // waves share the groups (chunks) of the same rows
constexpr int RANK_BITS = 4;         // bits per lookup of a column's rank
constexpr int RANK_UNROLL = 24 / RANK_BITS;   // lookups without a test
constexpr int RANK_MAX = (64 + RANK_BITS - 1) / RANK_BITS;
constexpr int PLAN_CHUNK = 32;       // groups per chunk (bits of a survival mask)
constexpr int PLAN_MAX_TERMS = 4096; // the term-by-term build's limit per row
constexpr int PLAN_SMALL_ROW = 64;   // longest row of the fill's compact lists
constexpr int FILL_U = 2;            // entries a thread of the fill has in flight
constexpr int PLAN_BIG = 24;         // a group of more terms (the diagonal) is summed per row

// A plan on the device, with what its kernels need to know of the spaces.
template <class W> struct Plan {
    const PlanTest<W> *tests;
    const int32_t *chunks;           // nchunk + 1 offsets into tests
    const PlanTerm<W> *terms;
    const double2 *vals;             // value of each term, the sign not applied
    const PlanGroup<W> *groups;
    const int32_t *rank;             // rank tables (plan_rank)
    int rank_len, nrank;             // their length, lookups per word
    int rank_off[RANK_MAX];
    int ngroups;
    int nchunk, gpc;                 // chunks (a multiple of the kernel's waves), groups per chunk
    int big;                         // group summed lane = row, or -1
    const PlanDens<W> *dens;         // its terms if all have constant signs and the same
    int ndens;                       // zero imaginary part, else none
    double dens_y;                   // that zero, signed
    int diag;                        // group of the diagonal when omega is added, or -1
    double2 omega;
    int64_t M;                       // rows
    const int64_t *left;             // valence words of the row space
    int64_t nleft;
    int nv, nc, nbits, nocc;         // nbits, nocc: the column basis
    int64_t nright;                  // its size
    int inter;                       // core-hole index valence * nc + slot
};

template <class W> __device__ __forceinline__ int plan_popc(W x) {
    if constexpr (sizeof(W) == 4) return __popc(x);
    else return __popcll(x);
}

template <int RK, class W>
__device__ __forceinline__ W plan_row_word(const Plan<W> &p, int64_t row) {
    const uint32_t r = (uint32_t)row;          // dimensions are below 2^31
    if (RK == ROW_PLAIN) return (W)p.left[r];
    const W full = (W)((W(1) << p.nc) - 1);
    if (RK == ROW_FULLCORE) return (W)((full << p.nv) | (W)p.left[r]);
    const uint32_t nl = (uint32_t)p.nleft, nc = (uint32_t)p.nc;
    const uint32_t v = p.inter ? r / nc : r % nl, k = p.inter ? r - v * nc : r / nl;
    return (W)(((full ^ (W(1) << (p.nc - 1 - k))) << p.nv) | (W)p.left[v]);   // src/ham.f90:419-421
}

// Order key of a column: ascending keys are ascending columns.
template <int CK, class W>
__device__ __forceinline__ W plan_key(const Plan<W> &p, W w) {
    if (CK == COL_PLAIN) return w;
    const W val = w & (W)((W(1) << p.nv) - 1);
    if (CK == COL_VALONLY) return val;
    return p.inter ? (W)((val << p.nc) | (w >> p.nv)) : w;
}

// Rank of a word of the column basis: sum of C(q_k, k + 1) over its orbitals
// q_0 < q_1 < ...  RANK_BITS of the word and the number of orbitals below them
// index a table (staged in LDS): six independent lookups for 24 orbitals, where a
// walk over the orbitals takes twelve dependent steps.  Six-bit tables (7 KB
// instead of 3) take a workgroup per CU: the fill below 1.14 for 1.05 ms.
template <class W>
__device__ __forceinline__ int32_t plan_rank(const Plan<W> &p, W val, const int32_t *s_rank) {
    constexpr uint32_t mask = (1u << RANK_BITS) - 1;
    int32_t l = 0;
    uint32_t k = 0;
#pragma unroll
    for (int j = 0; j < RANK_UNROLL; ++j) {   // past the last orbital: a zero entry
        const uint32_t c = (uint32_t)(val >> (RANK_BITS * j)) & mask;
        l += s_rank[p.rank_off[j] + (int)((k << RANK_BITS) | c)];
        k += __popc(c);
    }
    for (int j = RANK_UNROLL; j < p.nrank; ++j) {
        const uint32_t c = (uint32_t)(val >> (RANK_BITS * j)) & mask;
        l += s_rank[p.rank_off[j] + (int)((k << RANK_BITS) | c)];
        k += __popc(c);
    }
    return l;
}

// Column of a word.
template <int CK, class W>
__device__ __forceinline__ int32_t plan_col(const Plan<W> &p, W w, const int32_t *s_rank) {
    const W val = CK == COL_PLAIN ? w : w & (W)((W(1) << p.nv) - 1);
    const int32_t l = plan_rank<W>(p, val, s_rank);
    if (CK != COL_COREHOLE) return l;
    const W holes = (W)(((W(1) << p.nc) - 1) ^ (w >> p.nv));
    const int k = p.nc - 1 - ((sizeof(W) == 4 ? __ffs((unsigned)holes)
                                              : __ffsll((unsigned long long)holes)) - 1);
    return p.inter ? l * p.nc + k : (int32_t)(k * p.nright) + l;
}

template <class W>
__device__ __forceinline__ void plan_stage_rank(const Plan<W> &p, int32_t *s_rank) {
    const int4 *from = reinterpret_cast<const int4 *>(p.rank);
    int4 *to = reinterpret_cast<int4 *>(s_rank);
    for (int i = threadIdx.x; i < p.rank_len / 4; i += blockDim.x) to[i] = from[i];
}

// Which groups of chunk c have a surviving term on word w.  Chunk, test and
// group numbers are uniform over the wave, so the tests come by scalar loads
// and each costs two vector instructions for 64 rows.
template <class W>
__device__ __forceinline__ uint32_t plan_mask(const Plan<W> &p, int c, W w) {
    const int ib = p.chunks[c], ie = p.chunks[c + 1];
    uint32_t mask = 0;
#pragma unroll 2
    for (int i = ib; i < ie; ++i) {
        const PlanTest<W> &t = p.tests[i];
        const bool ok = ((w & t.m[0]) == t.v[0]) | ((w & t.m[1]) == t.v[1]);
        mask |= ok ? t.bit : 0u;
    }
    return mask;
}

__device__ __forceinline__ double plan_flip(double v, uint32_t sign) {
    return __hiloint2double(__double2hiint(v) ^ (int)sign, __double2loint(v));
}

template <class W>
__device__ __forceinline__ void plan_add_term(const PlanTerm<W> &t, double2 v, W w, double2 &acc) {
    if ((w & t.m) == t.v) {
        const uint32_t flip = (uint32_t)(plan_popc<W>(w & t.s) ^ t.neg) << 31;
        acc.x += plan_flip(v.x, flip & (t.neg << 1));
        acc.y += plan_flip(v.y, flip & t.neg);
    }
}

// Sum of a group's surviving terms in term order.  -0.0 + v is v bit for bit,
// so the sum is the reference's, which starts from the first survivor.
template <class W>
__device__ __forceinline__ double2 plan_sum(const Plan<W> &p, int tb, int te, W w) {
    double2 acc = make_double2(-0.0, -0.0);
#pragma unroll 2
    for (int t = tb; t < te; ++t) plan_add_term<W>(p.terms[t], p.vals[t], w, acc);
    return acc;
}

// Sum of terms first, first + step, ... of the big group; any: one survives.  SUMS: running
// sums of the density terms; 1 keeps the term order, 4 round less (the rounding of a
// hundred terms of one sign added one by one is the largest of a row's).
template <int SUMS, class W>
__device__ __forceinline__ double2 plan_big(const Plan<W> &p, int first, int step, W w, bool &any) {
    const PlanGroup<W> g = p.groups[p.big];
    if (p.ndens) {
        double acc[SUMS];
#pragma unroll
        for (int u = 0; u < SUMS; ++u) acc[u] = -0.0;
        auto take = [&](int t, double &a) {
            const PlanDens<W> d = p.dens[t];
            const bool ok = (w & d.m) == d.v;
            any |= ok;
            a += ok ? d.x : -0.0;
        };
        int t = first;
        if constexpr (SUMS == 1) {
#pragma unroll 4
            for (; t < p.ndens; t += step) take(t, acc[0]);
        } else {
            for (; t + (SUMS - 1) * step < p.ndens; t += SUMS * step)
#pragma unroll
                for (int u = 0; u < SUMS; ++u) take(t + u * step, acc[u]);
            for (; t < p.ndens; t += step) take(t, acc[0]);
#pragma unroll
            for (int h = SUMS / 2; h > 0; h /= 2)
#pragma unroll
                for (int u = 0; u < h; ++u) acc[u] += acc[u + h];
        }
        return make_double2(acc[0], any ? p.dens_y : -0.0);   // -0.0 + omega is omega bit for bit
    }
    double2 acc = make_double2(-0.0, -0.0);
#pragma unroll 2
    for (int t = g.tbeg + first; t < g.tend; t += step) {
        const PlanTerm<W> &tm = p.terms[t];
        any |= (w & tm.m) == tm.v;
        plan_add_term<W>(tm, p.vals[t], w, acc);
    }
    return acc;
}

__device__ __forceinline__ int plan_wave() {
    return __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
}

// Entries per row: the number of groups with a survivor.  maxrow gets the
// longest row.
template <int RK, class W>
__global__ __launch_bounds__(256) void k_plan_count(Plan<W> p, int64_t *counts, int *maxrow) {
    __shared__ int s_cnt[PLAN_WAVES][PLAN_ROWS];
    const int lane = threadIdx.x & 63, wave = plan_wave();
    const int64_t r = (int64_t)blockIdx.x * PLAN_ROWS + lane;
    const W w = r < p.M ? plan_row_word<RK, W>(p, r) : W(0);
    int n = 0;
    for (int c = wave; c < p.nchunk; c += PLAN_WAVES) n += __popc(plan_mask<W>(p, c, w));
    s_cnt[wave][lane] = n;
    __syncthreads();
    if (wave == 0) {
        n = 0;
        if (r < p.M) {
            for (int q = 0; q < PLAN_WAVES; ++q) n += s_cnt[q][lane];
            if (counts) counts[r] = n;
        }
        for (int off = 32; off > 0; off >>= 1) n = max(n, __shfl_xor(n, off, 64));
        // a stale read only costs an atomic that changes nothing
        if (lane == 0 && n > *(volatile int *)maxrow) atomicMax(maxrow, n);
    }
}

// Lists the row's surviving groups: entry e of row `lane` at list[e * 64 +
// lane] by emit(e, group), groups in plan order; returns the row's count.
// Every thread of the workgroup of NW waves calls it (barriers inside).
template <int NW, class W, class Emit>
__device__ __forceinline__ int plan_expand(const Plan<W> &p, W w, bool on, int (*s_cnt)[PLAN_ROWS],
                                           Emit emit) {
    const int lane = threadIdx.x & 63, wave = plan_wave();
    int n = 0;
    for (int c0 = 0; c0 < p.nchunk; c0 += NW) {
        const int c = c0 + wave;
        uint32_t mask = on ? plan_mask<W>(p, c, w) : 0u;
        __syncthreads();
        s_cnt[wave][lane] = __popc(mask);
        __syncthreads();
        int e = n;
        for (int q = 0; q < NW; ++q) {
            const int k = s_cnt[q][lane];
            if (q < wave) e += k;
            n += k;
        }
        while (mask) {
            emit(e++, c * p.gpc + __ffs((int)mask) - 1);
            mask &= mask - 1;
        }
    }
    return n;
}

// Fills the rows' columns and values.  A workgroup of four waves owns 64
// consecutive rows.  (1) lane = row: each wave finds the surviving groups of
// its chunks and lists (column key, group) per row in LDS; one wave sums the
// diagonal group, whose hundreds of density terms are the same for every lane.
// (2) lane = row: an entry's place in its row is the number of smaller keys.
// (3) lane = entry, in output order: sums its group's few terms, ranks its
// column and stores, so a wave writes 64 consecutive columns and values.
// LDS decides the workgroups per CU and with them the speed: lists of at most 64
// entries a row over at most 256 groups (SMALL) take 5 bytes an entry (32-bit
// words), the places in output order lying over the keys, and leave room for
// eight workgroups; other lists take 8.  The time goes to the integer
// instructions of (1) and (3) and their dependent loads, the 20 bytes per entry
// are written behind them.  Measured, count and fill: H_i norb 24 (2.7M rows,
// 44M entries) 0.08 + 0.74 ms (1.2 TB/s written; 8-byte lists 0.80), by the
// term-by-term kernel 16.1 + 21.4 ms; H_n norb 21 N 9 (2.1M rows, 50M entries)
// 0.11 + 1.05 ms (8-byte lists 1.48), before 27.9 + 36.9 ms.
template <bool SMALL, int RK, int CK, class W>
__global__ __launch_bounds__(256) void k_plan_fill(Plan<W> p, int cap,
                                                   const int64_t *__restrict__ rowptr,
                                                   int32_t *__restrict__ cols,
                                                   double2 *__restrict__ vals) {
    using G = typename std::conditional<SMALL, uint8_t, uint16_t>::type;
    extern __shared__ __attribute__((aligned(16))) char s_mem[];
    W *s_key = reinterpret_cast<W *>(s_mem);                                  // [cap][64]
    int32_t *s_rank = reinterpret_cast<int32_t *>(s_key + cap * PLAN_ROWS);   // rank_len
    G *s_grp = reinterpret_cast<G *>(s_rank + p.rank_len);                    // [cap][64]
    uint16_t *s_flat = SMALL ? reinterpret_cast<uint16_t *>(s_mem)            // [cap * 64]
                             : reinterpret_cast<uint16_t *>(s_grp + cap * PLAN_ROWS);
    __shared__ W s_w[PLAN_ROWS];
    __shared__ double2 s_big[PLAN_ROWS];
    __shared__ int s_cnt[PLAN_WAVES][PLAN_ROWS];
    const int lane = threadIdx.x & 63, wave = plan_wave();
    const int64_t r0 = (int64_t)blockIdx.x * PLAN_ROWS, r = r0 + lane;
    const bool on = r < p.M;
    const W w = on ? plan_row_word<RK, W>(p, r) : W(0);
    if (wave == 0) s_w[lane] = w;
    plan_stage_rank<W>(p, s_rank);
    if (p.big >= 0 && wave == PLAN_WAVES - 1) {
        bool any = false;
        s_big[lane] = plan_big<1, W>(p, 0, 1, w, any);
    }
    const int n = plan_expand<PLAN_WAVES, W>(p, w, on, s_cnt, [&](int e, int g) {
        if (e < cap) {
            s_key[e * PLAN_ROWS + lane] = plan_key<CK, W>(p, w ^ p.groups[g].flip);
            s_grp[e * PLAN_ROWS + lane] = (G)g;
        }
    });
    __syncthreads();
    const int64_t base = rowptr[r0];
    const int off = on ? (int)(rowptr[r] - base) : 0;
    // four entries a round: how many keys of the row are smaller
    auto places = [&](int i0) {
        W key[4];
        int below[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int i = i0 + u * PLAN_WAVES;
            key[u] = i < n ? s_key[i * PLAN_ROWS + lane] : W(0);
            below[u] = 0;
        }
        for (int j = 0; j < n; ++j) {
            const W kj = s_key[j * PLAN_ROWS + lane];
#pragma unroll
            for (int u = 0; u < 4; ++u) below[u] += kj < key[u];
        }
        return (uint32_t)(below[0] | below[1] << 8 | below[2] << 16 | below[3] << 24);
    };
    auto put = [&](int i0, uint32_t at) {
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int i = i0 + u * PLAN_WAVES;
            if (i < n) s_flat[off + (int)(at >> (8 * u) & 255)] = (uint16_t)(lane | (i << 6));
        }
    };
    if constexpr (SMALL) {   // the keys' room is written once they are all read
        constexpr int ROUNDS = PLAN_SMALL_ROW / (4 * PLAN_WAVES);
        uint32_t at[ROUNDS];
#pragma unroll
        for (int q = 0; q < ROUNDS; ++q) {
            const int i0 = wave + q * 4 * PLAN_WAVES;
            at[q] = i0 < n ? places(i0) : 0;
        }
        __syncthreads();
#pragma unroll
        for (int q = 0; q < ROUNDS; ++q) put(wave + q * 4 * PLAN_WAVES, at[q]);
    } else {
        for (int i0 = wave; i0 < n; i0 += 4 * PLAN_WAVES) put(i0, places(i0));
    }
    __syncthreads();
    const int64_t rend = r0 + PLAN_ROWS < p.M ? r0 + PLAN_ROWS : p.M;
    const int total = (int)(rowptr[rend] - base);
    for (int e0 = threadIdx.x; e0 < total; e0 += 256 * FILL_U) {
        int gi[FILL_U], row[FILL_U];
        W rw[FILL_U];
        PlanGroup<W> g[FILL_U];
#pragma unroll
        for (int u = 0; u < FILL_U; ++u) {
            const int e = e0 + 256 * u;
            const int f = s_flat[e < total ? e : e0];
            row[u] = f & 63;
            gi[u] = s_grp[(f >> 6) * PLAN_ROWS + row[u]];
            rw[u] = s_w[row[u]];
            g[u] = p.groups[gi[u]];
        }
#pragma unroll
        for (int u = 0; u < FILL_U; ++u) {
            const int e = e0 + 256 * u;
            if (e >= total) break;
            double2 acc = gi[u] == p.big ? s_big[row[u]] : plan_sum<W>(p, g[u].tbeg, g[u].tend, rw[u]);
            if (gi[u] == p.diag) acc = make_double2(acc.x + p.omega.x, acc.y + p.omega.y);
            cols[base + e] = plan_col<CK, W>(p, rw[u] ^ g[u].flip, s_rank);
            vals[base + e] = acc;
        }
    }
}

// ------------------------------------------------------------------ host side

struct PlanSpaces {
    int rk, ck;
    int nv, nc;
    const edx_basis *left, *right;
};

// A term as the device needs it, in 64-bit words; false if it never reaches
// the column space.
struct HostTerm {
    uint64_t m = 0, v = 0, f = 0, s = 0, group = 0;
    uint32_t neg = 0;
};

bool plan_term(const PlanSpaces &sp, uint32_t op, bool hop, bool negate, HostTerm &t) {
    const int pos[4] = {(int)(op & 63), (int)(op >> 8 & 63), (int)(op >> 16 & 63), (int)(op >> 24 & 63)};
    const int nops = hop ? 2 : 4;
    const int top = sp.ck == COL_PLAIN && sp.rk == ROW_PLAIN ? sp.right->nbits : sp.nv + sp.nc;
    int dval = 0, dcore = 0;
    for (int q = 0; q < nops; ++q) {
        const uint64_t bit = 1ull << pos[q], below = bit - 1;
        const bool filled = q < nops / 2;   // taken out first, then put in
        const bool now = (t.m & bit) ? ((t.v ^ t.f) & bit) != 0 : filled;
        if (now != filled) return false;    // a second operator of the same kind on one orbital
        if (!(t.m & bit)) {
            t.m |= bit;
            if (filled) t.v |= bit;
        }
        t.neg ^= (uint32_t)__builtin_popcountll(t.f & below) & 1u;
        t.s ^= below;
        t.f ^= bit;
        if (sp.rk == ROW_PLAIN || pos[q] < sp.nv) dval += filled ? -1 : 1;
        else dcore += filled ? -1 : 1;
    }
    if (negate) t.neg ^= 1u;
    if (top < 64 && (t.f >> top) != 0) return false;
    if (top < 64 && (t.v >> top) != 0) return false;   // needs an orbital no row has
    if (sp.left->nocc + dval != sp.right->nocc) return false;
    t.group = t.f;
    if (sp.ck == COL_VALONLY) t.group = t.f & ((1ull << sp.nv) - 1);
    if (sp.ck == COL_COREHOLE &&
        (sp.rk == ROW_COREHOLE ? sp.nc - 1 : sp.nc) + dcore != sp.nc - 1)
        return false;
    return true;
}

// A plan's device storage (one buffer) and description.
template <class W> struct PlanStore {
    Plan<W> p{};
    void *d_buf = nullptr;
    ~PlanStore() { edx::dfree(d_buf); }
    PlanStore() = default;
    PlanStore(const PlanStore &) = delete;
    PlanStore &operator=(const PlanStore &) = delete;
};

// The tables of plan_rank: for each RANK_BITS bits of a word, and each number of
// orbitals below them that a word of the basis can have, the part of the rank.
void plan_rank_tables(int nbits, int nocc, std::vector<int32_t> &tab, int *off, int *nrank) {
    std::vector<std::vector<int64_t>> C(nbits + 1, std::vector<int64_t>(nocc + 2, 0));
    for (int a = 0; a <= nbits; ++a) {
        C[a][0] = 1;
        for (int b = 1; b <= nocc + 1 && b <= a; ++b)
            C[a][b] = std::min(C[a - 1][b - 1] + C[a - 1][b], (int64_t)1 << 31);
    }
    *nrank = std::max((nbits + RANK_BITS - 1) / RANK_BITS, 1);
    const int words = 1 << RANK_BITS;
    for (int j = 0; j < RANK_MAX; ++j) {
        if (j >= *nrank) {   // nocc orbitals below and none here: entry 0 of the first row
            off[j] = -nocc * words;
            continue;
        }
        const int below = RANK_BITS * j;
        const int lo = std::max(0, nocc - (nbits - below)), hi = std::min(below, nocc);
        off[j] = (int)tab.size() - lo * words;
        for (int k0 = lo; k0 <= hi; ++k0)
            for (int c = 0; c < words; ++c) {
                int64_t l = 0;
                int k = k0;
                for (int b = 0; b < RANK_BITS; ++b)
                    if (c >> b & 1) {
                        ++k;   // a larger value is in no word's rank
                        if (below + b <= nbits && k <= nocc) l += C[below + b][k];
                    }
                tab.push_back(l < ((int64_t)1 << 31) ? (int32_t)l : 0);
            }
    }
}

// Terms of a group with the same test and parity mask have the same sign on
// every row up to one constant, so their sum may be taken here: summed in term
// order it is the row's own sum, or its negative, bit for bit (rounding is
// symmetric), as long as no row has survivors of two such classes, whose terms
// might alternate.  A part that sums to zero is +0 on every row unless all its
// terms are zeros of one sign (neg's flip flags).  Two-body terms come in four
// orders of their operators and two directions: eight terms become two.
struct TermClass {
    int lead;         // its first term
    double2 sum;      // in the lead's sign
    uint32_t flips;   // PLAN_FLIP_X, _Y
};

bool plan_merge_exact(const std::vector<HostTerm> &ht, const std::vector<double2> &hv,
                      const std::vector<int> &terms, std::vector<TermClass> &out) {
    out.clear();
    auto same_zero = [](double a, double b) {
        return a == 0.0 && b == 0.0 && std::signbit(a) == std::signbit(b);
    };
    for (int q : terms) {
        size_t c = 0;
        for (; c < out.size(); ++c) {
            const HostTerm &l = ht[out[c].lead];
            if (l.m == ht[q].m && l.v == ht[q].v && l.s == ht[q].s) break;
            if (((l.v ^ ht[q].v) & l.m & ht[q].m) == 0) return false;   // one row may have both
        }
        if (c == out.size()) {
            out.push_back(TermClass{q, hv[q], PLAN_FLIP_X | PLAN_FLIP_Y});
            continue;
        }
        TermClass &k = out[c];
        const double sg = ht[q].neg == ht[k.lead].neg ? 1.0 : -1.0;
        const double2 v = make_double2(sg * hv[q].x, sg * hv[q].y);
        if (!same_zero(hv[k.lead].x, v.x)) k.flips &= ~PLAN_FLIP_X;
        if (!same_zero(hv[k.lead].y, v.y)) k.flips &= ~PLAN_FLIP_Y;
        k.sum.x += v.x;
        k.sum.y += v.y;
    }
    for (TermClass &k : out) {
        if (k.sum.x != 0.0) k.flips |= PLAN_FLIP_X;
        if (k.sum.y != 0.0) k.flips |= PLAN_FLIP_Y;
    }
    return true;
}

// The terms that reach the column space, grouped by where they lead.
struct PlanTerms {
    struct Group {
        uint64_t key;
        int head, tail;   // its terms, chained by next in term order
    };
    std::vector<HostTerm> ht;
    std::vector<double2> hv;
    std::vector<int> next;
    std::vector<Group> groups;
};

// Groups the terms; false as soon as there are more than max_groups.  merge: terms
// that differ in their value only become one (the matrix-free apply, whose sums
// need not keep the term order).
bool plan_group(const PlanSpaces &sp, const uint32_t *ops, const double2 *tv, int nhop, int T,
                bool omega_on, bool negate, bool merge, double max_groups, PlanTerms &out) {
    auto &ht = out.ht;
    auto &hv = out.hv;
    auto &next = out.next;
    auto &groups = out.groups;
    ht.reserve(T);
    hv.reserve(T);
    next.reserve(T);
    int bits = 6;
    while ((1 << bits) < 2 * (T + 1)) ++bits;
    std::vector<int> table((size_t)1 << bits, -1);
    auto group_of = [&](uint64_t key) {
        for (int i = (int)(key * 0x9e3779b97f4a7c15ull >> (64 - bits));; i = (i + 1) & ((1 << bits) - 1)) {
            if (table[i] < 0) {
                table[i] = (int)groups.size();
                groups.push_back(PlanTerms::Group{key, -1, -1});
            }
            if (groups[table[i]].key == key) return table[i];
        }
    };
    if (omega_on) group_of(0);   // the diagonal, present in every row
    for (int t = 0; t < T; ++t) {
        HostTerm h;
        if (!plan_term(sp, ops[t], t < nhop, negate, h)) continue;
        PlanTerms::Group &g = groups[group_of(h.group)];
        if ((double)groups.size() > max_groups) return false;
        if (merge) {
            bool found = false;
            for (int q = g.head; q >= 0; q = next[q])
                if (ht[q].m == h.m && ht[q].v == h.v && ht[q].s == h.s) {
                    const double sg = ht[q].neg == h.neg ? 1.0 : -1.0;
                    hv[q].x += sg * tv[t].x;
                    hv[q].y += sg * tv[t].y;
                    found = true;
                    break;
                }
            if (found) continue;
        }
        const int q = (int)ht.size();
        (g.head < 0 ? g.head : next[g.tail]) = q;
        g.tail = q;
        ht.push_back(h);
        hv.push_back(tv[t]);
        next.push_back(-1);
    }
    return true;
}

// Entries of a mean row, from below: the largest share of rows that one term of
// each group survives on.
double plan_mean_row(const PlanSpaces &sp, const PlanTerms &pt) {
    const int n = sp.left->nbits, N = sp.left->nocc;
    auto falling = [](int x, int k) {   // x (x-1) ... (x-k+1), 0 if it runs out
        double r = 1.0;
        for (int i = 0; i < k; ++i) r *= std::max(x - i, 0);
        return r;
    };
    const uint64_t val = sp.rk == ROW_PLAIN ? ~0ull : (1ull << sp.nv) - 1;
    double rows = 0.0;
    for (const PlanTerms::Group &g : pt.groups) {
        double best = 0.0;
        for (int q = g.head; q >= 0; q = pt.next[q]) {
            const HostTerm &h = pt.ht[q];
            const int full = __builtin_popcountll(h.v & val), empty = __builtin_popcountll(h.m & val) - full;
            double share = falling(N, full) * falling(n - N, empty) / std::max(falling(n, full + empty), 1.0);
            const int cfull = __builtin_popcountll(h.v & ~val), cempty = __builtin_popcountll(h.m & ~val) - cfull;
            if (sp.rk == ROW_COREHOLE)
                share *= cempty == 0 ? (double)(sp.nc - cfull) / sp.nc : (cempty == 1 ? 1.0 / sp.nc : 0.0);
            if (sp.rk == ROW_FULLCORE && cempty) share = 0.0;
            best = std::max(best, share);
        }
        rows += best;
    }
    return rows;
}

// The plan of grouped terms.  waves: those of the kernels that expand it.
// exact_sums: a group's terms are summed in term order, bit for bit.
template <class W>
int plan_make(const PlanSpaces &sp, const PlanTerms &pt, bool omega_on, double2 omega, int waves,
              bool exact_sums, PlanStore<W> &out) {
    const auto &ht = pt.ht;
    const auto &hv = pt.hv;
    const auto &next = pt.next;
    const auto &groups = pt.groups;
    const int G = (int)groups.size();
    int nchunk = (G + PLAN_CHUNK - 1) / PLAN_CHUNK;
    nchunk = std::max((nchunk + waves - 1) / waves, 1) * waves;
    const int gpc = std::max((G + nchunk - 1) / nchunk, 1);
    std::vector<PlanTest<W>> tests;
    std::vector<int32_t> chunks(nchunk + 1, 0);
    std::vector<PlanTerm<W>> terms;
    std::vector<double2> vals;
    std::vector<PlanGroup<W>> dg(std::max(G, 1));
    int big = -1, nbig = PLAN_BIG;
    std::vector<std::pair<uint64_t, uint64_t>> kept;
    std::vector<TermClass> classes;
    std::vector<int> members;
    terms.reserve(ht.size());
    vals.reserve(ht.size());
    tests.reserve(ht.size());
    for (int c = 0; c < nchunk; ++c) {
        chunks[c] = (int32_t)tests.size();
        for (int g = c * gpc; g < std::min((c + 1) * gpc, G); ++g) {
            const PlanTerms::Group &gr = groups[g];
            members.clear();
            for (int q = gr.head; q >= 0; q = next[q]) members.push_back(q);
            PlanGroup<W> &d = dg[g];
            d.flip = 0;
            d.tbeg = (int32_t)terms.size();
            const bool exact = exact_sums && plan_merge_exact(ht, hv, members, classes);
            const size_t count = exact ? classes.size() : members.size();
            for (size_t i = 0; i < count; ++i) {
                const int q = exact ? classes[i].lead : members[i];
                const uint32_t flips = exact ? classes[i].flips : PLAN_FLIP_X | PLAN_FLIP_Y;
                terms.push_back(PlanTerm<W>{(W)ht[q].m, (W)ht[q].v, (W)ht[q].s, ht[q].neg | flips});
                vals.push_back(exact ? classes[i].sum : hv[q]);
                d.flip = (W)ht[q].f;
            }
            if (sp.ck == COL_VALONLY) d.flip = (W)gr.key;
            d.tend = (int32_t)terms.size();
            if (d.tend - d.tbeg > nbig) {
                nbig = d.tend - d.tbeg;
                big = g;
            }
            // survival tests, weakest first: one implied by a weaker one adds nothing
            kept.clear();
            if (omega_on && g == 0) {
                kept.emplace_back(0, 0);
            } else {
                for (int bits = 1; bits <= 4; ++bits)
                    for (int q : members) {
                        if (__builtin_popcountll(ht[q].m) != bits) continue;
                        bool implied = false;
                        for (auto &k : kept)
                            if ((ht[q].m & k.first) == k.first && (ht[q].v & k.first) == k.second) {
                                implied = true;
                                break;
                            }
                        if (!implied) kept.emplace_back(ht[q].m, ht[q].v);
                    }
            }
            for (size_t i = 0; i < kept.size(); i += 2) {
                PlanTest<W> q{};
                q.bit = 1u << (g - c * gpc);
                for (int u = 0; u < 2; ++u) {
                    const auto &k = kept[std::min(i + u, kept.size() - 1)];
                    q.m[u] = (W)k.first;
                    q.v[u] = (W)k.second;
                }
                tests.push_back(q);
            }
        }
    }
    chunks[nchunk] = (int32_t)tests.size();
    std::vector<PlanDens<W>> dens;
    double dens_y = 0.0;
    if (big >= 0) {
        for (int t = dg[big].tbeg; t < dg[big].tend; ++t) {
            const uint32_t neg = terms[t].neg;
            double2 v = vals[t];
            if ((neg & 1) && (neg & PLAN_FLIP_X)) v.x = -v.x;
            if ((neg & 1) && (neg & PLAN_FLIP_Y)) v.y = -v.y;
            if (t == dg[big].tbeg) dens_y = exact_sums ? v.y : 0.0;
            if (terms[t].s != 0 || v.y != 0.0 ||
                (exact_sums && std::signbit(v.y) != std::signbit(dens_y))) {
                dens.clear();
                break;
            }
            dens.push_back(PlanDens<W>{terms[t].m, terms[t].v, v.x});
        }
    }
    auto up = [](size_t b) { return (b + 63) / 64 * 64; };
    // two spare records: the scalar loads of the unrolled loop stay inside
    const size_t b_tests = up((tests.size() + 2) * sizeof(PlanTest<W>));
    const size_t b_chunks = up(chunks.size() * sizeof(int32_t));
    const size_t b_terms = up((terms.size() + 2) * sizeof(PlanTerm<W>));
    const size_t b_vals = up((vals.size() + 2) * sizeof(double2));
    const size_t b_groups = up(dg.size() * sizeof(PlanGroup<W>));
    Plan<W> &p = out.p;
    std::vector<int32_t> rank;
    plan_rank_tables(sp.right->nbits, sp.right->nocc, rank, p.rank_off, &p.nrank);
    const size_t b_rank = up(rank.size() * sizeof(int32_t));
    const size_t b_dens = up((dens.size() + 4) * sizeof(PlanDens<W>));
    std::vector<char> buf(b_tests + b_chunks + b_terms + b_vals + b_groups + b_rank + b_dens, 0);
    char *h = buf.data();
    const size_t o_chunks = b_tests, o_terms = o_chunks + b_chunks, o_vals = o_terms + b_terms,
                 o_groups = o_vals + b_vals, o_rank = o_groups + b_groups,
                 o_dens = o_rank + b_rank;
    if (!tests.empty()) memcpy(h, tests.data(), tests.size() * sizeof(PlanTest<W>));
    memcpy(h + o_chunks, chunks.data(), chunks.size() * sizeof(int32_t));
    if (!terms.empty()) {
        memcpy(h + o_terms, terms.data(), terms.size() * sizeof(PlanTerm<W>));
        memcpy(h + o_vals, vals.data(), vals.size() * sizeof(double2));
    }
    memcpy(h + o_groups, dg.data(), dg.size() * sizeof(PlanGroup<W>));
    memcpy(h + o_rank, rank.data(), rank.size() * sizeof(int32_t));
    if (!dens.empty()) memcpy(h + o_dens, dens.data(), dens.size() * sizeof(PlanDens<W>));
    out.d_buf = edx::dmalloc(buf.size(), "term plan");
    if (!out.d_buf) return EDX_ERR_NOMEM;
    EDX_HIP(edx::copy_sync(out.d_buf, h, buf.size(), hipMemcpyHostToDevice));
    char *d = (char *)out.d_buf;
    p.tests = (const PlanTest<W> *)d;
    p.chunks = (const int32_t *)(d + o_chunks);
    p.terms = (const PlanTerm<W> *)(d + o_terms);
    p.vals = (const double2 *)(d + o_vals);
    p.groups = (const PlanGroup<W> *)(d + o_groups);
    p.rank = (const int32_t *)(d + o_rank);
    p.rank_len = (int)rank.size();
    p.ngroups = G;
    p.nchunk = nchunk;
    p.gpc = gpc;
    p.big = big;
    p.dens = (const PlanDens<W> *)(d + o_dens);
    p.ndens = (int)dens.size();
    p.dens_y = dens_y;
    p.diag = omega_on ? 0 : -1;
    p.omega = omega;
    p.left = sp.left->d_words;
    p.nleft = sp.left->n;
    p.M = sp.rk == ROW_COREHOLE ? sp.left->n * sp.nc : sp.left->n;
    p.nv = sp.nv;
    p.nc = sp.nc;
    p.nbits = sp.right->nbits;
    p.nocc = sp.right->nocc;
    p.nright = sp.right->n;
    p.inter = edx::corehole_layout() == EDX_COREHOLE_INTERLEAVED;
    return EDX_OK;
}

// Whether the spaces have closed-form columns: complete bases of one valence
// width, and no orbital outside the words where columns ignore the core word.
bool plan_usable(const PlanSpaces &sp, const uint32_t *ops, int nhop, int T) {
    if (!sp.left->complete || !sp.right->complete || T > PLAN_MAX_TERMS) return false;
    if (sp.left->nbits != sp.right->nbits) return false;
    if (sp.rk != ROW_PLAIN && sp.left->nbits != sp.nv) return false;
    if (sp.ck == COL_VALONLY)
        for (int t = 0; t < T; ++t)
            for (int q = 0; q < (t < nhop ? 2 : 4); ++q)
                if ((int)(ops[t] >> (8 * q) & 63) >= sp.nv + sp.nc) return false;
    return true;
}

int plan_bits(const PlanSpaces &sp) {
    return sp.rk == ROW_PLAIN && sp.ck == COL_PLAIN ? sp.right->nbits : sp.nv + sp.nc;
}

constexpr int PLAN_LDS = 144 << 10;   // of 160 KB, with room for the static arrays

// Longest row the fill's lists can hold.
template <class W> int plan_max_row(const Plan<W> &p) {
    const int per = PLAN_ROWS * (int)(sizeof(W) + 4);
    return std::min((PLAN_LDS - p.rank_len * 4) / per, 255);
}

template <int RK, class W>
int plan_count(const Plan<W> &p, int64_t *counts, int *d_maxrow) {
    hipLaunchKernelGGL((k_plan_count<RK, W>), dim3((unsigned)((p.M + PLAN_ROWS - 1) / PLAN_ROWS)),
                       dim3(256), 0, edx::stream(), p, counts, d_maxrow);
    EDX_LAUNCH_CHECK();
    return EDX_OK;
}

template <bool SMALL, int RK, int CK, class W>
int plan_fill_launch(const Plan<W> &p, int cap, size_t entry, const int64_t *rowptr, int32_t *cols,
                     double2 *vals) {
    const size_t lds = (size_t)cap * PLAN_ROWS * entry + (size_t)p.rank_len * 4;
    if (lds > (64 << 10))
        EDX_HIP(hipFuncSetAttribute(reinterpret_cast<const void *>(k_plan_fill<SMALL, RK, CK, W>),
                                    hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    hipLaunchKernelGGL((k_plan_fill<SMALL, RK, CK, W>),
                       dim3((unsigned)((p.M + PLAN_ROWS - 1) / PLAN_ROWS)), dim3(256), lds,
                       edx::stream(), p, cap, rowptr, cols, vals);
    EDX_LAUNCH_CHECK();
    return EDX_OK;
}

template <int RK, int CK, class W>
int plan_fill(const Plan<W> &p, int maxrow, const int64_t *rowptr, int32_t *cols, double2 *vals) {
    const int cap = std::max((maxrow + 3) / 4 * 4, 4);
    if (cap <= PLAN_SMALL_ROW && p.ngroups <= 256)
        return plan_fill_launch<true, RK, CK, W>(p, cap, sizeof(W) + 1, rowptr, cols, vals);
    return plan_fill_launch<false, RK, CK, W>(p, cap, sizeof(W) + 4, rowptr, cols, vals);
}

}  // namespace
