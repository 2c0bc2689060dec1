// odemi_lu.h -- FP64 LU with partial pivoting of a matrix in LDS, factored by
// the workgroup of the FP64 Rodas5P kernels (256 threads, or 512 where they are
// built for eight waves), and the triangular solves with it.
//
// Every element sees the fma sequence of the sequential right-looking LU
// (a_ij -= l_ik u_kj, k ascending) and of the column-ordered substitutions, and
// every quotient is the IEEE one, so the results are those of the CPU
// restatement bit for bit; only who computes what and when is different.
//
// Bound: the instruction latency of one wave (a chain of 2 n substitution steps
// a solve, n pivot steps a factorization), one trajectory a workgroup.  Measured
// with these functions alone, one workgroup a CU: factorization 84 us with four
// waves, 79 us with eight at n = 128 (53 and 50 at 96, 28 and 27 at 64, 12 at 32);
// solve, one wave in both, 8.2 us (6.4, 4.4, 2.5).  96 chains of n = 8..128 with
// the element-by-element factorization and IEEE quotients in every step 43.2 ms,
// with this one 10.5 ms on four waves and 10.0 ms on eight from n = 96 on.
#pragma once

namespace odemi {

// Panel width.  The steps of a panel are unrolled (a lane's row stays in
// registers), so the width sets the size of the code that every panel runs
// through: 16 columns made 40 KB of it, which the instruction cache did not hold
// (3,000-5,000 cycles a pivot step).
constexpr int kLuNB = 8;

// 2^-400 <= |v| < 2^401, from the high word of v: quotients and reciprocals of
// such values need none of the scaling and fix-ups of the IEEE division.
__device__ __forceinline__ bool lu_in_range(unsigned hi) {
    return ((hi & 0x7fffffffu) - 0x26f00000u) < 0x32100000u;
}
__device__ __forceinline__ unsigned hi_word(double v) { return (unsigned)__double2hiint(v); }

// Values of a wave's LDS writes as its other lanes read them afterwards (LDS
// serves a wave's accesses in order; this orders them for the compiler).
__device__ __forceinline__ void lu_wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

typedef double lud4 __attribute__((ext_vector_type(4)));

// Pivot search of one step by the whole rule: the first maximum of |v| by
// position, a NaN at position k keeping that row and any other NaN losing.
// Returns the winning lane, its row slot in wq.
template <int NQ>
__device__ __forceinline__ int lu_search(const double (&x)[NQ], const int (&pos)[NQ], int k, int& wq) {
    unsigned long long key = 0;
    int cpos = 0x7fffffff, cq = 0;
#pragma unroll
    for (int q = 0; q < NQ; q++) {
        // bits of |v|, the high word one up; rows out of the search 0
        unsigned long long h = ((unsigned long long)__double_as_longlong(x[q]) & 0x7fffffffffffffffull) + (1ull << 32);
        if (x[q] != x[q]) h = (pos[q] == k) ? ~0ull : 0ull;
        if (pos[q] < k) h = 0ull;
        if (h > key || (h == key && pos[q] >= k && pos[q] < cpos)) { key = h; cpos = pos[q]; cq = q; }
    }
    const unsigned kh = (unsigned)(key >> 32), top = dpp_wave_max_u32(kh);
    const unsigned lo = (kh == top) ? (unsigned)key : 0u, ltop = dpp_wave_max_u32(lo);
    const bool in = kh == top && lo == ltop;
    const unsigned first = ~dpp_wave_max_u32(in ? ~(unsigned)cpos : 0u);
    const int wl = __ffsll((unsigned long long)__ballot(in && (unsigned)cpos == first)) - 1;
    wq = __builtin_amdgcn_readlane(cq, wl);
    return wl;
}

// The 8 (or n - k0 last) steps of the panel at column k0, by one wave: lane l
// holds the panel's entries of rows k0 + l + 64 q (n - k0 <= 64 NQ).  Rows stay
// in their lanes; pos is the position that the row interchanges would have
// moved them to: rows at positions below k are pivot rows already (-1: no row).
// One wave's issue bounds the step, so it takes as few instructions as it can:
// the search compares high words (lu_search only where several rows share the
// largest, or it is out of the range of the short reciprocal), and each lane
// refines the reciprocal of its own candidate beside the DPP maximum.  At the end
// the rows are stored at their positions, perm follows, and for the other columns
// tab[j] = offset (row * ld) of the row that became pivot row k0 + j,
// tab[8 + j] = offset of the position that row k0 + j moved to, -1: a pivot row.
template <int NQ>
__device__ __forceinline__ void lu_panel(double* A, int ld, int n, int k0, int* tab, int* perm) {
    const int l = threadIdx.x & 63;
    const int mc = min(kLuNB, n - k0);
    double v[NQ][kLuNB];
    int pos[NQ], pm[NQ];
#pragma unroll
    for (int q = 0; q < NQ; q++) {
        const int i = k0 + l + 64 * q, ic = min(i, n - 1);
        pos[q] = (i < n) ? i : -1;
        pm[q] = perm[ic];
        // columns past n (last panel) are read, never used: W is followed by the vectors
#pragma unroll
        for (int c = 0; c < kLuNB; c++) v[q][c] = A[ic * ld + k0 + c];
    }
#pragma unroll
    for (int kt = 0; kt < kLuNB; kt++) {
        if (kt >= mc) break;   // uniform
        const int k = k0 + kt;
        unsigned h[NQ], hm = 0;
        double cand = v[0][kt];
#pragma unroll
        for (int q = 0; q < NQ; q++) {
            h[q] = (pos[q] >= k) ? (hi_word(v[q][kt]) & 0x7fffffffu) : 0u;
            if (q > 0) cand = (h[q] > hm) ? v[q][kt] : cand;
            hm = max(hm, h[q]);
        }
        const double rc = rcp_nr(cand);
        const double ic = fma(fma(-cand, rc, 1.0), rc, rc);
        const unsigned top = dpp_wave_max_u32(hm);
        double icv = ic;
        asm volatile("" : "+v"(icv));   // computed here, beside the maximum, not behind the branch
        unsigned long long any = 0;
        int cnt = 0, wq = 0, wl;
#pragma unroll
        for (int q = 0; q < NQ; q++) {
            const unsigned long long m = __ballot(h[q] == top);
            if (q > 0) wq = m ? q : wq;
            cnt += __popcll(m);
            any |= m;
        }
        double inv;
        if (lu_in_range(top) && cnt == 1) {   // uniform
            wl = __ffsll(any) - 1;
            inv = wave_bcast(icv, wl);
        } else {
            double x[NQ], pv = 0.0;
#pragma unroll
            for (int q = 0; q < NQ; q++) x[q] = v[q][kt];
            wl = lu_search<NQ>(x, pos, k, wq);
#pragma unroll
            for (int q = 0; q < NQ; q++)
                if (wq == q) pv = wave_bcast(x[q], wl);
            inv = 1.0 / pv;
        }
        int wpos = 0;
        double pr[kLuNB];
#pragma unroll
        for (int q = 0; q < NQ; q++)
            if (wq == q) {   // uniform
                wpos = __builtin_amdgcn_readlane(pos[q], wl);
#pragma unroll
                for (int c = kt + 1; c < kLuNB; c++) pr[c] = wave_bcast(v[q][c], wl);
            }
#pragma unroll
        for (int q = 0; q < NQ; q++) {
            pos[q] = (pos[q] == k) ? wpos : pos[q];
            pos[q] = (wq == q && l == wl) ? k : pos[q];
            if (pos[q] > k) {
                const double m = v[q][kt] * inv;
                v[q][kt] = m;
#pragma unroll
                for (int c = kt + 1; c < kLuNB; c++) v[q][c] = fma(-m, pr[c], v[q][c]);
            }
        }
    }
    lu_wave_sync();
#pragma unroll
    for (int q = 0; q < NQ; q++)
        if (pos[q] >= 0) {
            const int i = k0 + l + 64 * q;
            double* row = A + pos[q] * ld + k0;
            if (mc == kLuNB) {   // uniform
#pragma unroll
                for (int c = 0; c < kLuNB; c++) row[c] = v[q][c];
            } else {
#pragma unroll
                for (int c = 0; c < kLuNB; c++)
                    if (c < mc) row[c] = v[q][c];
            }
            perm[pos[q]] = pm[q];
            if (pos[q] < k0 + mc) tab[pos[q] - k0] = i * ld;
            if (i < k0 + mc) tab[kLuNB + i - k0] = pos[q] >= k0 + mc ? pos[q] * ld : -1;
        }
}

// lu_panel with as few row slots as the n - k0 remaining rows need
template <int NQ>
__device__ __forceinline__ void lu_panel_rows(double* A, int ld, int n, int k0, int* tab, int* perm) {
    if constexpr (NQ > 1)
        if (n - k0 <= 64 * (NQ - 1)) return lu_panel_rows<NQ - 1>(A, ld, n, k0, tab, perm);
    lu_panel<NQ>(A, ld, n, k0, tab, perm);
}

// In-place LU with partial pivoting of the n x n leading block of A (stride
// ld), n <= 64 NQ.  perm[n]: the row gather, (P b)[i] = b[perm[i]].  tab[16]:
// scratch, 16-byte aligned.
//
// Blocked by 8 columns, because the element-by-element form spent its time in
// two workgroup barriers, a shuffled argmax and an LDS pass over the whole
// trailing matrix for each of the n pivots.  The panel's 8 steps run on one wave
// in registers (lu_panel).  Every wave owns the blocks of 16 columns
// w, w + waves, ...: one lane a column moves the 16 exchanged entries and solves the
// 8 x 8 unit triangle, then the wave updates its blocks of the trailing matrix
// on the matrix cores (2 v_mfma_f64_16x16x4 a 16 x 16 block, whose four products
// are added one after the other with one rounding each, as the fma chain does).
// Two workgroup barriers a panel.
template <int NQ>
__device__ __forceinline__ void wg_lu_blocked(double* A, int ld, int n, int* tab, int* perm) {
    constexpr int KC = kLuNB / 4;
    const int tid = threadIdx.x, NT = blockDim.x, NW = NT >> 6;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6), l = tid & 63, g = l >> 4, c16 = l & 15;
    for (int i = tid; i < n; i += NT) perm[i] = i;
    __syncthreads();
    for (int k0 = 0; k0 < n; k0 += kLuNB) {
        if (w == 0) lu_panel_rows<NQ>(A, ld, n, k0, tab, perm);
        __syncthreads();
        const int mc = min(kLuNB, n - k0), k1 = k0 + mc;
        // Row exchanges and U rows of the wave's blocks, two at a time: lanes 0-15
        // and 16-31 take a column each and bring in the pivot rows, lanes 32-63 the
        // same columns and move the displaced rows out.
        {
            const bool out = l >= 32;
            const double* T = A + k0 * ld + k0;
            double L[kLuNB][kLuNB];
            int from[kLuNB], to[kLuNB];
#pragma unroll
            for (int j = 0; j < kLuNB; j++) {   // mc < kLuNB only in the last panel: row n - 1 again
                const int top = (k0 + min(j, mc - 1)) * ld;
                const int s = tab[min(j, mc - 1)], d = tab[kLuNB + min(j, mc - 1)];
                from[j] = out ? top : s;
                to[j] = out ? d : top;
            }
#pragma unroll
            for (int j = 1; j < kLuNB; j++)
#pragma unroll
                for (int i = 0; i < j; i++) L[j][i] = T[min(j, mc - 1) * ld + i];
            for (int J = 16 * w; J < n; J += 32 * NW) {
                const int c = J + c16 + ((l & 16) ? 16 * NW : 0);
                if (c < n && (c < k0 || c >= k1)) {
                    double t[kLuNB];
#pragma unroll
                    for (int j = 0; j < kLuNB; j++) t[j] = A[from[j] + c];
                    if (c >= k1 && !out) {   // then mc == kLuNB
#pragma unroll
                        for (int j = 1; j < kLuNB; j++)
#pragma unroll
                            for (int i = 0; i < j; i++) t[j] = fma(-L[j][i], t[i], t[j]);
                    }
#pragma unroll
                    for (int j = 0; j < kLuNB; j++)
                        if (to[j] >= 0) A[to[j] + c] = t[j];
                }
            }
        }
        lu_wave_sync();
        for (int J = 16 * w; J < n; J += 16 * NW) {
            if (k1 >= n || J + 16 <= k1) continue;   // uniform
            const int c = J + c16;
            // The block's trailing rows: a 16 x 16 tile's values are loaded while the
            // one above is on the matrix cores.  Only the last tile can be short.
            const int jc = min(c, n - 1);
            const bool in = c >= k1 && c < n;
            double b[KC], a[KC], an[KC];
            lud4 d, e;
#pragma unroll
            for (int kc = 0; kc < KC; kc++) b[kc] = A[(k0 + 4 * kc + g) * ld + jc];
            const double* ra = A + (k1 + c16) * ld + k0 + g;
            double* rc[4];
#pragma unroll
            for (int r = 0; r < 4; r++) rc[r] = A + (k1 + 4 * r + g) * ld + jc;
            // tile at row I, whose row pointers are ra and rc
            auto load = [&](int I, double (&av)[KC], lud4& x) {
                if (I + 16 > n) {
                    ra = A + min(I + c16, n - 1) * ld + k0 + g;
#pragma unroll
                    for (int r = 0; r < 4; r++) rc[r] = A + min(I + 4 * r + g, n - 1) * ld + jc;
                }
#pragma unroll
                for (int kc = 0; kc < KC; kc++) av[kc] = -ra[4 * kc];
#pragma unroll
                for (int r = 0; r < 4; r++) x[r] = *rc[r];
            };
            load(k1, a, d);
            for (int I = k1; I < n; I += 16) {
                double* wr[4];
#pragma unroll
                for (int r = 0; r < 4; r++) wr[r] = rc[r];
                if (I + 16 < n) {
                    ra += 16 * ld;
#pragma unroll
                    for (int r = 0; r < 4; r++) rc[r] += 16 * ld;
                    load(I + 16, an, e);
                }
#pragma unroll
                for (int kc = 0; kc < KC; kc++) d = __builtin_amdgcn_mfma_f64_16x16x4f64(a[kc], b[kc], d, 0, 0, 0);
                if (I + 16 <= n) {   // uniform
                    if (in) {
#pragma unroll
                        for (int r = 0; r < 4; r++) *wr[r] = d[r];
                    }
                } else {
#pragma unroll
                    for (int r = 0; r < 4; r++)
                        if (in && I + 4 * r + g < n) *wr[r] = d[r];
                }
                d = e;
#pragma unroll
                for (int kc = 0; kc < KC; kc++) a[kc] = an[kc];
            }
        }
        __syncthreads();
    }
}

// x <- A^{-1} x (negated if NEG) with wg_lu_blocked's factors, by wave 0: lane l
// holds rows l + 64 q, a solved entry is broadcast with readlane, the factor's
// columns are read one chunk of 8 ahead, so the chain of a step is readlane and
// fma, and in the backward half the three fma of the quotient (each lane
// divides its own entry by its own pivot, whose reciprocal it refined once).
// Lanes then check that their dividend and pivot were in the range where that
// is the IEEE quotient; if one was not (or is -0, which the residual step would
// turn), x is left alone and false returned.  Wave 0 only.
template <int NQ, bool NEG>
__device__ __forceinline__ bool wave_lu_solve(const double* A, int ld, int n, const int* perm, double* x) {
    constexpr int CH = 8;
    const int l = threadIdx.x & 63;
    double b[NQ], piv[NQ], rp[NQ];
    const double* row[NQ];
#pragma unroll
    for (int q = 0; q < NQ; q++) {
        const int i = l + 64 * q;
        row[q] = A + min(i, n - 1) * ld;
        b[q] = (i < n) ? x[perm[i]] : 0.0;
        piv[q] = (i < n) ? row[q][i] : 1.0;
        rp[q] = rcp_nr(piv[q]);
    }
    // forward, unit lower triangle.  An entry goes on being updated after its
    // own step, so the solved ones are collected beside it.  Columns past n - 1
    // (up to 7, read behind W or in the next row) reach lanes past n only.
    const int ctop = (n - 1) & ~(CH - 1);
    double F[NQ][CH], G[NQ][CH], y[NQ];
#pragma unroll
    for (int q = 0; q < NQ; q++) {
        y[q] = b[q];
#pragma unroll
        for (int j = 0; j < CH; j++) F[q][j] = row[q][j];
    }
#pragma unroll
    for (int Q = 0; Q < NQ; Q++) {
        const int cend = min(64 * (Q + 1), n);
        for (int c0 = 64 * Q; c0 < cend; c0 += CH) {
            const int cn = min(c0 + CH, ctop);
#pragma unroll
            for (int q = Q; q < NQ; q++)
#pragma unroll
                for (int j = 0; j < CH; j++) G[q][j] = row[q][cn + j];
#pragma unroll
            for (int j = 0; j < CH; j++) {
                const int s = (c0 & 63) + j;
                const double xc = wave_bcast(b[Q], s);
                y[Q] = (l == s) ? b[Q] : y[Q];
#pragma unroll
                for (int q = Q; q < NQ; q++) b[q] = fma(-F[q][j], xc, b[q]);
            }
#pragma unroll
            for (int q = Q; q < NQ; q++)
#pragma unroll
                for (int j = 0; j < CH; j++) F[q][j] = G[q][j];
        }
    }
    // backward, upper triangle; the dividends are collected.  Columns past n: 0 * 0.
    int nl = n;
    asm("" : "+v"(nl));   // selected per lane, not branched around
#pragma unroll
    for (int q = 0; q < NQ; q++) {
        b[q] = (l + 64 * q < n) ? y[q] : 0.0;
        y[q] = b[q];
#pragma unroll
        for (int j = 0; j < CH; j++) {
            const double f = row[q][ctop + j];
            F[q][j] = (ctop + j < nl) ? f : 0.0;
        }
    }
#pragma unroll
    for (int Q = NQ - 1; Q >= 0; Q--) {
        for (int c0 = min(ctop, 64 * Q + 64 - CH); c0 >= 64 * Q; c0 -= CH) {
            const int cn = max(c0 - CH, 0);
#pragma unroll
            for (int q = 0; q <= Q; q++)
#pragma unroll
                for (int j = 0; j < CH; j++) G[q][j] = row[q][cn + j];
#pragma unroll
            for (int j = CH - 1; j >= 0; j--) {
                const int s = (c0 & 63) + j;
                y[Q] = (l == s) ? b[Q] : y[Q];
                const double xc = wave_bcast(div_by_rcp(b[Q], piv[Q], rp[Q]), s);
#pragma unroll
                for (int q = 0; q <= Q; q++) b[q] = fma(-F[q][j], xc, b[q]);
            }
#pragma unroll
            for (int q = 0; q <= Q; q++)
#pragma unroll
                for (int j = 0; j < CH; j++) F[q][j] = G[q][j];
        }
    }
    bool ok = true;
#pragma unroll
    for (int q = 0; q < NQ; q++) {
        const bool plus0 = __double_as_longlong(y[q]) == 0;
        ok = ok && (lu_in_range(hi_word(y[q])) || plus0) && lu_in_range(hi_word(piv[q]));
    }
    if (__ballot(!ok) != 0) return false;
#pragma unroll
    for (int q = 0; q < NQ; q++) {
        const int i = l + 64 * q;
        const double r = div_by_rcp(y[q], piv[q], rp[q]);
        if (i < n) x[i] = NEG ? -r : r;
    }
    return true;
}

}  // namespace odemi
