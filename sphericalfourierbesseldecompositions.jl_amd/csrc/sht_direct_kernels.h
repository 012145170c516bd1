// map2alm with its refinement iterations as one linear operator: the device side.
//
// Healpix's iteration a <- b + (1 - A S) a started from b = A delta is the polynomial
// P_J(A S) b, P_J(X) = sum_{j<=J} (1 - X)^j.  A S is C0 (dense per (m, parity), what ring
// sampling keeps on one m) plus the aliasing of short rings, which couples m to
// m' = +-m (mod npr).  With D = 1 - C0, S_m = Lam on the aliasing ring pairs kept for m
// (n_al x n_b), T_m = dOmega S_m^T and -K the coupling of ring values (k_alias_solve),
//   a = P_J(D) b + sum_j Z_j r_j,            Z_j = D^{J-1-j} T,
//   g_j = S P_j(D) b + sum_{i<j} Q_{j-1-i} r_i,  r_j = -K g_j,   Q_p = S D^p T,
// so every refined a comes from two products with tables laid out once per plan: X times
// [dOmega Lam P_J | dOmega Lam P_j S^T (j < J)], and [Z_0 .. Z_{J-1}] times the r_j.
// The iterated form ran a synthesis, an aliasing pass and a merged product per refinement.
//
// Which (ring pair, m) alias: lambda_lm falls off steeply beyond m ~ l sin(theta), and m and
// m' >= npr - m cannot both be inside it on a polar ring, so the product of the two lambdas
// is negligible on all but the first few ring pairs.  A pair of states is kept when
// dOmega npr mult max_l |lambda_lm| max_l' |lambda_l'm'| > 1e-18 (the entry of A S it makes, whose
// diagonal is ~1: what is dropped stays below an FP64 rounding of the coefficients).
#pragma once

// One batch of the row-addressed GEMM: C[crow + n][i] = alpha sum_k A[arow + k][i] B[k][n]
// (+ beta C) over the columns i in [col0, col0 + ncol) (ncol < 0: every column), with the row
// strides of A and C given at the launch.  dst: 0 -> C0, 1 -> C1.
struct RowGemm {
    const double* B;
    int64_t arow, crow;
    int32_t K, N, ldb, dst;
    int32_t col0, ncol;
};

// The GEMM of k_gemm_tall<FP64> on RowGemm batches (load-bound like it: 3 waves per SIMD).  One call with
// the folded table takes the place of the analysis and 2 niter refinement products.  159 shells, nside 128:
// 64 us; 219 shells, nside 256: 287 us.
__global__ __launch_bounds__(256, 3) void k_gemm_rows(const RowGemm* __restrict__ descs, int32_t cols,
                                                      const double* __restrict__ A, int64_t lda, double* C0,
                                                      int64_t ldc0, double* C1, int64_t ldc1, double alpha, double beta)
{
    __shared__ double As[GT_BK][GT_BM];
    __shared__ double Bs[GT_BK][GT_BNW];
    const RowGemm r = descs[blockIdx.z];
    const int ncol = r.ncol < 0 ? cols : r.ncol;
    const int i0 = blockIdx.x * GT_BM, n0 = blockIdx.y * GT_BNW;
    if (n0 >= r.N || i0 >= ncol) return;
    GemmDesc d;
    d.A = A + r.arow * lda + r.col0;
    d.B = r.B;
    const int64_t ldc = r.dst ? ldc1 : ldc0;
    d.C = (r.dst ? C1 : C0) + r.crow * ldc + r.col0;
    d.Cin = nullptr;
    d.K = r.K;
    d.N = r.N;
    d.lda = lda;
    d.ldb = r.ldb;
    d.ldc = ldc;
    d.A2 = d.B2 = nullptr;
    d.K1 = d.pad = 0;
    d.lda2 = d.ldb2 = 0;
    gemm_dispatch<false, false>(d, ncol, alpha, beta, i0, n0, As, Bs);
}

// Plan-time products: C = alpha A B (+ 1 when eye), any strides, one 16 x 16 tile per block.
struct SmallMM {
    const double *A, *B;
    double* C;
    int32_t M, N, K, eye;
    int64_t ars, acs, brs, bcs, crs, ccs;
    double alpha;
};
__global__ __launch_bounds__(256) void k_small_mm(const SmallMM* __restrict__ descs)
{
    __shared__ double As[16][17], Bs[16][17];
    const SmallMM d = descs[blockIdx.z];
    const int tx = threadIdx.x & 15, ty = threadIdx.x >> 4;
    const int i = blockIdx.y * 16 + ty, j = blockIdx.x * 16 + tx;
    if ((int)blockIdx.y * 16 >= d.M || (int)blockIdx.x * 16 >= d.N) return;
    double acc = 0.0;
    for (int k0 = 0; k0 < d.K; k0 += 16) {
        As[ty][tx] = (i < d.M && k0 + tx < d.K) ? d.A[i * d.ars + (k0 + tx) * d.acs] : 0.0;
        Bs[ty][tx] = (j < d.N && k0 + ty < d.K) ? d.B[(k0 + ty) * d.brs + j * d.bcs] : 0.0;
        __syncthreads();
#pragma unroll
        for (int k = 0; k < 16; ++k) acc = fma(As[ty][k], Bs[k][tx], acc);
        __syncthreads();
    }
    if (i < d.M && j < d.N) d.C[i * d.crs + j * d.ccs] = d.alpha * acc + ((d.eye && i == j) ? 1.0 : 0.0);
}

// An aliasing state: a kept (m, ring pair).  States are ordered by m, then ring pair; the
// states of one m are s0 .. s0 + na - 1.
struct AliasState {
    int32_t m, a, na, s0;  // a = s - s0
    int32_t e0, e1;        // couplings [e0, e1)
};
struct AliasTerm {
    int32_t s, pad;
    double cre, cim;  // coefficients of the partner's real and imaginary part
};

// h (J values per state and column) -> r: per column the J coupled steps
//   g_j = h_j + sum_{i<j} Q_{j-1-i} r_i,  r_j = sum of couplings of g_j.
// Columns alternate real and imaginary parts.  A column belongs to the sector of its l parity
// sg (parity of (m, l) blocks: (m + sg) & 1): sector blockIdx.y for split < 0, where sector sg's
// rows start at sg J S; else columns below split are of sector 0, the rest of sector 1, and the
// rows are shared.  Row of (s, j): J s0 + j na + a.  The values of CT columns (a power of two)
// stay in LDS over the J steps, with the states and couplings beside them, so that after one round
// of loads only the Q rows come from L2.  What bounds it is the chain of 2 J dependent phases
// over a few hundred states, not bytes (states, couplings and h read phase by phase: 115 us for
// 5028 columns and 441 states, 28 us for 320 columns; now 77 and 20 us).
__host__ __device__ inline size_t alias_lds(int32_t S, int32_t J, int32_t CT, int32_t nterm)
{
    return sizeof(double) * (size_t)(J + 1) * (size_t)S * (size_t)CT + sizeof(AliasTerm) * (size_t)nterm +
           sizeof(AliasState) * (size_t)S;
}
__global__ __launch_bounds__(1024) void k_alias_solve(int32_t S, int32_t J, int32_t L, int32_t CT, int32_t cols,
                                                      int32_t split, const AliasState* __restrict__ st, int32_t nterm,
                                                      const AliasTerm* __restrict__ term,
                                                      const double* __restrict__ Q, const int64_t* __restrict__ qoff,
                                                      const double* __restrict__ h, double* __restrict__ r, int64_t ld)
{
    extern __shared__ double alias_mem[];
    double* g = alias_mem;                     // [S][CT]
    double* rr = g + (int64_t)S * CT;          // [J][S][CT]: h_j, then r_j
    AliasTerm* tm = (AliasTerm*)(rr + (int64_t)J * S * CT);
    AliasState* sl = (AliasState*)(tm + nterm);
    const int c = threadIdx.x & (CT - 1), w0 = threadIdx.x / CT, nw = blockDim.x / CT;
    const int col = blockIdx.x * CT + c;
    const bool live = col < cols;
    const int sg = split < 0 ? (int)blockIdx.y : (col < split ? 0 : 1);
    const int64_t row0 = split < 0 ? (int64_t)sg * J * S : 0;
    const double* hc = h + row0 * ld + (live ? col : 0);
    for (int e = threadIdx.x; e < nterm; e += blockDim.x) tm[e] = term[e];
    for (int e = threadIdx.x; e < S; e += blockDim.x) sl[e] = st[e];
    for (int s = w0; s < S; s += nw) {
        const AliasState a = st[s];
        const bool some = live && !(a.m == L && ((a.m + sg) & 1));  // (lmax, odd) has no l: its h is never written
        for (int j = 0; j < J; ++j)
            rr[((int64_t)j * S + s) * CT + c] = some ? hc[((int64_t)J * a.s0 + j * a.na + a.a) * ld] : 0.0;
    }
    __syncthreads();
    for (int j = 0; j < J; ++j) {
        for (int s = w0; s < S; s += nw) {
            const AliasState a = sl[s];
            const int par = (a.m + sg) & 1;
            double v = rr[((int64_t)j * S + s) * CT + c];
            if (!(a.m == L && par == 1)) {
                const double* q = Q + qoff[2 * a.m + par] + (int64_t)a.a * a.na;
                for (int i = 0; i < j; ++i) {
                    const double* qr = q + (int64_t)(j - 1 - i) * a.na * a.na;
                    const double* ri = rr + ((int64_t)i * S + a.s0) * CT + c;
#pragma unroll 4
                    for (int e = 0; e < a.na; ++e) v = fma(qr[e], ri[e * CT], v);
                }
            }
            g[s * CT + c] = v;
        }
        __syncthreads();
        for (int s = w0; s < S; s += nw) {
            const int e0 = sl[s].e0, e1 = sl[s].e1;
            double v = 0.0;
            for (int e = e0; e < e1; ++e) v = fma((col & 1) ? tm[e].cim : tm[e].cre, g[tm[e].s * CT + c], v);
            rr[((int64_t)j * S + s) * CT + c] = v;
        }
        __syncthreads();
    }
    if (!live) return;
    double* rc = r + row0 * ld + col;
    for (int s = w0; s < S; s += nw) {
        const AliasState a = sl[s];
        for (int j = 0; j < J; ++j)
            rc[((int64_t)J * a.s0 + j * a.na + a.a) * ld] = rr[((int64_t)j * S + s) * CT + c];
    }
}
