// The mixed path over a common radial basis (radial.cpp): a galaxy adds w B_s(r) to the 10
// basis functions ("shells") s that are non-zero at its r, each shell is a HEALPix map, and
//   a_nlm = inv sum_s gamma_{nl,s} map2alm(D_s)_lm - w_ln map2alm(mask)_lm.
// 160 shell maps replace the 2514 per-(n, l) maps of a call at kmax 0.1, nside 128 (per-map
// scatter, transforms and Legendre steps 5.0 of 5.4 ms there), and everything runs in FP64:
// what is left of the mixed precision is the representation of the splines, 1.3e-8 of their
// largest value, below the FP32 rounding of the records it replaces (6e-8).
#pragma once

constexpr int SH_P = sfb::RADIAL_DEGREE, SH_W = SH_P + 1;  // 10 functions per galaxy
constexpr int SH_PT = 32;                                  // pixels per block
constexpr int SH_CH = 192;                                 // galaxies staged at a time
constexpr int SH_NT = 256;
constexpr int SH_SUB = SH_NT / SH_PT;

// LDS of a spread block: the tile, the staged values, their first shells, the knots and the
// reciprocal knot differences.
__host__ __device__ inline size_t sh_lds(int nc)
{
    return sizeof(double) * ((size_t)nc * SH_PT + (size_t)SH_CH * SH_W + (size_t)(nc + SH_W) * (SH_P + 1)) +
           sizeof(int) * SH_CH;
}

// D[s][p] = sum of w_i B_s(r_i) over the galaxies i of pixel p (ordered by pixel, then input),
// and D[nc][p] = mask[p].  A block owns SH_PT pixels and every shell of them in LDS: the
// galaxies of its pixels are one run of the sorted list.  Two phases per SH_CH galaxies: a
// thread per galaxy finds the interval (binary search over the breaks) and the 10 values
// (Cox-de Boor with tabulated reciprocals, no divisions); then a thread per (pixel, residue of
// s mod 8) adds its shells' values galaxy by galaxy, so every sum is in list order and no two
// threads share an address.  r outside the knots takes the end value (the reference's boundary
// extrapolation), NaN passes through.  Bound: LDS latency of the adds and the tile's HBM write
// (npix nc 8 B once; a row of a tile is 256 contiguous bytes).
template <bool UNIT>
__global__ __launch_bounds__(SH_NT) void k_shell_spread(int64_t npix, int32_t nc, const double* __restrict__ knots,
                                                        const double* __restrict__ recip,
                                                        const int32_t* __restrict__ pstart,
                                                        const uint32_t* __restrict__ idx,
                                                        const double* __restrict__ rtp, const double* __restrict__ w,
                                                        const double* __restrict__ mask, double* __restrict__ D)
{
    extern __shared__ double sh_mem[];
    double* tile = sh_mem;                      // [nc][SH_PT]
    double* val = tile + (size_t)nc * SH_PT;    // [SH_CH][SH_W]
    double* t = val + SH_CH * SH_W;             // nc + SH_W knots
    double* rc = t + nc + SH_W;                 // [SH_P][nc + SH_W]: 1 / (t[i+k] - t[i]) at (k-1, i)
    int* first = (int*)(rc + (size_t)SH_P * (nc + SH_W));
    const int nt = nc + SH_W, niv = nc - SH_P;
    const int64_t p0 = (int64_t)blockIdx.x * SH_PT;
    const int np = (int)min((int64_t)SH_PT, npix - p0);
    for (int e = threadIdx.x; e < nc * SH_PT; e += SH_NT) tile[e] = 0.0;
    const int g0 = pstart[p0], g1 = pstart[p0 + np];
    if (g1 > g0) {
        for (int e = threadIdx.x; e < nt; e += SH_NT) t[e] = knots[e];
        for (int e = threadIdx.x; e < SH_P * nt; e += SH_NT) rc[e] = recip[e];
    }
    const int pl = threadIdx.x % SH_PT, sub = threadIdx.x / SH_PT;
    const int a0 = pl < np ? pstart[p0 + pl] : 0, a1 = pl < np ? pstart[p0 + pl + 1] : 0;
    __syncthreads();
    for (int c0 = g0; c0 < g1; c0 += SH_CH) {
        const int n = min(SH_CH, g1 - c0);
        if ((int)threadIdx.x < n) {
            const int64_t gi = idx[c0 + threadIdx.x];
            double x = rtp[3 * gi];
            const double wt = UNIT ? 1.0 : w[gi];
            x = x < t[0] ? t[0] : (x > t[nt - 1] ? t[nt - 1] : x);
            int iv = 0;  // the interval: largest iv < niv with t[SH_P + iv] <= x (0 for NaN)
            for (int step = 256; step > 0; step >>= 1)
                if (iv + step < niv && t[SH_P + iv + step] <= x) iv += step;
            const double* ti = t + SH_P + iv;
            double b[SH_W];
            b[0] = wt;
#pragma unroll
            for (int k = 1; k <= SH_P; ++k) {
                double saved = 0.0;
#pragma unroll
                for (int j = 0; j < k; ++j) {
                    // right_{j+1} + left_{k-j} = t[i+1+j] - t[i+1+j-k]
                    const double tmp = b[j] * rc[(k - 1) * nt + (SH_P + iv + 1 + j - k)];
                    b[j] = fma(ti[1 + j] - x, tmp, saved);
                    saved = (x - ti[1 + j - k]) * tmp;
                }
                b[k] = saved;
            }
#pragma unroll
            for (int k = 0; k < SH_W; ++k) val[threadIdx.x * SH_W + k] = b[k];
            first[threadIdx.x] = iv;
        }
        __syncthreads();
        const int e1 = min(a1, c0 + n) - c0;
        for (int e = max(a0, c0) - c0; e < e1; ++e) {
            const int iv = first[e];
            const int k = (sub - iv) & (SH_SUB - 1);  // shells iv + k, iv + k + 8 are this thread's
            tile[(iv + k) * SH_PT + pl] += val[e * SH_W + k];
            if (k + SH_SUB < SH_W) tile[(iv + k + SH_SUB) * SH_PT + pl] += val[e * SH_W + k + SH_SUB];
        }
        __syncthreads();
    }
    for (int e = threadIdx.x; e < nc * SH_PT; e += SH_NT) {
        const int s = e / SH_PT, p = e % SH_PT;
        if (p < np) D[(int64_t)s * npix + p0 + p] = tile[e];
    }
    if (mask && (int)threadIdx.x < np) D[(int64_t)nc * npix + p0 + threadIdx.x] = mask[p0 + threadIdx.x];
}

// anlm[n, l, m] = inv sum_s gamma[q][s] Z[l, m][s] - w_ln[l, n] Z[l, m][nc], Z the refined
// coefficients of the shell maps (a layout, row stride ld, shell s at 2 s).  A block takes one
// l and SC_M values of m: their Z rows stay in LDS, and a thread sums one (n, m) over gamma's
// row, whose columns it shares with the other m.  A few MB and 0.1 GFLOP: latency-bound.
constexpr int SC_M = 8;
__global__ __launch_bounds__(256) void k_shell_contract(int32_t nmax, int32_t L, int32_t nc,
                                                        const double* __restrict__ gamma,
                                                        const int32_t* __restrict__ qbase,
                                                        const int32_t* __restrict__ lmaxn,
                                                        const int64_t* __restrict__ out_base,
                                                        const int64_t* __restrict__ aoff, int64_t ld,
                                                        const double* __restrict__ a, const double* __restrict__ wln,
                                                        double inv, double* __restrict__ out,
                                                        int32_t* __restrict__ flag)
{
    extern __shared__ double2 sc_z[];  // [SC_M][nc + 1]
    const int l = blockIdx.y, m0 = blockIdx.x * SC_M;
    if (m0 > l) return;
    const int nm = min(SC_M, l + 1 - m0), nz = nc + 1;
    for (int e = threadIdx.x; e < nm * nz; e += blockDim.x) {
        const int i = e / nz, s = e - i * nz, m = m0 + i;
        const int par = (l - m) & 1, j = (l - m) >> 1;
        sc_z[i * nz + s] = *(const double2*)(a + (aoff[m * 2 + par] + j) * ld + 2 * s);
    }
    __syncthreads();
    for (int e = threadIdx.x; e < nmax * SC_M; e += blockDim.x) {
        const int n = e / SC_M, i = e % SC_M;
        if (i >= nm || l > lmaxn[n]) continue;
        const int q = qbase[n] + l;
        const double* g = gamma + (int64_t)q * nc;
        const double2* z = sc_z + i * nz;
        double re = 0.0, im = 0.0;
        for (int s = 0; s < nc; ++s) {
            re = fma(g[s], z[s].x, re);
            im = fma(g[s], z[s].y, im);
        }
        const double wl = wln[(int64_t)n * (L + 1) + l];
        re = inv * re - wl * z[nc].x;
        im = inv * im - wl * z[nc].y;
        const int64_t o = 2 * (out_base[q] + m0 + i);
        out[o] = re;
        out[o + 1] = im;
        if (!isfinite(re) || !isfinite(im)) atomicOr(flag, 1);
    }
}

// The monopoles a_{n00} are differences of nearly equal sums (what a window leaves of a
// full-sky sum), so there the representation's error is taken out: part[n][chunk] = the
// exact spline sums sum_i w_i g_n0(r_i) of the galaxies in input order, FP64 records in LDS and
// the segment from the uniform knots (the scatter's rule, shells only exist on such knots).
// blockIdx = (chunk, n).  Bound by the random 32-byte record reads from LDS.
template <bool UNIT>
__global__ __launch_bounds__(512) void k_shell_mono(int64_t N, const double* __restrict__ r, const double* __restrict__ w,
                                                    const MapInfo* __restrict__ maps, const double4* __restrict__ rec4,
                                                    const int32_t* __restrict__ qbase, double* __restrict__ part)
{
    extern __shared__ double4 sm_rec[];  // slot 0: below the knots, 1 .. nk - 1: segments, nk: above
    __shared__ double red[8];
    const int q = qbase[blockIdx.y];
    const MapInfo mi = maps[q];
    const int nk = mi.nk;
    const double4* rq = rec4 + mi.koff + q;
    for (int j = threadIdx.x; j < nk - 1; j += blockDim.x) sm_rec[j + 1] = rq[j];
    if (threadIdx.x == 0) sm_rec[0] = rq[nk - 1];
    if (threadIdx.x == 1) sm_rec[nk] = rq[nk];
    __syncthreads();
    const double ainv = mi.invdx, c0 = -mi.xfirst * mi.invdx, top = (double)(nk - 1);
    const int64_t per = (N + gridDim.x - 1) / gridDim.x;
    const int64_t i0 = (int64_t)blockIdx.x * per, i1 = min(N, i0 + per);
    double s = 0.0;
    constexpr int U = 4;
    for (int64_t g0 = i0 + threadIdx.x; g0 < i1; g0 += U * (int64_t)blockDim.x) {
        double x[U], wt[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int64_t g = g0 + u * (int64_t)blockDim.x;
            x[u] = g < i1 ? r[g] : 0.0;
            wt[u] = g < i1 ? (UNIT ? 1.0 : w[g]) : 0.0;
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            if (g0 + u * (int64_t)blockDim.x >= i1) break;
            const double v = fma(x[u], ainv, c0), fl = floor(v);
            const int slot = (int)fmin(fmax(fl, -1.0), top) + 1;
            const double t = __builtin_isinf(v) ? 0.0 : v - fl;
            const double4 c = sm_rec[slot];  // (d, c, b, a); zero slopes outside the knots
            s = fma(wt[u], fma(t, fma(t, fma(t, c.w, c.z), c.y), c.x), s);
        }
    }
    for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o, 64);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = s;
    __syncthreads();
    if (threadIdx.x == 0) {
        double v = 0.0;
        for (int i = 0; i < (int)blockDim.x / 64; ++i) v += red[i];
        part[(int64_t)blockIdx.y * gridDim.x + blockIdx.x] = v;
    }
}

// a_{n00} += inv dOmega Y_00 (exact sum - sum_s gamma_s T_s), T_s = sum_p D_s(p) = the m = 0
// ring sums of shell s over the ring pairs.  (The refinements pass an error of the first
// analysis' monopole to a_00 one to one: (A S)_{00,00} = 1.)
__global__ __launch_bounds__(256) void k_shell_monofix(int32_t nc, int32_t K, int32_t nch, const double* __restrict__ X,
                                                       int64_t ld, const double* __restrict__ gamma,
                                                       const int32_t* __restrict__ qbase,
                                                       const int64_t* __restrict__ out_base,
                                                       const double* __restrict__ part, double scale,
                                                       double* __restrict__ out, int32_t* __restrict__ flag)
{
    __shared__ double red[4];
    const int n = blockIdx.x, q = qbase[n];
    double f = 0.0;
    for (int s = threadIdx.x; s < nc; s += blockDim.x) {
        double T = 0.0;
        for (int k = 0; k < K; ++k) T += X[(int64_t)k * ld + 2 * s];
        f = fma(gamma[(int64_t)q * nc + s], T, f);
    }
    for (int o = 32; o > 0; o >>= 1) f += __shfl_xor(f, o, 64);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = f;
    __syncthreads();
    if (threadIdx.x != 0) return;
    double S = 0.0;
    for (int c = 0; c < nch; ++c) S += part[(int64_t)n * nch + c];
    const int64_t o = 2 * out_base[q];
    const double a = out[o] + scale * (S - (red[0] + red[1] + red[2] + red[3]));
    out[o] = a;
    if (!isfinite(a)) atomicOr(flag, 1);
}
