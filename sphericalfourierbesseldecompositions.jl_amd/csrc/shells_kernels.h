// The mixed path over a common radial basis (radial.cpp): a galaxy adds w B_s(r) to the 10
// basis functions ("shells") s that are non-zero at its r, each shell is a HEALPix map, and
//   a_nlm = inv sum_s gamma_{nl,s} map2alm(D_s)_lm - w_ln map2alm(mask)_lm.
// 160 shell maps replace the 2514 per-(n, l) maps of a call at kmax 0.1, nside 128 (per-map
// scatter, transforms and Legendre steps 5.0 of 5.4 ms there), and everything runs in FP64:
// what is left of the mixed precision is the representation of the splines, 1.3e-8 of their
// largest value, below the FP32 rounding of the records it replaces (6e-8).
#pragma once

constexpr int SH_P = sfb::RADIAL_DEGREE, SH_W = SH_P + 1;  // 10 functions per galaxy
constexpr int SH_PT = 16;                                  // pixels per block: 128-byte rows of a shell
constexpr int SH_NT = 128;                                 // threads, and galaxies staged at a time
constexpr int SH_SUB = SH_NT / SH_PT;

// LDS of a spread block: the tile, the staged values, their first shells and the knots.
__host__ __device__ inline size_t sh_lds(int nc)
{
    return sizeof(double) * ((size_t)nc * SH_PT + (size_t)SH_NT * SH_W + (size_t)(nc + SH_W)) + sizeof(int) * SH_NT;
}

// 1 / d to FP64 rounding: the hardware's estimate and two Newton steps.
__device__ __forceinline__ double rcp64(double d)
{
    double r = __builtin_amdgcn_rcp(d);
    r = fma(fma(-d, r, 1.0), r, r);
    return fma(fma(-d, r, 1.0), r, r);
}

// D[s][p] = sum of w_i B_s(r_i) over the galaxies i of pixel p (r, w ordered by pixel, then
// input), and D[nc][p] = mask[p].  A block owns SH_PT pixels and every shell of them in LDS;
// the galaxies of its pixels are one run of the list.  Two phases per SH_NT galaxies: a thread
// per galaxy finds the interval (binary search over the breaks) and the 10 values (Cox-de Boor
// on the 18 knots around it); then a thread per (pixel, residue of s mod 8) adds its shells'
// values galaxy by galaxy with LDS adds that return nothing, so every sum is in list order and
// no two threads share an address.  r outside the knots takes the end value (the reference's
// boundary extrapolation), NaN passes through.
// Bound: the tile's HBM write (npix nc 8 B, once) and the latency of a block's phases, hence
// small blocks, four to a CU (32 pixels, 256 threads and tabulated reciprocals, two blocks to a
// CU, ran 121 us at N = 1e6, nside 128, nc 159 and 1025 us at 4e6, nside 256, nc 219; now 109
// and 515 us, 2.3 and 2.7 TB/s of the maps' write).
// PARTS: gridDim.y parts, for grids of few pixels with many galaxies each: part y takes its share of
// every block's run and writes its own maps (part y at D + y nc npix), which k_shell_sum adds up (a
// kernel of its own: the shares' divisions cost 4 of 99 us where there is one part).
template <bool PARTS>
__global__ __launch_bounds__(SH_NT) void k_shell_spread(int64_t npix, int32_t nc, const double* __restrict__ knots,
                                                        const int32_t* __restrict__ pstart,
                                                        const double* __restrict__ r_s, const double* __restrict__ w_s,
                                                        const double* __restrict__ mask, double* __restrict__ D,
                                                        double* __restrict__ Dmask)
{
    extern __shared__ double sh_mem[];
    double* tile = sh_mem;                      // [nc][SH_PT]
    double* val = tile + (size_t)nc * SH_PT;    // [SH_W][SH_NT]
    double* t = val + SH_NT * SH_W;             // nc + SH_W knots
    int* first = (int*)(t + nc + SH_W);
    const int nt = nc + SH_W, niv = nc - SH_P, tid = threadIdx.x;
    const int64_t p0 = (int64_t)blockIdx.x * SH_PT;
    const int np = (int)min((int64_t)SH_PT, npix - p0);
    const int pl = tid % SH_PT, sub = tid / SH_PT;
    int g0 = pstart[p0], g1 = pstart[p0 + np];
    if (PARTS) {
        const int64_t b0 = g0, run = g1 - g0;
        g0 = (int)(b0 + run * blockIdx.y / gridDim.y);
        g1 = (int)(b0 + run * (blockIdx.y + 1) / gridDim.y);
    }
    const int a0 = pl < np ? pstart[p0 + pl] : 0, a1 = pl < np ? pstart[p0 + pl + 1] : 0;
    for (int e = tid; e < nc * SH_PT; e += SH_NT) tile[e] = 0.0;
    if (g1 > g0)
        for (int e = tid; e < nt; e += SH_NT) t[e] = knots[e];
    for (int c0 = g0; c0 < g1; c0 += SH_NT) {
        const int n = min(SH_NT, g1 - c0);
        double x = 0.0, wt = 0.0;
        if (tid < n) {
            x = r_s[c0 + tid];
            wt = w_s[c0 + tid];
        }
        __syncthreads();  // the knots (and the last chunk's adds) are done
        if (tid < n) {
            x = x < t[0] ? t[0] : (x > t[nt - 1] ? t[nt - 1] : x);
            int iv = 0;  // the interval: largest iv < niv with t[SH_P + iv] <= x (0 for NaN)
#pragma unroll
            for (int step = 256; step > 0; step >>= 1)
                if (iv + step < niv && t[SH_P + iv + step] <= x) iv += step;
            double kn[2 * SH_P];  // t[iv + 1] .. t[iv + 18]; ti[m] = kn[m + 8] with ti = t + SH_P + iv
#pragma unroll
            for (int a = 0; a < 2 * SH_P; ++a) kn[a] = t[iv + 1 + a];
            double b[SH_W];
            b[0] = wt;
#pragma unroll
            for (int k = 1; k <= SH_P; ++k) {
                double saved = 0.0;
#pragma unroll
                for (int j = 0; j < k; ++j) {
                    const double hi = kn[1 + j + SH_P - 1], lo = kn[1 + j - k + SH_P - 1];
                    const double tmp = b[j] * rcp64(hi - lo);
                    b[j] = fma(hi - x, tmp, saved);
                    saved = (x - lo) * tmp;
                }
                b[k] = saved;
            }
#pragma unroll
            for (int k = 0; k < SH_W; ++k) val[k * SH_NT + tid] = b[k];
            first[tid] = iv;
        }
        __syncthreads();
        const int e1 = min(a1, c0 + n) - c0;
        for (int e = max(a0, c0) - c0; e < e1; ++e) {
            const int iv = first[e];
            const int k = (sub - iv) & (SH_SUB - 1);  // shells iv + k, iv + k + 8 are this thread's
            unsafeAtomicAdd(&tile[(iv + k) * SH_PT + pl], val[k * SH_NT + e]);
            if (k + SH_SUB < SH_W) unsafeAtomicAdd(&tile[(iv + k + SH_SUB) * SH_PT + pl], val[(k + SH_SUB) * SH_NT + e]);
        }
    }
    __syncthreads();
    if (PARTS) D += (int64_t)blockIdx.y * nc * npix;
    if (pl < np)
        for (int s = sub; s < nc; s += SH_SUB) D[(int64_t)s * npix + p0 + pl] = tile[s * SH_PT + pl];
    if ((!PARTS || blockIdx.y == 0) && tid < np) Dmask[p0 + tid] = mask[p0 + tid];
}

// D[e] = sum of the parts' maps in order, e < n = nc npix.  Bound by the parts' bytes.
__global__ __launch_bounds__(256) void k_shell_sum(int64_t n, int32_t parts, const double* __restrict__ part,
                                                   double* __restrict__ D)
{
    const int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= n) return;
    double v = part[e];
#pragma unroll 8
    for (int y = 1; y < parts; ++y) v += part[y * n + e];
    D[e] = v;
}

// The monopoles a_{n00} are differences of nearly equal sums (what a window leaves of a
// full-sky sum), so there the representation's error is taken out: part[n][chunk] = the
// exact spline sums sum_i w_i g_n0(r_i), FP64.  A block takes two n and one share of the galaxies:
// their (y, y'') at the knots in LDS, the segment from the uniform knots (the scatter's rule;
// shells only exist on such knots).  Bound by r and w from L2, once per pair of n, and the two
// random 16-byte reads per value (LDS 68% busy).  352 us at 4e6, 48 n (one n per block and 32-byte
// records: 482 us).
constexpr int SM_N = 2, SM_U = 4;
__global__ __launch_bounds__(1024) void k_shell_mono(int64_t N, int32_t nmx, const double* __restrict__ r,
                                                     const double* __restrict__ w, const MapInfo* __restrict__ maps,
                                                     const double4* __restrict__ rec, const int32_t* __restrict__ qbase,
                                                     double* __restrict__ part)
{
    extern __shared__ double2 sm_y[];  // (y, y'' h^2 / 6) of the first map's knots, then the second's
    __shared__ double red[SM_N][16];
    double s[SM_N], x0[SM_N], ainv[SM_N], top[SM_N];
    const double2* tab[SM_N];
    int off = 0;
#pragma unroll
    for (int v = 0; v < SM_N; ++v) {
        const MapInfo mi = maps[qbase[min((int)blockIdx.y * SM_N + v, nmx - 1)]];
        const double h2 = 1.0 / (6.0 * mi.invdx * mi.invdx);
        for (int j = threadIdx.x; j < mi.nk; j += blockDim.x) {
            const double4 c = rec[mi.koff + j];  // (x, y, y'', a)
            sm_y[off + j] = make_double2(c.y, c.z * h2);
        }
        tab[v] = sm_y + off;
        off += mi.nk;
        s[v] = 0.0;
        x0[v] = -mi.xfirst * mi.invdx;
        ainv[v] = mi.invdx;
        top[v] = (double)(mi.nk - 1);
    }
    __syncthreads();
    const int64_t per = (N + gridDim.x - 1) / gridDim.x;
    const int64_t i0 = (int64_t)blockIdx.x * per, i1 = min(N, i0 + per);
    for (int64_t g0 = i0 + threadIdx.x; g0 < i1; g0 += SM_U * (int64_t)blockDim.x) {
        double x[SM_U], wt[SM_U];
#pragma unroll
        for (int e = 0; e < SM_U; ++e) {  // SM_U galaxies' loads in flight
            const int64_t g = g0 + e * (int64_t)blockDim.x;
            x[e] = g < i1 ? r[g] : 0.0;
            wt[e] = g < i1 ? w[g] : 0.0;
        }
#pragma unroll
        for (int e = 0; e < SM_U; ++e)
#pragma unroll
            for (int v = 0; v < SM_N; ++v) {
                double u = fma(x[e], ainv[v], x0[v]);
                u = u < 0.0 ? 0.0 : (u > top[v] ? top[v] : u);  // the end values outside; NaN stays
                const int i = min((int)u, (int)top[v] - 1);
                const double B = u - (double)i, A = 1.0 - B;
                const double2 lo = tab[v][i], hi = tab[v][i + 1];
                const double g2 = fma(fma(A, A, -1.0) * A, lo.y, fma(B, B, -1.0) * B * hi.y);
                s[v] = fma(wt[e], fma(A, lo.x, fma(B, hi.x, g2)), s[v]);
            }
    }
#pragma unroll
    for (int v = 0; v < SM_N; ++v) {
        for (int o = 32; o > 0; o >>= 1) s[v] += __shfl_xor(s[v], o, 64);
        if ((threadIdx.x & 63) == 0) red[v][threadIdx.x >> 6] = s[v];
    }
    __syncthreads();
    if (threadIdx.x < SM_N && blockIdx.y * SM_N + threadIdx.x < nmx) {
        double v = 0.0;
        for (int i = 0; i < (int)blockDim.x / 64; ++i) v += red[threadIdx.x][i];
        part[((int64_t)blockIdx.y * SM_N + threadIdx.x) * gridDim.x + blockIdx.x] = v;
    }
}

// anlm[n, l, m] = inv sum_s gamma[q][s] Z[l, m][s] - w_ln[l, n] Z[l, m][nc], Z the refined
// coefficients of the shell maps (a layout, row stride ld, shell s at 2 s).  A block takes one
// l and SC_M values of m: their Z rows stay in LDS, and 32 lanes take the maps of this l (lq,
// cnt of them from l0) over gamma by shell, gt[l0 nc + s cnt + j].  A few MB and 0.1 GFLOP:
// latency-bound, 36 us at nside 128 (159 shells, 116 345 coefficients), 112 us at nside 256.  The monopoles (l = 0: a wave per map) add c00 inv (exact sum - sum_s gamma_s
// T_s), T_s = sum_p D_s(p) (at tsum[2 s]): the refinements pass an error of the first
// analysis' monopole to a_00 one to one.
// Aligned so that its 3.2 KB of code lie in one 4 KB page: where the linker had put the loop across two, the
// same instructions took 40 us.
constexpr int SC_M = 8;
__attribute__((aligned(4096))) __global__ __launch_bounds__(256) void k_shell_contract(int32_t L, int32_t nc, const double* __restrict__ gt,
                                                        const int32_t* __restrict__ lstart,
                                                        const int32_t* __restrict__ lq,
                                                        const MapInfo* __restrict__ maps,
                                                        const int64_t* __restrict__ out_base,
                                                        const int64_t* __restrict__ aoff, int64_t ld,
                                                        const double* __restrict__ a, const double* __restrict__ wln,
                                                        const double* __restrict__ tsum,
                                                        const double* __restrict__ mono, int32_t nch, double c00,
                                                        double inv, double* __restrict__ out,
                                                        int32_t* __restrict__ flag)
{
    extern __shared__ double2 sc_z[];  // [SC_M][nc + 1]
    const int l = blockIdx.y, m0 = blockIdx.x * SC_M;
    if (m0 > l) return;
    const int l0 = lstart[l], cnt = lstart[l + 1] - l0;
    const double* g = gt + (int64_t)l0 * nc;
    if (l == 0) {
        const int lane = threadIdx.x & 63;
        const double* z = a + aoff[0] * ld;
        for (int j = threadIdx.x >> 6; j < cnt; j += (int)blockDim.x >> 6) {
            const int q = lq[l0 + j], n = maps[q].n - 1;
            double re = 0.0, im = 0.0, ex = 0.0;
            for (int s = lane; s < nc; s += 64) {
                const double gs = g[(int64_t)s * cnt + j];
                re = fma(gs, z[2 * s], re);
                im = fma(gs, z[2 * s + 1], im);
                ex = fma(-gs, tsum[2 * s], ex);
            }
            for (int c = lane; c < nch; c += 64) ex += mono[(int64_t)n * nch + c];
            for (int o = 32; o > 0; o >>= 1) {
                re += __shfl_xor(re, o, 64);
                im += __shfl_xor(im, o, 64);
                ex += __shfl_xor(ex, o, 64);
            }
            if (lane == 0) {
                const double wl = wln[(int64_t)n * (L + 1)];
                re = inv * re - wl * z[2 * nc] + c00 * inv * ex;
                im = inv * im - wl * z[2 * nc + 1];
                out[2 * out_base[q]] = re;
                out[2 * out_base[q] + 1] = im;
                if (!isfinite(re) || !isfinite(im)) atomicOr(flag, 1);
            }
        }
        return;
    }
    const int nm = min(SC_M, l + 1 - m0), nz = nc + 1;
    for (int e = threadIdx.x; e < nm * nz; e += blockDim.x) {
        const int i = e / nz, s = e - i * nz, m = m0 + i;
        const int par = (l - m) & 1, j = (l - m) >> 1;
        sc_z[i * nz + s] = *(const double2*)(a + (aoff[m * 2 + par] + j) * ld + 2 * s);
    }
    __syncthreads();
    const int i = threadIdx.x >> 5;
    if (i >= nm) return;
    const double2* z = sc_z + i * nz;
    for (int j = threadIdx.x & 31; j < cnt; j += 32) {
        double re = 0.0, im = 0.0;
#pragma unroll 8
        for (int s = 0; s < nc; ++s) {
            const double gs = g[(int64_t)s * cnt + j];
            re = fma(gs, z[s].x, re);
            im = fma(gs, z[s].y, im);
        }
        const int q = lq[l0 + j];
        const double wl = wln[(int64_t)(maps[q].n - 1) * (L + 1) + l];
        re = inv * re - wl * z[nc].x;
        im = inv * im - wl * z[nc].y;
        const int64_t o = 2 * (out_base[q] + m0 + i);
        out[o] = re;
        out[o + 1] = im;
        if (!isfinite(re) || !isfinite(im)) atomicOr(flag, 1);
    }
}
