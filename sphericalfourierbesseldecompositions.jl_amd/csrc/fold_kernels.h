// The FP64 path per (n, l) map with the two hemispheres folded into one.
//
// A map of one l only needs the ring sums F_N(m) + (-1)^{l+m} F_S(m), and (-1)^m is a rotation of
// the southern ring by pi, i.e. by npr/2 pixels (npr is a multiple of 4 and both rings of a
// pair share their phase).  So the scatter sums the folded map
//   delta~(f) = delta(f) + (-1)^l delta(mirror pixel rotated by pi),  f north or equator,
// one real DFT per ring pair gives X_m, and with the refinements folded into the analysis table
// (sht_direct_kernels.h) only the row l' = l is needed:
//   a_lm = sum_k (dOmega Lam P_J)[k][l] X_m[k] + (aliasing correction).
// Half the map bytes and DFTs, a quarter of the ring coefficients (one parity, m <= l), and a
// dot product per coefficient in place of a product for every l' (70 at lmax 140).
//
// Columns: maps ordered by l parity, then l descending, so the maps with l >= m are a prefix
// of each parity's run for every m, and neighbouring columns share l.
#pragma once

struct FoldCol {
    int32_t q, l;     // the map and its l
    int32_t mtop;     // X kept for m <= mtop: max(l, largest aliasing m)
    int64_t out;      // index of a_{nl0}
};
// Per m: the analysis tables of the two l parities (block (m, par = (l + m) & 1)).
struct FoldM {
    int64_t lam[2], v[2];  // offsets of [K][nb] and [J na][nb] tables, by l parity
    int32_t nb[2], cnt[2]; // l per block; columns with l >= m, by l parity
    int32_t kc, s0, na, pad;
};

// The separable window of every slice lane, folded: even l in the first half, odd in the second.
__global__ void k_slice_win_fold(int64_t nlane, int64_t npf, const int2* __restrict__ pinfo,
                                 const int32_t* __restrict__ south, const double* __restrict__ win_a,
                                 double* __restrict__ pwin)
{
    const int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= nlane) return;
    double n = 0.0, s = 0.0;
    if (e < npf) {
        const int p = pinfo[e].x;
        n = win_a[p];
        s = south[p] >= 0 ? win_a[south[p]] : 0.0;
    }
    pwin[e] = n + s;
    pwin[nlane + e] = n - s;
}

// X_kf into every m = kf (mod npr) and, conjugated, m = -kf (mod npr), m <= Lm, with the ring
// phase (store_folded for one value).
template <bool TWPAD, typename TW>
__device__ __forceinline__ void store_fold1(double* __restrict__ X, int64_t ld, int32_t K, int32_t k, int npr, int shift,
                                            const TW* __restrict__ twr, int Lm, int kf, int c, double xr, double xi)
{
    const unsigned un2 = 2u * (unsigned)npr, dph = ((unsigned)npr * (unsigned)shift) % un2;
    for (int fam = 0; fam < 2; ++fam) {
        if (fam == 1 && (kf == 0 || 2 * kf == npr)) break;
        const int m0 = fam ? npr - kf : kf;
        unsigned ph = ((unsigned)m0 * (unsigned)shift) % un2;
        for (int m = m0; m <= Lm; m += npr, ph = min(ph + dph, ph + dph - un2)) {
            const TW w = twr[TWPAD ? twpad((int)ph) : (int)ph];
            double2 v;
            cmul_conj(xr, fam ? -xi : xi, (double)w.x, (double)w.y, v.x, v.y);
            *(double2*)(X + ((int64_t)m * K + k) * ld + 2 * c) = v;
        }
    }
}

// Equatorial ring pairs of folded maps: k_phi_fft with one sequence per map (TQ columns per
// block).  X[(m K + k) ld + 2 c].  Bound: FP64 butterflies (VALU 49% busy) and their LDS passes (42%).
// nside 128, 2514 maps: 561 us (unfolded, two sequences per map: 1.10 ms).
__global__ __launch_bounds__(512) void k_phi_fft_fold(const double* __restrict__ delta, int64_t npf, int32_t ncol,
                                                      int64_t ld, int32_t K, const RingDev* __restrict__ rings,
                                                      const double2* __restrict__ tw, double* __restrict__ X,
                                                      int32_t TQ, int32_t k0, int32_t logM,
                                                      const int32_t* __restrict__ mall,
                                                      const uint32_t* __restrict__ perm,
                                                      const FoldCol* __restrict__ cols, int32_t nring, int32_t ntile)
{
    extern __shared__ double2 zf_raw[];
    double2* zs = zf_raw;
    const int b = blockIdx.x, loc = b >> 3;
    const int unit = (((loc >> 3) << 3) + (b & 7)) * 8 + (loc & 7);  // runs of ring pairs per XCD, as k_phi_fft
    if (unit >= nring * ntile) return;
    const int k = k0 + unit % nring;
    const int c0 = (unit / nring) * TQ;
    const RingDev Rg = rings[k];
    const int N = Rg.npr, M = N >> 1, Mp = (int)fft_plen(M, sizeof(double));
    const int ltq = __ffs(TQ) - 1;
    const double2* twg = tw + Rg.tw_off;
    double2* twr = zs + TQ * Mp;
    constexpr int TQM = 8;
    int64_t base[TQM];
#pragma unroll
    for (int ql = 0; ql < TQM; ++ql) base[ql] = ql < TQ ? (int64_t)cols[min(c0 + ql, ncol - 1)].q * npf : 0;
    for (int e = threadIdx.x; e < M; e += blockDim.x) {
        const int rj = (int)(__brev((unsigned)e) >> (32 - logM));
        uint2 sl = make_uint2((uint32_t)(Rg.start_n + 2 * e), (uint32_t)(Rg.start_n + 2 * e + 1));
        if (perm) sl = *(const uint2*)(perm + Rg.start_n + 2 * e);
        double re[TQM], im[TQM];
#pragma unroll
        for (int ql = 0; ql < TQM; ++ql)
            if (ql < TQ) {
                re[ql] = delta[base[ql] + sl.x];
                im[ql] = delta[base[ql] + sl.y];
            }
#pragma unroll
        for (int ql = 0; ql < TQM; ++ql)
            if (ql < TQ) zs[ql * Mp + fpad<double>(rj)] = make_double2(re[ql], im[ql]);
    }
    for (int e = threadIdx.x; e <= N; e += blockDim.x) twr[twpad(e)] = twg[e];
    __syncthreads();
    fft_passes<double>(zs, TQ, M, Mp, N, logM, twr);
    const int Lk = mall[k];
    const int nm = min(Lk, M);
    for (int e = threadIdx.x; e < TQ * (nm + 1); e += blockDim.x) {
        const int m = e >> ltq, ql = e & (TQ - 1), c = c0 + ql;
        if (c >= ncol) continue;
        const int top = min(Lk, cols[c].mtop);
        if (m > top && N - m > top) continue;
        const double2* z = zs + ql * Mp;
        const double2 zm = z[fpad<double>(m & (M - 1))], zc = z[fpad<double>((M - m) & (M - 1))];
        const double er = 0.5 * (zm.x + zc.x), ei = 0.5 * (zm.y - zc.y);
        const double orr = 0.5 * (zm.y + zc.y), oi = -0.5 * (zm.x - zc.x);
        const double2 w = twr[twpad(2 * m)];
        const double xr = fma(w.x, orr, fma(w.y, oi, er)), xi = fma(w.x, oi, fma(-w.y, orr, ei));
        store_fold1<true>(X, ld, K, k, N, Rg.shift, twr, top, m, c, xr, xi);
    }
}

// Polar ring pairs of folded maps: k_phi_polar4 with one sequence per map (twice its maps per
// block for the same tiles).  Bound: VALU (57%: gathers, indexes, X stores) around the MFMA product, which
// takes even and odd sample parts (p4_product_sym).  nside 128, 2514 maps: 501 us (597 with the
// whole product, 1.20 ms unfolded).
template <int MTWMAX>
__global__ __launch_bounds__(256) void k_phi_polar4_fold(const double* __restrict__ delta, int64_t npf, int32_t ncol,
                                                         int64_t ld, int32_t K, const RingDev* __restrict__ rings,
                                                         const double2* __restrict__ tw, double* __restrict__ X,
                                                         const int32_t* __restrict__ mall,
                                                         const uint32_t* __restrict__ perm,
                                                         const FoldCol* __restrict__ cols, int32_t nring, int32_t ntile)
{
    extern __shared__ double2 pf_raw[];
    const int b = blockIdx.x, loc = b >> 3;
    const int unit = (((loc >> 2) << 3) + (b & 7)) * 4 + (loc & 3);
    if (unit >= nring * ntile) return;
    const int k = unit % nring;
    const RingDev Rg = rings[k];
    const int npr = Rg.npr, n2 = 2 * npr, ni = npr >> 2, nu = ni / 2 + 1;
    const int tq = p4_tq(ni, MTWMAX), TQ = 2 * tq;
    const int c0 = (unit / nring) * TQ;
    if (c0 >= ncol) return;
    const int ld1 = p4_ld(ni, (int)sizeof(double));
    const double2* twl = tw + Rg.tw_off;
    double* D = (double*)pf_raw;               // [TQ][ld1]: samples, then Y
    double2* twi = (double2*)(D + TQ * ld1);   // (cos, -sin)(2 pi v/i)
    for (int e = threadIdx.x; e < ni; e += blockDim.x) twi[e] = make_double2(twl[8 * e].x, -twl[8 * e].y);
    const int nv = npr >> 2;
    for (int e0 = threadIdx.x; e0 < TQ * nv; e0 += PH_UL * blockDim.x) {  // PH_UL fours in flight
        double4 v[PH_UL];
        uint4 sl[PH_UL];
#pragma unroll
        for (int u = 0; u < PH_UL; ++u) {
            const int e = min(e0 + u * (int)blockDim.x, TQ * nv - 1), p = (int)Rg.start_n + 4 * (e % nv);
            sl[u] = make_uint4(p, p + 1, p + 2, p + 3);
            if (perm) sl[u] = *(const uint4*)(perm + p);
        }
#pragma unroll
        for (int u = 0; u < PH_UL; ++u) {
            const int e = min(e0 + u * (int)blockDim.x, TQ * nv - 1);
            const double* dq = delta + (int64_t)cols[min(c0 + e / nv, ncol - 1)].q * npf;
            v[u] = make_double4(dq[sl[u].x], dq[sl[u].y], dq[sl[u].z], dq[sl[u].w]);
        }
#pragma unroll
        for (int u = 0; u < PH_UL; ++u) {
            const int e = e0 + u * blockDim.x;
            if (e < TQ * nv) *(double4*)(D + (e / nv) * ld1 + 4 * (e % nv)) = v[u];
        }
    }
    __syncthreads();
    p4_fold_samples(D, TQ, ni, ld1);
    __syncthreads();
    p4_product_tiles<MTWMAX>(D, twi, ni, ld1, tq);
    __syncthreads();
    const int Lk = mall[k];
    const int nkf = min(Lk, npr / 2) + 1;
    for (int e = threadIdx.x; e < TQ * nkf; e += blockDim.x) {
        const int ql = e % TQ, kf = e / TQ, c = c0 + ql;
        if (c >= ncol) continue;
        const int top = min(Lk, cols[c].mtop);
        if (kf > top && npr - kf > top) continue;
        int u = kf % ni;
        const bool cj = u > ni / 2;
        if (cj) u = ni - u;
        const double2* Y = (const double2*)(D + ql * ld1);
        double sr = 0.0, si = 0.0;
        unsigned iw = 0;
        const unsigned st2 = 2u * (unsigned)kf, un2 = (unsigned)n2;
#pragma unroll
        for (int ss = 0; ss < 4; ++ss, iw = min(iw + st2, iw + st2 - un2)) {
            const double2 w = twl[iw];
            double2 y = Y[ss * nu + u];
            if (cj) y.y = -y.y;
            sr = fma(y.x, w.x, fma(y.y, w.y, sr));
            si = fma(y.y, w.x, fma(-y.x, w.y, si));
        }
        store_fold1<false>(X, ld, K, k, npr, Rg.shift, twl, top, kf, c, sr, si);
    }
}

// a_lm of every map and m <= l from the ring coefficients and the aliasing steps' values r, and
// its place in the a_nlm vector.  A block takes one m, one l parity and 64 columns, its four waves
// a quarter of the ring pairs each (eight rows of X in flight per thread).  Bound: X read once
// (16 B per column, m <= l and ring pair).  nside 128, 2514 maps: 125 us; a product for every l' of
// each map in its place ran 680 us.
__global__ __launch_bounds__(256) void k_fold_rows(int32_t K, int32_t J, int64_t ld, const FoldM* __restrict__ fm,
                                                   const FoldCol* __restrict__ cols, int32_t neven,
                                                   const double* __restrict__ lam, const double* __restrict__ ZB,
                                                   const double* __restrict__ X, const double* __restrict__ r,
                                                   double* __restrict__ out, int32_t* __restrict__ flag)
{
    __shared__ double2 red[4][64];
    const int m = blockIdx.z, pi = blockIdx.y, lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const FoldM M = fm[m];
    const int i = blockIdx.x * 64 + lane;
    if ((int)blockIdx.x * 64 >= M.cnt[pi]) return;
    const bool live = i < M.cnt[pi];
    const int c = (pi ? neven : 0) + min(i, M.cnt[pi] - 1);
    const FoldCol C = cols[c];
    const int j = (C.l - m) >> 1, nb = M.nb[pi];
    const double* t = lam + M.lam[pi] + j;
    const double2* x = (const double2*)(X + (int64_t)m * K * ld) + c;
    const int64_t ld2 = ld >> 1;
    const int per = (K - M.kc + 3) / 4, k0 = M.kc + wv * per, k1 = min(K, k0 + per);
    double re = 0.0, im = 0.0;
#pragma unroll 8
    for (int k = k0; k < k1; ++k) {
        const double2 v = x[(int64_t)k * ld2];
        const double w = t[(int64_t)k * nb];
        re = fma(w, v.x, re);
        im = fma(w, v.y, im);
    }
    const double2* rr = (const double2*)(r + (int64_t)J * M.s0 * ld) + c;
    const double* z = ZB + M.v[pi] + j;
#pragma unroll 4
    for (int h = wv; h < J * M.na; h += 4) {
        const double2 v = rr[(int64_t)h * ld2];
        const double w = z[(int64_t)h * nb];
        re = fma(w, v.x, re);
        im = fma(w, v.y, im);
    }
    red[wv][lane] = make_double2(re, im);
    __syncthreads();
    if (wv || !live) return;
#pragma unroll
    for (int u = 1; u < 4; ++u) {
        re += red[u][lane].x;
        im += red[u][lane].y;
    }
    const int64_t o = 2 * (C.out + m);
    out[o] = re;
    out[o + 1] = im;
    if (!isfinite(re) || !isfinite(im)) atomicOr(flag, 1);
}

// ---- the transposed direction (adjoint): cotangent -> folded delta-bar maps ------------------

// h of the aliasing steps from the cotangent b = D_half c: h[s, j] = (U_j^T b)[state], b only at
// row l.  Zero where m > l.  13 us at nside 128 (h written once; launch and latency).
__global__ __launch_bounds__(256) void k_fold_coth(int32_t J, int32_t ncol, int64_t ld, const FoldM* __restrict__ fm,
                                                   const FoldCol* __restrict__ cols, int32_t neven,
                                                   const double* __restrict__ UB, const double* __restrict__ cot,
                                                   double* __restrict__ h)
{
    const int m = blockIdx.y, lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const FoldM M = fm[m];
    const int c = blockIdx.x * 64 + lane;
    if (c >= ncol || M.na == 0) return;
    const FoldCol C = cols[c];
    const int pi = c >= neven, H = J * M.na;
    double2 b = make_double2(0.0, 0.0);
    if (m <= C.l) {
        b = *(const double2*)(cot + 2 * (C.out + m));
        if (m) {
            b.x *= 0.5;
            b.y *= 0.5;
        } else {
            b.y = 0.0;  // Im a_l0 vanishes identically
        }
    }
    const double* u = UB + M.v[pi] + (int64_t)((C.l - m) >> 1) * H;
    double2* hh = (double2*)(h + (int64_t)J * M.s0 * ld) + c;
    for (int e = wv; e < H; e += 4) {
        const double w = m <= C.l ? u[e] : 0.0;
        hh[(int64_t)e * (ld >> 1)] = make_double2(w * b.x, w * b.y);
    }
}

// X_m[k] = (Lam P_J)[k][l] b_m + sum_h GZ[h][k] r_h, m <= mtop.  A block takes one m, 64 columns of one
// l parity and 32 ring pairs, a wave 8 of them: the aliasing tables' entries are wave-uniform
// (scalar loads; per-lane loads of them ran 548 us at nside 128).  Bound: X written once.
// nside 128, 2514 maps, FP32 X: 221 us (synthesis of every l' by products: 1.69 ms with the refinement).
template <typename R>
__global__ __launch_bounds__(256) void k_fold_synth(int32_t K, int32_t J, int32_t ncol, int64_t ld,
                                                    const FoldM* __restrict__ fm, const FoldCol* __restrict__ cols,
                                                    int32_t neven, const double* __restrict__ lamPT,
                                                    const double* __restrict__ GZ, const int64_t* __restrict__ gzoff,
                                                    const double* __restrict__ r, const double* __restrict__ cot,
                                                    R* __restrict__ X)
{
    const int m = blockIdx.z, lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const FoldM M = fm[m];
    const int te = (neven + 63) >> 6;  // tiles of the even maps, then of the odd ones
    const int pi = (int)blockIdx.x >= te;
    const int c = (pi ? neven + ((int)blockIdx.x - te) * 64 : (int)blockIdx.x * 64) + lane;
    const int k0 = blockIdx.y * 32 + wv * 8;
    if (c >= (pi ? ncol : neven) || k0 + 8 <= M.kc || k0 >= K) return;
    const FoldCol C = cols[c];
    if (m > C.mtop) return;
    double re[8], im[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) re[u] = im[u] = 0.0;
    if (m <= C.l) {
        double2 b = *(const double2*)(cot + 2 * (C.out + m));
        if (m) {
            b.x *= 0.5;
            b.y *= 0.5;
        } else {
            b.y = 0.0;
        }
        const double* t = lamPT + M.lam[pi] + (int64_t)((C.l - m) >> 1) * K + k0;
#pragma unroll
        for (int u = 0; u < 8; ++u)
            if (k0 + u < K) {
                re[u] = t[u] * b.x;
                im[u] = t[u] * b.y;
            }
    }
    if (M.na > 0 && M.nb[pi] > 0) {  // ((lmax, odd) has no l, hence no table)
        const double2* rr = (const double2*)(r + (int64_t)J * M.s0 * ld) + c;
        const double* gz = GZ + gzoff[2 * m + ((m + pi) & 1)] + k0;
        const int ku = min(8, K - k0);  // (K is even; 8 except on grids of fewer ring pairs)
        for (int e = 0; e < J * M.na; ++e) {
            const double2 v = rr[(int64_t)e * (ld >> 1)];
            const double* w = gz + (int64_t)e * K;
            if (ku == 8) {
#pragma unroll
                for (int u = 0; u < 8; ++u) {
                    re[u] = fma(w[u], v.x, re[u]);
                    im[u] = fma(w[u], v.y, im[u]);
                }
            } else {
#pragma unroll
                for (int u = 0; u < 8; ++u)
                    if (u < ku) {
                        re[u] = fma(w[u], v.x, re[u]);
                        im[u] = fma(w[u], v.y, im[u]);
                    }
            }
        }
    }
    typedef typename Vec2T<R>::T R2;
#pragma unroll
    for (int u = 0; u < 8; ++u)
        if (k0 + u < K && k0 + u >= M.kc) {
            R2 v;
            v.x = (R)re[u];
            v.y = (R)im[u];
            *(R2*)(X + ((int64_t)m * K + k0 + u) * ld + 2 * c) = v;
        }
}

// Equatorial ring pairs, inverse: k_phi_ifft with one sequence per map; out[q][f] in pixel order.
// Bound as k_phi_fft_fold.  nside 128, 2514 maps, FP32: 415 us (unfolded 1.09 ms).
template <typename R>
__global__ __launch_bounds__(512) void k_phi_ifft_fold(const R* __restrict__ X, int64_t npf, int32_t ncol, int64_t ld,
                                                       int32_t K, int32_t L, const RingDev* __restrict__ rings,
                                                       const double2* __restrict__ tw, double scale,
                                                       R* __restrict__ out, int32_t TQ, int32_t k0, int32_t logM,
                                                       const int32_t* __restrict__ mall,
                                                       const FoldCol* __restrict__ cols)
{
    typedef typename Vec2T<R>::T R2;
    extern __shared__ double2 zif_raw[];
    const int nqt = (ncol + TQ - 1) / TQ;
    const int b = blockIdx.x, loc = b >> 3;
    const int unit = (((loc >> 2) << 3) + (b & 7)) * 4 + (loc & 3);
    if (unit >= (K - k0) * nqt) return;
    const int k = k0 + unit / nqt;
    const int c0 = (unit - (unit / nqt) * nqt) * TQ;
    const RingDev Rg = rings[k];
    const int N = Rg.npr, M = N >> 1, Mp = (int)fft_plen(M, sizeof(R));
    const int ltq = __ffs(TQ) - 1;
    R2* zs = (R2*)zif_raw;
    R2* twr = zs + TQ * Mp;
    R2* hs = twr + tw_len(N);  // TQ x (L + 1): H_m per sequence
    const double2* twg = tw + Rg.tw_off;
    for (int e = threadIdx.x; e <= N; e += blockDim.x) {
        const double2 w = twg[e];
        twr[twpad(e)].x = (R)w.x;
        twr[twpad(e)].y = (R)w.y;
    }
    const int Lk = mall[k];
    for (int e = threadIdx.x; e < TQ * (L + 1); e += blockDim.x) {
        const int m = e >> ltq, ql = e & (TQ - 1), c = c0 + ql;
        R2 x;
        x.x = 0;
        x.y = 0;
        if (c < ncol && m <= min(Lk, cols[c].mtop)) x = *(const R2*)(X + ((int64_t)m * K + k) * ld + 2 * c);
        const R f = m ? (R)2 : (R)1;
        const double2 ph64 = twg[((unsigned)m * (unsigned)Rg.shift) % (2u * (unsigned)N)];  // e^{i m phi_0}
        const R phx = f * (R)ph64.x, phy = f * (R)ph64.y;
        R2 h;
        h.x = x.x * phx - x.y * phy;
        h.y = x.x * phy + x.y * phx;
        hs[ql * (L + 1) + m] = h;
    }
    __syncthreads();
    for (int e = threadIdx.x; e < TQ * M; e += blockDim.x) {
        const int f = e >> logM, kk = e & (M - 1);
        const R2* h = hs + f * (L + 1);
        auto spec = [&](int bb) -> R2 {
            R2 v;
            v.x = 0;
            v.y = 0;
            if (bb == 0) {
                v.x = (R)2 * h[0].x;
                return v;
            }
            if (bb <= L) v = h[bb];
            if (N - bb <= L) {
                v.x += h[N - bb].x;
                v.y -= h[N - bb].y;
            }
            return v;
        };
        const R2 xa = spec(kk), xb = spec(M - kk);
        const R er = (R)0.5 * (xa.x + xb.x), ei = (R)0.5 * (xa.y - xb.y);
        const R dr = (R)0.5 * (xa.x - xb.x), di = (R)0.5 * (xa.y + xb.y);
        const R2 w = twr[twpad(2 * kk)];
        const R orr = dr * w.x - di * w.y, oi = dr * w.y + di * w.x;
        const int rk = (int)(__brev((unsigned)kk) >> (32 - logM));
        R2 z;
        z.x = er - oi;
        z.y = -(ei + orr);
        zs[f * Mp + fpad<R>(rk)] = z;
    }
    __syncthreads();
    fft_passes<R>(zs, TQ, M, Mp, N, logM, twr);
    const R sc = (R)scale;
    for (int e = threadIdx.x; e < TQ * M; e += blockDim.x) {
        const int f = e >> logM, j = e & (M - 1), c = c0 + f;
        if (c >= ncol) continue;
        const R2 z = zs[f * Mp + fpad<R>(j)];
        R2 v;
        v.x = sc * z.x;
        v.y = -sc * z.y;
        *(R2*)(out + (int64_t)cols[c].q * npf + Rg.start_n + 2 * j) = v;
    }
}

// Polar ring pairs, inverse: k_phi_ipolar4 with one sequence per map.  Bound: the direct length-i DFTs
// (VALU) and their LDS reads (79% busy).  nside 128, 2514 maps, FP32: 345 us (unfolded 1.44 ms).
template <typename R>
__global__ __launch_bounds__(256) void k_phi_ipolar4_fold(const R* __restrict__ X, int64_t npf, int32_t ncol, int64_t ld,
                                                          int32_t K, const RingDev* __restrict__ rings,
                                                          const double2* __restrict__ tw, double scale,
                                                          R* __restrict__ out, int32_t TQMAX,
                                                          const int32_t* __restrict__ mall,
                                                          const FoldCol* __restrict__ cols, int32_t nring,
                                                          int32_t ntile)
{
    typedef typename Vec2T<R>::T R2;
    extern __shared__ double2 ipf_raw[];
    const int b = blockIdx.x, loc = b >> 3;
    const int unit = (((loc >> 2) << 3) + (b & 7)) * 4 + (loc & 3);
    if (unit >= nring * ntile) return;
    const int k = unit / ntile;
    const RingDev Rg = rings[k];
    const int npr = Rg.npr, ni = npr >> 2, n2 = 2 * npr, nu = ni / 2 + 1, njp = (ni + 1) / 2;
    const int TQ = min(TQMAX, (int)blockDim.x / njp);
    const int c0 = (unit - k * ntile) * TQ;
    if (c0 >= ncol) return;
    const double2* twl = tw + Rg.tw_off;
    R2* twi = (R2*)ipf_raw;    // (cos, sin)(2 pi v/i), v < i
    R2* Xb = twi + ni;         // [TQ][npr] folded spectrum
    R2* V = Xb + TQ * npr;     // [TQ][4][nu]
    for (int e = threadIdx.x; e < ni; e += blockDim.x) {
        twi[e].x = (R)twl[8 * e].x;
        twi[e].y = (R)twl[8 * e].y;
    }
    const int Lk = mall[k];
    const int nbh = npr / 2 + 1;
    for (int e = threadIdx.x; e < TQ * nbh; e += blockDim.x) {
        const int ql = e % TQ, bb = e / TQ, c = c0 + ql;
        R vr = 0, vi = 0;
        if (c < ncol) {
            const int top = min(Lk, cols[c].mtop);
            for (int sg = 0; sg < 2; ++sg) {  // m = +b (mod npr), then m = -b (mod npr) as conj
                const int m0 = sg ? (npr - bb) % npr : bb;
                for (int m = m0; m <= top; m += npr) {
                    const R2 x = *(const R2*)(X + ((int64_t)m * K + k) * ld + 2 * c);
                    const R f = m ? (R)2 : (R)1;
                    const double2 ph64 = twl[((unsigned)m * (unsigned)Rg.shift) % (unsigned)n2];  // e^{i m phi_0}
                    const R phx = f * (R)ph64.x, phy = f * (R)ph64.y;
                    vr += x.x * phx - x.y * phy;
                    const R hi = x.x * phy + x.y * phx;
                    vi += sg ? -hi : hi;
                }
            }
        }
        R2 v;
        v.x = vr;
        v.y = vi;
        Xb[ql * npr + bb] = v;
        if (bb > 0 && 2 * bb < npr) {
            v.y = -vi;
            Xb[ql * npr + npr - bb] = v;
        }
    }
    __syncthreads();
    for (int e = threadIdx.x; e < TQ * nu; e += blockDim.x) {
        const int f = e / nu, u = e - f * nu;
        ip4_radix<R>(Xb + f * npr, twl, ni, nu, u, V + f * 4 * nu);
    }
    __syncthreads();
    const int e = threadIdx.x;
    if (e >= TQ * njp) return;
    const int f = e / njp, jp = e - f * njp, c = c0 + f;
    if (c >= ncol) return;
    R y0[4], y1[4];
    const int j1 = ip4_outputs<R>(V + f * 4 * nu, twi, ni, nu, jp, y0, y1);
    const R sc = (R)scale;
    R* o = out + (int64_t)cols[c].q * npf + Rg.start_n;
#pragma unroll
    for (int ss = 0; ss < 4; ++ss) o[4 * jp + ss] = sc * y0[ss];
    if (j1 >= 0)
#pragma unroll
        for (int ss = 0; ss < 4; ++ss) o[4 * j1 + ss] = sc * y1[ss];
}

// Per galaxy and map range blockIdx.y (`step` runs of whole knot groups): part = (sum_q g_q(r) dbar_q,
// sum_q g'_q(r) dbar_q) on folded delta-bar maps and uniform knots.  Galaxies come in radius bins,
// by folded pixel inside a bin (a wave's delta-bar loads fall on a few lines); their segment slot
// and t are found from the radii once per knot group.  Of each map's records only the block's
// radial range is staged, so several maps fit in LDS at a time and each is staged from L2 for the
// radii that need it (any order of the galaxies is right); the next map's delta-bar is loaded
// while one is summed.
// Value and slope come from one Horner chain (5 fma); the slopes of a group share the segment's
// 1/h, applied once to their sum.  Outside the knots the pseudo-records' slopes are 0.  R = float:
// FP32 records, delta-bar and products, FP64 sums.
// Bound: VALU (82% busy in FP32, 19 instructions per galaxy and map), then the random 16-byte
// record reads from LDS.  1e6 galaxies, 2514 maps, FP32: 1.71 ms; whole tables staged, two
// at a time by 1024 threads, ran 2.87 ms and moved 5.4 GB past L2.
constexpr int VF_THR = 512;         // two blocks per CU: one sums while the other stages
constexpr int VF_MAPS = 16;          // maps per stage at most
constexpr int VF_LDS = 78 << 10;
constexpr int VF_BIN = 7 << 10;     // record bytes of one map in a radius bin (1e6 galaxies, 2514 maps, FP32, events
                                    // around the launch: one bin of 40 KB 3.18 ms, 10: 1.92, 7: 1.80, 5: 1.80; 2e5, 344 maps, FP64:
                                    // 153, 127, 125 and 124 us)
constexpr int VF_BLOCKS = 2048;     // blocks wanted (with the reduction of their sums, the same cases: 1024 1.98 ms
                                    // and 130 us, 2048 1.88 and 141, 4096 1.92 and 142)
template <typename R> struct VfGpt { static constexpr int N = sizeof(R) == 8 ? 4 : 8; };  // galaxies per thread
__device__ __forceinline__ float vf_flip(float d, uint32_t s) { return __uint_as_float(__float_as_uint(d) ^ s); }
__device__ __forceinline__ double vf_flip(double d, uint32_t s)
{
    return __hiloint2double(__double2hiint(d) ^ (int)s, __double2loint(d));
}
template <typename R>
__global__ __launch_bounds__(VF_THR, 4) void k_vjp_fold(int64_t N, int64_t npf, int32_t lds, int32_t step, int32_t nrange,
                                                      const double* __restrict__ r_s,
                                                      const uint32_t* __restrict__ pix_s,
                                                      const GroupInfo* __restrict__ groups,
                                                      const double* __restrict__ gx, const double* __restrict__ grh,
                                                      const int32_t* __restrict__ vgs, const int32_t* __restrict__ vgm,
                                                      const int2* __restrict__ vrange,
                                                      const MapInfo* __restrict__ maps,
                                                      const typename Vec4T<R>::T* __restrict__ rec4,
                                                      const R* __restrict__ dbar, double2* __restrict__ part)
{
    typedef typename Vec4T<R>::T R4;
    constexpr int GPT = VfGpt<R>::N, NW = VF_THR / 64;
    extern __shared__ double4 vf_raw[];  // lds bytes
    R4* tb = (R4*)vf_raw;
    __shared__ double rr[2 * NW];
    __shared__ int64_t base[VF_MAPS];  // first record of each staged map
    __shared__ int32_t mapq[VF_MAPS];
    const int64_t k0 = (int64_t)blockIdx.x * (VF_THR * GPT) + threadIdx.x;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    double aw[GPT], ar[GPT];
    uint32_t pf[GPT], south = 0;  // byte offsets of the pixels
    double rlo = INFINITY, rhi = -INFINITY;
    auto radius = [&](int u) { return r_s[min(k0 + VF_THR * u, N - 1)]; };  // past the end: computed and dropped
#pragma unroll
    for (int u = 0; u < GPT; ++u) {
        const double r = radius(u);
        const uint32_t px = pix_s[min(k0 + VF_THR * u, N - 1)];
        pf[u] = (px >> 1) * (uint32_t)sizeof(R);
        south |= (px & 1u) << u;
        aw[u] = ar[u] = 0.0;
        rlo = fmin(rlo, r);  // (NaN is passed over)
        rhi = fmax(rhi, r);
    }
    for (int o = 32; o > 0; o >>= 1) {
        rlo = fmin(rlo, __shfl_xor(rlo, o, 64));
        rhi = fmax(rhi, __shfl_xor(rhi, o, 64));
    }
    if ((threadIdx.x & 63) == 0) {
        rr[threadIdx.x >> 6] = rlo;
        rr[NW + (threadIdx.x >> 6)] = rhi;
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < NW; ++i) {
        rlo = fmin(rlo, rr[i]);
        rhi = fmax(rhi, rr[NW + i]);
    }
    const int g0 = vrange[blockIdx.y * step].x, g1 = vrange[min((int)(blockIdx.y + 1) * step, nrange) - 1].y;
    // delta-bar of the range's maps in order, one map ahead of the sums
    const int jend = vgs[g1];
    R dn[GPT];
    auto load_dbar = [&](int j) {
        const char* dq = (const char*)(dbar + (int64_t)vgm[min(j, jend - 1)] * npf);
#pragma unroll
        for (int u = 0; u < GPT; ++u) dn[u] = *(const R*)(dq + pf[u]);
    };
    load_dbar(vgs[g0]);
    for (int g = g0; g < g1; ++g) {
        const GroupInfo G = groups[g];
        const double ainv = G.invdx, c0 = -G.xfirst * G.invdx, top = (double)(G.nk - 1);
        // the block's slots: uniform-grid slots of its end radii, one to spare for the knots' rounding
        // (NaN radii only: slot 0)
        const double flo = fmin(fmax(floor(fma(rlo, ainv, c0)), -1.0), top);
        const double fhi = fmin(fmax(floor(fma(rhi, ainv, c0)), -1.0), top);
        const int lo = __builtin_amdgcn_readfirstlane(rlo <= rhi ? max((int)flo, 0) : 0);
        const int hi = __builtin_amdgcn_readfirstlane(rlo <= rhi ? min((int)fhi + 2, G.nk) : 0);
        const int nrec = hi - lo + 1;  // (nk + 1 records always fit)
        const int fit = min(VF_MAPS, lds / (nrec * (int)sizeof(R4)));
        // segment slot (0 and nk: outside) and t of a radius
        auto locate = [&](double r, double& t) -> int {
            // the end knots belong to the end segments (their slopes), outside is flat
            const double v = fma(r, ainv, c0), fl = fmin(fmax(floor(v), 0.0), top - 1.0);
            int i = (int)fl;  // NaN: segment 0, t NaN
            t = v - fl;
            if (sizeof(R) == 8 && r == r) {
                // the caller's knots and the correctly rounded t of k_seg_t (the uniform grid's t
                // is off by the knots' own rounding, 1e-13)
                const double* xs = gx + G.xoff;
                double x0 = xs[i], x1 = xs[i + 1];
                if (r < x0 && i > 0) {
                    x1 = x0;
                    x0 = xs[--i];
                } else if (r >= x1 && i < G.nk - 2) {
                    x0 = x1;
                    x1 = xs[++i + 1];
                }
                const double h = x1 - x0, n = r - x0, y = grh[G.xoff + i], q0 = n * y;
                t = fma(fma(-h, q0, n), y, q0);
            }
            if (r < G.xfirst || r > G.xlast) t = 0.0;
            return r < G.xfirst ? 0 : (r > G.xlast ? G.nk : i + 1);
        };
        int ii[GPT];
        R t[GPT];
        double gr[GPT];
#pragma unroll
        for (int u = 0; u < GPT; ++u) {
            double tt;
            ii[u] = min(max(locate(radius(u), tt) - lo, 0), nrec - 1);  // (clamped: NaN)
            t[u] = (R)tt;
            gr[u] = 0.0;
        }
        for (int j = vgs[g]; j < vgs[g + 1]; j += fit) {
            const int nm = min(fit, vgs[g + 1] - j);
            __syncthreads();  // the previous maps' records are no longer read
            if ((int)threadIdx.x < nm) {
                const int q = vgm[j + threadIdx.x];
                base[threadIdx.x] = maps[q].koff + q;
                mapq[threadIdx.x] = maps[q].l & 1;
            }
            __syncthreads();
            const int nch = (nrec + 63) >> 6;  // a wave copies 64 records of one map at a time
            for (int c = wave; c < nm * nch; c += NW) {
                const int v = c / nch, k = (c - v * nch) * 64 + lane, sl = lo + k;
                // slot 0 holds y_first (record nk - 1), 1 .. nk - 1 the segments, nk y_last
                const int64_t bq = base[v];
                const R4* rq = rec4 + (((int64_t)__builtin_amdgcn_readfirstlane((int)(bq >> 32)) << 32) |
                                       (uint32_t)__builtin_amdgcn_readfirstlane((int)bq));
                if (k < nrec) lds_rec_put(tb + v * nrec, nrec, k, rq[sl == 0 ? G.nk - 1 : (sl == G.nk ? sl : sl - 1)]);
            }
            __syncthreads();
            for (int v = 0; v < nm; ++v) {
                const int mq = __builtin_amdgcn_readfirstlane(mapq[v]);
                const uint32_t flip = (mq & 1) ? south : 0u;  // odd l: southern galaxies take -dbar
                R d[GPT];
#pragma unroll
                for (int u = 0; u < GPT; ++u) d[u] = vf_flip(dn[u], (flip >> u) << 31);
                load_dbar(j + v + 1);  // (a range's maps are consecutive)
                const R4* tv = tb + v * nrec;
#pragma unroll
                for (int u = 0; u < GPT; ++u) {
                    const R4 c = lds_rec_get(tv, nrec, ii[u]);  // (d, c, b, a)
                    const R x = t[u];
                    const R p1 = fma(x, c.w, c.z), p2 = fma(x, p1, c.y);
                    const R val = fma(x, p2, c.x);
                    const R slope = fma(x, fma(x, c.w, p1), p2);
                    if (sizeof(R) == 8) {
                        aw[u] = fma((double)val, (double)d[u], aw[u]);
                        gr[u] = fma((double)slope, (double)d[u], gr[u]);
                    } else {
                        aw[u] += (double)(val * d[u]);
                        gr[u] += (double)(slope * d[u]);
                    }
                }
            }
        }
#pragma unroll
        for (int u = 0; u < GPT; ++u)
            ar[u] = fma(gr[u], sizeof(R) == 8 ? grh[G.xoff + min(max(ii[u] + lo - 1, 0), G.nk - 2)] : ainv, ar[u]);
    }
#pragma unroll
    for (int u = 0; u < GPT; ++u) {
        const int64_t k = k0 + VF_THR * u;
        if (k < N) part[(int64_t)blockIdx.y * N + k] = make_double2(aw[u], ar[u]);
    }
}
