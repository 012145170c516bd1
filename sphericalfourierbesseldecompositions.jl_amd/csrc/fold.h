// The FP64 path on folded hemispheres: plan tables and launches (kernels: fold_kernels.h).
#pragma once

static size_t fold_fft_lds(int64_t nside, int32_t tq) { return 16 * ((size_t)tq * (size_t)fft_plen(2 * nside, 8) + (size_t)tw_len(4 * nside)); }
static size_t fold_ifft_lds(int64_t nside, int64_t L, int32_t tq, size_t vb)
{
    return 2 * vb * ((size_t)tq * (size_t)fft_plen(2 * nside, vb) + (size_t)tw_len(4 * nside) + (size_t)tq * (size_t)(L + 1));
}

static int fold_tables(sfb_plan* P)
{
    Fold& F = P->fold;
    const DirectSht& D = P->dir;
    F.ok = false;
    // (a slot's radius carries the hemisphere in its sign: k_sell_fill)
    if (!D.ok || !P->sell_ok || !(P->r_first >= 0.0)) return SFB_OK;
    const int64_t L = P->lmax, nside = P->nside;
    F.npf = 6 * nside * nside + 2 * nside;
    // launch shapes: three FFT blocks per CU (53 KB) while they hold more than one map.  nside 128, 2514
    // maps: 577 us forward and 432 inverse FP32; at 80 KB 575 and 433, at 26 KB 546 and 448; nside 64, 344
    // maps, FP64: 27.9 and 26.1 us, 26 KB 27.7 and 25.4.
    F.tq = 8;
    while (F.tq > 1 && fold_fft_lds(nside, F.tq) > 53 * 1024) F.tq /= 2;
    for (int f = 0; f < 2; ++f) {
        F.tqi[f] = 8;
        while (F.tqi[f] > 1 && fold_ifft_lds(nside, L, F.tqi[f], f ? 4 : 8) > 53 * 1024) F.tqi[f] /= 2;
    }
    size_t shp = 0;
    if ((int64_t)fold_fft_lds(nside, F.tq) > P->lds_max || (int64_t)fold_ifft_lds(nside, L, F.tqi[0], 8) > P->lds_max ||
        !polar4_fits(P, sizeof(double), &shp))
        return SFB_OK;
    F.shi = 0;  // inverse polar blocks (FP64 bytes)
    F.tqp = IP_TQMAX;
    for (int64_t i = 1; i < nside; ++i) {
        const int64_t njp = (i + 1) / 2, tq = std::min<int64_t>(IP_TQMAX, 256 / njp);
        F.shi = std::max(F.shi, sizeof(double2) * (size_t)(i + tq * 4 * i + tq * 4 * (i / 2 + 1)));
        F.tqp = std::min<int32_t>(F.tqp, (int32_t)tq);
    }
    if ((int64_t)F.shi > P->lds_max) return SFB_OK;
    int32_t mal = -1;
    for (int64_t m = 0; m <= L; ++m)
        if (D.na[(size_t)m] > 0) mal = (int32_t)m;
    std::vector<FoldCol> cols((size_t)P->nmaps);
    std::vector<int32_t> qs((size_t)P->nmaps);
    for (int32_t q = 0; q < (int32_t)P->nmaps; ++q) qs[(size_t)q] = q;
    std::stable_sort(qs.begin(), qs.end(), [&](int32_t a, int32_t b) {
        const int32_t la = P->maps[(size_t)a].l, lb = P->maps[(size_t)b].l;
        return (la & 1) != (lb & 1) ? (la & 1) < (lb & 1) : la > lb;
    });
    F.neven = 0;
    for (size_t c = 0; c < qs.size(); ++c) {
        const MapInfo& mi = P->maps[(size_t)qs[c]];
        F.neven += !(mi.l & 1);
        cols[c] = {qs[c], mi.l, std::max<int32_t>(mi.l, mal), P->out_base[(size_t)qs[c]]};
    }
    std::vector<FoldM> fm((size_t)(L + 1));
    F.maxcnt = 1;
    for (int64_t m = 0; m <= L; ++m) {
        FoldM& M = fm[(size_t)m];
        M = FoldM{};
        M.kc = P->kcut[(size_t)m];
        M.s0 = D.s0[(size_t)m];
        M.na = D.na[(size_t)m];
        for (int pi = 0; pi < 2; ++pi) {
            const size_t b = (size_t)(2 * m + ((m + pi) & 1));
            M.lam[pi] = P->lam_off[b];
            M.v[pi] = D.voff[b];
            M.nb[pi] = P->nb[b];
            for (const FoldCol& c : cols) M.cnt[pi] += (c.l & 1) == pi && c.l >= m;
            F.maxcnt = std::max(F.maxcnt, M.cnt[pi]);
        }
    }
    // h = X [dOmega Lam U]: per aliasing m, the columns of each l parity with their block's table
    std::vector<RowGemm> hg;
    F.maxh = 1;
    for (int64_t m = 0; m <= L; ++m)
        for (int pi = 0; pi < 2; ++pi) {
            const int64_t b = 2 * m + ((m + pi) & 1), kc = P->kcut[(size_t)m];
            const int32_t h = P->niter * D.na[(size_t)m], nc = pi ? (int32_t)P->nmaps - F.neven : F.neven;
            if (h == 0 || nc == 0 || P->nb[(size_t)b] == 0) continue;
            RowGemm d{};
            d.B = D.d_HB.as<double>() + D.hboff[(size_t)b] + kc * h;
            d.arow = m * P->K + kc;
            d.crow = (int64_t)P->niter * D.s0[(size_t)m];
            d.K = (int32_t)(P->K - kc);
            d.N = d.ldb = h;
            d.dst = 1;
            d.col0 = pi ? 2 * F.neven : 0;
            d.ncol = 2 * nc;
            hg.push_back(d);
            F.maxh = std::max(F.maxh, h);
        }
    F.n_h = (int32_t)hg.size();
    // the southern pixel of every folded one (-1 on the equator)
    std::vector<int32_t> south((size_t)F.npf, -1);
    for (const sfb::RingPair& R : sfb::ring_pairs(nside))
        if (R.start_s != R.start_n)
            for (int64_t j = 0; j < R.npr; ++j)
                south[(size_t)(R.start_n + (j + R.npr / 2) % R.npr)] = (int32_t)(R.start_s + j);
    int rc;
    if ((rc = F.d_cols.ensure(sizeof(FoldCol) * cols.size())) || (rc = F.d_m.ensure(sizeof(FoldM) * fm.size())) ||
        (rc = F.d_h.ensure(sizeof(RowGemm) * std::max<size_t>(1, hg.size()))) ||
        (rc = F.d_south.ensure(4 * south.size())) || (rc = F.d_gzoff.ensure(sizeof(int64_t) * D.hboff.size())))
        return rc;
    HIP_TRY(hipMemcpy(F.d_cols.p, cols.data(), sizeof(FoldCol) * cols.size(), hipMemcpyHostToDevice));
    HIP_TRY(hipMemcpy(F.d_m.p, fm.data(), sizeof(FoldM) * fm.size(), hipMemcpyHostToDevice));
    if (!hg.empty()) HIP_TRY(hipMemcpy(F.d_h.p, hg.data(), sizeof(RowGemm) * hg.size(), hipMemcpyHostToDevice));
    HIP_TRY(hipMemcpy(F.d_south.p, south.data(), 4 * south.size(), hipMemcpyHostToDevice));
    HIP_TRY(hipMemcpy(F.d_gzoff.p, D.hboff.data(), sizeof(int64_t) * D.hboff.size(), hipMemcpyHostToDevice));
    F.ok = true;
    return SFB_OK;
}

// Folded FP64 maps (d_delta, rows of npf) -> a_nlm in d_out.
static int fold_analysis(sfb_plan* P, double* d_out, hipStream_t st)
{
    Fold& F = P->fold;
    DirectSht& D = P->dir;
    const int32_t nq = (int32_t)P->nmaps, K = P->K, k_eq0 = (int32_t)(P->nside - 1);
    const int64_t ld = P->M2;
    {
        PhaseTimer timer(P, SFB_PHASE_PHI, st);
        const size_t sh = fold_fft_lds(P->nside, F.tq);
        const int32_t nring = K - k_eq0, ntile = (int32_t)nblk(nq, F.tq);
        HIP_TRY(hipFuncSetAttribute((const void*)k_phi_fft_fold, hipFuncAttributeMaxDynamicSharedMemorySize, (int)sh));
        hipLaunchKernelGGL(k_phi_fft_fold, dim3((unsigned)(64 * (((int64_t)nring * ntile + 63) / 64))),
                           dim3(F.tq * 2 * P->nside >= 2048 ? 512 : 256), sh, st, P->d_delta.as<double>(), F.npf, nq, ld, K,
                           P->d_rings.as<RingDev>(), P->d_tw.as<double2>(), P->d_X0.as<double>(), F.tq, k_eq0, P->logM,
                           P->d_mall.as<int32_t>(), P->delta_perm, F.d_cols.as<FoldCol>(), nring, ntile);
        LAUNCH_CHECK();
    }
    if (k_eq0 > 0) {
        PhaseTimer timer(P, SFB_PHASE_PHI_POLAR, st);
        size_t shp;
        int32_t gy;
        polar4_fits(P, sizeof(double), &shp, (nq + 1) / 2, &gy);  // two maps here per map of k_phi_polar4
        const dim3 grid((unsigned)(32 * (((int64_t)k_eq0 * gy + 31) / 32)));
        auto go = [&](auto kern) -> int {
            HIP_TRY(hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)shp));
            hipLaunchKernelGGL(kern, grid, dim3(256), shp, st, P->d_delta.as<double>(), F.npf, nq, ld, K,
                               P->d_rings.as<RingDev>(), P->d_tw.as<double2>(), P->d_X0.as<double>(),
                               P->d_mall.as<int32_t>(), P->delta_perm, F.d_cols.as<FoldCol>(), k_eq0, gy);
            LAUNCH_CHECK();
            return SFB_OK;
        };
        const int rc = p4_mtwmax(P->nside) > 4 ? go(k_phi_polar4_fold<8>) : go(k_phi_polar4_fold<4>);
        if (rc) return rc;
    }
    if (F.n_h > 0) {
        PhaseTimer timer(P, SFB_PHASE_RESIDUAL, st);
        direct_gemm(F.d_h, F.n_h, F.maxh, 2 * nq, P->d_X0.as<double>(), ld, nullptr, 0, D.d_h.as<double>(), ld, 0.0, st);
        LAUNCH_CHECK();
        const int rc = direct_alias(P, 2 * nq, ld, st, 2 * F.neven);
        if (rc) return rc;
    }
    PhaseTimer timer(P, SFB_PHASE_ANALYSIS, st);
    hipLaunchKernelGGL(k_fold_rows, dim3(nblk(F.maxcnt, 64), 2, (unsigned)(P->lmax + 1)), dim3(256), 0, st, K, P->niter, ld,
                       F.d_m.as<FoldM>(), F.d_cols.as<FoldCol>(), F.neven, D.d_lamP.as<double>(), D.d_ZB.as<double>(),
                       P->d_X0.as<double>(), D.d_r.as<double>(), d_out, P->d_flag.as<int32_t>());
    LAUNCH_CHECK();
    return SFB_OK;
}

// Cotangent of a_nlm -> folded delta-bar maps times scale in d_delta (rows of npf, pixel order).
template <typename R> static int fold_synthesis(sfb_plan* P, const double* d_cot, double scale, hipStream_t st)
{
    Fold& F = P->fold;
    DirectSht& D = P->dir;
    const int32_t nq = (int32_t)P->nmaps, K = P->K, L = (int32_t)P->lmax, k_eq0 = (int32_t)(P->nside - 1);
    const int64_t ld = P->M2;
    const unsigned gx = nblk(nq, 64);
    if (F.n_h > 0) {
        hipLaunchKernelGGL(k_fold_coth, dim3(gx, (unsigned)(L + 1)), dim3(256), 0, st, P->niter, nq, ld, F.d_m.as<FoldM>(),
                           F.d_cols.as<FoldCol>(), F.neven, D.d_UB.as<double>(), d_cot, D.d_h.as<double>());
        LAUNCH_CHECK();
        const int rc = direct_alias(P, 2 * nq, ld, st, 2 * F.neven);
        if (rc) return rc;
    }
    hipLaunchKernelGGL(k_fold_synth<R>, dim3(nblk(F.neven, 64) + nblk(nq - F.neven, 64), nblk(K, 32), (unsigned)(L + 1)), dim3(256), 0, st, K, P->niter, nq, ld,
                       F.d_m.as<FoldM>(), F.d_cols.as<FoldCol>(), F.neven, D.d_lamPT.as<double>(), D.d_GZ.as<double>(),
                       F.d_gzoff.as<int64_t>(), D.d_r.as<double>(), d_cot, P->d_X0.as<R>());
    LAUNCH_CHECK();
    if (k_eq0 > 0) {
        const int32_t ntile = (nq + F.tqp - 1) / F.tqp;
        const size_t shi = F.shi / (sizeof(double) / sizeof(R));
        HIP_TRY(hipFuncSetAttribute((const void*)k_phi_ipolar4_fold<R>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)shi));
        hipLaunchKernelGGL(k_phi_ipolar4_fold<R>, dim3((unsigned)(32 * (((int64_t)k_eq0 * ntile + 31) / 32))), dim3(256), shi,
                           st, P->d_X0.as<R>(), F.npf, nq, ld, K, P->d_rings.as<RingDev>(), P->d_tw.as<double2>(), scale,
                           P->d_delta.as<R>(), IP_TQMAX, P->d_mall.as<int32_t>(), F.d_cols.as<FoldCol>(), k_eq0, ntile);
        LAUNCH_CHECK();
    }
    const int32_t tqi = F.tqi[sizeof(R) == 4];
    const size_t sh = fold_ifft_lds(P->nside, L, tqi, sizeof(R));
    const int64_t units = (int64_t)(K - k_eq0) * nblk(nq, tqi);
    HIP_TRY(hipFuncSetAttribute((const void*)k_phi_ifft_fold<R>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)sh));
    hipLaunchKernelGGL(k_phi_ifft_fold<R>, dim3((unsigned)(32 * ((units + 31) / 32))),
                       dim3(tqi * 2 * P->nside >= 2048 ? 512 : 256), sh, st, P->d_X0.as<R>(), F.npf, nq, ld, K, L,
                       P->d_rings.as<RingDev>(), P->d_tw.as<double2>(), scale, P->d_delta.as<R>(), tqi, k_eq0, P->logM,
                       P->d_mall.as<int32_t>(), F.d_cols.as<FoldCol>());
    LAUNCH_CHECK();
    return SFB_OK;
}
