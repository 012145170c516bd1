// The mixed path over the common radial basis: plan tables and the per-call stages
// (kernels: shells_kernels.h).
#pragma once

// Takes the fitted basis (radial.cpp) into device tables; ok stays false without one.
static int shells_tables(sfb_plan* P, const sfb::RadialBasis& R, bool fitted)
{
    Shells& S = P->shells;
    S.ok = false;
    S.tried = true;
    // the maps' buffers hold the shells and the mask, and the blocks' tables fit in LDS
    if (!fitted || !P->seg_uniform || R.nc + 1 > P->nmaps || (int64_t)sh_lds(R.nc) > P->lds_max ||
        16 * SM_N * (int64_t)P->tbl_cap > P->lds_max - 1024)
        return SFB_OK;
    // the maps of each l, and their coefficients by shell
    std::vector<int32_t> lstart((size_t)P->lmax + 2, 0), lq;
    std::vector<double> gt(R.gamma.size());
    for (int64_t l = 0; l <= P->lmax; ++l) {
        for (int32_t q = 0; q < (int32_t)P->nmaps; ++q)
            if (P->maps[(size_t)q].l == l) lq.push_back(q);
        const int64_t l0 = lstart[(size_t)l], cnt = (int64_t)lq.size() - l0;
        lstart[(size_t)l + 1] = (int32_t)lq.size();
        for (int64_t j = 0; j < cnt; ++j)
            for (int64_t s = 0; s < R.nc; ++s)
                gt[(size_t)(l0 * R.nc + s * cnt + j)] = R.gamma[(size_t)(lq[(size_t)(l0 + j)] * (int64_t)R.nc + s)];
    }
    int r;
    S.tried = false;  // (until every table is there)
    if ((r = S.d_knots.ensure(sizeof(double) * R.t.size())) || (r = S.d_gamma.ensure(sizeof(double) * gt.size())) ||
        (r = S.d_lstart.ensure(4 * lstart.size())) || (r = S.d_lq.ensure(4 * lq.size())))
        return r;
    HIP_TRY(hipMemcpy(S.d_lstart.p, lstart.data(), 4 * lstart.size(), hipMemcpyHostToDevice));
    HIP_TRY(hipMemcpy(S.d_lq.p, lq.data(), 4 * lq.size(), hipMemcpyHostToDevice));
    HIP_TRY(hipMemcpy(S.d_knots.p, R.t.data(), sizeof(double) * R.t.size(), hipMemcpyHostToDevice));
    HIP_TRY(hipMemcpy(S.d_gamma.p, gt.data(), sizeof(double) * gt.size(), hipMemcpyHostToDevice));
    S.nc = R.nc;
    S.ok = S.tried = true;
    return SFB_OK;
}

// The basis and its tables for a plan that has none yet, from the splines it holds on the device
// (records (x, y, y'', .) of every knot).
static int shells_build(sfb_plan* P)
{
    if (P->shells.tried) return SFB_OK;
    sfb::RadialBasis basis;
    bool fitted = false;
    if (P->dir.ok) {
        try {
            const size_t n = (size_t)(P->maps.back().koff + P->maps.back().nk);
            std::vector<double> rec(4 * n), kx(n), ky(n), kypp(n);
            HIP_TRY(hipMemcpy(rec.data(), P->d_rec.p, sizeof(double) * rec.size(), hipMemcpyDeviceToHost));
            for (size_t i = 0; i < n; ++i) {
                kx[i] = rec[4 * i];
                ky[i] = rec[4 * i + 1];
                kypp[i] = rec[4 * i + 2];
            }
            std::vector<int64_t> off;
            for (const MapInfo& m : P->maps) off.push_back(m.koff);
            off.push_back((int64_t)n);
            fitted = sfb::radial_basis(P->nmaps, off.data(), kx.data(), ky.data(), kypp.data(), &basis,
                                       (int)std::min(16u, std::thread::hardware_concurrency()));
        } catch (const std::bad_alloc&) {
            return fail(SFB_ERR_NOMEM, "out of host memory for the radial basis");
        }
    }
    return shells_tables(P, basis, fitted);
}

// Parts of the spread's galaxy runs: blocks of 256 galaxies at least, 12 blocks per CU at most.  Spread
// at nside 16 with blocks of 256 / 512 / 1024 at least: 52 / 87 / 196 us for 3e5 galaxies, 508 / 509 / 506
// for 4e6; at nside 32, 1e6: 108 / 113 / 180 (the sum of the parts takes 5 to 7).
static int32_t shell_parts(int64_t N, int64_t npix)
{
    const int64_t nb = nblk(npix, SH_PT);
    return (int32_t)std::max<int64_t>(1, std::min<int64_t>(3072 / nb, N / (256 * nb)));
}

// One mixed cat2amln over the shells, enqueued on st (separable window).
static int shells_enqueue(sfb_plan* P, int64_t N, const double* d_rtp, const double* d_w, double nbar,
                          const double* d_mask, const double* d_wln, double* d_out, hipStream_t st)
{
    Shells& S = P->shells;
    const int32_t nc = S.nc, nq = nc + 1;
    int rc;
    if ((rc = catalog_stage(P, N, d_rtp, d_w, st, CAT_INPUT, false))) return rc;
    {
        PhaseTimer timer(P, SFB_PHASE_SCATTER, st);
        const size_t shm = sh_lds(nc);
        const int32_t parts = shell_parts(N, P->npix);
        const int64_t n = (int64_t)nc * P->npix;
        if (parts > 1 && (rc = S.d_part.ensure(sizeof(double) * (size_t)(parts * n)))) return rc;
        double* D = P->d_delta.as<double>();
        double* to = parts > 1 ? S.d_part.as<double>() : D;
        const auto spread = parts > 1 ? k_shell_spread<true> : k_shell_spread<false>;
        HIP_TRY(hipFuncSetAttribute((const void*)spread, hipFuncAttributeMaxDynamicSharedMemorySize, (int)shm));
        hipLaunchKernelGGL(spread, dim3(nblk(P->npix, SH_PT), (unsigned)parts), dim3(SH_NT), shm, st, P->npix,
                           nc, S.d_knots.as<double>(), P->d_pstart.as<int32_t>(), P->d_rs.as<double>(),
                           P->d_ws.as<double>(), d_mask, to, D + n);
        LAUNCH_CHECK();
        if (parts > 1) {
            hipLaunchKernelGGL(k_shell_sum, dim3(nblk(n, 256)), dim3(256), 0, st, n, parts, to, D);
            LAUNCH_CHECK();
        }
    }
    // the l = 0 maps' exact sums: about two blocks per CU over all n while their tables leave
    // room for two, whole blocks of galaxies each
    const int32_t nmx = (int32_t)P->nmax, npair = (nmx + SM_N - 1) / SM_N;
    const size_t shm_m = 16 * SM_N * (size_t)P->tbl_cap;
    const int32_t want = 2 * shm_m <= (size_t)P->lds_max ? 512 : 256;
    const int32_t nch = (int32_t)std::max<int64_t>(1, std::min<int64_t>((want + npair - 1) / npair, (N + 1023) / 1024));
    {
        PhaseTimer timer(P, SFB_PHASE_MONOPOLE, st);
        if ((rc = P->d_mono.ensure(sizeof(double) * (size_t)nmx * (size_t)nch))) return rc;
        HIP_TRY(hipFuncSetAttribute((const void*)k_shell_mono, hipFuncAttributeMaxDynamicSharedMemorySize, (int)shm_m));
        hipLaunchKernelGGL(k_shell_mono, dim3((unsigned)nch, (unsigned)npair), dim3(1024), shm_m, st, N, nmx,
                           P->d_rs.as<double>(), P->d_ws.as<double>(), P->d_maps.as<MapInfo>(), P->d_rec.as<double4>(),
                           P->d_qbase.as<int32_t>(), P->d_mono.as<double>());
        LAUNCH_CHECK();
    }
    P->delta_perm = nullptr;
    if ((rc = sht_stage(P, nq, st))) return rc;
    PhaseTimer timer(P, SFB_PHASE_PACK, st);
    const double domega = 4.0 * kPi / (double)P->npix, inv = 1.0 / (nbar * domega);
    const size_t shm = sizeof(double2) * SC_M * (size_t)nq;
    hipLaunchKernelGGL(k_shell_contract, dim3(nblk(P->lmax + 1, SC_M), (unsigned)(P->lmax + 1)), dim3(256), shm, st,
                       (int32_t)P->lmax, nc, S.d_gamma.as<double>(), S.d_lstart.as<int32_t>(), S.d_lq.as<int32_t>(),
                       P->d_maps.as<MapInfo>(), P->d_outbase.as<int64_t>(), P->d_aoff.as<int64_t>(), P->a_ld,
                       P->a_final, d_wln, P->dir.d_h.as<double>() + P->dir.hrows * P->a_ld, P->d_mono.as<double>(), nch,
                       domega / std::sqrt(4.0 * kPi), inv, d_out, P->d_flag.as<int32_t>());
    LAUNCH_CHECK();
    return SFB_OK;
}
