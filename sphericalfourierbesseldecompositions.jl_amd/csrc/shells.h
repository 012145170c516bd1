// The mixed path over the common radial basis: plan tables and the per-call stages
// (kernels: shells_kernels.h).
#pragma once

// Takes the fitted basis (radial.cpp) into device tables; ok stays false without one.
static int shells_tables(sfb_plan* P, const sfb::RadialBasis& R, bool fitted)
{
    Shells& S = P->shells;
    S.ok = false;
    // the maps' buffers hold the shells and the mask, and a block's tile fits in LDS
    if (!fitted || !P->seg_uniform || R.nc + 1 > P->nmaps || (int64_t)sh_lds(R.nc) > P->lds_max ||
        32 * (int64_t)(P->tbl_cap + 1) > P->lds_max - 1024)
        return SFB_OK;
    const int nt = R.nc + SH_W;
    std::vector<double> rc((size_t)SH_P * nt, 0.0);
    for (int k = 1; k <= SH_P; ++k)
        for (int i = 0; i + k < nt; ++i) {
            const double d = R.t[(size_t)(i + k)] - R.t[(size_t)i];
            rc[(size_t)(k - 1) * nt + i] = d > 0.0 ? 1.0 / d : 0.0;
        }
    int r;
    if ((r = S.d_knots.ensure(sizeof(double) * R.t.size())) || (r = S.d_recip.ensure(sizeof(double) * rc.size())) ||
        (r = S.d_gamma.ensure(sizeof(double) * R.gamma.size())))
        return r;
    HIP_TRY(hipMemcpy(S.d_knots.p, R.t.data(), sizeof(double) * R.t.size(), hipMemcpyHostToDevice));
    HIP_TRY(hipMemcpy(S.d_recip.p, rc.data(), sizeof(double) * rc.size(), hipMemcpyHostToDevice));
    HIP_TRY(hipMemcpy(S.d_gamma.p, R.gamma.data(), sizeof(double) * R.gamma.size(), hipMemcpyHostToDevice));
    S.nc = R.nc;
    S.ok = true;
    return SFB_OK;
}

// One mixed cat2amln over the shells, enqueued on st (separable window).
static int shells_enqueue(sfb_plan* P, int64_t N, const double* d_rtp, const double* d_w, double nbar,
                          const double* d_mask, const double* d_wln, double* d_out, hipStream_t st)
{
    const Shells& S = P->shells;
    const int32_t nc = S.nc, nq = nc + 1;
    int rc;
    if ((rc = catalog_stage(P, N, d_rtp, d_w, st, CAT_INPUT, false, false))) return rc;
    {
        PhaseTimer timer(P, SFB_PHASE_SCATTER, st);
        const size_t shm = sh_lds(nc);
        auto go = [&](auto kern) -> int {
            HIP_TRY(hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)shm));
            hipLaunchKernelGGL(kern, dim3(nblk(P->npix, SH_PT)), dim3(SH_NT), shm, st, P->npix, nc,
                               S.d_knots.as<double>(), S.d_recip.as<double>(), P->d_pstart.as<int32_t>(),
                               P->cat_idx, d_rtp, d_w, d_mask, P->d_delta.as<double>());
            LAUNCH_CHECK();
            return SFB_OK;
        };
        if ((rc = d_w ? go(k_shell_spread<false>) : go(k_shell_spread<true>))) return rc;
    }
    P->delta_perm = nullptr;
    if ((rc = sht_stage(P, nq, st))) return rc;
    const double domega = 4.0 * kPi / (double)P->npix, inv = 1.0 / (nbar * domega);
    {
        PhaseTimer timer(P, SFB_PHASE_PACK, st);
        const size_t shm = sizeof(double2) * SC_M * (size_t)nq;
        hipLaunchKernelGGL(k_shell_contract, dim3(nblk(P->lmax + 1, SC_M), (unsigned)(P->lmax + 1)), dim3(256), shm,
                           st, (int32_t)P->nmax, (int32_t)P->lmax, nc, S.d_gamma.as<double>(),
                           P->d_qbase.as<int32_t>(), P->d_lmaxn.as<int32_t>(), P->d_outbase.as<int64_t>(),
                           P->d_aoff.as<int64_t>(), P->a_ld, P->a_final, d_wln, inv, d_out, P->d_flag.as<int32_t>());
        LAUNCH_CHECK();
    }
    // the l = 0 maps' exact sums; chunks: two blocks per CU over all n (their tables are
    // 32 bytes per knot of LDS), whole waves of galaxies each
    PhaseTimer timer(P, SFB_PHASE_MONOPOLE, st);
    const int32_t nmx = (int32_t)P->nmax;
    const int32_t nch = (int32_t)std::max<int64_t>(1, std::min<int64_t>((512 + nmx - 1) / nmx, (N + 511) / 512));
    if ((rc = P->d_mono.ensure(sizeof(double) * (size_t)nmx * (size_t)nch))) return rc;
    const size_t shm = 32 * (size_t)(P->tbl_cap + 1);
    auto go = [&](auto kern) -> int {
        HIP_TRY(hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)shm));
        hipLaunchKernelGGL(kern, dim3((unsigned)nch, (unsigned)nmx), dim3(512), shm, st, N, P->d_rs.as<double>(), d_w,
                           P->d_maps.as<MapInfo>(), P->d_rec4.as<double4>(), P->d_qbase.as<int32_t>(),
                           P->d_mono.as<double>());
        LAUNCH_CHECK();
        return SFB_OK;
    };
    if ((rc = d_w ? go(k_shell_mono<false>) : go(k_shell_mono<true>))) return rc;
    hipLaunchKernelGGL(k_shell_monofix, dim3((unsigned)nmx), dim3(256), 0, st, nc, P->K, nch, P->d_X0.as<double>(),
                       P->a_ld, S.d_gamma.as<double>(), P->d_qbase.as<int32_t>(), P->d_outbase.as<int64_t>(),
                       P->d_mono.as<double>(), inv * domega / std::sqrt(4.0 * kPi), d_out, P->d_flag.as<int32_t>());
    LAUNCH_CHECK();
    return SFB_OK;
}
