// map2alm with its refinement iterations as one linear operator: plan tables and launches
// (the operator and its kernels: sht_direct_kernels.h).
#pragma once

// Limits of the folded form.  Beyond them (lmax well above nside, where whole equatorial
// rings alias, or many refinements) the tables [.. | J n_al] outgrow the iteration they
// replace and a column's states no longer fit in LDS: the iterated form stays (jacobi_stage).
constexpr int32_t DIRECT_MAX_NITER = 8, DIRECT_MAX_NAL = 48, DIRECT_MAX_STATES = 1536;

// Columns per k_alias_solve block: 4 (8: 80 us against 77 for 5028 columns at nside 128, 25 against 20
// for 320, 28 against 20 at nside 32), fewer when the states do not fit.
static inline int32_t direct_alias_ct(const DirectSht& D, int32_t J, int64_t lds_max)
{
    int32_t ct = 4;
    while (ct > 1 && (int64_t)alias_lds(D.S, J, ct, D.nterm) > lds_max) ct /= 2;
    return ct;
}

// Builds the operator's tables.  rowmax[m K + k] = max over l of |lambda_lm| on ring pair k.
static int direct_tables(sfb_plan* P, const std::vector<RingDev>& rd, const std::vector<double>& rowmax)
{
    const int64_t L = P->lmax;
    const int32_t K = P->K, J = P->niter;
    DirectSht& D = P->dir;
    D.ok = false;
    const double domega = 4.0 * kPi / (double)P->npix;
    std::vector<int32_t> ka((size_t)(L + 1), 0), na((size_t)(L + 1), 0), s0((size_t)(L + 2), 0);
    // kept states: (m, k) with a partner m' = m (mod npr), m' != m signed, whose product counts
    struct Pair { int32_t m, mp, k; double cre, cim; };
    std::vector<Pair> pairs;
    std::vector<int32_t> kb((size_t)(L + 1), 0);
    for (int64_t m = 0; m <= L; ++m) ka[(size_t)m] = K;
    if (J > 0)
        for (int32_t k = 0; k < P->K_al; ++k) {
            const int32_t npr = rd[(size_t)k].npr, sh = rd[(size_t)k].shift;
            const double wk = (k == K - 1) ? 1.0 : 2.0;  // north and south rings in one parity
            for (int64_t m = 0; m <= L; ++m)
                for (int64_t mp = m - ((m + L) / npr) * npr; mp <= L; mp += npr) {
                    if (mp == m) continue;
                    const int64_t ma = mp < 0 ? -mp : mp;
                    if (!(domega * npr * wk * rowmax[(size_t)(m * K + k)] * rowmax[(size_t)(ma * K + k)] > 1e-18))
                        continue;
                    const double sgn = ((((mp - m) / npr) * sh) & 1) ? -1.0 : 1.0;
                    const double c = -npr * wk * sgn;
                    pairs.push_back({(int32_t)m, (int32_t)ma, k, c, mp < 0 ? -c : c});
                    ka[(size_t)m] = std::min(ka[(size_t)m], k);
                    kb[(size_t)m] = std::max(kb[(size_t)m], k + 1);
                    if ((int64_t)pairs.size() > 64LL * DIRECT_MAX_STATES) return SFB_OK;
                }
        }
    for (int64_t m = 0; m <= L; ++m) {
        if (kb[(size_t)m] <= ka[(size_t)m]) ka[(size_t)m] = kb[(size_t)m] = 0;
        na[(size_t)m] = kb[(size_t)m] - ka[(size_t)m];
        s0[(size_t)m + 1] = s0[(size_t)m] + na[(size_t)m];
        if (na[(size_t)m] > DIRECT_MAX_NAL) return SFB_OK;
    }
    const int32_t S = s0[(size_t)L + 1];
    if (J > DIRECT_MAX_NITER || S > DIRECT_MAX_STATES) return SFB_OK;
    D.S = S;
    std::vector<AliasState> st((size_t)std::max(S, 1));
    for (int64_t m = 0; m <= L; ++m)
        for (int32_t a = 0; a < na[(size_t)m]; ++a)
            st[(size_t)(s0[(size_t)m] + a)] = {(int32_t)m, a, na[(size_t)m], s0[(size_t)m], 0, 0};
    std::vector<std::vector<AliasTerm>> by((size_t)std::max(S, 1));
    for (const Pair& p : pairs) {
        auto& v = by[(size_t)(s0[(size_t)p.m] + p.k - ka[(size_t)p.m])];
        const int32_t sp = s0[(size_t)p.mp] + p.k - ka[(size_t)p.mp];
        bool merged = false;
        for (AliasTerm& t : v)
            if (t.s == sp) {  // m' and -m' in one class
                t.cre += p.cre;
                t.cim += p.cim;
                merged = true;
            }
        if (!merged) v.push_back({sp, 0, p.cre, p.cim});
    }
    std::vector<AliasTerm> terms;
    for (int32_t s = 0; s < S; ++s) {
        st[(size_t)s].e0 = (int32_t)terms.size();
        terms.insert(terms.end(), by[(size_t)s].begin(), by[(size_t)s].end());
        st[(size_t)s].e1 = (int32_t)terms.size();
    }
    if (terms.empty()) terms.push_back({0, 0, 0.0, 0.0});
    D.nterm = (int32_t)terms.size();
    if ((int64_t)alias_lds(S, J, 1, D.nterm) > P->lds_max) return SFB_OK;
    // table offsets per block b = (m, parity)
    const int64_t nbat = 2 * (L + 1);
    std::vector<int64_t> hboff((size_t)nbat + 1, 0), voff((size_t)nbat + 1, 0), qoff((size_t)nbat + 1, 0);
    for (int64_t b = 0; b < nbat; ++b) {
        const int64_t a = na[(size_t)(b / 2)], n = P->nb[(size_t)b];
        hboff[(size_t)b + 1] = hboff[(size_t)b] + (n > 0 ? (int64_t)K * J * a : 0);
        voff[(size_t)b + 1] = voff[(size_t)b] + n * J * a;
        qoff[(size_t)b + 1] = qoff[(size_t)b] + std::max(J - 1, 0) * a * a;
    }
    int rc;
    struct Scratch {  // plan-time scratch, in two allocations
        DevBuf tab, mm;
        ~Scratch()
        {
            tab.release();
            mm.release();
        }
    } scratch;
    const int64_t icn = P->ic0_off.back();
    auto dbl = [](int64_t n) { return sizeof(double) * (size_t)std::max<int64_t>(1, n); };
    if ((rc = D.d_lamP.ensure(dbl(P->lam_size))) || (rc = D.d_lamPT.ensure(dbl(P->lam_size))) ||
        (rc = D.d_HB.ensure(dbl(hboff.back()))) || (rc = D.d_GZ.ensure(dbl(hboff.back()))) ||
        (rc = D.d_UB.ensure(dbl(voff.back()))) || (rc = D.d_ZB.ensure(dbl(voff.back()))) ||
        (rc = D.d_Q.ensure(dbl(qoff.back()))) || (rc = D.d_qoff.ensure(sizeof(int64_t) * qoff.size())) ||
        (rc = D.d_st.ensure(sizeof(AliasState) * st.size())) || (rc = D.d_term.ensure(sizeof(AliasTerm) * terms.size())) ||
        (rc = scratch.tab.ensure(dbl(voff.back() + 3 * icn))))
        return rc;
    double* const V = scratch.tab.as<double>();
    double *const I0 = V + voff.back(), *const P0 = I0 + icn, *const P1 = P0 + icn;
    HIP_TRY(hipMemcpy(D.d_qoff.p, qoff.data(), sizeof(int64_t) * qoff.size(), hipMemcpyHostToDevice));
    HIP_TRY(hipMemcpy(D.d_st.p, st.data(), sizeof(AliasState) * st.size(), hipMemcpyHostToDevice));
    HIP_TRY(hipMemcpy(D.d_term.p, terms.data(), sizeof(AliasTerm) * terms.size(), hipMemcpyHostToDevice));
    // one batched product over the blocks; f fills the descriptor of block b.  The products are
    // collected, uploaded together and launched in order.
    struct Launch { size_t at; unsigned n, gm, gn; };
    std::vector<SmallMM> all;
    std::vector<Launch> launches;
    auto batch = [&](auto f) {
        Launch l{all.size(), 0, 1, 1};
        for (int64_t b = 0; b < nbat; ++b) {
            if (P->nb[(size_t)b] <= 0) continue;
            SmallMM d{};
            d.alpha = 1.0;
            f(b, d);
            if (d.M <= 0 || d.N <= 0) continue;
            all.push_back(d);
            l.gm = std::max(l.gm, (unsigned)(d.M + 15) / 16);
            l.gn = std::max(l.gn, (unsigned)(d.N + 15) / 16);
            ++l.n;
        }
        if (l.n) launches.push_back(l);
    };
    auto lam = [&](int64_t b) { return P->d_lam.as<double>() + P->lam_off[(size_t)b]; };
    auto n_of = [&](int64_t b) { return P->nb[(size_t)b]; };
    auto a_of = [&](int64_t b) { return na[(size_t)(b / 2)]; };
    auto k_of = [&](int64_t b) { return (int64_t)ka[(size_t)(b / 2)]; };
    auto set = [](SmallMM& d, const double* A, int64_t ars, int64_t acs, const double* B, int64_t brs, int64_t bcs,
                  double* C, int64_t crs, int64_t ccs, int32_t M, int32_t N, int32_t Kk) {
        d.A = A; d.ars = ars; d.acs = acs; d.B = B; d.brs = brs; d.bcs = bcs;
        d.C = C; d.crs = crs; d.ccs = ccs; d.M = M; d.N = N; d.K = Kk;
    };
    // I0 = P0 = 1
    for (double* buf : {I0, P0})
        batch([&](int64_t b, SmallMM& d) {
        d.eye = 1;
        const int32_t n = n_of(b);
        set(d, nullptr, 0, 0, nullptr, 0, 0, buf + P->ic0_off[(size_t)b], n, 1, n, n, 0);
    });
    double *pc = P0, *pn = P1;
    for (int32_t j = 0; j < J; ++j) {
        const int64_t Jj = j;
        // U_j = P_j S^T and V_j = D^j S^T (V_0 = S^T), columns j na .. of the block's n x J na
        batch([&](int64_t b, SmallMM& d) {
            const int32_t n = n_of(b), a = a_of(b);
            set(d, pc + P->ic0_off[(size_t)b], n, 1, lam(b) + k_of(b) * n, 1, n,
                D.d_UB.as<double>() + voff[(size_t)b] + Jj * a, (int64_t)J * a, 1, n, a, n);
        });
        batch([&](int64_t b, SmallMM& d) {
            const int32_t n = n_of(b), a = a_of(b);
            double* v = V + voff[(size_t)b];
            if (j == 0)
                set(d, I0 + P->ic0_off[(size_t)b], n, 1, lam(b) + k_of(b) * n, 1, n, v,
                (int64_t)J * a, 1, n, a, n);
            else
                set(d, P->d_ic0.as<double>() + P->ic0_off[(size_t)b], n, 1, v + (Jj - 1) * a, (int64_t)J * a, 1,
                v + Jj * a, (int64_t)J * a, 1, n, a, n);
        });
        batch([&](int64_t b, SmallMM& d) {  // P_{j+1} = 1 + D P_j
            const int32_t n = n_of(b);
            d.eye = 1;
            set(d, P->d_ic0.as<double>() + P->ic0_off[(size_t)b], n, 1, pc + P->ic0_off[(size_t)b], n, 1,
                pn + P->ic0_off[(size_t)b], n, 1, n, n, n);
        });
        std::swap(pc, pn);
    }
    batch([&](int64_t b, SmallMM& d) {  // dOmega Lam P_J
        const int32_t n = n_of(b);
        d.alpha = domega;
        set(d, lam(b), n, 1, pc + P->ic0_off[(size_t)b], n, 1, D.d_lamP.as<double>() + P->lam_off[(size_t)b],
            n, 1, K, n, n);
    });
    batch([&](int64_t b, SmallMM& d) {  // its transpose without dOmega
        const int32_t n = n_of(b);
        set(d, lam(b), n, 1, pc + P->ic0_off[(size_t)b], n, 1,
            D.d_lamPT.as<double>() + P->lam_off[(size_t)b], 1, K, K, n, n);
    });
    batch([&](int64_t b, SmallMM& d) {  // dOmega Lam [U_0 .. U_{J-1}]
        const int32_t n = n_of(b), a = a_of(b);
        d.alpha = domega;
        set(d, lam(b), n, 1, D.d_UB.as<double>() + voff[(size_t)b], (int64_t)J * a, 1,
            D.d_HB.as<double>() + hboff[(size_t)b], (int64_t)J * a, 1, K, J * a, n);
    });
    for (int32_t j = 0; j < J; ++j) {
        const int64_t jr = J - 1 - j;  // Z_j and the adjoint's ring form take V_{J-1-j}
        batch([&](int64_t b, SmallMM& d) {
            const int32_t n = n_of(b), a = a_of(b);
            d.alpha = domega;
            set(d, V + voff[(size_t)b] + jr * a, 1, (int64_t)J * a,
                I0 + P->ic0_off[(size_t)b], n, 1,
                D.d_ZB.as<double>() + voff[(size_t)b] + (int64_t)j * a * n, n, 1, a, n, n);
        });
        batch([&](int64_t b, SmallMM& d) {
            const int32_t n = n_of(b), a = a_of(b);
            d.alpha = domega;
            set(d, V + voff[(size_t)b] + jr * a, 1, (int64_t)J * a, lam(b), 1, n,
                D.d_GZ.as<double>() + hboff[(size_t)b] + (int64_t)j * a * K, K, 1, a, K, n);
        });
        if (j + 1 < J) batch([&](int64_t b, SmallMM& d) {  // Q_j = dOmega S V_j
            const int32_t n = n_of(b), a = a_of(b);
            d.alpha = domega;
            set(d, lam(b) + k_of(b) * n, n, 1, V + voff[(size_t)b] + (int64_t)j * a,
                (int64_t)J * a, 1, D.d_Q.as<double>() + qoff[(size_t)b] + (int64_t)j * a * a, a,
                1, a, a, n);
        });
    }
    DevBuf& mm = scratch.mm;
    if ((rc = mm.ensure(sizeof(SmallMM) * std::max<size_t>(1, all.size())))) return rc;
    if (!all.empty()) HIP_TRY(hipMemcpy(mm.p, all.data(), sizeof(SmallMM) * all.size(), hipMemcpyHostToDevice));
    for (const Launch& l : launches) {
        hipLaunchKernelGGL(k_small_mm, dim3(l.gn, l.gm, l.n), dim3(256), 0, P->stream, mm.as<SmallMM>() + l.at);
        LAUNCH_CHECK();
    }
    HIP_TRY(hipStreamSynchronize(P->stream));  // done before the scratch is freed
    // launch descriptors.  Sector sg of block (m, par): l parity sg = (m + par) & 1.
    std::vector<RowGemm> ana, fix, syn, sfix;
    D.hrows = 2 * (int64_t)J * S;
    D.maxN = D.maxNs = D.maxNf = 1;
    for (int64_t b = 0; b < nbat; ++b) {
        const int64_t m = b / 2, n = P->nb[(size_t)b], kc = P->kcut[(size_t)m];
        if (n <= 0) continue;
        const int32_t a = na[(size_t)m], h = J * a;
        const int64_t sg = (m + b) & 1;
        const int64_t hrow = sg * J * (int64_t)S + (int64_t)J * s0[(size_t)m];
        RowGemm d{};
        d.ncol = -1;
        d.arow = b * K + kc;
        d.crow = P->aoff[(size_t)b];
        d.K = (int32_t)(K - kc);
        d.N = d.ldb = (int32_t)n;
        d.B = D.d_lamP.as<double>() + P->lam_off[(size_t)b] + kc * n;
        ana.push_back(d);
        // adjoint: a -> X over the ring pairs from kc on, a -> h
        RowGemm e = d;
        e.arow = P->aoff[(size_t)b];
        e.crow = b * K + kc;
        e.K = (int32_t)n;
        e.N = (int32_t)(K - kc);
        e.ldb = K;
        e.B = D.d_lamPT.as<double>() + P->lam_off[(size_t)b] + kc;
        syn.push_back(e);
        D.maxN = std::max<int32_t>(D.maxN, (int32_t)n);
        D.maxNs = std::max<int32_t>(D.maxNs, e.N);
        if (h == 0) continue;
        d.crow = hrow;
        d.dst = 1;
        d.N = d.ldb = h;
        d.B = D.d_HB.as<double>() + hboff[(size_t)b] + kc * h;
        ana.push_back(d);
        e.crow = hrow;
        e.dst = 1;
        e.N = e.ldb = h;
        e.B = D.d_UB.as<double>() + voff[(size_t)b];
        syn.push_back(e);
        D.maxN = std::max(D.maxN, h);
        D.maxNs = std::max(D.maxNs, h);
        // the corrections: r -> a, r -> X
        RowGemm f{};
        f.ncol = -1;
        f.arow = hrow;
        f.crow = P->aoff[(size_t)b];
        f.K = h;
        f.N = f.ldb = (int32_t)n;
        f.B = D.d_ZB.as<double>() + voff[(size_t)b];
        fix.push_back(f);
        f.crow = b * K + kc;
        f.N = (int32_t)(K - kc);
        f.ldb = K;
        f.B = D.d_GZ.as<double>() + hboff[(size_t)b] + kc;
        sfix.push_back(f);
        D.maxNf = std::max<int32_t>(D.maxNf, (int32_t)n);
    }
    {
        // one more row of h: sum over the ring pairs of the m = 0 coefficients, the maps' pixel
        // sums (the mixed path's monopoles)
        const std::vector<double> one((size_t)K, 1.0);
        if ((rc = D.d_one.ensure(sizeof(double) * one.size()))) return rc;
        HIP_TRY(hipMemcpy(D.d_one.p, one.data(), sizeof(double) * one.size(), hipMemcpyHostToDevice));
        RowGemm d{};
        d.ncol = -1;
        d.crow = D.hrows;
        d.dst = d.N = d.ldb = 1;
        d.K = K;
        d.B = D.d_one.as<double>();
        ana.push_back(d);
    }
    struct { DevBuf* d; std::vector<RowGemm>* v; int32_t* n; } up[] = {
        {&D.d_ana, &ana, &D.n_ana}, {&D.d_fix, &fix, &D.n_fix}, {&D.d_syn, &syn, &D.n_syn}, {&D.d_sfix, &sfix, &D.n_sfix}};
    for (auto& u : up) {
        *u.n = (int32_t)u.v->size();
        if ((rc = u.d->ensure(sizeof(RowGemm) * std::max<size_t>(1, u.v->size())))) return rc;
        if (!u.v->empty())
            HIP_TRY(hipMemcpy(u.d->p, u.v->data(), sizeof(RowGemm) * u.v->size(), hipMemcpyHostToDevice));
    }
    if ((rc = D.d_h.ensure(dbl((D.hrows + 1) * P->M2))) || (rc = D.d_r.ensure(dbl(D.hrows * P->M2)))) return rc;
    D.s0 = s0;
    D.hboff = hboff;
    D.voff = voff;
    D.na = na;
    D.ka = ka;
    D.ok = true;
    return SFB_OK;
}

static inline void direct_gemm(const DevBuf& desc, int32_t nbat, int32_t maxN, int32_t cols, const double* A, int64_t lda,
                               double* C0, int64_t ldc0, double* C1, int64_t ldc1, double beta, hipStream_t st)
{
    const dim3 g((unsigned)((cols + GT_BM - 1) / GT_BM), (unsigned)((maxN + GT_BNW - 1) / GT_BNW), (unsigned)nbat);
    hipLaunchKernelGGL(k_gemm_rows, g, dim3(256), 0, st, desc.as<RowGemm>(), cols, A, lda, C0, ldc0, C1, ldc1, 1.0, beta);
}

// The coupled aliasing steps h -> r of every column, both sectors.
static int direct_alias(sfb_plan* P, int32_t cols, int64_t ld, hipStream_t st, int32_t split = -1)
{
    DirectSht& D = P->dir;
    const int32_t J = P->niter;
    const int32_t ct = direct_alias_ct(D, J, P->lds_max);
    const size_t shm = alias_lds(D.S, J, ct, D.nterm);
    HIP_TRY(hipFuncSetAttribute((const void*)k_alias_solve, hipFuncAttributeMaxDynamicSharedMemorySize, (int)shm));
    hipLaunchKernelGGL(k_alias_solve, dim3(nblk(cols, ct), split < 0 ? 2u : 1u), dim3(1024), shm, st, D.S, J,
                       (int32_t)P->lmax, ct, cols, split, D.d_st.as<AliasState>(), D.nterm, D.d_term.as<AliasTerm>(),
                       D.d_Q.as<double>(), D.d_qoff.as<int64_t>(), D.d_h.as<double>(), D.d_r.as<double>(), ld);
    LAUNCH_CHECK();
    return SFB_OK;
}

// X0 (rows of ld values, the first cols used) -> refined a in d_a (rows of ld values).
static int direct_analysis(sfb_plan* P, int32_t cols, int64_t ld, hipStream_t st)
{
    DirectSht& D = P->dir;
    {
        PhaseTimer timer(P, SFB_PHASE_ANALYSIS, st);
        direct_gemm(D.d_ana, D.n_ana, D.maxN, cols, P->d_X0.as<double>(), ld, P->d_a.as<double>(), ld,
                    D.d_h.as<double>(), ld, 0.0, st);
        LAUNCH_CHECK();
    }
    if (D.n_fix > 0) {
        PhaseTimer timer(P, SFB_PHASE_RESIDUAL, st);
        int rc = direct_alias(P, cols, ld, st);
        if (rc) return rc;
        direct_gemm(D.d_fix, D.n_fix, D.maxNf, cols, D.d_r.as<double>(), ld, P->d_a.as<double>(), ld, nullptr, 0, 1.0, st);
        LAUNCH_CHECK();
    }
    P->a_final = P->d_a.as<double>();
    P->a_f32 = false;
    return SFB_OK;
}

// a (d_a) -> the refined iteration's ring coefficients S P_J(A S) a in X0.
static int direct_synthesis(sfb_plan* P, int32_t cols, int64_t ld, hipStream_t st)
{
    DirectSht& D = P->dir;
    direct_gemm(D.d_syn, D.n_syn, D.maxNs, cols, P->d_a.as<double>(), ld, P->d_X0.as<double>(), ld, D.d_h.as<double>(), ld,
                0.0, st);
    LAUNCH_CHECK();
    if (D.n_sfix > 0) {
        int rc = direct_alias(P, cols, ld, st);
        if (rc) return rc;
        direct_gemm(D.d_sfix, D.n_sfix, D.maxNs, cols, D.d_r.as<double>(), ld, P->d_X0.as<double>(), ld, nullptr, 0, 1.0,
                    st);
        LAUNCH_CHECK();
    }
    return SFB_OK;
}
