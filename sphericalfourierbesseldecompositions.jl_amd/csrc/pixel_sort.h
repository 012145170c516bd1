// Galaxies grouped by pixel with counting kernels: count (the atomic's return value is the
// galaxy's arrival rank in its pixel), scan, place, and a rank pass that puts every pixel's
// galaxies into a fixed order, so the result does not depend on the atomics' order.  Seven
// dispatches where two stable radix sorts took forty: the catalogue stage of a small call is
// launch-bound (1e5 galaxies at nside 32: ~49 dispatches of 3-7 us each).
//
// The rank pass compares a pixel's galaxies pairwise.  A catalogue with many galaxies in every
// pixel takes stable radix sorts instead (known from its size); a few crowded pixels
// do not: their rank costs little beside the sum over a pixel's galaxies in order that follows it, up
// to PS_CROWD galaxies (1.5e5 in one pixel, nside 64: 0.3 of 21.4 ms mixed, 0.65 of 21.3 ms in FP64).  A
// pixel beyond raises flag[2] bit 1 and the call is redone with the radix sorts.
#pragma once

// Mean galaxies per pixel above which the radix sorts run.  FP64 (by pixel and r, two sorts): at
// nside 16 the call takes 684 us with counting kernels against 795 with the sorts at 768 per folded
// pixel, 1310 against 1256 at 1536; nside 32 2765 / 3061 at 768.  Mixed (one sort, by pixel): 456 us
// either way at 96, nside 32; 198 / 222 at 48 and 460 / 525 at 144, nside 16; 340 / 332 at 24 and
// 1084 / 949 at 96, nside 64.  Any order (adjoint, in radius bins): 463 us either way at 638, nside 16
// mixed, 1315 / 828 at 2551 (the counters' atomics); 435 / 501 and 1450 / 1163 in FP64.
constexpr int PS_MEAN_R = 1024, PS_MEAN = 96, PS_MEAN_ANY = 640;
constexpr int PS_CROWD = 1 << 20; // galaxies of one pixel that the rank takes
constexpr int PS_WALK = 64;       // galaxies of a pixel up to which each lane walks them (call at 96 per
                                  // pixel, nside 32 FP64: 478 us; 128: 550, 256: 534)
constexpr int PS_OWN = 1024;      // galaxies a block ranks together in a giant pixel
constexpr int PS_GIANT = 4096;    // galaxies of a pixel from which blocks rank it (catalogue stage of 3e5 galaxies with one
                                  // such pixel, by wavefronts / by blocks: mixed 100 / 110 us at 3000, 124 / 117 at
                                  // 4000, 205 / 174 at 10000; FP64 135 / 149, 182 / 184 at 7000, 223 / 210)
constexpr int PS_CHUNK = 2048;    // pixels per scan block
constexpr int PS_SMALL = 32;      // scan blocks up to which each adds up the counts before it itself (one launch
                                  // less; 4 blocks: 5.0 us against 7.2 in two, 13: 8.2 / 9.1, 49: 17.8 / 9.3)

__global__ __launch_bounds__(256) void k_zero_counts(int64_t npix, int32_t* __restrict__ cnt, int32_t* __restrict__ flag)
{
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < npix) cnt[i] = 0;
    if (i < 4) flag[i] = 0;
}

// Radius bins in front of the pixels (bin major; n <= 1: none), for consumers that want a block's
// galaxies in a narrow radial range.  The bin of a galaxy only orders the list.
struct RadBins {
    int32_t n;
    uint32_t np2;      // folded pixels with the hemisphere bit: 2 npf per bin
    double r0, inv;    // bin = (r - r0) inv, clamped
};

// Arrival rank in a cell.  Atomics on one address take 7 ns each, one after another, so where lanes of a
// wavefront share a cell (a crowded or an ordered catalogue) one lane adds for all of its cell.  Shared
// cells are looked for among lanes whose numbers differ in one bit (192 of the 2016 pairs: ten lanes of one
// cell by chance are missed one time in a hundred, six one in four); a cell that is missed only takes its
// atomics one by one.  3e5 galaxies, nside 64, 1e4 / 3e4 / 1.5e5 of them in one pixel: 94 / 102 / 57 us (four
// cells tried by comparing with every lane: 114 / 236 / 157, and 1 us more at 5 galaxies per pixel).
__device__ __forceinline__ uint32_t arrival_rank(int32_t* __restrict__ cnt, uint32_t cell)
{
    const int lane = threadIdx.x & 63;
    uint64_t hit = 0;  // (lanes past the end hold anything: a false hit finds no company below)
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) hit |= __ballot(cell == (uint32_t)__shfl_xor((int)cell, d, 64));
    if (!hit) return (uint32_t)atomicAdd(cnt + cell, 1);
    uint64_t mine = 1ull << lane;
    while (hit) {
        const uint32_t c = (uint32_t)__builtin_amdgcn_readlane((int)cell, __ffsll((unsigned long long)hit) - 1);
        const uint64_t same = __ballot(cell == c);
        if (cell == c) mine = same;
        hit &= ~same;
    }
    const int lead = __ffsll((unsigned long long)mine) - 1;
    int32_t base = 0;
    if (lane == lead) base = atomicAdd(cnt + cell, (int32_t)__popcll(mine));
    return (uint32_t)(__shfl(base, lead, 64) + (int32_t)__popcll(mine & ((1ull << lane) - 1)));
}

// pixel (FOLD: folded, with the hemisphere in bit 0) and arrival rank of every galaxy.
// flag[1] |= 1 when an angle is not finite (the reference's floor(Int, NaN) throws).
template <bool FOLD>
__global__ __launch_bounds__(256) void k_count(int64_t N, const double* __restrict__ rtp, int64_t nside,
                                               int32_t* __restrict__ cnt, uint2* __restrict__ pr,
                                               int32_t* __restrict__ flag, RadBins rb)
{
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= N) return;
    const double th = rtp[3 * i + 1], ph = rtp[3 * i + 2];
    int64_t p = 0;
    if (isfinite(th) && isfinite(ph)) {
        p = ang2pix_ring_dev(nside, th, ph);
        p = min(max(p, (int64_t)0), 12 * nside * nside - 1);
    } else {
        atomicOr(flag + 1, 1);
    }
    uint32_t f = FOLD ? fold_pixel(p, nside) : (uint32_t)p;
    if (FOLD && rb.n > 1) f += rb.np2 * (uint32_t)fmin(fmax((rtp[3 * i] - rb.r0) * rb.inv, 0.0), (double)(rb.n - 1));
    pr[i] = make_uint2(f, arrival_rank(cnt, FOLD ? f >> 1 : f));
}

// per PS_CHUNK pixels: their galaxies, and the crowding flag
__global__ __launch_bounds__(256) void k_count_sums(int64_t npix, const int32_t* __restrict__ cnt,
                                                    int32_t* __restrict__ sums, int32_t* __restrict__ flag)
{
    __shared__ int32_t red[4];
    const int64_t p0 = (int64_t)blockIdx.x * PS_CHUNK;
    int32_t s = 0, big = 0;
    for (int u = 0; u < PS_CHUNK / 256; ++u) {
        const int64_t p = p0 + u * 256 + threadIdx.x;
        const int32_t c = p < npix ? cnt[p] : 0;
        s += c;
        big = max(big, c);
    }
    for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o, 64);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = s;
    if (flag && big > PS_CROWD) atomicOr(flag + 2, 2);
    __syncthreads();
    if (threadIdx.x == 0) sums[blockIdx.x] = red[0] + red[1] + red[2] + red[3];
}

// pstart[p] = galaxies before pixel p; pstart[npix] = N.  sums NULL (small grids, one launch
// less): a block adds up the counts before its chunk itself, and checks its own for crowding.
__global__ __launch_bounds__(256) void k_count_scan(int64_t npix, int32_t N, const int32_t* __restrict__ cnt,
                                                    const int32_t* __restrict__ sums, int32_t* __restrict__ pstart,
                                                    int32_t* __restrict__ flag)
{
    __shared__ int32_t part[256];
    constexpr int PT = PS_CHUNK / 256;
    const int t = threadIdx.x;
    int32_t before = 0;
    if (sums)
        for (int b = t; b < (int)blockIdx.x; b += 256) before += sums[b];
    else
#pragma unroll 8
        for (int p = t; p < (int)blockIdx.x * PS_CHUNK; p += 256) before += cnt[p];
    const int64_t p0 = (int64_t)blockIdx.x * PS_CHUNK + t * PT;
    int32_t c[PT], s = 0;
#pragma unroll
    for (int u = 0; u < PT; ++u) {
        c[u] = p0 + u < npix ? cnt[p0 + u] : 0;
        s += c[u];
        if (!sums && flag && c[u] > PS_CROWD) atomicOr(flag + 2, 2);
    }
    // the chunk's offset: the sum of `before` over the block
    for (int o = 32; o > 0; o >>= 1) before += __shfl_xor(before, o, 64);
    if ((t & 63) == 0) part[t >> 6] = before;
    __syncthreads();
    const int32_t base = part[0] + part[1] + part[2] + part[3];
    __syncthreads();
    part[t] = s;
    __syncthreads();
    for (int o = 1; o < 256; o <<= 1) {
        const int32_t v = t >= o ? part[t - o] : 0;
        __syncthreads();
        part[t] += v;
        __syncthreads();
    }
    int32_t run = base + part[t] - s;
#pragma unroll
    for (int u = 0; u < PT; ++u) {
        if (p0 + u < npix) pstart[p0 + u] = run;
        run += c[u];
    }
    if (blockIdx.x == 0 && t == 0) pstart[npix] = N;
}

// A galaxy at its place by arrival: everything the rank pass needs in one 32-byte sector, so
// the scattered writes touch one sector per galaxy (index and pixel placed alone, with the rank
// pass gathering r and w from the catalogue, ran 17 + 25 us at N = 1e6 and 64 + 166 us at 4e6).
struct alignas(32) CatSlot {
    double r, w;
    uint32_t i, pix;
};

__global__ __launch_bounds__(256) void k_place(int64_t N, const uint2* __restrict__ pr,
                                               const int32_t* __restrict__ pstart, const double* __restrict__ rtp,
                                               const double* __restrict__ w, int32_t sh, CatSlot* __restrict__ slot,
                                               uint32_t np2)
{
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= N) return;
    const uint2 q = pr[i];
    CatSlot c;
    c.r = rtp[3 * i];
    c.w = w ? w[i] : 1.0;
    c.i = (uint32_t)i;
    c.pix = np2 ? q.x % np2 : q.x;  // without the radius bin
    slot[(int64_t)pstart[q.x >> sh] + q.y] = c;
}

// Orders a wavefront's LDS accesses (its lanes run in step; only the compiler may reorder).
__device__ __forceinline__ void wave_lds_sync()
{
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// Sort key of a galaxy inside its pixel, northern ones first: ORDER 1 the input index, 2 r and
// the input index (31 bits).  No galaxy's key is the largest value.
struct RankKey {
    uint64_t a;
    uint32_t b;
};
template <int ORDER> __device__ __forceinline__ RankKey rank_key(const CatSlot& c)
{
    const uint64_t south = (uint64_t)(c.pix & 1u) << 63;
    if (ORDER == 1) return {south | c.i, 0};
    const uint64_t k = sortable_bits(c.r);
    return {south | k >> 1, (uint32_t)(k & 1) << 31 | c.i};
}
__device__ __forceinline__ bool rank_less(const RankKey& x, const RankKey& y)
{
    return (x.a < y.a) | ((x.a == y.a) & (x.b < y.b));
}

// The places of a giant pixel's galaxies [e, e + PS_OWN) (the pixel's run ends at s1), by a whole block:
// its own galaxies, sorted, stay in LDS and every galaxy of the pixel finds its place among them.  The list
// entries of its own galaxies are written.
struct RankLds {
    uint64_t a[PS_OWN];
    uint32_t b[PS_OWN], hist[PS_OWN];
    int32_t wsum[4];
};
// o before the own galaxy at place i (b decides ties of a: radii bit for bit the same)
template <int ORDER> __device__ __forceinline__ bool rank_before(const RankKey& o, const RankLds& L, int i)
{
    const uint64_t a = L.a[i];
    bool less = o.a < a;
    if (ORDER == 2 && o.a == a) less = o.b < L.b[i];
    return less;
}
template <int ORDER>
__device__ __forceinline__ void rank_block(const CatSlot* __restrict__ slot, int32_t e, int32_t s0, int32_t s1, RankLds& L,
                                           uint32_t* __restrict__ idx, uint32_t* __restrict__ pix_s,
                                           double* __restrict__ r_s, double* __restrict__ w_s)
{
    constexpr int U = PS_OWN / 256;
    const int t = threadIdx.x, lane = t & 63, wv = t >> 6, n = min(PS_OWN, s1 - e);
#pragma unroll
    for (int u = 0; u < U; ++u) {
        const int j = t + 256 * u;
        const RankKey k = j < n ? rank_key<ORDER>(slot[e + j]) : RankKey{~0ull, ~0u};
        L.a[j] = k.a;
        L.b[j] = k.b;
        L.hist[j] = 0;
    }
    __syncthreads();
    for (int m = 2; m <= PS_OWN; m <<= 1)  // bitonic sort
        for (int d = m >> 1; d > 0; d >>= 1) {
#pragma unroll
            for (int u = 0; u < U / 2; ++u) {
                const int q = t + 256 * u, i = ((q & ~(d - 1)) << 1) | (q & (d - 1));
                const RankKey x{L.a[i], L.b[i]}, y{L.a[i + d], L.b[i + d]};
                if (rank_less(y, x) == ((i & m) == 0)) {
                    L.a[i] = y.a;
                    L.b[i] = y.b;
                    L.a[i + d] = x.a;
                    L.b[i + d] = x.b;
                }
            }
            __syncthreads();
        }
    constexpr int V = 2;  // searches in flight
    int32_t none = 0;     // galaxies before every own one
    RankKey nx[V];
    auto load = [&](uint32_t c) {
#pragma unroll
        for (int u = 0; u < V; ++u) nx[u] = rank_key<ORDER>(slot[min(c + 256 * u, (uint32_t)s1 - 1)]);
    };
    load((uint32_t)s0 + t);
    for (uint32_t c = (uint32_t)s0 + t; c < (uint32_t)s1; c += 256 * V) {
        RankKey o[V];
        int at[V];  // own galaxies up to o
#pragma unroll
        for (int u = 0; u < V; ++u) {
            o[u] = nx[u];
            at[u] = 0;
        }
        load(c + 256 * V);
#pragma unroll
        for (int step = PS_OWN / 2; step > 0; step >>= 1)
#pragma unroll
            for (int u = 0; u < V; ++u) at[u] += rank_before<ORDER>(o[u], L, at[u] + step - 1) ? 0 : step;
#pragma unroll
        for (int u = 0; u < V; ++u) {
            at[u] += !rank_before<ORDER>(o[u], L, at[u]);
            if (c + 256 * u >= (uint32_t)s1) continue;
            if (at[u] == 0) ++none;
            else if (at[u] < PS_OWN) atomicAdd(&L.hist[at[u]], 1u);
        }
    }
    for (int o = 32; o > 0; o >>= 1) none += __shfl_xor(none, o, 64);
    if (lane == 0) atomicAdd(&L.hist[0], (uint32_t)none);
    __syncthreads();
    int32_t h[U], sum = 0;
#pragma unroll
    for (int u = 0; u < U; ++u) h[u] = sum += (int32_t)L.hist[U * t + u];
    int32_t inc = sum;
    for (int o = 1; o < 64; o <<= 1) {
        const int32_t v = __shfl_up(inc, o, 64);
        if (lane >= o) inc += v;
    }
    if (lane == 63) L.wsum[wv] = inc;
    __syncthreads();
    int32_t base = inc - sum;
    for (int i = 0; i < wv; ++i) base += L.wsum[i];
#pragma unroll
    for (int u = 0; u < U; ++u) L.hist[U * t + u] = (uint32_t)(base + h[u]);
    __syncthreads();
#pragma unroll
    for (int u = 0; u < U; ++u) {
        if (t + 256 * u >= n) continue;
        const CatSlot c = slot[e + t + 256 * u];
        const RankKey k = rank_key<ORDER>(c);
        int p = 0;  // place among the own galaxies
#pragma unroll
        for (int step = PS_OWN / 2; step > 0; step >>= 1) p += rank_less({L.a[p + step - 1], L.b[p + step - 1]}, k) ? step : 0;
        const int64_t f = (int64_t)s0 + L.hist[p];
        idx[f] = c.i;
        pix_s[f] = c.pix;
        r_s[f] = c.r;
        w_s[f] = c.w;
    }
    __syncthreads();  // the next pixel's galaxies take the LDS
}

// order inside a pixel: 0 as placed (where any order does), 1 by input index, 2 by (r, input
// index), the order of the reference's sums; in a folded pixel northern galaxies first, as the
// radix sorts leave them.  Writes the sorted list of input indices, and
// pixel, r and w in that order.
// Bound: the scattered 32-byte writes while pixels hold a few galaxies: each lane walks its own
// pixel's.  A wavefront that meets a crowded pixel takes its pixels one after another: its own
// galaxies of the pixel, sorted, stay in LDS, every other galaxy finds its place among them (seven
// LDS reads, 64 galaxies at a time), and a galaxy's rank is the sum of the places up to its own.  Pixels
// beyond PS_GIANT go to whole blocks, PS_OWN own galaxies at a time (1.5e5 in one pixel: 0.33 ms by input
// index and 0.66 by radius; by wavefronts 1.9 and 1.2), which costs the others one early barrier.
template <int ORDER>
__global__ __launch_bounds__(256, 8) void k_rank(int64_t N, const CatSlot* __restrict__ slot,
                                              const int32_t* __restrict__ pstart, int32_t sh,
                                              uint32_t* __restrict__ idx,
                                              uint32_t* __restrict__ pix_s, double* __restrict__ r_s,
                                              double* __restrict__ w_s)
{
    __shared__ RankLds lds;
    __shared__ int32_t lead[4][2];  // a wavefront's slots meet two giant pixels at most (-1: none)
    uint64_t(*own_a)[64] = (uint64_t(*)[64])lds.a;
    uint32_t(*own_b)[64] = (uint32_t(*)[64])lds.b, (*hist)[64] = (uint32_t(*)[64])lds.hist;
    const int64_t e0 = (int64_t)blockIdx.x * blockDim.x + threadIdx.x, e = min(e0, N - 1);
    const CatSlot me = slot[e];
    int64_t f = e;
    bool giant = false, giants = false;  // this galaxy's pixel; a set of own galaxies starts in this block
    if (ORDER) {
        const int32_t s0 = pstart[me.pix >> sh], s1 = pstart[(me.pix >> sh) + 1];
        giant = s1 - s0 > PS_GIANT && s1 - s0 <= PS_CROWD;
        {
            const int wv = threadIdx.x >> 6;
            const uint64_t at = __ballot(giant && e0 < N && ((int32_t)e - s0) % PS_OWN == 0), next = at & (at - 1);
            if ((threadIdx.x & 63) == 0) {
                lead[wv][0] = at ? (int32_t)e + __ffsll((unsigned long long)at) - 1 : -1;
                lead[wv][1] = next ? (int32_t)e + __ffsll((unsigned long long)next) - 1 : -1;
            }
            __syncthreads();
#pragma unroll
            for (int q = 0; q < 4; ++q) giants |= lead[q][0] >= 0;
        }
        int32_t before = 0;
        if (__ballot(s1 - s0 > PS_WALK) == 0) {
            const uint64_t k = sortable_bits(me.r);
            for (int32_t s = s0; s < s1; ++s) {
                const uint32_t i = slot[s].i, ps = slot[s].pix;
                if (ORDER == 2) {
                    const uint64_t ks = sortable_bits(slot[s].r);
                    before += ps < me.pix || (ps == me.pix && (ks < k || (ks == k && i < me.i)));
                } else {
                    before += ps < me.pix || (ps == me.pix && i < me.i);
                }
            }
        } else {  // (every lane is here, those past the end without a galaxy)
            const RankKey k = rank_key<ORDER>(me);
            const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
            for (uint64_t todo = __ballot(e0 < N); todo;) {
                const int l = __ffsll((unsigned long long)todo) - 1;
                const int32_t u0 = __builtin_amdgcn_readlane(s0, l), u1 = __builtin_amdgcn_readlane(s1, l);
                const uint64_t group = __ballot(s0 == u0 && e0 < N);
                todo &= ~group;
                if (u1 - u0 > PS_GIANT) continue;
                int p = 0;  // place among the wavefront's galaxies of this pixel
                for (uint64_t m = group; m; m &= m - 1) {
                    const int j = __ffsll((unsigned long long)m) - 1;
                    const RankKey o{(uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)(k.a >> 32), j) << 32 |
                                        (uint32_t)__builtin_amdgcn_readlane((int)k.a, j),
                                    (uint32_t)__builtin_amdgcn_readlane((int)k.b, j)};
                    p += rank_less(o, k);
                }
                own_a[wv][lane] = ~0ull;
                own_b[wv][lane] = ~0u;
                hist[wv][lane] = 0;
                wave_lds_sync();
                if (group >> lane & 1) {
                    own_a[wv][p] = k.a;
                    own_b[wv][p] = k.b;
                }
                wave_lds_sync();
                CatSlot nx = slot[min((uint32_t)(u0 + lane), (uint32_t)u1 - 1)];
                for (uint32_t c = (uint32_t)u0; c < (uint32_t)u1; c += 64) {
                    const RankKey o = rank_key<ORDER>(nx);
                    nx = slot[min(c + 64u + lane, (uint32_t)u1 - 1)];  // the next 64 in flight
                    int at = 0;  // own galaxies up to o
#pragma unroll
                    for (int step = 32; step > 0; step >>= 1)
                        at += rank_less(o, {own_a[wv][at + step - 1], own_b[wv][at + step - 1]}) ? 0 : step;
                    at += !rank_less(o, {own_a[wv][at], own_b[wv][at]});
                    if (c + lane < (uint32_t)u1 && at < 64) atomicAdd(&hist[wv][at], 1u);
                }
                wave_lds_sync();
                int32_t inc = (int32_t)hist[wv][lane];
                for (int o = 1; o < 64; o <<= 1) {
                    const int32_t v = __shfl_up(inc, o, 64);
                    if (lane >= o) inc += v;
                }
                inc = __shfl(inc, p, 64);
                if (group >> lane & 1) before = inc;
                wave_lds_sync();
            }
        }
        if (s1 - s0 <= PS_CROWD) f = (int64_t)s0 + before;  // (fuller: as placed, the call is redone)
    }
    if (e0 < N && !giant) {
        idx[f] = me.i;
        pix_s[f] = me.pix;
        r_s[f] = me.r;
        w_s[f] = me.w;
    }
    if (ORDER && giants) {
        __syncthreads();  // the wavefronts' use of the LDS
        for (int q = 0; q < 8; ++q) {
            const int32_t e1 = lead[q >> 1][q & 1];
            if (e1 < 0) continue;
            const uint32_t p1 = slot[e1].pix >> sh;
            rank_block<ORDER>(slot, e1, pstart[p1], pstart[p1 + 1], lds, idx, pix_s, r_s, w_s);
        }
    }
}

// Slices of the sliced layout from the counts: one block per window of SELL_SIGMA pixels orders
// them by count (descending) with a counting sort in LDS and writes the slices' lanes, widths and
// emptiest lanes.  Pixels of one count come in any order: a pixel's sum does not depend on its
// slot, and the slices' widths only on the counts' order.  (A bitonic sort of (count, pixel) keys,
// 55 barriers, ran 11 us; it stays for windows with a pixel of 1024 galaxies or more.)
__global__ __launch_bounds__(1024) void k_sell_window(int64_t npix, int32_t nslice, const int32_t* __restrict__ pstart,
                                                      int64_t* __restrict__ width, uint32_t* __restrict__ invperm,
                                                      int2* __restrict__ pinfo, int32_t* __restrict__ smin)
{
    static_assert(SELL_SIGMA == 1024, "one thread per pixel of a window");
    __shared__ int32_t bin[1024];   // pixels per bin (bin 0: the largest counts), then the bins' starts
    __shared__ int32_t wsum[16];
    __shared__ int32_t big;         // the window's largest count
    __shared__ int2 lane_pc[1024];  // (pixel, count) by position
    const int t = threadIdx.x, lane = t & 63, wv = t >> 6;
    const int64_t p0 = (int64_t)blockIdx.x * 1024;
    const bool in = p0 + t < npix;
    const int32_t c0 = in ? pstart[p0 + t + 1] - pstart[p0 + t] : 0;
    bin[t] = 0;
    lane_pc[t] = make_int2(0, 0);  // lanes past the last pixel: no pixel, no galaxies
    if (t == 0) big = 0;
    __syncthreads();
    int32_t mx = c0;
    for (int o = 32; o > 0; o >>= 1) mx = max(mx, __shfl_xor(mx, o, 64));
    if (lane == 0) atomicMax(&big, mx);
    __syncthreads();
    if (big < 1024) {  // a bin per count
        const int32_t b = big - c0;
        int32_t rank = 0;
        if (in) rank = atomicAdd(&bin[b], 1);
        __syncthreads();
        const int32_t n = bin[t];
        int32_t inc = n;
        for (int o = 1; o < 64; o <<= 1) {
            const int32_t v = __shfl_up(inc, o, 64);
            if (lane >= o) inc += v;
        }
        if (lane == 63) wsum[wv] = inc;
        __syncthreads();
        int32_t base = 0;
        for (int i = 0; i < wv; ++i) base += wsum[i];
        bin[t] = base + inc - n;
        __syncthreads();
        if (in) {
            const int32_t at = bin[b] + rank;
            lane_pc[at] = make_int2((int)(p0 + t), c0);
            invperm[p0 + t] = (uint32_t)(p0 + at);
        }
    } else {  // crowded: (count, pixel) keys by a bitonic sort
        uint32_t* key = (uint32_t*)bin;
        key[t] = in ? ((uint32_t)(0x1fffff - min(c0, 0x1fffff)) << 10) | (uint32_t)t : 0xffffffffu;
        __syncthreads();
        for (int k = 2; k <= 1024; k <<= 1)
            for (int j = k >> 1; j > 0; j >>= 1) {
                const int o = t ^ j;
                if (o > t) {
                    const uint32_t a = key[t], b = key[o];
                    if ((a > b) == ((t & k) == 0)) {
                        key[t] = b;
                        key[o] = a;
                    }
                }
                __syncthreads();
            }
        if (key[t] != 0xffffffffu) {
            const int l = (int)(key[t] & 1023u);
            lane_pc[t] = make_int2((int)(p0 + l), pstart[p0 + l + 1] - pstart[p0 + l]);
            invperm[p0 + l] = (uint32_t)(p0 + t);
        }
    }
    __syncthreads();
    const int64_t e = p0 + t;
    const int32_t s = (int32_t)(e >> 6);
    if (s >= nslice) return;  // whole wavefronts leave together
    const int2 pc = lane_pc[t];
    pinfo[e] = pc;
    int32_t c = pc.y, cmin = pc.y;
    for (int o = 32; o > 0; o >>= 1) {
        c = max(c, __shfl_xor(c, o, 64));
        cmin = min(cmin, __shfl_xor(cmin, o, 64));
    }
    if (lane == 0) {
        width[s] = 64 * (int64_t)c;
        smin[s] = cmin;
    }
}
