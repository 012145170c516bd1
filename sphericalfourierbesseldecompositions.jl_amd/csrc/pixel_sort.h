// Galaxies grouped by pixel with counting kernels: count (the atomic's return value is the
// galaxy's arrival rank in its pixel), scan, place, and a rank pass that puts every pixel's
// galaxies into a fixed order, so the result does not depend on the atomics' order.  Seven
// dispatches where two stable radix sorts took forty: the catalogue stage of a small call is
// launch-bound (1e5 galaxies at nside 32: ~49 dispatches of 3-7 us each).
//
// The rank pass compares a pixel's galaxies pairwise, so it is for pixels of up to PS_CROWD
// galaxies; a fuller one raises flag[2] bit 1 and the call is redone with the radix sorts
// (which the plan then keeps).
#pragma once

constexpr int PS_CROWD = 512;     // galaxies per pixel the pairwise rank takes
constexpr int PS_MEAN = 96;       // mean galaxies per pixel above which the radix sorts run at once
constexpr int PS_CHUNK = 2048;    // pixels per scan block
constexpr int PS_SMALL = 32;      // scan blocks up to which each adds up the counts before it itself

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

// Arrival rank in a cell.  Atomics on one address take 7 ns each, one after another, so where
// several lanes of a wavefront share a cell (a crowded or an ordered catalogue; four lanes are
// tried) one lane adds for all of its cell.
__device__ __forceinline__ uint32_t arrival_rank(int32_t* __restrict__ cnt, uint32_t cell)
{
    const uint64_t live = __ballot(1);
    const int lane = threadIdx.x & 63, nl = __popcll(live);  // lanes 0 .. nl - 1
    bool shared = false;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const uint32_t c = (uint32_t)__builtin_amdgcn_readlane((int)cell, (j * nl) >> 2);
        shared |= __popcll(__ballot(cell == c)) > 1;
    }
    if (!shared) return (uint32_t)atomicAdd(cnt + cell, 1);
    uint64_t mine = 0;
    for (uint64_t todo = live; todo;) {
        const uint32_t c = (uint32_t)__builtin_amdgcn_readlane((int)cell, __ffsll((unsigned long long)todo) - 1);
        const uint64_t same = __ballot(cell == c);
        if (cell == c) mine = same;
        todo &= ~same;
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

// order inside a pixel: 0 as placed (where any order does), 1 by input index, 2 by (r, input
// index), the order of the reference's sums; in a folded pixel northern galaxies first, as the
// radix sorts leave them.  Writes the sorted list of input indices, and
// pixel, r and w in that order.
template <int ORDER>
__global__ __launch_bounds__(256) void k_rank(int64_t N, const CatSlot* __restrict__ slot,
                                              const int32_t* __restrict__ pstart, int32_t sh,
                                              uint32_t* __restrict__ idx,
                                              uint32_t* __restrict__ pix_s, double* __restrict__ r_s,
                                              double* __restrict__ w_s)
{
    const int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= N) return;
    const CatSlot me = slot[e];
    int64_t f = e;
    if (ORDER) {
        const int32_t s0 = pstart[me.pix >> sh], s1 = pstart[(me.pix >> sh) + 1];
        if (s1 - s0 <= PS_CROWD) {  // (fuller: the call is redone)
            const uint64_t k = sortable_bits(me.r);
            int32_t before = 0;
            for (int32_t s = s0; s < s1; ++s) {
                const uint32_t i = slot[s].i, ps = slot[s].pix;
                if (ORDER == 2) {
                    const uint64_t ks = sortable_bits(slot[s].r);
                    before += ps < me.pix || (ps == me.pix && (ks < k || (ks == k && i < me.i)));
                } else {
                    before += ps < me.pix || (ps == me.pix && i < me.i);
                }
            }
            f = (int64_t)s0 + before;
        }
    }
    idx[f] = me.i;
    pix_s[f] = me.pix;
    r_s[f] = me.r;
    w_s[f] = me.w;
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
