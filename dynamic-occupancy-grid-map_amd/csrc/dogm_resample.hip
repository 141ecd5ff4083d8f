// Multinomial resampling on gfx950 (dogm/src/dogm.cu:386-423, resampling.cu:17-68).
//
// 1. Exact CDF over [posterior weights | birth weights]: tile totals and their scan give the
//    inclusive CDF value at the end of every 256-entry segment (the coarse index, four per
//    1024-entry scan tile); entries are not stored but recomputed per staged segment in the merge.
// 2. Sorted uniforms by exponential spacings: E_k for k = 0..N, exact prefix S_k, draw k is the
//    fraction S_k / S_N of the CDF total (spacing_draw in dogm_numerics.h).  Only the tile totals of E are
//    stored; the merge kernel regenerates E from the counter-based RNG (four E per Philox call).
// 3. Merge: a workgroup owns 1024 consecutive (hence sorted) draws.  Its ancestors lie between the
//    CDF segments holding its first and last draw; those are found by a two-level k-ary search over
//    the coarse index (two dependent loads instead of a 22-level binary search), the CDF entries of
//    those segments are rebuilt from the weights as 31-bit keys relative to the window (one wave per
//    segment), and every draw finds its ancestor among the keys (the reference's lower_bound); the few
//    draws whose key does not decide are resolved exactly.  The reference's resamplingKernel gather is
//    deferred: only the ancestors (and the new weight) are written, the next full step's prediction
//    reads each state through its ancestor, and anything else that reads the particles first has
//    k_materialize copy them.
// No atomics on global memory and no global sort: the result is a pure function of the inputs.
// Every vehicle of a step resamples from its own CDF with its own draws.
#include "dogm_device.h"

namespace dogm_hip
{

constexpr int RS_ITEMS = 4;
constexpr int RS_TILE = BLOCK * RS_ITEMS;  // draws per workgroup
// CDF entries staged in LDS per window: 8 segments (2048 entries, the built-in choice: 1024 draws mostly need one
// window) or 4 (the other choice of the tuning, 1% slower per step of 32 x 2e6 particles).  The float
// modes stage whole tiles (RS_FLOAT_SLICE_TILES per window).
constexpr int RS_WINDOW_NARROW = 4;
constexpr int RS_WINDOW_WIDE = 8;
constexpr int RS_FLOAT_SLICE_TILES = 2;
// Doubles per scan tile in the float modes' index (the envelope at the tile end and before it),
// spaced like the exact mode's segment ends so that vehicles of both kinds in one step keep
// disjoint index ranges.
constexpr int ENV_STRIDE = 2 * CDF_SEGS_PER_TILE;
// Doubles per scan tile in the float modes' tile totals, which lie in scan_tile_sum beside the exact
// vehicles' fixed-point prefixes.
constexpr int FSUM_STRIDE = sizeof(fx_t) / sizeof(double);

static_assert(RS_TILE == SCAN_TILE, "draw tiles and CDF tiles share the exact-scan tile size");

// What the merge's window keys cover: joint weights below 2^37 and a CDF below 2^38.  Four such weights (a thread's) sum
// to less than 2^39, so the first prefix outside the range shows as one at or above 2^38 or, wrapped, below 0.
constexpr float KEY_WEIGHT_MAX = 0x1p37f;

__device__ __forceinline__ bool beyond_keys(fx_t prefix)
{
    return (prefix >> (38 + FX_FRAC)) != 0;
}

struct SrcJointPos
{
    static constexpr bool kNonNeg = true;  // cdf_weight: +0 or positive
    DevScalars* scs;                       // null where the weights are only read again
    // Marks a vehicle beyond the keys (k_scan_top_resample clears the mark).
    __device__ void seen(int vehicle, const float (&v)[4], fx_t incl) const
    {
        if (fmaxf(fmaxf(v[0], v[1]), fmaxf(v[2], v[3])) >= KEY_WEIGHT_MAX || beyond_keys(incl))
            scs[vehicle].beyond_tiles = 1;
    }
    __device__ bool active(const VehDesc& d) const { return d.cdf_mode == CDF_EXACT; }
    __device__ int len(const VehDesc& d) const { return d.N + d.B; }
    __device__ void load4(const VehDesc& d, int p0, int cnt, float (&v)[4]) const
    {
        const int N = d.N;
        if (p0 + cnt <= N)
            load_run<4>(d.weight_array, p0, cnt, v);
        else if (p0 >= N && ((p0 - N) & 3) == 0)
            load_run<4>(d.birth.weight, p0 - N, cnt, v);
        else
        {
#pragma unroll
            for (int i = 0; i < 4; ++i)
                v[i] = i < cnt ? (p0 + i < N ? d.weight_array[p0 + i] : d.birth.weight[p0 + i - N]) : 0.0f;
        }
#pragma unroll
        for (int i = 0; i < 4; ++i)
            v[i] = cdf_weight(v[i]);
    }
};

// The spacings' exact prefixes S_k of the thread's four consecutive draws k = base + 4 threadIdx.x .. + 3, each
// handed to put(i, S_k) (multinomial draws; all threads of the workgroup call it).  Inside the workgroup's 1024
// draws the exponentials are summed in 64-bit units of 2^-48; the tile's prefix joins in 128 bits.
template <class Put>
__device__ __forceinline__ void spacing_prefixes(const VehDesc& d, int base, int n,
                                                 const fx_t* __restrict__ exp_tile_pre, const Put& put)
{
    __shared__ uint64_t s_w[BLOCK / WAVE];
    const int q0 = base + threadIdx.x * RS_ITEMS;
    float f[RS_ITEMS];
    resample_exponentials4(d.seed, d.inst, d.ep_rs, (uint32_t)(q0 >> 2), f);
    uint64_t e[RS_ITEMS];
    uint64_t sum = 0;
#pragma unroll
    for (int i = 0; i < RS_ITEMS; ++i)
    {
        e[i] = q0 + i < n ? exp_units(f[i]) : 0;
        sum += e[i];
    }
    const int lane = threadIdx.x & (WAVE - 1), wid = threadIdx.x / WAVE;
    const uint64_t incl = wave_inclusive_scan_u64(sum);
    if (lane == WAVE - 1)
        s_w[wid] = incl;
    __syncthreads();
    uint64_t run = incl - sum;
#pragma unroll
    for (int w = 0; w < BLOCK / WAVE - 1; ++w)
        run += w < wid ? s_w[w] : 0;
    const fx_t pre = exp_tile_pre[d.u0[SP_E] / SCAN_Q + base / RS_TILE];
#pragma unroll
    for (int i = 0; i < RS_ITEMS; ++i)
    {
        run += e[i];
        put(i, pre + fx_from_exp_units(run));
    }
}

// ---------------------------------------------------------------------------------------------
// Float CDF modes (precision study).  Per tile of 1024 joint weights: 4-element sequential folds
// per thread, the 64-lane DPP wave scan, sequential carries across the 4 waves, and a sequential
// prefix over the vehicle's tiles; element = ((tile prefix + wave carry) + thread's exclusive wave
// prefix) + thread-local prefix.  The running maximum (monotone envelope) is what the ancestor
// search sees.  The CDF is stored as doubles in the vehicle's CDF buffer; per tile, the coarse
// index holds (envelope at the tile end, envelope before the tile) as two doubles.
// ---------------------------------------------------------------------------------------------
template <class T>
struct CdfFloatMode;
template <>
struct CdfFloatMode<double>
{
    static constexpr int mode = CDF_FP64;
};
template <>
struct CdfFloatMode<float>
{
    static constexpr int mode = CDF_FP32;
};
template <>
struct CdfFloatMode<f32c>
{
    static constexpr int mode = CDF_FP32C;
};

// Thread fold, wave scan and wave carries of one tile: the thread's local prefixes, its wave
// carry (sum of the earlier waves' totals), its exclusive prefix inside the wave, and the tile total
// (on every thread).
template <class T>
__device__ __forceinline__ void tile_float_scan(const VehDesc& d, int p0, int cnt, T (&loc)[4], T* carry_out,
                                                T* excl_out, T* tile_total)
{
    __shared__ T s_w[BLOCK / WAVE];
    float f[4] = {0.0f, 0.0f, 0.0f, 0.0f};
    if (cnt > 0)
        SrcJointPos{nullptr}.load4(d, p0, cnt, f);
    T run = (T)0;
#pragma unroll
    for (int i = 0; i < 4; ++i)
    {
        run = run + (T)(i < cnt ? f[i] : 0.0f);
        loc[i] = run;
    }
    const int lane = threadIdx.x & (WAVE - 1);
    const int wid = threadIdx.x / WAVE;
    const T incl = wave_inclusive_scan_val(run);
    T excl = shfl_up1(incl);
    if (lane == 0)
        excl = (T)0;
    if (lane == WAVE - 1)
        s_w[wid] = incl;
    __syncthreads();
    T carry = (T)0;
    for (int w = 0; w < wid; ++w)
        carry = carry + s_w[w];
    T tot = (T)0;
#pragma unroll
    for (int w = 0; w < BLOCK / WAVE; ++w)
        tot = tot + s_w[w];
    __syncthreads();
    *carry_out = carry;
    *excl_out = excl;
    *tile_total = tot;
}

template <class T>
__global__ __launch_bounds__(BLOCK) void k_cdff_tiles(const VehDesc* __restrict__ descs,
                                                      const uint32_t* __restrict__ tab, double* __restrict__ tile_sum)
{
    const TileRef tr = tile_ref(tab, SCAN_Q, blockIdx.x);
    const VehDesc& d = descs[tr.v];
    if (d.cdf_mode != CdfFloatMode<T>::mode)
        return;
    const int n = d.N + d.B;
    const int p0 = tr.base + threadIdx.x * SCAN_ITEMS;
    const int cnt = max(0, min(SCAN_ITEMS, n - p0));
    T loc[4];
    T carry, ex, tot;
    tile_float_scan<T>(d, p0, cnt, loc, &carry, &ex, &tot);
    if (threadIdx.x == 0)
        tile_sum[FSUM_STRIDE * (size_t)blockIdx.x] = (double)tot;
}

// One workgroup per vehicle: sequential prefix over the vehicle's tile totals (the association of the float
// modes).  The additions are one dependent chain, so one thread does them; the others stage
// the totals in LDS and write the prefixes out, so that the chain waits for LDS reads issued ahead
// of it and not for one memory round trip per tile.  8600 tiles (2048^2 cells, 8e6 + 8e5 weights): FP64 692 us
// with every load and store in the chain, 124 us staged.
template <class T>
__global__ __launch_bounds__(BLOCK) void k_cdff_top(const VehDesc* __restrict__ descs,
                                                    const double* __restrict__ tile_sum, double* __restrict__ tile_pre)
{
    constexpr int CHUNK = 2048;  // totals staged at once
    constexpr int STEP = 16;     // totals read ahead of the chain
    __shared__ double s_x[CHUNK];
    const VehDesc& d = descs[blockIdx.x];
    if (d.cdf_mode != CdfFloatMode<T>::mode)
        return;
    const int t0 = d.u0[SP_J] / SCAN_Q;
    const int nt = d.nu[SP_J] / SCAN_Q;
    T run = (T)0;
    for (int c = 0; c < nt; c += CHUNK)
    {
        const int len = min(CHUNK, nt - c);
        __syncthreads();
        for (int i = threadIdx.x; i < CHUNK; i += BLOCK)
            s_x[i] = i < len ? tile_sum[FSUM_STRIDE * (size_t)(t0 + c + i)] : 0.0;
        __syncthreads();
        if (threadIdx.x == 0)
        {
            double x[STEP];
#pragma unroll
            for (int k = 0; k < STEP; ++k)
                x[k] = s_x[k];
            for (int i = 0; i < len; i += STEP)  // past len: zeros, whose prefixes are not written out
            {
                double next[STEP];
                const int n0 = min(i + STEP, CHUNK - STEP);
#pragma unroll
                for (int k = 0; k < STEP; ++k)
                    next[k] = s_x[n0 + k];
#pragma unroll
                for (int k = 0; k < STEP; ++k)
                {
                    const T before = run;
                    run = run + (T)x[k];
                    s_x[i + k] = (double)before;
                }
#pragma unroll
                for (int k = 0; k < STEP; ++k)
                    x[k] = next[k];
            }
        }
        __syncthreads();
        for (int i = threadIdx.x; i < len; i += BLOCK)
            tile_pre[t0 + c + i] = s_x[i];
    }
}

// Values, the envelope inside the tile, and the tile maximum (into env[ENV_STRIDE t]).
template <class T>
__global__ __launch_bounds__(BLOCK) void k_cdff_apply(const VehDesc* __restrict__ descs,
                                                      const uint32_t* __restrict__ tab,
                                                      const double* __restrict__ tile_pre, double* __restrict__ env)
{
    __shared__ T s_m[BLOCK / WAVE];
    const TileRef tr = tile_ref(tab, SCAN_Q, blockIdx.x);
    const VehDesc& d = descs[tr.v];
    if (d.cdf_mode != CdfFloatMode<T>::mode)
        return;
    const int n = d.N + d.B;
    const int p0 = tr.base + threadIdx.x * SCAN_ITEMS;
    const int cnt = max(0, min(SCAN_ITEMS, n - p0));
    T loc[4];
    T carry, ex, tot;
    tile_float_scan<T>(d, p0, cnt, loc, &carry, &ex, &tot);
    const T tp = (T)tile_pre[blockIdx.x];
    const int wid = threadIdx.x / WAVE;
    const T base = (tp + carry) + ex;
    T val[4];
    T mx = (T)0;
#pragma unroll
    for (int i = 0; i < 4; ++i)
    {
        val[i] = base + loc[i];
        if (i < cnt && val[i] > mx)
            mx = val[i];
    }
    // Exclusive running maximum over the earlier threads of the tile.
    const T wmax = wave_inclusive_max_val(mx);
    T before = shfl_up1(wmax);
    if ((threadIdx.x & (WAVE - 1)) == 0)
        before = (T)0;
    if ((threadIdx.x & (WAVE - 1)) == WAVE - 1)
        s_m[wid] = wmax;
    __syncthreads();
    for (int w = 0; w < wid; ++w)
        before = s_m[w] > before ? s_m[w] : before;
    T tmax = (T)0;
#pragma unroll
    for (int w = 0; w < BLOCK / WAVE; ++w)
        tmax = s_m[w] > tmax ? s_m[w] : tmax;
    double* cdf = reinterpret_cast<double*>(d.cdf.get());
#pragma unroll
    for (int i = 0; i < 4; ++i)
    {
        if (i < cnt)
        {
            const T e = val[i] > before ? val[i] : before;
            cdf[p0 + i] = (double)e;
            before = e;
        }
    }
    if (threadIdx.x == 0)
        env[ENV_STRIDE * (size_t)blockIdx.x] = (double)tmax;
}

// One workgroup per vehicle: the envelope across tiles, the total and the new particle weight.  The
// running maximum is exact in any order, so each thread takes a contiguous run of tiles and a block scan
// joins them (a tile maximum that is not above 0, NaN among them, leaves the envelope unchanged).
// 8600 tiles: 20 us, against 1628 us for one thread walking the tiles.
constexpr int ENV_BLOCK = 1024;

__global__ __launch_bounds__(ENV_BLOCK) void k_cdff_env(const VehDesc* __restrict__ descs, double* __restrict__ env,
                                                        DevScalars* __restrict__ scs)
{
    __shared__ double s_m[ENV_BLOCK / WAVE];
    const int v = blockIdx.x;
    const VehDesc& d = descs[v];
    if (d.cdf_mode == CDF_EXACT)
        return;
    const int t0 = d.u0[SP_J] / SCAN_Q;
    const int nt = d.nu[SP_J] / SCAN_Q;
    const int per = (nt + ENV_BLOCK - 1) / ENV_BLOCK;
    const int b0 = min(nt, (int)threadIdx.x * per), b1 = min(nt, b0 + per);
    double mx = 0.0;
#pragma unroll 4
    for (int t = b0; t < b1; ++t)
    {
        const double tm = env[ENV_STRIDE * (size_t)(t0 + t)];
        mx = tm > mx ? tm : mx;
    }
    const int lane = threadIdx.x & (WAVE - 1), wid = threadIdx.x / WAVE;
    const double wmax = wave_inclusive_max_val(mx);
    double run = shfl_up1(wmax);
    if (lane == 0)
        run = 0.0;
    if (lane == WAVE - 1)
        s_m[wid] = wmax;
    __syncthreads();
    double total = 0.0;
#pragma unroll
    for (int w = 0; w < ENV_BLOCK / WAVE; ++w)
    {
        const double x = s_m[w];
        if (w < wid)
            run = x > run ? x : run;
        total = x > total ? x : total;
    }
    for (int t = b0; t < b1; ++t)
    {
        double* e = env + ENV_STRIDE * (size_t)(t0 + t);
        const double tm = e[0];
        e[1] = run;
        run = tm > run ? tm : run;
        e[0] = run;
    }
    if (threadIdx.x == 0)
    {
        DevScalars* sc = scs + v;
        sc->ftotal = total;
        const float jm = (float)total;
        sc->new_weight = jm / (float)d.N;
    }
}

// Ancestor search over the float modes' envelope (doubles): the draw, the coarse index entry of a
// tile and a staged CDF value.
struct CdfFloatTr
{
    using V = double;
    __device__ static bool takes(const VehDesc& d) { return d.cdf_mode != CDF_EXACT; }
    __device__ static V draw(fx_t s_k, const Spacing& sp, const DevScalars* sc, int mode)
    {
        return cdf_float_draw(sc->ftotal, spacing_fraction(s_k, sp), mode);
    }
    __device__ static V incl(const void* ci, int t0, int t)
    {
        return static_cast<const double*>(ci)[ENV_STRIDE * (size_t)(t0 + t)];
    }
    __device__ static V value(const VehDesc& d, const void* ci, int t0, int j)
    {
        const double c = reinterpret_cast<const double*>(d.cdf.get())[j];
        const double b = static_cast<const double*>(ci)[ENV_STRIDE * (size_t)(t0 + j / SCAN_TILE) + 1];
        return c > b ? c : b;
    }
};

// Envelope entries staged in LDS (float modes).  Entry i sits at slot i + i / 32.
template <int LEN>
struct CdfStage
{
    double v[LEN + LEN / 32];
    __device__ static int slot(int i) { return i + (i >> 5); }
    __device__ void put(int i, double x) { v[slot(i)] = x; }
    __device__ double get(int i) const { return v[slot(i)]; }
    __device__ bool less(int i, double r) const { return v[slot(i)] < r; }
};

// Index of the first of n non-decreasing values value(0 .. n-1) that is >= r (n - 1 if none): a
// two-level k-ary search by the workgroup (the last value of each of up to BLOCK groups, then the
// values of one group).
template <class V, class Get>
__device__ int find_first_not_below(const Get& value, int n, V r, int* s_cnt)
{
    const int G = (n + BLOCK - 1) / BLOCK;  // values per group; at most BLOCK groups
    const int ng = (n + G - 1) / G;
    if (threadIdx.x == 0)
        s_cnt[0] = 0;
    __syncthreads();
    const int i = threadIdx.x;
    const bool below = i < ng && value(min(n - 1, (i + 1) * G - 1)) < r;
    const int groups_below = __syncthreads_count(below);
    const int g = min(groups_below, ng - 1);
    for (int j = threadIdx.x; j < G; j += BLOCK)
    {
        const int t = g * G + j;
        if (t < n && value(t) < r)
            atomicAdd(&s_cnt[0], 1);
    }
    __syncthreads();
    const int t = min(g * G + s_cnt[0], n - 1);
    __syncthreads();
    return t;
}

// The workgroup's draws r_k, k = base + threadIdx.x + i * BLOCK, in the float modes (item i of a thread is
// strided, so at every item a wave searches 64 consecutive draws), and s_rb = {first draw, last draw}.
template <class Draw, class Stage>
__device__ __forceinline__ void merge_draws(const VehDesc& d, const DevScalars* sc, int base, int n,
                                            const fx_t* __restrict__ exp_tile_pre, const Draw& draw, Stage& stage,
                                            double (&r)[RS_ITEMS], double* s_rb)
{
    const int last = min(base + RS_TILE, n) - 1;
    const Spacing sp = sc->spacing;
    if (d.draw_mode == DRAW_SYSTEMATIC)
    {
        const uint32_t u = systematic_u32(d.seed, d.inst, d.ep_rs);
#pragma unroll
        for (int i = 0; i < RS_ITEMS; ++i)
            r[i] = draw(systematic_s(base + (int)threadIdx.x + i * BLOCK, u), sp);
    }
    else
    {
        spacing_prefixes(d, base, n, exp_tile_pre,
                         [&](int i, fx_t s_k) { stage.put(threadIdx.x * RS_ITEMS + i, draw(s_k, sp)); });
        __syncthreads();
#pragma unroll
        for (int i = 0; i < RS_ITEMS; ++i)
            r[i] = stage.get(threadIdx.x + i * BLOCK);
    }
#pragma unroll
    for (int i = 0; i < RS_ITEMS; ++i)
    {
        const int k = base + (int)threadIdx.x + i * BLOCK;
        if (k == base)
            s_rb[0] = r[i];
        if (k == last)
            s_rb[1] = r[i];
    }
    __syncthreads();
}

// The smallest draw of the workgroup that has no ancestor yet (n if none), and its value in s_rb[0].
template <class V>
__device__ __forceinline__ int merge_next_draw(int base, int n, const int (&anc)[RS_ITEMS], const V (&r)[RS_ITEMS],
                                               int* s_kmin, V* s_rb)
{
    if (threadIdx.x == 0)
        *s_kmin = n;
    __syncthreads();
    int mine = n;
#pragma unroll
    for (int i = RS_ITEMS - 1; i >= 0; --i)
        if (anc[i] < 0 && base + (int)threadIdx.x + i * BLOCK < n)
            mine = base + (int)threadIdx.x + i * BLOCK;
    if (mine < n)
        atomicMin(s_kmin, mine);
    __syncthreads();
    const int kmin = *s_kmin;
    if (kmin < n)
    {
#pragma unroll
        for (int i = 0; i < RS_ITEMS; ++i)
            if (base + (int)threadIdx.x + i * BLOCK == kmin)
                s_rb[0] = r[i];
    }
    __syncthreads();
    return kmin;
}

// The resampled particles k = base + threadIdx.x + i * BLOCK, left by reference: the ancestor index (a draw
// without an ancestor, above the CDF total by rounding, takes the last joint entry) and the uniform new weight in
// weight[0].  The next full step's prediction reads the states through the ancestors, and every other reader first
// writes the set out (k_materialize).
__device__ __forceinline__ void merge_write(const VehDesc& d, const DevScalars* sc, int pph, int base, int n, int J,
                                            const int (&anc)[RS_ITEMS])
{
#pragma unroll
    for (int i = 0; i < RS_ITEMS; ++i)
    {
        const int k = base + i * BLOCK + (int)threadIdx.x;
        if (k < n)
            d.ancestors[k] = anc[i] < 0 ? J - 1 : min(anc[i], J - 1);
    }
    if (base == 0 && threadIdx.x == 0)
        d.part[pph ^ 1].weight[0] = sc->new_weight;
}

// Index of the first of n non-decreasing values value(0 .. n-1) that is >= r (n - 1 if none), for
// two values at once, found by one wave without a barrier: the lanes probe every s-th value (s =
// ceil(n / 64)); the probes below r form a prefix of k lanes, so the answer lies in [k s, (k + 1) s),
// whose values below r are then counted (ceil(s / 64) probes per lane).
template <class V, class Get>
__device__ __forceinline__ void wave_find2(const Get& value, int n, V r0, V r1, int* c0, int* c1)
{
    const int lane = threadIdx.x & (WAVE - 1);
    const int s = (n + WAVE - 1) / WAVE;
    const V p = value(min(n - 1, (lane + 1) * s - 1));
    const int b0 = __popcll(__ballot(p < r0)) * s;
    const int b1 = __popcll(__ballot(p < r1)) * s;
    int n0 = 0, n1 = 0;
    for (int q0 = 0; q0 < s; q0 += WAVE)
    {
        const int q = q0 + lane;
        const bool in0 = q < s && b0 + q < n, in1 = q < s && b1 + q < n;
        const V v0 = in0 ? value(b0 + q) : V(0), v1 = in1 ? value(b1 + q) : V(0);
        n0 += __popcll(__ballot(in0 && v0 < r0));
        n1 += __popcll(__ballot(in1 && v1 < r1));
    }
    *c0 = min(b0 + n0, n - 1);
    *c1 = min(b1 + n1, n - 1);
}

// The CDF in raw fixed-point units (value * 2^88) as a double; exact below 2^53 raw units.
__device__ __forceinline__ double fx_raw_f64(fx_t v)
{
    return fx_to_f64(v) * 0x1p88;
}

// A draw in raw units (an integer) as a fixed-point value.
__device__ __forceinline__ fx_t raw_fx(double raw)
{
    return fx_from_f64_nonneg(raw * 0x1p-88);
}

// Four joint weights in raw fixed-point units: fx_from_f32_nonneg as doubles (a 24-bit significand truncated to an
// integer), for weights below 2^39.
__device__ __forceinline__ void raw_weights(const float (&f)[SCAN_ITEMS], double (&v)[SCAN_ITEMS])
{
#pragma unroll
    for (int i = 0; i < SCAN_ITEMS; ++i)
        v[i] = trunc((double)f[i] * 0x1p88);
}

// The CDF index of a vehicle: the inclusive CDF value at the end of segment s, from the tile-local ends of
// the tile pass and the tiles' prefixes.
struct SegEnds
{
    const fx_t* local;     // [segments]
    const fx_t* tile_pre;  // [tiles]
    fx_t total;
    int tiles, segs;       // tiles and segments holding entries
    __device__ fx_t operator()(int s) const { return local[s] + tile_pre[s / CDF_SEGS_PER_TILE]; }

    // The first segments whose end is >= r0 and >= r1 (the last segment if none), by one wave without a barrier: a
    // search over the tile ends (each the next tile's prefix), then the ends inside the two tiles.
    __device__ void find2(fx_t r0, fx_t r1, int* s0, int* s1) const
    {
        const int lane = threadIdx.x & (WAVE - 1);
        const auto tile_end = [this](int t) { return t + 1 < tiles ? tile_pre[t + 1] : total; };
        int t0, t1;
        wave_find2<fx_t>(tile_end, tiles, r0, r1, &t0, &t1);
        // lanes 0 .. 3 hold the segment ends of tile t0, lanes 4 .. 7 those of t1
        const bool second = lane >= CDF_SEGS_PER_TILE;
        const int s = min((second ? t1 : t0) * CDF_SEGS_PER_TILE + (lane & (CDF_SEGS_PER_TILE - 1)), segs - 1);
        const uint64_t below = __ballot((*this)(s) < (second ? r1 : r0));
        *s0 = min(t0 * CDF_SEGS_PER_TILE + __popcll(below & 0xfull), segs - 1);
        *s1 = min(t1 * CDF_SEGS_PER_TILE + __popcll(below & 0xf0ull), segs - 1);
    }
};
static_assert(CDF_SEGS_PER_TILE == 4, "find2 tests a tile's segments with four lanes");

// First joint entry whose exact CDF value is >= r, by one wave: the coarse index gives the segment, the
// segment's entries are rebuilt exactly (the 64 lanes' four weights in fixed point, a 64-lane exact scan and the
// index entry before the segment) and those below r counted.
__device__ __forceinline__ int wave_exact_ancestor(const VehDesc& d, const SegEnds& seg_end, int J, fx_t r)
{
    const int lane = threadIdx.x & (WAVE - 1);
    int s, unused;
    seg_end.find2(r, r, &s, &unused);
    const int q0 = s * CDF_SEG + lane * SCAN_ITEMS;
    const int cnt = max(0, min(SCAN_ITEMS, J - q0));
    float f[SCAN_ITEMS] = {0.0f, 0.0f, 0.0f, 0.0f};
    if (cnt > 0)
        SrcJointPos{nullptr}.load4(d, q0, cnt, f);
    fx_t v[SCAN_ITEMS];
    fx_t sum = 0;
#pragma unroll
    for (int i = 0; i < SCAN_ITEMS; ++i)
    {
        v[i] = i < cnt ? fx_from_f32_nonneg(f[i]) : (fx_t)0;  // cdf_weight: sign bit clear
        sum += v[i];
    }
    fx_t run = wave_inclusive_scan_fx(sum) - sum + (s > 0 ? seg_end(s - 1) : (fx_t)0);
    int below = 0;
#pragma unroll
    for (int i = 0; i < SCAN_ITEMS; ++i)
    {
        run += v[i];
        below += __popcll(__ballot(i < cnt && run < r));
    }
    return s * CDF_SEG + below;
}

// The merge of a vehicle whose CDF is beyond the window keys (infinite weights count 2^38).  The 128-bit entries of
// `segs` segments (a window: 4 or 8) are rebuilt and searched, four segments at a time in the workgroup's 16 KB; a
// draw is resolved in the first window whose last entry is >= its value, by a branch-free binary search over
// the window padded to a power of two.  While the CDF is non-decreasing that is its lower bound.  Past the
// fixed-point range the sums wrap and the answer depends on the probes, so their order is fixed: the whole coarse
// index first, windows of a given length, halved from the front.  s_mem holds the workgroup's draws on entry.
// 2.2e5 joint weights, one of them infinite: 12.4 us (one by one, with wave_exact_ancestor, 457).
__device__ __forceinline__ void merge_beyond_keys(const VehDesc& d, const DevScalars* sc, const SegEnds& seg_end,
                                                  int pph, int base, int n, int J, int segs, uint64_t* s_mem)
{
    constexpr int NWAVE = BLOCK / WAVE;
    constexpr int HALF = NWAVE * CDF_SEG;  // entries staged at once, a segment per wave
    static_assert(HALF == RS_TILE, "the entries take the draws' bytes and as many again");
    __shared__ fx_t s_wr[NWAVE];
    __shared__ int s_wmin[NWAVE];
    int64_t* s_hi64 = reinterpret_cast<int64_t*>(s_mem);
    uint64_t* s_lo64 = s_mem + HALF;
    const double* s_r = reinterpret_cast<const double*>(s_mem);
    const int lane = threadIdx.x & (WAVE - 1), wid = wave_index();
    const auto put = [=](int i, fx_t x) {
        s_hi64[i] = (int64_t)(x >> 64);
        s_lo64[i] = (uint64_t)x;
    };
    const auto get = [=](int i) { return (fx_t)(((ufx_t)(uint64_t)s_hi64[i] << 64) | (ufx_t)s_lo64[i]); };
    const int last = min(base + RS_TILE, n) - 1;
    double r[RS_ITEMS];
    int anc[RS_ITEMS];
#pragma unroll
    for (int i = 0; i < RS_ITEMS; ++i)
    {
        r[i] = s_r[threadIdx.x + i * BLOCK];
        anc[i] = -1;
    }
    int s_lo, s_hi;
    wave_find2<fx_t>(seg_end, seg_end.segs, raw_fx(s_r[0]), raw_fx(s_r[last - base]), &s_lo, &s_hi);
    for (int s0 = s_lo; s0 <= s_hi;)
    {
        const int s1 = min(s0 + segs, s_hi + 1);  // window: segments [s0, s1)
        const int c0 = s0 * CDF_SEG;
        const int clen = min(J, s1 * CDF_SEG) - c0;
        const fx_t cmax = seg_end(s1 - 1), next_max = seg_end(min(s1 - 1 + segs, s_hi));
        const bool two = clen > HALF;
        const fx_t mid = two ? seg_end(s0 + NWAVE - 1) : (fx_t)0;  // entry HALF - 1: the first probe
        const int span = clen > 1 ? 1 << (32 - __clz(clen - 1)) : 1;
#pragma unroll 1
        for (int h = 0; h <= (two ? 1 : 0); ++h)
        {
            const int s = s0 + h * NWAVE + wid;
            const int q0 = s * CDF_SEG + lane * SCAN_ITEMS;
            float f[SCAN_ITEMS] = {0.0f, 0.0f, 0.0f, 0.0f};
            if (s < s1 && q0 < J)
                SrcJointPos{nullptr}.load4(d, q0, min(SCAN_ITEMS, J - q0), f);
            fx_t sum = 0;
#pragma unroll
            for (int i = 0; i < SCAN_ITEMS; ++i)
                sum += fx_from_f32_nonneg(f[i]);  // cdf_weight: sign bit clear; 0 past the entries
            fx_t run = wave_inclusive_scan_fx(sum) - sum + (s < s1 && s > 0 ? seg_end(s - 1) : (fx_t)0);
            __syncthreads();  // the searches (and the draws' staging) before are done
#pragma unroll
            for (int i = 0; i < SCAN_ITEMS; ++i)
            {
                run += fx_from_f32_nonneg(f[i]);
                put(wid * CDF_SEG + lane * SCAN_ITEMS + i, run);
            }
            __syncthreads();
#pragma unroll
            for (int i = 0; i < RS_ITEMS; ++i)
            {
                double raw = r[i];
                asm volatile("" : "+v"(raw));  // converted here and not once for all windows: four registers a draw less
                const fx_t ri = raw_fx(raw);
                const bool upper = two && mid < ri;
                if (anc[i] >= 0 || base + (int)threadIdx.x + i * BLOCK > last || cmax < ri || upper != (h != 0))
                    continue;
                // lo counts the entries below the draw; past the window the last entry stands for the ones missing.
                int lo = h * HALF;
                for (int step = two ? HALF / 2 : span >> 1; step > 0; step >>= 1)
                    if (get(min(lo + step, clen) - 1 - h * HALF) < ri)
                        lo += step;
                anc[i] = c0 + lo;
            }
        }
        if (s1 > s_hi)
            break;
        // The smallest unresolved draw: each wave's minimum (draw indices are distinct, so one lane holds it) with its
        // value, then the minimum over the waves.
        int mine = n;
        double rmine = 0.0;
#pragma unroll
        for (int i = RS_ITEMS - 1; i >= 0; --i)
        {
            const int k = base + (int)threadIdx.x + i * BLOCK;
            if (anc[i] < 0 && k <= last)
            {
                mine = k;
                rmine = r[i];
            }
        }
        int wmin = mine;
#pragma unroll
        for (int o = WAVE / 2; o > 0; o >>= 1)
            wmin = min(wmin, __shfl_xor(wmin, o, WAVE));
        if (wmin < n && mine == wmin)
            s_wr[wid] = raw_fx(rmine);
        if (lane == 0)
            s_wmin[wid] = wmin;
        __syncthreads();
        int kmin = n, kw = 0;
#pragma unroll
        for (int w = 0; w < NWAVE; ++w)
        {
            const int x = s_wmin[w];
            if (x < kmin)
            {
                kmin = x;
                kw = w;
            }
        }
        if (kmin >= n)
            break;
        const fx_t rmin = s_wr[kw];
        if (!(next_max < rmin))
        {
            s0 = s1;
        }
        else
        {
            int c, unused;
            wave_find2<fx_t>(seg_end, seg_end.segs, rmin, rmin, &c, &unused);
            s0 = max(s1, c);
        }
    }
    merge_write(d, sc, pph, base, n, J, anc);
}

// Exact-CDF merge.  The workgroup's ancestors lie in the CDF segments [s_lo, s_hi] holding its first and
// last draw; they are staged WSEG segments at a time (a window).  The answer is the exact lower bound in the 128-bit
// CDF, but nearly every comparison is decided by far fewer bits: a window stages one 31-bit key per entry,
// key(x) = floor((x - B0) 2^(30 - m)) with B0 the CDF before the window, W its exact total and m = msb(W), and
// the draws are compared by the same key.
//   - Weights, draws and their differences from B0 are formed in f64 in raw units (integers).  The rebuild's sums (a
//     wave scan of one segment from its exact index entry) are off by less than 2^-48 W.  B0 is subtracted in two
//     doubles, which hold it to 2^(msb(B0) - 106): at the smallest W that keys are used for (below) a draw's
//     difference is off by up to 2^-40 W, 2^-10 of a key.  Both keys are thus within 1 of the exact ones and two
//     keys at least 2 apart decide.  With W below 2^31 every value is an integer below 2^31 and the keys are exact.
//   - A draw within 1 of an entry's key (about 3e-6 of them: a window holds at most 2048 of 2^30 keys, and draws
//     fall in proportion to the CDF) is resolved by wave_exact_ancestor.
//   - A window whose total is below 2^-66 of a CDF above 2^107 raw units before it sends the draws that land in it
//     there (a draw lands in a window in proportion to its total).
//   - A vehicle with a weight of 2^37 or more, or with a CDF of 2^38 or more, may have sums that leave the fixed-point
//     range, which these bounds do not cover: merge_beyond_keys.
// Draws are sorted, so the resolved ones are a prefix: the next window starts at the segment of the first draw left.
// Bound by the vector ALU (Philox and logarithms of the draws, searches).  Before, windows held 128-bit
// entries (four 128-bit conversions and adds per lane and segment, 128-bit scans and two-word probes).
// 2e6 draws: 31.9 -> 22.1 us alone (3e5: 19.1 -> 15.2), 32 x 2e6 per step 3.4% off the whole step.
// Eight waves per SIMD are asked for: 64 vector and 78 scalar registers without memory spills; left to itself the
// compiler takes 99 scalar ones, and 16 x 2e6 draws 244 us instead of 221.
template <int WSEG>
__global__ __launch_bounds__(BLOCK, 8) void k_rs_merge_exact(const VehDesc* __restrict__ descs,
                                                          const uint32_t* __restrict__ tab, int pph,
                                                          const fx_t* __restrict__ exp_tile_pre,
                                                          const fx_t* __restrict__ seg_local,
                                                          const fx_t* __restrict__ cdf_pre,
                                                          const DevScalars* __restrict__ scs, int beyond_segs)
{
    constexpr int WLEN = WSEG * CDF_SEG;
    constexpr int NWAVE = BLOCK / WAVE;
    constexpr uint32_t PAD = 0xffffffffu;  // above every draw's key
    static_assert((WLEN & (WLEN - 1)) == 0, "the search halves the window");
    // The draws in raw units and the window's keys + margin; merge_beyond_keys takes the same bytes.
    constexpr int MEM = RS_TILE + WLEN / 2 > 2 * RS_TILE ? RS_TILE + WLEN / 2 : 2 * RS_TILE;
    __shared__ __attribute__((aligned(16))) uint64_t s_mem[MEM];
    double* s_r = reinterpret_cast<double*>(s_mem);
    uint32_t* s_key = reinterpret_cast<uint32_t*>(s_mem + RS_TILE);
    __shared__ int s_done[NWAVE];

    const TileRef tr = tile_ref(tab, RS_TILE / UNIT, blockIdx.x);
    const VehDesc& d = descs[tr.v];
    const int n = d.N;
    const int base = tr.base;
    if (base >= n || d.cdf_mode != CDF_EXACT)
        return;
    const DevScalars* sc = scs + tr.v;
    const int J = n + d.B;
    const int t0 = d.u0[SP_J] / SCAN_Q;
    const SegEnds seg_end{seg_local + (size_t)t0 * CDF_SEGS_PER_TILE, cdf_pre + t0, sc->cdf_total,
                          (J + SCAN_TILE - 1) / SCAN_TILE, (J + CDF_SEG - 1) / CDF_SEG};
    const int cnt_draws = min(RS_TILE, n - base);
    const int wid = threadIdx.x / WAVE;
    const int lane = threadIdx.x & (WAVE - 1);
    const Spacing sp = sc->spacing;
    // fx(total * u_k) as a double: the product truncated to an integer number of raw units.
    const auto raw_draw = [&sp](fx_t s_k) { return trunc(sp.total * spacing_fraction(s_k, sp) * 0x1p88); };
    if (d.draw_mode == DRAW_SYSTEMATIC)
    {
        const uint32_t u = systematic_u32(d.seed, d.inst, d.ep_rs);
#pragma unroll
        for (int i = 0; i < RS_ITEMS; ++i)
            s_r[threadIdx.x + i * BLOCK] = raw_draw(systematic_s(base + (int)threadIdx.x + i * BLOCK, u));
    }
    else
    {
        spacing_prefixes(d, base, n, exp_tile_pre,
                         [&](int i, fx_t s_k) { s_r[threadIdx.x * RS_ITEMS + i] = raw_draw(s_k); });
    }
    __syncthreads();
    if (sc->beyond_keys)
    {
        merge_beyond_keys(d, sc, seg_end, pph, base, n, J, beyond_segs, s_mem);
        return;
    }
    // Item i of a thread is draw base + threadIdx.x + i * BLOCK, so at every item a wave searches 64 consecutive draws,
    // whose probes read neighbouring keys, and the ancestors come out wave-contiguous.
    int anc[RS_ITEMS];
#pragma unroll
    for (int i = 0; i < RS_ITEMS; ++i)
        anc[i] = threadIdx.x + i * BLOCK < cnt_draws ? -1 : 0;
    int s_lo, s_hi;
    seg_end.find2(raw_fx(s_r[0]), raw_fx(s_r[cnt_draws - 1]), &s_lo, &s_hi);
    for (int s0 = s_lo;;)
    {
        const int s1 = min(s0 + WSEG, s_hi + 1);  // window: segments [s0, s1)
        const int c0 = s0 * CDF_SEG;
        const int clen = min(J, s1 * CDF_SEG) - c0;
        const fx_t B0 = s0 > 0 ? seg_end(s0 - 1) : (fx_t)0;
        const fx_t W = seg_end(s1 - 1) - B0;
        const int m = W > 0 ? 127 - clz128((ufx_t)W) : 0;
        const int mb = B0 > 0 ? 127 - clz128((ufx_t)B0) : 0;
        // Two doubles hold B0 exactly up to 107 bits, and to 2^-40 W while m >= mb - 66.
        const bool exact = mb > 106 && m < mb - 66;
        const double g = ldexp(1.0, 30 - m);
        const uint32_t margin = m <= 30 ? 0u : 1u;
        const double b_hi = exact ? 0.0 : fx_raw_f64(B0);
        const double b_lo = exact ? 0.0 : fx_raw_f64(B0 - raw_fx(b_hi));
#pragma unroll
        for (int q = 0; q < WSEG / NWAVE; ++q)
        {
            const int s = s0 + q * NWAVE + wid;
            uint32_t key[SCAN_ITEMS] = {PAD, PAD, PAD, PAD};
            if (s < s1)
            {
                const int q0 = s * CDF_SEG + lane * SCAN_ITEMS;
                const int cnt = max(0, min(SCAN_ITEMS, J - q0));
                float f[SCAN_ITEMS] = {0.0f, 0.0f, 0.0f, 0.0f};
                if (cnt > 0)
                    SrcJointPos{nullptr}.load4(d, q0, cnt, f);
                double v[SCAN_ITEMS];
                raw_weights(f, v);
                double sum = v[0];
#pragma unroll
                for (int i = 1; i < SCAN_ITEMS; ++i)
                    sum += v[i];
                const fx_t before = s > s0 ? seg_end(s - 1) - B0 : (fx_t)0;
                double run = wave_inclusive_scan_val(sum) - sum + fx_raw_f64(before);
#pragma unroll
                for (int i = 0; i < SCAN_ITEMS; ++i)
                {
                    run += v[i];
                    if (i < cnt)
                        key[i] = (uint32_t)(run * g) + margin;
                }
            }
            *reinterpret_cast<uint4*>(&s_key[(q * NWAVE + wid) * CDF_SEG + lane * SCAN_ITEMS]) =
                make_uint4(key[0], key[1], key[2], key[3]);
        }
        __syncthreads();
        // Keys below rk - margin (staged: below rk) are below the draw, keys from rk + 2 margin on are not.  The
        // thread's searches go step by step together (four LDS reads in flight).
        uint32_t rk[RS_ITEMS];
        int lo[RS_ITEMS];
#pragma unroll
        for (int i = 0; i < RS_ITEMS; ++i)
        {
            rk[i] = (uint32_t)fmin(fmax(((s_r[threadIdx.x + i * BLOCK] - b_hi) - b_lo) * g, 0.0), 2415919104.0);
            lo[i] = 0;
        }
#pragma unroll
        for (int step = WLEN / 2; step > 0; step >>= 1)
        {
#pragma unroll
            for (int i = 0; i < RS_ITEMS; ++i)
                lo[i] += s_key[lo[i] + step - 1] < rk[i] ? step : 0;
        }
        int left = 0;  // bit i: draw i is to be resolved exactly
#pragma unroll
        for (int i = 0; i < RS_ITEMS; ++i)
        {
            const uint32_t at = s_key[lo[i]];
            if (anc[i] < 0)
            {
                if (exact)
                    left |= 1 << i;
                else if (at >= rk[i] && at < rk[i] + 3u * margin)
                    left |= 1 << i;
                else if (at >= rk[i] && lo[i] < clen)
                    anc[i] = c0 + lo[i];
            }
        }
#pragma unroll
        for (int i = 0; i < RS_ITEMS; ++i)
        {
            uint64_t todo = __ballot((left >> i) & 1);
            while (todo)
            {
                const int l = __builtin_ctzll(todo);
                todo &= todo - 1;
                const int a = wave_exact_ancestor(d, seg_end, J, raw_fx(s_r[wid * WAVE + l + i * BLOCK]));
                if (lane == l)
                    anc[i] = a;
            }
        }
        if (s1 > s_hi)
            break;
        int done = 0;
#pragma unroll
        for (int i = 0; i < RS_ITEMS; ++i)
            done += __popcll(__ballot(anc[i] >= 0 && threadIdx.x + i * BLOCK < cnt_draws));
        if (lane == 0)
            s_done[wid] = done;
        __syncthreads();  // also: every search of this window is done
        done = 0;
#pragma unroll
        for (int w = 0; w < NWAVE; ++w)
            done += s_done[w];
        if (done >= cnt_draws)
            break;
        const fx_t rmin = raw_fx(s_r[done]);
        const int next_last = min(s1 - 1 + WSEG, s_hi);
        if (!(seg_end(next_last) < rmin))
        {
            s0 = s1;
        }
        else
        {
            int c, unused;
            seg_end.find2(rmin, rmin, &c, &unused);
            s0 = max(s1, c);
        }
    }
    merge_write(d, sc, pph, base, n, J, anc);
}

// Float-mode merge (precision study): the envelope is stored, so a window stages
// RS_FLOAT_SLICE_TILES tiles of it; the search and the window walk are those of the exact merge
// at tile granularity.
__global__ __launch_bounds__(BLOCK) __attribute__((amdgpu_waves_per_eu(4)))
void k_rs_merge_float(const VehDesc* __restrict__ descs, const uint32_t* __restrict__ tab, int pph,
                      const fx_t* __restrict__ exp_tile_pre, const void* __restrict__ cdf_incl,
                      const DevScalars* __restrict__ scs)
{
    using Tr = CdfFloatTr;
    constexpr int SLICE = RS_FLOAT_SLICE_TILES * SCAN_TILE;
    __shared__ CdfStage<SLICE> s_cdf;
    __shared__ double s_rb[2];
    __shared__ int s_cnt[1];
    __shared__ int s_kmin;

    const TileRef tr = tile_ref(tab, RS_TILE / UNIT, blockIdx.x);
    const VehDesc& d = descs[tr.v];
    const int n = d.N;
    const int base = tr.base;
    if (base >= n || !Tr::takes(d))
        return;
    const DevScalars* sc = scs + tr.v;
    const int J = n + d.B;
    double r[RS_ITEMS];
    merge_draws(
        d, sc, base, n, exp_tile_pre,
        [sc, &d](fx_t s_k, const Spacing& sp) { return Tr::draw(s_k, sp, sc, d.cdf_mode); }, s_cdf, r, s_rb);
    const int T = (J + SCAN_TILE - 1) / SCAN_TILE;
    const int t0 = d.u0[SP_J] / SCAN_Q;
    const auto tile_end = [cdf_incl, t0](int t) { return Tr::incl(cdf_incl, t0, t); };
    const int t_lo = find_first_not_below<double>(tile_end, T, s_rb[0], s_cnt);
    const int t_hi = find_first_not_below<double>(tile_end, T, s_rb[1], s_cnt);
    int anc[RS_ITEMS];
#pragma unroll
    for (int i = 0; i < RS_ITEMS; ++i)
        anc[i] = -1;
    for (int tc = t_lo; tc <= t_hi;)
    {
        const int tc_end = min(tc + RS_FLOAT_SLICE_TILES, t_hi + 1) - 1;
        const int c0 = tc * SCAN_TILE;
        const int clen = min(J, (tc_end + 1) * SCAN_TILE) - c0;
        __syncthreads();
        for (int i = threadIdx.x; i < clen; i += BLOCK)
            s_cdf.put(i, Tr::value(d, cdf_incl, t0, c0 + i));
        __syncthreads();
        const double cmax = s_cdf.get(clen - 1);
        const int span = clen > 1 ? 1 << (32 - __clz(clen - 1)) : 1;
#pragma unroll
        for (int i = 0; i < RS_ITEMS; ++i)
        {
            if (anc[i] < 0 && base + (int)threadIdx.x + i * BLOCK < n && !(cmax < r[i]))
            {
                int lo = 0;
                for (int step = span >> 1; step > 0; step >>= 1)
                {
                    const int j = lo + step - 1;
                    if (j < clen && s_cdf.less(j, r[i]))
                        lo += step;
                }
                anc[i] = c0 + lo;
            }
        }
        if (tc_end >= t_hi)
            break;
        const int kmin = merge_next_draw<double>(base, n, anc, r, &s_kmin, s_rb);
        if (kmin >= n)
            break;
        const double rmin = s_rb[0];
        const int next_end = min(tc_end + RS_FLOAT_SLICE_TILES, t_hi);
        if (!(tile_end(next_end) < rmin))
            tc = tc_end + 1;
        else
            tc = max(tc_end + 1, find_first_not_below<double>(tile_end, T, rmin, s_cnt));
    }
    merge_write(d, sc, pph, base, n, J, anc);
}

// Writes out a deferred resampled set (see merge_write): particle k of dst copied from its ancestor
// (particle anc[k] of src below n, birth particle anc[k] - n above) with the new weight, which the
// resampling left in dst.weight[0].
__global__ __launch_bounds__(BLOCK) void k_materialize(DevParticles dst, DevParticles src, DevParticles birth,
                                                       const int* __restrict__ anc, int n)
{
    const int k = blockIdx.x * BLOCK + threadIdx.x;
    if (k >= n)
        return;
    const int a = anc[k];
    const bool from_p = a < n;
    const int o = from_p ? a : a - n;
    const DevParticles& s = from_p ? src : birth;
    dst.pos[k] = s.pos[o];
    dst.vel[k] = s.vel[o];
    dst.idx[k] = word_index(s.idx[o]);
    dst.assoc[k] = s.assoc[o];
    if (k > 0)
        dst.weight[k] = dst.weight[0];
}

void run_materialize(Engine* E, const Vehicle* v)
{
    if (v->N <= 0)
        return;
    launch_begin(E, K_MATERIALIZE);
    hipLaunchKernelGGL(k_materialize, dim3(div_up(v->N, BLOCK)), dim3(BLOCK), 0, E->stream, v->part[0], v->part[1],
                       v->birth, v->ancestors, v->N);
    launch_end(E, K_MATERIALIZE);
}

// One workgroup per vehicle: half of its waves scan the joint CDF's tile totals (exact-CDF vehicles; prefixes in
// place), the other half the exponentials' (prefixes into exp_pre), then one thread derives the draws'
// mapping from both totals.  Bound by latency: a few dependent rounds of loads and 128-bit scans on one CU
// per vehicle.  2148 + 1954 tiles (2e6 particles): 20 us with one 256-thread workgroup doing both in turn
// and adding the prefixes into the four segment ends per tile, 8.4 us so.
__global__ __launch_bounds__(TOP_BLOCK) void k_scan_top_resample(const VehDesc* __restrict__ descs,
                                                                 fx_t* __restrict__ cdf_sum,
                                                                 const fx_t* __restrict__ exp_sum,
                                                                 fx_t* __restrict__ exp_pre,
                                                                 DevScalars* __restrict__ scs)
{
    constexpr int HALF = TOP_BLOCK / 2;
    __shared__ fx_t s_wave[2][HALF / WAVE];
    __shared__ fx_t s_total[2];
    __shared__ int s_beyond;
    const VehDesc& d = descs[blockIdx.x];
    if (threadIdx.x == 0)
        s_beyond = scs[blockIdx.x].beyond_tiles;  // beside the loads of the totals, not behind the scan
    const int half = threadIdx.x / HALF, tid = threadIdx.x % HALF;
    const int nj = d.cdf_mode == CDF_EXACT ? d.nu[SP_J] / SCAN_Q : 0;
    const int ne = d.draw_mode == DRAW_MULTINOMIAL ? d.nu[SP_E] / SCAN_Q : 0;
    const int rounds = max(top_rounds(nj, HALF), top_rounds(ne, HALF));
    bool beyond = false;
    const fx_t total = scan_tile_prefixes<HALF>(half ? exp_sum : cdf_sum, half ? exp_pre : cdf_sum,
                                                half ? d.u0[SP_E] / SCAN_Q : d.u0[SP_J] / SCAN_Q, half ? ne : nj, 1, tid,
                                                rounds, s_wave[half],
                                                [&](fx_t prefix) { beyond |= beyond_keys(prefix); });
    if (beyond && half == 0)
        s_beyond = 1;
    if (tid == 0)
        s_total[half] = total;
    __syncthreads();
    if (threadIdx.x == 0)
    {
        DevScalars* sc = scs + blockIdx.x;
        const fx_t cdf_total = s_total[0];
        // Systematic draws do not use the exponentials: S_N = N * 2^32 (dogm_numerics.h).
        sc->spacing = spacing_setup(ne ? s_total[1] : systematic_s(d.N, 0u), cdf_total);
        sc->cdf_total = cdf_total;
        sc->beyond_keys = s_beyond;
        sc->beyond_tiles = 0;
        if (nj)
        {
            const float jm = fx_to_f32(cdf_total);
            sc->new_weight = jm / (float)d.N;
        }
    }
}

void run_resampling(Engine* E, int pph, int modes, bool exp_done)
{
    const bool exact = modes & (1 << CDF_EXACT);
    const int jtiles = E->tiles(SP_J, SCAN_Q);
    const int etiles = exp_done ? 0 : E->tiles(SP_E, SCAN_Q);
    // Tile totals of the joint CDF (exact-CDF vehicles, with the tile-local segment ends of the coarse
    // index; the merge recomputes entries) and of the exponentials (multinomial draws) in one launch,
    // then both top-level scans in one launch.
    launch_begin(E, K_SCAN_TILES);
    hipLaunchKernelGGL(k_scan_tiles_exp<SrcJointPos>, dim3(jtiles + etiles), dim3(BLOCK), 0, E->stream,
                       SrcJointPos{E->scalars}, E->tab(SP_J), jtiles, E->scan_tile_sum, E->cdf_tile_incl, E->tab(SP_E),
                       E->exp_tile_sum, E->d_desc);
    launch_end(E, K_SCAN_TILES);
    launch_begin(E, K_SCAN_TOP);
    hipLaunchKernelGGL(k_scan_top_resample, dim3(E->m), dim3(TOP_BLOCK), 0, E->stream, E->d_desc, E->scan_tile_sum,
                       E->exp_tile_sum, E->scan_tile_pre, E->scalars);
    launch_end(E, K_SCAN_TOP);
    // Float modes: tile totals as doubles in scan_tile_sum (each in its tile's own entry), prefixes in the consumed
    // exponential totals (the exponentials' prefixes stay in scan_tile_pre for the merge).
    double* tsum = reinterpret_cast<double*>(E->scan_tile_sum);
    double* tpre = reinterpret_cast<double*>(E->exp_tile_sum);
    double* env = reinterpret_cast<double*>(E->cdf_tile_incl);
    auto float_mode = [&](auto tag) {
        using T = decltype(tag);
        launch_begin(E, K_CDF_WRITE);
        hipLaunchKernelGGL(k_cdff_tiles<T>, dim3(jtiles), dim3(BLOCK), 0, E->stream, E->d_desc, E->tab(SP_J), tsum);
        hipLaunchKernelGGL(k_cdff_top<T>, dim3(E->m), dim3(BLOCK), 0, E->stream, E->d_desc, tsum, tpre);
        hipLaunchKernelGGL(k_cdff_apply<T>, dim3(jtiles), dim3(BLOCK), 0, E->stream, E->d_desc, E->tab(SP_J), tpre,
                           env);
        launch_end(E, K_CDF_WRITE);
    };
    if (modes & (1 << CDF_FP64))
        float_mode(0.0);
    if (modes & (1 << CDF_FP32))
        float_mode(0.0f);
    if (modes & (1 << CDF_FP32C))
        float_mode(f32c(0));
    if (modes & ~(1 << CDF_EXACT))
        hipLaunchKernelGGL(k_cdff_env, dim3(E->m), dim3(ENV_BLOCK), 0, E->stream, E->d_desc, env, E->scalars);

    const int mt = E->tiles(SP_P, RS_TILE / UNIT);
    const bool wide = E->tune.merge_slice != 1;
    // Windows of merge_beyond_keys: 8 segments for launches of up to 4096 workgroups, 4 for larger ones.
    const int beyond_segs = (E->tune.merge_slice == 0 ? mt <= 4096 : wide) ? RS_WINDOW_WIDE : RS_WINDOW_NARROW;
    launch_begin(E, K_RS_MERGE);
    if (exact)
    {
        if (wide)
            hipLaunchKernelGGL(k_rs_merge_exact<RS_WINDOW_WIDE>, dim3(mt), dim3(BLOCK), 0, E->stream, E->d_desc,
                               E->tab(SP_P), pph, E->scan_tile_pre, E->cdf_tile_incl, E->scan_tile_sum, E->scalars,
                               beyond_segs);
        else
            hipLaunchKernelGGL(k_rs_merge_exact<RS_WINDOW_NARROW>, dim3(mt), dim3(BLOCK), 0, E->stream, E->d_desc,
                               E->tab(SP_P), pph, E->scan_tile_pre, E->cdf_tile_incl, E->scan_tile_sum, E->scalars,
                               beyond_segs);
    }
    if (modes & ~(1 << CDF_EXACT))
        hipLaunchKernelGGL(k_rs_merge_float, dim3(mt), dim3(BLOCK), 0, E->stream, E->d_desc, E->tab(SP_P), pph,
                           E->scan_tile_pre, (const void*)E->cdf_tile_incl, E->scalars);
    launch_end(E, K_RS_MERGE);
}

}  // namespace dogm_hip
