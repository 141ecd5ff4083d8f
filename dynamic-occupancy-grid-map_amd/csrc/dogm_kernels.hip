// Stage kernels of the DOGM particle-filter update on gfx950.
//
// Layout in HBM, per vehicle: particles structure-of-arrays (position, velocity, int cell index, float
// weight, uint8 association), grid cells structure-of-arrays (one array per field), measurement
// cells as given by the caller (16-byte AoS).  Every per-cell sum is an exact 128-bit fixed-point
// segmented reduction over the cell-sorted particles (dogm_device.h).  Step kernels find their
// vehicle and local tile through the step's work tables (dogm_internal.h).
#include "dogm_device.h"

namespace dogm_hip
{

// ---------------------------------------------------------------------------------------------
// Utility kernels
// ---------------------------------------------------------------------------------------------
__global__ __launch_bounds__(BLOCK) void k_fill_u32(unsigned* __restrict__ p, unsigned v, long long n)
{
    const long long i = (long long)blockIdx.x * BLOCK + threadIdx.x;
    if (i < n)
        p[i] = v;
}

void run_fill_u32(Engine* E, unsigned* p, unsigned v, long long n)
{
    if (n <= 0)
        return;
    launch_begin(E, K_FILL);
    hipLaunchKernelGGL(k_fill_u32, dim3(div_up(n, BLOCK)), dim3(BLOCK), 0, E->stream, p, v, n);
    launch_end(E, K_FILL);
}

struct TabArgs
{
    long long units[SP_COUNT];
};

// Expands the per-space unit prefixes of the step's vehicles (upre[s * (m + 1) + v]) into the
// work tables: entry i of space s = vehicle << 20 | local unit.
__global__ __launch_bounds__(BLOCK) void k_build_tables(const int* __restrict__ upre, int m, TabArgs a,
                                                        uint32_t* __restrict__ tab, long long total)
{
    const long long i = (long long)blockIdx.x * BLOCK + threadIdx.x;
    if (i >= total)
        return;
    int s = 0;
    long long u = i;
    while (s < SP_COUNT - 1 && u >= a.units[s])
    {
        u -= a.units[s];
        ++s;
    }
    const int* pre = upre + s * (m + 1);
    // last v in [0, m) with pre[v] <= u
    int lo = 0, count = m;
    while (count > 0)
    {
        const int step = count / 2;
        if (pre[lo + step + 1] <= u)
        {
            lo += step + 1;
            count -= step + 1;
        }
        else
        {
            count = step;
        }
    }
    tab[i] = ((uint32_t)lo << TAB_VEH_SHIFT) | (uint32_t)(u - pre[lo]);
}

void run_build_tables(Engine* E)
{
    TabArgs a{};
    long long total = 0;
    for (int s = 0; s < SP_COUNT; ++s)
    {
        a.units[s] = E->units[s];
        total += E->units[s];
    }
    if (total <= 0)
        return;
    launch_begin(E, K_BUILD_TABLES);
    hipLaunchKernelGGL(k_build_tables, dim3(div_up(total, BLOCK)), dim3(BLOCK), 0, E->stream, E->d_upre, E->m, a,
                       E->d_tab, total);
    launch_end(E, K_BUILD_TABLES);
}

// ---------------------------------------------------------------------------------------------
// Ego-motion compensation (dogm/src/kernel/ego_motion_compensation.cu:16-43), eager form for the
// single-vehicle pose update.  Inside an update step the shift is fused into predict and the
// occupancy update.
// ---------------------------------------------------------------------------------------------
__global__ __launch_bounds__(BLOCK) void k_move_particles(DevParticles P, int n, float mx, float my)
{
    const int i = blockIdx.x * BLOCK + threadIdx.x;
    if (i >= n)
        return;
    float2 s = P.pos[i];
    s.x = s.x - mx;
    s.y = s.y - my;
    P.pos[i] = s;
}

void run_move_particles(Engine* E, const Vehicle* v, float mx, float my)
{
    launch_begin(E, K_MOVE_PARTICLES);
    hipLaunchKernelGGL(k_move_particles, dim3(div_up(v->N, BLOCK)), dim3(BLOCK), 0, E->stream, v->part[0], v->N, mx,
                       my);
    launch_end(E, K_MOVE_PARTICLES);
}

// Metric ego compensation of one particle: position rotated by -dpsi about the grid centre and
// translated by whole cells, velocity rotated (a pure translation keeps positions exact).
__device__ __forceinline__ float4 ego_particle(float4 s, const EgoXform& t)
{
    if (t.sn == 0.0f && t.cs == 1.0f)
        return make_float4(s.x + t.tx, s.y + t.ty, s.z, s.w);
    const float dx = s.x - t.c, dy = s.y - t.c;
    const float rx = t.cs * dx + t.sn * dy;
    const float ry = t.cs * dy - t.sn * dx;
    const float vx = t.cs * s.z + t.sn * s.w;
    const float vy = t.cs * s.w - t.sn * s.z;
    return make_float4((t.c + rx) + t.tx, (t.c + ry) + t.ty, vx, vy);
}

// Source cell of destination cell c under the transform, by nearest cell: the cell containing
// c + R(dpsi) ((x + 0.5, y + 0.5) - c - t); -1 outside the grid.
__device__ __forceinline__ int ego_source_cell(int c, int gs, const EgoXform& t)
{
    const float qx = ((float)(c % gs) + 0.5f - t.c) - t.tx;
    const float qy = ((float)(c / gs) + 0.5f - t.c) - t.ty;
    const float sx = floorf(t.c + (t.cs * qx - t.sn * qy));
    const float sy = floorf(t.c + (t.sn * qx + t.cs * qy));
    const bool in = sx >= 0.0f && sx < (float)gs && sy >= 0.0f && sy < (float)gs;
    return in ? (int)sx + gs * (int)sy : -1;
}

__global__ __launch_bounds__(BLOCK) void k_ego_particles(DevParticles P, int n, EgoXform t)
{
    const int i = blockIdx.x * BLOCK + threadIdx.x;
    if (i >= n)
        return;
    const float2 p = P.pos[i], v = P.vel[i];
    const float4 s = ego_particle(make_float4(p.x, p.y, v.x, v.y), t);
    P.pos[i] = make_float2(s.x, s.y);
    P.vel[i] = make_float2(s.z, s.w);
}

void run_ego_particles(Engine* E, const Vehicle* v, const EgoXform& t)
{
    if (v->N <= 0)
        return;
    launch_begin(E, K_EGO_PARTICLES);
    hipLaunchKernelGGL(k_ego_particles, dim3(div_up(v->N, BLOCK)), dim3(BLOCK), 0, E->stream, v->part[0], v->N, t);
    launch_end(E, K_EGO_PARTICLES);
}

// The same transform on a grid field (nearest source cell; sources outside the grid give 0).
__global__ __launch_bounds__(BLOCK) void k_ego_field(const uint32_t* __restrict__ src, uint32_t* __restrict__ dst,
                                                     int gs, EgoXform t)
{
    const int c = blockIdx.x * BLOCK + threadIdx.x;
    if (c >= gs * gs)
        return;
    const int s = ego_source_cell(c, gs, t);
    dst[c] = s >= 0 ? src[s] : 0u;
}

void run_ego_field(Engine* E, const Vehicle* v, const void* src, void* dst, const EgoXform& t)
{
    launch_begin(E, K_EGO_FIELD);
    hipLaunchKernelGGL(k_ego_field, dim3(div_up(v->C, BLOCK)), dim3(BLOCK), 0, E->stream,
                       static_cast<const uint32_t*>(src), static_cast<uint32_t*>(dst), v->gs, t);
    launch_end(E, K_EGO_FIELD);
}

// new[x, y] = old[x + ix, y + iy] when 0 < x + ix < gs and 0 < y + iy < gs (strict lower bound,
// ego_motion_compensation.cu:38), else 0 (the reference memsets the grid first, dogm.cu:185).
__global__ __launch_bounds__(BLOCK) void k_shift_field(const uint32_t* __restrict__ src, uint32_t* __restrict__ dst,
                                                       int gs, int ix, int iy)
{
    const int c = blockIdx.x * BLOCK + threadIdx.x;
    if (c >= gs * gs)
        return;
    const int x = c % gs, y = c / gs;
    const int sx = x + ix, sy = y + iy;
    const bool in = sx > 0 && sx < gs && sy > 0 && sy < gs;
    dst[c] = in ? src[sx + gs * sy] : 0u;
}

void run_shift_field(Engine* E, const Vehicle* v, const void* src, void* dst, int ix, int iy)
{
    launch_begin(E, K_SHIFT_FIELD);
    hipLaunchKernelGGL(k_shift_field, dim3(div_up(v->C, BLOCK)), dim3(BLOCK), 0, E->stream,
                       static_cast<const uint32_t*>(src), static_cast<uint32_t*>(dst), v->gs, ix, iy);
    launch_end(E, K_SHIFT_FIELD);
}

// ---------------------------------------------------------------------------------------------
// Prediction (dogm/src/kernel/predict.cu:16-52), with the pending ego shift of the step fused in
// (moveParticlesKernel runs right before it in the reference).
// ---------------------------------------------------------------------------------------------
__device__ __forceinline__ int clamp_cell(float x, int gs)
{
    return (int)fminf(fmaxf(x, 0.0f), (float)(gs - 1));  // NaN gives cell 0
}

// Border cells: the cells whose coordinate predict clamps to, so the only ones that can hold out-of-grid
// particles (weight 0) beside in-grid ones.  For vehicles with per-cell weights their out-of-grid particles
// are counted in the born masses (as ints), which the occupancy update rewrites cell by cell after it has read
// the cell's count: zeroed beside predict, counted by k_cell_bounds.
__device__ __forceinline__ bool border_cell(int c, int gs)
{
    const int y = c / gs, x = c - y * gs;
    return x == 0 || y == 0 || x == gs - 1 || y == gs - 1;
}
__device__ __forceinline__ int* border_out(const VehDesc& d)
{
    return reinterpret_cast<int*>(d.born.get());
}

// start = end = -1 for the cells of work-table group `group` (THREADS x 4 cells), four cells per
// thread with 16-byte stores.  With valid occupancy bits only groups of four containing a cell that
// had particles are written (the others still hold -1, and rewriting -1 is harmless).
template <int THREADS>
__device__ __forceinline__ void reset_bounds_cells(const VehDesc* __restrict__ descs, const uint32_t* __restrict__ tab,
                                                   int group)
{
    const TileRef tr = tile_ref(tab, THREADS * 4 / UNIT, group);
    const VehDesc& d = descs[tr.v];
    const int c = tr.base + 4 * threadIdx.x;
    if (c >= d.C)
        return;
    if (d.wcell)
    {
        const int last = min(c + 3, d.C - 1);
        const int y = c / d.gs, x = c - y * d.gs;
        // a border cell among the four (a group that wraps into the next row holds one)
        if (y == 0 || x == 0 || x + 3 >= d.gs - 1 || last >= d.C - d.gs)
            for (int k = c; k <= last; ++k)
                border_out(d)[k] = 0;
    }
    if (d.nz_valid && ((d.nz[c >> 6] >> (c & 63)) & 0xfull) == 0)
        return;
    if (c + 4 <= d.C)
    {
        const int4 m1 = make_int4(-1, -1, -1, -1);
        *reinterpret_cast<int4*>(d.start + c) = m1;
        *reinterpret_cast<int4*>(d.end + c) = m1;
    }
    else
    {
        for (int k = c; k < d.C; ++k)
        {
            d.start[k] = -1;
            d.end[k] = -1;
        }
    }
}

// A workgroup covers one sort tile: PB threads of SORT_TILE / PB particles each (strided by PB).
// 512 x 4 (the built-in choice) gives a single 2e6-particle grid about 8 waves per SIMD to hide the
// Philox / Box-Muller latency; 256 x 8 is the other choice of the tuning.  Bound by memory where many vehicles
// share a launch (41 bytes a particle; 16 x 2e6: 329 us) and by latency below: with the item loop loading ahead,
// without its digit counts' global atomics and with the shorter quotient and root, 2e6 particles went from 35.5 to
// 23.8 us and 3e5 from 13.6 to 9.6; the item loop stays rolled (unrolled: 23.5 and 11.0).
//
// With passes > 0 the workgroup also counts the radix digits of the new cell indices (of every sort pass for the
// onesweep form, of the first for reduce-then-scan: `passes`).  Without thist the counts go to
// ghist[(vehicle * 4 + pass) * 256 + digit] (onesweep's one-time histogram; the sort passes' tile tickets are
// cleared too); with
// thist set (reduce-then-scan sort) it stores the first pass's digit counts of its tile as
// thist[digit * tiles + tile]: a workgroup covers exactly one sort tile, so the sort skips that
// upsweep.  With aos (the sort's gathering pass follows in the same step) the new state goes to the
// vehicle's CDF buffer, free until the resampling, as 16-byte (x, y, vx, vy) records, so that the
// gather reads one 16-byte record per particle at random instead of two 8-byte ones from two arrays;
// nothing else reads the positions or velocities in between.  The cell indices then carry the particles'
// flags (WORD_FLAGS), so the sort's first pass reads one word per particle and no association byte.
template <int PRED_BLOCK>
__global__ __launch_bounds__(PRED_BLOCK) void k_predict(const VehDesc* __restrict__ descs, const uint32_t* __restrict__ tab,
                                                   int pph, int passes, unsigned* __restrict__ ghist,
                                                   unsigned* __restrict__ tickets, unsigned* __restrict__ thist,
                                                   int tiles, int aos, const uint32_t* __restrict__ tab_c,
                                                   DevScalars* __restrict__ scs)
{
    constexpr int PRED_ITEMS = SORT_TILE / PRED_BLOCK;
    static_assert(PRED_ITEMS * PRED_BLOCK == SORT_TILE, "predict workgroups are the sort's tiles");
    if ((int)blockIdx.x >= tiles)
    {
        // The assignment's bounds reset, in workgroups after the particle tiles (memory work beside
        // the ALU-bound prediction).
        reset_bounds_cells<PRED_BLOCK>(descs, tab_c, (int)blockIdx.x - tiles);
        return;
    }
    __shared__ unsigned s_h[4][RADIX];
    if (passes > 0 && blockIdx.x == 0 && threadIdx.x < 4)
        tickets[threadIdx.x] = 0u;
    const TileRef tr = tile_ref(tab, SORT_Q, blockIdx.x);
    const VehDesc& d = descs[tr.v];
    const int n = d.N;
    if (tr.base == 0 && threadIdx.x == 0)
        scs[tr.v].born_odd = 0;  // until the occupancy update finds one
    if (tr.base >= n)
    {
        if (passes > 0 && thist)
            for (int i = threadIdx.x; i < RADIX; i += PRED_BLOCK)
                thist[(size_t)i * tiles + blockIdx.x] = 0u;
        return;
    }
    if (passes > 0)
    {
        for (int i = threadIdx.x; i < 4 * RADIX; i += PRED_BLOCK)
            (&s_h[0][0])[i] = 0u;
        __syncthreads();
    }
    const DescParticles P = d.part[pph];
    const DescParticles Q = d.part[pph ^ 1];  // sources of a deferred resampled set
    const DescParticles Bq = d.birth;
    const int gs = d.gs;
    const float dt = d.dt;
    const float zero = 0.0f, one = 1.0f;
    // The gathering pass forms the weight (always so for a deferred set: the host reads one
    // through its ancestors only in full steps, whose weights are uniform).
    const bool keep_w = aos && d.wuni;
    // Inputs of the thread's item `it` (past n: the last particle again, masked below).  A deferred resampled set
    // (see merge_write) is read through its ancestors, the state and association of part[pph ^ 1] below N and of the
    // birth set above.  Two items ahead of the arithmetic the ancestor is loaded, one ahead the state, so
    // neither is waited for.
    const bool gathered = d.rs_gather;
    const int* __restrict__ ancestors = d.ancestors;
    const float2 *lo_pos = (gathered ? Q : P).pos, *hi_pos = Bq.pos;
    const float2 *lo_vel = (gathered ? Q : P).vel, *hi_vel = Bq.vel;
    const uint8_t *lo_as = (gathered ? Q : P).assoc, *hi_as = Bq.assoc;
    const auto load_ancestor = [=](int it) {
        const int i = min(tr.base + it * PRED_BLOCK + (int)threadIdx.x, n - 1);
        return gathered ? ancestors[i] : i;
    };
    const auto load_state = [=](int a, float4& st, uint8_t& as) {
        const bool lo = a < n;
        const int o = lo ? a : a - n;
        const float2 p = (lo ? lo_pos : hi_pos)[o];
        const float2 v = (lo ? lo_vel : hi_vel)[o];
        as = aos ? (lo ? lo_as : hi_as)[o] : 0;
        st = make_float4(p.x, p.y, v.x, v.y);
    };
    float4 next;
    uint8_t next_assoc;
    load_state(load_ancestor(0), next, next_assoc);
    int a_next = load_ancestor(1);
#pragma unroll 1
    for (int it = 0; it < PRED_ITEMS; ++it)
    {
        const int i = tr.base + it * PRED_BLOCK + threadIdx.x;
        const bool valid = i < n;
        float4 s = next;
        const uint8_t assoc = next_assoc;
        load_state(a_next, next, next_assoc);  // the last round's repeats a valid particle
        a_next = load_ancestor(it + 2);
        if (d.move)
        {
            s.x = s.x - d.mx;
            s.y = s.y - d.my;
        }
        else if (d.xform_p)
        {
            s = ego_particle(s, d.xt);
        }
        const u32x4 r = draw(d.seed, d.inst, TAG_PREDICT, d.ep_pred, (uint32_t)i);
        float n0, n1, n2, n3;
        box_muller(r.x, r.y, &n0, &n1);
        box_muller(r.z, r.w, &n2, &n3);
        const float npx = normal_scale(n0, zero, d.sp), npy = normal_scale(n1, zero, d.sp);
        const float nvx = normal_scale(n2, zero, d.sv), nvy = normal_scale(n3, zero, d.sv);
        // glm mat4 * vec4 association ((c0 x + c1 y) + (c2 vx + c3 vy)) of the transposed constant velocity matrix
        // (dogm.cu:246-253).  In finite states the products with 0 add only zeros: they can change nothing
        // but the sign of a zero, and adding the noise (n * sd + 0, never -0) gives +0 for either.
        float4 o;
        const bool finite = fmaf(zero, s.x, fmaf(zero, s.y, fmaf(zero, s.z, zero * s.w))) == zero;
        if (__ballot(!finite) == 0)
        {
            o.x = (s.x + dt * s.z) + npx;
            o.y = (s.y + dt * s.w) + npy;
            o.z = s.z + nvx;
            o.w = s.w + nvy;
        }
        else
        {
            const float sx = (one * s.x + zero * s.y) + (dt * s.z + zero * s.w);
            const float sy = (zero * s.x + one * s.y) + (zero * s.z + dt * s.w);
            const float svx = (zero * s.x + zero * s.y) + (one * s.z + zero * s.w);
            const float svy = (zero * s.x + zero * s.y) + (zero * s.z + one * s.w);
            o.x = sx + npx;
            o.y = sy + npy;
            o.z = svx + nvx;
            o.w = svy + nvy;
        }
        const int cell = clamp_cell(o.x, gs) + gs * clamp_cell(o.y, gs);
        if (valid)
        {
            int word = cell;
            if (aos)
            {
                stream_store(reinterpret_cast<float4*>(d.cdf.get()) + i, o);
                word = (int)((unsigned)cell | (assoc ? WORD_ASSOC : 0u) |
                             (d.wcell && outside_grid(d, o) ? WORD_OUT : 0u));
            }
            else
            {
                P.pos[i] = make_float2(o.x, o.y);
                P.vel[i] = make_float2(o.z, o.w);
            }
            if (!keep_w)
                P.weight[i] = predicted_weight(d, P.weight[i], o);
            stream_store(&P.idx[i], word);
        }
        for (int ps = 0; ps < passes; ++ps)
            wave_count(s_h[ps], ((unsigned)cell >> (ps * RADIX_BITS)) & (RADIX - 1), valid);
    }
    if (passes > 0)
    {
        __syncthreads();
        if (thist)
        {
            for (int i = threadIdx.x; i < RADIX; i += PRED_BLOCK)
                thist[(size_t)i * tiles + blockIdx.x] = s_h[0][i];
            return;
        }
        unsigned* gh = ghist + (size_t)tr.v * 4 * RADIX;
        for (int i = threadIdx.x; i < passes * RADIX; i += PRED_BLOCK)
        {
            const unsigned v = (&s_h[0][0])[i];
            if (v)
                atomicAdd(&gh[i], v);
        }
    }
}

void run_predict(Engine* E, int pph, bool hist, bool aos)
{
    const int blocks = E->tiles(SP_P, SORT_Q);
    if (blocks <= 0)
        return;
    const bool onesweep = E->tune.sort == SORT_ONESWEEP;
    if (hist && onesweep)
    {
        if (!E->ghist_clean)
            run_fill_u32(E, E->sort_ghist, 0u, (long long)E->m * 4 * RADIX);
        E->ghist_clean = false;  // until the sort of this step has cleared them again
    }
    unsigned* thist = onesweep ? nullptr : E->sort_status;
    const int passes = hist ? (onesweep ? E->passes : 1) : 0;
    // With the assignment in the same step (hist), its bounds reset runs in extra workgroups.
    const int pb = E->tune.pred_block == 256 ? 256 : 512;
    const int resets = hist ? E->tiles(SP_C, pb * 4 / UNIT) : 0;
    launch_begin(E, K_PREDICT);
    if (pb == 256)
        hipLaunchKernelGGL(k_predict<256>, dim3(blocks + resets), dim3(256), 0, E->stream, E->d_desc, E->tab(SP_P),
                           pph, passes, E->sort_ghist, E->sort_tickets, thist, blocks, aos ? 1 : 0, E->tab(SP_C), E->scalars);
    else
        hipLaunchKernelGGL(k_predict<512>, dim3(blocks + resets), dim3(512), 0, E->stream, E->d_desc, E->tab(SP_P),
                           pph, passes, E->sort_ghist, E->sort_tickets, thist, blocks, aos ? 1 : 0, E->tab(SP_C), E->scalars);
    launch_end(E, K_PREDICT);
}

// ---------------------------------------------------------------------------------------------
// Assignment (dogm/src/dogm.cu:262-281, init.cu:86-93, particle_to_grid.cu:16-44)
// ---------------------------------------------------------------------------------------------
__global__ __launch_bounds__(BLOCK) void k_reset_bounds(const VehDesc* __restrict__ descs,
                                                        const uint32_t* __restrict__ tab)
{
    reset_bounds_cells<BLOCK>(descs, tab, blockIdx.x);
}

// Gathers the payload into sorted order and records first/last occurrence of every cell.
__global__ __launch_bounds__(BLOCK) void k_sort_gather(const VehDesc* __restrict__ descs,
                                                       const uint32_t* __restrict__ tab, int pph, int fin)
{
    const TileRef tr = tile_ref(tab, 1, blockIdx.x);
    const VehDesc& d = descs[tr.v];
    const int k = tr.base + threadIdx.x;
    const int n = d.N;
    if (k >= n)
        return;
    const DescParticles src = d.part[pph];
    const DescParticles dst = d.part[pph ^ 1];
    const int* skeys = d.sort_keys[fin];
    const int sv = d.sort_vals[fin][k];
    const int o = word_index(sv);
    const int key = skeys[k];
    const float w = src.weight[o];
    dst.pos[k] = src.pos[o];
    dst.vel[k] = src.vel[o];
    dst.weight[k] = w;
    dst.assoc[k] = word_assoc(sv);
    dst.idx[k] = key;
    d.weight_array[k] = w;
    if (k == 0 || skeys[k - 1] != key)
        d.start[key] = k;
    if (k == n - 1 || skeys[k + 1] != key)
        d.end[key] = k;
}

void run_assignment(Engine* E, int pph, bool hist_done, bool defer_bounds, bool write_wa)
{
    if (!hist_done)  // else predict's launch reset the bounds
    {
        launch_begin(E, K_RESET_BOUNDS);
        hipLaunchKernelGGL(k_reset_bounds, dim3(E->tiles(SP_C, 4)), dim3(BLOCK), 0, E->stream, E->d_desc,
                           E->tab(SP_C));
        launch_end(E, K_RESET_BOUNDS);
    }
    run_sort(E, pph, hist_done, defer_bounds, write_wa || !defer_bounds);
    if (defer_bounds)
        return;  // the last sort pass wrote the particles; the occupancy reduction records the bounds
    launch_begin(E, K_SORT_GATHER);
    hipLaunchKernelGGL(k_sort_gather, dim3(E->tiles(SP_P, 1)), dim3(BLOCK), 0, E->stream, E->d_desc, E->tab(SP_P),
                       pph, (E->passes - 1) & 1);
    launch_end(E, K_SORT_GATHER);
}

// ---------------------------------------------------------------------------------------------
// Occupancy / mass update (dogm/src/dogm.cu:283-298, mass_update.cu:16-93)
// ---------------------------------------------------------------------------------------------
// IT particles per thread (the tuning's seg_items); register budgets of six waves per SIMD for 8
// (no spills) and eight for 4.
template <int IT>
struct OccOp
{
    static constexpr int NCH = 1;
    static constexpr int ITEMS = IT;
    static constexpr int WAVES = IT == 8 ? 6 : 8;
    int pph;
    int bounds;  // record start_idx / end_idx (dogm.cu:262-281) when the assignment deferred them
    __device__ const int* keys(const VehDesc& d) const { return d.part[pph].idx; }
    __device__ void head(const VehDesc& d, int key, int p) const
    {
        if (bounds)
            d.start[key] = p;
    }
    __device__ void end(const VehDesc& d, int key, int p) const
    {
        if (bounds)
            d.end[key] = p;
    }
    __device__ void load(const VehDesc& d, int p0, int cnt, const int (&)[ITEMS], float (&v)[ITEMS][NCH]) const
    {
        // After the gathering sort pass of the same step the particles' weights equal weight_array
        // (which that pass may leave unwritten); otherwise weight_array is what the step starts from.
        float w[ITEMS];
        load_run<ITEMS>(bounds ? d.part[pph].weight : d.weight_array, p0, cnt, w);
#pragma unroll
        for (int i = 0; i < ITEMS; ++i)
            v[i][0] = w[i];
    }
    __device__ void finalize(const VehDesc& d, int key, const fx_t (&s)[1]) const { d.m_raw[key] = fx_to_f32(s[0]); }
    // A cell crossing tiles is marked with NaN (an exact sum is never NaN); the occupancy update
    // sums its tile partials.
    __device__ void cont(const VehDesc& d, int key) const { d.m_raw[key] = __builtin_nanf(""); }
};

// zero_empty: bit 0 writes mu_A = mu_UA = 0, bit 1 the five velocity moments = 0 for cells without
// particles (what the persistent-update and moments stages write there), when those stages run
// in the same step.  With both (a full update) the kernel also writes the occupancy bits, and with
// valid bits from the previous full update it skips the zeros of cells that were empty then (their
// fields are still zero in memory).
// Cells whose particles cross reduction tiles get their weight sum here from the reduction's tile
// partials (the first tile's tail, whole middle tiles, the last tile's head), as the fix-up pass
// would, and m_raw is written for them.
//
// Vehicles with per-cell weights (VehDesc::wcell): every in-grid particle of a cell has the weight
// w = persistence * prior and the out-of-grid ones (border cells only) weight 0, so the exact sums over a
// cell's particles are its counts times one fixed-point value (integer products: the same 128-bit sums, wrap
// included, as adding the particles one by one), and what the persistent update derives from them is
// formed here, one thread per cell.  cellrec then holds the two posterior weights of the cell's particles
// (in-grid, out-of-grid) and rho_p for the moments.  No per-particle reduction is left: the two segmented
// reductions and their fix-up took 39 us per frame at 1200 x 1200 cells and 2e6 particles (18 us per vehicle in
// a batch of 32); the cell bounds pass takes 5.6 (2.3) and this kernel 1 us more.
// One cell; returns its born mass rho_b.
__device__ __forceinline__ float mass_update_cell(const VehDesc& d, int c, int zero_empty, const SegCarry& carry,
                                                  int occ_tile, int pph)
{
    const int gs = d.gs;
    const float* free_src = d.free[0];
    const float one = 1.0f;
    float m_occ_pred = 0.0f;
    // Everything a cell reads is loaded before the first branch on it or store (75% of the wave cycles were
    // waits, for one load after the other).
    const int start = d.start[c], end = d.end[c];
    const unsigned long long was = zero_empty == 3 && d.nz_valid ? d.nz[c >> 6] : ~0ull;
    const float prior = d.wcell ? d.part[pph ^ 1].weight[0] : 0.0f;
    const dogm_measurement_cell mc = d.meas_in ? d.meas_in[c] : d.meas[c];
    float fprev;
    if (d.shifted)
    {
        const int x = c % gs, y = c / gs;
        const int sx = x + d.gx, sy = y + d.gy;
        fprev = (sx > 0 && sx < gs && sy > 0 && sy < gs) ? free_src[sx + gs * sy] : 0.0f;
    }
    else if (d.xform_g)
    {
        const int sc = ego_source_cell(c, gs, d.xt);
        fprev = sc >= 0 ? free_src[sc] : 0.0f;
    }
    else
    {
        fprev = free_src[c];
    }
    const bool occupied = start != -1;
    bool zero_fields = !occupied && zero_empty;
    if (zero_empty == 3)
    {
        // Work-table units are 256 cells, so each wave covers one aligned 64-cell word.
        zero_fields = zero_fields && ((was >> (c & 63)) & 1ull);
        const unsigned long long now = __ballot(occupied);
        if ((c & 63) == 0)
            d.nz[c >> 6] = now;
    }
    float w_in = 0.0f;  // per-cell weights: the in-grid particles' predicted weight, and the counts
    int n_in = 0, n_out = 0;
    if (occupied && d.wcell)
    {
        w_in = d.ps * prior;
        n_out = border_cell(c, gs) ? border_out(d)[c] : 0;
        n_in = end - start + 1 - n_out;
        m_occ_pred = fx_to_f32(fx_from_f32(w_in) * n_in);
    }
    else if (occupied)
    {
        const int OT = occ_tile;  // particles per reduction tile
        m_occ_pred = d.m_raw[c];
        if (m_occ_pred != m_occ_pred)  // marked: the cell crosses reduction tiles
        {
            const int ts = start / OT, te = end / OT;
            const int t0 = d.u0[SP_P] / (OT / UNIT);
            fx_t sum = carry.tail_partial[t0 + ts];
            for (int t = ts + 1; t < te; ++t)
                sum += carry.tail_partial[t0 + t];
            sum += carry.head_partial[t0 + te];
            m_occ_pred = fx_to_f32(sum);
            d.m_raw[c] = m_occ_pred;
        }
    }
    else if (zero_fields)
    {
        if (zero_empty & 1)
        {
            d.f[GF_MU_A][c] = 0.0f;
            d.f[GF_MU_UA][c] = 0.0f;
        }
        if (zero_empty & 2)
            for (int f = GF_MEAN_X; f <= GF_COVAR; ++f)
                d.f[f][c] = 0.0f;
    }
    const float m_raw_c = m_occ_pred;  // Σw of the cell before the clamp
    if (m_occ_pred > one)
        m_occ_pred = one;
    // The step's measurement grid, copied into the vehicle's buffer on the way when it comes from
    // the caller's device buffer (dogm.cu:205-215).
    if (d.meas_in)
        stream_store(&d.meas[c], mc);
    if ((zero_empty & 1) && occupied && !d.wcell)
        stream_store(&d.cellin[c], make_float2(mc.likelihood, m_raw_c));
    const float pB = d.pB;
    const float m_free_pred = fminf(d.alpha * fprev, one - m_occ_pred);
    const float unknown_pred = one - m_occ_pred - m_free_pred;
    const float meas_unknown = one - mc.free_mass - mc.occ_mass;
    const float K = m_free_pred * mc.occ_mass + m_occ_pred * mc.free_mass;
    const float occ_up =
        (m_occ_pred * meas_unknown + unknown_pred * mc.occ_mass + m_occ_pred * mc.occ_mass) / (one - K);
    const float free_up =
        (m_free_pred * meas_unknown + unknown_pred * mc.free_mass + m_free_pred * mc.free_mass) / (one - K);
    const float rho_b = (occ_up * pB * (one - m_occ_pred)) / (m_occ_pred + pB * (one - m_occ_pred));
    const float rho_p = occ_up - rho_b;
    if (occupied && d.wcell)
    {
        // mass_update.cu:51-59 (weights of overfull cells), update_persistent_particles.cu:16-87.
        const bool over = m_raw_c > one;
        const float wi = over ? w_in / m_raw_c : w_in;
        const float wo = over ? 0.0f / m_raw_c : 0.0f;
        const float lwi = mc.likelihood * wi, lwo = mc.likelihood * wo;
        fx_t sum = fx_from_f32(lwi) * n_in;
        if (n_out)
            sum += fx_from_f32(lwo) * n_out;
        const float acc = fx_to_f32(sum);
        const float mu_A = acc > 0.0f ? rho_p / acc : 0.0f;
        const float mu_UA = m_occ_pred > 0.0f ? rho_p / m_occ_pred : 0.0f;
        const float a = mc.p_A * mu_A, b = (one - mc.p_A) * mu_UA;
        d.f[GF_MU_A][c] = mu_A;
        d.f[GF_MU_UA][c] = mu_UA;
        d.cellrec[c] = make_float4(a * lwi + b * wi, a * lwo + b * wo, rho_p, 0.0f);
        // As the general path leaves it: an occupancy update on its own, after the resampling moved the particles,
        // reads it for cells that hold none now.
        stream_store(&d.m_raw[c], m_raw_c);
    }
    stream_store(&d.born[c], rho_b);
    stream_store(&d.f[GF_PERS][c], rho_p);
    stream_store(&d.f[GF_NEW_BORN][c], rho_b);
    stream_store(&d.free[1][c], free_up);
    stream_store(&d.f[GF_OCC][c], occ_up);
    stream_store(&d.f[GF_PRED][c], m_occ_pred);
    return rho_b;
}

// One workgroup per 256-cell unit.  With born_sums set (the births run in the same step), the unit's
// exact sum of born masses goes to born_sums[unit] for the births' top-level scan, which then needs no
// tile pass over the born masses.  With exp_sums set (the resampling runs in the same step), the
// workgroups after the `units` cell units compute the tile totals of the resampling's exponentials
// (ALU work beside the memory-bound cell update) into exp_sums.
__global__ __launch_bounds__(BLOCK) void k_mass_update(const VehDesc* __restrict__ descs,
                                                       const uint32_t* __restrict__ tab, int zero_empty,
                                                       SegCarry carry, int occ_tile, fx_t* __restrict__ born_sums,
                                                       int units, const uint32_t* __restrict__ tab_e,
                                                       fx_t* __restrict__ exp_sums, int pph,
                                                       DevScalars* __restrict__ scs)
{
    if ((int)blockIdx.x >= units)
    {
        exp_tile_body(descs, tab_e, (int)blockIdx.x - units, exp_sums);
        return;
    }
    const TileRef tr = tile_ref(tab, 1, blockIdx.x);
    const VehDesc& d = descs[tr.v];
    const int c = tr.base + threadIdx.x;
    float rho_b = 0.0f;
    if (c < d.C)
        rho_b = mass_update_cell(d, c, zero_empty, carry, occ_tile, pph);
    if (!(rho_b >= 0.0f && rho_b <= BORN_MAX))
        scs[tr.v].born_odd = 1;
    if (born_sums)
    {
        fx_t total;
        block_exclusive_scan_fx(c < d.C ? fx_from_f32(rho_b) : (fx_t)0, &total);
        if (threadIdx.x == 0)
            born_sums[blockIdx.x] = total;
    }
}

// Vehicles with per-cell weights: first / last occurrence of every cell in the sorted particles (dogm.cu:262-281)
// and the out-of-grid particles of the border cells.  Bound by the read of the cell words (4 N) and the
// scattered 4-byte bounds; BOUNDS_ITEMS consecutive words per thread in 16-byte loads.
constexpr int BOUNDS_ITEMS = 4;
constexpr int BOUNDS_Q = BLOCK * BOUNDS_ITEMS / UNIT;

__global__ __launch_bounds__(BLOCK) void k_cell_bounds(const VehDesc* __restrict__ descs,
                                                       const uint32_t* __restrict__ tab, int pph)
{
    const TileRef tr = tile_ref(tab, BOUNDS_Q, blockIdx.x);
    const VehDesc& d = descs[tr.v];
    const int n = d.N;
    if (!d.wcell || tr.base >= n)
        return;
    const int* words = d.part[pph].idx;
    const int p0 = tr.base + threadIdx.x * BOUNDS_ITEMS;
    const int cnt = max(0, min(BOUNDS_ITEMS, n - p0));
    const int lane = threadIdx.x & (WAVE - 1);
    int w[BOUNDS_ITEMS];
    load_run<BOUNDS_ITEMS>(words, p0, cnt, w, -1);
    bool any_out = false;
#pragma unroll
    for (int i = 0; i < BOUNDS_ITEMS; ++i)
        any_out |= i < cnt && word_out(w[i]);
    int key[BOUNDS_ITEMS];
#pragma unroll
    for (int i = 0; i < BOUNDS_ITEMS; ++i)
        key[i] = i < cnt ? word_index(w[i]) : -1;
    int kprev = __shfl_up(key[BOUNDS_ITEMS - 1], 1, WAVE);
    int knext = __shfl_down(key[0], 1, WAVE);
    if (lane == 0)
        kprev = p0 > 0 && p0 <= n ? word_index(words[p0 - 1]) : -1;
    if (lane == WAVE - 1)
        knext = p0 + BOUNDS_ITEMS < n ? word_index(words[p0 + BOUNDS_ITEMS]) : -1;
#pragma unroll
    for (int i = 0; i < BOUNDS_ITEMS; ++i)
    {
        if (i >= cnt)
            break;
        if (key[i] != (i == 0 ? kprev : key[i - 1]))
            d.start[key[i]] = p0 + i;
        if (key[i] != (i == BOUNDS_ITEMS - 1 ? knext : key[i + 1]))
            d.end[key[i]] = p0 + i;
    }
    if (__ballot(any_out) == 0)
        return;
    // Out-of-grid particles: one atomic per run of equal cells in a thread, or one per wave inside a
    // long run (a far ego jump puts whole sides of the grid into a few cells).
    int* out = border_out(d);
    const int first = __shfl(key[0], 0, WAVE);
    bool one_cell = true;
    int mine = 0;
#pragma unroll
    for (int i = 0; i < BOUNDS_ITEMS; ++i)
    {
        one_cell &= i >= cnt || key[i] == first;
        mine += i < cnt && word_out(w[i]) ? 1 : 0;
    }
    if (__ballot(!one_cell) == 0)
    {
#pragma unroll
        for (int s = WAVE / 2; s > 0; s >>= 1)
            mine += __shfl_xor(mine, s, WAVE);
        if (lane == 0 && mine)
            atomicAdd(&out[first], mine);
        return;
    }
    int run = 0;
#pragma unroll
    for (int i = 0; i < BOUNDS_ITEMS; ++i)
    {
        run += i < cnt && word_out(w[i]) ? 1 : 0;
        const bool last = i == BOUNDS_ITEMS - 1 || key[i + 1] != key[i];
        if (i < cnt && last && run)
            atomicAdd(&out[key[i]], run);
        if (last)
            run = 0;
    }
}

// normalize_weights (mass_update.cu:51-59) for cells whose predicted occupancy exceeds 1.
__global__ __launch_bounds__(BLOCK) void k_normalize(const VehDesc* __restrict__ descs,
                                                     const uint32_t* __restrict__ tab, int pph)
{
    const TileRef tr = tile_ref(tab, 1, blockIdx.x);
    const VehDesc& d = descs[tr.v];
    const int i = tr.base + threadIdx.x;
    if (i >= d.N)
        return;
    const DescParticles P = d.part[pph];
    const float m = d.m_raw[P.idx[i]];
    if (m > 1.0f)
    {
        const float w = d.weight_array[i] / m;
        d.weight_array[i] = w;
        P.weight[i] = w;
    }
}

void run_occupancy(Engine* E, int pph, int zero_empty, bool defer_normalize, bool bounds, bool born_sums,
                   bool exp_sums)
{
    if (E->any_wcell)
    {
        launch_begin(E, K_CELL_BOUNDS);
        hipLaunchKernelGGL(k_cell_bounds, dim3(E->tiles(SP_P, BOUNDS_Q)), dim3(BLOCK), 0, E->stream, E->d_desc,
                           E->tab(SP_P), pph);
        launch_end(E, K_CELL_BOUNDS);
    }
    if (E->any_general && E->tune.seg_items == 4)
        launch_segreduce(E, K_SEG_OCC, K_SEG_OCC_FIX, OccOp<4>{pph, bounds ? 1 : 0}, false);
    else if (E->any_general)
        launch_segreduce(E, K_SEG_OCC, K_SEG_OCC_FIX, OccOp<8>{pph, bounds ? 1 : 0}, false);
    launch_begin(E, K_MASS_UPDATE);
    const int units = E->tiles(SP_C, 1);
    const int etiles = exp_sums ? E->tiles(SP_E, SCAN_Q) : 0;
    hipLaunchKernelGGL(k_mass_update, dim3(units + etiles), dim3(BLOCK), 0, E->stream, E->d_desc, E->tab(SP_C),
                       zero_empty, E->seg, BLOCK * E->tune.seg_items, born_sums ? born_unit_sums(E) : (fx_t*)nullptr,
                       units, E->tab(SP_E), E->exp_tile_sum, pph, E->scalars);
    launch_end(E, K_MASS_UPDATE);
    if (defer_normalize)
        return;
    launch_begin(E, K_NORMALIZE);
    hipLaunchKernelGGL(k_normalize, dim3(E->tiles(SP_P, 1)), dim3(BLOCK), 0, E->stream, E->d_desc, E->tab(SP_P),
                       pph);
    launch_end(E, K_NORMALIZE);
}

// ---------------------------------------------------------------------------------------------
// Persistent particle update (dogm/src/dogm.cu:300-321, update_persistent_particles.cu:16-87)
// ---------------------------------------------------------------------------------------------
// Kernel1 (lw = likelihood * w, written to weight_array) is fused into the reduction's load.
// norm: normalize_weights (mass_update.cu:51-59) is applied here, when the occupancy update ran in the
// same step: w <- w / m_occ_pred for cells whose predicted occupancy exceeds 1 (the particle weight is
// rewritten; weight_array is overwritten by lw below either way).
template <int IT>
struct PersOp
{
    static constexpr int NCH = 1;
    static constexpr int ITEMS = IT;
    static constexpr int WAVES = IT == 8 ? 6 : 8;
    int pph;
    int norm;
    int rec;  // write the cell factors of the moments' posterior weights (cellrec)
    __device__ const int* keys(const VehDesc& d) const { return d.part[pph].idx; }
    __device__ void head(const VehDesc&, int, int) const {}
    __device__ void end(const VehDesc&, int, int) const {}
    __device__ void cont(const VehDesc&, int) const {}
    __device__ void load(const VehDesc& d, int p0, int cnt, const int (&key)[ITEMS], float (&v)[ITEMS][NCH]) const
    {
        float w[ITEMS], lw[ITEMS], lik[ITEMS];
        load_run<ITEMS>(d.part[pph].weight, p0, cnt, w);
        if (norm)
        {
            // The occupancy update of this step left (likelihood, Σw) per cell with particles; every
            // item's pair is loaded before the first store.
            float m[ITEMS];
#pragma unroll
            for (int i = 0; i < ITEMS; ++i)
            {
                const float2 ci = i < cnt ? d.cellin[key[i]] : make_float2(0.0f, 0.0f);
                lik[i] = ci.x;
                m[i] = ci.y;
            }
#pragma unroll
            for (int i = 0; i < ITEMS; ++i)
            {
                if (i < cnt && m[i] > 1.0f)
                {
                    w[i] = w[i] / m[i];
                    d.part[pph].weight[p0 + i] = w[i];
                }
            }
        }
        else
        {
#pragma unroll
            for (int i = 0; i < ITEMS; ++i)
                lik[i] = i < cnt ? d.meas[key[i]].likelihood : 0.0f;
        }
#pragma unroll
        for (int i = 0; i < ITEMS; ++i)
        {
            lw[i] = i < cnt ? lik[i] * w[i] : 0.0f;
            v[i][0] = lw[i];
        }
        store_run<ITEMS>(d.weight_array.get(), p0, cnt, lw);
    }
    __device__ void finalize(const VehDesc& d, int key, const fx_t (&s)[1]) const
    {
        const float acc = fx_to_f32(s[0]);
        const float rho_p = d.f[GF_PERS][key];
        const float mu_A = acc > 0.0f ? rho_p / acc : 0.0f;
        d.f[GF_MU_A][key] = mu_A;
        const float pred = d.f[GF_PRED][key];
        const float mu_UA = pred > 0.0f ? rho_p / pred : 0.0f;
        d.f[GF_MU_UA][key] = mu_UA;
        if (rec)
        {
            // The factors of w = (p_A mu_A) w_lik + ((1 - p_A) mu_UA) w_prior in that association
            // (update_persistent_particles.cu:76-87), and rho_p for the moments.
            const float pA = d.meas[key].p_A;
            d.cellrec[key] = make_float4(pA * mu_A, (1.0f - pA) * mu_UA, rho_p, 0.0f);
        }
    }
};

// Writes 0 into fields [f_lo, f_hi] of every cell without particles.
__global__ __launch_bounds__(BLOCK) void k_empty_cells(const VehDesc* __restrict__ descs,
                                                       const uint32_t* __restrict__ tab, int f_lo, int f_hi)
{
    const TileRef tr = tile_ref(tab, 1, blockIdx.x);
    const VehDesc& d = descs[tr.v];
    const int c = tr.base + threadIdx.x;
    if (c >= d.C || d.start[c] != -1)
        return;
    for (int f = f_lo; f <= f_hi; ++f)
        d.f[f][c] = 0.0f;
}

__global__ __launch_bounds__(BLOCK) void k_post_weights(const VehDesc* __restrict__ descs,
                                                        const uint32_t* __restrict__ tab, int pph)
{
    const TileRef tr = tile_ref(tab, 1, blockIdx.x);
    const VehDesc& d = descs[tr.v];
    const int i = tr.base + threadIdx.x;
    if (i >= d.N)
        return;
    const DescParticles P = d.part[pph];
    const int c = P.idx[i];
    const float pA = d.meas[c].p_A;
    d.weight_array[i] = pA * d.f[GF_MU_A][c] * d.weight_array[i] + (1.0f - pA) * d.f[GF_MU_UA][c] * P.weight[i];
}

void run_persistent(Engine* E, int pph, bool fused_normalize, bool empty_done, bool defer_post)
{
    if (!E->any_general)
        return;  // full steps only: the occupancy update did it all
    if (E->tune.seg_items == 4)
        launch_segreduce(E, K_SEG_PERS, K_SEG_PERS_FIX, PersOp<4>{pph, fused_normalize ? 1 : 0, defer_post ? 1 : 0});
    else
        launch_segreduce(E, K_SEG_PERS, K_SEG_PERS_FIX, PersOp<8>{pph, fused_normalize ? 1 : 0, defer_post ? 1 : 0});
    if (!empty_done)
    {
        launch_begin(E, K_EMPTY_CELLS);
        hipLaunchKernelGGL(k_empty_cells, dim3(E->tiles(SP_C, 1)), dim3(BLOCK), 0, E->stream, E->d_desc,
                           E->tab(SP_C), (int)GF_MU_A, (int)GF_MU_UA);
        launch_end(E, K_EMPTY_CELLS);
    }
    if (defer_post)
        return;
    launch_begin(E, K_POST_WEIGHTS);
    hipLaunchKernelGGL(k_post_weights, dim3(E->tiles(SP_P, 1)), dim3(BLOCK), 0, E->stream, E->d_desc, E->tab(SP_P),
                       pph);
    launch_end(E, K_POST_WEIGHTS);
}

// Born masses per cell (first-frame placement when init_only, births otherwise).
struct SrcBorn
{
    static constexpr bool kNonNeg = false;
    int init_only;
    __device__ bool active(const VehDesc& d) const { return !init_only || d.init; }
    __device__ int len(const VehDesc& d) const { return d.C; }
    __device__ void load4(const VehDesc& d, int p0, int cnt, float (&v)[4]) const { load_run<4>(d.born, p0, cnt, v); }
    __device__ void seen(int, const float (&)[4], fx_t) const {}
};

__device__ __forceinline__ int order_end_at(int j, fx_t prefix, const DevScalars* sc, int C, int v)
{
    if (sc->total == 0)
        return order_end_uniform(j, C, v);
    if (j == C - 1)
        return v;
    return order_end(prefix, sc->scale, v);
}

// First-frame placement: P_j only.
struct SinkOrders
{
    __device__ void apply4(const VehDesc& d, const DevScalars* sc, int p0, int cnt, const fx_t (&pre)[4],
                           const fx_t (&)[4]) const
    {
        int e[4];
#pragma unroll
        for (int i = 0; i < 4; ++i)
            e[i] = i < cnt ? order_end_at(p0 + i, pre[i], sc, d.C, d.N) : 0;
        store_run<4>(d.pend.get(), p0, cnt, e);
    }
};

// Birth placement and weights per cell (init_new_particles.cu:126-155).
struct SinkBirth
{
    __device__ void apply4(const VehDesc& d, const DevScalars* sc, int p0, int cnt, const fx_t (&pre)[4],
                           const fx_t (&own)[4]) const
    {
        float bm[4];
        load_run<4>(d.born, p0, cnt, bm);
        const int C = d.C, v = d.B;
        int e[4];
        float a[4], u[4];
#pragma unroll
        for (int i = 0; i < 4; ++i)
        {
            e[i] = 0;
            a[i] = 0.0f;
            u[i] = 0.0f;
            if (i < cnt)
            {
                const int j = p0 + i;
                e[i] = order_end_at(j, pre[i], sc, C, v);
                // P_{j-1}: the previous item's end, or recomputed from the exclusive prefix.
                const int s = j == 0 ? 0 : (i > 0 ? e[i - 1] : order_end_at(j - 1, pre[i] - own[i], sc, C, v));
                const int n = e[i] - s;
                if (n > 0)  // cells without birth slots keep w_A = w_UA = 0 and skip the measurement read
                {
                    const float pA = d.meas[j].p_A;
                    const int nu_A = (int)roundf((float)n * pA);
                    const int nu_UA = n - nu_A;
                    a[i] = nu_A > 0 ? (pA * bm[i]) / (float)nu_A : 0.0f;
                    u[i] = nu_UA > 0 ? ((1.0f - pA) * bm[i]) / (float)nu_UA : 0.0f;
                }
            }
        }
        store_run<4>(d.pend.get(), p0, cnt, e);
        store_run<4>(d.f[GF_W_A].get(), p0, cnt, a);
        store_run<4>(d.f[GF_W_UA].get(), p0, cnt, u);
    }
};

// ---------------------------------------------------------------------------------------------
// Birth particles (dogm/src/dogm.cu:323-348, init.cu:46-67, init_new_particles.cu:157-195)
// ---------------------------------------------------------------------------------------------

// Cell of birth slot k, j = first index with pend[j] > k (pend non-decreasing, pend[C - 1] = B), for
// the 64 consecutive slots k_first .. k_first + 63 of a wave (all lanes call it; k_last is the last
// valid slot).  Lanes 0-31 and 32-63 run 32-ary searches for the cells of k_first and k_last (one
// wave-wide load per round instead of one dependent load per binary-search level); when those cells
// are fewer than 65 apart, each lane holds one pend entry of the range and finds its own cell with a
// six-step search over the lanes, otherwise it binary-searches the range.
__device__ int wave_slot_cells(const int* __restrict__ pend, int C, int k_first, int k_last, int k, int lane)
{
    const int half = lane >> 5, hl = lane & 31;
    const int target = half ? k_last : k_first;
    int lo = 0, hi = C - 1;  // the answer lies in [lo, hi]
    while (__ballot(lo < hi))
    {
        const int step = (hi - lo + 31) >> 5;
        const int pos = lo + (hl + 1) * step - 1;
        const bool le = lo < hi && pos < hi && pend[pos] <= target;
        const unsigned long long bal = __ballot(le);
        const int cnt = __popcll((bal >> (32 * half)) & 0xffffffffull);
        if (lo < hi)
        {
            const int nlo = lo + cnt * step;
            hi = min(hi, nlo + step - 1);
            lo = nlo;
        }
    }
    const int jlo = __shfl(lo, 0, WAVE);
    const int jhi = __shfl(lo, 32, WAVE);
    const int r = jhi - jlo + 1;
    if (r <= WAVE)
    {
        const int pv = jlo + lane <= jhi ? pend[jlo + lane] : 0x7fffffff;
        int cnt = 0;  // entries of the range <= k
#pragma unroll
        for (int bit = WAVE / 2; bit > 0; bit >>= 1)
        {
            const int cand = cnt + bit;
            const int v = __shfl(pv, cand - 1, WAVE);
            if (v <= k)
                cnt = cand;
        }
        return jlo + cnt;
    }
    return jlo + upper_bound_i32(pend + jlo, r, k);
}

// What the birth cells of a full step leave for the birth particles, 64 consecutive slots (a block) per wave: the
// cell that holds the block's first slot, and in birth.idx the cells of the slots whose cell starts inside the
// block (with the association flag).  Every block and every such slot is written by exactly one cell.  The
// records lie in the CDF buffer, free between the sort and the resampling.
struct BirthBlock
{
    int cell;
    int s, e;  // the cell's slots [s, e)
    int nu_A;
};

__device__ __forceinline__ BirthBlock* birth_blocks(const VehDesc& d)
{
    return reinterpret_cast<BirthBlock*>(d.cdf.get());
}

// Marks of the 64-cell groups with birth slots (Vehicle::pend), four per unit.
__device__ __forceinline__ uint8_t* birth_marks(const VehDesc& d)
{
    return reinterpret_cast<uint8_t*>(d.pend.get());
}

// Particle-order ends of a full step whose born masses are out of range: in the cell inputs, which the persistent update
// has read by then (pend holds the marks).
__device__ __forceinline__ int* odd_ends(const VehDesc& d)
{
    return reinterpret_cast<int*>(d.cellin.get());
}

// full: the slots' cells as the birth cells of a full step left them; otherwise (a stage-by-stage call, or masses
// whose prefixes need not be monotone) searched in the particle-order ends.
__global__ __launch_bounds__(BLOCK) void k_birth_particles(const VehDesc* __restrict__ descs,
                                                           const uint32_t* __restrict__ tab,
                                                           const DevScalars* __restrict__ scs, int full)
{
    const TileRef tr = tile_ref(tab, 1, blockIdx.x);
    const VehDesc& d = descs[tr.v];
    const int B = d.B;
    const int lane = threadIdx.x & (WAVE - 1);
    const int k0 = tr.base + (threadIdx.x - lane);  // the wave's first slot
    if (k0 >= B)
        return;  // wave-uniform
    const int k = k0 + lane;
    int j;
    bool assoc;
    if (full && !scs[tr.v].born_odd)
    {
        if (k >= B)
            return;
        const int4 b = reinterpret_cast<const int4*>(birth_blocks(d))[k0 / WAVE];
        const int w = d.birth.idx[k];
        const bool spans = k < b.z;
        j = spans ? b.x : word_index(w);
        assoc = spans ? (k - b.y) <= b.w : word_assoc(w) != 0;
    }
    else
    {
        const int* pend = full ? odd_ends(d) : d.pend.get();
        j = wave_slot_cells(pend, d.C, k0, min(k0 + WAVE - 1, B - 1), k, lane);
        if (k >= B)
            return;
        const int s = j > 0 ? pend[j - 1] : 0;
        const int n = pend[j] - s;
        const int nu_A = (int)roundf((float)n * d.meas[j].p_A);
        assoc = (k - s) <= nu_A;
    }
    const u32x4 r = draw(d.seed, d.inst, TAG_BIRTH, d.ep_birth, (uint32_t)k);
    float n0, n1;
    box_muller(r.x, r.y, &n0, &n1);
    const int gs = d.gs;
    d.birth.pos[k] = make_float2((float)(j % gs) + 0.5f, (float)j / (float)gs + 0.5f);
    d.birth.vel[k] = make_float2(normal_scale(n0, 0.0f, d.sd_birth), normal_scale(n1, 0.0f, d.sd_birth));
    d.birth.idx[k] = j;
    d.birth.weight[k] = assoc ? d.f[GF_W_A][j] : d.f[GF_W_UA][j];
    d.birth.assoc[k] = assoc ? 1 : 0;
}

// ---------------------------------------------------------------------------------------------
// First-measurement initialisation (dogm/src/dogm.cu:217-241, init_new_particles.cu:76-124),
// for the vehicles of the step whose descriptor has `init` set.
// ---------------------------------------------------------------------------------------------
__global__ __launch_bounds__(BLOCK) void k_copy_masses(const VehDesc* __restrict__ descs,
                                                       const uint32_t* __restrict__ tab)
{
    const TileRef tr = tile_ref(tab, 1, blockIdx.x);
    const VehDesc& d = descs[tr.v];
    const int c = tr.base + threadIdx.x;
    if (d.init && c < d.C)
        d.born[c] = d.meas[c].occ_mass;
}

__global__ __launch_bounds__(BLOCK) void k_init_particles(const VehDesc* __restrict__ descs,
                                                          const uint32_t* __restrict__ tab)
{
    const TileRef tr = tile_ref(tab, 1, blockIdx.x);
    const VehDesc& d = descs[tr.v];
    const int k = tr.base + threadIdx.x;
    if (!d.init || k >= d.N)
        return;
    const int gs = d.gs;
    const int j = upper_bound_i32(d.pend, d.C, k);
    const u32x4 r = draw(d.seed, d.inst, TAG_INIT_PARTICLES, d.ep_init, (uint32_t)k);
    const float v = d.vmax;
    const DescParticles P = d.part[0];
    P.pos[k] = make_float2((float)(j % gs) + 0.5f, (float)(j / gs) + 0.5f);
    P.vel[k] = make_float2(-v + (v - -v) * uniform01(r.x), -v + (v - -v) * uniform01(r.y));
    P.idx[k] = j;
    P.weight[k] = 1.0f / (float)d.N;  // dogm.cu:228
    P.assoc[k] = 0;
}

void run_init_particles(Engine* E)
{
    launch_begin(E, K_COPY_MASSES);
    hipLaunchKernelGGL(k_copy_masses, dim3(E->tiles(SP_C, 1)), dim3(BLOCK), 0, E->stream, E->d_desc, E->tab(SP_C));
    launch_end(E, K_COPY_MASSES);
    run_exact_scan(E, SrcBorn{1}, SinkOrders{}, SCAN_ORDERS_N, K_INIT_CELLS, ONLY_INIT);
    launch_begin(E, K_INIT_PARTICLES);
    hipLaunchKernelGGL(k_init_particles, dim3(E->tiles(SP_P, 1)), dim3(BLOCK), 0, E->stream, E->d_desc,
                       E->tab(SP_P));
    launch_end(E, K_INIT_PARTICLES);
}

// ---------------------------------------------------------------------------------------------
// Statistical moments (dogm/src/dogm.cu:350-384, statistical_moments.cu:16-106)
// ---------------------------------------------------------------------------------------------
// Per-cell sums of the five velocity channels w vx, w vy, w vx^2, w vy^2, w vx vy (f32 products
// widened to f64) in one fixed association, independent of the launch shape and of the other
// vehicles of the step: a grid's sorted particles are cut into chunks of 256 (one wave64 per chunk,
// 4 consecutive particles per lane).
//   lane:   sequential fold restarting where a cell starts (the lane's first particle always starts it);
//   wave:   segmented inclusive scan of the lanes' last folds in six DPP steps (row shifts 1, 2, 4, 8
//           inside 16-lane rows, then lane 15 of rows 0 / 2 into rows 1 / 3, lane 31 into rows 2 / 3),
//           each adding the moved value only while no cell starts in between;
//   cell:   ending in lane l: its lane-local fold if it starts in lane l, else (scan of lane l - 1) +
//           fold;
//   chunks: a cell crossing chunks is the left fold ((first piece + whole middle chunk) + ...) + last
//           piece, summed by k_moments_fix from the chunks' carries.
// The float sums are then rounded once to f32 and finalised as in statistical_moments.cu:58-106.
// With post set (the persistent update ran in the same step) the posterior weights
// (update_persistent_particles.cu:76-87) are formed in the load: w = p_A mu_A lw + (1 - p_A) mu_UA
// w_prior, written to weight_array and used for the moments.
constexpr int MOM_CH = 5;
constexpr int MOM_ITEMS = 4;                  // consecutive particles per lane
constexpr int MOM_CHUNK = WAVE * MOM_ITEMS;   // particles per wave
static_assert(MOM_CHUNK == UNIT, "a moments chunk is one work-table unit");
constexpr uint8_t MC_CONT = 1;    // the chunk's last cell continues into the next chunk
constexpr uint8_t MC_NOHEAD = 2;  // no cell starts in the chunk

// rho_p = the cell's persistent occupancy mass (d.f[GF_PERS][key]).
__device__ __forceinline__ void mom_finalize(const VehDesc& d, int key, float rho_p, const float (&s)[MOM_CH])
{
    float mx = 0.0f, my = 0.0f, vx = 0.0f, vy = 0.0f, cv = 0.0f;
    if (rho_p > 0.0f)
    {
        const float inv = 1.0f / rho_p;
        mx = inv * s[0];
        my = inv * s[1];
        vx = inv * s[2] - mx * mx;
        vy = inv * s[3] - my * my;
        cv = inv * s[4] - mx * my;
    }
    d.f[GF_MEAN_X][key] = mx;
    d.f[GF_MEAN_Y][key] = my;
    d.f[GF_VAR_X][key] = vx;
    d.f[GF_VAR_Y][key] = vy;
    d.f[GF_COVAR][key] = cv;
}

template <int CTRL, int ROW_MASK>
__device__ __forceinline__ int dpp_i(int x)
{
    return __builtin_amdgcn_update_dpp(0, x, CTRL, ROW_MASK, 0xf, false);
}

// carry.flags[unit], and per unit MOM_CH doubles in carry.head_partial (piece of the chunk's first
// cell when that cell started in an earlier chunk) and carry.tail_partial (piece of its last cell).
// The first `top` workgroups (full steps) scan the birth orders, one vehicle each: single-workgroup latency (12 us at
// 1200 x 1200 cells) beside the particle work instead of in a launch of its own.
struct BirthTop
{
    int m;                  // vehicles
    const fx_t* unit_sums;  // born masses per cell unit
    fx_t* tile_pre;
    DevScalars* scalars;
};

// CELLS: the vehicles with per-cell weights (their records hold the posterior weights, so no prior or
// likelihood weights are read: 16 N instead of 24 N); else the others.  Bound by the latency of the cell
// records and of the f64 scans.  With the unit's index as a scalar (wave_index) the descriptor and its pointers take
// no vector registers and no vector loads: 19.5 -> 16.3 us at 2e6 particles, 66 registers for seven waves per
// SIMD; eight (4 registers spilled) take 17.9.
template <int WAVES_PER_WG, bool CELLS>
__global__ __launch_bounds__(WAVES_PER_WG* WAVE) __attribute__((amdgpu_waves_per_eu(7)))
void k_moments(const VehDesc* __restrict__ descs, const uint32_t* __restrict__ tab, int pph, int post,
               SegCarry carry, int top, BirthTop births)
{
    if ((int)blockIdx.x < top)
    {
        if ((int)blockIdx.x < births.m)
            scan_top_orders<WAVES_PER_WG * WAVE>(descs, blockIdx.x, births.unit_sums, births.tile_pre, births.scalars,
                                                 SCAN_ORDERS_B, ONLY_ALL, SCAN_Q);
        return;
    }
    const int lane = threadIdx.x & (WAVE - 1);
    const int unit = xcd_tile((int)blockIdx.x - top, (int)gridDim.x - top) * WAVES_PER_WG + wave_index();
    const TileRef tr = tile_ref(tab, 1, unit);
    const VehDesc& d = descs[tr.v];
    if (CELLS != (d.wcell != 0))
        return;
    const int n = d.N;
    const int base = tr.base;
    if (base >= n)
    {
        if (lane == 0)
            carry.flags[unit] = 0;  // padding chunk past the vehicle's particles
        return;                     // wave-uniform
    }
    const int p0 = base + lane * MOM_ITEMS;
    const int cnt = max(0, min(MOM_ITEMS, n - p0));
    const int* words = d.part[pph].idx;
    int word[MOM_ITEMS], key[MOM_ITEMS];
    load_run<MOM_ITEMS>(words, p0, cnt, word, -1);
#pragma unroll
    for (int i = 0; i < MOM_ITEMS; ++i)
        key[i] = i < cnt ? word_index(word[i]) : -1;
    int kprev = __shfl_up(key[MOM_ITEMS - 1], 1, WAVE);
    int knext = __shfl_down(key[0], 1, WAVE);
    if (lane == 0)
        kprev = base > 0 ? word_index(words[base - 1]) : -1;
    if (lane == WAVE - 1)
        knext = p0 + MOM_ITEMS < n ? word_index(words[p0 + MOM_ITEMS]) : -1;
    bool head[MOM_ITEMS], end[MOM_ITEMS], started[MOM_ITEMS];
    bool lh = false;
#pragma unroll
    for (int i = 0; i < MOM_ITEMS; ++i)
    {
        const int kp = i == 0 ? kprev : key[i - 1];
        const int kn = i == MOM_ITEMS - 1 ? knext : key[i + 1];
        head[i] = i < cnt && key[i] != kp;
        end[i] = i < cnt && key[i] != kn;
        lh = lh || head[i];
        started[i] = lh;
    }

    // The persistent masses of the cells ending here (and with post the cells' weight factors, which
    // carry them), loaded before any store so that they travel with the other loads instead of
    // waiting behind the weight_array stores.
    float rho[MOM_ITEMS];
    float w[MOM_ITEMS];
    if constexpr (CELLS)
    {
        // The cell record holds the posterior weights themselves (mass_update_cell).
#pragma unroll
        for (int i = 0; i < MOM_ITEMS; ++i)
        {
            float in = 0.0f, out = 0.0f;
            rho[i] = 0.0f;
            if (i < cnt)
            {
                const float4 cf = d.cellrec[key[i]];
                in = cf.x;
                out = cf.y;
                rho[i] = cf.z;
            }
            w[i] = word_out(word[i]) ? out : in;
        }
        store_run<MOM_ITEMS>(d.weight_array.get(), p0, cnt, w);
    }
    else
    {
        float4 cf[MOM_ITEMS];
#pragma unroll
        for (int i = 0; i < MOM_ITEMS; ++i)
        {
            cf[i] = post && i < cnt ? d.cellrec[key[i]] : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
            rho[i] = post ? cf[i].z : (end[i] ? d.f[GF_PERS][key[i]] : 0.0f);
        }
        load_run<MOM_ITEMS>(d.weight_array, p0, cnt, w);
        if (post)
        {
            float wp[MOM_ITEMS];
            load_run<MOM_ITEMS>(d.part[pph].weight, p0, cnt, wp);
#pragma unroll
            for (int i = 0; i < MOM_ITEMS; ++i)
                if (i < cnt)
                    w[i] = cf[i].x * w[i] + cf[i].y * wp[i];  // (p_A mu_A) w + ((1 - p_A) mu_UA) w_prior
            store_run<MOM_ITEMS>(d.weight_array.get(), p0, cnt, w);
        }
    }
    float vx[MOM_ITEMS], vy[MOM_ITEMS];
    {
        const float2* vel = d.part[pph].vel;
        if (cnt == MOM_ITEMS)
        {
            const float4 a = *reinterpret_cast<const float4*>(vel + p0);
            const float4 b = *reinterpret_cast<const float4*>(vel + p0 + 2);
            vx[0] = a.x; vy[0] = a.y; vx[1] = a.z; vy[1] = a.w;
            vx[2] = b.x; vy[2] = b.y; vx[3] = b.z; vy[3] = b.w;
        }
        else
        {
#pragma unroll
            for (int i = 0; i < MOM_ITEMS; ++i)
            {
                const float2 v = i < cnt ? vel[p0 + i] : make_float2(0.0f, 0.0f);
                vx[i] = v.x;
                vy[i] = v.y;
            }
        }
    }

    // Combine predicates of the six scan steps (the same for every channel): the source lane is in
    // range and no cell starts between it and this lane.
    bool comb[6];
    {
        const int row = lane >> 4, rl = lane & 15;
        int f = lh ? 1 : 0;
        int g;
        g = dpp_i<0x111, 0xf>(f); comb[0] = rl >= 1 && !f; f = rl >= 1 ? (f | g) : f;
        g = dpp_i<0x112, 0xf>(f); comb[1] = rl >= 2 && !f; f = rl >= 2 ? (f | g) : f;
        g = dpp_i<0x114, 0xf>(f); comb[2] = rl >= 4 && !f; f = rl >= 4 ? (f | g) : f;
        g = dpp_i<0x118, 0xf>(f); comb[3] = rl >= 8 && !f; f = rl >= 8 ? (f | g) : f;
        const bool b15 = row == 1 || row == 3, b31 = row >= 2;
        g = dpp_i<0x142, 0xa>(f); comb[4] = b15 && !f; f = b15 ? (f | g) : f;
        comb[5] = b31 && !f;
    }
    // The chunk's first cell started in an earlier chunk (lane 0's first particle is no cell start);
    // its first end is lane first_end_lane's particle first_i.
    const bool from_before = base > 0 && !(__ballot(head[0]) & 1ull);
    const uint64_t endlanes = __ballot(end[0] || end[1] || end[2] || end[3]);
    const int first_end_lane = endlanes ? __builtin_ctzll(endlanes) : WAVE;
    const int first_i = end[0] ? 0 : end[1] ? 1 : end[2] ? 2 : 3;
    const bool nohead = __ballot(lh) == 0;
    // The chunk's last cell continues into the next chunk: lane 63 holds 4 particles and the last
    // is no cell end.
    const bool cont = (__ballot(cnt == MOM_ITEMS && !end[MOM_ITEMS - 1]) >> (WAVE - 1)) & 1ull;

    float s32[MOM_ITEMS][MOM_CH];
#pragma unroll
    for (int c = 0; c < MOM_CH; ++c)
    {
        double r[MOM_ITEMS];
#pragma unroll
        for (int i = 0; i < MOM_ITEMS; ++i)
        {
            const float wv = w[i] * vx[i], wy = w[i] * vy[i];
            const float xf = c == 0 ? wv : c == 1 ? wy : c == 2 ? wv * vx[i] : c == 3 ? wy * vy[i] : wv * vy[i];
            const double x = (double)xf;
            if (i == 0)
                r[i] = x;
            else if (i < cnt)
                r[i] = head[i] ? x : r[i - 1] + x;
            else
                r[i] = r[i - 1];
        }
        double S = r[MOM_ITEMS - 1];
        { const double y = dpp_val<0x111, 0xf>(S); S = comb[0] ? y + S : S; }
        { const double y = dpp_val<0x112, 0xf>(S); S = comb[1] ? y + S : S; }
        { const double y = dpp_val<0x114, 0xf>(S); S = comb[2] ? y + S : S; }
        { const double y = dpp_val<0x118, 0xf>(S); S = comb[3] ? y + S : S; }
        { const double y = dpp_val<0x142, 0xa>(S); S = comb[4] ? y + S : S; }
        { const double y = dpp_val<0x143, 0xc>(S); S = comb[5] ? y + S : S; }
        const double E = __shfl_up(S, 1, WAVE);
#pragma unroll
        for (int i = 0; i < MOM_ITEMS; ++i)
        {
            const double v = (started[i] || lane == 0) ? r[i] : E + r[i];
            s32[i][c] = (float)v;
            if (end[i] && from_before && lane == first_end_lane && i == first_i)
                reinterpret_cast<double*>(carry.head_partial)[(size_t)unit * MOM_CH + c] = v;
        }
        if (lane == WAVE - 1 && cont)
            reinterpret_cast<double*>(carry.tail_partial)[(size_t)unit * MOM_CH + c] = S;
    }
    if (lane == 0)
        carry.flags[unit] = (uint8_t)((cont ? MC_CONT : 0) | (nohead ? MC_NOHEAD : 0));
#pragma unroll
    for (int i = 0; i < MOM_ITEMS; ++i)
    {
        if (!end[i])
            continue;
        if (from_before && lane == first_end_lane && i == first_i)
            continue;  // the cell started in an earlier chunk: k_moments_fix
        float s[MOM_CH];
#pragma unroll
        for (int c = 0; c < MOM_CH; ++c)
            s[c] = s32[i][c];
        mom_finalize(d, key[i], rho[i], s);
    }
}

// Cells crossing chunks: one thread per chunk u whose last cell starts in it and continues.
__device__ __forceinline__ void moments_fix_chunk(const VehDesc* __restrict__ descs, const uint32_t* __restrict__ tab,
                                                  int u, int units, int pph, const SegCarry& carry)
{
    if (u >= units)
        return;
    const uint8_t fl = carry.flags[u];
    if (!(fl & MC_CONT) || (fl & MC_NOHEAD))
        return;
    const double* tail = reinterpret_cast<const double*>(carry.tail_partial);
    const double* headp = reinterpret_cast<const double*>(carry.head_partial);
    double acc[MOM_CH];
#pragma unroll
    for (int c = 0; c < MOM_CH; ++c)
        acc[c] = tail[(size_t)u * MOM_CH + c];
    int j = u + 1;
    while ((carry.flags[j] & (MC_CONT | MC_NOHEAD)) == (MC_CONT | MC_NOHEAD))
    {
#pragma unroll
        for (int c = 0; c < MOM_CH; ++c)
            acc[c] = acc[c] + tail[(size_t)j * MOM_CH + c];
        ++j;
    }
    float s[MOM_CH];
#pragma unroll
    for (int c = 0; c < MOM_CH; ++c)
        s[c] = (float)(acc[c] + headp[(size_t)j * MOM_CH + c]);
    const TileRef tr = tile_ref(tab, 1, u);
    const VehDesc& d = descs[tr.v];
    const int key = word_index(d.part[pph].idx[tr.base + MOM_CHUNK - 1]);
    mom_finalize(d, key, d.f[GF_PERS][key], s);
}

__global__ __launch_bounds__(BLOCK) void k_moments_fix(const VehDesc* __restrict__ descs,
                                                       const uint32_t* __restrict__ tab, int units, int pph,
                                                       SegCarry carry)
{
    moments_fix_chunk(descs, tab, blockIdx.x * BLOCK + threadIdx.x, units, pph, carry);
}

constexpr int MOM_WAVES_PER_WG = 4;
static_assert(MOM_WAVES_PER_WG * WAVE == BLOCK, "the births' scan shares the moments' launch");

void run_moments(Engine* E, int pph, bool fused_post, bool empty_done, bool births_top)
{
    const int units = (int)E->units[SP_P];
    if (units > 0)
    {
        // The scan's workgroups come first (they are the longest), padded to whole rounds of the 8 XCDs.
        int top = births_top ? div_up(E->m, 8) * 8 : 0;
        const BirthTop bt{E->m, born_unit_sums(E), E->scan_tile_pre, E->scalars};
        const dim3 block(MOM_WAVES_PER_WG * WAVE);
        launch_begin(E, K_SEG_MOM);
        if (E->any_wcell)
        {
            hipLaunchKernelGGL((k_moments<MOM_WAVES_PER_WG, true>), dim3(top + units / MOM_WAVES_PER_WG), block, 0,
                               E->stream, E->d_desc, E->tab(SP_P), pph, 1, E->seg, top, bt);
            top = 0;
        }
        if (E->any_general)
            hipLaunchKernelGGL((k_moments<MOM_WAVES_PER_WG, false>), dim3(top + units / MOM_WAVES_PER_WG), block, 0,
                               E->stream, E->d_desc, E->tab(SP_P), pph, fused_post ? 1 : 0, E->seg, top, bt);
        launch_end(E, K_SEG_MOM);
        if (!births_top)
        {
            launch_begin(E, K_SEG_MOM_FIX);
            hipLaunchKernelGGL(k_moments_fix, dim3(div_up(units, BLOCK)), dim3(BLOCK), 0, E->stream, E->d_desc,
                               E->tab(SP_P), units, pph, E->seg);
            launch_end(E, K_SEG_MOM_FIX);
        }
    }
    if (empty_done)
        return;
    launch_begin(E, K_EMPTY_CELLS);
    hipLaunchKernelGGL(k_empty_cells, dim3(E->tiles(SP_C, 1)), dim3(BLOCK), 0, E->stream, E->d_desc, E->tab(SP_C),
                       (int)GF_MEAN_X, (int)GF_COVAR);
    launch_end(E, K_EMPTY_CELLS);
}

// Birth cells of a full step, 256 cells (a unit) per workgroup with one cell per lane (IT = 1) or per wave with
// four (IT = 4).  Cells without born mass have no births (equal prefixes round to equal particle orders), so
// a unit without any converts and rounds nothing; it only stores zero w_A and w_UA where the last full update
// left births.  The others hand their slots to the birth particles (BirthBlock), which then need no search over
// the particle-order ends, and those are not stored.
// Bound by the dependent chain of the few units with births (exact scan, roundings, the association
// probability, divisions, slots): IT = 1 spreads it over four times the waves, which wins while the launch leaves
// the GPU idle, IT = 4 has a quarter of the waves, which wins on large grids and batches.  Measured IT = 1 / IT = 4 in
// us by cell units of the launch: 245 (250 x 250) 8.5 / 10.6, 1024 (16 x 128 x 128) 9.9 / 11.9, 1407 (600 x 600) 9.6 /
// 11.2, 2823 (850 x 850) 11.5 / 12.0, 3907 (1000 x 1000) 12.9 / 12.3, 5000 (8 x 400 x 400) 18.6 / 16.1, 5625 (1200 x
// 1200) 14.7 / 12.8, 16384 (2048 x 2048) 33.1 / 27.7, 32768 (32 x 512 x 512) 79.6 / 47.0.  The line lies a little above
// where they meet (about 3000 units, 1% of the step between).  The birth particles went from 10.9 to 5.1 us at 2e5
// slots.
constexpr int BIRTH_WIDE_UNITS = 4096;

template <int IT>
__device__ __forceinline__ void birth_cells_unit(const VehDesc* __restrict__ descs, const uint32_t* __restrict__ tab,
                                                 int unit, const fx_t* __restrict__ tile_pre,
                                                 const fx_t* __restrict__ unit_sums,
                                                 const DevScalars* __restrict__ scs)
{
    constexpr int GROUP = WAVE / IT;  // lanes per 64 cells (one mark)
    const TileRef tr = tile_ref(tab, 1, unit);
    const VehDesc& d = descs[tr.v];
    const DevScalars* sc = scs + tr.v;
    const int C = d.C, v = d.B;
    if (tr.base >= C)
        return;
    const int lane = threadIdx.x & (WAVE - 1), wid = wave_index();
    const int w0 = tr.base + (IT == 1 ? wid * WAVE : 0);  // the wave's first cell
    const int p0 = w0 + lane * IT;
    const int cnt = max(0, min(IT, C - p0));
    // Every load that does not depend on a value comes first: the chain below is what bounds the kernel.
    float f[IT];
    load_run<IT>(d.born, p0, cnt, f);
    // The unit's prefix: its tile's plus the tile's earlier units (a vehicle's units start on a tile boundary).
    fx_t before = tile_pre[unit / SCAN_Q];
#pragma unroll
    for (int q = 0; q < SCAN_Q - 1; ++q)
    {
        const fx_t x = unit_sums[unit - unit % SCAN_Q + q];
        before += q < unit % SCAN_Q ? x : (fx_t)0;
    }
    const bool uniform = sc->total == 0;  // equal split over all cells
    const bool odd = sc->born_odd != 0;
    const bool all = uniform || odd || tr.base + UNIT >= C;  // (the last cell takes the remainder)
    uint8_t* mark = birth_marks(d) + w0 / WAVE;
    const uint32_t marks = w0 >= C ? 0u : IT == 1 ? *mark : *reinterpret_cast<const uint32_t*>(mark);
    const bool had = !d.marks_valid || marks != 0;
    fx_t run = 0;
    int e[IT], s[IT], nu_A[IT];
    float a[IT], u[IT];
    bool any = false, mass = false;
#pragma unroll
    for (int i = 0; i < IT; ++i)
    {
        e[i] = s[i] = nu_A[i] = 0;
        a[i] = u[i] = 0.0f;
        mass |= f[i] != 0.0f;
    }
    // With one cell per lane a wave's prefix needs the unit's other waves, so the unit decides together.
    const bool active = (IT == 1 ? __syncthreads_or(mass) : __ballot(mass) != 0) || all;
    if (active)
    {
        // Loaded beside the scan, not in the branch of a cell with births, behind it.
        float pA[IT];
#pragma unroll
        for (int i = 0; i < IT; ++i)
            pA[i] = i < cnt && (f[i] != 0.0f || all) ? d.meas[p0 + i].p_A : 0.0f;
        fx_t own[IT], sum = 0;
#pragma unroll
        for (int i = 0; i < IT; ++i)
        {
            own[i] = fx_from_f32(f[i]);
            sum += own[i];
        }
        const fx_t incl = wave_inclusive_scan_fx(sum);
        if constexpr (IT == 1)
        {
            __shared__ fx_t s_wave[BLOCK / WAVE];
            if (lane == WAVE - 1)
                s_wave[wid] = incl;
            __syncthreads();
#pragma unroll
            for (int w = 0; w < BLOCK / WAVE - 1; ++w)
                before += w < wid ? s_wave[w] : (fx_t)0;
        }
        run = before + incl - sum;
        // P_{j-1} of the lane's first cell, then P_j cell by cell.
        int prev = p0 == 0 || cnt == 0 ? 0 : order_end_at(p0 - 1, run, sc, C, v);
#pragma unroll
        for (int i = 0; i < IT; ++i)
        {
            const int j = p0 + i;
            run += own[i];
            s[i] = e[i] = prev;
            if (i < cnt)
            {
                if (f[i] != 0.0f || all)
                    e[i] = order_end_at(j, run, sc, C, v);
                const int n = e[i] - prev;
                if (n > 0)  // cells without birth slots keep w_A = w_UA = 0
                {
                    nu_A[i] = (int)roundf((float)n * pA[i]);
                    const int nu_UA = n - nu_A[i];
                    a[i] = nu_A[i] > 0 ? (pA[i] * f[i]) / (float)nu_A[i] : 0.0f;
                    u[i] = nu_UA > 0 ? ((1.0f - pA[i]) * f[i]) / (float)nu_UA : 0.0f;
                    any = true;
                }
                prev = e[i];
            }
        }
    }
    const uint64_t births = __ballot(any);
    if (had || births)
    {
        store_run<IT>(d.f[GF_W_A].get(), p0, cnt, a);
        store_run<IT>(d.f[GF_W_UA].get(), p0, cnt, u);
        if (cnt > 0 && lane % GROUP == 0)
            mark[lane / GROUP] = GROUP == WAVE ? births != 0 : ((births >> lane) & ((1ull << (GROUP & 63)) - 1)) != 0;
    }
    if (odd)
    {
        store_run<IT>(odd_ends(d), p0, cnt, e);  // the birth particles search
        return;
    }
    if (!births)
        return;
    // The slots [s, e) of a cell: those before the first block boundary one by one, then one record per block.
    int* words = d.birth.idx;
    BirthBlock* blocks = birth_blocks(d);
    const auto put = [&](int cell, int s0, int e0, int nu, int first, int step) {
        const int q0 = (s0 + WAVE - 1) / WAVE;
        for (int k = s0 + first; k < min(e0, q0 * WAVE); k += step)
            words[k] = (int)((unsigned)cell | ((k - s0) <= nu ? WORD_ASSOC : 0u));
        for (int q = q0 + first; q * WAVE < e0; q += step)
            blocks[q] = BirthBlock{cell, s0, e0, nu};
    };
#pragma unroll
    for (int i = 0; i < IT; ++i)
    {
        const bool many = e[i] - s[i] > 8;
        if (e[i] > s[i] && !many)
            put(p0 + i, s[i], e[i], nu_A[i], 0, 1);
        // Cells with many slots by the whole wave, one after the other.
        uint64_t todo = __ballot(many);
        while (todo)
        {
            const int l = __builtin_ctzll(todo);
            todo &= todo - 1;
            put(w0 + l * IT + i, __shfl(s[i], l, WAVE), __shfl(e[i], l, WAVE), __shfl(nu_A[i], l, WAVE), lane, WAVE);
        }
    }
}

// The birth cells of a full step, and in the workgroups after the `cell_groups` the moments of cells crossing
// chunks (both wait for the moments' launch only; as a launch of its own the latter took 4 to 5 us).
template <int IT>
__global__ __launch_bounds__(BLOCK) void k_birth_cells(const VehDesc* __restrict__ descs,
                                                       const uint32_t* __restrict__ tab_c, int cell_groups,
                                                       const fx_t* __restrict__ tile_pre,
                                                       const fx_t* __restrict__ unit_sums,
                                                       const DevScalars* __restrict__ scs,
                                                       const uint32_t* __restrict__ tab_p, int units, int pph,
                                                       SegCarry carry)
{
    const int group = blockIdx.x;
    if (group < cell_groups)
        birth_cells_unit<IT>(descs, tab_c, IT == 1 ? group : group * (BLOCK / WAVE) + wave_index(), tile_pre,
                             unit_sums, scs);
    else
        moments_fix_chunk(descs, tab_p, (group - cell_groups) * BLOCK + (int)threadIdx.x, units, pph, carry);
}

void run_births(Engine* E, bool moments_first, int pph)
{
    // With B = 0 the cell pass still runs (every cell gets n_j = 0 and w_A = w_UA = 0) and the
    // stage still consumes its RNG epoch, so the stream of later stages does not depend on B.
    if (moments_first)
    {
        const int cell_units = E->tiles(SP_C, 1), units = (int)E->units[SP_P], fix = div_up(units, BLOCK);
        const bool wide = cell_units > BIRTH_WIDE_UNITS;
        const int groups = wide ? cell_units / (BLOCK / WAVE) : cell_units;
        launch_begin(E, K_BIRTH_CELLS);
        if (wide)
            hipLaunchKernelGGL(k_birth_cells<4>, dim3(groups + fix), dim3(BLOCK), 0, E->stream, E->d_desc,
                               E->tab(SP_C), groups, E->scan_tile_pre, born_unit_sums(E), E->scalars, E->tab(SP_P),
                               units, pph, E->seg);
        else
            hipLaunchKernelGGL(k_birth_cells<1>, dim3(groups + fix), dim3(BLOCK), 0, E->stream, E->d_desc,
                               E->tab(SP_C), groups, E->scan_tile_pre, born_unit_sums(E), E->scalars, E->tab(SP_P),
                               units, pph, E->seg);
        launch_end(E, K_BIRTH_CELLS);
    }
    else
    {
        run_exact_scan(E, SrcBorn{0}, SinkBirth{}, SCAN_ORDERS_B, K_BIRTH_CELLS, ONLY_ALL);
    }
    const int blocks = E->tiles(SP_B, 1);
    if (blocks <= 0)
        return;
    launch_begin(E, K_BIRTH_PARTICLES);
    hipLaunchKernelGGL(k_birth_particles, dim3(blocks), dim3(BLOCK), 0, E->stream, E->d_desc, E->tab(SP_B), E->scalars,
                       moments_first ? 1 : 0);
    launch_end(E, K_BIRTH_PARTICLES);
}

// ---------------------------------------------------------------------------------------------
// Grid packing for read-back / injection (dogm_grid_cell AoS <-> structure-of-arrays)
// ---------------------------------------------------------------------------------------------
__global__ __launch_bounds__(BLOCK) void k_pack_grid(DevGrid G, dogm_grid_cell* __restrict__ out, int C)
{
    const int c = blockIdx.x * BLOCK + threadIdx.x;
    if (c >= C)
        return;
    dogm_grid_cell g;
    g.start_idx = G.start[c];
    g.end_idx = G.end[c];
    g.new_born_occ_mass = G.f[GF_NEW_BORN][c];
    g.pers_occ_mass = G.f[GF_PERS][c];
    g.free_mass = G.f[GF_FREE][c];
    g.occ_mass = G.f[GF_OCC][c];
    g.pred_occ_mass = G.f[GF_PRED][c];
    g.mu_A = G.f[GF_MU_A][c];
    g.mu_UA = G.f[GF_MU_UA][c];
    g.w_A = G.f[GF_W_A][c];
    g.w_UA = G.f[GF_W_UA][c];
    g.mean_x_vel = G.f[GF_MEAN_X][c];
    g.mean_y_vel = G.f[GF_MEAN_Y][c];
    g.var_x_vel = G.f[GF_VAR_X][c];
    g.var_y_vel = G.f[GF_VAR_Y][c];
    g.covar_xy_vel = G.f[GF_COVAR][c];
    out[c] = g;
}

__global__ __launch_bounds__(BLOCK) void k_unpack_grid(DevGrid G, const dogm_grid_cell* __restrict__ in, int C)
{
    const int c = blockIdx.x * BLOCK + threadIdx.x;
    if (c >= C)
        return;
    const dogm_grid_cell g = in[c];
    G.start[c] = g.start_idx;
    G.end[c] = g.end_idx;
    G.f[GF_NEW_BORN][c] = g.new_born_occ_mass;
    G.f[GF_PERS][c] = g.pers_occ_mass;
    G.f[GF_FREE][c] = g.free_mass;
    G.f[GF_OCC][c] = g.occ_mass;
    G.f[GF_PRED][c] = g.pred_occ_mass;
    G.f[GF_MU_A][c] = g.mu_A;
    G.f[GF_MU_UA][c] = g.mu_UA;
    G.f[GF_W_A][c] = g.w_A;
    G.f[GF_W_UA][c] = g.w_UA;
    G.f[GF_MEAN_X][c] = g.mean_x_vel;
    G.f[GF_MEAN_Y][c] = g.mean_y_vel;
    G.f[GF_VAR_X][c] = g.var_x_vel;
    G.f[GF_VAR_Y][c] = g.var_y_vel;
    G.f[GF_COVAR][c] = g.covar_xy_vel;
}

__global__ __launch_bounds__(BLOCK) void k_pack_state(DevParticles P, int n, float4* __restrict__ out)
{
    const int i = blockIdx.x * BLOCK + threadIdx.x;
    if (i >= n)
        return;
    const float2 p = P.pos[i], v = P.vel[i];
    out[i] = make_float4(p.x, p.y, v.x, v.y);
}

__global__ __launch_bounds__(BLOCK) void k_unpack_state(DevParticles P, int n, const float4* __restrict__ in)
{
    const int i = blockIdx.x * BLOCK + threadIdx.x;
    if (i >= n)
        return;
    const float4 s = in[i];
    P.pos[i] = make_float2(s.x, s.y);
    P.vel[i] = make_float2(s.z, s.w);
}

void run_pack_state(Engine* E, const DevParticles& p, int n, float4* out)
{
    if (n <= 0)
        return;
    launch_begin(E, K_PACK_STATE);
    hipLaunchKernelGGL(k_pack_state, dim3(div_up(n, BLOCK)), dim3(BLOCK), 0, E->stream, p, n, out);
    launch_end(E, K_PACK_STATE);
}

void run_unpack_state(Engine* E, const DevParticles& p, int n, const float4* in)
{
    if (n <= 0)
        return;
    launch_begin(E, K_UNPACK_STATE);
    hipLaunchKernelGGL(k_unpack_state, dim3(div_up(n, BLOCK)), dim3(BLOCK), 0, E->stream, p, n, in);
    launch_end(E, K_UNPACK_STATE);
}

void run_pack_grid(Engine* E, const Vehicle* v)
{
    launch_begin(E, K_PACK_GRID);
    hipLaunchKernelGGL(k_pack_grid, dim3(div_up(v->C, BLOCK)), dim3(BLOCK), 0, E->stream, v->grid, v->aos_tmp, v->C);
    launch_end(E, K_PACK_GRID);
}

void run_unpack_grid(Engine* E, const Vehicle* v)
{
    launch_begin(E, K_UNPACK_GRID);
    hipLaunchKernelGGL(k_unpack_grid, dim3(div_up(v->C, BLOCK)), dim3(BLOCK), 0, E->stream, v->grid, v->aos_tmp,
                       v->C);
    launch_end(E, K_UNPACK_GRID);
}

}  // namespace dogm_hip
