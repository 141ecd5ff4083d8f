// Measurement-grid generation on gfx950: the step before updateGrid.
//
// The reference turns a lidar scan into a measurement grid on the GPU through a polar inverse-sensor
// texture rendered into a Cartesian framebuffer with OpenGL (dogm/demo/simulator/mapping/
// laser_to_meas_grid.cu:25-70, kernel/measurement_grid.cu:46-132).  This generator ray-casts each
// beam straight into the Cartesian grid with a two-level inverse sensor model:
//   - every cell a beam samples (half-cell steps from the sensor, strictly before the return or
//     max_range) gets free mass `free_mass`;
//   - the cell of each return gets occupied mass `occ_mass` and no free mass;
//   - all other cells are unknown (0, 0); likelihood = p_A = 1 (measurement_grid.cu:129-130).
// The sensor sits at the grid centre; index = x + grid_size * y.  Positions are computed in f64 with
// one fixed operation order (centre + dir * dist, then / resolution, then floor), so the grid is a
// pure function of the ranges and the beam directions.
//
// Large calls take one launch (blockIdx.y = grid), a workgroup per square tile of cells: the beams that can cross the tile
// are found, their samples inside it marked in LDS, and every cell is then written once.
// Calls that this does not suit (lidar_form) take three launches, each over every grid of the call:
//   clear  16-byte stores of (0, 0, 1, 1) over the cells;
//   free   one thread per (beam, step) sample: an idempotent 4-byte store of free_mass;
//   occ    one thread per beam: occ_mass and free 0 at the return's cell (after every free store).
#include "dogm_internal.h"
#include "dogm_lidar_form.h"

#include <algorithm>
#include <cmath>
#include <cstring>
#include <memory>
#include <new>
#include <string>
#include <vector>

struct dogm_lidar
{
    dogm_lidar_params p{};
    int steps = 0;          // samples per beam
    double step = 0.0;      // sample spacing [m]
    double centre = 0.0;    // sensor position in grid metres (both axes)
    hipStream_t stream = nullptr;
    double* d_dir = nullptr;       // [4 * beams]: cos, sin, 1 / cos, 1 / sin
    double* d_ranges = nullptr;    // [cap * beams]
    double* h_ranges = nullptr;    // pinned staging
    dogm_measurement_cell** d_out = nullptr;  // [cap]
    dogm_measurement_cell** h_out = nullptr;  // pinned staging
    int cap = 0;
    std::string last_error;
};

namespace dogm_hip
{

struct LidarArgs
{
    int gs;
    int beams;
    int steps;
    double res;
    double step;
    double centre;
    double max_range;
    double inv_res;
    double inv_step;
    float occ_mass;
    float free_mass;
};

__global__ __launch_bounds__(BLOCK) void k_lidar_clear(dogm_measurement_cell* const* __restrict__ outs, int cells)
{
    const int c = blockIdx.x * BLOCK + threadIdx.x;
    if (c >= cells)
        return;
    *reinterpret_cast<float4*>(outs[blockIdx.y] + c) = make_float4(0.0f, 0.0f, 1.0f, 1.0f);
}

// End of the free samples: min(range, max_range); a NaN range has no free samples.
__device__ __forceinline__ double lidar_limit(double r, double max_range)
{
    return (r < max_range || r != r) ? r : max_range;
}

// floor(x / res).  The product with the rounded reciprocal is within 3 * 2^-53 of the quotient, relatively, so both
// lie between the same two integers unless one is nearer than that; the division is left to those.
__device__ __forceinline__ double cell_floor(double x, const LidarArgs& a)
{
    const double q = x * a.inv_res;
    if (fabs(q - rint(q)) > 0x1p-50 * fabs(q))
        return floor(q);
    return floor(x / a.res);
}

__global__ __launch_bounds__(BLOCK) void k_lidar_free(dogm_measurement_cell* const* __restrict__ outs,
                                                      const double* __restrict__ ranges,
                                                      const double* __restrict__ dir, LidarArgs a)
{
    const long long t = (long long)blockIdx.x * BLOCK + threadIdx.x;
    const long long n = (long long)a.beams * a.steps;
    if (t >= n)
        return;
    const int b = (int)(t / a.steps);
    const int k = (int)(t - (long long)b * a.steps);
    const double lim = lidar_limit(ranges[(size_t)blockIdx.y * a.beams + b], a.max_range);
    const double dist = (double)k * a.step;
    if (!(dist < lim))
        return;
    const double xs = a.centre + dir[b] * dist;
    const double ys = a.centre + dir[a.beams + b] * dist;
    const double fx = floor(xs / a.res), fy = floor(ys / a.res);
    if (!(fx >= 0.0 && fx < (double)a.gs && fy >= 0.0 && fy < (double)a.gs))
        return;
    const int c = (int)fx + a.gs * (int)fy;
    outs[blockIdx.y][c].free_mass = a.free_mass;
}

__global__ __launch_bounds__(BLOCK) void k_lidar_occ(dogm_measurement_cell* const* __restrict__ outs,
                                                     const double* __restrict__ ranges,
                                                     const double* __restrict__ dir, LidarArgs a)
{
    const int b = blockIdx.x * BLOCK + threadIdx.x;
    if (b >= a.beams)
        return;
    const double r = ranges[(size_t)blockIdx.y * a.beams + b];
    if (!(r <= a.max_range))
        return;  // no return within range (inf, NaN or beyond max_range)
    const double fx = floor((a.centre + dir[b] * r) / a.res);
    const double fy = floor((a.centre + dir[a.beams + b] * r) / a.res);
    if (!(fx >= 0.0 && fx < (double)a.gs && fy >= 0.0 && fy < (double)a.gs))
        return;
    const int c = (int)fx + a.gs * (int)fy;
    *reinterpret_cast<float2*>(&outs[blockIdx.y][c].free_mass) = make_float2(0.0f, a.occ_mass);
}

// One tile of T x T cells of one grid.  Each round of THREADS beams: a thread clips its beam against the tile (with
// half a cell and one sample of margin, far above rounding, so nothing is lost) and queues the samples that are
// left, and its return; then the waves take the queued beams in turn, a lane per sample.  The samples' positions
// and cells are computed as in k_lidar_free; marks are plain byte stores, free and occupied apart, so
// their order does not matter.
// Writes the grids once, where the three launches write every cell and then 4-byte pieces of most cache lines again.
// Side 64 and 512 threads: 32 x 1200 x 1200 cells (737 MB) from 1080 beams 262 us, side 32 384, side 16 1118, 1024
// threads 292 (three launches 464).  The tiles around the sensor walk every beam: a call of these grids from scans
// of a scene takes 194 us with them first and 238 grid after grid, where the last grid's are still at it when all
// is written (three launches 413).
constexpr int LIDAR_TILE = 64;
constexpr int LIDAR_THREADS = 512;

__global__ __launch_bounds__(LIDAR_THREADS) void k_lidar_tiles(dogm_measurement_cell* const* __restrict__ outs,
                                                               const double* __restrict__ ranges,
                                                               const double* __restrict__ dir, LidarArgs a,
                                                               int side, int count, int centre_first)
{
    constexpr int T = LIDAR_TILE, THREADS = LIDAR_THREADS;
    __shared__ __attribute__((aligned(16))) uint8_t s_free[T * T];
    __shared__ __attribute__((aligned(16))) uint8_t s_occ[T * T];
    __shared__ double s_dx[THREADS], s_dy[THREADS], s_lim[THREADS];
    __shared__ int2 s_k[THREADS];
    __shared__ int s_n;
    const int lane = threadIdx.x & (WAVE - 1), wid = threadIdx.x / WAVE;
    const int id = (int)blockIdx.x;
    int grid, tx, ty;
    if (centre_first)
    {
        // Rows and columns of tiles outwards from the sensor's, all grids at each.
        const int rank = id / count, mid = a.gs / 2 / T;
        const auto outwards = [=](int r) { return (mid + ((r & 1) ? (r + 1) / 2 : side - r / 2)) % side; };
        grid = id % count;
        tx = outwards(rank % side);
        ty = outwards(rank / side);
    }
    else
    {
        // Workgroups go to the 8 XCDs in turn.  An odd count along both sides spreads the busy middle tiles of every row
        // and grid over them; at a multiple of 8 they fall to two (24 x 1024 x 1024 cells 348 us, 219 with the odd
        // counts).
        const int stride = side | 1, t = id % (stride * stride);
        grid = id / (stride * stride);
        tx = t % stride;
        ty = t / stride;
        if (tx >= side || ty >= side)
            return;
    }
    const int x0 = tx * T, y0 = ty * T;
    for (int i = threadIdx.x; i < T * T / 4; i += THREADS)
    {
        reinterpret_cast<uint32_t*>(s_free)[i] = 0u;
        reinterpret_cast<uint32_t*>(s_occ)[i] = 0u;
    }
    // The tile's sides as seen from the sensor, half a cell outside.
    const double xa = ((double)x0 - 0.5) * a.res - a.centre, xb = ((double)(x0 + T) + 0.5) * a.res - a.centre;
    const double ya = ((double)y0 - 0.5) * a.res - a.centre, yb = ((double)(y0 + T) + 0.5) * a.res - a.centre;
    const double w = (double)min(T, a.gs - x0), h = (double)min(T, a.gs - y0);
    const auto mark = [&](uint8_t* map, double dx, double dy, double dist) {
        const double fx = cell_floor(a.centre + dx * dist, a) - (double)x0;
        const double fy = cell_floor(a.centre + dy * dist, a) - (double)y0;
        if (fx >= 0.0 && fx < w && fy >= 0.0 && fy < h)
            map[(int)fy * T + (int)fx] = 1;
    };
    for (int b0 = 0; b0 < a.beams; b0 += THREADS)
    {
        if (threadIdx.x == 0)
            s_n = 0;
        __syncthreads();
        const int b = b0 + threadIdx.x;
        if (b < a.beams)
        {
            const double dx = dir[b], dy = dir[a.beams + b];
            const double ix = dir[2 * (size_t)a.beams + b], iy = dir[3 * (size_t)a.beams + b];
            const double r = ranges[(size_t)grid * a.beams + b];
            const double lim = lidar_limit(r, a.max_range);
            // Distances at which the beam is inside (a direction of 0 gives infinite ones, empty if outside).
            const double xl = xa * ix, xh = xb * ix, yl = ya * iy, yh = yb * iy;
            const double lo = fmax(fmin(xl, xh), fmin(yl, yh)), hi = fmin(fmax(xl, xh), fmax(yl, yh));
            const double k_lo = fmax(floor(lo * a.inv_step) - 1.0, 0.0);
            const double k_hi = fmin(ceil(fmin(hi, lim) * a.inv_step) + 1.0, (double)(a.steps - 1));
            if (lim > 0.0 && k_lo <= k_hi)
            {
                const int j = atomicAdd(&s_n, 1);
                s_dx[j] = dx;
                s_dy[j] = dy;
                s_lim[j] = lim;
                s_k[j] = make_int2((int)k_lo, (int)k_hi);
            }
            // Negated so that directions that are not numbers are looked at too.
            if (r <= a.max_range && !(r + a.step < lo) && !(r - a.step > hi))
                mark(s_occ, dx, dy, r);
        }
        __syncthreads();
        const int jobs = s_n;
        for (int j = wid; j < jobs; j += THREADS / WAVE)
        {
            const double dx = s_dx[j], dy = s_dy[j], lim = s_lim[j];
            const int2 range = s_k[j];
            for (int k = range.x + lane; k <= range.y; k += WAVE)
            {
                const double dist = (double)k * a.step;
                if (dist < lim)
                    mark(s_free, dx, dy, dist);
            }
        }
        __syncthreads();
    }
    dogm_measurement_cell* out = outs[grid];
    for (int i = threadIdx.x; i < T * T; i += THREADS)
    {
        const int x = i % T, y = i / T;
        if (x0 + x >= a.gs || y0 + y >= a.gs)
            continue;
        const bool occ = s_occ[i] != 0;
        const float f = !occ && s_free[i] ? a.free_mass : 0.0f;
        *reinterpret_cast<float4*>(out + (x0 + x) + (size_t)a.gs * (y0 + y)) =
            make_float4(f, occ ? a.occ_mass : 0.0f, 1.0f, 1.0f);
    }
}

int lidar_grid_size(const dogm_lidar* l)
{
    return l->p.grid_size;
}

int lidar_beam_count(const dogm_lidar* l)
{
    return l->p.beam_count;
}

}  // namespace dogm_hip

using namespace dogm_hip;

namespace
{

int lfail(dogm_lidar* l, int code, const std::string& msg)
{
    if (l)
        l->last_error = msg;
    return code;
}

void lidar_release(dogm_lidar* l)
{
    if (l->stream)
        (void)hipStreamSynchronize(l->stream);
    (void)hipFree(l->d_dir);
    (void)hipFree(l->d_ranges);
    (void)hipFree(l->d_out);
    if (l->h_ranges)
        (void)hipHostFree(l->h_ranges);
    if (l->h_out)
        (void)hipHostFree(l->h_out);
    if (l->stream)
        (void)hipStreamDestroy(l->stream);
}

int lidar_reserve(dogm_lidar* l, int count)
{
    if (count <= l->cap)
        return DOGM_OK;
    const int cap = std::max(count, 2 * l->cap);
    (void)hipStreamSynchronize(l->stream);
    (void)hipFree(l->d_ranges);
    (void)hipFree(l->d_out);
    if (l->h_ranges)
        (void)hipHostFree(l->h_ranges);
    if (l->h_out)
        (void)hipHostFree(l->h_out);
    l->d_ranges = nullptr;
    l->d_out = nullptr;
    l->h_ranges = nullptr;
    l->h_out = nullptr;
    l->cap = 0;
    const size_t nr = (size_t)cap * (size_t)l->p.beam_count;
    if (hipMalloc(reinterpret_cast<void**>(&l->d_ranges), sizeof(double) * nr) != hipSuccess ||
        hipMalloc(reinterpret_cast<void**>(&l->d_out), sizeof(void*) * (size_t)cap) != hipSuccess ||
        hipHostMalloc(reinterpret_cast<void**>(&l->h_ranges), sizeof(double) * nr) != hipSuccess ||
        hipHostMalloc(reinterpret_cast<void**>(&l->h_out), sizeof(void*) * (size_t)cap) != hipSuccess)
        return lfail(l, DOGM_ERR_OUT_OF_MEMORY, "allocating lidar staging buffers");
    l->cap = cap;
    return DOGM_OK;
}

// The form of a call (lidar_form); the launches also where two grids overlap (a cell may then get marks of several
// scans) and where the resolution does not leave the tiles' clipping margins far above rounding.
LidarForm lidar_call_form(const dogm_lidar* l, int count, const double* ranges, dogm_measurement_cell* const* outs)
{
    const LidarForm form =
        lidar_form(l->p.grid_size, l->p.resolution, l->p.max_range, l->p.beam_count, count, ranges);
    if (form == LIDAR_LAUNCHES || !(l->p.resolution > 1e-100 && l->p.resolution < 1e100))
        return LIDAR_LAUNCHES;
    const uintptr_t bytes = sizeof(dogm_measurement_cell) * (uintptr_t)l->p.grid_size * (uintptr_t)l->p.grid_size;
    const std::unique_ptr<uintptr_t[]> at(new (std::nothrow) uintptr_t[count]);
    if (!at)
        return LIDAR_LAUNCHES;
    for (int i = 0; i < count; ++i)
        at[i] = reinterpret_cast<uintptr_t>(outs[i]);
    std::sort(at.get(), at.get() + count);
    for (int i = 1; i < count; ++i)
        if (at[i] - at[i - 1] < bytes)
            return LIDAR_LAUNCHES;
    return form;
}

}  // namespace

extern "C" {

int dogm_lidar_create(const dogm_lidar_params* p, const double* beam_cos, const double* beam_sin, dogm_lidar** out)
{
    if (!p || !out)
        return DOGM_ERR_INVALID_ARGUMENT;
    *out = nullptr;
    if (p->grid_size < 1 || p->grid_size > 46340 || p->beam_count < 1 || !(p->resolution > 0.0) ||
        !(p->max_range > 0.0) || !std::isfinite(p->max_range) || !std::isfinite(p->resolution))
        return DOGM_ERR_INVALID_ARGUMENT;
    if ((beam_cos == nullptr) != (beam_sin == nullptr))
        return DOGM_ERR_INVALID_ARGUMENT;
    dogm_lidar* l = new (std::nothrow) dogm_lidar();
    if (!l)
        return DOGM_ERR_OUT_OF_MEMORY;
    l->p = *p;
    l->step = 0.5 * p->resolution;
    l->steps = (int)std::ceil(p->max_range / l->step) + 1;
    l->centre = 0.5 * p->grid_size * p->resolution;
    if ((long long)l->steps * p->beam_count > (long long)INT32_MAX * 64)
    {
        delete l;
        return DOGM_ERR_INVALID_ARGUMENT;
    }
    std::vector<double> dir(4 * (size_t)p->beam_count);
    for (int b = 0; b < p->beam_count; ++b)
    {
        if (beam_cos)
        {
            dir[b] = beam_cos[b];
            dir[p->beam_count + b] = beam_sin[b];
        }
        else
        {
            // 360 degrees, beam b at 2 pi b / beam_count.
            const double ang = 2.0 * M_PI * (double)b / (double)p->beam_count;
            dir[b] = std::cos(ang);
            dir[p->beam_count + b] = std::sin(ang);
        }
    }
    for (size_t i = 0; i < 2 * (size_t)p->beam_count; ++i)
        dir[2 * (size_t)p->beam_count + i] = 1.0 / dir[i];
    int st = DOGM_OK;
    if (hipStreamCreateWithFlags(&l->stream, hipStreamNonBlocking) != hipSuccess)
        st = DOGM_ERR_HIP;
    else if (hipMalloc(reinterpret_cast<void**>(&l->d_dir), sizeof(double) * dir.size()) != hipSuccess)
        st = DOGM_ERR_OUT_OF_MEMORY;
    else if (hipMemcpy(l->d_dir, dir.data(), sizeof(double) * dir.size(), hipMemcpyHostToDevice) != hipSuccess)
        st = DOGM_ERR_HIP;
    else
        st = lidar_reserve(l, 1);
    if (st != DOGM_OK)
    {
        lidar_release(l);
        delete l;
        return st;
    }
    *out = l;
    return DOGM_OK;
}

void dogm_lidar_destroy(dogm_lidar* l)
{
    if (!l)
        return;
    lidar_release(l);
    delete l;
}

const char* dogm_lidar_last_error(const dogm_lidar* l)
{
    return l ? l->last_error.c_str() : "null lidar";
}

int dogm_lidar_generate_many(dogm_lidar* l, int count, const double* ranges, dogm_measurement_cell* const* device_out)
{
    if (!l)
        return DOGM_ERR_INVALID_ARGUMENT;
    if (count < 1 || count > 65535 || !ranges || !device_out)
        return lfail(l, DOGM_ERR_INVALID_ARGUMENT, "count must be in [1, 65535] with ranges and outputs");
    for (int i = 0; i < count; ++i)
        if (!device_out[i])
            return lfail(l, DOGM_ERR_INVALID_ARGUMENT, "output grid " + std::to_string(i) + " is null");
    int st = lidar_reserve(l, count);
    if (st != DOGM_OK)
        return st;
    const int beams = l->p.beam_count;
    const int gs = l->p.grid_size;
    std::memcpy(l->h_ranges, ranges, sizeof(double) * (size_t)count * beams);
    std::memcpy(l->h_out, device_out, sizeof(void*) * (size_t)count);
    if (hipMemcpyAsync(l->d_ranges, l->h_ranges, sizeof(double) * (size_t)count * beams, hipMemcpyHostToDevice,
                       l->stream) != hipSuccess ||
        hipMemcpyAsync(l->d_out, l->h_out, sizeof(void*) * (size_t)count, hipMemcpyHostToDevice, l->stream) !=
            hipSuccess)
        return lfail(l, DOGM_ERR_HIP, "uploading ranges");
    const LidarArgs a{gs,           beams,
                      l->steps,     l->p.resolution,
                      l->step,      l->centre,
                      l->p.max_range, 1.0 / l->p.resolution,
                      1.0 / l->step, l->p.occ_mass,
                      l->p.free_mass};
    const int cells = gs * gs;
    const LidarForm form = lidar_call_form(l, count, ranges, device_out);
    if (form != LIDAR_LAUNCHES)
    {
        const int side = div_up(gs, LIDAR_TILE), centre_first = form == LIDAR_TILES_CENTRE;
        const int stride = centre_first ? side : side | 1;
        hipLaunchKernelGGL(k_lidar_tiles, dim3(stride * stride * count), dim3(LIDAR_THREADS), 0, l->stream, l->d_out,
                           l->d_ranges, l->d_dir, a, side, count, centre_first);
    }
    else
    {
        const long long samples = (long long)beams * l->steps;
        hipLaunchKernelGGL(k_lidar_clear, dim3(div_up(cells, BLOCK), count), dim3(BLOCK), 0, l->stream, l->d_out, cells);
        hipLaunchKernelGGL(k_lidar_free, dim3(div_up(samples, BLOCK), count), dim3(BLOCK), 0, l->stream, l->d_out,
                           l->d_ranges, l->d_dir, a);
        hipLaunchKernelGGL(k_lidar_occ, dim3(div_up(beams, BLOCK), count), dim3(BLOCK), 0, l->stream, l->d_out,
                           l->d_ranges, l->d_dir, a);
    }
    hipError_t e = hipGetLastError();
    if (e == hipSuccess)
        e = hipStreamSynchronize(l->stream);
    if (e != hipSuccess)
        return lfail(l, DOGM_ERR_HIP, std::string("generating measurement grids: ") + hipGetErrorString(e));
    return DOGM_OK;
}

int dogm_lidar_generate(dogm_lidar* l, const double* ranges, dogm_measurement_cell* device_out)
{
    dogm_measurement_cell* outs[1] = {device_out};
    return dogm_lidar_generate_many(l, 1, ranges, outs);
}

}  // extern "C"
