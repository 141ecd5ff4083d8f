// Which form a call of the measurement-grid generator takes, by its sizes and ranges (host code only).
#pragma once

#include <cstddef>
#include <cstdint>

namespace dogm_hip
{

enum LidarForm
{
    LIDAR_LAUNCHES = 0,     // clear, free and occ launches over the grids
    LIDAR_TILES_GRIDS = 1,  // one launch of square tiles of cells, grid after grid
    LIDAR_TILES_CENTRE = 2, // the same, the tiles around the sensor of every grid first
};

// Measured over sides 64 to 4100, 256 to 1400 MB of cells, 180 to 4096 beams, ranges from blocked (2 to 10% of the side)
// to full (us: launches / tiles grid after grid / tiles centre first; ranges of 5 to 50% of the side if not said):
//  * The grids exceed the last-level cache (256 MB).  Below, the second write of the launches finds the cells there:
//    4 x 1200 x 1200 cells, 1080 beams 75 / 117.
//  * On sides below 192 every tile is near the sensor and walks most beams, which pays where the launches take many
//    samples for nothing: max_range of 0.4 of the side for one tile or few beams, of the whole side otherwise (1088 x
//    128, 1440 beams 1135 / 1325 / 1295, max_range of 3 sides 3622 / 1606 / 1600; 180 beams 312 / 262 / 256).
//  * A workgroup around the sensor walks every beam, 45 + 0.07 us per beam, which the rest of the call has to cover
//    (12.5 cells per beam and cell of the side, at most 23000 per beam; fewer where max_range is beyond the grid and
//    the launches take more samples): 1 x 4100, 1440 beams 88 / 142 / 128; 2 x 4100 201 / 192 / 143; 12 x 1200, 1440
//    beams, blocked 118 / 177 / 138, max_range of 3 sides 406 / 211 / 147; 22 x 900, 1440 beams 219 / 224 / 146.
//  * The beams cross 1.5% as many cells as there are.  The launches clear faster than the tiles write, and with few cells
//    to mark that is all: 113 x 900, 180 beams, blocked 354 / 406 / 401; 64 x 1200, 180 beams 411 / 296 / 302.
//    At most 4096 to 8191 ranges are looked at, so that this takes the host no time to speak of.
//  * Centre first hides those workgroups behind the others, grid after grid mixes them with writing ones and writes
//    neighbouring lines together, which wins once they are many (1.25 MB per beam): 25 x 1200, 720 beams 249 / 172 /
//    149; 113 x 900, 720 beams 674 / 383 / 438.
inline LidarForm lidar_form(int gs, double resolution, double max_range, int beams, int count, const double* ranges)
{
    const double cells = (double)gs * (double)gs * (double)count, bytes = 16.0 * cells;
    if (bytes <= 256.0 * 1048576.0)
        return LIDAR_LAUNCHES;
    const double most = max_range / (gs * resolution);
    if (gs < 192 && !(most >= (gs <= 64 || beams <= 3 * gs ? 0.4 : 1.0)))
        return LIDAR_LAUNCHES;
    if (cells * (most > 0.5 ? 2.0 * most : 1.0) < beams * (12.5 * gs < 23000.0 ? 12.5 * gs : 23000.0))
        return LIDAR_LAUNCHES;
    const size_t n = (size_t)count * (size_t)beams, step = n < 4096 ? 1 : n / 4096;
    double reach = 0.0;
    for (size_t i = 0; i < n; i += step)
    {
        const double r = ranges[i];
        reach += r > 0.0 ? (r < max_range ? r : max_range) : 0.0;
    }
    if (!((double)step * reach >= 0.015 * cells * resolution))
        return LIDAR_LAUNCHES;
    return bytes >= 1.25 * 1048576.0 * beams ? LIDAR_TILES_GRIDS : LIDAR_TILES_CENTRE;
}

}  // namespace dogm_hip
