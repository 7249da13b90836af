// Projection-guided window search for gfx950.
//
//   k_grid_build   Object::AssignFeaturesToGrid / PosInGrid (src/Object.cpp:
//                  182-201, :249-257): 30 x 30 cells, cell = round(x * 30/cols),
//                  keypoints outside [0,30) dropped, in-cell order = index.
//   k_window_knn   Object::ProjectBunchMapPoints (:208-236) per map point:
//                  R*Pw + t, z < 0 skip, pinhole project, GetFeaturesInArea
//                  (:263-308) in ix-major / iy / in-cell order, top-2 Hamming
//                  in that candidate order, FilterRatio + FilterThreshold.
//                  With direct positions instead of map points it is the
//                  query of Tracker::Wnd_Track (src/Tracker.cpp:339-353):
//                  GetFeaturesInArea(kp.pt, r, minLevel, maxLevel) then the
//                  same top-2 and filters.
// Included by mcv_api.hip.
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace mcv {

constexpr int kGrid = 30;
constexpr int kGridCells = kGrid * kGrid;
constexpr int kGridSortCap = 16384;

struct GridView {
    const float* kxy;       // n x 2
    const int32_t* koct;    // n octaves (read only by a level-filtered query)
    const uint8_t* kdesc;   // n x 32
    int n;
    int width, height;
    float inv_w, inv_h;     // (float)(30.0 / cols), (float)(30.0 / rows)
    int* cell_start;        // 901 entries
    int* cell_items;        // n entries (keypoint indices grouped by cell)
    float2* cell_xy;        // their positions
};

struct WindowCam {
    GridView grid;
    float R[9], t[3];
    float fx, fy, cx, cy;
    int32_t* out;           // n_points x 6
};

// the cameras of one launch, as kernel arguments
constexpr int kWindowCams = 8;
struct WindowCams {
    WindowCam c[kWindowCams];
};

// A stable counting sort by cell, one workgroup per camera: the keypoints are
// cut into one contiguous run per wave, each wave counts its run's cells
// (LDS), the counts are scanned over (cell, wave), and each wave places its
// run 64 keypoints at a time, the lanes of one cell ranked by ballots of the
// cell's bits.  Latency bound (one workgroup per camera, two trips to memory);
// a bitonic sort of (cell, index) with a one-thread scan took 75 us for 3
// cameras of 2000 keypoints.
__global__ __launch_bounds__(1024) void k_grid_build(WindowCams cams) {
    constexpr int kWaves = 16, kIter = kGridSortCap / 1024;
    __shared__ int s_cnt[kWaves][kGridCells];
    __shared__ int s_base[kGridCells];
    __shared__ int s_sum[kWaves];
    const GridView& G = cams.c[blockIdx.x].grid;
    const int n = G.n;
    const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int run = (n + 1023) / 1024 * 64;  // keypoints per wave: at most kIter * 64
    const int i0 = wv * run;
    for (int c = threadIdx.x; c < kWaves * kGridCells; c += 1024) s_cnt[0][c] = 0;
    float2 xy[kIter];
    int cell[kIter];
#pragma unroll
    for (int u = 0; u < kIter; u++) {
        const int i = i0 + 64 * u + lane;
        cell[u] = -1;
        if (64 * u < run && i < n) {
            const float x = G.kxy[2 * i], y = G.kxy[2 * i + 1];
            const int px = (int)roundf((x - 0.f) * G.inv_w);
            const int py = (int)roundf((y - 0.f) * G.inv_h);
            if (px >= 0 && px < kGrid && py >= 0 && py < kGrid) cell[u] = px * kGrid + py;
            xy[u] = make_float2(x, y);
        }
    }
    __syncthreads();
#pragma unroll
    for (int u = 0; u < kIter; u++)
        if (cell[u] >= 0) atomicAdd(&s_cnt[wv][cell[u]], 1);
    __syncthreads();
    {
        int sum = 0;
        if (threadIdx.x < kGridCells)
            for (int w = 0; w < kWaves; w++) {
                const int k = s_cnt[w][threadIdx.x];
                s_cnt[w][threadIdx.x] = sum;
                sum += k;
            }
        int incl = sum;
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
            const int y = __shfl_up(incl, o, 64);
            if (lane >= o) incl += y;
        }
        if (lane == 63) s_sum[wv] = incl;
        __syncthreads();
        int start = incl - sum;
        for (int w = 0; w < wv; w++) start += s_sum[w];
        // thread kGridCells, past the last cell: the total
        if (threadIdx.x <= kGridCells) G.cell_start[threadIdx.x] = start;
        if (threadIdx.x < kGridCells) s_base[threadIdx.x] = start;
    }
    __syncthreads();
#pragma unroll
    for (int u = 0; u < kIter; u++) {
        if (64 * u >= run) continue;  // wave-uniform
        const int c = cell[u];
        unsigned long long m = __ballot(c >= 0);
#pragma unroll
        for (int b = 0; b < 10; b++) {
            const unsigned long long on = __ballot((c >> b) & 1);
            m &= ((c >> b) & 1) ? on : ~on;
        }
        if (c >= 0) {
            const int rank = __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0));
            const int done = s_cnt[wv][c];
            // one wave's DS instructions run in order: the reads, then the first lanes' writes
            asm volatile("" ::: "memory");
            if (rank == 0) s_cnt[wv][c] = done + __builtin_popcountll(m);
            asm volatile("" ::: "memory");
            const int pos = s_base[c] + done + rank;
            G.cell_items[pos] = i0 + 64 * u + lane;
            G.cell_xy[pos] = xy[u];
        }
    }
}

struct WindowPoints {
    const float* pts;       // P x 3 map points, or null for direct positions
    const float* uv;        // P x 2 query positions (when pts is null)
    const uint8_t* pdesc;   // P x 32
    const int32_t* plevel;  // P (map points only)
    int P;
    float radius, ratio;
    int th;
    int nl;                 // scale-table entries (map points only)
    int min_level, max_level;  // GetFeaturesInArea's level filter (direct positions only)
    float scales[16];
};

// kLanes lanes per (camera, query).  The grid's items are ordered by (column of
// cells, row, keypoint), the order candidates are visited in, so the window is
// one run of items per column and an item's place in the grid orders it among
// the candidates; the lanes take the items of all columns together.  Output
// row: (kp0, d0, kp1, d1, n_candidates, match); a map point whose level is
// outside [0, nl) gets n_candidates = -1 and no match (the reference indexes
// mvScaleFactor with it).  Bound by the chain cell ranges -> positions ->
// descriptors of a query.  A wave per query that walked the cells one by one
// took 67 us for 3 cameras of 5000 queries and 2000 keypoints.
//
// Lanes by the queries of a launch: few queries leave lanes idle, so a query
// takes more of them, which shortens its walk over many candidates; from some
// ten thousand on they are better spent on queries.  us of a search, 16 / 32 / 64
// lanes: 1000 queries, 8000 keypoints in a twelfth of the image each way, radius
// 100: 489 / - / 137; 5000 so 488 / 250 / 158, 15000 512 / 362 / 402; 2000
// keypoints over the image, radius 400: 5000 queries 117 / 86 / 61, 10000 122 /
// 112 / 98, 15000 137 / 163 / 123; radius 15: 8000 queries 14.8 / 14.8 / 17.1,
// 20000 14.8 / 15.8 / 19.7.
constexpr int window_lanes(long long queries) { return queries <= 4096 ? 64 : queries <= 10240 ? 32 : 16; }

template <int kLanes>
__global__ __launch_bounds__(256) void k_window_knn(WindowCams cams, WindowPoints W) {
    const int lane = threadIdx.x % kLanes;
    const int p = blockIdx.x * (256 / kLanes) + threadIdx.x / kLanes;
    if (p >= W.P) return;
    const WindowCam& C = cams.c[blockIdx.y];
    const GridView& G = C.grid;
    int32_t* o = C.out + 6 * (long long)p;
    float u = 0.f, v = 0.f, r = 0.f;
    bool valid;
    if (W.pts) {
        // Pc = R * Pw + t: cv::Mat float gemm, products and sums in double,
        // one rounding to float per row
        const float* pw = W.pts + 3 * p;
        float Pc[3];
#pragma unroll
        for (int k = 0; k < 3; k++) {
            double s = 0.0;
            s += (double)C.R[3 * k] * (double)pw[0];
            s += (double)C.R[3 * k + 1] * (double)pw[1];
            s += (double)C.R[3 * k + 2] * (double)pw[2];
            Pc[k] = (float)(s + (double)C.t[k]);
        }
        const int lvl = W.plevel[p];
        if (lvl < 0 || lvl >= W.nl) {
            if (lane == 0) {
                o[0] = -1; o[1] = 999; o[2] = -1; o[3] = 999; o[4] = -1; o[5] = -1;
            }
            return;
        }
        valid = !(Pc[2] < 0.f);
        if (valid) {
            u = C.fx * Pc[0] / Pc[2] + C.cx;
            v = C.fy * Pc[1] / Pc[2] + C.cy;
            r = W.radius * W.scales[lvl];
        }
    } else {
        u = W.uv[2 * p];
        v = W.uv[2 * p + 1];
        r = W.radius;
        valid = true;
    }
    const bool check_levels = W.pts == nullptr && (W.min_level > 0 || W.max_level >= 0);
    uint32_t k0 = 999u << 22, k1 = 999u << 22;
    int ncand = 0;
    int nMinX = 0, nMaxX = -1, nMinY = 0, nMaxY = -1;
    if (valid && !(u != u || v != v) && !(u < 0 || v < 0 || u >= (float)G.width || v >= (float)G.height)) {
        nMinX = max(0, (int)floorf((u - 0.f - r) * G.inv_w));
        nMaxX = min(kGrid - 1, (int)ceilf((u - 0.f + r) * G.inv_w));
        nMinY = max(0, (int)floorf((v - 0.f - r) * G.inv_h));
        nMaxY = min(kGrid - 1, (int)ceilf((v - 0.f + r) * G.inv_h));
        if (!(nMinX < kGrid && nMaxX >= 0 && nMinY < kGrid && nMaxY >= 0)) nMaxX = -1;
    }
    if (nMaxX >= nMinX && nMaxY >= nMinY) {
        // 32 bytes at any 4-byte alignment
        typedef uint32_t __attribute__((ext_vector_type(4), aligned(4))) u32x4;
        const u32x4* qd = reinterpret_cast<const u32x4*>(W.pdesc + 32 * (long long)p);
        const u32x4 qa = qd[0], qb = qd[1];
        const int ncols = nMaxX - nMinX + 1;
        for (int j0 = 0; j0 < ncols; j0 += kLanes) {
            // lane j: column j0 + j's run of items
            const int nc = min(kLanes, ncols - j0);
            int a = 0, len = 0;
            if (lane < nc) {
                const int* cs = G.cell_start + (nMinX + j0 + lane) * kGrid;
                a = cs[nMinY];
                len = cs[nMaxY + 1] - a;
            }
            int incl = len;
#pragma unroll
            for (int s = 1; s < kLanes; s <<= 1) {
                const int y = __shfl_up(incl, s, kLanes);
                if (lane >= s) incl += y;
            }
            const int total = __shfl(incl, kLanes - 1, kLanes);
            const int first = incl - len;  // items of the columns before
            for (int t0 = 0; t0 < total; t0 += kLanes) {
                const int t = t0 + lane;
                int s = 0;
                for (int j = 0; j < nc; j++) {
                    const int fj = __shfl(first, j, kLanes), aj = __shfl(a, j, kLanes);
                    if (t >= fj) s = aj + (t - fj);
                }
                if (t >= total) continue;
                const int idx = G.cell_items[s];
                const float2 xy = G.cell_xy[s];
                const float dx = xy.x - u, dy = xy.y - v;
                bool in = fabsf(dx) < r && fabsf(dy) < r;
                if (check_levels) {
                    const int oct = G.koct[idx];
                    if (oct < W.min_level || (W.max_level >= 0 && oct > W.max_level)) in = false;
                }
                if (in) {
                    const u32x4* kd = reinterpret_cast<const u32x4*>(G.kdesc + 32 * (long long)idx);
                    const u32x4 ka = kd[0] ^ qa, kb = kd[1] ^ qb;
                    uint32_t d = 0;
#pragma unroll
                    for (int k = 0; k < 4; k++) d += __builtin_popcount(ka[k]) + __builtin_popcount(kb[k]);
                    const uint32_t key = (d << 22) | (uint32_t)s;
                    k1 = min(k1, max(k0, key));
                    k0 = min(k0, key);
                    ncand++;
                }
            }
        }
    }
    // merge the lanes' top-2 keys and candidate counts
#pragma unroll
    for (int off = kLanes / 2; off > 0; off >>= 1) {
        const uint32_t b0 = __shfl_xor(k0, off, kLanes), b1 = __shfl_xor(k1, off, kLanes);
        const uint32_t n1 = min(max(k0, b0), min(k1, b1));
        k0 = min(k0, b0);
        k1 = n1;
        ncand += __shfl_xor(ncand, off, kLanes);
    }
    if (lane != 0) return;
    auto kp_of = [&](uint32_t key) -> int {
        return (key >> 22) == 999u ? -1 : G.cell_items[key & ((1u << 22) - 1)];
    };
    const int d0 = (int)(k0 >> 22), d1 = (int)(k1 >> 22);
    const int kp0 = kp_of(k0), kp1 = kp_of(k1);
    int match = -1;
    if (ncand > 0 && (float)d0 / (float)d1 <= W.ratio && !((float)d0 > (float)W.th)) match = kp0;
    o[0] = kp0;
    o[1] = d0;
    o[2] = kp1;
    o[3] = d1;
    o[4] = ncand;
    o[5] = match;
}

}  // namespace mcv
