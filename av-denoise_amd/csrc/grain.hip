// Film-grain measurement (grain_measure, nl4d/kernels/grain.rs:243-513; constants
// nl4d/grain/consts.rs:1-45).
//
// Source grain is the motion-compensated difference of ring slots slot_next and slot_t over sqrt 2;
// one-frame grain is the high-pass std of slot_t over the 8x8 cell.  A cell that passes the flatness,
// band, clipping, interior, confidence and std gates adds one count to its brightness bin and std
// bucket of the source histogram (i32 atomics); a usable cell adds one to the one-frame histogram.
// Every cell writes its partial: the 46 lag sums of its mean-free source grain over the cell and a halo
// of 6 columns each side and 3 rows below (zeros when rejected), its pixel count and its strength group.
// Every f32 sum follows the reference's order: the cell sums are 64-slot halving trees, each lag sum
// adds the 64 pixels row by row; so the histograms and partials are bit-identical to the reference's.
//
// Lanes are columns: eight lanes hold a cell, a wave eight cells side by side, each lane its column's
// eight rows in registers, so a row is one coalesced load, the tree's three upper levels are adds of
// registers and its three lower ones DPP adds within eight lanes.

#include "common.h"

namespace avd {
namespace {

constexpr int kCell = 8, kHalo = 6, kHaloRows = 3, kLags = 46, kPartial = 48;
constexpr int kBuckets = 64, kBins = 16, kHist = kBins * kBuckets;
// A measuring workgroup's cells: a wave takes eight of a row.
constexpr int kGroupX = 16, kGroupY = 2, kMeasureThreads = kGroupX * kGroupY * kCell;
constexpr int kPlaneW = kGroupX * kCell + 2 * kHalo, kPlaneH = kGroupY * kCell + kHaloRows;

template <int CTRL>
__device__ __forceinline__ float dpp(float v)
{
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), CTRL, 0xf, 0xf, true));
}

// Lane l ^ 4, l ^ 2, l ^ 1 in turn: the lower levels of a cell's halving tree, whose total reaches all
// eight lanes (an add is the same both ways round).
__device__ __forceinline__ float sum8(float v)
{
    v += dpp<0x141>(dpp<0x1B>(v));  // row_half_mirror of quad_perm 3,2,1,0
    v += dpp<0x4E>(v);              // quad_perm 2,3,0,1
    v += dpp<0xB1>(v);              // quad_perm 1,0,3,2
    return v;
}

__device__ __forceinline__ float min8(float v)
{
    v = fminf(v, dpp<0x141>(v));
    v = fminf(v, dpp<0x4E>(v));
    return fminf(v, dpp<0xB1>(v));
}

__device__ __forceinline__ float max8(float v)
{
    v = fmaxf(v, dpp<0x141>(v));
    v = fmaxf(v, dpp<0x4E>(v));
    return fmaxf(v, dpp<0xB1>(v));
}

// The cell's 64-slot halving tree: a slot is row * 8 + column, so strides 32, 16 and 8 pair rows.
template <class F>
__device__ __forceinline__ float tree_cell(F row)
{
    return sum8(((row(0) + row(4)) + (row(2) + row(6))) + ((row(1) + row(5)) + (row(3) + row(7))));
}

// Rust's saturating float-to-u32 cast, for the brightness bins.
__device__ inline uint32_t sat_u32(float v) { return !(v >= 0.0f) ? 0u : v >= 4294967296.0f ? 0xFFFFFFFFu : (uint32_t)v; }

__device__ inline int shift_clamp(int v, int s, int limit) { return min(max(v + s, 0), limit - 1); }

__device__ inline uint32_t block_for(int cx, int cy, uint32_t bx, uint32_t by, uint32_t step)
{
    return min((uint32_t)(cx * kCell) / step, bx - 1) + min((uint32_t)(cy * kCell) / step, by - 1) * bx;
}

// The highest bucket whose lower edge is at or below s (bucket_for, grain.rs:193-205): lane lx of the
// cell holds the edges of buckets 8 lx to 8 lx + 7.
__device__ inline uint32_t bucket_for(float s, const float (&edge)[kBuckets / 8], int lx)
{
    int b = 0;
#pragma unroll
    for (int j = 0; j < kBuckets / 8; ++j) b = s >= edge[j] ? lx * (kBuckets / 8) + j : b;
    b = max(b, __builtin_amdgcn_update_dpp(0, b, 0x141, 0xf, 0xf, true));
    b = max(b, __builtin_amdgcn_update_dpp(0, b, 0x4E, 0xf, 0xf, true));
    b = max(b, __builtin_amdgcn_update_dpp(0, b, 0xB1, 0xf, 0xf, true));
    return (uint32_t)b;
}

__device__ inline uint32_t luma_bin(float mean) { return min(sat_u32(mean * (float)kBins), (uint32_t)kBins - 1); }

// A workgroup of four waves takes 16 x 2 cells.  An accepted cell is an interior one, so its halo lies in
// whole cells and holds those cells' own grain: the workgroup keeps one plane of grain in LDS, its own
// pixels and a rim, and no pixel is fetched per cell.  In the lag sums lane lx of a cell takes six or
// seven neighbouring lags of one row offset, whose windows share their fourteen plane values.
// Bound by VALU issue (the lag sums' ordered multiplies and adds are half of it) and the chain vector ->
// sample -> tree -> lags.  1920x1080, one wave per cell with shuffle trees, a lane per lag and 156 halo
// pixels fetched per cell: 120 us; this form 17 us.
__global__ __launch_bounds__(kMeasureThreads) void k_grain_measure(
    const float *__restrict__ ring, const float *__restrict__ out_t, const int32_t *__restrict__ saved_mv,
    const float *__restrict__ saved_conf, const float *__restrict__ edges, const float *__restrict__ luma_means,
    int *__restrict__ hist, float *__restrict__ partials, int W, int H, int C, int ch, uint32_t slot_t,
    uint32_t slot_next, uint32_t bx, uint32_t by, uint32_t step, uint32_t entry, int has_source, int has_luma_means,
    uint32_t means_bx, int luma_band)
{
    // The workgroup's counts gather in LDS and reach `hist` as one atomic per non-empty bin: a flat
    // region sends every cell to the same bin, where per-cell global atomics would serialise.
    __shared__ __align__(16) int s_hist[2 * kHist];  // cleared by 16-byte stores
    __shared__ int2 s_vec[kGroupY + 1][kGroupX + 2];  // the group's cells', the rim's cells' vectors
    __shared__ __align__(16) float s_grain[kPlaneH * kPlaneW];
    __shared__ __align__(16) float s_centre[kGroupY * kCell][kGroupX * kCell];  // mean-free
    const int t = (int)threadIdx.x, lane = t & 63, wave = t >> 6, lx = lane & 7;
    const int cells_x = W / kCell, cells_y = H / kCell;
    const int gx = (int)blockIdx.x * kGroupX, gy = (int)blockIdx.y * kGroupY;
    const int tcx = (wave & 1) * 8 + (lane >> 3), tcy = wave >> 1;  // the lane's cell in the group
    const bool live = gx + tcx < cells_x && gy + tcy < cells_y;
    const int cx = min(gx + tcx, cells_x - 1), cy = min(gy + tcy, cells_y - 1);
    const int x = cx * kCell + lx, oy = cy * kCell;
    const size_t plane = (size_t)W * H, row_len = (size_t)W * C;
    const float *ft = ring + (size_t)slot_t * plane * C + ch, *fnx = ring + (size_t)slot_next * plane * C + ch;
    const uint32_t blocks = bx * by, base = entry * blocks * 2;
    constexpr float kR2 = 0.70710677f;

    float cur[kCell], clean[kCell];
    {
        const size_t at = ((size_t)oy * W + x) * C;
#pragma unroll
        for (int r = 0; r < kCell; ++r) {
            cur[r] = ft[at + r * row_len];
            clean[r] = out_t[at + r * row_len + ch];
        }
    }
    const float conf = saved_conf[entry * blocks + block_for(cx, cy, bx, by, step)];
    float edge[kBuckets / 8] = {};
    if (has_source) {
#pragma unroll
        for (int j = 0; j < kBuckets / 8; ++j) edge[j] = edges[max(lx * (kBuckets / 8) + j, 1)];
    }
    for (int i = t; i < 2 * kHist / 4; i += kMeasureThreads) ((int4 *)s_hist)[i] = make_int4(0, 0, 0, 0);
    if (t < (kGroupY + 1) * (kGroupX + 2)) {
        const int vx = min(max(gx - 1 + t % (kGroupX + 2), 0), cells_x - 1);
        const int vy = min(gy + t / (kGroupX + 2), cells_y - 1);
        const uint32_t b = base + block_for(vx, vy, bx, by, step) * 2;
        s_vec[t / (kGroupX + 2)][t % (kGroupX + 2)] = make_int2(saved_mv[b], saved_mv[b + 1]);
    }
    __syncthreads();

    float nxt[kCell];
    {
        const int2 v = s_vec[tcy][tcx + 1];
        const float *column = fnx + (size_t)shift_clamp(x, v.x, W) * C;
#pragma unroll
        for (int r = 0; r < kCell; ++r) nxt[r] = column[shift_clamp(oy + r, v.y, H) * row_len];
    }
    // The rim: three rows below the group, then six columns on either side of all rows.  A pixel past
    // the last whole cell takes the nearest one's, which no accepted cell reads.
    constexpr int kBelow = kHaloRows * kGroupX * kCell, kRim = kBelow + 2 * kHalo * kPlaneH;
    constexpr int kRimSteps = (kRim + kMeasureThreads - 1) / kMeasureThreads;
    float rim[kRimSteps];
#pragma unroll
    for (int j = 0; j < kRimSteps; ++j) {
        const int f = t + kMeasureThreads * j, side = f - kBelow;
        const int ty = side < 0 ? kGroupY * kCell + f / (kGroupX * kCell) : min(side / (2 * kHalo), kPlaneH - 1);
        const int sx = side % (2 * kHalo);
        const int tx = side < 0 ? kHalo + f % (kGroupX * kCell) : sx < kHalo ? sx : sx + kGroupX * kCell;
        const int hx = min(max(gx * kCell + tx - kHalo, 0), cells_x * kCell - 1);
        const int hy = min(gy * kCell + ty, cells_y * kCell - 1);
        const int2 v = s_vec[hy / kCell - gy][hx / kCell - gx + 1];
        const float n = fnx[((size_t)shift_clamp(hy, v.y, H) * W + shift_clamp(hx, v.x, W)) * C];
        rim[j] = (n - ft[((size_t)hy * W + hx) * C]) * kR2;
        if (f < kRim) s_grain[ty * kPlaneW + tx] = rim[j];
    }

    float g[kCell];
#pragma unroll
    for (int r = 0; r < kCell; ++r) {
        g[r] = (nxt[r] - cur[r]) * kR2;
        s_grain[(tcy * kCell + r) * kPlaneW + kHalo + tcx * kCell + lx] = g[r];
    }
    // One-frame high pass (neighbour_squares, grain.rs:251-269): squared steps to the right and lower
    // neighbours inside the cell, relative to the origin sample.
    const float origin = __shfl(cur[0], lane & ~7);
    float fv[kCell], hp[kCell];
#pragma unroll
    for (int r = 0; r < kCell; ++r) fv[r] = cur[r] - origin;
#pragma unroll
    for (int r = 0; r < kCell; ++r) {
        const float right = dpp<0x101>(fv[r]) - fv[r];  // row_shl 1: the next lane
        hp[r] = lx + 1 < kCell ? right * right : 0.0f;
        if (r + 1 < kCell) hp[r] += (fv[r + 1] - fv[r]) * (fv[r + 1] - fv[r]);
    }

    const float sum = tree_cell([&](int r) { return g[r]; }), sum_sq = tree_cell([&](int r) { return g[r] * g[r]; });
    const float clean_sum = tree_cell([&](int r) { return clean[r]; }), hp_sum = tree_cell([&](int r) { return hp[r]; });
    float clean_lo = clean[0], clean_hi = clean[0], src_lo = fminf(cur[0], nxt[0]), src_hi = fmaxf(cur[0], nxt[0]);
#pragma unroll
    for (int r = 1; r < kCell; ++r) {
        clean_lo = fminf(clean_lo, clean[r]);
        clean_hi = fmaxf(clean_hi, clean[r]);
        src_lo = fminf(src_lo, fminf(cur[r], nxt[r]));
        src_hi = fmaxf(src_hi, fmaxf(cur[r], nxt[r]));
    }
    clean_lo = min8(clean_lo);
    clean_hi = max8(clean_hi);
    src_lo = min8(src_lo);
    src_hi = max8(src_hi);

    const float count = 64.0f;
    const float var = (sum_sq - sum * sum / count) / (count - 1.0f);
    const float grain_std = sqrtf(fmaxf(var, 0.0f));
    const float mean = clean_sum / count;
    const float frame_std = sqrtf(hp_sum / 224.0f);
    const float range = clean_hi - clean_lo;
    const bool interior = cx >= 1 && cx + 2 <= cells_x && cy + 2 <= cells_y;
    const bool band = !luma_band || (mean > 20.0f / 255.0f && mean < 235.0f / 255.0f);
    const bool usable = live && has_source && range < 5.0f / 255.0f && band && src_lo >= 4.0f / 255.0f &&
                        src_hi <= 251.0f / 255.0f;
    const bool passes = usable && interior && conf >= 0.8f && grain_std > 0.05f / 255.0f;
    const bool frame_passes = usable && (means_bx == 0 || has_luma_means);
    // Whole waves look the buckets up together: their eight lanes exchange.
    const uint32_t bucket = bucket_for(grain_std, edge, lx), frame_bucket = bucket_for(frame_std, edge, lx);
    if (lx == 0 && passes) atomicAdd(s_hist + luma_bin(mean) * kBuckets + bucket, 1);
    if (lx == 0 && frame_passes) {
        uint32_t bin = luma_bin(mean);
        if (means_bx > 0) {
            const uint32_t mb = (uint32_t)(cy * kCell / 16) * means_bx + (uint32_t)(cx * kCell / 16);
            bin = min(sat_u32(luma_means[mb * 3] / 16.0f), (uint32_t)kBins - 1);
        }
        atomicAdd(s_hist + kHist + bin * kBuckets + frame_bucket, 1);
    }
    const float gmean = sum / 64.0f;
#pragma unroll
    for (int r = 0; r < kCell; ++r) s_centre[tcy * kCell + r][tcx * kCell + lx] = g[r] - gmean;
    __syncthreads();

    // Lane lx takes the lags of row offset `row` from plane column `col` on: dy 0's seven, then six and
    // seven of each further row; lane 7 writes the count and the group.
    constexpr int kRun = 7;
    const int role = min(lx, 6), row = (role + 1) >> 1, col = role & 1 ? 0 : kHalo;
    float acc[kRun];
#pragma unroll
    for (int k = 0; k < kRun; ++k) acc[k] = 0.0f;
    if (__any(passes)) {
        const float *c_at = &s_centre[tcy * kCell][tcx * kCell];
        const float *n_at = s_grain + (tcy * kCell + row) * kPlaneW + tcx * kCell + col;
#pragma unroll 1
        for (int py = 0; py < kCell; ++py, c_at += kGroupX * kCell, n_at += kPlaneW) {
            __align__(16) float c[kCell], n[kCell + kRun - 1];
#pragma unroll
            for (int i = 0; i < kCell / 4; ++i) *(float4 *)(c + 4 * i) = ((const float4 *)c_at)[i];
#pragma unroll
            for (int i = 0; i < (kCell + kRun - 1) / 2; ++i) *(float2 *)(n + 2 * i) = ((const float2 *)n_at)[i];
#pragma unroll
            for (int i = 0; i < kCell + kRun - 1; ++i) n[i] -= gmean;
#pragma unroll
            for (int px = 0; px < kCell; ++px)
#pragma unroll
                for (int k = 0; k < kRun; ++k) acc[k] += c[px] * n[px + k];
        }
    }
    if (lx == 7) {
        acc[0] = 64.0f;
        acc[1] = (float)(bucket / 4);
    }
    if (live) {
        float *part = partials + ((size_t)cy * cells_x + cx) * kPartial;
        part += lx == 7 ? kLags : row == 0 ? 0 : kRun + (row - 1) * 13 + col;
#pragma unroll
        for (int k = 0; k < kRun; ++k)
            if (k < (lx == 7 ? 2 : col == 0 ? kRun - 1 : kRun)) part[k] = passes ? acc[k] : 0.0f;
    }

    for (int i = t; i < 2 * kHist; i += kMeasureThreads) {
        const int n = s_hist[i];
        if (n) atomicAdd(hist + i, n);
    }
}

// grain_reduce_partials (grain.rs:515-560): for each record lane, column t of 128 adds the lane of
// cells t, t + 128, ... in turn into its strength group's sum (the group clamped to 15), then each
// group's 128 columns fold by a halving tree (the 64-stride step through LDS, the rest as wave shuffles,
// the same slot pairs) and group g's total is added into chunk[record_offset + 47 g + lane].
//
// Workgroup (s, g) takes record lanes 16 s to 16 s + 15 of group g: four threads a column, four lanes a
// thread.  A cell of another group adds an exact +0.0 (a column starts at +0.0 and so never holds -0.0,
// which an added +0.0 would change).  The ordered columns keep a total in one workgroup, so the bound is
// one compute unit's fill rate: the lanes and the group of a cell lie in different cache lines.  32400
// cells: a workgroup per lane, a column's 16 groups in one thread, 61 us; four lanes of a group per
// workgroup 57 to 59; two groups in sixteen lanes 60; this split 50 to 52.
constexpr int kReduceThreads = 128, kGroups = 16, kRecordLen = kLags + 1;
constexpr int kSector = 16, kSectors = kPartial / kSector;

__global__ __launch_bounds__(4 * kReduceThreads) void k_grain_reduce(const float *__restrict__ partials,
                                                                     float *__restrict__ chunk,
                                                                     uint32_t record_offset, uint32_t cells)
{
    struct __attribute__((aligned(4))) Quad {  // the caller's floats: a single float's alignment
        float v[4];
    };
    __shared__ float s_col[kSector][kReduceThreads + 1];
    const uint32_t group = blockIdx.y, t = threadIdx.x >> 2, quad = threadIdx.x & 3;
    const float *part = partials + blockIdx.x * kSector + quad * 4, *groups = partials + kLags + 1;
    float acc[4] = {0.0f, 0.0f, 0.0f, 0.0f};
    constexpr uint32_t kBatch = 8;
    for (uint32_t c = t; c < cells; c += kBatch * kReduceThreads) {
        Quad v[kBatch];
        float gv[kBatch];
#pragma unroll
        for (uint32_t j = 0; j < kBatch; ++j) {
            const size_t at = (size_t)min(c + j * kReduceThreads, cells - 1) * kPartial;
            v[j] = *(const Quad *)(part + at);
            gv[j] = groups[at];
        }
#pragma unroll
        for (uint32_t j = 0; j < kBatch; ++j) {
            const bool mine = c + j * kReduceThreads < cells && min(sat_u32(gv[j]), (uint32_t)kGroups - 1) == group;
#pragma unroll
            for (int e = 0; e < 4; ++e) acc[e] += mine ? v[j].v[e] : 0.0f;
        }
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) s_col[quad * 4 + e][t] = acc[e];
    __syncthreads();
    const uint32_t wave = threadIdx.x >> 6, l = threadIdx.x & 63;
#pragma unroll
    for (uint32_t i = wave; i < kSector; i += 4 * kReduceThreads / 64) {
        float x = s_col[i][l] + s_col[i][l + 64];
#pragma unroll
        for (int stride = 32; stride >= 1; stride >>= 1) x += __shfl_down(x, stride);
        const uint32_t lane = blockIdx.x * kSector + i;
        if (l == 0 && lane < kRecordLen) chunk[record_offset + group * kRecordLen + lane] += x;
    }
}

// The AR(3) fit in f64 (undo_mean_removal, yule_walker, solve and quantise_ar, nl4d/grain/fit.rs:
// 79-300): one wave per 47-value record, its state in registers.  Each of the 20 mean-removal rounds
// has lane l < 46 add lag l's cell-mean term over the 91 cell offsets that reach a measured lag, in the
// reference's order: the lane's weights are 91 registers (zero where the offset lies past the cell) and
// the lags broadcast reads.  In the solve lane r holds row r of the 24 x 25 system; a row swap only
// exchanges the lanes' row numbers, the pivot is the last of equal maxima in row order (as
// Iterator::max_by keeps), and its row reaches the others by v_readlane.  Every f64 operation is the
// reference's, in its order, so the results are bit-identical.  Bound by the chain of 20 x 91 dependent
// adds, which a record cannot shorten; a segment's records run side by side.  16 records: 351 us
// with the index arithmetic, the system in LDS and the pivot in one lane, 32 us now.
__device__ __forceinline__ constexpr int fit_lane(int dy, int dx)
{
    if (dy < 0 || (dy == 0 && dx < 0)) {
        dy = -dy;
        dx = -dx;
    }
    if (dy > 3 || dx > 6 || dx < -6) return -1;
    return dy == 0 ? dx : 7 + (dy - 1) * 13 + dx + 6;
}

__device__ __forceinline__ double readlane_f64(double v, int lane)
{
    const uint64_t u = __builtin_bit_cast(uint64_t, v);
    const uint32_t lo = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)u, lane);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(u >> 32), lane);
    return __builtin_bit_cast(double, (uint64_t)hi << 32 | lo);
}

// AR_OFFSETS: dy -3..0, dx -3..3, the causal half.
__device__ __forceinline__ constexpr int ar_dy(int i) { return i < 21 ? -3 + i / 7 : 0; }
__device__ __forceinline__ constexpr int ar_dx(int i) { return i < 21 ? i % 7 - 3 : i - 24; }

constexpr int kWeights = 24, kCellTerms = 7 * 13;

__global__ __launch_bounds__(64) void k_grain_fit(const double *__restrict__ records, double *__restrict__ corrected,
                                                  double *__restrict__ weights, int32_t *__restrict__ quantised,
                                                  uint32_t *__restrict__ shifts, int32_t *__restrict__ solved)
{
    __shared__ __align__(16) double s_lag[kRecordLen + 1];
    const int lane = (int)threadIdx.x;
    const size_t r = blockIdx.x;
    const double *rec = records + r * kRecordLen;
    // One wave: LDS written by its lanes is read by them after a fence.
    auto sync = [] {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
    };
    const double raw = lane < kRecordLen ? rec[lane] : 0.0;
    const double zero_lag = readlane_f64(raw, 0);
    double lag = raw;
    if (zero_lag > 0.0) {
        const int dy = lane < 7 ? 0 : lane < 20 ? 1 : lane < 33 ? 2 : 3;
        const int dx = lane < 7 ? lane : (lane - 7) % 13 - 6;
        double share[kCellTerms];  // pairs / 4096 of cell offset (ty - dy, tx - dx)
#pragma unroll
        for (int k = 0; k < kCellTerms; ++k) {
            const int oy = abs(k / 13 - 3 - dy), ox = abs(k % 13 - 6 - dx);
            share[k] = oy <= 7 && ox <= 7 ? (double)((8 - oy) * (8 - ox)) / 4096.0 : 0.0;
        }
        const double measured = raw / zero_lag;
        double rho = lane == 0 ? 1.0 : measured;
        for (int round = 0; round < 20; ++round) {
            if (lane < kLags) s_lag[lane] = rho;
            sync();
            double term = 0.0;
#pragma unroll
            for (int k = 0; k < kCellTerms; ++k) term += share[k] * s_lag[fit_lane(k / 13 - 3, k % 13 - 6)];
            rho = measured * (1.0 - readlane_f64(term, 0)) + term;  // lane 0's term is the zero lag's
            sync();
        }
        if (lane < kLags) lag = rho * zero_lag;
    }
    if (lane < kRecordLen) {
        corrected[r * kRecordLen + lane] = lag;
        s_lag[lane] = lag;
    }
    sync();

    const double pixels = s_lag[kLags];
    bool ok = pixels > 0.0;
    double mine = 0.0;  // lane i's weight
    if (ok) {
        const int row_id = lane < kWeights ? lane : 0;
        const int row_dy = ar_dy(row_id), row_dx = ar_dx(row_id);
        double m[kWeights + 1];
#pragma unroll
        for (int j = 0; j < kWeights; ++j) m[j] = s_lag[fit_lane(row_dy - ar_dy(j), row_dx - ar_dx(j))] / pixels;
        m[kWeights] = s_lag[fit_lane(row_dy, row_dx)] / pixels;
        int at = lane < kWeights ? lane : -1;  // the row number this lane's row has now
        int order[kWeights];                   // the lane that holds row number i
#pragma unroll
        for (int col = 0; col < kWeights; ++col) {
            if (!ok) break;
            // The pivot: the last row of the largest magnitude, or row `col` itself when that is NaN.
            const double a = fabs(m[col]);
            const int here = __builtin_ctzll(__ballot(at == col));
            double top = at >= col && !isnan(a) ? a : -1.0;
#pragma unroll
            for (int x = 1; x < 32; x <<= 1) top = fmax(top, __shfl_xor(top, x));
            const double first = readlane_f64(a, here);
            int pivot = here;
            if (!isnan(first)) {
                const double largest = readlane_f64(top, 0);
                uint64_t tied = __ballot(at >= col && a == largest);
                int row = -1;
                while (tied) {  // ties are rare; the lanes' rows are in no order
                    const int l = __builtin_ctzll(tied);
                    const int l_row = __builtin_amdgcn_readlane(at, l);
                    if (l_row > row) {
                        row = l_row;
                        pivot = l;
                    }
                    tied &= tied - 1;
                }
            }
            pivot = __builtin_amdgcn_readfirstlane(pivot);
            if (readlane_f64(a, pivot) < 1e-18) {
                ok = false;
                break;
            }
            const int pivot_row = __builtin_amdgcn_readlane(at, pivot);
            if (lane == here) at = pivot_row;
            if (lane == pivot) at = col;
            order[col] = pivot;
            const double head = readlane_f64(m[col], pivot);
            if (at > col) {
                const double factor = m[col] / head;
#pragma unroll
                for (int j = col; j <= kWeights; ++j) m[j] -= factor * readlane_f64(m[j], pivot);
            }
        }
        if (ok) {
            double sol[kWeights];
#pragma unroll
            for (int i = kWeights - 1; i >= 0; --i) {
                double v = m[kWeights];
#pragma unroll
                for (int j = i + 1; j < kWeights; ++j) v -= m[j] * sol[j];
                sol[i] = readlane_f64(v / m[i], order[i]);
                if (lane == i) mine = sol[i];
            }
            ok = __ballot(lane < kWeights && !isfinite(mine)) == 0;
        }
    }
    uint32_t shift = 6;
    for (uint32_t cand = 9; cand >= 7; --cand) {
        const double v = round(mine * (double)(1u << cand));
        if (__ballot(lane < kWeights && !(v >= -128.0 && v <= 127.0)) == 0) {
            shift = cand;
            break;
        }
    }
    if (lane < kWeights) {
        const double v = ok ? fmin(fmax(round(mine * (double)(1u << shift)), -128.0), 127.0) : 0.0;
        weights[r * kWeights + lane] = ok ? mine : 0.0;
        quantised[r * kWeights + lane] = (int32_t)v;
    }
    if (lane == 0) {
        shifts[r] = ok ? shift : 0u;
        solved[r] = ok ? 1 : 0;
    }
}

// grain_save_vectors (grain.rs:50-75): one neighbour's vectors and confidences into saved entry
// `entry`, a grid-stride copy.
__global__ void k_grain_save_vectors(const int32_t *__restrict__ mv_field, const float *__restrict__ confidence,
                                     int32_t *__restrict__ saved_mv, float *__restrict__ saved_conf,
                                     uint32_t mv_offset, uint32_t conf_offset, uint32_t entry, uint32_t blocks)
{
    for (uint32_t b = blockIdx.x * blockDim.x + threadIdx.x; b < blocks; b += gridDim.x * blockDim.x) {
        const uint32_t s = entry * blocks + b;
        saved_mv[s * 2] = mv_field[mv_offset + b * 2];
        saved_mv[s * 2 + 1] = mv_field[mv_offset + b * 2 + 1];
        saved_conf[s] = confidence[conf_offset + b];
    }
}

// grain_project (grain_persistence.rs:54-153): a wave per eight neighbouring cells, eight lanes a cell.
// The eight pattern projections (pixel y * 8 + x added where the pattern bit is set, taken away where
// clear) and the denoised mean are the cell's 64-slot trees; lane p of the cell writes projection p of
// its history entry, lane 0 the flat flag behind them.  Bound by memory latency (two frames read once).
// 1920x1080, one wave per cell with shuffle trees: 32 us; this form 5.4 us.
constexpr int kProjections = 8, kEntry = kProjections + 1;

__global__ __launch_bounds__(256) void k_grain_project(const float *__restrict__ ring, const float *__restrict__ out,
                                                       const uint32_t *__restrict__ patterns,
                                                       float *__restrict__ history, int W, int H, int C, int ch,
                                                       uint32_t frame_slot, uint32_t history_slot, int luma_band)
{
    const int lane = (int)threadIdx.x & 63, lx = lane & 7, cells_x = W / kCell, cells_y = H / kCell;
    const int gx = (int)blockIdx.x * 8 + (lane >> 3), cy = (int)blockIdx.y * 4 + ((int)threadIdx.x >> 6);
    if (cy >= cells_y) return;  // a whole wave; the kernel has no barrier
    const int cx = min(gx, cells_x - 1);
    const size_t row_len = (size_t)W * C, at = ((size_t)cy * kCell * W + cx * kCell + lx) * C + ch;
    const float *src = ring + (size_t)frame_slot * H * row_len + at, *den = out + at;
    float sample[kCell], clean[kCell];
#pragma unroll
    for (int r = 0; r < kCell; ++r) {
        sample[r] = src[r * row_len];
        clean[r] = den[r * row_len];
    }
    float mine = 0.0f;
#pragma unroll
    for (int p = 0; p < kProjections; ++p) {
        // Row r's bit is bit (r % 4) * 8 + lx of word r / 4; a clear bit flips the sample's sign.
        const uint32_t low = ~patterns[p * 2] >> lx, high = ~patterns[p * 2 + 1] >> lx;
        const float v = tree_cell([&](int r) {
            const uint32_t flip = ((r < 4 ? low : high) << (31 - (r & 3) * 8)) & 0x80000000u;
            return __builtin_bit_cast(float, __builtin_bit_cast(uint32_t, sample[r]) ^ flip);
        });
        mine = lx == p ? v : mine;
    }
    const float clean_sum = tree_cell([&](int r) { return clean[r]; });
    float clean_lo = clean[0], clean_hi = clean[0], src_lo = sample[0], src_hi = sample[0];
#pragma unroll
    for (int r = 1; r < kCell; ++r) {
        clean_lo = fminf(clean_lo, clean[r]);
        clean_hi = fmaxf(clean_hi, clean[r]);
        src_lo = fminf(src_lo, sample[r]);
        src_hi = fmaxf(src_hi, sample[r]);
    }
    clean_lo = min8(clean_lo);
    clean_hi = max8(clean_hi);
    src_lo = min8(src_lo);
    src_hi = max8(src_hi);
    if (gx < cells_x) {
        const float mean = clean_sum / 64.0f, range = clean_hi - clean_lo;
        const bool band = !luma_band || (mean > 20.0f / 255.0f && mean < 235.0f / 255.0f);
        const bool flat = range < 5.0f / 255.0f && band && src_lo >= 4.0f / 255.0f && src_hi <= 251.0f / 255.0f;
        float *e = history + ((size_t)history_slot * cells_x * cells_y + (size_t)cy * cells_x + cx) * kEntry;
        e[lx] = mine;
        if (lx == 0) e[kProjections] = flat ? 1.0f : 0.0f;
    }
}

// grain_persist (grain_persistence.rs:155-230): workgroup (block, n) of 256 threads covers 1024
// cells at lag n + 1; thread t walks cells t, t + 256, t + 512, t + 768 of the block in turn, then
// each lane (count, auto, cross) folds by a 256-slot halving tree (the 128- and 64-stride steps
// through LDS, the rest as shuffles).
constexpr int kPersistThreads = 256, kPersistCells = 1024, kHistoryFrames = 9;

__global__ __launch_bounds__(kPersistThreads) void k_grain_persist(const float *__restrict__ history,
                                                                   float *__restrict__ partials, uint32_t now_slot,
                                                                   uint32_t cells, uint32_t blocks)
{
    __shared__ float s[3][kPersistThreads];
    const uint32_t t = threadIdx.x, block = blockIdx.x, lag = blockIdx.y;
    const uint32_t earlier = (now_slot + kHistoryFrames - 1 - lag) % kHistoryFrames;
    float count = 0.0f, auto_sum = 0.0f, cross_sum = 0.0f;
#pragma unroll
    for (uint32_t step = 0; step < kPersistCells / kPersistThreads; ++step) {
        const uint32_t cell = block * kPersistCells + t + step * kPersistThreads;
        if (cell < cells) {
            const float *now = history + ((size_t)now_slot * cells + cell) * kEntry;
            const float *ear = history + ((size_t)earlier * cells + cell) * kEntry;
            if (now[kProjections] * ear[kProjections] > 0.5f) {
                float sq = 0.0f, pr = 0.0f;
#pragma unroll
                for (int p = 0; p < kProjections; ++p) {
                    sq += now[p] * now[p] + ear[p] * ear[p];
                    pr += now[p] * ear[p];
                }
                count += 1.0f;
                auto_sum += sq * (1.0f / 1024.0f);
                cross_sum += pr * (1.0f / 512.0f);
            }
        }
    }
    s[0][t] = count;
    s[1][t] = auto_sum;
    s[2][t] = cross_sum;
    __syncthreads();
    if (t < 64) {
        float v[3];
#pragma unroll
        for (int l = 0; l < 3; ++l) {
            v[l] = (s[l][t] + s[l][t + 128]) + (s[l][t + 64] + s[l][t + 192]);
#pragma unroll
            for (int stride = 32; stride >= 1; stride >>= 1) v[l] += __shfl_down(v[l], stride);
        }
        if (t == 0) {
#pragma unroll
            for (int l = 0; l < 3; ++l) partials[((size_t)lag * blocks + block) * 3 + l] = v[l];
        }
    }
}

// grain_persist_reduce (grain_persistence.rs:232-279): workgroup n of 128 threads; thread t adds
// blocks t, t + 128, ... in turn per lane, then a 128-slot tree (the 64-stride step through LDS, the
// rest as shuffles), added into record[record_offset + 3 n + lane].
__global__ __launch_bounds__(kReduceThreads) void k_grain_persist_reduce(const float *__restrict__ partials,
                                                                         float *__restrict__ record,
                                                                         uint32_t record_offset, uint32_t blocks)
{
    __shared__ float s[3][kReduceThreads];
    const uint32_t t = threadIdx.x, lag = blockIdx.x;
    float acc[3] = {0.0f, 0.0f, 0.0f};
    for (uint32_t b = t; b < blocks; b += kReduceThreads)
#pragma unroll
        for (int l = 0; l < 3; ++l) acc[l] += partials[((size_t)lag * blocks + b) * 3 + l];
#pragma unroll
    for (int l = 0; l < 3; ++l) s[l][t] = acc[l];
    __syncthreads();
    if (t < 64) {
        float v[3];
#pragma unroll
        for (int l = 0; l < 3; ++l) {
            v[l] = s[l][t] + s[l][t + 64];
#pragma unroll
            for (int stride = 32; stride >= 1; stride >>= 1) v[l] += __shfl_down(v[l], stride);
        }
        if (t == 0) {
#pragma unroll
            for (int l = 0; l < 3; ++l) record[record_offset + lag * 3 + l] += v[l];
        }
    }
}

}  // namespace

uint32_t grain_partials_len(uint32_t width, uint32_t height)
{
    return (width / kCell) * (height / kCell) * kPartial;
}

hipError_t launch_grain_measure(const GrainMeasure &m, hipStream_t s)
{
    const uint32_t cells = (m.width / kCell) * (m.height / kCell);
    if (cells == 0) return hipSuccess;
    const dim3 groups(div_up(m.width / kCell, kGroupX), div_up(m.height / kCell, kGroupY));
    k_grain_measure<<<groups, kMeasureThreads, 0, s>>>(
        m.ring, m.denoised, m.saved_mv, m.saved_conf, m.edges, m.luma_means, m.hist, m.partials, (int)m.width,
        (int)m.height, (int)m.channels, (int)m.channel, m.slot_t, m.slot_next, m.blocks_x, m.blocks_y, m.step,
        m.source_entry, m.has_source ? 1 : 0, m.has_luma_means ? 1 : 0, m.means_blocks_x, m.luma_band ? 1 : 0);
    return hipGetLastError();
}

hipError_t launch_grain_reduce(const float *partials, uint32_t cells, float *chunk, uint32_t record_offset,
                               hipStream_t s)
{
    if (!partials || !chunk) return hipErrorInvalidValue;
    k_grain_reduce<<<dim3(kSectors, kGroups), 4 * kReduceThreads, 0, s>>>(partials, chunk, record_offset, cells);
    return hipGetLastError();
}

hipError_t launch_grain_fit(const double *records, uint32_t count, double *corrected, double *weights,
                            int32_t *quantised, uint32_t *shifts, int32_t *solved, hipStream_t s)
{
    if (!records || !corrected || !weights || !quantised || !shifts || !solved) return hipErrorInvalidValue;
    if (count == 0) return hipSuccess;
    k_grain_fit<<<count, 64, 0, s>>>(records, corrected, weights, quantised, shifts, solved);
    return hipGetLastError();
}

hipError_t launch_grain_save_vectors(const int32_t *mv_field, const float *confidence, int32_t *saved_mv,
                                    float *saved_conf, uint32_t mv_offset, uint32_t conf_offset, uint32_t entry,
                                    uint32_t blocks, hipStream_t s)
{
    if (!mv_field || !confidence || !saved_mv || !saved_conf) return hipErrorInvalidValue;
    if (blocks == 0) return hipSuccess;
    k_grain_save_vectors<<<std::min<uint32_t>((blocks + 255) / 256, 1024), 256, 0, s>>>(
        mv_field, confidence, saved_mv, saved_conf, mv_offset, conf_offset, entry, blocks);
    return hipGetLastError();
}

hipError_t launch_grain_project(const float *ring, const float *out, const uint32_t *patterns, float *history,
                                uint32_t width, uint32_t height, uint32_t channels, uint32_t channel,
                                uint32_t frame_slot, uint32_t history_slot, bool luma_band, hipStream_t s)
{
    const uint32_t cells = (width / kCell) * (height / kCell);
    if (cells == 0) return hipSuccess;
    k_grain_project<<<dim3(div_up(width / kCell, 8), div_up(height / kCell, 4)), 256, 0, s>>>(
        ring, out, patterns, history, (int)width, (int)height, (int)channels, (int)channel, frame_slot, history_slot,
        luma_band ? 1 : 0);
    return hipGetLastError();
}

uint32_t grain_persist_blocks(uint32_t cells) { return (cells + kPersistCells - 1) / kPersistCells; }

hipError_t launch_grain_persist(const float *history, float *partials, float *record, uint32_t record_offset,
                                uint32_t now_slot, uint32_t cells, uint32_t lags, hipStream_t s)
{
    const uint32_t blocks = grain_persist_blocks(cells);
    if (blocks == 0 || lags == 0) return hipSuccess;
    k_grain_persist<<<dim3(blocks, lags), kPersistThreads, 0, s>>>(history, partials, now_slot, cells, blocks);
    k_grain_persist_reduce<<<lags, kReduceThreads, 0, s>>>(partials, record, record_offset, blocks);
    return hipGetLastError();
}

}  // namespace avd
