// Spatial noise measurement: the two stages of the Immerkaer estimate
// (nlm_noise_partial / nlm_noise_reduce, noise/kernels/stats.rs:24-140; driven by
// noise/spatial.rs:93-125).
//
// Stage 1: per 32x8 tile of the frame (sixteen tile sums per workgroup).  Every interior pixel applies the 3x3 mask
//   [1 -2 1; -2 4 -2; 1 -2 1], which cancels affine content and leaves mostly noise, and the tile
//   sums the absolute responses of each channel into its own lane of the tile's two partials.
//   Border pixels, pixels past the frame and unused lanes contribute zero.
// Stage 2: one workgroup of 256 threads sums every partial into the two per-channel totals of row
//   `slot` of the results.
// Both sums are f32 in the reference's order (thread l of stage 2 adds partials l, l + 256, ... in
// turn; each total then adds its 256 thread sums in thread order, as does each tile in stage 1),
// so the totals are bit-identical to the reference's.  The work is one read of the frame (HBM).

#include <algorithm>
#include <mutex>
#include <type_traits>

#include "common.h"

namespace avd {

// The partials of the entry point that allocates nothing: a file-scope device array, one copy per
// GPU at its own address, resolved once per device by hipGetSymbolAddress.  Host code only ever
// uses that resolved address.  Every partial the reduce reads is written by the partial kernel of
// the same call first, so the array needs no clearing; calls that overlap on one GPU race on it.
__device__ __align__(256) float scratch[kNoiseScratchFloats];

namespace {

constexpr int kImmBlockX = 32, kImmBlockY = 8;  // the tile (noise/mod.rs:117-119)
constexpr int kImmLanes = 2;                    // partials per tile and totals per slot
constexpr int kReduceBlock = 256;               // stage 2's threads (noise/mod.rs:122)

// A workgroup takes sixteen tile sums: two tile rows of 256 / C columns.  Thread (column, channel)
// walks its column's sixteen rows with the rows above and below in registers and leaves the responses'
// magnitudes in one LDS plane per (tile, channel); then a lane per plane adds its tile's 256 in thread
// order.  Bound by that chain and the loads it waits for, hidden by the eight workgroups a CU holds.
// 3840x2160 luma: 18.6 us with a thread per pixel and eight tiles' chains per workgroup, 9.8 us now.
constexpr int kTileRows = 2, kPlanes = 16;
// Workgroups along y of a grid layer; a taller frame (past 2^19 rows) takes further layers along z, as a
// grid's y extent is limited to 16 bits.
constexpr uint32_t kGridRows = 1u << 15;
constexpr int kPlaneStride = kImmBlockX * kImmBlockY + 32;

// Where columns 4 g .. 4 g + 3 of row 0 of LDS plane i start: neighbouring planes 32 banks apart and the
// groups of every second plane permuted, so that the 64 columns a wave writes and the sixteen planes a
// lane each reads both cover all 64 banks.
__device__ __forceinline__ int imm_plane_at(int i, int g) { return i * kPlaneStride + 4 * (g ^ (i >> 1)); }

template <int C>
__global__ __launch_bounds__(256) void k_noise_partial(const float *__restrict__ ring, float *__restrict__ partials,
                                                       uint32_t frame, int W, int H)
{
    constexpr int kCols = 256 / C, kRows = kTileRows * kImmBlockY, kTilesX = kCols / kImmBlockX;
    __shared__ __align__(16) float s_abs[kPlanes * kPlaneStride];
    const int t = (int)threadIdx.x, c = t % C, col = t / C;
    const int tiles_x = (W + kImmBlockX - 1) / kImmBlockX, tiles_y = (H + kImmBlockY - 1) / kImmBlockY;
    const int group_y = (int)(blockIdx.z * kGridRows + blockIdx.y);
    if (group_y > (H - 1) / kRows) return;  // the last layer's surplus: whole workgroups
    const int x = (int)blockIdx.x * kCols + col, y0 = group_y * kRows;
    const size_t pitch = (size_t)W * C;
    const float *f = ring + (size_t)frame * W * H * C + c;
    const bool in_x = x >= 1 && x < W - 1;
    // Columns x - 1, x, x + 1 (all x where the mask does not apply: the response is dropped).
    const float *left = f + (size_t)(in_x ? x - 1 : min(x, W - 1)) * C, *right = left + (in_x ? 2 * C : 0);
    const float *mid = left + (in_x ? C : 0);
    float l[kRows + 2], m[kRows + 2], r[kRows + 2];
#pragma unroll
    for (int k = 0; k < kRows + 2; ++k) {
        const size_t at = (size_t)min(max(y0 + k - 1, 0), H - 1) * pitch;
        l[k] = left[at];
        m[k] = mid[at];
        r[k] = right[at];
    }
#pragma unroll
    for (int k = 0; k < kRows; ++k) {
        // The reference's expression order: centre 4 - (left + right + up + down) 2 + the corners.
        const float response = m[k + 1] * 4.0f - (l[k + 1] + r[k + 1] + m[k] + m[k + 2]) * 2.0f +
                               (l[k] + r[k] + l[k + 2] + r[k + 2]);
        const bool in = in_x && y0 + k >= 1 && y0 + k < H - 1;
        const int plane = ((k / kImmBlockY) * kTilesX + col / kImmBlockX) * C + c, px = col % kImmBlockX;
        s_abs[imm_plane_at(plane, px >> 2) + (px & 3) + (k % kImmBlockY) * kImmBlockX] = in ? fabsf(response) : 0.0f;
    }
    __syncthreads();
    // One wave adds, turned with the workgroup so that it is not always on the same SIMD.
    const int lane = t & 63;
    if (t >> 6 != (int)(blockIdx.x + blockIdx.y) % 4 || lane >= kPlanes) return;
    float sum = 0.0f;
#pragma unroll 2
    for (int row = 0; row < kImmBlockY; ++row) {
        float4 v[kImmBlockX / 4];
#pragma unroll
        for (int g = 0; g < kImmBlockX / 4; ++g)
            v[g] = *reinterpret_cast<const float4 *>(s_abs + imm_plane_at(lane, g) + row * kImmBlockX);
#pragma unroll
        for (int g = 0; g < kImmBlockX / 4; ++g) sum = (((sum + v[g].x) + v[g].y) + v[g].z) + v[g].w;
    }
    const int tx = (int)blockIdx.x * kTilesX + lane / C % kTilesX, ty = group_y * kTileRows + lane / C / kTilesX;
    if (tx < tiles_x && ty < tiles_y) {
        float *out = partials + ((size_t)ty * tiles_x + tx) * kImmLanes;
        out[lane % C] = sum;
        if (C == 1) out[1] = 0.0f;
    }
}

// Thread t adds partials t, t + 256, ... of both lanes in turn, 64 loads in flight at a time; then one
// lane per total adds the 256 thread sums.  3840x2160: 11.3 us with 32 loads of each lane apart and the
// thread sums read one by one, 7 us now.
struct Partial {  // of a tile's lanes; 4-byte aligned, as the caller's floats
    float x, y;
};

__global__ __launch_bounds__(kReduceBlock) void k_noise_reduce(const Partial *__restrict__ partials,
                                                                float *__restrict__ results, uint32_t slot,
                                                                uint32_t count)
{
    constexpr uint32_t kTail = 8;
    __shared__ __align__(16) float s_sum[kImmLanes][kReduceBlock];
    const uint32_t t = threadIdx.x;
    float sum0 = 0.0f, sum1 = 0.0f;
    uint32_t i = t;
    // Whole batches of a fixed size while one fits, so that no load waits for the batch's adds.
    auto batches = [&](auto size) {
        constexpr uint32_t n = decltype(size)::value;
#pragma unroll 1
        for (; i + (n - 1) * kReduceBlock < count; i += kReduceBlock * n) {
            Partial v[n];
#pragma unroll
            for (uint32_t u = 0; u < n; ++u) v[u] = partials[i + u * kReduceBlock];
#pragma unroll
            for (uint32_t u = 0; u < n; ++u) {
                sum0 += v[u].x;
                sum1 += v[u].y;
            }
        }
    };
    batches(std::integral_constant<uint32_t, 64>{});
    batches(std::integral_constant<uint32_t, 16>{});
#pragma unroll 1
    for (; i < count; i += kReduceBlock * kTail) {
        Partial v[kTail];
#pragma unroll
        for (uint32_t u = 0; u < kTail; ++u) v[u] = partials[min(i + u * kReduceBlock, count - 1)];
#pragma unroll
        for (uint32_t u = 0; u < kTail; ++u) {
            const bool in = i + u * kReduceBlock < count;
            sum0 = in ? sum0 + v[u].x : sum0;
            sum1 = in ? sum1 + v[u].y : sum1;
        }
    }
    s_sum[0][t] = sum0;
    s_sum[1][t] = sum1;
    __syncthreads();
    if (t < (uint32_t)kImmLanes) {
        float total = 0.0f;
#pragma unroll 16
        for (int k = 0; k < kReduceBlock; k += 4) {
            const float4 v = *reinterpret_cast<const float4 *>(&s_sum[t][k]);
            total = (((total + v.x) + v.y) + v.z) + v.w;
        }
        results[(size_t)slot * kImmLanes + t] = total;
    }
}

}  // namespace

uint32_t noise_partials_len(uint32_t width, uint32_t height)
{
    return ((width + kImmBlockX - 1) / kImmBlockX) * ((height + kImmBlockY - 1) / kImmBlockY) * kImmLanes;
}

hipError_t launch_noise_spatial(const float *ring, uint32_t width, uint32_t height, uint32_t channels,
                                uint32_t frame, float *partials, float *results, uint32_t slot, hipStream_t s)
{
    if (!ring || !partials || !results || width == 0 || height == 0 || (channels != 1 && channels != 2) ||
        (uint64_t)width * height * channels * (frame + 1ull) > (1ull << 40))
        return hipErrorInvalidValue;
    const uint32_t tiles_x = (width + kImmBlockX - 1) / kImmBlockX, tiles_y = (height + kImmBlockY - 1) / kImmBlockY;
    const uint32_t rows = div_up(height, kTileRows * kImmBlockY);
    const dim3 grid(div_up(width, 256 / channels), std::min(rows, kGridRows), div_up(rows, kGridRows));
    if (channels == 1)
        k_noise_partial<1><<<grid, 256, 0, s>>>(ring, partials, frame, (int)width, (int)height);
    else
        k_noise_partial<2><<<grid, 256, 0, s>>>(ring, partials, frame, (int)width, (int)height);
    k_noise_reduce<<<1, kReduceBlock, 0, s>>>(reinterpret_cast<const Partial *>(partials), results, slot,
                                              tiles_x * tiles_y);
    return hipGetLastError();
}

hipError_t noise_scratch_address(float **out)
{
    constexpr int kMaxDevices = 64;
    static std::mutex mu;
    static float *resolved[kMaxDevices] = {};
    int dev = -1;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return e;
    if (dev < 0 || dev >= kMaxDevices) return hipErrorInvalidDevice;
    std::lock_guard<std::mutex> lock(mu);
    if (!resolved[dev]) {
        void *ptr = nullptr;
        e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
        if (e != hipSuccess) return e;
        resolved[dev] = static_cast<float *>(ptr);
    }
    *out = resolved[dev];
    return hipSuccess;
}

// ---------------------------------------------------------------------------------------------
// Temporal block statistics (nlm_temporal_noise_stats, noise/kernels/stats.rs:142-604; record layout
// noise/temporal.rs:18-131; driven by run_temporal_noise_stats, noise/temporal.rs:206-257).
//
// The residual is frame slot_new minus frame slot_prev of the ring.  A record holds per channel sum_d
// and sum_d2, the lag-1 product sum of channel 0's row neighbours, channel 0's cell texture, the moved
// flag, four quarter records of channel 0 (sum_d, sum_d2, luma sum, flatness, luma min, luma max) and
// every further channel's texture.  Each f32 sum follows the reference's order: a lane total adds its
// 256 pixel values in pixel order, the gain check and the quarter sums are halving trees (slot s +
// stride into slot s, stride n/2 .. 1), cell means add their pixels row by row.  So the records are
// bit-identical to the reference's f32 records.
//
// k_temporal_stats: a workgroup takes 16 / C consecutive blocks: its threads sweep the blocks' rows into
// LDS (new and previous frame, and with motion the previous frame along each block's vector), then each
// wave runs one kind of ordered sum with a lane per (block, channel) or (block, quarter): sum_d with the
// cell means and textures, sum_d2, the lag-1 products, the quarter sums and extremes, the flatness grids
// with the first or, with motion, the last; before them, with motion, wave k tree k of the gain checks.  So
// the chains of 16 planes run side by side in one wave's lanes, in loops short enough for the instruction
// cache.  Bound by the chains' instruction issue.  3840x2160 with motion: a workgroup per block and a thread
// per pixel 114 us (each chain a few active lanes of a wave), a quarter per lane in registers, unrolled,
// 55 us (its thousands of instructions run once per wave, fetched cold), this form 30 us.
// k_temporal_small keeps a workgroup per block for frames of few blocks, where a workgroup's own chain is
// what takes the time: a two-channel 477x269 frame 4.9 us (6.2 with motion) against 6.2 (8.9) in sixteens.
// ---------------------------------------------------------------------------------------------

namespace {

constexpr int kTB = 16, kTQ = kTB / 2;  // a block's side and its quarters'
constexpr int kTThreads = 256;
constexpr int kTStride = kTB * kTB + 16;  // floats between planes; see plane_at
constexpr uint32_t kXcds = 8;
constexpr float kUnmeasuredFlatness = 3.0e38f;
constexpr float kCompensationGainMax = 0.5f;

// Where group g (four columns) of row 0 of plane i of an LDS array of 16x16 planes starts.  Planes sit
// 16 banks apart and every four planes permute the groups of a row, so the four planes a wave writes
// together (64 columns of a row) and the sixteen planes it reads together (a lane per plane, the same
// group) both cover all 64 banks.
__device__ __forceinline__ int plane_at(int i, int g) { return i * kTStride + 4 * (g ^ ((i >> 2) & 3)); }

__device__ __forceinline__ float4 lds4(const float *p) { return *reinterpret_cast<const float4 *>(p); }

// The mean squared step between adjacent 4x4-cell means fully inside a bw x bh block, or 0 with no
// such pair; `cells` holds the 16 means row-major (cell_texture, stats.rs:626-656).
__device__ __forceinline__ float cell_texture(const float (&cells)[16], int bw, int bh)
{
    const int cols = bw >> 2, rows = bh >> 2;
    float energy = 0.0f;
    int pairs = 0;
#pragma unroll
    for (int cy = 0; cy < 4; ++cy)
#pragma unroll
        for (int cx = 0; cx < 4; ++cx) {
            const bool here = cx < cols && cy < rows;
            if (cx < 3) {
                const float step = cells[cy * 4 + cx] - cells[cy * 4 + cx + 1];
                const bool both = here && cx + 1 < cols;
                energy = both ? energy + step * step : energy;
                pairs += both;
            }
            if (cy < 3) {
                const float step = cells[cy * 4 + cx] - cells[(cy + 1) * 4 + cx];
                const bool both = here && cy + 1 < rows;
                energy = both ? energy + step * step : energy;
                pairs += both;
            }
        }
    return pairs ? energy / (float)pairs : 0.0f;
}

// A halving tree over eight rows' values (r + 4, r + 2, r + 1), and over four columns' (c + 2, c + 1).
__device__ __forceinline__ float fold8(const float (&v)[8])
{
    return ((v[0] + v[4]) + (v[2] + v[6])) + ((v[1] + v[5]) + (v[3] + v[7]));
}
__device__ __forceinline__ float fold4(const float (&v)[4]) { return (v[0] + v[2]) + (v[1] + v[3]); }

// fminf / fmaxf without the quieting operation a load would get first: their operands hold no signalling
// NaN (which this instruction passes on, where it drops a quiet one).
__device__ __forceinline__ float min_f(float a, float b)
{
    float r;
    asm("v_min_f32 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
    return r;
}
__device__ __forceinline__ float max_f(float a, float b)
{
    float r;
    asm("v_max_f32 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
    return r;
}

template <int C, bool LUMA, bool COMP>
__global__ __launch_bounds__(kTThreads) void k_temporal_stats(const float *__restrict__ ring, float *__restrict__ stats,
                                                              const int32_t *__restrict__ mv, uint32_t slot_new,
                                                              uint32_t slot_prev, uint32_t mv_offset, uint32_t mv_step,
                                                              uint32_t mv_bx, uint32_t mv_by, int W, int H)
{
    constexpr int NB = 16 / C, kRec = 3 * C + 26, kPlane = 16 * kTStride;
    // Plane i C + c is block i's channel c.  With motion: the new frame, the previous one and the previous
    // one along the block's vector, from which the sums below take residual and mean once the gain check
    // has picked; without, the new frame, the residual and the mean themselves.
    __shared__ __align__(16) float s_new[kPlane], s_old[kPlane], s_mov[kPlane];
    __shared__ float s_gain[4][NB];
    __shared__ int s_vec[NB][2], s_follow[NB], s_matched[NB];
    const int t = (int)threadIdx.x, lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6);
    const uint32_t nbx = ((uint32_t)W + kTB - 1) / kTB, blocks = nbx * (((uint32_t)H + kTB - 1) / kTB);
    // Workgroups reach the eight XCDs round robin; XCD x takes a contiguous run of the row-major
    // blocks, so blocks that share a 128-byte row segment meet in one L2.
    const uint32_t xcd = blockIdx.x % kXcds, per = gridDim.x / kXcds, extra = gridDim.x % kXcds;
    const uint32_t first = (xcd * per + min(xcd, extra) + blockIdx.x / kXcds) * NB;
    const size_t plane = (size_t)W * H * C;
    const float *fn = ring + (size_t)slot_new * plane, *fp = ring + (size_t)slot_prev * plane;

    // Block i of the workgroup (the last block again past the end; nothing is written for it).
    struct Block {
        uint32_t b;
        int ox, oy, bw, bh;
        bool live;
    };
    auto block = [&](int i) {
        Block k;
        k.live = first + i < blocks;
        k.b = min(first + i, blocks - 1);
        k.ox = (int)(k.b % nbx) * kTB;
        k.oy = (int)(k.b / nbx) * kTB;
        k.bw = min(kTB, W - k.ox);
        k.bh = min(kTB, H - k.oy);
        return k;
    };

    // ---- the samples: thread t on column t % 16 (and channel) of block t / (16 C), row by row; what
    // lies outside the frame enters as 0.
    if constexpr (COMP) {
        if (t < NB) {
            const Block k = block(t);
            const uint32_t col = min((uint32_t)k.ox / mv_step, mv_bx - 1), row = min((uint32_t)k.oy / mv_step, mv_by - 1);
            const int32_t *v = mv + mv_offset + (size_t)(row * mv_bx + col) * 2;
            s_vec[t][0] = v[0];
            s_vec[t][1] = v[1];
        }
        __syncthreads();
    }
    {
        const int i = t / (kTB * C), lx = t % (kTB * C) / C, c = t % C;
        const int dst = plane_at(i * C + c, lx >> 2) + (lx & 3);
        const Block k = block(i);
        const size_t pitch = (size_t)W * C;
        const bool in_x = lx < k.bw;
        const int x = min(k.ox + lx, W - 1);
        const float *pn = fn + (size_t)k.oy * pitch + (size_t)x * C + c, *po = fp + (pn - fn), *pm = po;
        // Rows [m_lo, m_hi) of this column have their match in the frame.
        int m_lo = 0, m_hi = 0;
        if constexpr (COMP) {
            const long mx = (long)k.ox + lx + s_vec[i][0], my = (long)k.oy + s_vec[i][1];
            if (in_x && mx >= 0 && mx < W) {
                m_lo = (int)min(max(-my, 0l), (long)kTB);
                m_hi = (int)max(min((long)H - my, (long)k.bh), 0l);
                if (m_lo < m_hi) pm = fp + (my + m_lo) * (long)pitch + mx * C + c;
            }
        }
        float a[kTB], b[kTB], m[COMP ? kTB : 1];
#pragma unroll
        for (int r = 0; r < kTB; ++r) {
            a[r] = *pn;
            b[r] = *po;
            const size_t next = r + 1 < k.bh ? pitch : 0;  // rows past the frame read the last one again
            pn += next;
            po += next;
            if constexpr (COMP) {
                m[r] = *pm;
                pm += r >= m_lo && r + 1 < m_hi ? pitch : 0;
            }
        }
#pragma unroll
        for (int r = 0; r < kTB; ++r) {
            const bool in = in_x && r < k.bh;
            // Quiet, for the extremes: every other use only adds.
            s_new[dst + r * kTB] = in ? __builtin_canonicalizef(a[r]) : 0.0f;
            if constexpr (COMP) {
                s_old[dst + r * kTB] = in ? b[r] : 0.0f;
                // A pixel whose match leaves the frame takes no part: its residual along the vector is
                // new - new = 0 (a value that is not finite fails the check by its zero residual).
                s_mov[dst + r * kTB] = !in ? 0.0f : (r >= m_lo && r < m_hi ? m[r] : a[r]);
            } else {
                s_old[dst + r * kTB] = in ? a[r] - b[r] : 0.0f;
                s_mov[dst + r * kTB] = in ? 0.5f * (a[r] + b[r]) : 0.0f;
            }
        }
    }
    __syncthreads();

    if constexpr (COMP) {
        // The gain check (stats.rs:257-341): the block follows its vector when channel 0's residual
        // variance along it, over the pixels whose match stays in the frame, is at most half the
        // zero-vector variance, or when no match stays in the frame; a followed block whose shifted
        // extent leaves the frame is unmatched and writes zeros.  Wave k sums tree k (zero residuals,
        // their squares, residuals along the vector, their squares): lane (column quad, block) folds its
        // columns' sixteen rows (r + 8, r + 4, r + 2, r + 1), then columns c + 8 and c + 4 come from the
        // lanes 32 and 16 away and c + 2, c + 1 are its own.
        const int at = plane_at(min(lane & 15, NB - 1) * C, lane >> 4);
        const float *old = wave < 2 ? s_old : s_mov;
        float col[4][8], d[4][kTB];
#pragma unroll
        for (int r = 0; r < kTB; ++r) {
            const float4 n = lds4(s_new + at + r * kTB), o = lds4(old + at + r * kTB);
            d[0][r] = n.x - o.x, d[1][r] = n.y - o.y, d[2][r] = n.z - o.z, d[3][r] = n.w - o.w;
        }
        if (wave & 1) {
#pragma unroll
            for (int r = 0; r < kTB; ++r)
#pragma unroll
                for (int c = 0; c < 4; ++c) d[c][r] = d[c][r] * d[c][r];
        }
#pragma unroll
        for (int c = 0; c < 4; ++c)
#pragma unroll
            for (int r = 0; r < 8; ++r) col[c][r] = d[c][r] + d[c][r + 8];
        float v[4];
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            const float x = fold8(col[c]), y = x + __shfl_xor(x, 32);
            v[c] = y + __shfl_xor(y, 16);
        }
        if (lane < NB) s_gain[wave][lane] = fold4(v);
        __syncthreads();
        if (t < NB) {
            const Block k = block(t);
            const int vx = s_vec[t][0], vy = s_vec[t][1];
            const long left = (long)k.ox + vx, top = (long)k.oy + vy, right = left + k.bw, bottom = top + k.bh;
            const long span_w = max(min(right, (long)W) - max(left, 0l), 0l);
            const long span_h = max(min(bottom, (long)H) - max(top, 0l), 0l);
            const float matched_px = (float)(span_w * span_h), block_px = (float)(k.bw * k.bh);
            const float zmean = s_gain[0][t] / block_px;
            const float zvar = s_gain[1][t] / block_px - zmean * zmean;
            const float safe = fmaxf(matched_px, 1.0f);
            const float vmean = s_gain[2][t] / safe;
            const float vvar = s_gain[3][t] / safe - vmean * vmean;
            const bool follows = (vx != 0 || vy != 0) && (matched_px == 0.0f || vvar <= kCompensationGainMax * zvar);
            const bool fits = left >= 0 && right <= W && top >= 0 && bottom <= H;
            s_follow[t] = follows && fits;
            s_matched[t] = !(follows && !fits);
        }
        __syncthreads();
    }
    // An unmatched block's record is zero; a followed block's residual and mean are along its vector.
    auto matched = [&](int i) { return !COMP || s_matched[i] != 0; };
    auto old_of = [&](int i) { return COMP && s_follow[i] ? s_mov : s_old; };
    auto residual = [&](const float *old, int at) {
        const float4 o = lds4(old + at);
        if constexpr (!COMP) return o;
        const float4 n = lds4(s_new + at);
        return make_float4(n.x - o.x, n.y - o.y, n.z - o.z, n.w - o.w);
    };
    auto mean = [&](const float *old, int at) {
        if constexpr (!COMP) return lds4(s_mov + at);
        const float4 n = lds4(s_new + at), o = lds4(old + at);
        return make_float4(0.5f * (n.x + o.x), 0.5f * (n.y + o.y), 0.5f * (n.z + o.z), 0.5f * (n.w + o.w));
    };

    // The ordered sums, spread over the waves and turned with the workgroup so that the longest is not
    // always on the same SIMD: sum_d and the textures, sum_d2, the lag-1 products, the quarters.
    const int role = (wave + (int)blockIdx.x) & 3;
    if (role < 3) {
        // The pixel-order totals (stats.rs:400-410), a lane per plane, each d times nothing, d or its
        // right neighbour (0 past the block; only channel 0's lag is kept).
        const int pl = lane & 15, i = pl / C, c = pl % C;
        const Block k = block(i);
        const bool whole = __all(k.bw == kTB);
        if (lane < 16) {
            const float *old = old_of(i);
            float total = 0.0f;
            auto rows = [&](auto &&add) {
#pragma unroll 1
                for (int r = 0; r < kTB * kTB; r += kTB) {
                    float d[kTB];
#pragma unroll
                    for (int g = 0; g < 4; ++g) {
                        const float4 v = residual(old, plane_at(pl, g) + r);
                        d[4 * g] = v.x, d[4 * g + 1] = v.y, d[4 * g + 2] = v.z, d[4 * g + 3] = v.w;
                    }
                    add(d);
                }
            };
            if (role == 0)
                rows([&](const float (&d)[kTB]) {
#pragma unroll
                    for (int x = 0; x < kTB; ++x) total += d[x];
                });
            else if (role == 1)
                rows([&](const float (&d)[kTB]) {
#pragma unroll
                    for (int x = 0; x < kTB; ++x) total += d[x] * d[x];
                });
            else if (whole)
                rows([&](const float (&d)[kTB]) {
#pragma unroll
                    for (int x = 0; x < kTB - 1; ++x) total += d[x] * d[x + 1];
                });
            else
                rows([&](const float (&d)[kTB]) {
#pragma unroll
                    for (int x = 0; x < kTB - 1; ++x) total += x + 1 < k.bw ? d[x] * d[x + 1] : 0.0f;
                });
            if (k.live && (role < 2 || c == 0))
                stats[(size_t)k.b * kRec + role * C + c] = matched(i) ? total : 0.0f;
        }
        if (role > 0) return;
    }
    // A lane per (quarter, plane): the sixteen lanes of a DPP row read one plane each.
    const int q = lane >> 4, qx = (q & 1) * kTQ, qy = (q >> 1) * kTQ, pl = lane & 15;
    if (role == 0) {
        // The quarter's four cell means (write_cell_means, stats.rs:606-624), then the texture over the
        // block's sixteen.
        const int i = pl / C, c = pl % C;
        const Block k = block(i);
        const float *left = s_new + plane_at(pl, 2 * (q & 1)) + qy * kTB, *right = s_new + plane_at(pl, 2 * (q & 1) + 1) + qy * kTB;
        float own[4], cells[16];
#pragma unroll
        for (int cell = 0; cell < 4; ++cell) {
            float sum = 0.0f;
#pragma unroll
            for (int dy = 0; dy < 4; ++dy) {
                const float4 v = lds4((cell & 1 ? right : left) + (4 * (cell >> 1) + dy) * kTB);
                sum = (((sum + v.x) + v.y) + v.z) + v.w;
            }
            own[cell] = sum / 16.0f;
        }
#pragma unroll
        for (int cell = 0; cell < 4; ++cell)
#pragma unroll
            for (int from = 0; from < 4; ++from)
                cells[(2 * (from >> 1) + (cell >> 1)) * 4 + 2 * (from & 1) + (cell & 1)] = __shfl(own[cell], 16 * from + pl);
        const float texture = cell_texture(cells, k.bw, k.bh);
        if (k.live && q == 0) {
            float *out = stats + (size_t)k.b * kRec;
            out[c == 0 ? 2 * C + 1 : 2 * C + 26 + c] = matched(i) ? texture : 0.0f;
            if (c == 0) out[2 * C + 2] = COMP && s_follow[i] ? 1.0f : 0.0f;
        }
    }
    // The flatness goes with the textures where their wave is the shorter one.
    constexpr int kFlatRole = COMP ? 3 : 0;
    const int i = min(pl, NB - 1);
    const Block k = block(i);
    const bool write = k.live && pl < NB;
    float *quarter = stats + (size_t)k.b * kRec + 2 * C + 3 + 6 * q;
    if constexpr (!LUMA) {
        if (write && role == 3) {
#pragma unroll
            for (int f = 0; f < 6; ++f) quarter[f] = 0.0f;
        }
        return;
    }
    const float *old = old_of(i);
    const int half_at[2] = {plane_at(i * C, 2 * (q & 1)) + qy * kTB, plane_at(i * C, 2 * (q & 1) + 1) + qy * kTB};
    if (role == kFlatRole) {
        // Flatness (stats.rs:520-585): the quarter's 4x4 grid of 2x2 means of the temporal mean, each
        // cell's squared steps to its right and lower neighbour, a halving tree over the 16 cells, over
        // 24 pairs.
        float grid[4][4], e[4][4];
#pragma unroll
        for (int gy = 0; gy < 4; ++gy)
#pragma unroll
            for (int half = 0; half < 2; ++half) {
                const int at = half_at[half] + 2 * gy * kTB;
                const float4 a = mean(old, at), b = mean(old, at + kTB);
                grid[gy][2 * half] = (((a.x + a.y) + b.x) + b.y) / 4.0f;
                grid[gy][2 * half + 1] = (((a.z + a.w) + b.z) + b.w) / 4.0f;
            }
#pragma unroll
        for (int gy = 0; gy < 4; ++gy)
#pragma unroll
            for (int gx = 0; gx < 4; ++gx) {
                const float right = grid[gy][gx] - grid[gy][min(gx + 1, 3)], below = grid[gy][gx] - grid[min(gy + 1, 3)][gx];
                float v = 0.0f;
                if (gx < 3) v += right * right;
                if (gy < 3) v += below * below;
                e[gy][gx] = v;
            }
        float col[4];
#pragma unroll
        for (int gx = 0; gx < 4; ++gx) col[gx] = (e[0][gx] + e[2][gx]) + (e[1][gx] + e[3][gx]);
        const bool full = k.bw >= qx + kTQ && k.bh >= qy + kTQ;
        if (write) quarter[3] = !matched(i) ? 0.0f : full ? fold4(col) / 24.0f : kUnmeasuredFlatness;
    }
    if (role != 3) return;
    // The quarter's luma, sum_d and sum_d2 trees and its extremes over the pixels in the frame, four
    // columns at a time (columns c and c + 4 are the tree's first pairs).  The extremes start from NaN,
    // which any value replaces, so that a quarter of values past +-1e30 keeps its own and one of NaNs alone
    // is NaN; a pixel past the frame is +-1e30.
    float luma[4], sum_d[4], sum_d2[4], lo = __builtin_nanf(""), hi = lo;
#pragma unroll 1
    for (int half = 0; half < 2; ++half) {
        float n[4][8], d[4][8], d2[4][8];
        const int inside = k.bw - qx - 4 * half;  // columns of the four in the frame
#pragma unroll
        for (int r = 0; r < kTQ; ++r) {
            const int at = (half ? half_at[1] : half_at[0]) + r * kTB;
            const float4 a = lds4(s_new + at), b = residual(old, at);
            n[0][r] = a.x, n[1][r] = a.y, n[2][r] = a.z, n[3][r] = a.w;
            d[0][r] = b.x, d[1][r] = b.y, d[2][r] = b.z, d[3][r] = b.w;
#pragma unroll
            for (int c = 0; c < 4; ++c) d2[c][r] = d[c][r] * d[c][r];
        }
        if (__all(inside >= 4 && k.bh - qy >= kTQ)) {
#pragma unroll
            for (int r = 0; r < kTQ; ++r)
#pragma unroll
                for (int c = 0; c < 4; ++c) {
                    lo = min_f(lo, n[c][r]);
                    hi = max_f(hi, n[c][r]);
                }
        } else {
#pragma unroll
            for (int r = 0; r < kTQ; ++r)
#pragma unroll
                for (int c = 0; c < 4; ++c) {
                    const bool in = c < inside && qy + r < k.bh;
                    lo = min_f(lo, in ? n[c][r] : 1.0e30f);
                    hi = max_f(hi, in ? n[c][r] : -1.0e30f);
                }
        }
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            const float l = fold8(n[c]), s1 = fold8(d[c]), s2 = fold8(d2[c]);
            luma[c] = half ? luma[c] + l : l;
            sum_d[c] = half ? sum_d[c] + s1 : s1;
            sum_d2[c] = half ? sum_d2[c] + s2 : s2;
        }
    }
    if (write) {
        const bool m = matched(i);
        quarter[0] = m ? fold4(sum_d) : 0.0f;
        quarter[1] = m ? fold4(sum_d2) : 0.0f;
        quarter[2] = m ? fold4(luma) : 0.0f;
        quarter[4] = m ? lo : 0.0f;
        quarter[5] = m ? hi : 0.0f;
    }
}

// The same records a workgroup per block, thread t on pixel (t % 16, t / 16), for frames of few blocks: the
// samples take one round of loads, and after one barrier the four waves split the sums (wave 0 the pixel-order
// totals, wave 1 the textures, wave 2 the flatness grid, wave 3 the quarters; the first two steps of a
// 256-slot tree go through LDS, the rest are wave shuffles, which pair the same slots).  Bound by that chain,
// launch to last store, as every block runs at once.
constexpr int kTLaneStride = kTThreads + 1;  // lane-major totals: lanes land in different banks

__device__ __forceinline__ float tree_wave(float v)
{
#pragma unroll
    for (int stride = 32; stride >= 1; stride >>= 1) v += __shfl_down(v, stride);
    return v;
}

template <int C, bool LUMA, bool COMP>
__global__ __launch_bounds__(kTThreads) void k_temporal_small(const float *__restrict__ ring, float *__restrict__ stats,
                                                              const int32_t *__restrict__ mv, uint32_t slot_new,
                                                              uint32_t slot_prev, uint32_t mv_offset, uint32_t mv_step,
                                                              uint32_t mv_bx, uint32_t mv_by, int W, int H)
{
    constexpr int kLanes = 2 * C + 1, kRec = 3 * C + 26;
    __shared__ float s_lane[kLanes * kTLaneStride];
    __shared__ float s_val[C * kTThreads];                    // the new frame's values per channel
    __shared__ float s_quarter[LUMA ? 5 * kTThreads : 1];     // quarter-major: sum, d, d2, min, max
    __shared__ float s_mean[LUMA ? kTThreads : 1];            // the temporal mean of channel 0
    __shared__ float s_cells[C * 16];
    __shared__ float s_gain[COMP ? 4 * kTThreads : 1];
    __shared__ int s_shift[3];

    const int t = (int)threadIdx.x, lane = t & 63, wave = t >> 6, lx = t & (kTB - 1), ly = t >> 4;
    // Workgroups reach the eight XCDs round robin; XCD x takes a contiguous run of the row-major
    // blocks, so the two blocks sharing a 128-byte row segment meet in one L2.
    const uint32_t nbx = ((uint32_t)W + kTB - 1) / kTB, blocks = nbx * (((uint32_t)H + kTB - 1) / kTB);
    const uint32_t xcd = blockIdx.x % kXcds, per = blocks / kXcds, extra = blocks % kXcds;
    const uint32_t b = xcd * per + min(xcd, extra) + blockIdx.x / kXcds;
    const int ox = (int)(b % nbx) * kTB, oy = (int)(b / nbx) * kTB;
    const int bw = min(kTB, W - ox), bh = min(kTB, H - oy);
    const int x = ox + lx, y = oy + ly;
    const bool in_frame = x < W && y < H;
    const size_t plane = (size_t)W * H * C;
    const float *fn = ring + (size_t)slot_new * plane, *fp = ring + (size_t)slot_prev * plane;
    float *out = stats + (size_t)b * kRec;

    float nv[C], pv[C];
#pragma unroll
    for (int c = 0; c < C; ++c) nv[c] = pv[c] = 0.0f;
    if (in_frame) {
        const size_t at = ((size_t)y * W + x) * C;
#pragma unroll
        for (int c = 0; c < C; ++c) {
            nv[c] = fn[at + c];
            pv[c] = fp[at + c];
        }
    }

    int sx = 0, sy = 0;
    bool matched = true;
    float moved = 0.0f;
    if constexpr (COMP) {
        // The gain check (stats.rs:257-341): the block follows its vector when channel 0's residual
        // variance along it, over the pixels whose match stays in the frame, is at most half the
        // zero-vector variance, or when no match stays in the frame; a followed block whose shifted
        // extent leaves the frame is unmatched and writes zeros.
        const uint32_t col = min((uint32_t)ox / mv_step, mv_bx - 1), row = min((uint32_t)oy / mv_step, mv_by - 1);
        const int32_t *v = mv + mv_offset + (size_t)(row * mv_bx + col) * 2;
        const int vx = v[0], vy = v[1];
        float zr = 0.0f, vr = 0.0f;
        if (in_frame) {
            zr = nv[0] - pv[0];
            const long mx = (long)x + vx, my = (long)y + vy;
            if (mx >= 0 && mx < W && my >= 0 && my < H) vr = nv[0] - fp[((size_t)my * W + (size_t)mx) * C];
        }
        s_gain[t] = zr;
        s_gain[kTThreads + t] = zr * zr;
        s_gain[2 * kTThreads + t] = vr;
        s_gain[3 * kTThreads + t] = vr * vr;
        __syncthreads();
        if (wave == 0) {
            float sums[4];
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                const float *r = s_gain + k * kTThreads;
                sums[k] = tree_wave((r[lane] + r[lane + 128]) + (r[lane + 64] + r[lane + 192]));
            }
            if (lane == 0) {
                const long left = (long)ox + vx, top = (long)oy + vy, right = left + bw, bottom = top + bh;
                const long span_w = max(min(right, (long)W) - max(left, 0l), 0l);
                const long span_h = max(min(bottom, (long)H) - max(top, 0l), 0l);
                const float matched_px = (float)(span_w * span_h), block_px = (float)(bw * bh);
                const float zmean = sums[0] / block_px;
                const float zvar = sums[1] / block_px - zmean * zmean;
                const float safe = fmaxf(matched_px, 1.0f);
                const float vmean = sums[2] / safe;
                const float vvar = sums[3] / safe - vmean * vmean;
                const bool follows = (vx != 0 || vy != 0) && (matched_px == 0.0f || vvar <= kCompensationGainMax * zvar);
                const bool fits = left >= 0 && right <= W && top >= 0 && bottom <= H;
                s_shift[0] = follows ? vx : 0;
                s_shift[1] = follows ? vy : 0;
                s_shift[2] = follows && !fits ? 0 : 1;
            }
        }
        __syncthreads();
        sx = s_shift[0];
        sy = s_shift[1];
        matched = s_shift[2] != 0;
        moved = (sx != 0 || sy != 0) && matched ? 1.0f : 0.0f;
        if ((sx != 0 || sy != 0) && matched && in_frame) {
            const size_t at = ((size_t)(y + sy) * W + (x + sx)) * C;
#pragma unroll
            for (int c = 0; c < C; ++c) pv[c] = fp[at + c];
        }
    }

    const bool valid = in_frame && matched;
    float res[C];
#pragma unroll
    for (int c = 0; c < C; ++c) {
        res[c] = valid ? nv[c] - pv[c] : 0.0f;
        s_lane[c * kTLaneStride + t] = res[c];
        s_lane[(C + c) * kTLaneStride + t] = res[c] * res[c];
        s_val[c * kTThreads + t] = valid ? nv[c] : 0.0f;
    }
    // Pixel t + 1 is the row neighbour in the same wave whenever the pair lies inside the block.
    const float next = __shfl_down(res[0], 1);
    s_lane[2 * C * kTLaneStride + t] = valid && lx + 1 < bw ? res[0] * next : 0.0f;
    if constexpr (LUMA) {
        const int slot = ((ly >> 3) * 2 + (lx >> 3)) * 64 + (ly & 7) * 8 + (lx & 7);
        s_quarter[slot] = valid ? nv[0] : 0.0f;
        s_quarter[kTThreads + slot] = res[0];
        s_quarter[2 * kTThreads + slot] = res[0] * res[0];
        s_quarter[3 * kTThreads + slot] = valid ? nv[0] : 1.0e30f;
        s_quarter[4 * kTThreads + slot] = valid ? nv[0] : -1.0e30f;
        s_mean[t] = valid ? 0.5f * (nv[0] + pv[0]) : 0.0f;
    }
    __syncthreads();

    if (wave == 0) {
        // Lane totals (stats.rs:400-410): one lane per record lane adds the 256 pixels in order.
        if (lane < kLanes) {
            const float *v = s_lane + lane * kTLaneStride;
            float total = 0.0f;
#pragma unroll 32
            for (int k = 0; k < kTThreads; ++k) total += v[k];
            out[lane] = total;
        }
    } else if (wave == 1) {
        // Cell means of each channel (write_cell_means, stats.rs:606-624), then the textures.
        if (lane < 16 * C) {
            const int c = lane >> 4, cell = lane & 15, cx = cell & 3, cy = cell >> 2;
            const float *v = s_val + c * kTThreads;
            float sum = 0.0f;
#pragma unroll
            for (int dy = 0; dy < 4; ++dy)
#pragma unroll
                for (int dx = 0; dx < 4; ++dx) sum += v[(4 * cy + dy) * kTB + 4 * cx + dx];
            s_cells[lane] = sum / 16.0f;
        }
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        if (lane < C) {
            float cells[16];
#pragma unroll
            for (int i = 0; i < 16; ++i) cells[i] = s_cells[16 * lane + i];
            const float texture = cell_texture(cells, bw, bh);
            out[lane == 0 ? 2 * C + 1 : 2 * C + 26 + lane] = texture;
        }
        if (lane == 0) out[2 * C + 2] = moved;
    } else if (wave == 2) {
        float *flat = out + 2 * C + 3 + 3;
        if constexpr (LUMA) {
            // Flatness (stats.rs:520-585): the 8x8 grid of 2x2 means of the temporal mean, each
            // cell's squared steps to its right and lower neighbour inside its quarter, then per
            // quarter a halving tree over its 16 cells (stored quarter-major) over 24 pairs.
            const int gx = lane & 7, gy = lane >> 3;
            float cell = 0.0f;
#pragma unroll
            for (int dy = 0; dy < 2; ++dy)
#pragma unroll
                for (int dx = 0; dx < 2; ++dx) cell += s_mean[(2 * gy + dy) * kTB + 2 * gx + dx];
            cell = cell / 4.0f;
            const float right = __shfl_down(cell, 1), below = __shfl_down(cell, 8);
            float e = 0.0f;
            if ((gx & 3) != 3) e += (cell - right) * (cell - right);
            if ((gy & 3) != 3) e += (cell - below) * (cell - below);
            // Reorder the scores quarter-major: slot q * 16 + (gy % 4) * 4 + gx % 4.
            const int dest = ((gy >> 2) * 2 + (gx >> 2)) * 16 + (gy & 3) * 4 + (gx & 3);
            float q = __builtin_bit_cast(float, __builtin_amdgcn_ds_permute(dest * 4, __builtin_bit_cast(int, e)));
#pragma unroll
            for (int stride = 8; stride >= 1; stride >>= 1) q += __shfl_down(q, stride);
            if ((lane & 15) == 0) {
                const int quarter = lane >> 4;
                const bool full = bw >= ((quarter & 1) + 1) * 8 && bh >= ((quarter >> 1) + 1) * 8;
                flat[quarter * 6] = !matched ? 0.0f : full ? q / 24.0f : kUnmeasuredFlatness;
            }
        } else {
            if (lane < 4) flat[lane * 6] = 0.0f;
        }
    } else {
        float *quarters = out + 2 * C + 3;
        if constexpr (LUMA) {
#pragma unroll
            for (int quarter = 0; quarter < 4; ++quarter) {
                const float *qv = s_quarter + quarter * 64 + lane;
                const float luma = tree_wave(qv[0]);
                const float d = tree_wave(qv[kTThreads]);
                const float d2 = tree_wave(qv[2 * kTThreads]);
                float lo = qv[3 * kTThreads], hi = qv[4 * kTThreads];
#pragma unroll
                for (int stride = 32; stride >= 1; stride >>= 1) {
                    lo = fminf(lo, __shfl_xor(lo, stride));
                    hi = fmaxf(hi, __shfl_xor(hi, stride));
                }
                if (lane == 0) {
                    float *f = quarters + quarter * 6;
                    f[0] = matched ? d : 0.0f;
                    f[1] = matched ? d2 : 0.0f;
                    f[2] = matched ? luma : 0.0f;
                    f[4] = matched ? lo : 0.0f;
                    f[5] = matched ? hi : 0.0f;
                }
            }
        } else {
            if (lane < 24 && lane % 6 != 3) quarters[lane] = 0.0f;
        }
    }
}

__global__ void k_temporal_zero(float *__restrict__ dst, uint32_t len)
{
    for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < len; i += gridDim.x * blockDim.x) dst[i] = 0.0f;
}

template <int C, bool LUMA>
void launch_temporal_typed(uint32_t blocks, hipStream_t s, const float *ring, float *stats, const int32_t *mv,
                           uint32_t slot_new, uint32_t slot_prev, uint32_t mv_offset, uint32_t mv_step, uint32_t mv_bx,
                           uint32_t mv_by, int W, int H)
{
    // A workgroup per block while its chain costs less than the sixteen-plane one's: up to four workgroups per
    // CU, five with motion, where the latter's checks are the longer ones.  One channel, us by block / by
    // sixteen planes: 640x400 (1000 blocks) 5.8 / 6.0, 7.3 / 8.9 with motion; 640x480 (1200) 6.7 / 6.0, 8.3 /
    // 8.9; 768x432 (1296) 7.4 / 6.0, 8.9 / 8.9; 720x576 (1620) 8.1 / 6.1, 9.8 / 9.0; two channels the same.
    const bool small = blocks <= (mv ? 5u : 4u) * 256u;
    const dim3 grid(small ? blocks : div_up(blocks, 16 / C));
    auto launch = [&](auto kernel) {
        kernel<<<grid, kTThreads, 0, s>>>(ring, stats, mv, slot_new, slot_prev, mv_offset, mv_step, mv_bx, mv_by, W, H);
    };
    if (mv) launch(small ? k_temporal_small<C, LUMA, true> : k_temporal_stats<C, LUMA, true>);
    else launch(small ? k_temporal_small<C, LUMA, false> : k_temporal_stats<C, LUMA, false>);
}

}  // namespace

uint32_t temporal_stats_len(uint32_t width, uint32_t height, uint32_t channels)
{
    return ((width + kTB - 1) / kTB) * ((height + kTB - 1) / kTB) * (3 * channels + 26);
}

hipError_t launch_temporal_stats(const float *ring, uint32_t width, uint32_t height, uint32_t channels,
                                 uint32_t slot_new, uint32_t slot_prev, const int32_t *mv, uint32_t mv_offset,
                                 uint32_t mv_step, uint32_t mv_bx, uint32_t mv_by, bool luma_fields, float *stats,
                                 hipStream_t s)
{
    if (!ring || !stats || width == 0 || height == 0 || width > (1u << 20) || height > (1u << 20) ||
        (channels != 1 && channels != 2) || (mv && (mv_step == 0 || mv_bx == 0 || mv_by == 0)) ||
        (uint64_t)((width + kTB - 1) / kTB) * ((height + kTB - 1) / kTB) * (3 * channels + 26) > 0xFFFFFFFFull)
        return hipErrorInvalidValue;
    const uint32_t blocks = ((width + kTB - 1) / kTB) * ((height + kTB - 1) / kTB);
    const int W = (int)width, H = (int)height;
    if (channels == 1) {
        if (luma_fields) launch_temporal_typed<1, true>(blocks, s, ring, stats, mv, slot_new, slot_prev, mv_offset, mv_step, mv_bx, mv_by, W, H);
        else launch_temporal_typed<1, false>(blocks, s, ring, stats, mv, slot_new, slot_prev, mv_offset, mv_step, mv_bx, mv_by, W, H);
    } else {
        if (luma_fields) launch_temporal_typed<2, true>(blocks, s, ring, stats, mv, slot_new, slot_prev, mv_offset, mv_step, mv_bx, mv_by, W, H);
        else launch_temporal_typed<2, false>(blocks, s, ring, stats, mv, slot_new, slot_prev, mv_offset, mv_step, mv_bx, mv_by, W, H);
    }
    return hipGetLastError();
}

hipError_t launch_temporal_zero(float *stats, uint32_t len, hipStream_t s)
{
    if (!stats) return hipErrorInvalidValue;
    if (len == 0) return hipSuccess;
    const uint32_t blocks = std::min<uint32_t>((len + 255) / 256, 4096);
    k_temporal_zero<<<blocks, 256, 0, s>>>(stats, len);
    return hipGetLastError();
}

}  // namespace avd
