// NLMeans window kernels for gfx950.
//
// Semantics follow nlmeans/kernels/fused.rs: nlm_fused_single_window (:364-530) walks every
// offset q != 0 of the (2s+1)^2 window of a frame against itself; nlm_fused_pair_accumulate_window
// (:138-347) walks every q of one temporal pair, the forward frame at +q and the backward frame at
// -q.  Per offset the per-pixel distance is sum_c (x - y)^2 * scale (3 luma, 1.5 chroma) with
// clamp-to-edge reads, the patch distance is its (2P+1)^2 box sum, the weight is
// exp(-max(D - offset, 0) * h2) (times the block confidence on a pair), and each pixel gathers
// sum(w * y), sum(w) and max(w) in registers, added to the accumulators once.  nlm_finish
// (accumulate.rs:54-101) then blends in the centre with self_weight * max_w.
//
// MI355X layout.  The lanes of a wavefront are 64 adjacent distance rows and each lane walks COLS
// output columns, so the horizontal box sum runs in the lane's registers (2P fused multiply-adds that
// also apply the channel scale) and the vertical one is a chain of 2P v_add_f32 whose shifted operand
// is a DPP wave_shr:1 (lane l then holds the sum of rows l - 2P .. l, added top to bottom; lanes from
// 2P on own an output row).  Lanes on columns instead, the sums the other way round, cost two
// instructions per horizontal step, since no fused multiply-add takes a DPP operand as its addend, and
// recompute a 2P-row halo of them per COLS rows.  The neighbour frame(s) of the workgroup are staged
// in LDS with their (P + s) halo at an odd row pitch (64 lanes on 64 rows then hit distinct banks, and
// a lane's columns are immediate offsets), so the offset loop runs with no barrier.  COLS (8, 4 or 2)
// trades the 2P halo columns each lane recomputes (differences only) against the number of waves a
// small frame spreads over; every choice gives bit-identical sums, and the tuner picks one per window
// shape.  On planes up to 2^20 pixels each tile's offsets are split over SPLIT waves whose sums add in
// part order.  The sums leave through LDS, so global accumulators are read and written along rows.
// Bound by vector instruction issue: per pixel and offset about 2 (1 + 2P / COLS) for the differences,
// 4P + 1 for the box sums and 10 for the weight and the sums.  A wave's f32 add, subtract, multiply or
// multiply-add issues in about 2.3 cycles, a max or a DPP add in four, v_exp_f32 in eight (measured): 62
// cycles at P 2 and four columns, 77 at P 3.  Against lanes on columns (one pair or window of one frame,
// same sums): 640x360 P 2 S 7 81 -> 42 us (22 of issue: two waves per SIMD leave latency in the open),
// 1920x1080 P 3 S 4 pair 541 -> 266 us (185 of issue), P 4 S 2 pair with confidence 276 -> 120 us,
// two-channel 960x540 P 3 S 4 pair 300 -> 113 us.
// exp is v_exp_f32 (exp2) with log2(e) folded into h2 on the host.
#include <algorithm>

#include "common.h"

namespace avd {

namespace {

constexpr int kMaxP = 8;
constexpr int kMaxS = 8;

// Lane l reads lane l - 1; lane 0 reads 0.
__device__ __forceinline__ float wave_shr1(float v)
{
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x138, 0xf, 0xf, true));
}

__device__ __forceinline__ int clampi(int v, int hi) { return v < 0 ? 0 : (v > hi ? hi : v); }

// Shape of a workgroup: WX waves side by side, COLS output columns each, by SPLIT offset parts; its
// tile is 64 - 2P output rows high.
template <int C, int P, int COLS, int WX, int SPLIT>
struct Shape {
    static constexpr int kWidth = WX * COLS;         // output columns
    static constexpr int kRows = 64 - 2 * P;         // output rows
    static constexpr int kThreads = WX * SPLIT * 64;
    static constexpr int kDist = COLS + 2 * P;       // distance columns of a lane
    // Output elements a thread finishes: of the 64 x kWidth grid, element t + k kThreads.
    static constexpr int kElems = (64 * kWidth + kThreads - 1) / kThreads;
    // Lanes that stage one tile row: at least its columns at the largest search radius.
    static constexpr int kStage = kWidth + 2 * P + 2 * kMaxS <= 32 ? 32 : 64;
    static_assert(kWidth + 2 * P + 2 * kMaxS <= 64, "a tile row is staged by at most 64 lanes");
};

// Tile rows of a grid layer; taller frames take further layers along z, as a grid's y extent is limited to
// 16 bits (three million frame rows at patch radius 8).  The last layer's surplus tiles write nothing.
constexpr uint32_t kGridRows = 1u << 15;
inline dim3 tile_grid(uint32_t columns, uint32_t rows)
{
    return dim3(columns, std::min(rows, kGridRows), div_up(rows, kGridRows));
}

// Samples between rows of a staged tile: odd, so that lanes on consecutive rows fall on distinct banks.
__host__ __device__ inline int tile_pitch(int width, int P, int S) { return (width + 2 * P + 2 * S) | 1; }

// Loads the clamped (rows x cols) window of an interleaved frame from (x0, y0) into LDS, LANES lanes
// to a row and four rows of loads in flight.
template <int C, int THREADS, int LANES>
__device__ __forceinline__ void stage_tile(float *tile, const float *__restrict__ frame, int W, int H, int x0, int y0,
                                           int cols, int rows, int pitch)
{
    constexpr int kStep = THREADS / LANES, kBatch = 4;
    const int tx = threadIdx.x % LANES, first = threadIdx.x / LANES;
    const float *column = frame + (size_t)clampi(x0 + tx, W - 1) * C;
    for (int r = first; r < rows; r += kStep * kBatch) {
        float v[kBatch][C];
#pragma unroll
        for (int u = 0; u < kBatch; ++u) {
            const float *src = column + (size_t)clampi(y0 + min(r + u * kStep, rows - 1), H - 1) * W * C;
#pragma unroll
            for (int c = 0; c < C; ++c) v[u][c] = src[c];
        }
#pragma unroll
        for (int u = 0; u < kBatch; ++u) {
            const int row = r + u * kStep;
            if (row < rows && tx < cols) {
#pragma unroll
                for (int c = 0; c < C; ++c) tile[((size_t)row * pitch + tx) * C + c] = v[u][c];
            }
        }
    }
}

// The weights of this lane's COLS output pixels at one offset: the distances of row `nb` (the staged
// row of this lane at the offset) to `cen`, their (2P+1)^2 box sums and the exponential.  Every
// operation is spelled out (no contraction): the sums of all launch forms and tile shapes are the same.
template <int C, int P, int COLS>
__device__ __forceinline__ void offset_weights(const float *nb, const float (&cen)[COLS + 2 * P][C], float scale,
                                               float off, float h2l, float (&weight)[COLS])
{
#pragma clang fp contract(off)
    float sq[COLS + 2 * P];
#pragma unroll
    for (int i = 0; i < COLS + 2 * P; ++i) {
        const float e0 = cen[i][0] - nb[i * C];
        if constexpr (C == 1) {
            sq[i] = e0 * e0;
        } else {
            const float e1 = cen[i][1] - nb[i * C + 1];
            sq[i] = fmaf(e0, e0, e1 * e1);
        }
    }
    float h[COLS], d[COLS];
#pragma unroll
    for (int j = 0; j < COLS; ++j) {
        float a = scale * sq[j];
#pragma unroll
        for (int k = 1; k <= 2 * P; ++k) a = fmaf(scale, sq[j + k], a);
        h[j] = a;
        d[j] = a;
    }
    // Step by step over all columns, so that a DPP read never follows the write of its operand at once.
#pragma unroll
    for (int k = 0; k < 2 * P; ++k)
#pragma unroll
        for (int j = 0; j < COLS; ++j) d[j] = wave_shr1(d[j]) + h[j];
#pragma unroll
    for (int j = 0; j < COLS; ++j) weight[j] = __builtin_amdgcn_exp2f(-fmaxf(d[j] - off, 0.0f) * h2l);
}

// The offset loop of one window for this lane's COLS output pixels, into acc / ws / mw (zeroed here):
// every offset q (q != 0 for a single window) against the staged tile `tf` (the forward frame of a
// pair, or the frame itself) and, for a pair, `tb` (the backward frame at -q).  `cen` holds the lane's
// centre row of COLS + 2P distance columns.
template <int C, int P, int COLS, bool PAIR, bool CONF, int SPLIT>
__device__ __forceinline__ void window_sums(const NlmWindow &w, const float *tf, const float *tb, int pitch, int wave,
                                            int lane, int part, const float (&cen)[COLS + 2 * P][C],
                                            const float *__restrict__ lut, const float (&conf_fv)[COLS],
                                            const float (&conf_bv)[COLS], float (&acc)[COLS][C], float (&ws)[COLS],
                                            float (&mw)[COLS])
{
#pragma clang fp contract(off)
    const int S = w.S, side = 2 * S + 1;
    float scale = (C == 1) ? 3.0f : 1.5f;
    asm("" : "+s"(scale));  // in a register: a literal would double the size of every multiply-add
    const float h2l = w.h2_log2e;
#pragma unroll
    for (int j = 0; j < COLS; ++j) {
#pragma unroll
        for (int c = 0; c < C; ++c) acc[j][c] = 0.0f;
        ws[j] = 0.0f;
        mw[j] = 0.0f;
    }
    // Sample of this lane's first distance column, and of its first output pixel (the distance row P
    // above, P columns on), at offset 0; lanes below 2P own no output and read rows inside the tile.
    const int dist0 = (lane + S) * pitch + wave * COLS + S;
    const int gather0 = (max(lane, P) - P + S) * pitch + wave * COLS + P + S;
    // This wave's share of the offsets: the rows qy of part `part` of SPLIT consecutive runs of
    // offset rows.
    const int qy_lo = -S + part * side / SPLIT, qy_hi = -S + (part + 1) * side / SPLIT;
    for (int qy = qy_lo; qy < qy_hi; ++qy) {
        for (int qx = -S; qx <= S; ++qx) {
            if (!PAIR && qx == 0 && qy == 0) continue;
            const float off = PAIR ? w.offset : lut[(qy + S) * side + (qx + S)];
            const int q = qy * pitch + qx;
            float wf[COLS];
            offset_weights<C, P, COLS>(tf + (size_t)(dist0 + q) * C, cen, scale, off, h2l, wf);
            const float *gf = tf + (size_t)(gather0 + q) * C;
            if constexpr (PAIR) {
                float wb[COLS];
                offset_weights<C, P, COLS>(tb + (size_t)(dist0 - q) * C, cen, scale, off, h2l, wb);
                const float *gb = tb + (size_t)(gather0 - q) * C;
#pragma unroll
                for (int j = 0; j < COLS; ++j) {
                    float cf = wf[j], cb = wb[j], both;
                    if constexpr (CONF) {
                        cf = wf[j] * conf_fv[j];
                        cb = wb[j] * conf_bv[j];
                        both = fmaf(conf_fv[j], wf[j], cb);
                    } else {
                        both = cf + cb;
                    }
#pragma unroll
                    for (int c = 0; c < C; ++c)
                        acc[j][c] = fmaf(gb[j * C + c], cb, fmaf(gf[j * C + c], cf, acc[j][c]));
                    ws[j] += both;
                    mw[j] = fmaxf(mw[j], fmaxf(cf, cb));
                }
            } else {
#pragma unroll
                for (int j = 0; j < COLS; ++j) {
#pragma unroll
                    for (int c = 0; c < C; ++c) acc[j][c] = fmaf(gf[j * C + c], wf[j], acc[j][c]);
                    ws[j] += wf[j];
                    mw[j] = fmaxf(mw[j], wf[j]);
                }
            }
        }
    }
}

// Hands the window sums from the lanes that walked them to the threads that finish them: each field
// (the C channel sums, the weight sum, the largest weight) passes through `red`, LDS of SPLIT x 64 x
// (kWidth + 1) floats (the tiles are done with, so the caller passes their memory), and element k of
// a thread is pixel (t + k kThreads) of the 64 x kWidth grid, its parts joined in part order.  Every
// thread of the workgroup calls it.
template <int C, int P, int COLS, int WX, int SPLIT>
__device__ __forceinline__ void join_parts(float *red, int wave, int lane, int part, const float (&acc)[COLS][C],
                                           const float (&ws)[COLS], const float (&mw)[COLS],
                                           float (&out)[Shape<C, P, COLS, WX, SPLIT>::kElems][C + 2])
{
    using T = Shape<C, P, COLS, WX, SPLIT>;
    constexpr int kPitch = T::kWidth + 1, kPart = 64 * kPitch;
#pragma unroll
    for (int f = 0; f < C + 2; ++f) {
        __syncthreads();  // every wave is done with the tiles, or with the last field
        float *dst = red + part * kPart + lane * kPitch + wave * COLS;
#pragma unroll
        for (int j = 0; j < COLS; ++j) dst[j] = f < C ? acc[j][f < C ? f : 0] : (f == C ? ws[j] : mw[j]);
        __syncthreads();
#pragma unroll
        for (int k = 0; k < T::kElems; ++k) {
            const int e = min((int)threadIdx.x + k * T::kThreads, 64 * T::kWidth - 1);
            const float *src = red + (e / T::kWidth) * kPitch + e % T::kWidth;
            float v = src[0];
#pragma unroll
            for (int p = 1; p < SPLIT; ++p) v = f <= C ? v + src[p * kPart] : fmaxf(v, src[p * kPart]);
            out[k][f] = v;
        }
    }
}

// The pixel of element k of this thread, or false where it lies outside the tile's outputs.
template <int P, typename T>
__device__ __forceinline__ bool element_pixel(int k, int X0, int Y0, int W, int H, size_t &p)
{
    const int e = (int)threadIdx.x + k * T::kThreads, row = e / T::kWidth;
    const int ox = X0 + e % T::kWidth, oy = Y0 - 2 * P + row;
    p = (size_t)oy * W + ox;
    return row >= 2 * P && row < 64 && ox < W && oy < H;
}

// The centre samples of this lane's distance row from the staged centre tile.
template <int C, int P, int COLS>
__device__ __forceinline__ void read_centre(const float *tile, int pitch, int S, int wave, int lane,
                                            float (&cen)[COLS + 2 * P][C])
{
    const float *src = tile + (size_t)((lane + S) * pitch + wave * COLS + S) * C;
#pragma unroll
    for (int i = 0; i < COLS + 2 * P; ++i)
#pragma unroll
        for (int c = 0; c < C; ++c) cen[i][c] = src[i * C + c];
}

// The confidence of the blocks this lane's output pixels fall in.
template <int COLS>
__device__ __forceinline__ void load_conf(const NlmWindow &w, const float *__restrict__ conf, int ox, int oy,
                                          float (&out)[COLS])
{
    const float *row = conf + (size_t)min(clampi(oy, w.H - 1) / w.step, w.blocks_y - 1) * w.blocks_x;
#pragma unroll
    for (int j = 0; j < COLS; ++j) out[j] = row[min(clampi(ox + j, w.W - 1) / w.step, w.blocks_x - 1)];
}

// The finish of one pixel (accumulate.rs:54-101): the centre joins with self_weight times the largest
// weight, or stands alone where every weight vanished.
template <int C>
__device__ __forceinline__ void finish_pixel(const float *frame, const float *accum, float wsum, float maxw,
                                             float self_weight, float *out)
{
#pragma clang fp contract(off)
    const float sw = self_weight * maxw, den = fmaf(self_weight, maxw, wsum);
    if (den > 1e-30f) {
        const float inv = 1.0f / den;
#pragma unroll
        for (int c = 0; c < C; ++c) out[c] = fmaf(frame[c], sw, accum[c]) * inv;
    } else {
#pragma unroll
        for (int c = 0; c < C; ++c) out[c] = frame[c];
    }
}

// One window of a frame.  Its sums add to the accumulators, or start them (`fresh`); a single window
// with `out` is the frame's last and finishes it instead of storing the sums, so a frame's windows run
// with no launch to clear the accumulators and none to finish (1920x1080 4:2:0 HQ base, ten fills and
// two finishes fewer: 429 -> 407 us per frame; 10-bit temporal radius 2: 804 -> 781 us).
template <int C, int P, int COLS, int WX, bool PAIR, bool CONF, int SPLIT>
__global__ __launch_bounds__(WX * SPLIT * 64) void k_nlm(NlmWindow w, const float *__restrict__ centre,
                                                             const float *__restrict__ fwd, const float *__restrict__ bwd,
                                                             const float *__restrict__ lut,
                                                             const float *__restrict__ conf_f,
                                                             const float *__restrict__ conf_b, float *__restrict__ accum,
                                                             float *__restrict__ wsum, float *__restrict__ maxw,
                                                             bool fresh, float self_weight, float *__restrict__ out)
{
    using T = Shape<C, P, COLS, WX, SPLIT>;
    extern __shared__ float lds[];
    const int S = w.S, W = w.W, H = w.H;
    // Wave (wave, part): column run `wave` of the workgroup's WX, offset part `part` of SPLIT.
    const int lane = threadIdx.x & 63, id = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int wave = id % WX, part = id / WX;
    const int X0 = blockIdx.x * T::kWidth, Y0 = (int)(blockIdx.z * kGridRows + blockIdx.y) * T::kRows;

    // Tiles: columns X0-P-S .. X0+kWidth+P-1+S, rows Y0-P-S .. Y0+63-P+S.
    const int tcols = T::kWidth + 2 * P + 2 * S, trows = 64 + 2 * S, pitch = tile_pitch(T::kWidth, P, S);
    const int tx0 = X0 - P - S, ty0 = Y0 - P - S;
    float *tf = lds;
    float *tb = lds + (size_t)pitch * trows * C;
    float cen[T::kDist][C];
    stage_tile<C, T::kThreads, T::kStage>(tf, centre, W, H, tx0, ty0, tcols, trows, pitch);
    __syncthreads();
    read_centre<C, P, COLS>(tf, pitch, S, wave, lane, cen);
    if (PAIR) {
        __syncthreads();
        stage_tile<C, T::kThreads, T::kStage>(tf, fwd, W, H, tx0, ty0, tcols, trows, pitch);
        stage_tile<C, T::kThreads, T::kStage>(tb, bwd, W, H, tx0, ty0, tcols, trows, pitch);
        __syncthreads();
    }
    float conf_fv[COLS], conf_bv[COLS];
    if (CONF) {
        load_conf<COLS>(w, conf_f, X0 + wave * COLS, Y0 - 2 * P + lane, conf_fv);
        load_conf<COLS>(w, conf_b, X0 + wave * COLS, Y0 - 2 * P + lane, conf_bv);
    }
    float acc[COLS][C], ws[COLS], mw[COLS], sums[T::kElems][C + 2];
    window_sums<C, P, COLS, PAIR, CONF, SPLIT>(w, tf, tb, pitch, wave, lane, part, cen, lut, conf_fv, conf_bv, acc, ws,
                                               mw);
    join_parts<C, P, COLS, WX, SPLIT>(lds, wave, lane, part, acc, ws, mw, sums);
#pragma unroll
    for (int k = 0; k < T::kElems; ++k) {
        size_t p;
        if (!element_pixel<P, T>(k, X0, Y0, W, H, p)) continue;
        if (!fresh) {
#pragma unroll
            for (int c = 0; c < C; ++c) sums[k][c] = accum[p * C + c] + sums[k][c];
            sums[k][C] = wsum[p] + sums[k][C];
            sums[k][C + 1] = fmaxf(maxw[p], sums[k][C + 1]);
        }
        if (!PAIR && out) {
            finish_pixel<C>(centre + p * C, sums[k], sums[k][C], sums[k][C + 1], self_weight, out + p * C);
        } else {
#pragma unroll
            for (int c = 0; c < C; ++c) accum[p * C + c] = sums[k][c];
            wsum[p] = sums[k][C];
            maxw[p] = sums[k][C + 1];
        }
    }
}

// The batched form: one launch per frame and plane group walks every temporal pair (oldest first),
// then the single window, then the finish, with the window sums of each tile in registers.  Each
// window's sums start from zero and join the running totals in the plain form's order (the plain
// form adds every launch's sums to accumulators that start at zero), so the output is bit-identical
// to the plain launches' while the accumulators never reach memory.  The pair tiles are re-staged
// per pair; the single window stages the centre frame into the first of them.
template <int C, int P, int COLS, int WX, bool CONF, int SPLIT>
__global__ __launch_bounds__(WX * SPLIT * 64) void k_nlm_window(NlmWindow w, NlmFrames f,
                                                                const float *__restrict__ centre,
                                                                const float *__restrict__ lut, float self_weight,
                                                                float *__restrict__ out)
{
    using T = Shape<C, P, COLS, WX, SPLIT>;
    extern __shared__ float lds[];
    const int S = w.S, W = w.W, H = w.H;
    const int lane = threadIdx.x & 63, id = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int wave = id % WX, part = id / WX;
    const int X0 = blockIdx.x * T::kWidth, Y0 = (int)(blockIdx.z * kGridRows + blockIdx.y) * T::kRows;
    const int tcols = T::kWidth + 2 * P + 2 * S, trows = 64 + 2 * S, pitch = tile_pitch(T::kWidth, P, S);
    const int tx0 = X0 - P - S, ty0 = Y0 - P - S;
    float *tf = lds;
    float *tb = lds + (size_t)pitch * trows * C;
    float cen[T::kDist][C];
    stage_tile<C, T::kThreads, T::kStage>(tf, centre, W, H, tx0, ty0, tcols, trows, pitch);
    __syncthreads();
    read_centre<C, P, COLS>(tf, pitch, S, wave, lane, cen);

    float total[T::kElems][C + 2];
#pragma unroll
    for (int k = 0; k < T::kElems; ++k)
#pragma unroll
        for (int c = 0; c < C + 2; ++c) total[k][c] = 0.0f;
    float acc[COLS][C], ws[COLS], mw[COLS], sums[T::kElems][C + 2];
    float conf_fv[COLS], conf_bv[COLS];
    auto join = [&] {
        join_parts<C, P, COLS, WX, SPLIT>(lds, wave, lane, part, acc, ws, mw, sums);
#pragma unroll
        for (int k = 0; k < T::kElems; ++k) {
#pragma unroll
            for (int c = 0; c <= C; ++c) total[k][c] = total[k][c] + sums[k][c];
            total[k][C + 1] = fmaxf(total[k][C + 1], sums[k][C + 1]);
        }
    };
    for (int k = 0; k < f.pairs; ++k) {
        __syncthreads();  // every wave is done with the centre tile, or the previous pair's sums
        stage_tile<C, T::kThreads, T::kStage>(tf, f.fwd[k], W, H, tx0, ty0, tcols, trows, pitch);
        stage_tile<C, T::kThreads, T::kStage>(tb, f.bwd[k], W, H, tx0, ty0, tcols, trows, pitch);
        __syncthreads();
        if (CONF) {
            load_conf<COLS>(w, f.conf_f[k], X0 + wave * COLS, Y0 - 2 * P + lane, conf_fv);
            load_conf<COLS>(w, f.conf_b[k], X0 + wave * COLS, Y0 - 2 * P + lane, conf_bv);
        }
        window_sums<C, P, COLS, true, CONF, SPLIT>(w, tf, tb, pitch, wave, lane, part, cen, nullptr, conf_fv, conf_bv,
                                                   acc, ws, mw);
        join();
    }
    if (f.pairs > 0) {
        __syncthreads();
        stage_tile<C, T::kThreads, T::kStage>(tf, centre, W, H, tx0, ty0, tcols, trows, pitch);
        __syncthreads();
    }
    window_sums<C, P, COLS, false, false, SPLIT>(w, tf, tf, pitch, wave, lane, part, cen, lut, conf_fv, conf_bv, acc,
                                                 ws, mw);
    join();
#pragma unroll
    for (int k = 0; k < T::kElems; ++k) {
        size_t p;
        if (element_pixel<P, T>(k, X0, Y0, W, H, p))
            finish_pixel<C>(centre + p * C, total[k], total[k][C], total[k][C + 1], self_weight, out + p * C);
    }
}

template <int C>
__global__ __launch_bounds__(256) void k_finish(const float *__restrict__ frame, const float *__restrict__ accum,
                                                const float *__restrict__ wsum, const float *__restrict__ maxw,
                                                float self_weight, uint32_t pixels, float *__restrict__ out)
{
    for (uint32_t p = blockIdx.x * 256 + threadIdx.x; p < pixels; p += gridDim.x * 256) {
        const size_t at = (size_t)p * C;
        finish_pixel<C>(frame + at, accum + at, wsum[p], maxw[p], self_weight, out + at);
    }
}

// Waves side by side in a workgroup: four, within eight waves (column runs x offset parts); pairs of
// two-channel frames stage two tiles of twice the width, so they take two, within four waves.
constexpr int waves_for(int C, bool pair, int split)
{
    const int base = (pair && C == 2) ? 2 : 4, cap = C == 2 ? 4 : 8;
    return base * split > cap ? cap / split : base;
}

// Offset parts: each workgroup runs SPLIT waves per column run, each on a consecutive
// run of the window's offset rows, so a frame puts SPLIT times the waves on the chip.  Planes up to
// 2^20 pixels take four (one channel) or two (two channels, whose workgroups hold at most four waves);
// larger ones have waves enough with one: 640x360 makes 480 waves of eight columns at one part, 1920x1080
// about 4500 (when the line was drawn 640x360 ran 12.3k frames/s against 6.3k at one part, 1920x1080
// 4:2:0 643 frames/s against 620 with two parts for luma).  The part sums add in part order, the same
// for every tile shape and both launch forms, which therefore stay bit-identical: a plane's split is
// part of its result.
constexpr int offset_parts(int C) { return C == 1 ? 4 : 2; }
inline int offset_split(int W, int H, int C) { return (size_t)W * H <= (1u << 20) ? offset_parts(C) : 1; }

// LDS of a workgroup: its tile(s), or the part sums of one field while they join, whichever is larger.
size_t tile_bytes(int C, int P, int S, bool pair, int cols, int split, int waves)
{
    const int width = waves * cols;
    const size_t one = (size_t)tile_pitch(width, P, S) * (64 + 2 * S) * C * sizeof(float);
    const size_t parts = (size_t)split * 64 * (width + 1) * sizeof(float);
    return std::max(pair ? 2 * one : one, parts);
}

int device_lds_limit()
{
    static int limit = -1;
    if (limit < 0) {
        int dev = 0, v = 0;
        if (hipGetDevice(&dev) != hipSuccess ||
            hipDeviceGetAttribute(&v, hipDeviceAttributeMaxSharedMemoryPerBlock, dev) != hipSuccess)
            v = 64 * 1024;
        limit = v;
    }
    return limit;
}

// What one window launch works on (a single window's forward and backward frames are the frame itself).
struct Window {
    const float *centre, *fwd, *bwd, *lut, *conf_f, *conf_b;
    float *accum, *wsum, *maxw;
    bool fresh;
    float self_weight;
    float *out;
};

template <int C, int P, int COLS, int SPLIT>
hipError_t dispatch_split(const NlmWindow &w, const Window &a, bool pair, hipStream_t s)
{
    constexpr int WS = waves_for(C, false, SPLIT), WP = waves_for(C, true, SPLIT);
    const size_t lds = tile_bytes(C, P, w.S, pair, COLS, SPLIT, pair ? WP : WS);
    const dim3 grid = tile_grid(div_up(w.W, (pair ? WP : WS) * COLS), div_up(w.H, 64 - 2 * P));
    auto launch = [&](auto kernel, int waves) {
        kernel<<<grid, waves * SPLIT * 64, lds, s>>>(w, a.centre, a.fwd, a.bwd, a.lut, a.conf_f, a.conf_b, a.accum,
                                                     a.wsum, a.maxw, a.fresh, a.self_weight, a.out);
    };
    if (!pair) launch(k_nlm<C, P, COLS, WS, false, false, SPLIT>, WS);
    else if (a.conf_f && a.conf_b) launch(k_nlm<C, P, COLS, WP, true, true, SPLIT>, WP);
    else launch(k_nlm<C, P, COLS, WP, true, false, SPLIT>, WP);
    return hipGetLastError();
}

// One channel splits its offsets over four parts or none, two channels over two or none.
template <int C, int P, int COLS>
hipError_t dispatch_cols(const NlmWindow &w, const Window &a, bool pair, hipStream_t s)
{
    if (offset_split(w.W, w.H, C) > 1) return dispatch_split<C, P, COLS, offset_parts(C)>(w, a, pair, s);
    return dispatch_split<C, P, COLS, 1>(w, a, pair, s);
}

template <int C, int P>
hipError_t dispatch(const NlmWindow &w, const Window &a, bool pair, int variant, hipStream_t s)
{
    switch (variant) {
    case 1: return dispatch_cols<C, P, 4>(w, a, pair, s);
    case 2: return dispatch_cols<C, P, 2>(w, a, pair, s);
    default: return dispatch_cols<C, P, 8>(w, a, pair, s);
    }
}

template <int C>
hipError_t dispatch_p(const NlmWindow &w, const Window &a, bool pair, int variant, hipStream_t s)
{
    switch (w.P) {
    case 0: return dispatch<C, 0>(w, a, pair, variant, s);
    case 1: return dispatch<C, 1>(w, a, pair, variant, s);
    case 2: return dispatch<C, 2>(w, a, pair, variant, s);
    case 3: return dispatch<C, 3>(w, a, pair, variant, s);
    case 4: return dispatch<C, 4>(w, a, pair, variant, s);
    case 5: return dispatch<C, 5>(w, a, pair, variant, s);
    case 6: return dispatch<C, 6>(w, a, pair, variant, s);
    case 7: return dispatch<C, 7>(w, a, pair, variant, s);
    case 8: return dispatch<C, 8>(w, a, pair, variant, s);
    default: return hipErrorInvalidValue;
    }
}

template <int C, int P, int COLS, int SPLIT>
hipError_t dispatch_window_split(const NlmWindow &w, const NlmFrames &f, const float *centre, const float *lut,
                                 float self_weight, float *out, hipStream_t s)
{
    constexpr int WX = waves_for(C, true, SPLIT);
    const size_t lds = tile_bytes(C, P, w.S, f.pairs > 0, COLS, SPLIT, WX);
    const dim3 grid = tile_grid(div_up(w.W, WX * COLS), div_up(w.H, 64 - 2 * P));
    const bool conf = f.pairs > 0 && f.conf_f[0] != nullptr;
    if (conf)
        k_nlm_window<C, P, COLS, WX, true, SPLIT><<<grid, WX * SPLIT * 64, lds, s>>>(w, f, centre, lut, self_weight,
                                                                                    out);
    else
        k_nlm_window<C, P, COLS, WX, false, SPLIT><<<grid, WX * SPLIT * 64, lds, s>>>(w, f, centre, lut, self_weight,
                                                                                     out);
    return hipGetLastError();
}

template <int C, int P, int COLS>
hipError_t dispatch_window(const NlmWindow &w, const NlmFrames &f, const float *centre, const float *lut,
                           float self_weight, float *out, hipStream_t s)
{
    if (offset_split(w.W, w.H, C) > 1)
        return dispatch_window_split<C, P, COLS, offset_parts(C)>(w, f, centre, lut, self_weight, out, s);
    return dispatch_window_split<C, P, COLS, 1>(w, f, centre, lut, self_weight, out, s);
}

template <int C>
hipError_t dispatch_window_p(const NlmWindow &w, const NlmFrames &f, const float *centre, const float *lut,
                             float self_weight, float *out, int variant, hipStream_t s)
{
#define AVD_WINDOW_P(PP)                                                                                      \
    case PP:                                                                                                  \
        return variant == 1 ? dispatch_window<C, PP, 4>(w, f, centre, lut, self_weight, out, s)              \
                            : dispatch_window<C, PP, 8>(w, f, centre, lut, self_weight, out, s);
    switch (w.P) {
        AVD_WINDOW_P(0)
        AVD_WINDOW_P(1)
        AVD_WINDOW_P(2)
        AVD_WINDOW_P(3)
        AVD_WINDOW_P(4)
        AVD_WINDOW_P(5)
        AVD_WINDOW_P(6)
        AVD_WINDOW_P(7)
        AVD_WINDOW_P(8)
    default: return hipErrorInvalidValue;
    }
#undef AVD_WINDOW_P
}

}  // namespace

bool nlm_supported(int C, int P, int S)
{
    return (C == 1 || C == 2) && P >= 0 && P <= kMaxP && S >= 0 && S <= kMaxS &&
           tile_bytes(C, P, S, true, 8, 1, waves_for(C, true, 1)) <= (size_t)device_lds_limit();
}

hipError_t launch_nlm_single(const NlmWindow &w, const float *frame, const float *lut, float *accum, float *wsum,
                             float *maxw, hipStream_t s, int variant, bool fresh, float self_weight, float *out)
{
    if (!nlm_supported(w.C, w.P, w.S) || variant < 0 || variant >= kNlmVariants) return hipErrorInvalidValue;
    const Window a{frame, frame, frame, lut, nullptr, nullptr, accum, wsum, maxw, fresh, self_weight, out};
    return w.C == 1 ? dispatch_p<1>(w, a, false, variant, s) : dispatch_p<2>(w, a, false, variant, s);
}

hipError_t launch_nlm_pair(const NlmWindow &w, const float *centre, const float *fwd, const float *bwd,
                           const float *conf_f, const float *conf_b, float *accum, float *wsum, float *maxw,
                           hipStream_t s, int variant, bool fresh)
{
    if (!nlm_supported(w.C, w.P, w.S) || variant < 0 || variant >= kNlmVariants) return hipErrorInvalidValue;
    const Window a{centre, fwd, bwd, nullptr, conf_f, conf_b, accum, wsum, maxw, fresh, 0.0f, nullptr};
    return w.C == 1 ? dispatch_p<1>(w, a, true, variant, s) : dispatch_p<2>(w, a, true, variant, s);
}

hipError_t launch_nlm_window(const NlmWindow &w, const NlmFrames &f, const float *centre, const float *lut,
                             float self_weight, float *out, hipStream_t s, int variant)
{
    if (!nlm_supported(w.C, w.P, w.S) || variant < 0 || variant >= kNlmBatchedVariants || f.pairs < 0 ||
        f.pairs > kNlmMaxPairs || !centre || !lut || !out)
        return hipErrorInvalidValue;
    for (int k = 0; k < f.pairs; ++k)
        if (!f.fwd[k] || !f.bwd[k] || (f.conf_f[0] != nullptr) != (f.conf_f[k] != nullptr && f.conf_b[k] != nullptr))
            return hipErrorInvalidValue;
    if (w.C == 1) return dispatch_window_p<1>(w, f, centre, lut, self_weight, out, variant, s);
    return dispatch_window_p<2>(w, f, centre, lut, self_weight, out, variant, s);
}

hipError_t launch_nlm_finish(const float *frame, const float *accum, const float *wsum, const float *maxw,
                             float self_weight, uint32_t pixels, int C, float *out, hipStream_t s)
{
    unsigned g = div_up(pixels, 256);
    if (g > 4096) g = 4096;
    if (g < 1) g = 1;
    if (C == 1) k_finish<1><<<g, 256, 0, s>>>(frame, accum, wsum, maxw, self_weight, pixels, out);
    else k_finish<2><<<g, 256, 0, s>>>(frame, accum, wsum, maxw, self_weight, pixels, out);
    return hipGetLastError();
}

}  // namespace avd
