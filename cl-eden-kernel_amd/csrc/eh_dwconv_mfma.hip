// Depthwise uint8 convolution with 5x5 and 7x7 windows on the matrix cores (gfx950), channels-last tensors.
//
// On the vector units such a window is bound by instructions: 8-bit dot products need every channel's taps gathered into
// words first, 30 instructions per output at 5x5 (64 images of 144 channels at 56x56: 39 us, 22.6 here; the bytes take 11).
// The matrix form needs no gather.  One 16x16x64 product takes 16 pixels and, per pixel, 64 bytes: the 16 channels of a
// 16-byte piece at four neighbouring taps of a kernel row, read as they lie in memory; the other operand is diagonal
// (channel i of tap t only reaches output channel i), so 15 of 16 products multiply zeros, and 25 taps still cost seven
// products of 16 cycles per 256 outputs.  What is left on the vector units is the requantization.
//
//   workgroup   an output tile of 2 TH rows x 8 nx pixels in up to 64 channels; its input tile lies in LDS, one plane per
//               16-byte piece, as value - 128, pixels outside the image as the input zero point
//   wave        16 channels; walks input rows downwards for 8 columns in two strips of TH rows at once (lanes 0-7 and
//               8-15 of each 16), multiplies each row's operand by the weights of every kernel row it belongs to and
//               finishes the output row above in the shadow of the products
//   5x5         the fifth kernel column by itself: an operand of four rows at that column serves four of its taps, and the
//               same operand four rows further down the fifth
//
// Weights are stored as w - zp_w - d, d being zero unless one of the channel's differences leaves int8 (a byte's range
// spans 255, so some d always fits).  A channel with d adds d times its window's sum, taken from a running sum of the
// input rows (two more products per row, only in waves that hold such a channel).
#include <type_traits>

#include "eh_internal.h"

namespace eh {
namespace {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v4i_a4 __attribute__((ext_vector_type(4), aligned(4)));

constexpr int kStrips = 2, kColumns = 8;

struct DwTile {
    uint32_t tiles;                         // workgroups that have one
    int32_t cblocks, tiles_x, tiles_y;      // channel blocks, and tiles per image
    int32_t chunks, ch_per;                 // 16-byte channel pieces: of a pixel, of a workgroup
    int32_t nx, waves_per_chunk;            // groups of eight columns per tile; waves that share them
    int32_t rows, cols, plane;              // input tile; bytes per piece's plane in LDS
    int32_t rows_per_step;                  // tile rows the workgroup fetches at a time
    uint32_t in_bytes, out_bytes;
    FastDiv div_cblocks, div_tiles_x, div_tiles_y, div_ch, div_line;
};

// XCD x (workgroups x, x + 8, ...) takes the x-th eighth of the tiles: neighbouring tiles share input rows
__device__ __forceinline__ uint32_t xcd_contiguous_block() { return (blockIdx.x & 7u) * (gridDim.x >> 3) + (blockIdx.x >> 3); }

// 16 bytes, all zero but the one at `at`
__device__ __forceinline__ v4i one_byte(uint32_t byte, int at) {
    const int v = (int)(byte << (8 * (at & 3))), d = at >> 2;
    return v4i{d == 0 ? v : 0, d == 1 ? v : 0, d == 2 ? v : 0, d == 3 ? v : 0};
}

constexpr int kernel_columns(int k) { return (k + 3) / 4 * 4; }

// K: window.  S: stride.  TH: output rows per strip.  PC: one multiplier and shift per channel.  MODE: single-shift form of
// the requantization (1, 2) or the two-step form (0).  (One form has a register more than four waves per SIMD leave it: 224 channels at 32x64, 7x7, 35 images
// 22.4 us, held to four waves 19.8.)
template <int K, int S, int TH, bool PC, int MODE>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(K == 7 && S == 1 && TH == 4 && !PC && MODE == 2 ? 4 : 1))) void dw_mfma_kernel(const DwProblem p, const DwTile g) {
    constexpr int KF = kernel_columns(K), ROWS = (TH - 1) * S + K;
    constexpr bool COLUMN = K == 5;             // the fifth kernel column by itself
    constexpr int FX = KF / 4, FR = COLUMN ? 1 : FX;  // operands per input row; those that run along the row
    extern __shared__ __align__(16) uint8_t lds[];
    const uint32_t tile = xcd_contiguous_block();
    if (tile >= g.tiles) return;
    const uint32_t t1 = fastdiv(tile, g.div_cblocks), t2 = fastdiv(t1, g.div_tiles_x);
    const int cb = (int)(tile - t1 * (uint32_t)g.cblocks), tx = (int)(t1 - t2 * (uint32_t)g.tiles_x);
    const int img = (int)fastdiv(t2, g.div_tiles_y), ty = (int)t2 - img * g.tiles_y;
    const int oy0 = ty * TH * kStrips, ox0 = tx * g.nx * kColumns;
    const int iy0 = oy0 * S - p.pad_t, ix0 = ox0 * S - p.pad_l;
    const int chunk0 = cb * g.ch_per, n_chunks = g.chunks - chunk0 < g.ch_per ? g.chunks - chunk0 : g.ch_per;
    const int tid = threadIdx.x, lane = tid & 63, quarter = lane >> 4, lane16 = lane & 15;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    // ---- this wave's weights: lane16's channel at the taps of its quarter, requested ahead of the input tile
    const int chunk = wave / g.waves_per_chunk, first_x = wave - chunk * g.waves_per_chunk;
    const int c0 = (chunk0 + chunk) * 16, c_out = c0 + quarter * 4, cpad = g.chunks * 16;
    const bool works = chunk < n_chunks;
    uint32_t w_row[K][FR], w_col[2] = {0, 0}, d_neg = 0;
    int4 bias = make_int4(0, 0, 0, 0), mult = bias, shift = bias;
    if (works) {
        const uint8_t *w = p.w_mm + c0 + lane16;
#pragma unroll
        for (int ky = 0; ky < K; ++ky)
#pragma unroll
            for (int f = 0; f < FR; ++f) w_row[ky][f] = w[(ky * KF + f * 4 + quarter) * cpad];
        if constexpr (COLUMN) {
            w_col[0] = w[(quarter * KF + 4) * cpad];
            w_col[1] = w[(quarter == 0 ? 4 * KF + 4 : KF - 1) * cpad];  // (column KF - 1 is padding: zero)
        }
        d_neg = w[K * KF * cpad];
        bias = *reinterpret_cast<const int4 *>(p.bias_mm + c_out);
        if constexpr (PC) {
            const int ch = c_out < p.c ? c_out : 0;
            mult = *reinterpret_cast<const int4 *>(p.rq.pc_multiplier + ch);
            shift = *reinterpret_cast<const int4 *>(p.rq.pc_shift + ch);
        }
    }
    // ---- the input tile
    const int flip = p.io_flip ? 0 : (int)0x80808080u;  // to value - 128
    const int fill = (int)(((uint32_t)p.zp_in * 0x01010101u) ^ 0x80808080u);
    const uint32_t base = (uint32_t)img * (uint32_t)(p.h * p.w_ * p.c) + (uint32_t)chunk0 * 16u;
    const int line = g.cols * g.ch_per;  // 16-byte pieces of a tile row
    const auto in = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t *>(p.in), 0, (int)g.in_bytes, 0x00020000);
    constexpr int BATCH = 4;             // rows a thread has on their way
    auto fetch = [&](auto inside_c, auto whole_c) {
        constexpr bool INSIDE = decltype(inside_c)::value, WHOLE = decltype(whole_c)::value;
        const int y_first = g.rows_per_step > 1 ? (int)fastdiv((uint32_t)tid, g.div_line) : 0;
        if (y_first >= g.rows_per_step) return;
        for (int e = tid - y_first * line; e < line; e += (int)blockDim.x) {  // (one turn where a step takes whole rows)
            const int x = (int)fastdiv((uint32_t)e, g.div_ch), c = e - x * g.ch_per, ix = ix0 + x;
            const bool exists = INSIDE || ((unsigned)ix < (unsigned)p.w_ && c < n_chunks);
            // A piece that does not exist is loaded without a branch of its own: with one the compiler waited for each load before it
            // made the next.  (144 channels at 56x56, 64 images: 5x5 25.6 -> 24.7 us, at stride 2 16.0 -> 14.7, 7x7 36.3 -> 32.8; 88
            // at 100x100, 7x7 stride 2, 44 images 26.5 -> 22.6.)  Of pixels of whole pieces it is sent past the tensor's end, where
            // the bounds check gives zero, and the XOR that makes operands makes it the fill: one select in place of the clamps and
            // four more.  (The first and third again: 23.8 -> 22.6, 32.6 -> 30.2.)
            const int ixc = ix < 0 ? 0 : (ix < p.w_ ? ix : p.w_ - 1), cc = c < n_chunks ? c : 0;
            const uint32_t off0 = base + (uint32_t)((WHOLE ? ix : ixc) * p.c + (WHOLE ? c : cc) * 16), pitch = (uint32_t)(p.w_ * p.c);
            uint8_t *to = lds + c * g.plane + x * 16;
            for (int y0 = y_first; y0 < g.rows; y0 += g.rows_per_step * BATCH) {
                v4i v[BATCH];
                int mask[BATCH];
#pragma unroll
                for (int b = 0; b < BATCH; ++b) {
                    const int y = y0 + b * g.rows_per_step;
                    if constexpr (WHOLE) {
                        const bool there = y < g.rows && (INSIDE || (exists && (unsigned)(iy0 + y) < (unsigned)p.h));
                        mask[b] = there ? flip : fill;
                        v[b] = __builtin_amdgcn_raw_buffer_load_b128(in, (int)(there ? off0 + (uint32_t)(iy0 + y) * pitch : 0xFFFFFFF0u), 0, 0);
                    } else {
                        int iy = iy0 + (y < g.rows ? y : g.rows - 1);
                        iy = iy < 0 ? 0 : (iy < p.h ? iy : p.h - 1);
                        const uint32_t off = off0 + (uint32_t)iy * pitch;
                        if (off + 16u <= g.in_bytes) {
                            v[b] = *reinterpret_cast<const v4i_a4 *>(p.in + off);
                        } else {  // the tensor's last pixel, where it ends inside a piece
                            v[b] = v4i{0, 0, 0, 0};
#pragma unroll
                            for (int d = 0; d < 3; ++d)
                                if (off + 4u * d + 4u <= g.in_bytes) v[b][d] = *reinterpret_cast<const int *>(p.in + off + 4u * d);
                        }
                    }
                }
#pragma unroll
                for (int b = 0; b < BATCH; ++b) {
                    const int y = y0 + b * g.rows_per_step;
                    if constexpr (WHOLE) {
                        v[b] ^= v4i{mask[b], mask[b], mask[b], mask[b]};
                    } else {
                        const bool there = exists && (unsigned)(iy0 + y) < (unsigned)p.h;
                        v[b] = v4i{there ? v[b].x ^ flip : fill, there ? v[b].y ^ flip : fill, there ? v[b].z ^ flip : fill, there ? v[b].w ^ flip : fill};
                    }
                    if (y < g.rows) *reinterpret_cast<v4i *>(to + y * g.cols * 16) = v[b];
                }
            }
        }
    };
    if ((p.c & 15) != 0)
        fetch(std::false_type{}, std::false_type{});
    else if (iy0 >= 0 && iy0 + g.rows <= p.h && ix0 >= 0 && ix0 + g.cols <= p.w_ && n_chunks == g.ch_per)
        fetch(std::true_type{}, std::true_type{});
    else
        fetch(std::false_type{}, std::true_type{});
    __syncthreads();
    if (!works) return;
    v4i wf[K][FR], wc[2];
#pragma unroll
    for (int ky = 0; ky < K; ++ky)
#pragma unroll
        for (int f = 0; f < FR; ++f) wf[ky][f] = one_byte(w_row[ky][f], lane16);
    wc[0] = one_byte(w_col[0], lane16);
    wc[1] = one_byte(w_col[1], lane16);
    const RequantDev rq = p.rq;
    const int col = lane16 & (kColumns - 1), strip = lane16 / kColumns;
    const int pitch = g.cols * 16;
    const uint32_t out_pitch = (uint32_t)(p.wo * p.c);
    // pixels that do not exist are sent past the tensor's end, where the hardware's bounds check drops them: no branch per row
    const auto out = __builtin_amdgcn_make_buffer_rsrc(p.out, 0, (int)g.out_bytes, 0x00020000);
    auto walk = [&](auto d_c) {
        constexpr bool D = decltype(d_c)::value;  // some channel of the wave has d != 0
        v4i df[FX];
#pragma unroll
        for (int f = 0; f < FX; ++f) df[f] = one_byte(D && f * 4 + quarter < K ? d_neg : 0, lane16);
        for (int xg = first_x; xg < g.nx; xg += g.waves_per_chunk) {
            const int px = xg * kColumns + col;
            const uint8_t *src = lds + chunk * g.plane + ((strip * TH * S) * g.cols + px * S + quarter) * 16;
            // (quarter q of the column's operand: kernel row q)
            const uint8_t *src_col = lds + chunk * g.plane + ((strip * TH * S + quarter) * g.cols + px * S + 4) * 16;
            const int oy = oy0 + strip * TH, ox = ox0 + px;
            const int rows_here = ox < p.wo && c_out < p.c ? p.ho - oy : 0;
            const uint32_t dst = (((uint32_t)img * (uint32_t)p.ho + (uint32_t)oy) * (uint32_t)p.wo + (uint32_t)ox) * (uint32_t)p.c + (uint32_t)c_out;
            v4i acc[TH], past = v4i{0, 0, 0, 0}, past_out = past;  // past: -d times the sum of the rows so far
            auto finish = [&](int o) {
                v4i a = acc[o];
                if constexpr (D) a -= past_out;
                uint32_t v;
                if constexpr (PC && MODE == 0)
                    v = pack_bytes(requant_u8_channel(a.x, mult.x, shift.x, rq), requant_u8_channel(a.y, mult.y, shift.y, rq),
                                   requant_u8_channel(a.z, mult.z, shift.z, rq), requant_u8_channel(a.w, mult.w, shift.w, rq));
                else if constexpr (PC)
                    v = pack_bytes(requant_u8_channel_fast<MODE>(a.x, mult.x, shift.x, rq), requant_u8_channel_fast<MODE>(a.y, mult.y, shift.y, rq),
                                   requant_u8_channel_fast<MODE>(a.z, mult.z, shift.z, rq), requant_u8_channel_fast<MODE>(a.w, mult.w, shift.w, rq));
                else if constexpr (MODE == 0)
                    v = pack_bytes(requant_u8(a.x, rq), requant_u8(a.y, rq), requant_u8(a.z, rq), requant_u8(a.w, rq));
                else
                    v = requant4_fast<MODE>(a.x, a.y, a.z, a.w, 0, rq);
                __builtin_amdgcn_raw_buffer_store_b32(v ^ p.io_flip, out, (int)(o < rows_here ? dst + (uint32_t)o * out_pitch : 0xFFFFFFF0u), 0, 0);
            };
            v4i ahead[FX];
            auto load = [&](int row) {
#pragma unroll
                for (int f = 0; f < FX; ++f) ahead[f] = *reinterpret_cast<const v4i *>(COLUMN && f == 1 ? src_col + row * pitch : src + row * pitch + f * 64);
            };
            load(0);
#pragma unroll
            for (int row = 0; row < ROWS; ++row) {
                v4i x[FX];
#pragma unroll
                for (int f = 0; f < FX; ++f) x[f] = ahead[f];
                if (row + 1 < ROWS) load(row + 1);
                if constexpr (D) past_out = past;
                if (row % S == 0 && row / S < TH) {  // output row / S starts here
                    acc[row / S] = v4i{bias.x, bias.y, bias.z, bias.w};
                    if constexpr (D) acc[row / S] += past;
                }
#pragma unroll
                for (int f = 0; f < FX; ++f) {
                    if constexpr (D) past = __builtin_amdgcn_mfma_i32_16x16x64_i8(df[f], x[f], past, 0, 0, 0);
#pragma unroll
                    for (int ky = K - 1; ky >= 0; --ky)
                        if (f < FR && (row - ky) % S == 0 && row >= ky && (row - ky) / S < TH)
                            acc[(row - ky) / S] = __builtin_amdgcn_mfma_i32_16x16x64_i8(wf[ky][f < FR ? f : 0], x[f], acc[(row - ky) / S], 0, 0, 0);
                }
                if constexpr (COLUMN) {
                    if (row % S == 0 && row / S < TH) acc[row / S] = __builtin_amdgcn_mfma_i32_16x16x64_i8(wc[0], x[1], acc[row / S], 0, 0, 0);
                    if (row >= 4 && (row - 4) % S == 0 && (row - 4) / S < TH)
                        acc[(row - 4) / S] = __builtin_amdgcn_mfma_i32_16x16x64_i8(wc[1], x[1], acc[(row - 4) / S], 0, 0, 0);
                }
                if (row >= K && (row - K) % S == 0) finish((row - K) / S);  // complete since the row above
                __builtin_amdgcn_sched_barrier(0);  // (rows stay apart: hoisted operand loads would cost the registers of another wave)
            }
            past_out = past;
            finish(TH - 1);
        }
    };
    if (__builtin_amdgcn_ballot_w64(d_neg != 0) != 0)
        walk(std::true_type{});
    else
        walk(std::false_type{});
}

// weights [cout][K * K] -> w_mm[ky * KF + kx][cpad] (KF, cpad: the window's width and the channels rounded up to 4 and 16) as
// w - zp_w - d, then -d[cpad]; bias_mm[c] = bias - (zp_in - 128) * sum (w - zp_w)
__global__ void dw_pack_mfma_kernel(const uint8_t *w, const int32_t *bias, uint8_t *w_mm, int32_t *bias_mm, int32_t cout, int32_t cpad, int32_t k, int32_t zp_in,
                                    int32_t zp_w, int32_t w_signed) {
    const int oc = blockIdx.x * blockDim.x + threadIdx.x;
    if (oc >= cpad) return;
    const int kf = kernel_columns(k);
    auto value = [&](int ky, int kx) {
        const uint8_t raw = w[(size_t)oc * k * k + ky * k + kx];
        return (w_signed ? (int32_t)(int8_t)raw : (int32_t)raw) - zp_w;
    };
    int32_t sum = 0, lo = 0, hi = 0;
    if (oc < cout)
        for (int ky = 0; ky < k; ++ky)
            for (int kx = 0; kx < k; ++kx) {
                const int32_t v = value(ky, kx);
                sum += v;
                lo = v < lo ? v : lo;
                hi = v > hi ? v : hi;
            }
    // (the differences span at most 255, so what is left fits; d is at most 128, and -d is what is stored)
    const int32_t d = hi > 127 ? hi - 127 : lo < -128 ? lo + 128 : 0;
    for (int ky = 0; ky < k; ++ky)
        for (int kx = 0; kx < kf; ++kx) w_mm[(size_t)(ky * kf + kx) * cpad + oc] = (uint8_t)(oc < cout && kx < k ? value(ky, kx) - d : 0);
    w_mm[(size_t)k * kf * cpad + oc] = (uint8_t)-d;
    bias_mm[oc] = oc < cout ? (bias ? bias[oc] : 0) - (zp_in - 128) * sum : 0;
}

// The tile of a launch; its output rows per strip as the result.
int plan_tile(const DwProblem &p, DwTile *g) {
    const int K = p.kh, S = p.stride_h;
    g->chunks = (p.c + 15) / 16;
    const int groups = (p.wo + kColumns - 1) / kColumns;
    auto shape = [&](int th, int nx, int chunks_max) {
        if (groups == 1 || groups == 3) {  // pairs of column groups would leave one idle
            chunks_max = nx > 1 && chunks_max < 4 ? chunks_max * 2 : chunks_max;
            nx = 1;
        }
        g->cblocks = (g->chunks + chunks_max - 1) / chunks_max;
        g->ch_per = (g->chunks + g->cblocks - 1) / g->cblocks;
        g->cblocks = (g->chunks + g->ch_per - 1) / g->ch_per;
        g->nx = nx < groups ? nx : groups;
        g->tiles_x = (groups + g->nx - 1) / g->nx;
        g->tiles_y = (p.ho + th * kStrips - 1) / (th * kStrips);
        return (long)p.n * g->tiles_y * g->tiles_x * g->cblocks;
    };
    // Large tiles share halos, weights and setup, small ones fill the chip: the largest shape that leaves a tile or two for
    // every workgroup the chip holds at a time.  5x5, us by shape (rows of 7 or 4, column groups, pieces): 144 channels at
    // 56x56, 64 images 23.6 (7,2,4) 26.7 (7,7,3) 24.3 (7,1,4) 27 (4,2,2); 32 at 112x112, 32 images 11.5 (7,7,1) 12.1 (7,7,2);
    // 240 at 28x28, 16 images 5.9 (7,2,2) 6.3 (4,2,2); 480 at 14x14, 16 images 4.8 (4,2,2) 5.0 (7,1,2); 960 at 7x7, one image
    // 4.0 (4,1,2).  Other shapes were faster by 2.6 % on average over 33 layers.
    // At stride 2 the largest shapes would take half a CU's LDS; strips of seven rows that leave a quarter more of their
    // rows past the image than strips of four are not used (120 at 30x30, 30 images: 6.5 us (7,2,2), 6.0 (4,2,2); 192 at 80x80
    // stride 2, 6 images: 6.5 (4,2,2), 6.0 (4,1,2)).
    int th = 7;
    const bool short_strips = 4 * ((p.ho + 13) / 14 * 14) > 5 * ((p.ho + 7) / 8 * 8);
    long tiles = S == 2 || short_strips ? 0 : g->chunks > 2 ? shape(7, 2, 4) : shape(7, 7, 1);
    if (tiles < 768 && (short_strips || (tiles = shape(7, 2, 2)) < 512)) {
        th = 4;
        if ((tiles = shape(4, 2, 2)) < (S == 2 ? 640 : 256)) tiles = shape(4, 1, 2);
    }
    if (p.rq.fast == 0 && th == 7) {  // (the two-step form has the short strips only)
        th = 4;
        tiles = shape(4, 2, 2);
    }
    g->tiles = tiles < (1l << 31) - 8 ? (uint32_t)tiles : 0;
    g->waves_per_chunk = g->ch_per >= 3 ? 1 : 4 / g->ch_per;
    g->rows = (th * kStrips - 1) * S + K;
    g->cols = (g->nx * kColumns - 1) * S + K;
    // planes start on different banks, so that the pieces of a pixel are written side by side
    const int skew = g->ch_per == 1 ? 0 : (128 / g->ch_per + 15) / 16 * 16;
    g->plane = g->rows * g->cols * 16;
    g->plane += ((skew - g->plane) % 128 + 128) % 128;
    const int line = g->cols * g->ch_per, threads = g->ch_per * g->waves_per_chunk * 64;
    g->rows_per_step = line < threads ? threads / line : 1;
    g->in_bytes = (uint32_t)((size_t)p.n * p.h * p.w_ * p.c);
    g->out_bytes = (uint32_t)((size_t)p.n * p.ho * p.wo * p.c);
    g->div_cblocks = make_fastdiv((uint32_t)g->cblocks);
    g->div_tiles_x = make_fastdiv((uint32_t)g->tiles_x);
    g->div_tiles_y = make_fastdiv((uint32_t)g->tiles_y);
    g->div_ch = make_fastdiv((uint32_t)g->ch_per);
    g->div_line = make_fastdiv((uint32_t)line);
    return th;
}

}  // namespace

size_t dw_mfma_weight_bytes(int32_t cout, int32_t k) { return (size_t)(k * kernel_columns(k) + 1) * (size_t)((cout + 15) / 16 * 16); }

int launch_dw_pack_mfma(const uint8_t *w, const int32_t *bias, uint8_t *w_mm, int32_t *bias_mm, int32_t cout, int32_t k, int32_t zp_in, int32_t zp_w, int32_t w_signed,
                        hipStream_t stream) {
    if (cout <= 0) return EH_OK;
    const int cpad = (cout + 15) / 16 * 16;
    hipLaunchKernelGGL(dw_pack_mfma_kernel, dim3((cpad + 127) / 128), dim3(128), 0, stream, w, bias, w_mm, bias_mm, cout, cpad, k, zp_in, zp_w, w_signed);
    EH_HIP(hipGetLastError());
    return EH_OK;
}

// 3x3 windows stay on the vector units: nine taps are three dot products there and six products' worth of LDS trips here
// (240 channels at 28x28, 16 images: 4.5 us there, 5.2 here).
bool dw_mfma_applies(const DwProblem &p) {
    return p.w_mm != nullptr && p.kh == p.kw && (p.kh == 5 || p.kh == 7) && p.dil_h == 1 && p.dil_w == 1 && p.dm == 1 && (p.c & 3) == 0 &&
           p.stride_h == p.stride_w && (p.stride_h == 1 || p.stride_h == 2) && ((reinterpret_cast<uintptr_t>(p.in) | reinterpret_cast<uintptr_t>(p.out)) & 3) == 0 &&
           (size_t)p.n * p.h * p.w_ * p.c < (1ull << 31) && (size_t)p.n * p.ho * p.wo * p.cout < (1ull << 31);
}

int launch_dw_mfma(const DwProblem &p, hipStream_t stream) {
    DwTile g;
    const int th = plan_tile(p, &g);
    EH_REQUIRE(g.tiles != 0, "depthwise: grid too large");
    // (the column's operand reads three rows past the last tile row, the row's four pixels past its end: multiplied by zero)
    const size_t lds = (size_t)g.plane * g.ch_per + (size_t)3 * g.cols * 16 + 64;
    const dim3 grid((g.tiles + 7) / 8 * 8), block((unsigned)(g.ch_per * g.waves_per_chunk * 64));
    auto launch = [&](auto k_c, auto s_c, auto th_c, auto pc_c, auto mode_c) {
        auto kernel = dw_mfma_kernel<decltype(k_c)::value, decltype(s_c)::value, decltype(th_c)::value, decltype(pc_c)::value, decltype(mode_c)::value>;
        hipLaunchKernelGGL(kernel, grid, block, lds, stream, p, g);
    };
    using std::integral_constant;
    auto with_mode = [&](auto k_c, auto s_c, auto pc_c) {
        if (p.rq.fast == 0)
            launch(k_c, s_c, integral_constant<int, 4>{}, pc_c, integral_constant<int, 0>{});
        else if (p.rq.fast == 2)
            th == 4 ? launch(k_c, s_c, integral_constant<int, 4>{}, pc_c, integral_constant<int, 2>{})
                    : launch(k_c, s_c, integral_constant<int, 7>{}, pc_c, integral_constant<int, 2>{});
        else
            th == 4 ? launch(k_c, s_c, integral_constant<int, 4>{}, pc_c, integral_constant<int, 1>{})
                    : launch(k_c, s_c, integral_constant<int, 7>{}, pc_c, integral_constant<int, 1>{});
    };
    auto with_stride = [&](auto k_c, auto s_c) { p.rq.pc_multiplier ? with_mode(k_c, s_c, std::true_type{}) : with_mode(k_c, s_c, std::false_type{}); };
    auto with_window = [&](auto k_c) {
        p.stride_h == 1 ? with_stride(k_c, integral_constant<int, 1>{}) : with_stride(k_c, integral_constant<int, 2>{});
    };
    p.kh == 5 ? with_window(integral_constant<int, 5>{}) : with_window(integral_constant<int, 7>{});
    EH_HIP(hipGetLastError());
    return EH_OK;
}

}  // namespace eh
