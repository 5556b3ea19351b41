// Depthwise uint8 convolution (gfx950) on the vector units: 3x3 windows, and every window the matrix form
// (eh_dwconv_mfma.hip) does not take.
//
// Replaces the reference's depthwise kernels for the uint8 path
// (gpu/operators/cl_kernels/DepthwiseconvolutionKernels.cpp:1242-2290: generic
// depthwise_conv plus the 3x3 pad-merge specialisations) and their pad pass
// (PadConvertKernels.cpp:7-23).  Out-of-image taps read the input zero point,
// as the reference's padding does, so they contribute nothing.
//
// Channels-last fast path: one thread owns four adjacent channels of one output
// pixel, so a wavefront reads whole contiguous pixel rows.  Two taps of one
// channel are paired into a 16-bit dot product (v_dot2_i32_i16) against
// weights stored as (w - zp_w) int16 pairs; the input zero point is folded
// into the bias: sum (a - zi)(w - zw) = sum a (w - zw) - zi * sum (w - zw).
#include <type_traits>

#include "eh_internal.h"

namespace eh {
namespace {

typedef short v2s __attribute__((ext_vector_type(2)));

__device__ __forceinline__ int dot2(uint32_t a_pair, int32_t w_pair, int acc) {
    return __builtin_amdgcn_sdot2(__builtin_bit_cast(v2s, a_pair), __builtin_bit_cast(v2s, w_pair), acc, false);
}

// byte j of `lo` into bits 0..15 and byte j of `hi` into bits 16..31, zero extended
template <int J>
__device__ __forceinline__ uint32_t pair_bytes(uint32_t lo, uint32_t hi) {
    constexpr uint32_t sel = (0x0cu << 24) | ((4u + J) << 16) | (0x0cu << 8) | (uint32_t)J;
    return __builtin_amdgcn_perm(hi, lo, sel);
}

// The per-channel multipliers and shifts of four adjacent channels, read once per thread.
struct ChannelQuad {
    int4 m, s;
};
template <bool PC>
__device__ __forceinline__ ChannelQuad load_channel_quad(const RequantDev &rq, uint32_t ch) {
    ChannelQuad q{};
    if (PC && rq.pc_multiplier) {
        q.m = *reinterpret_cast<const int4 *>(rq.pc_multiplier + ch);
        q.s = *reinterpret_cast<const int4 *>(rq.pc_shift + ch);
    }
    return q;
}

// Four adjacent channels' accumulators to four output bytes.  With one multiplier and shift per channel
// (depthwise_conv_per_channel, gpu/operators/cl_kernels/DepthwiseconvolutionKernels.cpp:1323-1371) the four pairs
// come in `cq`.
template <bool PC = true>
__device__ __forceinline__ uint32_t requant4(int acc0, int acc1, int acc2, int acc3, const RequantDev &rq, const ChannelQuad &cq) {
    if (PC && rq.pc_multiplier)  // the two-step order; the single-shift form per channel is the dot product kernel's
        return pack_bytes(requant_u8_channel(acc0, cq.m.x, cq.s.x, rq), requant_u8_channel(acc1, cq.m.y, cq.s.y, rq),
                          requant_u8_channel(acc2, cq.m.z, cq.s.z, rq), requant_u8_channel(acc3, cq.m.w, cq.s.w, rq));
    if (rq.fast == 2) return requant4_fast<2>(acc0, acc1, acc2, acc3, 0, rq);
    if (rq.fast) return requant4_fast<1>(acc0, acc1, acc2, acc3, 0, rq);
    return pack_bytes(requant_u8(acc0, rq), requant_u8(acc1, rq), requant_u8(acc2, rq), requant_u8(acc3, rq));
}

// the per-channel single-shift form alone (rq.fast is 1 or 2)
__device__ __forceinline__ uint32_t requant4_channel_fast(int acc0, int acc1, int acc2, int acc3, const RequantDev &rq, const ChannelQuad &cq) {
    if (rq.fast == 2)
        return pack_bytes(requant_u8_channel_fast<2>(acc0, cq.m.x, cq.s.x, rq), requant_u8_channel_fast<2>(acc1, cq.m.y, cq.s.y, rq),
                          requant_u8_channel_fast<2>(acc2, cq.m.z, cq.s.z, rq), requant_u8_channel_fast<2>(acc3, cq.m.w, cq.s.w, rq));
    return pack_bytes(requant_u8_channel_fast<1>(acc0, cq.m.x, cq.s.x, rq), requant_u8_channel_fast<1>(acc1, cq.m.y, cq.s.y, rq),
                      requant_u8_channel_fast<1>(acc2, cq.m.z, cq.s.z, rq), requant_u8_channel_fast<1>(acc3, cq.m.w, cq.s.w, rq));
}

// Workgroups are dispatched round-robin over the 8 XCDs, each with its own L2.  Neighbouring output rows read
// the same input rows, so every XCD takes one contiguous eighth of the block range (launch grids are whole
// multiples of 8): a shared input row is then fetched from HBM into one L2 instead of two or three.
__device__ __forceinline__ uint32_t xcd_contiguous_block() { return (blockIdx.x & 7u) * (gridDim.x >> 3) + (blockIdx.x >> 3); }

// One output pixel's four adjacent channels per thread, any kernel size, stride and dilation (KH = 0: sizes from the
// problem).  SMALL: both tensors below 2^31 bytes, so the index is decoded with 32-bit multiplications and the taps'
// offsets are 32-bit (64-bit divisions and multiply-adds cost several times the rest of a small kernel's arithmetic).
template <int KH, int KW, bool SMALL>
__global__ __launch_bounds__(256) void dw_nhwc_vec4_kernel(const DwProblem p, const long total, const FastDiv div_cq, const FastDiv div_wo,
                                                           const FastDiv div_ho) {
    using Offset = std::conditional_t<SMALL, uint32_t, size_t>;
    const long idx = (long)xcd_contiguous_block() * 256 + threadIdx.x;
    if (idx >= total) return;
    const int cq_count = p.c >> 2;
    int cq, ox, oy, img;
    Offset pix;
    if constexpr (SMALL) {
        const uint32_t i = (uint32_t)idx, px = fastdiv(i, div_cq), t0 = fastdiv(px, div_wo), im = fastdiv(t0, div_ho);
        cq = (int)(i - px * (uint32_t)cq_count);
        ox = (int)(px - t0 * (uint32_t)p.wo);
        oy = (int)(t0 - im * (uint32_t)p.ho);
        img = (int)im;
        pix = px;
    } else {
        cq = (int)(idx % cq_count);
        const long px = idx / cq_count;
        ox = (int)(px % p.wo);
        const long t0 = px / p.wo;
        oy = (int)(t0 % p.ho), img = (int)(t0 / p.ho);
        pix = (Offset)px;
    }
    const int kh = KH ? KH : p.kh, kw = KW ? KW : p.kw;
    const int taps = kh * kw, pairs = (taps + 1) >> 1;
    const int iy0 = oy * p.stride_h - p.pad_t, ix0 = ox * p.stride_w - p.pad_l;
    const uint8_t *src = p.in + ((Offset)img * (Offset)(p.h * p.w_) * (Offset)p.c + (Offset)(cq * 4));
    const uint32_t fill = (uint32_t)p.zp_in * 0x01010101u;

    auto tap_at = [&](int ky, int kx) -> uint32_t {
        // loaded from a clamped address whatever the tap, so that the loads of several taps can be in flight together
        const int iy = iy0 + ky * p.dil_h, ix = ix0 + kx * p.dil_w;
        const int iyc = iy < 0 ? 0 : (iy >= p.h ? p.h - 1 : iy), ixc = ix < 0 ? 0 : (ix >= p.w_ ? p.w_ - 1 : ix);
        const uint32_t v = *reinterpret_cast<const uint32_t *>(src + ((Offset)iyc * (Offset)p.w_ + (Offset)ixc) * (Offset)p.c) ^ p.io_flip;
        return (unsigned)iy < (unsigned)p.h && (unsigned)ix < (unsigned)p.w_ ? v : fill;
    };
    const int4 b4 = *reinterpret_cast<const int4 *>(p.bias_folded + cq * 4);
    int acc0 = b4.x, acc1 = b4.y, acc2 = b4.z, acc3 = b4.w;
    auto accumulate = [&](int pr, uint32_t lo, uint32_t hi) {
        const int4 w4 = *reinterpret_cast<const int4 *>(p.w_pair + ((Offset)pr * (Offset)p.cout + (Offset)(cq * 4)));
        acc0 = dot2(pair_bytes<0>(lo, hi), w4.x, acc0);
        acc1 = dot2(pair_bytes<1>(lo, hi), w4.y, acc1);
        acc2 = dot2(pair_bytes<2>(lo, hi), w4.z, acc2);
        acc3 = dot2(pair_bytes<3>(lo, hi), w4.w, acc3);
    };
    if constexpr (KH != 0) {
#pragma unroll
        for (int pr = 0; pr < (KH * KW + 1) / 2; ++pr) {
            constexpr int kw_c = KW ? KW : 1;
            const int t = 2 * pr;
            accumulate(pr, tap_at(t / kw_c, t % kw_c), t + 1 < KH * KW ? tap_at((t + 1) / kw_c, (t + 1) % kw_c) : 0u);
        }
    } else {
        // taps in row-major order, two per step; (ky, kx) walk along without a division per tap
        int ky = 0, kx = 0;
        auto next = [&]() -> uint32_t {
            const uint32_t v = ky < kh ? tap_at(ky, kx) : 0u;
            if (++kx == kw) kx = 0, ++ky;
            return v;
        };
        int pr = 0;
        for (; pr + 4 <= pairs; pr += 4) {  // eight taps requested before the first is used
            uint32_t v[8];
#pragma unroll
            for (int i = 0; i < 8; ++i) v[i] = next();
#pragma unroll
            for (int i = 0; i < 4; ++i) accumulate(pr + i, v[2 * i], v[2 * i + 1]);
        }
        for (; pr < pairs; ++pr) {
            const uint32_t lo = next(), hi = next();
            accumulate(pr, lo, hi);
        }
    }
    *reinterpret_cast<uint32_t *>(p.out + (pix * (Offset)p.cout + (Offset)(cq * 4))) =
        requant4(acc0, acc1, acc2, acc3, p.rq, load_channel_quad<true>(p.rq, (uint32_t)cq * 4u)) ^ p.io_flip;
}

// 3x3, dilation 1, stride S in both directions: a thread owns four adjacent channels of FOUR
// horizontally adjacent output pixels.  The 3 x (3 * S + 3) input pixels they need are loaded
// once (every load is issued before the first use, from clamped in-image addresses; taps
// outside the image are then replaced by the input zero point), so the address arithmetic, the
// weight and bias loads and the border tests are shared by sixteen outputs.
template <int S, bool PC, bool FLIP>
__global__ __launch_bounds__(256) void dw3x3_nhwc_tile4_kernel(const DwProblem p, const uint32_t total, const int tiles_x,
                                                               const FastDiv div_cq, const FastDiv div_tiles, const FastDiv div_ho) {
    constexpr int TW = 4, IW = (TW - 1) * S + 3;
    const uint32_t idx = xcd_contiguous_block() * 256u + threadIdx.x;
    if (idx >= total) return;
    // idx -> (image, output row, tile of four output columns, channel quad), channel quad fastest;
    // all offsets fit 32 bits (the launcher checks the tensor sizes)
    const uint32_t cq_count = (uint32_t)p.c >> 2;
    uint32_t r = fastdiv(idx, div_cq);
    const uint32_t cq = idx - r * cq_count;
    const uint32_t r2 = fastdiv(r, div_tiles);
    const int tx = (int)(r - r2 * (uint32_t)tiles_x);
    const uint32_t img = fastdiv(r2, div_ho);
    const int oy = (int)(r2 - img * (uint32_t)p.ho);
    const int ox0 = tx * TW;
    const int iy0 = oy * S - p.pad_t, ix0 = ox0 * S - p.pad_l;
    const uint32_t fill = (uint32_t)p.zp_in * 0x01010101u;
    const uint32_t base = img * (uint32_t)(p.h * p.w_ * p.c) + cq * 4u;

    uint32_t col_off[IW];
    bool col_ok[IW];
#pragma unroll
    for (int x = 0; x < IW; ++x) {
        const int ix = ix0 + x;
        col_ok[x] = (unsigned)ix < (unsigned)p.w_;
        const int ixc = ix < 0 ? 0 : (ix >= p.w_ ? p.w_ - 1 : ix);
        col_off[x] = base + (uint32_t)ixc * (uint32_t)p.c;
    }
    uint32_t in[3][IW];
#pragma unroll
    for (int ky = 0; ky < 3; ++ky) {
        const int iy = iy0 + ky;
        const bool row_ok = (unsigned)iy < (unsigned)p.h;
        const int iyc = iy < 0 ? 0 : (iy >= p.h ? p.h - 1 : iy);
        const uint32_t row_off = (uint32_t)iyc * (uint32_t)(p.w_ * p.c);
#pragma unroll
        for (int x = 0; x < IW; ++x) {
            const uint32_t v = *reinterpret_cast<const uint32_t *>(p.in + (row_off + col_off[x]));
            in[ky][x] = row_ok && col_ok[x] ? (FLIP ? v ^ 0x80808080u : v) : fill;
        }
    }
    int4 w4[5];
#pragma unroll
    for (int pr = 0; pr < 5; ++pr) w4[pr] = *reinterpret_cast<const int4 *>(p.w_pair + ((uint32_t)pr * (uint32_t)p.cout + cq * 4u));
    const int4 b4 = *reinterpret_cast<const int4 *>(p.bias_folded + cq * 4u);
    uint8_t *dst = p.out + (((img * (uint32_t)p.ho + (uint32_t)oy) * (uint32_t)p.wo + (uint32_t)ox0) * (uint32_t)p.cout + cq * 4u);
    const RequantDev rq = p.rq;
#pragma unroll
    for (int j = 0; j < TW; ++j) {
        int acc0 = b4.x, acc1 = b4.y, acc2 = b4.z, acc3 = b4.w;
#pragma unroll
        for (int pr = 0; pr < 5; ++pr) {
            const int t0 = 2 * pr, t1 = 2 * pr + 1;
            const uint32_t lo = in[t0 / 3][j * S + t0 % 3];
            const uint32_t hi = t1 < 9 ? in[t1 / 3][j * S + t1 % 3] : 0u;
            acc0 = dot2(pair_bytes<0>(lo, hi), w4[pr].x, acc0);
            acc1 = dot2(pair_bytes<1>(lo, hi), w4[pr].y, acc1);
            acc2 = dot2(pair_bytes<2>(lo, hi), w4[pr].z, acc2);
            acc3 = dot2(pair_bytes<3>(lo, hi), w4[pr].w, acc3);
        }
        uint32_t o = requant4<PC>(acc0, acc1, acc2, acc3, rq, load_channel_quad<PC>(rq, cq * 4u));
        if (FLIP) o ^= 0x80808080u;
        if (ox0 + j < p.wo) *reinterpret_cast<uint32_t *>(dst + (uint32_t)j * (uint32_t)p.cout) = o;
    }
}

// byte J of three rows' words into bytes 0, 1, 2 of one word (byte 3 zero): the three vertical taps of one channel
template <int J>
__device__ __forceinline__ uint32_t column_bytes(uint32_t r0, uint32_t r1, uint32_t r2) {
    constexpr uint32_t sel01 = (0x0cu << 24) | (0x0cu << 16) | ((4u + J) << 8) | (uint32_t)J;
    constexpr uint32_t sel2 = (0x0cu << 24) | ((4u + J) << 16) | (1u << 8) | 0u;
    return __builtin_amdgcn_perm(r2, __builtin_amdgcn_perm(r1, r0, sel01), sel2);
}

// The same for the four channels of a column at once, in six permutes instead of eight: the first two rows are
// interleaved pairwise (channels 0 and 1 in one word, 2 and 3 in the other), and each channel's word then takes its
// pair and its byte of the third row.
__device__ __forceinline__ void column_words(uint32_t r0, uint32_t r1, uint32_t r2, uint32_t (&out)[4]) {
    const uint32_t t01 = __builtin_amdgcn_perm(r1, r0, 0x05010400u);  // r0.b0 r1.b0 r0.b1 r1.b1
    const uint32_t t23 = __builtin_amdgcn_perm(r1, r0, 0x07030602u);  // r0.b2 r1.b2 r0.b3 r1.b3
    out[0] = __builtin_amdgcn_perm(r2, t01, 0x0c040100u);
    out[1] = __builtin_amdgcn_perm(r2, t01, 0x0c050302u);
    out[2] = __builtin_amdgcn_perm(r2, t23, 0x0c060100u);
    out[3] = __builtin_amdgcn_perm(r2, t23, 0x0c070302u);
}

// The same tile with 8-bit dot products, for weights whose differences w - zp_w all fit int8 (per-tensor
// requantization): activations as a - 128, the three vertical taps of a channel and column gathered into one word
// once and used by every output that touches the column (v_dot4_i32_i8 against the column's three weights), the
// term (zp_in - 128) * sum (w - zp_w) folded into the bias.  Six instructions per output for the taps instead of ten.
// TW output pixels per thread: four, or eight for stride 1 on rows that are whole tiles of eight (the column words and
// the index arithmetic are then shared by twice as many outputs).
// PC: one multiplier and shift per channel, all inside the single-shift form's range (p.rq.fast != 0).
// FOLD: weights of any range.  The products are then unsigned dot products of the raw bytes a and w, and
//     sum (a - za)(w - zw) = sum a w - zw * sum a - za * sum w + 9 za zw
// with the last two terms folded into the bias and sum a (nine taps, those outside the image reading za) taken from
// per-column sums that neighbouring outputs share: one more dot product per column and channel.  p.zp_w is then the
// zero point of the uint8 values being multiplied (int8 weights: + 128).
// D: the dilation (stride 1 only).  2 or 4: the tile's outputs j and j + D share input columns, so it reads
// TW + 2 D columns.  0: any dilation, read from the problem; no column is shared then and the tile reads three groups of
// TW adjacent columns, one per kernel column (what remains shared is the index arithmetic, the weights and the
// border tests).
// GATHER: a pixel of the input holds p.gather_c channels, any number from four on, each read by as many output channels as the
// multiplier says, and one of the output p.out_c; p.c and p.cout count those of the padded weights.  A thread loads the word of a pixel that holds its quad's
// input channels from where it lies and brings the channels to their places with one permute.  (Before, by a copy of the input with
// each channel as often as it is read and whole quads, and a copy of the result without the padding, us: 103
// channels at 22x22, 3 images 10.2 -> 3.9; 143 at 56x56, 32 images 31.6 -> 15.7; 119 at 40x40 stride 2, int8 with a pair per channel, 58
// images 19.1 -> 7.1; 112 x 2 at 86x86 stride 2, 60 images 96 -> 27; 50 x 2 at 28x28, 4 images 7.7 -> 4.0.)
__device__ __forceinline__ int udot4(uint32_t a, uint32_t b, int acc) { return (int)__builtin_amdgcn_udot4(a, b, (uint32_t)acc, false); }

template <int S, bool FLIP, int TW = 4, bool PC = false, bool FOLD = false, int D = 1, bool GATHER = false>
__global__ __launch_bounds__(256) void dw3x3_nhwc_tile4_dot4_kernel(const DwProblem p, const uint32_t total, const int tiles_x,
                                                                    const FastDiv div_cq, const FastDiv div_tiles, const FastDiv div_ho) {
    static_assert(D == 1 || S == 1, "dilated tiles are stride 1");
    constexpr int IW = D ? (TW - 1) * S + 2 * D + 1 : 3 * TW;
    const int dil = D ? D : p.dil_w;
    // tile column x lies this many pixels right of the tile's first input column; output j's tap kx reads tile column col_of(j, kx)
    auto x_offset = [&](int x) { return D ? x : (x / TW) * dil + (x % TW); };
    auto col_of = [](int j, int kx) { return D ? j * S + kx * D : kx * TW + j; };
    const uint32_t idx = xcd_contiguous_block() * 256u + threadIdx.x;
    if (idx >= total) return;
    const uint32_t cq_count = (uint32_t)p.c >> 2;
    uint32_t r = fastdiv(idx, div_cq);
    const uint32_t cq = idx - r * cq_count;
    const uint32_t r2 = fastdiv(r, div_tiles);
    const int tx = (int)(r - r2 * (uint32_t)tiles_x);
    const uint32_t img = fastdiv(r2, div_ho);
    const int oy = (int)(r2 - img * (uint32_t)p.ho);
    const int ox0 = tx * TW;
    const int iy0 = oy * S - p.pad_t, ix0 = ox0 * S - p.pad_l;
    // what a tap outside the image reads, as an operand of the form in use: the input zero point (FOLD) or that minus 128
    const uint32_t fill = ((uint32_t)p.zp_in * 0x01010101u) ^ (FOLD ? 0u : 0x80808080u);
    // uint8 tensors hold a, int8 tensors a - 128: the signed form wants a - 128, the unsigned one a
    constexpr bool flip_loaded = FOLD ? FLIP : !FLIP;
    const int in_c = GATHER ? p.gather_c : p.c, out_c = GATHER ? p.out_c : p.cout;
    uint32_t first = cq * 4u, select = 0;
    if constexpr (GATHER) {
        // the word of a pixel that holds the quad's input channels, the last one that lies in the pixel whole, and their places in it
        const uint32_t channel = fastdiv(first, p.gather_div);
        const uint32_t start = channel < (uint32_t)in_c - 4u ? channel : (uint32_t)in_c - 4u;
#pragma unroll
        for (uint32_t j = 0; j < 4; ++j) {
            const uint32_t oc = first + j < (uint32_t)out_c ? first + j : (uint32_t)out_c - 1u;
            select |= (fastdiv(oc, p.gather_div) - start) << (8 * j);
        }
        first = start;
    }
    const uint32_t base = img * (uint32_t)(p.h * p.w_ * in_c) + first;
    using Word = std::conditional_t<GATHER, const u32_any_alignment, const uint32_t>;
    auto load = [&](const uint8_t *from) {
        const uint32_t v = *reinterpret_cast<Word *>(from);
        return GATHER ? __builtin_amdgcn_perm(0u, v, select) : v;
    };

    // (row pitch and pixel offsets stay below 2^24, which the launcher checks: 24-bit multiplies run at full rate,
    // 32-bit ones at a quarter of it)
    const int row_pitch = p.w_ * in_c;
    uint32_t in[3][IW];
    const bool inside = iy0 >= 0 && iy0 + 2 * dil < p.h && ix0 >= 0 && ix0 + x_offset(IW - 1) < p.w_;
    if (__builtin_amdgcn_ballot_w64(!inside) == 0) {
        // every window of the wave lies inside the image (most waves): no clamps, no selects, offsets that differ
        // between the loads by wave-uniform amounts; a wave with one window on the border takes the general path whole
        const uint8_t *src = p.in + (base + (uint32_t)__mul24(iy0, row_pitch) + (uint32_t)__mul24(ix0, in_c));
#pragma unroll
        for (int ky = 0; ky < 3; ++ky)
#pragma unroll
            for (int x = 0; x < IW; ++x) {
                const uint32_t v = load(src + (uint32_t)(ky * dil * row_pitch + x_offset(x) * in_c));
                in[ky][x] = flip_loaded ? v ^ 0x80808080u : v;
            }
    } else {
        uint32_t col_off[IW];
        bool col_ok[IW];
#pragma unroll
        for (int x = 0; x < IW; ++x) {
            const int ix = ix0 + x_offset(x);
            col_ok[x] = (unsigned)ix < (unsigned)p.w_;
            const int ixc = ix < 0 ? 0 : (ix >= p.w_ ? p.w_ - 1 : ix);
            col_off[x] = base + (uint32_t)__mul24(ixc, in_c);
        }
#pragma unroll
        for (int ky = 0; ky < 3; ++ky) {
            const int iy = iy0 + ky * dil;
            const bool row_ok = (unsigned)iy < (unsigned)p.h;
            const int iyc = iy < 0 ? 0 : (iy >= p.h ? p.h - 1 : iy);
            const uint32_t row_off = (uint32_t)__mul24(iyc, row_pitch);
#pragma unroll
            for (int x = 0; x < IW; ++x) {
                const uint32_t v = load(p.in + (row_off + col_off[x]));
                in[ky][x] = row_ok && col_ok[x] ? (flip_loaded ? v ^ 0x80808080u : v) : fill;
            }
        }
    }
    int4 wk[3];
#pragma unroll
    for (int kx = 0; kx < 3; ++kx) wk[kx] = *reinterpret_cast<const int4 *>((FOLD ? p.w_fold : p.w_trip) + ((uint32_t)kx * (uint32_t)p.cout + cq * 4u));
    const int4 b4 = *reinterpret_cast<const int4 *>((FOLD ? p.bias_fold : p.bias_trip) + cq * 4u);
    uint32_t col[IW][4];
    int cs[FOLD ? IW : 1][4];  // FOLD: sum of the column's three bytes
#pragma unroll
    for (int x = 0; x < IW; ++x) {
        column_words(in[0][x], in[1][x], in[2][x], col[x]);
        if constexpr (FOLD) {
#pragma unroll
            for (int c = 0; c < 4; ++c) cs[x][c] = udot4(col[x][c], 0x00010101u, 0);
        }
    }
    uint8_t *dst = p.out + (((img * (uint32_t)p.ho + (uint32_t)oy) * (uint32_t)p.wo + (uint32_t)ox0) * (uint32_t)out_c + cq * 4u);
    const RequantDev rq = p.rq;
    const ChannelQuad quad = load_channel_quad<PC>(rq, cq * 4u);
#pragma unroll
    for (int j = 0; j < TW; ++j) {
        int acc0 = b4.x, acc1 = b4.y, acc2 = b4.z, acc3 = b4.w;
#pragma unroll
        for (int kx = 0; kx < 3; ++kx) {
            if constexpr (FOLD) {
                acc0 = udot4(col[col_of(j, kx)][0], (uint32_t)wk[kx].x, acc0);
                acc1 = udot4(col[col_of(j, kx)][1], (uint32_t)wk[kx].y, acc1);
                acc2 = udot4(col[col_of(j, kx)][2], (uint32_t)wk[kx].z, acc2);
                acc3 = udot4(col[col_of(j, kx)][3], (uint32_t)wk[kx].w, acc3);
            } else {
                acc0 = __builtin_amdgcn_sdot4((int)col[col_of(j, kx)][0], wk[kx].x, acc0, false);
                acc1 = __builtin_amdgcn_sdot4((int)col[col_of(j, kx)][1], wk[kx].y, acc1, false);
                acc2 = __builtin_amdgcn_sdot4((int)col[col_of(j, kx)][2], wk[kx].z, acc2, false);
                acc3 = __builtin_amdgcn_sdot4((int)col[col_of(j, kx)][3], wk[kx].w, acc3, false);
            }
        }
        if constexpr (FOLD) {
            // (nine bytes times a zero point of at most 383: a 24-bit multiply-add)
            acc0 += __mul24(-p.zp_w, cs[col_of(j, 0)][0] + cs[col_of(j, 1)][0] + cs[col_of(j, 2)][0]);
            acc1 += __mul24(-p.zp_w, cs[col_of(j, 0)][1] + cs[col_of(j, 1)][1] + cs[col_of(j, 2)][1]);
            acc2 += __mul24(-p.zp_w, cs[col_of(j, 0)][2] + cs[col_of(j, 1)][2] + cs[col_of(j, 2)][2]);
            acc3 += __mul24(-p.zp_w, cs[col_of(j, 0)][3] + cs[col_of(j, 1)][3] + cs[col_of(j, 2)][3]);
        }
        uint32_t o = PC ? requant4_channel_fast(acc0, acc1, acc2, acc3, rq, quad) : requant4<false>(acc0, acc1, acc2, acc3, rq, quad);
        if (FLIP) o ^= 0x80808080u;
        if (ox0 + j < p.wo) {
            uint8_t *const to = dst + (uint32_t)j * (uint32_t)out_c;
            if constexpr (GATHER) {
                const int left = out_c - (int)cq * 4;
                if (left >= 4) {
                    *reinterpret_cast<u32_any_alignment *>(to) = o;
                } else {
#pragma unroll
                    for (int i = 0; i < 3; ++i)
                        if (i < left) to[i] = (uint8_t)(o >> (8 * i));
                }
            } else {
                *reinterpret_cast<uint32_t *>(to) = o;
            }
        }
    }
}

// Planar tensors, K x K windows, stride S, no dilation: a thread owns four horizontally adjacent outputs of R rows of one plane.
//
// A row of a plane is what 8-bit dot products want: an output's taps of a kernel row are neighbouring bytes, with no gather.  The thread
// loads the aligned words of each input row under its windows, shifts them to its first column by one byte alignment each, and replaces
// what lies outside the image by masks that are the same for all its rows.  Weights are the caller's bytes as uint8; their zero point
// enters through the windows' sums.  Bound by those instructions on large tensors, some 25 per output at 5x5.
// Before -> here, us.  Through channels-last and back, three launches: 3x3 29 images of 232 channels at 8x7 9.7 -> 4.0, 32 of 144 at 56x56
// 27.3 -> 13.0; 5x5 64 of 144 at 56x56 53.0 -> 37.5; 7x7 2 of 520 at 13x7 11.5 -> 3.6.  One output to a thread, where the channels were no
// multiple of four or had a multiplier: 5x5 3 of 171 at 103x103 76 -> 11.2, 7x7 8 of 64 x 2 at 40x40 35.8 -> 6.2.
template <int K, int S, int R, bool PC>
__global__ __launch_bounds__(256) void dw_planar_kernel(const DwProblem p, const uint32_t total, const int quads, const int bands, const FastDiv div_quads,
                                                        const FastDiv div_bands, const FastDiv div_cout, const FastDiv div_dm) {
    constexpr int F = (K + 3) / 4, ND = (3 * S + 4 * F - 1) / 4 + 1, ROWS = (R - 1) * S + K;  // words per kernel row, per input row; input rows
    const uint32_t idx = xcd_contiguous_block() * 256u + threadIdx.x;
    if (idx >= total) return;
    const uint32_t r = fastdiv(idx, div_quads), plane = fastdiv(r, div_bands);
    const int ox0 = (int)(idx - r * (uint32_t)quads) * 4, oy0 = (int)(r - plane * (uint32_t)bands) * R;
    const uint32_t img = fastdiv(plane, div_cout), oc = plane - img * (uint32_t)p.cout;
    const uint32_t in_plane = img * (uint32_t)p.c + fastdiv(oc, div_dm);
    const int ix0 = ox0 * S - p.pad_l, iy0 = oy0 * S - p.pad_t;
    // the tensor from the word that it starts in to the one that it ends in: an aligned word with a byte of the tensor may be read whole
    const uint32_t lead = (uint32_t)reinterpret_cast<uintptr_t>(p.in) & 3u;
    const auto in = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t *>(p.in) - lead, 0,
                                                      (int)((lead + (uint32_t)p.n * (uint32_t)p.c * (uint32_t)p.h * (uint32_t)p.w_ + 3u) & ~3u), 0x00020000);
    const uint32_t fill = (uint32_t)p.zp_in * 0x01010101u;
    uint32_t keep[ND], pad[ND];
#pragma unroll
    for (int i = 0; i < ND; ++i) {  // bytes of word i left of the image, and those up to its right edge
        const int lo = -ix0 - 4 * i, hi = p.w_ - ix0 - 4 * i;
        const uint32_t below = lo <= 0 ? 0u : lo >= 4 ? ~0u : (1u << (8 * lo)) - 1u, upto = hi <= 0 ? 0u : hi >= 4 ? ~0u : (1u << (8 * hi)) - 1u;
        keep[i] = upto & ~below;
        pad[i] = fill & ~keep[i];
    }
    // kernel rows as words of uint8 taps, zero past the last one
    const uint32_t w_flip = p.w_signed ? 0x80808080u : 0u;
    const uint8_t *w = p.w + (size_t)oc * (K * K);
    uint32_t wk[K][F];
#pragma unroll
    for (int ky = 0; ky < K; ++ky)
#pragma unroll
        for (int f = 0; f < F; ++f) {
            const int taps = K - 4 * f < 4 ? K - 4 * f : 4;
            const uint32_t v = *reinterpret_cast<const u32_any_alignment *>(w + ky * K + f * 4);  // (the plan's copy ends in four bytes of slack)
            wk[ky][f] = (v ^ w_flip) & (taps == 4 ? ~0u : (1u << (8 * taps)) - 1u);
        }
    const int bias = p.bias_folded[oc];
    ChannelQuad quad{};
    if constexpr (PC) {
        const int m = p.rq.pc_multiplier[oc], sh = p.rq.pc_shift[oc];
        quad.m = make_int4(m, m, m, m);
        quad.s = make_int4(sh, sh, sh, sh);
    }
    int acc[R][4], sum[R][4];
#pragma unroll
    for (int o = 0; o < R; ++o)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            acc[o][j] = bias;
            sum[o][j] = 0;
        }
    const int row0 = (int)(lead + in_plane * (uint32_t)(p.h * p.w_)) + ix0;
#pragma unroll
    for (int row = 0; row < ROWS; ++row) {
        const int iy = iy0 + row;
        const bool exists = (unsigned)iy < (unsigned)p.h;
        const int off = exists ? row0 + iy * p.w_ : 0, at = off < 0 ? 0 : off;  // (below zero: the tensor's first row, left of it)
        uint32_t d[ND + 1], x[ND];
        const int from = at & ~3;
        if constexpr (ND == 2) {
            const auto v = __builtin_amdgcn_raw_buffer_load_b96(in, from, 0, 0);
            d[0] = v[0], d[1] = v[1], d[2] = v[2];
        } else {
            const auto v = __builtin_amdgcn_raw_buffer_load_b128(in, from, 0, 0);
            d[0] = v[0], d[1] = v[1], d[2] = v[2], d[3] = v[3];
            if constexpr (ND == 4) d[4] = __builtin_amdgcn_raw_buffer_load_b32(in, from + 16, 0, 0);
        }
#pragma unroll
        for (int i = 0; i < ND; ++i) x[i] = __builtin_amdgcn_alignbyte(d[i + 1], d[i], (uint32_t)at);
        if (off < 0) {
#pragma unroll
            for (int i = ND - 1; i >= 0; --i) x[i] = __builtin_amdgcn_alignbyte(x[i], i ? x[i - 1] : 0u, (uint32_t)(4 + off));
        }
#pragma unroll
        for (int i = 0; i < ND; ++i) x[i] = exists ? ((x[i] ^ p.io_flip) & keep[i]) | pad[i] : fill;
        uint32_t win[4][F];
        int row_sum[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            row_sum[j] = 0;
#pragma unroll
            for (int f = 0; f < F; ++f) {
                const int b = j * S + f * 4;
                win[j][f] = (b & 3) == 0 ? x[b >> 2] : __builtin_amdgcn_alignbyte((b >> 2) + 1 < ND ? x[(b >> 2) + 1 < ND ? (b >> 2) + 1 : 0] : 0u, x[b >> 2], b & 3);
                const int taps = K - 4 * f < 4 ? K - 4 * f : 4;
                row_sum[j] = udot4(win[j][f], 0x01010101u >> (8 * (4 - taps)), row_sum[j]);
            }
        }
#pragma unroll
        for (int ky = 0; ky < K; ++ky) {
            if (row < ky || (row - ky) % S != 0 || (row - ky) / S >= R) continue;
            const int o = (row - ky) / S;
#pragma unroll
            for (int j = 0; j < 4; ++j) {
#pragma unroll
                for (int f = 0; f < F; ++f) acc[o][j] = udot4(win[j][f], wk[ky][f], acc[o][j]);
                sum[o][j] += row_sum[j];
            }
        }
    }
    const int zw = p.zp_w + (p.w_signed ? 128 : 0);
    const RequantDev rq = p.rq;
    const uint32_t out_plane = plane * (uint32_t)(p.ho * p.wo);
#pragma unroll
    for (int o = 0; o < R; ++o) {
        if (oy0 + o >= p.ho) break;
        int a[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) a[j] = acc[o][j] - __mul24(zw, sum[o][j]);  // (49 bytes times a zero point of at most 383)
        const uint32_t v = (PC && rq.fast ? requant4_channel_fast(a[0], a[1], a[2], a[3], rq, quad) : requant4<PC>(a[0], a[1], a[2], a[3], rq, quad)) ^ p.io_flip;
        uint8_t *dst = p.out + (out_plane + (uint32_t)(oy0 + o) * (uint32_t)p.wo + (uint32_t)ox0);
        if (ox0 + 4 <= p.wo) {
            *reinterpret_cast<u32_any_alignment *>(dst) = v;
        } else {
#pragma unroll
            for (int j = 0; j < 3; ++j)
                if (ox0 + j < p.wo) dst[j] = (uint8_t)(v >> (8 * j));
        }
    }
}

// One output element per thread; any depth multiplier, dilation, channel count.
// NHWC = true: channel fastest.  NHWC = false: planar NCHW, x fastest.
template <bool NHWC>
__global__ __launch_bounds__(256) void dw_scalar_kernel(const DwProblem p, const long total) {
    const long idx = (long)blockIdx.x * 256 + threadIdx.x;
    if (idx >= total) return;
    int oc, ox, oy, img;
    if (total < (1l << 31)) {  // (uniform) 32-bit divisions: a fraction of the 64-bit ones' instructions
        const uint32_t i = (uint32_t)idx, d0 = (uint32_t)(NHWC ? p.cout : p.wo), d2 = (uint32_t)(NHWC ? p.ho : p.cout);
        const uint32_t d1 = (uint32_t)(NHWC ? p.wo : p.ho);
        const uint32_t r0 = i / d0, r1 = r0 / d1, r2 = r1 / d2;
        const int f0 = (int)(i - r0 * d0), f1 = (int)(r0 - r1 * d1), f2 = (int)(r1 - r2 * d2);
        img = (int)r2;
        if (NHWC)
            oc = f0, ox = f1, oy = f2;
        else
            ox = f0, oy = f1, oc = f2;
    } else if (NHWC) {
        oc = (int)(idx % p.cout);
        long r = idx / p.cout;
        ox = (int)(r % p.wo);
        r /= p.wo;
        oy = (int)(r % p.ho);
        img = (int)(r / p.ho);
    } else {
        ox = (int)(idx % p.wo);
        long r = idx / p.wo;
        oy = (int)(r % p.ho);
        r /= p.ho;
        oc = (int)(r % p.cout);
        img = (int)(r / p.cout);
    }
    const int ic = oc / p.dm;
    int32_t acc = p.bias ? p.bias[oc] : 0;
    const int iy0 = oy * p.stride_h - p.pad_t, ix0 = ox * p.stride_w - p.pad_l;
    for (int ky = 0; ky < p.kh; ++ky) {
        const int iy = iy0 + ky * p.dil_h;
        if ((unsigned)iy >= (unsigned)p.h) continue;
        for (int kx = 0; kx < p.kw; ++kx) {
            const int ix = ix0 + kx * p.dil_w;
            if ((unsigned)ix >= (unsigned)p.w_) continue;
            const size_t a_idx = NHWC ? (((size_t)img * p.h + iy) * p.w_ + ix) * p.c + ic
                                      : (((size_t)img * p.c + ic) * p.h + iy) * p.w_ + ix;
            const int32_t a = (int32_t)(p.in[a_idx] ^ (p.io_flip & 0xFFu)) - p.zp_in;
            const uint8_t raw = p.w[((size_t)oc * p.kh + ky) * p.kw + kx];
            const int32_t w = (p.w_signed ? (int32_t)(int8_t)raw : (int32_t)raw) - p.zp_w;
            acc += a * w;
        }
    }
    p.out[idx] = (uint8_t)((p.rq.pc_multiplier ? requant_u8_channel(acc, p.rq.pc_multiplier[oc], p.rq.pc_shift[oc], p.rq)
                                                : requant_u8(acc, p.rq)) ^ (p.io_flip & 0xFFu));
}

__global__ void dw_pack_kernel(const uint8_t *w, const int32_t *bias, int32_t *w_pair, int32_t *bias_folded, int32_t cout,
                               int32_t taps, int32_t zp_in, int32_t zp_w, int32_t w_signed) {
    const int oc = blockIdx.x * blockDim.x + threadIdx.x;
    if (oc >= cout) return;
    int32_t sum = 0;
    const int pairs = (taps + 1) >> 1;
    for (int pr = 0; pr < pairs; ++pr) {
        auto value = [&](int t) {
            const uint8_t raw = w[(size_t)oc * taps + t];
            return (w_signed ? (int32_t)(int8_t)raw : (int32_t)raw) - zp_w;
        };
        const int32_t lo = value(2 * pr);
        const int32_t hi = 2 * pr + 1 < taps ? value(2 * pr + 1) : 0;
        sum += lo + hi;
        w_pair[(size_t)pr * cout + oc] = (int32_t)(((uint32_t)lo & 0xFFFFu) | ((uint32_t)hi << 16));
    }
    bias_folded[oc] = (bias ? bias[oc] : 0) - zp_in * sum;
}

// 3x3 weights [cout][9] -> w_trip[kx][cout]: the three vertical taps (w - zp_w, each known to fit int8) of column kx
// in bytes 0..2; bias_trip[c] = bias - (zp_in - 128) * sum (w - zp_w)
__global__ void dw_pack_trip_kernel(const uint8_t *w, const int32_t *bias, int32_t *w_trip, int32_t *bias_trip, int32_t cout,
                                    int32_t zp_in, int32_t zp_w, int32_t w_signed) {
    const int oc = blockIdx.x * blockDim.x + threadIdx.x;
    if (oc >= cout) return;
    int32_t sum = 0;
    for (int kx = 0; kx < 3; ++kx) {
        uint32_t word = 0;
        for (int ky = 0; ky < 3; ++ky) {
            const uint8_t raw = w[(size_t)oc * 9 + ky * 3 + kx];
            const int32_t v = (w_signed ? (int32_t)(int8_t)raw : (int32_t)raw) - zp_w;
            sum += v;
            word |= ((uint32_t)v & 255u) << (8 * ky);
        }
        w_trip[(size_t)kx * cout + oc] = (int32_t)word;
    }
    bias_trip[oc] = (bias ? bias[oc] : 0) - (zp_in - 128) * sum;
}

// 3x3 weights [cout][9] -> w_fold[kx][cout]: the three vertical taps of column kx as the uint8 values the unsigned
// form multiplies (int8 weights: byte + 128, `zp_w` being their zero point + 128) in bytes 0..2;
// bias_fold[c] = bias - zp_in * sum w + 9 * zp_in * zp_w
__global__ void dw_pack_fold_kernel(const uint8_t *w, const int32_t *bias, int32_t *w_fold, int32_t *bias_fold, int32_t cout,
                                    int32_t zp_in, int32_t zp_w, int32_t w_signed) {
    const int oc = blockIdx.x * blockDim.x + threadIdx.x;
    if (oc >= cout) return;
    int32_t sum = 0;
    for (int kx = 0; kx < 3; ++kx) {
        uint32_t word = 0;
        for (int ky = 0; ky < 3; ++ky) {
            const uint32_t v = (uint32_t)w[(size_t)oc * 9 + ky * 3 + kx] ^ (w_signed ? 0x80u : 0u);
            sum += (int32_t)v;
            word |= v << (8 * ky);
        }
        w_fold[(size_t)kx * cout + oc] = (int32_t)word;
    }
    bias_fold[oc] = (bias ? bias[oc] : 0) - zp_in * sum + 9 * zp_in * zp_w;
}

}  // namespace

int launch_dw_pack_fold(const uint8_t *w, const int32_t *bias, int32_t *w_fold, int32_t *bias_fold, int32_t cout, int32_t zp_in,
                        int32_t zp_w_u8, int32_t w_signed, hipStream_t stream) {
    if (cout <= 0) return EH_OK;
    hipLaunchKernelGGL(dw_pack_fold_kernel, dim3((cout + 127) / 128), dim3(128), 0, stream, w, bias, w_fold, bias_fold, cout, zp_in,
                       zp_w_u8, w_signed);
    EH_HIP(hipGetLastError());
    return EH_OK;
}

int launch_dw_pack(const uint8_t *w, const int32_t *bias, int32_t *w_pair, int32_t *bias_folded, int32_t cout,
                   int32_t taps, int32_t zp_in, int32_t zp_w, int32_t w_signed, hipStream_t stream) {
    if (cout <= 0) return EH_OK;
    hipLaunchKernelGGL(dw_pack_kernel, dim3((cout + 127) / 128), dim3(128), 0, stream, w, bias, w_pair, bias_folded, cout,
                       taps, zp_in, zp_w, w_signed);
    EH_HIP(hipGetLastError());
    return EH_OK;
}

int launch_dw_pack_trip(const uint8_t *w, const int32_t *bias, int32_t *w_trip, int32_t *bias_trip, int32_t cout, int32_t zp_in,
                        int32_t zp_w, int32_t w_signed, hipStream_t stream) {
    if (cout <= 0) return EH_OK;
    hipLaunchKernelGGL(dw_pack_trip_kernel, dim3((cout + 127) / 128), dim3(128), 0, stream, w, bias, w_trip, bias_trip, cout, zp_in, zp_w,
                       w_signed);
    EH_HIP(hipGetLastError());
    return EH_OK;
}

static long pairs_of(const DwProblem &p) { return ((long)p.kh * p.kw + 1) / 2; }

int launch_dwconv_nhwc(const DwProblem &caller_p, hipStream_t stream) {
    DwProblem p = caller_p;
    if (dw_mfma_applies(p)) return launch_dw_mfma(p, stream);
    const bool pc_two_step = p.rq.pc_multiplier != nullptr && !p.rq.fast;
    if (p.w_trip || pc_two_step) p.w_fold = nullptr;  // the signed form where it applies; per-channel pairs outside the single-shift range use the 16-bit kernel
    const long outs = (long)p.n * p.ho * p.wo * p.cout;
    if (outs <= 0) return EH_OK;
    const bool vec = p.dm == 1 && (p.c & 3) == 0 && (reinterpret_cast<uintptr_t>(p.in) & 3) == 0 &&
                     (reinterpret_cast<uintptr_t>(p.out) & 3) == 0;
    // (the dot product kernels index rows and pixels with 24-bit multiplies)
    const bool dot4_form = (p.w_trip || p.w_fold) && (p.rq.pc_multiplier == nullptr || p.rq.fast) && (long)p.w_ * p.c < (1l << 23) && p.h < (1 << 23);
    const bool dilated = p.dil_h > 1 && p.dil_h == p.dil_w && p.stride_h == 1 && dot4_form && (long)p.dil_h * p.w_ * p.c < (1l << 22);
    const bool tile3x3 = vec && p.kh == 3 && p.kw == 3 && ((p.dil_h == 1 && p.dil_w == 1) || dilated) && p.stride_h == p.stride_w &&
                         (p.stride_h == 1 || p.stride_h == 2) && (size_t)p.n * p.h * p.w_ * p.c < (1ull << 31) &&
                         (size_t)p.n * p.ho * p.wo * p.cout < (1ull << 31);
    if (tile3x3) {
        // zero point of the uint8 values the unsigned form multiplies (only here: the one-output-per-thread kernel reads
        // the weights as the caller quantized them)
        if (p.w_fold) p.zp_w += p.w_signed ? 128 : 0;
        const int tiles_x = (p.wo + 3) / 4;
        const long total = (long)p.n * p.ho * tiles_x * (p.c >> 2);
        const long blocks = (total + 255) / 256;
        EH_REQUIRE(total < (1l << 31), "depthwise: grid too large");
        const FastDiv d_cq = make_fastdiv((uint32_t)(p.c >> 2)), d_t = make_fastdiv((uint32_t)tiles_x), d_ho = make_fastdiv((uint32_t)p.ho);
        // per-channel pairs and int8 tensors are compile-time variants: the plain uint8 kernel pays for neither
        const bool pc = p.rq.pc_multiplier != nullptr, flip = p.io_flip != 0;
        auto pick = [&](auto stride_c) {
            constexpr int S = decltype(stride_c)::value;
            return pc ? (flip ? dw3x3_nhwc_tile4_kernel<S, true, true> : dw3x3_nhwc_tile4_kernel<S, true, false>)
                      : (flip ? dw3x3_nhwc_tile4_kernel<S, false, true> : dw3x3_nhwc_tile4_kernel<S, false, false>);
        };
        auto kernel = p.stride_h == 1 ? pick(std::integral_constant<int, 1>{}) : pick(std::integral_constant<int, 2>{});
        // 8-bit dot products: the signed form where every w - zp_w fits int8, else the unsigned form for any weights
        const bool fold = p.w_trip == nullptr;
        auto pick_dot4 = [&](auto s_tag, auto tw_tag) {
            constexpr int S = decltype(s_tag)::value, TW = decltype(tw_tag)::value;
            if (fold)
                return pc ? (flip ? dw3x3_nhwc_tile4_dot4_kernel<S, true, TW, true, true> : dw3x3_nhwc_tile4_dot4_kernel<S, false, TW, true, true>)
                          : (flip ? dw3x3_nhwc_tile4_dot4_kernel<S, true, TW, false, true> : dw3x3_nhwc_tile4_dot4_kernel<S, false, TW, false, true>);
            return pc ? (flip ? dw3x3_nhwc_tile4_dot4_kernel<S, true, TW, true> : dw3x3_nhwc_tile4_dot4_kernel<S, false, TW, true>)
                      : (flip ? dw3x3_nhwc_tile4_dot4_kernel<S, true, TW, false> : dw3x3_nhwc_tile4_dot4_kernel<S, false, TW, false>);
        };
        using tw4 = std::integral_constant<int, 4>;
        const bool dot4 = dot4_form;
        if (p.dil_h > 1) {
            // dilated, stride 1: the tiles that share columns for dilations 2 and 4, the three-group tile for the rest
            auto pick_dilated = [&](auto d_tag) {
                constexpr int D = decltype(d_tag)::value;
                if (fold)
                    return pc ? (flip ? dw3x3_nhwc_tile4_dot4_kernel<1, true, 4, true, true, D> : dw3x3_nhwc_tile4_dot4_kernel<1, false, 4, true, true, D>)
                              : (flip ? dw3x3_nhwc_tile4_dot4_kernel<1, true, 4, false, true, D> : dw3x3_nhwc_tile4_dot4_kernel<1, false, 4, false, true, D>);
                return pc ? (flip ? dw3x3_nhwc_tile4_dot4_kernel<1, true, 4, true, false, D> : dw3x3_nhwc_tile4_dot4_kernel<1, false, 4, true, false, D>)
                          : (flip ? dw3x3_nhwc_tile4_dot4_kernel<1, true, 4, false, false, D> : dw3x3_nhwc_tile4_dot4_kernel<1, false, 4, false, false, D>);
            };
            kernel = p.dil_h == 2   ? pick_dilated(std::integral_constant<int, 2>{})
                     : p.dil_h == 4 ? pick_dilated(std::integral_constant<int, 4>{})
                                    : pick_dilated(std::integral_constant<int, 0>{});
        } else if (dot4)
            kernel = p.stride_h == 1 ? pick_dot4(std::integral_constant<int, 1>{}, tw4{}) : pick_dot4(std::integral_constant<int, 2>{}, tw4{});
        if (dot4 && p.dil_h == 1 && p.stride_h == 1 && (p.wo & 7) == 0 && total >= (1l << 20)) {
            // large stride-1 layers with rows of whole eight-pixel tiles: eight outputs per thread
            const int tiles8 = p.wo / 8;
            const long total8 = (long)p.n * p.ho * tiles8 * (p.c >> 2);
            const FastDiv d_t8 = make_fastdiv((uint32_t)tiles8);
            auto kernel8 = pick_dot4(std::integral_constant<int, 1>{}, std::integral_constant<int, 8>{});
            hipLaunchKernelGGL(kernel8, dim3((unsigned)(((total8 + 255) / 256 + 7) / 8 * 8)), dim3(256), 0, stream, p, (uint32_t)total8, tiles8, d_cq, d_t8,
                               d_ho);
            EH_HIP(hipGetLastError());
            return EH_OK;
        }
        hipLaunchKernelGGL(kernel, dim3((unsigned)((blocks + 7) / 8 * 8)), dim3(256), 0, stream, p, (uint32_t)total, tiles_x, d_cq, d_t, d_ho);
    } else if (vec) {
        const long total = outs / 4;
        const long blocks = (total + 255) / 256;
        EH_REQUIRE(blocks < (1l << 31), "depthwise: grid too large");
        const bool small = (size_t)p.n * p.h * p.w_ * p.c < (1ull << 31) && outs < (1l << 31) && (size_t)pairs_of(p) * p.cout < (1ull << 30);
        const FastDiv d_cq = make_fastdiv((uint32_t)(p.c >> 2)), d_wo = make_fastdiv((uint32_t)p.wo), d_ho = make_fastdiv((uint32_t)p.ho);
        const bool k3 = p.kh == 3 && p.kw == 3;
        auto kernel = k3 ? (small ? dw_nhwc_vec4_kernel<3, 3, true> : dw_nhwc_vec4_kernel<3, 3, false>)
                         : (small ? dw_nhwc_vec4_kernel<0, 0, true> : dw_nhwc_vec4_kernel<0, 0, false>);
        hipLaunchKernelGGL(kernel, dim3((unsigned)((blocks + 7) / 8 * 8)), dim3(256), 0, stream, p, total, d_cq, d_wo, d_ho);
    } else {
        const long blocks = (outs + 255) / 256;
        EH_REQUIRE(blocks < (1l << 31), "depthwise: grid too large");
        hipLaunchKernelGGL((dw_scalar_kernel<true>), dim3((unsigned)blocks), dim3(256), 0, stream, p, outs);
    }
    EH_HIP(hipGetLastError());
    return EH_OK;
}

// The problem of a plan whose kernels' channels are not its tensors': the dot product form of 3x3 layers without dilation.
bool dw_gather_applies(const DwProblem &p) {
    return p.kh == 3 && p.kw == 3 && p.dil_h == 1 && p.dil_w == 1 && p.stride_h == p.stride_w && (p.stride_h == 1 || p.stride_h == 2) && (p.w_trip || p.w_fold) &&
           (p.rq.pc_multiplier == nullptr || p.rq.fast) && (long)p.w_ * p.c < (1l << 23) && p.h < (1 << 23) && p.gather_c >= 4 &&
           (size_t)p.n * p.h * p.w_ * p.c < (1ull << 31) && (size_t)p.n * p.ho * p.wo * p.cout < (1ull << 31);
}

int launch_dw_gather(const DwProblem &caller_p, hipStream_t stream) {
    DwProblem p = caller_p;
    const bool fold = p.w_trip == nullptr, pc = p.rq.pc_multiplier != nullptr, flip = p.io_flip != 0;
    if (fold) p.zp_w += p.w_signed ? 128 : 0;
    const int tiles_x = (p.wo + 3) / 4;
    const long total = (long)p.n * p.ho * tiles_x * (p.c >> 2);
    if (total <= 0) return EH_OK;
    auto pick = [&](auto stride_c) {
        constexpr int S = decltype(stride_c)::value;
        if (fold)
            return pc ? (flip ? dw3x3_nhwc_tile4_dot4_kernel<S, true, 4, true, true, 1, true> : dw3x3_nhwc_tile4_dot4_kernel<S, false, 4, true, true, 1, true>)
                      : (flip ? dw3x3_nhwc_tile4_dot4_kernel<S, true, 4, false, true, 1, true> : dw3x3_nhwc_tile4_dot4_kernel<S, false, 4, false, true, 1, true>);
        return pc ? (flip ? dw3x3_nhwc_tile4_dot4_kernel<S, true, 4, true, false, 1, true> : dw3x3_nhwc_tile4_dot4_kernel<S, false, 4, true, false, 1, true>)
                  : (flip ? dw3x3_nhwc_tile4_dot4_kernel<S, true, 4, false, false, 1, true> : dw3x3_nhwc_tile4_dot4_kernel<S, false, 4, false, false, 1, true>);
    };
    auto kernel = p.stride_h == 1 ? pick(std::integral_constant<int, 1>{}) : pick(std::integral_constant<int, 2>{});
    hipLaunchKernelGGL(kernel, dim3((unsigned)(((total + 255) / 256 + 7) / 8 * 8)), dim3(256), 0, stream, p, (uint32_t)total, tiles_x,
                       make_fastdiv((uint32_t)(p.c >> 2)), make_fastdiv((uint32_t)tiles_x), make_fastdiv((uint32_t)p.ho));
    EH_HIP(hipGetLastError());
    return EH_OK;
}

// (what a plan that keeps a caller's planar tensors planar has to be)
bool dw_planar_applies(const DwProblem &p) {
    return p.kh == p.kw && (p.kh == 3 || p.kh == 5 || p.kh == 7) && p.dil_h == 1 && p.dil_w == 1 && p.stride_h == p.stride_w &&
           (p.stride_h == 1 || p.stride_h == 2) && p.pad_l >= 0 && p.pad_l <= 3 && p.pad_t >= 0 && (size_t)p.n * p.c * p.h * p.w_ < (1ull << 31) - 64 &&
           (size_t)p.n * p.cout * p.ho * p.wo < (1ull << 31) - 64;
}

static int launch_dw_planar(const DwProblem &p, hipStream_t stream) {
    const int quads = (p.wo + 3) / 4;
    const long threads = (long)p.n * p.cout * quads;
    // Four rows to a thread share their input rows' loads and shifts; a launch that they would not fill has one.  One row and four, us, by
    // the threads of four: 6272 5x5 stride 2 4.3 and 5.6; 8320 7x7 3.6 and 4.9; 26912 3x3 4.0 and 4.0; 61440 7x7 stride 2 7.4 and 6.6;
    // 122880 5x5 6.9 and 6.1; 225792 3x3 6.8 and 5.6.
    const bool four = threads * ((p.ho + 3) / 4) >= 32768;
    auto launch = [&](auto k_c, auto s_c, auto r_c, auto pc_c) {
        constexpr int R = decltype(r_c)::value;
        const int bands = (p.ho + R - 1) / R;
        const uint32_t total = (uint32_t)(threads * bands);
        hipLaunchKernelGGL((dw_planar_kernel<decltype(k_c)::value, decltype(s_c)::value, R, decltype(pc_c)::value>), dim3(((total + 255) / 256 + 7) / 8 * 8), dim3(256), 0,
                           stream, p, total, quads, bands, make_fastdiv((uint32_t)quads), make_fastdiv((uint32_t)bands), make_fastdiv((uint32_t)p.cout),
                           make_fastdiv((uint32_t)p.dm));
    };
    using std::integral_constant;
    auto with_rows = [&](auto k_c, auto s_c) {
        auto with_pairs = [&](auto r_c) { p.rq.pc_multiplier ? launch(k_c, s_c, r_c, std::true_type{}) : launch(k_c, s_c, r_c, std::false_type{}); };
        four ? with_pairs(integral_constant<int, 4>{}) : with_pairs(integral_constant<int, 1>{});
    };
    auto with_stride = [&](auto k_c) { p.stride_h == 1 ? with_rows(k_c, integral_constant<int, 1>{}) : with_rows(k_c, integral_constant<int, 2>{}); };
    p.kh == 3 ? with_stride(integral_constant<int, 3>{}) : p.kh == 5 ? with_stride(integral_constant<int, 5>{}) : with_stride(integral_constant<int, 7>{});
    EH_HIP(hipGetLastError());
    return EH_OK;
}

int launch_dwconv_nchw(const DwProblem &p, hipStream_t stream) {
    const long outs = (long)p.n * p.ho * p.wo * p.cout;
    if (outs <= 0) return EH_OK;
    if (dw_planar_applies(p)) return launch_dw_planar(p, stream);
    const long blocks = (outs + 255) / 256;
    EH_REQUIRE(blocks < (1l << 31), "depthwise: grid too large");
    hipLaunchKernelGGL((dw_scalar_kernel<false>), dim3((unsigned)blocks), dim3(256), 0, stream, p, outs);
    EH_HIP(hipGetLastError());
    return EH_OK;
}

}  // namespace eh
