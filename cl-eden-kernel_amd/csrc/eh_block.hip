// Pointwise expansion + depthwise 3x3 as ONE launch (gfx950): the MobileNet-style block "1x1 convolution to C expanded
// channels, activation, requantization to uint8; then a 3x3 depthwise convolution over that tensor" without the
// expanded tensor ever leaving the CU.
//
// The reference runs the two operators one after the other on its queue (gpu/gpu_op_executor.cc:56-103:
// CLConvolution -> quantizedGemmBlocked writes the expanded tensor, CLDepthwiseConvolution ->
// depthwise_conv_3x3s2_pad_merge reads it back, cl_kernels/DepthwiseconvolutionKernels.cpp:1964-2083); at the block of
// BASELINE configs[2] the expanded tensor is 14.45 MB written and read again against 2.4 MB of input and 3.6 MB of
// output.  Here a workgroup owns a tile of TH x TW output pixels of one image:
//   0. the input pixels under the tile's windows ((TH - 1) * S + 3 rows by (TW - 1) * S + 3 columns, a few KB) are copied
//      to LDS with contiguous loads, beside the pointwise weights and bias;
//   1. the expanded pixels are computed by the matrix cores (one 32x32x32 int8 MFMA per 32 pixels and 32 channels; the
//      (pixel block, channel block) pairs are dealt out evenly over the four waves), requantized exactly as the
//      pointwise operator does it and written as uint8 into an LDS image [row][column][channel]; pixels outside the
//      image are written as the depthwise operator's input zero point, which is what its padding reads;
//   2. after one barrier the waves compute the depthwise outputs from that image on the matrix cores and store them.  One 16x16x64
//      product takes 16 pixels and, per pixel, 16 channels at up to four columns of a kernel row; its other operand is diagonal.
//      A wave takes 16 channels and walks down 16 columns of the tile (or 8 in two strips of rows, or 4 in four): an input row is
//      read once, multiplied by each kernel row that it meets, and the vector units are left with the requantization, some 20
//      instructions for 256 outputs.  (As 8-bit dot products, which want every channel's three rows gathered into a word first, a
//      thread's sixteen outputs were 300.)  Dot products -> walk, us: 24 -> 144 at 56x56, 23 images 16.1 -> 11.8; 64 -> 384 at
//      58x58, 16 images 32.7 -> 23; 16 -> 96 at 83x83, 21 images 21.4 -> 13.6; 56 -> 336 at 31x31, 18 images 13.4 -> 9.3; 120 -> 720
//      at 12x12, 18 images 9.2 -> 7.0; a pair per channel, 16 -> 96 at 104x97, 28 images 34.1 -> 26.6, 80 -> 480 at 36x36, 16 images
//      20.4 -> 15.0; at stride 2, where the expansion is most of the work, 24 -> 144 at 56x56, 32 images 11.3 and 11.3.
//      Small tiles at stride 2, and those that a caller asks for, are taken sixteen outputs at a time instead, wherever their rows end
//      (units_tile and pwdw_block_geometry have the rules).
// The rows and columns two neighbouring workgroups both need (the halo) are computed twice; nothing else is.  Tiles are
// cut in both directions because the halo of a stride-2 window costs (2 TH + 1)(2 TW + 1) / (4 TH TW): 1.53 for one full
// row of 28 outputs, 1.21 for 4 x 7.
// A depthwise channel needs only its own expanded channel, so the expanded channels are cut into ranges of whole
// 32-channel blocks as well: a workgroup is (tile, channel range), which keeps its LDS image small (four or more
// workgroups share a CU and overlap their stages) on layers with many channels; the input pixels are then staged once
// per range, which costs little (they are the narrow side of an expansion).
// Both stages produce bit for bit what the two stand-alone launches produce.
#include <type_traits>

#include "eh_internal.h"

namespace eh {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v16i __attribute__((ext_vector_type(16)));

namespace {

// S: depthwise stride.  FORM: how the depthwise stage multiplies (DwForm).  ROWSUM: the pointwise weights' zero point is not 128, so a pixel's byte sum enters.
// QM: pointwise requantization, 0 two-step order, 1 / 2 the single-shift forms.  KS: reduction steps of the pointwise
// stage when they are 1, 2 or 3 (a lane then keeps its pixel's operand bytes in registers across the channel blocks),
// 0 for any number (read from LDS for every product).
enum class DwForm {
    UNITS,  // small tiles at stride 2 or on request: sixteen outputs of the tile, wherever its rows end, by sixteen channels
    WALK    // the others: sixteen columns, down the tile's rows
};
// PC: one multiplier and shift per channel in both operators; the depthwise ones in the single-shift form, or in two steps.
enum class Pairs { TENSOR, CHANNEL, CHANNEL_TWO_STEP };
template <int S, DwForm FORM, bool ROWSUM, int QM, int KS, Pairs PAIRS>
__global__ __launch_bounds__(256) void pwdw_block_kernel(const GemmProblem pw, const DwProblem dw, const BlockGeom g) {
    constexpr bool WALK = FORM == DwForm::WALK, PC = PAIRS != Pairs::TENSOR, DW_TWO_STEP = PAIRS == Pairs::CHANNEL_TWO_STEP;
    const int ksteps = KS ? KS : g.ks;
    extern __shared__ __align__(16) uint8_t lds_raw[];
    v4i *b_s = reinterpret_cast<v4i *>(lds_raw);                              // [nb][ks][64 lanes]: pointwise weights, fragment order
    int32_t *bias_s = reinterpret_cast<int32_t *>(lds_raw + (size_t)g.nb * ksteps * 1024);  // [nb * 32]
    // PC: the pointwise stage's pairs beside the bias; the shifts as the bytes that requant4_channel wants or, two-step, as they are
    int32_t *pcm_s = bias_s + g.nb * 32, *pcf_s = pcm_s + g.nb * 32;
    uint8_t *pce_s = reinterpret_cast<uint8_t *>(pcf_s);
    uint8_t *img_s = lds_raw + g.image_off;                                   // [ih][iwp][cpitch] uint8 xor 0x80: operands
    const int nb_first = blockIdx.y * g.nb;                                   // this workgroup's channel range
    const int c_first = nb_first * 32;
    const int c_here = g.c - c_first < g.nb * 32 ? g.c - c_first : g.nb * 32;  // channels of the range that exist (a multiple of 16)
    const int nb_here = (c_here + 31) >> 5;
    const int cpitch = g.cpitch;

    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int r = lane & 31, half = lane >> 5;
    // every XCD takes a contiguous eighth of the tiles: the rows two neighbouring tiles share are then fetched into one L2
    const uint32_t tile = (blockIdx.x & 7u) * (gridDim.x >> 3) + (blockIdx.x >> 3);
    if (tile >= (uint32_t)g.total_tiles) return;
    const uint32_t t_row = fastdiv(tile, g.div_tiles_w);
    const int txw = (int)(tile - t_row * (uint32_t)g.tiles_w);
    const uint32_t img = fastdiv(t_row, g.div_tiles_y);
    const int ty = (int)(t_row - img * (uint32_t)g.tiles_y);
    const int oy0 = ty * g.th, ox_first = txw * g.tw;
    const int iy_first = oy0 * S - dw.pad_t, ix_first = ox_first * S - dw.pad_l;  // image coordinates of the LDS image's corner
    uint8_t *a_s = lds_raw + g.a_off;  // [pixels][a_pitch]: the input pixels' reduction bytes as signed operands (a ^ 0x80), 0 past the reduction length

    // The depthwise stage's units of (chunk of 16 channels, 16 output pixels or columns of output pixels), a contiguous share per
    // wave; lane (i, q) holds the weights of channel i of the chunk in kernel column q.  A wave's first chunk is requested ahead
    // of everything else.
    const int lane16 = lane & 15, quarter = lane >> 4, cpad = (g.c + 15) & ~15;
    const int out_pixels = g.th * g.tw, groups = WALK ? g.walk_groups : (out_pixels + 15) >> 4, w_uniform = __builtin_amdgcn_readfirstlane(wave);
    const int unit_first = ((c_here >> 4) * groups * w_uniform) >> 2, unit_last = ((c_here >> 4) * groups * (w_uniform + 1)) >> 2;
    struct DwPart {
        uint32_t w[3], neg;  // by kernel row; minus what the stored weights lack (dw_pack_mfma_kernel)
        int4 bias, mult, shift;
    };
    auto request_dw = [&](int chunk) {
        const int c0 = c_first + chunk * 16;
        DwPart d;
#pragma unroll
        for (int ky = 0; ky < 3; ++ky) d.w[ky] = dw.w_mm[(ky * 4 + quarter) * cpad + c0 + lane16];  // (column 3 is padding: zero)
        d.neg = dw.w_mm[12 * cpad + c0 + lane16];
        d.bias = *reinterpret_cast<const int4 *>(dw.bias_mm + c0 + quarter * 4);
        if constexpr (PC) {
            d.mult = *reinterpret_cast<const int4 *>(dw.rq.pc_multiplier + c0 + quarter * 4);
            d.shift = *reinterpret_cast<const int4 *>(dw.rq.pc_shift + c0 + quarter * 4);
        }
        return d;
    };
    int chunk = unit_first / groups, group = unit_first - chunk * groups;
    DwPart part{};
    if (unit_first < unit_last) part = request_dw(chunk);

    // ---- stage 0: weights, bias and the tile's input pixels into LDS (8-byte pieces: pixels start on 8-byte boundaries)
    auto inside_image = [&](int q, int &iy, int &ix) {
        const int ry = (int)fastdiv((uint32_t)q, g.div_iwp), rx = q - ry * g.iwp;
        iy = iy_first + ry;
        ix = ix_first + rx;
        return (unsigned)iy < (unsigned)pw.h && (unsigned)ix < (unsigned)pw.w;
    };
    {
        // The input pixels first, then the weights as direct-to-LDS copies, all on their way at once beside the bias.  A thread of a tile
        // that walks has two pieces on their way at a time, from clamped addresses without a branch: 24 -> 144 at 56x56 stride 2, 32
        // images, four pieces to a thread, 10.95 us one at a time and 10.8 so, on cold tensors 13.6 and 12.8.  (Four at a time cost a small
        // tile more instructions than they save trips: 40 -> 240 at 20x20 stride 2, six images, 5.13 us one at a time, 5.44 like that; 48
        // -> 288 at 33x33, four images 5.57 and 5.81; 64 -> 384 at 14x14, eight images 5.46 and 5.69.)
        const int ppp = ksteps * 4;  // 8-byte pieces per pixel
        const int pieces = g.pixels * ppp;
        constexpr int BATCH = WALK ? 2 : 1;
        for (int i0 = tid; i0 < pieces; i0 += 256 * BATCH) {
            uint2 v[BATCH];
            uint32_t to[BATCH];
            bool exists[BATCH];
#pragma unroll
            for (int b = 0; b < BATCH; ++b) {
                const int i = i0 + b * 256, q = KS ? i / (KS * 4) : (int)fastdiv((uint32_t)i, g.div_ppp), piece = i - q * ppp;
                int iy, ix;
                exists[b] = inside_image(q, iy, ix) && piece * 8 < pw.k;
                to[b] = (uint32_t)(q * g.a_pitch + piece * 8);
                v[b] = make_uint2(0u, 0u);
                const uint32_t from = ((img * (uint32_t)pw.h + (uint32_t)iy) * (uint32_t)pw.w + (uint32_t)ix) * (uint32_t)pw.cin + (uint32_t)pw.a_offset + (uint32_t)piece * 8u;
                if (WALK || exists[b]) v[b] = *reinterpret_cast<const uint2 *>(pw.a + (exists[b] ? from : 0u));
            }
#pragma unroll
            for (int b = 0; b < BATCH; ++b) {  // bytes past the reduction length, and whole pixels outside the image: operand 0
                const uint2 w = exists[b] ? make_uint2(v[b].x ^ pw.a_xor, v[b].y ^ pw.a_xor) : make_uint2(0u, 0u);
                if (b == 0 || i0 + b * 256 < pieces) *reinterpret_cast<uint2 *>(a_s + to[b]) = w;
            }
        }
        dma_linear<4>(pw.b + (size_t)nb_first * ksteps * 1024, lds_offset(lds_raw), nb_here * ksteps, w_uniform, lane);
        for (int i = tid; i < nb_here * 32; i += 256) bias_s[i] = pw.bias[c_first + i];
        if constexpr (PC) {  // (the per-channel arrays are padded to whole channel blocks)
            for (int i = tid; i < nb_here * 32; i += 256) {
                const int32_t m = pw.rq.pc_multiplier[c_first + i], sh = pw.rq.pc_shift[c_first + i];
                pcm_s[i] = m;
                if constexpr (QM != 0)
                    pce_s[i] = (uint8_t)(-2 - sh);
                else
                    pcf_s[i] = sh;
            }
        }
        wait_vmcnt<0>();
        __syncthreads();
    }

    // ---- stage 1: the expanded pixels into the LDS image.  Units of (pixel block, channel block), a contiguous share per wave.
    const uint32_t flip_store = 0x80808080u;  // the depthwise stage multiplies a - 128
    const uint32_t pad_word = ((uint32_t)dw.zp_in * 0x01010101u) ^ flip_store;
    const int blocks = (g.pixels + 31) >> 5;
    const RequantDev rq = pw.rq;
    {
        const int all = blocks * nb_here;
        const int first = (all * wave) >> 2, last = (all * (wave + 1)) >> 2;
        int blk = first / nb_here, nb = first - blk * nb_here;
        int loaded = -1, ncorr = 0, q = 0;
        bool ok = false;
        const uint8_t *arow = a_s;
        v4i held[KS ? KS : 1];
        for (int u = first; u < last; ++u) {
            if (blk != loaded) {  // this lane's pixel of the block: where its fragment bytes sit, its row-sum term, its place in the image
                loaded = blk;
                q = blk * 32 + r;
                int iy, ix;
                ok = q < g.pixels && inside_image(q, iy, ix);
                arow = a_s + (q < g.pixels ? q : g.pixels - 1) * g.a_pitch + half * 16;
                if constexpr (KS != 0) {
#pragma unroll
                    for (int ks = 0; ks < KS; ++ks) held[ks] = *reinterpret_cast<const v4i *>(arow + ks * 32);
                }
                if constexpr (ROWSUM) {
                    int rowsum = 0;
#pragma unroll
                    for (int ks = 0; ks < ksteps; ++ks) {
                        const v4i af = KS ? held[KS ? ks : 0] : *reinterpret_cast<const v4i *>(arow + ks * 32);
                        rowsum = __builtin_amdgcn_sdot4(af.x, 0x01010101, rowsum, false);
                        rowsum = __builtin_amdgcn_sdot4(af.y, 0x01010101, rowsum, false);
                        rowsum = __builtin_amdgcn_sdot4(af.z, 0x01010101, rowsum, false);
                        rowsum = __builtin_amdgcn_sdot4(af.w, 0x01010101, rowsum, false);
                    }
                    rowsum += __shfl_xor(rowsum, 32);  // the other half of every step's bytes
                    ncorr = -pw.zw * rowsum;
                }
            }
            const int32_t *bsrc = bias_s + nb * 32 + half * 16;
            v16i acc;
#pragma unroll
            for (int gq = 0; gq < 4; ++gq) {
                const int4 bb = *reinterpret_cast<const int4 *>(bsrc + gq * 4);
                acc[gq * 4 + 0] = bb.x;
                acc[gq * 4 + 1] = bb.y;
                acc[gq * 4 + 2] = bb.z;
                acc[gq * 4 + 3] = bb.w;
            }
            const v4i *bw = b_s + nb * ksteps * 64 + lane;
            if constexpr (KS != 0) {
#pragma unroll
                for (int ks = 0; ks < KS; ++ks) acc = __builtin_amdgcn_mfma_i32_32x32x32_i8(bw[ks * 64], held[ks], acc, 0, 0, 0);
            } else {
                for (int ks = 0; ks < ksteps; ++ks)
                    acc = __builtin_amdgcn_mfma_i32_32x32x32_i8(bw[ks * 64], *reinterpret_cast<const v4i *>(arow + ks * 32), acc, 0, 0, 0);
            }
            uint32_t packed[4];
            v4i e16 = {0, 0, 0, 0};
            if constexpr (PC && QM != 0) e16 = *reinterpret_cast<const v4i *>(pce_s + nb * 32 + half * 16);
#pragma unroll
            for (int gq = 0; gq < 4; ++gq) {
                if constexpr (PC) {
                    const int tab = nb * 32 + half * 16 + gq * 4;
                    const int4 cm = *reinterpret_cast<const int4 *>(pcm_s + tab);
                    if constexpr (QM != 0) {
                        packed[gq] = requant4_channel<QM>(acc[gq * 4 + 0] + ncorr, acc[gq * 4 + 1] + ncorr, acc[gq * 4 + 2] + ncorr, acc[gq * 4 + 3] + ncorr, cm,
                                                          (uint32_t)e16[gq], rq);
                    } else {
                        const int4 cf = *reinterpret_cast<const int4 *>(pcf_s + tab);
                        packed[gq] = pack_bytes(requant_u8_channel(acc[gq * 4 + 0] + ncorr, cm.x, cf.x, rq), requant_u8_channel(acc[gq * 4 + 1] + ncorr, cm.y, cf.y, rq),
                                                requant_u8_channel(acc[gq * 4 + 2] + ncorr, cm.z, cf.z, rq), requant_u8_channel(acc[gq * 4 + 3] + ncorr, cm.w, cf.w, rq));
                    }
                } else if constexpr (QM != 0) {
                    packed[gq] = requant4_fast<QM>(acc[gq * 4 + 0], acc[gq * 4 + 1], acc[gq * 4 + 2], acc[gq * 4 + 3], ncorr, rq);
                } else {
                    packed[gq] = pack_bytes(requant_u8(acc[gq * 4 + 0] + ncorr, rq), requant_u8(acc[gq * 4 + 1] + ncorr, rq),
                                            requant_u8(acc[gq * 4 + 2] + ncorr, rq), requant_u8(acc[gq * 4 + 3] + ncorr, rq));
                }
            }
            if (q < g.pixels && nb * 32 + half * 16 < c_here) {  // (channel counts are multiples of 16: a lane's sixteen channels exist or do not)
                const uint4 v = ok ? make_uint4(packed[0] ^ flip_store, packed[1] ^ flip_store, packed[2] ^ flip_store, packed[3] ^ flip_store)
                                   : make_uint4(pad_word, pad_word, pad_word, pad_word);
                *reinterpret_cast<uint4 *>(img_s + (uint32_t)q * (uint32_t)cpitch + (uint32_t)(nb * 32 + half * 16)) = v;
            }
            if (++nb == nb_here) {
                nb = 0;
                ++blk;
            }
        }
    }
    __syncthreads();

    // ---- stage 2: the depthwise outputs from the LDS image
    // As in eh_dwconv_mfma.hip: lane (i, q) fetches the sixteen channels of output pixel i's window at kernel column q, one
    // 16-byte piece per kernel row, and three products against diagonal weights leave every lane with four neighbouring
    // channels of one pixel.
    const int column = quarter < 3 ? quarter : 2;  // (the fourth column's weights are zero: any pixel will do)
    auto diagonal = [&](uint32_t byte) {
        const int v = (int)(byte << (8 * (lane16 & 3))), d = lane16 >> 2;
        return v4i{d == 0 ? v : 0, d == 1 ? v : 0, d == 2 ? v : 0, d == 3 ? v : 0};
    };
    auto product = [](const v4i &w, const v4i &x, const v4i &acc) { return __builtin_amdgcn_mfma_i32_16x16x64_i8(w, x, acc, 0, 0, 0); };
    const auto out = __builtin_amdgcn_make_buffer_rsrc(dw.out, 0, (int)((uint32_t)dw.n * (uint32_t)dw.ho * (uint32_t)dw.wo * (uint32_t)dw.cout), 0x00020000);
    const uint32_t out_pitch = (uint32_t)dw.wo * (uint32_t)dw.cout;
    for (int left = unit_last - unit_first; left > 0; group = 0, ++chunk) {
        v4i wf[3];
#pragma unroll
        for (int ky = 0; ky < 3; ++ky) wf[ky] = diagonal(part.w[ky]);
        const v4i df = diagonal(quarter < 3 ? part.neg : 0u);
        const bool lacks = __builtin_amdgcn_ballot_w64(part.neg != 0) != 0;
        const DwPart now = part;
        const uint32_t shift_bytes = PC && !DW_TWO_STEP ? channel_shift_bytes(now.shift) : 0u;
        // four channels' accumulators to four bytes
        const RequantDev &drq = dw.rq;
        auto finish = [&](auto mode_c, const v4i &a) {
            constexpr int MODE = decltype(mode_c)::value;  // single-shift form 1 or 2, or the two steps
            if constexpr (PC && MODE != 0)
                return requant4_channel<MODE>(a.x, a.y, a.z, a.w, now.mult, shift_bytes, drq);
            else if constexpr (PC)
                return pack_bytes(requant_u8_channel(a.x, now.mult.x, now.shift.x, drq), requant_u8_channel(a.y, now.mult.y, now.shift.y, drq),
                                  requant_u8_channel(a.z, now.mult.z, now.shift.z, drq), requant_u8_channel(a.w, now.mult.w, now.shift.w, drq));
            else if constexpr (MODE != 0)
                return requant4_fast<MODE>(a.x, a.y, a.z, a.w, 0, drq);
            else
                return pack_bytes(requant_u8(a.x, drq), requant_u8(a.y, drq), requant_u8(a.z, drq), requant_u8(a.w, drq));
        };
        auto with_mode = [&](auto body) {
            if constexpr (DW_TWO_STEP)
                body(std::integral_constant<int, 0>{});
            else if (drq.fast == 2)
                body(std::integral_constant<int, 2>{});
            else if (PC || drq.fast != 0)  // (the caller clears `fast` unless every channel's pair fits the four-channel form)
                body(std::integral_constant<int, 1>{});
            else
                body(std::integral_constant<int, 0>{});
        };
        const v4i bias = v4i{now.bias.x, now.bias.y, now.bias.z, now.bias.w}, none = v4i{0, 0, 0, 0};
        const int last_group = left < groups - group ? group + left : groups;
        left -= last_group - group;
        if (left > 0) part = request_dw(chunk + 1);  // (on its way under this chunk's products)
        const int c0 = c_first + chunk * 16;
        if constexpr (WALK) {
            // lanes 0-15 are 16 columns, or 8 in two strips of rows, or 4 in four
            const int strip = lane16 >> g.walk_log, rows = g.th >> (4 - g.walk_log);
            auto walk = [&](auto mode_c, auto lacks_c) {
                constexpr bool LACKS = decltype(lacks_c)::value;
                for (int grp = group; grp < last_group; ++grp) {
                    const int px = (grp << g.walk_log) + lane16 - (strip << g.walk_log), oy = oy0 + strip * rows, ox = ox_first + px;
                    const int at = px * S + column < g.iwp ? px * S + column : g.iwp - 1;  // (columns past the tile: not stored)
                    const uint8_t *src = img_s + (strip * rows * S * g.iwp + at) * cpitch + chunk * 16;
                    const int src_pitch = g.iwp * cpitch;
                    const int rows_here = px < g.tw && ox < dw.wo ? dw.ho - oy : 0;
                    uint32_t dst = ((img * (uint32_t)dw.ho + (uint32_t)oy) * (uint32_t)dw.wo + (uint32_t)ox) * (uint32_t)dw.cout + (uint32_t)(c0 + quarter * 4);
                    auto next = [&] {
                        const v4i x = *reinterpret_cast<const v4i *>(src);
                        src += src_pitch;
                        return x;
                    };
                    auto store = [&](const v4i &acc, int o) {
                        const uint32_t v = finish(mode_c, acc);
                        // (what is not the tile's is sent past the tensor's end, where the hardware drops it: no branch per row)
                        __builtin_amdgcn_raw_buffer_store_b32(v, out, (int)(o < rows_here ? dst : 0xFFFFFFF0u), 0, 0);
                        dst += out_pitch;
                    };
                    // an input row is multiplied by every kernel row it meets: two, or one, output rows are on their way beside the one it ends
                    if constexpr (S == 1) {
                        v4i x = next(), a0 = product(wf[0], x, bias), l0 = LACKS ? product(df, x, none) : none;
                        x = next();
                        v4i a1 = product(wf[1], x, a0), l1 = LACKS ? product(df, x, l0) : none;
                        a0 = product(wf[0], x, bias);
                        if constexpr (LACKS) l0 = product(df, x, none);
                        for (int o = 0; o < rows; ++o) {
                            x = next();
                            v4i done = product(wf[2], x, a1);
                            a1 = product(wf[1], x, a0);
                            a0 = product(wf[0], x, bias);
                            if constexpr (LACKS) {
                                done -= product(df, x, l1);
                                l1 = product(df, x, l0);
                                l0 = product(df, x, none);
                            }
                            store(done, o);
                        }
                    } else {
                        v4i x = next(), a = product(wf[0], x, bias), l = LACKS ? product(df, x, none) : none;
                        for (int o = 0; o < rows; ++o) {
                            const v4i x1 = next(), x2 = next();
                            v4i done = product(wf[2], x2, product(wf[1], x1, a));
                            a = product(wf[0], x2, bias);
                            if constexpr (LACKS) {
                                done -= product(df, x2, product(df, x1, l));
                                l = product(df, x2, none);
                            }
                            store(done, o);
                        }
                    }
                }
            };
            with_mode([&](auto mode_c) { lacks ? walk(mode_c, std::true_type{}) : walk(mode_c, std::false_type{}); });
        } else {
            for (int grp = group; grp < last_group; ++grp) {
                const int p = grp * 16 + lane16, pc = p < out_pixels ? p : out_pixels - 1;
                const int row = (int)fastdiv((uint32_t)pc, g.div_tw), col = pc - row * g.tw, oy = oy0 + row, ox = ox_first + col;
                const uint8_t *const src = img_s + (row * S * g.iwp + col * S + column) * cpitch + chunk * 16;
                v4i x[3];
#pragma unroll
                for (int ky = 0; ky < 3; ++ky) x[ky] = *reinterpret_cast<const v4i *>(src + ky * g.iwp * cpitch);
                v4i acc = bias;
#pragma unroll
                for (int ky = 0; ky < 3; ++ky) acc = product(wf[ky], x[ky], acc);
                if (lacks) {
                    v4i lack = none;
#pragma unroll
                    for (int ky = 0; ky < 3; ++ky) lack = product(df, x[ky], lack);
                    acc -= lack;
                }
                uint32_t o = 0;
                with_mode([&](auto mode_c) { o = finish(mode_c, acc); });
                if (p < out_pixels && oy < dw.ho && ox < dw.wo)
                    *reinterpret_cast<uint32_t *>(dw.out + (((img * (uint32_t)dw.ho + (uint32_t)oy) * (uint32_t)dw.wo + (uint32_t)ox) * (uint32_t)dw.cout +
                                                            (uint32_t)(c0 + quarter * 4))) = o;
            }
        }
    }
}

constexpr size_t kBlockLdsMax = 150 * 1024;

// Bytes per pixel of the LDS image for `nb` channel blocks of a layer of c channels: the channels of the widest range,
// stretched where needed so that the pitch in words is an odd multiple of four (stage 1 writes sixteen bytes per lane
// for 32 consecutive pixels; at an even multiple of four words those writes meet in a quarter of the banks).
int block_image_pitch(int nb, int c) {
    int words = (nb * 32 < c ? nb * 32 : c) / 4;
    if ((words & 7) == 0) words += 4;
    return words * 4;
}

size_t block_lds_bytes(int nb, int ks, int ih, int iwp, int c, uint32_t *a_off, uint32_t *image_off) {
    const size_t head = ((size_t)nb * ks * 1024 + (size_t)nb * 512 + 15) & ~(size_t)15;  // weights, bias, per-channel pairs
    const size_t a_bytes = ((size_t)ih * iwp * (ks * 32 + 16) + 15) & ~(size_t)15;
    if (a_off) *a_off = (uint32_t)head;
    if (image_off) *image_off = (uint32_t)(head + a_bytes);
    return head + a_bytes + (size_t)ih * iwp * block_image_pitch(nb, c);
}

}  // namespace

// What a depthwise layer has to be to end a fused launch, of what is fixed when its plan is made: those plans keep the matrix form of
// their weights.
bool pwdw_block_takes(const DwProblem &dw) {
    return dw.kh == 3 && dw.kw == 3 && dw.dil_h == 1 && dw.dil_w == 1 && dw.stride_h == dw.stride_w && (dw.stride_h == 1 || dw.stride_h == 2) && dw.dm == 1 &&
           dw.c == dw.cout && (dw.c & 15) == 0 && !dw.io_flip && dw.pad_t >= 0 && dw.pad_l >= 0 && dw.pad_t <= 2 && dw.pad_l <= 2;
}

// The pointwise problem is a one-tap problem of at most eight 32-byte reduction steps on whole dense images whose
// weights are packed in fragment order, the depthwise one a 3x3 channels-last layer of stride 1 or 2 on the pointwise
// output with the matrix form of its weights at hand; uint8 tensors; one requantization pair per operator, or one pair per
// channel in both.
bool pwdw_block_applies(const GemmProblem &pw, const DwProblem &dw) {
    if (pw.cfg.id != GEMM_THIN || pw.k_pad > 256 || pw.k > pw.k_pad || (pw.k & 7) != 0 || (pw.cin & 7) != 0 || pw.k != pw.cin) return false;
    if (pw.stride_h != 1 || pw.stride_w != 1 || pw.y_base != 0 || pw.x_base != 0 || pw.ho != pw.h || pw.wo != pw.w) return false;
    if (pw.a_xor != 0x80808080u || pw.out_xor != 0u || pw.residual) return false;
    if ((pw.rq.pc_multiplier != nullptr) != (dw.rq.pc_multiplier != nullptr)) return false;
    if (!pwdw_block_takes(dw) || dw.c != pw.n || dw.h != pw.h || dw.w_ != pw.w || dw.w_mm == nullptr) return false;
    if ((size_t)dw.n * dw.h * dw.w_ * pw.cin >= (1ull << 31) || (size_t)dw.n * dw.ho * dw.wo * dw.cout >= (1ull << 31)) return false;
    return block_lds_bytes(1, pw.k_pad / 32, 3, 3 * dw.stride_w + 3, dw.c, nullptr, nullptr) <= kBlockLdsMax;  // one row of four outputs, one channel block
}

// Whether the one launch beats the two.  The fused kernel computes the expanded pixels of a tile's halo twice and
// requantizes every expanded value on the vector ALU just as the stand-alone kernels do, so what it saves is the
// expanded tensor's trip through memory and one launch; whether that pays depends on the shape, and the answer here
// is a table of the shapes that were timed inside a network (MobileNetV2 at 224 x 224, 32 images per launch, each
// pair switched to the fused kernel on its own; microseconds per network pass against 345 with none fused):
//   image  in -> expanded  stride   change        image  in -> expanded  stride   change
//   112     16 ->  96        2      +6.4           14    64 -> 384         1      -0.8 / -0.4 / -0.8 / -0.5
//    56     24 -> 144        1      -3.1           14    96 -> 576         1      -0.3 / +1.5
//    56     24 -> 144        2      -4.6           14    96 -> 576         2      -0.6
//    28     32 -> 192        1      -3.3 / +1.3     7   160 -> 960         1      +0.1 / +1.2 / +0.8
//    28     32 -> 192        2      -1.1
// (changes within +-1.5 are noise.  With the listed pairs fused the pass takes 324.6; 14 x 14 64 -> 384 alone runs in 6.6 us against 8.0
// for the two launches, 28 x 28 32 -> 192 in 9.2 against 9.2 and at stride 2 in 6.8 against 7.8, 56 x 56 24 -> 144 in 20.9 against 21.1.)
// A shape that is not in the table runs as two launches.  (The figures are from before the depthwise stage's walk.  Since then, alone in a
// replayed graph, two launches against one, us: 32 images, 96 -> 576 at 14x14 8.5 and 8.4, at stride 2 7.0 and 7.3, 160 -> 960 at 7x7 7.1 and 6.8,
// 24 -> 144 at 56x56 18.6 and 17.0, 16 -> 96 at 112x112 35.8 and 33.6, at stride 2 23.7 and 23.0; 64 images, 24 -> 144 at 56x56 29.9 and 27.1, 96 -> 576 12.4
// and 11.6, 160 -> 960 8.7 and 8.9; 44 images, 16 -> 96 at 88x88 32.2 and 33.4.  Inside the network these pairs have not been timed again.)
bool pwdw_block_listed(int32_t images, int32_t image_h, int32_t image_w, int32_t in_channels, int32_t expanded_channels, int32_t stride) {
    // Below 32 images a launch is mostly latency, and one launch instead of two wins for the whole network:
    // MobileNetV2 with all 16 fitting pairs fused against the listed ones, 144 against 162 us at batch 1, 168 against 176
    // at 4, 206 against 222 at 8, 246 against 260 at 16, 288 against 294 at 24; at 32 it is a draw, 324.2 against 324.6.
    // (With the walk also alone and on large tensors: 31 images, 16 -> 96 at 112x112 34.8 and 34.3, 32 -> 192 at 56x56 21.5 and 19.8; 16 images, 24 -> 144
    // at 112x112 29.9 and 27.0, 16 -> 96 at 112x112 22.4 and 21.3; one image, 24 -> 144 at 224x224 11.3 and 9.7.)
    if (images < 32) return true;
    if (image_h != image_w) return false;
    struct Shape {
        int32_t image, in, expanded, stride;
    };
    static const Shape faster[] = {{56, 24, 144, 2}, {28, 32, 192, 1}, {28, 32, 192, 2}, {14, 64, 384, 1}};
    for (const Shape &s : faster)
        if (image_h == s.image && in_channels == s.in && expanded_channels == s.expanded && stride == s.stride) return true;
    return false;
}

bool pwdw_block_preferred(const GemmProblem &pw, const DwProblem &dw) {
    return pwdw_block_applies(pw, dw) && pwdw_block_listed(dw.n, dw.h, dw.w_, pw.k, dw.c, dw.stride_h);
}

namespace {

// The tile of a launch whose depthwise stage walks: the one that takes the least time by a count of its waves' instructions, each of
// which takes a SIMD some 2.3 + 1.1 w ns for the w waves it holds; a set of workgroups that a CU holds at a time (registers leave
// room for five, with a pair per channel four) takes a microsecond beside that.  The coefficients are fitted to 3900 tiles of eighteen
// layers; for those layers the tile chosen is 3 % slower than the fastest on average and 8 % at most.  How many workgroups a CU gets is
// counted as the hardware deals them out: an eighth of the tiles, rounded up, to an XCD of 32 CUs, and LDS in pieces of 1280 bytes.  Without
// the one, 152 -> 912 at 17x17, 11 images, a pair per channel, had 65 workgroups to an XCD where 64 fit, 15.3 us (9.55 now); without the other 24 ->
// 144 at 77x77 stride 2, 22 images, had two of 54336 bytes to a CU where three were counted on, 17.8 us (13.8).  364 drawn pairs: 1.8 % faster.
bool walk_tile(const GemmProblem &pw, const DwProblem &dw, int rows_per_tile, int cols_per_tile, int *th, int *tw, int *nb, int *walk_log, double *time_taken) {
    const int S = dw.stride_h, ks = pw.k_pad / 32, nb_all = (dw.c + 31) / 32, chunks_all = dw.c / 16;
    const double epilogue = pw.rq.pc_multiplier ? 1.42 : 1.0;
    const int held = pw.rq.pc_multiplier ? 4 : 5;
    auto shares = [](int a, int b) { return (a + b - 1) / b; };
    // tiles across the image and down it, as equal as columns and whole strips allow, the largest first.  (A launch finds its tile the
    // first time it runs: what a candidate needs is worked out ahead of the loops, and shapes that cannot win are not looked at.)
    constexpr int MOST = 32;  // rows and columns
    struct Cut {
        int size, pieces;
    } across[MOST], down[3][MOST];
    int n_across = 0, n_down[3] = {0, 0, 0};
    auto cut = [&](int extent, int fixed, int unit, int narrowest, Cut *to, int *count) {
        if (fixed > 0) {
            if (fixed % unit == 0) to[(*count)++] = Cut{fixed, shares(extent, fixed)};
            return;
        }
        const int whole = shares(extent, unit) * unit;
        for (int size = whole < MOST ? whole : MOST; size >= unit; size -= unit) {
            const int even = shares(extent, shares(extent, size) * unit) * unit;
            if (*count > 0 && (even == to[*count - 1].size || even < narrowest)) continue;
            to[(*count)++] = Cut{even, shares(extent, even)};
        }
    };
    cut(dw.wo, cols_per_tile, 1, 4, across, &n_across);  // (of four columns or more: a walk takes no fewer at a time)
    for (int lg = 4; lg >= 2; --lg) cut(dw.ho, rows_per_tile, 16 >> lg, 1, down[4 - lg], &n_down[4 - lg]);
    double best = -1;
    for (const size_t lds_max : {(size_t)64 * 1024, kBlockLdsMax}) {  // (above 64 KiB a launch sets an attribute of the kernel first)
        for (int cn = 1; cn <= nb_all; ++cn) {
            const int ranges = shares(nb_all, cn);
            if ((ranges - 1) * cn >= nb_all) continue;  // the same ranges with fewer blocks each
            const int chunks = cn * 2 < chunks_all ? cn * 2 : chunks_all;
            const size_t lds_fixed = block_lds_bytes(cn, ks, 0, 0, dw.c, nullptr, nullptr), lds_pixel = (size_t)(ks * 32 + 16 + block_image_pitch(cn, dw.c));
            for (int lg = 4; lg >= 2; --lg) {
                for (int i = 0; i < n_down[4 - lg]; ++i) {
                    const Cut d = down[4 - lg][i];
                    const int ih = (d.size - 1) * S + 3;
                    const double walk = 52.0 + 26.0 * epilogue * (d.size >> (4 - lg));
                    for (int j = 0; j < n_across; ++j) {
                        const Cut a = across[j];
                        const int pixels = ih * ((a.size - 1) * S + 3);
                        const size_t lds = lds_fixed + (size_t)pixels * lds_pixel + 15;
                        if (lds > lds_max) continue;
                        const double per_cu = (double)(((long)dw.n * d.pieces * a.pieces + 7) / 8 * ranges) / 32.0;  // (of an XCD with all its tiles)
                        if (best >= 0 && pixels < 80 && per_cu > held) break;  // (small tiles only where larger ones would leave CUs idle)
                        const double wave = 10 + 40.0 * cn + 40.0 * ((pixels * ks * 4 + 255) >> 8) + ((((pixels + 31) >> 5) * cn + 3) >> 2) * (67.0 * epilogue + 5.5 * ks) +
                                            ((chunks * ((a.size + (1 << lg) - 1) >> lg) + 3) >> 2) * walk;
                        const int fit = (int)((160 * 1024) / ((lds + 1279) / 1280 * 1280)), most = fit < held ? fit : held, full = (int)(per_cu / most);
                        auto time = [&](int waves) { return wave * (2.3 + 1.07 * waves) + 800; };
                        const int rest = (int)(per_cu - full * most + 0.999);
                        const double cost = full * time(most) + (rest > 0 ? time(rest) : 0);
                        if (best < 0 || cost < best) {
                            best = cost;
                            *th = d.size;
                            *tw = a.size;
                            *nb = cn;
                            *walk_log = lg;
                        }
                    }
                }
            }
        }
        *time_taken = best;
        if (best >= 0) return true;
    }
    return false;
}

// The tile of a stride-2 launch whose depthwise stage takes sixteen outputs at a time, where that is the faster one than the tile that walks, of
// which `walk` is the time: at stride 2 a walk meets a wave's columns in rows twice as long and keeps few of its lanes busy on a small tile.  One
// group of outputs to a tile, up to eight chunks of sixteen channels, a workgroup or more to every CU and no second round of them (smaller launches
// are latency either way).  Priced as walk_tile prices, but by the mean of the channel ranges, of which the last may be short; the coefficients
// are fitted to 700 drawn stride-2 layers with every such tile timed, and so are the prices up to which units are taken: with one reduction step 1.06
// of the walk's, with more 0.94, where units' time is 0.98 of the walk's from there to 1.00 and 1.07 at most; launches of more than 1.28 million outputs
// took 1.02 .. 1.11.  836 other drawn stride-2 layers: 308 take units, 0.96 of the walk's time on average, 0.87 .. 1.07, four of them above 1.04.
// us, walk and units:
// 24 -> 144 at 56x56, seven images 5.47 and 4.89, a pair per channel at 48x48, nine images 6.08 and 5.37; 16 -> 96 at 64x64, six images
// 5.07 and 4.53.  At stride 1 the walk takes 0.88 of the units' time, 0.95 with a pair per channel.
bool units_tile(const GemmProblem &pw, const DwProblem &dw, double walk, int *th, int *tw, int *nb) {
    const int ks = pw.k_pad / 32, nb_all = (dw.c + 31) / 32, chunks_all = dw.c / 16;
    const double epilogue = pw.rq.pc_multiplier ? 1.42 : 1.0;
    if ((int64_t)dw.n * dw.ho * dw.wo * dw.c > 5000 * 256) return false;
    bool found = false;
    walk *= ks == 1 ? 1.06 : 0.94;  // (the prices of the two forms meet there: timed, see above)
    for (int cn = 1; cn <= 4 && cn <= nb_all; ++cn) {
        const int ranges = (nb_all + cn - 1) / cn;
        if ((ranges - 1) * cn >= nb_all) continue;  // the same ranges with fewer blocks each
        const int last_blocks = nb_all - (ranges - 1) * cn, last_chunks = chunks_all - (ranges - 1) * cn * 2;
        for (int rows = 1; rows <= 8 && rows <= dw.ho; ++rows)
            for (int cols = (8 + rows - 1) / rows < 3 ? 3 : (8 + rows - 1) / rows; cols * rows <= 16 && cols <= dw.wo; ++cols) {
                const int ih = (rows - 1) * 2 + 3, iw = (cols - 1) * 2 + 3, pixels = ih * iw;
                const size_t lds = block_lds_bytes(cn, ks, ih, iw, dw.c, nullptr, nullptr);
                if (lds > (size_t)64 * 1024) continue;
                const long tiles = (long)dw.n * ((dw.ho + rows - 1) / rows) * ((dw.wo + cols - 1) / cols);
                const double per_cu = (double)((tiles + 7) / 8 * ranges) / 32.0;
                const int fit = (int)((160 * 1024) / ((lds + 1279) / 1280 * 1280)), most = fit < 5 ? fit : 5;
                if (per_cu < 1 || per_cu > 5) continue;
                auto range = [&](int blocks, int chunks) {
                    return 10 + 40.0 * blocks + 40.0 * ((pixels * ks * 4 + 255) >> 8) + ((((pixels + 31) >> 5) * blocks + 3) >> 2) * (67.0 * epilogue + 5.5 * ks) +
                           ((chunks + 3) >> 2) * (40.0 + 12.0 * epilogue);
                };
                const double wave = ((ranges - 1) * range(cn, cn * 2) + range(last_blocks, last_chunks)) / ranges;
                auto time = [&](int waves) { return wave * (2.3 + 1.07 * waves) + 800; };
                const int full = (int)(per_cu / most), rest = (int)(per_cu - full * most + 0.999);
                const double cost = full * time(most) + (rest > 0 ? time(rest) : 0);
                if (cost >= walk) continue;
                walk = cost;
                *th = rows;
                *tw = cols;
                *nb = cn;
                found = true;
            }
    }
    return found;
}

}  // namespace

bool pwdw_block_geometry(const GemmProblem &pw, const DwProblem &dw, int rows_per_tile, int cols_per_tile, BlockGeom *geom) {
    const int S = dw.stride_h;
    BlockGeom g;
    g.c = dw.c;
    g.ks = pw.k_pad / 32;
    g.a_pitch = g.ks * 32 + 16;
    const int nb_all = (dw.c + 31) / 32;
    if (rows_per_tile > (dw.ho < 16 ? dw.ho : 16) || cols_per_tile > (dw.wo < 64 ? dw.wo : 64)) return false;
    int th = rows_per_tile, tw = cols_per_tile, nb = 0;
    g.matrix = g.walk_log = g.walk_groups = 0;
    if (rows_per_tile > 0 && cols_per_tile > 0) {
        // A tile of the caller's may suit the units of sixteen outputs: a walk takes 16 columns at a time, or 8, or 4, and leaves the lanes of the
        // others idle.  Channel blocks of a unit's workgroup: as many as leave room for four workgroups in a CU's LDS, or as fit.
        for (const size_t lds_max : {(size_t)36 * 1024, kBlockLdsMax})
            for (int cn = nb_all; cn >= 1 && nb == 0; --cn)
                if (((nb_all + cn - 1) / cn - 1) * cn < nb_all && block_lds_bytes(cn, g.ks, (th - 1) * S + 3, (tw - 1) * S + 3, dw.c, nullptr, nullptr) <= lds_max) nb = cn;
        if (nb == 0) return false;
        // The line, on 900 requested tiles of drawn layers of up to 1.5 GFLOP, walk over units by the units of a workgroup (with a pair per channel): 2
        // 0.98 (1.02), 4 1.03 (1.03), 6 1.17 and half full ones 1.21 (0.97 and 1.07), 8 full 0.96 (0.96), 12 full 0.92 (0.99), beyond 0.77 (0.73).
        const int groups = (th * tw + 15) / 16, chunks = nb * 2 < dw.c / 16 ? nb * 2 : dw.c / 16, units = groups * chunks;
        g.matrix = units <= (pw.rq.pc_multiplier == nullptr ? 8 : S == 2 ? 6 : 3) && (units <= 4 || th * tw > groups * 8) ? 1 : 0;
    }
    double time_taken = 0;
    if (!g.matrix && !walk_tile(pw, dw, rows_per_tile, cols_per_tile, &th, &tw, &nb, &g.walk_log, &time_taken)) return false;
    if (rows_per_tile <= 0 && cols_per_tile <= 0 && S == 2 && units_tile(pw, dw, time_taken, &th, &tw, &nb)) g.matrix = 1, g.walk_log = 0;
    g.nb = nb;
    g.th = th;
    g.tw = tw;
    g.ih = (th - 1) * S + 3;
    g.iwp = (tw - 1) * S + 3;
    g.pixels = g.ih * g.iwp;
    g.tiles_y = (dw.ho + th - 1) / th;
    g.tiles_w = (dw.wo + tw - 1) / tw;
    g.total_tiles = dw.n * g.tiles_y * g.tiles_w;
    if (!g.matrix) g.walk_groups = (tw + (1 << g.walk_log) - 1) >> g.walk_log;
    g.div_iwp = make_fastdiv((uint32_t)g.iwp);
    g.div_tw = make_fastdiv((uint32_t)tw);
    g.div_tiles_y = make_fastdiv((uint32_t)g.tiles_y);
    g.div_tiles_w = make_fastdiv((uint32_t)g.tiles_w);
    g.div_ppp = make_fastdiv((uint32_t)(g.ks * 4));
    g.cpitch = block_image_pitch(g.nb, g.c);
    const size_t lds = block_lds_bytes(g.nb, g.ks, g.ih, g.iwp, g.c, &g.a_off, &g.image_off);
    if (lds > kBlockLdsMax) return false;
    *geom = g;
    return true;
}

// `g`: what pwdw_block_geometry gave for the pair (the search over tiles costs the host as much as the launch: callers keep it)
int launch_pwdw_block(const GemmProblem &pw, const DwProblem &dw, const BlockGeom &g, hipStream_t stream) {
    EH_REQUIRE(pwdw_block_applies(pw, dw), "block: the two operators do not fit the fused kernel");
    EH_REQUIRE((reinterpret_cast<uintptr_t>(pw.a) & 7) == 0 && (reinterpret_cast<uintptr_t>(dw.out) & 3) == 0, "block: unaligned tensors");
    EH_REQUIRE(g.c == dw.c && g.ks == pw.k_pad / 32, "block: geometry of another pair");
    const int S = dw.stride_h;
    const size_t lds = (size_t)g.image_off + (size_t)g.ih * g.iwp * g.cpitch;
    if (g.total_tiles <= 0) return EH_OK;
    const dim3 grid((unsigned)((g.total_tiles + 7) / 8 * 8), (unsigned)(((g.c + 31) / 32 + g.nb - 1) / g.nb));
    auto launch_pc = [&](auto s_c, auto form_c, auto rowsum_c, auto qm_c, auto ks_c, auto pc_c) {
        auto kernel = pwdw_block_kernel<decltype(s_c)::value, decltype(form_c)::value, decltype(rowsum_c)::value, decltype(qm_c)::value, decltype(ks_c)::value,
                                        decltype(pc_c)::value>;
        if (lds > 64 * 1024) {
            // (a driver call, made per launch of the tall-tile shapes only; the default tile height stays below 64 KiB)
            hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void *>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, (int)kBlockLdsMax);
            if (e != hipSuccess) return hip_fail(e, "hipFuncSetAttribute(pwdw_block_kernel)");
        }
        hipLaunchKernelGGL(kernel, grid, dim3(256), lds, stream, pw, dw, g);
        return (int)EH_OK;
    };
    auto launch = [&](auto s_c, auto form_c, auto rowsum_c, auto qm_c, auto ks_c) {
        using std::integral_constant;
        if (!pw.rq.pc_multiplier) return launch_pc(s_c, form_c, rowsum_c, qm_c, ks_c, integral_constant<Pairs, Pairs::TENSOR>{});
        return dw.rq.fast ? launch_pc(s_c, form_c, rowsum_c, qm_c, ks_c, integral_constant<Pairs, Pairs::CHANNEL>{})
                          : launch_pc(s_c, form_c, rowsum_c, qm_c, ks_c, integral_constant<Pairs, Pairs::CHANNEL_TWO_STEP>{});
    };
    auto with_ks = [&](auto s_c, auto form_c, auto rowsum_c, auto qm_c) {
        if (g.ks == 1) return launch(s_c, form_c, rowsum_c, qm_c, std::integral_constant<int, 1>{});
        if (g.ks == 2) return launch(s_c, form_c, rowsum_c, qm_c, std::integral_constant<int, 2>{});
        if (g.ks == 3) return launch(s_c, form_c, rowsum_c, qm_c, std::integral_constant<int, 3>{});
        return launch(s_c, form_c, rowsum_c, qm_c, std::integral_constant<int, 0>{});
    };
    auto with_qm = [&](auto s_c, auto form_c, auto rowsum_c) {
        if (pw.rq.fast == 2) return with_ks(s_c, form_c, rowsum_c, std::integral_constant<int, 2>{});
        if (pw.rq.fast == 1) return with_ks(s_c, form_c, rowsum_c, std::integral_constant<int, 1>{});
        return with_ks(s_c, form_c, rowsum_c, std::integral_constant<int, 0>{});
    };
    auto with_rowsum = [&](auto s_c, auto form_c) {
        return pw.zw != 0 ? with_qm(s_c, form_c, std::true_type{}) : with_qm(s_c, form_c, std::false_type{});
    };
    auto with_form = [&](auto s_c) {
        return g.matrix ? with_rowsum(s_c, std::integral_constant<DwForm, DwForm::UNITS>{}) : with_rowsum(s_c, std::integral_constant<DwForm, DwForm::WALK>{});
    };
    const int rc = S == 1 ? with_form(std::integral_constant<int, 1>{}) : with_form(std::integral_constant<int, 2>{});
    if (rc) return rc;
    EH_HIP(hipGetLastError());
    return EH_OK;
}

}  // namespace eh
