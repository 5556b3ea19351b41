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
//   2. after one barrier the threads compute the depthwise outputs from that image, four horizontally adjacent output
//      pixels of four channels per thread, with the arithmetic of the stand-alone depthwise kernel (8-bit dot products,
//      signed or unsigned form), and store them.
//      Small tiles (a network on few images) do this stage on the matrix cores: a thread's sixteen outputs are a chain of some 300
//      vector instructions that a workgroup of few such threads waits for.  28x28 32 -> 192 at stride 2, two images, 5.4 -> 4.2 us
//      (pwdw_block_geometry has the rule and both sides of it).
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

__device__ __forceinline__ int udot4(uint32_t a, uint32_t b, int acc) { return (int)__builtin_amdgcn_udot4(a, b, (uint32_t)acc, false); }

// the four channels of a column's three rows as four words of three bytes each (byte 3 zero)
__device__ __forceinline__ void column_words(uint32_t r0, uint32_t r1, uint32_t r2, uint32_t (&out)[4]) {
    const uint32_t t01 = __builtin_amdgcn_perm(r1, r0, 0x05010400u);
    const uint32_t t23 = __builtin_amdgcn_perm(r1, r0, 0x07030602u);
    out[0] = __builtin_amdgcn_perm(r2, t01, 0x0c040100u);
    out[1] = __builtin_amdgcn_perm(r2, t01, 0x0c050302u);
    out[2] = __builtin_amdgcn_perm(r2, t23, 0x0c060100u);
    out[3] = __builtin_amdgcn_perm(r2, t23, 0x0c070302u);
}

// S: depthwise stride.  FORM: how the depthwise stage multiplies (DwForm).  ROWSUM: the pointwise weights' zero point is not 128, so a pixel's byte sum enters.
// QM: pointwise requantization, 0 two-step order, 1 / 2 the single-shift forms.  KS: reduction steps of the pointwise
// stage when they are 1, 2 or 3 (a lane then keeps its pixel's operand bytes in registers across the channel blocks),
// 0 for any number (read from LDS for every product).
enum class DwForm {
    DOT,   // 8-bit dot products of a - 128 and w - zp_w
    FOLD,  // ... of the raw bytes: the unsigned form, for weights of any range
    MATRIX // on the matrix cores, weights of any range
};
template <int S, DwForm FORM, bool ROWSUM, int QM, int KS, bool PC>
__global__ __launch_bounds__(256) void pwdw_block_kernel(const GemmProblem pw, const DwProblem dw, const BlockGeom g) {
    constexpr bool FOLD = FORM == DwForm::FOLD, MATRIX = FORM == DwForm::MATRIX;
    const int ksteps = KS ? KS : g.ks;
    extern __shared__ __align__(16) uint8_t lds_raw[];
    v4i *b_s = reinterpret_cast<v4i *>(lds_raw);                              // [nb][ks][64 lanes]: pointwise weights, fragment order
    int32_t *bias_s = reinterpret_cast<int32_t *>(lds_raw + (size_t)g.nb * ksteps * 1024);  // [nb * 32]
    // PC (one multiplier and shift per channel in both operators): the pointwise stage's pairs beside the bias; the shifts as the
    // bytes that requant4_channel wants or, two-step, as they are
    int32_t *pcm_s = bias_s + g.nb * 32, *pcf_s = pcm_s + g.nb * 32;
    uint8_t *pce_s = reinterpret_cast<uint8_t *>(pcf_s);
    uint8_t *img_s = lds_raw + g.image_off;                                   // [ih][iwp][cpitch] uint8 (xor 0x80 for the signed form)
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

    // MATRIX: units of (chunk of 16 channels, 16 output pixels), a contiguous share per wave; lane (i, q) holds the weights of
    // channel i of the chunk in kernel column q.  A wave's first chunk is requested ahead of everything else.
    const int lane16 = lane & 15, quarter = lane >> 4, cpad = (g.c + 15) & ~15;
    const int out_pixels = g.th * g.tw, groups = (out_pixels + 15) >> 4, w_uniform = __builtin_amdgcn_readfirstlane(wave);
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
    if constexpr (MATRIX) {
        if (unit_first < unit_last) part = request_dw(chunk);
    }

    // ---- stage 0: weights, bias and the tile's input pixels into LDS (8-byte pieces: pixels start on 8-byte boundaries)
    auto inside_image = [&](int q, int &iy, int &ix) {
        const int ry = (int)fastdiv((uint32_t)q, g.div_iwp), rx = q - ry * g.iwp;
        iy = iy_first + ry;
        ix = ix_first + rx;
        return (unsigned)iy < (unsigned)pw.h && (unsigned)ix < (unsigned)pw.w;
    };
    {
        // The input pixels first, then the weights as direct-to-LDS copies, all on their way at once beside the bias.  (The pieces four
        // at a time behind the weights' copies, from clamped addresses without a branch, cost a small launch more instructions than they
        // save trips: 40 -> 240 at 20x20 stride 2, six images, 5.13 us as here, 5.44 like that; 48 -> 288 at 33x33, four images 5.57
        // and 5.81; 64 -> 384 at 14x14, eight images 5.46 and 5.69.)
        const int ppp = ksteps * 4;  // 8-byte pieces per pixel
        const int pieces = g.pixels * ppp;
        for (int i = tid; i < pieces; i += 256) {
            const int q = KS ? i / (KS * 4) : (int)fastdiv((uint32_t)i, g.div_ppp), piece = i - q * ppp;
            int iy, ix;
            uint2 v = make_uint2(0u, 0u);  // bytes past the reduction length, and whole pixels outside the image: operand 0
            if (inside_image(q, iy, ix) && piece * 8 < pw.k) {
                v = *reinterpret_cast<const uint2 *>(pw.a + (((img * (uint32_t)pw.h + (uint32_t)iy) * (uint32_t)pw.w + (uint32_t)ix) * (uint32_t)pw.cin +
                                                               (uint32_t)pw.a_offset + (uint32_t)piece * 8u));
                v.x ^= pw.a_xor;
                v.y ^= pw.a_xor;
            }
            *reinterpret_cast<uint2 *>(a_s + q * g.a_pitch + piece * 8) = v;
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
    const uint32_t flip_store = FOLD ? 0u : 0x80808080u;  // the signed depthwise forms read a - 128
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
    // four channels' accumulators to four bytes
    auto finish = [&](int a0, int a1, int a2, int a3, const int4 &m, const int4 &sh) {
        const RequantDev &drq = dw.rq;
        if constexpr (PC) {
            // (the caller clears `fast` unless every pair fits the four-channel form)
            if (drq.fast == 2) return requant4_channel<2>(a0, a1, a2, a3, m, channel_shift_bytes(sh), drq);
            if (drq.fast) return requant4_channel<1>(a0, a1, a2, a3, m, channel_shift_bytes(sh), drq);
            return pack_bytes(requant_u8_channel(a0, m.x, sh.x, drq), requant_u8_channel(a1, m.y, sh.y, drq), requant_u8_channel(a2, m.z, sh.z, drq),
                              requant_u8_channel(a3, m.w, sh.w, drq));
        }
        if (drq.fast == 2) return requant4_fast<2>(a0, a1, a2, a3, 0, drq);
        if (drq.fast) return requant4_fast<1>(a0, a1, a2, a3, 0, drq);
        return pack_bytes(requant_u8(a0, drq), requant_u8(a1, drq), requant_u8(a2, drq), requant_u8(a3, drq));
    };
    if constexpr (MATRIX) {
        // As in eh_dwconv_mfma.hip: lane (i, q) fetches the sixteen channels of output pixel i's window at kernel column q, one
        // 16-byte piece per kernel row, and three products against diagonal weights leave every lane with four neighbouring
        // channels of one pixel.
        const int column = quarter < 3 ? quarter : 2;  // (the fourth column's weights are zero: any pixel will do)
        auto diagonal = [&](uint32_t byte) {
            const int v = (int)(byte << (8 * (lane16 & 3))), d = lane16 >> 2;
            return v4i{d == 0 ? v : 0, d == 1 ? v : 0, d == 2 ? v : 0, d == 3 ? v : 0};
        };
        for (int left = unit_last - unit_first; left > 0; group = 0, ++chunk) {
            v4i wf[3];
#pragma unroll
            for (int ky = 0; ky < 3; ++ky) wf[ky] = diagonal(part.w[ky]);
            const v4i df = diagonal(quarter < 3 ? part.neg : 0u);
            const bool lacks = __builtin_amdgcn_ballot_w64(part.neg != 0) != 0;
            const DwPart now = part;
            const int last_group = left < groups - group ? group + left : groups;
            left -= last_group - group;
            if (left > 0) part = request_dw(chunk + 1);  // (on its way under this chunk's products)
            const int c0 = c_first + chunk * 16;
            for (int grp = group; grp < last_group; ++grp) {
                const int p = grp * 16 + lane16, pc = p < out_pixels ? p : out_pixels - 1;
                const int row = (int)fastdiv((uint32_t)pc, g.div_tw), col = pc - row * g.tw, oy = oy0 + row, ox = ox_first + col;
                const uint8_t *const src = img_s + (row * S * g.iwp + col * S + column) * cpitch + chunk * 16;
                v4i x[3];
#pragma unroll
                for (int ky = 0; ky < 3; ++ky) x[ky] = *reinterpret_cast<const v4i *>(src + ky * g.iwp * cpitch);
                v4i acc = v4i{now.bias.x, now.bias.y, now.bias.z, now.bias.w};
#pragma unroll
                for (int ky = 0; ky < 3; ++ky) acc = __builtin_amdgcn_mfma_i32_16x16x64_i8(wf[ky], x[ky], acc, 0, 0, 0);
                if (lacks) {
                    v4i lack = v4i{0, 0, 0, 0};
#pragma unroll
                    for (int ky = 0; ky < 3; ++ky) lack = __builtin_amdgcn_mfma_i32_16x16x64_i8(df, x[ky], lack, 0, 0, 0);
                    acc -= lack;
                }
                const uint32_t o = finish(acc.x, acc.y, acc.z, acc.w, now.mult, now.shift);
                if (p < out_pixels && oy < dw.ho && ox < dw.wo)
                    *reinterpret_cast<uint32_t *>(dw.out + (((img * (uint32_t)dw.ho + (uint32_t)oy) * (uint32_t)dw.wo + (uint32_t)ox) * (uint32_t)dw.cout +
                                                            (uint32_t)(c0 + quarter * 4))) = o;
            }
        }
        return;
    }
    constexpr int TW = 4, IW = (TW - 1) * S + 3;  // a thread's four adjacent output pixels
    const uint32_t cq_count = (uint32_t)c_here >> 2;
    const uint32_t units = (uint32_t)g.units_per_cq * cq_count;
    const uint32_t cq_first = (uint32_t)c_first >> 2;
    const FastDiv div_cq = blockIdx.y + 1 == gridDim.y ? g.div_cq_last : g.div_cq;
    for (uint32_t u = (uint32_t)tid; u < units; u += 256u) {
        const uint32_t t = fastdiv(u, div_cq);
        const uint32_t cql = u - t * cq_count, cq = cq_first + cql;  // channel quad within the range, and in the layer
        const uint32_t row = fastdiv(t, g.div_tx);
        const int tx = (int)(t - row * (uint32_t)g.tiles_x);
        const int oy = oy0 + (int)row, lx0 = tx * TW, ox0 = ox_first + lx0;  // lx0: first column within the workgroup's tile
        if (oy >= dw.ho) continue;
        uint32_t in[3][IW];
#pragma unroll
        for (int ky = 0; ky < 3; ++ky)
#pragma unroll
            for (int x = 0; x < IW; ++x) {
                int col = lx0 * S + x;
                col = col < g.iwp ? col : g.iwp - 1;  // columns past the last window belong to outputs that are not stored
                in[ky][x] = *reinterpret_cast<const uint32_t *>(img_s + (((int)row * S + ky) * g.iwp + col) * cpitch + (int)cql * 4);
            }
        int4 wk[3];
#pragma unroll
        for (int kx = 0; kx < 3; ++kx) wk[kx] = *reinterpret_cast<const int4 *>((FOLD ? dw.w_fold : dw.w_trip) + ((uint32_t)kx * (uint32_t)dw.cout + cq * 4u));
        const int4 b4 = *reinterpret_cast<const int4 *>((FOLD ? dw.bias_fold : dw.bias_trip) + cq * 4u);
        int4 dm = make_int4(0, 0, 0, 0), ds = dm;  // PC: the depthwise stage's four pairs
        if constexpr (PC) {
            dm = *reinterpret_cast<const int4 *>(dw.rq.pc_multiplier + cq * 4u);
            ds = *reinterpret_cast<const int4 *>(dw.rq.pc_shift + cq * 4u);
        }
        uint32_t colw[IW][4];
        int cs[FOLD ? IW : 1][4];
#pragma unroll
        for (int x = 0; x < IW; ++x) {
            column_words(in[0][x], in[1][x], in[2][x], colw[x]);
            if constexpr (FOLD) {
#pragma unroll
                for (int c = 0; c < 4; ++c) cs[x][c] = udot4(colw[x][c], 0x00010101u, 0);
            }
        }
        uint8_t *dst = dw.out + (((img * (uint32_t)dw.ho + (uint32_t)oy) * (uint32_t)dw.wo + (uint32_t)ox0) * (uint32_t)dw.cout + cq * 4u);
#pragma unroll
        for (int j = 0; j < TW; ++j) {
            int acc0 = b4.x, acc1 = b4.y, acc2 = b4.z, acc3 = b4.w;
#pragma unroll
            for (int kx = 0; kx < 3; ++kx) {
                if constexpr (FOLD) {
                    acc0 = udot4(colw[j * S + kx][0], (uint32_t)wk[kx].x, acc0);
                    acc1 = udot4(colw[j * S + kx][1], (uint32_t)wk[kx].y, acc1);
                    acc2 = udot4(colw[j * S + kx][2], (uint32_t)wk[kx].z, acc2);
                    acc3 = udot4(colw[j * S + kx][3], (uint32_t)wk[kx].w, acc3);
                } else {
                    acc0 = __builtin_amdgcn_sdot4((int)colw[j * S + kx][0], wk[kx].x, acc0, false);
                    acc1 = __builtin_amdgcn_sdot4((int)colw[j * S + kx][1], wk[kx].y, acc1, false);
                    acc2 = __builtin_amdgcn_sdot4((int)colw[j * S + kx][2], wk[kx].z, acc2, false);
                    acc3 = __builtin_amdgcn_sdot4((int)colw[j * S + kx][3], wk[kx].w, acc3, false);
                }
            }
            if constexpr (FOLD) {
                acc0 += __mul24(-dw.zp_w, cs[j * S][0] + cs[j * S + 1][0] + cs[j * S + 2][0]);
                acc1 += __mul24(-dw.zp_w, cs[j * S][1] + cs[j * S + 1][1] + cs[j * S + 2][1]);
                acc2 += __mul24(-dw.zp_w, cs[j * S][2] + cs[j * S + 1][2] + cs[j * S + 2][2]);
                acc3 += __mul24(-dw.zp_w, cs[j * S][3] + cs[j * S + 1][3] + cs[j * S + 2][3]);
            }
            const uint32_t o = finish(acc0, acc1, acc2, acc3, dm, ds);
            if (lx0 + j < g.tw && ox0 + j < dw.wo) *reinterpret_cast<uint32_t *>(dst + (uint32_t)j * (uint32_t)dw.cout) = o;
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
// output with the 8-bit dot product weights at hand; uint8 tensors; one requantization pair per operator, or one pair per
// channel in both.
bool pwdw_block_applies(const GemmProblem &pw, const DwProblem &dw) {
    if (pw.cfg.id != GEMM_THIN || pw.k_pad > 256 || pw.k > pw.k_pad || (pw.k & 7) != 0 || (pw.cin & 7) != 0 || pw.k != pw.cin) return false;
    if (pw.stride_h != 1 || pw.stride_w != 1 || pw.y_base != 0 || pw.x_base != 0 || pw.ho != pw.h || pw.wo != pw.w) return false;
    if (pw.a_xor != 0x80808080u || pw.out_xor != 0u || pw.residual) return false;
    if ((pw.rq.pc_multiplier != nullptr) != (dw.rq.pc_multiplier != nullptr)) return false;
    if (!pwdw_block_takes(dw) || dw.c != pw.n || dw.h != pw.h || dw.w_ != pw.w || (!dw.w_trip && !dw.w_fold)) return false;
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
// A shape that is not in the table runs as two launches.
bool pwdw_block_listed(int32_t images, int32_t image_h, int32_t image_w, int32_t in_channels, int32_t expanded_channels, int32_t stride) {
    // Below 32 images a launch is mostly latency, and one launch instead of two wins for the whole network:
    // MobileNetV2 with all 16 fitting pairs fused against the listed ones, 144 against 162 us at batch 1, 168 against 176
    // at 4, 206 against 222 at 8, 246 against 260 at 16, 288 against 294 at 24; at 32 it is a draw, 324.2 against 324.6.
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

bool pwdw_block_geometry(const GemmProblem &pw, const DwProblem &dw, int rows_per_tile, int cols_per_tile, BlockGeom *geom) {
    const int S = dw.stride_h;
    BlockGeom g;
    g.c = dw.c;
    g.ks = pw.k_pad / 32;
    g.a_pitch = g.ks * 32 + 16;
    const int nb_all = (dw.c + 31) / 32;
    // Tile shape and channel blocks per workgroup.  A workgroup's three stages run one after the other, so the stages
    // of different workgroups have to overlap on a CU: the shapes considered leave room for four or more workgroups in
    // a CU's LDS (measured: tiles of twice that size take twice as long at a batch of 256, however little halo they
    // recompute) and, where the problem is large enough, give the launch at least three workgroups per CU.  Among those
    // the one that computes the fewest pixel slots wins, counting the slots that pixel blocks of 32 and output tiles of
    // four leave empty and, at a lower weight, the input bytes staged again for every channel range.
    int th = rows_per_tile, tw = cols_per_tile, nb = nb_all;
    // Form of the depthwise stage.  The matrix form works in units of sixteen output pixels by sixteen channels, spread over the four
    // waves, the vector form in units of four by four, some 300 instructions each, one to a thread: with few of them a workgroup waits
    // for that chain, however few threads walk it.  With more than a matrix unit to a wave it is a matter of their fill and of their
    // epilogue, which a pair per channel doubles.  The same tiles, vector -> matrix form, us (with a pair per channel):
    //   up to 3 units  28x28 32 -> 192 stride 2, 2 images 5.4 -> 4.2 (6.1 -> 4.6), stride 1, 2 images 4.6 -> 4.3 (4.9 -> 4.6),
    //                  7x7 160 -> 960, 1 image 5.3 -> 4.55 (6.1 -> 5.05)
    //   4              56x56 24 -> 144 stride 2, 4 images 5.4 -> 4.75 (6.1 -> 5.5), 28x28 32 -> 192 stride 1, 4 images 4.7 -> 4.8
    //                  (5.25 -> 5.4), 14x14 64 -> 384, 4 images 4.9 -> 4.8 (5.35 -> 5.5), 7x7 160 -> 960, 4 images 5.4 -> 5.2 (5.85 -> 5.8)
    //   6, full        56x56 24 -> 144 stride 2, 6 images 5.8 -> 5.1 (6.6 -> 6.0), 28x28 32 -> 192, 8 images 6.2 -> 6.0 (6.8 -> 7.1), at
    //                  stride 2, 24 images 6.5 -> 6.0 (7.4 -> 7.15)
    //   6, half full   28x28 32 -> 192 stride 2, 8 images 5.2 -> 5.35 (5.6 -> 6.4), 14x14 96 -> 576, 4 images 5.2 -> 5.7 (5.9 -> 6.7)
    //   8, full        14x14 96 -> 576, 8 images 5.9 -> 5.6 (6.6 -> 6.7), 64 -> 384, 16 images 6.0 -> 6.05 (6.85 -> 7.3)
    //   9 and 10, full 56x56 24 -> 144 stride 2, 12 images 7.1 -> 7.5 (8.4 -> 9.2), 14x14 96 -> 576, 12 images 6.5 -> 6.6 (7.3 -> 8.0),
    //                  33x33 48 -> 288, 4 images 5.8 -> 6.2 (6.5 -> 7.6)
    const bool per_channel = pw.rq.pc_multiplier != nullptr;
    auto quads_of = [&](int blocks) { return blocks * 8 < dw.c / 4 ? blocks * 8 : dw.c / 4; };
    auto matrix_form = [&](int rows, int cols, int blocks) {
        const int groups = (rows * cols + 15) / 16, units = groups * (quads_of(blocks) / 4);
        return dw.w_mm != nullptr && units <= (!per_channel ? 8 : S == 2 ? 6 : 3) && (units <= 4 || rows * cols > groups * 8);
    };
    {
        double best = -1;
        int best_th = 1, best_tw = dw.wo < 4 ? dw.wo : 4, best_nb = 1;
        for (int pass = 0; pass < 3 && best < 0; ++pass)  // later passes: fewer workgroups, then anything that fits at all
            for (int cn = 1; cn <= nb_all; ++cn) {
                const int ranges = (nb_all + cn - 1) / cn;
                if ((ranges - 1) * cn >= nb_all) continue;  // the same ranges with fewer blocks each
                for (int ch = 1; ch <= dw.ho && ch <= 16; ++ch)
                    for (int cw = 1; cw <= dw.wo && cw <= 64; ++cw) {
                        if (rows_per_tile > 0 && ch != rows_per_tile) continue;
                        if (cols_per_tile > 0 && cw != cols_per_tile) continue;
                        const int ih = (ch - 1) * S + 3, iw = (cw - 1) * S + 3;
                        const size_t lds = block_lds_bytes(cn, g.ks, ih, iw, dw.c, nullptr, nullptr);
                        if (pass < 2 ? lds * 4 > 144 * 1024 : lds > kBlockLdsMax) continue;
                        const long wgs = (long)dw.n * ((dw.ho + ch - 1) / ch) * ((dw.wo + cw - 1) / cw) * ranges;
                        if (pass == 0 && wgs < 768) continue;
                        const int px = ih * iw;
                        const double tiles = (double)dw.n * ((dw.ho + ch - 1) / ch) * ((dw.wo + cw - 1) / cw);
                        const double stage1 = (double)((px + 31) / 32 * 32) * tiles / ((double)dw.n * dw.h * dw.w_);   // pixel slots computed per real pixel
                        // A tile of up to 128 vector units (half the threads) is priced by whole groups of sixteen outputs, a slot of them at
                        // three quarters, whichever form will run it: by the vector form's own slots the search prefers tiles of two outputs
                        // or four, whose chain is as long and whose halo is larger.  Tiles by groups and by slots, us (with a pair per
                        // channel): both matrix, 56x56 24 -> 144 stride 2, one image 4.15 and 4.5 (4.6 and 5.0); matrix and vector, 28x28
                        // 32 -> 192 stride 2, 16 images 5.0 and 5.8 (5.8 and 6.6); both vector, 56x56 24 -> 144 stride 2, two images 5.0 and
                        // 5.15 (5.3 and 5.35), 14x14 96 -> 576 stride 2, 24 images 6.2 and 6.3 (7.15 and 7.1).
                        const bool small = ch * ((cw + 3) / 4) * quads_of(cn) <= 128;
                        const double slots = small ? 0.75 * ((ch * cw + 15) / 16 * 16) : (double)(ch * ((cw + 3) / 4 * 4));
                        const double stage2 = slots * tiles / ((double)dw.n * dw.ho * dw.wo);  // output slots per real output
                        const double restage = (double)px * tiles * ranges * (g.ks * 32) / ((double)dw.n * dw.h * dw.w_ * dw.c);  // staged input bytes per expanded byte
                        const double cost = stage1 + 0.5 * stage2 + 2.0 * restage;
                        if (best < 0 || cost < best) {
                            best = cost;
                            best_th = ch;
                            best_tw = cw;
                            best_nb = cn;
                        }
                    }
            }
        if (best < 0) return false;
        th = best_th;
        tw = best_tw;
        nb = best_nb;
    }
    g.nb = nb;
    if (!(th >= 1 && th <= dw.ho && tw >= 1 && tw <= dw.wo)) return false;
    g.th = th;
    g.tw = tw;
    g.ih = (th - 1) * S + 3;
    g.iwp = (tw - 1) * S + 3;
    g.pixels = g.ih * g.iwp;
    g.tiles_x = (tw + 3) / 4;
    g.tiles_y = (dw.ho + th - 1) / th;
    g.tiles_w = (dw.wo + tw - 1) / tw;
    g.total_tiles = dw.n * g.tiles_y * g.tiles_w;
    g.units_per_cq = th * g.tiles_x;
    g.div_iwp = make_fastdiv((uint32_t)g.iwp);
    g.div_tx = make_fastdiv((uint32_t)g.tiles_x);
    g.div_tw = make_fastdiv((uint32_t)tw);
    g.div_tiles_y = make_fastdiv((uint32_t)g.tiles_y);
    g.div_tiles_w = make_fastdiv((uint32_t)g.tiles_w);
    g.div_ppp = make_fastdiv((uint32_t)(g.ks * 4));
    const int ranges = (nb_all + g.nb - 1) / g.nb;
    g.div_cq = make_fastdiv((uint32_t)(g.nb * 8 < g.c / 4 ? g.nb * 8 : g.c / 4));
    g.div_cq_last = make_fastdiv((uint32_t)((g.c - (ranges - 1) * g.nb * 32) / 4));
    g.cpitch = block_image_pitch(g.nb, g.c);
    g.matrix = matrix_form(th, tw, nb) ? 1 : 0;
    const size_t lds = block_lds_bytes(g.nb, g.ks, g.ih, g.iwp, g.c, &g.a_off, &g.image_off);
    if (lds > kBlockLdsMax) return false;
    *geom = g;
    return true;
}

// `g`: what pwdw_block_geometry gave for the pair (the search over tiles costs the host as much as the launch: callers keep it)
int launch_pwdw_block(const GemmProblem &pw, const DwProblem &caller_dw, const BlockGeom &g, hipStream_t stream) {
    EH_REQUIRE(pwdw_block_applies(pw, caller_dw), "block: the two operators do not fit the fused kernel");
    EH_REQUIRE((reinterpret_cast<uintptr_t>(pw.a) & 7) == 0 && (reinterpret_cast<uintptr_t>(caller_dw.out) & 3) == 0, "block: unaligned tensors");
    EH_REQUIRE(g.c == caller_dw.c && g.ks == pw.k_pad / 32, "block: geometry of another pair");
    DwProblem dw = caller_dw;
    if (dw.w_trip) dw.w_fold = nullptr;                 // the signed form where it applies, as the stand-alone launcher decides
    if (dw.w_fold) dw.zp_w += dw.w_signed ? 128 : 0;    // zero point of the uint8 values the unsigned form multiplies
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
        return pw.rq.pc_multiplier ? launch_pc(s_c, form_c, rowsum_c, qm_c, ks_c, std::true_type{}) : launch_pc(s_c, form_c, rowsum_c, qm_c, ks_c, std::false_type{});
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
        if (g.matrix) return with_rowsum(s_c, std::integral_constant<DwForm, DwForm::MATRIX>{});
        return dw.w_trip ? with_rowsum(s_c, std::integral_constant<DwForm, DwForm::DOT>{}) : with_rowsum(s_c, std::integral_constant<DwForm, DwForm::FOLD>{});
    };
    const int rc = S == 1 ? with_form(std::integral_constant<int, 1>{}) : with_form(std::integral_constant<int, 2>{});
    if (rc) return rc;
    EH_HIP(hipGetLastError());
    return EH_OK;
}

}  // namespace eh
