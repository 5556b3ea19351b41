// First-layer convolution: 3 input channels, 3x3 taps (any stride and padding),
// channels-last uint8.  The 27 reduction bytes of an output pixel are three runs
// of nine contiguous input bytes (one per kernel row), so no im2col staging is
// needed: a thread gathers them with three unaligned 12-byte reads, replaces the
// taps that fall outside the image by the input zero point, and holds them as
// seven signed dwords.  It then produces 16 output channels with v_dot4 against
// weight rows that are uniform across the wave (scalar loads), requantizes and
// writes 16 bytes.  Arithmetic is the implicit-GEMM one: a' = a ^ 0x80 against
// w - 128 with the zero-point terms folded into the bias and a per-pixel
// correction -(zp_w - 128) * sum(a').
//
// With 32 output channels or more the multiply-adds go to the matrix cores instead (conv_c3k3_mfma_kernel): a
// lane still gathers one pixel, the two halves of the wave then exchange half of what they gathered so that each
// of the wave's two 32-pixel blocks has its 27 (+5 zero) reduction bytes in 32x32x32 fragment form, and one
// v_mfma_i32_32x32x32_i8 per block and 32 channels leaves every lane with 16 consecutive channels of one pixel.
//
// A wavefront of 64 pixels x 32 channels is 358 vector instructions, 426 with a pair per channel (SQ_INSTS_VALU / SQ_WAVES; multiply,
// clamp and shift of a lane's 32 values are 96 of them): at 32 images 3.7 of the 7.9 us, the rest is waiting, 45 % of the waves' cycles.
// 224x224, stride 2, 32 channels, before and after the rows, the weights and the bias (and a channel's pair) were requested
// ahead of their first use: one image 3.95 -> 3.20 us, 32 images 9.31 -> 7.77, 64 images 13.54 -> 11.50; with a pair per
// channel 4.62 -> 3.47, 11.43 -> 9.76 and 18.74 -> 15.61 (14.41 with the four-channel requantization); 160x160 to 96
// channels, 8 images 8.81 -> 5.96.  With fewer than 32 channels: 224x224 to 16, 32 images 7.17 -> 6.89.
//
// Stands in for the reference's direct convolution kernels on this shape
// (gpu/operators/cl_kernels/DirectConvolutionKernel.cpp, 3x3 uint8 variants).
#include <type_traits>

#include "eh_internal.h"

namespace eh {
namespace {

typedef uint32_t u32_unaligned __attribute__((aligned(1)));
typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v16i __attribute__((ext_vector_type(16)));
typedef uint32_t u32x4_a4 __attribute__((ext_vector_type(4), aligned(4)));

// The 27 reduction bytes of output pixel m < p.m as seven dwords of a' = a ^ a_xor (the 28th byte zero), out-of-image
// taps reading the input zero point; `pixel` is where the output pixel lies in the output's rows.
//
// Every row is read, the ones outside the image from the nearest inside, and all three before the first is used: with
// each row's loads in a branch of its own the compiler waited for one row before it asked for the next.  Where twelve
// bytes would leave the tensor at its first or last pixels, the twelve inside are read and the bytes moved into place.
__device__ __forceinline__ void gather_c3k3(const GemmProblem &p, const uint32_t in_bytes, int m, uint32_t (&A)[7], uint32_t &pixel) {
    const int plane = p.ho * p.wo;
    const int img = (int)fastdiv((uint32_t)m, p.div_plane), rem = m - img * plane;
    const int oy = (int)fastdiv((uint32_t)rem, p.div_wo), ox = rem - oy * p.wo;
    pixel = (uint32_t)((img * p.out_h + (oy * p.out_sy + p.out_y0)) * p.out_w + (ox * p.out_sx + p.out_x0));
    const int iy0 = oy * p.stride_h + p.y_base, ix0 = ox * p.stride_w + p.x_base;
    const bool c0 = (unsigned)ix0 < (unsigned)p.w, c1 = (unsigned)(ix0 + 1) < (unsigned)p.w, c2 = (unsigned)(ix0 + 2) < (unsigned)p.w;
    // (tensors stay below 2 GiB: 32-bit offsets)
    uint32_t d[3][3];
    int past[3];  // how far a row's nine bytes lie past the twelve that were read
    const int last = (int)in_bytes - 12;
    if (last >= 0) {
#pragma unroll
        for (int ky = 0; ky < 3; ++ky) {
            const int iy = iy0 + ky, iyc = iy < 0 ? 0 : (iy < p.h ? iy : p.h - 1);
            const int a = ((img * p.h + iyc) * p.w + ix0) * 3, ac = a < 0 ? 0 : (a < last ? a : last);
            past[ky] = a - ac;
#pragma unroll
            for (int i = 0; i < 3; ++i) d[ky][i] = *reinterpret_cast<const u32_unaligned *>(p.a + ac + 4 * i);  // (a three-element vector would read sixteen bytes)
        }
        if (__builtin_amdgcn_ballot_w64((past[0] | past[1] | past[2]) != 0) != 0) {
#pragma unroll
            for (int ky = 0; ky < 3; ++ky)
#pragma unroll
                for (int step = 3; step <= 9; step += 3) {  // (a multiple of three, like every pixel's address and the tensor's length)
                    uint32_t &x = d[ky][0], &y = d[ky][1], &z = d[ky][2];
                    if (past[ky] >= step) {
                        x = __builtin_amdgcn_alignbyte(y, x, 3);
                        y = __builtin_amdgcn_alignbyte(z, y, 3);
                        z = z >> 24;
                    }
                    if (past[ky] <= -step) {
                        z = __builtin_amdgcn_alignbyte(z, y, 1);
                        y = __builtin_amdgcn_alignbyte(y, x, 1);
                        x = x << 24;
                    }
                }
        }
    } else {  // a tensor of three pixels at most
#pragma unroll
        for (int ky = 0; ky < 3; ++ky) {
            const int iy = iy0 + ky, iyc = iy < 0 ? 0 : (iy < p.h ? iy : p.h - 1);
            uint32_t lo = 0, mid = 0, hi = 0;
#pragma unroll 1
            for (int j = 0; j < 9; ++j) {  // the first byte is shifted in last
                const int b = ((img * p.h + iyc) * p.w + ix0) * 3 + 8 - j;
                const uint32_t v = b >= 0 && (uint32_t)b < in_bytes ? p.a[b] : 0u;
                hi = __builtin_amdgcn_alignbyte(hi, mid, 3);
                mid = __builtin_amdgcn_alignbyte(mid, lo, 3);
                lo = lo << 8 | v;
            }
            d[ky][0] = lo, d[ky][1] = mid, d[ky][2] = hi;
        }
    }
    uint32_t seg[3][3];  // per kernel row: bytes 0..8 = 3 pixels x 3 channels, the rest zero
#pragma unroll
    for (int ky = 0; ky < 3; ++ky) {
        const bool row_ok = (unsigned)(iy0 + ky) < (unsigned)p.h;
        const bool v0 = row_ok && c0, v1 = row_ok && c1, v2 = row_ok && c2;
        const uint32_t m0 = (v0 ? 0x00FFFFFFu : 0u) | (v1 ? 0xFF000000u : 0u);
        const uint32_t m1 = (v1 ? 0x0000FFFFu : 0u) | (v2 ? 0xFFFF0000u : 0u);
        const uint32_t m2 = v2 ? 0x000000FFu : 0u;
        seg[ky][0] = (d[ky][0] & m0) | (p.fill & ~m0);
        seg[ky][1] = (d[ky][1] & m1) | (p.fill & ~m1);
        seg[ky][2] = ((d[ky][2] & m2) | (p.fill & ~m2)) & 0xFFu;
    }
    A[0] = seg[0][0];
    A[1] = seg[0][1];
    A[2] = seg[0][2] | (seg[1][0] << 8);
    A[3] = __builtin_amdgcn_alignbyte(seg[1][1], seg[1][0], 3);
    A[4] = (__builtin_amdgcn_alignbyte(seg[1][2], seg[1][1], 3) & 0xFFFFu) | (seg[2][0] << 16);
    A[5] = __builtin_amdgcn_alignbyte(seg[2][1], seg[2][0], 2);
    A[6] = __builtin_amdgcn_alignbyte(seg[2][2], seg[2][1], 2);
#pragma unroll
    for (int i = 0; i < 7; ++i) A[i] ^= p.a_xor;
    A[6] &= 0x00FFFFFFu;
}

// Matrix-core form.  Grid: x = 256 pixels per workgroup (64 per wave).  With one multiplier and shift per channel,
// FAST means that every channel's pair is inside the single-shift form's range.
template <bool ROWSUM, bool FAST, bool PLANAR, bool PC>
__global__ __launch_bounds__(256) void conv_c3k3_mfma_kernel(const GemmProblem p, const uint32_t in_bytes) {
    const int lane = threadIdx.x & 63, r = lane & 31, half = lane >> 5;
    // every XCD (workgroups are dispatched round-robin over the 8 of them) takes one contiguous eighth of the
    // pixel range, so the input rows that neighbouring output rows share are fetched into one L2 only
    const int block = (int)((blockIdx.x & 7u) * (gridDim.x >> 3) + (blockIdx.x >> 3));
    const int m_own = block * 256 + threadIdx.x;  // the pixel this lane gathers
    // weight rows are stored plainly, [channel][32 bytes]: row `r` of the fragment is channel 16 h + 4 g + t of the block
    const int8_t *const w_own = p.b + (size_t)(16 * ((r >> 2) & 1) + 4 * (r >> 3) + (r & 3)) * 32 + half * 16;
    v4i wf;
    int4 bias[4], mult[4], shift[4];
    auto request = [&](int nb) {
        const int n = nb * 32 + half * 16;
        wf = *reinterpret_cast<const v4i *>(w_own + (size_t)nb * (32 * 32));
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            bias[g] = *reinterpret_cast<const int4 *>(p.bias + n + g * 4);
            if constexpr (PC) {  // (the arrays are padded past the last channel block)
                mult[g] = *reinterpret_cast<const int4 *>(p.rq.pc_multiplier + n + g * 4);
                shift[g] = *reinterpret_cast<const int4 *>(p.rq.pc_shift + n + g * 4);
            }
        }
    };
    request(0);  // on its way while the pixels are gathered
    uint32_t A[7], pixel_own;
    gather_c3k3(p, in_bytes, m_own < p.m ? m_own : p.m - 1, A, pixel_own);
    int rs_own = 0;
    if constexpr (ROWSUM) {
#pragma unroll
        for (int i = 0; i < 7; ++i) rs_own = __builtin_amdgcn_sdot4((int)A[i], 0x01010101, rs_own, false);
    }
    // Lanes 0..31 hold pixels 0..31 of the wave, lanes 32..63 pixels 32..63.  Block b's fragment wants, in lane
    // (r, half), reduction bytes 16 half .. 16 half + 15 of pixel 32 b + r: the lower lanes send the upper half of
    // their bytes up (block 0), the upper lanes send the lower half of theirs down (block 1).
    uint32_t got[4];
#pragma unroll
    for (int d = 0; d < 4; ++d) got[d] = (uint32_t)__shfl_xor((int)(half ? A[d] : (d < 3 ? A[4 + d] : 0u)), 32);
    v4i af[2];
    af[0] = half ? v4i{(int)got[0], (int)got[1], (int)got[2], (int)got[3]} : v4i{(int)A[0], (int)A[1], (int)A[2], (int)A[3]};
    af[1] = half ? v4i{(int)A[4], (int)A[5], (int)A[6], 0} : v4i{(int)got[0], (int)got[1], (int)got[2], (int)got[3]};
    const int rs_got = ROWSUM ? __shfl_xor(rs_own, 32) : 0;
    const uint32_t pixel_got = (uint32_t)__shfl_xor((int)pixel_own, 32);
    const int wave_base = m_own - lane;
    const RequantDev rq = p.rq;
    const int n_blocks = (p.n + 31) >> 5;
    for (int nb = 0; nb < n_blocks; ++nb) {
        const int n = nb * 32 + half * 16;
        if (nb != 0) request(nb);
#pragma unroll
        for (int b = 0; b < 2; ++b) {
            const int m = wave_base + 32 * b + r;  // the pixel whose 16 channels this lane finishes in block b
            const int ncorr = ROWSUM ? -p.zw * (b == half ? rs_own : rs_got) : 0;
            const size_t out_off = (size_t)(b == half ? pixel_own : pixel_got) * (size_t)p.ldc;
            // the accumulators start from the folded bias and the pixel's row-sum term: nothing left to add afterwards
            v16i acc;
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                acc[g * 4 + 0] = bias[g].x + ncorr;
                acc[g * 4 + 1] = bias[g].y + ncorr;
                acc[g * 4 + 2] = bias[g].z + ncorr;
                acc[g * 4 + 3] = bias[g].w + ncorr;
            }
            acc = __builtin_amdgcn_mfma_i32_32x32x32_i8(wf, af[b], acc, 0, 0, 0);
            uint32_t packed[4];
            auto produce = [&](auto mode_c) {
                constexpr int mode = decltype(mode_c)::value;
#pragma unroll
                for (int g = 0; g < 4; ++g) {
                    if constexpr (PC && mode != 0)
                        packed[g] = requant4_channel<mode>(acc[g * 4 + 0], acc[g * 4 + 1], acc[g * 4 + 2], acc[g * 4 + 3], mult[g], channel_shift_bytes(shift[g]), rq) ^ p.out_xor;
                    else if constexpr (PC) {
                        auto one = [&](int x, int32_t mu, int32_t sh) {
#if defined(__HIP_DEVICE_COMPILE__)
                            asm("" : "+v"(sh));  // (a channel's terms are worked out for each block: kept for both they would cost a wavefront)
#endif
                            return requant_u8_channel(x, mu, sh, rq);
                        };
                        packed[g] = pack_bytes(one(acc[g * 4 + 0], mult[g].x, shift[g].x), one(acc[g * 4 + 1], mult[g].y, shift[g].y),
                                               one(acc[g * 4 + 2], mult[g].z, shift[g].z), one(acc[g * 4 + 3], mult[g].w, shift[g].w)) ^
                                    p.out_xor;
                    } else if constexpr (mode != 0)
                        packed[g] = requant4_fast<mode>(acc[g * 4 + 0], acc[g * 4 + 1], acc[g * 4 + 2], acc[g * 4 + 3], 0, rq) ^ p.out_xor;
                    else
                        packed[g] = pack_bytes(requant_u8_as<mode>(acc[g * 4 + 0], rq), requant_u8_as<mode>(acc[g * 4 + 1], rq),
                                               requant_u8_as<mode>(acc[g * 4 + 2], rq), requant_u8_as<mode>(acc[g * 4 + 3], rq)) ^
                                    p.out_xor;
                }
            };
            if constexpr (!FAST)
                produce(std::integral_constant<int, 0>{});
            else if (rq.fast == 2)
                produce(std::integral_constant<int, 2>{});
            else
                produce(std::integral_constant<int, 1>{});
            if (m < p.m && n < p.n) {
                uint8_t *dst = p.out + out_off + n;
                const int cnt = p.n - n;
                if constexpr (PLANAR) {
                    store_bytes_planar(p.out, p.planar, out_off, n, packed, cnt);
                } else if (cnt >= 16 && (p.ldc & 3) == 0 && (reinterpret_cast<uintptr_t>(p.out) & 3) == 0) {
                    *reinterpret_cast<u32x4_a4 *>(dst) = u32x4_a4{packed[0], packed[1], packed[2], packed[3]};
                } else {
                    store_bytes_any_alignment(dst, packed, cnt < 16 ? cnt : 16);
                }
            }
        }
    }
}

template <bool ROWSUM, bool FAST, bool PLANAR>
__global__ __launch_bounds__(256) void conv_c3k3_kernel(const GemmProblem p, const uint32_t in_bytes) {
    const int m = blockIdx.x * 256 + threadIdx.x;
    if (m >= p.m) return;
    const int n0 = blockIdx.y * 16;
    // reduction order (kernel row, kernel column, channel): 27 bytes in seven dwords, the 28th byte is zero
    uint32_t A[7], pixel;
    gather_c3k3(p, in_bytes, m, A, pixel);
    int ncorr = 0;
    if constexpr (ROWSUM) {
        int rs = 0;
#pragma unroll
        for (int i = 0; i < 7; ++i) rs = __builtin_amdgcn_sdot4((int)A[i], 0x01010101, rs, false);
        ncorr = -p.zw * rs;
    }
    const RequantDev rq = p.rq;
    uint32_t packed[4];
    auto produce = [&](auto mode_c) {
    constexpr int mode = decltype(mode_c)::value;
#pragma unroll
    for (int g = 0; g < 4; ++g) {
        uint32_t o[4];
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            const int n = n0 + g * 4 + t;  // uniform across the wave: the weight row and bias come through the scalar unit
            const int *wrow = reinterpret_cast<const int *>(p.b + (size_t)n * 32);
            int acc = p.bias[n] + ncorr;
#pragma unroll
            for (int i = 0; i < 7; ++i) acc = __builtin_amdgcn_sdot4((int)A[i], wrow[i], acc, false);
            o[t] = mode == 0 && rq.pc_multiplier ? requant_u8_channel(acc, rq.pc_multiplier[n], rq.pc_shift[n], rq)
                                                 : requant_u8_as<mode>(acc, rq);
        }
        packed[g] = pack_bytes(o[0], o[1], o[2], o[3]) ^ p.out_xor;
    }
    };
    if constexpr (!FAST)
        produce(std::integral_constant<int, 0>{});
    else if (rq.fast == 2)
        produce(std::integral_constant<int, 2>{});
    else
        produce(std::integral_constant<int, 1>{});
    uint8_t *dst = p.out + (size_t)pixel * (size_t)p.ldc + n0;
    const bool aligned16 = (p.ldc & 15) == 0 && ((reinterpret_cast<uintptr_t>(p.out) & 15) == 0);
    if constexpr (PLANAR) {
        store_bytes_planar(p.out, p.planar, (size_t)(dst - p.out) - (size_t)n0, n0, packed, p.n - n0);
    } else if (aligned16 && n0 + 16 <= p.n) {
        *reinterpret_cast<uint4 *>(dst) = make_uint4(packed[0], packed[1], packed[2], packed[3]);
    } else {
        store_bytes_any_alignment(dst, packed, p.n - n0 < 16 ? p.n - n0 : 16);
    }
}

}  // namespace

int launch_conv_c3k3(const GemmProblem &p, hipStream_t stream) {
    EH_REQUIRE(p.k == 27 && p.k_pad == 32 && p.cin == 3, "conv_c3k3: not a 3-channel 3x3 problem");
    const size_t in_bytes = (size_t)p.h * p.w * 3;  // per image
    const int images = (p.m + p.ho * p.wo - 1) / (p.ho * p.wo);
    EH_REQUIRE(in_bytes * images < (1ull << 31), "conv_c3k3: input too large");
    const uint32_t total_bytes = (uint32_t)(in_bytes * images);
    const bool rowsum = p.zw != 0;
    bool fast = p.rq.fast != 0;
    auto launch_variant = [&](auto launch) {
        auto with_planar = [&](auto rs, auto f) { p.planar.out_plane ? launch(rs, f, std::true_type{}) : launch(rs, f, std::false_type{}); };
        auto with_fast = [&](auto rs) { fast ? with_planar(rs, std::true_type{}) : with_planar(rs, std::false_type{}); };
        rowsum ? with_fast(std::true_type{}) : with_fast(std::false_type{});
    };
    if (p.n >= 32) {  // the packed rows and the folded bias are padded to whole tiles of channels
        const dim3 grid_m(((p.m + 255) / 256 + 7) / 8 * 8);  // whole multiples of 8: see the kernel's block numbering
        launch_variant([&](auto rs, auto f, auto pl) {
            constexpr bool ROWSUM = decltype(rs)::value, FAST = decltype(f)::value, PLANAR = decltype(pl)::value;
            if (p.rq.pc_multiplier)
                hipLaunchKernelGGL((conv_c3k3_mfma_kernel<ROWSUM, FAST, PLANAR, true>), grid_m, dim3(256), 0, stream, p, total_bytes);
            else
                hipLaunchKernelGGL((conv_c3k3_mfma_kernel<ROWSUM, FAST, PLANAR, false>), grid_m, dim3(256), 0, stream, p, total_bytes);
        });
        EH_HIP(hipGetLastError());
        return EH_OK;
    }
    const dim3 grid((p.m + 255) / 256, (p.n + 15) / 16);
    if (p.rq.pc_multiplier) fast = false;  // this kernel's per-channel code is the two-step order
    launch_variant([&](auto rs, auto f, auto pl) {
        hipLaunchKernelGGL((conv_c3k3_kernel<decltype(rs)::value, decltype(f)::value, decltype(pl)::value>), grid, dim3(256), 0, stream, p, total_bytes);
    });
    EH_HIP(hipGetLastError());
    return EH_OK;
}

}  // namespace eh
