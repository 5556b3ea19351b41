// uint8 implicit GEMM for problems with few output tiles: a layer of a network at batch 1, a classifier head, a phase of a
// small transposed convolution, a fully connected layer on a few rows.
//
// Such a launch is latency: the tiled kernels put one 64 x 64 tile on a CU and walk its reduction slab by slab, each slab a
// trip through L2 into LDS (3x3 on 256 channels at 14 x 14, one image: 16 workgroups of nine slabs, 9.1 us).  Here a
// workgroup owns 32 pixels x 32 output channels and its eight waves share the reduction: wave w takes the 128-byte groups
// w, w + 8, ... and requests all of its operands (up to three groups at a time) straight into registers before it
// multiplies the first, so the whole reduction costs about one memory latency.  Weights are packed in MFMA fragment
// order; a lane's activation chunk of 16 channels lies inside one kernel tap, whose place follows from the chunk's
// number by two divisions, so there is no tap table to fetch first.  The eight partial tiles and the pixels' byte sums meet in LDS; every thread finishes two channels of one
// pixel, whose bias, per-channel pair and residual bytes it requested at the very start.
#include <type_traits>

#include "eh_internal.h"

namespace eh {
namespace {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v16i __attribute__((ext_vector_type(16)));

constexpr int kWaves = 8;
constexpr int kLanePitch = 20;  // int32 per lane of a partial tile: 16 and a gap that spreads 16-byte accesses over the banks

// What this kernel reads of a problem: fields of GemmProblem by the same names, and the taps' geometry.  (3x3 on 256 channels at
// 14 x 14, one image: 5.35 us with a GemmProblem that held the geometry, 376 bytes; 6.07 at 512 bytes; 5.30 with this one.)
struct FewProblem {
    const uint8_t *a;
    const int8_t *b;
    const int32_t *bias;
    uint8_t *out;
    const uint8_t *residual;
    int32_t m, n, k, k_pad;
    int32_t h, w, cin, ho, wo;
    int32_t stride_h, stride_w, y_base, x_base;
    FastDiv div_plane, div_wo;
    TapGeom tap;
    uint32_t fill, a_xor, out_xor;
    int32_t zw;
    int32_t out_h, out_w, out_sy, out_sx, out_y0, out_x0, ldc;
    union {
        AddDev radd;
        PlanarOut planar;
    };
    int32_t c_last;
    RequantDev rq;

    FewProblem() {}
    FewProblem(const TapProblem &p)
        : a(p.a), b(p.b), bias(p.bias), out(p.out), residual(p.residual), m(p.m), n(p.n), k(p.k), k_pad(p.k_pad), h(p.h), w(p.w), cin(p.cin), ho(p.ho), wo(p.wo),
          stride_h(p.stride_h), stride_w(p.stride_w), y_base(p.y_base), x_base(p.x_base), div_plane(p.div_plane), div_wo(p.div_wo), tap(p.tap), fill(p.fill),
          a_xor(p.a_xor), out_xor(p.out_xor), zw(p.zw), out_h(p.out_h), out_w(p.out_w), out_sy(p.out_sy), out_sx(p.out_sx), out_y0(p.out_y0), out_x0(p.out_x0),
          ldc(p.ldc), radd(p.radd), c_last(p.c_last), rq(p.rq) {}  // (radd's bytes are `planar` where that is in use)
};
static_assert(sizeof(FewProblem) == 328, "c_last lies in what alignment leaves free: 3x3 on 256 channels at 14 x 14, one image, 5.31 us; in front of the union 5.41");
struct FewBatch {
    FewProblem p[GemmBatch::MAX];
};
__device__ __forceinline__ const FewProblem &problem_of(const FewProblem &one) { return one; }
__device__ __forceinline__ const FewProblem &problem_of(const FewBatch &batch) { return batch.p[blockIdx.z]; }

// the value of lane (lane ^ 1) or (lane ^ 2): a permutation inside every four lanes
template <int X>
__device__ __forceinline__ int quad_xor(int v) {
    constexpr int perm = X == 1 ? (1 | 0 << 2 | 3 << 4 | 2 << 6) : (2 | 3 << 2 | 0 << 4 | 1 << 6);
    return __builtin_amdgcn_update_dpp(0, v, perm, 0xF, 0xF, true);
}
// lane U's value in every lane of its four
template <int U>
__device__ __forceinline__ int quad_lane(int v) {
    return __builtin_amdgcn_update_dpp(0, v, U | U << 2 | U << 4 | U << 6, 0xF, 0xF, true);
}
// Transposes, inside every four lanes, the 4 x 4 matrix whose row is the lane and whose column is the register.
__device__ __forceinline__ void quad_transpose(int &c0, int &c1, int &c2, int &c3, bool odd, bool high) {
    auto swap1 = [&](int &u0, int &u1) {
        const int t = quad_xor<1>(odd ? u0 : u1);
        u0 = odd ? t : u0;
        u1 = odd ? u1 : t;
    };
    auto swap2 = [&](int &u0, int &u2) {
        const int t = quad_xor<2>(high ? u0 : u2);
        u0 = high ? t : u0;
        u2 = high ? u2 : t;
    };
    swap1(c0, c1);
    swap1(c2, c3);
    swap2(c0, c2);
    swap2(c1, c3);
}

typedef uint16_t u16x2 __attribute__((ext_vector_type(2)));
typedef v4i v4i_any_alignment __attribute__((aligned(1)));

// sixteen bytes shifted down by `bytes` of them (0 .. 15)
__device__ __forceinline__ v4i shift_bytes_down(v4i v, uint32_t bytes) {
    const uint64_t lo = (uint64_t)(uint32_t)v.x | (uint64_t)(uint32_t)v.y << 32, hi = (uint64_t)(uint32_t)v.z | (uint64_t)(uint32_t)v.w << 32;
    const uint32_t n = bytes * 8, part = n & 63u;
    const uint64_t down = part ? lo >> part | hi << (64u - part) : lo, top = hi >> part;
    const uint64_t a = n < 64u ? down : top, b = n < 64u ? top : 0u;
    return v4i{(int)(uint32_t)a, (int)(uint32_t)(a >> 32), (int)(uint32_t)b, (int)(uint32_t)(b >> 32)};
}
// the low `count` (0 or less .. 16 or more) of sixteen bytes' places, word d of the four
__device__ __forceinline__ uint32_t byte_mask(int count, int d) {
    const int left = count - 4 * d;
    return left >= 4 ? ~0u : left <= 0 ? 0u : (1u << (8 * left)) - 1u;
}

// GROUPS: 128-byte groups of the reduction a wave has on their way together.  TAPS: the reduction runs over kernel taps that
// may lie outside the image (else: one tap inside it).  ROWSUM: the weights' zero point is not 128.  FAST: every
// requantization pair in use is inside the single-shift form's range (or is told at run time).  BATCHED: equally shaped
// problems along grid z.  FORM: where the chunks are (InputForm).
//
// Ragged and planar tensors used to be brought into whole chunks by a launch of their own, which for a small layer costs as much as the
// layer (figures at gemm_few_tiles_direct).
// A ragged chunk is sixteen bytes at any address; what lies behind the tap's channels is replaced by the input zero point, the
// byte that the padded copy held, and a chunk that would end behind the tensor is read from sixteen bytes before its end and
// shifted down.  A planar chunk is sixteen single bytes a plane apart, which neighbouring lanes read from neighbouring pixels.
template <int GROUPS, bool TAPS, bool ROWSUM, bool FAST, bool BATCHED, int FORM>
__global__ __launch_bounds__(kWaves * 64) void few_tiles_kernel(const std::conditional_t<BATCHED, FewBatch, FewProblem> arg, const int m_blocks, const int n_blocks,
                                                                const int tiles_per_xcd, const int m_fastest) {
    const FewProblem &p = problem_of(arg);
    static_assert(FORM != INPUT_PLANAR || GROUPS <= 3, "a planar group is many loads on their way already");
    __shared__ __align__(16) int32_t part_s[kWaves][64 * kLanePitch];
    __shared__ int32_t sum_s[ROWSUM ? kWaves * 2 : 1][32];
    const int tid = threadIdx.x, lane = tid & 63, r = lane & 31, half = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    // XCD x (workgroups x, x + 8, ...) takes the x-th run of tiles; the operand whose blocks run slowest is fetched into one L2 only
    const int tile = (int)(blockIdx.x & 7u) * tiles_per_xcd + (int)(blockIdx.x >> 3);
    if ((int)(blockIdx.x >> 3) >= tiles_per_xcd || tile >= m_blocks * n_blocks) return;
    const int slow = __builtin_amdgcn_readfirstlane(tile / (m_fastest ? m_blocks : n_blocks));
    const int fast_i = tile - slow * (m_fastest ? m_blocks : n_blocks);
    const int mb = m_fastest ? fast_i : slow, nb = m_fastest ? slow : fast_i;
    // products of 32 bytes to a group; PLANAR: one, for the registers that single bytes take and so that more waves have a share
    // (3x3 21 -> 21 at 3 x 65x47 5.95 us with two, 5.06 with one)
    constexpr int STEPS = FORM == INPUT_PLANAR ? 1 : 4;
    const int groups = (p.k_pad + STEPS * 32 - 1) >> (STEPS == 1 ? 5 : 7), chunks = p.k_pad >> 4;

    // ---- where this lane's pixel reads
    const int m_in = mb * 32 + r;
    const int m_c = m_in < p.m ? m_in : p.m - 1;  // (pixels past the last one repeat it; nothing of theirs is stored)
    int iy0, ix0, base;
    {
        const int img = (int)fastdiv((uint32_t)m_c, p.div_plane), rem = m_c - img * (p.ho * p.wo);
        const int oy = (int)fastdiv((uint32_t)rem, p.div_wo), ox = rem - oy * p.wo;
        iy0 = oy * p.stride_h + p.y_base;
        ix0 = ox * p.stride_w + p.x_base;
        if constexpr (FORM == INPUT_PLANAR)
            base = ((img * p.cin + p.tap.c0) * p.h + iy0) * p.w + ix0;
        else
            base = ((img * p.h + iy0) * p.w + ix0) * p.cin + p.tap.c0;
    }
    // Activation loads: four neighbouring lanes fetch 64 contiguous bytes of ONE pixel (the cache answers a 64-byte piece
    // per cycle; four pixels' pieces take four), pixel by pixel of the four, and exchange them afterwards.
    const int4 q_base = make_int4(quad_lane<0>(base), quad_lane<1>(base), quad_lane<2>(base), quad_lane<3>(base));
    const int4 q_iy = make_int4(quad_lane<0>(iy0), quad_lane<1>(iy0), quad_lane<2>(iy0), quad_lane<3>(iy0));
    const int4 q_ix = make_int4(quad_lane<0>(ix0), quad_lane<1>(ix0), quad_lane<2>(ix0), quad_lane<3>(ix0));
    const bool odd = (lane & 1) != 0, high = (lane & 2) != 0;
    const v4i *wsrc = reinterpret_cast<const v4i *>(p.b) + (size_t)nb * chunks * 32 + r;  // + 32 per 16-byte chunk
    v16i acc;
#pragma unroll
    for (int i = 0; i < 16; ++i) acc[i] = 0;
    int rowsum[4] = {0, 0, 0, 0};
    // ---- what this thread finishes: two channels of one pixel
    const int f_px = tid >> 4, f_pair = tid & 15;
    const int f_m = mb * 32 + f_px, f_n = nb * 32 + f_pair * 2;
    int2 f_bias, f_mult = make_int2(0, 0), f_shift = make_int2(0, 0);
    uint32_t f_res0 = 0, f_res1 = 0;
    size_t f_off = 0;
    bool requested = false;
    auto request_finish = [&]() {  // behind the first operands: a first touch of memory each, hidden under theirs
        if (requested) return;
        requested = true;
        f_bias = *reinterpret_cast<const int2 *>(p.bias + f_n);  // (padded to whole channel blocks, as the per-channel arrays are)
        if (p.rq.pc_multiplier) {
            f_mult = *reinterpret_cast<const int2 *>(p.rq.pc_multiplier + f_n);
            f_shift = *reinterpret_cast<const int2 *>(p.rq.pc_shift + f_n);
        }
        const int mm = f_m < p.m ? f_m : p.m - 1;
        const int img = (int)fastdiv((uint32_t)mm, p.div_plane), rem = mm - img * (p.ho * p.wo);
        const int oy = (int)fastdiv((uint32_t)rem, p.div_wo), ox = rem - oy * p.wo;
        f_off = (((size_t)img * p.out_h + (oy * p.out_sy + p.out_y0)) * p.out_w + (ox * p.out_sx + p.out_x0)) * (size_t)p.ldc + (size_t)f_n;
        if (p.residual && f_m < p.m && f_n < p.n) {
            f_res0 = p.residual[f_off];
            if (f_n + 1 < p.n) f_res1 = p.residual[f_off + 1];
        }
    };

    uint32_t last_start = 0;  // RAGGED: where the last sixteen bytes of the tensor start (the host leaves smaller tensors to the padded copy)
    if constexpr (FORM == INPUT_RAGGED) last_start = fastdiv((uint32_t)p.m, p.div_plane) * (uint32_t)(p.h * p.w) * (uint32_t)p.cin - 16u;
    for (int g0 = wave; g0 < groups; g0 += kWaves * GROUPS) {
        // Group g is the reduction's bytes 128 g .. 128 g + 127: chunks 8 g + 4 half + u meet in its u-th product.  (PLANAR: a quarter of that.)
        v4i bf[GROUPS][STEPS], af[GROUPS][STEPS];
        uint32_t inside[GROUPS];   // bit px: pixel px's tap lies inside; RAGGED: bits 8 + 4 px on by how many bytes its chunk was read too early
        int valid[GROUPS];         // RAGGED: bytes of the chunk that are the tap's own
        bool exists[GROUPS];
#pragma unroll
        for (int u = 0; u < GROUPS; ++u) {
            const int g = g0 + u * kWaves;
            if (g >= groups) break;  // (uniform across the wave)
            auto place = [&](int chunk, int &dy, int &dx, int &c) {
                c = chunk;
                dy = dx = 0;
                if constexpr (TAPS) {
                    const int tap = (int)fastdiv((uint32_t)chunk, p.tap.div_chunks);
                    const int ty = (int)fastdiv((uint32_t)tap, p.tap.div_nx), tx = tap - ty * p.tap.nx;
                    c = chunk - tap * p.tap.chunks;
                    dy = p.tap.dy0 + ty * p.tap.dys;
                    dx = p.tap.dx0 + tx * p.tap.dxs;
                }
            };
            inside[u] = 0;
            valid[u] = 16;
            if constexpr (FORM == INPUT_PLANAR) {
                // product t's chunk of this lane's own pixel, byte by byte
#pragma unroll
                for (int t = 0; t < STEPS; ++t) {
                    const int chunk = (g * 2 + half) * STEPS + t;
                    int dy, dx, c;
                    place(chunk, dy, dx, c);
                    exists[u] = chunk * 16 < p.k;
                    bool ok = exists[u];
                    if constexpr (TAPS) ok = ok && (unsigned)(iy0 + dy) < (unsigned)p.h && (unsigned)(ix0 + dx) < (unsigned)p.w;
                    const int here = c == p.tap.chunks - 1 ? p.c_last : 16;
                    const uint32_t plane = (uint32_t)(p.h * p.w);
                    uint32_t at = ok ? (uint32_t)(base + dy * p.w + dx) + (uint32_t)(c * 16) * plane : 0u;
                    u16x2 b[8];  // (two to a register)
#pragma unroll
                    for (int j = 0; j < 16; ++j) {
                        b[j >> 1][j & 1] = p.a[at];
                        at += ok && j + 1 < here ? plane : 0u;
                    }
                    // (taps outside the image and bytes behind the tap's channels: the input zero point; past the reduction: zero after the flip)
                    const uint32_t other = exists[u] ? p.fill : p.a_xor;
#pragma unroll
                    for (int d = 0; d < 4; ++d) {
                        const uint32_t mask = ok ? byte_mask(here, d) : 0u;
                        const uint32_t w = __builtin_amdgcn_perm(__builtin_bit_cast(uint32_t, b[2 * d + 1]), __builtin_bit_cast(uint32_t, b[2 * d]), 0x06040200u);
                        af[u][t][d] = (int)(((w & mask) | (other & ~mask)) ^ p.a_xor);
                    }
                }
            } else {
                // the chunk this lane fetches for each of the four pixels
                const int chunk = g * 8 + half * 4 + (lane & 3);
                exists[u] = chunk * 16 < p.k;
                int dy, dx, c;
                place(chunk, dy, dx, c);
                int off = chunk * 16;
                if constexpr (TAPS) off = (dy * p.w + dx) * p.cin + c * 16;
                if constexpr (FORM == INPUT_RAGGED) valid[u] = c == p.tap.chunks - 1 ? p.c_last : 16;
                auto fetch = [&](auto px_c, int b, int iy, int ix) {
                    constexpr int px = decltype(px_c)::value;
                    bool ok = exists[u];
                    if constexpr (TAPS) ok = ok && (unsigned)(iy + dy) < (unsigned)p.h && (unsigned)(ix + dx) < (unsigned)p.w;
                    inside[u] |= (uint32_t)ok << px;
                    if constexpr (FORM == INPUT_RAGGED) {
                        const uint32_t at = ok ? (uint32_t)(b + off) : 0u, from = at < last_start ? at : last_start;
                        inside[u] |= (at - from) << (8 + 4 * px);
                        af[u][px] = *reinterpret_cast<const v4i_any_alignment *>(p.a + from);
                    } else {
                        af[u][px] = *reinterpret_cast<const v4i *>(p.a + (size_t)(ok ? b + off : 0));
                    }
                };
                fetch(std::integral_constant<int, 0>{}, q_base.x, q_iy.x, q_ix.x);
                fetch(std::integral_constant<int, 1>{}, q_base.y, q_iy.y, q_ix.y);
                fetch(std::integral_constant<int, 2>{}, q_base.z, q_iy.z, q_ix.z);
                fetch(std::integral_constant<int, 3>{}, q_base.w, q_iy.w, q_ix.w);
            }
#pragma unroll
            for (int t = 0; t < STEPS; ++t) {
                const int wc = (g * 2 + half) * STEPS + t;
                bf[u][t] = wsrc[(size_t)(wc < chunks ? wc : chunks - 1) * 32];  // (past the packed rows: multiplied by zeros)
            }
        }
        request_finish();
#pragma unroll
        for (int u = 0; u < GROUPS; ++u) {
            if (g0 + u * kWaves >= groups) break;
            if constexpr (FORM == INPUT_PLANAR) {
                if constexpr (ROWSUM) {
#pragma unroll
                    for (int t = 0; t < STEPS; ++t)
#pragma unroll
                        for (int d = 0; d < 4; ++d) rowsum[0] = __builtin_amdgcn_sdot4(af[u][t][d], 0x01010101, rowsum[0], false);
                }
            } else {
                // taps outside the image read the input zero point; bytes past the reduction the one the flip turns into 0
                const int other = (int)(exists[u] ? p.fill ^ p.a_xor : 0u), flip = (int)p.a_xor;
                if constexpr (FORM == INPUT_RAGGED) {
                    if (__builtin_amdgcn_ballot_w64(inside[u] >> 8 != 0)) {  // (only where the wave reads the tensor's last bytes)
#pragma unroll
                        for (int px = 0; px < 4; ++px) af[u][px] = shift_bytes_down(af[u][px], (inside[u] >> (8 + 4 * px)) & 15u);
                    }
                }
                uint32_t mask[4];
#pragma unroll
                for (int d = 0; d < 4; ++d) mask[d] = FORM == INPUT_RAGGED ? byte_mask(valid[u], d) : ~0u;
#pragma unroll
                for (int px = 0; px < 4; ++px) {
                    const bool ok = (inside[u] >> px) & 1u;
#pragma unroll
                    for (int d = 0; d < 4; ++d) {
                        const uint32_t v = (uint32_t)(af[u][px][d] ^ flip);
                        af[u][px][d] = ok ? (int)(FORM == INPUT_RAGGED ? (v & mask[d]) | ((uint32_t)other & ~mask[d]) : v) : other;
                    }
                }
                if constexpr (ROWSUM) {
                    // (summed before the exchange: of pixel px by the lane that fetched it)
#pragma unroll
                    for (int px = 0; px < 4; ++px) {
                        rowsum[px] = __builtin_amdgcn_sdot4(af[u][px].x, 0x01010101, rowsum[px], false);
                        rowsum[px] = __builtin_amdgcn_sdot4(af[u][px].y, 0x01010101, rowsum[px], false);
                        rowsum[px] = __builtin_amdgcn_sdot4(af[u][px].z, 0x01010101, rowsum[px], false);
                        rowsum[px] = __builtin_amdgcn_sdot4(af[u][px].w, 0x01010101, rowsum[px], false);
                    }
                }
#pragma unroll
                for (int d = 0; d < 4; ++d) {
                    int c0 = af[u][0][d], c1 = af[u][1][d], c2 = af[u][2][d], c3 = af[u][3][d];
                    quad_transpose(c0, c1, c2, c3, odd, high);
                    af[u][0][d] = c0, af[u][1][d] = c1, af[u][2][d] = c2, af[u][3][d] = c3;
                }
            }
#pragma unroll
            for (int t = 0; t < STEPS; ++t) acc = __builtin_amdgcn_mfma_i32_32x32x32_i8(bf[u][t], af[u][t], acc, 0, 0, 0);
        }
    }
    request_finish();  // (a wave without a step of its own)
    // ---- the partial tiles meet in LDS
    int32_t *mine = part_s[wave] + lane * kLanePitch;
#pragma unroll
    for (int g = 0; g < 4; ++g) *reinterpret_cast<int4 *>(mine + g * 4) = make_int4(acc[g * 4], acc[g * 4 + 1], acc[g * 4 + 2], acc[g * 4 + 3]);
    if constexpr (ROWSUM) {
        if constexpr (FORM != INPUT_PLANAR) quad_transpose(rowsum[0], rowsum[1], rowsum[2], rowsum[3], odd, high);  // now four lanes' shares of this lane's own pixel
        sum_s[wave * 2 + half][r] = rowsum[0] + rowsum[1] + rowsum[2] + rowsum[3];
    }
    __syncthreads();
    const int src = ((f_pair >> 3) * 32 + f_px) * kLanePitch + ((f_pair * 2) & 15);
    int x0 = f_bias.x, x1 = f_bias.y;
#pragma unroll
    for (int w = 0; w < kWaves; ++w) {
        const int2 v = *reinterpret_cast<const int2 *>(part_s[w] + src);
        x0 += v.x;
        x1 += v.y;
    }
    if constexpr (ROWSUM) {
        int rs = 0;
#pragma unroll
        for (int w = 0; w < kWaves * 2; ++w) rs += sum_s[w][f_px];
        x0 -= p.zw * rs;
        x1 -= p.zw * rs;
    }
    const RequantDev rq = p.rq;
    uint32_t o0, o1;
    auto produce = [&](auto mode_c) {
        constexpr int mode = decltype(mode_c)::value;
        if (rq.pc_multiplier) {
            if constexpr (mode == 0) {
                o0 = requant_u8_channel(x0, f_mult.x, f_shift.x, rq);
                o1 = requant_u8_channel(x1, f_mult.y, f_shift.y, rq);
            } else {
                o0 = requant_u8_channel_fast<mode>(x0, f_mult.x, f_shift.x, rq);
                o1 = requant_u8_channel_fast<mode>(x1, f_mult.y, f_shift.y, rq);
            }
        } else {
            o0 = requant_u8_as<mode>(x0, rq);
            o1 = requant_u8_as<mode>(x1, rq);
        }
    };
    if (!FAST || (FORM != INPUT_CHUNKS && rq.fast == 0))
        produce(std::integral_constant<int, 0>{});
    else if (rq.fast == 2)
        produce(std::integral_constant<int, 2>{});
    else
        produce(std::integral_constant<int, 1>{});
    o0 ^= p.out_xor & 0xFFu;
    o1 ^= p.out_xor & 0xFFu;
    if (p.residual) {
        o0 = add_one(f_res0, o0, p.radd);
        o1 = add_one(f_res1, o1, p.radd);
    }
    const uint32_t two = o0 | (o1 << 8);
    const uint32_t other = (uint32_t)__shfl_xor((int)two, 1);  // the neighbour's two channels
    if (f_m >= p.m || f_n >= p.n) return;
    uint8_t *dst = p.out + f_off;
    if (f_n + 1 < p.n && ((f_n | 3) < p.n) && (p.ldc & 3) == 0 && (reinterpret_cast<uintptr_t>(p.out) & 3) == 0) {
        if ((f_pair & 1) == 0) *reinterpret_cast<uint32_t *>(dst) = two | (other << 16);
    } else if (!p.residual && p.planar.out_plane) {
        const uint32_t packed[4] = {two, 0, 0, 0};
        store_bytes_planar(p.out, p.planar, f_off - (size_t)f_n, f_n, packed, p.n - f_n < 2 ? 1 : 2);
    } else {
        dst[0] = (uint8_t)o0;
        if (f_n + 1 < p.n) dst[1] = (uint8_t)o1;
    }
}

}  // namespace

static long few_tiles_count(int64_t m, int64_t n) { return (long)(((m + 31) / 32) * ((n + 31) / 32)); }

// Activations in whole 16-byte chunks of one tap each, and at most two rounds of 32 x 32 tiles.  Against the direct-to-LDS
// tiles, in us: 3x3 on 256 channels at 14 x 14, images 1 / 4 / 8 (56 / 200 / 392 tiles) 9.3 / 9.1 / 9.1 -> 5.3 / 5.4 / 8.9; on
// 512 channels at 7 x 7, 1 / 16 images (32 / 400 tiles) 13.1 / 13.4 -> 7.1 / 12.5; fully connected 100 x 4096 x 1000 (128
// tiles) 9.8 -> 6.6, 1364 x 640 x 192 (258) 5.8 -> 4.8, 64 x 4096 x 4096 (256) 10.4 -> 7.4; deconvolution 4x4 stride 2
// 256 -> 128 at 16 x 16, one image (128 in four phases) 7.3 -> 5.0.  Beyond 8 KiB, where a wave's loads no longer travel together,
// the tiles win or lose by their number: 3x3 on 1024 channels at 7 x 7, one image (64 tiles, 9 KiB) 14.3 -> 11.1, fully connected
// 100 x 9216 x 1000 (128) 15.0 -> 10.0, but 128 x 16384 x 4096 (512) 24.7 -> 31.7, 200 x 65536 x 256 (56) 37.3 -> 49.9 and 3x3 on
// 1024 at 14 x 14, eight images (392, 9 KiB) 21.1 -> 21.0; such plans keep the tiles.
bool gemm_few_tiles_applies(int64_t m, int64_t n, int64_t k, int32_t siblings) {
    return m > 0 && few_tiles_count(m, n) * siblings <= 512 && k <= 8192;
}

// The one-tap, few-row and 3x3 patch kernels keep their weights in the same order, so that the choice can be made at the
// launch.  Up to one round of tiles this kernel is the faster one: 3x3 on 128 channels at 28 x 28, one image (100 tiles)
// 6.1 -> 4.6, on 64 at 28 x 28, four images (196) 4.7 -> 4.1, but eight (392) 4.7 -> 4.9; one tap 256 -> 64 at 14 x 14, eight
// images (98) 5.6 -> 4.0, 96 -> 576 (882) 4.3 -> 6.3; fully connected 64 x 1280 x 1000 7.3 -> 4.6, 64 x 3456 x 184 11.2 -> 6.0.
// The few-row kernel fetches a row's activations once per lane and step, which costs by the row, this one 32 rows' whether they
// exist or not.  Few rows -> here, us at 1000 channels: 32 x 4096 7.3 -> 6.4, 17 x 4096 6.1 -> 6.4, 16 x 4096 6.0 -> 6.3, 16 x 8192
// 9.1 -> 9.1, 16 x 9216 10.5 -> 9.6, 12 x 9216 9.7 -> 9.7, 10 x 9216 9.2 -> 9.6, 1 x 9216 8.5 -> 9.6; 12 x 25088 20.9 -> 20.7,
// 10 x 25088 19.9 -> 20.7, 1 x 25088 17.6 -> 20.7; 12 x 65536 50.3 -> 48.3, 10 x 65536 46.7 -> 48.0.
bool gemm_few_tiles_instead(const GemmProblem &p) {
    if (p.vec != 16 || (reinterpret_cast<uintptr_t>(p.a) & 15) != 0 || few_tiles_count(p.m, p.n) > 256) return false;
    if (p.cfg.id == GEMM_SKINNY) return p.m > 16 || (p.m > 10 && p.k > 8192);
    return p.cfg.id == GEMM_THIN || p.cfg.id == GEMM_CONV3X3;
}

// Against the copy and the kernel that reads it.  Drawn layers (some 1700, on both sides of every line; a replayed graph, where a second
// launch is cheapest), the time of reading directly over that of the copy; k: a tap's reduction with its padding, times the taps:
//   ragged  up to one round of tiles  k to 2500 0.60 .. 1.03; 2700 .. 3500 0.79 .. 1.06; beyond 0.86 .. 1.13, as four lanes' pieces of a pixel
//                                     meet more cache lines than whole chunks do.  Rows few enough for the few-row kernel: k 2000 .. 2560 0.73 .. 1.07,
//                                     2600 .. 3000 0.82 .. 1.14, 3500 .. 3650 1.05 .. 1.23
//           up to two                 k 400 .. 1024 0.66 .. 0.84; 1150 .. 1570 0.88 .. 1.33; one tap 600 .. 2208 0.39 .. 0.91
//           up to four                one tap, k 190 .. 240 0.69 .. 0.79; 144 1.08; 3x3 288 1.06, 864 1.12
//   planar  up to one                 k to 576 0.50 .. 0.97; 720 .. 1000 0.80 .. 1.28 (most of 7x7 on 16 channels 1.01 .. 1.18); 1100 .. 1600 1.04 .. 1.70,
//                                     4000 2.0 .. 2.8: sixteen loads to a chunk.  One tap 0.51 .. 1.01 to 1072
//           up to two                 k 288 0.70 .. 0.94; 400 0.84 .. 1.19, 0.97 on average; 432 0.76 .. 1.07; 576 0.82 .. 1.20; 640 .. 860 0.90 .. 1.35.  One tap
//                                     0.33 .. 0.96 to 576
//           800 tiles                 k 48 .. 160 0.57 .. 0.84; 288 .. 1150 1.10 .. 1.31; 800 tiles, 160 7.8 -> 8.1 us
// (planar 1x1 layers of one product keep to two rounds: 980 tiles 6.5 .. 7.6 us either way)
bool gemm_few_tiles_direct(int64_t m, int64_t n, int64_t k, int32_t taps, int32_t problems, int32_t form) {
    const long tiles = m > 0 ? few_tiles_count(m, n) * problems : 0;
    if (tiles <= 0) return false;
    const bool one_tap = taps == 1;
    if (form == INPUT_RAGGED) {
        if (tiles <= 256) return k <= (one_tap && m <= 16 ? 2560 : 3500);
        if (tiles <= 512) return k <= (one_tap ? 2208 : 1024);
        return tiles <= 1024 && one_tap && k > 144 && k <= 256;
    }
    if (tiles <= 256) return k <= (one_tap ? 1152 : 576);
    return tiles <= 512 ? k <= (one_tap ? 576 : 432) : tiles < 800 && k > 32 && k <= 256;
}

int launch_gemm_few_tiles(const TapProblem *ps, int count, hipStream_t stream) {
    const TapProblem &p = ps[0];
    EH_REQUIRE(count >= 1 && count <= GemmBatch::MAX, "few_tiles: batch of %d", count);
    int m_max = p.m;
    for (int i = 0; i < count; ++i) {
        EH_REQUIRE(ps[i].k_pad == p.k_pad && ps[i].n == p.n && ps[i].zw == p.zw && ps[i].rq.fast == p.rq.fast && ps[i].vec == 16 &&
                       (ps[i].k & 15) == 0 && (ps[i].k_pad & 31) == 0 && ps[i].k_pad >= ps[i].k && ps[i].k > 0 && ps[i].k % (ps[i].tap.chunks * 16) == 0 &&
                       ps[i].form == p.form && ps[i].c_last == p.c_last && ps[i].c_last >= 1 && ps[i].c_last <= 16,
                   "few_tiles: unsupported problem");
        if (p.form != INPUT_CHUNKS)
            EH_REQUIRE((int64_t)(ps[i].m / (ps[i].ho * ps[i].wo)) * ps[i].h * ps[i].w * ps[i].cin >= 16 && ps[i].tap.c0 + (ps[i].tap.chunks - 1) * 16 + ps[i].c_last <= ps[i].cin,
                       "few_tiles: channels %d .. of %d", ps[i].tap.c0, ps[i].cin);
        else
            EH_REQUIRE((reinterpret_cast<uintptr_t>(ps[i].a) & 15) == 0 && (ps[i].cin & 15) == 0 && (ps[i].tap.c0 & 15) == 0, "few_tiles: unaligned activations");
        m_max = ps[i].m > m_max ? ps[i].m : m_max;
    }
    const int m_blocks = (m_max + 31) / 32, n_blocks = (p.n + 31) / 32;
    const long tiles = (long)m_blocks * n_blocks;
    EH_REQUIRE(tiles > 0 && tiles < (1l << 28), "few_tiles: %ld tiles", tiles);
    const int per_xcd = (int)((tiles + 7) / 8);
    const int m_fastest = (long)p.n * p.k >= (long)p.m * p.cin ? 1 : 0;  // the larger operand's blocks run slowest
    const dim3 grid((unsigned)(per_xcd * 8), 1, (unsigned)count), block(kWaves * 64);
    const int groups = ((p.k_pad + (p.form == INPUT_PLANAR ? 31 : 127)) / (p.form == INPUT_PLANAR ? 32 : 128) + kWaves - 1) / kWaves;  // of the longest-working wave
    // one tap at the pixel itself, on an image it cannot leave
    bool inside = true;
    for (int i = 0; i < count; ++i)
        inside = inside && ps[i].tap.chunks * 16 == ps[i].k && ps[i].tap.dy0 == 0 && ps[i].tap.dx0 == 0 && ps[i].y_base == 0 && ps[i].x_base == 0 &&
                 (ps[i].ho - 1) * ps[i].stride_h < ps[i].h && (ps[i].wo - 1) * ps[i].stride_w < ps[i].w;
    FewBatch batch;
    if (count > 1)
        for (int i = 0; i < count; ++i) batch.p[i] = ps[i];
    auto launch = [&](auto groups_c, auto taps_c, auto rowsum_c, auto fast_c, auto form_c) {
        constexpr int S = decltype(groups_c)::value, I = decltype(form_c)::value;
        constexpr bool T = decltype(taps_c)::value, R = decltype(rowsum_c)::value, F = decltype(fast_c)::value;
        if (count > 1)
            hipLaunchKernelGGL((few_tiles_kernel<S, T, R, F, true, I>), grid, block, 0, stream, batch, m_blocks, n_blocks, per_xcd, m_fastest);
        else
            hipLaunchKernelGGL((few_tiles_kernel<S, T, R, F, false, I>), grid, block, 0, stream, FewProblem(p), m_blocks, n_blocks, per_xcd, m_fastest);
    };
    auto with_fast = [&](auto groups_c, auto taps_c, auto rowsum_c) {
        if (p.form == INPUT_RAGGED)
            launch(groups_c, taps_c, rowsum_c, std::true_type{}, std::integral_constant<int, INPUT_RAGGED>{});
        else if (p.form == INPUT_PLANAR)
            launch(groups_c, taps_c, rowsum_c, std::true_type{}, std::integral_constant<int, INPUT_PLANAR>{});
        else if (p.rq.fast != 0)
            launch(groups_c, taps_c, rowsum_c, std::true_type{}, std::integral_constant<int, INPUT_CHUNKS>{});
        else
            launch(groups_c, taps_c, rowsum_c, std::false_type{}, std::integral_constant<int, INPUT_CHUNKS>{});
    };
    auto with_rowsum = [&](auto groups_c, auto taps_c) {
        if (p.zw != 0)
            with_fast(groups_c, taps_c, std::true_type{});
        else
            with_fast(groups_c, taps_c, std::false_type{});
    };
    auto with_taps = [&](auto groups_c) {
        if (inside)
            with_rowsum(groups_c, std::false_type{});
        else
            with_rowsum(groups_c, std::true_type{});
    };
    if (groups <= 1)
        with_taps(std::integral_constant<int, 1>{});
    else if (groups <= 2)
        with_taps(std::integral_constant<int, 2>{});
    else
        with_taps(std::integral_constant<int, 3>{});
    EH_HIP(hipGetLastError());
    return EH_OK;
}

}  // namespace eh
