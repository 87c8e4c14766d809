// conv_pws.hip -- large pointwise convolutions (1x1, stride 1, no padding) on
// int8 MFMA (kernels/conv/kernel/ConvKernel.cpp:171-249).
//
// y[n][m][p] = sat16(wrap32([bias[m] << 8] + sum_c w[m][c] * x[n][c][p]) >> 8),
// then the optional fused Add / Relu / Relu6 epilogue.
//
// These layers move x, y and the residual and do little arithmetic per byte, so
// the kernel is built around its memory accesses: every one of them is 16 bytes
// of eight consecutive pixels.  A block owns eight or sixteen groups of
// eight pixels (groups running across images) and a range of output channels.
//   * x: a thread loads four channels of one group and turns the 4 x 8 int16
//     values into limb bytes, channels minor, with v_perm (a 4 x 4 byte
//     transpose per two pixels); the tile's limb planes of every channel sit in
//     LDS in the order that MFMA fragments are read, 16 bytes a lane.
//   * The pixels are the MFMA's rows and the output channels its columns: row r
//     of row tile t is pixel t of the group 4 (r % 4) + r / 4 (sixteen groups,
//     eight row tiles), or pixel 4 (r % 2) + t of the group 4 (r % 4 / 2) + r / 4
//     (eight groups, four tiles), so that a lane's results are runs of eight
//     pixels of one channel -- one 16-byte store, four neighbouring lanes 64
//     bytes -- with no trip through LDS.  The fused Add's operand is loaded the same way, ahead of
//     the products.
//   * w: a wave takes every W-th 16-channel column tile and loads its fragments
//     (16 k of a channel's row) from L2 one k step ahead.
// Planes whose pixel count is not a multiple of 8: an image's last group is read
// eight pixels before the plane's end and stores only the pixels its neighbour
// does not have.
//
// Measured against the block-tiled GEMM it replaces (which split the limbs of both
// operands into LDS and carried its sums through LDS as well): 64 -> 256 with a
// residual at 32 x 56 x 56 68 -> 26 us (116 MB: 4.4 TB/s), 256 -> 64 39 -> 19, 128 ->
// 512 at 28 x 28 42 -> 21, 215 -> 146 at 17 x 63 x 63 127 -> 52.  Blocks of 128
// pixels and four waves: 29 us on the first; stores through the cache 36.
//
// Limbs and the exact sum are the GEMM kernel's (gemm.hip): v = 256 vh + vl + 128,
//     sum a*b = 65536 S_hh + 256 S_mid + S_ll + 128 (sum a + sum b) - 16384 Kp
// over Kp = 64 * steps positions, every term mod 2^32, the accumulator's wrap.
#include "cm_internal.h"
#include "limbs.h"
#include "q88.h"

#include <algorithm>

namespace {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef short v2s __attribute__((ext_vector_type(2)));
typedef unsigned int v2u __attribute__((ext_vector_type(2)));
typedef unsigned int v4u __attribute__((ext_vector_type(4)));

constexpr uint32_t kMaxC = 512;                 // 8 k steps: 128 KB of LDS
constexpr uint64_t kStreamBytes = 80ull << 20;
constexpr int kNonTemporal = 2;                 // buffer access cache policy bit

struct PwsArgs {
    const int16_t* x;
    const int16_t* w;
    const int16_t* bias;
    int16_t* y;
    EpiArgs epi;
    uint32_t C, M, P;
    uint32_t nk;                 // k steps of 64
    uint32_t gpi, n_groups;      // pixel groups per image; in all
    uint32_t ct_per_block, n_ct; // 16-channel tiles per block; in all
    uint32_t x_bytes, w_bytes, y_bytes, b_bytes;   // whole tensors, below 2^31
    FastDiv div_gpi;
};

using limbs::bsum;

__device__ __forceinline__ uint32_t perm(uint32_t hi, uint32_t lo, uint32_t sel) {
    return __builtin_amdgcn_perm(hi, lo, sel);
}

// Eight pixels at byte offset `off` of which the last n are stored: one access
// for all eight, else 1 + 2 + 4 elements from the end.
template <int AUX>
__device__ __forceinline__ void store_tail(__amdgpu_buffer_rsrc_t rs, uint32_t off, uint32_t n, const uint32_t (&d)[4]) {
    if (n == 8u) {
        __builtin_amdgcn_raw_buffer_store_b128(v4u{d[0], d[1], d[2], d[3]}, rs, off, 0, AUX);
        return;
    }
    // the window moves down as pieces are taken off its end
    uint32_t w0 = d[0], w1 = d[1], w2 = d[2], w3 = d[3], end = off + 16u;
    if (n & 1u) {
        end -= 2u;
        __builtin_amdgcn_raw_buffer_store_b16((uint16_t)(w3 >> 16), rs, end, 0, 0);
        w3 = __builtin_amdgcn_alignbit(w3, w2, 16);
        w2 = __builtin_amdgcn_alignbit(w2, w1, 16);
        w1 = __builtin_amdgcn_alignbit(w1, w0, 16);
    }
    if (n & 2u) {
        end -= 4u;
        __builtin_amdgcn_raw_buffer_store_b32(w3, rs, end, 0, 0);
        w3 = w2;
        w2 = w1;
    }
    if (n & 4u) __builtin_amdgcn_raw_buffer_store_b64(v2u{w2, w3}, rs, end - 8u, 0, 0);
}

// G: pixel groups per block (8 or 16: 4 or 8 row tiles); W: waves.  AV: in_ch is
// a multiple of 8; NT: y is stored past the cache.
template <uint32_t G, uint32_t W, bool AV, bool NT>
__global__ __launch_bounds__(W * 64, G == 8 ? 4 : 2) void conv_pws(PwsArgs g) {
    constexpr uint32_t kPix = G * 8, kWaves = W;
    constexpr uint32_t RT = G / 2;                   // row tiles of 16 pixels
    constexpr uint32_t kStepBytes = kPix * 64 * 2;   // limb planes of one k step (64 channels)
    constexpr uint32_t SP = W * 4 / G;               // k steps staged by one pass of the block
    extern __shared__ __align__(16) uint8_t lds[];   // [k step][row tile][hi, lo][lane][16]
    __shared__ uint32_t part[4 * SP][kPix];          // channel sums of the pixels, per 16-channel group
    __shared__ uint32_t xsum[kPix];
    touch_lines(g);
    const uint32_t tid = threadIdx.x, lane = tid & 63u;
    const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(tid >> 6));
    const __amdgpu_buffer_rsrc_t xr = make_rsrc(g.x, g.x_bytes), wr = make_rsrc(g.w, g.w_bytes);
    const __amdgpu_buffer_rsrc_t yr = make_rsrc(g.y, g.y_bytes), br = make_rsrc(g.bias, g.b_bytes);
    const __amdgpu_buffer_rsrc_t ar = make_rsrc(g.epi.add, g.epi.add_mode == 1u ? g.y_bytes : 0u);
    const uint32_t r16 = lane & 15u, kg = lane >> 4;

    // ---- weights of (column tile ct, k step s): 16 k of this lane's channel
    const uint32_t ct_lo = blockIdx.y * g.ct_per_block;
    const uint32_t ct_hi = min(ct_lo + g.ct_per_block, g.n_ct);
    struct Raw { uint32_t w[8]; };
    auto load_w = [&](uint32_t ct, uint32_t s) {
        Raw r;
        const uint32_t m = ct * 16u + r16, k = s * 64u + kg * 16u;
        const uint32_t row = m < g.M && ct < ct_hi ? m * g.C * 2u : kOob;
#pragma unroll
        for (int q = 0; q < 2; ++q) {
            // a row's last vector is read eight values before its end and shifted down
            const uint32_t kk = k + q * 8u, kb = min(kk, g.C - 8u), sh = kk - kb;
            v4u v = __builtin_amdgcn_raw_buffer_load_b128(wr, (row + kb * 2u) | (uint32_t)(kk >= g.C) << 31, 0, 0);
            if (!AV && s + 1 == g.nk) {
                v = sh & 4u ? v4u{v[2], v[3], 0u, 0u} : v;
                v = sh & 2u ? v4u{v[1], v[2], v[3], 0u} : v;
                const uint32_t h = (sh & 1u) * 16u;
                v = v4u{__builtin_amdgcn_alignbit(v[1], v[0], h), __builtin_amdgcn_alignbit(v[2], v[1], h),
                        __builtin_amdgcn_alignbit(v[3], v[2], h), v[3] >> h};
            }
            r.w[4 * q] = v[0]; r.w[4 * q + 1] = v[1]; r.w[4 * q + 2] = v[2]; r.w[4 * q + 3] = v[3];
        }
        return r;
    };
    uint32_t ct = ct_lo + wave;
    Raw next = load_w(ct, 0);

    // ---- x tile: this thread's four channels (4 c4 .. of the wave's 16) of one group
    {
        const uint32_t c4 = tid & 3u, grp = (tid >> 2) % G;
        const uint32_t kq = (tid / (4u * G)) & 3u, sp = tid / (16u * G);
        const uint32_t gi = blockIdx.x * G + grp;
        const uint32_t n = fdiv(gi < g.n_groups ? gi : 0u, g.div_gpi), pg = gi - n * g.gpi;
        const uint32_t px = min(pg * 8u, g.P - 8u);
        const uint32_t base = gi < g.n_groups ? (n * g.C * g.P + px) * 2u : kOob;
        int32_t hs[8], ls[8];
#pragma unroll
        for (int t = 0; t < 8; ++t) hs[t] = ls[t] = 0;
        auto load_x = [&](uint32_t s, v4u (&d)[4]) {
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const uint32_t c = (s + sp) * 64u + kq * 16u + c4 * 4u + i;
                d[i] = __builtin_amdgcn_raw_buffer_load_b128(xr, c < g.C ? base + c * g.P * 2u : kOob, 0, 0);
            }
        };
        auto put = [&](uint32_t s, const v4u (&d)[4]) {
            // byte c4 * 4 of the fragment slot (k group, row) of each row tile
            if (SP > 1 && s + sp >= g.nk) return;
            const uint32_t row0 = G == 16 ? 4u * (grp & 3u) + (grp >> 2) : 4u * (grp & 3u) + 2u * (grp >> 2);
            uint8_t* to = lds + (s + sp) * kStepBytes + (kq * 16u + row0) * 16u + c4 * 4u;
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const uint32_t ab0 = perm(d[1][q], d[0][q], 0x06020400u), cd0 = perm(d[3][q], d[2][q], 0x06020400u);
                const uint32_t ab1 = perm(d[1][q], d[0][q], 0x07030501u), cd1 = perm(d[3][q], d[2][q], 0x07030501u);
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    const uint32_t sel = h ? 0x07060302u : 0x05040100u;
                    const uint32_t lo = perm(cd0, ab0, sel) ^ 0x80808080u, hi = perm(cd1, ab1, sel);
                    const int t = 2 * q + h;
                    hs[t] = bsum(hi, hs[t]);
                    ls[t] = bsum(lo, ls[t]);
                    // G = 8: pixels 4 .. 7 of a group are the next row of tiles 0 .. 3
                    uint8_t* at = to + (t % RT) * 2048 + (t / RT) * 16;
                    *reinterpret_cast<uint32_t*>(at) = hi;
                    *reinterpret_cast<uint32_t*>(at + 1024) = lo;
                }
            }
        };
        v4u d0[4], d1[4];
        load_x(0, d0);
        for (uint32_t s = 0; s < g.nk; s += 2 * SP) {
            load_x(s + SP, d1);
            put(s, d0);
            if (s + SP >= g.nk) break;
            load_x(s + 2 * SP, d0);
            put(s + SP, d1);
        }
        const uint32_t mine = (g.nk + SP - 1 - sp) / SP;   // steps this thread staged
        // sums over the k group's channels: the four lanes of a row
#pragma unroll
        for (int t = 0; t < 8; ++t) {
            uint32_t v = 256u * (uint32_t)hs[t] + (uint32_t)ls[t] + 128u * 4u * mine;
            v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0xB1, 0xF, 0xF, true);   // quad: lane ^ 1
            v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x4E, 0xF, 0xF, true);   // quad: lane ^ 2
            if (c4 == 0u) part[sp * 4u + kq][grp * 8u + t] = v;
        }
    }
    __syncthreads();
    if (tid < kPix) {
        uint32_t v = 0;
#pragma unroll
        for (uint32_t q = 0; q < 4 * SP; ++q) v += part[q][tid];
        xsum[tid] = 128u * v;
    }
    __syncthreads();

    // ---- this lane's output groups (e: group 4 e + kg), channel r16 of the tile
    constexpr int E = G / 4;
    uint32_t yoff[E], yn[E];
#pragma unroll
    for (int e = 0; e < E; ++e) {
        const uint32_t gi = blockIdx.x * G + 4u * e + kg;
        const uint32_t n = fdiv(gi < g.n_groups ? gi : 0u, g.div_gpi), pg = gi - n * g.gpi;
        const uint32_t px = min(pg * 8u, g.P - 8u);
        yoff[e] = gi < g.n_groups ? (n * g.M * g.P + px) * 2u : kOob;
        yn[e] = min(8u, g.P - pg * 8u);
    }
    const v2s lo2 = {(short)q88::act_lo(g.epi.act), (short)q88::act_lo(g.epi.act)};
    const v2s hi2 = {(short)q88::act_hi(g.epi.act), (short)q88::act_hi(g.epi.act)};
    const uint32_t kp_term = 16384u * 64u * g.nk;

    for (; ct < ct_hi; ct += kWaves) {
        const uint32_t m = ct * 16u + r16;
        const uint32_t mo = m < g.M ? m * g.P * 2u : kOob;   // yoff + mo: bit 31 when either is out
        const uint32_t b8 = q88::data_to_acc((int16_t)__builtin_amdgcn_raw_buffer_load_b16(br, m * 2u, 0, 0));
        v4u add[E];
        if (g.epi.add_mode == 1u) {
#pragma unroll
            for (int e = 0; e < E; ++e) {
                const uint32_t off = (yoff[e] | mo) >> 31 ? kOob : yoff[e] + mo;
                add[e] = __builtin_amdgcn_raw_buffer_load_b128(ar, off, 0, 0);
            }
        }
        v4i hh[RT], mid[RT], ll[RT];
#pragma unroll
        for (uint32_t t = 0; t < RT; ++t) hh[t] = mid[t] = ll[t] = v4i{0, 0, 0, 0};
        int32_t ws = 0;
        for (uint32_t s = 0; s < g.nk; ++s) {
            const Raw raw = next;
            next = s + 1 < g.nk ? load_w(ct, s + 1) : load_w(ct + kWaves, 0);
            v4i bh, bl;
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const uint32_t w0 = raw.w[2 * q], w1 = raw.w[2 * q + 1];
                bh[q] = (int)limbs::hi4(w0, w1);
                bl[q] = (int)limbs::lo4(w0, w1);
                ws = __builtin_amdgcn_sdot2(__builtin_bit_cast(v2s, w0), v2s{1, 1}, ws, false);
                ws = __builtin_amdgcn_sdot2(__builtin_bit_cast(v2s, w1), v2s{1, 1}, ws, false);
            }
            const uint8_t* f = lds + s * kStepBytes + lane * 16u;
#pragma unroll
            for (uint32_t t = 0; t < RT; ++t) {
                const v4i ah = *reinterpret_cast<const v4i*>(f + t * 2048);
                const v4i al = *reinterpret_cast<const v4i*>(f + t * 2048 + 1024);
                hh[t] = __builtin_amdgcn_mfma_i32_16x16x64_i8(ah, bh, hh[t], 0, 0, 0);
                mid[t] = __builtin_amdgcn_mfma_i32_16x16x64_i8(ah, bl, mid[t], 0, 0, 0);
                mid[t] = __builtin_amdgcn_mfma_i32_16x16x64_i8(al, bh, mid[t], 0, 0, 0);
                ll[t] = __builtin_amdgcn_mfma_i32_16x16x64_i8(al, bl, ll[t], 0, 0, 0);
            }
        }
        uint32_t wsum = (uint32_t)ws;   // over the four k groups of the channel
        wsum += (uint32_t)__shfl_xor((int)wsum, 16, 64);
        wsum += (uint32_t)__shfl_xor((int)wsum, 32, 64);
        const uint32_t cterm = 128u * wsum - kp_term + b8;
#pragma unroll
        for (int e = 0; e < E; ++e) {
            const uint32_t* xs = xsum + (4u * e + kg) * 8u;
            const v4u x0 = *reinterpret_cast<const v4u*>(xs), x1 = *reinterpret_cast<const v4u*>(xs + 4);
            int32_t v[8];
#pragma unroll
            for (int t = 0; t < 8; ++t) {
                const int tt = t % (int)RT, ee = G == 16 ? e : 2 * e + t / (int)RT;
                const uint32_t s = ((((uint32_t)hh[tt][ee] << 8) + (uint32_t)mid[tt][ee]) << 8) + (uint32_t)ll[tt][ee];
                v[t] = (int32_t)(s + cterm + (t < 4 ? x0[t & 3] : x1[t & 3])) >> 8;
            }
            uint32_t out[4];
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                v2s o = __builtin_bit_cast(v2s, __builtin_amdgcn_cvt_pk_i16(v[2 * q], v[2 * q + 1]));
                if (g.epi.add_mode == 1u) {
                    const uint32_t a = add[e][q];
                    o = __builtin_elementwise_add_sat(o, __builtin_bit_cast(v2s, a));
                }
                out[q] = __builtin_bit_cast(uint32_t, __builtin_elementwise_min(__builtin_elementwise_max(o, lo2), hi2));
            }
            if (((yoff[e] | mo) >> 31) == 0u) store_tail<NT ? kNonTemporal : 0>(yr, yoff[e] + mo, yn[e], out);
        }
    }
}

template <uint32_t G, uint32_t W, bool AV, bool NT>
int launch_one(const PwsArgs& g, dim3 grid, hipStream_t s) {
    constexpr uint32_t max_lds = (G == 8 ? 256 : kMaxC) / 64 * G * 1024;
    if constexpr (max_lds > (64u << 10)) {
        static bool attr_set[64] = {};
        int dev = 0;
        (void)hipGetDevice(&dev);
        if (dev >= 0 && dev < 64 && !attr_set[dev]) {
            if (hipFuncSetAttribute(reinterpret_cast<const void*>(&conv_pws<G, W, AV, NT>),
                                    hipFuncAttributeMaxDynamicSharedMemorySize, max_lds) != hipSuccess)
                return cm_set_error(CM_ERR_HIP, "conv_pws: cannot set the LDS size");
            attr_set[dev] = true;
        }
    }
    hipLaunchKernelGGL((conv_pws<G, W, AV, NT>), grid, dim3(W * 64), g.nk * G * 1024u, s, g);
    return cm_check_launch("conv_pws");
}

template <uint32_t G, uint32_t W>
int launch(PwsArgs& g, hipStream_t s) {
    // Every block takes all output channels while the pixel tiles alone give two
    // blocks per CU, else a share of them (whole column tiles per wave): the
    // limb planes are then staged once
    const uint32_t tiles = (g.n_groups + G - 1) / G;
    const uint32_t want = (2u * cm_cu_count() + tiles - 1) / tiles;
    g.ct_per_block = std::max(W, ((g.n_ct + want - 1) / want + W - 1) / W * W);
    const dim3 grid(tiles, (g.n_ct + g.ct_per_block - 1) / g.ct_per_block);
    // x, y and the Add's operand past a third of the Infinity Cache (256 MB): y
    // would not stay there, and is stored past it
    const bool nt = (uint64_t)g.x_bytes + (g.epi.add_mode ? 2u : 1u) * (uint64_t)g.y_bytes > kStreamBytes;
    if (g.C % 8 == 0) return nt ? launch_one<G, W, true, true>(g, grid, s) : launch_one<G, W, true, false>(g, grid, s);
    return nt ? launch_one<G, W, false, true>(g, grid, s) : launch_one<G, W, false, false>(g, grid, s);
}

}  // namespace

// Pointwise convolutions of planes of at least eight pixels, 8 to 512 input
// channels and tensors below 2 GiB; returns 1, launching nothing, for others.
int cm_conv_pws_launch(const int16_t* x, const int16_t* w, const int16_t* bias, int16_t* y, uint32_t batch,
                       uint32_t in_ch, uint32_t out_ch, uint32_t hw, const cm_epilogue_t* epi, const LaunchCtx& lc) {
    const uint64_t np = (uint64_t)batch * hw;
    const uint64_t x_bytes = 2ull * in_ch * np, y_bytes = 2ull * out_ch * np, w_bytes = 2ull * out_ch * in_ch;
    if (np == 0 || out_ch == 0 || in_ch < 8 || in_ch > kMaxC || hw < 8 || x_bytes >= 0x80000000ull ||
        y_bytes >= 0x80000000ull || w_bytes >= 0x80000000ull)
        return 1;
    if (lc.need) return CM_OK;   // no workspace
    PwsArgs g{};
    g.x = x; g.w = w; g.bias = bias; g.y = y; g.epi = cm_epi_args(epi);
    g.C = in_ch; g.M = out_ch; g.P = hw;
    g.nk = (in_ch + 63) / 64;
    g.gpi = (hw + 7) / 8;
    g.n_groups = batch * g.gpi;
    g.n_ct = (out_ch + 15) / 16;
    g.x_bytes = (uint32_t)x_bytes; g.w_bytes = (uint32_t)w_bytes; g.y_bytes = (uint32_t)y_bytes;
    g.b_bytes = bias ? out_ch * 2u : 0u;
    g.div_gpi = make_fastdiv(g.gpi);
    // Up to 256 channels (32 KB of limb planes) four blocks of 64 pixels share a
    // CU; above, one block of 128 pixels and eight waves: 512 -> 128 at 32 x 28 x
    // 28 17.0 us against 25.3 (256 -> 64 at 56 x 56: 30.0 against 19.3).
    return in_ch <= 256 ? launch<8, 4>(g, lc.s) : launch<16, 8>(g, lc.s);
}
