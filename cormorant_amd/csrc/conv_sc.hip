// conv_sc.hip -- convolutions of at most four input channels on int8 MFMA
// (kernels/conv/kernel/ConvKernel.cpp:160-169, 171-249, 333): the first layer of an
// image network.
//
// The patch GEMM (conv_pgemm.hip) gives every window tap sixteen channels of an
// MFMA's k range; with three channels five sixths of its products are zeros.  Here
// a k chunk of sixteen values is four neighbouring columns of a window row times
// four channels: input pixels sit in LDS as one dword of high and one of low limb
// bytes (byte c = channel c), so the sixteen bytes an MFMA lane supplies are four
// consecutive pixels of a patch row -- a 7 x 7 window is 14 chunks (four k steps)
// instead of 49, a 3 x 3 one 3 (one step) instead of 9.
//   * A block owns `rb` output rows x `cb` eight-column groups of one image, and up
//     to 64 output channels; a wave eight groups (64 pixels).
//   * Input rows are loaded once, 16 bytes of eight columns per channel, and
//     transposed to channel-minor limb dwords with v_perm.
//   * The pixels are the MFMA's rows and the output channels its columns, in the
//     order of conv_pws.hip (eight groups): a lane's results are runs of eight
//     pixels of one channel, stored as 16 bytes straight from the accumulators.
//   * Weights: their limb fragments are built in LDS by each block, from the raw
//     tensor or from the patch GEMM's packed planes (a tap's first dword), so packed
//     weights serve either kernel.  A position past the window, the channels or the
//     output channels holds weight 0.
// Measured: 16 x 3 x 224 x 224 -> 64, 7 x 7 stride 2: 55.8 us on the patch GEMM, 21.3 here
// (30 MB: 6 us at the card's copy rate; staging, products and stores of the one round of
// blocks follow each other); 3 -> 64, 3 x 3 at 16 x 224 x 224 102 -> 49; one 224 x 224
// image 29 -> 16.
// Sums: a 16-channel tile whose weights are all int8 takes two products,
//     sum w*x = 256 sum w*xh + sum w*xl + 128 sum w;
// others the four limb products and both sums of gemm.hip's identity, the pixel
// sums over the very positions that the products read (whatever a position of
// weight 0 holds cancels).  Every term mod 2^32, the accumulator's wrap.
#include "cm_internal.h"
#include "limbs.h"
#include "q88.h"
#include "runs.h"

#include <algorithm>

namespace {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef short v2s __attribute__((ext_vector_type(2)));
typedef unsigned int v4u __attribute__((ext_vector_type(4)));

constexpr uint32_t kMaxWaves = 8;
constexpr uint32_t kMaxCt = 4;      // 16-channel tiles per block
constexpr uint32_t kMaxSteps = 16;  // k steps of 4 chunks
constexpr uint32_t kLdsBytes = 78u << 10;   // two blocks per CU

struct ScArgs {
    const int16_t* x;
    const int16_t* w;        // raw weights, or null
    const uint8_t* wpk;      // packed limb planes (tb rows per tile, `steps` k steps), or null
    const int16_t* bias;
    int16_t* y;
    EpiArgs epi;
    uint32_t C, H, W, M, OH, OW, KW, taps, pt, pl;
    uint32_t parts, chunks, nk;          // chunks per window row; in all; k steps
    uint32_t rb, cb, nrb, ncb, gpr;      // block rows / groups, blocks per image, groups per row
    uint32_t prow, pitch, units, plane;  // patch rows, dwords per row, 8-column units, bytes per limb plane
    uint32_t ct_per_block, n_ct;
    uint32_t tb_log, steps;
    uint32_t w_off;          // LDS bytes ahead of the weight fragments: the patch, before it the raw weights
    uint32_t x_bytes, w_bytes, y_bytes, b_bytes;
    FastDiv div_units, div_cb, div_parts, div_blk, div_ncb, div_tgs, div_kw;
};

using limbs::bsum;

__device__ __forceinline__ uint32_t perm(uint32_t hi, uint32_t lo, uint32_t sel) {
    return __builtin_amdgcn_perm(hi, lo, sel);
}

// PK: weights from the packed planes.  Every load's validity is bit 31 of its offset: a
// select there becomes a branch around the load and a wait for all others behind it.
// ADD: a fused Add (its loads, behind a branch, would make every store wait for the last).
template <uint32_t S, bool PK, bool ADD>
__global__ __launch_bounds__(kMaxWaves * 64, 2) void conv_sc(ScArgs g) {
    extern __shared__ __align__(16) uint8_t lds[];
    // [patch hi][patch lo, or the raw weights][weights: tile][k step][hi, lo][lane][16][per wave: 64 pixel sums]
    __shared__ uint32_t tab[kMaxSteps * 4];
    __shared__ uint32_t wide[kMaxCt], bias8[kMaxCt * 16], term[kMaxCt * 16];
    touch_lines(g);
    const uint32_t tid = threadIdx.x, nthr = blockDim.x, lane = tid & 63u;
    const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(tid >> 6));
    uint8_t* wlds = lds + g.w_off;
    uint32_t* xs = reinterpret_cast<uint32_t*>(wlds + g.ct_per_block * g.nk * 2048u) + wave * 64u;
    const uint32_t n = fdiv(blockIdx.x, g.div_blk), blk = blockIdx.x - n * (g.nrb * g.ncb);
    const uint32_t rblk = fdiv(blk, g.div_ncb), cblk = blk - rblk * g.ncb;
    const uint32_t oh0 = rblk * g.rb, gc0 = cblk * g.cb;
    const uint32_t ct_lo = blockIdx.y * g.ct_per_block, cts = min(g.ct_per_block, g.n_ct - ct_lo);
    // the patch's first input column: a multiple of 8, at most the first window's;
    // it is stored `shift` pixels in, so that the windows of every fourth output
    // column start at a 16-byte boundary
    const int32_t first = (int32_t)(gc0 * 8u * S) - (int32_t)g.pl;
    const int32_t c_lo = first & ~7;
    const uint32_t shift = (uint32_t)(c_lo - first) & 3u;

    if (tid < kMaxSteps * 4u) {
        const uint32_t khi = fdiv(tid, g.div_parts), part = tid - khi * g.parts;
        tab[tid] = tid < g.chunks ? (khi * g.pitch + part * 4u) * 4u : 0u;
    }
    if (tid < kMaxCt) wide[tid] = 0u;
    // the bias goes through LDS: a load between the stores of two channel tiles would
    // wait for the stores before it
    if (tid < kMaxCt * 16u) {
        const __amdgpu_buffer_rsrc_t br = make_rsrc(g.bias, g.b_bytes);
        bias8[tid] = q88::data_to_acc((int16_t)__builtin_amdgcn_raw_buffer_load_b16(br, (ct_lo * 16u + tid) * 2u, 0, 0));
    }
    const __amdgpu_buffer_rsrc_t xr = make_rsrc(g.x, g.x_bytes);
    const __amdgpu_buffer_rsrc_t wr = make_rsrc(PK ? reinterpret_cast<const int16_t*>(g.wpk) : g.w, g.w_bytes);

    // ---- weights.  Memory is read in its own order (gathered in the fragments' order
    // each lane's dword was a cache line access of its own: 9 of 26 us): raw ones are
    // copied to where the patch comes later, packed ones a row's four taps by
    // neighbouring lanes.  A wave takes four taps of a 16-channel tile at a time.
    const uint32_t rows = min(cts * 16u, g.M - ct_lo * 16u), row_elems = g.C * g.taps;
    if constexpr (!PK) {
        const uint32_t at = ct_lo * 16u * row_elems, count = rows * row_elems;
        for (uint32_t i = tid; i < count / 8u; i += nthr)
            *reinterpret_cast<v4u*>(lds + i * 16u) = __builtin_amdgcn_raw_buffer_load_b128(wr, (at + i * 8u) * 2u, 0, 0);
        const uint32_t e = (count & ~7u) + tid;
        if (tid < (count & 7u))
            *reinterpret_cast<uint16_t*>(lds + e * 2u) = (uint16_t)__builtin_amdgcn_raw_buffer_load_b16(wr, (at + e) * 2u, 0, 0);
    }
    // positions without a weight hold the limbs of 0
    for (uint32_t i = tid; i < cts * g.nk * 128u; i += nthr) {
        const uint32_t z = i & 64u ? 0x80808080u : 0u;
        *reinterpret_cast<v4u*>(wlds + i * 16u) = v4u{z, z, z, z};
    }
    __syncthreads();
    {
        const uint32_t tgs = (g.taps + 3u) / 4u, nu = cts * tgs, waves = nthr >> 6;
        constexpr uint32_t kWb = 4;
        for (uint32_t r0 = wave; r0 < nu; r0 += kWb * waves) {
            uint32_t hi[kWb], lo[kWb];
#pragma unroll
            for (uint32_t u = 0; u < kWb; ++u) {
                const uint32_t r = r0 + u * waves, ct = fdiv(r, g.div_tgs);
                const uint32_t tap = (r - ct * tgs) * 4u + (lane & 3u), ml = ct * 16u + (lane >> 2);
                const uint32_t hole = (uint32_t)(r >= nu || ml >= rows || tap >= g.taps) << 31;
                if constexpr (PK) {
                    const uint32_t m = ct_lo * 16u + ml;
                    const uint32_t at = ((m >> g.tb_log) * g.steps + (tap >> 2)) * (128u << g.tb_log) +
                                        (m & ((1u << g.tb_log) - 1u)) * 64u + (tap & 3u) * 16u;
                    hi[u] = __builtin_amdgcn_raw_buffer_load_b32(wr, (at & 0x7FFFFFFFu) | hole, 0, 0);
                    lo[u] = __builtin_amdgcn_raw_buffer_load_b32(wr, ((at + (64u << g.tb_log)) & 0x7FFFFFFFu) | hole, 0, 0);
                } else {
                    const uint16_t* e = reinterpret_cast<const uint16_t*>(lds) + (hole ? 0u : ml * row_elems + tap);
                    uint32_t v[4];
#pragma unroll
                    for (uint32_t c = 0; c < 4; ++c) v[c] = c < g.C ? e[c * g.taps] : 0u;
                    const uint32_t w0 = limbs::pack2(v[0], v[1]), w1 = limbs::pack2(v[2], v[3]);
                    hi[u] = limbs::hi4(w0, w1);
                    lo[u] = limbs::lo4(w0, w1);
                }
            }
#pragma unroll
            for (uint32_t u = 0; u < kWb; ++u) {
                const uint32_t r = r0 + u * waves, ct = fdiv(r, g.div_tgs);
                const uint32_t tap = (r - ct * tgs) * 4u + (lane & 3u), ml = ct * 16u + (lane >> 2);
                if (r >= nu || ml >= rows || tap >= g.taps) continue;
                const uint32_t khi = fdiv(tap, g.div_kw), kwi = tap - khi * g.KW, chunk = khi * g.parts + (kwi >> 2);
                uint8_t* to = wlds + (ct * g.nk + (chunk >> 2)) * 2048u + ((chunk & 3u) * 16u + (ml & 15u)) * 16u + (kwi & 3u) * 4u;
                *reinterpret_cast<uint32_t*>(to) = hi[u];
                *reinterpret_cast<uint32_t*>(to + 1024u) = lo[u];
                // int8: the high byte is the low byte's sign (lo holds it with its top bit flipped)
                const uint32_t neg = (~lo[u] & 0x80808080u) >> 7;      // 1 in each byte whose value is >= 128
                if (hi[u] != neg * 0xFFu) wide[ct] = 1u;
            }
        }
    }
    if constexpr (!PK) __syncthreads();   // the raw weights make room for the patch

    // ---- patch: (row, unit of eight columns) per thread, two at a time
    {
        const uint32_t tasks = g.prow * g.units;
        const int32_t ih0 = (int32_t)(oh0 * S) - (int32_t)g.pt;
        auto load = [&](uint32_t t, v4u (&d)[4], uint32_t& sh) {
            const uint32_t row = fdiv(t, g.div_units), u = t - row * g.units;
            const uint32_t ih = (uint32_t)(ih0 + (int32_t)row), col = (uint32_t)(c_lo + (int32_t)(u * 8u));
            // a ragged row's last unit is read eight columns before its end, shifted down
            const uint32_t cb = min(col, g.W - 8u);
            const uint32_t ok = (uint32_t)(t < tasks) & (uint32_t)(ih < g.H) & (uint32_t)(col < g.W);
            sh = (col - cb) & (0u - ok);
            const uint32_t off = ((n * g.C * g.H + ih) * g.W + cb) * 2u, hole = (ok ^ 1u) << 31;
#pragma unroll
            for (uint32_t c = 0; c < 4; ++c)
                d[c] = __builtin_amdgcn_raw_buffer_load_b128(
                    xr, ((off + c * g.H * g.W * 2u) & 0x7FFFFFFFu) | hole | (uint32_t)(c >= g.C) << 31, 0, 0);
        };
        auto put = [&](uint32_t t, v4u (&d)[4], uint32_t sh) {
            if (t >= tasks) return;
            if (g.W % 8u != 0u) {
                const uint32_t h = (sh & 1u) * 16u;
#pragma unroll
                for (uint32_t c = 0; c < 4; ++c) {
                    v4u v = d[c];
                    v = sh & 4u ? v4u{v[2], v[3], 0u, 0u} : v;
                    v = sh & 2u ? v4u{v[1], v[2], v[3], 0u} : v;
                    d[c] = v4u{__builtin_amdgcn_alignbit(v[1], v[0], h), __builtin_amdgcn_alignbit(v[2], v[1], h),
                               __builtin_amdgcn_alignbit(v[3], v[2], h), v[3] >> h};
                }
            }
            const uint32_t row = fdiv(t, g.div_units), u = t - row * g.units;
            uint32_t hi[8], lo[8];
#pragma unroll
            for (uint32_t q = 0; q < 4; ++q) {
                const uint32_t ab0 = perm(d[1][q], d[0][q], 0x06020400u), cd0 = perm(d[3][q], d[2][q], 0x06020400u);
                const uint32_t ab1 = perm(d[1][q], d[0][q], 0x07030501u), cd1 = perm(d[3][q], d[2][q], 0x07030501u);
                lo[2 * q] = perm(cd0, ab0, 0x05040100u) ^ 0x80808080u;
                lo[2 * q + 1] = perm(cd0, ab0, 0x07060302u) ^ 0x80808080u;
                hi[2 * q] = perm(cd1, ab1, 0x05040100u);
                hi[2 * q + 1] = perm(cd1, ab1, 0x07060302u);
            }
            uint32_t* to = reinterpret_cast<uint32_t*>(lds + (row * g.pitch + u * 8u + shift) * 4u);
            uint32_t* tl = reinterpret_cast<uint32_t*>(lds + g.plane + (row * g.pitch + u * 8u + shift) * 4u);
#pragma unroll
            for (uint32_t q = 0; q < 8; ++q) {
                to[q] = hi[q];
                tl[q] = lo[q];
            }
        };
        for (uint32_t t = tid; t < tasks; t += 2u * nthr) {
            v4u d0[4], d1[4];
            uint32_t s0, s1;
            load(t, d0, s0);
            load(t + nthr, d1, s1);
            put(t, d0, s0);
            put(t + nthr, d1, s1);
        }
    }
    __syncthreads();
    // the products' constant per channel: 128 sum w, the bias, and for four products
    // the identity's last term
    for (uint32_t i = tid; i < cts * 64u; i += nthr) {
        const uint32_t ct = i >> 6, ln = i & 63u;
        int32_t sh = 0, sl = 0;
        for (uint32_t s = 0; s < g.nk; ++s) {
            const uint8_t* f = wlds + (ct * g.nk + s) * 2048u + ln * 16u;
            const v4i h = *reinterpret_cast<const v4i*>(f), l = *reinterpret_cast<const v4i*>(f + 1024u);
#pragma unroll
            for (uint32_t q = 0; q < 4; ++q) {
                const int hq = h[q], lq = l[q];
                sh = bsum((uint32_t)hq, sh);
                sl = bsum((uint32_t)lq, sl);
            }
        }
        uint32_t sum = 256u * (uint32_t)sh + (uint32_t)sl + 128u * 16u * g.nk;
        sum += (uint32_t)__shfl_xor((int)sum, 16, 64);
        sum += (uint32_t)__shfl_xor((int)sum, 32, 64);
        if (ln < 16u) {
            const bool fit2 = (wide[ct & ~1u] | wide[min(ct | 1u, cts - 1u)]) == 0u;
            term[ct * 16u + ln] = bias8[ct * 16u + ln] + 128u * sum - (fit2 ? 0u : 16384u * 64u * g.nk);
        }
    }
    __syncthreads();

    // ---- this lane's fragment row: group of the wave, pixel 4 (r16 % 2) + t
    const uint32_t r16 = lane & 15u, kg = lane >> 4;
    auto group = [&](uint32_t gw, uint32_t& row, uint32_t& ow, uint32_t& cnt) {   // group gw of the wave
        const uint32_t gl = wave * 8u + gw;
        row = fdiv(gl, g.div_cb);
        const uint32_t gc = gc0 + gl - row * g.cb;
        ow = gc * 8u;
        cnt = min(8u, g.OW - ow);
        return row < g.rb && oh0 + row < g.OH && gc < g.gpr;
    };
    uint32_t frow, fow, fcnt;
    const bool fok = group(4u * ((r16 >> 1) & 1u) + (r16 >> 2), frow, fow, fcnt);
    const uint32_t fbase =
        fok ? (frow * S * g.pitch + (uint32_t)((int32_t)((fow + 4u * (r16 & 1u)) * S) - (int32_t)g.pl - c_lo) + shift) * 4u : 0u;
    uint32_t yoff[2], yn[2];
#pragma unroll
    for (uint32_t e = 0; e < 2; ++e) {
        uint32_t row, ow;
        const bool ok = group(4u * e + kg, row, ow, yn[e]);
        yoff[e] = ok ? ((n * g.M * g.OH + oh0 + row) * g.OW + ow) * 2u : kOob;
    }
    const __amdgpu_buffer_rsrc_t yr = make_rsrc(g.y, g.y_bytes);
    const __amdgpu_buffer_rsrc_t ar = make_rsrc(g.epi.add, ADD ? g.y_bytes : 0u);
    const v2s lo2 = {(short)q88::act_lo(g.epi.act), (short)q88::act_lo(g.epi.act)};
    const v2s hi2 = {(short)q88::act_hi(g.epi.act), (short)q88::act_hi(g.epi.act)};
    // The chunk of four neighbouring pixels (t = 0 .. 3: S columns apart) from one
    // limb plane: their windows overlap, so four fragments are runs of the same
    // 4 + 3 S dwords, read as whole 16-byte vectors
    auto frags = [&](uint32_t off, v4i (&f)[4]) {
        constexpr uint32_t NV = S == 1 ? 2 : 3;
        int d[NV * 4];
#pragma unroll
        for (uint32_t q = 0; q < NV; ++q) {
            const v4i v = *reinterpret_cast<const v4i*>(lds + off + q * 16u);
            d[4 * q] = v[0]; d[4 * q + 1] = v[1]; d[4 * q + 2] = v[2]; d[4 * q + 3] = v[3];
        }
#pragma unroll
        for (uint32_t t = 0; t < 4; ++t) f[t] = v4i{d[t * S], d[t * S + 1], d[t * S + 2], d[t * S + 3]};
    };

    bool have_xs = false;
    auto pixel_sums = [&]() {   // of each of the wave's pixels, over the positions its chunks read
        uint32_t v[4] = {0u, 0u, 0u, 0u};
        for (uint32_t s = 0; s < g.nk; ++s) {
            const uint32_t off = fbase + tab[s * 4u + kg];
            v4i h[4], l[4];
            frags(off, h);
            frags(off + g.plane, l);
#pragma unroll
            for (uint32_t t = 0; t < 4; ++t) {
                int32_t sh = 0, sl = 0;
#pragma unroll
                for (uint32_t q = 0; q < 4; ++q) {
                    const int hq = h[t][q], lq = l[t][q];
                    sh = bsum((uint32_t)hq, sh);
                    sl = bsum((uint32_t)lq, sl);
                }
                v[t] += 256u * (uint32_t)sh + (uint32_t)sl + 128u * 16u;
            }
        }
#pragma unroll
        for (uint32_t t = 0; t < 4; ++t) {
            v[t] += (uint32_t)__shfl_xor((int)v[t], 16, 64);
            v[t] += (uint32_t)__shfl_xor((int)v[t], 32, 64);
            if (kg == 0u) xs[t * 16u + r16] = 128u * v[t];
        }
    };
    // sums of channel tile ct, finished and stored
    auto store = [&](uint32_t ct, const uint32_t (&v)[2][8]) {
        const uint32_t m = (ct_lo + ct) * 16u + r16;
        const uint32_t mo = m < g.M ? m * g.OH * g.OW * 2u : kOob;
#pragma unroll
        for (uint32_t e = 0; e < 2; ++e) {
            if ((yoff[e] | mo) >> 31) continue;
            const uint32_t off = yoff[e] + mo;
            v4u add = v4u{0u, 0u, 0u, 0u};
            if constexpr (ADD) add = runs::load_head(ar, off, yn[e]);
            v4u out;
#pragma unroll
            for (uint32_t q = 0; q < 4; ++q) {
                const uint32_t a = add[q];
                v2s o = __builtin_bit_cast(v2s, __builtin_amdgcn_cvt_pk_i16((int32_t)v[e][2 * q] >> 8, (int32_t)v[e][2 * q + 1] >> 8));
                if constexpr (ADD) o = __builtin_elementwise_add_sat(o, __builtin_bit_cast(v2s, a));
                out[q] = __builtin_bit_cast(uint32_t, __builtin_elementwise_min(__builtin_elementwise_max(o, lo2), hi2));
            }
            runs::store_head(yr, off, yn[e], out);
        }
    };

    for (uint32_t ct = 0; ct < cts; ct += 2) {
        const uint32_t c1 = min(ct + 1u, cts - 1u);   // an odd count's last tile is done twice, stored once
        const bool fit = (wide[ct] | wide[c1]) == 0u;
        const uint8_t* wf[2] = {wlds + ct * g.nk * 2048u + lane * 16u, wlds + c1 * g.nk * 2048u + lane * 16u};
        uint32_t v[2][2][8];
        if (__builtin_amdgcn_readfirstlane((int)fit)) {
            v4i h[4][2], l[4][2];
#pragma unroll
            for (uint32_t t = 0; t < 4; ++t)
#pragma unroll
                for (uint32_t i = 0; i < 2; ++i) {
                    const int c = (int)term[(i ? c1 : ct) * 16u + r16];
                    h[t][i] = v4i{0, 0, 0, 0};
                    l[t][i] = v4i{c, c, c, c};
                }
            for (uint32_t s = 0; s < g.nk; ++s) {
                const uint32_t off = fbase + tab[s * 4u + kg];
                v4i w8[2], ah[4], al[4];
#pragma unroll
                for (uint32_t i = 0; i < 2; ++i)
                    w8[i] = *reinterpret_cast<const v4i*>(wf[i] + s * 2048u + 1024u) ^ (int)0x80808080;
                frags(off, ah);
                frags(off + g.plane, al);
#pragma unroll
                for (uint32_t t = 0; t < 4; ++t)
#pragma unroll
                    for (uint32_t i = 0; i < 2; ++i) {
                        h[t][i] = __builtin_amdgcn_mfma_i32_16x16x64_i8(ah[t], w8[i], h[t][i], 0, 0, 0);
                        l[t][i] = __builtin_amdgcn_mfma_i32_16x16x64_i8(al[t], w8[i], l[t][i], 0, 0, 0);
                    }
            }
#pragma unroll
            for (uint32_t i = 0; i < 2; ++i) {
#pragma unroll
                for (uint32_t q = 0; q < 16; ++q)
                    v[i][q / 8][q % 8] = ((uint32_t)h[q % 4][i][q / 4] << 8) + (uint32_t)l[q % 4][i][q / 4];
            }
        } else {
            if (!have_xs) {
                pixel_sums();
                have_xs = true;
            }
            v4i hh[4][2], mid[4][2], ll[4][2];
#pragma unroll
            for (uint32_t t = 0; t < 4; ++t)
#pragma unroll
                for (uint32_t i = 0; i < 2; ++i) {
                    const int c = (int)term[(i ? c1 : ct) * 16u + r16];
                    hh[t][i] = mid[t][i] = v4i{0, 0, 0, 0};
                    ll[t][i] = v4i{c, c, c, c};
                }
            for (uint32_t s = 0; s < g.nk; ++s) {
                const uint32_t off = fbase + tab[s * 4u + kg];
                v4i bh[2], bl[2], ah[4], al[4];
#pragma unroll
                for (uint32_t i = 0; i < 2; ++i) {
                    bh[i] = *reinterpret_cast<const v4i*>(wf[i] + s * 2048u);
                    bl[i] = *reinterpret_cast<const v4i*>(wf[i] + s * 2048u + 1024u);
                }
                frags(off, ah);
                frags(off + g.plane, al);
#pragma unroll
                for (uint32_t t = 0; t < 4; ++t)
#pragma unroll
                    for (uint32_t i = 0; i < 2; ++i) {
                        hh[t][i] = __builtin_amdgcn_mfma_i32_16x16x64_i8(ah[t], bh[i], hh[t][i], 0, 0, 0);
                        mid[t][i] = __builtin_amdgcn_mfma_i32_16x16x64_i8(ah[t], bl[i], mid[t][i], 0, 0, 0);
                        ll[t][i] = __builtin_amdgcn_mfma_i32_16x16x64_i8(al[t], bl[i], ll[t][i], 0, 0, 0);
                        mid[t][i] = __builtin_amdgcn_mfma_i32_16x16x64_i8(al[t], bh[i], mid[t][i], 0, 0, 0);
                    }
            }
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
#pragma unroll
            for (uint32_t i = 0; i < 2; ++i) {
#pragma unroll
                for (uint32_t q = 0; q < 16; ++q) {
                    const uint32_t t = q % 4, e = q / 4;
                    v[i][q / 8][q % 8] = ((((uint32_t)hh[t][i][e] << 8) + (uint32_t)mid[t][i][e]) << 8) +
                                         (uint32_t)ll[t][i][e] + xs[t * 16u + kg * 4u + e];
                }
            }
        }
        store(ct, v[0]);
        if (ct + 1u < cts) store(ct + 1u, v[1]);
    }
}

template <uint32_t S, bool PK, bool ADD>
int launch(const ScArgs& g, dim3 grid, dim3 block, uint32_t lds, hipStream_t s) {
    static bool attr_set[64] = {};
    int dev = 0;
    (void)hipGetDevice(&dev);
    if (dev >= 0 && dev < 64 && !attr_set[dev]) {
        if (hipFuncSetAttribute(reinterpret_cast<const void*>(&conv_sc<S, PK, ADD>),
                                hipFuncAttributeMaxDynamicSharedMemorySize, kLdsBytes) != hipSuccess)
            return cm_set_error(CM_ERR_HIP, "conv_sc: cannot set the LDS size");
        attr_set[dev] = true;
    }
    hipLaunchKernelGGL((conv_sc<S, PK, ADD>), grid, block, lds, s, g);
    return cm_check_launch("conv_sc");
}

}  // namespace

// Convolutions of at most four input channels, windows of two or more taps and up
// to 16 x 16, dilation 1, the same stride (1 or 2) both ways, rows of at least eight
// columns; w raw, or wpk the patch GEMM's planes (tb rows a tile, `steps`
// k steps, of wpk_bytes).  Returns 1, launching nothing, for any other shape.
int cm_conv_sc_launch(const int16_t* x, const int16_t* w, const uint8_t* wpk, uint32_t wpk_bytes, uint32_t tb,
                      uint32_t steps, const int16_t* bias, int16_t* y, uint32_t batch, uint32_t in_ch, uint32_t in_h,
                      uint32_t in_w, uint32_t out_ch, uint32_t out_h, uint32_t out_w, uint32_t kh, uint32_t kw,
                      uint32_t sh, uint32_t sw, uint32_t dh, uint32_t dw, uint32_t pt, uint32_t pl,
                      const EpiArgs& epi, hipStream_t s) {
    const uint64_t x_bytes = 2ull * batch * in_ch * in_h * in_w, y_bytes = 2ull * batch * out_ch * out_h * out_w;
    if (in_ch == 0 || in_ch > 4 || kh * kw < 2 || kh > 16 || kw > 16 || dh != 1 || dw != 1 || sh != sw || sh == 0 ||
        sh > 2 || in_w < 8 || pt > 0xFFFFu || pl > 0xFFFFu || in_h > 0xFFFFu || out_h > 0xFFFFu ||
        in_w > 0xFFFFu || out_w > 0xFFFFu || x_bytes >= 0x80000000ull || y_bytes >= 0x80000000ull ||
        2ull * out_ch * in_ch * kh * kw >= 0x80000000ull)
        return 1;
    ScArgs g{};
    g.x = x; g.w = w; g.wpk = wpk; g.bias = bias; g.y = y; g.epi = epi;
    g.C = in_ch; g.H = in_h; g.W = in_w; g.M = out_ch; g.OH = out_h; g.OW = out_w;
    g.KW = kw; g.taps = kh * kw; g.pt = pt; g.pl = pl;
    g.parts = (kw + 3) / 4;
    g.chunks = kh * g.parts;
    g.nk = (g.chunks + 3) / 4;
    g.gpr = (out_w + 7) / 8;
    g.n_ct = (out_ch + 15) / 16;
    g.ct_per_block = std::min(g.n_ct, kMaxCt);
    while (tb > 1u << g.tb_log) ++g.tb_log;
    g.steps = steps;
    // Column groups per block: a whole row while it fits four waves, else equal shares
    const uint32_t most = 4 * 8;
    g.ncb = (g.gpr + most - 1) / most;
    g.cb = (g.gpr + g.ncb - 1) / g.ncb;
    // patch columns: the windows of cb * 8 pixels, up to 7 to the left of the first
    // (whole units), and what a chunk reads past its window's last tap
    g.units = (7 + (g.cb * 8 - 1) * sh + 4 * g.parts + 7) / 8;
    g.pitch = g.units * 8 + 4;   // and the shift to 16 bytes
    const uint32_t raw = w ? (g.ct_per_block * 32u * in_ch * kh * kw + 15u) & ~15u : 0u;
    auto plane_of = [&](uint32_t rb) { return (((rb - 1) * sh + kh) * g.pitch * 4u + 96u + 15u) & ~15u; };
    auto lds_of = [&](uint32_t rb) {
        return std::max(2u * plane_of(rb), raw) + g.ct_per_block * g.nk * 2048u + kMaxWaves * 256u;
    };
    if (g.nk > kMaxSteps) return 1;
    // Output rows per block within the LDS budget, fewer while the blocks leave CUs
    // idle.  A block reads kh - stride rows of its neighbour again: tall windows take up
    // to eight waves of pixels (7 x 7 at 112 columns: 21.3 us, 24.9 on four), others four
    // (3 x 3 at 224: 48.6 against 56.0).
    uint32_t rb = std::min<uint32_t>(out_h, std::max(1u, (kh > 4 ? kMaxWaves : 4u) * 8 / g.cb));
    const uint64_t ctb = (g.n_ct + g.ct_per_block - 1) / g.ct_per_block;
    auto blocks = [&](uint32_t r) { return (uint64_t)batch * ((out_h + r - 1) / r) * g.ncb * ctb; };
    while (rb > 1 && (lds_of(rb) > kLdsBytes || blocks(rb) < cm_cu_count())) --rb;
    if (lds_of(rb) > kLdsBytes || (uint64_t)batch * ((out_h + rb - 1) / rb) * g.ncb > 0x7FFFFFFFull || ctb > 65535u) return 1;
    g.rb = rb;
    g.nrb = (out_h + rb - 1) / rb;
    g.prow = (rb - 1) * sh + kh;
    g.plane = plane_of(rb);
    g.w_off = std::max(2u * g.plane, raw);
    g.x_bytes = (uint32_t)x_bytes; g.y_bytes = (uint32_t)y_bytes;
    g.w_bytes = w ? 2u * out_ch * in_ch * kh * kw : wpk_bytes;
    g.b_bytes = bias ? out_ch * 2u : 0u;
    g.div_tgs = make_fastdiv((g.taps + 3) / 4);
    g.div_kw = make_fastdiv(kw);
    g.div_units = make_fastdiv(g.units);
    g.div_cb = make_fastdiv(g.cb);
    g.div_parts = make_fastdiv(g.parts);
    g.div_blk = make_fastdiv(g.nrb * g.ncb);
    g.div_ncb = make_fastdiv(g.ncb);
    const uint32_t waves = (rb * g.cb + 7) / 8;
    const dim3 grid(batch * g.nrb * g.ncb, (uint32_t)ctb), block(waves * 64);
    const uint32_t lds = lds_of(rb);
    const bool add = epi.add_mode == 1u;
    if (sh == 1) return w ? add ? launch<1, false, true>(g, grid, block, lds, s) : launch<1, false, false>(g, grid, block, lds, s)
                          : add ? launch<1, true, true>(g, grid, block, lds, s) : launch<1, true, false>(g, grid, block, lds, s);
    return w ? add ? launch<2, false, true>(g, grid, block, lds, s) : launch<2, false, false>(g, grid, block, lds, s)
             : add ? launch<2, true, true>(g, grid, block, lds, s) : launch<2, true, false>(g, grid, block, lds, s);
}
