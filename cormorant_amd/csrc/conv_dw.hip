// conv_dw.hip -- depthwise 3x3 / 5x5 convolution streamed through registers
// (kernels/conv/kernel/ConvKernel.cpp:251-319).
//
// Output channel m of image n reads input channel m through its own K x K
// filter.  The work is a stream: x in, y out, K * K multiply-adds per output
// between them, so what bounds a kernel is first the memory rate and then the
// instructions per output.  Here
//   * a lane owns eight input columns of a row (one 16-byte load) and the
//     output columns above them (8 / S), a group of L lanes a whole row, and a
//     wave 64 / L groups -- one plane's strip of output rows each;
//   * the columns a window needs to either side are one dword of each
//     neighbouring lane (a wave shift by one lane), so nothing is loaded twice
//     and nothing goes through LDS;
//   * a wave does one strip of a few output rows and ends: all of its input
//     rows are loaded at once, and many short waves keep more loads in flight
//     than few long ones that prefetch their next rows (the K - S rows that
//     neighbouring strips share come from L2);
//   * two horizontal taps are one v_dot2_i32_i16 (int16 pairs into the wrapping
//     32-bit sum), 3 * 2 or 5 * 3 of them per output, on the loaded dwords as
//     they are: the weights are paired twice, for windows that start at an even
//     and at an odd column.
// Measured (against conv_dw_band, which staged every input in LDS and read it
// back one element at a time, nine reads and nine multiply-adds per output):
// 32 x 96 x 112 x 112, 3x3: 87 -> 27 us (154 MB: 5.7 TB/s, a large copy's rate);
// stride 2: 28.8 -> 16.7; 32 x 384 x 28 x 28, 5x5: 89 -> 13.7; ragged rows,
// 15 x 72 x 106 x 151, 5x5: 178 -> 21 us.  Strips of 2 / 4 / 8 / 16 input rows:
// 26.4 / 27.0 / 27.7 / 36 us on the first shape, 24.6 / 20.9 / 21.5 / 23.4 on the
// last, whose ragged rows cost most where the shared rows are many.
#include "cm_internal.h"
#include "q88.h"

#include <algorithm>

namespace {

constexpr uint32_t kThreads = 256;
constexpr uint32_t kWaves = kThreads / 64;
constexpr int kNonTemporal = 2;   // buffer access cache policy bit
constexpr int kRows = 4;   // a strip: kRows / S output rows, which advance over kRows input rows

typedef short v2s __attribute__((ext_vector_type(2)));
typedef unsigned int v2u __attribute__((ext_vector_type(2)));
typedef unsigned int v4u __attribute__((ext_vector_type(4)));

// From this size on (a third of the MI355X's 256 MB Infinity Cache) x and y
// together no longer stay there until they are used next, and y is stored past
// it: 31.2 -> 26.9 us at 154 MB, 17.1 -> 16.1 at 96 MB, but 12.4 -> 14.4 at 58 MB and 13.8 -> 27.4 at 38 MB (rows of 56 bytes:
// partial lines), which the cache holds.  Whole 16-byte rows only.
constexpr uint64_t kStreamBytes = 80ull << 20;

struct DwRows {
    const int16_t* x;
    const int16_t* w;
    const int16_t* bias;     // null: a zero-size range, read as 0
    int16_t* y;
    EpiArgs epi;
    uint32_t C, M, H, W, OH, OW, pt;
    uint32_t lanes, groups;          // lanes per row; groups per wave
    uint32_t n_strips;               // strips per plane
    uint32_t n_groups;               // planes * n_strips
    uint32_t x_bytes, y_bytes, b_bytes;   // whole tensors, below 2^31
    FastDiv div_lanes, div_strips, div_m;
};

__device__ __forceinline__ int32_t dot2(uint32_t x, uint32_t w, int32_t acc) {
    return __builtin_amdgcn_sdot2(__builtin_bit_cast(v2s, x), __builtin_bit_cast(v2s, w), acc, false);
}

// N (8 or 4) consecutive elements at byte offset `off`, of which the first `n`
// exist: one access when all do, else 4 + 2 + 1 elements, so that nothing past
// the row's last element is touched.
template <int N>
__device__ __forceinline__ void load_run(__amdgpu_buffer_rsrc_t rs, uint32_t off, uint32_t n, uint32_t (&d)[N / 2]) {
    if (n == (uint32_t)N) {
        if constexpr (N == 8) {
            const v4u v = __builtin_amdgcn_raw_buffer_load_b128(rs, off, 0, 0);
            d[0] = v[0]; d[1] = v[1]; d[2] = v[2]; d[3] = v[3];
        } else {
            const v2u v = __builtin_amdgcn_raw_buffer_load_b64(rs, off, 0, 0);
            d[0] = v[0]; d[1] = v[1];
        }
        return;
    }
#pragma unroll
    for (int q = 0; q < N / 2; ++q) {
        const uint32_t lo = __builtin_amdgcn_raw_buffer_load_b16(rs, 2u * q < n ? off + 4u * q : kOob, 0, 0);
        const uint32_t hi = __builtin_amdgcn_raw_buffer_load_b16(rs, 2u * q + 1u < n ? off + 4u * q + 2u : kOob, 0, 0);
        d[q] = (lo & 0xFFFFu) | hi << 16;
    }
}
template <int N, int AUX>
__device__ __forceinline__ void store_run(__amdgpu_buffer_rsrc_t rs, uint32_t off, uint32_t n, const uint32_t (&d)[N / 2]) {
    if (n == (uint32_t)N) {
        if constexpr (N == 8) __builtin_amdgcn_raw_buffer_store_b128(v4u{d[0], d[1], d[2], d[3]}, rs, off, 0, AUX);
        else __builtin_amdgcn_raw_buffer_store_b64(v2u{d[0], d[1]}, rs, off, 0, AUX);
        return;
    }
    uint32_t a = d[0], b = d[1];
    if constexpr (N == 8) {
        if (n & 4u) {
            __builtin_amdgcn_raw_buffer_store_b64(v2u{d[0], d[1]}, rs, off, 0, 0);
            a = d[2]; b = d[3];
            off += 8u;
        }
    }
    if (n & 2u) {
        __builtin_amdgcn_raw_buffer_store_b32(a, rs, off, 0, 0);
        a = b;
        off += 4u;
    }
    if (n & 1u) __builtin_amdgcn_raw_buffer_store_b16((uint16_t)a, rs, off, 0, 0);
}

// K x K window, stride S both ways, PL columns of padding on the left; TAIL: the
// row is not a whole number of 16-byte vectors; NT: non-temporal stores.
template <int K, int S, int PL, bool TAIL, bool NT>
__global__ __launch_bounds__(kThreads) void conv_dw_rows(DwRows g) {
    constexpr int OPL = 8 / S;         // output columns per lane
    constexpr int U = kRows / S;       // output rows per strip
    constexpr int IN = kRows - S + K;  // input rows they read
    constexpr int NP = (K + 1) / 2;    // dot products per window row
    touch_lines(g);
    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const uint32_t grp = fdiv(lane, g.div_lanes), j = lane - grp * g.lanes;
    const uint32_t gid = (blockIdx.x * kWaves + wave) * g.groups + grp;
    const bool valid = grp < g.groups && gid < g.n_groups;
    const uint32_t gsafe = valid ? gid : 0u;
    const uint32_t plane = fdiv(gsafe, g.div_strips), strip = gsafe - plane * g.n_strips;
    const uint32_t n = fdiv(plane, g.div_m), m = plane - n * g.M;
    const uint32_t r0 = strip * U;

    const __amdgpu_buffer_rsrc_t xr = make_rsrc(g.x, g.x_bytes);
    const __amdgpu_buffer_rsrc_t yr = make_rsrc(g.y, g.y_bytes);
    const __amdgpu_buffer_rsrc_t wr = make_rsrc(g.w, g.M * (uint32_t)(K * K) * 2u);
    const __amdgpu_buffer_rsrc_t br = make_rsrc(g.bias, g.b_bytes);

    // A row's last vector of a ragged row is read eight columns before the row's
    // end and shifted down (zeros come in past the row), so no read leaves the row
    const uint32_t col = j * 8u;
    const uint32_t cb = TAIL ? min(col, g.W - 8u) : col;
    const uint32_t shift = col - cb;
    const uint32_t xoff = valid && col < g.W ? ((n * g.C + m) * g.H * g.W + cb) * 2u : kOob;
    const uint32_t xrow = g.W * 2u;
    const int32_t ih0 = (int32_t)(r0 * S) - (int32_t)g.pt;
    v4u raw[IN];
#pragma unroll
    for (int i = 0; i < IN; ++i) {
        const uint32_t ih = (uint32_t)(ih0 + i);
        raw[i] = __builtin_amdgcn_raw_buffer_load_b128(xr, ih < g.H ? xoff + ih * xrow : kOob, 0, 0);
    }

    // the filter's rows as int16 pairs: we for windows starting at an even
    // column, wo for odd ones (a dword of zeros' half in front)
    uint32_t we[K][NP], wo[K][NP];
    {
        uint32_t t[K * K];
#pragma unroll
        for (int i = 0; i < K * K; ++i)
            t[i] = (uint16_t)__builtin_amdgcn_raw_buffer_load_b16(wr, (m * (uint32_t)(K * K) + i) * 2u, 0, 0);
#pragma unroll
        for (int r = 0; r < K; ++r)
#pragma unroll
            for (int q = 0; q < NP; ++q) {
                we[r][q] = t[r * K + 2 * q] | (2 * q + 1 < K ? t[r * K + 2 * q + 1] << 16 : 0u);
                wo[r][q] = (q > 0 ? t[r * K + 2 * q - 1] : 0u) | t[r * K + 2 * q] << 16;
            }
    }
    const int32_t acc0 = (int32_t)q88::data_to_acc((int16_t)__builtin_amdgcn_raw_buffer_load_b16(br, m * 2u, 0, 0));

    const uint32_t left_mask = j > 0u ? 0xFFFFFFFFu : 0u;
    const uint32_t right_mask = j + 1u < g.lanes ? 0xFFFFFFFFu : 0u;
    // E[r]: input row r of the strip as six dwords, column pairs -1 .. 4 of the lane
    uint32_t E[IN][6];
    auto place = [&](uint32_t (&e)[6], v4u d) {
        if constexpr (TAIL) {
            const bool s4 = (shift & 4u) != 0u, s2 = (shift & 2u) != 0u;
            d = s4 ? v4u{d[2], d[3], 0u, 0u} : d;
            d = s2 ? v4u{d[1], d[2], d[3], 0u} : d;
            const uint32_t h = (shift & 1u) * 16u;
            d = v4u{__builtin_amdgcn_alignbit(d[1], d[0], h), __builtin_amdgcn_alignbit(d[2], d[1], h),
                    __builtin_amdgcn_alignbit(d[3], d[2], h), d[3] >> h};
        }
        e[1] = d[0]; e[2] = d[1]; e[3] = d[2]; e[4] = d[3];
        // lane l takes lane l - 1's last dword and lane l + 1's first one
        e[0] = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)d[3], 0x138, 0xF, 0xF, true) & left_mask;
        e[5] = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)d[0], 0x130, 0xF, 0xF, true) & right_mask;
    };
#pragma unroll
    for (int i = 0; i < IN; ++i) place(E[i], raw[i]);

    const uint32_t ocol = j * OPL;
    const uint32_t on = ocol < g.OW ? min((uint32_t)OPL, g.OW - ocol) : (uint32_t)OPL;
    const uint32_t yrow = g.OW * 2u;
    const uint32_t yoff = valid && ocol < g.OW ? ((plane * g.OH + r0) * g.OW + ocol) * 2u : kOob;
    const __amdgpu_buffer_rsrc_t ar = make_rsrc(g.epi.add, g.epi.add_mode == 1u ? g.y_bytes : 0u);
    const v2s lo = {(short)q88::act_lo(g.epi.act), (short)q88::act_lo(g.epi.act)};
    const v2s hi = {(short)q88::act_hi(g.epi.act), (short)q88::act_hi(g.epi.act)};

    // the Add's operands of every row, ahead of the first store: a load between two
    // stores would wait for the store before it
    uint32_t add[U][OPL / 2];
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
        for (int q = 0; q < OPL / 2; ++q) add[u][q] = 0u;
    if (g.epi.add_mode == 1u) {
#pragma unroll
        for (int u = 0; u < U; ++u) load_run<OPL>(ar, r0 + u < g.OH ? yoff + u * yrow : kOob, on, add[u]);
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
        const uint32_t off = r0 + u < g.OH ? yoff + u * yrow : kOob;
        int32_t acc[OPL];
#pragma unroll
        for (int o = 0; o < OPL; ++o) acc[o] = acc0;
#pragma unroll
        for (int k = 0; k < K; ++k)
#pragma unroll
            for (int q = 0; q < NP; ++q)
#pragma unroll
                for (int o = 0; o < OPL; ++o) {
                    const int start = o * S - PL + 2;   // column of the window's first tap, from pair -1
                    const int d = start / 2 + q;
                    acc[o] = dot2(E[u * S + k][d], start % 2 ? wo[k][q] : we[k][q], acc[o]);
                }
        uint32_t out[OPL / 2];
#pragma unroll
        for (int q = 0; q < OPL / 2; ++q)
            out[q] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_pk_i16(acc[2 * q] >> 8, acc[2 * q + 1] >> 8));
#pragma unroll
        for (int q = 0; q < OPL / 2; ++q) {
            const v2s v = __builtin_elementwise_add_sat(__builtin_bit_cast(v2s, out[q]), __builtin_bit_cast(v2s, add[u][q]));
            out[q] = __builtin_bit_cast(uint32_t, __builtin_elementwise_min(__builtin_elementwise_max(v, lo), hi));
        }
        store_run<OPL, NT ? kNonTemporal : 0>(yr, off, on, out);
    }
}

template <int K, int S, int PL>
int launch(const DwRows& g, uint32_t blocks, hipStream_t s) {
    const dim3 grid(blocks), block(kThreads);
    const bool nt = (uint64_t)g.x_bytes + g.y_bytes > kStreamBytes;
    if (g.W % 8 != 0) hipLaunchKernelGGL((conv_dw_rows<K, S, PL, true, false>), grid, block, 0, s, g);
    else if (nt) hipLaunchKernelGGL((conv_dw_rows<K, S, PL, false, true>), grid, block, 0, s, g);
    else hipLaunchKernelGGL((conv_dw_rows<K, S, PL, false, false>), grid, block, 0, s, g);
    return cm_check_launch("conv_dw_rows");
}

}  // namespace

// Depthwise convolutions with a 3x3 or 5x5 window, dilation 1, the same stride
// (1 or 2) both ways and a left padding whose window columns reach at most one
// dword to either side of a lane's eight; returns 1, launching nothing, for any
// other.  Rows of 8 to 512 columns (one to 64 lanes); tensors below 2 GiB.
int cm_conv_dw_rows_launch(const int16_t* x, const int16_t* w, const int16_t* bias, int16_t* y, uint32_t batch,
                           uint32_t in_ch, uint32_t in_h, uint32_t in_w, uint32_t out_ch, uint32_t out_h,
                           uint32_t out_w, uint32_t kh, uint32_t kw, uint32_t sh, uint32_t sw, uint32_t dh,
                           uint32_t dw, uint32_t pt, uint32_t pl, const EpiArgs& epi, hipStream_t s) {
    const uint64_t planes = (uint64_t)batch * out_ch;
    const uint64_t x_bytes = 2ull * batch * in_ch * in_h * in_w, y_bytes = 2ull * planes * out_h * out_w;
    const bool shape = kh == kw && (kh == 3 || kh == 5) && sh == sw && (sh == 1 || sh == 2) && dh == 1 && dw == 1 &&
                       (kh == 3 ? pl <= 1 : pl == 2 || (pl == 1 && sh == 2)) && in_w >= 8 && in_w <= 512 &&
                       pt <= 0xFFFFu && in_h <= 0xFFFFu && out_h <= 0xFFFFu &&
                       x_bytes < 0x80000000ull && y_bytes < 0x80000000ull &&
                       2ull * out_ch * kh * kw < 0x80000000ull;
    if (!shape) return 1;
    const uint32_t opl = 8 / sw;
    const uint32_t lanes = std::max((in_w + 7) / 8, (out_w + opl - 1) / opl);
    if (lanes > 64) return 1;
    DwRows g{};
    g.x = x; g.w = w; g.bias = bias; g.y = y; g.epi = epi;
    g.C = in_ch; g.M = out_ch; g.H = in_h; g.W = in_w; g.OH = out_h; g.OW = out_w; g.pt = pt;
    g.lanes = lanes;
    g.groups = 64 / lanes;
    const uint32_t u = kRows / sh;
    g.n_strips = (out_h + u - 1) / u;
    if (planes * g.n_strips > 0x7FFFFFFFull) return 1;
    g.n_groups = (uint32_t)(planes * g.n_strips);
    g.x_bytes = (uint32_t)x_bytes; g.y_bytes = (uint32_t)y_bytes; g.b_bytes = bias ? out_ch * 2u : 0u;
    g.div_lanes = make_fastdiv(lanes);
    g.div_strips = make_fastdiv(g.n_strips);
    g.div_m = make_fastdiv(out_ch);
    const uint32_t per_block = kWaves * g.groups;
    const uint32_t blocks = (g.n_groups + per_block - 1) / per_block;
    if (kh == 3) {
        if (sh == 1) return pl == 0 ? launch<3, 1, 0>(g, blocks, s) : launch<3, 1, 1>(g, blocks, s);
        return pl == 0 ? launch<3, 2, 0>(g, blocks, s) : launch<3, 2, 1>(g, blocks, s);
    }
    if (sh == 1) return launch<5, 1, 2>(g, blocks, s);
    return pl == 1 ? launch<5, 2, 1>(g, blocks, s) : launch<5, 2, 2>(g, blocks, s);
}
