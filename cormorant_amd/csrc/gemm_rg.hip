// gemm_rg.hip -- dense Q8.8 MatMul on int8 MFMA for operands of any size and
// alignment (kernels/matmul/kernel/MatmulKernel.cpp:196-218):
//     C[bi] = sat16( wrap32( A[bi] x B[bi] ) >> 8 ),  int16 A [n][k], B [k][m].
//
// A block owns 32 WR rows x 64 WC columns of C and walks K in steps of 64.
//   * B goes through LDS: a thread loads 4 k x 4 columns (8-byte loads along the
//     rows, at any alignment), turns them into limb bytes, k minor, with v_perm (a
//     4 x 4 byte transpose per column pair) and writes them where the fragment
//     reads want them, 16 bytes a lane, into one of two buffers: one barrier a step.
//   * A is staged the same way in the form for many tiles (ALDS).  With few, a
//     launch is a chain of latencies, and a wave loads its 32 rows straight into
//     registers two steps ahead: an MFMA lane's operand, 16 consecutive k of a row,
//     is two 16-byte loads.  (That form costs a cache line access per 16 bytes,
//     since neighbouring lanes hold different rows.)
//   * The columns are the MFMA's rows and the rows of A its columns: result row r
//     of column tile t is column 4 (r % 2) + t of the eight-column group
//     4 (r % 4 / 2) + r / 4, so that a lane's results are runs of eight
//     neighbouring columns of one row of C: 16-byte stores straight from the
//     accumulators, no LDS tile.
// Ragged edges: the last 4 columns of B and the last 8 k of A are read that many
// values before the row's end and shifted down, so that no access leaves its row;
// C's last columns are stored in pieces.
//
// Measured against the 128 x 128 tiles of gemm.hip, whose loads are one element each
// where a size is odd and whose steps end in a transposing LDS store and a barrier per
// eight waves: 2000 x 1283 x 1001 75.8 -> 23.4 us (16 MB of split-K sums less), 32 x 1023^3
// 692 -> 214, 4096 x 4095 x 4095 1308 -> 289, 2000 x 1280 x 1000 26.1 -> 18.9, 96 x 197 x 64 x
// 197 24.3 -> 12.7 (HIP graphs of back-to-back calls).
//
// Limbs and the exact sum are those of gemm.hip: v = 256 vh + vl + 128,
//     sum a*b = 65536 S_hh + 256 S_mid + S_ll + 128 (sum_k a + sum_k b) - 16384 Kp
// over Kp = 64 * steps positions, every term mod 2^32 (the accumulator's wrap);
// |S_mid| < 2^15 per k, so K is at most 32768 here.
#include "cm_internal.h"
#include "limbs.h"
#include "q88.h"
#include "runs.h"

#include <algorithm>

namespace {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef short v2s __attribute__((ext_vector_type(2)));
typedef unsigned int v2u __attribute__((ext_vector_type(2)));
typedef unsigned int v4u __attribute__((ext_vector_type(4)));

struct RgArgs {
    const int16_t* a;
    const int16_t* b;
    int16_t* c;
    uint32_t* ws;                // split-K partial sums [split][row][ws_ld], or null
    EpiArgs epi;                 // add_mode 1: laid out like C; 2: one value per column
    uint32_t n, k, m, nk;
    uint64_t a_bs, b_bs, c_bs;   // elements between batches
    uint32_t tx, ty;             // column / row tiles
    uint32_t steps;              // k steps per split
    uint32_t ws_ld;              // m rounded up to 8
};

using limbs::bsum;
using limbs::hi4;
using limbs::lo4;
using runs::load_head;
using runs::store_head;

__device__ __forceinline__ uint32_t perm(uint32_t hi, uint32_t lo, uint32_t sel) {
    return __builtin_amdgcn_perm(hi, lo, sel);
}

// WR x WC waves of 32 x 64 outputs; KS groups of them take every KS-th k step and
// meet in LDS.  AK: k is a multiple of 8 (whole 16-byte pieces of an A row).  ALDS:
// A goes through LDS, one step of loads ahead, else through registers, two ahead.
template <uint32_t WR, uint32_t WC, uint32_t KS, bool ALDS, bool AK>
__global__ __launch_bounds__(WR * WC * KS * 64, 2) void gemm_rg(RgArgs g) {
    static_assert(ALDS ? KS == 1 : WC == 1, "A rows in registers belong to one wave");
    constexpr uint32_t kWaves = WR * WC, kT = kWaves * 64, BM = 32 * WR, BN = 64 * WC;
    constexpr uint32_t kBufA = ALDS ? BM * 64 * 2 : 0, kBufB = BN * 64 * 2;   // limb planes of a k step
    constexpr uint32_t kStage = kBufA + kBufB;
    constexpr uint32_t U = 4 / WR;                  // 4 x 4 units of B a thread stages per step
    constexpr uint32_t UA = ALDS ? BM * 4 / kT : 2; // units of one A row x 16 k per thread
    __shared__ __align__(16) uint8_t lds_all[KS * 2 * kStage];
    __shared__ uint32_t csum[BN], rsum[BM];
    touch_lines(g);
    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t wave_all = (uint32_t)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const uint32_t kz = KS == 1 ? 0u : wave_all / kWaves, wave = wave_all - kz * kWaves;
    const uint32_t tid = threadIdx.x - kz * kT;          // within the k group
    uint8_t* lds = lds_all + kz * 2u * kStage;
    const uint32_t wr = wave % WR, wc = wave / WR;
    const uint32_t r16 = lane & 15u, kg = lane >> 4;
    // XCD-aware order: workgroups are dealt round robin to the 8 XCDs; XCD x takes
    // the x-th contiguous share of the tiles, rows of tiles in groups of eight
    const uint32_t nb = gridDim.x, per = nb >> 3, rem = nb & 7u, xcd = blockIdx.x & 7u, idx = blockIdx.x >> 3;
    const uint32_t tt = xcd < rem ? xcd * (per + 1u) + idx : rem * (per + 1u) + (xcd - rem) * per + idx;
    const uint32_t gsize = 8u * g.tx, grp_t = tt / gsize, first = grp_t * 8u, in_grp = tt - grp_t * gsize;
    const uint32_t rows_in = min(g.ty - first, 8u);
    const uint32_t row0 = (first + in_grp % rows_in) * BM, col0 = (in_grp / rows_in) * BN;
    const uint32_t bz = g.ws ? 0u : blockIdx.y, split = g.ws ? blockIdx.y : 0u;
    const uint32_t s_lo = split * g.steps, s_hi = min(s_lo + g.steps, g.nk);
    const __amdgpu_buffer_rsrc_t ar = make_rsrc(g.a + (uint64_t)bz * g.a_bs, g.n * g.k * 2u);
    const __amdgpu_buffer_rsrc_t br = make_rsrc(g.b + (uint64_t)bz * g.b_bs, g.k * g.m * 2u);

    // ---- A: units of one row x 16 k (8 words): ALDS: four neighbouring lanes a row's
    // 128 bytes, else the MFMA's own order (row r16 of two row tiles, k chunk kg).
    // Vector loads at odd elements (2 bytes past a dword) are several times slower
    // than at even ones (2000 x 1283 x 1000: 47 us, 1282: 31), so a row that starts
    // there is read from one element earlier and shifted into place, its last element
    // by a load of its own (row 0 has no earlier element: it takes the slow loads).
    uint32_t arow[UA], ash[UA];
    const uint32_t ak = (ALDS ? tid & 3u : kg) * 16u;
    auto a_row = [&](uint32_t j) { return ALDS ? (j * kT + tid) >> 2 : wr * 32u + j * 16u + r16; };
#pragma unroll
    for (uint32_t j = 0; j < UA; ++j) {
        const uint32_t r = row0 + a_row(j);
        const uint32_t at = (uint32_t)((uintptr_t)g.a >> 1) + bz * (uint32_t)g.a_bs + r * g.k;
        ash[j] = !AK && r > 0u && (at & 1u) ? 16u : 0u;
        arow[j] = r < g.n ? r * g.k * 2u - ash[j] / 8u : kOob;
    }
    struct ARaw { v4u v[UA][2]; uint32_t x[UA]; };
    auto load_a = [&](uint32_t s, ARaw& d) {
        const uint32_t kk = s * 64u + ak;
        if constexpr (AK) {
#pragma unroll
            for (uint32_t q = 0; q < 2; ++q) {
                const uint32_t hole = (uint32_t)(kk + q * 8u >= g.k || s >= s_hi) << 31;
#pragma unroll
                for (uint32_t j = 0; j < UA; ++j)
                    d.v[j][q] = __builtin_amdgcn_raw_buffer_load_b128(ar, (arow[j] + (kk + q * 8u) * 2u) | hole, 0, 0);
            }
        } else {
            // the row's last 16 values stand in for a window that reaches past its end
            const uint32_t kb = min(kk, g.k - 16u);
            const uint32_t hole = (uint32_t)(kk >= g.k || s >= s_hi) << 31;
#pragma unroll
            for (uint32_t j = 0; j < UA; ++j) {
                const uint32_t off = (arow[j] + kb * 2u) | hole;
                d.v[j][0] = __builtin_amdgcn_raw_buffer_load_b128(ar, off, 0, 0);
                d.v[j][1] = __builtin_amdgcn_raw_buffer_load_b128(ar, off + 16u, 0, 0);
                d.x[j] = (uint16_t)__builtin_amdgcn_raw_buffer_load_b16(ar, ash[j] ? off + 32u : kOob, 0, 0);
            }
        }
    };
    int32_t rs[UA];
#pragma unroll
    for (uint32_t j = 0; j < UA; ++j) rs[j] = 0;
    // unit j of step s in place (its sum added to rs[j]), as limbs
    auto split_a = [&](uint32_t s, const ARaw& ra, uint32_t j, v4i& hi, v4i& lo) {
        uint32_t w[8];
#pragma unroll
        for (uint32_t e = 0; e < 8; ++e) w[e] = ra.v[j][e / 4][e % 4];
        if constexpr (!AK) {
#pragma unroll
            for (uint32_t e = 0; e < 8; ++e)
                w[e] = __builtin_amdgcn_alignbit(e < 7 ? w[e + 1] : ra.x[j], w[e], ash[j]);
            if (s + 1 >= g.nk) {   // shift a stand-in window down, zeros past the row's end
                const uint32_t kk = s * 64u + ak, sh = kk - min(kk, g.k - 16u);
#pragma unroll
                for (uint32_t b = 4; b > 0; b >>= 1)
#pragma unroll
                    for (uint32_t e = 0; e < 8; ++e) w[e] = sh & (2u * b) ? (e + b < 8 ? w[e + b] : 0u) : w[e];
#pragma unroll
                for (uint32_t e = 0; e < 8; ++e)
                    w[e] = __builtin_amdgcn_alignbit(e < 7 ? w[e + 1] : 0u, w[e], (sh & 1u) * 16u);
            }
        }
#pragma unroll
        for (uint32_t e = 0; e < 8; ++e) {
            const uint32_t v = w[e];
            rs[j] = __builtin_amdgcn_sdot2(__builtin_bit_cast(v2s, v), v2s{1, 1}, rs[j], false);
        }
#pragma unroll
        for (uint32_t q = 0; q < 4; ++q) {
            hi[q] = (int)hi4(w[2 * q], w[2 * q + 1]);
            lo[q] = (int)lo4(w[2 * q], w[2 * q + 1]);
        }
    };
    v4i ah[2], al[2], bh[4], bl[4];
    auto put_a = [&](uint32_t s, uint32_t buf, const ARaw& ra) {
#pragma unroll
        for (uint32_t j = 0; j < UA; ++j) {
            v4i hi, lo;
            split_a(s, ra, j, hi, lo);
            // fragment slot (k chunk, row), rows moved by the chunk so that the four
            // chunks of a row land in different banks
            const uint32_t row = a_row(j), q = tid & 3u;
            uint8_t* to = lds + buf * kStage + (row >> 4) * 2048u + (q * 16u + ((row & 15u) ^ q << 2)) * 16u;
            *reinterpret_cast<v4i*>(to) = hi;
            *reinterpret_cast<v4i*>(to + 1024u) = lo;
        }
    };
    // ---- B: units of 4 k x 4 columns; unit u: k group, column group
    // lanes 0-15 and 16-31 of a half wave: 16 column groups of two k groups
    struct BRaw { v2u v[U][4]; };
    uint32_t boff[U], bsh[U], bdst[U];
#pragma unroll
    for (uint32_t u = 0; u < U; ++u) {
        const uint32_t id = u * kT + tid;                    // 256 * WC units
        const uint32_t c4 = (id & 15u) | (WC == 2 ? (id >> 5 & 1u) << 4 : 0u);
        const uint32_t k4 = (id >> 4 & 1u) | (WC == 2 ? id >> 6 : id >> 5) << 1;
        const uint32_t col = col0 + c4 * 4u;
        const uint32_t cb = min(col, g.m - 4u);
        bsh[u] = min(col - cb, 4u) * 16u;
        boff[u] = col < g.m ? (k4 * 4u * g.m + cb) * 2u : kOob;
        const uint32_t grp = (c4 >> 1) & 7u, row = 4u * (grp & 3u) + 2u * (grp >> 2) + (c4 & 1u);
        bdst[u] = kBufA + (c4 >> 4) * (kBufB / WC) + ((k4 >> 2) * 16u + row) * 16u + (k4 & 3u) * 4u;
    }
    auto load_b = [&](uint32_t s, BRaw& d) {
#pragma unroll
        for (uint32_t u = 0; u < U; ++u) {
            // rows past K lie past the buffer and read 0; steps past the last too (the
            // whole offset in the vector operand: the range check covers it)
            const uint32_t at = (s < s_hi ? boff[u] : kOob) + s * 128u * g.m;
#pragma unroll
            for (uint32_t e = 0; e < 4; ++e)
                d.v[u][e] = __builtin_amdgcn_raw_buffer_load_b64(br, at + e * g.m * 2u, 0, 0);
        }
    };
    int32_t hs[U][4], ls[U][4];
#pragma unroll
    for (uint32_t u = 0; u < U; ++u)
#pragma unroll
        for (uint32_t e = 0; e < 4; ++e) hs[u][e] = ls[u][e] = 0;
    auto put_b = [&](uint32_t buf, const BRaw& d) {
#pragma unroll
        for (uint32_t u = 0; u < U; ++u) {
            uint8_t* to = lds + buf * kStage + bdst[u];
            uint32_t w[4][2];
#pragma unroll
            for (uint32_t e = 0; e < 4; ++e) {
                const uint64_t v = ((uint64_t)d.v[u][e][1] << 32 | d.v[u][e][0]) >> (bsh[u] & 63u);
                w[e][0] = (uint32_t)v;
                w[e][1] = (uint32_t)(v >> 32);
            }
#pragma unroll
            for (uint32_t q = 0; q < 2; ++q) {
                const uint32_t ab0 = perm(w[1][q], w[0][q], 0x06020400u), cd0 = perm(w[3][q], w[2][q], 0x06020400u);
                const uint32_t ab1 = perm(w[1][q], w[0][q], 0x07030501u), cd1 = perm(w[3][q], w[2][q], 0x07030501u);
#pragma unroll
                for (uint32_t h = 0; h < 2; ++h) {
                    const uint32_t sel = h ? 0x07060302u : 0x05040100u, t = 2 * q + h;
                    const uint32_t lo = perm(cd0, ab0, sel) ^ 0x80808080u, hi = perm(cd1, ab1, sel);
                    hs[u][t] = bsum(hi, hs[u][t]);
                    ls[u][t] = bsum(lo, ls[u][t]);
                    *reinterpret_cast<uint32_t*>(to + t * 2048u) = hi;
                    *reinterpret_cast<uint32_t*>(to + t * 2048u + 1024u) = lo;
                }
            }
        }
    };

    v4i hh[4][2], mid[4][2], ll[4][2];
#pragma unroll
    for (uint32_t t = 0; t < 4; ++t)
#pragma unroll
        for (uint32_t i = 0; i < 2; ++i) hh[t][i] = mid[t][i] = ll[t][i] = v4i{0, 0, 0, 0};
    auto read_frags = [&](uint32_t buf) {
        const uint8_t* st = lds + buf * kStage;
        if constexpr (ALDS) {
            const uint8_t* f = st + wr * 4096u + (kg * 16u + (r16 ^ kg << 2)) * 16u;
#pragma unroll
            for (uint32_t i = 0; i < 2; ++i) {
                ah[i] = *reinterpret_cast<const v4i*>(f + i * 2048u);
                al[i] = *reinterpret_cast<const v4i*>(f + i * 2048u + 1024u);
            }
        }
        const uint8_t* f = st + kBufA + wc * (kBufB / WC) + lane * 16u;
#pragma unroll
        for (uint32_t t = 0; t < 4; ++t) {
            bh[t] = *reinterpret_cast<const v4i*>(f + t * 2048u);
            bl[t] = *reinterpret_cast<const v4i*>(f + t * 2048u + 1024u);
        }
    };
    auto products = [&]() {
#pragma unroll
        for (uint32_t t = 0; t < 4; ++t)
#pragma unroll
            for (uint32_t i = 0; i < 2; ++i) {
                hh[t][i] = __builtin_amdgcn_mfma_i32_16x16x64_i8(bh[t], ah[i], hh[t][i], 0, 0, 0);
                mid[t][i] = __builtin_amdgcn_mfma_i32_16x16x64_i8(bh[t], al[i], mid[t][i], 0, 0, 0);
                ll[t][i] = __builtin_amdgcn_mfma_i32_16x16x64_i8(bl[t], al[i], ll[t][i], 0, 0, 0);
                mid[t][i] = __builtin_amdgcn_mfma_i32_16x16x64_i8(bl[t], ah[i], mid[t][i], 0, 0, 0);
            }
    };
    // Step s: its limb planes are in one buffer behind the barrier; the next step's
    // are written to the other one while its products run.
    uint32_t s = s_lo + kz;   // steps s, s + KS, ... (past the last they read 0)
    const uint32_t turns = (s_hi - s_lo + KS - 1) / KS;
    if constexpr (ALDS) {
        ARaw a;
        BRaw b;
        load_b(s, b);
        load_a(s, a);
        put_a(s, 0, a);
        put_b(0, b);
        load_a(s + 1, a);
        load_b(s + 1, b);
        for (uint32_t i = 0; i < turns; ++i, ++s) {
            __syncthreads();
            read_frags(i & 1u);
            __builtin_amdgcn_sched_barrier(0);
            put_a(s + 1, (i & 1u) ^ 1u, a);
            put_b((i & 1u) ^ 1u, b);
            load_a(s + 2, a);
            load_b(s + 2, b);
            products();
        }
    } else {
        // the other buffer's limb splits (VALU, LDS writes) in the shadow of the products
        auto mix = [&]() {
#pragma unroll
            for (int i = 0; i < 32; ++i) {
                __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);
                __builtin_amdgcn_sched_group_barrier(0x2, 2, 0);
                if (i % 4 == 3) __builtin_amdgcn_sched_group_barrier(0x200, 1, 0);
            }
            __builtin_amdgcn_sched_barrier(0);
        };
        auto split = [&](uint32_t s, const ARaw& a) {
#pragma unroll
            for (uint32_t i = 0; i < 2; ++i) split_a(s, a, i, ah[i], al[i]);
        };
        ARaw a0, a1;
        BRaw b0, b1;
        load_b(s, b0);
        load_a(s, a0);
        load_b(s + KS, b1);
        load_a(s + KS, a1);
        put_b(0, b0);
        load_b(s + 2 * KS, b0);
        for (uint32_t i = 0;;) {   // entered once at least: a loop that may not be spills 168 registers
            split(s, a0);
            load_a(s + 2 * KS, a0);
            __syncthreads();
            read_frags(0);
            __builtin_amdgcn_sched_barrier(0);
            put_b(1, b1);
            load_b(s + 3 * KS, b1);
            products();
            mix();
            if (i + 1 >= turns) break;
            split(s + KS, a1);
            load_a(s + 3 * KS, a1);
            __syncthreads();
            read_frags(1);
            __builtin_amdgcn_sched_barrier(0);
            put_b(0, b0);
            load_b(s + 4 * KS, b0);
            products();
            mix();
            s += 2 * KS;
            if ((i += 2) >= turns) break;
        }
    }

    // The lane number made opaque: what follows from it stays behind the loop instead
    // of being computed, and held in registers, ahead of it (168 of them spilled)
    uint32_t ln = lane;
    asm volatile("" : "+v"(ln));
#pragma unroll
    for (uint32_t t = 0; t < 4; ++t)
#pragma unroll
        for (uint32_t i = 0; i < 2; ++i)
            asm volatile("" : "+v"(hh[t][i]), "+v"(mid[t][i]), "+v"(ll[t][i]));
    const uint32_t er16 = ln & 15u, ekg = ln >> 4, et = wave * 64u + ln;
    // column sums of B and row sums of A: this thread's values, met in LDS
    __syncthreads();
    for (uint32_t i = (kz * kT + et); i < BN; i += KS * kT) csum[i] = 0u;
    for (uint32_t i = (kz * kT + et); i < BM; i += KS * kT) rsum[i] = 0u;
    __syncthreads();
#pragma unroll
    for (uint32_t u = 0; u < U; ++u) {
        const uint32_t id = u * kT + et;
        const uint32_t c4 = (id & 15u) | (WC == 2 ? (id >> 5 & 1u) << 4 : 0u);
#pragma unroll
        for (uint32_t e = 0; e < 4; ++e)
            atomicAdd(&csum[c4 * 4u + e], 256u * (uint32_t)hs[u][e] + (uint32_t)ls[u][e]);
    }
#pragma unroll
    for (uint32_t j = 0; j < UA; ++j) 
        atomicAdd(&rsum[ALDS ? (j * kT + et) >> 2 : wr * 32u + j * 16u + er16], (uint32_t)rs[j]);
    __syncthreads();

    const __amdgpu_buffer_rsrc_t cr = make_rsrc(g.c + (uint64_t)bz * g.c_bs, g.n * g.m * 2u);
    const __amdgpu_buffer_rsrc_t er = make_rsrc(g.epi.add + (g.epi.add_mode == 1u ? (uint64_t)bz * g.c_bs : 0u),
                                                g.epi.add_mode == 0u ? 0u : (g.epi.add_mode == 1u ? g.n : 1u) * g.m * 2u);
    const v2s lo2 = {(short)q88::act_lo(g.epi.act), (short)q88::act_lo(g.epi.act)};
    const v2s hi2 = {(short)q88::act_hi(g.epi.act), (short)q88::act_hi(g.epi.act)};
    // this lane's limb products of its row i, mod 2^32
    auto finish = [&](uint32_t i, uint32_t (&v)[2][8]) {
#pragma unroll
        for (uint32_t e = 0; e < 2; ++e)
#pragma unroll
            for (uint32_t t = 0; t < 8; ++t) {
                const uint32_t ee = 2 * e + t / 4, q = t % 4;
                v[e][t] = ((((uint32_t)hh[q][i][ee] << 8) + (uint32_t)mid[q][i][ee]) << 8) + (uint32_t)ll[q][i][ee];
            }
    };
    // The Add's operands of every output, ahead of the first store: a load between two
    // stores would wait for the store before it
    v4u addv[2][2];
#pragma unroll
    for (uint32_t i = 0; i < 2; ++i)
#pragma unroll
        for (uint32_t e = 0; e < 2; ++e) addv[i][e] = v4u{0u, 0u, 0u, 0u};
    if (g.epi.add_mode && !g.ws) {
#pragma unroll
        for (uint32_t i = 0; i < 2; ++i)
#pragma unroll
            for (uint32_t e = 0; e < 2; ++e) {
                const uint32_t r = row0 + wr * 32u + i * 16u + er16, col = col0 + wc * 64u + (4u * e + ekg) * 8u;
                const uint32_t cnt = r < g.n && col < g.m ? min(8u, g.m - col) : 0u;
                addv[i][e] = load_head(er, ((g.epi.add_mode == 1u ? r * g.m : 0u) + col) * 2u, cnt);
            }
    }
    // k groups: group kz finishes row tile kz, the other one hands it its sums
    uint32_t* ex = reinterpret_cast<uint32_t*>(lds_all);
    if constexpr (KS == 2) {
        static_assert(16 * kT * 4 <= 2 * kStage, "a group's sums fit the limb buffers");
#pragma unroll
        for (uint32_t i = 0; i < 2; ++i) {
            if (i == kz) continue;
            uint32_t v[2][8];
            finish(i, v);
#pragma unroll
            for (uint32_t q = 0; q < 16; ++q) ex[(i * 16u + q) * kT + et] = v[q / 8][q % 8];
        }
        __syncthreads();
    }
#pragma unroll
    for (uint32_t i = 0; i < 2; ++i) {
        if (KS == 2 && i != kz) continue;
        uint32_t sums[2][8];
        finish(i, sums);
        if constexpr (KS == 2) {
#pragma unroll
            for (uint32_t q = 0; q < 16; ++q) sums[q / 8][q % 8] += ex[(i * 16u + q) * kT + et];
        }
        const uint32_t rl = wr * 32u + i * 16u + er16, r = row0 + rl;
        // the limb sums of B lack 128 per staged k, which over the products' Kp
        // positions is the identity's last term; one step of zeros more was staged by
        // each group
        const uint32_t rterm = 128u * rsum[rl] + KS * 16384u * 64u;
#pragma unroll
        for (uint32_t e = 0; e < 2; ++e) {
            const uint32_t cl = wc * 64u + (4u * e + ekg) * 8u, col = col0 + cl;
            const v4u x0 = *reinterpret_cast<const v4u*>(&csum[cl]), x1 = *reinterpret_cast<const v4u*>(&csum[cl + 4]);
            uint32_t v[8];
#pragma unroll
            for (uint32_t t = 0; t < 8; ++t)
                v[t] = sums[e][t] + 128u * (t < 4 ? x0[t] : x1[t - 4]) + rterm;
            if (r >= g.n || col >= g.m) continue;
            if (g.ws) {
                uint32_t* p = g.ws + ((uint64_t)split * g.n + r) * g.ws_ld + col;
                *reinterpret_cast<v4u*>(p) = v4u{v[0], v[1], v[2], v[3]};
                *reinterpret_cast<v4u*>(p + 4) = v4u{v[4], v[5], v[6], v[7]};
                continue;
            }
            const uint32_t cnt = min(8u, g.m - col), off = (r * g.m + col) * 2u;
            const v4u add = addv[i][e];
            v4u out;
#pragma unroll
            for (uint32_t q = 0; q < 4; ++q) {
                const uint32_t av = add[q];
                v2s o = __builtin_bit_cast(v2s, __builtin_amdgcn_cvt_pk_i16((int32_t)v[2 * q] >> 8, (int32_t)v[2 * q + 1] >> 8));
                o = __builtin_elementwise_add_sat(o, __builtin_bit_cast(v2s, av));
                out[q] = __builtin_bit_cast(uint32_t, __builtin_elementwise_min(__builtin_elementwise_max(o, lo2), hi2));
            }
            store_head(cr, off, cnt, out);
        }
    }
}

template <uint32_t WR, uint32_t WC, uint32_t KS, bool ALDS>
int launch(RgArgs& g, uint32_t z, hipStream_t s) {
    g.tx = (g.m + 64u * WC - 1) / (64u * WC);
    g.ty = (g.n + 32u * WR - 1) / (32u * WR);
    const dim3 grid(g.tx * g.ty, z), block(WR * WC * KS * 64);
    if (g.k % 8 == 0) hipLaunchKernelGGL((gemm_rg<WR, WC, KS, ALDS, true>), grid, block, 0, s, g);
    else hipLaunchKernelGGL((gemm_rg<WR, WC, KS, ALDS, false>), grid, block, 0, s, g);
    return cm_check_launch("gemm_rg");
}

}  // namespace

// How many k splits (at most `splits`, what the workspace holds) of a product of
// nk steps pay here: as many as the blocks leave CUs for, when they take at least
// eight steps off a block (each costs ~0.7 us, the reduce launch 3.5-6): 2000 x 1283
// x 1001 (256 blocks) 23.8 us unsplit, 29.5 in two; 128 x 4096 x 4096 (64 blocks)
// 29.1 / 23.1 / 20.8 / 22.6 us in 2 / 3 / 4 / 8.
uint32_t cm_gemm_rg_splits(uint32_t n, uint32_t m, uint32_t nk, uint32_t splits) {
    const uint64_t blocks = (uint64_t)((n + 127) / 128) * ((m + 63) / 64);
    const uint32_t sp = (uint32_t)std::min<uint64_t>(splits, cm_cu_count() / blocks);
    return sp > 1 && nk - nk / sp >= 8 ? sp : 1u;
}

// One batch launch (z batches, or z splits of one product into `ws`) on this
// path, or 1 when it does not take the shape: at least 4 columns and 8 k (16 when
// not a multiple of 8), at most 32768 k, and each batch's operands below 2 GiB.
int cm_gemm_rg_launch(const int16_t* a, const int16_t* b, int16_t* c, uint32_t n, uint32_t k, uint32_t m,
                      uint64_t a_bs, uint64_t b_bs, uint64_t c_bs, uint32_t z, uint32_t* ws, uint32_t steps,
                      uint32_t ws_ld, const EpiArgs& epi, hipStream_t s) {
    const uint64_t lim = 1ull << 30;
    if ((k % 8 ? k < 16 : k < 8) || k > 32768 || m < 4 || (uint64_t)n * (k + 320) >= lim || (uint64_t)(k + 320) * m >= lim ||
        (uint64_t)n * m >= lim || z > 65535u)
        return 1;
    RgArgs g{};
    g.a = a; g.b = b; g.c = c; g.ws = ws; g.epi = epi;
    g.n = n; g.k = k; g.m = m; g.nk = (k + 63) / 64;
    g.a_bs = a_bs; g.b_bs = b_bs; g.c_bs = c_bs;
    g.steps = ws ? steps : g.nk;
    g.ws_ld = ws_ld;
    // 128 x 128 tiles with A in LDS once they fill the chip twice over several
    // steps: 4096 x 4095 x 4095 293 us against 389, 32 x 1023 x 1023 x 1023 214 against
    // 248, but 20.3 against 19.0 at 3000 x 100 x 3000.  64 x 64 tiles on two k groups
    // where 128 x 64 ones are half empty (n at most 64: 16 x 1280 x 20000 20.1
    // against 23.0) or leave CUs idle in a launch that does not split (11 x 448 x 2944
    // x 56 25.7 against 35.4, 12 x 197 x 197 x 64 6.8 against 8.0; with splits they
    // lose: 128 x 4096 x 4096 23.2 against 20.8).
    const uint64_t cus = cm_cu_count();
    auto tiles = [&](uint64_t bm, uint64_t bn) { return z * ((n + bm - 1) / bm) * ((m + bn - 1) / bn); };
    if (!ws && g.nk >= 4 && tiles(128, 128) >= 2 * cus) return launch<4, 2, 1, true>(g, z, s);
    if (n <= 64 || (!ws && z > 1 && tiles(128, 64) < cus)) return launch<2, 1, 2, false>(g, z, s);
    return launch<4, 1, 1, false>(g, z, s);
}
