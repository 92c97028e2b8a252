// skinny_any.hip -- a few token rows (2 <= M <= 32) on bf16 matrix cores for
// any width and both stored formats: y[m, r] = sum_k x[m, k] * w(r, k).
//
// skinny.hip is instantiated for the Qwen3 widths; every other width, and
// every bf16 weight, ran a kernel that holds four token rows at a time and
// decodes (or loads) the weights again for the next four, by VALU. Here K is a
// run-time value and the weights are read once:
//  * a chunk is 128 elements of K. MFMA operand B is 16 weight rows x 32 K,
//    operand A 16 tokens x 32 K (V_MFMA_F32_16X16X32_BF16), four MFMAs a chunk.
//    MXFP4: lane group g (= lane / 16) holds block g of the chunk and MFMA t
//    takes elements [32 g + 8 t, +8); bf16: MFMA t takes [32 t + 8 g, +8), so
//    that a load instruction reads 64 contiguous bytes of each row. A and B
//    share the order, so it changes nothing in the result;
//  * a workgroup of TW waves takes T 16-row tiles at a time and walks K in
//    slices of TW x NC chunks, NC adjacent ones a wave: the slice's activation
//    fragments are loaded (f32: split into three bf16 terms, exact products;
//    a wave that met tiny or non-finite ones does the set again with care for them)
//    once and used for all T tiles, whose sums stay in registers. The next
//    slice's (or the next tiles') weights of tile t are loaded as soon as tile
//    t's are used, so T tiles (or two slices) are in flight;
//  * with two or four MXFP4 chunks a wave, a load instruction takes 16 / NC rows
//    of 64 NC contiguous bytes (whole cache lines, half the requests) and the
//    wave's own LDS stage turns them into the MFMA layout;
//  * where one slice is all of K, the activations stay for every tile;
//  * the TW partial tiles are summed through LDS at the end, in wave order;
//  * loads go through buffer resources: token rows >= M, weight rows >= N and
//    elements past K read as zeros without touching memory. Scale bytes are
//    read as the aligned word that holds a lane's byte (rows of any width
//    start at any byte), with byte 0 past K.
// Bound by HBM on long weights, by the launch and one load latency on short
// ones.
#include <type_traits>

#include "mx4_device.h"
#include "mx4_kernels.h"

namespace mx4 {

namespace {

constexpr int kStreamed = 2;                  // weights are used once: do not keep them in the caches
constexpr int TW = 8;                         // waves per workgroup
typedef double f64x4 __attribute__((ext_vector_type(4)));

// The weights of a launch: up to four of one width sharing x, weight s owning
// the 16-row tiles [first[s], first[s + 1]).
struct Weights {
    const uint8_t* data[4];    // packed codes, or bf16 values
    const uint8_t* scales[4];  // null for bf16
    float* y[4];
    uint32_t n[4];
    uint32_t first[4];
    uint32_t count;
};
struct Pick {
    const uint8_t* data;
    const uint8_t* scales;
    float* y;
    uint32_t n, first;
};
__device__ __forceinline__ Pick pick(const Weights& g, uint32_t tile) {
    Pick p{g.data[0], g.scales[0], g.y[0], g.n[0], 0u};
#pragma unroll
    for (int q = 1; q < 4; ++q) {
        const bool in = q < (int)g.count && tile >= g.first[q];
        p.data = in ? g.data[q] : p.data;
        p.scales = in ? g.scales[q] : p.scales;
        p.y = in ? g.y[q] : p.y;
        p.n = in ? g.n[q] : p.n;
        p.first = in ? g.first[q] : p.first;
    }
    return p;
}

// Wait states between the last MFMAs and reads of their sums (see gemm.hip).
__device__ __forceinline__ void mfma_drain() {
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("s_nop 7\n\ts_nop 7\n\ts_nop 7");
    __builtin_amdgcn_sched_barrier(0);
}

// Between one lane's LDS writes and another's reads in the same wave: the LDS
// serves a wave's accesses in order, so this only keeps the compiler, which
// sees each lane's own addresses, from turning the order round.
__device__ __forceinline__ void wave_handover() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// FP4: weights are MXFP4 (else bf16). MT: token tiles of 16. NC: chunks per
// wave and slice. T: 16-row weight tiles per workgroup at a time.
// Workgroups with blockIdx.y = 1 take the token rows from 16 MT on.
template <bool FP4, bool XBF16, int MT, int NC, int T>
__global__ __launch_bounds__(64 * TW) void skinny_any_kernel(const void* __restrict__ x, uint32_t m_all, uint32_t k,
                                                             uint32_t tiles, uint32_t grid, const Weights g) {
    const uint32_t tok0 = blockIdx.y * 16 * MT;
    const uint32_t m = m_all - tok0 < 16u * MT ? m_all - tok0 : 16u * MT;
    constexpr int WL = FP4 ? 1 : 4;            // 16-byte weight loads per chunk
    constexpr int XP = XBF16 ? 1 : 3;          // bf16 terms of an activation
    constexpr uint32_t XB = XBF16 ? 2 : 4;
    constexpr int D = T > 1 ? T : 2;           // weight buffers
    const uint32_t lane = threadIdx.x % 64, col = lane % 16, gq = lane / 16;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
    const uint32_t nblk = k / 32, row_bytes = FP4 ? k / 2 : k * 2;
    const uint32_t slices = (k + 128 * TW * NC - 1) / (128 * TW * NC);
    const __amdgpu_buffer_rsrc_t xr = rsrc(static_cast<const uint8_t*>(x) + (size_t)tok0 * k * XB, m * k * XB);

    // element of K that lane group gq's piece t of chunk c starts with
    auto element = [](uint32_t gq, uint32_t c, int t) { return 128 * c + (FP4 ? 32 * gq + 8 * t : 32 * t + 8 * gq); };

    struct Unit {
        u32x4 w[NC][WL];
        uint32_t s[FP4 ? NC : 1];
        uint32_t shift;
    };
    // TRANS: load i holds rows (16 / NC) i + j, block b of the wave's run at lane
    // (4 NC) j + b. Its stage slot is turned so that the writes and the reads
    // of any 8 consecutive lanes fall in 8 different 16-byte bank groups.
    constexpr bool TRANS = FP4 && (NC == 2 || NC == 4);
    constexpr uint32_t RPL = 16 / NC, BPR = 4 * NC;  // rows per load, blocks per row of the run
    __shared__ u32x4 stage[TRANS ? TW : 1][TRANS ? 64 * NC : 1];
    auto slot = [&](uint32_t i, uint32_t j, uint32_t b) -> uint32_t {
        if constexpr (NC == 4) return 64 * i + 16 * j + ((b + 2 * j + (i & 1)) & 15);
        else return 64 * i + 8 * j + ((b + (j & ~1u)) & 7);
    };
    // the weights of slice `sl` of tile `tile` (tiles and slices past the end: zeros)
    auto load_at = [&](uint32_t lane, uint32_t tile, uint32_t sl, Unit& u) {
        const uint32_t col = lane % 16, gq = lane / 16;
        const bool valid = tile < tiles;
        const Pick p = pick(g, tile);
        const uint32_t row0 = valid ? (tile - p.first) * 16 : 0;
        const uint32_t rows = valid ? (p.n - row0 < 16u ? p.n - row0 : 16u) : 0;
        const __amdgpu_buffer_rsrc_t wr = rsrc(p.data + (size_t)row0 * row_bytes, rows * row_bytes);
        const uint32_t c0 = (sl * TW + wave) * NC;
        if constexpr (FP4) {
            // rows start at any byte, 16 of them at a multiple of 16: the tile
            // is as far off a word as the whole array
            const uint32_t mis = (uint32_t)((uintptr_t)p.scales & 3);
            const __amdgpu_buffer_rsrc_t sr =
                rsrc(p.scales - mis + (size_t)row0 * nblk, rows ? (rows * nblk + mis + 3) & ~3u : 0u);
            const uint32_t at = col * nblk + 4 * c0 + gq + mis;
            u.shift = 8 * (at & 3);
#pragma unroll
            for (int q = 0; q < NC; ++q) {
                const uint32_t blk = 4 * (c0 + q) + gq;
                u.s[q] = __builtin_amdgcn_raw_buffer_load_b32(sr, blk < nblk ? (at & ~3u) + 4 * q : kPastEnd, 0, 0);
                const uint32_t row = TRANS ? RPL * q + lane / BPR : col;
                const uint32_t wblk = TRANS ? 4 * c0 + lane % BPR : blk;
                u.w[q][0] = __builtin_amdgcn_raw_buffer_load_b128(wr, wblk < nblk ? row * row_bytes + 16 * wblk : kPastEnd, 0,
                                                                  kStreamed);
            }
        } else {
#pragma unroll
            for (int q = 0; q < NC; ++q)
#pragma unroll
                for (int t = 0; t < WL; ++t) {
                    const uint32_t e = element(gq, c0 + q, t);
                    u.w[q][t] = __builtin_amdgcn_raw_buffer_load_b128(wr, e < k ? col * row_bytes + 2 * e : kPastEnd, 0,
                                                                      kStreamed);
                }
        }
        __builtin_amdgcn_sched_barrier(0);
    };
    auto load = [&](uint32_t tile, uint32_t sl, Unit& u) { load_at(lane, tile, sl, u); };

    // Activation fragments of the slice in use. f32: `raw` holds the next
    // slice's values on their way from memory (4096 x 4096 at 7 rows 10.6 -> 9.6
    // us); bf16 fragments are loaded as they are used (a second set of registers
    // for them spills: 18432 x 3264 at 7 rows 13.0 -> 18.4 us).
    constexpr int H = XBF16 ? 1 : 2;  // 16-byte loads per piece
    u32x4 raw[XBF16 ? 1 : NC][4][MT][H];
    bf16x8 xa[NC][4][MT][XP];
    auto x_piece_at = [&](uint32_t lane, uint32_t sl, int q, int t, int j, u32x4 (&out)[H]) {
        const uint32_t col = lane % 16, e = element(lane / 16, (sl * TW + wave) * NC + q, t);
        const uint32_t off = e < k ? ((16 * j + col) * k + e) * XB : kPastEnd;
#pragma unroll
        for (int h = 0; h < H; ++h) out[h] = __builtin_amdgcn_raw_buffer_load_b128(xr, off + 16 * h, 0, 0);
    };
    auto x_piece = [&](uint32_t sl, int q, int t, int j, u32x4 (&out)[H]) { x_piece_at(lane, sl, q, t, j, out); };
    auto issue_x = [&](uint32_t sl) {
        if constexpr (XBF16) return;
#pragma unroll
        for (int q = 0; q < NC; ++q)
#pragma unroll
            for (int t = 0; t < 4; ++t)
#pragma unroll
                for (int j = 0; j < MT; ++j) x_piece(sl, q, t, j, raw[XBF16 ? 0 : q][t][j]);
        __builtin_amdgcn_sched_barrier(0);
    };
    bool care = false;  // f32: this lane's activations of some slice are not plain
    auto settle_x = [&](uint32_t sl) {
        float most = 0.0f;
#pragma unroll
        for (int q = 0; q < NC; ++q)
#pragma unroll
            for (int t = 0; t < 4; ++t)
#pragma unroll
                for (int j = 0; j < MT; ++j) {
                    if constexpr (XBF16) {
                        u32x4 v[H];
                        x_piece(sl, q, t, j, v);
                        xa[q][t][j][0] = __builtin_bit_cast(bf16x8, v[0]);
                    } else {
                        split3_finite(raw[q][t][j][0], raw[q][t][j][1], xa[q][t][j][0], xa[q][t][j][1], xa[q][t][j][2]);
                        take_most(raw[q][t][j][0], most);
                        take_most(raw[q][t][j][1], most);
                    }
                }
        if constexpr (!XBF16) {
            // (zeros for what is done again anyway: without this branch the compiler
            // takes more registers than there are with four tiles of bf16 weights)
            if (__any(!plain(most))) {
                care = true;
#pragma unroll
                for (int q = 0; q < NC; ++q)
#pragma unroll
                    for (int t = 0; t < 4; ++t)
#pragma unroll
                        for (int j = 0; j < MT; ++j)
#pragma unroll
                            for (int p = 0; p < 3; ++p) xa[q][t][j][p] = __builtin_bit_cast(bf16x8, u32x4{0u, 0u, 0u, 0u});
            }
        }
    };

    // A slice's chain of MFMAs starts from zero and is added to the running
    // sums in 64 bits when the tile's next one starts: as far from the exact sum
    // as the kernel that ran these shapes before, whose lanes each summed K / 64
    // products (one chain over K and a sum of the waves in 32 bits: up to 1.4
    // times as far).
    f64x4 sums[T][MT];
    f32x4 acc[T][MT], fine[XBF16 ? 1 : T][MT];  // fine: the mid and lo terms' products (f32 x)
    auto zero = [&]() {
#pragma unroll
        for (int t = 0; t < T; ++t)
#pragma unroll
            for (int j = 0; j < MT; ++j) {
                sums[t][j] = f64x4{0.0, 0.0, 0.0, 0.0};
                acc[t][j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
                if constexpr (!XBF16) fine[t][j] = acc[t][j];
            }
    };
    auto fold = [&](int i) {
#pragma unroll
        for (int j = 0; j < MT; ++j) {
            f32x4 v = acc[i][j];
            if constexpr (!XBF16) {
                v += fine[i][j];
                fine[i][j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
            }
#pragma unroll
            for (int r = 0; r < 4; ++r) sums[i][j][r] += (double)v[r];
            acc[i][j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
        }
    };
    auto compute = [&](const Unit& u, uint32_t sl, int i) {
        const uint32_t c0 = (sl * TW + wave) * NC;
        if (sl > 0) fold(i);
        u32x4 w4[FP4 ? NC : 1];
        if constexpr (TRANS) {
#pragma unroll
            for (int q = 0; q < NC; ++q) stage[wave][slot(q, lane / BPR, lane % BPR)] = u.w[q][0];
            wave_handover();
#pragma unroll
            for (int q = 0; q < NC; ++q) w4[q] = stage[wave][slot(col / RPL, col % RPL, 4 * q + gq)];
            wave_handover();
        } else if constexpr (FP4) {
#pragma unroll
            for (int q = 0; q < NC; ++q) w4[q] = u.w[q][0];
        }
#pragma unroll
        for (int q = 0; q < NC; ++q) {
            if (q == 2) {
                mfma_drain();
                fold(i);
            }
            float sc = 0.0f;
            if constexpr (FP4) {
                const uint32_t byte = 4 * (c0 + q) + gq < nblk ? (u.s[q] >> u.shift) & 0xffu : 0u;
                sc = __uint_as_float(byte << 23);
            }
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                bf16x8 b;
                if constexpr (FP4) b = decode8(w4[q][t], sc);
                else b = __builtin_bit_cast(bf16x8, u.w[q][t]);
#pragma unroll
                for (int j = 0; j < MT; ++j) {
                    acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(xa[q][t][j][0], b, acc[i][j], 0, 0, 0);
                    if constexpr (!XBF16) {
                        fine[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(xa[q][t][j][1], b, fine[i][j], 0, 0, 0);
                        fine[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(xa[q][t][j][2], b, fine[i][j], 0, 0, 0);
                    }
                }
            }
        }
    };

    uint32_t nan_tokens = 0;  // bf16 weights: token rows with a NaN among the wave's activations
    // the wave's sums of tile i of the set again, with the careful split and the
    // tiny lanes' values in a pass of their own; everything is loaded again
    auto again_with_care = [&](uint32_t tile, int i) {
        if constexpr (!XBF16) {
            static_assert(NC == 1 && MT == 1, "one chunk and one token tile of f32 activations");
            // (opaque: what follows from it is computed here, not kept in registers
            // over the sets)
            uint32_t lane = threadIdx.x % 64;
            asm volatile("" : "+v"(lane));
            sums[i][0] = f64x4{0.0, 0.0, 0.0, 0.0};
#pragma unroll 1
            for (uint32_t sl = 0; sl < slices; ++sl) {
                Unit u;
                load_at(lane, tile, sl, u);
                float most = 0.0f, sc = 0.0f;
#pragma unroll 1
                for (int t = 0; t < 4; ++t) {
                    u32x4 v[H];
                    x_piece_at(lane, sl, 0, t, 0, v);
                    take_most(v[0], most);
                    take_most(v[1], most);
                }
                if constexpr (!FP4) {
                    const uint64_t nan = __ballot(most != most);
                    nan_tokens |= (uint32_t)(nan | nan >> 16 | nan >> 32 | nan >> 48) & 0xffffu;
                }
                if constexpr (FP4) {
                    const uint32_t blk = 4 * (sl * TW + wave) + lane / 16;
                    sc = __uint_as_float((blk < nblk ? (u.s[0] >> u.shift) & 0xffu : 0u) << 23);
                }
#pragma unroll 1
                for (int pass = 0; pass < 2; ++pass) {
                    f32x4 whole{0.0f, 0.0f, 0.0f, 0.0f}, parts = whole;
#pragma unroll
                    for (int t = 0; t < 4; ++t) {
                        bf16x8 b, hi, mid, lo;
                        if constexpr (FP4) b = decode8(u.w[0][0][t], sc);
                        else b = __builtin_bit_cast(bf16x8, u.w[0][t]);
                        u32x4 v[H];
                        x_piece_at(lane, sl, 0, t, 0, v);
                        split3_pass(pass, all_tiny(most), v[0], v[1], hi, mid, lo);
                        whole = __builtin_amdgcn_mfma_f32_16x16x32_bf16(hi, b, whole, 0, 0, 0);
                        parts = __builtin_amdgcn_mfma_f32_16x16x32_bf16(mid, b, parts, 0, 0, 0);
                        parts = __builtin_amdgcn_mfma_f32_16x16x32_bf16(lo, b, parts, 0, 0, 0);
                        __builtin_amdgcn_sched_barrier(0);  // one piece's registers at a time
                    }
                    mfma_drain();
                    whole += parts;
#pragma unroll
                    for (int r = 0; r < 4; ++r) sums[i][0][r] += (double)whole[r] * (pass ? kTinyDown : 1.0);
                }
            }
        }
    };

    __shared__ f32x4 red[TW][T * MT][64];
    constexpr bool INF = !FP4 && !XBF16;  // inf weights want a second look (inf_and_no_nan)
    __shared__ uint32_t nans[INF ? TW : 1];
    // tile i of the set that starts at `tile`; sets follow one another `grid` T tiles apart
    Unit u[D];
    uint32_t tile = blockIdx.x;
    if (tile >= tiles) return;
    issue_x(0);
    if constexpr (T > 1) {
#pragma unroll
        for (int i = 0; i < T; ++i) load(tile + i * grid, 0, u[i]);
    } else {
        load(tile, 0, u[0]);
    }
    bool again = false;
    // the activations of slice sl into use, the next slice's on their way (one slice: they stay)
    auto turn_x = [&](uint32_t sl) {
        if (slices == 1 && again) return;
        settle_x(sl);
        if (slices > 1) issue_x(sl + 1 == slices ? 0 : sl + 1);
    };
    for (;;) {
        const uint32_t next = tile + grid * T;
        zero();
        if constexpr (T > 1) {
            for (uint32_t sl = 0; sl < slices; ++sl) {
                turn_x(sl);
                const bool end = sl + 1 == slices;
#pragma unroll
                for (int i = 0; i < T; ++i) {
                    compute(u[i], sl, i);
                    load((end ? next : tile) + i * grid, end ? 0 : sl + 1, u[i]);
                }
            }
        } else {
            // one tile a workgroup and no other set (the launcher sees to it):
            // slice sl in buffer sl % 2, the other one a slice ahead
            for (uint32_t sl = 0; sl < slices; sl += 2) {
                load(tile, sl + 1, u[1]);
                turn_x(sl);
                compute(u[0], sl, 0);
                if (sl + 1 == slices) break;
                load(tile, sl + 2, u[0]);
                turn_x(sl + 1);
                compute(u[1], sl + 1, 0);
            }
        }
        mfma_drain();
#pragma unroll
        for (int i = 0; i < T; ++i) fold(i);
        if constexpr (!XBF16) {
            if (__any(care)) {
#pragma unroll
                for (int i = 0; i < T; ++i) again_with_care(tile + i * grid, i);
                // what the next set has a use for, loaded again rather than kept meanwhile
                if constexpr (T > 1) {
                    issue_x(0);
                    if (slices == 1) settle_x(0);
#pragma unroll
                    for (int i = 0; i < T; ++i) load(next + i * grid, 0, u[i]);
                }
            }
        }
        if (again) __syncthreads();  // the last set's sums have been read
#pragma unroll
        for (int i = 0; i < T; ++i)
#pragma unroll
            for (int j = 0; j < MT; ++j) {
                if constexpr (INF)
                    if (i == 0 && lane == 0) nans[wave] = nan_tokens;
                red[wave][i * MT + j][lane] = __builtin_convertvector(sums[i][j], f32x4);
            }
        __syncthreads();
        for (uint32_t v = wave; v < (uint32_t)(T * MT); v += TW) {
            const uint32_t at = tile + (v / MT) * grid, j = v % MT;
            f64x4 sum = __builtin_convertvector(red[0][v][lane], f64x4);
#pragma unroll
            for (int w = 1; w < TW; ++w) sum += __builtin_convertvector(red[w][v][lane], f64x4);
            if (at < tiles) {
                const Pick p = pick(g, at);
                const uint32_t row = (at - p.first) * 16 + col;
                if (row < p.n) {
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        const uint32_t tok = 16 * j + 4 * gq + r;
                        if (tok < m) p.y[(size_t)(tok0 + tok) * p.n + row] = (float)sum[r];
                    }
                }
                if constexpr (INF) {
                    uint32_t nan_rows = 0;  // token rows with a NaN; weight rows with one beside those
#pragma unroll
                    for (int w = 0; w < TW; ++w) nan_rows |= nans[w];
                    uint64_t doubt = 0;
#pragma unroll
                    for (int r = 0; r < 4; ++r)
                        doubt |= __ballot(sum[r] != sum[r] && row < p.n && 4 * gq + r < m && !((nan_rows >> (4 * gq + r)) & 1));
                    doubt = (doubt | doubt >> 16 | doubt >> 32 | doubt >> 48) & 0xffffu;
                    if (doubt) wait_vm<0>();  // the sums below overwrite
                    uint32_t lane = threadIdx.x % 64;
                    asm volatile("" : "+v"(lane));  // (its addresses are not for keeping, see above)
                    while (doubt) {
                        const uint32_t rr = (at - p.first) * 16 + (uint32_t)__builtin_ctzll(doubt);
                        doubt &= doubt - 1;
                        const uint16_t* wrow = reinterpret_cast<const uint16_t*>(p.data) + (size_t)rr * k;
                        if (!inf_and_no_nan(wrow, k, lane)) continue;
                        for (uint32_t tok = 0; tok < m; ++tok) {
                            if ((nan_rows >> tok) & 1) continue;
                            const float whole = dot_whole(static_cast<const float*>(x) + (size_t)(tok0 + tok) * k, wrow, k, lane);
                            if (lane == 0) p.y[(size_t)(tok0 + tok) * p.n + rr] = whole;
                        }
                    }
                }
            }
        }
        if (T == 1 || next >= tiles) break;
        tile = next;
        again = true;
    }
}

template <bool FP4, bool XBF16, int MT, int NC, int T>
hipError_t go(const Weights& g, const void* x, uint32_t m, uint32_t k, uint32_t tiles, uint32_t grid, hipStream_t s) {
    hipLaunchKernelGGL((skinny_any_kernel<FP4, XBF16, MT, NC, T>), dim3(grid, (m + 16 * MT - 1) / (16 * MT)),
                       dim3(64 * TW), 0, s, x, m, k, tiles, grid, g);
    return hipGetLastError();
}

// Tiles a workgroup takes at a time (t), chunks a wave takes of a slice, and the
// workgroups of the launch. From a sweep of the three on MI355X over weights of
// 14 to 9500 tiles, K = 896 .. 12288, 7 and 29 rows (cold weights, recorded
// passes); times in us, before: the kernel that takes four rows at a time.
//  * one tile a workgroup while the CUs are not full, then two, then four, one
//    workgroup per CU that walks several sets (100000 x 1600 at 7 rows 27-29
//    against 38 with two per CU);
//  * bf16 x: as many chunks as make one slice of K, up to four (two for two
//    token tiles, or with one tile a workgroup): 18432 x 3264 at 7 rows 13.7
//    with four, 16.2 with two, 18.8 with one; 1600 x 1600 at 7 rows 4.1 (before
//    20), 8576 x 1600 at 29 rows 9.7;
//  * bf16 weights (four times the loads): one chunk, and one tile a workgroup
//    up to four workgroups per CU: 12288 x 2048 at 7 rows 16.0 against 20.9
//    with two of each; two of each with two token tiles;
//  * f32 x: one (two spill), the second token tile counted as tiles of their
//    own: 1600 x 1600 at 7 rows 6.1, 18432 x 3264 at 7 / 29 rows 29 / 59.
struct Shape {
    uint32_t t, chunks, grid;
};
Shape shape_rule(bool fp4, bool x_bf16, uint32_t m, uint32_t k, uint32_t tiles, int cus) {
    const uint32_t nc = (uint32_t)(cus > 0 ? cus : 256);
    const uint32_t mt = x_bf16 && m > 16 ? 2 : 1;               // token tiles of a workgroup
    const uint32_t per_wave = ((k + 127) / 128 + TW - 1) / TW;  // chunks of a row for each wave
    // the activations of a slice take 16 MT XP NC registers, the weights 5 NC (FP4) or 16 NC a tile
    const uint32_t most = x_bf16 ? 4 / mt : 1;
    const uint32_t halves = (m + 16 * mt - 1) / (16 * mt);
    uint32_t t = tiles * halves <= nc ? 1 : tiles * halves <= 2 * nc ? 2 : 4;
    uint32_t chunks = per_wave >= 3 ? 4u : per_wave;
    if (chunks > most) chunks = most;
    if (chunks > 2 && t == 1) chunks = 2;
    if (!fp4 && x_bf16) {
        chunks = mt == 2 && t > 1 ? chunks : 1;
        t = mt == 1 && tiles <= 4 * nc ? 1 : t > 2 ? 2 : t;
    }
    if (chunks == 4 || (chunks == 2 && mt == 1)) t = t > 2 ? 2 : t;
    uint32_t grid = (tiles + t - 1) / t;
    if (t > 1 && grid > (x_bf16 ? nc : 2 * nc)) grid = x_bf16 ? nc : 2 * nc;
    // the same number of sets for every workgroup
    const uint32_t sets = (tiles + grid * t - 1) / (grid * t);
    return {t, chunks, (tiles + sets * t - 1) / (sets * t)};
}

template <bool FP4, bool XBF16, int MT>
hipError_t go_shape(const Weights& g, const void* x, uint32_t m, uint32_t k, uint32_t tiles, int cus, hipStream_t s) {
    constexpr int kMost = XBF16 ? 4 / MT : 1;
    const Shape r = shape_rule(FP4, XBF16, m, k, tiles, cus);
#define MX4_SKINNY_ANY(C, T_)                                            \
    if constexpr (C <= kMost && (FP4 || !XBF16 || (T_ <= 2 && C == 1) || (T_ == 2 && MT == 2)) && \
                  (C == 1 || T_ <= 2 || MT == 2))                         \
        if (r.chunks == C && r.t == T_) return go<FP4, XBF16, MT, C, T_>(g, x, m, k, tiles, r.grid, s);
    MX4_SKINNY_ANY(1, 1) MX4_SKINNY_ANY(1, 2) MX4_SKINNY_ANY(1, 4) MX4_SKINNY_ANY(2, 1) MX4_SKINNY_ANY(2, 2)
    MX4_SKINNY_ANY(2, 4) MX4_SKINNY_ANY(4, 2)
#undef MX4_SKINNY_ANY
    return hipErrorNotSupported;
}

}  // namespace

bool skinny_any_supported(uint32_t m, uint32_t k, bool fp4) {
    // whole 16-byte pieces of every row; 32-bit offsets within a tile and within x
    return m >= 2 && m <= 32 && k >= 32 && k % (fp4 ? 32 : 8) == 0 && k <= (1u << 20);
}

// The tuned widths (skinny.hip). f32 activations: skinny.hip splits a token's
// values again for every 16-row tile, here once for up to four of them (us,
// skinny.hip / here: 8B gate|up at 7 / 29 rows 48 / 110 against 35 / 65, o 10.4 /
// 20.4 against 9.8 / 17.1, down 25.9 / 63 against 23 / 48; 4096 x 6144 at 6 rows
// 12.1 / 11.4, 4096 x 8192 15.9 / 15.0; 1.7B gate|up 17.1 / 37.3 against 11.1 /
// 24.8). At K = 2048 with a tile or less a CU and one token tile it stays ahead
// (1.7B q|k|v 6.3 against 6.7 us). It would at 11 to 16 rows there too (4096 rows,
// K = 4096 / 6144 / 8192 / 12288 at 16 rows 14.3 / 21.4 / 24.7 / 39.4 against 16.3 /
// 23.3 / 28.5 / 42.4), but its sums are two to four times as far from the exact
// ones (2.2e-7 against 0.5 to 1.1e-7), so those stay here. bf16 ones: up to 16 rows
// it stays ahead everywhere (its activations are resident too); beyond, where its
// weights are too long for one tile a workgroup and too short for the tile ring, it
// loads them for every tile (1.7B gate|up 20.8 against 10.5 us, 8B q|k|v 20.9
// against 13.2; with fewer tiles 11.2 against 11.4, with the ring 26.7 against 32).
bool skinny_any_faster(uint32_t m, uint32_t k, uint32_t tiles, bool x_bf16, int cus) {
    const uint32_t nc = (uint32_t)(cus > 0 ? cus : 256);
    if (!x_bf16) return m > 16 || k != 2048 || tiles > nc;
    // (the ring: two tiles for each of the workgroups of eight waves a CU)
    const uint32_t ring = k == 2048 ? 4 * nc : 2 * nc;
    return m > 16 && (k == 2048 || k == 4096) && tiles > nc && tiles < ring;
}

uint32_t mx4_rule_skinny_any(bool fp4, bool x_bf16, uint32_t m, uint32_t k, uint32_t tiles, int cus) {
    const Shape r = shape_rule(fp4, x_bf16, m, k, tiles, cus);
    return r.chunks * 10 + r.t;
}

hipError_t launch_skinny_any(const GemvArgs& a, const uint16_t* const* bf16, int cus) {
    const bool fp4 = bf16 == nullptr;
    if (!skinny_any_supported(a.m, a.k, fp4)) return hipErrorNotSupported;
    Weights g{};
    g.count = a.group ? a.group->count : 1;
    if (g.count < 1 || g.count > 4) return hipErrorNotSupported;
    uint32_t tiles = 0;
    for (uint32_t s = 0; s < g.count; ++s) {
        g.data[s] = !fp4 ? reinterpret_cast<const uint8_t*>(bf16[s]) : a.group ? a.group->packed[s] : a.packed;
        g.scales[s] = !fp4 ? nullptr : a.group ? a.group->scales[s] : a.scales;
        g.y[s] = a.group ? a.group->y[s] : a.y;
        g.n[s] = a.group ? a.group->n[s] : a.n;
        if (g.n[s] == 0) return hipErrorNotSupported;
        g.first[s] = tiles;
        tiles += (g.n[s] + 15) / 16;
    }
    // More than 16 rows: bf16 x takes both token tiles with one read of the
    // weights; f32 x (three terms a value) has no registers for two, and runs
    // the tiles as two halves of the grid.
#define MX4_SKINNY_ANY(F)                                                                        \
    if (!a.x_bf16) return go_shape<F, false, 1>(g, a.x, a.m, a.k, tiles, cus, a.stream);         \
    return a.m <= 16 ? go_shape<F, true, 1>(g, a.x, a.m, a.k, tiles, cus, a.stream)              \
                     : go_shape<F, true, 2>(g, a.x, a.m, a.k, tiles, cus, a.stream);
    if (fp4) {
        MX4_SKINNY_ANY(true)
    } else {
        MX4_SKINNY_ANY(false)
    }
#undef MX4_SKINNY_ANY
}

}  // namespace mx4
