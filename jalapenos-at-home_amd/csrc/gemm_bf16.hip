// gemm_bf16.hip -- bf16 weights, more than 32 token rows, on matrix cores:
// y[m, r] = sum_k x[m, k] * w(r, k), the `None` arm of engine/src/lib.rs:255.
//
// A workgroup owns a BM x BN output tile (token rows x weight rows) and walks K
// in stages of 64: BM rows of activations (128 bytes of bf16 or 256 of f32) and
// BN weight rows (128 bytes) come straight into LDS (direct-to-LDS buffer
// loads) into a ring of D stages, D - 1 in flight while one is computed, one
// barrier per stage. A wave owns TM x TN 32x32 tiles of
// V_MFMA_F32_32X32X16_BF16: lane l (row l % 32, half h = l / 32) takes elements
// [32 h, 32 h + 32) of the stage, MFMA s elements [32 h + 8 s, +8), for both
// operands alike. f32 activations are three bf16 terms (exact products; a workgroup that
// met tiny or non-finite ones does its work again with care for them).
//
// Two stages are summed from zero and added to the running sums in 64 bits: as
// far from the exact sum as the kernel that ran these shapes before, whose
// lanes each summed K / 64 products, or nearer (one chain over all of K would
// be up to twice as far, four stages 1.1 times at K = 1600).
//
// Bound by the LDS reads and the 64-bit additions beside the MFMAs (adding every
// four stages instead of two is 7% faster): a layer of hidden size 4096 at 300
// rows of bf16 4.85 -> 0.295 ms, 394 TFLOP/s; by VALU it was 23 TFLOP/s at every
// size.
//
// Loads go through buffer resources: token rows >= M, weight rows >= N and
// elements past K read as zeros without touching memory.
#include <type_traits>

#include "mx4_device.h"
#include "mx4_kernels.h"

namespace mx4 {

namespace {

constexpr int kBK = 64;                     // K elements per stage
constexpr int kFold = 2;                    // stages summed in 32 bits
// The weights of a launch: up to four of one width sharing x, weight s owning
// the column tiles [tile0[s], tile0[s + 1]) of the grid.
struct Weights {
    const uint16_t* w[4];
    float* y[4];
    uint32_t n[4];
    uint32_t tile0[4];
    uint32_t count;
};

// LDS rows of 16-byte slots, written by direct-to-LDS loads (lane l at slot
// base + l), so the layout is chosen by which chunk a lane loads: chunk c of
// row r sits in slot c ^ (r / 2 % 8) of a 128-byte row, c ^ (r % 16) of a
// 256-byte one. The 16 lanes that read one logical chunk at a time then fall in
// 16 different 16-byte bank groups.
template <int CPR>
__device__ __forceinline__ uint32_t turned(uint32_t row, uint32_t c) {
    return CPR == 8 ? c ^ ((row >> 1) & 7) : c ^ (row & 15);
}

// Wait states after the last MFMAs before their sums are read (see gemm.hip).
__device__ __forceinline__ void mfma_drain() {
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("s_nop 7\n\ts_nop 7\n\ts_nop 7\n\ts_nop 7");
    __builtin_amdgcn_sched_barrier(0);
}

template <bool XBF16, int WM, int WN, int TM, int TN>
struct Geometry {
    static constexpr int NW = WM * WN, NT = 64 * NW;
    static constexpr int BM = 32 * TM * WM, BN = 32 * TN * WN;
    static constexpr int XB = XBF16 ? 2 : 4;
    static constexpr int A_CPR = kBK * XB / 16, B_CPR = kBK * 2 / 16;  // 16-byte chunks per row
    static constexpr int A_BYTES = BM * A_CPR * 16, B_BYTES = BN * B_CPR * 16, STAGE = A_BYTES + B_BYTES;
    static constexpr int A_INSTR = BM * A_CPR / NT, B_INSTR = BN * B_CPR / NT, LPS = A_INSTR + B_INSTR;
    static constexpr int D = STAGE * 4 <= 160 * 1024 ? 4 : STAGE * 3 <= 160 * 1024 ? 3 : 2;
    static_assert(BM * A_CPR % NT == 0 && BN * B_CPR % NT == 0, "stage split");
    static_assert(D * STAGE <= 160 * 1024 && (D - 2) * LPS <= 63, "ring");
};

template <bool XBF16, int WM, int WN, int TM, int TN>
__global__ __launch_bounds__(64 * WM * WN) void gemm_bf16_kernel(const void* __restrict__ x, uint32_t m, uint32_t k,
                                                                 uint32_t tiles_n, uint32_t tiles, uint32_t kslice,
                                                                 float* __restrict__ part, const Weights g) {
    using G = Geometry<XBF16, WM, WN, TM, TN>;
    constexpr int D = G::D;
    __shared__ __attribute__((aligned(16))) uint8_t lds[D * G::STAGE];
    const uint32_t lane = threadIdx.x % 64, h = lane / 32, r32 = lane % 32;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
    const uint32_t wm = wave / WN, wn = wave % WN;
    // K split: workgroup b takes tile b % tiles over K slice b / tiles and
    // writes its partial tile to part[slice][m][n]
    const uint32_t slice = blockIdx.x / tiles, tile = blockIdx.x % tiles;
    uint32_t tn = tile % tiles_n, t0 = 0, n = g.n[0];
    const uint16_t* w = g.w[0];
    float* y = g.y[0];
#pragma unroll
    for (int q = 1; q < 4; ++q) {
        const bool in = q < (int)g.count && tn >= g.tile0[q];
        w = in ? g.w[q] : w;
        y = in ? g.y[q] : y;
        n = in ? g.n[q] : n;
        t0 = in ? g.tile0[q] : t0;
    }
    const uint32_t row0 = tile / tiles_n * G::BM, col0 = (tn - t0) * G::BN;
    const uint32_t k0 = slice * kslice, klen = k - k0 < kslice ? k - k0 : kslice;
    const uint32_t stages = (klen + kBK - 1) / kBK;
    if (part) y = part + (size_t)slice * m * n;
    const __amdgpu_buffer_rsrc_t xr = rsrc(x, m * k * G::XB);
    const __amdgpu_buffer_rsrc_t wr = rsrc(w, n * k * 2);

    // this lane's offsets (stage 0) and first element within the stage
    uint32_t a_off[G::A_INSTR], a_col[G::A_INSTR], b_off[G::B_INSTR], b_col[G::B_INSTR];
#pragma unroll
    for (int q = 0; q < G::A_INSTR; ++q) {
        const uint32_t p = (q * G::NW + wave) * 64 + lane, row = p / G::A_CPR, c = turned<G::A_CPR>(row, p % G::A_CPR);
        a_off[q] = ((row0 + row) * k + k0) * G::XB + c * 16;
        a_col[q] = c * 16 / G::XB;
    }
#pragma unroll
    for (int q = 0; q < G::B_INSTR; ++q) {
        const uint32_t p = (q * G::NW + wave) * 64 + lane, row = p / G::B_CPR, c = turned<G::B_CPR>(row, p % G::B_CPR);
        b_off[q] = ((col0 + row) * k + k0) * 2 + c * 16;
        b_col[q] = c * 8;
    }
    auto issue = [&](uint32_t st) {
        uint8_t* base = lds + st % D * G::STAGE;
        const uint32_t live = klen - st * kBK;
#pragma unroll
        for (int q = 0; q < G::A_INSTR; ++q)
            load_lds16(xr, (lds_ptr)(base + (q * G::NW + wave) * 1024),
                       a_col[q] < live ? a_off[q] + st * kBK * G::XB : kPastEnd);
#pragma unroll
        for (int q = 0; q < G::B_INSTR; ++q)
            load_lds16(wr, (lds_ptr)(base + G::A_BYTES + (q * G::NW + wave) * 1024),
                       b_col[q] < live ? b_off[q] + st * kBK * 2 : kPastEnd);
    };

    f64x16 acc[TM][TN];
    f32x16 sum[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                acc[i][j][r] = 0.0;
                sum[i][j][r] = 0.0f;
            }
    // the stages' sums so far into the running ones
    auto fold = [&](double scale) {
        mfma_drain();
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j)
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    acc[i][j][r] += (double)sum[i][j][r] * scale;
                    sum[i][j][r] = 0.0f;
                }
    };
    auto w_piece = [&](const uint8_t* base, int j, uint32_t s) {
        const uint32_t r = (wn * TN + j) * 32 + r32;
        return __builtin_bit_cast(bf16x8, *reinterpret_cast<const u32x4*>(
                                              base + G::A_BYTES + (r * G::B_CPR + turned<G::B_CPR>(r, 4 * h + s)) * 16));
    };
    // f32 x: eight values
    auto x_piece = [&](const uint8_t* base, int i, uint32_t s, u32x4& v0, u32x4& v1) {
        const uint32_t r = (wm * TM + i) * 32 + r32;
        const uint8_t* ap = base + r * G::A_CPR * 16;
        v0 = *reinterpret_cast<const u32x4*>(ap + turned<G::A_CPR>(r, 8 * h + 2 * s) * 16);
        v1 = *reinterpret_cast<const u32x4*>(ap + turned<G::A_CPR>(r, 8 * h + 2 * s + 1) * 16);
    };
    auto mac3 = [&](int i, int j, bf16x8 hi, bf16x8 mid, bf16x8 lo, bf16x8 b) {
        sum[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(lo, b, sum[i][j], 0, 0, 0);
        sum[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(mid, b, sum[i][j], 0, 0, 0);
        sum[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(hi, b, sum[i][j], 0, 0, 0);
    };
    bool care = false;  // f32 x: this lane's activations of some stage are not plain
    auto compute = [&](uint32_t st) {
        const uint8_t* base = lds + st % D * G::STAGE;
        float most[TM];
#pragma unroll
        for (int i = 0; i < TM; ++i) most[i] = 0.0f;
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            bf16x8 b[TN];
#pragma unroll
            for (int j = 0; j < TN; ++j) b[j] = w_piece(base, j, s);
#pragma unroll
            for (int i = 0; i < TM; ++i) {
                if constexpr (XBF16) {
                    const uint32_t r = (wm * TM + i) * 32 + r32;
                    const bf16x8 a = __builtin_bit_cast(bf16x8, *reinterpret_cast<const u32x4*>(
                                                                    base + r * G::A_CPR * 16 + turned<G::A_CPR>(r, 4 * h + s) * 16));
#pragma unroll
                    for (int j = 0; j < TN; ++j)
                        sum[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b[j], sum[i][j], 0, 0, 0);
                } else {
                    u32x4 v0, v1;
                    x_piece(base, i, s, v0, v1);
                    bf16x8 hi, mid, lo;
                    split3_finite(v0, v1, hi, mid, lo);
                    take_most(v0, most[i]);
                    take_most(v1, most[i]);
#pragma unroll
                    for (int j = 0; j < TN; ++j) mac3(i, j, hi, mid, lo, b[j]);
                }
            }
        }
        if constexpr (!XBF16) {
#pragma unroll
            for (int i = 0; i < TM; ++i) care |= !plain(most[i]);
        }
        if (st % kFold == kFold - 1 || st + 1 == stages) fold(1.0);
    };
    // the same with the careful split, the tiny lanes' values in a pass of their own
    bool nan_lane[TM];  // this lane's token row holds a NaN
#pragma unroll
    for (int i = 0; i < TM; ++i) nan_lane[i] = false;
    auto compute_careful = [&](uint32_t st) {
        const uint8_t* base = lds + st % D * G::STAGE;
        float most[TM];
#pragma unroll
        for (int i = 0; i < TM; ++i) {
            most[i] = 0.0f;
#pragma unroll 1
            for (uint32_t s = 0; s < 4; ++s) {
                u32x4 v0, v1;
                x_piece(base, i, s, v0, v1);
                take_most(v0, most[i]);
                take_most(v1, most[i]);
            }
            nan_lane[i] |= most[i] != most[i];
        }
#pragma unroll
        for (int pass = 0; pass < 2; ++pass) {
#pragma unroll 1
            for (uint32_t s = 0; s < 4; ++s)
#pragma unroll
                for (int i = 0; i < TM; ++i) {
                    u32x4 v0, v1;
                    x_piece(base, i, s, v0, v1);
                    bf16x8 hi, mid, lo;
                    split3_pass(pass, all_tiny(most[i]), v0, v1, hi, mid, lo);
#pragma unroll
                    for (int j = 0; j < TN; ++j) mac3(i, j, hi, mid, lo, w_piece(base, j, s));
                }
            fold(pass ? kTinyDown : 1.0);
        }
    };
    auto walk = [&](auto&& step) {
#pragma unroll
        for (int p = 0; p < D - 1; ++p)
            if ((uint32_t)p < stages) issue(p);
        for (uint32_t st = 0; st < stages; ++st) {
            const uint32_t ahead = stages - 1 - st;  // stages issued after st, at most D - 2
            if (ahead >= (uint32_t)(D - 2)) wait_vm<(D - 2) * G::LPS>();
            else if (D > 3 && ahead == 1) wait_vm<(D > 3 ? 1 : 0) * G::LPS>();
            else wait_vm<0>();
            lds_barrier();
            if (st + D - 1 < stages) issue(st + D - 1);
            step(st);
        }
    };
    walk(compute);
    if constexpr (!XBF16) {
        if (workgroup_any<G::NW>(__any(care), reinterpret_cast<uint32_t*>(lds), wave)) {
#pragma unroll
            for (int i = 0; i < TM; ++i)
#pragma unroll
                for (int j = 0; j < TN; ++j)
#pragma unroll
                    for (int r = 0; r < 16; ++r) {
                        acc[i][j][r] = 0.0;
                        sum[i][j][r] = 0.0f;
                    }
            walk(compute_careful);
        }
    }

    // lane l holds column l % 32 of a 32x32 tile and, in register r, row
    // 8 (r / 4) + 4 (l / 32) + r % 4
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) {
            const uint32_t tile_row = row0 + (wm * TM + i) * 32, tile_col = col0 + (wn * TN + j) * 32, col = tile_col + r32;
            uint64_t nan_rows = 0, doubt = 0;  // NaN activations by token row; columns with a NaN beside those
            if constexpr (!XBF16) {
                nan_rows = __ballot(nan_lane[i]);
                nan_rows |= nan_rows >> 32;
            }
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const uint32_t at = 8 * (r / 4) + 4 * h + r % 4, row = tile_row + at;
                const float v = (float)acc[i][j][r];
                if constexpr (!XBF16) doubt |= __ballot(v != v && row < m && col < n && !((nan_rows >> at) & 1));
                if (row < m && col < n) y[(size_t)row * n + col] = v;
            }
            if constexpr (!XBF16) {
                doubt = (doubt | doubt >> 32) & 0xffffffffu;
                if (doubt) wait_vm<0>();  // the sums below overwrite
                while (doubt) {
                    const uint32_t cc = tile_col + (uint32_t)__builtin_ctzll(doubt);
                    doubt &= doubt - 1;
                    const uint16_t* wrow = w + (size_t)cc * k + k0;
                    if (!inf_and_no_nan(wrow, klen, lane)) continue;
                    for (uint32_t at = 0; at < 32 && tile_row + at < m; ++at) {
                        if ((nan_rows >> at) & 1) continue;
                        const float p = dot_whole(static_cast<const float*>(x) + (size_t)(tile_row + at) * k + k0, wrow, klen, lane);
                        if (lane == 0) y[(size_t)(tile_row + at) * n + cc] = p;
                    }
                }
            }
        }
}

uint32_t slice_k(uint32_t k, uint32_t ks) {
    const uint32_t stages = (k + kBK - 1) / kBK;
    return (stages + ks - 1) / ks * kBK;
}

template <bool XBF16, int WM, int WN, int TM, int TN>
hipError_t go(Weights g, const void* x, uint32_t m, uint32_t k, uint32_t ks, float* part, hipStream_t s) {
    using G = Geometry<XBF16, WM, WN, TM, TN>;
    uint32_t tiles_n = 0;
    for (uint32_t q = 0; q < g.count; ++q) {
        g.tile0[q] = tiles_n;
        tiles_n += (g.n[q] + G::BN - 1) / G::BN;
    }
    const uint32_t tiles = tiles_n * ((m + G::BM - 1) / G::BM);
    hipLaunchKernelGGL((gemm_bf16_kernel<XBF16, WM, WN, TM, TN>), dim3(tiles * ks), dim3(G::NT), 0, s, x, m, k, tiles_n,
                       tiles, slice_k(k, ks), ks > 1 ? part : nullptr, g);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess || ks == 1) return e;
    return launch_split_sum(part, ks, m * g.n[0], g.y[0], s);
}

// The tile and K split (1 to 4 slices, one weight) with the least estimated
// time: whole rounds of workgroups, one per CU, times the tile's time for its
// stages, plus the pass that adds the slices. Stage times from a sweep of nine
// wave arrangements and 1-4 slices on the 1.7B and 8B shapes and 1600 x 4288 at
// 40 .. 800 rows on MI355X (cold weights). Eight waves, two a SIMD, so that one
// adds its 64-bit sums while the other multiplies: 128 x 128 with four waves of
// 2 x 2 tiles ran 24576 x 4096 at 200 rows in 152 us, eight of 1 x 2 in 94, 128 x
// 256 with eight of 2 x 2 in 80; 2048 x 6144 at 200 rows 18.9 us (128 x 64, four
// slices).
struct Plan {
    int tile = 0;
    uint32_t ks = 1;
    double us = 0.0;
};
Plan plan(const uint32_t* n, uint32_t count, uint32_t m, uint32_t k, bool x_bf16, int cus, uint64_t part_bytes) {
    struct Cand { int bm, bn; double stage_us; };
    const Cand cands[] = {{128, 128, x_bf16 ? 0.65 : 1.64}, {64, 128, x_bf16 ? 0.43 : 1.2}, {128, 64, x_bf16 ? 0.41 : 1.28},
                          {64, 64, x_bf16 ? 0.42 : 1.04}, {128, 256, 1.19}};
    const uint64_t nc = (uint64_t)(cus > 0 ? cus : 256);
    Plan best;
    for (int c = 0; c < 5; ++c) {
        // (128 x 256 of f32 activations does not fit the registers; 64 x 64 of bf16
        // ones takes as long as 128 x 64)
        if (c == (x_bf16 ? 3 : 4)) continue;
        uint64_t tiles = 0;
        for (uint32_t q = 0; q < count; ++q) tiles += (n[q] + cands[c].bn - 1) / cands[c].bn;
        tiles *= (m + cands[c].bm - 1) / cands[c].bm;
        for (uint32_t ks = 1; ks <= 4; ++ks) {
            if (ks > 1 && (count > 1 || (uint64_t)(ks - 1) * slice_k(k, ks) >= k || (uint64_t)ks * m * n[0] * 4 > part_bytes))
                continue;
            const double t = (double)((tiles * ks + nc - 1) / nc) * (4.0 + cands[c].stage_us * (slice_k(k, ks) / kBK)) +
                             (ks > 1 ? 3.0 + 4.0 * (ks + 1) * m * n[0] / 4e6 : 0.0);
            if (best.us == 0.0 || t < best.us) best = {c, ks, t};
        }
    }
    return best;
}

template <bool XBF16>
hipError_t dispatch(const Weights& g, const void* x, uint32_t m, uint32_t k, int cus, float* part, uint64_t part_bytes,
                    hipStream_t s) {
    const Plan p = plan(g.n, g.count, m, k, XBF16, cus, part ? part_bytes : 0);
    if constexpr (XBF16) {
        if (p.tile == 4) return go<XBF16, 2, 4, 2, 2>(g, x, m, k, p.ks, part, s);
    } else {
        if (p.tile == 3) return go<XBF16, 2, 2, 1, 1>(g, x, m, k, p.ks, part, s);
    }
    if (p.tile == 0) return go<XBF16, 4, 2, 1, 2>(g, x, m, k, p.ks, part, s);
    if (p.tile == 1) return go<XBF16, 2, 4, 1, 1>(g, x, m, k, p.ks, part, s);
    return go<XBF16, 4, 2, 1, 1>(g, x, m, k, p.ks, part, s);
}

}  // namespace

// Estimated time of a launch (measured ones are about 1.2 us shorter: small
// weights at 33 .. 300 rows 1024 x 64 10.7 / 9.2 f32, 12288 x 64 27.2 / 26.5 bf16).
double gemm_bf16_us(const uint32_t* n, uint32_t count, uint32_t m, uint32_t k, bool x_bf16, int cus, uint64_t part_bytes) {
    return plan(n, count, m, k, x_bf16, cus, part_bytes).us - 1.2;
}

uint32_t mx4_rule_gemm_bf16(const uint32_t* n, uint32_t count, uint32_t m, uint32_t k, bool x_bf16, int cus, uint64_t part_bytes) {
    static const uint32_t tiles[] = {42120, 24110, 42110, 22110, 24220};
    const Plan p = plan(n, count, m, k, x_bf16, cus, part_bytes);
    return tiles[p.tile] + p.ks;
}

bool gemm_bf16_supported(uint32_t m, uint32_t n, uint32_t k, bool x_bf16) {
    // rows of whole 16-byte pieces; 32-bit offsets over the padded operands
    return m >= 1 && n >= 1 && k >= 8 && k % 8 == 0 && (uint64_t)(m + 128) * k * (x_bf16 ? 2 : 4) < (1ull << 31) &&
           (uint64_t)(n + 128) * k * 2 < (1ull << 31);
}

hipError_t launch_gemm_bf16(const uint16_t* const* w, float* const* y, const uint32_t* n, uint32_t count, const void* x,
                            bool x_bf16, uint32_t m, uint32_t k, int cus, float* part, uint64_t part_bytes,
                            hipStream_t s) {
    if (count < 1 || count > 4) return hipErrorNotSupported;
    Weights g{};
    g.count = count;
    for (uint32_t q = 0; q < count; ++q) {
        if (!gemm_bf16_supported(m, n[q], k, x_bf16)) return hipErrorNotSupported;
        g.w[q] = w[q];
        g.y[q] = y[q];
        g.n[q] = n[q];
    }
    return x_bf16 ? dispatch<true>(g, x, m, k, cus, part, part_bytes, s)
                  : dispatch<false>(g, x, m, k, cus, part, part_bytes, s);
}

}  // namespace mx4
