// gemm.hip -- exact matrix-core GEMM for more than 32 token rows:
// y[m, r] = sum_k x[m, k] * w(r, k), f32 accumulation of exact products.
//
// The reference sends every projection with M > 32 token rows (and, through
// its per-call bridge, every M > 1) to a tiled FP32 GEMM that decodes the
// weights into threadgroup tiles (project_mxfp4, engine/src/matmul.metal:65-97;
// dispatch engine/src/gpu.rs:510-514, engine/src/metal.m:103-105). Here the
// multiply-accumulate runs on gfx950's V_MFMA_F32_32X32X16_BF16 while the
// weights stay 4-bit in HBM, in the stored row-major layout:
//  * a workgroup owns a BM x BN output tile (token rows x weight rows) and
//    walks K in stages of 128. Each stage's activations (BM rows x 256 bytes
//    of bf16) and weights (BN rows x 64 packed bytes + 4 scale bytes) are
//    loaded straight into LDS (direct-to-LDS buffer loads, whole rows per
//    instruction) into a ring of D stages, D - 1 of them in flight while one
//    is computed (one barrier per stage);
//  * a wave owns TM x TN 32x32 MFMA tiles. Lane l (row l % 32, half h = l / 32)
//    takes elements [64h, 64h + 64) of the stage for both operands; k-step s
//    of the stage contracts elements [64h + 8s, +8). The contraction is over
//    K, so this order, shared by A and B, changes nothing in the result;
//  * a weight lane reads its row's 32 packed bytes once per stage and decodes
//    8 elements per k-step with the hardware E2M1 converter, the E8M0 scale
//    folded in (exact in bf16 for scale bytes 2..252, which the dispatcher
//    guarantees);
//  * bf16 activations are exact operands; f32 activations are split into three
//    bf16 terms hi + mid + lo (24 significant bits), three MFMAs each, so every
//    product is exact and only the f32 summation order differs from the
//    reference's sequential loop (engine/src/lib.rs:240-266);
//  * every global load goes through a buffer resource: token rows >= M and
//    weight rows >= N read as zeros without touching memory, and their outputs
//    are not stored;
//  * widths that are no whole number of stages (any K % 32 == 0: the ANY
//    instances) zero the last stage's columns past K the same way, and take
//    the scale bytes, whose rows then start at any byte, as aligned words. With
//    f32 activations they look at each stage's largest magnitude a lane, and a
//    workgroup that met tiny or non-finite ones walks K again with care for them
//    (mx4_device.h): 1600 x 1600 at 77 rows 18.8 -> 13.5 us against a check (for
//    non-finite ones only) at every eight values, other shapes within 3%.
#include <algorithm>
#include <type_traits>
#include "mx4_device.h"
#include "mx4_kernels.h"

namespace mx4 {

namespace {

// Wait states after the last MFMAs before their accumulators are read (the
// compiler has placed such reads after a branch without them on gfx950).
__device__ __forceinline__ void mfma_drain() {
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("s_nop 7\n\ts_nop 7\n\ts_nop 7\n\ts_nop 7");
    __builtin_amdgcn_sched_barrier(0);
}

constexpr int kBK = 128;  // K elements per stage

// Stage layout in LDS (no padding): activations BM rows x A_CPR 16-byte slots,
// packed weights BN rows x 4 slots, then BN scale words. Slots are written by
// direct-to-LDS buffer loads, lane l of a load instruction at slot base + l,
// so the layout is chosen through which global chunk each lane loads: chunk c
// of row r sits in slot c ^ (r % 16) of an activation row and c ^ ((r / 4) % 4)
// of a weight row. The MFMA-operand reads (32 rows, one logical chunk) then
// spread over all LDS banks.
//
// ANY: K is any multiple of 32. A stage's four scale bytes of a row then lie
// anywhere in two aligned words, so the stage holds both and the reader shifts.
template <bool XBF16, int WM, int WN, int TM, int TN, int D, bool ANY>
struct Geometry {
    static constexpr int NW = WM * WN, NT = 64 * NW;
    static constexpr int BM = 32 * TM * WM, BN = 32 * TN * WN;
    static constexpr int XB = XBF16 ? 2 : 4;              // bytes per activation element
    static constexpr int A_CPR = kBK * XB / 16;           // 16-byte chunks per activation row
    static constexpr int A_BYTES = BM * A_CPR * 16, B_BYTES = BN * 4 * 16, S_BYTES = BN * (ANY ? 8 : 4);
    static constexpr int STAGE = A_BYTES + B_BYTES + S_BYTES;
    static constexpr int A_INSTR = BM * A_CPR / NT;       // 64-lane loads per wave per stage
    static constexpr int B_INSTR = BN * 4 / NT;
    static constexpr int S_WORDS = BN / NW * (ANY ? 2 : 1);  // scale words per wave per stage
    static constexpr int S_INSTR = (S_WORDS + 63) / 64;
    static constexpr int LPS = A_INSTR + B_INSTR + S_INSTR;  // vector memory instructions per stage
    static_assert(BM * A_CPR % NT == 0 && BN * 4 % NT == 0 && BN % NW == 0, "stage split");
    static_assert(D >= 2 && D <= 4 && (D - 2) * LPS <= 63, "vmcnt range");
    static_assert(D * STAGE <= 160 * 1024, "the stages must fit the LDS");
};

// Up to four weights of one width sharing x (q|k|v, gate|up at more than 32
// token rows) in one launch: weight s owns the column tiles [tile0[s],
// tile0[s + 1]) of the grid; a workgroup picks its weight with uniform
// selects. Passed as the trailing argument, so the leading scalars keep
// arriving preloaded; NoGemmSegs stands there for one weight. A K split's
// partials of weight s are m x n[s] floats from m x row0[s] on in each slice's
// m x rows.
struct NoGemmSegs {};
struct GemmSegs {
    const uint8_t* packed[4];
    const uint8_t* scales[4];
    float* y[4];
    uint32_t n[4];
    uint32_t tile0[4];
    uint32_t row0[4];
    uint32_t rows;
    uint32_t count;
};

template <bool XBF16, int WM, int WN, int TM, int TN, int D, bool ANY = false, class SG = NoGemmSegs>
__global__ __launch_bounds__(64 * WM * WN) void gemm_exact_kernel(const uint8_t* __restrict__ packed,
                                                                  const uint8_t* __restrict__ scales,
                                                                  const void* __restrict__ x, float* __restrict__ y,
                                                                  uint32_t m, uint32_t n, uint32_t k,
                                                                  uint32_t tiles_n, uint32_t tiles,
                                                                  uint32_t kslice, float* __restrict__ part,
                                                                  const SG group) {
    using G = Geometry<XBF16, WM, WN, TM, TN, D, ANY>;
    __shared__ __attribute__((aligned(16))) uint8_t lds[D * G::STAGE];
    const uint32_t lane = threadIdx.x % 64, h = lane / 32, r32 = lane % 32;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
    const uint32_t wm = wave / WN, wn = wave % WN;
    // K split: workgroup b takes tile b % tiles over K slice b / tiles and
    // writes its partial tile to part[slice][m][n] (summed afterwards in slice order)
    const uint32_t slice = blockIdx.x / tiles, tile = blockIdx.x % tiles;
    uint32_t tn = tile % tiles_n;
    const uint32_t tm = tile / tiles_n;
    uint32_t prow0 = 0, prows = n;  // a K split's partials
    if constexpr (std::is_same_v<SG, GemmSegs>) {
        // the column tile's weight, and the tile within it
        uint32_t t0 = 0;
        packed = group.packed[0];
        scales = group.scales[0];
        y = group.y[0];
        n = group.n[0];
        prows = group.rows;
#pragma unroll
        for (int q = 1; q < 4; ++q) {
            const bool in = q < (int)group.count && tn >= group.tile0[q];
            packed = in ? group.packed[q] : packed;
            scales = in ? group.scales[q] : scales;
            y = in ? group.y[q] : y;
            n = in ? group.n[q] : n;
            t0 = in ? group.tile0[q] : t0;
            prow0 = in ? group.row0[q] : prow0;
        }
        tn -= t0;
    }
    const uint32_t row0 = tm * G::BM, col0 = tn * G::BN;
    // (ANY: the last slice may be shorter, and its last stage ragged)
    const uint32_t k0 = slice * kslice;
    const uint32_t klen = ANY ? (k - k0 < kslice ? k - k0 : kslice) : kslice;
    const uint32_t stages = ANY ? (klen + kBK - 1) / kBK : klen / kBK;
    if (part) y = part + (size_t)slice * m * prows + (size_t)m * prow0;

    const __amdgpu_buffer_rsrc_t xr = rsrc(x, m * k * G::XB);
    const __amdgpu_buffer_rsrc_t pr = rsrc(packed, n * (k / 2));
    // ANY: whole aligned words from the one that holds the first scale byte on
    const uint32_t mis = ANY ? (uint32_t)((uintptr_t)scales & 3) : 0u;
    const __amdgpu_buffer_rsrc_t sr =
        ANY ? rsrc(scales - mis, (n * (k / 32) + mis + 3) & ~3u) : rsrc(scales, n * (k / 32));

    using Acc = std::conditional_t<ANY, f64x16, f32x16>;
    Acc acc[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[i][j][r] = 0;

    uint32_t s_shift[TN];  // ANY: bits before row j's first scale byte in its two words
#pragma unroll
    for (int j = 0; j < TN; ++j)
        s_shift[j] = 8 * (((col0 + (wn * TN + j) * 32 + r32) * (k / 32) + k0 / 32 + mis) & 3);
    bool care = false;  // ANY, f32 x: this lane's activations of some stage are not plain
    auto compute = [&](uint32_t st, uint32_t slot) {
        const uint8_t* base = lds + slot * G::STAGE;
        // ANY: blocks past K keep scale byte 0 (what follows the row in memory is no scale of theirs)
        const uint32_t live = klen - st * kBK;
        const uint32_t s_mask = ANY && live < (uint32_t)kBK ? (1u << (live / 4)) - 1 : ~0u;
        u32x4 wq[TN][2];
        uint32_t sw[TN];
#pragma unroll
        for (int j = 0; j < TN; ++j) {
            const uint32_t r = (wn * TN + j) * 32 + r32, f = (r >> 2) & 3;
            const uint8_t* bp = base + G::A_BYTES + r * 64;
            wq[j][0] = *reinterpret_cast<const u32x4*>(bp + ((2 * h) ^ f) * 16);
            wq[j][1] = *reinterpret_cast<const u32x4*>(bp + ((2 * h + 1) ^ f) * 16);
            if constexpr (ANY) {
                const uint2 two = *reinterpret_cast<const uint2*>(base + G::A_BYTES + G::B_BYTES + r * 8);
                sw[j] = __builtin_amdgcn_alignbit(two.y, two.x, s_shift[j]) & s_mask;
            } else {
                sw[j] = *reinterpret_cast<const uint32_t*>(base + G::A_BYTES + G::B_BYTES + r * 4);
            }
        }
        // ANY: a stage is summed from zero and the stages are summed in 64
        // bits. The kernel that ran these widths before summed K / 64 products
        // per lane and the lanes in a tree; one MFMA chain over all of K is
        // 1.2 to 2.5 times as far from the exact sum as that (K = 1600, bf16 /
        // f32 x: 1.5e-7 / 3.9e-7 against 6e-8 / 1.6e-7 relative), stages added
        // in 32 bits up to 1.7 times, in 64 bits no further. (The chains of
        // the other instances are what those widths always had.)
        f32x16 sum[ANY ? TM : 1][ANY ? TN : 1];
        float most[TM];
#pragma unroll
        for (int i = 0; i < TM; ++i) most[i] = 0.0f;
        auto mac = [&](int s, int i, int j, bf16x8 a, bf16x8 w, bool first) {
            if constexpr (ANY) {
                f32x16 c;
#pragma unroll
                for (int r = 0; r < 16; ++r) c[r] = 0.0f;
                if (!(s == 0 && first)) c = sum[i][j];
                sum[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, w, c, 0, 0, 0);
            } else {
                acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, w, acc[i][j], 0, 0, 0);
            }
        };
#pragma unroll
        for (int s = 0; s < 8; ++s) {
            bf16x8 b[TN];
#pragma unroll
            for (int j = 0; j < TN; ++j) {
                // elements [64h + 8s, +8) lie in block 2h + s / 4 of the stage
                const uint32_t sb = (sw[j] >> (8 * (2 * h + s / 4))) & 0xffu;
                b[j] = decode8(wq[j][s / 4][s % 4], __uint_as_float(sb << 23));
            }
#pragma unroll
            for (int i = 0; i < TM; ++i) {
                const uint32_t r = (wm * TM + i) * 32 + r32, sw16 = r % 16;
                const uint8_t* ap = base + r * (G::A_CPR * 16);
                if constexpr (XBF16) {
                    const uint32_t c = (8 * h + s) ^ sw16;
                    const bf16x8 a = __builtin_bit_cast(bf16x8, *reinterpret_cast<const u32x4*>(ap + c * 16));
#pragma unroll
                    for (int j = 0; j < TN; ++j) mac(s, i, j, a, b[j], true);
                } else {
                    const uint32_t c0 = (16 * h + 2 * s) ^ sw16, c1 = (16 * h + 2 * s + 1) ^ sw16;
                    const u32x4 v0 = *reinterpret_cast<const u32x4*>(ap + c0 * 16);
                    const u32x4 v1 = *reinterpret_cast<const u32x4*>(ap + c1 * 16);
                    bf16x8 hi, mid, lo;
                    if constexpr (ANY) {
                        split3_finite(v0, v1, hi, mid, lo);
                        take_most(v0, most[i]);
                        take_most(v1, most[i]);
                        // several tiles a wave: each split between the MFMAs of the one
                        // before it, and no further ahead (a branch keeps the compiler
                        // to that in fewer registers than a scheduling barrier)
                        if constexpr (TM * TN > 1)
                            if (__any(!(most[i] < __builtin_inff())))
                                hi = mid = lo = __builtin_bit_cast(bf16x8, u32x4{0u, 0u, 0u, 0u});
                    } else {
                        split3x8(v0, v1, hi, mid, lo);
                    }
#pragma unroll
                    for (int j = 0; j < TN; ++j) {
                        mac(s, i, j, hi, b[j], true);
                        mac(s, i, j, mid, b[j], false);
                        mac(s, i, j, lo, b[j], false);
                    }
                }
            }
        }
        if constexpr (ANY) {
            mfma_drain();
#pragma unroll
            for (int i = 0; i < TM; ++i)
#pragma unroll
                for (int j = 0; j < TN; ++j)
#pragma unroll
                    for (int r = 0; r < 16; ++r) acc[i][j][r] += (double)sum[i][j][r];
            if constexpr (!XBF16) {
#pragma unroll
                for (int i = 0; i < TM; ++i) care |= !plain(most[i]);
            }
        }
    };
    // the same with the careful split, the tiny lanes' values in a pass of their own
    auto compute_careful = [&](uint32_t st, uint32_t slot) {
        const uint8_t* base = lds + slot * G::STAGE;
        const uint32_t live = klen - st * kBK;
        const uint32_t s_mask = live < (uint32_t)kBK ? (1u << (live / 4)) - 1 : ~0u;
        auto x_piece = [&](int i, uint32_t s, u32x4& v0, u32x4& v1) {
            const uint32_t r = (wm * TM + i) * 32 + r32, c = 16 * h + 2 * s;
            const uint8_t* ap = base + r * (G::A_CPR * 16);
            v0 = *reinterpret_cast<const u32x4*>(ap + (c ^ (r % 16)) * 16);
            v1 = *reinterpret_cast<const u32x4*>(ap + ((c + 1) ^ (r % 16)) * 16);
        };
        float most[TM];
#pragma unroll
        for (int i = 0; i < TM; ++i) {
            most[i] = 0.0f;
#pragma unroll 1
            for (uint32_t s = 0; s < 8; ++s) {
                u32x4 v0, v1;
                x_piece(i, s, v0, v1);
                take_most(v0, most[i]);
                take_most(v1, most[i]);
            }
        }
#pragma unroll 1
        for (int pass = 0; pass < 2; ++pass) {
            f32x16 sum[TM][TN];
#pragma unroll
            for (int i = 0; i < TM; ++i)
#pragma unroll
                for (int j = 0; j < TN; ++j)
#pragma unroll
                    for (int r = 0; r < 16; ++r) sum[i][j][r] = 0.0f;
#pragma unroll 1
            for (uint32_t s = 0; s < 8; ++s) {
                bf16x8 b[TN];
#pragma unroll
                for (int j = 0; j < TN; ++j) {
                    const uint32_t r = (wn * TN + j) * 32 + r32, c = (2 * h + s / 4) ^ ((r >> 2) & 3);
                    const uint2 two = *reinterpret_cast<const uint2*>(base + G::A_BYTES + G::B_BYTES + r * 8);
                    const uint32_t sw = __builtin_amdgcn_alignbit(two.y, two.x, s_shift[j]) & s_mask;
                    b[j] = decode8(*reinterpret_cast<const uint32_t*>(base + G::A_BYTES + r * 64 + c * 16 + 4 * (s % 4)),
                                   __uint_as_float(((sw >> (8 * (2 * h + s / 4))) & 0xffu) << 23));
                }
#pragma unroll
                for (int i = 0; i < TM; ++i) {
                    u32x4 v0, v1;
                    x_piece(i, s, v0, v1);
                    bf16x8 hi, mid, lo;
                    split3_pass(pass, all_tiny(most[i]), v0, v1, hi, mid, lo);
#pragma unroll
                    for (int j = 0; j < TN; ++j) {
                        sum[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(hi, b[j], sum[i][j], 0, 0, 0);
                        sum[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(mid, b[j], sum[i][j], 0, 0, 0);
                        sum[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(lo, b[j], sum[i][j], 0, 0, 0);
                    }
                }
            }
            mfma_drain();
#pragma unroll
            for (int i = 0; i < TM; ++i)
#pragma unroll
                for (int j = 0; j < TN; ++j)
#pragma unroll
                    for (int r = 0; r < 16; ++r) acc[i][j][r] += (double)sum[i][j][r] * (pass ? kTinyDown : 1.0);
        }
    };

    // D-stage ring: stages st + 1 .. st + D - 2 stay in flight while stage st
    // is computed; stage st + D - 1 is issued into the slot stage st - 1 used,
    // after the barrier that ends every wave's reads of it
    auto walk = [&](auto&& step) {
        // (opaque: a second walk computes its offsets again, instead of the first
        // one's registers holding them)
        uint32_t lane = threadIdx.x % 64;
        if constexpr (ANY && !XBF16) asm volatile("" : "+v"(lane));
        // this lane's global offsets (stage 0) of its loads; LDS slot p = (q NW + wave) 64 + lane
        uint32_t a_goff[G::A_INSTR], b_goff[G::B_INSTR], s_goff[G::S_INSTR];
        uint32_t a_col[G::A_INSTR], b_col[G::B_INSTR];  // first element within the stage (ANY)
#pragma unroll
        for (int q = 0; q < G::A_INSTR; ++q) {
            const uint32_t p = (q * G::NW + wave) * 64 + lane, row = p / G::A_CPR, c = (p % G::A_CPR) ^ (row % 16);
            a_goff[q] = (row0 + row) * k * G::XB + k0 * G::XB + c * 16;
            a_col[q] = c * 16 / G::XB;
        }
#pragma unroll
        for (int q = 0; q < G::B_INSTR; ++q) {
            const uint32_t p = (q * G::NW + wave) * 64 + lane, row = p / 4, c = (p % 4) ^ ((row >> 2) & 3);
            b_goff[q] = (col0 + row) * (k / 2) + k0 / 2 + c * 16;
            b_col[q] = c * 32;
        }
#pragma unroll
        for (int q = 0; q < G::S_INSTR; ++q) {
            const uint32_t p = wave * G::S_WORDS + q * 64 + lane, row = ANY ? p / 2 : p;
            s_goff[q] = (col0 + row) * (k / 32) + k0 / 32 + mis;
            if (ANY) s_goff[q] = (s_goff[q] & ~3u) + 4 * (p % 2);
        }
        auto issue = [&](uint32_t st, uint32_t slot) {
            uint8_t* base = lds + slot * G::STAGE;
            const uint32_t live = klen - st * kBK;  // ANY: columns of the stage before K's end
#pragma unroll
            for (int q = 0; q < G::A_INSTR; ++q) {
                uint32_t off = a_goff[q] + st * kBK * G::XB;
                if (ANY) off = a_col[q] < live ? off : kPastEnd;
                load_lds16(xr, (lds_ptr)(base + (q * G::NW + wave) * 1024), off);
            }
#pragma unroll
            for (int q = 0; q < G::B_INSTR; ++q) {
                uint32_t off = b_goff[q] + st * (kBK / 2);
                if (ANY) off = b_col[q] < live ? off : kPastEnd;
                load_lds16(pr, (lds_ptr)(base + G::A_BYTES + (q * G::NW + wave) * 1024), off);
            }
            // the wave's scale words; lanes past them stay inactive, so they
            // write nothing into the next wave's words (the instruction still
            // counts once in vmcnt: lane 0 is always active)
#pragma unroll
            for (int q = 0; q < G::S_INSTR; ++q)
                if (q * 64 + lane < (uint32_t)G::S_WORDS)
                    load_lds4(sr, (lds_ptr)(base + G::A_BYTES + G::B_BYTES + (wave * G::S_WORDS + q * 64) * 4),
                              s_goff[q] + st * (kBK / 32));
        };
#pragma unroll
        for (int p = 0; p < D - 1; ++p)
            if ((uint32_t)p < stages) issue(p, p);
        for (uint32_t st = 0; st < stages; ++st) {
            const uint32_t ahead = stages - 1 - st;  // stages issued after st, at most D - 2
            if (ahead >= (uint32_t)(D - 2)) wait_vm<(D - 2) * G::LPS>();
            else if (D > 3 && ahead == 1) wait_vm<(D > 3 ? 1 : 0) * G::LPS>();
            else wait_vm<0>();
            lds_barrier();
            if (st + D - 1 < stages) issue(st + D - 1, (st + D - 1) % D);
            step(st, st % D);
        }
    };
    walk(compute);
    if constexpr (ANY && !XBF16) {
        if (workgroup_any<G::NW>(__any(care), reinterpret_cast<uint32_t*>(lds), wave)) {
#pragma unroll
            for (int i = 0; i < TM; ++i)
#pragma unroll
                for (int j = 0; j < TN; ++j)
#pragma unroll
                    for (int r = 0; r < 16; ++r) acc[i][j][r] = 0;
            walk(compute_careful);
        }
    }
    mfma_drain();

    // D[i][j] of a 32x32 tile: lane l holds column l % 32 and, in register r,
    // row 8 (r / 4) + 4 (l / 32) + r % 4
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) {
            const uint32_t col = col0 + (wn * TN + j) * 32 + r32;
            if (col >= n) continue;
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const uint32_t row = row0 + (wm * TM + i) * 32 + 8 * (r / 4) + 4 * h + r % 4;
                if (row < m) y[(size_t)row * n + col] = (float)acc[i][j][r];
            }
        }
}

// K of one of ks slices: whole stages, the last slice taking what is left.
uint32_t slice_k(uint32_t k, uint32_t ks) {
    const uint32_t stages = (k + kBK - 1) / kBK;
    return (stages + ks - 1) / ks * kBK;
}

// Can K be cut into ks slices that the kernel takes: equal ones of whole
// stages, or (K no whole number of stages) none of them empty.
bool slices_fit(uint32_t k, uint32_t ks) {
    if (k % kBK == 0) return k % (ks * kBK) == 0;
    return (uint64_t)(ks - 1) * slice_k(k, ks) < k;
}

// y = sum over the slices of part[s] (count floats each), in slice order.
__global__ __launch_bounds__(256) void split_sum_kernel(const float* __restrict__ part, uint32_t ks, uint32_t count,
                                                        float* __restrict__ y) {
    const uint32_t i = blockIdx.x * 256 + threadIdx.x;
    if (count % 4 == 0) {
        if (4 * i >= count) return;
        f32x4 a = *reinterpret_cast<const f32x4*>(part + 4 * i);
        for (uint32_t s = 1; s < ks; ++s) a += *reinterpret_cast<const f32x4*>(part + (size_t)s * count + 4 * i);
        *reinterpret_cast<f32x4*>(y + 4 * i) = a;
    } else {
        if (i >= count) return;
        float a = part[i];
        for (uint32_t s = 1; s < ks; ++s) a += part[(size_t)s * count + i];
        y[i] = a;
    }
}

// The same for a group: the slices of all its weights in one pass.
__global__ __launch_bounds__(256) void split_sum_group_kernel(const float* __restrict__ part, uint32_t ks, uint32_t m,
                                                              const GemmSegs g) {
    const uint32_t i = blockIdx.x * 256 + threadIdx.x, count = m * g.rows;
    if (i >= count) return;
    float a = part[i];
    for (uint32_t s = 1; s < ks; ++s) a += part[(size_t)s * count + i];
    float* y = g.y[0];
    uint32_t at = i;
#pragma unroll
    for (int q = 1; q < 4; ++q)
        if (q < (int)g.count && i >= m * g.row0[q]) {
            y = g.y[q];
            at = i - m * g.row0[q];
        }
    y[at] = a;
}

template <bool XBF16, int WM, int WN, int TM, int TN, bool ANY>
hipError_t go(const GemvArgs& a, uint32_t ks, float* part) {
    // deepest ring that fits: 3 stages of a 128 x 128 bf16 tile (121.5 KiB)
    using G2 = Geometry<XBF16, WM, WN, TM, TN, 2, ANY>;
    constexpr int D3 = G2::STAGE * 3 <= 160 * 1024 ? 3 : 2;
    constexpr int D = (G2::STAGE * 4 <= 160 * 1024 && 2 * G2::LPS <= 63) ? 4 : D3;
    using G = Geometry<XBF16, WM, WN, TM, TN, D, ANY>;
    const uint32_t tiles_m = (a.m + G::BM - 1) / G::BM;
    if (a.group) {
        // each weight of the group a run of column tiles
        GemmSegs sg{};
        uint32_t tiles_n = 0;
        sg.count = a.group->count;
        for (uint32_t s = 0; s < sg.count; ++s) {
            sg.packed[s] = a.group->packed[s];
            sg.scales[s] = a.group->scales[s];
            sg.y[s] = a.group->y[s];
            sg.n[s] = a.group->n[s];
            sg.tile0[s] = tiles_n;
            sg.row0[s] = sg.rows;
            tiles_n += (sg.n[s] + G::BN - 1) / G::BN;
            sg.rows += sg.n[s];
        }
        if (ks < 1) ks = 1;
        const uint32_t tiles = tiles_n * tiles_m;
        hipLaunchKernelGGL((gemm_exact_kernel<XBF16, WM, WN, TM, TN, D, ANY, GemmSegs>), dim3(tiles * ks), dim3(G::NT), 0,
                           a.stream, nullptr, nullptr, a.x, nullptr, a.m, 0u, a.k, tiles_n, tiles, slice_k(a.k, ks),
                           ks > 1 ? part : nullptr, sg);
        const hipError_t e = hipGetLastError();
        if (e != hipSuccess || ks == 1) return e;
        hipLaunchKernelGGL(split_sum_group_kernel, dim3((a.m * sg.rows + 255) / 256), dim3(256), 0, a.stream, part, ks,
                           a.m, sg);
        return hipGetLastError();
    }
    const uint32_t tiles_n = (a.n + G::BN - 1) / G::BN;
    const uint32_t tiles = tiles_n * tiles_m;
    if (ks < 1) ks = 1;
    hipLaunchKernelGGL((gemm_exact_kernel<XBF16, WM, WN, TM, TN, D, ANY>), dim3(tiles * ks), dim3(G::NT), 0, a.stream,
                       a.packed, a.scales, a.x, a.y, a.m, a.n, a.k, tiles_n, tiles, slice_k(a.k, ks),
                       ks > 1 ? part : nullptr, NoGemmSegs{});
    hipError_t e = hipGetLastError();
    if (e != hipSuccess || ks == 1) return e;
    return launch_split_sum(part, ks, a.m * a.n, a.y, a.stream);
}

// the instances that the shape rule picks from, for widths of whole stages and for any
template <bool XBF16, bool ANY>
hipError_t dispatch_rule(const GemvArgs& a, const GemmConfig& c, uint32_t ks, float* part) {
    if (c.wm == 2 && c.wn == 2 && c.tm == 2 && c.tn == 3) return go<XBF16, 2, 2, 2, 3, ANY>(a, ks, part);
    if (c.wm == 2 && c.wn == 2 && c.tm == 1 && c.tn == 1) return go<XBF16, 2, 2, 1, 1, ANY>(a, ks, part);
    // (bf16 of any width: eight_waves has others in their place)
    if constexpr (!(XBF16 && ANY)) {
        if (c.wm == 2 && c.wn == 2 && c.tm == 2 && c.tn == 2) return go<XBF16, 2, 2, 2, 2, ANY>(a, ks, part);
        if (c.wm == 1 && c.wn == 4 && c.tm == 2 && c.tn == 2) return go<XBF16, 1, 4, 2, 2, ANY>(a, ks, part);
        if (c.wm == 1 && c.wn == 4 && c.tm == 2 && c.tn == 1) return go<XBF16, 1, 4, 2, 1, ANY>(a, ks, part);
    }
    // (f32 of any width: picked by nothing)
    if constexpr (XBF16 || !ANY)
        if (c.wm == 2 && c.wn == 4 && c.tm == 1 && c.tn == 2) return go<XBF16, 2, 4, 1, 2, ANY>(a, ks, part);
    // (picked by eight_waves only)
    if constexpr (XBF16 == ANY) {
        if (c.wm == 4 && c.wn == 2 && c.tm == 1 && c.tn == 2) return go<XBF16, 4, 2, 1, 2, ANY>(a, ks, part);
        if (c.wm == 2 && c.wn == 4 && c.tm == 1 && c.tn == 1) return go<XBF16, 2, 4, 1, 1, ANY>(a, ks, part);
    }
    // a 128 x 256 tile of f32 activations would leave room for one stage only
    if constexpr (XBF16)
        if (c.wm == 2 && c.wn == 4 && c.tm == 2 && c.tn == 2) return go<XBF16, 2, 4, 2, 2, ANY>(a, ks, part);
    return hipErrorNotSupported;
}

// Eight waves, two a SIMD, for the same tile where one wave's conversions (f32
// activations, whole stages: 24576 x 4096 at 64 rows 96 -> 75 us, 12288 x 2048
// at 300 rows 58.6 -> 50.7) or 64-bit sums (bf16, any width: 8576 x 1600 at 200
// rows 27.5 -> 24.4 us) hold up its MFMAs. f32 at any width has both, and four
// waves measured faster (by a quarter at 8576 x 1600, 77 rows); bf16 of whole
// stages has neither, and runs the same in both.
GemmConfig eight_waves(GemmConfig c, bool x_bf16, bool any) {
    if (x_bf16 != any) return c;
    if (c.wm == 2 && c.wn == 2 && c.tm == 2 && c.tn == 2) c.wm = 4, c.tm = 1;
    else if (c.wm == 1 && c.wn == 4 && c.tm == 2) c.wm = 2, c.tm = 1;
    return c;
}

template <bool XBF16>
hipError_t dispatch(const GemvArgs& a, const GemmConfig& c, float* part) {
    // instances: (waves along M x along N, MFMA tiles per wave along M x N)
    const uint32_t ks = c.ks < 1 ? 1u : (uint32_t)c.ks;
    if (a.k % kBK != 0) return dispatch_rule<XBF16, true>(a, c, ks, part);
    if (c.wm == 2 && c.wn == 2 && c.tm == 2 && c.tn == 1) return go<XBF16, 2, 2, 2, 1, false>(a, ks, part);
    if (c.wm == 2 && c.wn == 2 && c.tm == 1 && c.tn == 2) return go<XBF16, 2, 2, 1, 2, false>(a, ks, part);
    if (c.wm == 4 && c.wn == 1 && c.tm == 1 && c.tn == 2) return go<XBF16, 4, 1, 1, 2, false>(a, ks, part);
    if (c.wm == 1 && c.wn == 4 && c.tm == 1 && c.tn == 2) return go<XBF16, 1, 4, 1, 2, false>(a, ks, part);
    if (c.wm == 1 && c.wn == 4 && c.tm == 1 && c.tn == 1) return go<XBF16, 1, 4, 1, 1, false>(a, ks, part);
    return dispatch_rule<XBF16, false>(a, c, ks, part);
}

}  // namespace

hipError_t launch_split_sum(const float* part, uint32_t ks, uint32_t count, float* y, hipStream_t s) {
    const uint32_t threads = count % 4 == 0 ? count / 4 : count;
    hipLaunchKernelGGL(split_sum_kernel, dim3((threads + 255) / 256), dim3(256), 0, s, part, ks, count, y);
    return hipGetLastError();
}

bool gemm_exact_supported(uint32_t m, uint32_t n, uint32_t k, bool x_bf16) {
    // 32-bit buffer offsets over x and the packed weights
    const uint64_t xb = (uint64_t)m * k * (x_bf16 ? 2 : 4);
    return m >= 1 && n >= 1 && k % kBK == 0 && k >= kBK && xb + 256 * k * 4 < (1ull << 31) &&
           (uint64_t)(n + 256) * (k / 2) < (1ull << 31);
}

bool gemm_any_supported(uint32_t m, uint32_t n, uint32_t k, bool x_bf16) {
    if (k % kBK == 0) return gemm_exact_supported(m, n, k, x_bf16);
    const uint64_t xb = (uint64_t)m * k * (x_bf16 ? 2 : 4);
    return m >= 1 && n >= 1 && k % 32 == 0 && k >= 32 && xb + 256 * k * 4 < (1ull << 31) &&
           (uint64_t)(n + 256) * (k / 2) < (1ull << 31);
}

// The few-token-row K split (a grid short of the CUs) takes at most 4 MiB of
// partials, the range its picks were measured in.
constexpr uint64_t kFewRowsSplitBytes = 4ull << 20;

// The arrangement and K split for a shape; part_bytes of scratch for partials.
static GemmConfig shape_rule(const GemvArgs& a, int cus, uint64_t part_bytes) {
    // column tiles of width bn over the weight (or over each weight of a group)
    auto col_tiles = [&](uint32_t bn) -> uint64_t {
        if (!a.group) return (a.n + bn - 1) / bn;
        uint64_t t = 0;
        for (uint32_t s = 0; s < a.group->count; ++s) t += (a.group->n[s] + bn - 1) / bn;
        return t;
    };
    GemmConfig c;
    // The tile with the least estimated time: whole rounds of workgroups
    // (one per CU) times the time one round of that tile takes. The round
    // times (µs at K = 4096, bf16 x) are from a sweep of every instance on
    // the Qwen3-8B q, gate and down weights at M = 64..2048 on MI355X
    // (cold weights); with them the pick was the fastest instance, or
    // within 2% of it, at every M of the sweep: gate at M = 384 / 768 /
    // 1536 128 x 192 (47 / 90 / 145 us, where the largest tile whose grid
    // reaches three quarters of the CUs takes 64 / 102 / 157 us), at 2048
    // 128 x 256 (176 us); q and down at M = 512 64 x 128 (23 / 64 us).
    // The larger tiles re-read fewer operand bytes per flop, the smaller
    // ones leave fewer CUs idle in the last round.
    struct Cand { int wm, wn, tm, tn, bm, bn; double round_us; };
    const Cand cands[] = {{2, 4, 2, 2, 128, 256, 50.0}, {2, 2, 2, 3, 128, 192, 46.0},
                          {1, 4, 2, 2, 64, 256, 33.5},  {2, 2, 2, 2, 128, 128, 34.5},
                          {1, 4, 2, 1, 64, 128, 22.0},  {2, 2, 1, 1, 64, 64, 16.5}};
    const uint64_t nc = (uint64_t)(cus > 0 ? cus : 256);
    const uint64_t want = nc * 3 / 4;
    // 128 x 256 has an instance for bf16 x only
    auto wide = [&](const Cand& cd) { return cd.bn == 256 && cd.bm == 128 && !a.x_bf16; };
    // A bf16 group of whole stages runs unsplit even when its tiles leave
    // CUs idle: one short round of them beats a split and the pass that
    // adds it (a small model's layer 28.0 against 30.3 us, 4096 wide at 48
    // rows 89.8 against 90.3), and its weights' separate launches.
    // A split saves time with K and costs it with the outputs, so that a group
    // cuts K only while its partials stay below 8 KiB for every element of K
    // (two weights of 1536 x 512, f32 x, at 64 rows 10.7 -> 8.7 us with 3 MiB in
    // four slices, at 200 and 300 rows 11.1 and 11.5 -> 13.0 and 20.5 with 5 and
    // 14 MiB; 2048 + 512 + 512 x 2048 at 300 rows 33.8 -> 30.0 with 14 MiB) and,
    // where the tiles are few, not into a second round of the CUs (768 + 192 +
    // 192 x 768 at 300 rows 14.6 -> 15.5 us).
    const bool may_split = !(a.group && a.x_bf16 && a.k % kBK == 0);
    if (a.group && part_bytes > 8192ull * a.k) part_bytes = 8192ull * a.k;
    uint32_t rows = a.n;  // weight rows, of all the group's weights
    if (a.group) {
        rows = 0;
        for (uint32_t s = 0; s < a.group->count; ++s) rows += a.group->n[s];
    }
    const Cand* best = nullptr;
    double best_t = 0.0;
    for (const Cand& cd : cands) {
        if (wide(cd)) continue;
        const uint64_t tiles = (uint64_t)((a.m + cd.bm - 1) / cd.bm) * col_tiles(cd.bn);
        const double t = (double)((tiles + nc - 1) / nc) * cd.round_us;
        if (!best || t < best_t) {
            best = &cd;
            best_t = t;
        }
    }
    // f32 activations, and bf16 ones on wide K (K >= 8192): the largest
    // tile whose workgroups, with K cut into 1-4 slices of whole stages,
    // make one round of at least three quarters of the CUs (the most
    // workgroups among equal tiles). Measured on the 8B q / gate / down
    // weights at 64..1024 rows (cold): f32 q at 256 / 512 rows 63.9 /
    // 113.0 -> 44.2 / 75.8 us, gate at 128 / 256 113.3 / 131.7 -> 53.2 /
    // 90.9, down at 256 / 512 184 / 329 -> 107 / 201; bf16 down at 384 /
    // 512 / 1024 60.7 / 66.0 / 101.7 -> 47.5 / 54.1 / 93.3. bf16 at K =
    // 4096 keeps the round-time pick (its splits measured slower there).
    if (!a.x_bf16 || a.k >= 8192) {
        const Cand* sel = nullptr;
        uint32_t sel_ks = 0;
        uint64_t sel_area = 0, sel_wgs = 0;
        for (const Cand& cd : cands) {
            if (wide(cd)) continue;
            const uint64_t tiles = (uint64_t)((a.m + cd.bm - 1) / cd.bm) * col_tiles(cd.bn);
            for (uint32_t ks = 1; ks <= 4; ++ks) {
                if (!slices_fit(a.k, ks)) continue;
                if (ks > 1 && (!may_split || (uint64_t)ks * a.m * rows * 4 > part_bytes)) continue;
                const uint64_t wgs = tiles * ks, area = (uint64_t)cd.bm * cd.bn;
                if (wgs > nc || wgs < want) continue;
                if (!sel || area > sel_area || (area == sel_area && wgs > sel_wgs)) {
                    sel = &cd;
                    sel_ks = ks;
                    sel_area = area;
                    sel_wgs = wgs;
                }
            }
        }
        if (sel) {
            c.wm = sel->wm; c.wn = sel->wn; c.tm = sel->tm; c.tn = sel->tn;
            c.ks = (int)sel_ks;
            return eight_waves(c, a.x_bf16, a.k % kBK != 0);
        }
    }
    const Cand pick = *best;
    c.wm = pick.wm; c.wn = pick.wn; c.tm = pick.tm; c.tn = pick.tn;
    // A grid still short of the CUs (few token rows): split K across up to
    // four workgroups per tile, each slice whole stages, when the partials
    // fit the scratch; a second small kernel adds them in slice order.
    const uint64_t tiles = (uint64_t)((a.m + pick.bm - 1) / pick.bm) * col_tiles(pick.bn);
    c.ks = 1;
    for (uint32_t ks = 4; ks >= 2 && tiles < want && may_split; --ks) {
        if (slices_fit(a.k, ks) && !(a.group && tiles * ks > nc) &&
            (uint64_t)ks * a.m * rows * 4 <= std::min(part_bytes, kFewRowsSplitBytes)) {
            c.ks = (int)ks;
            break;
        }
    }
    return eight_waves(c, a.x_bf16, a.k % kBK != 0);
}

hipError_t launch_gemm_exact(const GemvArgs& a, int cus, const GemmConfig* forced, float* part, uint64_t part_bytes) {
    if (a.group) {
        // a group: every weight supported, no explicit configuration
        if (forced && forced->wm) return hipErrorNotSupported;
        if (a.group->count < 1 || a.group->count > 4) return hipErrorNotSupported;
        for (uint32_t s = 0; s < a.group->count; ++s)
            if (!gemm_any_supported(a.m, a.group->n[s], a.k, a.x_bf16)) return hipErrorNotSupported;
    } else if (!gemm_any_supported(a.m, a.n, a.k, a.x_bf16)) {
        return hipErrorNotSupported;
    }
    GemmConfig c;
    if (forced && forced->wm) {
        c = *forced;
        // arrangements of the shape rule's own
        if ((c.wm == 4 && c.wn == 2) || (c.wm == 2 && c.wn == 4 && c.tm == 1 && c.tn == 1)) return hipErrorNotSupported;
        // an explicit K split: whole stages per slice and partials within the scratch
        if (c.ks > 1 && (a.k % ((uint32_t)c.ks * kBK) != 0 || !part ||
                         (uint64_t)c.ks * a.m * a.n * 4 > part_bytes))
            return hipErrorNotSupported;
    } else {
        c = shape_rule(a, cus, part ? part_bytes : 0);
    }
    return a.x_bf16 ? dispatch<true>(a, c, part) : dispatch<false>(a, c, part);
}

uint32_t mx4_rule_gemm_exact(const uint32_t* n, uint32_t count, uint32_t m, uint32_t k, bool x_bf16, int cus, uint64_t part_bytes) {
    GemvGroup g{};
    g.count = count;
    for (uint32_t i = 0; i < count; ++i) g.n[i] = n[i];
    GemvArgs a{nullptr, nullptr, nullptr, nullptr, m, n[0], k, x_bf16, nullptr};
    if (count > 1) a.group = &g;
    const GemmConfig c = shape_rule(a, cus, part_bytes);
    return (uint32_t)(c.wm * 10000 + c.wn * 1000 + c.tm * 100 + c.tn * 10 + c.ks);
}

}  // namespace mx4
