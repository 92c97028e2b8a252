// bf16.hip -- projections with bf16 (non-quantized) weights, the other arm of
// the reference's matmul: engine/src/lib.rs:240-266 with Tensor::bf16 weights
// (the `None` arm of lib.rs:255), which the Metal bridge takes when `scales`
// is NULL (engine/src/metal.rs:45-50, engine/src/metal.m:85-95).
//
// y[m, r] = sum_k x[m, k] * bf16_to_f32(w[r, k]), f32 accumulation. bf16 -> f32
// is exact (the top half of an f32), so the only difference from the
// reference's sequential loop is the summation order.
//
// One token row (decode): bf16_gemv_kernel streams the weights, up to four
// matrices that share x in a launch. Two to 32 rows run skinny_any.hip, more
// gemm_bf16.hip. Small weights, where those leave most of the chip idle
// (bf16_rows_faster, bf16_matmul_us), and rows that are not whole 16-byte pieces:
//
// One wave per weight row, MT tokens per wave: each lane streams 16-byte
// pieces (8 weights) of the row, fully coalesced, and reuses each piece for the
// MT activation rows; the wave then reduces with lane shuffles. Rows whose
// width is not a multiple of 8 (or is misaligned) take the element-wise form.
#include "mx4_device.h"
#include "mx4_kernels.h"

namespace mx4 {

namespace {

template <bool XBF16>
__device__ __forceinline__ void load_x8(const void* x, uint64_t elem, float (&v)[8]) {
    if constexpr (XBF16) {
        const u32x4 p = load_u32x4(static_cast<const uint8_t*>(x) + 2 * elem);
#pragma unroll
        for (int d = 0; d < 4; ++d) {
            v[2 * d] = bf16_bits_to_f32(p[d] & 0xffffu);
            v[2 * d + 1] = bf16_bits_to_f32(p[d] >> 16);
        }
    } else {
        const float* f = static_cast<const float*>(x) + elem;
        const f32x4 a = *reinterpret_cast<const f32x4*>(f);
        const f32x4 b = *reinterpret_cast<const f32x4*>(f + 4);
#pragma unroll
        for (int d = 0; d < 4; ++d) {
            v[d] = a[d];
            v[4 + d] = b[d];
        }
    }
}

template <bool XBF16>
__device__ __forceinline__ float load_x1(const void* x, uint64_t elem) {
    if constexpr (XBF16)
        return bf16_bits_to_f32(static_cast<const uint16_t*>(x)[elem]);
    else
        return static_cast<const float*>(x)[elem];
}

template <bool XBF16, int MT, bool VEC>
__global__ __launch_bounds__(256) void bf16_matmul_kernel(const uint16_t* __restrict__ w, const void* __restrict__ x,
                                                          float* __restrict__ y, uint32_t m, uint32_t n, uint32_t k) {
    const uint32_t lane = threadIdx.x % 64;
    const uint32_t row = blockIdx.x * 4 + threadIdx.x / 64;
    const uint32_t m0 = blockIdx.y * MT;
    if (row >= n) return;
    const uint16_t* wr = w + (uint64_t)row * k;
    float acc[MT];
#pragma unroll
    for (int q = 0; q < MT; ++q) acc[q] = 0.0f;
    if constexpr (VEC) {
        for (uint32_t c = lane; c < k / 8; c += 64) {
            const u32x4 p = load_u32x4(reinterpret_cast<const uint8_t*>(wr) + 16 * (uint64_t)c);
            float wv[8];
#pragma unroll
            for (int d = 0; d < 4; ++d) {
                wv[2 * d] = bf16_bits_to_f32(p[d] & 0xffffu);
                wv[2 * d + 1] = bf16_bits_to_f32(p[d] >> 16);
            }
#pragma unroll
            for (int q = 0; q < MT; ++q) {
                const uint32_t tok = m0 + q < m ? m0 + q : m - 1;
                float xv[8];
                load_x8<XBF16>(x, (uint64_t)tok * k + 8 * (uint64_t)c, xv);
#pragma unroll
                for (int e = 0; e < 8; ++e) acc[q] = __builtin_fmaf(xv[e], wv[e], acc[q]);
            }
        }
    } else {
        for (uint32_t e = lane; e < k; e += 64) {
            const float wv = bf16_bits_to_f32(wr[e]);
#pragma unroll
            for (int q = 0; q < MT; ++q) {
                const uint32_t tok = m0 + q < m ? m0 + q : m - 1;
                acc[q] = __builtin_fmaf(load_x1<XBF16>(x, (uint64_t)tok * k + e), wv, acc[q]);
            }
        }
    }
#pragma unroll
    for (int q = 0; q < MT; ++q) {
        const float v = wave_sum(acc[q]);
        if (lane == 0 && m0 + q < m) y[(uint64_t)(m0 + q) * n + row] = v;
    }
}

// bf16 element e of a 16-byte piece, as f32 bits.
__device__ __forceinline__ uint32_t half_up(const u32x4& v, int e) { return e % 2 ? v[e / 2] & 0xffff0000u : v[e / 2] << 16; }

// The same for token rows of small weights, which the matrix cores would take
// longer for: four chains of at most eight products a token row, then sums in 64
// bits, so that the outputs come out as near to the exact sums as theirs (bf16 x
// 0.33e-7 relative, f32 0.66e-7 at any K; one chain per lane 0.9e-7 to 1.3e-7 and
// 1.0e-7 at K = 1024 to 2.6e-7 at 12288). What binds are loads and launch: with all
// loads of a turn on their way at once it takes no longer than one chain does (1024 x
// 4096 at 8 rows of f32 7.8 us, 16 x 1024 2.8 or, bf16 x, 2.7 for 2.9).
template <bool XBF16>
__global__ __launch_bounds__(256) void bf16_matmul_fine_kernel(const uint16_t* __restrict__ w, const void* __restrict__ x,
                                                               float* __restrict__ y, uint32_t m, uint32_t n,
                                                               uint32_t k) {
    const uint32_t lane = threadIdx.x % 64;
    const uint32_t row = blockIdx.x * 4 + threadIdx.x / 64;
    const uint32_t m0 = blockIdx.y * 4;
    if (row >= n) return;
    double acc[4] = {};
    for (uint32_t c0 = lane; c0 < k / 8; c0 += 4 * 64) {
        float part[4][4] = {};
        for (uint32_t c = c0; c < k / 8 && c < c0 + 4 * 64; c += 64) {
            u32x4 xw[4][XBF16 ? 1 : 2];
            const u32x4 ww = load_u32x4(reinterpret_cast<const uint8_t*>(w) + 2 * ((uint64_t)row * k + 8 * (uint64_t)c));
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const uint32_t tok = m0 + q < m ? m0 + q : m - 1;
                const uint8_t* xp = static_cast<const uint8_t*>(x) + (XBF16 ? 2 : 4) * ((uint64_t)tok * k + 8 * (uint64_t)c);
#pragma unroll
                for (int h = 0; h < (XBF16 ? 1 : 2); ++h) xw[q][h] = load_u32x4(xp + 16 * h);
            }
            __builtin_amdgcn_sched_barrier(0);  // every load on its way before the first is waited for
#pragma unroll
            for (int q = 0; q < 4; ++q)
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    const float xv = __uint_as_float(XBF16 ? half_up(xw[q][0], e) : xw[q][XBF16 ? 0 : e / 4][e % 4]);
                    part[q][e % 4] = __builtin_fmaf(xv, __uint_as_float(half_up(ww, e)), part[q][e % 4]);
                }
        }
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            acc[q] += (double)(part[q][0] + part[q][1]);
            acc[q] += (double)(part[q][2] + part[q][3]);
        }
    }
    const uint32_t q = lane / 16;
    const double v = wave_sum4(acc, lane);
    if (lane % 16 == 0 && m0 + q < m) y[(uint64_t)(m0 + q) * n + row] = (float)v;
}

// One token row. A wave takes a row at a time, U x 512 elements of it per turn
// (U loads of 1 KiB), the next turn's loads (of this row or its next one) issued
// before this turn's products; x lies in LDS once per workgroup, filled by
// direct-to-LDS loads that are issued first. Bound by HBM: 24576 x 4096 (201 MB)
// 35.4 us, 5.7 TB/s; 4096 x 12288 20.1 us, 5.0 TB/s. A layer of hidden size 2048
// ran at 2.4 TB/s with a load waited for at a time and q, k, v and gate, up
// launched one by one. Two rows a wave measured the same or slower (12288 x 2048
// 11.1 against 10.5 us), two turns' worth of loads (U = 2) slower past K = 1024.
struct Bf16Group {
    const uint16_t* w[4];
    float* y[4];
    uint32_t n[4];
    uint32_t first[5];  // rows before each weight; first[count] .. first[4] are all of them
    uint32_t count;
};

template <bool XBF16, int U>
__global__ __launch_bounds__(512) void bf16_gemv_kernel(const void* __restrict__ x, uint32_t k, uint32_t turns,
                                                        uint32_t rows, uint32_t stride, const Bf16Group g) {
    extern __shared__ __attribute__((aligned(16))) uint8_t xl[];
    constexpr uint32_t XB = XBF16 ? 2 : 4;
    const uint32_t lane = threadIdx.x % 64;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
    {
        // turns x U x 512 elements, zeros past K
        const __amdgpu_buffer_rsrc_t xr = rsrc(x, k * XB);
        const uint32_t bytes = turns * U * 512 * XB;
        for (uint32_t c = wave * 1024; c < bytes; c += 8 * 1024) load_lds16(xr, (lds_ptr)(xl + c), c + 16 * lane);
        __builtin_amdgcn_sched_barrier(0);
    }
    struct Turn {
        u32x4 w[U];
    };
    auto pick = [&](uint32_t at, const uint16_t*& w, float*& y, uint32_t& row) {
        w = g.w[0];
        y = g.y[0];
        uint32_t first = 0;
#pragma unroll
        for (int q = 1; q < 4; ++q) {
            const bool in = q < (int)g.count && at >= g.first[q];
            w = in ? g.w[q] : w;
            y = in ? g.y[q] : y;
            first = in ? g.first[q] : first;
        }
        row = at - first;
    };
    // a row past the end loads zeros without touching memory
    auto load = [&](uint32_t at, uint32_t turn, Turn& t) {
        const uint16_t* w;
        float* y;
        uint32_t row;
        pick(at, w, y, row);
        const bool valid = at < rows;
        const __amdgpu_buffer_rsrc_t r = rsrc(w + (size_t)(valid ? row : 0) * k, valid ? k * 2 : 0);
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const uint32_t e = (turn * U + u) * 512 + 8 * lane;
            t.w[u] = __builtin_amdgcn_raw_buffer_load_b128(r, e < k ? 2 * e : kPastEnd, 0, 2);
        }
        __builtin_amdgcn_sched_barrier(0);
    };
    float acc = 0.0f;
    // (v_dot2_f32_bf16 keeps subnormal values and results)
    auto consume = [&](uint32_t turn, const Turn& t) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const uint8_t* xp = xl + ((turn * U + u) * 512 + 8 * lane) * XB;
            if constexpr (XBF16) {
                const u32x4 v = *reinterpret_cast<const u32x4*>(xp);
#pragma unroll
                for (int d = 0; d < 4; ++d)
                    acc = __builtin_amdgcn_fdot2_f32_bf16(as_bf16x2(t.w[u][d]), as_bf16x2(v[d]), acc, false);
            } else {
                const f32x4 a = *reinterpret_cast<const f32x4*>(xp), b = *reinterpret_cast<const f32x4*>(xp + 16);
                const float v[8] = {a[0], a[1], a[2], a[3], b[0], b[1], b[2], b[3]};
#pragma unroll
                for (int d = 0; d < 4; ++d) {
                    acc = __builtin_fmaf(v[2 * d], __uint_as_float(t.w[u][d] << 16), acc);
                    acc = __builtin_fmaf(v[2 * d + 1], __uint_as_float(t.w[u][d] & 0xffff0000u), acc);
                }
            }
        }
    };
    auto finish = [&](uint32_t at) {
        const uint16_t* w;
        float* y;
        uint32_t row;
        pick(at, w, y, row);
        float sums[1] = {acc};
        const float total = wave_reduce_rows<1>(sums, lane);
        if (lane == 0) y[row] = total;
        acc = 0.0f;
    };
    uint32_t at = blockIdx.x * 8 + wave, turn = 0;
    Turn a, b;
    load(at, 0, a);
    wait_vm<U>();  // x is in, the weights need not be
    __syncthreads();
    if (at >= rows) return;
    auto step = [&](const Turn& cur, Turn& nxt) -> bool {
        const bool last = turn + 1 == turns;
        const uint32_t next = last ? at + stride : at;
        load(next, last ? 0 : turn + 1, nxt);
        consume(turn, cur);
        if (last) {
            finish(at);
            if (next >= rows) return true;
        }
        at = next;
        turn = last ? 0 : turn + 1;
        return false;
    };
    for (;;) {
        if (step(a, b)) break;
        if (step(b, a)) break;
    }
}

template <bool XBF16, int U>
hipError_t go_gemv(const Bf16Group& g, const void* x, uint32_t k, uint32_t rows, uint32_t grid, hipStream_t s) {
    const uint32_t turns = (k + 512 * U - 1) / (512 * U);
    hipLaunchKernelGGL((bf16_gemv_kernel<XBF16, U>), dim3(grid), dim3(512), turns * U * 512 * (XBF16 ? 2 : 4), s, x, k,
                       turns, rows, grid * 8, g);
    return hipGetLastError();
}

template <bool XBF16, int MT>
hipError_t go(const uint16_t* w, const void* x, float* y, uint32_t m, uint32_t n, uint32_t k, bool vec,
              hipStream_t s) {
    dim3 grid((n + 3) / 4, (m + MT - 1) / MT);
    if (vec)
        hipLaunchKernelGGL((bf16_matmul_kernel<XBF16, MT, true>), grid, dim3(256), 0, s, w, x, y, m, n, k);
    else
        hipLaunchKernelGGL((bf16_matmul_kernel<XBF16, MT, false>), grid, dim3(256), 0, s, w, x, y, m, n, k);
    return hipGetLastError();
}

}  // namespace

bool bf16_gemv_supported(uint32_t k, bool x_bf16) {
    // rows of whole 16-byte pieces; x (rounded up to whole turns) in 64 KiB of LDS
    return k >= 8 && k % 8 == 0 && (k + 2047) / 2048 * 2048 * (x_bf16 ? 2 : 4) <= 65536;
}

hipError_t launch_bf16_gemv(const uint16_t* const* w, float* const* y, const uint32_t* n, uint32_t count, const void* x,
                            bool x_bf16, uint32_t k, int cus, hipStream_t s) {
    if (count < 1 || count > 4 || !bf16_gemv_supported(k, x_bf16)) return hipErrorNotSupported;
    uint32_t rows = 0;
    for (uint32_t i = 0; i < count; ++i) {
        if (n[i] == 0) return hipErrorNotSupported;
        rows += n[i];
    }
    const uint32_t nc = (uint32_t)(cus > 0 ? cus : 256);
    Bf16Group g{};
    g.count = count;
    for (uint32_t i = 0; i < count; ++i) {
        g.w[i] = w[i];
        g.y[i] = y[i];
        g.n[i] = n[i];
        g.first[i + 1] = g.first[i] + n[i];
    }
    for (uint32_t i = count; i < 4; ++i) g.first[i + 1] = g.first[count];
    // four workgroups of eight waves per CU, the same number of rows for every wave
    uint32_t grid = (rows + 7) / 8;
    if (grid > 4 * nc) grid = 4 * nc;
    const uint32_t each = (rows + grid * 8 - 1) / (grid * 8);
    grid = (rows + each * 8 - 1) / (each * 8);
    if (k <= 1024) return x_bf16 ? go_gemv<true, 2>(g, x, k, rows, grid, s) : go_gemv<false, 2>(g, x, k, rows, grid, s);
    return x_bf16 ? go_gemv<true, 4>(g, x, k, rows, grid, s) : go_gemv<false, 4>(g, x, k, rows, grid, s);
}

// Two to 32 token rows: the row-per-wave kernel has n waves for every four of
// them, skinny_any.hip a workgroup of eight for every 16 weight rows; it reads
// the weights once, which pays where they are long. From a sweep of 16 to 16384
// weight rows, K = 256 .. 12288 and 2 to 32 token rows on MI355X (cold weights,
// recorded passes; no call is more than 8% slower than the other kernel would be,
// where skinny_any alone took up to 2.9 times as long), us, this one / skinny_any:
//  * bf16 x: 2048 x 2048 at 4 rows 5.5 / 6.0, 4096 x 2048 7.4 / 6.8, 4096 x 4096
//    11.9 / 12.3; 1024 x 4096 at 16 rows 9.3 / 11.6, 2048 x 4096 15.2 / 12.2; 512
//    x 8192 at 32 rows 13.6 / 26.1, 1024 x 8192 25.2 / 26.6. Up to four rows it
//    reads the weights once too: short rows stay here at any number of them
//    (16384 x 512 8.6 / 9.6);
//  * f32 x: 2048 x 2048 at 4 rows 5.7 / 7.8, 4096 x 2048 10.7 / 8.7; 2048 x 1024
//    at 8 rows 5.1 / 5.6; 1024 x 4096 at 16 rows 13.5 / 16.2, 2048 x 4096 22.9 /
//    16.7; 512 x 4096 at 32 rows 11.2 / 15.9, 1024 x 4096 21.7 / 16.1.
bool bf16_rows_faster(uint32_t m, uint32_t n, uint32_t k, bool x_bf16, int cus) {
    const uint64_t four = (m + 3) / 4, waves = (uint64_t)n * four;
    if (x_bf16 && m <= 4 && k <= 512) return true;
    uint64_t most = x_bf16 ? 3072 + 640 * four : 2560 + 384 * four;
    if (x_bf16 && m <= 4 && k >= 4096) most = 4096;
    if (!x_bf16 && k <= 2048) most = most * (k <= 512 ? 6 : 5) / 4;
    if (k <= 256 && most > (x_bf16 ? 3584u : 6144u)) most = x_bf16 ? 3584 : 6144;
    return waves * 256 <= most * (uint64_t)(cus > 0 ? cus : 256);
}

// Estimated time of the row-per-wave kernel for more than a few token rows: its
// waves at the rate they are launched at or, from K = 780 (f32 x: 510) on, at that
// of their products (within 10% of 1.4 thousand measured calls near where the
// matrix cores take over: 640 x 1024 at 33 / 300 rows 5.0 / 30 us, 128 x 12288 at
// 128 rows of f32 29).
double bf16_matmul_us(uint32_t m, uint32_t n, uint32_t k, bool x_bf16, int cus) {
    const double waves = (double)n * ((m + 3) / 4) * 256.0 / (cus > 0 ? cus : 256);
    const double each = (x_bf16 ? 3.6e-7 : 5.5e-7) * k;
    return 2.2 + waves * (each > 2.8e-4 ? each : 2.8e-4);
}

hipError_t launch_bf16_matmul(const uint16_t* w, const void* x, bool x_bf16, float* y, uint32_t m, uint32_t n,
                              uint32_t k, bool fine, hipStream_t s) {
    if (m == 0 || n == 0 || k == 0) return hipSuccess;
    // 16-byte pieces need every row (weights and activations) to start 16-byte aligned
    const uint32_t xalign = x_bf16 ? 8 : 4;
    const bool vec = k % 8 == 0 && k % xalign == 0 && ((uintptr_t)w & 15) == 0 && ((uintptr_t)x & 15) == 0;
    if (vec && fine && m > 1) {
        dim3 grid((n + 3) / 4, (m + 3) / 4);
        if (x_bf16)
            hipLaunchKernelGGL((bf16_matmul_fine_kernel<true>), grid, dim3(256), 0, s, w, x, y, m, n, k);
        else
            hipLaunchKernelGGL((bf16_matmul_fine_kernel<false>), grid, dim3(256), 0, s, w, x, y, m, n, k);
        return hipGetLastError();
    }
    if (m == 1) return x_bf16 ? go<true, 1>(w, x, y, m, n, k, vec, s) : go<false, 1>(w, x, y, m, n, k, vec, s);
    return x_bf16 ? go<true, 4>(w, x, y, m, n, k, vec, s) : go<false, 4>(w, x, y, m, n, k, vec, s);
}

}  // namespace mx4
