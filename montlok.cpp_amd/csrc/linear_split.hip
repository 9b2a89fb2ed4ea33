// Dense linear y = x W^T (+ bias, + residual) with fp32 weights on the bf16
// matrix cores, to fp32 accuracy.
//
// An fp32 value times 2^24 is the exact sum of three bf16 values (8 + 8 + 8 bits
// of its 24-bit significand; each part is the rounding of what the ones before
// it left, so their magnitudes fall by 2^-9 a step; the factor keeps the third
// part of the smallest subnormal, 2^-149, a normal bf16 value), so with x and w
// so enlarged
//
//   x w = x1 w1 + (x1 w2 + x2 w1) + (x1 w3 + x2 w2 + x3 w1) + O(2^-26 x w)
//
// and six v_mfma_f32_32x32x16_bf16 form, with every product exact and fp32
// accumulation, what the fp32 form needs eight v_mfma_f32_32x32x2_f32 for,
// at 0.4 of the matrix-core time (2.2 PFLOP/s bf16 and 155 TFLOP/s fp32
// measured on this chip). The first term and the other five are summed apart
// and added at the end, then returned to scale by 2^-48: the large sum then
// takes one rounding per 16 k, and the error against float64 is 8.5e-8 (2-norm,
// N(0, 1) x, K = 256; 1.2e-7 at K = 512) where the fp32 forms it replaces have
// 2.9e-7 (4.1e-7). Operands of 2^104 and more and results of 2^80 and more do
// not fit the enlarged form; they go the way of infinities, below.
//
//   block  = 64 rows x 64 columns of y, 4 waves of 32 x 32; K in steps of 32.
//            Large calls: 128 x 128, 4 waves of 64 x 64 that multiply and 4 that
//            stage, two LDS buffers. Up to 256 blocks: 8 waves, two a tile.
//   stage  = 16-row pieces of x and W, whole 128-byte lines per load (the
//            MFMA operand order straight from memory takes every line in four
//            separate instructions: 20-25% slower), split in registers and
//            written as three bf16 planes in LDS, in the operand order.
//   D      = transposed products (W as the A operand): lane (g, l) of a wave
//            holds row l, columns 8 j + 4 g .. + 3 (j = 0..3), 16-byte stores.
//
// What bounds it: the bf16 products. On random data this card's clocks hold a
// large bf16 matrix product at 1.1 PFLOP/s, 183 TFLOP/s of these sums, and
// 65536 x 512 -> 256 takes 101 us in the big blocks (170 TFLOP/s). The small
// blocks keep the matrix cores 43% busy (27 KiB of LDS, 84 registers, five
// blocks a CU in different phases: a step and SIMD takes 220 cycles of
// products and about as many of splitting); a second LDS buffer there, or deeper
// prefetch in either, was slower. Against the fp32 forms: 7680 x 256 -> 1192
// 69 -> 39 us, 7680 x 512 -> 256 33 -> 18, 15360 x 256 -> 1192 112 -> 68,
// 15360 x 512 -> 256 51 -> 26.5 (the enlargement's multiply: 0 to 3% of these).
//
// A sum past that range, or with an infinite operand, is infinite or NaN here
// (the parts of an infinity are inf and NaN). A wave that holds such a result
// and no NaN in the x row that explains it forms its tile again on the fp32
// matrix cores (plain_tile) and takes those results from there: the fp32 form's
// values, infinite or NaN where its are. Rows with a NaN are ordinary input
// (bars that are missing), so looking for it has to be cheap, and a serial sum
// of a lane's 16 results is not: 7680 x 512 -> 256 with one such row 513 us so,
// 28 with the look and 37 with the tile (22 without the row); all rows 1900
// and 31.

#include "linear_args.h"
#include "mlk_common.h"

namespace mlk {
namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

constexpr int kPlanes = 3, kStep = 32, kBlock = 64;
constexpr float kUp = 0x1p24f, kDown = 0x1p-48f;  // x and W are split 2^24 times as large, the sums returned from 2^48
constexpr int kMaxNormGroups = 32;  // RMSNorm groups of a row (K = 256 in groups of 8)

// 16-byte units of the LDS image of a 32-row x 32-k tile: [k half][plane][lane group][32 rows]. The groups are
// 576 bytes apart, so that the eight lanes that write one row's two halves and groups hit different banks.
constexpr int kGroupUnits = 36, kTileUnits = 2 * kPlanes * 2 * kGroupUnits;
__device__ __forceinline__ unsigned unit(int tile, int half, int plane, int group) {
    return tile * kTileUnits + ((half * kPlanes + plane) * 2 + group) * kGroupUnits;
}

// Two floats to one plane's packed bf16 pair; v keeps what the pair leaves.
__device__ __forceinline__ uint32_t take_bf16(f32x2& v) {
    const uint32_t u = __builtin_bit_cast(uint32_t, __builtin_convertvector(v, bf16x2));
    v[0] -= __builtin_bit_cast(float, u << 16);
    v[1] -= __builtin_bit_cast(float, u & 0xffff0000u);
    return u;
}

// rms_norm's scale of each (row, group) of the block's 64 rows: per 4 floats (a^2 + b^2) + (c^2 + d^2) in fp64,
// the chunks of a group combined highest index bit first, as tile_rms_norm and rms_norm_vec_kernel do.
template <int GS>
__device__ __forceinline__ void norm_scales(const LinearArgs& p, int64_t row0, int groups, double* scale) {
    for (int u = threadIdx.x; u < kBlock * groups; u += blockDim.x) {
        const int64_t row = row0 + u / groups;
        const float* x = p.x + (row < p.rows ? row : p.rows - 1) * p.x_stride + (u % groups) * GS;
        double part[GS / 4];
#pragma unroll
        for (int c = 0; c < GS / 4; ++c) {
            const float4 f = *reinterpret_cast<const float4*>(x + 4 * c);
            const double a = f.x, b = f.y, e = f.z, d = f.w;
            part[c] = (a * a + b * b) + (e * e + d * d);
        }
#pragma unroll
        for (int n = GS / 8; n >= 1; n /= 2)
#pragma unroll
            for (int c = 0; c < n; ++c) part[c] += part[c + n];
        scale[u] = 1.0 / sqrt(part[0] / static_cast<double>(GS) + p.norm_eps);
    }
}

// A wave's 32 x 32 tile of sums on the fp32 matrix cores, as linear's fp32 forms take them: lane (g, l) passes the
// k 8 s + 4 g .. + 3 of its own row of x and of W (for GS > 0 normalised as norm_scales' row scales say), read from
// memory, and gets row l of x, W rows 8 j + 4 g .. + 3. All lanes of the wave are active.
template <int GS>
__device__ __forceinline__ f32x16 plain_tile(const float* x, const float* w, int K, int g, const double* scale, const float* norm_w) {
    constexpr int kAhead = 4;  // 8-wide steps whose loads are in flight together
    f32x16 sum;
#pragma unroll
    for (int c = 0; c < 16; ++c) sum[c] = 0.0f;
#pragma unroll 1
    for (int k0 = 0; k0 < K; k0 += 8 * kAhead) {
        float4 xv[kAhead], wv[kAhead];
#pragma unroll
        for (int s = 0; s < kAhead; ++s) {
            const int k = k0 + 8 * s + 4 * g, kc = k < K ? k : 0;
            xv[s] = *reinterpret_cast<const float4*>(x + kc);
            wv[s] = *reinterpret_cast<const float4*>(w + kc);
        }
#pragma unroll
        for (int s = 0; s < kAhead; ++s) {
            const int k = k0 + 8 * s + 4 * g;
            const bool live = k < K;
            float xs[4] = {xv[s].x, xv[s].y, xv[s].z, xv[s].w}, ws[4] = {wv[s].x, wv[s].y, wv[s].z, wv[s].w};
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                if constexpr (GS > 0) {
                    const int kc = live ? k : 0;
                    xs[j] = static_cast<float>((static_cast<double>(xs[j]) * scale[kc / GS]) * static_cast<double>(norm_w[kc + j]));
                }
                sum = __builtin_amdgcn_mfma_f32_32x32x2f32(live ? ws[j] : 0.0f, live ? xs[j] : 0.0f, sum, 0, 0, 0);
            }
        }
    }
    return sum;
}

// Whether row l of x (lanes l and l + 32, K floats) holds a NaN.
__device__ __forceinline__ bool row_has_nan(const float* x, int K, int g, int li) {
    constexpr int kAhead = 8;
    bool found = false;
#pragma unroll 1
    for (int k0 = 0; k0 < K; k0 += 8 * kAhead) {
        float4 v[kAhead];
#pragma unroll
        for (int s = 0; s < kAhead; ++s) {
            const int k = k0 + 8 * s + 4 * g;
            v[s] = *reinterpret_cast<const float4*>(x + (k < K ? k : 0));
        }
#pragma unroll
        for (int s = 0; s < kAhead; ++s) found = found || __builtin_isunordered(v[s].x, v[s].y) || __builtin_isunordered(v[s].z, v[s].w);
    }
    const uint64_t lanes = __ballot(found);
    return ((lanes | lanes >> 32) >> li & 1) != 0;
}

// FULL: K a multiple of the step. GS > 0: the grouped RMSNorm of x (groups of GS floats, at most kMaxNormGroups
// of them) applied to the staged values, bit for bit rms_norm then this kernel. SWIGLU: W holds 2 N rows, gate
// then up; a wave's W tile is 16 gate rows and the 16 up rows of the same columns, so that a lane holds both
// of its outputs' factors, and out = silu(gate) * up in fp64, rounded once (p.N = hidden columns of out). The
// 2 N columns then never reach memory: 7680 x 256 -> 2 x 512 36 us, against 38 for the linear and 13 for swiglu.
// T: the wave tile is (32 T) x (32 T), the block (64 T) x (64 T). T = 2 has four more waves that stage (PRODUCER
// below) while the first four multiply, with two LDS buffers and one barrier a step.
// PAIR (T = 1, few blocks): eight waves to the 64 x 64 block, two to a tile, one for each k half of a step; their
// sums meet in LDS.
template <bool FULL, int GS, bool SWIGLU, int T, bool PAIR>
__global__ __launch_bounds__(T == 1 && !PAIR ? 256 : 512, T == 2 ? 2 : 1) void linear_split_kernel(LinearArgs p, unsigned n_blocks) {
    static_assert(T == 1 || (GS == 0 && !PAIR), "the norm's prologue and the pairs are the 64 x 64 block's");
    constexpr int MS = PAIR ? 1 : 2;  // 8-row loads a staging wave issues per 64 rows
    constexpr int kRows = kBlock * T, kCols = SWIGLU ? kRows / 2 : kRows;  // rows, output columns of the block
    constexpr int kBuffer = 4 * T * kTileUnits;  // x tiles 0 .. 2 T - 1, then W tiles
    __shared__ uint4 frag[T * kBuffer];
    __shared__ double scale[GS > 0 ? kBlock * kMaxNormGroups : 1];
    const int lane = threadIdx.x & 63, li = lane & 31, g = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6) & 3;
    const int upper = __builtin_amdgcn_readfirstlane(threadIdx.x >> 8);  // 1: T = 2's staging waves, a pair's second
    const bool producer = T == 1 || upper == 1;
    // XCD x takes the x-th eighth of the blocks, column blocks of one row block side by side: a row block's x
    // is fetched into one L2.
    unsigned lin = blockIdx.x;
    if (gridDim.x % 8 == 0) lin = (lin % 8) * (gridDim.x / 8) + lin / 8;
    const int64_t row0 = static_cast<int64_t>(lin / n_blocks) * kRows;
    const int64_t n0 = static_cast<int64_t>(lin % n_blocks) * kCols;
    const int K = static_cast<int>(p.K);
    const int groups = GS > 0 ? K / GS : 0;
    const float* w = static_cast<const float*>(p.w);

    // Staging wave w takes rows 64 i + 16 w .. + 15 of x and of W: lane 8 r + c of a load holds k = 4 c .. + 3 of
    // row r (of 8), whole lines; byte offsets in 32 bits from the block's first row (strides checked at launch).
    const int sr = lane >> 3, sc = lane & 7;
    const char* base[2] = {reinterpret_cast<const char*>(p.x + row0 * p.x_stride), reinterpret_cast<const char*>(w + n0 * p.K)};
    unsigned off[2][T][MS];
    float4 v[2][T][MS], nw;
    bool live = true;  // of the fetched step (K a multiple of 4: a lane's 4 k are on one side of it)
    auto rows = [&]() {
#pragma unroll
        for (int i = 0; i < T; ++i)
#pragma unroll
            for (int m = 0; m < MS; ++m) {
                const int r = 64 * i + 16 * wave + 8 * (PAIR ? upper : m) + sr;
                off[0][i][m] = static_cast<unsigned>((row0 + r < p.rows ? r : p.rows - 1 - row0) * p.x_stride * 4) + 16 * sc;
                int64_t n = r;
                if constexpr (SWIGLU) {
                    const int64_t col = 32 * i + 16 * (wave >> 1) + 8 * (PAIR ? upper : m) + sr;
                    n = (n0 + col < p.N ? col : p.N - 1 - n0) + (wave & 1 ? p.N : 0);
                } else {
                    n = n0 + n < p.N ? n : p.N - 1 - n0;
                }
                off[1][i][m] = static_cast<unsigned>(n * p.K * 4) + 16 * sc;
            }
    };
    auto fetch = [&](int k0) {
        live = k0 + 4 * sc < K;
        const unsigned ko = FULL ? (k0 < K ? 4 * k0 : 0u) : (live ? 4 * k0 : 0u - 16 * sc);
#pragma unroll
        for (int o = 0; o < 2; ++o)
#pragma unroll
            for (int i = 0; i < T; ++i)
#pragma unroll
                for (int m = 0; m < MS; ++m)
                    v[o][i][m] = *reinterpret_cast<const float4*>(base[o] + static_cast<unsigned>(off[o][i][m] + ko));
        if constexpr (GS > 0) nw = *reinterpret_cast<const float4*>(p.norm_w + (live ? k0 + 4 * sc : 0));
    };
    // Values past K become zeros here and not at the load, whose wait would then stand in front of the products.
    auto stage = [&](int k0, int buffer) {
        uint2* dst = reinterpret_cast<uint2*>(frag + buffer * kBuffer);
#pragma unroll
        for (int o = 0; o < 2; ++o)
#pragma unroll
            for (int i = 0; i < T; ++i)
#pragma unroll
                for (int m = 0; m < MS; ++m) {
                    const int r8 = 8 * (PAIR ? upper : m) + sr;  // of the wave's 16 rows
                    float4 f = v[o][i][m];
                    if (GS > 0 && o == 0) {
                        const int k = live ? k0 + 4 * sc : 0;
                        const double s = scale[(16 * wave + r8) * groups + k / (GS > 0 ? GS : 1)];
                        f.x = static_cast<float>((static_cast<double>(f.x) * s) * static_cast<double>(nw.x));
                        f.y = static_cast<float>((static_cast<double>(f.y) * s) * static_cast<double>(nw.y));
                        f.z = static_cast<float>((static_cast<double>(f.z) * s) * static_cast<double>(nw.z));
                        f.w = static_cast<float>((static_cast<double>(f.w) * s) * static_cast<double>(nw.w));
                    }
                    if (!FULL && !live) f = float4{0.0f, 0.0f, 0.0f, 0.0f};
                    f32x2 lo = {f.x * kUp, f.y * kUp}, hi = {f.z * kUp, f.w * kUp};
                    const unsigned slot = unit(2 * (o * T + i) + (wave >> 1), sc >> 2, 0, (sc >> 1) & 1) + 16 * (wave & 1) + r8;
#pragma unroll
                    for (int q = 0; q < kPlanes; ++q) dst[2 * (slot + q * 2 * kGroupUnits) + (sc & 1)] = uint2{take_bf16(lo), take_bf16(hi)};
                }
    };

    const int wm = wave & 1, wn = wave >> 1;
    f32x16 acc[T][T], low[T][T];  // [x tile][W tile]
#pragma unroll
    for (int i = 0; i < T; ++i)
#pragma unroll
        for (int j = 0; j < T; ++j)
#pragma unroll
            for (int c = 0; c < 16; ++c) acc[i][j][c] = low[i][j][c] = 0.0f;
    auto multiply = [&](int buffer) {
        const uint4* src = frag + buffer * kBuffer;
#pragma unroll
        for (int hh = 0; hh < (PAIR ? 1 : 2); ++hh) {
            const int h = PAIR ? upper : hh;
            bf16x8 xf[T][kPlanes], wf[T][kPlanes];
#pragma unroll
            for (int q = 0; q < kPlanes; ++q)
#pragma unroll
                for (int i = 0; i < T; ++i) {
                    xf[i][q] = __builtin_bit_cast(bf16x8, src[unit(wm * T + i, h, q, g) + li]);
                    wf[i][q] = __builtin_bit_cast(bf16x8, src[unit(2 * T + wn * T + i, h, q, g) + li]);
                }
#pragma unroll
            for (int order = 0; order < kPlanes; ++order)
#pragma unroll
                for (int q = 0; q <= order; ++q)
#pragma unroll
                    for (int i = 0; i < T; ++i)
#pragma unroll
                        for (int j = 0; j < T; ++j) {
                            f32x16& c = order == 0 ? acc[i][j] : low[i][j];
                            c = __builtin_amdgcn_mfma_f32_32x32x16_bf16(wf[j][q], xf[i][order - q], c, 0, 0, 0);
                        }
        }
    };

    if constexpr (T == 1) {
        rows();
        fetch(0);
        if constexpr (GS > 0) {
            norm_scales<(GS > 0 ? GS : 8)>(p, row0, groups, scale);
            __syncthreads();
        }
        if constexpr (FULL) {  // (apart: left in the loop, the compiler keeps a second set of sums, four blocks a CU)
            stage(0, 0);
            __syncthreads();
            fetch(kStep);
            multiply(0);
        }
        for (int k0 = FULL ? kStep : 0; k0 < K; k0 += kStep) {
            if (k0 > 0) __syncthreads();
            stage(k0, 0);
            __syncthreads();
            fetch(k0 + kStep);
            multiply(0);
        }
    } else if (producer) {
        rows();
        fetch(0);
        stage(0, 0);
        fetch(kStep);
        int buffer = 1;
        for (int k0 = 0; k0 < K; k0 += kStep, buffer ^= 1) {
            __syncthreads();
            stage(k0 + kStep, buffer);  // (past K: loads of the first columns, not read)
            fetch(k0 + 2 * kStep);
        }
        return;
    } else {
        int buffer = 0;
        for (int k0 = 0; k0 < K; k0 += kStep, buffer ^= 1) {
            __syncthreads();
            multiply(buffer);
        }
    }

    if constexpr (PAIR) {
        // (the fragments of the last step are done with: their LDS takes the second waves' sums)
        float* part = reinterpret_cast<float*>(frag) + wave * 16 * 64 + lane;
        static_assert(sizeof(frag) >= 4 * 16 * 64 * sizeof(float), "the sums fit the fragments' LDS");
        __syncthreads();
        if (upper == 1) {
#pragma unroll
            for (int c = 0; c < 16; ++c) part[64 * c] = acc[0][0][c] + low[0][0][c];
        }
        __syncthreads();
        if (upper == 1) return;
#pragma unroll
        for (int c = 0; c < 16; ++c) low[0][0][c] += part[64 * c];
    }
    const bool vec_out = (reinterpret_cast<uintptr_t>(p.out) & 15) == 0 && p.out_stride % 4 == 0 &&
                         (p.residual == nullptr ||
                          ((reinterpret_cast<uintptr_t>(p.residual) & 15) == 0 && p.res_stride % 4 == 0));
#pragma unroll
    for (int i = 0; i < T; ++i) {
        const int64_t row = row0 + 32 * (wm * T + i) + li;
        const float* xr = p.x + (row < p.rows ? row : p.rows - 1) * p.x_stride;
        bool looked = false, nan_row = false;  // (looked: the same in every lane)
#pragma unroll
        for (int t = 0; t < T; ++t) {
            f32x16& y = acc[i][t];
#pragma unroll
            for (int c = 0; c < 16; ++c) y[c] = (y[c] + low[i][t][c]) * kDown;
            // W row of accumulator element c (0 .. 15), and its column of out.
            auto w_row = [&](int c) -> int64_t {
                const int r = 8 * (c >> 2) + 4 * g + (c & 3);
                if constexpr (SWIGLU) return n0 + 16 * (wn * T + t) + (r & 15) + (r & 16 ? p.N : 0);
                return n0 + 32 * (wn * T + t) + r;
            };
            auto in_range = [&](int c) {
                if constexpr (SWIGLU) return w_row(c & 7) < p.N;
                return w_row(c) < p.N;
            };
            bool whole = true;
#pragma unroll
            for (int c = 0; c < 16; ++c) whole = whole && fabsf(y[c]) < INFINITY;
            bool again = __ballot(!whole) != 0;
            if (again) {
                if (!looked) nan_row = row_has_nan(xr, K, g, li);
                looked = true;
                again = __ballot(!whole && !nan_row) != 0;
            }
            if (again) {
                int64_t wr = n0 + (SWIGLU ? 16 * (wn * T + t) + (li & 15) : 32 * (wn * T + t) + li);
                wr = (wr < p.N ? wr : p.N - 1) + (SWIGLU && li >= 16 ? p.N : 0);
                f32x16& plain = low[i][t];
                plain = plain_tile<GS>(xr, w + wr * p.K, K, g, scale + (GS > 0 ? (32 * wm + li) * groups : 0), p.norm_w);
#pragma unroll
                for (int c = 0; c < 16; ++c) y[c] = fabsf(y[c]) < INFINITY ? y[c] : plain[c];
            }
            if (row >= p.rows) continue;
            if (p.bias != nullptr) {
#pragma unroll
                for (int c = 0; c < 16; ++c) y[c] += p.bias[in_range(c) ? w_row(c) : 0];
            }
#pragma unroll
            for (int j = 0; j < (SWIGLU ? 2 : 4); ++j) {
                const int64_t col = w_row(4 * j);
                if (col >= p.N) continue;
                f32x4 o = {y[4 * j], y[4 * j + 1], y[4 * j + 2], y[4 * j + 3]};
                if constexpr (SWIGLU) {
#pragma unroll
                    for (int c = 0; c < 4; ++c)
                        o[c] = static_cast<float>(silu_d(static_cast<double>(o[c])) * static_cast<double>(y[8 + 4 * j + c]));
                }
                float* dst = p.out + row * p.out_stride + col;
                const float* res = p.residual != nullptr ? p.residual + row * p.res_stride + col : nullptr;
                if (vec_out && col + 4 <= p.N) {
                    if (res != nullptr) o = *reinterpret_cast<const f32x4*>(res) + o;
                    *reinterpret_cast<f32x4*>(dst) = o;
                } else {
#pragma unroll
                    for (int c = 0; c < 4; ++c)
                        if (col + c < p.N) dst[c] = res != nullptr ? res[c] + o[c] : o[c];
                }
            }
        }
    }
}

template <int GS, bool SWIGLU, int T, bool PAIR = false>
void launch_blocks(const LinearArgs& p, hipStream_t stream) {
    const int64_t nb = ceil_div(p.N, (SWIGLU ? kBlock / 2 : kBlock) * T);
    const dim3 grid(static_cast<unsigned>(ceil_div(p.rows, kBlock * T) * nb)), threads(T == 1 && !PAIR ? 256 : 512);
    if (p.K % kStep == 0) {
        hipLaunchKernelGGL((linear_split_kernel<true, GS, SWIGLU, T, PAIR>), grid, threads, 0, stream, p, static_cast<unsigned>(nb));
    } else {
        hipLaunchKernelGGL((linear_split_kernel<false, GS, SWIGLU, T, PAIR>), grid, threads, 0, stream, p, static_cast<unsigned>(nb));
    }
}

// Whether rounds of 256 blocks of 128 x 128 (one a CU) are filled to nine tenths by the call's rows and columns.
// Then the big blocks, which split every operand half as often and multiply while they split, are the faster ones
// (15360 x 512 -> 256, 240 blocks: 28 us against 33; 65536 x 512 -> 256: 102 against 114; 7680 x 256 -> 1024, 480
// blocks: 30 against 32); otherwise their last round, or the columns past N, cost more than that (7680 x 256 ->
// 1192, 600 blocks: 41 against 36; 7680 x 512 -> 256, 120 blocks: 21 against 18).
bool fills_big_blocks(int64_t rows, int64_t w_rows) {
    const int64_t blocks = ceil_div(rows, 2 * kBlock) * ceil_div(w_rows, 2 * kBlock);
    const double held = static_cast<double>(ceil_div(blocks, 256) * 256) * (4 * kBlock * kBlock);
    return static_cast<double>(rows) * static_cast<double>(w_rows) >= 0.9 * held;
}

// Up to one 64 x 64 block a CU, a step is a chain of one wave a SIMD (load, split, products); eight waves halve its
// parts: 480 x 512 -> 256 13.1 -> 11.2 us, 3840 x 256 -> 256 (240 blocks) 8.7 -> 8.0, 3840 x 1024 -> 256 25.8 -> 21.2.
// Past that the second block of a CU fills the gaps as well: 2880 x 256 -> 352 (270 blocks) 10.0 in both, 5760 x 256 ->
// 256 (360) 10.4 against 10.7, 2880 x 256 -> 1192 (855) 17.7 against 20.0.
bool few_blocks(int64_t rows, int64_t w_rows) { return ceil_div(rows, kBlock) * ceil_div(w_rows, kBlock) <= 256; }

template <int GS, bool SWIGLU>
void launch(const LinearArgs& p, hipStream_t stream) {
    if constexpr (GS == 0) {
        if (fills_big_blocks(p.rows, SWIGLU ? 2 * p.N : p.N)) {
            launch_blocks<0, SWIGLU, 2>(p, stream);
            return;
        }
    }
    if (few_blocks(p.rows, SWIGLU ? 2 * p.N : p.N)) {
        launch_blocks<GS, SWIGLU, 1, true>(p, stream);
    } else {
        launch_blocks<GS, SWIGLU, 1>(p, stream);
    }
}

// 32-bit byte offsets from a block's first rows, and the grid.
bool fits(const LinearArgs& p, int64_t w_rows) {
    return p.K % 4 == 0 && p.x_stride < (int64_t{1} << 23) && p.K * (w_rows + 2 * kBlock) < (int64_t{1} << 30) &&
           ceil_div(p.rows, kBlock) * ceil_div(p.N, kBlock / 2) < (int64_t{1} << 31);
}

}  // namespace

bool linear_split_fits(const LinearArgs& p) { return fits(p, kBlock); }

void launch_linear_split(const LinearArgs& p, hipStream_t stream) { launch<0, false>(p, stream); }

void launch_linear_split_norm(const LinearArgs& p, int64_t group_size, hipStream_t stream) {
    switch (group_size) {
        case 8: launch<8, false>(p, stream); break;
        case 16: launch<16, false>(p, stream); break;
        case 32: launch<32, false>(p, stream); break;
        default: launch<64, false>(p, stream); break;
    }
}

bool linear_swiglu_fits(const LinearArgs& p) { return fits(p, 2 * p.N); }

void launch_linear_swiglu(const LinearArgs& p, hipStream_t stream) { launch<0, true>(p, stream); }

}  // namespace mlk
