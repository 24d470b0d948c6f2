// kt_split.hip -- products with quantized weights in fp32 precision on the bf16 matrix units.
//
// An integer weight q - zero has at most 8 significant bits, so it is a bf16 number
// exactly; an fp32 number is the exact sum of three bf16 numbers (its 24 significant bits
// cut into 8 + 8 + 8, the lower parts exact while they stay above 2^-126). A product of
// fp32 data and integer weights is therefore three v_mfma_f32_32x32x16_bf16 whose products
// are exact and whose sums are fp32: the precision of an fp32 multiply-add chain at a
// third of the bf16 rate (about 5 times the fp32 matrix rate).
//
//   forward: c[M x N] = a[M x K] . deq(W) (MatMul.multiplyQuantized, Engine/kotensor/src/main/
//   kotlin/MatMul.kt:479-485) of the shapes and alignments the fp16 GEMM does not take; the
//   scale of a k-group multiplies the group's sum.
//   transposed: dX[M x K] = dY[M x N] . deq(W)^T (MatMul.multiplyByQuantizedTransposed,
//   MatMul.kt:954-981). The sum runs over n, along which
//   the scale changes, so a lane multiplies its dY values by the scales of the k-group
//   first (one fp32 rounding, in the place of the one of deq(W)) and splits the product.
#include <algorithm>

#include "kt_common.h"
#include "kt_packed.h"
#include "kt_split.h"

namespace kt {
namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int THREADS = 256;
constexpr int STEP = 64;          // elements of the summed dimension per step
constexpr int PITCH = STEP + 8;   // halfs per LDS row: 16-byte reads of 16 consecutive rows hit all banks once
constexpr int MAX_SPLITS = 32;

// The dword at byte i of a row of `bytes` >= 4 bytes; bytes past the row's end are any.
__device__ __forceinline__ uint32_t load_end(const void* row, int32_t i, int32_t bytes) {
    const int32_t at = min(i, bytes - 4);
    return load_any<uint32_t>(static_cast<const uint8_t*>(row) + at) >> (8 * min(i - at, 3));
}

template <int I>
__device__ __forceinline__ float ubyte(uint32_t w) {
    return static_cast<float>((w >> (8 * I)) & 0xFFu);
}
// Eight unsigned bytes minus eight others (or minus 128) as bf16 integers.
__device__ __forceinline__ u32x4 diff8(uint32_t a0, uint32_t a1, uint32_t b0, uint32_t b1) {
    return u32x4{upper_halves(ubyte<0>(a0) - ubyte<0>(b0), ubyte<1>(a0) - ubyte<1>(b0)),
                 upper_halves(ubyte<2>(a0) - ubyte<2>(b0), ubyte<3>(a0) - ubyte<3>(b0)),
                 upper_halves(ubyte<0>(a1) - ubyte<0>(b1), ubyte<1>(a1) - ubyte<1>(b1)),
                 upper_halves(ubyte<2>(a1) - ubyte<2>(b1), ubyte<3>(a1) - ubyte<3>(b1))};
}
__device__ __forceinline__ u32x4 diff8_128(uint32_t a0, uint32_t a1) {
    return u32x4{upper_halves(ubyte<0>(a0) - 128.0f, ubyte<1>(a0) - 128.0f),
                 upper_halves(ubyte<2>(a0) - 128.0f, ubyte<3>(a0) - 128.0f),
                 upper_halves(ubyte<0>(a1) - 128.0f, ubyte<1>(a1) - 128.0f),
                 upper_halves(ubyte<2>(a1) - 128.0f, ubyte<3>(a1) - 128.0f)};
}

// Of the rows (bit r: row first + r of a [.. x width]) that hold elements of a wave's `nans`
// (element e of a block of 16: row 8 (e / 4) + 4 (lane / 32) + e % 4), those with a NaN among the
// columns [from, to) or [from2, to2): their sums are NaNs.
__device__ __forceinline__ uint32_t nan_rows(uint64_t nans, const float* a, size_t width, int32_t from, int32_t to, int32_t from2,
                                             int32_t to2) {
    const int32_t ln = threadIdx.x & 63;
    uint32_t mine = static_cast<uint32_t>(nans | nans >> 16 | nans >> 32 | nans >> 48) & 0xFFFFu, rows = 0;
#pragma unroll
    for (int e = 0; e < 16; ++e) {
        const uint64_t hit = __ballot(mine >> e & 1);
        rows |= ((hit & 0xFFFFFFFFull) ? 1u : 0u) << (8 * (e >> 2) + (e & 3));
        rows |= (hit >> 32 ? 1u : 0u) << (8 * (e >> 2) + 4 + (e & 3));
    }
    uint32_t found = 0;
    for (; rows; rows &= rows - 1) {
        const int32_t r = __builtin_ctz(rows);
        const float* row = a + r * width;
        bool nan = false;
        for (int32_t j = from + ln; j < to; j += 64) nan = nan || row[j] != row[j];
        for (int32_t j = from2 + ln; j < to2; j += 64) nan = nan || row[j] != row[j];
        if (__ballot(nan)) found |= 1u << r;
    }
    return found;
}

struct SplitArgs {
    const float* a;       // [M x N] dY
    const uint8_t* q;
    const float* s;
    const int8_t* z;
    float* out;           // [M x K], or the slices' sums [splits][M][K]
    int32_t M, K, N, bpr, g, G, tiles_m, splits, steps, steps_per_split, run, accumulate;
};

// Workgroup (tile of 32 WM rows of dY and 128 WK weight rows, slice of n): each of the
// four waves owns 32 rows x 128 weight rows (k), wave w row block w % WM and k tile w / WM.
// A step is 64 n: for INT4 32 bytes of each weight row (32 low-nibble and 32 high-nibble
// columns), for INT8 64 bytes. The workgroup turns them into bf16 integers in LDS once
// (q - zero; INT8 rows are dequantized without zero points, as dequantizeRow does); a
// wave's own dY values stay in registers, multiplied by the scales and split there once
// per scale group of its k tile (GB 32-row blocks of weights share a group).
// A step's 12 matrix products of a block start from zero and their sum joins the running
// sum with one fp32 add: few roundings lie on the long sum (one running sum in the matrix
// unit over all of a slice had 3.0e-7 of the 2-norm at N = 8192 where this has 1.15e-7 and
// the row-by-row kernel 1.26e-7).
// Bound by vector ALU work: about 700 instructions per wave and step, two thirds of them the
// splits, beside 48 matrix products (35% of the matrix units' time). M = 512, K = 2048,
// N = 8192, INT4: the call with the slices' sum 76 us at g = 64, 226 TFLOP/s (row by row on
// the vector ALU: 2850 us), 70 at g = 128, 97 at g = 32; traced one by one the two kernels
// take 75.7 and 8.6 us.
template <int BITS, int WM, int GB>
__global__ void __launch_bounds__(THREADS, 2) transposed_split_kernel(SplitArgs p) {
    constexpr int WK = 4 / WM, TK = 128 * WK, GW = 4 / GB, GT = WK * GW;
    constexpr int SB = BITS == 4 ? 32 : 64;    // bytes of a weight row per step
    constexpr int ROWS = TK / 128;             // weight rows a thread converts (half a row's bytes each)
    constexpr int WV = SB / 32;                // 16-byte loads of a half row
    constexpr int SN = (GT * STEP + THREADS - 1) / THREADS;  // scales (zero points) a thread stages
    __shared__ __attribute__((aligned(16))) uint16_t bs[TK * PITCH];
    __shared__ __attribute__((aligned(16))) float ss[GT * STEP];
    // zero points + 128 of two steps: a step's are read while the next one's are written
    __shared__ __attribute__((aligned(16))) uint8_t zs[BITS == 4 ? 2 : 1][BITS == 4 ? GT * STEP : 16];
    const int32_t sp = blockIdx.x % p.splits, tile = blockIdx.x / p.splits;
    const int32_t m0 = (tile % p.tiles_m) * 32 * WM, k0 = (tile / p.tiles_m) * TK;
    const int32_t t = threadIdx.x, ln = t & 63, hl = ln >> 5;
    const int32_t wave = __builtin_amdgcn_readfirstlane(t >> 6);
    const int32_t wm = wave % WM, wk = wave / WM;
    const int32_t slice_end = min((sp + 1) * p.steps_per_split, p.steps);
    const int32_t N = p.N, bpr = p.bpr;

    // Operands are addressed as a base of the wave plus a lane's 32-bit byte offset.
    // This lane's dY row (a row past M repeats the last; its sums are dropped).
    const int32_t row_a = m0 + 32 * wm;
    const char* abase = reinterpret_cast<const char*>(p.a + static_cast<size_t>(min(row_a, p.M - 1)) * N);
    const uint32_t a_off = static_cast<uint32_t>(max(min(ln & 31, p.M - 1 - row_a), 0)) * N * 4u;
    // The weight rows and half (16 or 32 bytes of the step) this thread converts.
    const int32_t r0 = t >> 1, hf = t & 1;
    const char* wbase = reinterpret_cast<const char*>(p.q) + static_cast<size_t>(k0) * bpr;
    uint32_t w_off[ROWS];
#pragma unroll
    for (int i = 0; i < ROWS; ++i) w_off[i] = static_cast<uint32_t>(min(r0 + 128 * i, p.K - 1 - k0)) * bpr;
    // The scales (zero points) it stages: element e of [GT][STEP], column sc_c of the step.
    const int32_t g0 = k0 / p.g;
    const char* sbase = reinterpret_cast<const char*>(p.s + static_cast<size_t>(g0) * N);
    const char* zbase = reinterpret_cast<const char*>(p.z) + (BITS == 4 ? static_cast<size_t>(g0) * N : 0);
    const int32_t sc_c = t % STEP;  // THREADS % STEP == 0
    uint32_t sc_row[SN];
#pragma unroll
    for (int i = 0; i < SN; ++i) {
        const int32_t gi = min((t + THREADS * i) / STEP, GT - 1);
        sc_row[i] = static_cast<uint32_t>(min((k0 + 32 * GB * gi) / p.g, p.G - 1) - g0) * N;
    }

    u32x4 w[ROWS][WV];
    float sv[SN];
    uint32_t zv[SN];
    // Column of element c of the step at byte column j0 (bases advance by whole steps).
    auto column = [&](int32_t j0, int32_t c) { return BITS == 4 && c >= 32 ? bpr + j0 + c - 32 : j0 + c; };
    auto valid = [&](int32_t n, int32_t c) { return n < N && (BITS == 8 || c >= 32 || n < bpr); };
    const uint32_t sc_n = BITS == 4 && sc_c >= 32 ? bpr + sc_c - 32 : sc_c;
    auto load_w = [&](int32_t x) {  // a step whose columns all exist
        const int32_t j0 = x * SB;
#pragma unroll
        for (int i = 0; i < ROWS; ++i)
#pragma unroll
            for (int v = 0; v < WV; ++v) w[i][v] = load_any<u32x4>(wbase + j0 + (w_off[i] + hf * (SB / 2) + 16 * v));
#pragma unroll
        for (int i = 0; i < SN; ++i) sv[i] = load_any<float>(sbase + 4 * static_cast<int64_t>(j0) + (sc_row[i] + sc_n) * 4u);
    };
    auto load_z = [&](int32_t x) {
        if constexpr (BITS == 4) {
            const int32_t n = column(x * SB, sc_c);  // may lie past the end
#pragma unroll
            for (int i = 0; i < SN; ++i) zv[i] = static_cast<uint8_t>(zbase[sc_row[i] + static_cast<uint32_t>(min(n, N - 1))]);
        }
    };
    auto store_z = [&](int32_t x) {
        if constexpr (BITS == 4) {
#pragma unroll
            for (int i = 0; i < SN; ++i)
                if (t + THREADS * i < GT * STEP) zs[x & 1][t + THREADS * i] = static_cast<uint8_t>(zv[i] ^ 0x80u);
        }
    };
    auto load_a = [&](float (&a)[8], int32_t x, int u) {  // a step whose columns all exist
        const int32_t j0 = x * SB;
        const char* src = abase + 4 * static_cast<int64_t>(BITS == 4 && u >= 2 ? bpr + j0 - 32 : j0) + (a_off + (64u * u + 32u * hl));
        const f32x4 v0 = load_any<f32x4>(src), v1 = load_any<f32x4>(src + 16);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            a[e] = v0[e];
            a[4 + e] = v1[e];
        }
    };
    auto convert = [&](int32_t x) {
#pragma unroll
        for (int i = 0; i < ROWS; ++i) {
            uint16_t* row = bs + (r0 + 128 * i) * PITCH;
            const uint8_t* zr = BITS == 4 ? zs[x & 1] + ((r0 + 128 * i) / (32 * GB)) * STEP + 16 * hf : nullptr;
#pragma unroll
            for (int c = 0; c < 2 * WV; ++c) {  // 8 bytes: columns 8 c .. of the half row
                const uint32_t w0 = w[i][c / 2][2 * (c & 1)], w1 = w[i][c / 2][2 * (c & 1) + 1];
                if constexpr (BITS == 8) {
                    *reinterpret_cast<u32x4*>(row + 32 * hf + 8 * c) = diff8_128(w0 ^ 0x80808080u, w1 ^ 0x80808080u);
                } else {  // a nibble and a zero point, both plus 128
                    const uint2 zl = *reinterpret_cast<const uint2*>(zr + 8 * c);
                    const uint2 zh = *reinterpret_cast<const uint2*>(zr + 32 + 8 * c);
                    *reinterpret_cast<u32x4*>(row + 16 * hf + 8 * c) =
                        diff8((w0 & 0x0F0F0F0Fu) | 0x80808080u, (w1 & 0x0F0F0F0Fu) | 0x80808080u, zl.x, zl.y);
                    *reinterpret_cast<u32x4*>(row + 32 + 16 * hf + 8 * c) =
                        diff8(((w0 >> 4) & 0x0F0F0F0Fu) | 0x80808080u, ((w1 >> 4) & 0x0F0F0F0Fu) | 0x80808080u, zh.x, zh.y);
                }
            }
        }
#pragma unroll
        for (int i = 0; i < SN; ++i)
            if (t + THREADS * i < GT * STEP) ss[t + THREADS * i] = sv[i];
    };

    f32x16 acc[4];
    float a[4][8];

    // Products of one step; dY of step `next` is loaded as the registers become free. Per
    // scale group the lower parts' products come first and the upper parts' last, so only
    // four roundings of the step's sum are at its full size. Operands are made while the
    // matrix products before them run (one product, then a few vector instructions, in
    // turn: a wave that waits for the matrix unit issues nothing else).
    auto multiply = [&](int32_t next, auto load) {
        bf16x8 upper[2][4], lower[2][2], b[2][GB];
        auto operand = [&](int gi, int u, int x) {
            return __builtin_bit_cast(bf16x8, *reinterpret_cast<const u32x4*>(
                                                  bs + (wk * 128 + (gi * GB + x) * 32 + (ln & 31)) * PITCH + 16 * u + 8 * hl));
        };
        auto prepare = [&](auto ic) {  // the parts of stage i = 4 (scale group) + u, 16 n each
            constexpr int i = decltype(ic)::value, gi = i / 4, u = i % 4;
            const float* sc = ss + (wk * GW + gi) * STEP + 16 * u + 8 * hl;
            const f32x4 s0 = *reinterpret_cast<const f32x4*>(sc), s1 = *reinterpret_cast<const f32x4*>(sc + 4);
#pragma unroll
            for (int x = 0; x < GB; ++x) b[i & 1][x] = operand(gi, u, x);
            float v[8];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                v[e] = a[u][e] * s0[e];
                v[4 + e] = a[u][4 + e] * s1[e];
            }
            if constexpr (decltype(load)::value && gi == GW - 1) load_a(a[u], next, u);
            bf16x8 part[3];
            split3(v, part);
            upper[gi & 1][u] = part[0];
            lower[i & 1][0] = part[1];
            lower[i & 1][1] = part[2];
        };
        constexpr int SPLIT_VALU = 8 + 44;  // vector instructions of a stage's parts
        f32x16 sum[GB];
        prepare(std::integral_constant<int, 0>{});
        __builtin_amdgcn_sched_barrier(0);
        static_for<0, GW>([&](auto gc) {
            constexpr int gi = decltype(gc)::value;
#pragma unroll
            for (int x = 0; x < GB; ++x)
#pragma unroll
                for (int e = 0; e < 16; ++e) sum[x][e] = 0.0f;
            static_for<0, 4>([&](auto uc) {
                constexpr int u = decltype(uc)::value, i = 4 * gi + u;
#pragma unroll
                for (int h = 1; h >= 0; --h)
#pragma unroll
                    for (int x = 0; x < GB; ++x)
                        sum[x] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(lower[i & 1][h], b[i & 1][x], sum[x], 0, 0, 0);
                if constexpr (u < 3) {
                    prepare(std::integral_constant<int, i + 1>{});
                    __builtin_amdgcn_sched_group_barrier(0x100, 2 + GB, 0);  // the LDS reads
                    static_for<0, 2 * GB>([&](auto) {
                        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);  // one product
                        __builtin_amdgcn_sched_group_barrier(0x002, (SPLIT_VALU + 2 * GB - 1) / (2 * GB), 0);
                    });
                    __builtin_amdgcn_sched_barrier(0);
                }
            });
            // the upper parts (their weight operands read again)
            bf16x8 bu[4][GB];
#pragma unroll
            for (int u = 0; u < 4; ++u)
#pragma unroll
                for (int x = 0; x < GB; ++x) {
                    bu[u][x] = operand(gi, u, x);
                    sum[x] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(upper[gi & 1][u], bu[u][x], sum[x], 0, 0, 0);
                }
            if constexpr (gi + 1 < GW) {
                prepare(std::integral_constant<int, 4 * gi + 4>{});
                __builtin_amdgcn_sched_group_barrier(0x100, 2 + 2 * GB, 0);
                static_for<0, 6 * GB>([&](auto kc) {
                    __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                    if constexpr (decltype(kc)::value < 3 * GB) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
                    __builtin_amdgcn_sched_group_barrier(0x002, (SPLIT_VALU + 6 * GB - 1) / (6 * GB), 0);
                });
            }
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int x = 0; x < GB; ++x)
#pragma unroll
                for (int e = 0; e < 16; ++e) acc[gi * GB + x][e] += sum[x][e];
        });
    };

    // The slice in runs of at most p.run steps, each run's sums added to the output (the
    // slice's sums) on their own, so that no sum has more than p.run terms of a step.
    const int32_t all_whole = min(bpr / SB, BITS == 4 ? (N - bpr) / SB : p.steps);  // steps whose columns all exist
    float* out = p.out + static_cast<size_t>(p.splits > 1 ? sp : 0) * p.M * p.K;
    bool add = p.splits == 1 && p.accumulate;
    for (int32_t begin = sp * p.steps_per_split; begin < slice_end; begin += p.run, add = true) {
        const int32_t end = min(begin + p.run, slice_end), whole = min(end, all_whole);
#pragma unroll
        for (int b = 0; b < 4; ++b)
#pragma unroll
            for (int e = 0; e < 16; ++e) acc[b][e] = 0.0f;
        // whole steps, loads one step ahead; then the row's end
        if (begin < whole) {
            load_z(begin);
            load_w(begin);
#pragma unroll
            for (int u = 0; u < 4; ++u) load_a(a[u], begin, u);
            __syncthreads();  // the last run's zero points are read
            store_z(begin);
            load_z(begin + 1);
            for (int32_t x = begin; x < whole; ++x) {
                const int32_t next = min(x + 1, whole - 1);
                __syncthreads();  // the previous step's tile is read, this step's zero points are written
                convert(x);
                store_z(x + 1);
                __syncthreads();
                load_w(next);
                load_z(x + 2);
                multiply(next, std::true_type{});
            }
        }
        for (int32_t x = max(begin, whole); x < end; ++x) {
            const int32_t j0 = x * SB;
            load_z(x);
#pragma unroll
            for (int i = 0; i < ROWS; ++i)
#pragma unroll
                for (int v = 0; v < WV; ++v)
#pragma unroll
                    for (int d = 0; d < 4; ++d) w[i][v][d] = load_end(wbase + w_off[i], j0 + hf * (SB / 2) + 16 * v + 4 * d, bpr);
#pragma unroll
            for (int i = 0; i < SN; ++i) {
                const int32_t n = column(j0, sc_c);
                const float v = load_any<float>(sbase + (sc_row[i] + static_cast<uint32_t>(min(n, N - 1))) * 4u);
                sv[i] = valid(n, sc_c) ? v : 0.0f;
            }
#pragma unroll
            for (int u = 0; u < 4; ++u)
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    const int32_t c = 16 * u + 8 * hl + e, n = column(j0, c);
                    const float v = load_any<float>(abase + (a_off + static_cast<uint32_t>(min(n, N - 1)) * 4u));
                    a[u][e] = valid(n, c) ? v : 0.0f;
                }
            store_z(x);
            __syncthreads();  // the last tile is read, the zero points are written
            convert(x);
            __syncthreads();
            multiply(x, std::false_type{});
        }

        // Element e of block b: row 8 (e / 4) + 4 hl + e % 4, weight row 32 b + l % 32.
        int32_t el = ln;  // (opaque: its addresses are made here, not kept through the steps)
        asm volatile("" : "+v"(el));
        const int32_t m_e = m0 + 32 * wm + 4 * (el >> 5), k_e = k0 + wk * 128 + (el & 31);
        uint64_t nans = 0;
#pragma unroll
        for (int b = 0; b < 4; ++b) {
            const int32_t k = k_e + 32 * b;
            float* d = out + (static_cast<size_t>(m_e) * p.K + k);
            float old[16];  // all of a block's loads before its stores, from `out` itself where it has no element
#pragma unroll
            for (int e = 0; e < 16; ++e) old[e] = 0.0f;
            if (add) {
#pragma unroll
                for (int e = 0; e < 16; ++e) {
                    const int32_t m = m_e + 8 * (e >> 2) + (e & 3);
                    old[e] = *(m < p.M && k < p.K ? d + static_cast<size_t>(8 * (e >> 2) + (e & 3)) * p.K : out);
                }
            }
#pragma unroll
            for (int e = 0; e < 16; ++e) {
                const int32_t m = m_e + 8 * (e >> 2) + (e & 3);
                if (m < p.M && k < p.K) {
                    if (acc[b][e] != acc[b][e]) nans |= uint64_t{1} << (16 * b + e);
                    else d[static_cast<size_t>(8 * (e >> 2) + (e & 3)) * p.K] = old[e] + acc[b][e];
                }
            }
        }
        // A NaN may come from splitting an infinity: such an element is summed in fp32, term by
        // term, so that infinities and NaNs come out as the products give them; up to the first
        // NaN of 16 terms, and not at all where the row holds one (M = 512, 2048 <- 8192: with a NaN in
        // every row 0.17 ms, an infinity in one row 0.18, in every row 2.6; row by row 2.8 whatever dY).
        if (!__ballot(nans != 0)) continue;
        const int32_t j0 = begin * SB, j1 = min(end * SB, bpr);
        const uint32_t found = nan_rows(nans, p.a + static_cast<size_t>(row_a) * N, N, j0, j1, BITS == 4 ? bpr + j0 : 0, BITS == 4 ? min(bpr + j1, N) : 0);
        while (nans) {
            const int32_t i = __builtin_ctzll(nans), b = i >> 4, e = i & 15;
            nans &= nans - 1;
            const int32_t m = m_e + 8 * (e >> 2) + (e & 3), k = k_e + 32 * b;
            const float* dy = p.a + static_cast<size_t>(m) * N;
            const uint8_t* q = p.q + static_cast<size_t>(k) * bpr;
            const size_t row = static_cast<size_t>(k / p.g) * N;
            float sum = found >> (m - row_a) & 1 ? __builtin_nanf("") : 0.0f;
            int32_t j = j0;
            const int32_t wide = BITS == 8 ? j1 : min(j1, N - bpr);  // bytes with both columns
            for (; j + 16 <= wide && sum == sum; j += 16) {
                const u32x4 w = load_any<u32x4>(q + j);
                u32x4 zl, zh;
                if constexpr (BITS == 4) {
                    zl = load_any<u32x4>(p.z + row + j);
                    zh = load_any<u32x4>(p.z + row + bpr + j);
                }
#pragma unroll
                for (int c = 0; c < 16; ++c) {
                    auto byte = [&](const u32x4& v) { return static_cast<int32_t>(v[c / 4] << (24 - 8 * (c % 4))) >> 24; };
                    if constexpr (BITS == 8) {
                        sum = fmaf(dy[j + c], p.s[row + j + c] * static_cast<float>(byte(w)), sum);
                    } else {
                        sum = fmaf(dy[j + c], p.s[row + j + c] * static_cast<float>((byte(w) & 0xF) - byte(zl)), sum);
                        const int32_t n = bpr + j + c;
                        sum = fmaf(dy[n], p.s[row + n] * static_cast<float>((byte(w) >> 4 & 0xF) - byte(zh)), sum);
                    }
                }
            }
            for (; j < j1 && sum == sum; ++j) {
                if constexpr (BITS == 8) {
                    sum = fmaf(dy[j], p.s[row + j] * static_cast<float>(static_cast<int8_t>(q[j])), sum);
                } else {
                    sum = fmaf(dy[j], p.s[row + j] * static_cast<float>((q[j] & 0xF) - p.z[row + j]), sum);
                    const int32_t n = bpr + j;
                    if (n < N) sum = fmaf(dy[n], p.s[row + n] * static_cast<float>((q[j] >> 4) - p.z[row + n]), sum);
                }
            }
            float* d = out + static_cast<size_t>(m) * p.K + k;
            *d = add ? *d + sum : sum;
        }
    }
}

// ---- forward: c[M x N] = (accumulate ? c : 0) + alpha a[M x K] . deq(W) (+ bias) ------------
struct ForwardArgs {
    const float* a;
    const uint8_t* q;
    const float* s;
    const int8_t* z;
    float* c;         // or the slices' sums [splits][M][N]
    const float* bias;
    int32_t M, K, N, bpr, g, G, tiles_m, splits, steps, steps_per_split, accumulate;
    float alpha;
};

// Workgroup (tile of 32 WM rows of a and 128 WN columns, slice of k): each wave owns 32
// rows x 128 columns; for INT4 64 bytes of a weight row: 64 low-nibble columns and the 64
// high-nibble columns of the same bytes. A step is 64 k. The weights come to LDS transposed
// ([column][k], so that a lane's operand is 16 contiguous bytes): a thread takes 4 (INT4:
// 2) byte columns of 8 rows, and byte j of lane cq's columns goes to LDS row 32 j + cq, so
// that 32 lanes write 32 consecutive rows (no bank conflicts) and a lane ends with the sums
// of adjacent columns. The scale is constant along a group's k, so the group's sum is
// scaled, with one fp32 multiply-add: SC steps of 16 k share a scale (4 or 2).
// Bound by the steps' conversions and splits (vector ALU, 350 instructions a wave and step)
// beside 48 matrix products, at few rows by the conversions and the slices' sum:
// M = 512, 2048 -> 8191, INT4 g = 64 75 to 81 us, 220 TFLOP/s (generic_matmul 2784 us); M = 37,
// 1000 -> 2999 18 us with the call (163); M = 1, 14336 -> 20001 INT8 120 us, 2.4 TB/s (5104).
template <int BITS, bool ZP, int WM, int SC>
__global__ void __launch_bounds__(THREADS, 2) forward_split_kernel(ForwardArgs p) {
    constexpr int WN = 4 / WM, TN = 128 * WN;
    constexpr int TB = BITS == 4 ? 64 : 128;  // byte columns of a wave's tile
    constexpr int W = TB / 32;                // byte columns a thread converts
    __shared__ __attribute__((aligned(16))) uint16_t bs[TN * PITCH];
    const int32_t sp = blockIdx.x % p.splits, tile = blockIdx.x / p.splits;
    const int32_t m0 = (tile % p.tiles_m) * 32 * WM, j0 = (tile / p.tiles_m) * TB * WN;
    const int32_t t = threadIdx.x, ln = t & 63, hl = ln >> 5;
    const int32_t wave = __builtin_amdgcn_readfirstlane(t >> 6);
    const int32_t wm = wave % WM, wn = wave / WM;
    const int32_t begin = sp * p.steps_per_split, end = min(begin + p.steps_per_split, p.steps);
    const int32_t K = p.K, N = p.N, bpr = p.bpr;

    // This lane's row of a (a row past M repeats the last; its sums are dropped).
    const int32_t row_a = m0 + 32 * wm;
    const char* abase = reinterpret_cast<const char*>(p.a + static_cast<size_t>(min(row_a, p.M - 1)) * K);
    const uint32_t a_off = static_cast<uint32_t>(max(min(ln & 31, p.M - 1 - row_a), 0)) * K * 4u;
    // The bytes a thread converts: rows 8 rq .. + 7 of the step, W bytes from byte column
    // j0 + cq W of each tile (past the row's end the last W bytes, shifted into place).
    const int32_t cq = t & 31, rq = t >> 5;
    uint32_t w_at[WN], w_shift[WN];
#pragma unroll
    for (int i = 0; i < WN; ++i) {
        const int32_t j = j0 + TB * i + W * cq;
        w_at[i] = min(j, bpr - W);
        w_shift[i] = 8 * min(j - static_cast<int32_t>(w_at[i]), W - 1);
    }
    // Columns of this lane's sums: block b of the wave's tile.
    auto column = [&](int32_t lane, int b) {
        const int32_t j = j0 + TB * wn + W * (lane & 31) + b % W;
        return BITS == 4 && b >= 2 ? bpr + j : j;
    };
    auto exists = [&](int32_t n, int b) { return n < N && (BITS == 8 || b >= 2 || n < bpr); };

    uint32_t w[WN][8], zlo[WN], zhi[WN];
    float sc[4 / SC][4], sc_next[4 / SC][4];
    auto load_w = [&](int32_t x) {
        const int32_t k0 = x * STEP;
        const char* base = reinterpret_cast<const char*>(p.q) + static_cast<size_t>(k0) * bpr;
        const size_t zrow = static_cast<size_t>(min(k0 + 8 * rq, K - 1) / p.g) * N;
#pragma unroll
        for (int i = 0; i < WN; ++i) {
#pragma unroll
            for (int r = 0; r < 8; ++r) {
                const char* src = base + (static_cast<uint32_t>(min(8 * rq + r, K - 1 - k0)) * bpr + w_at[i]);
                if constexpr (BITS == 8) w[i][r] = load_any<uint32_t>(src) >> w_shift[i];
                else w[i][r] = static_cast<uint32_t>(load_any<uint16_t>(src)) >> w_shift[i];
            }
            if constexpr (ZP) {
                const int32_t j = j0 + TB * i + W * cq;
                const char* zr = reinterpret_cast<const char*>(p.z) + zrow;
                const int32_t lo = min(j, N - W), hi = min(bpr + j, N - W);
                if constexpr (BITS == 8) {
                    zlo[i] = load_any<uint32_t>(zr + lo) >> (8 * min(j - lo, W - 1));
                } else {
                    zlo[i] = static_cast<uint32_t>(load_any<uint16_t>(zr + lo)) >> (8 * min(j - lo, W - 1));
                    zhi[i] = static_cast<uint32_t>(load_any<uint16_t>(zr + hi)) >> (8 * min(bpr + j - hi, W - 1));
                }
            }
        }
    };
    auto load_scales = [&](int32_t x, float (&d)[4 / SC][4]) {
#pragma unroll
        for (int h = 0; h < 4 / SC; ++h)
#pragma unroll
            for (int b = 0; b < 4; ++b) {
                const int32_t gi = min(x * STEP + 16 * SC * h, K - 1) / p.g;
                d[h][b] = p.s[static_cast<size_t>(gi) * N + min(column(ln, b), N - 1)];
            }
    };
    auto convert = [&]() {
#pragma unroll
        for (int i = 0; i < WN; ++i)
            static_for<0, W>([&](auto jc) {
                constexpr int j = decltype(jc)::value;
                // byte j of the eight rows minus the zero point, both plus 128
                auto put = [&](int block, uint32_t zero, auto value) {
                    const float zf = ZP ? static_cast<float>(zero) : 128.0f;
                    u32x4 d;
#pragma unroll
                    for (int r = 0; r < 4; ++r) d[r] = upper_halves(value(w[i][2 * r]) - zf, value(w[i][2 * r + 1]) - zf);
                    *reinterpret_cast<u32x4*>(bs + (128 * i + 32 * block + cq) * PITCH + 8 * rq) = d;
                };
                if constexpr (BITS == 8) {
                    put(j, ((zlo[i] >> (8 * j)) & 0xFFu) ^ 0x80u, [](uint32_t v) { return ubyte<j>(v ^ 0x80808080u); });
                } else {
                    put(j, ((zlo[i] >> (8 * j)) & 0xFFu) ^ 0x80u, [](uint32_t v) { return ubyte<j>((v & 0x0F0Fu) | 0x8080u); });
                    put(2 + j, ((zhi[i] >> (8 * j)) & 0xFFu) ^ 0x80u, [](uint32_t v) { return ubyte<j>(((v >> 4) & 0x0F0Fu) | 0x8080u); });
                }
            });
    };
    float a[4][8];
    auto load_a = [&](int32_t x, int u) {  // a step inside K
        const char* src = abase + static_cast<int64_t>(x) * (4 * STEP) + (a_off + (64u * u + 32u * hl));
        const f32x4 v0 = load_any<f32x4>(src), v1 = load_any<f32x4>(src + 16);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            a[u][e] = v0[e];
            a[u][4 + e] = v1[e];
        }
    };

    f32x16 acc[4];
#pragma unroll
    for (int b = 0; b < 4; ++b)
#pragma unroll
        for (int e = 0; e < 16; ++e) acc[b][e] = 0.0f;

    // Products of one step: while the matrix products of 16 k run, the next 16 k of a are
    // split (and those of step `next` loaded in their place).
    auto multiply = [&](int32_t next, auto load) {
        bf16x8 part[2][3], b[2][4];
        auto prepare = [&](auto uc) {
            constexpr int u = decltype(uc)::value;
#pragma unroll
            for (int x = 0; x < 4; ++x)
                b[u & 1][x] = __builtin_bit_cast(bf16x8, *reinterpret_cast<const u32x4*>(
                                                             bs + (128 * wn + 32 * x + (ln & 31)) * PITCH + 16 * u + 8 * hl));
            split3(a[u], part[u & 1]);
            if constexpr (decltype(load)::value) load_a(next, u);
        };
        f32x16 sum[4];
        prepare(std::integral_constant<int, 0>{});
        __builtin_amdgcn_sched_barrier(0);
        static_for<0, 4>([&](auto uc) {
            constexpr int u = decltype(uc)::value;
            if constexpr (u % SC == 0) {
#pragma unroll
                for (int x = 0; x < 4; ++x)
#pragma unroll
                    for (int e = 0; e < 16; ++e) sum[x][e] = 0.0f;
            }
#pragma unroll
            for (int h = 2; h >= 0; --h)
#pragma unroll
                for (int x = 0; x < 4; ++x)
                    sum[x] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(part[u & 1][h], b[u & 1][x], sum[x], 0, 0, 0);
            if constexpr (u < 3) {
                prepare(std::integral_constant<int, u + 1>{});
                __builtin_amdgcn_sched_group_barrier(0x100, 4, 0);
                static_for<0, 12>([&](auto) {
                    __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                    __builtin_amdgcn_sched_group_barrier(0x002, 4, 0);
                });
            }
            __builtin_amdgcn_sched_barrier(0);
            if constexpr (u % SC == SC - 1) {
#pragma unroll
                for (int x = 0; x < 4; ++x)
#pragma unroll
                    for (int e = 0; e < 16; ++e) acc[x][e] = fmaf(sc[u / SC][x], sum[x][e], acc[x][e]);
            }
        });
    };

    const int32_t whole = min(end, K / STEP);
    if (begin < whole) {
        load_scales(begin, sc);
        load_w(begin);
#pragma unroll
        for (int u = 0; u < 4; ++u) load_a(begin, u);
        for (int32_t x = begin; x < whole; ++x) {
            const int32_t next = min(x + 1, whole - 1);
            __syncthreads();  // the previous step's tile is read
            convert();
            __syncthreads();
            load_w(next);
            load_scales(next, sc_next);
            multiply(next, std::true_type{});
#pragma unroll
            for (int h = 0; h < 4 / SC; ++h)
#pragma unroll
                for (int b = 0; b < 4; ++b) sc[h][b] = sc_next[h][b];
        }
    }
    if (whole < end) {  // K's end: a is zero past it
        const int32_t x = whole;
        load_scales(x, sc);
        load_w(x);
#pragma unroll
        for (int u = 0; u < 4; ++u)
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const int32_t k = x * STEP + 16 * u + 8 * hl + e;
                const float v = load_any<float>(abase + (a_off + static_cast<uint32_t>(min(k, K - 1)) * 4u));
                a[u][e] = k < K ? v : 0.0f;
            }
        __syncthreads();
        convert();
        __syncthreads();
        multiply(x, std::false_type{});
    }

    // Element e of block b: row 8 (e / 4) + 4 hl + e % 4, column column(l, b).
    const bool direct = p.splits == 1;
    float* out = p.c + static_cast<size_t>(direct ? 0 : sp) * p.M * N;
    auto finish = [&](float v, float old, int32_t n) {
        if (!direct) return v;
        const float o = fmaf(p.alpha, v, p.accumulate ? old : 0.0f);
        return p.bias ? o + p.bias[n] : o;
    };
    uint64_t nans = 0;
#pragma unroll
    for (int b = 0; b < 4; ++b) {
        const int32_t n = column(ln, b);
        if (!exists(n, b)) continue;
#pragma unroll
        for (int e = 0; e < 16; ++e) {
            const int32_t m = row_a + 8 * (e >> 2) + 4 * hl + (e & 3);
            if (m >= p.M) continue;
            float* d = out + static_cast<size_t>(m) * N + n;
            if (acc[b][e] != acc[b][e]) nans |= uint64_t{1} << (16 * b + e);
            else *d = finish(acc[b][e], direct && p.accumulate ? *d : 0.0f, n);
        }
    }
    // A NaN may come from splitting an infinity: such an element is summed as
    // generic_matmul does, term by term, up to the first group whose sum is a NaN, and not at
    // all where the row of a holds one (M = 512, 2048 -> 8191: with a NaN in every row 0.17 ms, an
    // infinity in one row 0.09, in every row 0.45; summed whole 13; generic_matmul 2.8).
    if (!__ballot(nans != 0)) return;
    const int32_t k_begin = begin * STEP, k_end = min(end * STEP, K);
    const uint32_t found = nan_rows(nans, p.a + static_cast<size_t>(row_a) * K, K, k_begin, k_end, 0, 0);
    while (nans) {
        const int32_t i = __builtin_ctzll(nans), b = i >> 4, e = i & 15;
        nans &= nans - 1;
        const int32_t m = row_a + 8 * (e >> 2) + 4 * hl + (e & 3), n = column(ln, b);
        const float* row = p.a + static_cast<size_t>(m) * K;
        const uint8_t* q = p.q + (BITS == 4 && b >= 2 ? n - bpr : n);
        float sum = found >> (m - row_a) & 1 ? __builtin_nanf("") : 0.0f;
        for (int32_t k1 = k_begin; k1 < k_end && sum == sum;) {
            const int32_t gi = k1 / p.g, k2 = min((gi + 1) * p.g, k_end);
            float part = 0.0f, rsum = 0.0f;
#pragma unroll 8
            for (; k1 < k2; ++k1) {
                const int32_t byte = q[static_cast<size_t>(k1) * bpr];
                const int32_t raw = BITS == 8 ? static_cast<int8_t>(byte) : b >= 2 ? byte >> 4 : byte & 0xF;
                part = fmaf(row[k1], static_cast<float>(raw), part);
                rsum += row[k1];
            }
            const size_t at = static_cast<size_t>(gi) * N + n;
            sum = fmaf(p.s[at], fmaf(ZP ? -static_cast<float>(p.z[at]) : -0.0f, rsum, part), sum);
        }
        float* d = out + static_cast<size_t>(m) * N + n;
        *d = finish(sum, direct && p.accumulate ? *d : 0.0f, n);
    }
}

// out = (accumulate ? out : 0) + alpha times the slices' sums, in a fixed order (+ bias of
// rows of N).
__global__ void __launch_bounds__(THREADS)
    slices_reduce_kernel(const float* __restrict__ part, int32_t splits, int64_t total, float* __restrict__ out,
                         int32_t accumulate, float alpha, const float* __restrict__ bias, int32_t N) {
    const int64_t i = static_cast<int64_t>(blockIdx.x) * THREADS + threadIdx.x;
    if (i >= total) return;
    float sum = 0.0f;
    for (int32_t s0 = 0; s0 < splits; s0 += 8) {  // eight at a time, added as a tree
        float v[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) v[u] = s0 + u < splits ? part[(s0 + u) * total + i] : 0.0f;
        sum += ((v[0] + v[1]) + (v[2] + v[3])) + ((v[4] + v[5]) + (v[6] + v[7]));
    }
    const float o = fmaf(alpha, sum, accumulate ? out[i] : 0.0f);
    out[i] = bias ? o + bias[i % N] : o;
}

int32_t launch_slices_reduce(const float* part, int32_t splits, int32_t m, int32_t n, float* out, int32_t accumulate,
                             float alpha, const float* bias, hipStream_t st) {
    const int64_t total = static_cast<int64_t>(m) * n, blocks = (total + THREADS - 1) / THREADS;
    if (blocks > INT32_MAX) return fail(KT_ERR_SHAPE, "grid of %lld blocks is out of range", static_cast<long long>(blocks));
    slices_reduce_kernel<<<static_cast<uint32_t>(blocks), THREADS, 0, st>>>(part, splits, total, out, accumulate, alpha,
                                                                          bias, n);
    KT_LAUNCHED("qmatmul: slices reduce");
    return KT_OK;
}

// Slices of `steps` for a grid of `tiles` workgroups, from the shape alone: two workgroups per
// CU, as far as the slices' sums (slice: bytes of one) fit SLICES_LIMIT.
void choose_slices(int64_t tiles, int32_t steps, size_t slice, int32_t* splits, int32_t* per_slice) {
    int64_t want = (2 * cu_count() + tiles - 1) / tiles;
    want = std::min<int64_t>(std::min<int64_t>(want, MAX_SPLITS), std::min<int64_t>(steps, SLICES_LIMIT / slice));
    *per_slice = ceil_div(steps, static_cast<int32_t>(std::max<int64_t>(want, 1)));
    *splits = ceil_div(steps, *per_slice);
}

template <int BITS, bool ZP, int WM>
void launch_forward_tiles(const ForwardArgs& p, uint32_t blocks, hipStream_t st) {
    if (p.g % 64 == 0) forward_split_kernel<BITS, ZP, WM, 4><<<blocks, THREADS, 0, st>>>(p);
    else forward_split_kernel<BITS, ZP, WM, 2><<<blocks, THREADS, 0, st>>>(p);
}
template <int BITS, bool ZP>
void launch_forward_rows(int32_t wm, const ForwardArgs& p, uint32_t blocks, hipStream_t st) {
    if (wm == 4) launch_forward_tiles<BITS, ZP, 4>(p, blocks, st);
    else if (wm == 2) launch_forward_tiles<BITS, ZP, 2>(p, blocks, st);
    else launch_forward_tiles<BITS, ZP, 1>(p, blocks, st);
}

template <int BITS, int WM>
void launch_transposed_tiles(const SplitArgs& p, uint32_t blocks, hipStream_t st) {
    if constexpr (WM == 4) {  // (the smaller row tiles would spill registers)
        if (p.g % 128 == 0) {
            transposed_split_kernel<BITS, WM, 4><<<blocks, THREADS, 0, st>>>(p);
            return;
        }
    }
    if (p.g % 64 == 0) transposed_split_kernel<BITS, WM, 2><<<blocks, THREADS, 0, st>>>(p);
    else transposed_split_kernel<BITS, WM, 1><<<blocks, THREADS, 0, st>>>(p);
}

}  // namespace

// The row-by-row kernel (kt_misc.hip) stays for small work, where it needs one launch and no
// slices: 2048 -> 2048 at M = 1 11.7 us against 14.1 here (both with the call), 896 -> 4864
// 13.8 against 18.8, M = 16 512 -> 512 9.9 against 12.1; 2048 -> 8192 at M = 1 28 against 23,
// M = 16 94 against 26, M = 37 1000 -> 2999 52 against 17, M = 200 640 -> 100 30 against 14.
bool transposed_split_preferred(int32_t m, const WeightView& w) {
    if (w.g % 32 != 0 || w.bpr < 4 || w.N > 1 << 22) return false;  // whole groups per block; 32-bit lane offsets
    const int64_t wgs = static_cast<int64_t>(ceil_div(m, 8)) * w.K;  // of the row-by-row kernel
    return wgs > 8192 || wgs * w.N > 6 << 20;
}

int32_t launch_transposed_split(const float* dy, int32_t m, const WeightView& w, float* dx, int32_t accumulate,
                                hipStream_t st) {
    SplitArgs p{dy, w.q, w.s, w.z, dx, m, w.K, w.N, w.bpr, w.g, w.G, 0, 1, 0, 0, 0, accumulate};
    const int32_t wm = m > 64 ? 4 : m > 32 ? 2 : 1;
    p.tiles_m = ceil_div(m, 32 * wm);
    const int64_t tiles = static_cast<int64_t>(p.tiles_m) * ceil_div(w.K, 128 * (4 / wm));
    p.steps = ceil_div(w.bpr, w.bits == 4 ? 32 : 64);
    const size_t slice = static_cast<size_t>(m) * w.K * sizeof(float);
    const int64_t max_blocks = tiles * MAX_SPLITS;
    if (max_blocks > INT32_MAX) return fail(KT_ERR_SHAPE, "grid of %lld blocks is out of range", static_cast<long long>(max_blocks));
    choose_slices(tiles, p.steps, slice, &p.splits, &p.steps_per_split);
    CallScratch area;
    if (p.splits > 1) {
        if (const int32_t status = area.take(CALL_SLICES, st, p.splits * slice)) return status;
        if (area.ptr) {
            p.out = static_cast<float*>(area.ptr);
        } else {
            // No scratch to have (CallScratch): one slice, or the row-by-row kernel where the few
            // workgroups of one slice would take longer. Row by row / one slice, 2048 -> 8192:
            // M = 1 28 / 460 us, 32 225 / 479, 48 334 / 362, 64 446 / 394, 512 2822 / 361; M = 200
            // 640 -> 100 30 / 19, M = 8 9000 -> 2000 60 / 129.
            if (int64_t{ceil_div(m, 8)} * w.K * w.N < int64_t{p.steps} * (7 << 17)) return launch_transposed_rows(dy, m, w, dx, accumulate, st);
            p.splits = 1;
            p.steps_per_split = p.steps;
        }
    }
    // Runs: no longer a sequence of sums than the row-by-row kernel's N / 256, or 16 steps
    // (28 steps in one run at N = 3584 had 1.19e-7 of the 2-norm against its 1.04e-7, two
    // runs of 14 have 1.01e-7; each run after a slice's first takes about 7 us).
    p.run = ceil_div(p.steps_per_split, ceil_div(p.steps_per_split, std::max(16, p.steps / 4)));
    const uint32_t blocks = static_cast<uint32_t>(tiles * p.splits);
    if (w.bits == 4)
        wm == 4   ? launch_transposed_tiles<4, 4>(p, blocks, st)
        : wm == 2 ? launch_transposed_tiles<4, 2>(p, blocks, st)
                  : launch_transposed_tiles<4, 1>(p, blocks, st);
    else
        wm == 4   ? launch_transposed_tiles<8, 4>(p, blocks, st)
        : wm == 2 ? launch_transposed_tiles<8, 2>(p, blocks, st)
                  : launch_transposed_tiles<8, 1>(p, blocks, st);
    const hipError_t err = hipGetLastError();
    int32_t status = err == hipSuccess ? KT_OK : hip_fail(err, "qmatmul_transposed: split kernel");
    if (area.ptr && status == KT_OK) status = launch_slices_reduce(p.out, p.splits, m, w.K, dx, accumulate, 1.0f, nullptr, st);
    return status;
}

// generic_matmul (kt_misc.hip: one thread per output, k in sequence: 0.13 to 0.16 us a k up to
// about 4000 waves, more with their number) stays for short sums, where this kernel's 12 to
// 17 us of a step or two are longer. Generic / here, with the call, INT4: 64 rows 32 -> 70
// 5.8 / 15.0 us, 64 -> 70 9.6 / 13.9, 80 -> 257 14.5 / 15.3, 88 -> 70 12.6 / 14.6, 96 -> 257
// 16.9 / 15.3; 1000 rows 64 -> 257 14.5 / 13.5, 64 -> 999 26 / 14; 4000 rows 48 -> 70 15.0 /
// 15.8, 64 -> 70 19 / 14; 16 rows 80 -> 257 14.3 / 14.5, 88 -> 257 15.6 / 14.5; one row
// 64 -> 70 9.1 / 12, 72 -> 257 12.2 / 12.4, 80 -> 257 13.4 / 12.5.
bool forward_split_preferred(int32_t m, const WeightView& w) {
    const int64_t waves = static_cast<int64_t>(m) * ceil_div(w.N, 64);  // of generic_matmul
    if (w.K <= (m > 16 ? 88 : m > 4 ? 80 : 72) && w.K * waves <= 410 << 10) return false;
    // 32 k share a scale, the clamped loads lie in a row; 32-bit lane offsets
    return w.g % 32 == 0 && w.N >= 8 && w.K <= 1 << 22 && w.bpr <= 1 << 24;
}

int32_t launch_forward_split(const float* a, int32_t m, const WeightView& w, float* c, int32_t accumulate, float alpha,
                             const float* bias, hipStream_t st) {
    ForwardArgs p{a, w.q, w.s, w.z, c, bias, m, w.K, w.N, w.bpr, w.g, w.G, 0, 1, 0, 0, accumulate, alpha};
    const int32_t wm = m > 64 ? 4 : m > 32 ? 2 : 1;
    p.tiles_m = ceil_div(m, 32 * wm);
    const int64_t tiles = static_cast<int64_t>(p.tiles_m) * ceil_div(w.bpr, (w.bits == 4 ? 64 : 128) * (4 / wm));
    p.steps = ceil_div(w.K, STEP);
    const size_t slice = static_cast<size_t>(m) * w.N * sizeof(float);
    const int64_t max_blocks = tiles * MAX_SPLITS;
    if (max_blocks > INT32_MAX) return fail(KT_ERR_SHAPE, "grid of %lld blocks is out of range", static_cast<long long>(max_blocks));
    choose_slices(tiles, p.steps, slice, &p.splits, &p.steps_per_split);
    CallScratch area;
    if (p.splits > 1) {
        if (const int32_t status = area.take(CALL_SLICES, st, p.splits * slice)) return status;
        if (area.ptr) {
            p.c = static_cast<float*>(area.ptr);
        } else {  // no scratch to have (CallScratch): one slice (3 us a step of 64 k; generic_matmul 9)
            p.splits = 1;
            p.steps_per_split = p.steps;
        }
    }
    const uint32_t blocks = static_cast<uint32_t>(tiles * p.splits);
    if (w.bits == 4) launch_forward_rows<4, true>(wm, p, blocks, st);
    else if (w.z) launch_forward_rows<8, true>(wm, p, blocks, st);
    else launch_forward_rows<8, false>(wm, p, blocks, st);
    const hipError_t err = hipGetLastError();
    int32_t status = err == hipSuccess ? KT_OK : hip_fail(err, "qmatmul: split kernel");
    if (area.ptr && status == KT_OK) status = launch_slices_reduce(p.c, p.splits, m, w.N, c, accumulate, alpha, bias, st);
    return status;
}

}  // namespace kt
