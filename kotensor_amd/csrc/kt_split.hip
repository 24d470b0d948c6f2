// kt_split.hip -- products with quantized weights in fp32 precision on the bf16 matrix units.
//
// An integer weight q - zero has at most 8 significant bits, so it is a bf16 number
// exactly; an fp32 number is the exact sum of three bf16 numbers (its 24 significant bits
// cut into 8 + 8 + 8, the lower parts exact while they stay above 2^-126). A product of
// fp32 data and integer weights is therefore three v_mfma_f32_32x32x16_bf16 whose products
// are exact and whose sums are fp32: the precision of an fp32 multiply-add chain at a
// third of the bf16 rate (about 5 times the fp32 matrix rate).
//
//   transposed: dX[M x K] = dY[M x N] . deq(W)^T (MatMul.multiplyByQuantizedTransposed,
//   Engine/kotensor/src/main/kotlin/MatMul.kt:954-981). The sum runs over n, along which
//   the scale changes, so a lane multiplies its dY values by the scales of the k-group
//   first (one fp32 rounding, in the place of the one of deq(W)) and splits the product.
#include <algorithm>

#include "kt_common.h"
#include "kt_packed.h"

namespace kt {
namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

constexpr int THREADS = 256;
constexpr int STEP = 64;          // elements of the summed dimension per step
constexpr int PITCH = STEP + 8;   // halfs per LDS row: 16-byte reads of 16 consecutive rows hit all banks once
constexpr int MAX_SPLITS = 32;

// 16 bytes at any alignment (dword accesses need none in global memory).
template <typename T>
__device__ __forceinline__ T load_any(const void* p) {
    T v;
    __builtin_memcpy(&v, p, sizeof(T));
    return v;
}

// The dword at byte i of a row of `bytes` >= 4 bytes; bytes past the row's end are any.
__device__ __forceinline__ uint32_t load_end(const void* row, int32_t i, int32_t bytes) {
    const int32_t at = min(i, bytes - 4);
    return load_any<uint32_t>(static_cast<const uint8_t*>(row) + at) >> (8 * min(i - at, 3));
}

// The upper halves of two floats in one dword: their bf16 truncations.
__device__ __forceinline__ uint32_t upper_halves(float lo, float hi) {
    return __builtin_amdgcn_perm(__builtin_bit_cast(uint32_t, hi), __builtin_bit_cast(uint32_t, lo), 0x07060302u);
}
// v minus its bf16 truncation, exact. (One v_dot2_f32_bf16 does the same, but runs on the
// matrix unit: four of them beside a 32x32x16 product took 63 cycles, four multiply-adds 38.)
__device__ __forceinline__ float below_upper(float v) {
    return v - __builtin_bit_cast(float, __builtin_bit_cast(uint32_t, v) & 0xFFFF0000u);
}

// Eight finite fp32 numbers as three bf16 operands, p = part[0] + part[1] + part[2]. An
// infinity makes a NaN of its lower parts; the callers look for NaN sums.
__device__ __forceinline__ void split3(const float (&p)[8], bf16x8 (&part)[3]) {
    u32x4 h, m, l;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const float a = p[2 * i], b = p[2 * i + 1];
        h[i] = upper_halves(a, b);
        const float ra = below_upper(a), rb = below_upper(b);
        m[i] = upper_halves(ra, rb);
        l[i] = upper_halves(below_upper(ra), below_upper(rb));
    }
    part[0] = __builtin_bit_cast(bf16x8, h);
    part[1] = __builtin_bit_cast(bf16x8, m);
    part[2] = __builtin_bit_cast(bf16x8, l);
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
// N = 8192, INT4 g = 64: 76 us, 220 TFLOP/s, plus 8 us for the slices' sum (row by row on
// the vector ALU: 2850 us); g = 128 63 us, g = 32 96 us.
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
        // term, so that infinities and NaNs come out as the products give them.
        while (nans) {
            const int32_t i = __builtin_ctzll(nans), b = i >> 4, e = i & 15;
            nans &= nans - 1;
            const int32_t m = m_e + 8 * (e >> 2) + (e & 3), k = k_e + 32 * b;
            const float* dy = p.a + static_cast<size_t>(m) * N;
            const uint8_t* q = p.q + static_cast<size_t>(k) * bpr;
            const size_t row = static_cast<size_t>(k / p.g) * N;
            float sum = 0.0f;
            for (int32_t j = begin * SB; j < min(end * SB, bpr) && sum == sum; ++j) {
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

// out = (accumulate ? out : 0) + the slices' sums, in a fixed order.
__global__ void __launch_bounds__(THREADS)
    slices_reduce_kernel(const float* __restrict__ part, int32_t splits, int64_t total, float* __restrict__ out,
                         int32_t accumulate) {
    const int64_t i = static_cast<int64_t>(blockIdx.x) * THREADS + threadIdx.x;
    if (i >= total) return;
    float sum = 0.0f;
    for (int32_t s0 = 0; s0 < splits; s0 += 8) {  // eight at a time, added as a tree
        float v[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) v[u] = s0 + u < splits ? part[(s0 + u) * total + i] : 0.0f;
        sum += ((v[0] + v[1]) + (v[2] + v[3])) + ((v[4] + v[5]) + (v[6] + v[7]));
    }
    out[i] = accumulate ? out[i] + sum : sum;
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
    // Slices of n: two workgroups per CU.
    int64_t splits = (2 * cu_count() + tiles - 1) / tiles;
    splits = std::min<int64_t>(std::min<int64_t>(splits, MAX_SPLITS), p.steps);
    const size_t slice = static_cast<size_t>(m) * w.K * sizeof(float);
    if (splits > 1 && !workspace_fits(st, splits * slice)) splits = 1;
    p.steps_per_split = ceil_div(p.steps, static_cast<int32_t>(splits));
    p.splits = ceil_div(p.steps, p.steps_per_split);
    // Runs: no longer a sequence of sums than the row-by-row kernel's N / 256, or 16 steps
    // (28 steps in one run at N = 3584 had 1.19e-7 of the 2-norm against its 1.04e-7, two
    // runs of 14 have 1.01e-7; each run after a slice's first takes about 7 us).
    p.run = ceil_div(p.steps_per_split, ceil_div(p.steps_per_split, std::max(16, p.steps / 4)));
    if (p.splits > 1) {
        void* ws = nullptr;
        const int32_t status = workspace(st, p.splits * slice, &ws);
        if (status) return status;
        p.out = static_cast<float*>(ws);
    }
    const int64_t blocks64 = tiles * p.splits;
    if (blocks64 > INT32_MAX) return fail(KT_ERR_SHAPE, "grid of %lld blocks is out of range", static_cast<long long>(blocks64));
    const uint32_t blocks = static_cast<uint32_t>(blocks64);
    if (w.bits == 4)
        wm == 4   ? launch_transposed_tiles<4, 4>(p, blocks, st)
        : wm == 2 ? launch_transposed_tiles<4, 2>(p, blocks, st)
                  : launch_transposed_tiles<4, 1>(p, blocks, st);
    else
        wm == 4   ? launch_transposed_tiles<8, 4>(p, blocks, st)
        : wm == 2 ? launch_transposed_tiles<8, 2>(p, blocks, st)
                  : launch_transposed_tiles<8, 1>(p, blocks, st);
    KT_LAUNCHED("qmatmul_transposed: split kernel");
    if (p.splits > 1) {
        const int64_t total = static_cast<int64_t>(m) * w.K;
        slices_reduce_kernel<<<static_cast<uint32_t>((total + THREADS - 1) / THREADS), THREADS, 0, st>>>(
            p.out, p.splits, total, dx, accumulate);
        KT_LAUNCHED("qmatmul_transposed: reduce");
    }
    return KT_OK;
}

}  // namespace kt
