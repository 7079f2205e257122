// FLASH_ATTN_EXT for heads of 388 .. 512 dimensions (the VAE's middle block:
// one head of 512) over many positions, with the products in split FP16 on
// v_mfma_f32_32x32x16_f16 where attention.hip's wide forms take them on the
// single-precision MFMA, a sixteenth of its rate.
//
// Operands.  Each query, key and value x is scaled by an exact power of two
// and taken as h = fp16(x), l = fp16(x - h): 22 bits of x, and each product as
// h h' + h l' + l h' in one accumulator.  One accumulator is enough because
// every scale brings a group's greatest magnitude into [2^14, 2^15): an l is
// normal (11 bits of its own) for every x within 2^17 of the greatest of its
// group, and is 2^-40 of that greatest off at most below.  The groups: a
// query's or a key's own dimensions (the scales come back with the score, a
// factor of the query's and one of the key's); for the values, whose sum over
// the keys must share one scale, a tile of 32 keys, whose exponent the
// exponentials take on (2^(E_tile - E_run), E_run the greatest so far; where a
// tile raises it the outputs are rescaled, as they are where the running
// maximum moves).  The exponentials go in as 2^10 exp2(x - m), m moved only
// where a score passes it by 2^4 or more: below 2^14, their l normal down to
// 2^-13 of one where E_tile is E_run.  Their sum is of the unsplit numbers,
// eight at a time in single precision, then in double.
//
// What the 2^-40 is worth depends on the numbers beside an x and on its weight,
// so a workgroup first looks at the spans of its operands (split_holds) and
// takes a split of keys whose numbers lie too far apart, or are not finite, in
// single precision from the operands as they stand.  Error against 64 bits, of
// sum |p v|, 1024 positions: keys whose values lie 2^16, 2^20, 2^24 above the
// others and have no weight, all split 1.7e-6, 1.9e-5, 4.0e-4; dimensions
// 2^(+-16) apart 2.6e-3; queries' dimensions 2^(+-16) apart and the keys' the
// other way 8.7e-4; in single precision 1.1e-6 or less, all of them.
//
// Kernels.  attention512_tiles_kernel splits the keys and values once, into
// the order in which the products' waves load them (a wave's 1 KB of an MFMA
// operand in a row).  attention512_kernel: a workgroup of eight waves takes 64
// queries of a head and a split of the keys in steps of 64.  Scores: wave
// (key tile of 32, quarter of the dimensions) with its quarter of both query
// tiles held for the whole split, the high parts in registers and the low
// parts in LDS, the keys' operands straight from L2 into registers, each read
// by one wave only; the quarters meet in LDS.  Softmax: a wave eight keys, a lane a query.  Outputs: a wave
// 64 dimensions of all 64 queries (64 accumulators), the values' operands
// straight from L2, the exponentials from LDS.  attention512_combine_kernel
// merges the splits of the keys.
//
// What bounds it: a step of 64 keys is 6144 cycles of MFMA on each SIMD and
// 256 KB past the L1 (4096 cycles at 64 bytes), and takes about 12500: the
// products run at 62% of the MFMA's rate (timestamps of each phase), and
// between them the waves of a SIMD wait together for the softmax and its three
// barriers, about 2900.  Halving the loads changed 3%.  One head of 512 over
// 4096 positions: 702 -> 126 us a pass (traced one by one, on a slower card: the
// products 678 -> 123, the merge of half as many splits 46 -> 10, the tiles 12),
// error against 64 bits 9.0e-7 -> 4.4e-7; 1024 positions 165 -> 45 us, of which the spans are
// 2.  In single precision, where a value lies 2^20 above the others: 489 us
// (706 by attention_wide2_kernel) and 93 (166).  Slower: the next
// step's scores beside the softmax or after the outputs with no barrier between
// (132 and 149 us for the kernel, the registers spilled).

#include "attention.h"
#include "host.h"
#include "profile.h"

namespace sdhip {

namespace {

constexpr int kDims = 512;      // the dimensions of a head, zeros past its own
constexpr int kBlockQ = 64;     // a workgroup's queries
constexpr int kStepKeys = 64;   // the keys of a step
constexpr int kTileKeys = 32;   // the keys of a tile: an MFMA operand's rows
constexpr int kWaves = 8;
constexpr int kPart = 1024;     // bytes of one part of an MFMA operand of a wave
constexpr int kTileBytes = kTileKeys * kDims * 4;  // a tile of split keys or of split values
constexpr int kExpShift = 10;   // the exponentials' scale, 2^10

constexpr float kFinite = 3.402823466e38f;

// The exponent e that brings finite m >= 0 into [2^14, 2^15) as m 2^-e (0
// for m = 0 or infinity), held where 2^e, 2^-e and their product with such an m
// are normal.
__device__ __forceinline__ int scale_exponent(float m) {
    int k = 0;
    frexpf(m, &k);
    k -= 15;
    return m > 0.0f && m <= kFinite ? (k < -110 ? -110 : k) : 0;
}

// |x|, NaN as infinity: a maximum over these is infinite where one is not finite.
__device__ __forceinline__ float magnitude(float x) {
    const float a = fabsf(x);
    return a <= kFinite ? a : INFINITY;
}

__device__ __forceinline__ void split8(const float (&x)[8], float f, half8 &hi, half8 &lo) {
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        _Float16 h, l;
        split_scaled(x[i] * f, h, l);
        hi[i] = h;
        lo[i] = l;
    }
}

// ------------------------------------------------------------------ keys and values

// What the tiles' kernel writes: the queries' tiles [b h][tile][step of 16
// dimensions][part][lane][8], lane = query % 32 + 32 (dimension / 8 % 2); the
// keys' likewise; the values' [b hk][tile][step of 16 keys][32 dimensions][part][lane][8], lane =
// dimension % 32 + 32 (key / 8 % 2); each query's and key's factor 2^e; each
// tile of values' exponent; and each tile's span, from which the products'
// kernel sees whether the split holds its numbers: its greatest magnitude
// (infinite where a number is not finite) and, of values, the least of its keys'
// and dimensions' own greatest (split_values_span).
struct Span {
    float most, least;
};

struct Tiles {
    char *q, *k, *v;
    float *qf;    // [b h][query tile][32]
    float *kf;    // [b hk][tile][32]
    int32_t *ve;  // [b hk][tile]
    float *qm;    // [b h][query tile]
    float *km;    // [b hk][tile]
    Span *vs;     // [b hk][tile]
    int64_t tiles, qtiles;
};

__device__ __forceinline__ float max_over_block(float v, float *scratch) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v = fmaxf(v, __shfl_xor(v, off, 64));
    if ((threadIdx.x & 63) == 0) scratch[threadIdx.x >> 6] = v;
    __syncthreads();
    float m = scratch[0];
#pragma unroll
    for (int w = 1; w < 8; ++w) m = fmaxf(m, scratch[w]);
    return m;
}

// The least of a tile of values' rows and columns: of the greatest magnitude of
// each key and of each dimension, those of zeros alone left out.  x is a
// thread's dimension, m its greatest, `count` the tile's keys.  A dimension's
// greatest of fewer than eight numbers may well be small: 2^10 times it.
// `scratch` takes 8 x 32 floats and 8.
__device__ __forceinline__ float split_values_span(const float (&x)[4][8], float m, int64_t count, float *scratch) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    // The keys' greatest over the wave's 64 dimensions: halves of the keys go
    // to halves of the lanes, five times.
    float key[32];
#pragma unroll
    for (int i = 0; i < 32; ++i) key[i] = magnitude(x[i >> 3][i & 7]);
#pragma unroll
    for (int step = 0; step < 5; ++step) {
        const int n = 16 >> step;
        const bool upper = (lane & (2 * n)) != 0;
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            if (i >= n) continue;
            const float low = key[i], high = key[i + n];
            const float mine = upper ? high : low, other = upper ? low : high;
            key[i] = fmaxf(mine, __shfl_xor(other, 2 * n, 64));
        }
    }
    scratch[32 * wave + (lane >> 1)] = fmaxf(key[0], __shfl_xor(key[0], 1, 64));
    const auto positive = [](float v) { return v > 0.0f ? v : INFINITY; };
    float least = positive(count < 8 ? m * 1024.0f : m);
    __syncthreads();
    if (wave == 0) {
        float k = 0.0f;
#pragma unroll
        for (int w = 0; w < 8; ++w) k = fmaxf(k, scratch[32 * w + (lane & 31)]);
        least = fminf(least, positive(k));
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) least = fminf(least, __shfl_xor(least, off, 64));
    if (lane == 0) scratch[256 + wave] = least;
    __syncthreads();
#pragma unroll
    for (int w = 0; w < 8; ++w) least = fminf(least, scratch[256 + w]);
    return least;
}

// A tile of 32 queries or keys, rows of `row` floats from p on (`count` of
// them live): a thread row tid / 16, runs of 8 dimensions 8 (tid % 16) + 128 u.
__device__ __forceinline__ void split_rows(const float *p, int64_t row, int64_t count, int64_t d, char *out,
                                           float *factor, float *most, float *scratch) {
    const int tid = threadIdx.x;
    const int r = tid >> 4, run = tid & 15;
    const bool live = r < count;
    p += (live ? r : 0) * row;
    float x[4][8];
    float m = 0.0f;
#pragma unroll
    for (int u = 0; u < 4; ++u)
#pragma unroll
        for (int q = 0; q < 2; ++q) {
            const int at = 8 * run + 128 * u + 4 * q;
            float4v v = float4v{};
            if (live && at < d) v = *reinterpret_cast<const float4v *>(p + at);
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                x[u][4 * q + i] = v[i];
                m = fmaxf(m, magnitude(v[i]));
            }
        }
#pragma unroll
    for (int off = 8; off > 0; off >>= 1) m = fmaxf(m, __shfl_xor(m, off, 16));
    const int e = scale_exponent(m);
    const float f = ldexpf(1.0f, -e);
    if (run == 0) factor[r] = ldexpf(1.0f, e);
#pragma unroll
    for (int u = 0; u < 4; ++u) {
        const int at = run + 16 * u;  // the run of 8 dimensions
        half8 hi, lo;
        split8(x[u], f, hi, lo);
        char *to = out + (at >> 1) * (2 * kPart) + (r + 32 * (at & 1)) * 16;
        *reinterpret_cast<half8 *>(to) = hi;
        *reinterpret_cast<half8 *>(to + kPart) = lo;
    }
    m = max_over_block(m, scratch);
    if (tid == 0) *most = m;
}

// A block of 512 threads a tile of 32 keys (blockIdx.y 0), their values (1) or
// 32 queries (2), 32 numbers a thread held in registers between the maximum
// and the split.  Bound by HBM: at 4096 positions it moves 25 MB in and out.
__global__ __launch_bounds__(512) void attention512_tiles_kernel(AttentionArgs a, Tiles t) {
    __shared__ float scratch[8 * 32 + 16];
    const int tid = threadIdx.x;
    const int64_t block = blockIdx.x;
    if (blockIdx.y == 2) {
        if (block >= t.qtiles * a.h * a.b) return;
        const int64_t bh = block / t.qtiles, q0 = (block - bh * t.qtiles) * kTileKeys;
        const int64_t bi = bh / a.h, hi = bh - bi * a.h;
        split_rows(a.q + bi * a.qnb3 + hi * a.qnb2 + q0 * a.qnb1, a.qnb1, a.lq - q0, a.d, t.q + block * kTileBytes,
                   t.qf + block * kTileKeys, t.qm + block, scratch);
        return;
    }
    if (block >= t.tiles * a.hk * a.b) return;
    const int64_t bh = block / t.tiles, key0 = (block - bh * t.tiles) * kTileKeys;
    const int64_t bi = bh / a.hk, kh = bh - bi * a.hk;
    if (blockIdx.y == 0) {
        split_rows(static_cast<const float *>(a.k) + bi * a.knb3 + kh * a.knb2 + key0 * a.knb1, a.knb1, a.lk - key0,
                   a.d, t.k + block * kTileBytes, t.kf + block * kTileKeys, t.km + block, scratch);
        return;
    }
    float x[4][8];
    // Values: a thread dimension tid, the 32 keys in runs of 8.
    const bool dim = tid < a.dv;
    const float *p = static_cast<const float *>(a.v) + bi * a.vnb3 + kh * a.vnb2 + (dim ? tid : 0);
    float m = 0.0f;
#pragma unroll
    for (int r = 0; r < 4; ++r)
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const int64_t key = key0 + 8 * r + i;
            const float v = dim && key < a.lk ? p[key * a.vnb1] : 0.0f;
            x[r][i] = v;
            m = fmaxf(m, magnitude(v));
        }
    const float own = m;
    m = max_over_block(m, scratch + 8 * 32 + 8);
    const int e = scale_exponent(m);
    const float f = ldexpf(1.0f, -e);
    char *out = t.v + block * kTileBytes;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        half8 hi, lo;
        split8(x[r], f, hi, lo);
        char *to = out + ((r >> 1) * 16 + (tid >> 5)) * (2 * kPart) + ((tid & 31) + 32 * (r & 1)) * 16;
        *reinterpret_cast<half8 *>(to) = hi;
        *reinterpret_cast<half8 *>(to + kPart) = lo;
    }
    const float least = split_values_span(x, own, a.lk - key0, scratch);
    if (tid == 0) {
        t.ve[block] = e;
        t.vs[block] = Span{m, least};
    }
}

// ------------------------------------------------------------------ products

// A split's maximum (of the scores times log2 e), sum and output of each query.
struct Partial {
    double *l;  // [b h][split][lq]
    float *m;
    float *o;   // [b h][split][lq][dv]
};

constexpr int kScoreRow = 72;  // floats of a key's row of partial scores: rows 4 apart 32 banks apart

struct Shared {
    union {
        float scores[4][kStepKeys][kScoreRow];  // [quarter][key][query]
        double sums[kWaves][kBlockQ];
    };
    union {
        _Float16 p[kStepKeys / 16][2][2][64][8];  // [step][query tile][part][lane][8]
        float p32[kStepKeys][kBlockQ];            // the exponentials of the single-precision products
    };
    _Float16 ql[4][8][2][64][8];  // the queries' low parts: [quarter][step][query tile][lane][8]
    float most[kWaves][kBlockQ];
};
static_assert(sizeof(Shared) <= 160 * 1024, "LDS of a CU");

// Whether two FP16 parts hold the numbers of a workgroup's split: all finite, of
// magnitudes whose scales are exact, the queries' and keys' such that what l
// leaves off a score (2^-40 of their greatest product a dimension, 512 of them)
// stays under 2^-21, and the values' keys and dimensions all within 2^-8 of the
// greatest, since that is what an l of theirs and the exponentials' part for the
// tiles' scales leave off (2^-40 of it, and 2^-27 of a product).  Elsewhere -- a
// masked key's -infinity, a key or a dimension far above the others -- the
// products are of single precision.  N(0, 1) values stay within 2^-3.
//
// Its barrier is also that of the queries' low parts in LDS.
__device__ __forceinline__ bool split_holds(const AttentionArgs &a, const Tiles &t, Shared &sh, int64_t first,
                                            int64_t begin, int64_t end, float qm) {
    const int tid = threadIdx.x, wave = tid >> 6;
    float km = 0.0f, vm = 0.0f, least = INFINITY;
    for (int64_t i = begin + tid; i < end; i += 64 * kWaves) {
        const Span v = t.vs[first + i];
        km = fmaxf(km, t.km[first + i]);
        vm = fmaxf(vm, v.most);
        least = fminf(least, v.least);
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
        km = fmaxf(km, __shfl_xor(km, off, 64));
        vm = fmaxf(vm, __shfl_xor(vm, off, 64));
        least = fminf(least, __shfl_xor(least, off, 64));
    }
    if ((tid & 63) == 0) {
        sh.most[wave][0] = km;
        sh.most[wave][1] = vm;
        sh.most[wave][2] = least;
    }
    __syncthreads();
#pragma unroll
    for (int w = 0; w < kWaves; ++w) {
        km = fmaxf(km, sh.most[w][0]);
        vm = fmaxf(vm, sh.most[w][1]);
        least = fminf(least, sh.most[w][2]);
    }
    const auto exact = [](float m) { return m == 0.0f || (m >= 1e-28f && m <= 1e28f); };
    const bool holds = exact(qm) && exact(km) && exact(vm) && qm * km * fabsf(a.scale) <= 256.0f &&
                       least * 256.0f >= vm;
    return __builtin_amdgcn_readfirstlane(holds) != 0;
}

__global__ __launch_bounds__(512, 2) void attention512_kernel(AttentionArgs a, Tiles t, int64_t splits,
                                                              int64_t split_tiles, Partial part) {
    extern __shared__ __attribute__((aligned(16))) char lds[];
    Shared &sh = *reinterpret_cast<Shared *>(lds);
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int col = lane & 31, half = lane >> 5;
    const int ktile = wave & 1, quarter = wave >> 1;

    const uint32_t b = xcd_swizzle(blockIdx.x, gridDim.x);
    const uint32_t qb = b % static_cast<uint32_t>(a.qblocks);
    const uint32_t rest = b / static_cast<uint32_t>(a.qblocks);
    const int64_t sp = rest % splits;
    const int64_t bh = rest / splits;
    const int64_t hi = bh % a.h;
    const int64_t bi = bh / a.h;
    const int64_t kbh = bi * a.hk + hi / (a.h / a.hk);
    const int64_t q0 = static_cast<int64_t>(qb) * kBlockQ;
    const int64_t tile_begin = sp * split_tiles;
    const int64_t tile_end = tile_begin + split_tiles < t.tiles ? tile_begin + split_tiles : t.tiles;

    // The wave's quarter of both query tiles, the high parts into registers, the
    // low ones into LDS, and its first keys: on their way while the spans are
    // looked at.  A lane's query in the softmax is q0 + lane.
    const int64_t qtile = bh * t.qtiles + 2 * static_cast<int64_t>(qb);
    const bool two = 2 * static_cast<int64_t>(qb) + 1 < t.qtiles;  // the second query tile exists
    half8 qh[2][8];
#pragma unroll
    for (int qt = 0; qt < 2; ++qt) {
        const char *p = t.q + (qtile + (two ? qt : 0)) * kTileBytes + quarter * (8 * 2 * kPart) + lane * 16;
#pragma unroll
        for (int s = 0; s < 8; ++s) {
            qh[qt][s] = *reinterpret_cast<const half8 *>(p + s * (2 * kPart));
            if (ktile == 0) {
                *reinterpret_cast<half8 *>(&sh.ql[quarter][s][qt][lane][0]) =
                    *reinterpret_cast<const half8 *>(p + s * (2 * kPart) + kPart);
            }
        }
    }
    const char *kbase = t.k + kbh * t.tiles * kTileBytes + quarter * (8 * 2 * kPart) + lane * 16;
    const auto load_k = [&](int64_t tile, int s, half8 (&f)[2]) {
        const char *p = kbase + (tile + ktile < tile_end ? tile + ktile : tile) * kTileBytes + s * (2 * kPart);
        f[0] = *reinterpret_cast<const half8 *>(p);
        f[1] = *reinterpret_cast<const half8 *>(p + kPart);
    };
    half8 kf[4][2];
#pragma unroll
    for (int s = 0; s < 4; ++s) load_k(tile_begin, s, kf[s]);
    const bool split = split_holds(a, t, sh, kbh * t.tiles, tile_begin, tile_end,
                                   two ? fmaxf(t.qm[qtile], t.qm[qtile + 1]) : t.qm[qtile]);

    float16v o[2][2];  // [dimension tile][query tile]
#pragma unroll
    for (int dt = 0; dt < 2; ++dt)
#pragma unroll
        for (int qt = 0; qt < 2; ++qt) o[dt][qt] = float16v{};
    float m = -INFINITY;  // of query q0 + lane
    double l = 0.0;       // of query q0 + lane, the wave's keys
    int erun = -1000;     // the outputs' exponent (the block's)
    if (split) {
        const float qscale =
            a.scale * 1.44269504088896341f * t.qf[qtile * kTileKeys + (two || lane < kTileKeys ? lane : 0)];
        const char *vbase = t.v + kbh * t.tiles * kTileBytes + wave * (2 * 2 * kPart) + lane * 16;
        const float *kfbase = t.kf + kbh * t.tiles * kTileKeys;
        const int32_t *vebase = t.ve + kbh * t.tiles;
        // The values' operands of step s (16 keys): [dimension tile][part].
        const auto load_v = [&](int64_t tile, int s, half8 (&f)[2][2]) {
            const int64_t vt = tile + (s >> 1) < tile_end ? tile + (s >> 1) : tile;
            const char *p = vbase + vt * kTileBytes + (s & 1) * (16 * 2 * kPart);
#pragma unroll
            for (int dt = 0; dt < 2; ++dt)
#pragma unroll
                for (int u = 0; u < 2; ++u) f[dt][u] = *reinterpret_cast<const half8 *>(p + (2 * dt + u) * kPart);
        };

        for (int64_t tile = tile_begin; tile < tile_end; tile += 2) {
            // The scores of the wave's key tile over its quarter of the dimensions.
            float16v s2[2] = {float16v{}, float16v{}};
#pragma unroll
            for (int s = 0; s < 8; ++s) {
                const half8 h = kf[s & 3][0], lo = kf[s & 3][1];
                half8 ql[2];
#pragma unroll
                for (int qt = 0; qt < 2; ++qt) ql[qt] = *reinterpret_cast<const half8 *>(&sh.ql[quarter][s][qt][lane][0]);
#pragma unroll
                for (int qt = 0; qt < 2; ++qt)
                    s2[qt] = __builtin_amdgcn_mfma_f32_32x32x16_f16(h, qh[qt][s], s2[qt], 0, 0, 0);
#pragma unroll
                for (int qt = 0; qt < 2; ++qt)
                    s2[qt] = __builtin_amdgcn_mfma_f32_32x32x16_f16(lo, qh[qt][s], s2[qt], 0, 0, 0);
#pragma unroll
                for (int qt = 0; qt < 2; ++qt)
                    s2[qt] = __builtin_amdgcn_mfma_f32_32x32x16_f16(h, ql[qt], s2[qt], 0, 0, 0);
                __builtin_amdgcn_sched_barrier(0);
                if (s < 4) load_k(tile, s + 4, kf[s]);
                __builtin_amdgcn_sched_barrier(0);
            }
            // The keys' factors and the values' exponents of the wave's eight
            // keys, then the first half of the values' operands.
            const int64_t own = tile + (wave >> 2) < tile_end ? tile + (wave >> 2) : tile;
            const int64_t key0 = tile * kTileKeys + 8 * wave;
            const float4v f0 = *reinterpret_cast<const float4v *>(kfbase + own * kTileKeys + 8 * (wave & 3));
            const float4v f1 = *reinterpret_cast<const float4v *>(kfbase + own * kTileKeys + 8 * (wave & 3) + 4);
            const int e0 = vebase[tile], e1 = vebase[tile + 1 < tile_end ? tile + 1 : tile];
            half8 vf[2][2][2];
            load_v(tile, 0, vf[0]);
            load_v(tile, 1, vf[1]);
#pragma unroll
            for (int qt = 0; qt < 2; ++qt)
#pragma unroll
                for (int e = 0; e < 16; ++e)
                    sh.scores[quarter][32 * ktile + tile_row(e) + 4 * half][32 * qt + col] = s2[qt][e];
            lds_barrier();
            float x[8];
            float mx = -INFINITY;
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                const int key = 8 * wave + j;
                const float sum = (sh.scores[0][key][lane] + sh.scores[1][key][lane]) +
                                  (sh.scores[2][key][lane] + sh.scores[3][key][lane]);
                const float f = j < 4 ? f0[j & 3] : f1[j & 3];
                x[j] = key0 + j < a.lk ? (sum * f) * qscale : -INFINITY;
                mx = fmaxf(mx, x[j]);
            }
            sh.most[wave][lane] = mx;
            lds_barrier();
#pragma unroll
            for (int w = 0; w < kWaves; ++w) mx = fmaxf(mx, sh.most[w][lane]);
            const float mnew = mx > m + 4.0f ? mx : m;
            const int etile = e0 > e1 ? e0 : e1;
            const int enew = etile > erun ? etile : erun;
            // The rescaling, the same on every wave: exact in the values'
            // exponent, and zero while there is nothing to rescale.
            if (__any(mnew != m) || enew != erun) {
                const float fe = erun < -999 ? 0.0f : ldexpf(1.0f, erun - enew);
                const float fm = m == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(m - mnew);
                l *= static_cast<double>(fm);
                const float f = fm * fe;
#pragma unroll
                for (int qt = 0; qt < 2; ++qt) {
                    const float fq = __shfl(f, 32 * qt + col, 64);
#pragma unroll
                    for (int dt = 0; dt < 2; ++dt) o[dt][qt] *= fq;
                }
                m = mnew;
                erun = enew;
            }
            {
                const float fv = ldexpf(1.0f, (wave >> 2 ? e1 : e0) - erun + kExpShift);
                half8 ph, pl;
                float p[8];
                const float mref = m == -INFINITY ? 0.0f : m;  // scores of -inf so far: zeros
#pragma unroll
                for (int j = 0; j < 8; ++j) {
                    p[j] = __builtin_amdgcn_exp2f(x[j] - mref);
                    _Float16 h, lo;
                    split_scaled(p[j] * fv, h, lo);
                    ph[j] = h;
                    pl[j] = lo;
                }
                l += static_cast<double>(((p[0] + p[1]) + (p[2] + p[3])) + ((p[4] + p[5]) + (p[6] + p[7])));
                const int to = (lane & 31) + 32 * (wave & 1);
                *reinterpret_cast<half8 *>(&sh.p[wave >> 1][half][0][to][0]) = ph;
                *reinterpret_cast<half8 *>(&sh.p[wave >> 1][half][1][to][0]) = pl;
            }
            lds_barrier();
            // O^T += V^T P^T, 16 keys a step.
            const int64_t next = tile + 2 < tile_end ? tile + 2 : tile;
#pragma unroll
            for (int s = 0; s < 4; ++s) {
                half8 pq[2][2];  // [query tile][part]
#pragma unroll
                for (int qt = 0; qt < 2; ++qt)
#pragma unroll
                    for (int u = 0; u < 2; ++u) pq[qt][u] = *reinterpret_cast<const half8 *>(&sh.p[s][qt][u][lane][0]);
                half8 (&f)[2][2] = vf[s & 1];
#pragma unroll
                for (int u = 0; u < 3; ++u)
#pragma unroll
                    for (int dt = 0; dt < 2; ++dt)
#pragma unroll
                        for (int qt = 0; qt < 2; ++qt)
                            o[dt][qt] = __builtin_amdgcn_mfma_f32_32x32x16_f16(f[dt][u == 1], pq[qt][u == 2], o[dt][qt],
                                                                               0, 0, 0);
                __builtin_amdgcn_sched_barrier(0);
                if (s < 2) {
                    load_v(tile, s + 2, f);
                } else {
                    load_k(next, 2 * s - 4, kf[2 * s - 4]);
                    load_k(next, 2 * s - 3, kf[2 * s - 3]);
                }
                __builtin_amdgcn_sched_barrier(0);
            }
        }
    } else {
        // The same steps in single precision on v_mfma_f32_32x32x2_f32, from the
        // operands as they stand: a lane four dimensions of its rows at a time,
        // taken by four MFMAs (the two halves of the wave 4 apart), each into sums
        // of its own, of 32 products, a quarter of the others' rounding.
        const float qscale = a.scale * 1.44269504088896341f;
        const float *qp[2];
#pragma unroll
        for (int qt = 0; qt < 2; ++qt) {
            const int64_t i = q0 + 32 * qt + col < a.lq ? q0 + 32 * qt + col : a.lq - 1;
            qp[qt] = a.q + bi * a.qnb3 + hi * a.qnb2 + i * a.qnb1;
        }
        const int64_t kh = kbh - bi * a.hk;
        const float *kg = static_cast<const float *>(a.k) + bi * a.knb3 + kh * a.knb2;
        const float *vg = static_cast<const float *>(a.v) + bi * a.vnb3 + kh * a.vnb2;
        for (int64_t tile = tile_begin; tile < tile_end; tile += 2) {
            const int64_t first = tile * kTileKeys;
            // The split's keys of the step: a last tile alone is half of one.
            const int64_t end = tile_end * kTileKeys < a.lk ? tile_end * kTileKeys : a.lk;
            const int64_t key = first + kTileKeys * ktile + col;
            const float *kp = kg + (key < end ? key : end - 1) * a.knb1;
            float16v s2[4][2];
#pragma unroll
            for (int u = 0; u < 4; ++u)
#pragma unroll
                for (int qt = 0; qt < 2; ++qt) s2[u][qt] = float16v{};
#pragma unroll 1
            for (int s = 0; s < 16; ++s) {
                const int dim = 128 * quarter + 8 * s + 4 * half;
                float4v kx = float4v{}, qx[2] = {float4v{}, float4v{}};
                if (dim < a.d) {
                    kx = *reinterpret_cast<const float4v *>(kp + dim);
#pragma unroll
                    for (int qt = 0; qt < 2; ++qt) qx[qt] = *reinterpret_cast<const float4v *>(qp[qt] + dim);
                }
#pragma unroll
                for (int u = 0; u < 4; ++u)
#pragma unroll
                    for (int qt = 0; qt < 2; ++qt)
                        s2[u][qt] = __builtin_amdgcn_mfma_f32_32x32x2f32(kx[u], qx[qt][u], s2[u][qt], 0, 0, 0);
            }
#pragma unroll
            for (int qt = 0; qt < 2; ++qt)
#pragma unroll
                for (int e = 0; e < 16; ++e)
                    sh.scores[quarter][32 * ktile + tile_row(e) + 4 * half][32 * qt + col] =
                        (s2[0][qt][e] + s2[1][qt][e]) + (s2[2][qt][e] + s2[3][qt][e]);
            lds_barrier();
            float x[8];
            float mx = m;
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                const int at = 8 * wave + j;
                const float sum = (sh.scores[0][at][lane] + sh.scores[1][at][lane]) +
                                  (sh.scores[2][at][lane] + sh.scores[3][at][lane]);
                x[j] = first + at < end ? sum * qscale : -INFINITY;
                mx = fmaxf(mx, x[j]);
            }
            sh.most[wave][lane] = mx;
            lds_barrier();
#pragma unroll
            for (int w = 0; w < kWaves; ++w) mx = fmaxf(mx, sh.most[w][lane]);
            if (__any(mx != m)) {
                const float fm = m == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(m - mx);
                l *= static_cast<double>(fm);
#pragma unroll
                for (int qt = 0; qt < 2; ++qt) {
                    const float fq = __shfl(fm, 32 * qt + col, 64);
#pragma unroll
                    for (int dt = 0; dt < 2; ++dt) o[dt][qt] *= fq;
                }
                m = mx;
            }
            const float mref = m == -INFINITY ? 0.0f : m;
            float p[8];
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                p[j] = __builtin_amdgcn_exp2f(x[j] - mref);
                sh.p32[8 * wave + j][lane] = p[j];
            }
            l += static_cast<double>(((p[0] + p[1]) + (p[2] + p[3])) + ((p[4] + p[5]) + (p[6] + p[7])));
            lds_barrier();
#pragma unroll 4
            for (int s = 0; s < kStepKeys / 2; ++s) {
                const int at = 2 * s + half;
                float vx[2] = {0.0f, 0.0f};
#pragma unroll
                for (int dt = 0; dt < 2; ++dt) {
                    const int dim = 64 * wave + 32 * dt + col;
                    if (dim < a.dv && first + at < end) vx[dt] = vg[(first + at) * a.vnb1 + dim];
                }
#pragma unroll
                for (int qt = 0; qt < 2; ++qt) {
                    const float px = sh.p32[at][32 * qt + col];
#pragma unroll
                    for (int dt = 0; dt < 2; ++dt)
                        o[dt][qt] = __builtin_amdgcn_mfma_f32_32x32x2f32(vx[dt], px, o[dt][qt], 0, 0, 0);
                }
            }
        }
        erun = kExpShift;  // the outputs stand as they are
    }

    // The sum of each query over the waves' keys.
    __syncthreads();
    sh.sums[wave][lane] = l;
    __syncthreads();
    l = 0.0;
#pragma unroll
    for (int w = 0; w < kWaves; ++w) l += sh.sums[w][lane];
    const int64_t at0 = (bh * splits + sp) * a.lq + q0;
    if (part.o != nullptr && wave == 0 && q0 + lane < a.lq) {
        part.m[at0 + lane] = m;
        part.l[at0 + lane] = l;
    }
    const float unscale = ldexpf(1.0f, erun - kExpShift);
    const float factor = part.o != nullptr ? 1.0f : static_cast<float>(1.0 / l);
#pragma unroll
    for (int qt = 0; qt < 2; ++qt) {
        const float fq = __shfl(factor, 32 * qt + col, 64);
        const int64_t i = q0 + 32 * qt + col;
        if (i >= a.lq) continue;
        float *out = part.o != nullptr ? part.o + (at0 + 32 * qt + col) * a.dv
                                       : a.y + bi * a.ynb3 + i * a.ynb2 + hi * a.ynb1;
#pragma unroll
        for (int dt = 0; dt < 2; ++dt)
#pragma unroll
            for (int e4 = 0; e4 < 4; ++e4) {
                const int dim = 64 * wave + 32 * dt + 8 * e4 + 4 * half;
                if (dim < a.dv) {
                    float4v r;
#pragma unroll
                    for (int u = 0; u < 4; ++u) r[u] = (o[dt][qt][4 * e4 + u] * unscale) * fq;
                    *reinterpret_cast<float4v *>(out + dim) = r;
                }
            }
    }
}

// The splits merged: each split's sum and output times 2^(its maximum - the
// greatest), the sum in double, the output times the sum's reciprocal rounded
// to single precision.  A wave a query, float4 a lane.
__global__ __launch_bounds__(256) void attention512_combine_kernel(AttentionArgs a, int64_t splits, Partial part) {
    const int64_t item = static_cast<int64_t>(blockIdx.x) * 4 + (threadIdx.x >> 6);  // (b h) lq + i
    const int lane = threadIdx.x & 63;
    if (item >= a.b * a.h * a.lq) return;
    const int64_t bh = item / a.lq, i = item - bh * a.lq;
    const int64_t hi = bh % a.h, bi = bh / a.h;
    const int64_t first = bh * splits * a.lq + i;
    float mx = -INFINITY;
    for (int64_t sp = 0; sp < splits; ++sp) mx = fmaxf(mx, part.m[first + sp * a.lq]);
    double l = 0.0;
    float4v acc[2] = {float4v{}, float4v{}};
    for (int64_t sp = 0; sp < splits; ++sp) {
        const int64_t at = first + sp * a.lq;
        const float ms = part.m[at];
        const float w = ms == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(ms - mx);
        l += part.l[at] * static_cast<double>(w);
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            const int64_t e = 4 * lane + 256 * u;
            if (e < a.dv) acc[u] += *reinterpret_cast<const float4v *>(part.o + at * a.dv + e) * w;
        }
    }
    const float reciprocal = static_cast<float>(1.0 / l);
    float *out = a.y + bi * a.ynb3 + i * a.ynb2 + hi * a.ynb1;
#pragma unroll
    for (int u = 0; u < 2; ++u) {
        const int64_t e = 4 * lane + 256 * u;
        if (e < a.dv) *reinterpret_cast<float4v *>(out + e) = acc[u] * reciprocal;
    }
}

// ------------------------------------------------------------------ host

struct Layout {
    int64_t tiles, qtiles, splits, split_tiles;
    size_t q, k, v, qf, kf, ve, qm, km, vs, l, m, o, total;
};

Layout layout_of(const AttentionArgs &a) {
    Layout w{};
    w.tiles = ceil_div(a.lk, kTileKeys);
    w.qtiles = ceil_div(a.lq, kTileKeys);
    // One workgroup a CU: splits of the keys, an even number of tiles each,
    // until the workgroups fill the device once.
    const int64_t blocks = ceil_div(a.lq, kBlockQ) * a.h * a.b;
    int64_t sp = compute_units() / blocks;
    sp = sp < w.tiles / 4 ? sp : w.tiles / 4;
    sp = sp < 1 ? 1 : sp;
    w.split_tiles = round_up(ceil_div(w.tiles, sp), 2);
    w.splits = ceil_div(w.tiles, w.split_tiles);
    size_t at = 0;
    const auto take = [&](int64_t bytes) {
        const size_t here = at;
        at += static_cast<size_t>(round_up(bytes, 256));
        return here;
    };
    const int64_t heads = a.b * a.hk;
    w.q = take(a.b * a.h * w.qtiles * kTileBytes);
    w.qf = take(a.b * a.h * w.qtiles * kTileKeys * 4);
    w.k = take(heads * w.tiles * kTileBytes);
    w.v = take(heads * w.tiles * kTileBytes);
    w.kf = take(heads * w.tiles * kTileKeys * 4);
    w.ve = take(heads * w.tiles * 4);
    w.qm = take(a.b * a.h * w.qtiles * 4);
    w.km = take(heads * w.tiles * 4);
    w.vs = take(heads * w.tiles * static_cast<int64_t>(sizeof(Span)));
    if (w.splits > 1) {
        const int64_t n = a.b * a.h * w.splits * a.lq;
        w.l = take(n * 8);
        w.m = take(n * 4);
        w.o = take(n * a.dv * 4);
    }
    w.total = at;
    return w;
}

}  // namespace

// The shapes: heads of 388 .. 512 dimensions, a multiple of 4, single precision
// operands, and 256 pairs of 64 queries by 64 keys or more, one a CU.  Smaller
// calls keep the wide form on the single-precision MFMA, whose bits are those
// of attention_generic=1, although this form is faster there too (512 x 512
// positions: 36 us against 157).
bool attention512_shape(const AttentionArgs &a) {
    if (a.khalf || a.vhalf || a.bf16 || tuning().attention_generic != 0 || tuning().attention_fp32 != 0) return false;
    if (a.d <= 384 || a.d > kDims || a.dv <= 384 || a.dv > kDims || a.d % 4 != 0 || a.dv % 4 != 0) return false;
    const int64_t qblocks = ceil_div(a.lq, kBlockQ) * a.h * a.b;
    if (qblocks * ceil_div(a.lk, kStepKeys) < 256) return false;
    // The grids' first dimensions, in threads, stay below 2^32.
    return qblocks < (int64_t{1} << 20) && ceil_div(a.lk, kTileKeys) * a.b * a.hk < (int64_t{1} << 22) &&
           a.b * a.h * a.lq < (int64_t{1} << 25);
}

bool attention512_taken(const AttentionArgs &a) {
    const auto aligned = [](const void *p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; };
    return attention512_shape(a) && a.qnb1 % 4 == 0 && a.qnb2 % 4 == 0 && a.qnb3 % 4 == 0 && a.knb1 % 4 == 0 &&
           a.knb2 % 4 == 0 && a.knb3 % 4 == 0 && aligned(a.q) && aligned(a.k) && aligned(a.y);
}

size_t attention512_work_bytes(const AttentionArgs &a) { return layout_of(a).total; }

hipError_t launch_attention512(AttentionArgs a, void *work, hipStream_t stream) {
    const Layout w = layout_of(a);
    a.qblocks = ceil_div(a.lq, kBlockQ);
    char *base = static_cast<char *>(work);
    Tiles t{};
    t.q = base + w.q;
    t.qf = reinterpret_cast<float *>(base + w.qf);
    t.qtiles = w.qtiles;
    t.k = base + w.k;
    t.v = base + w.v;
    t.kf = reinterpret_cast<float *>(base + w.kf);
    t.ve = reinterpret_cast<int32_t *>(base + w.ve);
    t.qm = reinterpret_cast<float *>(base + w.qm);
    t.km = reinterpret_cast<float *>(base + w.km);
    t.vs = reinterpret_cast<Span *>(base + w.vs);
    t.tiles = w.tiles;
    Partial part{};
    if (w.splits > 1) {
        part.l = reinterpret_cast<double *>(base + w.l);
        part.m = reinterpret_cast<float *>(base + w.m);
        part.o = reinterpret_cast<float *>(base + w.o);
    }
    static const hipError_t attr = hipFuncSetAttribute(reinterpret_cast<const void *>(&attention512_kernel),
                                                       hipFuncAttributeMaxDynamicSharedMemorySize,
                                                       static_cast<int>(sizeof(Shared)));
    if (attr != hipSuccess) return attr;
    {
        KernelScope scope("attention.tiles", stream);
        const int64_t qt = w.qtiles * a.h, kt = w.tiles * a.hk;
        SDHIP_LAUNCH(attention512_tiles_kernel, dim3(static_cast<uint32_t>((qt > kt ? qt : kt) * a.b), 3), dim3(512),
                     0, stream, a, t);
        const hipError_t err = hipGetLastError();
        if (err != hipSuccess) return err;
    }
    KernelScope scope("attention", stream);
    SDHIP_LAUNCH(attention512_kernel, dim3(static_cast<uint32_t>(a.qblocks * a.h * a.b * w.splits)),
                 dim3(64 * kWaves), sizeof(Shared), stream, a, t, w.splits, w.split_tiles, part);
    if (w.splits > 1) {
        SDHIP_LAUNCH(attention512_combine_kernel, dim3(static_cast<uint32_t>(ceil_div(a.b * a.h * a.lq, 4))),
                     dim3(256), 0, stream, a, w.splits, part);
    }
    return hipGetLastError();
}

}  // namespace sdhip
