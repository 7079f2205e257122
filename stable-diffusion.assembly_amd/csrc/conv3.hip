// 3x3 convolutions at stride 1 of FP16 kernels, directly: an implicit product
// of the nine taps on v_mfma_f32_16x16x32_f16, one pass over the image, for the
// sizes where F(4x4, 3x3) spends its time on the launches and the bytes between
// its transforms and products rather than on the products it saves.
//
// Precision.  The weights are exact FP16 operands.  Each input x is scaled by
// an exact power of two 2^-E and taken as h = fp16(x), l = fp16(x - h), two
// MFMAs a product: 22 bits of x.  E is the workgroup's own and follows its
// inputs as they come: it brings the greatest |x| so far into [2^13, 2^15), and
// where a later chunk of channels passes that, the sums are rescaled (exactly)
// and E raised.  So l is normal for every x within 2^15 of the greatest and
// 2^-40 of that greatest off at most below, and no pass over the image is needed
// before the products.  Against 64 bits this is nearer than F(4x4), whose
// transforms round and amplify.
//
// An output whose kernels are small on the greatest channels needs the others'
// own bits.  So the fetching waves also look for the least of a chunk's channels'
// greatest |x|, and where that is below 2^-2 take the chunk two or three times,
// 2^28 apart (store): 22 bits of each channel's greatest in the tile, the channels
// up to 2^72 apart.  Channels 2^24 and 2^40 apart and kernels of zero on the great
// ones, by one scale alone: 3.3e-5 and 0.45 of sum |x w| off; so, 5.1e-7.  That
// look, two numbers an operation and over the lanes without LDS, costs nothing in
// the forms of few tiles and 1 .. 2% of the 256 x 128 one, whose code it takes past
// the instruction cache (by shuffles 1 .. 3%; the second pass's code in a loop that
// is not unrolled 1% less there and twice the time below).  The second pass costs 16
// of 38 us at 320->320, 64x64, and 115 of 227 at 128->128, 520x768; a third 15 and
// 115.  Not held:
// a channel's rows further apart than its greatest's 2^-40, and kernels of FP16's
// last bits alone (all below 2^-22; 4.4e-6 of sum |x w|, where F(4x4) scales them
// first and has 1.8e-6).
//
// Shape.  A workgroup takes tiles of kRows x 16 outputs of an image by kOc
// output channels.  Its first waves compute, WP x WO x KS of them: WP groups of
// RW rows, WO groups of 16 NO channels, KS groups of input channels (each its
// own chunk of 32 at a time, their sums added through LDS at the end), so that
// small images fill the CUs with tiles whose waves still hold 64 or more
// accumulators.  Its last four waves fetch: a chunk's inputs, with their
// border, two chunks ahead into registers, their greatest magnitude found, and
// a chunk ahead split into LDS, [part][position][32 channels], two buffers, one
// barrier a chunk.  So a computing wave waits for no input: the memory counter
// is in order, and weights loaded behind inputs from HBM waited for those (kw0
// of the first version's chunks: 8600 cycles of the 3000 its MFMAs take).
// A fragment is 16 positions of a row by 32 channels; an input row's serves the
// three taps above each other of its column.  The weights, laid out as
// [chunk][tap][oc][32] by a first launch, go from L2 straight into registers, a
// column of taps ahead.
//
// What bounds it (timestamps of the waves, cycles).  A chunk of the 256 x 128
// form is 9216 cycles of MFMA on each SIMD and takes 11400, the MFMA's rate at
// 81%; a tile's end, 25000, is HBM's, every CU reading its residual and writing
// its outputs at once: 128->128 at 520x768 with a residual 595 -> 285 us (a call
// among others on new inputs each, the weights not kept, as all the times here),
// of which the bytes (614 MB, once each) are 119 at a copy's rate.  The 64 x 160
// form has one computing wave on a SIMD, 8300 cycles a pair of chunks of 5760 of
// MFMA, a start of 10000 and an end of 13500: 320->320 at 64x64, two images,
// 47.6 -> 35.4 us.  Not faster: two workgroups of 128 x 128 a CU (332 us at
// 520x768), the residual's lines read ahead by the fetching waves (298), stores
// past the caches (293), raised priority for either kind of wave.
// 16-byte piece p of a position's 64 bytes lies at p ^ (position / 4 % 4), so that
// the 16 consecutive positions of a fragment lie in 16 groups of banks for each
// piece; the counter still has 3.4 conflicts an LDS instruction in the 64 x 160
// form (reads, the fetching waves' writes and the exchange together).

#include <type_traits>

#include "conv3.h"
#include "host.h"
#include "kernels.h"
#include "profile.h"

namespace sdhip {

namespace {

constexpr int kCols = 16;          // outputs of a tile's row
constexpr int kPitch = kCols + 2;  // its inputs
constexpr int kChunk = 32;         // input channels of a chunk
constexpr int kFetchWaves = kChunk / 8;
constexpr int kLevelBits = 28;     // between the scales of a chunk's levels
constexpr int kMostLevels = 3;

template <int RW_, int NO_, int WP_, int WO_, int KS_, int FETCH>
struct Shape {
    static constexpr int RW = RW_, NO = NO_, WP = WP_, WO = WO_, KS = KS_;
    static constexpr int kFetch = FETCH;         // the waves that fetch inputs
    static constexpr int kWaves = WP * WO * KS;  // that compute
    static constexpr int kThreads = 64 * (kWaves + kFetch);
    static constexpr int kRows = RW * WP;
    static constexpr int kOc = 16 * NO * WO;
    static constexpr int kPos = (kRows + 2) * kPitch;
    static constexpr int kPosPer = (kPos + 63) / 64;  // a fetching lane's positions
    static constexpr int kPer = KS * kPosPer;         // and its items, 8 channels of a position
    static constexpr int kPlane = kPos * 2 * kChunk;  // bytes of one part of a chunk
    static constexpr int kBuffer = KS * 2 * kPlane;
    static constexpr int kExchange = KS > 1 ? kWaves * RW * NO * 1024 : 0;
    static constexpr int kLds = 2 * kBuffer > kExchange ? 2 * kBuffer : kExchange;
    static constexpr int kOwn = RW * NO / KS;  // the tiles of 16 x 16 a wave finishes
    static_assert(RW * NO % KS == 0, "whole tiles a group");
    static_assert(kFetch == kChunk / 8, "a fetching wave takes 8 channels of a chunk");
    static_assert(kLds + 256 <= 160 * 1024, "LDS of a CU");
};

// 256 outputs by 128 channels, eight computing waves: images of many tiles.
using Wide = Shape<8, 2, 2, 4, 1, kFetchWaves>;
// 64 outputs by 160 channels, four computing waves.
using Mid = Shape<4, 5, 1, 2, 2, kFetchWaves>;
// 64 outputs by 80 channels, four computing waves: few tiles.
using Narrow = Shape<4, 5, 1, 1, 4, kFetchWaves>;

struct Conv3Args {
    WinogradArgs a;
    const _Float16 *w;  // [chunk][3 kw + kh][oc][32]
    int32_t chunks, tiles_x, tiles_y;
    uint32_t tiles;    // of every image and block of output channels
    uint32_t xbytes;   // an image's, from its first element past its last
    uint32_t wbytes;
    int32_t vec_y;     // rows of whole aligned quads: float4 stores
    uint32_t vec_step;  // bit s: step s's operand in float4
};

__device__ __forceinline__ int scale_exponent(float m) {
    int k = 0;
    frexpf(m, &k);
    k -= 15;
    return m > 0.0f ? (k < -110 ? -110 : k) : -110;
}

// ------------------------------------------------------------------ weights

// [oc][ic][kh][kw] into [ic / 32][3 kw + kh][oc][ic % 32], a thread a kernel.  Bound
// by latency at 320 x 320 kernels (4.8 us; a thread eight kernels, 16-byte reads
// and writes: 5.1).
__global__ __launch_bounds__(256) void conv3_weights_kernel(const _Float16 *__restrict__ w, int64_t oc, int64_t ic,
                                                            _Float16 *__restrict__ out) {
    const int64_t c = static_cast<int64_t>(blockIdx.x) * kChunk + (threadIdx.x & 31);
    const int64_t o = static_cast<int64_t>(blockIdx.y) * 8 + (threadIdx.x >> 5);
    if (o >= oc) return;
    const _Float16 *k = w + (o * ic + c) * 9;
    _Float16 g[9];
#pragma unroll
    for (int i = 0; i < 9; ++i) g[i] = k[i];
#pragma unroll
    for (int t = 0; t < 9; ++t)
        out[((static_cast<int64_t>(blockIdx.x) * 9 + t) * oc + o) * kChunk + (threadIdx.x & 31)] = g[t % 3 * 3 + t / 3];
}

// ------------------------------------------------------------------ products

// A tile's place.  Consecutive tiles are neighbours of one block of output
// channels, whose weights and border rows an XCD's L2 then holds.
struct Place {
    int img, x0, y0, ob;
};

template <class S>
__device__ __forceinline__ Place place_of(const Conv3Args &p, uint32_t tile) {
    const uint32_t plane_tiles = static_cast<uint32_t>(p.tiles_x * p.tiles_y);
    const uint32_t spatial = plane_tiles * static_cast<uint32_t>(p.a.n);
    const uint32_t ob = tile / spatial;
    uint32_t rest = tile - ob * spatial;
    const uint32_t img = rest / plane_tiles;
    rest -= img * plane_tiles;
    const uint32_t ty = rest / static_cast<uint32_t>(p.tiles_x);
    return {static_cast<int>(img), static_cast<int>(rest - ty * p.tiles_x) * kCols, static_cast<int>(ty) * S::kRows,
            static_cast<int>(ob)};
}

// What the fetching waves hand over beside the buffers.
struct Handover {
    struct alignas(8) {
        float most;   // a chunk's greatest |x|, by wave,
        float least;  // and the least of its channels' greatest
    } range[2][kFetchWaves];
    struct alignas(8) {
        int e;      // a buffer's exponent,
        int again;  // and whether the next holds what it leaves of the same chunk
    } of[2];
};

// Magnitudes are compared as the bits of |x|, whose order is theirs (infinities
// and NaN above all others, from kInfinite on).
constexpr uint32_t kInfinite = 0x7f800000u;

__device__ __forceinline__ uint32_t greater(uint32_t a, uint32_t b) { return a > b ? a : b; }

// The lanes' values OFF (16, 32) apart: of `low`'s upper and `high`'s lower runs
// of OFF lanes swapped, the greater of both: `low`'s over each pair of lanes on
// the lower, `high`'s on the upper.
template <int OFF>
__device__ __forceinline__ uint32_t swapped_greater(uint32_t low, uint32_t high) {
    const auto r = OFF == 32 ? __builtin_amdgcn_permlane32_swap(low, high, false, false)
                             : __builtin_amdgcn_permlane16_swap(low, high, false, false);
    return greater(r[0], r[1]);
}

// The value of the lane's partner OFF (1, 2, 4, 8) apart (for 4 the eight lanes
// mirrored: a pair has different upper halves all the same).
template <int OFF>
__device__ __forceinline__ uint32_t partner(uint32_t v) {
    constexpr int kCtrl = OFF == 1 ? 0xB1 : OFF == 2 ? 0x4E : OFF == 4 ? 0x141 : 0x128;
    const int i = static_cast<int>(v);
    return static_cast<uint32_t>(__builtin_amdgcn_update_dpp(i, i, kCtrl, 0xF, 0xF, false));
}

// Of the N values v, the lanes' own and then the greatest over pairs of lanes
// OFF apart: halves of the values on halves of the lanes, down to one value, then
// that value over the lanes that hold it.
template <int OFF, int N>
__device__ __forceinline__ void meet_lanes(uint32_t *v, int lane) {
    constexpr int H = N > 1 ? N / 2 : 1;
#pragma unroll
    for (int i = 0; i < H; ++i) {
        const uint32_t low = v[i], high = N > 1 ? v[i + H] : v[i];
        if constexpr (OFF >= 16) {
            v[i] = swapped_greater<OFF>(low, high);
        } else {
            const bool upper = (lane & OFF) != 0;
            v[i] = greater(upper ? high : low, partner<OFF>(upper ? low : high));
        }
    }
    if constexpr (OFF > 1) meet_lanes<OFF / 2, H>(v, lane);
}

// The greatest over the lanes that hold different ones of N values.
template <int OFF, int N>
__device__ __forceinline__ uint32_t over_lanes(uint32_t v) {
    if constexpr (OFF >= 16) {
        v = swapped_greater<OFF>(v, v);
    } else {
        v = greater(v, partner<OFF>(v));
    }
    if constexpr (N > 2) v = over_lanes<OFF / 2, N / 2>(v);
    return v;
}

// Of N magnitudes a lane, the greatest over the wave's lanes of each: the most and
// the least positive of those (kInfinite if there is none).
template <int N>
__device__ __forceinline__ void wave_range(uint32_t (&v)[N], int lane, uint32_t &most, uint32_t &least) {
    meet_lanes<32, N>(v, lane);
    most = over_lanes<32, N>(v[0]);
    least = ~over_lanes<32, N>(~(v[0] != 0 ? v[0] : kInfinite));
}

// The fetching waves: `count` tiles from `tile` on, `stride` apart.
template <class S>
__device__ __forceinline__ void fetch_inputs(const Conv3Args &p, uint32_t tile, uint32_t stride, int count, int steps,
                                             char *lds, Handover &hand) {
    constexpr int KS = S::KS;
    constexpr uint32_t kPast = 0x80000000u;  // past any image (xbytes is below 2^31): reads zero
    const WinogradArgs &a = p.a;
    const int tid = static_cast<int>(threadIdx.x) - 64 * S::kWaves;
    const int lane = tid & 63, wave = tid >> 6;
    const uint32_t channel = static_cast<uint32_t>(a.xnb2) * 4;  // bytes of a channel's plane
    // A wave's items: channels 8 wave .. + 7 of each of the step's KS chunks at
    // every position of the tile's inputs, 64 positions at a time; the positions'
    // offsets in the image, past it where they lie outside.
    uint32_t from[S::kPosPer];
    __amdgpu_buffer_rsrc_t rsrc;
    const auto locate = [&](uint32_t t) {
        const Place at = place_of<S>(p, t);
        rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(a.x) + static_cast<int64_t>(at.img) * a.xnb3, 0,
                                                 static_cast<int>(p.xbytes), 0x00020000);
#pragma unroll
        for (int u = 0; u < S::kPosPer; ++u) {
            const int pos = lane + 64 * u;
            const int py = pos / kPitch, px = pos - py * kPitch;
            const int iy = at.y0 + py - a.p1, ix = at.x0 + px - a.p0;
            const bool in = pos < S::kPos && iy >= 0 && iy < a.ih && ix >= 0 && ix < a.iw;
            from[u] = in ? static_cast<uint32_t>(iy) * static_cast<uint32_t>(a.xnb1) * 4 + static_cast<uint32_t>(ix) * 4 +
                               8u * wave * channel
                         : kPast;
        }
    };
    float x[S::kPer][8];
    const auto load = [&](int sc) {
#pragma unroll
        for (int u = 0; u < S::kPer; ++u) {
            const int chunk = sc * KS + u / S::kPosPer;
            const uint32_t at = KS > 1 && chunk >= p.chunks ? kPast : from[u % S::kPosPer];
#pragma unroll
            for (int i = 0; i < 8; ++i)
                x[u][i] = __builtin_bit_cast(
                    float, __builtin_amdgcn_raw_buffer_load_b32(
                               rsrc, at, static_cast<uint32_t>(chunk * kChunk + i) * channel, 0));
        }
    };
    // Of the chunk in registers: the greatest |x|, and the least of its channels'
    // own greatest (those of zeros alone left out); of its finite numbers, where
    // some are not.
    const auto find_most = [&](int slot) {
        uint32_t c[8 * KS];
        uint32_t most, least;
#pragma unroll
        for (int k = 0; k < KS; ++k)
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                // One operation for two numbers: |.| is part of it, and a NaN
                // goes through.
                float m = fabsf(x[k * S::kPosPer][i]);
#pragma unroll
                for (int u = 1; u < S::kPosPer; ++u)
                    m = __builtin_elementwise_maximum(m, fabsf(x[k * S::kPosPer + u][i]));
                c[8 * k + i] = __builtin_bit_cast(uint32_t, m);
            }
        wave_range(c, lane, most, least);
        if (__builtin_expect(__builtin_amdgcn_readfirstlane(most) >= kInfinite, 0)) {
#pragma unroll
            for (int k = 0; k < KS; ++k)
#pragma unroll
                for (int i = 0; i < 8; ++i) {
                    c[8 * k + i] = 0;
#pragma unroll
                    for (int u = 0; u < S::kPosPer; ++u) {
                        const uint32_t m = __builtin_bit_cast(uint32_t, x[k * S::kPosPer + u][i]) & 0x7fffffffu;
                        c[8 * k + i] = greater(c[8 * k + i], m < kInfinite ? m : 0);
                    }
                }
            wave_range(c, lane, most, least);
        }
        if (lane == 0) {
            hand.range[slot][wave].most = __builtin_bit_cast(float, most);
            hand.range[slot][wave].least = __builtin_bit_cast(float, least);
        }
    };
    // The chunk's exponent: the tile's so far unless an input passes 2^15
    // times it, then one bit of room above the chunk's.  Where a channel's
    // greatest then lies below 2^-2, from where on l is below FP16's normal range,
    // the chunk goes into the buffers twice: what h leaves, where it is below 2^-14
    // and so no l of that range, follows 2^28 times as great, and once more where
    // that channel is still below.  (A subnormal l beside it would not do: the MFMA
    // aligns the product of a subnormal by the exponent of the least normal number,
    // 2^-14, and cuts the sums of small products off there.)  Returns whether the
    // chunk goes on.
    int erun = -1000;
    int level = 0;       // of the chunk in registers
    float reach = 0.0f;  // the least of the channels' greatest at its scale
    const auto store = [&](int buf, int slot, bool first) {
        float f = 1.0f;
        if (level == 0) {
            float m = hand.range[slot][0].most;
            reach = hand.range[slot][0].least;
#pragma unroll
            for (int w = 1; w < S::kFetch; ++w) {
                m = fmaxf(m, hand.range[slot][w].most);
                reach = fminf(reach, hand.range[slot][w].least);
            }
            const int e = scale_exponent(m);
            erun = first || e > erun ? e + 1 : erun;
            f = ldexpf(1.0f, -erun);
            reach = ldexpf(reach, -erun);
        }
        const bool again = __builtin_amdgcn_readfirstlane(level + 1 < kMostLevels && reach < 0.25f) != 0;
        if (tid == 0) {
            hand.of[buf].e = erun - kLevelBits * level;
            hand.of[buf].again = again;
        }
        const auto normal = [](float v) { return fabsf(v) >= 0x1p-14f ? v : 0.0f; };
        const auto put = [&](auto keep) {
#pragma unroll
            for (int u = 0; u < S::kPer; ++u) {
                const int pos = lane + 64 * (u % S::kPosPer);
                if (pos >= S::kPos) continue;
                half8 hi, lo;
#pragma unroll
                for (int i = 0; i < 8; ++i) {
                    _Float16 h, l;
                    const float s = x[u][i] * f;
                    split_scaled(s, h, l);
                    if constexpr (decltype(keep)::value) {
                        const float hf = normal(static_cast<float>(h)), lf = normal(s - hf);
                        const bool whole = fabsf(hf) >= 0x1p-14f && fabsf(lf) >= 0x1p-14f;
                        h = static_cast<_Float16>(hf);
                        l = static_cast<_Float16>(whole ? lf : 0.0f);
                        x[u][i] = whole ? 0.0f : (s - hf) * 0x1p28f;
                    }
                    hi[i] = h;
                    lo[i] = l;
                }
                char *d = lds + buf * S::kBuffer + u / S::kPosPer * 2 * S::kPlane + pos * 64 +
                          16 * (wave ^ ((pos >> 2) & 3));
                *reinterpret_cast<half8 *>(d) = hi;
                *reinterpret_cast<half8 *>(d + S::kPlane) = lo;
            }
        };
        if (__builtin_expect(again, 0)) {
            put(std::true_type{});
            reach *= 0x1p28f;
            ++level;
        } else {
            put(std::false_type{});
            level = 0;
        }
        return again;
    };
    static_assert(kLevelBits == 28, "what a level leaves, times 2^28");
    const int chunks = count * steps;  // of all the tiles
    int sc = 0;                        // of the chunk in registers, in its tile,
    int at = 0;                        // and of all
    // The next buffer, and the loads of the chunk after it.
    const auto next = [&](int buf) {
        if (store(buf, at & 1, sc == 0)) return;
        if (++at == chunks) return;
        if (++sc == steps) {
            sc = 0;
            tile += stride;
            locate(tile);
        }
        load(sc);
    };
    locate(tile);
    load(0);
    find_most(0);
    lds_barrier();
    next(0);
    lds_barrier();
    for (int g = 0;; ++g) {  // buffer g & 1 is the computing waves'
        const bool last = at == chunks;
        if (g == 0) {  // the second chunk's greatest, beside the first's products
            if (!last && level == 0) find_most(at & 1);
            lds_barrier();
        }
        if (!last) {
            next((g + 1) & 1);
            if (at < chunks && level == 0) find_most(at & 1);
        }
        if (KS > 1 && last) {  // the computing waves' exchange: a workgroup of several groups takes one tile
            lds_barrier();
            lds_barrier();
        }
        lds_barrier();
        if (last) break;
    }
}

// A tile's outputs: the groups' sums added, scaled back, the chain, stored.
template <class S>
__device__ __forceinline__ void finish(const Conv3Args &p, const Place &at, int oc0, int wp, int wo, int kg, int wave,
                                       int lane, int erun, float4v (&acc)[S::RW][S::NO], char *lds) {
    constexpr int RW = S::RW, NO = S::NO, KS = S::KS;
    const WinogradArgs &a = p.a;
    const int col = lane & 15, quad = lane >> 4;
    const int img = at.img, x0 = at.x0, y0 = at.y0;
    // The groups' sums: each wave writes the tiles it does not finish, and adds
    // the others' of those it does.
    float4v v[S::kOwn];
    if constexpr (KS > 1) {
        // Over the buffers: every wave's reads of them are done, and a
        // workgroup of several groups takes one tile.
        float4v *ex = reinterpret_cast<float4v *>(lds);
        lds_barrier();
#pragma unroll
        for (int j = 0; j < RW * NO; ++j)
            if (j % KS != kg) ex[(wave * RW * NO + j) * 64 + lane] = acc[j / NO][j % NO];
        lds_barrier();
#pragma unroll
        for (int q = 0; q < S::kOwn; ++q) {
#pragma unroll
            for (int g = 0; g < KS; ++g)
                if (g == kg) v[q] = acc[(KS * q + g) / NO][(KS * q + g) % NO];
#pragma unroll
            for (int g = 1; g < KS; ++g) {
                const int other = (kg + g) % KS * (S::WP * S::WO) + wo * S::WP + wp;
                v[q] += ex[(other * RW * NO + KS * q + kg) * 64 + lane];
            }
        }
    } else {
#pragma unroll
        for (int q = 0; q < S::kOwn; ++q) v[q] = acc[q / NO][q % NO];
    }

    // Four or fewer tiles at a time, every load of a step of the chain before any
    // of its values is used: tile q is outputs x .. x + 3 of a row and channel.
    constexpr int kGroup = S::kOwn % 4 == 0 ? 4 : 5;
    static_assert(S::kOwn % kGroup == 0, "whole groups");
    const int x = x0 + 4 * quad;
    const int xc = x + 3 < a.ow ? x : static_cast<int>(a.ow) - 4;  // of a quad, where the rows are whole quads
    const int64_t ynb[4] = {1, a.ynb1, a.ynb2, a.ynb3};
#pragma unroll
    for (int q0 = 0; q0 < S::kOwn; q0 += kGroup) {
        int row[kGroup], och[kGroup];
        float4v t[kGroup];
#pragma unroll
        for (int q = 0; q < kGroup; ++q) {
            const int j = KS * (q0 + q) + kg;
            const int yy = y0 + wp * RW + j / NO, oc = oc0 + 16 * (j % NO) + col;
            row[q] = yy < a.oh ? yy : static_cast<int>(a.oh) - 1;
            och[q] = oc < a.oc ? oc : static_cast<int>(a.oc) - 1;
#pragma unroll
            for (int e = 0; e < 4; ++e) t[q][e] = ldexpf(v[q0 + q][e], erun);
        }
        // The values of a tensor at the tiles' outputs: in one piece, or each on
        // its own.
        const auto read = [&](const float *from, const int64_t *nb, bool vec, float4v(&o)[kGroup]) {
            const float *base = from + img * nb[3];
            if (vec) {
#pragma unroll
                for (int q = 0; q < kGroup; ++q)
                    o[q] = *reinterpret_cast<const float4v *>(base + och[q] * nb[2] + row[q] * nb[1] + xc);
            } else {
#pragma unroll
                for (int q = 0; q < kGroup; ++q)
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        const int xe = x + e < a.ow ? x + e : static_cast<int>(a.ow) - 1;
                        o[q][e] = base[och[q] * nb[2] + row[q] * nb[1] + xe * nb[0]];
                    }
            }
        };
        if (a.from_redirect) {
            float4v o[kGroup];
            read(a.y, ynb, p.vec_y, o);
#pragma unroll
            for (int q = 0; q < kGroup; ++q)
#pragma unroll
                for (int e = 0; e < 4; ++e) t[q][e] = __fadd_rn(o[q][e], t[q][e]);
        }
#pragma unroll 1
        for (int s = 0; s < a.chain.count; ++s) {
            const DevStep &st = a.chain.steps[s];
            if (st.kind == kSilu) {
#pragma unroll
                for (int q = 0; q < kGroup; ++q)
#pragma unroll
                    for (int e = 0; e < 4; ++e) t[q][e] = silu(t[q][e]);
                continue;
            }
            float4v o[kGroup];
            if (st.nb[0] == 0) {
                const float *base = st.operand + img * st.nb[3];
#pragma unroll
                for (int q = 0; q < kGroup; ++q) {
                    const float f = base[och[q] * st.nb[2] + row[q] * st.nb[1]];
                    o[q] = float4v{f, f, f, f};
                }
            } else {
                read(st.operand, st.nb, (p.vec_step >> s) & 1, o);
            }
#pragma unroll
            for (int q = 0; q < kGroup; ++q)
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    t[q][e] = st.kind == kAdd ? __fadd_rn(t[q][e], o[q][e]) : __fmul_rn(t[q][e], o[q][e]);
        }
#pragma unroll
        for (int q = 0; q < kGroup; ++q) {
            const int j = KS * (q0 + q) + kg;
            if (y0 + wp * RW + j / NO >= a.oh || oc0 + 16 * (j % NO) + col >= a.oc || x >= a.ow) continue;
            float *out = a.y + img * a.ynb3 + och[q] * a.ynb2 + row[q] * a.ynb1 + x;
            if (p.vec_y) {
                *reinterpret_cast<float4v *>(out) = t[q];
            } else {
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    if (x + e < a.ow) out[e] = t[q][e];
            }
        }
        __builtin_amdgcn_sched_barrier(0);
    }
}

template <class S>
__global__ __launch_bounds__(S::kThreads, S::kThreads / 256) void conv3_kernel(Conv3Args p) {
    constexpr int RW = S::RW, NO = S::NO, KS = S::KS;
    extern __shared__ __attribute__((aligned(16))) char lds[];
    __shared__ Handover hand;
    const WinogradArgs &a = p.a;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int steps = (p.chunks + KS - 1) / KS;
    uint32_t tile = xcd_swizzle(blockIdx.x, gridDim.x);
    const int count = static_cast<int>((p.tiles - tile + gridDim.x - 1) / gridDim.x);
    if (wave >= S::kWaves) {
        fetch_inputs<S>(p, tile, gridDim.x, count, steps, lds, hand);
        return;
    }
    const int wp = wave % S::WP, wo = wave / S::WP % S::WO, kg = wave / (S::WP * S::WO);
    const int col = lane & 15, quad = lane >> 4;

    // The wave's weights of column kw of a chunk's taps: NO fragments of 16
    // output channels by the chunk's 32 input channels a tap (channels past the
    // last read it again).
    const __amdgpu_buffer_rsrc_t w_rsrc = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<_Float16 *>(p.w), 0, static_cast<int>(p.wbytes), 0x00020000);
    const uint32_t tap_bytes = static_cast<uint32_t>(a.oc) * 64u;
    half8 wf[2][3][NO];
    const auto load_w = [&](int set, int oc0, int sc, int kw) {
        int chunk = sc * KS + kg;
        chunk = chunk < p.chunks ? chunk : p.chunks - 1;
        const uint32_t at = static_cast<uint32_t>(chunk * 9 + 3 * kw) * tap_bytes;
#pragma unroll
        for (int o = 0; o < NO; ++o) {
            const int oc = oc0 + 16 * o + col;
            const uint32_t row = static_cast<uint32_t>(oc < a.oc ? oc : static_cast<int>(a.oc) - 1) * 64u + 16u * quad;
#pragma unroll
            for (int kh = 0; kh < 3; ++kh)
                wf[set][kh][o] = __builtin_bit_cast(
                    half8, __builtin_amdgcn_raw_buffer_load_b128(w_rsrc, row, at + kh * tap_bytes, 0));
        }
    };
    const auto oc_of = [&](int ob) { return ob * S::kOc + wo * 16 * NO; };

    float4v acc[RW][NO];
    // A chunk's products, its first column's weights in set 0; the next chunk's
    // are loaded beside its last column and moved there.
    const auto chunk = [&](const char *buf, bool first, int oc0, int sc, int oc_next, int sc_next) {
#pragma unroll
        for (int kw = 0; kw < 3; ++kw) {
            const int set = kw & 1;
            if (kw == 1 && first) lds_barrier();  // the fetching waves' (fetch_inputs)
            half8 x[2][2];
            const int pos0 = opaque(wp * RW * kPitch + kw + col);  // not thirty addresses held over the chunks
            const auto read = [&](int r) {
                const int pos = pos0 + r * kPitch;
                const char *f = buf + pos * 64 + 16 * (quad ^ ((pos >> 2) & 3));
                x[r & 1][0] = *reinterpret_cast<const half8 *>(f);
                x[r & 1][1] = *reinterpret_cast<const half8 *>(f + S::kPlane);
            };
            read(0);
            if (kw < 2) {
                load_w(set ^ 1, oc0, sc, kw + 1);
            } else {
                load_w(set ^ 1, oc_next, sc_next, 0);
            }
#pragma unroll
            for (int r = 0; r < RW + 2; ++r) {
                if (r + 1 < RW + 2) read(r + 1);
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int part = 0; part < 2; ++part)
#pragma unroll
                    for (int kh = 0; kh < 3; ++kh) {
                        if (r - kh < 0 || r - kh >= RW) continue;
#pragma unroll
                        for (int o = 0; o < NO; ++o)
                            acc[r - kh][o] = __builtin_amdgcn_mfma_f32_16x16x32_f16(x[r & 1][part], wf[set][kh][o],
                                                                                   acc[r - kh][o], 0, 0, 0);
                    }
                __builtin_amdgcn_sched_barrier(0);
            }
        }
#pragma unroll
        for (int kh = 0; kh < 3; ++kh)
#pragma unroll
            for (int o = 0; o < NO; ++o) wf[0][kh][o] = wf[1][kh][o];
    };

    Place at = place_of<S>(p, tile);
    int oc0 = oc_of(at.ob);
    load_w(0, oc0, 0, 0);
    lds_barrier();
    lds_barrier();
    int g = 0;
    for (int left = count; left > 0; --left) {
        int erun = 0;
        const Place next = place_of<S>(p, left > 1 ? tile + gridDim.x : tile);
        const int oc_next = oc_of(next.ob);
#pragma unroll
        for (int r = 0; r < RW; ++r)
#pragma unroll
            for (int o = 0; o < NO; ++o) acc[r][o] = float4v{};
        bool first = true;
        for (int sc = 0; sc < steps; ++g) {
            if (!first) lds_barrier();
            const int e = __builtin_amdgcn_readfirstlane(hand.of[g & 1].e);
            const int after = __builtin_amdgcn_readfirstlane(hand.of[g & 1].again) ? sc : sc + 1;
            if (!first && e != erun) {
                const float f = ldexpf(1.0f, erun - e);
#pragma unroll
                for (int r = 0; r < RW; ++r)
#pragma unroll
                    for (int o = 0; o < NO; ++o) acc[r][o] *= f;
            }
            erun = e;
            const char *buf = lds + (g & 1) * S::kBuffer + kg * 2 * S::kPlane;
            const bool last = after == steps;
            chunk(buf, g == 0, oc0, sc, last ? oc_next : oc0, last ? 0 : after);
            sc = after;
            first = false;
        }
        finish<S>(p, at, oc0, wp, wo, kg, wave, lane, erun, acc, lds);
        lds_barrier();
        tile += gridDim.x;
        at = next;
        oc0 = oc_next;
    }
}

// ------------------------------------------------------------------ host

template <class S>
int64_t blocks_of(const WinogradArgs &a) {
    return ceil_div(a.ow, kCols) * ceil_div(a.oh, S::kRows) * a.n * ceil_div(a.oc, S::kOc);
}

// What a form takes on one CU, in thousands of cycles (timestamps of the three
// kernels): a step of the input channels, and a tile's beginning and end; and in
// microseconds of the whole launch, fitted as direct_faster's comment says: of
// each round of workgroups, and of its tiles as they fill the device.
struct Cost {
    double step, tile;
    double us_step, us_tile, us_full_step, us_full_tile;
};

constexpr Cost kCosts[3] = {
    {11.4, 26.0, 3.2, 12.0, 2.9, 0.0},  // Wide
    {8.5, 14.0, 3.3, 7.8, 0.9, 0.0},    // Mid
    {9.7, 14.0, 4.4, 7.1, 0.4, 0.8},    // Narrow
};

struct Work {
    double cycles, us;  // of the products' launch
};

template <class S>
Work work_of(const WinogradArgs &a, const Cost &c) {
    const double filled = static_cast<double>(blocks_of<S>(a)) / compute_units();
    const double rounds = static_cast<double>(ceil_div(blocks_of<S>(a), compute_units()));
    const double steps = static_cast<double>(ceil_div(a.ic, kChunk * S::KS));
    return {rounds * (steps * c.step + c.tile) + 12.0,
            1.3 + rounds * (steps * c.us_step + c.us_tile) + filled * (steps * c.us_full_step + c.us_full_tile)};
}

// The form of the least cycles: 1 Wide, 2 Mid, 3 Narrow.
int shape_of(const WinogradArgs &a, Work &work) {
    const Work w[3] = {work_of<Wide>(a, kCosts[0]), work_of<Mid>(a, kCosts[1]), work_of<Narrow>(a, kCosts[2])};
    int best = 0;
    for (int i = 1; i < 3; ++i)
        if (w[i].cycles < w[best].cycles) best = i;
    work = w[best];
    return best + 1;
}

// F(4x4)'s microseconds, its weights kept in the store or not: on few tiles the
// small images' kernels, bound by the weights; else the launches; the inputs
// and outputs (in millions), more where rows are not whole quads; the scales'
// pass, a workgroup a channel, by single numbers where planes are not whole quads;
// the weights' transform; the products by their rounds of workgroups and their
// work; and what the passes between them hold past the last-level cache.
double winograd4_us(const WinogradArgs &a, bool kept) {
    const double kernels = static_cast<double>(a.ic * a.oc) / 1e6;
    if (a.tiles <= 16) return kept ? 30.0 + 17.5 * kernels : 29.0 + 19.4 * kernels;
    if (a.tiles <= 32) return kept ? 33.0 + 22.3 * kernels : 31.0 + 24.4 * kernels;
    const double in = static_cast<double>(a.n * a.ic * a.ih * a.iw) / 1e6;
    const double out = static_cast<double>(a.n * a.oc * a.oh * a.ow) / 1e6;
    const double ragged = a.ow % 4 != 0 ? 1.0 : 0.0;
    const double scales =
        a.ih * a.iw % 4 != 0 || a.xnb1 != a.iw ? static_cast<double>(a.n * a.ih * a.iw) / 1e3 : 0.0;
    const int64_t blocks = 36 * ceil_div(a.oc, 64) * ceil_div(a.tiles, 128);
    const double rounds = static_cast<double>(ceil_div(blocks, 2 * compute_units()) * a.ic) / 1e3;
    const double products = static_cast<double>(blocks * a.ic) / 1e6;
    const double held = 144.0 * kernels + 144.0 * static_cast<double>((a.ic + a.oc) * a.tiles) / 1e6 + 4.0 * (in + out);
    const double past = held > 200.0 ? (held - 200.0) / 100.0 : 0.0;
    if (kept) {
        return 20.2 + (3.3 + 0.6 * ragged) * in + (3.0 + 1.6 * ragged) * out + 1.3 * scales + 5.5 * kernels +
               10.5 * rounds + 19.7 * products + 8.8 * past;
    }
    return 21.0 + (2.7 + 1.4 * ragged) * in + (2.2 + 1.5 * ragged) * out + 1.2 * scales + 34.6 * kernels +
           3.1 * rounds + 32.0 * products + 25.0 * past;
}

// Whether the products here take less than F(4x4), by the sum of both cases, the
// weights kept in the store and not, and by each (kept, within 2%): whichever of
// them a call finds it takes the same path, so that its outputs do not depend on
// the store or on a capture.  The times above were fitted to 297 shapes of the
// UNet's and the VAE's levels, whole and ragged, with a spread of 3% for this
// form and 4% for F(4x4).  Of those taken here none is slower by more than 2.4%
// without the store; kept, one by 7% (12% faster without), the rest by 3.6% at
// most (the look at the channels, later, adds 0 .. 2% to this form).  Measured, F(4x4) and here, us, without the store and kept (images first):
//   2 320->320 64x64   45.2 34.9   45.7 31.2   1 128->128 520x768   551  231    545  234
//   1 640->1280 16x16  45.2 42.2   45.9 31.7   1 256->256 115x91   66.4 55.8   65.3 52.1
//   1 1280->1280 16x16 61.2 67.7   58.9 55.7   1 256->256 196x151  99.0  112    104  108
//   2 640->320 72x80   88.0  105   90.7 99.7   1 512->256 128x128  82.2 89.9   85.0 86.7
//   2 1920->640 32x32   106 94.7   80.7 86.3   1 512->512 114x85    107  103    105 99.4
//   2 2560->1280 32x32  322  210    184  191   1 128->256 104x102  40.6 41.6   42.7 38.8
bool direct_faster(const WinogradArgs &a) {
    Work work;
    shape_of(a, work);
    const double here = work.us + (a.ow % 4 != 0 ? 1.3 * static_cast<double>(a.n * a.oc * a.oh * a.ow) / 1e6 : 0.0);
    const double weights = 3.4 + 4.9 * static_cast<double>(a.ic * a.oc) / 1e6;  // the pass over them
    const double kept = winograd4_us(a, true), made = winograd4_us(a, false);
    return here + weights <= made && here <= 1.02 * kept && 2.0 * here + weights <= kept + made;
}

int64_t weight_bytes(const WinogradArgs &a) { return a.ic * a.oc * 18; }

// An image's floats from its first past its last.
int64_t image_floats(const WinogradArgs &a) { return (a.ic - 1) * a.xnb2 + (a.ih - 1) * a.xnb1 + a.iw; }

template <class S>
hipError_t launch(Conv3Args &p, hipStream_t stream) {
    static const hipError_t attr = hipFuncSetAttribute(reinterpret_cast<const void *>(&conv3_kernel<S>),
                                                       hipFuncAttributeMaxDynamicSharedMemorySize, S::kLds);
    if (attr != hipSuccess) return attr;
    p.tiles_x = static_cast<int32_t>(ceil_div(p.a.ow, kCols));
    p.tiles_y = static_cast<int32_t>(ceil_div(p.a.oh, S::kRows));
    p.tiles = static_cast<uint32_t>(blocks_of<S>(p.a));
    // A workgroup a CU, tile after tile, where one holds all the input
    // channels' groups; else one a tile.
    const uint32_t cus = static_cast<uint32_t>(compute_units());
    const uint32_t blocks = S::KS == 1 && p.tiles > cus ? cus : p.tiles;
    SDHIP_LAUNCH(conv3_kernel<S>, dim3(blocks), dim3(S::kThreads), S::kLds, stream, p);
    return hipGetLastError();
}

}  // namespace

bool conv3_shape(const WinogradArgs &a) {
    const Tuning &t = tuning();
    if (a.m != 4 || a.w32 != nullptr || t.winograd_fp32 || t.conv3x3_direct == 0) return false;
    if (a.ic % kChunk != 0 || a.ic < 128 || a.oc < 128) return false;
    if (a.xnb1 < a.iw || a.xnb2 < 1 || a.xnb3 < 0 || a.n < 1) return false;
    // Offsets in an image, in the weights and of blocks in 31 bits.
    if (image_floats(a) * 4 >= (int64_t{1} << 31) - 64 || weight_bytes(a) >= (int64_t{1} << 31) - 64) return false;
    return blocks_of<Narrow>(a) < (int64_t{1} << 22) && direct_faster(a);
}

// One pass reads the inputs while it writes the outputs: not in place.
bool conv3_taken(const WinogradArgs &a) {
    if (!conv3_shape(a)) return false;
    const int64_t x_floats = (a.n - 1) * a.xnb3 + image_floats(a);
    const int64_t y_floats = (a.n - 1) * a.ynb3 + (a.oc - 1) * a.ynb2 + (a.oh - 1) * a.ynb1 + a.ow;
    return !spans_overlap(a.x, static_cast<size_t>(x_floats) * 4, a.y, static_cast<size_t>(y_floats) * 4);
}

size_t conv3_work_size(const WinogradArgs &a) { return static_cast<size_t>(round_up(weight_bytes(a), 256)); }

sdhip_status conv3(const WinogradArgs &a, void *work, hipStream_t stream) {
    Conv3Args p{};
    p.a = a;
    p.chunks = static_cast<int32_t>(a.ic / kChunk);
    p.xbytes = static_cast<uint32_t>(image_floats(a) * 4);
    p.wbytes = static_cast<uint32_t>(weight_bytes(a));
    const auto quads = [](const float *t, int64_t nb1, int64_t nb2, int64_t nb3) {
        return (reinterpret_cast<uintptr_t>(t) & 15) == 0 && nb1 % 4 == 0 && nb2 % 4 == 0 && nb3 % 4 == 0;
    };
    p.vec_y = a.ow % 4 == 0 && quads(a.y, a.ynb1, a.ynb2, a.ynb3);
    for (int s = 0; s < a.chain.count; ++s) {
        const DevStep &st = a.chain.steps[s];
        if (st.kind != kSilu && a.ow % 4 == 0 && st.nb[0] == 1 && quads(st.operand, st.nb[1], st.nb[2], st.nb[3]))
            p.vec_step |= 1u << s;
    }
    // The weights in the products' order, kept in the store when it has room,
    // as Winograd's transformed ones are.
    const int64_t wne[4] = {3, 3, a.ic, a.oc};
    const int64_t wnb[4] = {2, 6, 18, 18 * a.ic};
    bool ready = false;
    void *kept = store_entry(a.w, SDHIP_TYPE_F16, wne, wnb, kStoreConv3, 0, static_cast<size_t>(weight_bytes(a)),
                             static_cast<size_t>(weight_bytes(a)), stream, ready);
    _Float16 *wt = static_cast<_Float16 *>(kept != nullptr ? kept : work);
    p.w = wt;
    if (!ready) {
        KernelScope scope("conv3x3.weights", stream);
        SDHIP_LAUNCH(conv3_weights_kernel,
                     dim3(static_cast<uint32_t>(p.chunks), static_cast<uint32_t>(ceil_div(a.oc, 8))), dim3(256), 0, stream,
                     a.w, a.oc, a.ic, wt);
        const hipError_t err = hipGetLastError();
        if (err != hipSuccess) return launched(err, "conv2d weights");
        if (kept != nullptr) store_publish(kept);
    }
    KernelScope scope("conv3x3.products", stream);
    Work unused;
    const int shape = shape_of(a, unused);
    const hipError_t err = shape == 1 ? launch<Wide>(p, stream) : shape == 2 ? launch<Mid>(p, stream) : launch<Narrow>(p, stream);
    return launched(err, "conv2d 3x3");
}

}  // namespace sdhip
