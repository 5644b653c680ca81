// sr_texture.h -- TextureData::CreateFromRGBA8 (Texture.cpp:119-199) on the
// device: the 32x32 Morton tiling of every level and the mip chain, each mip
// resized from the base level with stb_image_resize's Mitchell filter as
// stbir_resize_uint8 computes it (Texture.cpp:196).
//
// The resize is separable and rounds after each pass: a horizontal pass
// weights every input row into a row of float4 as wide as the level
// (k_mip_rows), a vertical pass weights those rows into the level's texels,
// encodes them and writes them at their tiled addresses (k_mip_cols), with
// the same float operations in the same order as the library. Every level is
// made by the same two launches (level 1 of a large texture by two more).
//
// Sizes are powers of two, so a level is 2^s times smaller than the base
// along an axis and its filter is the same for every output: input texel j
// reaches the four outputs K - 3 .. K, K = floor((j + 1.5 * 2^s) / 2^s), and
// with a = j + 1.5 * 2^s - K * 2^s its weight in output K - q is weight
// a + q * 2^s of the filter (filter offsets are exact in float; the library's
// contributor ranges floor((j + 0.5) / 2^s -+ 1.5) are K - 3 and K).
// A sum over up to 4 * 2^s texels has one order, so a line (a row; in the
// second pass a column) is a serial chain. A lane therefore walks a line's
// texels once, in order, for one channel, with the four open outputs' sums in
// registers: 16 lines x 4 channels a wave, the weights the same for all of
// them (staged through LDS), each texel decoded once for its four weights. Lines are cut into
// segments of whole outputs (at least 256 texels, plus the 3 * 2^s that the
// neighbours share), so the low levels, which have the work, run as many
// short chains and the high ones, which have 4 * 2^s taps but few outputs,
// as few long ones, all at the same time. Before, a thread per output read
// every tap (source, weight and texel) with one load after another, level
// after level: 1024^2 took 4,300 us in these kernels (2.7 ms rows, 1.6 ms
// columns) and 4 IEEE divisions a tap.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace srg {

// x (even bits) or y (odd bits) of a 10-bit Morton index inside a 32x32 tile.
__device__ __forceinline__ uint32_t morton_compact5(uint32_t m)
{
    m &= 0x155u;
    m = (m | (m >> 1)) & 0x133u;
    m = (m | (m >> 2)) & 0x10Fu;
    m = (m | (m >> 4)) & 0x01Fu;
    return m;
}

// The inverse: the low 5 bits of v at the even bit positions.
__device__ __forceinline__ uint32_t morton_spread5(uint32_t v)
{
    v = (v | (v << 4)) & 0x10Fu;
    v = (v | (v << 2)) & 0x133u;
    v = (v | (v << 1)) & 0x155u;
    return v;
}

// TileTexture (Texture.cpp:73-101) of the linear RGBA8 base level (its sides
// are multiples of 32), and zeros in the `nzero` words that follow the levels
// whose sides are: the levels with texels of 32-aligned padding, which
// k_mip_cols does not write.
__global__ __launch_bounds__(256) void k_tex_tile(const uint32_t* __restrict__ src, uint32_t w, uint32_t* __restrict__ dst,
                                                  uint32_t tiles_w, uint32_t ntexels, uint32_t* __restrict__ zero,
                                                  uint32_t nzero)
{
    const uint32_t t = blockIdx.x * 256u + threadIdx.x;
    if (t < ntexels) {
        const uint32_t tile = t >> 10, m = t & 1023u;
        const uint32_t x = ((tile % tiles_w) << 5) | morton_compact5(m);
        const uint32_t y = ((tile / tiles_w) << 5) | morton_compact5(m >> 1);
        dst[t] = src[(size_t)y * w + x];
    } else if (t - ntexels < nzero) {
        zero[t - ntexels] = 0u;
    }
}

// A level of a pass. Workgroups [block, next level's block) of the launch are
// its (line group of 16, segment) pairs, segments innermost.
struct MipPass {
    uint32_t block;
    uint32_t log2_scale;  // s: the axis is 2^s times shorter on this level
    uint32_t out;         // outputs of a line
    uint32_t lines;       // lines (rows; columns in the second pass)
    uint32_t seg;         // outputs of a segment
    uint32_t segs;        // segments of a line
    uint32_t rows_at;     // first float4 of the level's rows
    uint32_t dst_at;      // second pass: first word of the level in the texture
};
constexpr uint32_t kMaxMips = 14;
struct MipPasses {
    MipPass level[kMaxMips];
    uint32_t n;
};
constexpr uint32_t kMipSegTexels = 256;
// First float4 of the weights of scale s >= 1: 2^s of them, (weights a, a +
// 2^s, a + 2 * 2^s, a + 3 * 2^s) for a = 0 .. 2^s - 1.
__host__ __device__ constexpr uint32_t mip_weights_at(uint32_t s) { return (1u << s) - 2u; }

// Plain vectors: arrays of HIP's float4 / uint4 held over a loop go to scratch.
typedef float MipF4 __attribute__((ext_vector_type(4)));
typedef uint32_t MipU4 __attribute__((ext_vector_type(4)));
typedef MipU4 MipU4Any __attribute__((aligned(4)));  // four texels from any texel on

// The lines of a one-wave workgroup: outputs [k0, k1) of the filter of scale
// s over lines of `in` texels. The texels and their weights come in stages of
// STAGE through LDS (the loads of the next stage are in flight while this one
// is summed; a stage wholly past an end of the line is its edge texel and
// loads nothing, as on the highest levels, most of whose taps are clamped).
//   fetch(j0)      starts the loads of texels j0 .. j0 + STAGE - 1
//   commit()       puts them in LDS
//   get(i, v)      this lane's values of texels i .. i + 15 of the stage
//   edge(j)        this lane's value of texel j, from memory
//   emit(k, sum)   takes a finished output
template <int32_t STAGE, class Fetch, class Commit, class Get, class Edge, class Emit>
__device__ __forceinline__ void mip_line(uint32_t s, int32_t in, int32_t k0, int32_t k1, const MipF4* __restrict__ weights,
                                         MipF4* s_w, Fetch fetch, Commit commit, Get get, Edge edge, Emit emit)
{
    constexpr int32_t C = 16, NW = STAGE / 64;
    const int32_t scale = 1 << s, half3 = 3 << (s - 1);
    const int32_t a0 = k0 * scale, a1 = (k1 + 3) * scale;  // a = j + half3 over the segment
    const int32_t lane = (int32_t)threadIdx.x;
    auto clamped = [&](int32_t a) { return a + STAGE <= half3 || a - half3 >= in; };
    MipF4 wreg[NW];
    auto fetch_weights = [&](int32_t a) {
#pragma unroll
        for (int32_t i = 0; i < NW; ++i) wreg[i] = weights[(a + i * 64 + lane) & (scale - 1)];
    };
    float s0 = 0.0f, s1 = 0.0f, s2 = 0.0f, s3 = 0.0f;  // the sums of outputs K, K - 1, K - 2, K - 3
    fetch_weights(a0);
    if (!clamped(a0)) fetch(a0 - half3);
    for (int32_t A = a0; A < a1; A += STAGE) {
        const bool flat = clamped(A);
        float v[C];
        if (flat) {
            const float e = edge(A < half3 ? 0 : in - 1);
#pragma unroll
            for (int32_t i = 0; i < C; ++i) v[i] = e;
        } else {
            commit();
        }
#pragma unroll
        for (int32_t i = 0; i < NW; ++i) s_w[i * 64 + lane] = wreg[i];
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
        if (A + STAGE < a1) {
            fetch_weights(A + STAGE);
            if (!clamped(A + STAGE)) fetch(A + STAGE - half3);
        }
        const int32_t end = min(A + STAGE, a1);
        for (int32_t a = A; a < end; a += C) {
            const MipF4* w = s_w + (a - A);
            if (!flat) get(a - A, v);
            if (s >= 4) {  // the 16 texels have one K
                const int32_t K = a >> s;
                if (K >= k0 + 3 && K < k1) {
#pragma unroll
                    for (int32_t i = 0; i < C; ++i) {
                        const MipF4 f = w[i];
                        s0 = s0 + v[i] * f.x;
                        s1 = s1 + v[i] * f.y;
                        s2 = s2 + v[i] * f.z;
                        s3 = s3 + v[i] * f.w;
                    }
                } else {  // at the segment's ends: only its own outputs
                    const int32_t qlo = max(0, K - (k1 - 1)), qhi = min(3, K - k0);
                    auto one = [&](float& sum, uint32_t q) {
#pragma unroll
                        for (int32_t i = 0; i < C; ++i) sum = sum + v[i] * w[i][q];
                    };
                    if (qlo <= 0 && qhi >= 0) one(s0, 0);
                    if (qlo <= 1 && qhi >= 1) one(s1, 1);
                    if (qlo <= 2 && qhi >= 2) one(s2, 2);
                    if (qlo <= 3 && qhi >= 3) one(s3, 3);
                }
                if (((a + C) & (scale - 1)) == 0) {
                    if (K - 3 >= k0) emit(K - 3, s3);
                    s3 = s2;
                    s2 = s1;
                    s1 = s0;
                    s0 = 0.0f;
                }
            } else {
                // several outputs end among the 16 texels; the sums of outputs
                // that are not this segment's are dropped
#pragma unroll
                for (int32_t i = 0; i < C; ++i) {
                    const int32_t ai = a + i;
                    if (ai < a1) {
                        const MipF4 f = w[i];
                        s0 = s0 + v[i] * f.x;
                        s1 = s1 + v[i] * f.y;
                        s2 = s2 + v[i] * f.z;
                        s3 = s3 + v[i] * f.w;
                        if (((ai + 1) & (scale - 1)) == 0) {
                            const int32_t k = (ai >> s) - 3;
                            if (k >= k0) emit(k, s3);
                            s3 = s2;
                            s2 = s1;
                            s1 = s0;
                            s0 = 0.0f;
                        }
                    }
                }
            }
        }
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");  // the stage is read before the next is written
    }
}

__device__ __forceinline__ const MipPass& mip_pass_of(const MipPasses& P, uint32_t b)
{
    uint32_t i = 0;
    while (i + 1 < P.n && P.level[i + 1].block <= b) ++i;
    return P.level[i];
}

// Horizontal pass (stbir__resample_horizontal_downsample,
// stb_image_resize.h:1526-1655): rows[y][k] of every level, accumulated from
// 0 in the order of the input texels. One wave: 16 input rows x 4 channels of
// one segment. A byte is decoded as b / 255, by the reciprocal with one
// correction step (equal to the division for every byte).
__global__ __launch_bounds__(64) void k_mip_rows(const uint32_t* __restrict__ src, uint32_t w, MipPasses P,
                                                 const MipF4* __restrict__ weights, float* __restrict__ rows)
{
    const MipPass& L = mip_pass_of(P, blockIdx.x);
    const uint32_t b = blockIdx.x - L.block, seg = b % L.segs, line = (b / L.segs) * 16u + (threadIdx.x >> 2);
    const uint32_t sh = (threadIdx.x & 3u) * 8u, line0 = (b / L.segs) * 16u;
    // 16 rows x 256 texels, rows 260 words apart: the 16 rows' 16-byte reads
    // fall on different banks
    constexpr int32_t kStage = 256, kRow = 260;
    __shared__ __align__(16) uint32_t s_px[16 * kRow];
    __shared__ MipF4 s_w[kStage];
    const int32_t in = (int32_t)w, lane = (int32_t)threadIdx.x;
    MipU4 reg[16];
    float* out = rows + ((size_t)L.rows_at + (size_t)line * L.out) * 4u + (threadIdx.x & 3u);
    auto decode = [&](uint32_t px) {
        const float v = (float)((px >> sh) & 255u), q = v * (1.0f / 255.0f);
        return __builtin_fmaf(__builtin_fmaf(-255.0f, q, v), 1.0f / 255.0f, q);
    };
    mip_line<kStage>(
        L.log2_scale, in, (int32_t)(seg * L.seg), (int32_t)min((seg + 1u) * L.seg, L.out),
        weights + mip_weights_at(L.log2_scale), s_w,
        [&](int32_t j0) __attribute__((always_inline)) {
            const bool inside = j0 >= 0 && j0 + kStage <= in;
#pragma unroll
            for (int32_t r = 0; r < 16; ++r) {
                const uint32_t* row = src + (size_t)(line0 + (uint32_t)r) * w;
                const int32_t j = j0 + 4 * lane;
                if (inside) {
                    reg[r] = *(const MipU4Any*)(row + j);
                } else {
                    reg[r] = MipU4{ row[min(max(j, 0), in - 1)], row[min(max(j + 1, 0), in - 1)],
                                    row[min(max(j + 2, 0), in - 1)], row[min(max(j + 3, 0), in - 1)] };
                }
            }
        },
        [&]() __attribute__((always_inline)) {
#pragma unroll
            for (int32_t r = 0; r < 16; ++r) *(MipU4*)&s_px[r * kRow + 4 * lane] = reg[r];
        },
        [&](int32_t i, float v[16]) __attribute__((always_inline)) {
            const MipU4* p = (const MipU4*)&s_px[(lane >> 2) * kRow + i];
#pragma unroll
            for (int32_t k = 0; k < 4; ++k) {
                const MipU4 t = p[k];
                v[4 * k] = decode(t.x);
                v[4 * k + 1] = decode(t.y);
                v[4 * k + 2] = decode(t.z);
                v[4 * k + 3] = decode(t.w);
            }
        },
        [&](int32_t j) __attribute__((always_inline)) { return decode(src[(size_t)line * w + (uint32_t)j]); },
        [&](int32_t k, float sum) __attribute__((always_inline)) { out[(size_t)k * 4u] = sum; });
}

// STBIR__ENCODE_LINEAR8 (stb_image_resize.h:1743): saturate, * 255 in float,
// + 0.5 in double, truncate.
__device__ __forceinline__ uint32_t encode_u8(float f)
{
    f = f < 0.0f ? 0.0f : (f > 1.0f ? 1.0f : f);
    return (uint32_t)(int)((double)(f * 255.0f) + 0.5);
}

// Vertical pass, encode and tiling of every level
// (stbir__resample_vertical_downsample, :1987-2066, and the encode of
// :1695-1760). One wave: 16 columns x 4 channels of one segment; the four
// channels of a texel meet in one lane, which writes it.
__global__ __launch_bounds__(64) void k_mip_cols(const float* __restrict__ rows, uint32_t h, MipPasses P,
                                                 const MipF4* __restrict__ weights, uint32_t* __restrict__ dst)
{
    const MipPass& L = mip_pass_of(P, blockIdx.x);
    const uint32_t b = blockIdx.x - L.block, seg = b % L.segs, x = (b / L.segs) * 16u + (threadIdx.x >> 2);
    const uint32_t c = threadIdx.x & 3u;
    const bool inside = x < L.lines;  // levels narrower than 16 columns
    const float* col = rows + ((size_t)L.rows_at + (inside ? x : 0u)) * 4u + c;
    const uint32_t tiles_w = (L.lines + 31u) >> 5, tx = (x >> 5) * 1024u + morton_spread5(x & 31u);
    // 64 rows x 16 columns x 4 channels
    constexpr int32_t kStage = 64;
    __shared__ __align__(16) float s_v[kStage * 64];
    __shared__ MipF4 s_w[kStage];
    const int32_t in = (int32_t)h, lane = (int32_t)threadIdx.x;
    // a float4 (one texel of a row) per lane, four rows per load
    const MipF4* src = (const MipF4*)rows + L.rows_at;
    const uint32_t lx = min((b / L.segs) * 16u + (threadIdx.x & 15u), L.lines - 1u);
    MipF4 reg[16];
    mip_line<kStage>(
        L.log2_scale, in, (int32_t)(seg * L.seg), (int32_t)min((seg + 1u) * L.seg, L.out),
        weights + mip_weights_at(L.log2_scale), s_w,
        [&](int32_t j0) __attribute__((always_inline)) {
#pragma unroll
            for (int32_t r = 0; r < 16; ++r) {
                const int32_t j = min(max(j0 + 4 * r + (lane >> 4), 0), in - 1);
                reg[r] = src[(size_t)j * L.lines + lx];
            }
        },
        [&]() __attribute__((always_inline)) {
#pragma unroll
            for (int32_t r = 0; r < 16; ++r) *(MipF4*)&s_v[(4 * r + (lane >> 4)) * 64 + (lane & 15) * 4] = reg[r];
        },
        [&](int32_t i, float v[16]) __attribute__((always_inline)) {
#pragma unroll
            for (int32_t k = 0; k < 16; ++k) v[k] = s_v[(i + k) * 64 + lane];
        },
        [&](int32_t j) __attribute__((always_inline)) { return col[(size_t)j * L.lines * 4u]; },
        [&](int32_t k, float sum) __attribute__((always_inline)) {
            uint32_t v = encode_u8(sum) << (8u * c);
            v |= __shfl_xor(v, 1, 64);
            v |= __shfl_xor(v, 2, 64);
            const uint32_t y = (uint32_t)k;
            if (c == 0 && inside)
                dst[L.dst_at + (y >> 5) * tiles_w * 1024u + tx + (morton_spread5(y & 31u) << 1)] = v;
        });
}

}  // namespace srg
