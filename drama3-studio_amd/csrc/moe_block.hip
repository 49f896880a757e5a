// The rest of the MoE block around the routed experts (decode sizes): the
// router GEMV, the sigmoid-gated shared expert and the residual adds of
// BackboneDecodeGraph._route_impl / _shared_impl / _post_impl
// (src/drama_low_vram/backbone_graph.py:317-337), in the compute dtype bf16
// with every nn.Linear / elementwise boundary rounded as torch rounds it:
//   logits = bf16(x Wr^T)            -> fp32 for the router softmax
//   sgate  = bf16(sigmoid(bf16(x ws^T)))
//   act    = bf16(bf16(silu(bf16(x Wg^T))) * bf16(x Wu^T))
//   shared = bf16(sgate * bf16(act Wd^T))
//   out    = bf16(after_mixer + bf16(experts + shared))
// Dot products accumulate in fp32.
//
// Two launches bracket the routed experts: block_pre (router logits, shared
// gate, shared gate/up + SiLU) and block_post (shared down, gating, adds).
// Each is a batched GEMV: one wave per weight row (gate/up: the gate row and
// its up row), the row held in registers (16 bytes per lane per 512 columns:
// 64 bytes per lane for a 2048-wide bf16 row) while the token rows stream
// past it in chunks of kBlkTokens, read straight from global memory (every
// wave reads the same few kilobytes, so they stay in L2) with the row's own
// loads: one memory round trip at batch 1.  Sums are wave-wide by DPP.
//
// Calls of many tokens (block_tiled) take the tiled form of the same two
// launches (block_gemm_*_kernel below): the work is then a small dense GEMM
// and the GEMV's fp32 multiply-adds bound it.
#include <algorithm>

#include "common.hpp"
#include "kernels.hpp"

namespace dmoe {

namespace {

constexpr int kBlkWaves = 4, kBlkThreads = kBlkWaves * kWave;
constexpr int kBlkTokens = 2;           // token rows held in registers per chunk
// Calls of at most this many tokens take the GEMV (block_tiled).
constexpr int kBlkGemvTokens = 10;
constexpr int kBlkMaxK = 4096;          // reduction length (hidden or shared intermediate)

__device__ __forceinline__ float bf16v(uint16_t h) { return __uint_as_float((uint32_t)h << 16); }
__device__ __forceinline__ uint16_t to_bf16(float v) { return __builtin_bit_cast(uint16_t, (__bf16)v); }

// dot of this lane's 8-element slices (bf16 pairs in v4i) accumulated into acc.
__device__ __forceinline__ float dot8(const v4i& w, const v4i& x, float acc) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const uint32_t a = (uint32_t)w[i], b = (uint32_t)x[i];
        acc = fmaf(__uint_as_float(a << 16), __uint_as_float(b << 16), acc);
        acc = fmaf(__uint_as_float(a & 0xFFFF0000u), __uint_as_float(b & 0xFFFF0000u), acc);
    }
    return acc;
}

constexpr int kBlkChunks = kBlkMaxK / (kWave * 8);  // 16-byte pieces per lane of a kBlkMaxK row

// This lane's 16-byte pieces of a row (columns (c * 64 + lane) * 8 .. +7),
// every load issued at once; pieces past K are zero.
__device__ __forceinline__ void load_row(const uint16_t* w, int K, v4i (&v)[kBlkChunks]) {
    const int lane = threadIdx.x % kWave;
#pragma unroll
    for (int c = 0; c < kBlkChunks; ++c) {
        const int k = (c * kWave + lane) * 8;
        v[c] = k < K ? *(const v4i*)&w[k] : v4i{0, 0, 0, 0};
    }
}

// y[t] = sum_k w[k] x_t[k] for tokens t < n of a chunk whose rows are
// already in registers; every lane gets all sums.
template <int NT>
__device__ __forceinline__ void row_dots(const v4i (&wv)[kBlkChunks], const v4i (&xv)[NT][kBlkChunks], int n,
                                         float (&y)[NT]) {
#pragma unroll
    for (int t = 0; t < NT; ++t) {
        y[t] = 0.0f;
        if (t < n) {
#pragma unroll
            for (int c = 0; c < kBlkChunks; ++c) y[t] = dot8(wv[c], xv[t][c], y[t]);
        }
        y[t] = wave_sum_dpp(y[t]);
    }
}

// The chunk's token rows (t < n) straight from global memory (L2-resident:
// every wave reads the same few kilobytes), issued with the weight loads.
template <int NT>
__device__ __forceinline__ void load_tokens(const uint16_t* x, int64_t stride, int t0, int n, int K,
                                            v4i (&xv)[NT][kBlkChunks]) {
#pragma unroll
    for (int t = 0; t < NT; ++t) {
        if (t < n) load_row(x + (int64_t)(t0 + t) * stride, K, xv[t]);
        else {
#pragma unroll
            for (int c = 0; c < kBlkChunks; ++c) xv[t][c] = v4i{0, 0, 0, 0};
        }
    }
}

__global__ __launch_bounds__(kBlkThreads) void block_pre_kernel(BlockPreArgs a) {
    const int lane = threadIdx.x % kWave;
    const int H = a.hidden, E = a.experts, I = a.shared_inter;
    // rows: 0 .. E-1 router, E shared gate, E + 1 + j shared gate/up pair j
    const int rows = E + 1 + I;
    for (int r = blockIdx.x * kBlkWaves + threadIdx.x / kWave; r < rows; r += gridDim.x * kBlkWaves) {
        const bool pair = r > E;
        const int j = r - E - 1;
        v4i wv[kBlkChunks], uv[kBlkChunks];
        load_row(r < E ? a.router_w + (int64_t)r * a.router_row_stride
                       : r == E ? a.sgate_w : a.sg_w + (int64_t)j * a.sg_row_stride, H, wv);
        if (pair) load_row(a.su_w + (int64_t)j * a.su_row_stride, H, uv);
        for (int t0 = 0; t0 < a.tokens; t0 += kBlkTokens) {
            const int n = min(kBlkTokens, a.tokens - t0);
            v4i xv[kBlkTokens][kBlkChunks];
            load_tokens(a.x, a.x_row_stride, t0, n, H, xv);
            float y[kBlkTokens];
            row_dots(wv, xv, n, y);
            if (r < E) {
                // every lane holds every sum; lane t writes token t
#pragma unroll
                for (int t = 0; t < kBlkTokens; ++t)
                    if (lane == t && t < n) a.logits[(int64_t)(t0 + t) * a.logits_row_stride + r] = bf16_round(y[t]);
            } else if (r == E) {
#pragma unroll
                for (int t = 0; t < kBlkTokens; ++t)
                    if (lane == t && t < n) {
                        const float g = bf16_round(y[t]);
                        a.sgate[t0 + t] = to_bf16(1.0f / (1.0f + expf(-g)));
                    }
            } else {
                float u[kBlkTokens];
                row_dots(uv, xv, n, u);
#pragma unroll
                for (int t = 0; t < kBlkTokens; ++t)
                    if (lane == t && t < n) {
                        const float g = bf16_round(y[t]), up = bf16_round(u[t]);
                        const float sg = bf16_round(g / (1.0f + expf(-g)));
                        a.act[(int64_t)(t0 + t) * a.act_row_stride + j] = to_bf16(sg * up);
                    }
            }
        }
    }
}

__global__ __launch_bounds__(kBlkThreads) void block_post_kernel(BlockPostArgs a) {
    const int lane = threadIdx.x % kWave;
    const int H = a.hidden, I = a.shared_inter;
    for (int r = blockIdx.x * kBlkWaves + threadIdx.x / kWave; r < H; r += gridDim.x * kBlkWaves) {
        v4i wv[kBlkChunks];
        load_row(a.sd_w + (int64_t)r * a.sd_row_stride, I, wv);
        for (int t0 = 0; t0 < a.tokens; t0 += kBlkTokens) {
            const int n = min(kBlkTokens, a.tokens - t0);
            v4i xv[kBlkTokens][kBlkChunks];
            load_tokens(a.act, a.act_row_stride, t0, n, I, xv);
            float y[kBlkTokens];
            row_dots(wv, xv, n, y);
#pragma unroll
            for (int t = 0; t < kBlkTokens; ++t)
                if (lane == t && t < n) {
                    const int64_t tt = t0 + t;
                    const float s = bf16_round(bf16v(a.sgate[tt]) * bf16_round(y[t]));
                    const float e = bf16v(a.experts[tt * a.experts_row_stride + r]);
                    const float m = bf16_round(e + s);
                    a.out[tt * a.out_row_stride + r] = to_bf16(bf16v(a.residual[tt * a.residual_row_stride + r]) + m);
                }
        }
    }
}

// ------------------------------------------------------------ many tokens
// Tile = 64 token rows x 64 weight rows, 4 waves of 2 x 2 MFMA tiles (32 x 32)
// each, K in steps of 128 columns double-buffered in LDS through registers:
// step s + 1 is in flight while step s is multiplied, one barrier per step;
// two workgroups per CU (64 KB of LDS each) cover each other's waits.  The
// serial chain of 16 + 6 steps bounds these shapes (509 tokens: pre 3.5 GFLOP
// over 10 MB in 20 us, post 1.6 GFLOP over 10 MB in 12; 18 and 12 at 64);
// four steps in flight measured no better.
// The 16-byte chunk c of tile row r sits at chunk c ^ (r % 16), so the 16 rows
// of an operand read touch all banks.  Columns past K and rows past the
// matrices are zero.
constexpr int kBgTile = 64;             // token rows and weight rows of a tile
constexpr int kBgK = 128;               // columns per step
constexpr int kBgChunks = kBgK / 8;     // 16-byte chunks of a tile row per step
constexpr int kBgLoads = kBgTile * kBgChunks / kBlkThreads;  // 16-byte loads per thread, operand and step
static_assert(kBlkWaves == 4 && kBgChunks == 16, "wave tiling and swizzle");

struct BlockGemmLds {
    v4i a[2][kBgTile * kBgChunks];
    v4i b[2][kBgTile * kBgChunks];
};

// acc[mi][ni] = rows 32 (wave / 2) + 16 mi + .. of A times rows 32 (wave % 2) +
// 16 ni + .. of B; a_row(r) / b_row(r) give tile row r's source (null: zeros).
template <class ARow, class BRow>
__device__ __forceinline__ void block_gemm_tile(BlockGemmLds& s, int K, ARow a_row, BRow b_row, v4f (&acc)[2][2]) {
    const int lane = threadIdx.x % kWave, wave = threadIdx.x / kWave, col = lane % 16, grp = lane / 16;
    const int chunk = threadIdx.x % kBgChunks, row0 = threadIdx.x / kBgChunks;
    constexpr int kRowStep = kBlkThreads / kBgChunks;
    const uint16_t *ap[kBgLoads], *bp[kBgLoads];
#pragma unroll
    for (int i = 0; i < kBgLoads; ++i) {
        ap[i] = a_row(row0 + i * kRowStep);
        bp[i] = b_row(row0 + i * kRowStep);
    }
    v4i av[kBgLoads], bv[kBgLoads];
    auto load = [&](int k0) {
        const int k = k0 + chunk * 8;
        const bool in = k < K;
#pragma unroll
        for (int i = 0; i < kBgLoads; ++i) {
            av[i] = in && ap[i] ? *(const v4i*)(ap[i] + k) : v4i{0, 0, 0, 0};
            bv[i] = in && bp[i] ? *(const v4i*)(bp[i] + k) : v4i{0, 0, 0, 0};
        }
    };
    auto stage = [&](int buf) {
#pragma unroll
        for (int i = 0; i < kBgLoads; ++i) {
            const int r = row0 + i * kRowStep, at = r * kBgChunks + (chunk ^ (r % 16));
            s.a[buf][at] = av[i];
            s.b[buf][at] = bv[i];
        }
    };
#pragma unroll
    for (int mi = 0; mi < 2; ++mi) acc[mi][0] = acc[mi][1] = v4f{0, 0, 0, 0};
    const int ar = 32 * (wave / 2) + col, br = 32 * (wave % 2) + col;
    load(0);
    stage(0);
    for (int k0 = 0, buf = 0; k0 < K; k0 += kBgK, buf ^= 1) {
        const bool more = k0 + kBgK < K;
        if (more) load(k0 + kBgK);
        lds_barrier();  // this step is staged; the other buffer's readers are past it
#pragma unroll
        for (int t = 0; t < kBgK / 32; ++t) {
            const int c = (4 * t + grp) ^ col;
            const v4i a0 = s.a[buf][ar * kBgChunks + c], a1 = s.a[buf][(ar + 16) * kBgChunks + c];
            const v4i b0 = s.b[buf][br * kBgChunks + c], b1 = s.b[buf][(br + 16) * kBgChunks + c];
            acc[0][0] = mfma_bf16(__builtin_bit_cast(v8bf, a0), __builtin_bit_cast(v8bf, b0), acc[0][0]);
            acc[0][1] = mfma_bf16(__builtin_bit_cast(v8bf, a0), __builtin_bit_cast(v8bf, b1), acc[0][1]);
            acc[1][0] = mfma_bf16(__builtin_bit_cast(v8bf, a1), __builtin_bit_cast(v8bf, b0), acc[1][0]);
            acc[1][1] = mfma_bf16(__builtin_bit_cast(v8bf, a1), __builtin_bit_cast(v8bf, b1), acc[1][1]);
        }
        if (more) stage(buf ^ 1);
    }
}

// Column tiles: first the router rows with the shared gate as row E, then
// tiles of 32 shared gate/up columns (tile rows 32 q + c: gate columns 16 q + c,
// 32 q + 16 + c: the up rows, so SiLU * up stays in one lane).
constexpr int kBgActCols = 32;
inline __host__ __device__ int block_router_tiles(int experts) { return (experts + 1 + kBgTile - 1) / kBgTile; }

__global__ __launch_bounds__(kBlkThreads, 2) void block_gemm_pre_kernel(BlockPreArgs a) {
    __shared__ BlockGemmLds s;
    const int lane = threadIdx.x % kWave, wave = threadIdx.x / kWave, col = lane % 16, grp = lane / 16;
    const int E = a.experts, I = a.shared_inter, m0 = blockIdx.y * kBgTile;
    const int router_tiles = block_router_tiles(E);
    const bool router = (int)blockIdx.x < router_tiles;
    const int n0 = router ? blockIdx.x * kBgTile : (blockIdx.x - router_tiles) * kBgActCols;
    v4f acc[2][2];
    block_gemm_tile(
        s, a.hidden,
        [&](int r) { return m0 + r < a.tokens ? a.x + (int64_t)(m0 + r) * a.x_row_stride : nullptr; },
        [&](int r) -> const uint16_t* {
            if (router) {
                const int n = n0 + r;
                return n < E ? a.router_w + (int64_t)n * a.router_row_stride : n == E ? a.sgate_w : nullptr;
            }
            const int j = n0 + 16 * (r / 32) + r % 16;
            if (j >= I) return nullptr;
            return r % 32 < 16 ? a.sg_w + (int64_t)j * a.sg_row_stride : a.su_w + (int64_t)j * a.su_row_stride;
        },
        acc);
#pragma unroll
    for (int mi = 0; mi < 2; ++mi) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int64_t t = m0 + 32 * (wave / 2) + 16 * mi + 4 * grp + i;
            if (t >= a.tokens) continue;
            if (router) {
#pragma unroll
                for (int ni = 0; ni < 2; ++ni) {
                    const int n = n0 + 32 * (wave % 2) + 16 * ni + col;
                    const float y = bf16_round(acc[mi][ni][i]);
                    if (n < E) a.logits[t * a.logits_row_stride + n] = y;
                    else if (n == E) a.sgate[t] = to_bf16(1.0f / (1.0f + expf(-y)));
                }
            } else {
                const int j = n0 + 16 * (wave % 2) + col;
                const float g = bf16_round(acc[mi][0][i]), up = bf16_round(acc[mi][1][i]);
                if (j < I) a.act[t * a.act_row_stride + j] = to_bf16(bf16_round(g / (1.0f + expf(-g))) * up);
            }
        }
    }
}

__global__ __launch_bounds__(kBlkThreads, 2) void block_gemm_post_kernel(BlockPostArgs a) {
    __shared__ BlockGemmLds s;
    const int lane = threadIdx.x % kWave, wave = threadIdx.x / kWave, col = lane % 16, grp = lane / 16;
    const int H = a.hidden, m0 = blockIdx.y * kBgTile, n0 = blockIdx.x * kBgTile;
    v4f acc[2][2];
    block_gemm_tile(
        s, a.shared_inter,
        [&](int r) { return m0 + r < a.tokens ? a.act + (int64_t)(m0 + r) * a.act_row_stride : nullptr; },
        [&](int r) { return n0 + r < H ? a.sd_w + (int64_t)(n0 + r) * a.sd_row_stride : nullptr; }, acc);
#pragma unroll
    for (int mi = 0; mi < 2; ++mi) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int64_t t = m0 + 32 * (wave / 2) + 16 * mi + 4 * grp + i;
            if (t >= a.tokens) continue;
            const float sg = bf16v(a.sgate[t]);
#pragma unroll
            for (int ni = 0; ni < 2; ++ni) {
                const int n = n0 + 32 * (wave % 2) + 16 * ni + col;
                if (n >= H) continue;
                const float sh = bf16_round(sg * bf16_round(acc[mi][ni][i]));
                const float m = bf16_round(bf16v(a.experts[t * a.experts_row_stride + n]) + sh);
                a.out[t * a.out_row_stride + n] = to_bf16(bf16v(a.residual[t * a.residual_row_stride + n]) + m);
            }
        }
    }
}

}  // namespace

bool block_fits(int hidden, int shared_inter) {
    return hidden >= 8 && hidden <= kBlkMaxK && hidden % 8 == 0 && shared_inter >= 8 && shared_inter <= kBlkMaxK &&
           shared_inter % 8 == 0;
}

// The GEMV's time grows with its tokens and, once its rows fill the chip, with
// the rows; the tiled kernel's with its 128-column steps, which run in series.
// `tokens` x `rows` (at least `fill`, the rows that cost no more than fewer) is
// held against their crossing, (per_step * steps + base) / 10 tokens.  Measured,
// GEMV / tiled: pre at hidden 2048, 1665 rows 13.9 / 16.5 us at 11 tokens, 16.9
// / 16.8 at 14, 61 / 18 at 64; at 4096, 3329 rows 27.6 / 28.9 at 12, 34.7 / 28.8
// at 16; at 256, 145 rows 14.0 / 6.5 at 11.  Post at inter 2048, 512 rows 16.6 /
// 18.5 at 20, 19.1 / 18.6 at 24; at 768, 2048 rows 12.4 / 9.4 at 11.  The tiled
// grid's y dimension bounds it above.
static bool block_tiled(int tokens, int rows, int fill, int k, int per_step, int base) {
    const int64_t steps = (k + kBgK - 1) / kBgK;
    return tokens > kBlkGemvTokens && tokens <= 65535 * kBgTile &&
           (int64_t)tokens * std::max(rows, fill) * 10 > (per_step * steps + base) * fill;
}

void launch_block_pre(const BlockPreArgs& a, int cus, hipStream_t stream) {
    if (block_tiled(a.tokens, a.experts + 1 + 2 * a.shared_inter, 1664, a.hidden, 8, 13)) {
        const dim3 tiles(block_router_tiles(a.experts) + (a.shared_inter + kBgActCols - 1) / kBgActCols,
                         (a.tokens + kBgTile - 1) / kBgTile);
        hipLaunchKernelGGL(block_gemm_pre_kernel, tiles, dim3(kBlkThreads), 0, stream, a);
        return;
    }
    const int rows = a.experts + 1 + a.shared_inter;
    const int grid = std::max(1, std::min(4 * cus, (rows + kBlkWaves - 1) / kBlkWaves));
    hipLaunchKernelGGL(block_pre_kernel, dim3(grid), dim3(kBlkThreads), 0, stream, a);
}

void launch_block_post(const BlockPostArgs& a, int cus, hipStream_t stream) {
    if (block_tiled(a.tokens, a.hidden, 2048, a.shared_inter, 12, 38)) {
        const dim3 tiles((a.hidden + kBgTile - 1) / kBgTile, (a.tokens + kBgTile - 1) / kBgTile);
        hipLaunchKernelGGL(block_gemm_post_kernel, tiles, dim3(kBlkThreads), 0, stream, a);
        return;
    }
    const int grid = std::max(1, std::min(4 * cus, (a.hidden + kBlkWaves - 1) / kBlkWaves));
    hipLaunchKernelGGL(block_post_kernel, dim3(grid), dim3(kBlkThreads), 0, stream, a);
}

}  // namespace dmoe
