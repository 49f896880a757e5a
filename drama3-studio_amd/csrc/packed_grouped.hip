// Packed-integer expert banks for many route pairs: tiled grouped GEMMs on
// 8-bit MFMA operands over the moe_align tile map.  INT8 ConvRot (mode 1), W6A8
// (2) and W4A8 codebook (3) multiply on i8 MFMA, W4A8-g128 (4) and W6A8-g128
// (5) on FP8 MFMA, each under the arithmetic of its decode kernels:
//   modes 1-3: INT8 rows x INT8 weights (decoded exactly as packed_decode.hpp
//              does), int32 sums, y = bf16(acc * s_a * s_channel); gate/up:
//              act = bf16(bf16(silu(gate)) * up); down: * route weight (fp32);
//   modes 4-5: FP8 rows x integer levels exact in E4M3 (wfmt.hpp), per
//              128-column block acc = fma(dot * s_x, s_w, acc); gate/up rounded
//              through the compute dtype, h = silu(gate) * up, FP8 per
//              128-group; down: * route weight (fp32).  Gate/up sums as the
//              decode kernel's waves do (kDecodeUpWaves chains, added in
//              order), so a route row's value does not depend on how its call
//              was split: bit for bit that of a decode call.
// Replaces the reference's Triton _quant_gemm over large batches
// (src/drama_low_vram/quantized_kernels.py:115-214).
//
// Workgroup = (64-row tile of one expert's sorted pairs, 128 weight rows), 4
// waves; a wave owns two 16-row MFMA column tiles (gate/up: 16 gate rows and
// the matching 16 up rows, so SiLU * up is a register epilogue).  The weight
// stream bounds these calls, so weights go straight from global memory into
// the registers of the one wave that uses them and are decoded once per tile;
// a block's registers take the same block of the next K step as soon as it is
// decoded.  Activation rows (shared by the waves) go through a double-buffered
// LDS tile, loaded the same step ahead, one barrier per step.  Row tiles past
// the expert's last pair are skipped in 16-row units (1 to 4 of them).
// Modes 4-5 store the hidden fp32; one pass quantizes it for the down kernel.
//
// Measured gate/up + down against the column-group kernel (modes 1-3: 16 columns
// a workgroup, 16 rows a pass) and consecutive decode calls (4-5), E 128 H 2048
// I 768: INT8 197 tokens 276 + 313 -> 87 + 57 us (4.2 TB/s), W6A8 512 tokens 201
// + 194 -> 117 + 72 us, a W6A8-g128 layer at 301 tokens 2419 -> 201 us.  INT8
// waits for its one K step of loads; decode instructions and their latency bound
// the 6-bit formats.  (Small banks: see tiled_projection in abi.cpp.)
#include <algorithm>
#include <type_traits>

#include "common.hpp"
#include "fp8_util.hpp"
#include "kernels.hpp"
#include "packed_decode.hpp"
#include "tile_map.hpp"

namespace dmoe {

namespace {

// Four waves (128 weight rows): more, smaller workgroups even out the chip's
// last ones (8 waves measured 97 instead of 67 us for W6A8-g128 down at 301
// tokens).
constexpr int kPgWaves = 4, kPgThreads = kPgWaves * kWave;
constexpr int kPgMaxHiddenBlocks = kMaxInter / 128;

constexpr int pg_sub(int mode, bool gateup) { return (mode == 2 || mode == 3) && gateup ? 2 : 1; }
constexpr int pg_groups(int mode, bool gateup) { return gateup && mode >= 2 ? 3 : 4; }

template <int MODE, bool GATEUP>
struct Fmt {
    static constexpr bool kFp8 = MODE >= 4;
    static constexpr int kWf = MODE == 4 ? kWfInt4 : kWfInt6;
    // pg_sub, pg_groups: 128-column blocks of a K step, workgroups per CU (3:
    // 168 registers, 4: 128).  Measured for W6A8 gate/up at 512 tokens (2, 3)
    // 112 us vs (1, 4) 127, down 75 vs 68.7; INT8 90.6 + 64.2 vs 89.8 + 60.6
    // (197 tokens).
    static constexpr int kSub = pg_sub(MODE, GATEUP);
    // Sums along K of the group-128 gate/up: the decode kernel's waves each sum
    // a chain of K blocks and add the chains in wave order.  Two sums a result
    // need 3 workgroups' registers (at 4 they spill: a W6A8-g128 layer at 301
    // tokens 277 us).
    static constexpr int kChains = kFp8 && GATEUP ? kDecodeUpWaves : 0;
    using Acc = std::conditional_t<kFp8, v4f, v4i>;
};

template <int MODE, bool GATEUP>
struct alignas(16) PackedLds {
    uint8_t a[2][Fmt<MODE, GATEUP>::kSub][kGroupM * 128];  // [buffer][128-column block of the step]: swizzled 16-byte chunks
    int pair[kGroupM];                     // original pair of each tile row (-1: past the expert)
    float sa[kGroupM], wt[kGroupM];        // its activation scale and route weight
    // modes 4-5 down: hidden scale of each block and row
    float rs[MODE >= 4 && !GATEUP ? kPgMaxHiddenBlocks : 1][kGroupM];
    int8_t tab[MODE == 3 ? 256 * 16 : 16]; // mode 3: INT8 weight of (scale byte, code)
};

// One lane's weight bytes of one row and 128-column block.
template <int MODE, bool FP8 = (MODE >= 4)>
struct BlockRaw {
    PackedRaw v;
};
template <int MODE>
struct BlockRaw<MODE, true> {
    WRaw<MODE == 4 ? kWfInt4 : kWfInt6> v;
    uint32_t scale;  // fp16 bits
};

// An expert's weights and scales as a wave-uniform base plus 32-bit offsets.
struct RowBase {
    const uint8_t *w, *sc;
};

// 128-column block kb of the row at byte offsets wo (its 16-byte slice grp
// included) and so: the bytes fetch_wrow / load_wraw give.
template <int MODE>
__device__ __forceinline__ BlockRaw<MODE> fetch_block(const RowBase& rb, uint32_t wo, uint32_t ho, uint32_t so, int kb) {
    BlockRaw<MODE> r;
    if constexpr (MODE == 1) {
        const uint8_t* w = rb.w + (wo + (uint32_t)kb * 128u);
        r.v.a = *(const v4i*)w;
        r.v.b = *(const v4i*)(w + 16);
    } else {
        const v4i lo = *(const v4i*)(rb.w + (wo + (uint32_t)kb * 64u));
        v2i hi = {0, 0};
        if constexpr (MODE == 2 || MODE == 5) hi = *(const v2i*)(rb.w + (ho + (uint32_t)kb * 32u));
        const uint32_t sc = *(const uint16_t*)(rb.sc + (so + (uint32_t)kb * ((MODE >= 4) ? 2u : 8u)));
        if constexpr (!(MODE >= 4)) {
            r.v.a = lo;
            r.v.b = v4i{hi[0], hi[1], 0, 0};
            r.v.x = sc;
        } else {
            if constexpr (MODE == 4) {
                r.v.v = lo;
            } else {
                r.v.lo = lo;
                r.v.hi = hi;
            }
            r.scale = sc;
        }
    }
    return r;
}

// The tile (m0, mc rows of expert e) x 128 weight rows, MT 16-row units of it.
// OPEN (kChains): chains summed side by side; it divides the K blocks.  A chain's
// blocks lie eight apart, so one chain at a time finds the pieces of a cache line
// of W6A8-g128's high parts steps apart, and with two streams of both planes in
// use the lines overflow an XCD's L2 (TCC misses of a launch 3.7 -> 6.3 M).  Open chains
// visit neighbouring blocks; the registers hold 4 chains up to 32 rows, 2 up to
// 48 and one above (2 above: 51 spills).  A layer at 40 / 128 / 600 tokens
// uniform and 301 Zipf, E 128 H 2048 I 768: one chain 169 / 190 / 207 / 208 us,
// 4 up to 32 rows 158 / 175 / 201 / 204, with 2 up to 48 156 / 172 / 197 / 203
// (W4A8-g128, one plane: 112 / 130 / 148 / 151 -> 111 / 129 / 145 / 150).
template <int MODE, bool GATEUP, int MT, int OPEN = 1>
__device__ __forceinline__ void packed_tile(const PackedGroupedArgs& a, PackedLds<MODE, GATEUP>& s, int e, int m0, int mc,
                                            int ct) {
    using F = Fmt<MODE, GATEUP>;
    constexpr int kSub = F::kSub;
    const QuantProjArgs& p = a.p;
    const int lane = threadIdx.x % kWave, wave = threadIdx.x / kWave;
    const int col = lane % 16, grp = lane / 16;
    const int half = p.N / 2, KB = p.K / 128, steps = KB / kSub;
    // this lane's two weight rows (rows past the matrix repeat its last; not stored)
    const int n0 = GATEUP ? ct * (kPgWaves * 16) + wave * 16 + col : ct * (kPgWaves * 32) + wave * 32 + col;
    int n[2];
    n[0] = min(n0, (GATEUP ? half : p.N) - 1);
    n[1] = GATEUP ? half + n[0] : min(n0 + 16, p.N - 1);
    // activation chunks of this thread: 16 bytes of tile rows ar + q * kRowStep
    // (rows past the last pair repeat it)
    constexpr int kRowStep = kPgThreads / 8, kChunks = (16 * MT + kRowStep - 1) / kRowStep;
    const int ar = threadIdx.x / 8, ac = threadIdx.x % 8;
    constexpr bool kByPosition = F::kFp8 && !GATEUP;  // the FP8 hidden rows lie in sorted order
    const uint8_t* asrc[kChunks];
#pragma unroll
    for (int q = 0; q < kChunks; ++q) {
        const int pos = m0 + min(ar + q * kRowStep, mc - 1);
        asrc[q] = (const uint8_t*)p.x + (int64_t)(kByPosition ? pos : p.order[pos] / p.row_div) * p.x_row_stride + ac * 16;
    }
    const int aoff = ar * 128 + ((ac ^ (ar % 8)) * 16);  // kRowStep is a multiple of 8: the same swizzle
    const RowBase rb{p.w + (int64_t)e * p.w_se, p.s + (int64_t)e * p.s_se};
    uint32_t wo[2], so[2];
#pragma unroll
    for (int c = 0; c < 2; ++c) {
        wo[c] = (uint32_t)n[c] * (uint32_t)p.w_sn + grp * (MODE == 1 ? 32 : 16);
        so[c] = (uint32_t)n[c] * (uint32_t)p.s_sn + (F::kFp8 ? 0 : grp * 2);
    }
    const uint32_t high = p.K / 2 - grp * 8;  // from a row's low slice to its 2-bit high slice (grp * 16 -> + grp * 8)

    v4i areg[kSub][kChunks];
    BlockRaw<MODE> raw[kSub][2];  // [block][row]
    auto load_a = [&](int st) {
#pragma unroll
        for (int b = 0; b < kSub; ++b)
#pragma unroll
            for (int q = 0; q < kChunks; ++q) areg[b][q] = *(const v4i*)(asrc[q] + (st * kSub + b) * 128);
    };
    auto stage_a = [&](int buf) {
#pragma unroll
        for (int b = 0; b < kSub; ++b)
#pragma unroll
            for (int q = 0; q < kChunks; ++q) *(v4i*)&s.a[buf][b][aoff + q * kRowStep * 128] = areg[b][q];
    };
    auto load_b = [&](int st, int b, int c) { raw[b][c] = fetch_block<MODE>(rb, wo[c], wo[c] + high, so[c], st * kSub + b); };
    // kChains: `part` are the open chains and acc the sum of the chains before them
    constexpr int MP = F::kChains ? MT : 1;
    typename F::Acc acc[MT][2], part[OPEN][MP][2];
#pragma unroll
    for (int mi = 0; mi < MT; ++mi) acc[mi][0] = acc[mi][1] = typename F::Acc{0, 0, 0, 0};
#pragma unroll
    for (int j = 0; j < OPEN; ++j)
#pragma unroll
        for (int mi = 0; mi < MP; ++mi) part[j][mi][0] = part[j][mi][1] = typename F::Acc{0, 0, 0, 0};

    // Multiply step st; a weight block's registers take the same block of step
    // `next` as soon as it is decoded.
    auto compute = [&](int st, int next, int buf, auto open) {
        const int o0 = ((2 * grp) ^ (col % 8)) * 16, o1 = ((2 * grp + 1) ^ (col % 8)) * 16;
#pragma unroll
        for (int b = 0; b < kSub; ++b) {
            const uint8_t* at = s.a[buf][b] + col * 128;
            __builtin_amdgcn_sched_barrier(0);  // one block's operands live at a time
            if constexpr (!F::kFp8) {
                PackedRow w[2];
#pragma unroll
                for (int c = 0; c < 2; ++c) {
                    if constexpr (MODE == 3) decode_w4a8_tab(raw[b][c].v, s.tab, w[c]);
                    else decode_wrow<MODE, false>(raw[b][c].v, n[c], nullptr, w[c]);
                    if constexpr (MODE != 1) load_b(next, b, c);
                }
#pragma unroll
                for (int mi = 0; mi < MT; ++mi) {
                    const v4i a0 = *(const v4i*)(at + mi * 16 * 128 + o0), a1 = *(const v4i*)(at + mi * 16 * 128 + o1);
#pragma unroll
                    for (int c = 0; c < 2; ++c) {
                        acc[mi][c] = mfma_i8(a0, w[c].r[0], acc[mi][c]);
                        acc[mi][c] = mfma_i8(a1, w[c].r[1], acc[mi][c]);
                    }
                }
                // INT8 products read the loaded registers themselves, so these
                // are reloaded after them (before them the loop copied every
                // block and waited for it: a layer at 197 tokens 186 -> 179 us;
                // two or three steps ahead, at 3 workgroups per CU: 192).
                if constexpr (MODE == 1) {
                    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                    for (int c = 0; c < 2; ++c) load_b(next, b, c);
                }
            } else {
                const v4f zero = {0, 0, 0, 0};
#pragma unroll
                for (int c = 0; c < 2; ++c) {
                    // Converted here, not in the multiply-adds below: the loaded
                    // word would stay live past the reload, which then takes
                    // another register and a wait and a copy at the loop's end.
                    float sw = f16_to_f32((uint16_t)raw[b][c].scale);
                    asm volatile("" : "+v"(sw));
                    v8i lo, hi;
                    if (c > 0) __builtin_amdgcn_sched_barrier(0);
                    expand_w<F::kWf>(raw[b][c].v, lo, hi);
                    load_b(next, b, c);
#pragma unroll
                    for (int mi = 0; mi < MT; ++mi) {
                        const v4i a0 = *(const v4i*)(at + mi * 16 * 128 + o0), a1 = *(const v4i*)(at + mi * 16 * 128 + o1);
                        const v8i av = {a0[0], a0[1], a0[2], a0[3], a1[0], a1[1], a1[2], a1[3]};
                        const v4f rs = *(const v4f*)(GATEUP ? &s.sa[16 * mi + 4 * grp] : &s.rs[GATEUP ? 0 : st * kSub + b][16 * mi + 4 * grp]);
                        v4f d = mfma_fp8(av, lo, zero);
                        if constexpr (MODE == 5) d = mfma_fp8(av, hi, d);
                        v4f& sum = F::kChains ? part[decltype(open)::value][F::kChains ? mi : 0][c] : acc[mi][c];
#pragma unroll
                        for (int i = 0; i < 4; ++i) sum[i] = fmaf(d[i] * rs[i], sw, sum[i]);
                    }
                }
            }
        }
    };

    load_a(0);
#pragma unroll
    for (int b = 0; b < kSub; ++b)
#pragma unroll
        for (int c = 0; c < 2; ++c) load_b(0, b, c);
    if (threadIdx.x < kGroupM) {
        const int r = threadIdx.x, pr = p.order[m0 + min(r, mc - 1)];
        s.pair[r] = r < mc ? pr : -1;
        if (p.sa) s.sa[r] = p.sa[pr / p.row_div];
        if (p.weighted) s.wt[r] = load_as_f32(p.weights, pr, p.w_dtype);
    }
    if constexpr (MODE == 3) {  // entry 16 * scale byte + code; a thread's entries share the code
        const float level = *(const float*)(p.s + (int64_t)e * p.s_se + (int64_t)(threadIdx.x % 16) * p.s_sn + p.K / 16 + 4);
        for (int i = threadIdx.x; i < 256 * 16; i += kPgThreads) s.tab[i] = q8(level, e4m3((uint32_t)i / 16));
    }
    if constexpr (F::kFp8 && !GATEUP) {
        for (int i = threadIdx.x; i < kGroupM * KB; i += kPgThreads) {
            const int r = i / KB, kb = i % KB;
            s.rs[kb][r] = a.hs[(int64_t)(m0 + min(r, mc - 1)) * KB + kb];
        }
    }
    stage_a(0);
    // The barrier makes this step's activation rows visible; the buffer staged
    // into was read before it.  The last step loads itself again: no branch
    // around the loads, so the waits stay counted and never drain them.
    // the chains that end with this step go into the sum
    auto close_chains = [&] {
#pragma unroll
        for (int j = 0; j < OPEN; ++j) {
#pragma unroll
            for (int mi = 0; mi < MP; ++mi) {
#pragma unroll
                for (int c = 0; c < 2; ++c) {
                    acc[mi][c] += part[j][mi][c];
                    part[j][mi][c] = typename F::Acc{0, 0, 0, 0};
                }
            }
        }
    };
    constexpr int kC = F::kChains ? F::kChains : 1;
    if constexpr (OPEN == 1) {
        for (int i = 0, st = 0, buf = 0; i < steps; ++i, buf ^= 1) {
            // kChains: blocks w, w + kChains, .. of one chain w after the other
            const bool end = F::kChains == 0 || st + kC >= steps;
            const int after = F::kChains == 0 ? st + 1 : end ? st % kC + 1 : st + kC;
            const int next = i + 1 < steps ? after : st;
            load_a(next);
            lds_barrier();
            compute(st, next, buf, std::integral_constant<int, 0>{});
            if constexpr (F::kChains > 0) {
                if (end) close_chains();
            }
            stage_a(buf ^ 1);
            st = next;
        }
    } else {
        // OPEN neighbouring blocks st .., one of each open chain; after the
        // chains' last ones the next chains open
        for (int i = 0, st = 0; i < steps; i += OPEN) {
            const bool end = st + kC >= steps;
            const int after = end ? st % kC + OPEN : st + kC, last = i + OPEN < steps ? after : st + OPEN - 1;
            auto step = [&](auto open) {
                constexpr int J = decltype(open)::value;
                const int next = J + 1 < OPEN ? st + J + 1 : last;
                load_a(next);
                lds_barrier();
                compute(st + J, next, J % 2, open);
                if constexpr (J + 1 == OPEN) {
                    if (end) close_chains();
                }
                stage_a(J % 2 ^ 1);
            };
            step(std::integral_constant<int, 0>{});
            step(std::integral_constant<int, 1>{});
            if constexpr (OPEN == 4) {
                step(std::integral_constant<int, 2>{});
                step(std::integral_constant<int, 3>{});
            }
            st = after;
        }
    }

    // epilogue: a lane holds column `col` of each 16 x 16 result, rows 4 grp + i
    {
        float sb[2] = {1.0f, 1.0f};
        if constexpr (!F::kFp8) {
            sb[0] = channel_scale<MODE>(p, e, n[0]);
            sb[1] = channel_scale<MODE>(p, e, n[1]);
        }
#pragma unroll
        for (int mi = 0; mi < MT; ++mi) {
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int r = 16 * mi + 4 * grp + i, pr = s.pair[r];
                if (pr < 0) continue;
                float y[2];
                if constexpr (F::kFp8) {
                    y[0] = acc[mi][0][i];
                    y[1] = acc[mi][1][i];
                } else {
                    const float sa = s.sa[r];
                    y[0] = bf16_round((float)acc[mi][0][i] * sa * sb[0]);
                    y[1] = bf16_round((float)acc[mi][1][i] * sa * sb[1]);
                }
                if constexpr (GATEUP && F::kFp8) {
                    const float h = silu_f32(round_through(y[0], a.gu_dtype)) * round_through(y[1], a.gu_dtype);
                    if (n0 < half) a.h32[(int64_t)(m0 + r) * half + n0] = h;
                } else if constexpr (GATEUP) {
                    const float act = bf16_round(bf16_round(y[0] / (1.0f + expf(-y[0]))) * y[1]);
                    if (n0 < half) p.act[(int64_t)pr * half + n0] = __builtin_bit_cast(uint16_t, (__bf16)act);
                } else {
                    const float wt = s.wt[r];
#pragma unroll
                    for (int c = 0; c < 2; ++c) {
                        const int nc = n0 + 16 * c;
                        if (nc >= p.N) continue;
                        const int64_t o = (int64_t)pr * p.out_row_stride + nc;
                        if (p.weighted) ((float*)p.out)[o] = y[c] * wt;
                        else ((uint16_t*)p.out)[o] = __builtin_bit_cast(uint16_t, (__bf16)y[c]);
                    }
                }
            }
        }
    }
}

// Column tiles of N weight rows.
template <bool GATEUP>
__host__ __device__ constexpr int pg_cols(int N) {
    constexpr int kCols = kPgWaves * (GATEUP ? 16 : 32);
    return ((GATEUP ? N / 2 : N) + kCols - 1) / kCols;
}

template <int MODE, bool GATEUP>
__global__ __launch_bounds__(kPgThreads, pg_groups(MODE, GATEUP)) void packed_grouped_kernel(PackedGroupedArgs a) {
    __shared__ PackedLds<MODE, GATEUP> s;
    TileWork t;
    if (!take_tile(a, pg_cols<GATEUP>(a.p.N), t)) return;
    const int e = __builtin_amdgcn_readfirstlane(t.e), m0 = __builtin_amdgcn_readfirstlane(t.m0), mc = t.mc, ct = t.ct;
    if constexpr (Fmt<MODE, GATEUP>::kChains > 0) {
        if (a.p.K % 512 == 0 && mc <= 48) {
            if (mc <= 16) packed_tile<MODE, GATEUP, 1, 4>(a, s, e, m0, mc, ct);
            else if (mc <= 32) packed_tile<MODE, GATEUP, 2, 4>(a, s, e, m0, mc, ct);
            else packed_tile<MODE, GATEUP, 3, 2>(a, s, e, m0, mc, ct);
            return;
        }
    }
    if (mc <= 16) packed_tile<MODE, GATEUP, 1>(a, s, e, m0, mc, ct);
    else if (mc <= 32) packed_tile<MODE, GATEUP, 2>(a, s, e, m0, mc, ct);
    else if (mc <= 48) packed_tile<MODE, GATEUP, 3>(a, s, e, m0, mc, ct);
    else packed_tile<MODE, GATEUP, 4>(a, s, e, m0, mc, ct);
}

}  // namespace

// Whole K steps, and an expert's rows within 32-bit byte offsets.
bool packed_grouped_fits(int mode, int N, int K, int64_t w_sn, int64_t s_sn) {
    return mode >= 1 && mode <= 5 && K % (128 * std::max(pg_sub(mode, true), pg_sub(mode, false))) == 0 && N * w_sn < (int64_t(1) << 32) &&
           N * s_sn < (int64_t(1) << 32);
}

template <int MODE, bool GATEUP>
static void launch_mode(const PackedGroupedArgs& a, hipStream_t stream) {
    const dim3 grid(tile_grid(a.max_tiles, pg_cols<GATEUP>(a.p.N)));
    hipLaunchKernelGGL((packed_grouped_kernel<MODE, GATEUP>), grid, dim3(kPgThreads), 0, stream, a);
}

void launch_packed_grouped(const PackedGroupedArgs& a, hipStream_t stream) {
    auto go = [&](auto gateup) {
        constexpr bool kGateUp = decltype(gateup)::value;
        switch (a.p.mode) {
            case 1: launch_mode<1, kGateUp>(a, stream); break;
            case 2: launch_mode<2, kGateUp>(a, stream); break;
            case 3: launch_mode<3, kGateUp>(a, stream); break;
            case 4: launch_mode<4, kGateUp>(a, stream); break;
            default: launch_mode<5, kGateUp>(a, stream); break;
        }
    };
    if (a.p.gateup) go(std::true_type{});
    else go(std::false_type{});
}

}  // namespace dmoe
