// mid_kernel: products of 9-48 tokens (batches of sequences, verification of several drafts); included by kernels.hip.
//
// D = X . W^T on v_mfma_f32_32x32x16_bf16 with the prefill kernel's operand layout (A: 32 tokens, B: two 16-row tiles)
// and skinny_kernel's exact arithmetic: weights as bf16 (128 + q), the group's zero point and scale after its MFMAs.
// What bounds it: memory requests. Against a weight's bytes stand the activations, m x 256 bytes per group for each
// workgroup (at 20 tokens as much as two tiles' codes), and both come through the same queues; elimination builds of
// the [gate; up] product (34816 x 5120, int4) at 20 tokens took 21 us without activations and arithmetic, 28 us with
// the activations, 31 us in all. So a workgroup stages a step's activations once in LDS for its WT waves side by side
// over tiles, while the step before is computed, and K is split over the workgroup's WK wave rows (their sums meet in
// LDS) before it is split over the grid: few f32 partials (skinny_kernel's plain products write one per 4 groups, 34 at
// K = 17408, 14 MB at 20 tokens, which their consumer reads again).
//
// The sum of a group's activations, which the zero point multiplies, costs 32 two-wide dots per token block on the
// VALU or 8 MFMAs against ones. Each wave takes the dots of 8 / WT of the group's A fragments, the WT shares meet in
// LDS behind a barrier placed after the group's MFMAs, and one f32 MFMA (K = 2: the two lane halves' sums) subtracts
// the product with the zero points.
//
// Same-box graph replays, us per product against skinny_kernel (plain: with add_rmsnorm over the partials), at 12 / 20 /
// 32 tokens: [gate; up] 19456 x 2560 int4 17.5 / 21.3 / 22.8 -> 12.8 / 13.5 / 14.9, int8 25.5 / 28 / 30.5 -> 15 / 16.5 /
// 19.2, bf16 28.9 / 35.3 / 36.7 -> 20.3 / 21.6 / 24.8; 34816 x 5120 int4 27.6 / 38.2 / 41.4 -> (not taken) / 32.7 / 38.4,
// int8 43.8 / 53.4 / 57.3 -> 39.1 / 43.3 / 47.8; (5120, 17408) plain int4 21.8 / 26.7 / 33.1 -> 20.2 / 21.1 / 22.0, int8
// 28 / 33 / 40.5 -> 25 / 26 / 27.8; (2560, 9728) bf16 21.2 / 24.6 / 27.8 -> 16.2 / 17 / 18; whole rows (6144, 5120) int4
// 25 / 35 / 38.7 -> 10.8 / 13.8 / 15.9.
// Measured and not kept: three steps of weights in flight instead of one (the ring's registers, more barriers: 32.8 us
// for 29.8 on [gate; up]); waves with activations of their own and no barrier (33.3 us; the activations' traffic).
#pragma once

struct MidArgs {
    const uint8_t* codes;
    const void* scales;
    const uint16_t* zeros;
    const __bf16* x;
    const int32_t* xrows;  // argmax: x row of token t (null: t)
    void* y;
    unsigned long long* table;  // argmax
    int ldx, ldy;
    int tiles, G, m, valid;
    int steps, spp;  // steps of K (2^gs_shift groups each) and steps per split
    int gs_shift;
    uint32_t mask, magic;
};

// groups per wave and step: 4 KiB of codes of the wave's two tiles
template <int F>
__host__ __device__ constexpr int mid_ng() { return (F & (F_I8 | F_BF16)) ? 1 : 2; }

// LDS bytes of one step's activations: 2^gs_shift groups of ceil(m / 4) quads of 256-byte rows
__host__ __device__ inline int mid_xbytes(int m, int gs_shift) { return ((m + 3) / 4) * 1024 << gs_shift; }

// F, EPI: as skinny_kernel; TB: blocks of 32 tokens; WT: waves side by side over tiles, two tiles each (blockDim.x =
// 64 WT, blockDim.y = WK wave rows over K); LORA: with an adapter, whose arguments come in `ll`.
// (at least two waves per SIMD: the MFMA accumulators stay in VGPRs, as in skinny_m1_kernel)
template <int F, int EPI, int TB, int WT, bool LORA>
static __global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2))) void mid_kernel(
    MidArgs a, std::conditional_t<LORA, Launch, NoLora> ll) {
    extern __shared__ __attribute__((aligned(1024))) uint8_t msmem[];
    constexpr int NG = mid_ng<F>(), CW = CodeWords<F>::N;
    const int lane = threadIdx.x & 63, wt = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wk = __builtin_amdgcn_readfirstlane(threadIdx.y), WK = blockDim.y;
    const int NW = WT * WK, wave = wk * WT + wt;
    const int l32 = lane & 31, lh = lane >> 5, l16 = lane & 15;
    const int T = a.tiles, G = a.G;
    // the workgroup's tokens: all of them, or (narrow_launch) block blockIdx.z of 32 TB
    const int M = min(a.m - 32 * TB * (int)blockIdx.z, 32 * TB);
    const __bf16* const x0 = a.x + (size_t)(32 * TB) * blockIdx.z * a.ldx;
    const int tile0 = (blockIdx.x * WT + wt) * 2;
    const int tt = min(tile0 + (l32 >> 4), T - 1);
    const int s0 = blockIdx.y * a.spp, s1 = min(s0 + a.spp, a.steps);
    const int quads4 = (M + 3) >> 2, GS = 1 << a.gs_shift, XB = quads4 * 1024 << a.gs_shift;
    float* const xsums = (float*)(msmem + 2 * XB);  // [wave row][group][token block][lane][WT]
    int* const xtab = (int*)(xsums + WK * NG * TB * 64 * WT);  // argmax: the tokens' rows of x
    uint32_t magic;
    asm volatile("v_mov_b32 %0, %1" : "=v"(magic) : "s"(a.magic));
    const uint32_t mask = a.mask;

    if constexpr (EPI == EPI_ARGMAX) {  // (read once: an index load in every step would wait for the weights in flight)
        for (int i = wave * 64 + lane; i < M; i += NW * 64) xtab[i] = a.xrows ? a.xrows[i] : i;
        __syncthreads();
    }
    // one step's activations, global -> LDS directly, into buffer `buf`: row r of a group (256 bytes) holds token
    // min(r, M - 1), its 16-byte chunk k at slot k ^ (r % 16), so that the 16 rows of a read hit all banks once
    auto stage = [&](int s, int buf) __attribute__((always_inline)) {
        for (int p = wave; p < quads4 << a.gs_shift; p += NW) {
            const int gi = p & (GS - 1), q = p >> a.gs_shift;
            const int g = min((s << a.gs_shift) + gi, G - 1);
            const int slot = 4 * q + (lane >> 4), row = min(slot, M - 1);
            const size_t xr = EPI == EPI_ARGMAX ? (size_t)xtab[row] : (size_t)row;
            const __bf16* src = x0 + xr * a.ldx + (size_t)g * QG + 8 * ((lane & 15) ^ (slot & 15));
            __builtin_amdgcn_global_load_lds((const void*)src, (lds_ptr)(msmem + buf * XB + (gi * quads4 + q) * 1024), 16,
                                             0, 0);
        }
    };
    const uint32_t cg = (uint32_t)(((size_t)tt * G * 64 * CW + 16 * lh + l16) * 16);
    struct W {
        u32x4 c[NG][2][CW];
        uint32_t s[NG], z;
    };
    auto load = [&](int s, W& w) __attribute__((always_inline)) {
        const int gb = (s << a.gs_shift) + wk * NG;
        const int gq = NG == 2 ? min(gb, (G - 1) & ~1) : min(gb, G - 1);
        if constexpr (!(F & F_BF16)) {
            const size_t si = scale_idx(tt, T, gq, l16);
            if constexpr (NG == 2 && (F & F_S32) != 0) {
                const unsigned long long v =
                    __builtin_nontemporal_load((const unsigned long long*)((const float*)a.scales + si));
                w.s[0] = (uint32_t)v, w.s[1] = (uint32_t)(v >> 32);
            } else if constexpr (NG == 2) {
                w.s[0] = __builtin_nontemporal_load((const uint32_t*)((const uint16_t*)a.scales + si));
            } else {
                w.s[0] = (F & F_S32) ? __builtin_nontemporal_load((const uint32_t*)a.scales + si)
                                     : __builtin_nontemporal_load((const uint16_t*)a.scales + si);
            }
            if (F & F_ZP) w.z = __builtin_nontemporal_load(a.zeros + zero_idx(tt, T, gq, l16));
        }
#pragma unroll
        for (int gi = 0; gi < NG; gi++) {
            const uint8_t* cb = a.codes + (size_t)min(gb + gi, G - 1) * 64 * CW * 16;
#pragma unroll
            for (int pc = 0; pc < 2; pc++)
#pragma unroll
                for (int h = 0; h < CW; h++)
                    w.c[gi][pc][h] = __builtin_nontemporal_load((const u32x4*)(cb + cg + (h * 64 + 32 * pc) * 16));
        }
    };
    f32x16 acc[TB][1];
#pragma unroll
    for (int b = 0; b < TB; b++)
#pragma unroll
        for (int e = 0; e < 16; e++) acc[b][0][e] = 0.0f;
    // LDS offset of the lane's first A fragment of token block b in a group
    int xr[TB];
#pragma unroll
    for (int b = 0; b < TB; b++) {
        const int r = min(32 * b + l32, M - 1);
        xr[b] = r * 256 + 16 * (lh ^ (r & 15));
    }
    auto scale = [&](const W& w, int gi) __attribute__((always_inline)) {
        if constexpr ((F & F_S32) != 0 || NG == 1) return __uint_as_float((F & F_S32) ? w.s[gi] : w.s[gi] << 16);
        else return __uint_as_float(gi ? (w.s[0] & 0xffff0000u) : (w.s[0] << 16));
    };
    auto compute = [&](int s, int buf, const W& w) __attribute__((always_inline)) {
        const int gb = (s << a.gs_shift) + wk * NG;
        constexpr bool SUM = !(F & F_BF16);
#pragma unroll
        for (int gi = 0; gi < NG; gi++) {
            const uint8_t* xg = msmem + buf * XB + (wk * NG + gi) * quads4 * 1024;
            auto frag = [&](int kk) __attribute__((always_inline)) -> bf16x8 {
                const int pc = kk & 1, i = kk >> 1;
                if (F & F_BF16) return __builtin_bit_cast(bf16x8, w.c[gi][pc][i % CW]);
                if (F & F_I8)
                    return i8_biased(w.c[gi][pc][(i >> 1) % CW][2 * (i & 1)], w.c[gi][pc][(i >> 1) % CW][2 * (i & 1) + 1]);
                return i4_biased(w.c[gi][pc][0][i], mask, magic);
            };
            const bool valid = gb + gi < G;  // wave-uniform
            f32x16 d[TB];
            float* const xs = xsums + (size_t)((wk * NG + gi) * TB) * 64 * WT;
            if (SUM && valid) {
                // the wave's share of the group's activation sums: 8 / WT of its A fragments, every lane its token's
                const bf16x2 one2 = __builtin_bit_cast(bf16x2, 0x3F803F80u);
#pragma unroll
                for (int b = 0; b < TB; b++) {
                    float sum[2] = {0.0f, 0.0f};
#pragma unroll
                    for (int k = 0; k < 8 / WT; k++) {
                        const u32x4 v = *(const u32x4*)(xg + (xr[b] ^ ((wt * (8 / WT) + k) << 5)));
#pragma unroll
                        for (int j = 0; j < 4; j++) {
                            const uint32_t p = v[j];  // (a copy: bit_cast of a vector's element takes element 0)
                            sum[j & 1] = __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2, p), one2, sum[j & 1], false);
                        }
                    }
                    xs[(b * 64 + lane) * WT + wt] = sum[0] + sum[1];
#pragma unroll
                    for (int e = 0; e < 16; e++) d[b][e] = 0.0f;
                }
            }
            if (valid) {
#pragma unroll
                for (int kk = 0; kk < 8; kk++) {
                    const bf16x8 bw = frag(kk);
#pragma unroll
                    for (int b = 0; b < TB; b++) {
                        const u32x4 xa = *(const u32x4*)(xg + (xr[b] ^ (kk << 5)));
                        if constexpr (SUM) d[b] = mfma32(xa, bw, d[b]);
                        else acc[b][0] = mfma32(xa, bw, acc[b][0]);
                    }
                }
            }
            if constexpr (SUM) {
                const float sc = scale(w, gi);
                const float ncz = (F & F_I8) ? -128.0f : (F & F_ZP) ? -(float)(128 + (int)((w.z >> (4 * ((gb + gi) & 3))) & 15u)) : -136.0f;
                if (WT > 1) {
                    __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0): this wave's sums are written
                    asm volatile("s_barrier" ::: "memory");
                }
                if (valid)
#pragma unroll
                for (int b = 0; b < TB; b++) {
                    const float* r = xs + (b * 64 + lane) * WT;
                    float sum = r[0];
#pragma unroll
                    for (int k = 1; k < WT; k++) sum += r[k];
                    d[b] = __builtin_amdgcn_mfma_f32_32x32x2f32(sum, ncz, d[b], 0, 0, 0);
#pragma unroll
                    for (int e = 0; e < 16; e++) acc[b][0][e] = __builtin_fmaf(sc, d[b][e], acc[b][0][e]);
                }
            }
        }
    };

    // each step's loads are issued a step ahead, into the buffer and registers of the step before it (whose readers have
    // passed the barrier)
    W w0, w1;
    stage(s0, 0);
    load(s0, w0);
    if constexpr (LORA) {
        // the adapter's delta (on split 0), shared by the wave rows, while the first step is on its way
        if (EPI == EPI_SILU || blockIdx.y == 0) lora_item32<EPI == EPI_SILU, TB, 1>(ll, tile0, 32 * TB * blockIdx.z, acc, nullptr, 0, wk, WK);
    }
    for (int s = s0; s < s1; s += 2) {
        __builtin_amdgcn_s_waitcnt(0);
        __syncthreads();
        if (s + 1 < s1) {
            stage(s + 1, 1);
            __builtin_amdgcn_sched_barrier(0);
            load(s + 1, w1);
        }
        compute(s, 0, w0);
        if (s + 1 >= s1) break;
        __builtin_amdgcn_s_waitcnt(0);
        __syncthreads();
        if (s + 2 < s1) {
            stage(s + 2, 0);
            __builtin_amdgcn_sched_barrier(0);
            load(s + 2, w0);
        }
        compute(s + 1, 1, w1);
    }

    // one accumulator register (bv: token block bv / 16, register bv % 16) of the finished sums
    const int tile = tile0 + (l32 >> 4), out = tile * TILE + l16;
    const bool tile_ok = tile < T;
    auto emit = [&](int bv, float val) __attribute__((always_inline)) {
        const int tok = 32 * (bv >> 4) + 8 * ((bv & 15) >> 2) + 4 * lh + (bv & 3);
        if (EPI == EPI_SILU) {
            const float up = __shfl_xor(val, 8);
            if (tile_ok && l16 < 8 && tok < M)
                ((__bf16*)a.y)[(size_t)tok * a.ldy + tile * 8 + l16] = (__bf16)(silu(val) * up);
        } else {
            if (tile_ok && tok < M)
                __builtin_nontemporal_store(val, (float*)a.y + ((size_t)blockIdx.y * a.m + 32 * TB * blockIdx.z + tok) * a.ldy + out);
            if (EPI == EPI_ARGMAX) {
                unsigned long long k = tile_ok && tok < M && out < a.valid ? argmax_key(val, out) : 0;
#pragma unroll
                for (int o = 1; o < 32; o <<= 1) k = max_u64(k, __shfl_xor(k, o));
                if (l32 == 0 && tok < M && k) argmax_spread_max(a.table, tok, k);
            }
        }
    };
    if (WK == 1) {
#pragma unroll
        for (int b = 0; b < TB; b++)
#pragma unroll
            for (int v = 0; v < 16; v++)
                if (32 * b + 8 * (v >> 2) + (v & 3) < M) emit(16 * b + v, acc[b][0][v]);
        return;
    }
    __syncthreads();  // the last step's readers are done
    float* red = (float*)msmem + (size_t)wave * TB * 16 * 64 + lane;
#pragma unroll
    for (int b = 0; b < TB; b++)
#pragma unroll
        for (int v = 0; v < 16; v++) red[(16 * b + v) * 64] = acc[b][0][v];
    __syncthreads();
    // each of a column's waves finishes its share of the registers: the K waves' sums in order
    for (int bv = wk; bv < 16 * TB; bv += WK) {
        if (32 * (bv >> 4) + 8 * ((bv & 15) >> 2) + (bv & 3) >= M) continue;
        const float* rp = (const float*)msmem + ((size_t)wt * TB * 16 + bv) * 64 + lane;
        float v = 0.0f;
        for (int k = 0; k < WK; k++) v += rp[(size_t)k * WT * TB * 16 * 64];
        emit(bv, v);
    }
}

template <int F, int EPI, int TB, int WT>
static hipError_t mid_launch(const Launch& l) {
    const int tiles = l.rows / TILE, G = l.cols / QG, wt = WT, wk = l.waves / wt;
    MidArgs a{};
    a.codes = (const uint8_t*)l.codes;
    a.scales = l.scales;
    a.zeros = l.zeros;
    a.x = (const __bf16*)l.x;
    a.xrows = l.xrows;
    a.y = l.y;
    a.table = l.argmax_table;
    a.ldx = l.ldx, a.ldy = l.ldy;
    a.tiles = tiles, a.G = G, a.m = l.m, a.valid = l.valid;
    int gs = wk * mid_ng<F>(), sh = 0;
    while ((1 << sh) < gs) sh++;
    a.gs_shift = sh;
    a.steps = (G + gs - 1) / gs;
    a.spp = (a.steps + l.split - 1) / l.split;
    a.mask = l.nib_mask, a.magic = l.bf16_magic;
    const size_t lds = std::max((size_t)mid_xbytes(l.m, sh) * 2 + (size_t)gs * TB * 64 * 4 * WT + (EPI == EPI_ARGMAX ? 64 * 4 : 0), wk > 1 ? (size_t)wt * wk * TB * 4096 : 0);
    const dim3 grid((tiles + 2 * wt - 1) / (2 * wt), l.split), block(64 * wt, wk);
    if (l.lora_rank) {
        if constexpr (EPI != EPI_ARGMAX)
            hipLaunchKernelGGL((mid_kernel<F, EPI, TB, WT, true>), grid, block, lds, l.stream, a, l);
    } else {
        hipLaunchKernelGGL((mid_kernel<F, EPI, TB, WT, false>), grid, block, lds, l.stream, a, NoLora{});
    }
    hipError_t e = hipGetLastError();
    if (e == hipSuccess && EPI == EPI_ARGMAX) e = argmax_fold(l, l.m);
    return e;
}

// the kernel of a launch whose partition (api.hip mid_partition) is l.tile_waves x l.waves / l.tile_waves, l.split
template <int F, int EPI>
static hipError_t mid_epi(const Launch& l) {
    auto go = [&](auto TBc) {
        constexpr int TB = decltype(TBc)::value;
        // (the widths that mid_partition gives: 8 for split-K products, and int4 above 32 tokens 2 or 4 columns)
        constexpr bool narrow = TB == 1 || mid_ng<F>() == 1;
        if (l.tile_waves == 4) return mid_launch<F, EPI, TB, 4>(l);
        if (l.tile_waves == 2) return mid_launch<F, EPI, TB, 2>(l);
        if constexpr (narrow) {
            if (l.tile_waves == 1) return mid_launch<F, EPI, TB, 1>(l);
        }
        if constexpr (narrow && EPI == EPI_PLAIN) {
            if (l.tile_waves == 8) return mid_launch<F, EPI, TB, 8>(l);
        }
        return hipErrorInvalidConfiguration;
    };
    if constexpr (EPI != EPI_ARGMAX) {  // (the argmax: up to 32 tokens)
        if (l.m > 32) return go(std::integral_constant<int, 2>{});
    }
    return go(std::integral_constant<int, 1>{});
}

// y = the sum of `splits` partials of n4 float4 each, in order (y of any alignment). (A template, so that only the object
// of the format that launches it holds it.)
template <int F>
static __global__ __launch_bounds__(64) void sum_narrow_kernel(const float* x, int splits, size_t n4, float* y) {
    const size_t i = (size_t)blockIdx.x * 64 + threadIdx.x;
    if (i >= n4) return;
    constexpr int B = 16;  // partials loaded ahead of their adds
    f32x4 v = {0.0f, 0.0f, 0.0f, 0.0f};
    for (int s0 = 0; s0 < splits; s0 += B) {
        f32x4 p[B];
#pragma unroll
        for (int j = 0; j < B; j++)
            if (s0 + j < splits) p[j] = ((const f32x4*)x)[(size_t)(s0 + j) * n4 + i];
#pragma unroll
        for (int j = 0; j < B; j++)
            if (s0 + j < splits) v += p[j];
    }
#pragma unroll
    for (int e = 0; e < 4; e++) y[4 * i + e] = v[e];
}

// Plain products of more than 48 tokens on dense bf16 matrices of few rows (up to NARROW_TILES tiles: a LoRA adapter's
// stacked A, a DeltaNet in_ba projection), on mid_kernel over blocks of 32 tokens: the prefill kernel's 64 x 128 items
// are a handful there, each walking all of K. Bound by the activations, read once; so K is split over the grid until
// the launch has a few hundred workgroups, and a second launch (sum_narrow) adds the partials, kept in the stream-K
// scratch, into one row of sums per token: split 1 to the caller (whose fused adapter epilogue then stages it in LDS).
// An adapter of the product itself is added to split 0's sums before them, as in mid_kernel's other products, so that
// outputs without a delta keep the order of their sums.
// Kernel trace at 333 tokens, 32 x 5120 / 16 x 17408: 29.7 us (24 items) -> 6.3 + 4.8 / 6.4 + 4.8 us (55 / 187
// workgroups, then the sum). Over 16-256 rows, K 1024-17408 and 49-2048 tokens it is 0.2-1.0 times the prefill kernel's
// time with the sum of its partials (256 x 5120 at 49 / 333 / 2048 15.5 / 17.5 / 38.5 -> 9.3 / 11.4 / 24.0), 1.04 at one
// corner (256 x 1024 at 2048 11.9 -> 12.4).
template <int F>
static hipError_t narrow_launch(const Launch& l) {
    static_assert(F == F_BF16, "dense bf16");
    const int pairs = (l.rows / TILE + 1) / 2, wt = pairs >= 4 ? 4 : pairs >= 2 ? 2 : 1;
    MidArgs a{};
    a.codes = (const uint8_t*)l.codes;
    a.x = (const __bf16*)l.x;
    a.y = l.narrow > 1 ? (void*)l.sk_part : l.y;
    a.ldx = l.ldx, a.ldy = l.ldy;
    a.tiles = l.rows / TILE, a.G = l.cols / QG, a.m = l.m;
    const int wk = 8 / wt;
    a.gs_shift = wt == 4 ? 1 : wt == 2 ? 2 : 3;
    a.steps = (a.G + wk - 1) / wk;
    a.spp = (a.steps + l.narrow - 1) / l.narrow;
    const size_t lds = std::max((size_t)mid_xbytes(32, a.gs_shift) * (a.spp > 1 ? 2 : 1), (size_t)8 * 4096);
    const dim3 grid((pairs + wt - 1) / wt, l.narrow, (l.m + 31) / 32), block(64 * wt, wk);
    auto go = [&](auto WTc) {
        constexpr int WT = decltype(WTc)::value;
        if (l.lora_rank) hipLaunchKernelGGL((mid_kernel<F, EPI_PLAIN, 1, WT, true>), grid, block, lds, l.stream, a, l);
        else hipLaunchKernelGGL((mid_kernel<F, EPI_PLAIN, 1, WT, false>), grid, block, lds, l.stream, a, NoLora{});
    };
    if (wt == 4) go(std::integral_constant<int, 4>{});
    else if (wt == 2) go(std::integral_constant<int, 2>{});
    else go(std::integral_constant<int, 1>{});
    if (hipError_t e = hipGetLastError(); e != hipSuccess || l.narrow == 1) return e;
    const size_t n4 = (size_t)l.m * l.rows / 4;
    hipLaunchKernelGGL(sum_narrow_kernel<F>, dim3((unsigned)((n4 + 63) / 64)), dim3(64), 0, l.stream, l.sk_part, l.narrow, n4,
                       (float*)l.y);
    return hipGetLastError();
}
