// Expert-grouped GEMMs in f32 on the bf16 matrix cores (gfx950).
//
// gfx950 has no f32 matrix rate above its vector FMA rate (157 TFLOP/s
// nominal; the vector form of this kernel reached 62 TFLOP/s at Nomic
// T=4096), while a bf16 MFMA runs 16 times that rate. Every f32 value is
// therefore split into three bf16 parts, 2^16 x = h + m + l: h = bf16(2^16 x),
// m and l likewise of what is left, all rounded to nearest even, the
// differences exact, so that the parts hold all 24 significand bits (split2). A
// product is summed from the six part products of relative size 2^-18 and
// above (l*h, h*l, m*m, m*h, h*m, h*h, smallest first), accumulated in f32 by
// the MFMA; the dropped ones (m*l, l*m, l*l) are below 2^-26 of it, a quarter
// of one f32 rounding (a sum of one single product comes within 1 ulp, where an
// FMA's is within 1/2: 2.6e-8 against 2.5e-8 rms; two products and more are closer
// than with FMAs). Summing 16 k per MFMA also rounds the running sum
// fewer times than one FMA per k did. Error against 64 bits (2-norm,
// relative): Nomic T=4096 4.0e-7 against 1.2e-6 for the vector kernel, Qwen3
// T=200 4.2e-7 against 1.2e-6, Qwen3-30B-A3B T=400 4.6e-7 against 1.3e-6 (with
// the small part products in the same accumulators as h*h: 1.0e-6 at Nomic
// T=4096, and 5 % less time).
// Measured, vector kernel -> this one: Nomic T=4096 fc1 547 -> 299 us, fc2
// 664 -> 241 us (193 f32 TFLOP/s in 1.16 PFLOP/s of bf16 products), step 1205
// -> 539 us; Qwen3 T=600 1035 -> 507 us, Qwen3-30B-A3B T=1000 1795 -> 841 us.
// Bound: the matrix cores at the clock the chip holds under them (without the
// loads and the splits the same loop takes 214 us for that fc1).
//
// Values the split cannot hold (infinities, NaN, magnitudes from 2^111) give a
// non-finite sum in every output they enter; such sums (and those from 2^96,
// which overflow scaled) are recomputed with plain f32 FMAs from the operands in
// memory, so non-finite inputs give what the vector kernel gave; rows with a NaN
// need only be found (redo_non_finite). A sixteenth of the rows clean / NaN / all
// infinite: Nomic T=64 47 / 75 / 87 us, T=4096 531 / 584 / 683, Qwen3 T=600 506 /
// 586 / 909 (the vector kernel 98 / 1198 / 1022, whatever the values).
//
// moe_f32_gemm<BM, MODE>: BM x 128 block tile, 256 threads, v_mfma 32x32x16.
//  BM = 128: 2 x 2 waves of 64 x 64, K in steps of 32;
//  BM = 32 (few rows per expert): 4 waves side by side, K in steps of 64.
// For the gate/up GEMM the 128-column weight panel is 64 gate columns then
// the same 64 up columns; a wave's columns are matching gate and up columns
// (64 output columns per workgroup).
// Per K step: global -> registers (16-byte loads, one step ahead), split and
// store the bf16 parts to LDS (three planes per operand), barrier, MFMAs,
// barrier. Two (or more) workgroups share a CU, so one's loads and splits run
// under another's MFMAs: 6 MFMAs per f32 product block against 5.5 vector
// instructions per element split (each element of a 128 x 128 tile feeds 128
// products), i.e. about half as many vector as matrix cycles.
// LDS layout: 16-byte chunks of 8 consecutive k; chunk c of row (or column) r
// at [c][slot(r, c)], slot = r with its low 3 bits xored by (r / 8) and c, so
// that the 8-lane groups of every 16-byte LDS access land in 8 distinct
// bank groups: fragment reads (32 consecutive rows of one chunk), A and
// [N,K] stores (a row's chunks side by side) and [K,N] stores (a thread
// holds 8 k-rows x 4 columns, which the pairwise conversion transposes for
// free: it packs two k of one column).
//  * A rows are gathered (gate/up, fc1: the pair's token row) or sorted rows
//    (down, fc2: the intermediate in pair order).
//  * Few tiles: K is split over up to 16 workgroups per tile, which meet in
//    the ordered fixup (splitk_fixup), so results stay deterministic.
//  * Epilogues as the other kernels: act(gate) * up or act(x) into the
//    intermediate; w * acc added with one f32 atomic per element and pair
//    into the accumulator (down, fc2).
// Requires K % 4 == 0, N % 4 == 0 and 16-byte aligned operands (checked on
// the host; other shapes take moe_simt_gemm).
#include "cm_lds.hpp"

namespace cm {

using namespace lds;

namespace {

template <int BM, int MODE>
__global__ __launch_bounds__(256, 2) void moe_f32_gemm(GemmArgs a) {
    constexpr int BN = 128;
    constexpr int BK = f32_tile_k(BM);
    constexpr int NCH = BK / 8;  // 8-k chunks per step
    constexpr bool DUAL = (MODE == kGateUp);
    constexpr bool GATHER = (MODE == kGateUp || MODE == kFc1);
    constexpr bool BNK = (MODE == kFc2);
    constexpr bool ATOMIC = (MODE == kDown || MODE == kFc2);
    constexpr int BNO = DUAL ? BN / 2 : BN;  // output columns per workgroup
    constexpr int MB = BM == 128 ? 2 : 1, NB = BM == 128 ? 2 : 1;
    constexpr int A_CHUNKS = NCH * BM, B_CHUNKS = NCH * BN;
    // staging: BM = 128 gives the weights to threads 0..127 and A to the
    // others (32 values each); BM = 32 gives every thread 32 weights and 8 of A
    constexpr bool HALVES = BM == 128;
    constexpr int ST = HALVES ? 128 : 256;       // threads per operand
    constexpr int A_PER = A_CHUNKS / ST;         // A chunks per thread
    constexpr int BQ_PER = B_CHUNKS / 4 / ST;    // [K,N]: 8 k x 4 columns per thread
    constexpr int BC_PER = B_CHUNKS / ST;        // [N,K]: chunks per thread
    static_assert(A_PER * ST == A_CHUNKS && BQ_PER == 1 && BC_PER == 4 && A_PER <= 4, "f32 staging");
    __shared__ __attribute__((aligned(16))) u32x4 sA[3][A_CHUNKS];
    __shared__ __attribute__((aligned(16))) u32x4 sB[3][B_CHUNKS];
    __shared__ long long s_row[BM];
    __shared__ int32_t s_tok[ATOMIC ? BM : 1];
    __shared__ float s_w[ATOMIC ? BM : 1];

    clear_share(a.zero_f32, a.zero_n);
    const int live = *a.num_tiles * a.n_tiles;
    const int nsplit = adaptive_split(a.ksplit, a.split_target, live, (a.K + BK - 1) / BK);
    const int lg = xcd_logical(live * nsplit);
    if (lg < 0) return;
    const int tile = lg / nsplit, ks = lg - tile * nsplit;
    const int mt = tile / a.n_tiles, nt = tile - mt * a.n_tiles;
    const int r0 = a.tile_row[mt];
    const int e = a.tile_exp[mt];
    const int m_valid = min(BM, a.offsets[e + 1] - r0);
    const int K = a.K, N = a.N, n0 = nt * BNO;
    const int tid = threadIdx.x, lane = tid & 63, lr = lane & 31, lh = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = BM == 128 ? wave >> 1 : 0, wn = BM == 128 ? wave & 1 : wave;
    const float* A = reinterpret_cast<const float*>(a.A);
    const float* B0 = reinterpret_cast<const float*>(a.B0) + (long long)e * a.strideB;
    const float* B1 = DUAL ? reinterpret_cast<const float*>(a.B1) + (long long)e * a.strideB : B0;
    if (tid < BM) {
        // (rows past the group's end repeat its first row; never stored)
        const int r = r0 + (tid < m_valid ? tid : 0);
        const int p = a.sorted_pair[r];
        s_row[tid] = (long long)(GATHER ? p / a.k_top : r) * K;
        if constexpr (ATOMIC) {
            s_tok[tid] = p / a.k_top;
            s_w[tid] = a.routing_w[p];
        }
    }
    __syncthreads();

    // this split's K steps
    const int nk_all = (K + BK - 1) / BK;
    const int per_split = (nk_all + nsplit - 1) / nsplit;
    const int kc0 = min(nk_all, ks * per_split);
    const int nk = min(nk_all, kc0 + per_split) - kc0;

    auto slot = [](int r, int c) { return r ^ ((r >> 3) & 7) ^ (c * (8 / NCH)); };
    const bool do_b = !HALVES || tid < ST, do_a = !HALVES || tid >= ST;
    const int st = HALVES ? tid & (ST - 1) : tid;

    // global addresses of this thread's share of the K step at k = 0
    // (columns past N re-read the last ones; never stored)
    const float* pA[A_PER];
#pragma unroll
    for (int i = 0; i < A_PER; ++i) {
        const int it = st + ST * i;
        pA[i] = A + s_row[it / NCH] + 8 * (it % NCH);
    }
    const float* pB[BNK ? BC_PER : 1];
    const int bq = st & 31, bc = st >> 5;  // [K,N]: column quad and chunk
    if constexpr (BNK) {
#pragma unroll
        for (int i = 0; i < BC_PER; ++i) {
            const int it = st + ST * i;
            pB[i] = B0 + (long long)min(n0 + it / NCH, N - 1) * a.ldb + 8 * (it % NCH);
        }
    } else {
        const int col = min(n0 + 4 * (DUAL ? bq & 15 : bq), N - 4);
        pB[0] = (DUAL && bq >= 16 ? B1 : B0) + (long long)(8 * bc) * a.ldb + col;
    }

    f32x4 rb[8], ra[HALVES ? 1 : 2 * A_PER];
    f32x4* const va = HALVES ? rb : ra;  // (HALVES: a thread stages one operand only)
    auto fetch = [&](int kc) {
        const int k0 = kc * BK;
        const bool tail = k0 + BK > K;
        const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
        if (do_b) {
            if constexpr (BNK) {
#pragma unroll
                for (int i = 0; i < BC_PER; ++i) {
                    const int k = k0 + 8 * ((st + ST * i) % NCH);
                    const float* p = pB[i] + k0;
#pragma unroll
                    for (int h = 0; h < 2; ++h) {
                        if (!tail || k + 4 * h < K) rb[2 * i + h] = *reinterpret_cast<const f32x4*>(p + 4 * h);
                        else rb[2 * i + h] = zero;
                    }
                }
            } else {
                const float* p = pB[0] + (long long)k0 * a.ldb;
#pragma unroll
                for (int t = 0; t < 8; ++t) {
                    if (!tail || k0 + 8 * bc + t < K) rb[t] = *reinterpret_cast<const f32x4*>(p + (long long)t * a.ldb);
                    else rb[t] = zero;
                }
            }
        }
        if (do_a) {
#pragma unroll
            for (int i = 0; i < A_PER; ++i) {
                const int k = k0 + 8 * ((st + ST * i) % NCH);
                const float* p = pA[i] + k0;
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    if (!tail || k + 4 * h < K) va[2 * i + h] = *reinterpret_cast<const f32x4*>(p + 4 * h);
                    else va[2 * i + h] = zero;
                }
            }
        }
    };
    // split 8 values (consecutive k) into the three planes' chunk
    auto put = [&](auto& plane, int at, const float (&v)[8]) {
        u32x4 h, m, l;
        split8(v, h, m, l);
        plane[0][at] = h;
        plane[1][at] = m;
        plane[2][at] = l;
    };
    auto stash = [&]() {
        if (do_b) {
            if constexpr (BNK) {
#pragma unroll
                for (int i = 0; i < BC_PER; ++i) {
                    const int it = st + ST * i, r = it / NCH, c = it % NCH;
                    const f32x4 x = rb[2 * i], y = rb[2 * i + 1];
                    const float v[8] = {x[0], x[1], x[2], x[3], y[0], y[1], y[2], y[3]};
                    put(sB, c * BN + slot(r, c), v);
                }
            } else {
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    float v[8];
#pragma unroll
                    for (int t = 0; t < 8; ++t) v[t] = rb[t][j];
                    put(sB, bc * BN + slot(4 * bq + j, bc), v);
                }
            }
        }
        if (do_a) {
#pragma unroll
            for (int i = 0; i < A_PER; ++i) {
                const int it = st + ST * i, r = it / NCH, c = it % NCH;
                const f32x4 x = va[2 * i], y = va[2 * i + 1];
                const float v[8] = {x[0], x[1], x[2], x[3], y[0], y[1], y[2], y[3]};
                put(sA, c * BM + slot(r, c), v);
            }
        }
    };

    // panel column of this lane in column block nb: BM = 128: 32 columns of
    // the wave's 64 (gate/up: nb = 0 gate, 1 up of the same 32); BM = 32: 32
    // of the panel (gate/up: lanes 0..15 gate, 16..31 up of the same 16)
    auto panel_col = [&](int nb) {
        if constexpr (BM == 128) return DUAL ? nb * 64 + wn * 32 + lr : wn * 64 + nb * 32 + lr;
        else return DUAL ? (lr >> 4) * 64 + wn * 16 + (lr & 15) : wn * 32 + lr;
    };
    // h*h apart from the five small part products, whose sum (2^-8 of it) then
    // adds no roundings at the full sum's magnitude
    f32x16 acc[MB][NB], small[MB][NB];
#pragma unroll
    for (int i = 0; i < MB; ++i)
#pragma unroll
        for (int j = 0; j < NB; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[i][j][r] = small[i][j][r] = 0.f;
    // a wave whose rows all lie past the group's end only stages
    const bool rows_live = BM == 32 || wm * 64 < m_valid;

    if (nk > 0) fetch(kc0);
    for (int s = 0; s < nk; ++s) {
        stash();
        __syncthreads();
        if (s + 1 < nk) fetch(kc0 + s + 1);
        if (rows_live) {
#pragma unroll
            for (int kk = 0; kk < BK / 16; ++kk) {
                const int c = 2 * kk + lh;
                u32x4 af[3][MB], bf[3][NB];
#pragma unroll
                for (int pl = 0; pl < 3; ++pl) {
#pragma unroll
                    for (int i = 0; i < MB; ++i) af[pl][i] = sA[pl][c * BM + slot(wm * 64 + i * 32 + lr, c)];
#pragma unroll
                    for (int j = 0; j < NB; ++j) bf[pl][j] = sB[pl][c * BN + slot(panel_col(j), c)];
                }
                constexpr int PA[5] = {2, 0, 1, 1, 0}, PB[5] = {0, 2, 1, 0, 1};
#pragma unroll
                for (int q = 0; q < 5; ++q)
#pragma unroll
                    for (int i = 0; i < MB; ++i)
#pragma unroll
                        for (int j = 0; j < NB; ++j)
                            small[i][j] = mfma32<kBF16>(af[PA[q]][i], bf[PB[q]][j], small[i][j]);
#pragma unroll
                for (int i = 0; i < MB; ++i)
#pragma unroll
                    for (int j = 0; j < NB; ++j) acc[i][j] = mfma32<kBF16>(af[0][i], bf[0][j], acc[i][j]);
            }
        }
        __syncthreads();
    }

#pragma unroll
    for (int i = 0; i < MB; ++i)
#pragma unroll
        for (int j = 0; j < NB; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[i][j][r] = (acc[i][j][r] + small[i][j][r]) * kSplitUnscale;

    // Non-finite sums again with f32 FMAs (see the top). Register
    // i of lane l: row 8(i/4) + 4(l/32) + i%4 of the block, column l%32.
    auto row_of = [&](int mb, int i) { return wm * 64 + mb * 32 + 8 * (i >> 2) + 4 * lh + (i & 3); };
#pragma unroll
    for (int mb = 0; mb < MB; ++mb)
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) {
            bool bad = false;
#pragma unroll
            for (int i = 0; i < 16; ++i) bad |= !__builtin_isfinite(acc[mb][nb][i]);
            if (__builtin_expect(__any(bad), 0)) {
                const int pc = panel_col(nb);
                const int col = min(n0 + (DUAL ? pc & 63 : pc), N - 1);
                const float* b = ((DUAL && pc >= 64) ? B1 : B0) + (BNK ? (long long)col * a.ldb : col);
                const long long step = BNK ? 1 : a.ldb;
                redo_non_finite<16, 32>(
                    lane, kc0 * BK, min(K, (kc0 + nk) * BK),
                    [&](int q) {
                        float v = acc[mb][nb][0];
#pragma unroll
                        for (int i = 1; i < 16; ++i) v = q == i ? acc[mb][nb][i] : v;
                        return v;
                    },
                    [&](int q, float v) {
#pragma unroll
                        for (int i = 0; i < 16; ++i) acc[mb][nb][i] = q == i ? v : acc[mb][nb][i];
                    },
                    [&](int q, int k) { return *reinterpret_cast<const f32x4*>(A + s_row[row_of(mb, q)] + k); },
                    [&](int k) { return b[k * step]; });
            }
        }

    if (nsplit > 1 && !splitk_fixup<MB, NB, 4, 4, (BM == 32)>(a, acc, tile * nsplit, tile, ks, nsplit, wave, lane))
        return;

#pragma unroll
    for (int mb = 0; mb < MB; ++mb) {
        if constexpr (DUAL) {
            float* C = reinterpret_cast<float*>(a.C) + (long long)r0 * N;
#pragma unroll
            for (int i = 0; i < 16; ++i) {
                const int m = row_of(mb, i);
                if constexpr (BM == 128) {
                    const int col = n0 + wn * 32 + lr;
                    if (m < m_valid && col < N)
                        C[(long long)m * N + col] = act_f32(acc[mb][0][i], a.act) * acc[mb][NB - 1][i];
                } else {
                    // the up value sits 16 lanes on
                    const int col = n0 + wn * 16 + (lr & 15);
                    const float up = xor_lane<16>(acc[mb][0][i]);
                    if (lr < 16 && m < m_valid && col < N) C[(long long)m * N + col] = act_f32(acc[mb][0][i], a.act) * up;
                }
            }
        } else {
#pragma unroll
            for (int nb = 0; nb < NB; ++nb) {
                const int col = n0 + panel_col(nb);
#pragma unroll
                for (int i = 0; i < 16; ++i) {
                    const int m = row_of(mb, i);
                    if (m >= m_valid || col >= N) continue;
                    if constexpr (!ATOMIC) {
                        reinterpret_cast<float*>(a.C)[(long long)(r0 + m) * N + col] = act_f32(acc[mb][nb][i], a.act);
                    } else {
                        unsafeAtomicAdd(reinterpret_cast<float*>(a.C) + (long long)s_tok[m] * N + col,
                                        s_w[m] * acc[mb][nb][i]);
                    }
                }
            }
        }
    }
}

}  // namespace

template <int MODE>
static hipError_t launch_f32_mode(int cfg, const GemmArgs& a, hipStream_t stream) {
    const long long nwg_l = split_grid((long long)a.m_tiles_max * a.n_tiles, a);
    if (nwg_l > 0x7fffffffLL) return hipErrorInvalidValue;
    const int nwg = (int)nwg_l;
    if (nwg <= 0) return hipSuccess;
    if (cfg == kF32Rows32)
        hipLaunchKernelGGL((moe_f32_gemm<32, MODE>), dim3(nwg), dim3(256), 0, stream, a);
    else
        hipLaunchKernelGGL((moe_f32_gemm<128, MODE>), dim3(nwg), dim3(256), 0, stream, a);
    return hipGetLastError();
}

hipError_t launch_moe_gemm_f32(int mode, int cfg, const GemmArgs& a, hipStream_t stream) {
    switch (mode) {
        case kGateUp: return launch_f32_mode<kGateUp>(cfg, a, stream);
        case kFc1: return launch_f32_mode<kFc1>(cfg, a, stream);
        case kDown: return launch_f32_mode<kDown>(cfg, a, stream);
        case kFc2: return launch_f32_mode<kFc2>(cfg, a, stream);
        default: return hipErrorInvalidValue;  // the expert-set path is MFMA-only
    }
}

}  // namespace cm
