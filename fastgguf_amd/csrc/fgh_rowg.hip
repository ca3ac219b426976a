// fgh_rowg.hip - Q4_K and Q5_K matrices times 2..64 tokens in the decode kernels' own fp32 orders
// (fgh_q4k.hip), on f16 MFMA: the matmuls that the reference runs token by token (matmul,
// fastgguf.c:3004-3017: every batch below 8 tokens, and Q5_K at every batch, which has no prompt
// GEMM there). Outputs equal the per-token decode kernel's bit for bit.
//
// Per (row, token, block) the orders need integers (dot_q4_K_q8k 1118-1153, dot_q5_K_q8k
// 1178-1230, dot_q4Kx8 2322-2358):
//   row order   eight lane partials  u_k = sum_g sc_g sum_{j < 4} q[32 g + 4 k + j] y[..]  and
//               four min partials    m_2p bs_2p + m_2p+1 bs_2p+1
//   repacked    their sums over k and p
// One lane partial is a sum over 8 sub-blocks x 4 positions: exactly the K = 32 of
// v_mfma_f32_16x16x32_f16. Lane (kg, .) of an operand holds the 4 positions of sub-blocks 2 kg and
// 2 kg + 1, A = 16 tokens' activations, B = 16 rows' weights times their 6-bit scales. A weight
// times its scale (31 * 63 = 1953) and an activation (127) are exact in f16, and every sum an
// integer below 2^23 (8 * 4 * 1953 * 127), so D is the partial as a float, with no conversion. (On
// int8 MFMA a scaled weight needs two or three operands, a recombination and a conversion per
// partial.) Repacked: lane groups 0..3 and 4..7 accumulate apart, each below 2^24 (15.4 M), and one
// add rounds their sum as the reference's conversion does. The mins: 32-value sums split 64 bh + bl
// against (64 m, m) in 16x16x16 MFMAs, one per min lane with the other lanes' weights zero.
// The fp32 chains of a (token, row) then run in block order in one lane: lane (q, n) holds tokens
// 4 q .. 4 q + 3 of row n.
//
// A launch of gemm-like shape: workgroup = 4 wavefronts of one 16-row tile each (no split of a row:
// its chains run over all blocks), NG groups of 16 tokens per wavefront; the activation records
// (8.6 KB per block and group, written by rowg_quant_kernel in fragment order) go through two LDS
// stages, requested D blocks ahead in registers; each wavefront keeps a ring of R blocks of its
// weights. The block loop is straight-line code (loads past the end repeat the last block), so
// its waits are exact counts.
// NG = 2 where that still gives most compute units a workgroup, since a block's weights are unpacked
// once per wavefront (about 130 VALU instructions, Q5_K 230, against 56 per group); with 4 groups
// the 192 chain registers would lie in accumulation registers, two moves for every fma (measured:
// 49.7 us).
// Bound (counters): two groups, Q5_K 14336 x 4096, 64 tokens (31 us after a quantizer launch of 4): VALU
// issue, 42.7 k of the 63.5 k cycles that a SIMD is busy (matrix pipe 10.8 k). One group, Q4_K, 5 tokens (12 us
// after a launch of 3.5): the latency of a block's steps in the one wavefront of a SIMD, which issues for half
// of its life, waits a third of it for results of MFMAs and fmas and a sixth for memory.
#include "fgh_internal.h"

namespace fgh {

namespace {

typedef _Float16 h2 __attribute__((ext_vector_type(2)));
typedef _Float16 h4 __attribute__((ext_vector_type(4)));
typedef _Float16 h8 __attribute__((ext_vector_type(8)));
typedef float f4 __attribute__((ext_vector_type(4)));
typedef uint32_t u4 __attribute__((ext_vector_type(4)));

// The activation records of block b of 16 tokens (group t: records t nb + b of both arrays):
//   fragments, 8192 B   A fragments of lane group k at 1024 k: lane (kg, token) its 8 values,
//                       sub-blocks 2 kg (lo) and 2 kg + 1 (hi) at positions 4 k + j:
//                       lo0 lo2 hi0 hi2 lo1 lo3 hi1 hi3
//   then, after all fragments, 576 B: [0, 512) min fragments, lane (kg, token) bh, bl of sub-block
//                       2 kg, then of 2 kg + 1; [512, 576) yd of the 16 tokens
constexpr int RG_FRAG = 8192, RG_SMALL = 576, RG_YD = 512;

// Q8_K quantization of the tokens (quantize_q8k, fastgguf.c:773-793, as q8k_store_b) into records:
// grid (blocks, groups of 16 tokens), 16 threads per token. Tokens past T are zeros.
__global__ __launch_bounds__(256) void rowg_quant_kernel(const float *__restrict__ X, int64_t ldx, int nb, int T,
                                                         uint8_t *__restrict__ act) {
    const int b = blockIdx.x, tl = threadIdx.x & 15, m = threadIdx.x >> 4, tok = (int)blockIdx.y * 16 + m;
    const size_t ri = (size_t)blockIdx.y * nb + b;
    uint8_t *rec = act + ri * RG_FRAG, *sm = act + (size_t)gridDim.y * nb * RG_FRAG + ri * RG_SMALL;
    float v[16];
    if (tok < T) {
        XRound xr;
        q8k_load_b(X + (size_t)tok * ldx, b, true, xr);
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            v[4 * u] = xr.v[u].x; v[4 * u + 1] = xr.v[u].y; v[4 * u + 2] = xr.v[u].z; v[4 * u + 3] = xr.v[u].w;
        }
    } else {
#pragma unroll
        for (int u = 0; u < 16; ++u) v[u] = 0.0f;
    }
    float amax = 0.0f;
#pragma unroll
    for (int u = 0; u < 16; ++u) amax = fmaxf(amax, fabsf(v[u]));
    amax = fmaxf(amax, dpp_ror_f32(amax, 8));
    amax = fmaxf(amax, dpp_ror_f32(amax, 4));
    amax = fmaxf(amax, dpp_ror_f32(amax, 2));
    amax = fmaxf(amax, dpp_ror_f32(amax, 1));
    const float d = amax / 127.0f;
    const float id = d > 0.0f ? 1.0f / d : 0.0f;
    // values 16 tl .. + 15: sub-block tl / 2, lane groups 4 (tl & 1) + u, positions 4 (..) + j
    const int kg = tl >> 2, i = (tl >> 1) & 1;
    int s = 0;
#pragma unroll
    for (int u = 0; u < 4; ++u) {
        int q[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            q[j] = (int)(int8_t)q8_round(v[4 * u + j] * id);
            s += q[j];
        }
        uint8_t *f = rec + 1024 * (4 * (tl & 1) + u) + 16 * (16 * kg + m) + 4 * i;
        *(h2 *)f = (h2){(_Float16)q[0], (_Float16)q[2]};
        *(h2 *)(f + 8) = (h2){(_Float16)q[1], (_Float16)q[3]};
    }
    s += dpp_xor1(s);  // threads 2 g, 2 g + 1: the 32 values of sub-block g
    if ((tl & 1) == 0) *(h2 *)(sm + 8 * (16 * kg + m) + 4 * i) = (h2){(_Float16)(s >> 6), (_Float16)(s & 63)};
    if (tl == 0) ((float *)(sm + RG_YD))[m] = d;
}

// one lane's weights of one block: pieces 0 and 1 of chunk kg of its row (the layout's swap undone
// in the addresses), its row's meta and, Q5_K only, the fifth bits of its chunk
struct RgW {
    uint4 p0, p1, m;
    uint2 h;
};
template <int TYPE, int AUX>
__device__ __forceinline__ void rg_load(const uint8_t *blk, uint32_t o0, uint32_t o1, uint32_t L, bool live, RgW &w) {
    const BufRes r = buf_res(blk, live ? (TYPE == T_Q5_K ? Q5K_TILE : Q4K_TILE) : 0);
    w.p0 = bld16<AUX>(r, o0);
    w.p1 = bld16<AUX>(r, o1);
    w.m = bld16<AUX>(r, 16 * (L >> 2));
    if (TYPE == T_Q5_K) w.h = bld8<AUX>(r, 2304 + 8 * L);
}
__device__ __forceinline__ h2 as_h2(uint32_t v) { return __builtin_bit_cast(h2, v); }
// bits (t, t + 16) of w moved to bits (4, 20): fifth bits of a pair of values
template <int T>
__device__ __forceinline__ uint32_t fifth2(uint32_t w) {
    return T <= 4 ? w << (4 - (T <= 4 ? T : 4)) : w >> ((T > 4 ? T : 4) - 4);
}
// register k of an operand: lane group k's 4 low and 4 high values of the chunk, times their scales.
// M, F, E: 0x000f000f, 0x00100010 and 0x64006400 in registers (a value or-ed with E is 1024 + value, exact in f16;
// with literals the compiler takes two instructions for one v_and_or_b32)
template <int TYPE, int D>  // D: the register's index in the layout's fifth-bit words
__device__ __forceinline__ h8 rg_operand(uint32_t q, uint32_t M, uint32_t F, uint32_t E, uint32_t fl, uint32_t fh, h2 sl, h2 ol, h2 sh,
                                         h2 oh) {
    uint32_t l02 = (q & M) | E, h02 = ((q >> 4) & M) | E, l13 = ((q >> 8) & M) | E, h13 = ((q >> 12) & M) | E;
    if (TYPE == T_Q5_K) {
        l02 = (fifth2<D>(fl) & F) | l02;
        l13 = (fifth2<D + 8>(fl) & F) | l13;
        h02 = (fifth2<D>(fh) & F) | h02;
        h13 = (fifth2<D + 8>(fh) & F) | h13;
    }
    const h2 a = __builtin_elementwise_fma(as_h2(l02), sl, ol), b = __builtin_elementwise_fma(as_h2(h02), sh, oh);
    const h2 c = __builtin_elementwise_fma(as_h2(l13), sl, ol), e = __builtin_elementwise_fma(as_h2(h13), sh, oh);
    return (h8){a.x, a.y, b.x, b.y, c.x, c.y, e.x, e.y};
}

struct RgArgs {
    const uint8_t *W;
    float *Y;
    const uint8_t *act;
    int64_t rows, gpm, groups, ldy;
    int nb, T, tg;  // tg: groups of 16 tokens
};

template <int ORDER, int TYPE, int NG, int R, int D, int AUX>
__global__ __launch_bounds__(256, 2) void rowg_kernel(RgArgs a) {
    constexpr int STAGE = NG * RG_FRAG + 4096;  // fragments, then 256 pieces of which NG * 36 are the small records
    constexpr int NA = ORDER == 1 ? 1 : 8, NM = ORDER == 1 ? 1 : 4;
    constexpr int NS = NG == 1 ? 3 : 2;  // LDS stages: with 3 a block's fragments are read during the block before it
    static_assert(R % 2 == 0 && R % D == 0, "the stages rotate within a ring round");
    extern __shared__ __align__(16) uint8_t smem[];
    const int tid = threadIdx.x, l = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int nb = a.nb, tg0 = (int)blockIdx.y * NG;
    const int64_t tile = (int64_t)blockIdx.x * 4 + wave;
    const bool live = tile < a.groups;
    const uint32_t tc = (uint32_t)(live ? tile : a.groups - 1), gpm = (uint32_t)a.gpm;
    const uint32_t mi = (uint32_t)__builtin_amdgcn_readfirstlane((int)(tc / gpm)), lt = tc - mi * gpm;
    constexpr int TB = TYPE == T_Q5_K ? Q5K_TILE : Q4K_TILE;
    const uint8_t *W0 = a.W + ((size_t)mi * nb * gpm + lt) * TB;
    const size_t bstride = (size_t)gpm * TB;
    const int kg = l >> 4, n = l & 15;
    const uint32_t L = 4 * n + kg;
    const uint32_t o0 = (kg >= 2 ? 1280u : 256u) + 16 * L, o1 = (kg >= 2 ? 256u : 1280u) + 16 * L;

    // (1) the ring's first blocks, then the records of blocks 0 .. D
    RgW ring[R];
#pragma unroll
    for (int r = 0; r < R; ++r) rg_load<TYPE, AUX>(W0 + (size_t)min(r, nb - 1) * bstride, o0, o1, L, live && r < nb, ring[r]);
    struct Rec {
        uint4 f[2 * NG], s;
    } st[D];
    // this thread's piece of the small records: piece tid % 36 of group tid / 36 (past the last group:
    // a piece that is not read back); a group past the last token group repeats it
    const uint8_t *small = a.act + (size_t)a.tg * nb * RG_FRAG +
                           (tid < 36 * NG ? (uint32_t)min(tg0 + tid / 36, a.tg - 1) * (uint32_t)(nb * RG_SMALL) + 16 * (tid % 36) : 0u);
    int first[NG];  // the records of block 0 of each group
#pragma unroll
    for (int g = 0; g < NG; ++g) first[g] = __builtin_amdgcn_readfirstlane(min(tg0 + g, a.tg - 1) * nb);
    auto rec_load = [&](int b, Rec &r) {
#pragma unroll
        for (int g = 0; g < NG; ++g) {
            const BufRes fr = buf_res(a.act + (size_t)(uint32_t)(first[g] + b) * RG_FRAG, RG_FRAG);
            r.f[2 * g] = bld16(fr, 16 * tid);
            r.f[2 * g + 1] = bld16(fr, 4096 + 16 * tid);
        }
        r.s = *(const uint4 *)(small + (uint32_t)(b * RG_SMALL));
    };
    auto rec_store = [&](int b, const Rec &r) {
        uint8_t *dst = smem + (b % NS) * STAGE + 16 * tid;
#pragma unroll
        for (int g = 0; g < NG; ++g) {
            *(uint4 *)(dst + g * RG_FRAG) = r.f[2 * g];
            *(uint4 *)(dst + g * RG_FRAG + 4096) = r.f[2 * g + 1];
        }
        *(uint4 *)(dst + NG * RG_FRAG) = r.s;
    };
    // blocks 0 .. NS - 2 into their stages, D blocks from there requested
    rec_load(0, st[0]);
#pragma unroll
    for (int i = 1; i < D; ++i) rec_load(min(i, nb - 1), st[i]);
#pragma unroll
    for (int i = 0; i < NS - 1; ++i) {
        rec_store(i, st[i % D]);
        rec_load(min(i + D, nb - 1), st[i % D]);
    }
    __syncthreads();

    f4 acc[NG][NA], macc[NG][NM];
#pragma unroll
    for (int g = 0; g < NG; ++g) {
#pragma unroll
        for (int k = 0; k < NA; ++k) acc[g][k] = (f4){0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int p = 0; p < NM; ++p) macc[g][p] = (f4){0.0f, 0.0f, 0.0f, 0.0f};
    }
    const f4 Z = {0.0f, 0.0f, 0.0f, 0.0f};
    const int shs = 16 * (kg & 1);
    const uint32_t hm = kg >= 2 ? 0xFFFFFFFFu : 0u;
    uint32_t M = 0x000f000fu, F = 0x00100010u, E = 0x64006400u;
    asm("" : "+s"(M));
    asm("" : "+s"(F));
    asm("" : "+v"(E));
    struct Frags {  // NG == 1: a block's fragments, min fragments and yd
        h8 a[8];
        h4 m;
        f4 yd;
    } fr[NG == 1 ? 2 : 1];
    auto frag_read = [&](int b, Frags &f) {
        const uint8_t *S = smem + (b % NS) * STAGE, *Sm = S + NG * RG_FRAG;
#pragma unroll
        for (int k = 0; k < 8; ++k) f.a[k] = *(const h8 *)(S + 1024 * k + 16 * l);
        f.m = *(const h4 *)(Sm + 8 * l);
        f.yd = *(const f4 *)(Sm + RG_YD + 16 * kg);
    };
    auto blk = [&](const RgW &w, int b, const Frags &f) {
        const uint8_t *S = smem + (b % NS) * STAGE, *Sm = S + NG * RG_FRAG;
        // scales and mins of sub-blocks 2 kg, 2 kg + 1 (scale_min_k4, fastgguf.c:466-472): both forms,
        // the lane's one selected bitwise; as f16 by 1024 + v - 1024
        const uint32_t A = w.m.y >> shs, B = w.m.z >> shs, C = w.m.w >> shs;
        const uint32_t scp = (((C & 0x0f0fu) | ((A >> 2) & 0x3030u)) & hm) | (A & 0x3f3fu & ~hm);
        const uint32_t mnp = ((((C >> 4) & 0x0f0fu) | ((B >> 2) & 0x3030u)) & hm) | (B & 0x3f3fu & ~hm);
        const h2 k1024 = {(_Float16)1024.0f, (_Float16)1024.0f};
        const h2 sc = as_h2(__builtin_amdgcn_perm(0u, scp, 0x0C010C00u) | E) - k1024;  // (sc_2kg, sc_2kg+1)
        const h2 mn = as_h2(__builtin_amdgcn_perm(0u, mnp, 0x0C010C00u) | E) - k1024;
        const h2 so = sc * -k1024, m64 = mn * (_Float16)64.0f;
        const h2 sl = {sc.x, sc.x}, sh = {sc.y, sc.y}, ol = {so.x, so.x}, oh = {so.y, so.y};
        const h4 MB = {m64.x, mn.x, m64.y, mn.y};
        const float d = fp16_bits_to_f32(w.m.x & 0xFFFF), dmin = fp16_bits_to_f32(w.m.x >> 16);
        uint32_t fl = 0, fh = 0;
        if (TYPE == T_Q5_K) {  // lanes kg >= 2 hold their chunk's halves swapped: so are their bit indices
            fl = ((((w.h.x >> 4) & 0x0f0f0f0fu) | ((w.h.x & 0x0f0f0f0fu) << 4)) & hm) | (w.h.x & ~hm);
            fh = ((((w.h.y >> 4) & 0x0f0f0f0fu) | ((w.h.y & 0x0f0f0f0fu) << 4)) & hm) | (w.h.y & ~hm);
        }
        const uint32_t q[8] = {w.p0.x, w.p0.y, w.p0.z, w.p0.w, w.p1.x, w.p1.y, w.p1.z, w.p1.w};
        f4 fd[NG], fm[NG];
        auto scales = [&]() {
#pragma unroll
            for (int g = 0; g < NG; ++g) {
                const f4 yd = NG == 1 ? f.yd : *(const f4 *)(Sm + g * RG_SMALL + RG_YD + 16 * kg);  // tokens 4 (l / 16) .. + 3
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    fd[g][r] = d * yd[r];
                    fm[g][r] = dmin * yd[r];
                }
            }
        };
        auto frag = [&](int g, int k) { return *(const h8 *)(S + g * RG_FRAG + 1024 * k + 16 * l); };
        f4 half[NG][2];  // repacked: the halves of sumi
        auto add = [&](auto kk, int g, const h8 &A, const h8 &Bk) {
            constexpr int k = decltype(kk)::value;
            if constexpr (ORDER == 1) {
                half[g][k / 4] = __builtin_amdgcn_mfma_f32_16x16x32_f16(A, Bk, k % 4 ? half[g][k / 4] : Z, 0, 0, 0);
            } else {
                const f4 u = __builtin_amdgcn_mfma_f32_16x16x32_f16(A, Bk, Z, 0, 0, 0);
#pragma unroll
                for (int r = 0; r < 4; ++r) acc[g][k][r] = __builtin_fmaf(fd[g][r], u[r], acc[g][k][r]);
            }
        };
        if constexpr (NG == 1) {
            scales();
            for_seq([&](auto kk) {
                constexpr int k = decltype(kk)::value;
                add(kk, 0, f.a[k], rg_operand<TYPE, k>(q[k], M, F, E, fl, fh, sl, ol, sh, oh));
            }, std::make_integer_sequence<int, 8>{});
        } else {
            scales();
            for_seq([&](auto kk) {
                constexpr int k = decltype(kk)::value;
                const h8 Bk = rg_operand<TYPE, k>(q[k], M, F, E, fl, fh, sl, ol, sh, oh);
#pragma unroll
                for (int g = 0; g < NG; ++g) add(kk, g, frag(g, k), Bk);
            }, std::make_integer_sequence<int, 8>{});
        }
#pragma unroll
        for (int g = 0; g < NG; ++g) {
            const h4 MA = NG == 1 ? f.m : *(const h4 *)(Sm + g * RG_SMALL + 8 * l), hz = {0, 0, 0, 0};
            if constexpr (ORDER == 1) {
                const f4 mt = __builtin_amdgcn_mfma_f32_16x16x16f16(MA, MB, Z, 0, 0, 0);
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    acc[g][0][r] = __builtin_fmaf(fd[g][r], half[g][0][r] + half[g][1][r], acc[g][0][r]);
                    macc[g][0][r] = __builtin_fmaf(fm[g][r], mt[r], macc[g][0][r]);
                }
            } else {
#pragma unroll
                for (int p = 0; p < 4; ++p) {  // min lane p alone: the other lanes' weights zero
                    const f4 mt = __builtin_amdgcn_mfma_f32_16x16x16f16(MA, kg == p ? MB : hz, Z, 0, 0, 0);
#pragma unroll
                    for (int r = 0; r < 4; ++r) macc[g][p][r] = __builtin_fmaf(fm[g][r], mt[r], macc[g][p][r]);
                }
            }
        }
        // the sums end here: the compiler would gather the fmas of a whole ring round at its end, and
        // spill what they wait for
#pragma unroll
        for (int g = 0; g < NG; ++g) {
#pragma unroll
            for (int k = 0; k < NA; ++k) asm volatile("" : "+v"(acc[g][k]));
#pragma unroll
            for (int p = 0; p < NM; ++p) asm volatile("" : "+v"(macc[g][p]));
        }
    };
    // block b; the records of block b + NS - 1 into their stage, those of block b + NS - 1 + D and the
    // weights of block b + R requested
    auto step = [&](int b, RgW &w, Rec &r, const Frags &f, Frags &next) {
        rec_store(b + NS - 1, r);
        rec_load(min(b + NS - 1 + D, nb - 1), r);
        if constexpr (NG == 1) frag_read(b + 1, next);
        __builtin_amdgcn_sched_barrier(0);
        blk(w, b, f);
        rg_load<TYPE, AUX>(W0 + (size_t)min(b + R, nb - 1) * bstride, o0, o1, L, live && b + R < nb, w);
        lds_barrier();
        __builtin_amdgcn_sched_barrier(0);
    };
    if constexpr (NG == 1) frag_read(0, fr[0]);
    constexpr int NF = NG == 1 ? 2 : 1;
    int b0 = 0;
    for (; b0 + R <= nb; b0 += R) {
#pragma unroll
        for (int r = 0; r < R; ++r) step(b0 + r, ring[r], st[(r + NS - 1) % D], fr[r % NF], fr[(r + 1) % NF]);
    }
#pragma unroll
    for (int r = 0; r < R - 1; ++r)
        if (b0 + r < nb) step(b0 + r, ring[r], st[(r + NS - 1) % D], fr[r % NF], fr[(r + 1) % NF]);  // uniform
    const int64_t row = (int64_t)lt * 16 + n;
    if (!live || row >= a.rows) return;
#pragma unroll
    for (int g = 0; g < NG; ++g)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int tok = 16 * (tg0 + g) + 4 * kg + r;
            float y;
            if constexpr (ORDER == 1) {
                y = acc[g][0][r] - macc[g][0][r];
            } else {  // hsum8(acc) - hsum4(macc), fastgguf.c:797-806 and 1089-1095
                const float h8s = ((acc[g][0][r] + acc[g][4][r]) + (acc[g][1][r] + acc[g][5][r])) +
                                  ((acc[g][2][r] + acc[g][6][r]) + (acc[g][3][r] + acc[g][7][r]));
                y = h8s - ((macc[g][0][r] + macc[g][1][r]) + (macc[g][2][r] + macc[g][3][r]));
            }
            if (tok < a.T) a.Y[(size_t)tok * a.ldy + (int64_t)mi * a.rows + row] = y;
        }
}

template <int ORDER, int TYPE, int NG, int R, int D, int AUX>
hipError_t rg_launch(const RgArgs &a, hipStream_t s) {
    const dim3 grid((unsigned)((a.groups + 3) / 4), (unsigned)((a.tg + NG - 1) / NG));
    rowg_kernel<ORDER, TYPE, NG, R, D, AUX><<<grid, 256, (NG == 1 ? 3 : 2) * (NG * RG_FRAG + 4096), s>>>(a);
    return hipGetLastError();
}
template <int ORDER, int TYPE>
hipError_t rg_launch_type(const RgArgs &a, int num_cu, hipStream_t s) {
    const int64_t wg = (a.groups + 3) / 4;
    if (a.tg == 1) return rg_launch<ORDER, TYPE, 1, ORDER == 1 ? 6 : 4, 2, WNT>(a, s);  // the weights are read once
    if constexpr (TYPE == T_Q5_K) {
        if (wg * ((a.tg + 1) / 2) >= num_cu * 3 / 4) return rg_launch<ORDER, TYPE, 2, 4, 1, 0>(a, s);
        return rg_launch<ORDER, TYPE, 1, 4, 2, 0>(a, s);
    }
    return hipErrorInvalidValue;  // Q4_K: from 8 tokens the prompt GEMM
}

}  // namespace

size_t rowg_act_bytes(int nb, int T) { return (size_t)((T + 15) / 16) * nb * (RG_FRAG + RG_SMALL); }

// Whether these kernels take less time than the per-token decode launches: both sides from what they
// measured on MI355X (us; 1740 calls: 62 shapes from 512 x 2048 to 3584 x 18944 and 60851 x 256, 2..7
// tokens, Q5_K 2..64). The decode launches walk a row's blocks in rounds of one wavefront per SIMD (a
// tile and token each; shorter launches split their tiles and are never slower), more slowly where an XCD's
// L2 doesn't hold its share of the matrix for the next token. These walk all blocks of a row in one
// wavefront, up to two per SIMD.
//                                   decode -> these     rule        decode -> these     rule
//   Q4_K repacked  14336 x 4096   4 16.7   16.6  decode   5 20.0   16.4  these
//   Q4_K row order 14336 x 4096   4 18.7   19.4  decode   5 21.5   19.2  these
//   Q4_K repacked   8192 x 8192   6 20.7   24.1  decode   7 25.3   24.2  these
//   Q5_K           14336 x 4096   4 20.8   23.6  decode   5 24.4   23.5  these
//   Q5_K           12464 x 5888   3 28.1   30.2  decode   5 41.2   29.9  these
//   Q5_K            4096 x 14336 12 46.9   62.1  decode  17 71.7   60.4  these
//   Q5_K            1024 x 4096  64 18.9   22.0  decode
//   Q5_K           14336 x 4096                          64 263.2  36.3  these
// In one of those calls it picks these kernels where they are 4 % slower, in none more; in 10 it keeps decode
// launches that are 8 to 18 % slower.
bool rowg_pays(int type, int order, int64_t groups, int nb, int T, int num_cu) {
    struct Fit {
        double base, block, round_block, round, far, one, one2;
    };
    const Fit f = type == T_Q5_K ? Fit{2.4, 0.051, 0.216, 0.462, 1.373, 0.97, 1.6}
                  : order == 1   ? Fit{2.265, 0.079, 0.175, 0.262, 1.185, 0.54, 1.07}
                                 : Fit{2.68, 0.229, 0.151, 0.32, 1.275, 0.72, 1.2};
    const int64_t simds = 4 * (int64_t)num_cu;
    const bool far = decode_l2_mib((double)groups * nb * (type == T_Q5_K ? Q5K_TILE : Q4K_TILE), (groups + 3) / 4) > 5.8;
    const double rounds = (double)((groups * T + simds - 1) / simds);
    const double before = f.base + f.block * nb + rounds * (f.round_block * (far ? f.far : 1.0) * nb + f.round);
    const int tg = (T + 15) / 16;
    const bool two = tg > 1 && (groups + 3) / 4 * ((tg + 1) / 2) >= num_cu * 3 / 4;
    const int64_t waves = groups * (two ? (tg + 1) / 2 : tg);
    const double one = two ? 1.17 : tg > 1 ? 0.95 : f.one;    // a block, at up to one wavefront per SIMD
    const double more = two ? 1.7 : tg > 1 ? 1.43 : f.one2;  // and at up to two, for each such round
    const double block = waves <= simds ? one : more * (double)((waves + 2 * simds - 1) / (2 * simds));
    return before > (two ? 8.0 : 6.6) + block * nb;
}

hipError_t launch_rowg(int type, int order, const RowgArgs &r, int num_cu, hipStream_t s) {
    if ((type != T_Q4_K && type != T_Q5_K) || r.nb < 1 || r.T < 1 || r.T > 64 || r.groups < 1 || r.gpm < 1 ||
        r.groups % r.gpm != 0 || r.gpm * 16 < r.rows || !r.W || !r.X || !r.Y || !r.act || (type == T_Q5_K && order != 0) ||
        (r.groups + 3) / 4 > 0x7fffffff)
        return hipErrorInvalidValue;
    const int tg = (r.T + 15) / 16;
    rowg_quant_kernel<<<dim3((unsigned)r.nb, (unsigned)tg), 256, 0, s>>>(r.X, r.ldx, r.nb, r.T, r.act);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    const RgArgs a{r.W, r.Y, r.act, r.rows, r.gpm, r.groups, r.ldy, r.nb, r.T, tg};
    if (type == T_Q5_K) return rg_launch_type<0, T_Q5_K>(a, num_cu, s);
    return order == 1 ? rg_launch_type<1, T_Q4_K>(a, num_cu, s) : rg_launch_type<0, T_Q4_K>(a, num_cu, s);
}

}  // namespace fgh
