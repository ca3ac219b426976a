// fgh_attn.hip - attention over an fp32 KV ring cache on gfx950, bit-exact with the reference's
// attn_rows (fastgguf.c:3273-3326): its vector path (hd % 32 == 0) and its per-row path (any
// other head size up to 256).
//
// Rows are (token, head) pairs: row i = t * n_head + h reads q / writes o at i * hd and the K / V
// head (h / G) * hd of each cache row (G = n_head / n_head_kv, the GQA grouping of the reference's
// forward, 4770-4790), over the positions st[t]..en[t] (slot p % cap). Three launches:
//   scores   8 chains per key: chain l runs fma over q[8m + l] k[8m + l] (att_qk_kern,
//            3227-3246), then hsum4_ps's tree ((a0+a1)+(a2+a3))+((a4+a5)+(a6+a7)) (3187-3190),
//            times scale; other head sizes dot_f32v's order (1618-1632): 8-lane chains s0 over
//            values 16 i + l and s1 over 16 i + 8 + l, one more group of 8 into s0, hsum_ps of
//            s0 + s1, then the last hd % 8 values one fma each, times scale (3313-3315)
//   softmax  one workgroup per row (softmax_vec, 3194-3219): the maximum, exp_neg_ps (3168-3184)
//            over whole groups of 8 and libm's expf over the tail, the sum as 8 ordered lane sums
//            (lane l over e[8g + l]) added in hsum_ps's tree then the tail in order, and every
//            value times 1 / sum
//   values   one lane per output element (att_v_kern, 3249-3270): acc = fma(w_p, v_p[c], acc)
//            over the positions in order
// The value sums are one dependent chain per (row, element) over every position: the
// reference's order, which no split over positions keeps. What bounds them is the latency of
// their operands, so the kernel keeps many tiles of V in flight per workgroup and runs the
// chains out of LDS. Head sizes up to 256; for hd % 32 == 0, kv_dim % 4 == 0 and 16-byte aligned
// pointers; other head sizes read K and (when a 16-byte read would not be aligned) V value by value.
#include <hip/hip_runtime.h>

#include "fgh_internal.h"

namespace fgh {

// exp_neg_ps (fastgguf.c:3168-3184) on one value: Cephes polynomial after x = max(x, -87),
// fx = floor(x log2(e) + 0.5), and 0 for x <= -87
__device__ __forceinline__ float exp_neg_ref(float x) {
    const bool keep = x > -87.0f;
    x = x > -87.0f ? x : -87.0f;
    const float fx = floorf(__builtin_fmaf(x, 1.44269504088896341f, 0.5f));
    x = __builtin_fmaf(-fx, 0.693359375f, x);
    x = __builtin_fmaf(-fx, -2.12194440e-4f, x);
    float y = 1.9875691500E-4f;
    y = __builtin_fmaf(y, x, 1.3981999507E-3f);
    y = __builtin_fmaf(y, x, 8.3334519073E-3f);
    y = __builtin_fmaf(y, x, 4.1665795894E-2f);
    y = __builtin_fmaf(y, x, 1.6666665459E-1f);
    y = __builtin_fmaf(y, x, 5.0000001201E-1f);
    const float xx = x * x, x1 = x + 1.0f;
    y = __builtin_fmaf(y, xx, x1);
    const float e = __builtin_bit_cast(float, (uint32_t)((int)fx + 127) << 23);
    return keep ? y * e : 0.0f;
}

// the rows' ranges: n = en - st + 1, or 0 when the range is empty, longer than the cache or than
// the score buffer (such a row gets NaN outputs)
__device__ __forceinline__ int row_len(const AttnArgs &a, int tok) {
    const int n = a.en[tok] - a.st[tok] + 1;
    return n >= 1 && n <= a.cap && n <= a.max_len ? n : 0;
}
__device__ __forceinline__ int64_t kv_slot(int p, int cap) { return (int64_t)(((p % cap) + cap) % cap); }

// A group is R rows that read the same K / V head kh: group q of head kh holds j = R q .. R q + R - 1
// of the head's n_tok * G rows, j = t * G + g (token t, query head kh * G + g). The scores and the
// value sums of a group run over the union lo..hi of its rows' ranges, as attn_rows runs its 4-row
// calls; a position outside a row's own range has weight 0, and fma(0, v, acc) = acc, so every
// row's sums are those of its own range.
struct GroupRow {
    int row, st, en;  // row = -1: no such row; en < st: no valid range
};
__device__ __forceinline__ GroupRow group_row(const AttnArgs &a, int n_tok, int R, int grp, int kh, int r) {
    const int G = a.n_head / a.n_head_kv, j = grp * R + r;
    GroupRow g{-1, 0, -1};
    if (j < n_tok * G) {
        const int t = j / G;
        g.row = t * a.n_head + kh * G + (j - t * G);
        if (row_len(a, t) > 0) {
            g.st = a.st[t];
            g.en = a.en[t];
        }
    }
    return g;
}
// A group's ranges, found by every wavefront for itself: lane r (mod R) reads row r's range, so the
// group costs one round of loads, and lane exchanges reduce them. R: 4, 16, 32 or 64.
struct GroupSpan {
    int lo, hi;        // the union of the rows' ranges; hi < lo: none is valid
    int in_lo, in_hi;  // the positions inside every valid row's range
    GroupRow mine;     // row lane % R
    GroupRow first;    // the first row with a valid range
    __device__ __forceinline__ bool any() const { return hi >= lo; }
    __device__ __forceinline__ GroupRow row(int r) const {  // r: any lane-dependent row
        return GroupRow{__shfl(mine.row, r, 64), __shfl(mine.st, r, 64), __shfl(mine.en, r, 64)};
    }
    __device__ __forceinline__ GroupRow urow(int r) const {  // r: uniform
        return GroupRow{__builtin_amdgcn_readlane(mine.row, r), __builtin_amdgcn_readlane(mine.st, r),
                        __builtin_amdgcn_readlane(mine.en, r)};
    }
};
__device__ __forceinline__ GroupSpan group_span(const AttnArgs &a, int n_tok, int R, int grp, int kh) {
    GroupSpan s;
    const int lane = threadIdx.x & 63, r = lane & (R - 1);
    s.mine = group_row(a, n_tok, R, grp, kh, r);
    const bool ok = s.mine.en >= s.mine.st;
    int lo = ok ? s.mine.st : 0x7fffffff, hi = ok ? s.mine.en : -0x7fffffff;
    int il = ok ? s.mine.st : -0x7fffffff, ih = ok ? s.mine.en : 0x7fffffff;
    for (int o = 1; o < R; o <<= 1) {
        lo = min(lo, __shfl_xor(lo, o, 64));
        hi = max(hi, __shfl_xor(hi, o, 64));
        il = max(il, __shfl_xor(il, o, 64));
        ih = min(ih, __shfl_xor(ih, o, 64));
    }
    s.lo = __builtin_amdgcn_readfirstlane(lo);
    s.hi = __builtin_amdgcn_readfirstlane(hi);
    s.in_lo = __builtin_amdgcn_readfirstlane(il);
    s.in_hi = __builtin_amdgcn_readfirstlane(ih);
    const uint64_t valid = __builtin_amdgcn_ballot_w64(ok);
    s.first = s.urow(valid ? __builtin_ctzll(valid) : 0);
    return s;
}

typedef float av4 __attribute__((ext_vector_type(4)));  // a native vector: kept in registers when staged
typedef float av4u __attribute__((ext_vector_type(4), aligned(4)));  // a 16-byte load at a 4-byte boundary

// ---- scores ----
// K = 1 MFMAs run the 8 lane chains: chain l of every (row, key) pair of a tile is one accumulator
// register set, and dimension d adds q_d k_d to chain d % 8, each as one fmaf, dimension after
// dimension (subnormals, infinities and NaN included; the tests compare bits, as for the values). K tiles
// of 64 keys go through LDS: 1 KB loads of whole rows in, one 16-byte read of 4 dimensions per key out.

// K rows of positions p0 .. p0 + 63 (past hi: hi's row) into dst[64][HD + 4], NT threads: pieces
// j B .. j B + B - 1 of each thread
template <int HD, int NT>
struct KTile {
    static constexpr int Q = HD / 4, N = 64 * Q / NT, B = N > 32 ? N / 2 : N;  // 16-byte pieces per row, per thread, at a time
    av4 v[B];
    __device__ __forceinline__ void load(const AttnArgs &a, int kh, int p0, int hi, int t, int j) {
        const float *kb = a.k + (int64_t)kh * HD;
        const int s0 = __builtin_amdgcn_readfirstlane((int)kv_slot(p0, a.cap));
        if (p0 + 63 <= hi && s0 + 64 <= a.cap) {  // uniform: no wrap, no clamp
#pragma unroll
            for (int i = 0; i < B; ++i) {
                const int e = t + (i + j * B) * NT;
                v[i] = *(const av4 *)(kb + (int64_t)(s0 + e / Q) * a.kv_dim + 4 * (e % Q));
            }
        } else {
#pragma unroll
            for (int i = 0; i < B; ++i) {
                const int e = t + (i + j * B) * NT;
                v[i] = *(const av4 *)(kb + kv_slot(min(p0 + e / Q, hi), a.cap) * a.kv_dim + 4 * (e % Q));
            }
        }
    }
    __device__ __forceinline__ void store(int t, int j, float *dst) const {
#pragma unroll
        for (int i = 0; i < B; ++i) {
            const int e = t + (i + j * B) * NT;
            *(av4 *)&dst[(e / Q) * (HD + 4) + 4 * (e % Q)] = v[i];
        }
    }
    __device__ __forceinline__ void copy(const AttnArgs &a, int kh, int p0, int hi, int t, float *dst) {
#pragma unroll
        for (int j = 0; j < N / B; ++j) {
            load(a, kh, p0, hi, t, j);
            store(t, j, dst);
        }
    }
};

// hsum4_ps's tree over the 8 chains
__device__ __forceinline__ float chain_tree(float a0, float a1, float a2, float a3, float a4, float a5, float a6, float a7) {
    return ((a0 + a1) + (a2 + a3)) + ((a4 + a5) + (a6 + a7));
}

// scores of 16 rows or more per K head: grid (K heads, groups of 16 NW rows, key chunks), NW
// wavefronts. Wavefront w multiplies rows 16 w .. + 15 of the group with a tile of 64 keys by
// v_mfma_f32_16x16x1: A = q (one register holds 4 dimensions x 16 rows; cbsz = 2 broadcasts the
// dimension's block to all four), B = K (lane = key), 8 chains x 16 registers of sums, in flight
// one after another. The next tile's loads are in flight
// in registers while a tile is multiplied (head sizes up to 128).
// 64 tokens x 32 heads over 8, 4096 positions, hd 128: 35 us. One 32-cycle MFMA per dimension and 16
// rows x 64 keys is about 15 of them (counters: the matrix pipe is busy 32.8 k cycles a SIMD); with two
// wavefronts a SIMD the rest is the range search, the q loads, the tiles' two barriers and the epilogue.
template <int HD, int NW>
__global__ __launch_bounds__(64 * NW, NW == 4 && HD <= 192 ? 2 : 1) void attn_scores16_kernel(AttnArgs a, int n_tok) {
    __shared__ __attribute__((aligned(16))) float kt[64 * (HD + 4)];
    typedef float av16 __attribute__((ext_vector_type(16)));
    const int kh = blockIdx.x, grp = blockIdx.y, tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const GroupSpan sp = group_span(a, n_tok, 16 * NW, grp, kh);
    if (!sp.any()) return;
    float q[HD / 4];
    {
        const GroupRow g = sp.row(16 * wave + (lane & 15));
        const float *qp = a.q + (int64_t)(g.en >= g.st ? g.row : sp.first.row) * HD + (lane >> 4);
#pragma unroll
        for (int i = 0; i < HD / 4; ++i) q[i] = qp[4 * i];
    }
    // the rows of this lane's sums: register 4 b + i = row 4 (lane / 16) + i, key 16 b + lane % 16
    float *out[4];
    int st[4], en[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const GroupRow g = sp.row(16 * wave + 4 * (lane >> 4) + i);
        st[i] = g.st;
        en[i] = g.en;
        out[i] = a.s + (int64_t)g.row * a.max_len - g.st;
    }
    KTile<HD, 64 * NW> tile;
    constexpr bool AHEAD = NW == 4 && HD <= 128;  // registers for the next tile beside 8 x 16 sums
    const int step = (int)gridDim.z * 64;
    int p0 = sp.lo + (int)blockIdx.z * 64;
    if (AHEAD && p0 <= sp.hi) tile.load(a, kh, p0, sp.hi, tid, 0);
    for (; p0 <= sp.hi; p0 += step) {
        if constexpr (AHEAD) {
            tile.store(tid, 0, kt);
            lds_barrier();
            if (p0 + step <= sp.hi) tile.load(a, kh, p0 + step, sp.hi, tid, 0);
        } else {
            tile.copy(a, kh, p0, sp.hi, tid, kt);
            lds_barrier();
        }
        av16 acc[8], zero;  // a chain's first MFMA adds to a constant 0
#pragma unroll
        for (int i = 0; i < 16; ++i) zero[i] = 0.0f;
        const float *kr = kt + lane * (HD + 4);
        for_seq([&](auto d) {
            constexpr int D = decltype(d)::value;
            const av4 k = *(const av4 *)(kr + 4 * D);
            acc[4 * (D & 1) + 0] = __builtin_amdgcn_mfma_f32_16x16x1f32(q[D], k.x, D < 2 ? zero : acc[4 * (D & 1) + 0], 2, 0, 0);
            acc[4 * (D & 1) + 1] = __builtin_amdgcn_mfma_f32_16x16x1f32(q[D], k.y, D < 2 ? zero : acc[4 * (D & 1) + 1], 2, 1, 0);
            acc[4 * (D & 1) + 2] = __builtin_amdgcn_mfma_f32_16x16x1f32(q[D], k.z, D < 2 ? zero : acc[4 * (D & 1) + 2], 2, 2, 0);
            acc[4 * (D & 1) + 3] = __builtin_amdgcn_mfma_f32_16x16x1f32(q[D], k.w, D < 2 ? zero : acc[4 * (D & 1) + 3], 2, 3, 0);
        }, std::make_integer_sequence<int, HD / 4>{});
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const int p = p0 + 16 * (r / 4) + (lane & 15), i = r & 3;
            const float t = chain_tree(acc[0][r], acc[1][r], acc[2][r], acc[3][r], acc[4][r], acc[5][r], acc[6][r], acc[7][r]);
            if (p >= st[i] && p <= en[i]) out[i][p] = t * a.scale;
        }
        lds_barrier();
    }
}

// scores of fewer rows (decode): grid (K heads, key chunks), 2 wavefronts that work alone. A wavefront
// takes a tile of 64 keys into its own part of LDS and multiplies it with the head's rows, 4 at a
// time, by v_mfma_f32_4x4x1 (one register holds 16 dimensions x 4 rows of q): K is read once
// whatever the rows. 32 heads over 8, 4096 positions, hd 128: 6.7 us; K's bytes are 2.5 of them. Every tile
// is in flight at once, two wavefronts a CU: a wavefront's one pass bounds it, 43 % of its life waits
// for its tile and 36 % issues VALU work (1667 instructions: addresses, LDS stores, the trees).
template <int HD>
__global__ __launch_bounds__(128) void attn_scores4_kernel(AttnArgs a, int n_tok) {
    __shared__ __attribute__((aligned(16))) float kt[2][64 * (HD + 4)];
    const int kh = blockIdx.x, tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int rows = n_tok * (a.n_head / a.n_head_kv);  // at most 16
    const GroupSpan sp = group_span(a, n_tok, 16, 0, kh);
    if (!sp.any()) return;
    constexpr int NQ = (HD + 15) / 16;
    for (int p0 = sp.lo + (int)(2 * blockIdx.y + wave) * 64; p0 <= sp.hi; p0 += (int)gridDim.y * 128) {
        for (int r0 = 0; r0 < rows; r0 += 4) {
            float q[NQ];
            const GroupRow mq = sp.row(r0 + (lane & 3));
            const float *qp = a.q + (int64_t)(mq.en >= mq.st ? mq.row : sp.first.row) * HD + (lane >> 2);
#pragma unroll
            for (int i = 0; i < NQ; ++i) q[i] = qp[16 * i];
            if (r0 == 0) {
                KTile<HD, 64> tile;
                tile.copy(a, kh, p0, sp.hi, lane, kt[wave]);
                __builtin_amdgcn_wave_barrier();  // the lanes of one wavefront share the tile: its LDS accesses are in order
            }
            av4 acc[8];
#pragma unroll
            for (int l = 0; l < 8; ++l) acc[l] = (av4){0.0f, 0.0f, 0.0f, 0.0f};
            const float *kr = kt[wave] + lane * (HD + 4);
            for_seq([&](auto d) {
                constexpr int D = decltype(d)::value;
                const av4 k = *(const av4 *)(kr + 4 * D);
                constexpr int B = 4 * (D & 1), Q = D / 4, J = 4 * (D % 4);
                acc[B + 0] = __builtin_amdgcn_mfma_f32_4x4x1f32(q[Q], k.x, acc[B + 0], 4, J + 0, 0);
                acc[B + 1] = __builtin_amdgcn_mfma_f32_4x4x1f32(q[Q], k.y, acc[B + 1], 4, J + 1, 0);
                acc[B + 2] = __builtin_amdgcn_mfma_f32_4x4x1f32(q[Q], k.z, acc[B + 2], 4, J + 2, 0);
                acc[B + 3] = __builtin_amdgcn_mfma_f32_4x4x1f32(q[Q], k.w, acc[B + 3], 4, J + 3, 0);
            }, std::make_integer_sequence<int, HD / 4>{});
            const int p = p0 + lane;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const GroupRow g = sp.urow(r0 + i);
                const float t = chain_tree(acc[0][i], acc[1][i], acc[2][i], acc[3][i], acc[4][i], acc[5][i], acc[6][i], acc[7][i]);
                if (p >= g.st && p <= g.en) a.s[(int64_t)g.row * a.max_len + (p - g.st)] = t * a.scale;
            }
        }
    }
}

template <int HD>
static void scores_launch(const AttnArgs &a, int n_tok, hipStream_t s) {
    const int rows_kv = n_tok * (a.n_head / a.n_head_kv), tiles = (a.max_len + 63) / 64;
    const unsigned kvh = (unsigned)a.n_head_kv;
    if (rows_kv < 16) {
        attn_scores4_kernel<HD><<<dim3(kvh, (unsigned)std::min((tiles + 1) / 2, 65535)), 128, 0, s>>>(a, n_tok);
        return;
    }
    // key chunks: about 512 workgroups of 4 wavefronts (2 per CU), each keeping its q over its tiles
    const int nw = rows_kv <= 16 ? 1 : rows_kv <= 32 ? 2 : 4, groups = (rows_kv + 16 * nw - 1) / (16 * nw);
    const unsigned ch = (unsigned)std::min((int64_t)tiles, std::max((int64_t)1, (int64_t)2048 / nw / ((int64_t)kvh * groups)));
    const dim3 g(kvh, (unsigned)groups, ch);
    if (nw == 1) attn_scores16_kernel<HD, 1><<<g, 64, 0, s>>>(a, n_tok);
    else if (nw == 2) attn_scores16_kernel<HD, 2><<<g, 128, 0, s>>>(a, n_tok);
    else attn_scores16_kernel<HD, 4><<<g, 256, 0, s>>>(a, n_tok);
}

// scores of the per-row path (hd % 32 != 0): thread = one key of the group's
// union, the q rows from LDS, K read value by value (any head size and offset), dot_f32v's order
template <int R>
__global__ __launch_bounds__(256) void attn_scores_row_kernel(AttnArgs a, int n_tok) {
    __shared__ float qs[R][256];
    const int grp = blockIdx.y, kh = blockIdx.z, tid = threadIdx.x;
    const GroupSpan sp = group_span(a, n_tok, R, grp, kh);
    if (!sp.any()) return;
    const int lo = sp.lo, hi = sp.hi;
    const int hd = a.hd;
    for (int i = tid; i < R * hd; i += 256) {
        const int r = i / hd, x = i - r * hd;
        const GroupRow g = group_row(a, n_tok, R, grp, kh, r);
        qs[r][x] = g.en >= g.st ? a.q[(size_t)g.row * hd + x] : 0.0f;
    }
    __syncthreads();
    const int64_t kvo = (int64_t)kh * hd;
    for (int p = lo + (int)blockIdx.x * 256 + tid; p <= hi; p += (int)gridDim.x * 256) {
        const float *kp = a.k + kv_slot(p, a.cap) * a.kv_dim + kvo;
        float s0[R][8], s1[R][8];
#pragma unroll
        for (int r = 0; r < R; ++r)
#pragma unroll
            for (int l = 0; l < 8; ++l) s0[r][l] = s1[r][l] = 0.0f;
        int i = 0;
        for (; i + 16 <= hd; i += 16) {
            float k0[8], k1[8];
#pragma unroll
            for (int l = 0; l < 8; ++l) {
                k0[l] = kp[i + l];
                k1[l] = kp[i + 8 + l];
            }
#pragma unroll
            for (int r = 0; r < R; ++r)
#pragma unroll
                for (int l = 0; l < 8; ++l) {
                    s0[r][l] = __builtin_fmaf(qs[r][i + l], k0[l], s0[r][l]);
                    s1[r][l] = __builtin_fmaf(qs[r][i + 8 + l], k1[l], s1[r][l]);
                }
        }
        if (i + 8 <= hd) {
#pragma unroll
            for (int l = 0; l < 8; ++l) {
                const float k0 = kp[i + l];
#pragma unroll
                for (int r = 0; r < R; ++r) s0[r][l] = __builtin_fmaf(qs[r][i + l], k0, s0[r][l]);
            }
            i += 8;
        }
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const GroupRow g = sp.urow(r);
            if (p >= g.st && p <= g.en) {
                float v[8];
#pragma unroll
                for (int l = 0; l < 8; ++l) v[l] = s0[r][l] + s1[r][l];
                float t = ((v[0] + v[4]) + (v[1] + v[5])) + ((v[2] + v[6]) + (v[3] + v[7]));  // hsum_ps
                for (int j = i; j < hd; ++j) t = __builtin_fmaf(qs[r][j], kp[j], t);
                a.s[(size_t)g.row * a.max_len + (p - g.st)] = t * a.scale;
            }
        }
    }
}

// softmax: one workgroup per row, in place over the row's scores. A row of up to SM_RES positions
// stays in LDS (sized min(max_len, SM_RES) at launch, so short rows leave room for more
// workgroups per CU) from its one load to its one store: maximum, exponentials, lanes 0..7 of
// wavefront 0 running the 8 ordered sums, then every value times 1 / sum. Longer rows go
// through LDS SM_RES positions at a time, the 8 sums carried across the chunks. 1024 threads for
// few rows (decode: a CU holds one row), 256 for prompt batches.
constexpr int SM_RES = 12288;
__device__ __forceinline__ float sum8_tree(float v) {  // lanes 0..7: hsum_ps's tree
    v = v + __shfl_xor(v, 4, 8);                       // (v0 + v4), (v1 + v5), ...
    v = v + __shfl_xor(v, 1, 8);
    return v + __shfl_xor(v, 2, 8);  // ((v0 + v4) + (v1 + v5)) + ((v2 + v6) + (v3 + v7))
}
// v += e[8g + l], g < ng: 16 values read while the 16 before them are added, one wait per batch
// (the adds are the bound: 4096 positions are 512 dependent adds)
__device__ __forceinline__ float lane_sum(const float *e, int ng, int l, float v) {
    const int n16 = ng & ~15;
    float t0[16], t1[16];
    auto read = [&](float *t, int g) {
        const float *p = e + 8 * g + l;
#pragma unroll
        for (int u = 0; u < 16; ++u) t[u] = p[8 * u];
        __builtin_amdgcn_sched_barrier(0);
    };
    auto add = [&](const float *t) {
        __builtin_amdgcn_s_waitcnt(0xC87F);  // lgkmcnt 8: the next batch's 8 paired reads may be in flight
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int u = 0; u < 16; ++u) v += t[u];
        __builtin_amdgcn_sched_barrier(0);
    };
    int g = 0;
    if (n16) {
        read(t0, 0);
        for (; g + 32 <= n16; g += 32) {
            read(t1, g + 16);
            add(t0);
            read(t0, g + 32 < n16 ? g + 32 : 0);  // past the end: any batch, not added
            add(t1);
        }
        if (g < n16) add(t0);
    }
    for (g = n16; g < ng; ++g) v += e[8 * g + l];
    return v;
}
template <int NT>
__device__ __forceinline__ float wg_max(float mx, float *red) {  // every thread of NT calls it
    for (int o = 1; o < 64; o <<= 1) mx = fmaxf(mx, __shfl_xor(mx, o, 64));
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = mx;
    __syncthreads();
#pragma unroll
    for (int w = 0; w < NT / 64; ++w) mx = fmaxf(mx, red[w]);
    return mx;
}
template <int NT>
__global__ __launch_bounds__(NT) void attn_softmax_kernel(AttnArgs a) {
    extern __shared__ float e[];  // min(max_len, SM_RES) values
    __shared__ float red[NT / 64];
    __shared__ float total;
    const int row = blockIdx.x, tok = row / a.n_head, tid = threadIdx.x;
    const int n = row_len(a, tok);
    if (n == 0) return;
    float *s = a.s + (size_t)row * a.max_len;
    const int nv = n & ~7;  // whole groups of 8
    const bool resident = n <= SM_RES;
    float mx = -__builtin_inff();
    if (resident) {
#pragma unroll 4
        for (int i = tid; i < n; i += NT) {
            const float x = s[i];
            e[i] = x;
            mx = fmaxf(mx, x);
        }
    } else {
        for (int i = tid; i < n; i += NT) mx = fmaxf(mx, s[i]);
    }
    mx = wg_max<NT>(mx, red);
    if (resident) {
        // whole groups and the tail apart, 4 values of a thread at a time: 2048 rows of 4096 positions
        // take 18.3 us instead of 20.1
#pragma unroll 4
        for (int i = tid; i < nv; i += NT) e[i] = exp_neg_ref(e[i] - mx);
        if (nv + tid < n) e[nv + tid] = expf_ref(e[nv + tid] - mx);
        __syncthreads();
        if (tid < 8) {
            float v = sum8_tree(lane_sum(e, nv / 8, tid, 0.0f));
            if (tid == 0) {
                for (int i = nv; i < n; ++i) v += e[i];  // the tail, in order
                total = v;
            }
        }
        __syncthreads();
        const float sum = total;
        const float inv = 1.0f / sum;
        const float f = sum > 0.0f ? inv : 1.0f;
#pragma unroll 4
        for (int i = tid; i < n; i += NT) s[i] = e[i] * f;
        return;
    }
    float v = 0.0f;
    for (int c0 = 0; c0 < n; c0 += SM_RES) {
        const int cn = min(SM_RES, n - c0);
        for (int i = tid; i < cn; i += NT) {
            const float x = s[c0 + i] - mx;
            const float ev = c0 + i < nv ? exp_neg_ref(x) : expf_ref(x);
            e[i] = ev;
            s[c0 + i] = ev;
        }
        __syncthreads();
        if (tid < 8) {
            v = lane_sum(e, (min(c0 + cn, nv) - c0) / 8, tid, v);
            if (c0 + cn == n) {  // the last chunk holds the tail
                v = sum8_tree(v);
                if (tid == 0) {
                    for (int i = nv; i < n; ++i) v += e[i - c0];
                    total = v;
                }
            }
        }
        __syncthreads();
    }
    const float sum = total;
    if (sum > 0.0f) {
        const float inv = 1.0f / sum;
        for (int i = tid; i < n; i += NT) s[i] = s[i] * inv;
    }
}

// ---- values: loaders shared by the two kernels below ----
// V of a tile of TP positions: a loading thread takes 4 columns of the chunk at every PS-th position
// from its own. Positions are uniform over the workgroup, so a tile that neither passes hi nor
// wraps around the ring is one scalar base plus a fixed 32-bit offset per thread and pass; the
// others clamp every position to hi's slot (a valid address: positions past hi are never summed).
// The values go to LDS transposed ([column][position]): a chain reads 4 positions of its column at
// a time. 16 lanes at consecutive positions x 4 column quads write all 64 banks.
// VB = 0: V in fp32 (a.v); VB = 2, 4, 8: V as TurboQuant records (a.vq), decoded to centroids
// (int8 codes for VB = 8) through an LDS table when a tile is stored.
// SC: V read value by value (hd or kv_dim not a multiple of 4: a 16-byte read would not be
// aligned), columns past hd reading the thread's first column.
template <int TP, int PS, int VB, bool SC>
struct AvLoader {
    static constexpr int M = TP / PS;  // passes per tile
    struct Stage {
        av4 v[VB ? 1 : M];
        uint32_t k[VB ? M : 1];
    };
    const uint8_t *base;  // the chunk's first column of the K / V head, slot 0
    int64_t stride;       // bytes per slot
    uint32_t off;         // this thread's column, bytes from base
    int sc1, sc2, sc3, lp, cap, hi, slot_hi;
    bool wide;            // a tile's byte offsets may exceed 32 bits: clamped form only
    // quad: the thread's columns 4 quad .. + 3 of the chunk at cc; pos: its first position
    __device__ __forceinline__ void init(const AttnArgs &a, int kh, int cc, int quad, int pos, int hi_) {
        const int lc = quad * 4, lcol = cc + lc < a.hd ? lc : -cc;  // columns past hd read column 0
        lp = pos;
        if constexpr (VB == 0) {
            base = (const uint8_t *)(a.v + (int64_t)kh * a.hd);
            stride = (int64_t)a.kv_dim * 4;
            off = (uint32_t)(cc + lcol) * 4;
            sc1 = cc + lc + 1 < a.hd ? 1 : 0;
            sc2 = cc + lc + 2 < a.hd ? 2 : 0;
            sc3 = cc + lc + 3 < a.hd ? 3 : 0;
        } else {
            const int vrec = 4 + a.hd * VB / 8;  // record bytes; the slot's records back to back
            base = a.vq + (int64_t)kh * vrec + 4;
            stride = (int64_t)a.n_head_kv * vrec;
            off = (uint32_t)(cc + lcol) * VB / 8;
        }
        cap = a.cap;
        hi = hi_;
        slot_hi = (int)kv_slot(hi_, a.cap);
        wide = stride * TP > 0x7fffffff;
    }
    __device__ __forceinline__ void one(Stage &s, int m, const uint8_t *p) const {
        if constexpr (VB == 0 && SC) {
            const float *vp = (const float *)p;
            s.v[m] = (av4){vp[0], vp[sc1], vp[sc2], vp[sc3]};
        } else if constexpr (VB == 0)
            s.v[m] = *(const av4 *)p;
        else if constexpr (VB == 8)
            s.k[m] = *(const uint32_t *)p;
        else if constexpr (VB == 4)
            s.k[m] = *(const uint16_t *)p;
        else
            s.k[m] = *p;
    }
    __device__ __forceinline__ void load(Stage &s, int p0) const {
        const int s0 = __builtin_amdgcn_readfirstlane((int)kv_slot(p0, cap));
        if (p0 + TP - 1 <= hi && s0 + TP <= cap && !wide) {  // uniform
            const uint8_t *tb = base + s0 * stride;
            const uint32_t st = (uint32_t)stride, o = off + (uint32_t)lp * st;
#pragma unroll
            for (int m = 0; m < M; ++m) one(s, m, tb + (o + (uint32_t)(m * PS) * st));
        } else {
#pragma unroll
            for (int m = 0; m < M; ++m) {
                const int p = p0 + lp + m * PS;
                one(s, m, base + (p <= hi ? kv_slot(p, cap) : slot_hi) * stride + off);
            }
        }
    }
    // the 4 values of pass m; tab: 4 bits: the centroid pairs of a code byte; 2 bits: the centroids
    __device__ __forceinline__ av4 value(const Stage &s, int m, const float2 *tab) const {
        if constexpr (VB == 0) return s.v[m];
        else if constexpr (VB == 8) {
            const uint32_t c = s.k[m];
            return (av4){(float)(int8_t)c, (float)(int8_t)(c >> 8), (float)(int8_t)(c >> 16), (float)(int8_t)(c >> 24)};
        } else {
            const uint32_t c = s.k[m];
            const float2 x = tab[VB == 4 ? c & 255 : c & 15], y = tab[VB == 4 ? c >> 8 : c >> 4];
            return (av4){x.x, x.y, y.x, y.y};
        }
    }
    // a tile into LDS: dst = [column 0 of the thread's quad][its first position], rows of P floats
    template <int P>
    __device__ __forceinline__ void store(const Stage &s, float *dst, const float2 *tab) const {
#pragma unroll
        for (int m = 0; m < M; ++m) {
            const av4 v = value(s, m, tab);
#pragma unroll
            for (int i = 0; i < 4; ++i) dst[i * P + m * PS] = v[i];
        }
    }
    static __device__ __forceinline__ void table(float2 *tab, int t, int nthreads) {
        if constexpr (VB == 4)
            for (int i = t; i < 256; i += nthreads) tab[i] = make_float2(kvq_centroid4(i & 15), kvq_centroid4(i >> 4));
        if constexpr (VB == 2)
            for (int i = t; i < 16; i += nthreads) tab[i] = make_float2(kvq_centroid2(i & 3), kvq_centroid2(i >> 2));
    }
};

// The weights of a tile: thread t takes 4 consecutive positions of one row per pass. A tile inside
// every valid row's range reads them unmasked; otherwise each position is clamped into the row's
// scores and masked to 0 outside its range. A row without a valid range has weight 0 and reads a
// valid row's scores.
struct AvWeights {
    const float *row;  // row + position = this row's weight
    int st, en, in_lo, in_hi;
    bool valid;
    __device__ __forceinline__ void init(const AttnArgs &a, const GroupSpan &sp, int r) {
        in_lo = sp.in_lo;
        in_hi = sp.in_hi;
        const GroupRow g = sp.row(r);
        valid = g.en >= g.st;
        st = valid ? g.st : sp.first.st;
        en = valid ? g.en : sp.first.en;
        row = a.s + (int64_t)(valid ? g.row : sp.first.row) * a.max_len - st;
    }
    __device__ __forceinline__ bool inside(int p0, int n) const { return p0 >= in_lo && p0 + n - 1 <= in_hi; }
    // positions p .. p + 3; in: the whole tile is inside every valid row's range (uniform)
    __device__ __forceinline__ av4 load(int p, bool in) const {
        if (in) return *(const av4u *)(row + p);
        av4 w;
#pragma unroll
        for (int i = 0; i < 4; ++i) w[i] = row[min(max(p + i, st), en)];
        return w;
    }
    __device__ __forceinline__ av4 mask(av4 w, int p, bool in) const {
        if (!in) {
#pragma unroll
            for (int i = 0; i < 4; ++i) w[i] = p + i >= st && p + i <= en ? w[i] : 0.0f;
        }
        return valid ? w : (av4){0.0f, 0.0f, 0.0f, 0.0f};
    }
};

// values of prompt batches: grid (K heads, groups of 16 rows, 64-column chunks), 4 chain wavefronts
// and 8 loading wavefronts. Chain wavefront w sums rows 4 w .. 4 w + 3 of the group over the
// chunk's 64 columns with v_mfma_f32_4x4x1: its 16 blocks are 16 groups of 4 columns, K = 1 is one
// position, so one instruction adds w_p v_p to 256 sums, each as one fmaf (subnormals, infinities and
// NaN included), in the position's turn. cbsz = 4
// broadcasts one of 16 blocks of the weight register to all: one register holds 16 positions x 4
// rows, one LDS read. The reads of 16 positions are issued before the MFMAs of the 16 before them,
// one wait per batch. The loaders hold 4 tiles of 128 positions in flight in registers (all
// workgroups of a head reach a tile at about the same time, so each tile comes from beyond the L2)
// and fill the other LDS buffer while the chain wavefronts sum; one barrier per tile.
// PR: the reference's per-row path (hd % 32 != 0, fastgguf.c:3318-3323): each row's chain walks
// only its own positions st..en, so a position of another row of the group adds nothing to it (not
// even fma(0, v, acc), which is NaN for a non-finite v and turns -0 into +0); the vector path's
// att_v_kern walks the group's whole span with zero weights, as the chains do without PR
// 64 tokens x 32 heads over 8, 4096 positions, hd 128: 50 us, 1.5 (3200 to 3600 cycles) a tile. The chain,
// one dependent MFMA of 12.2 cycles per position, is 1560 of them, 1950 with the LDS reads of 4 wavefronts
// a CU. By the counters the LDS is active for a third of the time (a quarter of that bank conflicts) and the
// matrix pipe for less: neither is the bound; all wavefronts together spend half their cycles in waits
// (the tile's barrier, loads, LDS).
constexpr int AP_T = 128, AP_P = AP_T + 4, AP_W = AP_T + 16;  // positions per tile, LDS rows of V and of the weights
template <int VB, bool SC, bool PR>
__global__ __launch_bounds__(768) void attn_values16_kernel(AttnArgs a, int n_tok) {
    typedef AvLoader<AP_T, 32, VB, SC> Loader;
    __shared__ __attribute__((aligned(16))) float vt[2][64 * AP_P];
    __shared__ __attribute__((aligned(16))) float wt[2][16 * AP_W];  // [row][position]
    __shared__ float2 tab[VB == 4 ? 256 : 16];
    const int kh = blockIdx.x, grp = blockIdx.y, cc = (int)blockIdx.z * 64, tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const GroupSpan sp = group_span(a, n_tok, 16, grp, kh);
    if (!sp.any()) {
        for (int r = 0; wave < 4 && r < 4; ++r) {
            const GroupRow g = sp.urow(4 * wave + r);
            if (g.row >= 0 && cc + lane < a.hd) a.o[(size_t)g.row * a.hd + cc + lane] = __builtin_nanf("");
        }
        return;
    }
    const int lo = sp.lo, hi = sp.hi, span = hi - lo + 1, nt = (span + AP_T - 1) / AP_T;
    if (VB == 2 || VB == 4) {
        Loader::table(tab, tid, 768);
        __syncthreads();
    }
    if (wave >= 4) {  // loaders
        const int t = tid - 256, wr = t >> 5, wp = (t & 31) * 4;
        const int quad = (t & 3) + 4 * ((t >> 6) & 3), pos = ((t & 63) >> 2) + 16 * (t >> 8);
        Loader ld;
        AvWeights lw;
        ld.init(a, kh, cc, quad, pos, hi);
        lw.init(a, sp, wr);
        struct Stage {
            typename Loader::Stage v;
            av4 w;
        } s0, s1, s2, s3;
        auto load = [&](int k, Stage &s) {
            const int p0 = lo + k * AP_T;
            if (k < nt) {
                s.w = lw.load(p0 + wp, lw.inside(p0, AP_T));
                ld.load(s.v, p0);
            }
        };
        auto store = [&](int k, Stage &s) {
            const int p0 = lo + k * AP_T;
            if (k < nt) {
                *(av4 *)&wt[k & 1][wr * AP_W + wp] = lw.mask(s.w, p0 + wp, lw.inside(p0, AP_T));
                ld.template store<AP_P>(s.v, &vt[k & 1][4 * quad * AP_P + pos], tab);
            }
        };
        load(0, s0);
        load(1, s1);
        load(2, s2);
        load(3, s3);
        store(0, s0);
        load(4, s0);
        lds_barrier();
        auto step = [&](int k, Stage &s) {  // while tile k is summed: tile k + 1 stored, k + 5 requested
            if (k < nt) {
                store(k + 1, s);
                load(k + 5, s);
                lds_barrier();
            }
        };
        for (int k = 0; k < nt; k += 4) {
            step(k, s1);
            step(k + 1, s2);
            step(k + 2, s3);
            step(k + 3, s0);
        }
        return;
    }
    __builtin_amdgcn_s_setprio(1);
    av4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
    int rst[4], ren[4], in_lo = lo, in_hi = hi;  // PR: the ranges of this wavefront's rows
    if (PR) {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const GroupRow g = sp.urow(4 * wave + r);
            const bool ok = g.en >= g.st;  // a row without a range: its sums are not stored
            rst[r] = ok ? g.st : lo;
            ren[r] = ok ? g.en : hi;
            in_lo = max(in_lo, rst[r]);
            in_hi = min(in_hi, ren[r]);
        }
    }
    lds_barrier();
    for (int k = 0; k < nt; ++k) {
        const int p0 = lo + k * AP_T, cnt = min(AP_T, span - k * AP_T);
        const float *vs = vt[k & 1] + lane * AP_P;
        const float *ws = wt[k & 1] + (4 * wave + (lane & 3)) * AP_W + (lane >> 2);
        struct Batch {  // 16 positions
            float w;
            av4 v[4];
        } x, y;
        auto read = [&](Batch &s, int g) {
            s.w = ws[16 * g];
#pragma unroll
            for (int q = 0; q < 4; ++q) s.v[q] = *(const av4 *)(vs + 16 * g + 4 * q);
            __builtin_amdgcn_sched_barrier(0);
        };
        auto sum = [&](const Batch &s) {
            for_seq([&](auto j) { acc = __builtin_amdgcn_mfma_f32_4x4x1f32(s.w, s.v[j() / 4][j() % 4], acc, 4, j(), 0); },
                  std::make_integer_sequence<int, 16>{});
            __builtin_amdgcn_sched_barrier(0);
        };
        if (cnt == AP_T && (!PR || (p0 >= in_lo && p0 + AP_T - 1 <= in_hi))) {
            read(x, 0);
#pragma unroll
            for (int g = 0; g < AP_T / 16; g += 2) {
                read(y, g + 1);
                __builtin_amdgcn_s_waitcnt(0xC57F);  // lgkmcnt 5: y's reads may be in flight
                __builtin_amdgcn_sched_barrier(0);
                sum(x);
                if (g + 2 < AP_T / 16) {
                    read(x, g + 2);
                    __builtin_amdgcn_s_waitcnt(0xC57F);
                    __builtin_amdgcn_sched_barrier(0);
                }
                sum(y);
            }
        } else {
            for (int g = 0; 16 * g < cnt; ++g) {
                read(x, g);
                for_seq([&](auto j) {
                    const int p = p0 + 16 * g + j();
                    if (p <= hi) {
                        const av4 old = acc;
                        acc = __builtin_amdgcn_mfma_f32_4x4x1f32(x.w, x.v[j() / 4][j() % 4], acc, 4, j(), 0);
                        if (PR) {
#pragma unroll
                            for (int r = 0; r < 4; ++r) acc[r] = p >= rst[r] && p <= ren[r] ? acc[r] : old[r];
                        }
                    }
                }, std::make_integer_sequence<int, 16>{});
            }
        }
        lds_barrier();
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const GroupRow g = sp.urow(4 * wave + r);
        if (g.row >= 0 && cc + lane < a.hd)
            a.o[(size_t)g.row * a.hd + cc + lane] = g.en >= g.st ? acc[r] : __builtin_nanf("");
    }
}

// acc = fma(w of lane 16 r + n, v[n], acc) for n = 0 .. 15 in order, r the lane's group of 16: the
// broadcast is part of the instruction (row_newbcast on its first operand)
__device__ __forceinline__ void fmac16_bcast(float &acc, float w, const av4 &a, const av4 &b, const av4 &c, const av4 &d) {
#define FGH_FM(n, i) "v_fmac_f32_dpp %0, %1, %" #i " row_newbcast:" #n " row_mask:0xf bank_mask:0xf\n"
    asm volatile("s_nop 1\n" FGH_FM(0, 2) FGH_FM(1, 3) FGH_FM(2, 4) FGH_FM(3, 5) FGH_FM(4, 6) FGH_FM(5, 7) FGH_FM(6, 8)
                     FGH_FM(7, 9) FGH_FM(8, 10) FGH_FM(9, 11) FGH_FM(10, 12) FGH_FM(11, 13) FGH_FM(12, 14)
                         FGH_FM(13, 15) FGH_FM(14, 16) FGH_FM(15, 17)
                 : "+&v"(acc)
                 : "v"(w), "v"(a.x), "v"(a.y), "v"(a.z), "v"(a.w), "v"(b.x), "v"(b.y), "v"(b.z), "v"(b.w), "v"(c.x),
                   "v"(c.y), "v"(c.z), "v"(c.w), "v"(d.x), "v"(d.y), "v"(d.z), "v"(d.w));
#undef FGH_FM
}

// values of small batches (decode): grid (K heads, groups of 4 rows, 16-column chunks), one chain
// wavefront and 4 loading wavefronts. Lane 16 r + c of the chain wavefront sums row r, column c:
// the narrow chunk gives a decode step of 8 K / V heads 64 workgroups, and V lies transposed in
// LDS ([column][position]), so one 16-byte read feeds 4 positions and the 4 rows share it; the
// row's weight comes in by a lane broadcast inside the fma. The reads of the next 32 positions
// are issued before the 32 fmas of the current ones, one wait for the whole batch.
// 32 heads over 8, 4096 positions, hd 128: 18.5 us. 4096 dependent fmas per lane are 9 to 12 of them (about
// 5.3 cycles each, 7 with the reads); the rest is the range search, the first tiles' way from memory
// and the loaders' stores (a quarter of the LDS cycles are bank conflicts).
constexpr int AD_T = 256, AD_P = AD_T + 4;  // positions per tile, LDS row (16 columns of 16 bytes cover all banks)
template <int VB, bool SC, bool PR>
__global__ __launch_bounds__(320) void attn_values4_kernel(AttnArgs a, int n_tok) {
    typedef AvLoader<AD_T, 64, VB, SC> Loader;
    __shared__ __attribute__((aligned(16))) float vt[2][16 * AD_P];
    __shared__ __attribute__((aligned(16))) float wt[2][4 * AD_P];
    __shared__ float2 tab[VB == 4 ? 256 : 16];
    const int kh = blockIdx.x, grp = blockIdx.y, cc = (int)blockIdx.z * 16, tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int r = lane >> 4, c = lane & 15;
    const GroupSpan sp = group_span(a, n_tok, 4, grp, kh);
    const GroupRow me = sp.row(r);
    if (!sp.any()) {
        if (wave == 0 && me.row >= 0 && cc + c < a.hd) a.o[(size_t)me.row * a.hd + cc + c] = __builtin_nanf("");
        return;
    }
    const int lo = sp.lo, hi = sp.hi, span = hi - lo + 1, nt = (span + AD_T - 1) / AD_T;
    if (VB == 2 || VB == 4) {
        Loader::table(tab, tid, 320);
        __syncthreads();
    }
    if (wave > 0) {  // loaders
        const int t = tid - 64;
        Loader ld;
        AvWeights lw;
        ld.init(a, kh, cc, t & 3, t >> 2, hi);
        lw.init(a, sp, t >> 6);
        struct Stage {
            typename Loader::Stage v;
            av4 w;
        } s0, s1;
        auto load = [&](int k, Stage &s) {
            const int p0 = lo + k * AD_T;
            s.w = lw.load(p0 + 4 * lane, lw.inside(p0, AD_T));
            ld.load(s.v, p0);
        };
        auto store = [&](int k, Stage &s) {
            const int b = k & 1, p0 = lo + k * AD_T;
            *(av4 *)&wt[b][(t >> 6) * AD_P + 4 * lane] = lw.mask(s.w, p0 + 4 * lane, lw.inside(p0, AD_T));
            ld.template store<AD_P>(s.v, &vt[b][(t & 3) * 4 * AD_P + (t >> 2)], tab);
        };
        load(0, s0);
        if (nt > 1) load(1, s1);
        store(0, s0);
        if (nt > 2) load(2, s0);
        lds_barrier();
        auto step = [&](int k, Stage &s) {  // while tile k is summed: tile k + 1 stored, k + 3 requested
            if (k + 1 < nt) {
                store(k + 1, s);
                if (k + 3 < nt) load(k + 3, s);
            }
            lds_barrier();
        };
        for (int k = 0; k < nt; k += 2) {
            step(k, s1);
            if (k + 1 < nt) step(k + 1, s0);
        }
        return;
    }
    __builtin_amdgcn_s_setprio(1);
    float acc = 0.0f;
    const bool ok = me.en >= me.st;
    const int rst = ok ? me.st : lo, ren = ok ? me.en : hi;
    const int in_lo = sp.in_lo, in_hi = sp.in_hi;
    lds_barrier();
    for (int k = 0; k < nt; ++k) {
        const int b = k & 1, p0 = lo + k * AD_T, cnt = min(AD_T, span - k * AD_T);
        const av4 *vs = (const av4 *)(vt[b] + c * AD_P);
        const float *ws = wt[b] + r * AD_P;
        struct Batch {  // 32 positions
            av4 v[8];
            float w0, w1;
        } x, y;
        auto read = [&](Batch &s, int i) {
            s.w0 = ws[32 * i + c];
            s.w1 = ws[32 * i + 16 + c];
#pragma unroll
            for (int q = 0; q < 8; ++q) s.v[q] = vs[8 * i + q];
            __builtin_amdgcn_sched_barrier(0);
        };
        auto sum = [&](Batch &s) {
            fmac16_bcast(acc, s.w0, s.v[0], s.v[1], s.v[2], s.v[3]);
            fmac16_bcast(acc, s.w1, s.v[4], s.v[5], s.v[6], s.v[7]);
            __builtin_amdgcn_sched_barrier(0);
        };
        if (cnt == AD_T && (!PR || (p0 >= in_lo && p0 + AD_T - 1 <= in_hi))) {
            read(x, 0);
#pragma unroll
            for (int i = 0; i < AD_T / 32; i += 2) {
                read(y, i + 1);
                __builtin_amdgcn_s_waitcnt(0xCA7F);  // lgkmcnt 10: y's reads may be in flight
                __builtin_amdgcn_sched_barrier(0);
                sum(x);
                if (i + 2 < AD_T / 32) {
                    read(x, i + 2);
                    __builtin_amdgcn_s_waitcnt(0xCA7F);
                    __builtin_amdgcn_sched_barrier(0);
                }
                sum(y);
            }
        } else {
            int i = 0;
            for (; 32 * i + 32 <= cnt; ++i) {
                const int q0 = p0 + 32 * i;
                if (PR && !(q0 >= in_lo && q0 + 31 <= in_hi)) break;
                read(x, i);
                sum(x);
            }
            for (int j = 32 * i; j < cnt; ++j) {
                const float s = __builtin_fmaf(ws[j], ((const float *)vs)[j], acc);
                acc = !PR || (p0 + j >= rst && p0 + j <= ren) ? s : acc;
            }
        }
        lds_barrier();
    }
    if (me.row >= 0 && cc + c < a.hd) a.o[(size_t)me.row * a.hd + cc + c] = ok ? acc : __builtin_nanf("");
}

template <int VB, bool SC, bool PR>
static void values_launch(const AttnArgs &a, int n_tok, hipStream_t s) {
    const int rows_kv = n_tok * (a.n_head / a.n_head_kv);
    const unsigned kvh = (unsigned)a.n_head_kv;
    // K heads along x: workgroups go to the 8 XCDs in turn, so with 8 K heads every XCD's L2 holds
    // one head's V
    if (rows_kv >= 64)
        attn_values16_kernel<VB, SC, PR>
            <<<dim3(kvh, (unsigned)((rows_kv + 15) / 16), (unsigned)((a.hd + 63) / 64)), 768, 0, s>>>(a, n_tok);
    else
        attn_values4_kernel<VB, SC, PR>
            <<<dim3(kvh, (unsigned)((rows_kv + 3) / 4), (unsigned)((a.hd + 15) / 16)), 320, 0, s>>>(a, n_tok);
}

hipError_t launch_attention_values(const AttnArgs &a, int n_tok, hipStream_t s) {
    if (n_tok < 1 || a.hd < 1 || a.hd > 256 || a.n_head_kv < 1 || a.n_head % a.n_head_kv != 0 || a.max_len < 1)
        return hipErrorInvalidValue;
    const int rows_kv = n_tok * (a.n_head / a.n_head_kv);
    if ((rows_kv + 3) / 4 > 65535 || a.n_head_kv > 65535) return hipErrorInvalidValue;
    // 16-byte V reads need 4-value columns and rows; TurboQuant records need a multiple of 32
    const bool sc = a.hd % 4 != 0 || a.kv_dim % 4 != 0 || (uintptr_t)a.v % 16 != 0, pr = a.hd % 32 != 0;
    if (a.vq) {
        if (pr || sc) return hipErrorInvalidValue;
        if (a.vbits == 8) values_launch<8, false, false>(a, n_tok, s);
        else if (a.vbits == 4) values_launch<4, false, false>(a, n_tok, s);
        else if (a.vbits == 2) values_launch<2, false, false>(a, n_tok, s);
        else return hipErrorInvalidValue;
        return hipGetLastError();
    }
    if (!a.v) return hipErrorInvalidValue;
    if (pr) {  // the per-row path
        if (sc) values_launch<0, true, true>(a, n_tok, s);
        else values_launch<0, false, true>(a, n_tok, s);
    } else {
        if (sc) return hipErrorInvalidValue;  // hd % 32 == 0: launch_attention asks for aligned K, the caller for V
        values_launch<0, false, false>(a, n_tok, s);
    }
    return hipGetLastError();
}

hipError_t launch_attention(const AttnArgs &a, int n_tok, hipStream_t s) {
    if (n_tok < 1 || a.hd < 1 || a.hd > 256 || a.n_head_kv < 1 || a.n_head % a.n_head_kv != 0 || a.max_len < 1)
        return hipErrorInvalidValue;
    const bool vec = a.hd % 32 == 0;  // the reference's vector path: 16-byte reads of q and K
    if (vec && (a.kv_dim % 4 != 0 || ((uintptr_t)a.q | (uintptr_t)a.k) % 16 != 0)) return hipErrorInvalidValue;
    const int rows_kv = n_tok * (a.n_head / a.n_head_kv);  // rows per K / V head
    if ((rows_kv + 3) / 4 > 65535 || a.n_head_kv > 65535) return hipErrorInvalidValue;
    const unsigned kb = (unsigned)std::min((a.max_len + 255) / 256, 1024);
    const dim3 kvh(1, 1, (unsigned)a.n_head_kv);
    if (!vec)
        attn_scores_row_kernel<4><<<dim3(kb, (unsigned)((rows_kv + 3) / 4), kvh.z), 256, 0, s>>>(a, n_tok);
    else {
        switch (a.hd / 32) {
        case 1: scores_launch<32>(a, n_tok, s); break;
        case 2: scores_launch<64>(a, n_tok, s); break;
        case 3: scores_launch<96>(a, n_tok, s); break;
        case 4: scores_launch<128>(a, n_tok, s); break;
        case 5: scores_launch<160>(a, n_tok, s); break;
        case 6: scores_launch<192>(a, n_tok, s); break;
        case 7: scores_launch<224>(a, n_tok, s); break;
        default: scores_launch<256>(a, n_tok, s); break;
        }
    }
    const int rows = n_tok * a.n_head;
    const size_t lds = (size_t)std::min(a.max_len, SM_RES) * 4;
    if (rows <= 256) attn_softmax_kernel<1024><<<rows, 1024, lds, s>>>(a);
    else attn_softmax_kernel<256><<<rows, 256, lds, s>>>(a);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    return launch_attention_values(a, n_tok, s);
}

}  // namespace fgh
