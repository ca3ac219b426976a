// fgh_kvq.hip - the TurboQuant KV cache on gfx950 (fastgguf.c:3341-3513 and forward's attention
// step over it, 4726-4735 and 4760-4846), bit-exact with the compiled reference.
//
// Records: one per (slot, K / V head), KVQ_REC = 4 + hd * bits / 8 bytes: the float scale, then
// the codes (8 bits: int8; 4 bits: low nibble first; 2 bits: low bits first). A slot holds the
// n_head_kv records of one position back to back. The rotation R x = H(D x) / sqrt(hd) (signs D
// of xorshift64*, kvq_init 3363-3372; butterflies kvq_fwht 3375-3386) of a row runs in one wavefront by
// lane exchanges (rotate_wave), so every value sees the reference's additions.
//
// Attention (hd a power of 2, 32..256):
//   q rows rotated (4763)                                    kvq_rotate_gather_kernel (16 rows and
//                                                            more per K / V head), else in kvq_scores_kernel
//   scores: kvq_dot_k (3447-3462) times scale, per key       kvq_scores_kernel
//   softmax_inplace (3147-3156), then w' = w * s_V(p)         kvq_softmax_kernel
//   o = fma(w', centroid, o) over the positions in order     attn_values (fgh_attn.hip), which
//                                                            decodes the V codes as it stages them
//   output rows rotated back (4846)                           kvq_rotate_kernel
// kvq_axpy_v (3465-3489) adds fma(w * s, value, o) for each position with w != 0; w' = w * s is
// that product, and a position with w = 0 gets w' = 0 (not 0 * s, which an inf or NaN scale would
// turn into NaN) and adds fma(0, centroid, o) = o, so the value chains of the fp32 attention give
// its sums. No fp32 copy of the cache is made.
#include <hip/hip_runtime.h>

#include "fgh_internal.h"

namespace fgh {

namespace {

struct SignTable {
    float v[1024];
    constexpr SignTable() : v() {
        uint64_t s = 0x243F6A8885A308D3ULL;
        for (int i = 0; i < 1024; ++i) {
            uint64_t x = s;
            x ^= x >> 12;
            x ^= x << 25;
            x ^= x >> 27;
            s = x;
            v[i] = ((x * 0x2545F4914F6CDD1DULL) >> 63) ? 1.0f : -1.0f;
        }
    }
};
__constant__ SignTable kvq_sign = SignTable();

__device__ __forceinline__ int64_t slot_of(int p, int cap) { return (int64_t)(((p % cap) + cap) % cap); }

// The rotation (or its inverse) of one row in one wavefront: lane l holds values l + 64 e (hd 32:
// lanes 0..31, value l). Butterflies up to 32 apart are lane exchanges, wider ones stay in the
// lane; every value sees the reference's additions (lower: a + b, upper: a - b).
constexpr int KVQ_E = 4;  // hd <= 256
__device__ __forceinline__ void rotate_wave(float (&x)[KVQ_E], int hd, bool inverse) {
    const int lane = threadIdx.x & 63, ne = hd < 64 ? 1 : hd / 64;
    if (!inverse)
#pragma unroll
        for (int e = 0; e < KVQ_E; ++e) x[e] = x[e] * kvq_sign.v[lane + 64 * e];
#pragma unroll
    for (int len = 1; len < 64; len <<= 1) {
        if (len < hd) {
#pragma unroll
            for (int e = 0; e < KVQ_E; ++e)
                if (e < ne) {
                    const float o = __shfl_xor(x[e], len, 64);
                    x[e] = lane & len ? o - x[e] : x[e] + o;
                }
        }
    }
    if (hd >= 128) {
#pragma unroll
        for (int e = 0; e < KVQ_E; e += 2) {
            const float p = x[e], q = x[e + 1];
            x[e] = p + q;
            x[e + 1] = p - q;
        }
    }
    if (hd >= 256) {
#pragma unroll
        for (int e = 0; e < 2; ++e) {
            const float p = x[e], q = x[e + 2];
            x[e] = p + q;
            x[e + 2] = p - q;
        }
    }
    const float inv = 1.0f / sqrtf((float)hd);
#pragma unroll
    for (int e = 0; e < KVQ_E; ++e) x[e] = inverse ? x[e] * inv * kvq_sign.v[lane + 64 * e] : x[e] * inv;
}
__device__ __forceinline__ void row_load(float (&x)[KVQ_E], const float *src, int hd) {
    const int lane = threadIdx.x & 63;
#pragma unroll
    for (int e = 0; e < KVQ_E; ++e) x[e] = lane + 64 * e < hd ? src[lane + 64 * e] : 0.0f;
}

// the number of midpoints below u: the first code whose upper midpoint u does not pass
// (kvq_enc4 / kvq_enc2; a NaN passes none)
__device__ __forceinline__ uint32_t code4(float u) {
    uint32_t c = 0;
#pragma unroll
    for (int i = 0; i < 15; ++i) c += u > (kvq_centroid4(i) + kvq_centroid4(i + 1)) * 0.5f ? 1u : 0u;
    return c;
}
__device__ __forceinline__ uint32_t code2(float u) {
    uint32_t c = 0;
#pragma unroll
    for (int i = 0; i < 3; ++i) c += u > (kvq_centroid2(i) + kvq_centroid2(i + 1)) * 0.5f ? 1u : 0u;
    return c;
}

// sum += p[0], p[1], .. p[n - 1] in order (n a multiple of 32, p in LDS, 16-byte aligned): 32 values
// read while the 32 before them are added, one wait per batch. All lanes run the same sum.
__device__ __forceinline__ float ordered_sum(const float *p, int n, float sum) {
    typedef float kv4 __attribute__((ext_vector_type(4)));
    kv4 t0[8], t1[8];
    auto read = [&](kv4 *t, int i) {
        const kv4 *q = (const kv4 *)(p + i);
#pragma unroll
        for (int u = 0; u < 8; ++u) t[u] = q[u];
        __builtin_amdgcn_sched_barrier(0);
    };
    auto add = [&](const kv4 *t) {
        __builtin_amdgcn_s_waitcnt(0xC87F);  // lgkmcnt 8: the next batch may be in flight
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            sum += t[u].x;
            sum += t[u].y;
            sum += t[u].z;
            sum += t[u].w;
        }
        __builtin_amdgcn_sched_barrier(0);
    };
    if (n <= 0) return sum;
    read(t0, 0);
    int i = 0;
    for (; i + 64 <= n; i += 64) {
        read(t1, i + 32);
        add(t0);
        read(t0, i + 64 < n ? i + 64 : 0);  // past the end: any batch, not added
        add(t1);
    }
    if (i < n) add(t0);
    return sum;
}

// store: grid (tokens, K / V heads, 2: K then V), one wavefront. Rotates the head slice of the
// token's new K or V row and writes its record into slot pos % cap (kvq_quant_slice 3415-3444):
// each lane encodes its own values, and the lanes of a 32-bit word combine theirs by exchanges.
// The reference writes token after token: where two tokens of a call share a slot, only the
// later one writes.
__global__ __launch_bounds__(64) void kvq_store_kernel(KvqStoreArgs a, int n_tok) {
    __shared__ __attribute__((aligned(16))) float sq[256];
    const int tok = blockIdx.x, kh = blockIdx.y, isv = blockIdx.z, lane = threadIdx.x, hd = a.hd;
    float x[KVQ_E];
    row_load(x, (isv ? a.v : a.k) + (size_t)tok * a.stride + (size_t)kh * hd, hd);
    const int64_t my_slot = slot_of(a.pos[tok], a.cap);
    bool later = false;
    for (int t = tok + 1 + lane; t < n_tok; t += 64) later |= slot_of(a.pos[t], a.cap) == my_slot;
    if (__builtin_amdgcn_ballot_w64(later)) return;  // the whole wavefront
    const int bits = isv ? a.vbits : a.kbits;
    rotate_wave(x, hd, false);
    float s;
    if (bits == 8) {
        float amax = 0.0f;
#pragma unroll
        for (int e = 0; e < KVQ_E; ++e)
            if (lane + 64 * e < hd) amax = fmaxf(amax, fabsf(x[e]));
        for (int o = 1; o < 64; o <<= 1) amax = fmaxf(amax, __shfl_xor(amax, o, 64));
        s = amax / 127.0f;
    } else {  // the squares in parallel, their sum in order
#pragma unroll
        for (int e = 0; e < KVQ_E; ++e)
            if (lane + 64 * e < hd) sq[lane + 64 * e] = x[e] * x[e];
        __syncthreads();
        s = sqrtf(ordered_sum(sq, hd, 0.0f) / (float)hd);
    }
    const float inv = s > 0.0f ? 1.0f / s : 0.0f;
    const int rec = 4 + hd * bits / 8;
    uint8_t *dst = (isv ? a.vq : a.kq) + my_slot * (int64_t)(a.n_head_kv * rec) + (int64_t)kh * rec;
    if (lane == 0) *(float *)dst = s;
    uint32_t *words = (uint32_t *)(dst + 4);
    const int per = 32 / bits;  // codes per 32-bit word: per adjacent lanes
#pragma unroll
    for (int e = 0; e < KVQ_E; ++e) {
        if (64 * e >= hd) break;  // uniform
        const float u = x[e] * inv;
        uint32_t v = bits == 8 ? (uint32_t)(uint8_t)(int8_t)(int)rintf(u) : bits == 4 ? code4(u) : code2(u);
        v <<= bits * (lane & (per - 1));
        for (int o = 1; o < per; o <<= 1) v |= (uint32_t)__shfl_xor((int)v, o, 64);
        if ((lane & (per - 1)) == 0 && lane + 64 * e < hd) words[(lane + 64 * e) / per] = v;
    }
}

__device__ __forceinline__ int kvq_row_len(const KvqAttnArgs &a, int tok) {
    const int n = a.en[tok] - a.st[tok] + 1;
    return n >= 1 && n <= a.cap && n <= a.max_len ? n : 0;
}

// the V scales that some token's range reads, gathered: out[head * cap + slot]. A wavefront takes 64
// slots of one head; lane t looks at tokens t, t + 64, .. for a range that meets them, and without one
// nothing is read or written (a short range on a long ring would pay for every record of the cache).
struct KvqGather {
    KvqAttnArgs a;
    float *out;  // null: none
    int n_tok;
    unsigned wgs;  // workgroups, 4 wavefronts each
};
static unsigned kvq_gather_wgs(int cap, int n_head_kv) { return (unsigned)(((int64_t)((cap + 63) / 64) * n_head_kv + 3) / 4); }
__device__ __forceinline__ void kvq_gather(const KvqGather &g) {
    const KvqAttnArgs &a = g.a;
    const int w = (int)blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int kvh = w % a.n_head_kv, s0 = w / a.n_head_kv * 64, sl = s0 + lane;
    if (s0 >= a.cap) return;
    bool used = false;
    for (int t = lane; t < (g.n_tok + 63) / 64 * 64; t += 64) {  // uniform
        if (t < g.n_tok) {
            const int n = kvq_row_len(a, t), f = (int)slot_of(a.st[t], a.cap);  // slots f .. f + n - 1, around the ring
            used = n > 0 && ((f < s0 + 64 && f + n > s0) || f + n - a.cap > s0);
        }
        if (__builtin_amdgcn_ballot_w64(used)) break;
    }
    if (!__builtin_amdgcn_ballot_w64(used) || sl >= a.cap) return;
    const int rec = 4 + a.hd * a.vbits / 8;
    g.out[(int64_t)kvh * a.cap + sl] = *(const float *)(a.vq + ((int64_t)sl * a.n_head_kv + kvh) * rec);
}
// rows of hd values rotated (inverse = false) or rotated back: one wavefront per row, 4 rows per
// workgroup
__device__ __forceinline__ void rotate_rows(const float *in, float *out, int hd, int rows, bool inverse, unsigned wg) {
    const int row = (int)wg * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (row >= rows) return;
    float x[KVQ_E];
    row_load(x, in + (size_t)row * hd, hd);
    rotate_wave(x, hd, inverse);
#pragma unroll
    for (int e = 0; e < KVQ_E; ++e)
        if (lane + 64 * e < hd) out[(size_t)row * hd + lane + 64 * e] = x[e];
}
__global__ __launch_bounds__(256) void kvq_rotate_kernel(const float *in, float *out, int hd, int rows, bool inverse) {
    rotate_rows(in, out, hd, rows, inverse, blockIdx.x);
}
// the query rows rotated; the first g.wgs workgroups gather V scales
__global__ __launch_bounds__(256) void kvq_rotate_gather_kernel(KvqGather g) {
    if (blockIdx.x < g.wgs) kvq_gather(g);
    else rotate_rows(g.a.q, g.a.qr, g.a.hd, g.n_tok * g.a.n_head, false, blockIdx.x - g.wgs);
}

// Groups of R rows that read one K / V head kh: j = R q .. R q + R - 1 of the head's n_tok * G
// rows, j = t * G + g (token t, query head kh * G + g); the scores of a group run over the union
// of its rows' ranges and are stored for each row's own range.
struct KvqRow {
    int row, st, en;  // row = -1: no such row; en < st: no valid range
};
__device__ __forceinline__ KvqRow kvq_group_row(const KvqAttnArgs &a, int n_tok, int R, int grp, int kh, int r) {
    const int G = a.n_head / a.n_head_kv, j = grp * R + r;
    KvqRow g{-1, 0, -1};
    if (j < n_tok * G) {
        const int t = j / G;
        g.row = t * a.n_head + kh * G + (j - t * G);
        if (kvq_row_len(a, t) > 0) {
            g.st = a.st[t];
            g.en = a.en[t];
        }
    }
    return g;
}

// scores: grid of key blocks, groups of R rows and K / V heads, 256 threads; thread = one key of the
// group's union for its R rows: each record's codes are loaded and looked up once for R chains
// in kvq_dot_k's order, then times s, times scale. R = 16 for prompt batches. R = 4 (decode): each
// wavefront rotates one of the rows itself, while its keys' records are on their way: 10.8 us at 32
// heads, 4096 positions, hd 128, against 9.7 and a rotation launch of 4.0. (With 16 rows per group
// every key block would rotate 4 per wavefront.) A record's words are requested 8 ahead of their
// use. Bound at decode: latency, 128 workgroups of one wavefront a SIMD, which waits for half of its life;
// twice the workgroups of 128 threads took 11.5 us against 11.3.
// The grid has key blocks for max_len keys; those past the range leave before they load a record.
// R = 16: heads are the grid's fastest index, key blocks its slowest. With key blocks fastest the few
// workgroups of a short range all went to one XCD (32 or 64 blocks a group, 8 XCDs in turn): 64 tokens x
// 32 heads at the start of a ring of max_len 8192 took 77.9 us, now 38.2, and 4096 of 4096 positions
// 180.8, now 177.9. R = 4 keeps key blocks fastest: a full range of 4096 positions is 54.2 us so (16
// heads over 8, hd 256), 57.2 the other way.
template <int R>
__global__ __launch_bounds__(256) void kvq_scores_kernel(KvqAttnArgs a, int n_tok) {
    __shared__ float q[R][256];
    __shared__ float c4[16];
    const int grp = blockIdx.y, kh = R == 16 ? blockIdx.x : blockIdx.z, tid = threadIdx.x, hd = a.hd;
    const int kb = R == 16 ? blockIdx.z : blockIdx.x, nkb = R == 16 ? gridDim.z : gridDim.x;
    // every wavefront finds the group's ranges for itself: lane r (mod R) reads row r's, one round of
    // loads, and lane exchanges reduce them. R = 4: its own row of q is on its way meanwhile
    const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    float x[KVQ_E] = {0.0f, 0.0f, 0.0f, 0.0f};
    if (R == 4) {
        const int G = a.n_head / a.n_head_kv, j = grp * R + wave, t = j / G;
        if (t < n_tok) row_load(x, a.q + ((size_t)t * a.n_head + kh * G + (j - t * G)) * hd, hd);
    }
    const KvqRow mine = kvq_group_row(a, n_tok, R, grp, kh, lane & (R - 1));
    const bool ok = mine.en >= mine.st;
    int lo = ok ? mine.st : 0x7fffffff, hi = ok ? mine.en : -0x7fffffff;
    for (int o = 1; o < R; o <<= 1) {
        lo = min(lo, __shfl_xor(lo, o, 64));
        hi = max(hi, __shfl_xor(hi, o, 64));
    }
    lo = __builtin_amdgcn_readfirstlane(lo);
    hi = __builtin_amdgcn_readfirstlane(hi);
    if (hi < lo || (int64_t)lo + (int64_t)kb * 256 > hi) return;  // the whole workgroup: no key of its own
    KvqRow rows[R];
#pragma unroll
    for (int r = 0; r < R; ++r)
        rows[r] = KvqRow{__builtin_amdgcn_readlane(mine.row, r), __builtin_amdgcn_readlane(mine.st, r), __builtin_amdgcn_readlane(mine.en, r)};
    constexpr int CW = 8;
    const int rec = 4 + hd * a.kbits / 8, nw = hd * a.kbits / 32;
    const uint32_t *w = nullptr;
    uint32_t cur[CW], nxt[CW];
    float s = 0.0f;
    auto words = [&](uint32_t (&d)[CW], int c) {  // words c .. c + 7, the last one past the record's end
#pragma unroll
        for (int u = 0; u < CW; ++u) d[u] = w[min(c + u, nw - 1)];
    };
    auto start = [&](int p) {  // key p's scale and first words (past hi: hi's)
        const uint8_t *rp = a.kq + slot_of(min(p, hi), a.cap) * (int64_t)(a.n_head_kv * rec) + (int64_t)kh * rec;
        w = (const uint32_t *)(rp + 4);
        s = *(const float *)rp;
        words(cur, 0);
    };
    int p = lo + kb * 256 + tid;
    start(p);
    if constexpr (R == 4) {
        rotate_wave(x, hd, false);
#pragma unroll
        for (int e = 0; e < KVQ_E; ++e) q[wave][lane + 64 * e] = x[e];  // past hd, and rows without a range: not used
    } else {
        for (int i = tid; i < R * hd; i += 256) {
            const int r = i / hd, x = i - r * hd;
            const KvqRow g = kvq_group_row(a, n_tok, R, grp, kh, r);
            q[r][x] = g.en >= g.st ? a.qr[(size_t)g.row * hd + x] : 0.0f;
        }
    }
    if (tid < 16) c4[tid] = kvq_centroid4(tid);
    __syncthreads();
    for (; p <= hi; p += nkb * 256) {
        float acc[R];
#pragma unroll
        for (int r = 0; r < R; ++r) acc[r] = 0.0f;
        for (int c = 0; c < nw; c += CW) {
            if (c + CW < nw) words(nxt, c + CW);
#pragma unroll
            for (int u = 0; u < CW; ++u) {
                if (c + u >= nw) break;  // uniform
                const uint32_t v = cur[u];
                if (a.kbits == 8) {
                    const int i = 4 * (c + u);
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        const float k = (float)(int8_t)(v >> (8 * j));
#pragma unroll
                        for (int r = 0; r < R; ++r) acc[r] = __builtin_fmaf(q[r][i + j], k, acc[r]);
                    }
                } else {
                    const int i = 8 * (c + u);
#pragma unroll
                    for (int j = 0; j < 8; j += 2) {
                        const float clo = c4[(v >> (4 * j)) & 15], chi = c4[(v >> (4 * j + 4)) & 15];
#pragma unroll
                        for (int r = 0; r < R; ++r)
                            acc[r] = acc[r] + __builtin_fmaf(q[r][i + j], clo, q[r][i + j + 1] * chi);
                    }
                }
            }
#pragma unroll
            for (int u = 0; u < CW; ++u) cur[u] = nxt[u];
        }
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const KvqRow g = rows[r];
            if (p >= g.st && p <= g.en) a.s[(size_t)g.row * a.max_len + (p - g.st)] = acc[r] * s * a.scale;
        }
        if (p + nkb * 256 <= hi) start(p + nkb * 256);
    }
}

// softmax_inplace over each row's scores, then each weight times its position's V scale. The sum is
// one ordered chain per row: about 5 cycles per position out of LDS. 1024 threads for few rows
// (decode: a CU holds one row), 256 for prompt batches.
constexpr int KVQ_RES = 12288;
template <int NT>
__global__ __launch_bounds__(NT) void kvq_softmax_kernel(KvqAttnArgs a, const float *scales) {
    extern __shared__ __attribute__((aligned(16))) float e[];  // min(max_len, KVQ_RES) values: rows up to that length stay in LDS
    __shared__ float red[NT / 64];
    __shared__ float total;
    const int row = blockIdx.x, tok = row / a.n_head, h = row - tok * a.n_head, tid = threadIdx.x;
    const int n = kvq_row_len(a, tok);
    if (n == 0) return;
    float *s = a.s + (size_t)row * a.max_len;
    const bool resident = n <= KVQ_RES;
    float mx = -__builtin_inff();
#pragma unroll 4
    for (int i = tid; i < n; i += NT) {
        const float x = s[i];
        if (resident) e[i] = x;
        mx = fmaxf(mx, x);
    }
    for (int o = 1; o < 64; o <<= 1) mx = fmaxf(mx, __shfl_xor(mx, o, 64));
    if ((tid & 63) == 0) red[tid >> 6] = mx;
    __syncthreads();
#pragma unroll
    for (int w = 0; w < NT / 64; ++w) mx = fmaxf(mx, red[w]);
    // decode rows: the first NT exponentials here, the others while wavefront 0 sums those (20.2 ->
    // 17.4 us, 32 rows of 4096 positions)
    const bool split = NT == 1024 && resident && n > NT;
    for (int i = tid; i < (split ? NT : n); i += NT) {
        if (resident) e[i] = expf_ref(e[i] - mx);
        else s[i] = expf_ref(s[i] - mx);
    }
    // the V scales of this thread's first positions, in flight while the sum runs; n <= cap: the ring
    // wraps at most once. scales: gathered by the launch before, [K / V head][slot]
    const int kvh = h / (a.n_head / a.n_head_kv), rec = 4 + a.hd * a.vbits / 8;
    const uint8_t *vr = scales ? (const uint8_t *)(scales + (int64_t)kvh * a.cap) : a.vq + (int64_t)kvh * rec;
    const int64_t stride = scales ? 4 : (int64_t)a.n_head_kv * rec;
    const int64_t s0 = slot_of(a.st[tok], a.cap);
    auto vscale = [&](int i) {
        const int64_t sl = s0 + i < a.cap ? s0 + i : s0 + i - a.cap;
        return *(const float *)(vr + sl * stride);
    };
    constexpr int PF = 4;
    float pf[PF];
#pragma unroll
    for (int k = 0; k < PF; ++k) pf[k] = vscale(min(tid + k * NT, n - 1));
    __syncthreads();
    float head = 0.0f;  // wavefront 0: the sum of the first NT
    if (split) {
        if (tid < 64) head = ordered_sum(e, NT, 0.0f);
        else
            for (int i = NT + tid - 64; i < n; i += NT - 64) e[i] = expf_ref(e[i] - mx);
        __syncthreads();
    }
    if (tid < 64) {
        float sum = head;
        int i = 0;
        if (resident) {
            const int from = split ? NT : 0, to = n & ~31;
            sum = ordered_sum(e + from, to - from, sum);
            for (i = to; i < n; ++i) sum += e[i];
        } else {  // 32 values loaded ahead of their adds
            for (; i + 32 <= n; i += 32) {
                float t[32];
#pragma unroll
                for (int u = 0; u < 32; ++u) t[u] = s[i + u];
#pragma unroll
                for (int u = 0; u < 32; ++u) sum += t[u];
            }
            for (; i < n; ++i) sum += s[i];
        }
        if (tid == 0) total = sum;
    }
    __syncthreads();
    const float sum = total, inv = 1.0f / sum;
    auto weigh = [&](int i, float sv) {
        const float ev = resident ? e[i] : s[i];
        const float w = sum > 0.0f ? ev * inv : ev;
        // kvq_axpy_v skips a zero weight (fastgguf.c:4829-4831): stored as 0, never 0 * s_V, so a V
        // record whose scale is inf or NaN adds nothing where the reference adds nothing
        s[i] = w == 0.0f ? 0.0f : w * sv;
    };
#pragma unroll
    for (int k = 0; k < PF; ++k)
        if (tid + k * NT < n) weigh(tid + k * NT, pf[k]);
    for (int i = tid + PF * NT; i < n; i += NT) weigh(i, vscale(i));
}

}  // namespace

hipError_t launch_kvq_store(const KvqStoreArgs &a, int n_tok, hipStream_t s) {
    if (n_tok < 1 || a.hd < 32 || a.hd > 256 || (a.hd & (a.hd - 1)) || (a.kbits != 4 && a.kbits != 8) ||
        (a.vbits != 2 && a.vbits != 4 && a.vbits != 8) || a.n_head_kv < 1 || a.n_head_kv > 65535)
        return hipErrorInvalidValue;
    kvq_store_kernel<<<dim3((unsigned)n_tok, (unsigned)a.n_head_kv, 2), 64, 0, s>>>(a, n_tok);
    return hipGetLastError();
}

hipError_t launch_kvq_attention(const KvqAttnArgs &a, int n_tok, hipStream_t s) {
    const int rows = n_tok * a.n_head;
    if (n_tok < 1 || a.hd < 32 || a.hd > 256 || (a.hd & (a.hd - 1)) || (a.kbits != 4 && a.kbits != 8) ||
        (a.vbits != 2 && a.vbits != 4 && a.vbits != 8) || a.n_head_kv < 1 || a.n_head % a.n_head_kv != 0 ||
        a.max_len < 1 || rows > 65535)
        return hipErrorInvalidValue;
    const int rows_kv = n_tok * (a.n_head / a.n_head_kv);
    const unsigned kb = (unsigned)std::min((a.max_len + 255) / 256, 1024);
    // prompt batches: every row reads its head's V scales, a cache line each out of the records. Those
    // of the rows' ranges are gathered once, into the scratch that the value chains fill later, where
    // that holds the ring's and the rows may read them 4 times and more (64 tokens, 32 heads, 4096
    // positions: the call 196.2 -> 186.3 us; 16 heads over 2, 1000 positions of 8-bit records 55.3 -> 52.6).
    float *scales = nullptr;
    if (rows_kv >= 16) {
        const int64_t ns = (int64_t)a.n_head_kv * a.cap;
        if (ns <= (int64_t)rows * a.hd && 4 * ns <= (int64_t)rows * a.max_len && ns <= 0x3fffffff) scales = a.orot;
        const KvqGather g{a, scales, n_tok, scales ? kvq_gather_wgs(a.cap, a.n_head_kv) : 0u};
        kvq_rotate_gather_kernel<<<g.wgs + (unsigned)((rows + 3) / 4), 256, 0, s>>>(g);
        kvq_scores_kernel<16><<<dim3((unsigned)a.n_head_kv, (unsigned)((rows_kv + 15) / 16), kb), 256, 0, s>>>(a, n_tok);
    } else
        kvq_scores_kernel<4><<<dim3(kb, (unsigned)((rows_kv + 3) / 4), (unsigned)a.n_head_kv), 256, 0, s>>>(a, n_tok);
    const size_t lds = (size_t)std::min(a.max_len, KVQ_RES) * 4;
    if (rows <= 256) kvq_softmax_kernel<1024><<<rows, 1024, lds, s>>>(a, scales);
    else kvq_softmax_kernel<256><<<rows, 256, lds, s>>>(a, scales);
    AttnArgs v{nullptr, a.orot, nullptr, nullptr, a.s, a.st, a.en, a.n_head, a.n_head_kv, a.hd,
               a.n_head_kv * a.hd, a.cap, a.max_len, 1.0f};
    v.vq = a.vq;  // the value chains decode the V records' codes themselves
    v.vbits = a.vbits;
    hipError_t e = launch_attention_values(v, n_tok, s);
    if (e != hipSuccess) return e;
    kvq_rotate_kernel<<<(rows + 3) / 4, 256, 0, s>>>(a.orot, a.o, a.hd, rows, true);
    return hipGetLastError();
}

}  // namespace fgh
