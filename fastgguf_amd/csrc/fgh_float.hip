// fgh_float.hip - the decode matvec for the float weight types F32, F16 and BF16 on fp32
// activations (dot_row fastgguf.c:2207-2214: dot_f32v 1618-1632, dot_f16_row 1645-1656 and the
// BF16 loop 2209-2213; the reference's own GPU path runs these types too, gpu_kernel_for 1745).
//
// Each row kernel runs C fp32 fma chains over the row, chain k over the values C j + k in order
// (no quantization of x), then sums the chains with a fixed tree and runs the last values one
// fma each:
//   F32:  C = 16 (dot_f32v's two 8-lane accumulators s0 = chains 0..7, s1 = chains 8..15), one
//         more 8-value group into s0 when 8 values remain, hsum_ps(s0 + s1), then the last n % 8
//         values (gcc's contraction of `s += a[i] * b[i]`)
//   F16:  C = 8, the values converted exactly (vcvtph2ps), hsum_ps, then the last n % 8 values
//   BF16: C = 1, one chain over the whole row (the value is its 16 bits above 16 zero bits)
// hsum_ps(v) = ((v0 + v4) + (v1 + v5)) + ((v2 + v6) + (v3 + v7)) (fastgguf.c:797-806).
//
// A wavefront holds one row tile, lane L = C r + k taking chain k of tile row r (64 / C rows per
// tile), and walks the row's steps in order through a ring of R 16-byte loads. A step is 1 KB:
// V = 16 / value bytes values per lane, lane L's values u = 0..V-1 of step s being the row's
// values C (V s + u) + k (tile layout below), so a step is V consecutive values of each chain.
// x is staged once per workgroup in LDS in the same order (value C (V s + u) + k at float
// (C s + k) V + u), so a lane reads its step's V activations with one or two 16-byte LDS reads
// (the rows of a wavefront read the same addresses). The last, partial step runs each value on
// the chain its position takes in the reference, and the lane of chain 0 runs the scalar tail
// from the tile in global memory after the tree. Rows are independent, and every row's fp32
// operations are the reference's, in its order: the outputs are bit-identical.
//
// BF16's one chain per row makes its launch latency-bound: about 11 ns per value of the row on
// MI355X (46 us at 4096 values) whatever the row count, against 9.9 us for F16 at 4096 x 4096.
//
// Tiles (upload, fl_relayout_kernel): step s of row tile t of matrix m at
// ((m * steps + s) * tiles per matrix + t) * 1 KB, lane L's 16 bytes at 16 L; values past the
// row's end and rows past the matrix's end are zeros (never on a chain).
#include <algorithm>
#include <type_traits>

#include "fgh_internal.h"

namespace fgh {

namespace {

template <int TYPE>
struct Fl {
    static constexpr int C = TYPE == T_F32 ? 16 : TYPE == T_F16 ? 8 : 1;  // chains per row
    static constexpr int V = TYPE == T_F32 ? 4 : 8;                      // values per lane and step
    static constexpr int CV = C * V;                                     // a row's values per step
    static constexpr int TR = 64 / C;                                    // rows per tile
};
static_assert(Fl<T_F32>::CV == fl_step_elems(T_F32) && Fl<T_F16>::CV == fl_step_elems(T_F16) &&
                  Fl<T_BF16>::CV == fl_step_elems(T_BF16),
              "step geometry");
static_assert(Fl<T_F32>::TR == fl_tile_rows(T_F32) && Fl<T_F16>::TR == fl_tile_rows(T_F16) &&
                  Fl<T_BF16>::TR == fl_tile_rows(T_BF16),
              "tile geometry");

// DPP row_shl:k, the value of lane + k within its 16-lane row (lanes without a source read 0)
__device__ __forceinline__ float shl(float v, int k) {
    const int iv = __builtin_bit_cast(int, v);
    int o;
    switch (k) {
    case 1: o = __builtin_amdgcn_update_dpp(0, iv, 0x101, 0xF, 0xF, true); break;
    case 2: o = __builtin_amdgcn_update_dpp(0, iv, 0x102, 0xF, 0xF, true); break;
    case 4: o = __builtin_amdgcn_update_dpp(0, iv, 0x104, 0xF, 0xF, true); break;
    default: o = __builtin_amdgcn_update_dpp(0, iv, 0x108, 0xF, 0xF, true); break;
    }
    return __builtin_bit_cast(float, o);
}

// a lane's 16 bytes of one step; live = false: zeros without a memory access
__device__ __forceinline__ uint4 fl_load(const uint8_t *step, uint32_t lane, bool live) {
    return bld16<WNT>(buf_res(step, live ? FL_TILE : 0), 16 * lane);
}

// value u of a lane's 16 bytes, as fp32 (each conversion exact)
template <int TYPE>
__device__ __forceinline__ float fl_val(const uint4 &w, int u) {
    const uint32_t d[4] = {w.x, w.y, w.z, w.w};
    if (TYPE == T_F32) return __builtin_bit_cast(float, d[u]);
    const uint32_t p = d[u >> 1];
    if (TYPE == T_BF16) return __builtin_bit_cast(float, (u & 1) ? p & 0xFFFF0000u : p << 16);
    return fp16_bits_to_f32((u & 1) ? p >> 16 : p & 0xFFFFu);
}
// one value of the row in the tile layout (the scalar tail), by its position e
template <int TYPE>
__device__ __forceinline__ float fl_val_at(const uint8_t *T0, size_t sstride, int r, int e) {
    using F = Fl<TYPE>;
    const int s = e / F::CV, rem = e - s * F::CV, u = rem / F::C, kk = rem - u * F::C;
    const uint8_t *p = T0 + (size_t)s * sstride + 16 * (F::C * r + kk) + fl_value_bytes(TYPE) * u;
    if (TYPE == T_F32) return *(const float *)p;
    const uint32_t h = *(const uint16_t *)p;
    return TYPE == T_BF16 ? __builtin_bit_cast(float, h << 16) : fp16_bits_to_f32(h);
}

// where value e of the row sits in the LDS copy of x (and in a lane's step: lane C r + kk, value u)
template <int TYPE>
__device__ __forceinline__ int fl_xpos(int e) {
    using F = Fl<TYPE>;
    const int s = e / F::CV, rem = e - s * F::CV, u = rem / F::C, kk = rem - u * F::C;
    return (s * F::C + kk) * F::V + u;
}

// is value u of chain k in step s on its chain (and not in the scalar tail or past the row)?
template <int TYPE>
__device__ __forceinline__ bool on_chain(int s, int u, int k, int n) {
    using F = Fl<TYPE>;
    const int j = F::V * s + u;  // the chain's j-th value: position C j + k
    if (TYPE == T_F32) return 16 * j + 16 <= n || (k < 8 && 16 * j + 8 <= n);
    if (TYPE == T_F16) return 8 * j + 8 <= n;
    return j < n;
}

__device__ __forceinline__ int fl_tensor_of(const MvArgs &a, int64_t g) {
    int ti = 0;
#pragma unroll
    for (int q = 1; q < 4; ++q)
        if (q < a.nt && g >= a.t[q].gfirst) ti = q;
    return ti;
}

}  // namespace

// Workgroup = TPW row tiles, one wavefront each; grid = (tiles over all tensors / TPW, token
// slots). a.nb = the row's values n, a.ntile = its steps.
template <int TYPE, int R, int TPW>
__global__ __launch_bounds__(64 * TPW) void fl_mv_kernel(MvArgs a) {
    using F = Fl<TYPE>;
    extern __shared__ __align__(16) uint8_t smem[];
    float *xs = (float *)smem;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int r = lane / F::C, k = lane - r * F::C;
    const int n = a.nb, nst = a.ntile;
    const int tok = blockIdx.y;
    const int64_t tile = (int64_t)blockIdx.x * TPW + wave;
    const bool live = tile < a.groups;
    const int64_t tc = live ? tile : a.groups - 1;
    const int ti = fl_tensor_of(a, tc);
    const uint32_t lt = (uint32_t)(tc - a.t[ti].gfirst), tpm = (uint32_t)a.t[ti].gpm;
    const uint32_t mi = (a.sel ? (uint32_t)a.sel[tok] : 0u) + lt / tpm, tt = lt % tpm;
    const size_t sstride = (size_t)tpm * FL_TILE;
    const uint8_t *T0 = a.t[ti].W + ((size_t)mi * nst * tpm + tt) * FL_TILE;

    // (1) the ring's first R steps, (2) x into LDS in the lanes' order while they load
    uint4 ring[R];
#pragma unroll
    for (int q = 0; q < R; ++q) ring[q] = fl_load(T0 + (size_t)min(q, nst - 1) * sstride, (uint32_t)lane, q < nst);
    const float *x = a.x + (size_t)(tok / a.xdiv) * a.ldx;
    const int npad = nst * F::CV;
    for (int e0 = tid; e0 < npad; e0 += 4 * 64 * TPW) {
        float v[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int e = e0 + q * 64 * TPW;
            v[q] = e < n ? x[e] : 0.0f;
        }
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int e = e0 + q * 64 * TPW;
            if (e < npad) xs[fl_xpos<TYPE>(e)] = v[q];
        }
    }
    __syncthreads();

    float acc = 0.0f;
    const int nwhole = n / F::CV;  // steps whose every value is on its chain (nst - 1 or nst)
    // the activations of step s from LDS (the last step's for s past it)
    auto xload = [&](int s, float (&xv)[8]) {
        const float4 *xp = (const float4 *)(xs + (size_t)(min(s, nst - 1) * F::C + k) * F::V);
        const float4 x0 = xp[0];
        xv[0] = x0.x, xv[1] = x0.y, xv[2] = x0.z, xv[3] = x0.w;
        if (F::V == 8) {
            const float4 x1 = xp[1];
            xv[4] = x1.x, xv[5] = x1.y, xv[6] = x1.z, xv[7] = x1.w;
        } else {
            xv[4] = xv[5] = xv[6] = xv[7] = 0.0f;
        }
    };
    // whole rounds of R whole steps, refilling the ring (a refill past the last step loads
    // nothing), straight-line code without a test; then the last steps (at most R, already in the
    // ring), each value tested against its chain. Step s's activations are in xb[s % XD], loaded
    // XD steps ahead (one step ahead left each step waiting for its LDS reads: BF16's one chain
    // ran 28 cycles per value).
    constexpr int XD = 4;
    static_assert(R % XD == 0, "the activation buffers rotate within a round");
    float xb[XD][8];
#pragma unroll
    for (int q = 0; q < XD; ++q) xload(q, xb[q]);
    int b0 = 0;
    for (; b0 + R <= nwhole; b0 += R) {
#pragma unroll
        for (int q = 0; q < R; ++q) {
#pragma unroll
            for (int u = 0; u < F::V; ++u) acc = __builtin_fmaf(fl_val<TYPE>(ring[q], u), xb[q % XD][u], acc);
            ring[q] = fl_load(T0 + (size_t)min(b0 + q + R, nst - 1) * sstride, (uint32_t)lane, b0 + q + R < nst);
            xload(b0 + q + XD, xb[q % XD]);
        }
    }
#pragma unroll
    for (int q = 0; q < R; ++q)
        if (b0 + q < nst) {  // uniform
            const int st = b0 + q;
#pragma unroll
            for (int u = 0; u < F::V; ++u)
                if (on_chain<TYPE>(st, u, k, n)) acc = __builtin_fmaf(fl_val<TYPE>(ring[q], u), xb[q % XD][u], acc);
            xload(st + XD, xb[q % XD]);
        }

    // the chains' tree (hsum_ps of s0 + s1 for F32, of the 8 chains for F16), then the scalar tail
    float res = acc;
    if (TYPE == T_F32) res = res + shl(res, 8);  // v_k = s0_k + s1_k
    if (TYPE != T_BF16) {
        res = res + shl(res, 4);  // (v_k + v_k+4), k < 4
        res = res + shl(res, 1);  // (v0 + v4) + (v1 + v5) at k = 0, the other pair at k = 2
        res = res + shl(res, 2);
    }
    const int64_t rows = a.t[ti].rows, row = (int64_t)tt * F::TR + r;
    if (live && k == 0 && row < rows) {
        if (TYPE != T_BF16) {
            const int t0 = TYPE == T_F32 ? 16 * (n / 16) + (n % 16 >= 8 ? 8 : 0) : 8 * (n / 8);
            for (int e = t0; e < n; ++e) res = __builtin_fmaf(fl_val_at<TYPE>(T0, sstride, r, e), xs[fl_xpos<TYPE>(e)], res);
        }
        a.t[ti].y[(size_t)tok * a.ldy + (int64_t)(lt / tpm) * rows + row] = res;
    }
}

// ---- upload: file rows -> tiles, one thread per destination 16 bytes ----
__global__ void fl_relayout_kernel(int type, const uint8_t *__restrict__ src, uint8_t *__restrict__ dst, int64_t rows,
                                   int64_t cols, int steps, int64_t gpm, int64_t units) {
    const int C = type == T_F32 ? 16 : type == T_F16 ? 8 : 1, V = type == T_F32 ? 4 : 8, TR = 64 / C;
    const int vb = fl_value_bytes(type);
    for (int64_t o = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; o < units; o += (int64_t)gridDim.x * blockDim.x) {
        const int64_t t = o >> 6;  // = (m * steps + s) * gpm + gl
        const int L = (int)(o & 63);
        const int64_t mt = t / gpm, gl = t - mt * gpm;
        const int64_t m = mt / steps;
        const int s = (int)(mt - m * steps);
        const int r = L / C, k = L - r * C;
        const int64_t row = gl * TR + r;
        uint8_t b[16];
#pragma unroll
        for (int q = 0; q < 16; ++q) b[q] = 0;
        if (row < rows)
            for (int u = 0; u < V; ++u) {
                const int64_t e = (int64_t)C * (V * s + u) + k;
                if (e < cols) {
                    const uint8_t *p = src + ((m * rows + row) * cols + e) * vb;
                    for (int q = 0; q < vb; ++q) b[vb * u + q] = p[q];
                }
            }
        uint4 w;
        __builtin_memcpy(&w, b, 16);
        ((uint4 *)dst)[o] = w;
    }
}

// ---- host side ----
size_t fl_lds_bytes(int type, int64_t cols) {
    const int64_t steps = (cols + fl_step_elems(type) - 1) / fl_step_elems(type);
    return (size_t)steps * fl_step_elems(type) * 4;
}
// One wavefront per tile (the chains are serial), a ring of 16 steps (16 KB in flight per
// wavefront). Tiles per workgroup: F16 4, BF16 2, F32 4 from 2 to 8 tiles per compute unit and 2
// otherwise. Measured (graph of back-to-back launches over >= 512 MB of copies, rings of 8, 16
// and 32 x 1, 2 and 4 tiles per workgroup, at 14336 x 4096, 4096 x 4096, 4096 x 14336 and
// 1024 x 4096): a ring of 16 was the fastest or within 2 % everywhere; F32 4096 x 4096 (1024
// tiles) 13.2 us with 4 tiles against 14.9 with 2, 14336 x 4096 (3584) 37.3 with 2 against 38.5,
// 1024 x 4096 (256) 8.3 with 2 against 9.2 and 10.5 with 1.
MvShape fl_matvec_shape(int type, int64_t tiles, int64_t cols, int num_cu) {
    const int tpw = type == T_F16    ? 4
                    : type == T_BF16 ? 2
                    : tiles >= 2 * (int64_t)num_cu && tiles <= 8 * (int64_t)num_cu ? 4
                                                                                   : 2;
    return MvShape{1, 16, tpw, fl_lds_bytes(type, cols)};
}

template <int TYPE, int R, int TPW>
static hipError_t fl_launch(const MvArgs &a, int ntok, size_t lds, hipStream_t s) {
    const unsigned wg = (unsigned)((a.groups + TPW - 1) / TPW);
    fl_mv_kernel<TYPE, R, TPW><<<dim3(wg, ntok), 64 * TPW, lds, s>>>(a);
    return hipGetLastError();
}
template <int TYPE, int R>
static hipError_t fl_launch_r(const MvShape &sh, const MvArgs &a, int ntok, hipStream_t s) {
    switch (sh.TPW) {
    case 4: return fl_launch<TYPE, R, 4>(a, ntok, sh.lds, s);
    case 2: return fl_launch<TYPE, R, 2>(a, ntok, sh.lds, s);
    default: return fl_launch<TYPE, R, 1>(a, ntok, sh.lds, s);
    }
}
template <int TYPE>
static hipError_t fl_launch_type(const MvArgs &a, int ntok, int num_cu, hipStream_t s) {
    const MvShape sh = fl_matvec_shape(TYPE, a.groups * ntok, a.nb, num_cu);
    if (sh.lds > GEMM_LDS_MAX || sh.R != 16) return hipErrorInvalidValue;
    return fl_launch_r<TYPE, 16>(sh, a, ntok, s);
}
hipError_t launch_fl_matvec(int type, const MvArgs &a, int ntok, int num_cu, hipStream_t s) {
    if (a.nb < 1 || a.ntile != (a.nb + fl_step_elems(type) - 1) / fl_step_elems(type) || a.dump_s)
        return hipErrorInvalidValue;
    switch (type) {
    case T_F32: return fl_launch_type<T_F32>(a, ntok, num_cu, s);
    case T_F16: return fl_launch_type<T_F16>(a, ntok, num_cu, s);
    case T_BF16: return fl_launch_type<T_BF16>(a, ntok, num_cu, s);
    default: return hipErrorInvalidValue;
    }
}
hipError_t launch_fl_relayout(int type, const uint8_t *src, uint8_t *dst, int64_t rows, int64_t cols, int steps,
                              int64_t gpm, int64_t total, hipStream_t s) {
    if (!fl_kind(type) || total % 16) return hipErrorInvalidValue;
    const int64_t units = total / 16, want = (units + 255) / 256;
    const unsigned grid = (unsigned)(want < 65536 ? want : 65536);
    fl_relayout_kernel<<<grid, 256, 0, s>>>(type, src, dst, rows, cols, steps, gpm, units);
    return hipGetLastError();
}

// ---- several tokens (matmul): the same chains on fp32 MFMAs of K = 1 ----
// The reference multiplies float matrices token by token (matmul, fastgguf.c:3004-3017), each chain
// an ordered run of fmas. v_mfma_f32_*x1 adds one product to every sum of its tile, each as one
// fmaf (subnormals, infinities and NaN included), so a chain of rank-1
// updates over the values in order is the reference's chain for 16 rows x 16 tokens at once.
// F32 / F16: v_mfma_f32_16x16x1 with its 4 blocks as 4 chains: lane 16 b + i of A holds row i's
// value of chain 4 h + b, lane 16 b + t of B token t's activation; a lane then holds all chains of
// 4 rows x 1 token, so the final tree needs no exchange. BF16 has one chain per row: A = tokens
// (one register holds 4 positions x 16 tokens, the position's block broadcast), B = 64 rows.
// Workgroup = 4 wavefronts on 4 row tiles, sharing stages of 4096 activations in LDS (NT groups of 16
// tokens x 4 / NT steps of 64 values), loaded a stage ahead; grid.y = chunks of NT groups.
// Counters, 64 tokens: F32 and F16 14336 x 2048 (70 and 52 us) keep the matrix pipe busy for 57 k cycles a SIMD,
// about 27 us; their wavefronts wait to issue for 52 and 62 % of their lives (half of the LDS cycles are bank
// conflicts, but the LDS is active for a sixth of the time). BF16 4096 x 4096 (107 us): one
// dependent MFMA per value, 62 cycles each.
typedef float fm4 __attribute__((ext_vector_type(4)));
typedef float fm4u __attribute__((ext_vector_type(4), aligned(4)));
typedef float fm16 __attribute__((ext_vector_type(16)));

struct FlMmArgs {
    const uint8_t *W;
    const float *X;
    float *Y;
    int64_t rows, gpm, ldx, ldy;  // rows and tiles per matrix
    int n, nst, T;                // values per row, steps, tokens
    uint32_t wpm;                 // wavefront tiles per matrix
    int64_t groups;               // wavefront tiles
    uint32_t xbytes;              // X up to its last value (below 2 GiB)
};

// NT groups of 16 tokens per wavefront, SB steps of 64 values per stage (NT SB = 4: 16 KB)
template <int TYPE, int NT>
__global__ __launch_bounds__(256, NT == 4 ? 1 : 2) void fl_mm_kernel(FlMmArgs a) {
    using F = Fl<TYPE>;
    constexpr int SB = 4 / NT, HN = F::C / 4, VQ = F::V / 4, R = TYPE == T_F32 ? 4 : 8, TW = 16 / F::TR;
    static_assert(F::CV == 64 && R % SB == 0, "stage geometry");
    __shared__ __attribute__((aligned(16))) float xs[2][4096];  // [step][group][h][u / 4][lane][u % 4]
    const int tid = threadIdx.x, l = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int n = a.n, nst = a.nst, tok0 = (int)blockIdx.y * 16 * NT;
    const int64_t wt = (int64_t)blockIdx.x * 4 + wave;
    const bool live = wt < a.groups;
    const uint32_t tc = (uint32_t)(live ? wt : a.groups - 1), mi = (uint32_t)__builtin_amdgcn_readfirstlane((int)(tc / a.wpm)), wl = tc - mi * a.wpm;
    const int b = l >> 4, i = l & 15;
    // A: row i of the wavefront's 16 rows: row i % TR of tile TW wl + i / TR
    const uint32_t tile = wl * TW + (uint32_t)(i / F::TR);
    const bool rlive = live && tile < (uint32_t)a.gpm;
    const size_t sstride = (size_t)a.gpm * FL_TILE;
    const uint8_t *M0 = a.W + (size_t)mi * nst * sstride;  // the matrix
    // a lane whose tile does not exist reads past the buffer's end: zeros, no access
    const uint32_t off = rlive ? tile * FL_TILE + 16 * (F::C * (i % F::TR) + b) : 0x80000000u;
    auto wload = [&](int s, uint4 (&w)[HN]) {
        const BufRes r = buf_res(M0 + (size_t)min(s, nst - 1) * sstride, live && s < nst ? (uint32_t)sstride : 0u);
#pragma unroll
        for (int h = 0; h < HN; ++h) w[h] = bld16(r, off + 64 * h);
    };
    uint4 ring[R][HN];
#pragma unroll
    for (int q = 0; q < R; ++q) wload(q, ring[q]);
    // activations: thread (t, q) takes values 4 q .. + 3 of token t of each group and step
    const int xt = tid >> 4, xq = tid & 15;
    fm4 xr[4];
    // one buffer over all tokens; a quad that is not whole lies past the chains (the scalar tail reads
    // X itself) and, like one past the row, is out of the buffer's range: zeros, no access, no branch
    const BufRes xb = buf_res((const uint8_t *)a.X, a.xbytes);
    auto xload = [&](int st) {  // stage st: steps SB st .. + SB - 1
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int s = SB * st + j / NT, tok = min(tok0 + 16 * (j % NT) + xt, a.T - 1), e = 64 * s + 4 * xq;
            const uint4 v = bld16(xb, e + 4 <= n ? 4u * ((uint32_t)tok * (uint32_t)a.ldx + (uint32_t)e) : 0x80000000u);
            xr[j] = (fm4){__uint_as_float(v.x), __uint_as_float(v.y), __uint_as_float(v.z), __uint_as_float(v.w)};
        }
    };
    auto xstore = [&](int st) {
        float *d = xs[st & 1];
        const int k0 = (4 * xq) % F::C, u = (4 * xq) / F::C;  // 4 adjacent chains of value u
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
            for (int c = 0; c < 4; ++c)
                d[(((j * HN) + (k0 >> 2)) * VQ + (u >> 2)) * 256 + (16 * c + xt) * 4 + (u & 3)] = xr[j][c];
    };
    fm16 acc[NT][HN];
#pragma unroll
    for (int g = 0; g < NT; ++g)
#pragma unroll
        for (int h = 0; h < HN; ++h)
#pragma unroll
            for (int e = 0; e < 16; ++e) acc[g][h][e] = 0.0f;
    const int nstage = (nst + SB - 1) / SB;
    xload(0);
    xstore(0);
    if (nstage > 1) xload(1);
    lds_barrier();
    // a step: its activations read, its weights converted (each into a register of its own: an MFMA in
    // flight holds its operands), then the MFMAs; all: every value of the step is on its chain
    auto step = [&](auto all, int s0, int q, uint4 (&w)[HN]) {  // step s0 + q, s0 a multiple of R
        constexpr bool whole = decltype(all)::value;
        const int s = s0 + q;
        const float *x = xs[(s / SB) & 1] + (size_t)(q % SB) * NT * HN * VQ * 256 + 4 * l;
        if (q % SB == 0) {  // a new stage
            if (s / SB + 1 < nstage) xstore(s / SB + 1);
            xload(min(s / SB + 2, nstage - 1));
        }
        fm4 xv[NT][HN][VQ];
#pragma unroll
        for (int g = 0; g < NT; ++g)
#pragma unroll
            for (int h = 0; h < HN; ++h)
#pragma unroll
                for (int q = 0; q < VQ; ++q) xv[g][h][q] = *(const fm4 *)(x + ((g * HN + h) * VQ + q) * 256);
        float wv[HN][F::V];
#pragma unroll
        for (int h = 0; h < HN; ++h)
#pragma unroll
            for (int u = 0; u < F::V; ++u) wv[h][u] = fl_val<TYPE>(w[h], u);
        wload(s + R, w);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int u = 0; u < F::V; ++u)
#pragma unroll
            for (int h = 0; h < HN; ++h)
                if (whole || on_chain<TYPE>(s, u, 4 * h, n)) {  // the 4 chains of h agree
#pragma unroll
                    for (int g = 0; g < NT; ++g)
                        acc[g][h] = __builtin_amdgcn_mfma_f32_16x16x1f32(wv[h][u], xv[g][h][u >> 2][u & 3], acc[g][h], 0, 0, 0);
                }
        if (q % SB == SB - 1) lds_barrier();
        __builtin_amdgcn_sched_barrier(0);
    };
    int s0 = 0;
    for (; 64 * (s0 + R) <= n; s0 += R) {  // whole rounds: straight-line code
#pragma unroll
        for (int q = 0; q < R; ++q) step(std::true_type{}, s0, q, ring[q]);
    }
#pragma unroll
    for (int q = 0; q < R; ++q)
        if (s0 + q < nst) step(std::false_type{}, s0, q, ring[q]);  // uniform over the workgroup
    // lane (q, t): rows 4 q + r, token t; register 4 b + r of acc[.][h] is chain 4 h + b
#pragma unroll
    for (int g = 0; g < NT; ++g) {
        const int tok = tok0 + 16 * g + i;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            float v[8];
#pragma unroll
            for (int k = 0; k < 8; ++k) {
                v[k] = acc[g][k >> 2][4 * (k & 3) + r];
                if constexpr (TYPE == T_F32) v[k] = v[k] + acc[g][2 + (k >> 2)][4 * (k & 3) + r];  // s0_k + s1_k
            }
            float y = ((v[0] + v[4]) + (v[1] + v[5])) + ((v[2] + v[6]) + (v[3] + v[7]));
            const int64_t row = (int64_t)wl * 16 + 4 * b + r;
            if (live && row < a.rows && tok < a.T) {
                const int t0 = TYPE == T_F32 ? 16 * (n / 16) + (n % 16 >= 8 ? 8 : 0) : 8 * (n / 8);
                const uint8_t *T0 = M0 + (size_t)(row / F::TR) * FL_TILE;
                for (int e = t0; e < n; ++e)
                    y = __builtin_fmaf(fl_val_at<TYPE>(T0, sstride, (int)(row % F::TR), e), a.X[(size_t)tok * a.ldx + e], y);
                a.Y[(size_t)tok * a.ldy + (int64_t)mi * a.rows + row] = y;
            }
        }
    }
}

// BF16: a wavefront holds 64 rows (lane = row: the decode tile) x 16 tokens, stages of 128 values of
// the tokens in LDS ([value / 4][lane]: lane 16 c + t of an A register is position 4 q + c of token t)
__global__ __launch_bounds__(256) void fl_mm_bf16_kernel(FlMmArgs a) {
    using F = Fl<T_BF16>;
    constexpr int SV = 128, SS = SV / F::CV, R = 16, TB = 16;  // values and steps per stage, ring, tokens
    static_assert(R == SS, "a ring round is a stage");
    __shared__ __attribute__((aligned(16))) float xs[2][SV * TB];
    const int tid = threadIdx.x, l = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int n = a.n, nst = a.nst, tok0 = (int)blockIdx.y * TB;
    const int64_t wt = (int64_t)blockIdx.x * 4 + wave;
    const bool live = wt < a.groups;
    const uint32_t tc = (uint32_t)(live ? wt : a.groups - 1), mi = (uint32_t)__builtin_amdgcn_readfirstlane((int)(tc / a.wpm)), wl = tc - mi * a.wpm;
    const size_t sstride = (size_t)a.gpm * FL_TILE;
    const uint8_t *T0 = a.W + (size_t)mi * nst * sstride + (size_t)wl * FL_TILE;
    const int nstage = (n + SV - 1) / SV;
    uint4 ring[R];
#pragma unroll
    for (int q = 0; q < R; ++q) ring[q] = fl_load(T0 + (size_t)min(q, nst - 1) * sstride, (uint32_t)l, live && q < nst);
    const BufRes xb = buf_res((const uint8_t *)a.X, a.xbytes);  // past the row: out of range, zeros
    fm4 xr[2];  // thread (t, q): values 4 q .. + 3 of tokens t and t + 8
    auto xload = [&](int st) {
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const int t = (tid >> 5) + 8 * j, e = SV * st + 4 * (tid & 31);
            const uint32_t o = 4u * ((uint32_t)min(tok0 + t, a.T - 1) * (uint32_t)a.ldx + (uint32_t)e);
            if (n % 4 == 0 || st + 1 < nstage) {  // uniform: whole quads
                const uint4 v = bld16(xb, e < n ? o : 0x80000000u);
                xr[j] = (fm4){__uint_as_float(v.x), __uint_as_float(v.y), __uint_as_float(v.z), __uint_as_float(v.w)};
            } else {
#pragma unroll
                for (int c = 0; c < 4; ++c)
                    xr[j][c] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(xb, e + c < n ? (int)(o + 4 * c) : (int)0x80000000u, 0, 0));
            }
        }
    };
    auto xstore = [&](int st) {
        float *d = xs[st & 1] + 64 * (tid & 31) + (tid >> 5);
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int c = 0; c < 4; ++c) d[16 * c + 8 * j] = xr[j][c];
    };
    fm16 acc;
#pragma unroll
    for (int e = 0; e < 16; ++e) acc[e] = 0.0f;
    xload(0);
    xstore(0);
    if (nstage > 1) xload(1);
    lds_barrier();
    auto run = [&](auto all, int st) {  // a stage; all: every value of it exists (no test per value)
        constexpr bool whole = decltype(all)::value;
        if (st + 1 < nstage) xstore(st + 1);
        xload(min(st + 2, nstage - 1));
        const float *x = xs[st & 1] + l;
        const int cnt = min(SV, n - st * SV);
#pragma unroll
        for (int q = 0; q < SS; ++q) {
            // the step's operands in registers of their own, then its MFMAs
            float w[8];
#pragma unroll
            for (int u = 0; u < 8; ++u) w[u] = fl_val<T_BF16>(ring[q], u);
            const float x0 = x[64 * (2 * q)], x1 = x[64 * (2 * q + 1)];
            const int s = SS * st + q;
            ring[q] = fl_load(T0 + (size_t)min(s + R, nst - 1) * sstride, (uint32_t)l, live && s + R < nst);
            __builtin_amdgcn_sched_barrier(0);
#define FL_B(u, X, J) \
    if (whole || 8 * q + u < cnt) acc = __builtin_amdgcn_mfma_f32_16x16x1f32(X, w[u], acc, 2, J, 0);
            FL_B(0, x0, 0) FL_B(1, x0, 1) FL_B(2, x0, 2) FL_B(3, x0, 3)
            FL_B(4, x1, 0) FL_B(5, x1, 1) FL_B(6, x1, 2) FL_B(7, x1, 3)
#undef FL_B
        }
        lds_barrier();
    };
    int st = 0;
    for (; SV * (st + 1) <= n; ++st) run(std::true_type{}, st);
    if (st < nstage) run(std::false_type{}, st);
    // register 4 b + r: token 4 (l / 16) + r of row 16 b + l % 16
#pragma unroll
    for (int e = 0; e < 16; ++e) {
        const int tok = tok0 + 4 * (l >> 4) + (e & 3);
        const int64_t row = (int64_t)wl * 64 + 16 * (e >> 2) + (l & 15);
        if (live && row < a.rows && tok < a.T) a.Y[(size_t)tok * a.ldy + (int64_t)mi * a.rows + row] = acc[e];
    }
}

// groups of 16 tokens per wavefront: the most that still fill the compute units; F32's 16 chains
// leave room for one
static int fl_mm_nt(int type, int64_t groups, int tg, int num_cu) {
    int nt = type != T_F16 ? 1 : tg >= 3 ? 4 : tg;
    while (nt > 1 && (groups + 3) / 4 * ((tg + nt - 1) / nt) < num_cu * 3 / 4) nt >>= 1;
    return nt;
}
// Whether these kernels take less time than the per-token decode launches: both sides from what they
// measured on MI355X (us; 1012 calls a type: 59 shapes from 256 x 256 to 11008 x 4096, 151936 x 128 and
// 602 x 12608, 2..64 tokens). The decode launches take a wavefront per tile and token: a part per tile, the
// scalar tail, and one per value that grows with what an XCD's L2 meets of the matrix, up to 2 MiB and again
// to 8 (F16 3120 x 4192, 98 workgroups a token: 16 tokens 55.8; 4096 x 4096, 128 of them: 38.4). These walk a
// row in one wavefront: rounds of one per SIMD.
//                        decode -> these   rule           decode -> these   rule
//   F32   640 x 2048   40  15.6   20.0  decode
//   F32   512 x 4096   40  22.0   34.5  decode
//   F32  4096 x 4096    4  33.0   35.9  decode      8  65.2   36.0  these
//   F32 14336 x 2048                                64 991.1   69.9  these
//   F16  3072 x 3072   14  18.2   22.9  decode     24  25.2   22.8  these
//   F16 14336 x 2048                                64 379.4   50.2  these
//   BF16 4096 x 4096   48 100.2  107.1  decode     64 139.2  107.4  these
//   BF16 14336 x 2048   8  39.3   56.9  decode     64 291.8   56.8  these
// In three of those calls it picks these kernels where they are 3 % slower, in none more; in 36 it keeps
// decode launches that are 8 to 43 % slower (BF16 16400 x 1024 at 8 tokens the most).
bool fl_matmul_pays(int type, int64_t rows, int n, int T, int num_cu) {
    struct Fit {
        double base, chain, tile, value, l2, far, tail;  // chain, value, l2, far: per 1000 values of a row
    };
    const Fit f = type == T_F32   ? Fit{2.8, 0.08, 0.711, 0.333, 0.52, 0.78, 0.57}
                  : type == T_F16 ? Fit{2.6, 1.4, 0.57, 0.35, 0.12, 0.78, 0.5}
                                  : Fit{2.85, 0.8, 1.0, 2.8, 1.6, 7.27, 0.1};
    const double simds = 4.0 * num_cu, k = n / 1000.0;
    const int64_t tiles = (rows + fl_tile_rows(type) - 1) / fl_tile_rows(type);
    const int tpw = fl_matvec_shape(type, tiles * T, n, num_cu).TPW;
    const double mib = decode_l2_mib((double)rows * n * (type == T_F32 ? 4 : 2), (tiles + tpw - 1) / tpw);
    const double value = f.value + f.l2 * std::min(mib, 2.0) / 2 + f.far * (std::min(std::max(mib, 2.0), 8.0) - 2) / 6;
    const double before = f.base + f.chain * k + tiles * T / simds * (value * k + f.tile + (n % 8 ? f.tail : 0.0));
    const int tg = (T + 15) / 16;
    const int64_t groups = (rows + (type == T_BF16 ? 63 : 15)) / (type == T_BF16 ? 64 : 16);
    const int nt = fl_mm_nt(type, groups, tg, num_cu);
    const double rounds = (double)((groups * ((tg + nt - 1) / nt) + 4 * num_cu - 1) / (4 * num_cu));
    if (type == T_BF16) return before > 3 + rounds * (1 + 0.0258 * n);
    return before > 3 + rounds * (1 + (type == T_F32 ? 0.48 : 0.375 * nt) * ((n + 63) / 64)) + (n % 8 ? 2.5 : 0.0);
}
template <int TYPE>
static hipError_t fl_mm_launch(const FlMmArgs &a, int num_cu, hipStream_t s) {
    const int tg = (a.T + 15) / 16, nt = fl_mm_nt(TYPE, a.groups, tg, num_cu);
    const dim3 g((unsigned)((a.groups + 3) / 4), (unsigned)((tg + nt - 1) / nt));
    if constexpr (TYPE != T_F32) {
        if (nt == 4) fl_mm_kernel<TYPE, 4><<<g, 256, 0, s>>>(a);
        if (nt == 2) fl_mm_kernel<TYPE, 2><<<g, 256, 0, s>>>(a);
    }
    if (nt == 1) fl_mm_kernel<TYPE, 1><<<g, 256, 0, s>>>(a);
    return hipGetLastError();
}
hipError_t launch_fl_matmul(int type, const RowgArgs &r, int num_cu, hipStream_t s) {
    if (!fl_kind(type) || r.nb < 1 || r.T < 1 || r.T > 64 || r.groups < 1 || r.gpm < 1 || r.groups % r.gpm != 0 ||
        r.gpm * fl_tile_rows(type) < r.rows || !r.W || !r.X || !r.Y)
        return hipErrorInvalidValue;
    const int64_t mats = r.groups / r.gpm;
    const int tw = type == T_BF16 ? 1 : 16 / fl_tile_rows(type);
    FlMmArgs a{r.W, r.X, r.Y, r.rows, r.gpm, r.ldx, r.ldy, r.nb, (r.nb + fl_step_elems(type) - 1) / fl_step_elems(type), r.T,
               (uint32_t)((r.gpm + tw - 1) / tw), 0, 0};
    a.groups = mats * a.wpm;
    const int64_t xb = 4 * ((r.T - 1) * r.ldx + r.nb);
    if (xb > 0x7fffffff) return hipErrorInvalidValue;
    a.xbytes = (uint32_t)xb;
    if ((a.groups + 3) / 4 > 0x7fffffff || r.gpm * FL_TILE > 0x7fffffff) return hipErrorInvalidValue;
    if (type == T_F32) return fl_mm_launch<T_F32>(a, num_cu, s);
    if (type == T_F16) return fl_mm_launch<T_F16>(a, num_cu, s);
    const unsigned wg = (unsigned)((a.groups + 3) / 4);
    fl_mm_bf16_kernel<<<dim3(wg, (unsigned)((a.T + 15) / 16)), 256, 0, s>>>(a);
    return hipGetLastError();
}

}  // namespace fgh
