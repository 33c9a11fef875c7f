// ts_proj.hip -- the attention output projection with the residual add, for gfx950 (f16
// weights).
//
// Replaces main_attn_proj (src/backend/bindless/sh_layer_v1.wgsl:763-821, F16 branch
// :777-781): for every token, dot = Wo a over attn_dim = n_head * head_dim inputs (the
// attention output after the split-K combine), stashed raw when asked (the reference keeps it
// for Gemma-2's post-attention norm, :812-815), and added to the residual stream:
// act = act + dot (:818-820).  Same matrix-core loops as the QKV projection (ts_gemm.h):
//   * enough 64-row tiles: one workgroup per 64 x 256 tile over all of attn_dim, the result
//     added to act straight from the accumulators;
//   * one or two rows: ts_gemv.h, one kernel;
//   * few tiles (decode): 32 x 256 tiles with attn_dim split across workgroups (f32
//     partials), then a kernel that sums the partials in split order and adds them to act.
// Taking the combine's output rather than the decode partials is deliberate: every column
// tile reads all of a token's attention output, so folding the combine into this kernel would
// redo it (n_split-fold reads of the partials) once per column tile.
#include "ts_gemm.h"
#include "ts_gemv.h"
#include "ts_internal.h"
#include "ts_kquant.h"

namespace ts {
namespace {

constexpr int kPT = 256;        // columns per tile
constexpr int kMaxPSplit = kKqMaxSplit;  // most splits of the reduction

struct ProjArgs {
    const float *a;      // [M][K] attention output
    const _Float16 *w;   // [N][K]
    const uint8_t *bw;   // the same rows as GGUF K-quant blocks (the K-quant kernel)
    size_t brow;         // bytes of one block row
    float *act;          // [M][N], += dot
    float *stash;        // [M][N] raw dot, or null
    float *part;         // [n_split][RT][CT][32][256] partials, or null
    int M, N, K;
    int KW;              // weight row length: K (f16 rows) or 2 K (hi then lo planes)
    int RT, CT, kps, n_split, n_wg;
};

__device__ inline void proj_tile_of(const ProjArgs &p, int id, int &rt, int &ct, int &sp) {
    const int per = (p.n_wg + 7) / 8;
    const int lin = (id % 8) * per + id / 8;  // a contiguous run of column tiles per XCD
    rt = lin % p.RT;
    ct = (lin / p.RT) % p.CT;
    sp = lin / (p.RT * p.CT);
}

// 64-row tiles over all of K; the epilogue from the accumulators.  The residuals of a 32 x 32
// block are loaded together before any of them is used (one by one, each a trip to memory, they
// took as long as the whole product of a 96-long reduction: 51 us of 2048 x 6144 outputs).
// T: 0 for f16 rows (4 waves of 64 columns), else the GGUF block type (8 waves of 32).
template <int T>
__global__ __launch_bounds__(T == 0 ? 256 : 512, 2) void proj_tile_kernel(ProjArgs p) {
    constexpr int CB = T == 0 ? 2 : 1;
    __shared__ __align__(16) std::conditional_t<T == 0, GemmTiles, KqRowTiles> sm;
    int rt, ct, sp;
    proj_tile_of(p, blockIdx.x, rt, ct, sp);
    if (sp >= 1) return;
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, j = lane & 31, hf = lane >> 5;
    const int row0 = 64 * rt, col0 = kPT * ct;
    floatx16 acc[2][CB];
    if constexpr (T == 0) {
        const int si = tid >> 2, sc = tid & 3;
        const _Float16 *ws[4];
#pragma unroll
        for (int i = 0; i < 4; i++) ws[i] = p.w + (size_t)min(col0 + si + 64 * i, p.N - 1) * p.KW + tile_k(sc);
        gemm_tile_core(sm, p.a + (size_t)min(row0 + si, p.M - 1) * p.K + tile_k(sc), ws, p.KW / kTK, p.K / kTK, tid, acc);
    } else {
        floatx16 c[2];
        gemm_tile_blocks<T>(sm, p.a + (size_t)min(row0 + (tid >> 3), p.M - 1) * p.K + 8 * (tid & 7),
                            p.bw + (size_t)min(col0 + 32 * wave + j, p.N - 1) * p.brow, p.K / 256, tid, c);
        acc[0][0] = c[0];
        acc[1][0] = c[1];
    }
#pragma unroll
    for (int rb = 0; rb < 2; rb++)
#pragma unroll
        for (int cb = 0; cb < CB; cb++) {
            const int col = col0 + 32 * (CB * wave + cb) + j;
            const int r0 = row0 + 32 * rb + 4 * hf;
            float res[16];
#pragma unroll
            for (int e = 0; e < 16; e++)
                res[e] = p.act[(size_t)min(r0 + 8 * (e >> 2) + (e & 3), p.M - 1) * p.N + min(col, p.N - 1)];
#pragma unroll
            for (int e = 0; e < 16; e++) {
                const int row = r0 + 8 * (e >> 2) + (e & 3);
                if (row >= p.M || col >= p.N) continue;
                const size_t i = (size_t)row * p.N + col;
                if (p.stash) p.stash[i] = acc[rb][cb][e];
                p.act[i] = res[e] + acc[rb][cb][e];
            }
        }
}

// One split of the reduction on a 32-row tile; the partial to the scratch buffer.
__global__ __launch_bounds__(256) void proj_split_kernel(ProjArgs p) {
    __shared__ __align__(16) SplitTiles sm;
    int rt, ct, sp;
    proj_tile_of(p, blockIdx.x, rt, ct, sp);
    if (sp >= p.n_split) return;
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, j = lane & 31, hf = lane >> 5;
    const int row0 = 32 * rt, col0 = kPT * ct + 64 * wave;
    const int kb = sp * p.kps;
    const int nbat = (min(kb + p.kps, p.KW) - kb) / (4 * kKC);
    const int si = tid >> 3, sc = tid & 7;
    const float *xs = row0 + si < p.M ? p.a + (size_t)(row0 + si) * p.K + 8 * sc : nullptr;
    const _Float16 *const wp[2] = {p.w + (size_t)min(col0 + j, p.N - 1) * p.KW + kb + 32 * hf,
                                   p.w + (size_t)min(col0 + 32 + j, p.N - 1) * p.KW + kb + 32 * hf};
    floatx16 acc[2];
    gemm_split_core(sm, xs, kb / kKC, p.K / kKC, wp, nbat, tid, acc);
    float *dst = p.part + (((size_t)sp * p.RT + rt) * p.CT + ct) * (32 * kPT);
#pragma unroll
    for (int cb = 0; cb < 2; cb++)
#pragma unroll
        for (int e = 0; e < 16; e++)
            dst[(8 * (e >> 2) + 4 * hf + (e & 3)) * kPT + 64 * wave + 32 * cb + j] = acc[cb][e];
}

// The same with the weights as GGUF K-quant blocks read in the loop (gemm_split_kq); slices of
// whole super-blocks, one slice where 256 tiles or more do not take the tile kernel (kq_tiles, or an
// output that shares memory with the input).
template <int T>
__global__ __launch_bounds__(256) void proj_split_kq_kernel(ProjArgs p) {
    __shared__ __align__(16) KqTiles sm[2];
    int rt, ct, sp;
    proj_tile_of(p, blockIdx.x, rt, ct, sp);
    if (sp >= p.n_split) return;
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, j = lane & 31, hf = lane >> 5;
    const int row0 = 32 * rt, col0 = kPT * ct + 64 * wave;
    const int kb = sp * p.kps;
    const int nbat = (min(kb + p.kps, p.K) - kb) / 256;
    const int si = tid >> 3, sc = tid & 7;
    const float *xs = row0 + si < p.M ? p.a + (size_t)(row0 + si) * p.K + kb + 8 * sc : nullptr;
    const size_t boff = (size_t)(kb / 256) * KQ<T>::BYTES;
    const uint8_t *const wb[2] = {p.bw + (size_t)min(col0 + j, p.N - 1) * p.brow + boff,
                                  p.bw + (size_t)min(col0 + 32 + j, p.N - 1) * p.brow + boff};
    floatx16 acc[2];
    gemm_split_blocks<T>(sm, xs, wb, nbat, tid, acc);
    float *dst = p.part + (((size_t)sp * p.RT + rt) * p.CT + ct) * (32 * kPT);
#pragma unroll
    for (int cb = 0; cb < 2; cb++)
#pragma unroll
        for (int e = 0; e < 16; e++)
            dst[(8 * (e >> 2) + 4 * hf + (e & 3)) * kPT + 64 * wave + 32 * cb + j] = acc[cb][e];
}

// One or two rows (decode): 8 R output columns per workgroup, complete in one kernel (ts_gemv.h).
template <int T, int MB, int R>
__global__ __launch_bounds__(256) void proj_gemv_kernel(ProjArgs p) {
    extern __shared__ __align__(16) float sx[];
    __shared__ float red[4 * 8 * R * MB];
    const int tid = threadIdx.x, g = (tid & 63) >> 3;
    const int n0 = (blockIdx.x * 8 + g) * R;
    const uint8_t *row[R];
    float res[R][MB], out[R][MB];
#pragma unroll
    for (int r = 0; r < R; r++) {
        const int n = min(n0 + r, p.N - 1);
        if constexpr (T == kGemvF16 || T == kGemvF16x2)
            row[r] = reinterpret_cast<const uint8_t *>(p.w + (size_t)n * p.KW);
        else
            row[r] = p.bw + (size_t)n * p.brow;
#pragma unroll
        for (int m = 0; m < MB; m++) res[r][m] = tid < 64 ? p.act[(size_t)min(m, p.M - 1) * p.N + n] : 0.0f;
    }
    gemv_rows<T, MB, R>(sx, red, p.a, p.M, p.K, p.K, row, (size_t)p.K * 2, tid, out);
    if (tid >= 64 || (tid & 7)) return;
#pragma unroll
    for (int r = 0; r < R; r++)
#pragma unroll
        for (int m = 0; m < MB; m++) {
            if (n0 + r >= p.N || m >= p.M) continue;
            const size_t i = (size_t)m * p.N + n0 + r;
            if (p.stash) p.stash[i] = out[r][m];
            p.act[i] = res[r][m] + out[r][m];
        }
}

// Sum of the partials of NR rows of one tile in split order, added to act.
constexpr int kPRows = 4;  // rows per workgroup of the sum (4 vs 8: config 3 14.1 vs 15.0 us, config 2 11.5 vs 12.2)
__global__ __launch_bounds__(256) void proj_reduce_kernel(ProjArgs p) {
    constexpr int NR = kPRows;
    __shared__ __align__(16) float tile[NR][kPT + 4];
    const int tix = blockIdx.x / (32 / NR), r0 = (blockIdx.x % (32 / NR)) * NR;
    const int rt = tix % p.RT, ct = tix / p.RT;
    if (32 * rt + r0 >= p.M) return;
    const int tid = threadIdx.x;
    const size_t stride = (size_t)p.RT * p.CT * (32 * kPT) / 4;
    const float4 *src = reinterpret_cast<const float4 *>(p.part) + ((size_t)rt * p.CT + ct) * (32 * kPT / 4) +
                        r0 * (kPT / 4);
    // the residual this thread updates (row r0 + i, column tid of the tile), read while the
    // partials stream in
    const int col = kPT * ct + tid;
    float res[NR];
#pragma unroll
    for (int i = 0; i < NR; i++) {
        const int row = 32 * rt + r0 + i;
        res[i] = (row < p.M && col < p.N) ? p.act[(size_t)row * p.N + col] : 0.0f;
    }
    sum_partials<NR, kMaxPSplit>(src, stride, p.n_split, &tile[0][0], kPT + 4, tid);
    __syncthreads();
#pragma unroll
    for (int i = 0; i < NR; i++) {
        const int row = 32 * rt + r0 + i;
        if (row >= p.M || col >= p.N) continue;
        const float v = tile[i][tid];
        const size_t idx = (size_t)row * p.N + col;
        if (p.stash) p.stash[idx] = v;
        p.act[idx] = res[i] + v;
    }
}

__global__ __launch_bounds__(256) void fill_zero_kernel(float4 *p, size_t n4) {
    for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < n4; i += (size_t)gridDim.x * 256)
        p[i] = make_float4(0.f, 0.f, 0.f, 0.f);
}

}  // namespace

static void proj_gemv(int t, const ProjArgs &p, hipStream_t st) {
    gemv_dispatch(t, gemv_mb(p.M), [&](auto tc, auto mc) {
        constexpr int T = decltype(tc)::value, MB = decltype(mc)::value, R = gemv_r(MB);
        proj_gemv_kernel<T, MB, R><<<(p.N + 8 * R - 1) / (8 * R), 256, gemv_lds(MB, p.K), st>>>(p);
    });
}

// Zeroes n floats (n a multiple of 4, p 16-byte aligned) with a kernel, so that a caller may
// capture it in a graph.
hipError_t launch_fill_zero(float *p, size_t n, hipStream_t st) {
    if (n % 4 || ((uintptr_t)p & 15)) return hipErrorInvalidValue;
    if (n == 0) return hipSuccess;
    const size_t n4 = n / 4;
    fill_zero_kernel<<<(int)std::min<size_t>((n4 + 255) / 256, 4096), 256, 0, st>>>(reinterpret_cast<float4 *>(p), n4);
    return hipGetLastError();
}

ProjPlan proj_plan(int M, int K, int N) {
    ProjPlan p;
    p.CT = (N + kPT - 1) / kPT;
    p.kps = K;
    p.n_split = 1;
    p.part_bytes = 0;
    const int rt32 = (M + 31) / 32;
    const int tiles = rt32 * p.CT;
    if (tiles < 256 && K % 256 == 0 && K >= 512) {
        p.RT = rt32;
        const int want = std::min(kMaxPSplit, std::max(2, (512 + tiles - 1) / tiles));
        const int nbat = K / 256;
        const int per = (nbat + want - 1) / want;
        p.kps = per * 256;
        p.n_split = (nbat + per - 1) / per;
        p.part_bytes = (uint64_t)p.n_split * tiles * 32 * kPT * sizeof(float);
        return p;
    }
    p.RT = (M + 63) / 64;
    return p;
}

ProjPlan proj_plan_kq(int ggml_type, int M, int K, int N, bool in_place) {
    ProjPlan p;
    p.in_place = in_place;
    p.CT = (N + kPT - 1) / kPT;
    p.RT = (M + 31) / 32;
    const int tiles = p.RT * p.CT;
    if (kq_tiles(ggml_type, tiles, K) && !in_place) {
        p.RT = (M + 63) / 64;
        p.kps = K;
        p.n_split = 1;
        p.part_bytes = 0;
        return p;
    }
    const KqSlices s = kq_slices(tiles, K);
    p.kps = s.kps;
    p.n_split = s.n_split;
    p.part_bytes = s.bytes;
    return p;
}

uint64_t proj_part_bytes_kq(int ggml_type, int M, int K, int N) {
    const int CT = (N + kPT - 1) / kPT, RT = (M + 31) / 32;
    uint64_t most = 0;
    for (int rt = 1; rt <= RT && !kq_tiles(ggml_type, rt * CT, K); rt++)
        most = std::max(most, kq_slices(rt * CT, K).bytes);
    return most;
}

hipError_t launch_proj_kq(const float *a, int M, int K, int ggml_type, const void *w, int N, float *act,
                          float *stash, const ProjPlan &plan, float *part, hipStream_t st) {
    if (K % 256 != 0 || M <= 0 || N <= 0 || (plan.part_bytes > 0 && !part) || !kq_type(ggml_type))
        return hipErrorInvalidValue;
    ProjArgs p;
    p.a = a;
    p.w = nullptr;
    p.bw = static_cast<const uint8_t *>(w);
    p.brow = (size_t)(K / 256) * kq_bytes(ggml_type);
    p.act = act;
    p.stash = stash;
    p.part = part;
    p.M = M;
    p.N = N;
    p.K = K;
    p.KW = K;
    p.RT = plan.RT;
    p.CT = plan.CT;
    p.kps = plan.kps;
    p.n_split = plan.n_split;
    p.n_wg = plan.RT * plan.CT * plan.n_split;
    if (gemv_fits(ggml_type, M, K, N) && plan.part_bytes > 0 && !plan.in_place) {
        proj_gemv(ggml_type, p, st);
        return hipGetLastError();
    }
    const int grid = (p.n_wg + 7) / 8 * 8;
    kq_dispatch(ggml_type, [&](auto tc) {
        constexpr int T = decltype(tc)::value;
        if (plan.part_bytes == 0)
            proj_tile_kernel<T><<<grid, 512, 0, st>>>(p);
        else
            proj_split_kq_kernel<T><<<grid, 256, 0, st>>>(p);
    });
    if (plan.part_bytes > 0) proj_reduce_kernel<<<plan.RT * plan.CT * (32 / kPRows), 256, 0, st>>>(p);
    return hipGetLastError();
}

hipError_t launch_proj(const float *a, int M, int K, const uint16_t *w, int N, float *act, float *stash,
                       const ProjPlan &plan, float *part, int planes, hipStream_t st) {
    if (K % kKC != 0 || M <= 0 || N <= 0 || (planes != 1 && planes != 2)) return hipErrorInvalidValue;
    ProjArgs p;
    p.a = a;
    p.w = reinterpret_cast<const _Float16 *>(w);
    p.bw = nullptr;
    p.brow = 0;
    p.act = act;
    p.stash = stash;
    p.part = part;
    p.M = M;
    p.N = N;
    p.K = K;
    p.KW = planes * K;
    p.RT = plan.RT;
    p.CT = plan.CT;
    p.kps = plan.kps;
    p.n_split = plan.n_split;
    p.n_wg = plan.RT * plan.CT * plan.n_split;
    const int grid = (p.n_wg + 7) / 8 * 8;
    if (plan.n_split == 1) {
        proj_tile_kernel<0><<<grid, 256, 0, st>>>(p);
    } else if (gemv_fits(planes == 2 ? kGemvF16x2 : kGemvF16, M, K, N) && !plan.in_place) {
        proj_gemv(planes == 2 ? kGemvF16x2 : kGemvF16, p, st);
    } else {
        proj_split_kernel<<<grid, 256, 0, st>>>(p);
        proj_reduce_kernel<<<plan.RT * plan.CT * (32 / kPRows), 256, 0, st>>>(p);
    }
    return hipGetLastError();
}

}  // namespace ts
