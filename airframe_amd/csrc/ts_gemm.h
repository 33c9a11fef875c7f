// ts_gemm.h -- the matrix-core loops shared by the projection kernels (the QKV projection
// with the append as epilogue, and the attention output projection): C = X W^T with X f32
// [M][K] split hi + lo into f16 and W f16 [N][K] row-major, on v_mfma_f32_32x32x16_f16.
//
// Operand layout of the 32x32x16 instruction used throughout: lane (j = lane % 32,
// hf = lane / 32) supplies row j of A and column j of B with 8 consecutive k; within a chunk of
// 64, k-step q of lane half hf covers k = 32 hf + 8 q .. + 7, so a lane's B operands of one
// chunk are 64 contiguous bytes of its weight row.  D register 4q + r of a 32 x 32 block is
// row 8q + 4hf + r, column j.
#pragma once
#include <type_traits>

#include "ts_mfma.h"

namespace ts {
namespace {

typedef float floatx16 __attribute__((ext_vector_type(16)));

constexpr int kKC = 64;     // k per chunk
constexpr int kAStr = 72;   // LDS row stride of the x tiles (f16): 144 B spreads the rows' banks

// The 8 x values of one staging thread as hi and lo f16 halves.
__device__ inline void split8(const float4 &u, const float4 &v, half8 &hi, half8 &lo) {
    const float x[8] = {u.x, u.y, u.z, u.w, v.x, v.y, v.z, v.w};
#pragma unroll
    for (int e = 0; e < 8; e++) {
        const _Float16 h = (_Float16)x[e];
        hi[e] = h;
        lo[e] = (_Float16)(x[e] - (float)h);
    }
}

__device__ inline void zero(floatx16 &a) {
#pragma unroll
    for (int e = 0; e < 16; e++) a[e] = 0.0f;
}

// LDS of the tile loop: three chunks of kTK k of 64 x rows (hi/lo) and 256 weight rows, rows
// unpadded.  A row's four 16-byte slots are permuted by row (tile_slot) so that the 16 rows
// that one phase of an operand read or a staging write touches at one slot cover all 64 banks.
constexpr int kTK = 32;
struct GemmTiles {
    _Float16 hi[3][64][kTK];
    _Float16 lo[3][64][kTK];
    _Float16 w[3][256][kTK];
};
// f16 index inside tile row r of slot s (8 k).
__device__ inline int tile_slot(int r, int s) { return 8 * (s ^ ((r >> 2) & 3)); }
// Chunk c holds k 0-15 and 32-47 of its 64 (c even) or the other half, so that the k-steps of two
// chunks are those of the slice loop (k 8q.. and 32 + 8q.. together) and the sums have the same
// bits; slot s of a chunk starts tile_k(s) behind tile_chunk(c).
__device__ inline size_t tile_chunk(int c) { return (size_t)(c >> 1) * 64 + (c & 1) * 16; }
__device__ inline int tile_k(int s) { return 8 * (s & 1) + 32 * (s >> 1); }

#define TS_SGB(mask, n) __builtin_amdgcn_sched_group_barrier(mask, n, 0)
constexpr int kValu = 2, kMfma = 8, kVmemRead = 0x20, kDsRead = 0x100, kDsWrite = 0x200;

// 64 rows x 256 columns over nch chunks of kTK, 256 threads: wave w accumulates rows 32 rb + ..,
// columns 64 w + 32 cb + .. in acc[rb][cb].  Staging thread tid owns slot tid % 4 of x row tid / 4
// and of weight rows tid / 4 + 64 i: xs / ws[i] point at its k (tile_k) of chunk 0 (a row past the tile's last
// one points at any valid row: what it adds up to is not used).  xwrap: x has xwrap chunks and
// weight chunk c multiplies x chunk c mod xwrap (nch = 2 xwrap: rows of two weight planes, hi
// then lo, against the same x; nch = xwrap: one plane).
//
// Both operands go through LDS, read from memory whole cache lines at a time (a weight row per
// lane, straight into the operands, kept the address path busier than the matrix cores).  Chunk c
// is multiplied from one LDS buffer while chunk c + 2 goes from registers into another and
// chunk c + 5 is loaded into those registers; the third buffer already holds chunk c + 1, so that
// its first operands are read before the barrier and no matrix instruction waits for LDS
// behind it.  The instruction groups spread the staging's VALU, LDS and memory instructions
// between the matrix instructions of the same wave (two waves per SIMD do not cover for each
// other between barriers).  Nothing in the loop is conditional (a skipped load would make every
// wait for memory a wait for all of it): past the end the last chunk is loaded and stored again.
// 2048 x 6144 outputs, 2560 long: 198 us with the weight rows loaded into the operands, 187 now;
// 2048 x 2560, 4096 long: 199, 149 (all CUs together reach about 1.1 PFLOP/s on f16 matrix
// instructions; chunks of 32 k in a row took 164 and 134, but add in another order, and a last bit
// moves a key or value next to a code's edge).
// Its loads bound it (counters, 2048 x 6144): of the CUs' busy cycles the address path works 91%, ~50
// cycles for a load of 1 KB, the matrix cores 39% and LDS 30%.  A chunk takes two 32-byte pieces of
// a weight row's 128-byte line and the next chunk the other two, a step later.  128-row tiles (8
// waves, or 4 of 64 x 128) were slower.
__device__ __forceinline__ void gemm_tile_core(GemmTiles &sm, const float *xs, const _Float16 *const (&ws)[4],
                                               int nch, int xwrap, int tid, floatx16 (&acc)[2][2]) {
    const int wave = tid >> 6, lane = tid & 63, j = lane & 31, hf = lane >> 5;
    const int si = tid >> 2, sc = tid & 3;
    struct Stage {
        float4 x[2];
        half8 w[4];
    };
    struct Ops {
        half8 ah[2], al[2], b[2];
    };
    auto load = [&](Stage &g, int c) {
        c = min(c, nch - 1);
        const int cx = c >= xwrap ? c - xwrap : c;
        const size_t kx = tile_chunk(cx), kw = tile_chunk(c);
        g.x[0] = *reinterpret_cast<const float4 *>(xs + kx);
        g.x[1] = *reinterpret_cast<const float4 *>(xs + kx + 4);
#pragma unroll
        for (int i = 0; i < 4; i++) g.w[i] = *reinterpret_cast<const half8 *>(ws[i] + kw);
    };
    auto store_x = [&](int buf, const Stage &g) {
        const int at = tile_slot(si, sc);
        half8 h, l;
        split8(g.x[0], g.x[1], h, l);
        *reinterpret_cast<half8 *>(&sm.hi[buf][si][at]) = h;
        *reinterpret_cast<half8 *>(&sm.lo[buf][si][at]) = l;
    };
    auto store_w = [&](int buf, const Stage &g) {
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const int r = si + 64 * i;
            *reinterpret_cast<half8 *>(&sm.w[buf][r][tile_slot(r, sc)]) = g.w[i];
        }
    };
    auto fetch = [&](Ops &o, int buf, int q) {
#pragma unroll
        for (int rb = 0; rb < 2; rb++) {
            const int r = 32 * rb + j, at = tile_slot(r, 2 * hf + q);
            o.ah[rb] = *reinterpret_cast<const half8 *>(&sm.hi[buf][r][at]);
            o.al[rb] = *reinterpret_cast<const half8 *>(&sm.lo[buf][r][at]);
        }
#pragma unroll
        for (int cb = 0; cb < 2; cb++) {
            const int r = 64 * wave + 32 * cb + j;
            o.b[cb] = *reinterpret_cast<const half8 *>(&sm.w[buf][r][tile_slot(r, 2 * hf + q)]);
        }
    };
    auto multiply = [&](const Ops &o) {
#pragma unroll
        for (int rb = 0; rb < 2; rb++)
#pragma unroll
            for (int cb = 0; cb < 2; cb++)
                acc[rb][cb] = __builtin_amdgcn_mfma_f32_32x32x16_f16(o.ah[rb], o.b[cb], acc[rb][cb], 0, 0, 0);
#pragma unroll
        for (int rb = 0; rb < 2; rb++)
#pragma unroll
            for (int cb = 0; cb < 2; cb++)
                acc[rb][cb] = __builtin_amdgcn_mfma_f32_32x32x16_f16(o.al[rb], o.b[cb], acc[rb][cb], 0, 0, 0);
    };
#pragma unroll
    for (int rb = 0; rb < 2; rb++)
#pragma unroll
        for (int cb = 0; cb < 2; cb++) zero(acc[rb][cb]);
    Stage g[3];
    Ops o[2];
#pragma unroll
    for (int u = 0; u < 3; u++) load(g[u], u);
#pragma unroll
    for (int u = 0; u < 2; u++) {
        store_x(u, g[u]);
        store_w(u, g[u]);
        load(g[u], 3 + u);
    }
    __syncthreads();
    fetch(o[0], 0, 0);
    // chunk c in buffer u = c mod 3 (a constant, so that g and o stay in registers)
    auto step = [&](auto uc, int c) {
        constexpr int u = decltype(uc)::value, v = (u + 2) % 3;
        fetch(o[1], u, 1);
        store_x(v, g[v]);
        multiply(o[0]);
#pragma unroll
        for (int i = 0; i < 6; i++) {
            TS_SGB(kMfma, 1);
            TS_SGB(kDsRead, 1);
            TS_SGB(kValu, 5);
        }
#pragma unroll
        for (int i = 0; i < 2; i++) {
            TS_SGB(kMfma, 1);
            TS_SGB(kValu, 6);
            TS_SGB(kDsWrite, 1);
        }
        __builtin_amdgcn_sched_barrier(0);
        fetch(o[0], (u + 1) % 3, 0);
        store_w(v, g[v]);
        load(g[v], c + 5);
        multiply(o[1]);
#pragma unroll
        for (int i = 0; i < 4; i++) {
            TS_SGB(kMfma, 1);
            TS_SGB(kDsRead, 1);
            TS_SGB(kDsWrite, 1);
        }
#pragma unroll
        for (int i = 0; i < 2; i++) {
            TS_SGB(kMfma, 1);
            TS_SGB(kDsRead, 1);
            TS_SGB(kValu, 4);
            TS_SGB(kVmemRead, 1);
        }
#pragma unroll
        for (int i = 0; i < 2; i++) {
            TS_SGB(kMfma, 1);
            TS_SGB(kValu, 4);
            TS_SGB(kVmemRead, 2);
        }
        __builtin_amdgcn_sched_barrier(0);
        __syncthreads();
    };
    int c = 0;
    for (; c + 3 <= nch; c += 3) {
        step(std::integral_constant<int, 0>{}, c);
        step(std::integral_constant<int, 1>{}, c + 1);
        step(std::integral_constant<int, 2>{}, c + 2);
    }
    if (c < nch) step(std::integral_constant<int, 0>{}, c);
    if (c + 1 < nch) step(std::integral_constant<int, 1>{}, c + 1);
}

// LDS of gemm_split_core: x of one batch (4 chunks) as hi/lo.
struct SplitTiles {
    _Float16 hi[4][32][kAStr];
    _Float16 lo[4][32][kAStr];
};

// One slice of the reduction for a 32 x 256 tile, 256 threads, in batches of 4 chunks (256 k)
// loaded in one go -- x into LDS as hi/lo (shared by the 4 waves), the weights straight into B
// operands -- so a batch costs one memory round trip, then 64 MFMAs per wave.  Wave w
// accumulates columns 64 w + 32 cb + .. in acc[cb].  Staging thread (si = tid / 8, sc = tid % 8)
// owns 8 floats of x row si per chunk (xs at chunk 0 of the row, null: a zero row); the slice
// starts at weight chunk c0, and weight chunk c multiplies x chunk c mod xwrap (as in
// gemm_tile_core); wp[cb]: the lane's weight row of column block cb at chunk c0, offset 32 hf.
__device__ __forceinline__ void gemm_split_core(SplitTiles &sm, const float *xs, int c0, int xwrap,
                                                const _Float16 *const (&wp)[2], int nbat, int tid,
                                                floatx16 (&acc)[2]) {
    constexpr int NB = 4;
    const int lane = tid & 63, j = lane & 31, hf = lane >> 5;
    const int si = tid >> 3, sc = tid & 7;
    zero(acc[0]);
    zero(acc[1]);
    for (int b = 0; b < nbat; b++) {
        const int ko = b * NB * kKC;
        float4 xu[NB], xv[NB];
        half8 wb[NB][2][4];
#pragma unroll
        for (int c = 0; c < NB; c++) {
            xu[c] = make_float4(0.f, 0.f, 0.f, 0.f);
            xv[c] = xu[c];
            if (xs) {
                int cx = c0 + b * NB + c;
                cx = cx >= xwrap ? cx - xwrap : cx;
                xu[c] = *reinterpret_cast<const float4 *>(xs + cx * kKC);
                xv[c] = *reinterpret_cast<const float4 *>(xs + cx * kKC + 4);
            }
#pragma unroll
            for (int cb = 0; cb < 2; cb++)
#pragma unroll
                for (int q = 0; q < 4; q++)
                    wb[c][cb][q] = *reinterpret_cast<const half8 *>(wp[cb] + ko + c * kKC + 8 * q);
        }
        if (b > 0) __syncthreads();  // the previous batch's x tiles are no longer read
#pragma unroll
        for (int c = 0; c < NB; c++) {
            half8 h, l;
            split8(xu[c], xv[c], h, l);
            *reinterpret_cast<half8 *>(&sm.hi[c][si][8 * sc]) = h;
            *reinterpret_cast<half8 *>(&sm.lo[c][si][8 * sc]) = l;
        }
        __syncthreads();
#pragma unroll
        for (int c = 0; c < NB; c++)
#pragma unroll
            for (int q = 0; q < 4; q++) {
                const half8 ah = *reinterpret_cast<const half8 *>(&sm.hi[c][j][32 * hf + 8 * q]);
                const half8 al = *reinterpret_cast<const half8 *>(&sm.lo[c][j][32 * hf + 8 * q]);
#pragma unroll
                for (int cb = 0; cb < 2; cb++) {
                    acc[cb] = __builtin_amdgcn_mfma_f32_32x32x16_f16(ah, wb[c][cb][q], acc[cb], 0, 0, 0);
                    acc[cb] = __builtin_amdgcn_mfma_f32_32x32x16_f16(al, wb[c][cb][q], acc[cb], 0, 0, 0);
                }
            }
    }
}

// Deterministic sum of n_split partial tiles (split stride `stride` float4s) of NR rows x 256
// columns starting at src, into tile[NR][tstr] of LDS: every thread issues the loads of all
// splits of two float4 before adding them, in split order.  256 threads.
template <int NR, int MAXS>
__device__ __forceinline__ void sum_partials(const float4 *src, size_t stride, int n_split, float *tile, int tstr,
                                             int tid) {
    constexpr int PER = NR / 4;            // float4 of the rows per thread
    constexpr int U = PER < 2 ? PER : 2;   // float4 per pass
#pragma unroll
    for (int pass = 0; pass < PER / U; pass++) {
        float4 v[U][MAXS];
#pragma unroll
        for (int u = 0; u < U; u++)
#pragma unroll
            for (int sp = 0; sp < MAXS; sp++)
                if (sp < n_split) v[u][sp] = src[sp * stride + (U * pass + u) * 256 + tid];
#pragma unroll
        for (int u = 0; u < U; u++) {
            float4 acc = v[u][0];
#pragma unroll
            for (int sp = 1; sp < MAXS; sp++)
                if (sp < n_split) {
                    acc.x = acc.x + v[u][sp].x;
                    acc.y = acc.y + v[u][sp].y;
                    acc.z = acc.z + v[u][sp].z;
                    acc.w = acc.w + v[u][sp].w;
                }
            const int e4 = (U * pass + u) * 256 + tid;
            *reinterpret_cast<float4 *>(tile + (e4 / 64) * tstr + 4 * (e4 % 64)) = acc;
        }
    }
}

}  // namespace
}  // namespace ts
