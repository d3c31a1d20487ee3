// Recompute backward for f32 storage where the LDS-staged kernels (backward.hip) would leave most of
// the chip idle: dK/dV and dQ on v_mfma_f32_32x32x2_f32, no value rounded below f32.
//
// Bound by the f32 matrix pipe (one 32x32x2 product every 64 clocks): a 32 x 32 block of D 128
// takes 256 of them for dK/dV against 128 row loads that the L2 holds, so operands go straight
// from memory into registers, every wave works by itself, and the whole design is about giving
// every SIMD a share of the blocks:
//   bwd_f32_dkdv  one workgroup per (batch, kv head, 32 keys) and chunk of the (query head, 32
//                 queries) blocks that see them; its four waves take the chunk's blocks in turn and
//                 are added up in LDS. More than one chunk: partial dK, dV in a workspace.
//   bwd_f32_dq    one workgroup per (batch, query head, 32 queries), its waves taking the key
//                 blocks in turn; further workgroups add up the partials of dK and dV in chunk
//                 order. No atomics, one writer per element: results repeat bit for bit.
// Staged through LDS with 128 keys (or queries) to a workgroup, B1 Hq8 Hkv2 S512 D64 causal put 8
// workgroups on the chip for dK/dV (293 us) and 32 for dQ (69 us); 19.9 and 19.2 us here, and the
// whole backward 366 -> 41; D 128 646 -> 75, Hq32 Hkv8 B2 S1024 D128 1311 -> 677 us.
#include "common.hpp"
#include "kernels.hpp"

#include <algorithm>

namespace fa {
namespace {

struct Frag32 {
    float v[16];
};

// Lane l = 32 g + c holds, for row (or column) c, the 16 contracted elements kidx(g, t); the
// accumulator keeps row kidx(g, r) of column c in register r, i.e. an accumulator is the operand
// of the next product that contracts over its rows.
__device__ __forceinline__ int kidx32(int g, int t) { return 8 * (t >> 2) + 4 * g + (t & 3); }

__device__ __forceinline__ f32x16_t mma32(const Frag32& a, const Frag32& b, f32x16_t acc) {
#pragma unroll
    for (int t = 0; t < 16; ++t)
        acc = __builtin_amdgcn_mfma_f32_32x32x2f32(a.v[t], b.v[t], acc, 0, 0, 0);
    return acc;
}

// The 32 rows of a tile as a buffer resource: rows from `rows` on read as zeros, so that no load
// needs a clamp or a select. Loads need dword alignment only.
typedef __amdgpu_buffer_rsrc_t Tile;
__device__ __forceinline__ Tile tile_of(const void* base, int64_t row0, int row_bytes, int rows) {
    return __builtin_amdgcn_make_buffer_rsrc((uint8_t*)base + row0 * row_bytes, (short)0,
                                             rows * row_bytes, 0x00020000);
}

// Columns col0 + kidx(g, t) of row c, zeros past D (FULL: D is the padded width).
template <bool FULL>
__device__ __forceinline__ Frag32 row_frag(Tile t, int col0, int D, int g, int c) {
    Frag32 f;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const int col = col0 + 8 * j + 4 * g;
        const int off = FULL || col < D ? (c * D + col) * 4 : (int)0x7fffff00;
        const u32x4_t x = __builtin_amdgcn_raw_buffer_load_b128(t, off, 0, 0);
#pragma unroll
        for (int i = 0; i < 4; ++i)
            f.v[4 * j + i] = FULL || col + i < D ? __uint_as_float(x[i]) : 0.0f;
    }
    return f;
}

// Column col of rows kidx(g, t). (Columns past D hold other rows' values: they only reach columns
// past D of the result, which are never stored.)
__device__ __forceinline__ Frag32 col_frag(Tile tl, int col, int D, int g) {
    Frag32 f;
#pragma unroll
    for (int t = 0; t < 16; ++t)
        f.v[t] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(
            tl, (4 * g * D + col) * 4, (8 * (t >> 2) + (t & 3)) * D * 4, 0));
    return f;
}

// Adds up the waves' 32 x DPAD results (register r of block m: row kidx(g, r), column 32 m + c)
// and hands element (row, column) to put().
template <int DPAD, int NW, typename Put>
__device__ __forceinline__ void reduce_waves(float* lds, const f32x16_t (&acc)[DPAD / 32], int D,
                                             Put&& put) {
    const int tid = threadIdx.x, lane = tid & 63, g = lane >> 5, c = lane & 31, wave = tid >> 6;
    __syncthreads();
#pragma unroll
    for (int m = 0; m < DPAD / 32; ++m)
#pragma unroll
        for (int r = 0; r < 16; ++r)
            lds[(wave * 32 + kidx32(g, r)) * DPAD + 32 * m + c] = acc[m][r];
    __syncthreads();
    for (int e = tid; e < 32 * DPAD; e += 64 * NW) {
        float s = lds[e];
#pragma unroll
        for (int w = 1; w < NW; ++w) s += lds[w * 32 * DPAD + e];
        if (e % DPAD < D) put(e / DPAD, e % DPAD, s);
    }
}

template <int DPAD, bool FULL>
__global__ __launch_bounds__(256, DPAD == 128 ? 1 : 2) void bwd_f32_dkdv(BackwardArgs a,
                                                                         BackwardSplit sp) {
    constexpr int MB = DPAD / 32;
    __shared__ float lds[4 * 32 * DPAD];
    const int tid = threadIdx.x, lane = tid & 63, g = lane >> 5, c = lane & 31;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int S = a.seq, D = a.head_dim, nq = (S + 31) / 32, nbk = a.batch * a.kv_heads;
    // early key blocks first: under a causal mask they see the most queries
    const int bkv = blockIdx.x % nbk;
    int kb, part;
    sp.coords(blockIdx.x / nbk, nq, a.group, a.causal, kb, part);
    const int qb0 = a.causal ? kb : 0, nqv = nq - qb0, items = a.group * nqv;
    const int first = part * sp.chunk, last = min(items, first + sp.chunk);
    const int b = bkv / a.kv_heads, kvh = bkv - b * a.kv_heads;
    const int k0 = kb * 32;
    const int64_t krow0 = (int64_t)bkv * S;
    const int64_t qhead0 = ((int64_t)b * a.q_heads + (int64_t)kvh * a.group) * S;
    const float c2 = a.scale * kLog2e;

    Frag32 kf[MB], vf[MB];
    {
        const Tile kt = tile_of(a.k, krow0 + k0, 4 * D, min(32, S - k0));
        const Tile vt = tile_of(a.v, krow0 + k0, 4 * D, min(32, S - k0));
#pragma unroll
        for (int m = 0; m < MB; ++m) {
            kf[m] = row_frag<FULL>(kt, 32 * m, D, g, c);
            vf[m] = row_frag<FULL>(vt, 32 * m, D, g, c);
        }
    }
    f32x16_t dk[MB], dv[MB];
#pragma unroll
    for (int m = 0; m < MB; ++m) {
        dk[m] = (f32x16_t)0.0f;
        dv[m] = (f32x16_t)0.0f;
    }
    // Loads run ahead of the products that need them, in the order the fences fix: the next block's
    // rows under this block's dV/dK products (D 128: one wave per SIMD has the registers, and
    // nothing else hides their latency), the columns of block m + 1 under the products of m.
    // (D 128 takes all 512 registers and twelve more, 16-byte pieces of K and V that are read again
    // from scratch memory once a block, of 16384 clocks; the lane offsets are opaque in the loop, or
    // ten to fifteen of them would be kept there too.)
    constexpr bool AHEAD = DPAD == 128;
    struct At {
        Tile q, o, ld;
        int qb, rows;
    };
    auto tiles = [&](int it) {
        At t;
        const int hh = it / nqv;
        t.qb = qb0 + it - hh * nqv;
        t.rows = min(32, S - t.qb * 32);
        const int64_t row0 = qhead0 + (int64_t)hh * S + t.qb * 32;
        t.q = tile_of(a.q, row0, 4 * D, t.rows);
        t.o = tile_of(a.dout, row0, 4 * D, t.rows);
        t.ld = tile_of(a.ld, row0, 8, t.rows);
        return t;
    };
    Frag32 qr[MB], dr[MB];
    auto load_rows = [&](const At& t) {
        int row = c;
        if (AHEAD) asm volatile("" : "+v"(row));
#pragma unroll
        for (int m = 0; m < MB; ++m) {
            qr[m] = row_frag<FULL>(t.q, 32 * m, D, g, row);
            dr[m] = row_frag<FULL>(t.o, 32 * m, D, g, row);
        }
    };
    if (AHEAD && first + wave < last) load_rows(tiles(first + wave));
    for (int it = first + wave; it < last; it += 4) {
        const At t = tiles(it);
        int cc = c, gg = g;
        if (AHEAD) asm volatile("" : "+v"(cc), "+v"(gg));
        if (!AHEAD) load_rows(t);
        u32x4_t ld[8];  // (LSE log2 e, delta) of rows kidx(g, 2 i), kidx(g, 2 i + 1)
#pragma unroll
        for (int i = 0; i < 8; ++i)
            ld[i] = __builtin_amdgcn_raw_buffer_load_b128(
                t.ld, (8 * (i >> 1) + 4 * gg + 2 * (i & 1)) * 8, 0, 0);
        f32x16_t s = (f32x16_t)0.0f, dp = (f32x16_t)0.0f;
#pragma unroll
        for (int m = 0; m < MB; ++m) {
            s = mma32(qr[m], kf[m], s);
            dp = mma32(dr[m], vf[m], dp);
        }
        __builtin_amdgcn_sched_barrier(0);
        Frag32 oc = col_frag(t.o, cc, D, gg), qc = col_frag(t.q, cc, D, gg);
        __builtin_amdgcn_sched_barrier(0);
        // Rows past the sequence: dO = 0 and delta = 0, so they add nothing.
        Frag32 pf, df;
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            const u32x4_t l = ld[i >> 1];
            float p = fast_exp2(fmaf(s[i], c2, -__uint_as_float(l[2 * (i & 1)])));
            if (a.causal && t.qb == kb && cc > kidx32(gg, i)) p = 0.0f;
            pf.v[i] = p;
            df.v[i] = p * (dp[i] - __uint_as_float(l[2 * (i & 1) + 1]));
        }
        if (AHEAD && it + 4 < last) load_rows(tiles(it + 4));
#pragma unroll
        for (int m = 0; m < MB; ++m) {
            const Frag32 om = oc, qm = qc;
            __builtin_amdgcn_sched_barrier(0);
            if (m + 1 < MB) {
                oc = col_frag(t.o, 32 * (m + 1) + cc, D, gg);
                qc = col_frag(t.q, 32 * (m + 1) + cc, D, gg);
            }
            __builtin_amdgcn_sched_barrier(0);
            dv[m] = mma32(pf, om, dv[m]);
            dk[m] = mma32(df, qm, dk[m]);
        }
    }
    // one chunk: the gradients themselves; else this chunk's partials (dK, then dV)
    const bool whole = items <= sp.chunk;
    float* const pp = sp.part + (int64_t)blockIdx.x * 64 * D;
    reduce_waves<DPAD, 4>(lds, dk, D, [&](int r, int d, float x) {
        if (!whole) pp[r * D + d] = x;
        else if (k0 + r < S) ((float*)a.dk)[(krow0 + k0 + r) * D + d] = x * a.scale;
    });
    reduce_waves<DPAD, 4>(lds, dv, D, [&](int r, int d, float x) {
        if (!whole) pp[(32 + r) * D + d] = x;
        else if (k0 + r < S) ((float*)a.dv)[(krow0 + k0 + r) * D + d] = x;
    });
}

// dK (which = 0) or dV of one (batch * kv head, 32 keys) with several chunks: the partials in chunk
// order.
__device__ __forceinline__ void add_partials(const BackwardArgs& a, const BackwardSplit& sp,
                                             int block) {
    const int S = a.seq, D = a.head_dim, nkb = (S + 31) / 32;
    const int split = sp.split_blocks(nkb, a.group, a.causal);
    const int which = block & 1, at = block >> 1, bkv = at / split, kb = at - bkv * split;
    const int items = a.group * (nkb - (a.causal ? kb : 0));
    const int n = (items + sp.chunk - 1) / sp.chunk;
    const int64_t step = (int64_t)64 * D * a.batch * a.kv_heads;
    const float* const base = sp.part + (int64_t)bkv * 64 * D + which * 32 * D;
    const BackwardSplit::Walk first(sp, kb, nkb, a.group, a.causal);
    const float scale = which ? 1.0f : a.scale;
    float* out = (float*)(which ? a.dv : a.dk) + ((int64_t)bkv * S + kb * 32) * D;
    const int count = min(32, S - kb * 32) * D;
    if (a.vec) {
        for (int e = threadIdx.x * 4; e < count; e += blockDim.x * 4) {
            BackwardSplit::Walk at_chunk = first;
            f32x4_t s = *(const f32x4_t*)(base + at_chunk.slot * step + e);
#pragma unroll 8
            for (int i = 1; i < n; ++i) {
                at_chunk.next();
                s += *(const f32x4_t*)(base + at_chunk.slot * step + e);
            }
            *(f32x4_t*)(out + e) = s * scale;
        }
    } else {
        for (int e = threadIdx.x; e < count; e += blockDim.x) {
            BackwardSplit::Walk at_chunk = first;
            float s = base[at_chunk.slot * step + e];
#pragma unroll 8
            for (int i = 1; i < n; ++i) {
                at_chunk.next();
                s += base[at_chunk.slot * step + e];
            }
            out[e] = s * scale;
        }
    }
}

template <int DPAD, int NW, bool FULL>
__global__ __launch_bounds__(64 * NW, DPAD == 128 ? 1 : 2) void bwd_f32_dq(BackwardArgs a,
                                                                           BackwardSplit sp,
                                                                           int n_dq) {
    constexpr int MB = DPAD / 32;
    __shared__ float lds[NW * 32 * DPAD];
    if ((int)blockIdx.x >= n_dq) {
        add_partials(a, sp, blockIdx.x - n_dq);
        return;
    }
    const int tid = threadIdx.x, lane = tid & 63, g = lane >> 5, c = lane & 31;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int S = a.seq, D = a.head_dim, nq = (S + 31) / 32, nbh = a.batch * a.q_heads;
    // causal: the last query blocks see the most keys and dispatch first
    const int qb = a.causal ? nq - 1 - (int)(blockIdx.x / nbh) : (int)(blockIdx.x / nbh);
    const int bh = blockIdx.x % nbh, b = bh / a.q_heads, kvh = (bh - b * a.q_heads) / a.group;
    const int q0 = qb * 32, rows = min(32, S - q0);
    const int64_t qrow0 = (int64_t)bh * S + q0, krow0 = ((int64_t)b * a.kv_heads + kvh) * S;
    const float c2 = a.scale * kLog2e;

    Frag32 qf[MB], of[MB];
    const Tile qt = tile_of(a.q, qrow0, 4 * D, rows), ot = tile_of(a.dout, qrow0, 4 * D, rows);
#pragma unroll
    for (int m = 0; m < MB; ++m) {
        qf[m] = row_frag<FULL>(qt, 32 * m, D, g, c);
        of[m] = row_frag<FULL>(ot, 32 * m, D, g, c);
    }
    const float2 ld = a.ld[qrow0 + min(c, rows - 1)];
    f32x16_t dq[MB];
#pragma unroll
    for (int m = 0; m < MB; ++m) dq[m] = (f32x16_t)0.0f;
    const int nkb = a.causal ? qb + 1 : nq;
    constexpr bool AHEAD = DPAD == 128;  // (as in bwd_f32_dkdv)
    Frag32 kr[MB], vr[MB];
    auto load_rows = [&](int kb) {
        const int keys = min(32, S - kb * 32);
        const Tile kt = tile_of(a.k, krow0 + kb * 32, 4 * D, keys);
        const Tile vt = tile_of(a.v, krow0 + kb * 32, 4 * D, keys);
#pragma unroll
        for (int m = 0; m < MB; ++m) {
            kr[m] = row_frag<FULL>(kt, 32 * m, D, g, c);
            vr[m] = row_frag<FULL>(vt, 32 * m, D, g, c);
        }
    };
    if (AHEAD && wave < nkb) load_rows(wave);
    for (int kb = wave; kb < nkb; kb += NW) {
        const int keys = min(32, S - kb * 32);
        const Tile kt = tile_of(a.k, krow0 + kb * 32, 4 * D, keys);
        if (!AHEAD) load_rows(kb);
        f32x16_t s = (f32x16_t)0.0f, dp = (f32x16_t)0.0f;
#pragma unroll
        for (int m = 0; m < MB; ++m) {
            s = mma32(kr[m], qf[m], s);
            dp = mma32(vr[m], of[m], dp);
        }
        __builtin_amdgcn_sched_barrier(0);
        Frag32 kc = col_frag(kt, c, D, g);
        __builtin_amdgcn_sched_barrier(0);
        Frag32 df;
#pragma unroll
        for (int t = 0; t < 16; ++t) {
            const int key = kidx32(g, t);
            float p = fast_exp2(fmaf(s[t], c2, -ld.x));
            if (key >= keys || (a.causal && kb == qb && key > c)) p = 0.0f;
            df.v[t] = p * (dp[t] - ld.y);
        }
        if (AHEAD && kb + NW < nkb) load_rows(kb + NW);
#pragma unroll
        for (int m = 0; m < MB; ++m) {
            const Frag32 km = kc;
            __builtin_amdgcn_sched_barrier(0);
            if (m + 1 < MB) kc = col_frag(kt, 32 * (m + 1) + c, D, g);
            __builtin_amdgcn_sched_barrier(0);
            dq[m] = mma32(df, km, dq[m]);
        }
    }
    reduce_waves<DPAD, NW>(lds, dq, D, [&](int r, int d, float x) {
        if (r < rows) ((float*)a.dq)[(qrow0 + r) * D + d] = x * a.scale;
    });
}

template <int DPAD, int NW, bool FULL>
void launch_v(const BackwardArgs& a, const BackwardSplit& sp, hipStream_t s) {
    const int nb = (a.seq + 31) / 32, nbk = a.batch * a.kv_heads;
    hipLaunchKernelGGL((bwd_f32_dkdv<DPAD, FULL>),
                       dim3((unsigned)(sp.workgroups(nb, a.group, a.causal) * nbk)), dim3(256), 0,
                       s, a, sp);
    const int n_dq = nb * a.batch * a.q_heads;
    const int n_add = 2 * sp.split_blocks(nb, a.group, a.causal) * nbk;
    hipLaunchKernelGGL((bwd_f32_dq<DPAD, NW, FULL>), dim3((unsigned)(n_dq + n_add)), dim3(64 * NW), 0, s,
                       a, sp, n_dq);
}

template <int DPAD, int NW>
void launch_d(const BackwardArgs& a, const BackwardSplit& sp, hipStream_t s) {
    if (a.head_dim == DPAD) launch_v<DPAD, NW, true>(a, sp, s);
    else launch_v<DPAD, NW, false>(a, sp, s);
}

}  // namespace

// Whether the LDS-staged kernels (backward.hip: one workgroup per 128 keys, four waves share the
// tiles) are the faster ones: where those workgroups fill the chip. `filled` is the part of the CUs'
// time that they keep busy, one to a CU; over 400 shapes the ratio of the two follows it (us for the
// backward, staged / these):
//   D 128: 0.62 (H32 B2 S500 causal) 276 / 253, 0.75 (B4 S200 causal) 145 / 155, 1 (B4 S384 causal)
//     267 / 326, (B4 S200) 148 / 214; Hq32 Hkv8 S2048 causal, 0.27, 2529 / 1218; over long sequences,
//     whose chunks come out even, from 0.78 (B2 H8 S1500, 0.75, 707 / 661, H4 S6000, 0.73, 2722 /
//     2431; H24 S2048 causal, 0.80, 957 / 987);
//   64 < D < 128, where these load and multiply the padding too: D 96, 0.50 (B2 S384 causal) 208 / 197,
//     0.62 (B2 S500 causal) 266 / 316, 1 (B4 S200) 139 / 261;
//   D <= 64, where a CU holds two of them: with that chip filled too (D 64, H32 B4 S500 292 / 318, B8
//     S384 causal 254 / 276, B8 S500 576 / 650; not B4 S384 causal 129 / 118, B6 S384 251 / 221), or up
//     to 256 keys without a mask, a few tiles to a workgroup, once (B4 S200 85.5 / 94.9). Between 33 and
//     63 dims, where these load half the padding, a little earlier (D 40: B4 S500 causal 202 / 215, but
//     D 24 113 / 102), to 512 keys (B2 S500 152 / 161) and with one key block (B8 S100 causal 52 / 60;
//     not at 0.75, B12 S60 53 / 46, although B6 S100 51 / 56). At D 32 and 64 not with long sequences
//     (B4 S1000 1059 / 1085, B4 H16 S2048 causal 1132 / 1095; D 40 B4 S1000 1034 / 1138).
static bool staged_f32(const BackwardArgs& a) {
    const int64_t nkb = (a.seq + 127) / 128, n = (int64_t)a.batch * a.kv_heads * nkb;
    const int64_t cus = device_cus();
    if (n < cus / 2) return false;
    const int64_t longest = a.group * nkb, units = (int64_t)a.batch * a.kv_heads;
    const double tiles = (double)units * (a.causal ? 0.5 * longest * (nkb + 1) : longest * nkb);
    BackwardSplit one{};
    one.set_chunk(longest, longest, (int)nkb, a.group, a.causal, units, 0);
    auto filled = [&](int64_t places) {
        return tiles / (double)(places * backward_time(one, (int)nkb, a, places, 0, 0));
    };
    if (a.head_dim > 64) return filled(cus) >= (a.head_dim < 128 ? 0.55 : a.seq < 1024 ? 0.7 : 0.78);
    const bool full = a.head_dim == 64 || a.head_dim == 32, padded = a.head_dim > 32 && !full;
    return (a.seq < 1500 || !full) && filled(cus) >= 0.9 &&
           (filled(2 * cus) >= (padded ? 0.6 : 0.7) || (padded && a.seq <= 128) ||
            (!a.causal && a.seq <= (padded ? 512 : 256)));
}

// Blocks a wave takes: the total over the waves that the chip holds at once (one per SIMD at
// D 128, two below), so a launch is one round of about equal workgroups and the partials of a
// small problem stay a few MB (at most one chunk more than the round has workgroups, twice for
// the causal taper).
BackwardSplit backward_f32_split(const BackwardArgs& a, uint64_t limit) {
    const int64_t nq = (a.seq + 31) / 32, nbk = (int64_t)a.batch * a.kv_heads;
    const int64_t blocks = a.causal ? nq * (nq + 1) / 2 : nq * nq;
    const int64_t waves = (int64_t)device_cus() * 4 * (a.head_dim > 64 ? 1 : 2);
    const int64_t per_wave = std::max<int64_t>(1, (nbk * a.group * blocks + waves - 1) / waves);
    BackwardSplit sp{};
    if (staged_f32(a)) return sp;
    const int64_t longest = a.group * nq;
    sp.set_chunk(4 * per_wave, longest, (int)nq, a.group, a.causal, nbk, 64 * a.head_dim);
    if (sp.bytes > limit)  // one chunk: no partials
        sp.set_chunk(longest, longest, (int)nq, a.group, a.causal, nbk, 64 * a.head_dim);
    return sp;
}

void launch_backward_f32(const BackwardArgs& a, const BackwardSplit& sp, hipStream_t s) {
    if (a.head_dim <= 32) launch_d<32, 8>(a, sp, s);
    else if (a.head_dim <= 64) launch_d<64, 8>(a, sp, s);
    else launch_d<128, 4>(a, sp, s);
}

}  // namespace fa
