// attention.hip -- the exact attention face (gpu_attention.rs:451-570
// GpuContext::attention): f32 softmax(Q K^T / sqrt(d)) V with GQA and
// causal masking, the quality reference the reference serves over
// cubek-attention and the engine's tiled decode face
// (engine/mod.rs:1041-1067 gqa_attention_tiled).
//
// Contract kept from the reference: Q is taken unscaled and 1/sqrt(head_dim)
// applied here; query head h reads kv head h / (n_heads / n_kv_heads) (the
// reference materialises that repeat on the host, here it is an index);
// causal masks key j for query i when j + seq_q > i + seq_kv (bottom-right
// aligned, so seq_q = 1 attends to every key); a row with every key masked
// is 0/0 = NaN, as the NumPy reference's is.  Same validation, messages and
// u32 index ceiling as the reference's face.
//
// att_tile (below) serves head dims up to 128 on the f32 matrix cores; other
// shapes, and a few queries over few keys (att_rows_faster), run att_exact, one workgroup per (batch, head, query row): the
// row's query in LDS, keys
// in chunks of ATT_CHUNK -- a thread per key for the scores (dot products in
// 16-channel partial sums), the chunk's max and sum by workgroup reductions,
// an online softmax across chunks in f32, and a thread per output channel
// summing p_j v[j][c] over the chunk's keys in 32-key partial sums (blocked
// sums keep f32 rounding growing with the square root of the length).  It is
// what the quantised schemes are measured against.
#include <math.h>

#include <type_traits>

#include "qbk_internal.h"

#pragma clang fp contract(off)

namespace qbk {

#define ATT_THREADS 256
#define ATT_CHUNK 1024
#define ATT_MAXD 1024

struct AttArgs {
    const float *q, *k, *v;
    float *out;
    size_t H, Hk, Sq, Skv, d, dv;
    int causal;
    float scale;
    // element strides of k and v: between consecutive keys of a kv head and
    // between kv heads (head-major (B, Hkv, Skv, d): d and Skv d; a decoder
    // block's row-major cache (rows, Hkv d): Hkv d and d)
    size_t k_tok, k_head, v_tok, v_head;
    uint32_t BH;  // att_tile: batches times heads
};

__device__ __forceinline__ float att_block_max(float v, float *red) {
    for (int o = 32; o >= 1; o >>= 1) v = fmaxf(v, __shfl_xor(v, o, 64));
    __syncthreads();
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
    __syncthreads();
    float r = red[0];
    for (int w = 1; w < ATT_THREADS / 64; w++) r = fmaxf(r, red[w]);
    return r;
}

__device__ __forceinline__ float att_block_sum(float v, float *red) {
    for (int o = 32; o >= 1; o >>= 1) v += __shfl_xor(v, o, 64);
    __syncthreads();
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
    __syncthreads();
    float r = red[0];
    for (int w = 1; w < ATT_THREADS / 64; w++) r += red[w];
    return r;
}

__global__ void __launch_bounds__(ATT_THREADS) att_exact(AttArgs a) {
    __shared__ float qs[ATT_MAXD];
    __shared__ float ps[ATT_CHUNK];
    __shared__ float red[ATT_THREADS / 64];
    const size_t row = blockIdx.x;  // (b * H + h) * Sq + i
    const size_t i = row % a.Sq, bh = row / a.Sq, b = bh / a.H, h = bh % a.H;
    const size_t bk = b * a.Hk + h / (a.H / a.Hk);
    const float *qr = a.q + row * a.d;
    const float *kb = a.k + bk * a.k_head;
    const float *vb = a.v + bk * a.v_head;
    const int tid = threadIdx.x;
    for (size_t c = tid; c < a.d; c += ATT_THREADS) qs[c] = qr[c];
    // keys visible to query i: j < i + 1 + (Skv - Sq), i.e. j + Sq <= i + Skv
    size_t kend = a.Skv;
    if (a.causal) kend = i + a.Skv >= a.Sq ? (i + a.Skv - a.Sq + 1 < a.Skv ? i + a.Skv - a.Sq + 1 : a.Skv) : 0;
    float m = -INFINITY, l = 0.0f;
    float acc[ATT_MAXD / ATT_THREADS];
#pragma unroll
    for (int u = 0; u < ATT_MAXD / ATT_THREADS; u++) acc[u] = 0.0f;
    __syncthreads();
    for (size_t j0 = 0; j0 < kend; j0 += ATT_CHUNK) {
        const size_t j1 = j0 + ATT_CHUNK < kend ? j0 + ATT_CHUNK : kend;
        float cmax = -INFINITY;
        for (size_t j = j0 + tid; j < j1; j += ATT_THREADS) {
            const float *kr = kb + j * a.k_tok;
            float s = 0.0f;
            for (size_t c0 = 0; c0 < a.d; c0 += 16) {  // blocked: 16-term partials
                float sp = 0.0f;
                const size_t c1 = c0 + 16 < a.d ? c0 + 16 : a.d;
                for (size_t c = c0; c < c1; c++) sp += qs[c] * kr[c];
                s += sp;
            }
            s = s * a.scale;
            ps[j - j0] = s;
            cmax = fmaxf(cmax, s);
        }
        cmax = att_block_max(cmax, red);
        const float mn = fmaxf(m, cmax);
        const float alpha = m == -INFINITY ? 0.0f : expf(m - mn);
        float part = 0.0f;
        for (size_t j = j0 + tid; j < j1; j += ATT_THREADS) {
            const float p = expf(ps[j - j0] - mn);
            ps[j - j0] = p;
            part += p;
        }
        part = att_block_sum(part, red);  // its barriers also publish ps
        l = l * alpha + part;
#pragma unroll
        for (int u = 0; u < ATT_MAXD / ATT_THREADS; u++) {
            const size_t c = tid + (size_t)u * ATT_THREADS;
            if (c >= a.dv) break;
            float sacc = 0.0f;
            for (size_t jb = j0; jb < j1; jb += 32) {  // blocked: 32-term partials
                float sp = 0.0f;
                const size_t je = jb + 32 < j1 ? jb + 32 : j1;
                for (size_t j = jb; j < je; j++) sp += ps[j - j0] * vb[j * a.v_tok + c];
                sacc += sp;
            }
            acc[u] = acc[u] * alpha + sacc;
        }
        m = mn;
        __syncthreads();  // ps is rewritten by the next chunk
    }
#pragma unroll
    for (int u = 0; u < ATT_MAXD / ATT_THREADS; u++) {
        const size_t c = tid + (size_t)u * ATT_THREADS;
        if (c >= a.dv) break;
        a.out[row * a.dv + c] = acc[u] / l;
    }
}

// ---- the same on the f32 matrix cores --------------------------------------
//
// att_exact's arithmetic in f32 throughout, for head and value dims of at
// most 128 whose rows take 16-byte loads.  A query row a workgroup reads every
// key and value once per query, and a thread per key walks its key's row
// alone; here a wave takes 16 QT queries of one head against 32 keys at a
// time on v_mfma_f32_16x16x4_f32 (f32 products and sums), and the waves of a
// workgroup split the keys (tiles of 32 round robin), so that a few queries
// over many keys fill the chip as well; each keeps its own running max, sum
// and output, merged through LDS at the end.
//   S = K Q^T: A row = key, B column = query; a lane's float4 of channels
//     16 s + 4 G .. feeds four MFMAs, of both operands.  Lane (col, G) gets
//     keys 4 G .. 4 G + 3 of a 16-key tile for query col;
//   O^T += V^T P^T: MFMA i of a tile takes keys 4 G + i, whose p are lane
//     (col, G)'s i-th: P never leaves its lane.  A lane's float4 of channels
//     64 h + 4 m .. feeds four MFMAs, whose outputs leave lane (col, G) the
//     16 consecutive channels 64 h + 16 G .. of query col.
// The sums stay blocked as in att_exact: a score in 16-channel partial sums,
// the output in sums over 32 keys added to the running one.
// A masked key's p is 0 and its value is not to be touched (0 x inf): tiles
// that hold masked keys and a value that is not finite go key by key
// (att_tile_masked), all others through the MFMAs.
// What bounds it: the operands' way into registers (a 1 KB wave load takes
// about 40 cycles of the CU's, which the f32 MFMAs, 32 cycles each for 2048
// FLOP, only half cover: without the loads 2 x 777 queries run at 154 TFLOP/s,
// the card's f32 rate).  Measured, a row a workgroup -> here: 16 / 8 heads, 777
// queries over 1300 keys, d 128, causal 5.33 -> 0.103 ms; one query of 32 / 8
// heads over 700 keys 128 -> 28 us (over a block's cache, whose rows hold all
// heads, 227 -> 29 under the profiler).
#define ATT_TILE_K 32  // keys a wave takes at a time
#define ATT_WAVES 8    // waves a workgroup, the key tiles among them

typedef float att_f32x4_t __attribute__((ext_vector_type(4)));

__device__ __forceinline__ float att_max4(float v) {  // over lanes l, l ^ 16, l ^ 32, l ^ 48
    const auto a = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    const float m = fmaxf(__uint_as_float(a[0]), __uint_as_float(a[1]));
    const auto b = __builtin_amdgcn_permlane32_swap(__float_as_uint(m), __float_as_uint(m), false, false);
    return fmaxf(__uint_as_float(b[0]), __uint_as_float(b[1]));
}
__device__ __forceinline__ float att_sum4(float v) {
    const auto a = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    const float m = __uint_as_float(a[0]) + __uint_as_float(a[1]);
    const auto b = __builtin_amdgcn_permlane32_swap(__float_as_uint(m), __float_as_uint(m), false, false);
    return __uint_as_float(b[0]) + __uint_as_float(b[1]);
}

// The reference r that a query's p = exp(s - r) share: n ln 2 for an integer
// n, the least at or above the running max, in two parts.  Moving it scales by
// a power of two, exactly, so running sums and the merge of the waves add no
// rounding (with r the max itself each wave's factor carried an exp's error
// into the result) -- as long as hi + lo is n ln 2 for every n: the high part,
// 355 / 512, has nine significant bits, so n times it is exact to n = 2^15,
// and n times the low part is off by 2^-23 of n 2.1e-4 at most.  (A high part
// of fifteen bits was exact to n = 512 only: scores of 600 to 3500 then cost
// 2e-5 to 3e-5 of the result.)  Past |max| = 4096 (n lo nears 1 there), and at
// infinities, r is the max and n is infinite.
struct AttRef {
    float n, hi, lo;
};
__device__ __forceinline__ AttRef att_ref(float m) {
    if (fabsf(m) < 4096.0f) {
        const float n = ceilf(m * 1.44269504088896341f);
        return AttRef{n, n * 0.693359375f, n * -2.12194440054690583e-4f};
    }
    return AttRef{INFINITY, m, 0.0f};
}
// exp(a - b), the factor of sums held at a on b; 0 where a holds none
__device__ __forceinline__ float att_rescale(const AttRef &a, const AttRef &b) {
    if (a.hi == -INFINITY) return 0.0f;
    if (a.n < INFINITY && b.n < INFINITY) return ldexpf(1.0f, (int)(a.n - b.n));
    return expf((a.hi - b.hi) + (a.lo - b.lo));
}

// One tile's part of O for 16 queries, key by key: keys a query does not see
// add nothing, whatever their values.  p of key 16 kt + 4 G + i is in lane
// (col, G).
template <int NH>
__device__ __forceinline__ void att_tile_masked(const float *vb, size_t v_tok, uint32_t dv, uint32_t j0, uint32_t kend_wg,
                                             uint32_t kend, const float p[ATT_TILE_K / 4], int lane,
                                             att_f32x4_t (*part)[4]) {
    const int col = lane & 15, G = lane >> 4;
    for (int hh = 0; hh < NH; hh++)
        for (int j = 0; j < 4; j++) part[hh][j] = att_f32x4_t{0, 0, 0, 0};
    for (uint32_t kk = 0; kk < ATT_TILE_K && j0 + kk < kend_wg; kk++) {
        float pk = 0.0f;
#pragma unroll
        for (int e = 0; e < ATT_TILE_K / 4; e++)
            if ((uint32_t)e == 4 * (kk / 16) + kk % 4) pk = p[e];
        pk = __shfl(pk, col + 16 * (int)(kk % 16 / 4), 64);
        const bool see = j0 + kk < kend;
        const float *vr = vb + (size_t)(j0 + kk) * v_tok;
        for (int hh = 0; hh < NH; hh++)
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const uint32_t c = 64 * hh + 16 * G + 4 * i;
                if (c >= dv) continue;
                const att_f32x4_t v = *(const att_f32x4_t *)(vr + c);
#pragma unroll
                for (int j = 0; j < 4; j++)
                    if (see) part[hh][j][i] += pk * v[j];
            }
    }
}

// DT: 16-channel steps of the head dim; NH: 64-channel halves of the value
// dim; QW: 16-query tiles of a workgroup, its other waves splitting the keys.
template <int DT, int NH, int QW>
__global__ void __launch_bounds__(64 * ATT_WAVES, 2) att_tile(AttArgs a) {
    constexpr int KT = ATT_TILE_K / 16, KW = ATT_WAVES / QW;
    __shared__ AttRef refs[ATT_WAVES][16];
    __shared__ float ls[ATT_WAVES][16];
    __shared__ __attribute__((aligned(16))) float ob[ATT_WAVES][16][64];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int col = lane & 15, G = lane >> 4, qw = wave % QW, kw = wave / QW;
    // the longest key ranges first, heads innermost
    const uint32_t BH = a.BH, nq = (uint32_t)((a.Sq + 16 * QW - 1) / (16 * QW));
    const uint32_t bh = blockIdx.x % BH, qi = nq - 1 - blockIdx.x / BH;
    const size_t b = bh / a.H, h = bh % a.H;
    const size_t bk = b * a.Hk + h / (a.H / a.Hk);
    const uint32_t Sq = (uint32_t)a.Sq, Skv = (uint32_t)a.Skv, d = (uint32_t)a.d, dv = (uint32_t)a.dv;
    const uint32_t qg = qi * (16 * QW), q0 = qg + 16 * qw;  // the workgroup's first query, the wave's
    const float *kb = a.k + bk * a.k_head, *vb = a.v + bk * a.v_head;
    // keys visible to query i: j < i + 1 + Skv - Sq (none below 0)
    auto visible = [&](uint32_t i) {
        if (!a.causal) return Skv;
        const int64_t e = (int64_t)i + 1 + Skv - Sq;
        return e < 0 ? 0u : e < (int64_t)Skv ? (uint32_t)e : Skv;
    };
    const uint32_t qlast = q0 + 15 < Sq ? q0 + 15 : Sq - 1;
    // a wave past the last query has no keys (and only takes part in the merge)
    const uint32_t kend_wg = q0 < Sq ? visible(qlast) : 0, kend_min = q0 < Sq ? visible(q0) : 0;
    const uint32_t iq = q0 + col < Sq ? q0 + col : Sq - 1;  // past the last: it repeats the last one, stores nothing
    const uint32_t kend = visible(iq);
    att_f32x4_t qf[DT];
    {
        const float *qr = a.q + ((size_t)bh * a.Sq + iq) * a.d;
#pragma unroll
        for (int s = 0; s < DT; s++) {
            qf[s] = *(const att_f32x4_t *)(qr + (16u * s < d ? 16 * s : 0) + 4 * G);
        }
    }
    att_f32x4_t o[NH][4];
    float m = -INFINITY, l = 0.0f;
    AttRef ref = att_ref(m);
#pragma unroll
    for (int hh = 0; hh < NH; hh++)
#pragma unroll
        for (int j = 0; j < 4; j++) o[hh][j] = att_f32x4_t{0, 0, 0, 0};
    // Rows are addressed from a uniform pointer (scalar registers) plus one
    // lane offset; a tile that runs past the range (its last) clamps each
    // lane's row to the range's last.  Keys load a tile ahead, under the
    // P V MFMAs.
    const uint32_t k_tok = (uint32_t)a.k_tok, v_tok = (uint32_t)a.v_tok;
    uint32_t vc[NH];  // this lane's first channel of a half (channels past dv repeat the first)
#pragma unroll
    for (int hh = 0; hh < NH; hh++) vc[hh] = 64u * hh + 4 * col < dv ? 64 * hh + 4 * col : 0;
    att_f32x4_t kf[KT][DT];
    auto load_k = [&](uint32_t j0) {
        const uint32_t last = kend_wg - 1 - j0;  // >= 0: the tile's first key is in the range
#pragma unroll
        for (int kt = 0; kt < KT; kt++) {
            const uint32_t row = 16 * kt + col;
            const float *kt0 = kb + (size_t)j0 * k_tok;
            const uint32_t off = (row < last ? row : last) * k_tok + 4 * G;
#pragma unroll
            for (int s = 0; s < DT; s++)
                kf[kt][s] = *(const att_f32x4_t *)(kt0 + (16u * s < d ? 16 * s : 0) + off);
        }
    };
    // One tile.  edge: some of its keys are masked for some query.  The keys
    // of the tile at jn load under the P V MFMAs (jn past the range: none).
    auto tile = [&](uint32_t j0, uint32_t jn, auto edge) {
        // values of the tile's keys, under the S MFMAs
        att_f32x4_t vf[KT][4][NH];
        {
            const uint32_t last = kend_wg - 1 - j0;
            const float *vt0 = vb + (size_t)j0 * v_tok;
#pragma unroll
            for (int kt = 0; kt < KT; kt++)
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    const uint32_t row = 16 * kt + 4 * G + i;
                    const uint32_t off = (row < last ? row : last) * v_tok;
#pragma unroll
                    for (int hh = 0; hh < NH; hh++) vf[kt][i][hh] = *(const att_f32x4_t *)(vt0 + off + vc[hh]);
                }
        }
        __builtin_amdgcn_sched_barrier(0);
        float p[4 * KT];
        {
            att_f32x4_t acc[KT];
#pragma unroll
            for (int kt = 0; kt < KT; kt++) acc[kt] = att_f32x4_t{0, 0, 0, 0};
#pragma unroll
            for (int s = 0; s < DT; s++)
                if (16u * s < d) {
                    att_f32x4_t sp[KT];  // 16-term partial sums, as att_exact's
#pragma unroll
                    for (int kt = 0; kt < KT; kt++) sp[kt] = att_f32x4_t{0, 0, 0, 0};
#pragma unroll
                    for (int e = 0; e < 4; e++)
#pragma unroll
                        for (int kt = 0; kt < KT; kt++)
                            sp[kt] = __builtin_amdgcn_mfma_f32_16x16x4f32(kf[kt][s][e], qf[s][e], sp[kt], 0, 0, 0);
#pragma unroll
                    for (int kt = 0; kt < KT; kt++) acc[kt] += sp[kt];
                }
#pragma unroll
            for (int kt = 0; kt < KT; kt++)
#pragma unroll
                for (int e = 0; e < 4; e++) p[4 * kt + e] = acc[kt][e] * a.scale;
        }
        if (!edge) load_k(jn);
        __builtin_amdgcn_sched_barrier(0);
        bool slow = false;
        if constexpr (edge) {
#pragma unroll
            for (int e = 0; e < 4 * KT; e++)
                if (j0 + 16 * (e / 4) + 4 * G + e % 4 >= kend) p[e] = -INFINITY;
            bool fin = true;
#pragma unroll
            for (int kt = 0; kt < KT; kt++)
#pragma unroll
                for (int i = 0; i < 4; i++)
#pragma unroll
                    for (int hh = 0; hh < NH; hh++)
#pragma unroll
                        for (int e = 0; e < 4; e++) fin = fin & (fabsf(vf[kt][i][hh][e]) < INFINITY);
            slow = !__all(fin);
        }
        float cmax = -INFINITY;
#pragma unroll
        for (int e = 0; e < 4 * KT; e++) cmax = fmaxf(cmax, p[e]);
        const float mn = fmaxf(m, att_max4(cmax));
        if (__any(mn > m)) {  // some query's max moved
            const AttRef to = mn > m ? att_ref(mn) : ref;
            const float alpha = att_rescale(ref, to);
            l *= alpha;
#pragma unroll
            for (int hh = 0; hh < NH; hh++)
#pragma unroll
                for (int j = 0; j < 4; j++) o[hh][j] *= alpha;
            m = mn;
            ref = to;
        }
        float part = 0.0f;
#pragma unroll
        for (int e = 0; e < 4 * KT; e++) {
            const float x = expf((p[e] - ref.hi) - ref.lo);
            p[e] = p[e] == -INFINITY ? 0.0f : x;
            part += p[e];
        }
        l += part;
        if constexpr (edge) {
            if (slow) {
                att_f32x4_t sum[NH][4];
                att_tile_masked<NH>(vb, a.v_tok, dv, j0, kend_wg, kend, p, lane, sum);
#pragma unroll
                for (int hh = 0; hh < NH; hh++)
#pragma unroll
                    for (int j = 0; j < 4; j++) o[hh][j] += sum[hh][j];
                return;
            }
        }
#pragma unroll
        for (int hh = 0; hh < NH; hh++) {
            att_f32x4_t sum[4];
#pragma unroll
            for (int j = 0; j < 4; j++) sum[j] = att_f32x4_t{0, 0, 0, 0};
#pragma unroll
            for (int kt = 0; kt < KT; kt++)
#pragma unroll
                for (int i = 0; i < 4; i++)
#pragma unroll
                    for (int j = 0; j < 4; j++)
                        sum[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(vf[kt][i][hh][j], p[4 * kt + i], sum[j], 0, 0, 0);
#pragma unroll
            for (int j = 0; j < 4; j++) o[hh][j] += sum[j];
        }
    };
    // the tiles every query sees in full, then the edge's (two at most)
    uint32_t j0 = kw * ATT_TILE_K;
    if (j0 + ATT_TILE_K <= kend_min) {
        load_k(j0);
        for (; j0 + ATT_TILE_K <= kend_min; j0 += KW * ATT_TILE_K) {
            const uint32_t jn = j0 + KW * ATT_TILE_K;
            tile(j0, jn < kend_wg ? jn : j0, std::false_type{});
        }
    }
    for (; j0 < kend_wg; j0 += KW * ATT_TILE_K) {
        load_k(j0);
        tile(j0, 0, std::true_type{});
    }
    // merge the waves: every wave's output and sum on the largest reference
    const float lsum = att_sum4(l);
    if (G == 0) {
        refs[wave][col] = ref;
        ls[wave][col] = lsum;
    }
    __syncthreads();
    // the largest reference of query q of the workgroup's query tile t
    auto largest = [&](int t, int q) {
        AttRef r = refs[t][q];
#pragma unroll
        for (int w = 1; w < KW; w++) {
            const AttRef x = refs[w * QW + t][q];
            if (x.hi > r.hi) r = x;
        }
        return r;
    };
    const float f = att_rescale(ref, largest(qw, col));
#pragma unroll
    for (int hh = 0; hh < NH; hh++) {
        if (hh) __syncthreads();  // the first half's sums are read
#pragma unroll
        for (int i = 0; i < 4; i++) {
            att_f32x4_t v;
#pragma unroll
            for (int j = 0; j < 4; j++) v[j] = o[hh][j][i] * f;
            *(att_f32x4_t *)&ob[wave][col][16 * G + 4 * i] = v;
        }
        __syncthreads();
        for (int x = tid; x < QW * 16 * 64; x += 64 * ATT_WAVES) {
            const int t = x / 1024, q = x / 64 % 16, c = x % 64;
            const uint32_t i = qg + 16 * t + q;
            if (i >= Sq || 64u * hh + c >= dv) continue;
            const AttRef M = largest(t, q);
            float L = 0.0f, sum = 0.0f;
#pragma unroll
            for (int w = 0; w < KW; w++) {
                L += ls[w * QW + t][q] * att_rescale(refs[w * QW + t][q], M);
                sum += ob[w * QW + t][q][c];
            }
            a.out[((size_t)bh * a.Sq + i) * a.dv + 64 * hh + c] = sum / L;
        }
    }
}

// Whether att_tile serves the call: 16-byte rows of queries, keys and values.
static bool att_tile_fits(const AttArgs &a) {
    return a.d <= 128 && a.dv <= 128 && (a.d | a.dv) % 16 == 0 && (a.k_tok | a.v_tok | a.k_head | a.v_head) % 4 == 0 &&
           a.k_tok <= 0x1000000u && a.v_tok <= 0x1000000u &&
           (((uintptr_t)a.q | (uintptr_t)a.k | (uintptr_t)a.v) & 15) == 0 && a.Sq <= 0x40000000u &&
           a.Skv <= 0x40000000u;
}

// Whether att_exact is the faster of the two for a shape that att_tile fits: a
// few queries of many heads over few keys.  A workgroup of att_tile has a CU
// to itself and takes 3.7 us however few keys there are (value dims past 64:
// 7.5 us), while the rows of att_exact share one and cost by their keys.
// Measured over 3150 shapes (heads 32 to 16384, queries 1 to 16, keys 1 to
// 128, d 16 to 128), row kernel against tiles, us: 4096 heads of d 64, one
// query, 1 key 18, 66; 32 keys 48, 68; 48 keys 82, 75; two queries, 16 keys 63,
// 72; four queries, 8 keys 93, 69; d 128, one query, 32 keys 68, 124; 48 keys
// 125, 140; 64 keys 162, 136.  Up to 256 heads every workgroup of att_tile has a CU
// at once and only rows of 16 channels or fewer are better off by themselves.
// (Heads: batches times heads.)
static bool att_rows_faster(const AttArgs &a, size_t B) {
    if (a.Sq > 16 || a.Skv > 64) return false;
    const size_t BH = B * a.H, w = (a.d + a.dv) / 2;
    const bool small = a.d <= 64 && a.dv <= 64;
    if (BH <= 256) return w <= 16 && a.Skv <= 8 && BH * a.Sq <= 1024;
    if (BH < 768 && a.Skv * w > (small ? 512 : 2048)) return false;
    return a.Sq * (20 + w + a.Skv * (2 + w / 16)) <= (small ? 360 : 730);
}

static int att_tile_launch(AttArgs a, size_t B, hipStream_t st) {
    a.BH = (uint32_t)(B * a.H);
    // More query tiles a workgroup share each key's and value's way through
    // the L1 but leave fewer workgroups: 16 / 8 heads, d 128, 1300 keys (us
    // for 1, 2, 4 tiles): 777 queries causal 124, 107, 127; 2 x 777 not causal
    // 291, 279, 255; 400 queries of d 80 over 700 keys 56, 47, 47; 64 queries
    // 44 each.
    // Tiles that hold no query leave their waves idle, so no more of them than
    // there are queries for where the keys need the waves: 4096 single queries
    // (us for 1 and 4 tiles) over 32 keys of d 64 68, 72; 64 keys 72, 91; 128
    // keys 82, 137; 16 queries of 1024 heads over 32 keys 25, 21 (the merge of
    // eight waves' outputs); 64 keys 27, 28.
    int qw = div_ceil(a.Sq, 64) * B * a.H >= 400 ? 4 : div_ceil(a.Sq, 32) * B * a.H >= 150 ? 2 : 1;
    if (a.Skv >= 32 + 6 * a.Sq)
        while (qw > 1 && 8 * (size_t)qw >= a.Sq) qw /= 2;
    const size_t grid = div_ceil(a.Sq, 16 * (size_t)qw) * B * a.H;
    if (grid > 0x7FFFFFFFull) return fail(QBK_ERR_VALIDATION, "attention: too many query tiles for one launch");
    const bool small = a.d <= 64 && a.dv <= 64;
#define ATT_GO(QW)                                                                                        \
    if (small)                                                                                            \
        hipLaunchKernelGGL((att_tile<4, 1, QW>), dim3((unsigned)grid), dim3(64 * ATT_WAVES), 0, st, a);   \
    else                                                                                                  \
        hipLaunchKernelGGL((att_tile<8, 2, QW>), dim3((unsigned)grid), dim3(64 * ATT_WAVES), 0, st, a);
    if (qw == 4) {
        ATT_GO(4)
    } else if (qw == 2) {
        ATT_GO(2)
    } else {
        ATT_GO(1)
    }
#undef ATT_GO
    QBK_HIP(hipGetLastError());
    return QBK_OK;
}

// gpu_attention.rs:466-509: validation in the reference's order and words,
// then the u32 index ceiling of its device face.
static int validate_exact(const qbk_attn_shape *s, const size_t *lens) {
    if (!s) return fail(QBK_ERR_VALIDATION, "null shape");
    if (s->batch == 0 || s->n_heads == 0 || s->n_kv_heads == 0)
        return fail(QBK_ERR_VALIDATION, "attention requires non-empty batch and head dimensions");
    if (s->n_heads % s->n_kv_heads != 0)
        return fail(QBK_ERR_VALIDATION, fmt("n_kv_heads must divide n_heads: n_heads=%zu, n_kv_heads=%zu",
                                            s->n_heads, s->n_kv_heads));
    if (s->seq_q == 0 || s->seq_kv == 0 || s->head_dim == 0 || s->val_dim == 0)
        return fail(QBK_ERR_VALIDATION, "attention requires non-empty sequence and head dimensions");
    const size_t eq = s->batch * s->n_heads * s->seq_q * s->head_dim;
    const size_t ek = s->batch * s->n_kv_heads * s->seq_kv * s->head_dim;
    const size_t ev = s->batch * s->n_kv_heads * s->seq_kv * s->val_dim;
    const std::string dbg = fmt("AttentionShape { batch: %zu, n_heads: %zu, n_kv_heads: %zu, seq_q: %zu, seq_kv: "
                                "%zu, head_dim: %zu, val_dim: %zu }",
                                s->batch, s->n_heads, s->n_kv_heads, s->seq_q, s->seq_kv, s->head_dim, s->val_dim);
    if (lens) {
        if (lens[0] != eq)
            return fail(QBK_ERR_VALIDATION, fmt("query must hold %zu values for %s, got %zu", eq, dbg.c_str(), lens[0]));
        if (lens[1] != ek)
            return fail(QBK_ERR_VALIDATION, fmt("key must hold %zu values for %s, got %zu", ek, dbg.c_str(), lens[1]));
        if (lens[2] != ev)
            return fail(QBK_ERR_VALIDATION, fmt("value must hold %zu values for %s, got %zu", ev, dbg.c_str(), lens[2]));
    }
    size_t largest = eq > ek ? eq : ek;
    largest = largest > ev ? largest : ev;
    if ((uint64_t)largest > 0xFFFFFFFFull)
        return fail(QBK_ERR_VALIDATION, "attention inputs exceed the device u32 index ceiling (4294967295); use "
                                        "the CPU reference face");
    if (s->head_dim > ATT_MAXD || s->val_dim > ATT_MAXD)
        return fail(QBK_ERR_VALIDATION, fmt("attention on this device supports head_dim and val_dim up to %d, "
                                            "got head_dim=%zu, val_dim=%zu",
                                            ATT_MAXD, s->head_dim, s->val_dim));
    return QBK_OK;
}

static int launch_exact(const qbk_attn_shape *s, const float *q, const float *k, const float *v, int causal,
                        float *out, hipStream_t st) {
    AttArgs a{q, k, v, out, s->n_heads, s->n_kv_heads, s->seq_q, s->seq_kv, s->head_dim, s->val_dim, causal ? 1 : 0,
              1.0f / sqrtf((float)s->head_dim), s->head_dim, s->seq_kv * s->head_dim, s->val_dim,
              s->seq_kv * s->val_dim};
    const size_t rows = s->batch * s->n_heads * s->seq_q;
    if (rows > 0x7FFFFFFFull) return fail(QBK_ERR_VALIDATION, "attention: too many query rows for one launch");
    if (att_tile_fits(a) && !att_rows_faster(a, s->batch)) return att_tile_launch(a, s->batch, st);
    hipLaunchKernelGGL(att_exact, dim3((unsigned)rows), dim3(ATT_THREADS), 0, st, a);
    QBK_HIP(hipGetLastError());
    return QBK_OK;
}

// One query position of every head over rows 0 .. rows - 1 of a decoder
// block's row-major cache (f32 [rows][Hk hd] keys and values): the engine's
// tiled decode face (engine/mod.rs:1041-1067: seq_q = 1, so every cached key
// is visible), reading the cache in place rather than gathered head-major.
int attention_exact_cache(const float *q, const float *kc, const float *vc, size_t H, size_t Hk, size_t hd,
                          size_t rows, float *out, hipStream_t st) {
    if (rows == 0 || H == 0 || Hk == 0 || H % Hk != 0 || hd == 0 || hd > ATT_MAXD)
        return fail(QBK_ERR_VALIDATION, "exact cache attention: bad shape");
    AttArgs a{q, kc, vc, out, H, Hk, 1, rows, hd, hd, 0, 1.0f / sqrtf((float)hd), Hk * hd, hd, Hk * hd, hd};
    if (att_tile_fits(a) && !att_rows_faster(a, 1)) return att_tile_launch(a, 1, st);
    hipLaunchKernelGGL(att_exact, dim3((unsigned)H), dim3(ATT_THREADS), 0, st, a);
    QBK_HIP(hipGetLastError());
    return QBK_OK;
}

}  // namespace qbk

using namespace qbk;

extern "C" {

int qbk_attention(qbk_ctx *ctx, const qbk_attn_shape *shape, const float *q, size_t q_len, const float *k,
                  size_t k_len, const float *v, size_t v_len, int causal, float *out) {
    int rc;
    const size_t lens[3] = {q_len, k_len, v_len};
    if ((rc = validate_exact(shape, lens))) return rc;
    if (!q || !k || !v || !out) return fail(QBK_ERR_VALIDATION, "null argument");
    if ((rc = bind(ctx))) return rc;
    const size_t no = shape->batch * shape->n_heads * shape->seq_q * shape->val_dim;
    DevBuf dq, dk, dv, dout;
    CallStream cs;
    if ((rc = dq.alloc(q_len * 4)) || (rc = dk.alloc(k_len * 4)) || (rc = dv.alloc(v_len * 4)) ||
        (rc = dout.alloc(no * 4)) || (rc = cs.create()))
        return rc;
    QBK_HIP(hipMemcpyAsync(dq.p, q, q_len * 4, hipMemcpyHostToDevice, cs.s));
    QBK_HIP(hipMemcpyAsync(dk.p, k, k_len * 4, hipMemcpyHostToDevice, cs.s));
    QBK_HIP(hipMemcpyAsync(dv.p, v, v_len * 4, hipMemcpyHostToDevice, cs.s));
    if ((rc = launch_exact(shape, (const float *)dq.p, (const float *)dk.p, (const float *)dv.p, causal,
                           (float *)dout.p, cs.s)))
        return rc;
    QBK_HIP(hipMemcpyAsync(out, dout.p, no * 4, hipMemcpyDeviceToHost, cs.s));
    QBK_HIP(hipStreamSynchronize(cs.s));
    return QBK_OK;
}

int qbk_attention_dev(qbk_ctx *ctx, const qbk_attn_shape *shape, const float *q, const float *k, const float *v,
                      int causal, float *out, void *stream) {
    int rc;
    if ((rc = validate_exact(shape, nullptr))) return rc;
    if (!q || !k || !v || !out) return fail(QBK_ERR_VALIDATION, "null argument");
    if ((rc = bind(ctx))) return rc;
    return launch_exact(shape, q, k, v, causal, out, (hipStream_t)stream);
}

}  // extern "C"
