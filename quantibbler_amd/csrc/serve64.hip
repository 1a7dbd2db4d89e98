// serve64.hip -- the factor linear at fp32 serving (engine/mod.rs:393-436,
// PackedLayer::apply), one token:
//
//   z = f64(s2 * x);  t = Vb^T z;  u = Ub t  (f64, in element order);
//   y = f32(u) * s1 + bias
//
// The reference's contract pins the order of each row's sum, so a row is one
// chain of K dependent f64 additions however many lanes there are, and the
// chain is the time (a decoder block's projections, 4096 wide with an FFN of
// 14336 at 0.55 bit a weight, hold 32,285 steps one after another).  On the
// VALU a step is the addition (6.3 cycles of a lone wave) and the two
// operations that put the sign on (5.4 each), 17 in all; a thread per row
// over row bitplanes took about 80.  Here the chain runs on
// v_mfma_f64_4x4x4_4b_f64, of which a dependent one takes 21-23 cycles for
// four steps.  The instruction adds its four products one after another, k
// ascending, each with its own rounding -- checked on gfx950 bit for bit
// against an fma chain (2048 steps, exponents over 2^40), and by the tests
// against the oracle -- and a product by +-1 is exact, so the sums are the
// reference's.
//
// A wave takes 16 rows (the MFMA's 4 blocks of 4): A = their signs as +-1.0,
// lane (row % 16, G) holding k = 4 s + G of step s; B = z, the same in all
// four columns.  VALU work does not run under an f64 MFMA (each interleaved
// operation cost its own time and the MFMA's wait again: 42-50 cycles a
// step of four), so the signs of eight MFMAs are formed at once, one byte
// operation each.  Signs and z go to LDS by direct loads, a chunk of 16
// slices (2048 k) ahead.
// Measured: stage 1 of a 4096 x 14336 layer of rank 1733 (14336 steps) 65 us,
// 4.6 ns a step; the decoder block at fp32 serving over 700 cached rows, exact
// attention, 4.82 -> 0.233 ms a token.
#include <mutex>

#include "factor_internal.h"

#pragma clang fp contract(off)

namespace qbk {

// Signs of a stage for these kernels: word [row / 16][k / 128][lane], lane
// (row % 16, G): bit 8 (s % 4) + s / 4 set when row's sign at k = 4 s + G is
// -1, so that (w << (7 - g)) & 0x80808080 holds the sign bits of steps 4 g ..
// 4 g + 3 on top of its bytes.  Formed on the device from the fp4 decode
// layout (repack_q4) on a layer's first fp32-serving call.
__global__ void q4_to_f64(const uint32_t *q4, uint32_t n_groups, uint32_t ns, uint32_t *out) {
    const size_t idx = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= (size_t)n_groups * ns * 64) return;
    const uint32_t lane = (uint32_t)(idx % 64), G = lane / 16, l15 = lane % 16;
    const size_t s = idx / 64 % ns, rg = idx / 64 / ns;  // 16-row group rg: row tile rg % 4 of 64-row group rg / 4
    uint32_t w[4];
    for (int g = 0; g < 4; g++) w[g] = q4[((rg / 4 * ns + s) * 64 + 16 * g + l15) * 4 + rg % 4];
    uint32_t o = 0;
    for (uint32_t st = 0; st < 32; st++) {
        const uint32_t k = 4 * st + G;  // the inverse of kq4: k = 64 (g & 1) + 32 (e >> 4) + 16 (g >> 1) + e % 16
        const uint32_t g = 2 * ((k >> 4) & 1) + ((k >> 6) & 1), e = 16 * ((k >> 5) & 1) + (k & 15);
        o |= ((w[g] >> (4 * (e & 7) + (e >> 3))) & 1u) << (8 * (st % 4) + st / 4);
    }
    out[idx] = o;
}

#define F64_CH 16  // slices of 128 k a chunk

// The sign of the +-1.0 V: its top byte 0x3f with the sign bit that byte B of
// BITS holds, its other bytes kept.
#define F64_SIGN(V, BITS, B)                                                                                 \
    {                                                                                                        \
        union {                                                                                              \
            double d;                                                                                        \
            uint32_t u[2];                                                                                   \
        } x_;                                                                                                \
        x_.d = V;                                                                                            \
        asm volatile("v_or_b32_sdwa %0, %1, %2 dst_sel:BYTE_3 dst_unused:UNUSED_PRESERVE src0_sel:BYTE_0 src1_sel:BYTE_" #B \
            : "+v"(x_.u[1])                                                                                  \
            : "v"(top), "v"(BITS));                                                                          \
        V = x_.d;                                                                                            \
    }

struct F64Stage {
    const uint32_t *bits;
    const double *z;      // [ns] slices in f64_pos order, zero past the valid K
    double *t;            // stage 1: out, f64_pos order, zero past rows (to a multiple of 128)
    float *y;             // stage 2: out
    const float *s1, *bias, *resid;
    uint32_t ns, rows, wg0;
};
struct F64Args {
    F64Stage l[F64_MAXL];
};

template <bool OUT>
__global__ void __launch_bounds__(64) f64_stage(F64Args a) {
    __shared__ __attribute__((aligned(16))) uint8_t wl[2][F64_CH * 256], zl[2][F64_CH * 1024];
    const int lane = threadIdx.x, G = lane >> 4;
    int li = 0;
#pragma unroll
    for (int i = 1; i < F64_MAXL; i++)
        if (blockIdx.x >= a.l[i].wg0) li = i;
    const F64Stage L = a.l[li];
    const uint32_t rg = blockIdx.x - L.wg0, ns = L.ns;
    // D: lane 16 i + 4 b + j holds row 4 b + i of column j
    const uint32_t row = 16 * rg + (lane & 12) + G;
    double acc = 0.0;
    if (OUT || 16 * rg < L.rows) {
        const uint32_t *bits = L.bits + (size_t)rg * ns * 64 + lane * 4;
        const double *z = L.z + lane * 2;
        // +-1.0 of the next eight steps, in pairs whose other seven bytes stay
        double sg[8];
        uint32_t top = 0x3f;
#pragma unroll
        for (int j = 0; j < 8; j++) {
            sg[j] = 1.0;
            asm("" : "+v"(sg[j]));
        }
        asm("" : "+v"(top));
        // a chunk's signs (1 KB: 4 slices) and z (1 KB a slice); the last
        // piece of signs may run on into the next group's (the array is padded)
        auto issue = [&](uint32_t c, int buf) {
            const uint32_t s0 = c * F64_CH, cs = ns - s0 < F64_CH ? ns - s0 : F64_CH;
#pragma unroll
            for (uint32_t p = 0; p < F64_CH / 4; p++)
                if (4 * p < cs)
                    __builtin_amdgcn_global_load_lds((const void *)(bits + (size_t)(s0 + 4 * p) * 64),
                                                     (__attribute__((address_space(3))) void *)&wl[buf][p * 1024], 16, 0, 0);
#pragma unroll
            for (uint32_t p = 0; p < F64_CH; p++)
                if (p < cs)
                    __builtin_amdgcn_global_load_lds((const void *)(z + (size_t)(s0 + p) * 128),
                                                     (__attribute__((address_space(3))) void *)&zl[buf][p * 1024], 16, 0, 0);
        };
        const uint32_t nc = (ns + F64_CH - 1) / F64_CH;
        issue(0, 0);
        for (uint32_t c = 0; c < nc; c++) {
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            __syncthreads();  // one wave: the chunk's direct loads have landed
            const int buf = (int)(c & 1);
            if (c + 1 < nc) issue(c + 1, buf ^ 1);
            const uint32_t cs = ns - c * F64_CH < F64_CH ? ns - c * F64_CH : F64_CH;
            const double2 *zp = (const double2 *)zl[buf] + G;
            const uint32_t *wp = (const uint32_t *)wl[buf] + lane;
            double2 za[8], zb[8];
            uint32_t w = wp[0];
#pragma unroll
            for (int t = 0; t < 8; t++) za[t] = zp[4 * t];
            auto step = [&](const double2 *zz, int g0) {  // steps 4 g0 .. 4 g0 + 15
#pragma unroll
                for (int q = 0; q < 2; q++) {
                    const uint32_t b0 = (w << (7 - g0 - 2 * q)) & 0x80808080u, b1 = (w << (6 - g0 - 2 * q)) & 0x80808080u;
                    F64_SIGN(sg[0], b0, 0) F64_SIGN(sg[1], b0, 1) F64_SIGN(sg[2], b0, 2) F64_SIGN(sg[3], b0, 3)
                    F64_SIGN(sg[4], b1, 0) F64_SIGN(sg[5], b1, 1) F64_SIGN(sg[6], b1, 2) F64_SIGN(sg[7], b1, 3)
                    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                    for (int j = 0; j < 8; j++)
                        acc = __builtin_amdgcn_mfma_f64_4x4x4f64(sg[j], j & 1 ? zz[4 * q + j / 2].y : zz[4 * q + j / 2].x, acc, 0,
                                                                 0, 0);
                    __builtin_amdgcn_sched_barrier(0);
                }
            };
            for (uint32_t sl = 0; sl < cs; sl++) {
#pragma unroll
                for (int t = 0; t < 8; t++) zb[t] = zp[64 * sl + 4 * (8 + t)];
                __builtin_amdgcn_sched_barrier(0);
                step(za, 0);
                const uint32_t sn = sl + 1 < cs ? sl + 1 : sl;
                const uint32_t wn = wp[64 * sn];
#pragma unroll
                for (int t = 0; t < 8; t++) za[t] = zp[64 * sn + 4 * t];
                __builtin_amdgcn_sched_barrier(0);
                step(zb, 4);
                w = wn;
            }
        }
    }
    if (lane & 3) return;  // column 0 of four equal ones
    if constexpr (OUT) {
        if (row >= L.rows) return;
        float y = (float)acc * L.s1[row] + L.bias[row];
        if (L.resid) y = y + L.resid[row];
        L.y[row] = y;
    } else {
        L.t[f64_pos(row)] = row < L.rows ? acc : 0.0;
    }
}

// z = f64(s2 * x), an f32 product widened, zero past din
__global__ void f64_in(const float *x, const float *s2, double *z, uint32_t din) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= ((din + 127) & ~127u)) return;
    z[f64_pos(i)] = i < din ? (double)(s2[i] * x[i]) : 0.0;
}

int factor_f64_ready(const qbk_factor *L, hipStream_t s) {
    static std::mutex mu;
    std::lock_guard<std::mutex> lock(mu);
    if (L->u_f64) return QBK_OK;
    qbk_factor *M = const_cast<qbk_factor *>(L);
    void *pu = nullptr, *pv = nullptr;
    const uint32_t gu = (uint32_t)(L->dout_p / 16), gv = (uint32_t)(L->r_p / 16);
    const uint32_t nu = (uint32_t)(L->r_q / 128), nv = (uint32_t)(L->din_q / 128);
    const size_t wu = (size_t)gu * nu * 64, wv = (size_t)gv * nv * 64;
    // 1 KB past the end: a chunk's last piece reads whole fours of slices
    QBK_HIP(hipMalloc(&pu, wu * 4 + 1024));
    M->allocs.push_back(pu);
    QBK_HIP(hipMalloc(&pv, wv * 4 + 1024));
    M->allocs.push_back(pv);
    hipLaunchKernelGGL(q4_to_f64, dim3((unsigned)div_ceil(wu, 256)), dim3(256), 0, s, L->u_q4, gu, nu, (uint32_t *)pu);
    QBK_HIP(hipGetLastError());
    hipLaunchKernelGGL(q4_to_f64, dim3((unsigned)div_ceil(wv, 256)), dim3(256), 0, s, L->vt_q4, gv, nv, (uint32_t *)pv);
    QBK_HIP(hipGetLastError());
    QBK_HIP(hipStreamSynchronize(s));
    M->vt_f64 = (uint32_t *)pv;
    M->u_f64 = (uint32_t *)pu;
    return QBK_OK;
}

size_t factor_f64_scratch(const qbk_factor *const *L, int n) {
    size_t d = 0;
    for (int i = 0; i < n; i++) d += L[i]->din_q + L[i]->r_q;
    return d;
}

double *factor_f64_z(const qbk_factor *const *L, int i, double *scratch) {
    for (int k = 0; k < i; k++) scratch += L[k]->din_q + L[k]->r_q;
    return scratch;
}

int factor_f64_staged(const qbk_factor *const *L, int n, float *const *y, const float *resid, double *scratch,
                      hipStream_t s) {
    F64Args a{}, b{};
    uint32_t g1 = 0, g2 = 0;
    for (int i = 0; i < F64_MAXL; i++) {
        if (i >= n) {
            a.l[i].wg0 = b.l[i].wg0 = 0xffffffffu;
            continue;
        }
        double *z = factor_f64_z(L, i, scratch), *t = z + L[i]->din_q;
        a.l[i] = F64Stage{L[i]->vt_f64, z, t, nullptr, nullptr, nullptr, nullptr, (uint32_t)(L[i]->din_q / 128),
                          (uint32_t)L[i]->r, g1};
        b.l[i] = F64Stage{L[i]->u_f64, t, nullptr, y[i], L[i]->s1, L[i]->bias, resid, (uint32_t)(L[i]->r_q / 128),
                          (uint32_t)L[i]->dout, g2};
        g1 += (uint32_t)(L[i]->r_q / 16);
        g2 += (uint32_t)div_ceil(L[i]->dout, 16);
    }
    hipLaunchKernelGGL(f64_stage<false>, dim3(g1), dim3(64), 0, s, a);
    QBK_HIP(hipGetLastError());
    hipLaunchKernelGGL(f64_stage<true>, dim3(g2), dim3(64), 0, s, b);
    QBK_HIP(hipGetLastError());
    return QBK_OK;
}

int factor_f64_run(const qbk_factor *L, const float *x, float *y, double *scratch, hipStream_t s) {
    hipLaunchKernelGGL(f64_in, dim3((unsigned)div_ceil(L->din_q, 256)), dim3(256), 0, s, x, (const float *)L->s2,
                       factor_f64_z(&L, 0, scratch), (uint32_t)L->din);
    QBK_HIP(hipGetLastError());
    return factor_f64_staged(&L, 1, &y, nullptr, scratch, s);
}

}  // namespace qbk
