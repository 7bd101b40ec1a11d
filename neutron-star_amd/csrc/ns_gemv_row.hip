// ns_gemv_row.hip -- decode (batch 1) dequant-fused GEMV on ROW_MAJOR tensors, for gfx950.
//
// Replaces gemma_q4k_mv_fast / gemma_q6k_mv_fast (metal/gemma4.metal:55-100, selected by matmul batch==1
// at metal_engine.mm:272) for the tensors that stay in GGUF order: the attention projections and an
// lm-head that was not re-tiled.
//
// What bounds it: a 4-9 MB projection is over before the memory system is saturated, so the launch
// ramp and one round trip of loads are most of the time.  The slab kernel (lane = row) reads 64 rows
// with 16 bytes each per load instruction, 64 or more cache lines apart, and runs one super-block per
// wave in sequence with a cross-wave sum: 18-22 us for the 2,048- and 4,096-row projections.  Here a
// row's blocks lie across the lanes: a lane takes one 16-byte qs chunk (Q4_K: 8 lanes per
// super-block) or the 48 bytes of one 64-weight quarter (Q6_K: 4 lanes per super-block), so a load
// instruction reads contiguous bytes, a wave covers 16 super-blocks of a row in one round of loads and
// keeps its share of x (64 values per lane) in registers over all its rows.  Rows longer than 16
// super-blocks split over kw waves of the workgroup, whose sums meet in LDS in wave order.
//
// The arithmetic per weight is the slab kernel's (ns_gemv.hip): quants as fp16 subnormals into fp32
// mixed-precision FMAs, scales and mins once per 16 values of x.  Lane sums are added in a fixed
// order, so results are deterministic.
#include <type_traits>

#include "ns_internal.hpp"
#include "ns_quant.hpp"

namespace ns {
namespace {

constexpr int kSpan = 16;  // super-blocks of a row one wave covers

template <int CTRL>
__device__ __forceinline__ float dpp_add(float v) {
    return v + __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, v), CTRL, 0xF, 0xF, false));
}
// Sum over the wave, wave-uniform: lane ^ 1, ^ 2, the other quad, the other half of 16 lanes (DPP
// quad_perm, row_half_mirror, row_mirror), then the four rows of 16 lanes.
__device__ __forceinline__ float wave_sum(float v) {
    v = dpp_add<0xB1>(v);
    v = dpp_add<0x4E>(v);
    v = dpp_add<0x141>(v);
    v = dpp_add<0x140>(v);
    const auto rl = [&](int l) { return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), l)); };
    return (rl(0) + rl(16)) + (rl(32) + rl(48));
}

// One lane's bytes of one row.
struct RowQ4 {
    u32x4 hdr[2], qs[2];  // super-blocks lane/8 and 8 + lane/8 of the wave's span, chunk 1 + lane%8
};
struct RowQ6 {
    // super-block lane/4, half h = lane%4 / 2, t = lane%2: ql chunks 4h+t and 4h+2+t, qh chunk 8+2h+t and
    // the scales, each as the dword-aligned 16 bytes at or below it and the next dword
    u32x4 c[4];
    uint32_t n[4], d;
};

// MW: most waves per workgroup; R rows per step.  Four waves: two rows per step and the next step's in
// flight.  Rows of more than 64 super-blocks take up to 16 waves (128 VGPRs each): one row at a time.
template <int TYPE, int MW, int R>
__global__ __launch_bounds__(64 * MW) void gemv_row_kernel(
    const uint8_t *__restrict__ w, const float *__restrict__ x, float *__restrict__ out, uint32_t rows, uint32_t nb,
    uint32_t kw, uint32_t steps) {
    constexpr bool Q4 = TYPE == Q4_K;
    __shared__ float part[2][MW][R];
    const uint32_t lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t rg = (blockDim.x >> 6) / kw, wr = wave / kw, wkk = wave % kw;  // row groups; this wave's
    const uint32_t b0 = wkk * kSpan;
    // rows of step s: first(s) .. +R-1; consecutive steps of one wave are a whole grid apart
    auto first = [&](uint32_t s) { return ((s * gridDim.x + blockIdx.x) * rg + wr) * R; };

    // Super-blocks past the row's end (the last wave's span) re-read the row's last one and add nothing.
    constexpr int NB = Q4 ? 2 : 1;
    uint32_t blk[NB];
    bool in[NB];
#pragma unroll
    for (int k = 0; k < NB; ++k) {
        const uint32_t b = b0 + (Q4 ? 8 * uint32_t(k) + (lane >> 3) : lane >> 2);
        in[k] = b < nb;
        blk[k] = __builtin_elementwise_min(b, nb - 1);
    }
    using Row = typename std::conditional<Q4, RowQ4, RowQ6>::type;
    auto load = [&](uint32_t r, Row &q) {
        const uint64_t row = __builtin_elementwise_min(r, rows - 1);
        if constexpr (Q4) {
#pragma unroll
            for (int k = 0; k < 2; ++k) {
                const u32x4 *p = reinterpret_cast<const u32x4 *>(w + (row * nb + blk[k]) * kQ4Bytes);
                q.hdr[k] = p[0];
                q.qs[k] = p[1 + (lane & 7)];
            }
        } else {
            const uint32_t h = (lane >> 1) & 1, t = lane & 1;
            const uint8_t *p = w + (row * nb + blk[0]) * kQ6Bytes;
            const uint8_t *al = reinterpret_cast<const uint8_t *>(reinterpret_cast<uintptr_t>(p) & ~uintptr_t(3));
            // the next dword of a piece is only used (and then inside the block) when the block is
            // 2 bytes past a dword; otherwise the piece's own last dword is read again
            const uint32_t nx = reinterpret_cast<uintptr_t>(p) & 2 ? 16 : 12;
            const uint32_t off[4] = {16 * (4 * h + t), 16 * (4 * h + 2 + t), 16 * (8 + 2 * h + t), 192};
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                const uint32_t *s = reinterpret_cast<const uint32_t *>(al + off[k]);
                q.c[k] = u32x4{s[0], s[1], s[2], s[3]};
                q.n[k] = *reinterpret_cast<const uint32_t *>(al + off[k] + nx);
            }
            q.d = *reinterpret_cast<const uint16_t *>(p + 208);
        }
    };

    // ---- the first rows in flight, then the lane's x
    constexpr bool PRE = MW <= 4;
    Row cur[R], nxt[PRE ? R : 1];
#pragma unroll
    for (int i = 0; i < R; ++i) load(first(0) + uint32_t(i), cur[i]);
    __builtin_amdgcn_sched_barrier(0);
    float xv[64];   // Q4_K [k][low | high nibbles][16]; Q6_K [quarter][16]
    float xs[4];    // their sums over 16
#pragma unroll
    for (int g = 0; g < 4; ++g) {
        const uint32_t base = Q4 ? blk[(g >> 1) % NB] * kQK + 64 * ((lane & 7) >> 1) + 32 * uint32_t(g & 1) + 16 * (lane & 1)
                                 : blk[0] * kQK + 128 * ((lane >> 1) & 1) + 32 * uint32_t(g) + 16 * (lane & 1);
        const float4 *p = reinterpret_cast<const float4 *>(x + base);
        float s = 0.f;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const float4 v = p[i];
            xv[16 * g + 4 * i] = v.x;
            xv[16 * g + 4 * i + 1] = v.y;
            xv[16 * g + 4 * i + 2] = v.z;
            xv[16 * g + 4 * i + 3] = v.w;
            s += (v.x + v.y) + (v.z + v.w);
        }
        xs[g] = s;
    }

    auto dot = [&](const Row &q) -> float {
        float tot = 0.f;
        if constexpr (Q4) {
            const uint32_t sh = 8 * (lane & 2);  // 16 * (p & 1), p = lane%8 / 2: groups 2p and 2p + 1
            const bool hi = (lane & 4) != 0;      // p >= 2
#pragma unroll
            for (int k = 0; k < 2; ++k) {
                float A = 0.f, B = 0.f;
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const uint32_t wv = q.qs[k][i], w8 = wv >> 8;
                    const float *xl = xv + 32 * k + 4 * i, *xh = xl + 16;
                    A = __builtin_fmaf(lo_half(wv & 0x000F000Fu), xl[0], A);
                    A = __builtin_fmaf(lo_half(w8 & 0x000F000Fu), xl[1], A);
                    A = __builtin_fmaf(hi_half(wv & 0x000F000Fu), xl[2], A);
                    A = __builtin_fmaf(hi_half(w8 & 0x000F000Fu), xl[3], A);
                    B = __builtin_fmaf(lo_half(wv & 0x00F000F0u), xh[0], B);
                    B = __builtin_fmaf(lo_half(w8 & 0x00F000F0u), xh[1], B);
                    B = __builtin_fmaf(hi_half(wv & 0x00F000F0u), xh[2], B);
                    B = __builtin_fmaf(hi_half(w8 & 0x00F000F0u), xh[3], B);
                }
                // the two groups' 6-bit scales and mins (q4_scales for a lane-varying group pair)
                const uint32_t s0 = q.hdr[k].y >> sh, s1 = q.hdr[k].z >> sh, s2 = q.hdr[k].w >> sh;
                const uint32_t sc = hi ? (s2 & 0x0F0Fu) | ((s0 >> 2) & 0x3030u) : s0 & 0x3F3Fu;
                const uint32_t mn = hi ? ((s2 >> 4) & 0x0F0Fu) | ((s1 >> 2) & 0x3030u) : s1 & 0x3F3Fu;
                // low nibbles carry 2^-24, high nibbles 2^-20
                const float sq = float(byte_of(sc, 0)) * 16777216.0f * A + float(byte_of(sc, 1)) * 1048576.0f * B;
                const float sm = float(byte_of(mn, 0)) * xs[2 * k] + float(byte_of(mn, 1)) * xs[2 * k + 1];
                const float v = lo_half(q.hdr[k].x) * sq - hi_half(q.hdr[k].x) * sm;
                tot += in[k] ? v : 0.f;
            }
        } else {
            float A[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const uint32_t a = q.c[0][i], b = q.c[1][i], hq = q.c[2][i];
#pragma unroll
                for (int odd = 0; odd < 2; ++odd) {
                    const uint32_t aa = odd ? a >> 8 : a, bb = odd ? b >> 8 : b;
                    const uint32_t h4 = odd ? hq >> 4 : hq << 4, h2 = odd ? hq >> 6 : hq << 2;
                    const uint32_t e0 = (aa & 0x000F000Fu) | (h4 & 0x00300030u);
                    const uint32_t e2 = (aa & 0x00F000F0u) | (h4 & 0x03000300u);
                    const uint32_t e1 = (bb & 0x000F000Fu) | (h2 & 0x00300030u);
                    const uint32_t e3 = (bb & 0x00F000F0u) | (h2 & 0x03000300u);
                    const float *xo = xv + 4 * i + odd;
                    A[0] = __builtin_fmaf(hi_half(e0), xo[2], __builtin_fmaf(lo_half(e0), xo[0], A[0]));
                    A[1] = __builtin_fmaf(hi_half(e1), xo[18], __builtin_fmaf(lo_half(e1), xo[16], A[1]));
                    A[2] = __builtin_fmaf(hi_half(e2), xo[34], __builtin_fmaf(lo_half(e2), xo[32], A[2]));
                    A[3] = __builtin_fmaf(hi_half(e3), xo[50], __builtin_fmaf(lo_half(e3), xo[48], A[3]));
                }
            }
            // scale of quarter g: 8h + 2g + t, i.e. byte t of each half of dwords 2h, 2h + 1
            const uint32_t t8 = 8 * (lane & 1);
            const uint32_t sa = ((lane & 2) ? q.c[3].z : q.c[3].x) >> t8, sb = ((lane & 2) ? q.c[3].w : q.c[3].y) >> t8;
            const float sc[4] = {float(int8_t(byte_of(sa, 0))), float(int8_t(byte_of(sa, 2))),
                                 float(int8_t(byte_of(sb, 0))), float(int8_t(byte_of(sb, 2)))};
#pragma unroll
            for (int g = 0; g < 4; ++g)  // quarters 0, 1 carry 2^-24, quarters 2, 3 carry 2^-20
                tot = __builtin_fmaf(sc[g], __builtin_fmaf(A[g], g >= 2 ? 1048576.0f : 16777216.0f, -32.0f * xs[g]), tot);
            tot = in[0] ? lo_half(q.d) * tot : 0.f;
        }
        return tot;
    };
    // Q6_K: shift the pieces down to the block's 2-byte alignment (the tensor is 4-byte aligned, so the
    // parity of the block's index)
    auto fix = [&](uint32_t r, Row &q) {
        if constexpr (!Q4) {
            const uint64_t row = __builtin_elementwise_min(r, rows - 1);
            const uint32_t sh = 16 * uint32_t((row * nb + blk[0]) & 1);
#pragma unroll
            for (int k = 0; k < 4; ++k) {
#pragma unroll
                for (int i = 0; i < 3; ++i) q.c[k][i] = __builtin_amdgcn_alignbit(q.c[k][i + 1], q.c[k][i], sh);
                q.c[k][3] = __builtin_amdgcn_alignbit(q.n[k], q.c[k][3], sh);
            }
        }
    };

    auto step = [&](uint32_t s, Row (&q)[R], auto &next) {
        const uint32_t r = first(s);
        if constexpr (PRE) {
            if (s + 1 < steps) {  // uniform over the grid
                const uint32_t rn = first(s + 1);
#pragma unroll
                for (int i = 0; i < R; ++i) load(rn + uint32_t(i), next[i]);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        float v[R];
#pragma unroll
        for (int i = 0; i < R; ++i) {
            fix(r + uint32_t(i), q[i]);
            v[i] = wave_sum(dot(q[i]));
        }
        if (kw == 1) {
            const float o = lane == 0 ? v[0] : v[R - 1];
            if (lane < R && r + lane < rows) out[r + lane] = o;
            return;
        }
        if (lane == 0)
#pragma unroll
            for (int i = 0; i < R; ++i) part[s & 1][wave][i] = v[i];
        __syncthreads();  // every wave runs every step; the other half of `part` is free by the next one
        if (wkk == 0 && lane < R && r + lane < rows) {
            float sum = 0.f;
            for (uint32_t k = 0; k < kw; ++k) sum += part[s & 1][wave + k][lane];
            out[r + lane] = sum;
        }
    };
    if constexpr (PRE) {
        for (uint32_t s = 0; s < steps; ++s) {
            step(s, cur, nxt);
            if (++s == steps) break;
            step(s, nxt, cur);
        }
    } else {
        for (uint32_t s = 0; s < steps; ++s) {
            if (s > 0)
#pragma unroll
                for (int i = 0; i < R; ++i) load(first(s) + uint32_t(i), cur[i]);
            step(s, cur, cur);
        }
    }
}

}  // namespace

// Where this kernel is the faster one: rows of up to 256 super-blocks (16 waves of 16); the slab kernel where a
// test asks for one of its grids.  While the rows do not fill the device the ramp and the round trip decide, and
// this kernel takes 0.3-1.0 of the slab kernel's time at every length.  Beyond, a row costs a wave the same
// whatever its length, so the lanes have to be in use; the slab kernel's time follows the super-blocks.  MI355X,
// this kernel's time over the slab kernel's:
//   Q4_K  32,768 rows: 2.07 at 1 super-block, 1.20 at 4, 0.81 at 5, 0.40 at 16, 0.68 at 17, 1.17 at 65, 0.93 at
//         80, 0.58 at 128;  8,192 rows: 0.87 at 1 and at 4, 1.09 at 65, 0.93 at 72
//   Q6_K  98,304 rows: 4.87 at 1, 1.23 at 8, 1.00 at 9, 0.71 at 16, 1.12 at 17, 0.84 at 28;  49,152 rows: 1.07 at
//         36, 0.89 at 48, 1.60 at 72;  16,384 rows: 1.30 at 6, 0.86 at 9, 0.93 at 17, 1.04 at 112, 0.82 at 128;
//         8,192 rows: 1.13 at 4, 0.99 at 5, 1.41 at 72
// (rows of 5 to 7 waves run few waves per CU, the one workgroup's)
bool gemv_row_eligible(int type, int layout, uint32_t cols, uint32_t rows, const Tuning &t) {
    const uint32_t nb = cols / kQK, kw = (nb + kSpan - 1) / kSpan;
    if (layout != ROW_MAJOR || t.gemv_row == 0 || nb > 16 * kSpan || t.gemv_pf >= 0 || t.gemv_waves != 0 ||
        t.gemv_whole == 0 || t.gemv_qslab == 0)
        return false;
    if (rows <= 4096) return true;
    if (type == Q4_K) return kw > 4 ? nb > 80 : nb >= 5 || rows <= 8192;
    if (kw > 4) return nb >= 128;
    if (rows <= 21504) return nb >= (rows <= 8192 ? 5 : 9);
    return kw == 1 ? nb >= 9 : nb * 5 >= kw * kSpan * 4;  // a second wave's lanes mostly in use
}

hipError_t launch_gemv_row(int type, const uint8_t *w, const float *x, float *out, uint32_t cols, uint32_t rows,
                           hipStream_t stream) {
    const uint32_t nb = cols / kQK, kw = (nb + kSpan - 1) / kSpan;
    const bool wide = kw > 4;
    const uint32_t waves = wide ? kw : kw == 3 ? 3 : 4, per = wide ? 1 : waves / kw * 2;  // rows per workgroup and step
    const uint32_t wgs = (rows + per - 1) / per, cap = uint32_t(device_cus()) * (wide ? 1 : 2);
    const uint32_t steps = (wgs + cap - 1) / cap;
    const dim3 grid((wgs + steps - 1) / steps), block(64 * waves);
    if (type == Q4_K) {
        if (wide) gemv_row_kernel<Q4_K, 16, 1><<<grid, block, 0, stream>>>(w, x, out, rows, nb, kw, steps);
        else gemv_row_kernel<Q4_K, 4, 2><<<grid, block, 0, stream>>>(w, x, out, rows, nb, kw, steps);
    } else {
        if (wide) gemv_row_kernel<Q6_K, 16, 1><<<grid, block, 0, stream>>>(w, x, out, rows, nb, kw, steps);
        else gemv_row_kernel<Q6_K, 4, 2><<<grid, block, 0, stream>>>(w, x, out, rows, nb, kw, steps);
    }
    return hipGetLastError();
}

}  // namespace ns
