// ns_gemm_skinny.hip -- prefill GEMM for few tokens (one 32- to 128-token tile per workgroup) on
// fp16 MFMA, for gfx950: CDNA4 layout in both accumulation modes, ROW_MAJOR in the FP32 mode.
//
// Replaces, for small batches, the same reference kernels as ns_gemm_reg.hip, ns_gemm_f16.hip and
// ns_gemm.hip (metal/gemma4.metal:263-301, 373-395, 432-490; metal_engine.mm:274, :288-289, :311).
//
// What bounds it: below ~100 tokens the weight bytes (a 256-token tile spent most of its matrix
// work on padding, and the 120 column tiles of the gate/up pair left half the CUs idle), so the
// work is split over the weights and the token tile is only as tall as the batch needs.
//
// Work split.  A workgroup is 8 waves = WC column groups x WK groups of super-blocks.  Each wave
// owns 64 columns (2 MFMA tiles; for the gate/up pair 32 gate rows and the same 32 up rows) and
// walks every WK-th super-block of the workgroup's K range alone; the WK partial sums meet in LDS
// at the end, in a fixed order.  So 64 * WC columns keep all eight waves streaming weights, and the
// gate/up pair needs no reduction between workgroups.  A shape with too few columns to fill the
// device splits K over kparts workgroups as well; the last of them to arrive adds the parts in
// part order (no workgroup ever waits for another).
//
// A wave decodes its own B fragments from raw blocks in registers: lane l holds weight row l%32
// and, of each pair of 16-byte qs (ql, qh) chunks, the chunk l/32, so one 16-byte load per chunk
// pair feeds four fragments.  The MFMA sums over k in any order as long as A and B agree on it:
// fragment (group g, e) covers k = 32g + 16(l/32) + 8e + 0..7 for both block types.  x goes
// through LDS by DMA in stages of KS columns per wk group, two buffers; rows are stored with their
// 16-byte chunks XOR-swizzled so the fragment reads are conflict-free.
//
// Arithmetic.  FP16 mode: the tiles of ns_tile16.hpp, accumulated across super-blocks; the row
// scale comes from every wave reading the block factors of its share of the row first.  FP32
// mode: fragments are exact integers times a power of two (Q4_K sc*q*2^-14; Q6_K sc*(v-32)*2^-16,
// one rounding past 11 bits as in ns_gemm.hip), summed per super-block in S, and y += d*S in fp32.
// The Q4_K min term -dmin * sum_g m_g * (sum of x over group g) needs no pass over x ahead of the
// GEMM: each lane has the 16 values per group that its own A fragments hold added up in fp32 (by
// 4x4x4 MFMAs), splits the eight sums exactly into three bf16 pieces, and three bf16 MFMAs multiply
// them by the m_g (exact in bf16) and add the two lane halves.
#include <algorithm>
#include <type_traits>

#include "ns_internal.hpp"
#include "ns_quant.hpp"
#include "ns_tile16.hpp"

namespace ns {
namespace {

typedef _Float16 half4_t __attribute__((ext_vector_type(4)));
typedef _Float16 half8_t __attribute__((ext_vector_type(8)));
typedef __bf16 bf8_t __attribute__((ext_vector_type(8)));
typedef float float4_t __attribute__((ext_vector_type(4)));
typedef float float16_t __attribute__((ext_vector_type(16)));
typedef __amdgpu_buffer_rsrc_t rsrc_t;

constexpr int kWaves = 8;
constexpr int kThreads = 64 * kWaves;
constexpr int NJ = 2;  // 32-column MFMA tiles per wave
constexpr int kMaxSeg = 3;

// Up to three matrices that share x (Q, K and V): one run of column tiles each.
struct Args {
    const uint8_t *w[kMaxSeg], *up;
    void *out[kMaxSeg];
    uint32_t rows[kMaxSeg], ct_end[kMaxSeg];
    uint32_t q6_seg;  // the mixed kernel: the segment whose matrix is Q6_K
    void *copy;       // a second output of the last segment (tied V), or nullptr
    const uint16_t *x;
    float *partial;
    uint32_t *counters;
    uint32_t cols, batch, ntok, ncol, kparts;
};

__device__ __forceinline__ rsrc_t make_rsrc(const void *p, uint32_t bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(p), 0, int(bytes), 0x00020000);
}
__device__ __forceinline__ u32x4 bload16(rsrc_t r, uint32_t off, uint32_t soff) {
    return __builtin_amdgcn_raw_buffer_load_b128(r, int(off), int(soff), 0);
}
__device__ __forceinline__ uint32_t bload4(rsrc_t r, uint32_t off, uint32_t soff) {
    return __builtin_amdgcn_raw_buffer_load_b32(r, int(off), int(soff), 0);
}
__device__ __forceinline__ uint32_t bload2(rsrc_t r, uint32_t off, uint32_t soff) {
    return __builtin_amdgcn_raw_buffer_load_b16(r, int(off), int(soff), 0);
}

// One LDS DMA instruction: 16 bytes per lane into the 1 KiB at lds.
__device__ __forceinline__ void dma16(rsrc_t r, u32x4 *lds, uint32_t voff, uint32_t soff) {
    __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (__attribute__((address_space(3))) void *)lds, 16, voff, soff, 0, 0);
}

template <int N>
__device__ __forceinline__ void vm_wait() {
    static_assert(N >= 0 && N < 64, "vmcnt is 6 bits");
    __builtin_amdgcn_s_waitcnt((N & 15) | ((N >> 4) << 14) | (7 << 4) | (15 << 8));
}
// The bare barrier (no wait for loads in flight); signal fences keep memory accesses on their side.
__device__ __forceinline__ void bare_barrier() {
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
    __builtin_amdgcn_s_barrier();
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
}
__device__ __forceinline__ void lds_barrier() {
    __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0)
    bare_barrier();
}

__device__ __forceinline__ float round_f16p(float v) {
    uint32_t b = __builtin_bit_cast(uint32_t, v);
    b = (b + 0x0fffu + ((b >> 13) & 1u)) & 0xffffe000u;
    return __builtin_bit_cast(float, b);
}
__device__ __forceinline__ uint32_t bits(half2_t v) { return __builtin_bit_cast(uint32_t, v); }
__device__ __forceinline__ half2_t h2(uint32_t v) { return __builtin_bit_cast(half2_t, v); }

// One lane's raw bytes of one super-block of one column: the chunks of its lane half.
struct RawQ4 {
    u32x4 hdr, qs[4];  // qs[p]: chunk 1 + 2p + l/32 (groups 2p low nibbles, 2p+1 high)
};
struct RawQ6 {
    u32x4 ql[4];  // [2h + q]: chunk 4h + 2q + l/32 (quarters q low nibbles, q + 2 high)
    u32x4 qh[2];  // [h]: chunk 8 + 2h + l/32
    u32x4 sc;
    uint32_t d;
    uint32_t x[7];  // ROW_MAJOR: the dword after each 16-byte piece (blocks are 2-byte aligned)
};

// A workgroup's work item and the LDS its kernel holds for it.
struct Item {
    uint32_t tt, kp, tile, seg, ct;
};
__device__ __forceinline__ Item work_item(const Args &a) {
    // XCD-aware order: workgroup L runs on XCD L % 8, which takes a contiguous run of the work items
    // q = (ct * kparts + kp) * ntok + tt, so the token tiles that share weights share an L2.
    const uint32_t nwg = gridDim.x, w8 = nwg / 8, L = blockIdx.x;
    const uint32_t q = L < 8 * w8 ? (L % 8) * w8 + L / 8 : L;
    Item it;
    it.tt = q % a.ntok;
    const uint32_t g = q / a.ntok, ctg = g / a.kparts;
    it.kp = g % a.kparts;
    it.tile = ctg * a.ntok + it.tt;
    it.seg = ctg < a.ct_end[0] ? 0u : ctg < a.ct_end[1] ? 1u : 2u;
    it.ct = ctg - (it.seg == 0 ? 0u : a.ct_end[it.seg - 1]);
    return it;
}
struct Shared {
    float rmax[kWaves][NJ][32];
    uint32_t last_flag;
};
// u32x4 of one x buffer: a stage for every wk group, and what the final sum of a token tile needs
template <int MI, int WK>
constexpr int buf_len() {
    constexpr int x = WK * 32 * MI * (MI * WK <= 8 ? 128 : 64) / 8, red = kWaves * NJ * 16 * 64 / 4;
    return x > red ? x : red;
}

// WC column groups x WK super-block groups of waves; MI 32-token tiles.
template <int TYPE, int LAYOUT, int ACC, bool PAIR, int MI, int WK, bool EX>
__device__ __forceinline__ void skinny_body(const Args &a, const Item &item, u32x4 *X0, u32x4 *X1, Shared &sh) {
    constexpr bool Q4 = TYPE == Q4_K, F16 = ACC == ACC_FP16, ROW = LAYOUT == ROW_MAJOR;
    constexpr int WC = kWaves / WK, TT = 32 * MI;
    constexpr int KS = MI * WK <= 8 ? 128 : 64;      // columns of x per stage
    constexpr int NS = 256 / KS, CR = KS / 8;         // stages per super-block, 16-byte chunks per x row
    constexpr int RPI = 64 / CR;                      // x rows one DMA instruction fills
    constexpr int ND = TT / RPI / WC;                 // DMA instructions per wave and stage
    constexpr int kXBuf = WK * TT * CR;               // u32x4 per buffer
    static_assert(TT % (RPI * WC) == 0 && 2 * kXBuf * 16 <= 131072, "x stages");
    using Raw = typename std::conditional<Q4, RawQ4, RawQ6>::type;
    static_assert(kXBuf <= buf_len<MI, WK>(), "x buffer");
    // EX: sc*(v-32) in two exact fragments (see factors)
    static_assert(!EX || (TYPE == Q6_K && ACC == ACC_FP32), "EX");

    const uint32_t tid = threadIdx.x, lane = tid & 63, hl = lane >> 5, ln = lane & 31;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t wc = wave % WC, wk = wave / WC;
    const uint32_t tt = item.tt, kp = item.kp, tile = item.tile, seg = item.seg, ct = item.ct;
    const uint32_t rows = a.rows[seg], cols = a.cols, batch = a.batch, t0 = tt * TT;
    const uint32_t nb = cols / kQK, kparts = a.kparts;
    const uint32_t sb0 = kp * nb / kparts, sb1 = (kp + 1) * nb / kparts;
    const uint32_t iters = (sb1 - sb0 + WK - 1) / WK;

    constexpr uint32_t kRowsPerTile = PAIR ? WC * 32 : WC * 64;
    auto brow = [&](int j) -> uint32_t {
        if constexpr (PAIR) return ct * kRowsPerTile + wc * 32 + ln;  // j 0 = gate, 1 = up
        else return ct * kRowsPerTile + wc * 64 + uint32_t(j) * 32 + ln;
    };
    const uint32_t wbytes = rows * nb * block_bytes(TYPE);
    const uint8_t *const w0 = a.w[seg], *const w1 = PAIR ? a.up : a.w[seg];
    const uint32_t xbytes = batch * cols * 2;

    // ---- weight addressing: the lane's part is a VGPR, the super-block's a uniform offset.  Rows past
    // `rows` lie past the descriptor's range and read zeros.
    constexpr uint32_t kRegion = kRowTile * block_bytes(TYPE);
    uint32_t voff[NJ];  // first byte of block (row, 0); CDNA4: of its chunk 0
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
        const uint32_t r = brow(j);
        voff[j] = ROW ? r * nb * block_bytes(TYPE) : uint32_t(region_offset(TYPE, r / kRowTile, 0, nb)) + (r % kRowTile) * 16;
    }
    // byte offset, past voff + the super-block's uniform part, of chunk c
    auto chunk = [](uint32_t c) { return c * (ROW ? 16u : 1024u); };
    constexpr uint32_t kBlkStep = ROW ? block_bytes(TYPE) : kRegion;
    // live = 0 (past the last block): the range is the tensor's first block step, from uniform offset 0, so all
    // but the first rows' loads read zeros and touch no memory.  No instruction's uniform offset passes the
    // range: the check compares with their difference.
    auto load_raw = [&](uint32_t sb, bool live, Raw (&raw)[NJ]) {
        const uint32_t so = live ? sb * kBlkStep : 0;
        const rsrc_t wsrc0 = make_rsrc(w0, live ? wbytes : kBlkStep),
                     wsrc1 = make_rsrc(w1, live ? wbytes : kBlkStep);
        auto wsrc = [&](int j) { return (PAIR && j == 1) ? wsrc1 : wsrc0; };
#pragma unroll
        for (int j = 0; j < NJ; ++j) {
            if constexpr (Q4) {
                raw[j].hdr = bload16(wsrc(j), voff[j], so);
#pragma unroll
                for (int p = 0; p < 4; ++p) raw[j].qs[p] = bload16(wsrc(j), voff[j] + chunk(hl), so + chunk(1 + 2 * p));
            } else if constexpr (!ROW) {
#pragma unroll
                for (int c = 0; c < 4; ++c) raw[j].ql[c] = bload16(wsrc(j), voff[j] + chunk(hl), so + chunk(2 * c));
#pragma unroll
                for (int h = 0; h < 2; ++h) raw[j].qh[h] = bload16(wsrc(j), voff[j] + chunk(hl), so + chunk(8 + 2 * h));
                raw[j].sc = bload16(wsrc(j), voff[j], so + chunk(12));
                // d of row r: region + 13 KiB + 2*(r%64) = voff - 14*(r%64) + 13 KiB
                raw[j].d = bload2(wsrc(j), voff[j] - 14 * (brow(j) % kRowTile), so + kQ6Chunks * 1024);
            } else {
                // 210-byte blocks: the dword-aligned address at or below each piece, five dwords
                const uint32_t blk = voff[j] + so, al = blk & ~3u;
                const uint32_t lo = al + 16 * hl;
#pragma unroll
                for (int c = 0; c < 4; ++c) {
                    raw[j].ql[c] = bload16(wsrc(j), lo + 32 * c, 0);
                    raw[j].x[c] = bload4(wsrc(j), lo + 32 * c + 16, 0);
                }
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    raw[j].qh[h] = bload16(wsrc(j), lo + 128 + 32 * h, 0);
                    raw[j].x[4 + h] = bload4(wsrc(j), lo + 128 + 32 * h + 16, 0);
                }
                raw[j].sc = bload16(wsrc(j), al + 192, 0);
                raw[j].x[6] = bload4(wsrc(j), al + 208, 0);
                raw[j].d = bload2(wsrc(j), blk + 208, 0);
            }
        }
    };
    // vector loads of load_raw: the x DMA issued before them has landed once only these are in flight
    constexpr int kRawLoads = NJ * (Q4 ? 5 : ROW ? 15 : 8);
    // ROW_MAJOR Q6_K: shift the five dwords of each piece down to the block's 2-byte alignment
    auto fix_raw = [&](uint32_t sb, Raw (&raw)[NJ]) {
        if constexpr (!Q4 && ROW) {
#pragma unroll
            for (int j = 0; j < NJ; ++j) {
                const uint32_t by = ((voff[j] + sb * kBlkStep) & 2u) * 8u;
                auto shift = [&](u32x4 &v, uint32_t hi) {
#pragma unroll
                    for (int i = 0; i < 3; ++i) v[i] = __builtin_amdgcn_alignbit(v[i + 1], v[i], by);
                    v[3] = __builtin_amdgcn_alignbit(hi, v[3], by);
                };
#pragma unroll
                for (int c = 0; c < 4; ++c) shift(raw[j].ql[c], raw[j].x[c]);
#pragma unroll
                for (int h = 0; h < 2; ++h) shift(raw[j].qh[h], raw[j].x[4 + h]);
                shift(raw[j].sc, raw[j].x[6]);
            }
        }
    };

    // ---- x staging: instruction i of wave wc fills rows (wc*ND + i)*RPI .. of group wk's tile; lane l
    // writes position l%CR of row +l/CR and fetches the chunk that the swizzle puts there.
    auto swz = [](uint32_t R) { return CR == 16 ? (R & 15) : ((R >> 1) & 7); };
    // The swizzle repeats every 16 rows: where registers are short (Q4_K FP32 mode; spills else), the offsets
    // of the first 16 / RPI instructions serve the others, at an add each.
    constexpr int NX = Q4 && !F16 && 16 / RPI < ND ? 16 / RPI : ND;
    uint32_t xoff[NX];
#pragma unroll
    for (int i = 0; i < NX; ++i) {
        const uint32_t R = (wc * ND + uint32_t(i)) * RPI + lane / CR, c = (lane % CR) ^ swz(R);
        xoff[i] = ((t0 + R) * cols + 8 * c) * 2;
    }
    auto xbuf = [&](int b) -> u32x4 * { return b ? X1 : X0; };
    auto dma_x = [&](uint32_t sb, bool live, int st) {
        const uint32_t so = live ? (sb * kQK + uint32_t(st) * KS) * 2 : 0;
        const rsrc_t xsrc = make_rsrc(a.x, live ? xbytes : 0);
        uint32_t xo[NX];
#pragma unroll
        for (int i = 0; i < NX; ++i) {
            xo[i] = xoff[i];
            if constexpr (NX < ND) asm volatile("" : "+v"(xo[i]));  // the sums below are formed here, not kept in registers
        }
#pragma unroll
        for (int i = 0; i < ND; ++i)
            dma16(xsrc, xbuf(st & 1) + wk * (TT * CR) + (wc * ND + uint32_t(i)) * 64, xo[i % NX] + uint32_t(i / NX) * 32 * cols, so);
    };
    // A fragment of token tile i: row 32i + ln, chunk 4*gq + 2*hl + e of the stage
    const uint32_t a0 = wk * (TT * CR) + ln * CR, asw = (2 * hl) ^ swz(ln);
    auto load_a = [&](int b, int i, int gq, int e) -> half8_t {
        return __builtin_bit_cast(half8_t, xbuf(b)[a0 + uint32_t(i) * 32 * CR + ((4 * gq + e) ^ asw)]);
    };

    // ---- prologue: the first super-block in flight, then (FP16 mode) the row scales
    auto sb_of = [&](uint32_t it) { return sb0 + it * WK + wk; };
    Raw raw[NJ];
    float c24[NJ], inv_c[NJ];
    auto first_loads = [&]() {  // in this order: the main loop's first wait counts the raw loads
        dma_x(sb_of(0), sb_of(0) < sb1, 0);
        __atomic_signal_fence(__ATOMIC_SEQ_CST);
        __builtin_amdgcn_sched_barrier(0);
        load_raw(sb_of(0), sb_of(0) < sb1, raw);
        __atomic_signal_fence(__ATOMIC_SEQ_CST);
        __builtin_amdgcn_sched_barrier(0);
    };
    if constexpr (F16) {
        // this wave's share of the rows' block factors: super-blocks 2*(wk + WK*u) + hl
        const rsrc_t wsrc0 = make_rsrc(w0, wbytes), wsrc1 = make_rsrc(w1, wbytes);
        auto wsrc = [&](int j) { return (PAIR && j == 1) ? wsrc1 : wsrc0; };
        float M[NJ] = {};
        for (uint32_t u0 = 0; 2 * WK * u0 < nb; u0 += 2) {
            uint32_t dd[2][NJ];
#pragma unroll
            for (int u = 0; u < 2; ++u) {
                const uint32_t b = __builtin_elementwise_min(2 * (wk + WK * (u0 + uint32_t(u))) + hl, nb - 1);
#pragma unroll
                for (int j = 0; j < NJ; ++j) {
                    if constexpr (Q4) dd[u][j] = bload4(wsrc(j), voff[j] + b * kBlkStep, 0);
                    else dd[u][j] = bload2(wsrc(j), voff[j] - 14 * (brow(j) % kRowTile) + b * kBlkStep + kQ6Chunks * 1024, 0);
                }
            }
#pragma unroll
            for (int u = 0; u < 2; ++u)
#pragma unroll
                for (int j = 0; j < NJ; ++j) {
                    const float m = __builtin_fabsf(lo_half(dd[u][j]));
                    M[j] = __builtin_fmaxf(M[j], Q4 ? __builtin_fmaxf(m, __builtin_fabsf(hi_half(dd[u][j]))) : m);
                }
            if (u0 == 0) first_loads();  // behind the first factors
        }
#pragma unroll
        for (int j = 0; j < NJ; ++j) {
            M[j] = __builtin_fmaxf(M[j], __shfl_xor(M[j], 32));
            if (hl == 0) sh.rmax[wave][j][ln] = M[j];
        }
        lds_barrier();
#pragma unroll
        for (int j = 0; j < NJ; ++j) {
            float m = 0.f;
#pragma unroll
            for (int k = 0; k < WK; ++k) m = __builtin_fmaxf(m, sh.rmax[uint32_t(k) * WC + wc][j][ln]);
            row_scale(m, c24[j], inv_c[j], !Q4);
        }
    } else {
        first_loads();
    }

    float16_t acc[MI][NJ];
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int j = 0; j < NJ; ++j)
#pragma unroll
            for (int v = 0; v < 16; ++v) acc[i][j][v] = 0.f;

    // ---- per super-block factors of column j, and its fragments (group grp, e)
    struct Factors {
        half2_t A2[NJ][EX ? 8 : 1], B2[NJ][EX ? 8 : 1];  // EX: the odd unit of the scale
        half2_t A[NJ][8], B[NJ][8];  // per group; Q4_K FP32 mode: A alone; Q4_K FP16 mode: per group pair
    };
    auto factors = [&](const Raw (&r)[NJ], Factors &F) {
#pragma unroll
        for (int j = 0; j < NJ; ++j) {
            if constexpr (Q4) {
                const Q4Scales sc = q4_scales(r[j].hdr.y, r[j].hdr.z, r[j].hdr.w);
                if constexpr (F16) {
                    const half2_t dc = q4_dc(r[j].hdr.x, c24[j]), mc = q4_mc22(r[j].hdr.x, c24[j]);
                    const uint32_t m03 = sc.m03 << 2, m47 = sc.m47 << 2;
#pragma unroll
                    for (int p = 0; p < 4; ++p) {  // group pair 2p, 2p + 1 (its A times 2^-4)
                        const Q4Factors g = q4_factors(p < 2 ? sc.sc03 : sc.sc47, p < 2 ? m03 : m47, p & 1, dc, mc);
                        F.A[j][p] = g.A;
                        F.B[j][p] = g.B;
                    }
                } else {
                    // q*2^-24 (low nibbles) or 16q*2^-24 (high) times this = sc*q*2^-14, exact
#pragma unroll
                    for (int gg = 0; gg < 8; ++gg)
                        F.A[j][gg] = splat(_Float16(float(q4_sc(sc, gg)) * (gg & 1 ? 64.0f : 1024.0f)));
                }
            } else {
                const float d = lo_half(r[j].d);
#pragma unroll
                for (int gg = 0; gg < 8; ++gg) {
                    // group gg = 4h + Q of this lane half: scale 8h + 2Q + hl
                    const int sc = int8_t(byte_of(r[j].sc[gg >> 1] >> (8 * hl), 2 * (gg & 1)));
                    if constexpr (F16) {
                        const float dc = d * c24[j], dm = -32.0f * d * (c24[j] * 5.9604644775390625e-08f);
                        F.A[j][gg] = splat(_Float16(dc * float(sc)));
                        F.B[j][gg] = splat(_Float16(dm * float(sc)));
                    } else {
                        // v*2^-24 * sc*2^8 - sc*2^-11 = sc*(v-32)*2^-16, rounded once where |sc| > 64 makes
                        // it 12 bits; EX takes sc without its lowest bit (11 bits) and that bit apart
                        const int s1 = EX ? sc & ~1 : sc;
                        F.A[j][gg] = splat(_Float16(float(s1) * 256.0f));
                        F.B[j][gg] = splat(_Float16(float(s1) * -0.00048828125f));
                        if constexpr (EX) {
                            F.A2[j][gg] = splat(_Float16(float(sc & 1) * 256.0f));
                            F.B2[j][gg] = splat(_Float16(float(sc & 1) * -0.00048828125f));
                        }
                    }
                }
            }
        }
    };
    auto frag = [&](const Raw &r, const auto &A, const auto &B, int grp, int e) -> half8_t {
        u32x4 f;
#pragma unroll
        for (int d = 0; d < 2; ++d) {
            if constexpr (Q4) {
                const uint32_t w = r.qs[grp >> 1][2 * e + d];
                if constexpr (F16) {
                    uint32_t lo[2], hi[2];  // (the two groups of a pair share the unpack: common subexpressions)
                    q4_f16x8(w, Q4Factors{A[grp >> 1], B[grp >> 1]}, lo, hi);
                    f[2 * d] = grp & 1 ? hi[0] : lo[0];
                    f[2 * d + 1] = grp & 1 ? hi[1] : lo[1];
                } else {
                    const uint32_t p = __builtin_amdgcn_perm(w, w, 0x03010200u);  // bytes [b0, b2, b1, b3]
                    const uint32_t m = grp & 1 ? 0x00F000F0u : 0x000F000Fu;
                    f[2 * d] = bits(h2(p & m) * A[grp]);
                    f[2 * d + 1] = bits(h2((p >> 8) & m) * A[grp]);
                }
            } else {
                const int h = grp >> 2, Q = grp & 3;
                const uint32_t ql = r.ql[2 * h + (Q & 1)][2 * e + d], qh = r.qh[h][2 * e + d];
                const uint32_t lo4 = (Q >= 2 ? ql >> 4 : ql) & 0x0F0F0F0Fu;
                const uint32_t hb = Q == 0 ? qh << 4 : Q == 1 ? qh << 2 : Q == 2 ? qh : qh >> 2;
                uint32_t o[2];
                q6_f16x4(lo4 | (hb & 0x30303030u), A[grp], B[grp], o);
                f[2 * d] = o[0];
                f[2 * d + 1] = o[1];
            }
        }
        return __builtin_bit_cast(half8_t, f);
    };
    auto mfma = [](half8_t x, half8_t w, const float16_t &c) { return __builtin_amdgcn_mfma_f32_32x32x16_f16(x, w, c, 0, 0, 0); };

    // ---- main loop.  Stage s = (iteration, st): x(s) has been requested one stage earlier and, at
    // st 0, the super-block's raw blocks once those of the iteration before were consumed.  Wait for
    // this wave's share of x(s) (leaving the raw loads issued after it in flight), meet the other
    // waves of the column groups at the barrier (which also puts every read of buffer (s+1) % 2, at
    // stage s-1, before the DMA that refills it), request x(s+1), then compute.  (A second set of raw
    // registers, filled one super-block earlier, changed nothing: 20.3 us either way for the FP16 pair
    // at 5 tokens, and the FP32 pair took 23.0 instead of 21.5.)
    constexpr bool kMin = Q4 && !F16;
    // The 32-token tile (which also takes batch 2-4) has the registers for short chains of sums: one per half of
    // the super-block, per quarter for row-major Q4_K, added up in T (each once the next is under way, the last
    // after the loads), and one for EX's small second fragments.  Together with the pairwise sum over the waves and
    // the min term's small pieces first, error against 64 bits at 3 tokens of 3840 x 4096, in brackets that of the
    // small-batch kernel: row-major Q4_K 1.09e-7 (1.12e-7; in halves 1.18e-7, in one chain 1.55e-7), Q6_K
    // 1.01e-7 (1.04e-7; in one chain 1.42e-7), CDNA4 Q4_K 1.18e-7 (1.40e-7).  Quarters everywhere took 0.5-2% more time.
    constexpr bool kShort = !F16 && MI == 1;
    constexpr int kChain = !kShort ? 8 : Q4 && ROW ? 2 : 4;  // in groups of 32
    auto group_sum = [](int s, half4_t sel, half4_t xv, float4_t c) {  // s is a constant once unrolled
        return s == 0   ? __builtin_amdgcn_mfma_f32_4x4x4f16(sel, xv, c, 4, 0, 0)
               : s == 1 ? __builtin_amdgcn_mfma_f32_4x4x4f16(sel, xv, c, 4, 1, 0)
               : s == 2 ? __builtin_amdgcn_mfma_f32_4x4x4f16(sel, xv, c, 4, 2, 0)
                        : __builtin_amdgcn_mfma_f32_4x4x4f16(sel, xv, c, 4, 3, 0);
    };
    // The group sums of x by 4x4x4 MFMAs (16 independent 4x4 blocks): a lane's four x values are one column
    // and its column of D stays with the lane, so D's row s takes group 4h + s where A is ones in row s alone.
    // A's block s (lanes 4s..) holds that selector, broadcast to all blocks.  (As mixed-precision FMAs they
    // were 256 of the 680 VALU instructions per super-block at 64 tokens, and as many wait states: row-major
    // projections at 384 tokens 27.6 us then, 26.7 now, Q4_K downs at 64-512 tokens 21.0-91.7 us, 20.0-87.0.)
    const _Float16 one = lane >> 2 == (lane & 3) ? _Float16(1.0f) : _Float16(0.0f);
    const half4_t ones{one, one, one, one};
    for (uint32_t it = 0; it < iters; ++it) {
        const uint32_t sb = sb_of(it), sbn = sb_of(it + 1);
        const bool valid = sb < sb1, more = sbn < sb1;  // wave-uniform
        Factors F;
        float16_t S[F16 ? 1 : MI][NJ], S2[EX ? NJ : 1], T[kShort ? NJ : 1];
        float4_t P[kMin ? MI : 1][2];  // group sums of this lane half's x: groups 4h + slot
#pragma unroll
        for (int st = 0; st < NS; ++st) {
            __builtin_amdgcn_sched_barrier(0);
            if (st == 0) vm_wait<kRawLoads>();
            else vm_wait<0>();
            if constexpr (WC > 1) bare_barrier();
            else __atomic_signal_fence(__ATOMIC_SEQ_CST);
            if (st + 1 < NS) dma_x(sb, valid, st + 1);
            else dma_x(sbn, more, 0);
            if (st == 0) {
                // the factors are formed here, behind the DMA: without the pin the compiler hoists
                // them, and their wait for the raw blocks, above the barrier
#pragma unroll
                for (int j = 0; j < NJ; ++j) {
                    if constexpr (Q4) asm volatile("" : "+v"(raw[j].hdr));
                    else asm volatile("" : "+v"(raw[j].sc), "+v"(raw[j].d));
                }
                fix_raw(sb, raw);
                factors(raw, F);
            }
            __builtin_amdgcn_sched_barrier(0);
            if (valid) {
#pragma unroll
                for (int gq = 0; gq < KS / 32; ++gq) {
                    const int grp = st * (KS / 32) + gq;
#pragma unroll
                    for (int e = 0; e < 2; ++e) {
                        half8_t av[MI], fb[NJ], fb2[EX ? NJ : 1];
#pragma unroll
                        for (int i = 0; i < MI; ++i) av[i] = load_a(st & 1, i, gq, e);
#pragma unroll
                        for (int j = 0; j < NJ; ++j) {
                            fb[j] = frag(raw[j], F.A[j], F.B[j], grp, e);
                            if constexpr (EX) fb2[j] = frag(raw[j], F.A2[j], F.B2[j], grp, e);
                        }
#pragma unroll
                        for (int i = 0; i < MI; ++i) {
                            if constexpr (kMin) {
                                float4_t p = grp % 4 == 0 && e == 0 ? float4_t{} : P[i][grp / 4];
                                p = group_sum(grp % 4, ones, __builtin_shufflevector(av[i], av[i], 0, 1, 2, 3), p);
                                P[i][grp / 4] = group_sum(grp % 4, ones, __builtin_shufflevector(av[i], av[i], 4, 5, 6, 7), p);
                            }
#pragma unroll
                            for (int j = 0; j < NJ; ++j) {
                                if constexpr (F16) acc[i][j] = mfma(av[i], fb[j], acc[i][j]);
                                else S[i][j] = mfma(av[i], fb[j], grp % kChain == 0 && e == 0 ? float16_t{} : S[i][j]);
                                if constexpr (EX) S2[j] = mfma(av[i], fb2[j], grp == 0 && e == 0 ? float16_t{} : S2[j]);
                                if constexpr (kShort) {
                                    if (grp % kChain == kChain - 1 && grp < 7 && e == 1) T[j] = grp < kChain ? S[i][j] : T[j] + S[i][j];
                                }
                            }
                        }
                    }
                }
            }
        }
        float d[NJ], dmin[NJ];
        bf8_t mb[NJ];
        if constexpr (!F16) {
#pragma unroll
            for (int j = 0; j < NJ; ++j) {
                if constexpr (Q4) {
                    d[j] = lo_half(raw[j].hdr.x) * 16384.0f;
                    dmin[j] = hi_half(raw[j].hdr.x);
                    const Q4Scales sc = q4_scales(raw[j].hdr.y, raw[j].hdr.z, raw[j].hdr.w);
                    u32x4 m;
#pragma unroll
                    for (int k = 0; k < 4; ++k)  // bf16 of an integer below 64: the upper half of its fp32
                        m[k] = __builtin_amdgcn_perm(__builtin_bit_cast(uint32_t, float(q4_m(sc, 2 * k + 1))),
                                                     __builtin_bit_cast(uint32_t, float(q4_m(sc, 2 * k))), 0x07060302u);
                    // formed before the next blocks are requested: a header still in use would be loaded
                    // elsewhere and copied, which waits for the load just issued
                    asm volatile("" : "+v"(d[j]), "+v"(dmin[j]), "+v"(m));
                    mb[j] = __builtin_bit_cast(bf8_t, m);
                } else {
                    d[j] = lo_half(raw[j].d) * 65536.0f;
                    asm volatile("" : "+v"(d[j]));
                }
            }
        }
        // the raw blocks are consumed: request the next super-block's
        __builtin_amdgcn_sched_barrier(0);
        load_raw(sbn, more, raw);
        __atomic_signal_fence(__ATOMIC_SEQ_CST);
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (!F16) {
            if (valid) {
#pragma unroll
                for (int i = 0; i < MI; ++i) {
#pragma unroll
                    for (int j = 0; j < NJ; ++j)
#pragma unroll
                        for (int v = 0; v < 16; ++v) {
                            float sum = S[i][j][v];
                            if constexpr (kShort) sum = T[j][v] + sum;
                            if constexpr (EX) sum += S2[j][v];
                            acc[i][j][v] = __builtin_fmaf(d[j], sum, acc[i][j][v]);
                        }
                    if constexpr (kMin) {
                        // P = hi + mid + lo, each exact in bf16 (8 of the 24 bits at a time)
                        u32x4 pc[3];
#pragma unroll
                        for (int k = 0; k < 4; ++k) {
                            uint32_t pb[3][2];
#pragma unroll
                            for (int u = 0; u < 2; ++u) {
                                float r = P[i][k / 2][2 * (k & 1) + u];
#pragma unroll
                                for (int z = 0; z < 3; ++z) {
                                    pb[z][u] = __builtin_bit_cast(uint32_t, r) & 0xffff0000u;
                                    r -= __builtin_bit_cast(float, pb[z][u]);
                                }
                            }
#pragma unroll
                            for (int z = 0; z < 3; ++z) pc[z][k] = __builtin_amdgcn_perm(pb[z][1], pb[z][0], 0x07060302u);
                        }
#pragma unroll
                        for (int j = 0; j < NJ; ++j) {
                            float16_t mn{};
#pragma unroll
                            for (int z = 0; z < 3; ++z)  // MI 1: the smallest piece first (MI 2 has no register to spare)
                                mn = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf8_t, pc[kShort ? 2 - z : z]), mb[j],
                                                                             mn, 0, 0, 0);
#pragma unroll
                            for (int v = 0; v < 16; ++v) acc[i][j][v] = __builtin_fmaf(-dmin[j], mn[v], acc[i][j][v]);
                        }
                    }
                }
            }
        }
    }
    // Nothing may land in the buffers the sums now go through, and every wave is past its reads.
    vm_wait<0>();
    bare_barrier();

    // ---- the WK partial sums of each column group: wave wk finishes elements v = wk*VP .. +VP-1 of
    // every tile (32x32 D layout: lane holds column ln and token 8*(v/4) + 4*hl + v%4)
    constexpr int VP = 16 / WK;
    float fin[MI][VP][NJ];
#pragma unroll
    for (int i = 0; i < MI; ++i) {
        float *red = reinterpret_cast<float *>(xbuf(i & 1));  // [wave][v][j][64]
#pragma unroll
        for (int v = 0; v < 16; ++v)
#pragma unroll
            for (int j = 0; j < NJ; ++j) red[((wave * 16 + v) * NJ + j) * 64 + lane] = acc[i][j][v];
        lds_barrier();
#pragma unroll
        for (int u = 0; u < VP; ++u)
#pragma unroll
            for (int j = 0; j < NJ; ++j) {
                float s[WK];
#pragma unroll
                for (int k = 0; k < WK; ++k) s[k] = red[(((uint32_t(k) * WC + wc) * 16 + wk * VP + u) * NJ + j) * 64 + lane];
                if constexpr (kShort) {  // pairwise
#pragma unroll
                    for (int m = 1; m < WK; m *= 2)
#pragma unroll
                        for (int k = 0; k < WK; k += 2 * m) s[k] += s[k + m];
                } else {
#pragma unroll
                    for (int k = 1; k < WK; ++k) s[0] += s[k];
                }
                fin[i][u][j] = F16 ? s[0] * inv_c[j] : s[0];
            }
    }

    void *const copy = a.ct_end[seg] == a.ncol ? a.copy : nullptr;
    auto write_out = [&]() {
#pragma unroll
        for (int i = 0; i < MI; ++i)
#pragma unroll
            for (int u = 0; u < VP; ++u) {
                const uint32_t v = wk * VP + uint32_t(u), t = t0 + uint32_t(i) * 32 + 8 * (v >> 2) + 4 * hl + (v & 3);
                if (t >= batch) continue;
                if constexpr (PAIR) {
                    const uint32_t r = brow(0);
                    const float gv = F16 ? round_f16p(fin[i][u][0]) : fin[i][u][0];
                    const float uv = F16 ? round_f16p(fin[i][u][1]) : fin[i][u][1];
                    if (r < rows) static_cast<_Float16 *>(a.out[0])[size_t(t) * rows + r] = _Float16(gelu_tanh(gv) * uv);
                } else {
#pragma unroll
                    for (int j = 0; j < NJ; ++j) {
                        const uint32_t r = brow(j);
                        if (r >= rows) continue;
                        const float y = F16 ? round_f16p(fin[i][u][j]) : fin[i][u][j];
                        static_cast<float *>(a.out[seg])[size_t(t) * rows + r] = y;
                        if (copy) static_cast<float *>(copy)[size_t(t) * rows + r] = y;
                    }
                }
            }
    };
    if (kparts == 1) {
        write_out();
        return;
    }

    // ---- split K over workgroups: parts [tile][kp][i][u][j][thread], added by the last to arrive.
    // Device-coherent atomic stores and loads; the wait completes them before the arrival counts.
    constexpr uint32_t kPart = MI * VP * NJ * kThreads;
    float *mine = a.partial + (size_t(tile) * kparts + kp) * kPart;
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int u = 0; u < VP; ++u)
#pragma unroll
            for (int j = 0; j < NJ; ++j)
                __hip_atomic_store(&mine[((i * VP + u) * NJ + j) * kThreads + tid], fin[i][u][j], __ATOMIC_RELAXED,
                                   __HIP_MEMORY_SCOPE_AGENT);
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
    __builtin_amdgcn_s_waitcnt(0);
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
    __syncthreads();
    if (tid == 0)
        sh.last_flag = __hip_atomic_fetch_add(&a.counters[tile], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == kparts - 1;
    __syncthreads();
    if (!sh.last_flag) return;
    if (tid == 0) __hip_atomic_store(&a.counters[tile], 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    const float *parts = a.partial + size_t(tile) * kparts * kPart;
    for (uint32_t p0 = 0; p0 < kparts; p0 += 4) {  // four parts per round trip, added in part order
        float pv[4][MI][VP][NJ];
#pragma unroll
        for (int z = 0; z < 4; ++z) {
            const float *p = parts + size_t(__builtin_elementwise_min(p0 + uint32_t(z), kparts - 1)) * kPart;
#pragma unroll
            for (int i = 0; i < MI; ++i)
#pragma unroll
                for (int u = 0; u < VP; ++u)
#pragma unroll
                    for (int j = 0; j < NJ; ++j)
                        pv[z][i][u][j] = __hip_atomic_load(&p[((i * VP + u) * NJ + j) * kThreads + tid], __ATOMIC_RELAXED,
                                                           __HIP_MEMORY_SCOPE_AGENT);
        }
#pragma unroll
        for (int i = 0; i < MI; ++i)
#pragma unroll
            for (int u = 0; u < VP; ++u)
#pragma unroll
                for (int j = 0; j < NJ; ++j) {
                    float s = p0 == 0 ? 0.f : fin[i][u][j];
#pragma unroll
                    for (int z = 0; z < 4; ++z) s = p0 + uint32_t(z) < kparts ? s + pv[z][i][u][j] : s;
                    fin[i][u][j] = s;
                }
    }
    write_out();
}

// The exact Q6_K form, where batch 2-4 runs here (its own kernels are exact): row-major tensors (9-13 us
// against 14-15 us there) and V beside Q and K.  On the CDNA4 layout alone it loses (the down projection:
// 17.0 us at 2-4 tokens against 16.5 on the small-batch kernel, and 17.4 against 15.0 rounded at 5).
template <int TYPE, int LAYOUT, int ACC, int MI>
constexpr bool kExact = TYPE == Q6_K && ACC == ACC_FP32 && LAYOUT == ROW_MAJOR && MI == 1;

// (Two instances spill: Q6_K in the FP16 mode with 128-token tiles 12 bytes per lane, the row-major mixed kernel
// with 64-token tiles and WK 8 8 bytes.  Scratch accesses count as vector memory instructions too, in order, so
// they can only make the counted waits of the main loop stricter.)
template <int TYPE, int LAYOUT, int ACC, bool PAIR, int MI, int WK>
__global__ __launch_bounds__(kThreads) void gemm_skinny_kernel(const Args a) {
    // two LDS objects, so that the compiler does not take a DMA into one for a write to the other
    __shared__ __attribute__((aligned(16))) u32x4 X0[buf_len<MI, WK>()], X1[buf_len<MI, WK>()];
    __shared__ Shared sh;
    skinny_body<TYPE, LAYOUT, ACC, PAIR, MI, WK, kExact<TYPE, LAYOUT, ACC, MI>>(a, work_item(a), X0, X1, sh);
}

// Q, K and V in one launch where V is Q6_K (FP32 mode): a workgroup takes its matrix's form of the body.
template <int LAYOUT, int MI, int WK>
__global__ __launch_bounds__(kThreads) void gemm_skinny_mixed_kernel(const Args a) {
    __shared__ __attribute__((aligned(16))) u32x4 X0[buf_len<MI, WK>()], X1[buf_len<MI, WK>()];
    __shared__ Shared sh;
    const Item item = work_item(a);
    if (item.seg == a.q6_seg) skinny_body<Q6_K, LAYOUT, ACC_FP32, false, MI, WK, MI == 1>(a, item, X0, X1, sh);
    else skinny_body<Q4_K, LAYOUT, ACC_FP32, false, MI, WK, false>(a, item, X0, X1, sh);
}

struct Plan {
    uint32_t mi, wk, ntok, ncol, kparts;
    uint32_t cost;  // the model's estimate, tenths of a microsecond
};

uint32_t col_tiles(const uint32_t *rows, int nseg, bool pair, uint32_t wk) {
    const uint32_t per = (kWaves / wk) * (pair ? 32 : 64);
    uint32_t n = 0;
    for (int s = 0; s < nseg; ++s) n += (rows[s] + per - 1) / per;
    return n;
}

// Token tile, wave split and split K, by a cost model in tenths of a microsecond fitted to MI355X
// timings of the gate/up pair, the down projections and 2,048- and 4,096-row projections at 5 to 512
// tokens (within ~10% of them).  A call costs ~6 us of launch, ramp and tail; each round of workgroups
// (one per CU) ~6 us more and, per super-block a wave walks, kIter[kind][MI]: bound by the weight
// bytes at 32 tokens, by the matrix and decode work above.  Splitting K over workgroups (only to fill
// the first round) adds the hand-off, whose last arrival reads every part.
Plan plan_skinny(int type, uint32_t cols, const uint32_t *rows, int nseg, uint32_t batch, bool pair, bool f16,
                 const Tuning &t) {
    static constexpr uint32_t kIter[3][3] = {{25, 45, 0}, {22, 38, 0}, {23, 36, 80}};  // FP32 Q4_K, FP32 Q6_K, FP16
    const uint32_t *iter_cost = kIter[f16 ? 2 : type == Q6_K ? 1 : 0];
    Plan best{};
    const uint32_t nb = cols / kQK, cus = uint32_t(device_cus());
    const uint32_t forced = t.gemm_kparts >= 1 && uint32_t(t.gemm_kparts) <= nb ? uint32_t(t.gemm_kparts) : 0;
    uint32_t best_cost = ~0u;
    for (uint32_t m = 0; m < (f16 ? 3u : 2u); ++m) {
        const uint32_t mi = 1u << m, ntok = (batch + 32 * mi - 1) / (32 * mi);
        // without a forced tile: the shortest one that holds the batch, or a shorter one
        if (t.skinny_mi > 0 ? mi != uint32_t(t.skinny_mi) : m > 0 && batch <= 16 * mi) continue;
        for (uint32_t wk : {4u, 8u}) {
            if (wk == 8 && mi == 4) continue;  // no room for its x stages
            if (t.skinny_wk > 0 && uint32_t(t.skinny_wk) != wk && mi < 4) continue;
            const uint32_t ncol = col_tiles(rows, nseg, pair, wk), tiles = ncol * ntok;
            // of the parts that leave a wave as many super-blocks, the fewest
            for (uint32_t kp = forced ? forced : 1, iters = 0; kp <= nb && (forced || kp == 1 || tiles * kp <= cus);
                 kp = iters > 1 && !forced ? (nb + (iters - 1) * wk - 1) / ((iters - 1) * wk) : nb + 1) {
                const uint32_t rounds = (tiles * kp + cus - 1) / cus;
                iters = (nb + kp * wk - 1) / (kp * wk);
                const uint32_t cost = 60 + rounds * (60 + iters * iter_cost[m]) + (kp > 1 ? 10 + 4 * kp * mi : 0);
                if (cost < best_cost) {
                    best_cost = cost;
                    best = Plan{mi, wk, ntok, ncol, kp, cost};
                }
            }
        }
    }
    if (best.wk == 0) {  // a forced tile this mode does not have
        Tuning plain = t;
        plain.skinny_mi = plain.skinny_wk = 0;
        return plan_skinny(type, cols, rows, nseg, batch, pair, f16, plain);
    }
    return best;
}

// What a call takes, in microseconds, here and on the FP32-mode tile kernel that would run instead
// (ns_gemm_reg.hip for Q4_K on CDNA4, else ns_gemm.hip): least squares of the logarithms over 7,000 timings of
// random shapes each, weighted to where the two are close (there within 17% in 90 of 100).
//   here   call + rounds * (wg + super-blocks a wave walks * sb[32- or 64-token tile]) + part per K part and
//          32 tokens + mb per MB of output; rounds of one workgroup per CU, past the first by size plus `over`
//   tile   call + rounds * (wg + super-blocks * sb) + part_mb per MB of K parts (padded to tiles) + x_mb per MB
//          of x + col per super-block of columns (the group sums ahead) + last per K part that a last arrival
//          reads + mb; ns_gemm_reg.hip runs two workgroups per CU, from sb[0] alone to sb[1] together
struct Route {
    double call, wg, sb[2], part, over, mb;
    struct {
        double call, wg, sb[2], over, part_mb, x_mb, col, last, mb;
    } tile;
};
const Route &route_of(int type, int layout, bool pair) {
    static constexpr Route kPair{3.73, 1.71, {3.9, 6.01}, 0.29, 0.07, 0.4, {8.73, 0, {5.71, 7.75}, 0.22, 0.32, 0.18, 0.21, 1.19, 0.65}};
    static constexpr Route kQ4{2.7, 1.05, {3.83, 5.82}, 0.52, 0.24, 0.38, {9.91, 0, {5.16, 7.88}, 0.26, 0.33, 0.16, 0.24, 0.77, 0.15}};
    static constexpr Route kQ6{1.9, 1.81, {4.06, 5.25}, 0.62, 0.36, 0.3, {3.3, 0.71, {6.79, 6.79}, 0.68, 0.28, 0.05, 0.36, 1.02, 0.19}};
    static constexpr Route kQ4Row{3.16, 0.55, {4.68, 6.26}, 0.54, 0.24, 0.36, {8.3, 0, {8.78, 8.78}, 0.61, 0.31, 0.02, 0.33, 1.45, 0.19}};
    static constexpr Route kQ6Row{2.69, 0, {9.21, 9.01}, 0.62, 0.28, 0.08, {7.56, 3.17, {29.52, 29.52}, 0.54, 1.23, 0, 0.28, 1.23, 0.19}};
    if (layout == ROW_MAJOR) return type == Q4_K ? kQ4Row : kQ6Row;
    return pair ? kPair : type == Q4_K ? kQ4 : kQ6;
}
double out_mb(const uint32_t *rows, int nseg, uint32_t batch, bool pair) {
    double n = 0;
    for (int s = 0; s < nseg; ++s) n += rows[s];
    return n * batch * (pair ? 2 : 4) * 1e-6;
}
double skinny_us(const Route &r, const Plan &p, uint32_t cols, const uint32_t *rows, int nseg, uint32_t batch, bool pair) {
    const uint32_t nb = cols / kQK, iters = ((nb + p.kparts - 1) / p.kparts + p.wk - 1) / p.wk;
    const double q = double(p.ntok * p.ncol) * p.kparts / device_cus();
    return r.call + (q <= 1 ? 1 : q + r.over) * (r.wg + iters * r.sb[p.mi == 1 ? 0 : 1]) +
           (p.kparts > 1 ? r.part * p.kparts * p.mi : 0) + r.mb * out_mb(rows, nseg, batch, pair);
}
double tile_us(const Route &r, int type, int layout, uint32_t cols, uint32_t rows, uint32_t batch, bool pair, const Tuning &t) {
    const auto &c = r.tile;
    const bool reg = layout == CDNA4 && type == Q4_K;
    const TileGrid g = reg ? gemm_reg_grid(cols, rows, batch, pair, t) : gemm_grid(type, cols, rows, batch, pair, ACC_FP32, t);
    const double n = double(g.tiles) * g.kparts, q = n / device_cus();
    const uint32_t nb = cols / kQK, sb = (nb + g.kparts - 1) / g.kparts;
    const double rounds = reg ? (q <= 2 ? 1 : q / 2 + c.over) : (q <= 1 ? 1 : q + c.over);
    const double step = c.sb[0] + (c.sb[1] - c.sb[0]) * std::min(std::max(q - 1, 0.0), 1.0);
    const bool scatter = (g.tokens / 32) % g.kparts == 0 && q <= (reg ? 2 : 1);
    return c.call + rounds * (c.wg + sb * step) + (g.kparts > 1 ? c.part_mb * n * g.tokens * 256 * 4e-6 : 0) +
           c.x_mb * batch * cols * 2e-6 + c.col * nb + (g.kparts > 1 && !scatter ? c.last * g.kparts : 0) +
           c.mb * out_mb(&rows, 1, batch, pair);
}

template <int TYPE, int LAYOUT, int ACC, bool PAIR>
hipError_t launch_mi(const Plan &p, const Args &a, hipStream_t stream) {
    const dim3 grid(p.ntok * p.ncol * p.kparts), block(kThreads);
    if (p.mi == 1) {
        if (p.wk == 8) gemm_skinny_kernel<TYPE, LAYOUT, ACC, PAIR, 1, 8><<<grid, block, 0, stream>>>(a);
        else gemm_skinny_kernel<TYPE, LAYOUT, ACC, PAIR, 1, 4><<<grid, block, 0, stream>>>(a);
    } else if (p.mi == 2) {
        if (p.wk == 8) gemm_skinny_kernel<TYPE, LAYOUT, ACC, PAIR, 2, 8><<<grid, block, 0, stream>>>(a);
        else gemm_skinny_kernel<TYPE, LAYOUT, ACC, PAIR, 2, 4><<<grid, block, 0, stream>>>(a);
    } else {
        if constexpr (ACC == ACC_FP16) gemm_skinny_kernel<TYPE, LAYOUT, ACC, PAIR, 4, 4><<<grid, block, 0, stream>>>(a);
        else return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

template <int LAYOUT>
hipError_t launch_mixed(const Plan &p, const Args &a, hipStream_t stream) {
    const dim3 grid(p.ntok * p.ncol * p.kparts), block(kThreads);
    if (p.mi == 1) {
        if (p.wk == 8) gemm_skinny_mixed_kernel<LAYOUT, 1, 8><<<grid, block, 0, stream>>>(a);
        else gemm_skinny_mixed_kernel<LAYOUT, 1, 4><<<grid, block, 0, stream>>>(a);
    } else if (p.mi == 2) {
        if (p.wk == 8) gemm_skinny_mixed_kernel<LAYOUT, 2, 8><<<grid, block, 0, stream>>>(a);
        else gemm_skinny_mixed_kernel<LAYOUT, 2, 4><<<grid, block, 0, stream>>>(a);
    } else {
        return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

}  // namespace

// Whether this kernel is the faster one.  FP16 mode: by its plan's estimate against the tile kernel's
// (gate/up 128 tokens: 44 us here, 50 there; 225: 75 / 65; downs 225: 43-46 / 48-55; 320: 63-67 / 63).
// FP32 mode: by the two estimates of Route, 5% for their error.  Over 37,000 random shapes (256 to 32,768
// columns, 64 to 262,144 rows, 5 to 2,048 tokens) the choice is more than 5% slower than the tile kernels in
// 0.2% of them (0.5% for Q4_K on CDNA4) and more than 5% slower than this kernel in 1%; it takes 0.362 of the tile
// kernels' time (geometric mean), the better one of each two 0.361.  MI355X, this kernel against them (us):
//   gate/up 192 tokens: 81 / 94, 225: 106 / 95;  downs 512: 78-96 / 105-127, 775: 157-180 / 134-145
//   4096 x 3840, 1536 tokens: 89 / 114, row-major 93 / 95;  2048: 121 / 103, row-major 125 / 106
//   256 columns: 65,536 rows at 71 tokens 55 / 23 (the pair), Q6_K at 217 62 / 20
bool gemm_skinny_eligible(int type, int layout, int acc, uint32_t cols, uint32_t rows, uint32_t batch, bool pair,
                          const Tuning &t) {
    if (t.gemm_skinny == 0) return false;
    if (layout == NSMFFN || (layout == ROW_MAJOR && (acc == ACC_FP16 || pair))) return false;
    if (t.gemm_skinny > 0) return batch <= uint32_t(t.gemm_skinny);
    if (t.gemm_q4_reg == 0 && type == Q4_K && acc == ACC_FP32) return false;  // the LDS-tile kernel is asked for
    if (batch > 2048) return false;  // beyond what was measured
    Tuning plain = t;  // a forced number of K parts does not change the kernel
    plain.gemm_kparts = 0;
    const Plan p = plan_skinny(type, cols, &rows, 1, batch, pair, acc == ACC_FP16, plain);
    // (and a bound: past two rounds the weights are read once per token tile from beyond L2, which the
    // estimate leaves out: downs at 600 tokens 124-130 us here, 109 there)
    if (acc == ACC_FP16) return p.cost <= std::min(800u, gemm_f16_cost(cols, rows, batch, pair, plain));
    // one super-block and up to two workgroups per CU, which the estimate has in turn: 10.8 us here, 15.3 there
    if (type == Q4_K && layout == CDNA4 && cols == kQK && p.mi == 1 && p.ncol * p.ntok <= 2 * uint32_t(device_cus())) return true;
    const Route &r = route_of(type, layout, pair);
    return skinny_us(r, p, cols, &rows, 1, batch, pair) <= 0.95 * tile_us(r, type, layout, cols, rows, batch, pair, plain);
}

namespace {

// Batch 2-4: x comes by 16-byte DMA, and no small-batch kernel is asked for.
bool small_batch_possible(int type, const void *x, uint32_t batch, const Tuning &t) {
    return batch >= 2 && batch <= 4 && reinterpret_cast<uintptr_t>(x) % 16 == 0 && t.gemm_skinny != 0 &&
           (t.gemm_q4_reg != 0 || type != Q4_K) && t.mt_mfma != 0 && t.mt_parts <= 0 && t.mt_slabs <= 0 && t.mt_spw <= 0;
}

// What the small-batch kernels take at 2 and at 3-4 fp16 tokens, in microseconds: call, per super-block of columns
// (its serial part) and per 1,024 super-blocks (fitted as Route; within 20%).
double small_us(int type, int layout, uint32_t cols, uint32_t rows, uint32_t batch) {
    static constexpr double k[2][2][2][3] = {{{{7.0, 0.082, 0.0908}, {8.0, 0.11, 0.098}}, {{8.7, 0.103, 0.0928}, {8.1, 0.098, 0.1086}}},
                                             {{{10.0, 0.087, 0.0285}, {10.0, 0.087, 0.0285}}, {{8.2, 0.097, 0.0358}, {8.2, 0.097, 0.0358}}}};
    const double *c = k[layout == CDNA4][type == Q6_K][batch > 2];
    const uint32_t nb = cols / kQK;
    return c[0] + c[1] * nb + c[2] * (double(rows) * nb / 1024);
}

}  // namespace

// Row-major tensors by the two estimates (but for Q4_K at 2 tokens by 5% more, as that of the small-batch kernel is
// low); short rows, whose estimates are loose, stay there.  Q6_K of many super-blocks, and many Q6_K rows at 3-4
// tokens, are always here, where the small-batch kernel may take 1.5 times what its estimate has and this one does
// not (21,504 rows: 2,304 columns at 3 tokens 27 us here, 48 there, 15,360 at 2 tokens 140 / 208).  Over 31,300
// random shapes the choice is more than 5% slower than the small-batch kernels in 0.9% of them, and more than 5%
// slower than this one in 2.1% (2,048 x 3,840 at 3 tokens 9.4 us here, 12.4 there; Q6_K 64 x 3,840 13 / 10, 65,536 x
// 2,304 55 / 76).  Q4_K on CDNA4:
// here but for tall matrices of up to 15 super-blocks, which the small-batch kernel walks with a wave per slab and
// no hand-off (at up to two slabs per CU 0.58-1.00 of its time, at 65,536-262,144 rows 1.1-2.0 of it).  Q6_K on
// CDNA4: not exact here (kExact).
bool skinny_small_batch(int type, int layout, uint32_t cols, uint32_t rows, const void *x, uint32_t batch, const Tuning &t) {
    if (layout == NSMFFN || (type == Q6_K && layout == CDNA4) || !small_batch_possible(type, x, batch, t)) return false;
    if (t.gemm_skinny > 0) return batch <= uint32_t(t.gemm_skinny);
    const uint32_t nb = cols / kQK;
    if (layout == CDNA4) return nb > 15 || rows <= 2 * uint32_t(device_cus()) * kRowTile;
    if (type == Q6_K && ((batch > 2 && nb >= 3 && rows >= 20480) || (nb >= 6 && uint64_t(rows) * nb >= 61440))) return true;
    if (nb < (type == Q4_K ? 2u : 6u)) return false;
    Tuning plain = t;
    plain.gemm_kparts = 0;
    return skinny_us(route_of(type, layout, false), plan_skinny(type, cols, &rows, 1, batch, false, false, plain), cols, &rows, 1,
                     batch, false) <= (type == Q4_K && batch == 2 ? 1.0 : 1.05) * small_us(type, layout, cols, rows, batch);
}

// Q, K and V (or Q and a K that is V too) in one launch: against the launches of their own that they would take.
bool skinny_qkv_eligible(int layout, uint32_t cols, const uint32_t *rows, int nseg, int last_type, const void *x,
                         uint32_t batch, const Tuning &t) {
    if (t.gemm_skinny == 0 || layout == NSMFFN || t.gemm_q4_reg == 0 || batch > 2048) return false;
    const bool small = batch <= 4;
    if (small && !small_batch_possible(Q4_K, x, batch, t)) return false;
    if (t.gemm_skinny > 0) return batch <= uint32_t(t.gemm_skinny);
    Tuning plain = t;
    plain.gemm_kparts = 0;
    double total = 0;
    for (int s = 0; s < nseg; ++s) total += rows[s];
    Route mix = route_of(Q4_K, layout, false);
    if (last_type == Q6_K)  // by the share of the column tiles that are Q6_K
        for (int m = 0; m < 2; ++m) mix.sb[m] += (route_of(Q6_K, layout, false).sb[m] - mix.sb[m]) * (rows[nseg - 1] / total);
    const double together =
        skinny_us(mix, plan_skinny(Q4_K, cols, rows, nseg, batch, false, false, plain), cols, rows, nseg, batch, false);
    if (together <= 18) return true;  // less than the launches alone, and the host would take longer to find out
    double apart = last_type ? 0 : 4;  // a tied V is a copy of K
    for (int s = 0; s < nseg; ++s) {
        const int type = s == nseg - 1 && last_type ? last_type : Q4_K;
        const Route &r = route_of(type, layout, false);
        const double own = skinny_us(r, plan_skinny(type, cols, rows + s, 1, batch, false, false, plain), cols, rows + s, 1, batch, false);
        if (!small) apart += std::min(own, tile_us(r, type, layout, cols, rows[s], batch, false, plain));
        else apart += skinny_small_batch(type, layout, cols, rows[s], x, batch, t) ? own : small_us(type, layout, cols, rows[s], batch);
    }
    return together <= apart;
}

void gemm_skinny_workspace_need(int type, uint32_t cols, const uint32_t *rows, int nseg, uint32_t batch, bool pair,
                                int acc, const Tuning &t, size_t *part_floats, size_t *counters) {
    const Plan p = plan_skinny(type, cols, rows, nseg, batch, pair, acc == ACC_FP16, t);
    const size_t tiles = size_t(p.ncol) * p.ntok;
    *part_floats = p.kparts > 1 ? tiles * p.kparts * (p.mi * 32 * (kWaves / p.wk) * 64) : 0;
    *counters = p.kparts > 1 ? tiles : 0;
}

hipError_t launch_gemm_skinny(int type, int layout, int acc, const uint8_t *const *w, const uint8_t *up, void *const *out,
                              const uint32_t *rows, int nseg, const uint16_t *x, uint32_t cols, uint32_t batch,
                              float *partial, uint32_t *counters, const Tuning &t, hipStream_t stream, int last_type,
                              void *copy) {
    const bool pair = up != nullptr, f16 = acc == ACC_FP16;
    const bool mixed = last_type != 0 && last_type != type;  // Q4_K matrices, then one of Q6_K
    if (nseg < 1 || nseg > kMaxSeg || (pair && nseg != 1)) return hipErrorInvalidValue;
    if (mixed && (type != Q4_K || f16 || pair || nseg < 2)) return hipErrorInvalidValue;
    const Plan p = plan_skinny(type, cols, rows, nseg, batch, pair, f16, t);
    Args a{};
    uint32_t ct = 0;
    for (int s = 0; s < kMaxSeg; ++s) {
        const int z = s < nseg ? s : nseg - 1;
        a.w[s] = w[z];
        a.out[s] = out[z];
        a.rows[s] = rows[z];
        if (s < nseg) ct += col_tiles(rows + s, 1, pair, p.wk);
        a.ct_end[s] = ct;
    }
    a.up = up;
    a.q6_seg = uint32_t(nseg - 1);
    a.copy = copy;
    a.x = x;
    a.partial = partial;
    a.counters = counters;
    a.cols = cols;
    a.batch = batch;
    a.ntok = p.ntok;
    a.ncol = p.ncol;
    a.kparts = p.kparts;
    if (mixed)
        return layout == CDNA4 ? launch_mixed<CDNA4>(p, a, stream)
               : layout == ROW_MAJOR ? launch_mixed<ROW_MAJOR>(p, a, stream) : hipErrorInvalidValue;
    if (layout == CDNA4) {
        if (pair)
            return f16 ? launch_mi<Q4_K, CDNA4, ACC_FP16, true>(p, a, stream) : launch_mi<Q4_K, CDNA4, ACC_FP32, true>(p, a, stream);
        if (type == Q4_K)
            return f16 ? launch_mi<Q4_K, CDNA4, ACC_FP16, false>(p, a, stream) : launch_mi<Q4_K, CDNA4, ACC_FP32, false>(p, a, stream);
        return f16 ? launch_mi<Q6_K, CDNA4, ACC_FP16, false>(p, a, stream) : launch_mi<Q6_K, CDNA4, ACC_FP32, false>(p, a, stream);
    }
    if (layout != ROW_MAJOR || f16 || pair) return hipErrorInvalidValue;
    return type == Q4_K ? launch_mi<Q4_K, ROW_MAJOR, ACC_FP32, false>(p, a, stream)
                        : launch_mi<Q6_K, ROW_MAJOR, ACC_FP32, false>(p, a, stream);
}

}  // namespace ns
