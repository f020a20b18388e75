// Prefill GEMM, bf16 variant: Y[M, N] = X[M, K] . bf16(W)[N, K]^T
// with fp32 accumulation, W the exactly decoded weights of Q8_0, Q4_0, Q4_K or Q6_K blocks
// (semantics: quantMatvec per row of X, QuantizedOps.java:27 / CpuBackend.java:708-725).
//
// Structure:
//  - Tile 32 TM x 32 WV per workgroup of WV waves. Wave w owns columns [32 w, +32) for all rows:
//    TM v_mfma_f32_32x32x16_bf16 accumulators, no partial tiles to add at the end. With WV = 4
//    two workgroups share a CU (one's barriers, prologue and stores are covered by the other's
//    matrix work); with WV = 8 the two waves of a SIMD share X. Small grids: WV = 2 and KG groups
//    of such waves in a workgroup, which split its range of K.
//  - K advances in stages of two 32-blocks. Lane (r, h) = (lane % 32, lane / 32) supplies block
//    h of the stage, elements 8 p .. 8 p + 7 to the stage's MFMA p = 0..3, for A (X) and B (W)
//    alike: every lane dequantizes one whole block of one W row, so the scale decode is paid
//    once per 32 weights, and each weight is dequantized once per workgroup.
//  - Everything goes straight from global memory into LDS (buffer_load ... lds): X as two stage
//    buffers of rows of 128 bytes (16-byte chunk c of row r at slot c ^ ((r / 2) % 8): the 16
//    rows of a quarter-wave read fall on distinct banks); W in units of two stages, 64 bytes of
//    4-bit quants per row (chunk c of row r at slot c ^ ((r / 4) % 4)) or 128 of Q8_0's (placed
//    as X's rows), Q6_K's high bits as 32 bytes per row, and the scale words. A wave loads the W
//    rows it uses itself, so W needs no barrier; X needs one per stage.
//  - Dequantization to the decoder's fp32 value and then bf16 (round to nearest even). 4- and
//    6-bit codes: a field masked into the low bits of an fp16 is the subnormal q 2^-24 (q 2^-20
//    for a high nibble), and v_fma_mix_f32 computes fma(q 2^-24, s 2^24, o) = fma(q, s, o) with
//    one rounding and no conversion:
//      Q4_0  w = d (q - 8)                 = fma(d, q, -8 d)       (exact)
//      Q4_K  w = fl((d sc) q - dmin m)     = fma(d sc, q, -dmin m) (d sc q is exact in fp32)
//      Q6_K  w = fl((d sc) (q - 32))       = fma(d sc, q, -32 d sc)
//      Q8_0  w = d q                                               (exact)
//  - Stage i: wait for X of stage i, barrier, issue X of stage i + 1 (into the buffer of stage
//    i - 1) and the W unit that is read next but one, then the MFMAs of stage i. The B operands
//    of MFMA p + 1 are dequantized between those of p (the next stage's first ones at the end),
//    so the vector ALU works in the shadow of the matrix core.
//  - The LDS buffers are separate __shared__ arrays and the stage loop is unrolled over their
//    common period, so the compiler knows which loads write the buffer a read touches.
// Loads past K, past the workgroup's K range, or of rows past M or N return zeros (out-of-range
// offsets); zero quants with zero scales decode to 0.
// grid = (ceil(M / (32 TM)) * ceil(N / (32 WV)), S) workgroups of 64 WV threads: S K splits of
// split_stages stages each (a multiple of 4 when S > 1; partial tiles go to part[s][M][N], added
// by sum_splits_kernel). Requires K % 64 == 0 (Q8_0), K % 128 == 0 (Q4_0) or K % 256 == 0,
// M * K * 2 < 2^31, and N * K (Q8_0) or N * K / 2 < 2^31.
#pragma once

#include <type_traits>

#include "gemm_wide.h"

namespace j4q {
namespace gt {

using gw::bf16x2;
using gw::bf16x8;
using gw::dma16;
using gw::dma4;
using gw::f32x2;
using gw::kOob;
using gw::lds_barrier;
using gw::load_order;
using gw::make_rsrc;
using gw::u32x2;
using gw::u32x4;
using gw::wait_vm_lgkm0;
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef _Float16 half2_t __attribute__((ext_vector_type(2)));

constexpr float kTwo24 = 16777216.0f, kTwo20 = 1048576.0f;

// bf16(fma(q, s, off)) of the four codes in the fp16 subnormals (even: elements 0, 2; odd: 1, 3).
__device__ __forceinline__ u32x2 deq4(uint32_t even, uint32_t odd, float s, float off) {
    const half2_t e = __builtin_bit_cast(half2_t, even), o = __builtin_bit_cast(half2_t, odd);
    const float f0 = __builtin_fmaf((float)e.x, s, off), f1 = __builtin_fmaf((float)o.x, s, off);
    const float f2 = __builtin_fmaf((float)e.y, s, off), f3 = __builtin_fmaf((float)o.y, s, off);
    u32x2 r;
    r[0] = __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2{f0, f1}), bf16x2));
    r[1] = __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2{f2, f3}), bf16x2));
    return r;
}

// A W unit of a tile in LDS: two stages (four 32-blocks) of the 32 WV rows of W that the tile's waves
// use, loaded by the wave that uses them: quants, Q6_K's high bits, scale words (one array, so few
// that the compiler tracks the loads into each of them apart).
template <int FMT, int WV>
struct WUnit {
    static constexpr int QR = FMT == Q8_0 ? 128 : 64;              // bytes of quants per row
    static constexpr int QL = QR / 32;                             // their loads per wave
    static constexpr int kLoads = QL + (FMT == Q6_K ? 3 : 1);      // all loads per wave
    static constexpr int kH = 32 * WV * QR;                        // offset of the high bits
    static constexpr int kS = kH + (FMT == Q6_K ? 32 * WV * 32 : 0);      // ... of the scale words
    static constexpr int kSlot = FMT == Q4_K ? 1024 : FMT == Q6_K ? 512 : 256;  // scale words of one wave
    static constexpr int kBytes = kS + WV * kSlot;

    __amdgpu_buffer_rsrc_t qr, hr, sr;
    uint32_t qoff[QL], hoff, soff, doff;
    int wave;

    // 16-byte chunk c of row r sits at slot c ^ swz(r): the rows of a quarter-wave read fall on
    // distinct banks.
    static __device__ __forceinline__ int swz(int row) { return QR == 128 ? (row >> 1) & 7 : (row >> 2) & 3; }

    // nw: the wave's first row of W.
    __device__ __forceinline__ void init(const QMat &w, int nw, int wave_, int lane) {
        const int N = (int)w.rows, K = (int)w.cols, nsb = K / 256;
        wave = wave_;
        // Quants: a load fills 1024 / QR rows (QR / 16 lanes a row); the slot of a lane holds the
        // chunk that the row's swizzle puts there.
        const uint32_t qrow = FMT == Q8_0 ? (uint32_t)K : (uint32_t)(K / 2);
        qr = make_rsrc(w.qs, (uint64_t)N * qrow);
#pragma unroll
        for (int j = 0; j < QL; j++) {
            const int row = j * (1024 / QR) + lane / (QR / 16), c = (lane % (QR / 16)) ^ swz(row), n = nw + row;
            qoff[j] = n < N ? (uint32_t)n * qrow + (uint32_t)c * 16u : kOob;
        }
        // Q6_K high bits: lane L: 16-byte half L % 2 of the unit's 32 bytes of row L / 2.
        const int n2 = nw + (lane >> 1);
        hr = make_rsrc(w.qh, FMT == Q6_K ? (uint64_t)N * (uint64_t)K / 4u : 0);
        hoff = n2 < N ? (uint32_t)n2 * (uint32_t)(K / 4) + (uint32_t)(lane & 1) * 16u : kOob;
        // Scale words into this wave's slot:
        //  Q8_0, Q4_0: lane L: dword L % 2 of the unit's four fp16 d of row L / 2;
        //  Q4_K: lane r < 32: row r's 16-byte superblock record (the other lanes write zeros behind:
        //        a branch around them would blur the compiler's wait counts);
        //  Q6_K: lane L: dword L % 2 of the unit's eight int8 group scales of row L / 2; then lane
        //        r < 32: the aligned dword holding row r's fp16 superblock d (the d section follows
        //        the sc section in the matrix's allocation, so one buffer resource from sc to the
        //        end of d's 256-byte-aligned section serves both).
        const uint32_t d_rel = FMT == Q6_K ? (uint32_t)(w.d - w.sc) : 0u;
        sr = make_rsrc(w.sc, FMT == Q6_K ? (uint64_t)d_rel + align256((uint64_t)N * (uint64_t)nsb * 2u)
                                         : (uint64_t)N * (uint64_t)(K / 16));
        soff = doff = kOob;
        if constexpr (FMT == Q4_K) {
            if (lane < 32 && nw + lane < N) soff = (uint32_t)(nw + lane) * (uint32_t)(K / 16);
        } else {
            if (n2 < N) soff = (uint32_t)n2 * (uint32_t)(K / 16) + (uint32_t)(lane & 1) * 4u;
            if (FMT == Q6_K && lane < 32 && nw + lane < N) doff = d_rel + (uint32_t)(nw + lane) * (uint32_t)(nsb * 2);
        }
    }
    // Unit u (stages 2 u and 2 u + 1) into wb; zeros when not live.
    __device__ __forceinline__ void load(int u, bool live, uint8_t *wb) const {
        uint8_t *const slot = wb + kS + wave * kSlot;
        const uint32_t uu = live ? (uint32_t)u : 0u;
#pragma unroll
        for (int j = 0; j < QL; j++) dma16(qr, wb + (wave * QL + j) * 1024, live ? qoff[j] : kOob, uu * (uint32_t)QR);
        if constexpr (FMT == Q6_K) {
            dma16(hr, wb + kH + wave * 1024, live ? hoff : kOob, uu * 32u);
            dma4(sr, slot, live && soff != kOob ? soff + uu * 8u : kOob);
            dma4(sr, slot + 256, live && doff != kOob ? (doff + (uu >> 1) * 2u) & ~3u : kOob);
        } else if constexpr (FMT == Q4_K) {
            dma16(sr, slot, live ? soff : kOob, (uu >> 1) * 16u);
        } else {
            dma4(sr, slot, live && soff != kOob ? soff + uu * 8u : kOob);
        }
    }
};

template <int FMT, int WV, int TM>
struct Tile {
    static constexpr int BM = 32 * TM, BN = 32 * WV;
    static constexpr int XL = 4 * TM / WV;  // X loads per wave and stage
    static constexpr int kX = BM * 128;
    static_assert(4 * TM % WV == 0, "whole X loads per wave");
};

// KG = 2 or 4 (WV = 2; KG = 2 also WV = 4): as many groups of waves, each with buffers of its own, take a part
// of the range of K each (split_stages, a multiple of 4; K a multiple of 256). Their sums meet through LDS, a
// quarter of the rows of a 32-row tile or a half in each group, and are added in group order.
template <int FMT, int WV, int TM, int KG = 1>
__global__ void __launch_bounds__(64 * WV * KG, 2)
gemm_tile(QMat w, const uint16_t *__restrict__ x, float *__restrict__ y, int M, int split_stages,
          float *__restrict__ part) {
    using T = Tile<FMT, WV, TM>;
    using U = WUnit<FMT, WV>;
    constexpr int BM = T::BM, BN = T::BN, QR = U::QR, WL = U::kLoads, XL = T::XL;
    static_assert(2 * KG * (T::kX + U::kBytes) <= 163840, "LDS");
    __shared__ __attribute__((aligned(1024))) uint8_t xs0[KG * T::kX], xs1[KG * T::kX];
    __shared__ __attribute__((aligned(1024))) uint8_t ws0[KG * U::kBytes], ws1[KG * U::kBytes];
    const int N = (int)w.rows, K = (int)w.cols;
    const int kg = KG > 1 ? __builtin_amdgcn_readfirstlane((int)threadIdx.x / (64 * WV)) : 0;  // K group
    const int sbeg = ((int)blockIdx.y * KG + kg) * split_stages, send = sbeg + split_stages, all = K / 64;
    const int ns = send < all ? send : all;  // stages [sbeg, ns)
    const int nl = KG > 1 ? send : ns;       // K groups run the same number (zeros past ns), for the barriers
    // Workgroup b runs on XCD b % 8, and each XCD takes a contiguous range of tiles. Tiles go
    // down groups of 4 row tiles (a row tile's X costs about twice a column tile's W), so the
    // tiles that one XCD runs at a time share both in its L2.
    const int mt = (M + BM - 1) / BM, total = (int)gridDim.x, nt = total / mt;
    int tile = (int)blockIdx.x;
    if (total % 8 == 0) tile = (tile % 8) * (total / 8) + tile / 8;
    const int mg = tile / (4 * nt), gm = mt - 4 * mg < 4 ? mt - 4 * mg : 4, rem = tile - 4 * mg * nt;
    const int m0 = (4 * mg + rem % gm) * BM, n0 = (rem / gm) * BN;

    const int lane = (int)threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6) % WV;
    const int r32 = lane & 31, h = lane >> 5;

    // X load j of this wave fills rows 8 (WV j + wave) .. + 7 of the stage buffer; lane L fills
    // slot L % 8 of row 8 (WV j + wave) + L / 8, which holds chunk (L % 8) ^ ((row / 2) % 8).
    const __amdgpu_buffer_rsrc_t xr = make_rsrc(x, (uint64_t)M * (uint64_t)K * 2u);
    uint32_t xoff[XL];
#pragma unroll
    for (int j = 0; j < XL; j++) {
        const int row = 8 * (WV * j + wave) + (lane >> 3), c = (lane & 7) ^ ((row >> 1) & 7);
        xoff[j] = m0 + row < M ? (uint32_t)(m0 + row) * (uint32_t)K * 2u + (uint32_t)c * 16u : kOob;
    }
    const int nw = n0 + 32 * wave;  // this wave's first column
    const int nsb = K / 256;
    U unit;
    unit.init(w, nw, wave, lane);

    // The loads of stage i of X, and of W unit u (stages 2 u and 2 u + 1).
    auto load_x = [&](int i, uint8_t *xb) __attribute__((always_inline)) {
        const uint32_t so = i < ns ? (uint32_t)i * 128u : 0u;
#pragma unroll
        for (int j = 0; j < XL; j++) dma16(xr, xb + (WV * j + wave) * 1024, i < ns ? xoff[j] : kOob, so);
    };
    auto load_w = [&](int u, uint8_t *wb) __attribute__((always_inline)) { unit.load(u, 2 * u < ns, wb); };

    // One block of one W row as it lies in LDS; scale s and offset o of its elements 0..15 and
    // 16..31 (s carries the power of two of the codes' units).
    struct Raw {
        u32x4 q[U::QL / 2];
        u32x2 hi;
        u32x4 s;
    };
    struct Scale {
        float s[2], o[2];
    };
    // Stage j's block h of row r32, from its unit's buffer.
    auto read_raw = [&](int j, const uint8_t *wb, Raw &o) __attribute__((always_inline)) {
        const int swz = U::swz(r32), blk = 2 * (j & 1) + h;  // blk: block within the unit
        const uint8_t *const row = wb + (32 * wave + r32) * QR, *const slot = wb + U::kS + wave * U::kSlot;
#pragma unroll
        for (int c = 0; c < U::QL / 2; c++)
            o.q[c] = *reinterpret_cast<const u32x4 *>(row + (((U::QL / 2 * blk + c) ^ swz) << 4));
        if constexpr (FMT == Q4_K) o.s = *reinterpret_cast<const u32x4 *>(slot + r32 * 16);
        else o.s[0] = *reinterpret_cast<const uint16_t *>(slot + r32 * 8 + blk * 2);
        if constexpr (FMT == Q6_K) {
            o.hi = *reinterpret_cast<const u32x2 *>(wb + U::kH + (32 * wave + r32) * 32 + blk * 8);
            o.s[1] = *reinterpret_cast<const uint32_t *>(slot + 256 + r32 * 4);
        }
    };
    auto decode_scale = [&](int j, const Raw &raw, Scale &c) __attribute__((always_inline)) {
        if constexpr (FMT == Q8_0) {
            c.s[0] = half_bits_to_float(raw.s[0]);
        } else if constexpr (FMT == Q4_0) {
            const float d = half_bits_to_float(raw.s[0]);
            c.s[0] = d * kTwo24;
            c.s[1] = d * kTwo20;
            c.o[0] = c.o[1] = -8.0f * d;
        } else if constexpr (FMT == Q4_K) {
            const int jsb = 2 * (j & 3) + h;
            const uint32_t sc = __builtin_amdgcn_ubfe(raw.s[1], 4 * jsb, 4) | (__builtin_amdgcn_ubfe(raw.s[3], 2 * jsb, 2) << 4);
            const uint32_t mn = __builtin_amdgcn_ubfe(raw.s[2], 4 * jsb, 4) | (__builtin_amdgcn_ubfe(raw.s[3], 16 + 2 * jsb, 2) << 4);
            const float d1 = half_bits_to_float(raw.s[0] & 0xFFFFu) * (float)sc;
            c.s[0] = d1 * kTwo24;
            c.s[1] = d1 * kTwo20;
            c.o[0] = c.o[1] = -(half_bits_to_float(raw.s[0] >> 16) * (float)mn);
        } else {
            const uint32_t odd = ((uint32_t)(nw + r32) * (uint32_t)nsb + (uint32_t)(j >> 2)) & 1u;
            const float d = half_bits_to_float(odd ? raw.s[1] >> 16 : raw.s[1] & 0xFFFFu);
            const float da = d * (float)(int8_t)(raw.s[0] & 0xFFu), db = d * (float)(int8_t)(raw.s[0] >> 8);
            c.s[0] = da * kTwo24;
            c.o[0] = -32.0f * da;
            c.s[1] = db * kTwo20;
            c.o[1] = -32.0f * db;
        }
    };
    // Operand p: elements 8 p .. 8 p + 7 of the block.
    auto operand = [&](const Raw &raw, const Scale &c, int p) __attribute__((always_inline)) -> bf16x8 {
        if constexpr (FMT == Q8_0) {
            return gw::dequant8(u32x2{raw.q[p >> 1][2 * (p & 1)], raw.q[p >> 1][2 * (p & 1) + 1]}, c.s[0]);
        } else {
            const int hi = p >> 1, d0 = 2 * (p & 1);
            u32x4 r;
#pragma unroll
            for (int k = 0; k < 2; k++) {
                const uint32_t v = raw.q[0][d0 + k], t = v >> 8;
                const uint32_t mask = hi ? 0x00F000F0u : 0x000F000Fu;
                uint32_t even = v & mask, odd = t & mask;
                if constexpr (FMT == Q6_K) {
                    // ql dwords d0, d0 + 1 share qh dword p % 2; the odd one's fields sit 8 bits on
                    const uint32_t hw = k ? __builtin_amdgcn_alignbit(raw.hi[p & 1], raw.hi[p & 1], 8) : raw.hi[p & 1];
                    const uint32_t hm = hi ? 0x03000300u : 0x00300030u;
                    even |= hw & hm;
                    odd |= (hw >> 2) & hm;
                }
                const u32x2 f = deq4(even, odd, c.s[hi], c.o[hi]);
                r[2 * k] = f[0];
                r[2 * k + 1] = f[1];
            }
            return __builtin_bit_cast(bf16x8, r);
        }
    };

    f32x16 acc[TM];
#pragma unroll
    for (int t = 0; t < TM; t++) acc[t] = f32x16{};
    const int aoff = r32 * 128, asw = (r32 >> 1) & 7;
    auto read_a = [&](const uint8_t *xb, int p, bf16x8 (&a)[TM]) __attribute__((always_inline)) {
#pragma unroll
        for (int t = 0; t < TM; t++)
            a[t] = *reinterpret_cast<const bf16x8 *>(xb + t * 32 * 128 + aoff + (((4 * h + p) ^ asw) << 4));
    };
    Raw raw[2];   // this lane's block of the current stage and of the next one
    Scale sc[2];
    bf16x8 b[2];  // B operands of MFMA p and p + 1
    // Stage number S of the period (S = (i - sbeg) % 4), so the buffers are constants. It reads
    // stage i + 1's block of unit (i + 1) / 2; odd stages load the unit after it. At the start,
    // what may be outstanding is what was issued after X of stage i: a unit, first read in stage
    // i + 1.
    auto stage = [&](auto S_, int i) __attribute__((always_inline)) {
        constexpr int S = decltype(S_)::value, cur = S & 1;
        uint8_t *const xb = (cur ? xs1 : xs0) + kg * T::kX, *const xn = (cur ? xs0 : xs1) + kg * T::kX;
        constexpr int ur = (S + 1) / 2 % 2, un = (S + 3) / 2 % 2;
        uint8_t *const wc = (ur ? ws1 : ws0) + kg * U::kBytes, *const wn = (un ? ws1 : ws0) + kg * U::kBytes;
        wait_vm_lgkm0<S % 2 == 0 ? WL : 0>();
        lds_barrier();
        bf16x8 a[2][TM];
        read_a(xb, 0, a[0]);
        read_raw(i + 1, wc, raw[cur ^ 1]);
        load_x(i + 1, xn);
        load_order();  // X first: the wait at an even stage leaves the newest unit of W outstanding
        if constexpr (S % 2 == 1) load_w((i + 3) / 2, wn);
        // issue the loads first (not where that costs registers: Q6_K at 256 rows would spill)
        if constexpr (TM < 8 || FMT != Q6_K) __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int p = 0; p < 4; p++) {
            if (p < 3) read_a(xb, p + 1, a[(p + 1) & 1]);
            if (p == 1) decode_scale(i + 1, raw[cur ^ 1], sc[cur ^ 1]);
#pragma unroll
            for (int t = 0; t < TM; t++) acc[t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[p & 1][t], b[p & 1], acc[t], 0, 0, 0);
            b[(p + 1) & 1] = p < 3 ? operand(raw[cur], sc[cur], p + 1) : operand(raw[cur ^ 1], sc[cur ^ 1], 0);
        }
        // computed here, between the MFMAs, although the last stage does not use it
        asm volatile("" : "+v"(b[0]));
    };

    // Prologue: what the stages before the first would have issued, in their order, then the
    // first stage's block and first operand.
    load_w(sbeg / 2, ws0 + kg * U::kBytes);
    load_order();
    load_x(sbeg, xs0 + kg * T::kX);
    load_order();
    load_w(sbeg / 2 + 1, ws1 + kg * U::kBytes);
    wait_vm_lgkm0<XL + WL>();
    asm volatile("" ::: "memory");
    read_raw(sbeg, ws0 + kg * U::kBytes, raw[0]);
    decode_scale(sbeg, raw[0], sc[0]);
    b[0] = operand(raw[0], sc[0], 0);
    // Whole periods in the loop: with an exit between stages the compiler takes the loads in flight at
    // the loop's head for any stage's, and waits there for all of them (2048 x 14336 x 4096 Q4_K 230 ->
    // 228 us, 512 x 4096 x 4096 31.9 -> 30.8).
#define J4Q_STAGE(S) stage(std::integral_constant<int, S>{}, i + S);
    int i = sbeg;
    for (; i + 4 <= nl; i += 4) {
        J4Q_STAGE(0) J4Q_STAGE(1) J4Q_STAGE(2) J4Q_STAGE(3)
    }
    if constexpr (KG == 1 && (FMT == Q8_0 || FMT == Q4_0)) {
        if (i < ns) {
            J4Q_STAGE(0)
            if (i + 1 < ns) {
                J4Q_STAGE(1)
                if (i + 2 < ns) J4Q_STAGE(2)
            }
        }
    }
#undef J4Q_STAGE
    __builtin_amdgcn_s_waitcnt(0);  // no LDS load outlives the workgroup
    // Result element v of tile t: row 32 t + 8 (v / 4) + 4 h + v % 4, column r32.
    float *const out = part ? part + (int64_t)blockIdx.y * M * N : y;
    const int col = nw + r32;
    if constexpr (KG > 1) {
        // elements 4 q .. 4 q + 3 of the tiles: through the X buffers, which hold them exactly (KG = 2: the two
        // quarters that a group gives away)
        static_assert((KG == 4 && WV == 2) || (KG == 2 && WV <= 4), "the groups' quarters in the X buffers");
        typedef float f32x4 __attribute__((ext_vector_type(4)));
        auto at = [&](int g, int t, int q) __attribute__((always_inline)) -> f32x4 & {
            if (KG == 2) return reinterpret_cast<f32x4 *>(q % 2 ? xs1 : xs0)[((g * TM + t) * WV + wave) * 64 + lane];
            return reinterpret_cast<f32x4 *>(q < 2 ? xs0 : xs1)[(((g * TM + t) * 2 + q % 2) * WV + wave) * 64 + lane];
        };
        auto quarter = [&](int t, int q) __attribute__((always_inline)) {
            return f32x4{acc[t][4 * q], acc[t][4 * q + 1], acc[t][4 * q + 2], acc[t][4 * q + 3]};
        };
        __syncthreads();
#pragma unroll
        for (int t = 0; t < TM; t++)
#pragma unroll
            for (int q = 0; q < 4; q++)
                if (q / (4 / KG) != kg) at(kg, t, q) = quarter(t, q);
        __syncthreads();
#pragma unroll
        for (int t = 0; t < TM; t++)
#pragma unroll
            for (int q = 0; q < 4; q++) {
                if (q / (4 / KG) != kg) continue;
                f32x4 s = kg == 0 ? quarter(t, q) : at(0, t, q);
#pragma unroll
                for (int g = 1; g < KG; g++) s += kg == g ? quarter(t, q) : at(g, t, q);
#pragma unroll
                for (int v = 0; v < 4; v++) {
                    const int row = m0 + 32 * t + 8 * q + 4 * h + v;
                    if (row < M && col < N) out[(int64_t)row * N + col] = s[v];
                }
            }
        return;
    }
#pragma unroll
    for (int t = 0; t < TM; t++)
#pragma unroll
        for (int v = 0; v < 16; v++) {
            const int row = m0 + 32 * t + 8 * (v >> 2) + 4 * h + (v & 3);
            if (row < M && col < N) out[(int64_t)row * N + col] = acc[t][v];
        }
}

}  // namespace gt
}  // namespace j4q
