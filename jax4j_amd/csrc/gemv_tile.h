// Batched GEMV for more rows than one launch of gemv_mfma.h takes: y[b][n] = sum_k W[n, k] x[b][k]
// (+ add[b][n]) with W streamed once for 32 or 64 rows of x, split-layout weights, exact codes.
//
// The 16-row kernel streams and unpacks W once per 16 rows, and is bound by that unpacking (140
// vector instructions per 16 x 256 weights). Here the unpacked codes of a 32 x 32 block feed the
// products of up to 64 rows. Measured (us, 16-row launches -> this): 61 rows Q6_K 4096 x 14336 83.4 ->
// 42.7 (35 the tile kernel, 5 each the split of x and the sum of the K splits), Q4_K 4096 x 4096 36.9
// -> 21.5, 64 rows Q4_K 28672 x 4096 97 -> 67, 256 rows Q4_K 4096 x 4096 153 -> 39, 48 rows Q8_0
// 11008 x 4096 54.5 -> 32.5. The tile kernel is bound by no one unit: at 64 x 28672 x 4096 the matrix
// cores are busy 18 of 61 us, the vector units about 20, and the two waves of a SIMD overlap them
// only in part; without its loads it takes 45.
//
// Arithmetic (as gemv_mfma.h): x is scaled per row and K split by a power of two 2^e (max |x| 2^e over
// the split's 512 to 1024 columns of the row in [2^14, 2^15)) and split into hi + lo fp16 by
// split_x_kernel: 22 significant bits for elements down to 2^-16 of that maximum (2^-12 for elements
// 16..31 of a 4- or 6-bit block, stored times 1/16), below it an absolute error of up to 2^-39 (2^-35)
// of the maximum. The error of a row's sums hardly shows it, but that of an output whose weight at a far
// larger element is zero; other splits' sums do not depend on that element. The codes
// enter the MFMA as exact fp16 integers (Q4_K's as subnormals q 2^-24), so products are exact; each
// block's sum C = sum q' x' comes out of the matrix core and one FMA with the block's fp32 scale
// folds it into the accumulator. Codes of Q8_0, Q4_0 and Q6_K carry their offset (q - 8, q - 32);
// Q4_K's min term is a 32 x 32 x 2 fp32 MFMA per stage over the block sums of x'.
//
// Structure (as gemm_tile.h, whose W units it loads): tile 32 TM rows of x x 128 rows of W per
// workgroup of 4 waves, two workgroups or more per CU, K in stages of two 32-blocks through LDS.
// Lane (r, h) supplies elements 8 h .. + 7 (MFMA q = 0) and 16 + 8 h .. + 7 (q = 1) of a block, so that
// an MFMA sums over one block: 4 MFMAs per block and 32 rows of x (q, hi / lo), one fold of 16 FMAs.
// A block's fold runs under the next block's MFMAs. split_x_kernel stores each 4 elements as 0, 2,
// 1, 3 (the order in which masking a dword of codes yields them) and, for the 4-bit quants, elements
// 16..31 of a block times 1/16 (their codes sit at bits 4..7).
// grid = (ceil(B / (32 TM)) * ceil(N / 128), S): S K splits of split_stages stages (a multiple of
// 4 when S > 1) to part[s][B][N], added by sum_windows_kernel. Requires K as gemm_tile.h.
#pragma once

#include "gemm_tile.h"

namespace j4q {
namespace gvt {

using gt::WUnit;
using gw::dma16;
using gw::dma4;
using gw::dma4s;
using gw::kOob;
using gw::lds_barrier;
using gw::load_order;
using gw::make_rsrc;
using gw::u32x2;
using gw::u32x4;
using gw::wait_vm_lgkm0;
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef _Float16 h2 __attribute__((ext_vector_type(2)));
typedef _Float16 h4 __attribute__((ext_vector_type(4)));
typedef _Float16 h8 __attribute__((ext_vector_type(8)));

// Columns [64 per s, 64 per (s + 1)) of row r of x [rows, K], r = blockIdx.x, s = blockIdx.y, as hi and lo
// fp16 in the layout above (lo `lo_off` halves after hi), 2^-e to unscale[s rows + r], and with sums
// the sums of x 2^e over every 32-block. K % 64 == 0, per <= 16: a thread per 4 elements. What bounds
// it is the memory latency, paid once: x stays in registers between the maximum and the conversion.
template <bool SIXTEENTH>
__global__ void __launch_bounds__(256)
split_x_kernel(const float *__restrict__ x, int K, int per, _Float16 *__restrict__ hi, int64_t lo_off, float *__restrict__ unscale,
               float *__restrict__ sums) {
    __shared__ float wmax[4];
    const int tid = (int)threadIdx.x, i = 16 * per * (int)blockIdx.y + tid;  // this thread's 4 elements
    const bool in = tid < 16 * per && i < K / 4;
    const f32x4 raw = in ? reinterpret_cast<const f32x4 *>(x + (int64_t)blockIdx.x * K)[i] : f32x4{};
    float v = fmaxf(fmaxf(fabsf(raw.x), fabsf(raw.y)), fmaxf(fabsf(raw.z), fabsf(raw.w)));
#pragma unroll
    for (int o = 32; o > 0; o /= 2) v = fmaxf(v, __shfl_xor(v, o));
    if ((tid & 63) == 0) wmax[tid >> 6] = v;
    __syncthreads();
    v = fmaxf(fmaxf(wmax[0], wmax[1]), fmaxf(wmax[2], wmax[3]));
    int e = 0;
    if (v > 0.f && v <= 3.402823466e38f) {
        int E;
        (void)frexpf(v, &E);
        e = 15 - E;
        e = e < -126 ? -126 : (e > 127 ? 127 : e);
    }
    const float sx = ldexpf(1.0f, e);
    if (tid == 0) unscale[blockIdx.y * gridDim.x + blockIdx.x] = ldexpf(1.0f, -e);
    if (!in) return;
    const f32x4 a = raw * sx;
    const f32x4 b = SIXTEENTH && (i & 4) ? a * 0.0625f : a;
    const h4 h = __builtin_convertvector(f32x4{b.x, b.z, b.y, b.w}, h4);
    const f32x4 back = __builtin_convertvector(h, f32x4);
    const int64_t o = (int64_t)blockIdx.x * (K / 4) + i;
    reinterpret_cast<h4 *>(hi)[o] = h;
    reinterpret_cast<h4 *>(hi + lo_off)[o] = __builtin_convertvector(f32x4{b.x, b.z, b.y, b.w} - back, h4);
    if (sums) {  // the 8 lanes of a block (K % 32 == 0: all of them are here)
        float t = (a.x + a.y) + (a.z + a.w);
        t += __shfl_xor(t, 1);
        t += __shfl_xor(t, 2);
        t += __shfl_xor(t, 4);
        if ((i & 7) == 0) sums[o >> 3] = t;
    }
}

// ALL: a workgroup takes every K split in turn (grid.y = 1) and adds their sums in its registers, in the
// order and with the roundings of sum_windows_kernel, so results are the same bit for bit.
template <int FMT, int TM, bool ALL>
__global__ void __launch_bounds__(256, 2)
gemv_tile(QMat w, const uint16_t *__restrict__ xs, const float *__restrict__ unscale, const float *__restrict__ sums,
          const float *add, float *y, int B, int split_stages, float *__restrict__ part) {
    using U = WUnit<FMT, 4>;
    constexpr int BM = 32 * TM, BN = 128, QR = U::QR, WL = U::kLoads;
    constexpr bool MIN = FMT == Q4_K;                      // a min term
    constexpr int XL = 2 * TM + (MIN ? TM : 0);            // X loads per wave and stage
    constexpr int kX = 2 * BM * 128, kXs = kX + (MIN ? 4 * TM * 256 : 0);
    constexpr int GS = FMT == Q6_K ? 4 : 2;                // folds per stage (Q6_K: a scale per 16)
    // Which of hi (0) and lo (1) a block's sum starts with. The matrix core aligns C and the products
    // of one MFMA to the largest exponent and drops what lies below, so the small lo products go
    // first - except with Q4_K's subnormal codes, whose products count as 2^10 larger there than
    // they are (error against 64 bits at 61 x 4096 x 4096: lo first 3.3e-5, hi first 4.1e-6; Q4_0's
    // offset codes 1.4e-7).
    constexpr int kFirst = MIN ? 0 : 1;
    __shared__ __attribute__((aligned(1024))) uint8_t xs0[kXs], xs1[kXs];
    __shared__ __attribute__((aligned(1024))) uint8_t ws0[U::kBytes], ws1[U::kBytes];
    const int N = (int)w.rows, K = (int)w.cols;
    const int sbeg = ALL ? 0 : (int)blockIdx.y * split_stages, send = sbeg + split_stages, all = K / 64;
    const int ns = ALL || send > all ? all : send;  // stages [sbeg, ns)
    // each XCD takes a contiguous range of tiles, row tiles of x fastest: they share the W rows
    const int mt = (B + BM - 1) / BM, total = (int)gridDim.x;
    int tile = (int)blockIdx.x;
    if (total % 8 == 0) tile = (tile % 8) * (total / 8) + tile / 8;
    const int m0 = (tile % mt) * BM, n0 = (tile / mt) * BN;

    const int lane = (int)threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int r32 = lane & 31, h = lane >> 5;

    // X load j of this wave (hi, then the same rows of lo) fills rows 8 (4 j + wave) .. + 7; lane L
    // fills slot L % 8 of row 8 (4 j + wave) + L / 8, which holds chunk (L % 8) ^ ((row / 2) % 8).
    const uint32_t lo_off = (uint32_t)B * (uint32_t)K * 2u;
    const __amdgpu_buffer_rsrc_t xr = make_rsrc(xs, 2u * (uint64_t)lo_off);
    uint32_t xoff[TM];
#pragma unroll
    for (int j = 0; j < TM; j++) {
        const int row = 8 * (4 * j + wave) + (lane >> 3), c = (lane & 7) ^ ((row >> 1) & 7);
        xoff[j] = m0 + row < B ? (uint32_t)(m0 + row) * (uint32_t)K * 2u + (uint32_t)c * 16u : kOob;
    }
    // Block sums, a copy per wave: dword TM (2 (row % 32) + block of the stage) + row / 32.
    const __amdgpu_buffer_rsrc_t mr = make_rsrc(sums, MIN ? (uint64_t)B * (uint64_t)(K / 32) * 4u : 0);
    uint32_t moff[TM];
#pragma unroll
    for (int t = 0; t < TM; t++) {
        const int d = 64 * t + lane, row = m0 + 32 * (d % TM) + d / (2 * TM);
        moff[t] = row < B ? (uint32_t)row * (uint32_t)(K / 32) * 4u + (uint32_t)(d / TM & 1) * 4u : kOob;
    }
    const int nw = n0 + 32 * wave;  // this wave's first row of W
    const int nsb = K / 256;
    U unit;
    unit.init(w, nw, wave, lane);

    auto load_x = [&](int i, uint8_t *xb) __attribute__((always_inline)) {
        const bool live = i < ns;
        const uint32_t so = live ? (uint32_t)i * 128u : 0u;
#pragma unroll
        for (int j = 0; j < TM; j++) {
            dma16(xr, xb + (4 * j + wave) * 1024, live ? xoff[j] : kOob, so);
            dma16(xr, xb + BM * 128 + (4 * j + wave) * 1024, live ? xoff[j] : kOob, so + lo_off);
        }
        if constexpr (MIN) {
#pragma unroll
            for (int t = 0; t < TM; t++)
                dma4s(mr, xb + kX + (wave * TM + t) * 256, live ? moff[t] : kOob, live ? (uint32_t)i * 8u : 0u);
        }
    };
    auto load_w = [&](int u, uint8_t *wb) __attribute__((always_inline)) { unit.load(u, 2 * u < ns, wb); };

    // The stage's two blocks of row r32 of W as this lane uses them: 8 bytes of codes (Q8_0: of
    // each half), a dword of Q6_K's high bits, and the scale words.
    struct Raw {
        u32x2 q[2][FMT == Q8_0 ? 2 : 1];
        uint32_t hi[2];
        u32x4 s;
    };
    auto read_raw = [&](int j, const uint8_t *wb, Raw &o) __attribute__((always_inline)) {
        const int swz = U::swz(r32), e = j & 1;
        const uint8_t *const row = wb + (32 * wave + r32) * QR, *const slot = wb + U::kS + wave * U::kSlot;
#pragma unroll
        for (int c = 0; c < 2; c++) {
            const int blk = 2 * e + c;
#pragma unroll
            for (int k = 0; k < U::QL / 2; k++)
                o.q[c][k] = *reinterpret_cast<const u32x2 *>(row + (((U::QL / 2 * blk + k) ^ swz) << 4) + 8 * h);
        }
        if constexpr (FMT == Q6_K) {
            const u32x4 v = *reinterpret_cast<const u32x4 *>(wb + U::kH + (32 * wave + r32) * 32 + e * 16);
            o.hi[0] = h ? v[1] : v[0];
            o.hi[1] = h ? v[3] : v[2];
        }
        if constexpr (FMT == Q4_K) {
            o.s = *reinterpret_cast<const u32x4 *>(slot + r32 * 16);
        } else {
            o.s[0] = *reinterpret_cast<const uint32_t *>(slot + r32 * 8 + 4 * e);
            if constexpr (FMT == Q6_K) o.s[1] = *reinterpret_cast<const uint32_t *>(slot + 256 + r32 * 4);
        }
    };
    // Scale of fold g of stage j (block g; Q6_K: group g of the stage's four), and Q4_K's min of
    // block h.
    auto scale_of = [&](int j, int g, const Raw &raw) __attribute__((always_inline)) -> float {
        if constexpr (FMT == Q8_0 || FMT == Q4_0) {
            return half_bits_to_float(g ? raw.s[0] >> 16 : raw.s[0] & 0xFFFFu);
        } else if constexpr (FMT == Q4_K) {
            const int jsb = 2 * (j & 3) + g;
            const uint32_t sc = __builtin_amdgcn_ubfe(raw.s[1], 4 * jsb, 4) | (__builtin_amdgcn_ubfe(raw.s[3], 2 * jsb, 2) << 4);
            return half_bits_to_float(raw.s[0] & 0xFFFFu) * (float)sc * gt::kTwo24;
        } else {
            const uint32_t odd = ((uint32_t)(nw + r32) * (uint32_t)nsb + (uint32_t)(j >> 2)) & 1u;
            const float d = half_bits_to_float(odd ? raw.s[1] >> 16 : raw.s[1] & 0xFFFFu);
            return d * (float)(int8_t)(raw.s[0] >> (8 * g));
        }
    };
    auto min_of = [&](int j, const Raw &raw) __attribute__((always_inline)) -> float {
        const int jsb = 2 * (j & 3) + h;
        const uint32_t mn = __builtin_amdgcn_ubfe(raw.s[2], 4 * jsb, 4) | (__builtin_amdgcn_ubfe(raw.s[3], 16 + 2 * jsb, 2) << 4);
        return half_bits_to_float(raw.s[0] >> 16) * (float)mn;
    };
    // Operand q of block c: exact fp16 codes.
    auto operand = [&](const Raw &raw, int c, int q) __attribute__((always_inline)) -> h8 {
        u32x4 r;
#pragma unroll
        for (int k = 0; k < 2; k++) {
            uint32_t even, odd;
            _Float16 off;
            if constexpr (FMT == Q8_0) {
                const uint32_t v = raw.q[c][q][k] ^ 0x80808080u;
                even = (v & 0x00FF00FFu) | 0x64006400u;
                odd = ((v >> 8) & 0x00FF00FFu) | 0x64006400u;
                off = (_Float16)-1152.0f;
            } else {
                const uint32_t v = raw.q[c][0][k], mask = q ? 0x00F000F0u : 0x000F000Fu;
                even = v & mask;
                odd = (v >> 8) & mask;
                if constexpr (FMT == Q6_K) {
                    const uint32_t hw = k ? __builtin_amdgcn_alignbit(raw.hi[c], raw.hi[c], 8) : raw.hi[c];
                    const uint32_t hm = q ? 0x03000300u : 0x00300030u;
                    even |= hw & hm;
                    odd |= (hw >> 2) & hm;
                }
                if constexpr (FMT != Q4_K) {
                    even |= 0x64006400u;
                    odd |= 0x64006400u;
                }
                off = (_Float16)(FMT == Q4_0 ? (q ? -1152.0f : -1032.0f) : (q ? -1536.0f : -1056.0f));
            }
            if constexpr (FMT != Q4_K) {
                even = __builtin_bit_cast(uint32_t, __builtin_bit_cast(h2, even) + h2{off, off});
                odd = __builtin_bit_cast(uint32_t, __builtin_bit_cast(h2, odd) + h2{off, off});
            }
            r[2 * k] = even;
            r[2 * k + 1] = odd;
        }
        return __builtin_bit_cast(h8, r);
    };

    f32x16 acc[TM], corr[MIN ? TM : 1], sum[2][TM];  // sum: the block sums of two folds in turn
    float fs[2] = {0.f, 0.f};                        // ... and their scales
#pragma unroll
    for (int t = 0; t < TM; t++) acc[t] = sum[1][t] = f32x16{};
    if constexpr (MIN) {
#pragma unroll
        for (int t = 0; t < TM; t++) corr[t] = f32x16{};
    }
    const int aoff = r32 * 128, asw = (r32 >> 1) & 7;
    auto read_a = [&](const uint8_t *xb, int c, int q, h8 (&a)[2][TM]) __attribute__((always_inline)) {
#pragma unroll
        for (int l = 0; l < 2; l++)
#pragma unroll
            for (int t = 0; t < TM; t++)
                a[l][t] = *reinterpret_cast<const h8 *>(xb + (l * BM + 32 * t) * 128 + aoff + (((4 * c + 2 * q + h) ^ asw) << 4));
    };
    auto fold = [&](int k) __attribute__((always_inline)) {
#pragma unroll
        for (int t = 0; t < TM; t++)
#pragma unroll
            for (int v = 0; v < 16; v++) acc[t][v] = __builtin_fmaf(fs[k], sum[k][t][v], acc[t][v]);
    };
    Raw raw[2];  // the blocks of the current stage and of the next one
    // Stage number S of the period, buffers and waits as in gemm_tile.h.
    auto stage = [&](auto S_, int i) __attribute__((always_inline)) {
        constexpr int S = decltype(S_)::value, cur = S & 1;
        uint8_t *const xb = cur ? xs1 : xs0, *const xn = cur ? xs0 : xs1;
        constexpr int ur = (S + 1) / 2 % 2, un = (S + 3) / 2 % 2;
        uint8_t *const wc = ur ? ws1 : ws0, *const wn = un ? ws1 : ws0;
        wait_vm_lgkm0<S % 2 == 0 ? WL : 0>();
        lds_barrier();
        h8 a[4][2][TM], b[4];
        read_a(xb, 0, 0, a[0]);
        read_raw(i + 1, wc, raw[cur ^ 1]);
        load_x(i + 1, xn);
        load_order();  // X first: the wait at an even stage leaves the newest unit of W outstanding
        if constexpr (S % 2 == 1) load_w((i + 3) / 2, wn);
        __builtin_amdgcn_sched_barrier(0);  // issue the loads first
#pragma unroll
        for (int p = 0; p < 4; p++) {  // block p / 2, operand p % 2
            const int c = p >> 1, q = p & 1, g = GS == 4 ? p : c, k = g & 1;
            if (p < 3) read_a(xb, (p + 1) >> 1, (p + 1) & 1, a[p + 1]);
            b[p] = operand(raw[cur], c, q);
            const bool first = GS == 4 || q == 0, last = GS == 4 || q == 1;
            if (first) fs[k] = scale_of(i, g, raw[cur]);
#pragma unroll
            for (int t = 0; t < TM; t++)
                sum[k][t] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a[p][kFirst][t], b[p], first ? f32x16{} : sum[k][t], 0, 0, 0);
#pragma unroll
            for (int l = GS == 4 ? p : 2 * c; last && l <= p; l++)
#pragma unroll
                for (int t = 0; t < TM; t++)
                    sum[k][t] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a[l][!kFirst][t], b[l], sum[k][t], 0, 0, 0);
            if (first) fold(k ^ 1);  // the fold before, under these MFMAs
            if (MIN && p == 1) {
                const float mn = min_of(i, raw[cur]);
                typedef float fv __attribute__((ext_vector_type(TM)));
                const fv sx = reinterpret_cast<const fv *>(xb + kX + wave * TM * 256)[2 * r32 + h];
#pragma unroll
                for (int t = 0; t < TM; t++) corr[t] = __builtin_amdgcn_mfma_f32_32x32x2f32(sx[t], mn, corr[t], 0, 0, 0);
            }
        }
    };

    // The sum of split s of element v of tile t (row 32 t + 8 (v / 4) + 4 h + v % 4 of x), unscaled.
    auto unscaled = [&](int s, int t, int v) __attribute__((always_inline)) -> float {
        // both halves' scales by uniform loads, which do not wait for the loads into LDS
        const int row = m0 + 32 * t + 8 * (v >> 2) + (v & 3), last = B - 1;
        const float *const u = unscale + (int64_t)s * B;
        const float u0 = u[row < last ? row : last], u1 = u[row + 4 < last ? row + 4 : last];
        float r = acc[t][v];
        if constexpr (MIN) r -= corr[t][v];
        return r * (h ? u1 : u0);
    };
    f32x16 run[ALL ? TM : 1];
    int split = 0, left = split_stages;  // ALL: the current split, and its stages still to come
    if constexpr (ALL) {
#pragma unroll
        for (int t = 0; t < TM; t++)
#pragma unroll
            for (int v = 0; v < 16; v++) run[t][v] = -0.f;
    }
    auto flush = [&]() __attribute__((always_inline)) {
        fold(1);
        fs[1] = 0.f;
#pragma unroll
        for (int t = 0; t < TM; t++) {
#pragma unroll
            for (int v = 0; v < 16; v++) run[t][v] += unscaled(split, t, v);
            acc[t] = sum[1][t] = f32x16{};
            if constexpr (MIN) corr[t] = f32x16{};
        }
        split++;
        left = split_stages;
    };

    load_w(sbeg / 2, ws0);
    load_order();
    load_x(sbeg, xs0);
    load_order();
    load_w(sbeg / 2 + 1, ws1);
    wait_vm_lgkm0<XL + WL>();
    asm volatile("" ::: "memory");
    read_raw(sbeg, ws0, raw[0]);
#define J4Q_STAGE(S) stage(std::integral_constant<int, S>{}, i + S);
    int i = sbeg;
    for (; i + 4 <= ns; i += 4) {
        J4Q_STAGE(0) J4Q_STAGE(1) J4Q_STAGE(2) J4Q_STAGE(3)
        if constexpr (ALL) {
            left -= 4;
            if (left == 0) flush();
        }
    }
    if constexpr (FMT == Q8_0 || FMT == Q4_0) {
        if (i < ns) {
            J4Q_STAGE(0)
            if (i + 1 < ns) {
                J4Q_STAGE(1)
                if (i + 2 < ns) J4Q_STAGE(2)
            }
        }
    }
#undef J4Q_STAGE
    if constexpr (ALL) {
        if (split * split_stages < all) flush();
    } else {
        fold(1);  // GS is even: the last fold of a stage is its number 1
    }
    __builtin_amdgcn_s_waitcnt(0);  // no LDS load outlives the workgroup

    float *const out = part ? part + (int64_t)blockIdx.y * B * N : y;
    const int col = nw + r32;
    if (col >= N) return;
#pragma unroll
    for (int t = 0; t < TM; t++)
#pragma unroll
        for (int v = 0; v < 16; v++) {
            const int row = m0 + 32 * t + 8 * (v >> 2) + 4 * h + (v & 3);
            if (row < B) {
                const float r = ALL ? run[t][v] : unscaled((int)blockIdx.y, t, v);
                const int64_t o = (int64_t)row * N + col;
                out[o] = !part && add ? r + add[o] : r;
            }
        }
}

}  // namespace gvt
}  // namespace j4q
