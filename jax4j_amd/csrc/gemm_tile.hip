// Prefill GEMM, bf16 variant: picks the tile and the K split of the LDS-tiled kernel
// (gemm_tile.h) for the shape, and the kernels of gemm_wide.h where they are faster (Q8_0).
#include "j4q_common.h"
#include "gemm_tile.h"

namespace j4q {
namespace {

// The tiles, and what one stage of one workgroup takes in us on MI355X: few workgroups, each
// alone on its CU (few); one on every CU (all: the chip's clock and its memory are shared); and as
// a share of the CU's time when every CU runs several, one after another or side by side (shared).
// From sweeps of Q4_K, Q4_0 and Q8_0 over N = 700 .. 14336, K = 1024 .. 14336, M = 8 .. 2048.
struct Cost {
    int waves, tm;
    float few, all, shared;
};
constexpr Cost kCost[] = {{4, 1, .33f, .38f, .26f}, {4, 2, .38f, .43f, .34f}, {4, 3, .45f, .50f, .43f},
                          {4, 4, .47f, .57f, .51f}, {4, 5, .58f, .68f, .63f}, {8, 4, .62f, 1.02f, 1.0f},
                          {8, 8, 1.2f, 1.75f, 1.75f}};
// Workgroups of K groups of two waves (64 columns) or four, one per CU: what the launch, the prologue and the sums
// of the groups take, and a stage of all groups, as above; Q6_K's decoding comes on top. Fitted to 162
// sizes (N = 350 .. 15000, K = 512 .. 14336, M = 4 .. 1500), times 1.09, by which the figures above are too
// large at those sizes. us a call of the 64-column kernel of 8 waves that
// was here before, of the shapes above, and of these: Q4_K 950 x 1040 x 2560 16.9, 17.2, 12.4; 17 x 2267 x 768
// 5.4, 6.6, 5.3; 24 x 14336 x 4096 18.2, 15.7, 12.6; 128 x 4096 x 2048 23.0, 11.7, 8.2; Q6_K 950 x 1040 x 2560
// 16.7, 19.2, 14.0.
struct Group {
    int waves, tm, groups;
    float base, few, all, q6_few, q6_all;
};
constexpr Group kGroups[] = {{2, 1, 2, 2.98f, .355f, .428f, .059f, .081f}, {2, 2, 2, 3.44f, .412f, .492f, .081f, .102f},
                             {2, 1, 4, 3.20f, .565f, .700f, .155f, .200f}, {2, 2, 4, 3.72f, .641f, .792f, .164f, .223f},
                             {2, 3, 4, 4.13f, .762f, 1.035f, .158f, .164f}, {4, 2, 2, 3.80f, .590f, .700f, .130f, .170f}};
constexpr int kCus = 256;  // of an MI355X; a constant, so that results do not depend on the device

// The fastest shape by a model of the launch: the stages that the busiest CU runs (Q6_K's take
// longer to decode, Q8_0's to load), a launch's fixed 3 us, and with K split the sum kernel: 2 us,
// a quarter per split, and its traffic (the partial products written and read, the result written)
// at 5.5 MB/us. Over the sweeps (38 sizes) its choice takes 1.2 % longer than the best of all
// shapes on average, 11 % at worst (with the groups of kGroups, 162 sizes: 0.5 %). Splits are whole
// multiples of four stages, and their workspace is at most 32 MiB; a Q8_0 call takes no workspace, so
// it does not split.
GemmShape pick(int id, const QMat &w, int64_t m, bool split, float *us_out) {
    const int64_t n = w.rows, ns = w.cols / 64;
    const float alone_add = id == Q6_K ? .12f : id == Q8_0 ? .05f : 0.f, shared_add = id == Q6_K ? .09f : id == Q8_0 ? .05f : 0.f;
    GemmShape best;
    float best_us = 0.f;
    for (const Cost &c : kCost) {
        const int64_t tiles = ((m + 32 * c.tm - 1) / (32 * c.tm)) * ((n + 32 * c.waves - 1) / (32 * c.waves));
        int64_t last = 0;
        for (int64_t want = 1; want <= (split && id != Q8_0 ? 16 : 1); want++) {
            const int64_t per = want == 1 ? ns : ((ns + want - 1) / want + 3) / 4 * 4, s = (ns + per - 1) / per;
            if (s == last || (s > 1 && s * m * n * 4 > (32ll << 20))) continue;
            last = s;
            const int64_t groups = tiles * s, rounds = (groups + kCus - 1) / kCus;
            float us = rounds <= 1 ? c.few + (c.all - c.few) * (float)groups / kCus + alone_add : (float)rounds * (c.shared + shared_add);
            us = us * (float)per + 3.0f;
            if (s > 1) us += 2.0f + .25f * (float)s + (float)((2 * s + 1) * m * n * 4) / 5.5e6f;
            if (!best.tm || us < best_us) {
                best_us = us;
                best = GemmShape{c.waves, c.tm, (int)s, (int)per, 1, 0};
            }
        }
    }
    // At most a tile per CU without the sum kernel: K in groups of waves of a workgroup (kGroups).
    if (id != Q8_0 && ns % 4 == 0) {
        for (const Group &c : kGroups) {
            const int64_t tiles = ((m + 32 * c.tm - 1) / (32 * c.tm)) * ((n + 32 * c.waves - 1) / (32 * c.waves)), per = ((ns + c.groups - 1) / c.groups + 3) / 4 * 4;
            if (tiles > kCus) continue;
            const float few = c.few + (id == Q6_K ? c.q6_few : 0.f), all = c.all + (id == Q6_K ? c.q6_all : 0.f);
            const float us = (few + (all - few) * (float)tiles / kCus) * (float)per + c.base;
            if (us < best_us) {
                best_us = us;
                best = GemmShape{c.waves, c.tm, 1, (int)per, c.groups, 0};
            }
        }
    }
    *us_out = best_us;
    return best;
}

// y[i] = ((part[0][i] + part[1][i]) + ...) for i < n: the K splits' partial products added
// in split order (deterministic). A thread takes four consecutive elements when n % 4 == 0
// (every split then starts 16-byte aligned; y is), else one.
__global__ void __launch_bounds__(256)
sum_splits_kernel(const float *__restrict__ part, int splits, int64_t n, float *__restrict__ y) {
    typedef float f32x4 __attribute__((ext_vector_type(4)));
    const int64_t stride = (int64_t)gridDim.x * 256;
    if (n % 4 == 0) {
        for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n / 4; i += stride) {
            f32x4 v = reinterpret_cast<const f32x4 *>(part)[i];
            for (int r = 1; r < splits; r++) v += reinterpret_cast<const f32x4 *>(part + (int64_t)r * n)[i];
            reinterpret_cast<f32x4 *>(y)[i] = v;
        }
        return;
    }
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += stride) {
        float v = part[i];
        for (int r = 1; r < splits; r++) v += part[(int64_t)r * n + i];
        y[i] = v;
    }
}

template <int FMT>
hipError_t launch_fmt(const QMat &w, const uint16_t *x, float *y, int64_t m, const GemmShape &t, const Workspace &ws, hipStream_t s) {
    const int64_t tiles = ((m + 32 * t.tm - 1) / (32 * t.tm)) * ((w.rows + 32 * t.waves - 1) / (32 * t.waves));
    if (tiles > 0x7fffffff || ws.bytes < t.workspace) return hipErrorInvalidValue;
    const dim3 grid((unsigned)tiles, (unsigned)t.splits);
    float *const part = t.splits > 1 ? ws.ptr : nullptr;
    bool launched = false;
#define J4Q_TILE(WV, TM)                                                                              \
    if (t.waves == WV && t.tm == TM && t.groups == 1) {                                               \
        gt::gemm_tile<FMT, WV, TM><<<grid, 64 * WV, 0, s>>>(w, x, y, (int)m, t.split_stages, part);   \
        launched = true;                                                                              \
    }
    J4Q_TILE(4, 1)
    J4Q_TILE(4, 2)
    J4Q_TILE(4, 3)
    J4Q_TILE(4, 4)
    J4Q_TILE(4, 5)
    J4Q_TILE(8, 4)
    J4Q_TILE(8, 8)
#undef J4Q_TILE
    if constexpr (FMT != Q8_0) {
#define J4Q_GROUPS(WV, TM, KG)                                                                              \
    if (t.waves == WV && t.tm == TM && t.groups == KG) {                                                    \
        gt::gemm_tile<FMT, WV, TM, KG><<<grid, 64 * WV * KG, 0, s>>>(w, x, y, (int)m, t.split_stages, part); \
        launched = true;                                                                                    \
    }
        J4Q_GROUPS(2, 1, 2)
        J4Q_GROUPS(2, 2, 2)
        J4Q_GROUPS(2, 1, 4)
        J4Q_GROUPS(2, 2, 4)
        J4Q_GROUPS(2, 3, 4)
        J4Q_GROUPS(4, 2, 2)
#undef J4Q_GROUPS
    }
    if (!launched) return hipErrorInvalidValue;
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess || t.splits == 1) return e;
    const int64_t n = m * w.rows;
    const int64_t blocks = ((n % 4 == 0 ? n / 4 : n) + 255) / 256;
    return launch_with_event(sum_splits_kernel, dim3((unsigned)(blocks < 2048 ? blocks : 2048)), dim3(256), s, ws.done, ws.ptr, t.splits, n, y);
}

}  // namespace

bool gemm_bf16_supported(int id, int64_t cols) {
    switch (id) {
    case Q8_0: return cols % 32 == 0;
    case Q4_0: return cols % 128 == 0;
    case Q4_K:
    case Q6_K: return cols % 256 == 0;
    default: return false;
    }
}

GemmShape gemm_bf16_shape(int id, const QMat &w, int64_t m, bool split) {
    if (!gemm_bf16_supported(id, w.cols) || m <= 0 || w.rows <= 0 || (id == Q8_0 && w.cols % 64 != 0)) return GemmShape{};
    float us = 0.f;
    GemmShape t = pick(id, w, m, split, &us);
    if (id == Q8_0 && choose_q8_bf16(w, m).us <= 1.05f * us) return GemmShape{};
    t.workspace = t.splits > 1 ? (uint64_t)t.splits * (uint64_t)m * (uint64_t)w.rows * 4u : 0;
    return t;
}

hipError_t launch_gemm_bf16(int id, const QMat &w, const uint16_t *x, float *y, int64_t m, const GemmShape &t,
                            const Workspace &ws, hipStream_t s) {
    if (m <= 0 || w.rows <= 0) return hipSuccess;
    if (id == Q8_0 && !t.tm) return launch_gemm_q8_bf16(w, x, y, m, s);
    if (!gemm_bf16_supported(id, w.cols) || (uint64_t)m * (uint64_t)w.cols * 2u > 0x7fffffffull ||
        (uint64_t)w.rows * (uint64_t)w.cols / (id == Q8_0 ? 1u : 2u) > 0x7fffffffull)
        return hipErrorInvalidValue;
    switch (id) {
    case Q8_0: return launch_fmt<Q8_0>(w, x, y, m, t, ws, s);
    case Q4_0: return launch_fmt<Q4_0>(w, x, y, m, t, ws, s);
    case Q4_K: return launch_fmt<Q4_K>(w, x, y, m, t, ws, s);
    case Q6_K: return launch_fmt<Q6_K>(w, x, y, m, t, ws, s);
    default: return hipErrorInvalidValue;
    }
}

}  // namespace j4q
