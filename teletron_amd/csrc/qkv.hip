// The QK-norm call site as one kernel per direction: the fused projection mixed [B, S, H, 3 * C] holds q, k and v
// of a head side by side (teletron/models/dit/dit_attention.py:149-214); q and k leave RMS-normalised over C as
// contiguous [B, H, S, C] tensors, optionally rotated, and backward assembles the projection's gradient in place.
//
//   forward   q, k read from mixed (512 contiguous bytes per head and token at C = 128 two-byte), both written
//   backward  the gradients of q, k, v and the projection's q, k read; d mixed written whole (768 contiguous bytes);
//             dweight of both norms as per-workgroup partial sums, one column reducer for the two
//
// Arithmetic and rounding points are those of rmsnorm.hip; a head's row is owned by LANES lanes (8, 16, 32 or 64),
// 16 bytes per lane, 64 / LANES consecutive tokens of one head per wavefront.  The row statistic is formed again in
// backward from the row it has to read anyway (the same operations, hence the same bits), so nothing but the
// projection itself is kept between the passes.
#include "norm_device.h"
#include "norm_host.h"
#include "rope_device.h"

// What bounds both kernels is the memory system under a transposing mix of reads and writes: at [1, 29700, 24, 3 * 128]
// two-byte forward moves its 730 MB in 124 us (5.9 TB/s) and backward its 1.46 GB in 258 us (5.7), where plain streams
// reach 6.2-6.3, and that only if what is WRITTEN at a time is contiguous: forward therefore runs its workgroups along the
// tokens of one head at a time (one-shot), backward along the heads of one token group at a time.  Measured there, against
// one kernel per tensor (two forward; two backward, one copy of the value gradient, two reducers): forward 124 against 150
// us, with tables 137 against 151; backward 258 against 297, with tables 262 against 303.
//
// Forward: wavefronts of a workgroup along the tokens (1 << LOG2 of the four; the others along heads and samples) and heads
// per wavefront (HR).  With tables, two heads of one token group share the 1 KiB of table per token (one head 143 us, three
// 136, four 149; two heads with two / four wavefronts along the tokens 139 / 155).  Without tables four consecutive token
// groups of one head (tokens along two / one wavefronts: 127 us) or of two, whichever keeps the chip busier: two heads per
// wavefront double what a wavefront has in flight, which wins once every compute unit has four workgroups of one head to
// choose from (1500 x 24 x 128 bf16 10.0 -> 9.3 us, 3000 x 16 x 64 6.9 -> 6.2; below, half the wavefronts is what counts:
// 256 x 24 x 128 3.4 / 3.6) and loses on long streams of whole rows (6000 x 24 x 128 29.1 either way, 29700 128 / 131).
// Rows that leave lanes empty keep gaining (5208 x 12 x 80 12.1 -> 10.9, 30000 53.3 -> 50.3, 52083 90.8 -> 90.1).
// Where there are fewer token groups, or fewer heads and samples, than the split asks for, the launch moves wavefronts to
// the other side instead of leaving them idle (4096 x 1 token x 24 heads x 128: 77 us with three of four idle, 43 now; one
// rotated head of 300000 tokens 216 / 106).
#ifndef TTN_QKV_FWD_TOKEN_WAVES_LOG2
#define TTN_QKV_FWD_TOKEN_WAVES_LOG2 (ROPE ? 0 : 2)
#endif
#ifndef TTN_QKV_FWD_TWO_HEADS_FROM
#define TTN_QKV_FWD_TWO_HEADS_FROM 4  // workgroups of one head per compute unit
#endif
#ifndef TTN_QKV_FWD_TWO_HEADS_BELOW
#define TTN_QKV_FWD_TWO_HEADS_BELOW (FULL ? 32 : 1 << 20)
#endif
// Forward, tokens a multiple of 4 KiB apart in the projection: the pieces of one head then lie at one offset of the
// memory's 4 KiB interleave, and a launch that walks all tokens of one head before the next reads from a part of the
// channels only.  There it takes the heads of 2048 tokens before the next 2048 (bf16, 16 x 128: 24414 tokens 85.9 -> 74.1 us,
// 8000 27.7 -> 25.9; 32 x 64 86.2 -> 76.7; fp32 16 x 64 84.0 -> 75.1; 1024 or 4096 tokens at a time within 3 %).  Other strides
// are better off with the longest contiguous writes (24 x 128 128 us, 133 in pieces), and so are fewer than three such
// pieces (4000 tokens 15.2 / 15.6) and rotated four-byte rows, whose two heads are 2.5 KiB in one run (91.9 / 94.3).
constexpr int64_t kInterleave = 4096, kTileTokens = 2048;
// Forward with tables: dynamic LDS the kernel does not touch, as a throttle on a long grid whose workgroups are all busy:
// five to a compute unit stream better than eight (24 heads, 29700 tokens 142.5 -> 135.7 us, 7681 39.2 -> 38.1, 4000 22.3 ->
// 21.8; four the same, six 138).  A short grid wants every wavefront (2500 tokens 15.5 / 15.9), and so does one whose heads leave
// wavefronts of a workgroup idle (12 heads, 30000 tokens 74.7 / 77.9).
#ifndef TTN_QKV_FWD_ROPE_LDS
#define TTN_QKV_FWD_ROPE_LDS 32768
#endif
#ifndef TTN_QKV_FWD_ROPE_LDS_FROM
#define TTN_QKV_FWD_ROPE_LDS_FROM 10  // workgroups per compute unit
#endif
// Backward: persistent, for the column sums.  Two workgroups per compute unit keep 10 MB requested (three: 271, four
// 278 us; one with the next step's rows requested ahead 263-272).  The wavefront waits for its rows, works and
// writes; the other wavefront of its SIMD overlaps it (a second row buffer: 266-269 us).
#ifndef TTN_QKV_BWD_BLOCKS_PER_CU
#define TTN_QKV_BWD_BLOCKS_PER_CU 2
#endif
// From this many steps per wavefront on, a step's rows are requested only when the stores of the step before have left the
// wavefront: its reads and writes then take turns at the memory, as in the dense backward kernels (24 heads, 29700 tokens
// 265 -> 251 us, 50000 451 -> 416, with tables 266 -> 259; 48828 x 16 x 64 151 -> 142; 39062 x 16 x 80 185 -> 182).  Shorter walks
// are latency and lose the overlap (5000 tokens 49.5 / 49.9, 3000 32.6 / 33.4; 8000 73.7 / 73.3).
#ifndef TTN_QKV_BWD_DRAIN_FROM
#define TTN_QKV_BWD_DRAIN_FROM 24
#endif
// Consecutive steps of a wavefront that are neighbouring heads: with tables the rows it has fetched then serve more than
// one head (runs of one 271, two 260, three 261, six 267 us); without tables runs only spread the writes (two: 261).
#ifndef TTN_QKV_BWD_RUN
#define TTN_QKV_BWD_RUN (Rope::kOn ? 2 : 1)
#endif

namespace ttn {

constexpr int kLoadNt = 2;  // cache policy of the row loads: non-temporal
constexpr int kRowWavesLog2 = 2;
static_assert(1 << kRowWavesLog2 == kRowWaves);

// FULL: the row fills its LANES lanes, so its length is known at compile time.
template <typename T, int LANES_, bool FULL>
struct HeadGeom {
    static constexpr int VEC = Elem<T>::VEC;
    static constexpr int LANES = LANES_;
    static constexpr int CHUNKS = 1;
    static constexpr int RPW = kWaveSize / LANES;
    static __device__ __forceinline__ int cols(int c) { return FULL ? VEC * LANES : c; }
};

template <typename T, int LANES>
__device__ __forceinline__ float row_rstd(const u32x4 &x, int C, float eps) {
    float v[Elem<T>::VEC];
    Elem<T>::unpack(x, v);
    float ss = 0.0f;
#pragma unroll
    for (int j = 0; j < Elem<T>::VEC; ++j) ss = fmaf(v[j], v[j], ss);
    ss = group_sum<LANES>(ss);
    return 1.0f / sqrtf(ss / (float)C + eps);
}

template <typename T, int LANES, bool FULL, typename Rope, int HR>
__global__ __launch_bounds__(kRowThreads) void qkv_fwd_kernel(T *__restrict__ q, T *__restrict__ k,
                                                              const T *__restrict__ mixed, const T *__restrict__ wq,
                                                              const T *__restrict__ wk, const Rope rope, int64_t S, int H,
                                                              uint32_t head_groups, uint32_t outer, int tw_log2, int c_arg,
                                                              float eps) {
    using G = HeadGeom<T, LANES, FULL>;
    using E = Elem<T>;
    constexpr bool ROPE = Rope::kOn;
    constexpr int VEC = G::VEC, RPW = G::RPW;
    const int C = G::cols(c_arg);
    const int lane = threadIdx.x & 63;
    const int sub = lane / LANES;
    const int l = lane % LANES;
    const int wave = wave_id_in_block();
    const bool in = FULL || l * VEC < C;
    // a wavefront's place among the token groups and among the (sample, group of HR heads) pairs
    const int token_wave = wave & ((1 << tw_log2) - 1), outer_wave = wave >> tw_log2, outer_waves = kRowWaves >> tw_log2;
    const int64_t s0 = ((((int64_t)blockIdx.z * gridDim.x + blockIdx.x) << tw_log2) + token_wave) * RPW;
    const bool ok = in && s0 + sub < S;
    const uint32_t from = (uint32_t)sub * (uint32_t)(H * 3 * C * (int)sizeof(T)) + l * 16;
    const uint32_t to = (uint32_t)(sub * C * (int)sizeof(T)) + l * 16;
    const u32x4 zero{0, 0, 0, 0};

    for (uint32_t first = blockIdx.y * outer_waves; first < outer; first += gridDim.y * outer_waves) {
        // a wavefront past the last pair works along on zeros: leaving early slows the others of its workgroup (7681 tokens
        // x 12 heads with tables 21.0 instead of 20.4 us)
        const uint32_t y = first + outer_wave;
        const bool mine = y < outer;
        const int64_t b = y / head_groups;
        const int h0 = (int)(y % head_groups) * HR;
        const T *src = mixed + ((b * S + s0) * H + h0) * 3 * C;
        u32x4 xr[HR][2];
#pragma unroll
        for (int i = 0; i < HR; ++i) {
            const RowReader<kLoadNt> rq(src + i * 3 * C, from), rk(src + (i * 3 + 1) * C, from);
            const bool here = ok && mine && h0 + i < H;
            xr[i][0] = here ? rq.get(0) : zero;
            xr[i][1] = here ? rk.get(0) : zero;
        }
        RopeRows<ROPE, 1, VEC> rot;
        if constexpr (ROPE) rot.fetch(rope, ok, s0 + sub, C, l, LANES);
        u32x4 w[2];
        w[0] = in ? load16(reinterpret_cast<const u32x4 *>(wq) + l) : zero;
        w[1] = in ? load16(reinterpret_cast<const u32x4 *>(wk) + l) : zero;
#pragma unroll
        for (int i = 0; i < HR; ++i) {
            const int64_t row0 = (b * H + h0 + i) * S + s0;
#pragma unroll
            for (int t = 0; t < 2; ++t) {
                const float r = row_rstd<T, LANES>(xr[i][t], C, eps);
                float v[VEC], wv[VEC];
                E::unpack(xr[i][t], v);
                E::unpack(w[t], wv);
#pragma unroll
                for (int j = 0; j < VEC; ++j) v[j] *= r;
                E::round(v);  // y = the normalised row in the element type
#pragma unroll
                for (int j = 0; j < VEC; ++j) v[j] *= wv[j];
                if constexpr (ROPE) {
                    if (rot.on) {
                        E::round(v);  // the norm's output in the element type, which the rotation reads
                        rotate_pairs_forward<VEC>(v, rot.c[0], rot.s[0]);
                    }
                }
                const RowWriter<0> out((t ? k : q) + row0 * C, to);
                if (ok && mine && h0 + i < H) out.put(0, E::pack(v));
            }
        }
    }
}

// gq / gk / gv may be null (that output was not used): its slice of d mixed is zero, as is its dweight.
template <typename T, int LANES, bool FULL, typename Rope, bool DRAIN>
__global__ __launch_bounds__(kRowThreads) void qkv_bwd_kernel(
    T *__restrict__ dmixed, float *__restrict__ partial, const T *__restrict__ gq, const T *__restrict__ gk,
    const T *__restrict__ gv, const T *__restrict__ mixed, const T *__restrict__ wq, const T *__restrict__ wk,
    const Rope rope, int64_t S, uint32_t H, uint32_t token_groups, uint32_t units, int c_arg, float eps) {
    using G = HeadGeom<T, LANES, FULL>;
    using E = Elem<T>;
    constexpr int VEC = G::VEC, RPW = G::RPW;
    __shared__ __align__(16) float lds[kRowWaves][2][LANES * VEC];
    const int C = G::cols(c_arg);
    const int lane = threadIdx.x & 63;
    const int sub = lane / LANES;
    const int l = lane % LANES;
    const int wave = wave_id_in_block();
    const bool in = FULL || l * VEC < C;
    const uint32_t mixed_lane = (uint32_t)sub * (H * 3u * (uint32_t)C * (uint32_t)sizeof(T)) + l * 16;
    const uint32_t dense_lane = (uint32_t)(sub * C * (int)sizeof(T)) + l * 16;
    const u32x4 zero{0, 0, 0, 0};
    const uint32_t waves = gridDim.x * kRowWaves, me = blockIdx.x * kRowWaves + wave;
    const bool has[3] = {gq != nullptr, gk != nullptr, gv != nullptr};

    const u32x4 w[2] = {in ? load16(reinterpret_cast<const u32x4 *>(wq) + l) : zero,
                        in ? load16(reinterpret_cast<const u32x4 *>(wk) + l) : zero};
    float acc[2][VEC];
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int j = 0; j < VEC; ++j) acc[t][j] = 0.0f;

    // heads fastest, so that what the wavefronts of the chip write at a time is one contiguous region of d mixed
    constexpr uint32_t kRun = TTN_QKV_BWD_RUN;
    [[maybe_unused]] RopeRows<Rope::kOn, 1, VEC> rot;
    [[maybe_unused]] uint32_t rot_group = 0xffffffffu;
    const uint32_t runs = (units + kRun - 1) / kRun;
    const uint32_t steps = runs > me ? ((runs - me + waves - 1) / waves) * kRun : 0;
    for (uint32_t step = 0; step < steps; ++step) {
        const uint32_t u = (step / kRun * waves + me) * kRun + step % kRun;
        const uint32_t h = u % H, rest = u / H;
        const uint32_t tg = rest % token_groups;
        const int64_t b = rest / token_groups;
        const int64_t s0 = (int64_t)tg * RPW;
        const bool exists = s0 + sub < S && u < units;  // this lane's token
        const bool ok = in && exists;
        const int64_t at = ((b * S + s0) * H + h) * 3 * C;
        const int64_t dense = ((b * H + h) * S + s0) * C;
        u32x4 g[3], x[2];
        if constexpr (DRAIN) wait_memory_ops<0>();
        {
            const RowReader<kLoadNt> rgq(gq + dense, dense_lane), rgk(gk + dense, dense_lane), rgv(gv + dense, dense_lane);
            const RowReader<kLoadNt> rxq(mixed + at, mixed_lane), rxk(mixed + at + C, mixed_lane);
            g[0] = (ok && has[0]) ? rgq.get(0) : zero;
            g[1] = (ok && has[1]) ? rgk.get(0) : zero;
            x[0] = ok ? rxq.get(0) : zero;
            x[1] = ok ? rxk.get(0) : zero;
            g[2] = (ok && has[2]) ? rgv.get(0) : zero;
        }
        if constexpr (Rope::kOn) {
            if (tg != rot_group) rot.fetch(rope, in && s0 + sub < S, s0 + sub, C, l, LANES);
            rot_group = tg;
            // the gradients arrive rotated: back through the rotation first
            if (rot.on) {
#pragma unroll
                for (int t = 0; t < 2; ++t) {
                    float gvv[VEC];
                    E::unpack(g[t], gvv);
                    rotate_pairs_backward<E, VEC>(gvv, rot.c[0], rot.s[0]);
                    g[t] = E::pack(gvv);
                }
            }
        }
        u32x4 d[3] = {zero, zero, g[2]};
#pragma unroll
        for (int t = 0; t < 2; ++t) {
            if (!has[t]) continue;
            const u32x4 gy = packed_products<T>(g[t], w[t]);  // rnd(g * w)
            float dot = 0.0f;
            if constexpr (kHasDot2<T>) {
#pragma unroll
                for (int i = 0; i < 4; ++i) dot = dot2<T>(gy[i], x[t][i], dot);
            } else {
                float gyv[VEC], xv[VEC];
                E::unpack(gy, gyv);
                E::unpack(x[t], xv);
#pragma unroll
                for (int j = 0; j < VEC; ++j) dot = fmaf(gyv[j], xv[j], dot);
            }
            dot = group_sum<LANES>(dot);
            const float rstd = row_rstd<T, LANES>(x[t], C, eps);
            const float r = exists ? rstd : 0.0f;  // rows past the end must add nothing, whatever eps is
            const float coef = -((dot / (float)C) * r * r * r);
            float gyv[VEC], xv[VEC], o[VEC], y[VEC];
            E::unpack(gy, gyv);
            E::unpack(x[t], xv);
#pragma unroll
            for (int j = 0; j < VEC; ++j) {
                o[j] = fmaf(xv[j], coef, gyv[j] * r);
                y[j] = xv[j] * r;
            }
            d[t] = E::pack(o);
            add_columns<T>(acc[t], packed_products<T>(g[t], E::pack(y)));  // dw += rnd(g * rnd(y))
        }
        const RowWriter<0> wd[3] = {{dmixed + at, mixed_lane}, {dmixed + at + C, mixed_lane}, {dmixed + at + 2 * C, mixed_lane}};
        if (ok) {
#pragma unroll
            for (int t = 0; t < 3; ++t) wd[t].put(0, d[t]);
        }
    }

    // the workgroup's partial row: tokens of a wavefront folded, then wavefronts in order
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int j = 0; j < VEC; ++j) {
            const float v = fold_rows_of_wave<LANES>(acc[t][j]);
            if (sub == 0) lds[wave][t][l * VEC + j] = v;
        }
    __syncthreads();
    for (int i = threadIdx.x; i < 2 * C; i += kRowThreads) {
        const int t = i >= C, c = t ? i - C : i;
        partial[(int64_t)blockIdx.x * 2 * C + i] = ((lds[0][t][c] + lds[1][t][c]) + lds[2][t][c]) + lds[3][t][c];
    }
}

// ------------------------------------------------------------------ host side

static int head_lanes(int pieces) { return pieces <= 8 ? 8 : pieces <= 16 ? 16 : pieces <= 32 ? 32 : 64; }

static int qkv_pieces(int64_t cols, int dtype) { return (int)(cols / (16 / (int64_t)elem_bytes(dtype))); }

static int64_t qkv_bwd_blocks(int64_t units, int cus) {
    const int64_t want = (units + kRowWaves - 1) / kRowWaves, most = (int64_t)cus * TTN_QKV_BWD_BLOCKS_PER_CU;
    return want < most ? want : most;
}

struct QkvSizes {
    int64_t B, S, H, cols;
    int lanes;
    int64_t token_groups() const { return (S + kWaveSize / lanes - 1) / (kWaveSize / lanes); }
    int64_t units() const { return B * token_groups() * H; }
};

template <typename T, int LANES, bool FULL, typename Rope, int HR>
static void launch_qkv_fwd_heads(const QkvSizes &z, int cus, void *q, void *k, const void *mixed, const void *wq, const void *wk,
                                 const Rope &rope, float eps, hipStream_t stream) {
    constexpr bool ROPE = Rope::kOn;
    const int64_t head_groups = (z.H + HR - 1) / HR, outer = z.B * head_groups;
    int tw_log2 = TTN_QKV_FWD_TOKEN_WAVES_LOG2;  // no more wavefronts along the tokens than there are groups of them,
    while (tw_log2 > 0 && (1 << (tw_log2 - 1)) >= z.token_groups()) --tw_log2;
    // nor across them than there are groups of heads
    while (tw_log2 < kRowWavesLog2 && (kRowWaves >> (tw_log2 + 1)) >= outer) ++tw_log2;
    const int tw = 1 << tw_log2, outer_waves = kRowWaves >> tw_log2;
    const int64_t along = (z.token_groups() + tw - 1) / tw, across = (outer + outer_waves - 1) / outer_waves;
    // the grid is walked along the tokens of a layer, then across, then layer by layer
    int64_t layers = (along + kMostBlocks - 1) / kMostBlocks;
    const int64_t tiles = z.S / kTileTokens < 65535 ? z.S / kTileTokens : 65535;
    if (z.H * 3 * z.cols * (int64_t)sizeof(T) % kInterleave == 0 && !(ROPE && sizeof(T) == 4) && tiles >= 3 && tiles > layers)
        layers = tiles;
    const dim3 grid((unsigned)((along + layers - 1) / layers), (unsigned)(across < 65535 ? across : 65535), (unsigned)layers);
    const bool throttle = ROPE && outer % outer_waves == 0 && along * across >= (int64_t)cus * TTN_QKV_FWD_ROPE_LDS_FROM;
    RowKernelProfile prof(stream);
    qkv_fwd_kernel<T, LANES, FULL, Rope, HR><<<grid, dim3(kRowThreads), throttle ? TTN_QKV_FWD_ROPE_LDS : 0, stream>>>(
        (T *)q, (T *)k, (const T *)mixed, (const T *)wq, (const T *)wk, rope, z.S, (int)z.H, (uint32_t)head_groups, (uint32_t)outer,
        tw_log2, (int)z.cols, eps);
}

template <typename T, int LANES, bool FULL, typename Rope>
static void launch_qkv_fwd(const QkvSizes &z, int cus, void *q, void *k, const void *mixed, const void *wq, const void *wk,
                           const Rope &rope, float eps, hipStream_t stream) {
    const int64_t blocks = z.units() / kRowWaves;  // of one head per wavefront
    if (Rope::kOn || (z.H > 1 && blocks >= (int64_t)cus * TTN_QKV_FWD_TWO_HEADS_FROM &&
                      blocks < (int64_t)cus * (TTN_QKV_FWD_TWO_HEADS_BELOW)))
        launch_qkv_fwd_heads<T, LANES, FULL, Rope, 2>(z, cus, q, k, mixed, wq, wk, rope, eps, stream);
    else if constexpr (!Rope::kOn)
        launch_qkv_fwd_heads<T, LANES, FULL, Rope, 1>(z, cus, q, k, mixed, wq, wk, rope, eps, stream);
}

template <typename T, int LANES, bool FULL, typename Rope>
static void launch_qkv_bwd(const QkvSizes &z, int64_t blocks, void *dmixed, void *ws, const void *gq, const void *gk,
                           const void *gv, const void *mixed, const void *wq, const void *wk, const Rope &rope, float eps,
                           hipStream_t stream) {
    RowKernelProfile prof(stream);
    const bool drain = z.units() >= blocks * kRowWaves * TTN_QKV_BWD_DRAIN_FROM;
    const auto kernel = drain ? qkv_bwd_kernel<T, LANES, FULL, Rope, true> : qkv_bwd_kernel<T, LANES, FULL, Rope, false>;
    kernel<<<dim3((unsigned)blocks), dim3(kRowThreads), 0, stream>>>(
        (T *)dmixed, (float *)ws, (const T *)gq, (const T *)gk, (const T *)gv, (const T *)mixed, (const T *)wq,
        (const T *)wk, rope, z.S, (uint32_t)z.H, (uint32_t)z.token_groups(), (uint32_t)z.units(), (int)z.cols, eps);
}

static int check_qkv(const char *who, int64_t B, int64_t S, int64_t H, int64_t cols, int dtype, const float *cos,
                     const float *sin, int64_t rope_tokens, QkvSizes *z) {
    if (B < 0 || S < 0 || H < 0 || cols <= 0)
        return fail(TT_NORM_EINVAL, "%s: B=%lld S=%lld H=%lld cols=%lld", who, (long long)B, (long long)S, (long long)H,
                    (long long)cols);
    if (!tt_qkv_rmsnorm_supported(cols, dtype))
        return fail(TT_NORM_EUNSUPPORTED, "%s: cols=%lld dtype=%d (a head's row must be at most 64 whole 16-byte pieces)",
                    who, (long long)cols, dtype);
    if (rope_tokens < 0 || rope_tokens > S)
        return fail(TT_NORM_EINVAL, "%s: rope_tokens=%lld outside [0, S=%lld]", who, (long long)rope_tokens, (long long)S);
    if (rope_tokens > 0) {
        if (cols != 128) return fail(TT_NORM_EUNSUPPORTED, "%s: the rotation is built for cols 128 (the head dimension) only", who);
        if (!cos || !sin) return fail(TT_NORM_EINVAL, "%s: null cos/sin table", who);
        if (!aligned16(cos) || !aligned16(sin)) return fail(TT_NORM_EALIGN, "%s: cos/sin table not 16-byte aligned", who);
    }
    // a wavefront's tokens are addressed with 32-bit byte offsets from the first of them
    if (H * 3 * cols > kMaxRowStrideBytes / (int64_t)elem_bytes(dtype))
        return fail(TT_NORM_EINVAL, "%s: a token of the projection exceeds 256 MiB", who);
    *z = QkvSizes{B, S, H, cols, head_lanes(qkv_pieces(cols, dtype))};
    if (z->token_groups() > 0x7fffffffLL || z->units() > 0x7fffffffLL) return fail(TT_NORM_EINVAL, "%s: grid too large", who);
    return TT_NORM_OK;
}

static int check_qkv_ptrs(const char *who, std::initializer_list<const void *> ptrs) {
    for (const void *p : ptrs) {
        if (!p) return fail(TT_NORM_EINVAL, "%s: null pointer", who);
        if (!aligned16(p)) return fail(TT_NORM_EALIGN, "%s: pointer %p not 16-byte aligned", who, p);
    }
    return TT_NORM_OK;
}

}  // namespace ttn

using namespace ttn;

// CALL(T, LANES, FULL, Rope, rope) for the run-time (dtype, lanes, full row, rotation)
#define TTN_QKV_LANES(T, CALL)                                                                                    \
    do {                                                                                                          \
        constexpr int kHead = 128 / Elem<T>::VEC;                                                                 \
        if (rope.tokens > 0) { CALL(T, kHead, true, RopeTable, rope); }                                           \
        else if (z.lanes == 8) { if (full) { CALL(T, 8, true, NoRope, NoRope{}); } else { CALL(T, 8, false, NoRope, NoRope{}); } }    \
        else if (z.lanes == 16) { if (full) { CALL(T, 16, true, NoRope, NoRope{}); } else { CALL(T, 16, false, NoRope, NoRope{}); } } \
        else if (z.lanes == 32) { if (full) { CALL(T, 32, true, NoRope, NoRope{}); } else { CALL(T, 32, false, NoRope, NoRope{}); } } \
        else { if (full) { CALL(T, 64, true, NoRope, NoRope{}); } else { CALL(T, 64, false, NoRope, NoRope{}); } } \
    } while (0)
#define TTN_QKV_DISPATCH(CALL)                                      \
    do {                                                            \
        if (dtype == TT_NORM_BF16) TTN_QKV_LANES(bf16_t, CALL);     \
        else if (dtype == TT_NORM_F16) TTN_QKV_LANES(f16_t, CALL);  \
        else TTN_QKV_LANES(float, CALL);                            \
    } while (0)

extern "C" {

int tt_qkv_rmsnorm_supported(int64_t cols, int dtype) {
    return (tt_norm_supported(cols, dtype) && qkv_pieces(cols, dtype) <= kWaveSize) ? 1 : 0;
}

int tt_qkv_rmsnorm_forward(void *q, void *k, const void *mixed, const void *weight_q, const void *weight_k,
                           const float *cos, const float *sin, int64_t rope_tokens, int64_t B, int64_t S, int64_t H,
                           int64_t cols, double eps, int dtype, void *stream) {
    const char *who = "tt_qkv_rmsnorm_forward";
    QkvSizes z;
    int st = check_qkv(who, B, S, H, cols, dtype, cos, sin, rope_tokens, &z);
    if (st != TT_NORM_OK) return st;
    if (z.units() == 0) return TT_NORM_OK;
    st = check_qkv_ptrs(who, {q, k, mixed, weight_q, weight_k});
    if (st != TT_NORM_OK) return st;
    int known = TT_NORM_OK;
    int cus = current_device_cus(&known);
    if (known != TT_NORM_OK) cus = 256;  // chooses the split only; without a device the launch itself reports it
    const bool full = qkv_pieces(cols, dtype) == z.lanes;
    const RopeTable rope{cos, sin, rope_tokens};
#define CALL(T, L, F, R, r) launch_qkv_fwd<T, L, F, R>(z, cus, q, k, mixed, weight_q, weight_k, r, (float)eps, (hipStream_t)stream)
    TTN_QKV_DISPATCH(CALL);
#undef CALL
    return check_launch("qkv forward launch");
}

size_t tt_qkv_rmsnorm_backward_workspace_bytes(int64_t B, int64_t S, int64_t H, int64_t cols, int dtype) {
    if (B <= 0 || S <= 0 || H <= 0 || !tt_qkv_rmsnorm_supported(cols, dtype)) return 0;
    int st = TT_NORM_OK;
    const int cus = current_device_cus(&st);
    if (st != TT_NORM_OK) return 0;
    const QkvSizes z{B, S, H, cols, head_lanes(qkv_pieces(cols, dtype))};
    return (size_t)qkv_bwd_blocks(z.units(), cus) * 2 * cols * sizeof(float);
}

int tt_qkv_rmsnorm_backward(void *dmixed, void *dweight_q, void *dweight_k, const void *dq, const void *dk,
                            const void *dv, const void *mixed, const void *weight_q, const void *weight_k,
                            const float *cos, const float *sin, int64_t rope_tokens, int64_t B, int64_t S, int64_t H,
                            int64_t cols, double eps, int dtype, void *workspace, size_t workspace_bytes, void *stream) {
    const char *who = "tt_qkv_rmsnorm_backward";
    QkvSizes z;
    int st = check_qkv(who, B, S, H, cols, dtype, cos, sin, rope_tokens, &z);
    if (st != TT_NORM_OK) return st;
    if (!dweight_q || !dweight_k) return fail(TT_NORM_EINVAL, "%s: null dweight", who);
    const hipStream_t s = (hipStream_t)stream;
    // empty input: the parameter gradients are empty sums, written by the reducer over zero partial rows
    if (z.units() == 0) return launch_colreduce(dweight_q, dweight_k, nullptr, nullptr, 1, 0, cols, 2 * cols, dtype, s);
    st = check_qkv_ptrs(who, {dmixed, mixed, weight_q, weight_k});
    if (st != TT_NORM_OK) return st;
    for (const void *p : {dq, dk, dv})
        if (!aligned16(p)) return fail(TT_NORM_EALIGN, "%s: pointer %p not 16-byte aligned", who, p);
    const int cus = current_device_cus(&st);
    if (st != TT_NORM_OK) return st;
    const int64_t blocks = qkv_bwd_blocks(z.units(), cus);
    const size_t need = (size_t)blocks * 2 * cols * sizeof(float);
    if (!workspace || workspace_bytes < need)
        return fail(TT_NORM_EWORKSPACE, "%s: workspace %zu B < required %zu B", who, workspace_bytes, need);
    if (!aligned16(workspace)) return fail(TT_NORM_EALIGN, "%s: workspace %p not 16-byte aligned", who, workspace);
    const bool full = qkv_pieces(cols, dtype) == z.lanes;
    const RopeTable rope{cos, sin, rope_tokens};
#define CALL(T, L, F, R, r)                                                                                        \
    launch_qkv_bwd<T, L, F, R>(z, blocks, dmixed, workspace, dq, dk, dv, mixed, weight_q, weight_k, r, (float)eps, s)
    TTN_QKV_DISPATCH(CALL);
#undef CALL
    st = check_launch("qkv backward launch");
    if (st != TT_NORM_OK) return st;
    return launch_colreduce(dweight_q, dweight_k, nullptr, (const float *)workspace, 1, (int)blocks, cols, 2 * cols, dtype, s);
}

}  // extern "C"
