// RMSNorm and AdaLN for any row width: cols a multiple of one 16-byte access
// (8 two-byte or 4 four-byte elements), up to 1024 accesses per row (8192 / 4096
// columns), for bf16, fp16 and fp32.  The widths and types the tuned kernels in
// rmsnorm.hip / adaln.hip are not built for land here, so that smaller models
// (other hidden sizes and head dimensions) still run fused.
//
// Same arithmetic and rounding points as the tuned kernels, same row -> lane
// geometry, but the width is a run-time argument: a row is laid over a padded
// geometry of LANES x CHUNKS accesses (the smallest instantiated one that holds
// it) and every lane knows which of its accesses fall inside the row.  Accesses
// outside read zeros and write nothing.  The parameter-gradient reduction is
// the same fixed-order two-stage scheme, so results are bit-identical from run
// to run.
#include <hip/hip_runtime.h>

#include "norm_device.h"
#include "norm_host.h"

// Rows of a full wavefront (33 pieces and more) are read and written through buffer resources that end with the row, and
// the backward kernels with registers for a second row (rows of up to six accesses; gated from three on) request it between
// the two passes of the current one; what bounds them is the memory system and, below some 50 MB per tensor, the fixed
// cost of a launch (ramp, last rows, flush of the column sums).
// Measured as calls with the reducer behind them, against plain masked loads, no request ahead, two or three workgroups
// per compute unit and one wavefront at a time in the flush: AdaLN backward 12000 x 1536 bf16 30.4 -> 25.1 us,
// 8 x 1025 x 1536 fp16 26.4 -> 21.1, 12000 x 1024 24.5 -> 20.1, 40000 x 2560 149 -> 104 (five accesses per lane instead
// of six, one of them empty), 30000 x 1536 fp32 105 -> 96; RMSNorm backward 12000 x 2560 51.7 -> 36.5; gated backward
// 12000 x 2560 94 -> 71.  The packed forms of the products (widerow.hip) measure the same here.

// Cache policy (sc0 = 1, nt = 2, sc1 = 16) of full-wavefront rows: loads and forward stores non-temporal, backward
// stores write-through as well (plain non-temporal: 1536 columns 184 instead of 182 us, 1024 196 / 186; strided views of
// 6144 columns 140.6 / 137.4, of 4096 82.7 / 82.9, of 8192 and of 4096 fp32 the same).
#ifndef TTN_ANY_LOAD_POLICY
#define TTN_ANY_LOAD_POLICY 2
#endif
#ifndef TTN_ANY_FWD_STORE_POLICY
#define TTN_ANY_FWD_STORE_POLICY 2
#endif
#ifndef TTN_ANY_BWD_STORE_POLICY
#define TTN_ANY_BWD_STORE_POLICY 18
#endif
// The same for rows of part of a wavefront: 1 = write-through (RowWriter<1>), 0 = plain streaming store.
#ifndef TTN_ANY_FWD_STORE
#define TTN_ANY_FWD_STORE 0
#endif
#ifndef TTN_ANY_BWD_STORE
#define TTN_ANY_BWD_STORE 1
#endif
// Into a strided view the rows of neighbouring heads come from different wavefronts: a row that does not end with a 128-byte
// line then shares one, which the L2 puts together only if it is not written through (39062 x 16 x 80 bf16 101.8 -> 89.7 us;
// rows of whole lines the same either way, 48828 x 16 x 64 65.4 / 65.0).
#ifndef TTN_ANY_STRIDED_BWD_STORE
#define TTN_ANY_STRIDED_BWD_STORE 0
#endif
// AdaLN forward of two-byte rows whose grid of one row per wavefront is larger than what the chip holds at a time: rows
// per wavefront, which share the modulation row (100000 x 1024 bf16 one row 79.5, two 75.3 us; 30000 x 768 23.2 / 21.6;
// 12000 x 1024 12.2 / 11.1).  A grid that fits gets longer with a second row (64 x 64 x 1024 fp32 8.6 instead of 7.0 us,
// 6000 x 1024 bf16 7.6 / 7.3).  The gated form and four-byte rows, with twice the bytes per row of the modulation, gain
// nothing or lose (gated 100000 x 1024 138.3 / 141.6, 30000 x 1024 fp32 81.4 / 84.4; 20000 x 1536 fp32 42.9 / 43.9).
#ifndef TTN_ANY_ADALN_FWD_ROWS
#define TTN_ANY_ADALN_FWD_ROWS 2
#endif
// Backward workgroups per compute unit by accesses per lane (1 to 6).  One with the next row requested ahead beats two
// and three without from three accesses on (12000 x 2560: 37.5 against 41.2 us), and writes fewer partial rows.  Rows of
// one access take four: with a second row buffer in flight six only add partial rows and contention (RMSNorm backward
// 200000 x 256 bf16 with six 65.7 us, four 57.8, three 55.8; 100000 x 512 61.7 / 57.5 / 55.2), while three lose on strided
// views of short rows (9000 x 16 x 96: 26.2 with four, 27.3 with three).
#ifndef TTN_ANY_BWD_BLOCKS
#define TTN_ANY_BWD_BLOCKS {4, 2, 1, 1, 1, 1}
#endif

namespace ttn {

constexpr int kLoad = TTN_ANY_LOAD_POLICY, kFwdStore = TTN_ANY_FWD_STORE_POLICY, kBwdStore = TTN_ANY_BWD_STORE_POLICY;

template <typename T, int LANES_, int CHUNKS_>
struct PadGeom {
    static constexpr int VEC = Elem<T>::VEC;
    static constexpr int LANES = LANES_;
    static constexpr int CHUNKS = CHUNKS_;
    static constexpr int RPW = kWaveSize / LANES;
    static_assert(LANES >= kMinRowLanes, "the host's row-stride cap assumes at most kMaxRowsPerWave rows per wavefront");
    static_assert(LANES == 8 || LANES == 16 || LANES == 32 || LANES == 64, "row must fill an aligned lane group");
    static_assert(LANES == 64 || CHUNKS == 1, "only full wavefronts take several accesses per lane");
};

// Which of this lane's accesses lie inside a row of `pieces` 16-byte pieces.
template <typename G>
struct LaneMask {
    bool in[G::CHUNKS];
    __device__ __forceinline__ LaneMask(int l, int pieces) {
#pragma unroll
        for (int k = 0; k < G::CHUNKS; ++k) in[k] = k * G::LANES + l < pieces;
    }
};

// The rows of one wavefront step: full wavefronts read their one row through a bounded resource, narrower rows
// through per-lane addresses.  row_base is the lane's row.
template <typename G>
__device__ __forceinline__ void load_row(u32x4 (&dst)[G::CHUNKS], const void *row_base, int l, bool ok,
                                         const LaneMask<G> &m, uint32_t bytes) {
    if constexpr (G::LANES == kWaveSize) {
        const BoundedRow<kLoad> row(row_base, ok ? bytes : 0, l);
#pragma unroll
        for (int k = 0; k < G::CHUNKS; ++k) dst[k] = row.get(k * G::LANES);
    } else {
        const u32x4 *p = reinterpret_cast<const u32x4 *>(row_base) + l;
#pragma unroll
        for (int k = 0; k < G::CHUNKS; ++k) dst[k] = (ok && m.in[k]) ? load16_stream(p + k * G::LANES) : u32x4{0, 0, 0, 0};
    }
}

// Writes of one wavefront step: `first` is the wavefront's first row, lane_bytes the distance to the lane's piece.
template <typename G, int THROUGH, int POLICY>
struct RowOut {
    static constexpr bool kBounded = G::LANES == kWaveSize;
    std::conditional_t<kBounded, BoundedRow<POLICY>, RowWriter<THROUGH>> w;
    __device__ __forceinline__ RowOut(void *first, uint32_t lane_bytes, int l, uint32_t bytes)
        : w([&] {
              if constexpr (kBounded)
                  return BoundedRow<POLICY>(first, bytes, l);
              else
                  return RowWriter<THROUGH>(first, lane_bytes);
          }()) {}
    __device__ __forceinline__ void put(int k, bool ok, const LaneMask<G> &m, const u32x4 &v) const {
        if constexpr (kBounded)
            w.put(k * G::LANES, v);
        else if (ok && m.in[k])
            w.put(k * G::LANES, v);
    }
};

template <typename G>
__device__ __forceinline__ void load_param(u32x4 (&dst)[G::CHUNKS], const void *base, int l, const LaneMask<G> &m) {
    const u32x4 *p = reinterpret_cast<const u32x4 *>(base) + l;
#pragma unroll
    for (int k = 0; k < G::CHUNKS; ++k) dst[k] = m.in[k] ? load16(p + k * G::LANES) : u32x4{0, 0, 0, 0};
}

// Workgroup-level flush of per-lane column sums: rows of a wavefront folded by
// shuffles; then, one set at a time, every wavefront deposits its sums in an LDS region
// of its own and all threads add the four regions in wavefront order into the fp32 row of
// NSETS*C partial sums.  lds holds kRowWaves*C floats.
template <typename G, int NSETS>
__device__ __forceinline__ void flush_partials_anywidth(float (&acc)[NSETS][G::CHUNKS][G::VEC],
                                                        float *__restrict__ partial_row, float *lds, int C,
                                                        const LaneMask<G> &m) {
    constexpr int VEC = G::VEC, LANES = G::LANES, CHUNKS = G::CHUNKS;
    const int lane = threadIdx.x & 63;
    const int sub = lane / LANES;
    const int l = lane % LANES;
    const int wave = wave_id_in_block();
#pragma unroll
    for (int s = 0; s < NSETS; ++s)
#pragma unroll
        for (int k = 0; k < CHUNKS; ++k)
#pragma unroll
            for (int j = 0; j < VEC; ++j) acc[s][k][j] = fold_rows_of_wave<LANES>(acc[s][k][j]);
#pragma unroll
    for (int s = 0; s < NSETS; ++s) {
        if (s > 0) __syncthreads();  // the set before has been read
        if (sub == 0) {
#pragma unroll
            for (int k = 0; k < CHUNKS; ++k) {
                if (!m.in[k]) continue;
                float *p = lds + wave * C + (k * LANES + l) * VEC;
#pragma unroll
                for (int q = 0; q < VEC / 4; ++q) {
                    // copies the compiler cannot see through: a 16-byte store must not pin the accumulators to
                    // groups of four consecutive registers for the whole kernel
                    float a0 = acc[s][k][4 * q], a1 = acc[s][k][4 * q + 1], a2 = acc[s][k][4 * q + 2], a3 = acc[s][k][4 * q + 3];
                    asm volatile("" : "+v"(a0), "+v"(a1), "+v"(a2), "+v"(a3));
                    *reinterpret_cast<u32x4 *>(p + 4 * q) = u32x4{as_u32(a0), as_u32(a1), as_u32(a2), as_u32(a3)};
                }
            }
        }
        __syncthreads();
        for (int i = threadIdx.x; i < C / 4; i += kRowThreads) {
            u32x4 part[kRowWaves], sum;
#pragma unroll
            for (int w = 0; w < kRowWaves; ++w) part[w] = *reinterpret_cast<const u32x4 *>(lds + w * C + 4 * i);
#pragma unroll
            for (int j = 0; j < 4; ++j)
                sum[j] = as_u32(((as_f32(part[0][j]) + as_f32(part[1][j])) + as_f32(part[2][j])) + as_f32(part[3][j]));
            *reinterpret_cast<u32x4 *>(partial_row + s * C + 4 * i) = sum;
        }
    }
}

// ------------------------------------------------------------------ RMSNorm

template <typename T, int LANES, int CHUNKS, typename Map>
__global__ __launch_bounds__(kRowThreads) void anywidth_rmsnorm_fwd_kernel(
    T *__restrict__ out, float *__restrict__ rstd, const T *__restrict__ x, const T *__restrict__ w,
    const Map map, int C, float eps) {
    using G = PadGeom<T, LANES, CHUNKS>;
    using E = Elem<T>;
    constexpr int VEC = G::VEC, RPW = G::RPW;
    const int lane = threadIdx.x & 63;
    const int sub = lane / LANES;
    const int l = lane % LANES;
    const int wave = wave_id_in_block();
    const LaneMask<G> m(l, C / VEC);
    const uint32_t row_bytes = (uint32_t)(C * (int)sizeof(T));

    u32x4 wr[CHUNKS];
    load_param<G>(wr, w, l, m);

    const int64_t groups = map.template groups<RPW>();
    const int64_t stride = (int64_t)gridDim.x * kRowWaves;
    for (int64_t grp = (int64_t)blockIdx.x * kRowWaves + wave; grp < groups; grp += stride) {
        keep_packed(wr);
        const RowAddr at = map.template locate<RPW>(grp, sub, C);
        const int64_t row = at.row;
        const bool ok = at.ok;
        u32x4 xr[CHUNKS];
        load_row<G>(xr, x + at.xoff, l, ok, m, row_bytes);

        float ss = 0.0f;
#pragma unroll
        for (int k = 0; k < CHUNKS; ++k) {
            float v[VEC];
            E::unpack(xr[k], v);
#pragma unroll
            for (int j = 0; j < VEC; ++j) ss = fmaf(v[j], v[j], ss);
        }
        ss = group_sum<LANES>(ss);
        const float r = 1.0f / sqrtf(ss / (float)C + eps);
        if (ok && l == 0) rstd[row] = r;

        // the wavefront's rows are consecutive in out: base = its first row
        const RowOut<G, TTN_ANY_FWD_STORE, kFwdStore> wo(out + map.template locate<RPW>(grp, 0, C).row * C,
                                              (uint32_t)(sub * C * (int)sizeof(T)) + l * 16, l, row_bytes);
#pragma unroll
        for (int k = 0; k < CHUNKS; ++k) {
            float v[VEC], wv[VEC];
            E::unpack(xr[k], v);
            E::unpack(wr[k], wv);
#pragma unroll
            for (int j = 0; j < VEC; ++j) v[j] *= r;
            E::round(v);  // y = normalised row in the element type
#pragma unroll
            for (int j = 0; j < VEC; ++j) v[j] *= wv[j];
            wo.put(k, ok, m, E::pack(v));
        }
    }
}

template <typename T, int LANES, int CHUNKS, typename Map>
__global__ __launch_bounds__(kRowThreads) void anywidth_rmsnorm_bwd_kernel(
    T *__restrict__ dx, float *__restrict__ partial, const T *__restrict__ g, const T *__restrict__ x,
    const T *__restrict__ w, const float *__restrict__ rstd, const Map map, int C) {
    using G = PadGeom<T, LANES, CHUNKS>;
    using E = Elem<T>;
    constexpr int VEC = G::VEC, RPW = G::RPW;
    extern __shared__ __align__(16) float lds[];
    const int lane = threadIdx.x & 63;
    const int sub = lane / LANES;
    const int l = lane % LANES;
    const int wave = wave_id_in_block();
    const LaneMask<G> m(l, C / VEC);
    const uint32_t row_bytes = (uint32_t)(C * (int)sizeof(T));

    u32x4 wr[CHUNKS];
    load_param<G>(wr, w, l, m);
    float acc[1][CHUNKS][VEC];
#pragma unroll
    for (int k = 0; k < CHUNKS; ++k)
#pragma unroll
        for (int j = 0; j < VEC; ++j) acc[0][k][j] = 0.0f;

    struct Row {
        u32x4 g[CHUNKS], x[CHUNKS];
        float r;
        RowAddr at;
        int64_t doff0;
    };
    const int64_t groups = map.template groups<RPW>();
    const int64_t stride = (int64_t)gridDim.x * kRowWaves;
    auto fetch = [&](Row &b, int64_t grp) {
        b.at = map.template locate<RPW>(grp, sub, C);
        b.doff0 = map.template locate<RPW>(grp, 0, C).doff;
        load_row<G>(b.g, g + b.at.row * C, l, b.at.ok, m, row_bytes);
        load_row<G>(b.x, x + b.at.xoff, l, b.at.ok, m, row_bytes);
        b.r = b.at.ok ? rstd[b.at.row] : 0.0f;
    };
    auto process = [&](Row &b, auto &&between_passes) {
        keep_packed(wr);
        const float r = b.r;
        // pass 1: gy = rnd(g*w) kept packed; row dot  sum_c gy * x
        u32x4 gyp[CHUNKS];
        float dot = 0.0f;
#pragma unroll
        for (int k = 0; k < CHUNKS; ++k) {
            gyp[k] = packed_products<T>(b.g[k], wr[k]);
            if constexpr (kHasDot2<T>) {
#pragma unroll
                for (int i = 0; i < 4; ++i) dot = dot2<T>(gyp[k][i], b.x[k][i], dot);
            } else {
                float gy[VEC], xv[VEC];
                E::unpack(gyp[k], gy);
                E::unpack(b.x[k], xv);
#pragma unroll
                for (int j = 0; j < VEC; ++j) dot = fmaf(gy[j], xv[j], dot);
            }
        }
        dot = group_sum<LANES>(dot);
        between_passes();
        // dx = r*(gy - xhat * mean_c(gy*xhat)) = gy*r + x*coef
        const float coef = -((dot / (float)C) * r * r * r);
        // the second pass unpacks the row again rather than holding pass 1's fp32 copies live
        keep_packed(b.g);
        keep_packed(b.x);
        keep_packed(gyp);

        // dx goes through its own strides: base = the wavefront's first row, the lane adds its row's distance
        const RowOut<G, (std::is_same<Map, DenseRows>::value ? TTN_ANY_BWD_STORE : TTN_ANY_STRIDED_BWD_STORE), kBwdStore> wd(
            dx + b.doff0, (uint32_t)((b.at.doff - b.doff0) * (int64_t)sizeof(T)) + l * 16, l, row_bytes);
#pragma unroll
        for (int k = 0; k < CHUNKS; ++k) {
            float gy[VEC], xv[VEC], o[VEC], y[VEC];
            E::unpack(gyp[k], gy);
            E::unpack(b.x[k], xv);
#pragma unroll
            for (int j = 0; j < VEC; ++j) {
                o[j] = fmaf(xv[j], coef, gy[j] * r);
                y[j] = xv[j] * r;
            }
            wd.put(k, b.at.ok, m, E::pack(o));
            add_columns<T>(acc[0][k], packed_products<T>(b.g[k], E::pack(y)));  // dw += rnd(g * rnd(y))
        }
    };
    row_pipeline<CHUNKS <= 6 ? 2 : 1, true, Row>(
        (int64_t)blockIdx.x * kRowWaves + wave, groups, stride, fetch, process, [] {});
    flush_partials_anywidth<G, 1>(acc, partial + (int64_t)blockIdx.x * C, lds, C, m);
}

// -------------------------------------------------------------------- AdaLN

// GATED = true: the normalised row is first formed as h2 = rnd(x + rnd(attn * gate[b])) (the gated residual
// update that precedes the norm in the transformer blocks) and written out too.
template <typename T, int LANES, int CHUNKS, bool GATED>
__global__ __launch_bounds__(kRowThreads) void anywidth_adaln_fwd_kernel(
    T *__restrict__ out, float *__restrict__ mean, float *__restrict__ rstd, const T *__restrict__ x,
    const T *__restrict__ scale, const T *__restrict__ shift, T *__restrict__ h2_out, const T *__restrict__ attn,
    const T *__restrict__ gate, int64_t rows_per_sample, const SampleLayout lay, int blocks_per_sample, int C,
    float eps) {
    using G = PadGeom<T, LANES, CHUNKS>;
    using E = Elem<T>;
    constexpr int VEC = G::VEC, RPW = G::RPW;
    const int lane = threadIdx.x & 63;
    const int sub = lane / LANES;
    const int l = lane % LANES;
    const int wave = wave_id_in_block();
    const int64_t b = blockIdx.x / blocks_per_sample;  // sample this workgroup serves
    const int slot = blockIdx.x % blocks_per_sample;
    const LaneMask<G> m(l, C / VEC);
    const uint32_t row_bytes = (uint32_t)(C * (int)sizeof(T));

    // Two orders of the requests.  Two-byte rows ask for the modulation row first and form t = rnd(1 + scale) behind the
    // row's statistics, which then wait for neither (row first, t before the statistics: 3000 x 1536 bf16 6.5 instead of
    // 6.0 us, 4400 x 1536 8.2 / 7.6, gated 30000 x 768 40.9 / 35.0).  Four-byte rows, with half the arithmetic per byte,
    // ask for the row first and wait for all of it before they start, which keeps the chip's reads apart from its writes
    // (3700 x 1024 fp32 6.3 us, the other order 7.7).  Rows of one access are walked by a persistent grid: t once per
    // wavefront.
    constexpr bool kRowFirst = sizeof(T) == 4 && CHUNKS > 1;
    constexpr bool kFormLate = sizeof(T) == 2 && CHUNKS > 1;
    u32x4 tr[CHUNKS], hr[CHUNKS];
    [[maybe_unused]] u32x4 qr[GATED ? CHUNKS : 1];
    auto one_plus = [](const u32x4 &raw) -> u32x4 {
        float v[VEC];
        E::unpack(raw, v);
#pragma unroll
        for (int j = 0; j < VEC; ++j) v[j] = 1.0f + v[j];
        return E::pack(v);
    };

    const int64_t groups = (rows_per_sample + RPW - 1) / RPW;
    const int64_t stride = (int64_t)blocks_per_sample * kRowWaves;
    const uint32_t lane_bytes = (uint32_t)(sub * lay.row_stride * C * (int64_t)sizeof(T)) + l * 16;
    u32x4 xr[CHUNKS];
    [[maybe_unused]] u32x4 ar[GATED ? CHUNKS : 1];
    auto fetch = [&](int64_t i) {
        const int64_t rs = i * RPW + sub;
        const int64_t at = lay.row(b, rs) * C;
        load_row<G>(xr, x + at, l, rs < rows_per_sample, m, row_bytes);
        if constexpr (GATED) load_row<G>(ar, attn + at, l, rs < rows_per_sample, m, row_bytes);
    };
    int64_t grp = (int64_t)slot * kRowWaves + wave;
    if constexpr (kRowFirst) {
        if (grp < groups) fetch(grp);
    }
    load_param<G>(tr, scale + b * C, l, m);
    load_param<G>(hr, shift + b * C, l, m);
    if constexpr (GATED) load_param<G>(qr, gate + b * C, l, m);
    if constexpr (!kRowFirst) {
        if (grp < groups) fetch(grp);
    }
    if constexpr (!kFormLate) {
#pragma unroll
        for (int k = 0; k < CHUNKS; ++k) tr[k] = one_plus(tr[k]);
    }

    for (; grp < groups; grp += stride) {
        keep_packed(tr);
        keep_packed(hr);
        if constexpr (GATED) keep_packed(qr);
        const int64_t rs = grp * RPW + sub;
        const bool ok = rs < rows_per_sample;
        const int64_t row = lay.row(b, rs);
        const int64_t first = lay.row(b, grp * RPW) * C;  // the wavefront's first row: base of what it writes
        if constexpr (GATED) {
            const RowOut<G, TTN_ANY_FWD_STORE, kFwdStore> wh(h2_out + first, lane_bytes, l, row_bytes);
#pragma unroll
            for (int k = 0; k < CHUNKS; ++k) {
                float hv[VEC], av[VEC], gv[VEC];
                E::unpack(xr[k], hv);
                E::unpack(ar[k], av);
                E::unpack(qr[k], gv);
#pragma unroll
                for (int j = 0; j < VEC; ++j) av[j] *= gv[j];
                E::round(av);  // attn * gate materialised in the element type
#pragma unroll
                for (int j = 0; j < VEC; ++j) hv[j] += av[j];
                xr[k] = E::pack(hv);  // h2: the new residual stream, and the row that is normalised
                wh.put(k, ok, m, xr[k]);
            }
        }

        float s = 0.0f;
#pragma unroll
        for (int k = 0; k < CHUNKS; ++k) {
            if constexpr (kHasDot2<T>) {  // row sum straight from the packed pairs
#pragma unroll
                for (int i = 0; i < 4; ++i) s = dot2<T>(xr[k][i], kOnesPair<T>, s);
            } else {
                float v[VEC];
                E::unpack(xr[k], v);
#pragma unroll
                for (int j = 0; j < VEC; ++j) s += v[j];
            }
        }
        const float mu = group_sum<LANES>(s) / (float)C;
        float q = 0.0f;
#pragma unroll
        for (int k = 0; k < CHUNKS; ++k) {
            float v[VEC];
            E::unpack(xr[k], v);
            if (m.in[k]) {  // padding must not count as (0 - mu)^2
#pragma unroll
                for (int j = 0; j < VEC; ++j) {
                    const float d = v[j] - mu;
                    q = fmaf(d, d, q);
                }
            }
        }
        const float r = 1.0f / sqrtf(group_sum<LANES>(q) / (float)C + eps);
        if (ok && l == 0) {
            mean[row] = mu;
            rstd[row] = r;
        }

        const float nmr = -(mu * r);
        const RowOut<G, TTN_ANY_FWD_STORE, kFwdStore> wo(out + first, lane_bytes, l, row_bytes);
#pragma unroll
        for (int k = 0; k < CHUNKS; ++k) {
            float v[VEC], tv[VEC], hv[VEC];
            E::unpack(xr[k], v);
            E::unpack(kFormLate ? one_plus(tr[k]) : tr[k], tv);
            E::unpack(hr[k], hv);
#pragma unroll
            for (int j = 0; j < VEC; ++j) v[j] = centred<T>(v[j], mu, r, nmr);
            E::round(v);  // xn
#pragma unroll
            for (int j = 0; j < VEC; ++j) v[j] *= tv[j];
            E::round(v);  // xn * (1 + scale)
#pragma unroll
            for (int j = 0; j < VEC; ++j) v[j] += hv[j];
            wo.put(k, ok, m, E::pack(v));
        }
        if (grp + stride < groups) fetch(grp + stride);
    }
}

// GATED: x is the saved h2; dx = dh = rnd(rnd(dx of the norm) + e) with e the gradient arriving at h2 from
// its other use (may be null), da = rnd(dh * gate[b]) is written too and dgate[b] += rnd(dh * attn) is a
// third set of column sums.  RES: dx = rnd(rnd(dx of the norm) + e), e the gradient the input receives
// from its other consumer.  (Same forms as the tuned kernels.)
template <typename T, int LANES, int CHUNKS, bool GATED, bool RES>
__global__ __launch_bounds__(kRowThreads) void anywidth_adaln_bwd_kernel(
    T *__restrict__ dx, float *__restrict__ partial, const T *__restrict__ g, const T *__restrict__ x,
    const T *__restrict__ scale, const float *__restrict__ mean, const float *__restrict__ rstd,
    T *__restrict__ da, const T *__restrict__ e, const T *__restrict__ attn, const T *__restrict__ gate,
    int64_t rows_per_sample, const SampleLayout lay, int blocks_per_sample, int C) {
    static_assert(!(GATED && RES), "the gated form handles e itself");
    static_assert(CHUNKS <= 6, "wider dense rows run on the wide-row kernels");
    constexpr int NSETS = GATED ? 3 : 2;
    using G = PadGeom<T, LANES, CHUNKS>;
    using E = Elem<T>;
    constexpr int VEC = G::VEC, RPW = G::RPW;
    extern __shared__ __align__(16) float lds[];
    const int lane = threadIdx.x & 63;
    const int sub = lane / LANES;
    const int l = lane % LANES;
    const int wave = wave_id_in_block();
    const int64_t b = blockIdx.x / blocks_per_sample;
    const int slot = blockIdx.x % blocks_per_sample;
    const LaneMask<G> m(l, C / VEC);
    const uint32_t row_bytes = (uint32_t)(C * (int)sizeof(T));

    u32x4 tr[CHUNKS];  // t = rnd(1 + scale[sample]), formed behind the first row's requests
    load_param<G>(tr, scale + b * C, l, m);
    [[maybe_unused]] u32x4 qr[GATED ? CHUNKS : 1];
    if constexpr (GATED) load_param<G>(qr, gate + b * C, l, m);

    // Gated, rows of three accesses and more: attn and e have one register buffer, which is asked to hold the next row's piece as
    // soon as the current row's has been used, as in adaln.hip (with g and x, one row at a time: 43402 x 1152 bf16 115.6 us,
    // now 106.0; 3906 x 1536 22.4 / 20.5; 24414 x 2048 111.6 / 110.0; 8 x 1025 x 1536 fp16 38.5 / 37.1).  Narrower rows
    // take them with g and x, one row at a time (ahead: 48828 x 1024 112.6 / 115.2, 50000 x 512 62.8 / 64.4), and so does
    // the residual form, which has registers for two rows (ahead it gains 2-4 % at most widths and loses 8 % at 1152).
    constexpr bool kAhead = GATED && CHUNKS >= 3;
    [[maybe_unused]] u32x4 an[kAhead ? CHUNKS : 1], en[kAhead ? CHUNKS : 1];
    [[maybe_unused]] int64_t next_row = 0;
    [[maybe_unused]] bool next_ok = false;
    [[maybe_unused]] auto request_operands = [&](int k) {
        __builtin_amdgcn_sched_barrier(0);  // spread over the second pass
        const uint32_t bytes = next_ok ? row_bytes : 0;
        an[k] = BoundedRow<kLoad>(attn + next_row * C, bytes, l).get(k * LANES);
        en[k] = BoundedRow<kLoad>(e + next_row * C, e != nullptr ? bytes : 0, l).get(k * LANES);
    };
    auto prepare = [&] {
        if constexpr (kAhead) {
#pragma unroll
            for (int k = 0; k < CHUNKS; ++k) request_operands(k);
        }
#pragma unroll
        for (int k = 0; k < CHUNKS; ++k) {
            float v[VEC];
            E::unpack(tr[k], v);
#pragma unroll
            for (int j = 0; j < VEC; ++j) v[j] = 1.0f + v[j];
            tr[k] = E::pack(v);
        }
    };

    float acc[NSETS][CHUNKS][VEC];  // [0] = dscale, [1] = dshift, [2] = dgate
#pragma unroll
    for (int s = 0; s < NSETS; ++s)
#pragma unroll
        for (int k = 0; k < CHUNKS; ++k)
#pragma unroll
            for (int j = 0; j < VEC; ++j) acc[s][k][j] = 0.0f;

    struct Row {
        u32x4 g[CHUNKS], x[CHUNKS];
        u32x4 e[(GATED || RES) && !kAhead ? CHUNKS : 1], a[GATED && !kAhead ? CHUNKS : 1];
        float r, mu;
        int64_t first;  // element offset of the wavefront's first row
        bool ok;
    };
    const int64_t groups = (rows_per_sample + RPW - 1) / RPW;
    const int64_t stride = (int64_t)blocks_per_sample * kRowWaves;
    const uint32_t lane_bytes = (uint32_t)(sub * lay.row_stride * C * (int64_t)sizeof(T)) + l * 16;
    auto fetch = [&](Row &q, int64_t grp) {
        const int64_t rs = grp * RPW + sub;
        q.ok = rs < rows_per_sample;
        const int64_t row = lay.row(b, rs);
        q.first = lay.row(b, grp * RPW) * C;
        load_row<G>(q.g, g + row * C, l, q.ok, m, row_bytes);
        load_row<G>(q.x, x + row * C, l, q.ok, m, row_bytes);
        if constexpr ((GATED || RES) && !kAhead) load_row<G>(q.e, e + row * C, l, q.ok && e != nullptr, m, row_bytes);
        if constexpr (GATED && !kAhead) load_row<G>(q.a, attn + row * C, l, q.ok, m, row_bytes);
        if constexpr (kAhead) {
            next_row = wave_uniform(row);
            next_ok = q.ok;
        }
        const int64_t srow = LANES == kWaveSize ? wave_uniform(row) : row;
        q.r = q.ok ? rstd[srow] : 0.0f;
        q.mu = q.ok ? mean[srow] : 0.0f;
    };
    // As in adaln.hip, a row's first pass waits for the stores of the row before it, which pays where a third tensor is read
    // (residual: 24414 x 2048 bf16 74.1 -> 71.5 us, 43402 x 1152 81.2 -> 78.6, 1953 x 2560 17.3 -> 15.9, 8 x 1025 x 1536 fp16
    // 26.6 -> 26.0).  The plain form loses 1-2 % and the gated one, whose operands are then waited for too, up to 7 %.
    constexpr bool kDrain = RES && LANES == kWaveSize && CHUNKS >= 2;
    auto process = [&](Row &q, auto &&between_passes) {
        keep_packed(tr);
        if constexpr (kDrain) wait_memory_ops<0>();
        const float r = q.r, mu = q.mu;
        const float nmr = -(mu * r);  // xhat = x*r + nmr
        // pass 1: gx = rnd(g*t) kept packed; s1 = sum_c gx; s2 = sum_c gx * xhat
        // (padding: g = 0 there, so gx = 0 and neither sum sees xhat = nmr)
        u32x4 gxp[CHUNKS];
        float s1 = 0.0f, s2 = 0.0f;
#pragma unroll
        for (int k = 0; k < CHUNKS; ++k) {
            gxp[k] = packed_products<T>(q.g[k], tr[k]);
            if constexpr (kHasDot2<T>) {
                // straight from the packed pairs; s2 holds sum_c gx * x here, turned into sum_c gx * xhat below
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    s1 = dot2<T>(gxp[k][i], kOnesPair<T>, s1);
                    s2 = dot2<T>(gxp[k][i], q.x[k][i], s2);
                }
            } else {
                float gv[VEC], xv[VEC];
                E::unpack(gxp[k], gv);
                E::unpack(q.x[k], xv);
#pragma unroll
                for (int j = 0; j < VEC; ++j) {
                    s1 += gv[j];
                    s2 = fmaf(gv[j], centred<T>(xv[j], mu, r, nmr), s2);
                }
            }
        }
        s1 = group_sum<LANES>(s1);
        s2 = group_sum<LANES>(s2);
        if constexpr (kAhead) next_ok = false;  // until the next row is asked for
        between_passes();
        if constexpr (kHasDot2<T>) s2 = r * (s2 - mu * s1);
        const float m1 = s1 / (float)C, m2 = s2 / (float)C;
        // dx = r*(gx - m1 - xhat*m2) = r*gx + x*K1 + K0
        const float k1 = -(r * m2), k0 = -(r * m1);
        const float K1 = k1 * r;
        const float K0 = fmaf(k1, nmr, k0);

        // the second pass unpacks the row again rather than holding pass 1's fp32 copies live
        keep_packed(q.g);
        keep_packed(q.x);
        keep_packed(gxp);
        const RowOut<G, (TTN_ANY_BWD_STORE && !GATED), kBwdStore> wd(dx + q.first, lane_bytes, l, row_bytes);
        const RowOut<G, 0, kBwdStore> wa(GATED ? da + q.first : nullptr, lane_bytes, l, row_bytes);
        if constexpr (GATED) keep_packed(qr);
#pragma unroll
        for (int k = 0; k < CHUNKS; ++k) {
            float gx[VEC], xv[VEC], o[VEC], xn[VEC];
            E::unpack(gxp[k], gx);
            E::unpack(q.x[k], xv);
#pragma unroll
            for (int j = 0; j < VEC; ++j) {
                o[j] = fmaf(r, gx[j], fmaf(xv[j], K1, K0));
                xn[j] = centred<T>(xv[j], mu, r, nmr);
            }
            if constexpr (GATED || RES) {
                float ev[VEC];
                E::round(o);  // the norm's dx, materialised in the element type
                E::unpack(kAhead ? en[k] : q.e[k], ev);
#pragma unroll
                for (int j = 0; j < VEC; ++j) o[j] += ev[j];
            }
            const u32x4 dxp = E::pack(o);
            wd.put(k, q.ok, m, dxp);
            if constexpr (GATED) {
                float av[VEC], qv[VEC];
                E::unpack(dxp, o);  // dh as stored
                E::unpack(kAhead ? an[k] : q.a[k], av);
                E::unpack(qr[k], qv);
#pragma unroll
                for (int j = 0; j < VEC; ++j) {
                    qv[j] *= o[j];
                    av[j] *= o[j];
                }
                wa.put(k, q.ok, m, E::pack(qv));
                E::round(av);  // dh*attn materialised in the element type before the column sum
#pragma unroll
                for (int j = 0; j < VEC; ++j) acc[2][k][j] += av[j];
            }
            if constexpr (kAhead) request_operands(k);
            add_columns<T>(acc[1][k], q.g[k]);                                    // dshift += g (padding: g = 0)
            add_columns<T>(acc[0][k], packed_products<T>(q.g[k], E::pack(xn)));  // dscale += rnd(g * rnd(xhat))
        }
    };
    row_pipeline<GATED && !kAhead ? 1 : 2, true, Row>((int64_t)slot * kRowWaves + wave, groups, stride, fetch, process,
                                          prepare);
    flush_partials_anywidth<G, NSETS>(acc, partial + (int64_t)blockIdx.x * (NSETS * C), lds, C, m);
}

// ---------------------------------------------------------------- dispatch

constexpr int kMaxPieces = 1024;  // 16-byte accesses per row: 64 lanes x 16

bool anywidth_supported(int64_t cols, int dtype) {
    if (dtype != TT_NORM_BF16 && dtype != TT_NORM_F32 && dtype != TT_NORM_F16) return false;
    const int vec = 16 / (int)elem_bytes(dtype);
    return cols > 0 && cols % vec == 0 && cols / vec <= kMaxPieces;
}

// The smallest instantiated geometry that holds `pieces` accesses.
struct GeomChoice {
    int lanes, chunks;
};
static GeomChoice choose_geometry(int pieces) {
    if (pieces <= 8) return {8, 1};
    if (pieces <= 16) return {16, 1};
    if (pieces <= 32) return {32, 1};
    const int need = (pieces + 63) / 64;
    for (int c : {1, 2, 3, 4, 5, 6, 8, 12, 16})
        if (need <= c) return {64, c};
    return {0, 0};
}

// Calls F<T, LANES, CHUNKS>::run(args...) for the run-time (dtype, geometry).
#define TTN_ANYWIDTH_GEOMS(X, T) \
    X(T, 8, 1) X(T, 16, 1) X(T, 32, 1) X(T, 64, 1) X(T, 64, 2) X(T, 64, 3) X(T, 64, 4) X(T, 64, 5) X(T, 64, 6) X(T, 64, 8) X(T, 64, 12) X(T, 64, 16)

template <template <typename, int, int> class F, typename... Args>
static int dispatch(int dtype, GeomChoice gc, Args... args) {
#define TTN_TRY(T, L, K) \
    if (gc.lanes == L && gc.chunks == K) return F<T, L, K>::run(args...);
    if (dtype == TT_NORM_BF16) {
        TTN_ANYWIDTH_GEOMS(TTN_TRY, bf16_t)
    } else if (dtype == TT_NORM_F16) {
        TTN_ANYWIDTH_GEOMS(TTN_TRY, f16_t)
    } else {
        TTN_ANYWIDTH_GEOMS(TTN_TRY, float)
    }
#undef TTN_TRY
    return fail(TT_NORM_EUNSUPPORTED, "no kernel geometry for %d lanes x %d accesses", gc.lanes, gc.chunks);
}

// Launch policy.  Forward: narrow rows (one access per lane) use a persistent grid of 16 workgroups
// per compute unit, wider rows one row per wavefront (AdaLN: see share_modulation).  Backward is
// persistent (column sums live in registers); the grid shrinks as rows widen so that each compute unit
// keeps about the same number of bytes in flight.
constexpr int kOneShotAny = 1 << 20;
static int fwd_blocks_per_cu(int chunks) { return chunks == 1 ? 16 : kOneShotAny; }
static int bwd_blocks_per_cu(int chunks) {
    constexpr int blocks[] = TTN_ANY_BWD_BLOCKS;
    return chunks > 6 ? 1 : blocks[chunks - 1];
}

static GeomChoice geometry_for(int64_t cols, int dtype) {
    return choose_geometry((int)(cols / (16 / (int)elem_bytes(dtype))));
}

// Grid for (batch, rows_per_sample) under geometry gc; status != OK on failure.
static int plan_for(RowPlan *plan, int64_t batch, int64_t rows_per_sample, GeomChoice gc, bool backward) {
    int st = TT_NORM_OK;
    const int cus = current_device_cus(&st);
    if (st != TT_NORM_OK) return st;
    *plan = make_row_plan(batch, rows_per_sample, kWaveSize / gc.lanes,
                          backward ? bwd_blocks_per_cu(gc.chunks) : fwd_blocks_per_cu(gc.chunks), cus);
    if (plan->blocks > kMostBlocks && batch <= kMostBlocks) {  // the kernels walk whatever the grid leaves
        plan->blocks_per_sample = (int)(kMostBlocks / batch);
        plan->blocks = batch * plan->blocks_per_sample;
    }
    if (plan->blocks > 0x7fffffffLL) return fail(TT_NORM_EINVAL, "grid too large");
    return TT_NORM_OK;
}

// A grid of one row per wavefront that the chip cannot hold at once: TTN_ANY_ADALN_FWD_ROWS rows per wavefront instead.
constexpr int kMostResident = 8;  // workgroups of four wavefronts that fill a compute unit
static int share_modulation(RowPlan *plan, int resident) {
    int st = TT_NORM_OK;
    const int cus = current_device_cus(&st);
    if (st != TT_NORM_OK) return st;
    const int64_t batch = plan->blocks / plan->blocks_per_sample;
    if (plan->blocks > (int64_t)cus * resident) {
        plan->blocks_per_sample = (plan->blocks_per_sample + TTN_ANY_ADALN_FWD_ROWS - 1) / TTN_ANY_ADALN_FWD_ROWS;
        plan->blocks = batch * plan->blocks_per_sample;
    }
    return TT_NORM_OK;
}

template <typename Map>
struct RmsOn {  // the RMSNorm kernels over one kind of row map
    template <typename T, int LANES, int CHUNKS>
    struct Fwd {
        static int run(const RowPlan &p, void *out, float *rstd, const void *x, const void *w, const Map &map, int C,
                       double eps, hipStream_t stream) {
            if constexpr (CHUNKS > 6 && std::is_same<Map, DenseRows>::value) {  // run on the wide-row kernels
                return fail(TT_NORM_EUNSUPPORTED, "RMSNorm: dense rows of more than six 16-byte accesses per lane");
            } else {
                RowKernelProfile prof(stream);
                anywidth_rmsnorm_fwd_kernel<T, LANES, CHUNKS, Map><<<dim3((unsigned)p.blocks), dim3(kRowThreads), 0, stream>>>(
                    (T *)out, rstd, (const T *)x, (const T *)w, map, C, (float)eps);
                return TT_NORM_OK;
            }
        }
    };
    template <typename T, int LANES, int CHUNKS>
    struct Bwd {
        static int run(const RowPlan &p, void *dx, void *ws, const void *g, const void *x, const void *w,
                       const float *rstd, const Map &map, int C, hipStream_t stream) {
            if constexpr (CHUNKS > 6 && std::is_same<Map, DenseRows>::value) {
                return fail(TT_NORM_EUNSUPPORTED, "RMSNorm backward: dense rows of more than six 16-byte accesses per lane");
            } else {
                RowKernelProfile prof(stream);
                anywidth_rmsnorm_bwd_kernel<T, LANES, CHUNKS, Map>
                    <<<dim3((unsigned)p.blocks), dim3(kRowThreads), (size_t)kRowWaves * C * sizeof(float), stream>>>(
                        (T *)dx, (float *)ws, (const T *)g, (const T *)x, (const T *)w, rstd, map, C);
                return TT_NORM_OK;
            }
        }
    };
};

struct AdalnExtra {  // operands of the gated / residual forms (null otherwise)
    void *h2_or_da;   // forward: h2 out; backward: dattn out
    const void *e;    // backward: the other gradient (dh2 or dres), may be null for the gated form
    const void *attn;
    const void *gate;
};

template <bool GATED, bool RES>
struct AdalnOn {
    template <typename T, int LANES, int CHUNKS>
    struct Fwd {
        static int run(const RowPlan &p, void *out, float *mean, float *rstd, const void *x, const void *scale,
                       const void *shift, const AdalnExtra &ex, int64_t rows_per_sample, SampleLayout lay, int C,
                       double eps, hipStream_t stream) {
            if constexpr (CHUNKS > 6) {  // wider dense rows run on the wide-row kernels
                return fail(TT_NORM_EUNSUPPORTED, "AdaLN: rows of more than six 16-byte accesses per lane");
            } else {
                RowPlan q = p;
                if constexpr (!GATED && sizeof(T) == 2 && CHUNKS > 1) {
                    static const int resident =
                        resident_blocks_per_cu(anywidth_adaln_fwd_kernel<T, LANES, CHUNKS, GATED>, kMostResident);
                    const int st = share_modulation(&q, resident);
                    if (st != TT_NORM_OK) return st;
                }
                RowKernelProfile prof(stream);
                anywidth_adaln_fwd_kernel<T, LANES, CHUNKS, GATED><<<dim3((unsigned)q.blocks), dim3(kRowThreads), 0, stream>>>(
                    (T *)out, mean, rstd, (const T *)x, (const T *)scale, (const T *)shift, (T *)ex.h2_or_da,
                    (const T *)ex.attn, (const T *)ex.gate, rows_per_sample, lay, q.blocks_per_sample, C, (float)eps);
                return TT_NORM_OK;
            }
        }
    };
    template <typename T, int LANES, int CHUNKS>
    struct Bwd {
        static int run(const RowPlan &p, void *dx, void *ws, const void *g, const void *x, const void *scale,
                       const float *mean, const float *rstd, const AdalnExtra &ex, int64_t rows_per_sample,
                       SampleLayout lay, int C, hipStream_t stream) {
            if constexpr (CHUNKS > 6) {
                return fail(TT_NORM_EUNSUPPORTED, "AdaLN backward: rows of more than six 16-byte accesses per lane");
            } else {
                RowKernelProfile prof(stream);
                anywidth_adaln_bwd_kernel<T, LANES, CHUNKS, GATED, RES>
                    <<<dim3((unsigned)p.blocks), dim3(kRowThreads), (size_t)kRowWaves * C * sizeof(float), stream>>>(
                        (T *)dx, (float *)ws, (const T *)g, (const T *)x, (const T *)scale, mean, rstd,
                        (T *)ex.h2_or_da, (const T *)ex.e, (const T *)ex.attn, (const T *)ex.gate, rows_per_sample,
                        lay, p.blocks_per_sample, C);
                return TT_NORM_OK;
            }
        }
    };
};

template <typename Map>
static int rmsnorm_forward_on(void *out, float *rstd, const void *x, const void *w, const Map &map, int64_t rows,
                              int64_t cols, double eps, int dtype, hipStream_t stream) {
    if (rows == 0) return TT_NORM_OK;
    const GeomChoice gc = geometry_for(cols, dtype);
    RowPlan p;
    int st = plan_for(&p, 1, rows, gc, false);
    if (st != TT_NORM_OK) return st;
    st = dispatch<RmsOn<Map>::template Fwd>(dtype, gc, p, out, rstd, x, w, map, (int)cols, eps, stream);
    return st != TT_NORM_OK ? st : check_launch("rmsnorm forward launch");
}

int anywidth_rmsnorm_forward(void *out, float *rstd, const void *x, const void *w, int64_t rows, int64_t cols,
                             double eps, int dtype, hipStream_t stream) {
    if (widerow_takes(cols, dtype)) return widerow_rmsnorm_forward(out, rstd, x, w, rows, cols, eps, dtype, stream);
    return rmsnorm_forward_on(out, rstd, x, w, DenseRows{rows}, rows, cols, eps, dtype, stream);
}

int anywidth_rmsnorm_forward_strided(void *out, float *rstd, const void *x, const void *w, const Strided3Rows &map,
                                     int64_t cols, double eps, int dtype, hipStream_t stream) {
    return rmsnorm_forward_on(out, rstd, x, w, map, map.n0 * map.n1 * map.n2, cols, eps, dtype, stream);
}

static size_t backward_scratch(int64_t batch, int64_t rows_per_sample, int64_t cols, int dtype, int nsets) {
    if (batch <= 0 || rows_per_sample <= 0 || !anywidth_supported(cols, dtype)) return 0;
    RowPlan p;
    if (plan_for(&p, batch, rows_per_sample, geometry_for(cols, dtype), true) != TT_NORM_OK) return 0;
    size_t need = (size_t)p.blocks * nsets * cols * sizeof(float);
    if (widerow_takes(cols, dtype)) {  // dense rows take the other kernels, strided views these
        const size_t wide = widerow_backward_workspace_bytes(batch, rows_per_sample, cols, dtype, nsets);
        if (wide == 0) return 0;
        if (wide > need) need = wide;
    }
    return need;
}

size_t anywidth_rmsnorm_backward_workspace_bytes(int64_t rows, int64_t cols, int dtype) {
    return backward_scratch(1, rows, cols, dtype, 1);
}

template <typename Map>
static int rmsnorm_backward_on(void *dx, void *dw, const void *g, const void *x, const void *w, const float *rstd,
                               const Map &map, int64_t rows, int64_t cols, int dtype, void *ws, size_t ws_bytes,
                               hipStream_t stream) {
    if (rows == 0) return launch_colreduce(dw, nullptr, nullptr, nullptr, 1, 0, cols, cols, dtype, stream);
    const GeomChoice gc = geometry_for(cols, dtype);
    RowPlan p;
    int st = plan_for(&p, 1, rows, gc, true);
    if (st != TT_NORM_OK) return st;
    const size_t need = (size_t)p.blocks * cols * sizeof(float);
    if (!ws || ws_bytes < need)
        return fail(TT_NORM_EWORKSPACE, "rmsnorm backward: workspace %zu B < required %zu B", ws_bytes, need);
    if (!aligned16(ws)) return fail(TT_NORM_EALIGN, "rmsnorm backward: workspace %p not 16-byte aligned", ws);
    st = dispatch<RmsOn<Map>::template Bwd>(dtype, gc, p, dx, ws, g, x, w, rstd, map, (int)cols, stream);
    if (st != TT_NORM_OK) return st;
    st = check_launch("rmsnorm backward launch");
    if (st != TT_NORM_OK) return st;
    return launch_colreduce(dw, nullptr, nullptr, (const float *)ws, 1, p.blocks_per_sample, cols, cols, dtype,
                            stream);
}

int anywidth_rmsnorm_backward(void *dx, void *dw, const void *g, const void *x, const void *w,
                              const float *rstd, int64_t rows, int64_t cols, int dtype, void *ws,
                              size_t ws_bytes, hipStream_t stream) {
    if (widerow_takes(cols, dtype))
        return widerow_rmsnorm_backward(dx, dw, g, x, w, rstd, rows, cols, dtype, ws, ws_bytes, stream);
    return rmsnorm_backward_on(dx, dw, g, x, w, rstd, DenseRows{rows}, rows, cols, dtype, ws, ws_bytes, stream);
}

int anywidth_rmsnorm_backward_strided(void *dx, void *dw, const void *g, const void *x, const void *w,
                                      const float *rstd, const Strided3Rows &map, int64_t cols, int dtype,
                                      void *ws, size_t ws_bytes, hipStream_t stream) {
    return rmsnorm_backward_on(dx, dw, g, x, w, rstd, map, map.n0 * map.n1 * map.n2, cols, dtype, ws, ws_bytes,
                               stream);
}

static SampleLayout layout_of(int64_t batch, int64_t rows_per_sample, bool seq_first) {
    return seq_first ? SampleLayout{1, batch} : SampleLayout{rows_per_sample, 1};
}

bool anywidth_wide_forms_supported(int64_t cols, int dtype) {
    if (!anywidth_supported(cols, dtype)) return false;
    // rows of up to six accesses per lane here; wider dense rows on the wide-row kernels
    return geometry_for(cols, dtype).chunks <= 6 || widerow_takes(cols, dtype);
}

template <bool GATED>
static int adaln_forward_any(void *out, float *mean, float *rstd, const void *x, const void *scale,
                             const void *shift, const AdalnExtra &ex, int64_t batch, int64_t rows_per_sample,
                             int64_t cols, double eps, int dtype, bool seq_first, hipStream_t stream) {
    if (rows_per_sample == 0) return TT_NORM_OK;
    const GeomChoice gc = geometry_for(cols, dtype);
    RowPlan p;
    int st = plan_for(&p, batch, rows_per_sample, gc, false);
    if (st != TT_NORM_OK) return st;
    st = dispatch<AdalnOn<GATED, false>::template Fwd>(dtype, gc, p, out, mean, rstd, x, scale, shift, ex, rows_per_sample,
                                                       layout_of(batch, rows_per_sample, seq_first), (int)cols, eps,
                                                       stream);
    return st != TT_NORM_OK ? st : check_launch("adaln forward launch");
}

int anywidth_adaln_forward(void *out, float *mean, float *rstd, const void *x, const void *scale,
                           const void *shift, int64_t batch, int64_t rows_per_sample, int64_t cols, double eps,
                           int dtype, hipStream_t stream, bool seq_first) {
    if (widerow_takes(cols, dtype))
        return widerow_adaln_forward(out, mean, rstd, x, scale, shift, batch, rows_per_sample, cols, eps, dtype, seq_first,
                                     stream);
    return adaln_forward_any<false>(out, mean, rstd, x, scale, shift, AdalnExtra{nullptr, nullptr, nullptr, nullptr},
                                    batch, rows_per_sample, cols, eps, dtype, seq_first, stream);
}

int anywidth_gated_adaln_forward(void *h2, void *out, float *mean, float *rstd, const void *h, const void *attn,
                                 const void *gate, const void *scale, const void *shift, int64_t batch,
                                 int64_t rows_per_sample, int64_t cols, double eps, int dtype, hipStream_t stream) {
    if (widerow_takes(cols, dtype))
        return widerow_gated_adaln_forward(h2, out, mean, rstd, h, attn, gate, scale, shift, batch, rows_per_sample, cols,
                                           eps, dtype, stream);
    return adaln_forward_any<true>(out, mean, rstd, h, scale, shift, AdalnExtra{h2, nullptr, attn, gate}, batch,
                                   rows_per_sample, cols, eps, dtype, false, stream);
}

size_t anywidth_adaln_backward_workspace_bytes(int64_t batch, int64_t rows_per_sample, int64_t cols, int dtype) {
    return backward_scratch(batch, rows_per_sample, cols, dtype, 2);
}

template <bool GATED, bool RES>
static int adaln_backward_any(void *dx, void *dscale, void *dshift, void *dgate, const void *g, const void *x,
                              const void *scale, const float *mean, const float *rstd, const AdalnExtra &ex,
                              int64_t batch, int64_t rows_per_sample, int64_t cols, int dtype, void *ws,
                              size_t ws_bytes, bool seq_first, hipStream_t stream) {
    constexpr int NSETS = GATED ? 3 : 2;
    if (rows_per_sample == 0)
        return launch_colreduce(dscale, dshift, dgate, nullptr, batch, 0, cols, NSETS * cols, dtype, stream);
    const GeomChoice gc = geometry_for(cols, dtype);
    RowPlan p;
    int st = plan_for(&p, batch, rows_per_sample, gc, true);
    if (st != TT_NORM_OK) return st;
    const size_t need = (size_t)p.blocks * NSETS * cols * sizeof(float);
    if (!ws || ws_bytes < need)
        return fail(TT_NORM_EWORKSPACE, "adaln backward: workspace %zu B < required %zu B", ws_bytes, need);
    if (!aligned16(ws)) return fail(TT_NORM_EALIGN, "adaln backward: workspace %p not 16-byte aligned", ws);
    st = dispatch<AdalnOn<GATED, RES>::template Bwd>(dtype, gc, p, dx, ws, g, x, scale, mean, rstd, ex, rows_per_sample,
                                                     layout_of(batch, rows_per_sample, seq_first), (int)cols, stream);
    if (st != TT_NORM_OK) return st;
    st = check_launch("adaln backward launch");
    if (st != TT_NORM_OK) return st;
    return launch_colreduce(dscale, dshift, dgate, (const float *)ws, batch, p.blocks_per_sample, cols, NSETS * cols,
                            dtype, stream);
}

int anywidth_adaln_backward(void *dx, void *dscale, void *dshift, const void *g, const void *x,
                            const void *scale, const float *mean, const float *rstd, int64_t batch,
                            int64_t rows_per_sample, int64_t cols, int dtype, void *ws, size_t ws_bytes,
                            hipStream_t stream, bool seq_first) {
    if (widerow_takes(cols, dtype))
        return widerow_adaln_backward(dx, dscale, dshift, g, x, scale, mean, rstd, batch, rows_per_sample, cols, dtype, ws,
                                      ws_bytes, seq_first, stream);
    return adaln_backward_any<false, false>(dx, dscale, dshift, nullptr, g, x, scale, mean, rstd,
                                            AdalnExtra{nullptr, nullptr, nullptr, nullptr}, batch, rows_per_sample, cols,
                                            dtype, ws, ws_bytes, seq_first, stream);
}

int anywidth_adaln_backward_residual(void *dx, void *dscale, void *dshift, const void *g, const void *dres,
                                     const void *x, const void *scale, const float *mean, const float *rstd,
                                     int64_t batch, int64_t rows_per_sample, int64_t cols, int dtype, void *ws,
                                     size_t ws_bytes, hipStream_t stream) {
    if (widerow_takes(cols, dtype))
        return widerow_adaln_backward_residual(dx, dscale, dshift, g, dres, x, scale, mean, rstd, batch, rows_per_sample,
                                               cols, dtype, ws, ws_bytes, stream);
    return adaln_backward_any<false, true>(dx, dscale, dshift, nullptr, g, x, scale, mean, rstd,
                                           AdalnExtra{nullptr, dres, nullptr, nullptr}, batch, rows_per_sample, cols, dtype,
                                           ws, ws_bytes, false, stream);
}

size_t anywidth_gated_adaln_backward_workspace_bytes(int64_t batch, int64_t rows_per_sample, int64_t cols, int dtype) {
    return backward_scratch(batch, rows_per_sample, cols, dtype, 3);
}

int anywidth_gated_adaln_backward(void *dh, void *dattn, void *dgate, void *dscale, void *dshift, const void *g,
                                  const void *dh2, const void *h2, const void *attn, const void *gate,
                                  const void *scale, const float *mean, const float *rstd, int64_t batch,
                                  int64_t rows_per_sample, int64_t cols, int dtype, void *ws, size_t ws_bytes,
                                  hipStream_t stream) {
    if (widerow_takes(cols, dtype))
        return widerow_gated_adaln_backward(dh, dattn, dgate, dscale, dshift, g, dh2, h2, attn, gate, scale, mean, rstd,
                                            batch, rows_per_sample, cols, dtype, ws, ws_bytes, stream);
    return adaln_backward_any<true, false>(dh, dscale, dshift, dgate, g, h2, scale, mean, rstd,
                                           AdalnExtra{dattn, dh2, attn, gate}, batch, rows_per_sample, cols, dtype, ws,
                                           ws_bytes, false, stream);
}

}  // namespace ttn
