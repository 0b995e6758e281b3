// Stand-alone IIR filter (the TritonIIR operator), forward or time reversed:
// one filter in parallel form (one scan pass), or a cascade of full biquads
// (all sections in one pass, iir_cascade_kernel).
#include <utility>

#include "iir.hpp"

namespace pesq {

template <bool kRev>
struct SingleMode {
    static constexpr int kInputs = 1;
    static constexpr int kOutputs = 1;
    static constexpr bool kRamp = false;
    static constexpr bool kReverse = kRev;
    static constexpr bool kAccumulates = false;
    static constexpr bool kSegments = false;
    static constexpr bool kObserver = true;
    using In = float;
    using Out = float;

    const float *x;
    float *y;
    int64_t len;

    __device__ __forceinline__ const float *src(int row, int) const { return x + int64_t(row) * len; }
    __device__ __forceinline__ float *dst(int row, int) const { return y + int64_t(row) * len; }
    __device__ __forceinline__ void inputs(double, const float *in, double &xa, double &xb) const {
        xa = in[0];
        xb = 0.0;
    }
    __device__ __forceinline__ void setup(int, double *, int) const {}
    __device__ __forceinline__ void compute(double, double ya, double, double &, const double *,
                                            float *out) const {
        out[0] = static_cast<float>(ya);
    }
    __device__ __forceinline__ void finish(int, int, double) const {}
};

template <int NS, bool kRev>
static int launch_single(const float *x, float *y, int64_t rows, int64_t len,
                         const IirTable *table, double *aggr, hipStream_t stream) {
    SingleMode<kRev> m{x, y, len};
    return launch_scan<NS, 0>(m, table, aggr, rows, len, true, true, stream);
}

template <bool kRev>
static int dispatch(int sections, const float *x, float *y, int64_t rows, int64_t len,
                    const IirTable *table, double *aggr, hipStream_t stream) {
    switch (sections) {
        case 1: return launch_single<1, kRev>(x, y, rows, len, table, aggr, stream);
        case 2: return launch_single<2, kRev>(x, y, rows, len, table, aggr, stream);
        case 3: return launch_single<3, kRev>(x, y, rows, len, table, aggr, stream);
        case 4: return launch_single<4, kRev>(x, y, rows, len, table, aggr, stream);
        case 5: return launch_single<5, kRev>(x, y, rows, len, table, aggr, stream);
        case 6: return launch_single<6, kRev>(x, y, rows, len, table, aggr, stream);
        case 7: return launch_single<7, kRev>(x, y, rows, len, table, aggr, stream);
        case 8: return launch_single<8, kRev>(x, y, rows, len, table, aggr, stream);
        default: break;
    }
    set_error("unsupported section count %d", sections);
    return PESQ_ERR_ARGUMENT;
}

// A cascade of one section: a full biquad through the scan kernels.
template <bool kRev>
struct BiquadMode {
    static constexpr int kInputs = 1;
    static constexpr int kOutputs = 1;
    static constexpr bool kRamp = false;
    static constexpr bool kReverse = kRev;
    static constexpr bool kAccumulates = false;
    static constexpr bool kSegments = false;
    static constexpr bool kObserver = true;
    using In = float;
    using Out = float;

    const float *x;
    float *y;
    int64_t len;

    __device__ __forceinline__ const float *src(int row, int) const { return x + int64_t(row) * len; }
    __device__ __forceinline__ float *dst(int row, int) const { return y + int64_t(row) * len; }
    __device__ __forceinline__ void inputs(double, const float *in, double &xa, double &xb) const {
        xa = static_cast<double>(in[0]);
        xb = 0.0;
    }
    __device__ __forceinline__ void setup(int, double *, int) const {}
    __device__ __forceinline__ void compute(double, double ya, double, double &, const double *,
                                            float *out) const {
        out[0] = static_cast<float>(ya);
    }
    __device__ __forceinline__ void finish(int, int, double) const {}
};

// --------------------------------------------------------------------------
// Cascades of two and more biquads.
//
// A wavefront holds a block of kSegmentSpan samples of a row, 32 per lane as
// doubles, and runs the sections over it one after the other: each section's
// chunk end states (4 operations per sample), their scan over the lanes and the
// recursion (5 per sample), whose outputs are the next section's inputs,
// so no signal between the sections leaves the registers.  A block's start
// states (two per section) depend on the row's earlier blocks through all
// sections before them, so rows of more than one block take three launches:
// the blocks run from zero states (kOutput false) to their end states, a
// workgroup per row carries these over the row (s_(b+1) = T s_b + e_(b+1), T the
// cascade's transfer over a block), and the blocks run again from their true
// starts.  The blocks of a row do not depend on the other rows: a row's result
// is the same in any batch.
//
// Bound by issue and the sections' serial chains: 345 VALU instructions per
// section and 2048 samples in the states pass, 383 in the output pass.  One scan pass per
// section, with float64 signals through memory between them, took 445
// us for 8 sections over 24 rows of 160001 samples, forward and adjoint; this
// form takes 119 us with the host's share (states 18, starts 12, output 24 us per
// direction).
// --------------------------------------------------------------------------
struct CascadeArgs {
    const float *x;
    float *y;
    const IirTable *tables;
    double *states;  // [rows][blocks][2 sections]: end states of the block before, then starts
    int64_t rows, len;
    int sections, blocks;
};

template <bool kRev, bool kOutput>
__global__ void __launch_bounds__(kSegmentWaves *kWave, 3) iir_cascade_kernel(CascadeArgs a) {
    extern __shared__ double powers[];  // [section][kCarryPowers][4]: A^(kSegmentChunk m)
    __shared__ __attribute__((aligned(16))) float stages[kSegmentWaves][kStageFloats];
    const int wave = wave_index();
    const int lane = static_cast<int>(threadIdx.x) % kWave;
    // the states pass has nothing to do for a row's last block
    const int per_row = kOutput ? a.blocks : a.blocks - 1;
    const int64_t id = int64_t(blockIdx.x) * kSegmentWaves + wave;
    const bool live = id < a.rows * per_row;
    const int64_t row = live ? id / per_row : 0;
    const int blk = live ? static_cast<int>(id - row * per_row) : 0;
    const float *src = a.x + row * a.len;
    const int64_t lo = segment_lo<kRev>(blk, a.len);
    Vec4 raw[kSegmentChunk / 4];
    if (segment_full(lo, a.len)) segment_load(src + lo, lane, raw);
    for (int i = threadIdx.x; i < a.sections * kCarryPowers; i += kSegmentWaves * kWave) {
        const int k = i / kCarryPowers, power = i - k * kCarryPowers;
        const IirTable &t = a.tables[k];
        const double *p = power < kWave / 2 ? t.lane_pw[0][2 * power] : t.pw[kLevelBlock][0];
#pragma unroll
        for (int e = 0; e < 4; ++e) powers[4 * i + e] = p[e];
    }
    __syncthreads();
    if (!live) return;  // whole wavefronts; no barrier follows
    float *stage = stages[wave];
    float *own = stage + (kRev ? kWave - 1 - lane : lane) * kStageChunk;
    stage_in(stage, raw, src, lo, a.len, lane);
    wave_lds_fence();
    double y[kSegmentChunk];
#pragma unroll
    for (int g = 0; g < kSegmentChunk / 4; ++g) {
        float v[4];
        chunk_read<kRev>(own, g, v);
#pragma unroll
        for (int i = 0; i < 4; ++i) y[4 * g + i] = static_cast<double>(v[i]);
    }
    double *states = a.states + (row * a.blocks + blk) * 2 * a.sections;
    const double *c5 = powers + 4 * ((lane & 15) + 1);
    const double *c6 = powers + 4 * (lane >= 32 ? lane - 31 : 0);
#pragma unroll 1
    for (int k = 0; k < a.sections; ++k) {
        const ConstDoubles pw = (ConstDoubles)(&a.tables[k].pw[0][0][0]);
        Coeffs<0, 1, true> c;
        c.load_scalar(a.tables[k], a.tables[k].c0a);
        Bank<1> z;
        z.zero();
#pragma unroll
        for (int i = 0; i < kSegmentChunk; ++i) c.advance(z, y[i]);
        double pu = 0.0, pv = 0.0;  // the block's start state
        if constexpr (kOutput) {
            if (blk > 0) {
                pu = states[2 * k];
                pv = states[2 * k + 1];
            }
            const ConstDoubles q = scan_powers(pw, 0, 0);
            const double fu = lane == 0 ? pu : 0.0, fv = lane == 0 ? pv : 0.0;
            z.u[0] = fma(q[0], fu, fma(q[1], fv, z.u[0]));
            z.v[0] = fma(q[2], fu, fma(q[3], fv, z.v[0]));
        }
        using std::integral_constant;
        auto level = [&](auto ctrl, int j) {
            const ConstDoubles q = scan_powers(pw, j, 0);
            const double ou = dpp_move<decltype(ctrl)::value, 0xF>(z.u[0]);
            const double ov = dpp_move<decltype(ctrl)::value, 0xF>(z.v[0]);
            z.u[0] = fma(q[0], ou, fma(q[1], ov, z.u[0]));
            z.v[0] = fma(q[2], ou, fma(q[3], ov, z.v[0]));
        };
        level(integral_constant<int, 0x111>{}, 0);
        level(integral_constant<int, 0x112>{}, 1);
        level(integral_constant<int, 0x114>{}, 2);
        level(integral_constant<int, 0x118>{}, 3);
        auto carry_level = [&](auto ctrl, auto mask, const double *p) {
            const double2 q0 = *reinterpret_cast<const double2 *>(p + 4 * kCarryPowers * k);
            const double2 q1 = *reinterpret_cast<const double2 *>(p + 4 * kCarryPowers * k + 2);
            const double ou = dpp_move<decltype(ctrl)::value, decltype(mask)::value>(z.u[0]);
            const double ov = dpp_move<decltype(ctrl)::value, decltype(mask)::value>(z.v[0]);
            z.u[0] = fma(q0.x, ou, fma(q0.y, ov, z.u[0]));
            z.v[0] = fma(q1.x, ou, fma(q1.y, ov, z.v[0]));
        };
        carry_level(integral_constant<int, 0x142>{}, integral_constant<int, 0xA>{}, c5);
        carry_level(integral_constant<int, 0x143>{}, integral_constant<int, 0xC>{}, c6);
        if constexpr (!kOutput) {
            // the block's end state, where the next block's start will stand
            if (lane == kWave - 1) {
                states[2 * a.sections + 2 * k] = z.u[0];
                states[2 * a.sections + 2 * k + 1] = z.v[0];
            }
            if (k + 1 == a.sections) return;
        }
        Bank<1> s;
        const double before_u = dpp_move<0x138, 0xF>(z.u[0]);  // wave_shr:1, all lanes active
        const double before_v = dpp_move<0x138, 0xF>(z.v[0]);
        s.u[0] = lane == 0 ? pu : before_u;
        s.v[0] = lane == 0 ? pv : before_v;
#pragma unroll
        for (int i = 0; i < kSegmentChunk; ++i) y[i] = c.step(s, y[i]);
    }
    if constexpr (kOutput) {
#pragma unroll
        for (int g = 0; g < kSegmentChunk / 4; ++g) {
            float v[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) v[i] = static_cast<float>(y[4 * g + i]);
            chunk_write<kRev>(own, g, v);
        }
        wave_lds_fence();
        stage_out(a.y + row * a.len, stage, lo, a.len, lane);
    }
}

// Start states of a row's blocks from the end states of the blocks before
// them, in place, one workgroup per row: s_(b+1) = T s_b + e_(b+1).  The steps are
// serial, so a long row is shared out (StartsPlan): a group of lanes carries the
// blocks of its share from a zero state, the states at the shares' first blocks
// follow from those ends with T^per = (T^(8^level))^hops, and each group carries
// its blocks again from its true start.
//
// Lane i of a group holds row i of T (kN >= 2 sections columns, zero past them)
// and state i, which the others take by lane broadcasts: groups of 16 lanes, four
// shares per wavefront, up to 8 sections, else a wavefront per share.  The end
// states of kStartsGroup blocks are loaded while the ones before them are
// carried.  Bound by the issue of the steps on one CU, about 0.1 us each, and 6 us
// of loads.  1 row of 2880000 samples (1407 blocks), 2 sections: 18.3 us, the
// filter 38 (170 with one wavefront carrying every block of the row, 48 with a
// scan per section); 1 row of 960000, 8 sections: 24.6 us, the filter 54 (104,
// 100).
constexpr int kStartsGroup = 16;  // blocks carried without a branch; divides per

struct StartsPlan {
    int shares, per;  // blocks of a share (the last one's may be fewer)
    int level, hops;  // per = hops 8^level
};

// The plan of fewest serial steps: a share's blocks twice, and hops for every
// share before the last.
static StartsPlan starts_plan(int blocks, int most) {
    const int count = blocks - 1;
    StartsPlan best{1, count, 0, count};
    int cost = count - 8;  // the shared form's barrier and loads of T
    for (int level = 0, unit = 1; level < kCascadeLevels; ++level, unit *= 8) {
        const int quantum = unit < kStartsGroup ? kStartsGroup / unit : 1;
        int hops = (count + most * unit - 1) / (most * unit);
        hops = (hops + quantum - 1) / quantum * quantum;
        const int per = hops * unit, shares = (count + per - 1) / per;
        if (2 * per + (shares - 1) * hops < cost) {
            cost = 2 * per + (shares - 1) * hops;
            best = {shares, per, level, hops};
        }
    }
    return best;
}

// lane j of the lane's group (of 16: DPP row_newbcast, or of the whole wavefront)
template <int kLanes, int j>
__device__ __forceinline__ double group_lane(double v) {
    if constexpr (kLanes == 16) return dpp_move<0x150 + j, 0xF>(v);
    return read_lane(v, j);
}
// e + sum_j t[j] (v of the group's lane j)
template <int kLanes, int kN, int... j>
__device__ __forceinline__ double group_product(const double (&t)[kN], double v, double e,
                                                std::integer_sequence<int, j...>) {
    double acc[4] = {e, 0.0, 0.0, 0.0};
    ((acc[j % 4] = fma(t[j], group_lane<kLanes, j>(v), acc[j % 4])), ...);
    return (acc[0] + acc[1]) + (acc[2] + acc[3]);
}

template <int kN>
struct Starts {
    static constexpr int kLanes = kN <= 16 ? 16 : kWave;     // of a share
    static constexpr int kPerWave = kWave / kLanes;          // shares
    static constexpr int kWaves = 8;                         // at most, by registers
};

template <int kN>
__global__ void __launch_bounds__(kWave *Starts<kN>::kWaves)
    iir_cascade_starts_kernel(CascadeArgs a, StartsPlan plan) {
    using S = Starts<kN>;
    __shared__ double ends[S::kWaves * kWave];
    static_assert(kN >= 4 && kN <= S::kLanes, "a lane per state");
    const int n = 2 * a.sections;
    const int lane = static_cast<int>(threadIdx.x) % S::kLanes;
    const int share = static_cast<int>(threadIdx.x) / S::kLanes;
    const bool mine = lane < n && share < plan.shares;
    const int at = lane < n ? lane : 0;
    double t[kN];
    auto transfer = [&](int level) {
#pragma unroll
        for (int j = 0; j < kN; ++j) {
            const double v = a.tables[at / 2].cascade[level][at % 2][j];
            t[j] = lane < n && j < n ? v : 0.0;
        }
    };
    // T state + e, state j broadcast to the group
    auto carry = [&](double state, double e) {
        return group_product<S::kLanes>(t, state, e, std::make_integer_sequence<int, kN>{});
    };
    const int first = 1 + share * plan.per;
    const int left = a.blocks - first;  // (at most 0 past the shares)
    const int count = plan.per < left ? plan.per : left;
    double *row = a.states + int64_t(blockIdx.x) * a.blocks * n + at;
    auto load = [&](int b0, double (&e)[kStartsGroup]) {
#pragma unroll
        for (int q = 0; q < kStartsGroup; ++q) {
            // (past the shares count <= 0: the row's last block)
            e[q] = row[int64_t(first + (b0 + q < count ? b0 + q : count - 1)) * n];
        }
    };
    // a share's blocks from `state`: the state after them (of a whole share)
    auto run = [&](double state, auto written) {
        double e[kStartsGroup], next[kStartsGroup];
        load(0, e);
        for (int b0 = 0; b0 < plan.per; b0 += kStartsGroup) {
            load(b0 + kStartsGroup, next);
#pragma unroll
            for (int q = 0; q < kStartsGroup; ++q) {
                state = carry(state, mine ? e[q] : 0.0);
                if constexpr (decltype(written)::value) {
                    if (mine && b0 + q < count) row[int64_t(first + b0 + q) * n] = state;
                }
                e[q] = next[q];
            }
        }
        return state;
    };
    transfer(0);
    double start = 0.0;
    if (plan.shares > 1) {  // uniform over the grid
        ends[threadIdx.x] = run(0.0, std::false_type{});
        __syncthreads();
        transfer(plan.level);
        for (int s = 0; s + 1 < plan.shares; ++s) {
            const double e = ends[s * S::kLanes + lane];
            double v = start;
            for (int h = 1; h < plan.hops; ++h) v = carry(v, 0.0);
            v = carry(v, e);
            start = s < share ? v : start;
        }
        transfer(0);
    }
    run(start, std::true_type{});
}

template <int kN>
static void launch_starts(const CascadeArgs &a, hipStream_t stream) {
    using S = Starts<kN>;
    const StartsPlan plan = starts_plan(a.blocks, S::kWaves * S::kPerWave);
    const int waves = static_cast<int>(cdiv(plan.shares, int64_t(S::kPerWave)));
    hipLaunchKernelGGL(iir_cascade_starts_kernel<kN>, dim3(static_cast<unsigned>(a.rows)),
                       dim3(kWave * waves), 0, stream, a, plan);
}

template <bool kRev>
static int cascade(const float *x, float *y, int64_t rows, int64_t len, const IirTable *tables,
                   int count, double *workspace, hipStream_t stream) {
    if (count == 1) {
        BiquadMode<kRev> m{x, y, len};
        return launch_scan<1, 0>(m, tables, workspace, rows, len, true, true, stream);
    }
    CascadeArgs a{x, y, tables, workspace, rows, len, count,
                  static_cast<int>(cdiv(len, kSegmentSpan))};
    const size_t lds = size_t(count) * kCarryPowers * 4 * sizeof(double);
    const dim3 block(kSegmentWaves * kWave);
    auto groups = [&](int64_t per_row) {
        return dim3(static_cast<unsigned>(cdiv(rows * per_row, kSegmentWaves)));
    };
    if (a.blocks > 1) {
        hipLaunchKernelGGL((iir_cascade_kernel<kRev, false>), groups(a.blocks - 1), block, lds,
                           stream, a);
        PESQ_CHECK_LAUNCH("iir cascade states");
        if (count <= 2) {
            launch_starts<4>(a, stream);
        } else if (count <= 4) {
            launch_starts<8>(a, stream);
        } else if (count <= 8) {
            launch_starts<16>(a, stream);
        } else if (count <= 16) {
            launch_starts<32>(a, stream);
        } else {
            launch_starts<64>(a, stream);
        }
        PESQ_CHECK_LAUNCH("iir cascade starts");
    }
    hipLaunchKernelGGL((iir_cascade_kernel<kRev, true>), groups(a.blocks), block, lds, stream, a);
    PESQ_CHECK_LAUNCH("iir cascade output");
    return PESQ_OK;
}

// doubles of the workspace that hold the states
static int64_t cascade_state_doubles(int64_t rows, int64_t len, int sections) {
    const int64_t blocks = cdiv(len, kSegmentSpan);
    return sections > 1 && blocks > 1 ? rows * blocks * 2 * sections : 0;
}

}  // namespace pesq

using namespace pesq;

extern "C" int pesq_iir_cascade_workspace(int64_t rows, int64_t len, int sections,
                                          size_t *bytes) {
    PESQ_CHECK_ARG(rows >= 0 && len >= 0 && bytes != nullptr, "invalid sizes");
    PESQ_CHECK_ARG(sections >= 1 && sections <= PESQ_IIR_MAX_CASCADE,
                   "a cascade has 1..%d sections", PESQ_IIR_MAX_CASCADE);
    const int64_t nblk = cdiv(len, kBlockSpan);
    PESQ_CHECK_ARG(rows * nblk < (int64_t(1) << 31), "too many rows x blocks for one launch");
    const int64_t mid = sections == 1 ? 0 : (sections == 2 ? 1 : 2) * rows * len;
    const int64_t size = scan_workspace_doubles(rows, nblk, 1) + mid;
    const int64_t states = cascade_state_doubles(rows, len, sections);
    *bytes = size_t(size > states ? size : states) * sizeof(double);
    return PESQ_OK;
}

extern "C" int pesq_iir_cascade_apply(const float *x, float *y, int64_t rows, int64_t len,
                                      const void *cascade_tables, int sections, int reverse,
                                      void *workspace, hipStream_t stream) {
    PESQ_CHECK_ARG(x && y && cascade_tables && workspace, "null pointer argument");
    PESQ_CHECK_ARG(rows >= 0 && len >= 0, "invalid sizes");
    PESQ_CHECK_ARG(sections >= 1 && sections <= PESQ_IIR_MAX_CASCADE,
                   "a cascade has 1..%d sections", PESQ_IIR_MAX_CASCADE);
    if (rows == 0 || len == 0) return PESQ_OK;
    const int64_t nblk = cdiv(len, kBlockSpan);
    PESQ_CHECK_ARG(rows * nblk < (int64_t(1) << 31), "too many rows x blocks for one launch");
    const IirTable *tables = static_cast<const IirTable *>(cascade_tables);
    double *ws = static_cast<double *>(workspace);
    return reverse ? cascade<true>(x, y, rows, len, tables, sections, ws, stream)
                   : cascade<false>(x, y, rows, len, tables, sections, ws, stream);
}

extern "C" int pesq_iir_workspace(int64_t rows, int64_t len, size_t *bytes) {
    PESQ_CHECK_ARG(rows >= 0 && len >= 0 && bytes != nullptr, "invalid sizes");
    const int64_t nblk = cdiv(len, kBlockSpan);
    PESQ_CHECK_ARG(rows * nblk < (int64_t(1) << 31), "too many rows x blocks for one launch");
    *bytes = size_t(scan_workspace_doubles(rows, nblk)) * sizeof(double);
    return PESQ_OK;
}

// The kernels are compiled per section count; the caller packed the table and
// passes its section count, so no device memory is read on the host.
extern "C" int pesq_iir_apply(const float *x, float *y, int64_t rows, int64_t len,
                                const void *iir_table, int sections, int reverse,
                                void *workspace, hipStream_t stream) {
    PESQ_CHECK_ARG(x && y && iir_table && workspace, "null pointer argument");
    PESQ_CHECK_ARG(rows >= 0 && len >= 0, "invalid sizes");
    if (rows == 0 || len == 0) return PESQ_OK;
    PESQ_CHECK_ARG(rows * cdiv(len, kBlockSpan) < (int64_t(1) << 31),
                   "too many rows x blocks for one launch");
    const IirTable *table = static_cast<const IirTable *>(iir_table);
    double *aggr = static_cast<double *>(workspace);
    return reverse ? dispatch<true>(sections, x, y, rows, len, table, aggr, stream)
                   : dispatch<false>(sections, x, y, rows, len, table, aggr, stream);
}
