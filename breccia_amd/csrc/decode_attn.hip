// Paged decode attention for gfx950: what the split-K kernels of decode_attn_mfma.hip share -- the
// cut of a batch into work-groups, the merge kernel, the launch.  Together they replace the
// reference's four dispatches (scores -> softmax -> split apply -> reduce:
// crates/breccia-kernels/shaders/qsa_attn_scores_small.comp, ops_softmax.comp,
// qsa_attn_apply_split.comp, qsa_attn_apply_reduce.comp) and must agree with its f64 CPU attend
// (crates/breccia-kernels/src/qsa/cpu.rs:197-246).
//
// Shape of the work: for one (sequence, kv head) every K row and V row is read once and used by
// all q heads of the group -- an HBM-bound stream.  A work-group of four waves owns one (entry, kv
// head, page range); a wave owns whole pages (16 cells); the four waves' running (m, l, O) are
// folded in LDS and written as one partial per work-group; the merge kernel combines the page
// ranges of a head and applies sigmoid(gate).
#include <atomic>
#include <type_traits>

#include "decode_attn_common.hpp"
#include "gate.hpp"
#include "lane_groups.hpp"

namespace bkv {

namespace {

struct MergeParams {
    const AttnBatch* bd;  // DESC: the batch is read from this device-resident copy
    const float* part_o;
    const float* part_ml;
    const float* gate;
    float* out;
    int64_t gate_seq_stride, gate_head_stride;
    int32_t n_kv, n_q, group;
    uint32_t inv_group16;  // small_divisor_inverse(group)
};
// What the merge needs of a batch, as an argument (kFewEntries: why there are two).
template <int N>
struct MergeArgs : MergeParams {
    int32_t splits[N], wg_base[N];
};
template <int N>
static MergeArgs<N> merge_args(const MergeParams& mp, const AttnBatch& b) {
    MergeArgs<N> args{};
    static_cast<MergeParams&>(args) = mp;
    for (int i = 0; i < b.n; ++i) {
        args.splits[i] = b.splits[i];
        args.wg_base[i] = b.wg_base[i];
    }
    return args;
}

constexpr int kMergeWaves = 4;
constexpr int kMergeCols = 64;                  // columns of a work-group
constexpr int kMergeGroups = kMergeWaves * 4;   // 16 lanes, 4 columns each, sum splits i, i + kMergeGroups, ...
constexpr int kMergeInFlight = 6;               // partial rows a lane requests at most per round

// A lane's share of a head: splits at, at + kMergeGroups, ... under a maximum of its own.
struct MergeSum {
    f4 o = f4{0.0f, 0.0f, 0.0f, 0.0f};
    float l = 0.0f, m = -INFINITY;
};
// exp2(x - ref), and 0 where nothing has been attended yet (both -inf)
__device__ __forceinline__ float weight_of(float x, float ref) { return __builtin_amdgcn_exp2f(x - (ref == -INFINITY ? 0.0f : ref)); }

// N rounds of kMergeGroups splits from split s0 on, everything requested before the first use and without branches:
// past the end the last split is requested again and counts as zeros (not by its weight alone: 0 x inf is NaN).
template <int N>
__device__ __forceinline__ void merge_rounds(const float* po, const float* pml, uint32_t lane_at, uint32_t ostride, uint32_t mlstride, int s0, int splits,
                                             MergeSum& a) {
    float m[N], l[N];
    f4 v[N];
#pragma unroll
    for (int u = 0; u < N; ++u) {
        const uint32_t s = (uint32_t)min(s0 + u * kMergeGroups, splits - 1);
        const float2 ml = *reinterpret_cast<const float2*>(pml + s * mlstride);
        m[u] = ml.x, l[u] = ml.y;
    }
#pragma unroll
    for (int u = 0; u < N; ++u) {
        const uint32_t s = (uint32_t)min(s0 + u * kMergeGroups, splits - 1);
        v[u] = *reinterpret_cast<const f4*>(po + (s * ostride + lane_at));
    }
    __builtin_amdgcn_sched_barrier(0);
    float mx = a.m;
#pragma unroll
    for (int u = 0; u < N; ++u) {
        const bool mine = s0 + u * kMergeGroups < splits;
        m[u] = mine ? m[u] : -INFINITY;
        l[u] = mine ? l[u] : 0.0f;
        v[u] = mine ? v[u] : f4{0.0f, 0.0f, 0.0f, 0.0f};
        mx = fmaxf(mx, m[u]);
    }
    const float keep = weight_of(a.m, mx);
    a.o *= keep;
    a.l *= keep;
    a.m = mx;
#pragma unroll
    for (int u = 0; u < N; ++u) {
        const float f = weight_of(m[u], mx);
        a.o += v[u] * f;
        a.l = fmaf(f, l[u], a.l);
    }
}

// One work-group per (entry, q head, quarter of the columns).  The kernel is a chain of trips -- arguments, partial
// results, output -- and what stands between them.  Every 16 lanes keep a maximum of their own and everything meets once,
// at the end, and a quarter of a head is what one compute unit takes in a quarter of the time (64 bytes a clock).  Against a
// work-group of 16 waves a head, (m, l) staged in LDS and the maximum agreed ahead of the sums, a launch in a kernel trace
// takes 3.1 us instead of 4.2 for one sequence of 4096 cells (65 splits), 3.0 instead of 3.9 for four of up to 2048; for
// eight of up to 32k it takes 4.6 as before.
// N: entries of the batch in the arguments, 0: the batch is in device memory (DESC).
template <int N>
__global__ __launch_bounds__(64 * kMergeWaves) void decode_attn_merge_kernel(const std::conditional_t<N == 0, MergeParams, MergeArgs<N>> P) {
    constexpr bool DESC = N == 0;
    __shared__ __attribute__((aligned(16))) float red[kMergeWaves][kMergeCols];
    __shared__ __attribute__((aligned(16))) float red_m[kMergeWaves], red_l[kMergeWaves];
    // grid (q heads x quarters, entries): no division at the head of a kernel that is all latency, and every argument
    // is asked for at once
    const int e = blockIdx.y;
    const int h = blockIdx.x / (kHd / kMergeCols);
    const int col = blockIdx.x % (kHd / kMergeCols) * kMergeCols;
    int splits, base;
    if constexpr (DESC) {
        const batch_desc_ptr D = (batch_desc_ptr)(uintptr_t)P.bd;
        splits = D->splits[e];
        base = D->wg_base[e];
    } else {
        splits = P.splits[e];
        base = P.wg_base[e];
    }
    asm volatile("" ::"s"(splits), "s"(base), "s"(P.part_o), "s"(P.part_ml), "s"(P.gate), "s"(P.out), "s"(P.gate_seq_stride), "s"(P.gate_head_stride),
                 "s"(P.n_kv), "s"(P.n_q), "s"(P.group), "s"(P.inv_group16));
    const int kvh = small_div(h, P.inv_group16);
    const int hl = h - kvh * P.group;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    // the gate of the element this thread writes at the end is requested with the partial rows, not after
    // the sums (a trip to memory at the tail of a kernel that is all latency)
    float gt = 0.0f;
    if (P.gate && wave == 0) gt = P.gate[(size_t)e * P.gate_seq_stride + (size_t)h * P.gate_head_stride + col + lane];
    const size_t head = ((size_t)(base + kvh) * P.group + hl);  // the first split's row
    // floats between consecutive splits; the workspace is 33.6 MB, 32 bits hold any offset in it
    const uint32_t ostride = (uint32_t)(P.n_kv * P.group * kHd), mlstride = (uint32_t)(P.n_kv * P.group * 2);
    static_assert((uint64_t)kMaxWgs * 8 * kHd * sizeof(float) < (1ull << 32), "32-bit offsets");
    const float* const po = P.part_o + head * kHd + col;
    const float* const pml = P.part_ml + head * 2;
    const uint32_t lane_at = 4u * (uint32_t)(lane & 15);
    const int at = threadIdx.x >> 4;
    MergeSum a;
    const auto rounds = [&](auto n, int s0) { merge_rounds<decltype(n)::value>(po, pml, lane_at, ostride, mlstride, s0, splits, a); };
    if (splits <= kMergeGroups) {
        rounds(std::integral_constant<int, 1>(), at);
    } else if (splits <= 2 * kMergeGroups) {
        rounds(std::integral_constant<int, 2>(), at);
    } else if (splits <= 4 * kMergeGroups) {
        rounds(std::integral_constant<int, 4>(), at);
    } else {
        for (int s0 = 0; s0 < splits; s0 += kMergeInFlight * kMergeGroups) rounds(std::integral_constant<int, kMergeInFlight>(), s0 + at);
    }
    // the four 16-lane groups of a wave, then the waves
    const float m_wave = max_over_lane_groups(a.m);
    const float f = weight_of(a.m, m_wave);
    f4 o;
#pragma unroll
    for (int k = 0; k < 4; ++k) o[k] = sum_over_lane_groups(a.o[k] * f);
    const float l_wave = sum_over_lane_groups(a.l * f);
    if (lane < 16) *reinterpret_cast<f4*>(&red[wave][4 * lane]) = o;
    if (lane == 0) {
        red_m[wave] = m_wave;
        red_l[wave] = l_wave;
    }
    __syncthreads();
    if (wave != 0) return;
    const f4 m = *reinterpret_cast<const f4*>(red_m), l = *reinterpret_cast<const f4*>(red_l);
    const float mx = fmaxf(fmaxf(m[0], m[1]), fmaxf(m[2], m[3]));
    float r = 0.0f, lt = 0.0f;
#pragma unroll
    for (int w = 0; w < kMergeWaves; ++w) {
        const float fw = weight_of(m[w], mx);
        r = fmaf(red[w][lane], fw, r);
        lt = fmaf(l[w], fw, lt);
    }
    r = lt > 0.0f ? r / lt : 0.0f;
    if (P.gate) r *= sigmoid(gt);
    P.out[((size_t)e * P.n_q + h) * kHd + col + lane] = r;
}

}  // namespace

// The limits a plan of this pool geometry works under.  The partial-result workspace holds
// max_wgs x 8 head rows and a work-group writes `group` of them.
AttnPlanLimits attn_plan_limits(int32_t n_cu, int32_t max_wgs, int32_t n_kv, int32_t group) {
    AttnPlanLimits lim;
    lim.per_page = n_kv;
    lim.gran = kWaves;
    // All work-groups should be resident at once (one generation): a handful of left-over
    // work-groups would run alone after the rest and double the kernel's time.  Two work-groups
    // fit a compute unit (registers and LDS of the kernels).
    lim.target = (n_cu > 0 ? n_cu : 256) * 2;
    lim.max_wgs = group > 8 ? (int32_t)((int64_t)max_wgs * 8 / group) : max_wgs;
    return lim;
}

int32_t plan_attn(const bkv_pool* p, int32_t n_q_head, AttnBatch& b, int32_t sel_groups, int32_t max_wgs) {
    const AttnPlanLimits lim =
        attn_plan_limits(p->n_cu, max_wgs > 0 ? max_wgs : p->max_wgs, p->g.n_kv, n_q_head / p->g.n_kv);
    return plan_attn_ranges(lim, kPage, sel_groups, b);
}

// ---- partial results without an allocation -----------------------------------------------------
// For callers that may not allocate device memory (a stream under capture, a tight serving loop):
// the split-K partials of bkv_decode_attn_static live in this array, one copy per GPU, held from
// the moment the library is loaded until the process ends.  Host code never uses the array's name
// as an address: each device's copy has its own address, looked up once per device below.
struct AttnStaticScratch {
    float o[(size_t)kStaticWgs * 8 * kHd];
    float ml[(size_t)kStaticWgs * 8 * 2];
};
static __device__ __align__(256) unsigned char scratch[sizeof(AttnStaticScratch)];

constexpr int kMaxDevices = 64;
// One address per device, looked up once; pools may be created from several threads at once, so the
// table is atomic (two threads that race on one device store the same address).
static std::atomic<void*> g_scratch_ptr[kMaxDevices];

// Makes `device` current for the lookup (every GPU holds its own copy of the array at its own
// address) and restores the caller's device afterwards.
hipError_t attn_static_scratch_init(int device) {
    if (device < 0 || device >= kMaxDevices) return hipErrorInvalidDevice;
    if (g_scratch_ptr[device].load(std::memory_order_acquire)) return hipSuccess;
    int current = -1;
    hipError_t e = hipGetDevice(&current);
    if (e != hipSuccess) return e;
    if (current != device) {
        e = hipSetDevice(device);
        if (e != hipSuccess) return e;
    }
    void* ptr = nullptr;
    e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
    if (current != device) {
        const hipError_t back = hipSetDevice(current);
        if (e == hipSuccess) e = back;
    }
    if (e != hipSuccess) return e;
    g_scratch_ptr[device].store(ptr, std::memory_order_release);
    return hipSuccess;
}

bool attn_static_scratch(int device, float** o, float** ml) {
    if (device < 0 || device >= kMaxDevices) return false;
    void* ptr = g_scratch_ptr[device].load(std::memory_order_acquire);
    if (!ptr) return false;
    AttnStaticScratch* s = static_cast<AttnStaticScratch*>(ptr);
    *o = s->o;
    *ml = s->ml;
    return true;
}

hipError_t launch_decode_attn(bkv_pool* p, int32_t layer, const AttnBatch& b, const AttnArgs& a,
                              hipStream_t stream) {
    const int32_t n_kv = p->g.n_kv;
    const int32_t group = a.n_q_head / n_kv;
    AttnKernelParams kp;
    kp.bd = a.desc;
    kp.kpool = p->k_layer[(size_t)layer];
    kp.vpool = p->v_layer[(size_t)layer];
    kp.tables = p->table_dev;
    kp.q = a.q;
    kp.part_o = a.ws_o ? a.ws_o : p->part_o;
    kp.part_ml = a.ws_ml ? a.ws_ml : p->part_ml;
    kp.max_pages_per_seq = p->desc.max_pages_per_seq;
    kp.n_kv = n_kv;
    kp.n_q = a.n_q_head;
    kp.group = group;
    kp.inv_kv16 = small_divisor_inverse(n_kv);
    kp.scale_log2e = a.scale * kLog2e;
    kp.ids = a.ids;
    kp.counts = a.counts;
    kp.id_stride = a.id_stride;
    kp.max_ids = a.max_ids;
    kp.new_k = a.new_k;
    kp.new_v = a.new_v;
    kp.kpool_w = p->k_layer[(size_t)layer];
    kp.vpool_w = p->v_layer[(size_t)layer];
    const bool sel = a.ids != nullptr;
    const bool step = a.new_k != nullptr;
    const int32_t total = a.desc ? a.desc_grid : b.wg_base[b.n];
    // one work-group per unit, every head of the kv head in it; while the pool times its kernels,
    // the events ride on the dispatch
    hipEvent_t ev_start = nullptr, ev_stop = nullptr;
    if (a.timed) (void)timer_dispatch_events(p, BKV_STAGE_ATTN_SPLIT, &ev_start, &ev_stop);
    hipError_t err = launch_decode_attn_mfma(kp, b, p->g.layout, step, sel, total, stream, ev_start, ev_stop);
    if (err != hipSuccess) return err;
    MergeParams mp;
    mp.bd = a.desc;
    mp.part_o = kp.part_o;
    mp.part_ml = kp.part_ml;
    mp.gate = a.gate;
    mp.out = a.out;
    mp.gate_seq_stride = a.gate_seq_stride;
    mp.gate_head_stride = a.gate_head_stride;
    mp.n_kv = n_kv;
    mp.n_q = a.n_q_head;
    mp.group = group;
    mp.inv_group16 = small_divisor_inverse(group);
    const dim3 mgrid((unsigned)a.n_q_head * (kHd / kMergeCols), (unsigned)b.n), mblock(64 * kMergeWaves);
    const auto merge = [&](auto kernel, const auto& args) {
        if (a.timed && !a.desc)
            launch_staged(p, BKV_STAGE_ATTN_MERGE, kernel, mgrid, mblock, 0, stream, args);
        else
            hipLaunchKernelGGL(kernel, mgrid, mblock, 0, stream, args);
    };
    if (a.desc) merge(decode_attn_merge_kernel<0>, mp);
    else if (b.n <= kFewEntries) merge(decode_attn_merge_kernel<kFewEntries>, merge_args<kFewEntries>(mp, b));
    else merge(decode_attn_merge_kernel<kMaxBatch>, merge_args<kMaxBatch>(mp, b));
    return hipGetLastError();
}

// ---- a decode step that re-plans itself on the device ------------------------------------------
// One wave, lane i = entry i: every entry moves on by one cell and the batch is cut again with the
// arithmetic of plan_attn_ranges (attn_plan.hpp) -- the sums and the running offsets as wave
// reductions -- so that a replayed launch reads what a fresh call would have been given, bit for
// bit.  An entry that would pass the last cell the plan was checked for stops the advance
// (nothing moves, the status word says so).
__device__ __forceinline__ long long wave_sum(long long v) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
    return v;
}
__device__ __forceinline__ long long wave_max(long long v) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
        const long long o = __shfl_xor(v, off, 64);
        v = o > v ? o : v;
    }
    return v;
}
__global__ __launch_bounds__(64) void step_advance_kernel(StepDesc* d, AttnPlanLimits lim, int32_t page_cells) {
    static_assert(kMaxBatch <= 64, "one lane per entry");
    const int i = threadIdx.x;
    const int n = d->b.n;
    const bool live = i < n;
    int pos = live ? d->b.pos[i] : 0;
    const bool past = live && pos + 1 > d->horizon[i];
    if (__builtin_amdgcn_ballot_w64(past) != 0) {
        if (i == 0) d->status = 1;
        return;
    }
    pos += 1;
    const long long per_page = lim.per_page, gran = lim.gran;
    const long long min_total = (long long)n * per_page;
    long long target = lim.target < lim.max_wgs ? lim.target : lim.max_wgs;
    if (target < min_total) target = min_total;
    const long long pages = live ? pos / page_cells + 1 : 0;
    const long long total_pages = wave_sum(pages), max_pages = wave_max(pages);
    long long pps = (total_pages * per_page + target - 1) / target;
    pps = (pps + gran - 1) / gran * gran;
    if (pps < gran) pps = gran;
    long long my_splits = 0, each = gran, total = 0;
    for (;;) {
        if (live) {
            const long long splits = (pages + pps - 1) / pps;
            // even the ranges out inside the entry, keeping whole groups of `gran` pages
            each = (pages + splits - 1) / splits;
            each = (each + gran - 1) / gran * gran;
            my_splits = (pages + each - 1) / each;
        }
        total = wave_sum(my_splits * per_page);
        if (total <= target || pps >= max_pages) break;
        pps += gran;
    }
    // first work-group of every entry: the sum over the entries before it
    long long incl = my_splits * per_page;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
        const long long o = __shfl_up(incl, off, 64);
        if (i >= off) incl += o;
    }
    if (live) {
        d->b.pos[i] = pos;
        d->b.splits[i] = (int32_t)my_splits;
        d->b.pps[i] = (int32_t)each;
        d->b.wg_base[i] = (int32_t)(incl - my_splits * per_page);
    }
    if (i == 0) {
        d->b.wg_base[n] = (int32_t)total;
        d->steps += 1u;
    }
}

hipError_t launch_step_advance(StepDesc* d, const AttnPlanLimits& lim, int32_t page_cells, hipStream_t stream) {
    hipLaunchKernelGGL(step_advance_kernel, dim3(1), dim3(64), 0, stream, d, lim, page_cells);
    return hipGetLastError();
}

}  // namespace bkv
