// Batched Local_Alignment on gfx950: a persistent grid of single-wave
// workgroups pulls alignment tasks from a device counter; every task is one
// daligner Local_Alignment (dalign/align.c:1922-2060), computed by one half
// of a wave64 (la_pack.hpp).
//
// Device-resident batch (mi_la_batch_device):
//   * inputs stay in HBM: 2-bit packed reads and MiLaTask records;
//   * each finished task reserves its A and B traces in a compact trace arena
//     with one 64-bit atomic and copies them there, so the output is exactly
//     the traces produced (no worst-case per-task slots, no clearing);
//   * tasks whose band outgrows the 128 diagonals of the first instantiation's
//     wide window or their pebble pool append themselves to a device retry
//     list and are re-run by a wider one (256 / 1,024 diagonals, larger
//     pools); only the retry count comes back to the host between levels;
//   * before a launch every task it covers is marked LA_UNRUN, so a launch
//     stopped early (watchdog flag) can never leave a stale record behind;
//   * the scratch of each half (pebble pools, chain points, trace staging) is one
//     workspace carved per level.  The library keeps a grown workspace per
//     device, so repeated calls allocate nothing.
#pragma once
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdio>
#include <cstring>

#include "la_pack.hpp"
#include "mi_common.h"

namespace mi {

constexpr int LA_SPACE = 6;   // the call's trace arena is full (task not written)
constexpr int LA_UNRUN = 7;   // the launch stopped before reaching the task

struct BatchScratch {
    Peb* pools;
    int pool_cap;
    Peb* pts;
    int pts_cap;
    uint16_t* latr;   // per slot: 4 * maxtp u16 (A and B traces, each with maxtp before and after its origin)
    int latr_cap;
    int slots;        // alignments a wave holds, each with a slot of scratch
};

// Arguments of a launch, read through the kernarg segment.
struct BatchArgs {
    const MiLaTask* tasks;
    const int* order;
    int norder;
    const uint64_t* pk;
    DevSpec sp;
    MiLaResult* res;
    uint16_t* arena;
    long long arena_cap;
    unsigned long long* arena_top;
    int* retry;
    int* nretry;
    BatchScratch ws;
    int* counter;
    unsigned long long* work;
    const int* abort_flag;
};

// The tasks of a launch as the packed aligner's job (la_pack.hpp): half h of
// workgroup b owns scratch slot ws.slots b + h.
// (NCH: each kernel has its own copy, so its registers fit that kernel's.)
template <int NCH>
struct BatchJob {
    const BatchArgs* args;
    int* ti;   // LDS: the task of each half

    __device__ bool next(PackLds& L, int h)
    {
        const KernArgs<BatchArgs>* a = kern_args(args);
        const int lane = __lane_id();
        PackSlot& S = L.slot[h];
        const int ab = uni(__atomic_load_n(a->abort_flag, __ATOMIC_RELAXED));
        if (ab) return false;
        // every lane executes the atomic (only lane 0 adds 1), so no lane-dependent branch precedes the broadcast
        const int t = uni(atomicAdd(a->counter, lane == 0 ? 1 : 0));
        if (t >= a->norder) return false;
        const int i = a->order ? uni(a->order[t]) : t;
        if (lane == 0) {
            const MiLaTask tk = a->tasks[i];
            const int slot = a->ws.slots * blockIdx.x + h;
            const int TS = a->sp.tspace;
            const int maxtp = 2 * ((tk.alen > tk.blen ? tk.alen : tk.blen) / TS + 2);
            uint16_t* latr = a->ws.latr + (size_t)slot * a->ws.latr_cap;
            // Local_Alignment's borders (dalign/align.c:1966-1985): lbord/hbord < 0
            // leave the wave unbounded, except that a read aligned to itself may not
            // reach the main diagonal
            const bool selfie = (tk.aword == tk.bword && tk.selfie);
            S.minp = (tk.lbord < 0) ? ((selfie && tk.low >= 0) ? 1 : -INT32_MAX) : tk.low - tk.lbord;
            S.maxp = (tk.hbord < 0) ? ((selfie && tk.hgh <= 0) ? -1 : INT32_MAX) : tk.hgh + tk.hbord;
            S.prio = a->order ? queue_priority(t, a->norder) : 0;
            S.A = a->pk + tk.aword;
            S.B = a->pk + tk.bword;
            S.alen = tk.alen;
            S.blen = tk.blen;
            S.comp = tk.comp;
            S.low = tk.low;
            S.hgh = tk.hgh;
            S.anti = tk.anti;
            S.pool = a->ws.pools + (size_t)slot * a->ws.pool_cap;
            S.pool_cap = 4 * maxtp > a->ws.latr_cap ? 0 : a->ws.pool_cap;   // 0: no room for the trace, LA_POOL
            S.pts = a->ws.pts + (size_t)slot * 2 * a->ws.pts_cap;
            S.pts_cap = a->ws.pts_cap;
            S.atr = latr + maxtp;
            S.btr = latr + 3 * maxtp;
            S.maxtp = maxtp;
            ti[h] = i;
        }
        return true;
    }

    __device__ void done(PackLds& L, int h)
    {
        const KernArgs<BatchArgs>* a = kern_args(args);
        const int lane = __lane_id();
        PackSlot& S = L.slot[h];
        const int i = uni(ti[h]);
        int status = uni(S.res.status);
        const int na = status == LA_OK ? uni(S.res.atlen) : 0, nb = status == LA_OK ? uni(S.res.btlen) : 0;
        const int need = na + nb;
        long long off = 0;
        if (status == LA_OK) {
            const unsigned long long o = atomicAdd(a->arena_top, lane == 0 ? (unsigned long long)need : 0ull);
            off = uni((long long)o);
            if (off + need > a->arena_cap) {
                status = LA_SPACE;
            } else {
                const uint16_t* ta = uni(S.atr) + uni(S.res.afirst);
                const uint16_t* tb = uni(S.btr) + uni(S.res.bfirst);
                uint16_t* out = a->arena + off;
                for (int q = lane; q < na; q += 64) out[q] = ta[q];
                for (int q = lane; q < nb; q += 64) out[na + q] = tb[q];
            }
        } else if (status == LA_WIDE || status == LA_POOL) {
            const int q = uni(atomicAdd(a->nretry, lane == 0 ? 1 : 0));
            if (lane == 0) a->retry[q] = i;
        }
        if (lane == 0) {
            MiLaResult r = {};
            r.status = status;
            if (status == LA_OK) {
                r.abpos = S.res.abpos;
                r.bbpos = S.res.bbpos;
                r.aepos = S.res.aepos;
                r.bepos = S.res.bepos;
                r.diffs = S.res.diffs;
                r.b_abpos = S.res.b_abpos;
                r.b_bbpos = S.res.b_bbpos;
                r.b_aepos = S.res.b_aepos;
                r.b_bepos = S.res.b_bepos;
                r.atlen = na;
                r.btlen = nb;
            }
            r.atrace = off;
            r.btrace = off + (status == LA_OK ? na : 0);
            r.cells = S.cells;
            r.snake = S.snake;
            a->res[i] = r;
            atomicAdd(&a->work[0], (unsigned long long)S.cells);
            atomicAdd(&a->work[1], (unsigned long long)S.snake);
        }
        wave_sync();
    }
};

// A persistent grid of single-wave workgroups; with one slot a wave the upper
// halves stay idle.
template <int NCH>
__global__ __launch_bounds__(64, NCH == 2 ? kPackWaves : 1) void la_batch_kernel(BatchArgs)
{
    __shared__ PackLds L;
    __shared__ int ti[2];
    const BatchArgs* args = kernarg_ptr<BatchArgs>();
    const KernArgs<BatchArgs>* a = kern_args(args);
    DevSpec sp;
    sp.table = a->sp.table;
    sp.score = a->sp.score;
    sp.tspace = a->sp.tspace;
    sp.ave_path = a->sp.ave_path;
    pack_tables(L, sp);
    pack_run<NCH>(L, BatchJob<NCH>{args, ti}, a->ws.slots == 2, a->abort_flag);
}

// status of every task a launch covers := LA_UNRUN
static __global__ void k_la_mark_unrun(const int* __restrict__ order, int n, MiLaResult* __restrict__ res)
{
    const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) res[order ? order[i] : (int)i].status = LA_UNRUN;
}

// out[0] = max read length, out[1] = tasks whose reads leave the packed
// buffer or whose band is empty, out[2] = tasks still LA_UNRUN (results)
static __global__ void k_la_check(const MiLaTask* __restrict__ tasks, int n, long long npacked, int* out)
{
    const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const MiLaTask s = tasks[i];
    const bool bad = s.aword < 1 || s.bword < 1 || s.alen < 0 || s.blen < 0 || s.hgh < s.low ||
                     s.aword + (s.alen + 31) / 32 + 2 > npacked || s.bword + (s.blen + 31) / 32 + 2 > npacked;
    if (bad) atomicAdd(&out[1], 1);
    else atomicMax(&out[0], s.alen > s.blen ? s.alen : s.blen);
}

static __global__ void k_la_count_unrun(const MiLaResult* __restrict__ res, int n, int* out)
{
    const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n && res[i].status == LA_UNRUN) atomicAdd(&out[2], 1);
}

// Queue order for a batch whose caller gives none: the tasks by classes of
// their shorter read's length, longest first, so no long alignment starts when
// the queue is nearly empty.  (In task order 62 % of the CUs were busy over a
// launch of 20,000 tasks of 1 - 60 kb, 23.3 ms, with this one 20.9; 400,000
// tasks 53.9 and 48.5.)  cls[0..255]: counts, then the next free place of each
// class, zero at the start.
constexpr int kLenClasses = 256;

__device__ __forceinline__ int len_class(const MiLaTask& t, int maxlen)
{
    const int len = t.alen < t.blen ? t.alen : t.blen;
    return kLenClasses - 1 - (int)((long long)len * (kLenClasses - 1) / (maxlen > 0 ? maxlen : 1));
}

static __global__ __launch_bounds__(256) void k_la_class_counts(const MiLaTask* __restrict__ tasks, int n, int maxlen,
                                                                int* __restrict__ cls)
{
    __shared__ int h[kLenClasses];
    h[threadIdx.x] = 0;
    __syncthreads();
    const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) atomicAdd(&h[len_class(tasks[i], maxlen)], 1);
    __syncthreads();
    if (h[threadIdx.x]) atomicAdd(&cls[threadIdx.x], h[threadIdx.x]);
}

static __global__ __launch_bounds__(256) void k_la_class_starts(int* __restrict__ cls)
{
    __shared__ int s[kLenClasses];
    const int t = threadIdx.x, c = cls[t];
    s[t] = c;
    __syncthreads();
    for (int o = 1; o < kLenClasses; o <<= 1) {
        const int u = t >= o ? s[t - o] : 0;
        __syncthreads();
        s[t] += u;
        __syncthreads();
    }
    cls[t] = s[t] - c;
}

static __global__ __launch_bounds__(256) void k_la_class_order(const MiLaTask* __restrict__ tasks, int n, int maxlen,
                                                               int* __restrict__ cls, int* __restrict__ order)
{
    const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) order[atomicAdd(&cls[len_class(tasks[i], maxlen)], 1)] = (int)i;
}

// ---- workspace ----------------------------------------------------------------
// One batch call needs: a few counters, two retry lists of ntasks ints, and per
// level the per-wave scratch of that level's grid.  Level l runs window NCH[l]
// with pool PCAP[l] pebbles on at most GRID[l] waves.

struct Level {
    int nch;
    int pool_cap;
    int waves;   // upper bound; the scratch may cap it
};
constexpr int kWideLevel = 2;   // the first level of kWideNch

// Alignments a wave holds at level L when n tasks run and the scratch has room
// for `fit`.  One where every task gets a wave of its own, and where the
// scratch leaves SIMDs without a wave: two alignments in lock step take longer
// than one, so they are worth it only where waves share a SIMD.
// (The 64 MiB of mi_la_batch_device_noalloc hold about 120: with two a wave
// 4,000 tasks of 1 - 60 kb took 23.2 ms and 200,000 of 0.3 - 1 kb 220 ms, with
// one 16.3 and 160 ms.)
static int wave_slots(const Level& L, long long n, long long fit, int cus)
{
    return n > L.waves && fit > 4LL * cus ? 2 : 1;
}

static const int kCounterBytes = 4096;   // 256 bytes of counters, then the length classes of a queue

constexpr size_t kCarveSlack = 3 * 256;   // what a level's three pieces lose to their alignment, at most

static size_t align_up(size_t x) { return (x + 255) & ~(size_t)255; }

static size_t slot_bytes(int pool_cap, int pts_cap, int latr_cap)
{
    return (size_t)pool_cap * sizeof(Peb) + (size_t)2 * pts_cap * sizeof(Peb) + (size_t)latr_cap * sizeof(uint16_t);
}

// carve n slots of scratch at p (256-byte aligned pieces)
static BatchScratch carve(char* p, int n, int pool_cap, int pts_cap, int latr_cap)
{
    BatchScratch s;
    s.pool_cap = pool_cap;
    s.pts_cap = pts_cap;
    s.latr_cap = latr_cap;
    s.pools = (Peb*)p;
    p += align_up((size_t)n * pool_cap * sizeof(Peb));
    s.pts = (Peb*)p;
    p += align_up((size_t)n * 2 * pts_cap * sizeof(Peb));
    s.latr = (uint16_t*)p;
    s.slots = 1;
    return s;
}

static size_t carve_bytes(int n, int pool_cap, int pts_cap, int latr_cap)
{
    return align_up((size_t)n * pool_cap * sizeof(Peb)) + align_up((size_t)n * 2 * pts_cap * sizeof(Peb)) +
           align_up((size_t)n * latr_cap * sizeof(uint16_t));
}

static int launch_level(int nch, int grid, const MiLaTask* tasks, const int* order, int n, const uint64_t* pk,
                        const DevSpec& sp, MiLaResult* res, uint16_t* arena, long long arena_cap,
                        unsigned long long* arena_top, int* retry, int* nretry, const BatchScratch& ws, int* counter,
                        unsigned long long* work, const int* abort_flag, hipStream_t st)
{
    if (hipMemsetAsync(counter, 0, sizeof(int), st) != hipSuccess) return -1;
    if (hipMemsetAsync(nretry, 0, sizeof(int), st) != hipSuccess) return -1;
    hipLaunchKernelGGL(k_la_mark_unrun, dim3((n + 255) / 256), dim3(256), 0, st, order, n, res);
    const BatchArgs a{tasks, order, n, pk, sp, res, arena, arena_cap, arena_top, retry, nretry, ws, counter, work,
                      abort_flag};
    switch (nch) {
    case 2: hipLaunchKernelGGL(HIP_KERNEL_NAME(la_batch_kernel<2>), dim3(grid), dim3(64), 0, st, a); break;
    case 4: hipLaunchKernelGGL(HIP_KERNEL_NAME(la_batch_kernel<4>), dim3(grid), dim3(64), 0, st, a); break;
    case kWideNch: hipLaunchKernelGGL(HIP_KERNEL_NAME(la_batch_kernel<kWideNch>), dim3(grid), dim3(64), 0, st, a); break;
    default: return -1;
    }
    return hipGetLastError() == hipSuccess ? 0 : -1;
}

// Where a batch call's scratch lives: a buffer of `bytes` bytes.
struct ScratchArea {
    char* base;
    size_t bytes;
};

struct BatchPlan {
    int pts_cap, latr_cap;
    Level lv[4];
};

static BatchPlan make_plan(int maxlen, int tspace, int cus)
{
    BatchPlan p;
    // a chain holds one pebble per trace point of its read plus the root
    p.pts_cap = maxlen / tspace + 64;
    p.latr_cap = 4 * (2 * (maxlen / tspace + 2));
    const int w0 = mi_tuning().batch_waves_per_cu;
    const int w1 = mi_tuning().batch_wide_waves_per_cu;
    // bands of up to 128, 256 and 1,024 diagonals; a task re-runs at the
    // next level when its band outgrows the window or its pool fills
    p.lv[0] = Level{2, 1 << 15, cus * (w0 ? w0 : 4 * kPackWaves)};
    p.lv[1] = Level{4, 1 << 17, cus * (w1 ? w1 : 4)};
    p.lv[kWideLevel] = Level{kWideNch, 1 << 18, 256};
    p.lv[3] = Level{kWideNch, 1 << 20, 256};
    return p;
}

// Validates the tasks on the device: the longest read (sizes the per-wave
// scratch) or MI_ERR_ARG when a task's reads leave the packed buffer or its
// band is empty.  d_tmp: 3 device ints.
static int check_tasks(const MiLaTask* d_tasks, int ntasks, long long npacked, int* d_tmp, int* maxlen)
{
    hipStream_t st = 0;
    if (hipMemsetAsync(d_tmp, 0, 3 * sizeof(int), st) != hipSuccess) return MI_ERR_DEVICE;
    hipLaunchKernelGGL(k_la_check, dim3((ntasks + 255) / 256), dim3(256), 0, st, d_tasks, ntasks, npacked, d_tmp);
    int chk[3] = {0, 0, 0};
    if (hipMemcpyAsync(chk, d_tmp, sizeof(chk), hipMemcpyDeviceToHost, st) != hipSuccess ||
        hipStreamSynchronize(st) != hipSuccess)
        return MI_ERR_DEVICE;
    if (chk[1] != 0) {
        mi_set_error("batch: a task's reads lie outside the packed buffer or its band is empty");
        return MI_ERR_ARG;
    }
    *maxlen = chk[0];
    return 0;
}

// The level loop.  `area` holds the counters, the retry lists and the
// per-level wave scratch; levels whose full grid does not fit run fewer waves.
static int run_batch(DevSpec sp, const uint64_t* pk, const MiLaTask* tasks, int ntasks, int maxlen,
                     const int* order, MiLaResult* res, uint16_t* arena, long long arena_cap,
                     unsigned long long* d_arena_top, const ScratchArea& area, const int* abort_flag, bool watchdog,
                     long long* work, const char* who)
{
    char* p = area.base;
    int* ctr = (int*)p;   // [0] queue, [1] retry count, [2] unrun count
    unsigned long long* dwork = (unsigned long long*)(p + 64);
    p += kCounterBytes;
    int* lists[2];
    lists[0] = (int*)p;
    p += align_up((size_t)ntasks * sizeof(int));
    lists[1] = (int*)p;
    p += align_up((size_t)ntasks * sizeof(int));
    const size_t fixed = (size_t)(p - area.base);
    if (fixed > area.bytes) {
        mi_set_error("batch: task count exceeds the scratch");
        return MI_ERR_ARG;
    }
    hipStream_t st = 0;
    if (hipMemsetAsync(area.base, 0, kCounterBytes, st) != hipSuccess) return MI_ERR_DEVICE;
    int chk[3] = {0, 0, 0};
    // kernel time of each level (HIP events on the launch stream) when work is asked for
    static hipEvent_t ev[2] = {nullptr, nullptr};
    if (work) {
        for (int i = 0; i < 8; i++) work[i] = 0;
        for (int i = 0; i < 2; i++)
            if (ev[i] == nullptr && hipEventCreate(&ev[i]) != hipSuccess) return MI_ERR_DEVICE;
    }
    const BatchPlan plan = make_plan(maxlen, sp.tspace, mi_num_cus());
    sp.tspace = point_spacing(sp.tspace, maxlen);
    const int first = points24(sp.tspace, maxlen) ? 0 : kWideLevel;
    const int* cur = order;
    int n = ntasks;
    int which = 0;
    for (int level = first; level < 4 && n > 0; level++) {
        const Level& L = plan.lv[level];
        const size_t slot = slot_bytes(L.pool_cap, plan.pts_cap, plan.latr_cap), room = area.bytes - fixed;
        const long long fit = room > kCarveSlack ? (long long)((room - kCarveSlack) / slot) : 0;
        const int slots = wave_slots(L, n, fit, mi_num_cus());
        const long long g = std::min<long long>(std::min<long long>(L.waves, n), fit / slots);
        if (g <= 0) {
            mi_set_error("batch: scratch too small for one wave of this level");
            return MI_ERR_ARG;
        }
        BatchScratch ws = carve(area.base + fixed, slots * (int)g, L.pool_cap, plan.pts_cap, plan.latr_cap);
        ws.slots = slots;
        int* retry = lists[which];
        if (level == first && cur == nullptr && n > g) {
            // (the second list is free until the next level's retries)
            int* cls = (int*)(area.base + 256);
            const dim3 nb((n + 255) / 256), bt(256);
            hipLaunchKernelGGL(k_la_class_counts, nb, bt, 0, st, tasks, n, maxlen, cls);
            hipLaunchKernelGGL(k_la_class_starts, dim3(1), bt, 0, st, cls);
            hipLaunchKernelGGL(k_la_class_order, nb, bt, 0, st, tasks, n, maxlen, cls, lists[1]);
            if (hipGetLastError() != hipSuccess) return MI_ERR_DEVICE;
            cur = lists[1];
        }
        if (work && hipEventRecord(ev[0], st) != hipSuccess) return MI_ERR_DEVICE;
        if (launch_level(L.nch, (int)g, tasks, cur, n, pk, sp, res, arena, arena_cap, d_arena_top, retry, ctr + 1, ws,
                         ctr, dwork, abort_flag, st))
            return MI_ERR_DEVICE;
        if (work && hipEventRecord(ev[1], st) != hipSuccess) return MI_ERR_DEVICE;
        if (watchdog) {
            const int w = mi_wait_watchdog(st, who);
            if (w > 0) {
                mi_set_error("batch: kernel exceeded the watchdog deadline and was stopped");
                return MI_ERR_TIMEOUT;
            }
            if (w < 0) return MI_ERR_DEVICE;
        }
        int nr = 0;
        if (hipMemcpyAsync(&nr, ctr + 1, sizeof(int), hipMemcpyDeviceToHost, st) != hipSuccess ||
            hipStreamSynchronize(st) != hipSuccess)
            return MI_ERR_DEVICE;
        if (work) {
            float ms = 0.f;
            if (hipEventElapsedTime(&ms, ev[0], ev[1]) != hipSuccess) return MI_ERR_DEVICE;
            work[2 + level] = (long long)(ms * 1000.0);
            work[6] += nr;
        }
        cur = retry;
        n = nr;
        which ^= 1;
    }
    // tasks still wider than the widest level keep LA_WIDE / LA_POOL; a task
    // left LA_UNRUN means a launch was stopped from outside
    hipLaunchKernelGGL(k_la_count_unrun, dim3((ntasks + 255) / 256), dim3(256), 0, st, res, ntasks, ctr + 2);
    unsigned long long wk[2] = {0, 0};
    if (hipMemcpyAsync(chk, ctr + 2, sizeof(chk), hipMemcpyDeviceToHost, st) != hipSuccess ||
        hipMemcpyAsync(wk, dwork, sizeof(wk), hipMemcpyDeviceToHost, st) != hipSuccess ||
        hipStreamSynchronize(st) != hipSuccess)
        return MI_ERR_DEVICE;
    if (work) {
        work[0] = (long long)wk[0];
        work[1] = (long long)wk[1];
    }
    if (chk[2] != 0) {
        mi_set_error("batch: a launch stopped before reaching every task (abort flag raised)");
        return MI_ERR_TIMEOUT;
    }
    return 0;
}

}  // namespace mi
