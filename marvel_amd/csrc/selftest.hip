// Device self-tests of the wave64 building blocks the aligner relies on
// (cross-lane scans, neighbour gathers, ballots/mbcnt, the 2-bit snake
// matcher, the persistent task loop).  Each test writes plain per-lane /
// per-task outputs that the host checks against a CPU computation.
#include <hip/hip_runtime.h>

#include "la_wave.hpp"
#include "mi_common.h"

namespace mi {

// test 0: persistent loop scaffold -- outs[t] = 3*t + 1 for every task
__global__ __launch_bounds__(64) void st_persistent(int n, int* counter, int* outs, const int* abort_flag)
{
    for (;;) {
        const int t = __builtin_amdgcn_readfirstlane(atomicAdd(counter, __lane_id() == 0 ? 1 : 0));
        const int ab = __builtin_amdgcn_readfirstlane(__atomic_load_n(abort_flag, __ATOMIC_RELAXED));
        if (t >= n || ab) break;
        outs[t] = 3 * t + 1;   // every lane stores the same value
    }
}

// test 1: per wave, input v[64]; outputs per lane:
//   o[0] = exclusive suffix max (lanes above), o[1] = exclusive prefix min (lanes below),
//   o[2] = value of lane-1 (wrap), o[3] = value of lane+1 (wrap),
//   o[4] = readlane(v, lowest lane with v odd), o[5] = mbcnt rank among odd lanes,
//   o[6] = __any(v > thr), o[7] = popcount of ballot(v odd)
__global__ __launch_bounds__(64) void st_lanes(const int* in, int thr, int* out)
{
    const int lane = __lane_id();
    const int v = in[blockIdx.x * 64 + lane];
    int incl = v;
    for (int o = 1; o < 64; o <<= 1) {
        const int w = __shfl_down(incl, o, 64);
        if (lane + o < 64) incl = max(incl, w);
    }
    int excl = __shfl_down(incl, 1, 64);
    if (lane == 63) excl = -1;
    int inc2 = v;
    for (int o = 1; o < 64; o <<= 1) {
        const int w = __shfl_up(inc2, o, 64);
        if (lane - o >= 0) inc2 = min(inc2, w);
    }
    int exc2 = __shfl_up(inc2, 1, 64);
    if (lane == 0) exc2 = INT32_MAX;
    const int up = shfl_i(v, (lane + 63) & 63);
    const int dn = shfl_i(v, (lane + 1) & 63);
    const unsigned long long odd = __ballot(v & 1);
    int rl = -7;
    if (odd) rl = rdl(v, lowest_lane(odd));
    const int rank = prefix_rank(odd);
    const int any = __any(v > thr);
    int* o = out + (blockIdx.x * 64 + lane) * 8;
    o[0] = excl; o[1] = exc2; o[2] = up; o[3] = dn; o[4] = rl; o[5] = rank; o[6] = any; o[7] = __popcll(odd);
}

// test 2: snake matcher; per lane one query (x, y, lim, dir) on packed A/B
__global__ __launch_bounds__(64) void st_match(const uint64_t* A, const uint64_t* B, const int* q, int n, int* out)
{
    const int i = blockIdx.x * 64 + __lane_id();
    if (i >= n) return;
    const int x = q[4 * i], y = q[4 * i + 1], lim = q[4 * i + 2], dir = q[4 * i + 3];
    bool mism;
    const int s = dir > 0 ? match_fwd(A, B, x, y, lim, mism) : match_rev(A, B, x, y, lim, mism);
    out[2 * i] = s;
    out[2 * i + 1] = mism ? 1 : 0;
}

// value of lane (L-1) & 63 / (L+1) & 63: DPP wave_ror:1 / wave_rol:1, full-rate
// VALU moves (no LDS traffic).  All 64 lanes must be active.
// (every lane has a source, so no "old" value is needed: one v_mov_b32_dpp)
__device__ __forceinline__ int lane_below(int v) { return __builtin_amdgcn_mov_dpp(v, 0x13C, 0xF, 0xF, false); }
__device__ __forceinline__ int lane_above(int v) { return __builtin_amdgcn_mov_dpp(v, 0x134, 0xF, 0xF, false); }
// Wave-wide scans from DPP row moves (no LDS): row_shl:n / row_shr:n read
// lane L+n / L-n of the same 16-lane row, row_bcast:15 / :31 hand the last
// lane of a row (of two rows) to the next row(s).  Lanes without a source
// read 0 (bound_ctrl), the identity of max over non-negative values, so each
// level is a single v_max_i32 with a DPP operand.
template <int CTRL, int ROW_MASK = 0xF>
__device__ __forceinline__ int dpp0(int v)
{
    return __builtin_amdgcn_update_dpp(0, v, CTRL, ROW_MASK, 0xF, true);
}
// inclusive max over lanes >= L of x >= 0
__device__ __forceinline__ int suffix_max_nn(int x)
{
    x = max(x, dpp0<0x101>(x));   // row_shl:1
    x = max(x, dpp0<0x102>(x));   // row_shl:2
    x = max(x, dpp0<0x104>(x));   // row_shl:4
    x = max(x, dpp0<0x108>(x));   // row_shl:8
    // lane 16r now holds row r's maximum; lanes of row r add the rows above
    // it, selected with arithmetic masks (-1 / 0) rather than lane masks
    const int s1 = __builtin_amdgcn_readlane(x, 16), s2 = __builtin_amdgcn_readlane(x, 32);
    const int s3 = __builtin_amdgcn_readlane(x, 48);
    int row = __lane_id() >> 4;
    asm volatile("" : "+v"(row));   // keeps the row masks from being hoisted into (spilled) SGPR lane masks
    const int m1 = (row - 1) >> 31, m2 = (row - 2) >> 31, m3 = (row - 3) >> 31;
    return max(max(x, s1 & m1), max(s2 & m2, s3 & m3));
}
// inclusive max over lanes <= L of x >= 0
__device__ __forceinline__ int prefix_max_nn(int x)
{
    x = max(x, dpp0<0x111>(x));        // row_shr:1
    x = max(x, dpp0<0x112>(x));        // row_shr:2
    x = max(x, dpp0<0x114>(x));        // row_shr:4
    x = max(x, dpp0<0x118>(x));        // row_shr:8
    x = max(x, dpp0<0x142, 0xA>(x));   // row_bcast:15 into rows 1, 3
    x = max(x, dpp0<0x143, 0xC>(x));   // row_bcast:31 into rows 2, 3
    return x;
}
// value of lane L+1 / L-1; the lane without one (63 / 0) gets `edge`
// (DPP wave_shl:1 / wave_shr:1)
__device__ __forceinline__ int lane_above_or(int v, int edge) { return __builtin_amdgcn_update_dpp(edge, v, 0x130, 0xF, 0xF, false); }
__device__ __forceinline__ int lane_below_or(int v, int edge) { return __builtin_amdgcn_update_dpp(edge, v, 0x138, 0xF, 0xF, false); }
// inclusive max over lanes >= L (x >= -1).  GATHER: the lanes reversed by one
// ds_bpermute each way around the DPP prefix scan, for passes that run many
// waves per SIMD (the LDS pipe is idle there, the VALU is not); otherwise
// the DPP suffix scan, which keeps the two LDS round trips off the path of a
// wave that runs alone (the wider windows).
template <bool GATHER>
__device__ __forceinline__ int wave_suffix_max(int x)
{
    if constexpr (GATHER) {
        const int r = 63 - __lane_id();
        return __shfl(prefix_max_nn(__shfl(x + 1, r, 64)), r, 64) - 1;
    } else {
        return suffix_max_nn(x + 1) - 1;
    }
}
// inclusive min over lanes <= L (any x): the max of INT32_MAX - x >= 0
__device__ __forceinline__ int wave_prefix_min(int x) { return 2147483647 - prefix_max_nn(2147483647 - x); }

// fields of lane L + sel (sel in {-1, 0, +1}, wrapping like (L + sel) & 63)
__device__ __forceinline__ int pick3(int v, int sel)
{
    const int b = lane_below(v), a = lane_above(v);
    return sel < 0 ? b : (sel > 0 ? a : v);
}
// test 3: DPP lane moves; per lane: [lane_below(v), lane_above(v), the
// scans, the edge moves, the DPP suffix max, pick3 with sel = L % 3 - 1]
__global__ __launch_bounds__(64) void st_dpp(const int* in, int* out)
{
    const int lane = __lane_id();
    const int v = in[blockIdx.x * 64 + lane];
    int* o = out + (blockIdx.x * 64 + lane) * 8;
    o[0] = lane_below(v);
    o[1] = lane_above(v);
    // the aligner's scans: suffix max over values >= -1, prefix min over values >= 0
    o[2] = wave_suffix_max<true>(v);
    o[3] = wave_prefix_min(v < 0 ? 2147483647 : v);
    o[4] = lane_above_or(v, -7);
    o[5] = lane_below_or(v, -9);
    o[6] = wave_suffix_max<false>(v);
    o[7] = pick3(v, lane % 3 - 1);
}

}  // namespace mi

using namespace mi;

extern "C" int mi_selftest(int which, const void* in, long long nin, const void* in2, long long nin2,
                           const void* q, int nq, int arg, void* out, long long nout)
{
    void *din = nullptr, *din2 = nullptr, *dq = nullptr, *dout = nullptr;
    int* dctr = nullptr;
    int rc = MI_ERR_DEVICE;
    const int* abort_flag = mi_abort_flag_device();
    if (abort_flag == nullptr) return MI_ERR_DEVICE;
    if (nin > 0 && (hipMalloc(&din, nin) != hipSuccess || hipMemcpy(din, in, nin, hipMemcpyHostToDevice) != hipSuccess)) goto done;
    if (nin2 > 0 && (hipMalloc(&din2, nin2) != hipSuccess || hipMemcpy(din2, in2, nin2, hipMemcpyHostToDevice) != hipSuccess)) goto done;
    if (nq > 0 && (hipMalloc(&dq, 16LL * nq) != hipSuccess || hipMemcpy(dq, q, 16LL * nq, hipMemcpyHostToDevice) != hipSuccess)) goto done;
    if (hipMalloc(&dout, nout) != hipSuccess || hipMemset(dout, 0, nout) != hipSuccess) goto done;
    if (hipMalloc(&dctr, sizeof(int)) != hipSuccess || hipMemset(dctr, 0, sizeof(int)) != hipSuccess) goto done;
    switch (which) {
    case 0:
        hipLaunchKernelGGL(HIP_KERNEL_NAME(st_persistent), dim3(arg), dim3(64), 0, 0, (int)(nout / 4), dctr, (int*)dout, abort_flag);
        break;
    case 1:
        hipLaunchKernelGGL(HIP_KERNEL_NAME(st_lanes), dim3((int)(nin / 256)), dim3(64), 0, 0, (const int*)din, arg, (int*)dout);
        break;
    case 2:
        hipLaunchKernelGGL(HIP_KERNEL_NAME(st_match), dim3((nq + 63) / 64), dim3(64), 0, 0, (const uint64_t*)din + 1, (const uint64_t*)din2 + 1, (const int*)dq, nq,
                                         (int*)dout);
        break;
    case 3:
        hipLaunchKernelGGL(HIP_KERNEL_NAME(st_dpp), dim3((int)(nin / 256)), dim3(64), 0, 0, (const int*)din, (int*)dout);
        break;
    default:
        rc = MI_ERR_ARG;
        goto done;
    }
    if (hipGetLastError() != hipSuccess) goto done;
    if (mi_wait_watchdog(0, "mi_selftest") != 0) { rc = MI_ERR_TIMEOUT; goto done; }
    if (hipMemcpy(out, dout, nout, hipMemcpyDeviceToHost) != hipSuccess) goto done;
    rc = 0;
done:
    (void)hipFree(din);
    (void)hipFree(din2);
    (void)hipFree(dq);
    (void)hipFree(dout);
    (void)hipFree(dctr);
    return rc;
}
