// Building blocks of the wave64 furthest-reaching-point aligner (la_pack.hpp)
// on gfx950: constants and status codes, 2-bit sequence windows and match
// lengths, lane helpers, and the assembly of a pass's pebble chains
// (dalign/align.c:359-365, :970-1107, :1709-1901) into traces.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace mi {

constexpr int kPathLen = 60;
constexpr int kTrimMLag = 200;
constexpr int kWaveLag = 30;
// status codes of one alignment
constexpr int LA_OK = 0;
constexpr int LA_WIDE = 1;    // band wider than this instantiation's register window
constexpr int LA_POOL = 2;    // pebble pool or point scratch exhausted
constexpr int LA_UNDEF = 3;   // input drives the wave into a state the reference leaves undefined
constexpr int LA_CHAIN = 4;   // internal consistency check of a pebble chain failed
constexpr int LA_ABORT = 5;   // host watchdog asked the kernel to stop

struct DevSpec {
    const int16_t* table;   // [32768] suffix-positivity table, then the [32768] score table
    const int16_t* score;   // == table + 32768
    int tspace;
    int ave_path;
};

struct Peb {
    int up, diag, dif, mark;
};

// ---- sequence access -------------------------------------------------------
// 2-bit packed read: base i at bits 2*(i&31) of word (i>>5); one guard word
// before word 0 and two after the last word, so windows starting in
// [-32, len+32] stay inside the allocation.
// 16-base window starting at base p, read as 32-bit words of the same
// buffer (base i at bits 2*(i&15) of word i>>4): one funnel shift of the two
// words holding it.  Windows starting in [-32, len+32] stay inside the
// guard words.
__device__ __forceinline__ uint32_t win16(const uint32_t* pk, int p)
{
    const int q = p >> 4;
    return __builtin_amdgcn_alignbit(pk[q + 1], pk[q], (uint32_t)(2 * (p & 15)));
}

// forward: count of equal bases A[x+i] == B[y+i] for i < lim
__device__ __forceinline__ int match_fwd(const uint64_t* A, const uint64_t* B, int x, int y, int lim, bool& mism)
{
    const uint32_t* a = reinterpret_cast<const uint32_t*>(A);
    const uint32_t* b = reinterpret_cast<const uint32_t*>(B);
    int s = 0;
    mism = false;
    while (s < lim) {
        const uint32_t d = win16(a, x + s) ^ win16(b, y + s);
        if (d) {
            s += __builtin_ctz(d) >> 1;
            if (s < lim) mism = true;
            else s = lim;
            return s;
        }
        s += 16;
    }
    return lim;
}

// reverse: count of equal bases A[x-1-i] == B[y-1-i] for i < lim
__device__ __forceinline__ int match_rev(const uint64_t* A, const uint64_t* B, int x, int y, int lim, bool& mism)
{
    const uint32_t* a = reinterpret_cast<const uint32_t*>(A);
    const uint32_t* b = reinterpret_cast<const uint32_t*>(B);
    int s = 0;
    mism = false;
    while (s < lim) {
        const uint32_t d = win16(a, x - s - 16) ^ win16(b, y - s - 16);
        if (d) {
            s += __builtin_clz(d) >> 1;
            if (s < lim) mism = true;
            else s = lim;
            return s;
        }
        s += 16;
    }
    return lim;
}

// ---- cross-lane helpers ----------------------------------------------------
__device__ __forceinline__ int rdl(int v, int lane) { return __builtin_amdgcn_readlane(v, lane); }
__device__ __forceinline__ uint64_t rdl64(uint64_t v, int lane)
{
    uint32_t lo = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)v, lane);
    uint32_t hi = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(v >> 32), lane);
    return ((uint64_t)hi << 32) | lo;
}
// Order this wave's earlier global stores before its later loads (all
// lanes of one wave; no workgroup barrier, so several waves per workgroup may
// run independent alignments).
__device__ __forceinline__ void wave_sync()
{
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "workgroup");
    __builtin_amdgcn_wave_barrier();
}
__device__ __forceinline__ int lowest_lane(unsigned long long m) { return __ffsll((long long)m) - 1; }
__device__ __forceinline__ int highest_lane(unsigned long long m) { return 63 - __clzll(m); }
__device__ __forceinline__ int prefix_rank(unsigned long long m)
{
    return __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0));
}

// ---- trace assembly ----------------------------------------------------------
// Lane 0 rebuilds the A-view chain and lane 1 the B-view chain of one pass
// (the same code runs on both lanes with per-lane coordinates).  The chain
// from the tail pebble back to its root is copied tail first to the end of
// pts[0..pts_cap), so it reads root to tail from pts + pts_cap - (depth + 1),
// then walked like dalign/align.c:970-1107 (forward) or :1709-1901 (reverse).
//   tr     : trace origin (forward writes tr[0..], reverse prepends tr[-1..]);
//            it holds maxtp values on either side
//   fwdlen : (reverse only) length of the forward part already at tr[0..]
// Returns the new trace length / first index through *len / *first, or
// false for a chain that leaves the pool, outgrows pts_cap or needs more
// than maxtp trace values.
template <int DIR>
__device__ bool assemble_chain(const Peb* pool, int pool_used, Peb* pts_all, int pts_cap, int tail, bool isB, int mida,
                               int TS, int boff, int trimx, int trimy, int trimd, uint16_t* tr, int maxtp, int fwdlen,
                               int* len, int* first, int* root_diag)
{
    // copy the chain, tail first, until its root (up == -1); a chain that
    // leaves the pool or does not end within pts_cap links is reported,
    // never followed further
    int h = tail, nl = 0;
    while (h != -1) {
        if (h < 0 || h >= pool_used || nl >= pts_cap) return false;
        const Peb p = pool[h];
        pts_all[pts_cap - 1 - nl] = p;
        h = p.up;
        nl++;
    }
    if (nl == 0) return false;
    const int depth = nl - 1;
    if (2 * depth + 2 > maxtp) return false;
    const Peb* pts = pts_all + (pts_cap - nl);
    const int tprim = isB ? trimy : trimx;   // end-point coordinate along the trace axis
    const int tsec = isB ? trimx : trimy;    // and across it
    // secondary coordinate of a pebble: A-view -> y, B-view -> x
    auto sec = [&](const Peb& p) { return isB ? p.mark + p.diag : p.mark - p.diag; };
    *root_diag = pts[0].diag;
    if (DIR > 0) {
        const int k0 = pts[0].diag;
        int b = isB ? (mida + k0) / 2 : (mida - k0) / 2;
        int e = 0, n = 0, kk = k0;
        for (int i = 1; i <= depth; i++) {
            kk = pts[i].diag;
            const int a = sec(pts[i]);
            const int dd = pts[i].dif;
            tr[n++] = (uint16_t)(dd - e);
            tr[n++] = (uint16_t)(a - b);
            b = a;
            e = dd;
        }
        const int prim = isB ? b - kk : b + kk;
        if (prim != tprim) {
            tr[n++] = (uint16_t)(trimd - e);
            tr[n++] = (uint16_t)(tsec - b);
        } else if (b != tsec && n > 0) {
            tr[n - 1] = (uint16_t)(tr[n - 1] + (tsec - b));
            tr[n - 2] = (uint16_t)(tr[n - 2] + (trimd - e));
        }
        *len = n;
        *first = 0;
    } else {
        int kk = pts[0].diag;
        int b = sec(pts[0]);
        int e = 0, n = 0, i = 0;
        bool live = true;   // reference: h >= 0
        const int prim0 = isB ? b - kk : b + kk;
        if (prim0 % TS != (isB ? boff : 0)) {
            int a, dd;
            i = 1;
            if (i > depth) {
                a = tsec;
                dd = trimd;
                live = false;
            } else {
                kk = pts[i].diag;
                a = sec(pts[i]);
                dd = pts[i].dif;
            }
            if (fwdlen == 0) {
                tr[--n] = (uint16_t)(b - a);
                tr[--n] = isB ? (uint16_t)(b - a) : (uint16_t)(dd - e);   // dalign/align.c:1831-1832
            } else {
                tr[1] = (uint16_t)(tr[1] + (b - a));
                tr[0] = (uint16_t)(tr[0] + (dd - e));
            }
            b = a;
            e = dd;
        }
        if (live) {
            for (int q = i + 1; q <= depth; q++) {
                kk = pts[q].diag;
                const int a = sec(pts[q]);
                tr[--n] = (uint16_t)(b - a);
                const int dd = pts[q].dif;
                tr[--n] = (uint16_t)(dd - e);
                b = a;
                e = dd;
            }
            const int prim = isB ? b - kk : b + kk;
            if (prim != tprim) {
                tr[--n] = (uint16_t)(b - tsec);
                tr[--n] = (uint16_t)(trimd - e);
            } else if (b != tsec && (n < 0 || fwdlen > 0)) {
                tr[n + 1] = (uint16_t)(tr[n + 1] + (b - tsec));
                tr[n] = (uint16_t)(tr[n] + (trimd - e));
            }
        }
        *len = -n;
        *first = n;
    }
    return true;
}

struct LaResult {
    int abpos, bbpos, aepos, bepos, diffs;     // A-view path
    int b_abpos, b_bbpos, b_aepos, b_bepos;    // B-view path (diffs equal)
    int atlen, btlen;
    int afirst, bfirst;                        // trace start relative to the trace origins
    int status;
};

}  // namespace mi
