// Furthest-reaching-point aligner for gfx950 (CDNA4): two alignments per
// wave64, one on each 32-lane half.
//
// A daligner Local_Alignment (dalign/align.c:1922-2060) is a forward pass
// (dalign/align.c:369-1110) and a reverse pass (:1114-1916) of furthest-
// reaching waves.  The band of diagonals of a pass lives in registers, one
// diagonal per lane.
//
// Why halves: the bands of real overlaps are narrow -- 12 diagonals on
// average at 28 % pair error, 99.99 % of the steps at most 30 on reads of an
// iid genome, 93 % where the genome is full of repeats -- and the loop is
// bound by VALU issue where the GPU is full and by its chain of dependent
// memory and lane operations where it is not.  One alignment per wave leaves
// 80 % of the lanes without a diagonal; two per wave share every instruction.
//   * A half keeps its band in lanes 1..30 (lanes 0 and 31 always hold the
//     sentinel, so single-lane DPP moves over the whole wave never carry a
//     value from one half into the other).
//   * A pass whose band outgrows 30 diagonals takes the whole wave for a
//     while (wide_run: 64 NCH diagonals, the other half's registers wait) and
//     comes back to its half when the band is narrow again, so nothing is
//     computed twice.  Bands beyond 64 NCH diagonals report LA_WIDE and the
//     caller runs the alignment again with a larger NCH.
//   * Both directions run the same code: the reverse pass is the forward
//     pass of the reflected problem (x, y, k and V negated), which keeps
//     every comparison and tie of the reference's reverse loop; only the
//     sequence windows are read backwards.  The halves of a wave are mostly
//     in different passes.
//   * Lane L of a half holds diagonal k = ktop - L, so the reference's
//     visiting order (k descending) is lane order and the records ("strict
//     improvements of the best antidiagonal") are a DPP prefix maximum.
//   * What the reference tests against memory is carried instead: a
//     diagonal's trace-point thresholds and its pebbles' trace points as
//     small numbers (the 8 low bits of the number ride on the pebble's
//     index, see skip_points), so a wave that crosses trace points only stores; the
//     suffix-positivity test of the trim point (dalign/align.c:884-896) reads
//     a 10-bit table in LDS three times instead of a 128 KB table twice.
//   * What only changes at events lives in LDS, written by the lane that owns
//     the event: the trim point, the best point's y, the boundary point.
//
// What bounds it, on a full GPU: VALU issue -- 2.65e10 wave64 VALU
// instructions per report launch on the 5 Mbp / 30x block (195 per step of two
// alignments), 43 ms of the 45 ms it takes at one per SIMD every 4 cycles; one
// alignment per wave needed 5.2e10 and 96 ms (and 6.6 ms more for the pairs
// wider than 64 diagonals, run again at 128).  So the sets of lanes are kept as
// the compares' own masks (ballot, lane_in: an integer made of a condition and
// compared again takes 2 instructions more each), products are 24-bit, and the
// reads and the pool are addressed as HBM (a flat access also holds up every
// wait for LDS).  Where few alignments are left (repeat-rich
// blocks: one pair with 90 alignments one after another, 55 % of the CUs busy
// over the launch) it is the latency of one wave's step, about 1.5 us.
// Waves per SIMD, ms a pass against 6 (both in turn on one GPU):
//   4: 5 Mbp block 186 : 179, repeat-rich 201 : 207, 400,000 tasks that start
//      off their diagonal 54.2 : 48.4, 20,000 tasks 19.2 : 21.8
//   5: 197 : 189, 254 : 259, 50.6 : 49.1, 19.8 : 21.6
//   7: 177 : 174, 223 : 213, 47.6 : 48.0, 20.5 : 20.7 (spills in the loop)
//
// Persistent kernels: `Job` (a few pointers, passed by value) hands out
// alignments (next) and takes their results (done); PackSlot says what it
// fills in.  What happens between passes and in wide bands is called, not
// inlined, so the loop's registers are its own.
#pragma once
#include "la_wave.hpp"

namespace mi {

constexpr int kHalfBand = 30;          // diagonals a half holds (lanes 1..30)
constexpr int kNarrow = 18;            // a wide band this narrow returns to its half
constexpr int kOneChunk = 44;          // a wide band this narrow is kept in one 64-lane chunk, the others' steps are skipped
constexpr int kSentV = -(1 << 30);     // V of a lane without a diagonal
constexpr int kFar = 1 << 30;          // no border
constexpr int kPebIdx = 0xffffff;      // pebble index in HA / HB; the top 8 bits: its trace point's number
constexpr int kPoolMax = 1 << 24;
constexpr int kPackWaves = 6;          // waves per SIMD of the kernels with the smallest wide window (see the note above)
constexpr int kSufBits = 10;           // columns per lookup of the suffix table

// phases of a slot
constexpr int PH_IDLE = 0, PH_FWD = 1, PH_REV = 2;
// LA_* codes a pass ends with; this one asks for the whole wave
constexpr int LA_GROW = 100;

// One half's alignment, in LDS.
struct PackSlot {
    // the alignment, filled in by the job
    const uint64_t *A, *B;
    Peb* pool;
    Peb* pts;            // 2 pts_cap points
    uint16_t *atr, *btr; // trace origins (each with maxtp entries before and after)
    int alen, blen, comp, low, hgh, anti, minp, maxp;
    int pool_cap, pts_cap, maxtp;
    // the pass
    int phase;
    int mind;            // reverse pass: the diagonal of the forward B chain's root
    int status;          // LA_* it ended with
    int used, dif;       // pebbles, waves
    int fa, fb;          // forward trace lengths
    // the alignment's results
    long long cells, snake, steps, snake0;   // snake0: before the pass
    LaResult res;
    // a pass outside the loop's registers (see PackBand)
    int a, b, ktop, besta, lasta, navail, amin, bmax, running;
    int prio;            // the wave's priority while this alignment runs (queue_priority)
};

// A half's diagonals outside the loop's registers: while the other half is
// served, and on their way into and out of wide_run.
struct PackBand {
    int V[32], M[32], HA[32], HB[32], tA[32], tB[32];   // M: bit 16 set where the wave's snake ran into a read's end
    uint64_t N[32];
};
constexpr int kEnd = 1 << 16;

// What the loop writes at events, at the front of LDS (small offsets).
struct PackHot {
    int tr_c, tr_y, tr_d, tr_ha, tr_hb;           // trim point
    int best_y;                                   // y of the best antidiagonal's diagonal
    int mo_m, mo_c, mo_y, mo_d, mo_ha, mo_hb;     // boundary point (mo_m < 0: none)
    int pad[4];
};

struct PackLds {
    PackHot hot[2];
    int16_t suf[1 << kSufBits];   // smallest suffix sum of 10 columns given by their mismatches
    int w_all, w_match;           // score of a column: w_match for a match, w_match - w_all for a mismatch
    int many;                     // the last wave of a pass passed many trace points (see skip_points)
    DevSpec sp;
    PackSlot slot[2];
    PackBand band[2];
};

// A kernel's only argument, a struct, read where it is used by scalar loads
// through the kernarg segment, so none of it is held across the loop.
#ifndef MI_CPU_WAVE_EMU
template <class T>
using Glob = T __attribute__((address_space(1)));   // in HBM: pointers that come out of LDS would be flat otherwise
template <class T>
using KernArgs = const T __attribute__((address_space(4)));
template <class T>
__device__ __forceinline__ const T* kernarg_ptr()
{
    return (const T*)(KernArgs<T>*)__builtin_amdgcn_kernarg_segment_ptr();
}
#else
// the CPU wave emulator (tests/wave_emu) hands the launch's arguments over
template <class T>
using Glob = T;
template <class T>
using KernArgs = const T;
template <class T>
inline const T* kernarg_ptr() { return (const T*)emu::kernarg(); }
#endif

// the lanes where p holds: the compare's own mask (HIP's __ballot makes an integer of p and compares it again)
__device__ __forceinline__ unsigned long long ballot(bool p)
{
#ifndef MI_CPU_WAVE_EMU
    return __builtin_amdgcn_ballot_w64(p);
#else
    return __ballot(p);
#endif
}
__device__ __forceinline__ bool any_lane(bool p) { return ballot(p) != 0; }
// whether this lane is one of m's: the mask itself as the condition
__device__ __forceinline__ bool lane_in(unsigned long long m)
{
#ifndef MI_CPU_WAVE_EMU
    return __builtin_amdgcn_inverse_ballot_w64(m);
#else
    return (m >> __lane_id()) & 1;
#endif
}
typedef int Int4 __attribute__((vector_size(16)));   // a pebble as it is stored
static_assert(sizeof(Peb) == 16, "a pebble is stored as one vector");

__device__ __forceinline__ int uni(int v) { return __builtin_amdgcn_readfirstlane(v); }
template <class T>
__device__ __forceinline__ T* uni(T* p)
{
    const uint64_t v = (uint64_t)p;
    const uint32_t lo = (uint32_t)uni((int)(uint32_t)v), hi = (uint32_t)uni((int)(uint32_t)(v >> 32));
    return (T*)(((uint64_t)hi << 32) | lo);
}
__device__ __forceinline__ long long uni(long long v)
{
    const uint32_t lo = (uint32_t)uni((int)(uint32_t)v), hi = (uint32_t)uni((int)(uint32_t)((unsigned long long)v >> 32));
    return (long long)(((uint64_t)hi << 32) | lo);
}
template <class T>
__device__ __forceinline__ KernArgs<T>* kern_args(const T* p)
{
    return (KernArgs<T>*)uni(p);
}
// product of two factors below 2^23 (full rate; the 32-bit multiply takes four times as long)
__device__ __forceinline__ int mul24(int x, int y) { return __mul24(x, y); }
// Trace point t's place is t TS, in the narrower windows a 24-bit product.
// The hosts keep its factors below 2^23 there: point_spacing takes a spacing
// beyond every read down (no read has a point then, whatever the spacing), and
// what points24 still refuses -- reads of 2^23 bases or more -- starts at the
// widest window, whose kernel multiplies in 32 bits.
constexpr int kMul24 = 1 << 23;
constexpr int kWideNch = 16;
template <int NCH>
__device__ __forceinline__ int point_at(int t, int TS)
{
    if constexpr (NCH == kWideNch) return t * TS;
    else return mul24(t, TS);
}
static inline int point_spacing(int TS, int maxlen) { return TS >= kMul24 && maxlen < kMul24 - 1 ? kMul24 - 1 : TS; }
static inline bool points24(int TS, int maxlen) { return TS < kMul24 && maxlen / TS + 2 < kMul24; }
// value of lane `src`
__device__ __forceinline__ int bperm(int v, int src) { return __builtin_amdgcn_ds_bpermute(src << 2, v); }
__device__ __forceinline__ uint64_t bperm64(uint64_t v, int src)
{
    return ((uint64_t)(uint32_t)bperm((int)(uint32_t)(v >> 32), src) << 32) | (uint32_t)bperm((int)(uint32_t)v, src);
}
// lo on the lower half's lanes, hi on the upper half's (hm: 0 / -1), both wave-uniform
__device__ __forceinline__ int hsel(int hm, int lo, int hi)
{
    return (int)((unsigned)lo + ((unsigned)hm & ((unsigned)hi - (unsigned)lo)));
}
// Wave priority (0..3) by the place in the queue: the queues hold the longest
// alignments first, and a launch ends when the longest chain of waves does,
// so the waves that hold it issue before the others of their SIMD.
// (Without and with: 400,000 tasks 50.6 and 48.1 ms, 20,000 tasks 21.8 and
// 21.5, 4 Mbp block 11.9 and 11.7, 5 Mbp block 179 and 178; repeat-rich block,
// whose heavy pairs their seeds do not tell, 219 and 221.)
__device__ __forceinline__ int queue_priority(int t, int n)
{
    return t < n / 256 ? 3 : t < n / 32 ? 2 : t < n / 8 ? 1 : 0;
}
__device__ __forceinline__ void set_priority(int p)
{
#ifndef MI_CPU_WAVE_EMU
    if (p == 3) __builtin_amdgcn_s_setprio(3);
    else if (p == 2) __builtin_amdgcn_s_setprio(2);
    else if (p == 1) __builtin_amdgcn_s_setprio(1);
    else __builtin_amdgcn_s_setprio(0);
#endif
}
__device__ __forceinline__ uint32_t hmask(int hm, unsigned long long m)
{
    return (uint32_t)hsel(hm, (int)(uint32_t)m, (int)(uint32_t)(m >> 32));
}
__device__ __forceinline__ int top_bit(uint32_t m) { return 31 - __builtin_clz(m | 1u); }
__device__ __forceinline__ int low_bit(uint32_t m) { return __builtin_ctz(m | 0x80000000u); }

// inclusive prefix maximum over the lanes of each half / of the wave
template <int CTRL, int ROWS = 0xF>
__device__ __forceinline__ int dpp_max(int x)
{
    return max(x, __builtin_amdgcn_update_dpp(INT32_MIN, x, CTRL, ROWS, 0xF, false));
}
template <bool WAVE>
__device__ __forceinline__ int prefix_max(int x)
{
    x = dpp_max<0x111>(x);                        // row_shr:1, 2, 4, 8
    x = dpp_max<0x112>(x);
    x = dpp_max<0x114>(x);
    x = dpp_max<0x118>(x);
    x = dpp_max<0x142, 0xA>(x);                   // row_bcast:15 into rows 1, 3
    if constexpr (WAVE) x = dpp_max<0x143, 0xC>(x);   // row_bcast:31 into rows 2, 3
    return x;
}
// value of lane L - 1 / L + 1; lanes 0 / 63: anything / the sentinel
__device__ __forceinline__ int dpp_shr1(int v) { return __builtin_amdgcn_mov_dpp(v, 0x138, 0xF, 0xF, true); }
__device__ __forceinline__ int dpp_shl1(int v) { return __builtin_amdgcn_mov_dpp(v, 0x130, 0xF, 0xF, true); }
__device__ __forceinline__ int from_below(int v) { return __builtin_amdgcn_update_dpp(kSentV, v, 0x138, 0xF, 0xF, false); }
__device__ __forceinline__ int from_above(int v) { return __builtin_amdgcn_update_dpp(kSentV, v, 0x130, 0xF, 0xF, false); }

// Matching columns from (x, y) on in the pass's direction, at most lim (m: 0
// forward, -1 reverse; x and y in the pass's coordinates), on the lanes where
// `in` holds; every lane takes part.  32 bases a step: a second step is a
// round trip to memory for the whole wave, and with 16 bases one of its lanes
// asks for it in 9 of 10 steps at 16 % pair error (in 1 of 8 at 28 %).
// (16 and 32 bases: 20,000 tasks 22.4 and 21.5 ms; 400,000 tasks, the 5 Mbp
// and the repeat-rich block the same.)
typedef Glob<const uint32_t> SeqWord;
// the 32-base windows at x and y compared: bit pair i differs where base i does
__device__ __forceinline__ uint64_t seq_diff(SeqWord* A, SeqWord* B, int m, int x, int y)
{
    const int off = m & -31;
    const int p = (x ^ m) + off, q = (y ^ m) + off;   // reverse: the 32 bases before x
    SeqWord* a = A + (p >> 4);
    SeqWord* b = B + (q >> 4);
    const uint32_t a0 = a[0], a1 = a[1], a2 = a[2], b0 = b[0], b1 = b[1], b2 = b[2];
    const uint32_t lo = __builtin_amdgcn_alignbit(a1, a0, (uint32_t)(2 * p)) ^
                        __builtin_amdgcn_alignbit(b1, b0, (uint32_t)(2 * q));
    const uint32_t hi = __builtin_amdgcn_alignbit(a2, a1, (uint32_t)(2 * p)) ^
                        __builtin_amdgcn_alignbit(b2, b1, (uint32_t)(2 * q));
    const uint32_t d0 = m ? __builtin_bitreverse32(hi) : lo, d1 = m ? __builtin_bitreverse32(lo) : hi;
    return ((uint64_t)d1 << 32) | d0;
}
__device__ __forceinline__ int same_bases(uint64_t d) { return (d ? __builtin_ctzll(d) : 64) >> 1; }
__device__ __forceinline__ int snake_len(SeqWord* A, SeqWord* B, int m, int x, int y, int lim, bool in)
{
    int s = 0;
    if (in) s = same_bases(seq_diff(A, B, m, x, y));
    unsigned long long go = ballot(s == 32) & ballot(lim > 32);
    while (go) {
        int n = 0;
        if (lane_in(go)) n = same_bases(seq_diff(A, B, m, x + s, y + s));
        s += n;
        go = ballot(n == 32) & ballot(s < lim);
    }
    return min(s, lim);
}

// The last 61 columns of a path as mismatch bits, latest at bit 3, with bit 2
// set (the mismatch column every step begins with): one more mismatch and s
// matches.  m: matches among them.
__device__ __forceinline__ void add_columns(uint64_t& N, int& m, int s)
{
    const int sc = min(s, 61);
    m += __popcll(N >> (63 - sc)) - 1;
    N = (N << (sc + 1)) | 4;
}
constexpr uint64_t kColsInit = (1ull << 63) | 4;   // a mismatch, then 60 matches

// the smallest score of a suffix of the last 30 columns; >= 0: the path may be trimmed here (TABLE and SCORE of
// dalign/align.c:884-896)
__device__ __forceinline__ int min_suffix(const PackLds& L, int w_match, int w_all, uint64_t N)
{
    const uint32_t z = (uint32_t)(N >> 3) & 0x3fffffffu;
    const int s1 = 10 * w_match - mul24(__popc(z & 0x3ffu), w_all);
    const int s2 = 20 * w_match - mul24(__popc(z & 0xfffffu), w_all);
    const int q0 = L.suf[z & 0x3ffu], q1 = L.suf[(z >> 10) & 0x3ffu] + s1, q2 = L.suf[z >> 20] + s2;
    return min(q0, min(q1, q2));
}

__device__ __forceinline__ void pack_tables(PackLds& L, const DevSpec& sp)
{
    const int lane = __lane_id();
    for (int i = lane; i < (1 << kSufBits); i += 64) L.suf[i] = sp.table[(~i & 0x3ff) | 0x7c00];
    const int none = sp.table[32768], all = sp.table[32768 + 0x7fff];   // 15 mismatches / matches
    if (lane == 0) {
        L.sp = sp;
        L.w_match = all / 15;
        L.w_all = (all - none) / 15;
        L.many = 0;
    }
    // both halves idle: the loop reads every field of a slot, also of one that never gets an alignment
    int* z = (int*)L.slot;
    for (int i = lane; i < (int)(sizeof(L.slot) / sizeof(int)); i += 64) z[i] = 0;
    z = (int*)L.band;
    for (int i = lane; i < (int)(sizeof(L.band) / sizeof(int)); i += 64) z[i] = 0;
    z = (int*)L.hot;
    for (int i = lane; i < (int)(sizeof(L.hot) / sizeof(int)); i += 64) z[i] = 0;
    wave_sync();
    if (lane < 2) {
        L.slot[lane].phase = PH_IDLE;
        L.slot[lane].a = 1;
        L.slot[lane].amin = kFar;
        L.slot[lane].bmax = -kFar;
    }
    wave_sync();
}

// ---- many trace points in one wave ------------------------------------------------------
// A diagonal whose path reached trace point t (those below t are done) pushes a
// pebble there unless the path's pebble lies at or beyond t.  The 8 low bits
// of the pebble's number settle that while it lies less than 128 points beyond
// t (it is never more than one before t).  A diagonal takes a neighbour's
// path one wave after the neighbour got there and had by then, at least, come
// as far as the neighbour one wave earlier; so the pebble lies at most as many
// points beyond t as some diagonal passed in the wave before.  That is 128 or
// more only in an exact run of that length: both neighbours of a diagonal run
// through a tandem repeat in one wave, the diagonal itself stays.  So only a
// wave after one that passed kManyPoints points looks at the paths that end
// that many points beyond t (a pebble lies on its path), and reads the marks of
// their pebbles: pack_skip between two waves of the halves' loop, wide_run
// instead of the numbers.  (Looking in every wave that crosses trace points
// cost 2.7 % on the 5 Mbp block, 172.9 -> 177.7 ms a pass.)
constexpr int kManyPoints = 120;
constexpr unsigned kMany = 4;          // beside the halves to serve: `many` is set
__device__ __forceinline__ int many_points(int TS) { return TS <= INT32_MAX / kManyPoints ? kManyPoints * TS : INT32_MAX; }
// The first point from t on that lies beyond pebble h (point n lies at n TS + off): no point before it needs a pebble.
__device__ __forceinline__ int skip_points(const Glob<Int4>* pool, int h, int t, int TS, int off, int m)
{
    const int p = ((pool[h & kPebIdx][3] ^ m) - m) - off;   // the pebble's mark, in the pass's direction
    const int n = p / TS;
    return max(t, n - (n * TS > p ? 1 : 0) + 1);
}

// ---- a pass over the whole wave -----------------------------------------------------
// Takes the pass of slot h after the trim of a wave (its diagonals in L->band[h],
// lanes slot.a .. slot.b) and runs it with 64 NCH diagonals until its
// band is at most kNarrow wide (running = 1, the diagonals handed back before
// their wave's trace points and records) or it ends (running = 0, status).
// slot.dif < 0: the pass begins here, a forward pass from more diagonals than
// a half holds.
// Index i of the window (lane i & 63 of chunk i >> 6) holds diagonal kt - i.
template <int NCH>
__device__ __noinline__ void wide_run(PackLds* L, int h, const int* abort_flag)
{
    constexpr int W = 64 * NCH;
    const int lane = __lane_id();
    int many = uni(L->many);
    PackSlot& S = L->slot[h];
    PackHot& H = L->hot[h];
    PackBand& D = L->band[h];
    const int TS = uni(L->sp.tspace), ave = uni(L->sp.ave_path);
    const int alen = uni(S.alen), blen = uni(S.blen);
    const int m = uni(S.phase) == PH_REV ? -1 : 0;
    const int boff = uni(S.comp) ? blen % TS : 0;
    const int offB = (boff ^ m) - m;
    const int limA = alen & ~m, limB = blen & ~m;
    SeqWord* A = (SeqWord*)uni(S.A);
    SeqWord* B = (SeqWord*)uni(S.B);
    Glob<Int4>* pool = (Glob<Int4>*)uni(S.pool);
    const int w_match = uni(L->w_match), w_all = uni(L->w_all);
    const int cap = uni(S.pool_cap);
    int a = uni(S.a), b = uni(S.b), kt = uni(S.ktop), besta = uni(S.besta), lasta = uni(S.lasta), dif = uni(S.dif);
    int navail = uni(S.navail), amin = uni(S.amin), bmax = uni(S.bmax);
    int cells = 0, snake = 0, status = LA_OK;

    int V[NCH], M[NCH], HA[NCH], HB[NCH], tA[NCH], tB[NCH], y[NCH];
    uint64_t N[NCH];
    bool end[NCH];
    bool fresh = dif < 0, undef = false;
    if (fresh) {   // wave 0 (dalign/align.c:455-587)
        const int hi = uni(S.hgh), wd = hi - uni(S.low) + 1, mida = uni(S.anti);
        const int minp = uni(S.minp), maxp = uni(S.maxp);
        a = (W - wd) / 2;
        b = a + wd - 1;
        kt = hi + a;
        amin = maxp == INT32_MAX ? -kFar : kt - maxp;
        bmax = minp == -INT32_MAX ? kFar : kt - minp;
        dif = 0;
        besta = lasta = mida;
        navail = 2 * wd;
        if (wd > W) status = LA_WIDE;
#pragma unroll
        for (int j = 0; j < NCH; j++) {
            const int i = 64 * j + lane, k = kt - i;
            V[j] = kSentV;
            M[j] = HA[j] = HB[j] = tA[j] = tB[j] = y[j] = 0;
            N[j] = kColsInit;
            end[j] = false;
            const bool in = i >= a && i <= b && status == LA_OK;
            int lim = 0;
            if (in) {
                y[j] = (mida - k) >> 1;
                const int x = y[j] + k;
                const bool bad = y[j] < 0 || y[j] > blen || x < 0 || x > alen;
                undef |= bad;
                tA[j] = x / TS + 1;
                tB[j] = (y[j] + (TS - boff)) / TS;
                HA[j] = 2 * (i - a);
                HB[j] = HA[j] + 1;
                pool[HA[j]] = Int4{-1, k, 0, (tA[j] - 1) * TS};
                pool[HB[j]] = Int4{-1, k, 0, (tB[j] - 1) * TS + boff};
                HA[j] |= (int)((unsigned)(tA[j] - 1) << 24);
                HB[j] |= (int)((unsigned)(tB[j] - 1) << 24);
                M[j] = kPathLen;
                if (i == a) {
                    H.best_y = H.tr_y = y[j];
                    H.tr_c = mida;
                    H.tr_d = 0;
                    H.tr_ha = 0;
                    H.tr_hb = 1;
                    H.mo_m = -1;
                }
                lim = bad ? 0 : min(alen - x, blen - y[j]);
            }
            const int s = snake_len(A, B, 0, y[j] + k, y[j], lim, lim > 0);
            if (in) {
                end[j] = s == lim;
                snake += s + 1;
                y[j] += s;
                V[j] = 2 * y[j] + k;
            }
        }
        if (status == LA_OK && any_lane(undef)) status = LA_UNDEF;
    } else {
        const int wd = b - a + 1, d = (wd <= kOneChunk ? 64 - wd : W - wd) / 2 - a;
#pragma unroll
        for (int j = 0; j < NCH; j++) {
            const int i = 64 * j + lane - d;   // lane in the half
            const bool in = i >= a && i <= b;
            V[j] = in ? D.V[i & 31] : kSentV;
            M[j] = in ? D.M[i & 31] & (kEnd - 1) : 0;
            HA[j] = in ? D.HA[i & 31] : 0;
            HB[j] = in ? D.HB[i & 31] : 0;
            tA[j] = in ? D.tA[i & 31] : 0;
            tB[j] = in ? D.tB[i & 31] : 0;
            N[j] = in ? D.N[i & 31] : 0;
            y[j] = 0;
            end[j] = false;
        }
        a += d;
        b += d;
        kt += d;
        amin += d;
        bmax += d;
    }
    // chunks wholly outside the band hold sentinels only
    auto live = [&](int j) { return 64 * j <= b && 64 * j + 63 >= a; };

    while (status == LA_OK) {
        if (!fresh) {
            // ---- the next wave: band one wider on each side (dalign/align.c:645-743)
            const bool ea = a - 1 >= amin, eb = b + 1 <= bmax;
            int na = ea ? a - 1 : a, nb = eb ? b + 1 : b;
            const int wd = nb - na + 1;
            if (na < 0 || nb >= W || (NCH > 1 && wd <= kOneChunk && (na >> 6) != (nb >> 6))) {
                if (wd > W) {
                    status = LA_WIDE;
                    break;
                }
                const int d = na - (wd <= kOneChunk ? 64 - wd : W - wd) / 2;   // index i takes index i + d
                int v2[NCH], m2[NCH], ha2[NCH], hb2[NCH], ta2[NCH], tb2[NCH];
                uint64_t n2[NCH];
#pragma unroll
                for (int j = 0; j < NCH; j++) {
                    const int s = 64 * j + lane + d;
                    v2[j] = kSentV;
                    m2[j] = ha2[j] = hb2[j] = ta2[j] = tb2[j] = 0;
                    n2[j] = 0;
#pragma unroll
                    for (int q = 0; q < NCH; q++) {
                        const bool hit = s >= 64 * q && s < 64 * q + 64;
                        const int v_ = bperm(V[q], s & 63), m_ = bperm(M[q], s & 63), ha_ = bperm(HA[q], s & 63);
                        const int hb_ = bperm(HB[q], s & 63), ta_ = bperm(tA[q], s & 63), tb_ = bperm(tB[q], s & 63);
                        const uint64_t n_ = bperm64(N[q], s & 63);
                        if (hit) {
                            v2[j] = v_;
                            m2[j] = m_;
                            ha2[j] = ha_;
                            hb2[j] = hb_;
                            ta2[j] = ta_;
                            tb2[j] = tb_;
                            n2[j] = n_;
                        }
                    }
                }
#pragma unroll
                for (int j = 0; j < NCH; j++) {
                    V[j] = v2[j];
                    M[j] = m2[j];
                    HA[j] = ha2[j];
                    HB[j] = hb2[j];
                    tA[j] = ta2[j];
                    tB[j] = tb2[j];
                    N[j] = n2[j];
                }
                na -= d;
                nb -= d;
                kt -= d;
                amin -= d;
                bmax -= d;
            }
            a = na;
            b = nb;
            dif += 1;
            // ---- predecessors (dalign/align.c:760-791, :1498-1529) from the old values
            int am[NCH], ap[NCH];   // k - 1 (index + 1) and k + 1 (index - 1)
#pragma unroll
            for (int j = 0; j < NCH; j++) {
                am[j] = from_above(V[j]);
                ap[j] = from_below(V[j]);
                if (j + 1 < NCH) {
                    const int e = rdl(V[j + 1], 0);
                    if (lane == 63) am[j] = e;
                }
                if (j > 0) {
                    const int e = rdl(V[j - 1], 63);
                    if (lane == 0) ap[j] = e;
                }
            }
            // new end diagonals take the thresholds of their inner neighbour
            if (ea) {
                const int s = a + 1;
                int u = 0, w = 0;
#pragma unroll
                for (int j = 0; j < NCH; j++)
                    if ((s >> 6) == j) {
                        u = rdl(tA[j], s & 63);
                        w = rdl(tB[j], s & 63);
                    }
#pragma unroll
                for (int j = 0; j < NCH; j++)
                    if (64 * j + lane == a) {
                        tA[j] = u;
                        tB[j] = w;
                    }
            }
            if (eb) {
                const int s = b - 1;
                int u = 0, w = 0;
#pragma unroll
                for (int j = 0; j < NCH; j++)
                    if ((s >> 6) == j) {
                        u = rdl(tA[j], s & 63);
                        w = rdl(tB[j], s & 63);
                    }
#pragma unroll
                for (int j = 0; j < NCH; j++)
                    if (64 * j + lane == b) {
                        tA[j] = u;
                        tB[j] = w;
                    }
            }
            int gM[NCH], gHA[NCH], gHB[NCH];
            uint64_t gN[NCH];
#pragma unroll
            for (int j = 0; j < NCH; j++) {
                gM[j] = M[j];
                gHA[j] = HA[j];
                gHB[j] = HB[j];
                gN[j] = N[j];
                if (!live(j)) continue;
                const int mx = max(am[j], ap[j]);
                const int sel = V[j] < mx ? (am[j] >= ap[j] ? 1 : -1) : 0;
                const int src = (lane + sel) & 63;
                gM[j] = bperm(M[j], src);
                gHA[j] = bperm(HA[j], src);
                gHB[j] = bperm(HB[j], src);
                gN[j] = bperm64(N[j], src);
                if (j + 1 < NCH) {
                    const int m_ = rdl(M[j + 1], 0), ha_ = rdl(HA[j + 1], 0), hb_ = rdl(HB[j + 1], 0);
                    const uint64_t n_ = rdl64(N[j + 1], 0);
                    if (lane == 63 && sel == 1) {
                        gM[j] = m_;
                        gHA[j] = ha_;
                        gHB[j] = hb_;
                        gN[j] = n_;
                    }
                }
                if (j > 0) {
                    const int m_ = rdl(M[j - 1], 63), ha_ = rdl(HA[j - 1], 63), hb_ = rdl(HB[j - 1], 63);
                    const uint64_t n_ = rdl64(N[j - 1], 63);
                    if (lane == 0 && sel == -1) {
                        gM[j] = m_;
                        gHA[j] = ha_;
                        gHB[j] = hb_;
                        gN[j] = n_;
                    }
                }
            }
#pragma unroll
            for (int j = 0; j < NCH; j++) {
                M[j] = gM[j];
                HA[j] = gHA[j];
                HB[j] = gHB[j];
                N[j] = gN[j];
                end[j] = false;
                if (!live(j)) {
                    V[j] = kSentV;
                    continue;
                }
                const int i = 64 * j + lane, k = kt - i;
                const bool in = i >= a && i <= b;
                const int mx = max(am[j], ap[j]);
                int c = V[j] < mx ? mx + 1 : V[j] + 2;
                if (in) y[j] = (c - k) >> 1;
                const int x = y[j] + k, lim = in ? min(limA - x, limB - y[j]) : 0;
                undef |= lim < 0;
                const int s = max(snake_len(A, B, m, x, y[j], lim, lim > 0), 0);
                V[j] = kSentV;
                if (in) {
                    end[j] = s == lim;
                    snake += s + 1;
                    add_columns(N[j], M[j], s);
                    y[j] += s;
                    V[j] = 2 * y[j] + k;
                }
            }
            if (any_lane(undef)) {
                status = LA_UNDEF;
                break;
            }
            // ---- narrow again: back to the half
            if (b - a + 1 <= kNarrow) {
                bool e = false;
#pragma unroll
                for (int j = 0; j < NCH; j++) e |= end[j];
                if (!any_lane(e)) {
                    const int d = a - (1 + (kHalfBand - (b - a + 1)) / 2);
#pragma unroll
                    for (int j = 0; j < NCH; j++) {
                        const int i = 64 * j + lane - d;
                        if (i >= 0 && i < 32) {
                            D.V[i] = V[j];
                            D.M[i] = M[j];
                            D.HA[i] = HA[j];
                            D.HB[i] = HB[j];
                            D.tA[i] = tA[j];
                            D.tB[i] = tB[j];
                            D.N[i] = N[j];
                        }
                    }
                    if (lane == 0) {
                        S.a = a - d;
                        S.b = b - d;
                        S.ktop = kt - d;
                        S.amin = amin - d;
                        S.bmax = bmax - d;
                        S.besta = besta;
                        S.lasta = lasta;
                        S.dif = dif;
                        S.navail = navail;
                        S.running = 1;
                    }
                    break;
                }
            }
        }
        fresh = false;
        // ---- trace-point pebbles (dalign/align.c:826-878, :1562-1612)
        bool full = false;
        for (int n = 0;; n++) {   // n: points passed
            bool any = false;
            bool wA[NCH], wB[NCH];
#pragma unroll
            for (int j = 0; j < NCH; j++) {
                const int i = 64 * j + lane;
                const bool in = i >= a && i <= b;
                wA[j] = in && y[j] + kt - i >= point_at<NCH>(tA[j], TS);
                wB[j] = in && y[j] >= point_at<NCH>(tB[j], TS) + offB;
                any |= wA[j] | wB[j];
            }
            if (!any_lane(any)) {
                many = n >= kManyPoints ? 1 : 0;
                break;
            }
            if (many) wave_sync();   // pebbles of this wave's other lanes
#pragma unroll
            for (int j = 0; j < NCH; j++) {
                if (!live(j)) continue;
                const int k = kt - (64 * j + lane);
                bool pA = wA[j] && (dif == 0 || (int)(((unsigned)tA[j] << 24) - ((unsigned)HA[j] & ~(unsigned)kPebIdx)) > 0);
                bool pB = wB[j] && (dif == 0 || (int)(((unsigned)tB[j] << 24) - ((unsigned)HB[j] & ~(unsigned)kPebIdx)) > 0);
                if (many) {   // (see skip_points; the marks themselves)
                    if (wA[j]) pA = dif == 0 || ((pool[HA[j] & kPebIdx][3] ^ m) - m) < point_at<NCH>(tA[j], TS);
                    if (wB[j]) pB = dif == 0 || ((pool[HB[j] & kPebIdx][3] ^ m) - m) < point_at<NCH>(tB[j], TS) + offB;
                }
                const unsigned long long ba = ballot(pA), bb = ballot(pB);
                const int ca = __popcll(ba), cb = __popcll(bb);
                if (navail + ca + cb > cap) {
                    full = true;
                    break;
                }
                if (pA) {
                    const int q = navail + prefix_rank(ba);
                    pool[q] = Int4{HA[j] & kPebIdx, (k ^ m) - m, dif, ((tA[j] * TS) ^ m) - m};
                    HA[j] = q | (int)((unsigned)tA[j] << 24);
                }
                if (pB) {
                    const int q = navail + ca + prefix_rank(bb);
                    pool[q] = Int4{HB[j] & kPebIdx, (k ^ m) - m, dif, ((tB[j] * TS + offB) ^ m) - m};
                    HB[j] = q | (int)((unsigned)tB[j] << 24);
                }
                navail += ca + cb;
                if (wA[j]) tA[j] += 1;
                if (wB[j]) tB[j] += 1;
            }
            if (full) break;
        }
        if (full) {
            status = LA_POOL;
            break;
        }
        // ---- records in visiting order
        {
            int carry = besta;
#pragma unroll
            for (int j = 0; j < NCH; j++) {
                if (!live(j)) continue;
                const int incl = prefix_max<true>(V[j]);
                const int e = __builtin_amdgcn_update_dpp(carry, incl, 0x138, 0xF, 0xF, false);
                const bool rec = V[j] > max(e, carry);
                carry = max(carry, rdl(incl, 63));
                if (rec && V[j] == carry) H.best_y = y[j];
                const bool good = rec && (dif == 0 || M[j] >= ave);
                const unsigned long long bm = ballot(good);
                if (bm) {
                    lasta = rdl(V[j], highest_lane(bm));
                    const unsigned long long bt = ballot(good && (dif == 0 || min_suffix(*L, w_match, w_all, N[j]) >= 0));
                    if (bt && lane == highest_lane(bt)) {
                        H.tr_c = V[j];
                        H.tr_y = y[j];
                        H.tr_d = dif;
                        H.tr_ha = HA[j] & kPebIdx;
                        H.tr_hb = HB[j] & kPebIdx;
                    }
                }
            }
            besta = carry;
        }
        cells += b - a + 1;
        // ---- clips at the read ends (dalign/align.c:912-944, :1650-1686)
        int more = 1;
        {
            int la = -1, lb = INT32_MAX;   // lowest k that reached A's end, highest k that reached B's
            bool any = false;
#pragma unroll
            for (int j = 0; j < NCH; j++) {
                if (!live(j)) continue;
                const unsigned long long eb_ = ballot(end[j] && y[j] == limB);
                const unsigned long long ea_ = ballot(end[j] && y[j] != limB);
                if (ea_) la = 64 * j + highest_lane(ea_);
                if (eb_) lb = min(lb, 64 * j + lowest_lane(eb_));
                any |= (ea_ | eb_) != 0;
            }
            if (any) {
                wave_sync();
                const int by = uni(H.best_y);
                more = (by == limB || besta - by == limA) ? 0 : 1;
#pragma unroll
                for (int q = 0; q < 2; q++) {
                    const int at = q == 0 ? la : lb;
                    const bool hit = q == 0 ? (la >= a) : (lb <= b);   // (la = -1 / lb = INT32_MAX: none)
                    if (!hit) continue;
                    if (q == 0) a = at + 1;
                    else b = at - 1;
                    const int mo = uni(H.mo_m);
#pragma unroll
                    for (int j = 0; j < NCH; j++)
                        if (64 * j + lane == at && mo <= M[j]) {
                            H.mo_m = M[j];
                            H.mo_c = V[j];
                            H.mo_y = y[j];
                            H.mo_d = dif;
                            H.mo_ha = HA[j] & kPebIdx;
                            H.mo_hb = HB[j] & kPebIdx;
                        }
                    wave_sync();
                }
            }
        }
        // ---- WAVE_LAG trim of the band's ends (dalign/align.c:946-955, :1688-1697)
        {
            const int n = dif > 0 ? besta - kWaveLag : kSentV + 1;
            int na2 = INT32_MAX, nb2 = -1;
#pragma unroll
            for (int j = 0; j < NCH; j++) {
                const int i = 64 * j + lane;
                const unsigned long long bk = ballot(i >= a && i <= b && V[j] >= n);
                if (bk) {
                    na2 = min(na2, 64 * j + lowest_lane(bk));
                    nb2 = 64 * j + highest_lane(bk);
                }
            }
            a = na2;
            b = nb2;
        }
#pragma unroll
        for (int j = 0; j < NCH; j++) {
            const int i = 64 * j + lane;
            if (i < a || i > b) V[j] = kSentV;
        }
        // ---- go on?
        if (!(more && lasta >= besta - kTrimMLag)) break;
        if (b < a || dif > 2 * (alen + blen) + 1024) {
            status = LA_UNDEF;   // empty band with the loop still running
            break;
        }
        if ((dif & 255) == 255 && uni(__atomic_load_n(abort_flag, __ATOMIC_RELAXED))) {
            status = LA_ABORT;
            break;
        }
    }
    int t = snake;
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) t += __shfl_xor(t, o, 64);
    if (lane == 0) {
        S.snake += t;
        S.cells += cells;
        if (!S.running) {
            S.status = status;
            S.used = navail;
            S.dif = dif;
        } else if (many) L->many = 1;
    }
    wave_sync();
}

// ---- between passes ------------------------------------------------------------------

// The pass of slot h ended: its chains are assembled, then the reverse pass
// or the job's next alignment is set up (phase PH_IDLE: none left).
template <class Job>
__device__ __noinline__ void pack_service(Job job, PackLds* L, int h)
{
    const int lane = __lane_id();
    PackSlot& S = L->slot[h];
    const PackHot& H = L->hot[h];
    const int TS = uni(L->sp.tspace);
    const int phase = uni(S.phase);
    if (phase != PH_IDLE) {
        const bool rev = phase == PH_REV;
        int status = uni(S.status);
        if (lane == 0) {
            S.steps += S.dif + 1;
            if (status == LA_OK) S.snake0 = S.snake;
            else S.snake = S.snake0;   // a pass that failed counts its cells only
        }
        const int alen = uni(S.alen), blen = uni(S.blen), comp = uni(S.comp), anti = uni(S.anti);
        const int boff = comp ? blen % TS : 0;
        const int maxtp = uni(S.maxtp);
        uint16_t *atr = uni(S.atr), *btr = uni(S.btr);
        if (status == LA_OK) {
            const bool mo = uni(H.mo_m) >= 0;
            const int c = mo ? uni(H.mo_c) : uni(H.tr_c), yy = mo ? uni(H.mo_y) : uni(H.tr_y);
            const int trimd = mo ? uni(H.mo_d) : uni(H.tr_d);
            const int tha = mo ? uni(H.mo_ha) : uni(H.tr_ha), thb = mo ? uni(H.mo_hb) : uni(H.tr_hb);
            const int trimx = rev ? yy - c : c - yy, trimy = rev ? -yy : yy;
            Peb* pool = uni(S.pool);
            const int pts_cap = uni(S.pts_cap);
            const bool isB = lane == 1;
            Peb* pts = uni(S.pts) + (isB ? pts_cap : 0);
            int len = 0, first = 0, rootk = 0;
            bool ok = true;
            if (lane < 2) {
                if (!rev)
                    ok = assemble_chain<+1>(pool, S.used, pts, pts_cap, isB ? thb : tha, isB, anti, TS, boff, trimx,
                                            trimy, trimd, isB ? btr : atr, maxtp, 0, &len, &first, &rootk);
                else
                    ok = assemble_chain<-1>(pool, S.used, pts, pts_cap, isB ? thb : tha, isB, anti, TS, boff, trimx,
                                            trimy, trimd, isB ? btr : atr, maxtp, isB ? S.fb : S.fa, &len, &first,
                                            &rootk);
            }
            const int la = rdl(len, 0), lb = rdl(len, 1);
            if (__any(!ok)) {
                status = LA_CHAIN;
            } else if (!rev) {
                if (lane == 0) {
                    S.fa = la;
                    S.fb = lb;
                    S.res.aepos = trimx;
                    S.res.bepos = trimy;
                    S.res.diffs = trimd;
                    if (comp) {
                        S.res.b_abpos = blen - trimy;
                        S.res.b_bbpos = alen - trimx;
                    } else {
                        S.res.b_aepos = trimy;
                        S.res.b_bepos = trimx;
                    }
                }
                const int mind = rdl(rootk, 1);   // the B chain's root (dalign/align.c:1059-1061)
                if (lane == 0) {
                    S.mind = mind;
                    S.phase = PH_REV;
                }
                wave_sync();   // the pool is used again
                return;
            } else {
                const int af = rdl(first, 0), bf = rdl(first, 1);
                const int atlen = uni(S.fa) + la, btlen = uni(S.fb) + lb;
                if (lane == 0) {
                    S.res.afirst = af;
                    S.res.bfirst = bf;
                    S.res.atlen = atlen;
                    S.res.btlen = btlen;
                    S.res.abpos = trimx;
                    S.res.bbpos = trimy;
                    S.res.diffs += trimd;
                    if (comp) {
                        S.res.b_aepos = blen - trimy;
                        S.res.b_bepos = alen - trimx;
                    } else {
                        S.res.b_abpos = trimy;
                        S.res.b_bbpos = trimx;
                    }
                }
                wave_sync();
                if (comp) {   // B-view trace runs the other way (dalign/align.c:2004-2023)
                    uint16_t* t = btr + bf;
                    const int npair = btlen / 2;
                    for (int p = lane; p < npair / 2; p += 64) {
                        const int q = npair - 1 - p;
                        const uint16_t a0 = t[2 * p], a1 = t[2 * p + 1];
                        const uint16_t b0 = t[2 * q], b1 = t[2 * q + 1];
                        t[2 * p] = b0;
                        t[2 * p + 1] = b1;
                        t[2 * q] = a0;
                        t[2 * q + 1] = a1;
                    }
                    wave_sync();
                }
            }
        }
        if (lane == 0) S.res.status = status;
        wave_sync();
        job.done(*L, h);
    }
    const bool some = job.next(*L, h);
    if (lane == 0) {
        S.phase = some ? PH_FWD : PH_IDLE;
        S.cells = S.snake = S.steps = S.snake0 = 0;
    }
    wave_sync();
}

// Wave 0 of the pass of slot h (dalign/align.c:455-587, :1193-1322) into its
// PackBand, or the status that keeps the pass from starting.
static __device__ __noinline__ void pass_begin(PackLds* L, int h)
{
    const int lane = __lane_id(), sl = lane & 31;
    PackSlot& S = L->slot[h];
    PackHot& H = L->hot[h];
    PackBand& D = L->band[h];
    const int TS = uni(L->sp.tspace);
    const bool rev = uni(S.phase) == PH_REV;
    const int m = rev ? -1 : 0;
    const int alen = uni(S.alen), blen = uni(S.blen), mida = uni(S.anti), cap = uni(S.pool_cap);
    const int mind = uni(S.mind), minp = uni(S.minp), maxp = uni(S.maxp);
    const int lo = rev ? -mind : uni(S.low), hi = rev ? -mind : uni(S.hgh);
    const int boff = uni(S.comp) ? blen % TS : 0;
    const int wd = hi - lo + 1;
    const int a = 1 + (kHalfBand - wd) / 2, b = a + wd - 1, k = hi + a - sl;
    int status = LA_OK;
    if (2 * wd > cap || cap > kPoolMax) status = LA_POOL;
    else if (wd > kHalfBand) status = LA_GROW;
    bool bad = false;
    const bool in = status == LA_OK && lane >= a && lane <= b;
    int HA = 0, HB = 0, tA = 0, tB = 0, y = 0, lim = 0;
    if (in) {
        Glob<Int4>* pool = (Glob<Int4>*)S.pool;
        const int kr = (k ^ m) - m;
        const int yr = (mida - kr) >> 1, xr = yr + kr;
        bad = yr < 0 || yr > blen || xr < 0 || xr > alen;
        int ma, mb;   // the roots' marks
        if (!rev) {
            const int na = xr / TS, nb = (yr + (TS - boff)) / TS - 1;
            tA = na + 1;
            tB = nb + 1;
            ma = na * TS;
            mb = nb * TS + boff;
        } else {
            tA = -((xr + TS - 1) / TS - 1);
            tB = -((yr + (TS - boff) - 1) / TS - 1);
            ma = xr;
            mb = yr;
        }
        HA = 2 * (sl - a);
        HB = HA + 1;
        pool[HA] = Int4{-1, kr, 0, ma};
        pool[HB] = Int4{-1, kr, 0, mb};
        HA |= (int)((unsigned)(tA - 1) << 24);
        HB |= (int)((unsigned)(tB - 1) << 24);
        y = (yr ^ m) - m;
        if (sl == a) {
            H.best_y = H.tr_y = y;
            H.tr_c = rev ? -mida : mida;
            H.tr_d = 0;
            H.tr_ha = 0;
            H.tr_hb = 1;
            H.mo_m = -1;
        }
        lim = bad ? 0 : min((rev ? 0 : alen) - (y + k), (rev ? 0 : blen) - y);
    }
    int snake = snake_len((SeqWord*)uni(S.A), (SeqWord*)uni(S.B), m, y + k, y, lim, lim > 0);
    if (lane < 32) {
        // the columns of a first wave are matches only
        D.V[sl] = in ? 2 * (y + snake) + k : kSentV;
        D.M[sl] = kPathLen | (in && snake == lim ? kEnd : 0);
        D.HA[sl] = HA;
        D.HB[sl] = HB;
        D.tA[sl] = tA;
        D.tB[sl] = tB;
        D.N[sl] = kColsInit;
    }
    snake = in ? snake + 1 : 0;
    if (any_lane(bad)) status = LA_UNDEF;
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) snake += __shfl_xor(snake, o, 64);
    if (lane == 0) {
        // borders as lanes
        const int mn = rev ? (maxp == INT32_MAX ? -INT32_MAX : -maxp) : minp;
        const int mx = rev ? (minp == -INT32_MAX ? INT32_MAX : -minp) : maxp;
        S.amin = mx == INT32_MAX ? -kFar : hi + a - mx;
        S.bmax = mn == -INT32_MAX ? kFar : hi + a - mn;
        S.a = a;
        S.b = b;
        S.ktop = hi + a;
        S.navail = 2 * wd;
        S.dif = status == LA_GROW ? -1 : 0;   // (wide_run begins the pass)
        S.besta = S.lasta = rev ? -mida : mida;
        S.snake += snake;
        S.status = status;
    }
    wave_sync();
}

// The trace points that the paths in the PackBands have already are done.
// many: whether there were any, so that the next wave looks again.
template <int NCH>
__device__ __noinline__ void pack_skip(PackLds* L)
{
    const int lane = __lane_id(), sl = lane & 31;
    const PackSlot& S = L->slot[lane >> 5];
    PackBand& D = L->band[lane >> 5];
    const int TS = uni(L->sp.tspace), far = many_points(TS);
    const int m = S.phase == PH_REV ? -1 : 0;
    const int offB = ((S.comp ? S.blen % TS : 0) ^ m) - m;
    const int k = S.ktop - sl, y = (D.V[sl] - k) >> 1, tA = D.tA[sl], tB = D.tB[sl];
    const bool in = sl >= S.a && sl <= S.b;
    const bool fA = in && y + k - point_at<NCH>(tA, TS) >= far, fB = in && y - offB - point_at<NCH>(tB, TS) >= far;
    wave_sync();   // pebbles of the wave's other lanes
    Glob<Int4>* pool = (Glob<Int4>*)S.pool;
    if (fA) D.tA[sl] = skip_points(pool, D.HA[sl], tA, TS, 0, m);
    if (fB) D.tB[sl] = skip_points(pool, D.HB[sl], tB, TS, offB, m);
    if (lane == 0) L->many = 0;
    if (any_lane(fA || fB) && lane == 0) L->many = 1;
    wave_sync();
}

// The halves in `stopped` (bit 0: lanes 0..31): a pass that needs the wave
// gets it, one that ended is followed by the next.  Afterwards every slot
// holds a pass that goes on from its PackBand, or is idle with an empty band.
template <int NCH, class Job>
__device__ __noinline__ void pack_serve(Job job, PackLds* L, unsigned stopped, const int* abort_flag)
{
    const int lane = __lane_id();
    stopped = (unsigned)uni((int)stopped);
    for (int h = 0; h < 2; h++) {
        if (!((stopped >> h) & 1)) continue;
        PackSlot& S = L->slot[h];
        bool go = false;
        for (;;) {
            if (uni(S.phase) != PH_IDLE && uni(S.status) == LA_GROW) {
                wide_run<NCH>(L, h, abort_flag);
                go = uni(S.running) != 0;
                if (lane == 0) {
                    S.running = 0;
                    if (go) S.status = LA_OK;
                }
                wave_sync();
            }
            if (go) break;
            pack_service(job, L, h);
            if (uni(S.phase) == PH_IDLE) {
                if (lane == 0) {
                    S.a = 1;
                    S.b = 0;
                    S.amin = kFar;
                    S.bmax = -kFar;
                    S.prio = 0;
                }
                wave_sync();
                break;
            }
            pass_begin(L, h);
            go = uni(S.status) == LA_OK;
        }
    }
    set_priority(max(uni(L->slot[0].prio), uni(L->slot[1].prio)));
    if (uni(L->many)) pack_skip<NCH>(L);
}

// ---- the loop --------------------------------------------------------------------------
//
// `second`: the upper half takes alignments too.  A grid that has a wave for
// every alignment leaves it idle (the launch is then bound by its longest
// alignment, and a wave with one alignment steps faster than one with two).
template <int NCH, class Job>
__device__ __forceinline__ void pack_run(PackLds& L, Job job, bool second, const int* abort_flag)
{
    typedef unsigned long long Lanes;   // a set of lanes
    // What serving a half would have to keep is set again after it (see below).
    int lane = 0, sl = 0, hm = 0, TS = 0, ave = 0, w_all = 0, w_match = 0;
    PackSlot* S = nullptr;
    PackHot* H = nullptr;
    PackBand* D = nullptr;
    // per diagonal; V, M, N, HA, HB as the reference's V, M, T, HA, HB; tA / tB: the numbers of the next trace
    // points; rem: columns left to a read's end (0: the wave's snake ran into it)
    int V = kSentV, M = 0, HA = 0, HB = 0, tA = 0, tB = 0, y = 0, rem = 1;
    uint64_t N = 0;
    // per half (the same on its 32 lanes); an idle half has an empty band that no border lets grow
    int k = 0, a = 1, b = 0, besta = 0, lasta = 0, dif = 0, navail = 0, amin = kFar, bmax = -kFar;
    int limA = 0, limB = 0, m = 0, offB = 0, cap = 0;
    SeqWord *A = nullptr, *B = nullptr;
    Glob<Int4>* pool = nullptr;
    int ncell = 0, nsnake = 0;
    // wave-uniform
    Lanes act = 0, fresh = 0;                // halves with a pass; of these, in wave 0
    unsigned stopped = second ? 3u : 1u;     // halves to serve (bit 0: lanes 0..31), kMany
    unsigned tick = 0;

    for (;;) {
        if (stopped) {
            // Nothing stays in registers while the wave serves a half: the
            // other one's pass goes through LDS and everything else is set
            // again, so the loop does not pay for the registers of what it
            // calls.
            if (lane_in(act) && !((stopped >> (lane >> 5)) & 1)) {
                D->V[sl] = V;
                D->M[sl] = M | (rem == 0 ? kEnd : 0);
                D->HA[sl] = HA;
                D->HB[sl] = HB;
                D->tA[sl] = tA;
                D->tB[sl] = tB;
                D->N[sl] = N;
                if (sl == 0) {
                    S->a = a;
                    S->b = b;
                    S->ktop = k;
                    S->besta = besta;
                    S->lasta = lasta;
                    S->dif = dif;
                    S->navail = navail;
                    S->amin = amin;
                    S->bmax = bmax;
                }
            }
            if (tick) {   // (the first time there is nothing to hand over)
#pragma unroll
                for (int o = 16; o >= 1; o >>= 1) nsnake += __shfl_xor(nsnake, o, 64);
                if (sl == 0) {
                    S->cells += ncell;
                    S->snake += nsnake;
                }
            }
            wave_sync();
            pack_serve<NCH>(job, &L, stopped, abort_flag);
            stopped = uni(L.many) ? kMany : 0;
            lane = __lane_id();
#ifndef MI_CPU_WAVE_EMU
            asm volatile("" : "+v"(lane));   // computed here, not once before the loop
#endif
            sl = lane & 31;
            hm = -(lane >> 5);
            S = &L.slot[lane >> 5];
            H = &L.hot[lane >> 5];
            D = &L.band[lane >> 5];
            TS = uni(L.sp.tspace);
            ave = uni(L.sp.ave_path);
            w_all = uni(L.w_all);
            w_match = uni(L.w_match);
            const bool rev = S->phase == PH_REV;
            m = rev ? -1 : 0;
            limA = rev ? 0 : S->alen;
            limB = rev ? 0 : S->blen;
            const int boff = S->comp ? S->blen % TS : 0;
            offB = rev ? -boff : boff;
            A = (SeqWord*)S->A;
            B = (SeqWord*)S->B;
            pool = (Glob<Int4>*)S->pool;
            cap = S->pool_cap;
            a = S->a;
            b = S->b;
            k = S->ktop - sl;
            besta = S->besta;
            lasta = S->lasta;
            dif = S->dif;
            navail = S->navail;
            amin = S->amin;
            bmax = S->bmax;
            const bool in = sl >= a && sl <= b;
            V = in ? D->V[sl] : kSentV;
            M = D->M[sl];
            rem = in && (M & kEnd) ? 0 : 1;
            M &= kEnd - 1;
            HA = D->HA[sl];
            HB = D->HB[sl];
            tA = D->tA[sl];
            tB = D->tB[sl];
            N = D->N[sl];
            y = (V - k) >> 1;
            ncell = nsnake = 0;
            act = ballot(S->phase != PH_IDLE);
            if (!act) break;   // every half is idle
            fresh = act & ballot(dif == 0);
            wave_sync();
        }

        // ---- trace-point pebbles: wave 0 pushes always, later waves when the
        // inherited pebble does not already sit on the trace point
        // (dalign/align.c:521-563, :826-878, :1258-1297, :1562-1612)
        {
            const int x = y + k;
            int nA = point_at<NCH>(tA, TS), nB = point_at<NCH>(tB, TS) + offB;
            const Lanes in = ballot(sl >= a) & ballot(sl <= b);
            Lanes wA = in & ballot(x >= nA), wB = in & ballot(y >= nB);
            int n = 0;   // points passed
            while (wA | wB) {
                const Lanes pA = wA & (fresh | ballot((int)(((unsigned)tA << 24) - ((unsigned)HA & ~(unsigned)kPebIdx)) > 0));
                const Lanes pB = wB & (fresh | ballot((int)(((unsigned)tB << 24) - ((unsigned)HB & ~(unsigned)kPebIdx)) > 0));
                const int al = __popcll(pA & 0xffffffffull), bl = __popcll(pB & 0xffffffffull);
                const int ia = navail + prefix_rank(pA) - (hm & al);
                navail += hsel(hm, al, __popcll(pA >> 32));
                const int ib = navail + prefix_rank(pB) - (hm & bl);
                navail += hsel(hm, bl, __popcll(pB >> 32));
                const Lanes room = ballot(navail <= cap);   // (once there is none, the pass stops below)
                const int kr = (k ^ m) - m;
                if (lane_in(pA & room)) {
                    pool[(unsigned)ia] = Int4{HA & kPebIdx, kr, dif, (nA ^ m) - m};
                    HA = ia | (int)((unsigned)tA << 24);
                }
                if (lane_in(pB & room)) {
                    pool[(unsigned)ib] = Int4{HB & kPebIdx, kr, dif, (nB ^ m) - m};
                    HB = ib | (int)((unsigned)tB << 24);
                }
                tA += lane_in(wA) ? 1 : 0;
                tB += lane_in(wB) ? 1 : 0;
                nA = point_at<NCH>(tA, TS);
                nB = point_at<NCH>(tB, TS) + offB;
                wA &= ballot(x >= nA);
                wB &= ballot(y >= nB);
                n++;
            }
            if (n >= kManyPoints) {
                stopped = kMany;
                L.many = 1;
            }
        }

        // ---- records: strict improvements of besta in lane order
        {
            const int incl = prefix_max<false>(V);
            int e = dpp_shr1(incl);
            e = sl == 0 ? besta : max(e, besta);
            besta = max(besta, bperm(incl, lane | 31));
            const Lanes rec = ballot(V > e);
            if (lane_in(rec & ballot(V == besta))) H->best_y = y;
            const Lanes good = rec & (fresh | ballot(M >= ave));
            if (good) {
                const uint32_t mm = hmask(hm, good);
                const int lv = bperm(V, (lane & 32) + top_bit(mm));
                lasta = mm ? lv : lasta;
                const Lanes trim = good & (fresh | ballot(min_suffix(L, w_match, w_all, N) >= 0));
                if ((hmask(hm, trim) >> sl) == 1u) {   // the last one in visiting order
                    H->tr_c = V;
                    H->tr_y = y;
                    H->tr_d = dif;
                    H->tr_ha = HA & kPebIdx;
                    H->tr_hb = HB & kPebIdx;
                }
            }
        }
        ncell += b - a + 1;

        // ---- clips at the read ends (dalign/align.c:589-625, :912-944, :1327-1361, :1650-1686)
        Lanes over = 0;   // halves whose best path reached a read's end
        const Lanes end = ballot(rem == 0);
        if (end) {
            wave_sync();
            const Lanes eB = end & ballot(y == limB);
            const uint32_t mB = hmask(hm, eB), mA = hmask(hm, end & ~eB);
            const int by = H->best_y;
            over = ballot((mA | mB) != 0) & (ballot(by == limB) | ballot(besta - by == limA));
            const int la = mA ? top_bit(mA) : -1, lb = mB ? low_bit(mB) : 32;
            const bool hitA = mA && la >= a;
            if (hitA && sl == la && H->mo_m <= M) {
                H->mo_m = M;
                H->mo_c = V;
                H->mo_y = y;
                H->mo_d = dif;
                H->mo_ha = HA & kPebIdx;
                H->mo_hb = HB & kPebIdx;
            }
            wave_sync();
            const bool hitB = mB && lb <= b;
            if (hitB && sl == lb && H->mo_m <= M) {
                H->mo_m = M;
                H->mo_c = V;
                H->mo_y = y;
                H->mo_d = dif;
                H->mo_ha = HA & kPebIdx;
                H->mo_hb = HB & kPebIdx;
            }
            wave_sync();
            if (hitA) a = la + 1;
            if (hitB) b = lb - 1;
            if (sl < a || sl > b) V = kSentV;
        }

        // ---- WAVE_LAG trim of the band's ends (dalign/align.c:946-955, :1688-1697)
        int lag = besta - kWaveLag;
        if (fresh) lag = lane_in(fresh) ? kSentV + 1 : lag;
        const uint32_t mk = hmask(hm, ballot(V >= lag));
        a = low_bit(mk);    // (an empty band: 31 .. 0)
        b = top_bit(mk);
        V = lane_in(ballot(sl >= a) & ballot(sl <= b)) ? V : kSentV;

        // ---- go on?  Then the band grows by one diagonal on each side (dalign/align.c:645-743)
        const Lanes ea = ballot(a > amin), eb = ballot(b < bmax);
        int na = a - (lane_in(ea) ? 1 : 0), nb = b + (lane_in(eb) ? 1 : 0);
        const Lanes run = ballot(lasta >= besta - kTrimMLag) & ~over;
        Lanes stop = act & (~run | ballot(mk == 0) | ballot(nb - na >= kHalfBand) | ballot(navail > cap));
        Lanes aborted = 0;
        if ((++tick & 255u) == 0) {
            if (uni(__atomic_load_n(abort_flag, __ATOMIC_RELAXED))) aborted = ~0ull;
            stop |= act & (aborted | ballot(dif > 2 * (S->alen + S->blen) + 1024));
        }
        if (stop) {
            if (lane_in(stop)) {
                int st = LA_OK;
                if (navail > cap) st = LA_POOL;
                else if (lane_in(run)) {
                    if (mk == 0) st = LA_UNDEF;   // empty band with the loop still running
                    else if (lane_in(aborted)) st = LA_ABORT;
                    else if (nb - na >= kHalfBand) st = LA_GROW;
                    else st = LA_UNDEF;
                }
                if (st == LA_GROW) {
                    D->V[sl] = V;
                    D->M[sl] = M;
                    D->HA[sl] = HA;
                    D->HB[sl] = HB;
                    D->tA[sl] = tA;
                    D->tB[sl] = tB;
                    D->N[sl] = N;
                }
                if (sl == 0) {
                    S->status = st;
                    S->used = S->navail = navail;
                    S->dif = dif;
                    S->a = a;
                    S->b = b;
                    S->ktop = k;   // lane 0's diagonal
                    S->besta = besta;
                    S->lasta = lasta;
                    S->amin = amin;
                    S->bmax = bmax;
                }
                na = 1;
                nb = 0;
                V = kSentV;
            }
            wave_sync();
            act &= ~stop;
            if (stop & 0xffffffffull) stopped |= 1u;
            if (stop >> 32) stopped |= 2u;
        }
        // lanes 0 and 31 stay free: move the band to the middle of its half
        if (ballot(na < 1) | ballot(nb > kHalfBand)) {
            const bool mv = na < 1 || nb > kHalfBand;
            const int d = mv ? na - (1 + (kHalfBand - (nb - na + 1)) / 2) : 0;   // lane L takes lane L + d
            const int src = lane + d;
            const bool ok = (src >> 5) == (lane >> 5);
            const int v2 = bperm(V, src);
            M = bperm(M, src);
            HA = bperm(HA, src);
            HB = bperm(HB, src);
            tA = bperm(tA, src);
            tB = bperm(tB, src);
            N = bperm64(N, src);
            V = ok ? v2 : kSentV;
            na -= d;
            nb -= d;
            k -= d;
            amin -= d;
            bmax -= d;
        }
        dif += 1;
        fresh = 0;
        a = na;
        b = nb;

        // ---- the next wave: predecessors (dalign/align.c:760-791, :1498-1529)
        {
            const int am = dpp_shl1(V), ap = dpp_shr1(V);   // k - 1, k + 1
            // a new end diagonal takes the thresholds of its inner neighbour
            const int t0 = lane + (lane_in(ea & ballot(sl == a)) ? 1 : 0) - (lane_in(eb & ballot(sl == b)) ? 1 : 0);
            tA = bperm(tA, t0);
            tB = bperm(tB, t0);
            const int mx = max(am, ap);
            const bool take = V < mx;
            const int src = lane + (take ? (am >= ap ? 1 : -1) : 0);
            const int c = take ? mx + 1 : V + 2;
            M = bperm(M, src);
            HA = bperm(HA, src);
            HB = bperm(HB, src);
            N = bperm64(N, src);
            const Lanes in = ballot(sl >= a) & ballot(sl <= b) & act;
            y = (c - k) >> 1;
            const int lim = lane_in(in) ? min(limA - (y + k), limB - y) : 0;
            const Lanes undef = ballot(lim < 0);
            const int s = snake_len(A, B, m, y + k, y, lim, lim > 0);
            rem = lane_in(in) ? lim - s : 1;
            nsnake += lane_in(in) ? s + 1 : 0;
            add_columns(N, M, s);
            y += s;
            V = lane_in(in) ? 2 * y + k : kSentV;
            if (undef) {
                const uint32_t mu = hmask(hm, undef);
                if (mu && sl == 0) {
                    S->status = LA_UNDEF;
                    S->used = navail;
                    S->dif = dif - 1;
                }
                wave_sync();
                act &= ~ballot(mu != 0);
                if (undef & 0xffffffffull) stopped |= 1u;
                if (undef >> 32) stopped |= 2u;
            }
        }
    }
}

}  // namespace mi
