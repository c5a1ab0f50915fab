// report_thread (dalign/filter.c:1617-1989) on gfx950: one half-wave per read
// pair while it aligns, the whole wave for what happens between alignments.
//
// The reference walks a pair's seeds (sorted by apos) in 50 kb panels that
// overlap by 10 kb.  Per panel it scores diagonal bands (band = diag >> w),
// then visits the seeds in order and aligns a seed when its band has enough
// score and the seed lies beyond the end of the last alignment that covered
// its band (lasta).  Each alignment then raises lasta over its diagonal span.
//
// Here a half of a wave owns the pair (la_pack.hpp runs its alignments) and
// the wave serves it in between:
//   * band scores: 64 seeds at a time; lanes in the same band find each other
//     with ballots, take the previous seed's apos from the lane below (or
//     the band's lastp), add min(K, apos - prev) with atomics, and the last
//     lane of the band stores lastp -- the order the sequential loop implies;
//   * gating: the 64 seeds of a chunk test the condition together, the first
//     passing lane is aligned, lasta is raised in parallel over the span, and
//     testing resumes after that seed;
//   * redundant alignments of the pair are fused by lane 0
//     (dalign/filter.c:1249-1566) and the records are appended to the output.
// The band arrays (score | lastp | lasta) of a half use the reference's
// per-thread layout, so neighbour reads at the outer bands see the same
// cells; any access outside [mindiag, maxdiag] is counted as an edge event.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "filter_kernels.hpp"
#include "la_pack.hpp"
#include "records.h"

namespace mi {

// statuses of a pair
constexpr int RP_OK = 0;
constexpr int RP_RETRY = 1;    // needs a wider band window or bigger pools
constexpr int RP_UNDEF = 3;    // an alignment reached a reference-undefined state
constexpr int RP_ARENA = 4;    // per-wave match arena too small
constexpr int RP_OUT = 5;      // output arena full (records not written)

struct MPath {   // a kept alignment of the pair (dalign/align.h:76-83 fields)
    int tlen, diffs, abpos, bbpos, aepos, bepos;
    long long toff;   // offset of its u16 trace in the half's trace pool
};


struct ReportArgs {
    const Seed* hits;
    const long long* pstart;   // seed range of pair p: [pstart[p], pstart[p+1])
    const int* jobs;           // pair index of every job
    const int* order;          // jobs of this launch
    int norder;
    const uint64_t* pkA;
    const long long* w0A;
    const int* lenA;
    const uint64_t* pkB;
    const long long* w0B;
    const int* lenB;
    int afirst, bfirst, comp, self, symmetric, hgap_min;
    int K, binshift, hitmin, minhit, minover, tspace, small_trace;
    int mindiag, maxdiag, w;
    DevSpec sp;
    // scratch of each half
    int* bands;         // (3w + 2) ints, zero on entry, left zero on exit
    Peb* pools;
    int pool_cap;
    Peb* pts;
    int pts_cap;
    uint16_t* latr;     // alignment trace scratch: 4 * maxtp_all
    int maxtp_all;
    MPath* mpaths;      // 2 * mcap (A list then B list)
    int mcap;
    uint16_t* mtrace;   // mtcap values
    long long mtcap;
    // the band cell shared by lastp[maxdiag] and lasta[mindiag-1]: its value
    // when the job starts (null: 0), at the end, and whether the job used it
    const int* edge_in;
    int* edge_out;
    int* touch;
    // outputs
    OutRec* orecs;
    long long ocap;
    uint8_t* otr;
    long long otcap;
    unsigned long long* ocount;   // [0] records, [1] trace bytes
    int* status;                  // per job
    int* final_gen;               // per job: launch of its last successful run
    int gen;                      // this launch
    int* counter;
    const int* abort_flag;
    unsigned long long* stats;    // [0] seeds aligned, [1] cells, [2] snake, [3] edge events, [4] wave steps
    unsigned long long* job_work; // optional, per job: band cells + snake steps of its last successful run
    unsigned* redund;             // optional, per job: kRedundBranches counters of handle_redundancies
};

// ---- redundancy handling (dalign/filter.c:1249-1566), lane 0 ------------------

__device__ int entwine(const MPath* jp, const MPath* kp, const uint16_t* T, int TS, int* where)
{
    const uint16_t* jt = T + jp->toff;
    const uint16_t* kt = T + kp->toff;
    int mn = 10000, den = 0, y2 = jp->bbpos, b2 = kp->bbpos, ac, i, j, k;
    const int jseg = jp->abpos / TS, kseg = kp->abpos / TS;
    if (jseg < kseg) {
        ac = kseg * TS;
        j = 1 + 2 * (kseg - jseg);
        k = 1;
        for (i = 1; i < j; i += 2) y2 += jt[i];
    } else {
        ac = jseg * TS;
        k = 1 + 2 * (jseg - kseg);
        j = 1;
        for (i = 1; i < k; i += 2) b2 += kt[i];
    }
    const int ae = jp->aepos < kp->aepos ? jp->aepos : kp->aepos;
    for (;;) {
        ac += TS;
        if (ac >= ae) break;
        y2 += jt[j];
        b2 += kt[k];
        j += 2;
        k += 2;
        i = y2 > b2 ? y2 - b2 : b2 - y2;
        if (i <= mn) {
            mn = i;
            if (i == 0) *where = ac;
        }
        den += 1;
    }
    return den == 0 ? -1 : mn;
}

// p1 up to A coordinate `at`, then p2; appends the new trace at *top
__device__ bool fusion(MPath* p1, int at, const MPath* p2, uint16_t* T, long long* top, long long cap, int TS)
{
    const int k1 = 2 * ((at / TS) - (p1->abpos / TS));
    const int k2 = 2 * ((at / TS) - (p2->abpos / TS));
    const int len = k1 + (p2->tlen - k2);
    if (*top + len > cap) return false;
    uint16_t* d = T + *top;
    const uint16_t* s1 = T + p1->toff;
    const uint16_t* s2 = T + p2->toff;
    int n = 0, diff = 0;
    for (int k = 0; k < k1; k += 2) {
        d[n++] = s1[k];
        d[n++] = s1[k + 1];
        diff += s1[k];
    }
    for (int k = k2; k < p2->tlen; k += 2) {
        d[n++] = s2[k];
        d[n++] = s2[k + 1];
        diff += s2[k];
    }
    p1->aepos = p2->aepos;
    p1->bepos = p2->bepos;
    p1->diffs = diff;
    p1->toff = *top;
    p1->tlen = n;
    *top += len;
    return true;
}

// Branch counters of handle_redundancies (pass statistics):
//   0 j starts first, k reaches further: fused, A and B views, COMP      4 j contains k: k replaced
//   1 the same, not COMP                                                  5 same start, j longer: k replaced
//   2 the same, A view only                                               6 k starts first, j reaches further: fused, A and B, COMP
//   3 (unused)                                                            7 the same, not COMP; 8 the same, A view only
constexpr int kRedundBranches = 9;

__device__ int handle_redundancies(MPath* am, int n, MPath* bm, uint16_t* T, long long* top, long long cap, int TS,
                                   int comp, bool* ok, unsigned (&br)[kRedundBranches])
{
    int no = 0, j, k, aw = 0, bw = 0;
    for (j = 1; j < n; j++) {
        MPath* jp = am + j;
        for (k = no; k >= 0; k--) {
            MPath* kp = am + k;
            if (jp->abpos < kp->abpos) {
                if (!(kp->abpos <= jp->aepos && kp->bbpos <= jp->bepos)) continue;
                if (entwine(jp, kp, T, TS, &aw) != 0) continue;
                if (kp->aepos > jp->aepos) {
                    if (bm) {
                        if (comp) {
                            if (entwine(bm + k, bm + j, T, TS, &bw) != 0) continue;
                            *ok &= fusion(jp, aw, kp, T, top, cap, TS);
                            am[k] = *jp;
                            *ok &= fusion(bm + k, bw, bm + j, T, top, cap, TS);
                            br[0]++;
                        } else {
                            if (entwine(bm + j, bm + k, T, TS, &bw) != 0) continue;
                            *ok &= fusion(jp, aw, kp, T, top, cap, TS);
                            am[k] = *jp;
                            *ok &= fusion(bm + j, bw, bm + k, T, top, cap, TS);
                            bm[k] = bm[j];
                            br[1]++;
                        }
                    } else {
                        *ok &= fusion(jp, aw, kp, T, top, cap, TS);
                        am[k] = *jp;
                        br[2]++;
                    }
                } else {
                    am[k] = *jp;
                    if (bm) bm[k] = bm[j];
                    br[4]++;
                }
                break;
            } else {
                if (!(jp->abpos <= kp->aepos && jp->bbpos <= kp->bepos)) continue;
                if (entwine(kp, jp, T, TS, &aw) != 0) continue;
                if (kp->abpos == jp->abpos) {
                    if (kp->aepos < jp->aepos) {
                        am[k] = *jp;
                        if (bm) bm[k] = bm[j];
                        br[5]++;
                    }
                } else if (jp->aepos > kp->aepos) {
                    if (bm) {
                        if (comp) {
                            if (entwine(bm + j, bm + k, T, TS, &bw) != 0) continue;
                            *ok &= fusion(kp, aw, jp, T, top, cap, TS);
                            *ok &= fusion(bm + j, bw, bm + k, T, top, cap, TS);
                            bm[k] = bm[j];
                            br[6]++;
                        } else {
                            if (entwine(bm + k, bm + j, T, TS, &bw) != 0) continue;
                            *ok &= fusion(kp, aw, jp, T, top, cap, TS);
                            *ok &= fusion(bm + k, bw, bm + j, T, top, cap, TS);
                            br[7]++;
                        }
                    } else {
                        *ok &= fusion(kp, aw, jp, T, top, cap, TS);
                        br[8]++;
                    }
                }
                break;
            }
        }
        if (k < 0) {
            no += 1;
            am[no] = *jp;
            if (bm) bm[no] = bm[j];
        }
    }
    return no + 1;
}

// ---- the pair kernel --------------------------------------------------------------
//
// AUX: the instantiation that also fills job_work / redund (capture mode and
// the branch statistics).

// The pair a half works on, in LDS.
struct PairState {
    int active, in_panel, job, status;
    long long ps, pe;        // its seeds
    int ar, br, alen, blen, do_a, do_b;
    int novla, novlb, tmin, tmax, touched, band0;
    long long ttop, aligned, edges, cells, snake, steps;
    long long lidx, nidx, h2, f0;   // panel [lidx, nidx), start of the next one, next seed to test
    int amark2, prio;
};

// (NCH: each kernel has its own copy, so its registers fit that kernel's)
template <int NCH, bool AUX>
struct PairJob {
    const ReportArgs* args;
    PairState* ps;   // LDS, one per half

    typedef KernArgs<ReportArgs> KA;

    struct Bands {
        int *F, *score, *lastp, *lasta, *edge;
    };
    __device__ static Bands bands(KA* a, int slot)
    {
        // score[band], band in [mindiag-1, maxdiag+1]; edge: lastp[maxdiag] == lasta[mindiag-1]
        Bands b;
        b.F = a->bands + (size_t)slot * (3 * a->w + 2);
        b.score = b.F + 1 - a->mindiag;
        b.lastp = b.score + a->w;
        b.lasta = b.lastp + a->w;
        b.edge = b.F + 2 * a->w;
        return b;
    }

    // the next alignment of half h: of its pair, or of the next pair in the queue
    __device__ bool next(PackLds& L, int h)
    {
        KA* a = kern_args(args);
        const int lane = __lane_id();
        PairState& P = ps[h];
        const int slot = 2 * blockIdx.x + h;
        const Bands b = bands(a, slot);
        for (;;) {
            if (!uni(P.active)) {
                // all lanes take part in the atomic (lane 0 adds 1), so the exit is uniform
                const int t = uni(atomicAdd(a->counter, lane == 0 ? 1 : 0));
                const int ab = uni(__atomic_load_n(a->abort_flag, __ATOMIC_RELAXED));
                if (t >= a->norder || ab) return false;
                if (lane == 0) {
                    const int job = a->order[t], p = a->jobs[job];
                    P.job = job;
                    P.prio = queue_priority(t, a->norder);
                    P.ps = a->pstart[p];
                    P.pe = a->pstart[p + 1];
                    const Seed s0 = a->hits[P.ps];
                    P.ar = s0.aread;
                    P.br = s0.bread;
                    P.alen = a->lenA[s0.aread];
                    P.blen = a->lenB[s0.bread];
                    P.do_a = P.alen >= a->hgap_min;
                    P.do_b = a->symmetric && P.blen >= a->hgap_min && (P.ar != P.br || !a->self || !a->comp);
                    P.novla = P.novlb = 0;
                    P.ttop = 0;
                    P.status = RP_OK;
                    P.tmin = INT32_MAX;   // lasta cells raised by this pair
                    P.tmax = -INT32_MAX;
                    P.touched = 0;
                    P.aligned = P.edges = P.cells = P.snake = P.steps = 0;
                    P.nidx = P.ps;
                    P.amark2 = 0;
                    P.in_panel = 0;
                    P.active = 1;
                    *b.edge = a->edge_in ? a->edge_in[job] : 0;
                }
                wave_sync();
            }
            const long long pe = uni(P.pe);
            if (uni(P.in_panel)) {
                // gating in seed order (dalign/filter.c:1768-1893): a seed is
                // aligned when it lies beyond its band's lasta and the band
                // pair score reaches hitmin; 64 seeds are tested at once and
                // testing resumes after each aligned seed
                const long long lidx = uni(P.lidx), nidx = uni(P.nidx);
                long long f0 = uni(P.f0);
                while (f0 < nidx && uni(P.status) == RP_OK) {
                    const long long f = f0 + lane;
                    bool go = false;
                    if (f < nidx) {
                        const int ap = a->hits[f].apos, band = a->hits[f].diag >> a->binshift;
                        go = ap > b.lasta[band] && (b.score[band] + b.score[band + 1] >= a->hitmin ||
                                                    b.score[band] + b.score[band - 1] >= a->hitmin);
                    }
                    const unsigned long long gm = __ballot(go);
                    if (!gm) {
                        f0 += 64;
                        continue;
                    }
                    const long long fh = f0 + lowest_lane(gm);
                    if (lane == 0) {
                        const Seed sd = a->hits[fh];
                        P.f0 = fh + 1;
                        P.band0 = sd.diag >> a->binshift;
                        align(L.slot[h], P, a, slot, sd);
                    }
                    wave_sync();
                    return true;
                }
                // panel reset of the scored bands (dalign/filter.c:1895-1899)
                wave_sync();
                for (long long c = lidx; c < nidx; c += 64) {
                    const long long f = c + lane;
                    if (f < nidx) {
                        const int band = a->hits[f].diag >> a->binshift;
                        b.score[band] = 0;
                        b.lastp[band] = 0;
                    }
                }
                if (lane == 0) {
                    P.in_panel = 0;
                    P.nidx = P.h2;
                }
                wave_sync();
                continue;
            }
            const long long lidx = uni(P.nidx);
            if (lidx < pe && uni(P.status) == RP_OK) {
                panel(a, b, P, lidx, pe);
                continue;
            }
            finish(a, b, P, slot);
        }
    }

    // slot S's alignment of seed sd (lane 0)
    __device__ static void align(PackSlot& S, const PairState& P, KA* a, int slot, const Seed& sd)
    {
        const int dg = sd.diag;
        // a read against itself (-I, self forward pass: the same bases): the
        // wave may not reach the main diagonal (Local_Alignment's selfie
        // bounds, dalign/align.c:1966-1985)
        const bool selfie = a->self && !a->comp && P.ar == P.br;
        const int maxtp = 2 * ((P.alen > P.blen ? P.alen : P.blen) / a->tspace + 2);
        uint16_t* latr = a->latr + (size_t)slot * 4 * a->maxtp_all;
        S.prio = P.prio;
        S.A = a->pkA + a->w0A[P.ar];
        S.B = a->pkB + a->w0B[P.br];
        S.alen = P.alen;
        S.blen = P.blen;
        S.comp = a->comp;
        S.low = S.hgh = dg;
        S.anti = 2 * sd.apos - dg;
        S.minp = (selfie && dg >= 0) ? 1 : -INT32_MAX;
        S.maxp = (selfie && dg <= 0) ? -1 : INT32_MAX;
        S.pool = a->pools + (size_t)slot * a->pool_cap;
        S.pool_cap = a->pool_cap;
        S.pts = a->pts + (size_t)slot * 2 * a->pts_cap;
        S.pts_cap = a->pts_cap;
        S.atr = latr + maxtp;
        S.btr = latr + 3 * maxtp;
        S.maxtp = maxtp;
    }

    // The panel from seed lidx on: its end, the next one's start, its band scores.
    __device__ static void panel(KA* a, const Bands& b, PairState& P, long long lidx, long long pe)
    {
        const int lane = __lane_id();
        const int amark = uni(P.amark2) + 50000, amark2 = amark - 10000;
        // panel (dalign/filter.c:1740-1755): up to and including the first
        // seed beyond amark; the next panel starts after the last seed at
        // or before amark2
        long long pend = pe, h2 = lidx;
        for (long long c = lidx; c < pe; c += 64) {
            const long long f = c + lane;
            const int ap = (f < pe) ? a->hits[f].apos : INT32_MAX;
            const unsigned long long beyond = __ballot(f < pe && ap > amark);
            const unsigned long long within2 = __ballot(f < pe && ap <= amark2);
            if (within2) h2 = c + highest_lane(within2) + 1;
            if (beyond) {
                pend = c + lowest_lane(beyond) + 1;
                break;
            }
        }
        const bool scored = pend - lidx >= a->minhit;
        bool touched = false;
        long long edges = 0;
        if (scored) {
            // band scores (dalign/filter.c:1757-1766): each seed adds
            // min(K, apos - apos of the band's previous seed)
            for (long long c = lidx; c < pend; c += 64) {
                const long long f = c + lane;
                const bool v = f < pend;
                int ap = 0, band = a->mindiag;
                if (v) {
                    ap = a->hits[f].apos;
                    band = a->hits[f].diag >> a->binshift;
                }
                const unsigned bi = (unsigned)(band - a->mindiag);
                unsigned long long peers = __ballot(v);
#pragma unroll
                for (int q = 0; q < 16; q++) {
                    const unsigned long long m = __ballot((bi >> q) & 1);
                    peers &= ((bi >> q) & 1) ? m : ~m;
                }
                const unsigned long long below = peers & ((1ull << lane) - 1);
                const int prevl = below ? highest_lane(below) : lane;
                const int pap = __shfl(ap, prevl, 64);
                int prev = 0;
                if (v) prev = below ? pap : b.lastp[band];
                if (__any(v && band == a->maxdiag)) touched = true;
                edges += __popcll(__ballot(v && (band == a->mindiag || band == a->maxdiag)));
                wave_sync();
                if (v) {
                    const int d = ap - prev;
                    atomicAdd(&b.score[band], d >= a->K ? a->K : d);
                    if (lane == highest_lane(peers)) b.lastp[band] = ap;
                }
                wave_sync();
            }
        }
        if (lane == 0) {
            P.amark2 = amark2;
            P.lidx = lidx;
            P.h2 = h2;
            P.f0 = lidx;
            P.in_panel = scored;
            P.nidx = scored ? pend : h2;
            if (touched) P.touched = 1;
            P.edges += edges;
        }
        wave_sync();
    }

    // the alignment of half h ended (S.res)
    __device__ void done(PackLds& L, int h)
    {
        KA* a = kern_args(args);
        const int lane = __lane_id();
        PairState& P = ps[h];
        const PackSlot& S = L.slot[h];
        const int slot = 2 * blockIdx.x + h;
        const Bands b = bands(a, slot);
        const int TS = a->tspace;
        const int rs = uni(S.res.status);
        if (lane == 0) {
            P.cells += S.cells;
            P.snake += S.snake;
            P.steps += S.steps;
        }
        if (rs != LA_OK) {
            if (lane == 0)
                P.status = (rs == LA_WIDE || rs == LA_POOL || rs == LA_ABORT) ? RP_RETRY : RP_UNDEF;
            wave_sync();
            return;
        }
        const int abpos = uni(S.res.abpos), bbpos = uni(S.res.bbpos), aepos = uni(S.res.aepos),
                  bepos = uni(S.res.bepos);
        const int atlen = uni(S.res.atlen), btlen = uni(S.res.btlen);
        const uint16_t* ta = uni(S.atr) + uni(S.res.afirst);
        const uint16_t* tb = uni(S.btr) + uni(S.res.bfirst);
        const int band0 = uni(P.band0);
        // Diagonal_Span (dalign/filter.c:1568-1599) widened by one band on
        // each side and to the seed's band.  The walk over the trace points is
        // a prefix sum: 64 of them at a time.
        int lo = abpos - bbpos, hi = lo;
        {
            const int d1 = aepos - bepos;
            lo = min(lo, d1);
            hi = max(hi, d1);
            int dd = (abpos / TS) * TS - bbpos;
            const int n = atlen / 2 - 1;   // every pair but the last
            for (int c = 0; c < n; c += 64) {
                const int i = c + lane;
                int x = i < n ? TS - ta[2 * i + 1] : 0;
#pragma unroll
                for (int o = 1; o < 64; o <<= 1) {
                    const int u = __shfl_up(x, o, 64);
                    if (lane >= o) x += u;
                }
                x += dd;
                dd = rdl(x, 63);
                int mn = i < n ? x : lo, mx = i < n ? x : hi;
#pragma unroll
                for (int o = 32; o >= 1; o >>= 1) {
                    mn = min(mn, __shfl_xor(mn, o, 64));
                    mx = max(mx, __shfl_xor(mx, o, 64));
                }
                lo = min(lo, uni(mn));
                hi = max(hi, uni(mx));
            }
            lo = (lo >> a->binshift) - 1;
            hi = (hi >> a->binshift) + 1;
            if (band0 < lo) lo = band0;
            else if (band0 > hi) hi = band0;
        }
        const bool out = lo < a->mindiag, over = out || hi > a->maxdiag;
        // a consistent trace keeps the span within one band of the
        // array on each side; the clamp only guards the memory
        lo = max(lo, a->mindiag - 1);
        hi = min(hi, a->maxdiag + 1);
        for (int i = lane; i <= hi - lo; i += 64)
            if (aepos > b.lasta[lo + i]) b.lasta[lo + i] = aepos;
        const int do_a = uni(P.do_a), do_b = uni(P.do_b), na = uni(P.novla), nb = uni(P.novlb);
        long long ttop = uni(P.ttop);
        const bool keep = (aepos - abpos) + (bepos - bbpos) >= a->minover;
        const long long need = (do_a ? atlen : 0) + (do_b ? btlen : 0);
        const bool full = keep && (na >= a->mcap || nb >= a->mcap || ttop + need > a->mtcap);
        MPath* am = a->mpaths + (size_t)slot * 2 * a->mcap;
        MPath* bm = am + a->mcap;
        uint16_t* T = a->mtrace + (size_t)slot * a->mtcap;
        if (keep && !full) {
            if (do_a) {
                for (int i = lane; i < atlen; i += 64) T[ttop + i] = ta[i];
                if (lane == 0) am[na] = MPath{atlen, S.res.diffs, abpos, bbpos, aepos, bepos, ttop};
                ttop += atlen;
            }
            if (do_b) {
                for (int i = lane; i < btlen; i += 64) T[ttop + i] = tb[i];
                if (lane == 0)
                    bm[nb] = MPath{btlen, S.res.diffs, S.res.b_abpos, S.res.b_bbpos, S.res.b_aepos, S.res.b_bepos, ttop};
                ttop += btlen;
            }
        }
        if (lane == 0) {
            P.aligned += 1;
            if (over) P.edges += 1;
            if (out) P.touched = 1;
            P.tmin = min(P.tmin, lo);
            P.tmax = max(P.tmax, hi);
            if (full) P.status = RP_ARENA;
            else if (keep) {
                P.novla = na + (do_a ? 1 : 0);
                P.novlb = nb + (do_b ? 1 : 0);
                P.ttop = ttop;
            }
        }
        wave_sync();
    }

    // the pair is done: its records and statistics, its band arrays zero for the next one
    __device__ static void finish(KA* a, const Bands& b, PairState& P, int slot)
    {
        const int lane = __lane_id();
        const int job = uni(P.job), TS = a->tspace;
        int pstatus = uni(P.status);
        MPath* am = a->mpaths + (size_t)slot * 2 * a->mcap;
        MPath* bm = am + a->mcap;
        uint16_t* T = a->mtrace + (size_t)slot * a->mtcap;
        // per-pair lasta reset (dalign/filter.c:1905-1920): every raised cell
        // inside [mindiag, maxdiag] belongs to a run of non-zero cells through
        // a seed band of this pair, so the reference's walk clears exactly the
        // raised in-range cells; cells outside the range keep their value
        const int tmin = uni(P.tmin), tmax = uni(P.tmax);
        if (tmin <= tmax) {   // some alignment raised cells (tmin / tmax start empty)
            const int lo = max(tmin, a->mindiag), hi = min(tmax, a->maxdiag);
            for (int i = lane; i <= hi - lo; i += 64) b.lasta[lo + i] = 0;
            wave_sync();
        }
        if (pstatus == RP_OK) {
            // fuse redundant alignments (lane 0) and append the records
            bool ok = true;
            int na = uni(P.novla), nb = uni(P.novlb);
            if (lane == 0 && (AUX || na > 1 || nb > 1)) {
                unsigned br[kRedundBranches] = {};
                long long ttop = P.ttop;
                const int comp = a->comp;
                if (na > 1) {
                    if (nb > 1) na = nb = handle_redundancies(am, na, bm, T, &ttop, a->mtcap, TS, comp, &ok, br);
                    else na = handle_redundancies(am, na, nullptr, T, &ttop, a->mtcap, TS, comp, &ok, br);
                } else if (nb > 1)
                    nb = handle_redundancies(bm, nb, nullptr, T, &ttop, a->mtcap, TS, comp, &ok, br);
                if constexpr (AUX) {
                    if (a->redund)   // the job's last successful run overwrites earlier ones
                        for (int q = 0; q < kRedundBranches; q++) a->redund[(size_t)job * kRedundBranches + q] = br[q];
                }
            }
            ok = uni(ok ? 1 : 0) != 0;
            na = uni(na);
            nb = uni(nb);
            if (!ok) pstatus = RP_ARENA;
            else if (na + nb > 0) {
                wave_sync();
                long long tl = 0;
                for (int i = 0; i < na; i++) tl += am[i].tlen;
                for (int i = 0; i < nb; i++) tl += bm[i].tlen;
                const int tbytes = a->small_trace ? 1 : 2;
                const unsigned long long r0 = atomicAdd(&a->ocount[0], lane == 0 ? (unsigned long long)(na + nb) : 0ull);
                const unsigned long long t0 = atomicAdd(&a->ocount[1], lane == 0 ? (unsigned long long)(tl * tbytes) : 0ull);
                const unsigned long long rbase = (unsigned long long)uni((long long)r0);
                const unsigned long long tbase = (unsigned long long)uni((long long)t0);
                if (rbase + na + nb > (unsigned long long)a->ocap || tbase + tl * tbytes > (unsigned long long)a->otcap)
                    pstatus = RP_OUT;
                else {
                    const int ar = uni(P.ar) + a->afirst, br = uni(P.br) + a->bfirst;
                    unsigned long long to = tbase;
                    for (int i = 0; i < na + nb; i++) {
                        const bool isA = i < na;
                        const MPath m = isA ? am[i] : bm[i - na];
                        if (lane == 0) {
                            OutRec o;
                            o.tlen = m.tlen;
                            o.diffs = m.diffs;
                            o.abpos = m.abpos;
                            o.bbpos = m.bbpos;
                            o.aepos = m.aepos;
                            o.bepos = m.bepos;
                            o.flags = (uint32_t)a->comp;
                            o.aread = isA ? ar : br;
                            o.bread = isA ? br : ar;
                            o.local = isA ? i : i - na;
                            o.job = job;
                            o.toff = (long long)to;
                            o.gen = a->gen;
                            o.pad = 0;
                            a->orecs[rbase + i] = o;
                        }
                        // Compress_TraceTo8 (dalign/align.c:3352-3360) when the spacing is <= 125
                        for (int q = lane; q < m.tlen; q += 64) {
                            const uint16_t x = T[m.toff + q];
                            if (tbytes == 1) a->otr[to + q] = (uint8_t)x;
                            else {
                                a->otr[to + 2 * q] = (uint8_t)(x & 0xff);
                                a->otr[to + 2 * q + 1] = (uint8_t)(x >> 8);
                            }
                        }
                        to += (unsigned long long)m.tlen * tbytes;
                    }
                }
            }
        }
        wave_sync();
        const int eout = *b.edge;
        if (lane == 0) {
            a->status[job] = pstatus;
            if (pstatus == RP_OK) a->final_gen[job] = a->gen;
            a->edge_out[job] = eout;
            a->touch[job] = P.touched;
            if (pstatus == RP_OK) {
                atomicAdd(&a->stats[0], (unsigned long long)P.aligned);
                atomicAdd(&a->stats[1], (unsigned long long)P.cells);
                atomicAdd(&a->stats[2], (unsigned long long)P.snake);
                atomicAdd(&a->stats[3], (unsigned long long)P.edges);
                atomicAdd(&a->stats[4], (unsigned long long)P.steps);
                if constexpr (AUX) {
                    if (a->job_work) a->job_work[job] = (unsigned long long)(P.cells + P.snake);
                }
            }
        }
        // leave the band arrays zero for the next job: the edge cell and the
        // pad always, everything when the pair stopped early
        const int W3 = 3 * a->w + 2;
        if (pstatus != RP_OK) {
            wave_sync();
            for (int i = lane; i < W3; i += 64) b.F[i] = 0;
        } else if (lane == 0) {
            *b.edge = 0;
            b.F[W3 - 1] = 0;
        }
        if (lane == 0) P.active = 0;
        wave_sync();
    }
};

// A persistent grid of single-wave workgroups, two pairs in flight on each
// (one where the grid has a wave for every pair).
template <int NCH, bool AUX>
__global__ __launch_bounds__(64, NCH == 2 ? kPackWaves : 1) void k_report(ReportArgs)
{
    __shared__ PackLds L;
    __shared__ PairState ps[2];
    const ReportArgs* args = kernarg_ptr<ReportArgs>();
    KernArgs<ReportArgs>* a = kern_args(args);
    if (__lane_id() < 2) ps[__lane_id()].active = 0;
    DevSpec sp;
    sp.table = a->sp.table;
    sp.score = a->sp.score;
    sp.tspace = a->sp.tspace;
    sp.ave_path = a->sp.ave_path;
    pack_tables(L, sp);
    pack_run<NCH>(L, PairJob<NCH, AUX>{args, ps}, a->norder > (int)gridDim.x, a->abort_flag);
}

}  // namespace mi
