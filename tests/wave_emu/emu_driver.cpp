// Runs the batched aligner (marvel_amd/csrc/la_batch.hip over la_pack.hpp) on
// the CPU wave emulator over a la_vectors task file and writes a la_vectors
// result file (plus a status word per task).  TEST INFRASTRUCTURE ONLY.
#include <algorithm>
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <vector>

#include "../../include/marvl_align.h"

int main(int argc, char** argv)
{
    if (argc < 3) return 1;
    FILE* in = fopen(argv[1], "rb");
    FILE* out = fopen(argv[2], "wb");
    const int only = argc > 3 ? atoi(argv[3]) : -1;
    if (!in || !out) return 1;
    int32_t n, ts;
    int64_t nb;
    MiAlignParams prm;
    if (fread(&n, 4, 1, in) != 1 || fread(&prm.ave_corr, 8, 1, in) != 1 || fread(&ts, 4, 1, in) != 1 ||
        fread(prm.freq, 16, 1, in) != 1 || fread(&nb, 8, 1, in) != 1)
        return 1;
    prm.trace_space = ts;
    std::vector<char> seq(nb);
    if (fread(seq.data(), 1, nb, in) != (size_t)nb) return 1;
    std::vector<uint64_t> packed(1, 0);
    auto pack = [&](int64_t off, int len) {
        const long long at = (long long)packed.size();
        packed.resize(packed.size() + (len + 31) / 32 + 2, 0);
        for (int j = 0; j < len; j++) packed[at + (j >> 5)] |= (uint64_t)(seq[off + j] & 3) << (2 * (j & 31));
        return at;
    };
    std::vector<MiLaTask> tasks;
    long long ntr = 16;
    for (int i = 0; i < n; i++) {
        int64_t ao, bo;
        int32_t v[8];
        if (fread(&ao, 8, 1, in) != 1 || fread(&bo, 8, 1, in) != 1 || fread(v, 4, 8, in) != 8) return 1;
        if (only >= 0 && i != only) continue;
        MiLaTask t = {};
        t.alen = v[0];
        t.blen = v[1];
        t.comp = v[2];
        t.low = v[3];
        t.hgh = v[4];
        t.anti = v[5];
        t.lbord = v[6];
        t.hbord = v[7];
        t.aword = pack(ao, t.alen);
        t.bword = pack(bo, t.blen);
        ntr += 4LL * (std::max(t.alen, t.blen) / ts + 2);
        tasks.push_back(t);
    }
    packed.push_back(0);
    const int m = (int)tasks.size();
    std::vector<MiLaResult> res(m);
    std::vector<uint16_t> tr(ntr);
    const int rc = mi_la_batch_host(&prm, packed.data(), (long long)packed.size(), tasks.data(), m, res.data(), tr.data(),
                                    ntr);
    if (rc != 0) {
        fprintf(stderr, "mi_la_batch_host: %d (%s)\n", rc, mi_last_error());
        return 1;
    }
    for (const MiLaResult& r : res) {
        int32_t f[13] = {r.abpos,   r.bbpos,   r.aepos,   r.bepos, r.diffs,  r.atlen, r.b_abpos,
                         r.b_bbpos, r.b_aepos, r.b_bepos, r.diffs, r.btlen, r.status};
        if (r.status)
            for (int q = 0; q < 12; q++) f[q] = 0;
        fwrite(f, 4, 13, out);
        if (!r.status) {
            fwrite(tr.data() + r.atrace, 2, r.atlen, out);
            fwrite(tr.data() + r.btrace, 2, r.btlen, out);
        }
    }
    fclose(out);
    return 0;
}
