// CPU check of the factorization's streams (windows and phases, built by
// glu_plan.hip) on a pattern: every slot, place and position a chunk names is
// in range, no two lanes of a step write one value, no lane reads a value
// another lane writes in the same step, every product is written once before
// it is subtracted; and the emulated steps equal the updates taken one at a
// time in schedule order (step by step, a step's columns as level_idx lists
// them) bit for bit, with and without replaced pivots.
//
//   factor_streams_check <pattern file> <window values> <bin values> <reverse: 0 | 1>
//
// The pattern file holds the arrays of Symbolic_Matrix (sym_c_ptr, sym_r_idx,
// l_col_ptr, csr_r_ptr, csr_c_idx, csr_diag_ptr, level_ptr, level_idx), each as
// a uint64 count followed by uint32 values.  reverse lists each level's columns
// the other way round (a pattern of the caller's may).  Compiled together with
// the library's host objects (this file includes glu_plan.hip itself).
#include "glu_plan.hip"
#include <cstdio>
#include <random>

using namespace glu;

static std::vector<uint32_t> rd(FILE *f)
{
    uint64_t k;
    if (fread(&k, 8, 1, f) != 1) exit(2);
    std::vector<uint32_t> v(k);
    if (k && fread(v.data(), 4, k, f) != k) exit(2);
    return v;
}

[[noreturn]] static void die(const char *what, size_t a = 0, size_t b = 0)
{
    printf("%s (%zu, %zu)\n", what, a, b);
    exit(1);
}

static float gesp(float d, float pert) { return std::fabs(d) < pert ? pert : d; }

// The values of one window or bin while its streams run.
struct Lds {
    std::vector<float> v;
    std::vector<uint64_t> read, written;   // 1 + step * kWho + who, by slot
    static constexpr uint64_t kWho = 1u << 24;
    uint32_t nslot = 0;
    void load(uint32_t slot, uint64_t step, uint64_t who, float &out)
    {
        if (slot >= nslot + kWinExtra) die("slot out of range", slot, nslot);
        if (slot < nslot) {
            if (written[slot] / kWho == step + 1 && written[slot] % kWho != who) die("a value is read in the step that writes it", slot, step);
            // (one reader is enough to refuse a later writer, unless it is the writer itself)
            if (read[slot] / kWho != step + 1 || read[slot] % kWho == who) read[slot] = (step + 1) * kWho + who;
            else read[slot] = (step + 1) * kWho + kWho - 1;   // two readers
        }
        out = v[slot];
    }
    void store(uint32_t slot, uint64_t step, uint64_t who, float x)
    {
        if (slot >= nslot + kWinExtra) die("slot out of range", slot, nslot);
        if (slot >= nslot) {
            if (slot < nslot + 2) die("a constant is written", slot, step);
            return;   // a target that nothing reads
        }
        if (written[slot] / kWho == step + 1) die("a value is written twice in a step", slot, step);
        if (read[slot] / kWho == step + 1 && read[slot] % kWho != who) die("a value is written in a step that reads it", slot, step);
        written[slot] = (step + 1) * kWho + who;
        v[slot] = x;
    }
};

// One window's (out: a bin's) streams over the values.
static void run_window(const Window &w, uint32_t waves, std::vector<float> &val, float pert, std::vector<float> *out,
                       std::vector<uint8_t> *made)
{
    if (w.wptr.size() != waves + 1 || w.wptr[0] != 0 || w.wptr.back() != w.hdr.size() || w.prog.size() != 512 * w.hdr.size())
        die("stream sizes");
    Lds S;
    S.nslot = (uint32_t)w.pos.size();
    if (S.nslot + kWinExtra > 0x10000) die("slots exceed 16 bits", S.nslot);
    S.v.assign(S.nslot + kWinExtra, 0.f);
    S.read.assign(S.nslot, 0);
    S.written.assign(S.nslot, 0);
    for (uint32_t i = 0; i < S.nslot; ++i) {
        if (w.pos[i] >= val.size() || (i && w.pos[i] <= w.pos[i - 1])) die("positions", i);
        S.v[i] = val[w.pos[i]];
    }
    S.v[S.nslot + 1] = 1.f;
    const uint32_t steps = (uint32_t)(w.l1 - w.l0);
    std::vector<uint32_t> at(waves);
    std::vector<std::array<float, 64>> acc(waves);
    for (uint32_t v = 0; v < waves; ++v) at[v] = w.wptr[v];
    for (uint32_t step = 0; step <= steps; ++step) {
        uint64_t who = 0;   // lanes of the step (a chain of chunks keeps its lanes)
        for (uint32_t v = 0; v < waves; ++v) {
            uint64_t chain = 0;
            for (; at[v] < w.wptr[v + 1] && (w.hdr[at[v]] & ((1u << kWinKindShift) - 1u)) == step; ++at[v]) {
                const uint32_t kind = w.hdr[at[v]] >> kWinKindShift;
                const uint16_t *p = &w.prog[512 * (size_t)at[v]];
                if (kind == kWinOut ? !out || step != steps : step == steps) die("a chunk's step", step, kind);
                if (kind == kWinCol || kind == kWinOut) chain = who, who += 64;
                for (uint32_t ln = 0; ln < 64; ++ln) {
                    const uint16_t *e = p + 8 * ln;
                    auto value = [&](uint32_t i, uint64_t id) {
                        float x;
                        S.load(e[i], step, id, x);
                        return x;
                    };
                    if (kind == kWinCol) {
                        const float l = value(0, chain + ln) / gesp(value(1, chain + ln), pert);
                        for (uint32_t k = 2; k < 8; k += 2) {
                            const float t = value(k + 1, chain + ln);
                            const float u = value(k, chain + ln);
                            S.store(e[k + 1], step, chain + ln, t + (-(l * u)));
                        }
                    } else if (kind == kWinOut) {
                        const float l = value(0, chain + ln) / gesp(value(1, chain + ln), pert);
                        for (uint32_t k = 0; k < 2; ++k) {
                            uint32_t o;
                            std::memcpy(&o, e + 4 + 2 * k, 4);
                            if (o == ~0u) continue;
                            if (o >= out->size() || (*made)[o]++) die("a product's place", o, out->size());
                            (*out)[o] = l * value(2 + k, chain + ln);
                        }
                    } else if (kind == kWinMerge) {
                        if (ln == 0 && (e[1] & kWinFirst)) chain = who, who += 64;
                        if (e[1] & kWinFirst) acc[v][ln] = value(0, chain + ln);
                        for (uint32_t k = 2; k < 8; k += 3) {
                            const float l = value(k, chain + ln), u = value(k + 1, chain + ln), d = value(k + 2, chain + ln);
                            acc[v][ln] = acc[v][ln] + (-(l / gesp(d, pert) * u));
                        }
                        if (e[1] & kWinLast) S.store(e[0], step, chain + ln, acc[v][ln]);
                    } else if (ln % 16 == 0) {   // 16 lanes an entry: all their sources here
                        if (ln == 0 && (e[7] & kWinFirst)) chain = who, who += 64;
                        if (e[7] & kWinFirst) acc[v][ln] = value(6, chain + ln);
                        for (uint32_t half = 0; half < (kind == kWinGroup ? 2u : 1u); ++half)
                            for (uint32_t j = 0; j < 16; ++j) {
                                const uint16_t *s = e + 8 * j + 3 * half;
                                if ((e[7] & (kWinFirst | kWinLast)) && (e[8 * j + 6] != e[6] || e[8 * j + 7] != e[7])) die("lanes of an entry", ln);
                                float l, u, d;
                                S.load(s[0], step, chain + ln, l);
                                S.load(s[1], step, chain + ln, u);
                                S.load(s[2], step, chain + ln, d);
                                acc[v][ln] = acc[v][ln] - (l / gesp(d, pert) * u);
                            }
                        if (e[7] & kWinLast) S.store(e[6], step, chain + ln, acc[v][ln]);
                    }
                }
            }
        }
    }
    for (uint32_t v = 0; v < waves; ++v)
        if (at[v] != w.wptr[v + 1]) die("a stream's steps are not in order", v);
    for (uint32_t i = 0; i < S.nslot; ++i) val[w.pos[i]] = S.v[i];
}

static void run_phase(const Phase &ph, std::vector<float> &val, float pert)
{
    std::vector<float> out(ph.nout);
    std::vector<uint8_t> made(ph.nout, 0), bin_of(val.size(), 0), sub(val.size(), 0);
    for (const Window &w : ph.bin) {
        if (w.l1 - w.l0 != ph.l1 - ph.l0 || w.pos.size() > ph.nslot) die("a bin's steps or values");
        for (uint32_t q : w.pos)
            if (bin_of[q]++) die("a value in two bins", q);
        run_window(w, kPhaseWaves, val, pert, &out, &made);
    }
    auto product = [&](size_t o) {
        if (o >= out.size() || made[o]++ != 1) die("a product is missing or taken twice", o);
        return out[o];
    };
    auto target = [&](uint32_t t) {
        if (t >= val.size() || bin_of[t] || sub[t]++) die("an assembled entry", t);
    };
    for (const AsmWave &e : ph.wav) {
        target(e.tgt);
        for (uint32_t k = 0; k < e.cnt; ++k) val[e.tgt] = val[e.tgt] - product(e.base + (size_t)k);
    }
    for (size_t g = 0; g < ph.grp.size(); ++g)
        for (uint32_t ln = 0; ln < 64; ++ln) {
            const uint32_t t = ph.tgt[64 * g + ln], cnt = ph.cnt[64 * g + ln];
            if (t == ~0u) continue;
            target(t);
            if (cnt > ph.grp[g].y) die("products of a group", g);
            for (uint32_t k = 0; k < cnt; ++k) val[t] = val[t] - product(ph.grp[g].x + 64 * (size_t)k + ln);
        }
    for (uint8_t m : made)
        if (m == 1) die("a product is not used");
}

int main(int argc, char **argv)
{
    if (argc < 5) return 2;
    const uint32_t budget = (uint32_t)atoi(argv[2]), bin_values = (uint32_t)atoi(argv[3]), waves = 16;
    FILE *f = fopen(argv[1], "rb");
    if (!f) return 2;
    auto cp = rd(f), ri = rd(f), ld = rd(f), rp = rd(f), ci = rd(f), rdg = rd(f), lp = rd(f), li = rd(f);
    fclose(f);
    std::vector<int32_t> level_ptr(lp.begin(), lp.end()), level_idx(li.begin(), li.end());
    if (atoi(argv[4]))
        for (size_t l = 0; l + 1 < level_ptr.size(); ++l)
            std::reverse(level_idx.begin() + level_ptr[l], level_idx.begin() + level_ptr[l + 1]);
    glu_pattern P{};
    P.n = (uint32_t)ld.size();
    P.nnz = (uint32_t)ri.size();
    P.num_lev = (int)level_ptr.size() - 1;
    P.sym_c_ptr = cp.data(), P.sym_r_idx = ri.data(), P.l_col_ptr = ld.data();
    P.csr_r_ptr = rp.data(), P.csr_c_idx = ci.data(), P.csr_diag_ptr = rdg.data();
    P.level_ptr = level_ptr.data(), P.level_idx = level_idx.data();
    std::string err;
    Tables T;
    int64_t updates = 0;
    if (!validate_pattern(P, err) || !build_factor_tables(P, T, updates, err)) die(err.c_str());
    std::vector<Window> wins;
    choose_windows(T, P.num_lev, P.nnz, budget, kDefaultFuseUnits, 1, waves, wins);
    std::vector<Phase> phases;
    const std::vector<uint32_t> umap = T.umap;   // (the phases write places over theirs)
    choose_phases(P, T, wins.empty() ? 0 : std::min(wins[0].l0, P.num_lev), bin_values, phases);
    size_t lane = 0, wave = 0, bins = 0, most = 0, busiest = 0;   // busiest: chunks of a phase's longest bin a step
    int steps = 0;
    for (const Phase &ph : phases) {
        lane += 64 * ph.grp.size();
        for (const Window &w : ph.bin) busiest = std::max(busiest, w.hdr.size() / (size_t)(ph.l1 - ph.l0));
        wave += ph.wav.size();
        bins += ph.bin.size();
        most = std::max<size_t>(most, ph.nslot);
        steps = ph.l1;
    }
    printf("n=%u levels=%d windows=%zu phases=%zu steps=%d bins=%zu largest=%zu lane_entries=%zu wave_entries=%zu busiest=%zu\n", P.n,
           P.num_lev, wins.size(), phases.size(), steps, bins, most, lane, wave, busiest);
    if (most > bin_values) die("a bin's values exceed the limit", most, bin_values);
    std::mt19937 g(11);
    std::uniform_real_distribution<float> U(-1.f, 1.f);
    std::vector<float> v0(P.nnz);
    for (auto &x : v0) x = U(g);
    for (uint32_t c = 0; c < P.n; ++c) v0[ld[c]] = (c % 7 == 3 ? 1e-3f : 3.f) + std::fabs(U(g)) * (c % 7 == 3 ? 1e-3f : 1.f);
    for (const float pert : {0.f, 0.01f}) {
        std::vector<float> got = v0, want = v0;
        auto plain = [&](std::vector<float> &v, int l) {   // step l, one update at a time
            for (int t = P.level_ptr[l]; t < P.level_ptr[l + 1]; ++t) {
                const uint32_t k = (uint32_t)P.level_idx[t], d = ld[k], L = cp[k + 1] - d - 1, u0 = rdg[k] + 1;
                for (uint32_t jj = 0; jj < rp[k + 1] - u0; ++jj)
                    for (uint32_t ii = 0; ii < L; ++ii) {
                        const float m = v[d + 1 + ii] / gesp(v[d], pert);
                        float &x = v[umap[T.moff[k] + (uint64_t)jj * L + ii]];
                        x = x + (-(m * v[T.upos[u0 + jj]]));
                    }
            }
        };
        for (int l = 0; l < P.num_lev; ++l) plain(want, l);
        int l = 0;
        auto up_to = [&](int e) {
            for (; l < e; ++l) plain(got, l);
        };
        for (const Phase &ph : phases) {
            up_to(ph.l0);
            run_phase(ph, got, pert);
            l = ph.l1;
        }
        for (const Window &w : wins) {
            up_to(w.l0);
            run_window(w, waves, got, pert, nullptr, nullptr);
            l = w.l1;
        }
        up_to(P.num_lev);
        for (uint32_t q = 0; q < P.nnz; ++q)
            if (std::memcmp(&got[q], &want[q], 4)) die("a value differs from the updates in schedule order", q);
    }
    printf("ok: streams equal the updates in schedule order bit for bit\n");
    return 0;
}
