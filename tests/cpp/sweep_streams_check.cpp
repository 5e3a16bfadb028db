// CPU check of the sweeps' streams (build_sw and choose_split in
// glu_plan.hip) on a pattern: the emulated sweeps of A x = b (L, U) and
// A' x = b (U', L'), run step by step over the streams' chunks, equal the
// row-by-row solve bit for bit where a row's products are subtracted in order
// (the exact solve), and agree with it in FP64 to the rounding of a sum where
// they are added (the refinement); the plan builder's own check accepts the
// streams and refuses planted mistakes.
//
//   sweep_streams_check <pattern file> <rows a workgroup holds, 0: all> <waves>
//
// With a limit, the sweeps are split: head parts, the tail, products formed
// between them.  The pattern file holds sym_c_ptr, sym_r_idx, l_col_ptr,
// csr_r_ptr, csr_c_idx, csr_diag_ptr, each as a uint64 count followed by
// uint32 values.  Compiled together with the library's host objects (this
// file includes glu_plan.hip itself).
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

// A sweep's value copy and right-hand sides (by lane of its streams).
struct Run {
    const SwHost *S;
    std::vector<float> val, rhs;
    bool div;
    Run(const SwHost &s, const std::vector<float> &lu, bool d) : S(&s), rhs(s.meta.size(), 0.f), div(d)
    {
        for (uint32_t q : s.vsrc) val.push_back(q == UINT32_MAX ? 0.f : lu[q]);
    }
    void products(const std::vector<float> &lu, const std::vector<float> &x)
    {
        for (const SwProd &q : S->prod) val[q.val] = lu[q.vpos] * x[q.col];
    }
};

// One part's sweep: right-hand sides set, results by slot into xs.
static void part_steps(const Run &R, const SwPart &P, bool tree, std::vector<float> &xs)
{
    const SwHost &S = *R.S;
    xs.assign(P.nslot + 2, std::nanf(""));
    xs[P.nslot] = 0.f;
    xs[P.nslot + 1] = 1.f;
    struct Open {
        float acc[64], first;
    };
    std::vector<std::array<Open, 2>> open(S.nwave);
    std::vector<uint32_t> f(S.nwave), u(S.nwave), f2(S.nwave), u2(S.nwave), left(S.nwave);
    for (uint32_t w = 0; w < S.nwave; ++w) {
        const uint4 d = S.wave[P.wp + w];
        left[w] = d.x, f[w] = d.y, f2[w] = d.z, u[w] = d.w & 255u, u2[w] = d.w >> 8;
    }
    for (uint32_t step = 0; step < P.steps; ++step) {
        std::vector<std::pair<uint32_t, float>> done;   // seen by the steps after this one
        for (uint32_t w = 0; w < S.nwave; ++w)
            for (; left[w] && (S.meta[f[w]].w & kSwStepMask) == step; --left[w]) {
                const uint4 *m = &S.meta[f[w]];
                const float *v = &R.val[(size_t)f[w] * S.per_lane];
                const uint32_t h = m[0].w, n = u[w];
                auto entry = [&](uint32_t lane, uint32_t e) {
                    const uint32_t q = e < 2 ? m[lane].x : m[lane].y;
                    return v[4 * lane + e] * xs[(e & 1) ? q >> 16 : q & 0xffffu];
                };
                auto finish = [&](uint32_t slot, uint32_t lane, float x) {
                    done.push_back({slot, R.div ? x / v[4 * n + lane] : x});
                };
                if (h & kSwLong) {
                    Open &o = open[w][(h & kSwTrack) ? 1 : 0];
                    const uint32_t count = m[0].z >> kSwCountShift;
                    if (h & kSwFirst) {
                        o.first = R.rhs[f[w]];
                        for (uint32_t l = 0; l < 64; ++l) o.acc[l] = l || tree ? 0.f : o.first;
                    }
                    for (uint32_t k = 0; k < count; ++k) {
                        if (!(m[k % 64].z & (kSwEntry << (k / 64)))) die("an entry's mark is missing", step, k);
                        if (tree) o.acc[k % 64] += entry(k % 64, k / 64);
                        else o.acc[0] = o.acc[0] - entry(k % 64, k / 64);
                    }
                    if (h & kSwLast) {
                        float s = 0.f;
                        for (float a : o.acc) s += a;
                        finish(m[0].z & 0xffffu, 0, tree ? o.first - s : o.acc[0]);
                    }
                } else
                    for (uint32_t lane = 0; lane < n;) {
                        const uint32_t z = m[lane].z, g = 1u << ((z >> 16) & 7u);
                        if (z & kSwOn) {
                            float a = R.rhs[f[w] + lane], s = 0.f;
                            for (uint32_t k = 0; k < 4 * g; ++k) {
                                a = a - entry(lane + k / 4, k % 4);
                                s += entry(lane + k / 4, k % 4);
                            }
                            const bool sum = tree && (z & kSwTree);   // its pivot at the first lane, else at the last
                            finish(z & 0xffffu, sum ? lane : lane + g - 1, sum ? R.rhs[f[w] + lane] - s : a);
                        }
                        lane += g;
                    }
                // (the stream's links: a chunk names the one two after it)
                f[w] = f2[w], u[w] = u2[w];
                f2[w] = m[1].w, u2[w] = m[2].w;
            }
        for (const auto &d : done) xs[d.first] = d.second;
    }
    for (uint32_t l : left)
        if (l) die("a chunk never runs", l);
}

int main(int argc, char **argv)
{
    if (argc < 4) return 2;
    const uint32_t cap = (uint32_t)atoi(argv[2]), waves = (uint32_t)atoi(argv[3]);
    FILE *fp = fopen(argv[1], "rb");
    if (!fp) return 2;
    auto cp = rd(fp), ri = rd(fp), ld = rd(fp), rp = rd(fp), ci = rd(fp), dg = rd(fp);
    fclose(fp);
    glu_pattern P{};
    const uint32_t n = P.n = (uint32_t)ld.size();
    const uint32_t nnz = P.nnz = (uint32_t)ri.size();
    P.sym_c_ptr = cp.data(), P.sym_r_idx = ri.data(), P.l_col_ptr = ld.data();
    P.csr_r_ptr = rp.data(), P.csr_c_idx = ci.data(), P.csr_diag_ptr = dg.data();
    std::vector<uint32_t> upos(nnz), cursor(rp.begin(), rp.end() - 1);
    for (uint32_t c = 0; c < n; ++c)
        for (uint32_t q = cp[c]; q < cp[c + 1]; ++q) upos[cursor[ri[q]]++] = q;
    // entries {column, position} of a row in the order it consumes them
    using Row = std::vector<uint2>;
    const auto row = [&](int q, uint32_t r) {
        Row o;
        if (q == 0) for (uint32_t k = rp[r]; k < dg[r]; ++k) o.push_back(make_uint2(ci[k], upos[k]));
        if (q == 1) for (uint32_t k = rp[r + 1]; k > dg[r] + 1; --k) o.push_back(make_uint2(ci[k - 1], upos[k - 1]));
        if (q == 2) for (uint32_t k = cp[r]; k < ld[r]; ++k) o.push_back(make_uint2(ri[k], k));
        if (q == 3) for (uint32_t k = cp[r + 1]; k > ld[r] + 1; --k) o.push_back(make_uint2(ri[k - 1], k - 1));
        return o;
    };
    const bool divs[4] = {false, true, true, false};
    const bool whole = cap == 0;
    SwSplit spl;
    if (whole) {
        spl.tail.part_of.assign(n, 0);
        spl.tail.count.assign(1, n);
        for (uint32_t r = 0; r < n; ++r) spl.tail.slot_of.push_back(r);
    } else if (!choose_split(P, cap, waves, spl)) {
        printf("no split\n");
        return 0;
    }
    for (const SwParts *p : {&spl.head, &spl.tail})
        for (uint32_t k : p->count)
            if (!whole && k > cap) die("a part's rows exceed the limit", k, cap);
    SwHost hd[4], tl[4];
    uint64_t lanes = 0, slots = 0, longest = 0, waited = 0, least = 0;
    int planted = 0, caught = 0;
    for (int q = 0; q < 4; ++q) {
        TriHost H;
        tri_levels(n, q % 2 ? -1 : +1, [&](uint32_t r, auto f) {
            for (const uint2 &e : row(q, r)) f(e.x);
        }, [&](uint32_t r) { return (uint32_t)row(q, r).size(); }, H);
        for (uint32_t l : H.len) longest = std::max<uint64_t>(longest, l);
        DfHost D;
        build_df(H, [&](uint32_t r, Row &o) { o = row(q, r); }, divs[q], [&](uint32_t r) { return ld[r]; }, !whole, D);
        std::string err;
        build_sw(H, D, n, divs[q], spl.tail, waves, tl[q]);
        if (!check_sw(tl[q], nnz, "tail", err)) die(err.c_str());
        if (!whole) {
            build_sw(H, D, n, divs[q], spl.head, kHeadWaves, hd[q]);
            if (!check_sw(hd[q], nnz, "head", err)) die(err.c_str());
        }
        lanes += tl[q].meta.size() + hd[q].meta.size();
        slots += D.idx.size();
        // (glu_refine_noalloc's scratch rests on this)
        if (whole && 3 * (uint64_t)tl[q].meta.size() > D.idx.size() + 64 * (uint64_t)n)
            die("lanes exceed a third of the slots and 64 a row", tl[q].meta.size(), D.idx.size());
        // chunks every step waits for: the most a wave has, and the fewest that could be
        if (whole) {
            const SwHost &S = tl[q];
            std::vector<uint32_t> total(S.part[0].steps), most(S.part[0].steps);
            size_t c = 0;
            for (uint32_t w = 0; w < waves; ++w) {
                std::vector<uint32_t> mine(S.part[0].steps);
                for (uint32_t k = 0; k < S.wave[w].x; ++k, ++c) ++mine[S.hdr[c] & kSwStepMask];
                for (uint32_t k = 0; k < mine.size(); ++k) total[k] += mine[k], most[k] = std::max(most[k], mine[k]);
            }
            for (uint32_t k = 0; k < total.size(); ++k) waited += most[k], least += std::max(1u, (total[k] + waves - 1) / waves);
        }
        // planted mistakes: a slot or a value position past the end, a step
        // too early, a chunk left out, a right-hand side elsewhere
        const SwHost &S = tl[q];
        auto plant = [&](auto change) {
            SwHost bad = S;
            change(bad);
            ++planted;
            std::string e2;
            caught += !check_sw(bad, nnz, "planted", e2);
        };
        plant([&](SwHost &b) { b.meta[0].x |= 0xffffu; });
        plant([&](SwHost &b) { b.vsrc[0] = nnz; });
        plant([&](SwHost &b) { b.rpos[0] ^= 1; });
        plant([&](SwHost &b) { --b.part[0].steps; });
        plant([&](SwHost &b) {
            uint32_t w = 0;
            while (!b.wave[w].x) ++w;
            --b.wave[w].x;
        });
        for (uint32_t c = 0; c < S.hdr.size(); ++c)   // a chunk with entries of its own part, at the first step
            if ((S.hdr[c] & kSwStepMask) && (S.meta[S.first[c]].x & 0xffffu) < S.part[0].nslot) {
                plant([&](SwHost &b) { b.meta[b.first[c]].w = b.hdr[c] &= ~kSwStepMask; });
                break;
            }
    }
    std::mt19937 g(5);
    std::uniform_real_distribution<float> U(-1.f, 1.f);
    std::vector<float> lu(nnz), b(n);
    for (uint32_t c = 0; c < n; ++c)   // rows and columns of both factors sum to less than a half
        for (uint32_t q = cp[c]; q < cp[c + 1]; ++q) lu[q] = 0.5f * U(g) / (float)longest;
    for (uint32_t c = 0; c < n; ++c) lu[ld[c]] = (c & 1 ? 1.f : -1.f) * (1.f + std::fabs(U(g)));
    for (float &v : b) v = U(g);
    for (int t = 0; t < 2; ++t)
        for (const bool tree : {false, true}) {
            std::vector<float> x(n, std::nanf("")), seq = b, xs;
            std::vector<double> ref(b.begin(), b.end());
            for (int q = 2 * t; q < 2 * t + 2; ++q)
                for (uint32_t i = 0; i < n; ++i) {
                    const uint32_t r = q % 2 ? n - 1 - i : i;
                    for (const uint2 &e : row(q, r)) {
                        seq[r] = seq[r] - lu[e.y] * seq[e.x];
                        ref[r] -= (double)lu[e.y] * ref[e.x];
                    }
                    if (divs[q]) seq[r] = seq[r] / lu[ld[r]], ref[r] /= lu[ld[r]];
                }
            auto sweep = [&](Run &R, const std::vector<float> &rhs) {
                for (const SwPart &p : R.S->part) {
                    for (uint32_t k = 0; k < p.nslot; ++k) R.rhs[R.S->rpos[p.s0 + k]] = rhs[R.S->row[p.s0 + k]];
                    part_steps(R, p, tree, xs);
                    for (uint32_t k = 0; k < p.nslot; ++k) x[R.S->row[p.s0 + k]] = xs[k];
                }
            };
            const int q0 = 2 * t, q1 = q0 + 1;
            Run h0(hd[q0], lu, divs[q0]), t0(tl[q0], lu, divs[q0]), t1(tl[q1], lu, divs[q1]), h1(hd[q1], lu, divs[q1]);
            if (!whole) sweep(h0, b);
            t0.products(lu, x);
            sweep(t0, b);
            sweep(t1, x);
            h1.products(lu, x);
            if (!whole) sweep(h1, x);
            // a row's rounding errors are at most (entries + 3) u times its
            // sum of magnitudes, at most 2; later rows take half of them on
            const double tol = 8.0 * (longest + 3) * std::ldexp(1.0, -24);
            for (uint32_t r = 0; r < n; ++r)
                if (tree ? !(std::fabs(x[r] - ref[r]) <= tol) : std::memcmp(&x[r], &seq[r], 4) != 0)
                    die("a row differs", r, (size_t)(2 * t + tree));
        }
    if (whole) printf("chunks waited for: %llu of at least %llu\n", (unsigned long long)waited, (unsigned long long)least);
    printf("ok n=%u parts=%zu tail=%u lanes=%llu slots=%llu planted=%d caught=%d: streams equal the row-by-row solve bit for bit\n",
           n, spl.head.count.size(), spl.tail.count[0], (unsigned long long)lanes, (unsigned long long)slots, planted, caught);
    return planted == caught ? 0 : 1;
}
