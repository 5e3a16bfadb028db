// CPU check of glu_refine_noalloc's scratch (noalloc_layout in glu_plan.hip):
// every order whose ready-bit tables are within GLU_NOALLOC_SCRATCH_BYTES is
// served.  First the bound the layout rests on, from the builders themselves:
// a sweep of m rows of `len` entries has at most (slots + 64 m) / 3 lanes, its
// rows side by side in one level or one a level.  Then the layout at the sizes
// at which it is largest.  Compiled together with the library's host objects
// (this file includes glu_plan.hip itself).
#include "glu_plan.hip"
#include <cstdio>

using namespace glu;

struct Size {
    double lanes, slots;   // a row
};

// m rows of len entries each on `first` rows without any; chain: each also on
// the row before it
static void sizes(uint32_t first, uint32_t m, uint32_t len, bool chain, bool long_lanes, uint64_t &lanes, uint64_t &slots)
{
    const uint32_t n = first + m;
    std::vector<std::vector<uint2>> rows(n);
    for (uint32_t i = 0; i < m; ++i)
        for (uint32_t k = 0; k < len; ++k) {
            const bool before = chain && i && k + 1 == len;
            rows[first + i].push_back(make_uint2(before ? first + i - 1 : k, 0u));
        }
    TriHost H;
    tri_levels(n, +1, [&](uint32_t r, auto f) {
        for (const uint2 &e : rows[r]) f(e.x);
    }, [&](uint32_t r) { return (uint32_t)rows[r].size(); }, H);
    DfHost D;
    build_df(H, [&](uint32_t r, std::vector<uint2> &o) { o = rows[r]; }, false, [](uint32_t) { return 0u; }, long_lanes, D);
    SwParts Q;
    Q.part_of.assign(n, 0);
    Q.count.assign(1, n);
    for (uint32_t r = 0; r < n; ++r) Q.slot_of.push_back(r);
    SwHost S;
    build_sw(H, D, n, false, Q, 16, S);
    lanes = S.meta.size();
    slots = D.idx.size();
}

int main()
{
    constexpr uint32_t kRows = 64;
    for (uint32_t len = 0; len <= 1100; len += len < 700 ? 1 : 37)
        for (const bool chain : {false, true}) {
            if (chain && len == 0) continue;
            const uint32_t first = std::max(len, 1u);
            uint64_t l0, s0, l1, s1;
            sizes(first, 0, 0, false, false, l0, s0);
            sizes(first, kRows, len, chain, false, l1, s1);
            // (a task's last rows and a level's last chunk: up to 64 lanes
            // more, or slots less, than the rows alone)
            if (3.0 * (double)(l1 - l0) > (double)(s1 - s0) + 64.0 * kRows + 6 * 64.0) {
                printf("len %u chain %d: %llu lanes, %llu slots\n", len, chain, (unsigned long long)(l1 - l0), (unsigned long long)(s1 - s0));
                return 1;
            }
        }
    // one workgroup: the largest n, every split of the limit between the two
    // sweeps, lanes at the bound
    size_t most = 0;
    for (const uint32_t n : {5000u, 20000u, 39718u})
        for (const int krylov : {0, 1, 4})
            for (uint32_t part = 0; part <= 10; ++part) {
                glu_plan p;
                p.n = n;
                p.krylov = krylov;
                const uint64_t fixed = (4 + 2 * (uint64_t)(krylov ? 3 * krylov + 1 : 0)) * n + 64 + 6 * 64;
                const uint64_t total = GLU_NOALLOC_SCRATCH_BYTES / 4;
                if (fixed >= total) continue;
                const uint64_t x = (total - fixed) * part / 10, y = total - fixed - x;
                const uint64_t lx = (x + 64 * (uint64_t)n) / 3, ly = (y + 64 * (uint64_t)n) / 3;
                for (int t = 0; t < 2; ++t) {
                    p.scratch_nval[t] = x + y + n + 64;
                    p.rhs_len[t] = (uint32_t)std::max(lx, ly);
                }
                p.df_nval = p.tdf_nval = (uint32_t)(4 * lx + 5 * ly);
                for (int t = 0; t < 2; ++t) {
                    const NoallocLayout L = noalloc_layout(p, 2, t);
                    if (L.limit > GLU_NOALLOC_SCRATCH_BYTES || L.bytes > kScratchBytes || L.split) {
                        printf("n=%u krylov=%d: limit %zu, layout %zu\n", n, krylov, L.limit, L.bytes);
                        return 1;
                    }
                    most = std::max(most, L.bytes);
                }
            }
    printf("one workgroup: at most %zu of %zu bytes\n", most, (size_t)kScratchBytes);
    // split sweeps: 95,000 rows in dense blocks of 129 (rows of 0 to 128
    // entries, one a level in every part), whose streams do not fit
    {
        glu_plan p;
        p.n = 95000;
        uint64_t lanes = 0, slots = 0;
        for (uint32_t len = 0; len < 129; ++len) {
            uint64_t l0, s0, l1, s1;
            const uint32_t first = std::max(len, 1u);
            sizes(first, 0, 0, false, true, l0, s0);
            sizes(first, 64, len, false, true, l1, s1);   // (a level of 64 such rows: lane rows)
            slots += (s1 - s0) / 64;
            sizes(first, 1, len, false, true, l1, s1);
            lanes += l1 - l0;
        }
        const double per_row = (double)p.n / 129;
        p.has_split = true;
        for (int t = 0; t < 2; ++t) {
            p.scratch_nval[t] = (uint64_t)(2 * slots * per_row) + p.n + 64;
            p.rhs_len[t] = (uint32_t)(lanes * per_row);
            p.split[t].nval = (uint32_t)(9 * lanes * per_row);
        }
        p.df_nval = p.tdf_nval = (uint32_t)p.scratch_nval[0];
        for (int t = 0; t < 2; ++t) {
            const NoallocLayout L = noalloc_layout(p, 1, t);
            printf("split: limit %zu, streams %zu values, layout %zu (%s)\n", L.limit, (size_t)p.split[t].nval, L.bytes,
                   L.split ? "split" : "one workgroup");
            if (L.limit > GLU_NOALLOC_SCRATCH_BYTES || L.bytes > kScratchBytes) return 1;
        }
        p.split[0].nval = (uint32_t)(kScratchBytes / 4);   // certainly beyond it
        const NoallocLayout L = noalloc_layout(p, 1, 0);
        if (L.split || L.nval != p.df_nval || L.bytes > L.limit) return 1;
    }
    printf("ok\n");
    return 0;
}
