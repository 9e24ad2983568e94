// Sums over several eq factors, sum_g eq(rho_g, x) P_g(x), on the CPU through tests/cpp/emu/hip/hip_runtime.h under the host sanitizers:
// wsum_kernel (a round that is a launch of its own) and slice_kernel with SliceArgsEqs (the rounds resident in LDS, one or two a trip).
// Every sum is compared with q_g(t) = sum_x' R_g(x') P_g(t, x') worked out by plain loops from the terms, R_g from its definition.
// The programs are built as the library builds them (program.hpp), from terms that are also evaluated one by one; programs of random lists of
// terms are walked by a plain stack machine besides.
#include <algorithm>
#include <chrono>
#include <memory>
#include <thread>
#include <vector>

#include "dpsumcheck.h"
#include "kernels.hpp"
#include "program.hpp"

using gl::E2;
using gl::u32;
using gl::u64;

static u64 sm_state = 99;
static u64 splitmix()
{
    sm_state += 0x9E3779B97F4A7C15ull;
    u64 z = sm_state;
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
    return z ^ (z >> 31);
}
static u64 felt()
{
    for (;;) {
        const u64 v = splitmix();
        if (v < gl::P) return v;
    }
}
static E2 felt2() { return gl::e2(felt(), felt()); }
typedef std::vector<E2> Table;
static Table fold(const Table &s, E2 r)
{
    Table o(s.size() / 2);
    for (size_t i = 0; i < o.size(); i++) o[i] = gl::add(s[2 * i], gl::mul(r, gl::sub(s[2 * i + 1], s[2 * i])));
    return o;
}
struct Term {
    E2 coeff;
    std::vector<u32> slots;
};
static std::vector<dpk::PolyOp> program_of(const std::vector<Term> &terms)
{
    std::vector<dpk::ProgramTerm> ts(terms.size());
    for (size_t i = 0; i < terms.size(); i++) {
        ts[i].coeff = terms[i].coeff;
        ts[i].n = (uint8_t)terms[i].slots.size();
        for (size_t f = 0; f < terms[i].slots.size(); f++) ts[i].slot[f] = (uint8_t)terms[i].slots[f];
    }
    std::vector<dpk::PolyOp> ops;
    dpk::program_root(ts.data(), (u32)ts.size(), ops);
    return ops;
}
static E2 eval(const std::vector<Term> &terms, const std::vector<Table> &tabs, size_t pair, u64 t)
{
    E2 g = gl::e2_zero();
    for (const Term &tm : terms) {
        E2 prod = tm.coeff;
        for (u32 f : tm.slots) prod = gl::mul(prod, gl::add(tabs[f][2 * pair], gl::mul_base(gl::sub(tabs[f][2 * pair + 1], tabs[f][2 * pair]), t)));
        g = gl::add(g, prod);
    }
    return g;
}
static u32 degree_of(const std::vector<Term> &terms)
{
    u32 d = 0;
    for (const Term &t : terms) d = std::max(d, (u32)t.slots.size());
    return d;
}
// eq(rho_{first..}, i) over `bits` variables
static E2 eq_at(const std::vector<E2> &rho, u32 first, u32 bits, u64 i)
{
    E2 v = gl::e2_one();
    for (u32 b = 0; b < bits; b++) v = gl::mul(v, ((i >> b) & 1) ? rho[first + b] : gl::sub(gl::e2_one(), rho[first + b]));
    return v;
}

static int failures = 0;

// ---- programs of random lists of terms: the value, the depth, the coefficients' classes and the number of products ----
static void check_programs()
{
    bool ok = true;
    for (u32 rep = 0; rep < 3000 && ok; rep++) {
        const u32 n_tabs = 1 + (u32)(splitmix() % (rep % 3 == 0 ? (u32)dpk::SL_MAX_TABS : 4u)), n_terms = (u32)(splitmix() % 65), most = 1 + (u32)(splitmix() % DPS_MAX_DEGREE);
        std::vector<E2> val;
        for (u32 k = 0; k < n_tabs; k++) val.push_back(felt2());
        std::vector<Term> terms;
        E2 want = gl::e2_zero();
        u32 degree = 0, factors = 0;
        for (u32 i = 0; i < n_terms; i++) {
            const u32 cls = (u32)(splitmix() % 4);
            Term t{cls == 0 ? felt2() : gl::e2(cls == 1 ? 1 : cls == 2 ? gl::P - 1 : felt(), 0), {}};
            for (u32 f = (u32)(splitmix() % (most + 1)); f > 0; f--) t.slots.push_back((u32)(splitmix() % n_tabs));
            E2 prod = t.coeff;
            for (u32 sl : t.slots) prod = gl::mul(prod, val[sl]);
            want = gl::add(want, prod);
            degree = std::max(degree, (u32)t.slots.size()), factors += (u32)t.slots.size();
            terms.push_back(t);
        }
        const std::vector<dpk::PolyOp> ops = program_of(terms);
        std::vector<E2> acc;
        u32 products = 0;
        for (const dpk::PolyOp &o : ops) {
            const u32 kind = o.code & 3, depth = (o.code >> 2) & 15, cls = (o.code >> 6) & 3, slot = o.code >> 8;
            const E2 c = gl::e2(o.c0, o.c1);
            if (kind == dpk::POLY_OP_ENTER) {
                ok = ok && acc.size() == depth && (depth == 0 || depth < degree);
                acc.push_back(c);
            } else if (kind == dpk::POLY_OP_LEAF) {
                ok = ok && acc.size() == depth + 1 && slot < n_tabs && o.w == gl::mul_small(c.c1, (u32)gl::W) &&
                     cls == (c.c1 ? dpk::POLY_COEFF_ANY : c.c0 == 1 ? dpk::POLY_COEFF_ONE : c.c0 == gl::P - 1 ? dpk::POLY_COEFF_MINUS_ONE : dpk::POLY_COEFF_BASE);
                if (ok) acc.back() = gl::add(acc.back(), gl::mul(val[slot], c)), products++;
            } else {
                ok = ok && acc.size() == depth + 1 && depth > 0 && slot < n_tabs;
                if (!ok) break;
                const E2 child = acc.back();
                acc.pop_back();
                acc.back() = gl::add(acc.back(), gl::mul(child, val[slot])), products++;
            }
        }
        ok = ok && acc.size() == 1 && gl::eq(acc[0], want) && products <= factors;
        if (!ok) printf("program %u: %u terms over %u tables\n", rep, n_terms, n_tabs);
    }
    printf("%-60s : %s\n", "programs of random lists of terms", ok ? "ok" : "MISMATCH");
    if (!ok) failures++;
}

// ---- wsum_kernel: one round over 2^log_pairs pairs by `blocks` workgroups ----
struct Launch {
    bool factored = false;     // the weights as products of a low and a high table
    int mail = 0;              // a launch made ahead: 1, the challenge comes by mail, 2, by mail through the relay
    std::vector<u32> only{};   // workgroups that are run (none: all), whose partial sums are compared instead of the launch's
};
template <int NF, bool SKIP1, bool BASE, int REST>
static void run_round(const char *name, u32 log_pairs, u32 blocks, u32 n_tabs, std::vector<std::vector<Term>> polys, bool folds, bool base_tabs, Launch how = Launch())
{
    constexpr int NS = dpk::wsum_sums(NF, SKIP1, REST);
    const size_t n_pairs = (size_t)1 << log_pairs;
    const u32 G = (u32)polys.size();
    dpk::WsumArgs a;
    memset(&a, 0, sizeof a);
    std::vector<Table> src(n_tabs, Table(n_pairs * (folds ? 4 : 2))), tabs;
    std::vector<std::vector<u64>> s0(n_tabs), s1(n_tabs), d0(n_tabs), d1(n_tabs);
    const E2 r = felt2();
    for (u32 k = 0; k < n_tabs; k++) {
        for (E2 &x : src[k]) x = base_tabs ? gl::e2(felt(), 0) : felt2();
        for (E2 &x : src[k]) s0[k].push_back(x.c0), s1[k].push_back(x.c1);
        tabs.push_back(folds ? fold(src[k], r) : src[k]);
        d0[k].assign(2 * n_pairs, 7), d1[k].assign(2 * n_pairs, 7);
        a.tab[k] = dpk::PolyTab{s0[k].data(), base_tabs ? nullptr : s1[k].data(), folds ? d0[k].data() : nullptr, folds ? d1[k].data() : nullptr,
                                folds ? dpk::POLY_PAIR_FOLD : dpk::POLY_PAIR, 0};
    }
    a.n_tabs = n_tabs, a.n_eqs = G, a.n_pairs = n_pairs, a.r0 = r.c0, a.r1 = r.c1;
    std::vector<dpk::PolyOp> ops;
    for (u32 g = 0; g < G; g++) {
        a.degree[g] = degree_of(polys[g]);
        auto p = program_of(polys[g]);
        a.op_begin[g] = (u32)ops.size();
        ops.insert(ops.end(), p.begin(), p.end());
        a.op_end[g] = (u32)ops.size();
        bool base = true;
        for (const Term &t : polys[g]) base = base && t.coeff.c1 == 0;
        if (base) a.base_program |= 1u << g;
    }
    std::copy(ops.begin(), ops.end(), a.ops);
    std::vector<std::vector<E2>> rho(G), R(G);
    std::vector<std::vector<u64>> q0(G), q1(G), lq0(G), lq1(G), hq0(G), hq1(G);
    const size_t lows = (size_t)1 << dpk::EQ_LO_BITS;
    for (u32 g = 0; g < G; g++) {
        if (how.factored) {
            // (the streamed table is not to be read)
            for (size_t i = 0; i < lows; i++) lq0[g].push_back(felt()), lq1[g].push_back(felt());
            for (size_t i = 0; i < (n_pairs + lows - 1) / lows; i++) hq0[g].push_back(felt()), hq1[g].push_back(felt());
            for (size_t i = 0; i < n_pairs; i++)
                R[g].push_back(gl::mul(gl::e2(hq0[g][i / lows], hq1[g][i / lows]), gl::e2(lq0[g][i % lows], lq1[g][i % lows])));
            a.lq0[g] = lq0[g].data(), a.lq1[g] = lq1[g].data(), a.hq0[g] = hq0[g].data(), a.hq1[g] = hq1[g].data();
            continue;
        }
        for (u32 v = 0; v < log_pairs; v++) rho[g].push_back(felt2());
        for (size_t i = 0; i < n_pairs; i++) R[g].push_back(eq_at(rho[g], 0, log_pairs, i)), q0[g].push_back(R[g][i].c0), q1[g].push_back(R[g][i].c1);
        a.q0[g] = q0[g].data(), a.q1[g] = q1[g].data();
    }
    std::vector<u64> partial((size_t)2 * NS * blocks, 0), out(64, 0), dyn((size_t)n_tabs * (BASE ? 2 : 4) * dpk::BLOCK), mail(64, 0), relay(dpk::MAIL_RELAY_WORDS, 0);
    u32 counter = 0;
    if (how.mail) {
        // the mail is there before the launch (workgroups run one after the other here); the arguments hold no challenge
        a.r0 = a.r1 = 0x1234;
        a.wait_first = 1, a.mail = mail.data(), a.relay = how.mail == 2 ? relay.data() : nullptr, a.spin_limit = 1u << 30;
        mail[dpk::MAIL_R] = r.c0, mail[dpk::MAIL_R + 1] = r.c1, mail[dpk::MAIL_SKIP1] = SKIP1 ? 1 : 0;
        u64 chk = 17;
        for (u32 m = dpk::MAIL_R; m < (u32)dpk::MAIL_WORDS; m++) chk ^= dpk::mail_mix(mail[m], m);
        mail[dpk::MAIL_CHK] = chk, mail[dpk::MAIL_SEQ] = 17;
    }
    dpk::FastFin ff;
    memset(&ff, 0, sizeof ff);
    ff.partial = partial.data(), ff.n_blocks = blocks, ff.out_host = out.data(), ff.seq = 17, ff.counter = &counter;
    gridDim = dim3(blocks), blockDim = dim3(dpk::BLOCK);
    const bool whole = how.only.empty();
    if (whole)
        for (u32 b = 0; b < blocks; b++) how.only.push_back(b);
    for (u32 b : how.only) {
        emu::default_group.reset(dpk::BLOCK);
        emu::default_group.dyn = dyn.data();
        std::vector<std::thread> th;
        for (u32 t = 0; t < (u32)dpk::BLOCK; t++)
            th.emplace_back([&, t, b] {
                threadIdx = dim3(t);
                blockIdx = dim3(b, 0, 0);
                dpk::wsum_kernel<NF, SKIP1, BASE, REST>(a, partial.data(), ff);
            });
        for (auto &x : th) x.join();
    }
    bool ok = true;
    if (whole) {
        ok = out[dpk::WSUM_SEQ_SLOT] == 17 && counter == 0;
        u64 chk = 17;
        for (u32 i = 0; i < 2 * NS; i++) chk ^= dpk::rotl64(out[i], i + 1);
        ok = ok && chk == out[dpk::WSUM_CHK_SLOT];
    }
    const size_t stride = (size_t)blocks * dpk::BLOCK;
    // sum of the pairs of workgroups [b, b + n)
    auto compare = [&](u32 b, u32 n, auto &&word) {
        const u32 n0 = SKIP1 ? NF : NF + 1;
        for (u32 g = 0; g < G; g++)
            for (u32 t = 0; t <= a.degree[g]; t++) {
                if (g == 0 && t == 1 && SKIP1) continue;
                const u32 s = g == 0 ? (SKIP1 && t > 0 ? t - 1 : t) : n0 + (g - 1) * dpk::wsum_rest(NF, REST) + t;
                E2 want = gl::e2_zero();
                for (size_t first = (size_t)b * dpk::BLOCK; first < n_pairs; first += stride)
                    for (size_t i = first; i < std::min(n_pairs, first + (size_t)n * dpk::BLOCK); i++) want = gl::add(want, gl::mul(R[g][i], eval(polys[g], tabs, i, t)));
                if (!gl::eq(want, gl::e2(word(2 * s), word(2 * s + 1)))) ok = false, printf("%s: workgroup %u factor %u point %u\n", name, b, g, t);
            }
        for (u32 k = 0; k < n_tabs && folds; k++)
            for (size_t first = (size_t)b * dpk::BLOCK; first < n_pairs; first += stride)
                for (size_t i = 2 * first; i < 2 * std::min(n_pairs, first + (size_t)n * dpk::BLOCK); i++) ok = ok && d0[k][i] == tabs[k][i].c0 && d1[k][i] == tabs[k][i].c1;
    };
    if (whole)
        compare(0, blocks, [&](u32 w) { return out[w]; });
    else
        for (u32 b : how.only) compare(b, 1, [&](u32 w) { return partial[(size_t)w * blocks + b]; });
    printf("%-60s 2^%u pairs, %u workgroups : %s\n", name, log_pairs, blocks, ok ? "ok" : "MISMATCH");
    if (!ok) failures++;
}

// ---- slice_kernel: all rounds from round 1, `wide` workgroups and then one ----
template <int NF>
static void run_resident(const char *name, u32 n_vars, u32 wide, u32 n_tabs, std::vector<std::vector<Term>> polys, u32 base_tabs, bool doubles, u32 last_left)
{
    const u32 G = (u32)polys.size(), n_gpu = n_vars - last_left;
    std::vector<Table> state(n_tabs, Table((size_t)1 << n_vars));
    std::vector<std::vector<u64>> s0(n_tabs), s1(n_tabs), h0(n_tabs), h1(n_tabs);
    for (u32 f = 0; f < n_tabs; f++)
        for (E2 &x : state[f]) x = f < base_tabs ? gl::e2(felt(), 0) : felt2(), s0[f].push_back(x.c0), s1[f].push_back(x.c1);
    std::vector<std::vector<E2>> rho(G);
    std::vector<std::vector<u64>> e0(G, std::vector<u64>((size_t)2 << n_vars)), e1 = e0;
    for (u32 g = 0; g < G; g++) {
        for (u32 v = 0; v < n_vars; v++) rho[g].push_back(felt2());
        for (u32 l = 0; l <= n_vars; l++)
            for (u64 i = 0; i < (u64)1 << (n_vars - l); i++) {
                const E2 v = eq_at(rho[g], l, n_vars - l, i);
                const size_t off = ((size_t)2 << n_vars) - ((size_t)2 << (n_vars - l)) + i;
                e0[g][off] = v.c0, e1[g][off] = v.c1;
            }
    }
    dpk::SliceArgsEqs a;
    memset(&a, 0, sizeof a);
    std::vector<dpk::PolyOp> ops;
    u32 sums = 0;
    a.n_eqs = G;
    for (u32 g = 0; g < G; g++) {
        auto p = program_of(polys[g]);
        a.op_begin[g] = (u32)ops.size();
        ops.insert(ops.end(), p.begin(), p.end());
        a.op_end[g] = (u32)ops.size();
        a.degree[g] = degree_of(polys[g]);
        a.off_q[g] = sums;
        sums += a.degree[g] + 1;
        a.geq0[g] = e0[g].data(), a.geq1[g] = e1[g].data();
    }
    a.n_sums1 = sums;
    for (u32 g = 0; g < G; g++) a.off_d[g] = sums, sums += (g == 0 ? a.degree[g] : a.degree[g] + 1) * (a.degree[g] + 1);
    a.n_sums2 = sums;
    memcpy(a.terms, ops.data(), ops.size() * sizeof(dpk::PolyOp));
    // the trips: of two rounds where the workgroups hold a quad and `doubles`
    std::vector<std::pair<u32, bool>> trips;
    u32 j = 1, pend = 0, n1 = 0;
    u64 len = ((u64)1 << n_vars) / wide;
    if (wide > 1) {
        for (;;) {
            const bool dbl = doubles && len >= 4 && j + 1 < n_gpu;
            if (dbl) a.dbl_mask |= 1u << trips.size();
            trips.push_back({j, dbl});
            pend = dbl ? 2 : 1, j += pend;
            if ((len >> pend) < 2 || j >= n_gpu) break;
            len >>= pend;
        }
        n1 = (u32)trips.size();
        len = (len * wide) >> pend;
    }
    const u64 handed = wide > 1 ? len << pend : 0;
    u32 k2 = 0;
    while (j <= n_gpu) {
        const bool dbl = doubles && len >= 4 && j + 1 <= n_gpu;
        if (dbl) (wide > 1 ? a.dbl_mask2 : a.dbl_mask) |= 1u << k2;
        k2++;
        trips.push_back({j, dbl});
        j += dbl ? 2 : 1;
        len >>= dbl ? 2 : 1;
    }
    a.n_trips = wide > 1 ? n1 : k2;
    a.n_trips2 = wide > 1 ? k2 : 0;
    std::vector<u64> hw0((size_t)G * (handed + 8)), hw1 = hw0;
    a.hw0 = hw0.data(), a.hw1 = hw1.data(), a.hw_stride = (u32)handed + 8;
    for (u32 f = 0; f < n_tabs; f++) {
        h0[f].assign(handed + 1, 0), h1[f].assign(handed + 1, 0);
        a.s0[f] = s0[f].data(), a.s1[f] = f < base_tabs ? nullptr : s1[f].data();
        a.h0[f] = h0[f].data(), a.h1[f] = h1[f].data();
    }
    std::vector<u64> mail(64, 0), relay(dpk::MAIL_RELAY_WORDS, 0), area(dpk::SL_AREA_WORDS, 0), fin(dpk::SL_FIN_AREA_WORDS, 0),
        gctr((size_t)dpk::SL_MAX_GROUPS * dpk::SL_GROUP_WORDS * dpk::SL_CTR_STRIDE, 0);
    u32 gate = 0;
    a.src_len = (u64)1 << n_vars, a.n_vars = n_vars, a.j0 = 1, a.mail = mail.data(), a.relay = relay.data(), a.spin_limit = 1u << 24, a.finish = 1, a.first_go = 2;
    a.out_host = area.data(), a.fin_out = fin.data(), a.seq0 = 500, a.ctr = gctr.data(), a.gate = &gate, a.n_tabs = n_tabs;
    const u32 cap = (u32)(a.src_len / wide);
    gridDim = dim3(wide), blockDim = dim3(dpk::BLOCK);
    std::vector<std::thread> th;
    std::vector<std::unique_ptr<emu::Group>> groups;
    std::vector<std::vector<u64>> lds(wide, std::vector<u64>(dpk::slice_lds_words(n_tabs, cap, dpk::BLOCK, G, dpk::SliceArgsEqs::TERMS), 0xAAAAAAAAAAAAAAAAull));
    for (u32 b = 0; b < wide; b++) {
        groups.emplace_back(new emu::Group());
        groups.back()->reset(dpk::BLOCK);
        groups.back()->dyn = lds[b].data();
        emu::Group *g = groups.back().get();
        for (u32 t = 0; t < (u32)dpk::BLOCK; t++)
            th.emplace_back([=] {
                emu::group = g;
                threadIdx = dim3(t);
                blockIdx = dim3(b, 0, 0);
                dpk::slice_kernel<NF, true, true, dpk::BLOCK, dpk::SliceArgsEqs>(a);
            });
    }
    bool ok = true;
    std::vector<u64> seen(4 * dpk::SL_MAX_SUMS, 0);
    E2 before[2] = {gl::e2_zero(), gl::e2_zero()};  // the last two challenges, the older first
    std::vector<Table> last_state;
    for (size_t k = 0; k < trips.size() && ok; k++) {
        const u32 r = trips[k].first;
        const bool dbl = trips[k].second;
        const u64 seq = 500 + r - 1;
        if (k > 0) {
            mail[dpk::MAIL_R] = before[1].c0, mail[dpk::MAIL_R + 1] = before[1].c1, mail[dpk::MAIL_RA] = before[0].c0, mail[dpk::MAIL_RA + 1] = before[0].c1;
            mail[dpk::MAIL_SKIP1] = 1;
            u64 chk = seq;
            for (u32 i = dpk::MAIL_R; i < (u32)dpk::MAIL_WORDS; i++) chk ^= dpk::mail_mix(mail[i], i);
            mail[dpk::MAIL_CHK] = chk;
            __atomic_store_n(&mail[dpk::MAIL_SEQ], seq, __ATOMIC_SEQ_CST);
        }
        const u32 ns = dbl ? a.n_sums2 : a.n_sums1;
        std::vector<u64> cnt(4 * ns, 0);
        const auto t0 = std::chrono::steady_clock::now();
        for (u32 c = 0; c < 4 * ns && ok;) {
            if (c >= 4 && c < 8) {
                c++;
                continue;
            }
            const u64 v = __atomic_load_n(&area[c], __ATOMIC_SEQ_CST);
            if ((v >> 56) == dpk::sl_tag(seq)) {
                const u64 now = v & dpk::SL_CTR_MASK;
                cnt[c] = now - (k < n1 ? seen[c] : 0);
                seen[c] = now;
                area[c++] = 0;
            } else if (std::chrono::steady_clock::now() - t0 > std::chrono::seconds(60)) {
                printf("%s: no result for the trip of round %u\n", name, r);
                ok = false;
            } else {
                std::this_thread::sleep_for(std::chrono::microseconds(200));
            }
        }
        auto sum_at = [&](u32 i) {
            u64 limb[2];
            for (int l = 0; l < 2; l++) {
                const unsigned __int128 t = (unsigned __int128)cnt[4 * i + 2 * l] + ((unsigned __int128)cnt[4 * i + 2 * l + 1] << 32);
                limb[l] = gl::reduce128((u64)t, (u64)(t >> 64));
            }
            return gl::e2(limb[0], limb[1]);
        };
        auto direct = [&](const std::vector<Table> &tabs, u32 round, u32 g, u32 t) {
            E2 v = gl::e2_zero();
            for (size_t p = 0; p < tabs[0].size() / 2; p++) v = gl::add(v, gl::mul(eq_at(rho[g], round, n_vars - round, p), eval(polys[g], tabs, p, t)));
            return v;
        };
        for (u32 g = 0; g < G && ok; g++) {
            for (u32 t = 0; t <= a.degree[g]; t++)
                if (!(g == 0 && t == 1) && !gl::eq(sum_at(a.off_q[g] + t), direct(state, r, g, t))) ok = false, printf("%s: round %u factor %u point %u\n", name, r, g, t);
            const u32 npt = g == 0 ? a.degree[g] : a.degree[g] + 1;
            for (u32 smp = 0; smp <= a.degree[g] && dbl; smp++) {
                std::vector<Table> tmp;
                for (auto &t : state) tmp.push_back(fold(t, gl::e2(smp, 0)));
                for (u32 ti = 0; ti < npt; ti++)
                    if (!gl::eq(sum_at(a.off_d[g] + smp * npt + ti), direct(tmp, r + 1, g, g == 0 && ti > 0 ? ti + 1 : ti)))
                        ok = false, printf("%s: round %u factor %u sample %u point %u\n", name, r + 1, g, smp, ti);
            }
        }
        last_state = state;
        for (u32 q = 0; q < (dbl ? 2u : 1u); q++) {
            before[0] = before[1], before[1] = felt2();
            for (auto &t : state) t = fold(t, before[1]);
        }
    }
    if (!ok) __atomic_store_n(&mail[dpk::MAIL_SEQ], dpk::MAIL_ABORT_SEQ, __ATOMIC_SEQ_CST);
    for (auto &t : th) t.join();
    if (ok) {
        const u32 left = (u32)last_state[0].size();
        for (u32 f = 0; f < n_tabs; f++)
            for (u32 e = 0; e < left; e++)
                if (fin[2 * (f * left + e)] != last_state[f][e].c0 || fin[2 * (f * left + e) + 1] != last_state[f][e].c1) ok = false;
        for (u64 c : gctr) ok = ok && c == 0;
    }
    printf("%-60s n=%u, %u workgroups, %zu trips : %s\n", name, n_vars, wide, trips.size(), ok ? "ok" : "MISMATCH");
    if (!ok) failures++;
}

int main()
{
    const E2 one = gl::e2_one(), minus = gl::e2(gl::P - 1, 0), half = gl::e2(1234567, 0);
    // the linking sum's shape: v - b^2 v + c b^2 + d b, and s v + s' b
    const std::vector<Term> lp{{one, {0}}, {minus, {1, 1, 0}}, {half, {1, 1}}, {gl::e2(77, 0), {1}}}, ll{{felt2(), {0}}, {felt2(), {1}}};
    const std::vector<Term> p4{{felt2(), {0, 1, 2, 2}}, {felt2(), {2, 3}}, {felt2(), {}}, {one, {3}}}, p2{{felt2(), {0, 3}}, {minus, {1}}}, p1{{half, {2}}, {felt2(), {}}};
    check_programs();
    run_round<3, false, true, 1>("two factors, base tables", 9, 2, 2, {lp, ll}, false, true);
    run_round<3, true, true, 1>("the same, p(1) from the claim, a single workgroup", 5, 1, 2, {lp, ll}, false, true);
    run_round<3, true, false, 1>("base tables folded on the way in", 9, 2, 2, {lp, ll}, true, true);
    run_round<3, true, false, 1>("extension tables folded on the way in", 8, 1, 2, {lp, ll}, true, false);
    run_round<4, true, false, 2>("three factors of degrees 4, 2 and 1", 9, 3, 4, {p4, p2, p1}, true, false);
    run_round<4, false, false, 2>("the same unfolded, every point, one pair", 0, 1, 4, {p4, p2, p1}, false, false);
    run_round<3, true, false, 0>("one factor, extension tables folded on the way in", 9, 2, 4, {lp}, true, false);
    run_round<3, false, true, 0>("the same unfolded over base tables, every point", 6, 1, 4, {lp}, false, true);
    run_round<2, true, false, 2>("degrees 2 and 2 over base tables", 7, 1, 4, {p2, p2}, false, true);
    // a lane takes several pairs, one behind the other
    run_round<3, true, false, 1>("two factors, several pairs a lane", 10, 2, 2, {lp, ll}, true, true);
    run_round<3, false, false, 1>("the same, every point, the challenge by mail", 10, 1, 2, {lp, ll}, true, true, {.mail = 1});
    run_round<4, true, false, 2>("three factors, several pairs a lane, mail through the relay", 10, 3, 4, {p4, p2, p1}, true, false, {.mail = 2});
    run_round<4, false, false, 2>("the same, every point", 9, 1, 4, {p4, p2, p1}, true, false);
    run_round<2, true, false, 2>("degrees 2 and 2, several pairs a lane", 9, 1, 4, {p2, p2}, true, false);
    run_round<3, false, true, 0>("one factor unfolded, several pairs a lane", 9, 1, 4, {lp}, false, true);
    // the weights as a low and a high table: workgroups of a launch whose stride is a run of the low table, two runs of pairs
    run_round<3, true, true, 1>("two factors, base tables, factored weights", 17, 256, 2, {lp, ll}, false, true, {.factored = true, .only = {0, 255}});
    run_round<3, false, false, 1>("two factors folded, every point, factored weights", 17, 256, 2, {lp, ll}, true, false, {.factored = true, .mail = 2, .only = {0, 77}});
    run_round<4, true, false, 2>("three factors folded, factored weights", 17, 256, 4, {p4, p2, p1}, true, false, {.factored = true, .only = {0, 255}});
    run_round<3, true, false, 0>("one factor folded, factored weights", 17, 256, 4, {lp}, true, false, {.factored = true, .only = {0, 128}});
    run_resident<3>("resident, two factors, trips of two rounds", 7, 1, 2, {lp, ll}, 2, true, 0);
    run_resident<3>("resident, one round a trip, the last two rounds left out", 6, 1, 2, {lp, ll}, 1, false, 2);
    run_resident<3>("resident, four workgroups, then one", 9, 4, 2, {lp, ll}, 0, true, 2);
    run_resident<2>("resident, degrees 2 and 2, more pairs than lanes", 10, 1, 4, {p2, p2}, 4, true, 3);
    run_resident<4>("resident, three factors of degrees 4, 2 and 1, two workgroups", 7, 2, 4, {p4, p2, p1}, 1, false, 1);
    printf("%s\n", failures ? "FAILED" : "all cases ok");
    return failures ? 1 : 0;
}
