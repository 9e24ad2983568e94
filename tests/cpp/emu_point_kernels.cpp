// The kernels that take their weights from a point -- axis_point_{col,wide,row,short}_kernel, eval_point_kernel, combine_kernel,
// eval_tables_kernel -- run on the CPU through tests/cpp/emu/hip/hip_runtime.h, one workgroup after the other with one host thread
// per lane, and compared with plain loops over the definitions.  Every buffer is exactly as large as the launch may use, so that the
// sanitizers see an entry too far.  Built with the host sanitizers and a fill pattern for uninitialised locals by
// tests/test_kernel_emulation.py.
#include <thread>
#include <vector>

#include "dpsumcheck.h"
#include "kernels.hpp"

using gl::E2;
using gl::u32;
using gl::u64;

static u64 sm_state = 4242;
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
static int failures = 0;
static void report(const char *name, bool ok)
{
    printf("%-90s : %s\n", name, ok ? "ok" : "MISMATCH");
    fflush(stdout);
    if (!ok) failures++;
}

template <class K, class... A>
static void launch(dim3 grid, K kernel, A... args)
{
    gridDim = grid;
    blockDim = dim3(dpk::BLOCK);
    for (u32 y = 0; y < grid.y; y++)
        for (u32 x = 0; x < grid.x; x++) {
            emu::default_group.reset(dpk::BLOCK);
            std::vector<std::thread> th;
            for (u32 t = 0; t < (u32)dpk::BLOCK; t++)
                th.emplace_back([=] {
                    threadIdx = dim3(t);
                    blockIdx = dim3(x, y, 0);
                    kernel(args...);
                });
            for (auto &t : th) t.join();
        }
}

static std::vector<E2> random_point(u32 m)
{
    std::vector<E2> p(m);
    for (auto &x : p) x = felt2();
    return p;
}
static void put_point(u64 *out, const std::vector<E2> &p)
{
    for (size_t i = 0; i < p.size(); i++) out[2 * i] = p[i].c0, out[2 * i + 1] = p[i].c1;
}
static E2 eq_at(const std::vector<E2> &p, u64 k)
{
    E2 v = gl::e2_one();
    for (size_t b = 0; b < p.size(); b++) v = gl::mul(v, ((k >> b) & 1) ? p[b] : gl::sub(gl::e2_one(), p[b]));
    return v;
}
// the same as a table
static std::vector<E2> eq_table(const std::vector<E2> &p)
{
    std::vector<E2> t{gl::e2_one()};
    for (size_t b = 0; b < p.size(); b++) {
        const size_t n = t.size();
        t.resize(2 * n);
        for (size_t i = 0; i < n; i++) {
            const E2 hi = gl::mul(t[i], p[b]);
            t[n + i] = hi;
            t[i] = gl::sub(t[i], hi);
        }
    }
    return t;
}

// a table of one of the kinds of entries
struct Entries {
    int kind;  // 0 base, 1 extension, 8 int64, 2 int16
    std::vector<u64> c0, c1;
    std::vector<int64_t> i64;
    std::vector<int16_t> i16;
    Entries(int k, size_t n) : kind(k)
    {
        for (size_t i = 0; i < n; i++) {
            if (k == 8) i64.push_back((int64_t)(splitmix() % 4096) - 2048);
            if (k == 2) i16.push_back((int16_t)(splitmix() & 0xFFFF));
            if (k <= 1) c0.push_back(felt());
            if (k == 1) c1.push_back(felt());
        }
    }
    const void *p0() const { return kind == 8 ? (const void *)i64.data() : kind == 2 ? (const void *)i16.data() : (const void *)c0.data(); }
    const u64 *p1() const { return kind == 1 ? c1.data() : nullptr; }
    E2 at(size_t i) const
    {
        if (kind == 8) return gl::e2(gl::from_i64(i64[i]), 0);
        if (kind == 2) return gl::e2(gl::from_i64(i16[i]), 0);
        return gl::e2(c0[i], kind == 1 ? c1[i] : 0);
    }
};

enum Way { COL, WIDE, ROW, SHORT };
// A tensor of `dims`, stored with `padded` dims, one axis contracted (-1: none).  `row_len`, `padded_len`: how the outputs are laid
// out.  COL: `per_slice` values of k a workgroup (0: all); ROW: steps of 512 a workgroup, `waves` wavefronts an output; WIDE,
// SHORT: `blocks` workgroups that go over all outputs
template <int KIND>
static void axis(const char *name, Way way, std::vector<u64> dims, std::vector<u64> padded, int ax, u64 row_len, u64 padded_len, u64 per_slice, u32 waves, u32 blocks)
{
    const u32 n = (u32)dims.size();
    std::vector<u64> strides(n, 1);
    u64 size = 1;
    for (u32 d = n; d-- > 0;) strides[d] = size, size *= padded[d];
    // (as much of the storage as the unpadded region reaches)
    u64 last = 1;
    for (u32 d = 0; d < n; d++) last += (dims[d] - 1) * strides[d];
    const Entries in(KIND, last);
    dpk::AxisPointArgs a;
    memset(&a, 0, sizeof a);
    a.in0 = in.p0(), a.in1 = in.p1();
    a.K = a.P = a.C = 1;
    for (int d = 0; d < (int)n; d++) {
        if (d == ax) {
            a.K = dims[d], a.stride_k = strides[d];
        } else if (d < ax) {
            a.pre_dims[a.n_pre] = dims[d], a.pre_strides[a.n_pre++] = strides[d], a.P *= dims[d];
        } else {
            a.post_dims[a.n_post] = dims[d], a.post_strides[a.n_post++] = strides[d], a.C *= dims[d];
        }
    }
    while (ax >= 0 && ((u64)1 << a.m) < a.K) a.m++;
    const auto point = random_point(a.m);
    put_point(a.p, point);
    const u64 outputs = a.P * a.C, rows = outputs / row_len;
    a.row_len = row_len, a.padded_len = padded_len, a.n_pads = rows * (padded_len - row_len);
    std::vector<u64> o0(rows * padded_len, ~0ull), o1(rows * padded_len, ~0ull);
    a.o0 = o0.data(), a.o1 = o1.data();
    a.waves_per_out = waves;
    a.n_slices = 1;
    const u64 steps = (a.K + 511) / 512, units = way == ROW ? steps : a.K;
    a.k_per_slice = per_slice ? per_slice : units;
    if (way == COL || way == ROW) a.n_slices = (u32)((units + a.k_per_slice - 1) / a.k_per_slice);
    const u64 tiles = (a.C + 63) / 64;
    dim3 grid(way == COL ? (u32)(a.P * tiles) : way == ROW ? (u32)((outputs + 4 / waves - 1) / (4 / waves)) : blocks, a.n_slices);
    std::vector<u64> p0((size_t)a.n_slices * outputs, ~0ull), p1(p0);
    std::vector<u32> counters(grid.x, 0);
    if (a.n_slices > 1) a.part0 = p0.data(), a.part1 = p1.data(), a.counters = counters.data();
    if (way == COL) launch(grid, dpk::axis_point_col_kernel<KIND>, a);
    if (way == WIDE) launch(grid, dpk::axis_point_wide_kernel<KIND>, a);
    if (way == ROW) launch(grid, dpk::axis_point_row_kernel<KIND>, a);
    if (way == SHORT) {
        if (a.K <= 64)
            launch(grid, dpk::axis_point_short_kernel<KIND, 1>, a);
        else if (a.K <= 128)
            launch(grid, dpk::axis_point_short_kernel<KIND, 2>, a);
        else
            launch(grid, dpk::axis_point_short_kernel<KIND, 4>, a);
    }
    bool ok = true;
    for (u32 c : counters) ok = ok && c == 0;
    const auto weights = eq_table(point);
    auto offset = [](u64 flat, u32 n_dims, const u64 *d, const u64 *s) {
        u64 off = 0;
        for (u32 i = n_dims; i-- > 0;) off += flat % d[i] * s[i], flat /= d[i];
        return off;
    };
    for (u64 o = 0; o < outputs && ok; o++) {
        const u64 base = offset(o / a.C, a.n_pre, a.pre_dims, a.pre_strides) + offset(o % a.C, a.n_post, a.post_dims, a.post_strides);
        E2 want = gl::e2_zero();
        for (u64 k = 0; k < a.K; k++) want = gl::add(want, gl::mul(in.at(base + k * a.stride_k), weights[k]));
        const u64 at = o / row_len * padded_len + o % row_len;
        ok = gl::eq(want, gl::e2(o0[at], o1[at]));
    }
    for (u64 r = 0; r < rows; r++)
        for (u64 c = row_len; c < padded_len; c++) ok = ok && o0[r * padded_len + c] == 0 && o1[r * padded_len + c] == 0;
    report(name, ok);
}

template <int KIND>
static void evaluate(u32 n, u32 blocks)
{
    const Entries t(KIND, (size_t)1 << n);
    const auto point = random_point(n);
    std::vector<u64> area(dpk::WS_OFF_PARTIAL + 2 * blocks, 0), out(64, 0);
    dpk::EvalArgs a;
    memset(&a, 0, sizeof a);
    a.t0 = t.p0(), a.t1 = t.p1();
    a.n = n;
    a.n_rows = n > dpk::EVAL_LO_BITS ? 1ull << (n - dpk::EVAL_LO_BITS) : 1;
    a.rows_per_block = a.n_rows / blocks;
    put_point(a.p, point);
    dpk::FastFin ff;
    memset(&ff, 0, sizeof ff);
    ff.partial = area.data() + dpk::WS_OFF_PARTIAL;
    ff.n_blocks = blocks;
    ff.out_host = out.data();
    ff.seq = 77;
    ff.counter = reinterpret_cast<u32 *>(area.data() + dpk::WS_OFF_COUNTER);
    const auto weights = eq_table(point);
    E2 want = gl::e2_zero();
    for (size_t i = 0; i < weights.size(); i++) want = gl::add(want, gl::mul(t.at(i), weights[i]));
    bool ok = true;
    for (int pass = 0; pass < 2; pass++) {  // (the second finds the counter the first one left)
        out[0] = out[1] = ~0ull;
        launch(dim3(blocks), dpk::eval_point_kernel<KIND>, a, ff);
        ok = ok && gl::eq(want, gl::e2(out[0], out[1])) && out[dpk::HOST_SEQ_SLOT] == 77 && *ff.counter == 0;
    }
    char name[80];
    snprintf(name, sizeof name, "evaluation of 2^%u entries of kind %d, %u workgroups", n, KIND, blocks);
    report(name, ok);
}

struct Item {
    int what;  // 0 base table, 1 extension table, 2 eq table
    u32 vars;
};
// tables of 2^n entries from lists of items, descriptors in the arguments or in memory
template <int STEPS>
static void combine(const char *name, u32 n, std::vector<std::vector<Item>> tables, bool inside, u32 blocks)
{
    std::vector<dpk::CombJob> jobs;
    std::vector<dpk::CombItem> items;
    std::vector<u64> points;
    std::vector<Entries> kept;
    for (auto &t : tables)
        for (auto &it : t) kept.emplace_back(it.what == 1 ? 1 : 0, it.what == 2 ? 0 : (size_t)1 << it.vars);
    std::vector<std::vector<u64>> o0(tables.size(), std::vector<u64>((size_t)1 << n, ~0ull)), o1(o0);
    std::vector<std::vector<E2>> want;
    size_t at = 0;
    for (size_t j = 0; j < tables.size(); j++) {
        jobs.push_back(dpk::CombJob{o0[j].data(), o1[j].data(), (u32)items.size(), (u32)tables[j].size()});
        want.emplace_back((size_t)1 << n, gl::e2_zero());
        for (auto &it : tables[j]) {
            const Entries &e = kept[at++];
            const E2 c = felt2();
            dpk::CombItem d;
            memset(&d, 0, sizeof d);
            d.c0 = c.c0, d.c1 = c.c1, d.len = (u64)1 << it.vars, d.n_bits = it.vars;
            std::vector<E2> values;
            if (it.what == 2) {
                const auto p = random_point(it.vars);
                d.point_off = (u32)points.size();
                for (auto &x : p) points.push_back(x.c0), points.push_back(x.c1);
                values = eq_table(p);
            } else {
                d.t0 = e.c0.data(), d.t1 = e.p1();
                for (size_t i = 0; i < d.len; i++) values.push_back(e.at(i));
            }
            items.push_back(d);
            for (size_t i = 0; i < values.size(); i++) want[j][i] = gl::add(want[j][i], gl::mul(c, values[i]));
        }
    }
    std::vector<u64> words;
    auto add = [&](const void *p, size_t bytes) { words.insert(words.end(), (const u64 *)p, (const u64 *)p + bytes / 8); };
    add(jobs.data(), jobs.size() * sizeof jobs[0]);
    add(items.data(), items.size() * sizeof items[0]);
    words.insert(words.end(), points.begin(), points.end());
    dpk::CombArgs a;
    memset(&a, 0, sizeof a);
    a.n_out = (u64)1 << n, a.n_jobs = (u32)jobs.size(), a.n_items = (u32)items.size();
    if (inside) {
        if (words.size() > dpk::COMB_INLINE_WORDS) abort();
        memcpy(a.words, words.data(), words.size() * 8);
    } else {
        a.src = words.data();
    }
    launch(dim3(blocks, (u32)jobs.size()), dpk::combine_kernel<STEPS>, a);
    bool ok = true;
    for (size_t j = 0; j < jobs.size(); j++)
        for (size_t i = 0; i < want[j].size(); i++) ok = ok && gl::eq(want[j][i], gl::e2(o0[j][i], o1[j][i]));
    report(name, ok);
}

static void evaluate_tables(std::vector<Item> tables, u32 shares)
{
    u32 most = 0;
    for (auto &t : tables) most = std::max(most, t.vars);
    const auto point = random_point(most);
    std::vector<Entries> kept;
    std::vector<dpk::EvalTable> desc;
    for (auto &t : tables) kept.emplace_back(t.what, (size_t)1 << t.vars);
    for (size_t i = 0; i < tables.size(); i++) desc.push_back(dpk::EvalTable{kept[i].c0.data(), kept[i].p1(), tables[i].vars, 0});
    std::vector<u64> partial(2 * tables.size() * shares, ~0ull), fin(dpk::SL_FIN_AREA_WORDS, 0);
    u32 counter = 0;
    dpk::EvalTablesArgs a;
    memset(&a, 0, sizeof a);
    a.tables = desc.data(), a.n_tables = (u32)desc.size(), a.shares = shares;
    a.partial = partial.data(), a.counter = &counter, a.fin_out = fin.data(), a.seq = 55;
    put_point(a.p, point);
    launch(dim3(shares, (u32)desc.size()), dpk::eval_tables_kernel, a);
    bool ok = counter == 0 && fin[dpk::SL_FIN_SEQ_SLOT] == 55;
    u64 chk = 55;
    for (size_t i = 0; i < tables.size(); i++) {
        E2 want = gl::e2_zero();
        const auto weights = eq_table(std::vector<E2>(point.begin(), point.begin() + tables[i].vars));
        for (size_t k = 0; k < weights.size(); k++) want = gl::add(want, gl::mul(kept[i].at(k), weights[k]));
        ok = ok && gl::eq(want, gl::e2(fin[2 * i], fin[2 * i + 1]));
        chk ^= dpk::sl_fin_mix(fin[2 * i], (u32)(2 * i)) ^ dpk::sl_fin_mix(fin[2 * i + 1], (u32)(2 * i + 1));
    }
    ok = ok && fin[dpk::SL_FIN_CHK_SLOT] == chk;
    char name[80];
    snprintf(name, sizeof name, "%zu tables at a point, %u shares each", tables.size(), shares);
    report(name, ok);
}

int main()
{
    // the weights as the tests' tables make them are the definition's
    {
        const auto p = random_point(5);
        const auto t = eq_table(p);
        bool ok = true;
        for (u64 k = 0; k < 32; k++) ok = ok && gl::eq(t[k], eq_at(p, k));
        report("eq table against the definition", ok);
    }
    axis<8>("tiles: one workgroup a tile, rows padded, stored padded", COL, {3, 70, 40}, {4, 128, 64}, 1, 40, 64, 0, 1, 0);
    axis<2>("tiles: two of them, k shared by three workgroups", COL, {70, 100}, {70, 100}, 0, 100, 128, 24, 1, 0);
    axis<1>("tiles: more values than weights are made for together, shared", COL, {600, 33}, {600, 33}, 0, 33, 33, 301, 1, 0);
    axis<0>("tiles: a tile of one axis before and two behind", COL, {2, 9, 5, 7}, {2, 16, 5, 8}, 1, 35, 64, 0, 1, 0);
    axis<8>("a thread an output: several passes, rows padded", WIDE, {2, 9, 300}, {2, 16, 512}, 1, 300, 512, 0, 1, 2);
    axis<1>("a thread an output: extension entries, two axes around", WIDE, {5, 3, 77}, {5, 4, 77}, 1, 385, 385, 0, 1, 1);
    axis<2>("a thread an output: as many values as weights", WIDE, {128, 40}, {128, 40}, 0, 40, 64, 0, 1, 1);
    axis<0>("a thread an output: nothing contracted", WIDE, {3, 5, 20}, {4, 8, 32}, -1, 100, 128, 0, 1, 1);
    axis<8>("rows: a wavefront an output", ROW, {5, 1100}, {8, 2048}, 1, 5, 8, 0, 1, 0);
    axis<2>("rows: two wavefronts an output, three steps", ROW, {5, 1100}, {5, 1100}, 1, 5, 8, 0, 2, 0);
    axis<1>("rows: four wavefronts an output, fewer steps than wavefronts", ROW, {3, 1030}, {3, 1030}, 1, 3, 4, 0, 4, 0);
    axis<0>("rows: adjacent outputs, four wavefronts", ROW, {2, 700, 3}, {2, 1024, 4}, 1, 6, 8, 0, 4, 0);
    axis<1>("rows: shared by three workgroups", ROW, {2, 2900}, {2, 2900}, 1, 2, 2, 2, 4, 0);
    axis<8>("rows: shared, one output of one axis", ROW, {4000}, {4000}, 0, 1, 1, 5, 4, 0);
    axis<8>("short rows: 64 values, several passes", SHORT, {75, 64}, {128, 64}, 1, 75, 128, 0, 1, 1);
    axis<1>("short rows: one value", SHORT, {41, 1}, {41, 1}, 1, 41, 64, 0, 1, 1);
    axis<2>("short rows: 100 values, adjacent outputs", SHORT, {7, 100, 3}, {8, 128, 4}, 1, 3, 4, 0, 1, 1);
    axis<0>("short rows: 200 values", SHORT, {19, 200}, {19, 256}, 1, 19, 32, 0, 1, 2);
    evaluate<0>(0, 1);
    evaluate<1>(1, 1);
    evaluate<8>(5, 1);
    evaluate<2>(10, 1);
    evaluate<0>(11, 1);
    evaluate<1>(13, 2);
    evaluate<8>(14, 4);
    combine<1>("combined tables: one entry", 0, {{{0, 0}, {1, 0}, {2, 0}}}, true, 1);
    combine<1>("combined tables: shorter than a row, zero-padded items", 4, {{{0, 4}, {1, 2}, {2, 3}, {2, 0}, {1, 0}}, {{2, 4}}}, true, 1);
    combine<1>("combined tables: rows of 512, more workgroups than one, descriptors in memory", 12, {{{2, 12}, {0, 11}, {1, 12}, {2, 9}, {2, 11}, {2, 12}}, {{1, 10}}}, false, 3);
    combine<2>("combined tables: rows of 1024", 13, {{{2, 13}, {1, 13}, {2, 12}}}, true, 2);
    {
        std::vector<Item> many;
        for (u32 i = 0; i < 70; i++) many.push_back(Item{(int)(i % 3), 3});
        combine<1>("combined tables: more items than are staged together", 3, {many, {{2, 3}}}, false, 1);
    }
    evaluate_tables({{0, 0}, {1, 4}, {0, 11}}, 1);
    evaluate_tables({{1, 13}, {0, 12}, {1, 3}, {0, 0}}, 4);
    printf("%s\n", failures ? "FAILED" : "all cases ok");
    return failures ? 1 : 0;
}
