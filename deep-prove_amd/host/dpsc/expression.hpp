// Symbolic sum-of-products over registered tables, mirroring the Expression type
// the reference's provers build (WitIn / Constant / Challenge with + - *):
// zkml/src/layers/einsum/op_info.rs:137-199, zkml/src/lookup/logup_gkr/circuit.rs:245-284,
// zkml/src/iop/same_poly.rs:94-104.  Challenge(id, pow, scalar, offset) evaluates to
// scalar * challenges[id]^pow + offset.
#pragma once
#include <algorithm>
#include <map>
#include <memory>
#include <stdexcept>
#include <vector>

#include "field.hpp"

namespace dpsc {

struct Monomial {
    F coeff;
    std::vector<uint16_t> wits;  // sorted table indices, repeats allowed
};

class Expression {
public:
    enum class Kind { WitIn, Constant, Challenge, Sum, Product, Neg };

    static Expression WitIn(uint16_t id)
    {
        Expression e(Kind::WitIn);
        e.n_->id = id;
        return e;
    }
    static Expression Constant(const F &c)
    {
        Expression e(Kind::Constant);
        e.n_->scalar = c;
        return e;
    }
    static Expression Challenge(uint16_t id, size_t pow, const F &scalar, const F &offset)
    {
        Expression e(Kind::Challenge);
        e.n_->id = id;
        e.n_->pow = pow;
        e.n_->scalar = scalar;
        e.n_->offset = offset;
        return e;
    }
    static Expression ZERO() { return Constant(F::zero()); }
    static Expression ONE() { return Constant(F::one()); }

    Expression operator+(const Expression &o) const { return binary(Kind::Sum, o); }
    Expression operator*(const Expression &o) const { return binary(Kind::Product, o); }
    Expression operator-(const Expression &o) const { return *this + (-o); }
    Expression operator-() const
    {
        Expression e(Kind::Neg);
        e.n_->a = n_;
        return e;
    }

    // Flatten to monomials with the challenges substituted.  Equal products of
    // tables are merged; monomials whose coefficient cancels to zero are dropped.
    std::vector<Monomial> to_monomials(const std::vector<F> &challenges) const
    {
        std::vector<Monomial> out;
        for_each_monomial(challenges, [&](const F &c, const uint16_t *wits, size_t n) { out.push_back(Monomial{c, std::vector<uint16_t>(wits, wits + n)}); });
        return out;
    }
    // The same, handed to fn(coefficient, table indices, their number) in the order of the index lists.  A layer of five fraction trees is flattened in
    // 1.4 us this way, with a vector of indices for every product on the way and a map of them in 8.4.
    template <class Fn>
    void for_each_monomial(const std::vector<F> &challenges, Fn &&fn) const
    {
        std::vector<Flat> flat;
        flat.reserve(64);
        if (!flatten(*n_, F::one(), challenges, flat)) {
            // (products of more tables than the short form holds)
            std::map<std::vector<uint16_t>, F> acc;
            for (auto &m : expand(*n_, challenges)) acc[m.wits] += m.coeff;
            for (auto &kv : acc)
                if (!kv.second.is_zero()) fn(kv.second, kv.first.data(), kv.first.size());
            return;
        }
        std::sort(flat.begin(), flat.end(), [](const Flat &x, const Flat &y) { return std::lexicographical_compare(x.wits, x.wits + x.n, y.wits, y.wits + y.n); });
        for (size_t i = 0; i < flat.size();) {
            F c = flat[i].coeff;
            size_t j = i + 1;
            for (; j < flat.size() && flat[j].n == flat[i].n && std::equal(flat[i].wits, flat[i].wits + flat[i].n, flat[j].wits); j++) c += flat[j].coeff;
            if (!c.is_zero()) fn(c, flat[i].wits, (size_t)flat[i].n);
            i = j;
        }
    }

    // utils::eval_by_expr_with_instance restricted to what the callers pass:
    // witness evaluations and challenges (zkml/src/lookup/logup_gkr/prover.rs:43-58)
    F evaluate(const std::vector<F> &wit_evals, const std::vector<F> &challenges) const { return eval(*n_, wit_evals, challenges); }

    size_t degree() const
    {
        size_t d = 0;
        for (auto &m : to_monomials_symbolic()) d = std::max(d, m);
        return d;
    }

private:
    struct Node {
        Kind kind;
        uint16_t id = 0;
        size_t pow = 0;
        F scalar, offset;
        std::shared_ptr<const Node> a, b;
    };
    std::shared_ptr<Node> n_;
    explicit Expression(Kind k) : n_(std::make_shared<Node>()) { n_->kind = k; }
    Expression binary(Kind k, const Expression &o) const
    {
        Expression e(k);
        e.n_->a = n_;
        e.n_->b = o.n_;
        return e;
    }
    static F challenge_value(const Node &n, const std::vector<F> &ch)
    {
        if (n.id >= ch.size()) throw std::out_of_range("Expression: challenge index out of range");
        return n.scalar * ch[n.id].pow(n.pow) + n.offset;
    }
    // A monomial of at most MAX_FLAT tables, in place: what a product costs is its coefficient
    static constexpr size_t MAX_FLAT = 8;
    struct Flat {
        F coeff;
        uint32_t n;
        uint16_t wits[MAX_FLAT];  // sorted
    };
    // Appends scale * (the node's monomials) to `out`; false: one has more than MAX_FLAT tables
    static bool flatten(const Node &n, const F &scale, const std::vector<F> &ch, std::vector<Flat> &out)
    {
        if (scale.is_zero()) return true;
        auto constant = [&](const F &c) {
            if (!c.is_zero()) out.push_back(Flat{scale * c, 0, {}});
            return true;
        };
        switch (n.kind) {
        case Kind::WitIn: out.push_back(Flat{scale, 1, {n.id}}); return true;
        case Kind::Constant: return constant(n.scalar);
        case Kind::Challenge: return constant(challenge_value(n, ch));
        case Kind::Neg: return flatten(*n.a, -scale, ch, out);
        case Kind::Sum: return flatten(*n.a, scale, ch, out) && flatten(*n.b, scale, ch, out);
        case Kind::Product: {
            // a constant scales the other factor, a single table goes into each of its monomials
            for (const Node *c : {n.a.get(), n.b.get()}) {
                const Node &other = c == n.a.get() ? *n.b : *n.a;
                if (c->kind == Kind::Constant || c->kind == Kind::Challenge) {
                    const F v = c->kind == Kind::Constant ? c->scalar : challenge_value(*c, ch);
                    if (!v.is_zero()) return flatten(other, scale * v, ch, out);
                }
                if (c->kind != Kind::WitIn) continue;
                const size_t from = out.size();
                if (!flatten(other, scale, ch, out)) return false;
                for (size_t x = from; x < out.size(); x++) {
                    Flat &m = out[x];
                    if (m.n == MAX_FLAT) return false;
                    size_t i = m.n++;
                    for (; i > 0 && m.wits[i - 1] > c->id; i--) m.wits[i] = m.wits[i - 1];
                    m.wits[i] = c->id;
                }
                return true;
            }
            // both factors' monomials behind what is there, their products behind those, then down over the factors
            const size_t at = out.size();
            if (!flatten(*n.a, F::one(), ch, out)) return false;
            const size_t mid = out.size();
            if (!flatten(*n.b, scale, ch, out)) return false;
            const size_t end = out.size();
            for (size_t x = at; x < mid; x++)
                for (size_t y = mid; y < end; y++) {
                    const Flat p = out[x], q = out[y];
                    Flat m;
                    m.coeff = p.n == 0 && p.coeff == F::one() ? q.coeff : q.n == 0 && q.coeff == F::one() ? p.coeff : p.coeff * q.coeff;
                    if (m.coeff.is_zero()) continue;
                    if (p.n + q.n > MAX_FLAT) return false;
                    m.n = p.n + q.n;
                    std::merge(p.wits, p.wits + p.n, q.wits, q.wits + q.n, m.wits);
                    out.push_back(m);
                }
            out.erase(out.begin() + (ptrdiff_t)at, out.begin() + (ptrdiff_t)end);
            return true;
        }
        }
        return true;
    }
    static std::vector<Monomial> expand(const Node &n, const std::vector<F> &ch)
    {
        std::vector<Monomial> out;
        expand_into(n, F::one(), ch, out);
        return out;
    }
    // appends scale * (the node's monomials) to `out`: long sums (one `+` per term, as the provers build them)
    // cost one pass, not one copy of everything so far per `+`
    static void expand_into(const Node &n, const F &scale, const std::vector<F> &ch, std::vector<Monomial> &out)
    {
        if (scale.is_zero()) return;
        switch (n.kind) {
        case Kind::WitIn: out.push_back(Monomial{scale, {n.id}}); return;
        case Kind::Constant:
            if (!n.scalar.is_zero()) out.push_back(Monomial{scale * n.scalar, {}});
            return;
        case Kind::Challenge: {
            const F c = challenge_value(n, ch);
            if (!c.is_zero()) out.push_back(Monomial{scale * c, {}});
            return;
        }
        case Kind::Neg: expand_into(*n.a, -scale, ch, out); return;
        case Kind::Sum:
            expand_into(*n.a, scale, ch, out);
            expand_into(*n.b, scale, ch, out);
            return;
        case Kind::Product: {
            std::vector<Monomial> v, w;
            expand_into(*n.a, F::one(), ch, v);
            expand_into(*n.b, scale, ch, w);
            out.reserve(out.size() + v.size() * w.size());
            for (auto &x : v)
                for (auto &y : w) {
                    Monomial m{x.coeff * y.coeff, x.wits};
                    if (m.coeff.is_zero()) continue;
                    m.wits.insert(m.wits.end(), y.wits.begin(), y.wits.end());
                    std::sort(m.wits.begin(), m.wits.end());
                    out.push_back(std::move(m));
                }
            return;
        }
        }
    }
    static F eval(const Node &n, const std::vector<F> &w, const std::vector<F> &ch)
    {
        switch (n.kind) {
        case Kind::WitIn:
            if (n.id >= w.size()) throw std::out_of_range("Expression: witness index out of range");
            return w[n.id];
        case Kind::Constant: return n.scalar;
        case Kind::Challenge: return challenge_value(n, ch);
        case Kind::Neg: return -eval(*n.a, w, ch);
        case Kind::Sum: return eval(*n.a, w, ch) + eval(*n.b, w, ch);
        case Kind::Product: return eval(*n.a, w, ch) * eval(*n.b, w, ch);
        }
        return F::zero();
    }
    std::vector<size_t> to_monomials_symbolic() const
    {
        std::vector<size_t> out;
        degrees(*n_, out);
        return out;
    }
    static void degrees(const Node &n, std::vector<size_t> &out)
    {
        switch (n.kind) {
        case Kind::WitIn: out.push_back(1); break;
        case Kind::Constant:
        case Kind::Challenge: out.push_back(0); break;
        case Kind::Neg: degrees(*n.a, out); break;
        case Kind::Sum:
            degrees(*n.a, out);
            degrees(*n.b, out);
            break;
        case Kind::Product: {
            std::vector<size_t> x, y;
            degrees(*n.a, x);
            degrees(*n.b, y);
            size_t mx = 0, my = 0;
            for (auto v : x) mx = std::max(mx, v);
            for (auto v : y) my = std::max(my, v);
            out.push_back(mx + my);
            break;
        }
        }
    }
};

}  // namespace dpsc
