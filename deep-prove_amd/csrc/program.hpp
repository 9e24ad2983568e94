// The nested programs of sums of several terms, built on the host (kernels.hpp says how they are walked).
#pragma once
#include <cstring>
#include <utility>
#include <vector>

#include "kernels.hpp"  // (behind dpsumcheck.h)

namespace dpk {

// Nested (Horner) form of a sum of terms: the table found in most of the remaining terms is factored out of them, recursively.
struct ProgramTerm {
    E2 coeff;
    uint8_t n, slot[DPS_MAX_FACTORS];  // remaining factors, as slots below SL_MAX_TABS
};

inline PolyOp program_op(u32 kind, u32 d, u32 slot, E2 c)
{
    PolyOp op;
    memset(&op, 0, sizeof op);
    op.c0 = c.c0;
    op.c1 = c.c1;
    op.w = gl::mul_small(c.c1, (u32)gl::W);
    const u32 cls = c.c1 ? POLY_COEFF_ANY : c.c0 == 1 ? POLY_COEFF_ONE : c.c0 == gl::P - 1 ? POLY_COEFF_MINUS_ONE : POLY_COEFF_BASE;
    op.code = kind | d << 2 | (kind == POLY_OP_LEAF ? cls : 0) << 6 | slot << 8;
    return op;
}

// Appends the operations of the node of depth `depth` with these terms, each of at least one factor (their order is not kept); returns
// its number of products.
inline u32 program_build(ProgramTerm *t, u32 n, u32 depth, std::vector<PolyOp> &ops)
{
    u32 products = 0;
    while (n) {
        uint8_t count[SL_MAX_TABS] = {0};
        u32 best = t[0].slot[0];
        for (u32 i = 0; i < n; i++)
            for (u32 f = 0; f < t[i].n; f++) {
                const u32 sl = t[i].slot[f];
                bool again = false;
                for (u32 q = 0; q < f; q++) again = again || t[i].slot[q] == sl;
                if (again) continue;
                count[sl]++;
                if (count[sl] > count[best] || (count[sl] == count[best] && sl < best)) best = sl;
            }
        // its terms to the front, those that end here behind the others among them
        u32 inner = 0, with = 0;
        E2 ending = gl::e2_zero();
        for (u32 i = 0; i < n; i++) {
            ProgramTerm &p = t[i];
            u32 f = 0;
            while (f < p.n && p.slot[f] != best) f++;
            if (f == p.n) continue;
            p.slot[f] = p.slot[--p.n];
            if (p.n) {
                std::swap(t[i], t[with]);
                std::swap(t[with++], t[inner++]);
            } else {
                ending = gl::add(ending, p.coeff);
                std::swap(t[i], t[with++]);
            }
        }
        if (inner) {
            ops.push_back(program_op(POLY_OP_ENTER, depth + 1, 0, ending));
            products += program_build(t, inner, depth + 1, ops);
            ops.push_back(program_op(POLY_OP_LEAVE, depth + 1, best, gl::e2_zero()));
        } else {
            ops.push_back(program_op(POLY_OP_LEAF, depth, best, ending));
        }
        products++;
        t += with, n -= with;
    }
    return products;
}

// A whole program: its first operation enters the root with the constant.  Returns the number of products.
inline u32 program_root(ProgramTerm *t, u32 n, std::vector<PolyOp> &ops)
{
    E2 root = gl::e2_zero();
    u32 m = 0;
    for (u32 i = 0; i < n; i++)
        if (t[i].n)
            std::swap(t[i], t[m++]);
        else
            root = gl::add(root, t[i].coeff);
    ops.push_back(program_op(POLY_OP_ENTER, 0, 0, root));
    return program_build(t, m, 0, ops);
}

}  // namespace dpk
