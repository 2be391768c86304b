// recompute_temporaries on z = c / s with c = v[:, None] + v[None, :] (v made and freed in the list): prints the rewritten
// list, one instruction a line, bases by name.
#include <cstdio>
#include <map>
#include <set>
#include <vector>

#include <bohrium/bh_opcode.h>

#include "ve_hip/rewrite.hpp"

using namespace bohrium;

int main() {
    const int64_t n = 1500;
    bh_base w(n, bh_type::FLOAT32), v(n, bh_type::FLOAT32), c(n * n, bh_type::FLOAT32), q(n * n, bh_type::FLOAT32),
        s(n, bh_type::FLOAT32), z(n * n, bh_type::FLOAT32);
    std::map<const bh_base *, const char *> names{{&w, "w"}, {&v, "v"}, {&c, "c"}, {&q, "q"}, {&s, "s"}, {&z, "z"}};
    auto full = [&](bh_base *b) { return bh_view(b, 0, 2, {n, n}, {n, 1}); };
    auto one = [&](bh_base *b) { return bh_view(b, 0, 1, {n}, {1}); };
    auto rows = [&](bh_base *b) { return bh_view(b, 0, 2, {n, n}, {1, 0}); };
    auto cols = [&](bh_base *b) { return bh_view(b, 0, 2, {n, n}, {0, 1}); };
    std::vector<bh_instruction> program{
        {BH_ADD, {one(&v), one(&w), one(&w)}},     {BH_ADD, {full(&c), rows(&v), cols(&v)}},
        {BH_MULTIPLY, {full(&q), full(&c), full(&c)}}, {BH_ADD_REDUCE, {one(&s), full(&q), bh_view()}},
        {BH_FREE, {one(&q)}},                      {BH_FREE, {one(&v)}},
        {BH_DIVIDE, {full(&z), full(&c), rows(&s)}}, {BH_FREE, {one(&c)}},
        {BH_FREE, {one(&s)}}};
    program[3].constant = bh_constant::make(1, bh_type::INT64);
    std::vector<bh_instruction *> list;
    for (bh_instruction &i : program) list.push_back(&i);
    vehip::RewriteStore store;
    std::printf("rewritten %d\n", vehip::recompute_temporaries(list, store, std::set<bh_base *>()));
    for (const bh_instruction *i : list) {
        std::printf("%s", bh_opcode_text(i->opcode));
        for (const bh_view &o : i->operand)
            std::printf(" %s", o.isConstant() ? "const" : names.count(o.base) ? names[o.base] : "again");
        std::printf("\n");
    }
    return 0;
}
