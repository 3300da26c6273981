// Prints a model's product rules and the tables the kernels read (build_plan,
// build_lin_plan and moment_table in imr-mlp_amd/csrc/model.cpp) as plain
// text for the host tests in test_capi_host.py:
//   K B T K4 dummy red0 pad M
//   basic: B lines "mu a b c";  times: T lines "l r c o"
//   forward and reverse rules: a step table each ("nlev nsteps", the
//   level_step line, nsteps * 64 lines "x y")
//   linear fit: "dummy one L0 nL priv nslots nchunks S", slot_basic, map,
//   chunk_s0, chunk_scalar, slot_mask, slot_L, then the step tables of the
//   forward rules and of the Jacobian (nchunks -1: no linear plan)
//   moment tables: the count, then per degree "nu entries groups", the table
//   and its shifts
#include "mtpx_internal.hpp"

#include <cstdio>
#include <fstream>
#include <sstream>

template <class T>
static void line(const std::vector<T> &v)
{
    for (T x : v)
        std::printf("%lld ", (long long)x);
    std::printf("\n");
}

static void table(const std::vector<int> &level_step, const std::vector<int> &steps)
{
    std::printf("%zu %zu\n", level_step.size() - 1, steps.size() / (2 * mtpx::kWave));
    line(level_step);
    for (size_t i = 0; i < steps.size(); i += 2)
        std::printf("%d %d\n", steps[i], steps[i + 1]);
}

int main(int argc, char **argv)
{
    if (argc != 2) {
        std::fprintf(stderr, "usage: %s model.mtp\n", argv[0]);
        return 2;
    }
    std::ifstream f(argv[1]);
    std::stringstream ss;
    ss << f.rdbuf();
    mtpx::Model m;
    mtpx::Plan p;
    std::string err;
    if (!mtpx::parse_mtp(ss.str(), m, err) || !mtpx::build_plan(m, p, err)) {
        std::fprintf(stderr, "%s\n", err.c_str());
        return 1;
    }
    std::printf("%d %d %d %d %d %d %d %d\n", m.K, m.B, m.T, p.K4, p.dummy, p.red0,
                mtpx::kRulePad, m.M);
    line(m.basic);
    line(m.times);
    table(p.fwd_level_step, p.fwd_steps);
    table(p.bwd_level_step, p.bwd_steps);
    mtpx::LinPlan lp;
    const bool lin = mtpx::build_lin_plan(m, p, lp, err);
    std::printf("%d %d %d %d %d %d %d %d\n", lp.dummy, lp.one, lp.L0, lp.nL, lp.priv, p.nslots,
                lin ? lp.nchunks : -1, m.S);
    if (lin) {
        line(p.slot_basic);
        line(m.map);
        line(lp.chunk_s0);
        line(lp.chunk_scalar);
        line(lp.slot_mask);
        line(lp.slot_L);
        table(lp.fwd_level_step, lp.fwd_steps);
        table(lp.level_step, lp.steps);
    }
    std::vector<int> degrees;
    for (int nu : {3, 6, 8})
        if (nu >= p.numax_all)
            degrees.push_back(nu);
    std::printf("%zu\n", degrees.size());
    for (int nu : degrees) {
        std::vector<unsigned short> tab;
        std::vector<unsigned> shift;
        unsigned groups;
        mtpx::moment_table(m, p, nu, tab, shift, groups);
        std::printf("%d %zu %u\n", nu, tab.size() / mtpx::kWave, groups);
        line(tab);
        line(shift);
    }
    return 0;
}
