// Prints the split size, units and partial slots that the step packer chooses for
// each step of STEPS_FILE (the format of step_plan_fuzz.cpp): first "fresh" lines,
// a planner of its own for every step, then "shared" lines, one planner for all of
// them in order, twice over.
#include <cstdio>
#include <cstdlib>
#include <vector>

#include "gsp_step_plan.h"

int main(int argc, char** argv) {
    if (argc < 2) return 2;
    FILE* f = std::fopen(argv[1], "rb");
    if (!f) return 2;
    auto rd = [&](std::vector<int32_t>& v, size_t n) {
        v.resize(n);
        return n == 0 || std::fread(v.data(), sizeof(int32_t), n, f) == n;
    };
    struct Step {
        std::vector<int32_t> h, positions, q_lens, token_counts, offsets, ids;
    };
    std::vector<int32_t> head;
    if (!rd(head, 2) || head[0] != 0x53505347) return 2;
    std::vector<Step> steps((size_t)head[1]);
    for (Step& s : steps) {
        if (!rd(s.h, 11)) return 2;
        const size_t b = (size_t)s.h[6];
        if (!rd(s.positions, b) || (s.h[8] && !rd(s.q_lens, b)) || !rd(s.token_counts, b) || !rd(s.offsets, b + 1) ||
            !rd(s.ids, (size_t)s.h[9]))
            return 2;
    }
    std::fclose(f);
    gsp::PlanOptions opt;
    opt.num_cus = 256;
    auto plan = [&](gsp::StepPlanner& p, const Step& s, const char* kind, size_t i) {
        gsp::PlanPool pool;
        pool.total_blocks = s.h[0];
        pool.heads_kv = s.h[1];
        pool.head_dim = s.h[2];
        pool.v_head_dim = s.h[3];
        pool.block_size = s.h[4];
        pool.kv_dtype = s.h[5];
        pool.layers = s.h[10];
        gsp_step_desc d{};
        d.num_rows = s.h[6];
        d.positions = s.positions.data();
        d.q_lens = s.h[8] ? s.q_lens.data() : nullptr;
        d.token_counts = s.token_counts.data();
        d.bt_offsets = s.offsets.data();
        d.bt_ids = s.ids.data();
        d.n_bt_ids = (int32_t)s.ids.size();
        d.max_seq_len = s.h[7];
        gsp::StepPlan out;
        const int rc = p.plan(pool, &d, opt, out);
        std::printf("%s %zu %d %d %d %lld\n", kind, i, rc, out.target, out.num_units, (long long)out.num_slots);
    };
    for (size_t i = 0; i < steps.size(); ++i) {
        gsp::StepPlanner p;
        plan(p, steps[i], "fresh", i);
    }
    gsp::StepPlanner shared;
    for (int pass = 0; pass < 2; ++pass)
        for (size_t i = 0; i < steps.size(); ++i) plan(shared, steps[i], "shared", i);
    return 0;
}
