// The launch plans' host arithmetic behind C names, for test_plans_cpu.py.
#include "attention_plan.h"
#include "gemm_plan.h"

extern "C" uint32_t plan_split_first_block(uint32_t blocks, uint32_t split, uint32_t splits) {
    return hyperion::hip::split_first_block(blocks, split, splits);
}

// One GEMM call: kernel (0 few rows, 1 the 128-row tiles, 2 the 256-row tiles), k splits (few
// rows: waves per tile) and column tiles per wave (few rows; else 0). ns: the segments' widths.
extern "C" void plan_gemm(uint32_t m, uint32_t k, uint32_t nseg, const uint32_t* ns, uint32_t dual, uint32_t cus,
                          uint32_t* out) {
    hyperion::hip::GemmShape g{m, (k + 127u) / 128u, nseg, {}, dual != 0u};
    for (uint32_t i = 0; i < nseg; ++i) g.n[i] = ns[i];
    if (hyperion::hip::few_rows(g, cus)) {
        const hyperion::hip::FewRowShape f = hyperion::hip::few_row_shape(g, cus);
        out[0] = 0u;
        out[1] = f.splits;
        out[2] = f.tiles;
        return;
    }
    const hyperion::hip::GemmChoice c = hyperion::hip::choose_gemm(g, cus);
    // (as launch_split: no empty split)
    const uint32_t per = (g.pairs + c.ksplit - 1u) / c.ksplit;
    out[0] = static_cast<uint32_t>(c.kernel);
    out[1] = (g.pairs + per - 1u) / per;
    out[2] = 0u;
}
