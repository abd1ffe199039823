// The launch plans' host arithmetic behind C names, for test_plans_cpu.py.
#include "attention_plan.h"

extern "C" uint32_t plan_split_first_block(uint32_t blocks, uint32_t split, uint32_t splits) {
    return hyperion::hip::split_first_block(blocks, split, splits);
}
