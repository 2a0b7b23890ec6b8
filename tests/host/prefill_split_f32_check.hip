// prefill_split_check.h with the settings of the fp32 kernel, two and three
// workgroups per compute unit.
#include "prefill_f32.hip"

#include "prefill_split_check.h"

int main() {
  return SplitCheck<clv::SplitCfg>().run(clv::kRows, 512, 10000) |
         SplitCheck<clv::SplitCfg>().run(clv::kRows, 768, 10000);
}
