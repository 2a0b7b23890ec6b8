// prefill_split_check.h with the settings of the 16-bit kernel.
#include "prefill_mfma.hip"

#include "prefill_split_check.h"

int main() { return SplitCheck<clv::SplitCfg>().run(clv::kRows, 256, 20000); }
