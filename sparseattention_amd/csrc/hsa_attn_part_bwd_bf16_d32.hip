#include "hsa_attn_part_inst.h"
namespace hsa {
HSA_PART_FUSED_INSTANTIATE(BF16, 32)
}  // namespace hsa
