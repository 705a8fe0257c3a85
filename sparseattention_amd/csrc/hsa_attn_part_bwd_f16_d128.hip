#include "hsa_attn_part_inst.h"
namespace hsa {
HSA_PART_FUSED_INSTANTIATE(F16, 128)
}  // namespace hsa
