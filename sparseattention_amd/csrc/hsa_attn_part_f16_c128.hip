#include "hsa_attn_part_inst.h"
namespace hsa {
HSA_PART_INSTANTIATE(F16, 128, 128)
}  // namespace hsa
