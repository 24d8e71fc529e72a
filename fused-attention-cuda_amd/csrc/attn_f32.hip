// attn_f32.hip -- stage 3, fp32 compute: fp32 inputs on split bf16 operands, fp16 inputs on fp32 MFMA.
#include "attn_kernel.h"
#include "attn_split32.h"

namespace fa {
VariantList variants_s3_f32() { return split32::table(); }
VariantList variants_s3_f16() { return kern::s3_table<_Float16>(); }
}  // namespace fa
