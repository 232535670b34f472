#include "dcn_backward_input_host.h"

namespace dcn {

#define INSTANTIATE(T, ND, S) template int backward_input_offset<T, ND, S>(const Geometry&, const S*, const S*, const S*, const S*, T*, T*, void*, size_t, hipStream_t, unsigned, bool*, Prep*);
INSTANTIATE(float, 3, Bf16) INSTANTIATE(float, 3, Fp16)

}  // namespace dcn
