#include "dcn_forward_host.h"

namespace dcn {

#define INSTANTIATE(T, ND, S) template int forward<T, ND, S>(const Geometry&, const S*, const S*, const S*, const S*, S*, void*, size_t, hipStream_t, bool*, bool);
INSTANTIATE(float, 2, Bf16) INSTANTIATE(float, 3, Bf16) INSTANTIATE(float, 2, Fp16) INSTANTIATE(float, 3, Fp16)

}  // namespace dcn
