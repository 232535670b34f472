#include "dcn_backward_input_host.h"

namespace dcn {

#define INSTANTIATE(T, ND, S) template int backward_input_offset<T, ND, S>(const Geometry&, const S*, const S*, const S*, const S*, T*, T*, void*, size_t, hipStream_t, unsigned, bool*, Prep*);
INSTANTIATE(float, 3, float)

}  // namespace dcn
