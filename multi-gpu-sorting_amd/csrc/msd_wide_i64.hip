// Three-pass path of i64 keys (msd_wide_kernels.hpp).
#include "msd_wide_kernels.hpp"

namespace mgs {

template int wide_launch<MGS_KEY_I64, MGS_VAL_NONE>(const void*, void*, void*, const void*, void*, void*, size_t, char*,
                                                 const WideLayout&, uint32_t*, uint32_t, hipStream_t, Marks&);
template int wide_launch<MGS_KEY_I64, MGS_VAL_U32>(const void*, void*, void*, const void*, void*, void*, size_t, char*,
                                                 const WideLayout&, uint32_t*, uint32_t, hipStream_t, Marks&);
template int wide_launch<MGS_KEY_I64, MGS_VAL_U64>(const void*, void*, void*, const void*, void*, void*, size_t, char*,
                                                 const WideLayout&, uint32_t*, uint32_t, hipStream_t, Marks&);

}  // namespace mgs
