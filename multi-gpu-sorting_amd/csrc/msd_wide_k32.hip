// Three-pass path of 4-byte keys with payloads (msd_wide_kernels.hpp).
#include "msd_wide_kernels.hpp"

namespace mgs {

template int wide_launch<MGS_KEY_U32, MGS_VAL_U32>(const void*, void*, void*, const void*, void*, void*, size_t, char*,
                                                 const WideLayout&, uint32_t*, uint32_t, hipStream_t, Marks&);
template int wide_launch<MGS_KEY_U32, MGS_VAL_U64>(const void*, void*, void*, const void*, void*, void*, size_t, char*,
                                                 const WideLayout&, uint32_t*, uint32_t, hipStream_t, Marks&);
template int wide_launch<MGS_KEY_I32, MGS_VAL_U32>(const void*, void*, void*, const void*, void*, void*, size_t, char*,
                                                 const WideLayout&, uint32_t*, uint32_t, hipStream_t, Marks&);
template int wide_launch<MGS_KEY_I32, MGS_VAL_U64>(const void*, void*, void*, const void*, void*, void*, size_t, char*,
                                                 const WideLayout&, uint32_t*, uint32_t, hipStream_t, Marks&);

}  // namespace mgs
