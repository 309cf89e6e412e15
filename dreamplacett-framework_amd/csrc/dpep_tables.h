// dpep_tables.h -- the twiddle tables' device function, shared by the kernel a
// context builds its tables with (dpep_spectral.hip) and the no-alloc entry
// point's opening kernel (dpep_noalloc.hip): both get bitwise the same tables.
#pragma once

#include <hip/hip_runtime.h>

namespace dpep {

// Entry i of the tables of a length-L transform (twiddle_elems, post_elems).
template <typename T>
__device__ __forceinline__ void table_entry(int L, int i, T* __restrict__ tw,
                                            T* __restrict__ post)
{
    double s, c;
    if (i < L) {
        sincospi(2.0 * (double)i / (double)L, &s, &c);
        tw[2 * i] = (T)c;
        tw[2 * i + 1] = (T)-s;
    }
    if (i <= L / 2) {
        sincospi((double)i / (2.0 * (double)L), &s, &c);
        post[2 * i] = (T)c;
        post[2 * i + 1] = (T)-s;
    }
}

}  // namespace dpep
