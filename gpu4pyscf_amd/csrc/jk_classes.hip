// Instantiates the class kernels of one part of the angular-class list;
// compiled once per part (-DJK_PART=0..7) so that the parts build in
// parallel.  Parts: 0 = li <= 1, 1 to 3 = li 2 by lj, 4 to 7 = li 3 by lj.
#include "jk_class_kernels.h"

#ifndef JK_PART
#error "JK_PART must be defined (0..7)"
#endif

static constexpr bool in_part(int li, int lj)
{
    return JK_PART == (li <= 1 ? 0 : li == 2 ? 1 + lj : 4 + lj);
}

template <int I, int J, int K, int L>
static const ClassInfo *info_if_in_part()
{
    if constexpr (in_part(I, J)) return class_info<I, J, K, L>();
    else return nullptr;
}

#define JK_CASE(I, J, K, L) \
    case ((I)*125 + (J)*25 + (K)*5 + (L)): return info_if_in_part<I, J, K, L>();

#define JK_CASE_TYPE const ClassInfo *
#include "jk_dispatch.inc"

#define JK_CAT2(a, b) a##b
#define JK_CAT(a, b) JK_CAT2(a, b)

const ClassInfo *JK_CAT(jk_class_info_part, JK_PART)(int key)
{
    return dispatch_class(key);
}
