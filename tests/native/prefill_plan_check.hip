// prefill_plan_check.hip -- the tile a prefill launch takes (kq_launch.h),
// for the CPU tests: it launches nothing.  Built by inferno_hip.build into
// tests/native/_build/libsdig_check.so.
#include "kq_launch.h"

extern "C" int prefill_wide_rows_of(int T, int inner, int outer, int ncu)
{
    return ihip::prefill_wide_rows(T, inner, outer, ncu);
}

extern "C" int prefill_thin_of(int T, int inner, int outer, int ncu)
{
    return ihip::prefill_thin(T, inner, outer, ncu);
}
