// gemv_plan_check.hip -- the kernel a GEMV launch takes (kq_gemv_plan.h), for
// the CPU tests: it launches nothing.  Built by inferno_hip.build into
// tests/native/_build/libsdig_check.so.
#include "kq_gemv_plan.h"

extern "C" int norm_takes_wide_of(int type, int nblk, int outer, int ncu)
{
    return ihip::norm_takes_wide(type, nblk, outer, ncu);
}
