// Narrow scans of bf16 matrices.
#include "lbi_scan_narrow_kernel.h"

template int lbi::scan_narrow::launch_type<lbi::bf16_raw>(const void*, void*, const void*, void*, int, int, int, int, bool, const ScanPlan&,
                                               hipStream_t);
