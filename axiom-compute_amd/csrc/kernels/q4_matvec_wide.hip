// The one-pass matvec kernels for workgroups of 9 to 12 waves: the entry points
// of q4_matvec.hip under the same names, in a code object of their own (see
// kOnePassWide there for why).
#define AXH_WIDE_ONE_PASS
#include "q4_matvec.hip"
