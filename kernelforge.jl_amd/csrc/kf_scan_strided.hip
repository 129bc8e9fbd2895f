// The strided scans (a strided source, or a destination that takes no whole
// vectors): the kernels of kf_scan.hip with STRIDED, in an object of their
// own so that both halves compile in parallel (1.6 minutes each; 4.3 as one).
#define KF_SCAN_STRIDED 1
#include "kf_scan.hip"
