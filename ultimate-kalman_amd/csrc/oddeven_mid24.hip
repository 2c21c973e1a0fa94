/*
 * oddeven_mid24.hip -- elimination phases for n = 21 .. 24 (see
 * oddeven_mid.h; a translation unit of its own so that the kernels compile in parallel).
 */
#include "oddeven_mid.h"

UKMID_DEFINE(6)
