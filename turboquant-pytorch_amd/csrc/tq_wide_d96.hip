#include "tq_wide_kernel.h"

TQ_WIDE_DEFINE(96)
