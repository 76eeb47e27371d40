// gd_rules.h -- bounds that the kernels test, as functions which the CPU tests call
// too.
#pragma once
#include "gd_rng.h"

// The offset of any lane in n rows of Rp floats each fits 32 bits, in bytes.
GD_HD bool gd_rows_fit(int n, int Rp) { return (uint64_t)n * (uint64_t)Rp <= (1ull << 30); }

// Queue entries [at, at + n) of the stepping kernel lie in a queue of `limit`.  `at`
// is a difference of two counters that run on from launch to launch: after a
// launch that failed it can be negative (the launch queued fewer entries than the
// host has counted), which here is a number close to 2^32.
GD_HD bool gd_queue_room(uint32_t at, uint32_t n, uint32_t limit) { return at < limit && n <= limit - at; }
