// Device utilities shared by the libtgx translation units.
#pragma once
#include "tgx_internal.h"

// Zero two device ranges (bytes, multiples of four) in one launch.
int tgx_zero2(tgx_ctx* ctx, void* p, size_t np, void* q, size_t nq);

// Exclusive prefix sum of n int32 values into int64 offsets; out has n + 1
// entries (out[n] is the total). total, when not NULL, is pinned host memory
// that the scan's kernel stores the total into (valid once the stream has been
// synchronised; a copy of its own costs a launch and its gap). The block totals
// go to tmp, or to the context's own scratch when tmp is NULL; scans that may
// run on different streams at once must each bring their own.
int tgx_scan_i32(tgx_ctx* ctx, const int* in, int64_t* out, int64_t n, int64_t* total, dbuf* tmp = nullptr);
// The same for several arrays of n values at once (one launch for all of them up
// to 8,192 values, two up to 65,536, three each above).
constexpr int TGX_SCAN_TASKS = 16;
constexpr int TGX_SCAN_BLOCK = 1024;  // values whose total is one word of tmp
// Words of tmp that the scan of one array of n values uses, whatever its launches.
constexpr int64_t tgx_scan_tmp_words(int64_t n) { return (n + TGX_SCAN_BLOCK - 1) / TGX_SCAN_BLOCK + 2; }
struct tgx_scan_task {
  const int* in;
  int64_t* out;
  int64_t* tot;
};
struct tgx_scan_tasks {
  tgx_scan_task t[TGX_SCAN_TASKS];
};
int tgx_scan_many(tgx_ctx* ctx, const tgx_scan_tasks& ts, int count, int64_t n, dbuf* tmp);

// Partial sums of n doubles into TGX_SUM_PARTS device values, each over a fixed
// contiguous slice in a fixed tree (summed on the host in order).
constexpr int TGX_SUM_PARTS = 256;
int tgx_device_sum_launch(tgx_ctx* ctx, const double* d_x, int64_t n, double* d_part);

// Streaming device-to-device copy of `bytes` (a multiple of 16) by k_hbm_copy.
int tgx_hbm_copy(tgx_ctx* ctx, const void* src, void* dst, size_t bytes);
