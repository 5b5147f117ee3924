// Internals shared by the translation units of libdqcrt.so (not installed).
#pragma once

#include <hip/hip_runtime.h>

#include "dogqc_amd.h"

namespace dqcrt {

// Record a message for dqc_last_error() on this thread and return `code`.
int fail(int code, const char* fmt, ...);
int hipFail(hipError_t e, const char* what);

// A loaded plan module: its three C-ABI entry points.
struct Module {
    void* handle;
    const char* (*describe)(void);
    int (*layout)(const dqc_plan_inputs*, const dqc_plan_tuning*, dqc_plan_layout*);
    int (*enqueue)(const dqc_plan_inputs*, const dqc_plan_tuning*, void*, uint64_t, void*, void* const*);
};

// After a run: enlarge in `tun` every table the status reports too small
// (hash tables grow fourfold, since the number of keys that did not fit is
// unknown; multimaps, temp tables, long-list queues and the result get
// their exact counts).  Returns true when the run has to be repeated.
bool adjustForRetry(const dqc_plan_layout& L, const dqc_plan_status& st, dqc_plan_tuning* tun);

// The plan's layout, within `limit` bytes if it can be: a workspace too large
// does without the memory that the plan takes only to be faster when the
// tuning leaves the choice to it (the record segments of partitioned
// group-bys, then join filters: part_agg and join_filter 0, set to -1 here).
// The caller looks whether L->ws_bytes fits.
int layoutWithin(const Module* m, const dqc_plan_inputs* in, dqc_plan_tuning* tun, uint64_t limit,
                 dqc_plan_layout* L);

// Sets the two fields layoutWithin may have changed back, so that a caller's
// tuning keeps what it asked for.
struct KeepChoices {
    dqc_plan_tuning* tun;
    int32_t part_agg, join_filter;
    explicit KeepChoices(dqc_plan_tuning* t) : tun(t), part_agg(t->part_agg), join_filter(t->join_filter) {}
    ~KeepChoices() { tun->part_agg = part_agg; tun->join_filter = join_filter; }
};

// Workspaces of dqc_query_run.  A workspace handed out is an allocation of
// its own (hipMalloc); one that is released waits here for the next run that
// fits it, because allocating and freeing costs more than most plans: 0.3 ms
// for 100 MB and more, and 8 ms where the process holds gigabytes (a TPC-H Q18
// call at SF1 9.0 ms, 0.34 ms with waiting workspaces).
//   * bounded: at most 2 GiB and 16 blocks wait, the oldest are freed first;
//     a larger workspace is freed at once; a run takes no block of more than
//     twice its size and 4 MB, so a small result that is kept holds no large one;
//   * given back: blocks no run has asked for in 256 acquisitions are freed,
//     all when an allocation of this library fails, when the last plan
//     module is unloaded and when the program asks (dqc_workspace_trim), for
//     instance before another allocator of the process needs the memory;
//   * released like hipFree: the device's pending work is waited for, so work
//     on any stream that still reads the results has ended before the memory
//     is handed out again;
//   * safe with several threads (a lock around the list) and devices (a block
//     goes only to runs on its own device).
int wsAcquire(void** ptr, uint64_t bytes);
int wsRelease(void* ptr);
void wsTrim();
void wsForget(void* ptr);

}  // namespace dqcrt

#define HIP_CHECK(expr, what)                                      \
    do {                                                           \
        hipError_t _e = (expr);                                    \
        if (_e != hipSuccess) return dqcrt::hipFail(_e, what);     \
    } while (0)
