/*
 * dogqc_amd C ABI: the drop-in boundary of the MI355X execution backend.
 *
 * Two kinds of shared library export these symbols:
 *
 *  1. Every compiled plan module (one .so per plan, generated by the HIP
 *     translator) exports the dqc_plan_* functions.  Together they replace the
 *     per-query program the reference generates and runs as a subprocess: its
 *     main() with mmap, cudaMalloc, HT init kernels, H2D copies, the kernel
 *     launch sequence and the result print (dogqc/codegen.py:121-159, 209-218;
 *     dogqc/gpuio.py:5-58).
 *
 *  2. libdqcrt.so (the runtime) exports the dqc_* functions: HBM-resident
 *     column loading, plan-module loading, the run-with-retry driver, hipGraph
 *     capture and the serving loop.
 *
 * All pointers are plain device or host addresses; streams, events and graphs
 * are passed as opaque void* (hipStream_t / hipEvent_t / hipGraphExec_t).
 * Functions return 0 on success and a negative DQC_E* code on failure; they
 * never exit the process (the reference's ERROR macro does, util.h:2-5).
 * dqc_last_error() returns the calling thread's last message.
 */
#ifndef DOGQC_AMD_H
#define DOGQC_AMD_H

#include <stdint.h>

#ifdef __cplusplus
extern "C" {
#endif

#define DQC_MAX_PIPES 32
#define DQC_MAX_HTS 32
#define DQC_MAX_RESULT_COLS 64
#define DQC_MAX_TEMPS 8
#define DQC_MAX_STEPS 128
#define DQC_PROFILE_BUCKETS 65

enum {
    DQC_OK = 0,
    DQC_EINVAL = -1,     /* bad argument or input binding */
    DQC_EHIP = -2,       /* a HIP runtime call failed */
    DQC_EIO = -3,        /* file or mmdb format error */
    DQC_EOVERFLOW = -4,  /* a table stayed too small after all retries */
    DQC_ENOMEM = -5,     /* workspace does not fit or exceeds a budget */
    DQC_ELOAD = -6       /* plan module could not be loaded */
};

/* status word bits, first field of dqc_plan_status */
#define DQC_ST_HT_OVERFLOW 0x1u
#define DQC_ST_MM_OVERFLOW 0x2u
#define DQC_ST_RESULT_OVERFLOW 0x4u

/* ---------------------------------------------------------------------------
 * Plan module ABI
 * ------------------------------------------------------------------------- */

/* Input binding.  Tables and columns are numbered in the order listed by
 * dqc_plan_describe().  A STRING column occupies two slots (uint64 offsets
 * [rows+1], then the char heap).  Replaces the per-column map_memory_file /
 * cudaMalloc / cudaMemcpy triple of the generated main()
 * (dogqc/cudaTranslator.py:138-166; dogqc/gpuio.py:19-21). */
typedef struct dqc_plan_inputs {
    int32_t ntables;
    int32_t ncols;
    const int64_t* table_rows;
    const void* const* cols;
} dqc_plan_inputs;

/* Per-run tuning.  Zero means "plan default" everywhere.  Replaces the fixed
 * launch shape KernelCall.defaultGridSize/defaultBlockSize (kernel.py:10-11),
 * the refill threshold of LaneRefill (cudaDivergenceBuffer.py:15) and the
 * cfg htSizeFactor (relationalAlgebra.py:453-455) with per-pipeline values. */
typedef struct dqc_plan_tuning {
    int32_t grid[DQC_MAX_PIPES];             /* workgroups per pipeline kernel */
    int32_t refill_threshold[DQC_MAX_PIPES]; /* 1..64 active lanes (lane refills, push-down probes that gather) */
    int32_t lds_slots[DQC_MAX_PIPES];        /* LDS group slots (power of 2); -1 = no LDS tier */
    int32_t lds_replicas[DQC_MAX_PIPES];     /* LDS accumulator replicas (power of 2, <= 64) */
    float ht_factor[DQC_MAX_HTS];            /* multiplies htSizeFactor / the 2x agg factor */
    int64_t ht_capacity[DQC_MAX_HTS];        /* explicit slot count */
    int64_t mm_entries[DQC_MAX_HTS];         /* explicit multimap entry capacity */
    int64_t result_capacity;                 /* explicit result row capacity */
    int64_t temp_capacity[DQC_MAX_TEMPS];    /* explicit temp-table row capacities */
    int64_t split_capacity[DQC_MAX_HTS];     /* explicit capacity of a push-down join's long-list queue */
    int32_t split_threshold[DQC_MAX_PIPES];  /* matches above which a probe row's list is split (0 = 1024) */
    int32_t profile;                         /* 1 = fill lane-activity histograms */
    int32_t xcd_replicas;                    /* global group-by accumulator copies: 0 = plan default,
                                                1 = one copy, 2/4/8 = copies by workgroup index */
    int32_t census;                          /* 1 = count the occupied slots of every hash table
                                                into dqc_plan_status.ht_fill after the plan */
    int32_t part_agg;                        /* partitioned group-by (plans translated with it): 0 = when
                                                the group count (ht_capacity / 2, else the plan's numgroups)
                                                exceeds 2048 and 65536 rows or more are estimated
                                                to reach it, -1 = never, n > 0 = n partitions */
    int32_t join_filter;                     /* filter of the build keys of selective unique joins: n > 0 =
                                                n KB (in LDS when it fits), 0 = the size the plan was
                                                translated with, else 16 bits per key in device memory for
                                                a join whose lane refill gathers the rows that pass it,
                                                else none; < 0 = none */
    int32_t part_build;                      /* partitioned unique-join build (plans translated with it):
                                                n > 0 = n partitions, else none */
    int32_t reserved[2];
} dqc_plan_tuning;

/* Written by the device into the first bytes of the workspace.  Replaces the
 * device printf on a full hash table (hashing.cuh:95-97, 117-118, 266-268)
 * and the after-the-fact output size check (cudaTranslator.py:609-610).
 * result_count and temp_count[] count every appended row, also those beyond
 * the capacity, so a count above the capacity asks for a retry with exactly
 * that many rows.  A temp table's scans read its count from here. */
typedef struct dqc_plan_status {
    uint32_t flags;
    uint32_t ht_overflow_mask;
    uint32_t mm_overflow_mask;
    uint32_t reserved;
    uint64_t result_count;
    uint64_t mm_total[DQC_MAX_HTS];
    uint64_t temp_count[DQC_MAX_TEMPS];
    uint64_t split_count[DQC_MAX_HTS];   /* probe rows queued as long match lists, per push-down join */
    uint64_t ht_fill[DQC_MAX_HTS];       /* occupied slots of each unique-join / group-by table
                                            (with tuning.census; the keys a table really holds) */
} dqc_plan_status;

typedef struct dqc_plan_layout {
    uint64_t ws_bytes;
    int32_t nsteps;                   /* kernel launches per enqueue */
    int32_t nhts;
    int64_t ht_capacity[DQC_MAX_HTS];
    int64_t mm_entries[DQC_MAX_HTS];
    int64_t result_capacity;
    int32_t nresult;
    int32_t nprofile;                 /* lane-activity histograms */
    uint64_t result_offset[DQC_MAX_RESULT_COLS];
    uint64_t profile_offset;          /* nprofile x DQC_PROFILE_BUCKETS uint64 counters */
    int32_t ntemps;                   /* temp tables (createtemp), in describe() order */
    int32_t ntempcols;
    int64_t temp_capacity[DQC_MAX_TEMPS];
    uint64_t temp_offset[DQC_MAX_RESULT_COLS]; /* columns of all temp tables, in describe() order */
    int64_t split_capacity[DQC_MAX_HTS];  /* long-list queue capacity per push-down join (0 = none) */
} dqc_plan_layout;

/* JSON description of the module: tables, column slots, result schema,
 * pipelines and launch steps.  Replaces reading the generated source. */
const char* dqc_plan_describe(void);

/* Workspace size, table capacities and result placement for given inputs. */
int dqc_plan_layout_of(const dqc_plan_inputs* in, const dqc_plan_tuning* tun, dqc_plan_layout* out);

/* Enqueue every kernel of the plan on `stream` (asynchronous, no allocation,
 * no host synchronisation, so it can be captured into a hipGraph).  The
 * workspace (at least 16-byte aligned, as hipMalloc's 256 bytes are; else
 * DQC_EINVAL) is initialised by the plan's own init kernel.  If step_events is
 * not NULL it must hold nsteps+1 events, recorded before each launch and
 * after the last.  Replaces the launch sequence of the generated main()
 * (codegen.py:143-146). */
int dqc_plan_enqueue(const dqc_plan_inputs* in, const dqc_plan_tuning* tun, void* ws, uint64_t ws_bytes,
                     void* stream, void* const* step_events);

/* ---------------------------------------------------------------------------
 * Runtime (libdqcrt.so)
 * ------------------------------------------------------------------------- */

const char* dqc_last_error(void);

/* Select the device and report its compute units and memory. */
int dqc_device_init(int device, int32_t* compute_units, uint64_t* hbm_bytes);
int dqc_malloc(void** ptr, uint64_t bytes);
int dqc_free(void* ptr);
int dqc_memcpy_h2d(void* dst, const void* src, uint64_t bytes);
int dqc_memcpy_d2h(void* dst, const void* src, uint64_t bytes);
int dqc_memset(void* dst, int value, uint64_t bytes);
int dqc_stream_create(void** stream);
int dqc_stream_destroy(void* stream);
int dqc_stream_sync(void* stream);
int dqc_event_create(void** event);
int dqc_event_destroy(void* event);
int dqc_event_elapsed_ms(void* start, void* stop, float* ms);
int dqc_event_record(void* event, void* stream);

/* Load the payload of one mmdb column file into a new device allocation
 * (the reader of mappedmalloc.h:69-82 plus the H2D copy of gpuio.py:19-21).
 * *bytes receives the payload size. */
int dqc_mmdb_load(const char* path, void** dptr, uint64_t* bytes);

/* Plan modules (replaces CodeGenerator.execute, codegen.py:209-218). */
int dqc_module_load(const char* so_path, void** module);
int dqc_module_unload(void* module);
const char* dqc_module_describe(void* module);
int dqc_query_layout(void* module, const dqc_plan_inputs* in, const dqc_plan_tuning* tun, dqc_plan_layout* out);
int dqc_query_enqueue(void* module, const dqc_plan_inputs* in, const dqc_plan_tuning* tun, void* ws,
                      uint64_t ws_bytes, void* stream, void* const* step_events);

typedef struct dqc_query_result {
    void* ws;                   /* device workspace holding the result columns */
    uint64_t ws_bytes;
    dqc_plan_layout layout;
    dqc_plan_status status;
    int32_t retries;
} dqc_query_result;

/* Run a plan to completion on `stream`: allocate the workspace (or take a
 * released one, of at most twice the size and 4 MB), enqueue, synchronise, and on a full hash table, multimap, temp table or result buffer enlarge
 * it (tuning is updated in place) and run again, up to max_retries times. */
int dqc_query_run(void* module, const dqc_plan_inputs* in, dqc_plan_tuning* tun, void* stream,
                  int32_t max_retries, dqc_query_result* res);
/* Give a result's workspace back.  Up to 2 GiB of released workspaces wait in
 * the library for later runs; dqc_workspace_trim frees them all. */
int dqc_query_release(dqc_query_result* res);
int dqc_workspace_trim(void);

/* Workspace size of dqc_query_run_noalloc: a static device array compiled
 * into libdqcrt.so, one copy per GPU the library runs on, held until the
 * process ends. */
#define DQC_NOALLOC_WS_BYTES (64ull << 20)

/* dqc_query_run without any allocation.  No counterpart in the reference:
 * it is for callers that cannot allocate device memory (code under stream
 * capture, tight serving loops, hosts that forbid hipMalloc).  The plan runs
 * in the library's static workspace; a plan whose workspace (the layout's
 * ws_bytes) exceeds DQC_NOALLOC_WS_BYTES, also after a retry enlarged its
 * tables, runs without the memory it takes only to be faster (what part_agg
 * and join_filter left at 0 let it choose) and is rejected with DQC_ENOMEM
 * if that is not enough.  The caller passes one device buffer
 * per result column (out_cols, in describe() order, each holding out_rows
 * rows of its column's type); the result rows are copied there and a result
 * of more than out_rows rows fails with DQC_EOVERFLOW.  res receives the
 * layout, status and retry count; res->ws stays NULL (nothing to release).
 * Calls on one GPU share the workspace: they are serialised by a lock, and
 * the call returns after its stream has finished.  No hipMalloc, hipFree or
 * allocating library routine is called. */
int dqc_query_run_noalloc(void* module, const dqc_plan_inputs* in, dqc_plan_tuning* tun, void* stream,
                          int32_t max_retries, void* const* out_cols, int64_t out_rows, dqc_query_result* res);

/* Capture one dqc_plan_enqueue into an executable hipGraph. */
int dqc_graph_create(void* module, const dqc_plan_inputs* in, const dqc_plan_tuning* tun, void* ws,
                     uint64_t ws_bytes, void* stream, void** graph_exec);
int dqc_graph_launch(void* graph_exec, void* stream);
int dqc_graph_destroy(void* graph_exec);

/* ---------------------------------------------------------------------------
 * Serving loop: continuous batching of plan runs on one GPU (no counterpart
 * in the reference, which runs one query per process, codegen.py:209-218).
 *
 * Queries are submitted with an arrival time; a scheduler thread admits a
 * query once it has arrived, one of `slots` HIP streams is free and its
 * workspace (hash tables, multimaps, temp tables, result: the layout's
 * ws_bytes) fits the device arena, then enqueues the plan and its status
 * readback on that stream.  Finished queries free their slot and arena
 * space for the next arrivals while the others keep running, so the work
 * of different queries overlaps on the device.  Heavy queries (large
 * workspaces, which go with large inputs) can be limited to a few at a time
 * so they do not slow each other down by competing for caches and
 * bandwidth, while light queries overlap with them; a slot is kept free for
 * a waiting heavy query.  A query whose tables
 * overflowed is re-admitted with enlarged tables.  slots = 1 gives the
 * one-query-at-a-time baseline.  Input columns are shared, read-only and
 * resident in HBM for the server's lifetime.
 * ------------------------------------------------------------------------- */
typedef struct dqc_serve_config {
    int32_t slots;            /* concurrent queries (HIP streams, default priority), 1..64 */
    int32_t max_retries;      /* per query, on a full table */
    uint64_t arena_bytes;     /* device memory for query workspaces: the admission budget */
    int32_t bypass_ms;        /* later arrivals may pass a query waiting for memory this long (0 = strict FIFO) */
    int32_t size_feedback;    /* 1: size tables from what earlier queries of the same module needed */
    int32_t max_heavy;        /* queries with a workspace of heavy_bytes or more run at most this many at once */
    uint64_t heavy_bytes;     /* (0 = no limit); lighter queries fill the other slots */
    int32_t max_batch;        /* up to this many waiting queries with the same batched plan run as
                                 one batch (<= 1: never; at most DQC_SERVE_MAX_BATCH) */
    int32_t batch_ratio;      /* a waiting query joins the first waiting query's batch only if their
                                 driving row counts are within this factor (<= 0: any size); a batch
                                 takes as long as its largest member, so a much smaller query is
                                 better run on its own */
    double batch_min_share;   /* a batch runs only while its members other than the largest hold at
                                 least this share of the largest's driving rows; otherwise the
                                 largest leaves the batch and runs on its own (<= 0: no such rule).
                                 A batch costs more than its largest member alone, and a large
                                 query batched with little else pays that for almost nothing */
} dqc_serve_config;

#define DQC_SERVE_MAX_BATCH 32

typedef struct dqc_serve_request {
    void* module;                   /* from dqc_module_load */
    dqc_plan_inputs inputs;         /* copied at submit; the column memory must stay valid */
    const dqc_plan_tuning* tuning;  /* copied at submit; NULL = plan defaults */
    int64_t arrival_ns;             /* arrival, as an offset from dqc_serve_start */
    int32_t keep_result;            /* 1: keep the workspace (the result) until dqc_serve_release */
    /* Optional batched plan of the same query: queries with the same module
     * and batch_module may run as one batch that scans their largest
     * prefixes once (members ordered by growing prefixes).  The batched
     * module reads, for each of its tables j, batch_table_map[j] >= 0: the
     * largest member's row count of this module's table batch_table_map[j];
     * -1: its `__batch` table (one row per member).  For each of its columns
     * c, batch_col_prefix[c] = -1: the pointer batch_cols[c]; j >= 0: the
     * members' row counts of its table j (int64 per member, filled by the
     * server). */
    int32_t batch_ntables;
    void* batch_module;
    const void* const* batch_cols;
    const int32_t* batch_col_prefix;
    const int32_t* batch_table_map;
    int32_t batch_ncols;
    int32_t reserved;
} dqc_serve_request;

enum { DQC_SERVE_PENDING = 0, DQC_SERVE_RUNNING = 1, DQC_SERVE_DONE = 2, DQC_SERVE_FAILED = 3 };

typedef struct dqc_serve_record {
    int64_t arrival_ns;   /* offsets from dqc_serve_start */
    int64_t admit_ns;     /* last (re)admission */
    int64_t done_ns;      /* the run finished and its status reached the host */
    int32_t state;        /* DQC_SERVE_* */
    int32_t retries;
    int32_t error;        /* DQC_E* code when failed */
    int32_t slot;
    void* ws;             /* workspace holding the result (keep_result), else NULL once done */
    uint64_t ws_bytes;
    int32_t batch_size;   /* > 1: ran in a batch of this many queries; ws, layout and status are the
                             batch's (of the batched module), shared by its members */
    int32_t batch_index;  /* this query's member index in the batch (members by growing prefixes) */
    dqc_plan_layout layout;
    dqc_plan_status status;
} dqc_serve_record;

int dqc_serve_create(const dqc_serve_config* cfg, void** server);
/* Thread-safe; allowed before and after dqc_serve_start. */
int dqc_serve_submit(void* server, const dqc_serve_request* req, int64_t* id);
/* Start the clock and the scheduler thread. */
int dqc_serve_start(void* server);
/* Block until every submitted query is done or failed (timeout_ms < 0: no limit). */
int dqc_serve_wait(void* server, int64_t timeout_ms);
int dqc_serve_record_of(void* server, int64_t id, dqc_serve_record* out);
/* Return a kept workspace to the arena. */
int dqc_serve_release(void* server, int64_t id);
/* Wait for running queries, stop the scheduler, free streams, arena and records. */
int dqc_serve_destroy(void* server);

#ifdef __cplusplus
}
#endif
#endif
