// prepare_tasks: device-built compact task table (request, query offset) per query tile.
//
// Reference: oscar_ascend/kernels.py:222-287 (`_prepare_tasks_kernel`, `prepare_tasks`).
// One workgroup per program (request). Each workgroup recomputes the exclusive prefix sum of
// tile counts of the requests before it, so no inter-workgroup communication is needed and
// the table is identical for any program execution order.
//
// prepare_step: the whole per-step metadata fill (query starts, lengths, slots, counts, table
// and tasks) as one launch. Latency-bound: a few KB and one prefix sum, so its cost is the
// launches: one kernel that reads the scheduler's tensors itself (4 us) in place of five copies
// and fills and the task kernel makes a step 7 to 10 us shorter (four layers of one 700-token
// request 118 -> 110 us, of 117 ragged requests 196 -> 186 us).
#include "common.h"

namespace oscar {
namespace {

struct TaskArgs {
  const int32_t* qstarts;  // step form: the scheduler's
  const int32_t* counts;   // step form: unused (reqs, active)
  int32_t* tasks;
  int32_t* task_count;
  int64_t capacity;
  int32_t limit;  // requests that may contribute: min(next_pow2(max_reqs), max_reqs)
  int32_t query_tile;
  const int32_t* source;
  int64_t source_stride;
  int32_t* table;
  int64_t table_stride;
  int64_t copy_columns;
  // Step form: the counts (host values) and the sources and destinations of the copies.
  int32_t reqs, active;
  const int32_t* seq_lens;
  const int64_t* slots;
  int32_t* qstarts_out;
  int32_t* seq_lens_out;
  int64_t* slots_out;
  int32_t* counts_out;
};

// Slots one workgroup of the step form copies.
constexpr int kStepSlots = 4 * kThreads;

__device__ __forceinline__ int tiles_of(const TaskArgs& a, int r, int active) {
  const int start = min(a.qstarts[r], active);
  const int end = min(a.qstarts[r + 1], active);
  return cdiv(max(end - start, 0), a.query_tile);
}

template <bool kStep>
__global__ __launch_bounds__(kThreads) void prepare_tasks_kernel(const TaskArgs a) {
  __shared__ int s_before[kThreads / kWave], s_all[kThreads / kWave];
  const int req = blockIdx.x;
  const int nr = kStep ? a.reqs : a.counts[0], active = kStep ? a.active : a.counts[1];
  if constexpr (kStep) {
    // Workgroup b copies slots [b kStepSlots, ...); the first one also the per-request rows.
#pragma unroll
    for (int k = 0; k < kStepSlots / kThreads; ++k) {
      const int64_t i = static_cast<int64_t>(req) * kStepSlots + k * kThreads + threadIdx.x;
      if (i < active) a.slots_out[i] = a.slots[i];
    }
    if (req == 0) {
      for (int i = threadIdx.x; i <= nr; i += kThreads) {
        a.qstarts_out[i] = a.qstarts[i];
        if (i < nr) a.seq_lens_out[i] = a.seq_lens[i];
      }
      if (threadIdx.x < 2) a.counts_out[threadIdx.x] = threadIdx.x ? active : nr;
    }
  }
  if (a.source && req < min(nr, a.limit)) {
    for (int64_t c = threadIdx.x; c < a.copy_columns; c += kThreads)
      a.table[req * a.table_stride + c] = a.source[req * a.source_stride + c];
  }
  const int live = min(nr, a.limit);
  int before = 0, all = 0;
  for (int r = threadIdx.x; r < live; r += kThreads) {
    const int t = tiles_of(a, r, active);
    all += t;
    if (r < req) before += t;
  }
#pragma unroll
  for (int m = 32; m >= 1; m >>= 1) {
    before += __shfl_xor(before, m, kWave);
    all += __shfl_xor(all, m, kWave);
  }
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  if (lane == 0) {
    s_before[wave] = before;
    s_all[wave] = all;
  }
  __syncthreads();
  before = s_before[0] + s_before[1] + s_before[2] + s_before[3];
  all = s_all[0] + s_all[1] + s_all[2] + s_all[3];
  if (req == 0 && threadIdx.x == 0) a.task_count[0] = all;
  const int count = req < live ? tiles_of(a, req, active) : 0;
  for (int j = threadIdx.x; j < count; j += kThreads) {
    const int64_t idx = static_cast<int64_t>(before) + j;
    if (idx < a.capacity) {
      a.tasks[2 * idx] = req;
      a.tasks[2 * idx + 1] = j * a.query_tile;
    }
  }
}

}  // namespace
}  // namespace oscar

namespace oscar {
namespace {

// Requests that may contribute tasks: min(next_pow2(max_reqs), max_reqs).
int32_t request_limit(int64_t max_reqs) {
  int64_t lanes = 1;
  while (lanes < max_reqs) lanes <<= 1;
  return static_cast<int32_t>(lanes < max_reqs ? lanes : max_reqs);
}

}  // namespace
}  // namespace oscar

extern "C" int oscar_prepare_tasks(const int32_t* qstarts, const int32_t* counts, int32_t* tasks,
                                   int32_t* task_count, int64_t task_capacity, int64_t max_reqs,
                                   int32_t query_tile, int64_t programs,
                                   const int32_t* source_table, int64_t source_stride,
                                   int32_t* table, int64_t table_stride, int64_t copy_columns,
                                   void* stream) {
  using namespace oscar;
  if (max_reqs < 1 || query_tile < 1 || programs < 1 || task_capacity < 0 || copy_columns < 0)
    return OSCAR_E_SHAPE;
  if (!qstarts || !counts || !tasks || !task_count) return OSCAR_E_NULL;
  if (source_table && (!table || copy_columns > table_stride)) return OSCAR_E_SHAPE;
  if (max_reqs > (1ll << 30) || programs > (1ll << 30)) return OSCAR_E_SHAPE;
  TaskArgs a{};
  a.qstarts = qstarts;
  a.counts = counts;
  a.tasks = tasks;
  a.task_count = task_count;
  a.capacity = task_capacity;
  a.limit = request_limit(max_reqs);
  a.query_tile = query_tile;
  a.source = source_table;
  a.source_stride = source_stride;
  a.table = table;
  a.table_stride = table_stride;
  a.copy_columns = source_table ? copy_columns : 0;
  hipLaunchKernelGGL(prepare_tasks_kernel<false>, dim3(static_cast<unsigned>(programs)), dim3(kThreads),
                     0, as_stream(stream), a);
  return static_cast<int>(hipGetLastError());
}

extern "C" int oscar_prepare_step(const int32_t* src_qstarts, const int32_t* src_seq_lens,
                                  const int64_t* src_slots, const int32_t* src_table,
                                  int64_t src_table_stride, int64_t copy_columns,
                                  int32_t num_reqs, int32_t num_tokens, int64_t max_reqs,
                                  int64_t max_tokens, int32_t query_tile, int32_t* qstarts,
                                  int32_t* seq_lens, int64_t* slots, int32_t* table,
                                  int64_t table_stride, int32_t* counts, int32_t* tasks,
                                  int32_t* task_count, int64_t task_capacity, void* stream) {
  using namespace oscar;
  if (max_reqs < 1 || max_reqs > (1ll << 30) || query_tile < 1 || task_capacity < 0 ||
      num_reqs < 0 || num_reqs > max_reqs || num_tokens < 0 || num_tokens > max_tokens ||
      copy_columns < 0 || copy_columns > table_stride)
    return OSCAR_E_SHAPE;
  if (!src_qstarts || !src_table || !qstarts || !seq_lens || !slots || !table || !counts ||
      !tasks || !task_count || (num_reqs && !src_seq_lens) || (num_tokens && !src_slots))
    return OSCAR_E_NULL;
  TaskArgs a{};
  a.qstarts = src_qstarts;
  a.tasks = tasks;
  a.task_count = task_count;
  a.capacity = task_capacity;
  a.limit = request_limit(max_reqs);
  a.query_tile = query_tile;
  a.source = src_table;
  a.source_stride = src_table_stride;
  a.table = table;
  a.table_stride = table_stride;
  a.copy_columns = copy_columns;
  a.reqs = num_reqs;
  a.active = num_tokens;
  a.seq_lens = src_seq_lens;
  a.slots = src_slots;
  a.qstarts_out = qstarts;
  a.seq_lens_out = seq_lens;
  a.slots_out = slots;
  a.counts_out = counts;
  const int programs = max(max(num_reqs, 1), (num_tokens + kStepSlots - 1) / kStepSlots);
  hipLaunchKernelGGL(prepare_tasks_kernel<true>, dim3(static_cast<unsigned>(programs)),
                     dim3(kThreads), 0, as_stream(stream), a);
  return static_cast<int>(hipGetLastError());
}
