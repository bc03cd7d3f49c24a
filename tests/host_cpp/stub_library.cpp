// A libmograd_hip without a GPU, for tests of the host path (tests/test_graph_host.py): host memory,
// a record of the calls, and a count of the blocks that were given back to the pool while a call was
// using them.  Only ADD and RELU compute; the others note their call and fill their results.
#include <unistd.h>

#include <atomic>
#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <string>

#include "mograd_hip.h"

namespace {

struct Block {
  int64_t bytes;
  bool live;
  int users;
};
std::mutex g_lock;
std::map<uintptr_t, Block> g_blocks;  // by address; memory is never reused, so that a late read is seen
std::string g_log;
std::atomic<int> g_violations{0};
std::atomic<int> g_pause_us{0};

Block* find(const void* p) {
  auto it = g_blocks.upper_bound(reinterpret_cast<uintptr_t>(p));
  return it == g_blocks.begin() ? nullptr : &std::prev(it)->second;
}
// A call that reads or writes `n` arrays, for as long as it lives.
struct Use {
  const void* p[4];
  int n;
  Use(std::initializer_list<const void*> list) : n(0) {
    std::lock_guard<std::mutex> hold(g_lock);
    for (const void* q : list) {
      p[n++] = q;
      Block* b = find(q);
      if (!b || !b->live) ++g_violations;
      else ++b->users;
    }
  }
  ~Use() {
    if (g_pause_us) usleep(static_cast<useconds_t>(g_pause_us.load()));
    std::lock_guard<std::mutex> hold(g_lock);
    for (int i = 0; i < n; ++i)
      if (Block* b = find(p[i])) --b->users;
  }
};
int note(const std::string& line) {
  std::lock_guard<std::mutex> hold(g_lock);
  g_log += line + "\n";
  return 0;
}
void fill(void* p, float v) {
  if (p) *static_cast<float*>(p) = v;
}
std::string num(double v) { return " " + std::to_string(v); }

}  // namespace

extern "C" {

// For the tests.
void stub_reset(int pause_us) {
  std::lock_guard<std::mutex> hold(g_lock);
  g_log.clear();
  g_violations = 0;
  g_pause_us = pause_us;
}
int stub_violations() { return g_violations; }
int64_t stub_log(char* out, int64_t size) {
  std::lock_guard<std::mutex> hold(g_lock);
  if (size > 0) std::strncpy(out, g_log.c_str(), static_cast<size_t>(size));
  return static_cast<int64_t>(g_log.size());
}

const char* mg_last_error(void) { return "stub"; }
int mg_init(int) { return 0; }
int mg_stream_create(mg_stream* s) { return *s = reinterpret_cast<void*>(16), 0; }
int mg_stream_destroy(mg_stream) { return 0; }
int mg_stream_sync(mg_stream) { return 0; }
int mg_copy_to_device(void* dst, const void* src, int64_t n, mg_stream) { return std::memcpy(dst, src, n), 0; }
int mg_copy_to_host(void* dst, const void* src, int64_t n, mg_stream) { return std::memcpy(dst, src, n), 0; }
int mg_copy_device(void* dst, const void* src, int64_t n, mg_stream) { return std::memcpy(dst, src, n), 0; }
int mg_pool_alloc(void** out, int64_t n) {
  *out = std::aligned_alloc(64, static_cast<size_t>((n + 127) / 64 * 64));
  std::lock_guard<std::mutex> hold(g_lock);
  g_blocks[reinterpret_cast<uintptr_t>(*out)] = Block{n, true, 0};
  return 0;
}
int mg_pool_free(void* p) {
  std::lock_guard<std::mutex> hold(g_lock);
  Block* b = find(p);
  if (!b) return 1;
  if (b->users > 0) ++g_violations;
  b->live = false;
  return 0;
}

int mg_add(const void* a, const void* b, void* dst, int64_t n, int, mg_stream) {
  Use use{a, b, dst};
  for (int64_t i = 0; i < n; ++i) static_cast<float*>(dst)[i] = static_cast<const float*>(a)[i] + static_cast<const float*>(b)[i];
  return note("add");
}
int mg_relu(const void* a, void* dst, int64_t n, int, mg_stream) {
  Use use{a, dst};
  for (int64_t i = 0; i < n; ++i) static_cast<float*>(dst)[i] = static_cast<const float*>(a)[i] > 0 ? static_cast<const float*>(a)[i] : 0;
  return note("relu");
}
int mg_linear_bwd_fused(const void* dy, const void* x, const void* w, void* dx, void* dw, void* db, int64_t, int64_t,
                        int64_t, int, int, int, mg_stream) {
  Use use{dy, x, w};
  fill(dx, 1), fill(dw, 2), fill(db, 3);
  return note(std::string("linear_bwd") + (dx ? " dx" : "") + (dw ? " dw" : "") + (db ? " db" : ""));
}
int mg_linear_bwd(const void* dy, const void* x, const void* w, void* dx, void* dw, void* db, int64_t M, int64_t N, int64_t K,
                  int dtype, mg_stream s) {
  return mg_linear_bwd_fused(dy, x, w, dx, dw, db, M, N, K, 0, 0, dtype, s);
}
int mg_layer_norm_fwd_stats(const void*, const void*, const void*, void*, float*, float*, int64_t rows, int64_t cols,
                            float eps, int, mg_stream) {
  return note("layer_norm_stats" + num(rows) + num(cols) + num(eps));
}
int mg_layer_norm_bwd_stats(const void*, const void*, const void*, const float*, const float*, void*, void*, void*,
                            int64_t rows, int64_t cols, int, mg_stream) {
  return note("layer_norm_bwd_stats" + num(rows) + num(cols));
}
int mg_matmul_bt(const void*, const void*, void*, int64_t, int64_t M, int64_t N, int64_t K, int64_t, int64_t, int64_t,
                 int64_t, int64_t, int64_t, int, mg_stream) {
  return note("matmul_bt" + num(M) + num(N) + num(K));
}
int mg_scatter_add(const void*, const void*, void*, int64_t, int64_t rows, int64_t row_size, int, int, mg_stream) {
  return note("scatter_add" + num(rows) + num(row_size));
}
int mg_flash_attn_fwd_packed(const void*, const void*, void*, float*, int64_t, int64_t, int64_t, int64_t, float scale,
                             int causal, int bias, int, mg_stream) {
  return note("attn_packed" + num(scale) + num(causal) + num(bias));
}
int mg_flash_attn_bwd_packed(const void*, const void*, const void*, const void*, const float*, void*, int64_t, int64_t,
                             int64_t, int64_t, float scale, int causal, int bias, int, mg_stream) {
  return note("attn_packed_bwd" + num(scale) + num(causal) + num(bias));
}
int mg_cross_entropy_ids(const void*, const void*, void* loss, int64_t rows, int64_t classes, int, int id_dtype,
                         mg_stream) {
  return fill(loss, 4), note("ce_ids" + num(rows) + num(classes) + " dtype " + std::to_string(id_dtype));
}
int mg_cross_entropy_grad_ids(const void*, const void*, const void*, void* grad, int64_t rows, int64_t classes, int, int,
                              mg_stream) {
  return fill(grad, 5), note("ce_grad_ids" + num(rows) + num(classes));
}
int mg_cross_entropy_fused_ids(const void* logits, const void* ids, const void* up, void* loss, void* grad, int64_t rows,
                               int64_t classes, int, int, mg_stream) {
  Use use{logits, ids, up};
  fill(loss, 4), fill(grad, 5);
  return note("ce_fused_ids" + num(rows) + num(classes));
}

}  // extern "C"
