// msm_combine (snarkrs_amd/csrc/runtime_impl.h) with the helper pool in this file's hands, for
// tests/test_msm_combine.py: rows k G of known k, combined while the pool
//   run    starts a thread per task,
//   late   starts none until the results are there and the rows are gone,
//   throw  refuses every task.
// Prints "ok" when every sum is the point it should be.
#include <cstdio>
#include <cstring>
#include <random>

#include "../../snarkrs_amd/csrc/runtime_impl.h"

using namespace g16;

static const char* mode;
static std::mutex tasks_mu;
static std::vector<std::function<void()>> tasks;
static std::vector<std::thread> threads;

namespace g16 {
void hip_check(hipError_t, const char*) {}
void set_last_error(const std::string&) {}
void msm_reduce_shape(const MsmPlan& p, int* rows, int* lg) {
  *lg = 2;
  *rows = p.c - 2;  // 2^(c - 1) buckets in groups of 4: one row and one per bit of the group
}
void host_pool_run(std::function<void()> fn) {
  if (!std::strcmp(mode, "throw")) throw std::bad_alloc();
  std::lock_guard<std::mutex> lk(tasks_mu);
  if (!std::strcmp(mode, "run")) threads.emplace_back(std::move(fn));
  else tasks.push_back(std::move(fn));
}
}  // namespace g16

static Xyzz<Fq> to_row(const Xyzz<Fq>& p) {  // the kernels' form (R' = 2^261)
  const auto q = hx::in(p);
  return hx::out<Fq>({hx::to_msm_form(q.X), hx::to_msm_form(q.Y), hx::to_msm_form(q.ZZ),
                      hx::to_msm_form(q.ZZZ)});
}

int main(int, char** argv) {
  mode = argv[1];
  std::mt19937_64 rng(3);
  Aff<Fq> g;
  g.x = fp_one<FqCfg>();
  g.y = add(g.x, g.x);  // (1, 2)
  const Xyzz<Fq> G = xyzz_from_aff(g);
  int bad = 0;
  for (int rep = 0; rep < 20; ++rep) {
    MsmPlan p;
    p.c = rep & 1 ? 8 : 5;
    p.windows = rep & 1 ? 9 : 16;
    p.merged = false;
    const int W = msm_bucket_sets(p);
    int rows, lg;
    msm_reduce_shape(p, &rows, &lg);
    std::vector<Xyzz<Fq>> at((size_t)W * rows);
    // sum over w, j of 2^e k, e = c w, or c w + lg + j - 1 past row 0; k small enough for 256 bits
    uint32_t want[8] = {};
    const auto add_shifted = [&](uint64_t k, int e) {
      for (int b = 0; b < 16; ++b)
        if (k >> b & 1) {
          uint64_t c = 1ull << ((e + b) & 31);
          for (int i = (e + b) >> 5; i < 8 && c; ++i) {
            c += want[i];
            want[i] = (uint32_t)c;
            c >>= 32;
          }
        }
    };
    for (int w = 0; w < W; ++w)
      for (int j = 0; j < rows; ++j) {
        const uint32_t k[8] = {(uint32_t)(rng() & 0xffff)};
        at[(size_t)w * rows + j] = to_row(host_mul(G, k));
        add_shifted(k[0], p.c * w + (j ? lg + j - 1 : 0));
      }
    const Aff<Fq> ref = host_to_aff(host_mul(G, want));
    std::atomic<int> wrong{0};
    const auto call = [&] {
      const Aff<Fq> got = host_to_aff(msm_combine(at.data(), p, 1 + rep % 3));
      wrong += std::memcmp(&got, &ref, sizeof got) != 0;
    };
    std::vector<std::thread> callers;
    for (int k = 0; k < 8; ++k) callers.emplace_back(call);
    for (auto& t : callers) t.join();
    bad += wrong.load() + (tasks.size() > 8u * (1 + rep % 3));
    at = std::vector<Xyzz<Fq>>();  // a helper that starts now must not need the rows
    for (auto& t : tasks) t();
    tasks.clear();
    for (auto& t : threads) t.join();
    threads.clear();
  }
  std::printf(bad ? "%d wrong\n" : "ok\n", bad);
  return bad != 0;
}
