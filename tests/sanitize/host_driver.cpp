// Exercises the library's host-only code -- the CPU Crout (lucore_cpu.cpp),
// RunInfo (run_info.cpp), the shape-table reader (lufqhe_table.cpp) and the
// pool of kept server buffers (kept_pool.hpp) --
// under AddressSanitizer and UndefinedBehaviorSanitizer, without a GPU.  The
// few library functions those files call are stubbed here.  Exit status 0
// when every call returns; the sanitizers abort on the first finding.
#include <atomic>
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <random>
#include <string>
#include <vector>

#include <memory>
#include <thread>

#include "../../include/lucore_cpu.hpp"
#include "../../include/lufqhe.h"
#include "../../lion-codes_amd/csrc/kept_pool.hpp"

extern "C" {
// stubs of the kernel tables: 4 candidate shapes per n
int32_t lufqhe_shape_count(int32_t n) { return (n >= 1 && n <= 64) ? 4 : 0; }
int32_t lufqhe_shape_info(int32_t n, int32_t shape, int32_t* lanes, int32_t* cols, int32_t* waves) {
  if (n < 1 || n > 64 || shape < 0 || shape > 3 || !lanes || !cols) return LUFQHE_ERROR_INVALID_VALUE;
  *lanes = 64;
  *cols = 2;
  if (waves) *waves = 1;
  return LUFQHE_SUCCESS;
}
int32_t lufqhe_shape_kernel(int32_t n, int32_t) { return n > 24; }
int32_t lufqhe_set_default_shape(int32_t, int32_t, int32_t, int32_t) { return LUFQHE_SUCCESS; }
const char* lufqhe_status_string(int32_t) { return "stub"; }
}

static std::string write_tmp(const char* name, const std::string& text) {
  const char* dir = std::getenv("TMPDIR");
  std::string p = std::string(dir ? dir : "/tmp") + "/" + name;
  FILE* f = std::fopen(p.c_str(), "wb");
  if (!f) std::exit(3);
  std::fwrite(text.data(), 1, text.size(), f);
  std::fclose(f);
  return p;
}

// The pool of buffers that idle servers keep: limits, order, and threads.
struct FakeBuf {
  static std::atomic<int> live;
  int owner;
  explicit FakeBuf(int o) : owner(o) { ++live; }
  ~FakeBuf() { --live; }
};
std::atomic<int> FakeBuf::live{0};

static int check_kept_pool() {
  using Pool = lufqhe::KeptPool<FakeBuf>;
  int o[40];
  auto make = [](int i) { return std::make_unique<FakeBuf>(i); };
  {
    Pool p(100);
    p.put(&o[0], make(0), 60);
    p.put(&o[1], make(1), 40);
    if (p.bytes(nullptr) != 100 || p.bytes(&o[0]) != 60 || FakeBuf::live != 2) return 20;
    p.put(&o[2], make(2), 30);  // the oldest makes room
    if (p.bytes(&o[0]) != 0 || p.bytes(&o[1]) != 40 || p.bytes(nullptr) != 70) return 21;
    p.put(&o[1], make(11), 50);  // one set per owner, now the newest
    if (p.bytes(&o[1]) != 50 || FakeBuf::live != 2) return 22;
    p.put(&o[3], make(3), 101);  // more than the limit is not kept, and costs nobody
    if (p.bytes(&o[3]) != 0 || p.bytes(nullptr) != 80 || FakeBuf::live != 2) return 23;
    p.put(&o[1], make(12), 101);  // nor is the owner's old set then
    if (p.bytes(&o[1]) != 0 || p.bytes(nullptr) != 30) return 24;
    auto b = p.take(&o[2]);
    if (!b || b->owner != 2 || p.take(&o[2]) || p.bytes(nullptr) != 0) return 25;
    p.put(&o[2], std::move(b), 100);
    if (!p.release(&o[2]) || p.release(&o[2]) || p.release(nullptr) || FakeBuf::live != 0) return 26;
    for (int i = 0; i < 40; ++i) p.put(&o[i], make(i), 1);
    if (p.bytes(nullptr) != Pool::kSets || FakeBuf::live != Pool::kSets || p.bytes(&o[23]) != 0 ||
        p.bytes(&o[24]) != 1)
      return 27;
    if (!p.release(nullptr) || FakeBuf::live != 0 || p.bytes(nullptr) != 0) return 28;
    std::vector<std::thread> th;
    std::atomic<int> wrong{0};
    for (int t = 0; t < 6; ++t)
      th.emplace_back([&, t] {
        for (int i = 0; i < 2000; ++i) {
          const int k = (7 * i + t) % 20;
          auto b = p.take(&o[k]);
          if (b && b->owner != k) ++wrong;
          p.put(&o[k], b ? std::move(b) : make(k), 1 + i % 30);
          if (i % 50 == t) p.release(i % 100 == t ? nullptr : &o[k]);
          if (p.bytes(nullptr) > 100) ++wrong;
        }
      });
    for (auto& t : th) t.join();
    if (wrong) return 29;
  }
  return FakeBuf::live == 0 ? 0 : 30;
}

int main(int argc, char** argv) {
  std::mt19937_64 rng(7);
  std::normal_distribution<double> g;
  for (int n = 1; n <= 64; ++n) {
    const int count = 7, ld = n + (n & 1);
    const int64_t stride = (int64_t)n * ld + 3;
    std::vector<double2> A((size_t)(count * stride + ld));
    for (auto& v : A) v = make_double2(g(rng), g(rng));
    for (int c = 0; c < n; ++c) A[(size_t)(2 * stride + c)].x = 0.0;  // a rejected row
    A[(size_t)(3 * stride)] = make_double2(NAN, INFINITY);
    std::vector<double2> det(count), mant(count);
    std::vector<int32_t> e(count), info(count);
    std::vector<int8_t> piv((size_t)count * n);
    for (int th : {1, 3})
      if (lufqhe_cpu_crout_det(A.data(), count, n, ld, stride, det.data(), mant.data(), e.data(),
                               info.data(), piv.data(), th) != LUFQHE_SUCCESS)
        return 4;
    double2 sum;
    int32_t bad;
    if (lufqhe_cpu_pair_sum(A.data(), count, n, ld, stride, &sum, &bad, 2) != LUFQHE_SUCCESS) return 5;
    std::vector<double2> one(A.begin(), A.begin() + (size_t)n * ld);
    double2 d1;
    LUCoreCPU::determinant(one.data(), &d1, n, ld);
    RunInfo ri(4, n, count, true);
    try {
      std::vector<double2> B((size_t)count * n * ri.getLoadSize());
      for (auto& v : B) v = make_double2(g(rng), g(rng));
      LUCoreCPU::CALL(B.data(), &sum, count, &ri, 0, 2);
    } catch (const LUCoreCPU::Error&) {
    }
  }
  if (const int bad_pool = check_kept_pool()) return bad_pool;
  // invalid arguments are refused without touching memory
  if (lufqhe_cpu_crout_det(nullptr, 3, 0, 1, 1, nullptr, nullptr, nullptr, nullptr, nullptr, 1) ==
      LUFQHE_SUCCESS)
    return 6;
  // the shape table: the committed one, then malformed files
  if (argc > 1 && lufqhe_load_shape_table(argv[1]) < 0) return 7;
  const char* bad_tables[] = {"", "{", "{\"entries\": [", "{\"entries\": [{\"n\": 99999999999}]}",
                              "{\"entries\": [{\"policy\": \"abs\", \"n\": \"32\", \"shape\": -4}]}",
                              "{\"entries\": [{\"n\": 8, \"shape\": 1, \"lanes\": 64, \"lane_cols\": 2",
                              "{\"entries\": [{}, {}, {\"n\":,}]}"};
  int i = 0;
  for (const char* t : bad_tables)
    (void)lufqhe_load_shape_table(write_tmp(("bad_table_" + std::to_string(i++)).c_str(), t).c_str());
  (void)lufqhe_load_shape_table("/nonexistent/shapes.json");
  std::printf("host driver: ok\n");
  return 0;
}
