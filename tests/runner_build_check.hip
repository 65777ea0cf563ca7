// CPU check of what the ADMM runner's build does when memory runs out
// (tests/test_runner_cpu.py builds and runs it; it stops where a GPU is
// visible).  Device memory is host memory here and no kernel runs: for every
// allocation of the two builds, the build is tried with that allocation
// refused, and with an exception in its place; each time the runner must come
// back off and empty, with every block given back and nothing recorded.  A
// launch that is refused (without a GPU all are) must be reported by runner_run.
#include "hip/runner.hip"

#include <set>

namespace osqp_hip {
static Runtime g_rt;
static std::set<void*> g_live;
static int g_at = 0, g_fail = -1, g_recorded = 0;
static bool g_throw = false;

Runtime& rt() { return g_rt; }
int check(hipError_t e, const char*, const char*, int) {  // launches fail without a GPU; only memory counts
  if (e == hipErrorOutOfMemory) g_recorded++;
  return 0;
}
void* dev_try_alloc(size_t bytes) {
  if (g_at++ == g_fail) {
    if (g_throw) throw std::bad_alloc();
    return nullptr;
  }
  void* p = calloc(1, bytes ? bytes : 1);
  g_live.insert(p);
  return p;
}
void* dev_alloc(size_t bytes) {
  void* p = dev_try_alloc(bytes);
  if (!p) g_recorded++;
  return p;
}
void dev_free(void* p) {
  if (!p) return;
  if (!g_live.erase(p)) fprintf(stderr, "FAIL: a block freed twice\n"), g_recorded++;
  free(p);
}
void upload(void* dst, const void* src, size_t bytes) { memcpy(dst, src, bytes); }
void download(void* dst, const void* src, size_t bytes) { memcpy(dst, src, bytes); }
}  // namespace osqp_hip

using namespace osqp_hip;

// m rows of `row` entries over n columns, and the diagonal as P
struct Problem {
  std::vector<int> arp, aci, prp, pci, krp, kci;
  std::vector<double> val;
  OSQPMatrix A, P;
  RunK K;
  Problem(int n, int m, int row) {
    for (int r = 0; r <= m; ++r) arp.push_back(r * row);
    for (int k = 0; k < m * row; ++k) aci.push_back(k % n);
    for (int j = 0; j <= n; ++j) prp.push_back(j);
    for (int j = 0; j < n; ++j) pci.push_back(j);
    for (int j = 0; j <= n; ++j) krp.push_back((int)((long long)m * row * j / n));
    kci.assign((size_t)m * row, 0);
    val.assign((size_t)m * row + n, 1.0);
    memset(&A, 0, sizeof(A));
    memset(&P, 0, sizeof(P));
    A.m = m;
    A.n = n;
    A.nnz = m * row;
    A.rp = arp.data();
    A.ci = aci.data();
    A.val = val.data();
    A.trp = krp.data();
    A.tci = kci.data();
    A.tval = val.data();
    P.m = P.n = n;
    P.nnz = n;
    P.rp = prp.data();
    P.ci = pci.data();
    P.val = val.data();
    K = RunK{krp.data(), kci.data(), val.data()};
  }
};

int main() {
  int devices = 0;
  if (hipGetDeviceCount(&devices) == hipSuccess && devices > 0) {
    fprintf(stderr, "a GPU is visible: device memory is not host memory here\n");
    return 2;
  }
  g_rt.num_cu = 256;
  int fails = 0;
  auto tries = [&](const char* name, Problem& p, int bits, bool one, int least) {
    for (bool thrown : {false, true}) {
      g_throw = thrown;
      int allocs = 0;
      for (g_fail = -1; g_fail < (allocs ? allocs : 1); ++g_fail) {
        Runner r;
        memset(&r, 0xAB, sizeof(r));
        g_at = 0;
        const int on = runner_build(&r, &p.A, &p.P, p.K, bits, one, 20);
        if (g_fail < 0) allocs = g_at;
        Runner zero;
        memset(&zero, 0, sizeof(zero));
        // (with no GPU the launch attribute is refused after the last allocation, so it is off there too)
        if (on || memcmp(&r, &zero, sizeof(r)) != 0 || !g_live.empty() || g_recorded) {
          fprintf(stderr, "FAIL %s, %d bits, allocation %d of %d%s: on %d, live %zu, recorded %d\n", name, bits, g_fail,
                  allocs, thrown ? " (exception)" : "", on, g_live.size(), g_recorded);
          fails++;
          g_live.clear();
          g_recorded = 0;
        }
      }
      printf("%s, %d bits, one %d: %d allocations\n", name, bits, (int)one, allocs);
      if (allocs < least) fprintf(stderr, "FAIL %s: %d allocations\n", name, allocs), fails++;
    }
  };
  Problem small(20, 40, 3), medium(2100, 100, 40), most(2100, 100, 40), past(2100, 100, 40);
  most.P.nnz = 64000000 - 4000;  // the line past which it is not built
  past.P.nnz = most.P.nnz + 1;
  for (int bits : {32, 64}) {
    tries("one workgroup", small, bits, true, bits == 32 ? 16 : 8);
    tries("several workgroups", medium, bits, false, 22);
    tries("several workgroups not asked for", medium, bits, true, 0);
    tries("at the most entries", most, bits, false, 4);
    tries("past the most entries", past, bits, false, 0);
  }
  for (int groups : {1, 32}) {
    Runner r;
    memset(&r, 0, sizeof(r));
    r.on = 1;
    r.n = 20;
    r.m = 40;
    r.bits = 64;
    r.G = groups;
    RunCall c;
    memset(&c, 0, sizeof(c));
    c.iters = 24;
    int z = -7;
    if (!runner_run(&r, &small.A, &small.P, small.K, c, &z) || z != -7)
      fprintf(stderr, "FAIL: a refused launch of %d workgroups went unnoticed\n", groups), fails++;
  }
  printf(fails ? "FAILURES: %d\n" : "all checks passed\n", fails);
  return fails ? 1 : 0;
}
