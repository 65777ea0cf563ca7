// CPU check of the batched engine's lane rows (tests/test_lane_rows_cpu.py
// builds and runs it; no GPU is used).  For every problem of a file of CSC
// problems it builds the stage image with the library's own host code, replays
// the setup kernel's derivation of the lane rows' columns and values
// (Solver::fill_group_values) and the product of each row (lane_piece), every
// index bounds-checked, and compares the FP32 and FP64 sums with the group
// walk's additions on the same row groups: equal to the bit.
// usage: lane_rows_check <problems file> [plant]   ("plant" moves one row's
// first-piece length in each image, which must then fail)
#include "serve/batch.hip"
using namespace osqp_serve;

static int fails = 0;
#define CHECK(c, ...) do { if (!(c)) { if (fails++ < 20) { fprintf(stderr, "FAIL %s:%d: ", __FILE__, __LINE__); fprintf(stderr, __VA_ARGS__); fprintf(stderr, "\n"); } } } while (0)

// the group walk's sum of a row whose first entry has slot `slot`: lane pieces
// in entry order, carried in from earlier lanes (at most three pieces: left to right)
template <typename T>
static T group_sum(const double* val, const int* ci, int len, int slot, const std::vector<T>& x) {
  T tot = 0;
  bool first = true;
  for (int k = 0; k < len;) {
    const int piece = std::min(len - k, kGroupPer - (slot + k) % kGroupPer);
    T acc = (T)val[k] * x[(size_t)ci[k]];
    for (int i = 1; i < piece; ++i) acc += (T)val[k + i] * x[(size_t)ci[k + i]];
    tot = first ? acc : tot + acc;
    first = false;
    k += piece;
  }
  return tot;
}

static long long n_rows = 0, n_pieces[4] = {0, 0, 0, 0};

template <typename T>
static void check(const char* name, const char* blk, size_t total, int rows, int cols, const GroupDims& d,
                  const Layout::Groups& o, size_t Orp, size_t Oci, size_t Oval) {
  const int* rp = (const int*)(blk + Orp);
  const int* ci = (const int*)(blk + Oci);
  const double* val = (const double*)(blk + Oval);
  const int* lsl = (const int*)(blk + o.lsl);
  const unsigned char* lc0 = (const unsigned char*)(blk + o.lc0);
  const int nls = lane_slices(rows);
  CHECK(nls <= kWave, "%s: slices", name);
  CHECK(o.lcol + 2 * (size_t)d.lane_slots <= total && o.lrv64 + 8 * (size_t)d.lane_slots <= total, "%s: lane block", name);
  std::vector<int> col((size_t)d.lane_slots, -1);
  std::vector<double> v((size_t)d.lane_slots, -1.0);
  for (int w = 0; w < nls * kWave; ++w) {
    const int r = w, at = lsl[2 * (w / kWave)] + w % kWave, steps = lsl[2 * (w / kWave) + 1];
    CHECK(steps == 1 || steps == 2 || steps == 4 || steps == 8 || steps == 16 || steps == 24, "%s: steps %d", name, steps);
    const int s0 = r < rows ? rp[r] : 0, c0 = r < rows ? lc0[r] : 0,
              len = c0 > 0 ? rp[r + 1] - s0 : 0;
    for (int k = 0; k < steps; ++k) {
      const int g = k / kGroupPer, q = g == 0 ? k : c0 + (g - 1) * kGroupPer + k % kGroupPer;
      const bool in = g == 0 ? k < c0 : q < len;
      const long long slot = at + (long long)k * kWave;
      CHECK(slot >= 0 && slot < d.lane_slots, "%s: slot %lld of %lld", name, slot, d.lane_slots);
      if (slot < 0 || slot >= d.lane_slots) return;
      CHECK(col[(size_t)slot] == -1, "%s: slot written twice", name);
      col[(size_t)slot] = in ? ci[s0 + q] : (len > 0 ? ci[s0] : 0);
      v[(size_t)slot] = in ? val[s0 + q] : 0.0;
    }
  }
  for (int c : col) CHECK(c >= 0 && c < cols, "%s: column %d", name, c);
  // the first slot of each row in its group
  const int* grow = (const int*)(blk + o.grow);
  const unsigned char* goff = (const unsigned char*)(blk + o.goff);
  std::vector<int> slot0((size_t)rows, -1);
  for (int i = 0; i < d.ng * kGroupSlots; ++i)
    if (grow[i] >= 0 && goff[i] == 0) slot0[(size_t)grow[i]] = i;
  std::vector<T> x((size_t)cols);
  for (int c = 0; c < cols; ++c) x[(size_t)c] = (T)std::sin(0.37 * c + 1.0);
  for (int r = 0; r < rows; ++r) {
    const int at = lsl[2 * (r / kWave)] + r % kWave, steps = lsl[2 * (r / kWave) + 1], len = rp[r + 1] - rp[r];
    CHECK((lc0[r] == 0) == (len > kLongRow), "%s: row %d of %d entries, first piece %d", name, r, len, lc0[r]);
    if (len > kLongRow) continue;  // a wavefront's, from the long-row list
    T tot = 0;
    for (int g = 0; g < steps; g += kGroupPer) {
      T acc = 0;
      for (int k = g; k < std::min(steps, g + kGroupPer); ++k) {
        const size_t s = (size_t)(at + k * kWave);
        const T pr = (T)v[s] * x[(size_t)col[s]];
        acc = k == g ? pr : acc + pr;
      }
      tot = g == 0 ? acc : tot + acc;
    }
    CHECK(slot0[(size_t)r] >= 0, "%s: row %d has no group slot", name, r);
    const T ref = group_sum<T>(val + rp[r], ci + rp[r], len, slot0[(size_t)r], x);
    CHECK(tot == ref, "%s: row %d: %.17g, groups %.17g", name, r, (double)tot, (double)ref);
    n_rows++;
    n_pieces[(slot0[(size_t)r] % kGroupPer + len + kGroupPer - 1) / kGroupPer]++;
  }
}

int main(int argc, char** argv) {
  if (argc < 2) return 2;
  FILE* f = fopen(argv[1], "rb");
  if (!f) return 2;
  const bool plant = argc > 2 && strcmp(argv[2], "plant") == 0;
  int np = 0, lanes = 0;
  if (fread(&np, 4, 1, f) != 1) return 2;
  for (int t = 0; t < np; ++t) {
    int n, m, want;
    if (fread(&n, 4, 1, f) != 1 || fread(&m, 4, 1, f) != 1 || fread(&want, 4, 1, f) != 1) return 2;
    std::vector<int> pp[2], pi[2];
    std::vector<double> px[2];
    OSQPCscMatrix M[2];
    for (int k = 0; k < 2; ++k) {
      int nnz;
      if (fread(&nnz, 4, 1, f) != 1) return 2;
      pp[k].resize(n + 1);
      pi[k].resize(nnz);
      px[k].resize(nnz);
      if (fread(pp[k].data(), 4, n + 1, f) != (size_t)n + 1 || fread(pi[k].data(), 4, nnz, f) != (size_t)nnz ||
          fread(px[k].data(), 8, nnz, f) != (size_t)nnz)
        return 2;
      M[k].m = k == 0 ? n : m;
      M[k].n = n;
      M[k].p = pp[k].data();
      M[k].i = pi[k].data();
      M[k].x = px[k].data();
      M[k].nzmax = M[k].nz = nnz;
      M[k].owned = 0;
    }
    std::vector<double> q(n, 0.0), l(m, -1.0), u(m, 1.0);
    for (int vbytes : {4, 8}) {
      HostData h;
      const Layout L = build_host(&h, vbytes, &M[0], q.data(), &M[1], l.data(), u.data(), nullptr, nullptr, false);
      const bool lane = want == 1 || (want == 2 && vbytes == 4);  // 2: in FP32 alone
      CHECK(h.gA.lanes == lane && h.gP.lanes == h.gA.lanes && h.gT.lanes == h.gA.lanes, "problem %d: lane rows %d", t,
            (int)h.gA.lanes);
      CHECK(bucket_of(h) == (lane ? kBuckets : 0) + size_bucket(n, m, h.nnzA, h.nnzP), "problem %d: bucket", t);
      if (!h.gA.lanes) continue;
      lanes++;
      std::vector<char> blk(L.total + 64, 0);
      memcpy(blk.data() + L.s_begin, h.img_ptr, L.s_end - L.s_begin);
      if (plant)
        for (int r = 0; r < m; ++r)
          if (((int*)(blk.data() + L.Arp))[r + 1] - ((int*)(blk.data() + L.Arp))[r] > 8) {
            unsigned char& c = ((unsigned char*)(blk.data() + L.gA.lc0))[r];
            c = c > 1 ? c - 1 : c + 1;
            break;
          }
      for (int pass = 0; pass < 2; ++pass) {
        auto one = [&](auto zero) {
          using T = decltype(zero);
          check<T>("P", blk.data(), L.lane_total, n, n, h.gP, L.gP, L.Prp, L.Pci, L.Pval);
          check<T>("A", blk.data(), L.lane_total, m, n, h.gA, L.gA, L.Arp, L.Aci, L.Aval);
          check<T>("At", blk.data(), L.lane_total, n, m, h.gT, L.gT, L.Trp, L.Tci, L.Tval);
        };
        if (pass == 0) one(0.0);
        else one(0.0f);
      }
    }
  }
  printf("problems with lane rows %d, rows %lld, by pieces %lld %lld %lld\n", lanes, n_rows, n_pieces[1], n_pieces[2],
         n_pieces[3]);
  CHECK(lanes > 0 && n_pieces[1] > 0 && n_pieces[2] > 0 && n_pieces[3] > 0, "nothing exercised");
  printf(fails ? "FAILURES: %d\n" : "all checks passed\n", fails);
  return fails ? 1 : 0;
}
