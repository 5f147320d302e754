// A queued patch whose id needs 31 bits through the rank test and the
// expansion (k_qr.hip, k_exact.hip), called directly on the CPU emulation of
// the library.  The mesh is five tets whose first vertex is number 2^30 + 3;
// its arrays are sparse mappings, of which only the entries in use exist.
#include <sys/mman.h>

#include "device.h"

using namespace sprg;

template <class T>
static T* sparse(size_t n)
{
  void* p = mmap(nullptr, n * sizeof(T), PROT_READ | PROT_WRITE, MAP_PRIVATE | MAP_ANONYMOUS | MAP_NORESERVE, -1, 0);
  if (p == MAP_FAILED) {
    perror("mmap");
    exit(2);
  }
  return static_cast<T*>(p);
}

int main()
{
  const int32_t c = (1 << 30) + 3;
  const int64_t nv = (int64_t)c + 1;
  // four tets around c whose centroids lie in a plane (the initial set has
  // rank 3) and one on an outer face, which completes it
  const int32_t tets[5][4] = {{c, 0, 2, 4}, {c, 2, 1, 4}, {c, 1, 3, 4}, {c, 3, 0, 4}, {0, 2, 4, 5}};
  const double at[6][3] = {{1, 0, 0}, {-1, 0, 0}, {0, 1, 0}, {0, -1, 0}, {0, 0, 1}, {1, 1, 1}};
  int32_t* const tv = sparse<int32_t>(4 * 5);
  int32_t* const off = sparse<int32_t>((size_t)nv + 1);
  int32_t* const v2t = sparse<int32_t>(4 * 5);
  double* const xyz = sparse<double>(3 * (size_t)nv);
  for (int t = 0; t < 5; ++t)
    for (int k = 0; k < 4; ++k) tv[4 * t + k] = tets[t][k];
  int n = 0;
  auto row = [&](int32_t v) {
    off[v] = n;
    for (int t = 0; t < 5; ++t)
      for (int k = 0; k < 4; ++k)
        if (tets[t][k] == v) v2t[n++] = t;
    off[v + 1] = n;
  };
  for (int32_t v = 0; v < 6; ++v) {
    row(v);
    for (int j = 0; j < 3; ++j) xyz[3 * v + j] = at[v][j];
  }
  row(c);
  FitArgs a = {};
  a.m.nv = nv;
  a.m.nt = 5;
  a.m.order = 1;
  a.m.straight = 1;
  a.m.tv = tv;
  a.m.xyz = xyz;
  a.m.v2t_off = off;
  a.m.v2t = v2t;
  a.fast = 1;
  a.q = 1;
  a.nc = 1;
  a.npatch = nv;
  a.shape.expand_blocks = 2;
  int32_t count[2 * NBUCKET + 2] = {}, status[5] = {}, xq[1] = {(int32_t)(c | 0x80000000u)}, xq_exact[1], fbq[1], big[1],
          x_patch[1] = {-1}, x_len[1] = {-7}, x_set[1024];
  int64_t x_off[1], cursor[2] = {};
  count[2 * NBUCKET] = 1;
  a.L.count = count;
  a.L.status = status;
  a.L.xq = xq;
  a.L.xq_exact = xq_exact;
  a.L.fbq = fbq;
  a.L.big = big;
  a.L.x_patch = x_patch;
  a.L.x_len = x_len;
  a.L.x_off = x_off;
  a.L.x_set = x_set;
  a.L.x_cursor = cursor;
  a.L.x_cap = 1024;
  a.L.cap = 1;
  if (launch_rank_test(a, 4, nullptr) || launch_expand(a, 4, nullptr)) return 2;
  printf("patch %d set of %d status %d tested %d deferred %d\n", x_patch[0], x_len[0], status[0], status[4], status[1]);
  bool ok = x_patch[0] == c && x_len[0] == 5 && status[0] == 0 && status[1] + status[4] == 1;
  for (int i = 0; ok && i < 5; ++i) ok = x_set[x_off[0] + i] == i;
  puts(ok ? "PASS" : "FAIL");
  return ok ? 0 : 1;
}
