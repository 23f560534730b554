// One react call by one group of lanes on the host, and the exponentials of the rates:
//   main MECH G FILL AT_END < doubles > doubles        main exp < arguments > results
#include <string>
#include "react_kernel.h"
#include "mech/drm19.h"
#include "mech/dodecane_lu.h"
#include "mech/lidryer.h"
#include <algorithm>
#include <cstring>
#include <unistd.h>
#include "tables.h"  // pack_blob, pack_jac_tabs of the library

namespace emu {
int lanes, cur;
bool at_end;
unsigned char fill;
std::vector<Region*> regions;
static ucontext_t ctx[kMaxLanes], main_ctx;
static std::vector<char> stacks[kMaxLanes];
static int kinds[kMaxLanes], left;
static uint64_t slots[2][kMaxLanes], turn[kMaxLanes];
static void (*body)();

template <class... A>
static void stop(const char* text, A... a) {
  fprintf(stderr, text, a...);
  _exit(3);
}
void yield() {
  const int me = cur;
  cur = (cur + 1) % lanes;
  swapcontext(&ctx[me], &ctx[cur]);
}
uint64_t* box() { return slots[turn[cur]++ & 1]; }
void meet(int kind) {
  kinds[cur] = kind;
  yield();
  for (int l = 0; cur == 0 && l < lanes; ++l)  // lane 0 is the first to go on
    if (kinds[l] != kind) stop("lane 0 is at operation %d, lane %d at %d\n", kind, l, kinds[l]);
}
void sync() {
  meet(9);
  if (cur == 0)
    for (Region* r : regions)
      for (size_t w = 0; w < r->words; ++w) {
        const uint32_t old = r->base[w];
        int by = -1;
        for (int l = 0; l < lanes; ++l)
          if (r->copy[l][w] != old) {
            if (by >= 0 && r->copy[l][w] != r->base[w])
              stop("lanes %d and %d store different values to word %zu\n", by, l, w);
            by = l;
            r->base[w] = r->copy[l][w];
          } else if (r->uniform && by >= 0) {
            stop("word %zu of the control block differs between lanes\n", w);
          }
        if (by >= 0)
          for (int l = 0; l < lanes; ++l) r->copy[l][w] = r->base[w];
      }
}
static void lane_main() {
  body();
  if (--left == 0) setcontext(&main_ctx);
  const int me = cur;
  cur = (cur + 1) % lanes;
  swapcontext(&ctx[me], &ctx[cur]);
}
static void run(void (*f)()) {
  body = f;
  left = lanes;
  for (int l = 0; l < lanes; ++l) {
    stacks[l].resize(1 << 20);
    getcontext(&ctx[l]);
    ctx[l].uc_stack.ss_sp = stacks[l].data();
    ctx[l].uc_stack.ss_size = stacks[l].size();
    ctx[l].uc_link = nullptr;
    makecontext(&ctx[l], lane_main, 0);
  }
  cur = 0;
  swapcontext(&main_ctx, &ctx[0]);
}
}  // namespace emu

static prk::KParams P;
static std::vector<unsigned char> blob, jtabs;
static const pr_mech_t* mech;

namespace prk {
unsigned char* emu_smem() {
  static std::vector<unsigned char> lds(1 << 20);  // the kernel's own copy of the blob, not read
  return lds.data();
}
const unsigned char* emu_blob(int from, int to) {
  static std::vector<std::pair<int, unsigned char*>> made;
  for (auto& m : made)
    if (m.first == from) return m.second;
  unsigned char* p = emu::guarded(to - from);
  memcpy(p, blob.data() + from, to - from);
  made.push_back({from, p});
  return p;
}
}  // namespace prk

template <int N, int R, int G>
static void launch() {
  emu::lanes = G;
  emu::run([] { prk::react_kernel<N, R, G, 2>(P); });
}

template <class T>
static std::vector<T> get(size_t n) {
  std::vector<T> v(n);
  if (fread(v.data(), sizeof(T), n, stdin) != n) exit(4);
  return v;
}

int main(int argc, char** argv) {
  if (argc == 2) {  // exp_n and log_2 of the arguments, two at a time
    emu::lanes = 1;
    const long n = get<long>(1)[0];
    std::vector<double> x = get<double>(n), out(2 * n);
    const prk::ExpK K = prk::exp_constants();
    for (long i = 0; i < n; i += 2) {
      const double a[2] = {x[i], x[i + 1]};
      double e[2], l[2];
      prk::exp_n<2>(K, a, e);
      prk::log_2(a[0], a[1], l[0], l[1]);
      for (int k = 0; k < 2; ++k) {
        out[i + k] = e[k];
        out[n + i + k] = l[k];
      }
    }
    fwrite(out.data(), 8, out.size(), stdout);
    return 0;
  }
  const std::string name = argv[1];
  const int G = atoi(argv[2]);
  emu::fill = (unsigned char)atoi(argv[3]);
  emu::at_end = atoi(argv[4]);
  mech = name == "LiDryer" ? &pr_lidryer : (name == "drm19" ? &pr_drm19 : &pr_dodecane_lu);
  const int N = mech->nsp;
  const long nc = get<long>(1)[0];
  const double dt = get<double>(1)[0];
  std::vector<double> in = get<double>((2 * N + 3) * nc), FC(nc, 0.0);
  blob = pack_blob(mech);
  size_t off[3];
  jtabs = pack_jac_tabs(mech, blob, off, &P.jt.nentry);
  P.jt.term = (const prk::JacTerm*)(jtabs.data() + off[0]);
  P.jt.entry = (const prk::JacEntry*)(jtabs.data() + off[1]);
  P.jt.slice = (const int32_t*)(jtabs.data() + off[2]);
  auto arr = [&](double* p, long ns) { return prk::Arr{p, nc, nc, ns, 0, 0, 0}; };
  prk::BoxDesc B{};
  B.nx = (int)nc;
  B.ny = 1;
  B.ncells = nc;
  B.rY = arr(in.data(), nc);
  B.rYsrc = arr(in.data() + N * nc, nc);
  B.T = arr(in.data() + 2 * N * nc, 0);
  B.rH = arr(in.data() + (2 * N + 1) * nc, 0);
  B.rHsrc = arr(in.data() + (2 * N + 2) * nc, 0);
  B.FC = arr(FC.data(), 0);
  B.dt = dt;
  unsigned int queue = 0, nfail = 0;
  unsigned long long stats[8] = {};
  std::vector<double> atolv(N + 1, 1e-10);
  P.boxes = &B;
  P.nbox = 1;
  P.ncells = nc;
  P.rtol = P.atol = 1e-10;
  P.atolv = atolv.data();
  P.max_order = 4;
  P.max_steps = 10000;
  P.blob = blob.data();
  P.blob_bytes = (int)blob.size();
  P.neff = mech->neff;
  P.ninc = mech->ninc;
  P.queue = &queue;
  P.nfail = &nfail;
  P.stats = stats;
  double slot = 0.0;
  P.gscr = &slot;  // the views do not use it
  if (name == "LiDryer" && G == 8) launch<PR_LIDRYER_NSP, PR_LIDRYER_NR, 8>();
  else if (name == "LiDryer" && G == 16) launch<PR_LIDRYER_NSP, PR_LIDRYER_NR, 16>();
  else if (name == "LiDryer" && G == 32) launch<PR_LIDRYER_NSP, PR_LIDRYER_NR, 32>();
  else if (name == "LiDryer" && G == 64) launch<PR_LIDRYER_NSP, PR_LIDRYER_NR, 64>();
  else if (name == "drm19" && G == 16) launch<PR_DRM19_NSP, PR_DRM19_NR, 16>();
  else if (name == "drm19" && G == 32) launch<PR_DRM19_NSP, PR_DRM19_NR, 32>();
  else if (name == "drm19" && G == 64) launch<PR_DRM19_NSP, PR_DRM19_NR, 64>();
  else if (name == "dodecane_lu" && G == 64) launch<PR_DODECANE_LU_NSP, PR_DODECANE_LU_NR, 64>();
  else return 5;
  std::vector<double> out(in.begin(), in.begin() + N * nc);
  out.insert(out.end(), in.begin() + 2 * N * nc, in.begin() + (2 * N + 2) * nc);
  out.insert(out.end(), FC.begin(), FC.end());
  out.push_back((double)nfail);
  fwrite(out.data(), 8, out.size(), stdout);
  return 0;
}
