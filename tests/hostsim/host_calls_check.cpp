// Sequences of calls a host program makes, through the product's host runtime
// built against the host-only HIP stand-in.  TEST SCAFFOLDING.
//   host_calls_check CHECK
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <string>
#include <thread>
#include <vector>

#include "../../include/wx_capi.h"
#include "../../walicxe2d_amd/csrc/wx_runtime.h"
#include "../../walicxe2d_amd/csrc/wx_surrogate.h"

#define launch_build_tables launch_build_tables_cpu
#define launch_transpose launch_transpose_cpu
#define launch_stageA launch_stageA_cpu
#define launch_stageB launch_stageB_cpu
#include "fake_kernels.cpp"
#undef launch_build_tables
#undef launch_transpose
#undef launch_stageA
#undef launch_stageB

static int g_builds = 0;   // launches of the device table builder
static const double *g_state = nullptr;   // tiles that no launch may write, and how many values
static size_t g_nstate = 0;
static int g_stage[2] = {0, 0};   // stage launches, by whether the general form is asked for
namespace wx {
int launch_stageA(const wx_params *P, int neq, QueueRef q, int grid, int bs, int persist, const double *U, double *Uh,
                  const double *Pc, DevScalars *S, hipStream_t st) {
  ++g_stage[q.general != 0];
  return launch_stageA_cpu(P, neq, q, grid, bs, persist, U, Uh, Pc, S, st);
}
int launch_stageB(const wx_params *P, int neq, QueueRef q, int grid, int bs, int persist, const int2 *ops,
                  const BlockRec *binfo, double *U, double *Uh, DevScalars *S, hipStream_t st) {
  ++g_stage[q.general != 0];
  return launch_stageB_cpu(P, neq, q, grid, bs, persist, ops, binfo, U, Uh, S, st);
}
int launch_transpose(int neq, int cap, const double *src, double *dst, int mode, int ld, hipStream_t st) {
  if (g_state && dst >= g_state && dst < g_state + g_nstate) {
    fprintf(stderr, "a launch writes the state\n");
    _Exit(1);
  }
  return launch_transpose_cpu(neq, cap, src, dst, mode, ld, st);
}
int launch_build_tables(const wx_params &p, const TreeRow *T, int nbmax, int nleaf_host, LbInfo *info, LbPart *part,
                        LbOut out, int wide, DevScalars *S, hipStream_t st) {
  ++g_builds;
  return launch_build_tables_cpu(p, T, nbmax, nleaf_host, info, part, out, wide, S, st);
}
}  // namespace wx

#define REQUIRE(x)                                              \
  do {                                                          \
    if (!(x)) {                                                 \
      char b[512] = "";                                         \
      wx_last_error(b, 512);                                    \
      fprintf(stderr, "line %d: %s (%s)\n", __LINE__, #x, b);   \
      _Exit(1);                                                 \
    }                                                           \
  } while (0)

static wx_params params(int rx, int ry, int nlevs, int nblocks, int otherb) {
  wx_params p{};
  p.neq = 4; p.nlevs = nlevs; p.nbrootx = rx; p.nbrooty = ry; p.nblocks = nblocks; p.otherb = otherb;
  p.cv = 1.5; p.gamma = 5. / 3.; p.cfl = 0.4; p.tol = 0.05; p.tol2 = 1.0;
  p.Tempsc = 1; p.Psc = 1; p.tsc = 1;
  for (int l = 0; l < nlevs; ++l) p.dx[l] = p.dy[l] = 1.0 / (16 * rx) / (1 << l);
  return p;
}

static wx_ctx *context(const wx_params &p) {
  wx_ctx *c = nullptr;
  REQUIRE(wx_create(&p, &c) == WX_OK);
  std::vector<double> u((size_t)(p.nbrootx * p.nbrooty + 1) * p.neq * 400, 1.0);
  REQUIRE(wx_basegrid(c, u.data(), p.nbrootx * p.nbrooty) == WX_OK);
  return c;
}

struct Tables {
  std::vector<int32_t> rec, o2, o1;
  bool operator==(const Tables &t) const { return rec == t.rec && o2 == t.o2 && o1 == t.o1; }
};
static Tables tables(wx_ctx *c) {
  int32_t n = 0;
  REQUIRE(wx_get_tables(c, &n, nullptr, nullptr, nullptr, 0) == WX_OK);
  Tables t{std::vector<int32_t>((size_t)n * 8), std::vector<int32_t>((size_t)n * 16), std::vector<int32_t>((size_t)n * 16)};
  REQUIRE(wx_get_tables(c, &n, t.rec.data(), t.o2.data(), t.o1.data(), n) == WX_OK);
  return t;
}

// A list from the host that leaves segments uncovered is refused; the
// library's own list afterwards gives the tables it gave before, the jet
// imposition flags of the leaf records included.
static void rejected_list() {
  for (int builder : {0, 1}) {
    wx_ctx *c = context(params(4, 3, 2, 100, 1));
    REQUIRE(wx_set_builder(c, builder) == WX_OK);
    REQUIRE(wx_locatebounds(c, nullptr) == WX_OK);
    const Tables want = tables(c);
    int flagged = 0;
    for (size_t l = 0; l < want.rec.size() / 8; ++l) flagged += want.rec[l * 8 + 4] & 1;
    REQUIRE(flagged > 0);
    REQUIRE(wx_set_bounds(c, nullptr, 0, 0) != WX_OK);
    REQUIRE(wx_locatebounds(c, nullptr) == WX_OK);
    REQUIRE(tables(c) == want);
    wx_destroy(c);
  }
}

struct Tree {
  int32_t nbmax = 0, nbleafs = 0;
  std::vector<int32_t> lp, leaf, ic;
};
static Tree tree(wx_ctx *c) {
  Tree t;
  REQUIRE(wx_info(c, &t.nbmax, &t.nbleafs, nullptr) == WX_OK);
  t.lp.resize((size_t)t.nbmax * 8);
  t.leaf.resize(t.nbmax);
  t.ic.resize((size_t)t.nbmax * 2);
  REQUIRE(wx_get_tree(c, t.lp.data(), t.leaf.data(), t.ic.data(), t.nbmax, &t.nbmax, &t.nbleafs) == WX_OK);
  return t;
}
static int upload_tree(wx_ctx *c, const Tree &t) {
  return wx_upload_tree(c, t.lp.data(), t.leaf.data(), t.ic.data(), t.nbmax, t.nbmax, t.nbleafs);
}

// Where the ops are built by default: a tree that is new as a whole counts as
// a change that rewrote much of it (on the device from 6 144 leaves up), a
// change of a few rows does not.
static void builder_of_new_trees() {
  for (int ry : {95, 96}) {   // 6 080 and 6 144 roots
    const int dev = ry == 96;
    wx_ctx *c = context(params(64, ry, 2, 64 * ry + 400, 0));
    g_builds = 0;
    REQUIRE(wx_locatebounds(c, nullptr) == WX_OK);
    REQUIRE(g_builds == dev);
    Tree t = tree(c);
    for (int32_t &x : t.ic) x += 16;
    REQUIRE(upload_tree(c, t) == WX_OK);
    REQUIRE(wx_locatebounds(c, nullptr) == WX_OK);
    REQUIRE(g_builds == 2 * dev);
    std::vector<signed char> f(64 * ry + 1, 0);
    f[70] = 1;
    wxsim_set_flags(f.data(), (int)f.size());
    int32_t changed = 0;
    REQUIRE(wx_admesh(c, &changed) == WX_OK && changed == 1);
    REQUIRE(wx_locatebounds(c, nullptr) == WX_OK);
    REQUIRE(g_builds == 2 * dev);
    wx_destroy(c);
  }
}

// wx_info's list length after an upload of a tree that nothing has looked at
// yet: no pointer of it is followed.
static void info_of_an_unchecked_tree() {
  wx_ctx *c = context(params(6, 5, 2, 200, 0));
  REQUIRE(wx_locatebounds(c, nullptr) == WX_OK);
  std::vector<signed char> f(201, 0);
  f[8] = 1;
  wxsim_set_flags(f.data(), (int)f.size());
  int32_t changed = 0, nbmax = 0, nbleafs = 0, n = 0;
  REQUIRE(wx_admesh(c, &changed) == WX_OK && changed == 1);
  REQUIRE(wx_locatebounds(c, nullptr) == WX_OK);   // brought up to date without the list
  Tree t = tree(c);
  for (int k = 4; k < 8; ++k) t.lp[(size_t)k * t.nbmax + 2] = 1 << 28;
  REQUIRE(upload_tree(c, t) == WX_OK);
  REQUIRE(wx_info(c, &nbmax, &nbleafs, &n) == WX_OK && nbmax == 34 && nbleafs == 33);
  wx_destroy(c);
}

// A download, of any size, reads the state and nothing else of it: no launch
// writes the tiles, and two threads may download one context at once.
static void downloads() {
  for (int n : {1, 4, 80, 2700}) {   // one piece, and two (12.8 KB a block, 32 MiB)
    wx_params p = params(n, 1, 1, n, 0);
    wx_ctx *c = context(p);
    Tree t = tree(c);
    const size_t m = (size_t)(n + 1) * p.neq * 400;
    std::vector<double> u(m), got[2];
    for (size_t k = 0; k < m; ++k) u[k] = (double)(k * 2654435761u % 1000003u);
    REQUIRE(wx_upload(c, u.data(), WX_LAYOUT_BLOCK, t.lp.data(), t.leaf.data(), t.ic.data(), n, n, n) == WX_OK);
    // the tiles: the one allocation that holds exactly the uploaded interior cell
    for (const auto &a : hipsim::allocs)
      if (a.second == m * sizeof(double) && ((const double *)a.first)[p.neq * 400] == u[p.neq * 400 + 2 * 20 + 2]) {
        g_state = (const double *)a.first;
        g_nstate = m;
      }
    REQUIRE(g_state);
    for (int rep = 0; rep < 2; ++rep) {
      std::thread th[2];
      for (int k = 0; k < 2; ++k)
        th[k] = std::thread([&, k] {
          got[k].assign(m, 0.0);
          for (int r = 0; r < (n < 100 ? 40 : 2); ++r)
            REQUIRE(wx_download(c, got[k].data(), nullptr, WX_LAYOUT_BLOCK, 0) == WX_OK && got[k] == u);
        });
      for (std::thread &x : th) x.join();
    }
    g_state = nullptr;
    wx_destroy(c);
  }
}

// The stages are asked for their general form where a run's constants lie
// outside the short divisions' range, on any level in use and in any instance.
static void general_form() {
  const double lo = 0x1p-64, hi = 0x1p64;
  struct { double cv, Tempsc, dx1; int general; } k[] = {
      {1.5, 1e4, 1.0, 0}, {lo, lo, lo, 0}, {1.5, hi, 1.0, 1}, {1.5, 1e4, hi, 1}, {0.99 * lo, 1e4, 1.0, 1}, {1.5, -1e4, 1.0, 1}};
  for (const auto &x : k) {
    wx_params p[2] = {params(2, 2, 2, 40, 0), params(2, 2, 2, 40, 0)};
    p[1].cv = x.cv;
    p[1].Tempsc = x.Tempsc;
    p[1].dx[1] = x.dx1;
    p[1].dx[2] = p[1].dy[3] = 1e300;   // levels not in use
    g_stage[0] = g_stage[1] = 0;
    wx_ctx *c = context(p[1]);
    double t, dt, z;
    REQUIRE(wx_step(c, 1, 0, &t, &dt, &z) == WX_OK);
    REQUIRE(g_stage[x.general] == 2 && g_stage[!x.general] == 0);
    wx_destroy(c);
    wx_ens *e = nullptr;
    REQUIRE(wx_ens_create(p, 2, &e) == WX_OK);
    std::vector<double> u((size_t)5 * p[0].neq * 400, 1.0);
    for (int i = 0; i < 2; ++i) REQUIRE(wx_ens_basegrid(e, i, u.data(), 4) == WX_OK);
    REQUIRE(wx_ens_step(e, 1, 0, &z) == WX_OK);
    REQUIRE(g_stage[x.general] == 4 && g_stage[!x.general] == 0);
    wx_ens_destroy(e);
  }
}

// wx_profile counts the dt reduction where it is a launch (above 512 leaves),
// not where stage A takes it.
static void profile_counts() {
  for (int rx : {32, 33}) {   // 512 and 528 roots
    wx_ctx *c = context(params(rx, 16, 1, rx * 16, 0));
    double ms[wx::NPROF], t, dt, z;
    int64_t n[wx::NPROF];
    REQUIRE(wx_profile(c, 1, ms, n, wx::NPROF) == WX_OK);
    REQUIRE(wx_step(c, 3, 0, &t, &dt, &z) == WX_OK);
    REQUIRE(wx_profile(c, -1, ms, n, wx::NPROF) == WX_OK);
    REQUIRE(n[wx::KID_STAGEA] == 3 && n[wx::KID_STAGEB] == 3 && n[wx::KID_FILLI] == 3);
    REQUIRE(n[wx::KID_DTRED] == (rx == 32 ? 0 : 3));
    wx_destroy(c);
  }
}

int main(int argc, char **argv) {
  const std::string what = argc > 1 ? argv[1] : "";
  if (what == "rejected_list") rejected_list();
  else if (what == "builder_of_new_trees") builder_of_new_trees();
  else if (what == "info_of_an_unchecked_tree") info_of_an_unchecked_tree();
  else if (what == "downloads") downloads();
  else if (what == "general_form") general_form();
  else if (what == "profile_counts") profile_counts();
  else return 2;
  return 0;
}
