// The tables kept up to date from the rows of each mesh change (update_leaves,
// update_ops in walicxe2d_amd/csrc/wx_mesh.cpp) against a full compilation of
// the same tree: leaf records, block records, both fills' ops and the list.
// A front of refinement sweeps over the mesh, with stray flags; now and then
// the ops are left to another builder for a change, the tree comes from the
// host again, or the list does.  TEST SCAFFOLDING.
//   update_check RX RY NLEVS OTHERB COMPAT BC_LEFT BC_BOTTOM ROUNDS
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <random>
#include <vector>

#include "../../walicxe2d_amd/csrc/wx_runtime.h"

using namespace wx;

int main(int argc, char **argv) {
  if (argc != 9) return 2;
  wx_params p{};
  p.neq = 5; p.nblocks = 20000; p.nbrootx = atoi(argv[1]); p.nbrooty = atoi(argv[2]); p.nlevs = atoi(argv[3]);
  p.otherb = atoi(argv[4]); p.compat = atoi(argv[5]); p.bc[0] = atoi(argv[6]); p.bc[2] = atoi(argv[7]);
  const int rounds = atoi(argv[8]);
  Mesh m;
  m.init(p);
  if (basegrid_tree(&m)) return 3;
  std::mt19937 rng(17);
  int from_rows = 0, changes = 0;
  for (int r = 0; r < rounds; ++r) {
    const bool was_valid = m.tables_valid;
    if (r % 11 == 5 && !was_valid) {   // ops built elsewhere for this change
      if (update_leaves(&m)) return 3;
    }
    if (r % 53 == 20) {                // the list from the host
      locatebounds(&m);
      m.bounds_external = true;
      m.tables_valid = false;
    }
    if (update_tables(&m)) { fprintf(stderr, "update failed: %s\n", last_error().c_str()); return 3; }
    changes += !was_valid;
    from_rows += !was_valid && m.ops_ok && m.list_stale;
    // the full compilation, from a copy of the tree
    const int32_t ld = m.nbmax;
    std::vector<int32_t> lp((size_t)ld * 8), leaf(ld), ic((size_t)ld * 2);
    int32_t nbmax = 0, nbleafs = 0;
    if (get_tree(&m, lp.data(), leaf.data(), ic.data(), ld, &nbmax, &nbleafs)) return 3;
    Mesh f;
    f.init(p);
    if (set_tree(&f, lp.data(), leaf.data(), ic.data(), ld, nbmax, nbleafs, nullptr)) return 3;
    locatebounds(&f);
    if (compile_tables(&f)) return 3;
    const size_t n = f.leaves.size();
    bool same = m.leaves.size() == n && !memcmp(m.leaves.data(), f.leaves.data(), n * sizeof(LeafRec)) &&
                m.binfo.size() == f.binfo.size() &&
                !memcmp(m.binfo.data(), f.binfo.data(), f.binfo.size() * sizeof(BlockRec)) && m.opsI_same == f.opsI_same;
    for (size_t l = 0; same && l < n; ++l)
      same = !memcmp(m.leaf_ops(l), &f.opsII[l * 8], 64) && (m.opsI_same || !memcmp(&m.opsI[l * 8], &f.opsI[l * 8], 64)) &&
             m.lidx[m.leaves[l].id] == (int)l;
    for (int nb = 1; same && nb <= nbmax; ++nb) same = m.lidx[nb] == f.lidx[nb];
    if (same && m.list_stale) locatebounds(&m);
    same = same && m.ninternal == f.ninternal && m.bounds == f.bounds;
    if (!same) { fprintf(stderr, "round %d: tables differ\n", r); return 1; }
    if (r % 37 == 30) {                // the tree comes from the host, with a leaf more or less flagged anew
      if (set_tree(&m, lp.data(), leaf.data(), ic.data(), ld, nbmax, nbleafs, nullptr)) return 3;
    }
    std::vector<int8_t> fl(n, 0);
    const double R = 0.9 * r / rounds * p.nbrooty * NY;
    for (size_t l = 0; l < n; ++l) {
      const LeafRec &q = f.leaves[l];
      const double sc = 1.0 / (1 << (q.level - 1));
      const double d = std::fabs(std::hypot((q.icx + 8) * sc - p.nbrootx * 8, (q.icy + 8) * sc - p.nbrooty * 8) - R);
      fl[l] = d < 6 + 10 * sc ? 1 : (d > 12 + 16 * sc ? 2 : 0);
      if (rng() % 499 == 0) fl[l] = (int8_t)(rng() % 3);
      if (fl[l] == 1 && q.level >= p.nlevs) fl[l] = 0;
    }
    std::vector<MeshOp> ops;
    if (admesh_from_flags(&m, fl.data(), ops)) { fprintf(stderr, "admesh: %s\n", last_error().c_str()); return 3; }
    m.new_ids.clear();
  }
  printf("%d changes, %d from the rows\n", changes, from_rows);
  return from_rows > 0 ? 0 : 4;   // the path under test ran
}
