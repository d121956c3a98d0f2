// C ABI of the MI355X SEM path: meshes, shots, batches and the two step
// paths (plain separate kernels; fused colour kernels in hipGraph blocks).
//
// Host-side responsibilities mirror the reference's set-up code:
//   sem_mesh_create     Mesh::read + setupGlobalDof (Mesh.cpp:31-51, :361-452),
//                       attachVertexCoordinates / attachMaterialProperties,
//                       Order2Newmark::initializeGlobalDofs mass (Order2Newmark.cpp:32-66)
//   sem_shot_add_*      Problem::initializeElements source/receiver attach
//                       (Problem.cpp:34-142; QuadP1/HexP1 checkHull + Newton)
//   sem_batch_run       the time loop (Main.cpp:45-66)
#include <hip/hip_runtime.h>

#include <algorithm>
#include <array>
#include <chrono>
#include <cmath>
#include <cstdio>
#include <cstring>
#include <map>
#include <mutex>
#include <numeric>
#include <string>
#include <tuple>
#include <vector>

#include "batch.h"

namespace sem {

static thread_local std::string g_error;
void set_error(const std::string &msg) { g_error = msg; }
int hip_check(hipError_t e, const char *what) {
  if (e == hipSuccess) return 0;
  set_error(std::string(what) + ": " + hipGetErrorString(e));
  return -2;
}

}  // namespace sem

using namespace sem;

// ====================================================================== helpers
namespace sem {
int set_device(int device) {
  int n = 0;
  if (hipGetDeviceCount(&n) != hipSuccess || n == 0) {
    set_error("no HIP device visible");
    return -4;
  }
  if (device < 0 || device >= n) {
    set_error("device index out of range");
    return -1;
  }
  HIPCHK(hipSetDevice(device));
  SEM_TRY(init_device_tables(device));
  return init_tile_tables(device);
}
}  // namespace sem

static bool is_affine(int dim, const double *v) {
  // All bilinear/trilinear cross terms of the P1 map vanish.
  double scale = 0;
  const int nv = dim == 2 ? 4 : 8;
  for (int i = 0; i < nv * dim; ++i) scale = std::max(scale, std::fabs(v[i]));
  const double tol = 1e-12 * (scale + 1.0);
  if (dim == 2) {
    for (int a = 0; a < 2; ++a)
      if (std::fabs(v[0 * 2 + a] - v[1 * 2 + a] + v[2 * 2 + a] - v[3 * 2 + a]) > tol) return false;
    return true;
  }
  static const double s[8][3] = {{-1, -1, -1}, {-1, 1, -1}, {1, 1, -1}, {1, -1, -1},
                                 {-1, -1, 1},  {1, -1, 1},  {1, 1, 1},  {-1, 1, 1}};
  for (int a = 0; a < 3; ++a) {
    double rs = 0, rt = 0, st = 0, rst = 0;
    for (int k = 0; k < 8; ++k) {
      double x = v[k * 3 + a];
      rs += s[k][0] * s[k][1] * x;
      rt += s[k][0] * s[k][2] * x;
      st += s[k][1] * s[k][2] * x;
      rst += s[k][0] * s[k][1] * s[k][2] * x;
    }
    if (std::fabs(rs) > tol || std::fabs(rt) > tol || std::fabs(st) > tol || std::fabs(rst) > tol)
      return false;
  }
  return true;
}

// Temporary device space of one step: the mesh's while it is created, else its own.
// A mesh whose temporaries are small shares no buffer: its allocations come from
// what the runtime keeps of released ones, and releasing them leaves more of that to
// the first batch behind.  Creation and first pass, ms, with a shared buffer, without:
// 100^2 acoustic quads (3 MB) 5.7, 5.3; 150x133 deformed elastic quads (7 MB) 10.1, 9.1;
// 27x25x23 order-3 elastic hexes (11 MB) 27.4, 30.2; operator on 24x23x22 deformed
// elastic hexes (18 MB) 10.9, 12.6; 31x30x29 deformed acoustic hexes (41 MB) 32.7, 35.1.
constexpr size_t kMinShared = (size_t)8 << 20;
struct TempSpace {
  unsigned char *p = nullptr;
  bool own = false;
  int get(sem_mesh *m, size_t bytes) {
    own = bytes > m->temp_bytes;
    if (own) return dalloc(&p, bytes);
    p = m->d_temp;
    return 0;
  }
  ~TempSpace() {
    if (own) dfree(p);
  }
};

// The Dirichlet flags of n words (node | flags, or kSlotEmpty) in place, a piece at
// a time through the host.
static int reflag_words(sem_mesh *m, uint32_t *d_words, size_t n, const std::vector<uint8_t> &dirichlet) {
  const size_t piece = (size_t)1 << 20;
  std::vector<uint32_t> words(std::min(n, piece));
  for (size_t i = 0; i < n; i += piece) {
    const size_t k = std::min(piece, n - i);
    HIPCHK(hipMemcpyAsync(words.data(), d_words + i, k * 4, hipMemcpyDeviceToHost, m->stream));
    HIPCHK(hipStreamSynchronize(m->stream));
    for (size_t j = 0; j < k; ++j)
      if (words[j] != kSlotEmpty)
        words[j] = (words[j] & ~kFlagDirichlet) | (dirichlet[words[j] & kNodeMask] ? kFlagDirichlet : 0u);
    HIPCHK(hipMemcpyAsync(d_words + i, words.data(), k * 4, hipMemcpyHostToDevice, m->stream));
    HIPCHK(hipStreamSynchronize(m->stream));
  }
  return 0;
}

// The gather map in the sorted (colour) order with its flags, built on the
// device: the first and last colour of every node from one pass per colour
// (a host loop over the element nodes took three times as long: 13 ms of the
// 102 ms set-up of 32^3 hexes).
static int upload_conn(sem_mesh *m) {
  const int64_t E = m->E, nd = m->nd;
  const bool built = m->d_conn != nullptr;
  if (!built) SEM_TRY(dalloc(&m->d_conn, E * nd, &m->bytes));
  TempSpace temp;  // gather map, order, first and last colours, Dirichlet mask
  if (int rc = temp.get(m, 4 * (size_t)(E * nd + E + 2 * m->G + (m->G + 3) / 4)))
    return built ? reflag_words(m, m->d_conn, (size_t)(E * nd), m->dirichlet) : rc;  // no memory for it: flags only
  int32_t *d_raw = reinterpret_cast<int32_t *>(temp.p);
  int32_t *d_perm = d_raw + E * nd, *d_span = d_perm + E;
  uint8_t *d_dir = m->dirichlet.empty() ? nullptr : reinterpret_cast<uint8_t *>(d_span + 2 * m->G);
  int rc = 0;
  auto up = [&](void *dst, const void *src, size_t n) {
    if (!rc) rc = hip_check(hipMemcpyAsync(dst, src, n, hipMemcpyHostToDevice, m->stream), "upload");
  };
  up(d_raw, m->conn.data(), (size_t)(E * nd) * 4);
  up(d_perm, m->perm.data(), (size_t)E * 4);
  if (d_dir) up(d_dir, m->dirichlet.data(), (size_t)m->G);
  if (!rc) rc = launch_fill_i32(2 * m->G, d_span, -1, m->stream);
  for (int c = 0; c < m->ncol && !rc; ++c)
    rc = launch_conn_span(m->col_start[c], m->col_start[c + 1] - m->col_start[c], (int)nd, c, d_perm, d_raw, d_span,
                          d_span + m->G, m->stream);
  for (int c = 0; c < m->ncol && !rc; ++c)
    rc = launch_conn_flags(m->col_start[c], m->col_start[c + 1] - m->col_start[c], (int)nd, c, d_perm, d_raw,
                           d_span, d_span + m->G, d_dir, m->d_conn, m->stream);
  if (!rc) rc = hip_check(hipStreamSynchronize(m->stream), "gather map");
  return rc;
}

int sem::ensure_pointwise(sem_mesh *m) {
  if (m->d_geo_p) return 0;
  const int gm = pointwise_mode(m);
  const int ngp = point_geo_count(m->dim, m->physics, gm);
  SEM_TRY(dalloc(&m->d_geo_p, (size_t)m->E * ngp * m->nd, &m->bytes));
  SEM_TRY(launch_point_geometry(m->dim, m->order, m->physics, gm, m->E, m->d_vtx, m->d_vpar,
                                ref_npar(m->dim, m->physics), m->d_geo_p, nullptr, m->stream));
  HIPCHK(hipStreamSynchronize(m->stream));
  return 0;
}

// Partial results of the element kernel: a node of several elements gets one
// per element, a class of nodes (those of m elements) copy after copy.  They
// take the place of the accumulator and the colour launches unless they need
// much more memory than it: from order 4 in 3-D and 3 in 2-D on they are at
// most 1.6 arrays of the nodes; at lower orders (up to 8 arrays) only up to
// 256 MiB per shot, beyond which the launches they save no longer matter (at
// that size a colour's launch runs for a hundred times its latency) and the
// colours stay; so they do for a node of 63 elements or more (the classes are
// counted on the device, one a lane; no mesh generator makes such a node).
static std::mutex mesh_lazy;  // batches prepared in several threads may share a mesh
constexpr double kMaxPartsPerNode = 1.6;
constexpr int64_t kMaxSmallParts = (int64_t)256 << 20;
int sem::ensure_elem_parts(sem_mesh *m) {
  std::lock_guard<std::mutex> lock(mesh_lazy);
  if (m->elem_parts >= 0) return 0;
  // elements per node; the nodes of each count, block of nodes by block
  const int nb = (int)((m->G + kClassNodes - 1) / kClassNodes);
  std::vector<int32_t> count((size_t)nb * kNodeClasses);
  TempSpace temp;  // elements per node, strides, counts, table
  SEM_TRY(temp.get(m, 4 * (2 * (size_t)m->G + count.size() + 3 * kNodeClasses)));
  int32_t *d_hits = reinterpret_cast<int32_t *>(temp.p);
  uint32_t *d_next = reinterpret_cast<uint32_t *>(d_hits), *d_stride = d_next + m->G;
  int32_t *d_count = d_hits + 2 * m->G;
  int rc = launch_fill_i32(m->G, d_hits, 0, m->stream);
  if (!rc) rc = launch_colour_touch(0, m->E, m->nd, m->d_conn, d_hits, m->stream);
  if (!rc) rc = launch_class_count(m->G, d_hits, d_count, m->stream);
  if (!rc) rc = hip_check(hipMemcpyAsync(count.data(), d_count, count.size() * 4, hipMemcpyDeviceToHost, m->stream), "copy");
  if (!rc) rc = hip_check(hipStreamSynchronize(m->stream), "sync");
  if (rc) return rc;
  std::vector<int64_t> n(kNodeClasses, 0);  // elements per node -> nodes
  for (int b = 0; b < nb; ++b)
    for (int k = 0; k < kNodeClasses; ++k) {
      const int32_t here = count[(size_t)b * kNodeClasses + k];
      count[(size_t)b * kNodeClasses + k] = (int32_t)n[k];  // the block's first within its class
      n[k] += here;
    }
  int64_t nodes = 0, parts = 0;
  std::vector<SharedClass> classes;
  std::vector<uint32_t> table(3 * kNodeClasses, 0);  // per class: first in the list, first part, nodes
  for (int k = 2; k < kNodeClasses; ++k) {
    if (!n[k]) continue;
    classes.push_back(SharedClass{k, n[k], nodes, parts});
    table[3 * k] = (uint32_t)nodes;
    table[3 * k + 1] = (uint32_t)parts;
    table[3 * k + 2] = (uint32_t)n[k];
    nodes += n[k];
    parts += k * n[k];
  }
  if ((parts > kMaxPartsPerNode * m->G && 4 * m->c * parts > kMaxSmallParts) || parts >= ((int64_t)1 << 32) ||
      n[kNodeClasses - 1]) {  // the last class: this many elements per node or more
    m->elem_parts = 0;
    return 0;
  }
  // one buffer: positions, shared nodes (from a cache line's start on)
  const size_t npos = ((size_t)m->E * m->nd + 63) / 64 * 64;
  SEM_TRY(dalloc(&m->d_epos, npos + nodes, &m->bytes));
  m->d_sh_node = m->d_epos + npos;
  rc = hip_check(hipMemcpyAsync(d_count, count.data(), count.size() * 4, hipMemcpyHostToDevice, m->stream), "upload");
  if (!rc) rc = hip_check(hipMemcpyAsync(d_count + count.size(), table.data(), table.size() * 4, hipMemcpyHostToDevice, m->stream), "upload");
  if (!rc) rc = launch_class_list(m->G, d_count, reinterpret_cast<const uint32_t *>(d_count + count.size()), d_next,
                                  d_stride, m->d_sh_node, m->stream);
  for (int c = 0; c < m->ncol && !rc; ++c)  // copies in the order of the colours
    rc = launch_elem_pos(m->col_start[c], m->col_start[c + 1] - m->col_start[c], m->nd, m->d_conn, d_stride,
                         d_next, m->d_epos, m->stream);
  if (!rc) rc = hip_check(hipStreamSynchronize(m->stream), "sync");
  if (rc) {
    dfree(m->d_epos);
    m->d_sh_node = nullptr;
    m->bytes -= (npos + nodes) * 4;
    return rc;
  }
  m->classes = classes;
  m->nparts = parts;
  m->elem_parts = 1;
  return 0;
}

// Tile shape: the first compiled shape of the preference list for this
// dimension/physics, or exactly SEM_TILE=x,y[,z] (no tiles if that shape has
// no kernel for the mesh's order).  Returns false when no shape applies.
static bool pick_tile(int dim, int order, int physics, int *T) {
  const char *env = getenv("SEM_TILE");
  if (env && *env) {
    int a = 0, b = 0, c = 1;
    if (sscanf(env, "%d,%d,%d", &a, &b, &c) < 2 || a <= 0 || b <= 0 || c <= 0) return false;
    T[0] = a; T[1] = b; T[2] = dim == 3 ? c : 1;
    return tile_kernel_info(dim, order, physics, T).lds_bytes > 0;
  }
  static const int pref2[][3] = {{16, 8, 1}, {8, 8, 1}};
  static const int pref3a[][3] = {{4, 4, 2}, {4, 2, 2}};
  static const int pref3e[][3] = {{4, 2, 2}, {2, 2, 2}};
  const int(*list)[3] = dim == 2 ? pref2 : (physics == SEM_ACOUSTIC ? pref3a : pref3e);
  const int cnt = 2;
  for (int i = 0; i < cnt; ++i) {
    T[0] = list[i][0]; T[1] = list[i][1]; T[2] = list[i][2];
    const TileKernelInfo k = tile_kernel_info(dim, order, physics, T);
    if (k.lds_bytes > 0 && k.lds_bytes <= 160 * 1024) return true;
  }
  return false;
}

// (groups hold these buffers and read both in every step: a mask set later
// acts on them too)
static void free_colour_tiles(sem_mesh *m);
static int reflag_colour_tiles(sem_mesh *m) {
  const ColourTiles &ct = m->ctiles;
  const size_t n = (size_t)m->tiles.ntiles * m->tiles.slots_per_tile;
  std::vector<uint8_t> dirichlet(m->G);
  for (int64_t g = 0; g < m->G; ++g) dirichlet[ct.to_internal[g]] = m->dirichlet[g];
  SEM_TRY(reflag_words(m, ct.d_words, n, dirichlet));
  return ct.d_words_lat ? reflag_words(m, ct.d_words_lat, n, dirichlet) : 0;
}
static int upload_tile_words(sem_mesh *m) {
  const TileSet &ts = m->tiles;
  if (!m->d_tile_words) SEM_TRY(dalloc(&m->d_tile_words, ts.words.size(), &m->tile_bytes));
  if (!m->d_tile_slot) SEM_TRY(dalloc(&m->d_tile_slot, m->tile_slots.size(), &m->tile_bytes));
  const bool dir = std::any_of(m->dirichlet.begin(), m->dirichlet.end(), [](uint8_t d) { return d != 0; });
  for (uint32_t &w : m->tile_slots) w = dir ? w | kSlotDirichlet : w & ~kSlotDirichlet;
  HIPCHK(hipMemcpyAsync(m->d_tile_slot, m->tile_slots.data(), m->tile_slots.size() * 4, hipMemcpyHostToDevice, m->stream));
  HIPCHK(hipMemcpyAsync(m->d_tile_words, ts.words.data(), ts.words.size() * 4, hipMemcpyHostToDevice, m->stream));
  HIPCHK(hipStreamSynchronize(m->stream));
  return 0;
}

// Where the tile kernel finds each word: its slot in the LDS lattice and, in
// the high half, the place of its total after the face passes -- in the
// results of the element of highest lattice position containing it.  Tiles of
// one extent and place in the box (inside, at a face, edge or corner) hold their
// words in the same lattice order and share one table, which stays in the
// caches: 4 bytes per slot less to read per tile and launch (one acoustic
// shot, 10 of 73 KB at 4x4x2 tiles, 9 of 50 KB at 16x8).  Row r of slot_of, the
// slots of the words in order, belongs to tile tiles[r] (empty: r itself).
static std::vector<uint32_t> number_tile_slots(const sem_mesh *m, const std::vector<uint16_t> &slot_of,
                                               const std::vector<int32_t> &tiles, std::vector<int32_t> &table) {
  const TileSet &ts = m->tiles;
  const int64_t rows = tiles.empty() ? ts.ntiles : (int64_t)tiles.size();
  table.resize(rows);
  const TileKernelInfo k = tile_kernel_info(m->dim, m->order, m->physics, ts.T);
  const int N = m->order, n = m->n, LX = ts.T[0] * N + 1, LY = ts.T[1] * N + 1;
  const int64_t NTL = ts.slots_per_tile;
  std::vector<uint32_t> slot;
  std::map<std::tuple<int, int, int>, std::vector<int32_t>> tables;  // per tile extent: the first row of each table
  for (int64_t t = 0; t < rows; ++t) {
    const TileInfo &ti = ts.info[tiles.empty() ? t : tiles[t]];
    std::vector<int32_t> &seen = tables[std::make_tuple(ti.ex, ti.ey, ti.ez)];
    const uint16_t *of = &slot_of[t * NTL];
    const auto same = [&](int32_t u) { return std::equal(of, of + NTL, &slot_of[u * NTL]); };
    const auto it = std::find_if(seen.begin(), seen.end(), same);
    if (it != seen.end()) {
      table[t] = table[*it];
      continue;
    }
    seen.push_back((int32_t)t);
    table[t] = (int32_t)(slot.size() / NTL);
    for (int64_t i = 0; i < NTL; ++i) {
      const int l = of[i], x = l % LX, y = (l / LX) % LY, z = l / (LX * LY);
      const int a = std::min(x / N, ti.ex - 1), b = std::min(y / N, ti.ey - 1), c = std::min(z / N, ti.ez - 1);
      const int e = a + ts.T[0] * (b + ts.T[1] * c);
      const int p = (x - a * N) + n * ((y - b * N) + n * (z - c * N));
      // (padding words lie outside the mesh: place 0, never used)
      const bool in = x <= ti.ex * N && y <= ti.ey * N && z <= ti.ez * N;
      slot.push_back((uint32_t)(x + k.lxp * y + k.lxyp * z) | (in ? (uint32_t)(e * k.elem_stride + p) << 16 : 0u));
    }
  }
  return slot;
}

// Numbering and words of the colour launches, built once.
int sem::ensure_colour_tiles(sem_mesh *m) {
  std::lock_guard<std::mutex> lock(mesh_lazy);
  ColourTiles &ct = m->ctiles;
  if (ct.valid || ct.unfit) return 0;
  const TileSet &ts = m->tiles;
  const TileKernelInfo k = tile_kernel_info(m->dim, m->order, m->physics, ts.T);
  const int ntl = (int)ts.slots_per_tile;
  const size_t nwords = (size_t)ts.ntiles * ntl;
  ColourTables c;
  colour_tile_tables(m, c);
  std::vector<int32_t> row;
  const std::vector<uint32_t> slots = number_tile_slots(m, c.slot_of, c.example, row);
  std::vector<ColourTile> tiles(ts.ntiles);
  ct.table.resize(ts.ntiles);
  for (int64_t t = 0; t < ts.ntiles; ++t) {
    ct.table[t] = row[c.type[t]];
    tiles[t] = ColourTile{c.type[t], ts.info[t].slots, ts.info[t].nval, c.first[t]};
  }
  size_t bytes = 0;
  int32_t bad = 0;
  TempSpace temp;  // tiles, tables in both orders, flag
  int rc = temp.get(m, tiles.size() * sizeof(ColourTile) + 8 * c.words.size() + 4);
  ColourTile *d_tiles = reinterpret_cast<ColourTile *>(temp.p);
  uint32_t *d_entries = reinterpret_cast<uint32_t *>(d_tiles + tiles.size()), *d_lat = d_entries + c.words.size();
  int32_t *d_bad = reinterpret_cast<int32_t *>(d_lat + c.lat.size());
  auto up = [&](void *dst, const auto &v) {
    if (!rc) rc = hip_check(hipMemcpyAsync(dst, v.data(), v.size() * sizeof(v[0]), hipMemcpyHostToDevice, m->stream), "upload");
  };
  if (!rc) rc = dalloc(&ct.d_words, nwords, &bytes);
  if (!rc && m->physics == SEM_ACOUSTIC) rc = dalloc(&ct.d_words_lat, nwords, &bytes);
  if (!rc) rc = dalloc(&ct.d_slot, slots.size(), &bytes);
  if (!rc) rc = dalloc(&ct.d_to_int, (size_t)m->G, &bytes);
  if (!rc) rc = dalloc(&ct.d_mi, (size_t)m->G, &bytes);
  up(d_tiles, tiles);
  up(d_entries, c.words);
  up(d_lat, c.lat);
  up(ct.d_slot, slots);
  const int nx = ts.nt[0], nxy = ts.nt[0] * ts.nt[1];
  int32_t *number = reinterpret_cast<int32_t *>(ct.d_mi);  // until the masses come
  if (!rc) rc = launch_fill_i32(1, d_bad, 0, m->stream);
  if (!rc) rc = launch_colour_words(ts.ntiles, ntl, nx, nxy, d_tiles, d_entries, ct.d_words, m->stream);
  if (!rc && ct.d_words_lat) rc = launch_colour_words(ts.ntiles, ntl, nx, nxy, d_tiles, d_lat, ct.d_words_lat, m->stream);
  if (!rc)
    rc = launch_colour_numbers(ts.ntiles, ntl, ts.T[0] * m->order + 1, ts.T[1] * m->order + 1, k.lxp, k.lxyp, d_tiles, d_lat,
                               m->d_tile_words, m->d_tile_slot, (uint32_t)ts.nown, (uint32_t)(ts.nown + ts.sh_n[0]),
                               (uint32_t)(ts.nown + ts.sh_n[0] + ts.sh_n[1]), number, d_bad, m->stream);
  if (!rc) rc = hip_check(hipMemcpyAsync(&bad, d_bad, 4, hipMemcpyDeviceToHost, m->stream), "copy");
  if (!rc) rc = hip_check(hipStreamSynchronize(m->stream), "sync");
  if (rc || bad) {
    free_colour_tiles(m);
    ct.unfit = !rc;
    return rc;
  }
  ct.to_internal.resize(m->G);
  rc = launch_compose_i32(m->G, m->d_to_int, number, ct.d_to_int, m->stream);
  if (!rc) rc = launch_permute_f32(m->G, ct.d_to_int, m->d_mi, ct.d_mi, m->stream);
  if (!rc) rc = hip_check(hipMemcpyAsync(ct.to_internal.data(), ct.d_to_int, (size_t)m->G * 4, hipMemcpyDeviceToHost, m->stream), "copy");
  if (!rc) rc = hip_check(hipStreamSynchronize(m->stream), "sync");
  if (!rc && !m->dirichlet.empty()) rc = reflag_colour_tiles(m);
  if (rc) {
    free_colour_tiles(m);
    return rc;
  }
  ct.valid = true;
  m->tile_bytes += bytes;
  m->bytes += bytes;
  return 0;
}

static void free_colour_tiles(sem_mesh *m) {
  ColourTiles &ct = m->ctiles;
  dfree(ct.d_words);
  dfree(ct.d_words_lat);
  dfree(ct.d_slot);
  dfree(ct.d_mi);
  dfree(ct.d_to_int);
  ct = ColourTiles();
}

void sem::free_tiles(sem_mesh *m) {
  free_colour_tiles(m);
  dfree(m->d_tile_words);
  dfree(m->d_tile_slot);
  dfree(m->d_sh_part);
  dfree(m->d_telem);
  dfree(m->d_mi_int);
  dfree(m->d_to_int);
  m->bytes -= std::min(m->bytes, m->tile_bytes);
  m->tile_bytes = 0;
  m->tiles = TileSet();
}

// Builds and uploads the tile path of an affine, logically Cartesian mesh,
// with the given tile shape or (shape null) the first of the preference list.
int sem::setup_tiles(sem_mesh *m, const int *shape) {
  free_tiles(m);
  const char *off = getenv("SEM_NO_TILES");
  if (!m->affine || (off && off[0] == '1')) return 0;
  int T[3];
  if (shape) {
    T[0] = shape[0]; T[1] = shape[1]; T[2] = m->dim == 3 ? shape[2] : 1;
    if (tile_kernel_info(m->dim, m->order, m->physics, T).lds_bytes == 0) {
      set_error("tile shape not compiled for this order and physics");
      return -1;
    }
  } else if (!pick_tile(m->dim, m->order, m->physics, T)) {
    return 0;
  }
  if (build_tiles(m, T[0], T[1], T[2], m->tiles) != 0) {
    m->tiles = TileSet();
    return 0;  // not eligible: the element kernel is used
  }
  const int rc = upload_tiles(m);
  m->bytes += m->tile_bytes;
  return rc;
}

int sem::upload_tiles(sem_mesh *m) {
  TileSet &ts = m->tiles;
  const int dim = m->dim, nv = m->nv, npar = ref_npar(dim, m->physics), kp = kernel_npar(dim, m->physics);
  // padded tile element order (padding repeats element 0; never read)
  const int64_t E = (int64_t)ts.elem_order.size();
  {
    std::vector<int32_t> table;
    m->tile_slots = number_tile_slots(m, ts.slot_of, {}, table);
    for (int64_t t = 0; t < ts.ntiles; ++t) ts.info[t].slots = table[t];
  }
  SEM_TRY(upload_tile_words(m));
  SEM_TRY(dalloc(&m->d_sh_part, ts.sh_part.size(), &m->tile_bytes));
  if (!ts.sh_part.empty())
    HIPCHK(hipMemcpyAsync(m->d_sh_part, ts.sh_part.data(), ts.sh_part.size() * 4, hipMemcpyHostToDevice, m->stream));
  // FP64 vertices in tile element order -> affine factors on the device
  std::vector<double> tv(E * nv * dim);
  std::vector<float> tp(E * nv * kp);
  for (int64_t i = 0; i < E; ++i) {
    const int64_t e = std::max<int32_t>(ts.elem_order[i], 0);
    std::copy_n(&m->vtx[e * nv * dim], nv * dim, &tv[i * nv * dim]);
    for (int k = 0; k < nv; ++k) {
      const double *src = &m->vpar[(e * nv + k) * npar];
      float *dst = &tp[(i * nv + k) * kp];
      if (m->physics == SEM_ACOUSTIC) dst[0] = (float)src[0];
      else if (dim == 2) for (int q = 0; q < 4; ++q) dst[q] = (float)src[1 + q];
      else for (int q = 0; q < 6; ++q) dst[q] = (float)src[q];
    }
  }
  // affine factors (FP64 on the device, FP32 out), then one array of
  // [affine factors | vertex material] per element for the tile kernel
  const int ng = affine_geo_count(dim, m->physics), ned = ng + nv * kp;
  double *d_tv = nullptr;
  float *d_tg = nullptr;
  std::vector<float> tg(E * ng), te(E * ned);
  SEM_TRY(dalloc(&d_tv, tv.size()));
  int rc = hip_check(hipMemcpyAsync(d_tv, tv.data(), tv.size() * 8, hipMemcpyHostToDevice, m->stream), "upload");
  if (!rc) rc = dalloc(&d_tg, tg.size());
  if (!rc) rc = launch_affine_geometry(dim, m->physics, E, d_tv, d_tg, m->stream);
  if (!rc) rc = hip_check(hipMemcpyAsync(tg.data(), d_tg, tg.size() * 4, hipMemcpyDeviceToHost, m->stream), "download");
  if (!rc) rc = hip_check(hipStreamSynchronize(m->stream), "sync");
  if (!rc) {
    // off-diagonal entries: J^-1 row-major (elastic), packed symmetric G (acoustic)
    static const int off_e2[] = {1, 2}, off_e3[] = {1, 2, 3, 5, 6, 7}, off_a2[] = {1}, off_a3[] = {1, 2, 4};
    const int *off = m->physics == SEM_ACOUSTIC ? (dim == 2 ? off_a2 : off_a3) : (dim == 2 ? off_e2 : off_e3);
    const int noff = m->physics == SEM_ACOUSTIC ? (dim == 2 ? 1 : 3) : (dim == 2 ? 2 : 6);
    bool diag = true;
    for (int64_t i = 0; i < E && diag; ++i)
      for (int k = 0; k < noff; ++k) diag = diag && tg[i * ng + off[k]] == 0.f;
    m->tile_diag = diag;
    for (int64_t i = 0; i < E; ++i) {
      std::copy_n(&tg[i * ng], ng, &te[i * ned]);
      std::copy_n(&tp[i * nv * kp], nv * kp, &te[i * ned + ng]);
    }
    rc = dalloc(&m->d_telem, te.size(), &m->tile_bytes);
  }
  if (!rc) rc = hip_check(hipMemcpyAsync(m->d_telem, te.data(), te.size() * 4, hipMemcpyHostToDevice, m->stream), "upload");
  dfree(d_tg);
  // inverse mass in the internal numbering
  if (!rc) rc = dalloc(&m->d_to_int, (size_t)m->G, &m->tile_bytes);
  if (!rc) rc = hip_check(hipMemcpyAsync(m->d_to_int, ts.to_internal.data(), m->G * 4, hipMemcpyHostToDevice, m->stream), "upload");
  if (!rc) rc = dalloc(&m->d_mi_int, (size_t)m->G, &m->tile_bytes);
  if (!rc) rc = launch_permute_f32(m->G, m->d_to_int, m->d_mi, m->d_mi_int, m->stream);
  if (!rc) rc = hip_check(hipStreamSynchronize(m->stream), "sync");
  dfree(d_tv);
  return rc;
}

static void mesh_free(sem_mesh *m) {
  if (!m) return;
  (void)hipSetDevice(m->device);
  if (m->stream) (void)hipStreamSynchronize(m->stream);
  dfree(m->d_conn);
  dfree(m->d_geo_e);
  dfree(m->d_par_e);
  dfree(m->d_geo_p);
  dfree(m->d_mi);
  dfree(m->d_vtx);
  dfree(m->d_vpar);
  dfree(m->d_tile_words);
  dfree(m->d_tile_slot);
  dfree(m->d_sh_part);
  dfree(m->d_epos);
  dfree(m->d_apply_buf);
  dfree(m->d_temp);
  dfree(m->d_telem);
  dfree(m->d_mi_int);
  dfree(m->d_to_int);
  free_colour_tiles(m);
  if (m->stream) (void)hipStreamDestroy(m->stream);
  delete m;
}

// ====================================================================== C ABI
extern "C" {

const char *sem_last_error(void) { return g_error.c_str(); }

int sem_device_count(int *count) {
  int n = 0;
  hipError_t e = hipGetDeviceCount(&n);
  *count = e == hipSuccess ? n : 0;
  return 0;
}

int64_t sem_reference_step_count(double duration, double dt, double *dt_out) {
  int64_t m = (int64_t)std::ceil(duration / dt);
  double h = duration / (double)m;
  if (dt_out) *dt_out = h;
  double t = 0;
  int64_t count = 0;
  while (t < duration) {
    t += h;
    ++count;
  }
  return count;
}

int sem_topology_build(int dim, int order, int64_t E, int64_t V, const int32_t *cells,
                       int32_t *conn, int32_t *colour, int64_t *info) {
  if (order < 1 || order > (dim == 2 ? kMaxOrder2D : kMaxOrder3D)) {
    set_error("Polynomial order " + std::to_string(order) + " not supported");
    return -1;
  }
  Topology T;
  SEM_TRY(build_topology(dim, order, E, V, cells, T));
  std::vector<int32_t> col;
  SEM_TRY(colour_elements(dim, E, V, cells, col));
  if (conn) std::copy(T.conn.begin(), T.conn.end(), conn);
  if (colour) std::copy(col.begin(), col.end(), colour);
  if (info) {
    info[0] = T.G;
    info[1] = E ? 1 + *std::max_element(col.begin(), col.end()) : 0;
    info[2] = T.NF;
    info[3] = T.NEd;
  }
  return 0;
}

int sem_mesh_create(sem_mesh **out, int device, int dim, int order, int physics, int64_t E,
                    int64_t V, const int32_t *cells, const double *coords, const double *vpar,
                    int quirks) {
  *out = nullptr;
  if (dim != 2 && dim != 3) { set_error("dim must be 2 or 3"); return -1; }
  if (physics != SEM_ACOUSTIC && physics != SEM_ELASTIC) { set_error("physics"); return -1; }
  if (order < 1 || order > (dim == 2 ? kMaxOrder2D : kMaxOrder3D)) {
    set_error("Polynomial order " + std::to_string(order) + " not supported");
    return -1;
  }
  if (E <= 0 || V <= 0 || !cells || !coords || !vpar) { set_error("empty mesh"); return -1; }
  SEM_TRY(set_device(device));
  auto *m = new sem_mesh();
  m->device = device;
  m->dim = dim;
  m->order = order;
  m->n = order + 1;
  m->nd = dim == 2 ? m->n * m->n : m->n * m->n * m->n;
  m->physics = physics;
  m->c = physics == SEM_ACOUSTIC ? 1 : dim;
  m->nv = dim == 2 ? 4 : 8;
  m->quirks = quirks;
  m->E = E;
  m->V = V;
  const int nv = m->nv, npar = ref_npar(dim, physics);
  int rc = 0;
  auto fail = [&](int r) { mesh_free(m); return r; };
  Topology T;
  if ((rc = build_topology(dim, order, E, V, cells, T))) return fail(rc);
  m->G = T.G;
  m->conn = std::move(T.conn);
  if ((rc = colour_elements(dim, E, V, cells, m->colour))) return fail(rc);
  m->ncol = 1 + *std::max_element(m->colour.begin(), m->colour.end());
  // sorted order: by colour, then element index
  m->col_start.assign(m->ncol + 1, 0);
  for (int64_t e = 0; e < E; ++e) ++m->col_start[m->colour[e] + 1];
  for (int c = 0; c < m->ncol; ++c) m->col_start[c + 1] += m->col_start[c];
  m->perm.resize(E);
  m->inv_perm.resize(E);
  {
    std::vector<int64_t> cur(m->col_start.begin(), m->col_start.end() - 1);
    for (int64_t e = 0; e < E; ++e) {
      int64_t sp = cur[m->colour[e]]++;
      m->perm[sp] = (int32_t)e;
      m->inv_perm[e] = (int32_t)sp;
    }
  }
  // host geometry (original order), validity and affinity
  m->vtx.resize(E * nv * dim);
  m->bbox.resize(E * 2 * dim);
  m->vpar.assign(vpar, vpar + E * nv * npar);
  bool affine = true;
  for (int64_t e = 0; e < E; ++e) {
    double *vx = &m->vtx[e * nv * dim];
    for (int k = 0; k < nv; ++k)
      for (int a = 0; a < dim; ++a) vx[k * dim + a] = coords[(int64_t)cells[e * nv + k] * dim + a];
    double J[9], ref[3] = {0, 0, 0};
    if (jacobian(dim, vx, ref, J) <= 0) {
      set_error("element " + std::to_string(e) + " has det J <= 0");
      return fail(-1);
    }
    for (int a = 0; a < dim; ++a) {
      double lo = vx[a], hi = vx[a];
      for (int k = 1; k < nv; ++k) {
        lo = std::min(lo, vx[k * dim + a]);
        hi = std::max(hi, vx[k * dim + a]);
      }
      m->bbox[e * 2 * dim + a] = lo;
      m->bbox[e * 2 * dim + dim + a] = hi;
    }
    if (affine && !is_affine(dim, vx)) affine = false;
  }
  m->affine = affine;
  bin_elements(m->bins, dim, E, m->bbox.data());
  // device upload (sorted order)
  if ((rc = hip_check(hipStreamCreateWithFlags(&m->stream, hipStreamNonBlocking), "stream"))) return fail(rc);
  const size_t mass_bytes = 8 * ((size_t)E * m->nd + (size_t)m->G);  // the largest of the temporaries
  if (mass_bytes > kMinShared) {
    if ((rc = dalloc(&m->d_temp, mass_bytes))) return fail(rc);
    m->temp_bytes = mass_bytes;
  }
  if ((rc = upload_conn(m))) return fail(rc);
  {
    std::vector<double> sv(E * nv * dim), sp(E * nv * npar);
    for (int64_t s = 0; s < E; ++s) {
      int64_t e = m->perm[s];
      std::copy_n(&m->vtx[e * nv * dim], nv * dim, &sv[s * nv * dim]);
      std::copy_n(&m->vpar[e * nv * npar], nv * npar, &sp[s * nv * npar]);
    }
    if ((rc = dalloc(&m->d_vtx, sv.size(), &m->bytes))) return fail(rc);
    if ((rc = dalloc(&m->d_vpar, sp.size(), &m->bytes))) return fail(rc);
    if ((rc = hip_check(hipMemcpyAsync(m->d_vtx, sv.data(), sv.size() * 8, hipMemcpyHostToDevice, m->stream), "upload"))) return fail(rc);
    if ((rc = hip_check(hipMemcpyAsync(m->d_vpar, sp.data(), sp.size() * 8, hipMemcpyHostToDevice, m->stream), "upload"))) return fail(rc);
    // kernel material set (FP32 vertex values)
    const int kp = kernel_npar(dim, physics);
    std::vector<float> pe(E * nv * kp);
    for (int64_t s = 0; s < E; ++s)
      for (int k = 0; k < nv; ++k) {
        const double *src = &sp[(s * nv + k) * npar];
        float *dst = &pe[(s * nv + k) * kp];
        if (physics == SEM_ACOUSTIC) dst[0] = (float)src[0];
        else if (dim == 2) for (int q = 0; q < 4; ++q) dst[q] = (float)src[1 + q];  // C11 C13 C33 C55
        else for (int q = 0; q < 6; ++q) dst[q] = (float)src[q];
      }
    if ((rc = dalloc(&m->d_par_e, pe.size(), &m->bytes))) return fail(rc);
    if ((rc = hip_check(hipMemcpyAsync(m->d_par_e, pe.data(), pe.size() * 4, hipMemcpyHostToDevice, m->stream), "upload"))) return fail(rc);
    if ((rc = hip_check(hipStreamSynchronize(m->stream), "sync"))) return fail(rc);
  }
  if (affine) {
    if ((rc = dalloc(&m->d_geo_e, (size_t)E * affine_geo_count(dim, physics), &m->bytes))) return fail(rc);
    if ((rc = launch_affine_geometry(dim, physics, E, m->d_vtx, m->d_geo_e, m->stream))) return fail(rc);
  }
  // FP64 mass: element contributions, colour-ordered assembly, reciprocal
  {
    TempSpace temp;
    if ((rc = temp.get(m, mass_bytes))) return fail(rc);
    double *me = reinterpret_cast<double *>(temp.p), *M = me + (size_t)E * m->nd;
    rc = launch_point_geometry(dim, order, physics, pointwise_mode(m), E, m->d_vtx, m->d_vpar, npar,
                               nullptr, me, m->stream);
    if (!rc) rc = launch_fill_f64(m->G, M, 0.0, m->stream);
    for (int c = 0; c < m->ncol && !rc; ++c)
      rc = launch_mass_scatter(m->col_start[c], m->col_start[c + 1] - m->col_start[c], m->nd,
                               m->d_conn, me, M, m->stream);
    if (!rc) rc = dalloc(&m->d_mi, (size_t)m->G, &m->bytes);
    if (!rc) rc = launch_reciprocal(m->G, M, m->d_mi, m->stream);
    if (!rc) rc = hip_check(hipStreamSynchronize(m->stream), "mass");
    if (rc) return fail(rc);
  }
  if (!affine && (rc = ensure_pointwise(m)) == -3) {  // the largest array: without the temporaries
    m->temp_bytes = 0;
    dfree(m->d_temp);
    rc = ensure_pointwise(m);
  }
  if (rc) return fail(rc);
  // what it keeps only makes the allocation-free operator faster: without the
  // memory for it the operator runs colour by colour
  if (setup_apply(m)) (void)hipGetLastError();
  m->temp_bytes = 0;
  dfree(m->d_temp);
  if ((rc = setup_tiles(m, nullptr))) return fail(rc);
  *out = m;
  return 0;
}

int sem_mesh_destroy(sem_mesh *m) {
  mesh_free(m);
  return 0;
}

int sem_mesh_info(const sem_mesh *m, int64_t *info) {
  info[0] = m->E; info[1] = m->G; info[2] = m->ncol; info[3] = m->c;
  info[4] = m->nd; info[5] = m->affine; info[6] = (int64_t)m->bytes; info[7] = m->dim;
  info[8] = m->tiles.valid ? m->tiles.ntiles : 0;
  info[9] = m->tiles.valid ? m->tiles.T[0] * 10000 + m->tiles.T[1] * 100 + m->tiles.T[2] : 0;
  // tile path traffic counts: lattice slots loaded, slots on the mesh, partial
  // results of shared nodes (each written once and read once)
  int64_t valid = 0;
  for (const TileInfo &ti : m->tiles.info) valid += ti.nval;
  info[10] = m->tiles.valid ? m->tiles.total_slots : 0;
  info[11] = valid;
  info[12] = info[13] = m->tiles.nparts;
  info[14] = m->tiles.valid ? m->tiles.elems_per_tile : 0;
  info[15] = m->tiles.valid && m->tile_diag;
  return 0;
}

int sem_mesh_get_conn(const sem_mesh *m, int32_t *conn) {
  std::copy(m->conn.begin(), m->conn.end(), conn);
  return 0;
}

int sem_mesh_get_colours(const sem_mesh *m, int32_t *colour) {
  std::copy(m->colour.begin(), m->colour.end(), colour);
  return 0;
}

int sem_mesh_get_inverse_mass(const sem_mesh *m, float *mi) {
  HIPCHK(hipSetDevice(m->device));
  HIPCHK(hipMemcpy(mi, m->d_mi, m->G * sizeof(float), hipMemcpyDeviceToHost));
  return 0;
}

int sem_mesh_get_node_coords(const sem_mesh *m, double *xyz) {
  Gll g = make_gll(m->order);
  const int dim = m->dim, n = m->n;
  for (int64_t e = 0; e < m->E; ++e) {
    const double *vx = &m->vtx[e * m->nv * dim];
    for (int p = 0; p < m->nd; ++p) {
      double ref[3] = {g.xi[p % n], g.xi[(p / n) % n], dim == 3 ? g.xi[p / (n * n)] : 0.0};
      double w[8];
      p1_weights(dim, ref, w);
      int32_t gid = m->conn[e * m->nd + p];
      for (int a = 0; a < dim; ++a) {
        double s = 0;
        for (int k = 0; k < m->nv; ++k) s += w[k] * vx[k * dim + a];
        xyz[(int64_t)gid * dim + a] = s;
      }
    }
  }
  return 0;
}

int sem_mesh_set_dirichlet(sem_mesh *m, const uint8_t *mask) {
  HIPCHK(hipSetDevice(m->device));
  m->dirichlet.assign(mask, mask + m->G);
  SEM_TRY(upload_conn(m));
  if (m->tiles.valid) {
    TileSet &ts = m->tiles;
    std::vector<uint8_t> dint(m->G, 0);
    for (int64_t g = 0; g < m->G; ++g) dint[ts.to_internal[g]] = m->dirichlet[g];
    for (auto &w : ts.words) {
      if (w == kSlotEmpty) continue;
      uint32_t node = w & kNodeMask;
      w = node | (dint[node] ? kFlagDirichlet : 0u);
    }
    SEM_TRY(upload_tile_words(m));
    if (m->ctiles.valid) SEM_TRY(reflag_colour_tiles(m));
  }
  return 0;
}

int sem_mesh_check_colouring(sem_mesh *m, int64_t *violations) {
  HIPCHK(hipSetDevice(m->device));
  int32_t *hits = nullptr;
  unsigned long long *viol = nullptr;
  SEM_TRY(dalloc(&hits, (size_t)m->G));
  int rc = dalloc(&viol, 1);
  if (!rc) rc = launch_fill_i32(m->G, hits, 0, m->stream);
  if (!rc) rc = hip_check(hipMemsetAsync(viol, 0, sizeof(unsigned long long), m->stream), "memset");
  for (int c = 0; c < m->ncol && !rc; ++c) {
    rc = launch_colour_touch(m->col_start[c], m->col_start[c + 1] - m->col_start[c], m->nd,
                             m->d_conn, hits, m->stream);
    if (!rc) rc = launch_colour_count(m->G, hits, viol, m->stream);
  }
  unsigned long long h = 0;
  if (!rc) rc = hip_check(hipMemcpyAsync(&h, viol, sizeof h, hipMemcpyDeviceToHost, m->stream), "copy");
  if (!rc) rc = hip_check(hipStreamSynchronize(m->stream), "sync");
  dfree(hits);
  dfree(viol);
  *violations = (int64_t)h;
  return rc;
}

}  // extern "C"

// ====================================================================== sources/receivers (host, FP64)
// The first element (in the caller's order) whose closed hull holds the point:
// the elements whose bounding box holds it are all listed, ascending, in the
// point's bin.  (A scan over every element took 10 us a point at 500^2 quads
// and 20-200 us at 64^3 hexes, twice per source and receiver.)
int sem::locate(const sem_mesh *m, const double *pt, int64_t *elem, double *ref) {
  const int dim = m->dim;
  const ElementBins &B = m->bins;
  bool nan = false;  // in no bin and no box: every element is asked
  for (int a = 0; a < dim; ++a) nan = nan || std::isnan(pt[a]);
  const int64_t bin = nan ? 0 : bin_of(B, dim, pt);
  const int64_t begin = nan ? 0 : B.start[bin], end = nan ? m->E : B.start[bin + 1];
  for (int64_t i = begin; i < end; ++i) {
    const int64_t e = nan ? i : B.elem[i];
    const double *bb = &m->bbox[e * 2 * dim];
    bool out = false;
    for (int a = 0; a < dim; ++a) out = out || pt[a] < bb[a] || pt[a] > bb[dim + a];
    if (out) continue;  // a convex element lies inside its bounding box
    const double *vx = &m->vtx[e * m->nv * dim];
    int in = check_hull(dim, pt, vx);
    if (in < 0) { set_error("poorly behaved element"); return -1; }
    if (in) {
      if (inverse_map(dim, pt, vx, ref)) {
        set_error("inverseCoordinateTransform failed to converge");
        return -1;
      }
      *elem = e;
      return 0;
    }
  }
  set_error("point outside the mesh: source or receiver not added");
  return -1;
}

// Nodal load per unit source-time function, nd x c column-major (FP64).
int sem::source_load(const sem_mesh *m, const SrcSpec &s, int64_t *elem, std::vector<double> &load) {
  double ref[3] = {0, 0, 0};
  SEM_TRY(locate(m, s.loc, elem, ref));
  const int dim = m->dim, n = m->n, nd = m->nd, c = m->c;
  const double *vx = &m->vtx[*elem * m->nv * dim];
  Gll g = make_gll(m->order);
  double l[3][kMaxN], dl[3][kMaxN];
  for (int a = 0; a < dim; ++a) {
    lagrange(g, ref[a], l[a]);
    lagrange_deriv(g, ref[a], dl[a]);
  }
  load.assign((size_t)nd * c, 0.0);
  if (s.kind == 0 || s.kind == 2) {
    const bool e3d_quirk = dim == 3 && m->physics == SEM_ELASTIC && (m->quirks & SEM_QUIRK_E3D_SOURCE);
    for (int p = 0; p < nd; ++p) {
      int P[3] = {p % n, (p / n) % n, dim == 3 ? p / (n * n) : 0};
      double lp = 1.0, wq = 1.0;
      for (int a = 0; a < dim; ++a) {
        lp *= l[a][P[a]];
        wq *= g.w[P[a]];
      }
      // getDeltaFunctionCoefficients divides by w detJ at the node; the
      // test-and-integrate of Scalar/Elastic2D multiplies it back; Elastic3D's
      // source term skips it (Elastic3D.cpp:126-133).
      double r3[3] = {g.xi[P[0]], g.xi[P[1]], dim == 3 ? g.xi[P[2]] : 0.0}, J[9];
      double det = jacobian(dim, vx, r3, J);
      double delta = lp / (wq * det);
      double val = e3d_quirk ? delta : delta * det * wq;
      for (int k = 0; k < c; ++k) load[(size_t)k * nd + p] = val * s.dir[k];
    }
  } else {
    if (m->physics != SEM_ELASTIC) { set_error("moment tensor needs elastic physics"); return -1; }
    double J[9], inv[9];
    jacobian(dim, vx, ref, J);
    invert(dim, J, inv);
    for (int p = 0; p < nd; ++p) {
      int P[3] = {p % n, (p / n) % n, dim == 3 ? p / (n * n) : 0};
      double gr[3];
      for (int a = 0; a < dim; ++a) {
        double v = dl[a][P[a]];
        for (int b = 0; b < dim; ++b)
          if (b != a) v *= l[b][P[b]];
        gr[a] = v;
      }
      double gx[3];
      for (int a = 0; a < dim; ++a) {
        double v = 0;
        for (int b = 0; b < dim; ++b) v += inv[a * dim + b] * gr[b];
        gx[a] = v;
      }
      for (int i = 0; i < dim; ++i) {
        double v = 0;
        for (int j = 0; j < dim; ++j) v += s.M[i * dim + j] * gx[j];
        load[(size_t)i * nd + p] = -v;
      }
    }
  }
  return 0;
}

double sem::ricker(double t, double amp, double f0, double t0) {
  const double factor = M_PI * M_PI * f0 * f0 * (t - t0) * (t - t0);
  return amp * ((1 - 2 * factor) * std::exp(-1 * factor));
}

