// Tiling of logically Cartesian meshes for the tile kernel.
//
// A tile is a box of Tx x Ty (x Tz) elements of the element lattice.  Its
// nodes form an (Tx N + 1) x (Ty N + 1) (x (Tz N + 1)) node lattice that the
// tile kernel stages in LDS; element (a,b,c) of the tile, node (i,j,k) sits
// at lattice slot (aN+i) + Lx ((bN+j) + Ly (cN+k)).  Tiles at the mesh edge
// keep the full box: their missing elements and slots are padding.  The
// slot -> global DOF table is filled from the DMPlex-compatible gather map
// and checked for consistency, so the tile path is used only when every
// element's reference axes follow the lattice axes.
//
// Tiles are coloured by lattice parity (2^dim colours; tiles of one colour
// share no node).  A node lies in one tile alone or is shared by 2, 4 or 8
// tiles (a tile face, edge or corner).  Nodes are renumbered: first those in
// one tile alone, tile by tile in slot order, so that the state a tile
// updates is one contiguous range; then the shared ones, class by class (2,
// 4, 8 tiles), each class by its nodes' first tile and there by face, edge or
// corner, so that the kernel that finishes them streams through every array.
// A tile's partial result for a shared node goes to copy k of the node's
// class, k the rank of the tile's colour among the node's tiles (the order in
// which the partial results are summed): part = base + k n_class + position
// in the class.  The words of a tile (node | Dirichlet flag) hold its own nodes first,
// then the shared ones, each part in the order of its nodes, each word with
// its lattice slot (slot_of); sh_part holds the shared words' partial-result
// positions.
#include <algorithm>
#include <array>
#include <cmath>
#include <cstring>
#include <map>
#include <tuple>

#include "sem_internal.h"

namespace sem {

int build_tiles(sem_mesh *m, int Tx, int Ty, int Tz, TileSet &ts) {
  ts = TileSet();
  const int dim = m->dim, N = m->order, n = m->n;
  const int64_t E = m->E;
  if (dim == 2) Tz = 1;
  // ---- element lattice from centroids and a common element size
  double lo[3] = {1e300, 1e300, 1e300}, h[3] = {0, 0, 0};
  for (int a = 0; a < dim; ++a) h[a] = m->bbox[dim + a] - m->bbox[a];
  for (int64_t e = 0; e < E; ++e)
    for (int a = 0; a < dim; ++a) {
      lo[a] = std::min(lo[a], m->bbox[e * 2 * dim + a]);
      double he = m->bbox[e * 2 * dim + dim + a] - m->bbox[e * 2 * dim + a];
      if (std::fabs(he - h[a]) > 1e-9 * std::max(1.0, std::fabs(h[a]))) return 1;  // not uniform
    }
  int64_t nel[3] = {1, 1, 1};
  std::vector<int64_t> lat(E * 3, 0);
  for (int64_t e = 0; e < E; ++e)
    for (int a = 0; a < dim; ++a) {
      double c = 0.5 * (m->bbox[e * 2 * dim + a] + m->bbox[e * 2 * dim + dim + a]);
      double f = (c - lo[a]) / h[a] - 0.5;
      int64_t k = (int64_t)std::llround(f);
      if (std::fabs(f - k) > 1e-6 || k < 0) return 1;
      lat[e * 3 + a] = k;
      nel[a] = std::max(nel[a], k + 1);
    }
  if (nel[0] * nel[1] * nel[2] != E) return 1;
  std::vector<int32_t> at(E, -1);  // lattice cell -> element
  for (int64_t e = 0; e < E; ++e) {
    int64_t id = lat[e * 3] + nel[0] * (lat[e * 3 + 1] + nel[1] * lat[e * 3 + 2]);
    if (at[id] >= 0) return 1;
    at[id] = (int32_t)e;
  }
  const int T[3] = {Tx, Ty, Tz};
  const int LX = Tx * N + 1, LY = Ty * N + 1, LZ = dim == 3 ? Tz * N + 1 : 1;
  const int64_t NTL = (int64_t)LX * LY * LZ;
  const int EPT = Tx * Ty * Tz;
  int64_t nt[3];
  for (int a = 0; a < 3; ++a) nt[a] = (nel[a] + T[a] - 1) / T[a];
  const int64_t ntiles = nt[0] * nt[1] * nt[2];
  if (ntiles * EPT > INT32_MAX || ntiles * NTL > ((int64_t)1 << 40)) return 1;
  ts.ntiles = ntiles;
  ts.slots_per_tile = NTL;
  ts.elems_per_tile = EPT;
  ts.total_slots = ntiles * NTL;
  ts.info.resize(ntiles);
  ts.elem_order.assign(ntiles * EPT, -1);
  // ---- per tile: element list (lattice order), slot -> PETSc node map
  std::vector<int32_t> slot_node(ntiles * NTL, -1);  // PETSc ids, -1 = padding
  for (int64_t tz = 0; tz < nt[2]; ++tz)
    for (int64_t ty = 0; ty < nt[1]; ++ty)
      for (int64_t tx = 0; tx < nt[0]; ++tx) {
        const int64_t t = tx + nt[0] * (ty + nt[1] * tz);
        TileInfo &ti = ts.info[t];
        ti.ex = (int)std::min<int64_t>(T[0], nel[0] - tx * T[0]);
        ti.ey = (int)std::min<int64_t>(T[1], nel[1] - ty * T[1]);
        ti.ez = dim == 3 ? (int)std::min<int64_t>(T[2], nel[2] - tz * T[2]) : 1;
        ti.colour = (int32_t)((tx & 1) | ((ty & 1) << 1) | (dim == 3 ? ((tz & 1) << 2) : 0));
        for (int c = 0; c < ti.ez; ++c)
          for (int b = 0; b < ti.ey; ++b)
            for (int a = 0; a < ti.ex; ++a) {
              const int64_t cell = (tx * T[0] + a) + nel[0] * ((ty * T[1] + b) + nel[1] * (tz * T[2] + c));
              const int32_t e = at[cell];
              ts.elem_order[t * EPT + a + Tx * (b + Ty * c)] = e;
              for (int p = 0; p < m->nd; ++p) {
                const int i = p % n, j = (p / n) % n, k = dim == 3 ? p / (n * n) : 0;
                const int64_t s = (a * N + i) + (int64_t)LX * ((b * N + j) + (int64_t)LY * (c * N + k));
                const int32_t g = m->conn[(int64_t)e * m->nd + p];
                int32_t &dst = slot_node[t * NTL + s];
                if (dst < 0) dst = g;
                else if (dst != g) return 1;  // reference axes do not follow the lattice
              }
            }
      }
  // ---- internal numbering (see above): own nodes tile by tile, then the
  // shared ones by class, first tile and position category (which lattice
  // faces of that tile hold it).  A first pass over the slots numbers the own
  // nodes and, within its class, each shared node.
  if (NTL > 65535) return 1;
  std::vector<int8_t> copies(m->G, 0);
  for (int64_t s = 0; s < ntiles * NTL; ++s)
    if (slot_node[s] >= 0) ++copies[slot_node[s]];
  for (int64_t g = 0; g < m->G; ++g)
    if (copies[g] != 1 && copies[g] != 2 && copies[g] != 4 && copies[g] != 8) return 1;
  const auto cls = [](int copies) { return copies == 2 ? 0 : copies == 4 ? 1 : 2; };
  std::vector<uint8_t> slot_xyz(NTL * 3);
  for (int64_t s = 0; s < NTL; ++s) {
    slot_xyz[3 * s] = (uint8_t)(s % LX);
    slot_xyz[3 * s + 1] = (uint8_t)((s / LX) % LY);
    slot_xyz[3 * s + 2] = (uint8_t)(s / ((int64_t)LX * LY));
  }
  ts.to_internal.assign(m->G, -1);
  ts.nown = 0;
  for (int q = 0; q < 3; ++q) ts.sh_n[q] = 0;
  std::vector<std::pair<int32_t, int32_t>> order;  // (category, node) of the nodes this tile is the first to hold
  for (int64_t t = 0; t < ntiles; ++t) {
    TileInfo &ti = ts.info[t];
    const int last[3] = {ti.ex * N, ti.ey * N, dim == 3 ? ti.ez * N : -1};  // last lattice index
    ti.own = (int32_t)ts.nown;
    order.clear();
    for (int64_t s = 0; s < NTL; ++s) {
      const int32_t g = slot_node[t * NTL + s];
      if (g < 0 || ts.to_internal[g] >= 0) continue;
      if (copies[g] == 1) {
        ts.to_internal[g] = (int32_t)ts.nown++;
        continue;
      }
      int cat = 0, w = 1;
      for (int a = 0; a < dim; ++a, w *= 3) {
        const int x = slot_xyz[3 * s + a];
        cat += w * (x == 0 ? 1 : x == last[a] ? 2 : 0);
      }
      order.emplace_back(cat, g);
    }
    std::stable_sort(order.begin(), order.end(), [](const auto &x, const auto &y) { return x.first < y.first; });
    for (const auto &o : order) ts.to_internal[o.second] = (int32_t)ts.sh_n[cls(copies[o.second])]++;
  }
  const int64_t nbase[3] = {ts.nown, ts.nown + ts.sh_n[0], ts.nown + ts.sh_n[0] + ts.sh_n[1]};
  const int64_t pbase[3] = {0, 2 * ts.sh_n[0], 2 * ts.sh_n[0] + 4 * ts.sh_n[1]};
  ts.nparts = pbase[2] + 8 * ts.sh_n[2];
  if (nbase[2] + ts.sh_n[2] != m->G || ts.nparts > INT32_MAX) return 1;
  for (int64_t g = 0; g < m->G; ++g)
    if (copies[g] > 1) ts.to_internal[g] += (int32_t)nbase[cls(copies[g])];
  // ---- per tile, the slots of its own nodes in the order of their internal
  // node (slot order), then the shared ones, then padding: the kernel's
  // threads take the slots in this order, so the lanes of a wave touch
  // consecutive nodes (the tile's own nodes, then the runs shared with its
  // neighbours) and every HBM access of the gather and the finish is
  // coalesced; slot_of gives each position's lattice slot.
  ts.words.assign(ntiles * NTL, kSlotEmpty);
  ts.slot_of.assign(ntiles * NTL, 0);
  int64_t nsw = 0;
  for (int64_t t = 0; t < ntiles; ++t) {
    uint32_t *words = &ts.words[t * NTL];
    uint16_t *slot = &ts.slot_of[t * NTL];
    TileInfo &ti = ts.info[t];
    order.clear();  // (internal node, slot) of the shared words
    int k = 0;
    int64_t pad = NTL;
    for (int64_t s = 0; s < NTL; ++s) {
      const int32_t g = slot_node[t * NTL + s];
      if (g < 0) {
        slot[--pad] = (uint16_t)s;
      } else if (copies[g] > 1) {
        order.emplace_back(ts.to_internal[g], (int32_t)s);
      } else {
        slot[k] = (uint16_t)s;
        words[k++] = (uint32_t)ts.to_internal[g];
      }
    }
    ti.nint = k;
    std::sort(order.begin(), order.end());
    for (const auto &o : order) {
      slot[k] = (uint16_t)o.second;
      words[k++] = (uint32_t)o.first;
    }
    ti.nval = k;
    ti.sh_off = (int32_t)nsw;
    nsw += ti.nval - ti.nint;
    if (!m->dirichlet.empty())
      for (int i = 0; i < k; ++i)
        if (m->dirichlet[slot_node[t * NTL + slot[i]]]) words[i] |= kFlagDirichlet;
  }
  // ---- partial-result positions of the shared words: copies in the order of
  // their tiles' colours
  ts.sh_part.assign(nsw, 0);
  {
    std::vector<int8_t> seen(m->G - ts.nown, 0);
    for (int c = 0; c < (1 << dim); ++c)
      for (int64_t t = 0; t < ntiles; ++t) {
        const TileInfo &ti = ts.info[t];
        if (ti.colour != c) continue;
        for (int k = ti.nint; k < ti.nval; ++k) {
          const int64_t g = ts.words[t * NTL + k] & kNodeMask;
          const int q = g < nbase[1] ? 0 : g < nbase[2] ? 1 : 2;
          ts.sh_part[ti.sh_off + k - ti.nint] = (int32_t)(pbase[q] + seen[g - ts.nown]++ * ts.sh_n[q] + (g - nbase[q]));
        }
      }
  }
  ts.elem_pos.assign(E, -1);
  for (int64_t i = 0; i < ntiles * EPT; ++i)
    if (ts.elem_order[i] >= 0) ts.elem_pos[ts.elem_order[i]] = (int32_t)i;
  ts.T[0] = Tx; ts.T[1] = Ty; ts.T[2] = Tz;
  for (int a = 0; a < 3; ++a) ts.nt[a] = (int)nt[a];
  ts.valid = true;
  return 0;
}

// Nodes are renumbered tile-major by the tile that finishes them (the last
// colour holding the node): each tile's nodes by position, its inside first and
// then one run per lower/upper face, edge and corner, so that a tile's state and
// each piece its neighbours share are contiguous.  The words of a tile come in
// the order of their nodes, padding last.
//
// All of it follows from a tile's place in the lattice: along an axis a node on
// a face shared with the next tile is finished by the odd one of the two, so its
// number is that tile's first plus its rank there, and ranks and order depend on the
// kinds of a tile and its neighbours alone (extent, parity, faces shared): some
// hundred tables at most, from which a device kernel writes every tile's words.
// (Numbering slot by slot on the host took 0.3 s for 64^3 elastic hexes and 3 s
// for 128^3 acoustic ones in the first large batch of a mesh.)
void colour_tile_tables(const sem_mesh *m, ColourTables &c) {
  const TileSet &ts = m->tiles;
  const int N = m->order, NTL = (int)ts.slots_per_tile;
  const int L[3] = {ts.T[0] * N + 1, ts.T[1] * N + 1, m->dim == 3 ? ts.T[2] * N + 1 : 1};
  // kinds of tiles along each axis, and of a tile with the two next to it
  struct Kind {
    int last;              // last node
    bool odd, low, high;   // parity; its faces are shared
    bool operator<(const Kind &o) const { return std::tie(last, odd, low, high) < std::tie(o.last, o.odd, o.low, o.high); }
  };
  std::vector<Kind> kinds[3];
  std::vector<std::array<int, 3>> hoods[3];  // kinds of (previous, own, next) tile, -1: none
  std::vector<int> hood[3];                  // of each tile of the axis
  for (int a = 0; a < 3; ++a) {
    const int n = ts.nt[a];
    std::vector<int> kind(n);
    std::map<Kind, int> kid;
    std::map<std::array<int, 3>, int> hid;
    for (int i = 0; i < n; ++i) {
      const int64_t stride = a == 0 ? 1 : a == 1 ? ts.nt[0] : (int64_t)ts.nt[0] * ts.nt[1];
      const TileInfo &ti = ts.info[i * stride];
      const int e = a == 0 ? ti.ex : a == 1 ? ti.ey : ti.ez;
      const Kind k{a < m->dim ? e * N : 0, (i & 1) != 0, i > 0, i < n - 1};
      const auto it = kid.emplace(k, (int)kinds[a].size());
      if (it.second) kinds[a].push_back(k);
      kind[i] = it.first->second;
    }
    for (int i = 0; i < n; ++i) {
      const std::array<int, 3> h{i > 0 ? kind[i - 1] : -1, kind[i], i < n - 1 ? kind[i + 1] : -1};
      const auto it = hid.emplace(h, (int)hoods[a].size());
      if (it.second) hoods[a].push_back(h);
      hood[a].push_back(it.first->second);
    }
  }
  // ranks of the nodes a tile of each kind finishes (-1: another does), and how many
  std::map<std::array<int, 3>, std::pair<std::vector<int32_t>, int32_t>> ranked;
  const auto ranks = [&](const std::array<int, 3> &id) -> const std::pair<std::vector<int32_t>, int32_t> & {
    auto &r = ranked[id];
    if (!r.first.empty()) return r;
    r.first.assign(NTL, -1);
    int lo[3], hi[3], last[3];
    for (int a = 0; a < 3; ++a) {
      const Kind &k = kinds[a][id[a]];
      last[a] = k.last;
      lo[a] = k.low && !k.odd ? 1 : 0;
      hi[a] = k.high && !k.odd ? k.last - 1 : k.last;
    }
    std::vector<std::pair<int, int32_t>> order;  // (position, slot)
    for (int z = lo[2]; z <= hi[2]; ++z)
      for (int y = lo[1]; y <= hi[1]; ++y)
        for (int x = lo[0]; x <= hi[0]; ++x) {
          const auto at = [&](int v, int a) { return v == 0 ? 1 : v == last[a] ? 2 : 0; };
          order.emplace_back(at(x, 0) + 3 * at(y, 1) + 9 * at(z, 2), x + L[0] * (y + L[1] * z));
        }
    std::sort(order.begin(), order.end());
    for (size_t i = 0; i < order.size(); ++i) r.first[order[i].second] = (int32_t)i;
    r.second = (int32_t)order.size();
    return r;
  };
  std::map<std::array<int, 3>, int32_t> tid;
  c.type.resize(ts.ntiles);
  c.first.resize(ts.ntiles);
  uint32_t next = 0;
  for (int64_t t = 0; t < ts.ntiles; ++t) {
    const std::array<int, 3> id{hood[0][t % ts.nt[0]], hood[1][t / ts.nt[0] % ts.nt[1]],
                                hood[2][t / ((int64_t)ts.nt[0] * ts.nt[1])]};
    const std::array<int, 3> h[3] = {hoods[0][id[0]], hoods[1][id[1]], hoods[2][id[2]]};
    c.first[t] = next;
    next += (uint32_t)ranks({h[0][1], h[1][1], h[2][1]}).second;
    const auto it = tid.emplace(id, (int32_t)tid.size());
    c.type[t] = it.first->second;
    if (!it.second) continue;
    // a new neighbourhood: the tile that finishes each node, its rank there, the
    // words' order (tiles in theirs, ranks)
    const size_t o = c.words.size();
    c.words.resize(o + NTL, kSlotEmpty);
    c.lat.resize(o + NTL, kSlotEmpty);
    std::vector<std::pair<uint32_t, int32_t>> order;  // (finishing tile and rank, slot)
    for (int z = 0; z <= kinds[2][h[2][1]].last; ++z)
      for (int y = 0; y <= kinds[1][h[1][1]].last; ++y)
        for (int x = 0; x <= kinds[0][h[0][1]].last; ++x) {
          const int v[3] = {x, y, z};
          int at[3], d[3], shared = 0;
          std::array<int, 3> owner;
          bool starts = true, ends = true;
          for (int a = 0; a < 3; ++a) {
            const Kind &k = kinds[a][h[a][1]];
            const bool low = k.low && v[a] == 0, high = k.high && v[a] == k.last;
            d[a] = k.odd ? 0 : low ? -1 : high ? 1 : 0;
            owner[a] = h[a][d[a] + 1];
            at[a] = d[a] == 0 ? v[a] : d[a] < 0 ? kinds[a][owner[a]].last : 0;
            shared += low || high;
            starts = starts && !((low || high) && k.odd);
            ends = ends && d[a] == 0;
          }
          const int32_t s = x + L[0] * (y + L[1] * z);
          const uint32_t key = (uint32_t)(d[0] + 1 + 3 * (d[1] + 1) + 9 * (d[2] + 1)) << kRankBits |
                               (uint32_t)ranks(owner).first[at[0] + L[0] * (at[1] + L[1] * at[2])];
          order.emplace_back(key, s);
          c.lat[o + s] = key | (uint32_t)shared << kSharedShift | (starts ? kFlagFirst : 0u) | (ends ? kFlagLast : 0u);
        }
    std::sort(order.begin(), order.end());
    c.slot_of.resize(o + NTL, 0);
    for (size_t k = 0; k < order.size(); ++k) {
      c.words[o + k] = c.lat[o + order[k].second];
      c.slot_of[o + k] = (uint16_t)order[k].second;
    }
    size_t k = order.size();
    for (int32_t s = 0; s < NTL; ++s)
      if (c.lat[o + s] == kSlotEmpty) c.slot_of[o + k++] = (uint16_t)s;
    c.example.push_back((int32_t)t);
  }
}

}  // namespace sem
