// Host check of the colour launches' node numbering (colour_tile_tables in
// salvus_amd/csrc/tiles.cpp): the words that its tables give every tile, as the
// device kernel expands them, are those of a numbering made node by node -- each
// tile in turn numbers the nodes of which it is the last colour, by place and
// slot -- for boxes of one to seven tiles along an axis, with and without a partial
// tile at the end.  Exits non-zero if any word differs.
#include <algorithm>
#include <array>
#include <cstdio>
#include <map>
#include <tuple>

#include "sem_internal.h"

using namespace sem;

static int failures = 0, boxes = 0;

static void check(int dim, int N, const int *T, const int *nel) {
  sem_mesh m;
  m.dim = dim;
  m.order = N;
  TileSet &ts = m.tiles;
  int L[3];
  ts.ntiles = ts.slots_per_tile = 1;
  for (int a = 0; a < 3; ++a) {
    ts.T[a] = T[a];
    ts.nt[a] = (nel[a] + T[a] - 1) / T[a];
    L[a] = a < dim ? T[a] * N + 1 : 1;
    ts.ntiles *= ts.nt[a];
    ts.slots_per_tile *= L[a];
  }
  const int NTL = (int)ts.slots_per_tile;
  // node by node: lattice point of the mesh -> first and last colour
  std::map<std::array<int, 3>, std::pair<int, int>> span;
  std::map<std::array<int, 3>, uint32_t> id;
  const auto each = [&](int64_t t, auto &&f) {  // f(slot, lattice point, place)
    const TileInfo &ti = ts.info[t];
    const int c[3] = {(int)(t % ts.nt[0]), (int)(t / ts.nt[0] % ts.nt[1]), (int)(t / (ts.nt[0] * ts.nt[1]))};
    const int last[3] = {ti.ex * N, ti.ey * N, dim == 3 ? ti.ez * N : 0};
    for (int z = 0; z <= last[2]; ++z)
      for (int y = 0; y <= last[1]; ++y)
        for (int x = 0; x <= last[0]; ++x) {
          const int v[3] = {x, y, z};
          std::array<int, 3> p{};
          int place = 0;
          for (int a = 0, w = 1; a < dim; ++a, w *= 3) {
            p[a] = c[a] * T[a] * N + v[a];
            place += w * (v[a] == 0 ? 1 : v[a] == last[a] ? 2 : 0);
          }
          f(x + L[0] * (y + L[1] * z), p, place);
        }
  };
  for (int64_t t = 0; t < ts.ntiles; ++t) {
    const int c[3] = {(int)(t % ts.nt[0]), (int)(t / ts.nt[0] % ts.nt[1]), (int)(t / (ts.nt[0] * ts.nt[1]))};
    TileInfo ti{};
    ti.ex = std::min(T[0], nel[0] - c[0] * T[0]);
    ti.ey = std::min(T[1], nel[1] - c[1] * T[1]);
    ti.ez = std::min(T[2], nel[2] - c[2] * T[2]);
    ti.colour = (c[0] & 1) | (c[1] & 1) << 1 | (c[2] & 1) << 2;
    ts.info.push_back(ti);
  }
  for (int64_t t = 0; t < ts.ntiles; ++t)
    each(t, [&](int, const std::array<int, 3> &p, int) {
      const int c = ts.info[t].colour;
      auto it = span.emplace(p, std::make_pair(c, c)).first;
      it->second.first = std::min(it->second.first, c);
      it->second.second = std::max(it->second.second, c);
    });
  uint32_t next = 0;
  for (int64_t t = 0; t < ts.ntiles; ++t) {
    std::vector<std::tuple<int, int, std::array<int, 3>>> mine;
    each(t, [&](int s, const std::array<int, 3> &p, int place) {
      if (span[p].second == ts.info[t].colour) mine.emplace_back(place, s, p);
    });
    std::sort(mine.begin(), mine.end());
    for (const auto &e : mine) id[std::get<2>(e)] = next++;
  }
  ColourTables c;
  colour_tile_tables(&m, c);
  const size_t types = c.example.size();
  long wrong = c.words.size() != types * NTL || c.lat.size() != c.words.size() || c.slot_of.size() != c.words.size();
  for (int64_t t = 0; t < ts.ntiles && !wrong; ++t) {
    std::vector<std::pair<int64_t, int>> order;  // (node, slot), empty slots last
    std::vector<uint32_t> lat(NTL, kSlotEmpty);
    std::vector<int> shared(NTL, 0);
    each(t, [&](int s, const std::array<int, 3> &p, int) {
      const auto &sp = span[p];
      lat[s] = id[p] | (sp.first == ts.info[t].colour ? kFlagFirst : 0u) | (sp.second == ts.info[t].colour ? kFlagLast : 0u);
      for (int a = 0; a < dim; ++a) shared[s] += p[a] % (T[a] * N) == 0 && p[a] > 0 && p[a] < nel[a] * N;
    });
    for (int s = 0; s < NTL; ++s) order.emplace_back(lat[s] == kSlotEmpty ? (int64_t)next + s : lat[s] & kNodeMask, s);
    std::sort(order.begin(), order.end());
    const size_t o = (size_t)c.type[t] * NTL;
    const auto word = [&](uint32_t w) {
      if (w == kSlotEmpty) return w;
      const int at = (w >> kRankBits) & 31;
      const int64_t u = t + (at % 3 - 1) + ts.nt[0] * (at / 3 % 3 - 1) + (int64_t)ts.nt[0] * ts.nt[1] * (at / 9 - 1);
      if (u < 0 || u >= ts.ntiles) return kSlotEmpty - 1;
      return (c.first[u] + (w & ((1u << kRankBits) - 1))) | (w & (kFlagFirst | kFlagLast));
    };
    if (c.type[t] < 0 || c.type[t] >= (int64_t)types) { ++wrong; break; }
    for (int k = 0; k < NTL; ++k) {
      wrong += c.slot_of[o + k] != order[k].second || word(c.words[o + k]) != lat[order[k].second];
      wrong += word(c.lat[o + k]) != lat[k];
      if (c.lat[o + k] != kSlotEmpty) wrong += (int)((c.lat[o + k] >> kSharedShift) & 3) != shared[k];
    }
  }
  ++boxes;
  if (wrong) {
    ++failures;
    std::printf("dim %d order %d tile %dx%dx%d box %dx%dx%d: %ld wrong\n", dim, N, T[0], T[1], T[2], nel[0], nel[1], nel[2], wrong);
  }
}

int main() {
  for (int order = 1; order <= 2; ++order) {
    const int T3[3][3] = {{4, 2, 2}, {2, 2, 2}, {1, 1, 1}};
    for (const auto &T : T3)
      for (const auto &n : {std::array<int, 3>{1, 1, 1}, {2, 1, 3}, {2, 2, 2}, {3, 2, 1}, {1, 4, 5}, {5, 4, 3}, {7, 3, 4}, {6, 7, 5}})
        for (int part = 0; part < 8; ++part) {
          int nel[3];
          for (int a = 0; a < 3; ++a) nel[a] = n[a] * T[a] - ((part >> a) & 1 && T[a] > 1 ? 1 : 0);
          check(3, order, T, nel);
        }
    const int T2[3] = {8, 4, 1};
    for (int x = 1; x <= 7; ++x)
      for (int y = 1; y <= 7; ++y)
        for (int cut = 0; cut <= 3; ++cut) {
          const int nel[3] = {x * 8 - cut, y * 4 - cut, 1};
          check(2, order, T2, nel);
        }
  }
  if (failures) std::printf("%d of %d boxes differ\n", failures, boxes);
  else std::printf("all %d boxes alike\n", boxes);
  return failures ? 1 : 0;
}
