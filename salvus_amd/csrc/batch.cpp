// Batches: shots advanced together through the plain path (one shot per
// launch: gather / stiffness / colour scatter / update) or the batched path
// (tile launches and element colour launches over every group of the batch, in
// hipGraph-captured step blocks).  The time loop is Main.cpp:45-66; the
// update is Order2Newmark.cpp:68-115.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <map>
#include <set>
#include <tuple>

#include "batch.h"

using namespace sem;

namespace sem {

int64_t field_pos(const Group &g, int64_t i) {
  if (!g.tiled) return i;
  const sem_mesh *m = g.mesh;
  const int64_t c = i / m->G, node = i - c * m->G;
  return c * m->G + (g.parts ? m->tiles.to_internal : m->ctiles.to_internal)[node];
}

void free_group(Group &g) {
  dfree(g.fields);
  dfree(g.d_src);
  dfree(g.d_stf);
  dfree(g.d_load);
  dfree(g.d_step);
  dfree(g.d_seis);
  dfree(g.d_trec);
  dfree(g.d_trec_w);
  dfree(g.ext);
  dfree(g.mi_own);
  g.recs.clear();
  g.rec_nodes.clear();
  g.rec_w.clear();
  g.bytes = 0;
}

void drop_graph(sem_batch *b) {
  if (b->graph) (void)hipGraphExecDestroy(b->graph);
  if (b->graph_def) (void)hipGraphDestroy(b->graph_def);
  if (b->tail) (void)hipGraphExecDestroy(b->tail);
  if (b->tail_def) (void)hipGraphDestroy(b->tail_def);
  b->graph = nullptr;
  b->graph_def = nullptr;
  b->tail = nullptr;
  b->tail_def = nullptr;
  b->tail_steps = 0;
}

// Default launch shape: elements per block so a block has ~128-256 threads.
int default_epb(int nd) {
  int best = 1;
  for (int epb = 1; epb * nd <= 512; ++epb)
    if (block_threads(nd, epb) <= 256) best = epb;
  return best;
}

// SEM_TILE_OCCUPANCY=normal|high: the tile kernels of acoustic meshes run one
// launch per colour, in the given variant (tests compare them).
static const char *tile_occupancy(const sem_mesh *m) {
  const char *e = m->physics == SEM_ACOUSTIC ? getenv("SEM_TILE_OCCUPANCY") : nullptr;
  return e && (!strcmp(e, "high") || !strcmp(e, "normal")) ? e : nullptr;
}

// Whether the launch that a group's tiles join holds so many of them that one
// launch per colour is faster (sets Group::heavy of `gi`).  With partial results
// a step is one launch over all tiles, but its gathers and stores of shared
// nodes cost bandwidth; with colours it is 8 launches, each with the latency
// of its rounds of workgroups, on a numbering that leaves every tile fewer and
// longer runs.  Measured on 3-D meshes (milliseconds a step with partial
// results, with colours), by tile shots per workgroup that the chip holds:
// 54: 4 shots of 48^3 elastic hexes 0.77, 0.85; 128: 4 of 64^3 1.72, 1.68, 8 of
// 64^3 acoustic 1.37, 1.36; 163: 4 of 100^3 order-3 acoustic 1.09, 1.05; 182: 4 of
// 72^3 2.57, 2.53; 216: 2 of 96^3 3.12, 2.81, 4 of 96^3 acoustic 2.34, 2.28; 256: 8
// of 64^3 3.30, 3.08; 455: 8 of 128^3 order-2 acoustic 1.89, 1.89; 864: 8 of 96^3
// 11.0, 10.1; 1280: 32 of 32^3 to 96^3 16.2, 14.6.  In 2-D (4 colours, few shared
// nodes) the former colour kernel was slower at every size: 8 of 1000^2 elastic
// 1.54, 1.71, 4 of 2000^2 acoustic 1.53, 1.78.
constexpr int64_t kHeavyTiles = 160;
static int weigh_group(sem_batch *b, int gi) {
  Group &g = b->groups[gi];
  const sem_mesh *m = g.mesh;
  g.heavy = false;
  if (b->path != SEM_PATH_FUSED || !m->tiles.valid || m->dim != 3) return 0;
  int per_cu = 1, cus = 1;
  SEM_TRY(tile_kernel_prepare(m->dim, m->order, m->physics, m->tiles.T, kTileParts, &per_cu));
  HIPCHK(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, b->device));
  int64_t work = 0;
  for (const Group &o : b->groups)
    if (o.mesh->tiles.valid && o.mesh->dim == m->dim && o.mesh->order == m->order && o.mesh->physics == m->physics &&
        std::equal(m->tiles.T, m->tiles.T + 3, o.mesh->tiles.T))
      work += o.mesh->tiles.ntiles * o.S;
  g.heavy = work >= kHeavyTiles * per_cu * cus;
  return 0;
}

// Shared-node results of one plane (shot and component) of a group.
static int64_t group_parts(const Group &g) {
  return !g.parts ? 0 : g.tiled ? g.mesh->tiles.nparts : g.mesh->nparts;
}

int route_group(sem_batch *b, int gi) {
  Group &g = b->groups[gi];
  sem_mesh *m = g.mesh;
  const bool fused = b->path == SEM_PATH_FUSED;
  SEM_TRY(weigh_group(b, gi));
  // tile kernel: 32-bit field offsets, 16-bit shot numbers and at most
  // kTileMaxSrc sources per tile
  g.tiled = fused && m->tiles.valid && (uint64_t)m->c * (uint64_t)m->G * (uint64_t)g.S < (1ull << 32) && g.S < 65536;
  int64_t nsrc = 0;
  for (int k : g.shots)
    for (const SrcSpec &sp : b->shots[k].srcs) nsrc += sp.kind == 2 ? m->c : 1;
  if (g.tiled && nsrc > kTileMaxSrc) {
    std::map<int64_t, int> per_tile;
    for (int sl = 0; sl < g.S && g.tiled; ++sl)
      for (auto &sp : b->shots[g.shots[sl]].srcs) {
        int64_t e;
        std::vector<double> ld;
        SEM_TRY(source_load(m, sp, &e, ld));
        int &cnt = per_tile[m->tiles.elem_pos[e] / m->tiles.elems_per_tile];
        cnt += sp.kind == 2 ? m->c : 1;  // a file source is one source per component
        if (cnt > kTileMaxSrc) {
          g.tiled = false;
          break;
        }
      }
  }
  // partial results at shared nodes take at most an accumulator's memory in a
  // lean group, else colour launches run on the accumulator; with both the
  // results are the same
  if (g.tiled) {
    g.parts = g.lean ? m->tiles.nparts <= m->G : !(g.heavy || tile_occupancy(m));
    if (!g.parts) SEM_TRY(ensure_colour_tiles(m));
    g.parts = g.parts || m->ctiles.unfit;
  } else {
    if (fused && !g.lean) SEM_TRY(ensure_elem_parts(m));
    g.parts = fused && m->elem_parts == 1 && g.S < 65536 && (!g.lean || m->nparts <= m->G);
  }
  g.routed = true;
  return 0;
}

int64_t shot_bytes(const Group &g, const Shot &s, int64_t nsteps) {
  const sem_mesh *m = g.mesh;
  int64_t n = 4 * m->c * (g.parts ? 4 * m->G + group_parts(g) : 5 * m->G) + 8;  // fields, step counter
  n += 4 * (int64_t)s.recs.size() * m->c * nsteps;
  if (g.parts) n += (int64_t)s.recs.size() * ((int64_t)sizeof(TileRec) + 4 * m->nd);
  for (const SrcSpec &p : s.srcs)
    n += (p.kind == 2 ? m->c : 1) * (4 * nsteps + 4 * (int64_t)m->nd * m->c + (int64_t)sizeof(SrcDev));
  return n;
}

int setup_group(sem_batch *b, int gi) {
  Group &g = b->groups[gi];
  sem_mesh *m = g.mesh;
  const int path = b->path;
  int rc = 0;
  if (!g.routed) SEM_TRY(route_group(b, gi));
  const size_t len = (size_t)m->c * m->G * g.S;
  // u, w, a_, kc and the partial results at shared nodes (written before they
  // are read in each step) or the accumulator; kc = 0 is two bf16 zeros;
  // w = v + dt/2 a_ from the shot's initial v and a_
  const int64_t nparts = group_parts(g);
  const size_t arrays = g.parts ? 4 * len + (size_t)g.S * m->c * nparts : 5 * len;
  // The first group's allocation holds the batch's space for the field read-out
  // too: one of its own would cost each batch 30 to 60 us, the first 300 to 600.
  // An allocation above 64 MiB costs 0.2 ms more and its release 0.3 (fields
  // of 2.3 M entries, 50 + 18 MB: 28.9 -> 29.5 ms for set-up, 470 steps and
  // release), so one below it stays there with a smaller space.
  const size_t at = (arrays + 63) / 64 * 64, most = ((size_t)64 << 20) / 4;
  if (gi == 0 && b->read_len && !g.lean) {
    const size_t room = at >= most ? b->read_len : std::max<size_t>((most - at) / 2, 128 << 10);
    const size_t n = std::min(b->read_len, room);
    if (dalloc(&g.fields, at + 2 * n, &g.bytes) == 0) {
      b->d_read = reinterpret_cast<double *>(g.fields + at);
      b->read_cap = n;
    }
  }
  if (!g.fields) SEM_TRY(dalloc(&g.fields, arrays, &g.bytes));  // (the read-out then runs on the host)
  std::vector<float> buf;
  const double half_dt = 0.5 * g.dt;
  for (int which = 0; which < (g.parts ? 4 : 5); ++which) {
    bool any = false;
    for (int sl = 0; sl < g.S && which < 3; ++sl) {
      const Shot &s = b->shots[g.shots[sl]];
      any |= !s.init[which].empty() || (which == 1 && !s.init[2].empty());
    }
    if (!any) {  // zero start: a fill kernel, no host buffer
      SEM_TRY(launch_fill_f32((int64_t)len, g.fields + which * len, 0.f, b->stream));
      continue;
    }
    buf.assign(len, 0.f);
    for (int sl = 0; sl < g.S; ++sl) {
      const Shot &s = b->shots[g.shots[sl]];
      const size_t cg = (size_t)m->c * m->G;
      const std::vector<double> &v0 = s.init[1], &a0 = s.init[2];
      if (which == 1) {
        if (v0.empty() && a0.empty()) continue;
        for (size_t i = 0; i < cg; ++i)
          buf[sl * cg + field_pos(g, i)] =
              (float)((v0.empty() ? 0.0 : v0[i]) + (a0.empty() ? 0.0 : half_dt * a0[i]));
        continue;
      }
      if (s.init[which].empty()) continue;
      for (size_t i = 0; i < cg; ++i) buf[sl * cg + field_pos(g, i)] = (float)s.init[which][i];
    }
    HIPCHK(hipMemcpyAsync(g.fields + which * len, buf.data(), len * 4, hipMemcpyHostToDevice, b->stream));
    HIPCHK(hipStreamSynchronize(b->stream));
  }
  // step counter
  SEM_TRY(dalloc(&g.d_step, 1, &g.bytes));
  {
    const int64_t zero = 0;
    HIPCHK(hipMemcpyAsync(g.d_step, &zero, 8, hipMemcpyHostToDevice, b->stream));
    HIPCHK(hipStreamSynchronize(b->stream));
  }
  // sources: STF tables in FP64 at the accumulated times t_n (Main.cpp:45,
  // Order2Newmark.cpp:112), stored FP32
  std::vector<SrcDev> src;
  std::vector<float> stf, load;
  std::vector<int64_t> rec_out;  // seismogram offsets of g.recs
  std::vector<int32_t> rec_elem;  // tiled: tile-order position of their elements
  int64_t seis = 0;
  g.rec_key = m->c | (m->nd << 8);
  const Gll gl = make_gll(m->order);
  for (int sl = 0; sl < g.S; ++sl) {
    Shot &s = b->shots[g.shots[sl]];
    s.group = gi;
    s.slot = sl;
    for (auto &sp0 : s.srcs) {
      // a file source is one unit-direction source per component with that
      // component's tabulated series as its source-time function
      const int parts = sp0.kind == 2 ? m->c : 1;
      for (int k = 0; k < parts; ++k) {
        SrcSpec sp = sp0;
        if (sp0.kind == 2) {
          sp.kind = 0;
          for (int q = 0; q < 3; ++q) sp.dir[q] = q == k ? 1.0 : 0.0;
        }
        int64_t e;
        std::vector<double> ld;
        SEM_TRY(source_load(m, sp, &e, ld));
        SrcDev d;
        d.elem = g.tiled ? m->tiles.elem_pos[e] : m->inv_perm[e];
        d.stf_off = (int32_t)stf.size();
        d.load_off = (int32_t)load.size();
        d.shot = sl;
        if (sp0.kind == 2) {
          // (a shot shorter than its group's step count: zeros past its end)
          for (int64_t n = 0; n < g.nsteps; ++n)
            stf.push_back(n < sp0.nser ? (float)sp0.series[k * sp0.nser + n] : 0.f);
        } else {
          double t = 0.0;
          for (int64_t n = 0; n < g.nsteps; ++n) {
            stf.push_back((float)ricker(t, sp.amp, sp.f0, sp.t0));
            t += g.dt;
          }
        }
        for (double v : ld) load.push_back((float)v);
        src.push_back(d);
      }
    }
    // receivers: Lagrange weights of the owning element at the receiver
    s.seis_off = seis;
    for (size_t r = 0; r < s.recs.size(); ++r) {
      int64_t e;
      double ref[3];
      SEM_TRY(locate(m, s.recs[r].data(), &e, ref));
      RecDev d;
      d.nodes_off = (int32_t)g.rec_nodes.size();
      for (int p = 0; p < m->nd; ++p) {
        const int32_t gid = m->conn[e * m->nd + p];
        g.rec_nodes.push_back((uint32_t)field_pos(g, gid));
      }
      d.w_off = (int32_t)g.rec_w.size();
      d.shot = sl;
      d.stride = (int32_t)(s.recs.size() * m->c);
      d.out = nullptr;
      d.u = g.fields + (size_t)sl * m->c * m->G;
      d.step = g.d_step;
      d.G = m->G;
      d.nsteps = g.nsteps;
      rec_out.push_back(seis + (int64_t)r * m->c);
      rec_elem.push_back(g.tiled ? m->tiles.elem_pos[e] : (int32_t)e);
      double l[3][kMaxN];
      for (int a = 0; a < m->dim; ++a) lagrange(gl, ref[a], l[a]);
      for (int p = 0; p < m->nd; ++p) {
        const int P[3] = {p % m->n, (p / m->n) % m->n, m->dim == 3 ? p / (m->n * m->n) : 0};
        double v = 1;
        for (int a = 0; a < m->dim; ++a) v *= l[a][P[a]];
        g.rec_w.push_back((float)v);
      }
      g.recs.push_back(d);
    }
    // rows for every step of the group (a server groups shots whose step
    // counts differ a little; a shot's own rows are the first s.nsteps)
    seis += (int64_t)s.recs.size() * m->c * g.nsteps;
  }
  // a tile's sources are one range of the list (order kept within a tile)
  g.tile_src.clear();
  if (g.tiled) {
    const int ept = m->tiles.elems_per_tile;
    std::stable_sort(src.begin(), src.end(),
                     [&](const SrcDev &x, const SrcDev &y) { return x.elem / ept < y.elem / ept; });
    for (const SrcDev &d : src) g.tile_src.push_back(d.elem / ept);
  }
  g.seis_len = seis;
  SEM_TRY(dalloc(&g.d_seis, (size_t)std::max<int64_t>(seis, 1), &g.bytes));
  SEM_TRY(launch_fill_f32(std::max<int64_t>(seis, 1), g.d_seis, 0.f, b->stream));
  for (size_t r = 0; r < g.recs.size(); ++r) g.recs[r].out = g.d_seis + rec_out[r];
  g.tile_rec.clear();
  std::vector<TileRec> trec;
  if (g.parts && !g.recs.empty()) {
    // tile kernel: by tile and shot; element kernel: by shot and element (an
    // item's elements are one range of them)
    const int ept = g.tiled ? m->tiles.elems_per_tile : 1;
    std::vector<int32_t> order(g.recs.size());
    for (size_t r = 0; r < order.size(); ++r) order[r] = (int32_t)r;
    auto key = [&](int32_t r) {
      return g.tiled ? std::make_pair(rec_elem[r] / ept, g.recs[r].shot) : std::make_pair(g.recs[r].shot, rec_elem[r]);
    };
    std::stable_sort(order.begin(), order.end(), [&](int32_t x, int32_t y) { return key(x) < key(y); });
    for (int32_t r : order) {
      const RecDev &d = g.recs[r];
      trec.push_back(TileRec{d.out, d.w_off, d.shot, d.stride, g.tiled ? rec_elem[r] % ept : rec_elem[r]});
      g.tile_rec.push_back(key(r));
    }
    SEM_TRY(dalloc(&g.d_trec, trec.size(), &g.bytes));
    SEM_TRY(dalloc(&g.d_trec_w, g.rec_w.size(), &g.bytes));
    HIPCHK(hipMemcpyAsync(g.d_trec, trec.data(), trec.size() * sizeof(TileRec), hipMemcpyHostToDevice, b->stream));
    HIPCHK(hipMemcpyAsync(g.d_trec_w, g.rec_w.data(), g.rec_w.size() * 4, hipMemcpyHostToDevice, b->stream));
  }
  g.nsrc = (int)src.size();
  SEM_TRY(dalloc(&g.d_src, src.size(), &g.bytes));
  SEM_TRY(dalloc(&g.d_stf, stf.size(), &g.bytes));
  SEM_TRY(dalloc(&g.d_load, load.size(), &g.bytes));
  if (!src.empty()) {
    HIPCHK(hipMemcpyAsync(g.d_src, src.data(), src.size() * sizeof(SrcDev), hipMemcpyHostToDevice, b->stream));
    HIPCHK(hipMemcpyAsync(g.d_stf, stf.data(), stf.size() * 4, hipMemcpyHostToDevice, b->stream));
    HIPCHK(hipMemcpyAsync(g.d_load, load.data(), load.size() * 4, hipMemcpyHostToDevice, b->stream));
  }
  if (path == SEM_PATH_PLAIN || (!m->affine && !g.tiled)) SEM_TRY(ensure_pointwise(m));
  GroupDev h{};
  h.conn = m->d_conn;
  if (g.tiled) {
    h.tile_words = g.parts ? m->d_tile_words : m->ctiles.d_words;
    h.tile_words_lat = m->ctiles.d_words_lat;
    h.tile_slot = g.parts ? m->d_tile_slot : m->ctiles.d_slot;
    h.telem = m->d_telem;
    h.sh_part = m->d_sh_part;
  }
  if (g.parts) {
    h.rec = g.d_trec;
    h.rec_w = g.d_trec_w;
    h.part = g.fields + 4 * len;
    h.part_stride = nparts;
    h.epos = m->d_epos;
    h.sh_node = m->d_sh_node;
  }
  h.geo_e = m->d_geo_e;
  h.par_e = m->d_par_e;
  h.geo_p = m->d_geo_p;
  h.mi = !g.tiled ? m->d_mi : g.parts ? m->d_mi_int : m->ctiles.d_mi;
  h.u = g.fields;
  h.w = g.fields + len;
  h.ap = g.fields + 2 * len;
  h.kc = reinterpret_cast<uint32_t *>(g.fields + 3 * len);
  // (with partial results: the result of an accumulate-only pass, in the place of a_)
  h.acc = g.fields + (g.parts ? 2 : 4) * len;
  h.src = g.d_src;
  h.stf = g.d_stf;
  h.load = g.d_load;
  h.nsrc = g.nsrc;
  h.S = g.S;
  h.c = m->c;
  h.G = m->G;
  h.nsteps = g.nsteps;
  h.step = g.d_step;
  h.dt = (float)g.dt;
  h.acl = (float)((1.0 / 2.0) * g.dt);           // Order2Newmark.cpp:89
  h.quirks = m->quirks;
  // a coupled shot (a group of its own): external load and combined mass
  {
    const Shot &s0 = b->shots[g.shots[0]];
    if (s0.coupled >= 0) {
      const std::vector<float> &mc = coupled_mass(b->couples[s0.coupled], m);
      std::vector<float> mo(m->G);
      for (int64_t i = 0; i < m->G; ++i) mo[field_pos(g, i)] = mc[i];
      SEM_TRY(dalloc(&g.mi_own, (size_t)m->G, &g.bytes));
      SEM_TRY(dalloc(&g.ext, len, &g.bytes));
      SEM_TRY(launch_fill_f32((int64_t)len, g.ext, 0.f, b->stream));
      HIPCHK(hipMemcpyAsync(g.mi_own, mo.data(), mo.size() * 4, hipMemcpyHostToDevice, b->stream));
      HIPCHK(hipStreamSynchronize(b->stream));
      h.mi = g.mi_own;
      h.ext = g.ext;
      h.ap_always = 1;
    }
  }
  if ((int)b->h_groups.size() <= gi) b->h_groups.resize(gi + 1);
  b->h_groups[gi] = h;
  HIPCHK(hipStreamSynchronize(b->stream));
  return rc;
}

static void release_plan(sem_batch *b) {
  for (auto &l : b->launches) {
    dfree(l.d_items);
    dfree(l.d_elems);
    dfree(l.d_tiles);
    dfree(l.d_nodes);
  }
  b->launches.clear();
  for (auto &r : b->recsets) {
    dfree(r.d_recs);
    dfree(r.d_nodes);
    dfree(r.d_w);
  }
  b->recsets.clear();
}

static void batch_release(sem_batch *b) {
  drop_graph(b);
  free_couples(b);
  for (auto &g : b->groups) free_group(g);
  b->groups.clear();
  b->h_groups.clear();
  release_plan(b);
  dfree(b->d_groups);
  b->d_groups_cap = 0;
  b->d_read = nullptr;
  dfree(b->d_uloc);
  dfree(b->d_aloc);
  b->uloc_cap = 0;
  for (auto e : b->ev) (void)hipEventDestroy(e);
  b->ev.clear();
  b->ev_launches = 0;
  b->prepared = false;
}

// Items of one tile launch: every tile of its groups, each for `spw` shots.
// A workgroup that takes several shots reads the tile's words and element
// data once for them and loads a shot's lattice behind the previous shot's
// work, so shots stay together where the tiles alone fill the chip
// `kTileRounds` times over; below that they are spread over workgroups.
constexpr int kTileRounds = 2;
// The launch samples its groups' receivers (sets rec_in_tile) where every item
// is one shot's and holds at most one receiver component per wave: then the
// weights arrive with the tile and the sampling adds about 1 us to the
// workgroups that hold receivers, against 4-6 us a step for a launch of its
// own behind the step.  With more shots or receivers in an item their samples
// would be a serial chain (100 receivers along 500^2 elastic quads, loaded on
// demand: 49 -> 55 us a step).
//
// Partial results of a launch of 3-D elastic tiles are stored past the caches
// where they take a good part of the last-level cache (256 MB): smaller ones are
// read back from it, larger ones only push out what the next tiles read.  MB of
// them, us a step with stores through the caches, past them (order 4): 6, 24^3
// hexes 37.0, 39.3; 15, 32^3 63.3, 68.3; 24, 4 shots of 24^3 101.6, 110.2; 29, 40^3
// 111-115, 117; 51, 48^3 207-209, 211.5; 59, 4 of 32^3 252.3, 253.2; 102, 2 of 48^3
// 419.8, 418.4; 119, 8 of 32^3 485.5, 482.5; 122, 64^3 466, 469; 245, 2 of 64^3
// 965, 949; 490, 4 of 64^3 1831, 1788; order 3: 40^3 61.2, 66.1; order 2: 48^3 53.7,
// 57.8.  (A branch at the store instead of a kernel mode: 0.4 % more on both sides.)
constexpr int64_t kMaxCachedParts = (int64_t)96 << 20;
static std::vector<TileItem> tile_items(sem_batch *b, const std::vector<int> &gis, int capacity, int waves) {
  int spw = 1;
  for (int gi : gis) spw = std::max(spw, b->groups[gi].S);
  auto count = [&](int k) {
    int64_t n = 0;
    for (int gi : gis) n += b->groups[gi].mesh->tiles.ntiles * ((b->groups[gi].S + k - 1) / k);
    return n;
  };
  while (spw > 1 && count(spw) < (int64_t)kTileRounds * capacity) spw = (spw + 1) / 2;
  std::vector<TileItem> items;
  items.reserve(count(spw));
  for (int gi : gis) {
    Group &g = b->groups[gi];
    const size_t begin = items.size();
    size_t src = 0, rec = 0;
    int most = 0;
    for (int64_t t = 0; t < g.mesh->tiles.ntiles; ++t) {
      const TileInfo &ti = g.mesh->tiles.info[t];
      TileItem it{};
      it.group = gi;
      it.tile = (int32_t)t;
      it.ex = (uint8_t)ti.ex;
      it.ey = (uint8_t)ti.ey;
      it.ez = (uint8_t)ti.ez;
      it.nint = (uint16_t)ti.nint;
      it.nval = (uint16_t)ti.nval;
      it.own = (uint32_t)ti.own;
      it.sh_off = ti.sh_off;
      it.slots = ti.slots;
      it.src = (int32_t)src;
      while (src < g.tile_src.size() && g.tile_src[src] == t) ++src;
      it.nsrc = (int32_t)src - it.src;
      for (int s = 0; s < g.S; s += spw) {
        it.s0 = (uint16_t)s;
        it.s1 = (uint16_t)std::min(s + spw, g.S);
        it.rec = (int32_t)rec;
        while (rec < g.tile_rec.size() && g.tile_rec[rec].first == t && g.tile_rec[rec].second < it.s1) ++rec;
        it.nrec = (int32_t)rec - it.rec;
        most = std::max(most, it.nrec * g.mesh->c);
        items.push_back(it);
      }
    }
    g.rec_in_tile = spw == 1 && most > 0 && most <= waves;
    if (!g.rec_in_tile)
      for (size_t i = begin; i < items.size(); ++i) items[i].nrec = 0;
  }
  return items;
}

// Items of the launch of one tile colour: a tile each, with every shot of its
// group.
static std::vector<TileItem> colour_items(const sem_batch *b, const std::vector<int> &gis, int colour) {
  std::vector<TileItem> items;
  for (int gi : gis) {
    const Group &g = b->groups[gi];
    const sem_mesh *m = g.mesh;
    for (int64_t t = 0; t < m->tiles.ntiles; ++t) {
      const TileInfo &ti = m->tiles.info[t];
      if (ti.colour != colour) continue;
      const auto src = std::equal_range(g.tile_src.begin(), g.tile_src.end(), (int32_t)t);
      TileItem it{};
      it.group = gi;
      it.tile = (int32_t)t;
      it.s1 = (uint16_t)g.S;
      it.ex = (uint8_t)ti.ex;
      it.ey = (uint8_t)ti.ey;
      it.ez = (uint8_t)ti.ez;
      it.slots = m->ctiles.table[t];
      it.src = (int32_t)(src.first - g.tile_src.begin());
      it.nsrc = (int32_t)(src.second - src.first);
      items.push_back(it);
    }
  }
  return items;
}

// Acoustic colour launches take the high-occupancy variant when it needs fewer
// rounds of workgroups over the CUs and a workgroup takes at most two shots: one
// of its workgroups runs about 1.2x as long as a normal one, more with the
// later shots, whose lattices it gathers in lattice order (ms a step normal, high:
// one shot of 128^3 1.50, 1.43; two of 112^3 1.96, 1.90; four of 96^3 2.28, 2.38;
// of 128^3 5.14, 5.35).  Both variants do the same arithmetic in the same order:
// results are identical.
static int colour_mode(const LaunchSet &L, const char *forced, int shots, int cus, int *mode) {
  int lo = 1, hi = 1;
  SEM_TRY(tile_kernel_prepare(L.dim, L.order, L.physics, L.T, kTileColours, &lo));
  *mode = kTileColours;
  if (L.physics != SEM_ACOUSTIC) return 0;
  SEM_TRY(tile_kernel_prepare(L.dim, L.order, L.physics, L.T, kTileColoursHigh, &hi));
  const auto rounds = [&](int64_t per_cu) { return (L.nitems + per_cu * cus - 1) / (per_cu * cus); };
  if (forced ? !strcmp(forced, "high") : shots <= 2 && 6 * rounds(hi) < 5 * rounds(lo)) *mode = kTileColoursHigh;
  return 0;
}

// Items of the shared-node launch behind it: 256 nodes of one class each, for
// every plane (shot and component) of the group where that leaves enough
// workgroups to fill the chip, else one item per plane; 512 nodes where there
// is one plane only (64^3 acoustic hexes 40 -> 29 us; more planes give a thread
// enough to load).
static std::vector<NodeItem> shared_items(const sem_batch *b, const std::vector<int> &gis, int cus) {
  auto classes = [&](int gi) {
    const Group &g = b->groups[gi];
    if (!g.tiled) return g.mesh->classes;
    const TileSet &ts = g.mesh->tiles;
    std::vector<SharedClass> c;
    int64_t node = ts.nown, part = 0;
    for (int q = 0; q < 3; ++q) {
      c.push_back(SharedClass{2 << q, ts.sh_n[q], node, part});
      node += ts.sh_n[q];
      part += (2 << q) * ts.sh_n[q];
    }
    return c;
  };
  int64_t total = 0;
  for (int gi : gis)
    for (const SharedClass &c : classes(gi)) total += (c.n + kSharedNodes - 1) / kSharedNodes;
  const bool whole = total >= 16 * (int64_t)cus;  // two rounds of 8 workgroups per CU
  std::vector<NodeItem> items;
  for (int gi : gis) {
    const Group &g = b->groups[gi];
    const int64_t per = kSharedNodes * (whole && g.S * g.mesh->c == 1 ? 2 : 1);
    for (const SharedClass &c : classes(gi))
      for (int64_t f = 0; f < c.n; f += per)
        for (int p = whole ? -1 : 0; p < (whole ? 0 : g.S * g.mesh->c); ++p)
          items.push_back(NodeItem{gi, (int32_t)std::min<int64_t>(per, c.n - f), c.m, p, c.node + f,
                                   c.part + f, c.n, g.tiled ? 0 : 1, 0});
  }
  return items;
}

// Items of one element launch over every element of its groups (in the
// caller's order, so that neighbours are near in time and share an L2), the
// shots of a group spread over workgroups as in tile_items.  The launch samples
// its groups' receivers under the same rule (one-shot items, at most one
// receiver component per wave): 3 receivers, 400 steps of 150x133 deformed
// elastic quads and a read-out 9.9 -> 8.9 ms, 250 steps of 31x30x29 deformed
// acoustic hexes 15.4 -> 15.1.
static std::vector<WorkItem> element_items(sem_batch *b, const std::vector<int> &gis, int capacity, int waves,
                                           std::vector<int32_t> &elems) {
  int spw = 1;
  for (int gi : gis) spw = std::max(spw, b->groups[gi].S);
  auto count = [&](int k) {
    int64_t n = 0;
    for (int gi : gis) n += (b->groups[gi].mesh->E + b->epb - 1) / b->epb * ((b->groups[gi].S + k - 1) / k);
    return n;
  };
  while (spw > 1 && count(spw) < (int64_t)kTileRounds * capacity) spw = (spw + 1) / 2;
  std::vector<WorkItem> items;
  elems.clear();
  for (int gi : gis) {
    Group &g = b->groups[gi];
    const sem_mesh *m = g.mesh;
    const int64_t base = (int64_t)elems.size();
    const size_t begin = items.size();
    int most = 0;
    elems.insert(elems.end(), m->inv_perm.begin(), m->inv_perm.end());
    for (int64_t f = 0; f < m->E; f += b->epb)
      for (int s = 0; s < g.S; s += spw) {
        const int32_t count = (int32_t)std::min<int64_t>(b->epb, m->E - f);
        auto at = [&](int64_t e) {
          return std::lower_bound(g.tile_rec.begin(), g.tile_rec.end(), std::make_pair((int32_t)s, (int32_t)e)) -
                 g.tile_rec.begin();
        };
        const int32_t rec = (int32_t)at(f), nrec = (int32_t)at(f + count) - rec;
        most = std::max(most, nrec * m->c);
        items.push_back(WorkItem{gi, (int32_t)(base + f), count, (uint16_t)s, (uint16_t)std::min(s + spw, g.S),
                                 (int32_t)f, rec, nrec, 0});
      }
    g.rec_in_tile = spw == 1 && most > 0 && most <= waves;
    if (!g.rec_in_tile)
      for (size_t i = begin; i < items.size(); ++i) items[i].nrec = 0;
  }
  return items;
}

// Launches of one step: per kernel key the tiles of tiled groups or the
// elements of the others, behind them the shared nodes of both; groups without
// partial results one colour at a time, each colour of all of them in one launch.
static int build_plan(sem_batch *b) {
  // key = (lane, tile? | diagonal geometry << 1, dim, order, physics,
  // geometry mode, tile shape); SEM_TILE_GENERAL=1 keeps the general tile
  // kernel
  const char *gen = getenv("SEM_TILE_GENERAL");
  const bool general = gen && gen[0] == '1';
  // lanes: SEM_LANES=k (1..4) splits the groups over k streams (not with
  // coupled pairs, whose two groups exchange loads every step)
  const char *ln = getenv("SEM_LANES");
  const int ngroups = (int)b->groups.size();
  std::vector<int> lane(ngroups, 0);
  b->lanes = ln && atoi(ln) > 0 ? std::min(atoi(ln), kMaxLanes) : 1;
  if (!b->couples.empty()) b->lanes = 1;
  b->lanes = std::min(b->lanes, std::max(1, ngroups));
  if (b->lanes > 1) {
    // largest first onto the lightest lane (work: elements x shots)
    std::vector<int> order(ngroups);
    for (int gi = 0; gi < ngroups; ++gi) order[gi] = gi;
    auto work = [&](int gi) { return (double)b->groups[gi].mesh->E * b->groups[gi].S; };
    std::stable_sort(order.begin(), order.end(), [&](int x, int y) { return work(x) > work(y); });
    std::vector<double> load(b->lanes, 0.0);
    for (int gi : order) {
      const int l = (int)(std::min_element(load.begin(), load.end()) - load.begin());
      lane[gi] = l;
      load[l] += work(gi);
    }
    while ((int)b->lane_streams.size() < b->lanes - 1) {
      hipStream_t st;
      if (hipStreamCreateWithFlags(&st, hipStreamNonBlocking) != hipSuccess) {
        set_error("stream creation failed");
        return -2;
      }
      b->lane_streams.push_back(st);
    }
    while (b->lane_ev.size() < (size_t)kMaxBlockSteps * kMaxLanes) {
      hipEvent_t e;
      HIPCHK(hipEventCreateWithFlags(&e, hipEventDisableTiming));
      b->lane_ev.push_back(e);
    }
  }
  std::map<std::tuple<int, int, int, int, int, int, int>, std::vector<int>> keys;
  for (int gi = 0; gi < ngroups; ++gi) {
    sem_mesh *m = b->groups[gi].mesh;
    const bool t = b->groups[gi].tiled;
    const int shape = t ? m->tiles.T[0] * 10000 + m->tiles.T[1] * 100 + m->tiles.T[2] : 0;
    const int tk = (t ? 1 + 2 * (int)(m->tile_diag && !general) : 0) + (b->groups[gi].parts ? 0 : 4);
    keys[std::make_tuple(lane[gi], tk, m->dim, m->order, m->physics, geo_mode(m), shape)].push_back(gi);
  }
  for (auto &l : b->launches) {
    dfree(l.d_items);
    dfree(l.d_elems);
    dfree(l.d_tiles);
    dfree(l.d_nodes);
  }
  b->launches.clear();
  int cus = 1;
  HIPCHK(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, b->device));
  std::map<int, std::vector<int>> shared;  // lane -> groups with partial results
  auto upload = [&](auto **dst, const auto &items) {
    SEM_TRY(dalloc(dst, items.size()));
    HIPCHK(hipMemcpyAsync(*dst, items.data(), items.size() * sizeof(items[0]), hipMemcpyHostToDevice, b->stream));
    HIPCHK(hipStreamSynchronize(b->stream));
    return 0;
  };
  // (a launch owns its items, also after an error)
  auto add = [&](const LaunchSet &L) {
    b->launches.push_back(L);
    return &b->launches.back();
  };
  for (auto &kv : keys) {
    LaunchSet L{};
    L.lane = std::get<0>(kv.first);
    L.kind = std::get<1>(kv.first) & 1 ? kLaunchTile : kLaunchElement;
    L.diag = (std::get<1>(kv.first) & 2) != 0;
    L.dim = std::get<2>(kv.first);
    L.order = std::get<3>(kv.first);
    L.physics = std::get<4>(kv.first);
    L.gmode = std::get<5>(kv.first);
    L.nd = L.dim == 2 ? (L.order + 1) * (L.order + 1) : (L.order + 1) * (L.order + 1) * (L.order + 1);
    L.c = L.physics == SEM_ACOUSTIC ? 1 : L.dim;
    const int shape = std::get<6>(kv.first);
    L.T[0] = shape / 10000;
    L.T[1] = (shape / 100) % 100;
    L.T[2] = shape % 100;
    const bool colours = (std::get<1>(kv.first) & 4) != 0;
    if (!colours) {
      auto &sg = shared[L.lane];
      sg.insert(sg.end(), kv.second.begin(), kv.second.end());
    }
    if (L.kind == kLaunchTile && colours) {
      int shots = 1;
      for (int gi : kv.second) shots = std::max(shots, b->groups[gi].S);
      for (int c = 0; c < (1 << L.dim); ++c) {
        const std::vector<TileItem> items = colour_items(b, kv.second, c);
        L.colour = c;
        L.nitems = (int)items.size();
        SEM_TRY(colour_mode(L, tile_occupancy(b->groups[kv.second[0]].mesh), shots, cus, &L.mode));
        if (!items.empty()) SEM_TRY(upload(&add(L)->d_tiles, items));
      }
    } else if (L.kind == kLaunchTile) {
      int per_cu = 1;
      SEM_TRY(tile_kernel_prepare(L.dim, L.order, L.physics, L.T, kTileParts, &per_cu));
      const int waves = tile_kernel_info(L.dim, L.order, L.physics, L.T).threads / 64;
      const std::vector<TileItem> items = tile_items(b, kv.second, per_cu * cus, waves);
      int64_t parts = 0;
      for (int gi : kv.second) parts += 4 * b->groups[gi].S * L.c * group_parts(b->groups[gi]);
      if (L.dim == 3 && L.physics == SEM_ELASTIC && parts > kMaxCachedParts) {
        L.mode = kTilePartsPast;
        SEM_TRY(tile_kernel_prepare(L.dim, L.order, L.physics, L.T, L.mode, &per_cu));
      }
      L.nitems = (int)items.size();
      SEM_TRY(upload(&add(L)->d_tiles, items));
    } else if (!colours) {
      std::vector<int32_t> elems;
      const int threads = block_threads(L.nd, b->epb);
      const std::vector<WorkItem> items = element_items(b, kv.second, 2048 / threads * cus, threads / 64, elems);
      L.nitems = (int)items.size();
      LaunchSet *l = add(L);
      SEM_TRY(upload(&l->d_items, items));
      SEM_TRY(upload(&l->d_elems, elems));
    } else {
      int ncol = 0;
      for (int gi : kv.second) ncol = std::max(ncol, b->groups[gi].mesh->ncol);
      for (int c = 0; c < ncol; ++c) {
        std::vector<WorkItem> items;
        for (int gi : kv.second) {
          const sem_mesh *m = b->groups[gi].mesh;
          const int64_t end = c < m->ncol ? m->col_start[c + 1] : 0;
          for (int64_t f = c < m->ncol ? m->col_start[c] : 0; f < end; f += b->epb)
            items.push_back(WorkItem{gi, (int32_t)f, (int32_t)std::min<int64_t>(b->epb, end - f), 0, 0, 0, 0, 0, 0});
        }
        L.colour = c;
        L.nitems = (int)items.size();
        SEM_TRY(upload(&add(L)->d_items, items));
      }
    }
  }
  for (auto &kv : shared) {  // behind every other launch of their lane
    const std::vector<NodeItem> items = shared_items(b, kv.second, cus);
    if (items.empty()) continue;
    LaunchSet L{};
    L.kind = kLaunchShared;
    L.lane = kv.first;
    L.nitems = (int)items.size();
    SEM_TRY(upload(&add(L)->d_nodes, items));
  }
  // launches of one step that kernel timing counts: tile and element launches
  // (a tile launch with the shared-node launch behind it), those of the same
  // kernel and colour in different lanes, which run side by side, once
  std::set<std::tuple<int, int, int, int, int, int, int, int, bool>> per_step;
  for (const auto &L : b->launches)
    if (L.kind != kLaunchShared)
      per_step.insert(std::make_tuple((int)L.kind, (int)L.diag, L.dim, L.order, L.physics, L.gmode,
                                      L.T[0] * 10000 + L.T[1] * 100 + L.T[2], L.colour, L.mode >= kTileColours));
  b->step_launches = (int)per_step.size();
  HIPCHK(hipStreamSynchronize(b->stream));
  return 0;
}

int finalize_groups(sem_batch *b, int epb_hint) {
  drop_graph(b);
  release_plan(b);
  SEM_TRY(setup_couples(b));
  // group table
  const size_t ng = b->groups.size();
  if (ng > b->d_groups_cap) {
    dfree(b->d_groups);
    const size_t cap = std::max<size_t>(std::max<size_t>(ng, 2 * b->d_groups_cap), 16);
    b->d_groups_cap = 0;
    SEM_TRY(dalloc(&b->d_groups, cap));
    b->d_groups_cap = cap;
  }
  if (ng)
    HIPCHK(hipMemcpyAsync(b->d_groups, b->h_groups.data(), ng * sizeof(GroupDev), hipMemcpyHostToDevice, b->stream));
  for (auto &g : b->groups) g.rec_in_tile = false;
  // launch plan
  if (b->path == SEM_PATH_PLAIN) {
    size_t mx = 0;
    for (auto &g : b->groups) mx = std::max(mx, (size_t)g.mesh->E * g.mesh->nd * g.mesh->c);
    if (mx > b->uloc_cap) {
      dfree(b->d_uloc);
      dfree(b->d_aloc);
      b->uloc_cap = 0;
      SEM_TRY(dalloc(&b->d_uloc, mx));
      SEM_TRY(dalloc(&b->d_aloc, mx));
      b->uloc_cap = mx;
    }
    b->epb = 0;
  } else {
    int nd_max = 1;
    for (auto &g : b->groups) nd_max = std::max(nd_max, g.mesh->nd);
    b->epb = epb_hint > 0 ? epb_hint : default_epb(nd_max);
    if (block_threads(nd_max, b->epb) > 512) { set_error("elements per block too large"); return -1; }
    SEM_TRY(build_plan(b));
    int64_t min_steps = INT64_MAX;
    for (auto &g : b->groups) min_steps = std::min(min_steps, std::max<int64_t>(g.nsteps, 1));
    if (b->groups.empty()) min_steps = 1;
    b->block_steps = (int)std::min<int64_t>(std::max<int64_t>(1, 4096 / std::max<int>(1, (int)b->launches.size())), kMaxBlockSteps);
    b->block_steps = std::max(1, std::min<int>(b->block_steps, (int)min_steps));
    // SEM_GRAPH_STEPS=k: steps per captured graph block (1..50)
    const char *gs = getenv("SEM_GRAPH_STEPS");
    if (gs && atoi(gs) > 0) b->block_steps = std::max(1, std::min(atoi(gs), kMaxBlockSteps));
  }
  // receiver sets, one per (components, nodes per element, sampled by the tile
  // launches or not)
  std::map<int, std::vector<int>> by_key;
  for (int gi = 0; gi < (int)ng; ++gi)
    if (!b->groups[gi].recs.empty())
      by_key[b->groups[gi].rec_key | (b->groups[gi].rec_in_tile ? 1 << 24 : 0)].push_back(gi);
  for (auto &kv : by_key) {
    std::vector<RecDev> rd;
    std::vector<uint32_t> nodes;
    std::vector<float> w;
    for (int gi : kv.second) {
      const Group &g = b->groups[gi];
      const int32_t noff = (int32_t)nodes.size(), woff = (int32_t)w.size();
      for (RecDev d : g.recs) {
        d.nodes_off += noff;
        d.w_off += woff;
        rd.push_back(d);
      }
      nodes.insert(nodes.end(), g.rec_nodes.begin(), g.rec_nodes.end());
      w.insert(w.end(), g.rec_w.begin(), g.rec_w.end());
    }
    RecSet R;
    R.C = kv.first & 0xffffff;
    R.in_tile = (kv.first >> 24) != 0;
    R.nrec = (int)rd.size();
    SEM_TRY(dalloc(&R.d_recs, rd.size()));
    SEM_TRY(dalloc(&R.d_nodes, nodes.size()));
    SEM_TRY(dalloc(&R.d_w, w.size()));
    HIPCHK(hipMemcpyAsync(R.d_recs, rd.data(), rd.size() * sizeof(RecDev), hipMemcpyHostToDevice, b->stream));
    HIPCHK(hipMemcpyAsync(R.d_nodes, nodes.data(), nodes.size() * 4, hipMemcpyHostToDevice, b->stream));
    HIPCHK(hipMemcpyAsync(R.d_w, w.data(), w.size() * 4, hipMemcpyHostToDevice, b->stream));
    HIPCHK(hipStreamSynchronize(b->stream));
    b->recsets.push_back(R);
  }
  HIPCHK(hipStreamSynchronize(b->stream));
  return 0;
}

// Receivers after the step at offset koff of a block whose last offset is
// `last`; where the tile or element launches sample, every step but the block's last is
// sampled inside the next step's launch.
static int enqueue_receivers(sem_batch *b, int koff, int last) {
  for (auto &R : b->recsets) {
    if (R.in_tile && koff != last) continue;
    RecArgs ra;
    ra.recs = R.d_recs;
    ra.nodes = R.d_nodes;
    ra.weights = R.d_w;
    ra.nrec = R.nrec;
    ra.nd = R.C >> 8;
    ra.koff = koff;
    ra.end = R.in_tile;
    SEM_TRY(launch_receivers(ra, R.C & 0xff, b->stream));
  }
  return 0;
}

int enqueue_fused_step(sem_batch *b, int koff, int ku_only, int last) {
  if (!ku_only) SEM_TRY(enqueue_couples(b));  // coupling loads from the velocities after the last step
  // timing: one event pair around all launches of the step (a pair
  // per launch would add its own overhead to short launches)
  const bool timed = b->timing && !ku_only && !b->launches.empty();
  if (timed) {
    hipEvent_t e0, e1;
    HIPCHK(hipEventCreate(&e0));
    HIPCHK(hipEventCreate(&e1));
    b->ev.push_back(e0);
    b->ev.push_back(e1);
    b->ev_launches += (int64_t)b->step_launches;
    HIPCHK(hipEventRecord(e0, b->stream));
  }
  // lanes: fork from the batch stream, launch, join back (events of this
  // step's slot; a captured block holds at most kMaxBlockSteps steps)
  const int nl = b->lanes;
  hipEvent_t *lev = nl > 1 ? &b->lane_ev[(size_t)(koff % kMaxBlockSteps) * kMaxLanes] : nullptr;
  if (nl > 1) {
    HIPCHK(hipEventRecord(lev[0], b->stream));
    for (int l = 1; l < nl; ++l) HIPCHK(hipStreamWaitEvent(b->lane_streams[l - 1], lev[0], 0));
  }
  for (auto &L : b->launches) {
    hipStream_t st = L.lane > 0 && L.lane < nl ? b->lane_streams[L.lane - 1] : b->stream;
    FusedArgs a{};
    a.groups = b->d_groups;
    a.items = L.d_items;
    a.elems = L.d_elems;
    a.tiles = L.d_tiles;
    a.nodes = L.d_nodes;
    a.nitems = L.nitems;
    a.epb = b->epb;
    a.koff = koff;
    a.ku_only = ku_only;
    a.ap_koff = last;
    a.pad = 0;
    auto go = [&]() {
      if (L.kind == kLaunchTile) return launch_tile(L.dim, L.order, L.physics, L.T, L.diag, L.mode, a, st);
      if (L.kind == kLaunchShared) return launch_shared(a, st);
      return launch_fused(L.dim, L.order, L.physics, L.gmode, L.nitems, b->epb, L.nd, L.c, a, st);
    };
    SEM_TRY(go());
  }
  for (int l = 1; l < nl; ++l) {
    HIPCHK(hipEventRecord(lev[l], b->lane_streams[l - 1]));
    HIPCHK(hipStreamWaitEvent(b->stream, lev[l], 0));
  }
  if (timed) HIPCHK(hipEventRecord(b->ev.back(), b->stream));
  if (ku_only) return 0;
  return enqueue_receivers(b, koff, last);
}

int enqueue_plain_step(sem_batch *b) {
  SEM_TRY(enqueue_couples(b));
  for (int gi = 0; gi < (int)b->groups.size(); ++gi) {
    Group &g = b->groups[gi];
    GroupDev &h = b->h_groups[gi];
    sem_mesh *m = g.mesh;
    SEM_TRY(launch_plain_gather(m->E, m->nd, m->c, m->G, m->d_conn, h.u, b->d_uloc, b->stream));
    PlainArgs a;
    a.conn = m->d_conn;
    a.geo_p = m->d_geo_p;
    a.uloc = b->d_uloc;
    a.aloc = b->d_aloc;
    a.src = g.d_src;
    a.stf = g.d_stf;
    a.load = g.d_load;
    a.step = g.d_step;
    a.nsrc = g.nsrc;
    a.epb = default_epb(m->nd);
    a.E = m->E;
    a.koff = 0;
    a.pad = 0;
    if (b->timing) {
      hipEvent_t e0, e1;
      HIPCHK(hipEventCreate(&e0));
      HIPCHK(hipEventCreate(&e1));
      b->ev.push_back(e0);
      b->ev.push_back(e1);
      ++b->ev_launches;
      HIPCHK(hipEventRecord(e0, b->stream));
      SEM_TRY(launch_plain_stiffness(m->dim, m->order, m->physics, pointwise_mode(m), m->E, m->nd, m->c, a, b->stream));
      HIPCHK(hipEventRecord(e1, b->stream));
    } else {
      SEM_TRY(launch_plain_stiffness(m->dim, m->order, m->physics, pointwise_mode(m), m->E, m->nd, m->c, a, b->stream));
    }
    SEM_TRY(launch_fill_f32((int64_t)m->c * m->G, h.acc, 0.f, b->stream));
    for (int c = 0; c < m->ncol; ++c)
      SEM_TRY(launch_plain_scatter(m->col_start[c], m->col_start[c + 1] - m->col_start[c], m->nd, m->c,
                                   m->G, m->d_conn, b->d_aloc, h.acc, b->stream));
    SEM_TRY(launch_plain_update(m->G, m->c, m->quirks, h.dt, h.mi, h.acc, h.ext, h.u, h.w, h.ap,
                                h.kc, b->stream));
  }
  SEM_TRY(enqueue_receivers(b, 0, 0));
  SEM_TRY(launch_advance((int)b->groups.size(), b->d_groups, 1, b->stream));
  return 0;
}

int capture_graph(sem_batch *b, int steps) {
  const bool full = steps == b->block_steps;
  if (full && b->graph) return 0;
  if (!full && b->tail && b->tail_steps == steps) return 0;
  hipGraphExec_t &exec = full ? b->graph : b->tail;
  hipGraph_t &def = full ? b->graph_def : b->tail_def;
  if (exec) (void)hipGraphExecDestroy(exec);
  if (def) (void)hipGraphDestroy(def);
  exec = nullptr;
  def = nullptr;
  HIPCHK(hipStreamBeginCapture(b->stream, hipStreamCaptureModeThreadLocal));
  int rc = 0;
  for (int k = 0; k < steps && !rc; ++k) rc = enqueue_fused_step(b, k, 0, steps - 1);
  if (!rc) rc = launch_advance((int)b->groups.size(), b->d_groups, steps, b->stream);
  hipGraph_t gdef = nullptr;
  hipError_t e = hipStreamEndCapture(b->stream, &gdef);
  if (rc) {
    if (gdef) (void)hipGraphDestroy(gdef);
    return rc;
  }
  HIPCHK(e);
  def = gdef;
  HIPCHK(hipGraphInstantiate(&exec, gdef, nullptr, nullptr, 0));
  if (!full) b->tail_steps = steps;
  return 0;
}

}  // namespace sem

// Full batched-path steps (state advances; step counters do not), each timed
// with HIP events after one warm step; returns the fastest step's
// milliseconds (the least disturbed sample).
static double time_steps(sem_batch *b, int reps) {
  std::vector<hipEvent_t> ev(reps + 1, nullptr);
  auto done = [&](double r) {
    for (auto e : ev)
      if (e) (void)hipEventDestroy(e);
    return r;
  };
  for (auto &e : ev)
    if (hipEventCreate(&e) != hipSuccess) return done(-1);
  if (enqueue_fused_step(b, 0, 0, 0)) return done(-1);
  (void)hipEventRecord(ev[0], b->stream);
  for (int r = 0; r < reps; ++r) {
    if (enqueue_fused_step(b, 0, 0, 0)) return done(-1);
    (void)hipEventRecord(ev[r + 1], b->stream);
  }
  if (hipEventSynchronize(ev[reps]) != hipSuccess) return done(-1);
  double best = 1e300;
  for (int r = 0; r < reps; ++r) {
    float ms = 0;
    if (hipEventElapsedTime(&ms, ev[r], ev[r + 1]) != hipSuccess) return done(-1);
    best = std::min(best, (double)ms);
  }
  return done(best);
}

// key: mesh, nsteps, dt and (coupled shots, which form groups of their own)
// the shot index
using Bucket = std::map<std::tuple<sem_mesh *, int64_t, double, int>, std::vector<int>>;
static Bucket buckets_of(const sem_batch *b) {
  Bucket bk;
  for (int i = 0; i < (int)b->shots.size(); ++i)
    bk[std::make_tuple(b->shots[i].mesh, b->shots[i].nsteps, b->shots[i].dt,
                       b->shots[i].coupled >= 0 ? i : -1)].push_back(i);
  return bk;
}

static int largest_bucket(const sem_batch *b) {
  size_t mx = 0;
  for (auto &kv : buckets_of(b)) mx = std::max(mx, kv.second.size());
  return (int)mx;
}

// Groups of up to max_s shots sharing mesh, nsteps and dt.
static void form_groups(sem_batch *b, int max_s) {
  b->groups.clear();
  for (auto &kv : buckets_of(b)) {
    auto &list = kv.second;
    for (size_t k = 0; k < list.size(); k += max_s) {
      Group g;
      g.mesh = std::get<0>(kv.first);
      g.nsteps = std::get<1>(kv.first);
      g.dt = std::get<2>(kv.first);
      for (size_t j = k; j < std::min(list.size(), k + (size_t)max_s); ++j) g.shots.push_back(list[j]);
      g.S = (int)g.shots.size();
      g.lean = b->lean;
      b->groups.push_back(g);
    }
  }
}

static int set_up_once(sem_batch *b, int max_s, int epb) {
  form_groups(b, max_s);
  b->h_groups.resize(b->groups.size());
  for (int gi = 0; gi < (int)b->groups.size(); ++gi) SEM_TRY(setup_group(b, gi));
  return finalize_groups(b, epb);
}

// Groups of up to max_s shots on the device; a batch that the device memory
// does not hold with every group's first choice of kernels is set up again in
// the least memory (and without the space for the read-out).
static int set_up(sem_batch *b, int max_s, int epb) {
  int rc = set_up_once(b, max_s, epb);
  if (rc != -3 || b->lean) return rc;
  const int path = b->path;
  batch_release(b);
  b->path = path;
  b->lean = true;
  return set_up_once(b, max_s, epb);
}

static Shot *get_shot(sem_batch *b, int shot) {
  if (shot < 0 || shot >= (int)b->shots.size()) {
    set_error("shot index out of range");
    return nullptr;
  }
  return &b->shots[shot];
}

static float *field_base(sem_batch *b, const Shot &s, int which) {
  Group &g = b->groups[s.group];
  const size_t len = (size_t)s.mesh->c * s.mesh->G * g.S;
  return g.fields + (size_t)which * len;
}

extern "C" {

int sem_batch_create(sem_batch **out, int device) {
  *out = nullptr;
  SEM_TRY(set_device(device));
  auto *b = new sem_batch();
  b->device = device;
  if (hipStreamCreateWithFlags(&b->stream, hipStreamNonBlocking) != hipSuccess) {
    delete b;
    set_error("stream creation failed");
    return -2;
  }
  *out = b;
  return 0;
}

int sem_batch_destroy(sem_batch *b) {
  if (!b) return 0;
  (void)hipSetDevice(b->device);
  (void)hipStreamSynchronize(b->stream);
  batch_release(b);
  for (auto e : b->lane_ev) (void)hipEventDestroy(e);
  for (auto st : b->lane_streams) (void)hipStreamDestroy(st);
  (void)hipStreamDestroy(b->stream);
  delete b;
  return 0;
}

int sem_batch_add_shot(sem_batch *b, sem_mesh *m, int64_t nsteps, double dt, int *shot) {
  if (b->prepared) { set_error("batch already prepared"); return -1; }
  if (m->device != b->device) { set_error("mesh and batch on different devices"); return -1; }
  if (nsteps < 0 || !(dt > 0)) { set_error("nsteps >= 0 and dt > 0 required"); return -1; }
  Shot s;
  s.mesh = m;
  s.nsteps = nsteps;
  s.dt = dt;
  b->shots.push_back(s);
  *shot = (int)b->shots.size() - 1;
  return 0;
}

int sem_shot_add_source(sem_batch *b, int shot, const double *loc, double amp, double f0,
                        double t0, const double *dir) {
  Shot *s = get_shot(b, shot);
  if (!s) return -1;
  if (b->prepared) { set_error("batch already prepared"); return -1; }
  SrcSpec sp{};
  sp.kind = 0;
  for (int a = 0; a < s->mesh->dim; ++a) sp.loc[a] = loc[a];
  sp.amp = amp; sp.f0 = f0; sp.t0 = t0;
  for (int k = 0; k < s->mesh->c; ++k) sp.dir[k] = dir ? dir[k] : (k == 0 ? 1.0 : 0.0);
  int64_t e;
  std::vector<double> load;
  SEM_TRY(source_load(s->mesh, sp, &e, load));  // validates placement now
  s->srcs.push_back(sp);
  return 0;
}

int sem_shot_add_file_source(sem_batch *b, int shot, const double *loc, int ncomp,
                             int64_t nsamples, const double *stf) {
  Shot *s = get_shot(b, shot);
  if (!s) return -1;
  if (b->prepared) { set_error("batch already prepared"); return -1; }
  if (ncomp != s->mesh->c) { set_error("file source needs one series per field component"); return -1; }
  if (nsamples < s->nsteps || !stf) { set_error("file source needs a sample for every step"); return -1; }
  SrcSpec sp{};
  sp.kind = 2;
  for (int a = 0; a < s->mesh->dim; ++a) sp.loc[a] = loc[a];
  sp.dir[0] = 1.0;
  int64_t e;
  std::vector<double> load;
  SEM_TRY(source_load(s->mesh, sp, &e, load));  // validates placement now
  sp.nser = nsamples;
  sp.series.assign(stf, stf + (size_t)ncomp * nsamples);
  s->srcs.push_back(std::move(sp));
  return 0;
}

int sem_shot_add_moment_source(sem_batch *b, int shot, const double *loc, const double *M,
                               double amp, double f0, double t0) {
  Shot *s = get_shot(b, shot);
  if (!s) return -1;
  if (b->prepared) { set_error("batch already prepared"); return -1; }
  SrcSpec sp{};
  sp.kind = 1;
  const int d = s->mesh->dim;
  for (int a = 0; a < d; ++a) sp.loc[a] = loc[a];
  for (int i = 0; i < d * d; ++i) sp.M[i] = M[i];
  sp.amp = amp; sp.f0 = f0; sp.t0 = t0;
  int64_t e;
  std::vector<double> load;
  SEM_TRY(source_load(s->mesh, sp, &e, load));
  s->srcs.push_back(sp);
  return 0;
}

int sem_shot_add_receiver(sem_batch *b, int shot, const double *loc) {
  Shot *s = get_shot(b, shot);
  if (!s) return -1;
  if (b->prepared) { set_error("batch already prepared"); return -1; }
  std::array<double, 3> r{0, 0, 0};
  for (int a = 0; a < s->mesh->dim; ++a) r[a] = loc[a];
  int64_t e;
  double ref[3];
  SEM_TRY(locate(s->mesh, r.data(), &e, ref));
  s->recs.push_back(r);
  return 0;
}

int sem_shot_set_field(sem_batch *b, int shot, int which, const double *vals) {
  Shot *s = get_shot(b, shot);
  if (!s) return -1;
  if (which < 0 || which > 2) { set_error("field selector"); return -1; }
  const size_t len = (size_t)s->mesh->c * s->mesh->G;
  if (!b->prepared) {
    s->init[which].assign(vals, vals + len);
    return 0;
  }
  // live update of this shot's slice; v and a_ live in the state as
  // w = v + dt/2 a_ and a_, so setting one keeps the other
  HIPCHK(hipSetDevice(b->device));
  Group &g = b->groups[s->group];
  const double half_dt = 0.5 * g.dt;
  std::vector<float> buf(len), wcur, acur;
  auto fetch = [&](int w, std::vector<float> &out) {
    out.resize(len);
    HIPCHK(hipMemcpyAsync(out.data(), field_base(b, *s, w) + (size_t)s->slot * len, len * 4,
                          hipMemcpyDeviceToHost, b->stream));
    HIPCHK(hipStreamSynchronize(b->stream));
    return 0;
  };
  if (which >= 1) {
    SEM_TRY(fetch(1, wcur));
    SEM_TRY(fetch(2, acur));
  }
  auto put = [&](int w) {
    HIPCHK(hipMemcpyAsync(field_base(b, *s, w) + (size_t)s->slot * len, buf.data(), len * 4,
                          hipMemcpyHostToDevice, b->stream));
    HIPCHK(hipStreamSynchronize(b->stream));
    return 0;
  };
  if (which == 0) {
    for (size_t i = 0; i < len; ++i) buf[field_pos(g, i)] = (float)vals[i];
    return put(0);
  }
  if (which == 1) {  // w = v_new + dt/2 a_
    for (size_t i = 0; i < len; ++i) {
      const size_t k = field_pos(g, i);
      buf[k] = (float)(vals[i] + half_dt * acur[k]);
    }
    return put(1);
  }
  // a_ new: w = (w - dt/2 a_old) + dt/2 a_new keeps v
  for (size_t i = 0; i < len; ++i) {
    const size_t k = field_pos(g, i);
    buf[k] = (float)((double)wcur[k] - half_dt * acur[k] + half_dt * vals[i]);
  }
  SEM_TRY(put(1));
  for (size_t i = 0; i < len; ++i) buf[field_pos(g, i)] = (float)vals[i];
  return put(2);
}

int sem_shot_get_field(sem_batch *b, int shot, int which, double *vals) {
  Shot *s = get_shot(b, shot);
  if (!s) return -1;
  if (which < 0 || which > 2) { set_error("field selector"); return -1; }
  const size_t len = (size_t)s->mesh->c * s->mesh->G;
  if (!b->prepared) {
    for (size_t i = 0; i < len; ++i) vals[i] = s->init[which].empty() ? 0.0 : s->init[which][i];
    return 0;
  }
  HIPCHK(hipSetDevice(b->device));
  Group &g = b->groups[s->group];
  const float *f = field_base(b, *s, which) + (size_t)s->slot * len;
  const float *ap = which == 1 ? field_base(b, *s, 2) + (size_t)s->slot * len : nullptr;  // v = w - dt/2 a_
  const double half_dt = 0.5 * g.dt;
  std::lock_guard<std::mutex> lock(b->read_mu);
  if (!b->d_read) {  // the same on the host
    std::vector<float> buf(len), abuf(ap ? len : 0);
    HIPCHK(hipMemcpyAsync(buf.data(), f, len * 4, hipMemcpyDeviceToHost, b->stream));
    if (ap) HIPCHK(hipMemcpyAsync(abuf.data(), ap, len * 4, hipMemcpyDeviceToHost, b->stream));
    HIPCHK(hipStreamSynchronize(b->stream));
    for (size_t i = 0; i < len; ++i) {
      const size_t k = field_pos(g, i);
      vals[i] = ap ? (double)buf[k] - half_dt * (double)abuf[k] : (double)buf[k];
    }
    return 0;
  }
  const int32_t *to = !g.tiled ? nullptr : g.parts ? s->mesh->d_to_int : s->mesh->ctiles.d_to_int;
  for (size_t i = 0; i < len; i += b->read_cap) {
    const size_t n = std::min(b->read_cap, len - i);
    SEM_TRY(launch_read_field((int64_t)n, (int64_t)i, s->mesh->G, to, f, ap, half_dt, b->d_read, b->stream));
    HIPCHK(hipMemcpyAsync(vals + i, b->d_read, n * 8, hipMemcpyDeviceToHost, b->stream));
  }
  HIPCHK(hipStreamSynchronize(b->stream));
  return 0;
}

int sem_batch_prepare(sem_batch *b, int path, int epb, int spg) {
  if (b->prepared) { set_error("batch already prepared"); return -1; }
  if (b->shots.empty()) { set_error("batch has no shots"); return -1; }
  if (path != SEM_PATH_PLAIN && path != SEM_PATH_FUSED) { set_error("path"); return -1; }
  HIPCHK(hipSetDevice(b->device));
  b->path = path;
  b->lean = false;
  // one field, read out in pieces of at most 32 MiB
  for (const Shot &s : b->shots) b->read_len = std::max(b->read_len, (size_t)s.mesh->c * s.mesh->G);
  b->read_len = std::min<size_t>(b->read_len, (size_t)4 << 20);
  auto fail = [&](int r) { batch_release(b); return r; };
  int rc = 0;
  // ---- shots per group: given, 1 on the plain path, or autotuned: every
  // power of two up to the largest bucket is set up and timed over full
  // steps (the state is rebuilt from the shot specifications afterwards)
  int max_s = path == SEM_PATH_PLAIN ? 1 : spg;
  if (max_s <= 0) {
    const int biggest = largest_bucket(b);
    max_s = std::min(biggest, 8);
    if (biggest > 1) {
      double best = 1e300;
      for (int cand = 1; cand <= std::min(biggest, 8); cand *= 2) {
        rc = set_up(b, cand, epb);
        const double t = rc ? -1 : time_steps(b, 3);
        batch_release(b);
        if (rc) return rc;
        if (t < 0) return fail(-2);
        if (t < best * 0.99) {
          best = t;
          max_s = cand;
        }
      }
      b->path = path;
    }
  }
  // ---- grouping: shots sharing mesh, nsteps and dt
  if ((rc = set_up(b, max_s, epb))) return fail(rc);
  if (path == SEM_PATH_FUSED && epb <= 0) {
    bool any_elem = false;
    int nd_max = 1;
    for (auto &g : b->groups) {
      any_elem |= !g.tiled;
      nd_max = std::max(nd_max, g.mesh->nd);
    }
    if (any_elem) {
      // autotune elements per block of the element kernel over full steps
      // (gather, operator and finish: the stiffness pass alone ranks them
      // differently), one candidate per distinct block size; the timed steps
      // advance the state, so it is rebuilt from the shot specifications
      double best = 1e300;
      int best_epb = b->epb, last = 0;
      for (int bt = 64; bt <= 512; bt += 64) {
        const int cand = bt / nd_max;
        if (cand < 1 || cand == last) continue;
        last = cand;
        b->epb = cand;
        if ((rc = build_plan(b))) return fail(rc);
        const double t = time_steps(b, 3);
        if (t < 0) return fail(-2);
        if (t < best * 0.99) {
          best = t;
          best_epb = cand;
        }
      }
      batch_release(b);
      b->path = path;
      if ((rc = set_up(b, max_s, best_epb))) return fail(rc);
    }
  }
  b->spg = max_s;
  // the full-block graph is captured here (capture runs nothing), so the
  // first run's whole blocks are already replays
  const char *ng = getenv("SEM_NO_GRAPH");
  if (path == SEM_PATH_FUSED && !(ng && ng[0] == '1') && (rc = capture_graph(b, b->block_steps)))
    return fail(rc);
  if ((rc = hip_check(hipStreamSynchronize(b->stream), "sync"))) return fail(rc);
  b->prepared = true;
  return 0;
}

int sem_batch_run(sem_batch *b, int64_t nsteps) {
  if (!b->prepared) { set_error("batch not prepared"); return -1; }
  HIPCHK(hipSetDevice(b->device));
  for (auto e : b->ev) (void)hipEventDestroy(e);
  b->ev.clear();
  b->ev_launches = 0;
  int64_t left = nsteps;
  if (b->path == SEM_PATH_PLAIN) {
    const char *tg = getenv("SEM_TIME_KERNELS");
    b->timing = tg && tg[0] == '1';
    for (int64_t k = 0; k < left; ++k) {
      std::lock_guard<std::mutex> lock(b->read_mu);
      SEM_TRY(enqueue_plain_step(b));
    }
  } else {
    const char *tg = getenv("SEM_TIME_KERNELS");
    b->timing = tg && tg[0] == '1';
    const char *ng = getenv("SEM_NO_GRAPH");
    const bool graphs = !(ng && ng[0] == '1') && !b->timing;
    while (left > 0) {
      std::lock_guard<std::mutex> lock(b->read_mu);  // no steps between the pieces of a read-out
      if (graphs) {  // full blocks, then one (cached) tail block
        const int k = (int)std::min<int64_t>(left, b->block_steps);
        SEM_TRY(capture_graph(b, k));
        HIPCHK(hipGraphLaunch(k == b->block_steps ? b->graph : b->tail, b->stream));
        left -= k;
      } else {
        const int k = (int)std::min<int64_t>(left, b->block_steps);
        for (int j = 0; j < k; ++j) SEM_TRY(enqueue_fused_step(b, j, 0, k - 1));
        SEM_TRY(launch_advance((int)b->groups.size(), b->d_groups, k, b->stream));
        left -= k;
      }
    }
  }
  HIPCHK(hipStreamSynchronize(b->stream));
  b->steps_done += nsteps;
  if (!b->ev.empty()) {
    double ms = 0;
    for (size_t i = 0; i + 1 < b->ev.size(); i += 2) {
      float t = 0;
      HIPCHK(hipEventElapsedTime(&t, b->ev[i], b->ev[i + 1]));
      ms += t;
    }
    b->kernel_ms = ms;
    b->kernel_launches = b->ev_launches;
  }
  b->timing = false;
  return 0;
}

int sem_shot_progress(sem_batch *b, int shot, int64_t *steps, double *time) {
  Shot *s = get_shot(b, shot);
  if (!s) return -1;
  int64_t st = 0;
  if (b->prepared) {
    HIPCHK(hipSetDevice(b->device));
    HIPCHK(hipMemcpy(&st, b->groups[s->group].d_step, 8, hipMemcpyDeviceToHost));
  }
  *steps = st;
  double t = 0;
  for (int64_t k = 0; k < st; ++k) t += s->dt;
  *time = t;
  return 0;
}

int sem_shot_get_seismograms(sem_batch *b, int shot, float *out) {
  Shot *s = get_shot(b, shot);
  if (!s) return -1;
  if (!b->prepared) { set_error("batch not prepared"); return -1; }
  const size_t n = s->recs.size() * s->mesh->c * s->nsteps;
  if (n == 0) return 0;
  HIPCHK(hipSetDevice(b->device));
  HIPCHK(hipMemcpy(out, b->groups[s->group].d_seis + s->seis_off, n * 4, hipMemcpyDeviceToHost));
  return 0;
}

int sem_batch_config(const sem_batch *b, int64_t *cfg) {
  cfg[0] = b->epb;
  cfg[1] = b->spg;
  cfg[2] = b->block_steps;
  cfg[3] = (int64_t)b->groups.size();
  int64_t tiled = 0;
  for (const auto &g : b->groups) tiled += g.tiled ? 1 : 0;
  cfg[4] = tiled;
  return 0;
}

int sem_batch_lanes(const sem_batch *b, int *lanes) {
  *lanes = b->prepared ? b->lanes : 0;
  return 0;
}

int sem_batch_kernel_time(const sem_batch *b, double *ms, int64_t *launches) {
  *ms = b->kernel_ms;
  *launches = b->kernel_launches;
  return 0;
}

int sem_mesh_autotune(sem_mesh *m, int reps, int shots, int64_t *shape) {
  *shape = 0;
  HIPCHK(hipSetDevice(m->device));
  if (!m->tiles.valid) return 0;  // element kernel: nothing to choose per mesh
  if (shots < 1 || shots > 64) { set_error("autotune shots must be 1..64"); return -1; }
  reps = std::max(reps, 1);
  int shapes[3 * 16];
  const int ns = tile_kernel_shapes(m->dim, m->order, m->physics, shapes, 16);
  double best = 1e300;
  int bi = -1;
  for (int i = 0; i < ns; ++i) {
    SEM_TRY(setup_tiles(m, &shapes[3 * i]));
    if (!m->tiles.valid) continue;
    sem_batch *b = nullptr;
    SEM_TRY(sem_batch_create(&b, m->device));
    int rc = 0;
    for (int s = 0; s < shots && !rc; ++s) {
      int k = 0;
      rc = sem_batch_add_shot(b, m, 2 * reps + 4, 1.0, &k);
    }
    if (!rc) rc = sem_batch_prepare(b, SEM_PATH_FUSED, default_epb(m->nd), shots);
    const double t = rc ? -1 : time_steps(b, 2 * reps);
    sem_batch_destroy(b);
    if (rc) return rc;
    if (t < 0) { set_error("autotune timing failed"); return -2; }
    if (t < best * 0.98) {
      best = t;
      bi = i;
    }
  }
  SEM_TRY(setup_tiles(m, bi >= 0 ? &shapes[3 * bi] : nullptr));
  if (m->tiles.valid) *shape = m->tiles.T[0] * 10000 + m->tiles.T[1] * 100 + m->tiles.T[2];
  return 0;
}

int sem_mesh_apply_stiffness(sem_mesh *m, int path, const float *u, float *ku) {
  HIPCHK(hipSetDevice(m->device));
  sem_batch *b = nullptr;
  SEM_TRY(sem_batch_create(&b, m->device));
  int shot = 0;
  int rc = sem_batch_add_shot(b, m, 1, 1.0, &shot);
  if (!rc) rc = sem_batch_prepare(b, path, path == SEM_PATH_FUSED ? default_epb(m->nd) : 0, 1);
  const size_t len = (size_t)m->c * m->G;
  std::vector<float> uin(u, u + len);
  if (!rc && b->groups[0].tiled)
    for (size_t i = 0; i < len; ++i) uin[field_pos(b->groups[0], i)] = u[i];
  if (!rc) rc = hip_check(hipMemcpyAsync(b->h_groups[0].u, uin.data(), len * 4, hipMemcpyHostToDevice, b->stream), "upload");
  if (!rc) {
    if (path == SEM_PATH_FUSED) {
      rc = enqueue_fused_step(b, 0, 1, 0);
    } else {
      GroupDev &h = b->h_groups[0];
      rc = launch_plain_gather(m->E, m->nd, m->c, m->G, m->d_conn, h.u, b->d_uloc, b->stream);
      PlainArgs a{};
      a.conn = m->d_conn;
      a.geo_p = m->d_geo_p;
      a.uloc = b->d_uloc;
      a.aloc = b->d_aloc;
      a.epb = default_epb(m->nd);
      a.E = m->E;
      if (!rc) rc = launch_plain_stiffness(m->dim, m->order, m->physics, pointwise_mode(m), m->E, m->nd, m->c, a, b->stream);
      if (!rc) rc = launch_fill_f32((int64_t)len, h.acc, 0.f, b->stream);
      for (int c = 0; c < m->ncol && !rc; ++c)
        rc = launch_plain_scatter(m->col_start[c], m->col_start[c + 1] - m->col_start[c], m->nd, m->c,
                                  m->G, m->d_conn, b->d_aloc, h.acc, b->stream);
    }
  }
  std::vector<float> acc(len);
  if (!rc) rc = hip_check(hipMemcpyAsync(acc.data(), b->h_groups[0].acc, len * 4, hipMemcpyDeviceToHost, b->stream), "copy");
  if (!rc) rc = hip_check(hipStreamSynchronize(b->stream), "sync");
  if (!rc)
    for (size_t i = 0; i < len; ++i) ku[i] = -acc[field_pos(b->groups[0], i)];
  sem_batch_destroy(b);
  return rc;
}

}  // extern "C"
