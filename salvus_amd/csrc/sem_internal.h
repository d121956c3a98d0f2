// Internal declarations of the MI355X SEM library (host + device).
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>
#include <memory>
#include <string>
#include <vector>

#include "../../include/salvus_sem.h"
#include "element_bins.h"
#include "tile_layout.h"

namespace sem {

// ---------------------------------------------------------------- limits
constexpr int kMaxOrder3D = 7;   // Hexahedra::mMaxOrder with the order-7 table
constexpr int kMaxOrder2D = 10;  // TensorQuad::mMaxOrder
constexpr int kMaxN = 11;

// Gather-map words carry three flags above the node index (G < 2^29); tile
// words the Dirichlet flag only.
constexpr uint32_t kNodeMask = (1u << 29) - 1;
constexpr uint32_t kFlagDirichlet = 1u << 29;  // zero the stiffness row only
constexpr uint32_t kFlagFirst = 1u << 30;      // first colour to touch the node: store
constexpr uint32_t kFlagLast = 1u << 31;       // last colour: finalise (mass + Newmark)
// Slot-table words of the tile kernel: LDS lattice slot, a flag set in every
// word of a mesh that has Dirichlet nodes (only then are the words of a tile's
// own nodes read for theirs), place of the total in the high half.
constexpr uint32_t kSlotMask = 0x7fffu, kSlotDirichlet = 0x8000u;
// Tile lattice slot outside the mesh (partial tile at the mesh edge).
constexpr uint32_t kSlotEmpty = 0xffffffffu;

// ---------------------------------------------------------------- errors
void set_error(const std::string &msg);
#define SEM_TRY(expr)                                   \
  do {                                                  \
    int _rc = (expr);                                   \
    if (_rc) return _rc;                                \
  } while (0)
int hip_check(hipError_t e, const char *what);
#define HIPCHK(x) SEM_TRY(::sem::hip_check((x), #x))

// ---------------------------------------------------------------- host maths (FP64)
struct Gll {
  int order = 0, n = 0;
  double xi[kMaxN], w[kMaxN], D[kMaxN * kMaxN];  // D[i*n+j] = l'_j(xi_i)
};
Gll make_gll(int order);
void lagrange(const Gll &g, double x, double *l);
void lagrange_deriv(const Gll &g, double x, double *dl);

// J rows d/dr, d/ds(, d/dt); returns det.
double jacobian(int dim, const double *vtx, const double *ref, double *J);
double invert(int dim, const double *J, double *inv);
void p1_weights(int dim, const double *ref, double *w);
// 1 inside/on hull, 0 outside, -1 degenerate element
int check_hull(int dim, const double *pt, const double *vtx);
int inverse_map(int dim, const double *pt, const double *vtx, double *ref);

// ---------------------------------------------------------------- mesh topology
struct Topology {
  int dim = 0, order = 0;
  int64_t E = 0, V = 0, NF = 0, NEd = 0, G = 0;
  std::vector<int32_t> conn;  // E x nd (original element order)
};
int build_topology(int dim, int order, int64_t E, int64_t V, const int32_t *cells, Topology &T);
int colour_elements(int dim, int64_t E, int64_t V, const int32_t *cells,
                    std::vector<int32_t> &colour);

// ---------------------------------------------------------------- device-side descriptors
// Global-memory view of a device pointer.  Pointers that kernels read out of
// structs in memory are generic, and generic (flat) accesses also count on
// the LDS wait counter, so every wait for an LDS read would also wait for all
// outstanding global loads; kernels access HBM through these views instead.
// (The host pass parses kernel bodies too; there the view is the plain pointer.)
#if defined(__HIP_DEVICE_COMPILE__)
template <class T>
using gptr = __attribute__((address_space(1))) T *;
#else
template <class T>
using gptr = T *;
#endif
template <class T>
__device__ __forceinline__ gptr<T> glb(T *p) {
  return (gptr<T>)p;
}

// Kahan compensations of u and v are stored as the two bf16 halves of one
// word (round to nearest even).  A compensation is the rounding error of the
// last update, at most half an ulp of the sum, so its leading 8 bits keep the
// compensated u and v within about one FP32 ulp over thousands of steps while
// the state moves 8 bytes less per component and node.
__device__ __forceinline__ uint32_t pack_comp(float cu, float cv) {
#if defined(__HIP_DEVICE_COMPILE__)
  typedef float f32x2 __attribute__((ext_vector_type(2)));
  typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
  const bf16x2 h = __builtin_convertvector(f32x2{cu, cv}, bf16x2);  // one v_cvt_pk_bf16_f32
  return __builtin_bit_cast(uint32_t, h);
#else
  return 0;
#endif
}
// Item of a workgroup: hardware block ids go round the 8 XCDs in turn, so each
// XCD takes one contiguous range of items (neighbouring tiles and elements
// share an L2).
__device__ __forceinline__ int xcd_item(int bid, int nb) {
  const int x = bid & 7, q = nb >> 3, r = nb & 7;
  return x * q + min(x, r) + (bid >> 3);
}
__device__ __forceinline__ float comp_u(uint32_t w) { return __uint_as_float(w << 16); }
__device__ __forceinline__ float comp_v(uint32_t w) { return __uint_as_float(w & 0xffff0000u); }

// One Newmark step of a node component in the (u, w = v + dt/2 a_) form:
// Kahan w += dt a, Kahan u += dt w with the packed compensations kc.  `twice`
// advances it a second time (the field-list quirk's x component).  Which
// products are fused is written out, so that every kernel that finishes a
// node rounds the same way: the first time dt a joins its compensation in one
// fused operation, the second time as a product of its own.
__device__ __forceinline__ void newmark(float &u, float &w, uint32_t &kc, float a, float dt, bool twice) {
  float kw = comp_v(kc), ku = comp_u(kc);
  float y = fmaf(dt, a, -kw);
  float t = w + y;
  kw = (t - w) - y;
  w = t;
  y = fmaf(dt, w, -ku);
  t = u + y;
  ku = (t - u) - y;
  u = t;
  if (twice) {
    const float da = dt * a;
    {
#pragma clang fp contract(off)
      y = da - kw;
    }
    t = w + y;
    kw = (t - w) - y;
    w = t;
    y = fmaf(dt, w, -ku);
    t = u + y;
    ku = (t - u) - y;
    u = t;
  }
  kc = pack_comp(ku, kw);
}

// Per-element factor counts.
// Affine geometry (one Jacobian per element): acoustic Gsym (dim*(dim+1)/2);
// elastic Jinv (dim^2) + detJ (1).
// Pointwise geometry (per GLL node): acoustic w*vp^2*Gsym; elastic 2D
// Jinv(4)+w detJ(1)+C11,C13,C33,C55(4); elastic 3D Jinv(9)+w detJ(1)+9 c's.
__host__ __device__ inline int affine_geo_count(int dim, int physics) {
  return physics == SEM_ACOUSTIC ? dim * (dim + 1) / 2 : dim * dim + 1;
}
// Geometry modes of the element kernels: pointwise factors, per-element
// affine factors, or pointwise factors for the reference's quad operator
// (SEM_QUIRK_QUAD_JACOBIAN on non-affine quads: J^-1 and w det J of the
// QuadP1.h:20-27 Jacobian per node, J^-1 applied at the output node).
enum { kGeoPoint = 0, kGeoAffine = 1, kGeoQuadRef = 2 };
// With kGeoQuadRef the acoustic factors are Jinv(4) + w det J vp^2 (1).
__host__ __device__ inline int point_geo_count(int dim, int physics, int gmode = kGeoPoint) {
  if (physics == SEM_ACOUSTIC) return gmode == kGeoQuadRef ? 5 : dim * (dim + 1) / 2;
  return dim == 2 ? 9 : 19;
}
// Vertex material the fused kernels interpolate on the fly (stiffness only):
// acoustic {VP}; Elastic2D {C11,C13,C33,C55}; Elastic3D {RHO,VPV,VPH,VSV,VSH,ETA}.
__host__ __device__ inline int kernel_npar(int dim, int physics) {
  if (physics == SEM_ACOUSTIC) return 1;
  return dim == 2 ? 4 : 6;
}
__host__ __device__ inline int ref_npar(int dim, int physics) {
  if (physics == SEM_ACOUSTIC) return 1;
  return dim == 2 ? 5 : 6;
}

struct SrcDev {
  int32_t elem;     // sorted element position
  int32_t stf_off;  // offset of this source's STF samples
  int32_t load_off; // offset of nd*c load weights
  int32_t shot;     // shot slot within the group
};

// A receiver as k_receivers samples it: with its shot's field and step
// counter, so that no group descriptor stands between it and its samples.
struct RecDev {
  int32_t nodes_off; // offset of the owning element's nd node ids (field numbering)
  int32_t w_off;     // offset of nd Lagrange weights
  int32_t shot;      // shot slot within the group
  int32_t stride;    // floats between consecutive steps (R_shot * c)
  float *out;        // this receiver's step-0, component-0 sample
  const float *u;    // its shot's displacement, G floats per component
  const int64_t *step;  // its group's step counter
  int64_t G, nsteps;
};

// A receiver as the launch of its tile or element samples it.
struct TileRec {
  float *out;        // this receiver's step-0, component-0 sample
  int32_t w_off;     // offset of nd Lagrange weights
  int32_t shot;      // shot slot within the group
  int32_t stride;    // floats between consecutive steps
  int32_t elem;      // element of the tile; its number in the caller's order (element kernel)
};

// One tile of a logically Cartesian mesh (see tiles.cpp).
struct TileInfo {
  int32_t ex, ey, ez;  // elements per axis in this tile
  int32_t colour;      // lattice parity colour
  int32_t nint, nval;  // words: nodes in this tile alone | shared nodes | padding (from nval on)
  int32_t own;         // internal number of its first own node (the others follow)
  int32_t sh_off;      // first entry of its shared words in sh_part
  int32_t slots;       // its slot table
};

// Work item of a tile launch: shots [s0, s1) of one tile, its sources
// [src, src + nsrc) of the group's list and, where the launch samples them,
// the receivers [rec, rec + nrec) of its one shot.
struct TileItem {
  int32_t group, tile;
  uint16_t s0, s1;
  uint8_t ex, ey, ez, pad;
  uint16_t nint, nval;
  uint32_t own;
  int32_t sh_off, slots, src, nsrc, rec, nrec;
};

// One group = shots sharing a mesh, fields shot-major:
// field[(s*c + comp)*G + g] (each shot's field contiguous).
struct GroupDev {
  const uint32_t *conn;   // E x nd (sorted order, flags)
  const float *geo_e;     // affine: E x ng
  const float *par_e;     // E x nv x kpar
  const float *geo_p;     // pointwise: E x ngp x nd
  const float *mi;        // G
  // Newmark state: u, w = v + dt/2 a_ (what the update reads), a_ (written
  // for read-out only: v = w - dt/2 a_)
  float *u, *w, *ap;
  uint32_t *kc;           // Kahan compensations of u and w (bf16 pair per word)
  float *acc;
  const SrcDev *src;
  const float *stf;
  const float *load;
  int32_t nsrc;
  int32_t S;
  int64_t G;
  int64_t nsteps;
  int64_t *step;          // device step counter of this group
  float dt, acl;           // acl = dt/2 (Order2Newmark.cpp:89), host conversions of w
  int32_t quirks;
  int32_t pad;
  // tile kernel (structured meshes): fields in tile-major node numbering
  const uint32_t *tile_words;   // per tile: own nodes, shared ones, padding (colours: in node order, with flags)
  const uint32_t *tile_words_lat;  // the same in lattice order (high-occupancy colour launches)
  const uint32_t *tile_slot;    // slot tables, of each word: LDS lattice slot | kSlotDirichlet | place in the element results << 16
  const float *telem;     // per element in tile order: affine factors, then vertex material
  // coupled shots (fluid-solid pairs): external load added to a node's sum
  // at its first colour, null otherwise; a_ stored every step (the coupling
  // reads the velocities v = w - dt/2 a_ after each step)
  const float *ext;
  int32_t ap_always;
  // partial results of nodes shared by tiles or elements:
  // part[(s*c + comp)*part_stride + position]; the positions of the tiles'
  // shared words, or of every element node ([e][nd], like conn) with the list
  // of shared nodes
  int32_t c;
  int64_t part_stride;
  float *part;
  const int32_t *sh_part;
  const uint32_t *epos;
  const uint32_t *sh_node;
  const TileRec *rec;  // receivers by tile and shot (element kernel: by shot and element)
  const float *rec_w;  // their Lagrange weights
};

// Work item of an element launch: shots [s0, s1) of `count` elements of one
// group, in the launch's element list from `first` on; of a colour launch: every
// shot (s1 = 0) of the elements at sorted positions from `first` on.
struct WorkItem {
  int32_t group, first, count;
  uint16_t s0, s1;
  int32_t elem;       // first element's number in the caller's order
  int32_t rec, nrec;  // receivers in its elements (one-shot items): range of the group's `rec`
  int32_t pad;
};

// Work item of the shared-node launch: `count` nodes (at most kSharedNodes, or
// any number of one plane) of one class -- the nodes of m tiles or elements --, plane (shot and component)
// `plane` or, negative, every plane.
constexpr int kSharedNodes = 256;
struct NodeItem {
  int32_t group, count, m, plane;
  int64_t node;    // first node, or (listed) its place in the group's node list
  int64_t part;    // position of its first partial result
  int64_t stride;  // from one copy of a node to the next (nodes of the class)
  int32_t listed, pad;
};

// A class of shared nodes: n nodes of m tiles or elements each.
struct SharedClass {
  int m;
  int64_t n, node, part;  // as in NodeItem
};

// Every tile has the full Tx x Ty (x Tz) element box and its whole node
// lattice: elements and slots beyond a partial tile at the mesh edge are
// padding (element order -1, slot word kSlotEmpty).
struct TileSet {
  bool valid = false;
  int T[3] = {0, 0, 0};
  int64_t ntiles = 0, total_slots = 0;
  int64_t slots_per_tile = 0;        // (Tx N + 1)(Ty N + 1)(Tz N + 1)
  int elems_per_tile = 0;            // Tx Ty Tz
  int nt[3] = {0, 0, 0};             // tiles along each axis (x fastest)
  std::vector<TileInfo> info;
  std::vector<uint32_t> words;       // per tile, own nodes then shared ones, each in node order:
                                     // internal node | Dirichlet flag, or kSlotEmpty
  std::vector<uint16_t> slot_of;     // lattice slot of each word
  // shared nodes: internal nodes from `nown` on, `sh_n` of each class (2, 4
  // and 8 tiles); partial results per plane, and the positions of the tiles'
  // shared words in it
  int64_t nown = 0, nparts = 0;
  int64_t sh_n[3] = {0, 0, 0};
  std::vector<int32_t> sh_part;
  std::vector<int32_t> to_internal;  // DMPlex DOF -> internal node
  std::vector<int32_t> elem_order;   // tile-order position -> element (-1: padding)
  std::vector<int32_t> elem_pos;     // element -> tile-order position
};

// What the colour launches over the same tiles need, in a node numbering of
// their own (words: node | flags, or kSlotEmpty).
struct ColourTiles {
  bool valid = false;
  bool unfit = false;                // neighbouring tiles do not share all their nodes: no such numbering
  std::vector<int32_t> table;        // slot table of each tile
  std::vector<int32_t> to_internal;  // DMPlex DOF -> node
  uint32_t *d_words = nullptr;       // per tile, in node order
  uint32_t *d_words_lat = nullptr;   // acoustic: the same words in lattice order
  uint32_t *d_slot = nullptr;
  float *d_mi = nullptr;
  int32_t *d_to_int = nullptr;
};

// Tables of every kind of tile neighbourhood (colour_tile_tables), a table per type of
// slots_per_tile entries: rank among the nodes that the finishing tile finishes,
// that tile's place (3 x 3 x 3 around this one), axes along which the node is
// shared, kFlagFirst and kFlagLast; or kSlotEmpty.
constexpr int kRankBits = 15, kSharedShift = 20;
struct ColourTables {
  std::vector<int32_t> type;      // of each tile
  std::vector<uint32_t> first;    // first node that each tile finishes
  std::vector<int32_t> example;   // a tile of each type
  std::vector<uint32_t> words;    // in the words' order
  std::vector<uint32_t> lat;      // in lattice order
  std::vector<uint16_t> slot_of;  // lattice slot of each word
};
struct ColourTile {  // a tile as the kernels below read it
  int32_t type, slots, nval;
  uint32_t first;
};

// Kernel argument blocks (passed by value; recorded by graph capture).
struct FusedArgs {
  const GroupDev *groups;
  const WorkItem *items;   // element kernel
  const int32_t *elems;    // element kernel: the items' elements (null: one colour, the items' sorted positions)
  const TileItem *tiles;   // tile kernel
  const NodeItem *nodes;   // shared-node kernel
  int64_t first, count;    // element kernel, one colour without items: its elements of group `group`
  const float *u;          // accumulate-only pass on a caller's buffers (out set): input
  float *out;              // and result
  int32_t group;
  int32_t negate;          // accumulate-only pass: the sums are stored negated
  int32_t nitems;
  int32_t epb;
  int32_t koff;      // step offset within the captured block
  int32_t ku_only;   // 1: accumulate -K u into acc on every colour (no update)
  int32_t ap_koff;   // a_ (read out only) is stored at this step offset of the
                     // block -- its last -- and at a shot's last step
  int32_t pad;
};

struct PlainArgs {
  const uint32_t *conn;
  const float *geo_p;
  const float *uloc;
  float *aloc;
  const SrcDev *src;
  const float *stf;
  const float *load;
  const int64_t *step;
  int32_t nsrc;
  int32_t epb;
  int64_t E;
  int32_t koff;
  int32_t pad;
};

struct RecArgs {
  const RecDev *recs;
  const uint32_t *nodes;
  const float *weights;
  int32_t nrec;
  int32_t nd;
  int32_t koff;
  int32_t end;  // 1: the end of a block whose other steps the tile launches
                // have sampled: after each group's last step of the block
                // (koff, or the group's own last step)
};

// ---------------------------------------------------------------- launchers (kernels.hip)
int init_device_tables(int device);
int launch_affine_geometry(int dim, int physics, int64_t E, const double *vtx, float *geo,
                           hipStream_t st);
int launch_point_geometry(int dim, int order, int physics, int gmode, int64_t E, const double *vtx,
                          const double *vpar, int npar, float *geo_p, double *me, hipStream_t st);
int launch_mass_scatter(int64_t first, int64_t count, int nd, const uint32_t *conn,
                        const double *me, double *M, hipStream_t st);
int launch_reciprocal(int64_t G, const double *M, float *mi, hipStream_t st);
int launch_fill_f64(int64_t n, double *p, double v, hipStream_t st);
int launch_fill_f32(int64_t n, float *p, float v, hipStream_t st);
int launch_fill_i32(int64_t n, int32_t *p, int32_t v, hipStream_t st);
int launch_colour_touch(int64_t first, int64_t count, int nd, const uint32_t *conn, int32_t *hits,
                        hipStream_t st);
int launch_colour_count(int64_t G, int32_t *hits, unsigned long long *viol, hipStream_t st);
// Threads per block for EPB elements of nd nodes (multiple of 64).
inline int block_threads(int nd, int epb) { return ((nd * epb + 63) / 64) * 64; }
inline size_t fused_lds_bytes(int dim, int nd, int c, int epb) {
  return sizeof(float) * (size_t)epb * c * nd * (1 + dim);
}
int launch_fused(int dim, int order, int physics, int gmode, int nitems, int epb, int nd, int c,
                 const FusedArgs &a, hipStream_t st);
// Finishes the nodes shared by several tiles or elements (after the tile and
// element launches): one workgroup per item (a.nodes).
int launch_shared(const FusedArgs &a, hipStream_t st);
// First and last colours of the nodes of one colour's elements; then the gather
// map of one colour's elements (sorted order) with its flags.
int launch_conn_span(int64_t first, int64_t count, int nd, int colour, const int32_t *perm, const int32_t *raw,
                     int32_t *lo, int32_t *hi, hipStream_t st);
int launch_conn_flags(int64_t first, int64_t count, int nd, int colour, const int32_t *perm, const int32_t *raw,
                      const int32_t *lo, const int32_t *hi, const uint8_t *dir, uint32_t *conn, hipStream_t st);
// Nodes by their number of elements (the last class: that many or more): counts
// per block of nodes, then the classes' lists and the nodes' partial results
// (hits_next: elements per node in, first position out).
constexpr int kNodeClasses = 64, kClassNodes = 1024;
int launch_class_count(int64_t G, const int32_t *hits, int32_t *count, hipStream_t st);
int launch_class_list(int64_t G, const int32_t *first, const uint32_t *table, uint32_t *hits_next, uint32_t *stride,
                      uint32_t *list, hipStream_t st);
// Partial-result positions of one colour's elements (next: every node's next).
int launch_elem_pos(int64_t first, int64_t count, int nd, const uint32_t *conn, const uint32_t *stride,
                    uint32_t *next, uint32_t *pos, hipStream_t st);
int launch_permute_f32(int64_t n, const int32_t *to, const float *src, float *dst, hipStream_t st);
// Words of the colour launches from the tables of the tiles' types; the number
// of every node from its number in `words`, whose nodes of one, two, four and eight
// tiles begin at 0 and class0..2 (*bad is set where the tiles share others); and
// to[i] = number[from[i]].
int launch_colour_words(int64_t ntiles, int ntl, int nx, int nxy, const ColourTile *tiles, const uint32_t *entries,
                        uint32_t *words, hipStream_t st);
int launch_colour_numbers(int64_t ntiles, int ntl, int lx, int ly, int lxp, int lxyp, const ColourTile *tiles,
                          const uint32_t *lat, const uint32_t *words, const uint32_t *slots, uint32_t class0,
                          uint32_t class1, uint32_t class2, int32_t *number, int32_t *bad, hipStream_t st);
int launch_compose_i32(int64_t n, const int32_t *from, const int32_t *number, int32_t *to, hipStream_t st);
int launch_plain_gather(int64_t E, int nd, int C, int64_t G, const uint32_t *conn, const float *u,
                        float *uloc, hipStream_t st);
int launch_plain_stiffness(int dim, int order, int physics, int gmode, int64_t E, int nd, int c,
                           const PlainArgs &a, hipStream_t st);
int launch_plain_scatter(int64_t first, int64_t count, int nd, int C, int64_t G,
                         const uint32_t *conn, const float *aloc, float *acc, hipStream_t st);
// Newmark update in the (u, w = v + dt/2 a_) form: w += dt a, u += dt w.
int launch_plain_update(int64_t G, int C, int quirks, float dt, const float *mi, const float *acc,
                        const float *ext, float *u, float *w, float *ap, uint32_t *kc, hipStream_t st);
int launch_receivers(const RecArgs &a, int C, hipStream_t st);
int launch_read_field(int64_t n, int64_t i0, int64_t G, const int32_t *to, const float *f, const float *ap,
                      double half_dt, double *out, hipStream_t st);
// Advances every group's step counter by k (clamped at its nsteps).
int launch_advance(int ngroups, const GroupDev *groups, int64_t k, hipStream_t st);

// ---------------------------------------------------------------- tile kernel (tile_kernels.hip)
// Modes of the tile kernel: every tile in one launch, partial results at nodes
// shared by tiles; the same with these stored past the caches (3-D elastic); one
// launch per tile colour, sums of shared nodes in HBM; the same with more waves per
// SIMD (acoustic).
enum { kTileParts, kTilePartsPast, kTileColours, kTileColoursHigh };
int init_tile_tables(int device);
struct TileKernelInfo {
  size_t lds_bytes;  // 0: no kernel compiled for this order and tile shape
  int threads;
  int lxp, lxyp;    // LDS lattice: slot of node (x, y, z) = x + lxp y + lxyp z
  int elem_stride;  // LDS words between the results of consecutive elements
};
TileKernelInfo tile_kernel_info(int dim, int order, int physics, const int *T);
// Compiled tile shapes for (dim, order, physics): up to max triples; returns the count.
int tile_kernel_shapes(int dim, int order, int physics, int *shapes, int max);
// Readies the kernel of this shape and mode (LDS limit) and returns its workgroups per CU.
int tile_kernel_prepare(int dim, int order, int physics, const int *T, int mode, int *per_cu);
// One workgroup per item (a.tiles).
int launch_tile(int dim, int order, int physics, const int *T, bool diag, int mode, const FusedArgs &a,
                hipStream_t st);

}  // namespace sem

// ---------------------------------------------------------------- public structs
struct sem_mesh {
  int device = 0, dim = 0, order = 0, n = 0, nd = 0, physics = 0, c = 0, nv = 0, quirks = 0;
  int64_t E = 0, V = 0, G = 0;
  int ncol = 0;
  bool affine = false;
  std::vector<int64_t> col_start;  // ncol+1 positions in sorted order
  std::vector<int32_t> perm;       // sorted position -> original element
  std::vector<int32_t> inv_perm;   // original element -> sorted position
  std::vector<int32_t> conn;       // original order E x nd (plain)
  std::vector<int32_t> colour;     // original order
  std::vector<double> vtx;         // original order E x nv x dim
  std::vector<double> vpar;        // original order E x nv x npar
  std::vector<double> bbox;        // original order E x 2 dim
  sem::ElementBins bins;           // point location
  std::vector<uint8_t> dirichlet;  // G (empty = none)
  // device
  hipStream_t stream = nullptr;
  uint32_t *d_conn = nullptr;      // sorted E x nd with flags
  float *d_geo_e = nullptr;        // affine per-element factors
  float *d_par_e = nullptr;        // per-element vertex material (kernel set)
  float *d_geo_p = nullptr;        // pointwise factors (lazy)
  float *d_mi = nullptr;
  // element kernel with partial results (ensure_elem_parts): shared-node
  // classes, partial results per plane, their positions ([e][nd], sorted) and
  // the shared nodes class by class
  int elem_parts = -1;             // 1 built, 0 not taken (memory), -1 not decided
  int64_t nparts = 0;
  std::vector<sem::SharedClass> classes;
  uint32_t *d_epos = nullptr, *d_sh_node = nullptr;  // (one buffer)
  // allocation-free operator on meshes small enough to keep partial results
  // for it (setup_apply): one buffer with the descriptor, the step counter (0),
  // the items and the partial results
  unsigned char *d_apply_buf = nullptr;
  sem::GroupDev *d_apply = nullptr;
  sem::WorkItem *d_apply_items = nullptr;
  int32_t *d_apply_elems = nullptr;
  sem::NodeItem *d_apply_nodes = nullptr;
  int apply_nitems = 0, apply_nnodes = 0;
  double *d_vtx = nullptr;         // sorted E x nv x dim (FP64)
  double *d_vpar = nullptr;        // sorted E x nv x npar (FP64)
  // tile path (logically Cartesian affine meshes)
  sem::TileSet tiles;
  uint32_t *d_tile_words = nullptr;
  uint32_t *d_tile_slot = nullptr;
  std::vector<uint32_t> tile_slots;  // its host copy
  int32_t *d_sh_part = nullptr;
  float *d_telem = nullptr, *d_mi_int = nullptr;
  int32_t *d_to_int = nullptr;  // DMPlex DOF -> internal node
  sem::ColourTiles ctiles;  // built by the first group that takes colour launches
  bool tile_diag = false;  // every element's affine factors diagonal (axis-aligned lattice)
  // while the mesh is created: one buffer for the steps' temporary data (an
  // allocation and a release of some 100 us each for every one of them otherwise)
  unsigned char *d_temp = nullptr;
  size_t temp_bytes = 0;
  size_t bytes = 0;       // device bytes held (tile path included)
  size_t tile_bytes = 0;  // of which the tile path
};

namespace sem {
struct Shot;
struct Group;
}  // namespace sem

struct sem_batch;

namespace sem {
// Geometry mode of a mesh's element kernels (kGeo*).
inline int geo_mode(const sem_mesh *m) {
  if (m->affine) return kGeoAffine;
  return (m->dim == 2 && (m->quirks & SEM_QUIRK_QUAD_JACOBIAN)) ? kGeoQuadRef : kGeoPoint;
}
// Mode of the pointwise factors (plain path, mass): the reference quad
// operator where it differs from the consistent one, else kGeoPoint.
inline int pointwise_mode(const sem_mesh *m) {
  return geo_mode(m) == kGeoQuadRef ? kGeoQuadRef : kGeoPoint;
}
// Tiles a logically Cartesian mesh; 0 = tiled, 1 = not eligible.
int build_tiles(sem_mesh *m, int Tx, int Ty, int Tz, TileSet &ts);
// Numbering and words of the colour launches by kinds of tiles.
void colour_tile_tables(const sem_mesh *m, ColourTables &c);
}  // namespace sem
