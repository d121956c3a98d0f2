// Allocation-free stiffness application: sem_mesh_apply_stiffness_noalloc.
//
// sem_mesh_apply_stiffness builds a one-shot batch (group descriptor, step
// counter, work items, fields) in freshly allocated device memory.  This
// variant takes device input and output buffers from the caller and keeps
// everything else beforehand, so callers that may not call hipMalloc (graph
// capture, tight serving loops) can use it.  It runs the element kernel on the
// DMPlex-ordered fields directly:
//  - on meshes whose partial results are little (setup_apply), in two launches --
//    every element, then the shared nodes -- with the descriptor, the partial
//    results and the items kept with the mesh since its creation;
//  - on larger ones colour by colour, with the descriptor and the step counter
//    in a file-scope device array; a colour's blocks take its elements in order
//    (no work items).  There a colour runs for long enough that its launch does
//    not matter, and a mesh keeps no second set of partial results.
// The sums run in the order of the colours in both, so results are the same.
// Every kernel here writes the scratch itself (no memset, no host copy), so the
// calls can be captured.  24x23x22 deformed elastic hexes: 8 colours with
// work-item and sign launches 121 us, the colours alone 98 us, two launches
// 71 us.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstring>
#include <mutex>

#include "batch.h"
#include "sem_internal.h"

namespace sem {
namespace {

// Scratch: [0, 256) group descriptor, [256, 512) step counter.
constexpr size_t kScratchBytes = 512;
// Largest number of blocks a colour may need: the entry point's documented
// limit (the kernel itself takes any number a launch does).
constexpr int64_t kMaxBlocks = 262112;
static_assert(sizeof(GroupDev) <= 256, "group descriptor exceeds its scratch slot");

static __device__ __align__(256) unsigned char scratch[kScratchBytes];

// Per-device address of `scratch` (hipGetSymbolAddress with that device
// current); the array's host-side name is not a device address.
std::mutex g_mu;
void *g_ptr[64] = {nullptr};

int scratch_ptr(int device, unsigned char **out) {
  std::lock_guard<std::mutex> lk(g_mu);
  if (device < 0 || device >= 64) { set_error("device index"); return -1; }
  if (!g_ptr[device]) {
    void *p = nullptr;
    hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !p) {
      set_error(std::string("scratch address: ") + hipGetErrorString(e));
      return -2;
    }
    g_ptr[device] = p;
  }
  *out = static_cast<unsigned char *>(g_ptr[device]);
  return 0;
}

__global__ void k_put_group(GroupDev g, GroupDev *dst, int64_t *step) {
  if (threadIdx.x == 0 && blockIdx.x == 0) {
    *dst = g;
    *step = 0;
  }
}

int launched(const char *what) {
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) {
    set_error(std::string(what) + ": " + hipGetErrorString(e));
    return -2;
  }
  return 0;
}

// A mesh keeps what the two launches need if that is little: at most 64 MiB of
// partial results, and less than a thousandth of the device's free memory with
// their positions, so that meshes whose owners never call the operator take no
// memory that is missed.  (Creating a mesh takes 0.8 ms for it.)
constexpr int64_t kMaxKeptParts = (int64_t)64 << 20;  // bytes

}  // namespace

int setup_apply(sem_mesh *m) {
  // partial results number at most one per element node, their positions one
  if (4 * m->c * m->E * m->nd > kMaxKeptParts) return 0;
  size_t free_bytes = 0, total = 0;
  if (hipMemGetInfo(&free_bytes, &total) != hipSuccess || 4 * (m->c + 1) * m->E * m->nd > (int64_t)(free_bytes / 1024))
    return 0;
  SEM_TRY(ensure_elem_parts(m));
  if (m->elem_parts != 1) return 0;
  const int epb = default_epb(m->nd);
  std::vector<WorkItem> items;
  for (int64_t f = 0; f < m->E; f += epb)
    items.push_back(WorkItem{0, (int32_t)f, (int32_t)std::min<int64_t>(epb, m->E - f), 0, 1, 0, 0, 0, 0});
  std::vector<NodeItem> nodes;
  for (const SharedClass &c : m->classes)
    for (int64_t f = 0; f < c.n; f += kSharedNodes)
      for (int p = 0; p < m->c; ++p)
        nodes.push_back(NodeItem{0, (int32_t)std::min<int64_t>(kSharedNodes, c.n - f), c.m, p, c.node + f,
                                 c.part + f, c.n, 1, 0});
  // descriptor and step counter, work items, node items, elements; partial results
  auto pad = [](size_t n) { return (n + 255) / 256 * 256; };
  const size_t o_items = 512, o_nodes = o_items + pad(items.size() * sizeof(WorkItem)),
               o_elems = o_nodes + pad(nodes.size() * sizeof(NodeItem)), o_part = o_elems + pad((size_t)m->E * 4);
  std::vector<unsigned char> host(o_part, 0);
  SEM_TRY(dalloc(&m->d_apply_buf, o_part + (size_t)(m->c * m->nparts) * 4, &m->bytes));
  GroupDev h{};
  h.conn = m->d_conn;
  h.geo_e = m->d_geo_e;
  h.par_e = m->d_par_e;
  h.geo_p = m->d_geo_p;
  h.mi = m->d_mi;
  h.S = 1;
  h.G = m->G;
  h.nsteps = 1;
  h.step = reinterpret_cast<int64_t *>(m->d_apply_buf + 256);
  h.quirks = m->quirks;
  h.c = m->c;
  h.part = reinterpret_cast<float *>(m->d_apply_buf + o_part);
  h.part_stride = m->nparts;
  h.epos = m->d_epos;
  h.sh_node = m->d_sh_node;
  std::memcpy(host.data(), &h, sizeof h);
  std::copy(items.begin(), items.end(), reinterpret_cast<WorkItem *>(host.data() + o_items));
  std::copy(nodes.begin(), nodes.end(), reinterpret_cast<NodeItem *>(host.data() + o_nodes));
  std::copy(m->inv_perm.begin(), m->inv_perm.end(), reinterpret_cast<int32_t *>(host.data() + o_elems));
  HIPCHK(hipMemcpyAsync(m->d_apply_buf, host.data(), o_part, hipMemcpyHostToDevice, m->stream));
  HIPCHK(hipStreamSynchronize(m->stream));
  m->d_apply = reinterpret_cast<GroupDev *>(m->d_apply_buf);
  m->d_apply_items = reinterpret_cast<WorkItem *>(m->d_apply_buf + o_items);
  m->d_apply_nodes = reinterpret_cast<NodeItem *>(m->d_apply_buf + o_nodes);
  m->d_apply_elems = reinterpret_cast<int32_t *>(m->d_apply_buf + o_elems);
  m->apply_nitems = (int)items.size();
  m->apply_nnodes = (int)nodes.size();
  return 0;
}

}  // namespace sem

using namespace sem;

extern "C" int sem_mesh_apply_stiffness_noalloc(sem_mesh *m, const float *u, float *ku, void *stream) {
  if (!m || !u || !ku) { set_error("null argument"); return -1; }
  const int epb = default_epb(m->nd);
  int64_t worst = 0;
  for (int c = 0; c < m->ncol; ++c)
    worst = std::max<int64_t>(worst, (m->col_start[c + 1] - m->col_start[c] + epb - 1) / epb);
  if (worst > kMaxBlocks) {
    set_error("mesh too large for the allocation-free stiffness: a colour needs " +
              std::to_string(worst) + " blocks, at most " + std::to_string(kMaxBlocks) +
              " are allowed (at most " + std::to_string(kMaxBlocks * epb) + " elements per colour)");
    return -1;
  }
  HIPCHK(hipSetDevice(m->device));
  hipStream_t st = stream ? static_cast<hipStream_t>(stream) : m->stream;
  FusedArgs a{};
  a.epb = epb;
  a.ku_only = 1;
  a.negate = 1;
  a.u = u;
  a.out = ku;
  if (m->d_apply) {
    a.groups = m->d_apply;
    a.items = m->d_apply_items;
    a.elems = m->d_apply_elems;
    a.nitems = m->apply_nitems;
    SEM_TRY(launch_fused(m->dim, m->order, m->physics, geo_mode(m), a.nitems, epb, m->nd, m->c, a, st));
    a.nodes = m->d_apply_nodes;
    a.nitems = m->apply_nnodes;
    SEM_TRY(launch_shared(a, st));
    if (!stream) HIPCHK(hipStreamSynchronize(st));
    return 0;
  }
  unsigned char *base = nullptr;
  SEM_TRY(scratch_ptr(m->device, &base));
  GroupDev *d_group = reinterpret_cast<GroupDev *>(base);
  int64_t *d_step = reinterpret_cast<int64_t *>(base + 256);

  GroupDev h{};
  h.conn = m->d_conn;
  h.geo_e = m->d_geo_e;
  h.par_e = m->d_par_e;
  h.geo_p = m->d_geo_p;
  h.mi = m->d_mi;
  h.S = 1;
  h.G = m->G;
  h.nsteps = 1;
  h.step = d_step;
  h.quirks = m->quirks;
  hipLaunchKernelGGL(k_put_group, dim3(1), dim3(64), 0, st, h, d_group, d_step);
  SEM_TRY(launched("stiffness descriptor"));
  a.groups = d_group;
  for (int c = 0; c < m->ncol; ++c) {
    a.first = m->col_start[c];
    a.count = m->col_start[c + 1] - a.first;
    a.nitems = (int32_t)((a.count + epb - 1) / epb);
    SEM_TRY(launch_fused(m->dim, m->order, m->physics, geo_mode(m), a.nitems, epb, m->nd, m->c, a, st));
  }
  if (!stream) HIPCHK(hipStreamSynchronize(st));
  return 0;
}
