// Column-mapped tile kernel of the MI355X SEM path (gfx950).
//
// Structured (logically Cartesian, affine) meshes are cut into tiles of
// TX x TY (x TZ) elements whose node lattice is staged in LDS; one workgroup
// takes one tile (for some or all shots of the group) and one launch takes
// every tile.  A step is two launches: k_tile computes every tile's results
// and finishes the nodes that lie in one tile alone; for a node shared by 2,
// 4 or 8 tiles each of them writes its partial result, and k_shared sums them
// in a fixed order and finishes the node.
// One thread owns one node column of one element: the column runs along the
// last reference axis (eta in 2-D, zeta in 3-D), so the derivative along it
// is a register-only product with wave-uniform D entries, and only the
// lateral derivatives read the LDS lattice.  Columns run in chunks of at most
// 512 threads, all chunks equally full.  Per shot:
//   gather  u of every lattice slot -> LDS (the first shot's with the tile's
//           words and element data; every later shot's, with the finish
//           inputs of the first slots, during the previous shot's face
//           passes, so each shot waits for one memory round trip);
//   column  reference gradient and J^-T flux per node; lateral fluxes go to
//           LDS, the column flux stays in registers; the test-and-integrate
//           result (-Ku, zero on Dirichlet rows, plus source loads) is
//           stored element-locally in LDS;
//   faces   element copies of shared nodes are summed in fixed passes along
//           x, y (and z), after which the element of highest lattice
//           position containing a node holds the tile's total for it;
//   finish  a slot shared with other tiles is stored as this tile's partial
//           result; any other is finished: a = mi f;
//           Kahan w += dt a; Kahan u += dt w; a_ = a, where w = v + dt/2 a_
//           is the state the update reads (Order2Newmark.cpp:68-115:
//           v += dt/2 (a + a_), u += dt v + dt^2/2 a, a_ = a, rewritten so
//           that a_ is only written).
// One launch over every tile, instead of one per tile colour with nodes
// finished by the last colour, fills the chip and takes one latency chain per
// step instead of 4 (2-D) or 8 (3-D).  Measured per step, one MI355X, colours ->
// now: 100^2 acoustic quads 33 -> 10.1 us, 4 shots of 331x287 acoustic quads 97 ->
// 39 us, 500^2 elastic quads 70 -> 52 us, 64^3 acoustic hexes 285 -> 202 us,
// 27x25x23 elastic hexes of order 3 78 -> 24 us, 8 shots of 32^3 elastic hexes
// 486 -> 456 us, 4 shots of 64^3 1833 -> 1808 us (there HBM runs at 3.5 of the 4.7
// TB/s of a copy in k_tile and at 4.3 in k_shared, and the VALU is 62 % busy: two
// 128-register workgroups a CU).  In large 3-D batches the launches' latencies
// matter no more and the scattered shared nodes cost bandwidth (k_tile 3.6 TB/s
// against 4.2): there the tiles run one launch per colour (MODE), on a node
// numbering of its own in which the tile that finishes a node holds it, with
// the sums of shared nodes in HBM between the colours; batch.cpp says from
// which size on.  32 shots of 32^3 to 96^3 elastic hexes: one launch 17.49 ms,
// colours 16.11.
// The operator is the one of TensorQuad.cpp:176-210/:350-397 and
// Hexahedra.cpp:579-754 (sum-factorised gradient, J^-T contraction,
// test-and-integrate) with Scalar.cpp:42-71, Elastic2D.cpp:53-82 and
// Elastic3D.cpp:33-54/:70-118 material laws.  All sums are in a fixed order,
// so results are reproducible bit for bit.
#include <hip/hip_runtime.h>

#include <atomic>
#include <cstring>

#include "sem_internal.h"
#include "tile_layout.h"

namespace sem {

namespace {

constexpr int kTileMaxN = 8;

// GLL points, weights and derivative matrix of order N evaluated at compile
// time, so that every wave-uniform table entry becomes an instruction
// literal.  Points: interior roots of P_N' by Newton from the Chebyshev-
// Gauss-Lobatto guesses; w_j = 2 / (N (N+1) P_N(x_j)^2); D[i][m] = l'_m(x_i)
// = P_N(x_i) / (P_N(x_m) (x_i - x_m)) off the diagonal, -+N(N+1)/4 at the
// two end points and 0 elsewhere on the diagonal.
constexpr double cx_cos(double x) {
  double term = 1.0, sum = 1.0;
  const double x2 = x * x;
  for (int k = 1; k < 40; ++k) {
    term *= -x2 / ((2.0 * k - 1.0) * (2.0 * k));
    sum += term;
  }
  return sum;
}

template <int N>
struct GllC {
  double x[N + 1], w[N + 1], D[(N + 1) * (N + 1)];
  constexpr GllC() : x(), w(), D() {
    const double pi = 3.14159265358979323846;
    double PN[N + 1] = {};
    for (int j = 0; j <= N; ++j) x[j] = -cx_cos(pi * j / N);
    for (int it = 0; it < 60; ++it)
      for (int j = 0; j <= N; ++j) {
        double p0 = 1.0, p1 = x[j];
        for (int k = 2; k <= N; ++k) {
          const double p2 = ((2.0 * k - 1.0) * x[j] * p1 - (k - 1.0) * p0) / k;
          p0 = p1;
          p1 = p2;
        }
        PN[j] = p1;
        if (j > 0 && j < N) x[j] -= (x[j] * p1 - p0) / ((N + 1) * p1);
      }
    for (int j = 0; j <= N; ++j) w[j] = 2.0 / (N * (N + 1.0) * PN[j] * PN[j]);
    for (int i = 0; i <= N; ++i)
      for (int m = 0; m <= N; ++m)
        D[i * (N + 1) + m] = i != m ? PN[i] / (PN[m] * (x[i] - x[m]))
                                    : (i == 0 ? -N * (N + 1.0) / 4.0 : (i == N ? N * (N + 1.0) / 4.0 : 0.0));
  }
};

// Compile-time table entries (arguments must be constants after unrolling).
template <int N>
__device__ __forceinline__ float gD(int i, int m) {
  constexpr GllC<N> g{};
  return (float)g.D[i * (N + 1) + m];
}
template <int N>
__device__ __forceinline__ float gW(int i) {
  constexpr GllC<N> g{};
  return (float)g.w[i];
}
template <int N>
__device__ __forceinline__ float gX(int i) {
  constexpr GllC<N> g{};
  return (float)g.x[i];
}

struct TileTables {
  float D[(kTileMaxN + 1) * (kTileMaxN + 1)];  // D[i*n+m] = l'_m(xi_i)
  float w[kTileMaxN + 1];
  float xi[kTileMaxN + 1];
};
__constant__ TileTables t_tab[kTileMaxN + 1];

// x, opaque to the compiler: what is computed from it inside a loop is not
// kept in registers across the loop
__device__ __forceinline__ uint32_t again(uint32_t x) {
  asm volatile("" : "+v"(x));
  return x;
}

// a + b never fused with a product feeding it (per-operation contract flag)
__device__ __forceinline__ float add_unfused(float a, float b) {
#pragma clang fp contract(off)
  return a + b;
}

// P1 vertices (QuadP1.h:98-108, HexP1.cpp:242-298): the multilinear weight
// of vertex v at (a, b[, t]) is prod (1 + s_i x_i) / 2^DIM with the vertex's
// signs s.  In 2-D the column coordinate t is eta.  Along the column the
// weights are linear in t, so the material is fixed by its values on the two
// end faces t = -1 and t = +1, where only that face's vertices take part.
template <int DIM>
__device__ __forceinline__ int p1_tsign(int v) {
  constexpr signed char ts[8] = {-1, -1, -1, -1, 1, 1, 1, 1};
  return DIM == 2 ? (v >= 2 ? 1 : -1) : ts[v];
}
// weight of vertex v on its own end face (t = its sign)
template <int DIM>
__device__ __forceinline__ float p1_face(int v, float a, float b) {
  if (DIM == 2) {
    const float sa = (v == 1 || v == 2) ? 1.f : -1.f;
    return 0.5f * (1.f + sa * a);
  }
  constexpr signed char hs[8][2] = {{-1, -1}, {-1, 1}, {1, 1}, {1, -1}, {-1, -1}, {1, -1}, {1, 1}, {-1, 1}};
  return 0.25f * (1.f + hs[v][0] * a) * (1.f + hs[v][1] * b);
}

// DG: every element's J^-1 (and, acoustic, its G = det J J^-1 J^-T) is
// diagonal (axis-aligned lattices), so the contractions keep their diagonal
// terms only; the terms dropped are exact zeros, so results are those of the
// general kernel.
// MODE: partial results at shared nodes (kTileParts; kTilePartsPast: stored past
// the caches), or one launch per tile colour with the sums of shared nodes in HBM
// (kTileColours; kTileColoursHigh: its acoustic high-occupancy variant).
template <int DIM, int N, int PHYS, int TX, int TY, int TZ, bool DG, int MODE>
__global__ void __launch_bounds__((TS<DIM, N, PHYS, TX, TY, TZ, MODE == kTileColoursHigh>::BT))
    __attribute__((amdgpu_waves_per_eu(TS<DIM, N, PHYS, TX, TY, TZ, MODE == kTileColoursHigh>::MINW)))
    k_tile(FusedArgs A) {
  constexpr bool HO = MODE == kTileColoursHigh, COL = MODE == kTileColours || HO;
  using T = TS<DIM, N, PHYS, TX, TY, TZ, HO>;
  constexpr int n = T::n, C = T::C, ND = T::ND, NL = T::NL;
  static_assert(HO || T::NIT == T::KF, "every slot's finish inputs are loaded ahead");
  extern __shared__ float lds[];
  float *su = lds;
  uint32_t *sw = reinterpret_cast<uint32_t *>(lds + T::O_SW);
  float *sF = lds + T::O_SF;
  float *sK = lds + T::O_SK;
  float *sE = lds + T::O_SE;
  int *sS = reinterpret_cast<int *>(lds + T::O_SS);  // {element, shot, stf_off, load_off} of each source
  float *sD = lds + T::O_SD;  // GLL derivative matrix

  // everything a workgroup needs to know of its tile comes with its item, so
  // that the tables, the tile's own nodes and the group's step counter are
  // loaded together, two dependent loads (item, group) after the start
  const TileItem W = glb(A.tiles)[xcd_item(blockIdx.x, gridDim.x)];
  const auto &G = glb(A.groups)[W.group];
  const int tid = threadIdx.x;
  const TileTables &TT = t_tab[N];
  // descriptor fields, read once: G sits in global memory, so a field read
  // after a global store would be reloaded (the compiler cannot rule out
  // aliasing), and waiting for that load would wait for every store before it
  const gptr<float> gu = glb(G.u);
  const gptr<float> gw = glb(G.w);
  const gptr<float> gap = glb(G.ap);
  const gptr<uint32_t> gkc = glb(G.kc);
  const gptr<float> gpart = glb(G.part), gacc = glb(G.acc);
  const gptr<const float> gext = glb(G.ext);
  const gptr<const uint32_t> gmi = (gptr<const uint32_t>)glb(G.mi);
  const int64_t PS = G.part_stride;
  const uint32_t GG = (uint32_t)G.G;
  const int ex = W.ex, ey = W.ey, ez = W.ez;
  // words of nodes in this tile alone (k < nint; node own + k), then shared
  // ones (k < nval), then padding
  const int nint = W.nint, nval = W.nval;
  const uint32_t own = W.own;
  const uint32_t s_end = W.s1;  // shots [s0, s1)
  const float gdt = G.dt;
  const bool upd = !A.ku_only, has_ext = G.ext != nullptr;
  const int64_t step = *glb(G.step) + A.koff;
  const bool over = step >= G.nsteps;

  // ---- the column this thread owns in every chunk
  const int ec = tid / T::NCOL;
  const int col = tid - ec * T::NCOL;
  const int ci = col % n;
  const int cj = DIM == 3 ? col / n : 0;
  // (loads of its quadrature data go out with the staging loads)
  const float wi = TT.w[ci], wj = DIM == 3 ? TT.w[cj] : 1.f;
  const float xa = TT.xi[ci], xb = DIM == 3 ? TT.xi[cj] : 0.f;

  // ---- once per tile: node words, element data, sources inside the tile,
  // and the lattice of the first shot (every later shot's lattice is loaded
  // during the previous shot's face passes).  Thread tid owns the tile words
  // k = tid + r BT, which come in node order, so a wave's global accesses
  // are coalesced.  Outside the column phase each thread writes and reads
  // only its own slots of su.
  // Per word: its LDS lattice slot and the place of its total in the element
  // results (low 15 bits and high half), and its inverse mass (own nodes) or
  // partial-result position (shared ones), kept for all the tile's shots.
  // (High occupancy: the words come in lattice order, so slots need no table,
  // and inverse masses are read with the other finish inputs.)
  uint32_t slr[HO ? 1 : T::NIT], mik[HO ? 1 : T::NIT];
  const auto slot = [&](int r) {  // (colours: -1 past the end)
    const int k = tid + r * T::BT;
    if constexpr (HO) return k < T::NTL ? T::lds_slot(k) : -1;
    else return COL && k >= T::NTL ? -1 : (int)(slr[r] & kSlotMask);
  };
  constexpr int NRW = (ND + 63) / 64;
  float rw[NRW];
  int rec_c = -1, rec_e = 0;
  gptr<float> rec_out = nullptr;
  {
    const gptr<const uint32_t> words = glb(HO ? G.tile_words_lat : G.tile_words) + (int64_t)W.tile * T::NTL;
    const gptr<const uint32_t> slots = glb(G.tile_slot) + (int64_t)W.slots * T::NTL;
    const gptr<const uint32_t> gpos = (gptr<const uint32_t>)glb(G.sh_part) + W.sh_off;
    uint32_t wv[T::NIT];  // node | flags (own nodes: see kSlotDirichlet below)
#pragma unroll
    for (int r = 0; r < T::NIT; ++r) {
      const int k = min(tid + r * T::BT, T::NTL - 1);
      if constexpr (COL) {
        wv[r] = tid + r * T::BT < T::NTL ? words[k] : kSlotEmpty;
        if constexpr (!HO) slr[r] = slots[k];
      } else {
        slr[r] = slots[k];
        // (own nodes need no word; every lane loads all the same, those of the own
        // nodes the first shared one: with a branch around it the compiler waits
        // for each word before the next load, 64^3 acoustic hexes 202 -> 220 us)
        const uint32_t word = words[max(k, min(nint, T::NTL - 1))];
        wv[r] = k >= nint ? word : own + k;
        const gptr<const uint32_t> src = k < nint ? gmi + own + k : gpos + (min(k, nval - 1) - nint);
        mik[r] = nval > nint || k < nint ? *src : 0u;
      }
    }
    constexpr int NEI = (T::E * T::NED + T::BT - 1) / T::BT;
    static_assert(n * n <= T::BT && kTileMaxSrc <= T::BT, "staged one entry per thread");
    const gptr<const float> te = glb(G.telem) + (int64_t)W.tile * (T::E * T::NED);
    float ev[NEI];
#pragma unroll
    for (int q = 0; q < NEI; ++q) ev[q] = te[min(tid + q * T::BT, T::E * T::NED - 1)];
    const float dv = TT.D[min(tid, n * n - 1)];
    // receivers of this item (one-shot items only, one wave per receiver
    // component): their weights come with the staging loads
    if (!COL) rec_c = (tid >> 6) < W.nrec * C && A.koff > 0 && upd ? (tid >> 6) % C : -1;
    if (!COL && rec_c >= 0) {
      const TileRec R = glb(G.rec)[W.rec + (tid >> 6) / C];
      const gptr<const float> w = glb(G.rec_w) + R.w_off;
#pragma unroll
      for (int q = 0; q < NRW; ++q) rw[q] = w[min((tid & 63) + 64 * q, ND - 1)];
      rec_e = R.elem;
      rec_out = glb(R.out) + (step - 1) * R.stride + rec_c;
    }
    float uv[T::NIT][C];
    if constexpr (COL && !HO) {
#pragma unroll
      for (int r = 0; r < T::NIT; ++r)
        mik[r] = wv[r] != kSlotEmpty && (wv[r] & kFlagLast) && upd ? gmi[wv[r] & kNodeMask] : 0u;
    }
#pragma unroll
    for (int r = 0; r < T::NIT; ++r) {
      const uint32_t g = wv[r] == kSlotEmpty ? own : (wv[r] & kNodeMask);
#pragma unroll
      for (int c = 0; c < C; ++c) uv[r][c] = gu[((uint32_t)W.s0 * C + c) * GG + g];
    }
    if (over) return;  // uniform across the block; every load above is in range all the same
    if (tid < W.nsrc) {
      const SrcDev sd = glb(G.src)[W.src + tid];
      sS[4 * tid + 0] = sd.elem - W.tile * T::E;
      sS[4 * tid + 1] = sd.shot;
      sS[4 * tid + 2] = sd.stf_off;
      sS[4 * tid + 3] = sd.load_off;
    }
    if (tid < n * n) sD[tid] = dv;
#pragma unroll
    for (int q = 0; q < NEI; ++q) {
      const int i = tid + q * T::BT;
      if (i < T::E * T::NED) sE[i] = ev[q];
    }
#pragma unroll
    for (int r = 0; r < T::NIT; ++r) {
      if (COL ? slot(r) < 0 : tid + r * T::BT >= nval) continue;
      const int l = slot(r);
      sw[l] = wv[r];
#pragma unroll
      for (int c = 0; c < C; ++c) su[c * T::NTLP + l] = uv[r][c];
    }
    if (!COL && (slr[0] & kSlotDirichlet)) {
#pragma unroll 1
      for (int k = tid; k < nint; k += T::BT) sw[slots[k] & kSlotMask] = words[k];
    }
  }

  const bool lane = ec < T::EC;
  const float wl = DIM == 3 ? wi * wj : wi;
  const int pl = ci + (DIM == 3 ? n * cj : 0);  // element-local index of the column's node 0

  const bool q3 = (C >= 2) && (G.quirks & SEM_QUIRK_NEWMARK3D);  // {x, y, x}: x twice, z never
  // a_ is only read out (v = w - dt/2 a_, a_ itself): stored at the block's
  // last step and at the shot's last step, where a read-out can follow
  const bool wap = A.koff == A.ap_koff || step + 1 >= G.nsteps || G.ap_always;

  // no staging load is left in flight: one that some path never reads would
  // make the loop below wait for every store before the reuse of its register
  __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0) expcnt(7) lgkmcnt(15)
  __syncthreads();  // tile data and the first shot's lattice staged

  // ---- receivers in this tile: su holds u after the previous step of the
  // block, sampled as k_receivers samples it (the same lanes and butterfly)
  if (!COL && rec_c >= 0) {
    const int ln = tid & 63;
    const int ea = rec_e % TX, eb = (rec_e / TX) % TY, ec3 = DIM == 3 ? rec_e / (TX * TY) : 0;
    const float *ue = su + rec_c * T::NTLP + ea * N + T::LXP * (eb * N) + (DIM == 3 ? T::LXYP * (ec3 * N) : 0);
    float sum = 0.f;
#pragma unroll
    for (int q = 0; q < NRW; ++q) {
      const int p = ln + 64 * q, pj = p / n;
      if (p < ND) sum = fmaf(rw[q], ue[(p - pj * n) + (DIM == 3 ? T::LXP * (pj % n) + T::LXYP * (pj / n) : T::LXP * pj)], sum);
    }
    for (int off = 32; off > 0; off >>= 1) sum += __shfl_xor(sum, off);
    if (ln == 0) *rec_out = sum;
  }

  for (uint32_t s = W.s0; s < s_end; ++s) {
    // ---- columns, one chunk of elements at a time
#pragma unroll 1
    for (int ch = 0; ch < T::NCH; ++ch) {
      if (ch > 0) __syncthreads();  // previous chunk has read its lateral fluxes
      const int e = ch * T::EC + ec;
      bool act = false;
      int ebase = 0;
      if (lane && e < T::E) {
        const int ea = e % TX, eb = (e / TX) % TY, ec3 = DIM == 3 ? e / (TX * TY) : 0;
        act = ea < ex && eb < ey && (DIM == 2 || ec3 < ez);
        ebase = ea * N + T::LXP * (eb * N) + (DIM == 3 ? T::LXYP * (ec3 * N) : 0);
      }
      const int cb = ebase + ci + (DIM == 3 ? T::LXP * cj : 0);  // lattice slot of node 0
      float *myF = sF + ec * T::SFE;
      float Fz[C][n];
      if (act) {
        const float *ed = sE + e * T::NED;
        float Dx[n], Dy[n];  // rows ci and cj of D, from LDS
#pragma unroll
        for (int m = 0; m < n; ++m) {
          Dx[m] = sD[ci * n + m];
          Dy[m] = DIM == 3 ? sD[cj * n + m] : 0.f;
        }
        float uc[C][n];
#pragma unroll
        for (int c = 0; c < C; ++c)
#pragma unroll
          for (int k = 0; k < n; ++k) uc[c][k] = su[c * T::NTLP + cb + k * T::CS];
        // vertex material at t: mA + mB t, from its end-face values
        float mA[T::KP], mB[T::KP];
        {
          float wf[T::NV];
#pragma unroll
          for (int v = 0; v < T::NV; ++v) wf[v] = 0.5f * p1_face<DIM>(v, xa, xb);
#pragma unroll
          for (int q = 0; q < T::KP; ++q) {
            float lo = 0.f, hi = 0.f;
#pragma unroll
            for (int v = 0; v < T::NV; ++v) {
              const float P = ed[T::NG + v * T::KP + q];
              if (p1_tsign<DIM>(v) < 0) lo = fmaf(wf[v], P, lo);
              else hi = fmaf(wf[v], P, hi);
            }
            mA[q] = hi + lo;
            mB[q] = hi - lo;
          }
          if constexpr (PHYS != SEM_ACOUSTIC && DIM == 3) {
            // every Elastic3D coefficient is proportional to rho: scaling rho
            // by w_i w_j det J (and by w_k below) puts the quadrature weight
            // into the stress, so the flux needs no scaling of its own
            const float sw = wl * ed[DIM * DIM];
            mA[0] *= sw;
            mB[0] *= sw;
          }
        }
#pragma unroll
        for (int k = 0; k < n; ++k) {
          const float tk = gX<N>(k), wk = gW<N>(k);
          float g[C][DIM];
#pragma unroll
          for (int c = 0; c < C; ++c) {
            const float *rx = su + c * T::NTLP + (cb - ci) + k * T::CS;
            float s0 = 0.f;
#pragma unroll
            for (int m = 0; m < n; ++m) s0 = fmaf(Dx[m], rx[m], s0);
            g[c][0] = s0;
            if (DIM == 3) {
              const float *ry = su + c * T::NTLP + (cb - T::LXP * cj) + k * T::CS;
              float s1 = 0.f;
#pragma unroll
              for (int m = 0; m < n; ++m) s1 = fmaf(Dy[m], ry[m * T::LXP], s1);
              g[c][NL > 1 ? 1 : 0] = s1;
            }
            float sz = 0.f;
#pragma unroll
            for (int m = 0; m < n; ++m) sz = fmaf(gD<N>(k, m), uc[c][m], sz);
            g[c][DIM - 1] = sz;
          }
          float F[C][DIM];
          if constexpr (PHYS == SEM_ACOUSTIC) {
            const float vp = fmaf(mB[0], tk, mA[0]);
            const float sc = wl * wk * vp * vp;  // Scalar.cpp:45
            const float *Gs = ed;
            if constexpr (DG && DIM == 2) {
              F[0][0] = sc * (Gs[0] * g[0][0]);
              F[0][1] = sc * (Gs[2] * g[0][1]);
            } else if constexpr (DG) {
              F[0][0] = sc * (Gs[0] * g[0][0]);
              F[0][NL > 1 ? 1 : 0] = sc * (Gs[3] * g[0][1]);
              F[0][DIM - 1] = sc * (Gs[5] * g[0][DIM - 1]);
            } else if constexpr (DIM == 2) {
              F[0][0] = sc * (Gs[0] * g[0][0] + Gs[1] * g[0][1]);
              F[0][1] = sc * (Gs[1] * g[0][0] + Gs[2] * g[0][1]);
            } else {
              F[0][0] = sc * (Gs[0] * g[0][0] + Gs[1] * g[0][1] + Gs[2] * g[0][DIM - 1]);
              F[0][NL > 1 ? 1 : 0] = sc * (Gs[1] * g[0][0] + Gs[3] * g[0][1] + Gs[4] * g[0][DIM - 1]);
              F[0][DIM - 1] = sc * (Gs[2] * g[0][0] + Gs[4] * g[0][1] + Gs[5] * g[0][DIM - 1]);
            }
          } else {
            const float *Ji = ed;  // Jinv[a*DIM+b]
            const float wdet = wl * wk * ed[DIM * DIM];
            float cm[9];
            if constexpr (DIM == 2) {  // C11, C13, C33, C55
#pragma unroll
              for (int q = 0; q < 4; ++q) cm[q] = fmaf(mB[q], tk, mA[q]);
            } else {  // Elastic3D.cpp:42-52
              float q6[6];
#pragma unroll
              for (int q = 0; q < 6; ++q) q6[q] = fmaf(mB[q], tk, mA[q]);
              q6[0] *= wk;
              const float c11 = q6[0] * q6[2] * q6[2], c33 = q6[0] * q6[1] * q6[1];
              const float c44 = q6[0] * q6[3] * q6[3], c66 = q6[0] * q6[4] * q6[4];
              const float c13 = q6[5] * (c11 - 2.f * c44);
              cm[0] = c11; cm[1] = c11 - 2.f * c66; cm[2] = c13; cm[3] = c11; cm[4] = c13;
              cm[5] = c33; cm[6] = c44; cm[7] = c44; cm[8] = c66;
            }
            float gx[DIM][DIM];
#pragma unroll
            for (int c = 0; c < DIM; ++c)
#pragma unroll
              for (int a = 0; a < DIM; ++a) {
                float v = 0.f;
                if constexpr (DG) {
                  v = Ji[a * DIM + a] * g[c < C ? c : 0][a];
                } else {
#pragma unroll
                  for (int b = 0; b < DIM; ++b) v = fmaf(Ji[a * DIM + b], g[c < C ? c : 0][b], v);
                }
                gx[c][a] = v;
              }
            float sig[DIM][DIM];
            if constexpr (DIM == 2) {  // Elastic2D.cpp:53-82
              // shear sums unfused: with diagonal J^-1 the terms are plain
              // products the compiler could otherwise fuse into the sum, and
              // the variants would round differently
              const float exx = gx[0][0], eyy = gx[1][1], sh = add_unfused(gx[0][1], gx[1][0]);
              // explicit fmaf: the same fused products in every variant
              sig[0][0] = fmaf(cm[1], eyy, cm[0] * exx);
              sig[1][1] = fmaf(cm[2], eyy, cm[1] * exx);
              sig[0][1] = sig[1][0] = cm[3] * sh;
            } else {  // Elastic3D.cpp:76-83, :106-118
              constexpr int Y = DIM > 2 ? 2 : 1;
              const float e0 = gx[0][0], e1 = gx[1][1], e2 = gx[Y][Y];
              const float e3 = add_unfused(gx[1][Y], gx[Y][1]), e4 = add_unfused(gx[0][Y], gx[Y][0]);
              const float e5 = add_unfused(gx[0][1], gx[1][0]);  // unfused, as in 2-D
              sig[0][0] = fmaf(cm[2], e2, fmaf(cm[1], e1, cm[0] * e0));  // fixed fusion, as in 2-D
              sig[1][1] = fmaf(cm[4], e2, fmaf(cm[3], e1, cm[1] * e0));
              sig[Y][Y] = fmaf(cm[5], e2, fmaf(cm[4], e1, cm[2] * e0));
              sig[1][Y] = sig[Y][1] = cm[6] * e3;
              sig[0][Y] = sig[Y][0] = cm[7] * e4;
              sig[0][1] = sig[1][0] = cm[8] * e5;
            }
#pragma unroll
            for (int c = 0; c < DIM; ++c)
#pragma unroll
              for (int a = 0; a < DIM; ++a) {
                float v = 0.f;
                if constexpr (DG) {
                  v = Ji[a * DIM + a] * sig[c][a];
                } else {
#pragma unroll
                  for (int b = 0; b < DIM; ++b) v = fmaf(Ji[b * DIM + a], sig[c][b], v);
                }
                F[c < C ? c : 0][a] = DIM == 3 ? v : wdet * v;
              }
          }
          const int p = pl + T::ES * k;
#pragma unroll
          for (int c = 0; c < C; ++c) {
#pragma unroll
            for (int a = 0; a < NL; ++a) myF[(c * NL + a) * ND + p] = F[c][a];
            Fz[c][k] = F[c][DIM - 1];
          }
        }
      }
      __syncthreads();
      float f[C][n];
      if (act) {
        float Dcx[n], Dcy[n];  // columns ci and cj of D
#pragma unroll
        for (int m = 0; m < n; ++m) {
          Dcx[m] = sD[m * n + ci];
          Dcy[m] = DIM == 3 ? sD[m * n + cj] : 0.f;
        }
#pragma unroll
        for (int k = 0; k < n; ++k) {
          const int p = pl + T::ES * k;
          const bool dir = (sw[cb + k * T::CS] & kFlagDirichlet) != 0;
#pragma unroll
          for (int c = 0; c < C; ++c) {
            const float *Fx = myF + (c * NL) * ND + (p - ci);  // F_x along the x line
            float ku = 0.f;
#pragma unroll
            for (int m = 0; m < n; ++m) ku = fmaf(Dcx[m], Fx[m], ku);
            if (DIM == 3) {
              const float *Fy = myF + (c * NL + (NL > 1 ? 1 : 0)) * ND + (p - n * cj);
#pragma unroll
              for (int m = 0; m < n; ++m) ku = fmaf(Dcy[m], Fy[m * n], ku);
            }
#pragma unroll
            for (int m = 0; m < n; ++m) ku = fmaf(gD<N>(m, k), Fz[c][m], ku);
            f[c][k] = dir ? 0.f : -ku;
          }
        }
        for (int j = 0; j < W.nsrc; ++j) {
          if (sS[4 * j + 0] != e || sS[4 * j + 1] != (int)s) continue;
          const float R = glb(G.stf)[sS[4 * j + 2] + step];
          const gptr<const float> ld = glb(G.load) + sS[4 * j + 3];
#pragma unroll
          for (int c = 0; c < C; ++c)
#pragma unroll
            for (int k = 0; k < n; ++k) f[c][k] = fmaf(ld[c * ND + pl + T::ES * k], R, f[c][k]);
        }
      }
      if (T::ALIAS && ch == T::NCH - 1) __syncthreads();  // lateral fluxes read before sK overwrites them
      if (act) {
#pragma unroll
        for (int c = 0; c < C; ++c)
#pragma unroll
          for (int k = 0; k < n; ++k) sK[e * T::SKE + c * ND + pl + T::ES * k] = f[c][k];
      }
    }
    __syncthreads();

    // ---- the own nodes' finish inputs (w = v + dt/2 a_ and the
    // compensations) and the next shot's lattice are loaded here so that
    // their latency overlaps the face passes
    // (colours: a node's sum so far too, for the first KF slots)
    constexpr int KF = HO ? T::KF : T::NIT;
    float vw[KF][C], prev[COL ? KF : 1][C];
    uint32_t kc[KF][C], mia[HO ? KF : 1];
    const auto load_slot = [&](int l, float(&p)[C], float(&w)[C], uint32_t(&q)[C], uint32_t *mi) {
      const uint32_t word = l >= 0 ? sw[l] : kSlotEmpty;
      const bool valid = word != kSlotEmpty;
      const uint32_t g = valid ? word & kNodeMask : 0u;
      const bool fin = valid && (word & kFlagLast) && upd;
      if (mi) *mi = fin ? gmi[g] : 0u;
#pragma unroll
      for (int c = 0; c < C; ++c) {
        const uint32_t idx = (s * C + c) * GG + g;
        p[c] = !valid ? 0.f : !(word & kFlagFirst) ? gacc[idx] : has_ext ? gext[idx] : 0.f;
        w[c] = fin ? gw[idx] : 0.f;
        q[c] = fin ? gkc[idx] : 0u;
      }
    };
#pragma unroll
    for (int r = 0; r < KF; ++r) {
      if constexpr (COL) {
        load_slot(slot(r), prev[r], vw[r], kc[r], HO ? &mia[HO ? r : 0] : nullptr);
      } else {
        const int k = tid + r * T::BT;
        const bool fin = upd && k < nint;
#pragma unroll
        for (int c = 0; c < C; ++c) {
          const uint32_t idx = (s * C + c) * GG + own + k;
          vw[r][c] = fin ? gw[idx] : 0.f;
          kc[r][c] = fin ? gkc[idx] : 0u;
        }
      }
    }
    const bool more = s + 1 < s_end;
    float nu[T::NIT][C];
#pragma unroll
    for (int r = 0; r < T::NIT; ++r) {
      const int l = slot(r);
      const bool ok = more && (COL ? l >= 0 && sw[l] != kSlotEmpty : tid + r * T::BT < nval);
      const uint32_t g = ok ? (sw[l] & kNodeMask) : 0u;
#pragma unroll
      for (int c = 0; c < C; ++c) nu[r][c] = ok ? gu[((s + 1) * C + c) * GG + g] : 0.f;
    }

    // ---- shared faces: x, then y, then z (fixed order)
#pragma unroll
    for (int ax = 0; ax < DIM; ++ax) {
      constexpr int NF = ND / n;
      for (int i = tid; i < T::E * NF; i += T::BT) {
        const int e = i / NF, q = i - e * NF;
        const int ea = e % TX, eb = (e / TX) % TY, ec3 = DIM == 3 ? e / (TX * TY) : 0;
        const bool valid = ea < ex && eb < ey && (DIM == 2 || ec3 < ez);
        int lo, p, pn;
        if (ax == 0) {         // node (0, q) gains the x-neighbour's (N, q)
          lo = ea > 0 ? e - 1 : -1;
          p = q * n;
          pn = p + N;
        } else if (ax == 1) {  // (i, 0, k) gains (i, N, k)
          lo = eb > 0 ? e - TX : -1;
          p = DIM == 3 ? (q % n) + n * n * (q / n) : q;
          pn = p + n * N;
        } else {               // (i, j, 0) gains (i, j, N)
          lo = ec3 > 0 ? e - TX * TY : -1;
          p = q;
          pn = q + n * n * N;
        }
        if (valid && lo >= 0) {
#pragma unroll
          for (int c = 0; c < C; ++c) sK[e * T::SKE + c * ND + p] += sK[lo * T::SKE + c * ND + pn];
        }
      }
      __syncthreads();
    }

    // every finish input (and the next lattice) has arrived: one wait on all
    // paths here, so that no slot's finish below waits for the stores of the
    // slots before it (stores count on the same counter, and the loads were
    // issued under branches the compiler's counting cannot follow)
    // (not in the high-occupancy variant, whose later slots load in the finish
    // loop: 0.5 % slower with the wait)
    if (!HO) __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0) expcnt(7) lgkmcnt(15)
    if constexpr (COL) {
      // ---- finish every slot: its total joins the node's sum over the colours;
      // the Newmark update at the last colour
      const auto finish_slot = [&](int l, uint32_t o, const float(&p)[C], float(&w)[C], uint32_t(&q)[C], uint32_t mi) {
        const uint32_t word = l >= 0 ? sw[l] : kSlotEmpty;
        if (word == kSlotEmpty) return;
        const bool first = (word & kFlagFirst) != 0, fin = (word & kFlagLast) && upd;
#pragma unroll
        for (int c = 0; c < C; ++c) {
          const uint32_t idx = (s * C + c) * GG + (word & kNodeMask);
          const float tot = sK[o + c * ND];
          const float sum = first && !has_ext ? tot : p[c] + tot;
          if (!fin) {
            gacc[idx] = sum;
            continue;
          }
          if (q3 && c == 2) continue;
          const float a = __uint_as_float(mi) * sum;
          float u = su[c * T::NTLP + l];
          newmark(u, w[c], q[c], a, gdt, q3 && c == 0);
          gu[idx] = u; gw[idx] = w[c]; gkc[idx] = q[c];
          if (wap) gap[idx] = a;
        }
      };
      // place of a lattice slot's total: the owner element's result
      const auto place = [&](int l) -> uint32_t {
        const int z = DIM == 3 ? l / T::LXYP : 0, rl = l - z * T::LXYP, y = rl / T::LXP, x = rl - y * T::LXP;
        const int ea = min(x / N, ex - 1), eb = min(y / N, ey - 1), ec3 = DIM == 3 ? min(z / N, ez - 1) : 0;
        return (ea + TX * (eb + TY * ec3)) * T::SKE + (x - ea * N) + n * ((y - eb * N) + n * (z - ec3 * N));
      };
#pragma unroll
      for (int r = 0; r < KF; ++r) {
        const int l = slot(r);
        finish_slot(l, HO ? place(max(l, 0)) : slr[HO ? 0 : r] >> 16, prev[r], vw[r], kc[r], HO ? mia[HO ? r : 0] : mik[HO ? 0 : r]);
      }
      if constexpr (HO) {
        constexpr int KB = 4;
#pragma unroll 1
        for (int r0 = KF; r0 < T::NIT; r0 += KB) {
          float p[KB][C], w[KB][C];
          uint32_t q[KB][C], mi[KB];
          int ls[KB];
#pragma unroll
          for (int r = 0; r < KB; ++r) {
            ls[r] = r0 + r < T::NIT ? slot(r0 + r) : -1;
            load_slot(ls[r], p[r], w[r], q[r], &mi[r]);
          }
#pragma unroll
          for (int r = 0; r < KB; ++r) finish_slot(ls[r], place(max(ls[r], 0)), p[r], w[r], q[r], mi[r]);
        }
      }
    }
    // ---- (partial results) finish every slot: its total is the face-summed result of its owner
    // element; this tile's partial result for a node shared with other tiles,
    // the Newmark update for any other
#pragma unroll
    for (int r = 0; r < (COL ? 0 : T::NIT); ++r) {
      const int k = tid + r * T::BT;
      if (k >= nval) continue;
      const uint32_t sv = again(slr[r]);
      const int l = sv & kSlotMask, o = sv >> 16;
#pragma unroll
      for (int c = 0; c < C; ++c) {
        const float tot = sK[o + c * ND];
        if (k >= nint) {
          const gptr<float> at = gpart + (int64_t)(s * C + c) * PS + again(mik[r]);
          if constexpr (MODE == kTilePartsPast) __builtin_nontemporal_store(tot, at);
          else *at = tot;
          continue;
        }
        const uint32_t idx = (s * C + c) * GG + own + k;
        if (!upd) {
          gap[idx] = tot;  // accumulate-only pass: its result takes the place of a_
          continue;
        }
        if (q3 && c == 2) continue;
        const float a = __uint_as_float(mik[r]) * (has_ext ? glb(G.ext)[idx] + tot : tot);
        float u = su[c * T::NTLP + l], w = vw[r][c];
        uint32_t k2 = kc[r][c];
        newmark(u, w, k2, a, gdt, q3 && c == 0);
        gu[idx] = u; gw[idx] = w; gkc[idx] = k2;
        if (wap) gap[idx] = a;
      }
    }
    if (!more) break;
    // own slots only: u of this shot has been read above
#pragma unroll
    for (int r = 0; r < T::NIT; ++r) {
      const int l = slot(r);
      if (COL ? l < 0 : tid + r * T::BT >= nval) continue;
#pragma unroll
      for (int c = 0; c < C; ++c) su[c * T::NTLP + l] = nu[r][c];
    }
    __syncthreads();  // next lattice staged; sK and sF free again
  }
}

template <int N>
void fill_tables(TileTables &t) {
  constexpr GllC<N> g{};
  for (int i = 0; i < (N + 1) * (N + 1); ++i) t.D[i] = (float)g.D[i];
  for (int i = 0; i <= N; ++i) {
    t.w[i] = (float)g.w[i];
    t.xi[i] = (float)g.x[i];
  }
}

}  // namespace

int init_tile_tables(int device) {
  static bool done[64] = {false};
  if (device < 0 || device >= 64) { set_error("device index"); return -1; }
  if (done[device]) return 0;
  TileTables host[kTileMaxN + 1];
  memset(host, 0, sizeof host);
  // the same compile-time tables the kernels use as literals
  fill_tables<1>(host[1]);
  fill_tables<2>(host[2]);
  fill_tables<3>(host[3]);
  fill_tables<4>(host[4]);
  fill_tables<5>(host[5]);
  fill_tables<6>(host[6]);
  fill_tables<7>(host[7]);
  fill_tables<8>(host[8]);
  hipError_t e = hipMemcpyToSymbol(HIP_SYMBOL(t_tab), host, sizeof host, 0, hipMemcpyHostToDevice);
  if (e != hipSuccess) { set_error(std::string("tile tables: ") + hipGetErrorString(e)); return -2; }
  done[device] = true;
  return 0;
}

static bool same_shape(const int *T, int tx, int ty, int tz) {
  return T[0] == tx && T[1] == ty && T[2] == tz;
}

template <class S>
static TileKernelInfo tile_info() {
  static_assert(S::NTLP <= (int)kSlotMask && S::E * S::SKE < 65536, "LDS slots take 15 bits, result places 16");
  TileKernelInfo r{};
  r.lds_bytes = sizeof(float) * (size_t)S::LDS;
  r.threads = S::BT;
  r.lxp = S::LXP;
  r.lxyp = S::LXYP;
  r.elem_stride = S::SKE;
  return r;
}

TileKernelInfo tile_kernel_info(int dim, int order, int physics, const int *T) {
  TileKernelInfo r{};
#define TKI(D, N, X, Y, Z)                                                                  \
  if (dim == D && order == N && same_shape(T, X, Y, D == 3 ? Z : 1)) {                      \
    r = physics == SEM_ACOUSTIC ? tile_info<TS<D, N, 0, X, Y, Z>>()                         \
                                : tile_info<TS<D, N, 1, X, Y, Z>>();                        \
  }
  SEM_TILE_KERNELS(TKI)
#undef TKI
  return r;
}

int tile_kernel_shapes(int dim, int order, int physics, int *shapes, int max) {
  int k = 0;
#define TSH(D, N, X, Y, Z)                                                                  \
  if (dim == D && order == N && k < max) {                                                  \
    const int T[3] = {X, Y, D == 3 ? Z : 1};                                                \
    if (tile_kernel_info(dim, order, physics, T).lds_bytes <= 160 * 1024) {                 \
      shapes[3 * k] = T[0];                                                                 \
      shapes[3 * k + 1] = T[1];                                                             \
      shapes[3 * k + 2] = T[2];                                                             \
      ++k;                                                                                  \
    }                                                                                       \
  }
  SEM_TILE_KERNELS(TSH)
#undef TSH
  return k;
}

// Sets the dynamic-LDS limit of a kernel above 64 KiB and returns how many
// of its workgroups one CU holds; once per device (a batch's set-up asks several
// times, at some 50 us each).
template <int D, int N, int P, int X, int Y, int Z, int MODE>
static int prep_one(int *per_cu) {
  static std::atomic<int> known[64];
  int dev = -1;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) { set_error("device index"); return -1; }
  if ((*per_cu = known[dev].load(std::memory_order_acquire)) > 0) return 0;
  using S = TS<D, N, P, X, Y, Z, MODE == kTileColoursHigh>;
  const size_t shm = sizeof(float) * (size_t)S::LDS;
  if (shm > 160 * 1024) { set_error("tile does not fit in LDS"); return -1; }
  const void *fn = (const void *)k_tile<D, N, P, X, Y, Z, false, MODE>;
  if (shm > 64 * 1024) {
    const void *fns[2] = {fn, (const void *)k_tile<D, N, P, X, Y, Z, true, MODE>};
    for (const void *f : fns) {
      hipError_t e = hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, (int)shm);
      if (e != hipSuccess) { set_error(std::string("tile LDS attribute: ") + hipGetErrorString(e)); return -2; }
    }
  }
  int nb = 0;
  hipError_t e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, fn, S::BT, shm);
  if (e != hipSuccess) { set_error(std::string("tile occupancy: ") + hipGetErrorString(e)); return -2; }
  *per_cu = nb > 0 ? nb : 1;
  known[dev].store(*per_cu, std::memory_order_release);
  return 0;
}

template <int D, int N, int P, int X, int Y, int Z>
static int prep_tile(int mode, int *per_cu) {
  if constexpr (P == SEM_ACOUSTIC)
    if (mode == kTileColoursHigh) return prep_one<D, N, P, X, Y, Z, kTileColoursHigh>(per_cu);
  if constexpr (D == 3 && P == SEM_ELASTIC)
    if (mode == kTilePartsPast) return prep_one<D, N, P, X, Y, Z, kTilePartsPast>(per_cu);
  return mode == kTileParts ? prep_one<D, N, P, X, Y, Z, kTileParts>(per_cu)
                            : prep_one<D, N, P, X, Y, Z, kTileColours>(per_cu);
}

int tile_kernel_prepare(int dim, int order, int physics, const int *T, int mode, int *per_cu) {
  int rc = 1;
#define TPR(D, N, X, Y, Z)                                                                  \
  if (rc == 1 && dim == D && order == N && same_shape(T, X, Y, D == 3 ? Z : 1))             \
    rc = physics == SEM_ACOUSTIC ? prep_tile<D, N, 0, X, Y, Z>(mode, per_cu)                \
                                 : prep_tile<D, N, 1, X, Y, Z>(mode, per_cu);
  SEM_TILE_KERNELS(TPR)
#undef TPR
  if (rc == 1) { set_error("tile kernel not compiled for this order/shape"); return -1; }
  return rc;
}

template <int D, int N, int P, int X, int Y, int Z, bool DG, int MODE>
static int go_mode(const FusedArgs &a, hipStream_t st) {
  using S = TS<D, N, P, X, Y, Z, MODE == kTileColoursHigh>;
  hipLaunchKernelGGL((k_tile<D, N, P, X, Y, Z, DG, MODE>), dim3(a.nitems), dim3(S::BT),
                     sizeof(float) * (size_t)S::LDS, st, a);
  return 0;
}

template <int D, int N, int P, int X, int Y, int Z, bool DG>
static int go_tile(int mode, const FusedArgs &a, hipStream_t st) {
  if constexpr (P == SEM_ACOUSTIC)
    if (mode == kTileColoursHigh) return go_mode<D, N, P, X, Y, Z, DG, kTileColoursHigh>(a, st);
  if constexpr (D == 3 && P == SEM_ELASTIC)
    if (mode == kTilePartsPast) return go_mode<D, N, P, X, Y, Z, DG, kTilePartsPast>(a, st);
  return mode == kTileParts ? go_mode<D, N, P, X, Y, Z, DG, kTileParts>(a, st)
                            : go_mode<D, N, P, X, Y, Z, DG, kTileColours>(a, st);
}

int launch_tile(int dim, int order, int physics, const int *T, bool diag, int mode, const FusedArgs &a,
                hipStream_t st) {
  if (a.nitems <= 0) return 0;
  int rc = 1;
#define TLN(D, N, X, Y, Z)                                                                  \
  if (rc == 1 && dim == D && order == N && same_shape(T, X, Y, D == 3 ? Z : 1))             \
    rc = physics == SEM_ACOUSTIC                                                            \
             ? (diag ? go_tile<D, N, 0, X, Y, Z, true>(mode, a, st)                         \
                     : go_tile<D, N, 0, X, Y, Z, false>(mode, a, st))                       \
             : (diag ? go_tile<D, N, 1, X, Y, Z, true>(mode, a, st)                         \
                     : go_tile<D, N, 1, X, Y, Z, false>(mode, a, st));
  SEM_TILE_KERNELS(TLN)
#undef TLN
  if (rc == 1) { set_error("tile kernel not compiled for this order/shape"); return -1; }
  if (rc) return rc;
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) { set_error(std::string("tile step: ") + hipGetErrorString(e)); return -2; }
  return 0;
}

}  // namespace sem
