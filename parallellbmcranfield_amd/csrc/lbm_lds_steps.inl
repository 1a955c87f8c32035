// lbm_lds_steps.inl — several plain steps per launch with the block of nodes
// held in LDS between them; included after lbm_kernels.inl.
#pragma once

namespace lbmdev {

struct LdsRules {
  const LdsList& l;
  const BNode* bn;
  __device__ double uo() const { return l.uo; }
  __device__ bool inlet() const { return true; }
  __device__ bool lid() const { return l.bits & LL_LID; }
  __device__ bool west() const { return l.bits & LL_WEST; }
  __device__ bool wall(int k) const { return (l.bits >> k) & 1u; }
  __device__ double q(int k) const { return bn[l.node].q[k]; }
  __device__ bool east() const { return l.bits & LL_EAST; }
};

// One step of one node from its streamed populations F, as pull_cell / the
// boundary list and finish_node<MODE 0> form it: r is the node's rule word
// (LdsRule), l its list rules where it is a list node, own(k) and up(k) its
// METAF[k] and its upstream neighbour's.  In the storage's raw units.
template <class S, int COLL, bool GEN, class Own, class Up>
__device__ inline void lds_node(typename S::R (&F)[9], uint32_t r, const LdsList& l,
                                const BNode* __restrict__ bn, const KParams& p, const CollPar& cp,
                                Own own, Up up, typename S::R (&out)[9]) {
  using R = typename S::R;
  bool still = false, list = false;  // still: V = 0 (east outlets)
  if constexpr (GEN) {
    if ((r & LR_CLASS) == LR_LIST) {
      list = true;
      still = l.bits & LL_EAST;
      const LdsRules rules{l, bn};
      if constexpr (S::SCALED) {
        const R sc = (R)p.scale_f, isc = (R)p.inv_scale_f;
#pragma unroll
        for (int k = 0; k < 9; k++) F[k] *= isc;
        apply_bc<S>(
            F, rules, p, [&](int k) { return own(k) * isc; }, [&](int k) { return up(k) * isc; });
#pragma unroll
        for (int k = 0; k < 9; k++) F[k] *= sc;
      } else {
        apply_bc<S>(F, rules, p, own, up);
      }
    } else if ((r & LR_CLASS) == LR_WALL) {
      wall_bounce(F, r);
    }
  }
  if constexpr (!S::DEV)
    node_f64<COLL>(F, still, p, out);
  else if constexpr (S::SCALED)
    node_dev<COLL>(F, p.rho0_f, p.scale_f, p.inv_scale_f, still, list, cp, out);
  else
    node_dev<COLL>(F, p.rho0_f, 1.f, 1.f, still, list, cp, out);
}

// The value of the lane DX to the left (DX = 1) or right (-1) in the wave; the
// wave's outermost lanes keep their own.
template <int DX, class R>
__device__ inline R lane_pull(R x) {
  if constexpr (DX == 0) return x;
  constexpr int CTRL = DX > 0 ? 0x138 : 0x130;  // wave_shr:1, wave_shl:1
  constexpr int WORDS = sizeof(R) / 4;
  struct Words {
    int w[WORDS];
  };
  Words a = __builtin_bit_cast(Words, x);
#pragma unroll
  for (int i = 0; i < WORDS; i++)
    a.w[i] = __builtin_amdgcn_update_dpp(a.w[i], a.w[i], CTRL, 0xf, 0xf, false);
  return __builtin_bit_cast(R, a);
}

// steps (1 .. halo + 1) plain steps of one block.  The workgroup works on a
// region of RX x RY nodes: the block's output nodes and `halo` nodes around
// them.  Step 1 pulls from METAF_t in memory and leaves its results in LDS;
// each later step pulls from LDS, holds its results in registers until every
// pull of the workgroup is done, and writes them back; the last step's
// results go to METAF_{t+steps}.  The margin that a step forms shrinks by one
// node per step, so every value it pulls was formed here.  A thread takes NPT
// nodes one above the other.  GEN: the region holds nodes that are not plain
// interior ones.
//
// What bounds it.  Small lattices: the latency of a launch (the block's table
// entry, rule words and pulls, one after the other) and of each step (LDS
// reads, the collision's dependent chain, two barriers); 129^2 FP64 BGK 4.12
// us per single-step launch, 1.50 us per step at seven a launch.  Large
// lattices: VALU issue and memory together.  A block of 64 x 32 nodes makes
// five steps of 56 x 24, forming 1.37 nodes per node kept and loading 1.52
// times what it keeps (1.36 from memory, by the counters), where k_three_steps
// reads 1.72 times the state per three steps and two-step launches 1.30 times
// per two: 4097^2 FP32 MRT 115.2 -> 63.2 us per step (145 -> 265 GLUPS), 2049^2
// 39.7 -> 19.2, 1025^2 15.2 -> 7.0 (6.5 with LANES); FP64 BGK 4097^2 274 -> 145
// (130 with LANES), 2049^2 72 -> 39 (37); FP16 BGK 4097^2 111.8 -> 56.4.  Those
// are runs from rest; on a developed field 4097^2 takes 69.5 (FP32), 139 (FP64
// BGK) and 59.3 (FP16), 2049^2 FP64 38.5: as many cycles and instructions at a
// lower clock (FP64 2.39 -> 2.21 GHz between iterations 500 and 5500).
// Counters: 4097^2 FP32 0.77 M cycles per launch, whose VALU instructions fill
// every issue slot of the SIMDs (104 % at four cycles each) beside 4.6 TB/s;
// 1025^2 60 %, 2.9 TB/s.
// LANES: 72 bytes of LDS per node and step's 18 accesses limited FP64
// to regions of 32 x 32, which form 1.69 nodes per node kept and read 1.78.
// Blocks of interior nodes now hold their state in registers, a wave 64 x 4
// nodes, and a third of the LDS accesses is left for two nodes per thread, a
// sixth for four: FP64 BGK 4097^2 146.5 -> 130.6 us per step, 2049^2 40.2 ->
// 37.0, 1025^2 11.2 -> 9.9; there memory and VALU issue bound it together
// (2049^2, counters: 34 bytes per node and step, 3.9 TB/s; issue slots 61 %
// full).  For FP32 and FP16 the same form at
// 32 x 32 with three workgroups per CU is the faster one up to 1.7 M and 3 M
// cells (FP32 MRT 970^2 6.4 -> 5.7 us); above, the DPP moves, which are VALU
// instructions, cost more than they save (FP32 MRT 4097^2 63.2 us against
// 68.8).  Eight and six nodes per thread were 20-40 % slower there.
// Ordinary stores: two blocks store parts of a cache line where they meet,
// and non-temporal stores gave those to memory one by one (4097^2 FP32 82.7
// against 63.2 us per step, FP64 165.6 against 144.8).
// Two workgroups of 1024 threads per CU need 64 VGPRs (waves_per_eu 8): at 128,
// with one, 1025^2 FP32 took 8.3 us per step against 6.7.  One LDS copy and two
// barriers per step; two copies and one barrier measured 0-25 % slower (half
// the workgroups per CU).
template <class S, int COLL, int NT, int RX, int NPT, bool GEN, bool LANES>
__device__ inline void lds_block(const typename S::T* __restrict__ src,
                                 typename S::T* __restrict__ dst,
                                 const uint32_t* __restrict__ rule, const LdsTile& tl,
                                 const LdsList* __restrict__ list, const BNode* __restrict__ bn,
                                 int halo, int steps, const KParams& p, uint32_t step0,
                                 typename S::R* lds) {
  using R = typename S::R;
  constexpr int RY = NT / RX * NPT, PL = RX * RY;
  const int lx = (int)threadIdx.x % RX, ly = (int)threadIdx.x / RX * NPT;
  const int gx = tl.x0 - halo + lx;
  const int cx = min(max(gx, tl.rx0), tl.rx1 - 1);
  const CollPar cp = coll_par(p, tl.inst);
  uint32_t rl[NPT];
  int idx[NPT], far[NPT];  // far: rows / columns outside the output nodes
  R v[NPT][9];
  LdsList ll{};
#pragma unroll
  for (int i = 0; i < NPT; i++) {
    const int gy = tl.y0 - halo + ly + i;
    const int cy = min(max(gy, tl.ry0), tl.ry1 - 1);
    idx[i] = cy * p.pitch + cx;
    far[i] = max(max(tl.x0 - gx, gx - (tl.x1 - 1)), max(tl.y0 - gy, gy - (tl.y1 - 1)));
    if constexpr (GEN)
      rl[i] = (gx == cx && gy == cy) ? rule[idx[i]] : 0u;
    else
      rl[i] = LR_INTERIOR | 0x1ffu;
  }
  // rows between the wave's rows and the output rows: the same in every lane
  constexpr int WR = (RX >= 64 ? 1 : 64 / RX) * NPT;
  const int w0 = __builtin_amdgcn_readfirstlane(tl.y0 - halo + ly);
  const int wfar = max(tl.y0 - (w0 + WR - 1), w0 - (tl.y1 - 1));
  // does the step that leaves `margin` nodes around the output form node i?
  // Blocks of interior nodes form every node of a wave that forms any (the
  // others come to nothing, and the wave's nodes share one instruction
  // stream).
  auto forms = [&](int i, int margin) {
    return GEN ? far[i] <= margin && (rl[i] & LR_CLASS) != 0u : true;
  };
  // the pulls of every node of the thread first, so that they are in flight
  // together
  if (wfar < steps) {
    if constexpr (GEN && NPT == 1) {
      // small lattices, where the latency of a launch counts: every load
      // before the rule word is known (a cell outside the lattice pulls as
      // the nearest one inside its ring)
      const int px = min(max(gx, tl.rx0 + 1), tl.rx1 - 2);
      const int py = min(max(tl.y0 - halo + ly, tl.ry0 + 1), tl.ry1 - 2);
      const int pidx = py * p.pitch + px;
      R own[9];
#pragma unroll
      for (int k = 0; k < 9; k++) {
        v[0][k] = S::load_raw(plane_word(src, p.plane, k, pidx - CX[k] - CY[k] * p.pitch));
        own[k] = S::load_raw(plane_word(src, p.plane, k, idx[0]));
      }
#pragma unroll
      for (int k = 0; k < 9; k++)
        if (!((rl[0] >> k) & 1)) v[0][k] = own[k];
      if ((rl[0] & LR_CLASS) == LR_LIST) ll = list[rl[0] >> LR_SHIFT];
    } else {
#pragma unroll
      for (int i = 0; i < NPT; i++) {
        if (GEN && far[i] >= steps) continue;
#pragma unroll
        for (int k = 0; k < 9; k++) {
          int off = -CX[k] - CY[k] * p.pitch;
          if (GEN && !((rl[i] >> k) & 1)) off = 0;
          v[i][k] = S::load_raw(plane_word(src, p.plane, k, idx[i] + off));
        }
      }
    }
#pragma unroll
    for (int i = 0; i < NPT; i++) {
      if (!forms(i, steps - 1)) continue;
      if constexpr (GEN && NPT > 1)
        if ((rl[i] & LR_CLASS) == LR_LIST) ll = list[rl[i] >> LR_SHIFT];
      R out[9];
      const int id = idx[i];
      lds_node<S, COLL, GEN>(
          v[i], rl[i], ll, bn, p, cp, [&](int k) { return S::load_raw(src + k * p.plane + id); },
          [&](int k) { return S::load_raw(src + k * p.plane + id - CX[k] - CY[k] * p.pitch); },
          out);
#pragma unroll
      for (int k = 0; k < 9; k++) v[i][k] = out[k];
    }
  }
  if constexpr (LANES) {
    // What a node pulls from its own thread's or its wave's nodes stays in
    // registers, across lanes by DPP moves: the lanes that get a wrong
    // neighbour are the region's outermost columns, which no step from the
    // second on has to form.  LDS carries what crosses the threads' upper and
    // lower edges, in two copies in turn, so that one barrier per step is
    // enough.
    static_assert(!GEN && RX <= 64);
    constexpr int NG = NT / RX, QL = (NG + 2) * RX;
    constexpr int SLOT[9] = {0, 0, 0, 0, 3, 1, 2, 4, 5};
    for (int t = 1; t < steps; t++) {
      R* const w = lds + 1 + (t & 1) * 6 * QL + ((int)threadIdx.x / RX + 1) * RX + lx;
      if (wfar <= steps - t) {
#pragma unroll
        for (int i = 0; i < NPT; i++) S::round_raw(v[i], idx[i], step0 + (uint32_t)(t - 1));
#pragma unroll
        for (int k = 0; k < 9; k++)
          if (CY[k] != 0) w[SLOT[k] * QL] = v[CY[k] > 0 ? NPT - 1 : 0][k];
      }
      __syncthreads();
      if (wfar < steps - t) {
        R below[9];  // the values before this step of the node below
#pragma unroll
        for (int i = 0; i < NPT; i++) {
          R F[9];
#pragma unroll
          for (int k = 0; k < 9; k++) {
            if (CY[k] > 0 && i == 0)
              F[k] = w[SLOT[k] * QL - CX[k] - RX];
            else if (CY[k] < 0 && i == NPT - 1)
              F[k] = w[SLOT[k] * QL - CX[k] + RX];
            else {
              const R x = CY[k] > 0 ? below[k] : (CY[k] < 0 ? v[i + 1 < NPT ? i + 1 : i][k] : v[i][k]);
              F[k] = CX[k] == 0 ? x : (CX[k] > 0 ? lane_pull<1>(x) : lane_pull<-1>(x));
            }
            below[k] = v[i][k];
          }
          lds_node<S, COLL, false>(
              F, rl[i], ll, bn, p, cp, [&](int) { return R(0); }, [&](int) { return R(0); }, v[i]);
        }
      }
    }
  } else {
    R* const w = lds + RX + 1 + ly * RX + lx;
    for (int t = 1; t < steps; t++) {
      // step t's results to LDS (a cell without a node keeps the solid value
      // it was loaded with)
      if (wfar <= steps - t) {
#pragma unroll
        for (int i = 0; i < NPT; i++) {
          const bool node = !GEN || (rl[i] & LR_CLASS) != 0u;
          if (GEN && (far[i] > steps - t || (t > 1 && !node))) continue;
          if (node) S::round_raw(v[i], idx[i], step0 + (uint32_t)(t - 1));
#pragma unroll
          for (int k = 0; k < 9; k++) w[k * PL + i * RX] = v[i][k];
        }
      }
      __syncthreads();
      if (wfar < steps - t) {
#pragma unroll
        for (int i = 0; i < NPT; i++) {
          if (!forms(i, steps - t - 1)) continue;
          const R* wi = w + i * RX;
          R F[9];
#pragma unroll
          for (int k = 0; k < 9; k++) F[k] = wi[k * PL - CX[k] - CY[k] * RX];
          if (GEN && (rl[i] & LR_CLASS) != LR_INTERIOR) {
#pragma unroll
            for (int k = 0; k < 9; k++)
              if (!((rl[i] >> k) & 1)) F[k] = wi[k * PL];
          }
          if constexpr (GEN && NPT > 1)
            if ((rl[i] & LR_CLASS) == LR_LIST) ll = list[rl[i] >> LR_SHIFT];
          lds_node<S, COLL, GEN>(
              F, rl[i], ll, bn, p, cp, [&](int k) { return wi[k * PL]; },
              [&](int k) { return wi[k * PL - CX[k] - CY[k] * RX]; }, v[i]);
        }
      }
      __syncthreads();
    }
  }
#pragma unroll
  for (int i = 0; i < NPT; i++) {
    if (far[i] > 0 || (GEN && (rl[i] & LR_CLASS) == 0u)) continue;
    S::store_raw(dst, idx[i], v[i], p, step0 + (uint32_t)(steps - 1));
  }
}

// PRX, PNPT: the regions of blocks of interior nodes, LANES: held in registers
template <class S, int COLL, int NT, int RX, int NPT, int WPE, int PRX = RX, int PNPT = NPT,
          bool LANES = false>
__global__ __launch_bounds__(NT, WPE) void k_lds_steps(
    const typename S::T* __restrict__ src, typename S::T* __restrict__ dst,
    const uint32_t* __restrict__ rule, const LdsTile* __restrict__ tiles,
    const LdsList* __restrict__ list, const BNode* __restrict__ bn, int halo, int steps,
    KParams p) {
  using R = typename S::R;
  // a row and a cell before and after (LANES: one row and one cell): pulls of
  // nodes that come to nothing
  constexpr int ALL = 9 * NT * NPT + 2 * (RX + 1), EDGES = 12 * (NT + 2 * PRX) + 2;
  __shared__ R lds[LANES && EDGES > ALL ? EDGES : ALL];
  const uint32_t step0 = step_number<S>(p);
  if constexpr (S::SR) {
    if (blockIdx.x == 0 && threadIdx.x == 0) p.seed[p.seed_slot ^ 1] = step0 + (uint32_t)steps;
  }
  const LdsTile tl = tiles[blockIdx.x];
  if (tl.x1 <= tl.x0) return;
  if (tl.plain)
    lds_block<S, COLL, NT, PRX, PNPT, false, LANES>(src, dst, rule, tl, list, bn, halo, steps, p, step0,
                                           lds);
  else
    lds_block<S, COLL, NT, RX, NPT, true, false>(src, dst, rule, tl, list, bn, halo, steps, p, step0,
                                          lds);
}

}  // namespace lbmdev
