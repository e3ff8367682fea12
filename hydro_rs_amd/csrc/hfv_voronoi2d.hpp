// 2D moving meshes rebuilt on the device: Space::volume_calculation (src/space.rs:236-263) for 2D, the
// reference's call of meshless_voronoi's Voronoi::build_partial with the step's active mask: only the
// active cells are built (their faces, including those with inactive neighbours), and every cell gets
// its CSR range over the faces that exist.  Included by hfv_api.hip.
//
// The tessellation is the host tessellator's (hydro_rs_amd/csrc/host/voronoi.cpp, which stands in for
// the crate) evaluated with the same operations in the same order, so the device mesh equals the host's
// bit for bit: every generator's cell is the initial region (the box, or a square of K bin widths around
// the generator on a periodic box) clipped by the bisectors of the generators of the (2K+1)^2 bins around
// its own, visited in increasing (squared distance, index, image code) order until no unvisited one can
// cut the cell (a quarter of its squared distance beyond every vertex), with K = 2, 3, .. (up to the whole
// grid) until the cell lies within K bin widths (and, periodic, has no wall edge).  Faces are emitted in
// the order of the emitting cell's polygon edges (v2_emits); face indices follow the cells; each cell's
// CSR lists its faces in ascending face index.
//
// Per step (simulations with vmesh = 2, while stepping; 3D: hfv_voronoi3d.hpp), after the drift and the predict:
//   k_mask (v_count_bin)        bin counts of the generators
//   k_v2_sum<0>, k_v2_bins,
//   k_v2_place                  bin starts; the generators grouped by bin (a counting sort)
//   k_v2_cells (3D: k_v3_cells) the active cells' polygons, volume, centroid and search radius
//                               (Particle::update_geometry, part.rs:151-158); the cell's emitted faces in a
//                               provisional order, and the chunk sums of their counts
//   k_v2_faces                  face indices in cell order, the face arrays, each cell's CSR entries in its
//                               bucket
//   k_v2_sum<1>, k_v2_conn      CSR offsets; the entries in ascending face order
// Each prefix sum over cells (or bins) is two levels: a kernel before leaves the sums of the chunks of
// HFV_BLOCK elements, and every block of the kernel that needs the sum adds up the chunks before its own
// (chunks_before; on large meshes k_v2_prefix has scanned them) and scans its chunk.  The rebuild was 18
// launches of 4-5 us each (counts, sums, scans, fill and sort apart) and is 7 in 2D: a 125^2 vortex with
// steered generators 218 -> 202 us a step, a Sedov 256^2 run to t = 0.004 121 -> 111.5 ms.
// Inactive cells keep their geometry and get new CSR ranges (the reference's note at space.rs:233-235).
#pragma once

namespace hfv {

#define HFV_PREFIX_BLOCK 1024
// A clip removes the vertices beyond a plane by more than this fraction of its offset (the host
// tessellator's threshold): vertices on it test as beyond by a rounding error on exact lattices.
#define HFV_CLIP_TOL 1e-12

// (squared distance, index, image code) order; the code compares as the host's memcmp of int8 codes
__device__ __forceinline__ bool v2_less(double ad2, int32_t aj, int32_t ak, double bd2, int32_t bj, int32_t bk) {
  if (ad2 != bd2) return ad2 < bd2;
  if (aj != bj) return aj < bj;
  return ak < bk;
}

__device__ __forceinline__ int32_t v2_shift_code(int s0, int s1) {
  return (s0 == 1 ? 1 : s0 == -1 ? 2 : 0) | ((s1 == 1 ? 1 : s1 == -1 ? 2 : 0) << 2);
}

// ---------------------------------------------------------------- prefix sums
// exclusive scan of one value per thread over a block of HFV_BLOCK threads; *total receives the sum
__device__ __forceinline__ int32_t block_excl_scan(int32_t v, int32_t* total) {
  __shared__ int32_t ws[HFV_BLOCK / 64];
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  int32_t x = v;
  for (int o = 1; o < 64; o <<= 1) {
    const int32_t y = __shfl_up(x, o, 64);
    if (lane >= o) x += y;
  }
  if (lane == 63) ws[wid] = x;
  __syncthreads();
  int32_t before = 0, tot = 0;
  for (int w = 0; w < HFV_BLOCK / 64; ++w) {
    if (w < wid) before += ws[w];
    tot += ws[w];
  }
  __syncthreads();
  *total = tot;
  return before + x - v;
}

// The sum of the simulation's chunk sums (array k of V.part) before chunk `chunk`, and of all of them (every thread
// gets both).  Each block reads every chunk sum: at most a few thousand words that the L2 holds, where a launch of
// its own to scan them costs 4-5 us.  Meshes of more chunks have them scanned (k_v2_prefix).
template <bool SCANNED>
__device__ __forceinline__ int32_t chunks_before(const V2Bufs& V, int k, const SimDesc& D, int s, int32_t chunk,
                                                 int32_t* total) {
  const int32_t* part = V.part[k];
  if (SCANNED) {
    *total = V.ptot[3 * s + k];
    return part[chunk];
  }
  __shared__ int32_t wb[HFV_BLOCK / 64], wt[HFV_BLOCK / 64];
  int32_t b = 0, t = 0;
  for (int32_t c = D.cchunk0 + (int32_t)threadIdx.x; c < D.cchunk1; c += HFV_BLOCK) {
    const int32_t v = part[c];
    t += v;
    if (c < chunk) b += v;
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    b += __shfl_xor(b, o);
    t += __shfl_xor(t, o);
  }
  if (__lane_id() == 0) {
    wb[threadIdx.x >> 6] = b;
    wt[threadIdx.x >> 6] = t;
  }
  __syncthreads();
  b = 0;
  t = 0;
#pragma unroll
  for (int w = 0; w < HFV_BLOCK / 64; ++w) {
    b += wb[w];
    t += wt[w];
  }
  __syncthreads();
  *total = t;
  return b;
}

// A simulation's entries beyond their cells' buckets.
__device__ __forceinline__ V2Over* v_over(const Batch& B, const SimDesc& D) { return (V2Over*)(B.F.fs + 4 * D.face_base); }

// Chunk sums of the bin counts (CSR 0) or of the cells' CSR entries (CSR 1).  (Added up by the counting
// atomics instead, they put hundreds of atomics on one address: 10-100 us.)  CSR 1 also chains the entries beyond
// the buckets to their cells.
template <int CSR>
__global__ void __launch_bounds__(HFV_BLOCK) k_v2_sum(Batch B, V2Bufs V) {
  const BlockJob J = B.cjobs[blockIdx.x];
  if (J.sim < 0) return;
  const int s = J.sim;
  const SimDesc& D = B.sims[s];
  if (!D.vmesh || !B.st[s].stepping) return;
  const int64_t k = (int64_t)J.lo - D.cell_base + threadIdx.x;
  const int64_t len = CSR ? D.n : (int64_t)D.vnb[0] * D.vnb[1] * D.vnb[2];
  const int32_t* a = CSR ? V.ccnt + D.cell_base : V.gcnt + D.cell_base + s;
  const uint32_t t = block_sum_u32(k < len ? (uint32_t)a[k] : 0u);
  if (threadIdx.x == 0) V.part[CSR ? 2 : 0][J.chunk] = (int32_t)t;
  if (CSR && k < len) {
    const int64_t no = min((int64_t)B.st[s].n_over, 2 * D.face_cap);
    V2Over* over = v_over(B, D);
    for (int64_t o = k; o < no; o += len) over[o].next = atomicExch(&V.gkey[over[o].cell], (int32_t)o);
  }
}

// The chunk sums (array k) of a simulation, scanned in place: one block per simulation.
__global__ void __launch_bounds__(HFV_PREFIX_BLOCK) k_v2_prefix(Batch B, V2Bufs V, int k) {
  const int s = blockIdx.x;
  const SimDesc& D = B.sims[s];
  if (!D.vmesh || !B.st[s].stepping) return;
  __shared__ int32_t ws[HFV_PREFIX_BLOCK / 64];
  int32_t* part = V.part[k];
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  int32_t carry = 0;
  for (int32_t c0 = D.cchunk0; c0 < D.cchunk1; c0 += HFV_PREFIX_BLOCK) {
    const int32_t c = c0 + (int32_t)threadIdx.x;
    const int32_t v = c < D.cchunk1 ? part[c] : 0;
    int32_t x = v;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const int32_t y = __shfl_up(x, o, 64);
      if (lane >= o) x += y;
    }
    if (lane == 63) ws[wid] = x;
    __syncthreads();
    int32_t before = 0, tot = 0;
    for (int w = 0; w < HFV_PREFIX_BLOCK / 64; ++w) {
      if (w < wid) before += ws[w];
      tot += ws[w];
    }
    if (c < D.cchunk1) part[c] = carry + before + x - v;
    carry += tot;
    __syncthreads();
  }
  if (threadIdx.x == 0) V.ptot[3 * s + k] = carry;
}

// Bin starts and placement cursors; the chunk sums of the emitted faces restart at zero.
template <bool SCANNED>
__global__ void __launch_bounds__(HFV_BLOCK) k_v2_bins(Batch B, V2Bufs V) {
  const BlockJob J = B.cjobs[blockIdx.x];
  if (J.sim < 0) return;
  const int s = J.sim;
  const SimDesc& D = B.sims[s];
  if (!D.vmesh || !B.st[s].stepping) return;
  if (threadIdx.x == 0) V.part[1][J.chunk] = 0;
  const int64_t nbins = (int64_t)D.vnb[0] * D.vnb[1] * D.vnb[2];  // <= n
  const int64_t k = (int64_t)J.lo - D.cell_base + threadIdx.x;
  int32_t* a = V.gcnt + D.cell_base + s;
  const int32_t v = k < nbins ? a[k] : 0;
  int32_t all, tot;
  const int32_t base = chunks_before<SCANNED>(V, 0, D, s, J.chunk, &all);
  const int32_t x = base + block_excl_scan(v, &tot);
  if (k < nbins) {
    a[k] = x;
    V.gfill[D.cell_base + s + k] = x;
  }
  if (J.chunk == D.cchunk1 - 1 && threadIdx.x == 0) a[nbins] = all;
}

__global__ void __launch_bounds__(HFV_BLOCK) k_v2_place(Batch B, V2Bufs V) {
  const BlockJob J = B.cjobs[blockIdx.x];
  if (J.sim < 0) return;
  const int s = J.sim;
  const SimDesc& D = B.sims[s];
  if (!D.vmesh || !B.st[s].stepping) return;
  const int64_t gi = (int64_t)J.lo + threadIdx.x;
  if (gi >= J.hi) return;
  const int32_t p = atomicAdd(&V.gfill[D.cell_base + s + V.gkey[gi]], 1);
  V.gord[D.cell_base + p] = (int32_t)(gi - D.cell_base);
}

// ---------------------------------------------------------------- cells, a team of lanes per cell
// 16 lanes, a DPP row, build one cell together.  The candidates of the (2K+1)^2 block are gathered into LDS
// once, ranked by (squared distance, index, image code) (each lane ranks every 16th against all), and clip
// the polygon in rank order.  The polygon lies in registers, lane k holding edge k and the vertex after it: a
// clip is one ballot, and where it cuts, one permute that closes the edges up, one for the next edge's plane,
// the lanes' vertices and a row maximum.  The finish takes each edge's terms on its own lane and adds them in
// order.  (A team's chain of candidates is what bounds the rebuild, most of all where few cells are
// active: with the next candidate a 4-stage team minimum over whole candidates and the polygon in LDS the
// kernel took 65 us on Sedov 256^2 with steered generators and 98 us on a 125^2 vortex, now 35 and 71.)
// Cells of more than HFV_V2_CAP candidates or 16 edges are built by v2_team_build, which rescans the bins for
// every candidate and keeps polygons of up to HFV_V2_TLW edges in LDS.  Both make the host tessellator's
// operations in its order, so the same bits.
#define HFV_V2_TEAM 16
#define HFV_V2_TLW 48
#define HFV_V2_CAP 96           // 3 blocks a CU; a 9 x 9-bin block (K = 4) at one generator per bin mostly fits
#define HFV_V2_SUB HFV_V2_TEAM  // blocks per cell chunk

template <int TL>
struct V2TeamPoly {
  double nx[TL], ny[TL], d[TL], vx[TL], vy[TL];
  int32_t nb[TL], code[TL];
};

// Voronoi::build_partial builds the active cells only: a face is emitted by the lower-index cell of a pair
// of active cells, by the active cell of a pair with an inactive one, and a wall by its cell.
__device__ __forceinline__ bool v2_emits(const Batch& B, int64_t cb, int32_t nb, int32_t i) {
  return nb < 0 || nb > i || !B.C.act[cb + nb];
}

// Place of a cell's cnt emitted faces in the provisional order: after those that its chunk has placed, in the
// chunk's share of the simulation's face capacity, or where the share is full in the common overflow (from F.nf on:
// v_faces_at).  -1 beyond the capacity.  (One cursor for the whole simulation instead is an atomic on one address
// per cell, about 20 ns each: it alone bounded the 3D cell kernel.)
__device__ __forceinline__ int32_t v_place_faces(const Batch& B, const V2Bufs& V, const SimDesc& D, SimStep& S, int chunk,
                                                 int cnt) {
  const int32_t share = (int32_t)(D.face_cap / (D.cchunk1 - D.cchunk0));
  const int32_t p = atomicAdd(&V.part[1][chunk], cnt);
  if (p + cnt <= share) return (int32_t)(D.face_base + (int64_t)(chunk - D.cchunk0) * share + p);
  const int32_t o = atomicAdd(&S.nf_tmp, cnt);
  return (int64_t)o + cnt <= D.face_cap ? (int32_t)(B.F.nf + D.face_base + o) : -1;
}

__device__ __forceinline__ V2Face* v_faces_at(const Batch& B, const V2Bufs& V, int32_t start) {
  const int32_t nf = (int32_t)B.F.nf;  // (below 2^30: CSR values hold a face and a side)
  return start < nf ? V.vf + (uint32_t)start : (V2Face*)B.F.rec + (uint32_t)(start - nf);
}

// The finished cell: area and centroid summed over the edges in order (the host tessellator's
// Cell2::finish), the emitted faces appended to vf in edge order, and the cell's geometry
// (Particle::update_geometry, part.rs:151-158).
template <int TL>
__device__ void v2_finish(const Batch& B, const V2Bufs& V, const SimDesc& D, SimStep& S, int chunk, int64_t gi,
                          int32_t i, double xi, double yi, double zi, const V2TeamPoly<TL>& P, int m) {
  const int64_t N = B.C.n, cb = D.cell_base;
  double area = 0., cx = 0., cy = 0., r2 = 0.;
  int cnt = 0;
  for (int k = 0; k < m; ++k) {
    const int km = k == 0 ? m - 1 : k - 1;
    const double ax = P.vx[km], ay = P.vy[km], bxx = P.vx[k], byy = P.vy[k];
    const double cr = ax * byy - bxx * ay;
    area += 0.5 * cr;
    cx = cx + (cr / 6.0) * (ax + bxx);
    cy = cy + (cr / 6.0) * (ay + byy);
    const double len = sqrt((bxx - ax) * (bxx - ax) + (byy - ay) * (byy - ay));
    if (len > 0. && v2_emits(B, cb, P.nb[k], i)) ++cnt;
    const double q = bxx * bxx + byy * byy;
    r2 = r2 < q ? q : r2;
  }
  const int32_t start = v_place_faces(B, V, D, S, chunk, cnt);
  if (start < 0) {
    V.femit[gi] = 0;
    atomicCAS(&B.cnt->err, 0, E_MESH);
    atomicCAS(&S.err, 0, E_MESH);
    return;
  }
  V.vst[gi] = start;
  V.femit[gi] = cnt;
  V2Face* out = v_faces_at(B, V, start);
  int q = 0;
  for (int k = 0; k < m; ++k) {
    const int km = k == 0 ? m - 1 : k - 1;
    const double ax = P.vx[km], ay = P.vy[km], bxx = P.vx[k], byy = P.vy[k];
    const double len = sqrt((bxx - ax) * (bxx - ax) + (byy - ay) * (byy - ay));
    if (!(len > 0.) || !v2_emits(B, cb, P.nb[k], i)) continue;
    const double inv = 1.0 / sqrt(P.nx[k] * P.nx[k] + P.ny[k] * P.ny[k]);
    V2Face f;
    f.area = len;
    f.cx = 0.5 * (ax + bxx);
    f.cy = 0.5 * (ay + byy);
    f.cz = 0.;
    f.nx = inv * P.nx[k];
    f.ny = inv * P.ny[k];
    f.nz = 0.;
    f.nb = P.nb[k] < 0 ? -1 : P.nb[k];
    f.code = P.code[k];
    out[q++] = f;
  }
  if (B.C.act[gi]) {
    B.C.vol[gi] = area;
    const double ia = area > 0. ? 1.0 / area : 0.;
    B.C.cen[gi] = xi + (area > 0. ? ia * cx : 0.);
    B.C.cen[N + gi] = yi + (area > 0. ? ia * cy : 0.);
    B.C.cen[2 * N + gi] = zi;
    B.C.srad[gi] = 1.5 * 2.0 * sqrt(r2);
  }
}

// LDS writes of a team visible to the team's next reads (a team is part of one wavefront)
__device__ __forceinline__ void team_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}
__device__ __forceinline__ uint32_t team_ballot(bool p, int tiw) {
  return (uint32_t)((__ballot(p) >> (HFV_V2_TEAM * tiw)) & ((1ull << HFV_V2_TEAM) - 1));
}

// vertex k: the intersection of edges k and k+1 (0 where they are parallel)
template <int TL>
__device__ __forceinline__ void team_recompute(V2TeamPoly<TL>& P, int m, int lane) {
#pragma unroll
  for (int t = 0; t < TL; t += HFV_V2_TEAM) {
    const int k = t + lane;
    if (k < m) {
      const int k1 = k + 1 == m ? 0 : k + 1;
      const double nx0 = P.nx[k], ny0 = P.ny[k], d0 = P.d[k], nx1 = P.nx[k1], ny1 = P.ny[k1], d1 = P.d[k1];
      const double det = nx0 * ny1 - ny0 * nx1;
      if (det == 0.0) {
        P.vx[k] = 0.;
        P.vy[k] = 0.;
      } else {
        P.vx[k] = (d0 * ny1 - d1 * ny0) / det;
        P.vy[k] = (nx0 * d1 - nx1 * d0) / det;
      }
    }
  }
  team_sync();
}

template <int TL>
__device__ __forceinline__ double team_rmax2(const V2TeamPoly<TL>& P, int m, int lane) {
  double r = 0.;
#pragma unroll
  for (int t = 0; t < TL; t += HFV_V2_TEAM) {
    const int k = t + lane;
    if (k < m) {
      const double q = P.vx[k] * P.vx[k] + P.vy[k] * P.vy[k];
      r = r < q ? q : r;
    }
  }
#pragma unroll
  for (int o = HFV_V2_TEAM / 2; o > 0; o >>= 1) {
    const double q = __shfl_xor(r, o, HFV_V2_TEAM);
    r = r < q ? q : r;
  }
  return r;
}

// Clip by the half-plane n.y <= dd: 0 no cut, 1 cut, -1 more than TL edges.  The run of outside vertices
// start .. start+nout-1 is contiguous; edges start+1 .. start+nout-1 go, the new edge follows edge start,
// and the list restarts at the first kept edge after the removed run.
template <int TL>
__device__ __forceinline__ int team_clip(V2TeamPoly<TL>& P, int& m, double a, double b, double dd, int32_t n_,
                                         int32_t c_, int lane, int tiw) {
  static_assert(TL <= 64 && TL % HFV_V2_TEAM == 0, "edge masks");
  uint64_t om = 0;
#pragma unroll
  for (int t = 0; t < TL; t += HFV_V2_TEAM) {
    const int k = t + lane;
    const bool o = k < m && (a * P.vx[k] + b * P.vy[k]) > dd + HFV_CLIP_TOL * dd;
    om |= (uint64_t)team_ballot(o, tiw) << t;
  }
  const int nout = __popcll(om);
  if (nout == 0 || nout == m) return 0;
  const int q = m - nout + 2;
  if (q > TL) return -1;
  const uint64_t full = m == 64 ? ~0ull : (1ull << m) - 1ull;
  const uint64_t prev = ((om << 1) | (om >> (m - 1))) & full;  // bit k: vertex k-1 is outside
  const uint64_t sm = om & ~prev;
  const int start = sm ? __builtin_ctzll(sm) : 0;
  const int keep = (start + nout) % m;
  constexpr int R = TL / HFV_V2_TEAM;
  double rx[R], ry[R], rd[R];
  int32_t rn[R], rc[R];
#pragma unroll
  for (int t = 0; t < R; ++t) {
    const int p = t * HFV_V2_TEAM + lane;
    if (p < q - 1) {
      int o = keep + p;
      o = o >= m ? o - m : o;
      rx[t] = P.nx[o];
      ry[t] = P.ny[o];
      rd[t] = P.d[o];
      rn[t] = P.nb[o];
      rc[t] = P.code[o];
    }
  }
  team_sync();
#pragma unroll
  for (int t = 0; t < R; ++t) {
    const int p = t * HFV_V2_TEAM + lane;
    if (p < q - 1) {
      P.nx[p] = rx[t];
      P.ny[p] = ry[t];
      P.d[p] = rd[t];
      P.nb[p] = rn[t];
      P.code[p] = rc[t];
    }
  }
  if (lane == 0) {
    P.nx[q - 1] = a;
    P.ny[q - 1] = b;
    P.d[q - 1] = dd;
    P.nb[q - 1] = n_;
    P.code[q - 1] = c_;
  }
  team_sync();
  m = q;
  team_recompute(P, m, lane);
  return 1;
}

// The candidate key and plane of one generator image (bins wrapped once on a periodic box).
struct V2Cand {
  double d2, rx, ry;
  int32_t j, k, code;
};

// Visit this lane's candidates of the (2K+1)^2 block: f(cand) for each.
template <class Fn>
__device__ __forceinline__ void v2_lane_candidates(const Batch& B, const SimDesc& D, const V2Bufs& V, int s, int32_t i,
                                                   double xi, double yi, double zi, int K, int lane, Fn&& f) {
  const int64_t N = B.C.n, cb = D.cell_base;
  const double* L = B.C.loc;
  const double bx = D.cfg.box[0], by = D.cfg.box[1], bz = D.cfg.box[2];
  const int nb0 = D.vnb[0], nb1 = D.vnb[1];
  const bool per = D.periodic != 0;
  const int bi0 = v2_bin(xi, D.vw[0], nb0), bi1 = v2_bin(yi, D.vw[1], nb1);
  const int32_t* gst = V.gcnt + cb + s;
  const int32_t* gord = V.gord + cb;
  const int side = 2 * K + 1;
  for (int bb = lane; bb < side * side; bb += HFV_V2_TEAM) {
    int b0 = bi0 + bb / side - K, b1 = bi1 + bb % side - K, s0 = 0, s1 = 0;
    if (b0 < 0 || b0 >= nb0) {
      if (!per) continue;
      if (b0 < 0) {
        b0 += nb0;
        s0 = -1;
      } else {
        b0 -= nb0;
        s0 = 1;
      }
      if (b0 < 0 || b0 >= nb0) continue;
    }
    if (b1 < 0 || b1 >= nb1) {
      if (!per) continue;
      if (b1 < 0) {
        b1 += nb1;
        s1 = -1;
      } else {
        b1 -= nb1;
        s1 = 1;
      }
      if (b1 < 0 || b1 >= nb1) continue;
    }
    const int key = b0 * nb1 + b1;
    const int32_t kk = ((s0 & 0xFF) << 16) | ((s1 & 0xFF) << 8);  // the host's memcmp order of the int8 codes
    const int32_t code = v2_shift_code(s0, s1);
    for (int32_t q = gst[key]; q < gst[key + 1]; ++q) {
      const int32_t j = gord[q];
      if (j == i && s0 == 0 && s1 == 0) continue;
      const int64_t gj = cb + j;
      const double xj = L[gj] + (double)s0 * bx, yj = L[N + gj] + (double)s1 * by, zj = L[2 * N + gj] + 0.0 * bz;
      V2Cand c;
      c.rx = xj - xi;
      c.ry = yj - yi;
      const double rz = zj - zi;
      c.d2 = c.rx * c.rx + c.ry * c.ry + rz * rz;
      c.j = j;
      c.k = kk;
      c.code = code;
      f(c);
    }
  }
}

// Team minimum of the lanes' best candidates (unique keys: every lane ends with the same one).
__device__ __forceinline__ void team_min(bool& have, V2Cand& b) {
#pragma unroll
  for (int o = HFV_V2_TEAM / 2; o > 0; o >>= 1) {
    const int oh = __shfl_xor((int)have, o, HFV_V2_TEAM);
    V2Cand c;
    c.d2 = __shfl_xor(b.d2, o, HFV_V2_TEAM);
    c.rx = __shfl_xor(b.rx, o, HFV_V2_TEAM);
    c.ry = __shfl_xor(b.ry, o, HFV_V2_TEAM);
    c.j = __shfl_xor(b.j, o, HFV_V2_TEAM);
    c.k = __shfl_xor(b.k, o, HFV_V2_TEAM);
    c.code = __shfl_xor(b.code, o, HFV_V2_TEAM);
    if (oh && (!have || v2_less(c.d2, c.j, c.k, b.d2, b.j, b.k))) {
      have = true;
      b = c;
    }
  }
}

// The cell of generator i with candidate bins within K, any number of candidates: 0 built, 1 retry with a
// larger K, 2 more than TL edges.
template <int TL>
__device__ int v2_team_build(const Batch& B, const SimDesc& D, const V2Bufs& V, int s, int32_t i, double xi,
                             double yi, double zi, int K, V2TeamPoly<TL>& P, int& m, double& r2, int lane, int tiw) {
  const double w0 = D.vw[0], w1 = D.vw[1];
  const bool per = D.periodic != 0;
  // initial region: the box, or K bin widths around the generator on a periodic box
  double reach = 0.;
  reach = reach < K * w0 ? K * w0 : reach;
  reach = reach < K * w1 ? K * w1 : reach;
  const double lox = per ? -reach : -xi, loy = per ? -reach : -yi;
  const double hix = per ? reach : D.cfg.box[0] - xi, hiy = per ? reach : D.cfg.box[1] - yi;
  if (lane < 4) {  // counter-clockwise: bottom, right, top, left (walls -3, -2, -4, -1)
    P.nx[lane] = lane == 1 ? 1. : lane == 3 ? -1. : 0.;
    P.ny[lane] = lane == 0 ? -1. : lane == 2 ? 1. : 0.;
    P.d[lane] = lane == 0 ? -loy : lane == 1 ? hix : lane == 2 ? hiy : -lox;
    P.nb[lane] = lane == 0 ? -3 : lane == 1 ? -2 : lane == 2 ? -4 : -1;
    P.code[lane] = 0;
  }
  team_sync();
  m = 4;
  team_recompute(P, m, lane);
  r2 = team_rmax2(P, m, lane);
  bool have_last = false;
  V2Cand last{};
  while (true) {
    bool have = false;
    V2Cand best{};
    auto consider = [&](const V2Cand& c) {
      if ((!have_last || v2_less(last.d2, last.j, last.k, c.d2, c.j, c.k)) &&
          (!have || v2_less(c.d2, c.j, c.k, best.d2, best.j, best.k))) {
        have = true;
        best = c;
      }
    };
    v2_lane_candidates(B, D, V, s, i, xi, yi, zi, K, lane, consider);
    team_min(have, best);
    if (!have || 0.25 * best.d2 > r2) break;  // security radius: the bisector lies beyond every vertex
    const int c = team_clip(P, m, best.rx, best.ry, 0.5 * best.d2, best.j, best.code, lane, tiw);
    if (c < 0) return 2;
    if (c > 0) r2 = team_rmax2(P, m, lane);
    have_last = true;
    last = best;
  }
  // completeness: every unvisited generator lies farther than K bin widths
  double minw = 1e300;
  minw = K * w0 < minw ? K * w0 : minw;
  minw = K * w1 < minw ? K * w1 : minw;
  if (4.0 * r2 > minw * minw) return 1;
  if (per) {  // a periodic cell must not touch the initial region
    bool wall = false;
#pragma unroll
    for (int t = 0; t < TL; t += HFV_V2_TEAM) {
      const int k = t + lane;
      if (k < m) {
        const int km = k == 0 ? m - 1 : k - 1;
        const double ex = P.vx[k] - P.vx[km], ey = P.vy[k] - P.vy[km];
        wall = wall || (P.nb[k] < 0 && sqrt(ex * ex + ey * ey) > 0.);
      }
    }
    if (team_ballot(wall, tiw)) return 1;
  }
  return 0;
}

struct V2TeamCands {
  double d2[HFV_V2_CAP], rx[HFV_V2_CAP], ry[HFV_V2_CAP];
  int32_t j[HFV_V2_CAP], k[HFV_V2_CAP];
  uint8_t ord[HFV_V2_CAP];  // candidate of each rank
  int32_t n;
};

// A team's polygon: this lane's edge (plane, neighbour, image code) and the vertex between it and the next.
struct V2RegPoly {
  double nx, ny, d, vx, vy;
  int32_t nb, code;
};

template <int CTRL>
__device__ __forceinline__ double row_max_step(double v) {
  const int lo = __double2loint(v), hi = __double2hiint(v);
  const double t = __hiloint2double(__builtin_amdgcn_update_dpp(hi, hi, CTRL, 0xf, 0xf, false),
                                    __builtin_amdgcn_update_dpp(lo, lo, CTRL, 0xf, 0xf, false));
  return v < t ? t : v;
}
// maximum over the team (a DPP row: row_ror 8, 4, 2, 1), in every lane
__device__ __forceinline__ double team_max(double v) {
  static_assert(HFV_V2_TEAM == 16, "a team is a DPP row");
  v = row_max_step<0x128>(v);
  v = row_max_step<0x124>(v);
  v = row_max_step<0x122>(v);
  return row_max_step<0x121>(v);
}

// every vertex from its edge and the next one (0 where they are parallel); the largest squared radius
__device__ __forceinline__ double v2_vertices(V2RegPoly& P, int m, int lane) {
  const int k1 = lane + 1 == m ? 0 : lane + 1;
  const double nx1 = __shfl(P.nx, k1, HFV_V2_TEAM), ny1 = __shfl(P.ny, k1, HFV_V2_TEAM), d1 = __shfl(P.d, k1, HFV_V2_TEAM);
  double r = 0.;
  if (lane < m) {
    const double det = P.nx * ny1 - P.ny * nx1;
    P.vx = 0.;
    P.vy = 0.;
    if (det != 0.0) {
      P.vx = (P.d * ny1 - d1 * P.ny) / det;
      P.vy = (P.nx * d1 - nx1 * P.d) / det;
    }
    const double q = P.vx * P.vx + P.vy * P.vy;
    r = r < q ? q : r;
  }
  return team_max(r);
}

// The candidates of the (2K+1)^2 block into LDS (any order: the rank orders them), each lane taking every 16th
// bin, four candidates' loads in flight: their count, or -1 beyond HFV_V2_CAP.
__device__ __forceinline__ int v2_gather(const Batch& B, const SimDesc& D, const V2Bufs& V, int s, int32_t i, double xi,
                                         double yi, double zi, int K, V2TeamCands& Q, int lane, int tiw) {
  const int64_t N = B.C.n, cb = D.cell_base;
  const double* L = B.C.loc;
  const double bx = D.cfg.box[0], by = D.cfg.box[1], bz = D.cfg.box[2];
  const int nb0 = D.vnb[0], nb1 = D.vnb[1];
  const bool per = D.periodic != 0;
  const int bi0 = v2_bin(xi, D.vw[0], nb0), bi1 = v2_bin(yi, D.vw[1], nb1);
  const int32_t* gst = V.gcnt + cb + s;
  const int32_t* gord = V.gord + cb;
  const int side = 2 * K + 1;
  if (lane == 0) Q.n = 0;
  team_sync();
  for (int bb = lane; bb < side * side; bb += HFV_V2_TEAM) {
    int b0 = bi0 + bb / side - K, b1 = bi1 + bb % side - K, s0 = 0, s1 = 0;
    bool skip = false;
    if (b0 < 0 || b0 >= nb0) {
      s0 = b0 < 0 ? -1 : 1;
      b0 -= s0 * nb0;
      skip = !per || b0 < 0 || b0 >= nb0;
    }
    if (b1 < 0 || b1 >= nb1) {
      s1 = b1 < 0 ? -1 : 1;
      b1 -= s1 * nb1;
      skip = skip || !per || b1 < 0 || b1 >= nb1;
    }
    if (skip) continue;
    const int key = b0 * nb1 + b1;
    const int32_t kk = ((s0 & 0xFF) << 16) | ((s1 & 0xFF) << 8);  // the host's memcmp order of the int8 codes
    const int32_t g0 = gst[key], g1 = gst[key + 1];
    for (int32_t q0 = g0; q0 < g1; q0 += 4) {
      int32_t jj[4];
      double x[4], y[4], z[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) jj[u] = q0 + u < g1 ? gord[q0 + u] : -1;
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int64_t gj = cb + (jj[u] < 0 ? 0 : jj[u]);
        x[u] = L[gj];
        y[u] = L[N + gj];
        z[u] = L[2 * N + gj];
      }
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        if (jj[u] < 0 || (jj[u] == i && s0 == 0 && s1 == 0)) continue;
        const double xj = x[u] + (double)s0 * bx, yj = y[u] + (double)s1 * by, zj = z[u] + 0.0 * bz;
        const double rx = xj - xi, ry = yj - yi, rz = zj - zi;
        const int at = atomicAdd(&Q.n, 1);
        if (at >= HFV_V2_CAP) continue;
        Q.d2[at] = rx * rx + ry * ry + rz * rz;
        Q.rx[at] = rx;
        Q.ry[at] = ry;
        Q.j[at] = jj[u];
        Q.k[at] = kk;
      }
    }
  }
  team_sync();
  const int n = Q.n;
  return n > HFV_V2_CAP ? -1 : n;
}

// ord[rank] = candidate, by squared distance (a non-negative double orders as its bits), and by the whole key
// where two squared distances are equal.
__device__ __forceinline__ void v2_rank(V2TeamCands& Q, int n, int lane, int tiw) {
  const int nown = (n + HFV_V2_TEAM - 1) / HFV_V2_TEAM;
  const uint64_t* D2 = reinterpret_cast<const uint64_t*>(Q.d2);
  for (int h = 0; h < nown; ++h) {
    const int a = lane + HFV_V2_TEAM * h;
    const int aa = a < n ? a : 0;
    const uint64_t od = D2[aa];
    int rk = 0, le = 0;
    for (int b = 0; b < n; b += 8) {
      uint64_t db[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) db[u] = b + u < n ? D2[b + u] : ~0ull;
#pragma unroll
      for (int u = 0; u < 8; ++u) {
        rk += db[u] < od ? 1 : 0;
        le += db[u] <= od ? 1 : 0;
      }
    }
    if (a < n && le - rk > 1) {  // (rare)
      const int32_t oj = Q.j[a], ok = Q.k[a];
      for (int b = 0; b < n; ++b)
        rk += D2[b] == od && (Q.j[b] < oj || (Q.j[b] == oj && Q.k[b] < ok)) ? 1 : 0;
    }
    if (a < n) Q.ord[rk] = (uint8_t)a;
  }
  team_sync();
}

// The cell of generator i with candidate bins within K: 0 built, 1 retry with a larger K, 2 too many
// candidates or edges.
__device__ __forceinline__ int v2_reg_build(const Batch& B, const SimDesc& D, const V2Bufs& V, int s, int32_t i,
                                            double xi, double yi, double zi, int K, V2TeamCands& Q, V2RegPoly& P, int& m,
                                            double& r2, int lane, int tiw) {
  const double w0 = D.vw[0], w1 = D.vw[1];
  const bool per = D.periodic != 0;
  // initial region: the box, or K bin widths around the generator on a periodic box
  double reach = 0.;
  reach = reach < K * w0 ? K * w0 : reach;
  reach = reach < K * w1 ? K * w1 : reach;
  const double lox = per ? -reach : -xi, loy = per ? -reach : -yi;
  const double hix = per ? reach : D.cfg.box[0] - xi, hiy = per ? reach : D.cfg.box[1] - yi;
  // counter-clockwise: bottom, right, top, left (walls -3, -2, -4, -1)
  P.nx = lane == 1 ? 1. : lane == 3 ? -1. : 0.;
  P.ny = lane == 0 ? -1. : lane == 2 ? 1. : 0.;
  P.d = lane == 0 ? -loy : lane == 1 ? hix : lane == 2 ? hiy : -lox;
  P.nb = lane == 0 ? -3 : lane == 1 ? -2 : lane == 2 ? -4 : -1;
  P.code = 0;
  P.vx = 0.;
  P.vy = 0.;
  m = 4;
  r2 = v2_vertices(P, m, lane);
  const int n = v2_gather(B, D, V, s, i, xi, yi, zi, K, Q, lane, tiw);
  if (n < 0) return 2;
  v2_rank(Q, n, lane, tiw);
  int a = n > 0 ? Q.ord[0] : 0;
  double cd2 = Q.d2[a], cx = Q.rx[a], cy = Q.ry[a];
  for (int q = 0; q < n; ++q) {
    if (0.25 * cd2 > r2) break;  // security radius: the bisector lies beyond every vertex
    const int now = a;
    const double ca = cx, cbb = cy, dd = 0.5 * cd2;
    a = Q.ord[q + 1 < n ? q + 1 : q];  // the next candidate, in flight during the clip
    cd2 = Q.d2[a];
    cx = Q.rx[a];
    cy = Q.ry[a];
    // clip by the half-plane (ca, cbb).y <= dd: the run of outside vertices start .. start+nout-1 is contiguous;
    // edges start+1 .. start+nout-1 go, the new edge follows edge start, and the list restarts at the first
    // kept edge after the removed run
    const bool out = lane < m && (ca * P.vx + cbb * P.vy) > dd + HFV_CLIP_TOL * dd;
    const uint32_t om = team_ballot(out, tiw);
    const int nout = __popc(om);
    if (nout == 0 || nout == m) continue;
    const int mq = m - nout + 2;
    if (mq > HFV_V2_TEAM) return 2;
    const uint32_t full = (1u << m) - 1u;
    const uint32_t prev = ((om << 1) | (om >> (m - 1))) & full;  // bit k: vertex k-1 is outside
    const uint32_t sm = om & ~prev;
    const int start = sm ? __builtin_ctz(sm) : 0;
    int src = start + nout;
    src = src >= m ? src - m : src;
    src += lane;
    src = src >= m ? src - m : src;  // (lanes past the kept edges read any lane)
    const double ex = __shfl(P.nx, src, HFV_V2_TEAM), ey = __shfl(P.ny, src, HFV_V2_TEAM), ed = __shfl(P.d, src, HFV_V2_TEAM);
    const int32_t en = __shfl(P.nb, src, HFV_V2_TEAM), ec = __shfl(P.code, src, HFV_V2_TEAM);
    const bool fresh = lane == mq - 1;
    const int32_t ck = Q.k[now];
    P.nx = fresh ? ca : ex;
    P.ny = fresh ? cbb : ey;
    P.d = fresh ? dd : ed;
    P.nb = fresh ? Q.j[now] : en;
    P.code = fresh ? v2_shift_code((int8_t)((ck >> 16) & 0xFF), (int8_t)((ck >> 8) & 0xFF)) : ec;
    m = mq;
    r2 = v2_vertices(P, m, lane);
  }
  // completeness: every unvisited generator lies farther than K bin widths
  double minw = 1e300;
  minw = K * w0 < minw ? K * w0 : minw;
  minw = K * w1 < minw ? K * w1 : minw;
  if (4.0 * r2 > minw * minw) return 1;
  if (per) {  // a periodic cell must not touch the initial region
    const int km = lane == 0 ? m - 1 : lane - 1;
    const double ex = P.vx - __shfl(P.vx, km, HFV_V2_TEAM), ey = P.vy - __shfl(P.vy, km, HFV_V2_TEAM);
    if (team_ballot(lane < m && P.nb < 0 && sqrt(ex * ex + ey * ey) > 0., tiw)) return 1;
  }
  return 0;
}

// v2_finish of a team's register polygon, each edge on its lane; the sums are added in edge order.
__device__ __forceinline__ void v2_reg_finish(const Batch& B, const V2Bufs& V, const SimDesc& D, SimStep& S, int chunk,
                                              int64_t gi, int32_t i, double xi, double yi, double zi, const V2RegPoly& P,
                                              int m, int lane, int tiw) {
  const int64_t N = B.C.n, cb = D.cell_base;
  const int km = lane == 0 ? m - 1 : lane - 1;
  const double ax = __shfl(P.vx, km, HFV_V2_TEAM), ay = __shfl(P.vy, km, HFV_V2_TEAM), bxx = P.vx, byy = P.vy;
  const double cr = ax * byy - bxx * ay;
  const double ta = 0.5 * cr, tx = (cr / 6.0) * (ax + bxx), ty = (cr / 6.0) * (ay + byy);
  const double len = sqrt((bxx - ax) * (bxx - ax) + (byy - ay) * (byy - ay));
  const bool emit = lane < m && len > 0. && v2_emits(B, cb, P.nb, i);
  double q = 0.;
  if (lane < m) {
    const double qq = bxx * bxx + byy * byy;
    q = q < qq ? qq : q;
  }
  const double r2 = team_max(q);
  double area = 0., cx = 0., cy = 0.;
  for (int k = 0; k < m; ++k) {
    area += __shfl(ta, k, HFV_V2_TEAM);
    cx = cx + __shfl(tx, k, HFV_V2_TEAM);
    cy = cy + __shfl(ty, k, HFV_V2_TEAM);
  }
  const uint32_t em = team_ballot(emit, tiw);
  const int cnt = __popc(em);
  int32_t start = 0;
  if (lane == 0) start = v_place_faces(B, V, D, S, chunk, cnt);
  start = __shfl(start, 0, HFV_V2_TEAM);
  if (start < 0) {
    if (lane == 0) {
      V.femit[gi] = 0;
      atomicCAS(&B.cnt->err, 0, E_MESH);
      atomicCAS(&S.err, 0, E_MESH);
    }
    return;
  }
  if (emit) {
    const double inv = 1.0 / sqrt(P.nx * P.nx + P.ny * P.ny);
    V2Face f;
    f.area = len;
    f.cx = 0.5 * (ax + bxx);
    f.cy = 0.5 * (ay + byy);
    f.cz = 0.;
    f.nx = inv * P.nx;
    f.ny = inv * P.ny;
    f.nz = 0.;
    f.nb = P.nb < 0 ? -1 : P.nb;
    f.code = P.code;
    v_faces_at(B, V, start)[__popc(em & ((1u << lane) - 1u))] = f;
  }
  if (lane != 0) return;
  V.vst[gi] = start;
  V.femit[gi] = cnt;
  if (B.C.act[gi]) {
    B.C.vol[gi] = area;
    const double ia = area > 0. ? 1.0 / area : 0.;
    B.C.cen[gi] = xi + (area > 0. ? ia * cx : 0.);
    B.C.cen[N + gi] = yi + (area > 0. ? ia * cy : 0.);
    B.C.cen[2 * N + gi] = zi;
    B.C.srad[gi] = 1.5 * 2.0 * sqrt(r2);
  }
}

// grid: HFV_V2_SUB blocks per cell chunk, HFV_BLOCK / HFV_V2_TEAM cells per block.
__global__ void __launch_bounds__(HFV_BLOCK) k_v2_cells(Batch B, V2Bufs V) {
  union Team {
    V2TeamCands q;
    V2TeamPoly<HFV_V2_TLW> wide;
  };
  __shared__ Team teams[HFV_BLOCK / HFV_V2_TEAM];
  const BlockJob J = B.cjobs[blockIdx.x / HFV_V2_SUB];
  if (J.sim < 0) return;
  const int s = J.sim;
  const SimDesc& D = B.sims[s];
  SimStep& S = B.st[s];
  if (D.vmesh != 2 || !S.stepping) return;
  const int team = threadIdx.x / HFV_V2_TEAM, lane = threadIdx.x % HFV_V2_TEAM;
  const int tiw = (threadIdx.x & 63) / HFV_V2_TEAM;
  const int64_t gi = (int64_t)J.lo + (blockIdx.x % HFV_V2_SUB) * (HFV_BLOCK / HFV_V2_TEAM) + team;
  if (gi >= J.hi) return;  // whole teams; no block barrier follows
  const int64_t N = B.C.n, cb = D.cell_base;
  const int32_t i = (int32_t)(gi - cb);
  if (lane == 0) V.ccnt[gi] = 0;
  if (!B.C.act[gi]) {  // unbuilt in a partial build
    if (lane == 0) V.femit[gi] = 0;
    return;
  }
  const double xi = B.C.loc[gi], yi = B.C.loc[N + gi], zi = B.C.loc[2 * N + gi];
  Team& T = teams[team];
  int m = 0, r = 1;
  double r2 = 0.;
  const int kmax = max(6, max(D.vnb[0], D.vnb[1]));
  {
    V2RegPoly P;
    for (int K = 2; K <= kmax && r == 1; ++K)
      r = v2_reg_build(B, D, V, s, i, xi, yi, zi, K, T.q, P, m, r2, lane, tiw);
    if (r == 0) {
      v2_reg_finish(B, V, D, S, J.chunk, gi, i, xi, yi, zi, P, m, lane, tiw);
      return;
    }
  }
  if (r == 2) {
    r = 1;
    for (int K = 2; K <= kmax && r == 1; ++K)
      r = v2_team_build<HFV_V2_TLW>(B, D, V, s, i, xi, yi, zi, K, T.wide, m, r2, lane, tiw);
  }
  if (lane != 0) return;
  if (r != 0) {
    V.femit[gi] = 0;
    atomicCAS(&B.cnt->err, 0, E_MESH);
    atomicCAS(&S.err, 0, E_MESH);
  } else {
    v2_finish(B, V, D, S, J.chunk, gi, i, xi, yi, zi, T.wide, m);
  }
}

// ---------------------------------------------------------------- faces and CSR
// The faces of a chunk's cells, in cell order after the faces of the chunks before: face arrays, and the
// entries of both cells into their buckets.  The block's threads take its faces in turn, whichever cell
// emitted them (a binary search of the cells' offsets in LDS).
// (Chaining the entries beyond the buckets here, and telling the two places of provisional faces apart for each
// face instead of each cell, this kernel took 19.3 us instead of 18.3 on a 125^2 vortex.)
template <bool SCANNED>
__global__ void __launch_bounds__(HFV_BLOCK) k_v2_faces(Batch B, V2Bufs V) {
  __shared__ int32_t offs[HFV_BLOCK];
  __shared__ const V2Face* starts[HFV_BLOCK];
  const BlockJob J = B.cjobs[blockIdx.x];
  if (J.sim < 0) return;
  const int s = J.sim;
  const SimDesc& D = B.sims[s];
  SimStep& S = B.st[s];
  if (!D.vmesh || !S.stepping) return;
  const int64_t cb = D.cell_base, NF = B.F.nf, N = B.C.n;
  const int64_t gi0 = (int64_t)J.lo + threadIdx.x;
  const bool in = gi0 < J.hi;
  int32_t all, tot;
  const int32_t base = chunks_before<SCANNED>(V, 1, D, s, J.chunk, &all);
  offs[threadIdx.x] = block_excl_scan(in ? V.femit[gi0] : 0, &tot);
  starts[threadIdx.x] = v_faces_at(B, V, in ? V.vst[gi0] : 0);
  const bool full = all > D.face_cap;
  const bool bad = full || S.err != 0;  // a failed cell emitted nothing: the simulation stops
  if (J.chunk == D.cchunk0 && threadIdx.x == 0) {
    B.eng[s].nf_mesh = bad ? 0 : all;
    if (full) {
      atomicCAS(&B.cnt->err, 0, E_MESH);
      atomicCAS(&S.err, 0, E_MESH);
    }
  }
  __syncthreads();
  if (bad) return;
  const Faces& F = B.F;
  for (int32_t t = threadIdx.x; t < tot; t += HFV_BLOCK) {
    int lo = 0;  // the last cell whose offset is <= t (earlier cells of the same offset emit nothing)
#pragma unroll
    for (int h = HFV_BLOCK / 2; h > 0; h >>= 1)
      if (offs[lo + h] <= t) lo += h;
    const int64_t gi = (int64_t)J.lo + lo;
    const int64_t f = D.face_base + base + t;
    const V2Face r = starts[lo][t - offs[lo]];
    F.area[f] = r.area;
    F.nrm[f] = r.nx;
    F.nrm[NF + f] = r.ny;
    F.nrm[2 * NF + f] = D.vmesh == 3 ? r.nz : 0.;
    F.fcen[f] = B.C.loc[gi] + r.cx;
    F.fcen[NF + f] = B.C.loc[N + gi] + r.cy;
    F.fcen[2 * NF + f] = D.vmesh == 3 ? B.C.loc[2 * N + gi] + r.cz : B.C.loc[2 * N + gi];
    const int32_t right = r.nb < 0 ? -1 : (int32_t)(cb + r.nb);
    F.left[f] = (int32_t)gi;
    F.right[f] = right;
    F.shc[f] = (uint8_t)r.code;
    auto put = [&](int32_t cell, int32_t conn, int32_t nbr) {
      const int32_t q = atomicAdd(&V.ccnt[cell], 1);
      if (q < HFV_BUCKET) {
        V.bkt[(int64_t)q * N + cell] = ((uint64_t)(uint32_t)conn << 32) | (uint32_t)nbr;
        return;
      }
      const int32_t o = atomicAdd(&S.n_over, 1);
      if (o < 2 * D.face_cap) v_over(B, D)[o] = V2Over{cell, conn, nbr, -1};
    };
    put((int32_t)gi, (int32_t)(f << 1), right);
    if (right >= 0) put(right, (int32_t)((f << 1) | 1), (int32_t)gi);
  }
}

// CSR offsets, and every cell's entries in ascending face order (then side): CSR values are distinct and
// non-negative, so the packed words order as they do.  The bin counts restart at zero.
template <bool SCANNED>
__global__ void __launch_bounds__(HFV_BLOCK) k_v2_conn(Batch B, V2Bufs V) {
  __shared__ uint64_t ent[HFV_BUCKET][HFV_BLOCK];  // [slot][thread]
  const BlockJob J = B.cjobs[blockIdx.x];
  if (J.sim < 0) return;
  const int s = J.sim;
  const SimDesc& D = B.sims[s];
  SimStep& S = B.st[s];
  if (!D.vmesh || !S.stepping) return;
  const int64_t gi = (int64_t)J.lo + threadIdx.x, N = B.C.n;
  const bool in = gi < J.hi;
  const int64_t bin = gi - D.cell_base;
  if (bin < (int64_t)D.vnb[0] * D.vnb[1] * D.vnb[2]) V.gcnt[D.cell_base + s + bin] = 0;
  const int m = in ? V.ccnt[gi] : 0;
  int32_t all, tot;
  const int32_t base = chunks_before<SCANNED>(V, 2, D, s, J.chunk, &all);
  const int32_t x = base + block_excl_scan(m, &tot);
  const bool full = all > D.conn_cap;
  const bool bad = full || S.err != 0;
  if (full && J.chunk == D.cchunk0 && threadIdx.x == 0) {
    atomicCAS(&B.cnt->err, 0, E_MESH);
    atomicCAS(&S.err, 0, E_MESH);
  }
  const int32_t e0 = (int32_t)D.conn_base + (bad ? 0 : x);
  if (in) B.F.off[gi] = e0;
  if (J.chunk == D.cchunk1 - 1) {  // offsets past the last cell: the slot's end of the CSR
    const int32_t end = (int32_t)D.conn_base + (bad ? 0 : all);
    for (int64_t k = D.n + threadIdx.x; k < D.noff; k += HFV_BLOCK) B.F.off[D.cell_base + k] = end;
  }
  if (bad || !in) return;  // (no block barrier follows)
  int32_t* c = B.F.conn;
  int32_t* nb = B.F.nbr;
  if (m <= HFV_BUCKET) {
    uint64_t* v = &ent[0][threadIdx.x];
    for (int k = 0; k < m; k += 4) {  // (four loads in flight)
      uint64_t w[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) w[u] = k + u < m ? V.bkt[(int64_t)(k + u) * N + gi] : 0;
#pragma unroll
      for (int u = 0; u < 4; ++u)
        if (k + u < m) v[(k + u) * HFV_BLOCK] = w[u];
    }
    for (int k = 1; k < m; ++k) {
      const uint64_t w = v[k * HFV_BLOCK];
      int j = k - 1;
      while (j >= 0 && v[j * HFV_BLOCK] > w) {
        v[(j + 1) * HFV_BLOCK] = v[j * HFV_BLOCK];
        --j;
      }
      v[(j + 1) * HFV_BLOCK] = w;
    }
    for (int k = 0; k < m; ++k) {
      const uint64_t w = v[k * HFV_BLOCK];
      c[e0 + k] = (int32_t)(w >> 32);
      nb[e0 + k] = (int32_t)(uint32_t)w;
    }
    return;
  }
  // more than the bucket holds: its entries and those that k_v2_sum chained to it, sorted in place in memory (with every
  // such cell searching the simulation's whole list, this kernel took 763 us on 262,144 random 3D generators and 5460
  // on 10^6; chained 237 and 682)
  int32_t o = 0;
  for (int32_t at = 0; at < m; ++at) {
    int32_t conn, nbr;
    if (at < HFV_BUCKET) {
      const uint64_t w = V.bkt[(int64_t)at * N + gi];
      conn = (int32_t)(w >> 32);
      nbr = (int32_t)(uint32_t)w;
    } else {
      const V2Over w = v_over(B, D)[at == HFV_BUCKET ? V.gkey[gi] : o];
      conn = w.conn;
      nbr = w.nbr;
      o = w.next;
    }
    int32_t j = e0 + at - 1;
    while (j >= e0 && c[j] > conn) {
      c[j + 1] = c[j];
      nb[j + 1] = nb[j];
      --j;
    }
    c[j + 1] = conn;
    nb[j + 1] = nbr;
  }
}

}  // namespace hfv
