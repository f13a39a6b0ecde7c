// bmx_kernels.hip -- gfx950 kernels of the particle-mechanics path.
//
// Data live in bin-sorted order.  A rebuild bins every particle
// (floor((x - plo) * dxi), src/interpolation/bmx_interp_K.H:55-56), counts
// bins with atomics, scans the counts, scatters (original index, slot)
// pairs, orders each bin by original index, gathers every per-particle array
// into the new order and builds the neighbor rows over the +-1 bin stencil
// in a flat layout, the rows of a force wave's tile of particles back to
// back.  Rows are visited in a fixed order (stencil offsets dz, dy, dx
// lexicographic, ascending original index inside a bin), so the force pass
// sums each particle's pair terms in an order that does not depend on
// thread scheduling.  The force kernel is a gather: particle i reads its row
// and adds only into its own accumulators, as the reference's force lambda
// does (src/des/bmx_pc_interaction.cpp:170-279), then applies the overdamped
// update (src/des/bmx_pc_interaction.cpp:311-449) in the same launch,
// writing the next state into the other half of a ping-pong pair.
#include <algorithm>
#include <type_traits>

#include "bmx_device.h"
#include "bmx_kernels.h"

namespace bmx {

namespace {

constexpr int kWave = 64;

__device__ __forceinline__ unsigned long long dbits(double x) {
  return (unsigned long long)__double_as_longlong(x);
}

// Hardware dispatches workgroup b to XCD b % 8.  With remap, XCD x instead
// works on a contiguous range of tiles, so neighbor gathers of adjacent
// tiles share that XCD's L2.
__device__ __forceinline__ int64_t tile_of(int remap) {
  int64_t b = blockIdx.x, nb = gridDim.x;
  if (!remap) return b;
  int64_t x = b & 7, r = b >> 3, per = nb >> 3, extra = nb & 7;
  return x * per + (x < extra ? x : extra) + r;
}

// Block-wide max / sum through LDS (sh: one slot per wave); every thread
// must call it; the result is valid in thread 0.
template <typename T>
__device__ __forceinline__ T block_max(T v, T *sh) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    T w = __shfl_xor(v, o, kWave);
    v = w > v ? w : v;
  }
  int lane = threadIdx.x & (kWave - 1), wid = threadIdx.x / kWave;
  if (lane == 0) sh[wid] = v;
  __syncthreads();
  if (threadIdx.x == 0)
    for (int w = 1; w < (int)(blockDim.x / kWave); w++) v = sh[w] > v ? sh[w] : v;
  return v;
}
template <typename T>
__device__ __forceinline__ T block_sum(T v, T *sh) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, kWave);
  int lane = threadIdx.x & (kWave - 1), wid = threadIdx.x / kWave;
  if (lane == 0) sh[wid] = v;
  __syncthreads();
  if (threadIdx.x == 0)
    for (int w = 1; w < (int)(blockDim.x / kWave); w++) v += sh[w];
  return v;
}

template <typename T>
__global__ void k_fill(T *p, int64_t n, T v) {
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (; i < n; i += stride) p[i] = v;
}

int grid_for(int64_t n, int block) {
  int64_t g = (n + block - 1) / block;
  if (g < 1) g = 1;
  return (int)g;
}
int grid_capped(int64_t n, int block) {
  int64_t g = (n + block - 1) / block;
  if (g < 1) g = 1;
  if (g > 65536) g = 65536;
  return (int)g;
}

// ------------------------------------------------------------- AoS I/O ---

__global__ void k_aos_unpack(const uint8_t *__restrict__ aos, AosLayout lay,
                             int64_t n, const int32_t *__restrict__ col,
                             const BoxGeom *__restrict__ boxes, BoxGeom g0,
                             StaticArrays st, DynArrays dy,
                             unsigned long long *stats) {
  __shared__ double shd[16];
  __shared__ unsigned long long shu[16];
  int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  double rmax = 0.0, lmax = 0.0;
  unsigned long long flags = 0, nbad = 0;
  if (t < n) {
  const uint8_t *r = aos + t * (int64_t)lay.stride;
  const double *pos = reinterpret_cast<const double *>(r + lay.pos);
  const double *rd = reinterpret_cast<const double *>(r + lay.rdata);
  const int32_t *id = reinterpret_cast<const int32_t *>(r + lay.idata);
  BoxGeom g = g0;
  if (col) g = boxes[col[t]];
  double x = wrap_axis(pos[0], g.plo[0], g.phi[0], g.L[0], g.periodic[0]);
  double y = wrap_axis(pos[1], g.plo[1], g.phi[1], g.L[1], g.periodic[1]);
  double z = wrap_axis(pos[2], g.plo[2], g.phi[2], g.L[2], g.periodic[2]);
  double rad = rd[rec::radius];
  dy.pos[t] = make_double4(x, y, z, rad);
  st.oid[t] = (int32_t)t;
  int ty = id[rec::cell_type];
  st.type[t] = ty;
  if (st.col) st.col[t] = col[t];
  bool bad = !(rad >= 0.0) || !(x == x) || !(y == y) || !(z == z);
  if (ty == rec::YEAST) flags |= 1ull;
  if (ty == rec::FUNGI) flags |= 2ull;
  if (rad >= 0.0) rmax = rad;
  if (dy.rod) {
    double L = rd[rec::c_length], th = rd[rec::theta], ph = rd[rec::phi];
    dy.rod[t] = make_double4(L, th, ph, rd[rec::area]);
    dy.trig[t] = trig_of(th, ph);
    st.bscale[t] = rd[rec::bond_scale];
    Topo tp;
    tp.n_bnds = id[rec::n_bnds];
    for (int b = 0; b < 4; b++) {
      tp.seg_id[b] = id[rec::seg1_id1 + b];
      tp.seg_cpu[b] = id[rec::seg1_id2 + b];
      tp.site[b] = id[rec::site1 + b];
    }
    tp.position = id[rec::position];
    tp.fuse_tip = id[rec::fuse_tip];
    tp.fix_site = id[rec::fix_site];
    tp.self_id = id[rec::id];
    tp.self_cpu = id[rec::cpu];
    tp.dltd = 0;
    tp.pad = 0;
    dy.topo[t] = tp;
    if (ty == rec::FUNGI) {
      if (L >= 0.0) lmax = L;
      if (tp.n_bnds < 0 || tp.n_bnds > 4 || !(L > 0.0)) bad = true;
    }
  }
  if (bad) nbad = 1;
  }
  rmax = block_max(rmax, shd);
  __syncthreads();
  lmax = block_max(lmax, shd);
  __syncthreads();
  nbad = block_sum(nbad, shu);
  __syncthreads();
  unsigned long long fy = block_max(flags & 1ull, shu);
  __syncthreads();
  unsigned long long ff = block_max(flags & 2ull, shu);
  if (threadIdx.x == 0) {
    if (rmax > 0.0) max_u64_to(&stats[0], dbits(rmax));
    if (lmax > 0.0) max_u64_to(&stats[1], dbits(lmax));
    if (fy) or_u64_to(&stats[2], 1ull);
    if (ff) or_u64_to(&stats[3], 1ull);
    if (nbad) atomicAdd(&stats[4], nbad);
  }
}

// Re-reads the selected fields of every bound particle from its record
// into the current sorted arrays (slot t holds original index st.oid[t]),
// the inverse of k_aos_pack for those fields; the sorted order, the static
// arrays and everything not selected are kept.  stats as in k_aos_unpack
// (maxima over the particles after the update, bad records).
__global__ void k_aos_refresh(const uint8_t *__restrict__ aos, AosLayout lay,
                              int64_t n, BoxGeom g, StaticArrays st,
                              DynArrays dy, uint32_t fields,
                              unsigned long long *stats) {
  __shared__ double shd[16];
  __shared__ unsigned long long shu[16];
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  double rmax = 0.0, lmax = 0.0;
  unsigned long long nbad = 0;
  if (t < n) {
    const int64_t o = st.oid[t];
    const uint8_t *r = aos + o * (int64_t)lay.stride;
    const double *pos = reinterpret_cast<const double *>(r + lay.pos);
    const double *rd = reinterpret_cast<const double *>(r + lay.rdata);
    const int32_t *id = reinterpret_cast<const int32_t *>(r + lay.idata);
    double4 p = dy.pos[t];
    if (fields & kFieldPositions) {
      p.x = wrap_axis(pos[0], g.plo[0], g.phi[0], g.L[0], g.periodic[0]);
      p.y = wrap_axis(pos[1], g.plo[1], g.phi[1], g.L[1], g.periodic[1]);
      p.z = wrap_axis(pos[2], g.plo[2], g.phi[2], g.L[2], g.periodic[2]);
    }
    if (fields & kFieldSizes) p.w = rd[rec::radius];
    dy.pos[t] = p;
    bool bad = !(p.w >= 0.0) || !(p.x == p.x) || !(p.y == p.y) || !(p.z == p.z);
    if (p.w >= 0.0) rmax = p.w;
    const int ty = st.type[t];
    if (dy.rod) {
      double4 rr = dy.rod[t];
      if (fields & kFieldSizes) {
        rr.x = rd[rec::c_length];
        rr.w = rd[rec::area];
        st.bscale[t] = rd[rec::bond_scale];
      }
      if (fields & kFieldOrientations) {
        rr.y = rd[rec::theta];
        rr.z = rd[rec::phi];
        dy.trig[t] = trig_of(rr.y, rr.z);
      }
      dy.rod[t] = rr;
      if (fields & kFieldBonds) {
        Topo tp;
        tp.n_bnds = id[rec::n_bnds];
        for (int b = 0; b < 4; b++) {
          tp.seg_id[b] = id[rec::seg1_id1 + b];
          tp.seg_cpu[b] = id[rec::seg1_id2 + b];
          tp.site[b] = id[rec::site1 + b];
        }
        tp.position = id[rec::position];
        tp.fuse_tip = id[rec::fuse_tip];
        tp.fix_site = id[rec::fix_site];
        tp.self_id = id[rec::id];
        tp.self_cpu = id[rec::cpu];
        tp.dltd = 0;
        tp.pad = 0;
        dy.topo[t] = tp;
      }
      if (ty == rec::FUNGI) {
        if (rr.x >= 0.0) lmax = rr.x;
        const int nb = dy.topo[t].n_bnds;
        if (nb < 0 || nb > 4 || !(rr.x > 0.0)) bad = true;
      }
      // lists that survive this call read it
      if (dy.near) dy.near[t] = near_of(p, ty, rr, dy.trig[t], dy.topo[t]);
    }
    if (bad) nbad = 1;
  }
  rmax = block_max(rmax, shd);
  __syncthreads();
  lmax = block_max(lmax, shd);
  __syncthreads();
  nbad = block_sum(nbad, shu);
  if (threadIdx.x == 0) {
    if (rmax > 0.0) max_u64_to(&stats[0], dbits(rmax));
    if (lmax > 0.0) max_u64_to(&stats[1], dbits(lmax));
    if (nbad) atomicAdd(&stats[4], nbad);
  }
}

// fc of the last step, six doubles per particle (force, then torque) in one
// 48-byte run at index t.  Sphere steps keep it in the order of the step, so
// that their stores are whole lines: 307,201 spheres 12.0 us for the pass
// that writes it and 17.4 for the pack that reads it, against 13.1 and 22.5
// in original order; 1M spheres with the chemistry state 34 against 48 for
// the writing pass.  A reorder before its use has it put into the original
// order (k_fc_to_orig).  Segment steps store it in original order: their
// passes reorder between a step and its readers (exchange, fusion), and
// beside the pair law the scattered store does not show.
__device__ __forceinline__ void store_fc(double *__restrict__ fc, int64_t t,
                                         double f0, double f1, double f2,
                                         double f3, double f4, double f5) {
  double2 *q = reinterpret_cast<double2 *>(fc + t * 6);
  q[0] = make_double2(f0, f1);
  q[1] = make_double2(f2, f3);
  q[2] = make_double2(f4, f5);
}
__global__ void k_fc_to_orig(const double *__restrict__ fc,
                             const int32_t *__restrict__ oid, int64_t n,
                             double *__restrict__ out) {
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= n) return;
  const double2 *a = reinterpret_cast<const double2 *>(fc + t * 6);
  double2 *b = reinterpret_cast<double2 *>(out + (int64_t)oid[t] * 6);
  const double2 x = a[0], y = a[1], z = a[2];
  b[0] = x;
  b[1] = y;
  b[2] = z;
}

__global__ void k_aos_pack(uint8_t *__restrict__ aos, AosLayout lay, int64_t n,
                           StaticArrays st, DynArrays dy,
                           const double *__restrict__ fc, int fc_orig,
                           double mob, int wrote_step, int any_fungi) {
  int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= n) return;
  int64_t o = st.oid[t];
  uint8_t *r = aos + o * (int64_t)lay.stride;
  double *pos = reinterpret_cast<double *>(r + lay.pos);
  double *rd = reinterpret_cast<double *>(r + lay.rdata);
  int32_t *id = reinterpret_cast<int32_t *>(r + lay.idata);
  double4 p = dy.pos[t];
  pos[0] = p.x;
  pos[1] = p.y;
  pos[2] = p.z;
  if (wrote_step) {
    const double *f = fc + (fc_orig ? o : t) * 6;
    rd[rec::velx] = mob * f[0];
    rd[rec::vely] = mob * f[1];
    rd[rec::velz] = mob * f[2];
    rd[rec::wx] = f[3];
    rd[rec::wy] = f[4];
    rd[rec::wz] = f[5];
    id[rec::fuse_flag] = 0;
    id[rec::split_flag] = 0;
    id[rec::new_flag] = 0;
  }
  if (any_fungi && st.type[t] == rec::FUNGI) {
    double4 rr = dy.rod[t];
    rd[rec::theta] = rr.y;
    rd[rec::phi] = rr.z;
    Topo tp = dy.topo[t];
    id[rec::n_bnds] = tp.n_bnds;
    for (int b = 0; b < 4; b++) {
      id[rec::seg1_id1 + b] = tp.seg_id[b];
      id[rec::seg1_id2 + b] = tp.seg_cpu[b];
      id[rec::site1 + b] = tp.site[b];
    }
    id[rec::position] = tp.position;
    id[rec::fix_site] = tp.fix_site;
    if (tp.dltd)
      for (int k = rec::dltd_site1; k <= rec::dltd_cpu2; k++) id[k] = -1;
  }
}

// inv[original index] = sorted position
__global__ void k_inverse(const int32_t *__restrict__ oid, int64_t n,
                          int32_t *__restrict__ inv) {
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t < n) inv[oid[t]] = (int32_t)t;
}

// What k_aos_pack and k_chem_pack write, in one pass in record order: a wave
// takes 64 consecutive records, gathers each one's values by its sorted
// position, lays them out in LDS and then stores them component by component,
// so that neighbouring lanes write neighbouring words of a record and the
// launch walks through memory once.  Bound by the records' memory: their
// 64-byte sectors are written in part, three of a sphere's seven (position,
// velocities, flags; the flags are read, and stored only where they are not
// zero yet: 99.6 us against 111 for storing them always).  1M spheres, with
// the inverse order: 112 us against 129 scattered from the sorted order, and
// 225 against 332 with the chemistry state.
struct PackWhat {
  int step;  // a step has run: velocities and flags
  int fc_orig;  // its fc is in original order
  int rel;   // CHEM: the layout holds the amounts taken from the fluid
};
template <bool FUNGI, bool CHEM>
struct PackShape {
  // pos 3, vel and w 6, FUNGI: theta, phi; CHEM: radius, (length,) area, vol,
  // gradient 3, rates 2, species 6, taken 3
  static constexpr int nd = 9 + (FUNGI ? 2 : 0) + (CHEM ? 17 + (FUNGI ? 1 : 0) : 0);
  static constexpr int ni = FUNGI ? 15 : 0;  // bonds 13, position, fix_site
  static constexpr size_t lds = kWave * (nd * sizeof(double) + ni * sizeof(int32_t));
};

template <bool FUNGI, bool CHEM>
__global__ __launch_bounds__(kWave) void k_aos_pack_wide(
    uint8_t *__restrict__ aos, AosLayout lay, int64_t n,
    const int32_t *__restrict__ inv, const int32_t *__restrict__ type,
    DynArrays dy, const double *__restrict__ fc,
    const double *__restrict__ state, double mob, PackWhat what) {
  using P = PackShape<FUNGI, CHEM>;
  constexpr int ND = P::nd, NI = P::ni;
  extern __shared__ __align__(16) unsigned char pack_lds[];
  double *val = reinterpret_cast<double *>(pack_lds);
  int32_t *iv = reinterpret_cast<int32_t *>(val + kWave * ND);
  const int lane = threadIdx.x;
  const int64_t o0 = (int64_t)blockIdx.x * kWave, o = o0 + lane;
  const int nrec = n - o0 < kWave ? (int)(n - o0) : kWave;
  const bool on = lane < nrec;
  bool fungi = false, reset = false;
  if (on) {
    const int64_t t = inv[o];
    const double4 p = dy.pos[t];
    double *v = val + lane * ND;
    int c = 0;
    v[c++] = p.x;
    v[c++] = p.y;
    v[c++] = p.z;
    double4 rr = make_double4(0.0, 0.0, 0.0, 0.0);
    if (FUNGI) {
      fungi = type[t] == rec::FUNGI;
      if (fungi) {
        rr = dy.rod[t];
        const Topo tp = dy.topo[t];
        int32_t *w = iv + lane * NI;
        w[0] = tp.n_bnds;
#pragma unroll
        for (int b = 0; b < 4; b++) {
          w[1 + b] = tp.seg_id[b];
          w[5 + b] = tp.seg_cpu[b];
          w[9 + b] = tp.site[b];
        }
        w[13] = tp.position;
        w[14] = tp.fix_site;
        reset = tp.dltd != 0;
      }
    }
    double4 a = rr, b = rr, d = rr, e = rr;
    if (CHEM) {
      const double4 *q = reinterpret_cast<const double4 *>(state + t * chem::stride);
      a = q[0];
      b = q[1];
      d = q[2];
      e = q[3];
      v[c++] = p.w;
      if (FUNGI) v[c++] = rr.x;
    }
    if (FUNGI) {
      v[c++] = rr.y;
      v[c++] = rr.z;
    }
    if (CHEM) {
      v[c++] = b.w;  // area
      v[c++] = a.w;  // vol
    }
    if (what.step) {
      const double *f = fc + (what.fc_orig ? o : t) * 6;
      v[c++] = mob * f[0];
      v[c++] = mob * f[1];
      v[c++] = mob * f[2];
      v[c++] = f[3];
      v[c++] = f[4];
      v[c++] = f[5];
    } else {
      c += 6;
    }
    if (CHEM) {
      v[c++] = d.z;  // gradient
      v[c++] = d.w;
      v[c++] = e.x;
      v[c++] = d.x;  // dadt, dvdt
      v[c++] = d.y;
      v[c++] = a.x;  // species and their increments
      v[c++] = a.y;
      v[c++] = a.z;
      v[c++] = b.x;
      v[c++] = b.y;
      v[c++] = b.z;
      v[c++] = e.y;  // taken from the fluid
      v[c++] = e.z;
      v[c++] = e.w;
    }
  }
  const unsigned long long segs = FUNGI ? __ballot(fungi) : 0ull;
  const unsigned long long dltd = FUNGI ? __ballot(reset) : 0ull;
  wave_lds_sync();
  // component c of a record: its real index (below 0: position 3 + index),
  // and whether only segments have it
  for (int i = lane; i < nrec * ND; i += kWave) {
    const int r = i / ND, c = i - r * ND;
    constexpr int c1 = 3, c2 = c1 + (CHEM ? (FUNGI ? 2 : 1) : 0),
                  c3 = c2 + (FUNGI ? 2 : 0), c4 = c3 + (CHEM ? 2 : 0), c5 = c4 + 6;
    int k;
    bool put = true, seg_only = false;
    if (c < c1) {
      k = c - 3;
    } else if (c < c2) {
      k = rec::radius + (c - c1);
      seg_only = c > c1;
    } else if (c < c3) {
      k = rec::theta + (c - c2);
      seg_only = true;
    } else if (c < c4) {
      k = rec::area + (c - c3);
    } else if (c < c5) {
      k = rec::velx + (c - c4);
      put = what.step != 0;
    } else if (c < c5 + 5) {
      k = rec::gx + (c - c5);
    } else {
      k = rec::first_data + (c - c5 - 5);
      put = what.rel || c < c5 + 11;
    }
    if (seg_only) put = (segs >> r) & 1ull;
    if (put) {
      uint8_t *q = aos + (o0 + r) * (int64_t)lay.stride +
                   (k < 0 ? lay.pos + 8 * (k + 3) : lay.rdata + 8 * k);
      *reinterpret_cast<double *>(q) = val[i];
    }
  }
  if (FUNGI) {
    // n_bnds .. position, then dltd_site1 .. dltd_cpu2 of reset segments and
    // fix_site
    constexpr int nb = rec::position - rec::n_bnds + 1;
    constexpr int NW = nb + rec::fix_site - rec::dltd_site1 + 1;
    for (int i = lane; i < nrec * NW; i += kWave) {
      const int r = i / NW, c = i - r * NW;
      const bool table = c < nb, site = c == NW - 1;
      if (((table || site ? segs : dltd) >> r) & 1ull)
        reinterpret_cast<int32_t *>(aos + (o0 + r) * (int64_t)lay.stride +
                                    lay.idata)[table ? rec::n_bnds + c : rec::dltd_site1 + (c - nb)] =
            table ? iv[r * NI + c] : (site ? iv[r * NI + nb] : -1);
    }
  }
  if (what.step) {
    for (int i = lane; i < 3 * nrec; i += kWave) {
      const int r = i / 3;
      int32_t *q = reinterpret_cast<int32_t *>(aos + (o0 + r) * (int64_t)lay.stride +
                                               lay.idata) + rec::fuse_flag + (i - 3 * r);
      if (*q) *q = 0;
    }
  }
}

// ------------------------------------------------------------- binning ---

// blocks of the bin count that take part in a folded displacement check
constexpr int kSkinBlocks = 64;
constexpr int kSkinGroup = 16;  // slots reduced together
template <bool MULTI>
__global__ void k_bin_count(const double4 *__restrict__ pos,
                            const int32_t *__restrict__ col,
                            const BoxGeom *__restrict__ boxes, BoxGeom g0,
                            int64_t n, int32_t *__restrict__ key,
                            int32_t *__restrict__ rank,
                            int32_t *__restrict__ count, SkinCheck sk) {
  // The input is in the order of the previous rebuild, so neighboring lanes
  // mostly share a bin: each run of equal bins in the wave takes its slots
  // with one atomic (the head's) and numbers its lanes from there.  Only the
  // slot set of a bin matters: the bins are sorted by original index next.
  const int64_t s = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const bool active = s < n;
  int b = -1;
  if (active) {
    const BoxGeom &g = MULTI ? boxes[col[s]] : g0;
    b = bin_of(pos[s], g);
    key[s] = b;
  }
  const int lane = threadIdx.x & (kWave - 1);
  const int prev = __shfl_up(b, 1, kWave);
  const bool head = active && (lane == 0 || prev != b);
  const unsigned long long heads = __ballot(head);
  const unsigned long long act = __ballot(active);
  // run of this lane: from the last head at or below it to the next head
  const unsigned long long below = heads & ((2ull << lane) - 1ull);
  const int first = 63 - __builtin_clzll(below | 1ull);
  const unsigned long long above = heads & ~((2ull << lane) - 1ull);
  const int stop = above ? __builtin_ctzll(above) : 64 - __builtin_clzll(act);
  int base = 0;
  if (head) base = atomicAdd(&count[b], stop - lane);
  base = __shfl(base, first, kWave);
  if (active) rank[s] = base + (lane - first);
  // the first kSkinBlocks blocks also reduce the displacement partials of
  // the period this rebuild ends, one share of every slot each, and clear
  // them (block-uniform branch: the block reductions synchronise).  Up to
  // kSkinGroup slots at a time: every load of the group is issued before
  // any reduction, and the group's block maxima share one barrier.
  const int nsb = gridDim.x < kSkinBlocks ? (int)gridDim.x : kSkinBlocks;
  if (sk.vpart && (int)blockIdx.x < nsb) {
    // blocks of 256 (launch_bin_count): four waves
    __shared__ double shd[kSkinGroup][256 / kWave];
    const int64_t chunk = (sk.stride + nsb - 1) / nsb;
    const int64_t c0 = blockIdx.x * chunk;
    const int64_t c1 = c0 + chunk < sk.stride ? c0 + chunk : sk.stride;
    const int wid = threadIdx.x / kWave;
    for (int g = 0; g < sk.nslots; g += kSkinGroup) {
      double m[kSkinGroup];
#pragma unroll
      for (int j = 0; j < kSkinGroup; j++) m[j] = 0.0;
      for (int64_t i = c0 + threadIdx.x; i < c1; i += blockDim.x) {
#pragma unroll
        for (int j = 0; j < kSkinGroup; j++) {
          if (g + j < sk.nslots) {
            double *v = sk.vpart + (int64_t)(g + j) * sk.stride + i;
            const double x = *v;
            m[j] = x > m[j] ? x : m[j];
            *v = 0.0;
          }
        }
      }
#pragma unroll
      for (int j = 0; j < kSkinGroup; j++) {
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) {
          const double w = __shfl_xor(m[j], o, kWave);
          m[j] = w > m[j] ? w : m[j];
        }
        if (lane == 0) shd[j][wid] = m[j];
      }
      __syncthreads();
      const int j = threadIdx.x;
      if (j < kSkinGroup && g + j < sk.nslots) {
        double mm = shd[j][0];
        for (int w = 1; w < (int)(blockDim.x / kWave); w++)
          mm = shd[j][w] > mm ? shd[j][w] : mm;
        if (mm > 0.0) atomicMax(&sk.slotmax[g + j], dbits(mm));
      }
      __syncthreads();
    }
  }
}

// Exclusive scan: 256 threads x 8 items per block, wave prefix by shuffles.
constexpr int kScanThreads = 256;
constexpr int kScanItems = 8;
static_assert(kScanItems == 8, "k_scan_local moves a thread's counts as two int4");
constexpr int kScanTile = kScanThreads * kScanItems;

template <typename T>
__device__ __forceinline__ T block_excl_scan(T s, T *wsum, T &total) {
  int lane = threadIdx.x & (kWave - 1), wid = threadIdx.x / kWave;
  T incl = s;
#pragma unroll
  for (int o = 1; o < kWave; o <<= 1) {
    T y = __shfl_up(incl, o, kWave);
    if (lane >= o) incl += y;
  }
  if (lane == kWave - 1) wsum[wid] = incl;
  __syncthreads();
  T pre = 0, tot = 0;
  int nw = blockDim.x / kWave;
  for (int w = 0; w < nw; w++) {
    if (w < wid) pre += wsum[w];
    tot += wsum[w];
  }
  total = tot;
  return pre + incl - s;
}

// The counts are consumed here: each is reset to zero once read, which
// leaves the count array cleared for the next binning.
__global__ __launch_bounds__(kScanThreads) void k_scan_local(
    int32_t *__restrict__ in, int32_t *__restrict__ out,
    int32_t *__restrict__ bsum, int64_t n, SkinCheck sk) {
  __shared__ int32_t wsum[kScanThreads / kWave];
  if (sk.vpart && blockIdx.x == 0 && threadIdx.x == 0) {
    // the folded displacement check: the slot maxima the bin count left,
    // summed in slot order (as k_skin_final)
    double total = 0.0;
    for (int sl = 0; sl < sk.nslots; sl++) {
      total += __longlong_as_double((long long)sk.slotmax[sl]);
      sk.slotmax[sl] = 0ull;
    }
    if (total > sk.limit) atomicOr(sk.err, ERRBIT_SKIN);
  }
  int64_t base = (int64_t)blockIdx.x * kScanTile + threadIdx.x * kScanItems;
  // a thread's 8 counts are 32 aligned bytes (the arrays are allocation
  // bases): two 16-byte loads and stores, element by element at the tail
  const bool whole = base + kScanItems <= n;
  int32_t x[kScanItems];
  if (whole) {
    int4 *vin = reinterpret_cast<int4 *>(in + base);
    const int4 a = vin[0], b = vin[1];
    x[0] = a.x; x[1] = a.y; x[2] = a.z; x[3] = a.w;
    x[4] = b.x; x[5] = b.y; x[6] = b.z; x[7] = b.w;
    vin[0] = make_int4(0, 0, 0, 0);
    vin[1] = make_int4(0, 0, 0, 0);
  } else {
#pragma unroll
    for (int i = 0; i < kScanItems; i++) {
      x[i] = 0;
      if (base + i < n) {
        x[i] = in[base + i];
        in[base + i] = 0;
      }
    }
  }
  int32_t v[kScanItems];
  int32_t s = 0;
#pragma unroll
  for (int i = 0; i < kScanItems; i++) {
    v[i] = s;
    s += x[i];
  }
  int32_t total;
  int32_t ex = block_excl_scan(s, wsum, total);
  if (whole) {
    int4 *vout = reinterpret_cast<int4 *>(out + base);
    vout[0] = make_int4(v[0] + ex, v[1] + ex, v[2] + ex, v[3] + ex);
    vout[1] = make_int4(v[4] + ex, v[5] + ex, v[6] + ex, v[7] + ex);
  } else {
#pragma unroll
    for (int i = 0; i < kScanItems; i++)
      if (base + i < n) out[base + i] = v[i] + ex;
  }
  if (threadIdx.x == 0) bsum[blockIdx.x] = total;
}

// Adds each tile's offset, the sum of the tile sums before it, which every
// block forms itself from the (L2-resident) tile sums, so no separate pass
// scans them; the last block also writes the grand total to out[n].
__global__ __launch_bounds__(kScanThreads) void k_scan_add(
    int32_t *__restrict__ out, const int32_t *__restrict__ bsum, int64_t nt,
    int64_t n) {
  __shared__ int32_t wsum[kScanThreads / kWave];
  int32_t part = 0;
  for (int64_t i = threadIdx.x; i < (int64_t)blockIdx.x; i += kScanThreads)
    part += bsum[i];
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) part += __shfl_xor(part, o, kWave);
  if ((threadIdx.x & (kWave - 1)) == 0) wsum[threadIdx.x / kWave] = part;
  __syncthreads();
  int32_t add = 0;
#pragma unroll
  for (int w = 0; w < kScanThreads / kWave; w++) add += wsum[w];
  if (threadIdx.x == 0 && (int64_t)blockIdx.x == nt - 1) out[n] = add + bsum[blockIdx.x];
  const int64_t base = (int64_t)blockIdx.x * kScanTile + threadIdx.x * kScanItems;
  if (base + kScanItems <= n) {  // 32 aligned bytes, as in k_scan_local
    int4 *v = reinterpret_cast<int4 *>(out + base);
    int4 a = v[0], b = v[1];
    a.x += add; a.y += add; a.z += add; a.w += add;
    b.x += add; b.y += add; b.z += add; b.w += add;
    v[0] = a;
    v[1] = b;
  } else {
    for (int i = 0; i < kScanItems; i++)
      if (base + i < n) out[base + i] += add;
  }
}

__global__ void k_bin_scatter(const int32_t *__restrict__ key,
                              const int32_t *__restrict__ rank,
                              const int32_t *__restrict__ start,
                              const int32_t *__restrict__ oid, int64_t n,
                              unsigned long long *__restrict__ permk) {
  int64_t s = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (s >= n) return;
  int64_t dst = (int64_t)start[key[s]] + rank[s];
  permk[dst] = ((unsigned long long)(uint32_t)oid[s] << 32) |
               (unsigned long long)(uint32_t)s;
}

// Orders each bin by original index and gathers the per-particle arrays
// into that order in one pass.  Thread j takes slot j of the scattered
// (bin-grouped, not yet ordered) entries (original index << 32 | old
// position): its place in its bin is the number of the bin's entries below
// it (the original indexes are distinct), and it copies its particle from
// the old position to that place.  A bin of more than kMaxBinSort
// particles is left in scatter order and reported as an overflow (its rows
// could not fit anyway), which bounds the work of every thread; after a
// non-finite force nothing is ordered.
constexpr int64_t kMaxBinSort = 1024;
__global__ void k_sort_gather(const unsigned long long *__restrict__ permk,
                              const int32_t *__restrict__ start, int64_t n,
                              StaticArrays ss, StaticArrays ds, DynArrays sd,
                              DynArrays dd, const int32_t *__restrict__ key,
                              int multi, int rods, int32_t *__restrict__ err,
                              const double *__restrict__ chem_src,
                              double *__restrict__ chem_dst) {
  const int64_t jt = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const bool on = jt < n;
  if (!on && !chem_src) return;
  const int64_t j = on ? jt : n - 1;  // (idle lanes help with the lines below)
  const unsigned long long e = permk[j];
  const int64_t s = (int64_t)(uint32_t)(e & 0xffffffffull);
  const int32_t b = key[s];
  const int64_t a = start[b], z = start[b + 1];
  int64_t t = j;
  if (z - a > kMaxBinSort) {
    if (on && j == a) atomicOr(err, ERRBIT_OVERFLOW);
  } else if (!(*err & ERRBIT_NAN)) {
    t = a;
    for (int64_t i = a; i < z; i++) t += permk[i] < e;
  }
  // native vectors: double4's members and whole copies together keep it in
  // memory (LDS)
  typedef double double4v __attribute__((ext_vector_type(4)));
  typedef int int4v __attribute__((ext_vector_type(4)));
  if (on) {
    const double4v p = reinterpret_cast<const double4v *>(sd.pos)[s];
    const int32_t ty = ss.type[s];
    reinterpret_cast<double4v *>(dd.pos)[t] = p;
    ds.oid[t] = ss.oid[s];
    ds.type[t] = ty;
    ds.key[t] = b;
    if (multi) ds.col[t] = ss.col[s];
    if (rods) {
      ds.bscale[t] = ss.bscale[s];
      const double4v rr = reinterpret_cast<const double4v *>(sd.rod)[s];
      const double4v tr = reinterpret_cast<const double4v *>(sd.trig)[s];
      reinterpret_cast<double4v *>(dd.rod)[t] = rr;
      reinterpret_cast<double4v *>(dd.trig)[t] = tr;
      const int4v *a = reinterpret_cast<const int4v *>(sd.topo + s);
      int4v *b = reinterpret_cast<int4v *>(dd.topo + t);
      const int4v x0 = a[0], x1 = a[1], x2 = a[2], x3 = a[3], x4 = a[4];
      b[0] = x0;
      b[1] = x1;
      b[2] = x2;
      b[3] = x3;
      b[4] = x4;
      // n_bnds, seg_id[4], seg_cpu[4], ..., self_id and self_cpu at 16 and 17
      dd.near[t] = near_of(p[0], p[1], p[2], p[3], ty, rr[0], tr[0], tr[1], tr[2], tr[3],
                           x0[0], x0[1], x0[2], x0[3], x1[0], x1[1], x1[2], x1[3], x2[0],
                           x4[0], x4[1]);
    }
  }
  if (chem_src) {
    // the chemistry state's 128-byte lines, 8 lanes to a line: 1M spheres
    // 59 us with the rest of the kernel, 98 with one lane copying a line
    const int lane = threadIdx.x & (kWave - 1), part = lane & 7;
    const int si = (int)s, ti = (int)t;
    int4v v[8];
#pragma unroll
    for (int k = 0; k < 8; k++) {
      const int from = __shfl(si, 8 * k + (lane >> 3), kWave);
      v[k] = reinterpret_cast<const int4v *>(chem_src + (int64_t)from * chem::stride)[part];
    }
#pragma unroll
    for (int k = 0; k < 8; k++) {
      const int to = __shfl(ti, 8 * k + (lane >> 3), kWave);
      const bool live = __shfl(on ? 1 : 0, 8 * k + (lane >> 3), kWave);
      if (live)
        reinterpret_cast<int4v *>(chem_dst + (int64_t)to * chem::stride)[part] = v[k];
    }
  }
}

// -------------------------------------------------------- neighbor rows ---

// Interaction reach of a particle: r_lm = reach_i + reach_j + W_A for equal
// cell types (K.H:23-40).
template <bool RODS>
__device__ __forceinline__ double reach_of(const double4 &p, int ty,
                                           const double4 *rod, int64_t u) {
  if (RODS && ty == rec::FUNGI) return 1.5 * rod[u].x;
  return p.w;
}

// Separation along axis A: the periodic image test of sep_axis when bit A of
// M is set, the plain difference otherwise (used only where no image can be
// involved on that axis, which gives the same bits).
template <int M, int A>
__device__ __forceinline__ double sep_m(double xi, double xj, const BoxGeom &g) {
  if (M & (1 << A)) return sep_axis(xi, xj, g.L[A], g.halfL[A], g.periodic[A]);
  return xi - xj;
}

// A particle's bin stencil as memory ranges of the sorted arrays, in the
// canonical order (oz, then oy, then ox).  Each (oz, oy) row of bins is one
// or two ranges: the x window [bx - 1, bx + 1] is contiguous in memory
// (bins are x-fastest) unless it wraps a periodic x face, where it splits
// into the bins before the face and the bins after it (piece 0 holds the
// bins of ox = -1 first).  Rows outside a non-periodic box are empty.
// Everything that does not change from range to range is formed once per
// particle, with the row offsets already multiplied out, so that moving to
// the next range costs a few full-rate selects and adds and the two loads
// of its bounds (no integer multiply, which runs at a quarter of the rate).
struct Stencil {
  // bin id of the first bin of z row cz (base + cz * nby * nbx) for
  // oz = -1, 0, 1, and cy * nbx for oy = -1, 0, 1; -1 outside the box
  // (named fields, not arrays: a select between array elements becomes an
  // indexed scratch access)
  int z0, z1, z2, y0, y1, y2;
  int xa0, xb0, xa1, xb1;  // x pieces [xa, xb) of every row
  int two;                 // 1 when a row has two pieces
};

__device__ __forceinline__ Stencil make_stencil(int bx, int by, int bz,
                                                const BoxGeom &g) {
  Stencil st;
  const int nbx = g.nbin[0], nby = g.nbin[1], nbz = g.nbin[2];
  auto zrow = [&](int cz) {
    if (g.periodic[2]) cz = cz < 0 ? cz + nbz : (cz >= nbz ? cz - nbz : cz);
    return (cz >= 0 && cz < nbz) ? g.bin_offset + cz * nby * nbx : -1;
  };
  auto ycol = [&](int cy) {
    if (g.periodic[1]) cy = cy < 0 ? cy + nby : (cy >= nby ? cy - nby : cy);
    return (cy >= 0 && cy < nby) ? cy * nbx : -1;
  };
  st.z0 = zrow(bz - 1);
  st.z1 = zrow(bz);
  st.z2 = zrow(bz + 1);
  st.y0 = ycol(by - 1);
  st.y1 = ycol(by);
  st.y2 = ycol(by + 1);
  const int lo = bx - 1, hi = bx + 2;  // [lo, hi) before any wrap
  st.xa1 = st.xb1 = 0;
  if (lo < 0) {
    if (g.periodic[0]) {
      st.xa0 = nbx - 1;
      st.xb0 = nbx;
      st.xb1 = hi < nbx ? hi : nbx;
    } else {
      st.xa0 = 0;
      st.xb0 = hi < nbx ? hi : nbx;
    }
  } else if (hi > nbx) {
    st.xa0 = lo;
    st.xb0 = nbx;
    if (g.periodic[0]) st.xb1 = hi - nbx;
  } else {
    st.xa0 = lo;
    st.xb0 = hi;
  }
  st.two = st.xb1 > st.xa1;
  return st;
}

// Memory range of range k of the stencil (k < 9 << two): row r = k >> two
// (oz = r / 3, oy = r % 3), piece k & two.  Fields are read into locals
// before they are selected, so that the selects are between values.
__device__ __forceinline__ int2 stencil_range(const Stencil st, int k,
                                              const int32_t *__restrict__ start) {
  const int z0 = st.z0, z1 = st.z1, z2 = st.z2;
  const int y0 = st.y0, y1 = st.y1, y2 = st.y2;
  const int r = k >> st.two, piece = k & st.two;
  // r / 3 as 11 r / 32 (exact for r < 9), with 24-bit multiplies, which
  // run at the full rate
  const int iz = (int)(__umul24((unsigned)r, 11u) >> 5);
  const int iy = r - (int)__umul24((unsigned)iz, 3u);
  const int zz = iz == 0 ? z0 : (iz == 1 ? z1 : z2);
  const int yy = iy == 0 ? y0 : (iy == 1 ? y1 : y2);
  if ((zz | yy) < 0) return make_int2(0, 0);
  const int xa0 = st.xa0, xa1 = st.xa1, xb0 = st.xb0, xb1 = st.xb1;
  const int row = zz + yy;
  const int xa = piece ? xa1 : xa0, xb = piece ? xb1 : xb0;
  return make_int2(start[row + xa], start[row + xb]);
}

// Bits 28..30 of a row count mark the axes (x, y, z) along which a neighbor
// of the particle can need a periodic image before the next rebuild: the
// axis is periodic and the particle's bin is within two bins of a face (or
// the box has fewer than six bins along it).  Force kernels test images
// only along the axes marked somewhere in the wave.
constexpr int kImgShift = 28;
constexpr int32_t kRowMask = (1 << kImgShift) - 1;
__device__ __forceinline__ int row_len(int32_t raw) { return raw & kRowMask; }
__device__ __forceinline__ int row_img(int32_t raw) { return (raw >> kImgShift) & 7; }

// OR of a 3-bit axis mask over the wave.
__device__ __forceinline__ int wave_or3(int m) {
  return (__any(m & 1) ? 1 : 0) | (__any(m & 2) ? 2 : 0) | (__any(m & 4) ? 4 : 0);
}


// Axes (bits) along which a candidate of a list build over the +-1 stencil of
// bin b3 (scan) or a neighbor before the next rebuild (force) can need a
// periodic image.
__device__ __forceinline__ void image_axes(const int b3[3], const BoxGeom &g,
                                           int &scan_img, int &force_img) {
#pragma unroll
  for (int a = 0; a < 3; a++) {
    if (!g.periodic[a]) continue;
    const int nb = g.nbin[a];
    if (!(nb >= 4 && b3[a] >= 1 && b3[a] + 1 < nb)) scan_img |= 1 << a;
    if (!(nb >= 6 && b3[a] >= 2 && b3[a] + 2 < nb)) force_img |= 1 << a;
  }
}

// One block builds the rows of one tile (blockDim.x / G particles), G lanes
// to a particle.  The lanes of a group load the bounds of the particle's 9
// (18 next to a periodic x face) stencil ranges at once, leave their running
// ends in LDS, and then test candidates k = sub, sub + G, ... of the
// concatenated ranges, kBuildUnroll of them in flight; a ballot gives the
// accepted ones their places, which keeps the rows in candidate order.
// Entries past the staged ones pass through global memory (nbr).
constexpr int kBuildRanges = 18;
constexpr int kBuildUnroll = 2;
__host__ __device__ constexpr int build_stage(int tile) {
  return tile >= 64 ? 9 : (tile >= 32 ? 17 : 33);
}
size_t build_lds(int tile) {
  return (size_t)tile * (sizeof(int2) * kBuildRanges +
                         sizeof(int32_t) * build_stage(tile));
}

template <bool MULTI, bool RODS, int G>
__global__ __launch_bounds__(256, 8) void k_build_rows(
    const double4 *__restrict__ pos, const int32_t *__restrict__ col,
    const int32_t *__restrict__ type, const double4 *__restrict__ rod,
    const BoxGeom *__restrict__ boxes, BoxGeom g0,
    const int32_t *__restrict__ start, const int32_t *__restrict__ key,
    int64_t n, int mode, double crit, double wa, double skin,
    int32_t *__restrict__ nbr, int32_t *__restrict__ ncnt, int64_t ncap,
    int32_t maxn, int32_t *__restrict__ err, int32_t *__restrict__ bstats,
    FlatRows flat, int remap) {
  extern __shared__ __align__(8) int32_t build_words[];
  const int lane = threadIdx.x & (kWave - 1), wv = threadIdx.x / kWave;
  const int nwv = blockDim.x / kWave, T = flat.tile;  // T = blockDim.x / G
  const int place = threadIdx.x / G, sub = threadIdx.x & (G - 1);
  const int S = build_stage(T);
  int2 *rng = reinterpret_cast<int2 *>(build_words) + place * kBuildRanges;
  int32_t *stage = build_words + 2 * kBuildRanges * T + place * S;
  const int64_t tile = tile_of(remap);
  const int64_t t = tile * T + place;
  const double was = wa + skin;
  // Candidates visited per particle are capped (a pile of particles in a few
  // bins would otherwise make this quadratic): a range that would pass the
  // cap is dropped with every later one, and the row reported as an
  // overflow.  After a non-finite force no rows are built.
  const int64_t scan_cap = 64 * (int64_t)maxn + 4096;
  const int cap = scan_cap < (1 << 30) ? (int)scan_cap : (1 << 30);
  const bool active = t < n && !(*err & ERRBIT_NAN);
  const int64_t tc = t < n ? t : n - 1;
  const unsigned long long gmask = ((1ull << G) - 1ull) << (lane & ~(G - 1));
  const unsigned long long below = (1ull << lane) - 1ull;
  int cnt = 0;
  // The row build over box g.  Several boxes: a wave whose particles all
  // lie in one box (all but the waves at colony boundaries) reads that box
  // once into scalar registers; the others read each particle's box.
  auto build = [&](const BoxGeom &g) {
    const double4 p = pos[tc];
    const double reach_i = RODS ? reach_of<true>(p, type[tc], rod, tc) : p.w;
    const int nbx = g.nbin[0], nby = g.nbin[1];
    const int lb = key[tc] - g.bin_offset;
    const int rr = lb / nbx;
    const int b3[3] = {lb % nbx, rr % nby, rr / nby};
    int scan_img = 0, force_img = 0;
    image_axes(b3, g, scan_img, force_img);
    const Stencil sc = make_stencil(b3[0], b3[1], b3[2], g);
    const int nq = active ? 9 << sc.two : 0;
    // the ranges' bounds, then rng[r] = (running end, first - begin)
    int total = 0;
    bool over = false;
    auto bounds = [&](auto nb_tag) {
      constexpr int NB = decltype(nb_tag)::value;
      int2 se[NB];
#pragma unroll
      for (int b = 0; b < NB; b++) {
        const int r = b * G + sub;
        se[b] = r < nq ? stencil_range(sc, r, start) : make_int2(0, 0);
      }
      int run = 0;
#pragma unroll
      for (int b = 0; b < NB; b++) {
        const int r = b * G + sub;
        const int len = se[b].y - se[b].x;
        int incl = len;
#pragma unroll
        for (int o = 1; o < G; o <<= 1) {
          const int w = __shfl_up(incl, o, G);
          if (sub >= o) incl += w;
        }
        const int end = run + incl;
        if (r < nq) {
          rng[r] = make_int2(end, se[b].x - (end - len));
          if (end <= cap) total = end;
        }
        run += __shfl(incl, G - 1, G);
      }
      over = run > cap;
    };
    if (__any(nq > 9))
      bounds(std::integral_constant<int, (18 + G - 1) / G>{});
    else
      bounds(std::integral_constant<int, (9 + G - 1) / G>{});
#pragma unroll
    for (int o = G >> 1; o > 0; o >>= 1) {
      const int w = __shfl_xor(total, o, G);
      total = w > total ? w : total;
    }
    wave_lds_sync();
    auto scan = [&](auto m_tag, auto crit_tag) {
      constexpr int M = decltype(m_tag)::value;
      constexpr bool CRIT = decltype(crit_tag)::value;
      int r = 0;
      int2 cur = rng[0];
      for (int k0 = sub; __any(k0 < total); k0 += kBuildUnroll * G) {
        int u[kBuildUnroll];
        bool ok[kBuildUnroll];
        double4 o[kBuildUnroll];
        double rj[kBuildUnroll];
#pragma unroll
        for (int j = 0; j < kBuildUnroll; j++) {
          const int k = k0 + j * G;
          ok[j] = k < total;
          while (ok[j] && k >= cur.x) cur = rng[++r];
          u[j] = ok[j] ? k + cur.y : (int)tc;
          o[j] = pos[u[j]];
          if (!CRIT) rj[j] = RODS ? reach_of<true>(o[j], type[u[j]], rod, u[j]) : o[j].w;
        }
#pragma unroll
        for (int j = 0; j < kBuildUnroll; j++) {
          const double d0 = sep_m<M, 0>(p.x, o[j].x, g);
          const double d1 = sep_m<M, 1>(p.y, o[j].y, g);
          const double d2 = sep_m<M, 2>(p.z, o[j].z, g);
          const double r2 = d0 * d0 + d1 * d1 + d2 * d2;
          bool in;
          if (CRIT) {
            in = r2 <= crit;  // BMXCheckPair (src/des/bmx_pc.H:76)
          } else {
            const double cut = reach_i + rj[j] + was;
            in = r2 <= cut * cut;
          }
          in = in && ok[j] && u[j] != (int)t;
          const unsigned long long m = __ballot(in) & gmask;
          const int k = cnt + __popcll(m & below);
          if (in && k < maxn) {
            if (k < S)
              stage[k] = u[j];
            else
              nbr[tc + (int64_t)k * ncap] = u[j];
          }
          cnt += __popcll(m);
        }
      }
    };
    const bool img = wave_or3(active ? scan_img : 0) != 0;
    auto run = [&](auto crit_tag) {
      if (img)
        scan(std::integral_constant<int, 7>{}, crit_tag);
      else
        scan(std::integral_constant<int, 0>{}, crit_tag);
    };
    if (mode == 1)
      run(std::true_type{});
    else
      run(std::false_type{});
    if (over && cnt <= maxn) cnt = maxn + 1;  // reported as an overflow
    if (sub == 0 && t < n) {
      ncnt[t] = active ? (cnt < maxn ? cnt : maxn) | (force_img << kImgShift) : 0;
      if (cnt > maxn) atomicOr(err, ERRBIT_OVERFLOW);
    }
  };
  if (MULTI) {
    const int32_t cl = col[tc];
    const int cw = __builtin_amdgcn_readfirstlane(cl);
    if (__all(t >= n || cl == cw)) {
      const BoxGeom gw = boxes[cw];
      build(gw);
    } else {
      build(boxes[cl]);
    }
  } else {
    build(g0);
  }
  // the rows back to back: offsets over the tile's particles, wave totals
  // through LDS, with the row statistics
  __shared__ int32_t wsum[256 / kWave], wmax[256 / kWave], wall[256 / kWave];
  const int kept = cnt < maxn ? cnt : maxn;
  int incl = wave_incl_scan64(sub == 0 ? kept : 0);
  int all = incl;
  if (__any(cnt > kept)) all = wave_incl_scan64(sub == 0 ? cnt : 0);
  int mx = cnt;
#pragma unroll
  for (int o = kWave / 2; o >= G; o >>= 1) {
    const int w = __shfl_xor(mx, o, kWave);
    mx = w > mx ? w : mx;
  }
  if (lane == kWave - 1) {
    wsum[wv] = incl;
    wmax[wv] = mx;
    wall[wv] = all;
  }
  // (also orders the staged entries, and those in global memory, before
  // other lanes read them)
  __syncthreads();
  for (int w = 0; w < wv; w++) incl += wsum[w];
  if (threadIdx.x == 0) {
    int tot = wsum[0], m = wmax[0], a = wall[0];
    for (int w = 1; w < nwv; w++) {
      tot += wsum[w];
      m = wmax[w] > m ? wmax[w] : m;
      a += wall[w];
    }
    flat.tot[tile] = tot;
    bstats[2 * blockIdx.x] = m;
    bstats[2 * blockIdx.x + 1] = a;
  }
  if (sub == 0 && t < n) flat.roff[t] = incl - kept;
  const int64_t b = tile * (int64_t)T * maxn + (incl - kept);
  for (int k = sub; k < kept; k += G) {
    flat.cidx[b + k] = k < S ? stage[k] : nbr[tc + (int64_t)k * ncap];
    flat.cown[b + k] = (uint8_t)place;
  }
}

// ------------------------------------------------------- force + update ---

// Separation of two spheres along the axes, with the image test of sep_m.
template <int M>
__device__ __forceinline__ void sphere_sep(const double4 &p, const double4 &o,
                                           const BoxGeom &g, double &d0,
                                           double &d1, double &d2) {
  d0 = sep_m<M, 0>(p.x, o.x, g);
  d1 = sep_m<M, 1>(p.y, o.y, g);
  d2 = sep_m<M, 2>(p.z, o.z, g);
}

// ------------------------------------------------- flat sphere force ---
//
// The sphere step (force lambda PCI:170-279 with the sphere law K.H:243-276
// and the wall K.H:1009-1030, then the update PCI:311-449) over the flat row
// layout, one tile (64 particles or fewer, see flat_tile) per wave; lanes
// below the tile size own a particle.  Lane l takes list entries l and l + 64
// of each window of 128: it loads the neighbor index and its owner lane, gathers the
// neighbor, reads the owner's position from LDS and applies the interaction
// test (K.H:23-40 with PCI:212).  Interacting pairs are packed into LDS
// slots by ballot, entry 0 of every lane first, so slot order is entry
// order; the cubic law then runs once per 64 packed pairs and leaves each
// term in its slot.  An owner's interacting entries occupy a contiguous run
// of slots, which it adds in row order: every particle sums its pair terms
// in its row's order, as a loop over the row would.
constexpr int kFlatWin = 2 * kWave;
constexpr size_t kFlatWaveBytes =
    kWave * sizeof(double4) + 4 * kFlatWin * sizeof(double);

// Largest step displacement dt*|vel| of the wave, one store per wave at its
// tile's index (the partial arrays hold one entry per tile), with no block
// barrier: waves that finish early do not wait for the block's slowest.  (One atomic maximum per wave into a few shared words instead
// measured 2.4 times slower on the 1M-sphere step: the atomics serialize.)
__device__ __forceinline__ void wave_vmax(double v2, double dt, double *vpart,
                                          int64_t tile, int lane, bool live) {
  const double m = wave_max_f64(v2);
  if (lane == 0 && live) vpart[tile] = dt * sqrt(m);
}



template <bool MULTI, int M>
__device__ __forceinline__ void flat_rows(
    int T, int P, int c, int64_t B, int lane, int f0u, int f1u, int f0o, int f1o,
    const int32_t *__restrict__ cidx, const uint8_t *__restrict__ cown,
    const double4 *__restrict__ pos_in, const double4 *sp, const int32_t *scol,
    double *q0s, double *q1s, double *q2s, double *qrs,
    const BoxGeom *__restrict__ boxes, const BoxGeom &g0, const ForceParams &fp,
    double &a0, double &a1, double &a2) {
  const unsigned long long below = (1ull << lane) - 1ull;
  // f0u, f1u, f0o, f1o: with one box, the first window's entries, loaded
  // by the caller (entries past the count are masked below)
  for (int w0 = 0; w0 < T; w0 += kFlatWin) {
    const int e0 = w0 + lane, e1 = e0 + kWave;
    const bool v0 = e0 < T, v1 = e1 < T;
    int u0 = 0, u1 = 0, o0 = 0, o1 = 0;
    if (!MULTI && w0 == 0) {
      u0 = v0 ? f0u : 0;
      u1 = v1 ? f1u : 0;
      o0 = v0 ? f0o : 0;
      o1 = v1 ? f1o : 0;
    } else {
      if (v0) {
        u0 = cidx[B + e0];
        o0 = cown[B + e0];
      }
      if (v1) {
        u1 = cidx[B + e1];
        o1 = cown[B + e1];
      }
    }
    const double4 q0 = pos_in[u0], q1 = pos_in[u1];
    const double4 p0 = sp[o0], p1 = sp[o1];
    const BoxGeom &ga = MULTI ? boxes[scol[o0]] : g0;
    const BoxGeom &gb = MULTI ? boxes[scol[o1]] : g0;
    double x0, y0, z0, x1, y1, z1;
    sphere_sep<M>(p0, q0, ga, x0, y0, z0);
    sphere_sep<M>(p1, q1, gb, x1, y1, z1);
    const double r20 = x0 * x0 + y0 * y0 + z0 * z0;
    const double r21 = x1 * x1 + y1 * y1 + z1 * z1;
    const double lim0 = p0.w + q0.w + fp.WA - 1.0e-15;  // r_lm - small_number
    const double lim1 = p1.w + q1.w + fp.WA - 1.0e-15;
    const bool i0 = v0 && r20 <= lim0 * lim0;
    const bool i1 = v1 && r21 <= lim1 * lim1;
    const unsigned long long b0 = __ballot(i0), b1 = __ballot(i1);
    const int n0 = __popcll(b0), ni = n0 + __popcll(b1);
    if (i0) {
      const int k = __popcll(b0 & below);
      q0s[k] = x0;
      q1s[k] = y0;
      q2s[k] = z0;
      qrs[k] = p0.w + q0.w;
    }
    if (i1) {
      const int k = n0 + __popcll(b1 & below);
      q0s[k] = x1;
      q1s[k] = y1;
      q2s[k] = z1;
      qrs[k] = p1.w + q1.w;
    }
    wave_lds_sync();
    for (int k = lane; k < ni; k += kWave) {  // the cubic law, packed
      const double d0 = q0s[k], d1 = q1s[k], d2 = q2s[k];
      const double r2 = d0 * d0 + d1 * d1 + d2 * d2;
      double fx = 0.0, fy = 0.0, fz = 0.0;
      sphere_pair(d0, d1, d2, r2, qrs[k], fp, fx, fy, fz);
      q0s[k] = fx;
      q1s[k] = fy;
      q2s[k] = fz;
    }
    wave_lds_sync();
    const int lo = P > w0 ? P : w0;
    const int hi = P + c < w0 + kFlatWin ? P + c : w0 + kFlatWin;
    if (lo < hi) {
      const int k1 = packed_before(hi - w0, b0, b1, n0);
      for (int k = packed_before(lo - w0, b0, b1, n0); k < k1; k++) {
        a0 += q0s[k];
        a1 += q1s[k];
        a2 += q2s[k];
      }
    }
    wave_lds_sync();
  }
}

template <bool MULTI>
__global__ __launch_bounds__(512, 6) void k_force_sphere_flat(
    const double4 *__restrict__ pos_in, double4 *__restrict__ pos_out,
    const int32_t *__restrict__ cidx, const uint8_t *__restrict__ cown,
    const int32_t *__restrict__ wtot, const int32_t *__restrict__ ncnt,
    int64_t n, int tsize, int32_t maxn, const int32_t *__restrict__ col,
    const BoxGeom *__restrict__ boxes, BoxGeom g0, ForceParams fp,
    double *__restrict__ fc, double *__restrict__ vmax,
    int32_t *__restrict__ err, int remap) {
  extern __shared__ __align__(16) unsigned char flat_lds[];
  const int lane = threadIdx.x & (kWave - 1);
  const int wv = threadIdx.x / kWave, nwv = blockDim.x / kWave;
  double4 *sp = reinterpret_cast<double4 *>(flat_lds) + wv * kWave;
  double *q0s = reinterpret_cast<double *>(flat_lds + nwv * kWave * sizeof(double4)) +
                wv * 4 * kFlatWin;
  double *q1s = q0s + kFlatWin, *q2s = q1s + kFlatWin, *qrs = q2s + kFlatWin;
  int32_t *scol = reinterpret_cast<int32_t *>(flat_lds + nwv * kFlatWaveBytes) +
                  wv * kWave;
  const int64_t tile = tile_of(remap) * nwv + wv;
  const int64_t t0 = tile * tsize, t = t0 + lane;
  const bool active = lane < tsize && t < n;
  // The wave's entries start at its tile's region (tsize * maxn entries).
  // Every load that does not depend on another is issued here, before
  // anything waits, from indexes valid for every lane (the last particle
  // for lanes past n, tile 0 for a wave past n): the row length, the wave's
  // entry count, the particle, its box and the first window of entries (a
  // tile's region, and the padding after the last one, is always
  // readable).  The one-box path takes the first window from these; the
  // per-entry-box path, which would spill with them live, reloads it.
  const bool live = t0 < n;  // the tile holds at least one particle
  const int64_t B = live ? t0 * maxn : 0;
  const int64_t tc = active ? t : n - 1;
  const int32_t raw_l = ncnt[tc];
  const int32_t T_l = wtot[live ? tile : 0];
  const double4 p_l = pos_in[tc];
  const int32_t col_l = MULTI ? col[tc] : 0;
  const int f0u = cidx[B + lane], f1u = cidx[B + kWave + lane];
  const int f0o = cown[B + lane], f1o = cown[B + kWave + lane];
  const int T = live ? T_l : 0;
  const int32_t raw = active ? raw_l : 0;
  const int wave_img = wave_or3(row_img(raw));
  const int c = row_len(raw);
  const int P = wave_incl_scan64(c) - c;
  const double4 p = active ? p_l : make_double4(0.0, 0.0, 0.0, 0.0);
  sp[lane] = p;
  if (MULTI) scol[lane] = active ? col_l : 0;
  // Several boxes: a wave whose particles all lie in one box (all but the
  // waves at colony boundaries) takes the one-box path with that box's
  // geometry, read once into scalar registers; the others read each
  // owner's box per entry.
  bool one_box = true;
  BoxGeom gw = g0;
  if (MULTI) {
    const int cw = __builtin_amdgcn_readfirstlane(col_l);  // lane 0 is active
    one_box = __all(!active || col_l == cw);
    if (one_box) gw = boxes[cw];
  }
  wave_lds_sync();
  double a0 = 0.0, a1 = 0.0, a2 = 0.0;
  if (one_box) {
    if (wave_img == 0)
      flat_rows<false, 0>(T, P, c, B, lane, f0u, f1u, f0o, f1o, cidx, cown,
                          pos_in, sp, scol, q0s, q1s, q2s, qrs, boxes, gw, fp,
                          a0, a1, a2);
    else if (wave_img == 1)
      flat_rows<false, 1>(T, P, c, B, lane, f0u, f1u, f0o, f1o, cidx, cown,
                          pos_in, sp, scol, q0s, q1s, q2s, qrs, boxes, gw, fp,
                          a0, a1, a2);
    else
      flat_rows<false, 7>(T, P, c, B, lane, f0u, f1u, f0o, f1o, cidx, cown,
                          pos_in, sp, scol, q0s, q1s, q2s, qrs, boxes, gw, fp,
                          a0, a1, a2);
  } else if (MULTI) {
    if (wave_img == 0)
      flat_rows<true, 0>(T, P, c, B, lane, f0u, f1u, f0o, f1o, cidx, cown,
                         pos_in, sp, scol, q0s, q1s, q2s, qrs, boxes, g0, fp,
                         a0, a1, a2);
    else if (wave_img == 1)
      flat_rows<true, 1>(T, P, c, B, lane, f0u, f1u, f0o, f1o, cidx, cown,
                         pos_in, sp, scol, q0s, q1s, q2s, qrs, boxes, g0, fp,
                         a0, a1, a2);
    else
      flat_rows<true, 7>(T, P, c, B, lane, f0u, f1u, f0o, f1o, cidx, cown,
                         pos_in, sp, scol, q0s, q1s, q2s, qrs, boxes, g0, fp,
                         a0, a1, a2);
  }
  double v2 = 0.0;
  if (active) {
    const BoxGeom &g = MULTI ? boxes[col_l] : g0;
    // growth surface (K.H:1009-1030); vcom x/y are zero
    a0 += 0.0;
    a1 += 0.0;
    a2 += wall_law(p.z, p.w, fp);
    double vx = fp.mob * a0, vy = fp.mob * a1, vz = fp.mob * a2;
    double x = p.x + fp.dt * vx, y = p.y + fp.dt * vy, z = p.z + fp.dt * vz;
    x = wrap_axis(x, g.plo[0], g.phi[0], g.L[0], g.periodic[0]);
    y = wrap_axis(y, g.plo[1], g.phi[1], g.L[1], g.periodic[1]);
    z = wrap_axis(z, g.plo[2], g.phi[2], g.L[2], g.periodic[2]);
    pos_out[t] = make_double4(x, y, z, p.w);
    if (fc) store_fc(fc, t, a0, a1, a2, 0.0, 0.0, 0.0);
    if (!(isfinite(a0) && isfinite(a1) && isfinite(a2))) atomicOr(err, ERRBIT_NAN);
    v2 = vx * vx + vy * vy + vz * vz;
  }
  if (vmax) wave_vmax(v2, fp.dt, vmax, tile, lane, live);
}

// Serial pass over one particle's row (the reference's per-particle
// neighbor loop): sphere pairs for yeast, segment pairs for
// hyphae, summed into acc in row order; ti is the particle's evolving
// record (rod_pair_i may repair a bond or promote a second segment).
template <bool MULTI>
__device__ void general_rows(int64_t t, const BoxGeom &g, const DynArrays &in,
                             const StaticArrays &st, const FlatRows &flat,
                             int32_t maxn, const int32_t *__restrict__ ncnt,
                             const ForceParams &fp, double acc[6], Topo &ti) {
  const int ty = st.type[t];
  const double4 p = in.pos[t];
  const double4 rod_i = in.rod[t];
  const int c = row_len(ncnt[t]);
  const int32_t *row = flat.cidx + row_base(flat, maxn, t);
  if (ty == rec::YEAST) {
    for (int k = 0; k < c; k++) {
      int u = row[k];
      if (st.type[u] != rec::YEAST) continue;  // r_lm = 0 (K.H:39)
      double4 o = in.pos[u];
      double d0 = sep_axis(p.x, o.x, g.L[0], g.halfL[0], g.periodic[0]);
      double d1 = sep_axis(p.y, o.y, g.L[1], g.halfL[1], g.periodic[1]);
      double d2 = sep_axis(p.z, o.z, g.L[2], g.halfL[2], g.periodic[2]);
      double r2 = d0 * d0 + d1 * d1 + d2 * d2;
      double rS = p.w + o.w;
      double lim = rS + fp.WA - 1.0e-15;
      if (r2 <= lim * lim)
        sphere_pair(d0, d1, d2, r2, rS, fp, acc[0], acc[1], acc[2]);
    }
  } else if (ty == rec::FUNGI) {
    RodSelf S;
    rod_self_init(S, rod_i, in.trig[t], p.w, st.bscale[t], fp.visc);
    for (int k = 0; k < c; k++) {
      int u = row[k];
      if (st.type[u] != rec::FUNGI) continue;
      double4 o = in.pos[u];
      double4 rod_j = in.rod[u];
      double d[3];
      d[0] = sep_axis(p.x, o.x, g.L[0], g.halfL[0], g.periodic[0]);
      d[1] = sep_axis(p.y, o.y, g.L[1], g.halfL[1], g.periodic[1]);
      d[2] = sep_axis(p.z, o.z, g.L[2], g.halfL[2], g.periodic[2]);
      double r2 = d[0] * d[0] + d[1] * d[1] + d[2] * d[2];
      double rlm = 1.5 * (rod_i.x + rod_j.x) + fp.WA;  // K.H:33-37
      double lim = rlm - 1.0e-15;
      if (r2 <= lim * lim) {
        Topo tj = in.topo[u];
        rod_pair_i(d, S, ti, tj, rod_j.x, o.w, st.bscale[u], in.trig[u], fp,
                   acc);
      }
    }
  }
}

// Surface term, overdamped update and outputs of one particle after its
// pair terms (K.H:1009-1282, PCI:311-449); returns |vel|^2.
__device__ double general_finish(int64_t t, const BoxGeom &g,
                                 const DynArrays &in, const DynArrays &out,
                                 const StaticArrays &st, const ForceParams &fp,
                                 double acc[6], Topo &ti,
                                 double *__restrict__ fc,
                                 int32_t *__restrict__ err) {
  const int ty = st.type[t];
  const double4 p = in.pos[t];
  const double4 rod_i = in.rod[t];
  const double4 tr_i = in.trig[t];
  if (ty == rec::YEAST) {
    acc[0] += 0.0;
    acc[1] += 0.0;
    acc[2] += wall_law(p.z, p.w, fp);
    acc[3] += 0.0;
    acc[4] += 0.0;
    acc[5] += 0.0;
  } else if (ty == rec::FUNGI) {
    RodSelf S;
    rod_self_init(S, rod_i, tr_i, p.w, st.bscale[t], fp.visc);
    double vs[3], ws[3];
    rod_surface(p, S, fp, vs, ws);
    acc[0] += vs[0];
    acc[1] += vs[1];
    acc[2] += vs[2];
    acc[3] += ws[0];
    acc[4] += ws[1];
    acc[5] += ws[2];
    ti.fix_site = 0;  // K.H:1060
  }
  double vx = fp.mob * acc[0], vy = fp.mob * acc[1], vz = fp.mob * acc[2];
  double x = p.x + fp.dt * vx, y = p.y + fp.dt * vy, z = p.z + fp.dt * vz;
  x = wrap_axis(x, g.plo[0], g.phi[0], g.L[0], g.periodic[0]);
  y = wrap_axis(y, g.plo[1], g.phi[1], g.L[1], g.periodic[1]);
  z = wrap_axis(z, g.plo[2], g.phi[2], g.L[2], g.periodic[2]);
  out.pos[t] = make_double4(x, y, z, p.w);
  if (ty == rec::FUNGI) {
    double th = rod_i.y, ph = rod_i.z;
    double w[3] = {acc[3], acc[4], acc[5]};
    rod_rotate(th, ph, tr_i, rod_i.x, w, fp.dt);
    const double4 rod_o = make_double4(rod_i.x, th, ph, rod_i.w);
    const double4 tr_o = trig_of(th, ph);
    out.rod[t] = rod_o;
    out.trig[t] = tr_o;
    if (out.near) out.near[t] = near_of(make_double4(x, y, z, p.w), ty, rod_o, tr_o, ti);
  } else {
    out.rod[t] = rod_i;
    out.trig[t] = tr_i;
    if (out.near)
      out.near[t] = near_of(make_double4(x, y, z, p.w), ty, rod_i, tr_i, ti);
  }
  out.topo[t] = ti;
  if (fc) {  // original order
    store_fc(fc, st.oid[t], acc[0], acc[1], acc[2], acc[3], acc[4], acc[5]);
  }
  bool fin = true;
#pragma unroll
  for (int k = 0; k < 6; k++) fin = fin && isfinite(acc[k]);
  if (!fin) atomicOr(err, ERRBIT_NAN);
  return vx * vx + vy * vy + vz * vz;
}

// ------------------------------------------------ flat general force ---
//
// Segments (and mixed colonies) over the flat row layout with tiles of at
// most kGTile particles, one tile per wave.  Per window of 128 entries a
// light pass reads one 64-byte sector per neighbor (SegNear), applies the
// interaction test, and finds the entries that act: spheres, pairs that may
// be bonded, and segments that may touch.  The other pairs' terms are zeros
// (a zero force through a finite mobility), which adding leaves out.  The
// entries that act queue up in LDS, in entry order; whenever 64 are queued
// they load the heavy data and run the pair law (rod_pair_forces,
// sphere_pair), each term into its LDS slot, and the tile's particles (the
// first lanes) add their runs of terms in row order.  The pair law is evaluated
// with the particle's record as it stands before its row; that is what the
// row loop sees unless an earlier pair of the row repaired a bond.  A tile
// where some pair repairs a bond is marked and recomputed row by row by
// k_force_general_redo (general_rows), so every result is the row loop's;
// keeping the row loop out of this kernel keeps its register budget low.
// Promotion of a second segment and the dltd reset do not depend on the
// order of the pairs.
//
// 200,000 segments (10.8 interacting pairs each, about three of which act):
// 93 us, half of it issuing vector instructions (28.5 M per launch), the
// rest waiting on dependent loads at three waves per SIMD.  With every
// interacting pair through the law it was 157 us and 55.3 M instructions.
// At 4 waves per SIMD 16 registers spill: 115 us.
constexpr int kGTile = 32;
constexpr int kGWin = 2 * kWave;
constexpr int kGPass = kWave;           // packed pairs per pass
constexpr int kGQueue = kGWin + kGPass; // entries that act, waiting
// LDS of an owner's SegNear, padded off the bank period
constexpr int kGNear = 80;
// LDS per wave: the terms of one pass (6 x 64), the tile's mobility matrices
// (18 per particle, formed once) and its SegNear, the queue (neighbor,
// owner) and the pass's promotion flags
size_t general_lds(int tile) {
  return 6 * kGPass * sizeof(double) +
         (size_t)tile * (18 * sizeof(double) + kGNear) +
         (2 * kGQueue + kGPass) * sizeof(int32_t);
}

template <bool MULTI>
__global__ __launch_bounds__(256, 3) void k_force_general_flat(
    DynArrays in, DynArrays out, StaticArrays st,
    const int32_t *__restrict__ cidx, const uint8_t *__restrict__ cown,
    const int32_t *__restrict__ wtot, int8_t *__restrict__ redo_tile,
    const int32_t *__restrict__ ncnt, int64_t n, int tsize, int32_t maxn,
    const BoxGeom *__restrict__ boxes, BoxGeom g0,
    ForceParams fp, double *__restrict__ fc, double *__restrict__ vmax,
    int32_t *__restrict__ err, int remap, int wave_bytes) {
  extern __shared__ __align__(16) unsigned char gen_lds[];
  const int lane = threadIdx.x & (kWave - 1);
  const int wv = threadIdx.x / kWave, nwv = blockDim.x / kWave;
  double *res = reinterpret_cast<double *>(gen_lds + wv * wave_bytes);
  double *mob = res + 6 * kGPass;  // mob[m * tsize + owner]: dii (m < 9), dij
  unsigned char *own = reinterpret_cast<unsigned char *>(mob + 18 * tsize);
  int32_t *qu = reinterpret_cast<int32_t *>(own + kGNear * tsize);
  int32_t *qo = qu + kGQueue;
  int32_t *pf = qo + kGQueue;
  const int64_t tile = tile_of(remap) * nwv + wv;
  const int64_t t0 = tile * tsize;
  const int64_t t = t0 + lane;
  const bool active = lane < tsize && t < n;
  int64_t B = 0;
  int T = 0;
  if (t0 < n) {
    B = t0 * maxn;
    T = wtot[tile];
  }
  const int32_t raw = active ? ncnt[t] : 0;
  const int c = row_len(raw);
  const int img = wave_or3(row_img(raw));  // axes that can need an image
  const int P = wave_incl_scan64(c) - c;
  if (active) {
    SegNear q = in.near[t];
    if (q.type == rec::FUNGI && c > 0) {
      // the two-site mobility of the segment, once (the pairs read it)
      RodSelf S;
      rod_self_geom(S, in.rod[t], in.trig[t], in.pos[t].w, st.bscale[t]);
      rod_self_mob(S, in.trig[t], fp.visc);
      double sum = 0.0;
#pragma unroll
      for (int a = 0; a < 3; a++)
#pragma unroll
        for (int b = 0; b < 3; b++) {
          mob[(3 * a + b) * tsize + lane] = S.dii[a][b];
          mob[(9 + 3 * a + b) * tsize + lane] = S.dij[a][b];
          sum += S.dii[a][b] + S.dij[a][b];
        }
      // a zero force leaves no term only through a finite mobility: with an
      // infinite radius here every pair goes through the law
      if (!isfinite(sum)) q.rad = __builtin_huge_valf();
    }
    *reinterpret_cast<SegNear *>(own + kGNear * lane) = q;
  }
  wave_lds_sync();
  const unsigned long long below = (1ull << lane) - 1ull;
  double acc[6] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
  bool paired = false, promoted = false, repair = false;
  int a_lo = 0, a_hi = 0;      // this owner's queued entries, counted from 0
  int queued = 0, passed = 0;  // entries queued and evaluated so far
  const float wa = (float)fp.WA;
  // bit 0: the pair interacts; bit 1: it acts
  auto light = [&](int o, int u, bool valid) -> int {
    if (!valid) return 0;
    const SegNear a = *reinterpret_cast<const SegNear *>(own + kGNear * o);
    const SegNear b = in.near[u];
    if (a.type != b.type || (a.type != rec::YEAST && a.type != rec::FUNGI)) return 0;
    const BoxGeom &g = MULTI ? boxes[st.col[t0 + o]] : g0;
    double d0 = a.x - b.x, d1 = a.y - b.y, d2 = a.z - b.z;
    if (img) {
      d0 = sep_axis(a.x, b.x, g.L[0], g.halfL[0], g.periodic[0]);
      d1 = sep_axis(a.y, b.y, g.L[1], g.halfL[1], g.periodic[1]);
      d2 = sep_axis(a.z, b.z, g.L[2], g.halfL[2], g.periodic[2]);
    }
    const double r2 = d0 * d0 + d1 * d1 + d2 * d2;
    const bool seg = a.type == rec::FUNGI;
    // K.H:33-37 and the sphere's r_lm
    const double lim = (seg ? 1.5 * (a.reach + b.reach) + fp.WA
                            : a.reach + b.reach + fp.WA) - 1.0e-15;
    if (!(r2 <= lim * lim)) return 0;
    if (seg && !may_bond(a.bonds, b.self) && !may_bond(b.bonds, a.self) &&
        cannot_touch(a, b, d0, d1, d2, wa))
      return 1;
    return 3;
  };
  // evaluates the first min(64, waiting) queued entries
  auto pass = [&]() {
    const int m = queued - passed < kGPass ? queued - passed : kGPass;
    if (lane < m) {
      const int ow = qo[lane];
      const int64_t u = qu[lane], ti_ = t0 + ow;
      const BoxGeom &g = MULTI ? boxes[st.col[ti_]] : g0;
      const double4 p = in.pos[ti_], o = in.pos[u];
      double d[3];
      d[0] = sep_axis(p.x, o.x, g.L[0], g.halfL[0], g.periodic[0]);
      d[1] = sep_axis(p.y, o.y, g.L[1], g.halfL[1], g.periodic[1]);
      d[2] = sep_axis(p.z, o.z, g.L[2], g.halfL[2], g.periodic[2]);
      double f[6] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
      int flag = 0;
      if (st.type[ti_] == rec::YEAST) {
        const double r2 = d[0] * d[0] + d[1] * d[1] + d[2] * d[2];
        sphere_pair(d[0], d[1], d[2], r2, p.w + o.w, fp, f[0], f[1], f[2]);
      } else {
        RodSelf S;
        rod_self_geom(S, in.rod[ti_], in.trig[ti_], p.w, st.bscale[ti_]);
        Topo tio = in.topo[ti_];
        const int pos0 = tio.position, nb0 = tio.n_bnds;
        double f1[3], f2[3], ri[3];
        {
          const Topo tj = in.topo[u];
          rod_pair_forces(d, S, tio, tj, in.rod[u].x, o.w, st.bscale[u],
                          in.trig[u], fp, f1, f2, ri);
        }
        if (tio.n_bnds != nb0) repair = true;
        if (tio.position != pos0) flag = 1;
#pragma unroll
        for (int a = 0; a < 3; a++)
#pragma unroll
          for (int b = 0; b < 3; b++) {
            S.dii[a][b] = mob[(3 * a + b) * tsize + ow];
            S.dij[a][b] = mob[(9 + 3 * a + b) * tsize + ow];
          }
        rod_pair_mobility(S, f1, f2, ri, f);
      }
#pragma unroll
      for (int q = 0; q < 6; q++) res[q * kGPass + lane] = f[q];
      pf[lane] = flag;
    }
    wave_lds_sync();
    const int k0 = a_lo > passed ? a_lo - passed : 0;
    const int k1 = a_hi < passed + m ? a_hi - passed : m;
    for (int k = k0; k < k1; k++) {
#pragma unroll
      for (int q = 0; q < 6; q++) acc[q] += res[q * kGPass + k];
      promoted = promoted || pf[k] != 0;
    }
    passed += m;
    wave_lds_sync();
  };
  for (int w0 = 0;;) {
    if (w0 < T) {
      const int e0 = w0 + lane, e1 = e0 + kWave;
      const bool v0 = e0 < T, v1 = e1 < T;
      int u0 = 0, u1 = 0, o0 = 0, o1 = 0;
      if (v0) {
        u0 = cidx[B + e0];
        o0 = cown[B + e0];
      }
      if (v1) {
        u1 = cidx[B + e1];
        o1 = cown[B + e1];
      }
      const int l0 = light(o0, u0, v0), l1 = light(o1, u1, v1);
      const unsigned long long i0 = __ballot(l0 & 1), i1 = __ballot(l1 & 1);
      const unsigned long long b0 = __ballot(l0 & 2), b1 = __ballot(l1 & 2);
      const int n0 = __popcll(b0), ni = n0 + __popcll(b1);
      const int qn = queued - passed;  // fewer than 64 wait here
      if (l0 & 2) {
        const int k = qn + __popcll(b0 & below);
        qu[k] = u0;
        qo[k] = o0;
      }
      if (l1 & 2) {
        const int k = qn + n0 + __popcll(b1 & below);
        qu[k] = u1;
        qo[k] = o1;
      }
      const int lo = P > w0 ? P : w0;
      const int hi = P + c < w0 + kGWin ? P + c : w0 + kGWin;
      if (lo < hi) {
        const int m0 = __popcll(i0);
        paired = paired || packed_before(hi - w0, i0, i1, m0) >
                               packed_before(lo - w0, i0, i1, m0);
        if (lo == P) a_lo = queued + packed_before(lo - w0, b0, b1, n0);
        a_hi = queued + packed_before(hi - w0, b0, b1, n0);
      }
      queued += ni;
      wave_lds_sync();
      w0 += kGWin;
    }
    const bool last = w0 >= T;
    while (queued - passed >= kGPass || (last && queued > passed)) {
      pass();
      // the entries behind the pass move to the front
      const int left = queued - passed;
      int u[2], o[2];
#pragma unroll
      for (int h = 0; h < 2; h++) {
        const int k = h * kWave + lane;
        u[h] = k < left ? qu[kGPass + k] : 0;
        o[h] = k < left ? qo[kGPass + k] : 0;
      }
      wave_lds_sync();
#pragma unroll
      for (int h = 0; h < 2; h++) {
        const int k = h * kWave + lane;
        if (k < left) {
          qu[k] = u[h];
          qo[k] = o[h];
        }
      }
      wave_lds_sync();
    }
    if (last) break;
  }
  // A tile with a bond repair is left to k_force_general_redo.
  const bool redo = __any(repair);
  if (lane == 0 && t0 < n) redo_tile[tile] = redo ? 1 : 0;
  double v2 = 0.0;
  if (active && !redo) {
    const BoxGeom &g = MULTI ? boxes[st.col[t]] : g0;
    Topo ti = in.topo[t];
    if (st.type[t] == rec::FUNGI && paired) {
      ti.dltd = 1;  // K.H:364-369
      if (promoted) ti.position = rec::INTERIOR;
    }
    v2 = general_finish(t, g, in, out, st, fp, acc, ti, fc, err);
  }
  if (vmax) wave_vmax(v2, fp.dt, vmax, tile, lane, t0 < n);
}

// The row loop for the particles of the tiles that the flat pass marked
// (a pair of the tile repairs a bond).  Runs after the flat pass on the
// same stream; its displacement maxima join the step's partials through an
// atomic max (non-negative doubles order as their bit patterns).
template <bool MULTI>
__global__ __launch_bounds__(256) void k_force_general_redo(
    DynArrays in, DynArrays out, StaticArrays st,
    const int8_t *__restrict__ redo_tile, FlatRows flat, int32_t maxn,
    const int32_t *__restrict__ ncnt, int64_t n,
    const BoxGeom *__restrict__ boxes, BoxGeom g0, ForceParams fp,
    double *__restrict__ fc, double *__restrict__ vmax,
    int32_t *__restrict__ err) {
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= n || !redo_tile[t / flat.tile]) return;
  const BoxGeom &g = MULTI ? boxes[st.col[t]] : g0;
  Topo ti = in.topo[t];
  double acc[6] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
  general_rows<MULTI>(t, g, in, st, flat, maxn, ncnt, fp, acc, ti);
  const double v2 = general_finish(t, g, in, out, st, fp, acc, ti, fc, err);
  if (vmax)
    atomicMax(reinterpret_cast<unsigned long long *>(vmax), dbits(fp.dt * sqrt(v2)));
}

// InitBonds: per segment, scan the row in order and append a bond for the
// first site pair closer than rlim (K.H:1285-1444 with rlim = 1e-7, PCI:508).
template <bool MULTI>
__global__ void k_init_bonds(DynArrays dy, StaticArrays st, FlatRows flat,
                             int32_t maxn, const int32_t *__restrict__ ncnt,
                             int64_t n, const BoxGeom *__restrict__ boxes,
                             BoxGeom g0, ForceParams fp,
                             int32_t *__restrict__ err) {
  int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= n || st.type[t] != rec::FUNGI) return;
  const BoxGeom &g = MULTI ? boxes[st.col[t]] : g0;
  const double rlim = 1.0e-7;
  double4 p = dy.pos[t];
  double4 rod_i = dy.rod[t];
  double4 tr = dy.trig[t];
  double Li = rod_i.x;
  double nxi = tr.y * tr.z, nyi = tr.y * tr.w, nzi = tr.x;
  Topo ti = dy.topo[t];
  int c = row_len(ncnt[t]);
  const int32_t *row = flat.cidx + row_base(flat, maxn, t);
  for (int k = 0; k < c; k++) {
    int u = row[k];
    if (st.type[u] != rec::FUNGI) continue;
    double4 o = dy.pos[u];
    double4 rod_j = dy.rod[u];
    double d[3];
    d[0] = sep_axis(p.x, o.x, g.L[0], g.halfL[0], g.periodic[0]);
    d[1] = sep_axis(p.y, o.y, g.L[1], g.halfL[1], g.periodic[1]);
    d[2] = sep_axis(p.z, o.z, g.L[2], g.halfL[2], g.periodic[2]);
    double r2 = d[0] * d[0] + d[1] * d[1] + d[2] * d[2];
    double lim = 1.5 * (Li + rod_j.x) + fp.WA - 1.0e-15;
    if (!(r2 <= lim * lim)) continue;
    double4 trj = dy.trig[u];
    double Lj = rod_j.x;
    double nxj = trj.y * trj.z, nyj = trj.y * trj.w, nzj = trj.x;
    double xi1 = d[0] - 0.5 * nxi * Li, yi1 = d[1] - 0.5 * nyi * Li,
           zi1 = d[2] - 0.5 * nzi * Li;
    double xi2 = d[0] + 0.5 * nxi * Li, yi2 = d[1] + 0.5 * nyi * Li,
           zi2 = d[2] + 0.5 * nzi * Li;
    double xj1 = -0.5 * nxj * Lj, yj1 = -0.5 * nyj * Lj, zj1 = -0.5 * nzj * Lj;
    double xj2 = 0.5 * nxj * Lj, yj2 = 0.5 * nyj * Lj, zj2 = 0.5 * nzj * Lj;
    // site pairs in the reference's order 1-1, 2-1, 1-2, 2-2
    for (int cse = 0; cse < 4; cse++) {
      bool i2 = (cse & 1) != 0, j2 = (cse & 2) != 0;
      double rx = (i2 ? xi2 : xi1) - (j2 ? xj2 : xj1);
      double ry = (i2 ? yi2 : yi1) - (j2 ? yj2 : yj1);
      double rz = (i2 ? zi2 : zi1) - (j2 ? zj2 : zj1);
      double r = sqrt(rx * rx + ry * ry + rz * rz);
      if (r < rlim) {
        int nb = ti.n_bnds;
        if (nb < 0 || nb > 3) {
          atomicOr(err, ERRBIT_BOND);
        } else {
          ti.seg_id[nb] = dy.topo[u].self_id;
          ti.seg_cpu[nb] = dy.topo[u].self_cpu;
          ti.site[nb] = i2 ? 2 : 1;
          ti.n_bnds = nb + 1;
        }
        break;
      }
    }
  }
  dy.topo[t].n_bnds = ti.n_bnds;
  for (int b = 0; b < 4; b++) {
    dy.topo[t].seg_id[b] = ti.seg_id[b];
    dy.topo[t].seg_cpu[b] = ti.seg_cpu[b];
    dy.topo[t].site[b] = ti.site[b];
  }
}

// Sum over the steps since the last rebuild of the largest displacement in
// any block bounds every particle's displacement; more than half the skin
// means a pair may have entered interaction range unlisted.  Stage 1: each
// block takes the per-slot max over a chunk of force blocks into slotmax
// (one atomic per slot per block, values >= 0 compare as integers).
// Block (x, y) takes slot y over a chunk of kSkinChunk force blocks.
constexpr int kSkinChunk = 4096;
__global__ __launch_bounds__(256) void k_skin_partial(
    double *__restrict__ vpart, int32_t stride, int clear,
    unsigned long long *__restrict__ slotmax) {
  __shared__ double shd[4];
  const int sl = blockIdx.y;
  const int64_t b0 = (int64_t)blockIdx.x * kSkinChunk;
  const int64_t b1 = b0 + kSkinChunk < stride ? b0 + kSkinChunk : stride;
  double m = 0.0;
  for (int64_t b = b0 + threadIdx.x; b < b1; b += blockDim.x) {
    double v = vpart[(int64_t)sl * stride + b];
    m = v > m ? v : m;
    if (clear) vpart[(int64_t)sl * stride + b] = 0.0;
  }
  m = block_max(m, shd);
  if (threadIdx.x == 0 && m > 0.0) atomicMax(&slotmax[sl], dbits(m));
}

// Stage 2: sum the slot maxima in slot order, compare, reset the slot
// maxima.
__global__ void k_skin_final(unsigned long long *__restrict__ slotmax,
                             int32_t nslots, double limit,
                             int32_t *__restrict__ err) {
  if (threadIdx.x != 0 || blockIdx.x != 0) return;
  double total = 0.0;
  for (int sl = 0; sl < nslots; sl++) {
    total += __longlong_as_double((long long)slotmax[sl]);
    slotmax[sl] = 0ull;
  }
  if (total > limit) atomicOr(err, ERRBIT_SKIN);
}

// ------------------------------------------------------------- exports ---

// fc from its kept layout (oid: the order of the step; null: original) to
// the reference's component-major fc[i + c * n]
__global__ void k_export_fc(const double *__restrict__ fc,
                            const int32_t *__restrict__ oid, int64_t n,
                            double *__restrict__ out) {
  int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= n) return;
  const int64_t o = oid ? oid[t] : t;
  for (int c = 0; c < 6; c++) out[c * n + o] = fc[t * 6 + c];
}
__global__ void k_export_pos(const double4 *__restrict__ pos,
                             const int32_t *__restrict__ oid, int64_t n,
                             double *__restrict__ out) {
  int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= n) return;
  int64_t o = oid[t];
  double4 p = pos[t];
  out[3 * o] = p.x;
  out[3 * o + 1] = p.y;
  out[3 * o + 2] = p.z;
}
__global__ void k_export_orient(const double4 *__restrict__ rod,
                                const int32_t *__restrict__ oid, int64_t n,
                                double *__restrict__ out) {
  int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= n) return;
  int64_t o = oid[t];
  double4 r = rod[t];
  out[2 * o] = r.y;
  out[2 * o + 1] = r.z;
}
__global__ void k_export_i32(const int32_t *__restrict__ v,
                             const int32_t *__restrict__ oid, int64_t n,
                             int32_t *__restrict__ out) {
  int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= n) return;
  out[oid[t]] = v[t];
}
__global__ void k_export_counts(const int32_t *__restrict__ ncnt,
                                const int32_t *__restrict__ oid, int64_t n,
                                int64_t *__restrict__ out) {
  int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= n) return;
  out[oid[t]] = row_len(ncnt[t]);
}
// Rows from the flat layout, in original order.
__global__ void k_export_nbr(FlatRows flat, int32_t maxn,
                             const int32_t *__restrict__ ncnt,
                             const int32_t *__restrict__ oid, int64_t n,
                             const int64_t *__restrict__ row_off,
                             int32_t *__restrict__ out) {
  int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= n) return;
  const int64_t b = row_base(flat, maxn, t);
  int64_t base = row_off[oid[t]];
  int c = row_len(ncnt[t]);
  for (int k = 0; k < c; k++) out[base + k] = oid[flat.cidx[b + k]];
}

}  // namespace

// ----------------------------------------------------------- launchers ---

hipError_t launch_fill_i32(int32_t *p, int64_t n, int32_t v, hipStream_t s) {
  if (n <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_fill<int32_t>, dim3(grid_capped(n, 256)), dim3(256), 0,
                     s, p, n, v);
  return hipGetLastError();
}
hipError_t launch_fill_u64(unsigned long long *p, int64_t n,
                           unsigned long long v, hipStream_t s) {
  if (n <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_fill<unsigned long long>, dim3(grid_capped(n, 256)),
                     dim3(256), 0, s, p, n, v);
  return hipGetLastError();
}

hipError_t launch_aos_unpack(const uint8_t *aos, AosLayout lay, int64_t n,
                             const int32_t *col, const BoxGeom *boxes,
                             BoxGeom g0, StaticArrays st, DynArrays dy,
                             unsigned long long *stats, hipStream_t s) {
  if (n <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_aos_unpack, dim3(grid_for(n, 256)), dim3(256), 0, s,
                     aos, lay, n, col, boxes, g0, st, dy, stats);
  return hipGetLastError();
}
hipError_t launch_aos_refresh(const uint8_t *aos, AosLayout lay, int64_t n,
                              BoxGeom g, StaticArrays st, DynArrays dy,
                              uint32_t fields, unsigned long long *stats,
                              hipStream_t s) {
  if (n <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_aos_refresh, dim3(grid_for(n, 256)), dim3(256), 0, s,
                     aos, lay, n, g, st, dy, fields, stats);
  return hipGetLastError();
}

// Records that outgrow the 256 MB Infinity Cache are packed in record order.
// Below, the scattered stores merge in the cache and the extra launch does
// not pay: 20,011 segments 7 us scattered, 14 in record order; 307,201
// spheres (138 MB) 22.5 and 27; 690,000 (309 MB) 77 and 76; 1M (448 MB) 129
// and 112.
constexpr int64_t kPackWide = 320ll << 20;

hipError_t launch_aos_pack(uint8_t *aos, AosLayout lay, int64_t n,
                           StaticArrays st, DynArrays dy, const double *fc,
                           int fc_orig, const double *state, int has_rel, double mob,
                           int wrote_step, int any_fungi, int32_t *inv,
                           hipStream_t s) {
  if (n <= 0) return hipSuccess;
  if (n * (int64_t)lay.stride <= kPackWide) {
    hipLaunchKernelGGL(k_aos_pack, dim3(grid_for(n, 256)), dim3(256), 0, s, aos,
                       lay, n, st, dy, fc, fc_orig, mob, wrote_step, any_fungi);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess || !state) return e;
    return launch_chem_pack(aos, lay, n, has_rel, state, st.oid, st.type, dy.pos,
                            dy.rod, s);
  }
  const PackWhat what{wrote_step, fc_orig, has_rel};
  hipLaunchKernelGGL(k_inverse, dim3(grid_for(n, 256)), dim3(256), 0, s, st.oid,
                     n, inv);
#define BMX_PACK(F, C)                                                        \
  hipLaunchKernelGGL((k_aos_pack_wide<F, C>), dim3(grid_for(n, kWave)), dim3(kWave), \
                     (PackShape<F, C>::lds), s, aos, lay, n, inv, st.type, dy, \
                     fc, state, mob, what)
  if (any_fungi && state)
    BMX_PACK(true, true);
  else if (any_fungi)
    BMX_PACK(true, false);
  else if (state)
    BMX_PACK(false, true);
  else
    BMX_PACK(false, false);
#undef BMX_PACK
  return hipGetLastError();
}

hipError_t launch_bin_count(const double4 *pos, const int32_t *col,
                            const BoxGeom *boxes, BoxGeom g0, int multi,
                            int64_t n, int32_t *key, int32_t *rank,
                            int32_t *count, hipStream_t s, SkinCheck sk) {
  if (n <= 0) return hipSuccess;
  if (multi)
    hipLaunchKernelGGL(k_bin_count<true>, dim3(grid_for(n, 256)), dim3(256), 0,
                       s, pos, col, boxes, g0, n, key, rank, count, sk);
  else
    hipLaunchKernelGGL(k_bin_count<false>, dim3(grid_for(n, 256)), dim3(256),
                       0, s, pos, col, boxes, g0, n, key, rank, count, sk);
  return hipGetLastError();
}

int64_t scan_scratch_elems(int64_t nb) {
  return (nb + kScanTile - 1) / kScanTile + 1;
}

hipError_t launch_scan(int32_t *count, int32_t *start, int64_t nb,
                       int32_t *scratch, hipStream_t s, SkinCheck sk) {
  int64_t nt = (nb + kScanTile - 1) / kScanTile;
  if (nt < 1) nt = 1;
  if (nt > 1024 * 64) return hipErrorInvalidValue;
  hipLaunchKernelGGL(k_scan_local, dim3((unsigned)nt), dim3(kScanThreads), 0,
                     s, count, start, scratch, nb, sk);
  hipLaunchKernelGGL(k_scan_add, dim3((unsigned)nt), dim3(kScanThreads), 0, s,
                     start, scratch, nt, nb);
  return hipGetLastError();
}

hipError_t launch_bin_scatter(const int32_t *key, const int32_t *rank,
                              const int32_t *start, const int32_t *oid,
                              int64_t n, unsigned long long *permk,
                              hipStream_t s) {
  if (n <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_bin_scatter, dim3(grid_for(n, 256)), dim3(256), 0, s,
                     key, rank, start, oid, n, permk);
  return hipGetLastError();
}
hipError_t launch_sort_gather(const unsigned long long *permk,
                              const int32_t *start, int64_t n,
                              StaticArrays src_s, StaticArrays dst_s,
                              DynArrays src_d, DynArrays dst_d,
                              const int32_t *key, int multi, int rods,
                              int32_t *err, hipStream_t s,
                              const double *chem_src, double *chem_dst) {
  if (n <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_sort_gather, dim3(grid_for(n, 256)), dim3(256), 0, s,
                     permk, start, n, src_s, dst_s, src_d, dst_d, key, multi,
                     rods, err, chem_src, chem_dst);
  return hipGetLastError();
}

int32_t tile_count(int64_t n, int tile) { return grid_for(n, tile); }

namespace {
// blocks of a force launch, one wave per tile
int force_blocks(int64_t n, int tile, int block) {
  return grid_for(tile_count(n, tile), block / kWave);
}
// Lanes per particle of the row build.  More lanes shorten each particle's
// chain of dependent loads, until the waves they make no longer fit the chip
// at once.  A block is one tile, at least one wave and at most 256 threads, so
// the tile bounds the choice: tiles of 64 take 2 or 4 lanes, of 32 2 to 8, of
// 16 4 to 16, of 8 8 or 16, and of 4 16 (the lines at 8,000 and 60,000 tell
// the tiles below 64 apart; sparse spheres have 4 lanes up to 400,000).
// Whole rebuilds, us, medians of runs that differ by 1 to 3, by lanes:
//                                       16      8      4      2
//   spheres, tiles of 64:    2,000                  33.7   36.8
//                           24,000                  35.8   38.9
//                          120,000                  43.9   45.2
//                          300,000                  63.5   65.2
//                        1,000,000                 136.9  134.7
//   tiles of 32:             5,000           31.9   34.5   38.1
//                           24,000           34.4   36.6   41.0
//                          120,000           49.1   47.2   48.0
//   tiles of 16:             5,000   33.5    35.4   39.9
//                           24,000   36.1    36.7   40.5
//                           90,000   54.2    50.0   50.1
//   segments, stencil rows,
//   tiles of 8:             20,000   28.2    28.2
//   tiles of 16:            40,000   34.5    32.0   32.6
//   tiles of 32:            60,000           35.1   35.3   38.8
//                          200,000           63.5   58.4   61.4
int build_lanes(int tile, int64_t n) {
  const int g = n > 400000 ? 2 : (n > 60000 ? 4 : (n > 8000 ? 8 : 16));
  return std::min(std::max(g, kWave / tile), 256 / tile);
}
}  // namespace

hipError_t launch_build_nbr(const double4 *pos, const int32_t *col,
                            const int32_t *type, const double4 *rod,
                            const BoxGeom *boxes, BoxGeom g0, int multi,
                            int rods, const int32_t *start, const int32_t *key,
                            int64_t n, int mode, double crit, double wa,
                            double skin, int32_t *nbr, int32_t *ncnt,
                            int64_t ncap, int32_t maxn, int32_t *err,
                            int32_t *bstats, FlatRows flat, int remap,
                            hipStream_t s) {
  if (n <= 0) return hipSuccess;
  const int G = build_lanes(flat.tile, n);
#define BMX_BUILD(M, RD, G_)                                                  \
  hipLaunchKernelGGL((k_build_rows<M, RD, G_>), dim3(tile_count(n, flat.tile)), \
                     dim3(flat.tile * G_), build_lds(flat.tile), s, pos, col, \
                     type, rod, boxes, g0, start, key, n, mode, crit, wa,     \
                     skin, nbr, ncnt, ncap, maxn, err, bstats, flat, remap)
#define BMX_BUILD_G(M, RD)                                                    \
  do {                                                                        \
    if (G == 2)                                                               \
      BMX_BUILD(M, RD, 2);                                                    \
    else if (G == 4)                                                          \
      BMX_BUILD(M, RD, 4);                                                    \
    else if (G == 8)                                                          \
      BMX_BUILD(M, RD, 8);                                                    \
    else                                                                      \
      BMX_BUILD(M, RD, 16);                                                   \
  } while (0)
  if (multi && rods)
    BMX_BUILD_G(true, true);
  else if (multi)
    BMX_BUILD_G(true, false);
  else if (rods)
    BMX_BUILD_G(false, true);
  else
    BMX_BUILD_G(false, false);
#undef BMX_BUILD_G
#undef BMX_BUILD
  return hipGetLastError();
}


// The tail of a call in one launch: the row statistics of a build since the
// last one (nblk > 0), then the error word (add: OR-ed in, so that calls
// enqueued back to back add up until the host reads and clears it), the
// longest row and the entry total (out: 4 words, in host memory mapped for
// the device where there is such memory), and the device's error word
// cleared.
__global__ __launch_bounds__(1024) void k_flags_out(
    const int32_t *__restrict__ bstats, int32_t nblk,
    int32_t *__restrict__ stats, unsigned long long *__restrict__ total,
    int32_t *__restrict__ err, int32_t *__restrict__ out, int add) {
  __shared__ int32_t shi[16];
  __shared__ unsigned long long shu[16];
  if (nblk > 0) {
    int m = 0;
    unsigned long long sm = 0;
    for (int b = threadIdx.x; b < nblk; b += blockDim.x) {
      int v = bstats[2 * b];
      m = v > m ? v : m;
      sm += (unsigned long long)bstats[2 * b + 1];
    }
    m = block_max(m, shi);
    __syncthreads();
    sm = block_sum(sm, shu);
    if (threadIdx.x == 0) {
      stats[0] = m;
      *total = sm;
    }
  }
  if (threadIdx.x == 0) {
    const unsigned long long tot = *total;
    out[0] = add ? out[0] | *err : *err;
    out[1] = stats[0];
    out[2] = (int32_t)(uint32_t)(tot & 0xffffffffull);
    out[3] = (int32_t)(uint32_t)(tot >> 32);
    *err = 0;
  }
}

// The error word of a mesh call, cleared behind it, and (maxima) the two
// size maxima of the chemistry, into mapped host memory.
__global__ void k_mesh_out(int32_t *__restrict__ err,
                           const unsigned long long *__restrict__ maxima,
                           int32_t *__restrict__ out_err,
                           unsigned long long *__restrict__ out_max) {
  out_err[0] = *err;
  *err = 0;
  if (maxima) {
    out_max[0] = maxima[0];
    out_max[1] = maxima[1];
  }
}
hipError_t launch_mesh_out(int32_t *err, const unsigned long long *maxima,
                           int32_t *out_err, unsigned long long *out_max,
                           hipStream_t s) {
  hipLaunchKernelGGL(k_mesh_out, dim3(1), dim3(1), 0, s, err, maxima, out_err,
                     out_max);
  return hipGetLastError();
}

hipError_t launch_flags_out(const int32_t *bstats, int32_t nblk, int32_t *stats,
                            unsigned long long *total, int32_t *err,
                            int32_t *out, int add, hipStream_t s) {
  hipLaunchKernelGGL(k_flags_out, dim3(1), dim3(nblk > 0 ? 1024 : kWave), 0, s,
                     bstats, nblk, stats, total, err, out, add);
  return hipGetLastError();
}

size_t flat_lds_bytes(int block, int multi) {
  return (size_t)(block / kWave) * (kFlatWaveBytes + (multi ? kWave * sizeof(int32_t) : 0));
}

hipError_t launch_force_sphere_flat(const double4 *pos_in, double4 *pos_out,
                                    const int32_t *cidx, const uint8_t *cown,
                                    const int32_t *wtot, const int32_t *ncnt,
                                    int64_t n, int tile, int32_t maxn,
                                    const int32_t *col,
                                    const BoxGeom *boxes, BoxGeom g0, int multi,
                                    ForceParams fp, double *fc, double *vmax,
                                    int32_t *err, LaunchShape ls,
                                    hipStream_t s) {
  if (n <= 0) return hipSuccess;
  const int b = ls.block;
  const size_t lds = flat_lds_bytes(b, multi);
  const int grid = force_blocks(n, tile, b);
  if (multi)
    hipLaunchKernelGGL(k_force_sphere_flat<true>, dim3(grid), dim3(b), lds, s,
                       pos_in, pos_out, cidx, cown, wtot, ncnt, n, tile, maxn,
                       col, boxes, g0, fp, fc, vmax, err, ls.remap);
  else
    hipLaunchKernelGGL(k_force_sphere_flat<false>, dim3(grid), dim3(b), lds, s,
                       pos_in, pos_out, cidx, cown, wtot, ncnt, n, tile, maxn,
                       col, boxes, g0, fp, fc, vmax, err, ls.remap);
  return hipGetLastError();
}

hipError_t launch_force_general(DynArrays in, DynArrays out, StaticArrays st,
                                FlatRows flat, int8_t *redo_tile,
                                const int32_t *ncnt, int64_t n, int32_t maxn,
                                const BoxGeom *boxes, BoxGeom g0, int multi,
                                ForceParams fp, double *fc, double *vmax,
                                int32_t *err, LaunchShape ls, hipStream_t s) {
  if (n <= 0) return hipSuccess;
  const int b = ls.block > 256 ? 256 : ls.block;
  const int grid = force_blocks(n, flat.tile, b);
  const int wave_bytes = (int)general_lds(flat.tile);
  const size_t lds = (size_t)(b / kWave) * wave_bytes;
  if (multi) {
    hipLaunchKernelGGL(k_force_general_flat<true>, dim3(grid), dim3(b), lds, s,
                       in, out, st, flat.cidx, flat.cown, flat.tot, redo_tile,
                       ncnt, n, flat.tile, maxn, boxes, g0, fp, fc, vmax, err,
                       ls.remap, wave_bytes);
    hipLaunchKernelGGL(k_force_general_redo<true>, dim3(grid_for(n, 256)),
                       dim3(256), 0, s, in, out, st, redo_tile, flat, maxn,
                       ncnt, n, boxes, g0, fp, fc, vmax, err);
  } else {
    hipLaunchKernelGGL(k_force_general_flat<false>, dim3(grid), dim3(b), lds, s,
                       in, out, st, flat.cidx, flat.cown, flat.tot, redo_tile,
                       ncnt, n, flat.tile, maxn, boxes, g0, fp, fc, vmax, err,
                       ls.remap, wave_bytes);
    hipLaunchKernelGGL(k_force_general_redo<false>, dim3(grid_for(n, 256)),
                       dim3(256), 0, s, in, out, st, redo_tile, flat, maxn,
                       ncnt, n, boxes, g0, fp, fc, vmax, err);
  }
  return hipGetLastError();
}

// Particles per tile, one wave per tile of the force pass.  A wave's time
// grows with the windows of 128 entries its tile holds, and every wave pays
// its own start and end, so a tile holds about one window, as long as the
// waves are resident at once (6 per SIMD: 6,144); beyond that, tiles grow
// until they are few enough or hold four windows, where the share of start
// and end is small.  Force pass, us, tiles of 64 / 32 / 16 / 8 / 4:
//   rows of 1:  n = 24,000: 4.2 / 4.4 / 4.8 / 5.3 / 7.1; 1M: 18.7 / 26.7 / 44
//   rows of 8:  24,000: 11.9 / 8.5 / 7.2 / 6.0 / 7.9;
//               120,000: 15.3 / 13.6 / 15.0 / 16.1; 1M: 59 / 62 / 74 / 92
//   rows of 72: 24,000: 57 / 32 / 21 / 15.0 / 14.0; 120,000: 73 / 52 / 45 / 42.5 / 47
// Segment waves carry far more per particle, so their tiles are as small as
// keeps the waves resident at once (3 per SIMD), 64 / 32 / 16 / 8 / 4:
//   5,000: - / 34 / 25 / 21.8 / 20.8; 20,000: 58 / 39 / 30 / 27.9 / 37;
//   40,000: 63 / 47 / 36 / 42; 60,000: 63 / 45 / 48 / 55;
//   200,000: 116 / 93 / 106 / 144
int flat_tile(int segments, int64_t n, double row) {
  int t = 4;
  if (segments) {
    while (t < kGTile && n > (int64_t)t * 3072) t *= 2;
    return t;
  }
  while (t < kWave && 2 * t * row <= kFlatWin) t *= 2;
  while (t < kWave && n > (int64_t)t * 6144 && t * row < 4 * kFlatWin) t *= 2;
  return t;
}
int64_t flat_entries(int64_t ncap, int tile, int32_t maxn) {
  // + one window: the force pass reads a window before it knows the count
  return (ncap + tile - 1) / tile * (int64_t)tile * maxn + kFlatWin;
}

hipError_t launch_init_bonds(DynArrays dy, StaticArrays st, FlatRows flat,
                             int32_t maxn, const int32_t *ncnt, int64_t n,
                             const BoxGeom *boxes, BoxGeom g0, int multi,
                             ForceParams fp, int32_t *err, hipStream_t s) {
  if (n <= 0) return hipSuccess;
  if (multi)
    hipLaunchKernelGGL(k_init_bonds<true>, dim3(grid_for(n, 128)), dim3(128),
                       0, s, dy, st, flat, maxn, ncnt, n, boxes, g0, fp, err);
  else
    hipLaunchKernelGGL(k_init_bonds<false>, dim3(grid_for(n, 128)), dim3(128),
                       0, s, dy, st, flat, maxn, ncnt, n, boxes, g0, fp, err);
  return hipGetLastError();
}

hipError_t launch_skin_check(double *vpart, int32_t nslots, int32_t stride,
                             double limit, int clear,
                             unsigned long long *slotmax, int32_t *err,
                             hipStream_t s) {
  int chunks = (stride + kSkinChunk - 1) / kSkinChunk;
  if (chunks < 1) chunks = 1;
  hipLaunchKernelGGL(k_skin_partial, dim3(chunks, nslots > 0 ? nslots : 1),
                     dim3(256), 0, s, vpart, stride, clear, slotmax);
  hipLaunchKernelGGL(k_skin_final, dim3(1), dim3(64), 0, s, slotmax, nslots,
                     limit, err);
  return hipGetLastError();
}

hipError_t launch_fc_to_orig(const double *fc, const int32_t *oid, int64_t n,
                             double *out, hipStream_t s) {
  if (n <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_fc_to_orig, dim3(grid_for(n, 256)), dim3(256), 0, s, fc,
                     oid, n, out);
  return hipGetLastError();
}
hipError_t launch_export_fc(const double *fc, const int32_t *oid, int64_t n,
                            double *out, hipStream_t s) {
  if (n <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_export_fc, dim3(grid_for(n, 256)), dim3(256), 0, s, fc,
                     oid, n, out);
  return hipGetLastError();
}
hipError_t launch_export_pos(const double4 *pos, const int32_t *oid, int64_t n,
                             double *out, hipStream_t s) {
  if (n <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_export_pos, dim3(grid_for(n, 256)), dim3(256), 0, s,
                     pos, oid, n, out);
  return hipGetLastError();
}
hipError_t launch_export_orient(const double4 *rod, const int32_t *oid,
                                int64_t n, double *out, hipStream_t s) {
  if (n <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_export_orient, dim3(grid_for(n, 256)), dim3(256), 0, s,
                     rod, oid, n, out);
  return hipGetLastError();
}
hipError_t launch_export_i32(const int32_t *v, const int32_t *oid, int64_t n,
                             int32_t *out, hipStream_t s) {
  if (n <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_export_i32, dim3(grid_for(n, 256)), dim3(256), 0, s, v,
                     oid, n, out);
  return hipGetLastError();
}
hipError_t launch_export_counts(const int32_t *ncnt, const int32_t *oid,
                                int64_t n, int64_t *out, hipStream_t s) {
  if (n <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_export_counts, dim3(grid_for(n, 256)), dim3(256), 0, s,
                     ncnt, oid, n, out);
  return hipGetLastError();
}
hipError_t launch_export_nbr(FlatRows flat, int32_t maxn, const int32_t *ncnt,
                             const int32_t *oid, int64_t n,
                             const int64_t *row_off, int32_t *out,
                             hipStream_t s) {
  if (n <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_export_nbr, dim3(grid_for(n, 256)), dim3(256), 0, s,
                     flat, maxn, ncnt, oid, n, row_off, out);
  return hipGetLastError();
}

}  // namespace bmx
