// bmx_exchange.hip -- ParticleExchange: transfer of the species A, B, C
// between bonded segments over the neighbour rows
// (src/des/bmx_pc_xchng.cpp:13-257; initExchange / evaluateExchange /
// applyIncrements, src/chemistry/bmx_chem_K.H:1951-2112).
//
// The concentrations, volumes and increments are the chemistry state's line
// of each particle, in sorted order; the rows, bond tables and radii are the
// sorted arrays of the last rebuild.  Each row adds only into its own
// increments, in row order: the neighbour is seen through a copy in the
// reference, so its side of the flux is dropped there too.
#include "bmx_device.h"
#include "bmx_kernels.h"

namespace bmx {

namespace {

__global__ void k_chem_unpack(const uint8_t *__restrict__ aos, AosLayout lay,
                              int64_t n, int has_rel,
                              const int32_t *__restrict__ oid,
                              double *__restrict__ state) {
  int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= n) return;
  const double *rd = reinterpret_cast<const double *>(
      aos + (int64_t)oid[t] * lay.stride + lay.rdata);
  double4 *q = reinterpret_cast<double4 *>(state + t * chem::stride);
  q[0] = make_double4(rd[rec::first_data], rd[rec::first_data + 1],
                      rd[rec::first_data + 2], rd[rec::vol]);
  q[1] = make_double4(rd[rec::first_data + 3], rd[rec::first_data + 4],
                      rd[rec::first_data + 5], rd[rec::area]);
  q[2] = make_double4(rd[rec::dadt], rd[rec::dvdt], rd[rec::gx], rd[rec::gy]);
  q[3] = has_rel ? make_double4(rd[rec::gz], rd[rec::first_data + 6],
                                rd[rec::first_data + 7], rd[rec::first_data + 8])
                 : make_double4(rd[rec::gz], 0.0, 0.0, 0.0);
}

// Walks the sorted arrays, so each record also gets its radius and, for a
// segment, its length from where the mechanics keep them.
__global__ void k_chem_pack(uint8_t *__restrict__ aos, AosLayout lay, int64_t n,
                            int has_rel, const double *__restrict__ state,
                            const int32_t *__restrict__ oid,
                            const int32_t *__restrict__ type,
                            const double4 *__restrict__ pos,
                            const double4 *__restrict__ rod) {
  int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= n) return;
  const int64_t o = oid[t];
  double *rd = reinterpret_cast<double *>(aos + o * (int64_t)lay.stride + lay.rdata);
  const double4 *q = reinterpret_cast<const double4 *>(state + t * chem::stride);
  const double4 a = q[0], b = q[1], c = q[2], d = q[3];
  rd[rec::radius] = pos[t].w;
  if (type[t] == rec::FUNGI) rd[rec::c_length] = rod[t].x;
  rd[rec::area] = b.w;
  rd[rec::vol] = a.w;
  rd[rec::gx] = c.z;
  rd[rec::gy] = c.w;
  rd[rec::gz] = d.x;
  rd[rec::dadt] = c.x;
  rd[rec::dvdt] = c.y;
  rd[rec::first_data] = a.x;
  rd[rec::first_data + 1] = a.y;
  rd[rec::first_data + 2] = a.z;
  rd[rec::first_data + 3] = b.x;
  rd[rec::first_data + 4] = b.y;
  rd[rec::first_data + 5] = b.z;
  if (has_rel) {
    rd[rec::first_data + 6] = d.y;
    rd[rec::first_data + 7] = d.z;
    rd[rec::first_data + 8] = d.w;
  }
}

// The flux of one species from i to j (evaluateExchange, bmx_chem_K.H:
// 2041-2068): the area-weighted difference, clamped so that neither side
// gives more than its share per bond.
__device__ __forceinline__ double species_flux(double c1, double c2, double area,
                                               double mt, double dt, double v1,
                                               double v2, int nb1, int nb2) {
  double d = (c1 - c2) * area * mt * dt;
  if (d / v1 > c1 / (double)nb1) d = c1 * v1 / (double)nb1;
  if (-d / v2 > c2 / (double)nb2) d = -c2 * v2 / (double)nb2;
  return d;
}

// One tile of the flat rows per wave.  A row lists every segment in reach,
// of which a few are bonded: per window of 64 entries each lane compares the
// hashed bonds of its entry's two segments (16 bytes of the neighbor's
// SegNear), the pairs that may be bonded queue up in LDS in entry order, and
// 64 at a time they compare the bond tables themselves and form the fluxes;
// the owners (the first lanes) add their runs of terms in row order.  Bound
// by the latency of a wave's few dependent loads: 100,003 segments 24 us
// against 105 with one lane walking each row through whole bond tables.
constexpr int kXQueue = 2 * 64;
struct XWave {
  unsigned long long bonds[64];  // the owners' SegNear fields
  uint32_t self[64];
  int32_t qu[kXQueue], qo[kXQueue];  // pairs that may be bonded
  double term[3][64];
};

__global__ __launch_bounds__(64) void k_exchange_rows(
    const double4 *__restrict__ pos, const SegNear *__restrict__ near,
    const Topo *__restrict__ topo, FlatRows flat, int32_t maxn,
    const int32_t *__restrict__ ncnt, int64_t n, double *__restrict__ state,
    double mtA, double mtB, double mtC, double dt) {
  __shared__ XWave w;
  const int lane = threadIdx.x;
  const int64_t tile = blockIdx.x;
  const int64_t t0 = tile * flat.tile, t = t0 + lane;
  const bool active = lane < flat.tile && t < n;
  const int64_t B = t0 * maxn;
  const int T = flat.tot[tile];
  const int c = active ? ncnt[t] & ((1 << 28) - 1) : 0;  // bits 28..30: image axes
  const int P = wave_incl_scan64(c) - c;
  bool seg = false;
  w.bonds[lane] = 0;
  w.self[lane] = 0;
  if (active) {
    const SegNear *q = near + t;
    seg = q->type == rec::FUNGI;
    w.bonds[lane] = q->bonds;  // no bonds: 0, in no pair below
    w.self[lane] = q->self;
  }
  wave_lds_sync();
  const unsigned long long below = (1ull << lane) - 1ull;
  double ia = 0.0, ib = 0.0, ic = 0.0;  // initExchange
  int a_lo = 0, a_hi = 0, queued = 0, passed = 0;
  for (int w0 = 0;;) {
    if (w0 < T) {
      const int e = w0 + lane;
      bool hit = false;
      int u = 0, o = 0;
      if (e < T) {
        u = flat.cidx[B + e];
        o = flat.cown[B + e];
        const SegNear *q = near + u;
        hit = q->type == rec::FUNGI && may_bond(w.bonds[o], q->self) &&
              may_bond(q->bonds, w.self[o]);
      }
      const unsigned long long b = __ballot(hit);
      if (hit) {
        const int k = queued - passed + __popcll(b & below);
        w.qu[k] = u;
        w.qo[k] = o;
      }
      const int lo = P > w0 ? P - w0 : 0, hi = P + c < w0 + 64 ? P + c - w0 : 64;
      if (lo < hi) {
        if (P >= w0) a_lo = queued + __popcll(b & ((1ull << lo) - 1ull));
        a_hi = queued + __popcll(hi == 64 ? b : b & ((1ull << hi) - 1ull));
      }
      queued += __popcll(b);
      wave_lds_sync();
      w0 += 64;
    }
    const bool last = w0 >= T;
    while (queued - passed >= 64 || (last && queued > passed)) {
      const int m = queued - passed < 64 ? queued - passed : 64;
      double da = 0.0, db = 0.0, dc = 0.0;
      if (lane < m) {
        const int64_t u = w.qu[lane], ti_ = t0 + w.qo[lane];
        const Topo ti = topo[ti_], tj = topo[u];
        bool bi = false, bj = false;
#pragma unroll
        for (int k = 0; k < 4; k++) {
          bi = bi || (k < ti.n_bnds && ti.seg_id[k] == tj.self_id &&
                      ti.seg_cpu[k] == tj.self_cpu);
          bj = bj || (k < tj.n_bnds && tj.seg_id[k] == ti.self_id &&
                      tj.seg_cpu[k] == ti.self_cpu);
        }
        if (bi && bj) {
          const double r1 = pos[ti_].w, r2 = pos[u].w;
          const double4 c1 = *reinterpret_cast<const double4 *>(state + ti_ * chem::stride);
          const double4 c2 = *reinterpret_cast<const double4 *>(state + u * chem::stride);
          const double area1 = kPi * r1 * r1, area2 = kPi * r2 * r2;
          const double area = 0.5 * (area1 + area2);
          da = species_flux(c1.x, c2.x, area, mtA, dt, c1.w, c2.w, ti.n_bnds, tj.n_bnds) / c1.w;
          db = species_flux(c1.y, c2.y, area, mtB, dt, c1.w, c2.w, ti.n_bnds, tj.n_bnds) / c1.w;
          dc = species_flux(c1.z, c2.z, area, mtC, dt, c1.w, c2.w, ti.n_bnds, tj.n_bnds) / c1.w;
        }
      }
      // (a pair that only looked bonded leaves zeros)
      w.term[0][lane] = da;
      w.term[1][lane] = db;
      w.term[2][lane] = dc;
      // the queue's later entries move to the front
      const int left = queued - passed - m;
      const int mu = lane < left ? w.qu[64 + lane] : 0;
      const int mo = lane < left ? w.qo[64 + lane] : 0;
      wave_lds_sync();
      if (lane < left) {
        w.qu[lane] = mu;
        w.qo[lane] = mo;
      }
      const int k1 = a_hi < passed + m ? a_hi - passed : m;
      for (int k = a_lo > passed ? a_lo - passed : 0; k < k1; k++) {
        ia -= w.term[0][k];
        ib -= w.term[1][k];
        ic -= w.term[2][k];
      }
      passed += m;
      wave_lds_sync();
    }
    if (last) break;
  }
  if (active && seg) {
    double *inc = state + t * chem::stride;
    inc[chem::dA] = ia;
    inc[chem::dB] = ib;
    inc[chem::dC] = ic;
  }
}

// applyIncrements (bmx_chem_K.H:2092-2112)
__global__ void k_exchange_apply(const int32_t *__restrict__ type, int64_t n,
                                 double *__restrict__ state) {
  int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= n || type[t] != rec::FUNGI) return;
  double *q = state + t * chem::stride;
  q[chem::A] += q[chem::dA];
  q[chem::B] += q[chem::dB];
  q[chem::C] += q[chem::dC];
}

int grid256(int64_t n) { return (int)((n + 255) / 256 > 0 ? (n + 255) / 256 : 1); }

}  // namespace

hipError_t launch_chem_unpack(const uint8_t *aos, AosLayout lay, int64_t n,
                              int has_rel, const int32_t *oid, double *state,
                              hipStream_t s) {
  if (n <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_chem_unpack, dim3(grid256(n)), dim3(256), 0, s, aos, lay,
                     n, has_rel, oid, state);
  return hipGetLastError();
}

hipError_t launch_chem_pack(uint8_t *aos, AosLayout lay, int64_t n,
                            int has_rel, const double *state,
                            const int32_t *oid, const int32_t *type,
                            const double4 *pos, const double4 *rod,
                            hipStream_t s) {
  if (n <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_chem_pack, dim3(grid256(n)), dim3(256), 0, s, aos, lay,
                     n, has_rel, state, oid, type, pos, rod);
  return hipGetLastError();
}

hipError_t launch_exchange(const double4 *pos, const int32_t *type,
                           const SegNear *near, const Topo *topo, FlatRows flat,
                           int32_t maxn, const int32_t *ncnt, int64_t n,
                           double *state, const double xpar[3], double dt,
                           hipStream_t s) {
  if (n <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_exchange_rows, dim3(tile_count(n, flat.tile)), dim3(64), 0,
                     s, pos, near, topo, flat, maxn, ncnt, n, state, xpar[0],
                     xpar[1], xpar[2], dt);
  hipLaunchKernelGGL(k_exchange_apply, dim3(grid256(n)), dim3(256), 0, s, type,
                     n, state);
  return hipGetLastError();
}

}  // namespace bmx
