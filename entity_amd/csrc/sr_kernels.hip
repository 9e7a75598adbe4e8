// sr_kernels.hip -- kernel-level SR pusher and current deposit over an
// arbitrary (unsorted) particle range, reading E/B from HBM and accumulating J
// at the reference's ghost-extended indices: per workgroup in an LDS window of
// doubles over the particles that are spatially close (then one FP32 atomic
// per touched entry), the others with FP32 atomics straight into J.
//
// These are the drop-ins for kernel::sr::Pusher_kernel and
// kernel::DepositCurrents_kernel; the fused, tile-windowed push+deposit of
// the engine step lives in push_deposit.hip.
#include "sr_particle.hpp"

#include <climits>

namespace ntt {
namespace {

constexpr int kBlock = 256;

struct PushArgs {
  ParticleView P;
  GlobalEM     F;
  int32_t      ngh, N[3];
  float        ndth, dt, dxm;
  PrtlBCs      bc;
  uint32_t*    err;
};

// state of particle k of the workgroup whose first particle is `base` (a
// uniform base and a 32-bit offset)
template <int D>
__device__ __forceinline__ void load_pushed(const ParticleView& P, int64_t base, uint32_t k,
                                            PState& s) {
  s.i[0] = (P.i1 + base)[k];
  s.i[1] = (P.i2 + base)[k];
  if constexpr (D == 3) s.i[2] = (P.i3 + base)[k];
  s.dx[0] = (P.dx1 + base)[k];
  s.dx[1] = (P.dx2 + base)[k];
  if constexpr (D == 3) s.dx[2] = (P.dx3 + base)[k];
  s.u[0] = (P.ux1 + base)[k];
  s.u[1] = (P.ux2 + base)[k];
  s.u[2] = (P.ux3 + base)[k];
}

template <int D>
__device__ __forceinline__ void store_pushed(const ParticleView& P, int64_t base, uint32_t k,
                                             const PState& s, int16_t tag) {
  (P.i1p + base)[k]  = s.ip[0];
  (P.dx1p + base)[k] = s.dxp[0];
  (P.i1 + base)[k]   = s.i[0];
  (P.dx1 + base)[k]  = s.dx[0];
  (P.i2p + base)[k]  = s.ip[1];
  (P.dx2p + base)[k] = s.dxp[1];
  (P.i2 + base)[k]   = s.i[1];
  (P.dx2 + base)[k]  = s.dx[1];
  if constexpr (D == 3) {
    (P.i3p + base)[k]  = s.ip[2];
    (P.dx3p + base)[k] = s.dxp[2];
    (P.i3 + base)[k]   = s.i[2];
    (P.dx3 + base)[k]  = s.dx[2];
  }
  (P.ux1 + base)[k] = s.u[0];
  (P.ux2 + base)[k] = s.u[1];
  (P.ux3 + base)[k] = s.u[2];
  if (s.tag != tag) (P.tag + base)[k] = s.tag;
}

// whether the gather of a particle at its cell and offsets stays in the
// arrays (offsets outside [0, 1], or NaN, would move the order-0 stencil)
template <int D, int O>
__device__ __forceinline__ bool gather_in_array(const PushArgs& a, const PState& s) {
  int lo, hi;
  interp_reach<O>(lo, hi);
  bool ok = true;
#pragma unroll
  for (int d = 0; d < D; ++d) {
    const int g = s.i[d] + a.ngh;
    if (g + lo < 0 || g + hi >= a.N[d] || !(s.dx[d] >= ZERO && s.dx[d] <= ONE)) ok = false;
  }
  return ok;
}

// One particle per thread.  Bound by the gather's loads through the caches
// (162 values per particle in 3D at order 2, a stencil row of 3 in one load):
// issued a component at a time (GlobalEMAhead), 1.7e7 particles in tile order on
// 128 x 128 x 64 cells take 0.81 ms (1.03 ms on average between re-sorts 4 steps
// apart; 1.56 ms with the compiler's own order, which waits for every row), 512
// x 512 cells at order 2 81 us (115).  139 registers, three wavefronts per SIMD:
// held to 128 or 96 registers it spills and takes 0.94 and 1.17 ms.
template <int D, int O, int ALG>
__global__ __launch_bounds__(kBlock) void k_sr_push(PushArgs a) {
  const int64_t  base = static_cast<int64_t>(blockIdx.x) * kBlock;
  const uint32_t k    = threadIdx.x;
  if (base + k >= a.P.n) return;
  const int16_t tag = (a.P.tag + base)[k];
  if (tag != NTT_TAG_ALIVE) {
    if (tag != NTT_TAG_DEAD) raise_device_error(a.err, NTT_DEVERR_INVALID_TAG);
    return;
  }
  PState s;
  s.tag = tag;
  load_pushed<D>(a.P, base, k, s);
  if constexpr (ALG != ALG_PHOTON) {
    if (!gather_in_array<D, O>(a, s)) {
      raise_device_error(a.err, NTT_DEVERR_OUT_OF_BOUNDS);
      return;
    }
  }
  sr_update<D, O, ALG>(GlobalEMAhead{ a.F }, a.ngh, a.ndth, a.dt, a.dxm, a.bc, s);
  store_pushed<D>(a.P, base, k, s, tag);
}

// J sink: hardware float atomics into the ghost-extended current array
struct GlobalJ {
  float*  d;
  int32_t N1, N2;
  int64_t cstride;
  int     i0 = 0, j0 = 0, k0 = 0;
  __device__ __forceinline__ void set_origin(int i, int j, int k) {
    i0 = i;
    j0 = j;
    k0 = k;
  }
  __device__ __forceinline__ void add_rel(int a, int b, int g, int c, float v) {
    add(i0 + a, j0 + b, k0 + g, c, v);
  }
  __device__ __forceinline__ void add(int i, int j, int k, int c, float v) {
    unsafeAtomicAdd(d + static_cast<int64_t>(i) +
                      static_cast<int64_t>(N1) * (static_cast<int64_t>(j) + static_cast<int64_t>(N2) * k) +
                      cstride * c,
                    v);
  }
};

struct DepositArgs {
  ParticleView P;
  GlobalJ      J;
  int32_t      ngh, N[3];
  float        charge, inv_dt;
  uint32_t*    err;
};

// Deposit of kDepThreads consecutive particles by one workgroup into an LDS
// window of doubles, which is then added to J with one FP32 atomic per non-zero
// entry.
//
// The window is placed over the workgroup's particles, or, where they do not
// fit one (a tile at the periodic boundary, whose wrapped particles deposit on
// the far side of the array; a workgroup that straddles rows of tiles), over
// those near the sample that most of the wavefronts' first particles are near.
// The particles it leaves out, and all of them where such a window would take
// fewer than kDepMin (its clearing and flush would cost more), are added to J
// directly.
//
// Every single-precision contribution of a particle in the window enters its
// sum as it is, whatever the other particles' weights; the sum is rounded once.
// (Sums of 32-bit fixed point in units of the heaviest particle's contribution,
// ds_add_u64 for ds_add_f64, took 0.86 instead of 1.04 ms at the size below, but
// lost what is small beside that particle: an error of 2.6e-4 in the J3 of a
// plasma of |u| = 1e-4, against 3e-8 with FP32 sums throughout.)
//
// In 3D (orders 1, 2) the accepted particles are reordered through an LDS
// list, as in the step's deposit (push_deposit.hip): particles whose stencil
// keeps its cells first (54 slots without per-slot branches at order 2), the
// others by the direction they shift along, each rank-major by bank class.
//
// Measured on 128 x 128 x 64 cells, 1.7e7 particles, order 2: 1.04 ms in tile
// order and 1.30 ms four steps after it was made, with equal weights or weights
// over four decades alike.  Giving the window up where a workgroup's box does not
// fit it, every particle added by its own lane's FP32 atomics, took 9.3 and
// 10.0 ms (the tiles at the periodic boundary).  In no order: 20 ms against 48.
// 512 x 512 cells, 4.2e6 particles, order 1: 74 and 83 us, against 135 and 205.
// kDepMin from 8 to 256: within 1% at 128 x 128 x 64 and 350 x 250 cells.
constexpr int kDepThreads = 512;
constexpr int kDepMin     = 64;

// LDS window (cells per dimension): 24.6 KB in 2D, 33.6 KB in 3D
template <int D> struct DepWin;
template <> struct DepWin<2> { static constexpr int W[3] = { 64, 16, 1 }; };
template <> struct DepWin<3> { static constexpr int W[3] = { 14, 10, 10 }; };

// window sink
template <int D>
struct LdsJd {
  static constexpr int W1 = DepWin<D>::W[0], W2 = DepWin<D>::W[1], WC = W1 * W2 * DepWin<D>::W[2];
  double* w;
  int     o1, o2, o3;
  int     base = 0;
  __device__ __forceinline__ int index(int i, int j, int k) const {
    return (i - o1) + W1 * ((j - o2) + W2 * (k - o3));
  }
  __device__ __forceinline__ void set_origin(int i, int j, int k) { base = index(i, j, k); }
  __device__ __forceinline__ void add_rel(int a, int b, int g, int c, float v) {
    atomicAdd(w + c * WC + base + a + W1 * (b + W2 * g), static_cast<double>(v));
  }
  __device__ __forceinline__ void add(int i, int j, int k, int c, float v) {
    atomicAdd(w + c * WC + index(i, j, k), static_cast<double>(v));
  }
};

template <bool MAX>
__device__ __forceinline__ int wave_reduce(int v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v = MAX ? max(v, __shfl_xor(v, o)) : min(v, __shfl_xor(v, o));
  return v;
}

// A particle of the deposit: its cells, offsets, charge
// coefficient and (2D) out-of-plane velocity.
template <int D>
struct DepParticle {
  int   i[D], ip[D];
  float x[D], xp[D];
  float coeff, vz;
};

// Loads particle p; false for dead ones and for those whose stencil leaves the
// ghost-extended array (reported and skipped).
template <int D, int O>
__device__ __forceinline__ bool load_deposit(const DepositArgs& a, int64_t base, uint32_t k,
                                             DepParticle<D>& q) {
  // the workgroup's first particle (uniform) plus a 32-bit offset
  auto at = [&](auto* v) { return (v + base)[k]; };
  if (base + k >= a.P.n || at(a.P.tag) == NTT_TAG_DEAD) return false;
  const int32_t* i[3]  = { a.P.i1, a.P.i2, a.P.i3 };
  const int32_t* ip[3] = { a.P.i1p, a.P.i2p, a.P.i3p };
  const float*   x[3]  = { a.P.dx1, a.P.dx2, a.P.dx3 };
  const float*   xp[3] = { a.P.dx1p, a.P.dx2p, a.P.dx3p };
  bool ok = true;
#pragma unroll
  for (int d = 0; d < D; ++d) {
    q.i[d]  = at(i[d]);
    q.ip[d] = at(ip[d]);
    q.x[d]  = at(x[d]);
    q.xp[d] = at(xp[d]);
  }
  q.coeff = at(a.P.w) * a.charge;
  q.vz    = ZERO;
  if constexpr (D == 2) {
    const float u[3] = { at(a.P.ux1), at(a.P.ux2), at(a.P.ux3) };
    q.vz = vp_out_of_plane(u);
  }
#pragma unroll
  for (int d = 0; d < D; ++d) {
    int lo, hi;
    deposit_extent<O>(q.i[d], q.x[d], q.ip[d], q.xp[d], lo, hi);
    if (lo + a.ngh < 0 || hi + a.ngh >= a.N[d]) ok = false;
  }
  if (!ok) raise_device_error(a.err, NTT_DEVERR_OUT_OF_BOUNDS);
  return ok;
}

template <int D, int O, class Sink>
__device__ __forceinline__ void deposit_one(Sink& J, int G, const DepParticle<D>& q,
                                            float inv_dt) {
  PState s;
#pragma unroll
  for (int d = 0; d < D; ++d) {
    s.i[d]   = q.i[d];
    s.ip[d]  = q.ip[d];
    s.dx[d]  = q.x[d];
    s.dxp[d] = q.xp[d];
  }
  if constexpr (O == 0) deposit_zigzag<D>(J, G, s, q.vz, q.coeff, inv_dt);
  else if constexpr (D == 2) deposit_esirkepov_2d<O>(J, G, s, q.vz, q.coeff, inv_dt);
  else deposit_esirkepov_3d<O>(J, G, s, q.coeff, inv_dt);
}

// value of lane l (uniform) in every lane
__device__ __forceinline__ int lane_value(int v, int l) { return __builtin_amdgcn_readlane(v, l); }
__device__ __forceinline__ float lane_value(float v, int l) {
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), l));
}

// entry s of v, s differing between the lanes (starting from zero, not v[0]: a
// choice between two entries becomes one of addresses, and v goes to scratch)
template <int M>
__device__ __forceinline__ float entry(const float (&v)[M], int s) {
  float r = ZERO;
#pragma unroll
  for (int k = 0; k < M; ++k) r = s == k ? v[k] : r;
  return r;
}

// The 3D Esirkepov deposit (O = 1, 2) of one particle, the same for the whole
// wavefront, straight into J: lane a + 4 b + 16 g takes stencil slot (a, b, g)
// of the three components.  Shapes, longitudinal coefficients and products are
// those of deposit_esirkepov_3d.
template <int O>
__device__ __forceinline__ void deposit_wave(const GlobalJ& J, int G, const DepParticle<3>& q,
                                             float inv_dt) {
  constexpr int M = O + 2;
  const int   lane = threadIdx.x & 63;
  const int   s[3] = { lane & 3, (lane >> 2) & 3, lane >> 4 };
  const float q3   = -(q.coeff * inv_dt) * THIRD;
  int         m[3], n[3];
  float       iS[3], fS[3], C[3];
  bool        in = true;
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    int   a, b;
    float Si[O + 1], Sf[O + 1], i[M], f[M], c[O + 1];
    shape_order<false, O, true>(q.ip[d], q.xp[d], a, Si);
    shape_order<false, O, true>(q.i[d], q.x[d], b, Sf);
    // for_deposit, with selects: the shape that starts further up begins at slot 1
#pragma unroll
    for (int k = 0; k < M; ++k) {
      i[k] = f[k] = ZERO;
      if (k <= O) {
        i[k] = a > b ? ZERO : Si[k];
        f[k] = b > a ? ZERO : Sf[k];
      }
      if (k > 0) {
        i[k] = a > b ? Si[k - 1] : i[k];
        f[k] = b > a ? Sf[k - 1] : f[k];
      }
    }
    m[d] = min(a, b);
    n[d] = (a == b) ? O : O + 1;
    in   = in && s[d] <= n[d];
    c[0] = q3 * (f[0] - i[0]);
#pragma unroll
    for (int k = 1; k <= O; ++k) c[k] = fmaf(q3, f[k] - i[k], c[k - 1]);
    iS[d] = entry(i, s[d]);
    fS[d] = entry(f, s[d]);
    C[d]  = entry(c, s[d]);
  }
  if (!in) return;
  GlobalJ w = J;
  w.set_origin(m[0] + G, m[1] + G, m[2] + G);
  float P[3], Q[3];
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    P[d] = fmaf(HALF, fS[d], iS[d]);
    Q[d] = fmaf(HALF, iS[d], fS[d]);
  }
  if (s[0] < n[0]) w.add_rel(s[0], s[1], s[2], 0, C[0] * fmaf(P[1], iS[2], Q[1] * fS[2]));
  if (s[1] < n[1]) w.add_rel(s[0], s[1], s[2], 1, C[1] * fmaf(P[0], iS[2], Q[0] * fS[2]));
  if (s[2] < n[2]) w.add_rel(s[0], s[1], s[2], 2, C[2] * fmaf(P[0], iS[1], Q[0] * fS[1]));
}

// A particle of the 3D list: cells relative to the window (5 bits and the
// move's 2 bits per direction), offsets after and before, coefficient.
struct DepListed {
  uint4 a, b;
};
constexpr int kDepRanks = 32, kDepCrossRanks = 8;
constexpr int kDepGroups = kDepRanks + 4 * kDepCrossRanks;
static_assert(kDepGroups == 64, "one wavefront scans the groups");

// Deposits the workgroup's accepted particles (one per thread) into the
// window through the list.  The caller has cleared the window, ctr and gsz and
// passed a barrier.
template <int O>
__device__ __forceinline__ void deposit_listed(LdsJd<3>& jw, const int* org, int G, bool live,
                                               const DepParticle<3>& q, float inv_dt,
                                               DepListed* list, uint32_t (*ctr)[32],
                                               uint32_t* gsz, uint32_t* gpos, uint32_t* counts) {
  const int tid = threadIdx.x, lane = tid & 63;
  uint32_t  cells = 0u;
  int       grp = 0;
  if (live) {
    uint32_t shift = 0u;
    int      slot = 0, stride = 1;
#pragma unroll
    for (int d = 0; d < 3; ++d) {
      int lo, hi;
      deposit_extent<O>(q.i[d], q.x[d], q.ip[d], q.xp[d], lo, hi);
      if (!deposit_stays<O>(q.i[d], q.x[d], q.ip[d], q.xp[d])) shift |= 1u << d;
      slot += (lo - org[d]) * stride;
      stride *= DepWin<3>::W[d];
      cells |= (static_cast<uint32_t>(q.i[d] - org[d]) |
                (static_cast<uint32_t>(q.ip[d] - q.i[d] + 1) << 5)) << (7 * d);
    }
    // 0: stays; 1, 2, 3: shifts along x, y, z only; 4: along several
    const int cls = shift == 0u ? 0 : (shift == 1u ? 1 : (shift == 2u ? 2 : (shift == 4u ? 3 : 4)));
    const uint32_t rank = atomicAdd(&ctr[cls][slot & 31], 1u);
    grp = cls == 0 ? static_cast<int>(min(rank, static_cast<uint32_t>(kDepRanks - 1)))
                   : kDepRanks + (cls - 1) * kDepCrossRanks +
                       static_cast<int>(min(rank, static_cast<uint32_t>(kDepCrossRanks - 1)));
    atomicAdd(&gsz[grp], 1u);
  }
  __syncthreads();
  if (tid < kDepGroups) {
    const uint32_t v = gsz[tid];
    uint32_t       incl = v;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const uint32_t t = __shfl_up(incl, o);
      if (lane >= o) incl += t;
    }
    gpos[tid] = incl - v;
    if (tid == kDepRanks - 1) counts[0] = incl;
    if (tid == kDepGroups - 1) counts[1] = incl;
  }
  __syncthreads();
  if (live) {
    DepListed e;
    e.a = make_uint4(cells, __float_as_uint(q.x[0]), __float_as_uint(q.x[1]),
                     __float_as_uint(q.x[2]));
    e.b = make_uint4(__float_as_uint(q.xp[0]), __float_as_uint(q.xp[1]),
                     __float_as_uint(q.xp[2]), __float_as_uint(q.coeff));
    list[atomicAdd(&gpos[grp], 1u)] = e;
  }
  __syncthreads();
  const int ns = static_cast<int>(counts[0]), nall = static_cast<int>(counts[1]);
  if (tid < nall) {
    const DepListed e = list[tid];
    PState          s;
#pragma unroll
    for (int d = 0; d < 3; ++d) {
      const uint32_t v = e.a.x >> (7 * d);
      s.i[d]  = static_cast<int>(v & 31u) + org[d];
      s.ip[d] = s.i[d] + static_cast<int>((v >> 5) & 3u) - 1;
    }
    s.dx[0]  = __uint_as_float(e.a.y);
    s.dx[1]  = __uint_as_float(e.a.z);
    s.dx[2]  = __uint_as_float(e.a.w);
    s.dxp[0] = __uint_as_float(e.b.x);
    s.dxp[1] = __uint_as_float(e.b.y);
    s.dxp[2] = __uint_as_float(e.b.z);
    const float coeff = __uint_as_float(e.b.w);
    if (tid < ns) deposit_esirkepov_3d_stay<O>(jw, G, s, coeff, inv_dt);
    else deposit_esirkepov_3d<O>(jw, G, s, coeff, inv_dt);
  }
}

template <int D, int O>
__global__ __launch_bounds__(kDepThreads) __attribute__((amdgpu_waves_per_eu(D == 3 && O > 0 ? 6 : 4)))
void k_deposit(DepositArgs a) {
  constexpr bool LIST = D == 3 && O > 0;
  constexpr int  W1 = DepWin<D>::W[0], W2 = DepWin<D>::W[1], W3 = DepWin<D>::W[2];
  constexpr int  WC = W1 * W2 * W3;
  constexpr int  kWaves = kDepThreads / 64;
  __shared__ double    jw[3 * WC];
  __shared__ int       red[2 * D + 1][kWaves];
  __shared__ int       smp[kWaves][4];  // a particle of each wavefront: stencil start, valid
  __shared__ int       best, taken;
  __shared__ DepListed list[LIST ? kDepThreads : 1];
  __shared__ uint32_t  ctr[LIST ? 5 : 1][32], gsz[LIST ? 64 : 1], gpos[LIST ? 64 : 1], counts[2];
  const int     tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  const int     G   = a.ngh;
  DepParticle<D> q;
  const bool     live =
    load_deposit<D, O>(a, static_cast<int64_t>(blockIdx.x) * kDepThreads, tid, q);
  int lo[3] = { 0, 0, 0 }, hi[3] = { 0, 0, 0 };
  if (live)
#pragma unroll
    for (int d = 0; d < D; ++d) deposit_extent<O>(q.i[d], q.x[d], q.ip[d], q.xp[d], lo[d], hi[d]);
  // a listed particle's move is held in two bits per direction
  bool want = live;
  if constexpr (LIST)
#pragma unroll
    for (int d = 0; d < D; ++d) want = want && abs(q.ip[d] - q.i[d]) <= 1;
  // over the workgroup (uniform): the box of the particles that are `in`, and
  // whether every live one is
  auto box = [&](bool in, int* l, int* h) -> bool {
#pragma unroll
    for (int d = 0; d < D; ++d) {
      const int bl = wave_reduce<false>(in ? lo[d] : INT_MAX);
      const int bh = wave_reduce<true>(in ? hi[d] : INT_MIN);
      if (lane == 0) {
        red[2 * d][wv]     = bl;
        red[2 * d + 1][wv] = bh;
      }
    }
    const bool all = __ballot(live && !in) == 0ull;
    if (lane == 0) red[2 * D][wv] = all;
    __syncthreads();
#pragma unroll
    for (int d = 0; d < D; ++d) {
      int bl = red[2 * d][0], bh = red[2 * d + 1][0];
#pragma unroll
      for (int w = 1; w < kWaves; ++w) {
        bl = min(bl, red[2 * d][w]);
        bh = max(bh, red[2 * d + 1][w]);
      }
      l[d] = __builtin_amdgcn_readfirstlane(bl);  // uniform: scalar registers
      h[d] = __builtin_amdgcn_readfirstlane(bh);
    }
    int every = red[2 * D][0];
#pragma unroll
    for (int w = 1; w < kWaves; ++w) every &= red[2 * D][w];
    return __builtin_amdgcn_readfirstlane(every) != 0;
  };
  if (tid == 0) best = taken = 0;
  for (int k = tid; k < 3 * WC; k += kDepThreads) jw[k] = 0.0;
  if constexpr (LIST)
    if (tid < 160 + kDepGroups) {
      if (tid < 160) ctr[tid >> 5][tid & 31] = 0u;
      else gsz[tid - 160] = 0u;
    }
  int  org[3] = { 0, 0, 0 }, top[3] = { 0, 0, 0 };
  bool fits = box(want, org, top);
  const bool empty = org[0] > top[0];  // nothing for the window
  fits = fits && !empty;
#pragma unroll
  for (int d = 0; d < D; ++d)
    fits = fits && static_cast<int64_t>(top[d]) - org[d] < DepWin<D>::W[d];
  if (!fits && !empty) {
    const uint64_t b = __ballot(want);
    if (lane == 0) smp[wv][3] = b != 0ull;
    if (b != 0ull && lane == __ffsll(static_cast<unsigned long long>(b)) - 1)
#pragma unroll
      for (int d = 0; d < D; ++d) smp[wv][d] = lo[d];
    __syncthreads();
    auto near_sample = [&](const int* x, int w) {
      bool in = true;
#pragma unroll
      for (int d = 0; d < D; ++d) in = in && abs(x[d] - smp[w][d]) < DepWin<D>::W[d];
      return in;
    };
    if (tid < kWaves && smp[tid][3]) {
      int n = 0;
      for (int w = 0; w < kWaves; ++w) n += smp[w][3] && near_sample(smp[tid], w);
      atomicMax(&best, n * kWaves + tid);
    }
    __syncthreads();
    const int ref = __builtin_amdgcn_readfirstlane(best) % kWaves;
    box(want && near_sample(lo, ref), org, top);
    // a box wider than the window: from a quarter window below the sample
#pragma unroll
    for (int d = 0; d < D; ++d)
      if (top[d] - org[d] >= DepWin<D>::W[d])
        org[d] = __builtin_amdgcn_readfirstlane(
          max(org[d], smp[ref][d] - DepWin<D>::W[d] / 4));
  }
  // the particles the window takes
  bool in = want;
#pragma unroll
  for (int d = 0; d < D; ++d) in = in && lo[d] >= org[d] && hi[d] < org[d] + DepWin<D>::W[d];
  const uint64_t out = __ballot(live && !in);
  {
    const uint64_t b = __ballot(in);
    if (lane == 0 && b != 0ull) atomicAdd(&taken, __popcll(b));
  }
  __syncthreads();
  const bool window = fits || __builtin_amdgcn_readfirstlane(taken) >= kDepMin;
  uint64_t   direct = window ? out : __ballot(live);
  if constexpr (LIST) {
#pragma unroll 1
    while (direct != 0ull) {
      const int l = __ffsll(static_cast<unsigned long long>(direct)) - 1;
      direct &= direct - 1;
      DepParticle<D> s;
#pragma unroll
      for (int d = 0; d < D; ++d) {
        s.i[d]  = lane_value(q.i[d], l);
        s.ip[d] = lane_value(q.ip[d], l);
        s.x[d]  = lane_value(q.x[d], l);
        s.xp[d] = lane_value(q.xp[d], l);
      }
      s.coeff = lane_value(q.coeff, l);
      deposit_wave<O>(a.J, G, s, a.inv_dt);
    }
  } else {
    if ((direct >> lane) & 1ull) {
      GlobalJ J = a.J;
      deposit_one<D, O>(J, G, q, a.inv_dt);
    }
  }
  if (!window) return;
  LdsJd<D> J{ jw, org[0] + G, org[1] + G, D == 3 ? org[2] + G : 0 };
  if constexpr (LIST) deposit_listed<O>(J, org, G, in, q, a.inv_dt, list, ctr, gsz, gpos, counts);
  else if (in) deposit_one<D, O>(J, G, q, a.inv_dt);
  __syncthreads();
  const int e1 = min(top[0] - org[0] + 1, W1), e2 = min(top[1] - org[1] + 1, W2);
  const int rows = (D == 3 ? min(top[2] - org[2] + 1, W3) : 1) * (W1 * W2);
  for (int e = tid; e < rows; e += kDepThreads) {
    const int z = e / (W1 * W2), t = e - z * (W1 * W2);
    const int y = t / W1, x = t - y * W1;
    if (x < e1 && y < e2) {
#pragma unroll
      for (int c = 0; c < 3; ++c) {
        const double v = jw[c * WC + e];
        if (v != 0.0)
          a.J.add(org[0] + G + x, org[1] + G + y, D == 3 ? org[2] + G + z : 0, c,
                  static_cast<float>(v));
      }
    }
  }
}

template <int D, int O, int ALG>
void launch_push(const PushArgs& a, hipStream_t st) {
  k_sr_push<D, O, ALG><<<grid_for(a.P.n, kBlock), kBlock, 0, st>>>(a);
}

template <int D, int ALG>
void launch_push_o(int order, const PushArgs& a, hipStream_t st) {
  if (order == 0) launch_push<D, 0, ALG>(a, st);
  else if (order == 1) launch_push<D, 1, ALG>(a, st);
  else launch_push<D, 2, ALG>(a, st);
}

}  // namespace

// Shared validation of pusher inputs, also used by the engine step.
ntt_status prepare_push(const ntt_sr_pusher_ctx_t* ctx, const ntt_prtl_bc_t* bc,
                        const ntt_particles_t* prtls, const ntt_field_t* em,
                        const ntt_minkowski_t* metric, int32_t shape_order, int* alg_out,
                        ParticleView* pv, FieldView* fv, PrtlBCs* bcs, float* ndth) {
  if (ctx == nullptr || bc == nullptr || metric == nullptr) return NTT_ERR_ARG;
  if (shape_order < 0 || shape_order > 2) return NTT_ERR_UNSUPPORTED;
  ntt_status s = make_field_view(em, 6, fv);
  if (s != NTT_OK) return s;
  const int D = em->dim;
  if (metric->dim != D || !(metric->dx > 0.0f)) return NTT_ERR_ARG;
  if (fv->ngh < 2) return NTT_ERR_ARG;
  const uint8_t fl = ctx->pusher_flags;
  if (fl == NTT_PUSHER_NONE) return NTT_ERR_ARG;  // "No particle pusher specified"
  if (fl & NTT_PUSHER_GCA) return NTT_ERR_UNSUPPORTED;
  int alg;
  if (fl == NTT_PUSHER_PHOTON) alg = ALG_PHOTON;
  else if (fl & NTT_PUSHER_BORIS) alg = ALG_BORIS;
  else if (fl & NTT_PUSHER_VAY) alg = ALG_VAY;
  else return NTT_ERR_ARG;
  if (alg != ALG_PHOTON && !(ctx->mass != 0.0f)) return NTT_ERR_ARG;
  s = make_particle_view(prtls, D, true, pv);
  if (s != NTT_OK) return s;
  const int ni[3] = { ctx->ni1, ctx->ni2, ctx->ni3 };
  const int na[3] = { fv->n1, fv->n2, fv->n3 };
  for (int d = 0; d < D; ++d) {
    if (ni[d] != na[d]) return NTT_ERR_ARG;
    for (int e = 0; e < 2; ++e) {
      const uint8_t b = bc->bc[d][e];
      const bool ok = b == NTT_PRTL_BC_PERIODIC || b == NTT_PRTL_BC_ABSORB ||
                      b == NTT_PRTL_BC_ATMOSPHERE || b == NTT_PRTL_BC_REFLECT ||
                      (d == 1 && b == NTT_PRTL_BC_AXIS);
      if (!ok) return NTT_ERR_UNSUPPORTED;
    }
    bcs->lo[d] = bc->bc[d][0];
    bcs->hi[d] = bc->bc[d][1];
    bcs->ni[d] = ni[d];
  }
  for (int d = D; d < 3; ++d) {
    bcs->lo[d] = bcs->hi[d] = 0;
    bcs->ni[d] = 1;
  }
  // normalized_dt_half (sr.hpp:111): HALF * (charge / mass) * omegaB0 * dt
  *ndth = HALF * (ctx->charge / ctx->mass) * ctx->omegaB0 * ctx->dt;
  *alg_out = alg;
  return NTT_OK;
}

ntt_status launch_sr_push(const ParticleView& pv, const FieldView& fv, const PrtlBCs& bcs,
                          int D, int order, int alg, float ndth, float dt, float dxm,
                          hipStream_t st) {
  if (pv.n == 0) return NTT_OK;
  uint32_t* err = device_error_word();
  if (err == nullptr) return NTT_ERR_HIP;
  PushArgs a;
  a.P = pv;
  a.F = GlobalEM{ fv.d, fv.N1, fv.N2, fv.cstride };
  a.ngh = fv.ngh;
  a.N[0] = fv.N1; a.N[1] = fv.N2; a.N[2] = fv.N3;
  a.ndth = ndth; a.dt = dt; a.dxm = dxm;
  a.bc = bcs;
  a.err = err;
  if (D == 2) {
    if (alg == ALG_BORIS) launch_push_o<2, ALG_BORIS>(order, a, st);
    else if (alg == ALG_VAY) launch_push_o<2, ALG_VAY>(order, a, st);
    else launch_push<2, 0, ALG_PHOTON>(a, st);
  } else {
    if (alg == ALG_BORIS) launch_push_o<3, ALG_BORIS>(order, a, st);
    else if (alg == ALG_VAY) launch_push_o<3, ALG_VAY>(order, a, st);
    else launch_push<3, 0, ALG_PHOTON>(a, st);
  }
  return check_launch();
}

ntt_status launch_deposit(const ParticleView& pv, const FieldView& J, int D, int order,
                          float charge, float dt, hipStream_t st) {
  if (pv.n == 0) return NTT_OK;
  uint32_t* err = device_error_word();
  if (err == nullptr) return NTT_ERR_HIP;
  DepositArgs a;
  a.P = pv;
  a.J = GlobalJ{ J.d, J.N1, J.N2, J.cstride };
  a.ngh = J.ngh;
  a.N[0] = J.N1; a.N[1] = J.N2; a.N[2] = J.N3;
  a.charge = charge;
  a.inv_dt = ONE / dt;
  a.err = err;
  const unsigned g = grid_for(pv.n, kDepThreads);
  if (D == 2) {
    if (order == 0) k_deposit<2, 0><<<g, kDepThreads, 0, st>>>(a);
    else if (order == 1) k_deposit<2, 1><<<g, kDepThreads, 0, st>>>(a);
    else k_deposit<2, 2><<<g, kDepThreads, 0, st>>>(a);
  } else {
    if (order == 0) k_deposit<3, 0><<<g, kDepThreads, 0, st>>>(a);
    else if (order == 1) k_deposit<3, 1><<<g, kDepThreads, 0, st>>>(a);
    else k_deposit<3, 2><<<g, kDepThreads, 0, st>>>(a);
  }
  return check_launch();
}

}  // namespace ntt

using namespace ntt;

extern "C" ntt_status ntt_sr_push(const ntt_sr_pusher_ctx_t* ctx, const ntt_prtl_bc_t* bc,
                                  const ntt_particles_t* prtls, const ntt_field_t* em,
                                  const ntt_minkowski_t* metric, int32_t shape_order,
                                  void* stream) {
  ParticleView pv;
  FieldView    fv;
  PrtlBCs      bcs;
  float        ndth;
  int          alg;
  ntt_status s = prepare_push(ctx, bc, prtls, em, metric, shape_order, &alg, &pv, &fv, &bcs, &ndth);
  if (s != NTT_OK) return s;
  return launch_sr_push(pv, fv, bcs, em->dim, shape_order, alg, ndth, ctx->dt, metric->dx,
                        as_stream(stream));
}

extern "C" ntt_status ntt_deposit_currents(const ntt_particles_t* prtls, ntt_field_t* cur,
                                           const ntt_minkowski_t* metric, float charge, float dt,
                                           int32_t shape_order, void* stream) {
  if (metric == nullptr) return NTT_ERR_ARG;
  if (shape_order < 0 || shape_order > 2) return NTT_ERR_UNSUPPORTED;
  FieldView J;
  ntt_status s = make_field_view(cur, 3, &J);
  if (s != NTT_OK) return s;
  if (metric->dim != cur->dim || !(dt > 0.0f)) return NTT_ERR_ARG;
  if (J.ngh < 2) return NTT_ERR_ARG;
  ParticleView pv;
  s = make_particle_view(prtls, cur->dim, cur->dim == 2, &pv);
  if (s != NTT_OK) return s;
  return launch_deposit(pv, J, cur->dim, shape_order, charge, dt, as_stream(stream));
}
