// rsg_resident.hip -- many RSG steps in one launch, for meshes whose state fits the LDS of the
// GPU's compute units.
//
// The two per-step launches cost a mesh of up to a few 100 k cells more in launch latency and
// in dependent memory round trips than in work.  Here one workgroup per tile (a compact box of
// cells, at most one tile per compute unit) keeps the tile's stresses and velocities in LDS
// for all steps.  Per step a tile
//   1. updates the nodes that touch no other tile's cells;
//   2. reads its halo (the other tiles' cells at its nodes) into LDS as the neighbour tiles
//      publish the step before;
//   3. updates its other nodes.  A node of several tiles is updated by each of them, from the
//      same values in the same order, so velocities are never exchanged and a step needs one
//      exchange instead of two;
//   4. updates the cells that other tiles read, publishing each, then the rest.
//
// Exchange across the XCDs' separate L2s: the words are written and read with agent-scope
// relaxed atomics.  The waves that write exported cells wait until their stores are out, and the
// last of them sets the tile's flag to the step; a reader loads a cell's words after it has seen
// the flag of the cell's tile.  The stresses after step g go to buffer g % 2: a tile that has the
// whole halo of step g knows that its neighbours have finished step g and so have read g - 1.
// Each flag has a cache line of its own, which only its readers poll.
//
// What bounds it: up to some 30,000 cells the exchange (store, flag, load: about 1.7 us a step) and
// the dependent latency of two updates; above, the FP64 arithmetic and the LDS reads of a tile
// (24 reads of 16 bytes a node).  Every byte of state stays on the chip, so memory does not.
// Aluminium block of 32,000 cells on an MI355X: 10.7 us a step with the per-step kernels, 5.3 here
// (FP64), 9.9 and 4.3 (FP32).
//
// The workgroups wait for each other, so they must all be on the GPU at once.  There are no more
// of them than compute units, and the host lets one resident launch run at a time, but another
// process or stream may hold part of the GPU.  So a launch first agrees: the last workgroup to
// start decides that the steps are made; one that has waited long decides that they are not, and
// all leave with nothing written.  A kernel of one workgroup follows each launch and makes the
// steps of such a one by itself, slowly, and tells the host not to try again.  (A cooperative
// launch would see to it too, but costs 20 us and the host's wait for it, and on ROCm 7 its queue
// slows the streams created after it: a batch's two lanes took 5.4 ms for 2.0 ms of work.)
#include "rsg_device.h"

namespace rsg {
namespace {

// 100 MHz ticks a wave waits for its neighbours before it gives up (10 s), and a workgroup for
// the others to start (20 ms).
constexpr uint64_t kWaitTicks = 1000000000ull;
constexpr uint64_t kStartTicks = 2000000ull;

// The decision of launch seq is 2 seq + 1 (its steps are made) or 2 seq.
__device__ __forceinline__ bool decided(uint32_t d, uint32_t seq) { return (d >> 1) == (seq & 0x7FFFFFFFu); }

// Whether the launch's steps are made, once decided.  Called by one thread of each workgroup, which
// was the last to start or not.
__device__ __forceinline__ bool agree(uint32_t* decision, uint32_t seq, bool last) {
  uint64_t t0 = 0;
  for (;;) {
    uint32_t d = __hip_atomic_load(decision, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (decided(d, seq)) return d & 1;
    const uint64_t t = wall_clock64();
    if (t0 == 0) t0 = t;
    if (last || t - t0 > kStartTicks)  // the first decision stands
      __hip_atomic_compare_exchange_strong(decision, &d, 2 * seq + (last ? 1u : 0u), __ATOMIC_RELAXED,
                                           __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
}

// Stress components of a slot, in the order node_rates reads them.
__device__ __forceinline__ constexpr int slot_comp(int k) {
  return k == 0 ? 0 : k == 1 ? 5 : k == 2 ? 4 : k == 3 ? 1 : k == 4 ? 3 : 2;
}

typedef uint32_t v4u __attribute__((ext_vector_type(4)));

// The 8 x 12-bit links of a record.
__device__ __forceinline__ void unpack12(const v4u& w, int (&c)[8]) {
  c[0] = w.x & 0xFFF;
  c[1] = (w.x >> 12) & 0xFFF;
  c[2] = (w.x >> 24) | ((w.y & 0xF) << 8);
  c[3] = (w.y >> 4) & 0xFFF;
  c[4] = (w.y >> 16) & 0xFFF;
  c[5] = (w.y >> 28) | ((w.z & 0xFF) << 4);
  c[6] = (w.z >> 8) & 0xFFF;
  c[7] = w.z >> 20;
}

typedef unsigned long long word;
__device__ __forceinline__ void put_word(word* p, word w) {
  __hip_atomic_store(p, w, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ word get_word(const word* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// One exchanged cell: its 6 stresses in slot order, 8 bytes a word.
template <typename T>
struct Packed {
  static constexpr int kWords = 6 * sizeof(T) / 8;
  word w[kWords];
  __device__ __forceinline__ void pack(const T (&o)[6]) {
    if constexpr (sizeof(T) == 8) {
#pragma unroll
      for (int k = 0; k < 6; k++) w[k] = (word)__double_as_longlong(o[k]);
    } else {
#pragma unroll
      for (int k = 0; k < 3; k++)
        w[k] = (word)__float_as_uint(o[2 * k]) | ((word)__float_as_uint(o[2 * k + 1]) << 32);
    }
  }
  __device__ __forceinline__ void unpack(T (&o)[6]) const {
    if constexpr (sizeof(T) == 8) {
#pragma unroll
      for (int k = 0; k < 6; k++) o[k] = __longlong_as_double((long long)w[k]);
    } else {
#pragma unroll
      for (int k = 0; k < 3; k++) {
        o[2 * k] = __uint_as_float((uint32_t)w[k]);
        o[2 * k + 1] = __uint_as_float((uint32_t)(w[k] >> 32));
      }
    }
  }
};

// Two consecutive components as one LDS access.
template <typename T>
__device__ __forceinline__ void put_slot(T* S, int i, const T (&v)[6]) {
  typedef T P __attribute__((ext_vector_type(2)));
  P* q = reinterpret_cast<P*>(S) + 3 * i;
#pragma unroll
  for (int p = 0; p < 3; p++) q[p] = P{v[2 * p], v[2 * p + 1]};
}

// Waits until every lane's flag (nullptr: none) has reached `want`; false when the wait ran out
// (here or in another workgroup).
__device__ __forceinline__ bool wait_flags(const uint32_t* flag, uint32_t want, int32_t* status) {
  uint64_t t0 = 0;
  for (uint32_t spin = 1;; spin++) {
    const uint32_t f = flag ? __hip_atomic_load(flag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) : want;
    if (__all((int32_t)(f - want) >= 0)) return true;
    if ((spin & 1023u) == 0) {
      const uint64_t t = wall_clock64();
      if (t0 == 0) t0 = t;
      const bool out = t - t0 > kWaitTicks;
      if (out) __hip_atomic_store(status + kResidentLost, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
      if (out || __hip_atomic_load(status + kResidentLost, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM)) return false;
    }
  }
}

// NKEY / CKEY: node and cell coefficients by class key (else per-entity arrays).  REC: the records
// are in LDS (else in a.work, which stays in the L2).
template <typename T, int THREADS, bool NKEY, bool CKEY, bool REC>
__global__ __launch_bounds__(THREADS) void resident_kernel(ResidentArgs<T> a) {
  extern __shared__ __align__(16) unsigned char smem[];
  typedef T P __attribute__((ext_vector_type(2)));
  T* const S = reinterpret_cast<T*>(smem);  // [max_set + 1][6]: own cells, halo, zero
  T* const V = S + 6 * (a.max_set + 1);     // [max_node][3]
  unsigned char* const rest = smem + ((6 * (a.max_set + 1) + 3 * a.max_node) * sizeof(T) + 15) / 16 * 16;
  // records: 8 x 12-bit links, then the key (or the id, for per-entity coefficients)
  v4u* nrec;
  if constexpr (REC)
    nrec = reinterpret_cast<v4u*>(rest);
  else
    nrec = reinterpret_cast<v4u*>(a.work) + (size_t)blockIdx.x * (a.max_node + a.max_cell);
  v4u* const crec = nrec + a.max_node;
  // marks of the special nodes and cells: 1 + the class of their source terms, a node's sensor
  uint8_t* const nmark = REC ? reinterpret_cast<uint8_t*>(crec + a.max_cell) : rest;
  uint8_t* const cmark = nmark + a.max_node;
  __shared__ double force[2][kResidentForces];  // of the even and the odd steps
  __shared__ int sensors;  // the tile records some
  __shared__ int published;  // waves that have published a step's exported cells, over all steps
  const ResidentTile tl = a.tiles[blockIdx.x];
  const int t = threadIdx.x;
  const int rt = t ^ (THREADS - 64);  // the waves in reverse order

  T* const Sg[6] = {a.s.S0, a.s.S1, a.s.S2, a.s.S3, a.s.S4, a.s.S5};
  auto load_stress = [&](int e, int slot) {
    T o[6];
#pragma unroll
    for (int q = 0; q < 6; q++) o[q] = Sg[slot_comp(q)][e];
    put_slot(S, slot, o);
  };
  __shared__ int go;  // the launch's steps are made
  bool last = false;
  if (t == 0) {
    sensors = published = 0;
    if (a.ntiles > 1)
      last = __hip_atomic_fetch_add(a.ctrl, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) + 1 ==
             a.seq * (uint32_t)a.ntiles;
  }
  __syncthreads();
  for (int i = t; i < tl.ncell; i += THREADS) {
    v4u r = reinterpret_cast<const v4u*>(a.crec)[tl.cell0 + i];
    const int e = (int)r.w;
    load_stress(e, i);
    int sp = -1;
    if constexpr (CKEY) {
      r.w = resolve_key(a.s, a.s.lkey ? a.s.lkey[4 * (size_t)e + 3] : a.s.key[e], sp);
      if (sp >= 0) r.w |= kSpecialKey;
    } else {
      const T x = a.s.dcx[e];
      if (is_boxed(x)) sp = unbox(x);
    }
    crec[i] = r;
    cmark[i] = sp >= 0 ? a.ccls[sp] + 1 : 0;
  }
  for (int i = t; i < tl.nhalo; i += THREADS) load_stress(a.hcell[tl.halo0 + i], tl.ncell + i);
  for (int i = t; i < tl.nnode; i += THREADS) {
    v4u r = reinterpret_cast<const v4u*>(a.nrec)[tl.node0 + i];
    const int n = (int)(r.w & ~kResidentOwner);
    int sp = -1;
    uint8_t mark = 0;
    const bool owner = r.w & kResidentOwner;
    if constexpr (NKEY) {
      r.w = resolve_key(a.v, a.v.lkey ? a.v.lkey[4 * (size_t)n + 3] : a.v.key[n], sp);
      if (sp >= 0) r.w |= kSpecialKey;
    } else {
      r.w = (uint32_t)n;
      const T x = a.v.idt[n];
      if (is_boxed(x)) sp = unbox(x);
    }
    if (sp >= 0) {
      mark = a.ncls[sp] + 1;
      if (owner && a.v.sp_sens[sp] >= 0) {
        mark |= kResidentSensor;
        sensors = 1;
      }
    }
    nrec[i] = r;
    nmark[i] = mark;
    V[3 * i] = a.v.V0[n];
    V[3 * i + 1] = a.v.V1[n];
    V[3 * i + 2] = a.v.V2[n];
  }
  if (t < 6) S[6 * (tl.ncell + tl.nhalo) + t] = T(0);  // where the links to missing cells point
  constexpr int W = Packed<T>::kWords;
  const int2 none = {0, 0};
  const int2 first = rt < tl.nhalo ? a.halo[tl.halo0 + rt] : none;  // exchange slot, tile
  // waves that publish exported cells each step
  const int pub_waves = min((tl.nexp + 63) / 64, THREADS / 64);

  const VelocityArgs<T>& va = a.v;
  const StressArgs<T>& sa = a.s;
  const double* now = force[0];  // this step's source terms
  auto node_update = [&](int i) {
    const v4u rec = nrec[i];
    T idt, sx, sy, sz;
    bool special = false;
    if constexpr (NKEY) {
      special = rec.w & kSpecialKey;
      const uint32_t k = rec.w & ~kSpecialKey;
      const uint32_t k0 = __builtin_amdgcn_readfirstlane(k);
      if (__all(k == k0)) {
        idt = as_const(va.cls)[k0 >> kMatShift];
        axis_spacings(as_const(va.axis), k0, sx, sy, sz);
      } else {
        idt = va.cls[k >> kMatShift];
        axis_spacings(va.axis, k, sx, sy, sz);
      }
    } else {
      idt = va.idt[rec.w];
      sx = va.dnx[rec.w];
      sy = va.dny[rec.w];
      sz = va.dnz[rec.w];
      if (is_boxed(idt)) {
        special = true;
        idt = va.sp_idt[unbox(idt)];
      }
    }
    int c[8];
    unpack12(rec, c);
    T r[3];
    node_rates(
        [&](int p, T(&f)[8], T(&g)[8]) {
          const P* q = reinterpret_cast<const P*>(S) + p;
#pragma unroll
          for (int k = 0; k < 8; k++) {
            const P w = q[3 * c[k]];
            f[k] = w.x;
            g[k] = w.y;
          }
        },
        sx, sy, sz, r);
    if (special) {
      const double* f = now + 3 * ((nmark[i] & ~kResidentSensor) - 1);
#pragma unroll
      for (int d = 0; d < 3; d++) r[d] = r[d] + (T)f[d];
    }
#pragma unroll
    for (int d = 0; d < 3; d++) V[3 * i + d] = V[3 * i + d] + idt * r[d];
  };

  auto moments = [&](int i, int sp, double (&m)[6]) {
    if (sp < 0) return;
    const double* f = now + a.cforce0 + 6 * (cmark[i] - 1);
#pragma unroll
    for (int q = 0; q < 6; q++) m[q] = f[q];
  };

  // Steps the cell in its slot; o: its new stresses in slot order.
  auto cell_update = [&](int i, T (&o)[6]) {
    const v4u rec = crec[i];
    int c[8];
    unpack12(rec, c);
    T s[6];
#pragma unroll
    for (int p = 0; p < 3; p++) {
      const P w = reinterpret_cast<const P*>(S)[3 * i + p];
      s[slot_comp(2 * p)] = w.x;
      s[slot_comp(2 * p + 1)] = w.y;
    }
    T d[6];
    double m[6] = {0, 0, 0, 0, 0, 0};
    int sp = -1;
    auto xy = [&](T(&f)[8], T(&g)[8]) {
#pragma unroll
      for (int k = 0; k < 8; k++) {
        f[k] = V[3 * c[k]];
        g[k] = V[3 * c[k] + 1];
      }
    };
    auto z = [&](T(&f)[8]) {
#pragma unroll
      for (int k = 0; k < 8; k++) f[k] = V[3 * c[k] + 2];
    };
    if constexpr (CKEY) {
      if (rec.w & kSpecialKey) sp = 0;
      const uint32_t k = rec.w & ~kSpecialKey;
      const uint32_t k0 = __builtin_amdgcn_readfirstlane(k);
      T sx, sy, sz;
      if (__all(k == k0))
        axis_spacings(as_const(sa.axis), k0, sx, sy, sz);
      else
        axis_spacings(sa.axis, k, sx, sy, sz);
      const uint32_t mat = k >> kMatShift;
      uint32_t m0 = k0 >> kMatShift;
      strain_rates<T>(xy, z, sx, sy, sz, d);
      moments(i, sp, m);
      // one pass per distinct material of the wavefront, its row through the scalar cache
      for (;;) {
        if (mat == m0) {
          voigt_update(sa.dt, as_const(sa.cls + (size_t)m0 * kMatRow), d, m, sp, s);
          break;
        }
        m0 = __builtin_amdgcn_readfirstlane(mat);
      }
    } else {
      const int e = (int)rec.w;
      T sx = sa.dcx[e];
      const T sy = sa.dcy[e], sz = sa.dcz[e];
      T cc[21];
#pragma unroll
      for (int q = 0; q < 21; q++)
        cc[q] = sa.C[sa.ldc ? (int64_t)q * sa.ldc + e : ((int64_t)(e >> 6) * 21 + q) * 64 + (e & 63)];
      if (is_boxed(sx)) {
        sp = 0;
        sx = sa.sp_dcx[unbox(sx)];
      }
      strain_rates<T>(xy, z, sx, sy, sz, d);
      moments(i, sp, m);
      voigt_update(sa.dt, cc, d, m, sp, s);
    }
#pragma unroll
    for (int q = 0; q < 6; q++) o[q] = s[slot_comp(q)];
    put_slot(S, i, o);
  };

  if (a.ntiles > 1) {
    if (t == 0) go = agree(a.ctrl + 1, a.seq, last);
    __syncthreads();
    if (!go) return;
  }

  bool alive = true;
  double f0 = t < a.nforce ? a.force[t] : 0.0;
#pragma unroll 1
  for (int k = 0; k < a.nsteps; k++) {
    now = force[k & 1];
    if (t < a.nforce) {
      force[k & 1][t] = f0;
      if (k + 1 < a.nsteps) f0 = a.force[(size_t)(k + 1) * a.nforce + t];
    }
    __syncthreads();  // the step before's stresses are in LDS, and its velocities are read
#pragma unroll 1
    for (int i = t; i < tl.nown; i += THREADS) node_update(i);
    if (tl.nhalo > 0) {
      if (k > 0) {
        const word* x = a.xbuf + (size_t)((a.epoch + k) & 1) * a.nexp * W;
        for (int i = rt; (i & ~63) < tl.nhalo; i += THREADS) {
          const bool on = i < tl.nhalo;
          const int2 h = i == rt || !on ? first : a.halo[tl.halo0 + i];
          if (alive)
            alive = wait_flags(on ? a.flag + (size_t)kFlagStride * h.y : nullptr, a.epoch + (uint32_t)k, a.status);
          asm volatile("" ::: "memory");  // the loads below stay behind the wait
          if (on) {
            Packed<T> w;
            T o[6];
#pragma unroll
            for (int q = 0; q < W; q++) w.w[q] = get_word(x + q * (size_t)a.nexp + h.x);
            w.unpack(o);
            put_slot(S, tl.ncell + i, o);
          }
        }
      }
      __syncthreads();  // the halo is in LDS
#pragma unroll 1
      for (int i = tl.nown + t; i < tl.nnode; i += THREADS) node_update(i);
    }
    __syncthreads();  // the velocities are in LDS, and the stresses are read
    const bool publish = k + 1 < a.nsteps;  // the last step's stresses go to the state alone
    word* const x = a.xbuf + (size_t)((a.epoch + k + 1) & 1) * a.nexp * W + tl.exp0;
#pragma unroll 1
    for (int i = t; i < tl.nexp; i += THREADS) {
      T o[6];
      cell_update(i, o);
      if (publish) {
        Packed<T> w;
        w.pack(o);
#pragma unroll
        for (int q = 0; q < W; q++) put_word(x + q * (size_t)a.nexp + i, w.w[q]);
      }
    }
    if (publish && tl.nexp > (t & ~63)) {
      // the wave whose stores are the last to be out sets the flag
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      if ((t & 63) == 0 && atomicAdd(&published, 1) == (k + 1) * pub_waves - 1)
        __hip_atomic_store(a.flag + (size_t)kFlagStride * blockIdx.x, a.epoch + (uint32_t)k + 1u, __ATOMIC_RELAXED,
                           __HIP_MEMORY_SCOPE_AGENT);
    }
#pragma unroll 1
    for (int i = tl.nexp + rt; i < tl.ncell; i += THREADS) {
      T o[6];
      cell_update(i, o);
    }
    if (sensors)  // this step's velocities stay in LDS until the next barrier
      for (int i = rt; i < tl.nnode; i += THREADS)
        if (nmark[i] & kResidentSensor) {
          const int n = (int)(a.nrec[4 * (size_t)(tl.node0 + i) + 3] & ~kResidentOwner);
          int sp;
          if constexpr (NKEY)
            resolve_key(va, va.lkey ? va.lkey[4 * (size_t)n + 3] : va.key[n], sp);
          else
            sp = unbox(va.idt[n]);
          double* out = va.trace + (size_t)k * a.row + 3 * va.sp_sens[sp];
#pragma unroll
          for (int d = 0; d < 3; d++) out[d] = (double)V[3 * i + d];
        }
  }
  __syncthreads();

  for (int i = t; i < tl.ncell; i += THREADS) {
    const int e = (int)a.crec[4 * (size_t)(tl.cell0 + i) + 3];
#pragma unroll
    for (int q = 0; q < 6; q++) Sg[slot_comp(q)][e] = S[6 * i + q];
  }
  for (int i = t; i < tl.nnode; i += THREADS) {
    const uint32_t w = a.nrec[4 * (size_t)(tl.node0 + i) + 3];
    if (!(w & kResidentOwner)) continue;
    const int n = (int)(w & ~kResidentOwner);
    a.v.V0[n] = V[3 * i];
    a.v.V1[n] = V[3 * i + 1];
    a.v.V2[n] = V[3 * i + 2];
  }
}

// The steps of a launch whose tiles did not get onto the GPU together, by one workgroup from
// memory: all nodes, then all cells, tile after tile.  Ends at once after any other launch.
template <typename T>
__global__ __launch_bounds__(1024) void resident_alone_kernel(ResidentArgs<T> a) {
  if (__hip_atomic_load(a.ctrl + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == 2 * a.seq + 1) return;
  const int t = threadIdx.x, threads = blockDim.x;
  T* const Sg[6] = {a.s.S0, a.s.S1, a.s.S2, a.s.S3, a.s.S4, a.s.S5};
  T* const Vg[3] = {a.v.V0, a.v.V1, a.v.V2};
  const VelocityArgs<T>& va = a.v;
  const StressArgs<T>& sa = a.s;
  for (int k = 0; k < a.nsteps; k++) {
    const double* now = a.force + (size_t)k * a.nforce;
    for (int b = 0; b < a.ntiles; b++) {
      const ResidentTile tl = a.tiles[b];
      for (int i = t; i < tl.nnode; i += threads) {
        const v4u rec = reinterpret_cast<const v4u*>(a.nrec)[tl.node0 + i];
        if (!(rec.w & kResidentOwner)) continue;
        const int n = (int)(rec.w & ~kResidentOwner);
        int c[8];
        unpack12(rec, c);
#pragma unroll
        for (int q = 0; q < 8; q++)  // slots to cells
          c[q] = c[q] < tl.ncell                ? (int)a.crec[4 * (size_t)(tl.cell0 + c[q]) + 3]
                 : c[q] < tl.ncell + tl.nhalo ? a.hcell[tl.halo0 + c[q] - tl.ncell]
                                              : -1;
        T idt, sx, sy, sz, r[3];
        int sp = -1;
        if (va.key || va.lkey) {
          const uint32_t key = resolve_key(va, va.lkey ? va.lkey[4 * (size_t)n + 3] : va.key[n], sp);
          idt = va.cls[key >> kMatShift];
          axis_spacings(va.axis, key, sx, sy, sz);
        } else {
          idt = va.idt[n];
          sx = va.dnx[n];
          sy = va.dny[n];
          sz = va.dnz[n];
          if (is_boxed(idt)) {
            sp = unbox(idt);
            idt = va.sp_idt[sp];
          }
        }
        node_rates(
            [&](int p, T(&f)[8], T(&g)[8]) {
#pragma unroll
              for (int q = 0; q < 8; q++) {
                f[q] = c[q] >= 0 ? Sg[slot_comp(2 * p)][c[q]] : T(0);
                g[q] = c[q] >= 0 ? Sg[slot_comp(2 * p + 1)][c[q]] : T(0);
              }
            },
            sx, sy, sz, r);
#pragma unroll
        for (int d = 0; d < 3; d++) {
          if (sp >= 0) r[d] = r[d] + (T)now[3 * a.ncls[sp] + d];
          Vg[d][n] = Vg[d][n] + idt * r[d];
          if (sp >= 0 && va.sp_sens[sp] >= 0) va.trace[(size_t)k * a.row + 3 * va.sp_sens[sp] + d] = (double)Vg[d][n];
        }
      }
    }
    __syncthreads();
    for (int b = 0; b < a.ntiles; b++) {
      const ResidentTile tl = a.tiles[b];
      for (int i = t; i < tl.ncell; i += threads) {
        const v4u rec = reinterpret_cast<const v4u*>(a.crec)[tl.cell0 + i];
        const int e = (int)rec.w;
        int c[8];
        unpack12(rec, c);
#pragma unroll
        for (int q = 0; q < 8; q++) c[q] = (int)(a.nrec[4 * (size_t)(tl.node0 + c[q]) + 3] & ~kResidentOwner);
        T sx, sy, sz, cc[21], d[6], s[6];
        int sp = -1;
        if (sa.key || sa.lkey) {
          const uint32_t key = resolve_key(sa, sa.lkey ? sa.lkey[4 * (size_t)e + 3] : sa.key[e], sp);
          axis_spacings(sa.axis, key, sx, sy, sz);
#pragma unroll
          for (int q = 0; q < 21; q++) cc[q] = sa.cls[(size_t)(key >> kMatShift) * kMatRow + q];
        } else {
          sx = sa.dcx[e];
          sy = sa.dcy[e];
          sz = sa.dcz[e];
          if (is_boxed(sx)) {
            sp = unbox(sx);
            sx = sa.sp_dcx[sp];
          }
#pragma unroll
          for (int q = 0; q < 21; q++)
            cc[q] = sa.C[sa.ldc ? (int64_t)q * sa.ldc + e : ((int64_t)(e >> 6) * 21 + q) * 64 + (e & 63)];
        }
        double m[6] = {0, 0, 0, 0, 0, 0};
#pragma unroll
        for (int q = 0; q < 6; q++) {
          if (sp >= 0) m[q] = now[a.cforce0 + 6 * a.ccls[sp] + q];
          s[q] = Sg[q][e];
        }
        strain_rates<T>(
            [&](T(&f)[8], T(&g)[8]) {
#pragma unroll
              for (int q = 0; q < 8; q++) {
                f[q] = Vg[0][c[q]];
                g[q] = Vg[1][c[q]];
              }
            },
            [&](T(&f)[8]) {
#pragma unroll
              for (int q = 0; q < 8; q++) f[q] = Vg[2][c[q]];
            },
            sx, sy, sz, d);
        voigt_update(sa.dt, cc, d, m, sp, s);
#pragma unroll
        for (int q = 0; q < 6; q++) Sg[q][e] = s[q];
      }
    }
    __syncthreads();
  }
  if (t == 0) __hip_atomic_store(a.status + kResidentAlone, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

template <typename T, int THREADS, bool NKEY, bool CKEY>
const void* resident_fn(bool rec) {
  return rec ? reinterpret_cast<const void*>(&resident_kernel<T, THREADS, NKEY, CKEY, true>)
             : reinterpret_cast<const void*>(&resident_kernel<T, THREADS, NKEY, CKEY, false>);
}
template <typename T, int THREADS>
const void* resident_fn(bool nkey, bool ckey, bool rec) {
  if (nkey) return ckey ? resident_fn<T, THREADS, true, true>(rec) : resident_fn<T, THREADS, true, false>(rec);
  return ckey ? resident_fn<T, THREADS, false, true>(rec) : resident_fn<T, THREADS, false, false>(rec);
}

template <typename T>
hipError_t launch_resident(const ResidentArgs<T>& a, int threads, hipStream_t st) {
  if (a.nsteps < 2 || a.ntiles <= 0 || a.nforce > kResidentForces || a.nforce > threads) return hipErrorInvalidValue;
  const bool nkey = a.v.key || a.v.lkey, ckey = a.s.key || a.s.lkey, rec = a.work == nullptr;
  const void* fn = threads == 256    ? resident_fn<T, 256>(nkey, ckey, rec)
                   : threads == 512  ? resident_fn<T, 512>(nkey, ckey, rec)
                   : threads == 1024 ? resident_fn<T, 1024>(nkey, ckey, rec)
                                     : nullptr;
  if (!fn) return hipErrorInvalidValue;
  const size_t lds = resident_lds_bytes(a.max_set, a.max_node, a.max_cell, sizeof(T), rec);
  void* args[1] = {const_cast<void*>(static_cast<const void*>(&a))};
  const hipError_t e = hipLaunchKernel(fn, dim3(a.ntiles), dim3(threads), args, lds, st);
  if (e != hipSuccess || a.ntiles == 1) return e;
  hipLaunchKernelGGL(resident_alone_kernel<T>, dim3(1), dim3(1024), 0, st, a);
  return hipGetLastError();
}

}  // namespace

hipError_t resident_limits(int* cus, size_t* lds) {
  int dev = 0, bytes = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e == hipSuccess) e = hipDeviceGetAttribute(cus, hipDeviceAttributeMultiprocessorCount, dev);
  if (e == hipSuccess) e = hipDeviceGetAttribute(&bytes, hipDeviceAttributeMaxSharedMemoryPerBlock, dev);
  if (e != hipSuccess) return e;
  *lds = (size_t)bytes;
  return hipSuccess;
}

hipError_t resident_after(hipStream_t s, hipEvent_t e) { return hipStreamWaitEvent(s, e, 0); }

hipError_t launch_resident_f64(const ResidentArgs<double>& a, int threads, hipStream_t s) {
  return launch_resident<double>(a, threads, s);
}
hipError_t launch_resident_f32(const ResidentArgs<float>& a, int threads, hipStream_t s) {
  return launch_resident<float>(a, threads, s);
}

}  // namespace rsg
