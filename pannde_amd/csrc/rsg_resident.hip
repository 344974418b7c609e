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
// relaxed atomics, and a word's arrival is its own signal: every word is kEmptyWord until it is
// written, and a reader loads a cell's words until none is empty, so a step has one trip through
// memory (store, load) between two tiles.  (A flag per tile instead, set when its stores are out
// and read before the words, made it three: see the figures below.)
// The stresses before step k of a launch are in buffer k % 4.  A tile that has its whole halo of
// step k - 1 knows that its neighbours, the readers of its cells, are done with k - 2's; at the
// start of step k it empties that buffer for k + 2 and waits for these stores before it publishes
// k + 1, so a reader that has a cell's words of k + 1 finds those of k + 2 empty or written.  All
// buffers are emptied before the workgroups agree on the start.
//
// A step reads memory for nothing but its halo: the class tables are in LDS, FP64 with reciprocals
// of the spacings (see Recip), because a load in an update waits behind the exchange's stores.
//
// What bounds it: up to some 30,000 cells the trip of the exchange and the dependent latency of two
// updates (node and cell about 2,000 cycles each, with a wave or two per SIMD); above, the
// arithmetic and the LDS reads of a tile (24 reads of 16 bytes a node).  Every byte of state stays
// on the chip, so memory does not.  Aluminium blocks on an MI355X, us a step FP64 / FP32, with the
// per-step kernels, with a flag per tile, spacings through the caches and IEEE divisions, and now:
// 480 cells 8.9/8.3, 4.5/2.8, 4.1/2.7; 32,000 cells 9.7/8.9, 4.5/3.6, 4.4/3.5; 131,000 cells
// 12.8/10.0, 7.4/4.9, 6.4/4.5; 259,000 cells 18.2/12.0, 12.3/7.9, 11.0/6.9.
// (Three lanes to a node and a cell, each with a third of the differences, gained nothing: 32,000
// cells 4.3 us, 3.6 in FP32; the LDS reads and their latency remain.)
//
// The workgroups wait for each other, so they must all be on the GPU at once.  There are no more
// of them than compute units, and the host lets one resident launch run at a time, but another
// process or stream may hold part of the GPU.  So a launch first agrees: the last workgroup to
// start decides that the steps are made; one that has waited long decides that they are not, and
// all leave with nothing written.  What was queued behind such a launch must not run on its state: a
// launch that the host queues behind one whose decision it does not know yet gets a kernel of one
// thread in front, which passes a refusal on.  The host reads the decisions when it waits for the
// handle anyway, and makes the steps of refused launches with the per-step kernels.
// (A cooperative launch would see to the start too, but costs 20 us and the host's wait for it, and on
// ROCm 7 its queue slows the streams created after it: a batch's two lanes took 5.4 ms for 2.0 ms of
// work.  Waiting for each decision before queuing more costs nothing on an idle GPU, but beside a busy
// batch each piece of work then waits for a turn of its own: 100 steps of 259,000 cells and their
// energy 82..136 ms against 55.)
#include <type_traits>

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
// was the last to start or not; the one that decides tells the host.
__device__ __forceinline__ bool agree(uint32_t* decision, int32_t* status, uint32_t seq, bool last) {
  uint64_t t0 = 0;
  for (;;) {
    uint32_t d = __hip_atomic_load(decision, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (decided(d, seq)) return d & 1;
    const uint64_t t = wall_clock64();
    if (t0 == 0) t0 = t;
    const uint32_t mine = 2 * seq + (last ? 1u : 0u);
    if ((last || t - t0 > kStartTicks) &&  // the first decision stands
        __hip_atomic_compare_exchange_strong(decision, &d, mine, __ATOMIC_RELAXED, __ATOMIC_RELAXED,
                                             __HIP_MEMORY_SCOPE_AGENT))
      __hip_atomic_store(status + kResidentDecision, (int32_t)mine, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
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
// What an exchange word holds until it is written: a NaN (two, in FP32) that no arithmetic gives.
// A stress that a caller gave these very bits is sent with another payload.
constexpr word kEmptyWord = 0xFFFADE17FFFADE17ull;
__device__ __forceinline__ word sent(word w) { return w == kEmptyWord ? w ^ 1 : w; }
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
#pragma unroll
    for (int k = 0; k < kWords; k++) w[k] = sent(w[k]);
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

// Loads the words of the exchanged cell at x (`on`: the lane has one), as often as it takes until
// every lane of the wave has its whole cell; false when the wait ran out (here or in another
// workgroup).
template <typename T>
__device__ __forceinline__ bool fetch_cell(const word* x, int nexp, bool on, int32_t* status, Packed<T>& w) {
  uint64_t t0 = 0;
  for (uint32_t spin = 1;; spin++) {
    if (on) {
      bool full = true;
#pragma unroll
      for (int q = 0; q < Packed<T>::kWords; q++) w.w[q] = get_word(x + q * (size_t)nexp);
#pragma unroll
      for (int q = 0; q < Packed<T>::kWords; q++) full &= w.w[q] != kEmptyWord;
      on = !full;
    }
    if (!__any(on)) return true;
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
  // spacings with their reciprocals in FP64
  using Sp = typename std::conditional<sizeof(T) == 8, Recip, float>::type;
  struct alignas(sizeof(T) == 8 ? 16 : 4) Entry {
    Sp s;
  };
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
  // the class tables: spacings of the nodes and the cells ([axis][class]), then dt/rho
  unsigned char* const after = cmark + a.max_cell;
  Entry* const naxis = reinterpret_cast<Entry*>(smem + ((after - smem) + 15) / 16 * 16);
  Entry* const caxis = naxis + 3 * kResidentClasses;
  T* const ncls = reinterpret_cast<T*>(caxis + 3 * kResidentClasses);
  __shared__ double force[2][kResidentForces];  // of the even and the odd steps
  // the tile's sensors, slot << 12 | node; more than the list holds are looked up every step
  constexpr int kListed = 32;
  __shared__ int sensors;
  __shared__ uint32_t sensor[kListed];
  const ResidentTile tl = a.tiles[blockIdx.x];
  const int t = threadIdx.x;
  const int rt = THREADS - 64 - (t & ~63) + (t & 63);  // the waves in reverse order

  T* const Sg[6] = {a.s.S0, a.s.S1, a.s.S2, a.s.S3, a.s.S4, a.s.S5};
  auto load_stress = [&](int e, int slot) {
    T o[6];
#pragma unroll
    for (int q = 0; q < 6; q++) o[q] = Sg[slot_comp(q)][e];
    put_slot(S, slot, o);
  };
  __shared__ int go;  // the launch's steps are made
  constexpr int W = Packed<T>::kWords;
  const size_t xstep = (size_t)W * a.nexp;  // words of an exchange buffer
  auto empty = [&](word* x) {
    for (int i = t; i < tl.nexp; i += THREADS)
#pragma unroll
      for (int q = 0; q < W; q++) put_word(x + q * (size_t)a.nexp + i, kEmptyWord);
  };
  bool last = false;
  for (int b = 0; b < 4; b++) empty(a.xbuf + b * xstep + tl.exp0);
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
  if (t == 0) {
    sensors = 0;
    if (a.ntiles > 1)
      last = __hip_atomic_fetch_add(a.ctrl, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) + 1 ==
             a.seq * (uint32_t)a.ntiles;
  }
  __syncthreads();
  if (a.tables && t < 3 * kResidentClasses) {
    const int at = t / kResidentClasses * kAxisClasses + t % kResidentClasses;
    if constexpr (NKEY) set_spacing(a.v.axis[at], naxis[t].s);
    if constexpr (CKEY) set_spacing(a.s.axis[at], caxis[t].s);
    if constexpr (NKEY)
      if (t < a.nmat) ncls[t] = a.v.cls[t];
  }
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
        const uint32_t slot = (uint32_t)a.v.sp_sens[sp];
        const int at = atomicAdd(&sensors, slot < 1u << 20 ? 1 : kListed + 1);
        if (at < kListed) sensor[at] = slot << 12 | (uint32_t)i;
      }
    }
    nrec[i] = r;
    nmark[i] = mark;
    V[3 * i] = a.v.V0[n];
    V[3 * i + 1] = a.v.V1[n];
    V[3 * i + 2] = a.v.V2[n];
  }
  if (t < 6) S[6 * (tl.ncell + tl.nhalo) + t] = T(0);  // where the links to missing cells point
  const int first = rt < tl.nhalo ? a.halo[tl.halo0 + rt] : 0;  // exchange slot

  const VelocityArgs<T>& va = a.v;
  const StressArgs<T>& sa = a.s;
  const double* now = force[0];  // this step's source terms
  // spacings of class key k, from LDS or through the caches
  auto spacings = [&](const Entry* table, const T* axis, uint32_t k, Sp (&sp)[3]) {
    if (a.tables) {
#pragma unroll
      for (int d = 0; d < 3; d++)
        sp[d] = table[d * kResidentClasses + ((k >> (14 - 7 * d)) & (kResidentClasses - 1))].s;
    } else {
      T x[3];
      axis_spacings(axis, k, x[0], x[1], x[2]);
#pragma unroll
      for (int d = 0; d < 3; d++) set_spacing(x[d], sp[d]);
    }
  };
  auto node_update = [&](int i) {
    const v4u rec = nrec[i];
    T idt;
    Sp sp[3];
    bool special = false;
    if constexpr (NKEY) {
      special = rec.w & kSpecialKey;
      const uint32_t k = rec.w & ~kSpecialKey;
      spacings(naxis, va.axis, k, sp);
      // (one read from a chosen address would be a flat load, which waits for all others)
      if (a.tables)
        idt = ncls[k >> kMatShift];
      else
        idt = as_const(va.cls)[k >> kMatShift];
    } else {
      idt = va.idt[rec.w];
      set_spacing(va.dnx[rec.w], sp[0]);
      set_spacing(va.dny[rec.w], sp[1]);
      set_spacing(va.dnz[rec.w], sp[2]);
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
          // one pair's reads at a time: all three do not fit the 128 registers of 1024 threads (and
          // spilling them cost 259,000 cells 13.7 us a step against 11.0)
          if constexpr (sizeof(T) == 8 && THREADS == 1024) asm volatile("" ::: "memory");
          const P* q = reinterpret_cast<const P*>(S) + p;
#pragma unroll
          for (int k = 0; k < 8; k++) {
            const P w = q[3 * c[k]];
            f[k] = w.x;
            g[k] = w.y;
          }
        },
        sp, r);
    if (special) {
      const double* f = now + 3 * ((nmark[i] & ~kResidentSensor) - 1);
#pragma unroll
      for (int d = 0; d < 3; d++) r[d] = r[d] + (T)f[d];
    }
#pragma unroll
    for (int d = 0; d < 3; d++) V[3 * i + d] = V[3 * i + d] + idt * r[d];
  };

  // Steps the cell in its slot; o: its new stresses in slot order.
  auto cell_update = [&](int i, T (&o)[6]) {
    const v4u rec = crec[i];
    int c[8];
    unpack12(rec, c);
    T s[6], d[6];
    auto own = [&]() {  // after the differences, which need the registers
      asm volatile("" ::: "memory");
#pragma unroll
      for (int p = 0; p < 3; p++) {
        const P w = reinterpret_cast<const P*>(S)[3 * i + p];
        s[slot_comp(2 * p)] = w.x;
        s[slot_comp(2 * p + 1)] = w.y;
      }
    };
    int sp = -1;
    double terms[6] = {0, 0, 0, 0, 0, 0};
    auto moments = [&]() {  // read at once: one wait for the six
      if (sp < 0) return;
      const double* f = now + a.cforce0 + 6 * (cmark[i] - 1);
#pragma unroll
      for (int q = 0; q < 6; q++) terms[q] = f[q];
    };
    auto m = [&](int q) { return terms[q]; };
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
    Sp sd[3];
    if constexpr (CKEY) {
      if (rec.w & kSpecialKey) sp = 0;
      const uint32_t k = rec.w & ~kSpecialKey;
      spacings(caxis, sa.axis, k, sd);
      // the first lane's material row is requested before the differences need it
      const uint32_t mat = k >> kMatShift;
      uint32_t m0 = __builtin_amdgcn_readfirstlane(mat);
      const auto row0 = as_const(sa.cls + (size_t)m0 * kMatRow);
      T c0[21];
#pragma unroll
      for (int q = 0; q < 21; q++) c0[q] = row0[q];
      strain_rates(xy, z, sd, d);
      own();
      moments();
      if (__all(mat == m0)) {
        voigt_update(sa.dt, c0, d, m, sp, s);
      } else {  // one pass per distinct material of the wavefront
        for (;;) {
          if (mat == m0) {
            voigt_update(sa.dt, as_const(sa.cls + (size_t)m0 * kMatRow), d, m, sp, s);
            break;
          }
          m0 = __builtin_amdgcn_readfirstlane(mat);
        }
      }
    } else {
      const int e = (int)rec.w;
      T sx = sa.dcx[e];
      const T sy = sa.dcy[e], sz = sa.dcz[e];
      T cc[21];
      cell_constants(sa, e, cc);
      if (is_boxed(sx)) {
        sp = 0;
        sx = sa.sp_dcx[unbox(sx)];
      }
      set_spacing(sx, sd[0]);
      set_spacing(sy, sd[1]);
      set_spacing(sz, sd[2]);
      strain_rates(xy, z, sd, d);
      own();
      moments();
      voigt_update(sa.dt, cc, d, m, sp, s);
    }
#pragma unroll
    for (int q = 0; q < 6; q++) o[q] = s[slot_comp(q)];
    put_slot(S, i, o);
  };

  if (a.ntiles > 1) {
    if (t == 0) go = agree(a.ctrl + 1, a.status, a.seq, last);
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
    if (k > 2 && k + 2 < a.nsteps) empty(a.xbuf + ((k + 2) % 4) * xstep + tl.exp0);
#pragma unroll 1
    for (int i = t; i < tl.nown; i += THREADS) node_update(i);
    if (tl.nhalo > 0) {
      if (k > 0) {
        const word* x = a.xbuf + (k % 4) * xstep;
        for (int i = rt; (i & ~63) < tl.nhalo; i += THREADS) {
          const bool on = i < tl.nhalo;
          const int h = i == rt || !on ? first : a.halo[tl.halo0 + i];
          Packed<T> w = {};
          if (alive) alive = fetch_cell<T>(x + h, a.nexp, on, a.status, w);
          if (on) {
            T o[6];
            w.unpack(o);
            put_slot(S, tl.ncell + i, o);
          }
        }
      }
      __syncthreads();  // the halo is in LDS
#pragma unroll 1
      for (int i = tl.nown + t; i < tl.nnode; i += THREADS) node_update(i);
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the emptied words are out
    __syncthreads();  // the velocities are in LDS, and the stresses are read
    const bool publish = k + 1 < a.nsteps;  // the last step's stresses go to the state alone
    word* const x = a.xbuf + ((k + 1) % 4) * xstep + tl.exp0;
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
#pragma unroll 1
    for (int i = tl.nexp + rt; i < tl.ncell; i += THREADS) {
      T o[6];
      cell_update(i, o);
    }
    // this step's velocities stay in LDS until the next barrier
    if (sensors <= kListed) {
      if (rt < sensors) {
        const uint32_t w = sensor[rt];
        double* out = va.trace + (size_t)k * a.row + 3 * (w >> 12);
#pragma unroll
        for (int d = 0; d < 3; d++) out[d] = (double)V[3 * (w & 0xFFF) + d];
      }
    } else {
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

// In front of launch seq: it is decided against if the launch before it was (the host learns of that
// one alone).
__global__ void pass_refusal(uint32_t* decision, uint32_t seq) {
  if (__hip_atomic_load(decision, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == 2 * (seq - 1))
    __hip_atomic_store(decision, 2 * seq, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
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
  const size_t lds = resident_lds_bytes(a.max_set, a.max_node, a.max_cell, sizeof(T), rec) +
                     (a.tables ? resident_table_bytes(sizeof(T)) : 0);
  void* args[1] = {const_cast<void*>(static_cast<const void*>(&a))};
  if (a.chained) {
    uint32_t* decision = a.ctrl + 1;
    uint32_t seq = a.seq;
    void* pass[2] = {&decision, &seq};
    const hipError_t e = hipLaunchKernel(reinterpret_cast<const void*>(&pass_refusal), dim3(1), dim3(1), pass, 0, st);
    if (e != hipSuccess) return e;
  }
  return hipLaunchKernel(fn, dim3(a.ntiles), dim3(threads), args, lds, st);
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

void forget_error() { (void)hipGetLastError(); }

hipError_t resident_after(hipStream_t s, hipEvent_t e) { return hipStreamWaitEvent(s, e, 0); }

hipError_t launch_resident_f64(const ResidentArgs<double>& a, int threads, hipStream_t s) {
  return launch_resident<double>(a, threads, s);
}
hipError_t launch_resident_f32(const ResidentArgs<float>& a, int threads, hipStream_t s) {
  return launch_resident<float>(a, threads, s);
}

}  // namespace rsg
