// resident_stub.cpp -- the resident kernel's and the state transfers' launchers on the CPU, over the host stand-ins for the
// HIP runtime (hip_host_stub.cpp).  TEST INFRASTRUCTURE ONLY: it walks the tiles, records, halo and
// exchange slots exactly as the kernel does (each tile with its own copy of its slots and nodes, the
// exported stresses through the four-buffer exchange), with every index checked, so a plan that
// steps a mesh correctly here gives the kernel the right data.
#include <hip/hip_runtime_api.h>

#include <algorithm>
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <vector>

#include "../../pannde_amd/csrc/rsg_internal.h"

namespace rsg {
namespace {

#define CHECK(c)                                                        \
  do {                                                                  \
    if (!(c)) {                                                         \
      std::fprintf(stderr, "resident plan: %s (line %d)\n", #c, __LINE__); \
      std::abort();                                                     \
    }                                                                   \
  } while (0)

const int kSlot[6] = {0, 5, 4, 1, 3, 2};
const int kFwd[3][4] = {{1, 2, 5, 6}, {2, 3, 6, 7}, {4, 5, 6, 7}};
const int kBwd[3][4] = {{0, 3, 4, 7}, {0, 1, 4, 5}, {0, 1, 2, 3}};

void links(const uint32_t* w, int (&c)[8]) {
  for (int k = 0; k < 8; k++) {
    c[k] = 0;
    for (int b = 0; b < 12; b++) c[k] |= (int)(w[(12 * k + b) / 32] >> ((12 * k + b) % 32) & 1u) << b;
  }
}
double d_of(const double (&f)[8], int ax, double sp) {
  double v = 0.0;
  for (int q = 0; q < 4; q++) v += f[kFwd[ax][q]] - f[kBwd[ax][q]];
  return v * 0.25 / sp;
}
float d_of(const float (&f)[8], int ax, float inv) {
  const int p[3][4] = {{0, 1, 2, 3}, {0, 1, 2, 3}, {0, 1, 2, 3}};
  float g[4];
  for (int q = 0; q < 4; q++) g[q] = f[kFwd[ax][p[ax][q]]] - f[kBwd[ax][p[ax][q]]];
  return ((g[0] + g[1]) + (g[2] + g[3])) * inv;
}
int tri(int i, int j) { return i <= j ? i * 6 - i * (i - 1) / 2 + (j - i) : tri(j, i); }

// Index of component q (in slot order) of exchange slot x of a buffer: 8-byte words, nexp apart.
template <typename T>
size_t at(const ResidentArgs<T>& a, int buffer, int x, int q) {
  const int per = 8 / (int)sizeof(T), words = 6 / per;
  return (((size_t)buffer * words + q / per) * a.nexp + x) * per + q % per;
}

template <typename T>
hipError_t run(const ResidentArgs<T>& a, int threads) {
  CHECK(threads == 256 || threads == 512 || threads == 1024);
  CHECK(a.nsteps >= 2 && a.ntiles > 0);
  T* const Sg[6] = {a.s.S0, a.s.S1, a.s.S2, a.s.S3, a.s.S4, a.s.S5};
  T* const Vg[3] = {a.v.V0, a.v.V1, a.v.V2};
  T* const xb = reinterpret_cast<T*>(a.xbuf);
  std::vector<std::vector<T>> S(a.ntiles), V(a.ntiles);
  auto key = [](const auto& x, int i) { return x.lkey ? x.lkey[4 * (size_t)i + 3] : x.key[i]; };
  for (int t = 0; t < a.ntiles; t++) {
    const ResidentTile& tl = a.tiles[t];
    CHECK(tl.ncell > 0 && tl.ncell <= a.max_cell && tl.nexp <= tl.ncell && tl.nown <= tl.nnode);
    CHECK(tl.ncell + tl.nhalo <= a.max_set && tl.nnode <= a.max_node && tl.exp0 + tl.nexp <= a.nexp);
    S[t].assign((size_t)6 * (tl.ncell + tl.nhalo + 1), T(0));
    V[t].resize((size_t)3 * tl.nnode);
    for (int i = 0; i < tl.ncell + tl.nhalo; i++) {
      const int e = i < tl.ncell ? (int)a.crec[4 * (size_t)(tl.cell0 + i) + 3] : a.hcell[tl.halo0 + i - tl.ncell];
      CHECK(e >= 0 && e < a.s.n);
      for (int q = 0; q < 6; q++) S[t][6 * i + q] = Sg[kSlot[q]][e];
    }
    for (int i = 0; i < tl.nnode; i++) {
      const int n = (int)(a.nrec[4 * (size_t)(tl.node0 + i) + 3] & ~kResidentOwner);
      CHECK(n < a.v.n);
      for (int d = 0; d < 3; d++) V[t][3 * i + d] = Vg[d][n];
    }
  }
  std::fill(xb, xb + (size_t)24 * a.nexp, T(NAN));  // empty
  for (int k = 0; k < a.nsteps; k++) {
    const double* force = a.force + (size_t)k * a.nforce;
    for (int t = 0; t < a.ntiles; t++) {
      const ResidentTile& tl = a.tiles[t];
      if (k > 0)
        for (int i = 0; i < tl.nhalo; i++) {
          const int x = a.halo[tl.halo0 + i];
          CHECK(x >= 0 && x < a.nexp && (x < tl.exp0 || x >= tl.exp0 + tl.nexp));
          for (int q = 0; q < 6; q++) S[t][6 * (tl.ncell + i) + q] = xb[at(a, k % 4, x, q)];
        }
      if (k > 2 && k + 2 < a.nsteps)
        for (int x = tl.exp0; x < tl.exp0 + tl.nexp; x++)
          for (int q = 0; q < 6; q++) xb[at(a, (k + 2) % 4, x, q)] = T(NAN);
      for (int i = 0; i < tl.nnode; i++) {
        const uint32_t* r = &a.nrec[4 * (size_t)(tl.node0 + i)];
        const int n = (int)(r[3] & ~kResidentOwner);
        int c[8];
        links(r, c);
        for (int q : c) CHECK(q <= tl.ncell + tl.nhalo && (i >= tl.nown || q < tl.ncell || q == tl.ncell + tl.nhalo));
        T idt, sp[3];
        int special = -1;
        if (a.v.key || a.v.lkey) {
          uint32_t w = key(a.v, n);
          if (w & kSpecialKey) {
            special = (int)(w & ~kSpecialKey);
            w = a.v.sp_key[special];
          }
          idt = a.v.cls[w >> kMatShift];
          for (int d = 0; d < 3; d++) sp[d] = a.v.axis[d * kAxisClasses + (w >> (14 - 7 * d) & (kAxisClasses - 1))];
        } else {
          idt = a.v.idt[n];
          sp[0] = a.v.dnx[n], sp[1] = a.v.dny[n], sp[2] = a.v.dnz[n];
          if (std::isnan(idt)) {
            uint64_t bits = 0;
            std::memcpy(&bits, &idt, sizeof(T));
            special = (int)(bits & (sizeof(T) == 8 ? 0xFFFFFFFFull : 0x3FFFFFull));
            idt = a.v.sp_idt[special];
          }
        }
        auto D = [&](int q, int ax) {
          T f[8];
          for (int b = 0; b < 8; b++) f[b] = S[t][6 * c[b] + q];
          return d_of(f, ax, sp[ax]);
        };
        T w[3] = {(D(0, 0) + D(1, 1)) + D(2, 2), (D(1, 0) + D(3, 1)) + D(4, 2), (D(2, 0) + D(4, 1)) + D(5, 2)};
        for (int d = 0; d < 3; d++) {
          if (special >= 0) {
            CHECK(3 * a.ncls[special] + d < a.cforce0);
            w[d] = w[d] + (T)force[3 * a.ncls[special] + d];
          }
          V[t][3 * i + d] = V[t][3 * i + d] + idt * w[d];
        }
        if (special >= 0 && (r[3] & kResidentOwner) && a.v.sp_sens[special] >= 0)
          for (int d = 0; d < 3; d++)
            a.v.trace[(size_t)k * a.row + 3 * a.v.sp_sens[special] + d] = (double)V[t][3 * i + d];
      }
    }
    for (int t = 0; t < a.ntiles; t++) {
      const ResidentTile& tl = a.tiles[t];
      for (int i = 0; i < tl.ncell; i++) {
        const uint32_t* r = &a.crec[4 * (size_t)(tl.cell0 + i)];
        const int e = (int)r[3];
        int c[8];
        links(r, c);
        for (int q : c) CHECK(q < tl.nnode);
        T sp[3], cc[21];
        int special = -1;
        if (a.s.key || a.s.lkey) {
          uint32_t w = key(a.s, e);
          if (w & kSpecialKey) {
            special = (int)(w & ~kSpecialKey);
            w = a.s.sp_key[special];
          }
          for (int q = 0; q < 21; q++) cc[q] = a.s.cls[(size_t)(w >> kMatShift) * kMatRow + q];
          for (int d = 0; d < 3; d++) sp[d] = a.s.axis[d * kAxisClasses + (w >> (14 - 7 * d) & (kAxisClasses - 1))];
        } else {
          const int width = a.s.crow ? kAxialEntries : 21;
          for (int j = 0; j < 21; j++) {
            const int q = a.s.crow ? axial_entry(j) : j;
            cc[j] = q < 0 ? a.s.crow[j]
                          : a.s.C[a.s.ldc ? (int64_t)q * a.s.ldc + e : ((int64_t)(e >> 6) * width + q) * 64 + (e & 63)];
          }
          sp[0] = a.s.dcx[e], sp[1] = a.s.dcy[e], sp[2] = a.s.dcz[e];
          if (std::isnan(sp[0])) {
            uint64_t bits = 0;
            std::memcpy(&bits, &sp[0], sizeof(T));
            special = (int)(bits & (sizeof(T) == 8 ? 0xFFFFFFFFull : 0x3FFFFFull));
            sp[0] = a.s.sp_dcx[special];
          }
        }
        auto D = [&](int q, int ax) {
          T f[8];
          for (int b = 0; b < 8; b++) f[b] = V[t][3 * c[b] + q];
          return d_of(f, ax, sp[ax]);
        };
        const T g[6] = {D(0, 0), D(1, 1), D(2, 2), D(2, 1) + D(1, 2), D(2, 0) + D(0, 2), D(1, 0) + D(0, 1)};
        for (int q = 0; q < 6; q++) {
          const int ks = kSlot[q];
          T acc = cc[tri(ks, 0)] * g[0] + cc[tri(ks, 1)] * g[1] + cc[tri(ks, 2)] * g[2] + cc[tri(ks, 3)] * g[3] +
                  cc[tri(ks, 4)] * g[4] + cc[tri(ks, 5)] * g[5];
          double m = 0.0;
          if (special >= 0) {
            CHECK(a.cforce0 + 6 * a.ccls[special] + ks < a.nforce);
            m = force[a.cforce0 + 6 * a.ccls[special] + ks];
          }
          T& s = S[t][6 * i + q];
          if (sizeof(T) == 8) {
            if (special >= 0) acc = acc + (T)m;
            s = s + a.s.dt * acc;
          } else {
            if (special >= 0) acc = acc + (T)((double)a.s.dt * m);
            s = s + acc;
          }
          if (i < tl.nexp && k + 1 < a.nsteps) xb[at(a, (k + 1) % 4, tl.exp0 + i, q)] = s;
        }
      }
    }
  }
  std::vector<char> cell(a.s.n, 0), node(a.v.n, 0);
  for (int t = 0; t < a.ntiles; t++) {
    const ResidentTile& tl = a.tiles[t];
    for (int i = 0; i < tl.ncell; i++) {
      const int e = (int)a.crec[4 * (size_t)(tl.cell0 + i) + 3];
      cell[e]++;
      for (int q = 0; q < 6; q++) Sg[kSlot[q]][e] = S[t][6 * i + q];
    }
    for (int i = 0; i < tl.nnode; i++) {
      const uint32_t w = a.nrec[4 * (size_t)(tl.node0 + i) + 3];
      if (!(w & kResidentOwner)) continue;
      node[w & ~kResidentOwner]++;
      for (int d = 0; d < 3; d++) Vg[d][w & ~kResidentOwner] = V[t][3 * i + d];
    }
  }
  for (char n : cell) CHECK(n == 1);  // each cell and node is written by exactly one tile
  for (char n : node) CHECK(n == 1);
  return hipSuccess;
}

}  // namespace

// RESIDENT_CUS compute units (default 256) with 160 KiB of LDS each.
hipError_t resident_limits(int* cus, size_t* lds) {
  const char* e = std::getenv("RESIDENT_CUS");
  *cus = e ? std::atoi(e) : 256;
  *lds = 160 * 1024;
  return hipSuccess;
}
hipError_t resident_after(hipStream_t, hipEvent_t) { return hipSuccess; }
hipError_t launch_resident_f64(const ResidentArgs<double>& a, int threads, hipStream_t) { return run(a, threads); }
hipError_t launch_resident_f32(const ResidentArgs<float>& a, int threads, hipStream_t) { return run(a, threads); }

// State transfers, as rsg_state.hip makes them.
template <typename T>
static hipError_t state(const StateArgs<T>& a, int64_t g0, int n, T* chunk, bool write) {
  CHECK(n > 0 && n <= kStateChunk && g0 >= 0 && g0 + n <= (int64_t)3 * a.nn + (int64_t)6 * a.nc);
  for (int i = 0; i < n; i++) {
    const int64_t g = g0 + i, v = (int64_t)3 * a.nn;
    T* x = g < v ? a.V[g / a.nn] + a.node_at[g % a.nn] : a.S[(g - v) / a.nc] + a.cell_at[(g - v) % a.nc];
    if (write)
      *x = chunk[i];
    else
      chunk[i] = *x;
  }
  return hipSuccess;
}
hipError_t launch_state_f64(const StateArgs<double>& a, int64_t g0, int n, double* c, bool w, hipStream_t) {
  return state(a, g0, n, c, w);
}
hipError_t launch_state_f32(const StateArgs<float>& a, int64_t g0, int n, float* c, bool w, hipStream_t) {
  return state(a, g0, n, c, w);
}

}  // namespace rsg
