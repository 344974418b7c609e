// rsg_internal.h -- device-side layout shared by the host code (rsg_host.cpp) and the
// kernels (rsg_kernels.hip).  Not part of the public ABI.
#pragma once

#include <hip/hip_runtime_api.h>

#include <cstdint>
#include <cstring>

namespace rsg {

// Kernel argument blocks.  All arrays are in the library's internal (locality) order.
//
// Coefficients come in one of two forms per kernel:
//  * class tables (key != nullptr): each entity holds a 32-bit key made of a material
//    class (bits 21..30: the cell's row of 21 C, or the node's dt/rho) and one spacing
//    class per axis (7 bits each: x at bit 14, y at bit 7, z at bit 0).  The material rows
//    and the three spacing tables are small and read through the caches; a wavefront's
//    cells usually share one material row, so those loads coalesce.  A key with bit 31 set
//    flags a special entity (source or sensor): its low bits index the special tables,
//    which hold the entity's full key;
//  * per-entity arrays (key == nullptr), for meshes with more than 1024 materials or 128
//    spacings along an axis: source and sensor entities are flagged without any extra
//    array, a node's dt/rho (idt) or a cell's x-spacing (dcx) being replaced by a quiet NaN
//    whose payload is the special index, and the special tables hold the real value.
// Either way ordinary entities cost no extra HBM bytes for the flag.
constexpr uint32_t kSpecialKey = 0x80000000u;
constexpr int kMatShift = 21;
constexpr int kMaxMaterials = 1024;
constexpr int kAxisClasses = 128;  // spacing classes per axis; tables are [3][kAxisClasses]
// Entries of the 21 that a material with axes along the coordinate axes has (C11, C12, C13, C22, C23,
// C33, C44, C55, C66).  Per-cell arrays hold these alone where each of the others is the same for
// all cells, as in a part whose stiffness varies but not its symmetry: 72 of 168 bytes a cell.
constexpr int kAxialEntries = 9;
constexpr int axial_entry(int j) {  // its place among them, or -1
  return j < 3 ? j : j == 6 ? 3 : j == 7 ? 4 : j == 11 ? 5 : j == 15 ? 6 : j == 18 ? 7 : j == 20 ? 8 : -1;
}
constexpr int kMatRow = 24;        // cell material row: the 21 C as the C array holds them, padded
constexpr uint32_t kNoLink = 0x3FF;  // packed 10-bit link: no neighbour
constexpr int kMaxPackedSet = 1022;  // largest staged set whose local indices fit 10 bits

// LDS of a velocity workgroup: 6 stress rows of max_u + 1 entries, the last one a zero that
// links to missing cells read.
inline size_t velocity_lds_bytes(int max_u, size_t elt) { return (size_t)6 * (max_u + 1) * elt; }

// First word of a batch work item: the instance slot (18 bits) and the number of steps of the
// current K-step block it takes (kmax <= 4096, bits 18..30, so the word stays non-negative);
// -1 marks an empty item.
constexpr int kItemSlotBits = 18;
constexpr int32_t kMaxBatchSlots = 1 << kItemSlotBits;
inline int32_t batch_item_word(int32_t slot, int32_t kmax) { return slot | (kmax << kItemSlotBits); }

inline uint32_t make_key(int mat, int ix, int iy, int iz) {
  return ((uint32_t)mat << kMatShift) | ((uint32_t)ix << 14) | ((uint32_t)iy << 7) | (uint32_t)iz;
}
template <typename T>
struct VelocityArgs {
  T* V0;
  T* V1;
  T* V2;
  const T* S0;  // Sxx
  const T* S1;  // Syy
  const T* S2;  // Szz
  const T* S3;  // Syz
  const T* S4;  // Sxz
  const T* S5;  // Sxy
  const T* idt;  // dt/rho_n, NaN-boxed for special nodes
  const T* dnx;  // FP64: node spacing dxn; FP32: 0.25/dxn
  const T* dny;
  const T* dnz;
  const int32_t* ncell;  // [n][8] connected cells by slot, -1 = none
  int32_t n;
  int32_t xcd;  // 1: remap workgroups so each XCD owns a contiguous range
  int32_t cpt;  // entities per thread: a workgroup covers cpt * blockDim.x nodes
  int32_t stream;  // 1: non-temporal loads of what a step reads once (links, keys, lists)
  // LDS staging (lconn != nullptr): per-block unique cell lists and 16-bit local links
  const int32_t* u_off;    // [nblocks+1]
  const int32_t* ulist;    // cells staged by each block
  const uint16_t* lconn;   // [n][8] block-local cell index by slot, 0xFFFF = none
  int32_t max_u;           // largest unique set of a block (LDS rows hold max_u + 1)
  int32_t uchunk;          // 1: ulist holds chunk words, start << 2 | (len - 1): runs of up to 4
                           // consecutive cells, each taking 4 LDS slots (slot 4c + k holds
                           // start + k for k < len); max_u and the links count slots
  // special nodes (sources and/or sensors)
  const T* sp_idt;         // [nsp] real dt/rho_n
  const int32_t* sp_off;   // [nsp][4] term ranges for directions 0,1,2
  const int32_t* sp_sens;  // [nsp] sensor slot or -1
  const int32_t* term;     // channel id per term
  const double* amp;       // [n_channels] amplitudes of this step
  double* trace;           // [n_sensors][3] row of this step
  // class tables (key or lkey != nullptr: idt, dnx..dnz and sp_idt are not used)
  const uint32_t* key;     // [n] material/spacing key, or kSpecialKey | special index
  const T* cls;            // [materials] dt/rho
  const T* axis;           // [3][kAxisClasses] node spacings as dnx..dnz hold them
  const uint32_t* sp_key;  // [nsp] key of each special node
  // LDS links and key in one 16-byte record (lkey != nullptr: lconn and key are not used):
  // words 0..2 hold the 8 block-local indices, 10 bits each (3 per word, kNoLink = none),
  // word 3 the key
  const uint32_t* lkey;    // [n][4]
};

template <typename T>
struct StressArgs {
  T* S0;
  T* S1;
  T* S2;
  T* S3;
  T* S4;
  T* S5;
  const T* V0;
  const T* V1;
  const T* V2;
  const T* C;    // [21][ldc]: FP64 C_IJ; FP32 dt*C_IJ (FP64 product, rounded)
  int64_t ldc;   // leading dimension of C (>= n), or 0 for the 64-cell blocked layout
  const T* crow;  // [21], where C holds kAxialEntries per cell: what the others are for all cells
  const T* dcx;  // FP64: cell spacing dxc (NaN-boxed for special cells); FP32: 0.25/dxc
  const T* dcy;
  const T* dcz;
  const int32_t* cnode;  // [n][8] vertices
  int32_t n;
  int32_t xcd;
  int32_t cpt;             // cells per thread
  int32_t stream;          // as for VelocityArgs (and the per-cell C)
  const int32_t* u_off;    // LDS staging: per-block unique node lists
  const int32_t* ulist;
  const uint16_t* lconn;   // [n][8] block-local vertex index
  int32_t max_u;
  T dt;  // used by the FP64 form only
  // special cells (stress sources)
  const T* sp_dcx;        // [nsp] real x-spacing value
  const int32_t* sp_off;  // [nsp][7] term ranges for Voigt components 0..5
  const int32_t* term;
  const double* amp;
  // class tables (key or lkey != nullptr: C, dcx..dcz and sp_dcx are not used)
  const uint32_t* key;     // [n] material/spacing key, or kSpecialKey | special index
  const T* cls;            // [materials][kMatRow]
  const T* axis;           // [3][kAxisClasses] cell spacings as dcx..dcz hold them
  const uint32_t* sp_key;  // [nsp] key of each special cell
  const uint32_t* lkey;    // [n][4] LDS links + key, as for VelocityArgs
};

// Energy arguments (rsg_energy.hip): FP64 accumulation, one partial per workgroup.
constexpr int kEnergyMaxBlocks = 1024;
template <typename T>
struct EnergyArgs {
  const T* V0;
  const T* V1;
  const T* V2;
  const double* node_m;    // node mass rho_n * dxn*dyn*dzn (FP64)
  int32_t nn;
  StressArgs<T> s;         // the stress kernel's arguments: S, n and the coefficient form
  const double* cell_vol;  // dxc*dyc*dzc (FP64)
  double inv_scale;        // 1 (FP64: C stored as C_IJ) or 1/dt (FP32: stored as dt*C_IJ)
  double* partial;         // [2][nblocks]
};

// One instance of a batch: its argument blocks plus where this K-step block's
// amplitudes and traces go.
template <typename T>
struct BatchDesc {
  VelocityArgs<T> v;
  StressArgs<T> s;
  const double* amp_base;  // [K][nch] amplitudes of the current K-step block
  double* trace_base;      // the instance's trace buffer, [rows][row] (nullptr: no sensors)
  int32_t nch;
  int32_t row;             // 3 * sensors
  int64_t trace_row0;      // first trace row of this K-step block
  int32_t kmax;            // steps of this K-step block the instance takes
  int32_t pad;
};

// Launchers (rsg_kernels.hip).  block = threads per block (64..1024, multiple of 64).
hipError_t launch_velocity_f64(const VelocityArgs<double>& a, int block, hipStream_t s);
hipError_t launch_velocity_f32(const VelocityArgs<float>& a, int block, hipStream_t s);
hipError_t launch_stress_f64(const StressArgs<double>& a, int block, hipStream_t s);
hipError_t launch_stress_f32(const StressArgs<float>& a, int block, hipStream_t s);
// Batched launch: grid workgroups walk table = n (instance, block) int32 pairs in launch
// order, 8-byte aligned, (-1, 0) for an empty item; lds selects LDS staging (max_u: the
// largest staged set of any instance), cpt the entities per thread (1, 2 or 4), km the
// coefficient form of every instance the table names (0 per-entity arrays, 1 class-table
// keys, 3 keys packed with the LDS links; kBatchCached added: ordinary loads of what a step
// reads once).  With graph != nullptr the launch is added to
// the graph as a kernel node that depends on *node (when not null) and *node becomes the
// new node; otherwise it is enqueued on s.
constexpr int kBatchCached = 8;
hipError_t launch_batch_f64(const BatchDesc<double>* d, const int32_t* table, int n, int k, int grid, int block,
                            bool lds, int max_u, int cpt, int km, bool velocity, hipStream_t s, hipGraph_t graph,
                            hipGraphNode_t* node);
hipError_t launch_batch_f32(const BatchDesc<float>* d, const int32_t* table, int n, int k, int grid, int block,
                            bool lds, int max_u, int cpt, int km, bool velocity, hipStream_t s, hipGraph_t graph,
                            hipGraphNode_t* node);
// Energy: partials into a.partial, then their fixed-order sum into out[0] (kinetic) and
// out[1] (strain); both device addresses.  nblocks <= kEnergyMaxBlocks.
hipError_t launch_energy_f64(const EnergyArgs<double>& a, int nblocks, double* out, hipStream_t s);
// Device address of the static work area of the allocation-free energy on `device` (2 *
// kEnergyMaxBlocks + 2 doubles), resolved with hipGetSymbolAddress on first use per device.
hipError_t energy_scratch(int device, double** out);
// Largest node or cell count the energy kernels' grid-stride indexing takes.
constexpr int32_t kEnergyMaxEntities = 0x7FFFFFFF - kEnergyMaxBlocks * 256;
hipError_t launch_energy_f32(const EnergyArgs<float>& a, int nblocks, double* out, hipStream_t s);

// ---------------------------------------------------------------- resident stepping
// Many steps in one launch (rsg_resident.hip): the mesh is cut into tiles of cells, one
// workgroup per tile, all of them on the GPU at once.  A tile holds the stresses of its cells
// and the velocities of its nodes (every vertex of its cells) in LDS for the whole launch, and
// each step reads from memory only the stresses of its halo: the other tiles' cells at its
// nodes.
constexpr int kResidentSlots = 4095;  // 12-bit local links: slot numbers stay at or below this

// One tile: ranges of the plan's arrays.  The exported cells (in some other tile's halo) come
// first among its cells, and the nodes whose 8 cells are all its own first among its nodes.
struct ResidentTile {
  int32_t cell0, ncell, nexp;  // cell records; how many of them are exported
  int32_t node0, nnode, nown;  // node records; how many of them touch no halo cell
  int32_t halo0, nhalo;        // halo entries
  int32_t exp0;                // exchange slot of the tile's first exported cell
  int32_t pad;
};
constexpr uint32_t kResidentOwner = 0x80000000u;  // node record: this tile writes the node's results

// Source terms: the special nodes (cells) with the same lists of channel terms share a class, and
// the host sums each class's terms once per step, 3 (6) values a class: a row of 3 * node classes
// + 6 * cell classes doubles.  Class numbers stay below 128.
constexpr int kResidentForces = 256;  // largest row
constexpr uint8_t kResidentSensor = 0x80;  // node mark: a sensor this tile records

// Status words: the last decision that a launch of several tiles came to, 2 seq + 1 when its steps are
// made and 2 seq when its tiles did not get onto the GPU together and nothing is written; 1 when a wait
// between tiles ran out (the state is lost).
constexpr int kResidentDecision = 0, kResidentLost = 1, kResidentStatus = 2;

template <typename T>
struct ResidentArgs {
  VelocityArgs<T> v;  // state, coefficients, sources and sensors as the per-step kernels take them
  StressArgs<T> s;    // (amp and trace: the first step's)
  const ResidentTile* tiles;
  const uint32_t* crec;  // [cells][4]: 8 x 12-bit local node indices, internal cell id
  const uint32_t* nrec;  // [tile nodes][4]: 8 x 12-bit local cell slots (own cells, halo, then the
                         // zero slot of missing cells), internal node id | kResidentOwner
  const int32_t* halo;   // exchange slot of each halo cell
  const int32_t* hcell;  // internal id of each halo cell
  unsigned long long* xbuf;  // [4][6 * sizeof(T) / 8][nexp]: exported stresses of four steps in turn
  uint32_t* ctrl;        // [2] (several tiles): tiles started, over all launches; the last decision
  uint32_t seq;          // number of the launch, from 1
  int32_t* status;       // [kResidentStatus], pinned
  int32_t nsteps;        // >= 2
  int32_t ntiles;
  int32_t nexp;
  int32_t max_set;       // largest number of slots of a tile, without the zero slot
  int32_t max_node;
  int32_t max_cell;
  uint32_t* work;        // [tiles][max_node + max_cell][4] when the records do not fit LDS, else null
  const double* force;   // [nsteps][nforce] summed source terms
  int32_t nforce;
  const uint8_t* ncls;   // class of each special node, 0 .. node classes - 1
  const uint8_t* ccls;   // class of each special cell
  int32_t cforce0;       // first cell value of a force row
  int32_t row;           // doubles from one step's trace row to the next's
  int32_t nmat;          // values of dt/rho in v.cls
  int32_t tables;        // 1: the class tables' spacings and dt/rho are held in LDS
  int32_t chained;       // 1: the host does not know the decision on the launch before; if that was
                         // refused, so is this one (for the launcher)
};

// The class tables in LDS, for meshes of at most kResidentClasses spacings along each axis and
// values of dt/rho: node and cell spacings (FP64: with their reciprocals) and dt/rho.
constexpr int kResidentClasses = 16;
inline size_t resident_table_bytes(size_t elt) {
  return kResidentClasses * ((size_t)6 * (elt == 8 ? 32 : 4) + elt);
}

// LDS of a tile's workgroup: its slots' stresses, its nodes' velocities, the marks and, with
// `records`, the records; without, the kernel keeps those in `work`.
inline size_t resident_lds_bytes(int max_set, int max_node, int max_cell, size_t elt, bool records) {
  const size_t state = ((size_t)6 * (max_set + 1) + (size_t)3 * max_node) * elt;
  return ((state + 15) / 16 * 16 + (size_t)(records ? 17 : 1) * (max_node + max_cell) + 15) / 16 * 16;
}
constexpr size_t kResidentStaticLds = 2 * kResidentForces * 8 + 192;  // and what it declares itself

// These launchers, and those of the state transfers, may be left out of builds of the host code alone
// (the sanitizers'), which step with the per-step kernels and reorder states on the host.  The
// library is built with RSG_LIBRARY, where one that is missing fails the link.
#ifdef RSG_LIBRARY
#define RSG_WEAK
#else
#define RSG_WEAK __attribute__((weak))
#endif
template <typename F>
bool linked(F* launcher) {
  return launcher != nullptr;
}
// Compute units of the current device, and LDS bytes a workgroup may take.
RSG_WEAK hipError_t resident_limits(int* cus, size_t* lds);
// Work queued on s from now on waits for the event.
RSG_WEAK hipError_t resident_after(hipStream_t s, hipEvent_t e);
// Drops the thread's last HIP error, where what failed is done without: the launchers that ask for
// the last error would report it as theirs.
RSG_WEAK void forget_error();
// threads: 256, 512 or 1024 per workgroup.
RSG_WEAK hipError_t launch_resident_f64(const ResidentArgs<double>& a, int threads, hipStream_t s);
RSG_WEAK hipError_t launch_resident_f32(const ResidentArgs<float>& a, int threads, hipStream_t s);

// ---------------------------------------------------------------- state transfers (rsg_state.hip)
template <typename T>
struct StateArgs {
  T* V[3];
  T* S[6];
  const int32_t* node_at;  // caller -> internal
  const int32_t* cell_at;
  int32_t nn, nc;
};
constexpr int kStateChunk = 1 << 18;  // values a chunk holds
// Moves values [g0, g0 + n) of the caller's V[3][nn], S[6][nc] from the state to a chunk of pinned
// host memory, or with `write` from the chunk to the state.
RSG_WEAK hipError_t launch_state_f64(const StateArgs<double>& a, int64_t g0, int n, double* chunk, bool write,
                                     hipStream_t s);
RSG_WEAK hipError_t launch_state_f32(const StateArgs<float>& a, int64_t g0, int n, float* chunk, bool write,
                                     hipStream_t s);

// NaN boxing of a special-table index.
inline double box_f64(int32_t idx) {
  uint64_t b = 0x7FF8000000000000ull | (uint64_t)(uint32_t)idx;
  double d;
  std::memcpy(&d, &b, 8);
  return d;
}
inline float box_f32(int32_t idx) {
  uint32_t b = 0x7FC00000u | (uint32_t)idx;
  float f;
  std::memcpy(&f, &b, 4);
  return f;
}
constexpr int32_t kMaxSpecialF32 = (1 << 22) - 1;

}  // namespace rsg
