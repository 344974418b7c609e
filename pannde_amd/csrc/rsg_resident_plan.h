// rsg_resident_plan.h -- cuts a mesh into the tiles of the resident kernel (rsg_resident.hip)
// and builds their records.  Host code.
#pragma once

#include <algorithm>
#include <atomic>
#include <cmath>
#include <cstdint>
#include <cstdlib>
#include <cstring>
#include <memory>
#include <new>
#include <utility>
#include <vector>

#include "rsg_internal.h"

namespace rsg {

struct ResidentMesh {
  int32_t nn, nc;
  const int32_t* cells;       // [nc][8] vertices, caller numbering
  const int32_t* node_cells;  // [nn][8] cells, -1 = none
  const int32_t* cell_of;     // internal -> caller
  const int32_t* cell_at;     // caller -> internal
  const int32_t* node_at;
  const double* x[3];
  double lo[3], h[3];  // corner and finest spacing of the mesh
};

// The plan's arrays as one block of bytes, each on a 256-byte boundary, so that they go to the device
// with one allocation and one copy.
struct ResidentPlan {
  int32_t ntiles = 0, nexp = 0, max_set = 0, max_node = 0, max_cell = 0;
  size_t tiles = 0, halo = 0, hcell = 0, nrec = 0, crec = 0, ctrl = 0, bytes = 0;  // offsets, total
  std::unique_ptr<char[]> block;
};

inline void pack12(const int (&l)[8], uint32_t* w) {
  w[0] = (uint32_t)l[0] | (uint32_t)l[1] << 12 | (uint32_t)l[2] << 24;
  w[1] = (uint32_t)l[2] >> 8 | (uint32_t)l[3] << 4 | (uint32_t)l[4] << 16 | (uint32_t)l[5] << 28;
  w[2] = (uint32_t)l[5] >> 4 | (uint32_t)l[6] << 8 | (uint32_t)l[7] << 20;
}

// Zeroed memory that is not touched until it is written.
struct ZeroTags {
  int32_t* p;
  explicit ZeroTags(size_t n) : p(static_cast<int32_t*>(std::calloc(n, sizeof(int32_t)))) {
    if (!p) throw std::bad_alloc();
  }
  ~ZeroTags() { std::free(p); }
  ZeroTags(const ZeroTags&) = delete;
  ZeroTags& operator=(const ZeroTags&) = delete;
};

// Cells to tiles, about nc / max_tiles each: slabs of equal cell counts along x, each cut the same
// way along y and each piece along z.  The counts per axis minimise what a tile of the mesh's
// extents computes and stages.  Returns the number of tiles used (empty ones are skipped).
template <typename Run>
int32_t resident_tiles(const ResidentMesh& m, int32_t max_tiles, Run&& run, std::vector<int32_t>& tile_of) {
  constexpr int32_t kBins = 4096;  // planes told apart along an axis
  const int tasks = (int)std::min<int64_t>(64, (m.nc + (1 << 15) - 1) / (1 << 15));
  const int64_t step = ((int64_t)m.nc + tasks - 1) / tasks;
  // planes: a cell's first vertex in units of the finest spacing, coarser for longer meshes
  std::vector<uint16_t> plane[3];
  double width[3];
  for (int d = 0; d < 3; d++) {
    plane[d].resize(m.nc);
    double hi = m.lo[d];
    for (int32_t n = 0; n < m.nn; n++) hi = std::max(hi, m.x[d][n]);
    width[d] = std::max(m.h[d], (hi - m.lo[d]) / (kBins - 1));
  }
  run(tasks, [&](int w) {
    for (int64_t c = w * step; c < std::min<int64_t>(m.nc, (w + 1) * step); c++)
      for (int d = 0; d < 3; d++) {
        const double q = (m.x[d][m.cells[8 * c]] - m.lo[d]) / width[d] + 0.5;
        plane[d][c] = (uint16_t)(q > 0 ? std::min(q, kBins - 1.0) : 0.0);
      }
  });
  // histograms over the planes there are: a mesh of 40 planes has bins for 40
  int32_t ext[3], bins[3];
  std::vector<int64_t> count[3];
  for (int d = 0; d < 3; d++) {
    bins[d] = 1 + *std::max_element(plane[d].begin(), plane[d].end());
    count[d].assign(bins[d], 0);
    for (int32_t c = 0; c < m.nc; c++) count[d][plane[d][c]]++;
    ext[d] = (int32_t)std::count_if(count[d].begin(), count[d].end(), [](int64_t v) { return v > 0; });
  }
  const double fill = (double)m.nc / ((double)ext[0] * ext[1] * ext[2]);
  int32_t p[3] = {1, 1, 1};
  double best = INFINITY;
  for (int32_t a = 1; a <= std::min(max_tiles, ext[0]); a++)
    for (int32_t b = 1; a * b <= max_tiles && b <= ext[1]; b++) {
      const int32_t c = std::min(max_tiles / (a * b), ext[2]);
      const double t[3] = {std::ceil((double)ext[0] / a), std::ceil((double)ext[1] / b), std::ceil((double)ext[2] / c)};
      const double cost = fill * t[0] * t[1] * t[2] + fill * (t[0] + 1) * (t[1] + 1) * (t[2] + 1) +
                          0.3 * (t[0] + 2) * (t[1] + 2) * (t[2] + 2);
      if (cost < best) {
        best = cost;
        p[0] = a, p[1] = b, p[2] = c;
      }
    }
  // piece of each of nb planes when their cells, cnt[q] per plane, are cut into n pieces
  auto cut = [](const int64_t* cnt, int32_t nb, int32_t n, uint16_t* piece) {
    int64_t total = 0, seen = 0;
    for (int32_t q = 0; q < nb; q++) total += cnt[q];
    for (int32_t q = 0; q < nb; q++) {
      // by the middle of the plane's cells, so whole planes go to the nearest piece
      piece[q] = total ? (uint16_t)std::min<int64_t>(n - 1, (int64_t)((seen + 0.5 * cnt[q]) * n / total)) : 0;
      seen += cnt[q];
    }
  };
  std::vector<uint16_t> px(bins[0]);
  cut(count[0].data(), bins[0], p[0], px.data());
  std::vector<int64_t> cy((size_t)p[0] * bins[1], 0);
  for (int32_t c = 0; c < m.nc; c++) cy[(size_t)px[plane[0][c]] * bins[1] + plane[1][c]]++;
  std::vector<uint16_t> py(cy.size());
  for (int32_t a = 0; a < p[0]; a++) cut(&cy[(size_t)a * bins[1]], bins[1], p[1], &py[(size_t)a * bins[1]]);
  auto column = [&](int32_t c) {
    const int32_t a = px[plane[0][c]];
    return a * p[1] + py[(size_t)a * bins[1] + plane[1][c]];
  };
  std::vector<int64_t> cz((size_t)p[0] * p[1] * bins[2], 0);
  for (int32_t c = 0; c < m.nc; c++) cz[(size_t)column(c) * bins[2] + plane[2][c]]++;
  std::vector<uint16_t> pz(cz.size());
  for (int32_t k = 0; k < p[0] * p[1]; k++) cut(&cz[(size_t)k * bins[2]], bins[2], p[2], &pz[(size_t)k * bins[2]]);
  tile_of.resize(m.nc);
  std::vector<int32_t> number((size_t)p[0] * p[1] * p[2], -1);
  int32_t n = 0;
  for (int32_t c = 0; c < m.nc; c++) {
    const int32_t k = column(c);
    int32_t& id = number[(size_t)k * p[2] + pz[(size_t)k * bins[2] + plane[2][c]]];
    if (id < 0) id = n++;
    tile_of[c] = id;
  }
  return n;
}

// The plan for at most max_tiles tiles; false when some tile does not fit (too many slots for
// 12-bit links, or more LDS than lds_limit) or the mesh has a node that no cell uses.  run(n, fn)
// calls fn(0) .. fn(n - 1), on threads.
template <typename Run>
bool build_resident_plan(const ResidentMesh& m, int32_t max_tiles, size_t lds_limit, size_t elt, Run&& run,
                         ResidentPlan& p) {
  std::vector<int32_t> tile_of;
  const int32_t nt = resident_tiles(m, max_tiles, run, tile_of);
  const int tasks = (int)std::min<int64_t>(64, ((int64_t)m.nc + (1 << 15) - 1) / (1 << 15));
  // nodes of more than one tile, and each node's owner (the tile of its first cell)
  std::vector<int32_t> owner(m.nn);
  std::vector<char> shared(m.nn);
  std::atomic<bool> ok{true};
  const int64_t nstep = ((int64_t)m.nn + tasks - 1) / tasks;
  run(tasks, [&](int w) {
    for (int64_t n = w * nstep; n < std::min<int64_t>(m.nn, (w + 1) * nstep); n++) {
      int32_t own = -1;
      char sh = 0;
      for (int k = 0; k < 8; k++) {
        const int32_t c = m.node_cells[8 * n + k];
        if (c < 0) continue;
        if (own < 0) own = tile_of[c];
        if (tile_of[c] != own) sh = 1;
      }
      if (own < 0) ok = false;
      owner[n] = own;
      shared[n] = sh;
    }
  });
  if (!ok) return false;
  // cells by tile, in internal order, the exported ones (with a shared vertex) first
  std::vector<char> exported(m.nc);
  const int64_t cstep = ((int64_t)m.nc + tasks - 1) / tasks;
  run(tasks, [&](int w) {
    for (int64_t c = w * cstep; c < std::min<int64_t>(m.nc, (w + 1) * cstep); c++) {
      char e = 0;
      for (int v = 0; v < 8; v++) e |= shared[m.cells[8 * c + v]];
      exported[c] = e;
    }
  });
  std::vector<ResidentTile> tiles(nt, ResidentTile{});
  for (int32_t c = 0; c < m.nc; c++) {
    tiles[tile_of[c]].ncell++;
    tiles[tile_of[c]].nexp += exported[c];
  }
  p.nexp = 0;
  for (int32_t t = 0, at = 0; t < nt; t++) {
    tiles[t].cell0 = at;
    tiles[t].exp0 = p.nexp;
    at += tiles[t].ncell;
    p.nexp += tiles[t].nexp;
  }
  std::vector<int32_t> tile_cells(m.nc), slot(m.nc), next(2 * (size_t)nt);
  for (int32_t t = 0; t < nt; t++) {
    next[2 * t] = 0;
    next[2 * t + 1] = tiles[t].nexp;
  }
  for (int32_t i = 0; i < m.nc; i++) {
    const int32_t c = m.cell_of[i], t = tile_of[c];
    slot[c] = next[2 * t + (exported[c] ? 0 : 1)]++;
    tile_cells[(size_t)tiles[t].cell0 + slot[c]] = c;
  }
  // each tile's nodes, halo and links
  struct Part {
    std::vector<uint32_t> nrec, crec;
    std::vector<int32_t> halo, hcell;
  };
  std::vector<Part> parts(nt);
  const int groups = (int)std::min<int32_t>(nt, std::min<int64_t>(8, ((int64_t)m.nc + (1 << 13) - 1) >> 13));
  run(groups, [&](int g) {
    // a node's (cell's) number in the tile that saw it last, on top of that tile's base
    ZeroTags node_tags(m.nn), cell_tags(m.nc);
    int32_t *const node_tag = node_tags.p, *const cell_tag = cell_tags.p;
    int32_t node_base = 1, cell_base = 1;
    std::vector<int32_t> nodes;
    std::vector<std::pair<int32_t, int32_t>> around;  // exchange slot, cell
    for (int32_t t = (int32_t)((int64_t)nt * g / groups); t < (int32_t)((int64_t)nt * (g + 1) / groups); t++) {
      ResidentTile& tl = tiles[t];
      Part& part = parts[t];
      const int32_t* own = &tile_cells[tl.cell0];
      nodes.clear();
      for (int pass = 0; pass < 2; pass++) {  // nodes of this tile alone, then shared ones
        for (int32_t i = 0; i < (pass ? tl.nexp : tl.ncell); i++)
          for (int v = 0; v < 8; v++) {
            const int32_t n = m.cells[8 * (size_t)own[i] + v];
            if (shared[n] != pass || node_tag[n] >= node_base) continue;
            node_tag[n] = node_base + (int32_t)nodes.size();
            nodes.push_back(n);
          }
        if (pass == 0) tl.nown = (int32_t)nodes.size();
      }
      tl.nnode = (int32_t)nodes.size();
      // the halo in order of its exchange slots, so a wave reads runs of them
      around.clear();
      for (size_t i = tl.nown; i < nodes.size(); i++)
        for (int k = 0; k < 8; k++) {
          const int32_t c = m.node_cells[8 * (size_t)nodes[i] + k];
          if (c < 0 || tile_of[c] == t || cell_tag[c] >= cell_base) continue;
          cell_tag[c] = cell_base;
          around.emplace_back(tiles[tile_of[c]].exp0 + slot[c], c);
        }
      std::sort(around.begin(), around.end());
      for (auto& x : around) {
        cell_tag[x.second] = cell_base + (int32_t)part.halo.size();
        part.halo.push_back(x.first);
        part.hcell.push_back(m.cell_at[x.second]);
      }
      tl.nhalo = (int32_t)part.halo.size();
      const int32_t zero = tl.ncell + tl.nhalo;
      if (zero > kResidentSlots || tl.nnode > kResidentSlots + 1) {
        ok = false;
        return;
      }
      part.nrec.resize(nodes.size() * 4);
      for (size_t i = 0; i < nodes.size(); i++) {
        int l[8];
        for (int k = 0; k < 8; k++) {
          const int32_t c = m.node_cells[8 * (size_t)nodes[i] + k];
          l[k] = c < 0 ? zero : tile_of[c] == t ? slot[c] : tl.ncell + cell_tag[c] - cell_base;
        }
        pack12(l, &part.nrec[4 * i]);
        part.nrec[4 * i + 3] = (uint32_t)m.node_at[nodes[i]] | (owner[nodes[i]] == t ? kResidentOwner : 0);
      }
      part.crec.resize((size_t)tl.ncell * 4);
      for (int32_t i = 0; i < tl.ncell; i++) {
        int l[8];
        for (int v = 0; v < 8; v++) l[v] = node_tag[m.cells[8 * (size_t)own[i] + v]] - node_base;
        pack12(l, &part.crec[4 * (size_t)i]);
        part.crec[4 * (size_t)i + 3] = (uint32_t)m.cell_at[own[i]];
      }
      node_base += tl.nnode;
      cell_base += tl.nhalo;
    }
  });
  if (!ok) return false;
  int32_t node0 = 0, halo0 = 0;
  for (int32_t t = 0; t < nt; t++) {
    ResidentTile& tl = tiles[t];
    tl.node0 = node0;
    tl.halo0 = halo0;
    node0 += tl.nnode;
    halo0 += tl.nhalo;
    p.max_set = std::max(p.max_set, tl.ncell + tl.nhalo);
    p.max_node = std::max(p.max_node, tl.nnode);
    p.max_cell = std::max(p.max_cell, tl.ncell);
  }
  if (resident_lds_bytes(p.max_set, p.max_node, p.max_cell, elt, false) + kResidentStaticLds > lds_limit) return false;
  p.ntiles = nt;
  auto place = [&](size_t bytes) {
    const size_t at = p.bytes;
    p.bytes += (bytes + 255) / 256 * 256;
    return at;
  };
  p.tiles = place(sizeof(ResidentTile) * nt);
  p.halo = place((size_t)4 * halo0);
  p.hcell = place((size_t)4 * halo0);
  p.nrec = place((size_t)16 * node0);
  p.crec = place((size_t)16 * m.nc);
  p.ctrl = place(16);
  p.block.reset(new char[p.bytes]);
  std::memcpy(p.block.get() + p.tiles, tiles.data(), sizeof(ResidentTile) * nt);
  std::memset(p.block.get() + p.ctrl, 0, 16);
  auto put = [&](size_t at, const auto& v) {
    if (!v.empty()) std::memcpy(p.block.get() + at, v.data(), v.size() * sizeof(v[0]));
  };
  run(groups, [&](int g) {
    for (int32_t t = (int32_t)((int64_t)nt * g / groups); t < (int32_t)((int64_t)nt * (g + 1) / groups); t++) {
      put(p.halo + (size_t)4 * tiles[t].halo0, parts[t].halo);
      put(p.hcell + (size_t)4 * tiles[t].halo0, parts[t].hcell);
      put(p.nrec + (size_t)16 * tiles[t].node0, parts[t].nrec);
      put(p.crec + (size_t)16 * tiles[t].cell0, parts[t].crec);
      parts[t] = Part();
    }
  });
  return true;
}

}  // namespace rsg
