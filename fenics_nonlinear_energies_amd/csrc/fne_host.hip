// Host-side plan-construction helpers (plain C++, no device code).
#include <algorithm>
#include <cstring>
#include <new>
#include <vector>

#include "fne_common.h"

extern "C" int fne_color_patch_elements(int32_t n_patch, const int64_t* pelem_ptr, const int64_t* rows,
                                        int32_t n_loc, int64_t n_rows, int32_t* colors) {
  if (n_patch < 0 || n_loc <= 0 || n_rows < 0 || (n_patch > 0 && (!pelem_ptr || !rows || !colors))) {
    fne_set_error("fne_color_patch_elements: invalid arguments");
    return FNE_EINVAL;
  }
  // rows of different patches are disjoint, so one mask per row serves all patches
  std::vector<uint64_t> mask(size_t(n_rows), 0ull);
  int max_colors = 0;
  for (int32_t p = 0; p < n_patch; ++p) {
    int patch_colors = 0;
    for (int64_t i = pelem_ptr[p]; i < pelem_ptr[p + 1]; ++i) {
      uint64_t used = 0ull;
      for (int a = 0; a < n_loc; ++a) {
        const int64_t r = rows[i * n_loc + a];
        if (r >= 0) {
          if (r >= n_rows) {
            fne_set_error("fne_color_patch_elements: row index out of range");
            return FNE_EINVAL;
          }
          used |= mask[size_t(r)];
        }
      }
      if (used == ~0ull) {
        fne_set_error("fne_color_patch_elements: more than 64 colors needed in one patch");
        return FNE_EINVAL;
      }
      const int c = __builtin_ctzll(~used);
      colors[i] = c;
      if (c + 1 > patch_colors) patch_colors = c + 1;
      for (int a = 0; a < n_loc; ++a) {
        const int64_t r = rows[i * n_loc + a];
        if (r >= 0) mask[size_t(r)] |= (1ull << c);
      }
    }
    if (patch_colors > max_colors) max_colors = patch_colors;
  }
  return max_colors;
}

// Greedy distance-2 colouring (see include/fne_hip.h).  forbid[c] holds the last row for which
// colour c was found in the distance-2 neighbourhood, so the marks need no clearing between rows.
extern "C" int fne_color_distance2(int32_t n, const int32_t* indptr, const int32_t* indices, int32_t* colors) {
  if (n < 0 || (n > 0 && (!indptr || !indices || !colors))) {
    fne_set_error("fne_color_distance2: invalid arguments");
    return FNE_EINVAL;
  }
  if (n == 0) return 0;
  if (indptr[0] != 0) {
    fne_set_error("fne_color_distance2: indptr[0] must be 0");
    return FNE_EINVAL;
  }
  for (int32_t i = 0; i < n; ++i) {
    if (indptr[i + 1] < indptr[i]) {
      fne_set_error("fne_color_distance2: indptr must be non-decreasing");
      return FNE_EINVAL;
    }
  }
  const int64_t nnz = indptr[n];
  for (int64_t k = 0; k < nnz; ++k) {
    if (indices[k] < 0 || indices[k] >= n) {
      fne_set_error("fne_color_distance2: column index out of range");
      return FNE_EINVAL;
    }
  }
  for (int32_t i = 0; i < n; ++i) colors[i] = -1;
  std::vector<int32_t> forbid;
  int32_t n_colors = 0;
  for (int32_t v = 0; v < n; ++v) {
    for (int32_t k = indptr[v]; k < indptr[v + 1]; ++k) {
      const int32_t u = indices[k];
      if (colors[u] >= 0) forbid[size_t(colors[u])] = v;
      for (int32_t kk = indptr[u]; kk < indptr[u + 1]; ++kk) {
        const int32_t w = indices[kk];
        if (colors[w] >= 0) forbid[size_t(colors[w])] = v;
      }
    }
    int32_t c = 0;
    while (c < n_colors && forbid[size_t(c)] == v) ++c;
    if (c == n_colors) {
      forbid.push_back(-1);
      ++n_colors;
    }
    colors[v] = c;
  }
  return n_colors;
}

// ---------------------------------------------------------------------------------------------
// Node patches of the tetrahedral assembly (FneNodePatches).  Everything that the kernel indexes
// with is checked here: element codes, the 3x3 block structure of the CSR pattern, slots and
// positions within their bit fields.  A mesh that passes takes the patches in every node ordering:
// elements on patch borders are evaluated again by each patch (2.3 evaluations per element on the
// 320x16x16 beam in Morton order), four times at most, in a random one, and that still beats the
// row gather over stored element matrices (160x8x8 fused FP32: Morton 17.2 us against 45.7, random
// 28.2 against 49.4).
// ---------------------------------------------------------------------------------------------
namespace {

// host arrays to be placed in one device allocation, each at a multiple of 256 bytes
struct HostParts {
  struct Part {
    const void* src;
    size_t n, at;
  };
  std::vector<Part> parts;
  size_t bytes = 0;

  template <typename T>
  size_t add(const std::vector<T>& v) {
    const size_t n = v.size() * sizeof(T), at = bytes;
    parts.push_back(Part{v.data(), n, at});
    bytes += (n + 255) / 256 * 256;
    return at;
  }

  int upload(char** out, const char* name) const {
    char* base = nullptr;
    if (hipMalloc(&base, std::max<size_t>(bytes, 256)) != hipSuccess) {
      fne_set_error(std::string(name) + ": hipMalloc of the schedule failed");
      return FNE_ENOMEM;
    }
    for (const Part& p : parts)
      if (p.n && hipMemcpy(base + p.at, p.src, p.n, hipMemcpyHostToDevice) != hipSuccess) {
        (void)hipFree(base);
        fne_set_error(std::string(name) + ": upload of the schedule failed");
        return FNE_EHIP;
      }
    // on the null stream, which a caller's stream need not wait for: done when this returns
    if (hipStreamSynchronize(nullptr) != hipSuccess) {
      (void)hipFree(base);
      fne_set_error(std::string(name) + ": upload of the schedule failed");
      return FNE_EHIP;
    }
    *out = base;
    return FNE_OK;
  }
};

struct NodePatchHost {
  std::vector<int32_t> pnode, pelem_ptr, pelem, pelem_node, pown, pair_ptr, extra_ptr;
  std::vector<uint32_t> pair, diag;  // pair: two words per unit
  std::vector<uint16_t> pair_items, extra, diag_items;
};

int node_patch_unsupported(const char* why) {
  fne_set_error(std::string("fne_plan_build_node_patches: ") + why);
  return FNE_EUNSUPPORTED;
}

// index of the vertex pair (a, b), a != b, among 01 02 03 12 13 23
int tet_pair_index(int a, int b) {
  if (a > b) std::swap(a, b);
  return a == 0 ? b - 1 : (a == 1 ? b + 1 : 5);
}

int build_node_patches(const fne_plan_desc& d, const int32_t* edof, const int32_t* indptr, const int32_t* indices,
                       NodePatchHost& h) {
  const int32_t ne = d.n_elem, nf = d.n_free;
  if (nf % 3 != 0) return node_patch_unsupported("free DOFs do not come in node triples");
  const int32_t nn = nf / 3;
  std::vector<int32_t> enode(static_cast<size_t>(ne) * 4);
  std::vector<int32_t> min_node(static_cast<size_t>(ne), nn);
  std::vector<int32_t> inc_ptr(static_cast<size_t>(nn) + 1, 0);
  for (int32_t e = 0; e < ne; ++e) {
    for (int a = 0; a < 4; ++a) {
      const int32_t c = edof[size_t(3 * a) * ne + e];
      if (edof[size_t(3 * a + 1) * ne + e] != c + 1 || edof[size_t(3 * a + 2) * ne + e] != c + 2)
        return node_patch_unsupported("node components are not consecutive");
      if (c < 0 || c + 2 >= int64_t(nf) + d.n_total) return node_patch_unsupported("element code out of range");
      const bool free_node = c < nf;
      if (free_node ? (c % 3 != 0) : ((c - nf) % 3 != 0)) return node_patch_unsupported("node components are not aligned");
      const int32_t node = free_node ? c / 3 : nn + (c - nf) / 3;
      enode[size_t(e) * 4 + a] = node;
      if (free_node) {
        ++inc_ptr[size_t(node) + 1];
        min_node[e] = std::min(min_node[e], node);
      }
    }
    const int32_t* v = &enode[size_t(e) * 4];
    for (int a = 0; a < 4; ++a)
      for (int b = a + 1; b < 4; ++b)
        if (v[a] == v[b] && v[a] < nn) return node_patch_unsupported("an element names a node twice");
  }
  if (nn > 0 && indptr[0] != 0) return node_patch_unsupported("indptr[0] is not 0");
  h.diag.assign(size_t(nn), 0);
  for (int32_t i = 0; i < nn; ++i) {
    const int32_t k0 = indptr[3 * i], len = indptr[3 * i + 1] - k0;
    if (len <= 0 || len % 3 != 0 || len > 3 * 255) return node_patch_unsupported("CSR rows are not made of node blocks");
    bool diag = false;
    for (int r = 1; r <= 2; ++r)
      if (indptr[3 * i + r + 1] - indptr[3 * i + r] != len) return node_patch_unsupported("CSR rows of a node differ");
    for (int32_t b = 0; b < len / 3; ++b) {
      const int32_t c = indices[k0 + 3 * b];
      if (b > 0 && c <= indices[k0 + 3 * b - 3]) return node_patch_unsupported("CSR columns are not ascending");
      if (c < 0 || c >= nf || c % 3 != 0) return node_patch_unsupported("CSR columns are not made of node blocks");
      for (int r = 0; r < 3; ++r)
        for (int k = 0; k < 3; ++k)
          if (indices[k0 + r * len + 3 * b + k] != c + k) return node_patch_unsupported("CSR rows of a node differ");
      if (c == 3 * i) {
        h.diag[i] = uint32_t(b);
        diag = true;
      }
    }
    if (!diag) return node_patch_unsupported("a CSR row has no diagonal block");
  }
  for (int32_t i = 0; i < nn; ++i) inc_ptr[size_t(i) + 1] += inc_ptr[i];
  std::vector<int32_t> inc(static_cast<size_t>(inc_ptr[nn]));
  {
    std::vector<int32_t> at(inc_ptr.begin(), inc_ptr.end() - 1);
    for (int32_t e = 0; e < ne; ++e)
      for (int a = 0; a < 4; ++a) {
        const int32_t node = enode[size_t(e) * 4 + a];
        if (node < nn) inc[size_t(at[node]++)] = 4 * e + a;
      }
  }
  std::vector<int32_t> lone;  // elements without a free node: energy only
  for (int32_t e = 0; e < ne; ++e)
    if (min_node[e] == nn) lone.push_back(e);
  size_t next_lone = 0;
  std::vector<int32_t> seen(static_cast<size_t>(ne), -1), slot(static_cast<size_t>(ne), -1);
  std::vector<int32_t> pos_of(static_cast<size_t>(nn), -1);
  std::vector<int32_t> own, halo;
  std::vector<std::vector<uint16_t>> block_items(256);
  h.pnode.push_back(0);
  h.pelem_ptr.push_back(0);
  h.pair_ptr.push_back(0);
  // small meshes: fewer nodes per patch, so that 512 workgroups (two per CU) have one
  const int32_t max_nodes = std::clamp((nn + 511) / 512, 8, kNodePatchNodes);
  int32_t n0 = 0;
  while (n0 < nn || next_lone < lone.size()) {
    const int32_t p = int32_t(h.pnode.size()) - 1;
    own.clear();
    halo.clear();
    int32_t n1 = n0;
    while (n1 < nn && n1 - n0 < max_nodes) {
      int fresh = 0;
      for (int32_t k = inc_ptr[n1]; k < inc_ptr[n1 + 1]; ++k) fresh += seen[inc[k] >> 2] != p;
      if (int(own.size() + halo.size()) + fresh > kNodePatchElems) break;
      for (int32_t k = inc_ptr[n1]; k < inc_ptr[n1 + 1]; ++k) {
        const int32_t e = inc[k] >> 2;
        if (seen[e] == p) continue;
        seen[e] = p;
        (min_node[e] >= n0 ? own : halo).push_back(e);
      }
      ++n1;
    }
    if (n1 == n0 && n0 < nn) return node_patch_unsupported("a node has more elements than a patch holds");
    while (next_lone < lone.size() && int(own.size() + halo.size()) < kNodePatchElems) own.push_back(lone[next_lone++]);
    std::sort(own.begin(), own.end());
    std::sort(halo.begin(), halo.end());
    int32_t s = 0;
    for (int32_t e : own) slot[e] = s++;
    for (int32_t e : halo) slot[e] = s++;
    h.pelem.insert(h.pelem.end(), own.begin(), own.end());
    h.pelem.insert(h.pelem.end(), halo.begin(), halo.end());
    for (size_t k = size_t(h.pelem_ptr.back()); k < h.pelem.size(); ++k)
      for (int a = 0; a < 4; ++a) h.pelem_node.push_back(enode[size_t(h.pelem[k]) * 4 + a]);
    h.pelem_ptr.push_back(int32_t(h.pelem.size()));
    h.pown.push_back(int32_t(own.size()));
    const size_t extra0 = h.extra.size() / 8;
    h.extra_ptr.push_back(int32_t(extra0));
    for (int32_t i = n0; i < n1; ++i) {
      const int32_t k0 = indptr[3 * i], nb = (indptr[3 * i + 1] - k0) / 3;
      for (int32_t b = 0; b < nb; ++b) {
        pos_of[indices[k0 + 3 * b] / 3] = b;
        block_items[b].clear();
      }
      // item k of the diagonal goes to thread k % 8 of the node; items past 32 to extra blocks
      const int32_t items = inc_ptr[i + 1] - inc_ptr[i];
      const size_t diag_more = items > 32 ? size_t(items - 32 + 7) / 8 : 0, diag_off = h.extra.size() / 8 - extra0;
      if (diag_more > 255 || (diag_more > 0 && diag_off > 65535)) return node_patch_unsupported("a node has too many elements");
      h.diag[i] |= uint32_t(diag_more << 8) | uint32_t((diag_more ? diag_off : 0) << 16);
      h.diag_items.resize(size_t(i + 1) * 32, kNodePatchZero);
      for (int32_t k = inc_ptr[i]; k < inc_ptr[i + 1]; ++k) {
        const int32_t e = inc[k] >> 2, a = inc[k] & 3, t = k - inc_ptr[i];
        const uint16_t diag_item = uint16_t(slot[e] | (a << 9));
        if (t < 32)
          h.diag_items[size_t(i) * 32 + size_t(t % 8) * 4 + size_t(t / 8)] = diag_item;
        else
          h.extra.push_back(diag_item);
        for (int b = 0; b < 4; ++b) {
          const int32_t j = enode[size_t(e) * 4 + b];
          if (b == a || j >= nn) continue;
          const int32_t q = pos_of[j];
          if (q < 0) return node_patch_unsupported("element coupling missing from the CSR pattern");
          block_items[q].push_back(uint16_t(slot[e] | (a << 9) | (b << 11) | (tet_pair_index(a, b) << 13)));
        }
      }
      h.extra.resize((extra0 + diag_off + diag_more) * 8, kNodePatchZero);
      for (int32_t b = 0; b < nb; ++b) {
        const int32_t j = indices[k0 + 3 * b] / 3;
        pos_of[j] = -1;
        if (j == i) continue;
        uint32_t twin = kNodePatchNone;
        if (j >= n0 && j < n1) {  // both nodes in the patch: the block of (j, i) is its transpose
          const int32_t t0 = indptr[3 * j], t1 = indptr[3 * j + 1];
          const int32_t* at = std::lower_bound(indices + t0, indices + t1, 3 * i);
          if (at == indices + t1 || *at != 3 * i) return node_patch_unsupported("the CSR pattern is not symmetric");
          if (j < i) continue;  // written with (j, i)
          twin = uint32_t(j - n0) | (uint32_t((at - (indices + t0)) / 3) << 6);
        }
        const std::vector<uint16_t>& it = block_items[b];
        const size_t first = std::min<size_t>(it.size(), 8), more = (it.size() - first + 7) / 8;
        const size_t off = h.extra.size() / 8 - extra0;
        if (more > 15 || (more > 0 && off > 1023)) return node_patch_unsupported("an edge has too many elements");
        h.pair.push_back(uint32_t(i - n0) | (uint32_t(b) << 6) | (uint32_t(first) << 14) | (uint32_t(more) << 18) |
                         (uint32_t(more ? off : 0) << 22));
        h.pair.push_back(twin);
        for (size_t t = 0; t < 8; ++t) h.pair_items.push_back(t < first ? it[t] : kNodePatchZero);
        for (size_t t = 8; t < 8 + 8 * more; ++t) h.extra.push_back(t < it.size() ? it[t] : kNodePatchZero);
      }
    }
    h.pair_ptr.push_back(int32_t(h.pair.size() / 2));
    h.pnode.push_back(n1);
    n0 = n1;
  }
  return FNE_OK;
}

int upload_node_patches(fne_plan* plan, const NodePatchHost& h) {
  FneNodePatches np;
  np.n_patch = int(h.pnode.size()) - 1;
  HostParts parts;
  const size_t o_pnode = parts.add(h.pnode), o_pep = parts.add(h.pelem_ptr), o_pe = parts.add(h.pelem),
               o_pn = parts.add(h.pelem_node), o_po = parts.add(h.pown), o_pp = parts.add(h.pair_ptr),
               o_pr = parts.add(h.pair), o_pi = parts.add(h.pair_items), o_xp = parts.add(h.extra_ptr),
               o_x = parts.add(h.extra), o_di = parts.add(h.diag_items), o_dg = parts.add(h.diag);
  char* base = nullptr;
  const int up = parts.upload(&base, "fne_plan_build_node_patches");
  if (up != FNE_OK) return up;
  double2* partials = nullptr;
  if (np.n_patch > plan->n_partials && hipMalloc(&partials, sizeof(double2) * np.n_patch) != hipSuccess) {
    (void)hipFree(base);
    fne_set_error("hipMalloc of reduction scratch failed");
    return FNE_ENOMEM;
  }
  if (partials) {
    (void)hipFree(plan->partials);
    plan->partials = partials;
    plan->n_partials = np.n_patch;
  }
  // the assembly stores no element matrices any more (the element vectors stay, for fne_hvp)
  if (plan->mc_h) (void)hipFree(plan->mc_h);
  plan->mc_h = nullptr;
  np.storage = base;
  np.pnode = reinterpret_cast<int32_t*>(base + o_pnode);
  np.pelem_ptr = reinterpret_cast<int32_t*>(base + o_pep);
  np.pelem = reinterpret_cast<int32_t*>(base + o_pe);
  np.pown = reinterpret_cast<int32_t*>(base + o_po);
  np.pelem_node = reinterpret_cast<int4*>(base + o_pn);
  np.pair_ptr = reinterpret_cast<int32_t*>(base + o_pp);
  np.pair = reinterpret_cast<uint2*>(base + o_pr);
  np.pair_items = reinterpret_cast<uint4*>(base + o_pi);
  np.extra_ptr = reinterpret_cast<int32_t*>(base + o_xp);
  np.extra = reinterpret_cast<uint4*>(base + o_x);
  np.diag_items = reinterpret_cast<uint2*>(base + o_di);
  np.diag = reinterpret_cast<uint32_t*>(base + o_dg);
  plan->np = np;
  return FNE_OK;
}

}  // namespace

extern "C" int fne_plan_build_node_patches(fne_plan* plan, const int32_t* edof, const int32_t* indptr,
                                           const int32_t* indices) {
  if (!plan || !edof || !indptr || !indices) {
    fne_set_error("fne_plan_build_node_patches: null pointer");
    return FNE_EINVAL;
  }
  const fne_plan_desc& d = plan->d;
  if (d.kind != FNE_KIND_NEOHOOKEAN || !(d.flags & FNE_FLAG_ROW_GATHER) || plan->np.storage)
    return node_patch_unsupported("needs a tetrahedral row-gather plan without node patches");
  if (d.n_elem <= 0 || d.n_free <= 0) return node_patch_unsupported("empty mesh");
  NodePatchHost h;
  try {
    const int rc = build_node_patches(d, edof, indptr, indices, h);
    if (rc != FNE_OK) return rc;
    return upload_node_patches(plan, h);
  } catch (const std::bad_alloc&) {
    fne_set_error("fne_plan_build_node_patches: out of host memory");
    return FNE_ENOMEM;
  }
}

// ---------------------------------------------------------------------------------------------
// Row units of the Mohr-Coulomb assembly (FneRowUnits), from the plan's row incidences.
// ---------------------------------------------------------------------------------------------
constexpr size_t kUnitWindow = 256;

extern "C" int fne_plan_build_row_units(fne_plan* plan, const int32_t* inc_ptr, const uint32_t* inc,
                                        const unsigned char* pos, const int32_t* indptr,
                                        const int32_t* indices) {
  if (!plan || !inc_ptr || !inc || !pos || !indptr || !indices) {
    fne_set_error("fne_plan_build_row_units: null pointer");
    return FNE_EINVAL;
  }
  const fne_plan_desc& d = plan->d;
  auto unsupported = [](const char* why) {
    fne_set_error(std::string("fne_plan_build_row_units: ") + why);
    return FNE_EUNSUPPORTED;
  };
  if (d.kind != FNE_KIND_MOHR_COULOMB || plan->units.unit || d.n_elem <= 0 || d.n_free <= 0 || !d.inc_ptr || !d.inc || !d.pitem)
    return unsupported("needs a Mohr-Coulomb plan with row incidences and without units");
  const int32_t nf = d.n_free;
  auto items_of = [&](int32_t r) { return inc_ptr[r + 1] - inc_ptr[r]; };
  auto len_of = [&](int32_t r) { return indptr[r + 1] - indptr[r]; };
  for (int32_t r = 0; r < nf; ++r) {
    if (items_of(r) < 0 || items_of(r) >= (1 << 22) || len_of(r) < 0 || len_of(r) > 254)
      return unsupported("row or incidence list too long");
    for (int32_t k = inc_ptr[r]; k < inc_ptr[r + 1]; ++k)
      if (int32_t(inc[k] >> 5) >= d.n_elem || int32_t(inc[k] & 31u) >= d.n_loc)
        return unsupported("incidence item out of range");
  }
  // rows r, r + 1 are the x and y rows of a node with the same columns and elements
  auto paired = [&](int32_t r) {
    if (r + 1 >= nf || items_of(r) != items_of(r + 1) || items_of(r) == 0 || len_of(r) != len_of(r + 1)) return false;
    for (int32_t k = 0; k < items_of(r); ++k) {
      const uint32_t a = inc[inc_ptr[r] + k];
      if ((a & 1u) || inc[inc_ptr[r + 1] + k] != a + 1u) return false;
    }
    const unsigned char *p = pos + size_t(inc_ptr[r]) * 32, *p1 = pos + size_t(inc_ptr[r + 1]) * 32;
    if (!std::equal(p, p1, p1)) return false;
    return std::equal(indices + indptr[r], indices + indptr[r + 1], indices + indptr[r + 1]);
  };
  try {
    std::vector<int4> unit;
    unit.reserve(size_t(nf) / 2 + 1);
    int64_t in_pairs = 0;
    for (int32_t r = 0; r < nf;) {
      const bool two = paired(r);
      in_pairs += two ? 2 : 0;
      unit.push_back(make_int4(indptr[r], inc_ptr[r], r, len_of(r) | (int(two) << 8) | (items_of(r) << 9)));
      r += two ? 2 : 1;
    }
    // with fewer rows in pairs the plan goes on with the row gather (FP32 P4, 32,000 elements: a Hessian of
    // pairs 101 us, of single units 125 to 146, by the row gather 109: even at three quarters)
    if (in_pairs < int64_t(nf) - nf / 4) return FNE_OK;
    // units with the same number of elements side by side: the lane groups of a wavefront then take
    // the same branches; in windows, so that neighbouring rows keep sharing element matrices
    for (size_t i = 0; i < unit.size(); i += kUnitWindow)
      std::stable_sort(unit.begin() + i, unit.begin() + std::min(unit.size(), i + kUnitWindow),
                       [](const int4& a, const int4& b) { return (a.w >> 9) < (b.w >> 9); });
    const size_t width = d.n_loc == 30 ? 32 : 16;
    size_t items = 0;
    for (const int4& w : unit) items += size_t(w.w >> 9);
    std::vector<uint32_t> uinc(items);
    std::vector<unsigned char> upos(items * width);
    items = 0;
    for (int4& w : unit) {
      const int from = w.y, n = w.w >> 9;
      w.y = int(items);
      for (int k = 0; k < n; ++k, ++items) {
        uinc[items] = inc[from + k];
        std::copy_n(pos + size_t(from + k) * 32, width, &upos[items * width]);
      }
    }
    HostParts parts;
    const size_t o_u = parts.add(unit), o_i = parts.add(uinc), o_p = parts.add(upos);
    char* base = nullptr;
    const int up = parts.upload(&base, "fne_plan_build_row_units");
    if (up != FNE_OK) return up;
    plan->units.storage = base;
    plan->units.unit = reinterpret_cast<int4*>(base + o_u);
    plan->units.inc = reinterpret_cast<uint32_t*>(base + o_i);
    plan->units.pos = reinterpret_cast<unsigned char*>(base + o_p);
    plan->units.n_unit = int(unit.size());
  } catch (const std::bad_alloc&) {
    fne_set_error("fne_plan_build_row_units: out of host memory");
    return FNE_ENOMEM;
  }
  return FNE_OK;
}
