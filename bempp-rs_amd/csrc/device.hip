// device.hip -- device-side runtime of the assembly engine: per-grid geometry
// caches in HBM, rule tables, kernel launches, and the host entry points
// (dense into device or host memory, singular COO).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <map>
#include <memory>
#include <mutex>
#include <tuple>

#include "core.hpp"
#include "kernels.hpp"
#include "kernels_mixed.hpp"

namespace bempp_amd {

#define HIP_CHECK(expr)                                                                           \
  do {                                                                                            \
    hipError_t _e = (expr);                                                                       \
    if (_e != hipSuccess) throw Error(std::string(#expr) + " failed: " + hipGetErrorString(_e)); \
  } while (0)

// ---------------------------------------------------------------------------
// Device caches
// ---------------------------------------------------------------------------
// FP64 data of a grid's cells for one regular rule: one upload, pts its start.
struct RuleData {
  double* pts = nullptr;        // [nc][Q][4]
  const double* vtx = nullptr;  // [nc][3][4] vertex offsets, class weights
  const double* gq = nullptr;   // [nc][groups][3] |o_q|^2 of the grouped rule points (rules taken in groups)
};

struct DeviceGridCache {
  int device = -1;
  double* geo = nullptr;          // [nc][kGeoStride]
  int* vid = nullptr;             // [nc][4]
  std::map<int, RuleData> rules;  // by regular point count
  int4* pairs = nullptr;          // adjacent pairs
  int npairs = -1;
  double max_radius = 0.0;        // largest centroid-to-vertex distance of any cell
  double min_radius = 0.0;        // smallest of the cells' radii
  double max_edge = 0.0;          // longest edge of any cell
  std::map<int, float*> pts32;    // regular point count -> [nc][Q][4] FP32 offsets from the centroid, w*jdet
  std::map<int, float*> vtx32;    // regular point count -> [nc][3][4] FP32 vertex offsets, class weights
  int2* near = nullptr;           // non-adjacent pairs the mixed-precision far test rejects,
  int nnear = -1;                 // grouped by (test block, trial block) of 64 cells
  int4* near_segs = nullptr;      // per block pair with near pairs: test block, trial block, first, count
  int nsegs = 0;
  unsigned char* far_tiles = nullptr;  // [nblocks][nblocks]: every cell pair of the tile is far
  std::vector<unsigned char> far_tiles_host;
  int far_tiles_ld = 0;
};

struct DeviceSpaceCache {
  int device = -1;
  int* dofs = nullptr;  // [nc][nb] int32
  // 64-cell blocks (tiled kernel with a P1 side), built on first use
  int* blk_off = nullptr;   // [nblocks + 1]
  int* blk_dofs = nullptr;  // unique DOFs per block, ascending
  int* ldof = nullptr;      // [nc][nb] position in the block's list
  int max_nd = -1;          // largest block DOF count
  // DOF blocks of the potential kernel (PotentialInputs), built on first use
  int* pot_off = nullptr;    // one allocation; the others point into it
  int* pot_cells = nullptr;
  int* pot_ldof = nullptr;
  int pot_nblocks = 0;
  int64_t pot_entries = -1;  // cells listed, with repetitions
};

void drop_device_geometry(DeviceGridCache* c) {
  int cur = 0;
  if (hipGetDevice(&cur) == hipSuccess && hipSetDevice(c->device) == hipSuccess) {
    (void)hipFree(c->geo);
    for (auto& kv : c->rules) (void)hipFree(kv.second.pts);
    for (auto& kv : c->pts32) (void)hipFree(kv.second);
    for (auto& kv : c->vtx32) (void)hipFree(kv.second);
    (void)hipFree(c->near);
    (void)hipFree(c->near_segs);
    (void)hipFree(c->far_tiles);
    (void)hipSetDevice(cur);
  }
  c->geo = nullptr;
  c->rules.clear();
  c->pts32.clear();
  c->vtx32.clear();
  c->near = nullptr;
  c->near_segs = nullptr;
  c->nnear = -1;
  c->far_tiles = nullptr;
}

void free_device_grid_cache(DeviceGridCache* c) {
  if (!c) return;
  drop_device_geometry(c);
  int cur = 0;
  if (hipGetDevice(&cur) == hipSuccess && hipSetDevice(c->device) == hipSuccess) {
    (void)hipFree(c->vid);
    (void)hipFree(c->pairs);
    (void)hipSetDevice(cur);
  }
  delete c;
}

void free_device_space_cache(DeviceSpaceCache* c) {
  if (!c) return;
  int cur = 0;
  if (hipGetDevice(&cur) == hipSuccess && hipSetDevice(c->device) == hipSuccess) {
    (void)hipFree(c->dofs);
    if (c->blk_off) (void)hipFree(c->blk_off);
    if (c->blk_dofs) (void)hipFree(c->blk_dofs);
    if (c->ldof) (void)hipFree(c->ldof);
    if (c->pot_off) (void)hipFree(c->pot_off);
    (void)hipSetDevice(cur);
  }
  delete c;
}

int device_count() {
  int n = 0;
  if (hipGetDeviceCount(&n) != hipSuccess) return 0;
  return n;
}

namespace {

int current_device() {
  int n = device_count();
  if (n <= 0) throw Error("no HIP device available: assembly requires an MI355X GPU (there is no CPU fallback)");
  int d = 0;
  HIP_CHECK(hipGetDevice(&d));
  return d;
}

// Set while an entry point that must not allocate device memory gathers its inputs:
// a cache that is not built yet then raises instead of being uploaded.
thread_local int t_no_device_alloc = 0;

// Uninitialised device array of n elements (at least one).
template <typename T>
T* device_array(size_t n) {
  if (t_no_device_alloc)
    throw Error("this entry point allocates no device memory, but the device data of this grid, space or rule "
                "is not built yet: make one ordinary call with the same assembler and spaces first");
  T* d = nullptr;
  HIP_CHECK(hipMalloc((void**)&d, std::max<size_t>(n, 1) * sizeof(T)));
  return d;
}

template <typename T>
T* upload(const std::vector<T>& h) {
  if (t_no_device_alloc)
    throw Error("this entry point allocates no device memory, but the device data of this grid, space or rule "
                "is not built yet: make one ordinary call with the same assembler and spaces first");
  T* d = nullptr;
  HIP_CHECK(hipMalloc((void**)&d, std::max<size_t>(h.size(), 1) * sizeof(T)));
  if (!h.empty()) HIP_CHECK(hipMemcpy(d, h.data(), h.size() * sizeof(T), hipMemcpyHostToDevice));
  return d;
}

// Per-cell geometry record: vertices, unit normal, jdet = |J0 x J1|, and
// curlJ_b = J1 d0(phi_b) - J0 d1(phi_b) for the P1 basis (constant on a flat cell).
void cell_record(const Grid& g, int64_t c, double* r) {
  const double* v[3];
  for (int m = 0; m < 3; ++m) v[m] = &g.points[3 * g.cells[3 * c + m]];
  double J0[3], J1[3];
  for (int d = 0; d < 3; ++d) {
    r[d] = v[0][d];
    r[3 + d] = v[1][d];
    r[6 + d] = v[2][d];
    J0[d] = v[1][d] - v[0][d];
    J1[d] = v[2][d] - v[0][d];
  }
  const double n[3] = {J0[1] * J1[2] - J0[2] * J1[1], J0[2] * J1[0] - J0[0] * J1[2], J0[0] * J1[1] - J0[1] * J1[0]};
  const double jdet = std::sqrt(n[0] * n[0] + n[1] * n[1] + n[2] * n[2]);
  if (!(jdet > 0.0)) throw Error("cell " + std::to_string(c) + " is degenerate (zero area)");
  for (int d = 0; d < 3; ++d) {
    r[9 + d] = n[d] / jdet;
    r[13 + d] = J0[d] - J1[d];  // basis 0: grad (-1,-1)
    r[16 + d] = J1[d];          // basis 1: grad (1,0)
    r[19 + d] = -J0[d];         // basis 2: grad (0,1)
  }
  r[12] = jdet;
  r[22] = r[23] = 0.0;
  double rad2 = 0.0;
  for (int d = 0; d < 3; ++d) r[dev::kGeoCentroid + d] = (v[0][d] + v[1][d] + v[2][d]) / 3.0;
  for (int m = 0; m < 3; ++m) {
    double s = 0.0;
    for (int d = 0; d < 3; ++d) s += (v[m][d] - r[dev::kGeoCentroid + d]) * (v[m][d] - r[dev::kGeoCentroid + d]);
    rad2 = std::max(rad2, s);
  }
  // slightly enlarged so that rounding never lets a quadrature point escape the bound
  r[dev::kGeoRadius] = std::sqrt(rad2) * (1.0 + 1e-12);
  for (int m = dev::kGeoRadius + 1; m < dev::kGeoStride; ++m) r[m] = 0.0;
}

DeviceGridCache* grid_cache(Grid& g, int device) {
  std::lock_guard<std::mutex> lk(g.cache_mutex);
  auto it = g.device_cache.find(device);
  DeviceGridCache* c = it != g.device_cache.end() ? it->second : nullptr;
  if (c && c->geo) return c;
  const int64_t nc = g.nc();
  std::vector<double> geo(nc * dev::kGeoStride);
  double max_radius = 0.0, min_radius = INFINITY, max_edge = 0.0;
  for (int64_t i = 0; i < nc; ++i) {
    double* r = &geo[i * dev::kGeoStride];
    cell_record(g, i, r);
    max_radius = std::max(max_radius, r[dev::kGeoRadius]);
    min_radius = std::min(min_radius, r[dev::kGeoRadius]);
    for (int m = 0; m < 3; ++m) {  // the J-scaled curls are the edge vectors
      const double* e = r + 13 + 3 * m;
      max_edge = std::max(max_edge, std::sqrt(e[0] * e[0] + e[1] * e[1] + e[2] * e[2]));
    }
  }
  if (!c) {
    std::vector<int> vid(nc * 4);
    for (int64_t i = 0; i < nc; ++i) {
      for (int m = 0; m < 3; ++m) vid[4 * i + m] = (int)g.cells[3 * i + m];
      vid[4 * i + 3] = -1;
    }
    auto fresh = std::make_unique<DeviceGridCache>();
    fresh->device = device;
    fresh->vid = upload(vid);
    c = g.device_cache[device] = fresh.release();
  }
  c->geo = upload(geo);
  c->max_radius = max_radius;
  c->min_radius = min_radius;
  c->max_edge = max_edge;
  return c;
}

// (capacity for `more` further values)
std::vector<double> rule_points(const Grid& g, int Q, const std::vector<double>& xi, const std::vector<double>& w,
                                size_t more) {
  const int64_t nc = g.nc();
  std::vector<double> pts;
  pts.reserve(nc * Q * 4 + more);
  pts.resize(nc * Q * 4);
  for (int64_t i = 0; i < nc; ++i) {
    const double* v0 = &g.points[3 * g.cells[3 * i]];
    const double* v1 = &g.points[3 * g.cells[3 * i + 1]];
    const double* v2 = &g.points[3 * g.cells[3 * i + 2]];
    double J0[3], J1[3];
    for (int d = 0; d < 3; ++d) {
      J0[d] = v1[d] - v0[d];
      J1[d] = v2[d] - v0[d];
    }
    const double cr[3] = {J0[1] * J1[2] - J0[2] * J1[1], J0[2] * J1[0] - J0[0] * J1[2],
                          J0[0] * J1[1] - J0[1] * J1[0]};
    const double jdet = std::sqrt(cr[0] * cr[0] + cr[1] * cr[1] + cr[2] * cr[2]);
    for (int p = 0; p < Q; ++p) {
      double* o = &pts[(i * Q + p) * 4];
      for (int d = 0; d < 3; ++d) o[d] = v0[d] + J0[d] * xi[2 * p] + J1[d] * xi[2 * p + 1];
      o[3] = w[p] * jdet;
    }
  }
  return pts;
}

// FP32 copies of the regular points as offsets from the cell centroid (mixed precision).
const float* grid_points32_for_rule(Grid& g, DeviceGridCache* c, int Q, const std::vector<double>& xi,
                                    const std::vector<double>& w) {
  std::lock_guard<std::mutex> lk(g.cache_mutex);
  auto it = c->pts32.find(Q);
  if (it != c->pts32.end()) return it->second;
  const int64_t nc = g.nc();
  std::vector<float> p32(nc * Q * 4);
  for (int64_t i = 0; i < nc; ++i) {
    const double* v0 = &g.points[3 * g.cells[3 * i]];
    const double* v1 = &g.points[3 * g.cells[3 * i + 1]];
    const double* v2 = &g.points[3 * g.cells[3 * i + 2]];
    double J0[3], J1[3], cen[3];
    for (int d = 0; d < 3; ++d) {
      J0[d] = v1[d] - v0[d];
      J1[d] = v2[d] - v0[d];
      cen[d] = (v0[d] + v1[d] + v2[d]) / 3.0;
    }
    const double cr[3] = {J0[1] * J1[2] - J0[2] * J1[1], J0[2] * J1[0] - J0[0] * J1[2],
                          J0[0] * J1[1] - J0[1] * J1[0]};
    const double jdet = std::sqrt(cr[0] * cr[0] + cr[1] * cr[1] + cr[2] * cr[2]);
    for (int p = 0; p < Q; ++p) {
      float* o = &p32[(i * Q + p) * 4];
      for (int d = 0; d < 3; ++d) o[d] = (float)((v0[d] + J0[d] * xi[2 * p] + J1[d] * xi[2 * p + 1]) - cen[d]);
      o[3] = (float)(w[p] * jdet);
    }
  }
  float* d = upload(p32);
  c->pts32[Q] = d;
  return d;
}

// Per cell, for the P0 tiles (rule points in orbit form c + t (V_k - c)): d_0 = V_0 - c,
// |d_0|^2; d_1 = V_1 - c, |d_1|^2; the class weights w * jdet, |d_2|^2 (12 values of type T).
template <typename T>
std::vector<T> vertex_records(const Grid& g, int Q, const std::vector<double>& w) {
  const int64_t nc = g.nc();
  std::vector<T> out(nc * 12, T(0));
  for (int64_t i = 0; i < nc; ++i) {
    const double* v[3] = {&g.points[3 * g.cells[3 * i]], &g.points[3 * g.cells[3 * i + 1]],
                          &g.points[3 * g.cells[3 * i + 2]]};
    double cen[3], d[3][3], J0[3], J1[3];
    for (int k = 0; k < 3; ++k) {
      cen[k] = (v[0][k] + v[1][k] + v[2][k]) / 3.0;
      J0[k] = v[1][k] - v[0][k];
      J1[k] = v[2][k] - v[0][k];
    }
    for (int m = 0; m < 3; ++m)
      for (int k = 0; k < 3; ++k) d[m][k] = v[m][k] - cen[k];
    const double cr[3] = {J0[1] * J1[2] - J0[2] * J1[1], J0[2] * J1[0] - J0[0] * J1[2],
                          J0[0] * J1[1] - J0[1] * J1[0]};
    const double jdet = std::sqrt(cr[0] * cr[0] + cr[1] * cr[1] + cr[2] * cr[2]);
    T* o = &out[i * 12];
    for (int m = 0; m < 2; ++m)
      for (int k = 0; k < 3; ++k) o[4 * m + k] = (T)d[m][k];
    for (int m = 0; m < 3; ++m)
      o[m == 2 ? 11 : 4 * m + 3] = (T)(d[m][0] * d[m][0] + d[m][1] * d[m][1] + d[m][2] * d[m][2]);
    for (int cl = 0; cl < dev::weight_classes(Q); ++cl) o[8 + cl] = (T)(w[dev::class_point(Q, cl)] * jdet);
  }
  return out;
}

const float* grid_vertex32_for_rule(Grid& g, DeviceGridCache* c, int Q, const std::vector<double>& w) {
  std::lock_guard<std::mutex> lk(g.cache_mutex);
  auto it = c->vtx32.find(Q);
  if (it != c->vtx32.end()) return it->second;
  float* d = upload(vertex_records<float>(g, Q, w));
  c->vtx32[Q] = d;
  return d;
}

// |o_q|^2 of the rule's grouped points (RuleGroups): o_k = p d_k + s d_{k+1}.
std::vector<double> group_radii(const Grid& g, int Q) {
  const RuleGroups rg = rule_groups(Q);
  const int64_t nc = g.nc();
  std::vector<double> out((size_t)nc * rg.groups.size() * 3);
  double* o = out.data();
  for (int64_t i = 0; i < nc; ++i) {
    double d[3][3];
    for (int k = 0; k < 3; ++k) {
      const double v[3] = {g.points[3 * g.cells[3 * i] + k], g.points[3 * g.cells[3 * i + 1] + k],
                           g.points[3 * g.cells[3 * i + 2] + k]};
      const double cen = (v[0] + v[1] + v[2]) / 3.0;
      for (int m = 0; m < 3; ++m) d[m][k] = v[m] - cen;
    }
    for (const RuleGroup& r : rg.groups)
      for (int m = 0; m < 3; ++m) {
        double s = 0.0;
        for (int k = 0; k < 3; ++k) {
          const double x = r.p * d[m][k] + r.s * d[(m + 1) % 3][k];
          s += x * x;
        }
        *o++ = s;
      }
  }
  return out;
}

// Template point count of the kernels for a rule of Q points: Q itself for the rules
// compiled with their point count (held in registers), 0 (point count at run time) otherwise.
int kernel_q(int Q) { return (Q == 1 || Q == 3 || Q == 6 || Q == 7) ? Q : 0; }

RuleData grid_rule_data(Grid& g, DeviceGridCache* c, int Q, const std::vector<double>& xi,
                        const std::vector<double>& w) {
  std::lock_guard<std::mutex> lk(g.cache_mutex);
  auto it = c->rules.find(Q);
  if (it != c->rules.end()) return it->second;
  const std::vector<double> records = vertex_records<double>(g, Q, w);
  const std::vector<double> radii = kernel_q(Q) == 0 ? group_radii(g, Q) : std::vector<double>();
  std::vector<double> all = rule_points(g, Q, xi, w, records.size() + radii.size());
  const size_t vtx = all.size(), gq = vtx + records.size();
  all.insert(all.end(), records.begin(), records.end());
  all.insert(all.end(), radii.begin(), radii.end());
  RuleData r;
  r.pts = upload(all);
  r.vtx = r.pts + vtx;
  if (kernel_q(Q) == 0) r.gq = r.pts + gq;
  return c->rules[Q] = r;
}

// The rule's groups as a device table (group_sum.hpp) for test and trial spaces of nbt and nbs
// functions per cell.
const double* group_table(int device, int Q, int nbt, int nbs, const RuleGroups& rg) {
  static std::mutex mu;
  static std::map<std::tuple<int, int, int, int>, double*> tables;
  std::lock_guard<std::mutex> lk(mu);
  const auto key = std::make_tuple(device, Q, nbt, nbs);
  auto it = tables.find(key);
  if (it != tables.end()) return it->second;
  std::vector<double> t;
  for (const RuleGroup& r : rg.groups) {
    double row[dev::kGroupStride] = {r.p, r.s, -2.0 * r.p, -2.0 * r.s, r.w, r.p * r.p};
    for (int side = 0; side < 2; ++side) {
      double* o = row + (side == 0 ? dev::kGrpTest : dev::kGrpTrial);
      const bool p1 = (side == 0 ? nbt : nbs) == 3;
      o[0] = p1 ? r.w * r.p : 0.0;
      o[1] = p1 ? r.w * r.s : 0.0;
      o[2] = p1 ? r.w * r.g : r.w;
    }
    t.insert(t.end(), row, row + dev::kGroupStride);
  }
  double* d = upload(t);
  tables[key] = d;
  return d;
}

// True when every point of the rule is c + t (V_k - c) with the tabulated t, k (orbit_t,
// orbit_vertex) and the weights follow the weight classes.
bool rule_in_orbit_form(int Q, const std::vector<double>& xi, const std::vector<double>& w) {
  for (int p = 0; p < Q; ++p) {
    if (w[p] != w[dev::class_point(Q, dev::weight_class(Q, p))]) return false;
    const double lam[3] = {1.0 - xi[2 * p] - xi[2 * p + 1], xi[2 * p], xi[2 * p + 1]};
    const double t = dev::orbit_t(Q, p);
    const int kv = dev::orbit_vertex(Q, p);
    for (int m = 0; m < 3; ++m)
      if (std::fabs(lam[m] - (m == kv ? (1.0 + 2.0 * t) / 3.0 : (1.0 - t) / 3.0)) > 1e-15) return false;
  }
  return true;
}

// Tiles (64-cell blocks a, b) whose cell pairs are all far for the mixed-precision split:
// with block centre C (mean centroid), rho (largest centroid distance from C) and rmax
// (largest cell radius), every pair has R >= |C_a - C_b| - rho_a - rho_b; the tile is
// flagged when that bound exceeds the far limit kNearFactor (rmax_a + rmax_b) by 0.1 %, far
// beyond the rounding of the per-pair test it replaces (no flagged pair can be near or
// adjacent, adjacent cells being closer than rad_i + rad_j). Flag 2: beyond kVeryFarFactor too.
const unsigned char* grid_far_tiles(Grid& g, DeviceGridCache* c, int* ld) {
  std::lock_guard<std::mutex> lk(g.cache_mutex);
  if (!c->far_tiles) {
    const int64_t nc = g.nc();
    const int nb = (int)((nc + dev::kTile - 1) / dev::kTile);
    std::vector<double> cen(3 * nc), rad(nc), bc(3 * nb, 0.0), rho(nb, 0.0), rmax(nb, 0.0);
    std::vector<double> rec(dev::kGeoStride);
    for (int64_t i = 0; i < nc; ++i) {
      cell_record(g, i, rec.data());
      for (int d = 0; d < 3; ++d) cen[3 * i + d] = rec[dev::kGeoCentroid + d];
      rad[i] = rec[dev::kGeoRadius];
      const int b = (int)(i / dev::kTile);
      for (int d = 0; d < 3; ++d) bc[3 * b + d] += cen[3 * i + d];
      rmax[b] = std::max(rmax[b], rad[i]);
    }
    for (int b = 0; b < nb; ++b) {
      const int64_t n = std::min<int64_t>(dev::kTile, nc - (int64_t)b * dev::kTile);
      for (int d = 0; d < 3; ++d) bc[3 * b + d] /= (double)n;
    }
    for (int64_t i = 0; i < nc; ++i) {
      const int b = (int)(i / dev::kTile);
      double s = 0.0;
      for (int d = 0; d < 3; ++d) s += (cen[3 * i + d] - bc[3 * b + d]) * (cen[3 * i + d] - bc[3 * b + d]);
      rho[b] = std::max(rho[b], std::sqrt(s));
    }
    std::vector<unsigned char> flags((size_t)nb * nb, 0);
    for (int a = 0; a < nb; ++a)
      for (int b = 0; b < nb; ++b) {
        double s = 0.0;
        for (int d = 0; d < 3; ++d) s += (bc[3 * a + d] - bc[3 * b + d]) * (bc[3 * a + d] - bc[3 * b + d]);
        const double lower = std::sqrt(s) - rho[a] - rho[b];
        const double radii = 1.001 * (rmax[a] + rmax[b]);
        flags[(size_t)a * nb + b] = lower >= dev::kVeryFarFactor * radii ? 2 : lower >= dev::kNearFactor * radii ? 1 : 0;
      }
    c->far_tiles = upload(flags);
    c->far_tiles_host = std::move(flags);
    c->far_tiles_ld = nb;
  }
  *ld = c->far_tiles_ld;
  return c->far_tiles;
}

// The mixed-precision near-pair list of a grid (non-adjacent pairs the far test rejects),
// built on the device from the candidate tiles (those not flagged all-far; see
// near_count_kernel / near_fill_kernel), grouped by tile: segs[s] = {test block, trial
// block, first pair, pair count} for each tile with near pairs.
const int2* grid_near_pairs(Grid& g, DeviceGridCache* c, int* n, const int4** segs, int* nsegs) {
  int ld = 0;
  (void)grid_far_tiles(g, c, &ld);
  std::lock_guard<std::mutex> lk(g.cache_mutex);
  if (c->nnear < 0) {
    const int nb = c->far_tiles_ld;
    std::vector<int2> cand;
    for (int a = 0; a < nb; ++a)
      for (int b = 0; b < nb; ++b)
        if (!c->far_tiles_host[(size_t)a * nb + b]) cand.push_back(make_int2(a, b));
    std::vector<int> counts(cand.size()), offsets(cand.size());
    std::vector<int4> sg;
    long long total = 0;
    int2* tiles = nullptr;
    int* dcounts = nullptr;
    int* doffsets = nullptr;
    int2* out = nullptr;
    auto cleanup = [&]() {
      (void)hipFree(tiles);
      (void)hipFree(dcounts);
      (void)hipFree(doffsets);
    };
    try {
      if (!cand.empty()) {
        tiles = upload(cand);
        dcounts = upload(counts);
        dev::NearBuildArgs B{};
        B.geo = c->geo;
        B.vid = c->vid;
        B.n = (int)g.nc();
        B.tiles = tiles;
        B.counts = dcounts;
        dev::near_count_kernel<><<<(unsigned)cand.size(), 256, 0, nullptr>>>(B);
        HIP_CHECK(hipGetLastError());
        HIP_CHECK(hipMemcpy(counts.data(), dcounts, counts.size() * sizeof(int), hipMemcpyDeviceToHost));
        for (size_t t = 0; t < cand.size(); ++t) {
          offsets[t] = (int)total;
          if (counts[t] > 0) sg.push_back(make_int4(cand[t].x, cand[t].y, (int)total, counts[t]));
          total += counts[t];
          if (total > INT32_MAX) throw Error("too many near pairs for the mixed-precision split");
        }
        if (total > 0) {
          doffsets = upload(offsets);
          out = device_array<int2>((size_t)total);
          B.offsets = doffsets;
          B.out = out;
          dev::near_fill_kernel<><<<(unsigned)cand.size(), 256, 0, nullptr>>>(B);
          HIP_CHECK(hipGetLastError());
          HIP_CHECK(hipStreamSynchronize(nullptr));
        }
      }
      c->near_segs = upload(sg);
    } catch (...) {
      cleanup();
      (void)hipFree(out);
      throw;
    }
    cleanup();
    c->near = out ? out : device_array<int2>(1);
    c->nnear = (int)total;
    c->nsegs = (int)sg.size();
  }
  *n = c->nnear;
  if (segs) *segs = c->near_segs;
  if (nsegs) *nsegs = c->nsegs;
  return c->near;
}

const int4* grid_pairs(Grid& g, DeviceGridCache* c, int* npairs) {
  std::lock_guard<std::mutex> lk(g.cache_mutex);
  if (c->npairs < 0) {
    std::vector<AdjacentPair> pairs;
    adjacent_pairs(g, pairs);
    // group by adjacency type: consecutive wavefronts then read the same rule table
    std::stable_sort(pairs.begin(), pairs.end(),
                     [](const AdjacentPair& x, const AdjacentPair& y) { return x.nshared < y.nshared; });
    std::vector<int4> p(pairs.size());
    for (size_t i = 0; i < p.size(); ++i) {
      const AdjacentPair& a = pairs[i];
      p[i] = make_int4(a.test, a.trial, a.nshared, a.perm);
    }
    c->pairs = upload(p);
    c->npairs = (int)p.size();
  }
  *npairs = c->npairs;
  return c->pairs;
}

const int* space_dofs(FunctionSpace& s, int device) {
  std::lock_guard<std::mutex> lk(s.cache_mutex);
  auto it = s.device_cache.find(device);
  if (it != s.device_cache.end()) return it->second->dofs;
  if (s.size > INT32_MAX) throw Error("function space too large for 32-bit DOF indices");
  std::vector<int> d(s.dofs.begin(), s.dofs.end());
  auto* c = new DeviceSpaceCache();
  c->device = device;
  c->dofs = upload(d);
  s.device_cache[device] = c;
  return c->dofs;
}

// Block DOF lists of a space for the tiled kernel with a P1 side: cells [64 t, 64 t + 64)
// form block t (consecutive cells of a refined mesh are a compact patch).
const DeviceSpaceCache* space_blocks(FunctionSpace& s, int device) {
  space_dofs(s, device);
  std::lock_guard<std::mutex> lk(s.cache_mutex);
  DeviceSpaceCache* c = s.device_cache.at(device);
  if (c->max_nd >= 0) return c;
  const int64_t nc = s.grid->nc();
  const int nb = s.nb;
  const int64_t nblk = (nc + dev::kTile - 1) / dev::kTile;
  std::vector<int> off(nblk + 1, 0), bd, ldof((size_t)nc * nb);
  int max_nd = 0;
  std::vector<int64_t> tmp;
  for (int64_t t = 0; t < nblk; ++t) {
    const int64_t c0 = t * dev::kTile, c1 = std::min(nc, c0 + dev::kTile);
    tmp.assign(s.dofs.begin() + c0 * nb, s.dofs.begin() + c1 * nb);
    std::sort(tmp.begin(), tmp.end());
    tmp.erase(std::unique(tmp.begin(), tmp.end()), tmp.end());
    for (int64_t cc = c0; cc < c1; ++cc)
      for (int a = 0; a < nb; ++a)
        ldof[cc * nb + a] = (int)(std::lower_bound(tmp.begin(), tmp.end(), s.dofs[cc * nb + a]) - tmp.begin());
    for (int64_t d : tmp) bd.push_back((int)d);
    off[t + 1] = (int)bd.size();
    max_nd = std::max(max_nd, (int)tmp.size());
  }
  c->blk_off = upload(off);
  c->blk_dofs = upload(bd);
  c->ldof = upload(ldof);
  c->max_nd = max_nd;
  return c;
}

// Canonical Sauter-Schwab rules for one Gauss order n, per device (kept for the
// life of the process: a few hundred KB).
struct RuleTable {
  double* aos = nullptr;  // one record of 6 per point (a0 a1 b0 b1 w pad)
  int total = 0;
  int off[4] = {0, 0, 0, 0};
  int n[4] = {0, 0, 0, 0};
};

const RuleTable& rule_table(int device, int n) {
  static std::mutex mu;
  static std::map<std::pair<int, int>, RuleTable> tables;
  std::lock_guard<std::mutex> lk(mu);
  auto it = tables.find({device, n});
  if (it != tables.end()) return it->second;
  RuleTable t;
  std::vector<double> parts[4];
  for (int m = 1; m <= 3; ++m) {
    canonical_pair_rule(m, n, parts[m]);
    t.off[m] = t.total;
    t.n[m] = (int)(parts[m].size() / 5);
    t.total += t.n[m];
  }
  std::vector<double> aos(6 * (size_t)t.total, 0.0);
  for (int m = 1; m <= 3; ++m)
    for (int i = 0; i < t.n[m]; ++i)
      for (int f = 0; f < 5; ++f) aos[6 * (size_t)(t.off[m] + i) + f] = parts[m][5 * i + f];
  t.aos = upload(aos);
  return tables.emplace(std::make_pair(device, n), t).first->second;
}

// Regular rule as a device table [Q][4] = barycentric coordinates (the P1 basis values)
// and weight of each point, per device and point count; read by the kernels that take
// the point count at run time.
const double* regular_rule_table(int device, int Q, const std::vector<double>& xi, const std::vector<double>& w) {
  static std::mutex mu;
  static std::map<std::pair<int, int>, double*> tables;
  std::lock_guard<std::mutex> lk(mu);
  auto it = tables.find({device, Q});
  if (it != tables.end()) return it->second;
  std::vector<double> t(4 * (size_t)Q);
  for (int p = 0; p < Q; ++p) {
    t[4 * p] = 1.0 - xi[2 * p] - xi[2 * p + 1];
    t[4 * p + 1] = xi[2 * p];
    t[4 * p + 2] = xi[2 * p + 1];
    t[4 * p + 3] = w[p];
  }
  double* d = upload(t);
  tables[{device, Q}] = d;
  return d;
}

// The same for the potential kernel: [Q][4] = weight x P1 basis values, weight.
const double* weighted_rule_table(int device, int Q, const std::vector<double>& xi, const std::vector<double>& w) {
  static std::mutex mu;
  static std::map<std::pair<int, int>, double*> tables;
  std::lock_guard<std::mutex> lk(mu);
  auto it = tables.find({device, Q});
  if (it != tables.end()) return it->second;
  std::vector<double> t(4 * (size_t)Q);
  for (int p = 0; p < Q; ++p) {
    t[4 * p] = w[p] * (1.0 - xi[2 * p] - xi[2 * p + 1]);
    t[4 * p + 1] = w[p] * xi[2 * p];
    t[4 * p + 2] = w[p] * xi[2 * p + 1];
    t[4 * p + 3] = w[p];
  }
  double* d = upload(t);
  tables[{device, Q}] = d;
  return d;
}

hipStream_t assembler_stream(const Assembler& a, int device) {
  auto& m = const_cast<Assembler&>(a);
  static std::mutex mu;
  std::lock_guard<std::mutex> lk(mu);
  if (!m.stream || m.device != device) {
    if (m.stream) {
      int cur = 0;
      (void)hipGetDevice(&cur);
      (void)hipSetDevice(m.device);
      (void)hipStreamDestroy((hipStream_t)m.stream);
      (void)hipSetDevice(cur);
    }
    hipStream_t s;
    HIP_CHECK(hipStreamCreateWithFlags(&s, hipStreamNonBlocking));
    m.stream = s;
    m.device = device;
  }
  return (hipStream_t)m.stream;
}

int out_type(DType d) {
  switch (d) {
    case kF64: return dev::kOutF64;
    case kC64: return dev::kOutC128;
    case kF32: return dev::kOutF32;
    default: return dev::kOutC64;
  }
}

int regular_points(const Options& o) {
  auto it = o.quadrature_degrees.find(kTriangle);
  if (it == o.quadrature_degrees.end()) throw Error("no regular quadrature degree set for triangles");
  return (int)it->second;
}

int singular_points(const Options& o) {
  auto it = o.singular_quadrature_degrees.find({kTriangle, kTriangle});
  if (it == o.singular_quadrature_degrees.end()) throw Error("no singular quadrature degree set for triangle pairs");
  return (int)it->second;
}

// LDS a workgroup of the LDS-accumulating tile kernels may use: all of the device's (160 KB on
// gfx950). A compact 64-cell P1 patch has ~45 DOFs (16 KB Laplace, 32 KB Helmholtz); 64
// consecutive cells of a mesh numbered in rows have 66 (35 KB, 70 KB), other orders more. Past
// 80 KB one workgroup remains per CU, still far ahead of the general kernel's nine global
// atomics per cell pair and part: Laplace DL P1 on a torus of 19110 cells
// in rows takes 12.0 ms so, 63.9 ms there.
size_t max_tile_lds(int device) {
  int bytes = 0;
  HIP_CHECK(hipDeviceGetAttribute(&bytes, hipDeviceAttributeMaxSharedMemoryPerBlock, device));
  return (size_t)bytes;
}

// Largest block of complex sums that the mixed-precision tiles with a P1 side take.
constexpr size_t kMixedTileLds = 62 * 1024;

// Tile coordinates (tile row = test block, tile column = trial block) for the
// P0 x P0 kernel: all tiles, or the upper triangle a <= b when symmetric.
// Cached per device and shape for the life of the process.
const int2* tile_list(int device, int nta, int ntb, bool symmetric, int* count) {
  static std::mutex mu;
  static std::map<std::tuple<int, int, int, bool>, std::pair<int2*, int>> cache;
  std::lock_guard<std::mutex> lk(mu);
  auto key = std::make_tuple(device, nta, ntb, symmetric);
  auto it = cache.find(key);
  if (it == cache.end()) {
    std::vector<int2> t;
    for (int b = 0; b < ntb; ++b)
      for (int a = 0; a < (symmetric ? std::min(b + 1, nta) : nta); ++a) t.push_back(make_int2(a, b));
    it = cache.emplace(key, std::make_pair(upload(t), (int)t.size())).first;
  }
  *count = it->second.second;
  return it->second.first;
}

// Workgroups a 64 x 64 tile is split over (a power of two up to 16, one trial cell per wavefront): as
// many as give at most `most` workgroups, so that few tiles still fill the 256 CUs. Past that more
// parts only repeat the prologue (and, P1, the clearing and flushing of the tile's sums).
// Measured with 1 / 2 / 4 / 8 / 16 parts, us:
//   P0 Helmholtz SL, 15 tiles: 65 / 43 / 32 / 26 / 24; 210: 84 / 76 / 73 / 69 / 74; 595: 181 / 159 / 159 /
//   164 / 169; 3240: 516 / 515 / 524 / 545 / 604. P0 Laplace SL, 15: 37 / 26 / 20 / 18 / 16; 210: 55 / 48 / 46 / 46 / 50
//   P1 Helmholtz DL, 25: 121 / 83 / 64 / 55 / 54; 400: 209 / 200 / 188 / 186 / 191; 1156: 457 / 456 / 456 / 481 / 558
//   P1 Laplace HS, 15: 67 / 52 / 45 / 41 / 40; 210: 101 / 92 / 91 / 95 / 106; 1653: 298 / 306 / 344 / 440 / 632
constexpr int kSplitP0 = 2400, kSplitP1 = 1600;
int tile_split(int ntiles, int most) {
  int split = 1;
  while (split < 16 && (long long)ntiles * split * 2 <= most) split *= 2;
  return split;
}

// ---- kernel dispatch: tiled P0 x P0 or general, by operator, kernel and phase mode ----
// CENTRED: phase tier (0: full reduction, 1: |k (r - R)| <= 0.5, 2: <= 0.25, 3: <= 1.5; tier 2
// for the tile kernels, the general kernel runs tier 1 there).
// mode: 0 general kernel (atomics per cell pair), 1 P0 x P0 tiles, 2 tiles with LDS
// accumulation (a P1 side; lds = dynamic LDS bytes).
template <int OP, bool HELM, int CENTRED>
void launch_q(int mode, int Q, dim3 grid, hipStream_t s, const dev::RegularArgs& A, const int2* tiles, int sym,
              int split, size_t lds) {
  constexpr int GC = CENTRED == 2 ? 1 : CENTRED;
#define BEMPP_LAUNCH(QQ)                                                                                        \
  if (mode == 0) dev::regular_kernel<QQ, OP, HELM, GC><<<grid, 256, 0, s>>>(A);                                 \
  else                                                                                                          \
    in_launches(grid.x, [&](long long first, unsigned n) {                                                      \
      if (mode == 1)                                                                                            \
        dev::regular_p0_tiled<QQ, OP, HELM, CENTRED><<<n * split, 256, 0, s>>>(A, tiles + first, sym, split);   \
      else                                                                                                      \
        dev::regular_tiled_lds<QQ, OP, HELM, CENTRED><<<n * split, 256, lds, s>>>(A, tiles + first, sym, split); \
    });
  switch (kernel_q(Q)) {
    case 1: BEMPP_LAUNCH(1); break;
    case 3: BEMPP_LAUNCH(3); break;
    case 6: BEMPP_LAUNCH(6); break;
    case 7: BEMPP_LAUNCH(7); break;
    default: BEMPP_LAUNCH(0); break;  // point count at run time
  }
#undef BEMPP_LAUNCH
}

template <bool HELM, int CENTRED>
void launch_op(int op, int mode, int Q, dim3 grid, hipStream_t s, const dev::RegularArgs& A, const int2* tiles,
               int sym, int split, size_t lds) {
  switch (op) {
    case kSL: launch_q<kSL, HELM, CENTRED>(mode, Q, grid, s, A, tiles, sym, split, lds); break;
    case kDL: launch_q<kDL, HELM, CENTRED>(mode, Q, grid, s, A, tiles, sym, split, lds); break;
    case kADL: launch_q<kADL, HELM, CENTRED>(mode, Q, grid, s, A, tiles, sym, split, lds); break;
    case kHS: launch_q<kHS, HELM, CENTRED>(mode, Q, grid, s, A, tiles, sym, split, lds); break;
    default: throw Error("operator not supported by the dense assembler");
  }
}

// Regular pairs: mode 1 the P0 x P0 tile kernel, mode 2 the LDS-accumulating tile kernel
// (grid = tile count), mode 0 the general kernel (grid = test blocks x trial chunks).
void launch_regular(int op, bool helm, int tier, int mode, int Q, dim3 grid, hipStream_t s,
                    const dev::RegularArgs& A, const int2* tiles = nullptr, int sym = 0, int split = 1, size_t lds = 0) {
  if (!helm) launch_op<false, 0>(op, mode, Q, grid, s, A, tiles, sym, split, lds);
  else if (tier == 2 && (mode == 1 || mode == 2)) launch_op<true, 2>(op, mode, Q, grid, s, A, tiles, sym, split, lds);
  else if (tier == 3) launch_op<true, 3>(op, mode, Q, grid, s, A, tiles, sym, split, lds);
  else if (tier >= 1) launch_op<true, 1>(op, mode, Q, grid, s, A, tiles, sym, split, lds);
  else launch_op<true, 0>(op, mode, Q, grid, s, A, tiles, sym, split, lds);
  HIP_CHECK(hipGetLastError());
}

// Mixed precision (P0 x P0, one grid): FP32 far-pair tiles, then the FP64 near-pair list.
// TIER: phase tier of the cell pairs (0: range-reduced FP32 phase and FP64 near pairs
// without centring; 1, 2: centred small-argument tiers).
template <int OP, bool HELM, int TIER>
void launch_mixed_q(int Q, dim3 grid, hipStream_t s, const dev::RegularArgs& A, const int2* tiles, int sym, int split,
                    const int2* near, int nnear) {
  dim3 ng((unsigned)((nnear + 255) / 256));
  constexpr int NC = HELM && TIER > 0 ? 1 : 0;  // the near-pair kernel runs tier 1 when centred
#define BEMPP_LAUNCH(QQ)                                                                      \
  dev::regular_p0_tiled_mixed<QQ, OP, HELM, TIER><<<dim3(grid.x * split), 256, 0, s>>>(A, tiles, sym, split); \
  if (nnear > 0) dev::near_pair_kernel<QQ, OP, HELM, NC><<<ng, 256, 0, s>>>(A, near, nnear);
  switch (Q) {
    case 1: BEMPP_LAUNCH(1); break;
    case 3: BEMPP_LAUNCH(3); break;
    case 6: BEMPP_LAUNCH(6); break;
    case 7: BEMPP_LAUNCH(7); break;
    default: throw Error("unsupported regular quadrature point count");
  }
#undef BEMPP_LAUNCH
}

template <bool HELM, int TIER>
void launch_mixed_op(int op, int Q, dim3 grid, hipStream_t s, const dev::RegularArgs& A, const int2* tiles, int sym,
                     int split, const int2* near, int nnear) {
  switch (op) {
    case kSL: launch_mixed_q<kSL, HELM, TIER>(Q, grid, s, A, tiles, sym, split, near, nnear); break;
    case kDL: launch_mixed_q<kDL, HELM, TIER>(Q, grid, s, A, tiles, sym, split, near, nnear); break;
    case kADL: launch_mixed_q<kADL, HELM, TIER>(Q, grid, s, A, tiles, sym, split, near, nnear); break;
    case kHS: launch_mixed_q<kHS, HELM, TIER>(Q, grid, s, A, tiles, sym, split, near, nnear); break;
    default: throw Error("operator not supported by the dense assembler");
  }
}

void launch_mixed(int op, bool helm, int tier, int Q, dim3 grid, hipStream_t s, const dev::RegularArgs& A,
                  const int2* tiles, int sym, int split, const int2* near, int nnear) {
  if (!helm) launch_mixed_op<false, 1>(op, Q, grid, s, A, tiles, sym, split, near, nnear);
  else if (tier == 2) launch_mixed_op<true, 2>(op, Q, grid, s, A, tiles, sym, split, near, nnear);
  else if (tier == 1) launch_mixed_op<true, 1>(op, Q, grid, s, A, tiles, sym, split, near, nnear);
  else launch_mixed_op<true, 0>(op, Q, grid, s, A, tiles, sym, split, near, nnear);
  HIP_CHECK(hipGetLastError());
}

template <bool HELM, bool P0P0, int TIER>
void launch_singular_t(int op, dim3 grid, hipStream_t s, const dev::SingularArgs& A) {
  switch (op) {
    case kSL: dev::singular_kernel<kSL, HELM, P0P0, TIER><<<grid, 256, 0, s>>>(A); break;
    case kDL: dev::singular_kernel<kDL, HELM, P0P0, TIER><<<grid, 256, 0, s>>>(A); break;
    case kADL: dev::singular_kernel<kADL, HELM, P0P0, TIER><<<grid, 256, 0, s>>>(A); break;
    case kHS: dev::singular_kernel<kHS, HELM, P0P0, TIER><<<grid, 256, 0, s>>>(A); break;
    default: throw Error("operator not supported by the dense assembler");
  }
}

template <bool HELM, int TIER>
void launch_singular_s(int op, bool p0p0, dim3 grid, hipStream_t s, const dev::SingularArgs& A) {
  if (p0p0) launch_singular_t<HELM, true, TIER>(op, grid, s, A);
  else launch_singular_t<HELM, false, TIER>(op, grid, s, A);
}

// tier (Helmholtz): Prepared::adjacent_tier
void launch_singular(int op, bool helm, bool p0p0, int tier, dim3 grid, hipStream_t s, const dev::SingularArgs& A) {
  if (!helm) launch_singular_s<false, 0>(op, p0p0, grid, s, A);
  else if (tier == 1) launch_singular_s<true, 1>(op, p0p0, grid, s, A);
  else if (tier == 3) launch_singular_s<true, 3>(op, p0p0, grid, s, A);
  else launch_singular_s<true, 0>(op, p0p0, grid, s, A);
  HIP_CHECK(hipGetLastError());
}

// Largest distance of a point of the rule from the centroid of a cell of radius 1: |1 - 3 a| of an
// S21 orbit (c + t (V_k - c), t = 1 - 3 a); for other points the offset is a non-negative
// combination of two vertex offsets with weights summing to 1 - 3 min(lambda).
double rule_radius(const RuleGroups& rg) {
  double t = 0.0;
  for (size_t m = 0; m < rg.groups.size(); ++m) {
    const RuleGroup& r = rg.groups[m];
    const double least = std::min(r.g, std::min(r.g + r.p, r.g + r.s));
    t = std::max(t, (int)m < rg.n21 ? std::fabs(r.p) : 1.0 - 3.0 * least);
  }
  return t;
}

}  // namespace

NoDeviceAllocScope::NoDeviceAllocScope() { ++t_no_device_alloc; }
NoDeviceAllocScope::~NoDeviceAllocScope() { --t_no_device_alloc; }

void check_assembler(const Assembler& a, const FunctionSpace& trial, const FunctionSpace& test) {
  if (a.op != kSL && a.op != kDL && a.op != kADL && a.op != kHS)
    throw Error("operator type not supported for dense assembly");
  if ((a.kind == kLaplace) == is_complex(a.dtype)) throw Error("dtype does not match the kernel");
  (void)trial;
  (void)test;
}

Prepared prepare(const Assembler& a, const FunctionSpace& trial_c, const FunctionSpace& test_c, void* out,
                 void* stream, bool caller_stream, bool regular) {
  check_assembler(a, trial_c, test_c);
  require_triangles(test_c, "this entry point");
  require_triangles(trial_c, "this entry point");
  auto& trial = const_cast<FunctionSpace&>(trial_c);
  auto& test = const_cast<FunctionSpace&>(test_c);
  auto& tgrid = const_cast<Grid&>(*test.grid);
  auto& sgrid = const_cast<Grid&>(*trial.grid);
  Prepared P{};
  P.device = current_device();
  P.stream = (stream || caller_stream) ? (hipStream_t)stream : assembler_stream(a, P.device);
  P.Q = regular_points(a.options);
  std::vector<double> xi, w;
  triangle_rule(P.Q, xi, w);
  const int nsing = singular_points(a.options);
  if (nsing < 1 || nsing > 64) throw Error("singular quadrature degree must be in [1, 64]");
  P.same_grid = test.grid == trial.grid;
  // the device sine/cosine reduces k r exactly only while k r <= 1e8
  if (a.kind == kHelmholtz) {
    double lo[3] = {1e300, 1e300, 1e300}, hi[3] = {-1e300, -1e300, -1e300};
    for (const Grid* g : {test.grid, trial.grid})
      for (int64_t v = 0; v < g->nv(); ++v)
        for (int d = 0; d < 3; ++d) {
          lo[d] = std::min(lo[d], g->points[3 * v + d]);
          hi[d] = std::max(hi[d], g->points[3 * v + d]);
        }
    double diag = 0.0;
    for (int d = 0; d < 3; ++d) diag += (hi[d] - lo[d]) * (hi[d] - lo[d]);
    if (!(std::fabs(a.k) * std::sqrt(diag) <= 1e8))
      throw Error("|k| times the mesh diameter exceeds 1e8 (or is not finite)");
  }

  DeviceGridCache* tc = grid_cache(tgrid, P.device);
  DeviceGridCache* sc = P.same_grid ? tc : grid_cache(sgrid, P.device);
  // |k (r - R)| <= |k| t (rad_test + rad_trial) for every quadrature-point pair of a regular cell
  // pair, t the rule's largest point radius in a cell of radius 1; the small-argument
  // sine/cosine needs this bound <= 0.25 (tier 2), 0.5 (tier 1) or 1.5 (tier 3), and beyond that
  // every point pair takes a full reduction (tier 0): Helmholtz single layer P0, 5120 cells, k = 10
  // (bound 0.69) takes 0.62 ms in tier 3, 0.83 ms in tier 0
  const RuleGroups rg = rule_groups(P.Q);
  const double phase_bound = std::fabs(a.k) * rule_radius(rg) * (tc->max_radius + sc->max_radius) * (1.0 + 1e-12);
  const bool centred = a.kind == kHelmholtz && dev::scalable(a.k, tc->max_radius + sc->max_radius);
  P.tier = !centred ? 0 : phase_bound <= 0.25 ? 2 : phase_bound <= 0.5 ? 1 : phase_bound <= 1.5 ? 3 : 0;
  // points of two cells sharing a vertex are at most two longest edges apart (each is within one
  // of the vertex)
  const double adjacent_bound = std::fabs(a.k) * 2.0 * tc->max_edge * (1.0 + 1e-12);
  P.adjacent_tier = a.kind != kHelmholtz || !P.same_grid ? 0 : adjacent_bound <= 0.5 ? 1 : adjacent_bound <= 1.5 ? 3 : 0;
  dev::RegularArgs& R = P.R;
  RuleData test_rule, trial_rule;
  if (regular) {
    test_rule = grid_rule_data(tgrid, tc, P.Q, xi, w);
    trial_rule = grid_rule_data(sgrid, sc, P.Q, xi, w);
  }
  R.test_pts = test_rule.pts;
  R.trial_pts = trial_rule.pts;
  R.nq = P.Q;
  R.rule_tab = regular_rule_table(P.device, P.Q, xi, w);
  // the FP64 P0 x P0 tiles compiled for a point count take both rules' points in orbit
  // form; other rules run the tiles with the point count at run time
  const bool compiled_q = kernel_q(P.Q) != 0;
  R.orbit_form = compiled_q && rule_in_orbit_form(P.Q, xi, w) ? 1 : 0;
  if (compiled_q && !R.orbit_form && test.nb == 1 && trial.nb == 1)
    throw Error("P0 tiles: quadrature rule not in the tabulated orbit form");
  R.test_vtx64 = test_rule.vtx;
  R.trial_vtx64 = trial_rule.vtx;
  // the same rule in groups of three points, for the P1 kernels and the rules that are not compiled
  R.groups = group_table(P.device, P.Q, test.nb, trial.nb, rg);
  R.n21 = rg.n21;
  R.ngroups = (int)rg.groups.size();
  R.wc = rg.wc;
  R.wc_test = test.nb == 3 ? rg.wc / 3.0 : rg.wc;
  R.wc_trial = trial.nb == 3 ? rg.wc / 3.0 : rg.wc;
  R.trial_gq = trial_rule.gq;
  // mixed precision: one grid (P0 x P0: p0 mixed tiles; a P1 side: LDS mixed tiles), rules
  // compiled for their point count; other rules assemble in FP64. The Laplace hypersingular
  // operator on P1 x P1 also stays in FP64: its cell-pair sum is the single-layer sum, which
  // the FP64 tiles take in orbit form, and with the P1 scatter around it that runs faster
  // than the FP32 point pairs of the mixed tiles (FP32 without packed math issues at the
  // FP64 rate)
  const bool laplace_hs_p1 = a.kind == kLaplace && a.op == kHS && test.nb == 3 && trial.nb == 3 && R.orbit_form;
  // The FP32 point pairs of the Helmholtz tiles are in lengths scaled by |k|: (|k| r)^-3 overflows below
  // |k| r = 1e-13 and |k|^3 underflows below |k| = 1e-13 (NaN from there on), so wavenumbers
  // that near to zero (k = 0 itself runs the Laplace tiles) stay in FP64.
  const double scaled = std::fabs(a.k) * std::min(1.0, tc->min_radius);
  const bool too_small = a.kind == kHelmholtz && a.k != 0.0 && scaled < 1e-12;
  P.mixed = a.options.precision == kMixed && P.same_grid && compiled_q && !laplace_hs_p1 && !too_small && regular;
  P.near = nullptr;
  P.nnear = 0;
  P.near_segs = nullptr;
  P.nsegs = 0;
  R.test_pts32 = R.trial_pts32 = nullptr;
  R.trial_vtx32 = nullptr;
  R.far_tiles = nullptr;
  R.far_tiles_ld = 0;
  if (P.mixed) {
    // the mixed P0 tiles sum point pairs per weight class and take the trial points in
    // orbit form (kernels_mixed.hpp)
    if (!rule_in_orbit_form(P.Q, xi, w))
      throw Error("mixed precision: quadrature rule not in the tabulated orbit form");
    R.test_pts32 = R.trial_pts32 = grid_points32_for_rule(tgrid, tc, P.Q, xi, w);
    R.trial_vtx32 = grid_vertex32_for_rule(tgrid, tc, P.Q, w);
    R.far_tiles = grid_far_tiles(tgrid, tc, &R.far_tiles_ld);
    P.near = grid_near_pairs(tgrid, tc, &P.nnear, &P.near_segs, &P.nsegs);
  }
  R.test_geo = tc->geo;
  R.trial_geo = sc->geo;
  R.test_vid = tc->vid;
  R.trial_vid = sc->vid;
  R.test_dofs = space_dofs(test, P.device);
  R.trial_dofs = space_dofs(trial, P.device);
  R.n_test = (int)tgrid.nc();
  R.n_trial = (int)sgrid.nc();
  R.nbt = test.nb;
  R.nbs = trial.nb;
  R.same_grid = P.same_grid ? 1 : 0;
  R.k = a.k;
  for (int p = 0; p < dev::kMaxQ; ++p)
    for (int b = 0; b < 3; ++b) R.phi[p][b] = 0.0;
  for (int p = 0; p < std::min(P.Q, dev::kMaxQ); ++p) {
    R.phi[p][0] = 1.0 - xi[2 * p] - xi[2 * p + 1];
    R.phi[p][1] = xi[2 * p];
    R.phi[p][2] = xi[2 * p + 1];
  }
  for (int p = 0; p < dev::kMaxQ; ++p)
    for (int b = 0; b < 3; ++b) {
      const bool on = p < P.Q;
      R.wphi_test[p][b] = on ? (float)(w[p] * (test.nb == 3 ? R.phi[p][b] : (b == 0 ? 1.0 : 0.0))) : 0.0f;
      R.wphi_trial[p][b] = on ? (float)(w[p] * (trial.nb == 3 ? R.phi[p][b] : (b == 0 ? 1.0 : 0.0))) : 0.0f;
    }
  R.out = out;
  R.ld = (long long)test.size;
  R.out_type = out_type(a.dtype);

  P.npairs = 0;
  if (P.same_grid) {
    const RuleTable& rt = rule_table(P.device, nsing);
    dev::SingularArgs& S = P.S;
    S.pairs = grid_pairs(tgrid, tc, &P.npairs);
    S.npairs = P.npairs;
    S.rule_aos = rt.aos;
    for (int m = 0; m < 4; ++m) {
      S.rule_off[m] = rt.off[m];
      S.rule_n[m] = rt.n[m];
    }
    S.test_geo = tc->geo;
    S.trial_geo = tc->geo;
    S.test_dofs = R.test_dofs;
    S.trial_dofs = R.trial_dofs;
    S.nbt = test.nb;
    S.nbs = trial.nb;
    S.k = a.k;
    S.out = out;
    S.ld = R.ld;
    S.out_type = R.out_type;
  }
  return P;
}

const int2* p0_tile_list(const Prepared& P, bool symmetric, int* ntiles, int* split) {
  const int nta = (P.R.n_test + dev::kTile - 1) / dev::kTile, ntb = (P.R.n_trial + dev::kTile - 1) / dev::kTile;
  const int2* t = tile_list(P.device, nta, ntb, symmetric, ntiles);
  *split = tile_split(*ntiles, kSplitP0);
  return t;
}

void apply_adjacent(const Assembler& a, const Prepared& P, const double* u, double* y, bool transpose) {
  if (P.npairs == 0) return;
  dev::SingularArgs S = P.S;
  S.mode = dev::kApply;
  S.out = y;
  S.u = u;
  S.transpose = transpose ? 1 : 0;
  launch_singular(a.op, a.kind == kHelmholtz, true, P.adjacent_tier, dim3((unsigned)((P.npairs + 3) / 4)), P.stream, S);
}

// Geometry, rule tables and adjacent pairs for the matrix-free kernels (gradient.hip).
GradientInputs gradient_inputs(const Assembler& a, const FunctionSpace& trial, const FunctionSpace& test,
                               void* stream, bool caller_stream) {
  Prepared P = prepare(a, trial, test, nullptr, stream, caller_stream);
  GradientInputs g{};
  g.R = P.R;
  g.pairs = P.S.pairs;
  g.npairs = P.npairs;
  g.rule_aos = P.S.rule_aos;
  for (int m = 0; m < 4; ++m) {
    g.rule_off[m] = P.S.rule_off[m];
    g.rule_n[m] = P.S.rule_n[m];
  }
  g.tier = P.tier;
  g.adjacent_tier = P.adjacent_tier;
  g.Q = P.Q;
  g.device = P.device;
  g.stream = P.stream;
  return g;
}

void assemble_device(const Assembler& a, const FunctionSpace& trial, const FunctionSpace& test, void* dev_out,
                     bool accumulate, void* stream) {
  if (!dev_out) throw Error("output pointer is null");
  if (test.grid->general() || trial.grid->general()) {
    // grids with quadrilateral cells: the general-cell kernels (FP64 for every precision mode)
    check_assembler(a, trial, test);
    (void)current_device();
    assemble_cells_device(a, trial, test, dev_out, accumulate, stream);
    return;
  }
  Prepared P = prepare(a, trial, test, dev_out, stream);
  P.stream = (hipStream_t)stream;  // device entry point: the caller's stream, NULL = the null stream
  const bool p0p0 = test.nb == 1 && trial.nb == 1;
  const long long n_out = (long long)test.size * (long long)trial.size * (is_complex(a.dtype) ? 2 : 1);
  // a P1 side: tiles with LDS accumulation when the blocks' DOF lists fit in LDS, else the general
  // kernel, which stores directly when every entry belongs to one cell pair
  const DeviceSpaceCache *tb = nullptr, *sb = nullptr;
  size_t lds = 0;
  bool tiles_fit = false, exclusive = p0p0;
  if (!p0p0) {
    tb = space_blocks(const_cast<FunctionSpace&>(test), P.device);
    sb = space_blocks(const_cast<FunctionSpace&>(trial), P.device);
    lds = (size_t)tb->max_nd * (size_t)sb->max_nd * sizeof(double) * (a.kind == kHelmholtz ? 2 : 1);
    // + the kernels' static LDS: the flush's copies of the blocks' DOF numbers (2 x 256 ints)
    // and the hypersingular kernels' curls (6 x 64 doubles)
    tiles_fit = lds + 2 * 256 * sizeof(int) + 6 * 64 * sizeof(double) <= max_tile_lds(P.device);
    exclusive = !tiles_fit && test.size == test.nb * (int64_t)P.R.n_test && trial.size == trial.nb * (int64_t)P.R.n_trial;
  }
  if (!exclusive && !accumulate) {
    // a fill kernel, not a memset node: the caller may capture this stream in a graph
    if (a.dtype == kF32 || a.dtype == kC32)
      dev::fill_zero_kernel<<<2048, 256, 0, P.stream>>>((float*)dev_out, n_out);
    else
      dev::fill_zero_kernel<<<2048, 256, 0, P.stream>>>((double*)dev_out, n_out);
    HIP_CHECK(hipGetLastError());
  }
  // regular pairs
  dev::RegularArgs R = P.R;
  R.mode = exclusive ? (accumulate ? dev::kAccumulate : dev::kStore) : dev::kAtomic;
  const int bx = (R.n_test + 255) / 256;
  // trial chunk: enough blocks to fill 256 CUs several times over (at least four cells / one, Helmholtz
  // single layer on discontinuous P1, 320 cells: 54 / 42 us)
  long long chunk = ((long long)bx * R.n_trial + 16383) / 16384;
  chunk = std::max(1LL, std::min(128LL, chunk));
  chunk = std::max(chunk, ((long long)R.n_trial + 65534) / 65535);
  R.trial_chunk = (int)chunk;
  dim3 grid(bx, (unsigned)((R.n_trial + chunk - 1) / chunk));
  auto& am = const_cast<Assembler&>(a);
  if (a.profiling) {
    for (int e = 0; e < 4; ++e)
      if (!am.events[e]) {
        hipEvent_t ev;
        HIP_CHECK(hipEventCreate(&ev));
        am.events[e] = ev;
      }
    am.events_recorded[0] = am.events_recorded[1] = false;
  }
  if (R.n_test > 0 && R.n_trial > 0) {
    if (a.profiling) HIP_CHECK(hipEventRecord((hipEvent_t)am.events[0], P.stream));
    if (p0p0) {
      // symmetric operators on one space: upper-triangle tiles, mirrored writes
      // (a P0 space is determined by its grid, so same grid means same space)
      const bool sym = (a.op == kSL || a.op == kHS) && P.same_grid;
      const int nta = (R.n_test + dev::kTile - 1) / dev::kTile, ntb = (R.n_trial + dev::kTile - 1) / dev::kTile;
      int ntiles = 0;
      const int2* tiles = tile_list(P.device, nta, ntb, sym, &ntiles);
      if (P.mixed) {
        launch_mixed(a.op, a.kind == kHelmholtz, P.tier, P.Q, dim3(ntiles), P.stream, R, tiles, sym ? 1 : 0,
                     tile_split(ntiles, kSplitP0), P.near, P.nnear);
      } else {
        launch_regular(a.op, a.kind == kHelmholtz, P.tier, 1, P.Q, dim3(ntiles), P.stream, R, tiles,
                       sym ? 1 : 0, tile_split(ntiles, kSplitP0));
      }
    } else {
      if (tiles_fit) {
        R.test_blk_off = tb->blk_off;
        R.test_blk_dofs = tb->blk_dofs;
        R.test_ldof = tb->ldof;
        R.trial_blk_off = sb->blk_off;
        R.trial_blk_dofs = sb->blk_dofs;
        R.trial_ldof = sb->ldof;
        // symmetric operators on one space (the DOF numbering is fixed by grid and family)
        const bool sym = (a.op == kSL || a.op == kHS) && P.same_grid && test.nb == trial.nb &&
                         test.degree == trial.degree && test.continuous == trial.continuous;
        const int nta = (R.n_test + dev::kTile - 1) / dev::kTile, ntb = (R.n_trial + dev::kTile - 1) / dev::kTile;
        int ntiles = 0;
        const int2* tiles = tile_list(P.device, nta, ntb, sym, &ntiles);
        // (blocks of many DOFs, as of meshes numbered in rows, are in FP64 whatever the precision asked for)
        if (P.mixed && (size_t)tb->max_nd * sb->max_nd * sizeof(double2) <= kMixedTileLds)
          launch_mixed_lds(a.op, a.kind == kHelmholtz, P.tier, P.Q, dim3(ntiles), P.stream, R, tiles, sym ? 1 : 0,
                           tile_split(ntiles, kSplitP1), lds, P.near, P.near_segs, P.nsegs);
        else
          launch_regular(a.op, a.kind == kHelmholtz, P.tier, 2, P.Q, dim3(ntiles), P.stream, R, tiles,
                         sym ? 1 : 0, tile_split(ntiles, kSplitP1), lds);
      } else {
        launch_regular(a.op, a.kind == kHelmholtz, P.tier, 0, P.Q, grid, P.stream, R);
      }
    }
    if (a.profiling) {
      HIP_CHECK(hipEventRecord((hipEvent_t)am.events[1], P.stream));
      am.events_recorded[0] = true;
    }
  }
  // adjacent pairs
  if (P.npairs > 0) {
    dev::SingularArgs S = P.S;
    S.mode = p0p0 ? dev::kAccumulate : dev::kAtomic;
    dim3 sg((unsigned)((P.npairs + 3) / 4));
    if (a.profiling) HIP_CHECK(hipEventRecord((hipEvent_t)am.events[2], P.stream));
    launch_singular(a.op, a.kind == kHelmholtz, p0p0, P.adjacent_tier, sg, P.stream, S);
    if (a.profiling) {
      HIP_CHECK(hipEventRecord((hipEvent_t)am.events[3], P.stream));
      am.events_recorded[1] = true;
    }
  }
}

void kernel_times(const Assembler& a, float* ms) {
  for (int k = 0; k < 2; ++k) {
    ms[k] = -1.0f;
    if (!a.events_recorded[k]) continue;
    HIP_CHECK(hipEventSynchronize((hipEvent_t)a.events[2 * k + 1]));
    HIP_CHECK(hipEventElapsedTime(&ms[k], (hipEvent_t)a.events[2 * k], (hipEvent_t)a.events[2 * k + 1]));
  }
}

// Refuses a device staging buffer larger than the free device memory with a clear error.
static void check_device_memory(size_t bytes, const char* what) {
  size_t free_b = 0, total_b = 0;
  HIP_CHECK(hipMemGetInfo(&free_b, &total_b));
  if (bytes > free_b)
    throw Error(std::string(what) + " needs " + std::to_string(bytes) + " bytes of device memory, " +
                std::to_string(free_b) + " of " + std::to_string(total_b) + " are free");
}

void assemble_host(const Assembler& a, const FunctionSpace& trial, const FunctionSpace& test, void* host_out) {
  if (!host_out) throw Error("output pointer is null");
  const int device = current_device();
  (void)device;
  const size_t bytes = (size_t)test.size * (size_t)trial.size * dtype_size(a.dtype);
  check_device_memory(bytes, "assembly into host memory (staged on the device)");
  void* d = nullptr;
  HIP_CHECK(hipMalloc(&d, std::max<size_t>(bytes, 1)));
  try {
    hipStream_t s = assembler_stream(a, device);
    if (bytes) HIP_CHECK(hipMemcpyAsync(d, host_out, bytes, hipMemcpyHostToDevice, s));
    assemble_device(a, trial, test, d, true, s);
    if (bytes) HIP_CHECK(hipMemcpyAsync(host_out, d, bytes, hipMemcpyDeviceToHost, s));
    HIP_CHECK(hipStreamSynchronize(s));
  } catch (...) {
    (void)hipFree(d);
    throw;
  }
  HIP_CHECK(hipFree(d));
}

template <int OP, bool HELM>
void launch_correction_q(int Q, dim3 grid, hipStream_t s, const dev::RegularArgs& R, const int4* pairs, int n,
                         double* out) {
  switch (Q) {
    case 1: dev::correction_kernel<1, OP, HELM><<<grid, 256, 0, s>>>(R, pairs, n, out); break;
    case 3: dev::correction_kernel<3, OP, HELM><<<grid, 256, 0, s>>>(R, pairs, n, out); break;
    case 6: dev::correction_kernel<6, OP, HELM><<<grid, 256, 0, s>>>(R, pairs, n, out); break;
    case 7: dev::correction_kernel<7, OP, HELM><<<grid, 256, 0, s>>>(R, pairs, n, out); break;
    default: dev::correction_kernel<0, OP, HELM><<<grid, 256, 0, s>>>(R, pairs, n, out); break;
  }
}

template <bool HELM>
void launch_correction(int op, int Q, dim3 grid, hipStream_t s, const dev::RegularArgs& R, const int4* pairs, int n,
                       double* out) {
  switch (op) {
    case kSL: launch_correction_q<kSL, HELM>(Q, grid, s, R, pairs, n, out); break;
    case kDL: launch_correction_q<kDL, HELM>(Q, grid, s, R, pairs, n, out); break;
    case kADL: launch_correction_q<kADL, HELM>(Q, grid, s, R, pairs, n, out); break;
    case kHS: launch_correction_q<kHS, HELM>(Q, grid, s, R, pairs, n, out); break;
    default: throw Error("operator not supported");
  }
}

// Values of the adjacent pairs in COO layout [npairs][nbt * nbs] (re, im), position
// pair * nbt * nbs + t + nbt * b: the Duffy rules (correction = false) or the regular rule
// (the singular correction). Returns a new device buffer; the caller frees it.
static double* adjacent_coo_values(const Assembler& a, const FunctionSpace& trial, const FunctionSpace& test,
                                   const Prepared& P, bool correction) {
  const size_t nvals = (size_t)P.npairs * test.nb * trial.nb;
  double* d = nullptr;
  HIP_CHECK(hipMalloc((void**)&d, nvals * 2 * sizeof(double)));
  try {
    if (correction) {
      const dim3 grid((unsigned)((P.npairs + 255) / 256));
      if (a.kind == kHelmholtz) launch_correction<true>(a.op, P.Q, grid, P.stream, P.R, P.S.pairs, P.npairs, d);
      else launch_correction<false>(a.op, P.Q, grid, P.stream, P.R, P.S.pairs, P.npairs, d);
    } else {
      dev::SingularArgs S = P.S;
      S.mode = dev::kCoo;
      S.out = d;
      dim3 sg((unsigned)((P.npairs + 3) / 4));
      launch_singular(a.op, a.kind == kHelmholtz, test.nb == 1 && trial.nb == 1, P.adjacent_tier, sg, P.stream, S);
    }
    HIP_CHECK(hipGetLastError());
  } catch (...) {
    (void)hipFree(d);
    throw;
  }
  return d;
}

void coo_to_csr_device(const double* vals, const int4* pairs, int npairs, const int* test_dofs, int nbt, int tstride,
                       const int* trial_dofs, int nbs, int sstride, int64_t nrows, int64_t ncols, DType dtype,
                       hipStream_t s, CsrHost& out);  // csr.hip

void assemble_singular_csr(const Assembler& a, const FunctionSpace& trial, const FunctionSpace& test, bool correction,
                           CsrHost& out) {
  if (test.grid->general() || trial.grid->general()) {
    check_assembler(a, trial, test);
    assemble_cells_singular_csr(a, trial, test, correction, assembler_stream(a, current_device()), out);
    return;
  }
  out.indptr.assign((size_t)test.size + 1, 0);
  out.indices.clear();
  out.data.clear();
  if (test.grid != trial.grid) return;  // no neighbouring cells across grids (:240-243)
  // (the Duffy rules read no regular-rule data: of 20480 cells 5.9 MB to build and upload)
  Prepared P = prepare(a, trial, test, nullptr, nullptr, false, correction);
  if (P.npairs == 0) return;
  double* d = adjacent_coo_values(a, trial, test, P, correction);
  try {
    coo_to_csr_device(d, P.S.pairs, P.npairs, P.S.test_dofs, test.nb, test.nb, P.S.trial_dofs, trial.nb, trial.nb,
                      test.size, trial.size, a.dtype, P.stream, out);
  } catch (...) {
    (void)hipFree(d);
    throw;
  }
  HIP_CHECK(hipFree(d));
}

// ---- potential (off-surface) operators ----
// The distinct blocks of a cell's DOFs, in the order of its DOFs.
static int cell_dof_blocks(const FunctionSpace& s, int64_t cell, int64_t (&blk)[3]) {
  int n = 0;
  for (int a = 0; a < s.nb; ++a) {
    const int64_t b = s.dofs[cell * s.nb + a] / kPotentialDofs;
    if (std::find(blk, blk + n, b) == blk + n) blk[n++] = b;
  }
  return n;
}

// Evaluations of the space's cells by blocks: the cells that the blocks list, with repetitions.
static int64_t potential_entries(FunctionSpace& s, int device) {
  space_dofs(s, device);
  std::lock_guard<std::mutex> lk(s.cache_mutex);
  DeviceSpaceCache* c = s.device_cache.at(device);
  if (c->pot_entries < 0) {
    int64_t blk[3], n = 0;
    for (int64_t cell = 0; cell < s.grid->nc(); ++cell) n += cell_dof_blocks(s, cell, blk);
    c->pot_entries = n;
  }
  return c->pot_entries;
}

// DOF blocks of a space for the potential kernel (PotentialInputs): each DOF belongs to one
// block, so the block's workgroups sum its entries over the listed cells and write each once.
static const DeviceSpaceCache* potential_blocks(FunctionSpace& s, int device) {
  space_dofs(s, device);
  std::lock_guard<std::mutex> lk(s.cache_mutex);
  DeviceSpaceCache* c = s.device_cache.at(device);
  if (c->pot_off) return c;
  const int64_t nc = s.grid->nc();
  const int nb = s.nb;
  const int64_t nblk = (s.size + kPotentialDofs - 1) / kPotentialDofs;
  std::vector<int> off(nblk + 1, 0);
  int64_t blk[3];
  for (int64_t cell = 0; cell < nc; ++cell)
    for (int m = cell_dof_blocks(s, cell, blk) - 1; m >= 0; --m) ++off[blk[m] + 1];
  for (int64_t b = 0; b < nblk; ++b) off[b + 1] += off[b];
  // one upload: off, cells, ldof back to back
  const size_t ne = (size_t)off[nblk];
  std::vector<int> lists(off), at(off.begin(), off.end() - 1);
  lists.resize(nblk + 1 + ne * (1 + nb));
  int* cells = lists.data() + nblk + 1;
  int* ldof = cells + ne;
  for (int64_t cell = 0; cell < nc; ++cell)
    for (int m = cell_dof_blocks(s, cell, blk) - 1; m >= 0; --m) {
      const int e = at[blk[m]]++;
      cells[e] = (int)cell;
      for (int a = 0; a < nb; ++a) {
        const int64_t d = s.dofs[cell * nb + a];
        ldof[(size_t)e * nb + a] = d / kPotentialDofs == blk[m] ? (int)(d % kPotentialDofs) : -1;
      }
    }
  c->pot_off = upload(lists);
  c->pot_cells = c->pot_off + nblk + 1;
  c->pot_ldof = c->pot_cells + ne;
  c->pot_nblocks = (int)nblk;
  return c;
}

static bool potential_blocks_built(FunctionSpace& s, int device) {
  std::lock_guard<std::mutex> lk(s.cache_mutex);
  auto it = s.device_cache.find(device);
  return it != s.device_cache.end() && it->second->pot_off;
}

PotentialInputs potential_inputs(const Assembler& a, const FunctionSpace& space_c, int64_t npoints, void* stream) {
  auto& space = const_cast<FunctionSpace&>(space_c);
  auto& grid = const_cast<Grid&>(*space.grid);
  const int device = current_device();
  PotentialInputs P{};
  P.Q = regular_points(a.options);
  std::vector<double> xi, w;
  triangle_rule(P.Q, xi, w);
  DeviceGridCache* gc = grid_cache(grid, device);
  const RuleData rule = grid_rule_data(grid, gc, P.Q, xi, w);
  P.pts = rule.pts;
  P.geo = gc->geo;
  P.rule_tab = weighted_rule_table(device, P.Q, xi, w);
  const RuleGroups rg = rule_groups(P.Q);
  P.vtx = rule.vtx;
  P.gq = rule.gq;
  P.groups = group_table(device, P.Q, space.nb, space.nb, rg);
  P.n21 = rg.n21;
  P.ngroups = (int)rg.groups.size();
  P.wc = rg.wc;
  P.wc_trial = space.nb == 3 ? rg.wc / 3.0 : rg.wc;
  // DOF blocks pay where cells share DOFs, but a cell at their borders is evaluated for each: 1.57 times on an
  // icosphere, 2.48 times in random cell order. Many evaluations, or few workgroups, cost more than the atomics of
  // taking the cells once. P1, 16 points, blocks / cells once: Laplace single layer, 306 workgroups of blocks,
  // 34.6 / 31 us, 480: 40 / 36.5, 3807: 193 / 280; Helmholtz double layer, 84: 48.5 / 30; 6 points, 90: 24.4 / 27.
  // By evaluations of rule points a cell, 5120 cells, 10007 points: Laplace single layer, 25: 555 / 986, 40:
  // 880 / 973 (1000 points: 111 / 99), 58: 1120 / 1050, 92: 1760 / 1028; Helmholtz double layer, 58: 3246 / 3999,
  // 92: 5104 / 3993; 50 points: Helmholtz double layer, 21 workgroups, 9: 23 / 16, 81 workgroups, 9: 23 / 25, 15:
  // 33 / 24, 321 workgroups, 15: 64 / 78; Laplace, 15: 31 / 26. Nothing is built while the stream is captured:
  // blocks only if an earlier call did.
  const long long pblocks = (npoints + 63) / 64, dblocks = (space.size + kPotentialDofs - 1) / kPotentialDofs;
  const long long groups = pblocks * dblocks;
  const bool shared_dofs = space.size < (int64_t)space.nb * grid.nc();
  bool blocks = shared_dofs && (P.Q <= dev::kMaxQ || groups >= 512);
  if (blocks) {
    const double evaluations = (double)potential_entries(space, device) / (double)grid.nc() * P.Q;
    blocks = evaluations <= (a.kind == kHelmholtz ? std::min(80.0, groups / 4.0 - 10.0)
                                                  : std::min(35.0, std::max(10.0, groups / 24.0)));
  }
  if (blocks && stream) {
    hipStreamCaptureStatus capture = hipStreamCaptureStatusNone;
    HIP_CHECK(hipStreamIsCapturing((hipStream_t)stream, &capture));
    blocks = capture == hipStreamCaptureStatusNone || potential_blocks_built(space, device);
  }
  if (blocks) {
    const DeviceSpaceCache* sc = potential_blocks(space, device);
    P.off = sc->pot_off;
    P.cells = sc->pot_cells;
    P.ldof = sc->pot_ldof;
    P.nblocks = sc->pot_nblocks;
  } else {
    P.ldof = space_dofs(space, device);
  }
  P.ncells = (int)grid.nc();
  P.nb = space.nb;
  P.ndofs = space.size;
  P.max_radius = gc->max_radius;
  P.rule_radius = rule_radius(rg);
  P.out_type = out_type(a.dtype);
  return P;
}

void assemble_potential_host(const Assembler& a, const FunctionSpace& space, const double* points, int64_t npoints,
                             void* host_out) {
  require_triangles(space, "potential assembly");
  if (npoints == 0) return;
  if (!points || !host_out) throw Error("points or output pointer is null");
  if (a.kind == kHelmholtz) {  // the device sine/cosine reduction is exact while k r <= 1e8
    double lo[3] = {1e300, 1e300, 1e300}, hi[3] = {-1e300, -1e300, -1e300};
    auto grow = [&](const double* x) {
      for (int d = 0; d < 3; ++d) {
        lo[d] = std::min(lo[d], x[d]);
        hi[d] = std::max(hi[d], x[d]);
      }
    };
    for (int64_t v = 0; v < space.grid->nv(); ++v) grow(&space.grid->points[3 * v]);
    for (int64_t j = 0; j < npoints; ++j) grow(points + 3 * j);
    double diag = 0.0;
    for (int d = 0; d < 3; ++d) diag += (hi[d] - lo[d]) * (hi[d] - lo[d]);
    if (!(std::fabs(a.k) * std::sqrt(diag) <= 1e8)) throw Error("|k| times the extent of mesh and points exceeds 1e8");
  }
  const int device = current_device();
  const size_t bytes = (size_t)npoints * (size_t)space.size * dtype_size(a.dtype);
  check_device_memory(bytes + (size_t)npoints * 3 * sizeof(double), "potential assembly into host memory");
  void* d = nullptr;
  double* dp = nullptr;
  HIP_CHECK(hipMalloc(&d, std::max<size_t>(bytes, 1)));
  try {
    HIP_CHECK(hipMalloc((void**)&dp, (size_t)npoints * 3 * sizeof(double)));
    hipStream_t s = assembler_stream(a, device);
    HIP_CHECK(hipMemcpyAsync(dp, points, (size_t)npoints * 3 * sizeof(double), hipMemcpyHostToDevice, s));
    if (bytes) HIP_CHECK(hipMemcpyAsync(d, host_out, bytes, hipMemcpyHostToDevice, s));
    assemble_potential_device(a, space, dp, npoints, d, true, s);
    if (bytes) HIP_CHECK(hipMemcpyAsync(host_out, d, bytes, hipMemcpyDeviceToHost, s));
    HIP_CHECK(hipStreamSynchronize(s));
  } catch (...) {
    (void)hipFree(d);
    if (dp) (void)hipFree(dp);
    throw;
  }
  HIP_CHECK(hipFree(d));
  HIP_CHECK(hipFree(dp));
}

Assembler::~Assembler() {
  for (void* e : events)
    if (e) (void)hipEventDestroy((hipEvent_t)e);
  if (stream) {
    int cur = 0;
    if (hipGetDevice(&cur) == hipSuccess) {
      (void)hipSetDevice(device);
      (void)hipStreamDestroy((hipStream_t)stream);
      (void)hipSetDevice(cur);
    }
  }
}

}  // namespace bempp_amd
