// 2-D patches: the elements of a mesh cut into compact groups, each advanced
// by one workgroup that sums its element forces in LDS.
//
// A point all of whose elements lie in one patch is interior to it: the
// patch's workgroup assembles its force, divides by the mass and applies the
// corrector and the next predictor, with no force leaving the chip.  Points
// shared by several patches (1 in 13 with 45 elements a patch, 1 in 9.5 with 21)
// are boundary points: every patch stores the element contributions of its
// boundary points, and the next launch sums them (in every patch that needs
// the point, all with the same operands), so one launch carries a time step
// and no grid-wide synchronisation is needed.  Boundary state and
// contributions are double-buffered by launch parity; interior state is
// updated in place.
//
// Device point order: the interior points of patch 0, of patch 1, ..., then
// all boundary points.  Within a patch the interior points are sorted by
// their number of contributions (1, 2, more), so a wavefront's lanes sum the
// same number of terms.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>
#include <cstring>
#include <unordered_map>
#include <vector>

#include "assembly.hpp"
#include "kernels.hpp"
#include "runtime.hpp"

namespace sfx {

// Most elements of a patch: five threads each, so that a workgroup is four
// wavefronts (one per SIMD of its CU) or, on small meshes, two.
constexpr int PATCH_LARGE = 51, PATCH_SMALL = 25;
// Limits of a patch (the kernel's LDS arrays): local points and boundary
// points.  A 7 x 7 block of quads has 841 and 112.
template <int PE> struct PatchCap {
  static constexpr int points = PE == PATCH_LARGE ? 960 : 512;
  static constexpr int boundary = PE == PATCH_LARGE ? 256 : 128;
};

// Everything a workgroup needs to start, in one scalar read.  The table
// fields are offsets into the 16-bit array `tab`; patches of equal
// connectivity share their tables.
struct PatchHead {
  int el0, nel;          // elements [el0, el0 + nel) of the plan's order
  int pt0, nint;         // interior points [pt0, pt0 + nint) of the device order
  int n1, n2;            // of which the first n1 have one contribution, the next n2 two
  int nb, b0;            // boundary points: entries [b0, b0 + nb) of bpt
  int be0, nbent;        // their contributions from this patch: slots bslot[be0 ...]
  int seg0, nseg;        // Stacey segments (element points)
  int src0, nsrc;        // source elements
  int rm0;               // receiver rows of the interior points (rmap[rm0 + l]), or -1
  int sim;               // simulation the patch belongs to
  int lidx;              // (nel, 5, 8): local point of each element row's 5 points (interior first, then boundary)
  int enta;              // (nint): first contribution of each interior point: element * 25 + point; colored
                         // also PE * 25 + Stacey segment, then 25 per source element
  int entb;              // (nint - n1): second contribution
  int off3;              // (nint - n1 - n2 + 1): further ones, offsets into ent3
  int ent3;
  int bent;              // (nbent): contributions of the boundary points
  float dt, dto2, dt2o2; // constants of the simulation
  int nstep, nsb;
  int pad[5];
};

// A boundary point of a patch: its index (bit 31 set in the owning patch) and
// its contributions [k0, k0 + n).
struct PatchPoint {
  int b, k0, n, pad;
};

// Host plan over one or several meshes (a batch).
struct PatchPlan {
  int pe = PATCH_LARGE;
  std::vector<PatchHead> head;
  std::vector<uint16_t> tab;
  std::vector<int32_t> elem;       // plan order -> element of its mesh
  std::vector<PatchPoint> bpt;     // boundary points of each patch
  std::vector<int32_t> boff;       // (nbnd + 1) contributions of each boundary point
  std::vector<int32_t> bslot;      // where each patch's boundary contributions go
  int nint = 0, nbnd = 0;          // interior and boundary points
  std::vector<int> patch_end;      // patches of the first k + 1 meshes
  // while meshes are added: the distinct tables, found by what they follow from
  // and by their contents
  struct Tables {
    std::vector<uint16_t> sig, bidx;  // bidx: boundary point of each boundary contribution
    int base = 0, enta = 0, entb = 0, off3 = 0, ent3 = 0, bent = 0;
    size_t size = 0;
  };
  std::vector<Tables> tables;
  std::unordered_multimap<uint64_t, int> by_shape, by_tables;
  std::vector<std::vector<int32_t>> device_of;  // per mesh: point -> device index (boundary ones offset by nint once finished)
  std::vector<std::vector<int32_t>> slot_of;    // per mesh: element -> position in elem
};

// Most elements a patch holds, chosen so that the chip has work for every CU:
// see patch2d.cpp for the measured line.
int patch_elements(int64_t nspec);

// Adds a mesh (its elastic elements, all of them) to the plan; key[e] orders
// the contributions of a point.  Sources and Stacey terms are part of their
// element's contribution or, colored, come before and after all of them, the
// order in which the colored kernels add to the acceleration.  Call
// finish_patches after the last mesh.
void add_patches(PatchPlan &plan, const HostAssembly &h, const std::vector<int32_t> &key, bool colored);
void finish_patches(PatchPlan &plan);
// Puts the points of a single-mesh plan in device order: gather, Stacey
// points, M^-1 and lattice_of of the assembly.
void renumber_points(HostAssembly &h, const PatchPlan &plan);

// Constants of one simulation.
struct PatchSim {
  float dt, dto2, dt2o2;
  int nstep, nsb, nrec;
  long long seis;  // offset of its samples
};

struct PatchTables {
  const PatchHead *head;
  const uint16_t *tab;
  const PatchPoint *bpt;
  const int *boff, *bslot;
  const PatchSim *sim;
  Geom2D geom;                    // plan order
  const float *kappa, *mu, *kmu;  // plan order; kmu: one pair per element, or null
  const int *seg_pt;              // local element * 25 + point of each Stacey segment
  const int *seg_loc;             // its local point
  const int *seg_off;             // entries [seg_off[s], seg_off[s + 1])
  const float *bnormal, *bweight, *brvp, *brvs;
  const int4 *src_el;             // source elements: local element, sources [y, z) of src_id
  const int *src_id;              // in application order within an element
  const float *src_array;         // (nsrc, 2, 25)
  const float *stf;               // stf[step * stf_step + id * stf_src]
  long long stf_step, stf_src;
  const int4 *rec;                // receivers by patch: row of rec_h, index within the simulation, simulation, element
  const float *rec_h;             // (., 25)
  const int *rp_of;               // (nrec, 25): row of snap of each receiver element point, or -1 - boundary point
  const int *rmap;
  int nrow;                       // rows of snap
  const int *rec_row;             // plan order: Stacey element of the adjoint's record, or -1
  const int *types;
  int ntypes;
  const float *minv;              // (2, np)
  float *snap;                    // (2, rows, 6): u, corrected v, a, by launch parity
  float *seismo;
  int nint, np, nbnd;
};

// u, v, a: the flat fields (2, np); the boundary part of u, v is state A, and
// ub: state B (u0, u1, v0, v1; nbnd each).  rb: contributions (2 buffers).
struct PatchState {
  float *u, *v, *a;
  float *ub;
  float2 *rb[2];
};

// One launch.  step: this launch's step index, *base added when given; next
// (when given) receives that sum plus one.
struct PatchLaunch {
  const int *base;
  int *next;
  int step;
  int rd;        // buffers read (0: A)
  int pending;   // the contributions of step - 1 are summed first
  int advance;   // 1: corrector and predictor; 0: only a = M^-1 f (seam calls)
  int store_a;   // advance: keep a as well
  int add_a;     // contracted form, no advance: the stored a joins the sums
  float *rec;    // contracted form: the Stacey elements' forces of step n go to rec + n * rec_stride, or null
  long long rec_stride;
};

// One launch of the combined adjoint + backward loop (contracted form).
struct PatchPairLaunch {
  int step, rd, pending;
  int top;           // sample index of step 0
  const float *rec;  // the Stacey elements' forces of this step
};
struct PatchPairTables {
  const int2 *adj_head;    // adjoint source elements of each patch: [x, y) of adj_el
  const int4 *adj_el;      // local element, sources [y, z) of adj_id
  const int *adj_id;
  const float *adj_array;  // (sources, 2, 25)
  const float *adj_stf;    // [step * adj_step + id]
  long long adj_step;
  const int *kslot;        // plan order: element of Kmu, Kkappa
  float *Kmu, *Kkappa, *R;
};

// Arrays laid one after the other (256-byte boundaries) for one copy.
struct PatchBlob {
  std::vector<char> bytes;
  size_t room(size_t n) {
    const size_t at = (bytes.size() + 255) / 256 * 256;
    if (at + n > bytes.capacity()) bytes.reserve(2 * (at + n));
    bytes.resize(at + n);
    return at;
  }
  template <class T> size_t add(const std::vector<T> &v) {
    const size_t at = room(v.size() * sizeof(T));
    if (!v.empty()) std::memcpy(bytes.data() + at, v.data(), v.size() * sizeof(T));
    return at;
  }
};
// Device copies of a plan and of what the kernel reads beside it, in three
// allocations: tables, properties (set again by upload_properties) and the
// kernel's own buffers.
struct PatchDevice {
  DevBuf<char> tables_mem, props_mem;
  DevBuf<float> work;                   // boundary state B, contributions (two buffers), snapshots (two)
  std::vector<int> patch_end, rec_end;  // patches and receivers of the first k + 1 meshes
  int pe = PATCH_LARGE;
  PatchTables t{};                      // device pointers into the above
  float *ub = nullptr;
  float2 *rb[2] = {nullptr, nullptr};

  // everything of the meshes in plan order; source and receiver ids count over
  // all meshes in order (sources in application order when by_order)
  void upload(const PatchPlan &plan, const std::vector<const HostAssembly *> &meshes, bool sources_by_order,
              const std::vector<PatchSim> &sims, hipStream_t s);
  // kappa, mu and the Stacey impedances again (their meshes' values changed)
  void upload_properties(const PatchPlan &plan, const std::vector<const HostAssembly *> &meshes, hipStream_t s);
  PatchState state(float *u, float *v, float *a) const { return PatchState{u, v, a, ub, {rb[0], rb[1]}}; }
};

// One launch over the first npatch patches, and the samples of step - 1 at the
// first nrec receivers when the launch is pending.  exact: every product and
// sum rounded on its own; otherwise contracted into fused multiply-adds.
void launch_patch_step(hipStream_t s, int pe, int npatch, int nrec, bool exact, const PatchTables &t,
                       const PatchState &st, const GllConst &q, const PatchLaunch &l);
// Boundary points, from the contributions in buffer rd: with advance the
// corrector and predictor into state A (a too with store_a), else a only.
// add_a: the stored a joins the sums.
void launch_patch_boundary(hipStream_t s, bool exact, const PatchTables &t, const PatchState &st, NewmarkConst nc,
                           int rd, int advance, int store_a, int add_a);
void launch_patch_pair(hipStream_t s, int pe, int npatch, int nrec, const PatchTables &t, const PatchState &adj,
                       const PatchState &bwd, const GllConst &q, const PatchPairLaunch &l, const PatchPairTables &p);
void launch_patch_pair_boundary(hipStream_t s, const PatchTables &t, const PatchState &adj, const PatchState &bwd,
                                NewmarkConst nc, int rd, float *R);
// dst[i] = src[index[i]] / dst[index[i]] = src[i]
void launch_take(hipStream_t s, int n, const int *index, const float *src, float *dst);
void launch_put(hipStream_t s, int n, const int *index, const float *src, float *dst);

}  // namespace sfx
