// Arguments and launch of the clip kernels (rpd_kernels.hip).
#pragma once
#include <hip/hip_runtime.h>

#include "rpd_device.h"

namespace rpd {

// Completeness certificate of the learned path, evaluated on each cell
// when its status is final (tet_off == nullptr: off).  The cells of a tet's
// sphere set partition the tet iff the set is closed under facet
// neighbours: every active bisector facet (seed, j) of a cell must have j
// in the set -- the tet's CSR members, or a pair (tet, j) of the sorted
// ext keys added since.  A missing pair goes to miss (past cap: the tet is
// flagged); a cell that ends in a failure status flags its tet; a tet with
// a cell is marked in has_cell.
struct CertArgs {
  const int64_t* tet_off;
  const int32_t* mem_ids;
  const uint64_t* ext;
  int64_t n_ext;
  uint64_t* miss;
  int32_t cap;
  int32_t* n_miss;
  uint8_t* flag;
  uint8_t* has_cell;
  // (a captured run: the candidates of the launch, on the device; the miss
  // list then holds min(cap, max(4096, 2 * *cap_n)) entries, as the eager
  // path sizes it)
  const int64_t* cap_n;
};

struct ClipArgs {
  DevMesh M;
  DevSites S;
  const Cand* cand;
  const int32_t* items;   // cell indices to process (nullptr: item_base +
                          // item)
  int64_t item_base;
  int64_t n_items;
  SlotView out;           // indexed by slot_base + item, or by the cell
                          // index when slot_by_cell
  int64_t slot_base;
  int32_t slot_by_cell;   // items in step-count order: slot = cell index,
                          // and no XCD regrouping of the blocks
  int32_t use_mask;
  int32_t force_exact;
  int32_t geometry;
  int32_t* rerun_large;   // list + counter (small tier)
  int32_t* n_rerun_large;
  int32_t* rerun_exact;
  int32_t* n_rerun_exact;
  // a captured pipeline: n_items is the launch's capacity and the count is
  // on the device (n_items_d64, or n_items_d32 minus n_sub); the re-run
  // lists hold cap_large / cap_exact entries, more set overflow[0]
  const int64_t* n_items_d64;
  const int32_t* n_items_d32;
  int64_t n_sub;
  int32_t cap_large, cap_exact;
  int32_t* overflow;
  unsigned long long* work;  // 64 x 4 spread counters, or nullptr
  CertArgs cert;
};

// Launches the clip of a.n_items cells with G cells per wavefront: tier 0
// the small tier with the capacities caps_id of rpd_run_cfg.small_caps,
// tier 1 full capacity, tier 2 full capacity with exact arithmetic.
hipError_t clip_launch(hipStream_t s, int tier, int G, const ClipArgs& a,
                       int caps_id);

}  // namespace rpd
