// fv_tables.h -- the host-side tables of the step and adjoint launches: work
// items and their CFL lane masks, the reference fold's cell subset, the
// per-instance descriptor fields and row tables, parameter checks.  Plain
// C++ with no HIP call, so it builds and runs on any host (the runtime links
// it into libfivonagi.so; tests/sanitize builds it alone with AddressSanitizer
// and UndefinedBehaviorSanitizer).
#ifndef FIVONAGI_FV_TABLES_H
#define FIVONAGI_FV_TABLES_H

#include <stddef.h>
#include <stdint.h>

#include <string>
#include <vector>

#include "../../include/fivonagi.h"
#include "fv_adjoint.h"
#include "fv_types.h"

namespace fvh {

// Cells whose cfl reaches cfl[0] under the reference's fold
// (common/main.cu:503-524), as a 0/1 byte per cell (offset i + j*nx).
std::vector<uint8_t> fold_subset(int nx, int ny);

// 0, or an error code with *why set: the parameters every entry point that
// sets up an instance accepts.
int check_params(const fivonagi_params& q, bool f64, std::string* why);

// The host side of one instance: every scalar field of its descriptor (the
// device pointers are left null) and the tables its device copies are made
// from.
struct HostInst {
  fv::InstDesc d;                    // scalar fields; device pointers null
  std::vector<double> ec, es, tab;   // edge drive (or aperture) and HIFU row tables
  std::vector<uint32_t> fold_bits;   // kCflBitmap: bit i + j*nx = cell counted
  bool ext = false;                  // needs the extended step kernel
  int taylor_ring = 0;               // ghost ring of a Taylor instance (0: none)
};
void host_inst(const fivonagi_params& q, bool f64, HostInst& h);

// A table of doubles as the bytes of the context's precision.
void table_bytes(const std::vector<double>& v, bool f64, char* out);

// Is cell (i, j) one the CFL reduction counts, for an instance's mask kind
// (fv::CflMask) and bitmap?  (The lane masks are formed word by word; this is
// what they are checked against.)
bool cfl_counted(int cfl_mask, const std::vector<uint32_t>& fold_bits, int nx, int i, int j);

// Rows per item of the in-step cut (see build_work): the smallest height
// (never below 12) whose total wave count over all instances fits target_waves.
int auto_rows(const std::vector<fivonagi_params>& ps, long target_waves);

// Heights, bottom to top, of the waves (at most max_waves) that share R rows of
// a strip in one workgroup.
std::vector<int> group_heights(int R, int max_waves);

// Row boundaries of one strip cut into `chunks` work items (skewed heights,
// `levels` levels, the first item at level rot; the in-step cut takes 0).
std::vector<int> chunk_bounds(int ny, int chunks, float skew, int levels, int rot);

// The work list of the step kernel.
struct WorkList {
  std::vector<fv::WorkItem> items;   // workgroup by workgroup in launch order, each bottom
                                     // to top
  std::vector<int32_t> group_first;  // workgroup g: items group_first[g] .. group_first[g+1]
  std::vector<uint64_t> rowmask;     // CFL lane mask per row of each strip (fv::WorkItem::mrow)
  std::vector<int> n_items;          // per instance
  float skew_used = 0.0f;
  bool rotate_used = false;
};
// The strips are cut in one of two ways (same results):
//   running on  the strips laid end to end, dealt to workgroups of up to
//               kGroupWaves waves of about equal march steps, one above the
//               other, which hand their seam rows over in LDS;
//   in step     one wave per item, every strip of an instance cut at the same
//               rows, auto_h (or the instance's rows_per_wave) rows each.
// cus, per_cu: the device's CUs and resident step waves per CU; skew < 0:
// automatic, as the choice of the cut then is; else rotate picks running on
// (instances that ask for different rows_per_wave are always cut in step).
// cell_bytes: bytes of state, in and out, per cell.
void build_work(const std::vector<fivonagi_params>& ps, const std::vector<int>& cfl_mask,
                const std::vector<std::vector<uint32_t>>& fold_bits, long cus, int per_cu,
                int auto_h, float skew, bool rotate, WorkList& out, int cell_bytes = 24);
// The items as the step kernel reads them: kGroupWaves places per workgroup
// (an unused place has no rows).
std::vector<fv::WorkItem> launch_items(const WorkList& wl, long cus);

// Work items of the adjoint's reverse march (fv_adjoint_march.hip): strips
// of 56 output columns cut into row ranges, items in instance and strip
// order; first[k] .. first[k+1] are instance k's items, and wave w runs items
// wave_first[w] .. wave_first[w+1] in turn.  rows_per_wave > 0: items of that
// many rows, one per wave; 0: waves of about equal cost, at most target_waves
// of them, a wave taking one or more items (the end of one strip and the
// start of the next).
void build_adj_items(const std::vector<fivonagi_params>& ps, long target_waves,
                     int rows_per_wave, std::vector<fv::AdjItem>& items,
                     std::vector<size_t>& first, std::vector<int32_t>& wave_first);

}  // namespace fvh

#endif  // FIVONAGI_FV_TABLES_H
