// fv_tables.cpp -- host-side tables of the step and adjoint launches (see
// fv_tables.h).  No HIP call: this file builds alone on any host.
#include "fv_tables.h"

#include <algorithm>
#include <cmath>
#include <cstring>

namespace fvh {

// Cells whose cfl reaches cfl[0] under the reference's fold
// (common/main.cu:503-524): follow each cell's value forward through the
// launches.  A launch of S threads moves slot p to p - S when S <= p < 2S and
// strands slots >= 2S.
std::vector<uint8_t> fold_subset(int nx, int ny) {
  const long N = (long)nx * ny;
  std::vector<long> strides;
  long sizered = N;
  while (sizered > 32) { sizered /= 2; strides.push_back((sizered / 16) * 16); }
  while (sizered > 2) { sizered /= 2; strides.push_back(sizered); }
  // Walk the folds backwards from cfl[0].  A fold of stride S sets slot
  // i < S to max(slot i, slot i + S) and leaves the slots >= S as they are,
  // so a later fold can read such a slot again (when its stride is more than
  // S/2, as where the two loops meet).  Slots past the grid hold no cell.
  std::vector<uint8_t> m(N, 0);
  m[0] = 1;
  for (auto it = strides.rbegin(); it != strides.rend(); ++it) {
    const long S = *it;
    for (long i = 0; i < S && i + S < N; ++i)
      if (m[i]) m[i + S] = 1;
  }
  return m;
}

// Parameters every entry point that sets up an instance accepts.
int check_params(const fivonagi_params& q, bool f64, std::string* why) {
  auto fail = [&](int code, const char* msg) {
    if (why) *why = msg;
    return code;
  };
  if (q.nx < 8 || q.ny < 8) return fail(FIVONAGI_ERR_ARG, "nx, ny must be >= 8");
  // the kernels address a field with 32-bit byte offsets: at most 4 GiB
  // per field (2^30 cells in FP32, 2^29 in FP64)
  if ((long)q.nx * q.ny > (f64 ? (1L << 29) : (1L << 30)))
    return fail(FIVONAGI_ERR_ARG, "grid too large (a field must fit 4 GiB)");
  if (!(q.dx > 0) || !(q.dy > 0) || !(q.dt0 > 0) || !(q.cfl_wish > 0))
    return fail(FIVONAGI_ERR_ARG, "dx, dy, dt0, cfl_wish must be > 0");
  if (q.bc < 0 || q.bc > 3) return fail(FIVONAGI_ERR_ARG, "unknown boundary kind");
  if (q.bc == FIVONAGI_BC_HIFU &&
      !(q.hifu_f > 0 && q.hifu_frec > 0 && q.hifu_a >= 0 && std::isfinite(q.hifu_ampl)))
    return fail(FIVONAGI_ERR_ARG, "hifu: hifu_f, hifu_frec must be > 0, hifu_a >= 0");
  if (q.cfl_mode < 0 || q.cfl_mode > 1) return fail(FIVONAGI_ERR_ARG, "unknown cfl mode");
  if (q.md_on != 0 && q.md_on != 1) return fail(FIVONAGI_ERR_ARG, "md_on must be 0 or 1");
  if (q.md_on && !(q.md_vx >= 0 && q.md_vy >= 0 && std::isfinite(q.md_vx) &&
                   std::isfinite(q.md_vy) && std::isfinite(q.md_t)))
    return fail(FIVONAGI_ERR_ARG, "moving window: md_vx, md_vy must be finite and >= 0");
  return 0;
}

// The host side of one instance: every scalar field of its descriptor (the
// device pointers are left null) and the tables its device copies are made
// from -- edge drive or HIFU aperture, CFL fold subset.
void host_inst(const fivonagi_params& q, bool f64, HostInst& h) {
  fv::InstDesc& d = h.d;
  std::memset(&d, 0, sizeof(d));
  const size_t n = (size_t)q.nx * q.ny;
  d.fp64 = f64 ? 1 : 0;
  d.hbeta_d = q.beta - 1.0;
  d.hifu_k_d = q.hifu_frec / 4.0;
  // edge drive amplitude/phase folded into amp*cos(phase), amp*sin(phase);
  // the HIFU aperture's AMPL and phase delay ISPW*phi_j the same way
  h.ec.assign(q.ny, 0.0);
  h.es.assign(q.ny, 0.0);
  h.tab.clear();
  const bool hifu = q.bc == FIVONAGI_BC_HIFU;
  const double ispw = 2.0 * 3.14159265358979323846 * q.hifu_frec;   // ISPW
  if (hifu) h.tab.assign(4 * (size_t)q.ny, 0.0);
  for (int j = 0; j < q.ny; ++j) {
    if (hifu) {
      // apps/hifu-beam/boundary.h:79-90
      const int width = (int)(q.hifu_a / q.dy);
      const int jp = j - 2;
      if (jp >= 0 && jp < width) {
        const double F = q.hifu_f, jp2 = (double)jp * jp;
        const double nd = std::sqrt(jp2 + F * F);
        const double phi = (q.dx * jp2) / (2.0 * F);
        h.ec[j] = q.hifu_ampl * std::cos(ispw * phi);
        h.es[j] = q.hifu_ampl * std::sin(ispw * phi);
        h.tab[4 * (size_t)j + 0] = phi;
        h.tab[4 * (size_t)j + 1] = F / nd;
        h.tab[4 * (size_t)j + 2] = -jp / nd;
        h.tab[4 * (size_t)j + 3] = 1.0;
      }
      continue;
    }
    const double a = q.edge_amp ? q.edge_amp[j] : 0.0;
    const double ph = q.edge_phase ? q.edge_phase[j] : 0.0;
    h.ec[j] = a * std::cos(ph);
    h.es[j] = a * std::sin(ph);
  }
  d.hifu_k = (float)(q.hifu_frec / 4.0);
  // CFL subset
  d.cfl_mask = fv::kCflAll;
  h.fold_bits.clear();
  if (q.cfl_mode == FIVONAGI_CFL_REFERENCE_FOLD) {
    std::vector<uint8_t> m = fold_subset(q.nx, q.ny);
    bool even = true;
    for (size_t o = 0; o < n && even; ++o) even = (m[o] != 0) == ((o & 1) == 0);
    if (even) {
      d.cfl_mask = fv::kCflEven;
    } else {
      h.fold_bits.assign((n + 31) / 32, 0u);
      for (size_t o = 0; o < n; ++o)
        if (m[o]) h.fold_bits[o >> 5] |= 1u << (o & 31);
      d.cfl_mask = fv::kCflBitmap;
    }
  }
  d.dt_seq = nullptr;
  d.dt_seq_len = 0;
  d.dx = q.dx; d.dy = q.dy; d.delta = q.delta;
  d.cfl_max = q.cfl_max; d.cfl_wish = q.cfl_wish; d.omega = q.omega;
  d.inv_dx = 1.0 / q.dx; d.inv_dy = 1.0 / q.dy;
  d.dif_x = q.delta / (q.dx * q.dx); d.dif_y = q.delta / (q.dy * q.dy);
  d.omega_turns = (hifu ? ispw : q.omega) / 6.283185307179586476925286766559;
  d.tay_rhoa = q.tay_rhoa; d.tay_c = q.tay_c;
  d.tay_cos = std::cos(q.tay_theta); d.tay_sin = std::sin(q.tay_theta);
  d.tay_yoff = q.tay_yoff; d.tay_jc = q.tay_jc;
  d.nx = q.nx; d.ny = q.ny; d.bc = q.bc;
  h.taylor_ring = q.bc == FIVONAGI_BC_TAYLOR ? 4 * q.nx + 4 * (q.ny - 4) : 0;
  d.beta2m2 = (float)(2.0 * (q.beta - 1.0));
  d.md_on = q.md_on;
  d.md_vx = q.md_vx; d.md_vy = q.md_vy; d.md_t = q.md_t;
  h.ext = hifu || q.md_on;
}

// A table of doubles as the bytes of the context's precision.
void table_bytes(const std::vector<double>& v, bool f64, char* out) {
  if (f64) {
    std::memcpy(out, v.data(), sizeof(double) * v.size());
  } else {
    for (size_t k = 0; k < v.size(); ++k) {
      const float f = (float)v[k];
      std::memcpy(out + sizeof(float) * k, &f, sizeof(float));
    }
  }
}

bool cfl_counted(int cfl_mask, const std::vector<uint32_t>& fold_bits, int nx, int i, int j) {
  const size_t o = (size_t)i + (size_t)j * (size_t)nx;
  if (cfl_mask == fv::kCflEven) return (o & 1u) == 0u;
  if (cfl_mask == fv::kCflBitmap) return (fold_bits[o >> 5] >> (o & 31u)) & 1u;
  return true;
}

static long strips_of(const fivonagi_params& p) {
  return (p.nx + fv::kStripCols - 1) / fv::kStripCols;
}

// Lane mask of row j of the strip at x0: bit kHalo + n set when the CFL
// reduction counts the output cell (x0 + n, j), columns 0 and past the grid
// left out.
static uint64_t lane_mask(int cfl_mask, const std::vector<uint32_t>& fold_bits, int nx, int x0,
                          int j) {
  const int n = std::min(fv::kStripCols, nx - x0);
  uint64_t m = ~(uint64_t)0;
  const size_t o = (size_t)x0 + (size_t)j * (size_t)nx;
  if (cfl_mask == fv::kCflEven) {
    m = (o & 1) ? 0xAAAAAAAAAAAAAAAAull : 0x5555555555555555ull;
  } else if (cfl_mask == fv::kCflBitmap) {
    // 64 bits from bit o of the bitmap (words past its end: no cells)
    const size_t w = o >> 5, e = fold_bits.size();
    const unsigned sh = o & 31;
    const uint64_t lo = fold_bits[w] | (uint64_t)(w + 1 < e ? fold_bits[w + 1] : 0) << 32;
    const uint64_t hi = w + 2 < e ? fold_bits[w + 2] : 0;
    m = sh ? lo >> sh | hi << (64 - sh) : lo;
  }
  m &= ((uint64_t)1 << n) - 1;             // n <= 58
  if (x0 == 0) m &= ~(uint64_t)1;
  return m << fv::kHalo;
}

// Rows per item of the in-step cut: the smallest height (never below 12) whose
// total wave count over all instances fits one resident round of the device
// (CUs x resident step waves per CU): every wave then starts at once, and
// taller work items repeat fewer halo rows.
int auto_rows(const std::vector<fivonagi_params>& ps, long target_waves) {
  for (int H = 12; H <= 4096; ++H) {
    long waves = 0;
    for (const auto& p : ps)
      waves += strips_of(p) * std::max(1L, std::lround((double)p.ny / H));
    if (waves <= target_waves) return H;
  }
  return 4096;
}

// Items of a strip of p in the in-step cut.
static int in_step_items(const fivonagi_params& p, int auto_h) {
  const int H = p.rows_per_wave > 0 ? p.rows_per_wave : auto_h;
  return std::max(1, std::min(p.ny, (int)std::lround((double)p.ny / H)));
}

// March steps of the slowest of n waves that share R rows of a strip, one
// above the other: a wave below another marches one step per row of its own,
// at least kSeamRows (its first rows are what it hands down) and 2 mod 3 (the
// march's unrolled rotation, fv_step.hip); the topmost marches past its end,
// about kTail rows' worth.
constexpr double kTail = 3.3;
constexpr int kSeamRows = 5;

std::vector<int> group_heights(int R, int max_waves) {
  const int n = std::max(1, std::min(max_waves, (R - 1) / kSeamRows + 1));
  std::vector<int> h(n);
  int left = R;
  for (int w = 0; w + 1 < n; ++w) {
    const int rest = n - 1 - w;                        // waves above this one
    const double even = (left + kTail) / (rest + 1);
    const int most = left - (rest - 1) * kSeamRows - 1;
    int H = kSeamRows + 3 * std::max(0, (int)std::floor((even - kSeamRows) / 3.0 + 0.5));
    while (H > most) H -= 3;
    h[w] = std::max(kSeamRows, H);
    left -= h[w];
  }
  h[n - 1] = left;
  return h;
}

// Row boundaries of one strip cut into `chunks` work items.  With skew > 0
// the items get `levels` height levels (item j: level (j + rot) % levels)
// with weights falling linearly from 1 + skew to 1 - skew (mean 1), so the
// strip keeps its number of items, some taller and some shorter.  (The in-step
// cut takes rot = 0: the same rows in every strip.)
std::vector<int> chunk_bounds(int ny, int chunks, float skew, int levels, int rot) {
  const int L = std::max(1, std::min(levels, chunks));
  std::vector<double> cum(chunks + 1, 0.0);
  for (int j = 0; j < chunks; ++j) {
    const int level = (j + rot) % L;
    const double w = (L > 1) ? 1.0 + (double)skew * (L - 1 - 2 * level) / (L - 1) : 1.0;
    cum[j + 1] = cum[j] + std::max(w, 0.05);
  }
  std::vector<int> b(chunks + 1);
  for (int j = 0; j <= chunks; ++j) b[j] = (int)std::lround((double)ny * cum[j] / cum[chunks]);
  b[0] = 0;
  b[chunks] = ny;
  // no empty item; the ends stay at 0 and ny (chunks <= ny)
  for (int j = 1; j < chunks; ++j) b[j] = std::max(b[j], b[j - 1] + 1);
  for (int j = chunks - 1; j >= 1; --j) b[j] = std::min(b[j], b[j + 1] - 1);
  return b;
}

// Height skew where every SIMD starts its full complement of waves: evens out
// the ends of four waves of which the oldest issues first (their speeds,
// measured on equal items: 1.09, 0.75, 0.46, 0.32 rows per us).  Step in us at
// skew 0 / 0.5 / 0.65: 4096x1024 38.7 / 36.9 / 37.0, 4096x2048 69.7 / 65.3 /
// 63.1, 8192x4096 263 / 237 / 231, 6000x5001 232 / 234 / 244.
constexpr float kAutoSkew = 0.5f;

// Largest state, in and out, that is cut "running on" (cut A below).  Up to the
// 256 MiB of the memory-side cache the step is bound by its instructions, and
// cut A repeats fewer of them and balances better: 4096x1024 (101 MB) 37.0 us
// against 40.5 for cut B, 4096x2048 (201 MB) 63 against 73.  Beyond it the
// lines at the strips' edges, which two strips read and write, must meet in
// the L2 while both march them, which needs cut B: 4096x4096 (403 MB) 147
// against 134, 8192x4096 (805 MB) 340 against 231.
constexpr long kRunningBytes = 256L << 20;

namespace {

// A row range of one strip.
struct Piece {
  int inst, x0, y0, rows, mrow;
  int waves;                               // that share it
};
// The pieces one workgroup marches.
struct Group {
  int n = 0;
  Piece p[fv::kGroupWaves];
  long rows() const {
    long r = 0;
    for (int j = 0; j < n; ++j) r += p[j].rows;
    return r;
  }
};

// weight of height level l of L: falling linearly from 1 + skew to 1 - skew
double level_weight(int l, int L, float skew) {
  return L > 1 ? std::max(1.0 + (double)skew * (L - 1 - 2 * l) / (L - 1), 0.05) : 1.0;
}

// Cut A, "running on": the strips, laid end to end, are dealt to groups whose
// waves march at most c * (the group's level weight) steps; a group that
// reaches the end of a strip with waves to spare goes on with the next one.
// emit: called with each group (count only: a no-op).  Returns their number.
template <class Emit>
long cut_running(const std::vector<Piece>& strips, double c, float skew, int levels, Emit emit) {
  long n = 0;
  Group cur;
  int left = 0;                            // waves of the current group to spare
  double cl = 0.0;
  auto start = [&]() {
    cl = std::max<double>(kSeamRows, c * level_weight((int)(n % levels), levels, skew));
    left = fv::kGroupWaves;
    cur.n = 0;
  };
  auto flush = [&]() {
    if (cur.n > 0) {
      emit(cur);
      ++n;
    }
    start();
  };
  start();
  for (const auto& s : strips)
    for (int y = 0; y < s.rows;) {
      const int rest = s.rows - y;
      const int need = std::max(1, (int)std::ceil((rest + kTail) / cl - 1e-9));
      Piece p{s.inst, s.x0, s.y0 + y, rest, s.mrow + y, need};
      if (need > left) {
        p.waves = left;
        p.rows = std::min(rest - 1, std::max(1, (int)std::floor(left * cl - kTail + 1e-9)));
      }
      cur.p[cur.n++] = p;
      left -= p.waves;
      y += p.rows;
      if (left == 0) flush();
    }
  flush();
  return n;
}

// Groups sorted tallest first, dealt C at a time to the C CUs of an XCD: the
// first and the last round stay in order (the last may leave the last CUs
// without a group), and in the rounds between the tallest group goes to the CU
// with the fewest rows.
void balance_rounds(std::vector<Group>& run, int C) {
  const int n = (int)run.size(), rounds = (n + C - 1) / C;
  if (rounds < 3) return;
  std::vector<long> load(C, 0);
  for (int j = 0; j < C; ++j) load[j] = run[j].rows();
  for (int g = (rounds - 1) * C; g < n; ++g) load[g % C] += run[g].rows();
  for (int r = 1; r + 1 < rounds; ++r) {
    std::vector<int> place(C);
    for (int j = 0; j < C; ++j) place[j] = j;
    std::stable_sort(place.begin(), place.end(), [&](int u, int v) { return load[u] < load[v]; });
    const std::vector<Group> round(run.begin() + r * C, run.begin() + (r + 1) * C);
    for (int j = 0; j < C; ++j) {
      run[r * C + place[j]] = round[j];
      load[place[j]] += round[j].rows();
    }
  }
}

}  // namespace

void build_work(const std::vector<fivonagi_params>& ps, const std::vector<int>& cfl_mask,
                const std::vector<std::vector<uint32_t>>& fold_bits, long cus, int per_cu,
                int auto_h, float skew, bool rotate, WorkList& out, int cell_bytes) {
  out.items.clear();
  out.rowmask.clear();
  out.group_first.assign(1, 0);
  out.n_items.assign(ps.size(), 0);
  // the strips, with their lane masks
  std::vector<Piece> strips;
  long bytes = 0, waves = 0;               // waves: of the in-step cut
  double rows = 0.0;
  int asked = 0;                           // rows per wave all instances ask for
  bool alike = true;
  for (int k = 0; k < (int)ps.size(); ++k) {
    const auto& p = ps[k];
    waves += strips_of(p) * in_step_items(p, auto_h);
    rows += (double)strips_of(p) * p.ny;
    const int a = std::max(0, p.rows_per_wave);
    if (k == 0) asked = a;
    alike = alike && a == asked;
    bytes += (long)cell_bytes * p.nx * p.ny;
    for (int s = 0; s < (int)strips_of(p); ++s) {
      const int x0 = s * fv::kStripCols;
      strips.push_back({k, x0, 0, p.ny, (int)out.rowmask.size(), 1});
      for (int j = 0; j < p.ny; ++j)
        out.rowmask.push_back(lane_mask(cfl_mask[k], fold_bits[k], p.nx, x0, j));
    }
  }
  // height levels = waves each SIMD starts in the launch's first round
  const long simds = 4 * cus;
  const int per_simd = std::max(1, per_cu / 4);
  const int levels = (int)std::max(1L, std::min<long>(per_simd, (waves + simds - 1) / simds));
  // automatic: skewed only when every SIMD starts its full complement of
  // waves (there the oldest-first issue order staggers their ends; with
  // fewer waves per SIMD they progress together)
  bool running = rotate;
  if (skew < 0.0f) {
    skew = (levels >= 4 && levels == per_simd) ? kAutoSkew : 0.0f;
    running = bytes <= kRunningBytes;
  }
  // cut A marches every strip alike: where instances ask for different rows per
  // wave, cut B gives each its own
  running = running && alike;
  out.skew_used = skew;
  out.rotate_used = rotate && skew > 0.0f;
  std::vector<Group> groups;
  if (running) {
    // the least steps per wave whose groups are all resident at once (to 0.4%).
    // A group holds four strips at most, so with very many strips no height
    // makes them fit: then the least whose groups take as few rounds of
    // residency as whole strips, one to a wave, do (from `whole` steps on even
    // the lowest level holds any strip in one wave)
    auto groups_at = [&](double c) {
      return cut_running(strips, c, skew, levels, [](const Group&) {});
    };
    int tallest = 0;
    for (const auto& s : strips) tallest = std::max(tallest, s.rows);
    const double whole = (tallest + kTail) / level_weight(levels - 1, levels, skew);
    const long room = std::max(1L, cus * per_simd);
    const long target = room * ((groups_at(whole) + room - 1) / room);
    auto fits = [&](double c) { return c >= whole || groups_at(c) <= target; };
    double c = kSeamRows;
    if (asked > 0) {
      c = std::max(kSeamRows, asked);
    } else if (!fits(c)) {
      double lo = std::max(c, rows / (double)(target * fv::kGroupWaves)), hi = 1.05 * lo;
      while (!fits(hi)) { lo = hi; hi = std::min(1.25 * hi, whole); }
      while (hi - lo > 0.004 * lo) {
        const double mid = 0.5 * (lo + hi);
        if (fits(mid)) hi = mid;
        else lo = mid;
      }
      c = hi;
    }
    cut_running(strips, c, skew, levels, [&](const Group& g) { groups.push_back(g); });
  } else {
    // Cut B, "in step": each strip into the same number of one-wave items, cut
    // at the same rows in every strip of an instance
    std::vector<Piece> items;
    for (const auto& s : strips) {
      const int chunks = in_step_items(ps[s.inst], auto_h);
      const std::vector<int> b = chunk_bounds(s.rows, chunks, skew, levels, 0);
      for (int j = 0; j < chunks; ++j)
        items.push_back({s.inst, s.x0, b[j], b[j + 1] - b[j], s.mrow + b[j], 1});
    }
    // each XCD's run tallest first (see below), four to a workgroup; equal
    // heights by rows, so that a workgroup's waves are neighbouring strips
    const int n = (int)items.size(), W = fv::kGroupWaves;
    const int wgs = (n + W - 1) / W, q = wgs >> 3, rem = wgs & 7;
    for (int x = 0; x < 8; ++x) {
      const int b = std::min(n, W * (x * q + std::min(x, rem)));
      const int e = std::min(n, b + W * (q + (x < rem ? 1 : 0)));
      std::stable_sort(items.begin() + b, items.begin() + e, [](const Piece& u, const Piece& v) {
        if (u.rows != v.rows) return u.rows > v.rows;
        return u.inst != v.inst ? u.inst < v.inst : u.y0 < v.y0;
      });
      std::vector<Group> run;
      for (int i = b; i < e; i += W) {
        Group g;
        while (g.n < W && i + g.n < e) { g.p[g.n] = items[i + g.n]; ++g.n; }
        run.push_back(g);
      }
      balance_rounds(run, (int)std::max(1L, cus / 8));
      groups.insert(groups.end(), run.begin(), run.end());
    }
  }
  // Launch order.  Workgroup b of a launch runs on XCD b % 8 and takes group
  // x*q + min(x, rem) + (b >> 3) (fv_step_kernel), so XCD x works through the
  // run of groups [x*q + min(x, rem), ...) in order, and within a run the
  // hardware starts groups in that order, one per CU, then the next round of
  // CU slots.  A SIMD issues for its oldest wave first, so the rounds take the
  // levels in turn, tallest first: the waves that start first get the most
  // rows, and a SIMD's waves finish together instead of leaving one wave alone
  // at the end.  Cut A: CU c of an XCD takes groups L c .. L c + L - 1 of the
  // run (neighbouring rows, equal sums); cut B was sorted above.
  std::vector<int> order(groups.size());
  {
    const int n = (int)groups.size(), q = n >> 3, rem = n & 7;
    for (int x = 0; x < 8; ++x) {
      const int b = x * q + std::min(x, rem), e = b + q + (x < rem ? 1 : 0);
      int at = b;
      const int L = running ? levels : 1;
      // the level pattern starts anew every L groups of the whole list
      for (int l = 0; l < L; ++l)
        for (int g = b; g < e; ++g)
          if (g % L == l) order[at++] = g;
    }
  }
  for (int g : order) {
    int used = 0;
    for (int j = 0; j < groups[g].n; ++j) {
      const Piece& pc = groups[g].p[j];
      const std::vector<int> h = group_heights(pc.rows, pc.waves);
      int y = pc.y0;
      for (size_t w = 0; w < h.size(); ++w) {
        fv::WorkItem it;
        it.inst = pc.inst;
        it.x0 = pc.x0;
        it.y0 = y;
        it.y1 = y + h[w];
        it.mrow = pc.mrow + (y - pc.y0);
        it.local = out.n_items[pc.inst]++;
        it.bc = ps[pc.inst].bc;
        it.role = used++ | (w + 1 < h.size() ? fv::kRoleAbove : 0);
        out.items.push_back(it);
        y = it.y1;
      }
    }
    out.group_first.push_back((int32_t)out.items.size());
  }
}

std::vector<fv::WorkItem> launch_items(const WorkList& wl, long cus) {
  fv::WorkItem none;
  std::memset(&none, 0, sizeof(none));
  const int n = (int)wl.group_first.size() - 1, W = fv::kGroupWaves;
  std::vector<fv::WorkItem> v((size_t)n * W, none);
  // the waves of a workgroup go to its CU's SIMDs in turn, and an XCD's
  // groups to its CUs in turn: each group's tallest wave takes the place of
  // the SIMD with the least steps so far
  const int C = (int)std::max(1L, cus / 8), q = n >> 3, rem = n & 7;
  for (int x = 0; x < 8; ++x) {
    const int b = x * q + std::min(x, rem), e = b + q + (x < rem ? 1 : 0);
    std::vector<double> load((size_t)C * W, 0.0);
    for (int g = b; g < e; ++g) {
      double* ld = &load[(size_t)((g - b) % C) * W];
      std::pair<double, int> waves[fv::kGroupWaves];
      int place[fv::kGroupWaves], m = 0;
      for (int i = wl.group_first[g]; i < wl.group_first[g + 1]; ++i)
        waves[m++] = {wl.items[i].y1 - wl.items[i].y0 +
                          (wl.items[i].role & fv::kRoleAbove ? 0.0 : kTail), -i};
      std::sort(waves, waves + m, [](const auto& u, const auto& w) { return u > w; });
      for (int j = 0; j < W; ++j) place[j] = j;
      std::sort(place, place + W, [&](int u, int w) {
        return ld[u] != ld[w] ? ld[u] < ld[w] : u < w;
      });
      for (int j = 0; j < m; ++j) {
        v[(size_t)g * W + place[j]] = wl.items[-waves[j].second];
        ld[place[j]] += waves[j].first;
      }
    }
  }
  return v;
}

void build_adj_items(const std::vector<fivonagi_params>& ps, long target_waves,
                     int rows_per_wave, std::vector<fv::AdjItem>& items,
                     std::vector<size_t>& first, std::vector<int32_t>& wave_first) {
  constexpr int kCols = 56;   // output columns per strip (a 4-column halo each side)
  // strip starts; the last one never falls on nx-2 or nx-1 (column nx-3's
  // wave also holds nx-2 and nx-1)
  auto strips = [&](int nx) {
    std::vector<int> b;
    for (int x = 0; x < nx; x += kCols) b.push_back(x);
    if (b.size() >= 2 && nx - b.back() <= 2) b.back() = nx - 3;
    b.push_back(nx);
    return b;
  };
  // a row cut never leaves row 2 apart from rows 0, 1, nor row ny-3 apart
  // from ny-2, ny-1 (a ghost copy and its source in one item)
  auto legal_cut = [](int cut, int ny) {
    if (cut == 1 || cut == 2) return 3;
    if (cut == ny - 2 || cut == ny - 1) return ny;
    return cut;
  };
  items.clear();
  wave_first.assign(1, 0);
  first.assign(ps.size() + 1, 0);
  if (rows_per_wave > 0) {
    // fixed heights: rows_per_wave rows per item, one item per wave
    const int H = std::max(8, rows_per_wave);
    for (size_t k = 0; k < ps.size(); ++k) {
      const auto& p = ps[k];
      const std::vector<int> sb = strips(p.nx);
      first[k] = items.size();
      for (size_t s = 0; s + 1 < sb.size(); ++s)
        for (int y = 0; y < p.ny;) {
          const int y1 = std::min(p.ny, legal_cut(std::min(p.ny, y + H), p.ny));
          items.push_back({(int32_t)k, sb[s], sb[s], sb[s + 1], y, y1});
          wave_first.push_back((int32_t)items.size());
          y = y1;
        }
    }
    first[ps.size()] = items.size();
    return;
  }
  // balanced: the strips of every instance, one after another, are cut into
  // waves of about equal cost, an item costing its rows plus kWarm for the
  // rows the march starts with before the first it emits; a wave may end one
  // strip and start the next (two items).  The least cost per wave whose
  // waves fit target_waves is found by bisection.
  constexpr int kWarm = 4, kMinRows = 8;
  auto pack = [&](long T, bool emit) {
    long waves = 0, left = 0;
    for (size_t k = 0; k < ps.size(); ++k) {
      const auto& p = ps[k];
      const std::vector<int> sb = strips(p.nx);
      if (emit) first[k] = items.size();
      for (size_t s = 0; s + 1 < sb.size(); ++s)
        for (int y = 0; y < p.ny;) {
          if (left - kWarm < kMinRows) {       // start a wave
            if (emit && waves > 0) wave_first.push_back((int32_t)items.size());
            ++waves;
            left = T;
          }
          const long take = std::min<long>(p.ny - y, left - kWarm);
          const int y1 = std::min(p.ny, legal_cut(y + (int)take, p.ny));
          if (emit) items.push_back({(int32_t)k, sb[s], sb[s], sb[s + 1], y, y1});
          left -= (y1 - y) + kWarm;
          y = y1;
        }
    }
    if (emit) {
      first[ps.size()] = items.size();
      wave_first.push_back((int32_t)items.size());
    }
    return waves;
  };
  long total = 0;
  for (const auto& p : ps) total += (long)(strips(p.nx).size() - 1) * (p.ny + kWarm);
  long lo = kWarm + kMinRows, hi = std::max(lo, total + kWarm + kMinRows);
  const long target = std::max(1L, target_waves);
  while (lo < hi) {                          // the least T with pack(T) <= target
    const long mid = lo + (hi - lo) / 2;
    if (pack(mid, false) <= target) hi = mid;
    else lo = mid + 1;
  }
  pack(lo, true);
}

}  // namespace fvh
