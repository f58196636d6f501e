// extern "C" entry points of libdmuon_amd.so (declared in include/dmuon_amd.h): argument
// validation, workspace planning and the launch sequence of one Muon group step.
#include <math.h>
#include <stdarg.h>
#include <stdio.h>

#include <mutex>
#include <string>
#include <utility>
#include <vector>

#include "../../include/dmuon_amd.h"
#include "dmuon_amd_internal.h"

using namespace dmuon;

// Scratch of dmuon_muon_step_group_noalloc: one static device array, of which the loader gives
// every GPU its own copy, held until the process ends. This file holds no kernels, so its code
// object -- the array with it -- is loaded onto a GPU by the first hipGetSymbolAddress there,
// not by the kernels of the other entry points. Host code never uses the array's name as an
// address (on the host it is a stand-in symbol): the device address of the current GPU's copy
// comes from hipGetSymbolAddress on the first call on that GPU and is kept per device
// (scratch_of_current_device).
static __device__ __align__(256) char scratch[DMUON_NOALLOC_SCRATCH_BYTES];

namespace {

thread_local std::string g_last_error;

int fail(const char* fmt, ...) __attribute__((format(printf, 1, 2)));
int fail(const char* fmt, ...) {
  char buf[512];
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(buf, sizeof(buf), fmt, ap);
  va_end(ap);
  g_last_error = buf;
  return 1;
}

int check_launch(hipError_t e, const char* what) {
  if (e != hipSuccess) return fail("%s: launch failed: %s", what, hipGetErrorString(e));
  return 0;
}

bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }
bool ld_ok(int64_t ld) { return ld > 0 && (ld % 8) == 0; }
bool stride_ok(int64_t s, int batch) { return batch <= 1 || (s >= 0 && (s % 8) == 0); }

int64_t round_up(int64_t x, int64_t m) { return (x + m - 1) / m * m; }
int64_t align256(int64_t b) { return round_up(b, 256); }

// Diagonal-tile work skipped by the exactly symmetric products (NtArgs::diag_skip): the
// m x m polynomials (K = m) skip every 16x16 block below the diagonal, the products X X^T
// (K = n, up to 14336) none. Measured on the c5 step, same box, against no skipping anywhere:
// polynomial class -3.1 ms (-2%); for X X^T skipping only the two idle waves cost +0.7 ms and
// skipping blocks +1.6 ms (a diagonal tile that finishes early takes its CU out of step with
// the tiles that share its operand panels in L2).
constexpr int kDiagSkipPoly = DIAG_SKIP_BLOCKS;
constexpr int kDiagSkipGram = DIAG_SKIP_NONE;

// The products X' = P X (direct) and Q X (Gram) read X itself as their k-major B operand
// (transposing LDS reads) instead of a transposed copy: the staging writes one fp16 copy of
// ns_in (12 B per element, not 14), and X ping-pongs between two buffers (such a product reads
// the current X across the whole K range, so the new X cannot overwrite it). The k-major loads
// address a matrix's whole X through one 32-bit buffer range, so m_pad * n_pad * 2 < 2^31
// bytes: 2^30 fp16 values per padded matrix, which plan() enforces.
constexpr int64_t kMaxXBytes = int64_t(1) << 31;

// Power-of-two scale of the fp16 NS operand X, both backends (entries of the normalised X are at
// most 1; the scale keeps the typical ~1/sqrt(mn) entries out of the fp16 subnormal range)
constexpr float kNsKx = 4096.f;

struct Workspace {
  uint16_t *X, *X2, *Am, *Pm;
  // Gram backend only: the two slots of the accumulated polynomial Q (or its transpose), P R
  uint16_t *Q0, *Q1, *Wm;
  float *partials, *scale, *est_old;
  // correction of a copy staged with an estimated scale (1 when staged exactly), and the
  // per-matrix "stage again" flags
  float *ratio, *ratio_sq;
  int* restage;
  int nparts;
  int64_t bytes;
};

// Carves the workspace of a group; base == nullptr only computes the size.
Workspace carve(char* base, int m_pad, int n_pad, int Rp, int Cp, int batch, int gram) {
  Workspace w{};
  int64_t off = 0;
  auto take = [&](int64_t bytes) {
    char* p = base ? base + off : nullptr;
    off += align256(bytes);
    return p;
  };
  const int64_t L = batch;
  const int64_t xs = (int64_t)m_pad * n_pad * 2;
  const int64_t as = (int64_t)m_pad * m_pad * 2;
  // X and the second X buffer the NS products write the next X into, both backends; Gram adds
  // the two Q slots and P R
  w.X = reinterpret_cast<uint16_t*>(take(L * xs));
  w.X2 = reinterpret_cast<uint16_t*>(take(L * xs));
  w.Am = reinterpret_cast<uint16_t*>(take(L * as));
  w.Pm = reinterpret_cast<uint16_t*>(take(L * as));
  if (gram) {
    w.Q0 = reinterpret_cast<uint16_t*>(take(L * as));
    w.Q1 = reinterpret_cast<uint16_t*>(take(L * as));
    w.Wm = reinterpret_cast<uint16_t*>(take(L * as));
  }
  w.nparts = pre_blocks_per_mat(Rp, Cp);
  w.partials = reinterpret_cast<float*>(take(L * w.nparts * 4));
  w.scale = reinterpret_cast<float*>(take(L * 4));
  w.est_old = reinterpret_cast<float*>(take(L * 4));
  w.ratio = reinterpret_cast<float*>(take(L * 4));
  w.ratio_sq = reinterpret_cast<float*>(take(L * 4));
  w.restage = reinterpret_cast<int*>(take(L * 4));
  w.bytes = off;
  return w;
}

// ---- launch profiler: optional hipEvent pairs around every kernel of run_group ----------------
// Single-threaded use only (like the launch path itself). Events are host objects; no device
// memory is allocated.
enum ProfClass {
  PC_PRE = 0, PC_NORM, PC_SYRK, PC_POLY, PC_GEMM, PC_FINAL, PC_ADAMW, PC_CLIP, PC_COUNT
};
struct ProfRec {
  int cls;
  hipEvent_t a, b;
  double flops, bytes;
};
struct Profiler {
  bool on = false;
  std::vector<hipEvent_t> pool;
  std::vector<ProfRec> recs;
  hipEvent_t take() {
    if (!pool.empty()) {
      hipEvent_t e = pool.back();
      pool.pop_back();
      return e;
    }
    hipEvent_t e = nullptr;
    if (hipEventCreate(&e) != hipSuccess) return nullptr;
    return e;
  }
};
Profiler g_prof;
// set while an entry point that must not allocate runs: the profiler records no events then
thread_local bool g_no_events = false;

template <class F>
int timed(int cls, double flops, double bytes, hipStream_t stream, const char* who, F&& launch) {
  if (!g_prof.on || g_no_events) return check_launch(launch(), who);
  hipEvent_t a = g_prof.take(), b = g_prof.take();
  if (!a || !b) return fail("%s: hipEventCreate failed", who);
  if (hipEventRecord(a, stream) != hipSuccess) return fail("%s: hipEventRecord failed", who);
  const int rc = check_launch(launch(), who);
  if (hipEventRecord(b, stream) != hipSuccess) return fail("%s: hipEventRecord failed", who);
  g_prof.recs.push_back({cls, a, b, flops, bytes});
  return rc;
}

int tri_tiles(int m_pad, int tile) {
  const int mt = m_pad / tile;
  return mt * (mt + 1) / 2;
}

// Output tile of a group's products, by the estimated time of its triangle products (the bulk
// of the work) in units of one 256-tile of work: a wave of 256-tiles gives every CU one tile (4
// units of 128-tile work), a wave of 128-tiles gives it two (2 units) at about 1/1.35 of the
// 256-tile rate (fitted to grouped Gram runs: 32 x 4096^2, 64 x 1024x4096, 64 and 128 x
// 1408x2048, one 2048x8192). Ceil'd waves charge the last, partial wave in full; the padding
// each tile size adds to m and n counts too. Measured on MI355X: one 4096^2 matrix runs 20%
// faster on 256-tiles (136 tiles on 256 CUs) than on 128-tiles (528 tiles on 512 slots), one
// 1024x16384 or 2048x8192 matrix 25-55% faster on 128-tiles, 128 experts of 1408x2048 5% faster
// on 256-tiles padded to 1536.
int auto_tile(int64_t m, int64_t n, int64_t batch, int num_cus) {
  const int64_t m256 = round_up(m, 256) / 256, m128 = round_up(m, 128) / 128;
  const int64_t t256 = batch * m256 * (m256 + 1) / 2, t128 = batch * m128 * (m128 + 1) / 2;
  const double npad = (double)round_up(n, 256) / (double)round_up(n, 128);
  const double c256 = 4.0 * (double)((t256 + num_cus - 1) / num_cus) * npad;
  const double c128 = 2.7 * (double)((t128 + 2 * num_cus - 1) / (2 * num_cus));
  return c256 <= c128 ? 256 : 128;
}

int plan(int rows, int cols, int batch, int tile_req, int num_cus, int gram, int* tile,
         int* m_pad, int* n_pad, int64_t* bytes) {
  if (rows <= 0 || cols <= 0 || batch <= 0)
    return fail("dmuon_ns_plan: rows, cols and batch must be positive (got %d, %d, %d)", rows,
                cols, batch);
  if (tile_req != 0 && tile_req != 128 && tile_req != 256)
    return fail("dmuon_ns_plan: tile must be 0 (auto), 128 or 256, got %d", tile_req);
  const int m = rows < cols ? rows : cols;
  const int n = rows < cols ? cols : rows;
  if (num_cus <= 0) num_cus = 256;
  int t = tile_req;
  if (t == 0) t = auto_tile(m, n, batch, num_cus);
  const int mp = (int)round_up(m, t), np = (int)round_up(n, t);
  if ((int64_t)mp * np * 2 >= kMaxXBytes)
    return fail("dmuon_ns_plan: a %d x %d matrix pads to %d x %d, %lld fp16 values; the NS "
                "kernels take at most 2^30 per matrix", rows, cols, mp, np, (long long)mp * np);
  const bool tall = rows > cols;
  const int Rp = tall ? np : mp, Cp = tall ? mp : np;
  Workspace w = carve(nullptr, mp, np, Rp, Cp, batch, gram);
  *tile = t;
  *m_pad = mp;
  *n_pad = np;
  *bytes = w.bytes;
  return 0;
}

// Estimated time (us) of the Newton-Schulz products of a call's groups on `tile`-tiles: each
// product is one launch over all of them, whose time is that of its longest tile or of its
// work spread over the machine, whichever is more, plus 2 us from launch to launch. A tile's time
// is fixed + slices of K (64 wide) at its kernel's rate, measured on MI355X as K sweeps (64 ..
// 8192) of triangle products with 36 .. 1020 tiles: 256-tiles 13 us + 1.0 per slice on a third of
// the CUs and 1.4 on all of them, 128-tiles one per CU 6 + 0.39 .. 0.46, two per CU 8 + 0.93 for
// the pair, 64-tiles 5 + 0.18 (two of them per CU take 1 .. 2 us less than the 128-tiles one per CU
// that stand for them here). Only the comparison of two splits matters. That one of the Q updates may
// run in the CUs the triangle launches leave idle (nt_fill_pays, up to four groups) is left out: with
// it counted, 59 of 400 random sets of 2 .. 9 shapes were split another way, and forty of those ran 0.7%
// slower in the mean (0.93 .. 1.15 of the time), the estimate's other errors being larger.
double groups_cost_us(const dmuon_muon_group* g, int n, int tile, int num_cus, bool gram) {
  // launches of one NS run of five steps: X X^T, m x m triangle products, Q updates, P X
  const double n_xx = gram ? 2 : 5, n_tri = gram ? 11 : 5, n_full = gram ? 3 : 0,
               n_px = gram ? 2 : 5;
  auto launch = [&](auto&& dims) {   // dims(group, tile): (tiles of one matrix, K)
    auto total = [&](int t) {
      double tiles = 0;
      for (int i = 0; i < n; ++i) tiles += dims(g[i], t).first * g[i].batch;
      return tiles;
    };
    int t = tile;
    double fixed = 13.0, slice = 0, slots = num_cus;
    auto busy = [&](double tiles) { return tiles < num_cus ? tiles / num_cus : 1.0; };
    if (tile == 256) slice = 0.85 + 0.55 * busy(total(256));
    else if (total(64) <= num_cus) t = 64, fixed = 5.0, slice = 0.18;
    else if (total(128) <= num_cus) fixed = 6.0, slice = 0.35 + 0.11 * busy(total(128));
    else fixed = 8.0, slice = 0.93, slots = 2.0 * num_cus;
    double longest = 0, sum = 0;
    for (int i = 0; i < n; ++i) {
      const std::pair<double, double> d = dims(g[i], t);
      const double us = fixed + slice * ceil(d.second / 64.0);
      longest = us > longest ? us : longest;
      sum += us * d.first * g[i].batch;
    }
    // a last wave that is partly empty: half a tile on average
    const double spread = sum / slots + (total(t) > slots ? 0.5 * longest : 0.0);
    return (spread > longest ? spread : longest) + 2.0;
  };
  // tiles along m and n: of the padded sides, 64-tiles of the sides rounded up to 64
  auto sides = [](const dmuon_muon_group& q, int t) {
    const int64_t m = q.rows < q.cols ? q.rows : q.cols, w = q.rows < q.cols ? q.cols : q.rows;
    return std::pair<double, double>((double)((m + t - 1) / t), (double)((w + t - 1) / t));
  };
  auto m_of = [](const dmuon_muon_group& q) { return (double)(q.rows < q.cols ? q.rows : q.cols); };
  auto n_of = [](const dmuon_muon_group& q) { return (double)(q.rows < q.cols ? q.cols : q.rows); };
  typedef std::pair<double, double> dims_t;
  const double tri_m = launch([&](const dmuon_muon_group& q, int t) {
    const double s = sides(q, t).first;
    return dims_t(s * (s + 1) / 2, m_of(q));
  });
  const double tri_n = launch([&](const dmuon_muon_group& q, int t) {
    const double s = sides(q, t).first;
    return dims_t(s * (s + 1) / 2, n_of(q));
  });
  const double full = launch([&](const dmuon_muon_group& q, int t) {
    const double s = sides(q, t).first;
    return dims_t(s * s, m_of(q));
  });
  const double px = launch([&](const dmuon_muon_group& q, int t) {
    const std::pair<double, double> s = sides(q, t);
    return dims_t(s.first * s.second, m_of(q));
  });
  bool small = gram && tile == kGramSmallSide;     // run_gram's one-workgroup form
  double matrices = 0;
  for (int i = 0; i < n; ++i) {
    small = small && m_of(g[i]) <= kGramSmallSide;
    matrices += g[i].batch;
  }
  const double squares = small ? 2 * (4.0 + 13.0 * ceil(matrices / num_cus))
                               : n_tri * tri_m + n_full * full;
  return n_xx * tri_n + squares + n_px * px;
}

// Tile, workspace and estimated time of several groups in one call. One group takes the tile
// plan() gives it; several the tile whose estimate is lower (either gives every matrix the same
// bits).
int plan_groups(const dmuon_muon_group* g, int n, int tile_req, int num_cus, int gram, int* tile,
                int64_t* bytes, double* cost_us) {
  if (num_cus <= 0) num_cus = 256;
  int t = tile_req, mp, np;
  int64_t total = 0, one;
  if (t == 0 && n > 1)
    t = groups_cost_us(g, n, 256, num_cus, gram) <= groups_cost_us(g, n, 128, num_cus, gram)
            ? 256 : 128;
  for (int i = 0; i < n; ++i) {
    if (plan(g[i].rows, g[i].cols, g[i].batch, t, num_cus, gram, tile, &mp, &np, &one)) return 1;
    total += one;
  }
  *bytes = total;
  if (cost_us) *cost_us = groups_cost_us(g, n, *tile, num_cus, gram);
  return 0;
}

// One group of a call: `batch` matrices of one oriented shape, their tables, workspace and the
// state of their Newton-Schulz iteration.
struct Group {
  void* const* g_ptrs; int g_dtype;
  float* const* buf_ptrs;
  float* const* est_ptrs;
  void* const* w_ptrs; int w_dtype;
  void* const* pub_ptrs; int pub_dtype;
  void* const* out_ptrs; int out_dtype;
  int rows, cols, batch, n_t, first_step;
  float lrs;
  // derived (group_setup)
  int m, n, m_pad, n_pad, km, kn, n_flip;
  bool tall;
  long long xs, as;
  Workspace w;
  // NS: the current X and the buffer the next one is written to, whether it is still the staged
  // one, the scale of the stored R (or A), the Q slots and the row form of a slot's Q
  uint16_t *x_cur, *x_nxt;
  bool x_staged;
  float rs;
  uint16_t* qslot[2];
  uint16_t* qbuf[2];
};

// What one call runs: up to kMaxGroups groups of different shapes, each product of the iteration
// one launch over all of them. The groups share the tile size, the coefficients and the restarts;
// a matrix's bits depend on none of the others.
struct Call {
  Group* g;
  int n, tile;
  hipStream_t stream;
  const char* who;
};

double syrk_flops(const Group& g) { return (double)g.batch * g.m * (g.m + 1.0) * g.n; }
double poly_flops(const Group& g) { return (double)g.batch * g.m * (g.m + 1.0) * g.m; }
double gemm_flops(const Group& g) { return 2.0 * g.batch * (double)g.m * g.m * g.n; }
double square_flops(const Group& g) { return 2.0 * g.batch * (double)g.m * g.m * g.m; }
double update_bytes(const Group& g) {
  const double elems = (double)g.rows * g.cols * g.batch;
  auto width = [](int dtype) { return dtype == DMUON_DTYPE_F32 ? 4.0 : 2.0; };
  return elems * ((g.w_ptrs ? 2.0 * width(g.w_dtype) : 0.0) +
                  (g.out_ptrs ? width(g.out_dtype) : 0.0) +
                  (g.pub_ptrs ? width(g.pub_dtype) : 0.0));
}

// The args of one product for each group of a call: fill(group, args) sets a group's operands.
template <class Fill>
void product_args(const Call& c, NtArgs* a, Fill&& fill) {
  for (int i = 0; i < c.n; ++i) {
    NtArgs& s = a[i];
    s = NtArgs{};
    s.elt = ELT_F16;
    s.L = c.g[i].batch;
    fill(c.g[i], s);
    s.mt = s.M / c.tile;
    s.nt = s.N / c.tile;
    s.tiles_per_mat = s.tri ? tri_tiles(s.M, c.tile) : s.mt * s.nt;
  }
}

// One product of the iteration over the groups of a call, work(group) its useful FLOPs; with
// `more`, tiles of that product too (launch_nt_fill).
template <class Fill>
int nt_product(const Call& c, int cls, double (*work)(const Group&), Fill&& fill,
               NtFill* more = nullptr, bool all = false) {
  NtArgs a[kMaxGroups];
  product_args(c, a, fill);
  double flops = 0.0, bytes = 0.0;
  for (int i = 0; i < c.n; ++i) {
    flops += work(c.g[i]) + (more && all ? square_flops(c.g[i]) : 0.0);
    if (cls == PC_FINAL) bytes += update_bytes(c.g[i]);
  }
  return timed(cls, flops, bytes, c.stream, c.who,
               [&] { return launch_nt_fill(a, c.n, more, all, c.tile, c.stream); });
}

// K loop lengths: the operands are zero past m (n), so the products multiply only m (n) rounded
// up to the 64-wide slice (km, kn), not the tile-padded m_pad (n_pad); rows and columns past
// that are never read, which live_rows / live_cols state.
void square_operands(const Group& g, NtArgs& s, const uint16_t* A, const uint16_t* B,
                     const uint16_t* C) {
  s.A = A; s.B = B; s.C = C;
  s.lda = s.ldb = s.ldc = s.ldd = s.lddt = g.m_pad;
  s.sA = s.sB = s.sC = s.sD = s.sDT = g.as;
  s.M = s.N = s.K = g.m_pad;
  s.k_loop = g.km;
  s.live_rows = s.live_cols = g.km < g.m_pad ? g.km : 0;
}

// D = alpha * A B^T + beta * C + diag * I, m x m, upper tiles mirrored (a symmetric result), and
// optionally D2 = D + diag2 * I
void symmetric_square(const Group& g, NtArgs& s, const uint16_t* A, const uint16_t* B,
                      const uint16_t* C, uint16_t* D, float alpha, float beta, float diag,
                      uint16_t* D2 = nullptr, float diag2 = 0.f) {
  square_operands(g, s, A, B, C);
  s.tri = 1; s.sym_exact = 1; s.diag_skip = kDiagSkipPoly;
  s.mode = EPI_SYM; s.alpha = alpha; s.beta = beta; s.diag = diag;
  s.c_in = C == A ? C_IS_A : C_NONE;   // C's tile is the A panel's last slices
  s.D = D; s.D2 = D2; s.diag2 = diag2;
}

// R = alpha X X^T. The staged X may carry an estimated scale: the first products that read it
// multiply by the per-matrix correction (ratio for X, ratio_sq for X X^T; 1 after an exact
// staging). Later X are exactly scaled.
void gram_of_x(const Group& g, NtArgs& s, uint16_t* R, float alpha) {
  s.alpha_dev = g.x_staged ? g.w.ratio_sq : nullptr;
  s.A = s.B = g.x_cur;
  s.lda = s.ldb = g.n_pad;
  s.sA = s.sB = g.xs;
  s.M = s.N = g.m_pad; s.K = g.n_pad; s.k_loop = g.kn;
  s.live_rows = s.live_cols = g.km < g.m_pad ? g.km : 0;
  s.tri = 1; s.sym_exact = 1; s.diag_skip = kDiagSkipGram;
  s.mode = EPI_SYM; s.alpha = alpha;
  s.D = R; s.ldd = g.m_pad; s.sD = g.as;
}

// X' = P X + beta X into the other X buffer (X is the k-major B operand, read across the whole K
// range, so the new X goes elsewhere)
void px_next(const Group& g, NtArgs& s, const uint16_t* P, float beta) {
  s.alpha_dev = g.x_staged ? g.w.ratio : nullptr;
  s.A = P; s.lda = g.m_pad; s.sA = g.as;
  s.B = g.x_cur; s.ldb = g.n_pad; s.sB = g.xs; s.b_kmajor = 1;
  s.M = g.m_pad; s.N = g.n_pad; s.K = g.m_pad; s.k_loop = g.km;
  s.live_rows = g.km < g.m_pad ? g.km : 0;
  s.live_cols = g.kn < g.n_pad ? g.kn : 0;
  s.alpha = 1.f; s.beta = beta;
  s.mode = EPI_NS;
  s.D = g.x_nxt; s.ldd = g.n_pad; s.sD = g.xs;
}
void x_advance(Call& c) {
  for (int i = 0; i < c.n; ++i) {
    std::swap(c.g[i].x_cur, c.g[i].x_nxt);
    c.g[i].x_staged = false;
  }
}

// the last product: U = (P X + beta X) / KX with the Muon update in the epilogue
void px_final(const Group& g, NtArgs& s, const uint16_t* P, float beta, float decay) {
  px_next(g, s, P, beta);
  s.alpha = 1.f / kNsKx;
  s.mode = EPI_FINAL;
  s.D = nullptr;
  s.out_ptrs = g.out_ptrs; s.out_dtype = g.out_dtype;
  s.w_ptrs = g.w_ptrs; s.w_dtype = g.w_dtype; s.decay = decay; s.lrs = g.lrs;
  s.pub_ptrs = g.pub_ptrs; s.pub_dtype = g.pub_dtype;
  s.m_real = g.m; s.n_real = g.n; s.transposed = g.tall ? 1 : 0; s.n_flip = g.n_flip;
}

// Direct NS on the same fp16 operands as the Gram form: X carries the power-of-two scale kNsKx
// throughout; the first A (eigenvalues ~1/m) carries kr until its polynomial.
int run_direct(Call& c, const float* coeffs, int T, float decay) {
  for (int it = 0; it < T; ++it) {
    const float ca = coeffs[3 * it], cb = coeffs[3 * it + 1], cc = coeffs[3 * it + 2];
    if (it > 0)
      for (int i = 0; i < c.n; ++i) c.g[i].rs = 1.f;
    // A = rs * X X^T of the normalised X (the stored X is kNsKx * X)
    if (nt_product(c, PC_SYRK, syrk_flops, [&](Group& g, NtArgs& s) {
          gram_of_x(g, s, g.w.Am, g.rs / (kNsKx * kNsKx));
        }))
      return 1;
    // P = c A A^T + b A
    if (nt_product(c, PC_POLY, poly_flops, [&](Group& g, NtArgs& s) {
          symmetric_square(g, s, g.w.Am, g.w.Am, g.w.Am, g.w.Pm, cc / (g.rs * g.rs), cb / g.rs,
                           0.f);
        }))
      return 1;
    // X' = P X + a X; the final step writes U = X' / kNsKx
    if (nt_product(c, it + 1 < T ? PC_GEMM : PC_FINAL, gemm_flops, [&](Group& g, NtArgs& s) {
          if (it + 1 < T) px_next(g, s, g.w.Pm, ca);
          else px_final(g, s, g.w.Pm, ca, decay);
          s.C = g.x_cur; s.ldc = g.n_pad; s.sC = g.xs;
        }))
      return 1;
    x_advance(c);
  }
  return 0;
}

// Gram-space NS (the reference's gram_newton_schulz, newton_schulz.py:333-448) on the fp16 NT
// kernels, for X (m x n, m <= n) staged as fp16(KX * ns_in / ||ns_in||). With R = X X^T and
// Z_i = c_i R^2 + b_i R, one NS step maps X to P_i X, P_i = Z_i + a_i I, so per step
//   Q <- P_i Q  (Q = P_i after a start or restart), the accumulated polynomial: Z Q^T + a Q
//   R <- P_i R P_i  when the next step is neither the last nor a restart:
//        W = Z R + a R, R = W Z + a W
//   restart at step i: X <- Q X, R = X X^T, Q reset;   finally U = Q X / KX
// Every symmetric product (R, Z, W, a fresh Q) is computed on the upper-triangle tiles and
// stored exactly symmetric (diagonal tiles included), so R R^T = R R and Z R^T = Z R hold to the
// bit; an R that is symmetric only to rounding costs up to 10x accuracy in fp16 emulation. Q's
// update is a full product: Q is a product of polynomials that no longer commute once rounded,
// and symmetrising it costs 3-8x accuracy on square matrices. fp16 as in the reference (bf16
// loses the small eigenvalues of R). Power-of-two scales keep every operand normal in fp16:
// X carries KX = 2^12 throughout, the first R (eigenvalues ~1/m) carries kr = 2^floor(log2 m)
// (at most 2^12) until its first update; all scale changes are folded into alpha / beta.
int run_gram(Call& c, const float* coeffs, int T, const int* restarts, int n_restarts,
             float decay) {
  auto is_restart = [&](int it) {
    for (int r = 0; r < n_restarts; ++r)
      if (restarts[r] == it) return true;
    return false;
  };
  // Q <- P Q = Z Q + a Q as a full product (Q is a product of polynomials that no longer
  // commute once rounded; its factor order must match R's). Z is symmetric, so the update runs
  // transposed, Q^T <- Q^T Z + a Q^T: Q^T is its A operand and its addend (the K loop takes the
  // addend's slices last), and the output is Q^T -- except for the last update before the Q X
  // that consumes Q, which writes only its transposed output, the row form Q that Q X reads.
  // A Q that is still P itself (after a start or restart) is symmetric and serves as either
  // form. Two slots, used in turn.
  auto q_args = [&](Group& g, NtArgs& s, int from, float a_, bool last) {
    const int to = 1 - from;
    square_operands(g, s, g.qslot[from], g.w.Pm, g.qslot[from]);
    s.mode = EPI_NS; s.alpha = 1.f; s.beta = a_;
    s.c_in = C_IS_A;                           // the addend is the A panel's last slices
    if (last) s.DT = g.qslot[to];              // Q, the row form
    else s.D = g.qslot[to];                    // Q^T
    g.qbuf[to] = g.qslot[to];
  };
  auto q_update = [&](int from, float a_, bool last) -> int {
    return nt_product(c, PC_POLY, square_flops,
                      [&](Group& g, NtArgs& s) { q_args(g, s, from, a_, last); });
  };
  // A Q update with R's update and another step behind it: W, R and the next Z do not read Q, so
  // its tiles may go where these triangle launches leave CUs idle, and what is left run with the
  // last of them (nt_fill_pays). One 4096^2 matrix: 136 tiles each on 256 CUs, so the 256 tiles of
  // the update cost no launch of their own. As a D-only product it is EPI_SYM's arithmetic without
  // a triangle (alpha = 1: the same bits). Needs a table entry per group.
  NtFill fill;
  bool filling = false;
  // iterations from it up to the next restart (or T): the Q updates the segment has left
  auto updates_left = [&](int it) {
    int end = it + 1;
    while (end < T && !is_restart(end)) ++end;
    return end - it;
  };
  auto gram = [&]() {
    return nt_product(c, PC_SYRK, syrk_flops, [&](Group& g, NtArgs& s) {
      gram_of_x(g, s, g.w.Am, g.rs / (kNsKx * kNsKx));
    });
  };
  int qs = -1;               // slot of the current Q, -1: none since the last (re)start
  if (gram()) return 1;
  // Matrices of at most 128 rows: a segment's m x m products in one launch, one workgroup per
  // matrix with everything in LDS (the same bits). All groups of the call, and segments of at
  // most kGramSmallSteps steps.
  bool small = c.tile == kGramSmallSide;
  for (int i = 0; i < c.n; ++i) small = small && c.g[i].m_pad == kGramSmallSide;
  for (int it = 0, end; small && it < T; it = end) {
    for (end = it + 1; end < T && !is_restart(end);) ++end;
    small = end - it <= kGramSmallSteps;
  }
  for (int it = 0; it < T; ++it) {
    if (it != 0 && is_restart(it) && qs >= 0) {
      if (nt_product(c, PC_GEMM, gemm_flops,
                     [&](Group& g, NtArgs& s) { px_next(g, s, g.qbuf[qs], 0.f); }))
        return 1;
      x_advance(c);
      for (int i = 0; i < c.n; ++i) c.g[i].rs = 1.f;
      if (gram()) return 1;
      qs = -1;
    }
    if (small) {
      GramSmallArgs a;
      a.n = c.n;
      a.steps = updates_left(it);
      for (int k = 0; k < 3 * a.steps; ++k) a.coeff[k] = coeffs[3 * it + k];
      int matrices = 0;
      double flops = 0.0;
      for (int i = 0; i < c.n; ++i) {
        Group& g = c.g[i];
        a.g[i] = GramSmallGroup{g.w.Am, g.qslot[0], matrices, g.km, g.rs};
        g.qbuf[0] = g.qslot[0];
        matrices += g.batch;
        flops += (3 * a.steps - 2) * poly_flops(g) + (a.steps - 1) * square_flops(g);
      }
      if (timed(PC_POLY, flops, 0.0, c.stream, c.who,
                [&] { return launch_gram_small(a, matrices, c.stream); }))
        return 1;
      qs = 0;
      it += a.steps - 1;
      continue;
    }
    const float ca = coeffs[3 * it], cb = coeffs[3 * it + 1], cc = coeffs[3 * it + 2];
    const bool evolve = it + 1 < T && !is_restart(it + 1);
    // Z = c R^2 + b R; after a (re)start also Q = Z + a I, as the epilogue's second output, or,
    // when R is not updated afterwards (Z itself is not needed), as the only one
    const bool fresh = qs < 0, only_q = fresh && !evolve;
    if (filling)   // the update still reads the old Z: the new one goes where W was
      for (int i = 0; i < c.n; ++i) std::swap(c.g[i].w.Pm, c.g[i].w.Wm);
    if (nt_product(c, PC_POLY, poly_flops, [&](Group& g, NtArgs& s) {
          uint16_t* R = g.w.Am;
          symmetric_square(g, s, R, R, R, only_q ? g.qslot[0] : g.w.Pm, cc / (g.rs * g.rs),
                           cb / g.rs, only_q ? ca : 0.f, fresh && evolve ? g.qslot[0] : nullptr,
                           fresh && evolve ? ca : 0.f);
          if (fresh) g.qbuf[0] = g.qslot[0];
        }, filling ? &fill : nullptr, true))
      return 1;
    filling = false;
    auto w_args = [&](Group& g, NtArgs& s) {   // W = Z R + a R (the stored R is rs times R)
      symmetric_square(g, s, g.w.Pm, g.w.Am, g.w.Am, g.w.Wm, 1.f, ca, 0.f);
    };
    if (!fresh && evolve && 2 * c.n <= kMaxGroups) {
      NtArgs tri[kMaxGroups];
      product_args(c, tri, w_args);
      product_args(c, fill.a, [&](Group& g, NtArgs& s) {
        q_args(g, s, qs, ca, false);
        s.mode = EPI_SYM;
      });
      fill.next = 0;
      filling = nt_fill_pays(tri, fill.a, c.n, c.tile, 0);
    }
    if (fresh) {
      qs = 0;
    } else if (filling) {
      qs = 1 - qs;
    } else {
      if (q_update(qs, ca, updates_left(it) == 1)) return 1;   // Q <- Z Q + a Q
      qs = 1 - qs;
    }
    if (evolve) {
      // W, then R = P R P = W Z + a W
      NtFill* more = filling ? &fill : nullptr;
      if (nt_product(c, PC_POLY, poly_flops, w_args, more) ||
          nt_product(c, PC_POLY, poly_flops, [&](Group& g, NtArgs& s) {
            symmetric_square(g, s, g.w.Wm, g.w.Pm, g.w.Wm, g.w.Am, 1.f / g.rs, ca / g.rs, 0.f);
          }, more))
        return 1;
      for (int i = 0; i < c.n; ++i) c.g[i].rs = 1.f;
    }
  }
  return nt_product(c, PC_FINAL, gemm_flops,
                    [&](Group& g, NtArgs& s) { px_final(g, s, g.qbuf[qs], 0.f, decay); });
}

// Momentum, norm and NS operands of every group of a call.
// A group's matrices share the m x n NS shape: [0, batch - n_t) are rows x cols and the last n_t
// are cols x rows (their transposes). Each orientation is staged into its slice of the
// workspace; everything after the staging sees one m x n batch, and the final epilogue writes
// each matrix back in its own orientation. (Square shapes have one orientation: the n_t part is
// staged and written like the rest.)
int run_stage(const Call& c, float mu, int nesterov, float eps) {
  PreArgs p[2 * kMaxGroups];
  int np = 0;
  bool est = false, exact = false;
  double pre_bytes = 0.0, st_bytes = 0.0, norm_bytes = 0.0;
  NormArgs na[kMaxGroups];
  for (int i = 0; i < c.n; ++i) {
    const Group& g = c.g[i];
    (g.est_ptrs ? est : exact) = true;
    for (int part = 0; part < 2; ++part) {
      const int l0 = part == 0 ? 0 : g.batch - g.n_t, L = part == 0 ? g.batch - g.n_t : g.n_t;
      if (L == 0) continue;
      const int r_ = part == 0 ? g.rows : g.cols, c_ = part == 0 ? g.cols : g.rows;
      const bool tall_ = r_ > c_;
      PreArgs& q = p[np++];
      q = PreArgs{};
      q.g_ptrs = g.g_ptrs + l0;
      q.g_dtype = g.g_dtype;
      q.buf_ptrs = g.buf_ptrs ? g.buf_ptrs + l0 : nullptr;
      q.est_ptrs = g.est_ptrs ? g.est_ptrs + l0 : nullptr;
      q.Y = q.YT = g.w.X + l0 * g.xs;
      q.ldy = tall_ ? g.m_pad : g.n_pad;
      q.ldyt = tall_ ? g.n_pad : g.m_pad;
      q.sY = q.sYT = g.xs;
      q.partials = g.w.partials + (long long)l0 * g.w.nparts;
      q.rows = r_;
      q.cols = c_;
      q.Rp = tall_ ? g.n_pad : g.m_pad;
      q.Cp = tall_ ? g.m_pad : g.n_pad;
      q.L = L;
      q.mu = mu;
      q.first_step = g.first_step;
      q.nesterov = nesterov;
      q.kx = kNsKx;
      q.scale = g.w.scale + l0;
      q.restage = g.est_ptrs ? g.w.restage + l0 : nullptr;
      q.est_old = g.w.est_old + l0;
      q.norm_group = i;
      q.norm_l0 = l0;
      // the NS products read X k-major, so only X is staged: by the direct write for a wide
      // orientation, by the transposed one for a tall orientation
      q.skip_y = tall_ ? 1 : 0;
      q.skip_yt = tall_ ? 0 : 1;
      // algorithmic bytes (what one ideal pass moves): gradient read, fp32 momentum read (not on
      // the first step) and write, one 2-byte copy of the normalised ns_in. The second pass's
      // re-read of the gradient and the new momentum (fp16 cannot hold an un-normalised
      // gradient, so the copy waits for the norm) is overhead, not counted.
      const double elems = (double)r_ * c_ * L;
      pre_bytes += elems * ((g.g_dtype == DMUON_DTYPE_F32 ? 4.0 : 2.0) +
                            (g.buf_ptrs ? (g.first_step ? 4.0 : 8.0) : 0.0) +
                            (g.est_ptrs ? 2.0 : 0.0));
      if (!g.est_ptrs) st_bytes += elems * 2.0;
    }
    na[i] = NormArgs{g.w.partials, g.w.nparts, g.batch, g.w.scale, g.w.est_old, g.est_ptrs,
                     g.w.ratio, g.w.ratio_sq, g.w.restage};
    norm_bytes += (double)g.batch * g.w.nparts * 4;
  }
  if (est && exact)
    return fail("%s: est_ptrs must be given for every group of a call or for none", c.who);
  // With est_ptrs (a per-matrix scale kept from the previous step) the first pass also writes
  // the fp16 copy as fp16(kx * est * ns_in); the norm finalize then keeps that copy when
  // r = scale / est is within [1/4, 4] (the first products multiply by r or r^2, and every copy
  // entry stays below kx / r <= 2^14) and otherwise flags the matrix for the second pass,
  // which then stages exactly as without an estimate.
  auto stage = [&](int st, bool flagged) {
    for (int k = 0; k < np; ++k) {
      p[k].stage = st;
      if (!flagged) p[k].restage = nullptr;
    }
  };
  const int* flags[2 * kMaxGroups];
  for (int k = 0; k < np; ++k) flags[k] = p[k].restage;
  stage(est ? PRE_EST : PRE_NORM, false);
  if (timed(PC_PRE, 0.0, pre_bytes, c.stream, c.who,
            [&] { return launch_pre_batch(p, np, c.stream); }))
    return 1;
  // small matrices: the norm and the exact staging in one launch
  if (norm_stage_pays(na, c.n, p, np)) {
    stage(PRE_F16, false);
    return timed(PC_NORM, 0.0, norm_bytes + st_bytes, c.stream, c.who,
                 [&] { return launch_norm_stage(na, c.n, p, np, eps, c.stream); });
  }
  if (timed(PC_NORM, 0.0, norm_bytes, c.stream, c.who,
            [&] { return launch_norm_finalize_est(na, c.n, eps, c.stream); }))
    return 1;
  for (int k = 0; k < np; ++k) p[k].restage = flags[k];
  stage(PRE_F16, est);
  return timed(PC_PRE, 0.0, st_bytes, c.stream, c.who,
               [&] { return launch_pre_batch(p, np, c.stream); });
}

// Argument checks and the workspace of a call's groups, `c.g[i]` holding the caller's fields.
// phases: PH_STAGE (momentum, norm, NS operand staging into the workspace), PH_APPLY (the NS
// products and the fused update / output from a staged workspace), or both.
enum { PH_STAGE = 1, PH_APPLY = 2 };
int group_setup(Call& c, int tile_req, int backend, void* workspace, int64_t workspace_bytes,
                int phases) {
  const char* who = c.who;
  const int gram = backend == DMUON_NS_GRAM;
  if (!workspace || !aligned16(workspace)) return fail("%s: workspace NULL or misaligned", who);
  int64_t off = 0;
  for (int i = 0; i < c.n; ++i) {
    Group& g = c.g[i];
    if (phases & PH_STAGE) {
      if (!g.g_ptrs) return fail("%s: g_ptrs is NULL", who);
      if (g.g_dtype != DMUON_DTYPE_F32 && g.g_dtype != DMUON_DTYPE_BF16)
        return fail("%s: unsupported gradient dtype code %d", who, g.g_dtype);
    }
    if (phases & PH_APPLY) {
      if (g.w_ptrs && g.w_dtype != DMUON_DTYPE_F32 && g.w_dtype != DMUON_DTYPE_BF16)
        return fail("%s: unsupported weight dtype code %d", who, g.w_dtype);
      if (g.out_ptrs && g.out_dtype != DMUON_DTYPE_F32 && g.out_dtype != DMUON_DTYPE_BF16)
        return fail("%s: unsupported output dtype code %d", who, g.out_dtype);
      if (g.pub_ptrs && !g.w_ptrs)
        return fail("%s: pub_ptrs needs w_ptrs (it copies the new W)", who);
      if (g.pub_ptrs && g.pub_dtype != DMUON_DTYPE_F32 && g.pub_dtype != DMUON_DTYPE_BF16)
        return fail("%s: unsupported publish dtype code %d", who, g.pub_dtype);
    }
    if (g.n_t < 0 || g.n_t > g.batch)
      return fail("%s: n_transposed=%d outside [0, batch=%d]", who, g.n_t, g.batch);
    int tile;
    int64_t need;
    if (plan(g.rows, g.cols, g.batch, tile_req, 0, gram, &tile, &g.m_pad, &g.n_pad, &need))
      return 1;
    c.tile = tile;                       // several groups come with the tile of their plan
    if (workspace_bytes - off < need)
      return fail("%s: workspace of %lld bytes is smaller than the %lld bytes planned", who,
                  (long long)workspace_bytes, (long long)(off + need));
    g.tall = g.rows > g.cols;
    g.m = g.tall ? g.cols : g.rows;
    g.n = g.tall ? g.rows : g.cols;
    g.km = (int)round_up(g.m, 64);
    g.kn = (int)round_up(g.n, 64);
    g.n_flip = g.rows == g.cols ? 0 : g.n_t;
    g.xs = (long long)g.m_pad * g.n_pad;
    g.as = (long long)g.m_pad * g.m_pad;
    g.w = carve(static_cast<char*>(workspace) + off, g.m_pad, g.n_pad,
                g.tall ? g.n_pad : g.m_pad, g.tall ? g.m_pad : g.n_pad, g.batch, gram);
    off += need;
    g.x_cur = g.w.X;
    g.x_nxt = g.w.X2;
    g.x_staged = true;
    int kr = 1;
    while (kr * 2 <= g.m && kr < 4096) kr *= 2;
    g.rs = (float)kr;                    // the stored R is rs * (X X^T of the normalised X)
    g.qslot[0] = g.qbuf[0] = g.w.Q0;
    g.qslot[1] = g.qbuf[1] = g.w.Q1;
  }
  return 0;
}

// The whole Newton-Schulz + optional update sequence of a call's groups; see
// dmuon_muon_step_group.
int run_groups(Call& c, float mu, int nesterov, float decay, const float* coeffs, int T,
               int backend, const int* restarts, int n_restarts, float eps, void* workspace,
               int64_t workspace_bytes, int tile_req, int phases = PH_STAGE | PH_APPLY) {
  const char* who = c.who;
  if (phases & PH_APPLY) {
    if (!coeffs || T <= 0)
      return fail("%s: need at least one (a, b, c) coefficient triple", who);
    if (n_restarts < 0 || (n_restarts > 0 && !restarts))
      return fail("%s: restart list NULL or of negative length", who);
  }
  if (backend != DMUON_NS_DIRECT && backend != DMUON_NS_GRAM)
    return fail("%s: unknown NS backend %d", who, backend);
  if (group_setup(c, tile_req, backend, workspace, workspace_bytes, phases)) return 1;
  if ((phases & PH_STAGE) && run_stage(c, mu, nesterov, eps)) return 1;
  if (!(phases & PH_APPLY)) return 0;
  return backend == DMUON_NS_GRAM ? run_gram(c, coeffs, T, restarts, n_restarts, decay)
                                  : run_direct(c, coeffs, T, decay);
}

// The update scale of a shape, lr * 0.2 sqrt(max(rows, cols)), and the weight decay factor: host
// scalars in double, rounded once to fp32, as torch does with Python-float arguments.
float update_scale(double lr, int rows, int cols) {
  return (float)(lr * (0.2 * sqrt((double)(rows > cols ? rows : cols))));
}
float decay_of(double lr, double wd) { return wd > 0.0 ? (float)(1.0 - lr * wd) : 1.f; }

// ---- scratch of dmuon_muon_step_group_noalloc (the array itself is at file scope above) --------
constexpr int64_t kScratchBytes = DMUON_NOALLOC_SCRATCH_BYTES;
constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
void* g_scratch_ptr[kMaxDevices] = {};

// The device address of the current GPU's copy of `scratch`, resolved once per device. The
// first resolution may load the library's code object, so it is not itself allocation-free:
// dmuon_noalloc_init does it at set-up. With `capture_stream_checked`, a first resolution while
// `stream` is being captured is refused instead (it would run inside the capture).
int scratch_of_current_device(const char* who, void** out, bool capture_stream_checked = false,
                              hipStream_t stream = nullptr) {
  int dev = -1;
  const hipError_t ge = hipGetDevice(&dev);
  if (ge != hipSuccess || dev < 0 || dev >= kMaxDevices)
    return fail("%s: no current HIP device (%s)", who, hipGetErrorString(ge));
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  if (!g_scratch_ptr[dev]) {
    if (capture_stream_checked) {
      hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
      if (hipStreamIsCapturing(stream, &cs) == hipSuccess && cs != hipStreamCaptureStatusNone)
        return fail("%s: first use on device %d while its stream is being captured: call "
                    "dmuon_noalloc_init() (or the entry point once, eagerly) on this device "
                    "before capturing", who, dev);
    }
    void* p = nullptr;
    const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !p)
      return fail("%s: hipGetSymbolAddress(scratch) failed on device %d: %s", who, dev,
                  hipGetErrorString(e));
    g_scratch_ptr[dev] = p;
  }
  *out = g_scratch_ptr[dev];
  return 0;
}

struct NoEvents {
  NoEvents() { g_no_events = true; }
  ~NoEvents() { g_no_events = false; }
};

}  // namespace

extern "C" {

const char* dmuon_last_error(void) { return g_last_error.c_str(); }

int dmuon_stream_copy(const void* src, void* dst, int64_t bytes, void* stream) {
  const char* who = "dmuon_stream_copy";
  if (bytes == 0) return 0;
  if (!src || !dst || bytes < 0) return fail("%s: NULL buffer or negative size", who);
  if (!aligned16(src) || !aligned16(dst) || bytes % 16)
    return fail("%s: buffers must be 16-byte aligned and the size a multiple of 16 (got %lld)",
                who, (long long)bytes);
  const uintptr_t s = reinterpret_cast<uintptr_t>(src), d = reinterpret_cast<uintptr_t>(dst);
  if (s < d + (uintptr_t)bytes && d < s + (uintptr_t)bytes)
    return fail("%s: source and destination overlap", who);
  return check_launch(launch_stream_copy(src, dst, bytes / 16, static_cast<hipStream_t>(stream)),
                      who);
}

int dmuon_profile_enable(int on) {
  g_prof.on = on != 0;
  return 0;
}

int dmuon_profile_collect(double* ms, int64_t* launches, double* flops, double* bytes,
                          int n_classes) {
  if (n_classes < PC_COUNT || !ms || !launches || !flops || !bytes)
    return fail("dmuon_profile_collect: need arrays of at least %d classes", (int)PC_COUNT);
  for (int c = 0; c < n_classes; ++c) {
    ms[c] = 0.0;
    launches[c] = 0;
    flops[c] = 0.0;
    bytes[c] = 0.0;
  }
  int rc = 0;
  for (const ProfRec& r : g_prof.recs) {
    float t = 0.f;
    if (hipEventSynchronize(r.b) != hipSuccess || hipEventElapsedTime(&t, r.a, r.b) != hipSuccess)
      rc = fail("dmuon_profile_collect: event query failed");
    ms[r.cls] += t;
    launches[r.cls] += 1;
    flops[r.cls] += r.flops;
    bytes[r.cls] += r.bytes;
    g_prof.pool.push_back(r.a);
    g_prof.pool.push_back(r.b);
  }
  g_prof.recs.clear();
  return rc;
}

int dmuon_abi_version(void) { return DMUON_ABI_VERSION; }

}  // extern "C"

namespace {

// 16-bit operand type of the product entry points: DMUON_DTYPE_BF16 or DMUON_DTYPE_F16
int elt_of(const char* who, int dtype, int* elt) {
  if (dtype == DMUON_DTYPE_BF16) { *elt = ELT_BF16; return 0; }
  if (dtype == DMUON_DTYPE_F16) { *elt = ELT_F16; return 0; }
  return fail("%s: operand dtype code %d is not a 16-bit type (bf16 %d, fp16 %d)", who, dtype,
              DMUON_DTYPE_BF16, DMUON_DTYPE_F16);
}

// The SYRK seam (syrk_or_cublas) for any M and K. The NT kernel reads whole tiles (M a
// multiple of the tile, K of the 64-wide slice) from 16-byte aligned rows; a call that does
// not meet that runs on zero-padded copies in the caller's workspace -- A [L][Mp][Kp], B (when
// it is another matrix), C [L][Mp][Mp] and D [L][Mp][Mp] -- and the M x M corner of the padded
// result is copied into D. Zero rows and columns of A and B leave the corner unchanged.
struct SyrkPlan {
  int tile, Mp, Kp;
  bool direct;                 // the caller's operands are used in place, as whole tiles
  bool edge;                   // they are used in place up to their real sides
  bool b_copy;
  int64_t offB, offC, offD, bytes;
};

// Whether two batches of matrices in row pitch ld and batch stride share any byte of the ranges
// they span.
bool spans_overlap(const void* a, int64_t lda, int64_t sa, int cols_a, const void* b, int64_t ldb,
                   int64_t sb, int cols_b, int rows, int batch) {
  auto last = [&](int64_t ld, int64_t s, int cols) {
    return 2 * ((batch > 1 ? (batch - 1) * s : 0) + (rows - 1) * ld + cols);
  };
  const intptr_t x = reinterpret_cast<intptr_t>(a), y = reinterpret_cast<intptr_t>(b);
  return x < y + last(ldb, sb, cols_b) && y < x + last(lda, sa, cols_a);
}

int syrk_plan(const char* who, const void* A, int64_t lda, int64_t strideA, const void* B,
              int64_t ldb, int64_t strideB, const void* C, int64_t ldc, int64_t strideC,
              const void* D, int64_t ldd, int64_t strideD, int M, int K, int batch, int tile_req,
              SyrkPlan* pl) {
  if (tile_req != 0 && tile_req != 128 && tile_req != 256)
    return fail("%s: tile must be 0 (automatic), 128 or 256, got %d", who, tile_req);
  if (M < 0 || K < 0 || batch < 0) return fail("%s: bad sizes M=%d K=%d batch=%d", who, M, K, batch);
  if (!A || !D) return fail("%s: A and D must be non-NULL", who);
  if (lda < K || ldb < K || ldd < M || (C && ldc < M))
    return fail("%s: leading dimension smaller than the row length", who);
  if (batch > 1 && (strideA < 0 || strideB < 0 || strideD < 0 || (C && strideC < 0)))
    return fail("%s: batch strides must be non-negative", who);
  if (D == A || D == B || (C && D == C)) return fail("%s: D must not alias A, B or C", who);
  // C is an M x M matrix; an operand is M x K. The two can be one matrix only when K == M
  // (the polynomial Z = c R R^T + b R); otherwise the epilogue would read an M x M addend
  // over an M x K operand's rows.
  if (C && (C == A || C == B) && K != M)
    return fail("%s: C aliases %s but K=%d != M=%d (an M x M addend cannot be an M x K operand)",
                who, C == A ? "A" : "B", K, M);
  int t = tile_req;
  if (t == 0) {
    t = auto_tile(M, K > 0 ? K : 1, batch, 256);
    if (t == 256 && round_up(M, 256) != round_up(M, 128)) t = 128;   // no padded copy for 256
  }
  pl->tile = t;
  pl->Mp = (int)round_up(M, t);
  pl->Kp = (int)round_up(K > 0 ? K : 1, 64);
  const bool b_same = B == A && ldb == lda && strideB == strideA;
  pl->direct = M % t == 0 && K % 64 == 0 && K > 0 && aligned16(A) && aligned16(B) &&
               aligned16(D) && (!C || aligned16(C)) && ld_ok(lda) && ld_ok(ldb) && ld_ok(ldd) &&
               (!C || ld_ok(ldc)) && stride_ok(strideA, batch) && stride_ok(strideB, batch) &&
               stride_ok(strideD, batch) && (!C || stride_ok(strideC, batch));
  pl->b_copy = !b_same;
  // Ragged operands in whole 16-byte chunks (M and K multiples of 8, aligned rows) are read and
  // written in place by the edge variant of the 128- and 64-tile kernels: one launch instead of
  // up to four (fp16 1000 x 3000, X X^T and its polynomial: 45.4 -> 28.1 us the pair, 3-6 us
  // for each copy). A product of more than two 128-tiles per CU (512: the plan of a call, like its
  // tile, is for 256 CUs, without a look at the device) keeps the copies and the 256-tile kernel,
  // which are small beside it.
  const int64_t mt = pl->Mp / 128;
  pl->edge = !pl->direct && t == 128 && M % 8 == 0 && K % 8 == 0 && K > 0 && aligned16(A) &&
             aligned16(B) && aligned16(D) && (!C || aligned16(C)) && ld_ok(lda) && ld_ok(ldb) &&
             ld_ok(ldd) && (!C || ld_ok(ldc)) && stride_ok(strideA, batch) &&
             stride_ok(strideB, batch) && stride_ok(strideD, batch) &&
             (!C || stride_ok(strideC, batch)) && 128 * lda * 2 < (1LL << 31) &&
             128 * ldb * 2 < (1LL << 31) && mt * (mt + 1) / 2 * batch <= 512;
  // The copies read everything before D is stored: a D that lies over an operand or the addend in
  // part (its own address is refused above) keeps them.
  pl->edge = pl->edge && !spans_overlap(A, lda, strideA, K, D, ldd, strideD, M, M, batch) &&
             !spans_overlap(B, ldb, strideB, K, D, ldd, strideD, M, M, batch) &&
             !(C && spans_overlap(C, ldc, strideC, M, D, ldd, strideD, M, M, batch));
  const int64_t L = batch, xa = L * pl->Mp * (int64_t)pl->Kp * 2, xd = L * pl->Mp * (int64_t)pl->Mp * 2;
  int64_t off = align256(xa);
  pl->offB = pl->b_copy ? off : 0;
  if (pl->b_copy) off += align256(xa);
  pl->offC = C ? off : 0;
  if (C) off += align256(xd);
  pl->offD = off;
  off += align256(xd);
  pl->bytes = pl->direct || pl->edge ? 0 : off;
  return 0;
}

int syrk_impl(const char* who, int elt, const void* A, int64_t lda, int64_t strideA,
              const void* B, int64_t ldb, int64_t strideB, const void* C, int64_t ldc,
              int64_t strideC, void* D, int64_t ldd, int64_t strideD, int M, int K, int batch,
              float alpha, float beta, float diag_add, const float* alpha_dev, int tile_req,
              void* workspace, int64_t workspace_bytes, hipStream_t stream) {
  if (batch == 0 || M == 0) return 0;
  if (!B) { B = A; ldb = lda; strideB = strideA; }
  SyrkPlan pl;
  if (syrk_plan(who, A, lda, strideA, B, ldb, strideB, C, ldc, strideC, D, ldd, strideD, M, K,
                batch, tile_req, &pl))
    return 1;
  NtArgs s{};
  s.elt = elt;
  s.M = pl.Mp; s.N = pl.Mp; s.K = pl.Kp; s.L = batch;
  s.mt = s.nt = pl.Mp / pl.tile; s.tiles_per_mat = tri_tiles(pl.Mp, pl.tile); s.tri = 1;
  s.mode = EPI_SYM; s.alpha = alpha; s.beta = C ? beta : 0.f; s.diag = diag_add;
  s.alpha_dev = alpha_dev;
  if (pl.direct || pl.edge) {
    s.A = static_cast<const uint16_t*>(A); s.lda = lda; s.sA = strideA;
    s.B = static_cast<const uint16_t*>(B); s.ldb = ldb; s.sB = strideB;
    s.C = static_cast<const uint16_t*>(C); s.ldc = ldc; s.sC = strideC;
    if (C && C == A && ldc == lda && (batch <= 1 || strideC == strideA) && K == M &&
        pl.Kp == pl.Mp)
      s.c_in = C_IS_A;
    if (pl.edge) {
      s.edge = 1; s.m_real = M; s.k_real = K;
      s.live_rows = s.live_cols = (int)round_up(M, 64);
    }
    s.D = static_cast<uint16_t*>(D); s.ldd = ldd; s.sD = strideD;
    return check_launch(launch_nt(s, pl.tile, stream), who);
  }
  if (!workspace)
    return fail("%s: M=%d, K=%d or the operand layout needs the padded path (M a multiple of "
                "the tile %d, K of 64, 16-byte aligned rows otherwise), which needs a workspace "
                "of %lld bytes (dmuon_syrk_workspace_size)", who, M, K, pl.tile,
                (long long)pl.bytes);
  if (!aligned16(workspace) || workspace_bytes < pl.bytes)
    return fail("%s: workspace misaligned or smaller than the %lld bytes of the padded path", who,
                (long long)pl.bytes);
  char* ws = static_cast<char*>(workspace);
  const long long sa = (long long)pl.Mp * pl.Kp, sd = (long long)pl.Mp * pl.Mp;
  uint16_t* Ap = reinterpret_cast<uint16_t*>(ws);
  uint16_t* Bp = pl.b_copy ? reinterpret_cast<uint16_t*>(ws + pl.offB) : Ap;
  uint16_t* Cp = C ? reinterpret_cast<uint16_t*>(ws + pl.offC) : nullptr;
  uint16_t* Dp = reinterpret_cast<uint16_t*>(ws + pl.offD);
  if (check_launch(launch_pad_copy(static_cast<const uint16_t*>(A), lda, strideA, Ap, pl.Kp, sa,
                                   M, K, pl.Mp, pl.Kp, batch, stream), who))
    return 1;
  if (pl.b_copy &&
      check_launch(launch_pad_copy(static_cast<const uint16_t*>(B), ldb, strideB, Bp, pl.Kp, sa,
                                   M, K, pl.Mp, pl.Kp, batch, stream), who))
    return 1;
  // C == A (K == M): the padded C is the padded copy of A itself, and its tile is the A panel's
  // last slices (NtArgs::c_in)
  const bool c_from_a = C && C == A && ldc == lda && (batch <= 1 || strideC == strideA) &&
                        K == M && pl.Kp == pl.Mp;
  if (C && !c_from_a &&
      check_launch(launch_pad_copy(static_cast<const uint16_t*>(C), ldc, strideC, Cp, pl.Mp, sd,
                                   M, M, pl.Mp, pl.Mp, batch, stream), who))
    return 1;
  s.A = Ap; s.lda = pl.Kp; s.sA = sa;
  s.B = Bp; s.ldb = pl.Kp; s.sB = sa;
  s.C = Cp; s.ldc = pl.Mp; s.sC = sd;
  if (c_from_a) { s.C = Ap; s.ldc = pl.Kp; s.sC = sa; s.c_in = C_IS_A; }
  s.D = Dp; s.ldd = pl.Mp; s.sD = sd;
  if (check_launch(launch_nt(s, pl.tile, stream), who)) return 1;
  return check_launch(launch_pad_copy(Dp, pl.Mp, sd, static_cast<uint16_t*>(D), ldd, strideD, M,
                                      M, M, M, batch, stream), who);
}

}  // namespace

extern "C" {

int dmuon_syrk_workspace_size(int dtype, const void* A, int64_t lda, int64_t strideA,
                              const void* B, int64_t ldb, int64_t strideB, const void* C,
                              int64_t ldc, int64_t strideC, const void* D, int64_t ldd,
                              int64_t strideD, int M, int K, int batch, int tile,
                              int64_t* workspace_bytes) {
  const char* who = "dmuon_syrk_workspace_size";
  int elt;
  if (!workspace_bytes) return fail("%s: NULL output", who);
  *workspace_bytes = 0;
  if (elt_of(who, dtype, &elt)) return 1;
  if (batch == 0 || M == 0) return 0;
  if (!B) { B = A; ldb = lda; strideB = strideA; }
  SyrkPlan pl;
  if (syrk_plan(who, A, lda, strideA, B, ldb, strideB, C, ldc, strideC, D, ldd, strideD, M, K,
                batch, tile, &pl))
    return 1;
  *workspace_bytes = pl.bytes;
  return 0;
}

int dmuon_syrk(int dtype, const void* A, int64_t lda, int64_t strideA, const void* B, int64_t ldb,
               int64_t strideB, const void* C, int64_t ldc, int64_t strideC, void* D, int64_t ldd,
               int64_t strideD, int M, int K, int batch, float alpha, float beta, float diag_add,
               const float* alpha_dev, int tile, void* workspace, int64_t workspace_bytes,
               void* stream) {
  const char* who = "dmuon_syrk";
  int elt;
  if (elt_of(who, dtype, &elt)) return 1;
  return syrk_impl(who, elt, A, lda, strideA, B, ldb, strideB, C, ldc, strideC, D, ldd, strideD,
                   M, K, batch, alpha, beta, diag_add, alpha_dev, tile, workspace,
                   workspace_bytes, static_cast<hipStream_t>(stream));
}

int dmuon_syrk_bf16(const void* A, int64_t lda, int64_t strideA, const void* B, int64_t ldb,
                    int64_t strideB, const void* C, int64_t ldc, int64_t strideC, void* D,
                    int64_t ldd, int64_t strideD, int M, int K, int batch, float alpha, float beta,
                    float diag_add, const float* alpha_dev, int tile, void* stream) {
  const char* who = "dmuon_syrk_bf16";
  if (batch == 0 || M == 0) return 0;
  if (tile != 128 && tile != 256) return fail("%s: tile must be 128 or 256, got %d", who, tile);
  if (M > 0 && M % tile) return fail("%s: M=%d is not a multiple of the tile %d", who, M, tile);
  if (K > 0 && K % 64) return fail("%s: K=%d is not a multiple of 64", who, K);
  if (!aligned16(A) || (B && !aligned16(B)) || !aligned16(D) || (C && !aligned16(C)))
    return fail("%s: operands must be 16-byte aligned", who);
  return syrk_impl(who, ELT_BF16, A, lda, strideA, B, ldb, strideB, C, ldc, strideC, D, ldd,
                   strideD, M, K, batch, alpha, beta, diag_add, alpha_dev, tile, nullptr, 0,
                   static_cast<hipStream_t>(stream));
}

static int gemm_common_checks(const char* who, const void* P, int64_t ldp, int64_t strideP,
                              const void* XT, int64_t ldxt, int64_t strideXT, const void* X,
                              int64_t ldx, int64_t strideX, int M, int N, int batch, int tile) {
  if (tile != 128 && tile != 256) return fail("%s: tile must be 128 or 256, got %d", who, tile);
  if (M <= 0 || N <= 0 || batch < 0) return fail("%s: bad sizes M=%d N=%d batch=%d", who, M, N, batch);
  if (M % tile || N % tile) return fail("%s: M=%d and N=%d must be multiples of the tile %d", who, M, N, tile);
  if (!P || (!XT && !X)) return fail("%s: P and one of XT / X must be non-NULL", who);
  if (!aligned16(P) || (XT && !aligned16(XT)) || (X && !aligned16(X)))
    return fail("%s: operands must be 16-byte aligned", who);
  if (!ld_ok(ldp) || ldp < M || (XT && (!ld_ok(ldxt) || ldxt < M)) || (X && (!ld_ok(ldx) || ldx < N)))
    return fail("%s: bad leading dimensions", who);
  if (!stride_ok(strideP, batch) || (XT && !stride_ok(strideXT, batch)) ||
      (X && !stride_ok(strideX, batch)))
    return fail("%s: batch strides must be non-negative multiples of 8", who);
  // XT == NULL: the product reads X itself as its k-major B operand (one 32-bit buffer range
  // per matrix)
  if (!XT && (int64_t)M * ldx * 2 >= (1LL << 31))
    return fail("%s: X read in place needs M * ldx * 2 < 2^31 bytes (pass XT instead)", who);
  return 0;
}

// B operand of the NS-GEMM exports: X^T when given, else X read k-major
static void gemm_b_operand(NtArgs& g, const void* XT, int64_t ldxt, int64_t strideXT,
                           const void* X, int64_t ldx, int64_t strideX) {
  if (XT) {
    g.B = static_cast<const uint16_t*>(XT); g.ldb = ldxt; g.sB = strideXT;
  } else {
    g.B = static_cast<const uint16_t*>(X); g.ldb = ldx; g.sB = strideX; g.b_kmajor = 1;
  }
}

static int ns_gemm_impl(const char* who, int elt, const void* P, int64_t ldp, int64_t strideP, const void* XT, int64_t ldxt,
                       int64_t strideXT, const void* X, int64_t ldx, int64_t strideX, void* Xout,
                       int64_t ldxo, int64_t strideXo, void* XTout, int64_t ldxto,
                       int64_t strideXTo, int M, int N, int batch, float alpha, float beta,
                       const float* alpha_dev, int tile, void* stream) {
  if (batch == 0) return 0;
  if (gemm_common_checks(who, P, ldp, strideP, XT, ldxt, strideXT, X, ldx, strideX, M, N, batch, tile))
    return 1;
  if (!Xout || !aligned16(Xout) || !ld_ok(ldxo) || ldxo < N || !stride_ok(strideXo, batch))
    return fail("%s: bad Xout", who);
  if (XTout && (!aligned16(XTout) || !ld_ok(ldxto) || ldxto < M || !stride_ok(strideXTo, batch)))
    return fail("%s: bad XTout", who);
  if (XT && XTout == XT) return fail("%s: XTout must not alias XT", who);
  if (Xout == P || (XT && Xout == XT)) return fail("%s: Xout must not alias P or XT", who);
  if (!XT && Xout == X) return fail("%s: Xout must not alias X when X is the B operand", who);
  NtArgs g{};
  g.elt = elt;
  g.A = static_cast<const uint16_t*>(P); g.lda = ldp; g.sA = strideP;
  gemm_b_operand(g, XT, ldxt, strideXT, X, ldx, strideX);
  g.M = M; g.N = N; g.K = M; g.L = batch;
  g.mt = M / tile; g.nt = N / tile; g.tiles_per_mat = g.mt * g.nt; g.tri = 0;
  g.mode = EPI_NS; g.alpha = alpha; g.beta = X ? beta : 0.f; g.alpha_dev = alpha_dev;
  g.C = static_cast<const uint16_t*>(X); g.ldc = ldx; g.sC = strideX;
  g.D = static_cast<uint16_t*>(Xout); g.ldd = ldxo; g.sD = strideXo;
  g.DT = static_cast<uint16_t*>(XTout); g.lddt = ldxto; g.sDT = strideXTo;
  return check_launch(launch_nt(g, tile, static_cast<hipStream_t>(stream)), who);
}

static int ns_gemm_final_impl(const char* who, int elt, const void* P, int64_t ldp, int64_t strideP, const void* XT,
                             int64_t ldxt, int64_t strideXT, const void* X, int64_t ldx,
                             int64_t strideX, int M, int N, int batch, float alpha, float beta,
                             const float* alpha_dev, int m_real, int n_real, int transposed,
                             void* const* out_ptrs, int out_dtype, void* const* w_ptrs,
                             int w_dtype, void* const* pub_ptrs, int pub_dtype, float decay,
                             float lrs, int tile, void* stream) {
  if (batch == 0) return 0;
  if (gemm_common_checks(who, P, ldp, strideP, XT, ldxt, strideXT, X, ldx, strideX, M, N, batch, tile))
    return 1;
  if (m_real <= 0 || n_real <= 0 || m_real > M || n_real > N)
    return fail("%s: real extent %dx%d outside the padded %dx%d", who, m_real, n_real, M, N);
  if (!out_ptrs && !w_ptrs) return fail("%s: nothing to write (out_ptrs and w_ptrs NULL)", who);
  if (out_ptrs && out_dtype != DMUON_DTYPE_F32 && out_dtype != DMUON_DTYPE_BF16)
    return fail("%s: unsupported output dtype %d", who, out_dtype);
  if (w_ptrs && w_dtype != DMUON_DTYPE_F32 && w_dtype != DMUON_DTYPE_BF16)
    return fail("%s: unsupported weight dtype %d", who, w_dtype);
  if (pub_ptrs && !w_ptrs) return fail("%s: pub_ptrs needs w_ptrs (it copies the new W)", who);
  if (pub_ptrs && pub_dtype != DMUON_DTYPE_F32 && pub_dtype != DMUON_DTYPE_BF16)
    return fail("%s: unsupported publish dtype %d", who, pub_dtype);
  NtArgs g{};
  g.elt = elt;
  g.A = static_cast<const uint16_t*>(P); g.lda = ldp; g.sA = strideP;
  gemm_b_operand(g, XT, ldxt, strideXT, X, ldx, strideX);
  g.M = M; g.N = N; g.K = M; g.L = batch;
  g.mt = M / tile; g.nt = N / tile; g.tiles_per_mat = g.mt * g.nt; g.tri = 0;
  g.mode = EPI_FINAL; g.alpha = alpha; g.beta = X ? beta : 0.f; g.alpha_dev = alpha_dev;
  g.C = static_cast<const uint16_t*>(X); g.ldc = ldx; g.sC = strideX;
  g.out_ptrs = out_ptrs; g.out_dtype = out_dtype;
  g.w_ptrs = w_ptrs; g.w_dtype = w_dtype; g.decay = decay; g.lrs = lrs;
  g.pub_ptrs = pub_ptrs; g.pub_dtype = pub_dtype;
  g.m_real = m_real; g.n_real = n_real; g.transposed = transposed ? 1 : 0;
  return check_launch(launch_nt(g, tile, static_cast<hipStream_t>(stream)), who);
}

int dmuon_ns_gemm(int dtype, const void* P, int64_t ldp, int64_t strideP, const void* XT,
                  int64_t ldxt, int64_t strideXT, const void* X, int64_t ldx, int64_t strideX,
                  void* Xout, int64_t ldxo, int64_t strideXo, void* XTout, int64_t ldxto,
                  int64_t strideXTo, int M, int N, int batch, float alpha, float beta,
                  const float* alpha_dev, int tile, void* stream) {
  int elt;
  if (elt_of("dmuon_ns_gemm", dtype, &elt)) return 1;
  return ns_gemm_impl("dmuon_ns_gemm", elt, P, ldp, strideP, XT, ldxt, strideXT, X, ldx, strideX,
                      Xout, ldxo, strideXo, XTout, ldxto, strideXTo, M, N, batch, alpha, beta,
                      alpha_dev, tile, stream);
}

int dmuon_ns_gemm_bf16(const void* P, int64_t ldp, int64_t strideP, const void* XT, int64_t ldxt,
                       int64_t strideXT, const void* X, int64_t ldx, int64_t strideX, void* Xout,
                       int64_t ldxo, int64_t strideXo, void* XTout, int64_t ldxto,
                       int64_t strideXTo, int M, int N, int batch, float alpha, float beta,
                       const float* alpha_dev, int tile, void* stream) {
  return ns_gemm_impl("dmuon_ns_gemm_bf16", ELT_BF16, P, ldp, strideP, XT, ldxt, strideXT, X, ldx,
                      strideX, Xout, ldxo, strideXo, XTout, ldxto, strideXTo, M, N, batch, alpha,
                      beta, alpha_dev, tile, stream);
}

int dmuon_ns_gemm_final(int dtype, const void* P, int64_t ldp, int64_t strideP, const void* XT,
                        int64_t ldxt, int64_t strideXT, const void* X, int64_t ldx,
                        int64_t strideX, int M, int N, int batch, float alpha, float beta,
                        const float* alpha_dev, int m_real, int n_real, int transposed,
                        void* const* out_ptrs, int out_dtype, void* const* w_ptrs, int w_dtype,
                        void* const* pub_ptrs, int pub_dtype, float decay, float lrs, int tile,
                        void* stream) {
  int elt;
  if (elt_of("dmuon_ns_gemm_final", dtype, &elt)) return 1;
  return ns_gemm_final_impl("dmuon_ns_gemm_final", elt, P, ldp, strideP, XT, ldxt, strideXT, X,
                            ldx, strideX, M, N, batch, alpha, beta, alpha_dev, m_real, n_real,
                            transposed, out_ptrs, out_dtype, w_ptrs, w_dtype, pub_ptrs, pub_dtype,
                            decay, lrs, tile, stream);
}

int dmuon_ns_gemm_final_bf16(const void* P, int64_t ldp, int64_t strideP, const void* XT,
                             int64_t ldxt, int64_t strideXT, const void* X, int64_t ldx,
                             int64_t strideX, int M, int N, int batch, float alpha, float beta,
                             const float* alpha_dev, int m_real, int n_real, int transposed,
                             void* const* out_ptrs, int out_dtype, void* const* w_ptrs,
                             int w_dtype, void* const* pub_ptrs, int pub_dtype, float decay,
                             float lrs, int tile, void* stream) {
  return ns_gemm_final_impl("dmuon_ns_gemm_final_bf16", ELT_BF16, P, ldp, strideP, XT, ldxt,
                            strideXT, X, ldx, strideX, M, N, batch, alpha, beta, alpha_dev, m_real,
                            n_real, transposed, out_ptrs, out_dtype, w_ptrs, w_dtype, pub_ptrs,
                            pub_dtype, decay, lrs, tile, stream);
}

int dmuon_muon_pre_partials(int Rp, int Cp) { return pre_blocks_per_mat(Rp, Cp); }

int dmuon_muon_pre(void* const* g_ptrs, int g_dtype, float* const* buf_ptrs, void* Y, int64_t ldy,
                   int64_t strideY, void* YT, int64_t ldyt, int64_t strideYT, float* partials,
                   int rows, int cols, int Rp, int Cp, int batch, float mu, int first_step,
                   int nesterov, void* stream) {
  const char* who = "dmuon_muon_pre";
  if (batch == 0) return 0;
  if (!g_ptrs || (!Y && !YT) || !partials) return fail("%s: NULL argument", who);
  if (g_dtype != DMUON_DTYPE_F32 && g_dtype != DMUON_DTYPE_BF16)
    return fail("%s: unsupported gradient dtype %d", who, g_dtype);
  if (rows <= 0 || cols <= 0 || batch < 0) return fail("%s: bad sizes", who);
  if (Rp % 64 || Cp % 64 || Rp < rows || Cp < cols)
    return fail("%s: padded extent %dx%d must be multiples of 64 covering %dx%d", who, Rp, Cp, rows, cols);
  if ((Y && (!aligned16(Y) || !ld_ok(ldy) || ldy < Cp || !stride_ok(strideY, batch))) ||
      (YT && (!aligned16(YT) || !ld_ok(ldyt) || ldyt < Rp || !stride_ok(strideYT, batch))))
    return fail("%s: bad Y/YT layout", who);
  PreArgs p{};
  p.g_ptrs = g_ptrs; p.g_dtype = g_dtype; p.buf_ptrs = buf_ptrs;
  p.Y = static_cast<uint16_t*>(Y); p.ldy = ldy; p.sY = strideY;
  p.YT = static_cast<uint16_t*>(YT); p.ldyt = ldyt; p.sYT = strideYT;
  p.skip_y = Y ? 0 : 1;
  p.skip_yt = YT ? 0 : 1;
  p.partials = partials;
  p.rows = rows; p.cols = cols; p.Rp = Rp; p.Cp = Cp; p.L = batch;
  p.mu = mu; p.first_step = first_step; p.nesterov = nesterov;
  return check_launch(launch_pre(p, static_cast<hipStream_t>(stream)), who);
}

int dmuon_norm_finalize(const float* partials, int nparts, int batch, float eps, float* scale,
                        float* scale_sq, void* stream) {
  const char* who = "dmuon_norm_finalize";
  if (batch == 0) return 0;
  if (!partials || !scale || !scale_sq || nparts <= 0 || batch < 0) return fail("%s: bad arguments", who);
  return check_launch(launch_norm_finalize(partials, nparts, batch, eps, scale, scale_sq,
                                           static_cast<hipStream_t>(stream)),
                      who);
}

int dmuon_muon_update(void* const* w_ptrs, int w_dtype, const void* const* u_ptrs, int u_dtype,
                      int64_t numel, int batch, float decay, float lrs, void* stream) {
  const char* who = "dmuon_muon_update";
  if (batch == 0 || numel == 0) return 0;
  if (!w_ptrs || !u_ptrs || numel < 0 || batch < 0) return fail("%s: bad arguments", who);
  if ((w_dtype != DMUON_DTYPE_F32 && w_dtype != DMUON_DTYPE_BF16) ||
      (u_dtype != DMUON_DTYPE_F32 && u_dtype != DMUON_DTYPE_BF16))
    return fail("%s: unsupported dtype", who);
  UpdateArgs u{};
  u.w_ptrs = w_ptrs; u.w_dtype = w_dtype; u.u_ptrs = u_ptrs; u.u_dtype = u_dtype;
  u.numel = numel; u.L = batch; u.decay = decay; u.lrs = lrs;
  return check_launch(launch_update(u, static_cast<hipStream_t>(stream)), who);
}

}  // extern "C"

namespace {

int adamw_checks(const char* who, int n, int64_t total, int p_dtype, int g_dtype, bool pub,
                 int pub_dtype, float bc2_sqrt) {
  if (n < 0 || total < 0) return fail("%s: negative tensor count or size", who);
  if ((p_dtype != DMUON_DTYPE_F32 && p_dtype != DMUON_DTYPE_BF16) ||
      (g_dtype != DMUON_DTYPE_F32 && g_dtype != DMUON_DTYPE_BF16))
    return fail("%s: unsupported dtype (p %d, g %d)", who, p_dtype, g_dtype);
  if (pub && pub_dtype != DMUON_DTYPE_F32 && pub_dtype != DMUON_DTYPE_BF16)
    return fail("%s: unsupported publish dtype %d", who, pub_dtype);
  if (!(bc2_sqrt > 0.f)) return fail("%s: bias correction must be positive", who);
  return 0;
}

// read p, g, m, v; write p, m, v and the forward copy
double adamw_bytes(int64_t total, int p_dtype, int g_dtype, bool pub, int pub_dtype) {
  const int pb = p_dtype == DMUON_DTYPE_F32 ? 4 : 2, gb = g_dtype == DMUON_DTYPE_F32 ? 4 : 2;
  const double qb = pub ? (pub_dtype == DMUON_DTYPE_F32 ? 4 : 2) : 0;
  return (double)total * (6.0 * pb + gb + qb);
}

}  // namespace

extern "C" {

int dmuon_adamw_multi(const int64_t* p_ptrs, const int64_t* g_ptrs, const int64_t* m_ptrs,
                      const int64_t* v_ptrs, const int64_t* pub_ptrs, const int64_t* offsets,
                      int n, int64_t total, int p_dtype, int g_dtype, int pub_dtype, int apply_wd,
                      float wd_scale, float beta1, float alpha1, float beta2, float alpha2,
                      float bc2_sqrt, float eps, float neg_step, void* stream) {
  const char* who = "dmuon_adamw_multi";
  if (n == 0 || total == 0) return 0;
  if (n < 0 || total < 0) return fail("%s: negative tensor count or size", who);
  if (!p_ptrs || !g_ptrs || !m_ptrs || !v_ptrs || !offsets)
    return fail("%s: pointer arrays must be non-NULL", who);
  if (adamw_checks(who, n, total, p_dtype, g_dtype, pub_ptrs != nullptr, pub_dtype, bc2_sqrt))
    return 1;
  AdamWArgs a{};
  a.p_ptrs = p_ptrs; a.g_ptrs = g_ptrs; a.m_ptrs = m_ptrs; a.v_ptrs = v_ptrs;
  a.pub_ptrs = pub_ptrs; a.pub_dtype = pub_dtype;
  a.offsets = offsets; a.n = n; a.total = total;
  a.p_dtype = p_dtype; a.g_dtype = g_dtype; a.apply_wd = apply_wd != 0;
  a.wd_scale = wd_scale; a.beta1 = beta1; a.alpha1 = alpha1; a.beta2 = beta2; a.alpha2 = alpha2;
  a.bc2_sqrt = bc2_sqrt; a.eps = eps; a.neg_step = neg_step;
  hipStream_t st = static_cast<hipStream_t>(stream);
  return timed(PC_ADAMW, 0.0, adamw_bytes(total, p_dtype, g_dtype, pub_ptrs != nullptr, pub_dtype),
               st, who, [&] { return launch_adamw(a, st); });
}

int dmuon_adamw_tensors(const int64_t* table, int n, int p_dtype, int g_dtype, int pub_dtype,
                        int apply_wd, float wd_scale, float beta1, float alpha1, float beta2,
                        float alpha2, float bc2_sqrt, float eps, float neg_step, void* stream) {
  const char* who = "dmuon_adamw_tensors";
  if (n == 0) return 0;
  if (n < 0 || !table) return fail("%s: negative tensor count or NULL table", who);
  bool pub = false;
  for (int t = 0; t < n; ++t) {
    const int64_t* r = table + 6 * (int64_t)t;
    if (r[5] < 0) return fail("%s: tensor %d has a negative size", who, t);
    if (r[5] > 0 && (!r[0] || !r[1] || !r[2] || !r[3]))
      return fail("%s: tensor %d has a NULL address", who, t);
    pub = pub || r[4] != 0;
  }
  if (adamw_checks(who, n, 0, p_dtype, g_dtype, pub, pub_dtype, bc2_sqrt)) return 1;
  AdamWArgs a{};
  a.pub_dtype = pub_dtype;
  a.p_dtype = p_dtype; a.g_dtype = g_dtype; a.apply_wd = apply_wd != 0;
  a.wd_scale = wd_scale; a.beta1 = beta1; a.alpha1 = alpha1; a.beta2 = beta2; a.alpha2 = alpha2;
  a.bc2_sqrt = bc2_sqrt; a.eps = eps; a.neg_step = neg_step;
  hipStream_t st = static_cast<hipStream_t>(stream);
  AdamWTable tab;
  for (int t0 = 0; t0 < n; t0 += kAdamWTable) {
    a.n = n - t0 < kAdamWTable ? n - t0 : kAdamWTable;
    tab.off[0] = 0;
    for (int t = 0; t < a.n; ++t) {
      const int64_t* r = table + 6 * (int64_t)(t0 + t);
      tab.p[t] = r[0]; tab.g[t] = r[1]; tab.m[t] = r[2]; tab.v[t] = r[3]; tab.q[t] = r[4];
      tab.off[t + 1] = tab.off[t] + r[5];
    }
    a.total = tab.off[a.n];
    if (timed(PC_ADAMW, 0.0, adamw_bytes(a.total, p_dtype, g_dtype, pub, pub_dtype), st, who,
              [&] { return launch_adamw_table(a, tab, st); }))
      return 1;
  }
  return 0;
}

static int clip_common(const int64_t* ptrs, const int64_t* numels, const int32_t* dtypes,
                       const int32_t* segments, const int32_t* job_tensor_ids,
                       const int64_t* job_offsets, int64_t n_jobs, int64_t chunk_size,
                       const char* who, ClipArgs* a) {
  if (chunk_size <= 0) return fail("%s: chunk_size must be positive", who);
  if (n_jobs < 0 || n_jobs > 0x7fffffff) return fail("%s: job count out of range", who);
  if (n_jobs > 0 && (!ptrs || !numels || !dtypes || !segments || !job_tensor_ids || !job_offsets))
    return fail("%s: metadata arrays must be non-NULL", who);
  a->ptrs = ptrs; a->numels = numels; a->dtypes = dtypes; a->segments = segments;
  a->job_tensor_ids = job_tensor_ids; a->job_offsets = job_offsets;
  a->n_jobs = n_jobs; a->chunk = chunk_size;
  return 0;
}

int dmuon_segmented_l2_norm_sq(const int64_t* ptrs, const int64_t* numels, const int32_t* dtypes,
                               const int32_t* segments, const int32_t* job_tensor_ids,
                               const int64_t* job_offsets, int64_t n_jobs, int64_t chunk_size,
                               float* local_sq, void* stream) {
  const char* who = "dmuon_segmented_l2_norm_sq";
  ClipArgs a{};
  if (clip_common(ptrs, numels, dtypes, segments, job_tensor_ids, job_offsets, n_jobs, chunk_size,
                  who, &a))
    return 1;
  if (n_jobs == 0) return 0;
  if (!local_sq) return fail("%s: local_sq must be non-NULL", who);
  a.local_sq = local_sq;
  hipStream_t st = static_cast<hipStream_t>(stream);
  return timed(PC_CLIP, 0.0, 0.0, st, who, [&] { return launch_clip_sumsq(a, st); });
}

int dmuon_segmented_scale(const int64_t* ptrs, const int64_t* numels, const int32_t* dtypes,
                          const int32_t* segments, const int32_t* job_tensor_ids,
                          const int64_t* job_offsets, int64_t n_jobs, int64_t chunk_size,
                          const float* coefs, void* stream) {
  const char* who = "dmuon_segmented_scale";
  ClipArgs a{};
  if (clip_common(ptrs, numels, dtypes, segments, job_tensor_ids, job_offsets, n_jobs, chunk_size,
                  who, &a))
    return 1;
  if (n_jobs == 0) return 0;
  if (!coefs) return fail("%s: coefs must be non-NULL", who);
  a.coefs = coefs;
  hipStream_t st = static_cast<hipStream_t>(stream);
  return timed(PC_CLIP, 0.0, 0.0, st, who, [&] { return launch_clip_scale(a, st); });
}

static int64_t clip_workspace(int64_t n_jobs, int64_t chunk_size, int n_tensors) {
  return 8 * (int64_t)n_tensors + 4 * n_jobs * clip_pieces(n_jobs, chunk_size);
}

int dmuon_clip_workspace_size(int64_t n_jobs, int64_t chunk_size, int n_tensors,
                              int64_t* workspace_bytes) {
  if (!workspace_bytes || n_jobs < 0 || n_jobs > 0x7fffffff || chunk_size <= 0 || n_tensors < 0)
    return fail("dmuon_clip_workspace_size: bad sizes or NULL output");
  *workspace_bytes = clip_workspace(n_jobs, chunk_size, n_tensors);
  return 0;
}

int dmuon_clip_norms(const int64_t* ptrs, const int64_t* numels, const int32_t* dtypes,
                     const int32_t* segments, const int32_t* job_tensor_ids,
                     const int64_t* job_offsets, const int32_t* first_job, int64_t n_jobs,
                     int64_t chunk_size, int n_tensors, int n_segments, double max_norm,
                     float* norms, float* coefs, uint8_t* clipped, uint8_t* found_inf,
                     void* workspace, int64_t workspace_bytes, void* stream) {
  const char* who = "dmuon_clip_norms";
  ClipArgs a{};
  if (clip_common(ptrs, numels, dtypes, segments, job_tensor_ids, job_offsets, n_jobs, chunk_size,
                  who, &a))
    return 1;
  if (n_tensors <= 0 || n_segments < 0) return fail("%s: needs tensors", who);
  if (!dtypes || !segments || !first_job || !norms || !coefs || !clipped || !found_inf)
    return fail("%s: NULL argument", who);
  const int64_t need = clip_workspace(n_jobs, chunk_size, n_tensors);
  if (!workspace || (reinterpret_cast<uintptr_t>(workspace) & 7) || workspace_bytes < need)
    return fail("%s: workspace NULL, misaligned or smaller than %lld bytes", who, (long long)need);
  ClipFinishArgs f{};
  f.tensor_sq = static_cast<double*>(workspace);
  f.partials = reinterpret_cast<const float*>(f.tensor_sq + n_tensors);
  f.first_job = first_job; f.dtypes = dtypes; f.segments = segments;
  f.n = n_tensors; f.n_segments = n_segments;
  f.pieces = clip_pieces(n_jobs, chunk_size);
  f.global = n_segments == 0;
  f.has_max = max_norm == max_norm;            // NaN: no limit
  f.max_norm = f.has_max ? (float)max_norm : 0.f;
  f.norms = norms; f.coefs = coefs; f.clipped = clipped; f.found_inf = found_inf;
  hipStream_t st = static_cast<hipStream_t>(stream);
  return timed(PC_CLIP, 0.0, 0.0, st, who, [&] { return launch_clip_norms(a, f, st); });
}

int dmuon_ns_plan(int rows, int cols, int batch, int tile_req, int num_cus, int backend,
                  int* tile, int* m_pad, int* n_pad, int64_t* workspace_bytes) {
  if (!tile || !m_pad || !n_pad || !workspace_bytes) return fail("dmuon_ns_plan: NULL output");
  if (backend != DMUON_NS_DIRECT && backend != DMUON_NS_GRAM)
    return fail("dmuon_ns_plan: unknown NS backend %d", backend);
  return plan(rows, cols, batch, tile_req, num_cus, backend == DMUON_NS_GRAM, tile, m_pad, n_pad,
              workspace_bytes);
}

// The one group of the single-group entry points.
static Group one_group(void* const* g_ptrs, int g_dtype, float* const* buf_ptrs,
                       float* const* est_ptrs, void* const* w_ptrs, int w_dtype,
                       void* const* pub_ptrs, int pub_dtype, int rows, int cols, int batch,
                       int n_transposed, int first_step, double lr) {
  Group g{};
  g.g_ptrs = g_ptrs; g.g_dtype = g_dtype;
  g.buf_ptrs = buf_ptrs; g.est_ptrs = est_ptrs;
  g.w_ptrs = w_ptrs; g.w_dtype = w_dtype;
  g.pub_ptrs = pub_ptrs; g.pub_dtype = pub_dtype;
  g.rows = rows; g.cols = cols; g.batch = batch; g.n_t = n_transposed;
  g.first_step = first_step;
  g.lrs = update_scale(lr, rows, cols);
  return g;
}

int dmuon_muon_step_group(void* const* g_ptrs, int g_dtype, float* const* buf_ptrs,
                          float* const* est_ptrs, void* const* w_ptrs, int w_dtype,
                          void* const* pub_ptrs, int pub_dtype, int rows, int cols, int batch,
                          int n_transposed, double lr, double mu, double wd, int nesterov,
                          int first_step,
                          const float* coeffs, int T, int backend, const int* restarts,
                          int n_restarts, float eps, void* workspace, int64_t workspace_bytes,
                          int tile, void* stream) {
  const char* who = "dmuon_muon_step_group";
  if (batch == 0) return 0;
  if (!buf_ptrs || !w_ptrs) return fail("%s: buf_ptrs and w_ptrs must be non-NULL", who);
  Group g = one_group(g_ptrs, g_dtype, buf_ptrs, est_ptrs, w_ptrs, w_dtype, pub_ptrs, pub_dtype,
                      rows, cols, batch, n_transposed, first_step, lr);
  Call c{&g, 1, 0, static_cast<hipStream_t>(stream), who};
  return run_groups(c, (float)mu, nesterov, decay_of(lr, wd), coeffs, T, backend, restarts,
                    n_restarts, eps, workspace, workspace_bytes, tile);
}

int dmuon_muon_step_group_noalloc(void* const* g_ptrs, int g_dtype, float* const* buf_ptrs,
                                  float* const* est_ptrs, void* const* w_ptrs, int w_dtype,
                                  void* const* pub_ptrs, int pub_dtype, int rows, int cols,
                                  int batch, int n_transposed, double lr, double mu, double wd,
                                  int nesterov,
                                  int first_step, const float* coeffs, int T, int backend,
                                  const int* restarts, int n_restarts, float eps, int tile,
                                  void* stream) {
  const char* who = "dmuon_muon_step_group_noalloc";
  if (batch == 0) return 0;
  if (!buf_ptrs || !w_ptrs) return fail("%s: buf_ptrs and w_ptrs must be non-NULL", who);
  if (backend != DMUON_NS_DIRECT && backend != DMUON_NS_GRAM)
    return fail("%s: unknown NS backend %d", who, backend);
  int t, mp, np_;
  int64_t need;
  if (plan(rows, cols, batch, tile, 0, backend == DMUON_NS_GRAM, &t, &mp, &np_, &need)) return 1;
  if (need > kScratchBytes)
    return fail("%s: this group needs %lld bytes of scratch, more than the %lld bytes the "
                "entry point holds per GPU; split the group or use dmuon_muon_step_group with "
                "a workspace", who, (long long)need, (long long)kScratchBytes);
  void* ws = nullptr;
  if (scratch_of_current_device(who, &ws, true, static_cast<hipStream_t>(stream))) return 1;
  NoEvents no_events;
  Group g = one_group(g_ptrs, g_dtype, buf_ptrs, est_ptrs, w_ptrs, w_dtype, pub_ptrs, pub_dtype,
                      rows, cols, batch, n_transposed, first_step, lr);
  Call c{&g, 1, 0, static_cast<hipStream_t>(stream), who};
  return run_groups(c, (float)mu, nesterov, decay_of(lr, wd), coeffs, T, backend, restarts,
                    n_restarts, eps, ws, kScratchBytes, tile);
}

int dmuon_noalloc_init(void** scratch_out, int64_t* scratch_bytes) {
  void* p = nullptr;
  if (scratch_of_current_device("dmuon_noalloc_init", &p)) return 1;
  if (scratch_out) *scratch_out = p;
  if (scratch_bytes) *scratch_bytes = kScratchBytes;
  return 0;
}

int dmuon_newton_schulz_group(void* const* g_ptrs, int g_dtype, void* const* out_ptrs,
                              int out_dtype, int rows, int cols, int batch, int n_transposed,
                              const float* coeffs,
                              int T, int backend, const int* restarts, int n_restarts, float eps,
                              void* workspace, int64_t workspace_bytes, int tile, void* stream) {
  const char* who = "dmuon_newton_schulz_group";
  if (batch == 0) return 0;
  if (!out_ptrs) return fail("%s: out_ptrs must be non-NULL", who);
  Group g = one_group(g_ptrs, g_dtype, nullptr, nullptr, nullptr, 0, nullptr, 0, rows, cols, batch,
                      n_transposed, 1, 0.0);
  g.out_ptrs = out_ptrs; g.out_dtype = out_dtype;
  Call c{&g, 1, 0, static_cast<hipStream_t>(stream), who};
  return run_groups(c, 0.f, 0, 1.f, coeffs, T, backend, restarts, n_restarts, eps, workspace,
                    workspace_bytes, tile);
}

int dmuon_newton_schulz_matrices(const void* const* g, int g_dtype, void* const* out,
                                 int out_dtype, int rows, int cols, int batch,
                                 const float* coeffs, int T, int backend, const int* restarts,
                                 int n_restarts, float eps, void* workspace,
                                 int64_t workspace_bytes, int tile, void* stream) {
  const char* who = "dmuon_newton_schulz_matrices";
  if (batch == 0) return 0;
  if (batch < 0 || !g || !out) return fail("%s: NULL address table or negative batch", who);
  const int64_t words = align256(16 * (int64_t)batch);
  if (!workspace || !aligned16(workspace) || workspace_bytes < words)
    return fail("%s: workspace NULL, misaligned or too small", who);
  for (int l = 0; l < batch; ++l)
    if (!g[l] || !out[l]) return fail("%s: NULL matrix address", who);
  int64_t* dev = static_cast<int64_t*>(workspace);
  hipStream_t st = static_cast<hipStream_t>(stream);
  TableWords t;
  for (int w0 = 0; w0 < 2 * batch; w0 += kTableWords) {
    const int nw = 2 * batch - w0 < kTableWords ? 2 * batch - w0 : kTableWords;
    for (int w = 0; w < nw; ++w) {
      const int l = w0 + w;
      t.w[w] = (int64_t)(l < batch ? reinterpret_cast<intptr_t>(g[l])
                                   : reinterpret_cast<intptr_t>(out[l - batch]));
    }
    if (check_launch(launch_write_table(t, nw, dev + w0, st), who)) return 1;
  }
  return dmuon_newton_schulz_group(reinterpret_cast<void* const*>(dev), g_dtype,
                                   reinterpret_cast<void* const*>(dev + batch), out_dtype, rows,
                                   cols, batch, 0, coeffs, T, backend, restarts, n_restarts, eps,
                                   static_cast<char*>(workspace) + words, workspace_bytes - words,
                                   tile, stream);
}

int dmuon_muon_stage_group(void* const* g_ptrs, int g_dtype, float* const* buf_ptrs,
                           float* const* est_ptrs, int rows, int cols, int batch,
                           int n_transposed, double mu, int nesterov, int first_step,
                           int backend, float eps, void* workspace, int64_t workspace_bytes,
                           int tile, void* stream) {
  const char* who = "dmuon_muon_stage_group";
  if (batch == 0) return 0;
  if (!buf_ptrs) return fail("%s: buf_ptrs must be non-NULL", who);
  Group g = one_group(g_ptrs, g_dtype, buf_ptrs, est_ptrs, nullptr, 0, nullptr, 0, rows, cols,
                      batch, n_transposed, first_step, 0.0);
  Call c{&g, 1, 0, static_cast<hipStream_t>(stream), who};
  return run_groups(c, (float)mu, nesterov, 1.f, nullptr, 0, backend, nullptr, 0, eps, workspace,
                    workspace_bytes, tile, PH_STAGE);
}

int dmuon_muon_apply_group(void* const* w_ptrs, int w_dtype, void* const* pub_ptrs,
                           int pub_dtype, int rows, int cols, int batch, int n_transposed,
                           double lr, double wd,
                           const float* coeffs, int T, int backend, const int* restarts,
                           int n_restarts, void* workspace, int64_t workspace_bytes, int tile,
                           void* stream) {
  const char* who = "dmuon_muon_apply_group";
  if (batch == 0) return 0;
  if (!w_ptrs) return fail("%s: w_ptrs must be non-NULL", who);
  Group g = one_group(nullptr, 0, nullptr, nullptr, w_ptrs, w_dtype, pub_ptrs, pub_dtype, rows,
                      cols, batch, n_transposed, 0, lr);
  Call c{&g, 1, 0, static_cast<hipStream_t>(stream), who};
  return run_groups(c, 0.f, 0, decay_of(lr, wd), coeffs, T, backend, restarts, n_restarts, 0.f,
                    workspace, workspace_bytes, tile, PH_APPLY);
}

// The groups of a several-shapes entry point, from the caller's descriptors.
static int caller_groups(const char* who, const dmuon_muon_group* groups, int n, double lr,
                         Group* out) {
  if (n < 1 || n > DMUON_MAX_GROUPS || !groups)
    return fail("%s: needs 1 .. %d groups, got %d", who, DMUON_MAX_GROUPS, n);
  for (int i = 0; i < n; ++i) {
    const dmuon_muon_group& d = groups[i];
    out[i] = one_group(d.g_ptrs, d.g_dtype, d.buf_ptrs, d.est_ptrs, d.w_ptrs, d.w_dtype,
                       d.pub_ptrs, d.pub_dtype, d.rows, d.cols, d.batch, d.n_transposed,
                       d.first_step, lr);
  }
  return 0;
}
static_assert(DMUON_MAX_GROUPS == kMaxGroups, "groups of a call and of a launch");

int dmuon_muon_plan_groups(const dmuon_muon_group* groups, int n, int tile, int num_cus,
                           int backend, int* tile_out, int64_t* workspace_bytes,
                           double* cost_us) {
  const char* who = "dmuon_muon_plan_groups";
  if (!groups || n < 1 || n > DMUON_MAX_GROUPS)
    return fail("%s: needs 1 .. %d groups, got %d", who, DMUON_MAX_GROUPS, n);
  if (!tile_out || !workspace_bytes) return fail("%s: NULL output", who);
  if (backend != DMUON_NS_DIRECT && backend != DMUON_NS_GRAM)
    return fail("%s: unknown NS backend %d", who, backend);
  return plan_groups(groups, n, tile, num_cus, backend == DMUON_NS_GRAM, tile_out,
                     workspace_bytes, cost_us);
}

int dmuon_muon_stage_groups(const dmuon_muon_group* groups, int n, double mu, int nesterov,
                            int backend, float eps, void* workspace, int64_t workspace_bytes,
                            int tile, void* stream) {
  const char* who = "dmuon_muon_stage_groups";
  Group g[kMaxGroups];
  if (caller_groups(who, groups, n, 0.0, g)) return 1;
  for (int i = 0; i < n; ++i)
    if (!g[i].buf_ptrs) return fail("%s: buf_ptrs must be non-NULL", who);
  if (n > 1 && tile != 128 && tile != 256)
    return fail("%s: several groups need the tile of their plan (128 or 256), got %d", who, tile);
  Call c{g, n, 0, static_cast<hipStream_t>(stream), who};
  return run_groups(c, (float)mu, nesterov, 1.f, nullptr, 0, backend, nullptr, 0, eps, workspace,
                    workspace_bytes, tile, PH_STAGE);
}

int dmuon_muon_apply_groups(const dmuon_muon_group* groups, int n, double lr, double wd,
                            const float* coeffs, int T, int backend, const int* restarts,
                            int n_restarts, void* workspace, int64_t workspace_bytes, int tile,
                            void* stream) {
  const char* who = "dmuon_muon_apply_groups";
  Group g[kMaxGroups];
  if (caller_groups(who, groups, n, lr, g)) return 1;
  for (int i = 0; i < n; ++i)
    if (!g[i].w_ptrs) return fail("%s: w_ptrs must be non-NULL", who);
  if (n > 1 && tile != 128 && tile != 256)
    return fail("%s: several groups need the tile of their plan (128 or 256), got %d", who, tile);
  Call c{g, n, 0, static_cast<hipStream_t>(stream), who};
  return run_groups(c, 0.f, 0, decay_of(lr, wd), coeffs, T, backend, restarts, n_restarts, 0.f,
                    workspace, workspace_bytes, tile, PH_APPLY);
}

}  // extern "C"
