// plan.cpp -- plan builder and executor.
//
// A sub-plan is the reference's recursion (algorithms/strassen.hpp:378-659)
// unrolled level by level.  Level l holds R^l nodes, each an (A, B, C)
// operand triple plus the node's multiplier.  Every node of a level has the
// same block shape (the floor split of linalg/linalg.hpp:179-184), so each
// level is one S and one T launch over all of its nodes; the base-case
// products of every node become one grouped GEMM launch; then, deepest level
// first, one W launch and one grouped launch of the peeling products.  This
// is the reference's BFS schedule (util/par_util.hpp:17-95) with every task
// of a level in one launch.
//
// Multipliers follow the reference exactly: the root carries alpha, a
// product whose S (T) column has a single coefficient c multiplies its
// node's multiplier by c (codegen/gen.py:614-621), base-case products and
// peeling products use the node's multiplier as alpha (linalg/linalg.hpp:266,
// 201-244).  beta reaches only the root's W stage and peeling; children use
// 0 (algorithms/strassen.hpp:459).  With num_steps = 0 the root is itself
// the base case, MatMul(A, B, C) with beta 0 (algorithms/strassen.hpp:385-388).
//
// Addresses are (role, offset) pairs resolved at launch time, so a plan is
// built and uploaded once per shape and replayed for any buffers.
#include "plan.hpp"

#include <algorithm>
#include <cstring>
#include <map>
#include <tuple>

namespace fmplan {

namespace {
thread_local std::string t_err;
const int64_t kLdAlign = 16;    // elements; 128 B for FP64
const int64_t kSlabAlign = 64;  // elements; keeps every buffer 256 B aligned

struct Node {
  FmOp a, b, c;
  double mu;
  // operand produced by a two-level stage and never stored: the workspace
  // offset of its view sub-blocks (-1 when the operand is stored)
  int64_t a_views = -1, b_views = -1;
};

FmOp op_make(int role, int64_t off, int64_t ld) {
  FmOp o;
  o.role = role;
  o.pad = 0;
  o.off = off;
  o.ld = ld;
  return o;
}

FmOp op_sub(const FmOp& o, int64_t i, int64_t j) { return op_make(o.role, o.off + i + j * o.ld, o.ld); }

FmGemmDesc gdesc(FmOp a, FmOp b, FmOp c, int64_t M, int64_t N, int64_t K, double alpha,
                 double beta) {
  FmGemmDesc d;
  memset(&d, 0, sizeof(d));
  d.a = a;
  d.b = b;
  d.c = c;
  d.M = (int32_t)M;
  d.N = (int32_t)N;
  d.K = (int32_t)K;
  d.alpha = alpha;
  d.beta = beta;
  return d;
}

// Two-level S/T stage over the nodes whose operands are `ops` (blocks
// rows x cols, sub-blocks rows2 x cols2).
Launch stage2_launch(LaunchKind kind, const FmAlgDesc* alg, std::vector<FmOp> ops, int64_t rows,
                     int64_t cols, int64_t rows2, int64_t cols2, int64_t out_off, int64_t out_ld,
                     int64_t out_slab, int64_t view_off, double x) {
  Launch L;
  L.kind = kind;
  L.alg = alg;
  L.stage = kind == LK_S2 ? FM_STAGE_S : kind == LK_T2 ? FM_STAGE_T : FM_STAGE_W;
  L.st.rows = (int32_t)rows;
  L.st.cols = (int32_t)cols;
  L.st.rows2 = (int32_t)rows2;
  L.st.cols2 = (int32_t)cols2;
  L.st.nodes = (int32_t)ops.size();
  L.st.out_off = out_off;
  L.st.out_ld = out_ld;
  L.st.out_slab = out_slab;
  L.st.view_off = view_off;
  L.st.x = x;
  L.st.beta = 0.0;
  L.vec_ok = 1;
  L.ops = std::move(ops);
  return L;
}

Launch stage_launch(fm_dtype dt, LaunchKind kind, const FmAlgDesc* alg, std::vector<FmOp> ops,
                    int64_t rows, int64_t cols, int64_t out_off, int64_t out_ld, int64_t out_slab,
                    double x, double beta) {
  Launch L;
  L.kind = kind;
  L.alg = alg;
  L.stage = kind == LK_S ? FM_STAGE_S : kind == LK_T ? FM_STAGE_T : FM_STAGE_W;
  L.st.rows = (int32_t)rows;
  L.st.cols = (int32_t)cols;
  L.st.nodes = (int32_t)ops.size();
  L.st.out_off = out_off;
  L.st.out_ld = out_ld;
  L.st.out_slab = out_slab;
  L.st.x = x;
  L.st.beta = beta;
  const int vmax = dt == FM_F64 ? 2 : 4;
  bool ok = rows % vmax == 0 && out_ld % vmax == 0 && out_slab % vmax == 0 && out_off % vmax == 0;
  for (const FmOp& o : ops) ok = ok && o.off % vmax == 0 && o.ld % vmax == 0;
  L.vec_ok = ok ? vmax : 1;
  L.ops = std::move(ops);
  return L;
}

// Peeling products of one node (linalg/linalg.hpp:201-244).  Strips wider than the
// thin kernels take (remainders of a split into more than FM_THIN_MAX + 1 blocks)
// are several products.
void peel_descs(const Node& nd, const Dims& D, int am, int ak, int an, double beta,
                std::vector<FmThinDesc>& out) {
  const int64_t erA = D.m % am, ecA = D.k % ak, ecB = D.n % an;
  auto mk = [&](FmThinKind kind, FmOp a, FmOp b, FmOp c, int64_t M, int64_t N, int64_t K, double bta) {
    if (M <= 0 || N <= 0) return;
    FmThinDesc d;
    memset(&d, 0, sizeof(d));
    d.a = a;
    d.b = b;
    d.c = c;
    d.M = (int32_t)M;
    d.N = (int32_t)N;
    d.K = (int32_t)K;
    d.kind = kind;
    d.alpha = nd.mu;
    d.beta = bta;
    out.push_back(d);
  };
  if (ecA > 0) {
    const int64_t row_dim = D.m - erA, col_dim = D.n - ecB, kk = D.k - ecA;
    mk(FM_THIN_K, op_sub(nd.a, 0, kk), op_sub(nd.b, kk, 0), nd.c, row_dim, col_dim, ecA, 1.0);
  }
  if (ecB > 0) {
    for (int64_t s = D.n - ecB; s < D.n; s += FM_THIN_MAX)
      mk(FM_THIN_N, nd.a, op_sub(nd.b, 0, s), op_sub(nd.c, 0, s), D.m, std::min<int64_t>(D.n - s, FM_THIN_MAX), D.k,
         beta);
  }
  if (erA > 0) {
    const int64_t nc = D.n - ecB;
    for (int64_t s = D.m - erA; s < D.m; s += FM_THIN_MAX)
      mk(FM_THIN_M, op_sub(nd.a, s, 0), nd.b, op_sub(nd.c, s, 0), std::min<int64_t>(D.m - s, FM_THIN_MAX), nc, D.k,
         beta);
  }
}

// One launch of peeling products, ordered by kind.  The products of one
// problem's level have one shape per kind, so a tile finds its product by
// division; a batch's are found by a search over tile_begin.
Launch thin_launch(std::vector<FmThinDesc> descs, fm_dtype dt) {
  std::stable_sort(descs.begin(), descs.end(),
                   [](const FmThinDesc& x, const FmThinDesc& y) { return x.kind < y.kind; });
  Launch L;
  L.kind = LK_THIN;
  L.stage = FM_STAGE_PEEL;
  L.th.uniform = 1;
  int32_t t = 0;
  size_t i = 0;
  for (int kind = 0; kind < 3; ++kind) {
    L.th.t0[kind] = t;
    L.th.d0[kind] = (int32_t)i;
    L.th.per[kind] = 1;
    const size_t first = i;
    for (; i < descs.size() && descs[i].kind == kind; ++i) {
      FmThinDesc& d = descs[i];
      int bm, bn;
      fm_thin_tile(dt == FM_F64, kind, d.K, &bm, &bn);
      d.tiles_m = (d.M + bm - 1) / bm;
      d.tile_begin = t;
      const int32_t per = d.tiles_m * ((d.N + bn - 1) / bn);
      t += per;
      L.th.per[kind] = per;
      if (d.M != descs[first].M || d.N != descs[first].N || d.K != descs[first].K) L.th.uniform = 0;
    }
  }
  L.th.ndesc = (int32_t)descs.size();
  L.th.total_tiles = t;
  L.tdescs = std::move(descs);
  return L;
}

// Every product a whole number of tiles and K slices, columns 16-byte aligned.
bool whole_tiles(fm_dtype dt, int cfg, const std::vector<FmGemmDesc>& prods) {
  if (fm_tile_planes(cfg)) return true;
  int bm, bn;
  fm_tile_dims(cfg, &bm, &bn);
  const int bk = fm_tile_bk(cfg), vl = dt == FM_F64 ? 2 : 4;
  for (const FmGemmDesc& d : prods)
    if (d.M % bm || d.N % bn || d.K % bk || d.K == 0 || d.a.off % vl || d.a.ld % vl ||
        d.b.off % vl || d.b.ld % vl)
      return false;
  return true;
}

// Every product fits the spread kernels' ANY variant: a 16-byte vector of
// rows and a whole K slice exist to load from, and the byte offsets of a
// tile's columns (two slices of A, the tile's columns of B) stay within 32
// bits.
bool any_tile(fm_dtype dt, int cfg, const FmGemmDesc& d) {
  int bm, bn;
  fm_tile_dims(cfg, &bm, &bn);
  const int64_t bk = fm_tile_bk(cfg), vl = dt == FM_F64 ? 2 : 4;
  const int64_t span = (int64_t(1) << 32) / elem_size(dt);
  return d.M >= vl && d.K >= bk && bm + 2 * bk * d.a.ld < span && 2 * bk + bn * d.b.ld < span;
}

bool any_tiles(fm_dtype dt, int cfg, const std::vector<FmGemmDesc>& prods) {
  if (!fm_tile_spread(cfg)) return false;
  for (const FmGemmDesc& d : prods)
    if (!any_tile(dt, cfg, d)) return false;
  return true;
}

bool depths_differ(const std::vector<FmGemmDesc>& prods) {
  for (const FmGemmDesc& d : prods)
    if (d.K != prods[0].K) return true;
  return false;
}

Launch gemm_launch(std::vector<FmGemmDesc> descs, int cfg, int stage, fm_dtype dt) {
  int bm, bn;
  fm_tile_dims(cfg, &bm, &bn);
  int32_t t = 0;
  bool uniform = true;
  for (FmGemmDesc& d : descs) {
    d.tiles_m = (int32_t)((d.M + bm - 1) / bm);
    d.tiles_n = (int32_t)((d.N + bn - 1) / bn);
    d.tile_begin = t;
    t += d.tiles_m * d.tiles_n;
    uniform = uniform && d.M == descs[0].M && d.N == descs[0].N;
  }
  Launch L;
  L.kind = LK_GEMM;
  L.stage = stage;
  L.gm.ndesc = (int32_t)descs.size();
  L.gm.total_tiles = t;
  L.gm.uniform = uniform ? 1 : 0;
  // The unpredicated whole-tile kernel needs every product whole and its
  // A/B column starts 16-byte aligned (the base pointers are checked at
  // launch); the spread kernels' ANY variant takes the others.
  L.vec_ok = 1;
  L.gm.chunk = depths_differ(descs) ? FM_XCD_CHUNK : 0;
  L.gm.full = whole_tiles(dt, cfg, descs) ? 1 : 0;
  L.gm.any = any_tiles(dt, cfg, descs) ? 1 : 0;
  L.cfg = cfg;
  L.gdescs = std::move(descs);
  return L;
}

// Leaf products on int8 digits: descriptors plus digit-plane workspace,
// appended at byte offset *ws_bytes (advanced).
fm_status ozaki_launch(int S, int tile, const std::vector<FmGemmDesc>& prods, size_t* ws_bytes,
                       Launch& L) {
  int32_t t = 0;
  int max_rows = 0, max_cols = 0;
  size_t off = (size_t)align_up((int64_t)*ws_bytes, 256);
  // kernel: FmTileCfg 64x64 forced selects the 16 x 16 x 64 one, 128x64
  // the 64 x 64-tile 32 x 32 x 32 one; otherwise 64 x 128 tiles of
  // 32 x 32 x 32 products (B digit planes padded to 128 columns)
  const int variant = tile == FM_TILE_64x64 ? 0 : tile == FM_TILE_128x64 ? 1 : 2;
  const int bn = variant == 2 ? 128 : 64;
  for (const FmGemmDesc& g : prods) {
    FmOzakiDesc d;
    memset(&d, 0, sizeof(d));
    d.a = g.a;
    d.b = g.b;
    d.c = g.c;
    d.M = g.M;
    d.N = g.N;
    d.K = g.K;
    d.Kp = (int32_t)align_up(g.K, 64);
    if (d.Kp > fm_ozaki_max_kp(S))
      return set_err(FM_ERR_SHAPE, "ozaki_int8: leaf K too large for exact int32 sums");
    d.rows_pad = (int32_t)align_up(g.M, 64);
    d.cols_pad = (int32_t)align_up(g.N, bn);
    d.tiles_m = d.rows_pad / 64;
    d.tiles_n = d.cols_pad / bn;
    d.tile_begin = t;
    t += d.tiles_m * d.tiles_n;
    d.alpha = g.alpha;
    d.beta = g.beta;
    d.a_slc = (int64_t)off;
    off += (size_t)S * d.rows_pad * d.Kp;
    d.b_slc = (int64_t)off;
    off += (size_t)S * d.cols_pad * d.Kp;
    d.a_exp = (int64_t)off;
    off += align_up(4 * (int64_t)d.rows_pad, 256);
    d.b_exp = (int64_t)off;
    off += align_up(4 * (int64_t)d.cols_pad, 256);
    max_rows = std::max(max_rows, d.rows_pad);
    max_cols = std::max(max_cols, d.cols_pad);
    L.odescs.push_back(d);
  }
  L.kind = LK_OZAKI;
  L.stage = FM_STAGE_LEAF;
  L.oz.ndesc = (int32_t)L.odescs.size();
  L.oz.total_tiles = t;
  L.oz.variant = variant;
  L.oz_slices = S;
  L.oz_rows = max_rows;
  L.oz_cols = max_cols;
  *ws_bytes = off;
  return FM_OK;
}

// Split-bf16 leaf products on slice planes: one preparation record per
// distinct operand (products that share an operand share its planes), the
// planes appended to the workspace at byte offset *ws_bytes (advanced).
Launch split_launch(std::vector<FmGemmDesc> prods, int cfg, size_t* ws_bytes) {
  int bm, bn;
  fm_tile_dims(cfg, &bm, &bn);
  Launch L;
  L.kind = LK_SPLIT;
  L.stage = FM_STAGE_LEAF;
  L.cfg = cfg;
  size_t off = (size_t)align_up((int64_t)*ws_bytes, 256);
  std::map<std::tuple<int, int64_t, int64_t, int, int, int>, int64_t> seen;
  int32_t prep_wgs = 0;
  auto planes = [&](const FmOp& src, int rows, int K, int pad_to, int kcontig, int32_t* plane_rows) {
    if (src.role == FM_ROLE_PLANES) {  // written by the S/T stage
      *plane_rows = (int32_t)src.ld;
      return src.off;
    }
    *plane_rows = (int32_t)align_up(rows, pad_to);
    const auto key = std::make_tuple(src.role, src.off, src.ld, rows, K, kcontig);
    auto it = seen.find(key);
    if (it != seen.end()) return it->second;
    FmSplitPrep r;
    memset(&r, 0, sizeof(r));
    r.src = src;
    r.rows = rows;
    r.K = K;
    r.rows_pad = (int32_t)align_up(rows, pad_to);
    r.Kp = (int32_t)align_up(K, 32);
    r.kcontig = kcontig;
    r.dst = (int64_t)off;
    off += (size_t)align_up((int64_t)r.rows_pad * r.Kp * 6, 256);
    r.wg_begin = prep_wgs;
    prep_wgs += fm_prep_wgs(r);
    L.spreps.push_back(r);
    seen.emplace(key, r.dst);
    return r.dst;
  };
  int32_t t = 0;
  bool uniform = true;
  for (const FmGemmDesc& g : prods) {
    FmSplitDesc d;
    memset(&d, 0, sizeof(d));
    d.c = g.c;
    d.M = g.M;
    d.N = g.N;
    d.K = g.K;
    d.Kp = (int32_t)align_up(g.K, 32);
    d.tiles_m = (g.M + bm - 1) / bm;
    d.tiles_n = (g.N + bn - 1) / bn;
    d.tile_begin = t;
    t += d.tiles_m * d.tiles_n;
    d.alpha = g.alpha;
    d.beta = g.beta;
    d.a_pl = planes(g.a, g.M, g.K, bm, 0, &d.a_rows);
    d.b_pl = planes(g.b, g.N, g.K, bn, 1, &d.b_rows);
    uniform = uniform && g.M == prods[0].M && g.N == prods[0].N;
    L.sdescs.push_back(d);
  }
  L.sp.ndesc = (int32_t)L.sdescs.size();
  L.sp.total_tiles = t;
  L.sp.uniform = uniform ? 1 : 0;
  L.sp.chunk = depths_differ(prods) ? FM_XCD_CHUNK : 0;
  L.sp.nprep = (int32_t)L.spreps.size();
  L.sp.prep_wgs = prep_wgs;
  L.sp.even_k = 1;
  for (const FmSplitDesc& d : L.sdescs)
    if ((d.Kp / 32) % 2 != 0) L.sp.even_k = 0;
  *ws_bytes = off;
  return L;
}

}  // namespace

fm_options g_defaults = {-1, 0, 0, 1, 1, 8};

fm_status check_options(const fm_options& o) {
  if (o.gemm_tile < -1 || o.gemm_tile >= FM_TILE_OPTIONS) return set_err(FM_ERR_INVALID_ARG, "unknown tile config");
  if (o.dfs_levels < -1) return set_err(FM_ERR_INVALID_ARG, "dfs_levels must be >= -1");
  if (o.stage_fusion < 0 || o.stage_fusion > 2)
    return set_err(FM_ERR_INVALID_ARG, "stage_fusion must be 0, 1 or 2");
  if (o.ozaki_slices < 6 || o.ozaki_slices > 8)
    return set_err(FM_ERR_INVALID_ARG, "ozaki_slices must be 6, 7 or 8");
  return FM_OK;
}

fm_status set_err(fm_status s, const std::string& msg) {
  t_err = msg;
  return s;
}
fm_status hip_err(hipError_t e, const char* what) {
  return set_err(FM_ERR_HIP, std::string(what) + ": " + hipGetErrorString(e));
}
const std::string& last_error() { return t_err; }
void clear_error() { t_err.clear(); }

int64_t align_up(int64_t v, int64_t a) { return (v + a - 1) / a * a; }
double round_scalar(double v, fm_dtype dt) { return dt == FM_F32 ? (double)(float)v : v; }
int elem_size(fm_dtype dt) { return dt == FM_F64 ? 8 : 4; }

// Tile of a grouped launch: smallest estimated time over the configurations.
namespace {
// Plain leaves: what one tile of a configuration costs a CU, in us on MI355X,
// measured on launches of 1 to 16 tiles per CU at K = 256 and 1024: us_k per
// unit of K and k0 units of K for its start and end, whether the CU holds one
// work group or several; and lat_k, the same for a tile that has its CU to
// itself and waits for its own loads (the small tiles).  Launches of 2 to 16 tiles
// a CU at these depths take 0.93 to 1.03 of what the figures say, on every tile.
// Whole-tile and ragged products cost the same on these kernels (FP64 128 x 128:
// 8192 x 8192 x 4096 71.7 TFLOP/s, 8190 x 8190 x 4090 70.0, 8191 x 8191 x 4091 69.7).
// edge: the predicated kernel of the same tile, for launches the spread kernels
// cannot take (M below a vector, K below a slice, columns past 32-bit offsets;
// -1: not offered).  4096 x 4096 x 15, 7 products of 4096 x 4096 x 14 and 16384 x
// 16384 x 8 on 64 x 64 tiles, on 128 x 128 ones: FP64 32.7, 213, 525 us and 32.3,
// 196, 422; FP32 24.4, 144, 319 us and 20.2, 118, 310.
// deep_k: the least K in a launch of more than kManyTiles.  There the operands
// come from HBM, and a tile of few slices costs more than the figures say: 7
// products of 150000 x 32 x N (K = 32) on 32 x 32 and on 128 x 64 tiles, N = 8 and
// 32, FP64 166, 213 and 123, 168 us, FP32 78, 91 and 68, 80; K = 64 FP64 209, 272 and
// 181, 222; K = 128 300, 387 and 301, 361, and the small tile is ahead beyond.  64 x
// 128 FP64 against 64 x 64 on 64 x K x 150000: K = 16 239 and 205 us, 32 292 and 265,
// 64 359 and 323, 256 770 and 779.
struct TileCand {
  int cfg;
  double us_k, k0, lat_k;
  int edge, deep_k;
};
const TileCand kF64Tiles[] = {{FM_TILE_PS_128x128_O2, 0.1257, 30, 0, FM_TILE_128x128_O2_U1, 0},
                              {FM_TILE_PS_128x256_W8, 0.2520, 30, 0, -1, 0},
                              {FM_TILE_PS_128x96_O2, 0.0960, 30, 0, -1, 0},
                              {FM_TILE_128x64, 0.0650, 34, 0, -1, 0},
                              {FM_TILE_64x128, 0.0645, 34, 0, -1, 65},
                              {FM_TILE_64x64, 0.0340, 32, 0.037, FM_TILE_64x64, 0},
                              {FM_TILE_PS_32x32_K32, 0.0103, 50, 0.0129, -1, 128}};
const TileCand kF32Tiles[] = {{FM_TILE_PS_128x256_W8, 0.1383, 44, 0, -1, 0},
                              {FM_TILE_PS_128x128_O2, 0.0695, 40, 0, FM_TILE_128x128_W8, 0},
                              {FM_TILE_128x64, 0.0368, 43, 0, -1, 0},
                              {FM_TILE_64x128, 0.0368, 43, 0, -1, 0},
                              {FM_TILE_64x64, 0.0192, 43, 0.0227, FM_TILE_64x64, 0},
                              {FM_TILE_PS_32x32_K32, 0.0057, 60, 0.0099, -1, 128}};
const int64_t kManyTiles = 16 * 256;  // 64 x 64 tiles: 16 per CU, the range measured

const TileCand* plain_cands(fm_dtype dt, size_t* n) {
  *n = dt == FM_F64 ? sizeof(kF64Tiles) / sizeof(kF64Tiles[0]) : sizeof(kF32Tiles) / sizeof(kF32Tiles[0]);
  return dt == FM_F64 ? kF64Tiles : kF32Tiles;
}
// a launch's own cost beside its tiles
const double kLaunchUs = 3.0;
const double kCopyBytesPerUs = 4.9e6;
// one work group to a CU: nothing covers its wait for operands that are not in
// L2 (strassen one level 2048^3 FP64: 4 of 7 leaves as 256 128 x 128 tiles and
// 3 as 64 x 64 ones 294 us, all on 64 x 64 tiles 266; one call's figure: with the
// operands in L2 such a launch takes 0.86 to 1.0 of the figures without it)
const double kAlonePenalty = 1.15;
// the predicated loop's time over the spread loop's
const double kEdgePenalty = 1.3;
// split-bf16: kernels on prepared slice planes (any shape: the planes are
// padded to whole tiles), throughput per tile area and resident work groups
// per CU
// (Strassen, two levels, 16384^3 FP32, i.e. 49 products of 4096^3, whole
// multiply: 251 TFLOP/s with B straight to registers, 232 and 229 with the
// LDS-staged 128 x 256 and 256 x 128 kernels)
struct SplitCand {
  int cfg;
  double eff;
  int per_cu;
};
const SplitCand kSplitTiles[] = {{FM_TILE_SP_128x256_BD, 1.00, 1},
                                 {FM_TILE_SP_256x128_IL, 0.92, 1},
                                 {FM_TILE_SP_128x256_IL, 0.92, 1},
                                 {FM_TILE_SP_128x128, 0.88, 2},
                                 {FM_TILE_SP_128x128_DB, 0.83, 1}};
const int kCUs = 256;

int64_t count_tiles(int cfg, const std::vector<FmGemmDesc>& prods) {
  int bm, bn;
  fm_tile_dims(cfg, &bm, &bn);
  int64_t tiles = 0;
  for (const FmGemmDesc& d : prods) tiles += (int64_t)((d.M + bm - 1) / bm) * ((d.N + bn - 1) / bn);
  return tiles;
}

// Estimated time of one launch of `prods` on candidate c (us).  Equal depths:
// the busiest CU's tiles.  Unequal depths: the CUs' mean, and half of the
// deepest tile for the end of the launch.  At least the time of the products'
// bytes (a strip reads a whole operand again), a fifth of which is not hidden
// behind the products of a compute-bound launch.
double cand_us(fm_dtype dt, const TileCand& c, const std::vector<FmGemmDesc>& prods, bool fits) {
  int bm, bn;
  fm_tile_dims(c.cfg, &bm, &bn);
  double work = 0, kmax = 0, kmin = 1e30, elems = 0;
  int64_t tiles = 0;
  for (const FmGemmDesc& d : prods) {
    const int64_t t = (int64_t)((d.M + bm - 1) / bm) * ((d.N + bn - 1) / bn);
    tiles += t;
    work += (double)t * (d.K + c.k0);
    kmax = std::max(kmax, (double)d.K);
    kmin = std::min(kmin, (double)d.K);
    elems += ((double)d.M + d.N) * d.K + (double)d.M * d.N;
  }
  const double mem = elems * elem_size(dt) / kCopyBytesPerUs;
  const double tile = c.us_k * (kmax + c.k0);
  const double busy = kmin < kmax      ? c.us_k * work / kCUs + 0.5 * tile
                      : tiles > kCUs ? tile * (double)((tiles + kCUs - 1) / kCUs)
                                     : tile * kAlonePenalty;
  const double t = std::max(busy, std::max(c.lat_k * kmax, mem)) + 0.2 * mem;
  return kLaunchUs + t * (fits ? 1.0 : kEdgePenalty);
}

bool too_shallow(const TileCand& c, const std::vector<FmGemmDesc>& prods) {
  if (c.deep_k == 0) return false;
  int depth = 0;
  for (const FmGemmDesc& d : prods) depth = std::max(depth, d.K);
  return depth < c.deep_k && count_tiles(FM_TILE_64x64, prods) > kManyTiles;
}

// The spread kernels of configuration cfg take the products.
bool spread_fits(fm_dtype dt, int cfg, const std::vector<FmGemmDesc>& prods) {
  return any_tiles(dt, cfg, prods) || whole_tiles(dt, cfg, prods);
}

// Split-bf16: rounds of per_cu work groups on each CU, in relative units.
double split_time(const SplitCand& c, int64_t tiles) {
  int bm, bn;
  fm_tile_dims(c.cfg, &bm, &bn);
  const int64_t slots = (int64_t)kCUs * c.per_cu;
  return (double)((tiles + slots - 1) / slots) * bm * bn * c.per_cu / c.eff;
}

// Best candidate for a product list and its estimated time.  The lists run
// from large tiles to small: a smaller one has to be estimated faster by
// `margin`, about what the estimates are good for.
int best_tile(fm_dtype dt, fm_mode mode, const std::vector<FmGemmDesc>& prods, double* t_out,
              double margin = 0.97) {
  int best = -1;
  double best_t = 0;
  auto offer = [&](int cfg, double t, double margin) {
    if (best < 0 || t < best_t * margin) {
      best = cfg;
      best_t = t;
    }
  };
  if (mode == FM_MODE_SPLIT_BF16) {
    for (const SplitCand& c : kSplitTiles) offer(c.cfg, split_time(c, count_tiles(c.cfg, prods)), 0.999);
  } else {
    size_t n;
    const TileCand* c = plain_cands(dt, &n);
    for (size_t i = 0; i < n; ++i) {
      if (too_shallow(c[i], prods)) continue;
      const bool fits = spread_fits(dt, c[i].cfg, prods);
      const int cfg = fits ? c[i].cfg : c[i].edge;
      if (cfg >= 0) offer(cfg, cand_us(dt, c[i], prods, fits), margin);
    }
  }
  if (t_out) *t_out = best_t;
  return best;
}

// Estimated time of `prods` on configuration cfg (negative: not a candidate)
// and the tiles one round of the launch holds.
double list_time(fm_dtype dt, fm_mode mode, int cfg, const std::vector<FmGemmDesc>& prods, int64_t* round) {
  *round = kCUs;
  if (mode == FM_MODE_SPLIT_BF16) {
    for (const SplitCand& c : kSplitTiles)
      if (c.cfg == cfg) {
        *round = (int64_t)kCUs * c.per_cu;
        return split_time(c, count_tiles(cfg, prods));
      }
    return -1;
  }
  size_t n;
  const TileCand* c = plain_cands(dt, &n);
  for (size_t i = 0; i < n; ++i)
    if (c[i].cfg == cfg || c[i].edge == cfg)
      return cand_us(dt, c[i], prods, c[i].cfg == cfg && spread_fits(dt, cfg, prods));
  return -1;
}

FmGemmDesc gsub(const FmGemmDesc& d, int64_t i0, int64_t j0, int64_t m, int64_t n) {
  return gdesc(op_sub(d.a, i0, 0), op_sub(d.b, 0, j0), op_sub(d.c, i0, j0), m, n, d.K, d.alpha,
               d.beta);
}

// One product that no spread kernel takes (a K of 8, a single row, columns past
// 32-bit offsets) would send a whole grouped launch to the predicated kernels:
// such products move to `odd`, a launch of their own, where that is estimated
// faster (63 products of 512 to 2048 a side and one of 2048 x 8 x 2048: FP64 4029 ->
// 3388 us, FP32 2244 -> 1792).  Returns the estimated time of all of them; *cfg is the tile of those
// that stay.
double set_apart(fm_dtype dt, std::vector<FmGemmDesc>& prods, std::vector<FmGemmDesc>& odd, int* cfg) {
  double t_one = 0, t_fit = 0, t_odd = 0;
  *cfg = best_tile(dt, FM_MODE_PLAIN, prods, &t_one);
  // (the widest tile: the slice depth of all but the smallest, the longest offsets)
  auto fits = [&](const FmGemmDesc& d) { return any_tile(dt, FM_TILE_PS_128x256_W8, d); };
  std::vector<FmGemmDesc> in, out;
  for (const FmGemmDesc& d : prods) (fits(d) ? in : out).push_back(d);
  if (in.empty() || out.empty()) return t_one;
  const int cfg_in = best_tile(dt, FM_MODE_PLAIN, in, &t_fit);
  (void)best_tile(dt, FM_MODE_PLAIN, out, &t_odd);
  if (t_fit + t_odd >= 0.99 * t_one) return t_one;
  prods = std::move(in);
  odd = std::move(out);
  *cfg = cfg_in;
  return t_fit + t_odd;
}

// Whole-tile carve-out: a ragged product's last tile row and column are
// partly empty.  Cutting each product into its whole-tile core and the row and
// column strips left over (a second launch, with the tile that fits them) is
// worth it when the emptiness is a large share; every output element is
// computed by the same K-ordered MFMA sequence either way.  Returns false
// (prods unchanged) when it does not pay or does not apply.
bool carve_full(const Plan& P, int cfg, std::vector<FmGemmDesc>& prods, std::vector<FmGemmDesc>& strips,
                std::vector<FmGemmDesc>& odd, int* cfg_core, int* cfg_strips) {
  if (P.tile >= 0 || P.mode != FM_MODE_PLAIN) return false;
  int64_t round;
  const double t_all = list_time(P.dtype, P.mode, cfg, prods, &round);
  size_t n;
  const TileCand* cands = plain_cands(P.dtype, &n);
  double best_t = 0.995 * t_all;
  std::vector<FmGemmDesc> core, st, st_odd, best_core, best_st, best_odd;
  for (size_t i = 0; i < n; ++i) {
    int bm, bn;
    fm_tile_dims(cands[i].cfg, &bm, &bn);
    core.clear();
    st.clear();
    st_odd.clear();
    for (const FmGemmDesc& d : prods) {
      const int64_t Mf = d.M / bm * bm, Nf = d.N / bn * bn;
      if (Mf > 0 && Nf > 0) core.push_back(gsub(d, 0, 0, Mf, Nf));
      if (d.N > Nf) st.push_back(gsub(d, 0, Nf, d.M, d.N - Nf));           // right strip, all rows
      if (d.M > Mf && Nf > 0) st.push_back(gsub(d, Mf, 0, d.M - Mf, Nf));  // bottom strip
    }
    if (core.empty() || st.empty() || too_shallow(cands[i], core)) continue;
    if (!spread_fits(P.dtype, cands[i].cfg, core)) continue;
    int cs;
    const double t_strips = set_apart(P.dtype, st, st_odd, &cs);
    const double t = cand_us(P.dtype, cands[i], core, true) + t_strips;
    if (t >= best_t) continue;
    best_t = t;
    best_core = core;
    best_st = st;
    best_odd = st_odd;
    *cfg_core = cands[i].cfg;
    *cfg_strips = cs;
  }
  if (best_core.empty()) return false;
  prods = std::move(best_core);
  strips = std::move(best_st);
  odd.insert(odd.end(), best_odd.begin(), best_odd.end());
  return true;
}
}  // namespace

// (a depth-first child changes its one launch to a smaller tile only for a
// tenth: its siblings' stages and leaves follow, and fill the machine again)
int pick_tile(const Plan& P, const std::vector<FmGemmDesc>& prods) {
  if (P.tile >= 0) return P.tile;
  return best_tile(P.dtype, P.mode, prods, nullptr, P.child ? 0.90 : 0.97);
}

// The GPU form of the reference's HYBRID remainder rule (util/par_util.hpp:
// 65-95: leaf tasks that do not fill the last round of threads run one at a
// time on all threads): when the products' tiles leave the last round of
// work groups part-empty, the products of that round move to a second
// launch with the tile that finishes them soonest.  Products stay whole, so
// every output element is computed by the same instructions either way.
void split_remainder(const Plan& P, int cfg, std::vector<FmGemmDesc>& prods,
                     std::vector<FmGemmDesc>& rest, int* cfg_rest) {
  if (P.tile >= 0 || P.mode == FM_MODE_OZAKI_INT8) return;
  int64_t round;
  const double t_one = list_time(P.dtype, P.mode, cfg, prods, &round);
  if (t_one < 0) return;
  const int64_t total = count_tiles(cfg, prods);
  const int64_t full = total / round * round;
  if (full == 0 || full == total) return;
  // a depth-first child whose tiles are all resident at once keeps the one
  // leaf launch its schedule is documented with
  if (P.child && P.mode == FM_MODE_PLAIN && total < 2 * round) return;
  // the longest prefix of products whose tiles fill whole rounds
  int bm, bn;
  fm_tile_dims(cfg, &bm, &bn);
  int64_t acc = 0;
  size_t cut = 0;
  while (cut < prods.size()) {
    const int64_t t = (int64_t)((prods[cut].M + bm - 1) / bm) * ((prods[cut].N + bn - 1) / bn);
    if (acc + t > full) break;
    acc += t;
    ++cut;
  }
  if (acc != full || cut == prods.size()) return;
  std::vector<FmGemmDesc> tail(prods.begin() + (std::ptrdiff_t)cut, prods.end());
  std::vector<FmGemmDesc> head(prods.begin(), prods.begin() + (std::ptrdiff_t)cut);
  double t_tail = 0;
  const int cr = best_tile(P.dtype, P.mode, tail, &t_tail);
  const double t_two = list_time(P.dtype, P.mode, cfg, head, &round) + t_tail;
  if (t_two >= t_one * 0.99) return;
  prods.resize(cut);
  rest = std::move(tail);
  *cfg_rest = cr;
}

// Depth-first top level (the reference's DFS order, algorithms/strassen.hpp:
// 404-463): the level-0 S/T stages, then each child's whole sub-plan in turn
// (its own stages, leaf launch and W stages), every child reusing one
// workspace region, then the level-0 W stage and peeling.  Arithmetic is
// that of the breadth-first plan; only the launch order and the workspace
// differ.
fm_status build_dfs(fm_dtype dt, const Problem& p, const std::vector<Dims>& dims, int64_t ws_base,
                    SubPlan& out) {
  const FmAlgDesc* alg = p.alg;
  const int R = alg->R, NS = alg->ns, NT = alg->nt;
  const FmOp A0 = op_make(p.role_a, p.off_a, p.lda), B0 = op_make(p.role_b, p.off_b, p.ldb),
             C0 = op_make(p.role_c, p.off_c, p.ldc);
  const Dims c = dims[1];
  const int64_t s_ld = align_up(c.m, kLdAlign), s_slab = align_up(s_ld * c.k, kSlabAlign);
  const int64_t t_ld = align_up(c.k, kLdAlign), t_slab = align_up(t_ld * c.n, kSlabAlign);
  const int64_t m_ld = align_up(c.m, kLdAlign), m_slab = align_up(m_ld * c.n, kSlabAlign);
  int64_t ws = ws_base;
  const int64_t s_off = ws;
  ws += NS * s_slab;
  const int64_t t_off = ws;
  ws += NT * t_slab;
  const int64_t m_off = ws;
  ws += R * m_slab;
  if (NS > 0)
    out.pre.push_back(stage_launch(dt, LK_S, alg, {A0}, c.m, c.k, s_off, s_ld, s_slab, p.x, 0.0));
  if (NT > 0)
    out.pre.push_back(stage_launch(dt, LK_T, alg, {B0}, c.k, c.n, t_off, t_ld, t_slab, p.x, 0.0));
  const int64_t child_base = ws;
  const size_t es = (size_t)elem_size(dt);
  size_t end_bytes = (size_t)ws * es;
  const double mu0 = round_scalar(p.alpha, dt);
  for (int r = 0; r < R; ++r) {
    const int ai = alg->a_index[r], bi = alg->b_index[r];
    const FmOp a = alg->a_kind[r] ? op_make(FM_ROLE_WS, s_off + ai * s_slab, s_ld)
                                  : op_sub(A0, (ai / alg->k) * c.m, (ai % alg->k) * c.k);
    const FmOp b = alg->b_kind[r] ? op_make(FM_ROLE_WS, t_off + bi * t_slab, t_ld)
                                  : op_sub(B0, (bi / alg->n) * c.k, (bi % alg->n) * c.n);
    Problem q = p;
    q.steps = p.steps - 1;
    q.dfs = p.dfs - 1;
    q.fuse_planes = false;
    q.m = c.m;
    q.k = c.k;
    q.n = c.n;
    q.role_a = a.role;
    q.off_a = a.off;
    q.lda = a.ld;
    q.role_b = b.role;
    q.off_b = b.off;
    q.ldb = b.ld;
    q.role_c = FM_ROLE_WS;
    q.off_c = m_off + r * m_slab;
    q.ldc = m_ld;
    const double mu = round_scalar(mu0 * round_scalar(alg->a_coef(r, p.x), dt), dt);
    q.alpha = round_scalar(mu * round_scalar(alg->b_coef(r, p.x), dt), dt);
    q.beta = 0.0;
    std::vector<SubPlan> child(1);
    fm_status st = build_subplan(dt, q, child_base, child[0]);
    if (st != FM_OK) return st;
    Plan seq;
    seq.dtype = dt;
    seq.mode = p.mode;
    seq.slices = p.slices;
    seq.tile = p.tile;
    seq.split_rem = p.split_rem;
    seq.child = true;
    st = assemble(seq, child, child_base + child[0].ws_elems);
    if (st != FM_OK) return st;
    for (Launch& L : seq.launches) out.pre.push_back(std::move(L));
    end_bytes = std::max(end_bytes, seq.ws_bytes);
  }
  const double bl = round_scalar(p.beta, dt);
  out.w.push_back(stage_launch(dt, LK_W, alg, {C0}, c.m, c.n, m_off, m_ld, m_slab, p.x, bl));
  out.peels.resize(1);
  peel_descs(Node{A0, B0, C0, mu0}, dims[0], alg->m, alg->k, alg->n, bl, out.peels[0]);
  out.depth = 1;
  out.leaf = dims.back();
  out.ws_elems = (int64_t)((end_bytes + es - 1) / es) - ws_base;
  return FM_OK;
}

fm_status build_subplan(fm_dtype dt, const Problem& p, int64_t ws_base, SubPlan& out) {
  out = SubPlan();
  const FmOp A0 = op_make(p.role_a, p.off_a, p.lda), B0 = op_make(p.role_b, p.off_b, p.ldb),
             C0 = op_make(p.role_c, p.off_c, p.ldc);
  if (!p.alg) {  // classical product, beta honoured (MatMul, linalg/linalg.hpp:261-269)
    out.leaves.push_back(gdesc(A0, B0, C0, p.m, p.n, p.k, round_scalar(p.alpha, dt),
                               round_scalar(p.beta, dt)));
    out.leaf = {p.m, p.k, p.n};
    return FM_OK;
  }
  const FmAlgDesc* alg = p.alg;
  const int L = p.steps;
  std::vector<Dims> dims(L + 1);
  dims[0] = {p.m, p.k, p.n};
  for (int l = 0; l < L; ++l) {
    dims[l + 1] = {dims[l].m / alg->m, dims[l].k / alg->k, dims[l].n / alg->n};
    if (dims[l + 1].m <= 0 || dims[l + 1].k <= 0 || dims[l + 1].n <= 0)
      return set_err(FM_ERR_SHAPE, "num_steps too deep for this shape: a block dimension "
                                   "reaches 0 at level " + std::to_string(l + 1));
  }
  if (p.dfs > 0 && L > 0) return build_dfs(dt, p, dims, ws_base, out);
  std::vector<std::vector<Node>> lv(L + 1);
  lv[0].push_back(Node{A0, B0, C0, round_scalar(p.alpha, dt)});
  std::vector<int64_t> m_off(L), m_ld(L), m_slab(L);
  int64_t ws = ws_base;
  const int R = alg->R, NS = alg->ns, NT = alg->nt;
  // Two-level stages: s2[l] (t2[l]) merges the S (T) stage of level l into
  // that of level l + 1.  Pairs are taken from the deepest level up (deeper
  // levels move more data); a pair needs level l + 1 free of peeling, which
  // would read the level-(l+1) operands that a two-level stage never stores.
  // w2[l]: the W stages of levels l + 1 and l run as one launch, and the
  // level-(l+1) products are never stored.
  std::vector<char> s2(L, 0), t2(L, 0), w2(L, 0);
  if (p.fuse) {
    const bool fs = (dt == FM_F64 ? alg->s2_d : alg->s2_f) != nullptr;
    const bool ft = (dt == FM_F64 ? alg->t2_d : alg->t2_f) != nullptr;
    const bool fw = (dt == FM_F64 ? alg->w2_d : alg->w2_f) != nullptr;
    for (int l = L - 2; l >= 0;) {
      const Dims c = dims[l + 1];
      if (c.m % alg->m == 0 && c.k % alg->k == 0 && c.n % alg->n == 0 && (fs || ft || fw)) {
        s2[l] = fs;
        t2[l] = ft;
        w2[l] = fw;
        l -= 2;
      } else {
        l -= 1;
      }
    }
  }
  // Split-bf16 leaves on slice planes: the two-level S (T) stage of the last
  // two levels writes the leaf operands' planes itself, padded to whole tiles of
  // every split kernel (256 rows) and whole 32-deep slices, and the preparation
  // pass covers only leaf operands that are sub-blocks of A (B).  Taken when
  // the leaves' preparation grid would fit one launch (else they split on the
  // fly, on the FP32 operands), for operands that need no padding, and for
  // padded ones
  // - of more than 128 rows and a K of one slice or more: padding then takes no
  //   more workspace than FP32 outputs with planes padded to 128 rows (leaves of
  //   65536 x 1 x 1 and 65536 x 2 x 1 took 6% and 4% more);
  // - of 2^18 elements, one wave per SIMD at 4 elements a lane: a lane forms
  //   every output of its elements in turn, and a smaller stage is that serial
  //   chain; and fewer than 2^31 with the padding, as the kernel counts them.
  // Measured, separate -> stage-written: strassen two levels 600^3 51 -> 81 us,
  // 1036^3 73 -> 94, 2048^3 211 -> 154, 3448^3 682 -> 589, 10008^3
  // 9917 -> 8710; grey424_26_206 two levels 12000^3 23222 -> 17516.
  bool s_pl = false, t_pl = false;
  if (p.fuse_planes && dt == FM_F32 && L >= 2) {
    const Dims d = dims[L];
    double leaves = 1.0;
    for (int l = 0; l < L; ++l) leaves *= R;
    const double wgs = leaves * (double)((d.m + d.n + 126) / 64) * (double)((d.k + 127) / 128);
    const bool fits = wgs <= 2147483647.0;
    const bool whole = d.m % 256 == 0 && d.n % 256 == 0 && d.k % 32 == 0;
    auto padded = [&](int64_t rows) {
      const int64_t elems = align_up(rows, 256) * align_up(d.k, 32);
      return rows > 128 && d.k >= 32 && elems >= (1 << 18) && elems < (int64_t(1) << 31);
    };
    s_pl = fits && (whole || padded(d.m)) && s2[L - 2] && alg->s2p_f != nullptr;
    t_pl = fits && (whole || padded(d.n)) && t2[L - 2] && alg->t2p_f != nullptr;
  }
  const FmOp virt = op_make(-1, 0, 0);
  for (int l = 0; l < L; ++l) {
    const Dims c = dims[l + 1];
    const int64_t Q = (int64_t)lv[l].size();
    const int64_t s_ld = align_up(c.m, kLdAlign), s_slab = align_up(s_ld * c.k, kSlabAlign);
    const int64_t t_ld = align_up(c.k, kLdAlign), t_slab = align_up(t_ld * c.n, kSlabAlign);
    // the last level's S (T) outputs and views as slice planes: bytes per
    // operand (c.m x c.k, 6 bytes an element), in FP32 workspace elements
    const bool spl = s_pl && l == L - 1, tpl = t_pl && l == L - 1;
    const int64_t s_rows = align_up(c.m, 256), t_rows = align_up(c.n, 256), pk = align_up(c.k, 32);
    const int64_t s_pb = align_up(s_rows * pk * 6, 256), t_pb = align_up(pk * t_rows * 6, 256);
    const int64_t s_step = spl ? s_pb / 4 : s_slab, t_step = tpl ? t_pb / 4 : t_slab;
    m_ld[l] = align_up(c.m, kLdAlign);
    m_slab[l] = align_up(m_ld[l] * c.n, kSlabAlign);
    const bool s_first = s2[l], s_second = l > 0 && s2[l - 1];
    const bool t_first = t2[l], t_second = l > 0 && t2[l - 1];
    const int64_t s_off = ws;
    if (!s_first) ws += Q * NS * s_step;
    const int64_t t_off = ws;
    if (!t_first) ws += Q * NT * t_step;
    const int64_t sv_off = ws;
    if (s_second) ws += Q * alg->a_nviews * s_step;
    const int64_t tv_off = ws;
    if (t_second) ws += Q * alg->b_nviews * t_step;
    m_off[l] = ws;
    if (!w2[l]) ws += Q * R * m_slab[l];
    lv[l + 1].reserve(Q * R);
    for (int64_t q = 0; q < Q; ++q) {
      Node& nd = lv[l][q];
      if (s_second && nd.a.role < 0) nd.a_views = sv_off + q * alg->a_nviews * s_step;
      if (t_second && nd.b.role < 0) nd.b_views = tv_off + q * alg->b_nviews * t_step;
      // a workspace operand, or (last level, planes) the byte offset of its planes
      auto s_op = [&](int64_t off) { return spl ? op_make(FM_ROLE_PLANES, off * 4, s_rows) : op_make(FM_ROLE_WS, off, s_ld); };
      auto t_op = [&](int64_t off) { return tpl ? op_make(FM_ROLE_PLANES, off * 4, t_rows) : op_make(FM_ROLE_WS, off, t_ld); };
      for (int r = 0; r < R; ++r) {
        Node ch;
        const int ai = alg->a_index[r], bi = alg->b_index[r];
        if (alg->a_kind[r])
          ch.a = s_first ? virt : s_op(s_off + (q * NS + ai) * s_step);
        else if (nd.a_views >= 0)
          ch.a = s_op(nd.a_views + alg->a_view_slot[ai] * s_step);
        else
          ch.a = op_sub(nd.a, (ai / alg->k) * c.m, (ai % alg->k) * c.k);
        if (alg->b_kind[r])
          ch.b = t_first ? virt : t_op(t_off + (q * NT + bi) * t_step);
        else if (nd.b_views >= 0)
          ch.b = t_op(nd.b_views + alg->b_view_slot[bi] * t_step);
        else
          ch.b = op_sub(nd.b, (bi / alg->n) * c.k, (bi % alg->n) * c.n);
        ch.c = w2[l] ? virt : op_make(FM_ROLE_WS, m_off[l] + (q * R + r) * m_slab[l], m_ld[l]);
        double mu = round_scalar(nd.mu * round_scalar(alg->a_coef(r, p.x), dt), dt);
        ch.mu = round_scalar(mu * round_scalar(alg->b_coef(r, p.x), dt), dt);
        lv[l + 1].push_back(ch);
      }
    }
    if (NS > 0 && s_second) {
      const Dims pc = dims[l];
      std::vector<FmOp> ops;
      for (const Node& nd : lv[l - 1]) ops.push_back(nd.a);
      if (spl) {
        Launch S = stage2_launch(LK_S2, alg, std::move(ops), pc.m, pc.k, c.m, c.k, s_off * 4, 0,
                                 s_pb, sv_off * 4, p.x);
        S.planes = 1;
        out.pre.push_back(std::move(S));
      } else {
        out.pre.push_back(stage2_launch(LK_S2, alg, std::move(ops), pc.m, pc.k, c.m, c.k, s_off,
                                        s_ld, s_slab, sv_off, p.x));
      }
    } else if (NS > 0 && !s_first) {
      std::vector<FmOp> ops;
      for (const Node& nd : lv[l]) ops.push_back(nd.a);
      out.pre.push_back(stage_launch(dt, LK_S, alg, std::move(ops), c.m, c.k, s_off, s_ld, s_slab,
                                     p.x, 0.0));
    }
    if (NT > 0 && t_second) {
      const Dims pc = dims[l];
      std::vector<FmOp> ops;
      for (const Node& nd : lv[l - 1]) ops.push_back(nd.b);
      if (tpl) {
        Launch T = stage2_launch(LK_T2, alg, std::move(ops), pc.k, pc.n, c.k, c.n, t_off * 4, 0,
                                 t_pb, tv_off * 4, p.x);
        T.planes = 1;
        out.pre.push_back(std::move(T));
      } else {
        out.pre.push_back(stage2_launch(LK_T2, alg, std::move(ops), pc.k, pc.n, c.k, c.n, t_off,
                                        t_ld, t_slab, tv_off, p.x));
      }
    } else if (NT > 0 && !t_first) {
      std::vector<FmOp> ops;
      for (const Node& nd : lv[l]) ops.push_back(nd.b);
      out.pre.push_back(stage_launch(dt, LK_T, alg, std::move(ops), c.k, c.n, t_off, t_ld, t_slab,
                                     p.x, 0.0));
    }
  }
  const Dims d = dims[L];
  for (const Node& nd : lv[L]) out.leaves.push_back(gdesc(nd.a, nd.b, nd.c, d.m, d.n, d.k, nd.mu, 0.0));
  out.leaf = d;
  out.w.resize(L);
  out.peels.resize(L);
  for (int l = L - 1; l >= 0; --l) {
    const Dims c = dims[l + 1];
    const double bl = l == 0 ? round_scalar(p.beta, dt) : 0.0;
    std::vector<FmOp> ops;
    for (const Node& nd : lv[l]) ops.push_back(nd.c);
    if (w2[l]) {
      // levels l + 1 and l in one launch; the level-(l+1) launch is dropped
      const Dims c2 = dims[l + 2];
      out.w[l + 1] = Launch();
      out.w[l + 1].kind = LK_NONE;
      Launch W = stage2_launch(LK_W2, alg, std::move(ops), c.m, c.n, c2.m, c2.n, m_off[l + 1],
                               m_ld[l + 1], m_slab[l + 1], 0, p.x);
      W.st.beta = bl;
      out.w[l] = std::move(W);
    } else {
      out.w[l] = stage_launch(dt, LK_W, alg, std::move(ops), c.m, c.n, m_off[l], m_ld[l],
                              m_slab[l], p.x, bl);
    }
    for (const Node& nd : lv[l]) peel_descs(nd, dims[l], alg->m, alg->k, alg->n, bl, out.peels[l]);
  }
  out.depth = L;
  out.ws_elems = ws - ws_base;
  return FM_OK;
}

namespace {
// The stage kernels walk a block's elements with 32-bit counters in a
// grid-stride loop; blocks of 2^31 elements or more are refused (only
// reachable with matrices near the device's memory size).
fm_status check_stage_size(const Launch& L) {
  if (L.kind == LK_GEMM || L.kind == LK_OZAKI || L.kind == LK_SPLIT || L.kind == LK_THIN ||
      L.kind == LK_NONE)
    return FM_OK;
  if (L.kind == LK_ST && (int64_t)L.st2.rows * L.st2.cols >= (int64_t(1) << 31))
    return set_err(FM_ERR_SHAPE, "a recursion block exceeds the stage kernels' 2^31 element limit; use more steps");
  const bool two = L.kind == LK_S2 || L.kind == LK_T2 || L.kind == LK_W2;
  const int64_t elems = two ? (int64_t)L.st.rows2 * L.st.cols2 : (int64_t)L.st.rows * L.st.cols;
  if (elems >= (int64_t(1) << 31))
    return set_err(FM_ERR_SHAPE, "a recursion block of " + std::to_string(elems) +
                                     " elements exceeds the stage kernels' 2^31 limit; use more steps");
  return FM_OK;
}
}  // namespace

namespace {
// Output slabs per node of a stage launch's layout (see FmNodeView).
void stage_slabs(const Launch& L, int* nout, int* nview) {
  const FmAlgDesc* g = L.alg;
  *nview = 0;
  switch (L.kind) {
    case LK_S: *nout = g->ns; break;
    case LK_T: *nout = g->nt; break;
    case LK_W: *nout = g->R; break;
    case LK_S2: *nout = g->R * g->ns; *nview = g->R * g->a_nviews; break;
    case LK_T2: *nout = g->R * g->nt; *nview = g->R * g->b_nviews; break;
    case LK_W2: *nout = g->R * g->R; break;
    default: *nout = 0; break;
  }
}

// One launch for stage launches of the same kind and algorithm from several
// problems (their block shapes may differ): per-node descriptors, the
// largest shape for the grid, 16-byte accesses only if every node allows
// them.  The kernels compute every node exactly as its own launch would.
Launch group_stages(std::vector<Launch>& ls, fm_dtype dt) {
  Launch G;
  const Launch& f = ls[0];
  G.kind = f.kind;
  G.alg = f.alg;
  G.stage = f.stage;
  G.st = f.st;
  G.st.rows = G.st.cols = G.st.rows2 = G.st.cols2 = 0;
  int vec = dt == FM_F64 ? 2 : 4;
  for (const Launch& L : ls) {
    int nout, nview;
    stage_slabs(L, &nout, &nview);
    vec = std::min(vec, L.vec_ok);
    G.st.rows = std::max(G.st.rows, L.st.rows);
    G.st.cols = std::max(G.st.cols, L.st.cols);
    G.st.rows2 = std::max(G.st.rows2, L.st.rows2);
    G.st.cols2 = std::max(G.st.cols2, L.st.cols2);
    for (size_t q = 0; q < L.ops.size(); ++q) {
      FmStageNode n;
      memset(&n, 0, sizeof(n));
      n.op = L.ops[q];
      n.rows = L.st.rows;
      n.cols = L.st.cols;
      n.rows2 = L.st.rows2;
      n.cols2 = L.st.cols2;
      n.out_off = L.st.out_off + (int64_t)q * nout * L.st.out_slab;
      n.out_ld = L.st.out_ld;
      n.out_slab = L.st.out_slab;
      n.view_off = L.st.view_off + (int64_t)q * nview * L.st.out_slab;
      n.x = L.st.x;
      n.beta = L.st.beta;
      G.snodes.push_back(n);
    }
  }
  G.st.nodes = (int32_t)G.snodes.size();
  G.vec_ok = vec;
  return G;
}

// Merge the stage launches of several problems: launches at the same
// position of their problems' sequences with the same kind, algorithm and
// (for W) beta class become one grouped launch; positions keep their order,
// so every problem's own stage order is kept.
void group_sequence(std::vector<std::vector<Launch>*> seqs, std::vector<Launch>& out, fm_dtype dt) {
  size_t depth = 0;
  for (auto* sq : seqs) depth = std::max(depth, sq->size());
  for (size_t i = 0; i < depth; ++i) {
    std::vector<std::pair<std::tuple<int, const FmAlgDesc*, int>, std::vector<Launch>>> groups;
    for (auto* sq : seqs) {
      if (i >= sq->size() || (*sq)[i].kind == LK_NONE) continue;
      Launch& L = (*sq)[i];
      const bool stage = L.kind == LK_S || L.kind == LK_T || L.kind == LK_W || L.kind == LK_S2 ||
                         L.kind == LK_T2 || L.kind == LK_W2;
      // A depth-first child's launches come from a plan of its own: its leaves,
      // its shared launches and its W stages that add K remainders have
      // descriptors that group_stages does not carry, and stay as they are.
      if (!stage || L.nupd > 0 || L.planes) {
        out.push_back(std::move(L));
        continue;
      }
      const auto key = std::make_tuple((int)L.kind, L.alg, L.st.beta != 0.0 ? 1 : 0);
      auto it = std::find_if(groups.begin(), groups.end(), [&](const auto& g) { return g.first == key; });
      if (it == groups.end()) {
        groups.emplace_back(key, std::vector<Launch>());
        it = groups.end() - 1;
      }
      it->second.push_back(std::move(L));
    }
    for (auto& g : groups) {
      if (g.second.size() == 1)
        out.push_back(std::move(g.second[0]));
      else
        out.push_back(group_stages(g.second, dt));
    }
  }
}
}  // namespace

namespace {
// Stages that move less than this run two to a launch (fm_st_stage, fm_w_strips,
// one element a lane): a launch of its own costs about 3 us, which these bytes
// no longer hide.  Measured, one level, whole call, apart -> together in us:
// strassen FP64 257^3 (2.4 MB of S and T) 22.6 -> 18.0, 801^3 (23 MB) 49.9 ->
// 43.6, 1201^3 (52 MB; W 32 MB) 96.7 -> 95.0, 1501^3 (81 MB; W 50 MB) 144.3 ->
// 145.3; grey522 FP64 1201^3 (63 MB; W 32 MB) 99.8 -> 92.0; smirnov333 FP32
// 1501^3 (52 MB; W 32 MB) 97.8 -> 91.0.
const double kSmallPairBytes = 64e6;  // S and T
const double kSmallWBytes = 40e6;     // W; the strips beside it likewise

double stage_bytes1(const Launch& L, fm_dtype dt) {  // one-level stages
  const FmAlgDesc* g = L.alg;
  const int slabs = L.kind == LK_S ? g->m * g->k + g->ns : L.kind == LK_T ? g->k * g->n + g->nt : g->R + g->m * g->n;
  return (double)elem_size(dt) * L.st.nodes * L.st.rows * L.st.cols * slabs;
}

// Append one problem's S/T stages, adjacent small S and T as one launch.
void append_pre(std::vector<Launch>& pre, std::vector<Launch>& out, fm_dtype dt) {
  for (size_t i = 0; i < pre.size(); ++i) {
    if (i + 1 < pre.size() && pre[i].kind == LK_S && pre[i + 1].kind == LK_T && pre[i].alg == pre[i + 1].alg &&
        stage_bytes1(pre[i], dt) + stage_bytes1(pre[i + 1], dt) <= kSmallPairBytes) {
      Launch L = std::move(pre[i]);
      Launch& T = pre[++i];
      L.kind = LK_ST;
      L.st2 = T.st;
      L.ops.insert(L.ops.end(), T.ops.begin(), T.ops.end());
      out.push_back(std::move(L));
    } else {
      out.push_back(std::move(pre[i]));
    }
  }
}

// Append one problem's W stage of a level and the level's peeling products: a
// one-level W stage adds the K remainders itself (up to the K split its kernel is
// built for), and takes the strips into its launch where both are small.
// The update saves a pass over C and costs W registers, most where K is split
// six ways (smirnov363 FP64: one wave a SIMD, three without); it was faster with
// every algorithm measured, K split 2 to 6 ways, remainders of 1 and the largest, beta
// 0 and 0.5.  Whole call, one level, update apart -> in W: smirnov363 4320 x 4321 x
// 4320 FP64 2170 -> 2110 us, FP32 1163 -> 1126, 9000 x 601 x 9000 2738 -> 2395 and 1497
// -> 1345; strassen 9000 x 601 x 9000 FP64 2108 -> 1772; 900 x 901 x 900 FP64 54.3 ->
// 47.1 (smirnov363), and the one loss, FP32 41.7 -> 42.3.
void append_w(Launch W, std::vector<FmThinDesc> peel, std::vector<Launch>& out, fm_dtype dt) {
  std::vector<FmThinDesc> strips;
  const bool adds = W.kind == LK_W && W.alg->k <= FM_THIN_MAX + 1;
  if (adds) {
    for (const FmThinDesc& d : peel)
      if (d.kind == FM_THIN_K) W.tdescs.push_back(d);
    W.nupd = (int)W.tdescs.size();  // one per node, in node order, or none
  }
  for (const FmThinDesc& d : peel)
    if (!adds || d.kind != FM_THIN_K) strips.push_back(d);
  if (strips.empty()) {
    out.push_back(std::move(W));
    return;
  }
  Launch T = thin_launch(std::move(strips), dt);
  double bytes = 0;
  for (const FmThinDesc& d : T.tdescs) bytes += (double)elem_size(dt) * ((double)d.M * d.K + (double)d.K * d.N);
  const bool k_apart = T.tdescs[0].kind == FM_THIN_K;  // it updates what W writes
  if (W.kind == LK_W && !k_apart && T.th.uniform && bytes <= kSmallWBytes && stage_bytes1(W, dt) <= kSmallWBytes) {
    W.kind = LK_WS;
    W.th = T.th;
    W.tdescs.insert(W.tdescs.end(), T.tdescs.begin(), T.tdescs.end());
    out.push_back(std::move(W));
  } else {
    out.push_back(std::move(W));
    out.push_back(std::move(T));
  }
}
}  // namespace

fm_status assemble(Plan& P, std::vector<SubPlan>& subs, int64_t ws_elems, int persistent_grid) {
  for (SubPlan& s : subs) {
    for (const Launch& L : s.pre) {
      const fm_status st = check_stage_size(L);
      if (st != FM_OK) return st;
    }
    for (const Launch& L : s.w) {
      const fm_status st = check_stage_size(L);
      if (st != FM_OK) return st;
    }
  }
  if (subs.size() > 1) {
    // several problems (a batch): one launch per stage position and kind
    std::vector<std::vector<Launch>*> seqs;
    for (SubPlan& s : subs) seqs.push_back(&s.pre);
    group_sequence(seqs, P.launches, P.dtype);
  } else {
    for (SubPlan& s : subs) append_pre(s.pre, P.launches, P.dtype);
  }
  std::vector<FmGemmDesc> leaves;
  for (SubPlan& s : subs) leaves.insert(leaves.end(), s.leaves.begin(), s.leaves.end());
  // products of unequal depth: deepest first (fm_xcd_tile)
  if (depths_differ(leaves))
    std::stable_sort(leaves.begin(), leaves.end(),
                     [](const FmGemmDesc& x, const FmGemmDesc& y) { return x.K > y.K; });
  size_t wsb = (size_t)ws_elems * elem_size(P.dtype);
  if (!leaves.empty()) {
    if (P.mode == FM_MODE_OZAKI_INT8) {
      Launch L;
      fm_status st = ozaki_launch(P.slices, P.tile, leaves, &wsb, L);
      if (st != FM_OK) return st;
      P.launches.push_back(std::move(L));
    } else {
      const bool several = persistent_grid == 0 && P.split_rem;  // leaf launches allowed
      std::vector<FmGemmDesc> rest, strips, odd;
      if (several && P.tile < 0 && P.mode == FM_MODE_PLAIN) {
        int cfg_fit;
        (void)set_apart(P.dtype, leaves, odd, &cfg_fit);
      }
      const int cfg = pick_tile(P, leaves);
      if (fm_tile_planes(cfg) && P.mode != FM_MODE_SPLIT_BF16)
        return set_err(FM_ERR_INVALID_ARG, "tile config " + std::to_string(cfg) + " is for split_bf16 leaves");
      // split_bf16 leaves off the slice planes run the in-loop kernel, which
      // has the 128 x 128, 64 x 64, 128 x 64, 64 x 128 and 128 x 128 (8-wave) tiles
      if (P.mode == FM_MODE_SPLIT_BF16 && !fm_tile_planes(cfg) && cfg != FM_TILE_128x128 &&
          cfg != FM_TILE_64x64 && cfg != FM_TILE_128x64 && cfg != FM_TILE_64x128 &&
          cfg != FM_TILE_128x128_W8)
        return set_err(FM_ERR_INVALID_ARG, "tile config " + std::to_string(cfg) +
                                               " has no split_bf16 kernel");
      int cfg_rest = cfg, cfg_main = cfg, cfg_strips = cfg;
      if (several) {
        (void)carve_full(P, cfg, leaves, strips, odd, &cfg_main, &cfg_strips);
        split_remainder(P, cfg_main, leaves, rest, &cfg_rest);
      }
      auto leaf = [&](std::vector<FmGemmDesc> prods, int c) {
        // the preparation launch is one flat grid of at most 2^31 - 1 work
        // groups (64 rows x 4 K slices each, per operand; an upper bound
        // here): beyond that the leaves split on the fly instead
        int64_t wgs = 0;
        for (const FmGemmDesc& d : prods)
          wgs += ((int64_t)d.M + d.N + 126) / 64 * ((d.K + 127) / 128);
        if (fm_tile_planes(c) && wgs > 2147483647LL) c = FM_TILE_128x128;
        if (fm_tile_planes(c)) return split_launch(std::move(prods), c, &wsb);
        return gemm_launch(std::move(prods), c, FM_STAGE_LEAF, P.dtype);
      };
      P.launches.push_back(leaf(std::move(leaves), cfg_main));
      P.launches.back().gm.grid = persistent_grid;
      P.launches.back().sp.grid = persistent_grid;
      if (!rest.empty()) P.launches.push_back(leaf(std::move(rest), cfg_rest));
      if (!strips.empty()) P.launches.push_back(leaf(std::move(strips), cfg_strips));
      if (!odd.empty()) {
        const int cfg_odd = pick_tile(P, odd);
        P.launches.push_back(leaf(std::move(odd), cfg_odd));
      }
    }
  }
  int maxd = 0;
  for (const SubPlan& s : subs) maxd = std::max(maxd, s.depth);
  for (int l = maxd - 1; l >= 0; --l) {
    std::vector<FmThinDesc> peel;
    std::vector<Launch> wl;
    for (SubPlan& s : subs) {
      if (s.depth <= l) continue;
      if (s.w[l].kind != LK_NONE) wl.push_back(std::move(s.w[l]));
      peel.insert(peel.end(), s.peels[l].begin(), s.peels[l].end());
    }
    if (wl.size() > 1) {
      // this level's W stages of every problem: grouped by kind, algorithm, beta class
      std::vector<std::vector<Launch>> one(wl.size());
      std::vector<std::vector<Launch>*> seqs;
      for (size_t i = 0; i < wl.size(); ++i) {
        one[i].push_back(std::move(wl[i]));
        seqs.push_back(&one[i]);
      }
      group_sequence(seqs, P.launches, P.dtype);
    } else if (wl.size() == 1 && subs.size() == 1) {
      append_w(std::move(wl[0]), std::move(peel), P.launches, P.dtype);
      continue;
    } else {
      for (Launch& L : wl) P.launches.push_back(std::move(L));
    }
    // peeling products are sums in the data type in every leaf mode
    if (!peel.empty()) P.launches.push_back(thin_launch(std::move(peel), P.dtype));
  }
  P.ws_bytes = wsb;
  return FM_OK;
}

Plan::~Plan() {
  if (dbuf) (void)hipFree(dbuf);
}

// Descriptors and the role table, packed into one host buffer; each
// launch records its offsets in it.
void Plan::pack(std::vector<char>& buf) {
  buf.clear();
  auto put = [&](const void* src, size_t bytes) {
    const size_t off = (size_t)align_up((int64_t)buf.size(), 256);
    buf.resize(off + bytes);
    if (bytes) memcpy(buf.data() + off, src, bytes);
    return off;
  };
  for (Launch& L : launches) {
    if (L.kind == LK_GEMM)
      L.dev_off = put(L.gdescs.data(), L.gdescs.size() * sizeof(FmGemmDesc));
    else if (L.kind == LK_OZAKI)
      L.dev_off = put(L.odescs.data(), L.odescs.size() * sizeof(FmOzakiDesc));
    else if (L.kind == LK_THIN)
      L.dev_off = put(L.tdescs.data(), L.tdescs.size() * sizeof(FmThinDesc));
    else if (L.kind == LK_SPLIT) {
      L.dev_off = put(L.sdescs.data(), L.sdescs.size() * sizeof(FmSplitDesc));
      L.dev_off2 = put(L.spreps.data(), L.spreps.size() * sizeof(FmSplitPrep));
    } else if (!L.snodes.empty())
      L.dev_off = put(L.snodes.data(), L.snodes.size() * sizeof(FmStageNode));
    else {
      L.dev_off = put(L.ops.data(), L.ops.size() * sizeof(FmOp));
      if (!L.tdescs.empty()) L.dev_off2 = put(L.tdescs.data(), L.tdescs.size() * sizeof(FmThinDesc));
    }
  }
  ext_off = put(ext.data(), ext.size() * sizeof(void*));
}

// Point every launch at its descriptors in a device copy of the packed buffer.
void Plan::bind(void* dev) {
  desc_base = dev;
  for (Launch& L : launches) {
    char* p = (char*)dev + L.dev_off;
    if (L.kind == LK_GEMM)
      L.gm.descs = reinterpret_cast<const FmGemmDesc*>(p);
    else if (L.kind == LK_OZAKI)
      L.oz.descs = reinterpret_cast<const FmOzakiDesc*>(p);
    else if (L.kind == LK_THIN)
      L.th.descs = reinterpret_cast<const FmThinDesc*>(p);
    else if (L.kind == LK_SPLIT) {
      L.sp.descs = reinterpret_cast<const FmSplitDesc*>(p);
      L.sp.preps = reinterpret_cast<const FmSplitPrep*>((char*)dev + L.dev_off2);
    } else if (!L.snodes.empty()) {
      L.st.node = reinterpret_cast<const FmStageNode*>(p);
      L.st.ops = nullptr;
    } else {
      L.st.ops = reinterpret_cast<const FmOp*>(p);
      L.st.node = nullptr;
      if (L.kind == LK_ST) {
        L.st2.ops = L.st.ops + L.st.nodes;
        L.st2.node = nullptr;
      }
      const FmThinDesc* t = reinterpret_cast<const FmThinDesc*>((char*)dev + L.dev_off2);
      L.st.upd = L.nupd > 0 ? t : nullptr;
      L.th.descs = t + L.nupd;
    }
  }
}

fm_status Plan::upload() {
  std::vector<char> buf;
  pack(buf);
  if (buf.empty()) return FM_OK;
  hipError_t e = hipMalloc(&dbuf, buf.size());
  if (e != hipSuccess) {
    dbuf = nullptr;
    return hip_err(e, "hipMalloc(plan)");
  }
  e = hipMemcpy(dbuf, buf.data(), buf.size(), hipMemcpyHostToDevice);
  if (e != hipSuccess) return hip_err(e, "hipMemcpy(plan)");
  bind(dbuf);
  return FM_OK;
}

// ---- profiling ---------------------------------------------------------------
namespace {
struct ProfRec {
  int stage;
  hipEvent_t e0, e1;
  int second = -1;  // the other stage of a shared launch: counted, its time is stage's
};
std::vector<ProfRec> g_prof_pending;
std::vector<hipEvent_t> g_event_pool;
fm_profile g_prof_acc;

hipEvent_t pool_event() {
  if (!g_event_pool.empty()) {
    hipEvent_t e = g_event_pool.back();
    g_event_pool.pop_back();
    return e;
  }
  hipEvent_t e = nullptr;
  if (hipEventCreate(&e) != hipSuccess) return nullptr;
  return e;
}
}  // namespace

bool g_prof_on = false;

fm_status profile_read(fm_profile* out) {
  fm_status st = FM_OK;
  for (ProfRec& r : g_prof_pending) {
    float ms = 0.f;
    hipError_t e = hipEventSynchronize(r.e1);
    if (e == hipSuccess) e = hipEventElapsedTime(&ms, r.e0, r.e1);
    if (e != hipSuccess && st == FM_OK) st = hip_err(e, "profile event");
    g_prof_acc.ms[r.stage] += ms;
    g_prof_acc.launches[r.stage] += 1;
    if (r.second >= 0) g_prof_acc.launches[r.second] += 1;
    g_event_pool.push_back(r.e0);
    g_event_pool.push_back(r.e1);
  }
  g_prof_pending.clear();
  if (out) *out = g_prof_acc;
  memset(&g_prof_acc, 0, sizeof(g_prof_acc));
  return st;
}

fm_status Plan::run(const void* A, const void* B, void* C, void* ws, hipStream_t s) const {
  FmBases bases;
  bases.p[FM_ROLE_A] = const_cast<void*>(A);
  bases.p[FM_ROLE_B] = const_cast<void*>(B);
  bases.p[FM_ROLE_C] = C;
  bases.p[FM_ROLE_WS] = ws;
  bases.ext = ext.empty() ? nullptr : reinterpret_cast<void* const*>((char*)desc_base + ext_off);
  bool aligned = true;
  for (int i = 0; i < 4; ++i) aligned = aligned && ((uintptr_t)bases.p[i] % 16 == 0);
  for (void* p : ext) aligned = aligned && ((uintptr_t)p % 16 == 0);
  for (const Launch& L : launches) {
    hipError_t e = hipSuccess;
    ProfRec pr{L.stage, nullptr, nullptr};
    if (L.kind == LK_ST) pr.second = FM_STAGE_T;
    if (L.kind == LK_WS) pr.second = FM_STAGE_PEEL;
    if (g_prof_on) {
      pr.e0 = pool_event();
      pr.e1 = pool_event();
      if (pr.e0) (void)hipEventRecord(pr.e0, s);
    }
    if (L.kind == LK_SPLIT && ((uintptr_t)ws % 16 != 0))
      return set_err(FM_ERR_INVALID_ARG, "split_bf16 leaves need a 16-byte aligned workspace");
    if (L.kind == LK_OZAKI || L.kind == LK_SPLIT) {
      // profiled: the plane preparation and the products are timed apart
      // (preparation as FM_STAGE_PREP)
      auto go = [&](int phases) {
        if (L.kind == LK_OZAKI) {
          FmOzakiArgs o = L.oz;
          o.bases = bases;
          return fm_ozaki_launch(L.oz_slices, o, L.oz_rows, L.oz_cols, phases, s);
        }
        FmSplitArgs a = L.sp;
        a.bases = bases;
        return fm_split_launch(L.cfg, a, phases, s);
      };
      if (g_prof_on && pr.e0 && pr.e1) {
        e = go(FM_PHASE_PREP);
        (void)hipEventRecord(pr.e1, s);
        g_prof_pending.push_back(ProfRec{FM_STAGE_PREP, pr.e0, pr.e1});
        pr.e0 = pool_event();
        pr.e1 = pool_event();
        if (pr.e0) (void)hipEventRecord(pr.e0, s);
        if (e == hipSuccess) e = go(FM_PHASE_PRODUCT);
      } else {
        e = go(FM_PHASE_ALL);
      }
    } else if (L.kind == LK_THIN) {
      FmThinArgs t = L.th;
      t.bases = bases;
      e = fm_thin_launch(dtype == FM_F64, t, s);
    } else if (L.kind == LK_GEMM) {
      FmGemmArgs g = L.gm;
      g.bases = bases;
      g.vec = (L.vec_ok && aligned) ? 1 : 0;
      if (mode == FM_MODE_SPLIT_BF16)
        e = fm_gemm_launch_bf16x3(L.cfg, g, s);
      else
        e = dtype == FM_F64 ? fm_gemm_launch_f64(L.cfg, g, s) : fm_gemm_launch_f32(L.cfg, g, s);
    } else if (L.kind == LK_ST) {
      FmStageArgs a = L.st, b = L.st2;
      a.bases = b.bases = bases;
      e = (dtype == FM_F64 ? L.alg->st_d : L.alg->st_f)(a, b, s);
    } else if (L.kind == LK_WS) {
      FmStageArgs a = L.st;
      FmThinArgs t = L.th;
      a.bases = t.bases = bases;
      e = (dtype == FM_F64 ? L.alg->ws_d : L.alg->ws_f)(a, t, s);
    } else {
      FmStageArgs a = L.st;
      a.bases = bases;
      a.vec = aligned ? L.vec_ok : 1;
      const FmAlgDesc* g = L.alg;
      FmStageLaunch fn;
      const bool d = dtype == FM_F64;
      switch (L.kind) {
        case LK_S: fn = d ? g->s_d : g->s_f; break;
        case LK_T: fn = d ? g->t_d : g->t_f; break;
        case LK_S2: fn = d ? g->s2_d : L.planes ? g->s2p_f : g->s2_f; break;
        case LK_T2: fn = d ? g->t2_d : L.planes ? g->t2p_f : g->t2_f; break;
        case LK_W2: fn = d ? g->w2_d : g->w2_f; break;
        default: fn = d ? g->w_d : g->w_f; break;
      }
      e = fn(a, s);
    }
    if (g_prof_on && pr.e0 && pr.e1) {
      (void)hipEventRecord(pr.e1, s);
      g_prof_pending.push_back(pr);
    }
    if (e != hipSuccess) return hip_err(e, "kernel launch");
  }
  return FM_OK;
}

}  // namespace fmplan
