// Kernel formation for contractions on the matrix cores: operand layouts, f32 repacks, grouped
// launches of one activation's projections, fused epilogues (lookup tables included) and the
// elementwise mul + sum spelling.
#include <algorithm>

#include "planner_internal.hpp"

namespace accy {
namespace planning {

namespace {

// Tile-row group of the direct-to-LDS contraction's tile walk (gemm::GroupM): 4 when A is the larger
// operand (m > n), so that each XCD reads each of its A panels once per round where B is at least 8
// tiles wide and the operand read again is the smaller one; else 8. ACCY_GEMM_GROUP_M overrides the
// choice (1, 2, 4, 8 or 16). (Grouped launches keep 8: with their G contractions per tile, 4
// measured slower for the decoder's q, k and v projections, 204 against 201 µs.)
int tile_group_m(int64_t m, int64_t n) {
  if (const char* e = std::getenv("ACCY_GEMM_GROUP_M")) {
    const int g = std::atoi(e);
    if (g == 1 || g == 2 || g == 4 || g == 8 || g == 16) return g;
  }
  return m > n ? 4 : 8;
}

}  // namespace

double Planner::macs(const GemmShape& gs) { return (double)gs.m * (double)gs.n * (double)gs.k * (double)gs.batch; }

// ---- strided views: a value that is a transpose / rename / broadcast of a buffer ----

bool Planner::gemm_shape(const Op& op, GemmShape& gs) const {
  const Type& L = g_.type(op.args[0]);
  const Type& R = g_.type(op.args[1]);
  if (!resolve_view(op.args[0], gs.a) || !resolve_view(op.args[1], gs.b)) return false;
  auto in = [](const std::vector<int64_t>& a, size_t d) { return std::find(a.begin(), a.end(), (int64_t)d) != a.end(); };
  std::vector<size_t> lb(op.lhs_batch.begin(), op.lhs_batch.end()), rb(op.rhs_batch.begin(), op.rhs_batch.end());
  std::vector<size_t> lc(op.lhs_contract.begin(), op.lhs_contract.end()),
      rc(op.rhs_contract.begin(), op.rhs_contract.end());
  std::vector<size_t> lf, rf;
  for (size_t i = 0; i < L.rank(); ++i)
    if (!in(op.lhs_contract, i) && !in(op.lhs_batch, i)) lf.push_back(i);
  for (size_t i = 0; i < R.rank(); ++i)
    if (!in(op.rhs_contract, i) && !in(op.rhs_batch, i)) rf.push_back(i);
  // Batch and contraction axes pair up one to one.
  for (size_t i = 0; i < lc.size(); ++i)
    if (L.dims[lc[i]].extent != R.dims[rc[i]].extent) return false;
  for (size_t i = 0; i < lb.size(); ++i)
    if (L.dims[lb[i]].extent != R.dims[rb[i]].extent) return false;
  // Size-one axes drop out; a batch or contraction axis of extent > 1 on one side only cannot be.
  gs.ga_b = Group::make(L.dims, gs.a.strides, lb);
  gs.gb_b = Group::make(R.dims, gs.b.strides, rb);
  gs.ga_m = Group::make(L.dims, gs.a.strides, lf);
  gs.gb_n = Group::make(R.dims, gs.b.strides, rf);
  gs.ga_k = Group::make(L.dims, gs.a.strides, lc);
  gs.gb_k = Group::make(R.dims, gs.b.strides, rc);
  gs.batch = gs.ga_b.extent();
  gs.m = gs.ga_m.extent();
  gs.n = gs.gb_n.extent();
  gs.k = gs.ga_k.extent();
  if (gs.gb_b.extent() != gs.batch || gs.gb_k.extent() != gs.k) return false;
  // Pairwise merging can differ between the two sides; the offset functions decompose the same
  // flattened index either way, since merged runs are row-major over the same logical axes.
  gs.multi = !(gs.ga_b.single() && gs.gb_b.single() && gs.ga_m.single() && gs.gb_n.single() && gs.ga_k.single() &&
               gs.gb_k.single());
  gs.a_b = gs.ga_b.stride();
  gs.b_b = gs.gb_b.stride();
  gs.a_m = gs.ga_m.stride();
  gs.b_n = gs.gb_n.stride();
  gs.a_k = gs.ga_k.stride();
  gs.b_k = gs.gb_k.stride();
  return true;
}

int Planner::dma_rows(int64_t extent) { return extent % 256 == 0 ? 256 : (extent % 128 == 0 ? 128 : 0); }

bool Planner::dma_operand(const Group& rows, const Group& k, const Group& batch, int64_t offset, int tile, bool& kc) {
  if (!rows.strides_multiple_of(1) || offset % 8 != 0) return false;
  auto aligned8 = [](const Group& g, bool skip_inner) {
    for (size_t i = 0; i < g.str.size(); ++i) {
      if (skip_inner && i + 1 == g.str.size()) continue;
      if (g.str[i] % 8 != 0) return false;
    }
    return true;
  };
  if (!aligned8(batch, false)) return false;
  if (k.inner_str() == 1 && k.inner_ext() % (k.single() ? 8 : 32) == 0 && aligned8(k, true) && aligned8(rows, false)) {
    kc = true;
    return true;
  }
  if (rows.inner_str() == 1 && rows.inner_ext() % tile == 0 && aligned8(rows, true) && aligned8(k, false)) {
    kc = false;
    return true;
  }
  return false;
}

bool Planner::dma_eligible(const GemmShape& gs, int& dm, int& dn, bool& a_kc, bool& b_kc) const {
  // at least as many K steps of 32 as pipeline stages; a last one that K does not fill only for
  // single-axis groups (the kernel clears what its loads read past K)
  if (gs.k < 128 || (gs.k % 32 != 0 && gs.multi) || std::getenv("ACCY_GEMM_NO_DMA")) return false;
  dm = dma_rows(gs.m);
  dn = dma_rows(gs.n);
  if (dm && dn)
    return dma_operand(gs.ga_m, gs.ga_k, gs.ga_b, gs.a.offset, dm, a_kc) &&
           dma_operand(gs.gb_n, gs.gb_k, gs.gb_b, gs.b.offset, dn, b_kc);
  // M or N not a multiple of 128: single-axis groups, tiles that reach past the end (the kernel clamps those
  // loads to the last row / chunk, so a row-contiguous operand's extent is a multiple of 8, and stores
  // only in range).
  if (gs.multi) return false;
  dm = dm ? dm : (gs.m > 128 ? 256 : 128);
  dn = dn ? dn : (gs.n > 128 ? 256 : 128);
  return dma_operand(gs.ga_m, gs.ga_k, gs.ga_b, gs.a.offset, 8, a_kc) &&
         dma_operand(gs.gb_n, gs.gb_k, gs.gb_b, gs.b.offset, 8, b_kc);
}

bool Planner::f32_layout_ok(const GemmShape& gs) {
  auto ok4 = [](int64_t x) { return x % 4 == 0; };
  return gs.a_k == 1 && gs.b_n == 1 && ok4(gs.a_m) && ok4(gs.b_k) && ok4(gs.a_b) && ok4(gs.b_b) &&
         ok4(gs.a.offset) && ok4(gs.b.offset);
}

int Planner::pack_f32(int slot, int64_t off, int64_t batch, int64_t R, int64_t C, int64_t sb, int64_t sr, int64_t sc) {
  const int dst = slots_.add(SlotInfo::Temp, -1, DType::f32, (uint64_t)(batch * R * C) * 4);
  KernelWriter w(g_, slots_, "i64_t");
  const std::string src = w.arg(slot, false), out = w.arg(dst, true);
  const std::string nm = name("pack", (uint32_t)dst);
  std::ostringstream k;
  const int64_t tr = (R + 63) / 64, tc = (C + 63) / 64;
  k << "extern \"C\" __global__ void __launch_bounds__(256) " << nm << "(" << w.params() << ") {\n"
    << "  const long b = blockIdx.y, r0 = (long)(blockIdx.x / " << tc << ") * 64, c0 = (long)(blockIdx.x % " << tc << ") * 64;\n"
    << "  const float* __restrict__ s = " << src << " + " << off << "L + b * " << sb << "L;\n"
    << "  float* __restrict__ d = " << out << " + b * " << R * C << "L;\n";
  if (sr == 1) {
    k << transpose_tile("float", R, C, sc, C, "s", "d", transpose_lanes(4, {R, C, sc, sb, off}));
  } else {
    k << "  const int t = threadIdx.x & 63, q = threadIdx.x >> 6;\n"
      << "  for (int r = q; r < 64; r += 4)\n"
      << "    if (r0 + r < " << R << "L && c0 + t < " << C << "L) d[(r0 + r) * " << C << "L + c0 + t] = s[(r0 + r) * " << sr
      << "L + (c0 + t) * " << sc << "L];\n";
  }
  k << "}\n";
  KernelStep ks;
  ks.source = k.str();
  ks.name = nm;
  ks.grid[0] = (uint32_t)(tr * tc);
  ks.grid[1] = (uint32_t)batch;
  ks.block[0] = 256;
  ks.klass = "pack";
  ks.label = "pack:slot" + std::to_string(slot);
  ks.algorithmic_bytes = 8.0 * (double)(batch * R * C);
  push(std::move(ks), w);
  return dst;
}

void Planner::pack_f32_operands(GemmShape& gs) {
  auto ok4 = [](int64_t x) { return x % 4 == 0; };
  if (!(gs.a_k == 1 && ok4(gs.a_m) && ok4(gs.a_b) && ok4(gs.a.offset))) {
    const int s = pack_f32(gs.a.slot, gs.a.offset, gs.batch, gs.m, gs.k, gs.a_b, gs.a_m, gs.a_k);
    gs.a = View{s, 0, {}};
    gs.a_b = gs.m * gs.k;
    gs.a_m = gs.k;
    gs.a_k = 1;
    gs.ga_b = Group{{gs.batch}, {gs.a_b}};
    gs.ga_m = Group{{gs.m}, {gs.a_m}};
    gs.ga_k = Group{{gs.k}, {1}};
  }
  if (!(gs.b_n == 1 && ok4(gs.b_k) && ok4(gs.b_b) && ok4(gs.b.offset))) {
    const int s = pack_f32(gs.b.slot, gs.b.offset, gs.batch, gs.k, gs.n, gs.b_b, gs.b_k, gs.b_n);
    gs.b = View{s, 0, {}};
    gs.b_b = gs.k * gs.n;
    gs.b_k = gs.n;
    gs.b_n = 1;
    gs.gb_b = Group{{gs.batch}, {gs.b_b}};
    gs.gb_k = Group{{gs.k}, {gs.b_k}};
    gs.gb_n = Group{{gs.n}, {1}};
  }
}

// Only the direct kernel needs another layout; the staged one reads every layout that has a unit stride. (us a pass, repacked /
// as they are: A along M 2048^3 165 / 152, 1024^3 31 / 23; B along K 4000 x 1024 x 1024 86 / 78, 64 x 8192 x 2048 50 / 31.
// With both along K and a split 128-wide tile the other way round: 2048 x 8192 x 1024 308 / 347, 3000 x 2048 x 2048 236 / 250.)
bool Planner::f32_packs(const GemmShape& gs) const {
  const Tile t = f32_tile(gs);
  bool a_kc, b_kc;
  return !t.bm || (t.bm == 128 && t.splits > 1 && staged_layout(gs, 4, a_kc, b_kc) && a_kc && b_kc);
}

bool Planner::f32_direct(const GemmShape& gs) {
  // 256 x 256 x 32 tiles, A K-contiguous and B N-contiguous with 16-byte aligned rows. Exact tiles, or
  // M / N off the tile grid (N a multiple of 4) when the problem is large (2^27 multiply-adds and more).
  // Large problems with another operand layout (an A stored M-contiguous, a B stored K-contiguous,
  // rows not 16-byte aligned) copy that operand into a contiguous temporary first (pack_f32).
  const bool exact = gs.m % 256 == 0 && gs.n % 256 == 0;
  const bool large = macs(gs) >= (double)(1ull << 27);
  if (gs.multi || !(exact || (large && gs.n % 4 == 0)) || gs.k % 32 != 0) return false;
  return f32_layout_ok(gs) || large;
}

bool Planner::staged_layout(const GemmShape& gs, int64_t vector, bool& a_kc, bool& b_kc) {
  auto operand = [vector](const Group& rows, const Group& k, bool& kc) {
    auto whole = [vector](const Group& g) { return g.inner_str() == 1 && (g.single() || g.inner_ext() % vector == 0); };
    kc = whole(k);
    return kc || whole(rows);
  };
  return operand(gs.ga_m, gs.ga_k, a_kc) && operand(gs.gb_n, gs.gb_k, b_kc);
}

// The staged f32 kernel's tile and K split by an estimate of its time in clocks: rounds of 256
// workgroups x a tile's products (128 multiply-adds per CU and clock, of which the kernel reaches about
// 76 %), or its operands' bytes at the 2800 B per clock that the L2s were seen to serve to 2048 waves and
// more, plus the first loads of each round and, where K is split, another launch and the partials'
// traffic. Measured (one box, us a pass; 128- / 64-wide tiles): 2048^3 167 / 182, 4096 x 1024 x
// 4096 303 / 307, 1000^3 78 (33 in 4 splits) / 28, 300 x 4000 x 700 292 / 87 (30 in 4 splits), 16 x 4096 x 4096
// 180 / 85 (19 as 32 x 64 tiles in 8 splits). The direct kernel's 256-wide tiles reach 137 TFLOP/s where
// they fill every round and the staged ones 100-114, so the line between them lies at 0.8 full
// rounds (2048^3, 64 tiles: 496 us).
Planner::Tile Planner::f32_tile(const GemmShape& gs) const {
  bool a_kc, b_kc;
  Tile best;
  if (!staged_layout(gs, 4, a_kc, b_kc)) return best;
  auto up = [](int64_t a, int64_t b) { return (a + b - 1) / b; };
  const int64_t direct = up(gs.m, 256) * up(gs.n, 256) * gs.batch;
  if (f32_direct(gs) && (double)direct >= 0.8 * 256.0 * (double)up(direct, 256)) return best;
  static const Tile kTiles[] = {{128, 128, 4, 2, 1}, {64, 64, 2, 2, 2}, {32, 64, 1, 2, 2}, {64, 32, 2, 1, 2}};
  double best_cost = 0;
  for (Tile t : kTiles) {
    const int64_t tiles = up(gs.m, t.bm) * up(gs.n, t.bn) * gs.batch, steps = up(gs.k, 32 * t.wk);
    if (!launchable((uint64_t)(tiles / gs.batch), 64 * t.wm * t.wn * t.wk)) continue;
    for (int splits = 1; splits <= (opt_.allow_split ? 64 : 1) && (splits == 1 || steps / splits >= 4); splits *= 2) {
      const int64_t per = up(steps, splits), used = up(steps, per);  // every split has a step
      const double groups = (double)(tiles * used), rounds = (double)up(tiles * used, 256);
      const double k = (double)per * 32 * t.wk;
      const double waves = groups * t.wm * t.wn * t.wk;
      const double products = rounds * t.bm * t.bn * k / (0.76 * 128.0);
      const double bytes = groups * (t.bm + t.bn) * k * 4.0 / (2800.0 * std::min(1.0, waves / 2048.0));
      double cost = std::max(products, bytes) + rounds * 2500.0;
      if (used > 1) cost += 6000.0 + (double)used * (double)(gs.m * gs.n * gs.batch) * 8.0 / 2100.0;
      if (!best.bm || cost < best_cost) {
        best = t;
        best.splits = (int)used;
        best.cost = best_cost = cost;
      }
    }
  }
  return best;
}

// The direct-to-LDS kernel's tile and K split by an estimate of its time in microseconds: a CU with its
// tile of 256 x 256, 128 x 256, 256 x 128 or 128 x 128 does 5.4, 4.6, 3.9 or 4.05 TFLOP/s (4096^3, every CU at
// work: 105, 117, 139, 135 us) and up to 1.45 times that where few CUs share the board's power, a round of 256 of
// them starts and drains in about 4 us, and a split costs a launch and the partials' traffic. Measured (one
// box, us a pass, 256 x 256 against 128 x 128): 2048 x 8192 x 2048 134 / 66, 3000 x 2048 x 2048 45.6 / 34.1 (128 x 256:
// 31.9), 1024^3 21.4 / 9.7, 512 x 4096 x 4096 69.6 / 30.8, 16 x 2048 x 8192 22.4 / 13.1.
Planner::Tile Planner::dma_tile(const GemmShape& gs) const {
  auto up = [](int64_t a, int64_t b) { return (a + b - 1) / b; };
  static const struct { int bm, bn; double rate; } kTiles[] = {{256, 256, 5.4}, {128, 256, 4.6}, {256, 128, 3.9}, {128, 128, 4.05}};
  const int64_t steps = up(gs.k, 32);
  Tile best;
  double best_cost = 0;
  for (const auto& t : kTiles) {
    if (gs.multi && (gs.m % t.bm != 0 || gs.n % t.bn != 0)) continue;
    if (!launchable((uint64_t)(up(gs.m, t.bm) * up(gs.n, t.bn)), 256)) continue;
    bool akc, bkc;
    if (!dma_operand(gs.ga_m, gs.ga_k, gs.ga_b, gs.a.offset, gs.m % t.bm == 0 ? t.bm : 8, akc) ||
        !dma_operand(gs.gb_n, gs.gb_k, gs.gb_b, gs.b.offset, gs.n % t.bn == 0 ? t.bn : 8, bkc))
      continue;
    for (int splits = 1; splits <= (opt_.allow_split ? 8 : 1); ++splits) {
      if (steps % splits != 0 || (splits > 1 && steps / splits < 8)) continue;
      const double groups = (double)(up(gs.m, t.bm) * up(gs.n, t.bn) * gs.batch) * splits;
      const double full = std::floor(groups / 256.0), rest = groups - 256.0 * full;
      // microseconds of one round of `active` workgroups
      auto round = [&](double active) {
        const double boost = active >= 256 ? 1.0 : std::min(1.45, 1.0 + 0.45 * (256.0 - active) / 128.0);
        return 2e-6 * t.bm * t.bn * 32.0 * (double)(steps / splits) / (t.rate * boost) + 4.0;
      };
      double cost = full * round(256) + (rest > 0 ? round(rest) : 0.0);
      if (splits > 1) cost += 3.0 + (double)splits * (double)(gs.m * gs.n * gs.batch) * 8.0 / 4e6;
      if (!best.bm || cost < best_cost) {
        best.bm = t.bm;
        best.bn = t.bn;
        best.splits = splits;
        best_cost = cost;
      }
    }
  }
  return best;
}

// The staged 16-bit kernel: 128 x 128 tiles, K split until two workgroups share every CU (each split keeps four
// steps of 64 at least).
Planner::Tile Planner::staged16_tile(const GemmShape& gs) const {
  auto up = [](int64_t a, int64_t b) { return (a + b - 1) / b; };
  Tile t;
  t.bm = t.bn = 128;
  const int64_t groups = up(gs.m, 128) * up(gs.n, 128) * gs.batch, steps = up(gs.k, 64);
  if (!launchable((uint64_t)(groups / gs.batch), 256)) return Tile();
  const int64_t want = opt_.allow_split ? std::max<int64_t>(1, std::min<int64_t>({512 / groups, steps / 4, 16})) : 1;
  t.splits = (int)up(steps, up(steps, want));
  t.cost = (double)up(groups, 512) * (1000.0 + 2500.0 * (double)steps);
  return t;
}

// Batches of a few rows and columns, and very many rows of few columns, leave a tile mostly empty; one thread per
// output folding k in order is then faster. Its time in clocks: k dependent steps (without reuse between
// lanes where each batch is one output), multiply-adds at what the lanes' loads allow (B read along n in vectors or not,
// 16-bit rows in whole vectors along k or not), the operands from memory. Measured (us a pass, tiles / folded):
// f32 65535 x (4 x 128 x 4) 397 / 48, 4194304 x 4 x 4 329 / 30, 1048576 x 16 x 8 87 / 32, 2 x 130 x 3 6.0 / 3.8, but
// 20000 x 130 x 9 7.8 / 15.8, 10000 x (20 x 130 x 20) 100 / 129; bf16 65535 x (4 x 128 x 4) 348 / 36, 3000000 x 3 x 3
// 98 / 16, 300000 x 300 x 3 131 / 92, but 1000 x (50 x 130 x 50) 16 / 115. A single round of the 16-bit kernel is as fast as a launch of the fold.
bool Planner::fold_wins(const GemmShape& gs, const Tile& t, bool f32, bool rows) {
  const int64_t tiles = (gs.m + 127) / 128 * ((gs.n + 127) / 128) * gs.batch;
  if (!f32 && !rows && tiles <= 512) return false;
  const bool along_n = gs.gb_n.inner_str() == 1 && gs.gb_n.inner_ext() % 4 == 0, along_k = gs.k % 4 == 0;
  const bool short_k = gs.gb_k.inner_str() == 1 && gs.k <= 32;  // B's rows share lines
  const double rate = f32 ? (along_n ? 1300 : short_k ? 1000 : 700) : along_n ? (along_k ? 2200 : 1200) : (along_k ? 1800 : 1000);
  const double step = gs.batch > 1 && gs.m == 1 && gs.n == 1 ? 350 : f32 ? 55 : 80;
  const double bytes = (double)gs.batch * (double)gs.k * (double)(gs.m + gs.n) * (f32 ? 4 : 2);
  // 16-bit operands read along fewer than eight rows or columns are loaded element by element
  bool a_kc, b_kc;
  const bool slow = !f32 && staged_layout(gs, 8, a_kc, b_kc) && ((!a_kc && gs.m < 8) || (!b_kc && gs.n < 8));
  const double rest = !f32 ? 1000 : gs.k % 64 ? 500 : -1500;  // a launch against the other's, the last K step's edges
  // Row kernels (us a pass, tiles / rows: f32 127 x 131 x 129 6.8 / 3.7, 64 x 2000 x 64 10.1 / 6.4, 300^3 9.7 / 20).
  if (rows) return macs(gs) / 560 < t.cost + rest;
  return std::max({step * (double)gs.k, macs(gs) / rate, bytes / 1400}) < (slow ? 3.5 : 1.0) * t.cost + rest;
}

bool Planner::gemm_eligible(const Op& op, GemmShape& gs, bool rows) const {
  if (!opt_.allow_gemm) return false;
  DType d = op.result.dtype;
  if (d != DType::bf16 && d != DType::f16 && d != DType::f32) return false;
  if (!gemm_shape(op, gs)) return false;
  if (gs.m == 0 || gs.n == 0 || gs.k == 0) return false;
  if (gs.batch > 65535) return false;  // the batch index is gridDim.y, at most 65535 on gfx950
  if (d == DType::f32) {
    bool akc, bkc;
    // Small and shallow contractions keep runCpu's serial k order: 962 x 67 x 130 takes 5.5 us there, a
    // launch's time, but a fold of k = 1000 on few threads hundreds (1000^3: 262 us).
    if (f32_direct(gs)) return true;
    if ((gs.k < 128 && macs(gs) < (double)(1ull << 23)) || !staged_layout(gs, 4, akc, bkc)) return false;
    const Tile t = f32_tile(gs);
    return t.bm && !fold_wins(gs, t, true, rows);
  }
  int dm, dn;
  bool akc, bkc;
  if (dma_eligible(gs, dm, dn, akc, bkc)) return dma_tile(gs).bm != 0;
  // Through registers at any alignment; a shallow contraction of rows that are not 16-byte aligned keeps
  // runCpu's serial k order, as small f32 ones do.
  if (!staged_layout(gs, 8, akc, bkc)) return false;
  const Tile t = staged16_tile(gs);
  if (!t.bm) return false;
  auto ok8 = [](int64_t x) { return x % 8 == 0; };
  const bool aligned = ok8(akc ? gs.k : gs.m) && ok8(bkc ? gs.k : gs.n);
  return aligned || ((gs.k >= 32 || macs(gs) >= (double)(1ull << 20)) && !fold_wins(gs, t, false, rows));
}

void Planner::mark_gemm_operands() {
  for (uint32_t v = 0; v < g_.ops.size(); ++v) {
    const Op& op = g_.ops[v];
    if (!live_[v] || op.kind != Kind::dot_general) continue;
    if (op.result.dtype != DType::bf16 && op.result.dtype != DType::f16 && op.result.dtype != DType::f32) continue;
    for (uint32_t a : op.args) {
      if (a == op.args[0] && attn_.count(v)) continue;  // the probabilities of a fused attention
      if (!view_chain_to_anchor(a)) needed_[a] = true;
    }
  }
}

bool Planner::view_chain_to_anchor(uint32_t v) const {
  const Op& op = g_.ops[v];
  switch (op.kind) {
    case Kind::transpose: case Kind::broadcast_in_dim: return view_chain_to_anchor(op.args[0]);
    case Kind::reshape: {
      const Type& it = g_.type(op.args[0]);
      if (it.rank() != op.result.rank()) return false;
      for (size_t k = 0; k < it.rank(); ++k)
        if (it.dims[k].extent != op.result.dims[k].extent) return false;
      return view_chain_to_anchor(op.args[0]);
    }
    case Kind::parameter: case Kind::dot_general: case Kind::reduce: case Kind::scatter_add: return true;
    default: return needed_[v];
  }
}

// ---- fused attention: dot(softmax_last(scale * dot(Q, K) [causal -inf mask]), V) ----

void Planner::dot(uint32_t v) {
  const Op& op = g_.ops[v];
  auto fused = attn_.find(v);
  if (fused != attn_.end()) {
    AttnLayout L;
    if (attention_layout(v, fused->second, L)) {
      attention(v, fused->second, L);
      return;
    }
    AttnLayout one;
    if (decode_layout(v, fused->second, one)) {
      attention_decode(v, fused->second, one);
      return;
    }
    // Operands the kernel cannot address: compute the absorbed values after all, in order.
    needed_[op.args[0]] = true;
    std::vector<uint32_t> inner = fused->second.inner;
    attn_.erase(fused);
    for (uint32_t u : inner) done_[u] = false;
    for (uint32_t u : inner)
      if (!done_[u]) process(u);
  }
  GemmShape gs;
  if (gemm_eligible(op, gs)) {
    if (op.result.dtype == DType::f32 && f32_direct(gs) && !f32_layout_ok(gs) && f32_packs(gs)) pack_f32_operands(gs);
    std::vector<std::pair<uint32_t, GemmShape>> group;
    if (gemm_siblings(v, gs, group)) {
      gemm_group(group);
      return;
    }
    gemm(v, gs);
    return;
  }
  dot_serial(v);
}

// ---- grouped contractions: several contractions of one activation in one launch ----

bool Planner::same_group(const Group& x, const Group& y) { return x.ext == y.ext && x.str == y.str; }

bool Planner::plain_store(uint32_t u) const {
  uint32_t t;
  return attn_.find(u) == attn_.end() && !epilogue_target(u, t);
}

bool Planner::gemm_siblings(uint32_t v, const GemmShape& gs, std::vector<std::pair<uint32_t, GemmShape>>& group) const {
  const Op& op = g_.ops[v];
  const DType d = op.result.dtype;
  if (op.kind != Kind::dot_general || (d != DType::bf16 && d != DType::f16) || gs.multi) return false;
  // The decoder's three projections: 175.5 µs grouped against 186.6 µs in three launches (C5, one
  // box). ACCY_GEMM_NO_GROUP plans separate launches.
  if (gs.m % 256 != 0 || gs.n % 256 != 0 || std::getenv("ACCY_GEMM_NO_GROUP")) return false;
  int dm = 0, dn = 0;
  bool akc = gs.a_k == 1, bkc = gs.b_k == 1;
  if (!dma_eligible(gs, dm, dn, akc, bkc) || dm != 256 || dn != 256 || !plain_store(v)) return false;
  group.assign(1, {v, gs});
  constexpr size_t kMaxGroup = 4;
  for (uint32_t u = v + 1; u < g_.ops.size() && group.size() < kMaxGroup; ++u) {
    const Op& uo = g_.ops[u];
    if (!live_[u] || done_[u] || uo.kind != Kind::dot_general || uo.args[0] != op.args[0] || uo.result.dtype != d)
      continue;
    GemmShape gu;
    if (!gemm_eligible(uo, gu) || gu.multi || !plain_store(u)) continue;
    if (gu.batch != gs.batch || gu.m != gs.m || gu.n != gs.n || gu.k != gs.k) continue;
    if (gu.a.slot != gs.a.slot || gu.a.offset != gs.a.offset || gu.a_b != gs.a_b || gu.a_m != gs.a_m ||
        gu.a_k != gs.a_k || gu.b_b != gs.b_b || gu.b_k != gs.b_k || gu.b_n != gs.b_n)
      continue;
    if (!same_group(gu.ga_b, gs.ga_b) || !same_group(gu.ga_m, gs.ga_m) || !same_group(gu.ga_k, gs.ga_k) ||
        !same_group(gu.gb_b, gs.gb_b) || !same_group(gu.gb_k, gs.gb_k) || !same_group(gu.gb_n, gs.gb_n))
      continue;
    int um = 0, un = 0;
    bool uak = gu.a_k == 1, ubk = gu.b_k == 1;
    if (!dma_eligible(gu, um, un, uak, ubk) || um != dm || un != dn || uak != akc || ubk != bkc) continue;
    group.push_back({u, gu});
  }
  return group.size() > 1;
}

void Planner::gemm_group(const std::vector<std::pair<uint32_t, GemmShape>>& group) {
  const uint32_t v = group[0].first;
  const GemmShape& gs = group[0].second;
  const DType d = g_.ops[v].result.dtype;
  const size_t G = group.size();
  KernelWriter w(g_, slots_, "i64_t");
  const std::string a = w.arg(gs.a.slot, false);
  std::vector<std::string> bs;
  std::ostringstream cases;
  const std::string cidx = "b * " + std::to_string(gs.m * gs.n) + "L + m * " + std::to_string(gs.n) + "L + n";
  std::string nm = name("gemm", v), label = "gemm:%" + std::to_string(v);
  for (size_t i = 0; i < G; ++i) {
    const uint32_t u = group[i].first;
    bs.push_back(w.arg(group[i].second.b.slot, false) + " + " + std::to_string(group[i].second.b.offset) + "L");
    const int out = slots_.slot_of[u] >= 0 ? slots_.slot_of[u] : temp_slot(u);
    cases << "      case " << i << ": return " << w.arg(out, true) << ";\n";
    if (i) label += "&%" + std::to_string(u);
  }
  const KernelWriter::Members members = w.members();
  std::ostringstream src;
  src << "#include \"gemm\"\n";
  src << "struct Epi_" << nm << " {\n" << members.decls
      << "  __device__ __forceinline__ u16_t* out(int g) const {\n"
      << "    switch (g) {\n" << cases.str() << "      default: return nullptr;\n    }\n  }\n"
      << "  __device__ __forceinline__ void operator()(u16_t* __restrict__ o, long b, long m, long n, float v) const {\n"
      << "    accy::" << (d == DType::bf16 ? "st_bf16" : "st_f16") << "(o, " << cidx << ", v);\n  }\n};\n";
  src << "struct Cfg_" << nm << " {\n"
      << "  static constexpr int DT = " << (d == DType::bf16 ? 0 : 1) << ";\n"
      << "  static constexpr long M = " << gs.m << ", N = " << gs.n << ", K = " << gs.k << ";\n"
      << "  static constexpr bool A_KC = " << (gs.a_k == 1 ? "true" : "false")
      << ", B_KC = " << (gs.b_k == 1 ? "true" : "false") << ";\n"
      << gs.ga_b.fn("a_b") << gs.ga_m.fn("a_m") << gs.ga_k.fn("a_k") << gs.gb_b.fn("b_b") << gs.gb_k.fn("b_k")
      << gs.gb_n.fn("b_n") << "  static constexpr int BM = 256, BN = 256, STAGES = 4;\n};\n";
  src << "extern \"C\" __global__ void __launch_bounds__(256) " << nm << "(" << w.params() << ") {\n"
      << "  const u16_t* const bs[" << G << "] = {";
  for (size_t i = 0; i < G; ++i) src << (i ? ", " : "") << bs[i];
  src << "};\n  accy::gemm::mma16_dma_group<Cfg_" << nm << ", " << G << ">(" << a << " + " << gs.a.offset
      << "L, bs, Epi_" << nm << "{" << members.inits << "});\n}\n";
  KernelStep k;
  k.source = src.str();
  k.name = nm;
  k.grid[0] = (uint32_t)(G * (size_t)((gs.m / 256) * (gs.n / 256)));
  k.grid[1] = (uint32_t)gs.batch;
  k.block[0] = 256;
  k.klass = "gemm";
  k.label = label;
  k.algorithmic_flops = 2.0 * (double)G * (double)gs.batch * (double)gs.m * (double)gs.n * (double)gs.k;
  push(std::move(k), w);
  for (const auto& member : group) finish(member.first);
}

void Planner::gemm(uint32_t v, const GemmShape& gs) {
  OutStrides os;
  os.b = gs.m * gs.n;
  os.m = gs.n;
  os.n = 1;
  gemm(v, gs, os);
}

// ---- contraction epilogues ----

bool Planner::epilogue_target(uint32_t v, uint32_t& target) const {
  if (needed_[v] || slots_.slot_of[v] >= 0) return false;
  const Type& vt = g_.type(v);
  std::vector<std::vector<uint32_t>> users(g_.ops.size());
  for (uint32_t u = v + 1; u < g_.ops.size(); ++u)
    if (live_[u] && !done_[u])
      for (uint32_t a : g_.ops[u].args) users[a].push_back(u);
  std::set<uint32_t> region = {v}, targets;
  std::vector<uint32_t> stack = {v};
  while (!stack.empty()) {
    uint32_t x = stack.back();
    stack.pop_back();
    for (uint32_t u : users[x]) {
      const Op& uo = g_.ops[u];
      bool elementwise = uo.kind == Kind::unary || uo.kind == Kind::binary || uo.kind == Kind::select ||
                         uo.kind == Kind::compare;
      if (!elementwise || !(uo.result.dims == vt.dims)) return false;
      if (needed_[u]) {
        targets.insert(u);
      } else if (!region.count(u)) {
        region.insert(u);
        stack.push_back(u);
      }
    }
  }
  if (targets.size() != 1) return false;
  const uint32_t u = *targets.begin();
  if (done_[u]) return false;
  target = u;
  return true;
}

bool Planner::lut_epilogue(uint32_t v, uint32_t target, DType d, DType td) const {
  auto b16 = [](DType t) { return t == DType::bf16 || t == DType::f16; };
  if (!b16(d) || !b16(td) || target == v || std::getenv("ACCY_GEMM_NO_LUT")) return false;
  std::set<uint32_t> seen;
  int ops = 0;
  std::function<bool(uint32_t)> ok = [&](uint32_t x) -> bool {
    if (x == v || seen.count(x)) return true;
    double c;
    if (splat_float(x, c)) return true;
    const Op& o = g_.ops[x];
    const bool ew = o.kind == Kind::unary || o.kind == Kind::binary || o.kind == Kind::select ||
                    o.kind == Kind::compare;
    if (!ew) return false;
    seen.insert(x);
    ++ops;
    for (uint32_t a : o.args)
      if (!ok(a)) return false;
    return true;
  };
  return ok(target) && ops >= 6;
}

void Planner::gemm(uint32_t v, const GemmShape& gs, const OutStrides& os) {
  const Op& op = g_.ops[v];
  DType d = op.result.dtype;
  const std::string cidx = "b * " + std::to_string(os.b) + "L + m * " + std::to_string(os.m) + "L + n * " +
                           std::to_string(os.n) + "L";
  std::string nm = name("gemm", v);
  uint32_t target = v;
  std::unique_ptr<KernelWriter> w;
  // Split along K: the contraction stores f32 sums of its part of K and split::sum adds them and runs the
  // epilogue, whose kernel then reads no operand.
  int dm = 0, dn = 0;
  bool akc = gs.a_k == 1, bkc = gs.b_k == 1;
  const bool dma = d != DType::f32 && dma_eligible(gs, dm, dn, akc, bkc);
  const Tile tile = d == DType::f32 ? f32_tile(gs) : dma ? dma_tile(gs) : staged16_tile(gs);
  if (d != DType::f32) {
    if (!dma) staged_layout(gs, 8, akc, bkc);
    dm = tile.bm;
    dn = tile.bn;
  }
  const bool split = tile.splits > 1;
  auto operands = [&](KernelWriter& kw) {
    kw.arg(gs.a.slot, false);
    kw.arg(gs.b.slot, false);
  };
  std::ostringstream epi;
  std::string table_members;  // a lookup-table epilogue's interface (gemm.h HasTable)
  // The fused epilogue (dot_general results only: os is their row-major layout).
  const bool rowmajor = os.b == gs.m * gs.n && os.m == gs.n && os.n == 1;
  if (op.kind == Kind::dot_general && rowmajor && epilogue_target(v, target)) {
    try {
      w.reset(new KernelWriter(g_, slots_, "i64_t"));
      if (!split) operands(*w);
      const Type& rt = op.result;
      const size_t nb = op.lhs_batch.size();
      const size_t nlf = rt.rank() - nb - (g_.type(op.args[1]).rank() - op.rhs_batch.size() - op.rhs_contract.size());
      std::vector<Dim> bd(rt.dims.begin(), rt.dims.begin() + (long)nb);
      std::vector<Dim> md(rt.dims.begin() + (long)nb, rt.dims.begin() + (long)(nb + nlf));
      std::vector<Dim> ndims(rt.dims.begin() + (long)(nb + nlf), rt.dims.end());
      std::vector<std::string> coords;
      for (auto& c : delinearize("b", bd)) coords.push_back(c);
      for (auto& c : delinearize("m", md)) coords.push_back(c);
      for (auto& c : delinearize("n", ndims)) coords.push_back(c);
      Scope sc(epi, "    ");
      w->provide = [&](uint32_t vid, const std::vector<std::string>& c, std::string& out) -> bool {
        if (vid != v) return false;
        if (c != coords) throw NotFusable("contraction value read at another index");
        out = "vv";
        return true;
      };
      const DType td = g_.type(target).dtype;
      if (lut_epilogue(v, target, d, td)) {
        // A 16-bit epilogue that is a function of the rounded contraction value alone: a table
        // kernel evaluates the same generated expression for all 65536 bit patterns, and the
        // contraction's epilogue is one lookup per element (bit-identical by construction).
        const int tslot = slots_.add(SlotInfo::Temp, -1, td, 65536u * 2u);
        KernelWriter tw(g_, slots_, "i64_t");
        tw.arg(tslot, true);
        std::ostringstream tk;
        Scope tsc(tk, "  ");
        tw.provide = [&](uint32_t vid, const std::vector<std::string>&, std::string& out) -> bool {
          if (vid != v) return false;
          out = "vv";
          return true;
        };
        const std::string tx = tw.value(target, coords, tsc);
        const std::string tnm = name("lut", target);
        std::ostringstream tsrc;
        tsrc << "extern \"C\" __global__ void __launch_bounds__(256) " << tnm << "(" << tw.params() << ") {\n"
             << "  const int i = (int)(blockIdx.x * 256 + threadIdx.x);\n"
             << "  const float vv = " << (d == DType::bf16 ? "accy::bf16_to_f32" : "accy::f16_to_f32") << "((u16_t)i);\n"
             << tk.str() << "  " << tw.store(tslot, "i", td, tx) << "\n}\n";
        KernelStep ts;
        ts.source = tsrc.str();
        ts.name = tnm;
        ts.grid[0] = 256;
        ts.block[0] = 256;
        ts.klass = "lut";
        ts.label = "lut:%" + std::to_string(target);
        ts.once = true;
        const std::string tab = w->arg(tslot, false);
        int out = slots_.slot_of[target] >= 0 ? slots_.slot_of[target] : temp_slot(target);
        const std::string dst = w->arg(out, true);
        const std::string idx = d == DType::bf16 ? "accy::f32_to_bf16(v)" : "accy::f32_to_f16(v)";
        epi << "    " << dst << "[" << cidx << "] = " << tab << "[" << idx << "];\n";
        table_members = "  static constexpr bool kTable = true;\n"
                        "  __device__ __forceinline__ const u16_t* table() const { return " + tab + "; }\n"
                        "  static __device__ __forceinline__ u16_t index(float v) { return " + idx + "; }\n"
                        "  __device__ __forceinline__ void put(long b, long m, long n, u16_t bits) const { " +
                        dst + "[" + cidx + "] = bits; }\n";
        push(std::move(ts), tw);
      } else {
        std::string x = w->value(target, coords, sc);
        int out = slots_.slot_of[target] >= 0 ? slots_.slot_of[target] : temp_slot(target);
        epi << sc.indent << w->store(out, cidx, td, x) << "\n";
      }
    } catch (const NotFusable&) {
      target = v;
      w.reset();
      epi.str("");
    }
  }
  if (!w) {
    w.reset(new KernelWriter(g_, slots_, "i64_t"));
    if (!split) operands(*w);
    int out = slots_.slot_of[v] >= 0 ? slots_.slot_of[v] : temp_slot(v);
    epi << "    " << w->store(out, cidx, d, "v") << "\n";
  }
  // A split contraction's own kernel: operands and partial sums.
  std::unique_ptr<KernelWriter> pw;
  std::string partial;
  if (split) {
    pw.reset(new KernelWriter(g_, slots_, "i64_t"));
    operands(*pw);
    const int part = slots_.add(SlotInfo::Temp, -1, DType::f32, (uint64_t)tile.splits * (uint64_t)(gs.batch * gs.m * gs.n) * 4);
    partial = pw->arg(part, true);
    w->arg(part, false);
  }
  KernelWriter& kw = split ? *pw : *w;
  const std::string a = kw.arg(gs.a.slot, false), b = kw.arg(gs.b.slot, false);
  // Epilogue functor: every buffer of the kernel as a member named like the kernel parameter.
  const KernelWriter::Members members = w->members();
  // A 16-bit epilogue that reads buffers besides A, B and its output (a residual, a bias) goes
  // through LDS in whole row segments (gemm.h staged_epilogue; measured on C5's MLP-down: 224 ->
  // 219.7 us). A plain store does not (58.2 against 60.3 us staged for C5's q projection).
  const std::string ps = w->params();
  const long nparams = ps.empty() ? 0 : 1 + (long)std::count(ps.begin(), ps.end(), ',');
  const bool staged = table_members.empty() && target != v && (d == DType::bf16 || d == DType::f16) && nparams > 3 &&
                      !std::getenv("ACCY_GEMM_NO_STAGE");
  std::ostringstream src;
  KernelStep k;
  std::string functor = "Epi_" + nm + "{" + members.inits + "}", part_struct;
  if (split) {
    part_struct = "struct Part_" + nm + " {\n  float* __restrict__ p;\n"
                  "  __device__ __forceinline__ void operator()(long b, long m, long n, float v) const {\n    p[(blockIdx.z * " +
                  std::to_string(gs.batch) + "L + b) * " + std::to_string(gs.m * gs.n) + "L + m * " + std::to_string(gs.n) +
                  "L + n] = v;\n  }\n};\n";
    functor = "Part_" + nm + "{" + partial + "}";
  }
  src << "#include \"gemm\"\n";
  src << "struct Epi_" << nm << " {\n" << members.decls
      << table_members << (staged ? "  static constexpr bool kStaged = true;\n" : "")
      << "  __device__ __forceinline__ void operator()(long b, long m, long n, float v) const {\n"
      << (target != v && table_members.empty() ? "    const float vv = " + round_to(d, "v") + ";\n" : "") << epi.str()
      << "  }\n};\n";
  if (d == DType::f32) {
    // f32 on v_mfma_f32_32x32x2_f32: 256 x 256 x 32 tiles straight to LDS, or staged tiles (f32_tile).
    src << "struct Cfg_" << nm << " {\n"
        << "  static constexpr long BATCH = " << gs.batch << ", M = " << gs.m << ", N = " << gs.n << ", K = " << gs.k << ";\n"
        << gs.ga_b.fn("a_b") << gs.ga_m.fn("a_m") << gs.ga_k.fn("a_k") << gs.gb_b.fn("b_b") << gs.gb_k.fn("b_k")
        << gs.gb_n.fn("b_n");
    if (tile.bm) {
      bool a_kc = false, b_kc = false;
      staged_layout(gs, 4, a_kc, b_kc);
      src << "  static constexpr bool A_KC = " << (a_kc ? "true" : "false") << ", B_KC = " << (b_kc ? "true" : "false")
          << ";\n  static constexpr int BM = " << tile.bm << ", BN = " << tile.bn << ", WAVES_M = " << tile.wm
          << ", WAVES_N = " << tile.wn << ", WAVES_K = " << tile.wk << ", SPLITS = " << tile.splits << ";\n";
    }
    src << "};\n";
    const int bm = tile.bm ? tile.bm : 256, bn = tile.bm ? tile.bn : 256;
    k.block[0] = tile.bm ? 64u * (uint32_t)(tile.wm * tile.wn * tile.wk) : 256u;
    k.grid[0] = (uint32_t)(((gs.m + bm - 1) / bm) * ((gs.n + bn - 1) / bn));
    k.grid[2] = (uint32_t)tile.splits;
    src << part_struct;
    src << "extern \"C\" __global__ void __launch_bounds__(" << k.block[0] << ") " << nm << "(" << kw.params() << ") {\n"
        << "  accy::gemm::mma32f<Cfg_" << nm << ">(" << a << " + " << gs.a.offset << "L, " << b << " + "
        << gs.b.offset << "L, " << functor << ");\n}\n";
  } else {
    // Direct-to-LDS pipeline (dma_eligible: every row start 16-byte aligned); otherwise the kernel that
    // stages through registers.
    src << "struct Cfg_" << nm << " {\n"
        << "  static constexpr int DT = " << (d == DType::bf16 ? 0 : 1) << ";\n"
        << "  static constexpr long BATCH = " << gs.batch << ", M = " << gs.m << ", N = " << gs.n << ", K = " << gs.k << ";\n"
        << "  static constexpr bool A_KC = " << (akc ? "true" : "false") << ", B_KC = " << (bkc ? "true" : "false")
        << ";\n"
        << gs.ga_b.fn("a_b") << gs.ga_m.fn("a_m") << gs.ga_k.fn("a_k") << gs.gb_b.fn("b_b") << gs.gb_k.fn("b_k")
        << gs.gb_n.fn("b_n");
    // Launch candidates of the direct-to-LDS kernel (bit-identical results: every output keeps its
    // k order and split): the N tile dma_tile chose, then the other of 256 and 128 where B's layout and
    // extent allow it. (256 x 128 with 3 stages and two workgroups per CU was measured too: its LDS
    // traffic per MFMA is half as large again as the 256 x 256 tile's, and it ran 20-40 % slower on
    // every benchmark contraction.) The source carries a placeholder until the candidate is chosen.
    std::vector<int> n_tiles{dn};
    if (dma && gs.n > 128) {
      const int other = 384 - dn;
      bool kc2 = bkc;
      if (dma_operand(gs.gb_n, gs.gb_k, gs.gb_b, gs.b.offset, gs.n % other == 0 || gs.multi ? other : 8, kc2) && kc2 == bkc &&
          (!gs.multi || gs.n % other == 0))
        n_tiles.push_back(other);
    }
    const bool placeholder = n_tiles.size() > 1;
    src << "  static constexpr int BM = " << dm << ", BN = " << (placeholder ? "ACCY_N_TILE" : std::to_string(dn));
    if (dma) src << ", STAGES = 4, GROUP_M = " << tile_group_m(gs.m, gs.n);
    if (!dma || split) src << ", SPLITS = " << tile.splits;
    src << ";\n};\n";
    src << part_struct << "extern \"C\" __global__ void __launch_bounds__(256) " << nm << "(" << kw.params()
        << ") {\n  accy::gemm::" << (dma ? "mma16_dma" : "mma16_staged") << "<Cfg_" << nm << ">(" << a << " + " << gs.a.offset
        << "L, " << b << " + " << gs.b.offset << "L, " << functor << ");\n}\n";
    k.grid[2] = (uint32_t)tile.splits;
    k.source = src.str();
    if (placeholder) {
      k.tuning_key = tuning_key("gemm", k.source, "m=" + std::to_string(gs.m) + ",n=" + std::to_string(gs.n) +
                                                      ",k=" + std::to_string(gs.k) + ",batch=" + std::to_string(gs.batch));
      k.candidate_count = (uint32_t)n_tiles.size();
      k.candidate = candidate_for(k.tuning_key, k.candidate_count);
      dn = n_tiles[k.candidate];
      const std::string mark = "ACCY_N_TILE";
      k.source.replace(k.source.find(mark), mark.size(), std::to_string(dn));
    }
    k.grid[0] = (uint32_t)(((gs.m + dm - 1) / dm) * ((gs.n + dn - 1) / dn));
    k.block[0] = 256;
  }
  if (k.source.empty()) k.source = src.str();
  k.name = nm;
  k.grid[1] = (uint32_t)gs.batch;
  k.klass = "gemm";
  k.label = "gemm:%" + std::to_string(v) + (target != v ? "+%" + std::to_string(target) : "");
  k.algorithmic_flops = 2.0 * macs(gs);
  push(std::move(k), kw);
  if (split) {
    KernelStep sum;
    sum.name = name("split_sum", v);
    const std::string both = plan_.steps.back().kernel.source;  // with the launch candidate chosen
    sum.source = both.substr(0, both.find("struct Part_")) + "extern \"C\" __global__ void __launch_bounds__(256) " + sum.name + "(" +
                 w->params() + ") {\n  accy::split::sum<Cfg_" + nm + ">(" + w->arg(pw->args.back(), false) + ", Epi_" + nm +
                 "{" + members.inits + "});\n}\n";
    sum.grid[0] = grid_for((uint64_t)(gs.batch * gs.m * gs.n), 256);
    sum.block[0] = 256;
    sum.klass = "gemm";
    sum.label = "split_sum:%" + std::to_string(target);
    push(std::move(sum), *w);
  }
  if (target != v) {
    done_[v] = true;
    finish(target);
  } else {
    finish(v);
  }
}

// ---- sum over k of mul(A, B): the same contraction, spelled elementwise ----

bool Planner::operand_of(uint32_t u, size_t rank, Operand& o) const {
  const Op& op = g_.ops[u];
  if (op.kind == Kind::broadcast_in_dim) {
    o.src = op.args[0];
    o.to_mul.assign(op.ints.begin(), op.ints.end());
  } else {
    if (op.result.rank() != rank) return false;
    o.src = u;
    o.to_mul.resize(rank);
    for (size_t i = 0; i < rank; ++i) o.to_mul[i] = (int)i;
  }
  return true;
}

bool Planner::mulsum(uint32_t v) {
  const Op& red = g_.ops[v];
  if ((Reducer)red.code != Reducer::sum) return false;
  const DType d = red.result.dtype;
  if (d != DType::f32 && d != DType::bf16 && d != DType::f16) return false;
  double init;
  if (!splat_float(red.args[1], init) || init != 0.0) return false;
  const Op& mul = g_.ops[red.args[0]];
  if (mul.kind != Kind::binary || (Binary)mul.code != Binary::mul || mul.result.dtype != d) return false;
  const Type& mt = mul.result;
  const size_t R = mt.rank();
  Operand A, B;
  if (!operand_of(mul.args[0], R, A) || !operand_of(mul.args[1], R, B)) return false;
  // For each mul dim: the A / B source dim that supplies it (-1 if broadcast there).
  std::vector<int> from_a(R, -1), from_b(R, -1);
  const Type& at = g_.type(A.src);
  const Type& bt = g_.type(B.src);
  for (size_t i = 0; i < A.to_mul.size(); ++i)
    if (at.dims[i].extent == mt.dims[(size_t)A.to_mul[i]].extent && at.dims[i].extent != 1) from_a[(size_t)A.to_mul[i]] = (int)i;
  for (size_t i = 0; i < B.to_mul.size(); ++i)
    if (bt.dims[i].extent == mt.dims[(size_t)B.to_mul[i]].extent && bt.dims[i].extent != 1) from_b[(size_t)B.to_mul[i]] = (int)i;
  std::vector<bool> reduced(R, false);
  for (int64_t a : red.ints) reduced[(size_t)a] = true;
  Op dot;
  dot.kind = Kind::dot_general;
  dot.args = {A.src, B.src};
  std::vector<Dim> batch_dims, lf_dims, rf_dims;
  std::vector<size_t> batch_mul, lf_mul, rf_mul;
  for (size_t i = 0; i < R; ++i) {
    if (mt.dims[i].extent == 1) {
      // Size-one axes: must not come from a real axis of both (nothing to contract or batch).
      continue;
    }
    const bool ia = from_a[i] >= 0, ib = from_b[i] >= 0;
    if (reduced[i]) {
      if (!ia || !ib) return false;
      dot.lhs_contract.push_back(from_a[i]);
      dot.rhs_contract.push_back(from_b[i]);
    } else if (ia && ib) {
      dot.lhs_batch.push_back(from_a[i]);
      dot.rhs_batch.push_back(from_b[i]);
      batch_dims.push_back(mt.dims[i]);
      batch_mul.push_back(i);
    } else if (ia) {
      lf_dims.push_back(mt.dims[i]);
      lf_mul.push_back(i);
    } else if (ib) {
      rf_dims.push_back(mt.dims[i]);
      rf_mul.push_back(i);
    } else {
      return false;
    }
  }
  // Source dims that are not used (size one, or broadcast away) must have extent one.
  auto covered = [](const std::vector<int>& from, size_t src_dim) {
    return std::find(from.begin(), from.end(), (int)src_dim) != from.end();
  };
  for (size_t i = 0; i < at.rank(); ++i)
    if (!covered(from_a, i) && at.dims[i].extent != 1) return false;
  for (size_t i = 0; i < bt.rank(); ++i)
    if (!covered(from_b, i) && bt.dims[i].extent != 1) return false;
  // The contraction's free dims must flatten in the order the sources hold them; the dot result
  // is [batch, lhs free, rhs free].
  dot.result.dtype = d;
  for (auto* g : {&batch_dims, &lf_dims, &rf_dims})
    for (const Dim& x : *g) dot.result.dims.push_back(x);
  if (dot.lhs_contract.empty()) return false;
  GemmShape gs;
  RowShape rows;
  if (!gemm_eligible(dot, gs, row_shape(v, rows) && prod(rows.T, 0, rows.T.size()) >= 64)) return false;
  // Matrix cores only pay when both output extents fill a tile; x * x summed over an axis (a
  // norm) stays a row reduction.
  if (gs.m < 32 || gs.n < 32) return false;
  // Output strides: the reduce result keeps the non-reduced mul dims in order.
  std::vector<int64_t> rstr = row_major_strides(red.result.dims);
  std::vector<int> res_pos(R, -1);
  for (size_t i = 0, r = 0; i < R; ++i)
    if (!reduced[i]) res_pos[i] = (int)r++;
  auto group = [&](const std::vector<size_t>& muls, int64_t& extent, int64_t& stride) {
    std::vector<Dim> dims;
    std::vector<int64_t> strides;
    std::vector<size_t> idx;
    for (size_t j = 0; j < muls.size(); ++j) {
      dims.push_back(mt.dims[muls[j]]);
      strides.push_back(rstr[(size_t)res_pos[muls[j]]]);
      idx.push_back(j);
    }
    return flatten(dims, strides, idx, extent, stride);
  };
  OutStrides os;
  int64_t e;
  if (!group(batch_mul, e, os.b) || !group(lf_mul, e, os.m) || !group(rf_mul, e, os.n)) return false;
  gemm(v, gs, os);
  return true;
}

}  // namespace planning
}  // namespace accy
