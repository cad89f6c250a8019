// Kernel formation for reductions: serial folds (whole or in chunks) and row kernels (several fused
// reductions over the trailing axes of one row space, one workgroup per row).
#include "planner_internal.hpp"

namespace accy {
namespace planning {

// ---- fold: one output per thread, serial left-to-right over the reduced index ----

namespace {

// A fold in chunks: a long range of few outputs, where a thread per output leaves most of the GPU idle. From a wave
// per SIMD on a thread per output is faster (us a pass, a thread / chunks: 300 x 262143 bf16 28 / 43, 600 x 100000 f32 35 / 40,
// 1000 x 60000 f32 44 / 38).
bool long_fold(uint64_t nred, uint64_t nout) { return nred >= 256 && nout * nred >= (1ull << 17) && nout < (1ull << 16); }

}  // namespace

void Planner::fold(uint32_t v) {
  const Op& op = g_.ops[v];
  const Type& in = g_.type(op.args[0]);
  const Type& rt = op.result;
  uint64_t nout = rt.elements();
  if (nout == 0) {
    temp_slot(v);
    finish(v);
    return;
  }
  std::vector<size_t> red, keep;
  for (size_t d = 0; d < in.rank(); ++d)
    (std::find(op.ints.begin(), op.ints.end(), (int64_t)d) != op.ints.end() ? red : keep).push_back(d);
  std::vector<Dim> rdims, kdims;
  for (size_t d : red) rdims.push_back(in.dims[d]);
  for (size_t d : keep) kdims.push_back(in.dims[d]);
  uint64_t nred = prod(rdims, 0, rdims.size());
  Reducer r = (Reducer)op.code;
  DType d = rt.dtype;
  // Few outputs over a long reduced range: one serial fold per output cannot fill the GPU (and keeps
  // too few loads in flight), so the range is folded in chunks and the chunks' partials folded in
  // order (fold_chunked).
  if (long_fold(nred, nout) && chunk_identity(d, r)) {
    const int out = temp_slot(v);
    fold_chunked(v, out, in, red, keep, rdims, kdims, nout, nred, r, d);
    finish(v);
    return;
  }
  // Later folds over the same axes of the same extents whose operands are ready join this one: one
  // launch, and what their elementwise operands share (loads, a sine) is evaluated once. Each output
  // keeps its own left-to-right order. (The README's mismatch and slope of eight guesses: 10.7 us a
  // pass in two launches, 7.5 us in one.)
  std::vector<uint32_t> group{v};
  const std::set<int64_t> axes(op.ints.begin(), op.ints.end());
  const bool long_range = long_fold(nred, nout);
  constexpr size_t kMaxFolds = 4;
  for (uint32_t u = v + 1; !long_range && u < (uint32_t)g_.ops.size() && group.size() < kMaxFolds; ++u) {
    const Op& uo = g_.ops[u];
    if (!live_[u] || done_[u] || uo.kind != Kind::reduce || !(g_.type(uo.args[0]).dims == in.dims)) continue;
    if (std::set<int64_t>(uo.ints.begin(), uo.ints.end()) != axes) continue;
    // a product of two broadcasts may be a contraction spelled elementwise (mulsum), planned at its turn
    const Op& x = g_.ops[uo.args[0]];
    if (x.kind == Kind::binary && (Binary)x.code == Binary::mul && g_.ops[x.args[0]].kind == Kind::broadcast_in_dim &&
        g_.ops[x.args[1]].kind == Kind::broadcast_in_dim)
      continue;
    group.push_back(u);
    try {
      KernelWriter trial(g_, slots_, itype());
      fold_body(trial, group, in, red, keep, rdims, kdims, nred, false);
    } catch (const NotFusable&) {
      group.pop_back();
    }
  }
  KernelWriter w(g_, slots_, itype());
  const std::string body = fold_body(w, group, in, red, keep, rdims, kdims, nred, true);
  const uint32_t B = 256;
  std::string nm = name("fold", v), label = "fold:%" + std::to_string(v);
  for (size_t i = 1; i < group.size(); ++i) label += "&%" + std::to_string(group[i]);
  std::ostringstream src;
  src << "extern \"C\" __global__ void __launch_bounds__(" << B << ") " << nm << "(" << w.params() << ") {\n"
      << "  typedef " << w.itype << " I;\n"
      << "  for (I o = (I)blockIdx.x * " << B << " + threadIdx.x; o < (I)" << nout << "; o += (I)gridDim.x * "
      << B << ") {\n"
      << body << "  }\n}\n";
  KernelStep k;
  k.source = src.str();
  k.name = nm;
  k.grid[0] = grid_for(nout, B, 65536);
  k.block[0] = B;
  k.klass = "fold";
  k.label = label;
  push(std::move(k), w);
  for (uint32_t u : group) finish(u);
}

std::string Planner::fold_body(KernelWriter& w, const std::vector<uint32_t>& group, const Type& in, const std::vector<size_t>& red,
                               const std::vector<size_t>& keep, const std::vector<Dim>& rdims, const std::vector<Dim>& kdims,
                               uint64_t nred, bool commit) {
  std::ostringstream body, steps, stores;
  Scope outer(body, "    "), inner(steps, "      ");
  std::vector<std::string> kc = delinearize("o", kdims), rc = delinearize("r", rdims);
  std::vector<std::string> full(in.rank());
  for (size_t i = 0; i < red.size(); ++i) full[red[i]] = rc[i];
  for (size_t i = 0; i < keep.size(); ++i) full[keep[i]] = kc[i];
  for (size_t i = 0; i < group.size(); ++i) {
    const Op& op = g_.ops[group[i]];
    const Reducer r = (Reducer)op.code;
    const DType d = op.result.dtype;
    const std::string at = acc_type(d, r), acc = "acc" + (i ? std::to_string(i) : std::string());
    const std::string init = w.value(op.args[1], {}, outer);
    body << "    " << at << " " << acc << " = (" << at << ")" << init << ";\n";
    const std::string x = w.value(op.args[0], full, inner);
    steps << "      " << acc << " = " << serial_fold_step(d, r, acc, x) << ";\n";
    if (!commit) continue;
    const int out = slots_.slot_of[group[i]] >= 0 ? slots_.slot_of[group[i]] : temp_slot(group[i]);
    const std::string res = is_int(d) ? "(" + std::string(compute_type(d)) + ")" + acc : round_to(d, acc);
    stores << "    " << w.store(out, "o", d, res) << "\n";
  }
  // (Unrolled by eight, a single fold ends in up to seven rows waited for one by one: 250 x 300 9.9 us, 6.0 as the compiler
  // unrolls it; products summed over 130 rows 6.6, 4.6. With more arithmetic per row it is the other way round: two
  // folds of 40 sines 7.2 us, 7.8; a softmax's folds of 57 keys 1.4 us more.)
  body << (group.size() > 1 || costly_inside(g_.ops[group[0]].args[0]) ? "#pragma unroll 8\n" : "") << "    for (I r = 0; r < (I)" << nred << "; ++r) {\n" << steps.str() << "    }\n" << stores.str();
  return body.str();
}

std::optional<std::string> Planner::chunk_identity(DType d, Reducer r) {
  if (is_float_domain(d)) return std::string(r == Reducer::sum ? "-0.0f" : "__builtin_nanf(\"\")");
  if (d == DType::f64) return std::string(r == Reducer::sum ? "-0.0" : "__builtin_nan(\"\")");
  if (r == Reducer::sum && (d == DType::i32 || d == DType::u32 || d == DType::i64 || d == DType::u64))
    return "(" + acc_type(d, r) + ")0";
  const bool mx = r == Reducer::max;
  switch (d) {
    case DType::i32: return std::string(mx ? "(-2147483647 - 1)" : "2147483647");
    case DType::u32: return std::string(mx ? "0u" : "4294967295u");
    case DType::i64: return std::string(mx ? "(-9223372036854775807LL - 1)" : "9223372036854775807LL");
    case DType::u64: return std::string(mx ? "0ull" : "18446744073709551615ull");
    default: return std::nullopt;
  }
}

DType Planner::partial_dtype(DType d, Reducer r) {
  if (is_float_domain(d)) return DType::f32;
  if (r == Reducer::sum && d == DType::i32) return DType::u32;
  if (r == Reducer::sum && d == DType::i64) return DType::u64;
  return d;
}

void Planner::fold_chunked(uint32_t v, int out, const Type& in, const std::vector<size_t>& red, const std::vector<size_t>& keep,
                           const std::vector<Dim>& rdims, const std::vector<Dim>& kdims, uint64_t nout, uint64_t nred, Reducer r,
                           DType d) {
  const Op& op = g_.ops[v];
  const uint32_t B = 256;
  // Four adjacent outputs per lane where they are adjacent in the input too; 64 lanes x 4 waves per workgroup,
  // each wave a quarter of the workgroup's chunk, put together in order in LDS. Many outputs one by one take all 256
  // lanes of one chunk instead, so that a workgroup reads whole lines (4000 x 30001 bf16: 66 us, 49; 1000 x 5001 the other way round: 6.7, 8.7).
  const bool flat = kdims.size() == 1 && keep.back() + 1 == in.rank() && nout % 4 == 0;
  const uint64_t parts = !flat && nout >= 8192 && nred > 512 && opt_.allow_split ? 1 : 4, lanes = B / parts;
  const uint64_t VEC = flat ? 4 : 1, tiles = (nout + lanes * VEC - 1) / (lanes * VEC);
  // One launch up to 512 reduced elements (256 x 4096 f32: 4.0 us, 6.0 in two launches); else two workgroups for every CU, of
  // 32 reduced elements each at least, or one of vectors, since the chunks' partials are then folded one by one (100000 x 64
  // f32: 512 chunks 37 us, 256 16; 1000000 x 4 43 and 66). A transcendental per element takes all the waves that there
  // can be (the sines of 300 x 30000 beside their cosines: 67 us in one launch, 33). (3000 x 2048 bf16 summed over 3000: one output per lane and
  // chunks of 256 and more took 24 us in two launches, now 13; 1142 x 1110, one thread per output before, 160 us, now 9.)
  const bool light = !costly_inside(op.args[0]);
  const uint64_t want = flat && light && nred < (1ull << 18) ? 256 : 512;
  uint64_t S = !opt_.allow_split || (light && nred <= 512) ? 1 : std::min<uint64_t>({(want + tiles - 1) / tiles, nred / 32, 65535});
  const uint64_t chunk = (nred + S - 1) / S, quarter = (chunk + parts - 1) / parts;
  S = (nred + chunk - 1) / chunk;
  const DType pd = partial_dtype(d, r);
  const std::string at = acc_type(d, r);
  const int part = S > 1 ? slots_.add(SlotInfo::Temp, -1, pd, S * nout * dtype_size(pd)) : -1;
  {
    KernelWriter w(g_, slots_, itype());
    std::ostringstream body, pre;
    std::vector<std::string> kc = flat ? std::vector<std::string>{"c"} : delinearize("c", kdims), rc = delinearize("r", rdims);
    std::vector<std::string> full(in.rank());
    for (size_t i = 0; i < red.size(); ++i) full[red[i]] = rc[i];
    for (size_t i = 0; i < keep.size(); ++i) full[keep[i]] = kc[i];
    std::string hoisted;
    std::map<std::string, std::string> hoisted_var;
    if (flat)
      w.leaf_hook = [&](int slot, const std::string& off, DType ld, Scope& sc, std::string& res) -> bool {
        const std::optional<std::string> base = quad_base(off);
        if (!base) return false;
        const std::string key = std::to_string(slot) + "|" + off;
        auto hv = hoisted_var.find(key);
        if (hv == hoisted_var.end()) {
          const std::string q = "q" + std::to_string(hoisted_var.size());
          hoisted += "      " + w.quad_load(slot, q, *base, ld) + "\n";
          hv = hoisted_var.emplace(key, q).first;
        }
        res = w.tmp();
        sc.out << sc.indent << "const " << compute_type(ld) << " " << res << " = " << KernelWriter::quad_elem(hv->second, "u", ld) << ";\n";
        return true;
      };
    Scope inner(body, "        ");
    const std::string x = w.value(op.args[0], full, inner);
    body << "        mine[u] = " << serial_fold_step(d, r, "mine[u]", x) << ";\n";
    w.leaf_hook = nullptr;
    Scope outer(pre, "  ");
    const std::string start = S > 1 ? *chunk_identity(d, r) : "(" + at + ")" + w.value(op.args[1], {}, outer);
    const std::string res = is_int(d) ? "(" + std::string(compute_type(d)) + ")acc" : round_to(d, "acc");
    const std::string store = S > 1 ? w.store(part, "s * (I)" + std::to_string(nout) + " + c", pd, "acc") : w.store(out, "c", d, res);
    std::string nm = name(S > 1 ? "fold_chunks" : "fold", v);
    std::ostringstream src;
    src << "extern \"C\" __global__ void __launch_bounds__(" << B << ") " << nm << "(" << w.params() << ") {\n"
        << "  typedef " << w.itype << " I;\n" << w.align_hints() << "  __shared__ " << at << " parts[" << parts << "][" << lanes * VEC << "];\n"
        << "  const I lane = (I)(threadIdx.x & " << lanes - 1 << "), wave = (I)(threadIdx.x / " << lanes << "), s = (I)blockIdx.y;\n"
        << "  const I c0 = ((I)blockIdx.x * " << lanes << " + lane) * " << VEC << ";\n"
        << "  const I last = s * (I)" << chunk << " + (I)" << chunk << " < (I)" << nred << " ? s * (I)" << chunk << " + (I)" << chunk
        << " : (I)" << nred << ";\n"
        << "  const I r0 = s * (I)" << chunk << " + wave * (I)" << quarter << ";\n"
        << "  const I r1 = r0 + (I)" << quarter << " < last ? r0 + (I)" << quarter << " : last;\n"
        << "  " << at << " mine[" << VEC << "];\n#pragma unroll\n  for (int u = 0; u < " << VEC << "; ++u) {\n    const " << at
        << " empty = " << *chunk_identity(d, r) << ";\n    mine[u] = empty;\n  }\n"
        << "  if (c0 < (I)" << nout << ") {\n#pragma unroll 8\n    for (I r = r0; r < r1; ++r) {\n" << hoisted
        << "#pragma unroll\n      for (int u = 0; u < " << VEC << "; ++u) {\n        const I c = c0 + u;\n" << body.str() << "      }\n    }\n  }\n"
        << "#pragma unroll\n  for (int u = 0; u < " << VEC << "; ++u) parts[wave][lane * " << VEC << " + u] = mine[u];\n  __syncthreads();\n"
        << pre.str() << "  for (I i = (I)threadIdx.x; i < " << lanes * VEC << "; i += " << B << ") {\n"
        << "    const I c = (I)blockIdx.x * " << lanes * VEC << " + i;\n    if (c >= (I)" << nout << ") continue;\n    " << at << " acc = " << start
        << ";\n#pragma unroll\n    for (int k = 0; k < " << parts << "; ++k) acc = " << serial_fold_step(d, r, "acc", "parts[k][i]") << ";\n    " << store << "\n  }\n}\n";
    KernelStep k;
    k.source = src.str();
    k.name = nm;
    k.grid[0] = (uint32_t)tiles;
    k.grid[1] = (uint32_t)S;
    k.block[0] = B;
    k.klass = "fold";
    k.label = "fold:%" + std::to_string(v) + (S > 1 ? " chunks" : "");
    push(std::move(k), w);
  }
  if (S == 1) return;
  {
    KernelWriter w(g_, slots_, itype());
    std::ostringstream body;
    Scope outer(body, "    ");
    std::string init = w.value(op.args[1], {}, outer);
    body << "    " << at << " acc = (" << at << ")" << init << ";\n"
         << "#pragma unroll 8\n    for (I s = 0; s < (I)" << S << "; ++s) acc = "
         << serial_fold_step(d, r, "acc", w.load(part, "s * (I)" + std::to_string(nout) + " + o", pd)) << ";\n";
    std::string res = is_int(d) ? "(" + std::string(compute_type(d)) + ")acc" : round_to(d, "acc");
    body << "    " << w.store(out, "o", d, res) << "\n";
    std::string nm = name("fold", v);
    std::ostringstream src;
    src << "extern \"C\" __global__ void __launch_bounds__(" << B << ") " << nm << "(" << w.params() << ") {\n"
        << "  typedef " << w.itype << " I;\n"
        << "  for (I o = (I)blockIdx.x * " << B << " + threadIdx.x; o < (I)" << nout << "; o += (I)gridDim.x * " << B
        << ") {\n" << body.str() << "  }\n}\n";
    KernelStep k;
    k.source = src.str();
    k.name = nm;
    k.grid[0] = grid_for(nout, B, 65536);
    k.block[0] = B;
    k.klass = "fold";
    k.label = "fold:%" + std::to_string(v);
    push(std::move(k), w);
  }
}

// ---- row group: fused reductions over trailing axes of one row space, one workgroup per row ----

bool Planner::row_shape(uint32_t v, RowShape& rs) const {
  const Op& op = g_.ops[v];
  if (op.kind != Kind::reduce) return false;
  const Type& in = g_.type(op.args[0]);
  std::vector<int64_t> red = op.ints;
  std::sort(red.begin(), red.end());
  size_t rank = in.rank(), nr = red.size();
  if (nr == 0) return false;
  for (size_t i = 0; i < nr; ++i)
    if (red[i] != (int64_t)(rank - nr + i)) return false;
  rs.K.assign(in.dims.begin(), in.dims.begin() + (rank - nr));
  rs.T.assign(in.dims.begin() + (rank - nr), in.dims.end());
  DType d = op.result.dtype;
  return is_float_domain(d) || d == DType::f64 || is_int(d);
}

bool Planner::row_group(uint32_t r0) {
  if (!opt_.allow_row) return false;
  RowShape rs;
  if (!row_shape(r0, rs)) return false;
  uint64_t tn = prod(rs.T, 0, rs.T.size()), kn = prod(rs.K, 0, rs.K.size());
  if (tn < 64 || kn == 0) return false;
  RowKernel rk;
  rk.reduces.push_back(r0);
  if (!try_row(rs, rk)) return false;
  size_t n = g_.ops.size();
  for (uint32_t v = r0 + 1; v < n; ++v) {
    if (!live_[v] || done_[v]) continue;
    RowShape o;
    if (g_.ops[v].kind == Kind::reduce && row_shape(v, o) && o.K == rs.K && o.T == rs.T) {
      rk.reduces.push_back(v);
      if (!try_row(rs, rk)) rk.reduces.pop_back();
    }
  }
  std::vector<Dim> full = rs.K;
  full.insert(full.end(), rs.T.begin(), rs.T.end());
  for (uint32_t v = r0 + 1; v < n; ++v) {
    if (!live_[v] || done_[v] || !needed_[v] || !is_inlinable(g_.ops[v].kind)) continue;
    const auto& dims = g_.type(v).dims;
    if (dims == rs.K) {
      rk.row_vals.push_back(v);
      if (!try_row(rs, rk)) rk.row_vals.pop_back();
    } else if (dims == full) {
      rk.full_vals.push_back(v);
      if (!try_row(rs, rk)) rk.full_vals.pop_back();
    }
  }
  // A reduction whose value no other kernel reads stays in the kernel's registers (no slot, no
  // store): C2's row maximum and sum, a norm's sum of squares. (Storing them cost 4.7 µs of C2's
  // 163 µs in a standalone harness.)
  std::set<uint32_t> inside(rk.reduces.begin(), rk.reduces.end());
  inside.insert(rk.row_vals.begin(), rk.row_vals.end());
  inside.insert(rk.full_vals.begin(), rk.full_vals.end());
  for (uint32_t v : rk.reduces)
    if (is_output_[v] || read_outside(v, inside)) temp_slot(v);
  for (uint32_t v : rk.row_vals) temp_slot(v);
  for (uint32_t v : rk.full_vals) temp_slot(v);
  KernelStep k = gen_row(rs, rk, true);
  push_row(std::move(k));
  for (uint32_t v : rk.reduces) finish(v);
  for (uint32_t v : rk.row_vals) finish(v);
  for (uint32_t v : rk.full_vals) finish(v);
  return true;
}

void Planner::push_row(KernelStep k) {
  share_reductions(k.source);
  k.args = last_args_;
  double bytes = 0;
  for (int s : k.args) bytes += (double)plan_.slots[(size_t)s].bytes;
  k.algorithmic_bytes = bytes;
  Step st;
  st.type = Step::Kernel;
  st.kernel = std::move(k);
  plan_.steps.push_back(std::move(st));
}

bool Planner::try_row(const RowShape& rs, const RowKernel& rk) {
  try {
    gen_row(rs, rk, false);
    return true;
  } catch (const NotFusable&) {
    return false;
  }
}

std::vector<int> Planner::reduction_passes(const RowKernel& rk) const {
  std::vector<int> pass(rk.reduces.size(), 0);
  std::map<uint32_t, int> needs;  // value: the first pass that can evaluate it
  std::function<int(uint32_t)> first_pass = [&](uint32_t v) -> int {
    const auto known = needs.find(v);
    if (known != needs.end()) return known->second;
    int p = 0;
    const auto own = std::find(rk.reduces.begin(), rk.reduces.end(), v);
    if (own != rk.reduces.end()) {
      p = pass[(size_t)(own - rk.reduces.begin())] + 1;
    } else if (is_inlinable(g_.ops[v].kind) && slots_.available(v) < 0) {
      for (uint32_t a : g_.ops[v].args) p = std::max(p, first_pass(a));
    }
    return needs[v] = p;
  };
  for (size_t j = 0; j < rk.reduces.size(); ++j)  // in program order: what j reads comes before it
    for (uint32_t a : g_.ops[rk.reduces[j]].args) pass[j] = std::max(pass[j], first_pass(a));
  return pass;
}

bool Planner::row_leaves_16bit() const {
  for (const auto& [key, uses] : probe_use_) {
    const DType d = plan_.slots[std::stoul(key)].dtype;  // keys are "slot|offset"
    const bool row_major = quad_base(key.substr(key.find('|') + 1)).has_value();
    if (uses.size() >= 2 && !(row_major && (d == DType::bf16 || d == DType::f16))) return false;
  }
  return true;
}

bool Planner::costly(uint32_t v) const {
  const Op& op = g_.ops[v];
  if (op.kind == Kind::binary) return (Binary)op.code == Binary::div || (Binary)op.code == Binary::pow;
  return op.kind == Kind::unary && (Unary)op.code != Unary::neg && (Unary)op.code != Unary::abs;
}

bool Planner::costly_inside(uint32_t v) const {
  std::set<uint32_t> seen;
  std::function<bool(uint32_t)> walk = [&](uint32_t x) {
    if (!seen.insert(x).second || slots_.available(x) >= 0 || !is_inlinable(g_.ops[x].kind)) return false;
    return costly(x) || std::any_of(g_.ops[x].args.begin(), g_.ops[x].args.end(), walk);
  };
  return walk(v);
}

uint64_t Planner::row_registers(uint64_t per_thread, bool pairs) const {
  std::map<int, uint64_t> live;  // pass: registers holding values needed after it
  auto count = [&](const std::set<int>& uses, bool bits16) {
    for (int p = *uses.begin(); p < *uses.rbegin(); ++p) live[p] += pairs && bits16 ? per_thread / 2 : per_thread;
  };
  for (const auto& leaf : probe_use_) count(leaf.second, dtype_size(plan_.slots[std::stoul(leaf.first)].dtype) == 2);
  for (const auto& kept : row_keep_) {
    const auto uses = probe_values_.find(kept.first);
    if (uses != probe_values_.end()) count(uses->second, dtype_size(g_.type(kept.first).dtype) == 2);
  }
  uint64_t most = 0;
  for (const auto& pass : live) most = std::max(most, pass.second);
  return most;
}

// Values of the whole row that cost more than a register to evaluate again (a transcendental, a division) and
// that a later pass reads too: the pass that computes them first leaves them in registers, as a row
// read by several passes is. The outermost such value is taken first (what it was computed from is
// then often not read again), while the arrays live between two passes hold at most 64 registers per
// thread. (Cross-entropy with its gradient, 2048 x 50257 bf16, whose gradient reads the exponentials: 217 us
// with one row to a CU, evaluated twice or kept, as its loads, arithmetic and stores then take turns;
// 151 us kept, in pairs, with two rows to a CU.)
void Planner::keep_row_values(const RowShape& rs, const RowKernel& rk, uint64_t per_thread, bool pairs) {
  std::set<uint32_t> refused;
  for (int round = 0; round < 8; ++round) {
    uint32_t best = 0;
    bool found = false;
    for (const auto& [v, uses] : probe_values_) {
      if (uses.size() < 2 || row_keep_.count(v) || refused.count(v) || !costly(v)) continue;
      best = v;  // in program order: the last is the outermost
      found = true;
    }
    if (!found) return;
    row_keep_[best] = *probe_values_.at(best).begin();
    gen_row(rs, rk, false);
    if (row_registers(per_thread, pairs) > 64) {
      row_keep_.erase(best);
      refused.insert(best);
      gen_row(rs, rk, false);
    }
  }
}

KernelStep Planner::gen_row(const RowShape& rs, const RowKernel& rk, bool commit) {
  uint64_t tn = prod(rs.T, 0, rs.T.size()), kn = prod(rs.K, 0, rs.K.size());
  // Reductions that need no other's result share one pass over the row: pass_of[j] is one more than the
  // latest pass whose result reduction j reads. (A pass for each made every one of them load, or keep
  // in registers, the same row and evaluate the same elementwise values again: the mismatch and its
  // slope over 8192 x 16384 took 694 us in two passes of a cached, fully unrolled row, 82 us in one.)
  const std::vector<int> pass_of = reduction_passes(rk);
  const int reduce_passes = 1 + *std::max_element(pass_of.begin(), pass_of.end());
  const size_t passes = (size_t)reduce_passes + (rk.full_vals.empty() ? 0 : 1);
  // Four consecutive elements per thread, also of rows whose length is no multiple of four (their vectors
  // begin at any element). Shorter ones than one vector per lane of a wave keep one element per thread
  // (30000 rows of 67 f16: 7.4 us against 9.0 with 17 of 64 lanes at work), rows of several axes too, and of several
  // passes those whose second iteration is mostly a partial one (layernorm of 100000 rows of 510 f32: 92 us in vectors,
  // 75; of 300: 48, 53; of 514: 75, 167).
  const bool flat = rs.T.size() == 1, partly = passes >= 2 && tn > 320 && tn < 512;
  const uint32_t VEC = tn % 4 == 0 || (flat && tn >= 256 && !partly) ? 4 : 1;
  uint64_t lanes = (tn + VEC - 1) / VEC;
  // Two waves per row: against one workgroup of four waves per row, C2's logsumexp went from 163-165 to
  // 159-161 µs and C1's tone from 58 to 56 µs on one box (four rounds), 162.0 -> 159.0 and 53.4 ->
  // 52.3 µs on another, and C2 161.5 -> 162.9 (C1 51.0 -> 50.2) on a third; 512 threads helped C2
  // alike but slowed C1 by 4 %, 1024 slowed C2 by 40 %. More workgroups per CU are in flight, each
  // meeting two waves at its barriers instead of four.
  uint32_t B = lanes >= 128 ? 128 : (uint32_t)std::max<uint64_t>(64, (lanes + 63) / 64 * 64);
  uint64_t E = (tn + (uint64_t)B * VEC - 1) / ((uint64_t)B * VEC);
  if (commit) {
    row_keep_.clear();
    gen_row(rs, rk, false);  // what the passes read
  }
  // Elements of a row that a thread may keep in registers: 64. 16-bit rows too long for that are kept two
  // elements to a register, up to 104 of them (with 128 the addresses and sums beside them spill:
  // 4096 x 32000 bf16 cross-entropy took 264 us with 256 threads of 128, 174 us with 512 of 64), or 128
  // where a row has no shorter share. 256 threads keep 64 also in pairs: two rows that a gradient reads would take 104
  // registers of each thread (us, 256 threads of 104 / 512 of 64: gradient of a softmax 1000 x 20000 bf16 52 / 35,
  // 3000 x 24000 160 / 113, of a layer norm 1000 x 20000 50 / 46, 3000 x 24000 158 / 166).
  const bool pairs_ok = commit && VEC == 4 && flat && row_leaves_16bit();
  auto keepable = [&](uint32_t threads) -> uint64_t { return !pairs_ok || threads <= 256 ? 64 : threads == 1024 ? 128 : 104; };
  // No more rows than CUs: as many threads per row as have a vector each, up to 1024, so that a CU has more than two
  // waves. (us a pass, 128 threads / now: logsumexp 1 x 100000 f32 61 / 14, tone 200 x 16384 19.2 / 7.7, 1 x 8395 10.1 /
  // 7.7; rows that 128 threads keep in registers stay at a launch's 7.3.) The line is where rows outnumber the CUs, not
  // where it pays: 512 threads are faster for up to about 1000 long rows as well (128 / 512: tone 300 x 16384 19.2 / 8.0,
  // 1000 x 16384 18.2 / 14.4, logsumexp 500 x 8192 5.8 / 4.1, but 2000 x 4096 6.5 / 7.0).
  // Up to 1024 rows that one pass reads take 256 or 512 threads with four vectors each: 128 threads hold the waves of
  // one or two rows per SIMD (sum, sum of squares and maximum, 128 / now: 500 x 32000 f32 22.4 / 11.2, bf16 21.9 / 9.8,
  // 1000 x 9000 f32 12.8 / 8.1; with fewer vectors each it loses, 600 x 6000 5.0 / 5.9).
  if (kn <= 256 || (passes == 1 && kn <= 1024))
    for (uint32_t wide : {1024u, 512u, 256u})
      if (kn <= 256 ? lanes >= wide : wide <= 512 && lanes >= 4 * wide) {
        B = wide;
        E = (tn + (uint64_t)B * VEC - 1) / ((uint64_t)B * VEC);
        break;
      }
  // A row read by several passes is kept in registers when each thread holds at most 64 (128) of its
  // elements; a row too long for that with 128 threads takes 256, 512 or 1024 threads if that makes it
  // fit (read once instead of once per pass; four waves per SIMD still have 128 registers each).
  if (passes >= 2 && E * VEC > keepable(B)) {
    for (uint32_t wide : {256u, 512u, 1024u}) {
      const uint64_t e = (tn + (uint64_t)wide * VEC - 1) / ((uint64_t)wide * VEC);
      if (e * VEC <= keepable(wide)) {
        B = wide;
        E = e;
        break;
      }
    }
  }
  // Short rows, many of them: one wave per row and four rows per workgroup. The row's reductions then
  // stay inside the wave (no LDS exchange, no barrier), and a CU keeps up to 32 rows in flight instead
  // of one row per workgroup of four waves. (A C5 RMS norm: 8192 rows of 2048 bf16.)
  uint32_t R = 1;
  if (lanes <= 512 && kn >= 4 * 256) {
    R = 4;
    B = 64;
    E = (tn + (uint64_t)B * VEC - 1) / ((uint64_t)B * VEC);
  }
  const std::string tid = R > 1 ? "(I)(threadIdx.x & 63)" : "(I)threadIdx.x";
  bool unrolled = E * VEC <= (passes >= 2 ? keepable(B) : 64);
  const bool pairs = pairs_ok && E * VEC > 64;  // (pairs cost an operation per element and pass)
  bool cache = unrolled && passes >= 2;
  // Where the threads' vectors do not cover the row exactly, the last iteration is written apart: its
  // vectors past the end move back to the last four elements, and the elements another vector holds are
  // skipped (c < cr). Every other iteration loads and stores whole vectors without a test. (Each
  // element tested and loaded by itself, as a row of several axes still is: cross-entropy and its
  // gradient over 2048 rows of 50257 bf16 took 681 us, now 151.)
  const bool partial = tn % ((uint64_t)B * VEC) != 0, tail = partial && flat && VEC == 4, guard = partial && !tail;
  const uint64_t whole = tail ? tn / ((uint64_t)B * VEC) : E;  // iterations without a test
  const bool any = tn % 4 != 0;
  KernelWriter w(g_, slots_, itype());
  std::vector<std::string> kc = delinearize("row", rs.K);
  std::vector<std::string> tc = delinearize("c", rs.T);
  std::vector<std::string> full = kc;
  full.insert(full.end(), tc.begin(), tc.end());
  // Row-varying leaves loaded by more than one pass are kept in registers.
  std::map<std::string, std::set<int>> leaf_use;
  std::map<std::string, std::string> leaf_array;
  std::map<std::string, int> leaf_first;
  int cur_pass = 0;
  uint64_t registers = 0;  // of the row, per thread
  std::string decls;
  std::set<std::string> declared;
  if (commit) {
    if (cache) keep_row_values(rs, rk, E * VEC, pairs);
    registers = row_registers(E * VEC, pairs);
    leaf_use = probe_use_;
    int na = 0;
    for (auto& [key, uses] : leaf_use) {
      if (cache && uses.size() >= 2) {
        leaf_array[key] = "cache" + std::to_string(na++);
        leaf_first[key] = *uses.begin();
      }
    }
  }
  std::map<std::string, std::set<int>> use_record;
  std::map<uint32_t, std::set<int>> value_use;
  // A load whose offset is `rest + c` (c the row's element index, rank-1 row) is written as
  // (ptr + rest + c0)[u] so that the VEC adjacent loads of one thread merge into one vector load.
  // The `rest` of an offset `(rest + c)` (empty optional when the offset has another form).
  auto row_rest = [&](const std::string& off) -> std::optional<std::string> {
    if (VEC == 1 || tc.size() != 1 || tc[0] != "c") return std::nullopt;
    return quad_base(off);
  };
  auto direct_load = [&](int slot, const std::string& off, DType d) -> std::string {
    const std::optional<std::string> base = row_rest(off);
    return base ? w.load_at(slot, *base, "u", d) : w.load(slot, off, d);
  };
  // Without a tail guard, a leaf read at `rest + c` is loaded for the thread's VEC elements at once,
  // at the top of the element iteration (one aligned vector load per input, issued before any of
  // the iteration's arithmetic), and each element takes its lane.
  const bool hoist = VEC == 4 && !guard;
  std::string hoisted;
  std::map<std::string, std::string> hoisted_var;
  int nquad = 0;
  // A leaf is streamed (loaded with the non-temporal hint) when this kernel reads each of its
  // elements exactly once: its buffer holds as many elements as the kernel's rows x row length and
  // its offset depends on the row (a buffer reached through broadcast_in_dim covers a subset of the
  // loop's axes, so an equal element count means no axis is broadcast and no element is shared
  // between rows), and one pass reads it (or the row is cached in registers after the first).
  auto mentions_row = [](const std::string& off) {
    for (size_t p = off.find("row"); p != std::string::npos; p = off.find("row", p + 1)) {
      const bool start = p == 0 || !(isalnum((unsigned char)off[p - 1]) || off[p - 1] == '_');
      const bool end = p + 3 == off.size() || !(isalnum((unsigned char)off[p + 3]) || off[p + 3] == '_');
      if (start && end) return true;
    }
    return false;
  };
  auto streamed = [&](int slot, const std::string& off, DType d, const std::string& key) {
    if (!commit) return false;
    const auto use = leaf_use.find(key);
    const bool once = leaf_array.count(key) > 0 || (use != leaf_use.end() && use->second.size() == 1);
    const uint64_t elems = plan_.slots[(size_t)slot].bytes / dtype_size(d);
    return once && elems == kn * tn && mentions_row(off);
  };
  auto reread = [](const std::string& array) {
    return "      accy::opaque(" + array + "[e * 2]);\n      accy::opaque(" + array + "[e * 2 + 1]);\n";
  };
  // The hoisted vector load of a leaf for this iteration (emitted once per pass), as the lane `u`.
  auto hoisted_elem = [&](int slot, const std::string& base, DType d, const std::string& key, bool stream) {
    auto hv = hoisted_var.find(key);
    if (hv == hoisted_var.end()) {
      std::string q = "q" + std::to_string(nquad++);
      hoisted += "      " + w.quad_load(slot, q, base, d, stream, any) + "\n";
      hv = hoisted_var.emplace(key, q).first;
    }
    return KernelWriter::quad_elem(hv->second, "u", d);
  };
  w.leaf_hook = [&](int slot, const std::string& off, DType d, Scope& sc, std::string& out) -> bool {
    bool varies = false;
    for (const auto& t : tc)
      if (t != "0" && off.find(t) != std::string::npos) varies = true;
    if (!varies) return false;
    std::string key = std::to_string(slot) + "|" + off;
    use_record[key].insert(cur_pass);
    auto it = leaf_array.find(key);
    if (it == leaf_array.end()) {
      std::string t = w.tmp();
      std::optional<std::string> base = hoist ? row_rest(off) : std::nullopt;
      std::string val = base ? hoisted_elem(slot, *base, d, key, streamed(slot, off, d, key)) : direct_load(slot, off, d);
      sc.out << sc.indent << "const " << compute_type(d) << " " << t << " = " << val << ";\n";
      out = t;
      return true;
    }
    std::string elem = it->second + "[e * " + std::to_string(VEC) + " + u]";
    const std::optional<std::string> pair_base = pairs && hoist && dtype_size(d) == 2 && is_float_domain(d) ? row_rest(off) : std::nullopt;
    if (pair_base) {
      // two 16-bit elements to a register, filled from the vector load at the top of the first pass's iteration
      if (leaf_first[key] == cur_pass && !hoisted_var.count(key)) {
        hoisted_elem(slot, *pair_base, d, key, streamed(slot, off, d, key));
        for (int i = 0; i < 2; ++i)
          hoisted += "      " + it->second + "[e * 2 + " + std::to_string(i) + "] = accy::pair_of(" + hoisted_var[key] + ", " + std::to_string(i) + ");\n";
        if (declared.insert(key).second) decls += "    u32_t " + it->second + "[" + std::to_string(E * 2) + "];\n";
      }
      if (leaf_first[key] != cur_pass && !hoisted_var.count(key)) {
        hoisted += reread(it->second);
        hoisted_var.emplace(key, it->second);
      }
      out = w.tmp();
      sc.out << sc.indent << "const float " << out << " = accy::" << (d == DType::bf16 ? "bf16_of(" : "f16_of(") << it->second
             << "[e * 2 + (u >> 1)], u);\n";
      return true;
    }
    if (leaf_first[key] == cur_pass) {
      // The cache is filled by the first pass; a streamed leaf through the hoisted vector load.
      const bool stream = streamed(slot, off, d, key);
      std::optional<std::string> base = hoist && (stream || tail) ? row_rest(off) : std::nullopt;
      sc.out << sc.indent << elem << " = " << (base ? hoisted_elem(slot, *base, d, key, stream) : direct_load(slot, off, d))
             << ";\n";
      if (declared.insert(key).second)
        decls += "    " + std::string(compute_type(d)) + " " + it->second + "[" + std::to_string(E * VEC) + "];\n";
    }
    out = elem;
    return true;
  };
  std::vector<std::string> red_var(rk.reduces.size());
  int passes_done = 0;
  w.provide = [&](uint32_t vid, const std::vector<std::string>& coords, std::string& out) -> bool {
    for (size_t j = 0; j < rk.reduces.size(); ++j) {
      if (rk.reduces[j] != vid) continue;
      if (pass_of[j] >= passes_done || coords != kc) throw NotFusable("reduction used outside its row");
      out = red_var[j];
      return true;
    }
    const Op& op = g_.ops[vid];
    if (!is_inlinable(op.kind) && slots_.available(vid) < 0) throw NotFusable("value not produced yet");
    if (coords == full && slots_.available(vid) < 0) {
      const auto kept = row_keep_.find(vid);
      if (kept != row_keep_.end() && cur_pass > kept->second) {
        value_use[vid].insert(cur_pass);
        const std::string array = "kept" + std::to_string(vid);
        const DType d = g_.type(vid).dtype;
        if (pairs && dtype_size(d) == 2 && is_float_domain(d) && hoisted_var.emplace(array, array).second) hoisted += reread(array);
        if (pairs && dtype_size(d) == 2 && is_float_domain(d))
          out = std::string(d == DType::bf16 ? "accy::bf16_of(" : "accy::f16_of(") + array + "[e * 2 + (u >> 1)], u)";
        else
          out = array + "[e * " + std::to_string(VEC) + " + u]";
        return true;
      }
      value_use[vid].insert(cur_pass);
    }
    return false;
  };
  std::ostringstream body;
  // The values kept for later passes, once the pass that computes them has done so.
  auto emit_kept = [&](std::ostringstream& to, Scope& sc) {
    for (const auto& [vid, pass] : row_keep_) {
      if (pass != cur_pass) continue;
      const std::string x = w.value(vid, full, sc), array = "kept" + std::to_string(vid);
      const DType d = g_.type(vid).dtype;
      if (pairs && dtype_size(d) == 2 && is_float_domain(d)) {  // rounded already: its 16 bits hold it exactly
        to << sc.indent << "accy::put_half(" << array << "[e * 2 + (u >> 1)], u, " << KernelWriter::bits(d, x) << ");\n";
        decls += "    u32_t " + array + "[" + std::to_string(E * 2) + "] = {};\n";
        continue;
      }
      to << sc.indent << array << "[e * " << VEC << " + u] = " << x << ";\n";
      decls += "    " + std::string(compute_type(d)) + " " + array + "[" + std::to_string(E * VEC) + "];\n";
    }
  };
  // Element loop: fully unrolled when the thread's elements are cached in registers across passes;
  // otherwise unrolled by a few iterations (all of them would keep every hoisted load live at once).
  // Launch candidates when not cached: the unroll factor (first = default); the source carries a
  // placeholder until the candidate is chosen.
  static const char* const kUnrollMark = "#pragma unroll ACCY_ELEMENT_UNROLL\n";
  const std::vector<int> unroll_candidates =
      cache ? std::vector<int>{0} : (unrolled ? std::vector<int>{4, 2, 1, 8} : std::vector<int>{2, 1, 4});
  std::string unroll = cache ? "#pragma unroll\n" : kUnrollMark;
  // A wide row's passes each compute their own offsets (carried from pass to pass they would take as many
  // registers as the row: 316 bytes of scratch for the loss above). A row of 256 threads carries them, unless its last
  // iteration is incomplete or it keeps 65 to 112 registers: us, computed / carried, for 1500 x 16384 f32 (whole, 128
  // to 192 registers) gradients of a softmax 66 / 55, of a layer norm 140 / 64, 1000 x 12288 bf16 softmax 35 / 21; for
  // 1000 x 12288 f32 (whole, 96) softmax 29 / 35; for 2000 x 16000 bf16 (incomplete, 192) layer norm 59 / 90.
  // Whole rows of 144 registers go either way (1000 x 12288 f32: layer norm 43 / 37, RMS norm 28 / 35).
  const bool wide = cache && (B >= 512 || (B == 256 && (tail || (registers > 64 && registers <= 112))));
  const std::string first_elem = "((I)e * " + std::to_string(B) + " + " + tid + ") * " + std::to_string(VEC);
  const std::string vec_elem = wide ? "(I)e * " + std::to_string(B * VEC) + " + t0" : first_elem;
  const std::string head = "      const I c0 = " + vec_elem + ";\n";
  const std::string elements = "#pragma unroll\n      for (int u = 0; u < " + std::to_string(VEC) + "; ++u) {\n        const I c = c0 + u;\n";
  // One element loop: the pass's hoisted loads, the per-element code and what follows a vector's elements;
  // then the last iteration with its own per-element code.
  auto emit_loop = [&](const std::string& inner_code, const std::string& after, const std::string& tail_code) {
    if (wide)
      body << "    {\n    u32_t t = threadIdx.x * " << VEC << "u;\n    accy::opaque(t);\n    const I t0 = (I)(t & " << B * VEC - 1 << "u);\n";
    if (whole)
      body << unroll << "    for (int e = 0; e < " << whole << "; ++e) {\n" << head << hoisted << elements
           << (guard ? "        if (c < (I)" + std::to_string(tn) + ") {\n" : "") << inner_code
           << (guard ? "        }\n      }\n" : "      }\n") << after
           << (wide && cur_pass > 0 ? "      __builtin_amdgcn_sched_barrier(0);\n" : "") << "    }\n";
    if (tail)
      body << "    {\n      const int e = " << whole << ";\n      const I cr = " << vec_elem << ", c0 = cr < (I)" << tn - VEC << " ? cr : (I)" << tn - VEC << ";\n"
           << hoisted << elements << "        if (c >= cr) {\n" << tail_code << "        }\n      }\n    }\n";
    if (wide) body << "    }\n";
    hoisted.clear();
    hoisted_var.clear();
  };
  std::string lds_decl;
  for (cur_pass = 0; cur_pass < reduce_passes; ++cur_pass) {
    std::ostringstream ib;
    Scope inner(ib, guard ? "          " : "        ");
    for (size_t j = 0; j < rk.reduces.size(); ++j) {
      if (pass_of[j] != cur_pass) continue;
      const Op& op = g_.ops[rk.reduces[j]];
      Reducer r = (Reducer)op.code;
      DType d = op.result.dtype;
      std::string at = acc_type(d, r);
      Scope pre(body, "    ");
      std::string init = w.value(op.args[1], {}, pre);
      std::string acc = "acc" + std::to_string(j);
      // Every thread folds its share of the row, then the shares are combined. max / min may start
      // every share from the init (it is idempotent under them); a sum takes the init once, in the
      // first thread's share, and the others start from the additive identity (-0 for floats, so
      // that a share of -0 elements stays -0).
      if (r == Reducer::sum) {
        const std::string zero = is_int(d) ? "(" + at + ")0" : (d == DType::f64 ? "-0.0" : "-0.0f");
        body << "    " << at << " " << acc << " = " << tid << " == 0 ? (" << at << ")" << init << " : " << zero << ";\n";
      } else {
        body << "    " << at << " " << acc << " = (" << at << ")" << init << ";\n";
      }
      std::string x = w.value(op.args[0], full, inner);
      ib << inner.indent << acc << " = " << fold_step(d, r, acc, x) << ";\n";
    }
    emit_kept(ib, inner);
    emit_loop(ib.str(), "", ib.str());
    for (size_t j = 0; j < rk.reduces.size(); ++j) {
      if (pass_of[j] != cur_pass) continue;
      const Op& op = g_.ops[rk.reduces[j]];
      Reducer r = (Reducer)op.code;
      DType d = op.result.dtype;
      std::string acc = "acc" + std::to_string(j);
      std::string lds = "lds" + std::to_string(j);
      lds_decl += "  __shared__ " + acc_type(d, r) + " " + lds + "[" + std::to_string(std::max<uint32_t>(B / 64, 1)) + "];\n";
      body << "    " << acc << " = accy::block_reduce<" << B << ">(" << acc << ", " << reducer_op(r) << ", " << lds
           << ");\n";
      red_var[j] = "red" + std::to_string(j);
      std::string res = is_int(d) ? "(" + std::string(compute_type(d)) + ")" + acc : round_to(d, acc);
      body << "    const " << compute_type(d) << " " << red_var[j] << " = " << res << ";\n";
      if (commit && slots_.slot_of[rk.reduces[j]] >= 0)
        body << "    if (" << tid << " == 0) " << w.store(slots_.slot_of[rk.reduces[j]], "row", d, red_var[j]) << "\n";
    }
    passes_done = cur_pass + 1;
  }
  if (!rk.row_vals.empty()) {
    body << "    if (" << tid << " == 0) {\n";
    Scope sc(body, "      ");
    for (uint32_t v : rk.row_vals) {
      std::string x = w.value(v, kc, sc);
      if (commit) body << "      " << w.store(slots_.slot_of[v], "row", g_.type(v).dtype, x) << "\n";
    }
    body << "    }\n";
  }
  if (!rk.full_vals.empty()) {
    cur_pass = reduce_passes;
    std::ostringstream ib;
    Scope sc(ib, guard ? "          " : "        ");
    std::string after, tail_stores;
    for (size_t i = 0; i < rk.full_vals.size(); ++i) {
      const uint32_t v = rk.full_vals[i];
      std::string x = w.value(v, full, sc);
      if (!commit) continue;
      const DType d = g_.type(v).dtype;
      const std::string store = sc.indent + w.store(slots_.slot_of[v], "row * (I)" + std::to_string(tn) + " + c", d, x) + "\n";
      if (!tail) {
        ib << store;
        continue;
      }
      // whole vectors are stored at once after their elements, the last iteration's element by element
      const std::string q = "out" + std::to_string(i), type = std::string(any ? "accy::QuadAny<" : "accy::Quad<") + storage_type(d) + ">";
      ib << sc.indent << q << ".v[u] = " << KernelWriter::bits(d, x) << ";\n";
      hoisted += "      " + type + " " + q + ";\n";
      after += "      *(" + type + "*)(" + w.arg(slots_.slot_of[v], true) + " + row * (I)" + std::to_string(tn) + " + c0) = " + q + ";\n";
      tail_stores += store;
    }
    emit_loop(ib.str(), after, ib.str() + tail_stores);
  }
  probe_use_ = use_record;
  probe_values_ = value_use;
  KernelStep k;
  if (!commit) return k;
  row_keep_.clear();
  std::string nm = name("row", rk.reduces[0]);
  std::ostringstream src;
  // A wide row kept in registers: four waves per SIMD, so that two workgroups of 512 threads share a CU and
  // one computes while the other loads or stores. Not where the row itself takes the 128 registers that this leaves a
  // thread (us, four waves / the compiler's choice: layer norm's gradient 3000 x 32000, 192 registers, f32 450 / 322,
  // bf16 380 / 223; with 120 and 512 threads 1000 x 20000 f32 58 / 67; softmax's 2000 x 16000 bf16, 128 and 256 threads,
  // 70 / 54).
  const bool four_waves = wide && registers <= (B >= 512 ? 128 : 112);
  src << "extern \"C\" __global__ void __launch_bounds__(" << B * R << ") "
      << (four_waves ? "__attribute__((amdgpu_waves_per_eu(4))) " : "") << nm << "(" << w.params() << ") {\n"
      << "  typedef " << w.itype << " I;\n" << w.align_hints() << lds_decl;
  if (R > 1)
    src << "  for (I row = (I)blockIdx.x * " << R << " + (I)(threadIdx.x >> 6); row < (I)" << kn
        << "; row += (I)gridDim.x * " << R << ") {\n";
  else if (wide && kn <= (1u << 20))
    // one row per workgroup; written as a loop, every vector's address is carried across it in registers
    src << "  {\n    const I row = blockIdx.x;\n";
  else
    src << "  for (I row = blockIdx.x; row < (I)" << kn << "; row += gridDim.x) {\n";
  src << decls << body.str() << "  }\n}\n";
  k.source = src.str();
  k.grid[0] = (uint32_t)std::min<uint64_t>((kn + R - 1) / R, 1u << 20);
  if (unroll_candidates.size() > 1) {
    k.tuning_key = tuning_key("row", k.source, "rows=" + std::to_string(kn) + ",cols=" + std::to_string(tn));
    k.candidate_count = (uint32_t)unroll_candidates.size();
    k.candidate = candidate_for(k.tuning_key, k.candidate_count);
    const std::string pragma = "#pragma unroll " + std::to_string(unroll_candidates[k.candidate]) + "\n";
    for (size_t at = k.source.find(kUnrollMark); at != std::string::npos; at = k.source.find(kUnrollMark, at))
      k.source.replace(at, std::strlen(kUnrollMark), pragma);
  }
  k.name = nm;
  k.block[0] = B * R;
  k.klass = "row";
  k.label = "row:%" + std::to_string(rk.reduces[0]);
  last_args_ = w.args;
  return k;
}

}  // namespace planning
}  // namespace accy
