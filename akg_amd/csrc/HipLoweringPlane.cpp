/**
 * Reductions over axes on both sides of the kept ones whose results meet the tensor again: a training batch norm over
 * N, H and W of [N, C, H, W] (family `plane_reduce`).
 *
 * The tensor is seen as [RO, K, RI]: channel k of the K kept ones is RO runs of RI adjacent elements. The streaming
 * reductions keep nothing of what they read, so such a description took one kernel per reduction, one per value made
 * of the sums and one for the result (five launches for a batch norm, the tensor read three times). Two forms here:
 *   one workgroup per channel: every chunk of the channel is loaded once, all loads in flight together, and stays in
 *     registers as it came from memory; every level of reductions is one walk over the resident chunks, the last walk
 *     stores the results. One launch, one read, one write.
 *   several workgroups per channel (a channel that the registers of a workgroup do not hold, or too few channels to
 *     keep the chip busy): one launch per level, whose workgroups read their part, the partial results of the levels in
 *     front (folded anew by every workgroup, in a fixed order) and leave their own. No counters, no atomics; what
 *     follows from the sums is computed where it is used.
 * A run whose length the chunk does not divide is walked in slots, the last one starting at RI - V; the elements it
 * shares with its neighbour are left out of the reductions and stored twice with the same value.
 *
 * Combiners and initial values are the reference's (MindSporeToLinalg.cpp:791-901); sums whose steps round (16-bit
 * floats) or wrap (narrow integers) are refused and run as before.
 */
#include <algorithm>
#include <sstream>

#include "HipLowering.h"

namespace akg {

namespace {

using lowering::computeTypeName;
using lowering::dtypeTag;

// How a tensor lies in [RO, K, RI]: one value, one per channel (with the reduced axes kept as 1, or dropped), all.
enum class Span { Scalar, Kept, Dropped, Full };

class PlaneEmitter {
 public:
  PlaneEmitter(const OpGraph &g, const LoweringOptions &o) : g_(g), opt_(o) {}

  LoweredKernel run() {
    analyse();
    pickSchedule();
    LoweredKernel k;
    k.kernelName = g_.name + "_kernel";
    src_ << "// Generated by the akg HIP lowering for gfx950. Op description: " << g_.name << "\n";
    src_ << "// family: plane_reduce, fusion class: " << operatorTemplateName(g_.operatorTemplate) << "\n";
    src_ << "#include \"akg_rt.hpp\"\n\n";
    if (parts_ == 0) {
      emitKernel(k.kernelName, 0, lastWalk_);
      k.grid[0] = static_cast<unsigned>(kept_);
    } else {
      for (int w = 0; w < lastWalk_; ++w) {
        KernelPhase phase;
        phase.kernelName = g_.name + "_level" + std::to_string(w);
        phase.grid[0] = static_cast<unsigned>(kept_ * parts_);
        phase.block[0] = static_cast<unsigned>(block_);
        emitKernel(phase.kernelName, w, w);
        k.earlierPhases.push_back(phase);
      }
      emitKernel(k.kernelName, lastWalk_, lastWalk_);
      k.grid[0] = static_cast<unsigned>(kept_ * (fullOutputs_ ? parts_ : 1));
      k.workspaceBytes = workspaceBytes_;
    }
    k.source = src_.str();
    k.family = KernelFamily::PlaneReduce;
    k.block[0] = static_cast<unsigned>(block_);
    k.algorithmicBytes = lowering::countAlgorithmicBytes(g_);
    k.shapeArgs = lowering::buildShapeArgs(g_);
    std::ostringstream note;
    note << "plane_reduce channels=" << kept_ << " runs=" << outer_ << "x" << inner_ << " vec=" << vec_
         << (overlap_ ? " (overlapping last chunk)" : "") << " block=" << block_ << " chunks/thread=" << chunks_
         << " levels=" << lastWalk_ << " workgroups/channel=" << std::max<int64_t>(1, parts_)
         << (parts_ == 0 ? " (resident)" : "") << " workspace=" << workspaceBytes_;
    k.scheduleNote = note.str();
    return k;
  }

 private:
  struct Val {
    bool defined = false;
    bool full = false;
    std::string ident;
  };

  const OpGraph &g_;
  const LoweringOptions &opt_;
  std::ostringstream src_;
  std::vector<int64_t> full_;      // shape of the reduced tensor
  std::vector<bool> reduced_;      // per dim of full_: a reduced one with more than one element
  int64_t outer_ = 1, kept_ = 1, inner_ = 1;
  std::vector<Span> span_;         // per tensor
  std::vector<int> level_;
  std::vector<bool> relaxed_;
  std::vector<Val> vals_;
  int lastWalk_ = 0;               // walks 0 .. lastWalk_: one per level of reductions, the last one stores
  bool fullOutputs_ = false;
  int vec_ = 8, block_ = 256, chunks_ = 1, overlap_ = 0;
  bool keepsUnpacked_ = false;     // the elements of a channel stay in registers as they are computed with, from walk to walk
  bool chunkBranch_ = false;       // a chunk beyond the channel is left out by a branch, not element by element
  int64_t slots_ = 1, parts_ = 0;  // slots of a run; workgroups per channel of the form with one launch per level (0: one, resident)
  std::vector<uint64_t> partialAt_;   // per tensor: byte offset of a reduction's partial results in the workspace
  uint64_t workspaceBytes_ = 0;
  int reduceCount_ = 0;

  void line(const std::string &s) { src_ << s << "\n"; }
  static bool isExtremum(const lowering::ReduceSpec &spec) { return spec.combiner == "akg::RedMax" || spec.combiner == "akg::RedMin"; }
  static std::string id(const char *prefix, int t) { return std::string(prefix) + std::to_string(t); }

  std::vector<int64_t> padded(const TensorValue &t, const std::string &what) const {
    std::vector<int64_t> s = t.shape;
    while (s.size() > full_.size() && s.front() == 1) s.erase(s.begin());
    if (s.size() > full_.size()) throw LoweringError(what + ": rank exceeds the reduced tensor's");
    s.insert(s.begin(), full_.size() - s.size(), 1);
    return s;
  }

  Span classify(const TensorValue &t, const std::string &what) const {
    if (t.numel() == 1) return Span::Scalar;
    std::vector<int64_t> keptShape = full_, dropped;
    for (size_t d = 0; d < full_.size(); ++d) {
      if (reduced_[d]) keptShape[d] = 1;
      else if (full_[d] > 1) dropped.push_back(full_[d]);
    }
    const std::vector<int64_t> s = padded(t, what);
    if (s == full_) return Span::Full;
    if (s == keptShape) return Span::Kept;
    std::vector<int64_t> real;
    for (int64_t n : t.shape) {
      if (n != 1) real.push_back(n);
    }
    if (real == dropped) return Span::Dropped;
    throw LoweringError(what + ": neither of the reduced tensor's shape nor one value per channel");
  }

  void analyse() {
    const OpNode *first = nullptr;
    for (const OpNode &op : g_.ops) {
      if (lowering::isReduceKind(op.kind)) {
        first = &op;
        break;
      }
    }
    if (first == nullptr) throw LoweringError("plane kernel: no reduction");
    full_ = g_.tensor(first->inputs[0]).shape;
    const auto reducedDims = [&](const OpNode &op) {
      std::vector<bool> r(full_.size(), false);
      for (int64_t a : op.axes) {
        if (a >= 0 && static_cast<size_t>(a) < full_.size() && full_[static_cast<size_t>(a)] > 1) r[static_cast<size_t>(a)] = true;
      }
      return r;
    };
    reduced_ = reducedDims(*first);
    int part = 0;   // 0: reduced dims in front, 1: the kept ones, 2: reduced dims behind
    for (size_t d = 0; d < full_.size(); ++d) {
      if (full_[d] == 1) continue;
      if (reduced_[d] && part == 1) part = 2;
      if (!reduced_[d] && part == 0) part = 1;
      if (!reduced_[d] && part == 2) throw LoweringError("plane kernel: kept axes on both sides of a reduced one");
      (part == 0 ? outer_ : part == 1 ? kept_ : inner_) *= full_[d];
    }
    if (outer_ < 2 || kept_ < 2 || inner_ < 2) throw LoweringError("plane kernel: not reduced on both sides of the kept axes");
    const size_t nt = g_.tensors.size();
    span_.assign(nt, Span::Scalar);
    level_.assign(nt, 0);
    for (size_t t = 0; t < nt; ++t) {
      const TensorValue &tv = g_.tensors[t];
      if (tv.isConst || (tv.inputIndex >= 0 && !tv.used)) continue;
      span_[t] = classify(tv, "tensor " + tv.name);
      if (tv.numel() * static_cast<int64_t>(dtypeSize(tv.dtype)) >= (1LL << 31)) throw LoweringError("plane kernel: tensor " + tv.name + " is 2 GiB or more");
    }
    for (const OpNode &op : g_.ops) {
      if (op.outputs.size() != 1) throw LoweringError("op " + op.name + ": multiple results are not supported");
      const int out = op.outputs[0];
      const Span so = span_[static_cast<size_t>(out)];
      int lv = 0;
      for (int in : op.inputs) lv = std::max(lv, level_[static_cast<size_t>(in)]);
      if (lowering::isReduceKind(op.kind)) {
        const TensorValue &in = g_.tensor(op.inputs[0]);
        if (in.shape != full_ || reducedDims(op) != reduced_) throw LoweringError("plane kernel: all reductions must run over the same axes of the same shape");
        if (so != Span::Kept && so != Span::Dropped) throw LoweringError("op " + op.name + ": result shape does not match");
        const DType od = g_.tensor(out).dtype;
        if (std::string(computeTypeName(in.dtype)) != computeTypeName(od)) throw LoweringError("op " + op.name + ": operand and result element types differ");
        const lowering::ReduceSpec spec = lowering::reduceSpec(op, od);
        if (spec.ordered || spec.roundEachStep) throw LoweringError("op " + op.name + ": steps that round or wrap to a narrow type keep their order");
        lv += 1;
      } else {
        if (!lowering::isElementwiseKind(op.kind) || op.kind == OpKind::Assign || op.kind == OpKind::Iota) {
          throw LoweringError("op " + op.name + ": not an elementwise op or a reduction");
        }
        for (int in : op.inputs) {
          if (g_.tensor(in).isConst) continue;
          const Span si = span_[static_cast<size_t>(in)];
          // a value per channel whose reduced axes were dropped would broadcast along the last axis: only a Reshape moves it
          const bool fits = si == Span::Scalar || si == so || (so == Span::Full && si == Span::Kept) ||
                            (op.kind == OpKind::Reshape && si != Span::Full && so != Span::Full);
          if (!fits) throw LoweringError("op " + op.name + ": operand does not broadcast along the channels");
        }
        if (op.kind == OpKind::Reshape && so != Span::Scalar && g_.tensor(op.inputs[0]).numel() == 1) {
          throw LoweringError("op Reshape: more than adding or dropping unit dimensions");
        }
      }
      level_[static_cast<size_t>(out)] = lv;
      lastWalk_ = std::max(lastWalk_, lv);
    }
    for (size_t i = 0; i < g_.outputs.size(); ++i) {
      const TensorValue &t = g_.tensor(g_.outputs[i]);
      const Span s = span_[static_cast<size_t>(g_.outputs[i])];
      if (t.producer < 0) throw LoweringError("output " + t.name + " is a kernel input");
      if (s == Span::Scalar) throw LoweringError("output " + t.name + ": a single value");
      fullOutputs_ = fullOutputs_ || s == Span::Full;
      for (size_t j = 0; j < i; ++j) {
        if (g_.outputs[j] == g_.outputs[i]) throw LoweringError("output " + t.name + " is listed twice");
      }
    }
    relaxed_ = lowering::relaxedPrecisionTensors(g_);
  }

  void pickSchedule() {
    if (opt_.extentAsArgument) throw LoweringError("plane kernel: no open extents");
    int widest = 1, fullBytes = 0, fullInputs = 0;
    for (size_t t = 0; t < g_.tensors.size(); ++t) {
      const TensorValue &tv = g_.tensors[t];
      if (tv.isConst || span_[t] != Span::Full || (tv.inputIndex < 0 && tv.outputIndex < 0)) continue;
      if (tv.inputIndex >= 0 && !tv.used) continue;
      widest = std::max(widest, static_cast<int>(dtypeSize(tv.dtype)));
      if (tv.inputIndex >= 0) {
        fullBytes += static_cast<int>(dtypeSize(tv.dtype));
        ++fullInputs;
      }
    }
    if (fullBytes == 0) throw LoweringError("plane kernel: no full-sized input");
    vec_ = 16 / widest;
    while (vec_ > 1 && vec_ > inner_) vec_ /= 2;
    slots_ = (inner_ + vec_ - 1) / vec_;
    overlap_ = static_cast<int>(slots_ * vec_ - inner_);
    const int64_t perChannel = outer_ * slots_;
    // Fewer than 16 channels leave more than fifteen of sixteen CUs idle in the first form, and channels of less than half a
    // wavefront of chunks most lanes: both keep one streaming kernel per level.
    if (kept_ < 16) throw LoweringError("plane kernel: fewer than 16 channels");
    if (perChannel < 32) throw LoweringError("plane kernel: channels of less than 32 chunks");
    const int regsPerChunk = std::max(1, fullBytes * vec_ / 4);
    const auto chunksFor = [&](int64_t work, int block) { return (work + block - 1) / block; };
    // One workgroup per channel: the smallest with at most eight chunks a thread, 1024 threads beyond. What bounds it is one
    // trip to memory and back with every load in flight, two workgroup-wide reductions and the store. Training batch
    // norm, us, one kernel per level and value -> this form (bytes of x and y at the rate of the largest streaming kernels):
    // bf16 [64,128,28,28] 18.5 -> 7.5 (4.0), [8,936,23,23] 20.1 -> 5.4 (2.5), [27,136,27,27] 16.3 -> 5.1 (1.7),
    // [64,1024,7,7] 17.1 -> 4.8 (2.0), f16 [128,512,14,14] 27.2 -> 11.1 (8.0; 1024 threads 11.9, 256 with 13 chunks 11.3).
    int block = 128;
    while (block < 1024 && chunksFor(perChannel, block) > 8) block *= 2;
    if (opt_.block >= 64 && opt_.block <= 1024 && (opt_.block & (opt_.block - 1)) == 0) block = opt_.block;
    const int64_t resident = chunksFor(perChannel, block);
    // Extrema of chunks of eight and sixteen: with a condition per element the compiler unpacks all chunks in front of it and spills
    // (range of f16 [125,700,28,28] 83.9 us, 62.2 with a branch per chunk; int8 53.6 -> 44.8). Not 8-bit chunks that share elements (int8
    // [2048,700,7,7] 48.3, 50.6 by branches) nor chunks of four (i32 [10,700,28,28]
    // 9.0, 10.1).
    for (const OpNode &op : g_.ops) {
      if (lowering::isReduceKind(op.kind) && isExtremum(lowering::reduceSpec(op, g_.tensor(op.outputs[0]).dtype))) chunkBranch_ = true;
    }
    chunkBranch_ = chunkBranch_ && vec_ >= 8 && (overlap_ == 0 || widest == 2);
    // The line between the forms. 64 registers of a 1024-thread workgroup hold 256 KiB as they came from memory. (Offsets and
    // flags are a few more per chunk: where narrow types or short runs make 24 and more small chunks a thread some of them
    // spill; with 256 channels and more that is still the faster form: range of int8 [32000,700,6] 352 us, 491 by level, 390 by one kernel
    // per level and value as before. It is the slower one for f32 results of int8 runs of six: [12288,700,6] 174, by such kernels 161.)
    // Few channels leave CUs idle in the resident form, and many elements a thread make that the longer way. us, resident / by level,
    // batch norms: 16 bits, [201,16,21,21] (88 elements a thread) 13.1 / 7.4, [931,24,9,9] 14.3 / 7.9, [73,21,32,36] 9.0 / 7.2, [38,28,19,105] 11.9 / 7.8, 27 of 29
    // with 9 .. 11 chunks a thread slower resident, by a quarter in the mean; 48 channels of 96 9.9 / 10.0, of 128 12.3 / 11.5, 38 of ragged runs [105,38,35,35]
    // 19.0 / 10.1; 64 channels of 128 12.6 / 12.8; f32, 9 .. 15 chunks, 13 norms a fifth faster resident, [61,31,33,17] 5.1 / 7.3, [57,29,23,47] 7.4 / 8.2.
    // With one level of reductions, resident / by level / one kernel per level and value: int8 range of [64,32,64,64] 17.2 / 7.0 / 11.5,
    // [30000,32,2,3] 91.7 / 24 / 25.4. Short runs, which share their lines, earlier: i32 range of [3072,16,6] 11.9 / 5.2 / 9.1,
    // with 128 channels and one level range of f16 [12288,128,6] 62 / 33 / 46, of i32 [6144,128,6] 33.5 / 20.6 / 30.5 (batch norms, of two
    // levels, stay: bf16 [16384,128,6] 54.6 / 61).
    const int64_t runBytes = inner_ * widest;
    const bool fewChannels = runBytes < 64 ? (kept_ <= 32 && perChannel > 4096) || (kept_ < 256 && resident > 8 && lastWalk_ == 1)
                             : kept_ <= 32 ? resident > 8 && (lastWalk_ == 1 || fullBytes < 4 * fullInputs || resident * vec_ >= 96)
                                           : kept_ <= 48 && lastWalk_ > 1 && resident * vec_ >= 120;
    if (resident * regsPerChunk <= 64 && opt_.split <= 1 && (!fewChannels || opt_.split == 1)) {
      block_ = block;
      chunks_ = static_cast<int>(resident);
      parts_ = 0;
      // Half of the registers may hold the elements as they are computed with: the walks behind the first then neither unpack them nor
      // compute what the walk before did (a batch norm's instructions are 4 of the 8 us of bf16 [64,128,28,28]: 809 -> 641, 8.0 -> 7.5 us).
      // A single input of 32-bit elements has nothing to unpack, and kept it is only longer alive (range of f32 [79,803,8,8] 4.4 -> 5.0). And with more
      // channels than CUs two workgroups of 1024 threads share one only with half of the registers: bf16 [19,766,51,51] 29.1 -> 32.0, f16 [24,989,44,44]
      // 31.0 -> 33.1.
      keepsUnpacked_ = resident * vec_ * fullInputs <= 65536 / block_ && !(fullInputs == 1 && fullBytes >= 4) && (block_ < 1024 || kept_ <= opt_.computeUnits);
      return;
    }
    // One launch per level: 128 bytes of loads in flight per thread, less where that leaves less than four workgroups per
    // CU. Bound by the passes over the tensor, one per level and one to store (a later pass is served by the last-level
    // cache in part): f32 [112,32,79,79] 90.5 -> 64.4 us (56 for the 3 + 1 passes), f16 [24,112,80,80] 33.3 -> 20.0, bf16
    // [100,16,100,100] 33.8 -> 19.0, [128,64,56,56] 42.4 -> 32.5; 512 threads or half the chunks are within 5 % of it. Short runs of few
    // channels: one workgroup per CU, as neighbours in a channel ask for the same lines (int8 [30000,32,2,3] 33 us with four, 24).
    block_ = opt_.block >= 64 && opt_.block <= 1024 && (opt_.block & (opt_.block - 1)) == 0 ? opt_.block : 256;
    int chunks = std::max(1, 32 / regsPerChunk);
    if (opt_.chunks > 0) chunks = opt_.chunks;
    while (opt_.chunks == 0 && chunks > 1 && kept_ * chunksFor(perChannel, block_ * chunks) < (runBytes < 64 && kept_ <= 32 ? 1 : 4) * opt_.computeUnits) chunks /= 2;
    if (opt_.split > 1) chunks = static_cast<int>(chunksFor(perChannel, static_cast<int>(std::min<int64_t>(opt_.split, 1 << 16)) * block_));
    if (chunks * regsPerChunk > 128) throw LoweringError("plane kernel: too many chunks per thread");
    chunks_ = chunks;
    parts_ = chunksFor(perChannel, block_ * chunks_);
    if (kept_ * parts_ >= (1LL << 31)) throw LoweringError("plane kernel: too many workgroups");
    partialAt_.assign(g_.tensors.size(), 0);
    for (const OpNode &op : g_.ops) {
      if (!lowering::isReduceKind(op.kind)) continue;
      partialAt_[static_cast<size_t>(op.outputs[0])] = workspaceBytes_;
      workspaceBytes_ += (static_cast<uint64_t>(kept_ * parts_) * 8 + 255) / 256 * 256;
    }
  }

  std::string operandExpr(int t) const {
    const TensorValue &tv = g_.tensor(t);
    if (tv.isConst) return lowering::literalFor(tv.dtype, tv.constValue);
    const Val &v = vals_[static_cast<size_t>(t)];
    if (!v.defined) throw LoweringError("tensor " + tv.name + " is used before it is computed");
    return v.full ? v.ident + "[e]" : v.ident;
  }

  bool ready(const OpNode &op) const {
    for (int in : op.inputs) {
      if (!g_.tensor(in).isConst && !vals_[static_cast<size_t>(in)].defined) return false;
    }
    return true;
  }

  // Elementwise ops on full-sized (or per-channel) values up to level `upto`, in description order.
  void emitOps(bool full, int upto, const std::string &ind) {
    for (const OpNode &op : g_.ops) {
      if (lowering::isReduceKind(op.kind)) continue;
      const int out = op.outputs[0];
      Val &v = vals_[static_cast<size_t>(out)];
      if (level_[static_cast<size_t>(out)] > upto || v.defined || !ready(op)) continue;
      bool anyFull = false;
      for (int in : op.inputs) anyFull = anyFull || (!g_.tensor(in).isConst && vals_[static_cast<size_t>(in)].full);
      if (anyFull != full) continue;
      if (op.kind == OpKind::Reshape || op.kind == OpKind::BroadcastTo) {
        if (g_.tensor(op.inputs[0]).isConst) throw LoweringError("op " + op.name + ": constant operand");
        v = vals_[static_cast<size_t>(op.inputs[0])];
        continue;
      }
      std::vector<std::string> operands;
      for (int in : op.inputs) operands.push_back(operandExpr(in));
      // (values per channel cost nothing, so they are never the approximate ones)
      const std::string expr = lowering::elementwiseExpr(g_, op, operands, full && relaxed_[static_cast<size_t>(out)]);
      const std::string ct = computeTypeName(g_.tensor(out).dtype);
      v.defined = true;
      v.full = full;
      v.ident = id(full ? "t" : "s", out);
      if (full) {
        src_ << ind << ct << " " << v.ident << "[V];  // " << op.name << " -> " << g_.tensor(out).name << "\n";
        src_ << ind << "#pragma unroll\n";
        src_ << ind << "for (int e = 0; e < V; ++e) " << v.ident << "[e] = " << expr << ";\n";
      } else {
        src_ << ind << "const " << ct << " " << v.ident << " = " << expr << ";  // " << op.name << " -> " << g_.tensor(out).name << "\n";
      }
    }
  }

  std::string scratchExpr(const std::string &ct) {
    if (block_ <= 64) return "static_cast<" + ct + " *>(nullptr)";
    return "reinterpret_cast<" + ct + " *>(akg_scratch[" + std::to_string(reduceCount_++ & 1) + "])";
  }

  // One kernel that runs the walks `from` .. `upto`: all of them (one workgroup per channel) or one.
  void emitKernel(const std::string &name, int from, int upto) {
    vals_.assign(g_.tensors.size(), Val());
    reduceCount_ = 0;
    const bool last = upto == lastWalk_;
    const bool walksData = from < lastWalk_ || fullOutputs_;   // the last launch of the second form may have values per channel only
    const int64_t parts = parts_ == 0 || (last && !fullOutputs_) ? 1 : parts_;
    src_ << "extern \"C\" __global__ __launch_bounds__(" << block_ << ") void " << name << "(";
    for (size_t i = 0; i < g_.inputs.size(); ++i) {
      src_ << (i ? ", " : "") << "const " << dtypeTag(g_.tensor(g_.inputs[i]).dtype) << "::storage *__restrict__ in" << i;
    }
    for (size_t i = 0; i < g_.outputs.size(); ++i) {
      src_ << ", " << dtypeTag(g_.tensor(g_.outputs[i]).dtype) << "::storage *__restrict__ out" << i;
    }
    if (parts_ != 0) src_ << ", unsigned char *__restrict__ akg_ws";
    src_ << ") {\n";
    src_ << "  constexpr int V = " << vec_ << ", BLOCK = " << block_ << ", CH = " << chunks_ << ";\n";
    src_ << "  constexpr unsigned K = " << kept_ << "u, RI = " << inner_ << "u, SLOTS = " << slots_ << "u, TOTAL = " << outer_ * slots_
         << "u, PARTS = " << parts << "u;\n";
    line("  const int tid = static_cast<int>(threadIdx.x);");
    // neighbouring channels share the cache lines in which a run ends and the next one begins: one XCD, one L2
    line("  const unsigned akg_wg = static_cast<unsigned>(akg::xcd_contiguous_id(static_cast<int>(blockIdx.x), static_cast<int>(K * PARTS)));");
    line("  const unsigned akg_k = akg_wg / PARTS;");
    if (block_ > 64) line("  __shared__ double akg_scratch[2][BLOCK / 64];");
    for (size_t i = 0; i < g_.inputs.size(); ++i) {
      const TensorValue &t = g_.tensor(g_.inputs[i]);
      if (t.used) src_ << "  const akg::Buffer b_in" << i << " = akg::make_buffer(in" << i << ", " << t.numel() * static_cast<int64_t>(dtypeSize(t.dtype)) << "L);\n";
    }
    if (last) {
      for (size_t i = 0; i < g_.outputs.size(); ++i) {
        const TensorValue &t = g_.tensor(g_.outputs[i]);
        src_ << "  const akg::Buffer b_out" << i << " = akg::make_buffer(out" << i << ", " << t.numel() * static_cast<int64_t>(dtypeSize(t.dtype)) << "L);\n";
      }
    }
    if (walksData) {
      src_ << "  unsigned akg_at[CH];   // first element of the chunk\n";
      src_ << "  bool akg_ok[CH];\n";
      if (overlap_) src_ << "  int akg_skip[CH];      // elements the chunk shares with the one before it\n";
      line("#pragma unroll");
      line("  for (int j = 0; j < CH; ++j) {");
      line("    const unsigned slot = ((akg_wg % PARTS) * CH + j) * BLOCK + tid;");
      line("    const unsigned run = slot / SLOTS, in_run = slot % SLOTS;");
      line("    akg_ok[j] = slot < TOTAL;");
      if (overlap_) {
        line("    const bool tail = in_run == SLOTS - 1;");
        src_ << "    akg_skip[j] = !akg_ok[j] ? V : tail ? " << overlap_ << " : 0;\n";
        line("    akg_at[j] = (run * K + akg_k) * RI + (tail ? RI - V : in_run * V);");
      } else {
        line("    akg_at[j] = (run * K + akg_k) * RI + in_run * V;");
      }
      line("  }");
    }
    // streamed past the caches where this kernel is the last to read them and the runs are whole 64-byte pieces
    for (size_t i = 0; i < g_.inputs.size(); ++i) {
      const int t = g_.inputs[i];
      const TensorValue &tv = g_.tensor(t);
      if (!tv.used) continue;
      const std::string tag = dtypeTag(tv.dtype);
      Val &v = vals_[static_cast<size_t>(t)];
      if (span_[static_cast<size_t>(t)] == Span::Full) {
        if (!walksData) continue;
        const bool stream = last && opt_.nonTemporal != 0 && (inner_ * static_cast<int64_t>(dtypeSize(tv.dtype))) % 64 == 0;
        src_ << "  akg::RawChunk<" << tag << ", V> p_in" << i << "[CH];  // " << tv.name << "\n";
        line("#pragma unroll");
        src_ << "  for (int j = 0; j < CH; ++j) akg::load_raw_chunk_if<" << tag << ", V, " << (stream ? "true" : "false") << ">(b_in" << i
             << ", akg_ok[j], akg_at[j], p_in" << i << "[j]);\n";
      } else {
        v.defined = true;
        v.ident = id("s_in", static_cast<int>(i));
        src_ << "  const " << computeTypeName(tv.dtype) << " " << v.ident << " = akg::load_one<" << tag << ">(b_in" << i << ", "
             << (span_[static_cast<size_t>(t)] == Span::Scalar ? "0" : "akg_k") << ");  // " << tv.name << "\n";
      }
    }
    // the levels in front of this kernel's: the partial results of the channel, folded in the same order by every workgroup
    for (const OpNode &op : g_.ops) {
      const int out = op.outputs[0];
      if (!lowering::isReduceKind(op.kind) || level_[static_cast<size_t>(out)] > from) continue;
      const DType od = g_.tensor(out).dtype;
      const lowering::ReduceSpec spec = lowering::reduceSpec(op, od);
      const std::string ct = computeTypeName(od), acc = id("acc", out);
      src_ << "  " << ct << " " << acc << " = " << spec.init << ";  // " << op.name << " -> " << g_.tensor(out).name << "\n";
      src_ << "  for (unsigned p = tid; p < " << parts_ << "u; p += BLOCK) " << acc << " = " << spec.combiner << "::apply(" << acc
           << ", reinterpret_cast<const " << ct << " *>(akg_ws + " << partialAt_[static_cast<size_t>(out)] << "L)[akg_k * " << parts_ << "u + p]);\n";
      src_ << "  " << acc << " = akg::group_reduce<" << spec.combiner << ", BLOCK, true>(" << acc << ", " << scratchExpr(ct) << ", tid);\n";
      Val &v = vals_[static_cast<size_t>(out)];
      v.defined = true;
      v.ident = acc;
    }
    for (int walk = from; walk <= upto; ++walk) emitWalk(walk, walk > from);
    if (last) {
      src_ << "  if (tid == 0" << (parts > 1 ? " && akg_wg % PARTS == 0" : "") << ") {\n";
      for (size_t i = 0; i < g_.outputs.size(); ++i) {
        const int t = g_.outputs[i];
        if (span_[static_cast<size_t>(t)] == Span::Full) continue;
        src_ << "    akg::store_one<" << dtypeTag(g_.tensor(t).dtype) << ">(b_out" << i << ", akg_k, " << operandExpr(t) << ");\n";
      }
      line("  }");
    }
    line("}\n");
  }

  void emitWalk(int walk, bool again) {
    std::vector<const OpNode *> reduces;
    for (const OpNode &op : g_.ops) {
      if (lowering::isReduceKind(op.kind) && level_[static_cast<size_t>(op.outputs[0])] == walk + 1) reduces.push_back(&op);
    }
    src_ << "  // ---- walk " << walk << " ----\n";
    emitOps(false, walk, "  ");
    const bool stores = walk == lastWalk_ && fullOutputs_;
    if (reduces.empty() && !stores) return;
    for (const OpNode *op : reduces) {
      const DType od = g_.tensor(op->outputs[0]).dtype;
      src_ << "  " << computeTypeName(od) << " acc" << op->outputs[0] << " = " << lowering::reduceSpec(*op, od).init << ";  // " << op->name << " -> "
           << g_.tensor(op->outputs[0]).name << "\n";
    }
    line("#pragma unroll");
    line("  for (int j = 0; j < CH; ++j) {");
    if (chunkBranch_) line("    if (!akg_ok[j]) continue;");
    for (size_t i = 0; i < g_.inputs.size(); ++i) {
      const int t = g_.inputs[i];
      const TensorValue &tv = g_.tensor(t);
      if (!tv.used || span_[static_cast<size_t>(t)] != Span::Full) continue;
      Val &v = vals_[static_cast<size_t>(t)];
      v.defined = v.full = true;
      v.ident = id("x", static_cast<int>(i));
      if (again && !keepsUnpacked_) src_ << "    akg::forget_unpacked(p_in" << i << "[j]);\n";
      src_ << "    " << computeTypeName(tv.dtype) << " " << v.ident << "[V];\n";
      src_ << "    akg::unpack_chunk(p_in" << i << "[j], " << v.ident << ");\n";
    }
    emitOps(true, walk, "    ");
    for (const OpNode *op : reduces) {
      const DType od = g_.tensor(op->outputs[0]).dtype;
      const lowering::ReduceSpec spec = lowering::reduceSpec(*op, od);
      const std::string acc = id("acc", op->outputs[0]);
      line("#pragma unroll");
      src_ << "    for (int e = 0; e < V; ++e) {\n";
      // (in a walk by branches an extremum takes the elements a chunk shares with its neighbour twice)
      const std::string taken = chunkBranch_ && (overlap_ == 0 || isExtremum(spec)) ? "" : overlap_ ? "if (e >= akg_skip[j]) " : "if (akg_ok[j]) ";
      src_ << "      " << taken << acc << " = " << spec.combiner << "::apply(" << acc << ", " << operandExpr(op->inputs[0]) << ");\n";
      src_ << "    }\n";
    }
    if (stores) {
      for (size_t i = 0; i < g_.outputs.size(); ++i) {
        const int t = g_.outputs[i];
        if (span_[static_cast<size_t>(t)] != Span::Full) continue;
        const std::string tag = dtypeTag(g_.tensor(t).dtype);
        const bool stream = opt_.nonTemporal != 0 && (inner_ * static_cast<int64_t>(dtypeSize(g_.tensor(t).dtype))) % 64 == 0;
        std::string src = vals_[static_cast<size_t>(t)].ident;
        if (!vals_[static_cast<size_t>(t)].full) {
          src = "akg_b" + std::to_string(i);
          src_ << "    " << computeTypeName(g_.tensor(t).dtype) << " " << src << "[V];\n";
          line("#pragma unroll");
          src_ << "    for (int e = 0; e < V; ++e) " << src << "[e] = " << operandExpr(t) << ";\n";
        }
        src_ << "    akg::store_chunk_if<" << tag << ", V, " << (stream ? "true" : "false") << ">(b_out" << i << ", akg_ok[j], akg_at[j], " << src << ");\n";
      }
    }
    line("  }");
    for (Val &v : vals_) {
      if (v.full) v = Val();   // full-sized values live inside one walk
    }
    for (const OpNode *op : reduces) {
      const int out = op->outputs[0];
      const DType od = g_.tensor(out).dtype;
      const lowering::ReduceSpec spec = lowering::reduceSpec(*op, od);
      const std::string ct = computeTypeName(od), acc = id("acc", out);
      src_ << "  " << acc << " = akg::group_reduce<" << spec.combiner << ", BLOCK, true>(" << acc << ", " << scratchExpr(ct) << ", tid);\n";
      if (parts_ != 0) {
        src_ << "  if (tid == 0) reinterpret_cast<" << ct << " *>(akg_ws + " << partialAt_[static_cast<size_t>(out)] << "L)[akg_wg] = " << acc << ";\n";
      }
      Val &v = vals_[static_cast<size_t>(out)];
      v.defined = true;
      v.ident = acc;
    }
  }
};

}  // namespace

LoweredKernel lowerPlaneToHip(const OpGraph &graph, const LoweringOptions &options) {
  PlaneEmitter emitter(graph, options);
  return emitter.run();
}

}  // namespace akg
