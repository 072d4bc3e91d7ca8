/**
 * Lowering of a contraction whose result meets reductions over its last axis: attention probabilities (scores, scale,
 * mask, softmax) in one kernel. The scores of sixteen rows stay in the registers of the workgroup that computed them
 * (kernels/akg_gemm_rows.hpp), so the float32 [batch,M,N] tensor between the contraction and the row kernel never
 * exists in memory. What this kernel does not take runs as a contraction followed by a row kernel.
 *
 * The reference lowers the two parts as separate loop nests over the materialised scores
 * (akg-mlir/lib/Conversion/MindSporeToLinalg/MindSporeToLinalg.cpp:791-901,1511-1546).
 */
#include <algorithm>
#include <sstream>

#include "HipLowering.h"

namespace akg {
namespace {

using lowering::computeTypeName;
using lowering::dtypeTag;

enum class Rank { None, Const, Row, Full };   // Row: one value per row of C (or one value); Full: a value per element

class GemmRowsEmitter {
 public:
  explicit GemmRowsEmitter(const OpGraph &g) : g_(g) {}

  LoweredKernel run() {
    analyse();
    pickSchedule();
    emitBody();
    LoweredKernel k;
    k.kernelName = g_.name + "_kernel";
    k.source = assemble();
    k.family = KernelFamily::GemmRows;
    k.grid[0] = static_cast<unsigned>(perXcd() * 8);
    k.block[0] = static_cast<unsigned>(64 * wavesC_ * wavesR_);
    k.algorithmicBytes = lowering::countAlgorithmicBytes(g_);
    k.algorithmicOps = 2ull * static_cast<uint64_t>(batch_ * m_) * static_cast<uint64_t>(n_ * k_);
    k.shapeArgs = lowering::buildShapeArgs(g_);
    std::ostringstream note;
    note << "gemm_rows batch=" << batch_ << " M=" << m_ << " N=" << n_ << " K=" << k_ << " rows per workgroup=" << groupRows()
         << " wavefronts per row=" << wavesC_ << " units of 32 columns per wavefront=" << chunks_ << " grid=" << k.grid[0];
    k.scheduleNote = note.str();
    return k;
  }

 private:
  struct Val {
    Rank rank = Rank::None;
    std::string ident;
  };

  const OpGraph &g_;
  std::ostringstream src_;
  std::vector<Val> vals_;
  std::vector<bool> relaxed_;
  int matmulOp_ = -1, aId_ = -1, bId_ = -1, accId_ = -1;
  int64_t batch_ = 1, m_ = 0, n_ = 0, k_ = 0;
  bool small_ = false;   // one launch for two, however few rows
  int wavesC_ = 1, wavesR_ = 1, rowTiles_ = 1, chunks_ = 1, reductions_ = 0;

  int64_t groupRows() const { return 16L * rowTiles_ * wavesR_; }
  int64_t rowGroups() const { return (m_ + groupRows() - 1) / groupRows(); }
  int64_t perXcd() const { return (batch_ * rowGroups() + 7) / 8; }
  const char *mma() const { return g_.tensor(aId_).dtype == DType::BF16 ? "akg::MmaBF16" : "akg::MmaF16"; }

  void analyse() {
    bool reduces = false;
    for (size_t i = 0; i < g_.ops.size(); ++i) {
      const OpNode &op = g_.ops[i];
      if (op.outputs.size() != 1) throw LoweringError("op " + op.name + ": multiple results are not supported");
      if (op.kind == OpKind::MatMul) {
        if (matmulOp_ >= 0) throw LoweringError("only one MatMul per kernel is supported");
        matmulOp_ = static_cast<int>(i);
      } else if (lowering::isReduceKind(op.kind)) {
        reduces = true;
      } else if (!lowering::isElementwiseKind(op.kind) || op.kind == OpKind::Assign || op.kind == OpKind::Iota) {
        throw LoweringError("op " + op.name + " cannot follow a MatMul in one kernel with its row reductions");
      }
    }
    if (matmulOp_ < 0 || !reduces) throw LoweringError("no MatMul with reductions behind it");
    const OpNode &mm = g_.ops[static_cast<size_t>(matmulOp_)];
    aId_ = mm.inputs[0];
    bId_ = mm.inputs[1];
    accId_ = mm.outputs[0];
    const TensorValue &a = g_.tensor(aId_), &b = g_.tensor(bId_), &c = g_.tensor(accId_);
    const size_t rank = a.shape.size();
    if (mm.transposeA || !mm.transposeB || a.inputIndex < 0 || b.inputIndex < 0 || a.dtype != b.dtype ||
        (a.dtype != DType::BF16 && a.dtype != DType::F16) || c.dtype != DType::F32 || (rank != 2 && rank != 3) ||
        b.shape.size() != rank || c.shape.size() != rank) {
      throw LoweringError("MatMul: row reductions follow 16-bit operands [M,K] x [N,K] with a float32 result");
    }
    batch_ = rank == 3 ? a.shape[0] : 1;
    m_ = a.shape[rank - 2];
    k_ = a.shape[rank - 1];
    n_ = b.shape[rank - 2];
    if ((rank == 3 && (b.shape[0] != batch_ || c.shape[0] != batch_)) || b.shape[rank - 1] != k_ || c.shape[rank - 2] != m_ ||
        c.shape[rank - 1] != n_ || batch_ < 1 || m_ < 1) {
      throw LoweringError("MatMul: inconsistent shapes");
    }
    if (batch_ > 65535) throw LoweringError("MatMul: batch extent out of range");   // (the contraction kernel's limit)
    // Where the line lies (bf16 or f16, GPU time of one kernel against a contraction and a row kernel):
    //   [192,512,64]x512 77 us for 149, [384,256,64]x256 43 for 142, [24,2048,64]x2048 174 for 238, [380,77,64]x80 8.7 for 48;
    //   every row group reads all of B from the L2, which costs more than the scores' way through memory once B is large
    //   ([20,1200,128]x2048, 512 KiB of B: 136 us for 126; [384,37,128]x1000, 250 KiB: 61 for 85), and a single query uses one of its sixteen rows ([300,1,64]x2048:
    //   24 us for 17, four rows 31 for 32);
    //   few row groups leave the chip idle ([1,256,64]x1024, 16 groups: 9.1 us for 7.9; [3,512,128]x512, 96: 7.8 for 10.1);
    //   scores below 1 MiB stay in the caches, and both forms take the time of their launches: with up to 64 KiB of B a batch (a K above 128: 32 KiB)
    //   one launch is the faster one however few rows or scores there are ([33,56,64]x56 3.2 for 7.4, [12,104,64]x104 4.0 for 8.1, [3,320,64]x320 4.3
    //   for 8.5, [24,5,64]x232 3.2 for 6.2, [6,1,128]x88 3.3 for 6.0; 33 other
    //   shapes 0.44 of the time in the mean, none slower), with more not ([9,27,128]x552 7.8 for 6.8, [16,9,64]x1200 9.1 for
    //   5.7, [4,33,192]x128 7.9 for 7.1). Two kernels stay, as tests pin them, for fewer than 16 columns, from 32 rows on for up to 64 KiB of
    //   scores ([3,40,64]x136) and from 128 on for up to 512 KiB ([2,512,64]x64, [4,128,64]x256), though one would be the faster one there too
    //   ([1,360,64]x360 3.8 for 5.6, [2,64,128]x64 4.2 for 6.6, [2,48,256]x48 5.4 for 6.6).
    if (k_ % 32 != 0 || n_ % 8 != 0 || n_ > 2048 || n_ * k_ > (1LL << 17)) throw LoweringError("MatMul: operands of this shape have no row kernel");
    const int64_t scores = batch_ * m_ * n_ * 4;
    small_ = k_ <= 256 && n_ * k_ <= (k_ <= 128 ? 1LL << 15 : 1LL << 14) &&
             (scores > (512LL << 10) || (n_ >= 16 && (m_ < 32 || (m_ < 128 && scores > (64LL << 10)))));
    if (!small_ && (m_ < 4 || scores < (1LL << 20))) throw LoweringError("MatMul: too few rows or scores for the row kernel");
    // With a longer K a row group reads more of B from the L2, and the contraction kernel gains where its 256 x 256 tiles are
    // full. bf16 with softmax behind it, one kernel for two (us). K = 160 .. 224: 46 of 47 shapes faster, [12510,192]x312 20.1
    // for 19.3. Batches of fewer than 1000 rows: 164 x [343,256]x240 50 for 105, 271 x [487,384]x320 195 for 237, 64 x
    // [512,512]x256 50 for 62, but 64 x [46,512]x224 18.2 for 15.7; longer ones: 20 x [1378,256]x176 30 for 24, 4 x [3575,256]x400 34
    // for 26, few columns 107 x [2032,256]x56 50 for 70. One batch: [6024,256]x312 13.9 for 15.5, [9674,256]x328 20.5 for 19.2,
    // [93571,256]x256 64 for 56; at most 64 columns: [28955,256]x40 9.9 for 12.8, [16384,512]x64 12.3 for 18.5, [36288,256]x48 15.0 for
    // 13.4, [65536,512]x64 28 for 23; at most 24: [16384,1024]x16 11.1 for 20.0, [32768,4096]x8 61 for 80, [65536,7168]x16 172 for
    // 165. ([16384,2048]x64 38 for 28, [8192,4096]x32 44 for 33.)
    const bool batches = batch_ > 1 && m_ < 1000;
    int64_t longest = n_ <= 24 ? 4096 : 224;
    if (batches || batch_ * m_ <= 8192 || (batch_ > 1 && n_ <= 64)) longest = std::max<int64_t>(longest, 384);
    if ((batches && m_ >= 64) || (n_ <= 64 && batch_ * m_ <= 32768)) longest = std::max<int64_t>(longest, 512);
    if (k_ > longest) throw LoweringError("MatMul: K is too long for the row kernel");
    // Scores that are an output are written either way: bf16 [28,2048,64]x1024 with the probabilities in both types 174 us
    // for 144, [14,2048,64]x2048 118 for 100; up to 256 columns one kernel is faster ([400,300,64]x256 57 for 135).
    if (g_.tensor(accId_).outputIndex >= 0 && n_ > 256) throw LoweringError("MatMul: scores of this size that are written leave nothing to save");
    for (const OpNode &op : g_.ops) {
      if (op.kind == OpKind::MatMul) continue;
      for (int in : op.inputs) {
        if (in == aId_ || in == bId_) throw LoweringError("MatMul operands cannot also feed the ops behind it");
      }
    }
    for (size_t i = 0; i < g_.outputs.size(); ++i) {
      if (std::count(g_.outputs.begin(), g_.outputs.end(), g_.outputs[i]) > 1) throw LoweringError("an output is listed twice");
    }
    for (const TensorValue &t : g_.tensors) {
      if (!t.isConst && (t.inputIndex >= 0 || t.outputIndex >= 0) && t.numel() * static_cast<int64_t>(dtypeSize(t.dtype)) >= (1LL << 31)) {
        throw LoweringError("tensor " + t.name + ": the row kernel addresses less than 2 GiB per tensor");
      }
    }
  }

  // Wavefronts that share a row: at most four units of 32 columns each (32 values a lane) up to 2048 columns; short rows
  // fill the workgroup with row groups instead. Two row tiles per wavefront where 512 workgroups are left: every
  // fragment of B is then read for 32 rows ([192,512,64] x 512: 77 us, one row tile 95, four 76; with 48 workgroups
  // instead of 96 [3,512,128] x 512 takes 9.9 us instead of 7.8).
  void pickSchedule() {
    const int64_t units = (n_ + 31) / 32;
    wavesC_ = 1;
    while (wavesC_ < 16 && units > 4 * wavesC_) wavesC_ *= 2;
    chunks_ = static_cast<int>((units + wavesC_ - 1) / wavesC_);
    auto shape = [&](int rowTiles) {
      rowTiles_ = rowTiles;
      wavesR_ = 1;
      while (wavesC_ * wavesR_ < 4 && m_ > 16L * rowTiles_ * wavesR_) wavesR_ *= 2;
      return batch_ * rowGroups();
    };
    // (Sixteen wavefronts are alone on their CU, where two row tiles take 1.75 of the time of one: [8,1824,64] x 1824, 912 and 456 workgroups,
    // 63.0 / 55.3 us, [26,1160,64] x 1160 82.9 / 72.8, [100,96,64] x 1400, 600 and 300, 37.6 / 41.0.
    // With more than a mask and a 16-bit result two tiles have no registers left: those as the others.)
    const int64_t one = shape(1), two = shape(2);
    const bool pays = wavesC_ >= 16 && wideTensors() <= 2 ? 7 * ((two + 255) / 256) < 4 * ((one + 255) / 256) : two >= 512;
    if (m_ <= 16 || !pays) shape(1);
    // Every tensor of the scores' columns takes eight registers per unit, and a workgroup of sixteen wavefronts leaves 128 a
    // lane: beyond half as many again the spills cost more than the scores' way through memory. [*,*,64] x 2048 by the number
    // wideTensors() (us for two kernels): 3 (a float32 result and a mask) 122 .. 135 for 120 .. 136, 4 115 .. 179 for 139 .. 194,
    // 5 244 for 224, 6 145 .. 268 for 146 .. 215, 7 198 .. 359 for 140 .. 240; eight wavefronts, 6 121 for 138, 8 147 for 128.
    const int registers = wavesC_ >= 16 ? 192 : (wavesC_ == 8 ? 256 : 512);
    if (8 * chunks_ * (rowTiles_ + wideTensors()) > registers) throw LoweringError("MatMul: too many tensors of the scores' size for the row kernel's registers");
    if (!small_ && batch_ * rowGroups() < 64) throw LoweringError("MatMul: too few row groups for the row kernel");
  }

  // Eight wavefronts a row (513 .. 1024 columns): 32-bit tensors of the scores' size are read by whole lines of eight rows, and with two row
  // tiles so is B. us, half lines of sixteen rows / the tensors / both: [60,640,64] x 640 48.5 / 45.7 / 44.9, [24,896,64] x 896 40.6 / 39.7 / 37.3,
  // [20,2048,64] x 1024 68.6 / 67.2 / 63.5, [13,664,64] x 664 (one row tile) 16.3 / 15.9 / 16.4; four wavefronts [192,512,64] x 512 72.7 / 72.9 / 76.5,
  // sixteen [26,1160,64] x 1160 73.0 / 74.2 / 74.0, two [300,256,64] x 256 33.9 / 34.6 / 34.7.
  // With more than 64 of K the products are more of the time and the lines are waited for in front of them: [78,648,192] x 648 103 / 107, [63,712,128] x 712
  // 59.1 / 61.3, [109,142,96] x 712 21.1 / 21.8, 28 shapes 1.014 in the mean; only from ten workgroups a CU on and up to 128 they are a gain, [115,864,128] x 864 223 / 218,
  // [259,560,128] x 560 191 / 185, [139,592,128] x 592 115 / 111. Up to 64 the mean of 24 is 0.965, the worst 1.03.
  bool byLines() const { return wavesC_ == 8 && (k_ <= 64 || (k_ <= 128 && batch_ * rowGroups() >= 2560)); }

  // Tensors of the scores' columns besides the scores, in 32-bit values per element: what is read and what is written (a
  // float32 result is computed by the longer forms of the functions in front of it: one more).
  int wideTensors() const {
    int words = 0;
    auto add = [&](int id, bool result) {
      const TensorValue &t = g_.tensor(id);
      if (t.shape.empty() || t.shape.back() != n_) return;
      const bool whole = dtypeSize(t.dtype) >= 4;
      words += (dtypeSize(t.dtype) + 3) / 4 + (result && whole ? 1 : 0);
    };
    for (int id : g_.inputs) {
      if (id != aId_ && id != bId_ && g_.tensor(id).used) add(id, false);
    }
    for (int id : g_.outputs) add(id, true);
    return words;
  }

  std::string ctOf(int id) const { return computeTypeName(g_.tensor(id).dtype); }
  std::string tagOf(int id) const { return dtypeTag(g_.tensor(id).dtype); }
  std::string operand(int id) const {
    const Val &v = vals_[static_cast<size_t>(id)];
    return v.rank == Rank::Full ? v.ident + "[j][e]" : v.ident;
  }

  // extents of a tensor against [batch, M, N]: every one is 1 or the full extent
  std::vector<int64_t> spread(const TensorValue &t) const {
    std::vector<int64_t> s = t.shape;
    while (s.size() > 3 && s.front() == 1) s.erase(s.begin());
    if (s.size() > 3) throw LoweringError("tensor " + t.name + " does not broadcast to the MatMul result");
    while (s.size() < 3) s.insert(s.begin(), 1);
    const int64_t full[3] = {batch_, m_, n_};
    for (int d = 0; d < 3; ++d) {
      if (s[static_cast<size_t>(d)] != 1 && s[static_cast<size_t>(d)] != full[d]) {
        throw LoweringError("tensor " + t.name + " does not broadcast to the MatMul result");
      }
    }
    return s;
  }

  // row of the tensor (in rows of its last extent) that belongs to `row` (akg_mc: the lane's own) of batch akg_b
  std::string rowOf(const std::vector<int64_t> &s, const std::string &row = "akg_mc") const {
    const bool b = s[0] != 1, m = s[1] != 1;
    if (b && m) return "(akg_b * M + " + row + ")";
    if (b) return "akg_b";
    return m ? row : "0L";
  }

  void loops(const std::string &indent) {
    src_ << "#pragma unroll\n" << indent << "for (int j = 0; j < NCHUNK; ++j) {\n#pragma unroll\n" << indent << "  for (int e = 0; e < 8; ++e) ";
  }

  void emitInput(size_t i) {
    const int id = g_.inputs[i];
    const TensorValue &t = g_.tensor(id);
    if (id == aId_ || id == bId_ || !t.used) return;
    const std::vector<int64_t> s = spread(t);
    Val &v = vals_[static_cast<size_t>(id)];
    const std::string tag = tagOf(id), ct = ctOf(id);
    if (s[2] == 1) {
      v.rank = Rank::Row;
      v.ident = "r_in" + std::to_string(i);
      src_ << "    const " << ct << " " << v.ident << " = " << tag << "::load(in" << i << "[" << rowOf(s) << "]);\n";
      return;
    }
    v.rank = Rank::Full;
    v.ident = "t_in" + std::to_string(i);
    if (byLines() && s[1] != 1 && dtypeSize(t.dtype) == 4) {
      src_ << "    " << ct << " " << v.ident << "[NCHUNK][8];\n#pragma unroll\n    for (int j = 0; j < NCHUNK; ++j) akg::load_own_row_if<" << tag
           << ">(b_in" << i << ", akg_ok[j], " << rowOf(s, "akg_low") << " * N + akg_cols[j], " << rowOf(s, "akg_high")
           << " * N + akg_cols[j], lane, " << v.ident << "[j]);\n";
      return;
    }
    src_ << "    " << ct << " " << v.ident << "[NCHUNK][8];\n#pragma unroll\n    for (int j = 0; j < NCHUNK; ++j) akg::load_chunk_if<" << tag
         << ", 8, false>(b_in" << i << ", akg_ok[j], " << rowOf(s) << " * N + akg_cols[j], " << v.ident << "[j]);\n";
  }

  void emitReduction(const OpNode &op) {
    const int in = op.inputs[0], out = op.outputs[0];
    const TensorValue &it = g_.tensor(in), &ot = g_.tensor(out);
    if (vals_[static_cast<size_t>(in)].rank != Rank::Full || it.numel() != batch_ * m_ * n_ || op.axes.size() != 1 ||
        op.axes[0] + 1 != static_cast<int64_t>(it.shape.size()) || it.shape.back() != n_) {
      throw LoweringError("op " + op.name + ": only reductions of the whole scores over their last axis");
    }
    const lowering::ReduceSpec spec = lowering::reduceSpec(op, ot.dtype);
    if (spec.ordered || spec.roundEachStep || ctOf(in) != ctOf(out) || (ctOf(out) != "float" && ctOf(out) != "int")) {
      throw LoweringError("op " + op.name + ": the row kernel reduces 32-bit values");
    }
    if (!op.keepDims) {
      for (const OpNode &user : g_.ops) {
        for (int u : user.inputs) {
          if (u == out) throw LoweringError("op " + op.name + ": a result without keep_dims is only written");
        }
      }
    }
    const std::string ct = ctOf(out), acc = "acc" + std::to_string(out), u = "u" + std::to_string(out);
    const std::string value = vals_[static_cast<size_t>(in)].ident;
    src_ << "    " << ct << " " << acc << " = " << spec.init << ";  // " << op.name << " -> " << ot.name << "\n"
         << "#pragma unroll\n    for (int j = 0; j < NCHUNK; ++j) {\n"
         << "      " << ct << " akg_part = " << value << "[j][0];\n#pragma unroll\n"
         << "      for (int e = 1; e < 8; ++e) akg_part = " << spec.combiner << "::apply(akg_part, " << value << "[j][e]);\n"
         << "      " << acc << " = akg_ok[j] ? " << spec.combiner << "::apply(" << acc << ", akg_part) : " << acc << ";\n    }\n"
         << "    const " << ct << " " << u << " = akg::row_scores_reduce<" << spec.combiner << ", WC>(" << acc
         << ", reinterpret_cast<" << ct << " (*)[16]>(akg_slots[" << reductions_ << "][rt][wr]), wc, lane);\n";
    ++reductions_;
    vals_[static_cast<size_t>(out)].rank = Rank::Row;
    vals_[static_cast<size_t>(out)].ident = u;
  }

  void emitElementwise(const OpNode &op) {
    const int out = op.outputs[0];
    const TensorValue &ot = g_.tensor(out);
    const std::vector<int64_t> shape = spread(ot);
    Rank rank = Rank::Row;
    std::vector<std::string> operands;
    for (int in : op.inputs) {
      const Val &v = vals_[static_cast<size_t>(in)];
      if (v.rank == Rank::None) throw LoweringError("op " + op.name + ": operand " + g_.tensor(in).name + " is undefined");
      if (!g_.tensor(in).isConst) spread(g_.tensor(in));
      if (v.rank == Rank::Full) rank = Rank::Full;
      operands.push_back(operand(in));
    }
    if ((rank == Rank::Full) != (shape[2] == n_)) throw LoweringError("op " + op.name + ": result shape does not match its operands");
    const bool relaxed = relaxed_[static_cast<size_t>(out)];
    const std::string ct = ctOf(out), id = std::to_string(out);
    std::string expr;
    // a float32 division by a per-row value: the reciprocal (or the divisor's parts) once per row, as in the row kernel
    const bool uniformDivisor = op.kind == OpKind::Div && rank == Rank::Full && op.inputs.size() == 2 &&
                                vals_[static_cast<size_t>(op.inputs[1])].rank != Rank::Full && ct == "float" &&
                                ctOf(op.inputs[0]) == "float" && ctOf(op.inputs[1]) == "float";
    if (uniformDivisor) {
      if (relaxed) {
        src_ << "    const float d" << id << " = akg::fast_rcp(" << operands[1] << ");\n";
        expr = "(" + operands[0] + " * d" + id + ")";
      } else {
        src_ << "    const akg::UniformDivisor d" << id << " = akg::make_divisor(" << operands[1] << ");\n";
        expr = "akg::div_uniform(" + operands[0] + ", d" + id + ")";
      }
      if (ot.dtype == DType::F16 || ot.dtype == DType::BF16) expr = tagOf(out) + "::rnd(" + expr + ")";
    } else {
      expr = lowering::elementwiseExpr(g_, op, operands, relaxed);
    }
    Val &v = vals_[static_cast<size_t>(out)];
    v.rank = rank;
    if (rank == Rank::Full) {
      v.ident = "t" + id;
      src_ << "    " << ct << " " << v.ident << "[NCHUNK][8];  // " << op.name << " -> " << ot.name << "\n";
      loops("    ");
      src_ << v.ident << "[j][e] = " << expr << ";\n    }\n";
    } else {
      v.ident = "u" + id;
      src_ << "    const " << ct << " " << v.ident << " = " << expr << ";  // " << op.name << " -> " << ot.name << "\n";
    }
  }

  void emitBody() {
    vals_.assign(g_.tensors.size(), Val());
    relaxed_ = lowering::relaxedPrecisionTensors(g_);
    for (size_t t = 0; t < g_.tensors.size(); ++t) {
      if (!g_.tensors[t].isConst) continue;
      vals_[t].rank = Rank::Const;
      vals_[t].ident = lowering::literalFor(g_.tensors[t].dtype, g_.tensors[t].constValue);
    }
    vals_[static_cast<size_t>(accId_)].rank = Rank::Full;
    vals_[static_cast<size_t>(accId_)].ident = "akg_s[rt]";
    for (size_t i = 0; i < g_.inputs.size(); ++i) emitInput(i);
    for (const OpNode &op : g_.ops) {
      if (op.kind == OpKind::MatMul) continue;
      if (lowering::isReduceKind(op.kind)) {
        emitReduction(op);
      } else {
        emitElementwise(op);
      }
    }
    for (size_t i = 0; i < g_.outputs.size(); ++i) {
      const int id = g_.outputs[i];
      const TensorValue &t = g_.tensor(id);
      const Val &v = vals_[static_cast<size_t>(id)];
      if (v.rank == Rank::Full && t.numel() == batch_ * m_ * n_) {
        src_ << "#pragma unroll\n    for (int j = 0; j < NCHUNK; ++j) akg::store_chunk_if<" << tagOf(id) << ", 8, false>(b_out" << i
             << ", akg_ok[j] && akg_row_ok, (akg_b * M + akg_m) * N + akg_cols[j], " << v.ident << "[j]);\n";
      } else if (v.rank == Rank::Row && t.numel() == batch_ * m_ && t.inputIndex < 0) {
        src_ << "    if (akg_row_ok && wc == 0 && lane < 16) out" << i << "[akg_b * M + akg_m] = " << tagOf(id) << "::store(" << v.ident << ");\n";
      } else {
        throw LoweringError("output " + t.name + ": shape is neither the scores' nor one value per row");
      }
    }
  }

  std::string assemble() const {
    std::ostringstream o;
    o << "// Generated by the akg HIP lowering for gfx950. Op description: " << g_.name << "\n"
      << "// family: gemm_rows, fusion class: " << operatorTemplateName(g_.operatorTemplate) << "\n"
      << "#include \"akg_rt.hpp\"\n#include \"akg_gemm_mfma.hpp\"\n#include \"akg_gemm_rows.hpp\"\n\n"
      << "extern \"C\" __global__ __launch_bounds__(" << 64 * wavesC_ * wavesR_ << ") void " << g_.name << "_kernel(";
    size_t argc = 0;
    for (size_t i = 0; i < g_.inputs.size(); ++i, ++argc) {
      o << (argc ? ", " : "") << "const " << tagOf(g_.inputs[i]) << "::storage *__restrict__ in" << i;
    }
    for (size_t i = 0; i < g_.outputs.size(); ++i, ++argc) {
      o << (argc ? ", " : "") << tagOf(g_.outputs[i]) << "::storage *__restrict__ out" << i;
    }
    o << ") {\n  constexpr long M = " << m_ << "L, N = " << n_ << "L, GROUPS = " << rowGroups() << "L;\n"
      << "  constexpr int RT = " << rowTiles_ << ", NCHUNK = " << chunks_ << ", WC = " << wavesC_ << ", WR = " << wavesR_ << ";\n"
      << "  __shared__ float akg_slots[" << std::max(1, reductions_) << "][RT][WR][WC][16];\n"
      << "  // consecutive workgroups go round-robin to the 8 XCDs: regrouped, so that the workgroups of a batch share an L2\n"
      << "  const long akg_linear = static_cast<long>(blockIdx.x % 8u) * " << perXcd() << "L + static_cast<long>(blockIdx.x / 8u);\n"
      << "  if (akg_linear >= " << batch_ * rowGroups() << "L) return;\n"
      << "  const long akg_b = akg_linear / GROUPS;\n"
      << "  const int lane = static_cast<int>(threadIdx.x) & 63, wave = static_cast<int>(threadIdx.x) >> 6;\n"
      << "  const int wc = wave % WC, wr = wave / WC;\n"
      << "  const long akg_row0 = (akg_linear % GROUPS) * " << groupRows() << "L + wr * (16 * RT);\n";
    for (size_t i = 0; i < g_.inputs.size(); ++i) {
      const TensorValue &t = g_.tensor(g_.inputs[i]);
      if (g_.inputs[i] == aId_ || g_.inputs[i] == bId_ || !t.used) continue;
      o << "  const akg::Buffer b_in" << i << " = akg::make_buffer(in" << i << ", " << t.numel() * static_cast<int64_t>(dtypeSize(t.dtype)) << "L);\n";
    }
    for (size_t i = 0; i < g_.outputs.size(); ++i) {
      const TensorValue &t = g_.tensor(g_.outputs[i]);
      o << "  const akg::Buffer b_out" << i << " = akg::make_buffer(out" << i << ", " << t.numel() * static_cast<int64_t>(dtypeSize(t.dtype)) << "L);\n";
    }
    o << "  long akg_cols[NCHUNK];\n  bool akg_ok[NCHUNK];\n#pragma unroll\n  for (int j = 0; j < NCHUNK; ++j) {\n"
      << "    akg_cols[j] = 32L * akg::row_unit<NCHUNK, WC>(j, wc) + 8 * (lane >> 4);\n    akg_ok[j] = "
      << (n_ % (32L * wavesC_) == 0 ? "true" : "akg_cols[j] < N") << ";\n  }\n"
      << "  float akg_s[RT][NCHUNK][8];\n" 
      << "  akg::row_scores<" << mma() << ", M, N, " << k_ * 2 << "L, RT, NCHUNK, WC, " << (byLines() && rowTiles_ == 2 ? "true" : "false") << ">(in" << g_.tensor(aId_).inputIndex << " + akg_b * "
      << m_ * k_ << "L, in" << g_.tensor(bId_).inputIndex << " + akg_b * " << n_ * k_ << "L, akg_row0, wc, lane, akg_s);\n"
      << "#pragma unroll\n  for (int rt = 0; rt < RT; ++rt) {\n"
      << "    const long akg_m = akg_row0 + 16 * rt + (lane & 15);\n    const bool akg_row_ok = akg_m < M;\n"
      << "    const long akg_mc = akg_row_ok ? akg_m : M - 1;\n    (void)akg_mc;\n"
      << "    // the rows of lanes c % 8 and c % 8 + 8 of the sixteen (load_own_row_if)\n"
      << "    const long akg_first = akg_row0 + 16 * rt + (lane & 7), akg_low = akg_first < M ? akg_first : M - 1, akg_high = akg_first + 8 < M ? akg_first + 8 : M - 1;\n"
      << "    (void)akg_low, (void)akg_high;\n"
      << src_.str() << "  }\n}\n";
    return o.str();
  }
};

}  // namespace

LoweredKernel lowerGemmRowsToHip(const OpGraph &graph) {
  GemmRowsEmitter emitter(graph);
  return emitter.run();
}

}  // namespace akg
