/**
 * Lowering of the Matmul fusion class: one MatMul (int8 x int8 -> int32, or bfloat16 / float16 operands with a
 * float32 accumulator) followed by an elementwise epilogue over [M,N].
 *
 * The reference lowers MatMul to linalg.matmul and then through the same generic loop mapping as everything else
 * (akg-mlir/lib/Conversion/MindSporeToLinalg/MindSporeToLinalg.cpp:1453-1546; no tensor-core path is wired into
 * its GPU pipeline). Here the contraction runs on the MFMA units (kernels/akg_gemm_mfma.hpp) and the ops that follow
 * it in the description are emitted as an epilogue functor applied to the accumulators in registers, so the
 * [M,N] int32 / float32 intermediates never exist in memory.
 *
 * Float MatMul: the reference accumulates in the MatMul's declared result type, element by element in k order
 * (zero-filled accumulator of the output type, MindSporeToLinalg.cpp:1520-1540). The MFMA kernels serve a declared
 * float32 result (their float32 sum differs from the reference's only in the order of the additions). A declared
 * float16 / bfloat16 result means a product and a sum rounded to 16 bits at every k, which no matrix unit computes:
 * such descriptions, and the shapes and element types the MFMA kernels do not take, go to the serial kernel of
 * kernels/akg_gemm_serial.hpp, which keeps the reference's order and rounding exactly.
 *
 * Epilogue operands are classified by how they vary over the output tile:
 *   Full   [M,N]      4-element chunk per (row, 4 columns), loaded / computed per output chunk
 *   Col    [N]/[1,N]  4 values per lane, loaded / computed once per lane (a lane owns 4 fixed columns)
 *   Row    [M,1]      one value per output row
 *   Scalar [1]        one value
 */
#include <algorithm>
#include <cmath>
#include <sstream>

#include "HipLowering.h"

namespace akg {
namespace {

using lowering::computeTypeName;
using lowering::dtypeTag;

enum class EpiRank { Const = 0, Scalar = 1, Row = 2, Col = 3, Full = 4 };

struct EpiVal {
  bool defined = false;
  EpiRank rank = EpiRank::Const;
  std::string ident;
};

class GemmEmitter {
 public:
  GemmEmitter(const OpGraph &g, const LoweringOptions &o) : g_(g), opt_(o) {}

  LoweredKernel run() {
    analyse();
    pickSplit();
    emit();
    LoweredKernel k;
    k.kernelName = g_.name + "_kernel";
    k.source = src_.str();
    k.family = KernelFamily::GemmEpilogue;
    const int64_t tiles = ((m_ + 255) / 256) * ((n_ + 255) / 256);
    const int64_t gridTiles = ((tiles + 7) / 8) * 8;
    if (serial_) {
      k.grid[0] = static_cast<unsigned>(((m_ + 63) / 64) * ((n_ + 16 * epiWidth() - 1) / (16 * epiWidth())));
      k.block[0] = 256;
    } else if (skinny_) {
      const int64_t strips = (n_ + stripCols() - 1) / stripCols();
      k.grid[0] = static_cast<unsigned>(strips * kSplit_);
      if (kSplit_ > 1) {
        const int64_t groups = strips * batch_;
        k.workspaceBytes = static_cast<uint64_t>((groups * 4 + 255) / 256 * 256 + groups * kSplit_ * m_ * 128 * 4);
      }
      k.block[0] = static_cast<unsigned>(skinnyWaves() * 64);
    } else if (tileM_ > 0) {
      const int64_t smallTiles = ((m_ + tileM_ - 1) / tileM_) * ((n_ + tileN_ - 1) / tileN_), smallGrid = (smallTiles + 7) / 8 * 8;
      k.grid[0] = static_cast<unsigned>(smallGrid * kSplit_);
      if (kSplit_ > 1) {
        k.workspaceBytes = static_cast<uint64_t>((smallGrid * 4 + 255) / 256 * 256 + smallTiles * kSplit_ * tileM_ * tileN_ * 4);
      }
      k.block[0] = 256;
    } else {
      k.grid[0] = static_cast<unsigned>(gridTiles * kSplit_);
      if (kSplit_ > 1) {
        const int64_t partRows = std::min<int64_t>(m_, 256);
        k.workspaceBytes = static_cast<uint64_t>((gridTiles * 4 + 255) / 256 * 256 + tiles * kSplit_ * partRows * 256 * 4);
      }
      k.block[0] = 512;
    }
    if (dyn_) {
      // the row count and the number of K splits travel as kernel arguments, and the workspace pointer is part of the
      // signature whether this shape set splits K or not
      k.scalarArgs.push_back(m_);
      k.scalarArgs.push_back(kSplit_);
      k.workspaceBytes = std::max<uint64_t>(k.workspaceBytes, 256);
    }
    k.grid[1] = static_cast<unsigned>(batch_);
    k.algorithmicBytes = lowering::countAlgorithmicBytes(g_);
    k.algorithmicOps = 2ull * static_cast<uint64_t>(batch_) * static_cast<uint64_t>(m_) * static_cast<uint64_t>(n_) *
                       static_cast<uint64_t>(k_);
    k.shapeArgs = lowering::buildShapeArgs(g_);
    std::ostringstream note;
    note << "gemm_epilogue batch=" << batch_ << " M=" << m_ << " N=" << n_ << " K=" << k_ << " transpose_b=" << (transB_ ? 1 : 0);
    if (serial_) {
      note << " serial: the reference's k-ordered sum in the declared type on the vector ALUs, tile=64x" << 16 * epiWidth()
           << " grid=" << k.grid[0];
    } else if (skinny_) {
      note << " skinny: strips of " << stripCols() << " columns, B " << (narrowCols_ > 0 ? (transB_ ? "by whole lines, all of K" : "transposed in registers, all of K") : skinnyLines() ? (streamsLines() ? "by whole lines past the caches" : "by whole lines") : "straight into MFMA operands")
           << ", mfma=" << mfmaName(narrowCols_ > 0) << " waves=" << skinnyWaves() << " grid=" << k.grid[0];
    } else if (tileM_ > 0) {
      const int unitM = tileM_ % 128 == 0 ? 128 : 64, unitN = tileN_ % 128 == 0 ? 128 : 64;
      note << " tile=" << unitM << "x" << unitN << "x" << stepK() / elemBytes() << " mfma=" << mfmaName(true) << " waves=2x2 grid=" << k.grid[0];
      if (tileM_ * tileN_ > unitM * unitN) note << " (" << tileM_ / unitM << "x" << tileN_ / unitN << " tiles a workgroup)";
    } else {
      note << " tile=256x256x" << stepK() / elemBytes() << " mfma=" << mfmaName(true) << " waves=" << (tallWavefrontTiles() ? "2x4" : "4x2") << " grid=" << k.grid[0];
    }
    if (kSplit_ > 1) note << " k_splits=" << kSplit_;
    if (roundedOnce_) note << " (AKG_HIP_MATMUL_F32_ACC: float32 accumulation rounded once to the declared 16-bit type, not the reference's per-step rounding)";
    if (dyn_) note << " (rows of A and K splits are kernel arguments: one code object for " << (skinny_ ? "up to " + std::to_string(skinnyBucket()) + " rows" : "more than 64 rows") << ")";
    k.scheduleNote = note.str();
    return k;
  }

 private:
  const OpGraph &g_;
  LoweringOptions opt_;
  std::ostringstream src_;
  int64_t m_ = 0, n_ = 0, k_ = 0, batch_ = 1;
  int kSplit_ = 1;  // workgroups per tile, each with a range of K steps (see pickSplit)
  int skinnyRows() const { return 64; }   // (96 rows: no faster than the tile kernel; 128: slower)
  int skinnyWaves() const { return narrowCols_ > 0 ? narrowWaves_ : (opt_.block == 512 ? 8 : 4); }
  // Units of a narrow strip in flight: of 64 columns of a [N,K] weight one takes 48 registers a lane and more, and eight wavefronts have 256. us, four
  // (up to 18 spilled) / three / two: bf16 32 x 1856 x 10496 11.6 / 9.7 / 9.2, f16 28 x 1344 x 12008 9.7 / 8.6 / 8.6, int8 16 x 3072 x 10708 8.6 / 8.2 / 8.0,
  // 90 products of 1 .. 32 rows 0.775 / 0.735 / 0.72 of the time on strips of 128 columns.
  int skinnyUnroll() const {
    if (opt_.chunks > 0) return opt_.chunks;
    return narrowCols_ > 0 && transB_ && !(narrowCols_ == 64 && narrowWaves_ == 8) ? 4 : 2;
  }
  int stripCols() const { return narrowCols_ > 0 ? narrowCols_ : 128; }
  // A [N,K] weight with a short K is read in 32-byte pieces, four per cache line, by instructions that follow each other:
  // with the non-temporal hint the line is not kept for the next piece. (skinnyLines() reads whole lines.)
  bool skinnyNonTemporal() const { return opt_.nonTemporal != 0 && !transB_; }
  // Where columns end inside a line, a piece of 128 bytes lies in two lines, and a short K gives the wavefronts uneven shares: a
  // weight of less than 4 MiB (all batches together) is then loaded as it is. Operands as they are and whole lines,
  // three such weights in turn / not used for 640 MB of traffic (us), of 207 sizes from 0.3 to 103 MiB: bf16 2 x 544 x 1024
  // (1.1 MiB) 5.0 and 5.6 / 5.6 and 5.9, 16 x 1184 x 1024 (2.3 MiB) 5.9 and 6.2 / 6.5 and 6.6, 39 x 3120 x 512 (3 MiB) 9.7 and 10.3 / 10.4
  // and 10.8, int8 16 x 1632 x 2048 (3.2 MiB) 6.3 and 6.7 / 6.8 and 7.2; above, bf16 16 x 2080 x 1024 (4.1 MiB) 6.4 and 6.5 / 7.4 and 7.1,
  // int8 16 x 3136 x 2048 (6.1 MiB) 7.1 and 6.8 / 8.5 and 7.9, bf16 16 x 4128 x 4096 12.3 and 11.9 / 14.5 and 12.9.
  int64_t weightBytes() const { return batch_ * n_ * k_ * elemBytes(); }
  bool skinnyLines() const {
    return transB_ && k_ * elemBytes() >= 128 * skinnyWaves() && (k_ * elemBytes() % 128 == 0 || weightBytes() >= (4LL << 20));
  }
  // Whole lines of a [N,K] weight are read once, so from 96 MiB on (all batches together) they are read past the caches. Below, the
  // last-level cache (256 MiB) may hold the weight beside others: the hint then costs what it gives otherwise. With the
  // hint and without, three such weights in turn / not used for 640 MB (us): bf16 2 x 2048 x 8192 (32 MiB) 10.5 and 10.2 / 10.8 and
  // 11.9, 16 x 3648 x 8704 (61 MiB) 15.8 and 14.3 / 16.3 and 17.5, 16 x 8192 x 4096 (64 MiB) 15.7 and 14.4 / 15.9 and 17.2,
  // 16 x 8192 x 5120 (80 MiB) 18.7 and 16.9 / 18.8 and 20.1; 16 x 8192 x 8704 (136 MiB) 27.3 and 30.1 / 26.4 and 29.0, int8 16 x 16384 x
  // 8704 27.7 and 30.4 / 26.6 and 29.4. A line that does not end with the column belongs to two of them and needs its second look.
  bool streamsLines() const {
    return opt_.nonTemporal != 0 && skinnyLines() && k_ * elemBytes() % 128 == 0 && weightBytes() >= (96LL << 20);
  }
  // ... as the kernel's last argument, behind the other ones that have defaults
  std::string linesArgument(const std::string &before) const {
    if (narrowCols_ > 0) return before + ", akg::NarrowStrips<" + std::to_string(narrowCols_) + ">()";
    if (!transB_) return "";
    return streamsLines() ? before + ", akg::StreamedLines()" : (skinnyLines() ? "" : before + ", akg::NoLines()");
  }
  bool serial_ = false;  // no MFMA kernel takes the description: gemm_serial (akg_gemm_serial.hpp)
  int epiWidth() const { return (serial_ && n_ % 4 != 0) ? 1 : 4; }   // adjacent result columns per epilogue call
  int tileM_ = 0, tileN_ = 0;   // gemm_small_tile: its tile (0: another kernel)
  int narrowCols_ = 0, narrowWaves_ = 8;   // gemm_skinny_narrow: columns of a strip (0: another kernel), wavefronts
  bool skinny_ = false;  // M <= 64: the kernel that streams B, without barriers (gemm_skinny)
  // A dynamic description (extents bound per call): M and the K split are kernel arguments, so the source - and with it
  // the code object - is the same for every token count; the skinny kernel comes in three sizes (16, 32, 64 rows).
  bool dyn_ = false;
  int skinnyBucket() const { return m_ <= 16 ? 16 : (m_ <= 32 ? 32 : 64); }
  bool transB_ = false;
  bool roundedOnce_ = false;   // a 16-bit declared MatMul result on the matrix units by the caller's switch
  int matmulOp_ = -1;
  int aId_ = -1, bId_ = -1, accId_ = -1;
  std::vector<EpiVal> vals_;
  std::vector<bool> relaxed_;
  std::ostringstream members_, prepare_, apply_;
  std::vector<int> assignOnly_;   // inputs that are only written (Assign destinations the description never reads)

  DType elem_ = DType::I8;  // operand element type: I8, BF16 or F16
  int elemBytes() const { return elem_ == DType::I8 ? 1 : 2; }
  const char *mmaTraits() const {
    return elem_ == DType::I8 ? "akg::MmaI8" : (elem_ == DType::BF16 ? "akg::MmaBF16" : "akg::MmaF16");
  }
  // the skinny kernel issues 32 x 32 MFMAs (32 bytes of K), the tile kernel 16 x 16 ones (64 bytes of K)
  const char *mfmaName(bool tileKernel) const {
    if (tileKernel) return elem_ == DType::I8 ? "i32_16x16x64_i8" : (elem_ == DType::BF16 ? "f32_16x16x32_bf16" : "f32_16x16x32_f16");
    return elem_ == DType::I8 ? "i32_32x32x32_i8" : (elem_ == DType::BF16 ? "f32_32x32x16_bf16" : "f32_32x32x16_f16");
  }
  std::string accType() const { return serial_ ? computeTypeName(g_.tensor(accId_).dtype) : (elem_ == DType::I8 ? "int" : "float"); }
  int stepK() const { return 128; }   // bytes of K in one step of the tile kernel
  // 2 x 4 wavefronts of 128 x 64 instead of 4 x 2 of 64 x 128: half as many transposing reads of a row-major B (which move
  // 8 bytes a lane) for twice the 16-byte reads of A. int8 4096 x 8192 x 8192: +1.0 %, bfloat16: -0.4 %.
  // (AKG_HIP_VARIANT bit 5 takes the other one.)
  bool tallWavefrontTiles() const { return (elem_ == DType::I8 && !transB_) != ((opt_.variant & 32) != 0); }

  // What one workgroup of the small-tile kernel computes: one 64 x 64, 64 x 128 or 128 x 128 tile, or several adjacent ones that
  // share their operands in LDS (192 x 128: three of 64 x 128, 192 x 192: nine of 64 x 64, 128 x 256: two of 128 x 128). In us, per step of
  // 128 bytes of K with one workgroup on a CU, with several, and behind the loop. A CU takes in 60 .. 70 GB/s of operands
  // from L2 and memory whatever its workgroups do with them (loads alone take 42 us of the 46 of 300 x 4096 x 11008): its L1
  // answers in order, so lines that are on their way from memory hold up those behind them. Larger workgroups take in less.
  struct SmallShape {
    int m, n;
    double alone, shared, end;
    int splits;   // 1, 2, 4 .. up to this many
  };
  static const std::vector<SmallShape> &smallShapes() {
    static const std::vector<SmallShape> shapes = {{64, 64, 0.208, 0.204, 0.26, 8}, {64, 128, 0.29, 0.304, 1.2, 2}, {128, 128, 0.396, 0.44, 2.1, 2},
                                                   {192, 128, 0.528, 0.666, 4.27, 1}, {192, 192, 0.771, 0.899, 5.9, 1}, {128, 256, 0.699, 0.815, 5.24, 1}};
    return shapes;
  }
  // Fitted to 55 products (M 65 .. 4055, K 512 .. 11008, both layouts, 8 and 16 bits) on every shape, 700 times in all: standard
  // deviation 7 %; the shape it takes is 2.5 % behind the fastest in the mean (int8 4055 x 1408 x 1784 the furthest: 20.5 for 18.2). A split costs its partials' way to memory and
  // back and the time of the workgroup that adds them; rows of a [K,N] weight that begin inside lines cost one line in ten.
  double smallTileTime(const SmallShape &w, int64_t split) const {
    if (m_ <= skinnyRows()) return narrowTileTime(w.n, split);
    const int64_t steps = (k_ * elemBytes() + 127) / 128, tiles = ((m_ + w.m - 1) / w.m) * ((n_ + w.n - 1) / w.n);
    const double perCu = static_cast<double>(tiles * split) / 256, whole = std::ceil(perCu), area = static_cast<double>(w.m * w.n);
    const double rounds = perCu <= 1 ? 1 : 0.78 * whole + 0.22 * perCu;
    double step = perCu <= 1 ? w.alone : w.shared * rounds;
    if (!transB_) step *= (n_ * elemBytes() % 128 != 0 ? 1.054 : 1.007) + (elemBytes() == 1 ? 0.3 : 0);
    const double time = 2.43 + static_cast<double>((steps + split - 1) / split) * step + w.end * rounds;
    return split == 1 ? time : time + (split <= 4 ? 1.78 : 2.9) + 0.113 * static_cast<double>(split) * area / 4096 + 0.363 * static_cast<double>(tiles * split) * area * 8 / 5e6;
  }
  // At most 64 rows, where one tile's rows are the product's: an estimate of its own, which skinnyTime and smallTileRowsTime
  // below go with.
  double narrowTileTime(int64_t bn, int64_t split) const {
    const int64_t steps = (k_ * elemBytes() + 127) / 128, tiles = (n_ + bn - 1) / bn;
    const double perCu = static_cast<double>(tiles * split) / 256, area = static_cast<double>(64 * bn);
    const double step = bn == 64 ? (perCu <= 1 ? 0.35 : 0.28) : 0.48, rounds = perCu <= 1 ? 1 : (perCu + std::ceil(perCu)) / 2;
    const double loop = static_cast<double>((steps + split - 1) / split) * step * rounds;
    return split == 1 ? 3 + loop : 5.5 + loop + 0.3 * static_cast<double>(split) * area / 4096 + static_cast<double>(tiles * split) * area * 8 / 5e6;
  }
  // ... and of the 256 x 256 kernel with `split` workgroups per tile: fitted to the same products (14 %), and with more than 256 rows and
  // ragged columns to 200 such (K and N 512 .. 16384, 8 %; 8-bit ones with dequantisation and GELU behind the sums, whose eight wavefronts
  // a CU have nothing to do beside it: 16-bit ones with GELU take 5 us a tile longer than without).
  double largeTileTime(int64_t split) const {
    const int64_t steps = (k_ * elemBytes() + 127) / 128, tiles = ((m_ + 255) / 256) * ((n_ + 255) / 256), perTile = (steps + split - 1) / split;
    const double perCu = static_cast<double>(tiles * split) / 256, whole = std::ceil(perCu), rows = static_cast<double>(std::min<int64_t>(m_, 256));
    if (m_ > 256 && n_ % 256 != 0 && !outgrowsLaunch(split)) {
      const double step = 1.478 * (transB_ ? 1 : 1.068) * (elemBytes() == 1 ? (transB_ ? 0.949 : 0.967) : 1), rounds = perCu <= 1 ? 1 : 0.87 * whole + 0.13 * perCu;
      const double time = rounds * (static_cast<double>(perTile) * step + (elemBytes() == 1 ? 13.45 : functionBehind() ? 12.54 : 7.54));
      return split == 1 ? time : time + 6.45 + 1.35 * static_cast<double>(split);
    }
    const double step = 1.45 * (transB_ ? 1 : 1.093) * (elemBytes() == 1 ? 1.356 : 1);
    const double time = whole * (static_cast<double>(perTile) * step + 7.35);
    return split == 1 ? time : time + 5.67 + 2.32 * static_cast<double>(split) * rows / 256 + 0.24 * static_cast<double>(tiles * split) * rows * 2048 / 5e6;
  }
  // Partials of the 256 x 256 kernel beyond the 16 MiB of a launch without allocations: below 2^26 elements of weight such products stay with the
  // estimate that small tiles were chosen by before there was one for ragged columns, as a caller of that launch would be refused
  // (bf16 8100 x 8128 x 384 with 67 MB of them: 91.7 us, 78.5 on small tiles).
  bool outgrowsLaunch(int64_t split) const {
    const int64_t tiles = ((m_ + 255) / 256) * ((n_ + 255) / 256);
    return split > 1 && k_ * n_ < (1LL << 26) && tiles * split * std::min<int64_t>(m_, 256) * 256 * 4 + tiles * 4 > (16LL << 20);
  }
  bool functionBehind() const {
    for (const OpNode &op : g_.ops) {
      if (op.kind == OpKind::Exp || op.kind == OpKind::Tanh || op.kind == OpKind::Log || op.kind == OpKind::Pow) return true;
    }
    return false;
  }
  // 33 .. 64 rows: time in us of the skinny kernel and of 64 x 64 tiles, fitted to 1256 measured products (both layouts, 8 and
  // 16 bits, K 512 .. 14336, N 1024 .. 16384; the first within 11 %, the second within a quarter; standard deviations 3 and 6 %).
  double skinnyTime(int64_t split) const {
    const double mb = static_cast<double>(k_ * n_ * elemBytes()) * 1e-6, rows = static_cast<double>(m_);
    const double groups = static_cast<double>((n_ + 127) / 128 * split);
    const bool wide = elemBytes() == 2;
    const double start = transB_ ? (wide ? 9.1 : 7.8) : (wide ? 7.0 : 5.9), rate = transB_ ? (wide ? 0.155 : 0.175) : (wide ? 0.179 : 0.224);
    const double perRow = (transB_ ? (wide ? 0.035 : 0.047) : 0.068) / 32, idle = transB_ ? 0.105 : (wide ? 0.16 : 0.136);
    const double pitch = !transB_ && n_ * elemBytes() % 128 != 0 ? 0.04 : 0;   // rows of B begin inside a cache line
    return start + mb * (rate + perRow * (rows - 33) + idle * std::max(0.0, 224 / groups - 1) + pitch) + 0.4 * static_cast<double>(split) * rows / 64;
  }
  double smallTileRowsTime(int64_t split) const {
    const int64_t steps = (k_ * elemBytes() + 127) / 128;
    const double perCu = static_cast<double>((n_ + 63) / 64 * split) / 256, mb = static_cast<double>(k_ * n_ * elemBytes()) * 1e-6;
    const bool transposing8 = elemBytes() == 1 && !transB_;
    const double step = perCu <= 1 ? (transposing8 ? 0.35 : 0.23) : (transposing8 ? 0.6 : 0.41), rate = transposing8 ? 0.17 : 0.113;
    return 2.7 + static_cast<double>((steps + split - 1) / split) * step + mb * rate + (split > 1 ? 1.8 + 0.25 * static_cast<double>(split) + 0.5 * perCu : 0);
  }
  // The small-tile kernel where its estimate is below that of the 256 x 256 kernel, on the workgroup with the lowest one, and
  // for 33 .. 64 rows where the skinny one is not estimated a twentieth faster ([N,K] weights, whose estimates scatter more: a tenth, and those of
  // 16 bits are the skinny kernel's from 60 Mi elements on, where 8192 x 8184 takes 36.3 us for 30.3). Measured (us, 256 x 256
  // tiles / one 64 x 64 .. 128 x 128 tile a workgroup / this): bf16 300 x 4096 x 11000 [K,N] 90 / 52 / 43, 948 x 5184 x 6608 129 / 80 / 74, 1113 x
  // 4352 x 7776 142 / 113 / 75, 2168 x 4416 x 2248 102 / 56 / 49, 1096 x 1408 x 4592 42 / 36 / 20, 2936 x 6400 x 808 70 / 55 / 45, 720 x 2496 x 1368 36 / 14.5 / 14.5; 45 products
  // that no constant was fitted to take 0.78 of the time on the average, the worst of them 248 x 6656 x 2256 (20.2 -> 21.5);
  // it is the slower one, and the estimates say so, for 3568 x 5056 x 3848 (137 / 193 / 167) and 1881 x 4160 x 7568 (118 / 152 / 125).
  // The skinny one is faster at 33 rows for [K,N] weights of bf16 8192 x 6144 (30.9 for 26.1), int8 4096 x 6144 (14.8 for 13.4) and 6144 x 9216
  // (27.9 for 20.0), for [N,K] of bf16 11008 x 5120 (34.1 for 28.1).
  // Weights below 2 MiB with K from 1024 on (256 columns: 512) and at most 512 rows x 768 of whole 256-wide columns (or whose sums are rounded once by request) and those
  // of whole 256-wide columns from 2^26 elements on keep the kernels and splits that tests pin, though small tiles would be the faster ones there for some rows: int8
  // 121 x 1344 x 768 takes 26.9 us for their 5.5, bf16 8192 x 8192 with 96 rows 50.7 for 41.5. Other weights below 2 MiB take them (us: whole
  // 256-wide columns f16 181 x 576 x 1280 27.8 -> 4.3, 8192 x 768 x 768 22.1 -> 17.5, int8 768 x 1408 x 512 31.3 -> 6.2, 2276 x 384 x 3072
  // 20.3 -> 11.6, 200 such products a third of the time in the mean, none slower; others bf16 85 x 1088 x 816 22.7 -> 4.9,
  // 365 x 1408 x 744 34.0 -> 7.4, 1096 x 1152 x 552 34.4 -> 7.0, int8 200 x 640 x 584 20.7 -> 4.5), and those of ragged columns from
  // 2^26 elements on (us: int8 [N,K] 320 x 8192 x 8200 72 -> 38, f16 69 x 9728 x 13872 111 -> 60, [K,N] 845 x 8128 x 8560 206 -> 124; 103 products 0.75 of the
  // time in the mean, 130 others 0.74; f16 [N,K] 1600 x 12160 x 7408 the slowest of them, 274 -> 301; with at most 256 rows where they are estimated a
  // fifth faster: f16 [K,N] 216 x 16128 x 8872, estimated 0.89, takes 141 on 256 x 256 tiles and 151). Narrow products of at most 64 rows (N < 1024) are the skinny kernel's.
  bool pickSmallTile() {
    if (serial_ || dyn_ || batch_ != 1 || opt_.split > 0 || (opt_.variant & (8 | 128))) return false;
    const int64_t elements = k_ * n_;
    const bool narrow = m_ <= skinnyRows();
    if (m_ <= 32 || (elements >= (1LL << 26) && (narrow || n_ % 256 == 0))) return false;
    if (!transB_ && elements * elemBytes() >= (1LL << 31)) return false;   // (the row of a [K,N] weight is a 31-bit offset)
    const bool fewWhole = n_ % 256 == 0 && n_ <= 768 && m_ <= 512 && k_ >= (n_ <= 256 ? 512 : 1024);
    if (elements * elemBytes() < (2LL << 20) && (narrow || fewWhole || roundedOnce_)) return false;
    if (narrow && n_ < 1024) return false;
    // (Rows of a [K,N] weight that are not whole 16-byte chunks: with 8 bits and more than 64 rows. us, 256 x 256 tiles -> small ones:
    // 219 x 3776 x 5640 38.5 -> 17.2, 836 x 4544 x 9240 97 -> 49, 104 x 768 x 9080 18.9 -> 6.8, 2002 x 3200 x 8280 108 -> 73. For
    // 16 bits a test pins the other kernel.)
    if (!transB_ && n_ * elemBytes() % 16 != 0 && (narrow || elemBytes() == 2)) return false;
    const int64_t steps = (k_ * elemBytes() + 127) / 128;
    // (columns that are whole 256-wide tiles pad nothing there: small ones from a quarter below on; 1200 x 8192 x 2048, which a test
    // pins, takes 59.6 us on them and 56.4 on 128 x 128)
    // What the estimates above leave out, the operands' and the result's way from and to memory, is the same for every small tile: with it
    // they are 2 % below 224 products measured, without 21 %. (Not those of 8-bit [K,N] weights, which are 5 % above as they are, nor with at most 256 rows or whole 256-wide
    // columns, where the other estimate leaves it out too, nor with 16 steps and less, where single tiles wait for it beside each other: with it
    // they are 14 % above for 16 bits and up to eight steps, without 3 % below.) us, taken without it
    // and on 256 x 256 tiles: f16 [N,K] 1600 x 12160 x 7408 311 / 277, 3931 x 2144 x 6224 123 / 111, int8 908 x 9600 x 12216 126 / 114; the other way round
    // int8 [N,K] 2390 x 640 x 5184 20.4 / 21.0, f16 710 x 7104 x 15856 183 / 197, bf16 with few steps 6345 x 448 x 5164 43.0 / 54.2, 3822 x 704 x 9200
    // 59.4 / 70.9, with GELU behind it 6660 x 128 x 3088 19.7 / 29.5, [K,N] 7633 x 832 x 2704 54.1 / 61.7.
    const bool transposing8 = elemBytes() == 1 && !transB_, moved = !transposing8 && m_ > 256 && n_ % 256 != 0 && steps > 16 && !outgrowsLaunch(largeTileSplit());
    const double traffic = moved ? (0.09 * static_cast<double>(elements * elemBytes()) + 0.19 * static_cast<double>(m_ * k_ * elemBytes()) + 0.18 * static_cast<double>(m_ * n_)) * 1e-6 : 0;
    double best = narrow ? 1e30 : (n_ % 256 == 0 ? 0.75 : elements >= (1LL << 26) && m_ <= 256 ? 0.8 : transposing8 && !outgrowsLaunch(largeTileSplit()) ? 1.1 : 1.0) * largeTileTime(largeTileSplit()) - traffic;
    for (const SmallShape &w : smallShapes()) {
      if ((narrow && w.m > 64) || k_ * elemBytes() * std::max(w.m, w.n) >= (1LL << 31)) continue;
      // (several tiles a workgroup from 17 steps on: for fewer, what comes behind the loop is a third of their time;
      // 464 x 576 x 10032 would take 11.8 us for 13.1, 645 x 1024 x 6008, whose tile a test pins, 16.0 for 20.2)
      if (w.m * w.n > 128 * 128 && steps <= 16) continue;
      const int64_t tiles = ((m_ + w.m - 1) / w.m) * ((n_ + w.n - 1) / w.n);
      // Partials stay within the 16 MiB of a launch without allocations, those of the larger tiles within 15. Where they do not, half as
      // many workgroups a tile, or one. us, K split as estimated / this: bf16 1130 x 12800 x 512 39.8 / 40.9 (47.6 on the tile estimated
      // next), 338 x 13712 x 1368 51.5 / 56.1, 71 x 14272 x 4496 43.6 / 49.5, int8 2518 x 2528 x 808 20.0 / 17.2, 5350 x 3280 x 552 30.3 / 22.7.
      const auto partialsFit = [&](int split) {
        const int64_t bytes = tiles * split * w.m * w.n * 4;
        return w.m * w.n > 64 * 128 ? bytes <= (15LL << 20) : bytes + tiles * 4 + 256 <= (16LL << 20);
      };
      for (int split = 1; split <= w.splits; split *= 2) {
        if (split > 1 && (split - 1) * ((steps + split - 1) / split) >= steps) continue;   // no empty split
        // (8-bit weights below 2 MiB with more than 16 steps: two workgroups a tile at least, where a test of workspaces wants one
        // and the launch without allocations has the memory; estimated 0.5 us slower, and 20.7 -> 6 us against 256 x 256 tiles)
        if (split == 1 && elemBytes() == 1 && steps > 16 && elements < (2LL << 20) && partialsFit(2)) continue;
        if (tiles * split * w.m * w.n * 4 >= (1LL << 30)) continue;
        int parts = split;
        if (!narrow && split > 1 && !partialsFit(split)) {
          parts = split / 2;
          if (parts == 1 || !partialsFit(parts)) continue;
        }
        const double t = smallTileTime(w, split) * (split > 1 ? 1.03 : 1);   // (as fast without a workspace is better)
        if (t >= best) continue;
        best = t;
        tileM_ = w.m;
        tileN_ = w.n;
        kSplit_ = parts;
      }
    }
    const bool large = transB_ && elemBytes() == 2 && elements >= (60LL << 20);
    if (skinnyTakes() && (large || skinnyTime(skinnySplit()) < (transB_ ? 0.9 : 0.95) * smallTileRowsTime(kSplit_))) tileM_ = tileN_ = 0;
    return tileM_ > 0;
  }

  bool skinnyTakes() const {
    return m_ <= skinnyRows() && (k_ * elemBytes()) % 32 == 0 && (transB_ || n_ % 4 == 0) && !(opt_.variant & 8);
  }
  int64_t skinnySplit() const {
    const int64_t strips = (n_ + 127) / 128, steps = k_ * elemBytes() / 32;
    int64_t want = opt_.split > 0 ? opt_.split : std::max<int64_t>(1, 256 / (strips * batch_));
    want = std::min<int64_t>(want, std::max<int64_t>(1, opt_.split > 0 ? steps : steps / 16));
    // (the last workgroup of a strip adds the partials of all its splits: 16 x 8192 x 1024 takes 10.1 us with 16
    // splits, 12.9 with the 32 that would fill the chip)
    want = std::min<int64_t>(want, 16);
    while (want > 1 && strips * batch_ * want * m_ * 128 * 4 >= (1LL << 30)) --want;
    return want;
  }

  // Few tiles and a long K (a skinny activation in front of a big weight matrix: M = 16 .. 1024 against 8192 x 8192
  // leaves 32 .. 128 of 256 CUs busy, and the time is that of streaming the weights through those few): split K over
  // enough workgroups to fill the chip, at least four K steps each.
  void pickSplit() {
    kSplit_ = 1;
    if (serial_) return;
    dyn_ = opt_.extentAsArgument && batch_ == 1;
    if (pickSmallTile()) {
      // (0.8: 32 products of a split K 0.57 .. 0.71 of the time, without a split 0.94 between 0.72 and 0.8, six of 34 slower by up to 9 %)
      if (m_ > skinnyRows() || !pickNarrow((kSplit_ > 1 ? 0.8 : 0.72) * smallTileRowsTime(kSplit_))) return;
      tileM_ = tileN_ = 0;
    }
    kSplit_ = 1;
    // At most 64 rows of A (and K a multiple of 32 bytes): the time is that of streaming B, which gemm_skinny reads
    // straight into MFMA operands, or a [N,K] one by whole lines through LDS of each wavefront (skinnyLines()); 256
    // workgroups of four wavefronts (one per CU: 16 x 8192 x 8192 bf16 with a [K,N] weight reaches 66 % of the HBM peak
    // with 4 splits of 64 strips, 59 % with 8, 48 % with 2; 8 wavefronts or more steps in flight change nothing), each
    // wavefront with at least 4 MFMA steps.
    // AKG_HIP_VARIANT bit 3 keeps the 256 x 256 tile kernel.
    skinny_ = skinnyTakes();
    if (skinny_) {
      if (narrowCols_ > 0) return;   // (instead of small tiles)
      kSplit_ = static_cast<int>(skinnySplit());
      if (pickNarrow(m_ <= 32 ? 0.92 * wideStripTime() : 0.85 * skinnyTime(kSplit_))) kSplit_ = 1;
      return;
    }
    if (batch_ != 1) return;
    kSplit_ = static_cast<int>(largeTileSplit());
  }

  // us of the narrow strips, fitted to 122 products of at most 64 rows on 16, 32 and 64 columns (575 in all, both layouts, 8 and 16
  // bits, 0.4 to 96 MB of weight; standard deviation 12 %): a start, what a CU takes in of the weight and of A (32 columns of
  // 16-bit k-rows are half lines), and the weight from memory.
  double narrowTime(int64_t cols) const {
    const double kb = static_cast<double>(k_ * elemBytes()) / 1024, mb = static_cast<double>(k_ * n_ * elemBytes()) * 1e-6;
    const double strips = static_cast<double>((n_ + cols - 1) / cols) / 256;
    const double perCu = (strips <= 1 ? 1 : 0.5 * (strips + std::ceil(strips))) * kb, rows = static_cast<double>(m_), width = static_cast<double>(cols);
    if (transB_) return 3.02 + perCu * (0.0104 * width + 0.014 * rows) + 0.091 * mb;
    if (elemBytes() == 1) return 2.74 + perCu * (0.0195 * width + 0.026 * rows) + 0.119 * mb;
    return cols == 32 ? 2.33 + perCu * (0.0173 * width + 0.0172 * rows) + 0.107 * mb : 2.4 + perCu * (0.0145 * width + 0.019 * rows) + 0.102 * mb;
  }
  // ... and of the strips of 128 columns for at most 32 rows (90 of the same products, 6 %).
  double wideStripTime() const {
    const double mb = static_cast<double>(k_ * n_ * elemBytes()) * 1e-6, rows = static_cast<double>(m_), splits = static_cast<double>(skinnySplit());
    const double idle = std::max(0.0, 224 / (static_cast<double>((n_ + 127) / 128) * splits) - 1);
    if (transB_) return 5.41 + mb * ((elemBytes() == 1 ? 0.147 : 0.135) + 0.00174 * rows) + 0.0068 * splits * rows;
    return 6.32 + mb * ((elemBytes() == 1 ? 0.235 : 0.15) + 0.00196 * rows - 0.094 * idle) + 0.0108 * splits * rows;
  }
  // Narrow strips, each the whole K of one workgroup, where they are estimated faster than the kernel that `other` us are the estimate
  // of: they save the exchange of partials (3 of 6 us), and lose where few strips leave CUs idle with a long K, or where the rows of A,
  // which every strip reads, weigh more than its columns. us, strips of 128 columns / narrow ones: bf16 [N,K] 8 x 640 x 1336 6.0 / 3.2,
  // 4 x 5056 x 2176 10.0 / 6.2, 32 x 7040 x 1832 13.7 / 11.0, 16 x 7360 x 3536 15.5 / 13.5; [K,N] 2 x 512 x 2912 5.3 / 3.4, 25 x 896 x 5656 9.2 / 5.2,
  // 16 x 2880 x 5408 11.3 / 7.7, 5 x 6592 x 560 8.1 / 12.7, 26 x 5248 x 8632 27 / 32; int8 [N,K] 9 x 2688 x 3760 7.7 / 4.4, [K,N] 1 x 1920 x
  // 4808 8.2 / 6.3; small tiles / narrow strips: int8 [K,N] 49 x 1856 x 11256 16.6 / 10.0, bf16 [N,K] 62 x 1536 x 5880 7.7 / 8.1. 390
  // other products that take them need 0.68 of the time in the geometric mean, int8 32 x 7616 x 6172 15.2 / 16.3 the slowest of them.
  // More than 32 rows only with the weights that were measured, up to 24 MiB. A weight that is read past the caches keeps its kernel, as does one of a description with an open
  // row count or of several batches. (AKG_HIP_VARIANT bit 8 keeps the strips of 128 columns.)
  bool pickNarrow(double other) {
    narrowCols_ = 0;
    if (dyn_ || batch_ != 1 || !skinnyTakes() || opt_.split > 0 || opt_.block > 0 || opt_.chunks > 0 || (opt_.variant & 256)) return false;
    const int64_t kBytes = k_ * elemBytes();
    if (kBytes % 64 != 0 || kBytes < 640 || weightBytes() >= ((m_ <= 32 ? 96LL : 24LL) << 20)) return false;
    // Rows of a [K,N] weight that lie a multiple of 256 bytes apart: the half lines that a strip asks for meet in few channels. us, strips
    // of 128 columns / narrow ones: int8 2 x 3584 x 5120 8.3 / 13.1, 8 x 2240 x 23552 15.0 / 20.6, f16 8 x 4096 x 8192 14.9 / 19.5, bf16 3 x 3584 x 3072
    // 8.9 / 10.9, int8 16 x 3584 x 4608 8.5 / 9.7, 4 x 2048 x 5120 7.0 / 8.5; within these limits 390 products 0.67 of the time, three slower by 2 % and more (1.03). Long
    // columns of a [N,K] weight that begin inside lines: bf16 4 x 5216 x 256 6.0 / 6.9, 2 x 6880 x 936 7.8 / 9.1, int8 2 x 13888 x 1008 8.0 / 8.9.
    if (!transB_ && n_ * elemBytes() % 256 == 0 && (kBytes > (n_ * elemBytes() % 1024 != 0 ? 3200 : elemBytes() == 1 ? 1600 : 2560) || weightBytes() >= (32LL << 20))) return false;
    if (transB_ && kBytes % 128 != 0 && kBytes > 8192 && m_ <= 32) return false;
    int64_t cols = 0;
    double best = other;
    for (const int64_t width : {16, 32, 64}) {
      if (!transB_ && width * elemBytes() < 64) continue;
      const double t = narrowTime(width);
      if (t < best) {
        best = t;
        cols = width;
      }
    }
    narrowCols_ = static_cast<int>(cols);
    // (eight wavefronts where each has two to four units of K: us, 17 x 1280 x 1368 4.36 on four and 4.23, 2 x 3584 x 4192 7.3 and 7.7)
    const int64_t units = (kBytes + 127) / 128;
    narrowWaves_ = m_ <= 32 && units >= 12 && units <= 32 ? 8 : 4;
    return cols > 0;
  }

  int64_t largeTileSplit() const {
    const int64_t tiles = ((m_ + 255) / 256) * ((n_ + 255) / 256);
    const int64_t steps = (k_ * elemBytes() + stepK() - 1) / stepK();
    int64_t want = opt_.split > 0 ? opt_.split : (tiles >= 192 ? 1 : std::min<int64_t>(16, (256 + tiles - 1) / tiles));
    want = std::max<int64_t>(1, std::min<int64_t>(want, opt_.split > 0 ? steps : steps / 4));
    const int64_t partRows = std::min<int64_t>(m_, 256);
    while (want > 1 && tiles * want * partRows * 256 * 4 >= (1LL << 30)) --want;
    if (opt_.split <= 0) {
      // the partials are written and read once: not more of them than four times the operands (2048^3 int8 with four
      // splits moved 134 MB of partials for 8 MB of operands and lost 12 %; bf16 with twice the operands gained 26 %)
      const int64_t operandBytes = (m_ * k_ + k_ * n_) * elemBytes();
      while (want > 1 && 2 * tiles * want * partRows * 256 * 4 > 4 * operandBytes) --want;
    }
    if (opt_.split <= 0) {
      // ... and the one workgroup that finishes a tile reads the partials of all its splits by itself: at most 1 MiB
      // of them (256 x 8192 x 8192: four splits 68.0 us bf16 / 47.3 us int8, eight 75.5 / 60.7; 128 rows: eight are best)
      want = std::min<int64_t>(want, std::max<int64_t>(1, (1LL << 20) / (partRows * 256 * 4)));
    }
    while (want > 1 && (want - 1) * ((steps + want - 1) / want) >= steps) --want;   // no empty split
    return std::max<int64_t>(1, want);
  }

  void analyse() {
    for (size_t i = 0; i < g_.ops.size(); ++i) {
      const OpNode &op = g_.ops[i];
      if (op.kind == OpKind::MatMul) {
        if (matmulOp_ >= 0) throw LoweringError("only one MatMul per kernel is supported");
        matmulOp_ = static_cast<int>(i);
      } else if (op.kind == OpKind::Unknown) {
        throw LoweringError("op " + op.name + " is not in the op table (mindspore.unknown cannot be legalized)");
      } else if (op.kind == OpKind::Unsupported || lowering::isReduceKind(op.kind)) {
        throw LoweringError("op " + op.name + " cannot be fused into a MatMul epilogue yet");
      }
    }
    const OpNode &mm = g_.ops[static_cast<size_t>(matmulOp_)];
    if (mm.transposeA) throw LoweringError("MatMul: transpose_a is not supported (as in the reference)");
    transB_ = mm.transposeB;
    aId_ = mm.inputs[0];
    bId_ = mm.inputs[1];
    accId_ = mm.outputs[0];
    const TensorValue &a = g_.tensor(aId_);
    const TensorValue &b = g_.tensor(bId_);
    const TensorValue &c = g_.tensor(accId_);
    if (a.inputIndex < 0 || b.inputIndex < 0) {
      throw LoweringError("MatMul operands must be kernel inputs (prologue fusion is not supported yet)");
    }
    if (a.dtype != b.dtype) throw LoweringError("MatMul: the operands must have one element type");
    if (a.dtype == DType::I8 && c.dtype == DType::I32) {
      elem_ = DType::I8;
    } else if ((a.dtype == DType::BF16 || a.dtype == DType::F16) && c.dtype == DType::F32) {
      elem_ = a.dtype;
    } else if ((a.dtype == DType::BF16 || a.dtype == DType::F16) && c.dtype == a.dtype && opt_.matmulF32Acc) {
      elem_ = a.dtype;   // the caller asked for the matrix units: float32 sum, rounded once (see LoweringOptions)
      roundedOnce_ = true;
    } else {
      // linalg.matmul converts both operands to the accumulator's element type: the same type, a wider integer, or a
      // wider float
      auto isIntType = [](DType t) { return t == DType::I8 || t == DType::I16 || t == DType::I32 || t == DType::I64; };
      const bool sameType = c.dtype == a.dtype && a.dtype != DType::Bool;
      const bool widerInt = isIntType(a.dtype) && isIntType(c.dtype) && dtypeSize(c.dtype) > dtypeSize(a.dtype);
      const bool widerFloat = isFloatType(a.dtype) && isFloatType(c.dtype) && dtypeSize(c.dtype) > dtypeSize(a.dtype);
      if (!sameType && !widerInt && !widerFloat) {
        throw LoweringError("MatMul: the result type must be the operands' type or a wider one of the same kind");
      }
      elem_ = a.dtype;
      serial_ = true;
    }
    // [M,K] x [K,N], or one leading batch dimension on all three ([B,M,K] x [B,K,N] -> [B,M,N]: linalg.batch_matmul,
    // MindSporeToLinalg.cpp:1511-1530); every batch is one grid.y slice of the same tile kernel.
    const size_t rank = a.shape.size();
    if ((rank != 2 && rank != 3) || b.shape.size() != rank || c.shape.size() != rank) {
      throw LoweringError("MatMul: operands and result must all be rank 2, or all rank 3 with one batch dimension");
    }
    const size_t o = rank - 2;
    batch_ = rank == 3 ? a.shape[0] : 1;
    if (rank == 3 && (b.shape[0] != batch_ || c.shape[0] != batch_)) throw LoweringError("MatMul: batch extents differ");
    if (batch_ < 1 || batch_ > 65535) throw LoweringError("MatMul: batch extent out of range");
    m_ = a.shape[o];
    k_ = a.shape[o + 1];
    n_ = transB_ ? b.shape[o] : b.shape[o + 1];
    const int64_t kb = transB_ ? b.shape[o + 1] : b.shape[o];
    if (kb != k_ || c.shape[o] != m_ || c.shape[o + 1] != n_) throw LoweringError("MatMul: inconsistent shapes");
    // rows of K that are not whole 16-byte pieces, N not a multiple of 4: shapes the MFMA kernels' loads do not take
    if ((k_ * elemBytes()) % 16 != 0 || n_ % 4 != 0) serial_ = true;
    if (serial_ && (m_ * k_ >= (1LL << 31) || k_ * n_ >= (1LL << 31) || m_ * n_ >= (1LL << 31))) {
      throw LoweringError("MatMul: operands of 2^31 elements and more need the MFMA kernels' shapes");
    }
    for (const OpNode &op : g_.ops) {
      if (op.kind == OpKind::MatMul) continue;
      for (int in : op.inputs) {
        if (in == aId_ || in == bId_) throw LoweringError("MatMul operands cannot also feed the epilogue");
      }
    }
    if (g_.tensor(accId_).outputIndex >= 0) {
      // the raw int32 product as an output is fine: it is just another Full value
    }
  }

  std::string ctOf(int id) const { return computeTypeName(g_.tensor(id).dtype); }
  std::string tagOf(int id) const { return dtypeTag(g_.tensor(id).dtype); }

  EpiRank classifyInput(const TensorValue &t) const {
    if (t.numel() == 1) return EpiRank::Scalar;
    // the result is addressed as [batch * M, N]: fold a leading batch dimension into the rows
    std::vector<int64_t> s = t.shape;
    while (s.size() > 3 && s.front() == 1) s.erase(s.begin());
    if (s.size() == 3) {
      if (s[0] == batch_ && s[1] == m_) {
        s = {batch_ * m_, s[2]};
      } else if (s[0] == 1 && (batch_ == 1 || s[1] == 1)) {
        s = {s[1], s[2]};
      } else {
        throw LoweringError("epilogue input " + t.name + " does not broadcast to the MatMul result");
      }
    }
    if (s.size() == 1) s.insert(s.begin(), 1);
    if (s.size() != 2) throw LoweringError("epilogue input " + t.name + ": rank exceeds the output's");
    const int64_t rows = batch_ * m_;
    if (s[0] == rows && s[1] == n_) return EpiRank::Full;
    if (s[0] == 1 && s[1] == n_) return EpiRank::Col;
    if (s[0] == rows && s[1] == 1) return EpiRank::Row;
    throw LoweringError("epilogue input " + t.name + " does not broadcast to the MatMul result");
  }

  std::string operand(int id) const {
    const EpiVal &v = vals_[static_cast<size_t>(id)];
    if (!v.defined) throw LoweringError("internal: epilogue operand " + g_.tensor(id).name + " undefined");
    if (v.rank == EpiRank::Full || v.rank == EpiRank::Col) return v.ident + "[e]";
    return v.ident;
  }

  void emit() {
    vals_.assign(g_.tensors.size(), EpiVal());
    relaxed_ = lowering::relaxedPrecisionTensors(g_);
    const bool nt = opt_.nonTemporal != 0;
    const std::string W = std::to_string(epiWidth());   // result columns per epilogue call

    // accumulators
    EpiVal &acc = vals_[static_cast<size_t>(accId_)];
    acc.defined = true;
    acc.rank = EpiRank::Full;
    acc.ident = "acc";
    const DType accDt = g_.tensor(accId_).dtype;
    if (!serial_ && (accDt == DType::F16 || accDt == DType::BF16)) {
      // a 16-bit MatMul result: the float32 sum is rounded to the declared type once
      acc.ident = "accr";
      apply_ << "    float accr[4];\n#pragma unroll\n    for (int e = 0; e < 4; ++e) accr[e] = " << dtypeTag(accDt)
             << "::rnd(acc[e]);\n";
    }

    // constants
    for (size_t t = 0; t < g_.tensors.size(); ++t) {
      if (!g_.tensors[t].isConst) continue;
      vals_[t].defined = true;
      vals_[t].rank = EpiRank::Const;
      vals_[t].ident = lowering::literalFor(g_.tensors[t].dtype, g_.tensors[t].constValue);
    }
    // inputs
    for (size_t i = 0; i < g_.inputs.size(); ++i) {
      const int id = g_.inputs[i];
      if (id == aId_ || id == bId_) continue;
      const TensorValue &t = g_.tensor(id);
      if (!t.used) continue;
      const EpiRank r = classifyInput(t);
      EpiVal &v = vals_[static_cast<size_t>(id)];
      v.defined = true;
      v.rank = r;
      const std::string tag = tagOf(id), ct = ctOf(id);
      members_ << "  const " << tag << "::storage *__restrict__ in" << i << ";\n";
      switch (r) {
        case EpiRank::Scalar:
          v.ident = "s_in" + std::to_string(i);
          members_ << "  " << ct << " " << v.ident << ";\n";
          prepare_ << "    " << v.ident << " = " << tag << "::load(in" << i << "[0]);\n";
          break;
        case EpiRank::Col:
          v.ident = "c_in" + std::to_string(i);
          members_ << "  " << ct << " " << v.ident << "[" << W << "];\n";
          prepare_ << "    akg::load_chunk<" << tag << ", " << W << ", false>(in" << i << " + col, " << v.ident << ");\n";
          break;
        case EpiRank::Row:
          v.ident = "r_in" + std::to_string(i);
          apply_ << "    const " << ct << " " << v.ident << " = " << tag << "::load(in" << i << "[grow]);\n";
          break;
        case EpiRank::Full:
          v.ident = "t_in" + std::to_string(i);
          apply_ << "    " << ct << " " << v.ident << "[" << W << "];\n";
          apply_ << "    akg::load_chunk<" << tag << ", " << W << ", " << (nt ? "true" : "false") << ">(in" << i << " + grow * " << n_
                 << "L + col, " << v.ident << ");\n";
          break;
        default:
          break;
      }
    }
    for (size_t i = 0; i < g_.outputs.size(); ++i) {
      members_ << "  " << tagOf(g_.outputs[i]) << "::storage *__restrict__ out" << i << ";\n";
    }
    // ops
    for (const OpNode &op : g_.ops) {
      if (op.kind == OpKind::MatMul) continue;
      if (op.outputs.size() != 1) throw LoweringError("op " + op.name + ": multiple results are not supported");
      const int outId = op.outputs[0];
      if (op.kind == OpKind::Assign) {
        // the value is stored over the destination (a kernel input as large as the MatMul result) besides being the
        // op's result: linalg.copy ins=value outs=destination (MindSporeToLinalg.cpp:495-524). Every thread writes
        // exactly the chunk of the destination that it has read (if the description reads it at all) before.
        const TensorValue &dst = g_.tensor(op.inputs[0]);
        if (dst.inputIndex < 0 || op.inputs[0] == aId_ || op.inputs[0] == bId_ || dst.dtype != g_.tensor(outId).dtype ||
            dst.numel() != batch_ * m_ * n_ || classifyInput(dst) != EpiRank::Full) {
          throw LoweringError("op " + op.name + ": in a MatMul fusion the destination must be a kernel input of the result's shape and type (not a MatMul operand)");
        }
        const EpiVal &value = vals_[static_cast<size_t>(op.inputs[1])];
        if (!value.defined) throw LoweringError("op " + op.name + ": value is undefined");
        const std::string ct = ctOf(outId), tag = tagOf(outId);
        EpiVal &v = vals_[static_cast<size_t>(outId)];
        v.defined = true;
        v.rank = EpiRank::Full;
        v.ident = "t" + std::to_string(outId);
        std::vector<std::string> operands = {"", operand(op.inputs[1])};
        apply_ << "    " << ct << " " << v.ident << "[" << W << "];  // " << op.name << " -> " << dst.name << "\n";
        apply_ << "#pragma unroll\n    for (int e = 0; e < " << W << "; ++e) " << v.ident << "[e] = "
               << lowering::elementwiseExpr(g_, op, operands, false) << ";\n";
        if (!g_.tensor(op.inputs[0]).used || !vals_[static_cast<size_t>(op.inputs[0])].defined) {
          members_ << "  const " << tag << "::storage *__restrict__ in" << dst.inputIndex << ";\n";
          assignOnly_.push_back(dst.inputIndex);
        }
        apply_ << "    akg::store_chunk<" << tag << ", " << W << ", false>(const_cast<" << tag << "::storage *>(in" << dst.inputIndex
               << ") + grow * " << n_ << "L + col, " << v.ident << ");\n";
        continue;
      }
      bool hasRow = false, hasCol = false, hasFull = false, hasScalar = false;
      for (int in : op.inputs) {
        const EpiVal &vi = vals_[static_cast<size_t>(in)];
        if (!vi.defined) throw LoweringError("op " + op.name + ": operand " + g_.tensor(in).name + " is undefined");
        hasRow |= vi.rank == EpiRank::Row;
        hasCol |= vi.rank == EpiRank::Col;
        hasFull |= vi.rank == EpiRank::Full;
        hasScalar |= vi.rank == EpiRank::Scalar;
      }
      EpiRank rank = EpiRank::Scalar;
      if (hasFull || (hasRow && hasCol)) {
        rank = EpiRank::Full;
      } else if (hasCol) {
        rank = EpiRank::Col;
      } else if (hasRow) {
        rank = EpiRank::Row;
      }
      (void)hasScalar;
      std::vector<std::string> operands;
      for (int in : op.inputs) operands.push_back(operand(in));
      const std::string expr = lowering::elementwiseExpr(g_, op, operands, relaxed_[static_cast<size_t>(outId)]);
      EpiVal &v = vals_[static_cast<size_t>(outId)];
      v.defined = true;
      v.rank = rank;
      const std::string ct = ctOf(outId);
      const std::string comment = "  // " + op.name + " -> " + g_.tensor(outId).name + "\n";
      switch (rank) {
        case EpiRank::Full:
          v.ident = "t" + std::to_string(outId);
          apply_ << "    " << ct << " " << v.ident << "[" << W << "];" << comment;
          apply_ << "#pragma unroll\n    for (int e = 0; e < " << W << "; ++e) " << v.ident << "[e] = " << expr << ";\n";
          break;
        case EpiRank::Col:
          v.ident = "c" + std::to_string(outId);
          members_ << "  " << ct << " " << v.ident << "[" << W << "];\n";
          prepare_ << "#pragma unroll\n    for (int e = 0; e < " << W << "; ++e) " << v.ident << "[e] = " << expr << ";" << comment;
          break;
        case EpiRank::Row:
          v.ident = "r" + std::to_string(outId);
          apply_ << "    const " << ct << " " << v.ident << " = " << expr << ";" << comment;
          break;
        default:
          v.ident = "s" + std::to_string(outId);
          members_ << "  " << ct << " " << v.ident << ";\n";
          prepare_ << "    " << v.ident << " = " << expr << ";" << comment;
          break;
      }
    }
    // stores
    for (size_t i = 0; i < g_.outputs.size(); ++i) {
      const int id = g_.outputs[i];
      const TensorValue &t = g_.tensor(id);
      const EpiVal &v = vals_[static_cast<size_t>(id)];
      if (!v.defined) throw LoweringError("output " + t.name + " is never computed");
      if (t.numel() != batch_ * m_ * n_ || v.rank != EpiRank::Full) {
        throw LoweringError("output " + t.name + ": only [M,N] outputs of a MatMul fusion are supported");
      }
      apply_ << "    akg::store_chunk<" << tagOf(id) << ", " << W << ", " << (nt ? "true" : "false") << ">(out" << i << " + grow * "
             << n_ << "L + col, " << v.ident << ");\n";
    }

    const std::string kname = g_.name + "_kernel";
    src_ << "// Generated by the akg HIP lowering for gfx950. Op description: " << g_.name << "\n";
    src_ << "// family: gemm_epilogue, fusion class: " << operatorTemplateName(g_.operatorTemplate) << "\n";
    src_ << "#include \"akg_rt.hpp\"\n#include \"" << (serial_ ? "akg_gemm_serial.hpp" : "akg_gemm_mfma.hpp") << "\"\n\n";
    src_ << "namespace {\nstruct Epilogue {\n" << members_.str();
    src_ << "  AKG_DEV void prepare(long col) {\n    (void)col;\n" << prepare_.str() << "  }\n";
    src_ << "  long row0;  // first row of this batch in the [batch * M, N] view of the result\n";
    src_ << "  AKG_DEV void apply(const " << accType() << " (&acc)[" << W << "], long row, long col) {\n"
         << "    const long grow = row0 + row;\n    (void)grow;\n" << apply_.str() << "  }\n";
    src_ << "};\n}  // namespace\n\n";
    src_ << "extern \"C\" __global__ __launch_bounds__(" << (serial_ ? 256 : (skinny_ ? skinnyWaves() * 64 : (tileM_ > 0 ? 256 : 512))) << ") void " << kname << "(";
    size_t argc = 0;
    for (size_t i = 0; i < g_.inputs.size(); ++i, ++argc) {
      src_ << (argc ? ", " : "") << "const " << tagOf(g_.inputs[i]) << "::storage *__restrict__ in" << i;
    }
    for (size_t i = 0; i < g_.outputs.size(); ++i, ++argc) {
      src_ << (argc ? ", " : "") << tagOf(g_.outputs[i]) << "::storage *__restrict__ out" << i;
    }
    if (dyn_) src_ << ", const long akg_m, const long akg_ksplit";
    if (kSplit_ > 1 || dyn_) src_ << ", unsigned *__restrict__ akg_ws";
    src_ << ") {\n  Epilogue epi;\n  const long akg_batch = static_cast<long>(blockIdx.y);\n";
    if (dyn_) {
      src_ << "  epi.row0 = 0L;   // (one batch)\n";
    } else {
      src_ << "  epi.row0 = akg_batch * " << m_ << "L;\n";
    }
    for (size_t i = 0; i < g_.inputs.size(); ++i) {
      const int id = g_.inputs[i];
      const bool written = std::find(assignOnly_.begin(), assignOnly_.end(), static_cast<int>(i)) != assignOnly_.end();
      if (id == aId_ || id == bId_ || (!g_.tensor(id).used && !written)) continue;
      src_ << "  epi.in" << i << " = in" << i << ";\n";
    }
    for (size_t i = 0; i < g_.outputs.size(); ++i) src_ << "  epi.out" << i << " = out" << i << ";\n";
    if (serial_) {
      src_ << "  akg::gemm_serial<" << tagOf(aId_) << ", " << tagOf(accId_) << ", " << m_ << "L, " << n_ << "L, " << k_ << "L, "
           << (transB_ ? "true" : "false") << ", " << W << ", Epilogue>(in" << g_.tensor(aId_).inputIndex << " + akg_batch * "
           << m_ * k_ << "L, in" << g_.tensor(bId_).inputIndex << " + akg_batch * " << k_ * n_ << "L, epi);\n}\n";
      return;
    }
    if (skinny_) {
      if (dyn_) {
        src_ << "  akg::gemm_skinny<" << mmaTraits() << ", " << skinnyBucket() << "L, " << n_ << "L, " << k_ << "L, " << (transB_ ? "true" : "false")
             << ", Epilogue, 1, " << skinnyWaves() << ", " << skinnyUnroll() << ", " << (skinnyNonTemporal() ? "true" : "false") << ", true>(in"
             << g_.tensor(aId_).inputIndex << ", in" << g_.tensor(bId_).inputIndex << ", epi, akg_ws, 0L, akg_m, static_cast<int>(akg_ksplit)" << linesArgument("") << ");\n}\n";
        return;
      }
      src_ << "  akg::gemm_skinny<" << mmaTraits() << ", " << m_ << "L, " << n_ << "L, " << k_ << "L, " << (transB_ ? "true" : "false")
           << ", Epilogue, " << kSplit_ << ", " << skinnyWaves() << ", " << skinnyUnroll() << ", " << (skinnyNonTemporal() ? "true" : "false") << ">(in" << g_.tensor(aId_).inputIndex << " + akg_batch * " << m_ * k_ << "L, in"
           << g_.tensor(bId_).inputIndex << " + akg_batch * " << k_ * n_ << "L, epi, " << (kSplit_ > 1 ? "akg_ws" : "nullptr")
           << ", akg_batch * " << (n_ + 127) / 128 << "L" << linesArgument(", 0L, 1") << ");\n}\n";
      return;
    }
    if (tileM_ > 0) {
      src_ << "  akg::gemm_small_tile<" << mmaTraits() << ", " << tileM_ << ", " << tileN_ << ", " << m_ << "L, " << n_ << "L, " << k_ << "L, "
           << (transB_ ? "true" : "false") << ", Epilogue, " << kSplit_ << ">(in" << g_.tensor(aId_).inputIndex << ", in"
           << g_.tensor(bId_).inputIndex << ", epi" << (kSplit_ > 1 ? ", akg_ws" : "") << ");\n}\n";
      return;
    }
    if (dyn_) {
      src_ << "  akg::gemm_256x256<" << mmaTraits() << ", 0L, " << n_ << "L, " << k_ << "L, " << (transB_ ? "true" : "false")
           << ", Epilogue, 1, " << (tallWavefrontTiles() ? 2 : 4) << ", true>(in" << g_.tensor(aId_).inputIndex << ", in" << g_.tensor(bId_).inputIndex
           << ", epi, akg_ws, akg_m, static_cast<int>(akg_ksplit));\n}\n";
      return;
    }
    src_ << "  akg::gemm_256x256<" << mmaTraits() << ", " << m_ << "L, " << n_ << "L, " << k_ << "L, " << (transB_ ? "true" : "false")
         << ", Epilogue, " << kSplit_ << (tallWavefrontTiles() ? ", 2" : "") << ">(in" << g_.tensor(aId_).inputIndex << " + akg_batch * " << m_ * k_ << "L, in" << g_.tensor(bId_).inputIndex
         << " + akg_batch * " << k_ * n_ << "L, epi" << (kSplit_ > 1 ? ", akg_ws" : "") << ");\n}\n";
  }
};

}  // namespace

LoweredKernel lowerGemmToHip(const OpGraph &graph, const LoweringOptions &options) {
  GemmEmitter emitter(graph, options);
  return emitter.run();
}

}  // namespace akg
