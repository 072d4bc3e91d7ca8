/**
 * UnsortedSegmentSum: out[ids[i], ...] += data[i, ...] for the index positions i in increasing order.
 *
 * The reference lowers it to a serial loop over the (collapsed) index positions that adds one data slice to the
 * accumulator slice its id names (MindSporeToLinalg.cpp:596-745). A GPU scatter with float atomics would add in arrival
 * order; this kernel keeps the reference's order, bit for bit, without atomics and without a zero-filled output.
 *
 * A workgroup owns a range of segments (and a tile of the slice) whose accumulators live in LDS. Every wavefront of it
 * scans ALL index positions, 64 lanes x 16 bytes of ids per load and several loads in flight, and ballots the lanes
 * whose ids fall into the range; the few matches are handled in ascending position order. For slices of up to four
 * elements the matching lane adds the whole slice itself (its data loads are issued before the serial part); for wider
 * slices thread t adds columns t, t + block, ... and only ever touches its own columns, so the wavefronts of a workgroup
 * repeat the (cheap) scan instead of sharing it and no barrier is needed. Either way the order per output element is
 * the serial one.
 * Ids outside [0, segments) match nobody and are dropped. The id array is read once per workgroup (from L2 after the
 * first), the data once overall.
 *
 * That scan costs (workgroups x positions) id reads. Inputs with many positions are grouped by segment first instead
 * (lowerSegmentSorted, lowerSegmentBucketed and lowerSegmentChunked below): same result, bit for bit.
 */
#include <algorithm>
#include <sstream>

#include "HipLowering.h"

namespace akg {

namespace {

// The shapes all schedules need.
struct SegmentShapes {
  const OpNode *op = nullptr;
  const TensorValue *data = nullptr, *ids = nullptr, *out = nullptr;
  int64_t positions = 0, segments = 0, slice = 0;
};

SegmentShapes checkSegmentSum(const OpGraph &g) {
  if (g.ops.size() != 1 || g.ops[0].kind != OpKind::SegmentSum || g.outputs.size() != 1 ||
      g.outputs[0] != g.ops[0].outputs[0]) {
    throw LoweringError("UnsortedSegmentSum can only be lowered as a kernel of its own (no fused neighbours yet)");
  }
  SegmentShapes sh;
  sh.op = &g.ops[0];
  const OpNode &op = *sh.op;
  sh.data = &g.tensor(op.inputs[0]);
  sh.ids = &g.tensor(op.inputs[1]);
  sh.out = &g.tensor(op.outputs[0]);
  if (sh.data->inputIndex < 0 || sh.ids->inputIndex < 0) throw LoweringError("op " + op.name + ": operands must be kernel inputs");
  if (sh.data->dtype != sh.out->dtype) throw LoweringError("op " + op.name + ": data and result element types differ");
  if (sh.out->dtype == DType::Bool) throw LoweringError("op " + op.name + ": bool data is not supported");
  sh.positions = sh.ids->numel();
  sh.segments = op.padValue;
  sh.slice = sh.positions > 0 ? sh.data->numel() / sh.positions : 0;
  if (sh.positions <= 0 || sh.slice <= 0 || sh.out->numel() != sh.segments * sh.slice) {
    throw LoweringError("op " + op.name + ": inconsistent shapes");
  }
  if (sh.positions >= (1LL << 31) || sh.out->numel() >= (1LL << 31) || sh.data->numel() >= (1LL << 40)) {
    throw LoweringError("op " + op.name + ": too large");
  }
  return sh;
}

// The three counting launches both grouped schedules share. The generated source must define POSITIONS, KEYS (counters
// per run), RUNS, RUN, W_HIST, W_TOTAL, W_START, as_segment() and key_of(segment):
//   <op>_count    workgroup b counts the keys of its run of positions (LDS counters) -> hist[b][key]
//   <op>_offsets  per key, the exclusive prefix of hist over b (in place) and the key's total
//   <op>_starts   exclusive prefix of the totals: where each key's list starts (and, at [KEYS], where the last one ends)
// Workgroups of the <op>_offsets launch for `keys` counters per run (see emitCountingLaunches).
int64_t offsetsGrid(int64_t keys) {
  const int64_t perWg = keys >= 4096 ? 16 : 4, groups = (keys + perWg - 1) / perWg;
  return (groups + 7) / 8 * 8;
}

void emitCountingLaunches(std::ostringstream &s, const std::string &name, const std::string &paramList, const std::string &idTag,
                          const std::string &idsName, int64_t runs, int64_t keys) {
  const int perStart = static_cast<int>((keys + 1023) / 1024);
  // ---- count ----
  s << "extern \"C\" __global__ __launch_bounds__(256) void " << name << "_count(" << paramList << ") {\n";
  s << "  __shared__ unsigned akg_cnt[KEYS];\n";
  s << "  const int tid = static_cast<int>(threadIdx.x), run = static_cast<int>(blockIdx.x);\n";
  s << "  for (int k = tid; k < KEYS; k += 256) akg_cnt[k] = 0u;\n";
  s << "  __syncthreads();\n";
  s << "  const int p0 = run * RUN, p1 = p0 + RUN < POSITIONS ? p0 + RUN : POSITIONS;\n";
  s << "#pragma unroll 4\n";
  s << "  for (int p = p0 + tid; p < p1; p += 256) {\n";
  s << "    const int id = as_segment(" << idTag << "::load(" << idsName << "[p]));\n";
  s << "    if (id >= 0) atomicAdd(&akg_cnt[key_of(id)], 1u);\n";
  s << "  }\n";
  s << "  __syncthreads();\n";
  s << "  for (int k = tid; k < KEYS; k += 256) akg_ws[W_HIST + static_cast<long>(run) * KEYS + k] = akg_cnt[k];\n";
  s << "}\n\n";

  // ---- offsets ----
  // A workgroup takes a few keys and splits the runs among its threads: KPW keys x (256 / KPW) slabs of runs. Few keys
  // (the bucketed schedule) take 4 a workgroup, so that the launch still fills the chip.
  const int keysPerWg = keys >= 4096 ? 16 : 4, slabs = 256 / keysPerWg;
  const int64_t runsPer = (runs + slabs - 1) / slabs;
  s << "extern \"C\" __global__ __launch_bounds__(256) void " << name << "_offsets(" << paramList << ") {\n";
  s << "  constexpr int PER = " << runsPer << ", KPW = " << keysPerWg << ", SLABS = " << slabs << ";   // runs per thread, keys per workgroup, threads a key\n";
  s << "  __shared__ unsigned akg_part[SLABS][KPW + 1];\n";
  s << "  const int tid = static_cast<int>(threadIdx.x), sl = tid % KPW, bl = tid / KPW;\n";
  s << "  // (workgroups of one XCD - launch order: workgroup b runs on XCD b mod 8 - take neighbouring keys, which share lines)\n";
  s << "  constexpr int GROUPS = (KEYS + KPW - 1) / KPW, PER_XCD = (GROUPS + 7) / 8;\n";
  s << "  const int group = static_cast<int>(blockIdx.x & 7u) * PER_XCD + static_cast<int>(blockIdx.x >> 3);\n";
  s << "  if (group >= GROUPS) return;   // (uniform)\n";
  s << "  const int seg = group * KPW + sl;\n";
  s << "  const int b0 = bl * PER < RUNS ? bl * PER : RUNS, b1 = b0 + PER < RUNS ? b0 + PER : RUNS;\n";
  s << "  unsigned *__restrict__ col = akg_ws + W_HIST + seg;\n";
  s << "  unsigned sum = 0u;\n";
  s << "  if (seg < KEYS) {\n";
  s << "#pragma unroll 8\n";
  s << "    for (int b = b0; b < b1; ++b) sum += col[static_cast<long>(b) * KEYS];\n";
  s << "  }\n";
  s << "  akg_part[bl][sl] = sum;\n";
  s << "  __syncthreads();\n";
  s << "  unsigned before = 0u;\n";
  s << "  for (int j = 0; j < bl; ++j) before += akg_part[j][sl];\n";
  s << "  if (seg >= KEYS) return;\n";
  s << "  if (bl == SLABS - 1) akg_ws[W_TOTAL + seg] = before + sum;\n";
  s << "  for (int b = b0; b < b1; b += 8) {\n";
  s << "    unsigned v[8];\n";
  s << "#pragma unroll\n";
  s << "    for (int j = 0; j < 8; ++j) v[j] = b + j < b1 ? col[static_cast<long>(b + j) * KEYS] : 0u;\n";
  s << "#pragma unroll\n";
  s << "    for (int j = 0; j < 8; ++j) {\n";
  s << "      if (b + j < b1) col[static_cast<long>(b + j) * KEYS] = before;\n";
  s << "      before += v[j];\n";
  s << "    }\n  }\n";
  s << "}\n\n";

  // ---- starts ----
  s << "extern \"C\" __global__ __launch_bounds__(1024) void " << name << "_starts(" << paramList << ") {\n";
  s << "  constexpr int PER = " << perStart << ";\n";
  s << "  __shared__ unsigned akg_scan[1024];\n";
  s << "  const int tid = static_cast<int>(threadIdx.x);\n";
  s << "  unsigned v[PER], sum = 0u;\n";
  s << "#pragma unroll\n";
  s << "  for (int j = 0; j < PER; ++j) {\n";
  s << "    const int seg = tid * PER + j;\n";
  s << "    v[j] = seg < KEYS ? akg_ws[W_TOTAL + seg] : 0u;\n";
  s << "    sum += v[j];\n";
  s << "  }\n";
  s << "  akg_scan[tid] = sum;\n";
  s << "  __syncthreads();\n";
  s << "  for (int d = 1; d < 1024; d <<= 1) {\n";
  s << "    const unsigned add = tid >= d ? akg_scan[tid - d] : 0u;\n";
  s << "    __syncthreads();\n";
  s << "    akg_scan[tid] += add;\n";
  s << "    __syncthreads();\n";
  s << "  }\n";
  s << "  unsigned run = akg_scan[tid] - sum;\n";
  s << "#pragma unroll\n";
  s << "  for (int j = 0; j < PER; ++j) {\n";
  s << "    const int seg = tid * PER + j;\n";
  s << "    if (seg < KEYS) akg_ws[W_START + seg] = run;\n";
  s << "    run += v[j];\n";
  s << "  }\n";
  s << "  if (tid == 1023) akg_ws[W_START + KEYS] = akg_scan[1023];\n";
  s << "}\n\n";

}

/**
 * Many positions: the scan above costs (workgroups x positions) id reads, which dominates from a few hundred thousand
 * positions on. Here the positions are first grouped by segment, in position order within a segment (a counting sort
 * whose passes only use integer counters, so nothing depends on arrival order), and then every output element is one
 * serial chain of additions over its segment's list, one lane per element, all elements in parallel:
 *
 *   <op>_count    workgroup b counts the ids of its run of positions per segment (LDS counters) -> hist[b][segment]
 *   <op>_offsets  per segment, the exclusive prefix of hist over b (in place) and the segment's total
 *   <op>_starts   exclusive prefix of the totals: where each segment's list starts
 *   <op>_place    one wavefront per run: lanes with equal ids rank themselves with ballots over the id's bits, so the
 *                 positions of a segment land in increasing order; position -> sorted[start + prefix + rank]
 *   <op>_kernel   lane c adds data[sorted[k], column] for k over its segment's list, in order, and stores the sum
 *
 * The five launches take the same arguments and share one workspace (histogram, totals, starts, sorted positions).
 */
LoweredKernel lowerSegmentSorted(const OpGraph &g, const LoweringOptions &options, const SegmentShapes &sh) {
  using lowering::computeTypeName;
  using lowering::dtypeTag;
  const TensorValue &data = *sh.data, &ids = *sh.ids, &out = *sh.out;
  const int64_t positions = sh.positions, segments = sh.segments, slice = sh.slice;
  const std::string ct = computeTypeName(out.dtype), tag = dtypeTag(out.dtype), idTag = dtypeTag(ids.dtype);
  const bool narrow = out.dtype == DType::F16 || out.dtype == DType::BF16 || out.dtype == DType::I8 || out.dtype == DType::I16;
  const std::string rndOpen = narrow ? tag + "::rnd(" : std::string("(");
  // Runs of positions: a multiple of 64 positions, at least 1024, at most 2048 runs. One wavefront places a run, and
  // the placement is bound by latency with few wavefronts and by the scattered partial-line writes with many (24.5
  // million positions of 12-byte rows: 512 runs 1.56 ms, 1024 1.06 ms, 2048 0.82 ms, 4096 1.03 ms for all launches).
  int64_t runs = options.split > 0 ? options.split : std::min<int64_t>(2048, std::max<int64_t>(1, positions / 1024));
  int64_t runLength = (positions + runs - 1) / runs;
  runLength = (runLength + 63) / 64 * 64;
  runs = (positions + runLength - 1) / runLength;
  int idBits = 1;
  while ((1LL << idBits) < segments) ++idBits;
  const int64_t chains = segments * slice;
  const int unroll = options.chunks > 0 ? options.chunks : 8;
  // Short slices (one 16-byte load per data row) are moved into segment order themselves; of wider ones only the
  // positions are.
  const int elemBytes = static_cast<int>(dtypeSize(out.dtype));
  const bool staged = slice * elemBytes <= 16;
  // workspace, in 4-byte words
  const int64_t wHist = 0, wTotal = wHist + runs * segments, wStart = wTotal + segments,
                wSorted = (wStart + segments + 1 + 3) / 4 * 4;   // 16-byte aligned
  const int64_t words = wSorted + (staged ? (positions * slice * elemBytes + 3) / 4 : positions);
  std::ostringstream s;
  s << "// Generated by the akg HIP lowering for gfx950. Op description: " << g.name << "\n";
  s << "// family: segment_sum (positions grouped by segment first), fusion class: " << operatorTemplateName(g.operatorTemplate) << "\n";
  s << "#include \"akg_rt.hpp\"\n\n";
  s << "namespace {\n";
  s << "constexpr int POSITIONS = " << positions << ", SEGMENTS = " << segments << ", KEYS = SEGMENTS, RUNS = " << runs << ", RUN = " << runLength
    << ", ID_BITS = " << idBits << ";\n";
  s << "constexpr long SLICE = " << slice << ", CHAINS = " << chains << ";\n";
  s << "constexpr long W_HIST = " << wHist << ", W_TOTAL = " << wTotal << ", W_START = " << wStart << ", W_SORTED = " << wSorted << ";\n";
  s << "using id_t = " << idTag << "::storage;\n";
  // ids as int: anything outside [0, SEGMENTS) becomes -1 (belongs to no segment and is dropped)
  if (ids.dtype == DType::I64) {
    s << "__device__ inline int as_segment(long v) { return v < 0 || v >= SEGMENTS ? -1 : static_cast<int>(v); }\n";
  } else {
    s << "__device__ inline int as_segment(int v) { return v < 0 || v >= SEGMENTS ? -1 : v; }\n";
  }
  s << "__device__ inline int key_of(int segment) { return segment; }\n";
  s << "}  // namespace\n\n";
  std::ostringstream params;
  for (size_t i = 0; i < g.inputs.size(); ++i) {
    params << (i ? ", " : "") << "const " << dtypeTag(g.tensor(g.inputs[i]).dtype) << "::storage *__restrict__ in" << i;
  }
  params << ", " << tag << "::storage *__restrict__ out0, unsigned *__restrict__ akg_ws";
  const std::string idsName = "in" + std::to_string(ids.inputIndex), dataName = "in" + std::to_string(data.inputIndex);

  emitCountingLaunches(s, g.name, params.str(), idTag, idsName, runs, segments);

  // ---- place ----
  s << "extern \"C\" __global__ __launch_bounds__(64) void " << g.name << "_place(" << params.str() << ") {\n";
  s << "  constexpr int U = 8;   // tiles of 64 positions whose ids are in flight together\n";
  s << "  __shared__ unsigned akg_next[SEGMENTS];\n";
  s << "  const int lane = static_cast<int>(threadIdx.x), run = static_cast<int>(blockIdx.x);\n";
  s << "  for (int k = lane; k < SEGMENTS; k += 64) {\n";
  s << "    akg_next[k] = akg_ws[W_START + k] + akg_ws[W_HIST + static_cast<long>(run) * SEGMENTS + k];\n";
  s << "  }\n";
  s << "  __syncthreads();\n";
  s << "  // one wavefront: its LDS accesses complete in program order, so the loop needs no barrier\n";
  s << "  const int p0 = run * RUN, p1 = p0 + RUN < POSITIONS ? p0 + RUN : POSITIONS;\n";
  s << "  const unsigned long long below = (1ull << lane) - 1ull;\n";
  if (staged) {
    // rows are copied in the widest unit that divides them (their values are not looked at)
    const int64_t rowBytes = slice * elemBytes;
    const int unitBytes = rowBytes % 4 == 0 ? 4 : rowBytes % 2 == 0 ? 2 : 1;
    s << "  using unit_t = " << (unitBytes == 4 ? "unsigned" : unitBytes == 2 ? "unsigned short" : "unsigned char") << ";\n";
    s << "  constexpr int UNITS = " << rowBytes / unitBytes << ";\n";
    s << "  const unit_t *__restrict__ rows = reinterpret_cast<const unit_t *>(" << dataName << ");\n";
    s << "  unit_t *__restrict__ placed = reinterpret_cast<unit_t *>(akg_ws + W_SORTED);\n";
  }
  s << "  for (int base = p0; base < p1; base += 64 * U) {\n";
  s << "    int id[U];\n";
  if (staged) s << "    unit_t row[U][UNITS];\n";
  s << "#pragma unroll\n";
  s << "    for (int u = 0; u < U; ++u) {\n";
  s << "      const int p = base + u * 64 + lane;\n";
  s << "      id[u] = p < p1 ? as_segment(" << idTag << "::load(" << idsName << "[p])) : -1;\n";
  if (staged) {
    s << "#pragma unroll\n";
    s << "      for (int c = 0; c < UNITS; ++c) row[u][c] = p < p1 ? rows[static_cast<long>(p) * UNITS + c] : unit_t(0);\n";
  }
  s << "    }\n";
  s << "#pragma unroll\n";
  s << "    for (int u = 0; u < U; ++u) {\n";
  s << "      if (base + u * 64 < p1) {   // (uniform; a guard and not a break, so that the tiles stay in registers)\n";
  s << "      // lanes of this tile with the same id as mine\n";
  s << "      unsigned long long same = __ballot(id[u] >= 0);\n";
  s << "#pragma unroll\n";
  s << "      for (int bit = 0; bit < ID_BITS; ++bit) {\n";
  s << "        const bool set = ((id[u] >> bit) & 1) != 0;\n";
  s << "        const unsigned long long with = __ballot(set);\n";
  s << "        same &= set ? with : ~with;\n";
  s << "      }\n";
  s << "      if (id[u] >= 0) {\n";
  s << "        const unsigned at = akg_next[id[u]];\n";
  s << "        const unsigned rank = static_cast<unsigned>(__popcll(same & below));\n";
  if (staged) {
    s << "#pragma unroll\n";
    s << "        for (int c = 0; c < UNITS; ++c) placed[static_cast<long>(at + rank) * UNITS + c] = row[u][c];\n";
  } else {
    s << "        akg_ws[W_SORTED + at + rank] = static_cast<unsigned>(base + u * 64 + lane);\n";
  }
  s << "        if ((same >> lane) >> 1 == 0ull) akg_next[id[u]] = at + rank + 1u;   // the group's highest lane\n";
  s << "      }\n";
  s << "      }\n";
  s << "    }\n";
  s << "  }\n";
  s << "}\n\n";

  // ---- chains ----
  // Short slices (one 16-byte load per data row): the wavefront of a few segments fetches 256 list entries per segment
  // and round with all its lanes (positions, then rows, many loads in flight), stages the rows in LDS, and one lane
  // per output element adds them in list order. Wide slices have enough output elements to hide the latency of a
  // plain loop per element, whose lanes read neighbouring columns of the same rows.
  int64_t segsPerWave = 1;
  if (staged) {
    segsPerWave = std::max<int64_t>(1, std::min<int64_t>(segments / 2048, 64 / slice));
    segsPerWave = std::min<int64_t>(segsPerWave, 8);
    s << "extern \"C\" __global__ __launch_bounds__(64) void " << g.name << "_kernel(" << params.str() << ") {\n";
    s << "  constexpr int S = " << segsPerWave << ", E = 256, ROW = " << slice << ";   // segments per wavefront, entries per round\n";
    s << "  __shared__ " << ct << " akg_tile[S * E * ROW];\n";
    s << "  const int lane = static_cast<int>(threadIdx.x), seg0 = static_cast<int>(blockIdx.x) * S;\n";
    s << "  const " << tag << "::storage *__restrict__ placed = reinterpret_cast<const " << tag << "::storage *>(akg_ws + W_SORTED);\n";
    s << "  unsigned from[S], upto[S], longest = 0u;\n";
    s << "#pragma unroll\n";
    s << "  for (int i = 0; i < S; ++i) {\n";
    s << "    const bool real = seg0 + i < SEGMENTS;\n";
    s << "    from[i] = real ? akg_ws[W_START + seg0 + i] : 0u;\n";
    s << "    upto[i] = real ? akg_ws[W_START + seg0 + i + 1] : 0u;\n";
    s << "    longest = upto[i] - from[i] > longest ? upto[i] - from[i] : longest;\n";
    s << "  }\n";
    s << "  // the output element of this lane, if it has one\n";
    s << "  const int cs = lane / ROW, cc = lane - cs * ROW;\n";
    s << "  const bool adds = lane < S * ROW && seg0 + cs < SEGMENTS;\n";
    s << "  unsigned mine = 0u;\n";
    s << "#pragma unroll\n";
    s << "  for (int i = 0; i < S; ++i) mine = cs == i ? upto[i] - from[i] : mine;\n";
    s << "  " << ct << " acc = " << lowering::literalFor(out.dtype, 0.0) << ";\n";
    s << "  for (unsigned r = 0; r < longest; r += E) {\n";
    s << "    " << ct << " v[S][4 * ROW];\n";
    s << "#pragma unroll\n";
    s << "    for (int i = 0; i < S; ++i) {\n";
    s << "      const unsigned k = from[i] + r + lane * 4;\n";
    s << "      if (k + 4 <= upto[i]) {\n";
    s << "        akg::load_chunk_unaligned<" << tag << ", 4 * ROW>(placed + static_cast<long>(k) * ROW, v[i]);\n";
    s << "      } else {\n";
    s << "#pragma unroll\n";
    s << "        for (int e = 0; e < 4 * ROW; ++e) {\n";
    s << "          if (k + e / ROW < upto[i]) v[i][e] = " << tag << "::load(placed[static_cast<long>(k) * ROW + e]);\n";
    s << "        }\n";
    s << "      }\n";
    s << "    }\n";
    s << "#pragma unroll\n";
    s << "    for (int i = 0; i < S; ++i) {\n";
    s << "      const unsigned k = from[i] + r + lane * 4;\n";
    s << "#pragma unroll\n";
    s << "      for (int e = 0; e < 4; ++e) {\n";
    s << "        if (k + e < upto[i]) {\n";
    s << "#pragma unroll\n";
    s << "          for (int c = 0; c < ROW; ++c) akg_tile[((i * E) + lane * 4 + e) * ROW + c] = v[i][e * ROW + c];\n";
    s << "        }\n";
    s << "      }\n";
    s << "    }\n";
    s << "    __syncthreads();\n";
    s << "    if (adds && r < mine) {\n";
    s << "      const int n = mine - r < static_cast<unsigned>(E) ? static_cast<int>(mine - r) : E;\n";
    s << "      const " << ct << " *__restrict__ row = akg_tile + cs * E * ROW + cc;\n";
    s << "      int j = 0;\n";
    s << "      for (; j + 8 <= n; j += 8) {\n";
    s << "        " << ct << " t[8];\n";
    s << "#pragma unroll\n";
    s << "        for (int u = 0; u < 8; ++u) t[u] = row[(j + u) * ROW];\n";
    s << "#pragma unroll\n";
    s << "        for (int u = 0; u < 8; ++u) acc = " << rndOpen << "akg::op_add(t[u], acc));\n";
    s << "      }\n";
    s << "      for (; j < n; ++j) acc = " << rndOpen << "akg::op_add(row[j * ROW], acc));\n";
    s << "    }\n";
    s << "    __syncthreads();\n";
    s << "  }\n";
    s << "  if (adds) out0[static_cast<long>(seg0 + cs) * ROW + cc] = " << tag << "::store(acc);\n";
    s << "}\n";
  } else {
    s << "extern \"C\" __global__ __launch_bounds__(256) void " << g.name << "_kernel(" << params.str() << ") {\n";
    s << "  constexpr int U = " << unroll << ";\n";
    s << "  const long c = static_cast<long>(blockIdx.x) * 256 + static_cast<long>(threadIdx.x);\n";
    s << "  if (c >= CHAINS) return;\n";
    s << "  const int seg = static_cast<int>(c / SLICE);\n";
    s << "  const long col = c - static_cast<long>(seg) * SLICE;\n";
    s << "  const unsigned *__restrict__ sorted = akg_ws + W_SORTED;\n";
    s << "  const " << tag << "::storage *__restrict__ data = " << dataName << " + col;\n";
    s << "  unsigned k = akg_ws[W_START + seg];\n";
    s << "  const unsigned end = akg_ws[W_START + seg + 1];\n";
    s << "  " << ct << " acc = " << lowering::literalFor(out.dtype, 0.0) << ";\n";
    s << "  for (; k + U <= end; k += U) {\n";
    s << "    unsigned p[U];\n";
    s << "    " << ct << " v[U];\n";
    s << "#pragma unroll\n";
    s << "    for (int u = 0; u < U; ++u) p[u] = sorted[k + u];\n";
    s << "#pragma unroll\n";
    s << "    for (int u = 0; u < U; ++u) v[u] = " << tag << "::load(data[static_cast<long>(p[u]) * SLICE]);\n";
    s << "#pragma unroll\n";
    s << "    for (int u = 0; u < U; ++u) acc = " << rndOpen << "akg::op_add(v[u], acc));\n";
    s << "  }\n";
    s << "  for (; k < end; ++k) acc = " << rndOpen << "akg::op_add(" << tag << "::load(data[static_cast<long>(sorted[k]) * SLICE]), acc));\n";
    s << "  out0[c] = " << tag << "::store(acc);\n";
    s << "}\n";
  }

  LoweredKernel k;
  k.kernelName = g.name + "_kernel";
  k.source = s.str();
  k.family = KernelFamily::SegmentSum;
  k.grid[0] = static_cast<unsigned>(staged ? (segments + segsPerWave - 1) / segsPerWave : (chains + 255) / 256);
  k.block[0] = staged ? 64 : 256;
  const auto phase = [&](const char *suffix, int64_t grid, unsigned block) {
    KernelPhase ph;
    ph.kernelName = g.name + suffix;
    ph.grid[0] = static_cast<unsigned>(grid);
    ph.block[0] = block;
    k.earlierPhases.push_back(ph);
  };
  phase("_count", runs, 256);
  phase("_offsets", offsetsGrid(segments), 256);
  phase("_starts", 1, 1024);
  phase("_place", runs, 64);
  k.workspaceBytes = static_cast<uint64_t>(words) * 4;
  k.algorithmicBytes = lowering::countAlgorithmicBytes(g);
  k.shapeArgs = lowering::buildShapeArgs(g);
  std::ostringstream note;
  note << "segment_sum positions=" << positions << " segments=" << segments << " slice=" << slice << " grouped by segment: runs="
       << runs << " of " << runLength << " positions, 5 launches";
  k.scheduleNote = note.str();
  return k;
}

// Device code both launches of the bucketed schedule share: a stable counting sort of a chunk by key inside a workgroup.
const char *const kChunkSort = R"AKG(
// Stable counting sort of a chunk of NW x TILES x 64 items by key, inside a workgroup of NW wavefronts. Item (w, u, lane)
// - wavefront, tile, lane, in this order of significance - has key[u] (negative: the item takes no part); the function
// returns its place among the sorted items in slot[u]. First every wavefront ranks its own items: lanes of a tile with
// the same key find each other with one ballot per key bit and stand behind the wavefront's running counter of that
// key (its LDS accesses complete in program order, so the counters need no barrier between the tiles). Then the
// counters are summed over the wavefronts and the keys (each key's run starts at a multiple of ALIGN), and every item
// adds where the run of its key and wavefront starts. On return start[k] is where key k's run starts, len[k] its
// length; a barrier has been passed since they were written. cnt: NW * KEYS counters, scan: NW words.
template <int NW, int KEYS, int KEY_BITS, int TILES, int ALIGN>
__device__ inline void chunk_sort(const int (&key)[TILES], unsigned (&slot)[TILES], unsigned short *cnt, unsigned *start,
                                  unsigned *len, unsigned *scan) {
  constexpr int THREADS = NW * 64, PER = (KEYS + THREADS - 1) / THREADS;
  const int tid = static_cast<int>(threadIdx.x), lane = tid & 63, w = tid >> 6;
  for (int k = tid; k < NW * KEYS; k += THREADS) cnt[k] = 0;
  __syncthreads();
  unsigned short *mine = cnt + w * KEYS;
#pragma unroll
  for (int u = 0; u < TILES; ++u) {
    const int k = key[u] >= 0 ? key[u] : 0;
    const unsigned long long part = __ballot(key[u] >= 0);
    unsigned lo = static_cast<unsigned>(part), hi = static_cast<unsigned>(part >> 32);   // lanes with the same key
#pragma unroll
    for (int bit = 0; bit < KEY_BITS; ++bit) {
      const unsigned mine_bit = static_cast<unsigned>(__builtin_amdgcn_sbfe(k, bit, 1));   // 0 or all ones
      const unsigned long long with = __ballot(mine_bit != 0u);
      lo &= ~(static_cast<unsigned>(with) ^ mine_bit);
      hi &= ~(static_cast<unsigned>(with >> 32) ^ mine_bit);   // lanes whose bit equals mine
    }
    slot[u] = 0u;
    if (key[u] >= 0) {
      const unsigned before = mine[k];
      slot[u] = __builtin_amdgcn_mbcnt_hi(hi, __builtin_amdgcn_mbcnt_lo(lo, before));
      mine[k] = static_cast<unsigned short>(before + static_cast<unsigned>(__popc(lo) + __popc(hi)));   // (the same from every lane of the key)
    }
  }
  __syncthreads();
  unsigned total[PER], sum = 0u;
#pragma unroll
  for (int j = 0; j < PER; ++j) {
    const int k = tid * PER + j;
    unsigned before = 0u;
    if (k < KEYS) {
#pragma unroll
      for (int h = 0; h < NW; ++h) {
        const unsigned c = cnt[h * KEYS + k];
        cnt[h * KEYS + k] = static_cast<unsigned short>(before);
        before += c;
      }
      len[k] = before;
    }
    total[j] = (before + ALIGN - 1) / ALIGN * ALIGN;
    sum += total[j];
  }
  unsigned incl = sum;
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const unsigned o = __shfl_up(incl, d);
    if (lane >= d) incl += o;
  }
  if (lane == 63) scan[w] = incl;
  __syncthreads();
  unsigned at = incl - sum;
#pragma unroll
  for (int j = 0; j < NW; ++j) at += j < w ? scan[j] : 0u;
#pragma unroll
  for (int j = 0; j < PER; ++j) {
    const int k = tid * PER + j;
    if (k < KEYS) {
      start[k] = at;
#pragma unroll
      for (int h = 0; h < NW; ++h) cnt[h * KEYS + k] += static_cast<unsigned short>(at);
    }
    at += total[j];
  }
  __syncthreads();
#pragma unroll
  for (int u = 0; u < TILES; ++u) {
    if (key[u] >= 0) slot[u] += mine[key[u]];
  }
}
)AKG";

// Values of a list that are in flight (add_list). Integers: with 48 the compiler, free to add them in any order, moves the requests together
// and spills nine registers and more (us, int32 956289 x 1 into 14006 17.0 before there was add_list / 18.0 with 48 / 16.2 with 16). Sums that are rounded
// to 16 bits at every addition: an addition is longer, and a short list waits for requests it has no use for. us, 48 / 16: 65101 x 4 into 1536 9.7 / 9.0,
// 63114 x 2 into 1173 9.5 / 8.8, 579545 x 2 into 16024 15.0 / 14.2, 41 with fewer than 512 positions a segment 0.98 in the mean, none of them slower by 2 %;
// beyond, 4405314 x 4 into 901 96 / 104, 5035400 x 4 into 1282 89 / 94, 19 such 1.03.
int addBlock(const SegmentShapes &sh, const std::string &computeType, bool rounds) {
  return computeType == "float" && (!rounds || sh.positions >= 512 * sh.segments) ? 48 : 16;
}

// Device code of the launches that add lists out of LDS.
const char *const kAddList = R"AKG(
// acc, then list[0] .. list[n - 1] added to it one after the other. `list` begins at a multiple of 16 bytes; up to ADD_BLOCK values behind
// its end are read and not added. A float addition takes 4.4 cycles and LDS up to 230, so every value is requested 44 additions ahead and the
// order is given: left to itself the compiler requests values in front of the last two additions before them (13.7 cycles an addition).
template <typename T, typename Add>
__device__ inline T add_list(const T *list, int n, T acc, Add add) {
  static_assert(sizeof(T) == 4, "four values a request");
  typedef T quad_t __attribute__((ext_vector_type(4)));
  constexpr int BLOCK = ADD_BLOCK, QUADS = BLOCK / 4;
  const quad_t *quads = reinterpret_cast<const quad_t *>(list);
  quad_t q[QUADS];
#pragma unroll
  for (int i = 0; i < QUADS; ++i) q[i] = quads[i];
  int j = 0;
  for (; j + BLOCK <= n; j += BLOCK) {
#pragma unroll
    for (int i = 0; i < QUADS; ++i) {
#pragma unroll
      for (int u = 0; u < 4; ++u) acc = add(q[i][u], acc);
      q[i] = quads[j / 4 + QUADS + i];
      __builtin_amdgcn_sched_barrier(0);
    }
  }
#pragma unroll
  for (int h = 0; h < BLOCK; h += 8) {
    if (j + h < n) {
#pragma unroll
      for (int u = h; u < h + 8; ++u) {
        const T sum = add(q[u / 4][u & 3], acc);
        acc = j + u < n ? sum : acc;
      }
    }
  }
  return acc;
}
)AKG";

/**
 * Very many positions of short rows (at most 12 bytes): grouping by segment in one step writes every row to a place of
 * its own, a partial cache line each time (24.5 million 12-byte rows: 1.07 GB written for 0.29 GB of rows). Here the
 * positions are first grouped by BUCKET, a few neighbouring segments, and the last step to the segment happens in LDS:
 *
 *   <op>_count / _offsets / _starts   as above, with the bucket as the key and chunks of 4096 positions as the runs
 *   <op>_place    a workgroup sorts its chunk by bucket in LDS (chunk_sort above) and copies the sorted chunk out, one
 *                 16-byte entry per position {row, segment}: a bucket's entries of one chunk are contiguous, so the
 *                 stores fill whole sectors
 *   <op>_kernel   a workgroup per bucket walks the bucket's entries, 4096 per round: the same sort, by segment now,
 *                 puts the rows' columns into LDS lists per segment, and one lane per output element adds its list
 *
 * Both sorts are stable, so the order per output element is the position order and the result is the serial loop's,
 * bit for bit.
 */
LoweredKernel lowerSegmentBucketed(const OpGraph &g, const LoweringOptions &, const SegmentShapes &sh, int bucketBits) {
  using lowering::computeTypeName;
  using lowering::dtypeTag;
  const TensorValue &data = *sh.data, &ids = *sh.ids, &out = *sh.out;
  const int64_t positions = sh.positions, segments = sh.segments, slice = sh.slice;
  const std::string ct = computeTypeName(out.dtype), tag = dtypeTag(out.dtype), idTag = dtypeTag(ids.dtype);
  const bool narrow = out.dtype == DType::F16 || out.dtype == DType::BF16 || out.dtype == DType::I8 || out.dtype == DType::I16;
  const std::string rndOpen = narrow ? tag + "::rnd(" : std::string("(");
  const int elemBytes = static_cast<int>(dtypeSize(out.dtype));
  const int64_t rowWords = slice * elemBytes / 4;
  const int64_t perBucket = 1LL << bucketBits, buckets = (segments + perBucket - 1) / perBucket;
  const int64_t chunk = 4096, chunks = (positions + chunk - 1) / chunk;
  int keyBits = 1;
  while ((1LL << keyBits) < buckets) ++keyBits;
  // workspace, in 4-byte words
  const int64_t wHist = 0, wTotal = wHist + chunks * buckets, wStart = wTotal + buckets,
                wSorted = (wStart + buckets + 1 + 3) / 4 * 4;   // 16-byte aligned
  const int64_t words = wSorted + positions * 4;

  std::ostringstream s;
  s << "// Generated by the akg HIP lowering for gfx950. Op description: " << g.name << "\n";
  s << "// family: segment_sum (positions grouped by bucket of segments first), fusion class: " << operatorTemplateName(g.operatorTemplate) << "\n";
  s << "#include \"akg_rt.hpp\"\n\n";
  s << "namespace {\n";
  s << "constexpr int POSITIONS = " << positions << ", SEGMENTS = " << segments << ", BUCKET_BITS = " << bucketBits << ", KEYS = " << buckets
    << ", KEY_BITS = " << keyBits << ", RUNS = " << chunks << ", RUN = " << chunk << ";\n";
  s << "constexpr int ROW = " << slice << ", ROW_WORDS = " << rowWords << ", NW = 8, TILES = RUN / (64 * NW);\n";
  s << "constexpr long W_HIST = " << wHist << ", W_TOTAL = " << wTotal << ", W_START = " << wStart << ", W_SORTED = " << wSorted << ";\n";
  s << "using id_t = " << idTag << "::storage;\n";
  if (ids.dtype == DType::I64) {
    s << "__device__ inline int as_segment(long v) { return v < 0 || v >= SEGMENTS ? -1 : static_cast<int>(v); }\n";
  } else {
    s << "__device__ inline int as_segment(int v) { return v < 0 || v >= SEGMENTS ? -1 : v; }\n";
  }
  s << "__device__ inline int key_of(int segment) { return segment >> BUCKET_BITS; }\n";
  s << "typedef unsigned entry_t __attribute__((ext_vector_type(4)));   // x, y, z: the row's words, zero filled; w: segment\n";
  s << kChunkSort;
  s << "}  // namespace\n\n";
  std::ostringstream params;
  for (size_t i = 0; i < g.inputs.size(); ++i) {
    params << (i ? ", " : "") << "const " << dtypeTag(g.tensor(g.inputs[i]).dtype) << "::storage *__restrict__ in" << i;
  }
  params << ", " << tag << "::storage *__restrict__ out0, unsigned *__restrict__ akg_ws";
  const std::string idsName = "in" + std::to_string(ids.inputIndex), dataName = "in" + std::to_string(data.inputIndex);

  emitCountingLaunches(s, g.name, params.str(), idTag, idsName, chunks, buckets);

  // ---- place ----
  // Workgroups that run at the same time on one XCD (launch order: workgroup b runs on XCD b mod 8) take neighbouring
  // chunks, whose entries are neighbours in every bucket: the line two chunks share is completed in that XCD's L2.
  const int64_t perXcd = (chunks + 7) / 8;
  s << "extern \"C\" __global__ __launch_bounds__(512) void " << g.name << "_place(" << params.str() << ") {\n";
  s << "  __shared__ entry_t akg_stage[RUN];\n";
  s << "  __shared__ unsigned short akg_cnt[NW * KEYS];\n";
  s << "  __shared__ unsigned akg_start[KEYS], akg_len[KEYS], akg_scan[NW];\n";
  s << "  const int tid = static_cast<int>(threadIdx.x), lane = tid & 63, w = tid >> 6;\n";
  s << "  const int run = static_cast<int>(blockIdx.x & 7u) * " << perXcd << " + static_cast<int>(blockIdx.x >> 3);\n";
  s << "  if (run >= RUNS) return;   // (uniform)\n";
  s << "  const int p0 = run * RUN + w * (64 * TILES);\n";
  s << "  const unsigned *__restrict__ rows = reinterpret_cast<const unsigned *>(" << dataName << ");\n";
  s << "  int id[TILES], key[TILES];\n  unsigned row[TILES][ROW_WORDS], slot[TILES];\n";
  s << "#pragma unroll\n";
  s << "  for (int u = 0; u < TILES; ++u) {\n";
  s << "    const int p = p0 + u * 64 + lane;\n";
  s << "    id[u] = p < POSITIONS ? as_segment(" << idTag << "::load(" << idsName << "[p])) : -1;\n";
  s << "    key[u] = id[u] >= 0 ? key_of(id[u]) : -1;\n";
  s << "#pragma unroll\n";
  s << "    for (int c = 0; c < ROW_WORDS; ++c) row[u][c] = p < POSITIONS ? rows[static_cast<long>(p) * ROW_WORDS + c] : 0u;\n";
  s << "  }\n";
  s << "  chunk_sort<NW, KEYS, KEY_BITS, TILES, 1>(key, slot, akg_cnt, akg_start, akg_len, akg_scan);\n";
  s << "#pragma unroll\n";
  s << "  for (int u = 0; u < TILES; ++u) {\n";
  s << "    if (id[u] >= 0) {\n";
  s << "      entry_t e = {0u, 0u, 0u, static_cast<unsigned>(id[u])};\n";
  s << "      e.x = row[u][0];\n";
  if (rowWords > 1) s << "      e.y = row[u][1];\n";
  if (rowWords > 2) s << "      e.z = row[u][2];\n";
  s << "      akg_stage[slot[u]] = e;\n";
  s << "    }\n";
  s << "  }\n";
  s << "  // where the bucket's entries of this chunk go, less where they are in the sorted chunk\n";
  s << "  unsigned valid = 0u;\n";
  s << "  for (int k = tid; k < KEYS; k += 64 * NW) {\n";
  s << "    if (k == KEYS - 1) akg_scan[0] = akg_start[k] + akg_len[k];\n";
  s << "    akg_start[k] = akg_ws[W_START + k] + akg_ws[W_HIST + static_cast<long>(run) * KEYS + k] - akg_start[k];\n";
  s << "  }\n";
  s << "  __syncthreads();\n";
  s << "  valid = akg_scan[0];\n";
  s << "  entry_t *__restrict__ placed = reinterpret_cast<entry_t *>(akg_ws + W_SORTED);\n";
  s << "  for (unsigned i = tid; i < valid; i += 64 * NW) {\n";
  s << "    const entry_t e = akg_stage[i];\n";
  s << "    placed[akg_start[key_of(static_cast<int>(e.w))] + i] = e;\n";
  s << "  }\n";
  s << "}\n\n";

  // ---- chains ----
  const int64_t chains = perBucket * slice, chainsPerWave = (chains + 7) / 8;
  s << "extern \"C\" __global__ __launch_bounds__(512) void " << g.name << "_kernel(" << params.str() << ") {\n";
  s << "  constexpr int S = 1 << BUCKET_BITS, PLANE = RUN + 4 * S + 8, CHAINS = " << chains << ", PER_WAVE = " << chainsPerWave << ";\n";
  s << "  __shared__ __attribute__((aligned(16))) " << ct << " akg_plane[ROW][PLANE];   // column c of the rows, lists per segment\n";
  s << "  __shared__ unsigned short akg_cnt[NW * S];\n";
  s << "  __shared__ unsigned akg_start[S], akg_len[S], akg_scan[NW];\n";
  s << "  const int tid = static_cast<int>(threadIdx.x), lane = tid & 63, w = tid >> 6, bucket = static_cast<int>(blockIdx.x);\n";
  s << "  const entry_t *__restrict__ placed = reinterpret_cast<const entry_t *>(akg_ws + W_SORTED);\n";
  s << "  const unsigned from = akg_ws[W_START + bucket], upto = akg_ws[W_START + bucket + 1];\n";
  s << "  constexpr unsigned LAST = POSITIONS - 1;\n";
  s << "  // the output element of this lane, if it has one: wavefront w adds chains w * PER_WAVE ...\n";
  s << "  const int chain = w * PER_WAVE + lane;\n";
  s << "  const bool has = lane < PER_WAVE && chain < CHAINS;\n";
  s << "  const int cs = has ? chain / ROW : 0, cc = has ? chain - cs * ROW : 0;\n";
  s << "  union cell_t { entry_t q; " << tag << "::storage v[16 / sizeof(" << tag << "::storage)]; };\n";
  s << "  typedef " << ct << " quad_t __attribute__((ext_vector_type(4)));\n";
  s << "  " << ct << " acc = " << lowering::literalFor(out.dtype, 0.0) << ";\n";
  s << "  for (unsigned r = from; r < upto; r += RUN) {\n";
  s << "    cell_t cur[TILES];\n";
  s << "    int key[TILES];\n";
  s << "    unsigned slot[TILES];\n";
  s << "    // (every load is issued, the address clamped to the workspace's last entry: no branch between the loads)\n";
  s << "#pragma unroll\n";
  s << "    for (int u = 0; u < TILES; ++u) {\n";
  s << "      const unsigned k = r + (w * TILES + u) * 64 + lane;\n";
  s << "      cur[u].q = __builtin_nontemporal_load(placed + (k < LAST ? k : LAST));\n";
  s << "    }\n";
  s << "#pragma unroll\n";
  s << "    for (int u = 0; u < TILES; ++u) {\n";
  s << "      const unsigned k = r + (w * TILES + u) * 64 + lane;\n";
  s << "      key[u] = k < upto ? static_cast<int>(cur[u].q.w) & (S - 1) : -1;\n";
  s << "    }\n";
  s << "    chunk_sort<NW, S, BUCKET_BITS, TILES, 4>(key, slot, akg_cnt, akg_start, akg_len, akg_scan);\n";
  s << "#pragma unroll\n";
  s << "    for (int u = 0; u < TILES; ++u) {\n";
  s << "      if (key[u] >= 0) {\n";
  s << "#pragma unroll\n";
  s << "        for (int c = 0; c < ROW; ++c) akg_plane[c][slot[u]] = " << tag << "::load(cur[u].v[c]);\n";
  s << "      }\n";
  s << "    }\n";
  s << "    __syncthreads();\n";
  s << "    if (has) {\n";
  s << "      const int n = static_cast<int>(akg_len[cs]);\n";
  s << "      const quad_t *__restrict__ list = reinterpret_cast<const quad_t *>(&akg_plane[cc][akg_start[cs]]);   // (a multiple of 4)\n";
  s << "      int j = 0;\n";
  s << "      for (; j + 8 <= n; j += 8) {\n";
  s << "        const quad_t a = list[j / 4], b = list[j / 4 + 1];\n";
  s << "#pragma unroll\n";
  s << "        for (int u = 0; u < 4; ++u) acc = " << rndOpen << "akg::op_add(a[u], acc));\n";
  s << "#pragma unroll\n";
  s << "        for (int u = 0; u < 4; ++u) acc = " << rndOpen << "akg::op_add(b[u], acc));\n";
  s << "      }\n";
  s << "      if (j < n) {   // (what lies behind the list's end is read, inside the plane, and not added)\n";
  s << "        const quad_t a = list[j / 4], b = list[j / 4 + 1];\n";
  s << "#pragma unroll\n";
  s << "        for (int u = 0; u < 8; ++u) {\n";
  s << "          const " << ct << " sum = " << rndOpen << "akg::op_add(u < 4 ? a[u & 3] : b[u & 3], acc));\n";
  s << "          acc = j + u < n ? sum : acc;\n";
  s << "        }\n";
  s << "      }\n";
  s << "    }\n";
  s << "    __syncthreads();\n";
  s << "  }\n";
  s << "  if (has && bucket * S + cs < SEGMENTS) out0[static_cast<long>(bucket * S + cs) * ROW + cc] = " << tag << "::store(acc);\n";
  s << "}\n";

  LoweredKernel k;
  k.kernelName = g.name + "_kernel";
  k.source = s.str();
  k.family = KernelFamily::SegmentSum;
  k.grid[0] = static_cast<unsigned>(buckets);
  k.block[0] = 512;
  const auto phase = [&](const char *suffix, int64_t grid, unsigned block) {
    KernelPhase ph;
    ph.kernelName = g.name + suffix;
    ph.grid[0] = static_cast<unsigned>(grid);
    ph.block[0] = block;
    k.earlierPhases.push_back(ph);
  };
  phase("_count", chunks, 256);
  phase("_offsets", offsetsGrid(buckets), 256);
  phase("_starts", 1, 1024);
  phase("_place", perXcd * 8, 512);
  k.workspaceBytes = static_cast<uint64_t>(words) * 4;
  k.algorithmicBytes = lowering::countAlgorithmicBytes(g);
  k.shapeArgs = lowering::buildShapeArgs(g);
  std::ostringstream note;
  note << "segment_sum positions=" << positions << " segments=" << segments << " slice=" << slice << " grouped by bucket of " << perBucket
       << " segments: " << buckets << " buckets, chunks=" << chunks << " of " << chunk << " positions, 5 launches";
  k.scheduleNote = note.str();
  return k;
}

// Device code of the chunked schedule: the rank of every item of a chunk among the items of its key.
const char *const kChunkRank = R"AKG(
// Stable counting sort of a chunk of NW x TILES x 64 items by key, as chunk_sort above, for many keys: the lanes of a tile
// with the same key find each other through a mask of lanes per key and wavefront in LDS (or the own bit in, read the
// mask, put it back to zero: three LDS accesses of the wavefront, which complete in program order) instead of one ballot
// per key bit - 40 vector instructions of a tile's 120 and, beside the loads of the next chunk, most of what the
// launch's time was. An or gives the same mask in any order. The key is the low half of key[u]. On return start[k] is where key k's run starts, start[KEYS]
// the number of items that take part. masks: NW * KEYS, zero on return; cnt: NW * KEYS; start: KEYS + 1; scan: NW words.
template <int NW, int KEYS, int TILES>
__device__ inline void chunk_rank(const int (&key)[TILES], unsigned (&slot)[TILES], unsigned long long *masks, unsigned short *cnt,
                                  unsigned short *start, unsigned *scan) {
  constexpr int THREADS = NW * 64, PER = (KEYS + THREADS - 1) / THREADS;
  const int tid = static_cast<int>(threadIdx.x), lane = tid & 63, w = tid >> 6;
  for (int k = tid; k < NW * KEYS; k += THREADS) {
    masks[k] = 0ull;
    cnt[k] = 0;
  }
  __syncthreads();
  const unsigned long long bit = 1ull << lane;
  unsigned long long *lanes = masks + w * KEYS;
  unsigned short *mine = cnt + w * KEYS;
#pragma unroll
  for (int u = 0; u < TILES; ++u) {
    slot[u] = 0u;
    if (key[u] >= 0) {
      const int k = key[u] & 0xffff;
      __hip_atomic_fetch_or(lanes + k, bit, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
      __builtin_amdgcn_wave_barrier();
      const unsigned long long same = __hip_atomic_load(lanes + k, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
      const unsigned before = mine[k];
      __builtin_amdgcn_wave_barrier();
      __hip_atomic_store(lanes + k, 0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
      slot[u] = __builtin_amdgcn_mbcnt_hi(static_cast<unsigned>(same >> 32), __builtin_amdgcn_mbcnt_lo(static_cast<unsigned>(same), before));
      mine[k] = static_cast<unsigned short>(before + static_cast<unsigned>(__popcll(same)));   // (the same from every lane of the key)
    }
    __builtin_amdgcn_wave_barrier();
  }
  __syncthreads();
  unsigned total[PER], sum = 0u;
#pragma unroll
  for (int j = 0; j < PER; ++j) {
    const int k = tid * PER + j;
    unsigned before = 0u;
    if (k < KEYS) {
#pragma unroll
      for (int h = 0; h < NW; ++h) {
        const unsigned c = cnt[h * KEYS + k];
        cnt[h * KEYS + k] = static_cast<unsigned short>(before);
        before += c;
      }
    }
    total[j] = before;
    sum += before;
  }
  unsigned incl = sum;
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const unsigned o = __shfl_up(incl, d);
    if (lane >= d) incl += o;
  }
  if (lane == 63) scan[w] = incl;
  __syncthreads();
  unsigned at = incl - sum;
#pragma unroll
  for (int j = 0; j < NW; ++j) at += j < w ? scan[j] : 0u;
#pragma unroll
  for (int j = 0; j < PER; ++j) {
    const int k = tid * PER + j;
    if (k < KEYS) {
      start[k] = static_cast<unsigned short>(at);
#pragma unroll
      for (int h = 0; h < NW; ++h) cnt[h * KEYS + k] += static_cast<unsigned short>(at);
    }
    at += total[j];
  }
  if (tid == THREADS - 1) start[KEYS] = static_cast<unsigned short>(at);
  __syncthreads();
#pragma unroll
  for (int u = 0; u < TILES; ++u) {
    if (key[u] >= 0) slot[u] += mine[key[u] & 0xffff];
  }
}
)AKG";

// The chunked schedule's sizes: buckets of perBucket segments, chunks of 512 * tiles positions.
struct ChunkedPlan {
  bool possible = false;
  int tiles = 8;
  int64_t perBucket = 1, buckets = 0, chunk = 0, chunks = 0, pitch = 0, rowWords = 0;
  int64_t wSegs = 0, wTable = 0, words = 0;   // workspace, in 4-byte words: rows, then segments within the bucket, then starts
};

ChunkedPlan planChunked(const SegmentShapes &sh, const LoweringOptions &options) {
  ChunkedPlan p;
  const int64_t rowBytes = sh.slice * static_cast<int64_t>(dtypeSize(sh.out->dtype));
  const bool wide = sh.out->dtype == DType::I64 || sh.out->dtype == DType::F64;
  if (wide || rowBytes % 4 != 0 || rowBytes > 16 || sh.slice > 4) return p;
  p.rowWords = rowBytes / 4;
  // two workgroups per CU in the last launch, which has one per bucket, where there are that many segments
  const int64_t most = options.split > 0 ? std::min(options.split, 768) : 2LL * options.computeUnits;
  p.perBucket = (sh.segments + most - 1) / most;
  if (p.perBucket > 64) return p;
  p.buckets = (sh.segments + p.perBucket - 1) / p.perBucket;
  p.tiles = options.chunks == 1 || options.chunks == 2 || options.chunks == 4 || options.chunks == 8 ? options.chunks : 8;
  // Chunks: small ones while there are few, for workgroups; larger ones then, for longer runs. us with chunks of 512 / 1024 /
  // 2048 / 4096 positions: 35304 x 1 into 1131 8.4 / 9.0 / 10.3 / 11.4, 86700 x 3 into 8856 11.0 / 10.0 / 12.0 / 13.6, 138073 x 1
  // into 998 14.1 / 12.3 / 11.6 / 12.6, 300000 x 3 into 5000 22.7 / 18.6 / 14.4 / 16.0, 1536784 x 4 into 12654 91 / 56 / 42 / 34.
  // (Rows of 16 bytes in chunks of 4096 spill 13 registers of <op>_place. Chunks of 2048 do not and are no faster: 12.5 million x 4 into
  // 2216 224.9 us, 224.7 with 4096, 20 million x 4 into 16384 335 and 314, 2 million x 4 into 32768 48 and 42.)
  if (options.chunks == 0) p.tiles = sh.positions < (1 << 16) ? 1 : sh.positions < (1 << 17) ? 2 : sh.positions < (1 << 19) ? 4 : 8;
  p.chunk = 512LL * p.tiles;
  p.chunks = (sh.positions + p.chunk - 1) / p.chunk;
  if (p.chunks * p.chunk >= (1LL << 31)) return p;
  p.pitch = (p.buckets + 1 + 7) / 8 * 8;
  p.wSegs = p.chunks * p.chunk * p.rowWords;
  p.wTable = p.wSegs + p.chunks * p.chunk / 4;
  p.words = p.wTable + p.chunks * p.pitch / 2;
  p.possible = true;
  return p;
}

/**
 * Short rows (4, 8, 12 or 16 bytes): chunks of positions sorted by bucket of segments where they lie. Two launches:
 *
 *   <op>_place    a workgroup takes chunks in turn, the loads of the next one in flight while it sorts this one by bucket
 *                 in LDS (chunk_rank above) and writes it out in one piece: the rows, one byte each for the segment within
 *                 the bucket, and a table of where every bucket's run starts. No counts are needed in front of it.
 *   <op>_kernel   a workgroup per bucket walks the runs of its bucket, chunk by chunk, as many per round as fit: the
 *                 runs' lengths are summed up, every entry is fetched from its run (neighbouring buckets run on one XCD
 *                 and share the lines in which a run ends and the next one begins), sorted by segment (chunk_sort) into
 *                 LDS lists, and one lane per output element adds its list.
 *
 * Both sorts are stable and chunks are taken in order, so every output element is the serial loop's chain of additions
 * over its positions, bit for bit.
 */
LoweredKernel lowerSegmentChunked(const OpGraph &g, const LoweringOptions &options, const SegmentShapes &sh, const ChunkedPlan &plan) {
  using lowering::computeTypeName;
  using lowering::dtypeTag;
  const TensorValue &data = *sh.data, &ids = *sh.ids, &out = *sh.out;
  const std::string ct = computeTypeName(out.dtype), tag = dtypeTag(out.dtype), idTag = dtypeTag(ids.dtype);
  const bool narrow = out.dtype == DType::F16 || out.dtype == DType::BF16 || out.dtype == DType::I8 || out.dtype == DType::I16;
  const std::string rndOpen = narrow ? tag + "::rnd(" : std::string("(");
  // Rounds of the last launch: 4096 entries on eight wavefronts; few entries per bucket: 2048 on four, or where chunks are 512 that many
  // on two, if those have a lane for every output element of the bucket (of which there are at most 256). A frequent segment takes as
  // many rounds as its positions: us, 100000 x 4 into 5000, rounds of 1024 / 2048 / 4096: ids as frequent as words 187 / 128 / 111 (136 by
  // segment), uniform ones 10.1 / 10.4 / 11.4; chunks of 512, 60000 x 4 into 16000 uniform, rounds of 512 / 2048: 8.4 / 9.2.
  const bool small = sh.positions / plan.buckets < 1024 && plan.tiles <= 4;
  const int64_t perBucket = plan.perBucket, chains = perBucket * sh.slice;
  const int nw = small ? (plan.tiles == 1 && chains <= 128 ? 2 : 4) : 8, tiles = small && plan.tiles == 1 ? static_cast<int>(plan.chunk) / (nw * 64) : 8;
  // (at least sixteen chains a wavefront: an addition is an instruction of the whole wavefront however few lanes add)
  const int64_t chainsPerWave = std::max<int64_t>(16, (chains + nw - 1) / nw);
  int keyBits = 1;
  while ((1LL << keyBits) < perBucket) ++keyBits;
  std::ostringstream s;
  s << "// Generated by the akg HIP lowering for gfx950. Op description: " << g.name << "\n";
  s << "// family: segment_sum (positions grouped by bucket of segments, chunk by chunk), fusion class: "
    << operatorTemplateName(g.operatorTemplate) << "\n";
  s << "#include \"akg_rt.hpp\"\n\n";
  s << "namespace {\n";
  s << "constexpr int POSITIONS = " << sh.positions << ", SEGMENTS = " << sh.segments << ", S = " << perBucket << ", KEYS = " << plan.buckets
    << ", CHUNKS = " << plan.chunks << ", PITCH = " << plan.pitch << ";\n";
  s << "constexpr int ROW = " << sh.slice << ", ROW_WORDS = " << plan.rowWords << ", NW = 8, TILES = " << plan.tiles << ", CHUNK = NW * TILES * 64;\n";
  s << "constexpr long W_SEGS = " << plan.wSegs << ", W_TABLE = " << plan.wTable << ";\n";
  if (ids.dtype == DType::I64) {
    s << "__device__ inline int as_segment(long v) { return v < 0 || v >= SEGMENTS ? -1 : static_cast<int>(v); }\n";
  } else {
    s << "__device__ inline int as_segment(int v) { return v < 0 || v >= SEGMENTS ? -1 : v; }\n";
  }
  s << "struct __attribute__((aligned(4))) row_t { unsigned w[ROW_WORDS]; };\n";
  s << "typedef unsigned quad_words __attribute__((ext_vector_type(4)));\n";
  s << "constexpr int ADD_BLOCK = " << addBlock(sh, ct, narrow) << ";\n" << kChunkSort << kAddList << kChunkRank;
  s << "}  // namespace\n\n";
  std::ostringstream params;
  for (size_t i = 0; i < g.inputs.size(); ++i) {
    params << (i ? ", " : "") << "const " << dtypeTag(g.tensor(g.inputs[i]).dtype) << "::storage *__restrict__ in" << i;
  }
  params << ", " << tag << "::storage *__restrict__ out0, unsigned *__restrict__ akg_ws";
  const std::string idsName = "in" + std::to_string(ids.inputIndex), dataName = "in" + std::to_string(data.inputIndex);

  // ---- place ----
  const int64_t placeGrid = std::min<int64_t>(plan.chunks, 2LL * options.computeUnits);
  s << "extern \"C\" __global__ __launch_bounds__(512, 4) void " << g.name << "_place(" << params.str() << ") {\n";
  s << "  // the lane masks of the ranking, then (a barrier later) the sorted rows and their segments\n";
  s << "  constexpr int MASK_BYTES = NW * KEYS * 8, STAGE_BYTES = CHUNK * (ROW_WORDS * 4 + 1);\n";
  s << "  __shared__ __attribute__((aligned(16))) unsigned char akg_stage[MASK_BYTES > STAGE_BYTES ? MASK_BYTES : STAGE_BYTES];\n";
  s << "  __shared__ unsigned short akg_cnt[NW * KEYS];\n";
  s << "  __shared__ __attribute__((aligned(16))) unsigned short akg_start[PITCH];\n";
  s << "  __shared__ unsigned akg_scan[NW];\n";
  s << "  const int tid = static_cast<int>(threadIdx.x), lane = tid & 63, w = tid >> 6;\n";
  s << "  const row_t *__restrict__ rows = reinterpret_cast<const row_t *>(" << dataName << ");\n";
  s << "  int next_id[TILES];\n  unsigned next_row[TILES][ROW_WORDS];\n";
  s << "  const auto fetch = [&](int chunk) {   // (positions behind the last one read the last one's row and take no part)\n";
  s << "#pragma unroll\n";
  s << "    for (int u = 0; u < TILES; ++u) {\n";
  s << "      const int p = chunk * CHUNK + (w * TILES + u) * 64 + lane, at = p < POSITIONS ? p : POSITIONS - 1;\n";
  s << "      const int id = as_segment(" << idTag << "::load(" << idsName << "[at]));\n";
  s << "      next_id[u] = p < POSITIONS ? id : -1;\n";
  s << "      const row_t r = rows[at];\n";
  s << "#pragma unroll\n";
  s << "      for (int c = 0; c < ROW_WORDS; ++c) next_row[u][c] = r.w[c];\n";
  s << "    }\n  };\n";
  s << "  fetch(static_cast<int>(blockIdx.x));\n";
  s << "  for (int chunk = static_cast<int>(blockIdx.x); chunk < CHUNKS; chunk += static_cast<int>(gridDim.x)) {\n";
  s << "    int key[TILES];\n    unsigned row[TILES][ROW_WORDS], slot[TILES];\n";
  s << "#pragma unroll\n";
  s << "    for (int u = 0; u < TILES; ++u) {\n";
  s << "      const unsigned bucket = static_cast<unsigned>(next_id[u]) / S;\n";
  s << "      // the bucket, and the segment within it in the upper half\n";
  s << "      key[u] = next_id[u] >= 0 ? static_cast<int>(bucket | (static_cast<unsigned>(next_id[u]) - bucket * S) << 16) : -1;\n";
  s << "#pragma unroll\n";
  s << "      for (int c = 0; c < ROW_WORDS; ++c) row[u][c] = next_row[u][c];\n";
  s << "    }\n";
  s << "    if (chunk + static_cast<int>(gridDim.x) < CHUNKS) fetch(chunk + static_cast<int>(gridDim.x));   // (uniform)\n";
  s << "    chunk_rank<NW, KEYS, TILES>(key, slot, reinterpret_cast<unsigned long long *>(akg_stage), akg_cnt, akg_start, akg_scan);\n";
  s << "    unsigned char *stage_segs = akg_stage + CHUNK * ROW_WORDS * 4;\n";
  s << "#pragma unroll\n";
  s << "    for (int u = 0; u < TILES; ++u) {\n";
  s << "      if (key[u] >= 0) {\n";
  s << "        unsigned *to = reinterpret_cast<unsigned *>(akg_stage) + slot[u] * ROW_WORDS;\n";
  s << "#pragma unroll\n";
  s << "        for (int c = 0; c < ROW_WORDS; ++c) to[c] = row[u][c];\n";
  s << "        stage_segs[slot[u]] = static_cast<unsigned char>(key[u] >> 16);\n";
  s << "      }\n    }\n";
  s << "    __syncthreads();\n";
  s << "    // whole 16-byte pieces; what they hold behind the last item is never looked at\n";
  s << "    const int valid = akg_start[KEYS];\n";
  s << "    const quad_words *staged = reinterpret_cast<const quad_words *>(akg_stage);\n";
  s << "    quad_words *to = reinterpret_cast<quad_words *>(akg_ws + static_cast<long>(chunk) * (CHUNK * ROW_WORDS));\n";
  s << "    for (int i = tid; i < (valid * ROW_WORDS + 3) / 4; i += NW * 64) to[i] = staged[i];\n";
  s << "    to = reinterpret_cast<quad_words *>(akg_ws + W_SEGS + static_cast<long>(chunk) * (CHUNK / 4));\n";
  s << "    for (int i = tid; i < (valid + 15) / 16; i += NW * 64) to[i] = reinterpret_cast<const quad_words *>(stage_segs)[i];\n";
  s << "    to = reinterpret_cast<quad_words *>(akg_ws + W_TABLE + static_cast<long>(chunk) * (PITCH / 2));\n";
  s << "    for (int i = tid; i < PITCH / 8; i += NW * 64) to[i] = reinterpret_cast<const quad_words *>(akg_start)[i];\n";
  s << "    __syncthreads();\n";
  s << "  }\n}\n\n";

  // ---- chains ----
  s << "extern \"C\" __global__ __launch_bounds__(" << nw * 64 << (small ? "" : ", 4") << ") void " << g.name << "_kernel(" << params.str() << ") {\n";
  s << "  constexpr int W = " << nw << ", T = " << tiles << ", CAP = W * T * 64, PLANE = CAP + 4 * S, CHAINS = " << chains
    << ", PER_WAVE = " << chainsPerWave << ";\n";
  s << "  static_assert(CAP >= CHUNK, \"a chunk's run of one bucket fits a round\");\n";
  s << "  static_assert(PER_WAVE <= 64 && W * PER_WAVE >= CHAINS, \"a lane for every output element\");\n";
  s << "  // a round's entries: whose run each is, and where entry k of the round is less k for every run\n";
  s << "  __shared__ unsigned short akg_run[CAP];\n  __shared__ unsigned akg_base[W * 64];\n";
  s << "  // column c of a round's rows from c * PLANE on, lists per segment; what add_list reads behind the last one\n";
  s << "  __shared__ __attribute__((aligned(16))) " << ct << " akg_plane[ROW * PLANE + ADD_BLOCK];\n";
  s << "  __shared__ unsigned short akg_cnt[W * S];\n";
  s << "  __shared__ unsigned akg_start[S], akg_len[S], akg_scan[W], akg_sums[W], akg_taken[W], akg_total[W];\n";
  s << "  const int tid = static_cast<int>(threadIdx.x), lane = tid & 63, w = tid >> 6;\n";
  s << "  const int bucket = akg::xcd_contiguous_id(static_cast<int>(blockIdx.x), KEYS);\n";
  s << "  const row_t *__restrict__ rows = reinterpret_cast<const row_t *>(akg_ws);\n";
  s << "  const unsigned char *__restrict__ segs = reinterpret_cast<const unsigned char *>(akg_ws + W_SEGS);\n";
  s << "  const unsigned short *__restrict__ table = reinterpret_cast<const unsigned short *>(akg_ws + W_TABLE) + bucket;\n";
  s << "  // the output element of this lane, if it has one: wavefront w adds chains w * PER_WAVE ...\n";
  s << "  const int chain = w * PER_WAVE + lane;\n";
  s << "  const bool has = lane < PER_WAVE && chain < CHAINS;\n";
  s << "  const int cs = has ? chain / ROW : 0, cc = has ? chain - cs * ROW : 0;\n";
  s << "  union cell_t { row_t r; " << tag << "::storage v[ROW_WORDS * 4 / sizeof(" << tag << "::storage)]; };\n";
  s << "  " << ct << " acc = " << lowering::literalFor(out.dtype, 0.0) << ";\n";
  s << "  unsigned first = 0u, behind = 0u;   // this thread's run of the round: entries first .. behind - 1 of its chunk\n";
  s << "  const auto look_up = [&](int chunk) {\n";
  s << "    const unsigned short *t = table + static_cast<long>(chunk < CHUNKS ? chunk : CHUNKS - 1) * PITCH;\n";
  s << "    first = t[0];\n    behind = t[1];\n";
  s << "  };\n";
  s << "  look_up(tid);\n";
  s << "  cell_t cur[T];\n  int segment[T];\n  unsigned total = 0u;   // the round on its way: its entries as they are, how many\n";
  s << "  int chunk0 = 0;\n";
  s << "  const auto next_round = [&]() {\n";
  s << "    const int chunk = chunk0 + tid;\n";
  s << "    const unsigned len = chunk < CHUNKS ? behind - first : 0u;\n";
  s << "    const unsigned at = static_cast<unsigned>(chunk) * CHUNK + first;\n";
  s << "    unsigned incl = len;\n";
  s << "#pragma unroll\n";
  s << "    for (int d = 1; d < 64; d <<= 1) {\n";
  s << "      const unsigned o = __shfl_up(incl, d);\n";
  s << "      if (lane >= d) incl += o;\n";
  s << "    }\n";
  s << "    if (lane == 63) akg_sums[w] = incl;\n";
  s << "    __syncthreads();\n";
  s << "#pragma unroll\n";
  s << "    for (int j = 0; j < W; ++j) incl += j < w ? akg_sums[j] : 0u;\n";
  s << "    // the chunks whose runs fit the round: those in front of the first one that does not (the first one always does)\n";
  s << "    const bool fits = chunk < CHUNKS && incl <= static_cast<unsigned>(CAP);\n";
  s << "    const int fitting = __popcll(__ballot(fits));\n";
  s << "    if (lane == (fitting > 0 ? fitting - 1 : 0)) {\n";
  s << "      akg_taken[w] = static_cast<unsigned>(fitting);\n";
  s << "      akg_total[w] = fitting > 0 ? incl : 0u;\n";
  s << "    }\n";
  s << "    // every run's entries, one after the other; runs of more than 32 by the whole wavefront\n";
  s << "    unsigned long long longer = __ballot(fits && len > 32u);\n";
  s << "    akg_base[tid] = at - (incl - len);\n";
  s << "    if (fits && len <= 32u) {\n";
  s << "      for (unsigned i = 0; i < len; ++i) akg_run[incl - len + i] = static_cast<unsigned short>(tid);\n";
  s << "    }\n";
  s << "    while (longer) {\n";
  s << "      const int b = __builtin_ctzll(longer);\n";
  s << "      longer &= longer - 1;\n";
  s << "      const unsigned n = __builtin_amdgcn_readlane(len, b), to = __builtin_amdgcn_readlane(incl, b) - n;\n";
  s << "      for (unsigned i = lane; i < n; i += 64) akg_run[to + i] = static_cast<unsigned short>(w * 64 + b);\n";
  s << "    }\n";
  s << "    __syncthreads();\n";
  s << "    int taken = 0;\n    total = 0u;\n";
  s << "#pragma unroll\n";
  s << "    for (int j = 0; j < W; ++j) {\n";
  s << "      taken += static_cast<int>(akg_taken[j]);\n";
  s << "      total = akg_total[j] > total ? akg_total[j] : total;\n";
  s << "    }\n";
  s << "    chunk0 += taken;\n";
  s << "    look_up(chunk0 + tid);   // (the next round's runs)\n";
  s << "  };\n";
  s << "  const auto fetch_round = [&]() {\n";
  s << "#pragma unroll\n";
  s << "    for (int u = 0; u < T; ++u) {\n";
  s << "      const unsigned k = (w * T + u) * 64 + lane;\n";
  s << "      const unsigned from = k < total ? akg_base[akg_run[k]] + k : 0u;   // (the workspace's first row where there is no entry)\n";
  s << "      cur[u].r = rows[from];\n";
  s << "      segment[u] = segs[from];\n";
  s << "    }\n";
  s << "  };\n";
  s << "  next_round();\n  fetch_round();\n";
  s << "  for (;;) {\n";
  s << "    int key[T];\n    unsigned slot[T];\n";
  s << "#pragma unroll\n";
  s << "    for (int u = 0; u < T; ++u) key[u] = static_cast<unsigned>((w * T + u) * 64 + lane) < total ? segment[u] : -1;\n";
  if (perBucket == 1) {   // (nothing to sort)
    s << "#pragma unroll\n";
    s << "    for (int u = 0; u < T; ++u) slot[u] = static_cast<unsigned>((w * T + u) * 64 + lane);\n";
    s << "    if (tid == 0) {\n      akg_start[0] = 0u;\n      akg_len[0] = total;\n    }\n";
  } else {
    s << "    chunk_sort<W, S, " << keyBits << ", T, 4>(key, slot, akg_cnt, akg_start, akg_len, akg_scan);\n";
  }
  s << "#pragma unroll\n";
  s << "    for (int u = 0; u < T; ++u) {\n";
  s << "      if (key[u] >= 0) {\n";
  s << "#pragma unroll\n";
  s << "        for (int c = 0; c < ROW; ++c) akg_plane[c * PLANE + slot[u]] = " << tag << "::load(cur[u].v[c]);\n";
  s << "      }\n";
  s << "    }\n";
  s << "    __syncthreads();\n";
  s << "    // The next round's entries are requested while this one's are added up, by the wavefronts that add behind their additions: requests\n";
  s << "    // wait for room in the CU's 32 KiB of lines on their way, and a round ends with its longest list.\n";
  s << "    const bool more = chunk0 < CHUNKS;   // (uniform)\n";
  s << "    if (more) next_round();\n";
  s << "    if (has) {\n";
  s << "      __builtin_amdgcn_s_setprio(3);\n";
  s << "      acc = add_list(akg_plane + cc * PLANE + akg_start[cs], static_cast<int>(akg_len[cs]), acc, [](" << ct << " v, " << ct << " sum) { return " << rndOpen
    << "akg::op_add(v, sum)); });\n";
  s << "      __builtin_amdgcn_s_setprio(0);\n";
  s << "    }\n";
  s << "    if (!more) break;\n";
  s << "    fetch_round();\n";
  s << "    __syncthreads();\n";
  s << "  }\n";
  s << "  if (has && bucket * S + cs < SEGMENTS) out0[static_cast<long>(bucket * S + cs) * ROW + cc] = " << tag << "::store(acc);\n";
  s << "}\n";

  LoweredKernel k;
  k.kernelName = g.name + "_kernel";
  k.source = s.str();
  k.family = KernelFamily::SegmentSum;
  k.grid[0] = static_cast<unsigned>(plan.buckets);
  k.block[0] = static_cast<unsigned>(nw * 64);
  KernelPhase place;
  place.kernelName = g.name + "_place";
  place.grid[0] = static_cast<unsigned>(placeGrid);
  place.block[0] = 512;
  k.earlierPhases.push_back(place);
  k.workspaceBytes = static_cast<uint64_t>(plan.words) * 4;
  k.algorithmicBytes = lowering::countAlgorithmicBytes(g);
  k.shapeArgs = lowering::buildShapeArgs(g);
  std::ostringstream note;
  note << "segment_sum positions=" << sh.positions << " segments=" << sh.segments << " slice=" << sh.slice << " chunks=" << plan.chunks << " of "
       << plan.chunk << " positions grouped by bucket of " << perBucket << " segments where they lie: " << plan.buckets << " buckets, 2 launches";
  k.scheduleNote = note.str();
  return k;
}

// Sizes of the schedule by records.
struct RecordPlan {
  bool possible = false;
  int64_t chunks = 0, stride = 0, pitch = 0, wTable = 0, words = 0;   // words of a chunk's records, entries of a table row
};

RecordPlan planRecords(const ChunkedPlan &chunked) {
  RecordPlan p;
  if (!chunked.possible) return p;
  p.chunks = chunked.chunks;
  // (a record's segments take whole words)
  p.stride = (chunked.chunk * chunked.rowWords + (chunked.chunk + 3 * chunked.buckets) / 4 + 4) / 4 * 4;
  p.pitch = (chunked.buckets + 1 + 7) / 8 * 8;
  p.wTable = p.chunks * p.stride;
  p.words = p.wTable + p.chunks * p.pitch / 2;
  p.possible = p.words < (1LL << 32) && p.stride <= 65535;   // (32-bit word numbers, 16-bit ones within a chunk)
  return p;
}

// Device code of the schedule by records. The emitter defines the constants and types in front of it.
const char *const kRecordCode = R"AKG(
// Words of a record of n entries: n bytes, the segments within the bucket, in whole words, then n rows.
__device__ inline unsigned record_words(unsigned n) { return n * ROW_WORDS + (n + 3u) / 4u; }
// ... and the entries of a record of that many words.
__device__ inline unsigned record_entries(unsigned words) { return words * 4u / (4u * ROW_WORDS + 1u); }

__device__ inline void place_records(const id_store *__restrict__ ids, const unsigned *__restrict__ data, unsigned *__restrict__ ws) {
  constexpr int THREADS = NW * 64, PER = (KEYS + THREADS - 1) / THREADS;
  // the lane masks of the ranking, then (a barrier later) the chunk's records
  constexpr int MASK_BYTES = NW * KEYS * 8, STAGE_BYTES = STRIDE * 4;
  __shared__ __attribute__((aligned(16))) unsigned char akg_stage[MASK_BYTES > STAGE_BYTES ? MASK_BYTES : STAGE_BYTES];
  __shared__ unsigned short akg_cnt[NW * KEYS];
  __shared__ __attribute__((aligned(16))) unsigned short akg_start[PITCH];   // where a record begins, in words
  __shared__ unsigned short akg_rows[KEYS];                                   // ... and its rows
  __shared__ unsigned akg_scan[NW];
  const int tid = static_cast<int>(threadIdx.x), lane = tid & 63, w = tid >> 6;
  const row_t *__restrict__ rows = reinterpret_cast<const row_t *>(data);
  const unsigned long long bit = 1ull << lane;
  unsigned long long *masks = reinterpret_cast<unsigned long long *>(akg_stage), *lanes = masks + w * KEYS;
  unsigned short *mine = akg_cnt + w * KEYS;
  int next_id[TILES];
  row_t next_row[TILES];
  const auto fetch = [&](int chunk, int u) {   // (positions behind the last one read the last one's row and take no part)
    const int p = chunk * CHUNK + (w * TILES + u) * 64 + lane, at = p < POSITIONS ? p : POSITIONS - 1;
    const int id = as_segment(load_id(ids, at));
    next_id[u] = p < POSITIONS ? id : -1;
    next_row[u] = rows[at];
  };
#pragma unroll
  for (int u = 0; u < TILES; ++u) fetch(static_cast<int>(blockIdx.x), u);
  for (int chunk = static_cast<int>(blockIdx.x); chunk < CHUNKS; chunk += static_cast<int>(gridDim.x)) {
    int key[TILES];   // the bucket, and the segment within it in the upper half
    row_t row[TILES];
    unsigned slot[TILES];
#pragma unroll
    for (int u = 0; u < TILES; ++u) {
      const unsigned bucket = static_cast<unsigned>(next_id[u]) / S;
      key[u] = next_id[u] >= 0 ? static_cast<int>(bucket | (static_cast<unsigned>(next_id[u]) - bucket * S) << 16) : -1;
      row[u] = next_row[u];
    }
    for (int k = tid; k < NW * KEYS; k += THREADS) {
      masks[k] = 0ull;
      akg_cnt[k] = 0;
    }
    __syncthreads();
    // rank among the wavefront's items of the bucket, as in chunk_rank; behind every tile its loads for the next chunk (all of them in
    // front waited for the stores of the chunk before: 13 of the 28 thousand cycles of a chunk)
    const int next = chunk + static_cast<int>(gridDim.x) < CHUNKS ? chunk + static_cast<int>(gridDim.x) : CHUNKS - 1;
#pragma unroll
    for (int u = 0; u < TILES; ++u) {
      slot[u] = 0u;
      if (key[u] >= 0) {
        const int k = key[u] & 0xffff;
        __hip_atomic_fetch_or(lanes + k, bit, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        __builtin_amdgcn_wave_barrier();
        const unsigned long long same = __hip_atomic_load(lanes + k, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        const unsigned before = mine[k];
        __builtin_amdgcn_wave_barrier();
        __hip_atomic_store(lanes + k, 0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        slot[u] = __builtin_amdgcn_mbcnt_hi(static_cast<unsigned>(same >> 32), __builtin_amdgcn_mbcnt_lo(static_cast<unsigned>(same), before));
        mine[k] = static_cast<unsigned short>(before + static_cast<unsigned>(__popcll(same)));   // (the same from every lane of the key)
      }
      __builtin_amdgcn_wave_barrier();
      fetch(next, u);
    }
    __syncthreads();
    unsigned count[PER], words = 0u;
#pragma unroll
    for (int j = 0; j < PER; ++j) {
      const int k = tid * PER + j;
      count[j] = 0u;
      if (k < KEYS) {
#pragma unroll
        for (int h = 0; h < NW; ++h) {
          const unsigned n = akg_cnt[h * KEYS + k];
          akg_cnt[h * KEYS + k] = static_cast<unsigned short>(count[j]);
          count[j] += n;
        }
      }
      words += record_words(count[j]);
    }
    unsigned incl = words;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
      const unsigned o = __shfl_up(incl, d);
      if (lane >= d) incl += o;
    }
    if (lane == 63) akg_scan[w] = incl;
    __syncthreads();
    unsigned at = incl - words;
#pragma unroll
    for (int j = 0; j < NW; ++j) at += j < w ? akg_scan[j] : 0u;
#pragma unroll
    for (int j = 0; j < PER; ++j) {
      const int k = tid * PER + j;
      if (k < KEYS) {
        akg_start[k] = static_cast<unsigned short>(at);
        akg_rows[k] = static_cast<unsigned short>(at + (count[j] + 3u) / 4u);
      }
      at += record_words(count[j]);
    }
    if (tid == THREADS - 1) akg_start[KEYS] = static_cast<unsigned short>(at);
    __syncthreads();
#pragma unroll
    for (int u = 0; u < TILES; ++u) {
      if (key[u] >= 0) {
        const int k = key[u] & 0xffff;
        const unsigned rank = slot[u] + mine[k];
        akg_stage[akg_start[k] * 4u + rank] = static_cast<unsigned char>(key[u] >> 16);
        unsigned *to = reinterpret_cast<unsigned *>(akg_stage) + akg_rows[k] + rank * ROW_WORDS;
#pragma unroll
        for (int c = 0; c < ROW_WORDS; ++c) to[c] = row[u].w[c];
      }
    }
    __syncthreads();
    // whole 16-byte pieces; what lies behind the segments of a record and behind the last record is never looked at
    const int pieces = (akg_start[KEYS] + 3) / 4;
    quad_words *out = reinterpret_cast<quad_words *>(ws + static_cast<long>(chunk) * STRIDE);
    for (int i = tid; i < pieces; i += THREADS) out[i] = reinterpret_cast<const quad_words *>(akg_stage)[i];
    out = reinterpret_cast<quad_words *>(ws + W_TABLE + static_cast<long>(chunk) * (PITCH / 2));
    for (int i = tid; i < PITCH / 8; i += THREADS) out[i] = reinterpret_cast<const quad_words *>(akg_start)[i];
    __syncthreads();
  }
}

__device__ inline void sum_records(const unsigned *__restrict__ ws, store_t *__restrict__ out0) {
  constexpr int PLANE = CAP + 4 * S;
  static_assert(PER_WAVE <= 64 && W * PER_WAVE >= CHAINS, "a lane for every output element");
  // row of entry k of the round: rows + k * ROW_WORDS; its segment: byte k - first of the record, `words` words in front of the rows
  struct run_t { unsigned rows; short first, words; };
  __shared__ unsigned short akg_run[CAP];             // whose run each entry of the round is
  __shared__ run_t akg_base[W * 64];
  // column c of a round's rows from c * PLANE on, lists per segment; what add_list reads behind the last one
  __shared__ __attribute__((aligned(16))) compute_t akg_plane[ROW * PLANE + ADD_BLOCK];
  __shared__ unsigned short akg_cnt[W * S];
  __shared__ unsigned akg_start[S], akg_len[S], akg_scan[W], akg_sums[W], akg_taken[W], akg_cut;
  const int tid = static_cast<int>(threadIdx.x), lane = tid & 63, w = tid >> 6;
  const int bucket = akg::xcd_contiguous_id(static_cast<int>(blockIdx.x), KEYS);
  const unsigned char *__restrict__ segs = reinterpret_cast<const unsigned char *>(ws);
  const unsigned short *__restrict__ table = reinterpret_cast<const unsigned short *>(ws + W_TABLE) + bucket;
  // the output element of this lane, if it has one: wavefront w adds chains w * PER_WAVE ...
  const int chain = w * PER_WAVE + lane;
  const bool has = lane < PER_WAVE && chain < CHAINS;
  const int cs = has ? chain / ROW : 0, cc = has ? chain - cs * ROW : 0;
  compute_t acc = 0;
  unsigned begin = 0u, behind = 0u;   // this thread's record of the round: words begin .. behind - 1 of its chunk
  const auto look_up = [&](int chunk) {
    const unsigned short *t = table + static_cast<long>(chunk < CHUNKS ? chunk : CHUNKS - 1) * PITCH;
    begin = t[0];
    behind = t[1];
  };
  look_up(tid);
  cell_t cur[T];
  int segment[T];
  unsigned total = 0u, skip = 0u;   // entries of the round on its way; entries of its first run that earlier rounds had
  int chunk0 = 0;
  const auto next_round = [&]() {
    const int chunk = chunk0 + tid;
    const unsigned all = chunk < CHUNKS ? record_entries(behind - begin) : 0u, had = tid == 0 ? skip : 0u, len = all - had;
    unsigned incl = len;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
      const unsigned o = __shfl_up(incl, d);
      if (lane >= d) incl += o;
    }
    if (lane == 63) akg_sums[w] = incl;
    if (tid == 0) akg_cut = 0u;
    __syncthreads();
    unsigned sum = 0u;
#pragma unroll
    for (int j = 0; j < W; ++j) {
      incl += j < w ? akg_sums[j] : 0u;
      sum += akg_sums[j];
    }
    // the round's last run may be cut; the next round begins inside it
    const unsigned excl = incl - len, left = excl < static_cast<unsigned>(CAP) ? CAP - excl : 0u, take = len < left ? len : left;
    const int whole = __popcll(__ballot(chunk < CHUNKS && incl <= static_cast<unsigned>(CAP)));
    if (lane == 0) akg_taken[w] = static_cast<unsigned>(whole);
    if (take > 0u && take < len) akg_cut = had + take;
    const unsigned word = static_cast<unsigned>(chunk) * static_cast<unsigned>(STRIDE) + begin;
    const int to_first = static_cast<int>(excl) - static_cast<int>(had);   // (a run beyond the round is not looked at)
    akg_base[tid] = {word + (all + 3u) / 4u - static_cast<unsigned>(to_first) * ROW_WORDS, static_cast<short>(to_first), static_cast<short>((all + 3u) / 4u)};
    // every run's entries, one after the other; runs of more than 32 by the whole wavefront
    unsigned long long longer = __ballot(take > 32u);
    if (take <= 32u) {
      for (unsigned i = 0; i < take; ++i) akg_run[excl + i] = static_cast<unsigned short>(tid);
    }
    while (longer) {
      const int b = __builtin_ctzll(longer);
      longer &= longer - 1;
      const unsigned n = __builtin_amdgcn_readlane(take, b), to = __builtin_amdgcn_readlane(excl, b);
      for (unsigned i = lane; i < n; i += 64) akg_run[to + i] = static_cast<unsigned short>(w * 64 + b);
    }
    __syncthreads();
    int taken = 0;
#pragma unroll
    for (int j = 0; j < W; ++j) taken += static_cast<int>(akg_taken[j]);
    total = sum < static_cast<unsigned>(CAP) ? sum : CAP;
    skip = akg_cut;
    chunk0 += taken;
    look_up(chunk0 + tid);   // (the next round's records)
  };
  const auto fetch_round = [&]() {
#pragma unroll
    for (int u = 0; u < T; ++u) {
      const int k = (w * T + u) * 64 + lane;
      const bool there = static_cast<unsigned>(k) < total;   // (the workspace's first words where there is no entry)
      const run_t run = akg_base[there ? akg_run[k] : 0];
      const unsigned from = there ? run.rows + static_cast<unsigned>(k) * ROW_WORDS : 0u;
      cur[u].r = *reinterpret_cast<const row_t *>(ws + static_cast<unsigned long>(from));
      const unsigned record = run.rows + static_cast<unsigned>(run.first * ROW_WORDS - run.words);
      if constexpr (S > 1) segment[u] = segs[there ? static_cast<unsigned long>(record) * 4u + static_cast<unsigned>(k - run.first) : 0ul];
    }
  };
  next_round();
  fetch_round();
  for (;;) {
    int key[T];
    unsigned slot[T];
#pragma unroll
    for (int u = 0; u < T; ++u) key[u] = static_cast<unsigned>((w * T + u) * 64 + lane) < total ? (S == 1 ? 0 : segment[u]) : -1;
    if constexpr (S == 1) {   // (nothing to sort)
#pragma unroll
      for (int u = 0; u < T; ++u) slot[u] = static_cast<unsigned>((w * T + u) * 64 + lane);
      if (tid == 0) {
        akg_start[0] = 0u;
        akg_len[0] = total;
      }
    } else {
      chunk_sort<W, S, KEY_BITS, T, 4>(key, slot, akg_cnt, akg_start, akg_len, akg_scan);
    }
#pragma unroll
    for (int u = 0; u < T; ++u) {
      if (key[u] >= 0) {
#pragma unroll
        for (int c = 0; c < ROW; ++c) akg_plane[c * PLANE + slot[u]] = load_value(cur[u].v[c]);
      }
    }
    __syncthreads();
    // The next round's entries are requested while this one's are added up, by the wavefronts that add behind their additions: requests
    // wait for room in the CU's 32 KiB of lines on their way, and a round ends with its longest list.
    const bool more = chunk0 < CHUNKS;   // (uniform)
    if (more) next_round();
    if (has) {
      __builtin_amdgcn_s_setprio(3);
      acc = add_list(akg_plane + cc * PLANE + akg_start[cs], static_cast<int>(akg_len[cs]), acc, [](compute_t v, compute_t sum) { return add_value(v, sum); });
      __builtin_amdgcn_s_setprio(0);
    }
    if (!more) break;
    fetch_round();
    __syncthreads();
  }
  if (has && bucket * S + cs < SEGMENTS) out0[static_cast<long>(bucket * S + cs) * ROW + cc] = store_value(acc);
}
)AKG";

/**
 * As lowerSegmentChunked, for more positions: a bucket's run in a chunk is one record, a byte for the segment of every entry, in whole
 * words, and the rows behind them. What bounds the last launch is not bytes but the lines its workgroups touch (a CU has 32
 * KiB of lines on their way) and its phases: a run of eight entries touches two lines now, three with the segments elsewhere.
 * The last run of a round may be cut, so rounds are full.
 */
LoweredKernel lowerSegmentRecords(const OpGraph &g, const LoweringOptions &options, const SegmentShapes &sh, const ChunkedPlan &plan, const RecordPlan &records) {
  using lowering::computeTypeName;
  using lowering::dtypeTag;
  const TensorValue &data = *sh.data, &ids = *sh.ids, &out = *sh.out;
  const std::string ct = computeTypeName(out.dtype), tag = dtypeTag(out.dtype), idTag = dtypeTag(ids.dtype);
  const bool narrow = out.dtype == DType::F16 || out.dtype == DType::BF16 || out.dtype == DType::I8 || out.dtype == DType::I16;
  const bool small = sh.positions / plan.buckets < 1024 && plan.tiles <= 4;
  const int64_t perBucket = plan.perBucket, chains = perBucket * sh.slice;
  const int nw = small ? (plan.tiles == 1 && chains <= 128 ? 2 : 4) : 8, tiles = small && plan.tiles == 1 ? static_cast<int>(plan.chunk) / (nw * 64) : 8;
  const int64_t chainsPerWave = std::max<int64_t>(16, (chains + nw - 1) / nw);
  int keyBits = 1;
  while ((1LL << keyBits) < perBucket) ++keyBits;
  std::ostringstream s;
  s << "// Generated by the akg HIP lowering for gfx950. Op description: " << g.name << "\n";
  s << "// family: segment_sum (positions grouped by bucket of segments, chunk by chunk, in records), fusion class: "
    << operatorTemplateName(g.operatorTemplate) << "\n";
  s << "#include \"akg_rt.hpp\"\n\n";
  s << "namespace {\n";
  s << "constexpr int POSITIONS = " << sh.positions << ", SEGMENTS = " << sh.segments << ", S = " << perBucket << ", KEYS = " << plan.buckets
    << ", CHUNKS = " << records.chunks << ", PITCH = " << records.pitch << ", STRIDE = " << records.stride << ";\n";
  s << "constexpr int ROW = " << sh.slice << ", ROW_WORDS = " << plan.rowWords << ", KEY_BITS = " << keyBits << ", NW = 8, TILES = " << plan.tiles
    << ", CHUNK = NW * TILES * 64;\n";
  s << "constexpr int W = " << nw << ", T = " << tiles << ", CAP = W * T * 64, CHAINS = " << chains << ", PER_WAVE = " << chainsPerWave << ";\n";
  s << "constexpr long W_TABLE = " << records.wTable << ";\n";
  s << "using id_store = " << idTag << "::storage;\nusing store_t = " << tag << "::storage;\nusing compute_t = " << ct << ";\n";
  s << "__device__ inline auto load_id(const id_store *ids, int at) { return " << idTag << "::load(ids[at]); }\n";
  s << "__device__ inline int as_segment(" << (ids.dtype == DType::I64 ? "long" : "int") << " v) { return v < 0 || v >= SEGMENTS ? -1 : static_cast<int>(v); }\n";
  s << "__device__ inline compute_t load_value(store_t v) { return " << tag << "::load(v); }\n";
  s << "__device__ inline store_t store_value(compute_t v) { return " << tag << "::store(v); }\n";
  s << "__device__ inline compute_t add_value(compute_t v, compute_t acc) { return " << (narrow ? tag + "::rnd(" : "(") << "akg::op_add(v, acc)); }\n";
  s << "struct __attribute__((aligned(4))) row_t { unsigned w[ROW_WORDS]; };\n";
  s << "union cell_t { row_t r; store_t v[ROW_WORDS * 4 / sizeof(store_t)]; };\n";
  s << "typedef unsigned quad_words __attribute__((ext_vector_type(4)));\n";
  s << "constexpr int ADD_BLOCK = " << addBlock(sh, ct, narrow) << ";\n" << kChunkSort << kAddList << kRecordCode;
  s << "}  // namespace\n\n";
  std::ostringstream params;
  for (size_t i = 0; i < g.inputs.size(); ++i) {
    params << (i ? ", " : "") << "const " << dtypeTag(g.tensor(g.inputs[i]).dtype) << "::storage *__restrict__ in" << i;
  }
  params << ", " << tag << "::storage *__restrict__ out0, unsigned *__restrict__ akg_ws";
  s << "extern \"C\" __global__ __launch_bounds__(512, 4) void " << g.name << "_place(" << params.str() << ") {\n  place_records(in" << ids.inputIndex
    << ", reinterpret_cast<const unsigned *>(in" << data.inputIndex << "), akg_ws);\n}\n\n";
  s << "extern \"C\" __global__ __launch_bounds__(" << nw * 64 << (small ? "" : ", 4") << ") void " << g.name << "_kernel(" << params.str() << ") {\n  sum_records(akg_ws, out0);\n}\n";

  LoweredKernel k;
  k.kernelName = g.name + "_kernel";
  k.source = s.str();
  k.family = KernelFamily::SegmentSum;
  k.grid[0] = static_cast<unsigned>(plan.buckets);
  k.block[0] = static_cast<unsigned>(nw * 64);
  KernelPhase place;
  place.kernelName = g.name + "_place";
  place.grid[0] = static_cast<unsigned>(std::min<int64_t>(records.chunks, 2LL * options.computeUnits));
  place.block[0] = 512;
  k.earlierPhases.push_back(place);
  k.workspaceBytes = static_cast<uint64_t>(records.words) * 4;
  k.algorithmicBytes = lowering::countAlgorithmicBytes(g);
  k.shapeArgs = lowering::buildShapeArgs(g);
  std::ostringstream note;
  note << "segment_sum positions=" << sh.positions << " segments=" << sh.segments << " slice=" << sh.slice << " chunks=" << records.chunks << " of "
       << plan.chunk << " positions grouped by bucket of " << perBucket << " segments in records: " << plan.buckets << " buckets, 2 launches";
  k.scheduleNote = note.str();
  return k;
}

LoweredKernel lowerSegmentScan(const OpGraph &g, const LoweringOptions &options, const SegmentShapes &sh) {
  using lowering::computeTypeName;
  using lowering::dtypeTag;
  const OpNode &op = *sh.op;
  const TensorValue &data = *sh.data, &ids = *sh.ids, &out = *sh.out;
  const int64_t positions = sh.positions, segments = sh.segments, slice = sh.slice;
  const std::string ct = computeTypeName(out.dtype), tag = dtypeTag(out.dtype), idTag = dtypeTag(ids.dtype);
  const bool narrow = out.dtype == DType::F16 || out.dtype == DType::BF16 || out.dtype == DType::I8 || out.dtype == DType::I16;
  const int accBytes = out.dtype == DType::I64 || out.dtype == DType::F64 ? 8 : 4;
  // Short slices: the lane that found the id adds the whole slice itself (its data loads are issued before the
  // serial part). Otherwise the threads of the workgroup share the columns of the slice.
  const bool laneOwned = slice <= 4;
  const int block = options.block > 0 ? options.block : (slice <= 64 ? 64 : 256);
  if (block % 64 != 0 || block > 1024 || (laneOwned && block != 64)) throw LoweringError("op " + op.name + ": unsupported block size");
  const int64_t sliceTile = std::min<int64_t>(slice, 8192 / (accBytes / 4));
  const int64_t sliceTiles = (slice + sliceTile - 1) / sliceTile;
  // segments per workgroup: about 1024 workgroups (every one of them scans all ids; measured on 24.5 million positions
  // into 4954 segments: 256 -> 36 ms, 512 -> 26 ms, 1024 -> 21.6 ms, 2048 -> 20.4 ms), bounded by 32 KB of accumulators
  const int64_t wantGroups = options.split > 0 ? options.split : 1024;
  int64_t segsPerWg = std::max<int64_t>(1, (segments * sliceTiles + wantGroups - 1) / wantGroups);
  segsPerWg = std::min<int64_t>(segsPerWg, std::max<int64_t>(1, 32768 / (sliceTile * accBytes)));
  const int64_t groups = (segments + segsPerWg - 1) / segsPerWg;
  if (groups >= (1LL << 31) || sliceTiles >= 65536) throw LoweringError("op " + op.name + ": too large");
  // ids per lane and load (one 16-byte load where the id type allows), loads in flight per lane
  const int idv = ids.dtype == DType::I32 ? 4 : ids.dtype == DType::I64 ? 2 : 1;
  const int unroll = options.chunks > 0 ? options.chunks : 4;
  const std::string rndOpen = narrow ? tag + "::rnd(" : std::string("(");
  std::ostringstream s;
  s << "// Generated by the akg HIP lowering for gfx950. Op description: " << g.name << "\n";
  s << "// family: segment_sum, fusion class: " << operatorTemplateName(g.operatorTemplate) << "\n";
  s << "#include \"akg_rt.hpp\"\n\n";
  s << "extern \"C\" __global__ __launch_bounds__(" << block << ") void " << g.name << "_kernel(";
  for (size_t i = 0; i < g.inputs.size(); ++i) {
    s << (i ? ", " : "") << "const " << dtypeTag(g.tensor(g.inputs[i]).dtype) << "::storage *__restrict__ in" << i;
  }
  s << ", " << tag << "::storage *__restrict__ out0) {\n";
  s << "  constexpr int POSITIONS = " << positions << ", SEGMENTS = " << segments << ", SEGS = " << segsPerWg << ";\n";
  s << "  constexpr long SLICE = " << slice << ";\n  constexpr int TILE = " << sliceTile << ", BLOCK = " << block
    << ", IDV = " << idv << ", U = " << unroll << ";\n";
  s << "  using id_t = " << idTag << "::storage;\n";
  s << "  struct __attribute__((aligned(sizeof(id_t) * IDV))) id_chunk { id_t v[IDV]; };\n";
  s << "  __shared__ " << ct << " akg_acc[SEGS * TILE];\n";
  s << "  const int tid = static_cast<int>(threadIdx.x), lane = tid & 63;\n";
  s << "  const int seg0 = static_cast<int>(blockIdx.x) * SEGS;\n";
  s << "  const int seg1 = seg0 + SEGS < SEGMENTS ? seg0 + SEGS : SEGMENTS;\n";
  s << "  const long col0 = static_cast<long>(blockIdx.y) * TILE;\n";
  s << "  const int cols = SLICE - col0 < TILE ? static_cast<int>(SLICE - col0) : TILE;\n";
  s << "  const id_t *__restrict__ ids = in" << ids.inputIndex << ";\n";
  s << "  const " << tag << "::storage *__restrict__ data = in" << data.inputIndex << ";\n";
  s << "  for (int k = tid; k < SEGS * TILE; k += BLOCK) akg_acc[k] = " << lowering::literalFor(out.dtype, 0.0) << ";\n";
  s << "  __syncthreads();\n";
  if (laneOwned) {
    s << "  // one wavefront: LDS accesses of a wavefront complete in program order, so the loop needs no barrier\n";
  } else {
    s << "  // from here on a thread reads and writes only its own accumulator columns: no further barrier\n";
  }
  // ids as int: anything outside [0, SEGMENTS) becomes -1 (matches nobody)
  const std::string toInt = ids.dtype == DType::I64
      ? "[](long v) { return v < 0 || v >= SEGMENTS ? -1 : static_cast<int>(v); }"
      : "[](int v) { return v; }";
  s << "  const auto as_int = " << toInt << ";\n";
  // The part every lane can load without a bounds check runs double-buffered: the ids of the next step are in flight
  // while the hits of the current one are handled. The last, partial step loads element by element.
  const auto emitHits = [&](const std::string &ind) {
    const std::string isHit = "(id[u][e] >= seg0 && id[u][e] < seg1)";
    if (laneOwned) {
      // first every data load of the step (all lanes, all chunks at once), then the additions in position order
      s << ind << "unsigned long long hits[U];\n";
      s << ind << ct << " v[U][IDV][" << slice << "];\n";
      s << ind << "#pragma unroll\n";
      s << ind << "for (int u = 0; u < U; ++u) {\n";
      s << ind << "  bool mine = false;\n";
      s << ind << "#pragma unroll\n";
      s << ind << "  for (int e = 0; e < IDV; ++e) mine = mine || " << isHit << ";\n";
      s << ind << "  hits[u] = __ballot(mine);\n";
      s << ind << "  if (hits[u] == 0) continue;\n";
      s << ind << "  const long mypos = static_cast<long>(base) + static_cast<long>(u * 64 + lane) * IDV;\n";
      s << ind << "#pragma unroll\n";
      s << ind << "  for (int e = 0; e < IDV; ++e) {\n";
      s << ind << "    if " << isHit << " {\n";
      s << ind << "#pragma unroll\n";
      s << ind << "      for (int c = 0; c < " << slice << "; ++c) v[u][e][c] = " << tag << "::load(data[(mypos + e) * SLICE + c]);\n";
      s << ind << "    }\n" << ind << "  }\n" << ind << "}\n";
      s << ind << "#pragma unroll\n";
      s << ind << "for (int u = 0; u < U; ++u) {\n";
      s << ind << "  unsigned long long todo = hits[u];\n";
      s << ind << "  while (todo) {   // ascending lanes = ascending positions\n";
      s << ind << "    const int b = __builtin_ctzll(todo);\n";
      s << ind << "    todo &= todo - 1;\n";
      s << ind << "    if (lane == b) {\n";
      s << ind << "#pragma unroll\n";
      s << ind << "      for (int e = 0; e < IDV; ++e) {\n";
      s << ind << "        if " << isHit << " {\n";
      s << ind << "          const int row = id[u][e] - seg0;\n";
      s << ind << "#pragma unroll\n";
      s << ind << "          for (int c = 0; c < " << slice << "; ++c) {\n";
      s << ind << "            akg_acc[row * TILE + c] = " << rndOpen << "akg::op_add(v[u][e][c], akg_acc[row * TILE + c]));\n";
      s << ind << "          }\n" << ind << "        }\n" << ind << "      }\n" << ind << "    }\n" << ind << "  }\n";
      s << ind << "}\n";
      return;
    }
    s << ind << "#pragma unroll\n";
    s << ind << "for (int u = 0; u < U; ++u) {\n";
    s << ind << "  bool mine = false;\n";
    s << ind << "#pragma unroll\n";
    s << ind << "  for (int e = 0; e < IDV; ++e) mine = mine || " << isHit << ";\n";
    s << ind << "  unsigned long long hits = __ballot(mine);\n";
    s << ind << "  if (hits == 0) continue;\n";
    s << ind << "  const long first = static_cast<long>(base) + static_cast<long>(u * 64) * IDV;   // lane 0, element 0\n";
    s << ind << "  while (hits) {   // ascending lanes, then ascending elements = ascending positions\n";
    s << ind << "    const int b = __builtin_ctzll(hits);\n";
    s << ind << "    hits &= hits - 1;\n";
    s << ind << "#pragma unroll\n";
    s << ind << "    for (int e = 0; e < IDV; ++e) {\n";
    s << ind << "      const int sid = __builtin_amdgcn_readlane(id[u][e], b);\n";
    s << ind << "      if (sid < seg0 || sid >= seg1) continue;\n";
    s << ind << "      const int row = sid - seg0;\n";
    s << ind << "      const long from = (first + b * IDV + e) * SLICE + col0;\n";
    s << ind << "      for (int c = tid; c < cols; c += BLOCK) {\n";
    s << ind << "        akg_acc[row * TILE + c] = " << rndOpen << "akg::op_add(" << tag
      << "::load(data[from + c]), akg_acc[row * TILE + c]));\n";
    s << ind << "      }\n" << ind << "    }\n" << ind << "  }\n";
    s << ind << "}\n";
  };
  s << "  constexpr int STEP = 64 * IDV * U, FULL = POSITIONS / STEP * STEP;\n";
  s << "  if (FULL > 0) {\n";
  s << "    id_chunk next[U];\n";
  s << "#pragma unroll\n";
  s << "    for (int u = 0; u < U; ++u) next[u] = *reinterpret_cast<const id_chunk *>(ids + (u * 64 + lane) * IDV);\n";
  s << "    for (int base = 0; base < FULL; base += STEP) {\n";
  s << "      int id[U][IDV];\n";
  s << "#pragma unroll\n";
  s << "      for (int u = 0; u < U; ++u) {\n";
  s << "#pragma unroll\n";
  s << "        for (int e = 0; e < IDV; ++e) id[u][e] = as_int(" << idTag << "::load(next[u].v[e]));\n";
  s << "      }\n";
  s << "      if (base + STEP < FULL) {\n";
  s << "#pragma unroll\n";
  s << "        for (int u = 0; u < U; ++u) next[u] = *reinterpret_cast<const id_chunk *>(ids + base + STEP + (u * 64 + lane) * IDV);\n";
  s << "      }\n";
  emitHits("      ");
  s << "    }\n  }\n";
  s << "  if (FULL < POSITIONS) {\n";
  s << "    constexpr int base = FULL;\n";
  s << "    int id[U][IDV];\n";
  s << "#pragma unroll\n";
  s << "    for (int u = 0; u < U; ++u) {\n";
  s << "#pragma unroll\n";
  s << "      for (int e = 0; e < IDV; ++e) {\n";
  s << "        const int p = base + (u * 64 + lane) * IDV + e;\n";
  s << "        id[u][e] = p < POSITIONS ? as_int(" << idTag << "::load(ids[p])) : -1;\n";
  s << "      }\n    }\n";
  emitHits("    ");
  s << "  }\n";
  s << "  for (int r = 0; r < seg1 - seg0; ++r) {\n";
  s << "    for (int c = tid; c < cols; c += BLOCK) {\n";
  s << "      out0[static_cast<long>(seg0 + r) * SLICE + col0 + c] = " << tag << "::store(akg_acc[r * TILE + c]);\n";
  s << "    }\n  }\n}\n";

  LoweredKernel k;
  k.kernelName = g.name + "_kernel";
  k.source = s.str();
  k.family = KernelFamily::SegmentSum;
  k.grid[0] = static_cast<unsigned>(groups);
  k.grid[1] = static_cast<unsigned>(sliceTiles);
  k.block[0] = block;
  k.algorithmicBytes = lowering::countAlgorithmicBytes(g);
  k.shapeArgs = lowering::buildShapeArgs(g);
  std::ostringstream note;
  note << "segment_sum positions=" << positions << " segments=" << segments << " slice=" << slice << " segments/workgroup=" << segsPerWg << " slice tile=" << sliceTile;
  k.scheduleNote = note.str();
  return k;
}

// Wide rows and at most 2^16 positions, as gradients of embedding tables have: one launch without a workspace. Workgroup (g, t)
// sums the segments congruent to g modulo GROUPS in column tile t, one column a thread:
//   it counts its positions per segment, lists them by segment and in their order (LDS), and walks the list with 64 rows in flight,
//   whatever segments they belong to; zeros for segments without positions it writes for its own or for a share of adjacent ones.
// Frequent ids are often neighbours (tokens by rank), so neighbouring segments go to different workgroups, and a workgroup's
// columns are at most 256. More positions than the list holds: by windows of the positions, the sums wait in the result
// between them.
// What bounds it is the chain of a frequent segment's rows where there is one (16000 x 128 into 1000: 1600 rows, 43 us; 69 us with
// addresses in vector registers, 112 us where every wait was for all 64 rows) and two scans of the ids by every workgroup where there
// is none. At most 1024 workgroups, four a CU: 512 and 2048 take 98 and 102 us for 89 (32768 x 1024 into 32768, uniform ids), 1536 take
// 85 for 72 (20000 x 768 into 30522). All tiles of a group on one CU, as they were launched, took 225 us for 124 (ids as frequent
// as words).
struct ListedPlan {
  int64_t tiles = 0, block = 0, groupBits = 0, keys = 0;
  bool possible = false;
};

ListedPlan planListed(const SegmentShapes &sh, const LoweringOptions &options) {
  ListedPlan plan;
  if (sh.slice <= 64 || sh.positions > (1 << 20) || options.block > 0) return plan;
  plan.tiles = (sh.slice + 255) / 256;
  plan.block = ((sh.slice + plan.tiles - 1) / plan.tiles + 63) / 64 * 64;
  plan.tiles = (sh.slice + plan.block - 1) / plan.block;
  if (plan.tiles == 1) plan.block = 256;   // (four wavefronts for the ids, whatever the columns)
  const int64_t want = options.split > 0 ? options.split : 1024;
  while (plan.groupBits < 24 && (2LL << plan.groupBits) * plan.tiles <= want && (1LL << plan.groupBits) < sh.segments) ++plan.groupBits;
  while (((sh.segments + (1LL << plan.groupBits) - 1) >> plan.groupBits) > 512) ++plan.groupBits;
  plan.keys = (sh.segments + (1LL << plan.groupBits) - 1) >> plan.groupBits;
  plan.possible = plan.tiles < 65536;
  return plan;
}

LoweredKernel lowerSegmentListed(const OpGraph &g, const SegmentShapes &sh, const ListedPlan &plan) {
  using lowering::computeTypeName;
  using lowering::dtypeTag;
  const TensorValue &ids = *sh.ids, &out = *sh.out;
  const std::string ct = computeTypeName(out.dtype), tag = dtypeTag(out.dtype), idTag = dtypeTag(ids.dtype);
  const bool narrow = out.dtype == DType::F16 || out.dtype == DType::BF16 || out.dtype == DType::I8 || out.dtype == DType::I16;
  std::ostringstream s;
  s << "// Generated by the akg HIP lowering for gfx950. Op description: " << g.name << "\n";
  s << "// family: segment_sum (positions listed by segment), fusion class: " << operatorTemplateName(g.operatorTemplate) << "\n";
  s << "#include \"akg_rt.hpp\"\n\n";
  s << "extern \"C\" __global__ __launch_bounds__(" << plan.block << ") void " << g.name << "_kernel(";
  for (size_t i = 0; i < g.inputs.size(); ++i) {
    s << (i ? ", " : "") << "const " << dtypeTag(g.tensor(g.inputs[i]).dtype) << "::storage *__restrict__ in" << i;
  }
  s << ", " << tag << "::storage *__restrict__ out0) {\n";
  s << "  constexpr int POSITIONS = " << sh.positions << ", SEGMENTS = " << sh.segments << ", BLOCK = " << plan.block << ", NW = BLOCK / 64;\n";
  s << "  constexpr int BITS = " << plan.groupBits << ", GROUPS = 1 << BITS, KEYS = " << plan.keys << ", LIST = 8192;\n";
  const int64_t idv = ids.dtype == DType::I32 ? 4 : ids.dtype == DType::I64 ? 2 : 1;
  // chunks of ids a lane has in flight: no more than there are, as every workgroup loads them all (eight for 2000 x 128 into 2000,
  // where there are two: 33 MB from L2, 2.5 of 8.5 us)
  const int64_t inFlight = std::min<int64_t>(8, (sh.positions + plan.block * idv - 1) / (plan.block * idv));
  s << "  constexpr int IDV = " << idv << ", U = " << inFlight << ";\n";
  // Segments without positions: a share of adjacent ones per workgroup, in pieces of up to 16 bytes, so that lines are written whole and by
  // one XCD. Finding out which ones have none costs two instructions an id and workgroup: with more than 4096 positions a workgroup
  // writes zeros for its own segments. us, uniform ids, own / share: 512 x 1000 into 32768 43.4 / 31.2 (rows of 4000 bytes), 800 x 1544
  // into 16000 34.7 / 27.0, 4096 x 128 into 4096 9.4 / 7.8, 8192 x 256 into 8000 11.8 / 13.1, 60000 x 200 into 9000 58 / 64.
  const bool byShare = sh.positions <= 4096;
  int64_t piece = 16 / static_cast<int64_t>(dtypeSize(out.dtype));
  while (sh.slice % piece != 0) piece /= 2;
  const int64_t workgroups = (1LL << plan.groupBits) * plan.tiles;
  s << "  constexpr int WORKGROUPS = " << workgroups << ", SHARE_ROWS = " << (sh.segments + workgroups - 1) / workgroups << ", PIECE = " << piece
    << ", PIECES = " << sh.slice / piece << ";\n";
  s << "  constexpr bool BY_SHARE = " << (byShare ? "true" : "false") << ";\n";
  s << "  constexpr long SLICE = " << sh.slice << ";\n";
  s << "  using id_t = " << idTag << "::storage;\n";
  s << "  using T = " << tag << ";\n  using ID = " << idTag << ";\n";
  s << "  using acc_t = " << ct << ";\n";
  s << "  const id_t *__restrict__ ids = in" << ids.inputIndex << ";\n";
  s << "  const T::storage *__restrict__ data = in" << sh.data->inputIndex << ";\n";
  s << "  const acc_t zero = " << lowering::literalFor(out.dtype, 0.0) << ";\n";
  // ids as int: anything outside [0, SEGMENTS) is nobody's
  s << "  const auto as_int = " << (ids.dtype == DType::I64 ? "[](long v) { return v < 0 || v >= SEGMENTS ? -1 : static_cast<int>(v); }"
                                                            : "[](int v) { return v; }") << ";\n";
  s << "  const auto add = [](acc_t v, acc_t acc) -> acc_t { return " << (narrow ? "T::rnd(" : "(") << "akg::op_add(v, acc)); };\n";
  s << R"(  struct __attribute__((aligned(sizeof(id_t) * IDV))) id_chunk { id_t v[IDV]; };
  __shared__ unsigned akg_count[NW * KEYS];   // [wavefront][key]: its positions, then where it lists the next one
  __shared__ unsigned akg_has[KEYS], akg_total;
  __shared__ unsigned akg_met[BY_SHARE ? SHARE_ROWS : 1];    // this workgroup's share of adjacent segments: which ones have positions
  __shared__ unsigned akg_list[LIST];         // key << 20 | position, by key
  const int tid = static_cast<int>(threadIdx.x), lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  // (the tiles of a group, of which all may be long, on different XCDs and CUs)
  const int group = static_cast<int>(blockIdx.x + 37 * blockIdx.y) & (GROUPS - 1);
  const long col = static_cast<long>(blockIdx.y) * BLOCK + tid;
  const bool has = col < SLICE;
  const unsigned from_col = static_cast<unsigned>(has ? col : SLICE - 1);
  const unsigned share_first = static_cast<unsigned>(akg::xcd_contiguous_id(static_cast<int>(blockIdx.y * gridDim.x + blockIdx.x), WORKGROUPS)) * SHARE_ROWS;
  const auto mine = [&](int id) { return static_cast<unsigned>(id) < static_cast<unsigned>(SEGMENTS) && (id & (GROUPS - 1)) == group; };
  // ids that fit are loaded once
  constexpr bool ONCE = POSITIONS <= LIST && POSITIONS <= NW * 64 * IDV * U;
  id_chunk chunk[U];
  const auto load = [&](int base) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int p = base + (u * 64 + lane) * IDV;
      if constexpr (POSITIONS % IDV == 0) {
        chunk[u] = *reinterpret_cast<const id_chunk *>(ids + (p < POSITIONS ? p : 0));
      } else if (p + IDV <= POSITIONS) {
        chunk[u] = *reinterpret_cast<const id_chunk *>(ids + p);
      } else {
#pragma unroll
        for (int e = 0; e < IDV; ++e) {
          if (p + e < POSITIONS) chunk[u].v[e] = ids[p + e];
        }
      }
    }
  };
  constexpr int SHARE = (POSITIONS + NW * 64 * IDV - 1) / (NW * 64 * IDV) * (64 * IDV);
  if (ONCE) load(wave * SHARE);
  // the ids of positions [from, upto), a contiguous share per wavefront, 64 * IDV at a time in ascending order
  const auto scan = [&](int from, int upto, auto &&meet, auto &&visit) {
    const int share = (upto - from + NW * 64 * IDV - 1) / (NW * 64 * IDV) * (64 * IDV);
    const int first = from + wave * share, end = first + share < upto ? first + share : upto;
    for (int base = first; base < end; base += 64 * IDV * U) {
      if (!ONCE) load(base);
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int p = base + (u * 64 + lane) * IDV;
        int key[IDV];
        bool any = false;
#pragma unroll
        for (int e = 0; e < IDV; ++e) {
          const int id = p + e < end ? as_int(ID::load(chunk[u].v[e])) : -1;
          meet(static_cast<unsigned>(id) - share_first);
          key[e] = mine(id) ? id >> BITS : -1;
          any = any || key[e] >= 0;
        }
        if (__ballot(any) != 0) visit(p, key);
      }
    }
  };
  const auto count = [&](int from, int upto, auto &&meet) {
    for (int k = tid; k < NW * KEYS; k += BLOCK) akg_count[k] = 0;
    __syncthreads();
    scan(from, upto, meet, [&](int, const int (&key)[IDV]) {
#pragma unroll
      for (int e = 0; e < IDV; ++e) {
        if (key[e] >= 0) atomicAdd(&akg_count[wave * KEYS + key[e]], 1u);
      }
    });
    __syncthreads();
    if (wave == 0) {
      unsigned run = 0;
      for (int k0 = 0; k0 < KEYS; k0 += 64) {
        const int k = k0 + lane;
        unsigned c[NW], sum = 0;
#pragma unroll
        for (int w = 0; w < NW; ++w) {
          c[w] = k < KEYS ? akg_count[w * KEYS + k] : 0;
          sum += c[w];
        }
        unsigned upto_here = sum;
#pragma unroll
        for (int d = 1; d < (KEYS < 64 ? KEYS : 64); d <<= 1) {
          const unsigned below = __shfl_up(upto_here, d);
          if (lane >= d) upto_here += below;
        }
        unsigned at = run + upto_here - sum;
        if (k < KEYS) {
          akg_has[k] = sum;
#pragma unroll
          for (int w = 0; w < NW; ++w) {
            akg_count[w * KEYS + k] = at;
            at += c[w];
          }
        }
        run += __builtin_amdgcn_readlane(upto_here, KEYS < 64 ? KEYS - 1 : 63);
      }
      if (lane == 0) akg_total = run;
    }
    __syncthreads();
    return __builtin_amdgcn_readfirstlane(static_cast<int>(akg_total));
  };
  const auto pass_by = [](unsigned) {};
  const auto place = [&](int from, int upto) {
    scan(from, upto, pass_by, [&](int p, int (&key)[IDV]) {
      for (;;) {   // one key at a time; its positions go up with the lanes, then with the elements
        int pick = -1;
#pragma unroll
        for (int e = 0; e < IDV; ++e) pick = key[e] >= 0 ? key[e] : pick;
        const unsigned long long left = __ballot(pick >= 0);
        if (left == 0) break;
        const int one = __builtin_ctzll(left), k = __builtin_amdgcn_readlane(pick, one);
        unsigned before = 0, all = 0;
#pragma unroll
        for (int e = 0; e < IDV; ++e) {
          const unsigned long long same = __ballot(key[e] == k);
          before += __builtin_popcountll(same & ((1ULL << lane) - 1));
          all += __builtin_popcountll(same);
        }
        unsigned at = 0;
        if (lane == one) at = atomicAdd(&akg_count[wave * KEYS + k], all);
        at = __builtin_amdgcn_readlane(at, one) + before;
#pragma unroll
        for (int e = 0; e < IDV; ++e) {
          if (key[e] == k) {
            akg_list[at++] = static_cast<unsigned>(k) << 20 | static_cast<unsigned>(p + e);
            key[e] = -1;
          }
        }
      }
    });
    __syncthreads();
  };
  const __amdgpu_buffer_rsrc_t rows = __builtin_amdgcn_make_buffer_rsrc(const_cast<T::storage *>(data), 0,
      static_cast<int>(POSITIONS * SLICE * sizeof(T::storage) < 0x7fffffffUL ? POSITIONS * SLICE * sizeof(T::storage) : 0x7fffffffUL), 0x00020000);
  const auto row_of = [&](int k) { return (static_cast<long>(k) << BITS | group) * SLICE + from_col; };
  struct AllAtOnce { enum { kGoesOn = 0 }; };
  struct ByWindows { enum { kGoesOn = 1 }; };
  const auto sum = [&](int n, auto how) {
    int current = -1;
    acc_t acc = zero, v[64];
    const auto fetch = [&](int q, unsigned entries) {   // eight rows of a chunk of 64 entries
      constexpr long BYTES = sizeof(T::storage);
      if constexpr (POSITIONS * SLICE * BYTES < (1L << 31)) {
        // one address for all lanes and one offset of a lane for all rows: two instructions a row
        const unsigned at = (entries & 0xfffffu) * static_cast<unsigned>(SLICE * BYTES);
        const int lane_at = static_cast<int>(from_col * BYTES);
#pragma unroll
        for (int u = q; u < q + 8; ++u) {
          const int row = __builtin_amdgcn_readlane(static_cast<int>(at), u);
          T::storage x;
          if constexpr (BYTES == 8) {
            const auto w = __builtin_amdgcn_raw_buffer_load_b64(rows, lane_at, row, 0);
            __builtin_memcpy(&x, &w, BYTES);
          } else if constexpr (BYTES == 4) {
            const auto w = __builtin_amdgcn_raw_buffer_load_b32(rows, lane_at, row, 0);
            __builtin_memcpy(&x, &w, BYTES);
          } else if constexpr (BYTES == 2) {
            const auto w = __builtin_amdgcn_raw_buffer_load_b16(rows, lane_at, row, 0);
            __builtin_memcpy(&x, &w, BYTES);
          } else {
            const auto w = __builtin_amdgcn_raw_buffer_load_b8(rows, lane_at, row, 0);
            __builtin_memcpy(&x, &w, BYTES);
          }
          v[u] = T::load(x);
        }
      } else {
#pragma unroll
        for (int u = q; u < q + 8; ++u) {
          const unsigned p = __builtin_amdgcn_readlane(entries, u) & 0xfffffu;
          v[u] = T::load((data + static_cast<long>(p) * SLICE)[from_col]);
        }
      }
    };
    const auto fold = [&](int q, unsigned entries, int left) {
      // (the list ascends: the last of eight in the current segment, all are)
      if (static_cast<int>(__builtin_amdgcn_readlane(entries, q + 7) >> 20) == current && q + 8 <= left) {
#pragma unroll
        for (int u = q; u < q + 8; ++u) acc = add(v[u], acc);
        return;
      }
#pragma unroll
      for (int u = q; u < q + 8; ++u) {
        if (u >= left) continue;
        const int k = static_cast<int>(__builtin_amdgcn_readlane(entries, u) >> 20);
        if (k != current) {
          if (current >= 0 && has) out0[row_of(current)] = T::store(acc);
          current = k;
          acc = zero;
          if constexpr (decltype(how)::kGoesOn) acc = T::load(out0[row_of(k)]);
        }
        acc = add(v[u], acc);
      }
    };
    const auto entries_at = [&](int i) { return akg_list[i + lane < n ? i + lane : n - 1]; };
    unsigned entries = entries_at(0);
    int i = 0;
    if (BY_SHARE && n <= 8) {
      // (the ways below jump over a part for every eight rows: 512 x 128 into 1000 4.1 us, 3.3 this way)
      fetch(0, entries);
      fold(0, entries, n);
      if (has) out0[row_of(current)] = T::store(acc);
      return;
    }
    if (n >= 128) {
      // eight rows are summed, the eight 64 behind them requested; no load is conditional, or the waits would be for all of them
#pragma unroll
      for (int q = 0; q < 64; q += 8) fetch(q, entries);
      for (; i + 128 <= n; i += 64) {
        const unsigned next = entries_at(i + 64);
#pragma unroll
        for (int q = 0; q < 64; q += 8) {
          fold(q, entries, 64);
          fetch(q, next);
        }
        entries = next;
      }
    } else {
#pragma unroll
      for (int q = 0; q < 64; q += 8) {
        if (q < n) fetch(q, entries);   // (entries beyond the list repeat its last one)
      }
    }
    for (; i < n; i += 64) {
      const unsigned next = entries_at(i + 64);
#pragma unroll
      for (int q = 0; q < 64; q += 8) {
        if (i + q < n) fold(q, entries, n - i);
        if (i + 64 + q < n) fetch(q, next);
      }
      entries = next;
    }
    if (has) out0[row_of(current)] = T::store(acc);
  };
  if constexpr (BY_SHARE) {
    for (int r = tid; r < SHARE_ROWS; r += BLOCK) akg_met[r] = 0;   // (a barrier follows)
  }
  const int n = count(0, POSITIONS, [&](unsigned r) {
    if (BY_SHARE && r < static_cast<unsigned>(SHARE_ROWS)) akg_met[r] = 1;
  });
  if constexpr (BY_SHARE) {
    struct __attribute__((aligned(sizeof(T::storage)))) zeros { T::storage v[PIECE]; };
    // (each workgroup begins elsewhere in its share: at a power-of-two distance they would all write to the same channels)
    constexpr int TRIPS = (SHARE_ROWS * PIECES + BLOCK - 1) / BLOCK;
    const int begin = static_cast<int>((blockIdx.x + blockIdx.y * gridDim.x) * 40503u % 65536u * TRIPS / 65536u);
    for (int trip = 0; trip < TRIPS; ++trip) {
      const int i = (trip + begin < TRIPS ? trip + begin : trip + begin - TRIPS) * BLOCK + tid, r = i / PIECES;
      if (r < SHARE_ROWS && share_first + r < static_cast<unsigned>(SEGMENTS) && akg_met[r] == 0) {
        *reinterpret_cast<zeros *>(out0 + static_cast<long>(share_first + r) * SLICE + (i - r * PIECES) * PIECE) = zeros{};
      }
    }
  } else {
    // (sums that go on from window to window begin with zeros)
    const bool all = POSITIONS > LIST && n > LIST;
    for (int k0 = 0; k0 < KEYS; k0 += 64) {
      const int k = k0 + lane;
      unsigned long long empty = __ballot(k < KEYS && (static_cast<long>(k) << BITS | group) < SEGMENTS && (all || akg_has[k] == 0));
      while (empty) {
        if (has) out0[row_of(k0 + __builtin_ctzll(empty))] = T::store(zero);
        empty &= empty - 1;
      }
    }
  }
  if (POSITIONS <= LIST || n <= LIST) {
    place(0, POSITIONS);
    if (n > 0) sum(n, AllAtOnce());
    return;
  }
  for (int from = 0; from < POSITIONS; from += LIST) {
    const int upto = from + LIST < POSITIONS ? from + LIST : POSITIONS;
    const int here = count(from, upto, pass_by);
    place(from, upto);
    if (here > 0) sum(here, ByWindows());
    __syncthreads();
  }
}
)";

  LoweredKernel k;
  k.kernelName = g.name + "_kernel";
  k.source = s.str();
  k.family = KernelFamily::SegmentSum;
  k.grid[0] = static_cast<unsigned>(1LL << plan.groupBits);
  k.grid[1] = static_cast<unsigned>(plan.tiles);
  k.block[0] = static_cast<unsigned>(plan.block);
  k.algorithmicBytes = lowering::countAlgorithmicBytes(g);
  k.shapeArgs = lowering::buildShapeArgs(g);
  std::ostringstream note;
  note << "segment_sum positions=" << sh.positions << " segments=" << sh.segments << " slice=" << sh.slice << " positions listed by segment: "
       << plan.keys << " segments/workgroup, column tiles=" << plan.tiles << " of " << plan.block;
  k.scheduleNote = note.str();
  return k;
}

}  // namespace

LoweredKernel lowerSegmentSumToHip(const OpGraph &g, const LoweringOptions &options) {
  const SegmentShapes sh = checkSegmentSum(g);
  // Grouping pays once the repeated id scan costs more than a few launches: from 2^16 positions on
  // (69 thousand positions into 4954 segments: 0.050 ms grouped, 0.069 ms scanned). Its LDS counters
  // hold one word per segment.
  const bool canGroup = sh.segments <= 16384 && sh.segments * sh.slice + 256 < (1LL << 31);
  const bool group = options.variant == 5 ? false : options.variant >= 2 ? canGroup : options.variant == 1 ? false : canGroup && sh.positions >= (1 << 16);
  // Short rows (4, 8 or 12 bytes, 4-byte arithmetic) into many segments: by bucket first. The bucket is the largest power
  // of two of segments whose output elements number at most 32; there are at most 640 buckets (the counters of a chunk
  // must leave room for two workgroups per CU) and, unless asked for, at least 96 (the last launch has one workgroup
  // per bucket: 1 to 4 million positions into 300 segments run 1.3 to 1.9 times slower than grouped by segment; 0.3 to
  // 4 million into 5000 segments 1.7 to 2.2 times faster, 24.5 million 1.9 times).
  const int64_t rowBytes = sh.slice * static_cast<int64_t>(dtypeSize(sh.out->dtype));
  const bool wide = sh.out->dtype == DType::I64 || sh.out->dtype == DType::F64;
  int bucketBits = 4;
  while (bucketBits > 0 && (sh.slice << bucketBits) > 32) --bucketBits;
  const int64_t buckets = (sh.segments + (1LL << bucketBits) - 1) >> bucketBits;
  const bool canBucket = group && !wide && rowBytes <= 12 && rowBytes % 4 == 0 && bucketBits >= 2 && buckets <= 640 && buckets >= 2;
  const bool bucketed = canBucket && (options.variant == 3 || (options.variant == 0 && buckets >= 96));
  // Short rows by chunks, two launches for five. From 2^19 positions on always; us, grouped by segment or by bucket -> by
  // chunk: 24.5 million x 3 into 4954 413 -> 300, 12.5 million x 4 into 2216 401 -> 226, 20 million x 4 into 16384 1665 -> 314,
  // 1.5 million x 4 into 12654 261 -> 30, 5 million x 1 into 300 234 -> 180, 600000 x 1 into 300 49 -> 31, x 3 into 16000 227 -> 17.
  // Below, where the positions would be grouped by segment and a bucket has several segments (244664 x 4 into 9073 82 -> 13,
  // 65974 x 1 into 13950 97 -> 8.9, 138073 x 1 into 998 29.6 -> 11.0, 200000 x 4 into 513 33.9 -> 14.5) or a row fewer than four elements
  // from 3 * 2^15 positions on (124495 x 1 into 384 25.6 -> 9.9, 511656 x 2 into 344 46 -> 19.5; a test pins 70000 x 3 into 500), where they would be grouped into fewer than 512 buckets (149736 x 3
  // into 2040 30.1 -> 11.4, 97239 x 2 into 3395 25.5 -> 10.2), and from 2^15 positions on instead of the scan (35304 x 1 into 1131
  // 42.0 -> 8.4, 33000 x 4 into 300 51 -> 9.1). The other two schedules would lose in between as well (300000 x 3 into 5000 36.7 by
  // bucket, 13.4 by chunk), but their launches are pinned by tests there. Nor may the workspace outgrow the 16 MiB of a
  // launch without allocations where the schedule it takes the place of stays within them, as the scan does, which has none:
  // 2 million x 3 into 20000 (26 MB by chunk) stays scanned, though that takes 1760 us for 32.
  const ChunkedPlan chunked = planChunked(sh, options);
  bool byChunk = chunked.possible && (options.variant == 4 || options.variant == 6);
  if (chunked.possible && options.variant == 0 && sh.positions >= (1 << 15)) {
    const bool many = sh.positions >= (1 << 19);
    byChunk = many || (group ? (bucketed ? buckets < 512 : chunked.perBucket > 1 || (sh.slice < 4 && sh.positions >= (3 << 15))) : sh.positions < (1 << 16));
    const int64_t runs = std::min<int64_t>(2048, std::max<int64_t>(1, sh.positions / 1024));   // (of the schedule by segment)
    const int64_t before = !group ? 0 : bucketed ? sh.positions * 4 : sh.positions * rowBytes / 4 + runs * sh.segments;
    if (chunked.words * 4 > (16 << 20) && before * 4 <= (16 << 20)) byChunk = false;
  }
  // In records from 2^21 positions on. us, rows and segments apart / records: 24.5 million x 3 into 4954 283 / 261, 20 million x 4 into
  // 16384 299 / 255, 14 million x 4 into 8656 208 / 180, 10.8 million x 1 into 5096 98 / 94, 2.7 million x 3 into 1909 42.2 / 41.5; below,
  // 1.7 million x 3 into 520 43.8 / 44.7, 838736 x 4 into 1311 25.5 / 26.3. Not where only the whole words of the segments take the workspace
  // beyond the 16 MiB of a launch without allocations. (AKG_HIP_VARIANT=6 takes them for any size.)
  const RecordPlan records = planRecords(chunked);
  const bool fits = records.words * 4 <= (16 << 20) || chunked.words * 4 > (16 << 20);
  if (byChunk && records.possible && (options.variant == 6 || (options.variant == 0 && options.chunks == 0 && fits && sh.positions >= (1 << 21)))) {
    return lowerSegmentRecords(g, options, sh, chunked, records);
  }
  if (byChunk) return lowerSegmentChunked(g, options, sh, chunked);
  if (bucketed) return lowerSegmentBucketed(g, options, sh, bucketBits);
  if (group) return lowerSegmentSorted(g, options, sh);
  // Wide rows listed by segment. us, ids as frequent as words (the k-th with 1 / k) and uniform ones, scanned -> listed: 32768 x 1024
  // into 32768 11600 -> 117 and 198 -> 92, 20000 x 768 into 30522 5780 -> 72 and 98 -> 52, 8192 x 256 into 8000 710 -> 22 and
  // 18.1 -> 11.8, 2048 x 1024 into 32000 745 -> 36 and 50 -> 33, 60000 x 200 into 9000 5690 -> 150 and 99 -> 58, 600 x 128 into 30000 48 ->
  // 6.6 and 8.1 -> 6.5, 512 x 1000 into 32768 205 -> 31 and 31 -> 31, 1500 x 400 into 3000 150 -> 9.2 and 7.2 -> 6.6. The least
  // there is, 512 x 128 into 1000, takes 14.5 -> 4.4 and 3.1 -> 3.3. Rows of 5 to 64 elements stay scanned, as a thread has a column of one row here:
  // fewer than 64 of a wavefront would work (32768 x 64 into 32768 43 us with uniform ids, 3730 with ids as frequent as words).
  const ListedPlan listed = planListed(sh, options);
  if (listed.possible && (options.variant == 5 || (options.variant == 0 && sh.positions >= 512))) return lowerSegmentListed(g, sh, listed);
  return lowerSegmentScan(g, options, sh);
}

}  // namespace akg
