/**
 * Scores of a contraction kept in registers for the row reductions behind them (attention probabilities: Q K^T, scale,
 * mask, softmax): C[M,N] = A[M,K] * B[N,K]^T, sixteen rows of A against all N columns in one workgroup, so that a row
 * of results is never written before its reductions are done.
 *
 * A unit is 16 rows x 32 columns: two 16 x 16 MFMAs per 64 bytes of K with the operands EXCHANGED (the columns of C, rows
 * of B, are the rows of the MFMA): lane (c = lane % 16, g = lane / 16) then owns row c of the tile, and with column
 * 8 (r / 4) + 4 h + r % 4 of the unit in row r of MFMA h it owns the EIGHT ADJACENT columns 8 g .. 8 g + 7: a mask or a
 * result is read and written 16 bytes a lane, whole lines over the four lanes of a row, and a row reduction ends with
 * two exchanges between lanes (distances 16 and 32) and one LDS step between the wavefronts of a row.
 * The wavefronts of a row take its units in pairs (row_unit). No LDS holds operands: B is read once per workgroup, straight into MFMA
 * fragments, from the L2 (the launch keeps the workgroups of a batch on one XCD).
 * What bounds it: memory (mask in, probabilities out) and the fragments of B, of which the L1s ask the L2s for as many lines
 * (1.57 million each): bf16 [192,512,64] x 512 with its mask takes 74 us, 4.4 TB/s of what has to move; as a contraction and a row kernel 149 us,
 * the float32 scores written and read in between. Measured and left out: the mask requested in front of the MFMAs (77 us
 * either way, more registers: 2048 columns 201 us for 174), non-temporal loads of it (86 us), non-temporal stores (79 us).
 */
#pragma once

namespace akg {

// Unit j of wavefront wc: neighbouring units in pairs where their number is even, so that the 16-bit results of a pair
// fill a whole cache line from one wavefront.
template <int NCHUNK, int WC>
AKG_DEV constexpr int row_unit(int j, int wc) {
  return NCHUNK % 2 == 0 ? ((j / 2) * WC + wc) * 2 + j % 2 : j * WC + wc;
}

// Two loads of 16 bytes a lane that touch whole lines of eight rows each: in the first, the lanes c = lane % 16 below 8 have piece p of row c,
// the others piece q of row c - 8; in the second piece p of row c + 8 and piece q of row c. Afterwards `first` is piece p and `second` piece
// q of the lane's own row c. (Rows of their own in either load, all sixteen of them half a line each, take twice as many of a CU's
// requests.)
AKG_DEV void own_row_pieces(v4i &first, v4i &second) {
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const int f = first[e], s = second[e];
    first[e] = __builtin_amdgcn_update_dpp(f, s, 0x128, 0xF, 0xC, false);    // lanes 8 .. 15 take from the lane 8 below
    second[e] = __builtin_amdgcn_update_dpp(s, f, 0x128, 0xF, 0x3, false);   // lanes 0 .. 7 from the lane 8 above
  }
}

// load_chunk_if of the eight adjacent 32-bit columns of the lane's own row, by whole lines: `low` is the index of these columns in the row
// of lane c % 8 of the sixteen, `high` in that of lane c % 8 + 8.
template <typename DT>
AKG_DEV void load_own_row_if(Buffer buf, bool ok, long low, long high, int lane, typename DT::compute (&dst)[8]) {
  typedef typename DT::storage S;
  static_assert(sizeof(S) == 4, "a chunk is two pieces");
  typedef BufferIo<16, kAuxDefault> Io;
  const u32 piece = 16u * ((static_cast<u32>(lane) >> 3) & 1u);
  v4i p = __builtin_bit_cast(v4i, Io::load(buf, ok ? static_cast<u32>(low) * 4u + piece : kBeyondEveryBuffer));
  v4i q = __builtin_bit_cast(v4i, Io::load(buf, ok ? static_cast<u32>(high) * 4u + piece : kBeyondEveryBuffer));
  own_row_pieces(p, q);
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const int a = p[e], b = q[e];
    dst[e] = DT::load(__builtin_bit_cast(S, a));
    dst[4 + e] = DT::load(__builtin_bit_cast(S, b));
  }
}

// A number (of 64-byte slabs of K) as a type.
template <int N>
struct SlabCount {
  static constexpr int value = N;
};

// s[rt][j] = the eight columns of unit row_unit(j, wc) (columns beyond N hold copies of column N - 1) in row
// row0 + 16 rt + lane % 16 (rows beyond M hold copies of row M - 1). KB: bytes of K per row, a multiple of 64. LINES: two slabs of K at a
// time from whole lines of B.
// Up to seven slabs of 64 bytes the rows of A stay in registers; a longer K is taken in blocks of four with the
// accumulators live, so the registers do not grow with K (bf16, 512 x 256 with softmax: 200 a lane at K = 512, 332 with all of K
// held, where K = 1024 and more spilled; K = 512 50 us either way, and the next block's rows requested beside the MFMAs of a block
// gave nothing).
template <typename Mma, long M, long N, long KB, int RT, int NCHUNK, int WC, bool LINES>
AKG_DEV void row_scores(const void *__restrict__ A, const void *__restrict__ B, long row0, int wc, int lane,
                        float (&s)[RT][NCHUNK][8]) {
  static_assert(KB % 64 == 0 && M * KB < (1L << 31) && N * KB < (1L << 31), "operand shapes of the fragments");
  constexpr int kSlabs = static_cast<int>(KB / 64);
  constexpr int kBlock = kSlabs <= 7 ? kSlabs : 4, kBlocks = kSlabs / kBlock, kRest = kSlabs % kBlock;
  const int c = lane & 15, g = lane >> 4;
  const char *a = static_cast<const char *>(A);
  const char *b = static_cast<const char *>(B);
  u32 aOff[RT];
#pragma unroll
  for (int rt = 0; rt < RT; ++rt) {
    const long row = row0 + 16 * rt + c;
    aOff[rt] = static_cast<u32>((row < M ? row : M - 1) * KB) + 16u * static_cast<u32>(g);
  }
  v4i qf[RT][kBlock];
  auto loadRows = [&](auto slabs, u32 at) {
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) {
#pragma unroll
      for (int i = 0; i < slabs.value; ++i) qf[rt][i] = *reinterpret_cast<const v4i *>(a + aOff[rt] + at + 64 * i);
    }
  };
  // The fragments of kBatch units are requested together, in front of their MFMAs (left alone, the compiler keeps two
  // loads in flight and the wavefront waits out the L2 once per MFMA).
  auto multiply = [&](auto slabs, u32 at, auto first) {   // (into s, which the first block starts)
    constexpr int kCount = slabs.value, kBatch = kCount >= 8 ? 1 : 8 / kCount;
#pragma unroll
    for (int j0 = 0; j0 < NCHUNK; j0 += kBatch) {
      v4i kf[kBatch][2][kCount];
#pragma unroll
      for (int j = j0; j < j0 + kBatch && j < NCHUNK; ++j) {
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          auto offsetOf = [&](int cc) {
            long col = 32L * row_unit<NCHUNK, WC>(j, wc) + 8 * (cc >> 2) + 4 * h + (cc & 3);
            if constexpr (N % (32L * WC) != 0) col = col < N ? col : N - 1;
            return static_cast<u32>(col * KB) + 16u * static_cast<u32>(g) + at;
          };
          constexpr int kPaired = LINES ? kCount / 2 * 2 : 0;   // eight columns a load, own_row_pieces below; the others sixteen
          if constexpr (kPaired > 0) {
            const u32 half = 64u * static_cast<u32>(c >> 3), low = offsetOf(c & 7) + half, high = offsetOf((c & 7) + 8) + half;
#pragma unroll
            for (int i = 0; i < kPaired; i += 2) {
              kf[j - j0][h][i] = *reinterpret_cast<const v4i *>(b + low + 64 * i);
              kf[j - j0][h][i + 1] = *reinterpret_cast<const v4i *>(b + high + 64 * i);
            }
          }
          if constexpr (kPaired < kCount) {
            const u32 off = offsetOf(c);
#pragma unroll
            for (int i = kPaired; i < kCount; ++i) kf[j - j0][h][i] = *reinterpret_cast<const v4i *>(b + off + 64 * i);
          }
        }
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int j = j0; j < j0 + kBatch && j < NCHUNK; ++j) {
        if constexpr (LINES) {
#pragma unroll
          for (int h = 0; h < 2; ++h) {
#pragma unroll
            for (int i = 0; i + 1 < kCount; i += 2) own_row_pieces(kf[j - j0][h][i], kf[j - j0][h][i + 1]);
          }
        }
#pragma unroll
        for (int rt = 0; rt < RT; ++rt) {
#pragma unroll
          for (int h = 0; h < 2; ++h) {
            typename Mma::acc4_v acc = {0, 0, 0, 0};
            const float *sum = s[rt][j] + 4 * h;
            if constexpr (first.value == 0) acc = typename Mma::acc4_v{sum[0], sum[1], sum[2], sum[3]};
#pragma unroll
            for (int i = 0; i < kCount; ++i) acc = Mma::mma16(kf[j - j0][h][i], qf[rt][i], acc);
#pragma unroll
            for (int v = 0; v < 4; ++v) s[rt][j][4 * h + v] = acc[v];
          }
        }
      }
    }
  };
  loadRows(SlabCount<kBlock>(), 0);
  multiply(SlabCount<kBlock>(), 0, SlabCount<1>());
#pragma unroll 1
  for (int t = 1; t < kBlocks; ++t) {
    const u32 at = static_cast<u32>(t) * (64 * kBlock);
    loadRows(SlabCount<kBlock>(), at);
    multiply(SlabCount<kBlock>(), at, SlabCount<0>());
  }
  if constexpr (kRest > 0) {
    loadRows(SlabCount<kRest>(), 64 * kBlock * kBlocks);
    multiply(SlabCount<kRest>(), 64 * kBlock * kBlocks, SlabCount<0>());
  }
}

// One value per row from the lanes' partial values: the four lanes of a row, then its WC wavefronts through `slots`
// (every reduction of a kernel has slots of its own, so one barrier each is enough).
template <typename Red, int WC, typename T>
AKG_DEV T row_scores_reduce(T v, T (*slots)[16], int wc, int lane) {
  v = Red::apply(v, lane_partner<16>(v));
  v = Red::apply(v, lane_partner<32>(v));
  if constexpr (WC > 1) {
    if (lane < 16) slots[wc][lane] = v;
    __syncthreads();
    T r = slots[0][lane & 15];
#pragma unroll
    for (int w = 1; w < WC; ++w) r = Red::apply(r, slots[w][lane & 15]);
    return r;
  }
  return v;
}

}  // namespace akg
