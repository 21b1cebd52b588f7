// engine_mfma128.hpp -- 128x128 fp32 output tile on the gfx950 matrix cores,
// fed by a 3-stage LDS ring of buffer_load_dwordx4 ... lds (direct-to-LDS, no
// VGPR staging).
//
// The fp32 matrix instructions give 157 TFLOP/s, the bf16 ones sixteen times
// that. Each operand is therefore split into three bf16 parts, x = hi + mid +
// lo, every part the round-to-nearest bf16 of what the former leave: 24
// significand bits in all, so x is represented exactly down to bf16's last bit
// (2^-133; the conversions and v_mfma_f32_32x32x16_bf16 keep denormals, in
// operands, products and sums). A product is the sum
// of the six part products down to 2^-16 of hi.hi (the three left out are
// below 2^-24 of it), accumulated in fp32 by v_mfma_f32_32x32x16_bf16, which
// rounds once per 8 products where the fp32 instructions round at every one.
// Error against 64 bits, uniform [-1, 1) operands, K = 256 / 992 / 4096:
// 2.3e-7 / 4.8e-7 / 1.0e-6 (fp32 chain 2.9e-7 / 5.6e-7 / 1.1e-6). Operands
// spread over 2^-30 .. 2^30, K = 64 / 992: 6.0e-8 / 2.2e-7 (5.1e-8 / 1.7e-7).
// The three-part split is that of Henry, Tang and Heinecke, "Leveraging the
// bfloat16 Artificial Intelligence Datatype For Higher-Precision Computations"
// (2019).
// What the parts cannot carry is computed with exact fp32 products instead
// (compute_exact, at the fp32 matrix rate and with the same poll sites):
//  - from the first k-stage on that holds an operand with bits below 2^-133
//    (below 2^-110, that is), which its parts lose, to the end of the tile;
//  - a tile that ends with an infinite or NaN accumulator (an operand or a sum
//    that is infinite, NaN, or above bf16's largest value), from k = 0.
// Both are decided by the tile's operands alone, so a tile's result does not
// depend on where it was checkpointed. 4096^3, with fp32 products throughout
// 975 us: ordinary operands 790, softmax weights (two fifths of them below
// 2^-110) 1037, all 1e-35 1020, one small operand per panel in the middle of K
// 880; an infinity at k = 0 1060-1100, a NaN at the end of K 1740 (both passes).
//
// Block: 256 threads = 4 wave64s in a 2x2 arrangement; each wave owns a
// 64x64 sub-tile held as 2x2 32x32 accumulators (64 VGPRs per lane).
// Stage: k depth KS=32 -> A stage 128x32 fp32 (16 KiB) + B stage 32x128 fp32
// (16 KiB); 3 stages = 96 KiB of the 160 KiB LDS, and 48 KiB of split operands
// (planes): 1 block per CU.
//
// What bounds it: a 16-deep k-step is 24 MFMAs per wave (768 matrix cycles)
// and, with each operand split once per block, 16 values per lane to split
// (6.5 vector instructions each). At 4096^3 it takes about 1.75 K cycles at
// 2.25 GHz: a wave issues in order, one per SIMD, and meets the LDS traffic of
// the planes (18 instructions per wave and step); without them 1.2 K, at 2.0
// GHz (the package then limits the clock). Splitting in every wave for itself
// (no planes, twice the vector work) is no faster, and 6% slower with polls.
// 4096^3: 970 -> 775-825 us, card by card; 1920x1408x992: 80 -> 54 (with the
// queue's part); 8192x8192x4096 with chunk polls: 4140 -> 3,280-3,330.
//
// LDS layouts (bank-conflict-free):
//  A stage: 128 rows x 128 B. 16-byte quad q of row r is stored at slot
//           q ^ aswz(r), aswz(r) = (r ^ ((r >> 3) & 1)) & 7: 8 (or 16)
//           consecutive rows reading the same quad hit 8 (16) different
//           16-byte bank groups, whether the LDS serves 128 B or 256 B per
//           cycle.
//  B stage: 32 rows x 512 B; 16-byte chunk c of row k is stored at slot
//           c ^ (((k >> 2) & 1) << 3). An operand read is 32 consecutive
//           dwords of row k for the lower half-wave and of row k+4 for the
//           upper one; the XOR moves the upper half by 128 B, so the two
//           halves never share a bank even when all 64 lanes are served in
//           one cycle.
//  planes:  a k-step's split operands, per 32-row block (0-3 of A, 4-7 of B)
//           and part 64 lanes x 16 B, in the lane order of the MFMA operand:
//           written and read by whole waves at 16 bytes per lane.
//
// k order: a k-step is two k-groups of 8; the lower half-wave supplies k =
// 0-3 of both, the upper one k = 4-7. The order is fixed, so a tile's result
// is a deterministic function of its inputs whatever worker computes it and
// however often it is checkpointed and resumed.
#pragma once
#include "device.hpp"

namespace apk {

typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
typedef float f32x2 __attribute__((ext_vector_type(2)));

struct EngMfma128 {
  static constexpr int TM = 128, TN = 128, KS = 32, NS = 3, GROUP = 1, THREADS = 256;
  // Waves per SIMD at most (1 block per CU (LDS-bound)): the register budget the
  // compiler may schedule for.
  static constexpr int WAVES_PER_SIMD = 1, BLOCKS_PER_CU = 1;
  static constexpr int MIN_WAVES_PER_SIMD = 1;  // occupancy the registers must allow
  static constexpr int A_STAGE = TM * KS * 4;               // bytes
  static constexpr int B_STAGE = KS * TN * 4;               // bytes
  static constexpr int STAGE = A_STAGE + B_STAGE;           // 32 KiB
  // The split operands of two k-steps (planes), behind the ring.
  static constexpr int BLOCK_PLANES = 3 * 64 * 16;          // one 32-row block: 3 KiB
  static constexpr int PLANES = 8 * BLOCK_PLANES;           // a k-step's: 24 KiB
  static constexpr int LDS_BYTES = NS * STAGE + 2 * PLANES; // 144 KiB
  static constexpr int LOADS_A = A_STAGE / (THREADS * 16);  // 4 per thread
  static constexpr int LOADS_B = B_STAGE / (THREADS * 16);  // 4 per thread
  static constexpr int LOADS = LOADS_A + LOADS_B;           // per stage
  static constexpr int ACC_PER_THREAD = 64;                 // floats
  static constexpr int ELEM_BYTES = 4;                      // fp32 operands
  // Epilogue: the whole tile is staged in LDS in one pass (row stride TN).
  static constexpr int STORE_PASSES = 1, PASS_ROWS = TM, STAGE_LD = TN;

  struct Acc {
    f32x16 c[2][2];
  };

  static __device__ __forceinline__ int aswz(int r) { return (r ^ ((r >> 3) & 1)) & 7; }
  static __device__ __forceinline__ int bswz(int k) { return ((k >> 2) & 1) << 3; }

  struct Ctx {
    i32x4 ra, rb;
    int K, N;
  };

  static __device__ __forceinline__ Ctx make_ctx(const void* A, const void* B,
                                                 int M, int N, int K) {
    Ctx c;
    c.ra = make_rsrc(A, (uint32_t)((size_t)M * K * 4));
    c.rb = make_rsrc(B, (uint32_t)((size_t)K * N * 4));
    c.K = K;
    c.N = N;
    return c;
  }

  static __device__ __forceinline__ void zero(Acc& a) {
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int r = 0; r < 16; ++r) a.c[i][j][r] = 0.0f;
  }

  // Direct-to-LDS loads of one k-stage. A load i (< 4) fills the 1 KiB
  // piece i*4 + wave of the A stage: rows 32*i + 8*wave + lane/8, quad slot
  // lane%8. B load i fills rows 8*i + 2*wave + lane/32, chunk slot lane%32.
  // Neither swizzle depends on the row bits that i changes, so each lane's
  // offset of load i is fixed per tile (Lane, one register per load) and
  // stage s only adds scalar offsets.
  struct Lane {
    uint32_t a[LOADS_A], b[LOADS_B];
  };
  static __device__ __forceinline__ Lane lane_offsets(const Ctx& c, int row0, int col0) {
    const int w = wave_id(), l = lane_id();
    const int ra = w * 8 + (l >> 3);
    const int qa = (l & 7) ^ aswz(ra);
    const int rb = w * 2 + (l >> 5);
    const int cq = (l & 31) ^ bswz(rb);
    const uint32_t a0 = (uint32_t)(((row0 + ra) * c.K + 4 * qa) * 4);
    const uint32_t b0 = (uint32_t)((rb * c.N + col0 + 4 * cq) * 4);
    Lane ln;
#pragma unroll
    for (int i = 0; i < LOADS_A; ++i) ln.a[i] = a0 + (uint32_t)(i * 32) * (uint32_t)c.K * 4u;
#pragma unroll
    for (int i = 0; i < LOADS_B; ++i) ln.b[i] = b0 + (uint32_t)(i * 8) * (uint32_t)c.N * 4u;
    return ln;
  }
  // The scalar parts of the loads of stage t into ring slot `slot`, formed
  // once per stage: this wave's 1 KiB piece of the slot (LDS; wave_lds is
  // the piece in slot 0) and the byte offsets of k-stage t in A (along a
  // row) and B (down the rows).
  struct Dst {
    uint32_t lds, ka, kb;
  };
  // A stage past the tile's end (t >= S) fetches stage S-1 again: nothing
  // reads that slot before it is refilled.
  static __device__ __forceinline__ Dst stage_dst(uint32_t wave_lds, const Ctx& c, int slot,
                                                  int t, int S) {
    const uint32_t k0 = (uint32_t)((t < S ? t : S - 1) * KS);
    return Dst{wave_lds + (uint32_t)(slot * STAGE), k0 * 4u, k0 * (uint32_t)c.N * 4u};
  }
  // Byte offset inside a ring slot of load i's piece: thread t's 16 bytes of
  // load i land at slot + dma_lds_off(i) + 16 t.
  static constexpr uint32_t dma_lds_off(int i) {
    return (uint32_t)(i < LOADS_A ? i * 4096 : A_STAGE + (i - LOADS_A) * 4096);
  }
  static __device__ __forceinline__ void issue_one(const Ctx& c, const Lane& ln, const Dst& d,
                                                   int i) {
    if (i < LOADS_A)
      dma_x4(c.ra, d.lds, dma_lds_off(i), ln.a[i], d.ka);
    else
      dma_x4(c.rb, d.lds, dma_lds_off(i), ln.b[i - LOADS_A], d.kb);
  }

  // Operands of k-group g (8 k values): one 16-byte A read per 32-row
  // block (the quad 2g+h of the lane's row), four B dwords per 32-column
  // block (compute_exact). The wave's blocks are numbered so that block 0 of A is another
  // one for its neighbour in the column, and block 0 of B for its neighbour
  // in the row (arow, bcol): each wave splits its blocks 0, and together the
  // four split every operand once.
  struct Frag {
    f32x4 a4[2];
    float bv[2][4];
  };
  static __device__ __forceinline__ int arow(int rb) {
    const int w = threadIdx.x >> 6;
    return (w & 1) * 64 + (rb ^ (w >> 1)) * 32;
  }
  static __device__ __forceinline__ int bcol(int cb) {
    const int w = threadIdx.x >> 6;
    return (w >> 1) * 64 + (cb ^ (w & 1)) * 32;
  }
  static __device__ __forceinline__ void load_frag(const char* abase, int g, Frag& f) {
    const int l = lane_id();
    const int lr = l & 31, h = l >> 5;
    const float* bbase = (const float*)(abase + A_STAGE);
#pragma unroll
    for (int rb = 0; rb < 2; ++rb) {
      const int row = arow(rb) + lr;
      const int q = (2 * g + h) ^ aswz(row);
      f.a4[rb] = *(const f32x4*)(abase + row * 128 + q * 16);
    }
    // Row k = 8g + 4h + s has bswz(k) = h << 3 for every s.
#pragma unroll
    for (int cb = 0; cb < 2; ++cb) {
      const int col = bcol(cb) + lr;
      const int cpos = (((col >> 2) ^ (h << 3)) << 2) | (col & 3);
#pragma unroll
      for (int s = 0; s < 4; ++s) f.bv[cb][s] = bbase[(8 * g + 4 * h + s) * TN + cpos];
    }
  }

  // A k-step is two k-groups (16 k). Its operands are split: x = hi + mid +
  // lo, each the round-to-nearest bf16 of what the former leave (24
  // significand bits in all), eight k values of a row (column) per lane --
  // the operand layout of v_mfma_f32_32x32x16_bf16, k in the order of the
  // two groups. A wave splits its own blocks (A's block 0 and B's block 0)
  // and takes the other two from the waves beside it, through LDS.
  struct Own {
    u32x4 a[3], b[3];  // 0 hi, 1 mid, 2 lo
  };
  struct Raw {
    f32x4 a[2];
    float b[8];
  };
  static constexpr int STEPS = KS / 16;       // k-steps per stage
  static constexpr int MF = 24;               // MFMAs of a step per wave
  static __device__ __forceinline__ void load_raw(const char* abase, int j, Raw& r) {
    const int l = lane_id();
    const int lr = l & 31, h = l >> 5;
    const float* bbase = (const float*)(abase + A_STAGE);
    const int row = arow(0) + lr, col = bcol(0) + lr;
    const int cpos = (((col >> 2) ^ (h << 3)) << 2) | (col & 3);
#pragma unroll
    for (int g = 0; g < 2; ++g)
      r.a[g] = *(const f32x4*)(abase + row * 128 + (((2 * (2 * j + g) + h) ^ aswz(row)) << 4));
#pragma unroll
    for (int g = 0; g < 2; ++g)
#pragma unroll
      for (int s = 0; s < 4; ++s) r.b[4 * g + s] = bbase[(16 * j + 8 * g + 4 * h + s) * TN + cpos];
  }
  // Splits the wave's blocks in 24 parts, three for each of 8 value pairs
  // (pairs 0-3 are A's, 4-7 B's): part 0 of a pair gives hi and what it
  // leaves, part 1 mid, part 2 lo. One part goes under each MFMA: five vector
  // instructions fit the 32 cycles of one, while more in a row, or two
  // MFMAs in a row, leave one of the two units idle (a wave issues in
  // order).
  struct Rest {
    float x0, x1;
  };
  // `seen` collects what the lowest parts were rounded from (lossy).
  static __device__ __forceinline__ void split_part(const Raw& r, int part, Own& d, Rest& rest,
                                                    unsigned& seen) {
    const int p = part / 3, e = 2 * (p & 3);  // elements e, e + 1
    u32x4* o = p < 4 ? d.a : d.b;
    if (part % 3 == 0) {
      const float x0 = p < 4 ? r.a[e >> 2][e & 3] : r.b[e];
      const float x1 = p < 4 ? r.a[e >> 2][(e & 3) + 1] : r.b[e + 1];
      const unsigned hi = pack(x0, x1);
      rest = Rest{x0 - low(hi), x1 - high(hi)};
      o[0][p & 3] = hi;
    } else if (part % 3 == 1) {
      const unsigned mid = pack(rest.x0, rest.x1);
      rest = Rest{rest.x0 - low(mid), rest.x1 - high(mid)};
      o[1][p & 3] = mid;
    } else {
      o[2][p & 3] = pack(rest.x0, rest.x1);
      seen |= __float_as_uint(rest.x0) | __float_as_uint(rest.x1);
    }
  }
  // This lane's 16 bytes of plane 0 of block `blk` (0-3 A's rows, 4-7 B's
  // columns) of k-step buffer `buf`; planes 1 and 2 follow 1 KiB apart.
  static __device__ __forceinline__ char* plane(char* ring, int buf, int blk) {
    return ring + NS * STAGE + buf * PLANES + blk * BLOCK_PLANES + lane_id() * 16;
  }
  static __device__ __forceinline__ int ablock(int rb) { return arow(rb) >> 5; }
  static __device__ __forceinline__ int bblock(int cb) { return 4 + (bcol(cb) >> 5); }
  static __device__ __forceinline__ void put(char* dst, const u32x4 (&v)[3]) {
#pragma unroll
    for (int i = 0; i < 3; ++i) *(u32x4*)(dst + i * 1024) = v[i];
  }
  static __device__ __forceinline__ void take(const char* src, u32x4 (&v)[3]) {
#pragma unroll
    for (int i = 0; i < 3; ++i) v[i] = *(const u32x4*)(src + i * 1024);
  }
  // Two values rounded to bf16 (one v_cvt_pk_bf16_f32), and back.
  static __device__ __forceinline__ unsigned pack(float x0, float x1) {
    const f32x2 v = {x0, x1};
    return __builtin_bit_cast(unsigned, __builtin_convertvector(v, bf16x2));
  }
  static __device__ __forceinline__ float low(unsigned u) { return __uint_as_float(u << 16); }
  static __device__ __forceinline__ float high(unsigned u) {
    return __uint_as_float(u & 0xffff0000u);
  }
  // MFMA m (< 24) of a k-step. Blocks in the order (own, own), (own, other),
  // (other, own), (other, other), each with its six products in ascending
  // size: mid.mid, lo.hi, hi.lo, mid.hi, hi.mid, hi.hi (the three left out
  // are below 2^-24 of hi.hi). The wave's own come first: the others' planes
  // arrive from LDS under them.
  static __device__ __forceinline__ void mma(const Own& own, const Own& other, int m, Acc& acc) {
    constexpr int PA[6] = {1, 2, 0, 1, 0, 0}, PB[6] = {1, 0, 2, 0, 1, 0};
    const int t = m % 6, rb = m / 12, cb = m / 6 & 1;
    const u32x4 a = (rb ? other : own).a[PA[t]], b = (cb ? other : own).b[PB[t]];
    acc.c[rb][cb] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
        __builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), acc.c[rb][cb], 0, 0, 0);
  }

  // The k-steps are software-pipelined three deep, across the stage barriers:
  // with one wave per SIMD nothing else covers an LDS round trip or a chain
  // of conversions. A phase runs the MFMAs of one k-step while it splits the
  // wave's own blocks of the next (read from the ring a phase earlier), puts
  // them into the planes, and reads the blocks of the one after; a barrier
  // later every wave takes the others' from the planes. What is left over
  // from one call to the next: the own split blocks of a step whose MFMAs are
  // to come (the others' lie in planes 0 by the next barrier) and the blocks
  // of the step after it, not yet split.
  struct Tail {
    Own own;
    Raw raw;
  };
  // How a tile is computed: with parts; from some stage on with exact
  // products; with exact products throughout. And what the stage whose MFMAs
  // are next turned out to be: LOSSY, it holds an operand that is more than
  // its parts; BROKEN, an accumulator is infinite or NaN already.
  enum { SPLIT = 0, EXACT_REST = 1, EXACT = 2 };
  enum { FINE = 0, LOSSY = 1, BROKEN = 2 };

  // Whether this lane's operands of a stage are more than their parts. Its
  // first k-step has been split: bf16 is the upper half of fp32, so lo is
  // exact where the lower half of what it was rounded from (`seen`) is zero.
  // The second has only been read (its MFMAs, like the first's, come after
  // the next barrier, and the stage's slot is refilled after that): `least`
  // is the smallest of 2 |x| - 1 as an integer, where a zero wraps to the
  // largest, and 2^-110 the smallest normal value without bits below 2^-133.
  static constexpr unsigned LEAST = 2u * ((127 - 110) << 23) - 1;
  static __device__ __forceinline__ bool lossy(unsigned seen, unsigned least) {
    return (seen & 0xffffu) != 0 || least < LEAST;
  }
  static __device__ __forceinline__ void watch(const Raw& r, int p, unsigned& least) {
    const int e = 2 * (p & 3);
    const unsigned x0 = __float_as_uint(p < 4 ? r.a[e >> 2][e & 3] : r.b[e]);
    const unsigned x1 = __float_as_uint(p < 4 ? r.a[e >> 2][(e & 3) + 1] : r.b[e + 1]);
    const unsigned t0 = 2 * x0 - 1, t1 = 2 * x1 - 1;
    const unsigned t = t0 < t1 ? t0 : t1;
    least = t < least ? t : least;
  }
  // A lane of the block marks stage s: verdict[s & 1] (LDS, both words zero
  // when the tile starts) is read after the next barrier. Two words: a wave
  // ahead of the others marks stage s + 1 while they still read s's.
  // Every 16 stages it also looks for a sum that is no longer finite, so that
  // a tile of infinite or NaN operands does not run to its end first: one
  // register per column block and every one of column block 0 meet any row
  // or column of them.
  static __device__ __forceinline__ void mark(int* verdict, int s, unsigned seen, unsigned least,
                                              const Acc& acc) {
    if (lossy(seen, least)) verdict[s & 1] = LOSSY;
    if ((s & 15) == 15) {
      float z = acc.c[0][1][0] * 0.0f;
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int r = 0; r < 16; ++r) z = fmaf(acc.c[i][0][r], 0.0f, z);
      if (!(z == 0.0f)) verdict[s & 1] = BROKEN;
    }
  }
  // Stage s's verdict, after the barrier that follows its call (uniform).
  static __device__ __forceinline__ int verdict_of(const int* verdict, int s) {
    return uniform(verdict[s & 1]);
  }

  static __device__ __forceinline__ void take_other(const char* ring, int buf, Own& other) {
    take(plane(const_cast<char*>(ring), buf, bblock(1)), other.b);
    take(plane(const_cast<char*>(ring), buf, ablock(1)), other.a);
    __builtin_amdgcn_sched_barrier(0);
  }
  // The MFMAs of the step whose blocks are `cur` and `other`; under MFMA m part
  // m of `raw` is split into `next` and planes `buf` (SPLIT_NEXT), `at(m)`
  // runs, and `mid(i)`, i = lo..lo+3, issues loads (four of them).
  template <bool SPLIT_NEXT, class At, class Mid>
  static __device__ __forceinline__ void phase(char* ring, int buf, const Own& cur,
                                               const Own& other, const Raw& raw, Own& next,
                                               unsigned& seen, Acc& acc, At&& at, int lo,
                                               Mid&& mid) {
    Rest rest;
#pragma unroll
    for (int m = 0; m < MF; ++m) {
      mma(cur, other, m, acc);
      __builtin_amdgcn_sched_barrier(0);
      if constexpr (SPLIT_NEXT) split_put(ring, buf, raw, m, next, rest, seen);
      at(m);
      __builtin_amdgcn_sched_barrier(0);
      if (m % 5 == 4 && m / 5 < LOADS / 2) {
        mid(lo + m / 5);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
  }
  // Part `part`; a block goes to the planes once its last part is done.
  static __device__ __forceinline__ void split_put(char* ring, int buf, const Raw& raw, int part,
                                                   Own& d, Rest& rest, unsigned& seen) {
    split_part(raw, part, d, rest, seen);
    if (part == 11) put(plane(ring, buf, ablock(0)), d.a);
    if (part == 23) put(plane(ring, buf, bblock(0)), d.b);
    __builtin_amdgcn_sched_barrier(0);
  }
  // Stage s in ring slot `slot` enters the empty pipeline. `mid(i)`, i =
  // 0..LOADS-1, issues the loads of a later stage.
  template <class Mid>
  static __device__ __forceinline__ void enter(char* ring, int slot, int s, const Acc& acc,
                                               Tail& t, int* verdict, Mid&& mid) {
    const char* abase = ring + slot * STAGE;
    Raw raw;
    Rest rest;
    unsigned seen = 0, least = ~0u;
    load_raw(abase, 0, raw);
    load_raw(abase, 1, t.raw);
#pragma unroll
    for (int i = 0; i < LOADS; ++i) mid(i);
#pragma unroll
    for (int p = 0; p < MF; ++p) split_put(ring, 0, raw, p, t.own, rest, seen);
#pragma unroll
    for (int p = 0; p < 8; ++p) watch(t.raw, p, least);
    mark(verdict, s, seen, least, acc);
  }
  // Stage s in ring slot `slot` enters the pipeline and the two steps of stage
  // s - 1, which must be FINE, leave it; `other`: the first step's blocks from
  // planes 0 (take_other; its reads also cover the way of that stage's verdict,
  // read from LDS ahead of them). `mid`'s loads are spread over the MFMAs.
  // Looking for lossy stages costs 4096^3 0.7%, a 256^3 urgent job 14.0 -> 14.4
  // us.
  template <class Mid>
  static __device__ __forceinline__ void stage(char* ring, int slot, int s, Own& other, Acc& acc,
                                               Tail& t, int* verdict, Mid&& mid) {
    static_assert(STEPS == 2 && LOADS == 8, "two phases per stage, four loads each");
    const char* abase = ring + slot * STAGE;
    Raw raw;
    Own odd;
    unsigned seen = 0, unused = 0, least = ~0u;
    phase<true>(ring, 1, t.own, other, t.raw, odd, unused, acc,
                [&](int m) { if (m == 6) load_raw(abase, 0, raw); }, 0, mid);
    lds_sync();
    take_other(ring, 1, other);
    phase<true>(ring, 0, odd, other, raw, t.own, seen, acc,
                [&](int m) {
                  if (m == 6) load_raw(abase, 1, t.raw);
                  if (m >= 9 && m % 2) watch(t.raw, (m - 9) / 2, least);
                },
                4, mid);
    mark(verdict, s, seen, least, acc);
  }
  // The two steps left over of a stage, before the accumulators are read: after
  // a barrier (every wave's planes), and if the stage is FINE.
  static __device__ __forceinline__ void finish_tail(char* ring, Acc& acc, const Tail& t) {
    Own odd, other;
    unsigned unused = 0;
    take_other(ring, 0, other);
    phase<true>(ring, 1, t.own, other, t.raw, odd, unused, acc, [](int) {}, 0, [](int) {});
    lds_sync();
    take_other(ring, 1, other);
    phase<false>(ring, 0, odd, other, t.raw, odd, unused, acc, [](int) {}, 0, [](int) {});
  }

  // Whether an accumulator of this lane is infinite or NaN.
  static __device__ __forceinline__ bool broken(const Acc& a) {
    float z[2] = {0.0f, 0.0f};
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int r = 0; r < 16; ++r) z[j] = fmaf(a.c[i][j][r], 0.0f, z[j]);
    return !(z[0] + z[1] == 0.0f);
  }
  // One k-stage with the exact fp32 products of v_mfma_f32_32x32x2_f32. The
  // operands of group g+1 are read from LDS while group g's MFMAs run;
  // `mid(i)`, i < LOADS, issues a later stage's loads under the first ones.
  template <class Mid>
  static __device__ __forceinline__ void compute_exact(const char* ring, int slot, Acc& acc,
                                                       Mid&& mid) {
    const char* abase = ring + slot * STAGE;
    constexpr int GG = KS / 8;
    Frag f[2];
    load_frag(abase, 0, f[0]);
#pragma unroll
    for (int g = 0; g < GG; ++g) {
      if (g + 1 < GG) load_frag(abase, g + 1, f[(g + 1) & 1]);
      __builtin_amdgcn_sched_barrier(0);
      const Frag& c = f[g & 1];
#pragma unroll
      for (int m = 0; m < 16; ++m) {
        const int s = m >> 2, rb = (m >> 1) & 1, cb = m & 1;
        acc.c[rb][cb] = __builtin_amdgcn_mfma_f32_32x32x2f32(c.a4[rb][s], c.bv[cb][s],
                                                             acc.c[rb][cb], 0, 0, 0);
        if ((m & 1) && g * 8 + (m >> 1) < LOADS) {
          __builtin_amdgcn_sched_barrier(0);
          mid(g * 8 + (m >> 1));
          __builtin_amdgcn_sched_barrier(0);
        }
      }
    }
  }

  // Output element (tile-relative row, col) of accumulator register e.
  static __device__ __forceinline__ void coord(int e, int& r, int& c) {
    const int l = lane_id();
    const int rb = e >> 5, cb = (e >> 4) & 1, q = e & 15;
    r = arow(rb) + 8 * (q >> 2) + 4 * (l >> 5) + (q & 3);
    c = bcol(cb) + (l & 31);
  }
  static __device__ __forceinline__ float get(const Acc& a, int e) {
    return a.c[e >> 5][(e >> 4) & 1][e & 15];
  }
  static __device__ __forceinline__ void set(Acc& a, int e, float v) {
    a.c[e >> 5][(e >> 4) & 1][e & 15] = v;
  }

  // The C tile straight from the accumulators: a register holds, in each
  // half-wave, 32 consecutive columns of one row, so one dword store writes
  // two whole 128-byte row segments, with no LDS and no barrier:
  // 256^3 urgent 14.7 -> 14.0 us, 4096^3 804 -> 778.
  // (A fingerprinted tile is staged in LDS instead.)
  static __device__ __forceinline__ void store_direct(const Acc& acc, float* C, int ldc,
                                                      int row0, int col0) {
    const int l = lane_id();
#pragma unroll
    for (int rb = 0; rb < 2; ++rb)
#pragma unroll
      for (int cb = 0; cb < 2; ++cb) {
        float* base = C + (size_t)(row0 + arow(rb) + 4 * (l >> 5)) * ldc + col0 + bcol(cb) + (l & 31);
#pragma unroll
        for (int q = 0; q < 16; ++q) base[(size_t)(8 * (q >> 2) + (q & 3)) * ldc] = acc.c[rb][cb][q];
      }
  }

  // Write the accumulators into LDS as the row-major TM x TN tile (the ring
  // is free once a tile's last stage has been computed).
  static __device__ __forceinline__ int pass_row(int, int rr) { return rr; }
  static __device__ __forceinline__ void stage_pass(const Acc& acc, char* lds, int) {
    const int l = lane_id();
    const int lr = l & 31, h = l >> 5;
    float* t = (float*)lds;
#pragma unroll
    for (int rb = 0; rb < 2; ++rb)
#pragma unroll
      for (int cb = 0; cb < 2; ++cb)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int row = arow(rb) + 8 * (r >> 2) + 4 * h + (r & 3);
          t[row * TN + bcol(cb) + lr] = acc.c[rb][cb][r];
        }
  }
};

}  // namespace apk
