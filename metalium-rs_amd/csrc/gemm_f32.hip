// F32 products at F32 precision, operands moved HBM -> LDS by DMA.
//
// Reference: Engine::matmul_dram / matmul_dram_batched over F32 operands
// (crates/burn-tt/src/server.rs:178-239).
//
// Two ways to multiply, by the size of a block's tile:
//  * 64 x 64 (a wavefront's 32 x 32) on v_mfma_f32_32x32x2f32, two k a
//    64-cycle instruction: the chip's 157 TF/s.  A k-tile of 32 is 1024 cycles
//    of it, less than a load from HBM takes, so `global_load_lds` fills NS LDS
//    stages ahead: NS - 1 k-tiles in flight, no staging registers, no LDS
//    stores, one barrier a k-tile.  The choice where blocks are few: a short
//    chain of latencies.
//  * 64 x 128 and 128 x 128 on v_mfma_f32_32x32x16_bf16: each value, read from
//    LDS, is split in registers into three BF16 parts (24 bits in all) and a
//    product taken as six of the nine part products, the others at most 2^-24
//    of it together: 6 x 32 cycles for 16 k against 512.  The 14 vector
//    operations a pair of values run between the MFMAs of the step before.  Two
//    blocks a CU, each two LDS stages: one's barrier and epilogue under the
//    other's products.
//
// us, against the register-staged 64 x 64 / 128 x 128 kernel it replaces:
// 4096^3 (accurate mode) 1059 -> 747 (184 TF/s; 737 at best), 2048 x 8192 x 256
// 79 -> 59, [256, 8192] over k 2000 transposed 138 -> 69, 16 x 512^3 44.0 ->
// 32.2, 1500^3 128 -> 63, 512^3 15.4 -> 10.4, 64 x 128 x 784 12.7 -> 9.8.  The
// error against float64 falls at each (4096 x 4096 x 512 4.1e-7 -> 3.4e-7, 2048
// x 768 x 256 2.9e-7 -> 1.7e-7).
//
// LDS tiles.  An operand whose k is contiguous lies as 128-byte rows of 32 k
// in 16-byte chunks, chunk c of row r at c ^ (r / 2 & 7); a lane's fragment is one
// chunk (four k of its row).  One whose rows are contiguous lies as it is,
// [k][rows], a lane reading its row's four k one by one.  Lane l holds row l %
// 32 of a fragment and, of each 8 (16) k, the half l / 32.
//
// EDGE 0: whole tiles and k-tiles, 16-byte DMA.  1: any M, N and K, 16-byte
// DMA (contiguous extents in fours): each lane's address is clamped to the
// last row or chunk, and in the last k-tile lanes past K read zeros.  2: the
// same by 4-byte DMA, for operands of any pitch and alignment.
#include "gemm_args.hpp"

namespace mi {

// Lanes past K read here.
__device__ __constant__ float f32_zeros[4] = {0.0f, 0.0f, 0.0f, 0.0f};

typedef __attribute__((address_space(3))) void lds_ptr_t;

// One operand's tile of ROWS rows x 32 k: this wavefront's share of its DMA
// instructions (64 lanes of VEC floats each; instruction i of wavefront w is
// number i NW + w of the tile).
template <int ROWS, bool KC, int NW, int EDGE>
struct F32Operand {
  static constexpr int VEC = EDGE == 2 ? 1 : 4;
  static constexpr int BYTES = ROWS * 128;
  static constexpr int INSTR = ROWS * 32 / (64 * VEC);
  static constexpr int PER = INSTR / NW;
  static_assert(INSTR % NW == 0, "DMA instructions over the wavefronts");
  uint32_t voff[PER];  // this lane's byte offset from the tile's base, a k-tile's position apart
  const char *base;
  int64_t step;  // bytes a k-tile

  // 16 lanes' 16-byte reads are served together over the 64 banks: rows of
  // one parity share theirs, so the swizzle runs over pairs of rows.
  __device__ __forceinline__ static int swz(int r) { return (r >> 1) & 7; }

  // Lane's place in the tile: row and k.
  __device__ __forceinline__ static void place(int i, int wave, int lane, int &r, int &k) {
    const int o = ((i * NW + wave) * 64 + lane) * VEC;
    if constexpr (KC) {
      r = o / 32;
      const int q = o % 32;
      k = 4 * ((q >> 2) ^ swz(r)) + (q & 3);
    } else {
      k = o / ROWS;
      r = o % ROWS;
    }
  }

  __device__ __forceinline__ void init(const float *src, int64_t ld, int64_t r0, int64_t rows, int wave, int lane) {
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      int r, k;
      place(i, wave, lane, r, k);
      if constexpr (EDGE) {
        const int64_t last = rows - r0 - (KC ? 1 : VEC);
        if (r > last) r = static_cast<int>(last);
      }
      voff[i] = static_cast<uint32_t>((KC ? r * ld + k : k * ld + r) * 4);
    }
    base = reinterpret_cast<const char *>(src + (KC ? r0 * ld : r0));
    step = KC ? 128 : ld * 128;
  }

  // The DMA of k-tile kt into `lds`; krem: k left from its start (32 or more
  // but in the last).
  __device__ __forceinline__ void load(int64_t kt, int64_t krem, char *lds, int wave, int lane) const {
    const char *b = base + kt * step;
    const uint64_t gb =
        static_cast<uint64_t>(static_cast<uint32_t>(
            __builtin_amdgcn_readfirstlane(static_cast<int>(reinterpret_cast<uintptr_t>(b))))) |
        (static_cast<uint64_t>(__builtin_amdgcn_readfirstlane(static_cast<int>(reinterpret_cast<uintptr_t>(b) >> 32)))
         << 32);
    const uint32_t lds0 = static_cast<uint32_t>(reinterpret_cast<uintptr_t>((lds_ptr_t *)(lds)));
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      const uint32_t m0v = __builtin_amdgcn_readfirstlane(lds0 + (i * NW + wave) * (256 * VEC));
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
      if (EDGE && krem < 32) {
        int r, k;
        place(i, wave, lane, r, k);
        const uint64_t a = k < krem ? gb + voff[i] : reinterpret_cast<uint64_t>(&f32_zeros[0]);
        if constexpr (VEC == 4)
          asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off" : : "s"(m0v), "v"(a) : "memory", "m0");
        else
          asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dword %1, off" : : "s"(m0v), "v"(a) : "memory", "m0");
      } else if constexpr (VEC == 4) {
        asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2"
                     : : "s"(m0v), "v"(voff[i]), "s"(gb) : "memory", "m0");
      } else {
        asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dword %1, %2"
                     : : "s"(m0v), "v"(voff[i]), "s"(gb) : "memory", "m0");
      }
#pragma clang diagnostic pop
    }
  }

  // Lane's four k 4 c .. 4 c + 3 (chunk c) of its row in the 32-row fragment
  // at row0.
  __device__ __forceinline__ static float4 chunk(const char *lds, int row0, int c, int lane) {
    const int r = row0 + (lane & 31);
    if constexpr (KC) {
      return *reinterpret_cast<const float4 *>(lds + r * 128 + ((c ^ swz(r)) << 4));
    } else {
      const float *f = reinterpret_cast<const float *>(lds) + 4 * c * ROWS + r;
      return make_float4(f[0], f[ROWS], f[2 * ROWS], f[3 * ROWS]);
    }
  }
};

// Two F32 values as three BF16 parts each, packed in pairs: each part the
// nearest BF16 of what the ones before leave.  The head leaves at most 2^-8 of
// the value, in 16 bits, the middle at most 2^-17, in 7, so the three hold its
// 24 bits, and the part products that are left out (middle times remainder and
// less) come to at most 2^-24 of a product, of either sign.  The values are
// taken with their sign turned where sg is 0x80000000.  A value below about
// 2^-110 leaves bits under BF16's least subnormal, 2^-133: the low halves of
// its remainder's word, collected in lost.
__device__ __forceinline__ void split3_pair(float x, float y, uint32_t sg, uint32_t &hi, uint32_t &mid, uint32_t &lo,
                                            uint32_t &lost) {
  const float a = __uint_as_float(__float_as_uint(x) ^ sg), b = __uint_as_float(__float_as_uint(y) ^ sg);
  hi = bf16x2_bits(a, b);
  const float ra = a - __uint_as_float(hi << 16), rb = b - __uint_as_float(hi & 0xffff0000u);
  mid = bf16x2_bits(ra, rb);
  const float la = ra - __uint_as_float(mid << 16), lb = rb - __uint_as_float(mid & 0xffff0000u);
  lo = bf16x2_bits(la, lb);
  // (In asm, or the compiler keeps every remainder to collect them as a tree:
  // 48 spilled registers on 128 x 128.)
  asm("v_or3_b32 %0, %1, %2, %0" : "+v"(lost) : "v"(la), "v"(lb));
}

struct Raw8 {  // a lane's eight k of one fragment
  float4 a, b;
};
struct Parts3 {
  uint4 p[3];  // heads, middles, remainders
};

__device__ __forceinline__ float at4(const float4 &v, int e) {
  return e == 0 ? v.x : e == 1 ? v.y : e == 2 ? v.z : v.w;
}
__device__ __forceinline__ float raw_at(const Raw8 &r, int e) { return at4(e < 4 ? r.a : r.b, e & 3); }

// Pair q (0 .. 3) of a fragment's eight values into its parts.
__device__ __forceinline__ void split_piece(const Raw8 &r, Parts3 &o, int q, uint32_t sg, uint32_t &lost) {
  if (q == 0) split3_pair(r.a.x, r.a.y, sg, o.p[0].x, o.p[1].x, o.p[2].x, lost);
  else if (q == 1) split3_pair(r.a.z, r.a.w, sg, o.p[0].y, o.p[1].y, o.p[2].y, lost);
  else if (q == 2) split3_pair(r.b.x, r.b.y, sg, o.p[0].z, o.p[1].z, o.p[2].z, lost);
  else split3_pair(r.b.z, r.b.w, sg, o.p[0].w, o.p[1].w, o.p[2].w, lost);
}

// At most M DMA instructions (63 where M is more: the counter's range) and no
// LDS read of this wavefront outstanding, then the workgroup's barrier,
// neither moved past by an LDS access.
template <int M>
__device__ __forceinline__ void wait_tile() {
  constexpr int N = M < 63 ? M : 63;
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_waitcnt((N & 15) | ((N >> 4) << 14) | (7 << 4));
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

// Scheduling directive: each of MF MFMAs followed by V vector operations.
template <int Q, int MF, int V>
__device__ __forceinline__ void spread() {
  if constexpr (Q < MF) {
    __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
    __builtin_amdgcn_sched_group_barrier(0x002, V, 0);
    spread<Q + 1, MF, V>();
  }
}

// The accumulators the k loop goes round: a sum of rounded sums errs less
// than one long sum.  Four of a 32 x 32 wave tile, two of a 32 x 64 one where
// the registers have room.
template <int TM, int TN, bool SPLIT, int EDGE>
constexpr int f32_accs() {
  return !SPLIT ? 4 : (TM * TN <= 2 && EDGE < 2 ? 2 : 1);
}

template <int BM, int BN, int WM, int WN, int NS, bool SPLIT, bool AK, bool BKC, int EDGE>
__global__ void __launch_bounds__(WM *WN * 64, 2) gemm_f32_kernel(GemmArgs g) {
  constexpr int NW = WM * WN;
  constexpr int WTM = BM / WM, WTN = BN / WN, TM = WTM / 32, TN = WTN / 32, TF = TM + TN;
  using OA = F32Operand<BM, AK, NW, EDGE>;
  using OB = F32Operand<BN, BKC, NW, EDGE>;
  constexpr int STAGE = OA::BYTES + OB::BYTES;
  constexpr int PER_TILE = OA::PER + OB::PER;
  extern __shared__ __attribute__((aligned(1024))) char smem[];

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave / WN, wn = wave % WN;
  int tm, tn;
  tile_of(blockIdx.x, g.tiles_m, g.tiles_n, &tm, &tn);
  const int64_t m0 = static_cast<int64_t>(tm) * BM, n0 = static_cast<int64_t>(tn) * BN;
  const int64_t z = blockIdx.y;
  const int64_t zo = z / g.per_group, zi = z - zo * g.per_group;
  const float *A = static_cast<const float *>(g.a) + zo * g.sa2 + zi * g.sa;
  const float *B = static_cast<const float *>(g.b) + zo * g.sb2 + zi * g.sb;
  int64_t cz = zo * g.sc2 + zi * g.sc;  // the result's first element
  int64_t Kz = g.K;
  if (g.kc > 0) {
    // Split-K slice blockIdx.z: k in [ks, ks + Kz), into slice z of [S, M, N].
    const int64_t ks = static_cast<int64_t>(blockIdx.z) * g.kc;
    Kz = g.K - ks < g.kc ? g.K - ks : g.kc;
    A += AK ? ks : ks * g.lda;
    B += BKC ? ks : ks * g.ldb;
    cz += static_cast<int64_t>(blockIdx.z) * g.M * g.ldc;
  }
  OA oa;
  OB ob;
  oa.init(A, g.lda, m0, g.M, wave, lane);
  ob.init(B, g.ldb, n0, g.N, wave, lane);

  constexpr int NA = f32_accs<TM, TN, SPLIT, EDGE>();
  f32x16 accs[NA][TM][TN];
#pragma unroll
  for (int a = 0; a < NA; ++a)
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j)
#pragma unroll
        for (int r = 0; r < 16; ++r) accs[a][i][j][r] = 0.0f;
  f32x16(&acc)[TM][TN] = accs[0];
  auto fold_accs = [&]() {
#pragma unroll
    for (int a = NA / 2; a >= 1; a /= 2)
#pragma unroll
      for (int b = 0; b < a; ++b)
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
          for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) accs[b][i][j][r] += accs[b + a][i][j][r];
  };

  const int64_t ktiles = (Kz + 31) / 32;
  auto load = [&](int64_t kt, int stage) {
    if (kt >= ktiles) return;
    char *s = smem + stage * STAGE;
    oa.load(kt, Kz - 32 * kt, s, wave, lane);
    ob.load(kt, Kz - 32 * kt, s + OA::BYTES, wave, lane);
  };
  // Fragment f (A's TM, then B's TN) of k step st: this lane's eight k.
  auto read = [&](const char *s, int f, int st, Raw8 &r) {
    const int c = 4 * st + 2 * (lane >> 5);
    if (f < TM) {
      r.a = OA::chunk(s, wm * WTM + 32 * f, c, lane);
      r.b = OA::chunk(s, wm * WTM + 32 * f, c + 1, lane);
    } else {
      r.a = OB::chunk(s + OA::BYTES, wn * WTN + 32 * (f - TM), c, lane);
      r.b = OB::chunk(s + OA::BYTES, wn * WTN + 32 * (f - TM), c + 1, lane);
    }
  };
  if constexpr (!SPLIT) {
#pragma unroll
    for (int s = 0; s < NS - 1; ++s) load(s, s);
    for (int64_t kt = 0; kt < ktiles; kt += NS) {
#pragma unroll
      for (int s = 0; s < NS; ++s) {
        if (s == 0 || kt + s < ktiles) {
          // Tile kt + s has landed everywhere, and the tile before it is read.
          if (kt + s + NS - 2 < ktiles) wait_tile<(NS - 2) * PER_TILE>();
          else wait_tile<0>();  // the last tiles: none in flight behind them
          const char *st = smem + s * STAGE;
          const int h = lane >> 5;
          float4 fa[2][TM], fb[2][TN];
          auto read4 = [&](int p, int buf) {
#pragma unroll
            for (int i = 0; i < TM; ++i) fa[buf][i] = OA::chunk(st, wm * WTM + 32 * i, 2 * p + h, lane);
#pragma unroll
            for (int j = 0; j < TN; ++j) fb[buf][j] = OB::chunk(st + OA::BYTES, wn * WTN + 32 * j, 2 * p + h, lane);
          };
          read4(0, 0);
          load(kt + s + NS - 1, (s + NS - 1) % NS);
#pragma unroll
          for (int p = 0; p < 4; ++p) {
            if (p < 3) read4(p + 1, (p + 1) & 1);
#pragma unroll
            for (int e = 0; e < 4; ++e)
#pragma unroll
              for (int i = 0; i < TM; ++i)
#pragma unroll
                for (int j = 0; j < TN; ++j)
                  accs[p % NA][i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(
                      at4(fa[p & 1][i], e), at4(fb[p & 1][j], e), accs[p % NA][i][j], 0, 0, 0);
          }
        }
      }
    }
    fold_accs();
  } else {
#pragma unroll
    for (int s = 0; s < NS; ++s) load(s < ktiles ? s : 0, s);
    // Step 0's parts and step 1's values of the first tile.
    // An MFMA drops, downward, the bits of a small product that lie below its
    // accumulator's last: a bias of 2^-8 of a rounding, but one that a sum over
    // a result's rows or columns (a bias gradient) would collect.  Odd rows of
    // A and odd columns of B are taken with their sign turned, so results of
    // either parity lean either way (sum over 2000 rows of a [2000, 8192] x
    // [8192, 256] product: error 1.7e-6 without, at most 4.5e-7 with).
    const uint32_t sg = static_cast<uint32_t>(lane & 1) << 31;
    Raw8 raw[2][TF];
    Parts3 part[2][TF];
    // Bits that the parts could not hold.  The last tile splits its other stage
    // once more, which holds the tile before it or (one tile) the tile itself.
    uint32_t lost = 0;
    static_assert(NS == 2, "the waits below");
    if (ktiles > 1) wait_tile<PER_TILE>();
    else wait_tile<0>();
#pragma unroll
    for (int f = 0; f < TF; ++f) read(smem, f, 0, raw[0][f]);
#pragma unroll
    for (int f = 0; f < TF; ++f) read(smem, f, 1, raw[1][f]);
#pragma unroll
    for (int f = 0; f < TF; ++f)
#pragma unroll
      for (int q = 0; q < 4; ++q) split_piece(raw[0][f], part[0][f], q, sg, lost);

    // Tile kt + s multiplies the parts at hand; its own stage is free (its
    // values were read a tile ago) and takes tile kt + s + NS, while the next
    // tile's values are read and split between the MFMAs.
    for (int64_t kt = 0; kt < ktiles; kt += NS) {
#pragma unroll
      for (int s = 0; s < NS; ++s) {
        if (s == 0 || kt + s < ktiles) {
          wait_tile<0>();
          load(kt + s + NS, s);
          const char *nst = smem + ((s + 1) % NS) * STAGE;
#pragma unroll
          for (int st = 0; st < 2; ++st) {
            // The products of BF16 parts that F32 precision needs, smallest
            // first: lo hi, mid mid, hi lo, mid hi, hi mid, hi hi.
            constexpr int PA[6] = {2, 1, 0, 1, 0, 0}, PB[6] = {0, 1, 2, 0, 1, 0};
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int f = 0; f < TF; ++f) read(nst, f, st, raw[st][f]);
            __builtin_amdgcn_sched_barrier(0);
            constexpr int MF = 6 * TM * TN;
#pragma unroll
            for (int q = 0; q < 4 * TF; ++q) split_piece(raw[st ^ 1][q / 4], part[st ^ 1][q / 4], q % 4, sg, lost);
#pragma unroll
            for (int q = 0; q < MF; ++q) {
              const int t = q / (TM * TN), i = q % (TM * TN) / TN, j = q % TN;
              accs[st % NA][i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
                  __builtin_bit_cast(bf16x8, part[st][i].p[PA[t]]),
                  __builtin_bit_cast(bf16x8, part[st][TM + j].p[PB[t]]), accs[st % NA][i][j], 0, 0, 0);
            }
            // The step's 14 operations a pair of values spread over its MFMAs.
            spread<0, MF, (56 * TF + MF - 1) / MF>();
            __builtin_amdgcn_sched_barrier(0);
          }
        }
      }
    }
    fold_accs();
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j)
#pragma unroll
        for (int r = 0; r < 16; ++r)
          acc[i][j][r] =  // a turned zero is +0 again
              __uint_as_float(__float_as_uint(acc[i][j][r]) ^ sg ^ (static_cast<uint32_t>(r & 1) << 31)) + 0.0f;

    // A result that is not finite came from an operand that is not, or from a
    // head rounded up to infinity: the parts of such a value are not F32
    // arithmetic on it, nor are those of a value too small for three, so the
    // tile is formed again on the F32 matrix cores (4096^3 737 us; with such a
    // value in every tile 1693).
    uint32_t bad = lost & 0xffffu;
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j)
#pragma unroll
        for (int r = 0; r < 16; ++r) bad |= (__float_as_uint(acc[i][j][r]) & 0x7f800000u) == 0x7f800000u;
    if (__syncthreads_or(static_cast<int>(bad))) {
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
          for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.0f;
      for (int64_t kt = 0; kt < ktiles; ++kt) {
        load(kt, 0);
        wait_tile<0>();
#pragma unroll 1
        for (int st = 0; st < 2; ++st) {
          Raw8 r8[TF];
#pragma unroll
          for (int f = 0; f < TF; ++f) read(smem, f, st, r8[f]);
#pragma unroll
          for (int e = 0; e < 8; ++e)
#pragma unroll
            for (int i = 0; i < TM; ++i)
#pragma unroll
              for (int j = 0; j < TN; ++j)
                acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(raw_at(r8[i], e), raw_at(r8[TM + j], e), acc[i][j], 0, 0, 0);
        }
        wait_tile<0>();
      }
    }
  }

  const int lrow = lane & 31, lhalf = lane >> 5;
  const bool epi = g.bias != nullptr || g.resid != nullptr;
#pragma unroll
  for (int i = 0; i < TM; ++i) {
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      const int64_t col = n0 + wn * WTN + j * 32 + lrow;
      const int64_t rb = m0 + wm * WTM + i * 32 + 4 * lhalf;
      float v[16];
#pragma unroll
      for (int r = 0; r < 16; ++r) v[r] = acc[i][j][r];
      if (epi) fragment_epilogue<EDGE != 0>(g, rb, col, v);
      auto store = [&](auto *c) {
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int64_t row = rb + 8 * (r >> 2) + (r & 3);
          if (EDGE && (row >= g.M || col >= g.N)) continue;
          if constexpr (sizeof(*c) == 2) c[cz + row * g.ldc + col] = f32_to_bf16_bits(v[r]);
          else c[cz + row * g.ldc + col] = v[r];
        }
      };
      if (g.out_bf16) store(static_cast<uint16_t *>(g.c));
      else store(static_cast<float *>(g.c));
    }
  }
}

template <int BM, int BN, int WM, int WN, int NS, bool SPLIT, bool AK, bool BKC, int EDGE>
static hipError_t launch_f32(const Plan &p, hipStream_t st) {
  constexpr int SMEM = NS * (BM + BN) * 128;
  auto kern = gemm_f32_kernel<BM, BN, WM, WN, NS, SPLIT, AK, BKC, EDGE>;
  static const hipError_t attr =
      hipFuncSetAttribute(reinterpret_cast<const void *>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, SMEM);
  if (attr != hipSuccess) return attr;
  GemmArgs g;
  g.a = p.a; g.b = p.b; g.c = p.c;
  g.M = p.M; g.N = p.N; g.K = p.K;
  g.lda = p.lda; g.ldb = p.ldb;
  g.ldc = p.ldc > 0 ? p.ldc : p.N;
  g.sa = p.sa; g.sb = p.sb; g.sc = p.sc;
  g.per_group = p.per_group > 0 ? p.per_group : p.batch;
  g.sa2 = p.sa2; g.sb2 = p.sb2; g.sc2 = p.sc2;
  g.kc = p.kc;
  g.out_bf16 = p.eo == MI_BF16;
  g.bias = p.bias; g.resid = p.resid; g.ldr = p.ldr;
  g.tiles_m = static_cast<int>((p.M + BM - 1) / BM);
  g.tiles_n = static_cast<int>((p.N + BN - 1) / BN);
  const dim3 grid(static_cast<unsigned>(g.tiles_m * g.tiles_n), static_cast<unsigned>(p.batch),
                  static_cast<unsigned>(p.splits));
  kern<<<grid, WM * WN * 64, SMEM, st>>>(g);
  return hipGetLastError();
}

template <int BM, int BN, int WM, int WN, int NS, bool SPLIT, int EDGE>
static hipError_t launch_f32_orient(const Plan &p, hipStream_t st) {
  const bool ak = !p.ta, bk = p.tb;
  if (ak && bk) return launch_f32<BM, BN, WM, WN, NS, SPLIT, true, true, EDGE>(p, st);
  if (ak && !bk) return launch_f32<BM, BN, WM, WN, NS, SPLIT, true, false, EDGE>(p, st);
  if (!ak && bk) return launch_f32<BM, BN, WM, WN, NS, SPLIT, false, true, EDGE>(p, st);
  return launch_f32<BM, BN, WM, WN, NS, SPLIT, false, false, EDGE>(p, st);
}

// Sixteen-byte DMA: pitches, item strides, pointers and contiguous extents in
// fours (split-K slices start on k-tiles).
static bool f32_quads(const Plan &p) {
  return p.lda % 4 == 0 && p.ldb % 4 == 0 && p.sa % 4 == 0 && p.sb % 4 == 0 && p.sa2 % 4 == 0 && p.sb2 % 4 == 0 &&
         !(reinterpret_cast<uintptr_t>(p.a) & 15) && !(reinterpret_cast<uintptr_t>(p.b) & 15) &&
         (p.ta ? p.M : p.K) % 4 == 0 && (p.tb ? p.K : p.N) % 4 == 0;
}

bool f32_pipe_fits(const Plan &p) {
  // Operands by 4-byte DMA over k up to 8 (one with its k contiguous): a k-tile
  // of 32 is mostly lanes past k, and the register-staged kernel, which loads
  // them not at all, sums in the same order.  us there / here: 4096 x 4096 x 1
  // 23.1 / 30.2, x 2 with B^T 23.2 / 30.5; over k 9 to 63 it is still ahead (k 9
  // 24.8 / 30.6) by up to a quarter, but one chain over k errs more (k 16
  // 7.4e-8 against 6.0e-8).
  if (p.K <= 8 && !f32_quads(p) && (!p.ta || p.tb)) return false;
  // A lane's byte offset in a tile is 32 bits: 128 rows of the pitch.
  return p.ea == MI_F32 && p.eb == MI_F32 && p.lda < (int64_t(1) << 22) && p.ldb < (int64_t(1) << 22);
}

// The tiles: 64 x 64 on the F32 matrix cores, 64 x 128 and 128 x 128 on BF16
// parts.  A block's k step of 16 takes c1 us with its CU to itself and c2 a
// block where it shares it, over c0 of launch, first loads and last stores
// (measured on whole tiles: 784 x 128 x 64 in 5.1, 7.6 and 9.8 us, 64 x 128
// over k 2048 unsliced 0.27, 0.46 and 0.63 a step; 4096^3 0.27, 0.43 and
// 0.70).  Edges cost every tile their guards.
struct F32Tile {
  int bm, bn;
  double c0, c1, c2;
};
static const F32Tile F32_TILES[3] = {{64, 64, 3.3, 0.27, 0.26}, {64, 128, 4.2, 0.46, 0.43}, {128, 128, 5.2, 0.63, 0.70}};

// Estimated time (us) of the plan on tile t in S slices: the steps of the
// busiest CU, and for slices the reduce (2.5 us and their bytes at 5 TB/s).
static double f32_time(const Plan &p, const F32Tile &t, int64_t S) {
  const int64_t kc = ((p.K + S - 1) / S + 63) / 64 * 64, slices = (p.K + kc - 1) / kc;
  const int64_t blocks = ((p.M + t.bm - 1) / t.bm) * ((p.N + t.bn - 1) / t.bn) * p.batch * slices;
  const int64_t n = (blocks + 255) / 256, k = slices > 1 ? kc : p.K;
  const bool edge = p.M % t.bm || p.N % t.bn || p.K % 32 || !f32_quads(p);
  double us = t.c0 + static_cast<double>(n * ((k + 31) / 32 * 2)) * (n == 1 ? t.c1 : t.c2);
  if (edge) us *= 1.15;
  if (slices > 1) us += 2.5 + static_cast<double>((2 * slices + 1) * p.M * p.N) * 4.0 / 5e6;
  return us;
}

// The best tile for S slices.  4-byte DMA leaves no registers for the largest.
// Sums of up to 32 products stay on the F32 matrix cores, where an outer
// product is one rounding (4096 x 1 x 4096: 2.5e-8 from float64 against 3.5e-8
// from parts); 4096 x 4096 over k 16 and 32 23.0 and 20.6 us against 27.1 and
// 20.9 on 128 x 128.
static int f32_tile(const Plan &p, int64_t S) {
  int best = 0;
  if (p.K <= 32) return best;
  for (int t = 1; t < (f32_quads(p) ? 3 : 2); ++t)
    if (f32_time(p, F32_TILES[t], S) < f32_time(p, F32_TILES[best], S)) best = t;
  return best;
}

int f32_pipe_slices(const Plan &p) {
  int best = 1;
  double us = f32_time(p, F32_TILES[f32_tile(p, 1)], 1);
  if (p.batch != 1) return 1;
  for (int S : {2, 3, 4, 6, 8, 12, 16, 24, 32}) {
    if (p.K / S < 128) break;
    const double v = f32_time(p, F32_TILES[f32_tile(p, S)], S);
    if (v < us) {
      us = v;
      best = S;
    }
  }
  return best;
}

// Tile t of edge form E.  One k-tile or two want blocks in flight, not
// stages: 64 x 64 in two (32 KB of LDS, five blocks a CU) up to k 64, four
// past it.
template <int E>
static hipError_t launch_f32_tile(const Plan &p, int t, hipStream_t st) {
  if constexpr (E < 2)
    if (t == 2) return launch_f32_orient<128, 128, 2, 2, 2, true, E>(p, st);
  if (t == 1) return launch_f32_orient<64, 128, 2, 2, 2, true, E>(p, st);
  if (p.K <= 64) return launch_f32_orient<64, 64, 2, 2, 2, false, E>(p, st);
  return launch_f32_orient<64, 64, 2, 2, 4, false, E>(p, st);
}

hipError_t run_f32_pipe(const Plan &p, hipStream_t st) {
  const int t = f32_tile(p, p.splits);
  if (!f32_quads(p)) return launch_f32_tile<2>(p, t, st);
  if (p.K % 32 || p.M % F32_TILES[t].bm || p.N % F32_TILES[t].bn) return launch_f32_tile<1>(p, t, st);
  return launch_f32_tile<0>(p, t, st);
}

}  // namespace mi
