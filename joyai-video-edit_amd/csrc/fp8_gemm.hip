// Row-wise scaled FP8 GEMM with bias (drop-in for the reference's
// fp8_scaled_mm, deploy/joyomni_ops/csrc/fp8_gemm.cu:1450-1546):
//   out[m, n] = round_out( scale_a[m] * (acc[m, n] * scale_b[n]) + bias[n] ),
//   acc[m, n] = sum_k A[m, k] * B[k, n]   (fp8 e4m3fn operands, fp32 accumulate)
// with A [M, K] row-major and B [K, N] column-major (each column's K bytes
// contiguous, i.e. B^T [N, K] row-major) — the epilogue order of the
// reference's visitor tree (fp8_gemm.cu:99-136: acc * scale_b, then
// scale_a * that + bias, round to nearest).
//
// Four kernels, chosen by plan_gemm from M, N, K and the CU count:
//   pair    many rows: eight waves on a tile of 96 to 256 rows x 256 columns;
//   small   a few hundred rows: tiles of 64x64 to 128x192, with split K for few
//           tiles and a long K;
//   stream  up to 80 rows: all of them by 16 to 64 columns, the waves sharing K;
//   staged  what the others' direct global->LDS loads do not take: K == 0,
//           scales_b not 16-byte or bias not 8-byte aligned, 256 operand rows of
//           4 GiB and more.

#include <atomic>
#include <type_traits>

#include "jo_device.hpp"
#include "jo_host.hpp"

namespace jo {
namespace {

typedef int i32x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int kBM = 256;
constexpr int kBN = 256;
constexpr int kBK = 128;                      // bytes of K per stage
constexpr int kStageBytes = (kBM + kBN) * kBK;  // A tile then B tile
constexpr int kChunksPerThread = kBM * kBK / 16 / kBlock;  // 8 (same for B)

struct GemmArgs {
  const uint8_t* a;  // [M, K], row stride lda (bytes)
  const uint8_t* b;  // B^T [N, K], row stride ldb (bytes)
  const float* sa;   // [M]
  const float* sb;   // [N]
  const void* bias;  // [N] out dtype, optional
  void* out;         // [M, N] out dtype, row stride ldo (elements)
  int64_t lda, ldb, ldo;
  int M, N, K;
  float* ws = nullptr;  // split K: fp32 partial products [splits, M, N]
  int group = 0;        // pair kernel: tile rows of a group (xcd_grouped_tile)
};

__device__ __forceinline__ int swz(int r) { return (r & 7) ^ ((r >> 3) & 1); }

// One 32x32x64 fp8 MFMA with unit block scales (lowered to the unscaled
// v_mfma_f32_32x32x64_f8f6f4).
__device__ __forceinline__ f32x16 mfma32(const i32x8& a, const i32x8& b, const f32x16& c) {
  return __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(a, b, c, 0, 0, 0, 0, 0, 0);
}

// One 16x16x128 fp8 MFMA with unit block scales.
__device__ __forceinline__ f32x4 mfma16(const i32x8& a, const i32x8& b, const f32x4& c) {
  return __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(a, b, c, 0, 0, 0, 0, 0, 0);
}

// Staged kernel: one 256-thread workgroup per 256x256 output tile; the four
// waves own 128x128 quadrants computed with v_mfma_f32_32x32x64_f8f6f4
// (4x4 MFMA tiles, 256 fp32 accumulators per lane). K advances in 128-byte
// stages: every thread loads 8 sixteen-byte chunks of A and 8 of B^T from
// HBM into registers for the next stage while the MFMAs run on the current
// one, then writes them to the other half of a double-buffered LDS tile
// (2 x 64 KB). LDS rows are 128 bytes; chunk c of row r is stored at chunk
// position c ^ (r % 8) ^ ((r / 8) % 2), so the 16 rows a 16-lane group
// reads with one ds_read_b128 fall in 16 distinct 16-byte bank groups.
template <class OutTag>
__global__ __launch_bounds__(kBlock, 1) void fp8_gemm_kernel(const GemmArgs g) {
  __shared__ __attribute__((aligned(16))) uint8_t smem[2 * kStageBytes];  // 2 stages
  const int tid = threadIdx.x;
  const int lane = tid % kWave;
  const int wave = tid / kWave;
  const int wm = wave & 1, wn = wave >> 1;
  const int m0 = blockIdx.y * kBM, n0 = blockIdx.x * kBN;

  // Global chunk q = tid + 256 j of a 256 x 128-byte tile: row q / 8, chunk q % 8.
  // Rows beyond M (N) read row M-1 (N-1): their results are never stored.
  // Chunks beyond K read as zero so they add nothing.
  const uint8_t* ga[kChunksPerThread];
  const uint8_t* gb[kChunksPerThread];
  int lds_off[kChunksPerThread];
#pragma unroll
  for (int j = 0; j < kChunksPerThread; ++j) {
    const int q = tid + kBlock * j;
    const int r = q >> 3, c = q & 7;
    const int ra = min(m0 + r, g.M - 1), rb = min(n0 + r, g.N - 1);
    ga[j] = g.a + static_cast<int64_t>(ra) * g.lda + c * 16;
    gb[j] = g.b + static_cast<int64_t>(rb) * g.ldb + c * 16;
    lds_off[j] = r * kBK + ((c ^ swz(r)) << 4);
  }
  const int stages = (g.K + kBK - 1) / kBK;
  u32x4 ra[kChunksPerThread], rb[kChunksPerThread];
  auto load_stage = [&](int s) {
    const int kb = s * kBK;
#pragma unroll
    for (int j = 0; j < kChunksPerThread; ++j) {
      const int c = (tid + kBlock * j) & 7;
      const bool in_k = kb + c * 16 < g.K;
      ra[j] = in_k ? ld16(ga[j] + kb) : u32x4{0u, 0u, 0u, 0u};
      rb[j] = in_k ? ld16(gb[j] + kb) : u32x4{0u, 0u, 0u, 0u};
    }
  };
  auto store_stage = [&](int buf) {
    uint8_t* base = smem + buf * kStageBytes;
#pragma unroll
    for (int j = 0; j < kChunksPerThread; ++j) {
      *reinterpret_cast<u32x4*>(base + lds_off[j]) = ra[j];
      *reinterpret_cast<u32x4*>(base + kBM * kBK + lds_off[j]) = rb[j];
    }
  };

  f32x16 acc[4][4];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.f;

  // Fragment read offsets: tile row (l % 32) of subtile i, chunk pair
  // (l / 32) * 2 + {0, 1} of k-slice s (4 chunks per 64-byte slice).
  const int fr = lane & 31, fh = lane >> 5;

  load_stage(0);
  store_stage(0);
  __syncthreads();
  for (int s = 0; s < stages; ++s) {
    const int buf = s & 1;
    if (s + 1 < stages) load_stage(s + 1);
    const uint8_t* As = smem + buf * kStageBytes;
    const uint8_t* Bs = As + kBM * kBK;
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) {
      i32x8 af[4], bf[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int r = wm * 128 + i * 32 + fr;
        const int c = ks * 4 + fh * 2;
        const u32x4 lo = *reinterpret_cast<const u32x4*>(As + r * kBK + ((c ^ swz(r)) << 4));
        const u32x4 hi = *reinterpret_cast<const u32x4*>(As + r * kBK + (((c + 1) ^ swz(r)) << 4));
        af[i] = i32x8{(int)lo.x, (int)lo.y, (int)lo.z, (int)lo.w, (int)hi.x, (int)hi.y, (int)hi.z, (int)hi.w};
      }
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int r = wn * 128 + j * 32 + fr;
        const int c = ks * 4 + fh * 2;
        const u32x4 lo = *reinterpret_cast<const u32x4*>(Bs + r * kBK + ((c ^ swz(r)) << 4));
        const u32x4 hi = *reinterpret_cast<const u32x4*>(Bs + r * kBK + (((c + 1) ^ swz(r)) << 4));
        bf[j] = i32x8{(int)lo.x, (int)lo.y, (int)lo.z, (int)lo.w, (int)hi.x, (int)hi.y, (int)hi.z, (int)hi.w};
      }
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] = mfma32(af[i], bf[j], acc[i][j]);
    }
    if (s + 1 < stages) store_stage(buf ^ 1);
    __syncthreads();
  }

  // Epilogue: lane holds column n = n0 + wn*128 + j*32 + (l % 32) of subtile
  // (i, j), rows m = m0 + wm*128 + i*32 + (e / 4)*8 + (l / 32)*4 + e % 4.
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int n = n0 + wn * 128 + j * 32 + fr;
    if (n >= g.N) continue;
    const float sbn = g.sb[n];
    const float bn = g.bias ? load_elem<OutTag>(g.bias, n) : 0.f;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        const int m = m0 + wm * 128 + i * 32 + (e >> 2) * 8 + fh * 4 + (e & 3);
        if (m < g.M) {
          const float t = acc[i][j][e] * sbn;
          store_elem<OutTag>(g.out, static_cast<int64_t>(m) * g.ldo + n, __builtin_fmaf(g.sa[m], t, bn));
        }
      }
    }
  }
}

// s_waitcnt limiting only the vector-memory counter to n (n < 64); s_waitcnt
// limiting only the LDS counter to 0.
#define JO_WAIT_VM(n) __builtin_amdgcn_s_waitcnt(0x0F70 | ((n) & 15) | (((n) >> 4) << 14))
#define JO_WAIT_LDS0() __builtin_amdgcn_s_waitcnt(0xC07F)

template <int PER>
__device__ __forceinline__ void wait_loads(int later) {
  if (later >= 2)
    JO_WAIT_VM(2 * PER);
  else if (later == 1)
    JO_WAIT_VM(PER);
  else
    JO_WAIT_VM(0);
}

// ---------------------------------------------------------------------------
// Pair kernel, the default for many rows: eight waves on a
// BM x 256 tile (BM a multiple of 16 from 96 to 256), two per SIMD, in a 2 x 4
// grid of wave tiles of 64 columns whose first row takes (BM / 16 + 1) / 2 of
// the 16-row blocks. K advances in 128-byte stages, one
// v_mfma_f32_16x16x128_f8f6f4 deep, through LDS slots that direct
// global->LDS loads fill (eight lanes a row: a 1 KB load covers eight whole
// 128-byte lines; half lines doubled the L1 -> L2 requests and cost 10%). Per
// stage s, one barrier:
//   MFMAs of the wave's first two column blocks  | reads of the rest of this
//                                                | stage's fragments
//   wait for those reads and for this wave's loads of stage s+1; barrier
//   MFMAs of the last two | loads of stage s+2 into the slot of stage s (every
//                         | wave holds its fragments now), reads of stage
//                         | s+1's first fragments into registers set free
// so every fragment register is loaded under MFMAs that do not need it.
// LDS rows are 128 bytes; chunk c of row r sits at chunk position
// c ^ ((r >> 1) & 7): the sixteen consecutive rows that lanes 0-15 read with one
// ds_read_b128 fall in sixteen distinct 16-byte bank groups. (The bank-conflict
// counter still stands at half of the LDS cycles, where the 32-row fragments of
// 32x32x64 in this layout count next to none.)
//
// What bounds it: idle matrix cores (busy for 0.46 to 0.62 of the cycles at
// 3120 rows: epilogues, rounds, the first stages) and the clock, which power holds
// at 1.9-2.1 GHz of 2.4: the same launches on zero operands take 102.7 us for
// 120.7 at 3120x12288x4096, 119.9 for 143.7 at 3120x4096x16384. From registers
// alone, on random operands, 16x16x128 reaches 4.5-4.6 PFLOP/s at 2.2 GHz and
// 32x32x64, whose accumulators move twice the bits per flop, 4.1-4.2 at 2.0 (5.0
// at 2.4 both on zeros). Four waves of 128 x 128, with a third less LDS traffic,
// measured 2-12% slower. Against the same tiles on 32x32x64 with 224 or 256 rows
// only, us, weights from HBM: 3120x12288x4096 130.4 -> 126.7, 3120x16384x4096 174.0
// -> 165.6, 3120x4096x16384 158.7 -> 153.9, 3120x4096x4096 45.5 -> 43.3, 4096^3 53.6
// -> 52.2, 1560x12288x4096 91.9 -> 67.3, 1560x4096x4096 32.8 -> 28.8, 512x12288x4096
// 32.0 -> 31.4 (cached 31.5 -> 26.2).
// ---------------------------------------------------------------------------
constexpr int kQBK = 128;  // bytes of K per stage

__device__ __forceinline__ int qswz(int r) { return (r >> 1) & 7; }

// fn(std::integral_constant<int, 0>) .. fn(std::integral_constant<int, N - 1>).
template <int N, int I = 0, class Fn>
__device__ __forceinline__ void static_for(Fn&& fn) {
  if constexpr (I < N) {
    fn(std::integral_constant<int, I>{});
    static_for<N, I + 1>(fn);
  }
}

// A K that is not a multiple of 128 (it is one of 16): the part of a stage that
// is left over at its end is taken first, so that the loops know nothing of
// it. Chunks past K read that stage's first chunk of their row instead (always
// inside the row), and A's are then zeroed in LDS by the lanes that loaded
// them: what B holds there is multiplied by zero (it is a value of the same
// row of B, so a NaN among them was in the sum already). The lane's chunk
// position is the same in every load slot of a wave: slots are NW apart (even)
// and A has an even number of them.
struct KTail {
  bool part;       // K is not whole stages
  int back;        // bytes from this lane's chunk back to the row's first, if its chunk is past K
  uint32_t first;  // K offset of stage 0's loads, from operand bases moved back by shift()
  __device__ __forceinline__ KTail(int K, int lane, int wave) {
    const int bytes = (K - 1) % kQBK + 1, pos = ((lane & 7) ^ qswz((wave & 1) * 8 + lane / 8)) * 16;
    part = bytes != kQBK;
    back = pos >= bytes ? pos : 0;
    first = part ? static_cast<uint32_t>((K + kQBK - 1) / kQBK * kQBK - back) : 0u;
  }
  // Stage t >= 1 then reads from t * 128 on: whole stage t - 1 if stage 0 is the part.
  __device__ __forceinline__ int shift() const { return part ? kQBK : 0; }
};

// Direct loads of one stage: BM rows of A then BN rows of B^T, 128 bytes
// each, written by (BM + BN) / 8 wave instructions of 1 KB (8 rows, eight
// lanes per row); slot L fills stage bytes L * 1024 .. +1024 and belongs to
// wave L % NW.
template <int BM, int BN, int NW>
struct PairLoads {
  static constexpr int kSlots = (BM + BN) / 8;
  static constexpr int kPerWave = (kSlots + NW - 1) / NW;
  static constexpr bool kEven = kSlots % NW == 0;
  const uint8_t* base[kPerWave];  // wave-uniform: the tile's first row of A or B^T
  uint32_t off[kPerWave];         // this lane's 16-byte chunk of each slot at K offset 0
  bool last;                      // the wave owns a slot kPerWave - 1 (always when kEven)
};

// LDS of a workgroup: the rings (later the staged output tile), then the row
// scales, column scales and bias of the tile.
constexpr int kScaleRows = 256;
template <int BM, int BN, int NW, int NBS>
constexpr int pair_ring_bytes() {
  constexpr int ring = (2 * BM + NBS * BN) * kQBK;
  constexpr int store = NW * ((BM / 16 + 1) / 2) * 16 * (BN / (NW / 2) * 2 + 16);
  return ring > store ? ring : store;
}

// The K loop and epilogue of a wave holding MI row blocks of 16 (from the
// tile's row row0 on). NBS: B stages go through a ring of NBS slots beside A's
// two, so B loads run NBS - 1 stages ahead and A loads one.
template <class OutTag, int BM, int BN, int NW, int MI, int NBS, bool LINES>
__device__ __forceinline__ void fp8_gemm_pair_tile(const GemmArgs& g, uint8_t* smem,
                                                   const PairLoads<BM, BN, NW>& ld, const KTail& kt, int wave,
                                                   int row0, int wn, int m0, int n0) {
  using Loads = PairLoads<BM, BN, NW>;
  constexpr int WCOLS = BN / (NW / 2);  // wave tile columns
  constexpr int J = WCOLS / 16;         // n-blocks of 16 per wave
  constexpr int JH = J / 2;             // n-blocks of a half stage
  // Ring layout. NBS = 2: slot t % 2 holds stage t's A rows then its B rows.
  // NBS = 3: two A slots, then three B slots.
  constexpr int kASlot = NBS == 2 ? (BM + BN) * kQBK : BM * kQBK;
  constexpr int kBSlot = NBS == 2 ? (BM + BN) * kQBK : BN * kQBK;
  constexpr int kBBase = NBS == 2 ? BM * kQBK : 2 * BM * kQBK;
  constexpr int PER = Loads::kPerWave;
  constexpr int NB = BN / 8 / NW;  // B loads of a wave a stage: the last NB of its slots
  static_assert(J >= 2 && J % 2 == 0 && MI >= 2 && MI <= 8, "tile shape");
  constexpr int kScaleOff = pair_ring_bytes<BM, BN, NW, NBS>();
  static_assert((NBS == 2 || NBS == 3) && (BN / 8) % NW == 0, "B ring");
  const int lane = threadIdx.x % kWave;
  const int stages = (g.K + kQBK - 1) / kQBK;
  // Load i of this wave is A (slot index below BM / 8; a wave's A loads come
  // first in its slot order) or B: known at compile time but for the one index
  // that the last A slots share with the first B slots.
  auto is_a = [&](auto ic) {
    constexpr int i = decltype(ic)::value;
    if constexpr ((i + 1) * NW <= BM / 8) return true;
    if constexpr (i * NW >= BM / 8) return false;
    return wave + i * NW < BM / 8;
  };
  // Load i of stage t at K offset koff, A to slot t % 2 and B to ring slot bslot.
  auto issue_one = [&](int t, int bslot, uint32_t koff, auto ic) {
    constexpr int i = decltype(ic)::value;
    if (Loads::kEven || i + 1 < PER || ld.last) {
      uint8_t* dst = is_a(ic) || NBS == 2 ? smem + (t & 1) * kASlot + (wave + i * NW) * 1024
                                          : smem + kBBase + bslot * kBSlot + (wave + i * NW - BM / 8) * 1024;
      __builtin_amdgcn_global_load_lds(ld.base[i] + (ld.off[i] + koff), (__attribute__((address_space(3))) void*)dst, 16, 0, 0);
    }
  };
  // The loads issued in stage s's second half: A of stage s + 2 and B of
  // stage s + NBS, the latter into the slot of stage s's B (bcur).
  auto issue_batch_one = [&](int s, int bcur, auto ic) {
    if (NBS == 2 || is_a(ic))
      issue_one(s + 2, 0, (s + 2) * kQBK, ic);
    else if (s + NBS < stages)
      issue_one(s + NBS, bcur, (s + NBS) * kQBK, ic);
  };

  f32x4 acc[MI][J];
#pragma unroll
  for (int i = 0; i < MI; ++i)
#pragma unroll
    for (int j = 0; j < J; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};

  // Fragment rows are row0 + i*16 + lane%16 (A) and wn*WCOLS + j*16 +
  // lane%16 (B): they differ from lane%16 by multiples of 16, so they share
  // its swizzle. Lane group lane/16 holds the 32 bytes of K from its chunk
  // pair on, in A and B alike.
  const int fr = lane & 15, fh = lane >> 4;
  const int q = qswz(fr);
  int offa[2], offb[2];  // [chunk of the pair]
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const int pos = ((fh * 2 + h) ^ q) << 4;
    offa[h] = (row0 + fr) * kQBK + pos;
    offb[h] = kBBase + (wn * WCOLS + fr) * kQBK + pos;
  }
  auto frag = [&](const uint8_t* lo_p, const uint8_t* hi_p) {
    const u32x4 lo = *reinterpret_cast<const u32x4*>(lo_p);
    const u32x4 hi = *reinterpret_cast<const u32x4*>(hi_p);
    return i32x8{(int)lo.x, (int)lo.y, (int)lo.z, (int)lo.w, (int)hi.x, (int)hi.y, (int)hi.z, (int)hi.w};
  };
  i32x8 af[MI], bf[J];
  auto read_a = [&](int s, int i) {
    const uint8_t* st = smem + (s & 1) * kASlot;
    af[i] = frag(st + offa[0] + i * 16 * kQBK, st + offa[1] + i * 16 * kQBK);
  };
  auto read_b = [&](int bslot, int j) {
    const uint8_t* st = smem + bslot * kBSlot;
    bf[j] = frag(st + offb[0] + j * 16 * kQBK, st + offb[1] + j * 16 * kQBK);
  };
  // Stage s's wait: this wave's LDS reads, and its loads up to stage s + 1's.
  // A of s + 1 came with the latest loads; with NBS = 3 only their tail, B of
  // s + 2, may stay in flight.
  auto wait_next = [&](int s) {
    JO_WAIT_LDS0();
    if (NBS == 3 && s + 2 < stages)
      JO_WAIT_VM(NB);
    else
      JO_WAIT_VM(0);
  };
  auto bare_barrier = [&]() {
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  };
  // B first: the accumulator is the transposed tile (a lane holds one output
  // row and four consecutive columns). MFMA t of a half: row block t / JH,
  // column block half * JH + t % JH.
  auto mfma_t = [&](int half, int t) {
    const int i = t / JH, j = half * JH + ((i & 1) ? JH - 1 - t % JH : t % JH);
    acc[i][j] = mfma16(bf[j], af[i], acc[i][j]);
  };
  constexpr int NT = MI * JH;     // MFMAs of a half
  constexpr int NA1 = MI / 2;     // A blocks read in the first half (the last ones)
  constexpr int NA0 = MI - NA1;   // A blocks read in the second half, for the next stage
  // Fragment f that the first half reads (of this stage), in the order of
  // need: A blocks NA0 .. MI-1, then the second half's B blocks.
  auto read_first = [&](int s, int bcur, int f) {
    if (f < NA1)
      read_a(s, NA0 + f);
    else
      read_b(bcur, JH + f - NA1);
  };
  constexpr int NF1 = NA1 + JH;
  // Stage s with stage s+1 present (NEXT) and stage s+2 present (MORE); bcur
  // and bnext are the ring slots of stage s's and stage s+1's B.
  constexpr int KB = BM == 256 ? 2 : 0;  // MFMAs of the second half before the barrier
  auto stage = [&](int s, int bcur, int bnext, auto next, auto more) {
    constexpr bool kNext = decltype(next)::value, kMore = decltype(more)::value;
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      mfma_t(0, t);
      if (t < NF1) read_first(s, bcur, t);
      __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
    for (int f = NT; f < NF1; ++f) read_first(s, bcur, f);
    __builtin_amdgcn_sched_barrier(0);
    wait_next(s);
#pragma unroll
    for (int t = 0; t < KB; ++t) mfma_t(1, t);
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (kNext) bare_barrier();
    static_for<NT - KB>([&](auto uc) {
      constexpr int u = decltype(uc)::value, t = KB + u;
      mfma_t(1, t);
      if constexpr (kMore && u < PER) issue_batch_one(s, bcur, uc);
      if constexpr (kNext) {
        // B blocks of the next first half, then A block i once its own MFMAs
        // of this half are out.
        if constexpr (u < JH) read_b(bnext, u);
        if constexpr (t % JH == JH - 1 && t / JH >= 1 && t / JH - 1 < NA0) read_a(s + 1, t / JH - 1);
      }
      __builtin_amdgcn_sched_barrier(0);
    });
    static_assert(PER <= NT - KB, "every load has an MFMA to follow");
  };
  static_assert(NA0 <= MI - 1 && NT - KB >= JH, "the second half reads every early fragment");

  using T = std::true_type;
  using F = std::false_type;
  // Prologue: stage 0, then what the second halves of stages -2 and -1 would
  // have issued (stage 1; with NBS = 3, A of 1 and B of 1 and 2, B before A
  // within a stage); stage 0 starts once its own loads are in.
  auto issue_part = [&](int t, bool a) {
    static_for<PER>([&](auto ic) {
      if (is_a(ic) == a) issue_one(t, t, t == 0 ? kt.first : t * kQBK, ic);
    });
  };
  auto issue = [&](int t) {
    static_for<PER>([&](auto ic) { issue_one(t, t, t == 0 ? kt.first : t * kQBK, ic); });
  };
  // The tile's scales and bias go to LDS first (4 bytes a lane, 64 lanes a
  // load), the oldest loads of all, so that the epilogue does not start with
  // a wait for memory.
  uint8_t* scales = smem + kScaleOff;
  {
    auto load4 = [&](const void* src, int at) {
      __builtin_amdgcn_global_load_lds(static_cast<const uint8_t*>(src), (__attribute__((address_space(3))) void*)(scales + at), 4, 0, 0);
    };
    static_assert(BN == 256 && NW == 8 && kScaleRows == 256, "one scale load a wave");
    if (wave < 4)
      load4(g.sa + min(m0 + wave * 64 + lane, g.M - 1), wave * 256);
    else
      load4(g.sb + min(n0 + (wave - 4) * 64 + lane, g.N - 1), wave * 256);
    if (g.bias && wave < 2)
      load4(static_cast<const uint16_t*>(g.bias) + min(n0 + (wave * 64 + lane) * 2, g.N - 2), 2048 + wave * 256);
  }
  // In flight after stage 0's loads: NB B loads per later B stage and this
  // wave's A loads of stage 1 (PER - NB; one fewer for a wave without a last
  // slot, which is always a B slot since every wave has NB of those).
  const bool full = Loads::kEven || ld.last;
  if constexpr (NBS == 2) {
    issue(0);
    if (stages > 1) issue(1);
    JO_WAIT_LDS0();
    if (full)
      wait_loads<PER>(stages > 1 ? 1 : 0);
    else
      wait_loads<PER - 1>(stages > 1 ? 1 : 0);
  } else {
    issue_part(0, false);
    issue_part(0, true);
    if (stages >= 3) {
      issue_part(1, false);
      issue_part(1, true);
      issue_part(2, false);
      JO_WAIT_LDS0();
      if (full)
        JO_WAIT_VM(2 * NB + PER - NB);
      else
        JO_WAIT_VM(2 * NB + PER - NB - 1);
    } else if (stages == 2) {
      issue(1);
      JO_WAIT_LDS0();
      if (full)
        JO_WAIT_VM(PER);
      else
        JO_WAIT_VM(PER - 1);
    } else {
      JO_WAIT_LDS0();
      JO_WAIT_VM(0);
    }
  }
  if (kt.part) {  // this wave's loads of stage 0 are in
    asm volatile("" ::: "memory");
    if (kt.back)
      static_for<PER>([&](auto ic) {
        if (is_a(ic)) *reinterpret_cast<u32x4*>(smem + (wave + decltype(ic)::value * NW) * 1024 + lane * 16) = u32x4{0u, 0u, 0u, 0u};
      });
    JO_WAIT_LDS0();
  }
  bare_barrier();
#pragma unroll
  for (int j = 0; j < JH; ++j) read_b(0, j);  // stage 0's slot
#pragma unroll
  for (int i = 0; i < NA0; ++i) read_a(0, i);
  int s = 0, bcur = 0, bnext = 1, bthen = NBS - 1;  // bthen: NBS = 3 only
  auto turn = [&]() {
    const int freed = bcur;
    bcur = bnext;
    bnext = NBS == 2 ? freed : bthen;
    bthen = freed;
  };
  for (; s + 2 < stages; ++s, turn()) stage(s, bcur, bnext, T{}, T{});
  if (s + 1 < stages) {
    stage(s++, bcur, bnext, T{}, F{});
    turn();
  }
  stage(s, bcur, bnext, F{}, F{});

  // Epilogue. Block (i, j) element e of a lane is row m0 + row0 + i*16 +
  // lane%16, column n0 + wn*WCOLS + j*16 + (lane/16)*4 + e. Each wave passes
  // its tile through its own part of the LDS (the ring is free once every
  // wave is past the barrier), one block of 16 rows at a time, so that rows
  // leave as whole 16-byte lane stores, WCOLS * 2 bytes (128: a whole line) a
  // row. No wave waits for another after the barrier.
  constexpr int kRowBytes = WCOLS * 2 + 16;
  constexpr int kWaveBytes = MI * 16 * kRowBytes;
  float sam[MI];
#pragma unroll
  for (int i = 0; i < MI; ++i) sam[i] = *reinterpret_cast<const float*>(scales + (row0 + i * 16 + fr) * 4);
  float sbq[J][4], bq[J][4];
#pragma unroll
  for (int j = 0; j < J; ++j) {
    const int c = wn * WCOLS + j * 16 + fh * 4;
    const u32x4 sbv = *reinterpret_cast<const u32x4*>(scales + kScaleRows * 4 + c * 4);
    const u32x2 braw = *reinterpret_cast<const u32x2*>(scales + kScaleRows * 4 + BN * 4 + c * 2);
    const u32x4 b4{braw.x, braw.y, 0u, 0u};
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      sbq[j][t] = elem<F32>(sbv, t);
      bq[j][t] = g.bias ? elem<OutTag>(b4, t) : 0.f;
    }
  }
  bare_barrier();  // this wave's LDS reads were all waited for by its last MFMAs
  constexpr int kMaxWave = ((BM / 16 + 1) / 2) * 16 * kRowBytes;
  static_assert(kWaveBytes <= kMaxWave, "wave region");
  uint8_t* mine = smem + wave * kMaxWave;
  constexpr int kLanesPerRow = WCOLS * 2 / 16;          // 16-byte lanes of a row
  constexpr int kRowsPerStore = kWave / kLanesPerRow;   // rows of a wave store
  const int sr = lane / kLanesPerRow, sc = lane % kLanesPerRow;
  auto stage_block = [&](int i) {
#pragma unroll
    for (int j = 0; j < J; ++j) {
      float o[8];
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        o[t] = __builtin_fmaf(sam[i], acc[i][j][t] * sbq[j][t], bq[j][t]);
        o[t + 4] = 0.f;
      }
      const u32x4 pk = pack<OutTag>(o);
      *reinterpret_cast<u32x2*>(mine + (i * 16 + fr) * kRowBytes + (j * 16 + fh * 4) * 2) = u32x2{pk.x, pk.y};
    }
  };
  // LINES: output rows start on 128-byte lines. Where they do not (N of no multiple
  // of 64) a wave's pieces end inside lines that the next wave completes, so they
  // are left to the L2 to join instead of written through: us, through / joined,
  // 4326x10968x640 57.7 / 40.7, 4066x4072x128 14.6 / 10.7, 3184x9384x1280 52.3 / 44.0.
  // Whole lines written through are not read again and stay out of the L2. A
  // kernel for each: with the choice in this loop 3120x4096x4096 took 43.8 us for
  // 42.7, with a copy of the loop for each behind another kernel 51.0 for 50.4.
  // A wave's LDS operations run in order, so block i's reads follow its
  // writes; block i + 1 is written before block i leaves.
  stage_block(0);
#pragma unroll
  for (int i = 0; i < MI; ++i) {
    if (i + 1 < MI) stage_block(i + 1);
    asm volatile("" ::: "memory");
#pragma unroll
    for (int r = i * 16; r < i * 16 + 16; r += kRowsPerStore) {
      const int m = m0 + row0 + r + sr, n = n0 + wn * WCOLS + sc * 8;
      const u32x4 v = *reinterpret_cast<const u32x4*>(mine + (r + sr) * kRowBytes + sc * 16);
      if (m < g.M && n < g.N) {
        uint16_t* dst = static_cast<uint16_t*>(g.out) + static_cast<int64_t>(m) * g.ldo + n;
        if constexpr (LINES)
          st16_nt(dst, v);
        else
          st16(dst, v);
      }
    }
  }
}

// Output tile of this workgroup. The dispatcher hands workgroup id (linear
// over the grid, x fastest) to XCD id % 8, and each XCD has its own L2, so
// consecutive ids are spread over the XCDs and the tiles an XCD runs
// together should share operand rows. XCD x gets a contiguous range of a
// grouped order (groups of `group` tile rows, column by column inside a
// group): the ~32 tiles it runs at once are five tile rows by six columns,
// eleven operand panels where the row-major order gives it two columns by
// sixteen rows, eighteen (3120x12288x4096 141.0 -> 137.5 us with groups of
// four, 4096^3 59.0 -> 58.1). group_rows picks the size.
__device__ __forceinline__ void xcd_grouped_tile(int group, int bm, int bn, int& m0, int& n0) {
  const int ntn = gridDim.x, ntm = gridDim.y, tiles = ntn * ntm;
  const int id = blockIdx.y * ntn + blockIdx.x;
  const int x = id & 7;
  const int t = x * (tiles >> 3) + min(x, tiles & 7) + (id >> 3);  // a bijection of [0, tiles)
  const int grp = t / (group * ntn);
  const int r0 = grp * group;
  const int rows = min(group, ntm - r0);
  const int w = t - grp * group * ntn;
  m0 = (r0 + w % rows) * bm;
  n0 = (w / rows) * bn;
}

template <class OutTag, int BM, int BN, int NW, int NBS, bool LINES>
__device__ __forceinline__ void fp8_gemm_pair_body(const GemmArgs& g) {
  using Loads = PairLoads<BM, BN, NW>;
  constexpr int RB = BM / 16;  // 16-row blocks: the first wave row takes (RB + 1) / 2
  static_assert(BM % 16 == 0 && BM >= 64 && BM <= 256, "tile rows");
  __shared__ __attribute__((aligned(1024))) uint8_t smem[pair_ring_bytes<BM, BN, NW, NBS>() + (kScaleRows + BN) * 4 + BN * 2];
  const int tid = threadIdx.x;
  const int lane = tid % kWave;
  const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
  // A 2 x NW/2 grid of wave tiles. A workgroup's waves are spread round-robin
  // over the CU's four SIMDs, so with NW = 8 waves w and w + 4 share a SIMD:
  // with an odd number of row blocks each SIMD runs a wave of each height.
  const int wm = wave / (NW / 2), wn = wave % (NW / 2);
  int m0, n0;
  xcd_grouped_tile(g.group, BM, BN, m0, n0);

  // Lane p of a slot fills row +p/8, chunk position p%8 with the global chunk
  // that belongs there. Rows beyond M (N) read row M-1 (N-1); they are never
  // stored. Wave-uniform 64-bit tile bases plus 32-bit lane offsets (the host
  // keeps 256 rows of A and B^T under 4 GB).
  Loads ld;
  const KTail kt(g.K, lane, wave);
#pragma unroll
  for (int i = 0; i < Loads::kPerWave; ++i) {
    const int slot = wave + i * NW;
    const bool is_a = slot < BM / 8;
    const int r = (is_a ? slot : slot - BM / 8) * 8 + lane / 8;
    const int row = is_a ? min(m0 + r, g.M - 1) - m0 : min(n0 + r, g.N - 1) - n0;
    ld.base[i] = (is_a ? g.a + static_cast<int64_t>(m0) * g.lda : g.b + static_cast<int64_t>(n0) * g.ldb) - kt.shift();
    ld.off[i] = static_cast<uint32_t>(row) * static_cast<uint32_t>(is_a ? g.lda : g.ldb) +
                (((lane & 7) ^ qswz(r)) * 16);
  }
  ld.last = Loads::kEven || wave + (Loads::kPerWave - 1) * NW < Loads::kSlots;
  constexpr int kUp = (RB + 1) / 2, kLow = RB / 2;
  if constexpr (kUp == kLow) {
    fp8_gemm_pair_tile<OutTag, BM, BN, NW, kUp, NBS, LINES>(g, smem, ld, kt, wave, wm * kUp * 16, wn, m0, n0);
  } else {
    if (wm == 0)
      fp8_gemm_pair_tile<OutTag, BM, BN, NW, kUp, NBS, LINES>(g, smem, ld, kt, wave, 0, wn, m0, n0);
    else
      fp8_gemm_pair_tile<OutTag, BM, BN, NW, kLow, NBS, LINES>(g, smem, ld, kt, wave, kUp * 16, wn, m0, n0);
  }
}

template <class OutTag, int BM, int BN, int NW, int NBS, bool LINES>
__global__ __launch_bounds__(NW * 64, 1) void fp8_gemm_pair_kernel(const GemmArgs g) {
  fp8_gemm_pair_body<OutTag, BM, BN, NW, NBS, LINES>(g);
}

// Tile rows of a group of xcd_grouped_tile: equal groups of at most five (six
// rows stay one group). Against four: [3120, 12288] x 4096 at fifteen tile
// rows 123.3 -> 121.5 us (three groups of five against 4 + 4 + 4 + 3),
// [512, 12288] x 4096 at five tile rows 28.8 -> 26.7 (one group: the weight
// leaves HBM once); two, three, eight and one group of all rows measured level
// or slower on eleven shapes.
int group_rows(int tile_rows) {
  if (tile_rows <= 6) return tile_rows;
  const int groups = (tile_rows + 4) / 5;
  return (tile_rows + groups - 1) / groups;
}

template <class OutTag, int BM, int BN, int NW, int NBS>
void launch_pair(const GemmArgs& args, hipStream_t stream) {
  GemmArgs g = args;
  g.group = group_rows((g.M + BM - 1) / BM);
  const dim3 grid((g.N + BN - 1) / BN, (g.M + BM - 1) / BM);
  if (g.ldo % 64 == 0 && aligned(g.out, 128))
    hipLaunchKernelGGL((fp8_gemm_pair_kernel<OutTag, BM, BN, NW, NBS, true>), grid, dim3(NW * 64), 0, stream, g);
  else
    hipLaunchKernelGGL((fp8_gemm_pair_kernel<OutTag, BM, BN, NW, NBS, false>), grid, dim3(NW * 64), 0, stream, g);
}

// The pair kernel at `rows` tile rows (a multiple of 16 from 96 to 256), B two
// stages ahead (NBS = 3) except at 256 rows, whose rings fill the LDS: a long
// K's operands come from HBM and the deeper ring covers their latency
// ([3120, 4096] x 16384 at 224 rows 174 -> 169 us, [1560, 4096] x 16384 at 192
// rows 146 -> 123), as it does the loads of the low tiles ([512, 12288] x 4096
// at 128 rows 28.3 -> 25.7); on multi-round grids of 208 and 224 rows it
// measured 0-1% slower (169.5 -> 171.0, 168.3 -> 170.8 at 3120x16384x4096).
template <class OutTag, int ROWS = 256>
void launch_pair_rows(const GemmArgs& g, hipStream_t stream, int rows) {
  if (rows == ROWS || ROWS == 96)
    launch_pair<OutTag, ROWS, 256, 8, (ROWS == 256 ? 2 : 3)>(g, stream);
  else if constexpr (ROWS > 96)
    launch_pair_rows<OutTag, ROWS - 16>(g, stream, rows);
}

// ---------------------------------------------------------------------------
// Small-tile kernel, for grids that the pair kernel's 256-column tiles would
// leave mostly idle (a few hundred rows: the text stream's Fp8Linear calls;
// [256, 4096] is 32 tiles of 128x256 for 256 CUs). NW waves on a BM x BN tile
// (64x64, 64x128, 128x128 or 128x192 with four) in a WGM x NW/WGM grid of wave
// tiles (WGM = 2); the 96-column tiles give each wave 32 x 96 (128x96: four
// waves down the rows, WGM = 4; 64x96: two waves, WGM = 2, two workgroups to a
// CU's LDS); K advances in 128-byte stages (whole lines, the pair kernel's LDS
// layout) through a ring of NST slots that direct loads fill NST-1 stages ahead;
// one barrier a stage.
// Its K loop streams (BM + BN) x 128 bytes a stage for BM x BN x 128 MACs, so
// it only pays where it brings CUs into play that the large tiles leave idle.
// ---------------------------------------------------------------------------
template <int BM, int BN, int NW>
struct SmallLoads {
  static constexpr int kSlots = (BM + BN) / 8;  // 1 KB wave loads (8 rows) a stage
  static constexpr int kPerWave = kSlots / NW;
  static_assert(kSlots % NW == 0, "load slots spread evenly over the waves");
  const uint8_t* base[kPerWave];  // wave-uniform: the tile's first row of A or B^T
  uint32_t off[kPerWave];         // this lane's 16-byte chunk of each slot at K offset 0
};

template <class OutTag, int BM, int BN, int NW, int NST, bool SPLIT, bool PART, int WGM>
__device__ __forceinline__ void fp8_gemm_small_body(const GemmArgs& g) {
  constexpr int WROWS = BM / WGM, WCOLS = BN / (NW / WGM);  // wave tile
  constexpr int MI = WROWS / 32, J = WCOLS / 32;
  constexpr int kStage = (BM + BN) * kQBK;
  constexpr int kRowBytes = BN * 2 + 16;  // padded LDS row of the staged output tile
  constexpr int kChunksPerRow = BN * 2 / 16;
  using Loads = SmallLoads<BM, BN, NW>;
  constexpr int PER = Loads::kPerWave;
  static_assert(NW % WGM == 0 && WROWS % 32 == 0 && WCOLS % 32 == 0 && MI >= 1 && J >= 1 &&
                    BM * kRowBytes <= NST * kStage && NST >= 2 && NST <= 4,
                "tile shape");
  __shared__ __attribute__((aligned(1024))) uint8_t smem[NST * kStage];
  const int tid = threadIdx.x;
  const int lane = tid % kWave;
  const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
  const int wm = wave % WGM, wn = wave / WGM;
  int m0, n0;
  // Groups of four tile rows, a constant (a size out of the arguments, loaded
  // before the first address is known, 19.6 -> 20.3 us at 256x12288x4096).
  xcd_grouped_tile(4, BM, BN, m0, n0);

  // Lane p of load slot L fills row 8L + p/8 of the stage (A rows, then B^T
  // rows), chunk position p%8, with the global chunk that belongs there; rows
  // beyond M (N) read row M-1 (N-1) and are never stored.
  Loads ld;
  // PART: K is not whole stages (a split K always is). A kernel of its own: with
  // the test at run time 256x12288x4096 took 20.2 us for 19.7, 777x3072x3072
  // 16.2 for 15.6.
  static_assert(!(SPLIT && PART), "a split K is whole stages");
  const KTail kt(PART ? g.K : kQBK, lane, wave);
#pragma unroll
  for (int i = 0; i < PER; ++i) {
    const int slot = wave + i * NW;
    const bool is_a = slot < BM / 8;
    const int r = (is_a ? slot : slot - BM / 8) * 8 + lane / 8;
    const int row = is_a ? min(m0 + r, g.M - 1) - m0 : min(n0 + r, g.N - 1) - n0;
    ld.base[i] = (is_a ? g.a + static_cast<int64_t>(m0) * g.lda : g.b + static_cast<int64_t>(n0) * g.ldb) - kt.shift();
    ld.off[i] = static_cast<uint32_t>(row) * static_cast<uint32_t>(is_a ? g.lda : g.ldb) +
                (((lane & 7) ^ qswz(r)) * 16);
  }
  // SPLIT: workgroup z of the grid's gridDim.z takes the z-th equal share of
  // the K stages and writes its partial product for the reduction kernel.
  const int stages = SPLIT ? g.K / kQBK / static_cast<int>(gridDim.z) : PART ? (g.K + kQBK - 1) / kQBK : g.K / kQBK;
  const int s0 = SPLIT ? static_cast<int>(blockIdx.z) * stages : 0;
  auto issue = [&](int s, uint32_t koff) {
    uint8_t* dst = smem + (s % NST) * kStage;
#pragma unroll
    for (int i = 0; i < PER; ++i)
      __builtin_amdgcn_global_load_lds(ld.base[i] + (ld.off[i] + koff),
                                       (__attribute__((address_space(3))) void*)(dst + (wave + i * NW) * 1024),
                                       16, 0, 0);
  };

  // Fragment rows wm*WROWS + i*32 + lane%32 (A) and wn*WCOLS + j*32 +
  // lane%32 (B): multiples of 32 apart, so they share lane%32's swizzle.
  const int fr = lane & 31, fh = lane >> 5;
  const int q = qswz(fr);
  int offa[2][2], offb[2][2];  // [half of the stage][chunk of the pair]
#pragma unroll
  for (int k = 0; k < 2; ++k)
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int pos = ((k * 4 + fh * 2 + h) ^ q) << 4;
      offa[k][h] = (wm * WROWS + fr) * kQBK + pos;
      offb[k][h] = BM * kQBK + (wn * WCOLS + fr) * kQBK + pos;
    }
  f32x16 acc[MI][J];
#pragma unroll
  for (int i = 0; i < MI; ++i)
#pragma unroll
    for (int j = 0; j < J; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.f;
  auto compute = [&](int s) {
    const uint8_t* st = smem + (s % NST) * kStage;
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      i32x8 af[MI], bf[J];
#pragma unroll
      for (int j = 0; j < J; ++j) {
        const u32x4 lo = *reinterpret_cast<const u32x4*>(st + offb[k][0] + j * 32 * kQBK);
        const u32x4 hi = *reinterpret_cast<const u32x4*>(st + offb[k][1] + j * 32 * kQBK);
        bf[j] = i32x8{(int)lo.x, (int)lo.y, (int)lo.z, (int)lo.w, (int)hi.x, (int)hi.y, (int)hi.z, (int)hi.w};
      }
#pragma unroll
      for (int i = 0; i < MI; ++i) {
        const u32x4 lo = *reinterpret_cast<const u32x4*>(st + offa[k][0] + i * 32 * kQBK);
        const u32x4 hi = *reinterpret_cast<const u32x4*>(st + offa[k][1] + i * 32 * kQBK);
        af[i] = i32x8{(int)lo.x, (int)lo.y, (int)lo.z, (int)lo.w, (int)hi.x, (int)hi.y, (int)hi.z, (int)hi.w};
      }
      // B first: the accumulator is the transposed tile (a lane holds one
      // output row, four of every eight columns).
#pragma unroll
      for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int j = 0; j < J; ++j) acc[i][j] = mfma32(bf[j], af[i], acc[i][j]);
    }
  };

  // At stage s the wave waits for its LDS reads (of stage s-1) and its own
  // loads of stage s (the younger stages stay in flight), then meets the other
  // waves: stage s is complete in LDS and every wave is done with the slot of
  // stage s-1, which then takes stage s+NST-1.
  if constexpr (PART) {
    issue(0, kt.first);
    for (int s = 1; s < NST - 1 && s < stages; ++s) issue(s, s * kQBK);
    wait_loads<PER>(min(stages - 1, NST - 2));
    asm volatile("" ::: "memory");
    if (kt.back)
#pragma unroll
      for (int i = 0; i < PER; ++i)
        if (wave + i * NW < BM / 8) *reinterpret_cast<u32x4*>(smem + (wave + i * NW) * 1024 + lane * 16) = u32x4{0u, 0u, 0u, 0u};
  } else {
    for (int s = 0; s < NST - 1 && s < stages; ++s) issue(s, (s0 + s) * kQBK);
  }
  for (int s = 0; s < stages; ++s) {
    JO_WAIT_LDS0();
    wait_loads<PER>(min(stages - 1 - s, NST - 2));
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    if (s + NST - 1 < stages) issue(s + NST - 1, (s0 + s + NST - 1) * kQBK);
    compute(s);
  }

  if constexpr (SPLIT) {
    // The partial tile as fp32: a lane's four consecutive columns per group
    // are one 16-byte store, and a row's 32 columns of a block (128 bytes)
    // leave in the four stores of one (i, j) back to back. Plain stores: the
    // reduction reads them back right away.
    float* wz = g.ws + static_cast<int64_t>(blockIdx.z) * g.M * g.N;
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
      for (int j = 0; j < J; ++j)
#pragma unroll
        for (int qq = 0; qq < 4; ++qq) {
          const int m = m0 + wm * WROWS + i * 32 + fr;
          const int n = n0 + wn * WCOLS + j * 32 + qq * 8 + fh * 4;
          // Each element through a scalar first: a bit_cast of a vector
          // element expression reads element 0 with this compiler.
          const float v0 = acc[i][j][qq * 4 + 0], v1 = acc[i][j][qq * 4 + 1];
          const float v2 = acc[i][j][qq * 4 + 2], v3 = acc[i][j][qq * 4 + 3];
          if (m < g.M && n < g.N)
            st16(wz + static_cast<int64_t>(m) * g.N + n,
                 u32x4{__builtin_bit_cast(uint32_t, v0), __builtin_bit_cast(uint32_t, v1),
                       __builtin_bit_cast(uint32_t, v2), __builtin_bit_cast(uint32_t, v3)});
        }
    return;
  }
  // Epilogue: the finished tile goes through LDS (free once every wave is past
  // the barrier) so that rows leave as whole 16-byte lane stores.
  float sam[MI];
#pragma unroll
  for (int i = 0; i < MI; ++i) sam[i] = g.sa[min(m0 + wm * WROWS + i * 32 + fr, g.M - 1)];
  float sbq[J][4][4], bq[J][4][4];
#pragma unroll
  for (int j = 0; j < J; ++j)
#pragma unroll
    for (int qq = 0; qq < 4; ++qq) {
      const int n = min(n0 + wn * WCOLS + j * 32 + qq * 8 + fh * 4, g.N - 4);  // N % 8 == 0
      const u32x4 sbv = ld16(g.sb + n);
      u32x4 b4{0u, 0u, 0u, 0u};
      if (g.bias) {
        const u32x2 braw = *reinterpret_cast<const u32x2*>(static_cast<const uint16_t*>(g.bias) + n);
        b4 = u32x4{braw.x, braw.y, 0u, 0u};
      }
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        sbq[j][qq][t] = elem<F32>(sbv, t);
        bq[j][qq][t] = g.bias ? elem<OutTag>(b4, t) : 0.f;
      }
    }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < MI; ++i)
#pragma unroll
    for (int j = 0; j < J; ++j)
#pragma unroll
      for (int qq = 0; qq < 4; ++qq) {
        float o[8];
#pragma unroll
        for (int t = 0; t < 4; ++t) {
          o[t] = __builtin_fmaf(sam[i], acc[i][j][qq * 4 + t] * sbq[j][qq][t], bq[j][qq][t]);
          o[t + 4] = 0.f;
        }
        const u32x4 pk = pack<OutTag>(o);
        const int rl = wm * WROWS + i * 32 + fr, cl = wn * WCOLS + j * 32 + qq * 8 + fh * 4;
        *reinterpret_cast<u32x2*>(smem + rl * kRowBytes + cl * 2) = u32x2{pk.x, pk.y};
      }
  __syncthreads();
  for (int c = tid; c < BM * kChunksPerRow; c += NW * kWave) {
    const int rl = c / kChunksPerRow, ch = c % kChunksPerRow;
    const int m = m0 + rl, n = n0 + ch * 8;
    if (m < g.M && n < g.N)
      st16_nt(static_cast<uint16_t*>(g.out) + static_cast<int64_t>(m) * g.ldo + n,
              *reinterpret_cast<const u32x4*>(smem + rl * kRowBytes + ch * 16));
  }
}

template <class OutTag, int BM, int BN, int NW, int NST, bool SPLIT, bool PART, int WGM>
__global__ __launch_bounds__(NW * 64) void fp8_gemm_small_kernel(const GemmArgs g) {
  fp8_gemm_small_body<OutTag, BM, BN, NW, NST, SPLIT, PART, WGM>(g);
}

// Split K, second pass: out[m, n] = epilogue of the sum over z of the
// partials ws[z, m, n], added in z order (so every run gives the same bits),
// eight columns a thread.
template <class OutTag>
__global__ __launch_bounds__(kBlock) void fp8_gemm_splitk_reduce(const GemmArgs g, int splits) {
  const int64_t cpr = g.N / 8;  // N % 8 == 0
  const int64_t c = static_cast<int64_t>(blockIdx.x) * kBlock + threadIdx.x;
  if (c >= static_cast<int64_t>(g.M) * cpr) return;
  const int64_t m = c / cpr;
  const int n = static_cast<int>(c - m * cpr) * 8;
  const int64_t plane = static_cast<int64_t>(g.M) * g.N;
  const float* p = g.ws + m * g.N + n;
  float acc[8];
  {
    const u32x4 lo = ld16(p), hi = ld16(p + 4);
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      acc[t] = elem<F32>(lo, t);
      acc[t + 4] = elem<F32>(hi, t);
    }
  }
  for (int z = 1; z < splits; ++z) {
    const u32x4 lo = ld16(p + z * plane), hi = ld16(p + z * plane + 4);
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      acc[t] += elem<F32>(lo, t);
      acc[t + 4] += elem<F32>(hi, t);
    }
  }
  const float sa = g.sa[m];
  const u32x4 s0 = ld16(g.sb + n), s1 = ld16(g.sb + n + 4);
  u32x4 braw{0u, 0u, 0u, 0u};
  if (g.bias) braw = ld16(static_cast<const uint16_t*>(g.bias) + n);
  float o[8];
#pragma unroll
  for (int t = 0; t < 8; ++t) {
    const float sb = t < 4 ? elem<F32>(s0, t) : elem<F32>(s1, t - 4);
    o[t] = __builtin_fmaf(sa, acc[t] * sb, g.bias ? elem<OutTag>(braw, t) : 0.f);
  }
  st16_nt(static_cast<uint16_t*>(g.out) + m * g.ldo + n, pack<OutTag>(o));
}

template <class OutTag, int BM, int BN, int NW, int NST, int WGM = 2>
void launch_small(const GemmArgs& g, hipStream_t stream, int splits = 1) {
  const dim3 grid((g.N + BN - 1) / BN, (g.M + BM - 1) / BM, splits);
  if (g.K % kQBK != 0) {  // never split
    hipLaunchKernelGGL((fp8_gemm_small_kernel<OutTag, BM, BN, NW, NST, false, true, WGM>), grid,
                       dim3(NW * 64), 0, stream, g);
    return;
  }
  if (splits == 1) {
    hipLaunchKernelGGL((fp8_gemm_small_kernel<OutTag, BM, BN, NW, NST, false, false, WGM>), grid,
                       dim3(NW * 64), 0, stream, g);
    return;
  }
  hipLaunchKernelGGL((fp8_gemm_small_kernel<OutTag, BM, BN, NW, NST, true, false, WGM>), grid, dim3(NW * 64),
                     0, stream, g);
  const int64_t chunks = static_cast<int64_t>(g.M) * (g.N / 8);
  hipLaunchKernelGGL((fp8_gemm_splitk_reduce<OutTag>), dim3(static_cast<unsigned>((chunks + kBlock - 1) / kBlock)),
                     dim3(kBlock), 0, stream, g, splits);
}

// ---------------------------------------------------------------------------
// Streaming kernel, for up to 80 rows: the weight is read once and that is
// what the time should go to. A workgroup of eight waves takes BM = 16 MB rows
// (all of them) x BN = 16 NB columns, so one wave's fragments are used by no
// other; its waves split K instead, wave w taking the 128-byte steps w, w + 8,
// ... of every row. Each brings its steps through an LDS region of its own
// (direct loads of whole lines, the pair kernel's row layout) and waits for
// nothing but its own loads: there is no barrier in the loop, and the other
// waves' loads are in flight meanwhile. The partial tiles meet in LDS at the
// end and are added in wave order (the same bits on every run).
// Measured against the small-tile kernel, us, weights from HBM / cached:
// 1x4096x4096 11.4 -> 6.8 / 10.0 -> 4.0, 40x4096x4096 11.9 -> 7.8 / 10.1 -> 5.9,
// 77x4096x4096 11.5 -> 9.7 / 10.1 -> 7.7, 77x12288x4096 16.8 -> 15.2 / 16.0 -> 12.4,
// 1x12288x4096 13.5 -> 11.8 / 10.7 -> 9.3, 24x3072x3072 9.5 -> 5.4 / 8.2 -> 3.6.
// About 4 us of it are the launch, the first loads' latency and the last
// exchange; at 77 rows every workgroup also reads 320 KB of A from its L2.
// Fragments loaded straight into registers in MFMA layout (64 bytes a row and
// load instead of whole lines) measured 20.4 / 17.8 at 77x12288x4096;
// nontemporal loads of B 14.9 / 14.3 (77x16384x4096 18.2 / 17.7): nothing of the
// weight is then found in the Infinity Cache on a repeat.
// ---------------------------------------------------------------------------
constexpr int kStreamLds = 152 * 1024;

constexpr int kStreamWaves = 8;
// Five row blocks: what four column blocks leave room for in LDS. Up to 128 rows
// would fit with fewer columns; between 81 and 127 that is not measured, 128 rows
// were slower.
constexpr int kStreamRows = 80;

template <int MB, int NB>
struct StreamShape {
  static constexpr int NW = kStreamWaves;
  static constexpr int kPitch = NB * 16 + 4;                 // floats of a staged row
  static constexpr int kBlock = NW * 16 * kPitch * 4;        // bytes of a staged row block
  static constexpr int kPass = kStreamLds / kBlock < MB ? kStreamLds / kBlock : MB;
  static constexpr int kStep = (MB + NB) * 2048;             // bytes of a wave's step
  static constexpr int kMain = NW * kStep > kPass * kBlock ? NW * kStep : kPass * kBlock;
  static constexpr int kScales = MB * 16 * 4 + NB * 16 * 4 + NB * 16 * 2;
  static_assert(NW * kStep <= kStreamLds && kMain + 1024 + kScales <= 160 * 1024, "LDS");
};

template <int MB, int NB>
__device__ __forceinline__ void fp8_gemm_stream_body(const GemmArgs& g, int out_bf16) {
  using Sh = StreamShape<MB, NB>;
  constexpr int NW = kStreamWaves;
  constexpr int BN = NB * 16;
  __shared__ __attribute__((aligned(1024))) uint8_t smem[Sh::kMain + Sh::kScales];
  const int tid = threadIdx.x;
  const int lane = tid % kWave;
  const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
  const int fr = lane & 15, fh = lane >> 4;
  const int n0 = blockIdx.x * BN;
  const int steps = g.K / kQBK, left = g.K % kQBK;  // whole steps, bytes of a last, partial one

  // Lane p of load slot L fills row 8 L + p / 8 of the step (A rows, then B^T
  // rows), chunk position p % 8, with the global chunk that belongs there.
  // Rows past M (N) read row M - 1 (N - 1) and are never stored.
  uint8_t* mine = smem + wave * Sh::kStep;
  uint32_t off[(MB + NB) * 2];
#pragma unroll
  for (int i = 0; i < (MB + NB) * 2; ++i) {
    const int r = (i < MB * 2 ? i : i - MB * 2) * 8 + lane / 8;
    const int row = i < MB * 2 ? min(r, g.M - 1) : min(n0 + r, g.N - 1) - n0;
    off[i] = static_cast<uint32_t>(row) * static_cast<uint32_t>(i < MB * 2 ? g.lda : g.ldb) +
             (((lane & 7) ^ qswz(r)) * 16);
  }
  const uint8_t* pb = g.b + static_cast<int64_t>(n0) * g.ldb;
  auto issue = [&](int s) {
#pragma unroll
    for (int i = 0; i < (MB + NB) * 2; ++i) {
      // A chunk past K reads the row's first chunk of the step.
      const int c = ((lane & 7) ^ qswz((i & 1) * 8 + lane / 8)) * 16;
      const uint32_t k = s * kQBK - (s == steps && c >= left ? c : 0);
      __attribute__((address_space(3))) void* dst = (__attribute__((address_space(3))) void*)(mine + i * 1024);
      __builtin_amdgcn_global_load_lds((i < MB * 2 ? g.a : pb) + (off[i] + k), dst, 16, 0, 0);
    }
  };
  // Scales and bias, the oldest loads of the last wave.
  uint8_t* scales = smem + Sh::kMain;
  if (wave == NW - 1) {
    auto load4 = [&](const void* src, int at) {
      __builtin_amdgcn_global_load_lds(static_cast<const uint8_t*>(src), (__attribute__((address_space(3))) void*)(scales + at), 4, 0, 0);
    };
#pragma unroll
    for (int r = 0; r < MB * 16; r += kWave)
      if (r + lane < MB * 16) load4(g.sa + min(r + lane, g.M - 1), r * 4);
    if (lane < BN) load4(g.sb + min(n0 + lane, g.N - 1), MB * 64);
    if (g.bias && lane < BN / 2) load4(static_cast<const uint16_t*>(g.bias) + min(n0 + lane * 2, g.N - 2), MB * 64 + BN * 4);
  }

  f32x4 acc[MB][NB];
#pragma unroll
  for (int i = 0; i < MB; ++i)
#pragma unroll
    for (int j = 0; j < NB; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  int at[2];
#pragma unroll
  for (int h = 0; h < 2; ++h) at[h] = fr * kQBK + (((fh * 2 + h) ^ qswz(fr)) << 4);
  const int all = steps + (left != 0 ? 1 : 0);
  if (wave < all) issue(wave);
  for (int s = wave; s < all; s += NW) {
    JO_WAIT_VM(0);
    asm volatile("" ::: "memory");
    i32x8 af[MB], bf[NB];
    auto frag = [&](int block) {
      const u32x4 lo = *reinterpret_cast<const u32x4*>(mine + block * 2048 + at[0]);
      const u32x4 hi = *reinterpret_cast<const u32x4*>(mine + block * 2048 + at[1]);
      return i32x8{(int)lo.x, (int)lo.y, (int)lo.z, (int)lo.w, (int)hi.x, (int)hi.y, (int)hi.z, (int)hi.w};
    };
#pragma unroll
    for (int j = 0; j < NB; ++j) bf[j] = frag(MB + j);
#pragma unroll
    for (int i = 0; i < MB; ++i) af[i] = frag(i);
    if (s == steps) {  // A past K: zero
#pragma unroll
      for (int i = 0; i < MB; ++i)
#pragma unroll
        for (int e = 0; e < 8; ++e)
          if ((fh * 2 + e / 4) * 16 >= left) af[i][e] = 0;
    }
    // The fragments are held before the region is filled again.
    JO_WAIT_LDS0();
    asm volatile("" ::: "memory");
    if (s + NW < all) issue(s + NW);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < MB; ++i)
#pragma unroll
      for (int j = 0; j < NB; ++j) acc[i][j] = mfma16(bf[j], af[i], acc[i][j]);
  }
  JO_WAIT_VM(0);  // a wave without steps may have loaded scales

  // Lane: row i*16 + lane%16 of the tile, columns j*16 + (lane/16)*4 .. +3.
  constexpr int kQuads = BN / 4;
  constexpr int kPlane = Sh::kPass * 16 * Sh::kPitch;
  float* part = reinterpret_cast<float*>(smem);
#pragma unroll
  for (int i0 = 0; i0 < MB; i0 += Sh::kPass) {
    __syncthreads();  // every wave is done with its region, or the previous pass
#pragma unroll
    for (int i = i0; i < i0 + Sh::kPass && i < MB; ++i)
#pragma unroll
      for (int j = 0; j < NB; ++j)
        *reinterpret_cast<f32x4*>(part + wave * kPlane + ((i - i0) * 16 + fr) * Sh::kPitch + j * 16 + fh * 4) = acc[i][j];
    __syncthreads();
    const int rows = (MB - i0 < Sh::kPass ? MB - i0 : Sh::kPass) * 16;
    for (int c = tid; c < rows * kQuads; c += NW * kWave) {
      const int r = c / kQuads, col = c % kQuads * 4, n = n0 + col, m = i0 * 16 + r;
      if (m >= g.M || n >= g.N) continue;
      const float* p = part + r * Sh::kPitch + col;
      f32x4 v = *reinterpret_cast<const f32x4*>(p);
#pragma unroll
      for (int w = 1; w < NW; ++w) v += *reinterpret_cast<const f32x4*>(p + w * kPlane);
      {
        const float sa = *reinterpret_cast<const float*>(scales + (i0 * 16 + r) * 4);
        const u32x4 sbv = *reinterpret_cast<const u32x4*>(scales + MB * 64 + col * 4);
        const u32x2 braw = *reinterpret_cast<const u32x2*>(scales + MB * 64 + BN * 4 + col * 2);
        const u32x4 b4{braw.x, braw.y, 0u, 0u};
        float o[8];
#pragma unroll
        for (int t = 0; t < 4; ++t) {
          const float bias = !g.bias ? 0.f : out_bf16 ? elem<BF16>(b4, t) : elem<F16>(b4, t);
          o[t] = __builtin_fmaf(sa, v[t] * elem<F32>(sbv, t), bias);
          o[t + 4] = 0.f;
        }
        const u32x4 pk = out_bf16 ? pack<BF16>(o) : pack<F16>(o);
        *reinterpret_cast<u32x2*>(static_cast<uint16_t*>(g.out) + static_cast<int64_t>(m) * g.ldo + n) = u32x2{pk.x, pk.y};
      }
    }
  }
}

template <int MB, int NB>
__global__ __launch_bounds__(kStreamWaves * 64, 1) void fp8_gemm_stream_kernel(const GemmArgs g, int out_bf16) {
  fp8_gemm_stream_body<MB, NB>(g, out_bf16);
}

// The widths that are built: three or four row blocks of 64 columns were the
// fastest choice on none of 220 shapes.
constexpr bool stream_built(int mb, int nb) { return nb <= 3 || mb <= 2 || mb == 5; }

// The kernel of mb x nb row and column blocks.
template <int MB = kStreamRows / 16, int NB = 4>
void launch_stream(const GemmArgs& g, int mb, int nb, int bf16, hipStream_t stream) {
  if constexpr (MB > 1) {
    if (mb < MB) return launch_stream<MB - 1, NB>(g, mb, nb, bf16, stream);
  }
  if constexpr (NB > 1) {
    if (nb < NB) return launch_stream<MB, NB - 1>(g, mb, nb, bf16, stream);
  }
  if constexpr (stream_built(MB, NB))
    hipLaunchKernelGGL((fp8_gemm_stream_kernel<MB, NB>), dim3((g.N + NB * 16 - 1) / (NB * 16)),
                       dim3(kStreamWaves * 64), 0, stream, g, bf16);
}

// CUs of the current device (queried once per device; 256, MI355X's count,
// if the query fails).
int cu_count() {
  static std::atomic<int> cached[64];
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 256;
  int n = cached[dev].load(std::memory_order_relaxed);
  if (n == 0) {
    if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0) n = 256;
    cached[dev].store(n, std::memory_order_relaxed);
  }
  return n;
}

// Launch shapes. kPair + rows: the eight-wave pair kernel with tiles of that
// many rows x 256 columns (a multiple of 16 from 96 to 256); 2: the
// register-staged kernel; 5, 6, 8, 10, 11, 12: the small-tile kernel.
// kStream + 16 NB: the streaming kernel with NB column blocks.
constexpr int kPair = 1000;
constexpr int kStream = 2000;

// Cost of a pair-kernel launch and of a small-tile one in the same unit, a
// small-tile kernel's operand bytes per K byte on the busiest CU (those run at
// about 49 KB/us a CU). The pair kernel's stage takes about 9.6 rows + 80
// cycles (measured 2450 at 256 rows, 2075 at 208, 1560 at 160, 1325 at 128: the
// MFMAs), a fifth of that in the unit above at ~2.1 GHz; low tiles are priced
// higher, by the 32 KB of B a stage that they wait on when the weight comes
// from HBM ([256, 16384] x 4096 in a whole MLP: 96-row tiles 4 us slower than
// the 128x128 ones, though level with cached weights).
// Up to 128 rows in one row of tiles and a long K: no two workgroups share B
// then, and a CU draws its 32 KB a stage from HBM in the time of 23,500, so 128x192
// tiles are faster where they fit one round (us, weights from HBM, 96- or
// 112-row tiles / 128x192: 74x39720x3840 36.2 / 33.4, 101x35392x4096 41.2 / 39.6;
// with K up to 1280 the pair kernel is: 71x32912x1024 12.3 / 13.2).
bool one_row(int M, int K) { return M <= 128 && K > 1280; }

int64_t pair_cost(int cus, int M, int N, int K, int rows) {
  const int64_t tiles = static_cast<int64_t>((M + rows - 1) / rows) * ((N + 255) / 256);
  int64_t stage = 96 * rows + 800 > 56 * rows + 8500 ? 96 * rows + 800 : 56 * rows + 8500;
  if (one_row(M, K) && M <= rows && stage < 23500) stage = 23500;
  return (tiles + cus - 1) / cus * stage / 50;
}

int64_t small_cost(int cus, int M, int N, int bm, int bn) {
  const int64_t tiles = static_cast<int64_t>((M + bm - 1) / bm) * ((N + bn - 1) / bn);
  return (tiles + cus - 1) / cus * (bm + bn);
}

// The default launch shape, the cheapest of: the pair kernel at every tile
// height (one workgroup per CU, so what counts is rounds of workgroups times
// the height, and a height that divides M into whole rounds wastes least: 3120
// rows are fifteen 208-row tiles, 240 workgroups for 256 CUs at N = 4096), and
// the small-tile kernel at 128x128, 128x96, 64x128, 64x96 or 64x64 where the
// 256-column tiles leave CUs idle (ties go to the smaller tile: two 64x64
// workgroups share a CU). The 96-column tiles cut N = 12288 into 128 columns
// of tiles, so 128 or 256 rows fill the 256 CUs. Measured on MI355X against
// the choice of 224- or 256-row tiles (32x32x64 MFMAs) and 128x192 / 128x256
// small tiles: [3120, 4096] x 4096 45.0 -> 42.7 us (208 rows), [1560, 12288] x
// 4096 78.4 -> 69.1 (160), [1560, 4096] x 4096 32.2 -> 25.9 (112), [1560, 4096]
// x 16384 118 -> 101 (112), [512, 12288] x 4096 30.6 -> 25.7 (128); the
// small tiles at M = 256: [256, 4096] x 4096 34.2 -> 11.4 us (64x64),
// [256, 12288] x 4096 42.4 -> 22.0 us (128x96).
int auto_shape(int cus, int M, int N, int K) {
  int shape = 0;
  int64_t best = INT64_MAX;
  for (int rows = 256; rows >= 96; rows -= 16) {
    const int64_t c = pair_cost(cus, M, N, K, rows);
    if (c < best) {
      best = c;
      shape = kPair + rows;
    }
  }
  // Larger tiles first: a tie goes to the smaller one.
  const int small[6][3] = {{12, 128, 192}, {5, 128, 128}, {10, 128, 96}, {8, 64, 128}, {11, 64, 96}, {6, 64, 64}};
  for (const auto& t : small) {
    if (t[0] == 12 && !one_row(M, K)) continue;
    const int64_t c = small_cost(cus, M, N, t[1], t[2]);
    if (c <= best) {
      best = c;
      shape = t[0];
    }
  }
  return shape;
}

// Split K, for few tiles and a long K (the text stream's MLP down: [256,
// 16384] x [16384, 4096] is 64 tiles of 128x128): S workgroups share each
// tile's K stages and write fp32 partials that a second kernel adds up in a
// fixed order (the same bits on every run) under the epilogue. Taken by the
// small-tile kernel at 128x128 or 64x64 when the caller passes a workspace of
// S x M x N x 4 bytes and it cuts the cost above by 15% or more: the busiest
// CU's operand bytes, plus the partials written and read back (they stay in
// the caches: counted at half an operand byte) and a fixed ~9 us for the
// second launch and the first one's tail (405 KB at the operand rate), fitted
// on MI355X: [64, 4096] x 16384 38.8 -> 22.5 us, [256, 4096] x 16384 39.2 ->
// 34.4 us, [512, 4096] x 16384 65.9 -> 51.7 us; [512, 4096] x 4096 stays
// unsplit (16.5 us; split in two, 20.6).
constexpr int64_t kSplitCap = int64_t{1} << 30;  // largest partial buffer a split uses

// Estimated time of the streaming kernel, ns: the launch, first loads and last
// exchange; the busiest CU's rows of A (72 KB/us) and columns of B (39 KB/us),
// or B at what HBM gives all CUs (5.25 TB/s) with a part of A beside it,
// whichever is longer; what a row block, a workgroup and a block of the exchange
// cost; and, with rows a multiple of 8 KB apart, whose lines fall on the same
// channels, 4 us where narrow tiles keep most CUs at it (64x8192x8192 21.9 us,
// x6144 14.8). The constants here and in plan_gemm are fitted to 770 shapes (1 to
// 80 rows, N 512 to 16384, K 512 to 16384), each of the four widths measured on
// each with the weight from HBM and cached: 0.96 of the time that the best
// choices save is saved, and four shapes are slower than with the kernel that
// streaming replaces, by 2-3% (80x8192x4096, x5120 and 64x9216x512) or with a
// cached weight only (16x3072x16384 13.6 -> 14.8; from HBM 16.5 -> 15.1).
int64_t stream_ns(int M, int N, int K, int nb) {
  const int64_t tiles = (N + nb * 16 - 1) / (nb * 16);  // at most one a CU
  const int64_t mb = (M + 15) / 16, a = mb * 16 * K, b = static_cast<int64_t>(nb) * 16 * K;
  const int64_t cu = a / 72 + b / 39, hbm = static_cast<int64_t>(N) * K * 4 / 21000 + a / 200;
  const int64_t channels = K % 8192 == 0 && mb >= 3 && nb <= 2 && tiles > 192 ? 4000 : 0;
  return 3000 + (cu > hbm ? cu : hbm) + 150 * mb + tiles + 36 * mb * nb + channels;
}

struct GemmPlan {
  int shape;
  int splits;
};

int64_t split_bytes(int M, int N, int splits) {
  return splits > 1 ? static_cast<int64_t>(splits) * M * N * 4 : 0;
}

int64_t shape_cost(int cus, int shape, int M, int N, int K) {
  switch (shape) {
    case 5: return small_cost(cus, M, N, 128, 128);
    case 6: return small_cost(cus, M, N, 64, 64);
    case 8: return small_cost(cus, M, N, 64, 128);
    case 10: return small_cost(cus, M, N, 128, 96);
    case 11: return small_cost(cus, M, N, 64, 96);
    case 12: return small_cost(cus, M, N, 128, 192);
    default: return pair_cost(cus, M, N, K, shape - kPair);
  }
}

// Cost of `splits` workgroups sharing each bm x bn small tile's K.
int64_t split_cost(int cus, int M, int N, int K, int bm, int bn, int splits) {
  const int64_t tiles = static_cast<int64_t>((M + bm - 1) / bm) * ((N + bn - 1) / bn);
  return (tiles * splits + cus - 1) / cus * (bm + bn) * (K / splits) + split_bytes(M, N, splits) / cus +
         405 * 1024;
}

// The launch shape that a JO_KNOB_GEMM_SHAPE value forces.
int knob_shape(int v) {
  constexpr int kShape[12] = {kPair + 256, kPair + 208, 2, kPair + 224, kPair + 160, 5, 6, kPair + 128, 8, kPair + 112, 10, 11};
  return kShape[v];
}

GemmPlan plan_gemm(const GemmArgs& g, int64_t ws_bytes) {
  const int forced = launch_knob(JO_KNOB_GEMM_SHAPE);
  const int fsplit = launch_knob(JO_KNOB_GEMM_SPLIT);
  const int cus = cu_count();
  GemmPlan p{forced >= 0 ? knob_shape(forced) : auto_shape(cus, g.M, g.N, g.K), 1};
  const int64_t room = ws_bytes < kSplitCap ? ws_bytes : kSplitCap;
  auto split_ok = [&](int sp) {
    return g.K > 0 && g.K % (kQBK * sp) == 0 && split_bytes(g.M, g.N, sp) <= room;
  };
  if (fsplit >= 1) {
    if ((p.shape == 5 || p.shape == 6) && split_ok(fsplit)) p.splits = fsplit;
    return p;
  }
  if (forced >= 0) return p;
  const int64_t unsplit = shape_cost(cus, p.shape, g.M, g.N, g.K) * g.K;
  int64_t best = -1;
  GemmPlan split{p.shape, 1};
  const int cand[2][3] = {{5, 128, 128}, {6, 64, 64}};
  for (const auto& c : cand)
    for (int sp = 2; sp <= 8; sp *= 2)
      if (split_ok(sp)) {
        const int64_t cost = split_cost(cus, g.M, g.N, g.K, c[1], c[2], sp);
        if (best < 0 || cost < best) {
          best = cost;
          split = GemmPlan{c[0], sp};
        }
      }
  const bool splits = best >= 0 && best * 20 < unsplit * 17;
  if (splits) p = split;
  // Few rows: the streaming kernel where it is estimated faster than the
  // choice so far: 4.25 us and its operand bytes at 54 KB/us a CU (59 with two
  // tile rows), or the weight at 5.3 TB/s; 1 us more for the two waves of 64x96
  // tiles; with a split 10 us for the two launches and 75 KB/us, or 30 where
  // workgroups share a CU (streaming was faster on every such shape). A weight
  // that comes from HBM decides most of them: 80x2048x6144 10.6 us split in four,
  // 12.3 streamed (cached 9.5 and 7.1). Only where one round of workgroups takes
  // all columns: past that the short K's measured up to half slower
  // (57x17632x128 5.1 -> 7.6).
  if (g.M <= kStreamRows) {
    const int64_t draw = unsplit / (g.M > 64 ? 59 : 54), weight = static_cast<int64_t>(g.N) * g.K / 5300;
    int64_t other = 4250 + (draw > weight ? draw : weight) + (p.shape == 11 ? 1000 : 0);
    if (splits) {
      const int64_t t = split.shape == 5 ? 128 : 64;
      const int64_t wgs = (g.M + t - 1) / t * ((g.N + t - 1) / t) * split.splits, per = (wgs + cus - 1) / cus;
      other = 10000 + per * 2 * t * (g.K / split.splits) / (per > 1 ? 30 : 75);
    }
    for (int nb = 1; nb <= 4; ++nb) {
      if (g.N > cus * nb * 16 || !stream_built((g.M + 15) / 16, nb)) continue;
      const int64_t ns = stream_ns(g.M, g.N, g.K, nb);
      if (ns < other) {
        other = ns;
        p = GemmPlan{kStream + nb * 16, 1};
      }
    }
  }
  return p;
}

template <class OutTag>
int launch_gemm(const GemmArgs& g, hipStream_t stream, int64_t ws_bytes) {
  const dim3 grid((g.N + kBN - 1) / kBN, (g.M + kBM - 1) / kBM);
  // K == 0 takes the register-staged kernel, which loads no operand bytes
  // when K is 0 and stores the epilogue of a zero accumulator (the bias).
  const bool direct_ok = g.K > 0 && aligned(g.sb, 16) && (g.bias == nullptr || aligned(g.bias, 8)) &&
                         256 * (g.lda > g.ldb ? g.lda : g.ldb) + g.K <= int64_t{UINT32_MAX};
  // The JO_KNOB_GEMM_SHAPE override forces a shape (knob_shape; results are the
  // same up to the fp32 accumulation order inside the matrix cores).
  const GemmPlan plan = plan_gemm(g, ws_bytes);
  const int shape = plan.shape;
  if (!direct_ok || shape == 2)
    hipLaunchKernelGGL((fp8_gemm_kernel<OutTag>), grid, dim3(kBlock), 0, stream, g);
  else if (shape == 5)
    launch_small<OutTag, 128, 128, 4, 4>(g, stream, plan.splits);
  else if (shape == 6)
    launch_small<OutTag, 64, 64, 4, 4>(g, stream, plan.splits);
  else if (shape == 8)
    launch_small<OutTag, 64, 128, 4, 4>(g, stream);
  else if (shape == 10)
    launch_small<OutTag, 128, 96, 4, 4, 4>(g, stream);
  else if (shape == 11)
    launch_small<OutTag, 64, 96, 2, 4, 2>(g, stream);
  else if (shape == 12)
    launch_small<OutTag, 128, 192, 4, 3>(g, stream);
  else if (shape < kStream)
    launch_pair_rows<OutTag>(g, stream, shape - kPair);
  else
    launch_stream(g, (g.M + 15) / 16, (shape - kStream) / 16, std::is_same<OutTag, BF16>::value, stream);
  return launch_status("fp8_scaled_mm");
}

}  // namespace
}  // namespace jo

using namespace jo;

namespace {
int fp8_scaled_mm_impl(const void* mat_a, int64_t lda, const void* mat_b, int64_t ldb,
                       const float* scales_a, const float* scales_b, const void* bias, void* out,
                       int64_t ldo, int64_t M, int64_t N, int64_t K, int out_dtype,
                       void* workspace, int64_t workspace_bytes, void* stream) {
  const char* op = "fp8_scaled_mm";
  JO_REQUIRE(out_dtype == JO_DTYPE_BF16 || out_dtype == JO_DTYPE_F16,
             "out_dtype must be Half or BFloat16");
  JO_REQUIRE(M >= 0 && N >= 0 && K >= 0 && M <= INT32_MAX && N <= INT32_MAX && K <= INT32_MAX,
             "%s: bad shape", op);
  JO_REQUIRE(K % 16 == 0, "mat_a must be multiple of 16 bytes for memory alignment");
  JO_REQUIRE(N % 8 == 0, "out must be multiple of 16 bytes for memory alignment");
  JO_REQUIRE(lda >= K && ldb >= K && ldo >= N && lda % 16 == 0 && ldb % 16 == 0 && ldo % 8 == 0,
             "%s: row strides must cover the rows and keep 16-byte alignment", op);
  if (M == 0 || N == 0) return JO_OK;
  // With K == 0 no operand byte is read (torch hands zero-size views over as
  // null pointers), and the output is the epilogue of a zero accumulator.
  JO_REQUIRE((K == 0 || (mat_a && mat_b)) && scales_a && scales_b && out, "%s: null pointer", op);
  JO_REQUIRE(aligned(mat_a, 16) && aligned(mat_b, 16) && aligned(out, 16),
             "%s: operands must be 16-byte aligned", op);
  JO_REQUIRE(workspace_bytes >= 0 && (workspace_bytes == 0 || (workspace && aligned(workspace, 16))),
             "%s: workspace must be 16-byte aligned (or 0 bytes)", op);
  GemmArgs g{static_cast<const uint8_t*>(mat_a), static_cast<const uint8_t*>(mat_b), scales_a,
             scales_b, bias, out, lda, ldb, ldo, static_cast<int>(M), static_cast<int>(N),
             static_cast<int>(K), static_cast<float*>(workspace)};
  hipStream_t st = static_cast<hipStream_t>(stream);
  return out_dtype == JO_DTYPE_BF16 ? launch_gemm<BF16>(g, st, workspace_bytes)
                                    : launch_gemm<F16>(g, st, workspace_bytes);
}
}  // namespace

extern "C" int jo_fp8_scaled_mm(const void* mat_a, int64_t lda, const void* mat_b, int64_t ldb,
                                const float* scales_a, const float* scales_b, const void* bias,
                                void* out, int64_t ldo, int64_t M, int64_t N, int64_t K,
                                int out_dtype, void* stream) {
  return fp8_scaled_mm_impl(mat_a, lda, mat_b, ldb, scales_a, scales_b, bias, out, ldo, M, N, K,
                            out_dtype, nullptr, 0, stream);
}

extern "C" int jo_fp8_scaled_mm_ws(const void* mat_a, int64_t lda, const void* mat_b,
                                   int64_t ldb, const float* scales_a, const float* scales_b,
                                   const void* bias, void* out, int64_t ldo, int64_t M, int64_t N,
                                   int64_t K, int out_dtype, void* workspace,
                                   int64_t workspace_bytes, void* stream) {
  return fp8_scaled_mm_impl(mat_a, lda, mat_b, ldb, scales_a, scales_b, bias, out, ldo, M, N, K,
                            out_dtype, workspace, workspace_bytes, stream);
}

// Allocation-free variant: the split-K partials go to this file-scope device
// array instead of a caller's workspace. Each GPU the library runs on holds
// its own copy (kScratchBytes) until the process ends. Host code never uses
// the array's name as an address (it is a host-side stand-in there): the
// device address comes from hipGetSymbolAddress, once per device.
constexpr int64_t kScratchBytes = int64_t{32} << 20;
static __device__ __align__(256) float scratch[kScratchBytes / 4];

namespace {
constexpr int kMaxDevices = 64;
std::atomic<void*> g_scratch[kMaxDevices];

// The current device's address of `scratch`, looked up on the first call on
// that device (with it current) and kept.
int scratch_address(void** out) {
  int dev = -1;
  const hipError_t ge = hipGetDevice(&dev);
  if (ge != hipSuccess || dev < 0 || dev >= kMaxDevices) {
    set_error("fp8_scaled_mm_noalloc: no usable current device (%s)", hipGetErrorString(ge));
    return JO_ERR_HIP;
  }
  void* p = g_scratch[dev].load(std::memory_order_acquire);
  if (p == nullptr) {
    const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess || p == nullptr) {
      set_error("fp8_scaled_mm_noalloc: hipGetSymbolAddress(scratch) failed on device %d: %s",
                dev, hipGetErrorString(e));
      return JO_ERR_HIP;
    }
    g_scratch[dev].store(p, std::memory_order_release);
  }
  *out = p;
  return JO_OK;
}
}  // namespace

extern "C" int64_t jo_fp8_scaled_mm_workspace_bytes(int64_t M, int64_t N, int64_t K) {
  if (M <= 0 || N <= 0 || K <= 0 || M > INT32_MAX || N > INT32_MAX || K > INT32_MAX) return 0;
  GemmArgs g{nullptr, nullptr, nullptr, nullptr, nullptr, nullptr, K, K, N,
             static_cast<int>(M), static_cast<int>(N), static_cast<int>(K)};
  const GemmPlan p = plan_gemm(g, kSplitCap);
  return split_bytes(g.M, g.N, p.splits);
}

extern "C" int jo_fp8_scaled_mm_plan(int64_t M, int64_t N, int64_t K, int32_t* plan) {
  JO_REQUIRE(M > 0 && N > 0 && K > 0 && M <= INT32_MAX && N <= INT32_MAX && K <= INT32_MAX,
             "fp8_scaled_mm_plan: bad shape");
  JO_REQUIRE(plan != nullptr, "fp8_scaled_mm_plan: null pointer");
  GemmArgs g{nullptr, nullptr, nullptr, nullptr, nullptr, nullptr, K, K, N,
             static_cast<int>(M), static_cast<int>(N), static_cast<int>(K)};
  const GemmPlan p = plan_gemm(g, kSplitCap);
  int kernel = JO_GEMM_SMALL, rows = 0, cols = 0;
  switch (p.shape) {
    case 2: kernel = JO_GEMM_STAGED; rows = kBM; cols = kBN; break;
    case 5: rows = 128; cols = 128; break;
    case 6: rows = 64; cols = 64; break;
    case 8: rows = 64; cols = 128; break;
    case 10: rows = 128; cols = 96; break;
    case 11: rows = 64; cols = 96; break;
    case 12: rows = 128; cols = 192; break;
    default:
      if (p.shape < kStream) {
        kernel = JO_GEMM_PAIR; rows = p.shape - kPair; cols = 256;
      } else {
        kernel = JO_GEMM_STREAM; rows = (g.M + 15) / 16 * 16; cols = p.shape - kStream;
      }
  }
  const int32_t found[4] = {kernel, rows, cols, p.splits};
  for (int i = 0; i < 4; ++i) plan[i] = found[i];
  return JO_OK;
}

extern "C" int jo_fp8_scaled_mm_noalloc(const void* mat_a, int64_t lda, const void* mat_b,
                                        int64_t ldb, const float* scales_a,
                                        const float* scales_b, const void* bias, void* out,
                                        int64_t ldo, int64_t M, int64_t N, int64_t K,
                                        int out_dtype, void* stream) {
  const int64_t need = jo_fp8_scaled_mm_workspace_bytes(M, N, K);
  JO_REQUIRE(need <= kScratchBytes,
             "fp8_scaled_mm_noalloc: the split-K partials of [%lld, %lld] x %lld need %lld bytes, "
             "more than the %lld-byte static scratch (jo_fp8_scaled_mm_ws takes a workspace of "
             "any size)",
             static_cast<long long>(M), static_cast<long long>(K), static_cast<long long>(N),
             static_cast<long long>(need), static_cast<long long>(kScratchBytes));
  void* ws = nullptr;
  if (need > 0) {
    const int st = scratch_address(&ws);
    if (st != JO_OK) return st;
  }
  return fp8_scaled_mm_impl(mat_a, lda, mat_b, ldb, scales_a, scales_b, bias, out, ldo, M, N, K,
                            out_dtype, ws, need, stream);
}
