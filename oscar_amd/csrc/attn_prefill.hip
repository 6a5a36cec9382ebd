// Causal GQA prefill over an optional INT2 history for gfx950 (MFMA bf16).
//
// Replaces oscar_ascend/kernels/prefill.py:69-72 / decode_kernel.py:70-117
// (fresh-only prefill: causal SDPA of the current chunk, original domain, bf16 out)
// and the long-continuation use of slab_attention.py:376-476 (history waves plus
// the causal current chunk, rotated domain, fp32 out + LSE).
//
// Query i (0-based in the chunk) sees keys [0, history + i + 1).
//
// Two launches when there is a history:
//   history_bf16_kernel  the history's K/V values with the reference rounding
//                        (q_dtype(fp16(code*scale + zero)), or the staged fp32 value
//                        when the seat's owner tag matches, prepare_kv.py:77) into a
//                        caller-provided bf16 workspace, once per call: every query
//                        tile of a long chunk reuses them;
//   prefill_kernel       flash attention over [workspace history | current chunk]: see there.
#include <type_traits>

#include "common.h"

namespace oscar {

namespace {

constexpr int kWaves = 4;
constexpr int kThreads = 256;
constexpr int kKeys = 32;
constexpr int kRows = 128;
constexpr float kLog2e = 1.4426950408889634f;
constexpr float kLn2 = 0.6931471805599453f;
constexpr int kLazy = 10;     // log2 of the largest row sum of a tile's probabilities before O is rescaled
// workgroups per CU the register budget of prefill_kernel<D> is set for
constexpr int prefill_wgs(int D) { return D == 256 ? 1 : 2; }
// PV runs on v_mfma_f32_32x32x16_f16 with P and V in fp16 for both query dtypes.  bf16
// V values (8-bit significands) are held as fp16(v * 2^-kVShift): exact for |v| from
// 2^-6 up to 2^23 (below, within 2^-17 absolutely), and O is scaled back by 2^kVShift.
constexpr int kVShift = 8;
typedef short __attribute__((ext_vector_type(4))) i16x4;
typedef __bf16 __attribute__((ext_vector_type(2))) bf16x2;
typedef _Float16 __attribute__((ext_vector_type(2))) f16x2;
typedef float __attribute__((ext_vector_type(2))) f32x2;

// the reference history value q_dtype(fp16(x)) (prepare_kv.py:77) as 16-bit bits
template <int QT>
__device__ __forceinline__ unsigned hist_bits(float x) {
  const __half h = __float2half_rn(x);
  if constexpr (QT == OSCAR_F16) return __half_as_ushort(h);
  else return f32_to_bf16_bits(__half2float(h));
}
// the PV operand bits of a value v already in the query dtype: fp16 as it is; a bf16
// value scaled by 2^-kVShift into fp16 (exact, see kVShift)
template <int QT>
__device__ __forceinline__ unsigned pv_bits(float v) {
  if constexpr (QT == OSCAR_F16) return f32_to_f16_bits(v);
  else return f32_to_f16_bits(v * (1.f / (1 << kVShift)));
}
// two packed bf16 values to their PV operand bits: fp16(v * 2^-kVShift), one
// mixed-precision multiply-add each
__device__ __forceinline__ unsigned pv_pair(unsigned w) {
  constexpr float k = 1.f / (1 << kVShift);
  unsigned d;
  asm volatile("v_fma_mixlo_f16 %0, %1, %2, 0" : "=v"(d) : "v"(w << 16), "s"(k));
  asm volatile("v_fma_mixhi_f16 %0, %1, %2, 0" : "+v"(d) : "v"(w & 0xffff0000u), "s"(k));
  return d;
}
template <int QT> struct QVec { typedef bf16x8 type; typedef bf16x2 pair; typedef __bf16 elem; };
template <> struct QVec<OSCAR_F16> { typedef f16x8 type; typedef f16x2 pair; typedef _Float16 elem; };

// four consecutive output elements from element i: the query dtype without a history
// (original domain), else fp32 rotated.  One store each, at whatever alignment the
// caller's output has.
template <int QT>
__device__ __forceinline__ void store_out(const oscar_prefill_args_v1& A, int64_t i, f32x4 v) {
  typedef u32x2 __attribute__((aligned(2))) u32x2_any;
  typedef f32x4 __attribute__((aligned(4))) f32x4_any;
  if (A.history != 0) {
    *(f32x4_any*)((float*)A.out + i) = v;
  } else {
    using Q2 = typename QVec<QT>::pair;
    *(u32x2_any*)((uint16_t*)A.out + i) =
        u32x2{__builtin_bit_cast(unsigned, __builtin_convertvector(f32x2{v[0], v[1]}, Q2)),
              __builtin_bit_cast(unsigned, __builtin_convertvector(f32x2{v[2], v[3]}, Q2))};
  }
}

// ---- balanced split of the key ranges (a workspace of oscar_prefill_workspace_bytes_v2)
// Query tile qt (kRows GQA rows) sees key tiles [0, kt(qt)), kt growing with qt under
// the causal mask.  One workgroup per tile leaves the chip unbalanced: the continuation
// of 15360 + 9256 tokens is 441 tiles of 481..771 key tiles on 256 CUs, a
// fresh 2048-token prefill 96 tiles (a third of the CUs).  The key range of a tile is
// instead cut into chunks of U key tiles (c U .. (c + 1) U), U a little over the work of
// half a CU, and every chunk is a unit (a workgroup takes one, or the same chunk of two
// neighbouring tiles); a tile with more than one chunk writes
// normalised partials + log2 LSEs, and prefill_merge_kernel combines them (FP32 LSE
// merge).  Units are numbered chunk-major, heaviest tile first within a chunk index,
// so the large units are dispatched first: the tiles that have a chunk c are the
// suffix qt >= qmin[c] (kt is non-decreasing in qt), and unit u of chunk class c
// (base[c] <= u < base[c + 1]) is tile ntq - 1 - (u - base[c]).
constexpr int kMaxChunks = 32;
constexpr int64_t kMinChunkTiles = 16;  // 512 keys: shorter chunks cost more in merge than they balance
constexpr int64_t kSplitCUs = 256;      // MI355X compute units
constexpr int64_t kUnitsPerCU = 2;

struct PrefillParams {
  oscar_prefill_args_v1 a;
  oscar_staging_v1 st;
  int has_stage;
  int group;
  int qtok;            // query tokens per workgroup
  uint16_t* hist_k;    // [history][Hk][D] bf16 history values (workspace)
  uint16_t* hist_v;
  // the split plan (split == 0: one unit per query tile, the whole key range)
  int split;
  int chunks;          // chunks of the heaviest tile
  int U;               // key tiles per chunk
  int ntq;             // query tiles
  int qmin1;           // first tile with two chunks (the split tiles are qt >= qmin1)
  int base[kMaxChunks + 1];
  int pbase[kMaxChunks + 1];  // first workgroup of chunk class c when a workgroup takes two query tiles
  float* part_o;       // [slot][Hk][kRows / 32][D / 32][4][64][4] normalised partial O of the split tiles'
                       // chunks, as the MFMA results lie (32 rows x 32 columns per 4 x 64 x 4)
  float* part_lse;     // [slot][Hk][kRows] log2-domain LSE of each partial
};

// key tiles seen by the last query of a tile ending at chunk token q1
__host__ __device__ inline int64_t tile_keys(int64_t hist, int64_t q1) { return (hist + q1 + kKeys - 1) / kKeys; }

struct SplitPlan {
  int chunks = 0, U = 0, ntq = 0, units = 0, qmin1 = 0;
  int base[kMaxChunks + 1] = {};
  int64_t slots = 0;   // partial slots per KV head
};

SplitPlan plan_split(int64_t hist, int64_t n, int64_t qtok, int64_t hk) {
  SplitPlan sp;
  if (n <= 0) return sp;
  const int64_t ntq = (n + qtok - 1) / qtok;
  auto kt = [&](int64_t qt) { return tile_keys(hist, (qt + 1) * qtok < n ? (qt + 1) * qtok : n); };
  int64_t work = 0;
  for (int64_t qt = 0; qt < ntq; ++qt) work += kt(qt);
  const int64_t kmax = kt(ntq - 1);
  int64_t U = (work * hk + kSplitCUs * kUnitsPerCU - 1) / (kSplitCUs * kUnitsPerCU);
  // a little over half a CU's share: the longest units, dispatched first, then fit one round
  // of the chip with the shorter ones filling the rest.  Exactly the share / with the term, in
  // us: 15360 + 9256 tokens of 6 heads on 1 1124 / 1050, 1600 over 8000 148 / 119, 3500 fresh
  // 102 / 72, 6000 fresh 169 / 175, 12 heads on 2, 3000 fresh 122 / 113, 24 on 4, 1600 fresh
  // 84 / 87, 8 heads of 128 on 1, 4000 fresh 76 / 64, 16 on 2, 4000 + 2000 119 / 112.  Two
  // thirds of the share and half of it: 15360 + 9256 13% and 6% above the term's.
  if (U + U / 32 + 3 < kmax) U += U / 32 + 3;
  if (U < kMinChunkTiles) U = kMinChunkTiles;
  if ((kmax + U - 1) / U > kMaxChunks) U = (kmax + kMaxChunks - 1) / kMaxChunks;
  const int64_t chunks = (kmax + U - 1) / U;
  if (chunks < 2 || ntq > (1 << 24) || U > (1 << 24)) return sp;
  sp.chunks = (int)chunks;
  sp.U = (int)U;
  sp.ntq = (int)ntq;
  // qmin[c]: first tile with kt > c U (kt non-decreasing in qt)
  int64_t qt = 0, units = 0;
  for (int c = 0; c < sp.chunks; ++c) {
    while (qt < ntq && kt(qt) <= c * U) ++qt;
    if (c == 1) sp.qmin1 = (int)qt;
    sp.base[c] = (int)units;
    units += ntq - qt;
  }
  sp.base[sp.chunks] = (int)units;
  sp.units = (int)units;
  sp.slots = units - sp.qmin1;  // every unit but the single-chunk tiles' (class 0, qt < qmin1)
  return sp;
}

constexpr int64_t kWsAlign = 256;
int64_t hist_bytes(int64_t history, int64_t hk, int64_t D) {
  return history > 0 ? (2 * history * hk * D * (int64_t)sizeof(uint16_t) + kWsAlign - 1) / kWsAlign * kWsAlign : 0;
}
int64_t split_bytes(const SplitPlan& sp, int64_t hk, int64_t D) {
  return sp.chunks < 2 ? 0 : sp.slots * hk * kRows * (D + 1) * (int64_t)sizeof(float);
}

// one wave per (history token, kv head): lane l holds elements E*l .. E*l+E-1
template <int D, int QT>
__global__ __launch_bounds__(256) void history_bf16_kernel(PrefillParams P) {
  constexpr int E = D / 64;
  const oscar_prefill_args_v1& A = P.a;
  const int64_t hk = A.num_kv_heads;
  const int64_t vec = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (vec >= A.history * hk) return;
  const int lane = threadIdx.x & 63;
  const int64_t p = vec / hk, h = vec % hk;
  const int64_t bs = A.cache.block_size;
  int64_t blk = A.block_table_row[p / bs];
  if (blk < 0 || blk >= A.cache.num_blocks) blk = 0;  // host validates; never fault
  const int64_t off = p % bs;
  int64_t seat = 0;
  bool staged = false;
  if (P.has_stage) {
    seat = (blk % P.st.rows) * bs + off;
    staged = P.st.owner[seat] == blk;
  }
  float kv[E], vv[E];
  if (staged) {
    const float* sk = P.st.stage_k + (seat * hk + h) * D + E * lane;
    const float* sv = P.st.stage_v + (seat * hk + h) * D + E * lane;
#pragma unroll
    for (int i = 0; i < E; ++i) { kv[i] = sk[i]; vv[i] = sv[i]; }
  } else {
    const uint8_t* ks = A.cache.k + blk * A.cache.k_stride[0] + off * A.cache.k_stride[1] + h * A.cache.k_stride[2];
    const uint8_t* vs = A.cache.v + blk * A.cache.v_stride[0] + off * A.cache.v_stride[1] + h * A.cache.v_stride[2];
    const unsigned m0 = *(const unsigned*)ks, m1 = *(const unsigned*)(ks + 4);
    const float sk = f16_bits_to_f32(m0 & 0xffff), zk = f16_bits_to_f32(m0 >> 16);
    const float sv = f16_bits_to_f32(m1 & 0xffff), zv = f16_bits_to_f32(m1 >> 16);
    const int e0 = E * lane;  // element e sits in byte e / 4, bits 2 (e % 4)
    const unsigned kb = ks[32 + e0 / 4], vb = vs[e0 / 4];
#pragma unroll
    for (int i = 0; i < E; ++i) {
      const int sh = 2 * ((e0 + i) & 3);
      kv[i] = __fadd_rn(__fmul_rn((float)((kb >> sh) & 3u), sk), zk);
      vv[i] = __fadd_rn(__fmul_rn((float)((vb >> sh) & 3u), sv), zv);
    }
  }
  unsigned kw[E / 2], vw[E / 2];
#pragma unroll
  for (int i = 0; i < E / 2; ++i) {
    kw[i] = hist_bits<QT>(kv[2 * i]) | (hist_bits<QT>(kv[2 * i + 1]) << 16);
    // V: the reference's history value in the query dtype, then the PV operand bits
    const unsigned v0 = hist_bits<QT>(vv[2 * i]), v1 = hist_bits<QT>(vv[2 * i + 1]);
    auto as_float = [](unsigned b) {
      return QT == OSCAR_F16 ? f16_bits_to_f32((unsigned short)b) : bf16_bits_to_f32((unsigned short)b);
    };
    vw[i] = pv_bits<QT>(as_float(v0)) | (pv_bits<QT>(as_float(v1)) << 16);
  }
  uint16_t* dk = P.hist_k + vec * D + E * lane;
  uint16_t* dv = P.hist_v + vec * D + E * lane;
  if constexpr (E == 4) {
    *(u32x2*)dk = u32x2{kw[0], kw[1]};
    *(u32x2*)dv = u32x2{vw[0], vw[1]};
  } else {
    *(unsigned*)dk = kw[0];
    *(unsigned*)dv = vw[0];
  }
}

// One 16-byte-per-lane LDS DMA: lane l's 16 bytes at `addr` land at LDS offset lds + 16 l.
// The wait is the caller's (vmcnt): the builtin form would make the compiler drain every
// load before each later LDS read.
__device__ __forceinline__ void dma16(unsigned lds, const void* addr) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off" ::"s"(lds), "v"(addr) : "m0", "memory");
}

// the same with a uniform base and a 32-bit byte offset
__device__ __forceinline__ void dma16(unsigned lds, uint64_t base, unsigned voff) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(lds), "v"(voff), "s"(base) : "m0", "memory");
}

// Every wave's LDS traffic is done and all but the last PENDING of this wave's DMA
// instructions have landed, then the workgroup barrier.
template <int PENDING>
__device__ __forceinline__ void tile_barrier() {
  asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(PENDING) : "memory");
}

// S (+)= K Q^T with S in VGPRs.  The builtin would put every accumulator of a kernel of
// more than 256 registers into AGPRs, and the softmax would copy S out; O stays there.
template <int QT, bool FIRST, class QV>
__device__ __forceinline__ void mfma_qk(f32x16& S, QV k, QV q) {
  if constexpr (QT == OSCAR_F16) {
    if constexpr (FIRST) asm volatile("v_mfma_f32_32x32x16_f16 %0, %1, %2, 0" : "=&v"(S) : "v"(k), "v"(q));
    else asm volatile("v_mfma_f32_32x32x16_f16 %0, %1, %2, %0" : "+v"(S) : "v"(k), "v"(q));
  } else {
    if constexpr (FIRST) asm volatile("v_mfma_f32_32x32x16_bf16 %0, %1, %2, 0" : "=&v"(S) : "v"(k), "v"(q));
    else asm volatile("v_mfma_f32_32x32x16_bf16 %0, %1, %2, %0" : "+v"(S) : "v"(k), "v"(q));
  }
}

// o *= f with o in an AGPR.  Written out so that O has no other home than the AGPRs: an
// ordinary product makes the compiler move all of O to VGPRs and back in every iteration.
__device__ __forceinline__ void scale_acc(float& o, float f) {
  float t;
  asm volatile("v_accvgpr_read_b32 %1, %0\n\tv_mul_f32 %1, %1, %2\n\tv_accvgpr_write_b32 %0, %1"
               : "+a"(o), "=&v"(t) : "v"(f));
}

// whole vectors in AGPRs here (vectors put together element by element would make the
// compiler carry O through the loop as single registers)
template <int N>
__device__ __forceinline__ void hold_acc(f32x16 (&o)[N]) {
#pragma unroll
  for (int b = 0; b < N; ++b) asm volatile("" : "+a"(o[b]));
}

// Flash attention of one unit: four waves, one per SIMD (D = 256), each with 32 NB query
// rows (tokens x heads of one KV head, GQA packed) over the unit's key tiles of 32.
// Per wave and tile: S^T = K Q^T (v_mfma_f32_32x32x16_bf16 / _f16, Q^T operands in
// registers), probabilities against a lazy reference max (fp32, log2 domain), O^T += V^T P^T
// on v_mfma_f32_32x32x16_f16 (P and V in fp16, see kVShift), V^T by ds_read_b64_tr_b16.
//
// Bound by the matrix cores' power and by what a wave can issue beside its MFMAs.  NB = 2
// needs 256 AGPRs (O) and all 256 VGPRs (Q^T 128, S 32, P 32, K operands two K-steps
// ahead; a third one spills Q^T), so one wave per SIMD, and that wave has to overlap its
// own MFMA and VALU work:
//  - PV of tile t - 1 runs beside the softmax of tile t, whose maximum is not waited for:
//    P is formed against the old reference, and only a row whose sum shows a large value
//    has it redone;
//  - an MFMA leaves room for about five other instructions (measured: 32.9 cycles with
//    four, 44 with eight, 5 each beyond), so the rest is dealt out between the MFMAs;
//  - the tile moves are LDS DMA (no registers, no ds_write), one beside every fourth MFMA
//    of QK (every second with NB = 1): issued together they cost 900 cycles a tile, spread
//    about 170;
//  - rare blocks (mask, moved reference, ragged tiles) are marked unlikely, so that the
//    loop is one run of code: in line they cost 800 of 3900 cycles a tile.
// Per K/V operand read from LDS NB MFMAs run.  15360 + 9256 tokens, 6 heads: 2.12 M cycles
// (1.04 to 1.1 ms at the 1.9 to 2.0 GHz the power allows), which is 3800 per 256 rows x 32
// keys of its longest units (558 key tiles), 2048 of them MFMA.  The layer's call with its
// other launches: 1880 us before (four waves of 32 rows, tiles through registers, one phase
// after the other), 1155 to 1200 us now, 0.98 PFLOP/s; a large library bf16 product reaches
// 1.2 to 1.36 on this card.
template <int D, int QT, int NB>
__global__ __launch_bounds__(kThreads, prefill_wgs(D)) void prefill_kernel(PrefillParams P) {
  using QV = typename QVec<QT>::type;    // one MFMA operand in the query dtype
  const oscar_prefill_args_v1& A = P.a;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int g = lane >> 5;
  const int G = P.group;
  const int kvh = blockIdx.y;
  const int64_t hist = A.history;
  const int64_t hk = A.num_kv_heads;
  // this wave's query tile qt and the workgroup's key tiles [kb, ke); slot >= 0: the
  // tile is split and this unit writes a partial.  NB == 2: waves 0-1 take the heavier
  // tile of a pair, waves 2-3 the next one (live: it has this chunk).
  int qt, kb = 0, ke, slot = -1;
  bool live = true;
  {
    const int u = blockIdx.x;
    int c = 0, idx;
    if (P.split) {
      const int* base = NB == 2 ? P.pbase : P.base;
#pragma unroll
      for (int cc = 1; cc < kMaxChunks; ++cc)
        if (cc < P.chunks && u >= base[cc]) c = cc;
      idx = NB * (u - base[c]);
      kb = c * P.U;
    } else {
      idx = NB * u;
    }
    const int qt_top = P.ntq - 1 - idx;  // heaviest (latest) query tiles first within a chunk class
    const int64_t q1_top = ((int64_t)qt_top + 1) * P.qtok;
    ke = (int)tile_keys(hist, q1_top < A.num_tokens ? q1_top : A.num_tokens);
    if (P.split && kb + P.U < ke) ke = kb + P.U;  // kb < ke (plan)
    if (NB == 2 && wave >= 2) {
      ++idx;
      live = idx < (P.split ? P.base[c + 1] - P.base[c] : P.ntq);
    }
    qt = live ? P.ntq - 1 - idx : qt_top;
    if (P.split && live && qt >= P.qmin1) slot = c == 0 ? idx : P.base[c] + idx - P.qmin1;
  }
  const int64_t q0 = (int64_t)qt * P.qtok;
  const int64_t q1 = (q0 + P.qtok < A.num_tokens) ? q0 + P.qtok : A.num_tokens;
  // this wave's own key tiles end at ke_own: the lighter tile of a pair may see fewer, and
  // must not multiply values past them (0 x inf; in the last of them see pv)
  int ke_own = (int)tile_keys(hist, q1);
  ke_own = !live || ke_own <= kb ? kb + 1 : ke_own < ke ? ke_own : ke;

  // Key tiles arrive by LDS DMA, 16 bytes a lane in lane order, so rows are not padded;
  // the 16-byte columns of a row are permuted instead (each lane asks for the column that
  // belongs at its place): K column c of key r at c ^ (r % 16), so that a row-per-lane
  // read covers all banks; V column c at c ^ 4 (r % VSW), so that the transpose reads of
  // 8 keys x 64 bytes do.  Three K tiles (t read, t + 1 and t + 2 in flight) and five V
  // tiles (t - 2 still read by slower waves, t - 1 read, t being converted to the PV
  // format, t + 1 and t + 2 in flight).
  constexpr int CPR = D / 8;             // 16-byte columns per key row
  constexpr int VSW = CPR / 4;           // 64-byte column groups per key row
  constexpr int ROWB = 2 * D;            // bytes per key row
  constexpr int TILEB = kKeys * ROWB;
  constexpr int RPI = 64 / CPR;          // key rows per DMA instruction
  constexpr int NDMA = kKeys / kWaves / RPI;  // DMA instructions per wave and tile
  constexpr int NK = 3, NV = 5;
  __shared__ __attribute__((aligned(1024))) uint8_t s_tiles[(NK + NV) * TILEB];
  typedef __attribute__((address_space(3))) uint8_t lds_u8;
  lds_u8* const lds = (lds_u8*)s_tiles;
  const unsigned lds0 = (unsigned)(uintptr_t)lds;
  const int hrow = (int)(hk * D * 2), crow = (int)(A.kv_stride_token * 2);  // bytes
  const uint64_t hist_k = (uint64_t)P.hist_k + kvh * ROWB, hist_v = (uint64_t)P.hist_v + kvh * ROWB;
  const uint64_t cur_k = (uint64_t)A.k + kvh * ROWB, cur_v = (uint64_t)A.v + kvh * ROWB;
  const unsigned ulane = lane;
  const int ihist = (int)hist, ikeys = (int)(hist + A.num_tokens);
  // a value behind a register the compiler cannot see through: what is derived from it is
  // computed where it is used instead of staying live across the loop, which has no
  // registers to spare
  auto fresh = [&](unsigned x) __attribute__((always_inline)) { asm volatile("" : "+v"(x)); return x; };
  // The DMAs of key tile kt: instruction i brings the key row r0 + RPI i of each lane.
  // Keys past the chunk read current-chunk row 0, finite data whose scores the causal mask
  // removes.  load_tile takes any tile; load_part is instruction i (K for i < NDMA, then
  // V) of a tile that lies within the history or within the chunk (a Tile).
  auto row0 = [&]() __attribute__((always_inline)) { return wave * (kKeys / kWaves) + fresh(ulane) / CPR; };
  const unsigned kcol = ((ulane % CPR) ^ (row0() & 15)) * 16, vcol = ((ulane % CPR) ^ (4 * (row0() % VSW))) * 16;
  auto load_tile = [&](int kt, unsigned kdst, unsigned vdst) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < NDMA; ++i) {
      const int p = kt * kKeys + (int)row0() + RPI * i;
      const bool in_hist = p < ihist;
      const int ci = p < ikeys ? p - ihist : 0;  // current-chunk index
      const uint64_t off = (uint64_t)(unsigned)(in_hist ? p : ci) * (unsigned)(in_hist ? hrow : crow);
      const unsigned lo = (wave * (kKeys / kWaves) + RPI * i) * ROWB;
      dma16(lds0 + kdst + lo, (const void*)((in_hist ? hist_k : cur_k) + off + (kcol ^ (unsigned)(RPI * i * 16))));
      dma16(lds0 + vdst + lo, (const void*)((in_hist ? hist_v : cur_v) + off + (vcol ^ (unsigned)(4 * (RPI * i % VSW) * 16))));
    }
  };
  struct Tile {
    uint64_t k, v;          // its first row
    unsigned pitch;         // bytes
    unsigned row;           // per lane: offset of row r0
    unsigned kdst, vdst;    // where it goes in LDS, this wave's part
  };
  auto whole = [&](int kt) __attribute__((always_inline)) {
    const int p0 = kt * kKeys;
    return p0 + kKeys <= ihist || (p0 >= ihist && p0 + kKeys <= ikeys);
  };
  auto tile_at = [&](int kt, unsigned kdst, unsigned vdst) __attribute__((always_inline)) {
    const int p0 = kt * kKeys;
    const bool in_hist = p0 < ihist;
    Tile t;
    t.pitch = (unsigned)(in_hist ? hrow : crow);
    const uint64_t off = (uint64_t)(unsigned)(in_hist ? p0 : p0 - ihist) * t.pitch;
    t.k = (in_hist ? hist_k : cur_k) + off;
    t.v = (in_hist ? hist_v : cur_v) + off;
    t.row = row0() * t.pitch;
    t.kdst = lds0 + kdst + wave * (kKeys / kWaves) * ROWB;
    t.vdst = lds0 + vdst + wave * (kKeys / kWaves) * ROWB;
    return t;
  };
  auto load_part = [&](const Tile& t, int i) __attribute__((always_inline)) {
    const bool v = i >= NDMA;
    i = v ? i - NDMA : i;
    const unsigned sw = (unsigned)((v ? 4 * (RPI * i % VSW) : RPI * i) * 16);
    dma16((v ? t.vdst : t.kdst) + RPI * i * ROWB, (v ? t.v : t.k) + (uint64_t)(RPI * i) * t.pitch,
          t.row + ((v ? vcol : kcol) ^ sw));
  };
  // bf16 current-chunk rows of a landed V tile to the PV format, in place (kVShift):
  // 16-byte part i of this thread's share
  constexpr int NCONV = TILEB / 16 / kThreads;
  constexpr int CONVROWS = kThreads * 16 / ROWB;  // key rows of one part, over the workgroup
  auto conv_at = [&](unsigned off, int i) __attribute__((always_inline)) {
    return (__attribute__((address_space(3))) u32x4*)(lds + off + (wave * 64 + fresh(ulane)) * 16 + i * kThreads * 16);
  };
  auto conv_keep = [&](int kt, int i) __attribute__((always_inline)) {
    // the history rows of a mixed tile are in the format
    return (int)((wave * 64 + fresh(ulane)) * 16 / ROWB) < ihist - kt * kKeys - CONVROWS * i;
  };
  auto converts = [&](int kt) __attribute__((always_inline)) { return QT == OSCAR_BF16 && kt * kKeys + kKeys > ihist; };
  auto k_tile = [&](int i) __attribute__((always_inline)) { return (unsigned)(i * TILEB); };
  auto v_tile = [&](int i) __attribute__((always_inline)) { return (unsigned)((NK + i) * TILEB); };
  auto next = [](int i, int ring) { return i + 1 == ring ? 0 : i + 1; };

  // in the order the loop waits for them
  load_tile(kb, k_tile(0), v_tile(0));
  load_tile(kb + 1, k_tile(1), v_tile(1));

  // this lane's row of a row block: row n of the query tile, query qi; computed again where
  // it is needed
  struct Row { int n, head; int64_t qi; bool ok; };
  auto row_of = [&](int nb) __attribute__((always_inline)) {
    const int rm = (int)(fresh(ulane) & 31);
    Row r;
    r.n = NB == 2 ? (wave & 1) * 64 + 32 * nb + rm : wave * 32 + rm;
    r.qi = q0 + r.n / G;
    r.head = kvh * G + r.n % G;
    r.ok = live && (r.n < P.qtok * G) && (r.qi < q1);
    return r;
  };
  // the wave's Q^T operands (K-step j) in registers for the whole key range: each
  // tile's QK then reads only K from LDS
  QV qreg[NB][D / 16];
#pragma unroll
  for (int nb = 0; nb < NB; ++nb) {
    const Row r = row_of(nb);
    const uint16_t* qrow = (const uint16_t*)A.q + (r.ok ? r.qi : 0) * A.q_stride_token + (int64_t)r.head * D;
#pragma unroll
    for (int j = 0; j < D / 16; ++j)
      qreg[nb][j] = __builtin_bit_cast(QV, r.ok ? *(const u32x4*)(qrow + 16 * j + 8 * g) : u32x4{0u, 0u, 0u, 0u});
  }
  const float c = A.scale * kLog2e;

  float m_run[NB], l_run[NB];
  f32x16 O[NB][D / 32];
#pragma unroll
  for (int nb = 0; nb < NB; ++nb) {
    m_run[nb] = -INFINITY;
    l_run[nb] = 0.f;
#pragma unroll
    for (int b = 0; b < D / 32; ++b)
#pragma unroll
      for (int r = 0; r < 16; ++r) O[nb][b][r] = 0.f;
    hold_acc(O[nb]);
  }

  f32x16 S[NB];
  u32x4 p_cur[NB][2], p_new[NB][2] = {};  // P^T of the tile before and of this one, fp16
  float lsum[NB];

  // ---- operands from a tile in LDS: K of K-step j; V of PV step i (output block i / 2, 16
  // keys i % 2).  KA / VA of them are read ahead of their MFMAs, the first ones before
  // the phase starts.
  constexpr int KA = NB == 2 ? 3 : 4, VA = 3;
  QV ka[KA];
  f16x8 va[VA];
  const unsigned krow = (ulane & 31) * ROWB, ksw = ((ulane >> 5) ^ (ulane & 15)) * 16;
  auto k_op = [&](unsigned off, int j) __attribute__((always_inline)) {
    return *(const __attribute__((address_space(3))) QV*)(lds + off + krow + (fresh(ksw) ^ (unsigned)(32 * j)));
  };
  const unsigned vkey = 4 * (ulane >> 5) + ((ulane & 15) >> 2);  // + 16 s + 8 h
  const unsigned vrow = vkey * ROWB + 32 * ((ulane >> 4) & 1) + 8 * (ulane & 3), vsw = 64 * (vkey % VSW);
  auto v_op = [&](unsigned off, int i) __attribute__((always_inline)) {
    const lds_u8* const at = lds + off + vrow + ((unsigned)(64 * (i >> 1)) ^ fresh(vsw)) + 16 * (i & 1) * ROWB;
    f16x8 v;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      auto t = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) i16x4*)(at + 8 * h * ROWB));
#pragma unroll
      for (int e = 0; e < 4; ++e) v[4 * h + e] = __builtin_bit_cast(_Float16, (unsigned short)t[e]);
    }
    return v;
  };
  auto k_ahead = [&](unsigned off) __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < KA - 1; ++j) ka[j] = k_op(off, j);
  };
  auto v_ahead = [&](unsigned off) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < VA - 1; ++i) va[i] = v_op(off, i);
  };
  // ---- S^T = K Q^T of the landed tile kt, whose first K operands are in ka; reads the
  // first V operands of the tile at `voff`, which PV takes next.
  // An MFMA takes 32 cycles of the wave's SIMD, in which the wave can issue about five
  // other instructions; more than that wait for nothing to overlap with.  The work that
  // is not PV's is therefore dealt out one piece per MFMA: the DMAs of tile `t` (LOAD),
  // the move of the last P to p_cur and the conversion of kt's V (CONV).
  auto qk = [&](int kt, unsigned off, unsigned voff, unsigned vconv, const Tile& t, auto conv, auto load) __attribute__((always_inline)) {
    constexpr bool CONV = decltype(conv)::value, LOAD = decltype(load)::value;
    constexpr int NS = D / 16;
    constexpr int MOVES = (8 * NB + NS - 1) / NS;  // per step, of the 8 NB registers of P
    u32x4 cx;
    bool keep = false;
    auto beside = [&](int j, int nb) __attribute__((always_inline)) {
      const int w = NB * j + nb;  // the MFMA of row block nb of K-step j
      if (nb == 0 && j + KA - 1 < NS) ka[(j + KA - 1) % KA] = k_op(off, j + KA - 1);
      if (nb == 0 && j == NS - 2) v_ahead(voff);
      if (LOAD && w % (NB * NS / (2 * NDMA)) == 0) load_part(t, w / (NB * NS / (2 * NDMA)));
      if constexpr (CONV) {
        constexpr int WPC = NB * NS / NCONV;  // MFMAs per 16-byte part
        const int i = w / WPC, q = w % WPC;
        if (q == 0) cx = *conv_at(vconv, i);
        if (q == WPC / 2) keep = conv_keep(kt, i);
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (q == WPC / 2 + e * (WPC / 2) / 4) {
            const unsigned w = pv_pair(cx[e]);
            cx[e] = keep ? cx[e] : w;
          }
        if (q == WPC - 1) *conv_at(vconv, i) = cx;
      }
      if (nb == NB - 1) {
#pragma unroll
        for (int e = MOVES * j; e < MOVES * (j + 1) && e < 8 * NB; ++e) {
          unsigned x;
          asm volatile("v_mov_b32 %0, %1" : "=v"(x) : "v"(p_new[e / 8][e / 4 % 2][e % 4]));
          p_cur[e / 8][e / 4 % 2][e % 4] = x;
        }
      }
    };
#pragma unroll
    for (int j = 0; j < NS; ++j) {
#pragma unroll
      for (int nb = 0; nb < NB; ++nb) {
        if (j == 0) mfma_qk<QT, true>(S[nb], ka[j % KA], qreg[nb][j]);
        else mfma_qk<QT, false>(S[nb], ka[j % KA], qreg[nb][j]);
        beside(j, nb);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    // the MFMAs' results are read by the VALU next
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) asm volatile("s_nop 15" : "+v"(S[nb]));
  };
  // masked keys get -inf scores (boundary tiles only).  Padding rows have zero queries
  // and are never written, so they need no mask.
  const int all_see = (int)(hist + q0 + 1);  // keys visible to every row of the wave's tile
  auto mask = [&](int kt) __attribute__((always_inline)) {
    const int k0 = kt * kKeys;
    if (__builtin_expect(k0 + kKeys <= all_see, 1)) return;
    const int ml = (int)(fresh(ulane) >> 5);
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) {
      const int lim = (int)(hist + row_of(nb).qi + 1) - k0 - 4 * ml;  // keys of the tile visible to this row
#pragma unroll
      for (int r = 0; r < 16; ++r) S[nb][r] = 8 * (r >> 2) + (r & 3) >= lim ? -INFINITY : S[nb][r];
    }
  };
  // p = 2^(S c - m) of element r (exp2 of -inf is 0; rows with no key yet have m = -inf and p = 0)
  auto prob = [&](int nb, int r, float nm) __attribute__((always_inline)) { return __builtin_amdgcn_exp2f(fmaf(S[nb][r], c, nm)); };
  auto neg_m = [&](int nb) __attribute__((always_inline)) { return m_run[nb] == -INFINITY ? 0.f : -m_run[nb]; };
  auto row_max = [&](int nb) __attribute__((always_inline)) {  // of the scores, over both halves of the row
    float mx = -INFINITY;
#pragma unroll
    for (int r = 0; r < 16; ++r) mx = fmaxf(mx, S[nb][r]);
    auto sw = __builtin_amdgcn_permlane32_swap(__float_as_uint(mx), __float_as_uint(mx), false, false);
    return fmaxf(__uint_as_float(sw[0]), __uint_as_float(sw[1])) * c;  // c > 0
  };
  auto put_p = [&](int nb, int r, float p0, float p1) __attribute__((always_inline)) {
    unsigned w = __builtin_bit_cast(unsigned, __builtin_convertvector(f32x2{p0, p1}, f16x2));
    asm volatile("" : "+v"(w));  // stays where it stands (else it sinks past the test for a moved reference)
    p_new[nb][r >> 3][(r & 7) >> 1] = w;
  };
  // the probabilities of S against the reference m_run, not beside anything (first tile,
  // moved reference)
  auto softmax = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) {
      const float nm = neg_m(nb);
      lsum[nb] = 0.f;
#pragma unroll
      for (int r = 0; r < 16; r += 2) {
        const float p0 = prob(nb, r, nm), p1 = prob(nb, r + 1, nm);
        lsum[nb] += p0 + p1;
        put_p(nb, r, p0, p1);
      }
    }
  };
  // ---- O^T += V^T P^T of the tile before, whose first V operands are in va, beside the
  // probabilities and row sums of this tile (SM); reads the first K operands of the tile
  // at `koff`.  Without SM: the wave's last tile, in which values of keys past its query
  // tile (a later tile's, and the pair's other tile reads them) are taken as zero: their
  // probabilities are, but an infinite value's product would be NaN.
  auto pv = [&](unsigned off, unsigned koff, auto sm) __attribute__((always_inline)) {
    constexpr bool SM = decltype(sm)::value;
    constexpr int NPV = D / 16;   // steps
    constexpr int EPS = 16 / NPV; // elements of S per row block and step
    float nm[NB], pe[NB][2];
    u32x4 seen[2] = {};  // all ones where the step's V operand is of a key of this wave's tile
    if constexpr (SM) {
#pragma unroll
      for (int nb = 0; nb < NB; ++nb) { nm[nb] = neg_m(nb); lsum[nb] = 0.f; }
    } else {
      const int lim = (int)(hist + q1) - (ke_own - 1) * kKeys - 4 * (int)(fresh(ulane) >> 5);
#pragma unroll
      for (int e = 0; e < 16; ++e) {  // keys 16 s + 8 h + 4 g + (e & 3)
        const int key = 16 * (e >> 3) + 8 * (e >> 2 & 1) + (e & 3);
        seen[e >> 3][e / 2 % 4] |= key < lim ? 0xffffu << 16 * (e & 1) : 0u;
      }
    }
    auto pair_done = [&](int nb, int r) __attribute__((always_inline)) {  // elements r - 1, r
      lsum[nb] += pe[nb][0] + pe[nb][1];
      put_p(nb, r - 1, pe[nb][0], pe[nb][1]);
    };
#pragma unroll
    for (int i = 0; i < NPV; ++i) {
#pragma unroll
      for (int nb = 0; nb < NB; ++nb) {
        f16x8 v = va[i % VA];
        if constexpr (!SM) v = __builtin_bit_cast(f16x8, __builtin_bit_cast(u32x4, v) & seen[i & 1]);
        O[nb][i >> 1] = __builtin_amdgcn_mfma_f32_32x32x16_f16(v, __builtin_bit_cast(f16x8, p_cur[nb][i & 1]), O[nb][i >> 1], 0, 0, 0);
        if (nb == 0 && i + VA - 1 < NPV) va[(i + VA - 1) % VA] = v_op(off, i + VA - 1);
        if (SM && nb == NB - 1 && i == NPV - 1) k_ahead(koff);
        if constexpr (SM) {
          // a pair's sum and packing beside the next step's element
#pragma unroll
          for (int e = 0; e < EPS; ++e) {
            const int r = EPS * i + e;
            if (r % 2 == 0 && r > 0) pair_done(nb, r - 1);
            pe[nb][r & 1] = prob(nb, r, nm[nb]);
            if (r == 15) pair_done(nb, r);
          }
        }
        __builtin_amdgcn_sched_barrier(0);
      }
    }
  };
  // ---- the first tile: its row maxima are the first references
  tile_barrier<2 * NDMA>();
  load_tile(kb + 2, k_tile(2), v_tile(2));
  k_ahead(k_tile(0));
  qk(kb, k_tile(0), v_tile(0), v_tile(0), Tile{}, std::integral_constant<bool, QT == OSCAR_BF16>{}, std::false_type{});
  mask(kb);
#pragma unroll
  for (int nb = 0; nb < NB; ++nb) m_run[nb] = row_max(nb);
  softmax();
#pragma unroll
  for (int nb = 0; nb < NB; ++nb) l_run[nb] = lsum[nb];
  tile_barrier<2 * NDMA>();  // as in the loop
  k_ahead(k_tile(1));
  // Iteration kt: QK of kt, then PV of kt - 1 beside the softmax of kt against the
  // reference as it stands.  A row whose probabilities turn out large (one above 2^kLazy
  // shows in their sum) or that had no visible key before moves its reference to its
  // maximum: O and l are rescaled and P is formed again (rare).
  int kr = 0, vr = 0;  // ring places of K(kt - 1) and V(kt - 1)
#pragma clang loop unroll(disable)
  for (int kt = kb + 1; kt < ke_own; ++kt) {
    const int k1 = next(kr, NK), v1 = next(vr, NV);
    // kt + 2 (past the last tile: that one again, never read) goes over K(kt - 1) and
    // V(kt - 3), read before the last barrier
    const int kn = kt + 2 < ke ? kt + 2 : ke - 1;
    const unsigned kdst = k_tile(kr), vdst = v_tile(vr < 2 ? vr + NV - 2 : vr - 2);
    if (__builtin_expect(!whole(kn), 0)) {
      load_tile(kn, kdst, vdst);
      qk(kt, k_tile(k1), v_tile(vr), v_tile(v1), Tile{}, std::integral_constant<bool, QT == OSCAR_BF16>{}, std::false_type{});
    } else if (converts(kt)) {
      qk(kt, k_tile(k1), v_tile(vr), v_tile(v1), tile_at(kn, kdst, vdst), std::true_type{}, std::true_type{});
    } else {
      qk(kt, k_tile(k1), v_tile(vr), v_tile(v1), tile_at(kn, kdst, vdst), std::false_type{}, std::true_type{});
    }
    // every wave is past QK of kt and PV of kt - 2; kt's V is in its format; kt + 1 has
    // landed (kt + 2's DMAs are outstanding)
    tile_barrier<2 * NDMA>();
    mask(kt);
    pv(v_tile(vr), k_tile(next(k1, NK)), std::true_type{});
    kr = k1;
    vr = v1;
    bool moved = false;
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) moved = moved || lsum[nb] > (float)(1 << kLazy) || m_run[nb] == -INFINITY;
    if (__builtin_expect(__any(moved), 0)) {
      asm volatile("s_nop 15\n\ts_nop 15");  // the PV MFMAs' results
#pragma unroll
      for (int nb = 0; nb < NB; ++nb) {
        const float mx = row_max(nb);
        const bool move = mx > m_run[nb];
        const float f = move ? exp2f(m_run[nb] - mx) : 1.f;
#pragma unroll
        for (int b = 0; b < D / 32; ++b)
#pragma unroll
          for (int r = 0; r < 16; ++r) {
            float o = O[nb][b][r];
            scale_acc(o, f);
            O[nb][b][r] = o;
          }
        hold_acc(O[nb]);
        l_run[nb] *= f;
        if (move) m_run[nb] = mx;
      }
      softmax();
    }
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) l_run[nb] += lsum[nb];
  }
  // the last tile (its V was converted before the last barrier)
#pragma unroll
  for (int nb = 0; nb < NB; ++nb) { p_cur[nb][0] = p_new[nb][0]; p_cur[nb][1] = p_new[nb][1]; }
  v_ahead(v_tile(vr));
  pv(v_tile(vr), 0, std::false_type{});
  // the other waves' tiles past this wave's own: its share of the moves and conversions
#pragma clang loop unroll(disable)
  for (int kt = ke_own; kt < ke; ++kt) {
    const int v1 = next(vr, NV), kn = kt + 2 < ke ? kt + 2 : ke - 1;
    load_tile(kn, k_tile(kr), v_tile(vr < 2 ? vr + NV - 2 : vr - 2));
    if (converts(kt)) {
      for (int i = 0; i < NCONV; ++i) {
        u32x4 x = *conv_at(v_tile(v1), i);
        const bool keep = conv_keep(kt, i);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const unsigned w = pv_pair(x[e]);
          x[e] = keep ? x[e] : w;
        }
        *conv_at(v_tile(v1), i) = x;
      }
    }
    tile_barrier<2 * NDMA>();
    kr = next(kr, NK);
    vr = v1;
  }
  tile_barrier<0>();  // no DMA may be in flight when the workgroup ends

  // ---- finalize: row n = lane's row; O^T block b register r holds d = 32b + out_row(r, g)
#pragma unroll
  for (int nb = 0; nb < NB; ++nb) {
    float l_tot;
    {
      auto sw = __builtin_amdgcn_permlane32_swap(__float_as_uint(l_run[nb]), __float_as_uint(l_run[nb]), false, false);
      l_tot = __uint_as_float(sw[0]) + __uint_as_float(sw[1]);
    }
    const Row row = row_of(nb);
    const int rg = (int)(fresh(ulane) >> 5);
    if (!row.ok) continue;
    // O back from the PV scale of bf16 V values (a power of two: exact)
    const float inv = (l_tot > 0.f) ? (QT == OSCAR_F16 ? 1.f : (float)(1 << kVShift)) / l_tot : 0.f;
    const float lse2 = (l_tot > 0.f) ? m_run[nb] + log2f(l_tot) : -INFINITY;
    if (slot >= 0) {
      // a chunk of a split tile: normalised O and its log2-domain LSE (-inf: no key of
      // the chunk visible to the row) for prefill_merge_kernel
      const int64_t block = ((int64_t)slot * hk + kvh) * (kRows / 32) + row.n / 32;
      float* po = P.part_o + block * 32 * D + 4 * fresh(ulane);
#pragma unroll
      for (int b = 0; b < D / 32; ++b)
#pragma unroll
        for (int r = 0; r < 16; r += 4)
          *(f32x4*)(po + (4 * b + (r >> 2)) * 256) = f32x4{O[nb][b][r] * inv, O[nb][b][r + 1] * inv,
                                                           O[nb][b][r + 2] * inv, O[nb][b][r + 3] * inv};
      if (rg == 0) P.part_lse[((int64_t)slot * hk + kvh) * kRows + row.n] = lse2;
      continue;
    }
    const int64_t obase = row.qi * A.out_stride_token + (int64_t)row.head * D;
#pragma unroll
    for (int b = 0; b < D / 32; ++b)
#pragma unroll
      for (int r = 0; r < 16; r += 4)
        store_out<QT>(A, obase + 32 * b + 8 * (r >> 2) + 4 * rg,
                      f32x4{O[nb][b][r] * inv, O[nb][b][r + 1] * inv, O[nb][b][r + 2] * inv, O[nb][b][r + 3] * inv});
    if (A.lse != nullptr && rg == 0) A.lse[row.qi * A.num_q_heads + row.head] = l_tot > 0.f ? lse2 * kLn2 : -INFINITY;
  }
}

// FP32 LSE merge of a split tile's chunk partials (slab_attention.py:341-356 applied
// over the chunks): wave (32 rows, 32 output columns), lane as in the MFMA result that the
// partials keep (row lane % 32, four times four columns).  Writes what the unsplit kernel
// writes for the row: the output (query dtype when there is no history, else fp32 rotated)
// and the LSE.  Bound by the partials' bytes: a chunk's 1 KB per lane group comes in one
// load (row by row, 16 bytes a lane 1 KB apart, 2048 fresh
// tokens 10.8 us, 8.6 us this way, their prefill kernel 39.1 and 37.5 us).
template <int D, int QT>
__global__ __launch_bounds__(256) void prefill_merge_kernel(PrefillParams P) {
  constexpr int NBK = D / 32, PER = NBK / 4;  // 32-column blocks; workgroups per 32 rows
  const oscar_prefill_args_v1& A = P.a;
  const int lane = threadIdx.x & 63, m = lane & 31, g = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int unit = blockIdx.x / PER, b = (blockIdx.x % PER) * 4 + wave;
  const int s = unit / (kRows / 32);  // split tile, heaviest first (its class-0 slot)
  const int rb = unit % (kRows / 32), n = 32 * rb + m;
  const int kvh = blockIdx.y;
  const int64_t hk = A.num_kv_heads;
  const int G = P.group;
  const int qt = P.ntq - 1 - s;
  const int64_t q0 = (int64_t)qt * P.qtok;
  const int64_t q1 = (q0 + P.qtok < A.num_tokens) ? q0 + P.qtok : A.num_tokens;
  const int64_t qi = q0 + n / G;
  if (n >= P.qtok * G || qi >= q1) return;
  const int nch = (int)((tile_keys(A.history, q1) + P.U - 1) / P.U);
  auto slot = [&](int c) { return (int64_t)(c == 0 ? s : P.base[c] + s - P.qmin1) * hk + kvh; };
  float M = -INFINITY;
  for (int c = 0; c < nch; ++c) M = fmaxf(M, P.part_lse[slot(c) * kRows + n]);
  f32x4 acc[4] = {};
  float L = 0.f;
  if (M != -INFINITY) {
    for (int c = 0; c < nch; ++c) {
      const float lc = P.part_lse[slot(c) * kRows + n];
      if (lc != -INFINITY) {
        const f32x4* po = (const f32x4*)(P.part_o + (slot(c) * (kRows / 32) + rb) * 32 * D) + 4 * b * 64 + lane;
        const float w = exp2f(lc - M);
        L += w;
#pragma unroll
        for (int q = 0; q < 4; ++q) acc[q] += po[64 * q] * w;
      }
    }
  }
  const float inv = L > 0.f ? 1.f / L : 0.f;
  const int head = kvh * G + n % G;
  const int64_t obase = qi * A.out_stride_token + (int64_t)head * D + 32 * b + 4 * g;
#pragma unroll
  for (int q = 0; q < 4; ++q) store_out<QT>(A, obase + 8 * q, acc[q] * inv);
  if (A.lse != nullptr && b == 0 && g == 0)
    A.lse[qi * A.num_q_heads + head] = L > 0.f ? (M + log2f(L)) * kLn2 : -INFINITY;
}

// Two query tiles per workgroup from this many units on (head dim 256, where a CU holds one
// workgroup).  One tile takes about two thirds of a pair's time per key tile, so up to one
// unit per CU a unit's latency counts; beyond it the unpaired units need a second round of
// the chip, which pairs do without up to 512 and halve the operand reads per MFMA after.
// The line lies an eighth above a round, since the last units in launch order are the short
// ones.  Unpaired / paired in us: fresh tokens of 6 heads on 1, 2048 (247 units) 44 / 53,
// 2200 (283) 53 / 55, 2400 (333) 67 / 55, 3000 (473) 76 / 63, 6000 (625) 196 / 178; 12 heads
// on 2, 1500 (288) 53 / 53, 1800 (398) 68 / 57; 8000 + 1600 (500) 144 / 121; 15360 + 9256
// 1.60 / 1.23 ms.  At head dim 128 two unpaired workgroups fit a CU and overlap each other
// (8000 + 4000 tokens, 16 heads on 2: 374 us against 380 us paired), so there are no pairs
// there.
constexpr int64_t kPairUnits = kSplitCUs + kSplitCUs / 8;
template <int D, int QT>
void launch_prefill(const PrefillParams& p, dim3 grid, bool pairs, hipStream_t s) {
  if constexpr (D == 256) {
    if (pairs) {
      hipLaunchKernelGGL((prefill_kernel<D, QT, 2>), grid, dim3(kThreads), 0, s, p);
      return;
    }
  }
  hipLaunchKernelGGL((prefill_kernel<D, QT, 1>), grid, dim3(kThreads), 0, s, p);
}

}  // namespace

}  // namespace oscar

using namespace oscar;

extern "C" int64_t oscar_prefill_workspace_bytes_v1(int64_t history, int64_t num_kv_heads, int64_t head_dim) {
  if (history <= 0) return 0;
  return 2 * history * num_kv_heads * head_dim * (int64_t)sizeof(uint16_t);
}

extern "C" int64_t oscar_prefill_workspace_bytes_v2(int64_t history, int64_t num_tokens, int64_t num_q_heads,
                                                     int64_t num_kv_heads, int64_t head_dim) {
  if (history < 0 || num_tokens < 0 || num_kv_heads < 1 || num_q_heads < num_kv_heads ||
      num_q_heads % num_kv_heads || (head_dim != 128 && head_dim != 256) || num_q_heads / num_kv_heads > kRows)
    return -22;
  const SplitPlan sp = plan_split(history, num_tokens, kRows / (num_q_heads / num_kv_heads), num_kv_heads);
  return hist_bytes(history, num_kv_heads, head_dim) + split_bytes(sp, num_kv_heads, head_dim);
}

extern "C" int oscar_prefill_plan_v1(int64_t history, int64_t num_tokens, int64_t num_q_heads, int64_t num_kv_heads,
                                     int32_t* out, int32_t cap) {
  if (!out || cap < 6 + kMaxChunks + 1 || history < 0 || num_tokens < 0 || num_kv_heads < 1 ||
      num_q_heads < num_kv_heads || num_q_heads % num_kv_heads || num_q_heads / num_kv_heads > kRows)
    return -22;
  const SplitPlan sp = plan_split(history, num_tokens, kRows / (num_q_heads / num_kv_heads), num_kv_heads);
  const int64_t head[6] = {sp.chunks, sp.U, sp.ntq, sp.qmin1, sp.units, sp.slots};
  for (int i = 0; i < 6; ++i) out[i] = (int32_t)head[i];
  for (int c = 0; c <= kMaxChunks; ++c) out[6 + c] = sp.base[c];
  return 0;
}

extern "C" int oscar_attn_prefill_v1(const oscar_prefill_args_v1* args, void* stream) {
  if (!args) return fail(-22, "oscar_attn_prefill_v1: null args");
  const oscar_prefill_args_v1& a = *args;
  if (a.num_tokens == 0) return 0;
  const int64_t D = a.head_dim;
  if (D != 128 && D != 256) return fail(-22, "oscar_attn_prefill_v1: head_dim %lld unsupported", (long long)D);
  if (!a.q || !a.k || !a.v || !a.out || a.num_tokens < 0 || a.num_kv_heads < 1 ||
      a.num_q_heads % a.num_kv_heads)
    return fail(-22, "oscar_attn_prefill_v1: invalid arguments");
  if (a.q_dtype != OSCAR_BF16 && a.q_dtype != OSCAR_F16)
    return fail(-22, "oscar_attn_prefill_v1: q_dtype must be OSCAR_BF16 or OSCAR_F16");
  const int G = (int)(a.num_q_heads / a.num_kv_heads);
  if (G > kRows) return fail(-22, "oscar_attn_prefill_v1: more than %d query heads per KV head", kRows);
  if (a.history < 0) return fail(-22, "oscar_attn_prefill_v1: negative history");
  if (a.history > 0 && (!a.cache.k || !a.cache.v || !a.block_table_row || a.cache.head_dim != D ||
                        a.cache.block_size < 1))
    return fail(-22, "oscar_attn_prefill_v1: history needs the cache and the block-table row");
  // streaming_attention.py:51-53
  if (a.history > 0 && (a.history + a.cache.block_size - 1) / a.cache.block_size > a.block_table_cols)
    return fail(-22, "oscar_attn_prefill_v1: Block table cannot cover the history");
  // q/k/v rows and the history workspace are read as 16-byte vectors
  if ((((uintptr_t)a.q) & 15) || (((uintptr_t)a.k) & 15) || (((uintptr_t)a.v) & 15) ||
      ((a.q_stride_token * 2) & 15) || ((a.kv_stride_token * 2) & 15))
    return fail(-22, "oscar_attn_prefill_v1: q/k/v rows must be 16-byte aligned");
  // the prefill kernel addresses history and chunk rows with 32-bit element offsets
  if ((a.history + 64) * a.num_kv_heads * D >= (1ll << 31) ||
      (a.num_tokens + 64) * a.kv_stride_token >= (1ll << 31))
    return fail(-22, "oscar_attn_prefill_v1: history or chunk too large for one call");
  const int64_t need = oscar_prefill_workspace_bytes_v1(a.history, a.num_kv_heads, D);
  if (a.history > 0 &&
      (a.workspace == nullptr || a.workspace_bytes < need || (((uintptr_t)a.workspace) & 15)))
    return fail(-22, "oscar_attn_prefill_v1: 16-byte aligned workspace of %lld bytes required", (long long)need);
  PrefillParams p{};
  p.a = a;
  p.has_stage = a.staging != nullptr;
  if (a.staging) p.st = *a.staging;
  p.group = G;
  p.qtok = kRows / G;
  if (a.history > 0) {
    p.hist_k = (uint16_t*)a.workspace;
    p.hist_v = p.hist_k + a.history * a.num_kv_heads * D;
  }
  // the balanced split when the workspace holds its partials (after the history values)
  const SplitPlan sp = plan_split(a.history, a.num_tokens, p.qtok, a.num_kv_heads);
  const int64_t hbytes = hist_bytes(a.history, a.num_kv_heads, D), sbytes = split_bytes(sp, a.num_kv_heads, D);
  p.ntq = (int)((a.num_tokens + p.qtok - 1) / p.qtok);
  if (sbytes > 0 && a.workspace != nullptr && (((uintptr_t)a.workspace) & 15) == 0 &&
      a.workspace_bytes >= hbytes + sbytes) {
    p.split = 1;
    p.chunks = sp.chunks;
    p.U = sp.U;
    p.qmin1 = sp.qmin1;
    for (int c = 0; c <= kMaxChunks; ++c) p.base[c] = sp.base[c];
    p.part_o = (float*)((char*)a.workspace + hbytes);
    p.part_lse = p.part_o + sp.slots * a.num_kv_heads * kRows * D;
  }
  hipStream_t s = (hipStream_t)stream;
  if (a.history > 0) {
    const unsigned hb = (unsigned)((a.history * a.num_kv_heads + 3) / 4);
    if (a.q_dtype == OSCAR_F16) {
      if (D == 256) hipLaunchKernelGGL((history_bf16_kernel<256, OSCAR_F16>), dim3(hb), dim3(256), 0, s, p);
      else hipLaunchKernelGGL((history_bf16_kernel<128, OSCAR_F16>), dim3(hb), dim3(256), 0, s, p);
    } else {
      if (D == 256) hipLaunchKernelGGL((history_bf16_kernel<256, OSCAR_BF16>), dim3(hb), dim3(256), 0, s, p);
      else hipLaunchKernelGGL((history_bf16_kernel<128, OSCAR_BF16>), dim3(hb), dim3(256), 0, s, p);
    }
    OSCAR_CHECK_LAUNCH("history_bf16_kernel");
  }
  const int units = p.split ? sp.units : p.ntq;
  const bool pairs = D == 256 && units * a.num_kv_heads > kPairUnits;
  for (int c = 0; c < p.chunks; ++c) p.pbase[c + 1] = p.pbase[c] + (sp.base[c + 1] - sp.base[c] + 1) / 2;
  const int wgs = !pairs ? units : p.split ? p.pbase[p.chunks] : (p.ntq + 1) / 2;
  const dim3 grid((unsigned)wgs, (unsigned)a.num_kv_heads);
  if (a.q_dtype == OSCAR_F16) {
    if (D == 256) launch_prefill<256, OSCAR_F16>(p, grid, pairs, s);
    else launch_prefill<128, OSCAR_F16>(p, grid, pairs, s);
  } else {
    if (D == 256) launch_prefill<256, OSCAR_BF16>(p, grid, pairs, s);
    else launch_prefill<128, OSCAR_BF16>(p, grid, pairs, s);
  }
  OSCAR_CHECK_LAUNCH("prefill_kernel");
  if (p.split) {
    const dim3 mgrid((unsigned)((p.ntq - p.qmin1) * (kRows / 32) * (D / 128)), (unsigned)a.num_kv_heads);
    if (a.q_dtype == OSCAR_F16) {
      if (D == 256) hipLaunchKernelGGL((prefill_merge_kernel<256, OSCAR_F16>), mgrid, dim3(256), 0, s, p);
      else hipLaunchKernelGGL((prefill_merge_kernel<128, OSCAR_F16>), mgrid, dim3(256), 0, s, p);
    } else {
      if (D == 256) hipLaunchKernelGGL((prefill_merge_kernel<256, OSCAR_BF16>), mgrid, dim3(256), 0, s, p);
      else hipLaunchKernelGGL((prefill_merge_kernel<128, OSCAR_BF16>), mgrid, dim3(256), 0, s, p);
    }
    OSCAR_CHECK_LAUNCH("prefill_merge_kernel");
  }
  return 0;
}
