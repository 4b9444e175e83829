// Paged prefill attention over scaled-FP8 pages (chunked / prefix-hit
// prefill): for every sequence i, query token j of its chunk sits at
// position prefix_i + j (prefix_i = context_len_i - query_len_i) and attends
// to keys 0..prefix_i + j of its paged history, which already holds the
// chunk's own K/V.  Restates prism_infer/ops/paged_attention_reference.py:
// 185-246 (gather :22-63, dequantisation :102-122, GQA :125-145): causal
// SDPA over the dequantised pages, output in q's dtype.  Dequantisation here
// is fp32 (payload * scale applied to the fp32 scores and to P), as the
// decode kernels do; the reference multiplies in q's dtype.
//
// Work layout.  A workgroup owns one kv head and one block of query tokens of
// one sequence; a wave owns 32 of the tokens and one of the G query heads of
// the kv head, so each K/V tile is read once into LDS for all of them (4 waves:
// 32 tokens for G = 4, 64 and 128 for G = 2 and 1; 8 waves for G = 8, or two
// workgroups of four, by the length of the tables).  Tiles of 64 keys
// go through four LDS stages: two tiles' loads are in flight beside the tile
// whose scores and the one whose softmax are computed.  Per tile a wave computes S^T = K Q^T with
// 32x32 MFMAs (bf16 queries: the fp8 MFMA 32x32x64 on the K bytes as they
// are, the query split into two fp8 terms that hold it exactly, products
// exact in fp32; f16 queries: v_mfma_f32_32x32x16_f16 on K converted to f16,
// exact; the key scale multiplies the rows of S^T), runs the online softmax
// per query column (log2 domain, lazy rescaling), and accumulates O^T += V^T
// P^T with v_mfma_f32_32x32x16_bf16, V^T coming from ds_read_b64_tr_b8 (fp8
// -> bf16 is exact) and P * v_scale entering as bf16, whose fp32 exponent
// range holds every v scale from the 1e-6 floor up.  Only tiles on the
// diagonal apply the causal mask.
//
// A query is one lane column from the scores to the output (S^T and O^T
// share it), so the running max, the sum and the rescaling of the
// accumulators are lane-local, and a column's max needs one lane swap.
//
// Few, long blocks (a short chunk behind a long prefix) leave most CUs idle:
// the keys of a block are then split over several workgroups, which write
// fp32 partials (max, sum, unnormalised output), merged by a second kernel
// (267 tokens behind 12000-token prefixes, 32 / 8 heads: 371 us on 88
// workgroups, 79 + 9.7 us split).
//
// Bound by VALU issue and dependency beside the MFMAs (busy 61% and 52% of the
// cycles): per 32 x 32 scores of a wave the MFMAs take 512 cycles (4 fp8 and 8
// bf16) and the softmax, the scales and the V conversion about 120
// instructions.  With 16x16 MFMAs (four lane groups per score column, outputs
// as query rows) the same work took 193: 4 x 2048 tokens behind 8192, 32 / 8
// heads, 1585 us; 1390 with this layout, and 1120 to 1190 (1040 to 1100
// TFLOP/s) with the next tile's scores spread over the softmax; 6 prompts of
// 61 to 1900 tokens 219 and 166 us.  Workgroups of one or two tiles spend most
// of their time on the lookup, the first loads and the masked tile, which costs
// 2.2 settled ones: 80 prompts of 100 tokens take 81 us, 68 with 16x16 MFMAs.
//
// Metadata stays on the device: each workgroup finds its sequence and query
// block from cu_seqlens_q with wave reductions, longest blocks first.
// Invalid lengths or block ids record the lowest offending sequence in
// status[0] (atomicMin); the host raises the reference's error for it.
#include "common.h"
#include "fp8_mfma.h"

#include <algorithm>

namespace prism {
namespace {

constexpr int kPfD = 128;                    // head dim
constexpr int kPfCols = 32;                  // query tokens per wave: the columns of a 32x32 MFMA
constexpr int kPfKT = 64;                    // keys per tile
constexpr int kPfMaxWaves = 8;               // GQA group size limit
constexpr float kPfSumLimit = 256.0f;        // largest sum of a lane's 32 weights that keeps the running max

typedef float floatx16 __attribute__((ext_vector_type(16)));
typedef int i32x2 __attribute__((ext_vector_type(2)));
typedef __attribute__((address_space(3))) i32x2 lds_i32x2;

struct PrefillArgs {
  const void* q;
  int64_t q_st, q_sh;  // elements (dim stride 1)
  const uint8_t* k;
  const uint8_t* v;
  int64_t k_sn, k_sp, k_sh, v_sn, v_sp, v_sh;  // bytes (dim stride 1)
  const float* ks;
  const float* vs;
  int64_t ks_sn, ks_sp, ks_sh, vs_sn, vs_sp, vs_sh;  // elements
  const int32_t* bt;
  int64_t bt_sb, bt_sn;
  const int32_t* ctx;
  const int32_t* cu_q;
  void* out;
  int64_t o_st, o_sh;
  int batch, num_heads, groups, page, num_blocks, width;
  float scale_log2;
  int* status;
  int* report;    // pinned: [0] set to 1 where a sequence is flagged, [1] and [2] the packed rows' extent; or null
  int out_vec;    // output rows can be stored 8 bytes at a time
  int splits;     // most workgroups per (block, kv head); the kernel takes as many of them as fill the chip
  int slots;      // workgroups that the chip holds at once
  int total_q;
  int* used;      // splits that the kernel took (written for the merge)
  float* part;    // [splits][total_q][num_heads][kPfD] unnormalised outputs, then [..][2] (max, sum)
};

// 16-byte chunk swizzle of a key row in LDS, by the key's index t.  gfx950
// LDS (measured with SQ_LDS_BANK_CONFLICT): 64 banks of 4 bytes (address bits
// 2..7); ds_read_b64 (and _tr_b8) serves lanes 0-31 and 32-63 in separate
// passes; ds_read_b128 serves 16 lanes per pass, the lanes whose bit 5 and
// parity of bits 2..4 agree.  A 128-byte key row puts bit 7 of the address
// at t & 1, so a row's 8 chunks cover one half of the banks and rows of
// opposite parity the other half.  With chunk ^= 4 t1 ^ t2 ^ 2 t3 both reads
// below are conflict-free under that model.  K rows (b128, lane (g, r): row
// r, chunk 2g + const): a pass holds every t1, t2, t3 once per row parity,
// eight distinct chunks.  V (transposed b64, a half wave: rows 4g + 0..3 and
// 8 more, chunks 2n and 2n + 1): t1, t3 and the chunk's own bit 0 vary.
__device__ __forceinline__ int pf_swz(int t) { return (((t >> 1) & 1) * 4) | ((t >> 2) & 1) | (((t >> 3) & 1) * 2); }

// A wave-uniform pointer, moved to SGPRs.
__device__ __forceinline__ const uint8_t* uniform_ptr(const uint8_t* p) {
  const uint64_t v = reinterpret_cast<uint64_t>(p);
  const uint32_t lo = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(v));
  const uint32_t hi = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(v >> 32));
  return reinterpret_cast<const uint8_t*>((static_cast<uint64_t>(hi) << 32) | lo);
}

// A uniform value in an SGPR.  Integer divisions come out of the VALU, and what
// depends on them (the tile loop's counters, addresses and branches) would
// stay there.
__device__ __forceinline__ int uniform_int(int v) { return __builtin_amdgcn_readfirstlane(v); }

__device__ __forceinline__ void flag_sequence(const PrefillArgs& a, int seq) {
  atomicMin(a.status, seq);
  if (a.report != nullptr) a.report[0] = 1;  // (every writer stores the same)
}

// Inclusive wave scan with f over lanes of non-negative values (0 is f's
// neutral element): row shifts, then the row ends broadcast onwards.
template <typename F>
__device__ __forceinline__ int wave_scan(int v, F f) {
  v = f(v, __builtin_amdgcn_update_dpp(0, v, 0x111, 0xF, 0xF, false));  // row_shr:1
  v = f(v, __builtin_amdgcn_update_dpp(0, v, 0x112, 0xF, 0xF, false));  // row_shr:2
  v = f(v, __builtin_amdgcn_update_dpp(0, v, 0x114, 0xF, 0xF, false));  // row_shr:4
  v = f(v, __builtin_amdgcn_update_dpp(0, v, 0x118, 0xF, 0xF, false));  // row_shr:8
  v = f(v, __builtin_amdgcn_update_dpp(0, v, 0x142, 0xA, 0xF, false));  // row_bcast:15 into rows 1 and 3
  return f(v, __builtin_amdgcn_update_dpp(0, v, 0x143, 0xC, 0xF, false));  // row_bcast:31 into rows 2 and 3
}

struct AddInt {
  __device__ int operator()(int x, int y) const { return x + y; }
};
struct MaxInt {
  __device__ int operator()(int x, int y) const { return max(x, y); }
};

template <typename F>
__device__ __forceinline__ int wave_reduce(int v, F f) {
  return __builtin_amdgcn_readlane(wave_scan(v, f), 63);
}

// Query blocks of sequence i (0 for a sequence with invalid lengths, which
// is flagged) and the level of its block 0: block j ends after about
// QT (level + j) keys.
template <int QT>
__device__ __forceinline__ int seq_blocks(const PrefillArgs& a, int i, bool flag, int& level0) {
  const int q0 = a.cu_q[i];
  const int qlen = a.cu_q[i + 1] - q0;
  const int ctx = a.ctx[i];
  if (qlen <= 0 || ctx < qlen || ctx > a.width * a.page) {
    if (flag) flag_sequence(a, i);
    level0 = 0;
    return 0;
  }
  level0 = (ctx - qlen) / QT + 1;
  return (qlen + QT - 1) / QT;
}

// A workgroup's work: query block, part of its keys, kv head.
struct PfWork {
  int seq, qblock, split, splits, head;
};

// Time of a launch, in units of 64 ns, whose longest block walks `tiles` tiles
// in s parts.  A tile takes a workgroup 1.2 us, 1.7 where a CU holds eight
// waves; parts cost a second launch and, for each of them, an fp32 row per
// (token, query head) written and read again (0.34 ns a row).  Measured split
// and not split, 1 to 8 query heads per kv head, 33 to 800 tokens behind 0 to
// 4096: parts for every free slot took 1.5 times as long where rows are many
// and tiles few (64 heads, 400 tokens: 41.7 against 27.8 us; 32 heads, 800
// tokens: 38.2 and 29.7), 0.3 of the time where it is the other way round (32
// heads, 33 tokens behind 4096: 27.6 and 91.9).
__host__ __device__ inline int split_cost(int s, int tiles, int wgs, int waves, int slots, int rows) {
  const int tile = waves == 8 || 2 * wgs * s > slots ? 27 : 19;
  return tiles * tile / s + (s > 1 ? 47 + s * (rows / 190) : 0);
}

// Workgroup id -> work, from the number of real blocks: heads fastest (so that
// the long blocks of all heads start first and, with 8 kv heads, each XCD
// reads one head's K/V), then the parts of the keys, then the block's rank.
// Returns the rank.  The keys are split, if that pays, into the cheapest number
// of parts that the chip has room for (lane s - 1 weighs s parts).
template <int NW>
__device__ __forceinline__ int pf_parts(const PrefillArgs& a, int kv_heads, int total, int tiles, PfWork& w) {
  w.splits = 1;
  if (a.splits > 1 && total > 0) {
    const int wgs = total * kv_heads;
    const int s = static_cast<int>(__lane_id()) + 1;
    constexpr int kMost = (1 << 24) - 1;
    const int cost = min(split_cost(s, min(tiles, kMost / 27), wgs, NW, a.slots, a.total_q * a.num_heads), kMost);
    const bool room = s == 1 || (s <= a.splits && s * wgs <= a.slots);
    w.splits = 64 - (wave_reduce(room ? ((kMost - cost) << 6) | (64 - s) : 0, MaxInt()) & 63);
  }
  const int per_block = kv_heads * w.splits;
  const int rank = uniform_int(static_cast<int>(blockIdx.x) / per_block);
  const int rest = static_cast<int>(blockIdx.x) - rank * per_block;
  w.split = uniform_int(rest / kv_heads);
  w.head = rest - w.split * kv_heads;
  return rank;
}

// Rank (0 first) -> (sequence, query block), the blocks with most keys first:
// the launch then ends on short blocks.  Blocks above a level u: a sum over
// the sequences; the rank's level comes from a binary search over u, its
// sequence from a scan over those with a block at that level.  Returns false
// for a workgroup beyond the real blocks.
template <int QT, int NW>
__device__ bool locate(const PrefillArgs& a, int kv_heads, bool flag, PfWork& w) {
  const int lane = __lane_id();
  if (a.batch <= 64) {  // one lane per sequence, loaded once
    int l0 = 0;
    const int n = lane < a.batch ? seq_blocks<QT>(a, lane, flag, l0) : 0;
    int lo = 0, hi = wave_reduce(n == 0 ? 0 : l0 + n, MaxInt());
    const int total = wave_reduce(n, AddInt());
    const int rank = pf_parts<NW>(a, kv_heads, total, (hi - 1) * QT / kPfKT + 1, w);
    if (rank >= total) return false;
    auto above = [&](int u) { return min(max(l0 + n - 1 - max(u, l0 - 1), 0), n); };
    // smallest u in [0, hi] with at most `rank` blocks above level u
    while (lo < hi) {
      const int mid = (lo + hi) / 2;
      if (wave_reduce(above(mid), AddInt()) <= rank) hi = mid;
      else lo = mid + 1;
    }
    const int at = (n > 0 && lo >= l0 && lo < l0 + n) ? 1 : 0;
    const int first = wave_reduce(above(lo), AddInt());
    const int incl = wave_scan(at, AddInt()) + first;
    const uint64_t hit = __builtin_amdgcn_ballot_w64(at && incl == rank + 1);
    const int l = __builtin_ctzll(hit);
    w.seq = __builtin_amdgcn_readfirstlane(l);
    w.qblock = lo - __builtin_amdgcn_readfirstlane(__shfl(l0, l));
    return true;
  }
  // larger batches: sequence by sequence, in reverse
  int total = 0, levels = 1, l0;
  for (int base = 0; base < a.batch; base += 64) {
    const int i = base + lane;
    const int n = i < a.batch ? seq_blocks<QT>(a, i, flag, l0) : 0;
    total += wave_reduce(n, AddInt());
    levels = max(levels, wave_reduce(n == 0 ? 0 : l0 + n, MaxInt()));
  }
  const int target = total - 1 - pf_parts<NW>(a, kv_heads, total, (levels - 1) * QT / kPfKT + 1, w);
  if (target < 0) return false;
  int before = 0;
  for (int base = 0; base < a.batch; base += 64) {
    const int i = base + lane;
    const int n = i < a.batch ? seq_blocks<QT>(a, i, false, l0) : 0;
    const int incl = wave_scan(n, AddInt()) + before;
    const uint64_t hit = __builtin_amdgcn_ballot_w64(i < a.batch && target < incl && target >= incl - n);
    if (hit != 0) {
      const int l = __builtin_ctzll(hit);
      w.seq = __builtin_amdgcn_readfirstlane(base + l);
      w.qblock = __builtin_amdgcn_readfirstlane(target - (__shfl(incl, l) - __shfl(n, l)));
      return true;
    }
    before = __shfl(incl, 63);
  }
  return false;
}

// Query operand (B of S^T = K Q^T).  Lane (g, c), g = lane / 32, holds query
// column c's dims 64 kh + 32 g .. + 31 for the two halves kh, the same dims as
// the K bytes it meets (row c of the block, LDS chunks 4 kh + 2 g and + 1).
//
// bf16 queries: the fp8 MFMA (32x32x64) on the K bytes as they are.  The
// column is scaled by 2^e so that its largest |q| lies in [128, 256) and
// split into two E4M3FN terms (hi, lo).  A bf16 value there is M * 2^k with
// an 8-bit M; hi rounds it to 4 significant bits, which leaves
// (M - 16 H) * 2^k with |M - 16 H| <= 8: at most 4 significant bits, held
// exactly by lo whenever 2^k is on E4M3FN's grid (elements of 2^-2 and up,
// 2^-10 of the column's largest), and within 2^-10 below (2^-18 of the
// largest), as a third term would be.  The MFMA's block scale of the operand
// takes 2^e back out, so that the scores of every column are in one unit and
// what turns them into log2 units (softmax scale and key scale) depends on
// the key alone.
//
// f16 queries (11 bits, which two terms do not hold): K converted to f16
// (exact) and v_mfma_f32_32x32x16_f16.
template <int QDT>
struct PfQOperand {
  i32x8 t[2][2];  // [lo, hi][half]
  int scale;      // 2^-e as the MFMA's E8M0 block scale, in every byte
};

template <>
struct PfQOperand<PRISM_DTYPE_F16> {
  f16x8 op[2][4];
};

template <int QDT>
__device__ __forceinline__ void pf_make_q(const u32x4 (&w)[2][4], PfQOperand<QDT>& q) {
  if constexpr (QDT == PRISM_DTYPE_F16) {
#pragma unroll
    for (int kh = 0; kh < 2; ++kh)
#pragma unroll
      for (int cc = 0; cc < 4; ++cc) q.op[kh][cc] = __builtin_bit_cast(f16x8, w[kh][cc]);
  } else {
    float mx = 0.f;
#pragma unroll
    for (int kh = 0; kh < 2; ++kh)
#pragma unroll
      for (int cc = 0; cc < 4; ++cc)
#pragma unroll
        for (int e = 0; e < 4; ++e)
          mx = fmaxf(mx, fmaxf(fabsf(bf16_bits_to_f32(w[kh][cc][e] & 0xFFFFu)), fabsf(bf16_bits_to_f32(w[kh][cc][e] >> 16))));
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(mx), __float_as_uint(mx), false, false);
    mx = fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
    // ilogb(mx) = frexp exponent - 1; clamped to E8M0's range (columns of
    // zeros, or of non-finite values, keep e = 0)
    const int e = (mx > 0.f && mx <= 3.0e38f) ? min(max(8 - __builtin_amdgcn_frexp_expf(mx), -120), 120) : 0;
    q.scale = (127 - e) * 0x01010101;
#pragma unroll
    for (int kh = 0; kh < 2; ++kh)
#pragma unroll
      for (int d = 0; d < 8; ++d) {
        const uint32_t w0 = w[kh][d / 2][2 * (d % 2)], w1 = w[kh][d / 2][2 * (d % 2) + 1];
        const float y[4] = {ldexpf(bf16_bits_to_f32(w0 & 0xFFFFu), e), ldexpf(bf16_bits_to_f32(w0 >> 16), e),
                            ldexpf(bf16_bits_to_f32(w1 & 0xFFFFu), e), ldexpf(bf16_bits_to_f32(w1 >> 16), e)};
        uint32_t parts[2];
        fp8_split<2>(y, parts);
        q.t[1][kh][d] = static_cast<int>(parts[0]);
        q.t[0][kh][d] = static_cast<int>(parts[1]);
      }
  }
}

// Two waves per SIMD: at most 256 VGPRs + AGPRs per lane.
// G: query heads of one kv head per workgroup; WHOLE: a tile lies in one page
// (page % 64 == 0), else its 16-key groups are looked up one by one.
constexpr int pf_waves(int g) { return g <= 4 ? 4 : 8; }
constexpr int pf_qtile(int g) { return kPfCols * pf_waves(g) / g; }

template <int QDT, int G, bool SCALED, bool WHOLE>
__global__ void __launch_bounds__(64 * pf_waves(G)) __attribute__((amdgpu_waves_per_eu(2)))
paged_prefill_kernel(const PrefillArgs a) {
  constexpr int NW = pf_waves(G);
  constexpr int QT = pf_qtile(G);
  constexpr int kRow = kPfD;                   // one key's payload row in LDS (bytes)
  constexpr int kPayload = kPfKT * kRow;       // K or V payload of a tile
  constexpr int kStage = 2 * kPayload + 2 * kPfKT * 4;
  __shared__ __attribute__((aligned(256))) uint8_t stages[4 * kStage];

  PfWork work;
  const bool found = locate<QT, NW>(a, a.num_heads / G, blockIdx.x == 0 && threadIdx.x < 64, work);
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    if (a.splits > 1) *a.used = work.splits;
    if (a.report != nullptr) {
      a.report[1] = a.cu_q[0];
      a.report[2] = a.cu_q[a.batch];
    }
  }
  if (!found) return;
  const int seq = uniform_int(work.seq), qblock = uniform_int(work.qblock);
  // two workgroups of a kv head (G is half its group) are kv_heads apart: with 8 kv heads on one XCD
  int h = uniform_int(work.head), qhead0 = h * G;
  if (G == 4 && a.groups == 8) {
    const int kv_heads = a.num_heads / 8, upper = h >= kv_heads;
    h -= upper * kv_heads;
    qhead0 = h * 8 + upper * G;
  }
  const int split = uniform_int(work.split), splits = uniform_int(work.splits);
  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid / 64);  // uniform: SGPR arithmetic below
  const int lane = tid % 64;
  const int c = lane % 32;
  const int g = lane / 32;
  const int qhead = qhead0 + wave % G;

  // sequence metadata in SGPRs: every branch on it below is uniform
  const int qs = __builtin_amdgcn_readfirstlane(a.cu_q[seq]);
  const int qlen = __builtin_amdgcn_readfirstlane(a.cu_q[seq + 1]) - qs;
  const int ctx = __builtin_amdgcn_readfirstlane(a.ctx[seq]);
  const int prefix = ctx - qlen;
  const int kend = prefix + min((qblock + 1) * QT, qlen);  // keys [0, kend) are needed
  const int qb0 = qblock * QT + wave / G * kPfCols;        // first query token of the wave
  const int qpos0 = prefix + qb0;                          // its position: query column 0
  const int qlast = qb0 < qlen ? qpos0 + kPfCols - 1 : -1; // no key past it is visible to the wave (no query: none at all)
  const int all_tiles = (kend + kPfKT - 1) / kPfKT;
  // this workgroup's tiles
  const int t0 = uniform_int(static_cast<int>(static_cast<int64_t>(all_tiles) * split / splits));
  const int t1 = uniform_int(static_cast<int>(static_cast<int64_t>(all_tiles) * (split + 1) / splits));
  const int32_t* bt_row = a.bt + static_cast<int64_t>(seq) * a.bt_sb;

  // the query's loads, then the first tiles', then the query's conversion
  const bool colv = qb0 + c < qlen;
  u32x4 qraw[2][4];
  {
    const uint16_t* src = static_cast<const uint16_t*>(a.q) + static_cast<int64_t>(qs + (colv ? qb0 + c : 0)) * a.q_st +
                          static_cast<int64_t>(qhead) * a.q_sh + 32 * g;
#pragma unroll
    for (int kh = 0; kh < 2; ++kh)
#pragma unroll
      for (int cc = 0; cc < 4; ++cc)
        qraw[kh][cc] = colv ? *reinterpret_cast<const u32x4*>(src + 64 * kh + 8 * cc) : u32x4{0u, 0u, 0u, 0u};
  }

  // ---- tile loads, straight into LDS (load-to-LDS, 16 B per lane): K rows,
  // V rows, K scales, V scales.  A wave's load covers 8 rows: LDS chunk x of
  // row t holds the row's global chunk x ^ swz(t).  Every load of a wave is
  // in one 16-key group and is all K or all V: a uniform 64-bit base (SGPRs)
  // plus a 32-bit per-lane offset that does not change from tile to tile.  The
  // base holds the row in its page and the offset the 8 rows from there, so
  // that both fit in 32 bits (the host checks that a page's rows of one head
  // span less than 2 GiB; a tile of several pages' rows may span more).
  // Asm so that the compiler's wait-count pass does not drain these loads
  // before each LDS read of the other stage.
  // (the 8-row groups of a wave have the parity of the wave: NW is even)
  uint32_t k_off, v_off;
  const int k_sp = static_cast<int>(a.k_sp), v_sp = static_cast<int>(a.v_sp);
  {
    const int part = (lane % 8) ^ pf_swz(8 * wave + lane / 8);
    k_off = static_cast<uint32_t>(lane / 8 * k_sp + part * 16);
    v_off = static_cast<uint32_t>(lane / 8 * v_sp + part * 16);
  }
  const uint8_t* k_head = a.k + h * a.k_sh;
  const uint8_t* v_head = a.v + h * a.v_sh;
  // waves 0 and 1 load the tile's K and V scales
  const float* s_head = wave ? a.vs + h * a.vs_sh : a.ks + h * a.ks_sh;
  const int64_t s_sn = wave ? a.vs_sn : a.ks_sn;
  const int s_sp = static_cast<int>(wave ? a.vs_sp : a.ks_sp);
  // Block ids: 64 consecutive entries of the table row in one register,
  // renewed every 64 pages; (pg, row) walk the pages without divisions.
  int pg = uniform_int(t0 * kPfKT / a.page);
  int row = t0 * kPfKT - pg * a.page;
  int ids_base = pg;
  auto load_ids = [&](int base) { return bt_row[static_cast<int64_t>(min(base + lane, a.width - 1)) * a.bt_sn]; };
  int ids = load_ids(ids_base);
  auto block_at = [&](int page) {
    if (page >= ids_base + 64) {
      ids_base = page;
      ids = load_ids(ids_base);
    }
    return __builtin_amdgcn_readlane(ids, page - ids_base);
  };
  auto load_chunks = [&](const uint8_t* base, uint32_t off, uint32_t lds) {
    asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1"
                 : : "v"(off), "s"(uniform_ptr(base)), "s"(lds) : "memory", "m0");
  };
  // Starts tile t's loads into stage st; returns whether all of a full tile's
  // loads were issued (wait_tiles counts on their number).
  auto issue_tile = [&](int t, uint8_t* st) -> bool {
    constexpr int kGroups = WHOLE ? 1 : kPfKT / 16;  // table lookups per tile
    constexpr int kGroupRows = kPfKT / kGroups;
    int blk[kGroups], row0[kGroups];
    bool ok = true;
#pragma unroll
    for (int x = 0; x < kGroups; ++x) {
      blk[x] = -1;
      row0[x] = row;
      if (WHOLE || t * kPfKT + x * kGroupRows < kend) {  // groups past the keys needed are not looked up
        blk[x] = block_at(pg);
        ok = ok && blk[x] >= 0 && blk[x] < a.num_blocks;
        row += kGroupRows;
        if (row == a.page) {
          row = 0;
          ++pg;
        }
      }
    }
    if (!ok) {
      if (tid == 0) flag_sequence(a, seq);
      return false;
    }
    const uint32_t st_lds = lds_addr(st) + static_cast<uint32_t>(wave) * 8 * kRow;
    constexpr int kLoads = 2 * kPfKT / 8 / NW;  // 8-row loads per wave, the first half of them K
#pragma unroll
    for (int l = 0; l < kLoads; ++l) {
      const bool isv = l >= kLoads / 2;
      const int tr = (isv ? l - kLoads / 2 : l) * NW * 8;  // the waves' first row in the tile
      const int wr = tr + wave * 8;                        // this wave's first row
      int b = blk[0], pr = row0[0] + wr;                   // its block and row in the page
      if constexpr (!WHOLE) {
        const int x = wr / 16;
#pragma unroll
        for (int y = 1; y < kGroups; ++y)
          if (x == y) b = blk[y], pr = row0[y] + wr - 16 * y;
        if (b < 0) continue;
      }
      const uint8_t* base = isv ? v_head + b * a.v_sn + pr * v_sp : k_head + b * a.k_sn + pr * k_sp;
      load_chunks(base, isv ? v_off : k_off,
                  __builtin_amdgcn_readfirstlane(st_lds + (isv ? kPayload : 0) + static_cast<uint32_t>(tr) * kRow));
    }
    if (wave < 2) {
      if constexpr (SCALED) {
        int b = blk[0], pr = row0[0];
        if constexpr (!WHOLE) {
#pragma unroll
          for (int y = 1; y < kGroups; ++y)
            if (lane / 16 == y) b = blk[y], pr = row0[y] - 16 * y;
        }
        const uint32_t lds = __builtin_amdgcn_readfirstlane(lds_addr(st) + 2 * kPayload + wave * kPfKT * 4);
        if constexpr (WHOLE) {
          const uint8_t* base = uniform_ptr(reinterpret_cast<const uint8_t*>(s_head + b * s_sn + pr * s_sp));
          asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dword %0, %1"
                       : : "v"(static_cast<uint32_t>(lane * s_sp * 4)), "s"(base), "s"(lds) : "memory", "m0");
        } else {
          const float* src = s_head + b * s_sn + (pr + lane) * s_sp;
          if (b >= 0)
            asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dword %0, off" : : "v"(src), "s"(lds)
                         : "memory", "m0");
        }
      } else {
        reinterpret_cast<float*>(st + 2 * kPayload)[wave * kPfKT + lane] = 1.f;
      }
    }
    return WHOLE || (t + 1) * kPfKT <= kend;
  };
  // A tile's K scales are multiplied by the softmax scale in log2 units, in
  // place, while the tile before it is computed: a score times its entry is
  // the exponent.
  auto scale_slot = [&](uint32_t st) { return reinterpret_cast<float*>(stages + st + 2 * kPayload) + lane; };
  // Waits for this wave's loads but those of the last tile issued.  They are
  // counted: a wave issues exactly kLoads loads for a tile, waves 0 and 1 one
  // more for its scales, whenever issue_tile returns true (`full`); otherwise,
  // and where no tile was issued, it waits for all.
  auto wait_tiles = [&](bool full) {
    constexpr int kLoads = 2 * kPfKT / 8 / NW;
    if (!full) __builtin_amdgcn_s_waitcnt(0xF70);                              // vmcnt(0)
    else if (SCALED && wave < 2) __builtin_amdgcn_s_waitcnt(0xF70 | (kLoads + 1));
    else __builtin_amdgcn_s_waitcnt(0xF70 | kLoads);
  };

  floatx16 acc[4];  // O^T: dims 32 n + 8 (r / 4) + 4 g + r % 4 of query column c
#pragma unroll
  for (int n = 0; n < 4; ++n)
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[n][r] = 0.f;
  // Columns without a query (all scores 0) start at 0: from -inf, which no key
  // of theirs would ever raise, every tile of the wave would count as rising
  // (8 query heads per kv head, 1000 tokens behind 8000: 468 against 271 us).
  float m_run = colv ? -INFINITY : 0.f, l_run = 0.f;

  // per-lane LDS offsets inside a stage, for keys 0..31 (32 rows further for
  // the rest); the lane's other chunks differ by an exclusive or
  const uint32_t k_rd = c * kRow + (((2 * g) ^ pf_swz(c)) << 4);
  uint32_t v_rd;
  {
    const int r = (lane % 16) >> 1;
    const int t = 8 * (r >> 2) + 4 * g + (r & 3);  // key of the 16-key group
    v_rd = kPayload + t * kRow + ((((lane / 16) % 2) ^ pf_swz(t)) << 4) + (lane & 1) * 8;
  }
  const uint32_t stage_base = lds_addr(stages);

  // A tile that could not be loaded (invalid block id) leaves its stage as it
  // was: the sequence is flagged and its rows are unspecified.
  uint32_t cur = 0, nxt = kStage, ahead = 2 * kStage, ld = 3 * kStage;  // stages of tiles t .. t + 3
  if (t0 < t1) issue_tile(t0, stages);
  if (t0 + 1 < t1) issue_tile(t0 + 1, stages + nxt);
  const bool full2 = t0 + 2 < t1 && issue_tile(t0 + 2, stages + ahead);
  PfQOperand<QDT> qop;
  pf_make_q<QDT>(qraw, qop);
  wait_tiles(full2);
  if (wave == 0) *scale_slot(cur) *= a.scale_log2;
  __syncthreads();
  // S^T = K Q^T of the tile at byte `st` of the LDS, in two chains of 32 keys
  // (b), each of four steps: the K bytes are the fp8 MFMA's A operand as they
  // are, smaller query term first; f16 queries take two 16-dim MFMAs a step.
  auto read_k = [&](uint32_t st, int b, u32x4 (&kw)[4]) {
#pragma unroll
    for (int x = 0; x < 4; ++x)
      kw[x] = *reinterpret_cast<const u32x4*>(stages + b * 32 * kRow + ((st + k_rd) ^ ((x % 2) << 4) ^ ((x / 2) << 6)));
  };
  auto qk_step = [&](int step, const u32x4 (&kw)[4], floatx16& sc) {
    if (step == 0)
#pragma unroll
      for (int r = 0; r < 16; ++r) sc[r] = 0.f;
    if constexpr (QDT == PRISM_DTYPE_F16) {
      const u32x4& w = kw[step];
#pragma unroll
      for (int y = 0; y < 2; ++y)
        sc = __builtin_amdgcn_mfma_f32_32x32x16_f16(fp8x8_to_f16x8(w[2 * y], w[2 * y + 1]),
                                                    qop.op[step / 2][2 * (step % 2) + y], sc, 0, 0, 0);
    } else {
      const int kh = step % 2;
      i32x8 ka;
#pragma unroll
      for (int x = 0; x < 8; ++x) ka[x] = static_cast<int>(kw[2 * kh + x / 4][x % 4]);
      sc = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(ka, qop.t[step / 2][kh], sc, 0, 0, 0, 0x7F7F7F7F, 0, qop.scale);
    }
  };

  bool first = true;  // no tile's scores seen yet
  floatx16 sa[2], sb[2];
#pragma unroll
  for (int b = 0; b < 2; ++b) {
    u32x4 kw[4];
    read_k(cur, b, kw);
#pragma unroll
    for (int step = 0; step < 4; ++step) qk_step(step, kw, sa[b]);
  }

  // One tile: the scores of the next one (MFMAs) are computed beside this
  // one's softmax (VALU).
  auto tile = [&](int t, floatx16 (&sc)[2], floatx16 (&sn)[2]) {
    // tile t + 3 streams into the stage last read by tile t - 1, which every
    // wave finished before the barrier that ended that iteration
    const bool full = t + 3 < t1 && issue_tile(t + 3, stages + ld);
    if (wave == 0 && t + 1 < t1) *scale_slot(nxt) *= a.scale_log2;
    const uint8_t* st = stages + cur;
    const int key0 = t * kPfKT;
    if (key0 <= qlast) {
      const float* scl = reinterpret_cast<const float*>(st + 2 * kPayload) + 4 * g;
      const bool both = key0 + 32 <= qlast;
      // V^T operands of 32 keys: v[m][n] for 16-key group m and dim tile n
      auto read_v = [&](int b, u32x2 (&v)[2][4]) {
#pragma unroll
        for (int m = 0; m < 2; ++m)
#pragma unroll
          for (int n = 0; n < 4; ++n)
            v[m][n] = __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr8_b64_v2i32(
                reinterpret_cast<lds_i32x2*>(stage_base + ((cur + v_rd) ^ (n << 5)) + (32 * b + 16 * m) * kRow)));
      };
      // Online softmax -> P (B of O^T += V^T P^T: the k-slots 8 g + 0..3 of
      // 16-key group m are keys 16 m + 4 g + 0..3, and 8 g + 4..7 the keys 8
      // further, the order the score rows come out in: row r of chain b is key
      // key0 + 32 b + 8 (r / 4) + 4 g + r % 4).
      //
      // P is first formed against the running max as it stands; the sum, which
      // is needed anyway, tells whether that was low enough (every p is at
      // most the lane's sum).  Only where it was not (or is no number: a score
      // of -inf against a running max of -inf weighs 0, not NaN), on the first
      // tile and on tiles with masked keys, are the scores' maxima taken and
      // the accumulators rescaled.
      bf16x8 pa[2][2];
      float ps;
      const bool masked = key0 + kPfKT - 1 > qpos0;  // (uniform) the diagonal or the block's end is in the tile
      //
      // An MFMA issues once the one before it is through, and holds its wave
      // until then.  So the eight of the next tile's scores are spread over
      // the softmax by hand: each slice is one of them (past the last tile on
      // stale bytes, for nothing), four scores' worth of softmax, and the LDS
      // reads of the slices after it.
      u32x4 kw[2][4];
      u32x2 vt[2][2][4];
      floatx4 ksv[2], vsv[2];
      read_k(nxt, 0, kw[0]);
      ksv[0] = *reinterpret_cast<const floatx4*>(scl);
      vsv[0] = *reinterpret_cast<const floatx4*>(scl + kPfKT);
      ps = 0.f;
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int x = 0; x < 8; ++x) {
        const int b = x / 4, i = x % 4;
        qk_step(i, kw[b], sn[b]);
        if (x < 7) {
          ksv[(x + 1) % 2] = *reinterpret_cast<const floatx4*>(scl + 32 * ((x + 1) / 4) + 8 * ((x + 1) % 4));
          vsv[(x + 1) % 2] = *reinterpret_cast<const floatx4*>(scl + kPfKT + 32 * ((x + 1) / 4) + 8 * ((x + 1) % 4));
        }
        if (x == 3) read_k(nxt, 1, kw[1]);  // (into the registers that chain 0 is done with)
        if (x == 6) read_v(0, vt[0]);
        float p[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          // v_exp_f32: arguments are at most 2^3 above the running max;
          // results below 2^-126 (flushed to 0) weigh nothing next to it
          p[j] = __builtin_amdgcn_exp2f(fmaf(sc[b][4 * i + j], ksv[x % 2][j], -m_run));
          pa[b][i / 2][4 * (i % 2) + j] = static_cast<__bf16>(p[j] * vsv[x % 2][j]);
        }
        ps += (p[0] + p[1]) + (p[2] + p[3]);
        __builtin_amdgcn_sched_barrier(0);
      }
      // (the pins keep the sums and the MFMAs in front of the branch)
      asm volatile("" : "+v"(ps), "+v"(pa[0][0]), "+v"(pa[0][1]), "+v"(pa[1][0]), "+v"(pa[1][1])
                   : "v"(sn[0]), "v"(sn[1]));
      if (first || masked || __builtin_amdgcn_ballot_w64(!(ps <= kPfSumLimit)) != 0) {
        first = false;
        // causal mask: key k is visible to column c iff it is at or before the
        // query's position; columns without a query see none, and their rows
        // are never written.  Keys past the block's last may hold any bytes
        // and scales (past the context, or not loaded).
        const int last = colv ? qpos0 + c - key0 - 4 * g : -1;  // last visible key, as a row offset
        float tmax = -INFINITY;
#pragma unroll
        for (int b = 0; b < 2; ++b)
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const floatx4 ksv = *reinterpret_cast<const floatx4*>(scl + 32 * b + 8 * i);
#pragma unroll
            for (int j = 0; j < 4; ++j) {
              const float x = sc[b][4 * i + j] * ksv[j];
              sc[b][4 * i + j] = 32 * b + 8 * i + j <= last ? x : -INFINITY;
              tmax = fmaxf(tmax, sc[b][4 * i + j]);
            }
          }
        {
          const auto sw = __builtin_amdgcn_permlane32_swap(__float_as_uint(tmax), __float_as_uint(tmax), false, false);
          tmax = fmaxf(__uint_as_float(sw[0]), __uint_as_float(sw[1]));
        }
        const float m_new = tmax > m_run ? tmax : m_run;
        // (no key seen: keep the accumulators, all zero, from (-inf) - (-inf))
        const float alpha = m_new > m_run ? __builtin_amdgcn_exp2f(m_run - m_new) : 1.f;
        m_run = m_new;
        l_run *= alpha;
#pragma unroll
        for (int n = 0; n < 4; ++n)
#pragma unroll
          for (int r = 0; r < 16; ++r) acc[n][r] *= alpha;
        const float m_use = (m_run == -INFINITY) ? 0.f : m_run;
        // Weights are dropped by the key's visibility and not by p, so that a
        // NaN stays one (compared anew: 32 lane masks kept from above would
        // fill the SGPRs).
        int seen = last;
        asm("" : "+v"(seen));
        ps = 0.f;
#pragma unroll
        for (int b = 0; b < 2; ++b)
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const floatx4 vsv = *reinterpret_cast<const floatx4*>(scl + kPfKT + 32 * b + 8 * i);
            float p[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) {
              p[j] = __builtin_amdgcn_exp2f(sc[b][4 * i + j] - m_use);  // 0 where masked
              pa[b][i / 2][4 * (i % 2) + j] = static_cast<__bf16>(32 * b + 8 * i + j <= seen ? p[j] * vsv[j] : 0.f);
            }
            ps += (p[0] + p[1]) + (p[2] + p[3]);
          }
      }
      l_run += ps;
      // O^T += V^T P^T
#pragma unroll
      for (int b = 0; b < 2; ++b) {
        if (b == 1 && !both) break;
        if (b == 0 && both) read_v(1, vt[1]);
        if (key0 + 32 * b + 32 > kend) {  // (uniform) 0 x a stray NaN would not be 0
          const int left = kend - key0 - 32 * b - 4 * g;
#pragma unroll
          for (int m = 0; m < 2; ++m)
#pragma unroll
            for (int half = 0; half < 2; ++half) {
              uint32_t keep = 0;
#pragma unroll
              for (int jj = 0; jj < 4; ++jj) keep |= (16 * m + 8 * half + jj < left) ? (0xFFu << (8 * jj)) : 0u;
#pragma unroll
              for (int n = 0; n < 4; ++n) vt[b][m][n][half] &= keep;
            }
        }
#pragma unroll
        for (int m = 0; m < 2; ++m)
#pragma unroll
          for (int n = 0; n < 4; ++n)
            acc[n] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fp8x8_to_bf16x8(vt[b][m][n][0], vt[b][m][n][1]), pa[b][m], acc[n],
                                                             0, 0, 0);
      }
    }
    wait_tiles(full);  // this wave's part of tile t + 2 has landed
    __syncthreads();
    const uint32_t done = cur;
    cur = nxt;
    nxt = ahead;
    ahead = ld;
    ld = done;
  };
  for (int t = t0; t < t1; t += 2) {
    tile(t, sa, sb);
    if (t + 1 < t1) tile(t + 1, sb, sa);
  }

  // ---- epilogue
  const auto lsw = __builtin_amdgcn_permlane32_swap(__float_as_uint(l_run), __float_as_uint(l_run), false, false);
  const float l_tot = __uint_as_float(lsw[0]) + __uint_as_float(lsw[1]);
  if (!colv) return;
  const int64_t tok = qs + qb0 + c;
  if (splits > 1) {
    const int64_t cell = (static_cast<int64_t>(split) * a.total_q + tok) * a.num_heads + qhead;
    float* dst = a.part + cell * kPfD + 4 * g;
#pragma unroll
    for (int n = 0; n < 4; ++n)
#pragma unroll
      for (int i = 0; i < 4; ++i)
        *reinterpret_cast<floatx4*>(dst + 32 * n + 8 * i) =
            floatx4{acc[n][4 * i], acc[n][4 * i + 1], acc[n][4 * i + 2], acc[n][4 * i + 3]};
    float* ml = a.part + static_cast<int64_t>(a.splits) * a.total_q * a.num_heads * kPfD + 2 * cell;
    if (g == 0) *reinterpret_cast<floatx2*>(ml) = floatx2{m_run, l_tot};
    return;
  }
  const float inv = l_tot == 0.f ? 0.f : 1.f / l_tot;  // (a NaN sum makes the row NaN)
  uint16_t* dst = static_cast<uint16_t*>(a.out) + tok * a.o_st + static_cast<int64_t>(qhead) * a.o_sh + 4 * g;
#pragma unroll
  for (int n = 0; n < 4; ++n)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      uint32_t o[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const float x = acc[n][4 * i + j] * inv;
        o[j] = (QDT == PRISM_DTYPE_F16) ? f32_to_f16_bits(x) : f32_to_bf16_bits(x);
      }
      acc[n][4 * i] = __uint_as_float(o[0] | (o[1] << 16));
      acc[n][4 * i + 1] = __uint_as_float(o[2] | (o[3] << 16));
    }
  if (a.out_vec) {
#pragma unroll
    for (int n = 0; n < 4; ++n)
#pragma unroll
      for (int i = 0; i < 4; ++i)
        *reinterpret_cast<u32x2*>(dst + 32 * n + 8 * i) =
            u32x2{__float_as_uint(acc[n][4 * i]), __float_as_uint(acc[n][4 * i + 1])};
    return;
  }
#pragma unroll
  for (int n = 0; n < 4; ++n)
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j)
        dst[32 * n + 8 * i + j] = static_cast<uint16_t>(__float_as_uint(acc[n][4 * i + j / 2]) >> (16 * (j & 1)));
}

// Merges the splits' partials: one wave per (token, query head), two dims per
// lane.  Rows outside every sequence hold no partials and are skipped, as is
// a row of an invalid sequence (the status word names it).
template <int QDT>
__global__ void __launch_bounds__(256) paged_prefill_merge_kernel(const PrefillArgs a) {
  const int64_t cell = static_cast<int64_t>(blockIdx.x) * 4 + threadIdx.x / 64;
  const int64_t cells = static_cast<int64_t>(a.total_q) * a.num_heads;
  if (cell >= cells) return;
  const int lane = threadIdx.x % 64;
  const int splits = *a.used;
  if (splits == 1) return;  // the outputs are written
  const int tok = static_cast<int>(cell / a.num_heads);
  if (tok < a.cu_q[0] || tok >= a.cu_q[a.batch]) return;
  // lane s holds split s's weight (at most 64 splits)
  const floatx2* ml = reinterpret_cast<const floatx2*>(a.part + a.splits * cells * kPfD) + cell;
  const floatx2 mine = lane < splits ? ml[lane * cells] : floatx2{-INFINITY, 0.f};
  // Parts without a visible key hold zeros and weigh nothing; a NaN sum goes
  // through whatever its part's weight is.
  const bool live = mine[1] != 0.f;
  float m = live ? mine[0] : -INFINITY;
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) m = fmaxf(m, __shfl_xor(m, off));
  const float weight = live ? __builtin_amdgcn_exp2f(mine[0] - m) : 0.f;
  const floatx2* row = reinterpret_cast<const floatx2*>(a.part) + cell * (kPfD / 2) + lane;
  float l = 0.f, o0 = 0.f, o1 = 0.f;
#pragma unroll 4
  for (int s = 0; s < splits; ++s) {
    const float w = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(weight), s));
    const floatx2 v = row[s * cells * (kPfD / 2)];
    l = fmaf(w, __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(mine[1]), s)), l);
    o0 = fmaf(w, v[0], o0);
    o1 = fmaf(w, v[1], o1);
  }
  const float inv = l == 0.f ? 0.f : 1.f / l;
  uint16_t* dst = static_cast<uint16_t*>(a.out) + static_cast<int64_t>(tok) * a.o_st +
                  (cell - static_cast<int64_t>(tok) * a.num_heads) * a.o_sh + 2 * lane;
  dst[0] = (QDT == PRISM_DTYPE_F16) ? f32_to_f16_bits(o0 * inv) : f32_to_bf16_bits(o0 * inv);
  dst[1] = (QDT == PRISM_DTYPE_F16) ? f32_to_f16_bits(o1 * inv) : f32_to_bf16_bits(o1 * inv);
}

// Query heads per workgroup: all of a kv head's, but 4 of 8 where the tables
// hold few keys.  Eight waves fill a CU, so that a workgroup's lookup, loads
// and output lie bare between its tiles; two of four waves hide each other's
// and read the keys twice.  64 / 8 heads, pages of 256: a prompt of 16 tokens
// 15.0 us with eight and 11.4 with four, 80 of 100 188 and 153, 4 of 2048 375
// and 353, 300 tokens behind 1000 (16 sequences) 261 and 258; behind 2000 405
// and 407, without scales 397 and 415; 4 x 2048 behind 8000 2290 and 2323,
// without scales 2235 and 2360.
constexpr int64_t kPfHalfKeys = 2048;
int heads_per_wg(int groups, int64_t capacity) { return groups == 8 && capacity <= kPfHalfKeys ? 4 : groups; }

// Query blocks that the launch provides for: every sequence may end in a
// partial block.
int64_t block_bound(int total_q, int batch, int g) { return ceil_div(total_q, pf_qtile(g)) + batch; }

// Workgroups that the chip holds at once: the kernel fits eight waves on a CU.
int64_t chip_slots(int g) { return static_cast<int64_t>(device_cu_count()) * 8 / pf_waves(g); }

// Most workgroups per (block, kv head), for the fewest blocks that total_q rows
// make: where these leave slots free, parts of at least 4 tiles of the longest
// context the tables can hold; 1 where no number of parts pays even for that
// one (shorter contexts gain less).  The kernel chooses by the real blocks.
int split_count(int total_q, int num_heads, int num_kv_heads, int64_t capacity) {
  const int g = heads_per_wg(num_heads / num_kv_heads, capacity);
  const int64_t slots = chip_slots(g), wgs = ceil_div(total_q, pf_qtile(g)) * (num_heads / g);
  const int most = static_cast<int>(std::min<int64_t>({slots / wgs, capacity / (4 * kPfKT), 64}));
  const int tiles = static_cast<int>(std::min<int64_t>(ceil_div(capacity, kPfKT), 1 << 24));
  auto cost = [&](int s) {  // (two parts or more: few workgroups, and so few rows)
    return split_cost(s, tiles, static_cast<int>(wgs), pf_waves(g), static_cast<int>(slots), total_q * num_heads);
  };
  for (int s = 2; s <= most; ++s)
    if (cost(s) < cost(1)) return most;
  return 1;
}

constexpr int64_t kPfPartOffset = 256;  // the partials follow the count of splits

int64_t split_workspace(int splits, int total_q, int num_heads) {
  return splits > 1 ? kPfPartOffset + static_cast<int64_t>(splits) * total_q * num_heads * (kPfD + 2) * 4 : 0;
}

template <int QDT, int G>
int launch_prefill(const PrefillArgs& a, bool scaled, hipStream_t stream) {
  int64_t blocks = block_bound(a.total_q, a.batch, G) * (a.num_heads / G);
  if (a.splits > 1) blocks = std::max<int64_t>(blocks, a.slots);  // split blocks never take more than the slots
  if (blocks > INT32_MAX) {
    set_error("prism_paged_prefill: too many query blocks for one launch");
    return PRISM_ERR_INVALID;
  }
  const dim3 grid(static_cast<unsigned>(blocks)), block(64 * pf_waves(G));
  const bool whole = a.page % kPfKT == 0;
  if (scaled && whole) hipLaunchKernelGGL((paged_prefill_kernel<QDT, G, true, true>), grid, block, 0, stream, a);
  else if (scaled) hipLaunchKernelGGL((paged_prefill_kernel<QDT, G, true, false>), grid, block, 0, stream, a);
  else if (whole) hipLaunchKernelGGL((paged_prefill_kernel<QDT, G, false, true>), grid, block, 0, stream, a);
  else hipLaunchKernelGGL((paged_prefill_kernel<QDT, G, false, false>), grid, block, 0, stream, a);
  if (int rc = check_launch("paged_prefill_kernel launch")) return rc;
  if (a.splits == 1) return PRISM_OK;
  const int64_t cells = static_cast<int64_t>(a.total_q) * a.num_heads;
  hipLaunchKernelGGL((paged_prefill_merge_kernel<QDT>), dim3(static_cast<unsigned>(ceil_div(cells, 4))), dim3(256), 0,
                     stream, a);
  return check_launch("paged_prefill_merge_kernel launch");
}

template <int QDT>
int dispatch_groups(const PrefillArgs& a, int g, bool scaled, hipStream_t stream) {
  switch (g) {
    case 1: return launch_prefill<QDT, 1>(a, scaled, stream);
    case 2: return launch_prefill<QDT, 2>(a, scaled, stream);
    case 4: return launch_prefill<QDT, 4>(a, scaled, stream);
    case 8: return launch_prefill<QDT, 8>(a, scaled, stream);
    default:
      set_error("prism_paged_prefill: GQA group size %d is not 1, 2, 4 or 8", a.groups);
      return PRISM_ERR_LAYOUT;
  }
}

}  // namespace

// Loads this file's code object now rather than at its first kernel launch.
int preload_paged_prefill() {
  hipFuncAttributes attr;
  return check_hip(hipFuncGetAttributes(&attr, reinterpret_cast<const void*>(&paged_prefill_kernel<PRISM_DTYPE_BF16, 4, true, true>)), "preload_paged_prefill");
}

}  // namespace prism

extern "C" int64_t prism_paged_prefill_workspace_bytes(int batch, int total_q, int num_heads, int num_kv_heads,
                                                       int page_size, int width) {
  using namespace prism;
  if (batch <= 0 || total_q <= 0 || num_heads <= 0 || num_kv_heads <= 0 || num_heads % num_kv_heads != 0 ||
      num_heads / num_kv_heads > kPfMaxWaves || page_size <= 0 || width < 0)
    return 0;
  const int64_t capacity = static_cast<int64_t>(width) * page_size;
  return split_workspace(split_count(total_q, num_heads, num_kv_heads, capacity), total_q, num_heads);
}

extern "C" int prism_paged_prefill_ws(const void* q, int q_dtype, const int64_t q_strides[3], const void* k_cache,
                                      const void* v_cache, int cache_dtype, const int64_t k_strides[4],
                                      const int64_t v_strides[4], const float* k_scale, const float* v_scale,
                                      const int64_t k_scale_strides[3], const int64_t v_scale_strides[3],
                                      const int32_t* block_tables, const int64_t bt_strides[2],
                                      const int32_t* context_lens, const int32_t* cu_seqlens_q, void* out,
                                      const int64_t out_strides[3], int batch, int total_q, int num_heads,
                                      int num_kv_heads, int head_dim, int page_size, int num_blocks, int width,
                                      float scale, int32_t* status, void* workspace, int64_t workspace_bytes, int32_t* report,
                                      void* stream_ptr) {
  using namespace prism;
  clear_error();
  if (batch < 0 || total_q < 0 || num_heads <= 0 || num_kv_heads <= 0 || page_size <= 0 || num_blocks < 0 ||
      width < 0) {
    set_error("prism_paged_prefill: invalid geometry");
    return PRISM_ERR_INVALID;
  }
  if (num_heads % num_kv_heads != 0 || num_heads / num_kv_heads > kPfMaxWaves) {
    set_error("prism_paged_prefill: num_heads=%d / num_kv_heads=%d must be an integer group of at most %d",
              num_heads, num_kv_heads, kPfMaxWaves);
    return PRISM_ERR_LAYOUT;
  }
  if (head_dim != kPfD) {
    set_error("prism_paged_prefill: head_dim must be %d, got %d", kPfD, head_dim);
    return PRISM_ERR_LAYOUT;
  }
  if (cache_dtype != PRISM_DTYPE_FP8_E4M3FN) {
    set_error("prism_paged_prefill: the cache must be FP8 E4M3FN (dtype code %d)", cache_dtype);
    return PRISM_ERR_LAYOUT;
  }
  if (q_dtype != PRISM_DTYPE_BF16 && q_dtype != PRISM_DTYPE_F16) {
    set_error("prism_paged_prefill: q must be bf16 or float16 (dtype code %d)", q_dtype);
    return PRISM_ERR_LAYOUT;
  }
  if (page_size % 16 != 0) {
    set_error("prism_paged_prefill: page size must be a multiple of 16, got %d", page_size);
    return PRISM_ERR_LAYOUT;
  }
  if ((k_scale == nullptr) != (v_scale == nullptr)) {
    set_error("prism_paged_prefill: K/V scale caches must be provided together");
    return PRISM_ERR_INVALID;
  }
  if (!q_strides || !k_strides || !v_strides || !bt_strides || !out_strides || !status ||
      (k_scale && (!k_scale_strides || !v_scale_strides))) {
    set_error("prism_paged_prefill: null argument");
    return PRISM_ERR_INVALID;
  }
  if (q_strides[2] != 1 || k_strides[3] != 1 || v_strides[3] != 1 || out_strides[2] != 1 ||
      !aligned(q, 16) || !aligned(k_cache, 16) || !aligned(v_cache, 16) || q_strides[0] % 8 || q_strides[1] % 8 ||
      k_strides[0] % 16 || k_strides[1] % 16 || k_strides[2] % 16 || v_strides[0] % 16 || v_strides[1] % 16 ||
      v_strides[2] % 16) {
    set_error("prism_paged_prefill: q, K/V and out need unit-stride head dims and 16-byte aligned rows");
    return PRISM_ERR_LAYOUT;
  }
  // tile loads address a page's rows of one head by a 32-bit offset
  if ((page_size - 1) * k_strides[1] + kPfD > INT32_MAX || (page_size - 1) * v_strides[1] + kPfD > INT32_MAX ||
      (k_scale && ((page_size - 1) * k_scale_strides[1] >= INT32_MAX / 4 ||
                   (page_size - 1) * v_scale_strides[1] >= INT32_MAX / 4))) {
    set_error("prism_paged_prefill: a page's token rows must span less than 2 GiB");
    return PRISM_ERR_LAYOUT;
  }
  if (batch == 0 || total_q == 0) return PRISM_OK;
  PrefillArgs a{};
  a.q = q;
  a.q_st = q_strides[0];
  a.q_sh = q_strides[1];
  a.k = static_cast<const uint8_t*>(k_cache);
  a.v = static_cast<const uint8_t*>(v_cache);
  a.k_sn = k_strides[0], a.k_sp = k_strides[1], a.k_sh = k_strides[2];
  a.v_sn = v_strides[0], a.v_sp = v_strides[1], a.v_sh = v_strides[2];
  a.ks = k_scale;
  a.vs = v_scale;
  if (k_scale) {
    a.ks_sn = k_scale_strides[0], a.ks_sp = k_scale_strides[1], a.ks_sh = k_scale_strides[2];
    a.vs_sn = v_scale_strides[0], a.vs_sp = v_scale_strides[1], a.vs_sh = v_scale_strides[2];
  }
  a.bt = block_tables;
  a.bt_sb = bt_strides[0];
  a.bt_sn = bt_strides[1];
  a.ctx = context_lens;
  a.cu_q = cu_seqlens_q;
  a.out = out;
  a.o_st = out_strides[0];
  a.o_sh = out_strides[1];
  a.batch = batch;
  a.num_heads = num_heads;
  a.groups = num_heads / num_kv_heads;
  a.page = page_size;
  a.num_blocks = num_blocks;
  a.width = width;
  a.scale_log2 = scale * 1.4426950408889634f;
  a.status = status;
  a.report = report;
  a.out_vec = aligned(out, 8) && out_strides[0] % 4 == 0 && out_strides[1] % 4 == 0;
  a.total_q = total_q;
  const int64_t capacity = static_cast<int64_t>(width) * page_size;
  const int g = heads_per_wg(a.groups, capacity);
  a.slots = static_cast<int>(chip_slots(g));
  a.splits = split_count(total_q, num_heads, num_kv_heads, capacity);
  // without scratch for the partials the keys are not split
  if (a.splits > 1 &&
      (workspace == nullptr || !aligned(workspace, 16) || workspace_bytes < split_workspace(a.splits, total_q, num_heads)))
    a.splits = 1;
  a.used = static_cast<int*>(workspace);
  a.part = a.splits > 1 ? reinterpret_cast<float*>(static_cast<uint8_t*>(workspace) + kPfPartOffset) : nullptr;
  hipStream_t stream = static_cast<hipStream_t>(stream_ptr);
  const bool scaled = k_scale != nullptr;
  if (q_dtype == PRISM_DTYPE_F16) return dispatch_groups<PRISM_DTYPE_F16>(a, g, scaled, stream);
  return dispatch_groups<PRISM_DTYPE_BF16>(a, g, scaled, stream);
}

extern "C" int prism_paged_prefill(const void* q, int q_dtype, const int64_t q_strides[3], const void* k_cache,
                                   const void* v_cache, int cache_dtype, const int64_t k_strides[4],
                                   const int64_t v_strides[4], const float* k_scale, const float* v_scale,
                                   const int64_t k_scale_strides[3], const int64_t v_scale_strides[3],
                                   const int32_t* block_tables, const int64_t bt_strides[2],
                                   const int32_t* context_lens, const int32_t* cu_seqlens_q, void* out,
                                   const int64_t out_strides[3], int batch, int total_q, int num_heads,
                                   int num_kv_heads, int head_dim, int page_size, int num_blocks, int width,
                                   float scale, int32_t* status, void* stream_ptr) {
  return prism_paged_prefill_ws(q, q_dtype, q_strides, k_cache, v_cache, cache_dtype, k_strides, v_strides, k_scale,
                                v_scale, k_scale_strides, v_scale_strides, block_tables, bt_strides, context_lens,
                                cu_seqlens_q, out, out_strides, batch, total_q, num_heads, num_kv_heads, head_dim,
                                page_size, num_blocks, width, scale, status, nullptr, 0, nullptr, stream_ptr);
}
