// Sparse shared-KV attention decode for MI355X (gfx950 / CDNA4).
//
// Replaces the reference's fused TileLang kernels (kernel.py:_build_swa /
// _build_cfa / _build_scfa and sparse_flash_mla_kernel.py:_build_swa/_hca/_csa)
// with one metadata-driven HIP kernel plus a split-KV merge kernel.
//
// Work decomposition
//   One workgroup per FA metadata row; it walks its items (query row x 32- or
//   64-head m-block) and, inside each, its blocks of the attended list [window
//   rows ++ compressed positions]. All query heads of a token share every
//   gathered KV row (shared KV, N2 = 1): a 32-row tile is loaded once into LDS
//   and read by every wave, as K for Q·Kᵀ and (first head_dim_v columns) as V
//   for P·V.
//
// Waves (one per SIMD; details at attn2_kernel): head groups of 32 heads x 2
// halves of d_qk / d_v.
//   Q·Kᵀ: each wave computes a partial Sᵀ[32 rows x 32 heads] over its half of
//         d_qk with v_mfma_f32_32x32x16 (A = K rows from LDS, B = Qᵀ held in
//         AGPRs); the two partials of a head group meet through LDS, so both
//         waves hold the same full Sᵀ.
//   softmax: exp2 domain on 32 rows (two tiles) x 1 head per lane, in
//         registers; the running max moves at every 64-row step whose max
//         exceeds it.
//   P·V:  each wave accumulates Oᵀ[its dv half x 32 heads] (A = Vᵀ via
//         ds_read_b64_tr_b16 from the row-major tile, B = Pᵀ straight from the
//         Sᵀ registers).
//
// Gather: global_load_lds_dwordx4 (16 B per lane straight into LDS, no VGPR
//   staging) into a 3-stage ring, issued between the Q·Kᵀ MFMAs; rows of a
//   tile are rotated by 16-byte chunks so both the Kᵀ reads (b128) and the
//   transposed V reads (tr_b16) are bank-conflict free. fp8 cache rows are
//   loaded into VGPRs instead and dequantized into the same bf16 layout.
//
// Numerics follow golden.py:156-200: fp32 scores, P rounded to the input
// dtype before P·V while the running sum uses fp32 P, out = acc / l rounded
// RNE, lse = m + ln(l). Split pieces emit (acc / l, lse) without the sink;
// the merge adds the sink once.
#include <hip/hip_runtime.h>
#include <math.h>
#include <stdint.h>
#include <string.h>

#include <mutex>
#include <string>
#include <type_traits>

#include "../../include/sas_mi355x.h"
#include "sas_items.h"

namespace sas {

static thread_local std::string g_last_error;
void set_error(const std::string& msg) { g_last_error = msg; }

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef short i16x4 __attribute__((ext_vector_type(4)));
typedef short i16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef int i32x2 __attribute__((ext_vector_type(2)));
typedef int i32x4 __attribute__((ext_vector_type(4)));
typedef int i32x8 __attribute__((ext_vector_type(8)));

#define SAS_LDS __attribute__((address_space(3)))
#define SAS_GLOBAL __attribute__((address_space(1)))

constexpr int TILE = 32;        // KV rows per pipeline stage
constexpr uint32_t ROW_INVALID = 0xFFFFFFFFu;
constexpr float LOG2E = 1.4426950408889634f;
constexpr float LN2 = 0.6931471805599453f;
#ifndef SAS_KPF
#define SAS_KPF 8  // K operand reads in flight per wave (attn2_kernel)
#endif
#ifndef SAS_PV_SPREAD
#define SAS_PV_SPREAD 0  // P·V MFMA order of the rescaling tile (attn2_kernel)
#endif
#ifndef SAS_VPF
#define SAS_VPF 4  // Vᵀ operands in flight per wave (attn2_kernel)
#endif

template <typename T> struct MfmaOps;
template <> struct MfmaOps<__bf16> {
  typedef bf16x8 vec8;
  static __device__ inline f32x16 mma(i16x8 a, i16x8 b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a),
                                                   __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
  }
  static __device__ inline short from_f32(float x) {
    return __builtin_bit_cast(short, (__bf16)x);
  }
};
template <> struct MfmaOps<_Float16> {
  typedef f16x8 vec8;
  static __device__ inline f32x16 mma(i16x8 a, i16x8 b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, a),
                                                  __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
  }
  static __device__ inline short from_f32(float x) {
    return __builtin_bit_cast(short, (_Float16)x);
  }
};

// LDS stage layout (one 32-row tile).
//   main part, dims 0..511: row r occupies MAIN_SLOTS = 68 sixteen-byte slots
//     (1088 B); its chunk c (dims 8c..8c+7) sits in slot c + rot(r) with
//     rot(r) = (r >> 2) & 3. One DMA instruction (64 lanes x 16 B) fills one
//     row, and every read address is one per-lane base plus an immediate.
//   rope part, dims 512..575 (head_dim 576): 8 slots per row after the main
//     part; chunk 64 + c' of row r sits in slot 8 r + ((c' + (r >> 1)) & 7), so
//     one DMA instruction fills 8 rows.
// With 64 banks x 4 B (16 sixteen-byte bank groups):
//   * Kᵀ reads (ds_read_b128, 16 lanes = rows r..r+15 at one chunk) hit bank
//     groups (4 r + rot(r) + c) mod 16 (main) or (8 r + ((c' + r/2) & 7)) mod 16
//     (rope), all distinct;
//   * Vᵀ reads (ds_read_b64_tr_b16, 32 lanes = 4 consecutive rows x 4 chunks)
//     start at 4 (r % 4) + rot(r) = {0, 4, 8, 12} + const, four disjoint spans.
constexpr int MAIN_SLOTS = 68;
constexpr int MAIN_ROW_BYTES = MAIN_SLOTS * 16;
constexpr int MAIN_BYTES = TILE * MAIN_ROW_BYTES;      // 34816
constexpr int ROPE_BYTES = TILE * 8 * 16;              // 4096
__device__ __host__ inline int row_rot(int r) { return (r >> 2) & 3; }
__device__ __host__ inline int main_row_base(int r) { return r * MAIN_ROW_BYTES + row_rot(r) * 16; }
__device__ __host__ inline int rope_slot(int r, int cr) { return 8 * r + ((cr + (r >> 1)) & 7); }

// Combine lane l with lane l ^ 32 in registers (v_permlane32_swap): both
// halves end up with the identical result.
__device__ inline float wave_max_pair(float v) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
__device__ inline float wave_sum_pair(float v) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);  // lower half + upper half
}

// Direct-to-LDS 16-byte loads: lane's data lands at M0 + lane * 16.
// Issued through inline asm so the compiler does not serialise them against
// unrelated LDS reads; completion is tracked by hand with s_waitcnt vmcnt.
// The compiler's hazard pass cannot see inside the asm, which therefore keeps two
// rules itself: an LDS DMA needs one wait state after the SALU write of M0 it reads,
// and a VMEM instruction five after a VALU write of an SGPR it reads. Row addresses
// come from v_readlane (a VALU write), so the DMA takes a copy made by an s_mov_b64:
// scalar instructions may read such an SGPR at once, and an SGPR written by one is
// interlocked. The s_mov_b64 is M0's wait state, too.
// Rows are fetched with the streaming cache policy (sc0 nt): each row is read
// once per workgroup (the second 64-head m-block of a token reads it on the
// same XCD shortly after), and the non-temporal fills shortened the stalls of
// the DMA issue on every tile (measured about 3.5 us of 66 at B = 64, H = 128).
__device__ inline void dma16_sbase(const void* sbase, uint32_t voff, uint32_t lds_base) {
  uint64_t base;
  asm volatile(
      "s_mov_b32 m0, %3\n\t"
      "s_mov_b64 %0, %2\n\t"
      "global_load_lds_dwordx4 %1, %0 sc0 nt\n\t"
      : "=&s"(base)
      : "v"(voff), "s"(sbase), "s"(lds_base)
      : "memory");
}
// dma16_sbase on the lanes of `lanes` only (lane i still writes lds_base + 16 i):
// exec is narrowed and restored inside the statement, so the compiler never sees
// it change
__device__ inline void dma16_sbase_lanes(const void* sbase, uint32_t voff, uint32_t lds_base,
                                         uint64_t lanes) {
  uint64_t saved, base;
  asm volatile(
      "s_mov_b64 %0, exec\n\t"
      "s_mov_b64 exec, %5\n\t"
      "s_mov_b32 m0, %4\n\t"
      "s_mov_b64 %1, %3\n\t"
      "global_load_lds_dwordx4 %2, %1 sc0 nt\n\t"
      "s_mov_b64 exec, %0\n\t"
      : "=&s"(saved), "=&s"(base)
      : "v"(voff), "s"(sbase), "s"(lds_base), "s"(lanes)
      : "memory");
}
__device__ inline void dma16_vaddr(const void* gptr, uint32_t lds_base) {
  asm volatile(
      "s_mov_b32 m0, %1\n\t"
      "s_nop 0\n\t"
      "global_load_lds_dwordx4 %0, off sc0 nt\n\t" ::"v"(gptr),
      "s"(lds_base)
      : "memory");
}

// A read-only kernel input at a wave-uniform address, as a scalar load (through
// the constant address space: the compiler cannot prove on its own that the
// kernel's stores leave these arrays alone, and would use a vector load).
__device__ inline int32_t ld_uniform(const int32_t* p) {
  return *(const __attribute__((address_space(4))) int32_t*)p;
}

// Query rows of the batches, in one of three forms (SAS_QLENS_*, told apart by the
// null pointers the launch leaves): `first` and `rows` arrays; cumulative row counts
// (first only: batch b's rows end where those of b + 1 begin); or as many rows in
// every batch (neither). Batch b starts at token start(first[b]) and has
// count(rows[b], first[b]) rows; reads of the unused arrays go to seqused_kv.
struct QRows {
  const int32_t *first, *rows;
  int uniform;      // rows of every batch, or -1
  bool cumulative;
  __device__ explicit QRows(const SasAttnArgs& a)
      : first(a.q_prefix ? a.q_prefix : a.seqused_kv),
        rows(!a.q_prefix ? a.seqused_kv : a.act_q_lens ? a.act_q_lens : a.q_prefix + 1),
        uniform(a.q_prefix ? -1 : a.total_tokens / a.batch),
        cumulative(a.q_prefix && !a.act_q_lens) {}
  __device__ int start(int b, int first_b) const { return uniform < 0 ? first_b : b * uniform; }
  __device__ int count(int rows_b, int first_b) const {
    return uniform >= 0 ? uniform : cumulative ? rows_b - first_b : rows_b;
  }
};

// Cumulative row counts: tokens outside [lo, hi) belong to no row of the schedule;
// their output and lse rows are zeroed, spread over the workgroups (a fill of every
// output row in front of the kernel took 12 us of a 128 x 128-head decode call). A
// launch may be for more FA rows than are in use: the shares of rows out of use go to
// the row in use before them, those before any to the first.
template <typename T>
__device__ inline void zero_unowned_rows(const SasAttnArgs& a, int lo, int hi, int wg, int nwg,
                                         int tid, int nthreads) {
  lo = lo < 0 ? 0 : (lo < a.total_tokens ? lo : a.total_tokens);
  hi = hi < lo ? lo : (hi < a.total_tokens ? hi : a.total_tokens);
  const int n = lo + a.total_tokens - hi;
  if (n == 0) return;
  auto out_of_use = [&](int row) { return a.metadata[row * SAS_FA_METADATA_SIZE] == 0; };
  int first = wg, end = wg + 1;
  while (end < nwg && out_of_use(end)) ++end;
  while (first > 0 && out_of_use(first - 1)) --first;
  if (first > 0) first = wg;
  for (int share = first; share < end; ++share)
    for (int r = share; r < n; r += nwg) {
      const size_t row = (size_t)(r < lo ? r : hi + r - lo) * a.num_heads;
      i32x4* out = (i32x4*)((T*)a.out + row * a.head_dim_v);
      for (int k = tid; k < a.num_heads * a.head_dim_v / 8; k += nthreads) out[k] = (i32x4){0, 0, 0, 0};
      for (int k = tid; k < a.num_heads; k += nthreads) a.lse[row + k] = 0.0f;
    }
}

template <int N>
__device__ inline void wait_vmcnt() {
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

// N dword loads and their vmcnt(0) wait in ONE asm statement. Loads issued by
// separate asm statements leave the compiler free to place code between a load
// and its wait; under register pressure that code can spill the destination
// register (storing its stale value) and reuse it, and the load then lands in a
// register that holds something else by then (an address, which faulted the GPU).
// Early-clobber outputs keep the destinations apart from the address operands.
template <int N>
__device__ inline void gather_dwords_wait(int (&v)[N], const int32_t* const (&p)[N]) {
  static_assert(N == 6 || N == 8, "gather_dwords_wait: 6 or 8 loads");
  if constexpr (N == 6) {
    asm volatile(
        "global_load_dword %0, %6, off\n\t"
        "global_load_dword %1, %7, off\n\t"
        "global_load_dword %2, %8, off\n\t"
        "global_load_dword %3, %9, off\n\t"
        "global_load_dword %4, %10, off\n\t"
        "global_load_dword %5, %11, off\n\t"
        "s_waitcnt vmcnt(0)"
        : "=&v"(v[0]), "=&v"(v[1]), "=&v"(v[2]), "=&v"(v[3]), "=&v"(v[4]), "=&v"(v[5])
        : "v"(p[0]), "v"(p[1]), "v"(p[2]), "v"(p[3]), "v"(p[4]), "v"(p[5])
        : "memory");
  } else {
    asm volatile(
        "global_load_dword %0, %8, off\n\t"
        "global_load_dword %1, %9, off\n\t"
        "global_load_dword %2, %10, off\n\t"
        "global_load_dword %3, %11, off\n\t"
        "global_load_dword %4, %12, off\n\t"
        "global_load_dword %5, %13, off\n\t"
        "global_load_dword %6, %14, off\n\t"
        "global_load_dword %7, %15, off\n\t"
        "s_waitcnt vmcnt(0)"
        : "=&v"(v[0]), "=&v"(v[1]), "=&v"(v[2]), "=&v"(v[3]), "=&v"(v[4]), "=&v"(v[5]),
          "=&v"(v[6]), "=&v"(v[7])
        : "v"(p[0]), "v"(p[1]), "v"(p[2]), "v"(p[3]), "v"(p[4]), "v"(p[5]), "v"(p[6]),
          "v"(p[7])
        : "memory");
  }
}

// Cache rows that a tile holds but the softmax masks (tile tails, -1 and
// out-of-range top-k ids) are read from this all-zero row instead of the
// pool: their P is 0, and 0 * V is only 0 when V is finite, which an
// unwritten pool row need not be. Large enough for every row format.
__device__ __attribute__((aligned(256))) unsigned char g_zero_row[1152];

// What the attention kernels are launched with: the call's arguments and the
// divisors of the index arithmetic as multipliers.
struct KernelArgs : SasAttnArgs {
  FastDiv ori_bs, cmp_bs, ratio;  // of the block sizes and cmp_ratio
};

// The launch's arguments, read again from the kernel argument segment. Each phase of an
// item (its geometry and rows, the epilogue, the merge) takes its own copy: the few
// scalar loads it needs hit the scalar cache, while arguments (and what the compiler
// derives from them outside the item loop) kept in registers across the tile loop
// overflow the scalar registers into lanes of vector registers, and that spilling
// alone was a third of the instructions before a call's first row loads.
__device__ __forceinline__ KernelArgs fresh_args() {
  typedef const __attribute__((address_space(4))) uint32_t* seg_p;
  seg_p p = (seg_p)__builtin_amdgcn_kernarg_segment_ptr();
  asm volatile("" : "+s"(p));
  KernelArgs a;
  static_assert(sizeof(KernelArgs) % 4 == 0, "whole words");
  uint32_t words[sizeof(KernelArgs) / 4];
#pragma unroll
  for (int i = 0; i < (int)(sizeof(KernelArgs) / 4); ++i) words[i] = p[i];
  __builtin_memcpy(&a, words, sizeof(a));
  // device memory, said so: the compiler takes it for granted of pointers in the
  // launch's own arguments only, and would access these with flat instructions (which
  // return out of order, so each wait for one is a wait for every access in flight,
  // the row DMAs included)
  auto dev = [](auto*& q) {
    typedef __typeof__(*q) SAS_GLOBAL* global_p;
    q = (__typeof__(q + 0))(global_p)(uintptr_t)q;
  };
  auto devv = [](const void*& q) { q = (const void*)(const char*)(const char SAS_GLOBAL*)(uintptr_t)q; };
  devv(a.q), devv(a.ori_kv), devv(a.cmp_kv);
  dev(a.ori_block_table), dev(a.cmp_block_table), dev(a.cmp_indices), dev(a.q_prefix);
  dev(a.act_q_lens), dev(a.seqused_kv), dev(a.sinks), dev(a.metadata), dev(a.lse);
  dev(a.workspace), dev(a.merge_sync);
  a.out = (void*)(char*)(char SAS_GLOBAL*)(uintptr_t)a.out;
  return a;
}

__device__ inline ItemGeom item_geom_at(const KernelArgs& a, int act_q, int act_kv, int s) {
  return item_geom_div(act_q, act_kv, s, a.ori_win_left, a.scenario, a.ratio, a.topk);
}

// Positions [c0, c0 + clen) of an item's list -> cache rows in LDS (rowid: row number,
// bit 31 set for the compressed cache, ROW_INVALID for masked positions; tmask: valid
// bits of each 32-row tile), by a workgroup of NT threads; entries past the last tile
// pair are left alone. Two dependent round trips at most (top-k ids, table words),
// each with all its loads in flight; landed() runs when the words have arrived.
//
// Scenario 3 stops at the first -1 among the scanned top-k slots (golden.py:48-53).
// The first chunk's own top-k loads double as the scan of its range; the slots
// outside it are loaded in the same batch, and the table loads are issued before the
// barrier that publishes the result (the cut is applied when the row ids are
// packed). The two first_neg slots alternate between scans, so a slot is reset
// without a barrier of its own.
//
// A short call spends most of its time up to its first row loads on instructions, not
// on memory: a 32-bit division by a number in a register is some 30 of them, 64 bits
// 100. Dividing by multiplication, leaving out positions past the list, forming row
// numbers once and reading arguments per phase (fresh_args) took the way from the
// kernel's entry to its first tile from 15.7 k to 13.2 k clocks (32 x 64-head window
// decode; that kernel 14.8 -> 13.7 us, MLA decode with two rows 110.5 -> 107.6,
// 13 sequences of fp8 rows with fp8 query products 41.5 -> 38.0, 8K prefill with
// top-k 1086 -> 1060).
struct Resolver {
  ItemGeom g;
  const int32_t *ori_tab, *cmp_tab;  // the batch's block-table rows (without a compressed
  int cmp_len;                       // cache the raw one again, whose words are not used)
  const int32_t* idx_row;            // the token's top-k ids, or null
  bool tok_ok;
  int jmax;                          // top-k slots to scan
  bool stop_pending;
  int cmp_stop;

  __device__ Resolver(const KernelArgs& a, const ItemGeom& geom, int b, int tok, bool ok, int p_hi)
      : g(geom), tok_ok(ok) {
    ori_tab = a.ori_block_table + (size_t)b * a.ori_table_len;
    cmp_tab = a.scenario >= 2 ? a.cmp_block_table + (size_t)b * a.cmp_table_len : ori_tab;
    cmp_len = a.scenario >= 2 ? a.cmp_table_len : a.ori_table_len;
    idx_row = a.scenario == 3 && a.cmp_indices && a.topk > 0
                  ? a.cmp_indices + (size_t)(ok ? tok : 0) * a.topk : nullptr;
    jmax = idx_row && p_hi > g.n_win ? min(p_hi - g.n_win, g.n_cmp) : 0;
    stop_pending = jmax > 0;
    cmp_stop = g.n_cmp;
  }

  template <int NT, int RCH, int LOADS, typename Landed>
  __device__ __forceinline__ void chunk(const KernelArgs& a, int c0, int clen, int tid,
                                        uint32_t* rowid, uint32_t* tmask, int* first_neg,
                                        int& item_par, Landed&& landed) {
    constexpr int PER = RCH / NT;              // positions per thread
    constexpr int SCAN_PER = LOADS - PER;      // slots outside the chunk in the first batch
    auto wanted = [&](int e) { return e == 0 || e * NT < clen + 2 * TILE; };  // uniform
    int cid[PER], word[PER], off[PER], sv0[SCAN_PER];
    const int own_lo = max(c0 - g.n_win, 0);
    const int own_hi = min(max(c0 + clen - g.n_win, own_lo), jmax);
    const int n_extra = stop_pending ? jmax - (own_hi - own_lo) : 0;
    auto extra_slot = [&](int x) { return x < own_lo ? x : x + (own_hi - own_lo); };
    if (idx_row) {
      // all loads issued and waited for in one asm statement (gather_dwords_wait)
      const int32_t* src[LOADS];
      int got[LOADS];
#pragma unroll
      for (int e = 0; e < PER; ++e) {
        const int jj = c0 + e * NT + tid - g.n_win;
        src[e] = idx_row + (jj < 0 ? 0 : (jj < a.topk ? jj : a.topk - 1));
      }
#pragma unroll
      for (int e = 0; e < SCAN_PER; ++e) {
        const int x = e * NT + tid;  // clamped into range; unused when n_extra == 0
        const int xc = x < n_extra ? x : (n_extra > 0 ? n_extra - 1 : 0);
        src[PER + e] = idx_row + (n_extra > 0 ? extra_slot(xc) : 0);
      }
      gather_dwords_wait(got, src);
#pragma unroll
      for (int e = 0; e < SCAN_PER; ++e) sv0[e] = got[PER + e];
#pragma unroll
      for (int e = 0; e < PER; ++e) {
        const int r = e * NT + tid;
        cid[e] = (r < clen && tok_ok && c0 + r >= g.n_win) ? got[e] : -1;
      }
    } else {
#pragma unroll
      for (int e = 0; e < PER; ++e) cid[e] = tok_ok ? c0 + e * NT + tid - g.n_win : -1;
    }
    if (stop_pending) {
      int mine = g.n_cmp;
#pragma unroll
      for (int e = 0; e < PER; ++e) {
        const int jj = c0 + e * NT + tid - g.n_win;
        if (jj >= 0 && jj < jmax && e * NT + tid < clen && cid[e] == -1 && jj < mine) mine = jj;
      }
#pragma unroll
      for (int e = 0; e < SCAN_PER; ++e) {
        const int x = e * NT + tid;
        if (x < n_extra && sv0[e] == -1 && extra_slot(x) < mine) mine = extra_slot(x);
      }
      for (int x0 = NT * SCAN_PER; x0 < n_extra; x0 += NT * SCAN_PER) {  // beyond the first round
        int v[SCAN_PER];
#pragma unroll
        for (int e = 0; e < SCAN_PER; ++e) {  // unconditional, clamped: all loads in flight at once
          const int x = x0 + e * NT + tid;
          v[e] = idx_row[extra_slot(x < n_extra ? x : n_extra - 1)];
        }
#pragma unroll
        for (int e = 0; e < SCAN_PER; ++e) {
          const int x = x0 + e * NT + tid;
          if (x < n_extra && v[e] == -1 && extra_slot(x) < mine) mine = extra_slot(x);
        }
      }
      if (mine < g.n_cmp) atomicMin(&first_neg[item_par], mine);
    }
    // block-table words (compiler-visible loads with in-bounds addresses); off: the
    // position's row within its block, -1 when it has none
#pragma unroll
    for (int e = 0; e < PER; ++e) {
      word[e] = off[e] = -1;
      if (!wanted(e)) continue;
      const int r = e * NT + tid;
      const bool win = c0 + r < g.n_win;
      const int key = win ? g.win_lo + c0 + r : cid[e];
      const int tlen = win ? a.ori_table_len : cmp_len;  // >= 1
      const FastDiv bs = {win ? a.ori_bs.mul : a.cmp_bs.mul, win ? a.ori_bs.shift : a.cmp_bs.shift};
      const int bi = key >= 0 ? bs.div(key) : 0;
      word[e] = (win ? ori_tab : cmp_tab)[bi < tlen ? bi : tlen - 1];
      if (r < clen && tok_ok && key >= 0 && bi < tlen && (win || key < g.thr))
        off[e] = key - bi * (win ? a.ori_block_size : a.cmp_block_size);
    }
    // every load so far (table words, query fragment) has landed, as the compiler sees it
    __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0) expcnt(7) lgkmcnt(15)
    landed();
    if (stop_pending) {
      __syncthreads();  // every thread's atomicMin is in
      cmp_stop = min(first_neg[item_par], g.n_cmp);
      if (tid == 0) first_neg[item_par ^ 1] = INT32_MAX;  // the next scan's slot
      item_par ^= 1;
      stop_pending = false;
    }
#pragma unroll
    for (int e = 0; e < PER; ++e) {
      if (!wanted(e)) continue;
      const int r = e * NT + tid;
      const bool win = c0 + r < g.n_win;
      const bool ok = off[e] >= 0 && word[e] >= 0 &&
                      word[e] < (win ? a.ori_block_num : a.cmp_block_num) &&
                      (win || c0 + r - g.n_win < cmp_stop);
      const int row = word[e] * (win ? a.ori_block_size : a.cmp_block_size) + off[e];
      // masked rows are read from the zero row
      rowid[r] = ok ? (uint32_t)row | (win ? 0u : 0x80000000u) : ROW_INVALID;
      const unsigned long long bal = __ballot(ok);
      if ((tid & 63) == 0) {
        tmask[r / TILE] = (uint32_t)bal;
        tmask[r / TILE + 1] = (uint32_t)(bal >> 32);
      }
    }
    __syncthreads();
  }
};

// Rows [0, nh) of a staging area of ROWS rows (SROW bytes apart, 1 KB each) to global
// memory, one row per store instruction: wave w of NW takes rows w, w + NW, ..., a
// batch read from LDS before it is stored. put(h, v): lane's 16 bytes of row h.
template <int ROWS, int NW, int SROW, typename Put>
__device__ __forceinline__ void rows_out(const unsigned char* stg, int nh, int w, int lane,
                                         Put&& put) {
  constexpr int N = ROWS / NW, BATCH = N < 8 ? N : 8;
  static_assert(ROWS % NW == 0 && N % BATCH == 0, "rows per wave");
#pragma unroll
  for (int k0 = 0; k0 < N; k0 += BATCH) {
    i32x4 v[BATCH];
#pragma unroll
    for (int k = 0; k < BATCH; ++k)
      v[k] = *(const i32x4*)(stg + (w + NW * (k0 + k)) * SROW + 16 * lane);
#pragma unroll
    for (int k = 0; k < BATCH; ++k)
      if (w + NW * (k0 + k) < nh) put(w + NW * (k0 + k), v[k]);
  }
}

// Device-built schedules (num_fd == SAS_SCHED_DEVICE): the summary is read from
// the metadata config row; num_fa and num_partial_slots are the launch and
// workspace capacities it must fit.
__device__ inline bool dev_sched_ok(const SasAttnArgs& a, int mb) {
  const int32_t* cfg = a.metadata + SAS_CFG_OFFSET;
  return cfg[0] == SAS_META_MAGIC && cfg[5] == a.num_heads && cfg[6] == mb &&
         cfg[2] >= 1 && cfg[2] <= a.num_fa && cfg[4] <= a.num_partial_slots &&
         cfg[3] >= 0 && cfg[3] <= SAS_AIV_CORE_NUM && cfg[1] >= 32 && cfg[1] % 32 == 0;
}
// An unusable device-built schedule: every output becomes NaN (one workgroup).
template <typename T>
__device__ void nan_fill(const SasAttnArgs& a, int tid, int nthreads) {
  const short qnan = __is_same(T, __bf16) ? (short)0x7FC0 : (short)0x7E00;
  const size_t rows = (size_t)a.total_tokens * a.num_heads;
  short* out = (short*)a.out;
  for (size_t k = tid; k < rows * a.head_dim_v; k += nthreads) out[k] = qnan;
  for (size_t k = tid; k < rows; k += nthreads) a.lse[k] = __builtin_nanf("");
}

// Split-KV partials: per (slot, head) the row acc / l as fp16, times a power-of-two
// scale that puts the row's largest |value| into [2^14, 2^15) (scaled up or
// down), then fp32 lse [slot][head] and fp32 inverse scales [slot][head].
// fp16's 11-bit significand keeps the merged result as close to golden as fp32
// partials do on the reference's input distribution, at half the bytes, and the
// two-sided normalisation keeps that true for rows of any magnitude: small rows
// are not left to fp16's subnormal range.
struct PartialScale {
  float scale, inv;
};
__device__ inline PartialScale partial_scale(float row_max) {
  if (row_max > 0.0f && row_max < INFINITY) {
    // row_max = 1.f * 2^e; e clamped to [-112, 127] so that scale = 2^(14 - e) and
    // inv = 2^(e - 14) are both normal floats (rows below 2^-112 are scaled by 2^126)
    int e = (int)((__float_as_uint(row_max) >> 23) & 0xFF) - 127;
    e = e < -112 ? -112 : e;
    return {__uint_as_float((uint32_t)(127 + 14 - e) << 23),
            __uint_as_float((uint32_t)(127 + e - 14) << 23)};
  }
  return {1.0f, 1.0f};  // an all-zero (or non-finite) row
}
__device__ inline float* partial_lse(const SasAttnArgs& a, int mb, int dv) {
  return (float*)((char*)a.workspace + (size_t)a.num_partial_slots * mb * dv * 2);
}

// ---------------------------------------------------------------------------
// Split-KV merge inside the attention kernel (SasAttnArgs.merge_sync)
// ---------------------------------------------------------------------------
// The pieces of a split item sit in consecutive FA rows and take consecutive
// partial slots in block order (both schedulers number slots in core order).
// A row whose first item starts at a block > 0 continues an item begun in the
// rows before it; its piece index is 1 + the number of rows just before it that
// also start inside that item. Lane l looks at row fa_row - 1 - l (the first 64
// rows; continued_piece_index walks further for items of more pieces).
struct ContScan {
  int b, m, j;  // start cursor of row fa_row - 1 - lane (b = -1: no such row)
};
__device__ inline ContScan cont_scan_load(const SasAttnArgs& a, int fa_row, int lane) {
  const int r = fa_row - 1 - lane;
  if (r < 0) return {-1, 0, 0};
  const int32_t* p = a.metadata + (size_t)r * SAS_FA_METADATA_SIZE;
  return {p[1], p[2], p[3]};
}
__device__ inline int continued_piece_index(const SasAttnArgs& a, int fa_row, int b, int m,
                                            ContScan first) {
  const int lane = threadIdx.x & 63;
  int k = 1;
  ContScan c = first;
  for (int r0 = fa_row - 1;; r0 -= 64) {
    const bool cont = c.b == b && c.m == m && c.j > 0;
    const uint64_t stop = ~(uint64_t)__ballot(cont);
    if (stop != 0) return k + __builtin_ctzll(stop);
    k += 64;
    c = cont_scan_load(a, r0 - 63, lane);  // rows r0 - 64 - lane
  }
}

// Partials that another workgroup merges are written and read with agent-scope
// coherent accesses (sc1: through to the device's coherence point, past the
// per-XCD L2 caches), so the hand-over needs no cache-wide writeback or
// invalidate: a piece waits for its stores to complete, then counts itself in;
// the merging piece reads after it has seen the count.
__device__ inline __amdgpu_buffer_rsrc_t partial_rsrc(const SasAttnArgs& a, int mb, int dv) {
  const int bytes = a.num_partial_slots * mb * (2 * dv + 8);  // the workspace (< 2^31)
  return __builtin_amdgcn_make_buffer_rsrc(a.workspace, 0, bytes, 0x00020000);
}
constexpr int CPOL_SC1 = 16;  // buffer instruction cache policy: agent-scope coherent
__device__ inline void partial_store16(__amdgpu_buffer_rsrc_t r, uint32_t off, i32x4 v) {
  __builtin_amdgcn_raw_buffer_store_b128(v, r, (int)off, 0, CPOL_SC1);
}
__device__ inline void partial_store4(__amdgpu_buffer_rsrc_t r, uint32_t off, float v) {
  __builtin_amdgcn_raw_buffer_store_b32(__float_as_int(v), r, (int)off, 0, CPOL_SC1);
}

// One thread counts a piece of the item in slots slot0, ... in at the item's counter
// merge_sync[slot0]: pieces in the low 32 bits and, from the item's final piece (which
// alone knows it), the piece count in the high ones. Returns the piece count to the
// piece that completes it, 0 to the others, and then the counter is zero again. Pieces
// are counted, not their blocks: every piece of the schedule counts itself in once
// (split_settle), so a counter returns to zero whatever lengths a call finds.
__device__ inline int split_count(const SasAttnArgs& a, int slot0, int slot, bool final_piece) {
  const unsigned long long add =
      1ull | (final_piece ? (unsigned long long)(uint32_t)(slot - slot0 + 1) << 32 : 0ull);
  unsigned long long* c = (unsigned long long*)a.merge_sync + slot0;
  const unsigned long long tot =
      __hip_atomic_fetch_add(c, add, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) + add;
  if ((uint32_t)tot != (uint32_t)(tot >> 32)) return 0;
  __hip_atomic_store(c, 0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  return (int)(tot >> 32);
}
__device__ inline bool split_slots_ok(const SasAttnArgs& a, int slot0, int slot) {
  return slot0 >= 0 && slot < a.num_partial_slots && slot0 < SAS_MERGE_SYNC_WORDS;
}
// Arrival of a piece whose partial every thread of the workgroup has stored (with
// partial_store16 / partial_store4); the piece that gets a count merges the item.
__device__ inline int split_arrive(const SasAttnArgs& a, int slot0, int slot, bool final_piece,
                                   int* lds_word) {
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // this thread's partial stores are done
  __syncthreads();
  if (threadIdx.x == 0) *lds_word = split_count(a, slot0, slot, final_piece);
  __syncthreads();
  return *lds_word;
}
// After a workgroup's items: the pieces of its row whose items the call does not have
// (fewer query rows than scheduled). `slot` is the next piece's; first: the row's first
// piece, which continues an item (cont_k), is not counted in; last: its last is not.
__device__ inline void split_settle(const SasAttnArgs& a, bool first, int cont_k, bool last, int slot) {
  if (threadIdx.x != 0) return;
  if (first) {
    const int k = cont_k < 0 ? -cont_k : cont_k;
    if (split_slots_ok(a, slot - k, slot)) split_count(a, slot - k, slot, cont_k > 0);
    ++slot;
  }
  if (last && split_slots_ok(a, slot, slot)) split_count(a, slot, slot, false);
}

// Merge of split item (token tok, head block hb; pieces in slots slot0 ..
// slot0 + npc - 1) by a workgroup of NW waves: wave w takes heads
// [w * MB / NW, +MB / NW) of the block in groups of G, lane l dims 8 l .. 8 l + 7
// of each; the loads of PB pieces are in flight together. The arithmetic is
// merge_task's (below) operation for operation (o starts at -0, so the first
// fused multiply-add rounds as merge_task's first product), so out and lse are
// bit-identical to the merge kernel's.
template <int DV, typename T, int MB, int NW>
__device__ void merge_item_here(const SasAttnArgs& a, int tok, int hb, int slot0, int npc) {
  constexpr int HPW = MB / NW;
  constexpr int G = HPW < 8 ? HPW : 8;  // heads per group
  constexpr int PB = 2;                 // pieces per batch of loads
  static_assert(DV == 512 && MB % NW == 0 && HPW % G == 0 && HPW <= 64, "merge layout");
  int tid = threadIdx.x;
  asm volatile("" : "+v"(tid));  // (nothing of the merge is formed before its call)
  const int lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int nh = min(MB, a.num_heads - hb * MB);
  const int hw0 = w * HPW;
  if (hw0 >= nh) return;
  const __amdgpu_buffer_rsrc_t rs = partial_rsrc(a, MB, DV);
  const uint32_t lse_off = (uint32_t)a.num_partial_slots * MB * DV * 2;  // bytes
  const uint32_t inv_off = lse_off + (uint32_t)a.num_partial_slots * MB * 4;
  auto ldf = [&](uint32_t off) -> float {
    return __int_as_float(__builtin_amdgcn_raw_buffer_load_b32(rs, (int)off, 0, CPOL_SC1));
  };
  // lse of head hw0 + lane (lanes < HPW; the others repeat head hw0)
  const int hk = hw0 + (lane < HPW && hw0 + lane < nh ? lane : 0);
  const int hq = hb * MB + hk;
  const float sink = a.sinks[hq];
  auto plse = [&](int i) { return ldf(lse_off + ((uint32_t)(slot0 + i) * MB + hk) * 4); };
  auto pinv = [&](int i) { return ldf(inv_off + ((uint32_t)(slot0 + i) * MB + hk) * 4); };
  constexpr int MAXL = 8;
  float lv[MAXL];
#pragma unroll
  for (int i = 0; i < MAXL; ++i) lv[i] = plse(i < npc ? i : npc - 1);
  float mx = fmaxf(sink, lv[0]);
#pragma unroll
  for (int i = 1; i < MAXL; ++i)
    if (i < npc) mx = fmaxf(mx, lv[i]);
  for (int i = MAXL; i < npc; ++i) mx = fmaxf(mx, plse(i));
  float l = -INFINITY;
  if (mx != -INFINITY) {
    float tot = __expf(sink - mx) + __expf(lv[0] - mx);
#pragma unroll
    for (int i = 1; i < MAXL; ++i)
      if (i < npc) tot += __expf(lv[i] - mx);
    for (int i = MAXL; i < npc; ++i) tot += __expf(plse(i) - mx);
    l = mx + __logf(tot);
  }
  // the weights of the wave's heads (lane k: head hw0 + k) for piece i
  auto wlane = [&](int i) -> float {
    const float li = plse(i);  // (lv[i] again: loaded beside the piece's data)
    return ((l == -INFINITY || li == -INFINITY) ? 0.0f : __expf(li - l)) * pinv(i);
  };
  const bool tok_ok = tok >= 0 && tok < a.total_tokens;
  for (int g0 = 0; g0 < HPW; g0 += G) {
    f32x4 o[G][2];
#pragma unroll
    for (int k = 0; k < G; ++k) o[k][0] = o[k][1] = (f32x4){-0.0f, -0.0f, -0.0f, -0.0f};
    for (int i0 = 0; i0 < npc; i0 += PB) {
      i32x4 v[PB][G];
#pragma unroll
      for (int j = 0; j < PB; ++j) {
        const int i = i0 + j < npc ? i0 + j : npc - 1;  // clamped: every load unconditional
#pragma unroll
        for (int k = 0; k < G; ++k) {
          const int h = hw0 + g0 + k < nh ? hw0 + g0 + k : nh - 1;
          const uint32_t off = (((uint32_t)(slot0 + i) * MB + h) * DV + 8 * lane) * 2;
          v[j][k] = __builtin_amdgcn_raw_buffer_load_b128(rs, (int)off, 0, CPOL_SC1);
        }
      }
      float wj[PB];
#pragma unroll
      for (int j = 0; j < PB; ++j) wj[j] = wlane(i0 + j < npc ? i0 + j : npc - 1);
      __builtin_amdgcn_sched_barrier(0);  // every load of the batch issued before the first use
#pragma unroll
      for (int j = 0; j < PB; ++j) {
        if (i0 + j >= npc) break;
#pragma unroll
        for (int k = 0; k < G; ++k) {
          const float wk = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(wj[j]), g0 + k));
          typedef _Float16 h16x8 __attribute__((ext_vector_type(8)));
          const h16x8 x = __builtin_bit_cast(h16x8, v[j][k]);
#pragma unroll
          for (int e = 0; e < 8; ++e)
            o[k][e >> 2][e & 3] = __builtin_fmaf(wk, (float)x[e], o[k][e >> 2][e & 3]);
        }
      }
    }
    if (tok_ok) {
#pragma unroll
      for (int k = 0; k < G; ++k) {
        if (hw0 + g0 + k >= nh) break;
        T* orow = (T*)a.out + ((size_t)tok * a.num_heads + hb * MB + hw0 + g0 + k) * DV + 8 * lane;
        const i16x8 pk = {MfmaOps<T>::from_f32(o[k][0][0]), MfmaOps<T>::from_f32(o[k][0][1]),
                          MfmaOps<T>::from_f32(o[k][0][2]), MfmaOps<T>::from_f32(o[k][0][3]),
                          MfmaOps<T>::from_f32(o[k][1][0]), MfmaOps<T>::from_f32(o[k][1][1]),
                          MfmaOps<T>::from_f32(o[k][1][2]), MfmaOps<T>::from_f32(o[k][1][3])};
        *(i16x8*)orow = pk;
      }
    }
  }
  if (tok_ok && lane < HPW && hw0 + lane < nh) a.lse[(size_t)tok * a.num_heads + hq] = l;
}

// fp8 cache rows (SAS_KV_FP8_DS_MLA): eight e4m3 values (one 8-byte word) times
// their block scale, each product rounded to bf16 (v_cvt_pk_f32_fp8 decodes OCP
// e4m3 exactly; v_mul_f32 and v_cvt_pk_bf16_f32 round to nearest even).
__device__ inline i16x8 fp8x8_dequant_bf16(uint2 v, float s) {
  typedef float f32x2 __attribute__((ext_vector_type(2)));
  typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
  const f32x2 f0 = __builtin_amdgcn_cvt_pk_f32_fp8(v.x, false);
  const f32x2 f1 = __builtin_amdgcn_cvt_pk_f32_fp8(v.x, true);
  const f32x2 f2 = __builtin_amdgcn_cvt_pk_f32_fp8(v.y, false);
  const f32x2 f3 = __builtin_amdgcn_cvt_pk_f32_fp8(v.y, true);
  const bf16x2 b0 = __builtin_convertvector((f32x2){f0[0] * s, f0[1] * s}, bf16x2);
  const bf16x2 b1 = __builtin_convertvector((f32x2){f1[0] * s, f1[1] * s}, bf16x2);
  const bf16x2 b2 = __builtin_convertvector((f32x2){f2[0] * s, f2[1] * s}, bf16x2);
  const bf16x2 b3 = __builtin_convertvector((f32x2){f3[0] * s, f3[1] * s}, bf16x2);
  typedef short s2 __attribute__((ext_vector_type(2)));
  const s2 w0 = __builtin_bit_cast(s2, b0), w1 = __builtin_bit_cast(s2, b1);
  const s2 w2 = __builtin_bit_cast(s2, b2), w3 = __builtin_bit_cast(s2, b3);
  return (i16x8){w0[0], w0[1], w1[0], w1[1], w2[0], w2[1], w3[0], w3[1]};
}

// fp8 Q·Kᵀ: a head's 512 latent query dims as e4m3 codes of q * (448 / amax)
// (one IEEE fp32 division per head, then an fp32 product per dim, clamped to ±448
// and rounded to nearest even by v_cvt_pk_fp8_f32), with sq = amax / 448 the
// factor that scales the scores back (both 1 for an all-zero head). The lane holds dims
// 128 blk + 32 g4 + 8 h + e of its head in qf[4 blk + h][e] (bf16 bits); the
// head's other dims sit in lanes l ^ 16, l ^ 32, l ^ 48. q8[blk] is the 16x16x128
// B operand of block blk: byte p = dim 128 blk + 32 g4 + p.
__device__ inline void quantize_q(const i16x8 (&qf)[18], i32x8 (&q8)[4], float& sq) {
  auto f32 = [](short v) { return __uint_as_float((uint32_t)(uint16_t)v << 16); };
  // amax on the bf16 bits (|x| orders as its low 15 bits), one k-step at a time:
  // fp32 conversions here would be kept for the quantization below, and the
  // scheduler would convert every dim at once, more than the registers of the
  // loop around this can hold
  typedef unsigned short u16x2 __attribute__((ext_vector_type(2)));
  u16x2 mb = {0, 0};
#pragma unroll
  for (int ks = 0; ks < 16; ++ks) {
    const i32x4 wv = __builtin_bit_cast(i32x4, qf[ks]);
#pragma unroll
    for (int e = 0; e < 4; ++e)
      mb = __builtin_elementwise_max(mb, __builtin_bit_cast(u16x2, wv[e] & 0x7FFF7FFF));
    __builtin_amdgcn_sched_barrier(0);
  }
  float amax = __uint_as_float((uint32_t)(mb[0] > mb[1] ? mb[0] : mb[1]) << 16);
  const auto r1 = __builtin_amdgcn_permlane16_swap(__float_as_uint(amax), __float_as_uint(amax),
                                                   false, false);
  amax = wave_max_pair(fmaxf(__uint_as_float(r1[0]), __uint_as_float(r1[1])));
  sq = amax > 0.0f ? amax / 448.0f : 1.0f;
  const float inv = amax > 0.0f ? 448.0f / amax : 1.0f;
#pragma unroll
  for (int blk = 0; blk < 4; ++blk)
#pragma unroll
    for (int d = 0; d < 8; ++d) {
      const i16x8 v = qf[4 * blk + (d >> 1)];
      float y[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) y[i] = fminf(fmaxf(f32(v[4 * (d & 1) + i]) * inv, -448.0f), 448.0f);
      int w = __builtin_amdgcn_cvt_pk_fp8_f32(y[0], y[1], 0, false);
      w = __builtin_amdgcn_cvt_pk_fp8_f32(y[2], y[3], w, true);
      q8[blk][d] = w;
      __builtin_amdgcn_sched_barrier(0);  // (one word at a time, as above)
    }
}

// ---------------------------------------------------------------------------
// Attention kernel, dims-split form (native bf16 / fp16 rows)
// ---------------------------------------------------------------------------
// Waves: NHG head groups of 32 heads x 2 halves of d_qk / d_v = 2*NHG waves,
// one per SIMD. Wave w -> head group hg = w % NHG, half dh = w / NHG; its
// partner (same heads, other half) is w ^ NHG.
//   Q·Kᵀ: partial Sᵀ[32 rows x 32 heads] over dims half dh (main dims
//         256dh..256dh+255 and, for d_qk 576, rope dims 512+32dh..+31), with
//         v_mfma_f32_32x32x16 (A = K rows from LDS, B = Qᵀ in VGPRs);
//   exchange: the two partials of a head group meet through LDS; each wave
//         adds the other's to its own (fp32 addition is commutative, so both
//         hold the identical Sᵀ and take identical softmax decisions);
//   softmax: two tiles (64 rows) per step, 32 rows x 1 head per lane, exp2
//         domain. A head's running max moves at every step whose max exceeds
//         it (golden.py:187-191's rule at 64-row tiles), so the largest score
//         seen so far has P = 1 exactly when P is rounded to the input type
//         (golden.py:192-196); the accumulator rescale is paid once per step;
//   P·V:  Oᵀ[dv half dh (256) x 32 heads] += Vᵀ·Pᵀ. Pᵀ is taken straight from
//         the Sᵀ registers: the accumulator holds rows 8(i/4) + 4(lane/32) +
//         i%4 in element i, which is the B-operand order of the Vᵀ reads
//         (k-step kq = elements 8kq..8kq+7).
// Per step (tiles a, b): barrier 1a (b landed, partials of a written), barrier
// 1b (partials of b written), barrier X (stage a free) and barrier 2 (stage b
// free, a + 2 landed). Ring of 3 stages: tile a + 2 is issued under the Q·Kᵀ
// of a into the stage tile a - 1 left, a + 3 under the P·V of b into stage a.
// Native rows only: fp8 rows run on attn3_kernel.
// PREF: launches whose batches hold several query rows (prefill, MTP); then a
// workgroup's consecutive items of one batch load the next item's query
// fragment during the current item's epilogue. Decode launches keep the
// simpler first-chunk load (measured faster for their short items).
template <int DQK, int DV, int NHG, typename T, int KVF, bool PREF>
__global__ __launch_bounds__(128 * NHG) void attn2_kernel(const KernelArgs a) {
  constexpr int NW = 2 * NHG;            // waves per workgroup
  constexpr int MB = 32 * NHG;           // heads per item (m-block)
  constexpr int NT = 64 * NW;            // threads
  constexpr bool ROPE = DQK == 576;      // 64 extra rope dims after the 512 main dims
  constexpr int ROWB = DQK * 2;          // bytes per cache row in HBM
  constexpr int NKS_MAIN = 16;           // k-steps over the 256 main dims of a half
  constexpr int NKS = NKS_MAIN + (ROPE ? 2 : 0);
  constexpr int DVB = DV / 2 / 32;       // 32-wide dv blocks per wave (8)
  constexpr int NSTG = 3;                // LDS ring depth
  constexpr int STAGE_BYTES = MAIN_BYTES + (ROPE ? ROPE_BYTES : 0);
  constexpr int ROWS_PER_WAVE = TILE / NW;             // main-part DMA instructions per wave
  constexpr int NROPE = ROPE ? TILE / 8 : 0;           // rope DMA instructions per tile
  constexpr int ROPE_PER_WAVE = NROPE / NW;            // 1 or 2 (0 for d_qk 512)
  constexpr int DMA_PER_TILE = ROWS_PER_WAVE + ROPE_PER_WAVE;  // this wave's per tile
  constexpr int RCH = 4 * NT;            // positions resolved into LDS at a time
  static_assert(DQK == 512 || DQK == 576, "head_dim");
  static_assert(DV == 512, "head_dim_v");
  static_assert((STAGE_BYTES % 1024) == 0, "stage alignment");
  static_assert(TILE % NW == 0 && NROPE % NW == 0, "DMA split");
  static_assert(DMA_PER_TILE <= 63, "vmcnt range");
  static_assert(KVF == SAS_KV_NATIVE, "native rows only (fp8 rows run on attn3_kernel)");
  typedef MfmaOps<T> Ops;

  __shared__ __attribute__((aligned(1024))) unsigned char kv_lds[NSTG * STAGE_BYTES];
  __shared__ __attribute__((aligned(16))) f32x4 xbuf[2][NW][4][64];  // partial Sᵀ of each wave, per tile of a pair
  __shared__ uint32_t rowid[RCH];
  __shared__ uint32_t tmask[RCH / TILE];
  __shared__ int merge_word;    // split_arrive's answer to the workgroup
  __shared__ int first_neg[2];  // first -1 of the top-k scan (the slots alternate between scans)

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int hg = w % NHG;
  const int dh = w / NHG;
  const int partner = w ^ NHG;
  const int hlocal = hg * 32 + (lane & 31);  // head within the item's m-block
  const int hblocks = (a.num_heads + MB - 1) / MB;  // 1 or 2 (the launch's check of m_base)
  const int hshift = hblocks - 1;
  const int hl = lane >> 5;
  // Kᵀ operand: row lane%32, main chunk 32dh + 2ks + hl (dims 256dh + 16ks + 8hl),
  // rope chunk 4dh + 2(ks - 16) + hl
  const int r_qk = lane & 31;
  const int qk_base = main_row_base(r_qk) + (32 * dh + hl) * 16;
  const int rope_off0 = MAIN_BYTES + rope_slot(r_qk, 4 * dh + hl) * 16;
  const int rope_off1 = MAIN_BYTES + rope_slot(r_qk, 4 * dh + 2 + hl) * 16;
  // Vᵀ operand (ds_read_b64_tr_b16): 16-lane group (lane>>4) reads rows
  // 4*hl + (lane&15)/4 (+16kq, +8) at dv 256dh + 16*((lane>>4)&1) + 4*(lane&3) (+32d).
  // Row r+16 has the same rotation as r; row r+8 (r%8 < 4) has rotation +2.
  const int tr_base = main_row_base(4 * hl + ((lane & 15) >> 2)) + dh * DV +
                      ((lane >> 4) & 1) * 32 + (lane & 3) * 8;

  // With at most 64 batches, every batch's lengths and query offset sit in one
  // lane each, loaded at the start beside the metadata row (they no longer wait
  // for it: the item's batch picks its lane).
  const QRows qrows(a);
  const bool lens_in_lanes = a.batch <= 64;
  int lane_aq = 0, lane_kv = 0, lane_qp = 0;
  if (lens_in_lanes) {
    const int lb = lane < a.batch ? lane : a.batch - 1;
    lane_aq = qrows.rows[lb];
    lane_kv = a.seqused_kv[lb];
    lane_qp = qrows.first[lb];
  }
  int s2b = a.s2_base;
  int nfa = a.num_fa;
  if (a.num_fd == SAS_SCHED_DEVICE) {
    if (!dev_sched_ok(a, MB)) {
      if (blockIdx.x == 0) nan_fill<T>(a, tid, NT);
      return;
    }
    s2b = a.metadata[SAS_CFG_OFFSET + 1];
    nfa = a.metadata[SAS_CFG_OFFSET + 2];  // rows in use (the grid is sized for num_fa)
  }
  // XCD-aware row mapping: consecutive FA rows (pieces of one item) share an XCD.
  const int per_xcd = (nfa + 7) >> 3;
  const int fa_row = (int)(blockIdx.x & 7) * per_xcd + (int)(blockIdx.x >> 3);
  if (fa_row >= nfa || (int)(blockIdx.x >> 3) >= per_xcd) return;
  const int32_t* fa = a.metadata + fa_row * SAS_FA_METADATA_SIZE;
  if (fa[0] == 0) return;
  // where the whole schedule ends (loaded beside this row's cursors)
  const int32_t* fa_last = a.metadata + (nfa - 1) * SAS_FA_METADATA_SIZE;
  int last_on = fa_last[0], last_b = fa_last[4], last_m = fa_last[5];
  int b = fa[1], m = fa[2];
  const int j_start = fa[3];
  const int b_end = fa[4], s_end = fa[5], j_end = fa[6];
  int slot = fa[7];
  const uint32_t kv_base = (uint32_t)(uintptr_t)kv_lds;
  // in-kernel merge: the start cursors of the rows before this one, when its
  // first item continues a split item (loaded beside the lengths)
  const bool merge_here = a.merge_sync != nullptr && a.workspace != nullptr;
  ContScan cscan = {-1, 0, 0};
  if (merge_here && j_start > 0) cscan = cont_scan_load(a, fa_row, lane);

  const char* ori_kv = (const char*)a.ori_kv;
  const char* cmp_kv = (const char*)(a.cmp_kv ? a.cmp_kv : a.ori_kv);
  const float sc = a.softmax_scale * LOG2E;
  if (tid < 2) first_neg[tid] = INT32_MAX;
  // piece index of the first item when it continues a split item, negative when the
  // item goes on in the next row (by the schedule, whatever the lengths are by now);
  // last_owed: the row's last piece, of an item that begins here, is not counted in
  int cont_k = 0;
  bool last_owed = merge_here && j_end > 0;
  if (merge_here && j_start > 0) {
    cont_k = continued_piece_index(a, fa_row, b, m, cscan);
    if (j_end > 0 && b == b_end && m == s_end) {
      cont_k = -cont_k;
      last_owed = false;
    }
  }
  __syncthreads();

  // Sinks of this lane's head in the (at most two) head blocks of an item,
  // loaded once: a load per item would also wait for the previous item's output
  // stores (one in-order counter covers loads and stores). They are first read
  // after the first item's resolution has waited for its loads, so their
  // latency is not on the start-up chain.
  const float sink_hb0 = hlocal < a.num_heads ? a.sinks[hlocal] : -INFINITY;
  const float sink_hb1 = MB + hlocal < a.num_heads ? a.sinks[MB + hlocal] : -INFINITY;
  // the lane-held lengths are waited for here, once: read first inside the item
  // loop, whose later iterations have output stores and query loads in flight,
  // they would make the head of every item wait for those
  lane_aq = qrows.count(lane_aq, lane_qp);
  lane_qp = qrows.start(lane, lane_qp);
  asm volatile("" : "+v"(lane_aq), "+v"(lane_kv), "+v"(lane_qp));
  // cumulative row counts: the tokens [tok_lo, tok_hi) of the schedule's rows
  int tok_lo = 0, tok_hi = a.total_tokens;
  if (qrows.cumulative) {
    while (last_on == 0) {  // (a row out of use: the last one before it, at most this one)
      fa_last -= SAS_FA_METADATA_SIZE;
      last_on = fa_last[0], last_b = fa_last[4], last_m = fa_last[5];
    }
    tok_lo = ld_uniform(qrows.first);
    const bool inside = last_b < a.batch;
    tok_hi = ld_uniform(qrows.first + (last_b < 0 ? 0 : (inside ? last_b : a.batch))) +
             (inside ? last_m >> hshift : 0);
  }
  int item_par = 0;  // which first_neg slot the next top-k scan uses
  bool first_item = true;
  // query fragment of this wave's dims half (B operand of Sᵀ = K·Qᵀ); the next
  // item's is loaded into it during the current item's last step (q_pref)
  i16x8 qf[NKS];
  bool q_pref = false;
  // a batch's lengths and query offset: from the lanes (at most 64 batches) or
  // by scalar loads, issued together (the index is clamped)
  auto batch_lens = [&](int bb, int& aq, int& akv, int& qp) {
    const int bc = bb < a.batch ? bb : a.batch - 1;
    if (lens_in_lanes) {
      aq = __builtin_amdgcn_readlane(lane_aq, bc);
      akv = __builtin_amdgcn_readlane(lane_kv, bc);
      qp = __builtin_amdgcn_readlane(lane_qp, bc);
    } else {
      const int first_b = ld_uniform(qrows.first + bc);
      aq = qrows.count(ld_uniform(qrows.rows + bc), first_b);
      akv = ld_uniform(a.seqused_kv + bc);
      qp = qrows.start(bc, first_b);
    }
  };
  // this wave's query fragment of (token, head); rows out of range read token 0's
  // first head: their scores only reach their own softmax column, never stored (and
  // nothing here waits for the loads)
  auto load_q = [&](int qtok, int qhead) {
    const bool ok = qtok >= 0 && qtok < a.total_tokens && qhead < a.num_heads;
    const short* qrow = (const short*)a.q + ((size_t)(ok ? qtok : 0) * a.num_heads +
                                             (ok ? qhead : 0)) * DQK;
#pragma unroll
    for (int ks = 0; ks < NKS; ++ks) {
      const int dim = ks < NKS_MAIN ? (256 * dh + 16 * ks + 8 * hl)
                                    : (512 + 32 * dh + 16 * (ks - NKS_MAIN) + 8 * hl);
      qf[ks] = *(const i16x8*)(qrow + dim);
    }
  };
  for (;;) {
    const KernelArgs a = fresh_args();
    const bool have_q = PREF && q_pref;
    q_pref = false;
    b = __builtin_amdgcn_readfirstlane(b);
    m = __builtin_amdgcn_readfirstlane(m);
    int act_q, act_kv, qpre;
    batch_lens(b, act_q, act_kv, qpre);
    // normalise the cursor: skip batches with no (more) query rows
    while (b < a.batch && b <= b_end && m >= act_q * hblocks) {
      ++b;
      m = 0;
      batch_lens(b, act_q, act_kv, qpre);
    }
    if (b >= a.batch || b > b_end || (b == b_end && m > s_end)) break;
    const bool is_end = (b == b_end && m == s_end);
    const int s = m >> hshift;
    const int head = (m - s * hblocks) * MB + hlocal;
    const bool head_ok = head < a.num_heads;
    if (is_end && j_end == 0) break;

    const int tok = qpre + s;
    const ItemGeom g = item_geom_at(a, act_q, act_kv, s);
    const int L = g.n_win + g.n_cmp;
    const bool partial = (first_item && j_start > 0) || is_end;
    const int blo = first_item ? j_start : 0;
    const int p_lo = blo * s2b;
    const int p_hi = is_end && (int64_t)j_end * s2b < L ? j_end * s2b : L;
    const bool tok_ok = tok >= 0 && tok < a.total_tokens;

    // ---- online-softmax state (golden.py:156-160 seeds m = sink, l = 1; the 1
    // goes to the lanes of the lower row half, whose row sums are added to the
    // upper half's at the end) ----
    const int hb = m - s * hblocks;
    // the next item of this workgroup, if it is the next query row or head block
    // of the same batch: its query fragment is loaded into qf once this item's
    // last Q·Kᵀ has read qf
    auto prefetch_next_q = [&]() -> bool {
      if (is_end) return false;
      int nb = b, nm = m + 1, aq, akv, qp;
      batch_lens(nb, aq, akv, qp);
      while (nb < a.batch && nb <= b_end && nm >= aq * hblocks) {
        ++nb;
        nm = 0;
        batch_lens(nb, aq, akv, qp);
      }
      if (nb >= a.batch || nb > b_end || (nb == b_end && nm > s_end)) return false;
      if (nb == b_end && nm == s_end && j_end == 0) return false;
      // only within a batch (prefill-like runs of query rows): for decode items of
      // other batches the early loads delayed this item's output stores by more
      // than they saved (SWA decode +4 %, A/B)
      if (nb != b) return false;
      const int ns = nm >> hshift;
      load_q(qp + ns, (nm - ns * hblocks) * MB + hlocal);
      return true;
    };
    // the sink seeds m_run once the item's first loads have been waited for
    auto seed_m = [&]() -> float {
      const float sink_v = hb == 0 ? sink_hb0 : sink_hb1;
      return partial ? -INFINITY : (head_ok ? sink_v * LOG2E : -INFINITY);
    };
    float m_run = -INFINITY;
    float l_part = (partial || hl != 0) ? 0.0f : 1.0f;
    f32x16 acc[DVB];
#pragma unroll
    for (int d = 0; d < DVB; ++d)
#pragma unroll
      for (int j = 0; j < 16; ++j) acc[d][j] = 0.0f;

    Resolver res(a, g, b, tok, tok_ok, p_hi);
    for (int c0 = p_lo; c0 < p_hi; c0 += RCH) {
      const int clen = (p_hi - c0) < RCH ? (p_hi - c0) : RCH;
      const int ntile = (clen + TILE - 1) / TILE;
      // query fragment of the item (first chunk, unless the previous item's last
      // step loaded it): compiler-visible loads issued before the resolution's
      // loads, so they land during its memory round trips; the compiler's wait
      // for the table words below covers them
      if (c0 == p_lo && !have_q) load_q(tok, head);
      // ---- positions -> cache rows (bit 31: compressed cache) ----
      res.template chunk<NT, RCH, 8>(a, c0, clen, tid, rowid, tmask, first_neg, item_par, [&] {
        if (c0 == p_lo) m_run = seed_m();
      });

      // ---- DMA issue for one tile into one ring stage ----
      // main part: wave w fills rows w, w + NW, ...; one 1 KB row per instruction
      // rope part: instruction i (wave i % NW) fills rows 8i..8i+7 (8 lanes per row)
      auto row_ptr = [&](uint32_t id) -> const char* {
        const char* base = (id & 0x80000000u) ? cmp_kv : ori_kv;
        const char* p = base + (size_t)(id & 0x7FFFFFFFu) * ROWB;
        return id == ROW_INVALID ? (const char*)g_zero_row : p;
      };
      auto lane_row = [&](uint64_t ptrs, int j) -> const char* {
        const uint32_t lo = __builtin_amdgcn_readlane((uint32_t)ptrs, j);
        const uint32_t hi = __builtin_amdgcn_readlane((uint32_t)(ptrs >> 32), j);
        return (const char*)(uintptr_t)(((uint64_t)hi << 32) | lo);
      };
      // The DMAs of one tile, as DMA_PER_TILE instructions per wave: the row
      // addresses are gathered first (dma_addrs), then instruction j goes out
      // with dma_one(j), so the instructions can be spread between MFMAs (a wave
      // that issues many back to back stalls on the memory pipeline).
      struct DmaAddrs {
        uint64_t main;                      // lane j < ROWS_PER_WAVE: this wave's j-th main row
        const char* rope[ROPE ? ROPE_PER_WAVE : 1];  // per lane: its 16-byte rope piece
        uint32_t sbase;
      };
      auto dma_addrs = [&](int tile) -> DmaAddrs {
        DmaAddrs d;
        d.sbase = kv_base + (tile % NSTG) * STAGE_BYTES;
        d.main = (uint64_t)(uintptr_t)row_ptr(
            rowid[tile * TILE + w + NW * (lane < ROWS_PER_WAVE ? lane : 0)]);
        if constexpr (ROPE) {
#pragma unroll
          for (int k = 0; k < ROPE_PER_WAVE; ++k) {
            const int i = w + NW * k;  // rope instruction: rows 8i..8i+7
            const int r = 8 * i + (lane >> 3);
            const int cr = ((lane & 7) - (r >> 1)) & 7;
            d.rope[k] = row_ptr(rowid[tile * TILE + r]) + 1024 + cr * 16;
          }
        }
        return d;
      };
      auto dma_one = [&](const DmaAddrs& d, int j) {
        if (j < ROWS_PER_WAVE) {
          const int r = w + NW * j;
          dma16_sbase(lane_row(d.main, j), (uint32_t)lane * 16u, d.sbase + main_row_base(r));
        } else if constexpr (ROPE) {
          const int k = j - ROWS_PER_WAVE;
          dma16_vaddr(d.rope[k], d.sbase + MAIN_BYTES + (w + NW * k) * 1024);
        }
      };
      auto issue = [&](int tile) {
        const DmaAddrs d = dma_addrs(tile);
#pragma unroll
        for (int j = 0; j < DMA_PER_TILE; ++j) dma_one(d, j);
      };

      // ---- prologue: tiles 0 and 1 into stages 0 and 1 (tile 1 reads the zero
      // row when the chunk has a single tile: its rows are masked) ----
      issue(0);
      issue(1);
      // tile 0 has landed (tile 1's DMAs may be in flight; the query fragment and
      // the table words were waited for during the resolution)
      wait_vmcnt<DMA_PER_TILE>();
      // the query fragment lives in AGPRs (the MFMAs read B operands from them
      // directly), leaving the VGPRs to the accumulators and prefetch buffers
#pragma unroll
      for (int ks = 0; ks < NKS; ++ks) asm volatile("" : "+a"(qf[ks]));
      __syncthreads();

      // Addresses of the DMAs of tile t (t >= 2), gathered ahead of their issue.
      // Branch-free past the chunk's last tile: those instructions read the zero
      // row into the stage they would fill, which nothing reads before the chunk ends.
      auto next_addrs = [&](int tile) -> DmaAddrs {
        const bool real = tile < ntile;
        DmaAddrs d = dma_addrs(real ? tile : 0);
        d.sbase = kv_base + (tile % NSTG) * STAGE_BYTES;
        if (!real) {
          d.main = (uint64_t)(uintptr_t)g_zero_row;
#pragma unroll
          for (int k = 0; k < (ROPE ? ROPE_PER_WAVE : 1); ++k) d.rope[k] = (const char*)g_zero_row;
        }
        return d;
      };
      typedef const unsigned char SAS_LDS* lds_p;
      auto stage = [&](int tile) -> lds_p {
        return (lds_p)(kv_base + (uint32_t)((tile % NSTG) * STAGE_BYTES));
      };

      // ---- partial Sᵀ of one tile over this wave's dims half ----
      // K operands read KPF k-steps ahead (enough LDS reads in flight for one wave
      // per SIMD to keep the LDS busy); with DMA, the instructions of `dd` go out
      // between the MFMAs (instruction j after MFMA j * NKS / DMA_PER_TILE)
      auto qk_tile = [&](lds_p sb, const DmaAddrs& dd, auto with_dma, auto&& extra) -> f32x16 {
        constexpr int KPF = SAS_KPF;
        const lds_p kb = sb + qk_base;
        auto kaddr = [&](int ks) -> const i16x8 SAS_LDS* {
          return (const i16x8 SAS_LDS*)(ks < NKS_MAIN
                                            ? kb + 32 * ks
                                            : sb + (ks == NKS_MAIN ? rope_off0 : rope_off1));
        };
        i16x8 kbuf[KPF];
#pragma unroll
        for (int i = 0; i < KPF; ++i) kbuf[i] = *kaddr(i);
        // two accumulator chains (even / odd k-steps): an MFMA that reads the
        // previous one's result waits for it to drain (about 58 instead of 32
        // cycles per 32x32x16 MFMA, measured)
        f32x16 s2[2];
#pragma unroll
        for (int j = 0; j < 16; ++j) s2[0][j] = s2[1][j] = 0.0f;
        // (scheduling fences keep each read KPF MFMAs ahead of its use; left
        // alone, the scheduler sinks the reads next to their MFMAs)
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int ks = 0; ks < NKS; ++ks) {
          const i16x8 kop = kbuf[ks % KPF];
          if (ks + KPF < NKS) kbuf[ks % KPF] = *kaddr(ks + KPF);
          s2[ks & 1] = Ops::mma(kop, qf[ks], s2[ks & 1]);
          if (ks == 4) extra();  // VALU work of the caller, under the MFMAs
          if constexpr (decltype(with_dma)::value) {
#pragma unroll
            for (int j = 0; j < DMA_PER_TILE; ++j)
              if ((j * NKS) / DMA_PER_TILE == ks) dma_one(dd, j);
          }
          __builtin_amdgcn_sched_barrier(0);
        }
        f32x16 st;
#pragma unroll
        for (int j = 0; j < 16; ++j) st[j] = s2[0][j] + s2[1][j];
        return st;
      };

      // ---- Oᵀ (+)= Vᵀ·Pᵀ of one tile over both 16-row k-steps ----
      // (Vᵀ operands read VPF MFMAs ahead; MFMA i = dv block i / 2, k-step i % 2;
      // with the rescale, each accumulator block is multiplied just before its
      // first MFMA; with DMA, instruction j of `dd` goes out after MFMA
      // j * NPV / DMA_PER_TILE)
      constexpr int VPF = SAS_VPF;
      struct VBuf { i16x8 v[VPF]; };
      // Vᵀ operand of MFMA i of a tile (spread order: all first k-steps, then all
      // second ones)
      auto vop = [&](lds_p sb, bool spread, int i) -> i16x8 {
        const lds_p vb = sb + tr_base;
        typedef i16x4 SAS_LDS* lds4;
        const int d = spread ? i % DVB : i >> 1, kq = spread ? i / DVB : i & 1;
        const i16x4 g0 = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
            (lds4)(vb + (16 * kq) * MAIN_ROW_BYTES + d * 64));
        const i16x4 g1 = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
            (lds4)(vb + (16 * kq + 8) * MAIN_ROW_BYTES + 32 + d * 64));
        return (i16x8){g0[0], g0[1], g0[2], g0[3], g1[0], g1[1], g1[2], g1[3]};
      };
      // the first VPF operands, read ahead of the tile's P·V (under other work)
      auto pv_pre = [&](lds_p sb, auto rescale) -> VBuf {
        constexpr bool SPREAD = SAS_PV_SPREAD || !decltype(rescale)::value;
        VBuf vb;
#pragma unroll
        for (int i = 0; i < VPF; ++i) vb.v[i] = vop(sb, SPREAD, i);
        return vb;
      };
      auto pv_tile = [&](lds_p sb, VBuf vbf, const i16x8 (&pkt)[2], float alpha, const DmaAddrs& dd,
                         auto rescale, auto with_dma) {
        constexpr int NPV = 2 * DVB;
        i16x8 (&vbuf)[VPF] = vbf.v;
        // (no scheduling fences here: the compiler's own interleaving of the
        // rescale multiplies with the MFMAs measured faster than fenced orders)
        // MFMA order: with SAS_PV_SPREAD (or without the rescale) all first k-steps,
        // then all second ones, so an accumulator's two MFMAs are DVB apart
        constexpr bool SPREAD = SAS_PV_SPREAD || !decltype(rescale)::value;
        auto vdk = [&](int i, int& d, int& kq) {
          if (SPREAD) { d = i % DVB; kq = i / DVB; } else { d = i >> 1; kq = i & 1; }
        };
#pragma unroll
        for (int i = 0; i < NPV; ++i) {
          int d, kq;
          vdk(i, d, kq);
          if constexpr (decltype(rescale)::value) {
            if (kq == 0) {
#pragma unroll
              for (int j = 0; j < 16; ++j) acc[d][j] *= alpha;
            }
          }
          const i16x8 aop = vbuf[i % VPF];
          if (i + VPF < NPV) vbuf[i % VPF] = vop(sb, SPREAD, i + VPF);
          acc[d] = Ops::mma(aop, pkt[kq], acc[d]);
          if constexpr (decltype(with_dma)::value) {
#pragma unroll
            for (int j = 0; j < DMA_PER_TILE; ++j)
              if ((j * NPV) / DMA_PER_TILE == i) dma_one(dd, j);
          }
        }
      };

      // Two tiles (64 rows) per softmax step, so the accumulator rescale and the
      // running-max bookkeeping are paid once per 64 rows (golden.py:187-191's
      // rule at 64-row tiles). Pair p = tiles a = 2p, b = 2p + 1 of the chunk (a
      // trailing odd tile pairs with a masked zero-row tile); the 3-stage ring
      // holds a, b and tile a + 2:
      //   Q·Kᵀ(a), DMAs of tile a + 2 between its MFMAs (into the stage tile
      //     a - 1 left); partial of a to LDS; wait for this wave's DMAs of b;
      //   barrier 1a (b in LDS);  Q·Kᵀ(b); partial of b to LDS;
      //   barrier 1b (both partials written);  softmax over the 64 rows;
      //   P·V(a) with the rescale;  barrier X (stage a free);
      //   P·V(b), DMAs of tile a + 3 between its MFMAs (into stage a);
      //   wait for this wave's DMAs of a + 2;  barrier 2 (stage b free, a + 2 in LDS).
      const int npair = (ntile + 1) >> 1;
      const bool last_chunk = c0 + RCH >= p_hi;
      DmaAddrs nd = next_addrs(2);
      for (int pp = 0; pp < npair; ++pp) {
        const int ta = 2 * pp;
        const lds_p sa = stage(ta);
        const lds_p sbt = stage(ta + 1);

        const f32x16 st0 = qk_tile(sa, nd, std::true_type{}, [] {});
#pragma unroll
        for (int j = 0; j < 4; ++j)
          xbuf[0][w][j][lane] = (f32x4){st0[4 * j], st0[4 * j + 1], st0[4 * j + 2], st0[4 * j + 3]};
        wait_vmcnt<DMA_PER_TILE>();  // this wave's share of tile b (a + 2's may be in flight)
        __syncthreads();             // barrier 1a: tile b in LDS, partials of a written
        // ---- full Sᵀ = own + partner's (the same float sums on both waves); tile
        // a's sums are formed under the Q·Kᵀ MFMAs of tile b ----
        float sv[32];
        f32x4 oa[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) oa[j] = xbuf[0][partner][j][lane];
        const f32x16 st1 = qk_tile(sbt, nd, std::false_type{}, [&] {
#pragma unroll
          for (int j = 0; j < 4; ++j)
#pragma unroll
            for (int e = 0; e < 4; ++e) sv[4 * j + e] = st0[4 * j + e] + oa[j][e];
        });
#pragma unroll
        for (int j = 0; j < 4; ++j)
          xbuf[1][w][j][lane] = (f32x4){st1[4 * j], st1[4 * j + 1], st1[4 * j + 2], st1[4 * j + 3]};
        const uint32_t tm0 = tmask[ta], tm1 = tmask[ta + 1];
        __syncthreads();  // barrier 1b: the partials of b are written
        const DmaAddrs nd3 = next_addrs(ta + 3);  // (rowid reads under the softmax)
        VBuf vba = pv_pre(sa, std::true_type{});   // (Vᵀ reads of P·V(a) under the softmax)
        {
          f32x4 o[4];
#pragma unroll
          for (int j = 0; j < 4; ++j) o[j] = xbuf[1][partner][j][lane];
#pragma unroll
          for (int j = 0; j < 4; ++j)
#pragma unroll
            for (int e = 0; e < 4; ++e) sv[16 + 4 * j + e] = st1[4 * j + e] + o[j][e];
        }
        // ---- online softmax (exp2 domain) on rows 8(i/4) + 4hl + i%4 of each tile ----
        // (masking only on tiles with invalid rows: tile tails, -1 / out-of-range ids;
        // the empty asm keeps this a branch, so full tiles skip the selects)
        if (__builtin_amdgcn_readfirstlane(tm0 & tm1) != 0xFFFFFFFFu) {
          asm volatile("");
          const uint32_t vm0 = tm0 >> (4 * hl), vm1 = tm1 >> (4 * hl);
#pragma unroll
          for (int i = 0; i < 16; ++i) {
            const int bit = 8 * (i / 4) + (i % 4);
            sv[i] = ((vm0 >> bit) & 1u) ? sv[i] : -INFINITY;
            sv[16 + i] = ((vm1 >> bit) & 1u) ? sv[16 + i] : -INFINITY;
          }
        }
        // max of the raw scores, then scaled: rounding is monotonic, so this is
        // the max of the scaled scores
        float mloc = -INFINITY;
#pragma unroll
        for (int i = 0; i < 32; ++i) mloc = fmaxf(mloc, sv[i]);
        mloc = wave_max_pair(mloc) * sc;
        const bool grow = mloc > m_run;
        const float m_new = grow ? mloc : m_run;
        const float alpha = grow ? __builtin_amdgcn_exp2f(m_run - m_new) : 1.0f;  // -inf -> 0
        m_run = m_new;
        l_part *= alpha;
        // a head with no key and no sink yet (m_run = -inf) has every score -inf:
        // subtracting 0 instead keeps its P at exactly 0
        const float m_sub = m_run == -INFINITY ? 0.0f : m_run;
        i16x8 pk0[2], pk1[2];
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          const float p = __builtin_amdgcn_exp2f(__builtin_fmaf(sv[i], sc, -m_sub));
          l_part += p;
          pk0[i / 8][i % 8] = Ops::from_f32(p);
        }
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          const float p = __builtin_amdgcn_exp2f(__builtin_fmaf(sv[16 + i], sc, -m_sub));
          l_part += p;
          pk1[i / 8][i % 8] = Ops::from_f32(p);
        }

        pv_tile(sa, vba, pk0, alpha, nd3, std::true_type{}, std::false_type{});
        VBuf vbb = pv_pre(sbt, std::false_type{});  // (read while the barrier waits)
        __syncthreads();  // barrier X: stage a is free
        pv_tile(sbt, vbb, pk1, alpha, nd3, std::false_type{}, std::true_type{});
        nd = next_addrs(ta + 4);
        wait_vmcnt<DMA_PER_TILE>();  // this wave's share of tile a + 2 (a + 3's in flight)
        __syncthreads();             // barrier 2: stage b free; tile a + 2 in LDS
      }
      wait_vmcnt<0>();  // the last (zero-row) DMAs have landed
      // the item's last Q·Kᵀ has read qf: the next item's query fragment goes out
      // now and lands under the epilogue (before the output stores, so waiting
      // for it does not wait for them)
      if constexpr (PREF) {
        if (last_chunk) q_pref = prefetch_next_q();
      }
    }

    if (p_lo >= p_hi) m_run = seed_m();  // an item with no rows: the sink alone
    // ---- row sums of the two row halves (lanes l and l ^ 32, same head) ----
    const float l_run = wave_sum_pair(l_part);

    // ---- epilogue: the item's rows go out through LDS (the ring is free once
    // every wave's last DMAs have landed), so every store instruction writes
    // whole rows ----
    __syncthreads();
    {
      const KernelArgs a = fresh_args();
      int w_e = w;  // (the rows' addresses are formed here, not before the item loop)
      asm volatile("" : "+s"(w_e));
      unsigned char* stg = kv_lds;
      const int nh = min(MB, a.num_heads - hb * MB);  // heads of this item
      int lane_e = lane, hl_e = hlocal, dv_e = dh * (DV / 2) + 4 * hl;
      asm volatile("" : "+v"(lane_e), "+v"(hl_e), "+v"(dv_e));
      if (!partial) {
        constexpr int SROW = DV * 2 + 16;  // staging row stride (bytes; 16-byte aligned rows)
        static_assert(MB * SROW <= NSTG * STAGE_BYTES, "output staging");
        const float inv = 1.0f / l_run;
#pragma unroll
        for (int d = 0; d < DVB; ++d)
#pragma unroll
          for (int g4 = 0; g4 < 4; ++g4) {
            const int dv = dv_e + 32 * d + 8 * g4;
            const i16x4 v = {Ops::from_f32(acc[d][4 * g4] * inv),
                             Ops::from_f32(acc[d][4 * g4 + 1] * inv),
                             Ops::from_f32(acc[d][4 * g4 + 2] * inv),
                             Ops::from_f32(acc[d][4 * g4 + 3] * inv)};
            *(i16x4*)(stg + hl_e * SROW + dv * 2) = v;
          }
        __syncthreads();
        if (tok_ok) {
          char* obase = (char*)((T*)a.out + ((size_t)tok * a.num_heads + hb * MB) * DV);
          rows_out<MB, NW, SROW>(stg, nh, w_e, lane_e, [&](int h, i32x4 v) {
            *(i32x4*)(obase + h * DV * 2 + 16 * lane_e) = v;
          });
          if (dh == 0 && hl == 0 && head_ok)
            a.lse[(size_t)tok * a.num_heads + hb * MB + hl_e] = (m_run + __log2f(l_run)) * LN2;
        }
      } else if (slot >= 0 && slot < a.num_partial_slots && a.workspace) {
        // fp16 partials (acc / l, scaled): the row max over both dv halves (lanes
        // l, l ^ 32 and the partner wave) picks the scale; rows staged whole, as
        // the outputs are
        constexpr int SROW = DV * 2 + 16;  // staging row stride (bytes; 16-byte aligned rows)
        static_assert(MB * SROW + 2 * MB * 4 <= NSTG * STAGE_BYTES, "partial staging");
        float* rmax = (float*)(stg + MB * SROW);
        const bool empty = !(l_run > 0.0f);
        const float inv = empty ? 0.0f : 1.0f / l_run;
        float amax = 0.0f;
#pragma unroll
        for (int d = 0; d < DVB; ++d)
#pragma unroll
          for (int j = 0; j < 16; ++j) amax = fmaxf(amax, fabsf(acc[d][j]));
        // max |acc| times inv is max |acc * inv| (rounding is monotonic)
        amax = wave_max_pair(amax) * inv;
        if (hl == 0) rmax[dh * MB + hl_e] = amax;
        __syncthreads();
        const PartialScale ps = partial_scale(fmaxf(rmax[hl_e], rmax[MB + hl_e]));
#pragma unroll
        for (int d = 0; d < DVB; ++d)
#pragma unroll
          for (int g4 = 0; g4 < 4; ++g4) {
            const int dv = dv_e + 32 * d + 8 * g4;
            i16x4 v;
#pragma unroll
            for (int e = 0; e < 4; ++e)
              v[e] = __builtin_bit_cast(short, (_Float16)(acc[d][4 * g4 + e] * inv * ps.scale));
            *(i16x4*)(stg + hl_e * SROW + dv * 2) = v;
          }
        __syncthreads();
        const float lse_piece = empty ? -INFINITY : (m_run + __log2f(l_run)) * LN2;
        if (merge_here) {
          // read by another workgroup in this launch: agent-coherent stores
          const __amdgpu_buffer_rsrc_t rs = partial_rsrc(a, MB, DV);
          const uint32_t base = (uint32_t)slot * MB * DV * 2;
          rows_out<MB, NW, SROW>(stg, nh, w_e, lane_e, [&](int h, i32x4 v) {
            partial_store16(rs, base + (uint32_t)(h * DV * 2 + 16 * lane_e), v);
          });
          if (dh == 0 && hl == 0 && head_ok) {
            const uint32_t lo = (uint32_t)a.num_partial_slots * MB * DV * 2;
            partial_store4(rs, lo + ((uint32_t)slot * MB + hl_e) * 4, lse_piece);
            partial_store4(rs, lo + ((uint32_t)(a.num_partial_slots + slot) * MB + hl_e) * 4,
                           ps.inv);
          }
        } else {
          char* wbase = (char*)a.workspace + (size_t)slot * MB * DV * 2;
          rows_out<MB, NW, SROW>(stg, nh, w_e, lane_e, [&](int h, i32x4 v) {
            *(i32x4*)(wbase + h * DV * 2 + 16 * lane_e) = v;
          });
          if (dh == 0 && hl == 0 && head_ok) {
            float* wl = partial_lse(a, MB, DV);
            wl[(size_t)slot * MB + hl_e] = lse_piece;
            wl[(size_t)(a.num_partial_slots + slot) * MB + hl_e] = ps.inv;
          }
        }
      }
    }
    if (partial && merge_here) {
      // the piece that completes the item merges it (bit-identical to merge_kernel)
      const KernelArgs a = fresh_args();
      const bool cont = first_item && j_start > 0;
      const int slot0 = cont ? slot - (cont_k < 0 ? -cont_k : cont_k) : slot;
      if (split_slots_ok(a, slot0, slot)) {
        const int npc = split_arrive(a, slot0, slot, cont && cont_k > 0, &merge_word);
        if (npc > 0) merge_item_here<DV, T, MB, NW>(a, tok, hb, slot0, npc);
      }
      if (!cont) last_owed = false;
    }
    if (partial) ++slot;
    first_item = false;
    if (is_end) break;
    ++m;
  }
  if (last_owed || (merge_here && first_item && j_start > 0))
    split_settle(a, first_item && j_start > 0, cont_k, last_owed, slot);
  zero_unowned_rows<T>(a, tok_lo, tok_hi, fa_row, nfa, tid, NT);
}

// ---------------------------------------------------------------------------
// Attention kernel, software-pipelined form (two waves per SIMD)
// ---------------------------------------------------------------------------
// Waves: NHG head groups of 32 heads x 4 = 4*NHG waves (two per SIMD at 64
// heads). Wave w -> head group hg = w / 4 and quarter wq = w % 4, with row half
// rh = wq % 2 and head half qh = wq / 2.
//   Q·Kᵀ:  Sᵀ[16 rows (16rh ..) x 16 heads (hg*32 + 16qh ..)] over the whole
//          d_qk with v_mfma_f32_16x16x32 (A = the wave's K rows from LDS, B = Qᵀ
//          in AGPRs), as two chains (even / odd k-steps) added at the end.
//   softmax: in registers, 4 rows x 1 head per lane; a head's 16 rows of the
//          wave sit in lanes l, l^16, l^32, l^48 (max / sum over them by
//          permlane swaps), the tile max over both row halves meets through
//          LDS. The running max moves at every tile whose max exceeds it
//          (golden.py:187-191's rule at 32-row tiles); both row halves hold the
//          same max, factor and running max of a head. Pᵀ (input type) of the
//          wave's rows and the rescale factors go to LDS.
//   P·V:   Oᵀ[dv quarter wq (128) x 32 heads of hg] += Vᵀ·Pᵀ with
//          v_mfma_f32_32x32x16 (A = Vᵀ via ds_read_b64_tr_b16, B = Pᵀ of the
//          head group from LDS).
// Pipeline, per tile t (4-stage ring):
//   phase A: Q·Kᵀ MFMAs of tile t + 1 with the softmax of tile t between them,
//            and the row DMAs of tile t + 3 (into the stage tile t - 1 left);
//            then the wave's row max of tile t + 1 per head to LDS;
//   barrier 1 (Pᵀ and factors of tile t, row maxima of t + 1 written);
//   phase B: tile max of t + 1; rescale and P·V of tile t; wait for this
//            wave's DMAs of tile t + 2;
//   barrier 2 (tile t + 2 in LDS, stage t and the exchange buffers free).
// Pᵀ of tile t lives in the rope part of stage t (read by Q·Kᵀ of tile t during
// phase A of t - 1, refilled by the DMAs issued in phase A of t + 1).
// fp8 rows (KVF = SAS_KV_FP8_DS_MLA): tile t + 2 is loaded into VGPRs in phase A
// and dequantized into its stage in phase B.
// LDS stage layout of the pipelined kernel (one 32-row tile). Main part: row r
// (dims 0..511, 1 KB) at ring_row_base(r): rows permuted within groups of four
// and offset by 0..3 sixteen-byte slots inside 1088-byte row slots. Rope part
// (dims 512..575): chunk c of row r at slot 8 r + (c ^ ((r >> 1) & 7)). Both were
// chosen by measuring SQ_LDS_BANK_CONFLICT on MI355X: the 16x16x32 K-operand
// reads (16 rows x 4 consecutive chunks per instruction), the transposed Vᵀ reads
// and the 32x32x16 K-operand reads are all conflict-free in it.
__device__ __host__ inline int ring_row_base(int r) {
  const int a = r >> 4, b = (r >> 2) & 3, c = r & 3;
  return (16 * a + 4 * b + ((c + (b >> 1)) & 3)) * MAIN_ROW_BYTES + 16 * (2 * (b & 1) + a);
}
__device__ __host__ inline int ring_rope_slot(int r, int c) { return 8 * r + (c ^ ((r >> 1) & 7)); }
// fp8 Q·Kᵀ stage: chunk swizzle of row r (row bits 1, 0, 2, 3 to chunk bits 0, 1, 2,
// 3). A K-operand read (ds_read_b128) has lane l at row 16 rh + l % 16, chunk
// 8 blk + 2 (l / 16) + h. A b128 read is served 16 lanes per cycle, the lanes of
// one parity in one 32-lane half (lane bits 0 and 5 fixed): fitted to
// SQ_LDS_BANK_CONFLICT over single-pattern probe kernels on MI355X (it is the
// only such grouping under which ring_row_base reads are conflict-free and the
// dims-split kernel's rotated layout and two earlier fp8 layouts are 2-way
// conflicted, as measured). Such a cycle holds 8 rows of one parity x 2 chunk
// pairs, which the swizzle spreads over the 16 bank groups.
__device__ __host__ inline int k8_swz(int r) {
  return ((r >> 1) & 1) | ((r & 1) << 1) | (((r >> 2) & 1) << 2) | (((r >> 3) & 1) << 3);
}
__device__ __host__ inline int k8_chunk(int r, int c) { return (c & 16) | ((c ^ k8_swz(r)) & 15); }

template <int DQK, int DV, int NHG, typename T, int KVF, bool QK8 = false>
__global__ __launch_bounds__(256 * NHG) void attn3_kernel(const KernelArgs a) {
  constexpr int NW = 4 * NHG;            // waves per workgroup
  constexpr int MB = 32 * NHG;           // heads per item (m-block)
  constexpr int NT = 64 * NW;            // threads
  constexpr bool ROPE = DQK == 576;      // 64 extra rope dims after the 512 main dims
  constexpr bool FP8 = KVF == SAS_KV_FP8_DS_MLA;
  constexpr int ROWB = FP8 ? SAS_FP8_ROW_BYTES : DQK * 2;  // bytes per cache row in HBM
  constexpr int ROPE_OFF = FP8 ? 528 : 1024;               // byte offset of the rope dims
  constexpr int NKS = DQK / 32;          // 16x16x32 k-steps over d_qk (18 or 16)
  constexpr int NKS_MAIN = 16;           // k-steps over the 512 main dims
  constexpr int DVQ = DV / 4;            // dv per wave (a quarter)
  constexpr int DVB = DVQ / 32;          // 32-wide dv blocks per wave (4)
  // LDS ring depth: the DMA path keeps tile it + 3 in flight; fp8 rows fill tile
  // it + 2 from registers, which three stages hold (the space of the fourth goes
  // to a longer row-id buffer and, in the fp8 Q·Kᵀ form, the e4m3 K stages)
  constexpr int NSTG = FP8 ? 3 : 4;
  constexpr int STAGE_BYTES = MAIN_BYTES + (ROPE ? ROPE_BYTES : 0);
  constexpr int PB_HG = 32 * 64;         // Pᵀ of one head group: 32 heads x 32 rows x 2 B
  // fp8 Q·Kᵀ (QK8): two stages of the tile's raw e4m3 dims 0..511 (row r at
  // r * 512, its 16-byte chunk c at chunk (c & 16) | ((c ^ k8_swz(r)) & 15), see
  // k8_swz) followed by the block scales as [block][row] floats
  constexpr int K8_ROW = 512;
  constexpr int K8_SCALES = TILE * K8_ROW;
  constexpr int K8_SSTRIDE = 36;  // floats per block of scales (the 4 writers of a row hit 4 banks)
  constexpr int K8_STAGE = K8_SCALES + 4 * K8_SSTRIDE * 4;
  constexpr int K8_BASE = NSTG * STAGE_BYTES + (ROPE ? 0 : NHG * PB_HG);
  constexpr int ROWS_PER_WAVE = TILE / NW;             // main-part DMA instructions per wave
  constexpr int NROPE = ROPE ? TILE / 8 : 0;           // rope DMA instructions per tile (4)
  constexpr int DMA_MAX = ROWS_PER_WAVE + (ROPE ? 1 : 0);  // per wave and tile (waves w < NROPE)
  // positions resolved into LDS at a time (fp8 rows with 64-head items: 2048, so a
  // 2048-row item is one chunk: one resolution, one pipeline start and, in the
  // fp8 Q·Kᵀ form, one quantization of the query)
  constexpr int RCH = (FP8 && NHG == 2) ? 2048 : 1024;
  static_assert(DQK == 512 || DQK == 576, "head_dim");
  static_assert(DV == 512, "head_dim_v");
  static_assert((STAGE_BYTES % 1024) == 0, "stage alignment");
  static_assert(TILE % NW == 0 && NROPE <= NW, "DMA split");
  static_assert(!ROPE || NHG * PB_HG <= ROPE_BYTES, "Pᵀ in the rope part of a stage");
  static_assert(!FP8 || (ROPE && __is_same(T, __bf16)), "fp8 rows: head_dim 576, bf16");
  static_assert(!QK8 || FP8, "fp8 Q·Kᵀ reads fp8 rows");
  constexpr int RPL = 2 * ROWS_PER_WAVE;  // fp8 rows: rope bytes per lane per tile (8 or 16)
  typedef uint32_t ropev __attribute__((ext_vector_type(RPL / 4)));
  typedef MfmaOps<T> Ops;
  typedef typename Ops::vec8 vec8;

  __shared__ __attribute__((aligned(1024))) unsigned char kv_lds[K8_BASE + (QK8 ? 2 * K8_STAGE : 0)];
  __shared__ float htab[NHG][32];     // per head: rescale factor of the tile / final m
  __shared__ float xmax[NHG][2][32];  // per head and row half: row max of a tile / final l
  __shared__ uint32_t rowid[RCH];
  __shared__ uint32_t tmask[RCH / TILE];
  __shared__ int first_neg[2];  // first -1 of the top-k scan (the slots alternate between scans)

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int hg = w >> 2;
  const int wq = w & 3;
  const int rh = wq & 1;
  const int qh = wq >> 1;
  const int r16 = lane & 15;
  const int g4 = lane >> 4;                  // 16-lane group
  const int hl = lane >> 5;
  const int hq = hg * 32 + 16 * qh + r16;    // softmax head within the m-block
  const int hp = hg * 32 + (lane & 31);      // P·V head within the m-block
  const bool has_rope = ROPE && w < NROPE;   // this wave issues rope DMA instruction w
  const int hblocks = (a.num_heads + MB - 1) / MB;  // 1 or 2 (the launch's check of m_base)
  const int hshift = hblocks - 1;
  // Kᵀ operand of 16x16x32 (A = 16 rows x 32 dims): row 16rh + r16, dims 32ks + 8g4
  const int k_row = 16 * rh + r16;
  const int k_base = ring_row_base(k_row) + 16 * g4;
  const int rope_k0 = MAIN_BYTES + 16 * ring_rope_slot(k_row, g4);
  const int rope_k1 = MAIN_BYTES + 16 * ring_rope_slot(k_row, 4 + g4);
  // Vᵀ operand (ds_read_b64_tr_b16) of k-step kq: the 16-lane group (lane>>4) reads
  // a 4-row block at dv 128wq + 16*((lane>>4)&1) + 4*(lane&3) (+32d); its first read
  // (k elements 0..3) takes rows 16kq + 12hl + (lane&15)/4, the second (elements
  // 4..7) rows 16kq + 8 - 4hl + (lane&15)/4 (lanes 32..63 take their two row blocks
  // in swapped order, which spreads the Pᵀ writes over all banks).
  const int tr_col = wq * DVQ * 2 + ((lane >> 4) & 1) * 32 + (lane & 3) * 8;
  const int tr_r = (lane & 15) >> 2;
  const int tr00 = ring_row_base(12 * hl + tr_r) + tr_col;
  const int tr01 = ring_row_base(8 - 4 * hl + tr_r) + tr_col;
  const int tr10 = ring_row_base(16 + 12 * hl + tr_r) + tr_col;
  const int tr11 = ring_row_base(24 - 4 * hl + tr_r) + tr_col;
  // Pᵀ buffer: head h (of the group) at 64 h, its rows in the P·V B-operand order
  // (k-step kq, lane half hl: chunk 2kq + hl holds rows 16kq + 12hl .. +3 in its
  // first half and rows 16kq + 8 - 4hl .. +3 in its second); chunk q of head h is
  // stored at chunk q ^ ((h >> 2) & 3). The wave writes rows 16rh + 4g4 + i of head
  // 16qh + r16: chunk 2rh + (g4 & 1), half (g4 & 1) ^ (g4 >> 1).
  const int pw_q = 2 * rh + (g4 & 1);
  const int pw_off = hg * PB_HG + (16 * qh + r16) * 64 + 16 * (pw_q ^ ((r16 >> 2) & 3)) +
                     8 * ((g4 & 1) ^ (g4 >> 1));
  const int pr_head = lane & 31;
  const int pr_off0 = hg * PB_HG + pr_head * 64 + 16 * ((0 + hl) ^ ((pr_head >> 2) & 3));
  const int pr_off1 = hg * PB_HG + pr_head * 64 + 16 * ((2 + hl) ^ ((pr_head >> 2) & 3));

  // with at most 64 batches, their lengths and query offsets in one lane each
  const QRows qrows(a);
  const bool lens_in_lanes = a.batch <= 64;
  int lane_aq = 0, lane_kv = 0, lane_qp = 0;
  if (lens_in_lanes) {
    const int lb = lane < a.batch ? lane : a.batch - 1;
    lane_aq = qrows.rows[lb];
    lane_kv = a.seqused_kv[lb];
    lane_qp = qrows.first[lb];
  }
  int s2b = a.s2_base;
  int nfa = a.num_fa;
  if (a.num_fd == SAS_SCHED_DEVICE) {
    if (!dev_sched_ok(a, MB)) {
      if (blockIdx.x == 0) nan_fill<T>(a, tid, NT);
      return;
    }
    s2b = a.metadata[SAS_CFG_OFFSET + 1];
    nfa = a.metadata[SAS_CFG_OFFSET + 2];  // rows in use (the grid is sized for num_fa)
  }
  // XCD-aware row mapping: consecutive FA rows (pieces of one item) share an XCD.
  const int per_xcd = (nfa + 7) >> 3;
  const int fa_row = (int)(blockIdx.x & 7) * per_xcd + (int)(blockIdx.x >> 3);
  if (fa_row >= nfa || (int)(blockIdx.x >> 3) >= per_xcd) return;
  const int32_t* fa = a.metadata + fa_row * SAS_FA_METADATA_SIZE;
  if (fa[0] == 0) return;
  // where the whole schedule ends (loaded beside this row's cursors)
  const int32_t* fa_last = a.metadata + (nfa - 1) * SAS_FA_METADATA_SIZE;
  int last_on = fa_last[0], last_b = fa_last[4], last_m = fa_last[5];
  int b = fa[1], m = fa[2];
  const int j_start = fa[3];
  const int b_end = fa[4], s_end = fa[5], j_end = fa[6];
  int slot = fa[7];
  const uint32_t kv_base = (uint32_t)(uintptr_t)kv_lds;

  const char* ori_kv = (const char*)a.ori_kv;
  const char* cmp_kv = (const char*)(a.cmp_kv ? a.cmp_kv : a.ori_kv);
  const float sc = a.softmax_scale * LOG2E;
  if (tid < 2) first_neg[tid] = INT32_MAX;
  __syncthreads();

  lane_aq = qrows.count(lane_aq, lane_qp);
  lane_qp = qrows.start(lane, lane_qp);
  asm volatile("" : "+v"(lane_aq), "+v"(lane_kv), "+v"(lane_qp));
  // cumulative row counts: the tokens [tok_lo, tok_hi) of the schedule's rows
  int tok_lo = 0, tok_hi = a.total_tokens;
  if (qrows.cumulative) {
    while (last_on == 0) {  // (a row out of use: the last one before it, at most this one)
      fa_last -= SAS_FA_METADATA_SIZE;
      last_on = fa_last[0], last_b = fa_last[4], last_m = fa_last[5];
    }
    tok_lo = ld_uniform(qrows.first);
    const bool inside = last_b < a.batch;
    tok_hi = ld_uniform(qrows.first + (last_b < 0 ? 0 : (inside ? last_b : a.batch))) +
             (inside ? last_m >> hshift : 0);
  }

  // Sinks of this lane's softmax head in the (at most two) head blocks of an
  // item, loaded once: a load per item would also wait for the previous item's
  // output stores (one in-order counter covers loads and stores). They are
  // first read after the first item's resolution has waited for its loads.
  const float sink_hb0 = hq < a.num_heads ? a.sinks[hq] : -INFINITY;
  const float sink_hb1 = MB + hq < a.num_heads ? a.sinks[MB + hq] : -INFINITY;
  int item_par = 0;  // which first_neg slot the next top-k scan uses
  bool first_item = true;
  for (;;) {
    const KernelArgs a = fresh_args();
    b = __builtin_amdgcn_readfirstlane(b);
    m = __builtin_amdgcn_readfirstlane(m);
    // the batch's lengths and query offset, loaded together (one scalar round
    // trip; the index is clamped, so past the last batch they are not used)
    int act_q, act_kv, qpre;
    auto load_batch = [&] {
      const int bc = b < a.batch ? b : a.batch - 1;
      if (lens_in_lanes) {
        act_q = __builtin_amdgcn_readlane(lane_aq, bc);
        act_kv = __builtin_amdgcn_readlane(lane_kv, bc);
        qpre = __builtin_amdgcn_readlane(lane_qp, bc);
        return;
      }
      const int first_b = ld_uniform(qrows.first + bc);
      act_q = qrows.count(ld_uniform(qrows.rows + bc), first_b);
      act_kv = ld_uniform(a.seqused_kv + bc);
      qpre = qrows.start(bc, first_b);
    };
    load_batch();
    // normalise the cursor: skip batches with no (more) query rows
    while (b < a.batch && b <= b_end && m >= act_q * hblocks) {
      ++b;
      m = 0;
      load_batch();
    }
    if (b >= a.batch || b > b_end || (b == b_end && m > s_end)) break;
    const bool is_end = (b == b_end && m == s_end);
    const int s = m >> hshift;
    const int hb = m - s * hblocks;
    if (is_end && j_end == 0) break;

    const int tok = qpre + s;
    const ItemGeom g = item_geom_at(a, act_q, act_kv, s);
    const int L = g.n_win + g.n_cmp;
    const bool partial = (first_item && j_start > 0) || is_end;
    const int blo = first_item ? j_start : 0;
    const int p_lo = blo * s2b;
    const int p_hi = is_end && (int64_t)j_end * s2b < L ? j_end * s2b : L;
    const bool tok_ok = tok >= 0 && tok < a.total_tokens;

    // query fragment of the wave's 16 heads (B operand of Sᵀ = K·Qᵀ)
    i16x8 qf[NKS];
    // fp8 Q·Kᵀ: the head's latent as e4m3 codes of q / sq (B operands of the four
    // 128-dim blocks), sq = amax / 448 over the head's 512 latent dims
    i32x8 q8[4];
    float sq = 1.0f;
    // ---- online-softmax state of head hq (golden.py:156-160 seeds m = sink,
    // l = 1; the 1 goes to the lanes of group 0 of the first row half, whose row
    // sums are added to the others' at the end) ----
    const bool hq_ok = hb * MB + hq < a.num_heads;
    // the sink seeds m_run once the item's first loads have been waited for
    auto seed_m = [&]() -> float {
      const float sink_v = hb == 0 ? sink_hb0 : sink_hb1;
      return partial ? -INFINITY : (hq_ok ? sink_v * LOG2E : -INFINITY);
    };
    float m_run = -INFINITY;
    float l_part = (partial || g4 != 0 || rh != 0) ? 0.0f : 1.0f;
    float mx = -INFINITY;
    f32x16 acc[DVB];
#pragma unroll
    for (int d = 0; d < DVB; ++d)
#pragma unroll
      for (int j = 0; j < 16; ++j) acc[d][j] = 0.0f;

    Resolver res(a, g, b, tok, tok_ok, p_hi);
    for (int c0 = p_lo; c0 < p_hi; c0 += RCH) {
      const int clen = (p_hi - c0) < RCH ? (p_hi - c0) : RCH;
      const int ntile = (clen + TILE - 1) / TILE;
      // query fragment of the item (first chunk): compiler-visible loads issued
      // before the resolution's loads, so they land during its memory round
      // trips; the compiler's wait for the table words below covers them.
      // (fp8 Q·Kᵀ: loaded and quantized again for every chunk, so nothing of the
      // query is carried across the chunk loop but its e4m3 form within a chunk:
      // a carried bf16 copy next to the e4m3 one spilled the resolution's registers)
      if (QK8 || c0 == p_lo) {
        const int head_q = hb * MB + hq;
        const bool hok = head_q < a.num_heads && tok_ok;
        // (rows out of range read token 0's first head: never stored)
        const short* qrow = (const short*)a.q + ((size_t)(hok ? tok : 0) * a.num_heads +
                                                 (hok ? head_q : 0)) * DQK;
#pragma unroll
        for (int ks = 0; ks < NKS; ++ks) {
          // (fp8 Q·Kᵀ: latent k-step 4 blk + h holds dims 128 blk + 32 g4 + 8 h, the
          // lane's quarter of e4m3 block blk)
          const int dim = (QK8 && ks < NKS_MAIN) ? 128 * (ks >> 2) + 32 * g4 + 8 * (ks & 3)
                                                 : 32 * ks + 8 * g4;
          qf[ks] = *(const i16x8*)(qrow + dim);
        }
      }
      // ---- positions -> cache rows (bit 31: compressed cache) ----
      res.template chunk<NT, RCH, RCH / NT + 4>(a, c0, clen, tid, rowid, tmask, first_neg, item_par, [&] {
        if (c0 == p_lo) m_run = seed_m();
        if constexpr (QK8) quantize_q(qf, q8, sq);
      });

      // ---- DMA issue for one tile into one ring stage ----
      // main part: wave w fills rows w, w + NW, ...; one 1 KB row per instruction
      // rope part: instruction i (wave i < NROPE) fills rows 8i..8i+7 (8 lanes per row)
      auto row_ptr = [&](uint32_t id) -> const char* {
        const char* base = (id & 0x80000000u) ? cmp_kv : ori_kv;
        const char* p = base + (size_t)(id & 0x7FFFFFFFu) * ROWB;
        return id == ROW_INVALID ? (const char*)g_zero_row : p;
      };
      auto lane_row = [&](uint64_t ptrs, int j) -> const char* {
        const uint32_t lo = __builtin_amdgcn_readlane((uint32_t)ptrs, j);
        const uint32_t hi = __builtin_amdgcn_readlane((uint32_t)(ptrs >> 32), j);
        return (const char*)(uintptr_t)(((uint64_t)hi << 32) | lo);
      };
      // The DMAs of one tile: the row addresses are gathered first (next_addrs),
      // then instruction j goes out with dma_one(j), so the instructions can be
      // spread between MFMAs.
      struct DmaAddrs {
        uint64_t main;     // lane j < ROWS_PER_WAVE: this wave's j-th main row
        const char* rope;  // per lane: its 16-byte rope piece (waves w < NROPE)
        uint32_t sbase;
      };
      // Addresses of the DMAs of tile t. Past the chunk's last tile the
      // instructions read the zero row into the stage they would fill, which
      // nothing reads before the chunk ends (keeps the vmcnt accounting uniform).
      auto next_addrs = [&](int tile) -> DmaAddrs {
        DmaAddrs d;
        const bool real = tile < ntile;
        d.sbase = kv_base + (tile % NSTG) * STAGE_BYTES;
        const int t0 = real ? tile : 0;
        d.main = (uint64_t)(uintptr_t)row_ptr(
            rowid[t0 * TILE + w + NW * (lane < ROWS_PER_WAVE ? lane : 0)]);
        d.rope = (const char*)g_zero_row;
        if constexpr (ROPE) {
          const int r = 8 * (w < NROPE ? w : 0) + (lane >> 3);  // rope instruction w: rows 8w..8w+7
          const int cr = (lane & 7) ^ ((r >> 1) & 7);           // the chunk slot lane & 7 holds
          d.rope = row_ptr(rowid[t0 * TILE + r]) + 1024 + cr * 16;
        }
        if (!real) {
          d.main = (uint64_t)(uintptr_t)g_zero_row;
          d.rope = (const char*)g_zero_row;
        }
        return d;
      };
      auto dma_one = [&](const DmaAddrs& d, int j) {
        if (j < ROWS_PER_WAVE) {
          const int r = w + NW * j;
          dma16_sbase(lane_row(d.main, j), (uint32_t)lane * 16u, d.sbase + ring_row_base(r));
        } else if constexpr (ROPE) {
          if (has_rope) dma16_vaddr(d.rope, d.sbase + MAIN_BYTES + w * 1024);
        }
      };
      auto issue = [&](const DmaAddrs& d) {
#pragma unroll
        for (int j = 0; j < DMA_MAX; ++j) dma_one(d, j);
      };
      // this wave's DMAs of all but the newest tile have landed
      auto wait_all_but_one_tile = [&]() {
        if (has_rope) wait_vmcnt<ROWS_PER_WAVE + 1>();
        else wait_vmcnt<ROWS_PER_WAVE>();
      };

      // ---- fp8 rows: VGPR loads, then dequantize into one ring stage ----
      // wave w takes rows w + NW j (j < ROWS_PER_WAVE): lane l loads bytes 8l..8l+7
      // (dims 8l..8l+7, scale l / 16) of each, and RPL rope bytes of row
      // w + NW (l / (128 / RPL)). Ordinary (L2-allocating) loads: the token's other
      // 64-head m-block reads the same rows on the same XCD shortly after, and
      // finds them in L2 (measured: 9 % fewer HBM bytes than streaming loads, at
      // +0.5 % kernel time).
      struct Fp8Tile {
        uint2 v[ROWS_PER_WAVE];
        float s[ROWS_PER_WAVE];
        ropev rope;
      };
      constexpr int ROPE_LPR = 128 / RPL;  // lanes per row for the rope bytes
      typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
      auto fp8_load = [&](Fp8Tile& f, int tile) {
        const uint64_t my_ptrs = (uint64_t)(uintptr_t)row_ptr(
            rowid[tile * TILE + w + NW * (lane < ROWS_PER_WAVE ? lane : 0)]);
        const char* rp = nullptr;
#pragma unroll
        for (int j = 0; j < ROWS_PER_WAVE; ++j) {
          const char* p = lane_row(my_ptrs, j);
          const u32x2 t = *((const SAS_GLOBAL u32x2*)(p + 8 * lane));
          f.v[j] = make_uint2(t[0], t[1]);
          f.s[j] = *((const SAS_GLOBAL float*)(p + 512 + 4 * (lane >> 4)));
          rp = (lane / ROPE_LPR == j) ? p : rp;
        }
        f.rope = *(
            (const SAS_GLOBAL ropev*)(rp + ROPE_OFF + (lane % ROPE_LPR) * RPL));
      };
      auto fp8_store = [&](const Fp8Tile& f, int tile) {
        unsigned char* sb = kv_lds + (tile % NSTG) * STAGE_BYTES;
#pragma unroll
        for (int j = 0; j < ROWS_PER_WAVE; ++j) {
          const int r = w + NW * j;
          *(i16x8*)(sb + ring_row_base(r) + 16 * lane) = fp8x8_dequant_bf16(f.v[j], f.s[j]);
        }
        if constexpr (QK8) {
          // the raw e4m3 bytes and the block scales into the tile's K8 stage
          unsigned char* kb8 = kv_lds + K8_BASE + (tile & 1) * K8_STAGE;
#pragma unroll
          for (int j = 0; j < ROWS_PER_WAVE; ++j) {
            const int r = w + NW * j;
            *(uint2*)(kb8 + r * K8_ROW + 16 * k8_chunk(r, lane >> 1) + 8 * (lane & 1)) = f.v[j];
            if ((lane & 15) == 0) *(float*)(kb8 + K8_SCALES + 4 * ((lane >> 4) * K8_SSTRIDE + r)) = f.s[j];
          }
        }
        // the lane's RPL rope bytes: whole 16-byte chunks (RPL 16; consecutive chunks
        // of a row need not be adjacent in the rotated rope layout, so one store
        // each) or half of one (RPL 8)
        const int r = w + NW * (lane / ROPE_LPR);
        const int b0 = (lane % ROPE_LPR) * RPL;  // byte offset within the row's rope
        if constexpr (RPL >= 16) {
          typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
#pragma unroll
          for (int k = 0; k < RPL / 16; ++k)
            *(u32x4*)(sb + MAIN_BYTES + ring_rope_slot(r, b0 / 16 + k) * 16) =
                (u32x4){f.rope[4 * k], f.rope[4 * k + 1], f.rope[4 * k + 2], f.rope[4 * k + 3]};
        } else {
          static_assert(RPL == 8, "rope bytes per lane");
          *(u32x2*)(sb + MAIN_BYTES + ring_rope_slot(r, b0 / 16) * 16 + (b0 & 8)) =
              (u32x2){f.rope[0], f.rope[1]};
        }
      };
      Fp8Tile fpt;

      typedef const unsigned char SAS_LDS* lds_p;
      auto stage_of = [&](int tile) -> lds_p {
        return (lds_p)(kv_base + (uint32_t)((tile % NSTG) * STAGE_BYTES));
      };
      auto pbuf_of = [&](int tile) -> uint32_t {
        return ROPE ? kv_base + (uint32_t)((tile % NSTG) * STAGE_BYTES + MAIN_BYTES)
                    : kv_base + (uint32_t)(NSTG * STAGE_BYTES);
      };
      // K operand of k-step ks (the wave's 16 rows) from stage sb
      auto kop = [&](lds_p sb, int ks) -> i16x8 {
        const lds_p p = ks < NKS_MAIN ? sb + k_base + 64 * ks
                                      : sb + (ks == NKS_MAIN ? rope_k0 : rope_k1);
        return *(const i16x8 SAS_LDS*)p;
      };
      // fp8 Q·Kᵀ: the e4m3 A operand of block blk (the wave's row k_row, bytes
      // 128 blk + 32 g4 .. + 31) from a K8 stage, and the scores of the wave's 16
      // rows x 16 heads from the four blocks' dot products d8, the rope part dr and
      // the row scales: s = sq * sum_blk sk[blk][row] * d8[blk] + dr
      auto k8_stage = [&](int tile) -> lds_p {
        return (lds_p)(kv_base + (uint32_t)(K8_BASE + (tile & 1) * K8_STAGE));
      };
      auto k8op = [&](lds_p kb8, int blk) -> i32x8 {
        const lds_p p = kb8 + k_row * K8_ROW;
        const i32x4 lo = *(const i32x4 SAS_LDS*)(p + 16 * k8_chunk(k_row, 8 * blk + 2 * g4));
        const i32x4 hi = *(const i32x4 SAS_LDS*)(p + 16 * k8_chunk(k_row, 8 * blk + 2 * g4 + 1));
        return (i32x8){lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
      };
      // block blk's scales of the wave's output rows 16 rh + 4 g4 + i (element i)
      auto k8scale = [&](lds_p kb8, int blk) -> f32x4 {
        return *(const f32x4 SAS_LDS*)(kb8 + K8_SCALES + 4 * (blk * K8_SSTRIDE + 16 * rh + 4 * g4));
      };
      auto mma8 = [&](i32x8 x, i32x8 y) -> f32x4 {
        // e4m3 x e4m3 (format selectors 0), no block scaling: v_mfma_f32_16x16x128_f8f6f4
        return __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(x, y, (f32x4){0.0f, 0.0f, 0.0f, 0.0f},
                                                                0, 0, 0, 0, 0, 0);
      };
      // s8 (+)= d * sk, element-wise (block 0 starts the sum: s8 = d * sk)
      auto scale_add = [&](f32x4& s8, f32x4 d, f32x4 sk, bool first) {
#pragma unroll
        for (int i = 0; i < 4; ++i) s8[i] = first ? d[i] * sk[i] : __builtin_fmaf(d[i], sk[i], s8[i]);
      };
      auto scores8 = [&](f32x4 s8, f32x4 dr) -> f32x4 {
        f32x4 r;
#pragma unroll
        for (int i = 0; i < 4; ++i) r[i] = __builtin_fmaf(s8[i], sq, dr[i]);
        return r;
      };
      auto mma16 = [&](i16x8 x, i16x8 y, f32x4 c) -> f32x4 {
        return __is_same(T, __bf16)
                   ? __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(vec8, x),
                                                             __builtin_bit_cast(vec8, y), c, 0, 0, 0)
                   : __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(vec8, x),
                                                            __builtin_bit_cast(vec8, y), c, 0, 0, 0);
      };
      // row max of a tile's scores over this wave's rows (lanes l, l^16, l^32,
      // l^48 hold the wave's 16 rows of the lane's head); rows the tile mask
      // marks invalid become -inf first
      auto row_max = [&](f32x4& x, int tile) -> float {
        const uint32_t tm = tmask[tile];
        if (__builtin_amdgcn_readfirstlane(tm) != 0xFFFFFFFFu) {
          const uint32_t vm = tm >> (16 * rh + 4 * g4);
#pragma unroll
          for (int i = 0; i < 4; ++i) x[i] = ((vm >> i) & 1u) ? x[i] : -INFINITY;
        }
        float mm = fmaxf(fmaxf(x[0], x[1]), fmaxf(x[2], x[3]));
        const auto r1 = __builtin_amdgcn_permlane16_swap(__float_as_uint(mm),
                                                         __float_as_uint(mm), false, false);
        mm = fmaxf(__uint_as_float(r1[0]), __uint_as_float(r1[1]));
        mm = wave_max_pair(mm);
        if (g4 == 0) xmax[hg][rh][16 * qh + r16] = mm;
        return mm;
      };

      // ---- prologue: tiles 0, 1, 2 in flight, Q·Kᵀ of tile 0 ----
      if constexpr (FP8) {
        // one tile's registers at a time (the loop holds one tile in flight too)
        fp8_load(fpt, 0);
        fp8_store(fpt, 0);
        if (ntile > 1) {
          fp8_load(fpt, 1);
          fp8_store(fpt, 1);
        }
      } else {
        issue(next_addrs(0));
        issue(next_addrs(1));
        issue(next_addrs(2));
        wait_all_but_one_tile();  // tiles 0 and 1 have landed (tile 2 may be in flight)
      }
      __syncthreads();
      f32x4 st;
      {
        const lds_p sb = stage_of(0);
        f32x4 ce = {0.0f, 0.0f, 0.0f, 0.0f}, co = {0.0f, 0.0f, 0.0f, 0.0f};
        if constexpr (QK8) {
          const lds_p kb8 = k8_stage(0);
          f32x4 s8 = ce;
#pragma unroll
          for (int blk = 0; blk < 4; ++blk)
            scale_add(s8, mma8(k8op(kb8, blk), q8[blk]), k8scale(kb8, blk), blk == 0);
          ce = mma16(kop(sb, NKS_MAIN), qf[NKS_MAIN], ce);
          ce = mma16(kop(sb, NKS_MAIN + 1), qf[NKS_MAIN + 1], ce);
          st = scores8(s8, ce);
        } else {
#pragma unroll
          for (int ks = 0; ks < NKS; ks += 2) {
            ce = mma16(kop(sb, ks), qf[ks], ce);
            co = mma16(kop(sb, ks + 1), qf[ks + 1], co);
          }
          st = ce + co;
        }
        const float own = row_max(st, 0);
        __syncthreads();
        mx = fmaxf(own, xmax[hg][rh ^ 1][16 * qh + r16]);
      }
      DmaAddrs nd;
      if constexpr (!FP8) nd = next_addrs(3);

      for (int it = 0; it < ntile; ++it) {
        const lds_p sb = stage_of(it);
        const uint32_t pb = pbuf_of(it);
        if constexpr (FP8) {
          if (it + 2 < ntile) fp8_load(fpt, it + 2);
        }
        // ---- phase A: softmax of tile it between the Q·Kᵀ MFMAs of tile it + 1 ----
        // (st holds tile it's scores, masked by row_max; mx its tile max)
        f32x4 sn;
        float own = -INFINITY;
        auto phase_a = [&](auto with_qk) {
          constexpr bool QK = decltype(with_qk)::value;
          constexpr int KPF = QK8 ? 1 : FP8 ? 3 : 6;
          const lds_p sbn = stage_of(it + 1);
          i16x8 kb[KPF];
          f32x4 ce = {0.0f, 0.0f, 0.0f, 0.0f}, co = {0.0f, 0.0f, 0.0f, 0.0f};
          // fp8 Q·Kᵀ: the e4m3 A operands two blocks ahead, the row scales
          const lds_p kb8n = QK8 ? k8_stage(it + 1) : sbn;
          i32x8 k8b[2];
          f32x4 s8, d8, skb;  // running block sum, last block's product and scales
          if constexpr (QK && QK8) {
            k8b[0] = k8op(kb8n, 0);
            k8b[1] = k8op(kb8n, 1);
          } else if constexpr (QK) {
#pragma unroll
            for (int i = 0; i < KPF; ++i) kb[i] = kop(sbn, i);
          }
          float p[4], alpha = 1.0f, m_sub = 0.0f;
          i16x4 pk;
          // softmax of tile it in slices: slice k runs after k-step k's MFMA
          auto slice = [&](int k) {
            if (k == 0) {
              const float mt = mx * sc;
              const bool grow = mt > m_run;
              const float m_new = grow ? mt : m_run;
              alpha = grow ? __builtin_amdgcn_exp2f(m_run - m_new) : 1.0f;  // -inf -> 0
              m_run = m_new;
              l_part *= alpha;
              // a head with no key and no sink yet (m_run = -inf) has every score
              // -inf: subtracting 0 instead keeps its P at exactly 0
              m_sub = m_new == -INFINITY ? 0.0f : m_new;
            } else if (k == 1) {
              // both row halves hold the same factor: the first writes it
              if (g4 == 0 && rh == 0) htab[hg][16 * qh + r16] = alpha;
            } else if (k == 2 || k == 3) {
#pragma unroll
              for (int e = 0; e < 2; ++e) {
                const int i = 2 * (k - 2) + e;
                p[i] = __builtin_amdgcn_exp2f(__builtin_fmaf(st[i], sc, -m_sub));
              }
            } else if (k == 4) {
              l_part += (p[0] + p[1]) + (p[2] + p[3]);
              pk = (i16x4){Ops::from_f32(p[0]), Ops::from_f32(p[1]), Ops::from_f32(p[2]),
                           Ops::from_f32(p[3])};
            } else if (k == 5) {
              *(i16x4 SAS_LDS*)(pb + pw_off) = pk;
            }
          };
          constexpr int DMA_AT = 6;  // first k-step with a DMA after it
          // fp8 Q·Kᵀ: steps 0..3 are the e4m3 blocks, 4 and 5 the rope k-steps
          constexpr int NSTEP = QK8 ? 6 : NKS > DMA_AT + DMA_MAX ? NKS : DMA_AT + DMA_MAX;
#pragma unroll
          for (int ks = 0; ks < NSTEP; ++ks) {
            if constexpr (QK && QK8) {
              // step k: block k's MFMA, then block k - 1's product scaled into the sum
              // (its MFMA has drained under block k's)
              if (ks < 4) {
                const f32x4 dn = mma8(k8b[ks & 1], q8[ks]);
                if (ks + 2 < 4) k8b[ks & 1] = k8op(kb8n, ks + 2);
                if (ks > 0) scale_add(s8, d8, skb, ks == 1);
                d8 = dn;
                skb = k8scale(kb8n, ks);
                if (ks == 3) kb[0] = kop(sbn, NKS_MAIN);
              } else {
                const i16x8 k0 = kb[0];
                if (ks == 4) {
                  kb[0] = kop(sbn, NKS_MAIN + 1);
                  scale_add(s8, d8, skb, false);
                }
                ce = mma16(k0, qf[NKS_MAIN + ks - 4], ce);
              }
            } else if constexpr (QK) {
              if (ks < NKS) {
                const i16x8 k0 = kb[ks % KPF];
                if (ks + KPF < NKS) kb[ks % KPF] = kop(sbn, ks + KPF);
                if (ks & 1) co = mma16(k0, qf[ks], co);
                else ce = mma16(k0, qf[ks], ce);
              }
            }
            slice(ks);
            // DMA instruction j of tile it + 3 after k-step DMA_AT + j
            if constexpr (!FP8) {
#pragma unroll
              for (int j = 0; j < DMA_MAX; ++j)
                if (j + DMA_AT == ks) dma_one(nd, j);
            }
            __builtin_amdgcn_sched_barrier(0);
          }
          if constexpr (QK) {
            if constexpr (QK8) sn = scores8(s8, ce);
            else sn = ce + co;
            own = row_max(sn, it + 1);
          }
        };
        if (it + 1 < ntile) phase_a(std::true_type{});
        else phase_a(std::false_type{});
        __syncthreads();  // barrier 1: Pᵀ, factors of tile it and row maxima of it + 1 in LDS
        DmaAddrs nd4;
        if constexpr (!FP8) nd4 = next_addrs(it + 4);  // (rowid reads under P·V)

        // ---- phase B: Oᵀ = alpha·Oᵀ + Vᵀ·Pᵀ over both 16-row k-steps ----
        {
          if (it + 1 < ntile) mx = fmaxf(own, xmax[hg][rh ^ 1][16 * qh + r16]);
          constexpr int VPF = FP8 ? 2 : SAS_VPF;
          constexpr int NPV = 2 * DVB;
          const float al = htab[hg][lane & 31];
          // (no head of the wave moved its maximum: the rescale by 1 is skipped;
          // measured -1.6 % on the fp8 long-context decode, while the same skip in
          // the dims-split kernel, whose P·V then needs a second copy, cost +8 %)
          const bool resc = __ballot(al != 1.0f) != 0;
          const i16x8 pq0 = *(const i16x8 SAS_LDS*)(pb + pr_off0);
          const i16x8 pq1 = *(const i16x8 SAS_LDS*)(pb + pr_off1);
          typedef i16x4 SAS_LDS* lds4;
          // MFMA i: dv block i % DVB, k-step i / DVB (independent accumulators back to back)
          auto vop = [&](int i) -> i16x8 {
            const int d = i % DVB, kq = i / DVB;
            const i16x4 g0 = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                (lds4)(sb + (kq ? tr10 : tr00) + d * 64));
            const i16x4 g1 = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                (lds4)(sb + (kq ? tr11 : tr01) + d * 64));
            return (i16x8){g0[0], g0[1], g0[2], g0[3], g1[0], g1[1], g1[2], g1[3]};
          };
          i16x8 vbuf[VPF];
#pragma unroll
          for (int i = 0; i < VPF; ++i) vbuf[i] = vop(i);
#pragma unroll
          for (int i = 0; i < NPV; ++i) {
            const int d = i % DVB, kq = i / DVB;
            if (kq == 0 && resc) {
#pragma unroll
              for (int j = 0; j < 16; ++j) acc[d][j] *= al;
            }
            const i16x8 aop = vbuf[i % VPF];
            if (i + VPF < NPV) vbuf[i % VPF] = vop(i + VPF);
            acc[d] = Ops::mma(aop, kq ? pq1 : pq0, acc[d]);
          }
        }
        if constexpr (FP8) {
          // tile it + 2 into its stage (tile it - 2's, free since barrier 2 of it - 2)
          if (it + 2 < ntile) fp8_store(fpt, it + 2);
        } else {
          // this wave's share of tile it + 2 has landed (tile it + 3's may be in flight)
          wait_all_but_one_tile();
        }
        __syncthreads();  // barrier 2: tile it + 2 in LDS; stage it and its Pᵀ free
        if constexpr (!FP8) nd = nd4;
        st = sn;
      }
      if constexpr (!FP8) {
        wait_vmcnt<0>();  // the last (zero-row) DMAs have landed ...
        __syncthreads();  // ... for every wave, before LDS is reused
      }
    }

    if (p_lo >= p_hi) m_run = seed_m();  // an item with no rows: the sink alone
    // ---- row sums of head hq over the wave's four lanes and both row halves;
    // (m, l) to the P·V layout (head hp = hg * 32 + lane % 32) ----
    {
      const auto r1 = __builtin_amdgcn_permlane16_swap(__float_as_uint(l_part),
                                                       __float_as_uint(l_part), false, false);
      const float l16 = __uint_as_float(r1[0]) + __uint_as_float(r1[1]);
      const float lq = wave_sum_pair(l16);
      if (g4 == 0) {
        xmax[hg][rh][16 * qh + r16] = lq;
        if (rh == 0) htab[hg][16 * qh + r16] = m_run;
      }
    }
    __syncthreads();
    const float m_fin = htab[hg][lane & 31];
    const float l_run = xmax[hg][0][lane & 31] + xmax[hg][1][lane & 31];
    const bool head_p_ok = hb * MB + hp < a.num_heads;

    // ---- epilogue: the item's rows go out through LDS (the ring is free), so
    // every store instruction writes whole rows ----
    {
      const KernelArgs a = fresh_args();
      int w_e = w;  // (the rows' addresses are formed here, not before the item loop)
      asm volatile("" : "+s"(w_e));
      unsigned char* stg = kv_lds;
      const int nh = min(MB, a.num_heads - hb * MB);  // heads of this item
      int lane_e = lane, hl_e = hp, dv_e = wq * DVQ + 4 * hl;
      asm volatile("" : "+v"(lane_e), "+v"(hl_e), "+v"(dv_e));
      if (!partial) {
        constexpr int SROW = DV * 2 + 16;  // staging row stride (bytes; 16-byte aligned rows)
        static_assert(MB * SROW <= NSTG * STAGE_BYTES, "output staging");
        const float inv = 1.0f / l_run;
#pragma unroll
        for (int d = 0; d < DVB; ++d)
#pragma unroll
          for (int q4 = 0; q4 < 4; ++q4) {
            const int dv = dv_e + 32 * d + 8 * q4;
            const i16x4 v = {Ops::from_f32(acc[d][4 * q4] * inv),
                             Ops::from_f32(acc[d][4 * q4 + 1] * inv),
                             Ops::from_f32(acc[d][4 * q4 + 2] * inv),
                             Ops::from_f32(acc[d][4 * q4 + 3] * inv)};
            *(i16x4*)(stg + hl_e * SROW + dv * 2) = v;
          }
        __syncthreads();
        if (tok_ok) {
          char* obase = (char*)((T*)a.out + ((size_t)tok * a.num_heads + hb * MB) * DV);
          rows_out<MB, NW, SROW>(stg, nh, w_e, lane_e, [&](int h, i32x4 v) {
            *(i32x4*)(obase + h * DV * 2 + 16 * lane_e) = v;
          });
          if (wq == 0 && hl == 0 && head_p_ok)
            a.lse[(size_t)tok * a.num_heads + hb * MB + hl_e] = (m_fin + __log2f(l_run)) * LN2;
        }
      } else if (slot >= 0 && slot < a.num_partial_slots && a.workspace) {
        // fp16 partials (acc / l, scaled): the row max over the four dv quarters
        // (lanes l, l ^ 32 of waves wq = 0..3) picks the scale; rows staged whole
        constexpr int SROW = DV * 2 + 16;  // staging row stride (bytes), as for the outputs
        static_assert(MB * SROW + 4 * MB * 4 <= NSTG * STAGE_BYTES, "partial staging");
        float* rmax = (float*)(stg + MB * SROW);
        const bool empty = !(l_run > 0.0f);
        const float inv = empty ? 0.0f : 1.0f / l_run;
        float amax = 0.0f;
#pragma unroll
        for (int d = 0; d < DVB; ++d)
#pragma unroll
          for (int j = 0; j < 16; ++j) amax = fmaxf(amax, fabsf(acc[d][j]));
        // max |acc| times inv is max |acc * inv| (rounding is monotonic)
        amax = wave_max_pair(amax) * inv;
        if (hl == 0) rmax[wq * MB + hl_e] = amax;
        __syncthreads();
        const PartialScale ps = partial_scale(fmaxf(fmaxf(rmax[hl_e], rmax[MB + hl_e]),
                                                    fmaxf(rmax[2 * MB + hl_e], rmax[3 * MB + hl_e])));
#pragma unroll
        for (int d = 0; d < DVB; ++d)
#pragma unroll
          for (int q4 = 0; q4 < 4; ++q4) {
            const int dv = dv_e + 32 * d + 8 * q4;
            i16x4 v;
#pragma unroll
            for (int e = 0; e < 4; ++e)
              v[e] = __builtin_bit_cast(short, (_Float16)(acc[d][4 * q4 + e] * inv * ps.scale));
            *(i16x4*)(stg + hl_e * SROW + dv * 2) = v;
          }
        __syncthreads();
        char* wbase = (char*)a.workspace + (size_t)slot * MB * DV * 2;
        rows_out<MB, NW, SROW>(stg, nh, w_e, lane_e, [&](int h, i32x4 v) {
          *(i32x4*)(wbase + h * DV * 2 + 16 * lane_e) = v;
        });
        if (wq == 0 && hl == 0 && head_p_ok) {
          float* wl = partial_lse(a, MB, DV);
          wl[(size_t)slot * MB + hl_e] = empty ? -INFINITY : (m_fin + __log2f(l_run)) * LN2;
          wl[(size_t)(a.num_partial_slots + slot) * MB + hl_e] = ps.inv;
        }
      }
    }
    __syncthreads();  // the staging area and the head tables are read out before the next item
    if (partial) ++slot;
    if (is_end) break;
    first_item = false;
    ++m;
  }
  zero_unowned_rows<T>(a, tok_lo, tok_hi, fa_row, nfa, tid, NT);
}

}  // namespace sas

#include "sas_attn_wide.h"

namespace sas {

// ---------------------------------------------------------------------------
// Split-KV merge: lse = log(e^sink + Σ e^lse_i), out = Σ e^(lse_i - lse) o_i
// ---------------------------------------------------------------------------
// Grid: (merge task, group of MERGE_HPB heads). Thread t owns head t / 32 of
// the group and the 8-column chunks (t % 32) + 32 k of its row (one 16-byte
// load of fp16 partials, one 16-byte store of outputs each): a half-wave reads
// 512 contiguous bytes per load. Each thread derives its head's weights itself
// (the piece lse values are the same words for its 32 lanes), so there is no
// LDS and no barrier, and the first two pieces' loads are in flight with the
// lse, sink and token loads.
constexpr int MERGE_HPB = 8;          // heads per workgroup
constexpr int MERGE_THREADS = 256;

template <int DV, typename T>
__device__ __forceinline__ void merge_task(const SasAttnArgs& a, int task) {
  constexpr int V4 = DV / 4;                              // float4 per head row
  constexpr int TPH = MERGE_THREADS / MERGE_HPB;          // threads per head (32)
  constexpr int PER = V4 / TPH;                           // float4 per thread (4)
  static_assert(V4 % (2 * TPH) == 0 && TPH <= 64 && 64 % TPH == 0, "merge tiling");
  const int32_t* fd = a.metadata + SAS_FD_OFFSET + task * SAS_FD_METADATA_SIZE;
  if (fd[0] == 0) return;
  const int mb = a.m_base;
  const int hblocks = (a.num_heads + mb - 1) / mb;
  const int b = fd[1], m = fd[2], slot0 = fd[3], npc = fd[4], h0 = fd[5], hn = fd[6];
  if (b < 0 || b >= a.batch || m < 0 || slot0 < 0 || npc < 1 ||
      slot0 + npc > a.num_partial_slots || h0 < 0 || hn < 1 || h0 + hn > mb)
    return;
  const int g0 = (int)blockIdx.y * MERGE_HPB;  // first head of this group within the task
  if (g0 >= hn) return;
  const int tid = threadIdx.x;
  const int hh = tid / TPH;
  const int c0 = tid % TPH;
  // rows past the task's last head (never stored) read that head's row instead
  const int hr = g0 + hh < hn ? g0 + hh : hn - 1;
  const int hloc = h0 + hr;                            // m-block slot of this thread's row
  const _Float16* wo = (const _Float16*)a.workspace;
  const float* wl = partial_lse(a, mb, DV);
  const float* wsc = wl + (size_t)a.num_partial_slots * mb;  // inverse scales
  typedef _Float16 h16x4 __attribute__((ext_vector_type(4)));
  typedef _Float16 h16x8 __attribute__((ext_vector_type(8)));
  auto piece = [&](int i, f32x4 (&v)[PER]) {
    const _Float16* src = wo + ((size_t)(slot0 + i) * mb + hloc) * DV + 8 * c0;
#pragma unroll
    for (int k = 0; k < PER / 2; ++k) {  // all of one piece's loads in flight together
      const h16x8 x = *(const h16x8*)(src + 8 * TPH * k);
      v[2 * k] = (f32x4){(float)x[0], (float)x[1], (float)x[2], (float)x[3]};
      v[2 * k + 1] = (f32x4){(float)x[4], (float)x[5], (float)x[6], (float)x[7]};
    }
  };
  auto plse = [&](int i) -> float { return wl[(size_t)(slot0 + i) * mb + hloc]; };
  auto pinv = [&](int i) -> float { return wsc[(size_t)(slot0 + i) * mb + hloc]; };
  const int s = m / hblocks;
  const int h = (m - s * hblocks) * mb + hloc;  // query head
  const bool store = g0 + hh < hn && h < a.num_heads;
  const float sink = a.sinks[h < a.num_heads ? h : a.num_heads - 1];
  const QRows qrows(a);
  const int tok = qrows.start(b, qrows.first[b]) + s;
  // lse = log(e^sink + Σ_i e^lse_i); weights e^(lse_i - lse); the sums keep the
  // piece order 0, 1, 2, ...
  f32x4 o[PER];
  float l = -INFINITY;
  auto weight = [&](float li) -> float {
    return (l == -INFINITY || li == -INFINITY) ? 0.0f : __expf(li - l);
  };
  if (npc <= 2) {
    // one or two pieces: both fetched before the weights are known
    f32x4 v0[PER], v1[PER];
    piece(0, v0);
    if (npc > 1) piece(1, v1);
    const float l0 = plse(0);
    const float l1 = npc > 1 ? plse(1) : -INFINITY;
    const float s0 = pinv(0);
    const float s1 = npc > 1 ? pinv(1) : 1.0f;
    float mx = fmaxf(sink, l0);
    if (npc > 1) mx = fmaxf(mx, l1);
    if (mx != -INFINITY) {  // else no key and no sink: lse -inf, every weight 0
      float tot = __expf(sink - mx) + __expf(l0 - mx);
      if (npc > 1) tot += __expf(l1 - mx);
      l = mx + __logf(tot);
    }
    const float w0 = weight(l0) * s0;  // the piece's inverse scale is a power of two
#pragma unroll
    for (int k = 0; k < PER; ++k)
      o[k] = (f32x4){w0 * v0[k][0], w0 * v0[k][1], w0 * v0[k][2], w0 * v0[k][3]};
    if (npc > 1) {
      const float w1 = weight(l1) * s1;
#pragma unroll
      for (int k = 0; k < PER; ++k)
#pragma unroll
        for (int e = 0; e < 4; ++e) o[k][e] = __builtin_fmaf(w1, v1[k][e], o[k][e]);
    }
  } else {
    // more pieces: their data in batches of PB with all loads of a batch in
    // flight together, the first MAXL lse values in one batch (a loop of one
    // piece per round trip costs a memory latency per piece)
    constexpr int PB = 4;
    constexpr int MAXL = 16;
    f32x4 vb[PB][PER];
    float sb[PB];
#pragma unroll
    for (int i = 0; i < PB; ++i) {
      piece(i < npc ? i : npc - 1, vb[i]);
      sb[i] = pinv(i < npc ? i : npc - 1);
    }
    float lv[MAXL];
#pragma unroll
    for (int i = 0; i < MAXL; ++i) lv[i] = plse(i < npc ? i : npc - 1);
    auto lse_of = [&](int i) -> float { return i < MAXL ? lv[i] : plse(i); };
    float mx = fmaxf(sink, lv[0]);
#pragma unroll
    for (int i = 1; i < MAXL; ++i)
      if (i < npc) mx = fmaxf(mx, lv[i]);
    for (int i = MAXL; i < npc; ++i) mx = fmaxf(mx, plse(i));
    if (mx != -INFINITY) {
      float tot = __expf(sink - mx) + __expf(lv[0] - mx);
#pragma unroll
      for (int i = 1; i < MAXL; ++i)
        if (i < npc) tot += __expf(lv[i] - mx);
      for (int i = MAXL; i < npc; ++i) tot += __expf(plse(i) - mx);
      l = mx + __logf(tot);
    }
    for (int i0 = 0; i0 < npc; i0 += PB) {
      if (i0 > 0) {
#pragma unroll
        for (int i = 0; i < PB; ++i) {
          piece(i0 + i < npc ? i0 + i : npc - 1, vb[i]);
          sb[i] = pinv(i0 + i < npc ? i0 + i : npc - 1);
        }
      }
#pragma unroll
      for (int i = 0; i < PB; ++i) {
        if (i0 + i >= npc) break;
        const float wi = weight(lse_of(i0 + i)) * sb[i];
#pragma unroll
        for (int k = 0; k < PER; ++k) {
          if (i0 + i == 0) {
            o[k] = (f32x4){wi * vb[i][k][0], wi * vb[i][k][1], wi * vb[i][k][2], wi * vb[i][k][3]};
          } else {
#pragma unroll
            for (int e = 0; e < 4; ++e) o[k][e] = __builtin_fmaf(wi, vb[i][k][e], o[k][e]);
          }
        }
      }
    }
  }
  if (!store || tok < 0 || tok >= a.total_tokens) return;
  T* orow = (T*)a.out + ((size_t)tok * a.num_heads + h) * DV + 8 * c0;
#pragma unroll
  for (int k = 0; k < PER / 2; ++k) {
    const i16x8 pk = {MfmaOps<T>::from_f32(o[2 * k][0]), MfmaOps<T>::from_f32(o[2 * k][1]),
                      MfmaOps<T>::from_f32(o[2 * k][2]), MfmaOps<T>::from_f32(o[2 * k][3]),
                      MfmaOps<T>::from_f32(o[2 * k + 1][0]), MfmaOps<T>::from_f32(o[2 * k + 1][1]),
                      MfmaOps<T>::from_f32(o[2 * k + 1][2]), MfmaOps<T>::from_f32(o[2 * k + 1][3])};
    *(i16x8*)(orow + 8 * TPH * k) = pk;
  }
  if (c0 == 0) a.lse[(size_t)tok * a.num_heads + h] = l;
}

// Tasks t = blockIdx.x, + gridDim.x, ... (one per workgroup column when the grid
// matches the task count; device-built schedules launch for the capacity).
template <int DV, typename T>
__global__ __launch_bounds__(MERGE_THREADS) void merge_kernel(const SasAttnArgs a) {
  int nfd = a.num_fd;
  if (nfd == SAS_SCHED_DEVICE) {
    if (!dev_sched_ok(a, a.m_base)) return;  // the attention kernel wrote NaN
    nfd = a.metadata[SAS_CFG_OFFSET + 3];
  }
  // Tasks in eight slices: column bx runs on XCD bx % 8 (workgroups go round-
  // robin over the 8 XCDs and the grid width is a multiple of 8) and takes the
  // tasks of slice bx % 8. The attention kernel keeps consecutive FA rows on
  // one XCD, so an evenly spread schedule leaves each slice's partials in that
  // XCD's L2.
  const int per = (nfd + 7) >> 3;
  const int cols = (int)gridDim.x >> 3;
  const int x = (int)blockIdx.x & 7;
  for (int j = (int)blockIdx.x >> 3; j < per; j += cols) {
    const int t = x * per + j;
    if (t < nfd) merge_task<DV, T>(a, t);
  }
}

// Launches whose sequences hold several query rows run two consecutive rows of
// 64 heads per workgroup on the 128-head kernel when each row attends a window
// and / or a dense compressed prefix: the two rows' lists then overlap in all but
// a position or two, so one gathered tile serves both (pieces of split items run
// alone). The rule reads only what a host- and a device-built schedule's launch
// both know, so both run the same kernel.
static bool row_pairs_ok(const SasAttnArgs& a) {
  return !(a.phases & SAS_PHASE_ROW_ITEMS) && a.kv_format == SAS_KV_NATIVE &&
         a.scenario <= 2 && a.num_heads <= 64 && a.m_base == 64 && a.total_tokens > a.batch;
}

template <int DQK, int NHG, typename T, int KVF>
static hipError_t launch_attn(const SasAttnArgs& args, hipStream_t st) {
  KernelArgs a;
  (SasAttnArgs&)a = args;
  a.ori_bs = FastDiv::of(a.ori_block_size);
  a.cmp_bs = a.scenario >= 2 ? FastDiv::of(a.cmp_block_size) : a.ori_bs;
  a.ratio = a.scenario >= 2 ? FastDiv::of(a.cmp_ratio) : a.ori_bs;
  const int phases = (a.phases & 3) == 0 ? 3 : (a.phases & 3);
  if (phases & 1) {
    const int per_xcd = (a.num_fa + 7) / 8;
    // native rows: one wave per SIMD (attn2_kernel); fp8 rows: the pipelined
    // two-waves-per-SIMD kernel, whose second wave hides the dequantization
    if constexpr (KVF == SAS_KV_FP8_DS_MLA && NHG == 4) {
      // 128-head items of fp8 rows: the 128-head kernel, dequantizing a raw ring
      if (a.phases & SAS_PHASE_FP8_QK)
        hipLaunchKernelGGL((wide_kernel<DQK, 512, T, KVF, false, true>), dim3(8 * per_xcd),
                           dim3(512), 0, st, a);
      else
        hipLaunchKernelGGL((wide_kernel<DQK, 512, T, KVF>), dim3(8 * per_xcd), dim3(512), 0, st, a);
    } else if constexpr (KVF == SAS_KV_FP8_DS_MLA) {
      if (a.phases & SAS_PHASE_FP8_QK)
        hipLaunchKernelGGL((attn3_kernel<DQK, 512, NHG, T, KVF, true>), dim3(8 * per_xcd),
                           dim3(256 * NHG), 0, st, a);
      else
        hipLaunchKernelGGL((attn3_kernel<DQK, 512, NHG, T, KVF>), dim3(8 * per_xcd),
                           dim3(256 * NHG), 0, st, a);
    } else if constexpr (NHG == 4) {
      // 128-head items: one workgroup of 8 waves holds every head of the token
      hipLaunchKernelGGL((wide_kernel<DQK, 512, T>), dim3(8 * per_xcd), dim3(512), 0, st, a);
    } else {
      if (a.phases & SAS_PHASE_PIPELINED)
        hipLaunchKernelGGL((attn3_kernel<DQK, 512, NHG, T, KVF>), dim3(8 * per_xcd),
                           dim3(256 * NHG), 0, st, a);
      else if (NHG == 2 && row_pairs_ok(a))  // two query rows of 64 heads per workgroup
        hipLaunchKernelGGL((wide_kernel<DQK, 512, T, SAS_KV_NATIVE, true>), dim3(8 * per_xcd),
                           dim3(512), 0, st, a);
      else if (a.total_tokens > a.batch)  // some batch holds several query rows
        hipLaunchKernelGGL((attn2_kernel<DQK, 512, NHG, T, KVF, true>), dim3(8 * per_xcd),
                           dim3(128 * NHG), 0, st, a);
      else
        hipLaunchKernelGGL((attn2_kernel<DQK, 512, NHG, T, KVF, false>), dim3(8 * per_xcd),
                           dim3(128 * NHG), 0, st, a);
    }
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
  }
  const bool dev = a.num_fd == SAS_SCHED_DEVICE;
  // the 128-head kernel and the native-row one-wave-per-SIMD kernel merge split
  // items themselves when given arrival counters
  const bool merged_in_attn =
      (NHG == 4 || (KVF == SAS_KV_NATIVE && !(a.phases & SAS_PHASE_PIPELINED))) &&
      a.merge_sync != nullptr && a.workspace != nullptr;
  if ((phases & 2) && (a.num_fd > 0 || dev) && !merged_in_attn) {
    const int groups = (a.m_base + MERGE_HPB - 1) / MERGE_HPB;  // head groups per task (upper bound)
    const int tasks = dev ? (a.num_fa < 256 ? a.num_fa : 256) : a.num_fd;  // columns; tasks strided
    const int cols = (tasks + 7) / 8 * 8;  // a multiple of the 8 XCDs
    hipLaunchKernelGGL((merge_kernel<512, T>), dim3(cols, groups), dim3(MERGE_THREADS), 0, st, args);
    return hipGetLastError();
  }
  return hipSuccess;
}

// Items carry m_base = 32 or 64 heads (one or two 32-head groups: attn2_kernel,
// 2 or 4 waves, one per SIMD) or 128 heads (wide_kernel, 8 waves, two per SIMD).
template <typename T>
static hipError_t dispatch_heads(const SasAttnArgs& a, hipStream_t st) {
  constexpr int NAT = SAS_KV_NATIVE;
  if (a.head_dim == 576)
    return a.m_base == 32   ? launch_attn<576, 1, T, NAT>(a, st)
           : a.m_base == 64 ? launch_attn<576, 2, T, NAT>(a, st)
                            : launch_attn<576, 4, T, NAT>(a, st);
  return a.m_base == 32   ? launch_attn<512, 1, T, NAT>(a, st)
         : a.m_base == 64 ? launch_attn<512, 2, T, NAT>(a, st)
                          : launch_attn<512, 4, T, NAT>(a, st);
}

// fp8 rows: head_dim 576, bf16 queries and outputs
static hipError_t dispatch_fp8(const SasAttnArgs& a, hipStream_t st) {
  constexpr int F8 = SAS_KV_FP8_DS_MLA;
  return a.m_base == 32   ? launch_attn<576, 1, __bf16, F8>(a, st)
         : a.m_base == 64 ? launch_attn<576, 2, __bf16, F8>(a, st)
                          : launch_attn<576, 4, __bf16, F8>(a, st);
}

}  // namespace sas

extern "C" int sas_attention_launch(const SasAttnArgs* a, void* stream) {
  return sas_attention_launch_lens(a, SAS_QLENS_ARRAYS, stream);
}

extern "C" int sas_attention_launch_lens(const SasAttnArgs* args, int q_lens, void* stream) {
  using sas::set_error;
  if (!args) {
    set_error("sas_attention_launch: null args");
    return SAS_E_INVALID;
  }
  if (q_lens < SAS_QLENS_ARRAYS || q_lens > SAS_QLENS_UNIFORM) {
    set_error("sas_attention_launch_lens: unknown form of the query row counts");
    return SAS_E_INVALID;
  }
  if (!args->q || !args->ori_kv || !args->ori_block_table ||
      (q_lens != SAS_QLENS_UNIFORM && !args->q_prefix) ||
      (q_lens == SAS_QLENS_ARRAYS && !args->act_q_lens) ||
      !args->seqused_kv || !args->sinks || !args->metadata || !args->out || !args->lse) {
    set_error("sas_attention_launch: null tensor pointer");
    return SAS_E_INVALID;
  }
  if (q_lens == SAS_QLENS_UNIFORM && args->batch > 0 && args->total_tokens % args->batch != 0) {
    set_error("sas_attention_launch_lens: total_tokens must be a multiple of batch");
    return SAS_E_INVALID;
  }
  // the kernels tell the forms apart by the null pointers (QRows)
  SasAttnArgs form = *args;
  if (q_lens != SAS_QLENS_ARRAYS) form.act_q_lens = nullptr;
  if (q_lens == SAS_QLENS_UNIFORM) form.q_prefix = nullptr;
  const SasAttnArgs* const a = &form;
  if (a->head_dim != 512 && a->head_dim != 576) {
    set_error("sas_attention_launch: head_dim must be 512 or 576");
    return SAS_E_UNSUPPORTED;
  }
  if (a->head_dim_v != 512) {
    set_error("sas_attention_launch: head_dim_v must be 512");
    return SAS_E_UNSUPPORTED;
  }
  if (a->num_heads < 1 || a->num_heads > 128 || (a->num_heads % 16) != 0) {
    set_error("sas_attention_launch: num_heads must be a multiple of 16 in [16, 128]");
    return SAS_E_UNSUPPORTED;
  }
  // heads per item: 32 up to 32 heads, 64 up to 64 heads, above that 128 (one item
  // holds the token's every head: the 128-head kernel) or 64; 64 only for native
  // rows run through the pipelined kernel (SAS_PHASE_PIPELINED)
  const bool item64 = (a->phases & SAS_PHASE_PIPELINED) != 0;
  const int want_mb = a->num_heads <= 32 ? 32 : (a->num_heads <= 64 || item64) ? 64 : 128;
  // above 64 heads items may also hold 64 heads (two per token)
  if (a->m_base != want_mb && !(want_mb == 128 && a->m_base == 64)) {
    set_error("sas_attention_launch: m_base must be 32 for <= 32 heads, 64 for <= 64 heads "
              "(or SAS_PHASE_PIPELINED), else 128 or 64");
    return SAS_E_INVALID;
  }
  if (a->scenario < 1 || a->scenario > 3 || (a->scenario >= 2 && (!a->cmp_kv ||
      !a->cmp_block_table || a->cmp_ratio < 1)) || (a->scenario == 3 && (!a->cmp_indices ||
      a->topk < 0))) {
    set_error("sas_attention_launch: scenario inputs missing");
    return SAS_E_INVALID;
  }
  if (a->phases < 0 || a->phases > 31) {
    set_error("sas_attention_launch: phases must be 0..31");
    return SAS_E_INVALID;
  }
  if ((a->phases & SAS_PHASE_FP8_QK) && a->kv_format != SAS_KV_FP8_DS_MLA) {
    set_error("sas_attention_launch: SAS_PHASE_FP8_QK needs fp8 cache rows (SAS_KV_FP8_DS_MLA)");
    return SAS_E_INVALID;
  }
  const bool dev_sched = a->num_fd == SAS_SCHED_DEVICE;
  if (a->num_fa < 1 || a->num_fa > SAS_AIC_CORE_NUM || (a->num_fd < 0 && !dev_sched) ||
      a->num_fd > SAS_AIV_CORE_NUM || a->s2_base < 32 || (a->s2_base % 32) != 0 ||
      ((a->num_fd > 0 || dev_sched) && (!a->workspace || a->num_partial_slots < 1))) {
    set_error("sas_attention_launch: inconsistent schedule");
    return SAS_E_INVALID;
  }
  if (a->merge_sync && (((uintptr_t)a->merge_sync & 7) != 0 ||
                        a->num_partial_slots > SAS_MERGE_SYNC_WORDS)) {
    set_error("sas_attention_launch: merge_sync must be 8-byte aligned and the schedule "
              "within SAS_MERGE_SYNC_WORDS partial slots");
    return SAS_E_INVALID;
  }
  if (a->ori_block_num < 1 || a->ori_block_size < 1 || a->ori_table_len < 1 || a->batch < 0 ||
      a->total_tokens < 0 || (a->scenario >= 2 && (a->cmp_block_num < 1 ||
      a->cmp_block_size < 1 || a->cmp_table_len < 1))) {
    set_error("sas_attention_launch: bad cache geometry");
    return SAS_E_INVALID;
  }
  if ((int64_t)a->ori_block_num * a->ori_block_size >= (1ll << 31) ||
      (int64_t)a->cmp_block_num * a->cmp_block_size >= (1ll << 31)) {
    set_error("sas_attention_launch: more than 2^31 cache rows");
    return SAS_E_UNSUPPORTED;
  }
  if (a->kv_format != SAS_KV_NATIVE && a->kv_format != SAS_KV_FP8_DS_MLA) {
    set_error("sas_attention_launch: unknown kv_format");
    return SAS_E_INVALID;
  }
  if (a->kv_format == SAS_KV_FP8_DS_MLA && (a->head_dim != 576 || a->dtype != SAS_DTYPE_BF16)) {
    set_error("sas_attention_launch: fp8 cache rows need head_dim 576 and bf16 queries");
    return SAS_E_UNSUPPORTED;
  }
  if (a->batch == 0 || a->total_tokens == 0) return SAS_OK;
  hipStream_t st = (hipStream_t)stream;
  hipError_t e = a->kv_format == SAS_KV_FP8_DS_MLA ? sas::dispatch_fp8(*a, st)
                 : a->dtype == SAS_DTYPE_FP16      ? sas::dispatch_heads<_Float16>(*a, st)
                                                   : sas::dispatch_heads<__bf16>(*a, st);
  if (e != hipSuccess) {
    set_error(std::string("sas_attention_launch: ") + hipGetErrorString(e));
    return SAS_E_HIP;
  }
  return SAS_OK;
}

// ---------------------------------------------------------------------------
// Allocation-free launch: the split-KV partials go to a fixed device array
// ---------------------------------------------------------------------------
namespace sas {
// One copy per device (the runtime places it when the library's code object is
// loaded; each device keeps it until the process ends). In host code `scratch`
// names a host-side stand-in: only the address from hipGetSymbolAddress, taken
// once per device with that device current, is passed to kernels.
__device__ __attribute__((aligned(256))) float scratch[SAS_NOALLOC_SCRATCH_BYTES / sizeof(float)];
constexpr int MAX_DEVICES = 64;
static float* g_scratch_ptr[MAX_DEVICES];
static std::mutex g_scratch_mu;

// Address of this device's scratch array (resolved on the first call per device).
static int scratch_ptr(float** out) {
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) {
    set_error(std::string("sas_attention_launch_noalloc: hipGetDevice: ") + hipGetErrorString(e));
    return SAS_E_HIP;
  }
  if (dev < 0 || dev >= MAX_DEVICES) {
    set_error("sas_attention_launch_noalloc: device index out of range");
    return SAS_E_UNSUPPORTED;
  }
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  if (!g_scratch_ptr[dev]) {
    void* p = nullptr;
    e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !p) {
      set_error(std::string("sas_attention_launch_noalloc: hipGetSymbolAddress: ") +
                hipGetErrorString(e));
      return SAS_E_HIP;
    }
    g_scratch_ptr[dev] = (float*)p;
  }
  *out = g_scratch_ptr[dev];
  return SAS_OK;
}
}  // namespace sas

extern "C" int sas_attention_launch_noalloc(const SasAttnArgs* a, void* stream) {
  if (!a) {
    sas::set_error("sas_attention_launch_noalloc: null args");
    return SAS_E_INVALID;
  }
  // the last SAS_MERGE_SYNC_WORDS words of the scratch array hold the in-kernel
  // merge's arrival counters (zero when the library is loaded, zero after each call)
  constexpr int64_t SYNC_BYTES = (int64_t)SAS_MERGE_SYNC_WORDS * 8;
  const int64_t need = sas_workspace_bytes(a->num_partial_slots, a->m_base, a->head_dim_v);
  if (need > (int64_t)SAS_NOALLOC_SCRATCH_BYTES - SYNC_BYTES) {
    sas::set_error("sas_attention_launch_noalloc: the schedule's split-KV workspace (" +
                   std::to_string(need) + " bytes for " + std::to_string(a->num_partial_slots) +
                   " partial slots) exceeds the fixed scratch of " +
                   std::to_string((long long)(SAS_NOALLOC_SCRATCH_BYTES - SYNC_BYTES)) + " bytes");
    return SAS_E_CAPACITY;
  }
  float* ws = nullptr;
  const int rc = sas::scratch_ptr(&ws);
  if (rc != SAS_OK) return rc;
  SasAttnArgs b = *a;
  b.workspace = ws;  // the caller's workspace pointer, if any, is not used
  // a non-null merge_sync asks for the in-kernel merge; its counters are the scratch's
  b.merge_sync = a->merge_sync
                     ? (uint64_t*)((char*)ws + SAS_NOALLOC_SCRATCH_BYTES - SYNC_BYTES)
                     : nullptr;
  return sas_attention_launch(&b, stream);
}

// ---------------------------------------------------------------------------
// Arrival counters for captured calls
// ---------------------------------------------------------------------------
namespace sas {
// Zero when the code object is loaded and zero again after every call that used
// them, so a graph that owns an array needs no fill in front of its kernels (a
// fill of 8 KB delayed each replay's attention by about 4.5 us).
__device__ unsigned long long g_sync_pool[SAS_MERGE_SYNC_POOL][SAS_MERGE_SYNC_WORDS];
struct SyncPool {
  char* base = nullptr;
  int used = 0;
  unsigned long long capture = 0;  // the capture and stream that took the last array
  hipStream_t stream = nullptr;
};
static SyncPool g_sync[MAX_DEVICES];
static std::mutex g_sync_mu;
}  // namespace sas

extern "C" uint64_t* sas_merge_sync_take(void* stream) {
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= sas::MAX_DEVICES) return nullptr;
  hipStreamCaptureStatus status = hipStreamCaptureStatusNone;
  unsigned long long capture = 0;
  if (hipStreamGetCaptureInfo((hipStream_t)stream, &status, &capture) != hipSuccess ||
      status != hipStreamCaptureStatusActive) {
    sas::set_error("sas_merge_sync_take: the stream is not capturing");
    return nullptr;
  }
  std::lock_guard<std::mutex> lock(sas::g_sync_mu);
  sas::SyncPool& p = sas::g_sync[dev];
  if (!p.base) {
    void* at = nullptr;
    if (hipGetSymbolAddress(&at, HIP_SYMBOL(sas::g_sync_pool)) != hipSuccess || !at) {
      sas::set_error("sas_merge_sync_take: hipGetSymbolAddress failed");
      return nullptr;
    }
    p.base = (char*)at;
  }
  // calls of one capture on one stream run one after another, so they may share an
  // array; those taken in turn with another stream's take more than one
  if (p.used == 0 || p.capture != capture || p.stream != (hipStream_t)stream) {
    if (p.used == SAS_MERGE_SYNC_POOL) {
      sas::set_error("sas_merge_sync_take: every array is taken");
      return nullptr;
    }
    ++p.used;
    p.capture = capture;
    p.stream = (hipStream_t)stream;
  }
  return (uint64_t*)(p.base + (size_t)(p.used - 1) * SAS_MERGE_SYNC_WORDS * 8);
}

extern "C" int sas_version(void) { return 115; }

extern "C" int sas_args_struct_size(void) { return (int)sizeof(SasAttnArgs); }

extern "C" const char* sas_last_error(void) { return sas::g_last_error.c_str(); }
