// attn_kernels.hip -- gfx950 (CDNA4) kernels for the bf16 flash-attention forward.
//
// Semantics follow the reference's attn_flash (liujiang833/transfer_station flash.c:727-864):
// kv = h / (Hq/Hkv) (flash.c:765,780); scores scale*Q.K with scale = 1/sqrtf(D) (flash.c:766);
// bottom-right causal mask j <= Sk-Sq+i (flash.c:783,535-543); online softmax per key block with
// alpha = exp(m_old - m_new), 0 on a row's first contributing block, state held on a fully
// masked block (flash.c:546-559); P rounded RNE to bf16 before P.V while l sums the unrounded
// fp32 p (flash.c:566-576); O = acc * (l > 0 ? 1/l : 0) for every row (flash.c:851-860).
// The implementation is this file's own: MFMA tiles, LDS staging and register-resident softmax.
//
// Exponentials run in the log2 domain: with c = scale*log2(e) and scores kept as raw dot
// products s, p = 2^(s*c - m*c) equals e^(scale*s - scale*m).
//
// Kernels:
//   attn_prefill_fast_kernel<DP,KT,NW,CAUSAL,VT,KH,UA>  MFMA prefill, D <= DP in {64, 96, 128,
//                                          192, 256}; one workgroup = NW waves x 32 rows, or (KH) 8
//                                          waves over 128 rows on key-tile halves; UA: tensors
//                                          without the 16-byte vector layout
//   attn_prefill_persist_kernel<DP,CAUSAL,KH> the same tile code at D <= 128, one 8-wave
//                                          workgroup per CU running its 256-row items back to
//                                          back (causal: pairs of a heavy and a light query
//                                          tile), or (KH) one causal pair of 128-row items on
//                                          key-tile halves
//   attn_decode_kernel<DP,CAUSAL,AL,VT,NTL,NRB> split-K decode for g*Sq <= 64 rows per kv head
//   attn_decode_vt_kernel<DP,CAUSAL,NTL,UA> the same from V^T, staged in LDS 512 keys at a time
//   attn_merge{2,w,}_kernel                log-sum-exp merge of split partials (2 splits / up to
//                                          64 / any, one workgroup per row)
//   attn_pack_v16_kernel<TK,VEC>           V [Hkv][Sk][D] -> V^T [Hkv][D][Sk]
// VT selects a pre-transposed V ([Hkv][D][Sk], pack_v_full's layout).
#include <hip/hip_runtime.h>
#include <stdarg.h>
#include <stdint.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>

#include <algorithm>
#include <atomic>
#include <type_traits>
#include <utility>

#include "attn_decode_rule.h"
#include "attn_flash.h"

namespace {

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(4))) short s16x4;
typedef __attribute__((ext_vector_type(16))) float f32x16;
typedef __attribute__((ext_vector_type(4))) float f32x4;
typedef __attribute__((ext_vector_type(4))) uint32_t u32x4;
typedef __attribute__((address_space(3))) s16x4 lds_s16x4;

constexpr float kNegInf = -__builtin_inff();

// Workgroup and work-item ids read straight from their registers. HIP's blockIdx / threadIdx /
// gridDim go through device-library functions that are built with IEEE mode on; this library
// is built with it off (-mno-amdgpu-ieee), so the compiler will not inline them, and each use
// would be an out-of-line call in the kernel's prologue. The workgroup count comes from the
// kernel's own arguments instead: reading the grid size from the dispatch packet
// (__builtin_amdgcn_grid_size_x) in every workgroup's prologue measured 2-22% slower.
// The two kernels that stage tiles by LDS-DMA (the fast prefill and the V^T decode) still take
// threadIdx.x, and with it one such call, on purpose. In a kernel without any call this
// compiler makes each LDS read of a tile wait (vmcnt) for the DMA of the next tile into the
// other buffer, which it cannot tell apart from this one: measured 3-15% slower on the prefill
// shapes. With the call it leaves that ordering to the kernel, which does it itself (each wave
// waits for its own DMA, vmcnt(0), before the barrier that ends a tile).
__device__ __forceinline__ int wg_id_x() { return (int)__builtin_amdgcn_workgroup_id_x(); }
__device__ __forceinline__ int wg_id_y() { return (int)__builtin_amdgcn_workgroup_id_y(); }
__device__ __forceinline__ int wg_id_z() { return (int)__builtin_amdgcn_workgroup_id_z(); }
__device__ __forceinline__ int wi_id_x() { return (int)__builtin_amdgcn_workitem_id_x(); }

// Workgroups are dispatched round-robin over the 8 XCDs (each with its own L2). Remap the
// hardware block id so that consecutive logical ids land on the same XCD: logical ids that
// share a kv head then share that XCD's L2 copy of K/V.
__device__ __forceinline__ int xcd_remap(int b, int n) {
    const int per = n >> 3, rem = n & 7;
    const int x = b & 7, i = b >> 3;
    return (x < rem) ? x * (per + 1) + i : rem * (per + 1) + (x - rem) * per + i;
}

// xcd_remap for a grid resident all at once at two workgroups per CU (n <= 2 * CUs). Each
// XCD hands its blocks to its R CUs in order, one slot per CU first, so XCD positions i and
// i + R share a CU (measured with a HW_ID probe: blocks b and b + 256 on MI355X). Reversing
// positions [R, n_x) pairs the first round's heaviest item with the second round's lightest,
// when the logical order is heaviest first. R = 0 gives xcd_remap.
__device__ __forceinline__ int xcd_remap_paired(int b, int n, int R) {
    const int per = n >> 3, rem = n & 7;
    const int x = b & 7, nx = (x < rem) ? per + 1 : per;
    int i = b >> 3;
    if (R > 0 && i >= R)
        i = R + (nx - 1 - i);
    return (x < rem) ? x * (per + 1) + i : rem * (per + 1) + (x - rem) * per + i;
}

// f(std::integral_constant<int, 0>{}), ..., f(std::integral_constant<int, N-1>{}): an unrolled loop
// whose index is a constant expression (needed for sched_group_barrier counts).
template <typename F, int... I>
__device__ __forceinline__ void static_for_impl(F &&f, std::integer_sequence<int, I...>) {
    (f(std::integral_constant<int, I>{}), ...);
}
template <int N, typename F> __device__ __forceinline__ void static_for(F &&f) {
    static_for_impl(f, std::make_integer_sequence<int, N>{});
}

__device__ __forceinline__ u32x4 zero4() {
    u32x4 z = {0u, 0u, 0u, 0u};
    return z;
}

// Unaligned vectors: gfx950 serves 16-byte global accesses at any element alignment, so tensors
// whose rows are not 16-byte aligned are read 16 bytes at a time too (element-wise loads, eight
// 2-byte loads and their packing per chunk, made such calls 6-15x slower). O is fp32: 4-aligned.
typedef u32x4 __attribute__((aligned(2))) u32x4_a2;
typedef f32x4 __attribute__((aligned(4))) f32x4_a4;

template <bool NT> __device__ __forceinline__ u32x4 load16_any(const uint16_t *p) {
    return NT ? __builtin_nontemporal_load(reinterpret_cast<const u32x4_a2 *>(p))
              : *reinterpret_cast<const u32x4_a2 *>(p);
}

// x as a value that the compiler takes for new here: what follows from it is computed where it is
// used, not hoisted out of the key loop and spilled.
__device__ __forceinline__ uint32_t opaque(uint32_t x) {
    asm volatile("" : "+v"(x));
    return x;
}

// v without its first n (0..8) of eight 16-bit elements, zeros behind.
__device__ __forceinline__ u32x4 drop_elems(u32x4 v, int n) {
    const int h = (n & 1) * 16;
    const bool n2 = n & 2, n4 = n & 4, n8 = n & 8;
    const uint32_t a0 = __builtin_amdgcn_alignbit(v[1], v[0], h);
    const uint32_t a1 = __builtin_amdgcn_alignbit(v[2], v[1], h);
    const uint32_t a2 = __builtin_amdgcn_alignbit(v[3], v[2], h), a3 = v[3] >> h;
    const uint32_t b0 = n2 ? a1 : a0, b1 = n2 ? a2 : a1, b2 = n2 ? a3 : a2, b3 = n2 ? 0u : a3;
    return u32x4{n8 ? 0u : n4 ? b2 : b0, n8 ? 0u : n4 ? b3 : b1, n4 || n8 ? 0u : b2,
                 n4 || n8 ? 0u : b3};
}

// Elements [i, i+8) of the n-element row at p one by one, zero-filled past n: rows of fewer than
// eight elements. load_rolled does it in a loop: code that hardly any call reaches.
__device__ __forceinline__ u32x4 load_short(const uint16_t *p, int i, int n) {
    if (i >= n)
        return zero4();
    uint32_t e[8];
#pragma unroll
    for (int j = 0; j < 8; ++j)
        e[j] = i + j < n ? (uint32_t)p[i + j] : 0u;
    return u32x4{e[0] | (e[1] << 16), e[2] | (e[3] << 16), e[4] | (e[5] << 16), e[6] | (e[7] << 16)};
}

__device__ __forceinline__ u32x4 load_rolled(const uint16_t *p, int i, int n) {
    u32x4 v = zero4();
#pragma unroll 1
    for (int j = min(n, i + 8) - 1; j >= i; --j)
        v = u32x4{(v[0] << 16) | p[j], __builtin_amdgcn_alignbit(v[1], v[0], 16),
                  __builtin_amdgcn_alignbit(v[2], v[1], 16),
                  __builtin_amdgcn_alignbit(v[3], v[2], 16)};
    return v;
}

// The first m (1..7) of eight 16-bit elements, zeros behind.
__device__ __forceinline__ u32x4 keep_elems(u32x4 v, int m) {
    auto w = [&](uint32_t x, int j) {
        return m >= 2 * j + 2 ? x : m == 2 * j + 1 ? x & 0xffffu : 0u;
    };
    return u32x4{w(v[0], 0), w(v[1], 1), w(v[2], 2), w(v[3], 3)};
}

// Elements [i, i+8) of the n-element row at p (n >= 8), at any alignment and without a read outside
// the row, in two steps: load_piece reads a piece that reaches past the row's end as its last
// eight elements, and trim_piece shifts it where it is used, zeros behind (a shift at the load
// would wait for it before the next piece's load is issued). Pieces past the end are zeros. ie
// (wave-uniform) bounds the elements of the wave's lanes.
template <bool NT = false>
__device__ __forceinline__ u32x4 load_piece(const uint16_t *p, int i, int n, int ie) {
    if (i >= n)
        return zero4();
    if ((n & 7) != 0 && ie > n)
        return load16_any<NT>(p + min(i, n - 8));
    return load16_any<NT>(p + i);
}

__device__ __forceinline__ u32x4 trim_piece(u32x4 v, int i, int n, int ie) {
    return (n & 7) != 0 && ie > n ? drop_elems(v, (int)opaque(min(max(i + 8 - n, 0), 8))) : v;
}

// Aligned tensors: eight consecutive bf16 of one row, columns [col, col+8), zero-filled past D or
// when !ok. D % 8 == 0 and a 16-byte aligned base, so one 16-byte load covers them.
// NT marks the load non-temporal (data read once: HBM streams such loads ≈ 15% faster).
template <bool NT = false>
__device__ __forceinline__ u32x4 load_row8(const uint16_t *base, size_t row, int col, int D,
                                           bool ok) {
    if (!ok || col >= D)
        return zero4();
    const uint16_t *p = base + row * (size_t)D + col;
    return NT ? __builtin_nontemporal_load(reinterpret_cast<const u32x4 *>(p))
              : *reinterpret_cast<const u32x4 *>(p);
}

// Aligned tensors: eight consecutive keys [key, key+8) of row d of a V^T head ([D][Sk], row stride
// Sk), zero-filled at d >= D or key >= klim. Sk % 8 == 0 and a 16-byte aligned base (with
// key % 8 == 0 and klim % 8 == 0 a chunk is then wholly inside or wholly outside).
template <bool NT = false>
__device__ __forceinline__ u32x4 load_vt8(const uint16_t *base, int d, int key, int Sk, int D,
                                          int klim) {
    if (d >= D || key >= klim)
        return zero4();
    const uint16_t *p = base + (size_t)d * Sk + key;
    return NT ? __builtin_nontemporal_load(reinterpret_cast<const u32x4 *>(p))
              : *reinterpret_cast<const u32x4 *>(p);
}

__device__ __forceinline__ bf16x8 as_bf16x8(u32x4 v) { return __builtin_bit_cast(bf16x8, v); }

__device__ __forceinline__ bf16x8 join_tr(s16x4 lo, s16x4 hi) {
    typedef __attribute__((ext_vector_type(8))) short s16x8;
    s16x8 r = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
    return __builtin_bit_cast(bf16x8, r);
}

// ds_read_b64_tr_b16: within each 16-lane group, lane i receives element r (r = 0..3) from
// row (4r + i/4) of the group's 16x4 matrix of 8-byte reads, element i%4. Lanes that address
// V[key0 + j/4][d0 + 4*(j%4)] therefore receive V[key0 + r][d0 + i]: four keys for one column.
__device__ __forceinline__ s16x4 lds_read_tr(const uint16_t *p) {
    return __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4 *)(p));
}

__device__ __forceinline__ float fast_exp2(float x) { return __builtin_amdgcn_exp2f(x); }

// max(a, b, c); with IEEE mode off the compiler emits v_max3_f32 or two v_max_f32. No inline
// asm here on purpose: these read MFMA results, and a VALU read of an MFMA result needs wait
// states that the hardware does not enforce; the compiler inserts them only for instructions it
// can see (an asm v_max3 right after the last Q.K^T MFMA read stale scores).
__device__ __forceinline__ float max3f(float a, float b, float c) { return fmaxf(fmaxf(a, b), c); }

// max(x[lane], x[lane ^ 32]), through ds_bpermute (compiler-managed waits). The row max runs on
// an item's first key tile and on rare recomputed tiles only, so the exchange's cost is small.
// Lane exchanges of a value with lane l ^ 16 or l ^ 32 on the VALU (v_permlane16_swap /
// v_permlane32_swap with the value as both operands), where __shfl_xor goes through the LDS
// crossbar and its wait (lgkmcnt) also waits for the wave's LDS reads in flight. Each lane gets
// the pair {its value, its partner's} in one order or the other, so max and sum (commutative)
// give exactly what fmaxf / + with the shuffled value give.
__device__ __forceinline__ float max_xor32(float x) {
    const unsigned u = __builtin_bit_cast(unsigned, x);
    const auto p = __builtin_amdgcn_permlane32_swap(u, u, false, false);
    return fmaxf(__builtin_bit_cast(float, (unsigned)p[0]), __builtin_bit_cast(float, (unsigned)p[1]));
}
__device__ __forceinline__ float sum_xor32(float x) {
    const unsigned u = __builtin_bit_cast(unsigned, x);
    const auto p = __builtin_amdgcn_permlane32_swap(u, u, false, false);
    return __builtin_bit_cast(float, (unsigned)p[0]) + __builtin_bit_cast(float, (unsigned)p[1]);
}
__device__ __forceinline__ float max_xor16(float x) {
    const unsigned u = __builtin_bit_cast(unsigned, x);
    const auto p = __builtin_amdgcn_permlane16_swap(u, u, false, false);
    return fmaxf(__builtin_bit_cast(float, (unsigned)p[0]), __builtin_bit_cast(float, (unsigned)p[1]));
}
__device__ __forceinline__ float sum_xor16(float x) {
    const unsigned u = __builtin_bit_cast(unsigned, x);
    const auto p = __builtin_amdgcn_permlane16_swap(u, u, false, false);
    return __builtin_bit_cast(float, (unsigned)p[0]) + __builtin_bit_cast(float, (unsigned)p[1]);
}

__device__ __forceinline__ void lds_wave_fence() {
    // Wave-private LDS reuse: finish this wave's outstanding LDS traffic and keep the compiler
    // from moving LDS accesses across this point.
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
}

// ------------------------------------------------------------------------------------------
// Prefill, D <= DP (64, 96, 128, 192 or 256); the head-dim columns D .. DP-1 are zero in the tiles and
// in Q, and are never stored. NW waves per workgroup (8: 256 query rows, two waves per SIMD; 4 on
// grids too small to fill the GPU; past DP = 128 4 waves are one per SIMD, which holds O and Q);
// wave w owns 32 query rows. Per key tile of KT keys (one online-softmax update per tile):
//   S^T[key][q] = K_tile . Q^T     (v_mfma_f32_32x32x16_bf16, A = K rows from LDS, B = Q regs)
//   each lane holds one query (q = lane%32) and 16 keys per 32-key sub-tile, so the row max is
//   an in-lane reduction plus one exchange with lane^32;
//   O^T[d][q] += V^T . P^T         (A = V^T via ds_read_b64_tr_b16 from row-major LDS,
//                                    B = P^T straight from the S^T registers)
// The S^T operand rows are permuted (bits 2 and 3 of the row swapped within each 16-row half)
// so that a lane's 8 P values for one 16-key MFMA step are 8 consecutive keys.
// VT: V arrives pre-transposed ([Hkv][D][Sk], pack_v_full's output). The tile is then staged
// d-major (DP rows of KT keys), and the V^T operand of the P.V MFMA is a plain 16-byte LDS read
// of 8 consecutive keys of one d row; the operand values, and so the result, are the same.
//   * UA = 0 (D % 8 == 0, 16-byte aligned tensors, kv heads below 2 GiB; V^T: Sk % 8 == 0):
//   * K/V tiles arrive through raw buffer loads whose range is the kv head's Sk*D*2 bytes, so a
//     key past Sk reads as zero without a branch. The whole byte offset travels in the VGPR
//     offset (the range-checked one); the scalar offset is always 0. They are LDS-DMA loads
//     straight into swizzled LDS tiles (no staging registers or LDS writes).
//   * the next 32-key sub-tile's K fragments are read from LDS between the current sub-tile's
//     MFMAs; the row max is a max3 tree plus a VALU lane exchange (max_xor32).
//   * row max on an item's first tile only: later tiles take p against the running max m and
//     test each lane's tile sum of p against kSumCap instead; a tile that fails is recomputed
//     and takes the row max (softmax_next below). So every p <= kSumCap, m only rises, and the
//     accumulator rescale (alpha != 1) runs only on those rare tiles, decided wave-uniformly.
//     In exact arithmetic the result is identical (softmax is shift-invariant).
//   * at DP = 64 such tiles without a mask are software-pipelined over their 32-key sub-tiles
//     (tile_pipelined below): the exponentials of one sub-tile beside the MFMAs of the next
//     sub-tile's Q.K^T and the previous one's P.V.
//   * causal: work items are dispatched heaviest first; on grids of at most one workgroup per
//     CU the key range of each upper-half query tile is split over two workgroups, which write
//     partials (m, l, acc) for attn_merge2_kernel instead of O.
//   * short query blocks under GQA (pack): the rows of a kv head's g query heads share query
//     tiles, each lane carrying its own head and query index.
//   * grids that do not fill the GPU evenly: a key split over several workgroups (partials
//     merged by attn_mergew_kernel), the slot-balanced head split (D <= 64: whole tiles and key
//     halves placed by XCD position), and key halves inside one workgroup (KH: 8 waves at
//     D >= 64; 12 waves over 192 packed rows at D <= 64, in place of the head split where such
//     workgroups fit one per CU).
// ------------------------------------------------------------------------------------------
// Bound on a lane's tile sum of p = 2^(s c - m c) taken against a stale m (and so on each p).
// 2^16: on peaked rows (config 5's Q ~ N(0, 16)) a cap of 2^8 / 2^12 / 2^16 sends 9.9% / 2.2% /
// 0.13% of wave-tiles to the recompute (CPU count on the benchmark's data); N(0,1) rows never
// reach it. p up to 2^16 costs no precision (fp32 and bf16 are relative), only 16 bits of the
// 128-bit exponent range of the fp32 accumulators.
constexpr float kSumCap = 65536.0f;

// The descriptor must live in scalar registers; its inputs are workgroup-uniform, and the
// readfirstlane makes that explicit so the compiler never falls back to a per-lane loop.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t make_rsrc(const void *base, uint32_t bytes) {
    const uint64_t a = reinterpret_cast<uint64_t>(base);
    const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)a);
    const uint32_t hi = __builtin_amdgcn_readfirstlane((uint32_t)(a >> 32));
    void *p = reinterpret_cast<void *>(((uint64_t)hi << 32) | lo);
    return __builtin_amdgcn_make_buffer_rsrc(p, (short)0, (int)__builtin_amdgcn_readfirstlane(bytes),
                                             0x00020000);
}

// LDS-DMA: 16 bytes per lane from buffer r at byte voff + IMM straight into LDS, lane i writing
// [lds + IMM + 16 i, +16) (the immediate offset moves both addresses; lds must be wave-uniform).
// Bytes past the buffer's range arrive as zero. Completion is counted by vmcnt.
// AUX is the cache policy: 0 ordinary, kDmaNT non-temporal (data read once).
constexpr int kDmaNT = 2;
template <int IMM, int AUX = 0>
__device__ __forceinline__ void dma16(__amdgpu_buffer_rsrc_t r, uint16_t *lds, uint32_t voff) {
    __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (__attribute__((address_space(3))) void *)lds, 16,
                                             voff, 0, IMM, AUX);
}

// Phase stamps of the prefill kernels, compiled in only with ATTN_PHASE_STAMPS=1 (the separate
// libattn_flash_stamps.so that transfer_station_amd/phases.py loads; the product library has
// none of this code). Wave 0 of each workgroup writes the 100 MHz real-time counter (and, in the
// per-tile kernel, its CU and key-tile count) into g_phase_stamps[workgroup][slot]; the slots
// of each kernel are listed where it writes them. Each stamp is one global store of one lane,
// issued where no kernel wait depends on an exact count of outstanding operations (before a
// tile's DMA, or before a full vmcnt(0) wait).
#ifndef ATTN_PHASE_STAMPS
#define ATTN_PHASE_STAMPS 0
#endif
[[maybe_unused]] constexpr int kPhaseSlots = 64;
#if ATTN_PHASE_STAMPS
__device__ unsigned long long *g_phase_stamps;
#endif
__device__ __forceinline__ void phase_value(int w, int lane, int slot, unsigned long long v) {
#if ATTN_PHASE_STAMPS
    if (w == 0 && lane == 0 && slot < kPhaseSlots)
        g_phase_stamps[(size_t)wg_id_x() * kPhaseSlots + slot] = v;
#else
    (void)w, (void)lane, (void)slot, (void)v;
#endif
}
__device__ __forceinline__ void phase_stamp(int w, int lane, int slot) {
#if ATTN_PHASE_STAMPS
    if (w == 0)
        phase_value(w, lane, slot, __builtin_amdgcn_s_memrealtime());
#else
    (void)w, (void)lane, (void)slot;
#endif
}
// The CU a workgroup runs on, as stamp data: XCC_ID above bits 15:8 of HW_ID (CU, SH and SE).
__device__ __forceinline__ unsigned long long phase_cu() {
#if ATTN_PHASE_STAMPS
    const unsigned hw = __builtin_amdgcn_s_getreg((31 << 11) | 4);   // HW_REG_HW_ID
    const unsigned xcc = __builtin_amdgcn_s_getreg((31 << 11) | 20); // HW_REG_XCC_ID
    return ((unsigned long long)(xcc & 15) << 8) | ((hw >> 8) & 0xff);
#else
    return 0;
#endif
}

// Workgroups per CU the launch bounds ask for: 8 waves in all, unless the two K and V tiles
// (8*KT*DP bytes of LDS), the O and Q registers (DP > 128) or the workgroup's own size (12
// waves) allow only one workgroup.
constexpr int prefill_wg_per_cu(int DP, int KT, int NW) {
    return (DP > 128 || 8 * KT * DP > 80 * 1024 || NW > 8) ? 1 : 8 / NW;
}

// KH (key halves, NW = 8): a workgroup of 4 * 32 query rows whose waves w and w + 4 take the
// same rows and the two halves of every key tile (KW = KT / 2 keys each, one wave of each SIMD
// per half), combined through LDS at the end. For grids too small for one 256-row workgroup
// per CU, this keeps two waves per SIMD and 128-key tiles where 4-wave workgroups would take
// 64-key tiles. NW = 12 (DP = 64, non-causal, packed rows): 6 * 32 rows per workgroup, waves
// w and w + 6 on the same rows, three waves per SIMD; one such workgroup per CU holds the
// rows of one and a half 128-row tiles with no partials to merge.
//
// UA = 1 (unaligned): tensors without the vector layout (D % 8 != 0, a base that is not 16-byte
// aligned, V^T rows of an odd key count, or a kv head past a buffer's 31-bit range). The same tiles
// and LDS layouts, but each 16-byte piece goes through registers: loaded at element alignment at the
// start of the tile before, put into LDS at its end. What bounds it is those loads (2-byte aligned
// ones cost 6% more than 4-byte aligned ones, which cost what 16-byte aligned ones do), the registers
// they hold (two pieces per thread and tensor on 64-key tiles at 8 waves; on 4 waves, or K waited
// for in mid-tile, 27-75% slower; D > 128 on 8 waves: kRing below) and the row max, which every tile takes: the largest weights
// of a row are then exactly 1 or close below (error against 64 bits 1.5e-3 of the result, 1.7e-3
// with the sum test, which was 8% faster). Same box, element-wise loads before -> now: 24 heads of
// 1000 rows over 2003 keys, D = 100, V^T with its pack 249 -> 57 us; 64 heads at 2k, D = 128, V^T
// of 2003 keys 950 -> 172 us; D = 100 causal 524 -> 118 us (aligned, D = 128: 126 us non-causal).
// UA = 2: rows shorter than a piece (D < 8), a row per 16-byte load with the rows behind it masked off.
// Against element-wise loads: 128 heads x 20 rows over 1720 keys at D = 7 66 -> 46 us, 8 heads x 317 rows
// over 817 keys 35 -> 26; calls of one tile from V^T stay 0.3-0.8 us above (4.5-7 us).
template <int DP, int KT, int NW, bool CAUSAL, bool VT, bool KH, int UA>
__global__ __launch_bounds__(NW * 64, prefill_wg_per_cu(DP, KT, NW)) void attn_prefill_fast_kernel(
    const uint16_t *__restrict__ Q, const uint16_t *__restrict__ K,
    const uint16_t *__restrict__ V, float *__restrict__ O, int Hq, int Hkv, int Sq, int Sk, int D,
    float c, int nqt, int split_first, float *__restrict__ pm, float *__restrict__ pl,
    float *__restrict__ pacc, int prows, int pack, int pair_r, int pipe, int nsplit, int nwg,
    int hsplit) {
    // D <= DP: head-dim columns D .. DP-1 of the tiles and of Q are zero.
    static_assert(DP % 32 == 0 && KT % 32 == 0, "tile shape");
    static_assert(!KH || (KT == 128 && ((NW == 8 && DP >= 64) || (NW == 12 && DP == 64 && !CAUSAL))),
                  "key halves: 8 waves (or 12 at DP = 64), 128-key tiles");
    static_assert(NW != 12 || KH, "12 waves: key halves only");
    // Software-pipelined tiles (tile_pipelined): D <= 64, key halves on 12 waves only.
    // 8 waves at DP > 128: two waves per SIMD of 256 registers each, 128 (96) of them O and 64 (48)
    // Q, where 4 waves have 512. What made room: K and V fragments go through a ring of RD, read RD
    // MFMAs ahead, instead of a whole sub-tile's and chunk's, and at DP = 256 (and unaligned) a tile is
    // 32 keys; RD is what fits (aligned: no spills; unaligned at 256: 5). One wave's softmax and LDS
    // latency then runs under the other's MFMAs, and a tile is read from L2 for 256 rows. Same
    // box, 4 -> 8 waves, 64 heads at 2k: D = 256 282 -> 232 us (1185 TFLOP/s), causal 160 -> 136, V^T
    // 322 -> 238, D = 192 220 -> 184; unaligned, D = 189 over 2003 keys 530 -> 253, D = 250 at 1000
    // rows 307 -> 154. Neither unit is full (counters at D = 256: MFMA busy 50% of the clocks, no LDS
    // conflicts): a tile's LDS reads take about as long as its MFMAs, and two waves per SIMD, in step
    // through a barrier per tile, overlap them in part.
    constexpr bool kRing = DP > 128 && NW == 8;
    constexpr int RD = !kRing ? 1 : DP < 256 ? 4 : UA ? 2 : VT ? 3 : 4;
    constexpr bool kPipe = DP <= 64 && (!KH || NW == 12) && !UA;
    constexpr int NR = KH ? NW / 2 : NW; // waves with distinct query rows
    constexpr int KW = KH ? KT / 2 : KT; // keys of a tile that one wave takes
    constexpr int BQ = NR * 32;         // query rows per workgroup
    // K and V (or V^T) tiles arrive by LDS-DMA in swizzled, unpadded layouts (below).
    __shared__ __attribute__((aligned(1024))) uint16_t Ks[2][KT * DP];
    __shared__ __attribute__((aligned(1024))) uint16_t Vs[2][KT * DP];
    __shared__ float kh_ml[KH ? 2 * NR * 64 : 1]; // KH: (m, l) of each second-half lane
    // KH: the second halves' o go to the buffer pair the last tile left idle (4 * KT * DP bytes,
    // KT / 32 waves' (DP / 32) * 16 * 64 floats) where they fit, else to an area of their own.
    constexpr int KHO = (KH && NR * DP * 32 * 4 > 4 * KT * DP) ? NR * DP * 32 : 1;
    __shared__ float kh_o[KHO];

    const int g = Hq / Hkv;
    const int L0 = xcd_remap_paired(wg_id_x(), nwg, pair_r); // nwg: the grid's workgroup count
    // Key split of an under-filled grid (nsplit > 1): item L of nit query-tile items, part sp of
    // its key tiles. Logical ids run split-major, so the items of one kv head that read the same
    // key range stay adjacent (one XCD, one L2 copy).
    const int nit = nwg / nsplit;
    const int sp = __builtin_amdgcn_readfirstlane(L0 / nit);
    const int L = L0 - sp * nit;
    // Work item of this workgroup: query head h, query tile qt and, for a tile whose key range
    // is split in two (causal grids too small to fill the GPU), the half `part` (-1: whole).
    // Causal work grows with the query tile, so the items of a kv head are dispatched heaviest
    // first: longest-first keeps the tail of the grid short.
    // pack (Sq below the workgroup's BQ rows, GQA groups): the g*Sq rows of a kv head are one
    // row space, row r being query r % Sq of head u*g + r / Sq, and qt tiles it in BQ rows, so
    // short query blocks fill whole tiles and a kv head's K/V is read once for all its heads.
    // hsplit > 0 (non-causal, two workgroups per CU, a grid of 16 R = two per CU of R CUs per
    // XCD): the tiles of heads below Hq - hsplit run whole, in the CUs' first slots (XCD
    // positions below R), and each tile of the last hsplit heads runs as two halves of its key
    // range in the remaining slots, so no CU holds more than one and a half tiles.
    int h, qt, part = -1, h0 = 0;
    if (hsplit > 0) {
        const int R = pair_r, b = wg_id_x(), x = b & 7, i = b >> 3;
        const int item = (i < R) ? x * R + i : 8 * R + x * R + (i - R);
        const int nwhole = (Hq - hsplit) * nqt;
        if (item < nwhole) {
            h = item / nqt;
            qt = item - h * nqt;
        } else {
            const int k = item - nwhole;
            if (k >= 2 * hsplit * nqt)
                return; // the grid rounds the items up to two per CU
            const int j = k >> 1;
            h0 = Hq - hsplit;
            h = h0 + j / nqt;
            qt = j - (j / nqt) * nqt;
            part = k & 1;
        }
    } else if (pack) {
        const int uu = L / nqt;
        qt = L - uu * nqt;
        h = uu * g;
    } else if (split_first < 0) {
        const int uu = L / (g * nqt);
        const int rr = L - uu * (g * nqt);
        qt = CAUSAL ? nqt - 1 - rr / g : rr / g;
        h = uu * g + (rr - (rr / g) * g);
    } else {
        // Per kv head: tiles qt >= split_first as two halves (work ~ (qt+1)/2 each), tiles below
        // whole (work qt+1); item k of the merged heaviest-first order, g query heads each.
        const int nsp = nqt - split_first;
        const int per = g * (split_first + 2 * nsp);
        const int uu = L / per;
        const int rr = L - uu * per;
        const int k = rr / g;
        h = uu * g + (rr - k * g);
        int ia = 0, ib = 0;
        for (int st = 0; st < k; ++st) {
            const bool a = ib >= split_first || (ia < 2 * nsp && nqt - ia / 2 >= 2 * (split_first - ib));
            ia += a ? 1 : 0;
            ib += a ? 0 : 1;
        }
        if (ib >= split_first || (ia < 2 * nsp && nqt - ia / 2 >= 2 * (split_first - ib))) {
            qt = nqt - 1 - ia / 2;
            part = ia & 1;
        } else {
            qt = split_first - 1 - ib;
        }
    }
    // Work-item values are workgroup-uniform; readfirstlane keeps them (and the loop control and
    // tile addresses derived from them) in scalar registers, where the integer divisions above
    // would otherwise leave them in VGPRs.
    const int u = __builtin_amdgcn_readfirstlane(h / g); // kv head

    const int tid = threadIdx.x, lane = tid & 63; // a library call on purpose: see wi_id_x
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6); // wave-uniform: LDS-DMA bases in SGPRs
    // Phase stamps (ATTN_PHASE_STAMPS builds): slot 0 at entry, 1 when Q and the first tile are
    // in, 2 after the first tile, 3 after the last, 4 after the key halves' hand-over, the last
    // slot once the O (or partial) stores have completed; slot 6 holds the CU, 7 the key tiles.
    phase_stamp(w, lane, 0);
    phase_value(w, lane, 6, phase_cu());
    const int wr = KH ? w % NR : w; // the wave's 32-row block of the workgroup's rows
    const int kh = KH ? w / NR : 0; // and its half of each key tile
    const int l32 = lane & 31, hi = lane >> 5;
    // This lane's row: query myq of head hl (valid if rvalid); the wave's valid rows have query
    // indices in [qmin, qmax] (causal limits), and the workgroup's at most qwg.
    int hl, myq, qmin, qmax, qwg;
    bool rvalid, wvalid;
    if (pack) {
        const int R = g * Sq;
        const int r = qt * BQ + wr * 32 + l32;
        rvalid = r < R;
        hl = h + (rvalid ? r / Sq : 0);
        myq = rvalid ? r - (r / Sq) * Sq : 0;
        const int r0 = qt * BQ + wr * 32, r1 = min(r0 + 31, R - 1);
        wvalid = r0 < R;
        const bool one = r0 / Sq == r1 / Sq;
        qmin = one ? r0 - (r0 / Sq) * Sq : 0;
        qmax = one ? r1 - (r1 / Sq) * Sq : Sq - 1;
        const int g0 = qt * BQ, g1 = min(g0 + BQ - 1, R - 1);
        qwg = (g0 / Sq == g1 / Sq) ? g1 - (g1 / Sq) * Sq : Sq - 1;
    } else {
        hl = h;
        myq = qt * BQ + wr * 32 + l32;
        rvalid = myq < Sq;
        qmin = qt * BQ + wr * 32;
        wvalid = qmin < Sq;
        qmax = min(qmin + 31, Sq - 1);
        qwg = min(qt * BQ + BQ - 1, Sq - 1);
    }
    const size_t qrow = (size_t)hl * Sq + myq; // row of Q and O

    const uint32_t kvbytes = (uint32_t)Sk * D * 2;
    const __amdgpu_buffer_rsrc_t rv = make_rsrc(V + (size_t)u * Sk * D, kvbytes); // V^T path

    bf16x8 qb[DP / 16];
    // Q rows arrive either by LDS-DMA into this wave's 32 x DP block of the K/V tiles' second
    // buffer (idle until tile kt0+1's DMA, which follows the barrier before the loop): each DMA
    // reads 1 KB of whole rows, where loading the operand layout directly takes 32 rows x 32
    // bytes per instruction. Chunk c of row r sits at slot c ^ (r & QSWZ), so the 32 lanes of an
    // operand read (32 rows, one chunk) hit distinct bank groups; chunks past D and rows past Sq
    // arrive as zeros. Measured (same box): c3 1k +1.9%, config 5 +1.9%, c3 4k causal +1.5%,
    // c3 2k +1%, c4 +0.8%, c3 4k +0.5% with 8 waves; the 4-wave kernels measured 0 to -2%
    // (c3 1k causal, chunked prefill), and they, packed tiles and DP = 256 load directly.
    constexpr int NQC = DP / 8; // 16-byte chunks per Q row
    constexpr int QSWZ = (NQC % 16 == 0) ? 15 : ((NQC % 8 == 0) ? 7 : 3);
    const bool qstage = !UA && NW == 8 && KT >= 16 * NW && DP <= 128 && !pack &&
                        (long)Sq * D * 2 < 0x7fffffffL;
    const uint16_t *qlds =
        NW == 8 ? (w < NW / 2 ? &Ks[1][0] : &Vs[1][0]) + (w % (NW / 2)) * 32 * DP : &Ks[1][0];
    if (qstage) {
        const __amdgpu_buffer_rsrc_t rq =
            make_rsrc(Q + (size_t)h * Sq * D, (uint32_t)Sq * (uint32_t)D * 2u);
        const uint32_t qr0 = (uint32_t)(qt * BQ + wr * 32);
#pragma unroll
        for (int b = 0; b < DP / 16; ++b) {
            const int sl = b * 64 + lane, r = sl / NQC, c = (sl - r * NQC) ^ (r & QSWZ);
            dma16<0>(rq, const_cast<uint16_t *>(qlds) + b * 512,
                     c * 8 < D ? (qr0 + r) * (uint32_t)D * 2u + (uint32_t)c * 16u : 0x80000000u);
        }
    } else {
#pragma unroll
        for (int kk = 0; kk < DP / 16; ++kk) {
            const int col = kk * 16 + hi * 8;
            u32x4 v = zero4();
            if constexpr (UA == 0)
                v = load_row8(Q, qrow, col, D, rvalid);
            else if (rvalid && col < D) {
                const uint16_t *q = Q + qrow * D;
                if constexpr (UA == 2)
                    v = load_short(q, col, D);
                else if ((D & 7) != 0 && kk * 16 + 16 > D) // shifted here: once per workgroup
                    v = drop_elems(load16_any<false>(q + min(col, D - 8)), max(col + 8 - D, 0));
                else
                    v = load16_any<false>(q + col);
            }
            qb[kk] = as_bf16x8(v);
        }
    }
    // Q stays in flight while the first tile's DMA is issued; one wait before the loop covers
    // both (below).

    int nkt = (Sk + KT - 1) / KT;
    int wave_maxkey = wvalid ? Sk - 1 : -1;
    if (CAUSAL) {
        const int maxkey = Sk - Sq + qwg;
        nkt = (maxkey < 0) ? 0 : min(nkt, maxkey / KT + 1);
        if (wvalid)
            wave_maxkey = min(Sk - 1, Sk - Sq + qmax);
    }
    wave_maxkey = __builtin_amdgcn_readfirstlane(wave_maxkey);
    qmin = __builtin_amdgcn_readfirstlane(qmin);
    const int lim = CAUSAL ? min(Sk - 1, Sk - Sq + myq) : Sk - 1;

    float m_run = kNegInf, l_run = 0.f;
    f32x16 o[DP / 32];
#pragma unroll
    for (int db = 0; db < DP / 32; ++db)
#pragma unroll
        for (int i = 0; i < 16; ++i)
            o[db][i] = 0.f;

    // LDS-DMA staging. Byte layout of a tile for key row r and 16-byte chunk c (d/8), and of a
    // V^T tile for d row e and 16-byte key chunk k (8 keys):
    //   K:   (r/8)*16*DP + (c/2)*256 + (r%8)*32 + ((c%2) ^ ((r/8)%2))*16
    //   V:   (r/4)*8*DP + (c/4)*256 + (r%4)*64 + (c%4)*16
    //   V^T: (e/8)*16*KT + (k/2)*256 + (e%8)*32 + ((k%2) ^ ((e/8)%2))*16
    // The 16 lanes of one pass of a 16-byte K or V^T read (16 rows, one chunk) and the 32 lanes
    // of one pass of an 8-byte transposed V read (4 rows x 64 bytes) hit distinct banks; operand
    // steps are immediates (K: 256 B per 16 d, 16*DP*4 B per 32 keys; V: 256 B per 32 d,
    // 8*DP*4 B per 16 keys; V^T: 256 B per 16 keys, 16*KT*4 B per 32 d); each 1 KB DMA block
    // reads whole 128-byte lines of K and V, or 128-byte runs of V^T rows. The NI blocks per
    // tensor go to the waves in contiguous runs of PW; this lane's source offsets within a tile:
    // A chunk of columns D and beyond gets an offset past the buffer's range and arrives as zero.
    constexpr int NI = KT * DP / 512;
    constexpr int PW = (NI + NW - 1) / NW;
    static_assert(PW >= 1 && PW <= 8, "DMA blocks per wave");
    const int nblk_w = max(0, min(PW, NI - w * PW)); // this wave's blocks (wave-uniform)
    uint32_t kso[PW], vso[PW];
#pragma unroll
    for (int k = 0; k < PW; ++k) {
        const int b = (w * PW + k) * 1024 + 16 * lane;
        {
            const int rg = b / (16 * DP), wi = b % (16 * DP);
            const int r = rg * 8 + (wi % 256) / 32;
            const int cc = 2 * (wi / 256) + (((wi % 32) / 16) ^ (rg & 1));
            kso[k] = (cc * 8 < D) ? (uint32_t)(r * D * 2 + cc * 16) : 0x80000000u;
        }
        {
            const int rgv = b / (8 * DP), wi = b % (8 * DP);
            const int r = rgv * 4 + (wi % 256) / 64;
            const int cc = 4 * (wi / 256) + (wi % 64) / 16;
            vso[k] = (cc * 8 < D) ? (uint32_t)(r * D * 2 + cc * 16) : 0x80000000u;
        }
    }
    // V^T: byte d*Sk*2 + (key chunk)*16 of the head for tile 0, and the chunk's first key. A
    // chunk at or past Sk (Sk % 8 == 0, so chunks never straddle it) would read the next d row:
    // it gets an offset beyond the buffer's range and arrives as zero.
    uint32_t vto[PW];
    int vtk[PW];
#pragma unroll
    for (int k = 0; k < PW; ++k) {
        const int b = (w * PW + k) * 1024 + 16 * lane;
        const int rg = b / (16 * KT), wi = b % (16 * KT);
        const int e = rg * 8 + (wi % 256) / 32;
        const int kc = 2 * (wi / 256) + (((wi % 32) / 16) ^ (rg & 1));
        vto[k] = (uint32_t)e * (uint32_t)Sk * 2u + (uint32_t)kc * 16u;
        vtk[k] = (e < D) ? kc * 8 : 0x7fffffff; // d rows past D: never in range
    }
    // K (or V) tile kt into LDS buffer buf. Row-major K and V: descriptors based at the tile
    // (scalar work), whose range still ends at the head's last byte, so the per-lane offsets stay
    // loop-invariant.
    auto dma_k = [&](int kt, int buf) {
        const uint32_t toff = (uint32_t)kt * KT * D * 2;
        const __amdgpu_buffer_rsrc_t rkt = make_rsrc(K + (size_t)u * Sk * D + (size_t)kt * KT * D,
                                                     kvbytes - toff);
#pragma unroll
        for (int k = 0; k < PW; ++k)
            if (NI % NW == 0 || k < nblk_w)
                dma16<0>(rkt, &Ks[buf][(w * PW + k) * 512], kso[k]);
    };
    // UA: this wave's pieces of a K (or V) tile into registers, and from there into LDS. Every load
    // stays inside its row: a piece that reaches past the row's end is read as the row's last
    // eight elements and shifted where it is put into LDS (shifting it at the load would wait for
    // it). One packed offset per piece is kept and made opaque where it is used.
    constexpr int UPW = UA ? PW : 1;
    constexpr bool TINY = UA == 2; // rows of fewer than eight elements
    u32x4 gk[UPW], gv[UPW];
    const uint16_t *Kh = K + (size_t)u * Sk * D, *Vh = V + (size_t)u * Sk * D;
    // Row-major piece k: (element offset of its eight elements in the tile) * 16 + how many of
    // them precede the piece. TINY: (row * 64 + first column).
    uint32_t kpk[UPW], vpk[UPW];
    uint32_t ktail = 0, vtail = 0; // bit k: piece k of some lane reaches past D (wave-uniform)
    if constexpr (UA != 0) {
        auto pack = [&](int r, int col, uint32_t &pk, uint32_t &tail, int k) {
            pk = TINY ? (uint32_t)(r * 64 + col)
                      : (uint32_t)(r * D + min(col, D - 8)) * 16u + (uint32_t)min(8, max(0, col + 8 - D));
            tail |= __builtin_amdgcn_ballot_w64(col + 8 > D) != 0 ? 1u << k : 0u;
        };
#pragma unroll
        for (int k = 0; k < PW; ++k) {
            const int b = (w * PW + k) * 1024 + 16 * lane;
            const int rk = b / (16 * DP), wk = b % (16 * DP), rw = b / (8 * DP), wv = b % (8 * DP);
            pack(rk * 8 + (wk % 256) / 32, 8 * (2 * (wk / 256) + (((wk % 32) / 16) ^ (rk & 1))),
                 kpk[k], ktail, k);
            pack(rw * 4 + (wv % 256) / 64, 8 * (4 * (wv / 256) + (wv % 64) / 16), vpk[k], vtail, k);
        }
        ktail = __builtin_amdgcn_readfirstlane(ktail);
        vtail = __builtin_amdgcn_readfirstlane(vtail);
    }
    // TINY: a row is one piece, the rows after it behind it; the head's last rows are read with its
    // last eight elements, at this offset from tile kt's first (below 0 where that tile is shorter).
    auto tiny_last = [&](int kt) {
        return (int)min((long)(Sk - kt * KT) * D, (long)KT * 8) - 8;
    };
    auto ua_rows = [&](const uint16_t *H, int kt, const uint32_t *pk, u32x4 *gr)
        __attribute__((always_inline)) {
        const uint16_t *T = H + (size_t)kt * KT * D;
        const uint32_t last = (uint32_t)((Sk - kt * KT) * (long)D > KT * DP ? KT * DP
                                                                            : (Sk - kt * KT) * D);
#pragma unroll
        for (int k = 0; k < PW; ++k)
            if (NI % NW == 0 || k < nblk_w) {
                const uint32_t x = opaque(pk[k]);
                if constexpr (TINY) {
                    const int r = (int)(x >> 6);
                    gr[k] = zero4();
                    if ((x & 63) == 0 && kt * KT + r < Sk)
                        gr[k] = (long)Sk * D < 8 ? load_rolled(T + r * D, 0, D)
                                                 : load16_any<false>(T + min(r * D, tiny_last(kt)));
                } else { // rows past the last key read its last elements
                    gr[k] = load16_any<false>(T + min(x >> 4, last - 8));
                }
            }
    };
    // Rows past the last key become zeros (their P is 0, and 0 times what was read may be NaN).
    auto put_rows = [&](uint16_t *tile, int kt, const uint32_t *pk, uint32_t tail, const u32x4 *gr)
        __attribute__((always_inline)) {
        const bool edge = !TINY && kt * KT + KT > Sk;
#pragma unroll
        for (int k = 0; k < PW; ++k)
            if (NI % NW == 0 || k < nblk_w) {
                u32x4 v = gr[k];
                if (TINY && (long)Sk * D >= 8) {
                    const int at = (int)(opaque(pk[k]) >> 6) * D;
                    v = keep_elems(drop_elems(v, min(8, max(0, at - tiny_last(kt)))), D);
                }
                if (!TINY && (tail >> k & 1))
                    v = drop_elems(v, (int)(opaque(pk[k]) & 15));
                if (edge)
                    v = (int)(opaque(pk[k]) >> 4) < (Sk - kt * KT) * D ? v : zero4();
                *reinterpret_cast<u32x4 *>(&tile[(w * PW + k) * 512 + lane * 8]) = v;
            }
    };
    // V^T piece k: d row e (past D: D - 1, never stored) and the eight keys from 8 kc of the tile.
    auto vt_piece = [&](int k, int &e, int &key) __attribute__((always_inline)) {
        const int b = (w * PW + k) * 1024 + 16 * (int)opaque((uint32_t)lane);
        const int rg = b / (16 * KT), wi = b % (16 * KT);
        e = min(rg * 8 + (wi % 256) / 32, D - 1);
        key = 8 * (2 * (wi / 256) + (((wi % 32) / 16) ^ (rg & 1)));
    };
    auto ua_vt = [&](int kt) __attribute__((always_inline)) {
#pragma unroll
        for (int k = 0; k < PW; ++k)
            if (NI % NW == 0 || k < nblk_w) {
                int e, key;
                vt_piece(k, e, key);
                key += kt * KT;
                const uint16_t *row = Vh + (size_t)e * Sk;
                if (Sk < 8)
                    gv[k] = load_rolled(row, key, Sk);
                else
                    gv[k] = load16_any<false>(row + min(key, Sk - 8));
            }
    };
    auto put_vt = [&](uint16_t *tile, int kt) __attribute__((always_inline)) {
        const bool edge = Sk >= 8 && kt * KT + KT > Sk;
#pragma unroll
        for (int k = 0; k < PW; ++k)
            if (NI % NW == 0 || k < nblk_w) {
                u32x4 v = gv[k];
                if (edge) {
                    int e, key;
                    vt_piece(k, e, key);
                    v = drop_elems(v, min(8, max(0, kt * KT + key + 8 - Sk)));
                }
                *reinterpret_cast<u32x4 *>(&tile[(w * PW + k) * 512 + lane * 8]) = v;
            }
    };
    auto dma_v = [&](int kt, int buf) {
        if constexpr (VT) {
            const int klim = Sk - kt * KT; // keys of this tile that exist
#pragma unroll
            for (int k = 0; k < PW; ++k)
                if (NI % NW == 0 || k < nblk_w)
                    dma16<0>(rv, &Vs[buf][(w * PW + k) * 512],
                             vtk[k] < klim ? vto[k] + (uint32_t)kt * KT * 2 : 0x80000000u);
        } else {
            const uint32_t toff = (uint32_t)kt * KT * D * 2;
            const __amdgpu_buffer_rsrc_t rvt =
                make_rsrc(V + (size_t)u * Sk * D + (size_t)kt * KT * D, kvbytes - toff);
#pragma unroll
            for (int k = 0; k < PW; ++k)
                if (NI % NW == 0 || k < nblk_w)
                    dma16<0>(rvt, &Vs[buf][(w * PW + k) * 512], vso[k]);
        }
    };

    const int kperm = (l32 & ~12) | ((l32 & 4) << 1) | ((l32 & 8) >> 1);
    const int g16 = lane >> 4, i16 = lane & 15;

    // Key tiles [kt0, kt1) of this item: all of them, or one half of a split tile's range.
    const int kt0 = __builtin_amdgcn_readfirstlane(
        (nsplit > 1) ? (int)((long)nkt * sp / nsplit) : (part == 1) ? nkt / 2 : 0);
    const int kt1 = __builtin_amdgcn_readfirstlane(
        (nsplit > 1) ? (int)((long)nkt * (sp + 1) / nsplit) : (part == 0) ? nkt / 2 : nkt);
    // Fragment offsets (elements) of this lane in a DMA-staged tile: K row t*32 + kperm,
    // chunk 2kk + hi; V rows cc*16 + 8hi + i16/4 (+4), columns db*32 + (g16&1)*16 + 4(i16&3).
    const int kfo = (kperm >> 3) * 8 * DP + (kperm & 7) * 16 + ((hi ^ ((kperm >> 3) & 1)) * 8);
    constexpr int KSUB = 32 * DP; // 32-key sub-tile step
    constexpr int KDK = 128;      // 16-d step
    // V^T operand: d row db*32 + l32, keys cc*16 + 8hi .. +8.
    const int vfo = VT ? (l32 >> 3) * 8 * KT + (l32 & 7) * 16 + ((hi ^ ((l32 >> 3) & 1)) * 8)
                       : hi * 8 * DP + (i16 >> 2) * 32 + (2 * (g16 & 1) + ((i16 & 3) >> 1)) * 8 +
                             (i16 & 1) * 4;

    f32x16 s[KW / 32];
    bf16x8 pk[KW / 16];
    // S^T = K_tile . Q^T for one key tile (LDS buffer buf) into s; the next 32-key sub-tile's K
    // fragments are read between this sub-tile's MFMAs.
    auto qk = [&](int buf) __attribute__((always_inline)) {
        const uint16_t *kb0 = &Ks[buf][kfo + kh * (KW / 32) * KSUB];
        if constexpr (kRing) {
            constexpr int NK = DP / 16, N = KW / 32 * NK;
            auto frag = [&](int f) {
                return as_bf16x8(
                    *reinterpret_cast<const u32x4 *>(kb0 + f / NK * KSUB + f % NK * KDK));
            };
            bf16x8 kr[RD];
#pragma unroll
            for (int f = 0; f < RD; ++f)
                kr[f] = frag(f);
            __builtin_amdgcn_sched_group_barrier(0x100, RD, 0);
#pragma unroll
            for (int f = 0; f < N; ++f) {
                if (f % NK == 0)
#pragma unroll
                    for (int i = 0; i < 16; ++i)
                        s[f / NK][i] = 0.f;
                s[f / NK] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kr[f % RD], qb[f % NK],
                                                                   s[f / NK], 0, 0, 0);
                if (f + RD < N)
                    kr[f % RD] = frag(f + RD);
            }
#pragma unroll
            for (int f = 0; f < N; ++f) {
                __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                if (f + RD < N)
                    __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
            }
            return;
        }
        bf16x8 ka[2][DP / 16];
#pragma unroll
        for (int kk = 0; kk < DP / 16; ++kk)
            ka[0][kk] = as_bf16x8(*reinterpret_cast<const u32x4 *>(kb0 + kk * KDK));
        __builtin_amdgcn_sched_group_barrier(0x100, DP / 16, 0);
#pragma unroll
        for (int t = 0; t < KW / 32; ++t) {
#pragma unroll
            for (int i = 0; i < 16; ++i)
                s[t][i] = 0.f;
#pragma unroll
            for (int kk = 0; kk < DP / 16; ++kk) {
                s[t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ka[t & 1][kk], qb[kk], s[t], 0, 0, 0);
                if (t + 1 < KW / 32)
                    ka[(t + 1) & 1][kk] = as_bf16x8(
                        *reinterpret_cast<const u32x4 *>(kb0 + (t + 1) * KSUB + kk * KDK));
            }
#pragma unroll
            for (int kk = 0; kk < DP / 16; ++kk) {
                __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                if (t + 1 < KW / 32)
                    __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
            }
        }
    };
    // Online softmax of the tile at key kbase, in three steps: mask, row max with lazy rescale of
    // (l, o), then p = 2^(s c - m c) into P (bf16, the B operand of P.V) and the lane's sum of
    // the fp32 p.
    // ME (may be an edge tile) false: the tile is known to need no mask, and none is compiled.
    // Per 32-key sub-tile, with wave-uniform tests: the wave's smallest key limit (its first
    // row's) leaves whole sub-tiles visible to every row, its largest (wave_maxkey) leaves whole
    // sub-tiles visible to none; only a sub-tile between the two is masked key by key.
    auto mask = [&](int kbase, auto me) __attribute__((always_inline)) {
        if (decltype(me)::value &&
            ((kbase + KW > Sk) || (CAUSAL && kbase + KW - 1 > Sk - Sq + qmin))) {
            const int lo = CAUSAL ? min(Sk - 1, Sk - Sq + qmin) : Sk - 1;
#pragma unroll
            for (int t = 0; t < KW / 32; ++t) {
                const int k0t = kbase + t * 32;
                if (k0t + 31 <= lo)
                    continue;
                if (k0t > wave_maxkey) {
#pragma unroll
                    for (int i = 0; i < 16; ++i)
                        s[t][i] = kNegInf;
                    continue;
                }
#pragma unroll
                for (int i = 0; i < 16; ++i) {
                    const int key = k0t + 16 * (i >> 3) + 8 * hi + (i & 7);
                    if (key > lim)
                        s[t][i] = kNegInf;
                }
            }
        }
    };
    // Row max: one max3 chain per 32-key sub-tile (two new scores per instruction), the chains
    // combined, the partner half-row through the VALU exchange; m rises to any larger tile max
    // (wave-uniform test), rescaling (l, o).
    auto row_max = [&]() __attribute__((always_inline)) {
        float mt[KW / 32];
#pragma unroll
        for (int t = 0; t < KW / 32; ++t) {
            float m = max3f(s[t][0], s[t][1], s[t][2]);
#pragma unroll
            for (int i = 3; i < 15; i += 2)
                m = max3f(m, s[t][i], s[t][i + 1]);
            mt[t] = fmaxf(m, s[t][15]);
        }
        float mx = mt[0];
#pragma unroll
        for (int j = 1; j < KW / 32; j += 2)
            mx = (j + 1 < KW / 32) ? max3f(mx, mt[j], mt[j + 1]) : fmaxf(mx, mt[j]);
        mx = max_xor32(mx);
        const bool raise = mx > m_run;
        if (__builtin_amdgcn_ballot_w64(raise) != 0) {
            const float mnew = raise ? mx : m_run;
            const float alpha = (mnew == m_run) ? 1.0f : fast_exp2((m_run - mnew) * c);
            l_run *= alpha;
#pragma unroll
            for (int db = 0; db < DP / 32; ++db)
                o[db] *= alpha;
            m_run = mnew;
        }
    };
    auto exps = [&]() __attribute__((always_inline)) -> float {
        const float mc = (m_run == kNegInf) ? 0.f : m_run * c;
        float ps[KW / 16];
#pragma unroll
        for (int t = 0; t < KW / 32; ++t)
#pragma unroll
            for (int hh = 0; hh < 2; ++hh) {
                float p[8];
#pragma unroll
                for (int j = 0; j < 8; ++j) {
                    p[j] = fast_exp2(fmaf(s[t][8 * hh + j], c, -mc));
                    pk[2 * t + hh][j] = (__bf16)p[j];
                }
                ps[2 * t + hh] = ((p[0] + p[1]) + (p[2] + p[3])) + ((p[4] + p[5]) + (p[6] + p[7]));
            }
        float psum = 0.f;
#pragma unroll
        for (int j = 0; j < KW / 16; ++j)
            psum += ps[j];
        return psum;
    };
    // O^T += V^T . P^T for the tile in LDS buffer buf. The V^T operand of 16-key chunk cc, d
    // block db: one 16-byte read (V^T tile) or two transposed 8-byte reads (row-major V tile).
    // Fragments are double-buffered a chunk ahead, so each read has the previous chunk's MFMAs
    // to land in; chunk 0 is read by pv_first before the softmax, under its exponentials.
    bf16x8 va[2][DP / 32];
    auto vfrag = [&](int buf, int cc, int db) -> bf16x8 {
        cc += kh * (KW / 16); // the wave's key half of the tile (KH)
        if (VT)
            return as_bf16x8(
                *reinterpret_cast<const u32x4 *>(&Vs[buf][vfo + cc * 128 + db * 32 * KT]));
        const uint16_t *vb = &Vs[buf][vfo + cc * 16 * DP + db * 128];
        return join_tr(lds_read_tr(vb), lds_read_tr(vb + 4 * DP));
    };
    bf16x8 vr[RD];
    auto pv_first = [&](int buf) {
        if constexpr (kRing) {
#pragma unroll
            for (int f = 0; f < RD; ++f)
                vr[f] = vfrag(buf, f / (DP / 32), f % (DP / 32));
            return;
        }
#pragma unroll
        for (int db = 0; db < DP / 32; ++db)
            va[0][db] = vfrag(buf, 0, db);
    };
    // Softmax of a tile after an item's first. Its p are taken against the running m with no
    // row max, and each lane's tile sum is tested instead: it bounds each of the lane's p, so a
    // sum of at most kSumCap keeps every p <= kSumCap. A tile that fails the test (or is not
    // finite) is recomputed from the K tile still in LDS and takes the row max, which brings
    // that row's p back to at most 1. Either way m only rises and never falls behind a score by
    // more than log2(kSumCap) / c. An item's first tile always takes the row max (the loop below
    // peels it), so m starts at its tile's maximum and a row whose first tile holds its largest
    // score keeps weight exactly 1. A row still at m = -inf after its first tile has no
    // admissible key in the item (keys only grow along the tiles), so its p stay 0.
    auto softmax_next = [&](int buf, int kbase, auto me) __attribute__((always_inline)) {
        mask(kbase, me);
        float psum = exps();
        if (__builtin_expect(__builtin_amdgcn_ballot_w64(!(psum <= kSumCap)) != 0, 0)) {
            qk(buf);
            pv_first(buf); // re-read, so the earlier fragments are not live across qk
            mask(kbase, me);
            row_max();
            psum = exps();
        }
        l_run += psum;
    };
    auto pv = [&](int buf) {
        if constexpr (kRing) {
            constexpr int ND = DP / 32, N = KW / 16 * ND;
#pragma unroll
            for (int f = 0; f < N; ++f) {
                o[f % ND] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vr[f % RD], pk[f / ND],
                                                                   o[f % ND], 0, 0, 0);
                if (f + RD < N)
                    vr[f % RD] = vfrag(buf, (f + RD) / ND, (f + RD) % ND);
            }
#pragma unroll
            for (int f = 0; f < N; ++f) {
                __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                if (f + RD < N)
                    __builtin_amdgcn_sched_group_barrier(0x100, VT ? 1 : 2, 0);
            }
            return;
        }
#pragma unroll
        for (int cc = 0; cc < KW / 16; ++cc) {
#pragma unroll
            for (int db = 0; db < DP / 32; ++db) {
                o[db] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(va[cc & 1][db], pk[cc], o[db], 0, 0,
                                                               0);
                if (cc + 1 < KW / 16)
                    va[(cc + 1) & 1][db] = vfrag(buf, cc + 1, db);
            }
#pragma unroll
            for (int db = 0; db < DP / 32; ++db) {
                __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                if (cc + 1 < KW / 16)
                    __builtin_amdgcn_sched_group_barrier(0x100, VT ? 1 : 2, 0);
            }
        }
    };

    // A tile after an item's first whose keys are all admissible for the wave (no mask), software
    // pipelined over its 32-key sub-tiles: with the row max gone from such tiles, the
    // exponentials of sub-tile t need only t's scores, so one block issues them beside the MFMAs
    // of Q.K^T for t+1 and P.V for t-1, and each wave overlaps its own VALU and MFMA work. Each
    // sub-tile's p sum is tested before its P.V; a sub-tile that fails takes the row max of its
    // own scores, rescales (l, o) and redoes its exponentials (l and o then hold sub-tiles < t
    // only, so the rescale covers everything accumulated).
    auto tile_pipelined = [&](int buf) __attribute__((always_inline)) {
        constexpr int NS = KW / 32;
        constexpr int NDB = DP / 32, NKK = DP / 16;
        const uint16_t *kb0 = &Ks[buf][kfo + kh * (KW / 32) * KSUB];
        bf16x8 ka[2][NKK];
        float mc = m_run * c; // m_run is finite: every row of the wave has had an admissible key
#pragma unroll
        for (int kk = 0; kk < NKK; ++kk)
            ka[0][kk] = as_bf16x8(*reinterpret_cast<const u32x4 *>(kb0 + kk * KDK));
#pragma unroll
        for (int i = 0; i < 16; ++i)
            s[0][i] = 0.f;
#pragma unroll
        for (int kk = 0; kk < NKK; ++kk) {
            s[0] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ka[0][kk], qb[kk], s[0], 0, 0, 0);
            if (NS > 1)
                ka[1][kk] = as_bf16x8(*reinterpret_cast<const u32x4 *>(kb0 + KSUB + kk * KDK));
        }
#pragma unroll
        for (int db = 0; db < NDB; ++db)
            va[0][db] = vfrag(buf, 0, db);
        static_for<NS>([&](auto T) __attribute__((always_inline)) {
            constexpr int t = decltype(T)::value;
            // MFMA work of this block: Q.K^T of sub-tile t+1 and P.V of sub-tile t-1.
            if constexpr (t + 1 < NS) {
#pragma unroll
                for (int i = 0; i < 16; ++i)
                    s[t + 1][i] = 0.f;
#pragma unroll
                for (int kk = 0; kk < NKK; ++kk) {
                    s[t + 1] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ka[(t + 1) & 1][kk], qb[kk],
                                                                       s[t + 1], 0, 0, 0);
                    if (t + 2 < NS)
                        ka[t & 1][kk] = as_bf16x8(*reinterpret_cast<const u32x4 *>(
                            kb0 + (t + 2) * KSUB + kk * KDK));
                }
            }
            if constexpr (t >= 1) {
#pragma unroll
                for (int cc = 2 * t - 2; cc < 2 * t; ++cc)
#pragma unroll
                    for (int db = 0; db < NDB; ++db) {
                        o[db] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(va[cc & 1][db], pk[cc],
                                                                       o[db], 0, 0, 0);
                        va[(cc + 1) & 1][db] = vfrag(buf, cc + 1, db);
                    }
            }
            // VALU work of this block: p of sub-tile t and its sum.
            float ps[2];
#pragma unroll
            for (int hh = 0; hh < 2; ++hh) {
                float p[8];
#pragma unroll
                for (int jj = 0; jj < 8; ++jj) {
                    p[jj] = fast_exp2(fmaf(s[t][8 * hh + jj], c, -mc));
                    pk[2 * t + hh][jj] = (__bf16)p[jj];
                }
                ps[hh] = ((p[0] + p[1]) + (p[2] + p[3])) + ((p[4] + p[5]) + (p[6] + p[7]));
            }
            // Interleave: one MFMA, then its share of the LDS reads and of the VALU work.
            constexpr int NMF = ((t + 1 < NS) ? NKK : 0) + ((t >= 1) ? 2 * NDB : 0);
            constexpr int NDS = ((t + 2 < NS) ? NKK : 0) + ((t >= 1) ? 2 * NDB * (VT ? 1 : 2) : 0);
            if constexpr (NMF > 0) {
#pragma unroll
                for (int m = 0; m < NMF; ++m) {
                    __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                    if constexpr (NDS > 0)
                        __builtin_amdgcn_sched_group_barrier(0x100, (NDS + NMF - 1) / NMF, 0);
                    __builtin_amdgcn_sched_group_barrier(0x002, 64 / NMF, 0);
                }
            }
            float psum = ps[0] + ps[1];
            if (__builtin_expect(__builtin_amdgcn_ballot_w64(!(psum <= kSumCap)) != 0, 0)) {
                float mx = max3f(s[t][0], s[t][1], s[t][2]);
#pragma unroll
                for (int i = 3; i < 15; i += 2)
                    mx = max3f(mx, s[t][i], s[t][i + 1]);
                mx = max_xor32(fmaxf(mx, s[t][15]));
                const bool raise = mx > m_run;
                if (__builtin_amdgcn_ballot_w64(raise) != 0) {
                    const float mnew = raise ? mx : m_run;
                    const float alpha = (mnew == m_run) ? 1.0f : fast_exp2((m_run - mnew) * c);
                    l_run *= alpha;
#pragma unroll
                    for (int db = 0; db < NDB; ++db)
                        o[db] *= alpha;
                    m_run = mnew;
                    mc = m_run * c;
                }
                psum = 0.f;
#pragma unroll
                for (int hh = 0; hh < 2; ++hh)
#pragma unroll
                    for (int jj = 0; jj < 8; ++jj) {
                        const float p = fast_exp2(fmaf(s[t][8 * hh + jj], c, -mc));
                        pk[2 * t + hh][jj] = (__bf16)p;
                        psum += p;
                    }
            }
            l_run += psum;
        });
        // P.V of the last sub-tile.
#pragma unroll
        for (int cc = 2 * NS - 2; cc < 2 * NS; ++cc)
#pragma unroll
            for (int db = 0; db < NDB; ++db) {
                o[db] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(va[cc & 1][db], pk[cc], o[db], 0, 0,
                                                               0);
                if (cc + 1 < 2 * NS)
                    va[(cc + 1) & 1][db] = vfrag(buf, cc + 1, db);
            }
    };

    // The staging of tile kt into buffer buf: by DMA at the start of the tile before it, or (UA)
    // loaded at that tile's start and put into LDS at its end.
    auto stage_begin = [&](int kt, int buf) __attribute__((always_inline)) {
        if constexpr (UA != 0) {
            ua_rows(Kh, kt, kpk, gk);
            if constexpr (VT)
                ua_vt(kt);
            else
                ua_rows(Vh, kt, vpk, gv);
        } else {
            dma_k(kt, buf);
            dma_v(kt, buf);
        }
    };
    auto stage_end = [&](int kt, int buf) __attribute__((always_inline)) {
        if constexpr (UA != 0) {
            __builtin_amdgcn_sched_barrier(0);
            put_rows(&Ks[buf][0], kt, kpk, ktail, gk);
            if constexpr (VT)
                put_vt(&Vs[buf][0], kt);
            else
                put_rows(&Vs[buf][0], kt, vpk, vtail, gv);
        }
    };
    if (kt0 < kt1) {
        stage_begin(kt0, 0);
        stage_end(kt0, 0);
    }
    // Q and this wave's DMA blocks of the first tile have landed. Q must be resident before the
    // loop: otherwise the compiler's wait at the loop's first MFMA also waits for the next tile's
    // prefetch (its count cannot tell the two apart). 0x0F70 = vmcnt(0), expcnt and lgkmcnt
    // unconstrained (gfx9 encoding).
    __builtin_amdgcn_s_waitcnt(0x0F70);
    if (qstage) {
#pragma unroll
        for (int kk = 0; kk < DP / 16; ++kk)
            qb[kk] = as_bf16x8(*reinterpret_cast<const u32x4 *>(
                qlds + l32 * DP + (((2 * kk + hi) ^ (l32 & QSWZ)) * 8)));
    }
    __syncthreads();
    phase_stamp(w, lane, 1);
    // One key tile: the next tile's DMA, then Q.K^T, softmax and P.V of this one (FIRST: the
    // item's first tile, whose softmax takes the row max; ME: the tile may need the mask).
    auto step = [&](int kt, auto first, auto me) __attribute__((always_inline)) {
        const int buf = (kt - kt0) & 1;
        // The other buffer's last readers finished before the barrier that ended tile kt-1.
        if (kt + 1 < kt1)
            stage_begin(kt + 1, buf ^ 1);
        const int kbase = kt * KT + kh * KW; // this wave's keys: [kbase, kbase + KW)
        const bool edge = decltype(me)::value &&
                          ((kbase + KW > Sk) || (CAUSAL && kbase + KW - 1 > Sk - Sq + qmin));
        if (kbase <= wave_maxkey) {
            // The pipelined path at DP <= 64 only: at larger DP it spills (two sub-tiles' K
            // fragments, S and the V read-ahead do not fit beside O and Q). Key halves take it
            // on 12 waves only (two 32-key sub-tiles per wave).
            if (kPipe && !decltype(first)::value && !edge && pipe) {
                if constexpr (kPipe)
                    tile_pipelined(buf);
            } else {
                qk(buf);
                pv_first(buf);
                if constexpr (UA || decltype(first)::value) {
                    mask(kbase, me);
                    row_max();
                    l_run += exps();
                } else {
                    softmax_next(buf, kbase, me);
                }
                pv(buf);
            }
        }
        // vmcnt(0): tile kt+1's DMA blocks have landed; the barrier publishes them and frees
        // buffer buf for tile kt+2. After the item's last tile there is neither: its epilogue
        // uses only the idle buffer (below), so each wave goes on without waiting for the others.
        if (kt + 1 < kt1) {
            stage_end(kt + 1, buf ^ 1);
            __builtin_amdgcn_s_waitcnt(0x0F70);
            __syncthreads();
        }
    };
    // kRing on 32-key tiles: the first two take the row max, so that m starts at the largest of 64
    // keys as on 64-key tiles (with one, causal errors against 64 bits grew from 1.33e-3 to 1.36e-3;
    // with two they are 1.32e-3).
    constexpr int NF = kRing && KT == 32 && !UA ? 2 : 1;
    if (kt0 < kt1)
        step(kt0, std::true_type{}, std::true_type{});
    if constexpr (NF == 2)
        if (kt0 + 1 < kt1)
            step(kt0 + 1, std::true_type{}, std::true_type{});
    phase_stamp(w, lane, 2);
    if constexpr (DP > 128 && !UA) {
        // Unmasked tiles in a loop with no rescale of O in it: with 512 registers O lives in
        // accumulation registers, and a rescale path in the loop had the register allocator copy
        // all of O out of them on every tile (128 v_accvgpr_read per 64-key tile at DP = 256). A
        // tile whose sum test fails leaves the loop, takes the row max outside and comes back.
        // Bit-identical; same box, 64 heads at 2k: D = 256 323 -> 295 us (933 TFLOP/s), causal
        // 194 -> 179. At 4 waves one wave per SIMD bounds it: its softmax, LDS reads and MFMAs take
        // turns (MFMA busy 35% of the clocks). Software-pipelined sub-tiles (8 or 12 fragments ahead)
        // measured 10% slower than these plain phases, alternating the two Q.K^T accumulators
        // within 1%.
        const int medge = CAUSAL ? min(Sk - KT, Sk - Sq + qmin - KT + 1) : Sk - KT;
        const int kt_e = __builtin_amdgcn_readfirstlane(medge < 0 ? 0 : medge / KT + 1);
        const int kt_m = __builtin_amdgcn_readfirstlane(wave_maxkey < 0 ? 0 : min(kt1, kt_e));
        auto finish = [&](int kt, int buf) __attribute__((always_inline)) {
            pv(buf);
            if (kt + 1 < kt1) {
                __builtin_amdgcn_s_waitcnt(0x0F70);
                __syncthreads();
            }
        };
        int kt = kt0 + NF;
        for (;;) {
            bool redo = false;
            for (; kt < kt_m; ++kt) {
                const int buf = (kt - kt0) & 1;
                if (kt + 1 < kt1)
                    stage_begin(kt + 1, buf ^ 1);
                qk(buf);
                pv_first(buf);
                const float psum = exps();
                redo = __builtin_amdgcn_ballot_w64(!(psum <= kSumCap)) != 0;
                if (__builtin_expect(redo, 0))
                    break;
                l_run += psum;
                finish(kt, buf);
            }
            if (!redo)
                break;
            const int buf = (kt - kt0) & 1;
            qk(buf);
            pv_first(buf);
            row_max();
            l_run += exps();
            finish(kt, buf);
            ++kt;
        }
        for (; kt < kt1; ++kt)
            step(kt, std::false_type{}, std::true_type{});
    } else if constexpr (NW == 4 && DP > 64) {
        // Tiles from kt_e on may need the mask (keys past Sk, or past the causal limit of the
        // wave's first row); the loop before them has no mask code. Measured (same box) on the
        // 4-wave 64-key-tile kernels: c3 1k causal +3.3%, Qwen3 4k causal +2.8%, 32 heads 2k
        // causal +2%, 16 heads 2k +1.5%, others within 0.5%. The 8-wave kernels lost 1.5-3.5%
        // with it (c3 4k, c3 causal, c4), so they keep one loop (at D <= 64 see below).
        const int medge = CAUSAL ? min(Sk - KT, Sk - Sq + qmin - KT + 1) : Sk - KT;
        const int kt_e = __builtin_amdgcn_readfirstlane(medge < 0 ? 0 : medge / KT + 1);
        int kt = kt0 + 1;
        for (; kt < min(kt1, kt_e); ++kt)
            step(kt, std::false_type{}, std::false_type{});
        for (; kt < kt1; ++kt)
            step(kt, std::false_type{}, std::true_type{});
    } else {
        int kt = kt0 + 1;
        if constexpr (kPipe) {
            // A wave with query rows runs its tiles before kt_e (no mask needed) in a loop of
            // their own whose body is the pipelined tile alone: with the general tile path in
            // the same loop body, the register allocator kept o in different registers on the
            // two paths and copied it in and out of each pipelined tile (36 v_mov per 64 keys on
            // 12 waves, 18 per 128 on 4 or 8). Bit-identical; same box: config 5 61.6 -> 56.2 us,
            // 40 heads of 1000 rows over 4000 keys +12%, D = 40 +11%, 128 heads at 1k +4.3%,
            // the head split's 4-wave grid +3.7%, 64 heads at 2k causal +3.1%.
            const int medge = CAUSAL ? min(Sk - KT, Sk - Sq + qmin - KT + 1) : Sk - KT;
            const int kt_e = __builtin_amdgcn_readfirstlane(medge < 0 ? 0 : medge / KT + 1);
            if (pipe && __builtin_amdgcn_readfirstlane(wave_maxkey) >= 0) {
                for (; kt < min(kt1, kt_e); ++kt) {
                    const int buf = (kt - kt0) & 1;
                    if (kt + 1 < kt1)
                        stage_begin(kt + 1, buf ^ 1);
                    tile_pipelined(buf);
                    // The same wait and barrier as the end of step().
                    if (kt + 1 < kt1) {
                        __builtin_amdgcn_s_waitcnt(0x0F70);
                        __syncthreads();
                    }
                }
            }
        }
        for (; kt < kt1; ++kt)
            step(kt, std::false_type{}, std::true_type{});
    }
    phase_stamp(w, lane, 3);
    phase_value(w, lane, 7, (unsigned long long)(kt1 - kt0));

    if constexpr (KH) {
        // The second-half wave of each row block hands its (m, l, o) to the first-half wave
        // through LDS: o into the buffer pair the last tile left idle ((kt1 - kt0) & 1: past
        // the barrier after its last reader, no DMA pending; 12 waves: kh_o), 16-byte pieces in
        // lane order, so
        // each lane reads back exactly its partner lane's values (same query, same d, same key
        // parity). After the barrier the first-half wave combines the two with log-sum-exp
        // weights against the larger m (a half with no admissible key has m = -inf, weight 0),
        // and only it goes on to the epilogue, which then stages O in the other buffer.
        const int nbx = (kt1 - kt0) & 1;
        float *xo = (KHO > 1) ? &kh_o[wr * DP * 32]
                              : reinterpret_cast<float *>((wr & 2) ? &Vs[nbx][0] : &Ks[nbx][0]) +
                                    (wr & 1) * (DP / 32) * 16 * 64;
        if (kh == 1) {
            kh_ml[wr * 128 + lane] = m_run;
            kh_ml[wr * 128 + 64 + lane] = l_run;
#pragma unroll
            for (int db = 0; db < DP / 32; ++db)
#pragma unroll
                for (int i4 = 0; i4 < 4; ++i4) {
                    f32x4 v = {o[db][4 * i4], o[db][4 * i4 + 1], o[db][4 * i4 + 2],
                               o[db][4 * i4 + 3]};
                    *reinterpret_cast<f32x4 *>(xo + ((db * 4 + i4) * 64 + lane) * 4) = v;
                }
        }
        __syncthreads();
        if (kh == 1)
            return;
        const float m2 = kh_ml[wr * 128 + lane], l2 = kh_ml[wr * 128 + 64 + lane];
        const float mn = fmaxf(m_run, m2);
        const float a1 = (m_run == kNegInf) ? 0.f : fast_exp2((m_run - mn) * c);
        const float a2 = (m2 == kNegInf) ? 0.f : fast_exp2((m2 - mn) * c);
        l_run = l_run * a1 + l2 * a2;
        m_run = mn;
#pragma unroll
        for (int db = 0; db < DP / 32; ++db)
#pragma unroll
            for (int i4 = 0; i4 < 4; ++i4) {
                const f32x4 v = *reinterpret_cast<const f32x4 *>(xo + ((db * 4 + i4) * 64 + lane) * 4);
#pragma unroll
                for (int j = 0; j < 4; ++j)
                    o[db][4 * i4 + j] = o[db][4 * i4 + j] * a1 + v[j] * a2;
            }
    }
    phase_stamp(w, lane, 4);
    const float lt = sum_xor32(l_run);
    // Columns d .. d+3 of a row of D floats: UA rows are 4-byte aligned and may end inside them.
    auto store4 = [&](float *row, int d, f32x4 v) __attribute__((always_inline)) {
        if constexpr (!UA) {
            if (d < D)
                *reinterpret_cast<f32x4 *>(row + d) = v;
        } else if (d + 4 <= D) {
            *reinterpret_cast<f32x4_a4 *>(row + d) = v;
        } else {
#pragma unroll
            for (int j = 0; j < 3; ++j)
                if (d + j < D)
                    row[d + j] = v[j];
        }
    };
    if (part >= 0 || nsplit > 1) {
        // Unnormalised partial of one key range: (m, l, acc) into slot (row, part) for the
        // log-sum-exp merge (attn_merge2_kernel / attn_merge_kernel).
        if (rvalid) {
            const size_t slot = (nsplit > 1)
                                    ? ((size_t)h * Sq + myq) * nsplit + sp
                                    : ((size_t)(h - h0) * prows + (myq - split_first * BQ)) * 2 +
                                          part;
            if (hi == 0) {
                pm[slot] = m_run;
                pl[slot] = lt;
            }
            float *prow = pacc + slot * D;
#pragma unroll
            for (int db = 0; db < DP / 32; ++db)
#pragma unroll
                for (int i4 = 0; i4 < 4; ++i4) {
                    const int d = db * 32 + i4 * 8 + 4 * hi;
                    f32x4 v = {o[db][4 * i4], o[db][4 * i4 + 1], o[db][4 * i4 + 2], o[db][4 * i4 + 3]};
                    store4(prow, d, v);
                }
        }
#if ATTN_PHASE_STAMPS
        __builtin_amdgcn_s_waitcnt(0x0F70); // the partial stores have completed
        phase_stamp(w, lane, kPhaseSlots - 1);
#endif
        return;
    }
    const float inv = (lt > 0.f) ? 1.0f / lt : 0.f;
    bool staged = false;
    if constexpr (KT >= 16 * NW && DP <= 128 && UA != 2) { // rows of D < 8 fit one 32-byte piece
        if (!pack) {
            staged = true;
            // O leaves through LDS. Each wave writes its rows there in the accumulator layout (a
            // lane pair per row) and reads them back as row pieces of NCP 16-byte chunks, so that
            // each store instruction writes 64 / NCP rows x NCP consecutive chunks of O, where the
            // accumulator layout writes 32 rows x 32 bytes. The staging area is the K/V buffer pair
            // that the last tile left idle, (kt1 - kt0) & 1: every wave passed the barrier after
            // its last reader, and no DMA writes it any more. So no wave waits for the others to
            // finish the last tile: one that is done stores its rows while the others still run
            // P.V. Each wave owns OWB bytes of it, DBP blocks of 32 columns, and stages its DP
            // columns in passes of that width. Chunk c of row r sits at slot c ^ key(r), so that
            // the 16 lanes of a write pass (16 rows, one chunk) or of a read pass hit 16 distinct
            // 16-byte bank groups: with NCP % 16 == 0 every row starts at group 0 and key runs over
            // 16 rows; with NCP % 16 == 8 rows alternate between groups 0 and 8 and key runs over
            // row pairs. At DP = 256 the staging loop's registers add spills to a kernel already at
            // the register ceiling, and packed tiles (short, HBM-bound query blocks) lost 1-4% with
            // the extra LDS round trip, so those store directly.
            constexpr int OWB = 4 * KT * DP / NW; // staging bytes per wave
            constexpr int DBP = (OWB / 4096 < DP / 32) ? OWB / 4096 : DP / 32; // blocks per pass
            static_assert(DBP >= 1 && DP % 32 == 0, "staging area");
            constexpr int NCP = DBP * 8; // chunks per row piece
            static_assert(NCP % 8 == 0, "swizzle");
            auto key = [](int r) { return (NCP % 16 == 0) ? (r & 15) : ((r >> 1) & 7); };
            const int nb = ((kt1 - kt0) & 1) ^ (KH ? 1 : 0); // KH: the idle pair holds o halves
            float *ob = reinterpret_cast<float *>(w < NW / 2 ? &Ks[nb][0] : &Vs[nb][0]) +
                        (w % (NW / 2)) * (OWB / 4);
            const int row0 = qt * BQ + wr * 32; // the wave's first row of the head
            float *obase = O + ((size_t)h * Sq + (size_t)row0) * D;
#pragma unroll
            for (int pass = 0; pass < (DP / 32 + DBP - 1) / DBP; ++pass) {
                if (pass > 0)
                    lds_wave_fence(); // the last pass's reads are done before its slots are reused
#pragma unroll
                for (int j = 0; j < DBP; ++j) {
                    const int db = pass * DBP + j;
                    if (db < DP / 32) {
#pragma unroll
                        for (int i4 = 0; i4 < 4; ++i4) {
                            const int c = j * 8 + i4 * 2 + hi;
                            f32x4 v = {o[db][4 * i4] * inv, o[db][4 * i4 + 1] * inv,
                                       o[db][4 * i4 + 2] * inv, o[db][4 * i4 + 3] * inv};
                            float *dst = ob + l32 * (NCP * 4) + ((c ^ key(l32)) * 4);
                            *reinterpret_cast<f32x4 *>(dst) = v;
                        }
                    }
                }
                lds_wave_fence(); // this wave's rows are in LDS before any lane reads another's
                const int col0 = pass * DBP * 32;
#pragma unroll
                for (int q = 0; q < NCP / 2; ++q) {
                    const int f = q * 64 + lane, r = f / NCP, c = f - r * NCP;
                    const f32x4 v =
                        *reinterpret_cast<const f32x4 *>(ob + r * (NCP * 4) + ((c ^ key(r)) * 4));
                    if (row0 + r < Sq)
                        store4(obase + (size_t)r * D, col0 + c * 4, v);
                }
            }
        }
    }
    if (!staged && rvalid) {
        float *orow = O + qrow * D;
#pragma unroll
        for (int db = 0; db < DP / 32; ++db)
#pragma unroll
            for (int i4 = 0; i4 < 4; ++i4) {
                const int d = db * 32 + i4 * 8 + 4 * hi;
                f32x4 v = {o[db][4 * i4] * inv, o[db][4 * i4 + 1] * inv, o[db][4 * i4 + 2] * inv,
                           o[db][4 * i4 + 3] * inv};
                store4(orow, d, v);
            }
    }
#if ATTN_PHASE_STAMPS
    __builtin_amdgcn_s_waitcnt(0x0F70); // the O stores have completed
    phase_stamp(w, lane, kPhaseSlots - 1);
#endif
}

// ------------------------------------------------------------------------------------------
// Prefill, persistent (D % 8 == 0, D <= DP = 128, at least two rounds of 8-wave workgroups;
// causal grids as pairs of a heavy and a light query tile, whose key tiles add up to the same
// count for every pair). The fast kernel runs one (query head, 256-row tile) item per
// workgroup, and each item pays a fixed cost outside its key loop: all CUs load Q and the first
// key tile at once (an HBM burst), store O at once, and wait for the next workgroup's dispatch.
// Here one 8-wave workgroup per CU runs its items back to back, and the key-tile pipeline
// continues across them:
//   * the next item's first K/V tile is the last tile's ordinary LDS-DMA prefetch;
//   * the next item's Q (registers) is loaded during the last tile, after its S^T, so it lands
//     under the softmax and P.V (the last tile takes the row max, so no recompute needs the
//     old Q);
//   * an item's O leaves as NOST = 16 buffer stores per lane (8 with KH; rows past Sq fall
//     outside the descriptor's range: the count never depends on the data), issued in the next
//     item's first tile after that tile's DMA; the wait for the DMA then leaves exactly those
//     stores in flight (vmcnt(NOST): vector memory operations complete in issue order), so the O write
//     burst drains under the next tile's compute. The stores are non-temporal and each writes
//     whole 128-byte lines (store_o), so O does not evict the K/V tiles from L2.
// Items of a CU follow the non-persistent grid's rounds: XCD x = b % 8 holds the logical items
// [xb, xb + nx) (kv-head-major, as xcd_remap deals them) and its i-th workgroup takes
// xb + i, xb + i + R, ... (R workgroups per XCD), so each round of an XCD shares one kv head's
// K/V in its L2 as before. The tile code is the fast kernel's (8 waves, 32 rows each, 128-key
// tiles, lazy rescale with the sum test; causal masks compared against immediates), for
// row-major V only: a V^T variant needs 4 more offset registers for its DMA, spills them, and
// its spill reloads then wait for the DMA in flight (measured 0.5-2.6% slower than the V^T fast
// kernel on c3 and c4).
// KH (causal grids of exactly two 128-row query tiles per CU, where the fast kernel runs key
// halves in two rounds): each workgroup runs one heavy/light pair of 128-row items, waves w and
// w + 4 on the same 32 rows and the two 64-key halves of every tile. At each item's end the
// two halves are merged through LDS (kh_put / kh_combine) and each wave stores half of its rows'
// columns. A pair's key-tile counts add up to an odd number, so the item of even count runs
// first: the buffer order stays a compile-time constant without a padding tile.
// ------------------------------------------------------------------------------------------
// s_waitcnt operand (gfx9 encoding) that waits until at most n vector memory operations of
// the wave are in flight, with no wait on expcnt or lgkmcnt.
constexpr int waitcnt_vm(int n) { return 0x0F70 | (n & 15) | ((n >> 4) << 14); }


template <int DP, bool CAUSAL, bool KH>
__global__ __launch_bounds__(512, 1) void attn_prefill_persist_kernel(
    const uint16_t *__restrict__ Q, const uint16_t *__restrict__ K,
    const uint16_t *__restrict__ V, float *__restrict__ O, int Hq, int Hkv, int Sq, int Sk, int D,
    float c, int nqt, int nitems, int nwg) {
    static_assert(DP % 32 == 0 && DP <= 128, "tile shape");
    static_assert(!KH || (CAUSAL && DP == 128), "key halves: causal pairs at DP = 128");
    // KH: items of 128 rows, waves w and w + 4 (one SIMD) on the same 32 rows and the two
    // 64-key halves of every tile (NR row blocks, KW keys per wave and tile).
    constexpr int KT = 128, NW = 8, NR = KH ? NW / 2 : NW, KW = KH ? KT / 2 : KT, BQ = NR * 32;
    // One variable per tile buffer: the compiler tells LDS accesses apart by variable only, so
    // with the two buffers of an array it would make each tile's first reads wait for the DMA
    // of the next tile into the other buffer.
    __shared__ __attribute__((aligned(1024))) uint16_t Ks0[KT * DP];
    __shared__ __attribute__((aligned(1024))) uint16_t Ks1[KT * DP];
    __shared__ __attribute__((aligned(1024))) uint16_t Vs0[KT * DP];
    __shared__ __attribute__((aligned(1024))) uint16_t Vs1[KT * DP];
    auto kbuf = [&](int buf) -> uint16_t * { return buf ? Ks1 : Ks0; }; // buf: a constant
    auto vbuf = [&](int buf) -> uint16_t * { return buf ? Vs1 : Vs0; };
    __shared__ float kh_ml[KH ? NW * 128 : 1]; // KH: (m, l) of each lane, for its partner wave

    const int g = Hq / Hkv;
    const int b = wg_id_x(), x = b & 7, xi = b >> 3, R = nwg >> 3; // nwg % 8 == 0
    // nitems units (items, or causal pairs of items) dealt to the XCDs in contiguous runs.
    const int per = nitems >> 3, rem = nitems & 7;
    const int xb = (x < rem) ? x * (per + 1) : rem * (per + 1) + (x - rem) * per;
    const int nx = per + (x < rem ? 1 : 0);
    const int nunits = (xi < nx) ? (nx - xi + R - 1) / R : 0;
    const int nmine = CAUSAL ? 2 * nunits : nunits; // items of this workgroup
    if (nmine == 0)
        return;
    // Key tiles of an item: all of them, or (causal) those up to its last row's limit,
    // Sk - Sq + its last row (Sk >= Sq). Even for every item (host), except with KH.
    auto nkt_of = [&](int qt) {
        if constexpr (CAUSAL)
            return (Sk - Sq + min(Sq - 1, qt * BQ + BQ - 1)) / KT + 1;
        return (Sk + KT - 1) / KT;
    };
    // Item k of this workgroup: query head h and query tile qt (BQ rows). Non-causal: the fast
    // kernel's order (kv head, then tile, then the g heads of the group). Causal (nqt even):
    // unit P is the pair of tiles nqt-1-p and p of one head (kv head, then p, then the head),
    // whose key tiles add up to the same count for every p, run heavy first: each workgroup
    // gets the same number of pairs and so the same work. KH (Sq % 128 == 0): the pair's
    // counts add up to an odd number, and the tile of even count runs first.
    auto item = [&](int k, int &h, int &qt) {
        if constexpr (CAUSAL) {
            const int np = nqt >> 1;
            const int P = xb + xi + (k >> 1) * R;
            const int uu = P / (g * np);
            const int rr = P - uu * (g * np);
            const int pp = rr / g;
            const bool swap = KH && (nkt_of(nqt - 1 - pp) & 1);
            qt = __builtin_amdgcn_readfirstlane(((k & 1) != swap) ? pp : nqt - 1 - pp);
            h = __builtin_amdgcn_readfirstlane(uu * g + (rr - pp * g));
        } else {
            const int L = xb + xi + k * R;
            const int uu = L / (g * nqt);
            const int rr = L - uu * (g * nqt);
            qt = __builtin_amdgcn_readfirstlane(rr / g);
            h = __builtin_amdgcn_readfirstlane(uu * g + (rr - (rr / g) * g));
        }
    };

    const int tid = threadIdx.x, lane = tid & 63; // a library call on purpose: see wi_id_x
    // & 7: the compiler then knows each wave's DMA blocks stay inside one tile buffer
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6) & 7;
    const int wr = KH ? (w & (NR - 1)) : w; // the wave's 32-row block of the item
    const int kh = KH ? (w >> 2) : 0;       // and its half of each key tile
    const int l32 = lane & 31, hi = lane >> 5, g16 = lane >> 4, i16 = lane & 15;

    const uint32_t qbytes = (uint32_t)Sq * (uint32_t)D * 2u; // one head of Q (O: twice; < 2^31)
    // Q rows of item (h, qt) for this lane's operand layout: 16-byte buffer loads, rows past Sq
    // and columns past D outside the descriptor's range (zeros), DP/16 loads whatever the data.
    bf16x8 qb[DP / 16];
    auto load_q = [&](int h, int qt) __attribute__((always_inline)) {
        const __amdgpu_buffer_rsrc_t rq = make_rsrc(Q + (size_t)h * Sq * D, qbytes);
        // r is made opaque here (and in store_o, and kbase in the last tile's mask): the
        // offsets and key compares are the same for every item, and hoisted out of the item
        // loop they would hold their registers (64 lane masks, 24 offsets) for the whole kernel.
        int r = wr * 32 + l32;
        asm volatile("" : "+v"(r));
        r += qt * BQ; // row of the head
        const int dlim = (r < Sq) ? D : 0;
#pragma unroll
        for (int kk = 0; kk < DP / 16; ++kk) {
            const int col = kk * 16 + hi * 8;
            const uint32_t off = (col < dlim) ? (uint32_t)(r * D + col) * 2u : 0x80000000u;
            qb[kk] = as_bf16x8(__builtin_bit_cast(
                u32x4, __builtin_amdgcn_raw_buffer_load_b128(rq, off, 0, 0)));
        }
    };

    // LDS-DMA source offsets of this wave's blocks (layouts as in attn_prefill_fast_kernel).
    constexpr int NI = KT * DP / 512;
    constexpr int PW = NI / NW;
    static_assert(PW * NW == NI && PW >= 1, "DMA blocks per wave");
    const uint32_t kvbytes = (uint32_t)Sk * D * 2;
    uint32_t kso[PW], vso[PW];
#pragma unroll
    for (int k = 0; k < PW; ++k) {
        const int bb = (w * PW + k) * 1024 + 16 * lane;
        {
            const int rg = bb / (16 * DP), wi = bb % (16 * DP);
            const int r = rg * 8 + (wi % 256) / 32;
            const int cc = 2 * (wi / 256) + (((wi % 32) / 16) ^ (rg & 1));
            kso[k] = (cc * 8 < D) ? (uint32_t)(r * D * 2 + cc * 16) : 0x80000000u;
        }
        {
            const int rgv = bb / (8 * DP), wi = bb % (8 * DP);
            const int r = rgv * 4 + (wi % 256) / 64;
            const int cc = 4 * (wi / 256) + (wi % 64) / 16;
            vso[k] = (cc * 8 < D) ? (uint32_t)(r * D * 2 + cc * 16) : 0x80000000u;
        }
    }
    // K and V tile kt of kv head u into LDS buffer buf: 2 * PW DMA instructions.
    auto dma_kv = [&](int u, int kt, int buf) __attribute__((always_inline)) {
        const uint32_t toff = (uint32_t)kt * KT * D * 2;
        const __amdgpu_buffer_rsrc_t rk =
            make_rsrc(K + (size_t)u * Sk * D + (size_t)kt * KT * D, kvbytes - toff);
        const __amdgpu_buffer_rsrc_t rv =
            make_rsrc(V + (size_t)u * Sk * D + (size_t)kt * KT * D, kvbytes - toff);
#pragma unroll
        for (int k = 0; k < PW; ++k)
            dma16<0>(rk, &kbuf(buf)[(w * PW + k) * 512], kso[k]);
#pragma unroll
        for (int k = 0; k < PW; ++k)
            dma16<0>(rv, &vbuf(buf)[(w * PW + k) * 512], vso[k]);
    };
    // Column blocks (32 wide) of O that one wave stores: all, or (KH) its half of them.
    constexpr int NDB = KH ? DP / 64 : DP / 32;
    constexpr int NOST = NDB * 4; // vector memory instructions of one store_o

    const int kperm = (l32 & ~12) | ((l32 & 4) << 1) | ((l32 & 8) >> 1);
    const int kfo = (kperm >> 3) * 8 * DP + (kperm & 7) * 16 + ((hi ^ ((kperm >> 3) & 1)) * 8);
    constexpr int KSUB = 32 * DP, KDK = 128;
    const int vfo =
        hi * 8 * DP + (i16 >> 2) * 32 + (2 * (g16 & 1) + ((i16 & 3) >> 1)) * 8 + (i16 & 1) * 4;

    float m_run = kNegInf, l_run = 0.f;
    f32x16 o[DP / 32];
#pragma unroll
    for (int db = 0; db < DP / 32; ++db)
#pragma unroll
        for (int i = 0; i < 16; ++i)
            o[db][i] = 0.f;
    f32x16 s[KW / 32];
    bf16x8 pk[KW / 16];
    bf16x8 va[2][DP / 32];

    // S^T = K_tile . Q^T (the next sub-tile's K fragments read between this one's MFMAs).
    auto qk = [&](int buf) __attribute__((always_inline)) {
        const uint16_t *kb0 = &kbuf(buf)[kfo + kh * (KW / 32) * KSUB];
        bf16x8 ka[2][DP / 16];
#pragma unroll
        for (int kk = 0; kk < DP / 16; ++kk)
            ka[0][kk] = as_bf16x8(*reinterpret_cast<const u32x4 *>(kb0 + kk * KDK));
        __builtin_amdgcn_sched_group_barrier(0x100, DP / 16, 0);
#pragma unroll
        for (int t = 0; t < KW / 32; ++t) {
#pragma unroll
            for (int i = 0; i < 16; ++i)
                s[t][i] = 0.f;
#pragma unroll
            for (int kk = 0; kk < DP / 16; ++kk) {
                s[t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ka[t & 1][kk], qb[kk], s[t], 0, 0, 0);
                if (t + 1 < KW / 32)
                    ka[(t + 1) & 1][kk] = as_bf16x8(
                        *reinterpret_cast<const u32x4 *>(kb0 + (t + 1) * KSUB + kk * KDK));
            }
#pragma unroll
            for (int kk = 0; kk < DP / 16; ++kk) {
                __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                if (t + 1 < KW / 32)
                    __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
            }
        }
    };
    // Keys past a row's limit take -inf: Sk - 1, or (causal) min(Sk - 1, Sk - Sq + row). The
    // wave's rows qmin .. qmin + 31 of item tile qt have limits from lo (its first row's) to
    // wmax (its last valid row's; -1 when it has none); sub-tiles wholly at or below lo are
    // skipped and sub-tiles wholly past wmax set at once (wave-uniform tests), so only a
    // sub-tile between the two is compared key by key.
    auto lims = [&](int qt, int &lo, int &wmax) {
        if constexpr (CAUSAL) {
            const int qmin = qt * BQ + wr * 32;
            lo = __builtin_amdgcn_readfirstlane(min(Sk - 1, Sk - Sq + qmin));
            wmax = __builtin_amdgcn_readfirstlane(
                qmin < Sq ? min(Sk - 1, Sk - Sq + min(Sq - 1, qmin + 31)) : -1);
        } else {
            lo = Sk - 1;
            wmax = Sk - 1;
        }
    };
    auto mask = [&](int kbase, int qt) __attribute__((always_inline)) {
        int lo, wmax;
        lims(qt, lo, wmax);
        if (kbase + KW - 1 > lo) {
            int lim = Sk - 1;
            if constexpr (CAUSAL) {
                int r = wr * 32 + l32;
                asm volatile("" : "+v"(r));
                lim = min(Sk - 1, Sk - Sq + qt * BQ + r);
            }
#pragma unroll
            for (int t = 0; t < KW / 32; ++t) {
                const int k0t = kbase + t * 32;
                if (k0t + 31 <= lo)
                    continue;
                if (k0t > wmax) {
#pragma unroll
                    for (int i = 0; i < 16; ++i)
                        s[t][i] = kNegInf;
                    continue;
                }
                if constexpr (CAUSAL) {
                    // key = k0t + 8 hi + 16 (i >> 3) + (i & 7) > lim, against one register and
                    // immediates (with the keys in registers the causal variant spills)
                    const int rel = lim - k0t - 8 * hi;
#pragma unroll
                    for (int i = 0; i < 16; ++i)
                        if (16 * (i >> 3) + (i & 7) > rel)
                            s[t][i] = kNegInf;
                } else {
#pragma unroll
                    for (int i = 0; i < 16; ++i)
                        if (k0t + 16 * (i >> 3) + 8 * hi + (i & 7) > lim)
                            s[t][i] = kNegInf;
                }
            }
        }
    };
    // fresh: an item's first tile, where l and o are still zero (o is then written, not
    // accumulated, by that tile's P.V): m rises with no rescale to apply.
    auto row_max = [&](auto fresh) __attribute__((always_inline)) {
        float mt[KW / 32];
#pragma unroll
        for (int t = 0; t < KW / 32; ++t) {
            float m = max3f(s[t][0], s[t][1], s[t][2]);
#pragma unroll
            for (int i = 3; i < 15; i += 2)
                m = max3f(m, s[t][i], s[t][i + 1]);
            mt[t] = fmaxf(m, s[t][15]);
        }
        float mx = mt[0];
#pragma unroll
        for (int j = 1; j < KW / 32; j += 2)
            mx = (j + 1 < KW / 32) ? max3f(mx, mt[j], mt[j + 1]) : fmaxf(mx, mt[j]);
        mx = max_xor32(mx);
        const bool raise = mx > m_run;
        if constexpr (decltype(fresh)::value) {
            m_run = raise ? mx : m_run;
        } else if (__builtin_amdgcn_ballot_w64(raise) != 0) {
            const float mnew = raise ? mx : m_run;
            const float alpha = (mnew == m_run) ? 1.0f : fast_exp2((m_run - mnew) * c);
            l_run *= alpha;
#pragma unroll
            for (int db = 0; db < DP / 32; ++db)
                o[db] *= alpha;
            m_run = mnew;
        }
    };
    auto exps = [&]() __attribute__((always_inline)) -> float {
        const float mc = (m_run == kNegInf) ? 0.f : m_run * c;
        float ps[KW / 16];
#pragma unroll
        for (int t = 0; t < KW / 32; ++t)
#pragma unroll
            for (int hh = 0; hh < 2; ++hh) {
                float p[8];
#pragma unroll
                for (int j = 0; j < 8; ++j) {
                    p[j] = fast_exp2(fmaf(s[t][8 * hh + j], c, -mc));
                    pk[2 * t + hh][j] = (__bf16)p[j];
                }
                ps[2 * t + hh] = ((p[0] + p[1]) + (p[2] + p[3])) + ((p[4] + p[5]) + (p[6] + p[7]));
            }
        float psum = 0.f;
#pragma unroll
        for (int j = 0; j < KW / 16; ++j)
            psum += ps[j];
        return psum;
    };
    auto vfrag = [&](int buf, int cc, int db) -> bf16x8 {
        cc += kh * (KW / 16); // the wave's key half of the tile (KH)
        const uint16_t *vb = &vbuf(buf)[vfo + cc * 16 * DP + db * 128];
        return join_tr(lds_read_tr(vb), lds_read_tr(vb + 4 * DP));
    };
    auto pv_first = [&](int buf) {
#pragma unroll
        for (int db = 0; db < DP / 32; ++db)
            va[0][db] = vfrag(buf, 0, db);
    };
    // fresh (an item's first tile): the first 16-key chunk starts the accumulators from zero.
    auto pv = [&](int buf, auto fresh) {
#pragma unroll
        for (int cc = 0; cc < KW / 16; ++cc) {
#pragma unroll
            for (int db = 0; db < DP / 32; ++db) {
                const f32x16 acc =
                    (decltype(fresh)::value && cc == 0) ? f32x16{} : o[db];
                o[db] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(va[cc & 1][db], pk[cc], acc, 0, 0,
                                                               0);
                if (cc + 1 < KW / 16)
                    va[(cc + 1) & 1][db] = vfrag(buf, cc + 1, db);
            }
#pragma unroll
            for (int db = 0; db < DP / 32; ++db) {
                __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                if (cc + 1 < KW / 16)
                    __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
            }
        }
    };
    // O of item (h, qt) from (o, l): NOST buffer stores whatever the data (none lands when
    // !valid: every offset is then outside the descriptor's range). KH: o[0 .. NDB) holds
    // (kh_combine) the wave's column blocks kh * NDB .. of the rows, the partner wave's the
    // others.
    // Each store writes whole 128-byte lines, non-temporally: a lane holds 16-byte chunks
    // hi, 2 + hi, 4 + hi, 6 + hi (i4 = 0..3) of its row's 32-column block, so two lane/register
    // bit swaps (row bit 4 with i4 bit 1 by v_permlane16_swap, row bit 3 with i4 bit 0 by two
    // bank-masked DPP moves from lane ^ 8) leave each register holding, per lane, chunk
    // c8 = hi + 2 (lane bit 3) + 4 (lane bit 4) of row (lane & 7) + 8 s0 + 16 s1: one store then
    // covers 8 rows x 128 bytes. Partial-line stores left through L2 (whole-line ones with the
    // ordinary policy measured within 1%), where they evicted the K/V tiles of the next items;
    // non-temporal partial lines were written back piecemeal (2.35x the bytes).
    auto store_o = [&](int h, int qt, bool valid) __attribute__((always_inline)) {
        const float lt = sum_xor32(l_run);
        const float inv = (lt > 0.f) ? 1.0f / lt : 0.f;
        const __amdgpu_buffer_rsrc_t ro = make_rsrc(O + (size_t)h * Sq * D, 2u * qbytes);
        int r = wr * 32 + (lane & 7);
        asm volatile("" : "+v"(r));
        r += qt * BQ; // row of the head for s0 = s1 = 0
        const int c8 = hi + 2 * ((lane >> 3) & 1) + 4 * ((lane >> 4) & 1);
#pragma unroll
        for (int db = 0; db < NDB; ++db) {
            float x[4][4]; // [s1 s0][j] after the swaps; [i4][j] before
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                float v[4];
#pragma unroll
                for (int i4 = 0; i4 < 4; ++i4)
                    v[i4] = o[db][4 * i4 + j] * inv;
#pragma unroll
                for (int a = 0; a < 2; ++a) { // row bit 4 <-> i4 bit 1
                    const auto sw = __builtin_amdgcn_permlane16_swap(
                        __builtin_bit_cast(unsigned, v[a]), __builtin_bit_cast(unsigned, v[a + 2]),
                        false, false);
                    v[a] = __builtin_bit_cast(float, (unsigned)sw[0]);
                    v[a + 2] = __builtin_bit_cast(float, (unsigned)sw[1]);
                }
#pragma unroll
                for (int s1 = 0; s1 < 2; ++s1) { // row bit 3 <-> i4 bit 0
                    // row_ror:8 reads lane ^ 8; the bank mask writes only the lanes with bit 3
                    // set (banks 2, 3 of each row: 0xc) or clear (0x3), the others keep old.
                    const int X = __builtin_bit_cast(int, v[2 * s1]);
                    const int Y = __builtin_bit_cast(int, v[2 * s1 + 1]);
                    x[2 * s1][j] =
                        __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(X, Y, 0x128, 0xf, 0xc, false));
                    x[2 * s1 + 1][j] =
                        __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(Y, X, 0x128, 0xf, 0x3, false));
                }
            }
#pragma unroll
            for (int q = 0; q < 4; ++q) { // q = 2 s1 + s0: rows + 8 s0 + 16 s1
                const int rq = r + 8 * (q & 1) + 16 * (q >> 1);
                // One column limit per lane (D, or 0 for a row to drop): a single compare per
                // store keeps the stores free of branches.
                const int dlim = (valid & (rq < Sq)) ? D : 0;
                const int d = (kh * NDB + db) * 32 + 4 * c8;
                const f32x4 v = {x[q][0], x[q][1], x[q][2], x[q][3]};
                const uint32_t off = (d < dlim) ? (uint32_t)(rq * D + d) * 4u : 0x80000000u;
                __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, v), ro, off, 0,
                                                       2 /* nt */);
            }
        }
    };
    // KH hand-over at an item's end, once every wave is past the barrier after the item's last
    // tile (buffer pair buf): kh_put leaves each wave's (m, l) in kh_ml and the NDB column
    // blocks its partner (w ^ 4: same rows, other key half) stores in the partner's own DMA
    // blocks of buf (PW KB of K, then PW KB of V; 16 fp32 per lane and block, in lane order);
    // after a barrier kh_combine merges them with log-sum-exp weights against the larger m (a
    // half with no admissible key has m = -inf: weight 0) into o[0 .. NDB). Each wave reads back
    // only its own DMA blocks, which its own next DMA into buf rewrites after those reads have
    // returned. Blocks are chosen by value (selects on kh), not by a register index that
    // depends on kh, which would move o to scratch memory.
    static_assert(!KH || PW * 512 * 2 == 16 * 64 * 4, "hand-over block = a wave's DMA blocks");
    auto kh_area = [&](int buf, int wave, int j) __attribute__((always_inline)) -> float * {
        return reinterpret_cast<float *>(&(j ? vbuf(buf) : kbuf(buf))[wave * PW * 512]);
    };
    auto kh_put = [&](int buf) __attribute__((always_inline)) {
        if constexpr (!KH)
            return;
        kh_ml[w * 128 + lane] = m_run;
        kh_ml[w * 128 + 64 + lane] = l_run;
#pragma unroll
        for (int j = 0; j < NDB; ++j) {
            const f32x16 t = kh ? o[j] : o[(NDB + j) % (DP / 32)]; // the partner's block j
#pragma unroll
            for (int i4 = 0; i4 < 4; ++i4) {
                const f32x4 v = {t[4 * i4], t[4 * i4 + 1], t[4 * i4 + 2], t[4 * i4 + 3]};
                *reinterpret_cast<f32x4 *>(kh_area(buf, w ^ 4, j) + (i4 * 64 + lane) * 4) = v;
            }
        }
    };
    auto kh_combine = [&](int buf) __attribute__((always_inline)) {
        if constexpr (!KH)
            return;
        const int p = w ^ 4;
        const float m2 = kh_ml[p * 128 + lane], l2 = kh_ml[p * 128 + 64 + lane];
        // Key half 0's and half 1's values, in that order in both waves: both get the same l.
        const float m0 = kh ? m2 : m_run, m1 = kh ? m_run : m2;
        const float l0 = kh ? l2 : l_run, l1 = kh ? l_run : l2;
        const float mn = fmaxf(m0, m1);
        const float a0 = (m0 == kNegInf) ? 0.f : fast_exp2((m0 - mn) * c);
        const float a1 = (m1 == kNegInf) ? 0.f : fast_exp2((m1 - mn) * c);
        l_run = __builtin_fmaf(l0, a0, l1 * a1);
#pragma unroll
        for (int j = 0; j < NDB; ++j) {
            const f32x16 t = kh ? o[(NDB + j) % (DP / 32)] : o[j]; // this wave's block j
#pragma unroll
            for (int i4 = 0; i4 < 4; ++i4) {
                const f32x4 v =
                    *reinterpret_cast<const f32x4 *>(kh_area(buf, w, j) + (i4 * 64 + lane) * 4);
#pragma unroll
                for (int jj = 0; jj < 4; ++jj) {
                    const float x0 = kh ? v[jj] : t[4 * i4 + jj];
                    const float x1 = kh ? t[4 * i4 + jj] : v[jj];
                    o[j][4 * i4 + jj] = __builtin_fmaf(x0, a0, x1 * a1);
                }
            }
        }
    };

    // Phase stamps (ATTN_PHASE_STAMPS builds): slot 0 at entry, 1 when the first item's Q and
    // tile are in, four per item (its start, the end of its first tile, the start and the end of
    // its last tile), the last slot once the final O stores have completed.
    phase_stamp(w, lane, 0);
    {
        int h0, qt0;
        item(0, h0, qt0);
        load_q(h0, qt0);
        dma_kv(__builtin_amdgcn_readfirstlane(h0 / g), 0, 0);
    }
    __builtin_amdgcn_s_waitcnt(0x0F70); // vmcnt(0): Q and tile 0 of the first item
    __syncthreads();
    phase_stamp(w, lane, 1);
    // One key tile kt of item k (kv head u, query tile qt): FIRST (kt = 0: the previous item's
    // O leaves, then the row max), LAST (kt = nkt - 1: the next item's tile 0 DMA and Q loads,
    // the mask, the row max) or neither (the sum test, a rare recompute). Item coordinates are
    // recomputed from the item index where needed rather than carried in registers.
    // Every item's nkt is even (host), so tile kt uses LDS buffer kt & 1 (KH: the item order
    // below fixes the buffers of odd counts): each step's buffers are constants, which lets the
    // compiler tell this tile's LDS reads from the next tile's DMA (with a run-time buffer index
    // it waits for that DMA before the first read). FIRST and LAST are one step for a KH item of
    // one key tile. Causal: FIRST and middle tiles are masked too where they reach past the
    // wave's first row's limit.
    auto step = [&](int u, int qt, int kt, int k, auto kbuf, auto kfirst, auto klast)
        __attribute__((always_inline)) {
        constexpr bool FIRST = decltype(kfirst)::value, LAST = decltype(klast)::value;
        constexpr int buf = decltype(kbuf)::value;
        const bool more = k + 1 < nmine;
        if constexpr (KH && FIRST) {
            // The previous item's key halves (left in buffer pair buf ^ 1 after its last tile),
            // before the DMA below rewrites that pair.
            if (k > 0) {
                kh_combine(buf ^ 1);
                __builtin_amdgcn_s_waitcnt(0xC07F); // lgkmcnt(0): the reads have returned
            }
        }
        // The next tile's DMA, the oldest vector memory operation of the tile.
        if (!LAST) {
            dma_kv(u, kt + 1, buf ^ 1);
        } else if (more) {
            int hn, qtn;
            item(k + 1, hn, qtn);
            dma_kv(__builtin_amdgcn_readfirstlane(hn / g), 0, buf ^ 1);
        }
        // The previous item's O (after this tile's DMA; for the first item the stores are
        // issued but land nowhere, which keeps this tile free of branches), then a fresh state.
        // KH issues them after this tile's S^T instead (its registers leave room to keep its O
        // half live across it): 0-2% faster, bit-identical.
        auto leave_o = [&]() __attribute__((always_inline)) {
            int hp, qtp;
            item(k > 0 ? k - 1 : 0, hp, qtp);
            store_o(hp, qtp, k > 0);
            m_run = kNegInf;
            l_run = 0.f; // o: written by this tile's P.V
        };
        if constexpr (FIRST && !KH)
            leave_o();
        int kbase = kt * KT;
        if constexpr (LAST || CAUSAL)
            asm volatile("" : "+s"(kbase));
        kbase += kh * KW; // the wave's first key of the tile
        int lo, wmax;
        lims(qt, lo, wmax);
        // Causal: a wave whose rows see no key of the last tile (the first half of the waves
        // when the query tile's limits are 128-key aligned) skips its softmax and P.V there
        // but still computes S^T: skipping that too made the compiler spill about 100
        // registers.
        qk(buf);
        if constexpr (FIRST && KH)
            leave_o();
        pv_first(buf);
        // The fast kernel's phase order: S^T, then the softmax, then P.V (letting the compiler
        // move the first sub-tile's exponentials between the later sub-tiles' MFMAs measured
        // slower: in-wave VALU between MFMAs delays the wave's own S^T).
        __builtin_amdgcn_sched_barrier(0);
        if (LAST && more) { // qb is free: this tile takes the row max, with no recompute
            int hn, qtn;
            item(k + 1, hn, qtn);
            load_q(hn, qtn);
        }
        if (FIRST || LAST) {
            if (!(CAUSAL && LAST) || kbase <= wmax) {
                if (LAST || CAUSAL)
                    mask(kbase, qt);
                row_max(std::integral_constant<bool, FIRST>{});
                l_run += exps();
            }
        } else {
            if constexpr (CAUSAL)
                mask(kbase, qt);
            float psum = exps();
            if (__builtin_expect(__builtin_amdgcn_ballot_w64(!(psum <= kSumCap)) != 0, 0)) {
                qk(buf);
                pv_first(buf);
                if constexpr (CAUSAL)
                    mask(kbase, qt);
                row_max(std::false_type{});
                psum = exps();
            }
            l_run += psum;
        }
        if (!(CAUSAL && LAST) || kbase <= wmax) {
            pv(buf, std::integral_constant<bool, FIRST>{});
        } else if constexpr (FIRST) {
            // (KH: an item of one key tile whose half has no key for this wave's rows.)
#pragma unroll
            for (int db = 0; db < DP / 32; ++db)
                o[db] = f32x16{};
        }
        if (!LAST || more) {
            // Wait for the next tile's DMA only: the O stores of tile 0 (NOST) are younger and
            // stay in flight. The last tile waits for everything (the next item's Q loads, issued
            // mid-tile, have landed by then), so each item starts with no vector memory operation
            // in flight: with one still pending at the item loop's head the compiler waits for it
            // before the first tile's LDS reads.
            if (FIRST && !LAST)
                __builtin_amdgcn_s_waitcnt(waitcnt_vm(NOST));
            else
                __builtin_amdgcn_s_waitcnt(0x0F70);
            __syncthreads();
        }
        if constexpr (KH && LAST) {
            if (!more)
                __syncthreads(); // every wave is done with buffer pair buf
            kh_put(buf);
            __syncthreads();
        }
    };
    using B0 = std::integral_constant<int, 0>;
    using B1 = std::integral_constant<int, 1>;
    // KH: one unit per workgroup (host), its item of even key-tile count first (item): that
    // one's tiles alternate from buffer 0 and end in buffer 1, so the other, of odd count,
    // starts in buffer 0 and ends there too, and every step's buffers stay constants. The two
    // items are written out rather than looped over: in a loop the compiler keeps values of
    // every step instance live across it, and spills.
    if constexpr (KH) {
        {
            int h, qt;
            item(0, h, qt);
            const int u = __builtin_amdgcn_readfirstlane(h / g);
            const int nkt = __builtin_amdgcn_readfirstlane(nkt_of(qt));
            phase_stamp(w, lane, 2);
            step(u, qt, 0, 0, B0{}, std::true_type{}, std::false_type{});
            phase_stamp(w, lane, 3);
            for (int kt = 1; kt + 1 < nkt; kt += 2) {
                step(u, qt, kt, 0, B1{}, std::false_type{}, std::false_type{});
                step(u, qt, kt + 1, 0, B0{}, std::false_type{}, std::false_type{});
            }
            phase_stamp(w, lane, 4);
            step(u, qt, nkt - 1, 0, B1{}, std::false_type{}, std::true_type{});
            phase_stamp(w, lane, 5);
        }
        {
            int h, qt;
            item(1, h, qt);
            const int u = __builtin_amdgcn_readfirstlane(h / g);
            const int nkt = __builtin_amdgcn_readfirstlane(nkt_of(qt));
            phase_stamp(w, lane, 6);
            if (nkt == 1) {
                step(u, qt, 0, 1, B0{}, std::true_type{}, std::true_type{});
                phase_stamp(w, lane, 7);
                phase_stamp(w, lane, 8);
            } else {
                step(u, qt, 0, 1, B0{}, std::true_type{}, std::false_type{});
                phase_stamp(w, lane, 7);
                for (int kt = 1; kt + 2 < nkt; kt += 2) {
                    step(u, qt, kt, 1, B1{}, std::false_type{}, std::false_type{});
                    step(u, qt, kt + 1, 1, B0{}, std::false_type{}, std::false_type{});
                }
                step(u, qt, nkt - 2, 1, B1{}, std::false_type{}, std::false_type{});
                phase_stamp(w, lane, 8);
                step(u, qt, nkt - 1, 1, B0{}, std::false_type{}, std::true_type{});
            }
            phase_stamp(w, lane, 9);
        }
    }
    for (int k = 0; !KH && k < nmine; ++k) {
        int h, qt;
        item(k, h, qt);
        const int u = __builtin_amdgcn_readfirstlane(h / g);
        const int nkt = __builtin_amdgcn_readfirstlane(nkt_of(qt));
        phase_stamp(w, lane, 2 + 4 * k);
        step(u, qt, 0, k, B0{}, std::true_type{}, std::false_type{});
        phase_stamp(w, lane, 3 + 4 * k);
        for (int kt = 1; kt + 1 < nkt; kt += 2) {
            step(u, qt, kt, k, B1{}, std::false_type{}, std::false_type{});
            step(u, qt, kt + 1, k, B0{}, std::false_type{}, std::false_type{});
        }
        phase_stamp(w, lane, 4 + 4 * k);
        step(u, qt, nkt - 1, k, B1{}, std::false_type{}, std::true_type{});
        phase_stamp(w, lane, 5 + 4 * k);
    }
    {
        int hl, qtl;
        item(nmine - 1, hl, qtl);
        if constexpr (KH)
            kh_combine(0); // the last tile's buffer pair
        store_o(hl, qtl, true);
    }
#if ATTN_PHASE_STAMPS
    __builtin_amdgcn_s_waitcnt(0x0F70); // the final O stores have completed
    phase_stamp(w, lane, kPhaseSlots - 1);
#endif
}

// Row padding (floats) of the decode kernels' 4-wave merge area [4][16][DP + kMergePad]. Each
// lane stores its O^T registers (rows r16 = lane % 16, columns 16db + 4grp .. +3) as 16 bytes;
// with unpadded rows (DP = 64 or 128 floats: a multiple of the 64 four-byte banks) the 16 lanes
// of a group hit the same 4 banks, a 16-way conflict (3.0 M conflict cycles per c2 decode
// dispatch); 4 floats of padding move each row 4 banks on, so the 16 lanes cover all 64.
constexpr int kMergePad = 4;

// The decode kernels' 4-wave merge of one 16-row block (its waves' o in om, their (m, l) in red_m and
// red_l): rows row .. row + Mb - 1 of kv head u's g * Sq, into O (nsplit == 1) or the partial slots of
// split sp. A thread takes 4 columns at a time: with single columns and a runtime division per
// element, a 16-row block took 8 passes over 4 exponentials and two divisions each, which was
// felt on short key ranges: 32 heads x 4 rows over 2000 keys at D = 64 9.2 -> 8.1 us, 128 kv heads x
// 64 rows over 1000 keys 26.1 -> 23.9.
template <int DP>
__device__ __forceinline__ void decode_merge(const float *om, const float (*red_m)[16],
                                             const float (*red_l)[16], float *__restrict__ O,
                                             float *__restrict__ pm, float *__restrict__ pl,
                                             float *__restrict__ pacc, int tid, int row, int Mb,
                                             int u, int g, int Sq, int D, float c, int nsplit,
                                             int sp) {
    for (int idx = tid; idx < Mb * (DP / 4); idx += 256) {
        const int r = idx / (DP / 4), d = 4 * (idx % (DP / 4));
        if (d >= D)
            continue;
        float mx = kNegInf;
#pragma unroll
        for (int ww = 0; ww < 4; ++ww)
            mx = fmaxf(mx, red_m[ww][r]);
        const float muse = (mx == kNegInf) ? 0.f : mx;
        f32x4 acc = {0.f, 0.f, 0.f, 0.f};
        float lsum = 0.f;
#pragma unroll
        for (int ww = 0; ww < 4; ++ww) {
            const float wgt = fast_exp2((red_m[ww][r] - muse) * c);
            const f32x4 x =
                *reinterpret_cast<const f32x4 *>(&om[(ww * 16 + r) * (DP + kMergePad) + d]);
#pragma unroll
            for (int j = 0; j < 4; ++j)
                acc[j] += wgt * x[j];
            lsum += wgt * red_l[ww][r];
        }
        const int gi = (row + r) / Sq;
        const size_t orow = (size_t)(u * g + gi) * Sq + (row + r - gi * Sq);
        float *dst;
        if (nsplit == 1) {
            const float inv = (lsum > 0.f) ? 1.0f / lsum : 0.f;
#pragma unroll
            for (int j = 0; j < 4; ++j)
                acc[j] *= inv;
            dst = O + orow * D + d;
        } else {
            const size_t slot = orow * nsplit + sp;
            if (d == 0) {
                pm[slot] = mx;
                pl[slot] = lsum;
            }
            dst = pacc + slot * D + d;
        }
        if (d + 4 <= D) {
            *reinterpret_cast<f32x4_a4 *>(dst) = acc;
        } else {
#pragma unroll
            for (int j = 0; j < 3; ++j)
                if (d + j < D)
                    dst[j] = acc[j];
        }
    }
}

// ------------------------------------------------------------------------------------------
// Decode (split-K). One workgroup per (kv head u, split sp, 16-row block rb) serves up to 16 of
// the M = g*Sq <= 64 query rows of that kv head from one read of its K/V range
// [sp*kps, min(sp*kps+kps, Sk)) (the row blocks of a range share it through L2). Waves
// take interleaved 32-key tiles, starting at a workgroup-dependent 128-key step; per tile
// (v_mfma_f32_16x16x32_bf16):
//   S^T[key][row] = K . Q^T  (A = K rows loaded from global straight into the operand layout)
//   O^T[d][row]  += V^T . P^T (A = V^T via ds_read_b64_tr_b16 from a wave-private LDS tile)
// The 4 waves merge in LDS; the workgroup writes O directly (nsplit == 1) or one partial
// (m, l, acc[D]) per row into the caller's scratch for the merge kernels (launch_merge).
// VT: V arrives as V^T ([Hkv][D][Sk]); the V^T operand (row d, 8 consecutive keys per lane) is
// then loaded from global memory straight into its register layout, like K, with no LDS tile.
// NTL: K and V are loaded non-temporally (decode_nt_loads decides).
// ------------------------------------------------------------------------------------------
// AL: 1 tensors with the 16-byte vector layout; 0 without, read in pieces (load_piece, trim_piece);
// 2 rows shorter than a piece (D < 8, or V^T of fewer than 8 keys), read element by element. What
// bounds AL = 0 at small head dims is latency, so no piece is shifted before all of a tile's are in
// flight (shifted at the load -> so): 256 kv heads x 300 keys at D = 14 13.6 -> 8.7 us from V^T, 8 kv
// heads x 777 keys at D = 100 10.4 -> 8.8.
// NRB: the row blocks one workgroup serves (rb counts groups of NRB); each K/V fragment is then read
// once for all of them. Each row's arithmetic is that of NRB = 1. Two blocks for three or four of a
// kv head (launch_decode_d): 64 rows over 4001 keys, 32 kv heads 28.6 -> 23.2 us, 128 kv heads over
// 1000 keys 23.9 -> 21.9. Measured and not taken: four blocks at once (one wave per SIMD cannot cover
// the load and MFMA latencies: 36.9 us), two blocks where there are two (24-32 heads' rows over 2000
// keys at D = 64 8.1 -> 9.0 us: half the workgroups), the next step's loads issued a step ahead
// (+5 to +12%, the registers take a wave per SIMD).
// Two waves per SIMD are asked for (one for AL = 2 from V^T at DP = 256, which hardly any call reaches):
// the 137-165 registers at DP = 128 then allow three, where no bound took 172-185 (512 kv heads x 4096
// keys 162.6 -> 159.6 us, 200 x 300 14.9 -> 12.3; 8 kv heads at D = 256 17.9 -> 13.1). No instance
// spills; at DP = 256 that takes kLate.
template <int DP, bool CAUSAL, int AL, bool VT, bool NTL, int NRB>
__global__ __launch_bounds__(256, DP == 256 && VT && AL == 2 ? 1 : 2) void attn_decode_kernel(
    const uint16_t *__restrict__ Q, const uint16_t *__restrict__ K,
    const uint16_t *__restrict__ V, float *__restrict__ O, float *__restrict__ pm,
    float *__restrict__ pl, float *__restrict__ pacc, int Hq, int Hkv, int Sq, int Sk, int D,
    float c, int nsplit, int kps, int nrb) {
    constexpr int VSTR = DP + 16;
    // Rows 8..15 and 24..31 of a V tile (odd row-octets) are stored rotated by VROT elements:
    // one 32-lane pass of a transposed read covers rows 8g .. 8g+3 and 8g+8 .. 8g+11, which any
    // row stride that keeps 16-byte chunks aligned puts on the same banks (2 conflict cycles per
    // read at DP = 128); rotated by half a 256-byte row they take the other 32 banks. At DP = 64
    // no rotation within the 128-byte row separates them, and the 2-way conflict stays.
    constexpr int VROT = (DP == 128) ? 64 : 0;
    constexpr int VNCH = 32 * DP / 8 / 64; // 16-byte chunks per lane per V tile
    constexpr int VTILE = 32 * VSTR;       // elements of one wave's V tile
    __shared__ __attribute__((aligned(16))) uint16_t Vw[4 * VTILE];
    __shared__ float red_m[NRB][4][16], red_l[NRB][4][16];
    // The 4-wave merge reuses the V tiles' memory as float [4][16][DP + 4] (kMergePad).
    static_assert(4 * 16 * (DP + kMergePad) * 4 <= 4 * VTILE * 2,
                  "merge area must fit in the V tiles");

    // Block = (kv head u, split sp, row block group rb): rows 16 NRB rb on of the kv head's M rows.
    // Groups of one (u, sp) are consecutive logical ids, kept on one XCD so that they share
    // its L2 copy of the K/V range.
    const int g = Hq / Hkv, M = g * Sq;
    // The grid is Hkv * nsplit * nrb workgroups.
    const int L = (nrb > 1) ? xcd_remap(wg_id_x(), Hkv * nsplit * nrb) : wg_id_x();
    const int rb = L % nrb, us = L / nrb;
    const int u = us / nsplit, sp = us % nsplit;
    const int tid = wi_id_x(), w = tid >> 6, lane = tid & 63;
    const int r16 = lane & 15, grp = lane >> 4;
    const int k0 = sp * kps, k1 = min(k0 + kps, Sk);
    const int row0 = 16 * NRB * rb;
    constexpr bool VEC = AL == 1;

    const uint16_t *Kh = K + (size_t)u * Sk * D;
    const uint16_t *Vh = V + (size_t)u * Sk * D;

    auto piece = [](const uint16_t *p, int i, int n, int ie) __attribute__((always_inline)) {
        return AL == 2 ? load_short(p, i, n) : load_piece<NTL>(p, i, n, ie);
    };
    auto trim = [](u32x4 v, int i, int n, int ie) __attribute__((always_inline)) {
        return AL == 0 ? trim_piece(v, i, n, ie) : v;
    };
    bf16x8 qb[NRB][DP / 32];
    int lim[NRB];
    float m_run[NRB], l_run[NRB];
    f32x4 o[NRB][DP / 16];
#pragma unroll
    for (int b = 0; b < NRB; ++b) {
        const int row = row0 + 16 * b + r16;
        const bool rvalid = row < M;
        const int gi = rvalid ? row / Sq : 0, qi = rvalid ? row % Sq : 0;
        const size_t qrow = (size_t)(u * g + gi) * Sq + qi;
        u32x4 qr[DP / 32];
#pragma unroll
        for (int kk = 0; kk < DP / 32; ++kk)
            qr[kk] = VEC ? load_row8(Q, qrow, kk * 32 + grp * 8, D, rvalid)
                         : piece(Q + qrow * D, kk * 32 + grp * 8, D, kk * 32 + 32);
#pragma unroll
        for (int kk = 0; kk < DP / 32; ++kk)
            qb[b][kk] = as_bf16x8(VEC || rvalid ? trim(qr[kk], kk * 32 + grp * 8, D, kk * 32 + 32)
                                                : zero4());
        lim[b] = CAUSAL ? min(Sk - 1, Sk - Sq + qi) : Sk - 1;
        m_run[b] = kNegInf;
        l_run[b] = 0.f;
#pragma unroll
        for (int db = 0; db < DP / 16; ++db)
            o[b][db] = f32x4{0.f, 0.f, 0.f, 0.f};
    }

    uint16_t *vt = &Vw[w * VTILE];
    // Each workgroup starts its walk over the 128-key steps at a different step: workgroups
    // then read different column ranges at the same time, which spreads a V^T input's
    // 2*Sk-byte-strided rows over more HBM channels. attn_decode_vt_kernel walks the same order.
    const int nsteps = (k1 - k0 + 127) / 128;
    const int rot = us % (nsteps > 0 ? nsteps : 1);
    auto tile_of = [&](int js) {
        const int step = (js + rot < nsteps) ? js + rot : js + rot - nsteps;
        return k0 + step * 128 + w * 32;
    };
    struct frags {
        u32x4 k[2][DP / 32];
        u32x4 v[VT ? DP / 16 : VNCH];
    };
    // At DP = 256 K, V, Q and O of a tile do not fit the 256 registers of two waves per SIMD unless both
    // tensors are aligned and V is row-major: there V is loaded once Q.K^T has freed K's registers.
    // Spilling instead (12 registers aligned, 90-112 unaligned) -> so, 64 kv heads: 16000 keys at
    // D = 256 from V^T 250 -> 227 us, 4000 keys at D = 131 from V^T 67 -> 39 (one wave per SIMD, no
    // spills, V loaded with K: 54).
    constexpr bool kLate = DP == 256 && (VT || !VEC);
    // Unaligned pieces (AL != 1) of keys past k1 are those of key k1 - 1: their scores are masked,
    // their V rows zeroed (trim_v).
    auto load_k = [&](int tb, frags &f) __attribute__((always_inline)) {
#pragma unroll
        for (int t = 0; t < 2; ++t) {
            const int key = tb + 8 * (r16 >> 2) + 4 * t + (r16 & 3);
#pragma unroll
            for (int kk = 0; kk < DP / 32; ++kk)
                f.k[t][kk] = VEC ? load_row8<NTL>(Kh, (size_t)key, kk * 32 + grp * 8, D, key < k1)
                                 : piece(Kh + (size_t)min(key, k1 - 1) * D, kk * 32 + grp * 8, D,
                                         kk * 32 + 32);
        }
    };
    auto load_v = [&](int tb, frags &f) __attribute__((always_inline)) {
        if constexpr (VT) {
            // lane: d row 16db + r16, keys tb + 8grp .. +7 (the k index of pk below).
            const int key = tb + 8 * grp;
#pragma unroll
            for (int db = 0; db < DP / 16; ++db) {
                const int d = db * 16 + (VEC ? r16 : (int)opaque(r16));
                if (VEC) {
                    f.v[db] = load_vt8<NTL>(Vh, d, key, Sk, D, k1);
                } else {
                    f.v[db] = zero4();
                    if (d < D) // rows past D are never stored
                        f.v[db] = piece(Vh + (size_t)d * Sk, key, k1, tb + 32);
                }
            }
        } else {
#pragma unroll
            for (int r = 0; r < VNCH; ++r) {
                const int cidx = lane + 64 * r;
                const int row = tb + cidx / (DP / 8), col = (cidx % (DP / 8)) * 8;
                f.v[r] = VEC ? load_row8<NTL>(Vh, (size_t)row, col, D, row < k1)
                             : piece(Vh + (size_t)min(row, k1 - 1) * D, col, D, DP);
            }
        }
    };
    auto trim_k = [&](frags &f) __attribute__((always_inline)) {
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
            for (int kk = 0; kk < DP / 32; ++kk)
                f.k[t][kk] = trim(f.k[t][kk], kk * 32 + grp * 8, D, kk * 32 + 32);
    };
    auto trim_v = [&](int tb, frags &f) __attribute__((always_inline)) {
        if constexpr (VT) {
#pragma unroll
            for (int db = 0; db < DP / 16; ++db)
                f.v[db] = trim(f.v[db], tb + 8 * grp, k1, tb + 32);
        } else {
#pragma unroll
            for (int r = 0; r < VNCH; ++r) {
                const int cidx = lane + 64 * r;
                const int row = tb + cidx / (DP / 8), col = (cidx % (DP / 8)) * 8;
                f.v[r] = trim(f.v[r], col, D, DP);
                if (!VEC && tb + 32 > k1)
                    f.v[r] = row < k1 ? f.v[r] : zero4();
            }
        }
    };
    auto put_v = [&](const frags &f) __attribute__((always_inline)) {
        if (!VT) {
            lds_wave_fence(); // previous tile's transposed reads are complete
#pragma unroll
            for (int r = 0; r < VNCH; ++r) {
                const int cidx = lane + 64 * r;
                const int row = cidx / (DP / 8), col = (cidx % (DP / 8)) * 8;
                const int colr = (col + VROT * ((row >> 3) & 1)) & (DP - 1);
                *reinterpret_cast<u32x4 *>(&vt[row * VSTR + colr]) = f.v[r];
            }
        }
    };
    auto compute = [&](int tb, frags &f) __attribute__((always_inline)) {
        bf16x8 pk[NRB];
#pragma unroll
        for (int b = 0; b < NRB; ++b) {
            f32x4 s[2];
#pragma unroll
            for (int t = 0; t < 2; ++t) {
                s[t] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int kk = 0; kk < DP / 32; ++kk)
                    s[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf16x8(f.k[t][kk]),
                                                                   qb[b][kk], s[t], 0, 0, 0);
            }
            if (kLate) { // NRB == 1
                __builtin_amdgcn_sched_barrier(0);
                load_v(tb, f);
            }
            // Register (t, i) of this lane holds key tb + 8grp + 4t + i for row r16.
            float mx = kNegInf;
#pragma unroll
            for (int t = 0; t < 2; ++t)
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const int key = tb + 8 * grp + 4 * t + i;
                    if (key >= k1 || key > lim[b])
                        s[t][i] = kNegInf;
                    mx = fmaxf(mx, s[t][i]);
                }
            mx = max_xor32(max_xor16(mx));
            const float mnew = fmaxf(m_run[b], mx);
            const float muse = (mnew == kNegInf) ? 0.f : mnew;
            const float alpha = fast_exp2((m_run[b] - muse) * c);
            const float mc = muse * c;
            float psum = 0.f;
#pragma unroll
            for (int t = 0; t < 2; ++t)
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const float p = fast_exp2(fmaf(s[t][i], c, -mc));
                    psum += p;
                    pk[b][4 * t + i] = (__bf16)p;
                }
            l_run[b] = alpha * l_run[b] + psum;
            m_run[b] = mnew;
#pragma unroll
            for (int db = 0; db < DP / 16; ++db)
                o[b][db] *= alpha;
        }
        if (kLate) {
            trim_v(tb, f);
            put_v(f);
        }
        if (!VT)
            lds_wave_fence(); // this tile's V is in LDS before the transposed reads
        // rows of this lane's reads: 8grp + r16/4 and 4 on, in row-octet grp
        const int vrot = VROT * (grp & 1);
        const uint16_t *vb0 = &vt[(8 * grp + (r16 >> 2)) * VSTR + 4 * (r16 & 3)];
#pragma unroll
        for (int db = 0; db < DP / 16; ++db) {
            bf16x8 a;
            if (VT) {
                a = as_bf16x8(f.v[db < (int)(sizeof f.v / sizeof f.v[0]) ? db : 0]);
            } else {
                // column 16db + 4(r16 % 4) + vrot, modulo DP (db * 16 < DP - VROT: no wrap)
                const uint16_t *vb = vb0 + db * 16 + ((db * 16 < DP - VROT) ? vrot : -vrot);
                a = join_tr(lds_read_tr(vb), lds_read_tr(vb + 4 * VSTR));
            }
#pragma unroll
            for (int b = 0; b < NRB; ++b)
                o[b][db] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, pk[b], o[b][db], 0, 0, 0);
        }
    };
    for (int js = 0; js < nsteps; ++js) {
        const int tb = tile_of(js);
        if (tb >= k1)
            continue;
        frags f;
        load_k(tb, f);
        if (!kLate)
            load_v(tb, f);
        trim_k(f);
        if (!kLate) {
            trim_v(tb, f);
            put_v(f);
        }
        compute(tb, f);
    }
#pragma unroll
    for (int b = 0; b < NRB; ++b)
        l_run[b] = sum_xor32(sum_xor16(l_run[b]));

    // Merge the 4 waves: O^T register (db, i) of this lane holds d = 16db + 4grp + i, row r16.
    float *om = reinterpret_cast<float *>(Vw); // [4][16][DP + kMergePad]
    if (grp == 0)
#pragma unroll
        for (int b = 0; b < NRB; ++b) {
            red_m[b][w][r16] = m_run[b];
            red_l[b][w][r16] = l_run[b];
        }
#pragma unroll
    for (int b = 0; b < NRB; ++b) {
        __syncthreads();
#pragma unroll
        for (int db = 0; db < DP / 16; ++db)
#pragma unroll
            for (int i = 0; i < 4; ++i)
                om[(w * 16 + r16) * (DP + kMergePad) + db * 16 + 4 * grp + i] = o[b][db][i];
        __syncthreads();
        const int rowb = row0 + 16 * b, Mb = min(16, M - rowb);
        decode_merge<DP>(om, red_m[b], red_l[b], O, pm, pl, pacc, tid, rowb, Mb, u, g, Sq, D, c,
                         nsplit, sp);
    }
}

// Decode from V^T ([Hkv][D][Sk], DP of 64 or 128): attn_decode_kernel's workgroups, rows, key order, S MFMAs and softmax, with the V^T
// operand staged through LDS by LDS-DMA. HBM serves pieces of strided rows faster the longer
// the piece: 128 rows 8 KB apart read in 256-byte pieces stream at about 4.7 TB/s, in 1 KB
// pieces at about 5.9 TB/s (contiguous: 6.2). The kernel therefore walks the keys in groups of
// 512 (four of attn_decode_kernel's 128-key steps, in its order) and stages each group's V^T
// as four tiles of DP/4 d rows x 512 keys, every d row of a tile one 1 KB DMA. Tile i of group
// G-1 is multiplied in the same barrier interval as step i of group G is scored, so each
// interval has one step of K fragments and one V^T tile in flight; the softmax weights and
// rescale factors of a group's four steps wait in registers for their tiles. Each 16-row block
// of the output is rescaled and accumulated step by step as in attn_decode_kernel, so the two
// kernels' outputs are bit-identical. The 16-byte chunks of a tile row e sit at slot
// c ^ (e % 16), so the 16 lanes of an operand read (16 d rows, one key chunk) hit 16 distinct
// bank groups. NTL: K loads and V^T DMA are non-temporal (decode_nt_loads decides).
// UA: 0 tensors with the 16-byte vector layout; 1 and 2 without, their V^T pieces loaded into
// registers and put into LDS at the interval's end: 1 for D % 8 == 0, whose K and Q rows end with a
// piece, 2 for other D, whose last pieces are shifted once they are waited for. One instance for both
// cost D % 8 == 0 2-4%: 16 sequences of 8 kv heads over 4001 keys at D = 128 52.7 us, now 51.3; D = 100
// 50.3 with the shift at the load, now 45.6.
template <int DP, bool CAUSAL, bool NTL, int UA>
__global__ __launch_bounds__(256, 2) void attn_decode_vt_kernel(
    const uint16_t *__restrict__ Q, const uint16_t *__restrict__ K,
    const uint16_t *__restrict__ V, float *__restrict__ O, float *__restrict__ pm,
    float *__restrict__ pl, float *__restrict__ pacc, int Hq, int Hkv, int Sq, int Sk, int D,
    float c, int nsplit, int kps, int nrb) {
    static_assert(DP == 64 || DP == 128, "tile shape");
    constexpr int GK = 512;          // keys per group: 4 steps of 128 (4 waves x 32 keys)
    constexpr int RQ = DP / 4;       // d rows per V^T tile
    constexpr int RPW = RQ / 4;      // tile rows (one 1 KB DMA each) per wave
    constexpr int DBT = RQ / 16;     // 16-row operand blocks per tile
    constexpr int TILE = RQ * GK;    // elements of one tile
    __shared__ __attribute__((aligned(1024))) uint16_t Vt[2][TILE];
    __shared__ float red_m[4][16], red_l[4][16];
    static_assert(4 * 16 * (DP + kMergePad) * 4 <= 2 * TILE * 2,
                  "merge area must fit in the V^T tiles");

    const int g = Hq / Hkv, M = g * Sq;
    // The grid is Hkv * nsplit * nrb workgroups.
    const int L = (nrb > 1) ? xcd_remap(wg_id_x(), Hkv * nsplit * nrb) : wg_id_x();
    const int rb = L % nrb, us = L / nrb;
    const int u = us / nsplit, sp = us % nsplit;
    const int tid = threadIdx.x, lane = tid & 63; // a library call on purpose: see wi_id_x
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int r16 = lane & 15, grp = lane >> 4;
    const int k0 = sp * kps, k1 = min(k0 + kps, Sk);
    const int row0 = 16 * rb, Mb = min(16, M - row0);

    const bool rvalid = row0 + r16 < M;
    const int gi = rvalid ? (row0 + r16) / Sq : 0, qi = rvalid ? (row0 + r16) % Sq : 0;
    const int h = u * g + gi;
    const uint16_t *Kh = K + (size_t)u * Sk * D;

    bf16x8 qb[DP / 32];
    const size_t qrow = (size_t)h * Sq + qi;
    // Columns [col, col+8) of row `row` of H, zeros if !ok or past D. UA = 2: columns that reach
    // past D are trimmed where they are used (trim_piece).
    auto row8 = [&](const uint16_t *H, size_t row, int col, bool ok, auto NT)
        __attribute__((always_inline)) {
        constexpr bool kN = decltype(NT)::value;
        if constexpr (UA == 0)
            return load_row8<kN>(H, row, col, D, ok);
        if (!ok || col >= D)
            return zero4();
        return load16_any<kN>(H + row * D + (UA == 2 ? min(col, D - 8) : col));
    };
    u32x4 qr[DP / 32];
#pragma unroll
    for (int kk = 0; kk < DP / 32; ++kk)
        qr[kk] = row8(Q, qrow, kk * 32 + grp * 8, rvalid, std::false_type{});
#pragma unroll
    for (int kk = 0; kk < DP / 32; ++kk)
        qb[kk] = as_bf16x8(UA == 2 ? trim_piece(qr[kk], kk * 32 + grp * 8, D, kk * 32 + 32) : qr[kk]);
    const int lim = CAUSAL ? min(Sk - 1, Sk - Sq + qi) : Sk - 1;

    float m_run = kNegInf, l_run = 0.f;
    f32x4 o[DP / 16];
#pragma unroll
    for (int db = 0; db < DP / 16; ++db)
        o[db] = f32x4{0.f, 0.f, 0.f, 0.f};

    // This lane's DMA sources: wave w brings tile rows w*RPW .. w*RPW+RPW-1; lane slot p of
    // tile row e receives source chunk p ^ (e % 16) (tiles start at multiples of 16 d rows, so
    // e % 16 is also the d row's). A chunk of a d row past D or of keys at or past k1 gets an
    // offset beyond the buffer's range and lands as zeros.
    const uint16_t *Vh = V + (size_t)u * D * Sk;
    const __amdgpu_buffer_rsrc_t rvt = make_rsrc(Vh, (uint32_t)D * Sk * 2);
    const uint32_t row_bytes = (uint32_t)Sk * 2u;
    uint32_t vsrc[RPW];
    int vkey[RPW];
#pragma unroll
    for (int k = 0; k < RPW; ++k) {
        const int e = w * RPW + k;
        const int cw = (lane ^ e) & 15; // chunk within its step; the step is lane / 16
        vsrc[k] = (uint32_t)e * row_bytes + (uint32_t)cw * 16u;
        vkey[k] = cw * 8;
    }
    // Steps in attn_decode_kernel's order (it starts at step us % nsteps), taken four at a
    // time: group j holds walk positions 4j .. 4j+3, consecutive keys except where the walk
    // wraps to the split's first step.
    const int nsteps = (k1 - k0 + 127) / 128;
    const int ngr = (nsteps + 3) / 4;
    const int rot = us % (nsteps > 0 ? nsteps : 1);
    auto step_of = [&](int js) { return (js + rot < nsteps) ? js + rot : js + rot - nsteps; };
    // UA: the tile's pieces go through registers (vr), loaded where the DMA would be issued and
    // written at the interval's end (put_tile).
    u32x4 vr[UA ? RPW : 1];
    auto dma_tile = [&](int j, int q, int buf) {
        const int pos = 4 * j + (lane >> 4); // this lane's walk position
        const int key0 = pos < nsteps ? k0 + step_of(pos) * 128 : k1;
        const int klim = k1 - key0; // keys of this lane's step inside the split
        if constexpr (UA) {
            // Every load stays inside its row's first k1 keys (k1 >= 8): a piece that reaches past
            // k1 reads the last eight and is shifted in put_tile. Rows past D are never stored.
#pragma unroll
            for (int k = 0; k < RPW; ++k)
                vr[k] = load16_any<NTL>(Vh + (size_t)min(q * RQ + w * RPW + k, D - 1) * Sk +
                                        min(key0 + vkey[k], k1 - 8));
            return;
        }
        const uint32_t base = (uint32_t)(q * RQ) * row_bytes + (uint32_t)key0 * 2u;
#pragma unroll
        for (int k = 0; k < RPW; ++k) {
            const bool ok = q * RQ + w * RPW + k < D && vkey[k] < klim;
            dma16<0, NTL ? kDmaNT : 0>(rvt, &Vt[buf][(w * RPW + k) * GK], ok ? vsrc[k] + base : 0x80000000u);
        }
    };
    auto put_tile = [&](int j, int buf) {
        const int pos = 4 * j + (lane >> 4);
        const int key0 = pos < nsteps ? k0 + step_of(pos) * 128 : k1;
        const bool may = __builtin_amdgcn_ballot_w64(key0 + 128 > k1) != 0;
#pragma unroll
        for (int k = 0; k < (UA ? RPW : 0); ++k) {
            if (may)
                vr[k] = drop_elems(vr[k], min(8, max(0, key0 + vkey[k] + 8 - k1)));
            *reinterpret_cast<u32x4 *>(&Vt[buf][(w * RPW + k) * GK + lane * 8]) = vr[k];
        }
    };
    u32x4 ka[2][DP / 32], kn[2][DP / 32];
    auto load_k = [&](int tb, u32x4 (&dst)[2][DP / 32]) {
#pragma unroll
        for (int t = 0; t < 2; ++t) {
            const int key = tb + 8 * (r16 >> 2) + 4 * t + (r16 & 3);
#pragma unroll
            for (int kk = 0; kk < DP / 32; ++kk)
                dst[t][kk] = row8(Kh, (size_t)key, kk * 32 + grp * 8, key < k1,
                                  std::integral_constant<bool, NTL>{});
        }
    };
    // kn, once it is waited for, into ka.
    auto take_k = [&]() {
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
            for (int kk = 0; kk < DP / 32; ++kk)
                ka[t][kk] = UA == 2 ? trim_piece(kn[t][kk], kk * 32 + grp * 8, D, kk * 32 + 32)
                                    : kn[t][kk];
    };

    bf16x8 pkp[4], pkc[4]; // softmax weights of the previous / current group's steps
    float alp[4], alc[4];  // their rescale factors
    int livep = 0, livec = 0; // bit st: step st of the previous / current group was scored
    int buf = 0;
    if (ngr > 0) {
        const int tb = k0 + step_of(0) * 128 + w * 32;
        if constexpr (UA == 2) {
            load_k(tb, kn);
            take_k();
        } else {
            load_k(tb, ka);
        }
    }
    for (int j = 0; j <= ngr; ++j) {
        const bool cur = j < ngr;
        const int nsub = cur ? min(4, nsteps - 4 * j) : 0;
        static_for<4>([&](auto I) {
            constexpr int i = decltype(I)::value;
            // What the previous interval issued (this interval's K step and V^T tile) has
            // landed in every wave; every wave is done with the other buffer.
            __builtin_amdgcn_s_waitcnt(0x0F70);
            __syncthreads();
            if (i < 3) {
                if (j > 0)
                    dma_tile(j - 1, i + 1, buf ^ 1);
            } else if (cur) {
                dma_tile(j, 0, buf ^ 1);
            }
            int tbn = -1;
            if (i + 1 < nsub)
                tbn = k0 + step_of(4 * j + i + 1) * 128 + w * 32;
            else if (i + 1 == nsub && j + 1 < ngr)
                tbn = k0 + step_of(4 * j + 4) * 128 + w * 32;
            if (tbn >= 0)
                load_k(tbn, kn);
            const int tb = i < nsub ? k0 + step_of(4 * j + i) * 128 + w * 32 : k1;
            if (tb < k1) {
                f32x4 s[2];
#pragma unroll
                for (int t = 0; t < 2; ++t) {
                    s[t] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                    for (int kk = 0; kk < DP / 32; ++kk)
                        s[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf16x8(ka[t][kk]),
                                                                       qb[kk], s[t], 0, 0, 0);
                }
                // Register (t, x) of this lane holds key tb + 8grp + 4t + x for row r16.
                float mx = kNegInf;
#pragma unroll
                for (int t = 0; t < 2; ++t)
#pragma unroll
                    for (int x = 0; x < 4; ++x) {
                        const int key = tb + 8 * grp + 4 * t + x;
                        if (key >= k1 || key > lim)
                            s[t][x] = kNegInf;
                        mx = fmaxf(mx, s[t][x]);
                    }
                mx = max_xor32(max_xor16(mx));
                const float mnew = fmaxf(m_run, mx);
                const float muse = (mnew == kNegInf) ? 0.f : mnew;
                alc[i] = fast_exp2((m_run - muse) * c);
                const float mc = muse * c;
                float psum = 0.f;
#pragma unroll
                for (int t = 0; t < 2; ++t)
#pragma unroll
                    for (int x = 0; x < 4; ++x) {
                        const float p = fast_exp2(fmaf(s[t][x], c, -mc));
                        psum += p;
                        pkc[i][4 * t + x] = (__bf16)p;
                    }
                l_run = alc[i] * l_run + psum;
                m_run = mnew;
                livec |= 1 << i;
            }
            // Tile i of the previous group: d rows i*RQ .. i*RQ+RQ-1 over its four steps.
            if (j > 0) {
#pragma unroll
                for (int st = 0; st < 4; ++st) {
                    if (!(livep & (1 << st)))
                        continue;
                    const int cs = st * 16 + w * 4 + grp; // this wave's 32 keys of step st
#pragma unroll
                    for (int dl = 0; dl < DBT; ++dl) {
                        const int db = i * DBT + dl, e = dl * 16 + r16;
                        o[db] *= alp[st];
                        const bf16x8 a = as_bf16x8(*reinterpret_cast<const u32x4 *>(
                            &Vt[buf][e * GK + ((cs ^ (e & 15)) * 8)]));
                        o[db] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, pkp[st], o[db], 0, 0, 0);
                    }
                }
            }
            // The next step's K fragments (waiting for them here leaves the loads in flight
            // under both halves of the interval).
            if (tbn >= 0)
                take_k();
            if (UA && (i < 3 ? j > 0 : cur))
                put_tile(i < 3 ? j - 1 : j, buf ^ 1);
            buf ^= 1;
        });
#pragma unroll
        for (int st = 0; st < 4; ++st) {
            pkp[st] = pkc[st];
            alp[st] = alc[st];
        }
        livep = livec;
        livec = 0;
    }
    l_run = sum_xor32(sum_xor16(l_run));

    // Merge the 4 waves (as attn_decode_kernel): O^T register (db, i) holds d = 16db + 4grp + i.
    __syncthreads();
    float *om = reinterpret_cast<float *>(&Vt[0][0]); // [4][16][DP + kMergePad]
    if (grp == 0) {
        red_m[w][r16] = m_run;
        red_l[w][r16] = l_run;
    }
#pragma unroll
    for (int db = 0; db < DP / 16; ++db)
#pragma unroll
        for (int i = 0; i < 4; ++i)
            om[(w * 16 + r16) * (DP + kMergePad) + db * 16 + 4 * grp + i] = o[db][i];
    __syncthreads();
    decode_merge<DP>(om, red_m, red_l, O, pm, pl, pacc, tid, row0, Mb, u, g, Sq, D, c, nsplit, sp);
}

// Merge of split-K partials. Partial row r owns slots r*nsplit .. r*nsplit+nsplit-1 and covers
// row q_off + r % rph of query head r / rph, so its O row is (r / rph) * Sq + q_off + r % rph
// (decode: rph = Sq, q_off = 0). Weights w_s = 2^((m_s - max m) c), O = sum w_s acc_s / sum w_s l_s.
__device__ __forceinline__ size_t merge_orow(long r, int rph, int q_off, int Sq) {
    return (size_t)(r / rph) * Sq + q_off + r % rph;
}

// Any nsplit up to kMergeMaxSplit: one workgroup of 256 threads per row. The split weights
// w_s = 2^((m_s - max m) c) / sum_s w_s l_s are computed once, by the whole workgroup, into LDS;
// then threads take (split group, column) pairs, so the loads of one thread's splits are
// independent and several groups share a column, and the groups' sums meet in LDS.
constexpr int kMergeMaxSplit = 512;
__global__ __launch_bounds__(256) void attn_merge_kernel(const float *__restrict__ pm,
                                                         const float *__restrict__ pl,
                                                         const float *__restrict__ pacc,
                                                         float *__restrict__ O, int D, int nsplit,
                                                         float c, int rph, int q_off, int Sq) {
    __shared__ float wsh[kMergeMaxSplit];
    __shared__ float red[256];
    __shared__ float wred[4];
    const long row = wg_id_x();
    const int tid = wi_id_x(), lane = tid & 63, wv = tid >> 6;
    const size_t orow = merge_orow(row, rph, q_off, Sq);
    const float *m = pm + row * nsplit;
    const float *l = pl + row * nsplit;
    auto block_reduce = [&](float v, bool is_max) -> float {
#pragma unroll
        for (int o = 32; o >= 1; o >>= 1) {
            const float x = __shfl_xor(v, o);
            v = is_max ? fmaxf(v, x) : v + x;
        }
        if (lane == 0)
            wred[wv] = v;
        __syncthreads();
        const float r = is_max ? fmaxf(fmaxf(wred[0], wred[1]), fmaxf(wred[2], wred[3]))
                               : (wred[0] + wred[1]) + (wred[2] + wred[3]);
        __syncthreads();
        return r;
    };
    float mx = kNegInf;
    for (int s = tid; s < nsplit; s += 256)
        mx = fmaxf(mx, m[s]);
    mx = block_reduce(mx, true);
    const float muse = (mx == kNegInf) ? 0.f : mx;
    float lpart = 0.f;
    for (int s = tid; s < nsplit; s += 256) {
        const float w = fast_exp2((m[s] - muse) * c);
        wsh[s] = w;
        lpart += w * l[s];
    }
    const float lsum = block_reduce(lpart, false); // its barriers also publish wsh
    const float inv = (lsum > 0.f) ? 1.0f / lsum : 0.f;
    // sg split groups per column (D <= 256, so sg * D <= 256 threads are busy).
    const int sg = 256 / D;
    const int g = tid / D, d = tid - g * D;
    const float *pr = pacc + (size_t)row * nsplit * D;
    float acc = 0.f;
    if (g < sg) {
        int s = g;
        for (; s + 3 * sg < nsplit; s += 4 * sg) {
            const float a0 = pr[(size_t)s * D + d], a1 = pr[(size_t)(s + sg) * D + d];
            const float a2 = pr[(size_t)(s + 2 * sg) * D + d], a3 = pr[(size_t)(s + 3 * sg) * D + d];
            acc += wsh[s] * a0 + wsh[s + sg] * a1 + wsh[s + 2 * sg] * a2 + wsh[s + 3 * sg] * a3;
        }
        for (; s < nsplit; s += sg)
            acc += wsh[s] * pr[(size_t)s * D + d];
    }
    red[tid] = acc;
    __syncthreads();
    if (g == 0) {
        float t = acc;
        for (int k = 1; k < sg; ++k)
            t += red[k * D + d];
        O[orow * D + d] = t * inv;
    }
}

// 3 <= nsplit <= kMergeWaveMaxSplit (the prefill key split and decode splits): lp lanes cover a
// row's columns in 4-float pieces (4 lp >= D; the last piece is the last four floats, so two
// lanes may write the same columns, with the same values) and ng groups of them its splits, so a row
// takes lp * ng threads and a workgroup 256 / (lp ng) rows; lp and ng are powers of two (lps, ngs).
// The launch is a chain of latencies, so everything is in flight at once: the (m, l) of each row's
// splits (a row per 16 lanes, or per wave past 16 splits), then NL splits' columns per thread
// without a branch, and only then the weights, which go through LDS, as the groups' sums do. One
// wave per row reading its splits one by one took 7.2 us for 32 rows x 64 splits at D = 128 (8
// workgroups); decode over 32768 keys 34.5 -> 29.9 us with this layout. A wave per row for the
// weights, and branches around the loads, cost short merges 1 to 2 us: 202 rows x 3 splits at
// D = 32 5.3 us, 10144 rows x 3 at D = 128 8.8.
constexpr int kMergeWaveMaxSplit = 64;
// max or sum over each 16 (all: 64) lanes of the wave, in every lane, on the VALU.
template <bool MAX> __device__ __forceinline__ float seg_all(float x, bool all) {
    auto op = [](float a, float b) { return MAX ? fmaxf(a, b) : a + b; };
    auto ror = [](float v, auto C) {
        const int u = __builtin_bit_cast(int, v);
        return __builtin_bit_cast(
            float, __builtin_amdgcn_update_dpp(u, u, decltype(C)::value, 0xf, 0xf, false));
    };
    x = op(x, ror(x, std::integral_constant<int, 0x128>{})); // row_ror:8, 4, 2, 1
    x = op(x, ror(x, std::integral_constant<int, 0x124>{}));
    x = op(x, ror(x, std::integral_constant<int, 0x122>{}));
    x = op(x, ror(x, std::integral_constant<int, 0x121>{}));
    if (all)
        x = MAX ? max_xor32(max_xor16(x)) : sum_xor32(sum_xor16(x));
    return x;
}
template <int NL>
__global__ __launch_bounds__(256) void attn_mergew_kernel(const float *__restrict__ pm,
                                                          const float *__restrict__ pl,
                                                          const float *__restrict__ pacc,
                                                          float *__restrict__ O, long rows, int D,
                                                          int nsplit, float c, int rph, int q_off,
                                                          int Sq, int lps, int ngs) {
    __shared__ float wsh[32][kMergeWaveMaxSplit]; // up to 32 rows (lp = 8: D <= 32)
    __shared__ __attribute__((aligned(16))) f32x4 red[256];
    const int tid = wi_id_x(), wv = tid >> 6, lane = tid & 63;
    const int ng = 1 << ngs, rpw = 256 >> (lps + ngs);
    const long row0 = (long)wg_id_x() * rpw;
    const int rl = tid >> (lps + ngs); // the thread's row of the workgroup
    const int g = (tid >> lps) & (ng - 1), d = 4 * (tid & ((1 << lps) - 1));
    const long row = row0 + rl;
    const bool mine = row < rows && d < D;

    const bool all = nsplit > 16;
    const int segs = all ? 6 : 4, sl = lane & ((1 << segs) - 1);
    const int step = 256 >> segs; // rows per pass of the workgroup
    auto slot_of = [&](int r) {
        return (size_t)min(row0 + r, rows - 1) * nsplit + min(sl, nsplit - 1);
    };
    int r = (wv << (6 - segs)) + (lane >> segs);
    float ms = pm[slot_of(r)], ls = pl[slot_of(r)];

    const float *pr = pacc + (size_t)min(row, rows - 1) * nsplit * D;
    f32x4 x[NL];
    auto load = [&](int s0) __attribute__((always_inline)) {
        const float *p[NL];
#pragma unroll
        for (int i = 0; i < NL; ++i)
            p[i] = pr + (size_t)min(s0 + g + i * ng, nsplit - 1) * D;
        if (D >= 4) {
#pragma unroll
            for (int i = 0; i < NL; ++i)
                x[i] = *reinterpret_cast<const f32x4_a4 *>(p[i] + min(d, D - 4));
        } else {
#pragma unroll
            for (int i = 0; i < NL; ++i)
                x[i] = f32x4{p[i][0], p[i][D > 1 ? 1 : 0], p[i][D - 1], 0.f};
        }
    };
    load(0);
    for (;; ms = pm[slot_of(r)], ls = pl[slot_of(r)]) {
        const bool in = sl < nsplit;
        const float mx = seg_all<true>(in ? ms : kNegInf, all);
        const float muse = (mx == kNegInf) ? 0.f : mx;
        const float w = in ? fast_exp2((ms - muse) * c) : 0.f;
        const float lw = seg_all<false>(in ? w * ls : 0.f, all);
        if (r < rpw)
            wsh[r][sl] = w * ((lw > 0.f) ? 1.0f / lw : 0.f);
        r += step;
        if (r - (lane >> segs) >= rpw)
            break;
    }
    __syncthreads();
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
    for (int s0 = 0;;) {
#pragma unroll
        for (int i = 0; i < NL; ++i) {
            const int s = s0 + g + i * ng;
            const bool in = s < nsplit;
            const float a = in ? wsh[rl][s] : 0.f;
#pragma unroll
            for (int j = 0; j < 4; ++j)
                acc[j] += a * (in ? x[i][j] : 0.f);
        }
        s0 += NL * ng;
        if (s0 >= nsplit)
            break;
        load(s0);
    }
    if (ng > 1) {
        red[tid] = acc;
        __syncthreads();
        if (g != 0)
            return;
        for (int k = 1; k < ng; ++k) {
            const f32x4 y = red[tid + (k << lps)];
#pragma unroll
            for (int j = 0; j < 4; ++j)
                acc[j] += y[j];
        }
    }
    if (!mine)
        return;
    float *o = O + merge_orow(row, rph, q_off, Sq) * D;
    if (D >= 4) {
        *reinterpret_cast<f32x4_a4 *>(o + min(d, D - 4)) = acc;
    } else {
#pragma unroll
        for (int j = 0; j < 3; ++j)
            if (j < D)
                o[j] = acc[j];
    }
}

// nsplit == 2 (the causal prefill split, the head split, two-part key splits): the two
// weights computed once per lane, columns as float4 when D % 4 == 0 and O and the partials are
// 16-byte aligned.
__global__ __launch_bounds__(256) void attn_merge2_kernel(const float *__restrict__ pm,
                                                          const float *__restrict__ pl,
                                                          const float *__restrict__ pacc,
                                                          float *__restrict__ O, long rows, int D,
                                                          float c, int rph, int q_off, int Sq,
                                                          int lpr) {
    // lpr lanes per row (a power of two, 4 <= lpr <= 64): 256 / lpr rows per workgroup, each
    // lane taking 16-byte pieces of its row (vec) or single columns. One row per wave in 8-byte
    // pieces left half the lanes idle at D = 64; this layout measured config 5 +2-4% (same box),
    // other split shapes within noise, with the same arithmetic per element.
    const int t = wi_id_x();
    const long row = (long)wg_id_x() * (256 / lpr) + t / lpr;
    const int lane = t & (lpr - 1);
    if (row >= rows)
        return;
    const size_t orow = merge_orow(row, rph, q_off, Sq);
    const float m0 = pm[2 * row], m1 = pm[2 * row + 1];
    const float mx = fmaxf(m0, m1);
    const float muse = (mx == kNegInf) ? 0.f : mx;
    const float w0 = fast_exp2((m0 - muse) * c), w1 = fast_exp2((m1 - muse) * c);
    const float lsum = w0 * pl[2 * row] + w1 * pl[2 * row + 1];
    const float inv = (lsum > 0.f) ? 1.0f / lsum : 0.f;
    const float a0 = w0 * inv, a1 = w1 * inv;
    const float *p0 = pacc + (size_t)row * 2 * D, *p1 = p0 + D;
    float *o = O + orow * D;
    if ((D & 3) == 0 && ((uintptr_t)O & 15u) == 0 && ((uintptr_t)pacc & 15u) == 0) {
        for (int d = 4 * lane; d < D; d += 4 * lpr) {
            const f32x4 x = *reinterpret_cast<const f32x4 *>(p0 + d);
            const f32x4 y = *reinterpret_cast<const f32x4 *>(p1 + d);
            f32x4 r;
#pragma unroll
            for (int j = 0; j < 4; ++j)
                r[j] = a0 * x[j] + a1 * y[j];
            *reinterpret_cast<f32x4 *>(o + d) = r;
        }
    } else {
        for (int d = lane; d < D; d += lpr)
            o[d] = a0 * p0[d] + a1 * p1[d];
    }
}

// V [Hkv][Sk][D] -> Vp [Hkv][D][Sk]: one workgroup per TK-key x 64-column tile. Key rows arrive as 16-byte loads into LDS;
// each thread then gathers 8 consecutive keys of one column and stores them as one 16-byte
// chunk, so each wave store writes 512 / TK columns x 2*TK contiguous bytes.
// The LDS tile has unpadded 128-byte rows, 16-byte chunk c of row r stored at chunk
// c ^ ((r >> 3) & 7). The gathers of a wave read one column chunk of TK/8 rows spaced 8 apart;
// the XOR sends each 8 consecutive such rows to 8 different chunks.
// VEC: D % 8 == 0, Sk % 8 == 0 and both tensors 16-byte aligned. Otherwise the same 16-byte pieces
// at element alignment, the ends of rows handled apart.
template <int TK, bool VEC>
__global__ __launch_bounds__(256) void attn_pack_v16_kernel(const uint16_t *__restrict__ V,
                                                            uint16_t *__restrict__ Vp, int Sk,
                                                            int D) {
    constexpr int TD = 64;
    constexpr int TPR = TK / 8; // threads per V^T row piece (8 keys each)
    static_assert(TK % 32 == 0 && TK <= 2048, "tile");
    __shared__ __attribute__((aligned(16))) uint16_t tile[TK * TD];
    const int kv = wg_id_z();
    const int k0 = wg_id_x() * TK, d0 = wg_id_y() * TD;
    const uint16_t *src = V + (size_t)kv * Sk * D;
    uint16_t *dst = Vp + (size_t)kv * D * Sk;
    const int tid = wi_id_x();
#pragma unroll
    for (int r = 0; r < TK / 32; ++r) {
        const int cidx = tid + 256 * r;
        const int row = cidx >> 3, ch = cidx & 7;
        const int k = k0 + row, d = d0 + ch * 8;
        u32x4 v = zero4();
        if (k < Sk && d < D)
            v = VEC ? __builtin_nontemporal_load(
                          reinterpret_cast<const u32x4 *>(src + (size_t)k * D + d))
                    : D < 8 ? load_short(src + (size_t)k * D, d, D)
                            : trim_piece(load_piece<true>(src + (size_t)k * D, d, D, d0 + TD), d, D,
                                         d0 + TD);
        *reinterpret_cast<u32x4 *>(&tile[row * TD + ((ch ^ (row >> 3)) & 7) * 8]) = v;
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < TK / 32; ++r) {
        const int dl = r * (256 / TPR) + tid / TPR, kc = (tid % TPR) * 8;
        const int d = d0 + dl, k = k0 + kc;
        // Rows kc .. kc+7 share (row >> 3) == kc / 8, hence one swizzled chunk.
        const int col = (((dl >> 3) ^ (kc >> 3)) & 7) * 8 + (dl & 7);
        if (d < D && k < Sk) {
            uint32_t e[8];
#pragma unroll
            for (int j = 0; j < 8; ++j)
                e[j] = tile[(kc + j) * TD + col];
            const u32x4 out = {e[0] | (e[1] << 16), e[2] | (e[3] << 16), e[4] | (e[5] << 16),
                               e[6] | (e[7] << 16)};
            uint16_t *q = dst + (size_t)d * Sk + k;
            if (VEC) {
                *reinterpret_cast<u32x4 *>(q) = out;
            } else if (k + 8 <= Sk) {
                *reinterpret_cast<u32x4_a2 *>(q) = out;
            } else {
#pragma unroll
                for (int j = 0; j < 7; ++j)
                    if (k + j < Sk)
                        q[j] = (uint16_t)e[j];
            }
        }
    }
}

// Calls f(std::integral_constant<bool, b>{}): turns a runtime flag into a template argument.
template <typename F> hipError_t with_flag(bool b, F &&f) {
    return b ? f(std::true_type{}) : f(std::false_type{});
}

// Plan recording (attn_flash_plan): while t_plan is set on the calling thread, each launch
// site writes one line per kernel it would launch ("name<template arguments> grid=x[,y,z]
// block=n", then the site's notes) into the caller's buffer instead of launching.
struct plan_buf {
    char *buf;
    size_t len, pos;
    bool truncated;
};
thread_local plan_buf *t_plan = nullptr;
const char *tf(bool b) { return b ? "true" : "false"; }

__attribute__((format(printf, 3, 4))) void plan_note(dim3 g, dim3 b, const char *fmt, ...) {
    plan_buf *p = t_plan;
    char line[256];
    va_list ap;
    va_start(ap, fmt);
    int n = vsnprintf(line, sizeof line, fmt, ap);
    va_end(ap);
    if (n < 0)
        n = 0;
    size_t used = (size_t)n < sizeof line ? (size_t)n : sizeof line - 1;
    int m = (g.y > 1 || g.z > 1)
                ? snprintf(line + used, sizeof line - used, " grid=%u,%u,%u block=%u\n", g.x, g.y,
                           g.z, b.x * b.y * b.z)
                : snprintf(line + used, sizeof line - used, " grid=%u block=%u\n", g.x,
                           b.x * b.y * b.z);
    used += (m > 0 && (size_t)m < sizeof line - used) ? (size_t)m : 0;
    if (p->pos + used + 1 > p->len) {
        p->truncated = true;
        return;
    }
    memcpy(p->buf + p->pos, line, used);
    p->pos += used;
    p->buf[p->pos] = '\0';
}

// Compute units of the current device (cached per device).
static int device_cus() {
    static int cus[64];
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64)
        return 256;
    if (cus[dev] <= 0) {
        int n = 0;
        if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess ||
            n <= 0)
            n = 256;
        cus[dev] = n;
    }
    return cus[dev];
}

hipError_t launch_merge(const float *pm, const float *pl, const float *pacc, float *O, long rows,
                        int D, int nsplit, float c, int rph, int q_off, int Sq, hipStream_t st) {
    if (rows <= 0 || rows > 0x7fffffffL || rph <= 0)
        return hipErrorInvalidValue;
    if (nsplit == 2) {
        // Lanes per row: the power of two covering D / 4 pieces of 16 bytes, 4 to 64.
        int lpr = 4;
        while (lpr < 64 && 4 * lpr < D)
            lpr *= 2;
        const long rpw = 256 / lpr; // rows per workgroup
        if (t_plan)
            plan_note(dim3((unsigned)((rows + rpw - 1) / rpw)), dim3(256), "attn_merge2_kernel");
        else
            hipLaunchKernelGGL(attn_merge2_kernel, dim3((unsigned)((rows + rpw - 1) / rpw)),
                               dim3(256), 0, st, pm, pl, pacc, O, rows, D, c, rph, q_off, Sq, lpr);
    }
    else if (nsplit <= kMergeWaveMaxSplit && D <= 256) {
        int lps = 3;
        while ((4 << lps) < D)
            ++lps;
        // Split groups per row: at most 8 loads per thread where the workgroup allows, and more
        // groups (down to two loads per thread) while the grid has fewer threads than the GPU.
        int ngs = 0;
        while (ngs + lps < 8 && ((8 << ngs) < nsplit ||
                                 ((4 << ngs) <= nsplit && rows << (lps + ngs) < 256L * device_cus())))
            ++ngs;
        const long rpw = 256 >> (lps + ngs), nwg = (rows + rpw - 1) / rpw;
        if (t_plan)
            plan_note(dim3((unsigned)nwg), dim3(256), "attn_mergew_kernel nsplit=%d", nsplit);
        else if (nsplit <= 4 << ngs)
            hipLaunchKernelGGL(attn_mergew_kernel<4>, dim3((unsigned)nwg), dim3(256), 0, st, pm, pl,
                               pacc, O, rows, D, nsplit, c, rph, q_off, Sq, lps, ngs);
        else
            hipLaunchKernelGGL(attn_mergew_kernel<8>, dim3((unsigned)nwg), dim3(256), 0, st, pm, pl,
                               pacc, O, rows, D, nsplit, c, rph, q_off, Sq, lps, ngs);
    } else if (nsplit <= kMergeMaxSplit && D <= 256) {
        if (t_plan)
            plan_note(dim3((unsigned)rows), dim3(256), "attn_merge_kernel nsplit=%d", nsplit);
        else
            hipLaunchKernelGGL(attn_merge_kernel, dim3((unsigned)rows), dim3(256), 0, st, pm, pl,
                               pacc, O, D, nsplit, c, rph, q_off, Sq);
    }
    else
        return hipErrorInvalidValue;
    return hipGetLastError();
}

// Short query blocks under GQA (Sq <= 64, g > 1): the g heads' rows of a kv head share query
// tiles instead of each head leaving all but one or two waves of its tile idle. Measured with
// 64 batches x 32 heads (8 kv heads), Sk = 4096, causal, against one tile per head: Sq = 24 /
// 32 / 48 / 64: 2.35x / 2.1x / 1.67x / 1.25x faster. From Sq ~ 100 up, one tile per head is
// faster, since its larger grid keeps every CU busy.
static bool prefill_pack(int Hq, int Hkv, int Sq) { return Hq / Hkv > 1 && Sq <= 64; }

// CUs per XCD for xcd_remap_paired when `on` and the n workgroups fill more than one slot per
// CU but fit in two (all resident at once); else 0 (plain xcd_remap). ATTN_PREFILL_PAIR=0 turns
// the pairing off for tuning sweeps.
static int prefill_pair_r(bool on, long n) {
    static int env = -1;
    if (env < 0) {
        const char *e = getenv("ATTN_PREFILL_PAIR");
        env = (e && atoi(e) == 0) ? 0 : 1;
    }
    const int cus = device_cus();
    if (!on || !env || cus % 8 != 0 || n <= cus || n > 2L * cus)
        return 0;
    return cus / 8;
}

// Software-pipelined key tiles in the fast prefill kernel (tile_pipelined); ATTN_PREFILL_PIPE=0
// (read once) turns them off for tuning sweeps.
static int prefill_pipe() {
    static int env = -1;
    if (env < 0) {
        const char *e = getenv("ATTN_PREFILL_PIPE");
        env = (e && atoi(e) == 0) ? 0 : 1;
    }
    return env;
}

// Key split of a prefill grid that fills at most half of one round of resident workgroups
// (few query tiles, long key ranges: chunked prefill, small batches): each query tile's key
// tiles are cut into nsplit near-equal parts, run as separate workgroups that write partials
// (m, l, acc) to the scratch, and a merge kernel (launch_merge) combines them. nsplit fills one round,
// keeps at least kSplitMinTiles key tiles per part and fits the scratch's partial slots.
// Causal grids take it only when the keys before the query block (Sk - Sq) are at least as many
// as the queries, so that query tiles attend similar key counts; triangular causal grids keep
// the split of their heavier query tiles (below). 1 = no split. ATTN_PREFILL_SPLIT=0 (read
// once) turns it off for tuning sweeps.
constexpr int kSplitMinTiles = 4;
static int prefill_key_split(long nblk, int wg_per_cu, int nkt, long rows, long slots, bool ok,
                             bool shape_ok) {
    static int env = -1;
    if (env < 0) {
        const char *e = getenv("ATTN_PREFILL_SPLIT");
        env = (e && atoi(e) == 0) ? 0 : 1;
    }
    const long resident = (long)device_cus() * wg_per_cu;
    if (!env || !ok || !shape_ok || nblk <= 0 || 2 * nblk > resident || rows <= 0)
        return 1;
    long ns = resident / nblk;
    ns = std::min(ns, (long)nkt / kSplitMinTiles);
    ns = std::min(ns, slots / rows);
    ns = std::min(ns, (long)kMergeMaxSplit);
    return ns >= 2 ? (int)ns : 1;
}

// Slot-balanced head split of a non-causal grid of n = Hq * nqt 128-row (4-wave) tiles with
// one to two tiles per CU (two such workgroups are resident per CU). Dispatched as they are,
// n - CUs of the CUs run two tiles and the rest one, so the grid takes two tiles' time. Instead
// every tile of the last hs heads runs as two workgroups over the halves of its key range
// (partials merged through the scratch): the n - hs * nqt whole tiles take the CUs' first
// slots and the halves fill the rest, so no CU runs more than one and a half tiles. hs is the
// largest count whose items fit two per CU; it must leave at most one whole tile per CU, and
// each half at least 2 * kSplitMinTiles key tiles. Returns hs, or 0 when it does not apply.
// Taken at DP <= 64 only, whose 4-wave workgroups keep 128-key tiles. Measured (same box, two
// runs each): config 5 78.5 -> 72.9 us (+7.5%), 40 heads x 1000 over 4000 keys at D = 64
// +3-4%; with 12 key tiles (6 per half, D = 40) -10%; with the 64-key tiles of wider 4-wave
// workgroups it lost (D = 128 -12%, D = 96 -15%).
// ATTN_PREFILL_HSPLIT=0 (read once) turns it off for tuning sweeps.
static int prefill_head_split(int Hq, int Sq, int nqt, int nkt, long slots, bool ok) {
    static int env = -1;
    if (env < 0) {
        const char *e = getenv("ATTN_PREFILL_HSPLIT");
        env = (e && atoi(e) == 0) ? 0 : 1;
    }
    const long cus = device_cus(), n = (long)Hq * nqt;
    if (!env || !ok || cus % 8 != 0 || nqt <= 0 || n <= cus || n >= 2 * cus ||
        nkt < 4 * kSplitMinTiles)
        return 0;
    const long hs = std::min((long)Hq, (2 * cus - n) / nqt);
    if (hs < 1 || n - hs * nqt > cus || 2 * hs * Sq > slots)
        return 0;
    return (int)hs;
}

// Non-causal grids at DP = 64 that take the head split may run instead as 12-wave key-halves
// workgroups of 192 rows (attn_prefill_fast_kernel, NW = 12), a kv head's g * Sq query rows
// tiled as one row space, one workgroup per CU, where they fit one round: each CU then holds
// at most 192 rows, as with the head split's one and a half 128-row tiles, but with three waves
// per SIMD, no partials to write and no merge kernel.
// ATTN_PREFILL_W12=0 (read once) keeps the head split for tuning sweeps.
static bool prefill_rows192(int Hq, int Hkv, int Sq) {
    static int env = -1;
    if (env < 0) {
        const char *e = getenv("ATTN_PREFILL_W12");
        env = (e && atoi(e) == 0) ? 0 : 1;
    }
    const long nwg = (long)Hkv * (((long)(Hq / Hkv) * Sq + 191) / 192);
    return env && device_cus() % 8 == 0 && nwg <= device_cus() &&
           (long)(Hq / Hkv) * Sq < 0x7fffffffL;
}

// A causal grid of at most one workgroup per CU is as slow as its heaviest query tile. Then the
// key range of each tile in the upper half (qt >= nqt/2) is split in two workgroups whose
// partials (m, l, acc) go to the caller's scratch and are merged, when the slots suffice.
template <int DP, int KT, int NW, bool CAUSAL, bool VT, bool KH = false, int UA = 0>
hipError_t launch_prefill_fast_nw(const uint16_t *Q, const uint16_t *K, const uint16_t *V,
                                  float *O, int Hq, int Hkv, int Sq, int Sk, int D, float c,
                                  float *pm, float *pl, float *pacc, long slots, hipStream_t st) {
    constexpr int BQ = (KH ? NW / 2 : NW) * 32;
    const int g = Hq / Hkv;
    const int pack = (NW == 12 || prefill_pack(Hq, Hkv, Sq)) ? 1 : 0; // 12 waves: packed rows
    const int nqt = pack ? (g * Sq + BQ - 1) / BQ : (Sq + BQ - 1) / BQ;
    long nblk = (long)(pack ? Hkv : Hq) * nqt;
    const int nsplit = prefill_key_split(nblk, prefill_wg_per_cu(DP, KT, NW), (Sk + KT - 1) / KT,
                                         (long)Hq * Sq, slots, pm && !pack,
                                         !CAUSAL || (long)Sk - Sq >= Sq);
    int split_first = -1, prows = 0;
    if (nsplit > 1) {
        nblk *= nsplit;
    } else if (CAUSAL && !pack && pm && nqt >= 2 && nblk <= device_cus() &&
               (!KH || (nblk + (long)Hq * (nqt - nqt / 2) <= device_cus() &&
                        (Sk + KT - 1) / KT >= 3 * kSplitMinTiles))) {
        // Key halves (8 waves per item) take the split only when the split grid still fits one
        // round and each half keeps at least 6 key tiles: 8 heads at 2k 28.2 -> 26.2 us with it,
        // 8 heads at 1536 +4%, 8 heads of 1500 at D = 96 +3% (against the 4-wave split); Qwen3 2k
        // (384 items on 256 CUs) 42 us with it, 33.8 without; Qwen3 1k (4-tile halves) 21.2
        // with it, 19.5 without. 8 heads at 1200 (10 key tiles) stays 7% behind the 4-wave split.
        const int sf = nqt / 2;
        const long pr = (long)Sq - (long)sf * BQ;
        if (pr > 0 && 2L * Hq * pr <= slots) {
            split_first = sf;
            prows = (int)pr;
            nblk = (long)Hq * (nqt + (nqt - sf));
        }
    }
    // Non-causal grids of one to two tiles per CU: whole tiles plus halves (prefill_head_split).
    const int hsplit =
        (!CAUSAL && DP <= 64 && nsplit == 1 && prefill_wg_per_cu(DP, KT, NW) == 2)
            ? prefill_head_split(Hq, Sq, nqt, (Sk + KT - 1) / KT, slots, pm && !pack)
            : 0;
    if (hsplit > 0) {
        split_first = 0;
        prows = Sq;
        nblk = 2L * device_cus();
    }
    if (nblk <= 0 || nblk > 0x7fffffffL)
        return hipErrorInvalidValue;
    // Causal items resident all at once, two per CU: pair heavy with light query tiles on each
    // CU (xcd_remap_paired). Measured on a 16-head 4k causal grid: see prefill_pair_r. The head
    // split places its items by XCD position itself and takes the CUs per XCD here.
    const int pair_r = hsplit > 0 ? device_cus() / 8
                                  : prefill_pair_r(CAUSAL && !pack && split_first < 0 &&
                                                       nsplit == 1 &&
                                                       prefill_wg_per_cu(DP, KT, NW) == 2,
                                                   nblk);
    if (t_plan)
        plan_note(dim3((unsigned)nblk), dim3(NW * 64),
                  "attn_prefill_fast_kernel<%d, %d, %d, %s, %s, %s%s> nsplit=%d split_first=%d "
                  "hsplit=%d pack=%d pair=%d",
                  DP, KT, NW, tf(CAUSAL), tf(VT), tf(KH), UA ? ", unaligned" : "", nsplit,
                  split_first, hsplit, pack, pair_r);
    else
        hipLaunchKernelGGL((attn_prefill_fast_kernel<DP, KT, NW, CAUSAL, VT, KH, UA>),
                           dim3((unsigned)nblk), dim3(NW * 64), 0, st, Q, K, V, O, Hq, Hkv, Sq, Sk,
                           D, c, nqt, split_first, pm, pl, pacc, prows, pack, pair_r,
                           prefill_pipe(), nsplit, (int)nblk, hsplit);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess)
        return e;
    if (nsplit > 1)
        return launch_merge(pm, pl, pacc, O, (long)Hq * Sq, D, nsplit, c, Sq, 0, Sq, st);
    if (hsplit > 0)
        return launch_merge(pm, pl, pacc, O + (size_t)(Hq - hsplit) * Sq * D, (long)hsplit * Sq,
                            D, 2, c, Sq, 0, Sq, st);
    if (split_first < 0)
        return e;
    return launch_merge(pm, pl, pacc, O, (long)Hq * prows, D, 2, c, prows, split_first * BQ, Sq,
                        st);
}

// Waves per workgroup for the fast prefill kernel: 8 (256 query rows, one workgroup per CU,
// two waves per SIMD), or 4 (128 rows; two workgroups fit a CU).
//  * Packed tiles (prefill_pack): 4 waves when a kv head's rows fit one 128-row tile or fill
//    128-row tiles better than 256-row ones.
//  * Otherwise 4 waves when 256-row tiles are nearly full (>= 90% of their rows are queries)
//    but would leave CUs idle: at most half as many 8-wave workgroups as CUs, or for causal
//    grids (uneven tiles) at most one per CU; and for causal grids whose query tiles attend
//    at most 1024 keys on average. Measured against 8 waves: 16 heads at 2k +21%,
//    Qwen3 causal 1k / 2k / 4k +18% / +9% / +7.5%, config 5 causal +24%. When 256-row tiles
//    are part empty (Sq = 128, 200), 4 waves add no parallelism and their 64-key tiles lose
//    11-20%; above the small-grid sizes 8 waves win by 5-9%.
// ATTN_PREFILL_WAVES=4 or =8 (read once) forces one for tuning sweeps.
static int prefill_waves_forced() {
    static int forced = -1;
    if (forced < 0) {
        const char *e = getenv("ATTN_PREFILL_WAVES");
        forced = (e && (atoi(e) == 4 || atoi(e) == 8)) ? atoi(e) : 0;
    }
    return forced;
}

static int prefill_waves(int Hq, int Hkv, int Sq, int Sk, bool causal, bool head_split) {
    if (const int forced = prefill_waves_forced())
        return forced;
    const int g = Hq / Hkv;
    if (prefill_pack(Hq, Hkv, Sq)) {
        const long R = (long)g * Sq; // rows per kv head
        const long t4 = (R + 127) / 128, t8 = (R + 255) / 256;
        return (R <= 128 || 4 * t4 < 8 * t8) ? 4 : 8; // fewer idle wave slots at 4 waves
    }
    const long t8 = (Sq + 255) / 256;
    const long n8 = (long)Hq * t8;
    const bool full = (long)Sq * 10 >= t8 * 256 * 9;
    // Causal query tiles attend Sk - Sq/2 keys on average; up to 1024 their fixed cost per
    // workgroup (prologue, O stores, dispatch) is large enough that two resident 4-wave
    // workgroups per CU, which overlap it, win against 8-wave per-tile workgroups: c3-shaped
    // 1k / 2k causal +15% / +3%, 4k -1%. (Where the persistent kernel's pairs fit, that kernel
    // runs instead: launch_prefill_fast_t.)
    const bool short_causal = causal && (long)Sk - Sq / 2 <= 1024;
    // head_split: the 4-wave grid takes the slot-balanced head split (prefill_head_split).
    return (head_split ||
            (full && (n8 <= (causal ? device_cus() : device_cus() / 2) || short_causal)))
               ? 4
               : 8;
}

// Key halves (attn_prefill_fast_kernel's KH): where 4-wave workgroups would run at D >= 64, an
// 8-wave workgroup serves the same 128 rows with 128-key tiles, each SIMD's two waves taking
// the two halves of every tile. Taken where it measured faster (same box, two runs each):
// non-causal grids of at most one 128-row tile per CU (16 heads at 2k 54.3 -> 39.8 us; there
// the 4-wave grid took the key split), and causal grids of exactly two such tiles per CU,
// which heaviest-first dispatch balances in two rounds (Qwen3 4k 89.9 -> 86.7 us), and causal
// grids of at most one tile per CU: those whose keys before the query block are at least as
// many as the queries take the key split like non-causal grids (16 heads of 1024 rows over
// 4096 keys 52.3 -> 48 us, 8 heads 36.5 -> 34.3 us, 512 rows over 8192 keys +1-6%, 128 or 256
// rows over 8k-16k keys within -1.5 to +1.5%), triangular ones the causal split only where it
// pays (launch_prefill_fast_nw): Qwen3 2k 36.8 -> 33.8 us, Qwen3 1k 21.6 -> 19.5 us, 8 heads
// at 2k 28.2 -> 26.2 us. Where it
// adds rounds it lost: c3 1k causal (1024 tiles) 53 -> 65 us, Qwen3 2k causal (256 tiles,
// 384 with the causal key split) 37.7 -> 42.8 us, 48 heads of 1000 rows over 4000 keys at
// D = 96 causal (384 tiles) -2 to -7%. On full grids key halves everywhere (forced) lost
// 10-18% against 256-row workgroups (c3 4k 0.975 -> 1.095 ms, c3 4k causal 0.577 -> 0.657 ms,
// c4 0.284 -> 0.319 ms): twice the workgroups, each with its fixed cost and a merge.
// At D = 64 (4-wave workgroups there keep 128-key tiles, two per CU) it measured: 32 heads at
// 1k 27.7 -> 15.7 us, 16 heads at 2k 37.4 -> 25.5 us, 24 heads of 512 rows over 4000 keys
// +18%, 16 heads at 2k / 4k causal +14% / +7%; config 1 (two key tiles) 6.5 -> 7.0 us, so at
// D = 64 key halves need at least four key tiles (no such limit was measured at D > 64, where
// the 4-wave alternative takes 64-key tiles). Slot-balanced head-split grids keep 4 waves.
// ATTN_PREFILL_KH=0 (read once) keeps the 4-wave workgroups and =2 takes key halves wherever
// 4 waves run at D >= 64 (with ATTN_PREFILL_WAVES=4: everywhere), for tuning sweeps.
static bool prefill_kh(int DP, int Hq, int Sq, int Sk, bool causal) {
    static int env = -1;
    if (env < 0) {
        const char *e = getenv("ATTN_PREFILL_KH");
        env = (e && (atoi(e) == 0 || atoi(e) == 2)) ? atoi(e) : 1;
    }
    const long n = (long)Hq * ((Sq + 127) / 128), cus = device_cus();
    return env == 2 || (env == 1 && (DP > 64 || Sk > 3 * 128) &&
                        (n <= cus || (causal && n == 2 * cus)));
}

// ATTN_PREFILL_KT=64 or =128 (read once) forces the prefill key tile for tuning sweeps: 64 keys
// on 8-wave workgroups, or 128 keys on 4-wave workgroups at D > 64 (one such workgroup per CU).
static int prefill_kt_forced() {
    static int forced = -1;
    if (forced < 0) {
        const char *e = getenv("ATTN_PREFILL_KT");
        forced = (e && (atoi(e) == 64 || atoi(e) == 128)) ? atoi(e) : 0;
    }
    return forced;
}

// The persistent prefill (attn_prefill_persist_kernel) for 8-wave grids of at least two rounds,
// non-causal or causal: ATTN_PREFILL_PERSIST=0 (read once) turns it off for tuning sweeps.
static int prefill_persist() {
    static int env = -1;
    if (env < 0) {
        const char *e = getenv("ATTN_PREFILL_PERSIST");
        env = (e && atoi(e) == 0) ? 0 : 1;
    }
    return env;
}

// Whether a grid suits the persistent prefill: at least two items (256-row query tiles) per
// CU; every item's key-tile count even and at least two (the kernel's compile-time buffer
// order); causal: Sk >= Sq (every row sees key 0) and an even tile count (the pairs).
static bool prefill_persist_fits(int Hq, int Sq, int Sk, int D, bool causal) {
    const int nqt = (Sq + 255) / 256;
    if ((long)Hq * nqt < 2L * device_cus() || (long)Sq * D * 4 >= 0x7fffffffL)
        return false;
    if (!causal)
        return Sk > 128 && ((Sk + 127) / 128) % 2 == 0;
    if (Sk < Sq || nqt % 2 != 0)
        return false;
    for (int qt = 0; qt < nqt; ++qt) {
        const int nk = (Sk - Sq + std::min(Sq - 1, qt * 256 + 255)) / 128 + 1;
        if (nk < 2 || nk % 2 != 0)
            return false;
    }
    return true;
}

// Whether a causal grid suits the persistent prefill with key halves: exactly two 128-row
// query tiles per CU (where the per-tile kernel would run key halves in two rounds), so that
// each workgroup runs one pair (the kernel's buffer order assumes at most one); whole tiles
// (Sq % 128 == 0: a pair's key-tile counts then add up to an odd number), an even tile count
// per head (the pairs) and Sk >= Sq (every row sees key 0).
static bool prefill_persist_kh_fits(int Hq, int Sq, int Sk, int D) {
    const int nqt = Sq / 128;
    return Sk >= Sq && Sq % 128 == 0 && nqt % 2 == 0 && device_cus() % 8 == 0 &&
           (long)Hq * nqt == 2L * device_cus() && (long)Sq * D * 4 < 0x7fffffffL;
}

// One workgroup per CU (a multiple of 8: each XCD takes the same count), each running its
// items of the 256-row tiling (KH: 128-row) back to back (causal: pairs of items).
template <int DP, bool CAUSAL, bool KH = false>
hipError_t launch_prefill_persist(const uint16_t *Q, const uint16_t *K, const uint16_t *V,
                                  float *O, int Hq, int Hkv, int Sq, int Sk, int D, float c,
                                  hipStream_t st) {
    constexpr int BQ = KH ? 128 : 256;
    const int nqt = (Sq + BQ - 1) / BQ;
    const long nunits = (long)Hq * nqt / (CAUSAL ? 2 : 1);
    const int nwg = device_cus() / 8 * 8;
    if (nunits <= 0 || nunits > 0x3fffffffL || nwg <= 0 || (KH && nunits > nwg))
        return hipErrorInvalidValue;
    if (t_plan)
        plan_note(dim3((unsigned)nwg), dim3(512),
                  "attn_prefill_persist_kernel<%d, %s, %s> units=%ld", DP, tf(CAUSAL), tf(KH),
                  nunits);
    else
        hipLaunchKernelGGL((attn_prefill_persist_kernel<DP, CAUSAL, KH>), dim3((unsigned)nwg),
                           dim3(512), 0, st, Q, K, V, O, Hq, Hkv, Sq, Sk, D, c, nqt, (int)nunits,
                           nwg);
    return hipGetLastError();
}

// 8 waves at D > 128 (attn_prefill_fast_kernel's kRing) instead of 4; either way a CU holds one
// workgroup. A round of 256-row workgroups takes 1.67 times a round of 128-row ones (D = 256 and 192,
// 64 heads at 2k), so 8 waves are taken where their rounds are under 4/7 of the others': 36 heads of 1024
// rows, D = 192, 103 -> 72 us, 128 heads of 400 rows 50 -> 38; one round either way (32
// heads of 1000 rows, D = 256) 77 with 4 waves, 85 with 8. Not where 256-row tiles are padded much more
// (300 rows, 128 heads: 213 and 218). Triangular causal grids are balanced heaviest first, down to
// their longest item: 8 waves where the larger of that and the mean load falls under 3/4 (48 heads
// at 2k 122 -> 106 us; 24 heads 70 with 4 waves, 88 with 8; 16 heads at 4k 141 and 159).
// Unaligned tensors (ua): a round takes the same time with both, so 8 waves wherever they
// need fewer tiles (16 heads of 200 rows 27.6 -> 28.6 us, 24 heads of 300 47 -> 43, of 1500 causal
// 100 -> 68, 4 heads of 700 over 5000 keys 68 -> 54).
static bool prefill_wide8(int Hq, int Hkv, int Sq, int Sk, bool causal, bool ua = false) {
    if (const int forced = prefill_waves_forced())
        return forced == 8;
    if (prefill_pack(Hq, Hkv, Sq))
        return false;
    const long cus = device_cus();
    const long t4 = (Sq + 127) / 128, t8 = (Sq + 255) / 256, n4 = Hq * t4, n8 = Hq * t8;
    if (ua)
        return t8 < t4;
    if (8 * t8 > 5 * t4)
        return false;
    if (causal && (long)Sk - Sq < Sq) {
        // std::max: HIP's host max takes int, and these products pass 2^31.
        auto load = [&](long n) { return std::max((long)Sk * cus, n * (Sk - Sq / 2)); };
        return 4 * load(n8) < 3 * load(n4);
    }
    return 7 * ((n8 + cus - 1) / cus) < 4 * ((n4 + cus - 1) / cus);
}

template <int DP, int KT, bool CAUSAL, bool VT>
hipError_t launch_prefill_fast_t(const uint16_t *Q, const uint16_t *K, const uint16_t *V, float *O,
                                 int Hq, int Hkv, int Sq, int Sk, int D, float c, float *pm,
                                 float *pl, float *pacc, long slots, hipStream_t st) {
    constexpr int KT4 = (DP > 64 && KT == 128) ? 64 : KT; // the 4-wave key tile (below)
    const bool hs = !CAUSAL && DP <= 64 && !prefill_pack(Hq, Hkv, Sq) &&
                    prefill_head_split(Hq, Sq, (Sq + 127) / 128, (Sk + KT4 - 1) / KT4,
                                       pm ? slots : 0, pm != nullptr) > 0;
    if constexpr (DP == 64 && KT == 128 && !CAUSAL)
        if (hs && !prefill_waves_forced() && prefill_rows192(Hq, Hkv, Sq))
            return launch_prefill_fast_nw<DP, KT, 12, CAUSAL, VT, true>(Q, K, V, O, Hq, Hkv, Sq, Sk,
                                                                        D, c, pm, pl, pacc, slots,
                                                                        st);
    const int nw = (DP <= 128) ? prefill_waves(Hq, Hkv, Sq, Sk, CAUSAL, hs) : 4;
    // Tuning override of the key tile (the other of 64 / 128 keys), non-V^T only; the counter
    // study that fixed the defaults runs through it.
    if constexpr (DP <= 128 && KT == 128 && !VT) {
        if (prefill_kt_forced() == 64 && nw == 8)
            return launch_prefill_fast_nw<DP, 64, 8, CAUSAL, VT>(Q, K, V, O, Hq, Hkv, Sq, Sk, D, c,
                                                                 pm, pl, pacc, slots, st);
        if (prefill_kt_forced() == 128 && nw == 4 && DP > 64)
            return launch_prefill_fast_nw<DP, 128, 4, CAUSAL, VT>(Q, K, V, O, Hq, Hkv, Sq, Sk, D,
                                                                  c, pm, pl, pacc, slots, st);
    }
    if constexpr (DP >= 64 && DP <= 128 && KT == 128)
        if (nw == 4 && !hs && !prefill_pack(Hq, Hkv, Sq) && prefill_kh(DP, Hq, Sq, Sk, CAUSAL)) {
            // Causal grids of two 128-row tiles per CU with row-major V run their key halves
            // persistent: each CU's heavy and light tile in one workgroup.
            if constexpr (DP == 128 && CAUSAL && !VT)
                if (prefill_persist() && prefill_persist_kh_fits(Hq, Sq, Sk, D))
                    return launch_prefill_persist<DP, CAUSAL, true>(Q, K, V, O, Hq, Hkv, Sq, Sk,
                                                                    D, c, st);
            return launch_prefill_fast_nw<DP, KT, 8, CAUSAL, VT, true>(Q, K, V, O, Hq, Hkv, Sq, Sk,
                                                                       D, c, pm, pl, pacc, slots,
                                                                       st);
        }
    // Grids of at least two rounds of 8-wave workgroups with row-major V whose items suit it
    // run persistent (attn_prefill_persist_kernel). So do causal grids that take 4-wave
    // workgroups for their short key ranges (prefill_waves) when their pairs of 256-row items
    // fill the CUs evenly (at most 10% of the pair slots idle): same box, 4-wave -> persistent,
    // c3 shape at 1k causal 47.4 -> 46.0 us, 1000 rows 47.1 -> 45.6, 2k 144.8 -> 140.0, 64 heads
    // at 2k 75.9 -> 72.7, MQA-like 128 heads over 8 kv heads at 1k 45.0 -> 45.9; unevenly
    // (96 heads at 1536: 288 pairs on 256 CUs) 67.6 -> 98.9.
    if constexpr (DP == 128 && KT == 128 && !VT) {
        bool persist = nw == 8;
        if (CAUSAL && nw == 4 && !prefill_waves_forced()) {
            const long units = (long)Hq * ((Sq + 255) / 256) / 2, nwg = device_cus() / 8 * 8;
            persist = nwg > 0 && 10 * (((units + nwg - 1) / nwg) * nwg - units) <= units;
        }
        if (persist && prefill_persist() && !prefill_pack(Hq, Hkv, Sq) &&
            prefill_persist_fits(Hq, Sq, Sk, D, CAUSAL))
            return launch_prefill_persist<DP, CAUSAL>(Q, K, V, O, Hq, Hkv, Sq, Sk, D, c, st);
    }
    if constexpr (DP <= 128 && KT * DP / 8 >= 512) // every thread of 8 waves stages a chunk
        if (nw == 8)
            return launch_prefill_fast_nw<DP, KT, 8, CAUSAL, VT>(Q, K, V, O, Hq, Hkv, Sq, Sk, D, c,
                                                                 pm, pl, pacc, slots, st);
    if constexpr (DP > 128)
        if (prefill_wide8(Hq, Hkv, Sq, Sk, CAUSAL))
            return launch_prefill_fast_nw<DP, DP == 192 ? 64 : 32, 8, CAUSAL, VT>(
                Q, K, V, O, Hq, Hkv, Sq, Sk, D, c, pm, pl, pacc, slots, st);
    // 4-wave workgroups at D > 64 take 64-key tiles: at 128 keys the tiles use 96-128 KB of LDS
    // and a CU could hold only one such workgroup (one wave per SIMD). At D > 128 the grids that
    // prefill_wide8 leaves take them, one workgroup per CU.
    return launch_prefill_fast_nw<DP, KT4, 4, CAUSAL, VT>(Q, K, V, O, Hq, Hkv, Sq, Sk, D, c, pm,
                                                          pl, pacc, slots, st);
}

// Unaligned tensors (UA): the aligned kernels' choice of workgroup, without the persistent and 12-wave
// variants. Key tiles: 64 keys on 4 and 8 waves at D in (64, 128] (two staged pieces per thread and
// tensor at 8 waves), 128 at D <= 64 and for key halves, 32 past D = 128.
template <int DP, int KT, bool CAUSAL, bool VT>
hipError_t launch_prefill_ua(const uint16_t *Q, const uint16_t *K, const uint16_t *V, float *O,
                             int Hq, int Hkv, int Sq, int Sk, int D, float c, float *pm, float *pl,
                             float *pacc, long slots, hipStream_t st) {
    constexpr int KT4 = (DP > 128) ? 32 : (DP > 64 && KT == 128) ? 64 : KT;
    if constexpr (DP == 64)
        if (D < 8)
            return launch_prefill_fast_nw<DP, KT4, 4, CAUSAL, VT, false, 2>(
                Q, K, V, O, Hq, Hkv, Sq, Sk, D, c, pm, pl, pacc, slots, st);
    if constexpr (DP <= 128) {
        const int nw = prefill_waves(Hq, Hkv, Sq, Sk, CAUSAL, false);
        if (nw == 4 && !prefill_pack(Hq, Hkv, Sq) && prefill_kh(DP, Hq, Sq, Sk, CAUSAL))
            return launch_prefill_fast_nw<DP, KT, 8, CAUSAL, VT, true, 1>(
                Q, K, V, O, Hq, Hkv, Sq, Sk, D, c, pm, pl, pacc, slots, st);
        if (nw == 8)
            return launch_prefill_fast_nw<DP, KT4, 8, CAUSAL, VT, false, 1>(
                Q, K, V, O, Hq, Hkv, Sq, Sk, D, c, pm, pl, pacc, slots, st);
    }
    if constexpr (DP > 128)
        if (prefill_wide8(Hq, Hkv, Sq, Sk, CAUSAL, true))
            return launch_prefill_fast_nw<DP, KT4, 8, CAUSAL, VT, false, 1>(
                Q, K, V, O, Hq, Hkv, Sq, Sk, D, c, pm, pl, pacc, slots, st);
    return launch_prefill_fast_nw<DP, KT4, 4, CAUSAL, VT, false, 1>(
        Q, K, V, O, Hq, Hkv, Sq, Sk, D, c, pm, pl, pacc, slots, st);
}

// DMA staging needs D % 8 == 0 with D <= DP, 16-byte vectors (vec; with V^T also
// Sk % 8 == 0, which the host folds into vec) and a kv head's bytes within a buffer's 31-bit
// range; other calls take the unaligned instances. D in (64, 96] takes the 96-wide instance and
// D in (128, 192] the 192-wide one, whose MFMA tiles waste less on padding (64 heads at 2k, D = 192
// in 256-wide tiles 294 us, in 192-wide ones 222; D = 160 causal 164 -> 121).
template <int DP, int KT>
hipError_t launch_prefill_dk(const uint16_t *Q, const uint16_t *K, const uint16_t *V, float *O,
                             int Hq, int Hkv, int Sq, int Sk, int D, int causal, int vec, int vt,
                             float c, float *pm, float *pl, float *pacc, long slots,
                             hipStream_t st) {
    const bool fast = vec && D % 8 == 0 && D <= DP && (long)Sk * D * 2 < 0x7fffffffL;
    return with_flag(causal != 0, [&](auto CA) {
        return with_flag(vt != 0, [&](auto VTF) {
            constexpr bool kC = decltype(CA)::value, kT = decltype(VTF)::value;
            auto go = [&](auto DPW) {
                constexpr int W = decltype(DPW)::value;
                return fast ? launch_prefill_fast_t<W, KT, kC, kT>(Q, K, V, O, Hq, Hkv, Sq, Sk, D,
                                                                   c, pm, pl, pacc, slots, st)
                            : launch_prefill_ua<W, KT, kC, kT>(Q, K, V, O, Hq, Hkv, Sq, Sk, D, c,
                                                               pm, pl, pacc, slots, st);
            };
            if constexpr (DP == 128)
                if (D <= 96)
                    return go(std::integral_constant<int, 96>{});
            if constexpr (DP == 256)
                if (D <= 192)
                    return go(std::integral_constant<int, 192>{});
            return go(std::integral_constant<int, DP>{});
        });
    });
}

template <int DP>
hipError_t launch_prefill_d(const uint16_t *Q, const uint16_t *K, const uint16_t *V, float *O,
                            int Hq, int Hkv, int Sq, int Sk, int D, int causal, int vec, int vt,
                            float c, float *pm, float *pl, float *pacc, long slots,
                            hipStream_t st) {
    // Key tiles of 128 keys up to D = 128, the largest that keeps two waves per SIMD. D in
    // (128, 256]: 64 keys (two 64-key K and V tiles fill 128 KB of LDS).
    return launch_prefill_dk<DP, DP == 256 ? 64 : 128>(Q, K, V, O, Hq, Hkv, Sq, Sk, D, causal, vec,
                                                       vt, c, pm, pl, pacc, slots, st);
}

// Non-temporal K/V loads in the decode kernels: only when every K/V byte is read by exactly one
// workgroup (one 16-row block per kv head, nrb == 1) over a long key range (kps keys). Row
// blocks that share a key range through L2 lose 16-31% with them (256 / 32 heads, Sq = 8,
// Sk = 4096; 1024 / 64 heads, Sq = 4, Sk = 8192), and short ranges (512-1024 keys per
// workgroup: 32 / 8 heads over 32768 keys, 64 / 8 heads over 65536) lose 4-6%. Long ranges of
// 4096 keys gain 2.4-5.7% (config 2) and up to 18% at D = 64. ATTN_DECODE_NT=0 or =1 (read
// once) forces them off or on for tuning sweeps.
constexpr int kDecodeNTMinKeys = 2048;
static bool decode_nt_loads(int nrb, int kps) {
    static int forced = -2;
    if (forced == -2) {
        const char *e = getenv("ATTN_DECODE_NT");
        forced = (e && (atoi(e) == 0 || atoi(e) == 1)) ? atoi(e) : -1;
    }
    if (forced >= 0)
        return forced == 1;
    return nrb == 1 && kps >= kDecodeNTMinKeys;
}

static bool decode_vt_staged() {
    static int on = -1;
    if (on < 0) {
        const char *e = getenv("ATTN_DECODE_VT_STAGED");
        on = (e && atoi(e) == 0) ? 0 : 1;
    }
    return on == 1;
}

template <int DP>
hipError_t launch_decode_d(const uint16_t *Q, const uint16_t *K, const uint16_t *V, float *O,
                           float *pm, float *pl, float *pacc, int Hq, int Hkv, int Sq, int Sk,
                           int D, int causal, int vec, int vt, float c, int nsplit, int kps,
                           int nrb, hipStream_t st) {
    const long nblk = (long)Hkv * nsplit * nrb;
    if (nblk <= 0 || nblk > 0x7fffffffL)
        return hipErrorInvalidValue;
    const bool ntl = decode_nt_loads(nrb, kps);
    const int blocks = attn_decode_cut_of(Hq, Hkv, Sq, Sk, nrb, DP).blocks;
    // The staged V^T kernel, for one row block per workgroup and more than one 128-key step: its
    // pipeline fills over five barrier intervals (8 kv heads over 776 keys in one-step splits 10.3 us,
    // attn_decode_kernel straight from V^T 8.2; over 777 keys 14.2 and 10.0; two steps and up it is
    // the faster one, 64 kv heads over 3001 keys 24.0 and 28.0). Its DMA offsets are 32-bit: a head's
    // aligned V^T must stay below 2 GiB. Grouped row blocks read V^T once straight from memory (32 kv
    // heads, 64 rows over 4000 keys: staged per block 33, this 25.5). Unaligned V^T passes through
    // registers on its way to LDS, padding rows too, so there the staged kernel needs D > 32 and more
    // than two steps: against attn_decode_kernel, 128 kv heads x 4001 keys at D = 100 46.4 and 54.9
    // us, at D = 20 1.15-1.2 times its time, with two steps at any D 1.0 to 1.4 times.
    if constexpr (DP <= 128)
        if (vt && blocks == 1 && kps > ATTN_DECODE_MIN_KEYS && decode_vt_staged() &&
            (vec ? (long)D * Sk * 2 < 0x7fffffffL : D > 32 && kps > 2 * ATTN_DECODE_MIN_KEYS))
            return with_flag(causal != 0, [&](auto CA) {
                return with_flag(ntl, [&](auto NT) {
                    auto launch = [&](auto UAF) {
                        constexpr bool kC = decltype(CA)::value, kN = decltype(NT)::value;
                        constexpr int kU = decltype(UAF)::value;
                        if (t_plan)
                            plan_note(dim3((unsigned)nblk), dim3(256),
                                      "attn_decode_vt_kernel<%d, %s, %s%s> nsplit=%d nrb=%d", DP,
                                      tf(kC), tf(kN), kU ? ", unaligned" : "", nsplit, nrb);
                        else
                            hipLaunchKernelGGL((attn_decode_vt_kernel<DP, kC, kN, kU>),
                                               dim3((unsigned)nblk), dim3(256), 0, st, Q, K, V, O,
                                               pm, pl, pacc, Hq, Hkv, Sq, Sk, D, c, nsplit, kps,
                                               nrb);
                        return hipGetLastError();
                    };
                    return vec          ? launch(std::integral_constant<int, 0>{})
                           : D % 8 == 0 ? launch(std::integral_constant<int, 1>{})
                                        : launch(std::integral_constant<int, 2>{});
                });
            });
    // The row-major instances at DP = 128 keep three workgroups on a CU. A grid a little past three
    // per CU then ends in a round of few workgroups, which long key ranges feel; where rounds of
    // two per CU are a fifth better filled, LDS that nobody uses holds the third one back. 400 heads x
    // 3560 keys at D = 96 (800 workgroups) two per CU 101.3, three 109.5, this 100.7 us; 420 x 6000
    // 173, 180, 174; at under 1024 keys per workgroup three stay ahead (400 x 1000 35.9, 35.3).
    auto hold_third = [&](long n) -> unsigned {
        const long c2 = 2L * device_cus(), c3 = 3L * device_cus();
        const bool two = n > c3 && kps >= 1024 &&
                         6 * ((n + c2 - 1) / c2 * c2) < 5 * ((n + c3 - 1) / c3 * c3);
        return two ? 17408 : 0; // with the kernel's 37376 bytes, three do not fit 160 KB
    };
    auto go = [&](auto NB) {
        constexpr int NRB = decltype(NB)::value;
        const int ng = (nrb + NRB - 1) / NRB; // row block groups
        const long n = (long)Hkv * nsplit * ng;
        auto launch = [&](auto CA, auto ALF, auto VTF, auto NT) {
            constexpr bool kC = decltype(CA)::value, kT = decltype(VTF)::value,
                           kN = decltype(NT)::value;
            constexpr int kA = decltype(ALF)::value;
            constexpr bool kThree = DP == 128 && kA != 2 && !kT && NRB == 1;
            if (t_plan)
                plan_note(dim3((unsigned)n), dim3(256),
                          "attn_decode_kernel<%d, %s, %s, %s, %s%s%s> nsplit=%d nrb=%d%s", DP,
                          tf(kC), tf(kA == 1), tf(kT), tf(kN), kA == 2 ? ", short" : "",
                          NRB == 2 ? ", 2 blocks" : "", nsplit, nrb,
                          kThree && hold_third(n) ? " two-per-cu=1" : "");
            else
                hipLaunchKernelGGL((attn_decode_kernel<DP, kC, kA, kT, kN, NRB>),
                                   dim3((unsigned)n), dim3(256), kThree ? hold_third(n) : 0, st, Q, K, V, O, pm, pl, pacc,
                                   Hq, Hkv, Sq, Sk, D, c, nsplit, kps, ng);
            return hipGetLastError();
        };
        return with_flag(causal != 0, [&](auto CA) {
            return with_flag(vt != 0, [&](auto VTF) {
                // Rows shorter than a piece: of Q, K and V (D < 8, so DP = 64) or of V^T.
                if constexpr (DP == 64 || decltype(VTF)::value)
                    if (!vec && (D < 8 || (vt && Sk < 8)))
                        return launch(CA, std::integral_constant<int, 2>{}, VTF, std::false_type{});
                return with_flag(ntl, [&](auto NT) {
                    return vec ? launch(CA, std::integral_constant<int, 1>{}, VTF, NT)
                               : launch(CA, std::integral_constant<int, 0>{}, VTF, NT);
                });
            });
        });
    };
    if constexpr (DP <= 128)
        if (blocks == 2)
            return go(std::integral_constant<int, 2>{});
    return go(std::integral_constant<int, 1>{});
}

} // namespace

// ---- extern "C" launchers called by the C host layer (attn_flash.c) -------------------------
// vt = 1: V is V^T [Hkv][D][Sk] (pack_v_full's layout); vec must then also imply Sk % 8 == 0.
// pm/pl/pacc: split partial slots in the caller's scratch (slots of them); NULL disables the
// causal key split.
extern "C" int attn_hip_launch_prefill(const uint16_t *Q, const uint16_t *K, const uint16_t *V,
                                       float *O, int Hq, int Hkv, int Sq, int Sk, int D,
                                       int causal, int vec, int vt, int dp, float c,
                                       float *pm, float *pl, float *pacc, long slots,
                                       void *stream) {
    hipStream_t st = (hipStream_t)stream;
    switch (dp) {
    case 64:
        return (int)launch_prefill_d<64>(Q, K, V, O, Hq, Hkv, Sq, Sk, D, causal, vec, vt, c,
                                         pm, pl, pacc, slots, st);
    case 128:
        return (int)launch_prefill_d<128>(Q, K, V, O, Hq, Hkv, Sq, Sk, D, causal, vec, vt, c,
                                          pm, pl, pacc, slots, st);
    case 256:
        return (int)launch_prefill_d<256>(Q, K, V, O, Hq, Hkv, Sq, Sk, D, causal, vec, vt, c,
                                          pm, pl, pacc, slots, st);
    default:
        return (int)hipErrorInvalidValue;
    }
}

// nrb: 16-row blocks per kv head (g*Sq rows); attn_decode_cut_of has how many a workgroup serves.
extern "C" int attn_hip_launch_decode(const uint16_t *Q, const uint16_t *K, const uint16_t *V,
                                      float *O, float *pm, float *pl, float *pacc, int Hq,
                                      int Hkv, int Sq, int Sk, int D, int causal, int vec, int vt,
                                      int dp, float c, int nsplit, int kps, int nrb,
                                      void *stream) {
    hipStream_t st = (hipStream_t)stream;
    switch (dp) {
    case 64:
        return (int)launch_decode_d<64>(Q, K, V, O, pm, pl, pacc, Hq, Hkv, Sq, Sk, D, causal, vec,
                                        vt, c, nsplit, kps, nrb, st);
    case 128:
        return (int)launch_decode_d<128>(Q, K, V, O, pm, pl, pacc, Hq, Hkv, Sq, Sk, D, causal,
                                         vec, vt, c, nsplit, kps, nrb, st);
    case 256:
        return (int)launch_decode_d<256>(Q, K, V, O, pm, pl, pacc, Hq, Hkv, Sq, Sk, D, causal,
                                         vec, vt, c, nsplit, kps, nrb, st);
    default:
        return (int)hipErrorInvalidValue;
    }
}

// Compute units of the current device, for the host layer's kernel choice.
extern "C" int attn_hip_device_cus(void) { return device_cus(); }

// Phase stamps (ATTN_PHASE_STAMPS builds only): the persistent prefill's later launches write
// kPhaseSlots 64-bit stamps per workgroup into buf (device memory of at least workgroups *
// slots * 8 bytes; NULL is not allowed). Returns the slot count, or -1 in a build without
// stamps or when the pointer cannot be set.
extern "C" int attn_hip_phase_stamps(void *buf) {
#if ATTN_PHASE_STAMPS
    if (!buf)
        return -1;
    unsigned long long *p = static_cast<unsigned long long *>(buf);
    if (hipMemcpyToSymbol(HIP_SYMBOL(g_phase_stamps), &p, sizeof p) != hipSuccess)
        return -1;
    return kPhaseSlots;
#else
    (void)buf;
    return -1;
#endif
}

// Plan recording for attn_flash_plan: between begin and end, the launchers of the calling
// thread write kernel lines into buf (NUL-terminated) instead of launching. end returns the
// length written, or -1 if buf was too small for every line.
namespace {
thread_local plan_buf t_plan_state;
}
extern "C" void attn_hip_plan_begin(char *buf, size_t len) {
    t_plan_state = plan_buf{buf, len, 0, false};
    if (len > 0)
        buf[0] = '\0';
    t_plan = &t_plan_state;
}
extern "C" long attn_hip_plan_end(void) {
    t_plan = nullptr;
    return t_plan_state.truncated ? -1L : (long)t_plan_state.pos;
}

extern "C" int attn_hip_launch_merge(const float *pm, const float *pl, const float *pacc,
                                     float *O, int rows, int D, int nsplit, float c, int Sq,
                                     void *stream) {
    return (int)launch_merge(pm, pl, pacc, O, rows, D, nsplit, c, Sq, 0, Sq, (hipStream_t)stream);
}

// Keys per pack tile: 128 (256-byte pieces of each V^T row per store). Measured on c3 4k V
// (inputs rotated past the Infinity Cache): 64 keys 14.1 us, 128 keys 12.65 us, 256 keys 14.4 us,
// 512 keys 17.8 us. Without the vector layout the same tiles read and write 16 bytes at element
// alignment; against 32 x 32 tiles of
// single elements, packing 6 heads of 2003 keys at D = 100 and attending 59.1 -> 56.8 us.
constexpr int kPackTK = 128;

extern "C" int attn_hip_launch_pack_v(const uint16_t *V, uint16_t *Vp, int Hkv, int Sk, int D,
                                      void *stream) {
    if (Hkv <= 0 || Sk <= 0 || D <= 0)
        return (int)hipErrorInvalidValue;
    const bool v16 = D % 8 == 0 && Sk % 8 == 0 && (((uintptr_t)V | (uintptr_t)Vp) & 15u) == 0;
    // The kv head is the grid's z index, at most 65535 per launch: larger Hkv runs in chunks
    // (each chunk's base stays 16-byte aligned, since Sk*D is a multiple of 8 on the v16 path).
    constexpr int kMaxZ = 65535;
    for (int h0 = 0; h0 < Hkv; h0 += kMaxZ) {
        const unsigned nh = (unsigned)std::min(kMaxZ, Hkv - h0);
        const size_t off = (size_t)h0 * Sk * D;
        constexpr int TK = kPackTK;
        dim3 grid((unsigned)((Sk + TK - 1) / TK), (unsigned)((D + 63) / 64), nh);
        if (v16)
            hipLaunchKernelGGL((attn_pack_v16_kernel<TK, true>), grid, dim3(256), 0,
                               (hipStream_t)stream, V + off, Vp + off, Sk, D);
        else
            hipLaunchKernelGGL((attn_pack_v16_kernel<TK, false>), grid, dim3(256), 0,
                               (hipStream_t)stream, V + off, Vp + off, Sk, D);
        const hipError_t e = hipGetLastError();
        if (e != hipSuccess)
            return (int)e;
    }
    return (int)hipSuccess;
}

// ---- allocation-free scratch (attn_flash_noalloc) -------------------------------------------
// The split-K partial slots of attn_flash_noalloc: the layout of a caller's attn_flash scratch
// at D = ATTN_NOALLOC_D_MAX, one copy per GPU, held until the process ends. The kernels write
// every slot they later read, so nothing in it has to start at zero. In host code the name
// `scratch` is a host-side stand-in, not a device address: the device address comes from
// hipGetSymbolAddress, once per device with that device current, and only that address is
// ever passed to a kernel.
static __device__ __align__(256) unsigned char scratch[ATTN_NOALLOC_SCRATCH_BYTES];

namespace {
constexpr int kMaxDevices = 64;
std::atomic<void *> g_scratch_addr[kMaxDevices]; // per device; zero until first resolved
} // namespace

// Device address and size of the current device's static scratch. Two threads that resolve it
// at once both store the same address, so no lock is needed.
extern "C" int attn_hip_static_scratch(void **ptr, size_t *bytes) {
    int dev = -1;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess)
        return (int)e;
    if (dev < 0 || dev >= kMaxDevices)
        return (int)hipErrorInvalidDevice;
    void *p = g_scratch_addr[dev].load(std::memory_order_acquire);
    if (!p) {
        e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess)
            return (int)e;
        if (!p)
            return (int)hipErrorInvalidSymbol;
        g_scratch_addr[dev].store(p, std::memory_order_release);
    }
    *ptr = p;
    *bytes = sizeof(scratch);
    return (int)hipSuccess;
}
