// w6a16.hip -- weight-only 6-bit GEMM / GEMV (W6A16) on gfx950, reading the reference's bit-plane format directly.
//
// Format (rwkv_next/kernels/int6_gemm.py:14-38, 73-112): a (K, N) weight, N contiguous, quantised symmetrically to
// q in [-32, 31] per (group of group_k rows, column) with an fp16 scale s, w ~ s q.  Stored as u = q + 32 in [0, 63]
// split over two byte planes per 64-row chunk c:
//     lo[c*32 + j][n] = (u[c*64 + j] & 15) | (u[c*64 + j + 32] & 15) << 4                         j < 32
//     hi[c*16 + j][n] = u[c*64 + j] >> 4 | (u[.. + j + 16] >> 4) << 2 | (u[.. + j + 32] >> 4) << 4
//                       | (u[.. + j + 48] >> 4) << 6                                                 j < 16
// C[b][m][n] = sum_k A[b][m][k] s[k / group_k][n] q[k][n] with fp32 accumulation (int6_gemm.py:156-215).
//
// Tile kernel (decode-sized M; every M on the planes): a workgroup of W wavefronts computes 16 MT rows x 16 NT columns,
// the wavefronts taking the 64-row chunks of K in turn, each on its own:
//   * weights are loaded straight into registers in the order the matrix instruction takes them (packed layout) or four
//     columns of eight rows a lane (planes) and become B operands of v_mfma_f32_16x16x32 without conversion
//     instructions: 0x4300 | u is the bf16 of 128 + u, exact, assembled for two values with one v_perm_b32.  One MFMA
//     pair per chunk and M tile against a constant B of -160 removes the bias (128 + u - 160 = q) exactly;
//   * the chunk's rows of A are loaded coalesced (128 bytes a row) and turned into A operands through the wavefront's own
//     LDS buffer;
//   * each chunk's fp32 tile is scaled by s (fp16) and accumulated; the wavefronts' tiles are summed through LDS, and
//     the tiles of several workgroups, where K is split over them, through the workspace, both in a fixed order.
// Wide kernel (145..256 rows, many columns) and large-M kernel (packed weights): described where they are defined.
// Rows m >= M read zeros and columns n >= N are clamped on load (they only feed outputs that are not stored).
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <algorithm>
#include <type_traits>
#include <utility>

#include "w6a16.h"
#include "w6a16_plan.h"
#include "wkv7_launch.h"

namespace w6 {
namespace {

typedef __bf16 bf8 __attribute__((ext_vector_type(8)));
typedef float f4 __attribute__((ext_vector_type(4)));
typedef uint32_t u4 __attribute__((ext_vector_type(4)));
typedef int v2i __attribute__((ext_vector_type(2)));
typedef __attribute__((address_space(3))) v2i lds_v2i;

struct Args {
    const uint16_t* a;
    int64_t sa_b, sa_m;
    const uint8_t *lo, *hi;
    int64_t sl_b, sh_b;
    const uint16_t* sc;
    int64_t ss_b;
    void* out;
    int64_t so_b, so_m;
    uint32_t* cnt;  // K split over workgroups: arrival counters, one per tile; zero between calls
    float* part;    // K split over workgroups: partial tiles [tile][split][rows][16 NT columns]
    int32_t B, M, N, K, group_k, out_dtype, n_strips;
    TileGrid grid;                   // tile kernel: M groups of 16 MT rows, columns of a workgroup's column tiles
    int32_t parts, per_part, groups;  // wavefronts that share K, chunks of the longest share, scale groups
    Divisor group;                   // chunk c's scale group is c over the chunks of a group
    float* rsum;                     // wide kernel: row-sum bias [batch][chain][mpad]
    int32_t mpad, chain_k, nchains;
    int32_t out_vec;  // large-M kernel: the output takes 8-byte (16-byte for fp32) stores of 4 adjacent columns
};

__device__ __forceinline__ float h2f(uint16_t h) { return (float)__builtin_bit_cast(_Float16, h); }

__device__ __forceinline__ f4 mfma(bf8 a, bf8 b, f4 c) { return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0); }

typedef _Float16 h8 __attribute__((ext_vector_type(8)));
typedef _Float16 h2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf2 __attribute__((ext_vector_type(2)));

// Activation element types.  The 6-bit code u becomes an exact MFMA operand 2^e + u with no conversion instruction
// (the code byte beside a constant high byte), and one MFMA pair per chunk against the constant -(2^e + 32) takes the
// offset out again: 2^e + u - (2^e + 32) = q exactly.  bf16 (the model's activations): 128 + u, high bytes 0x43,
// offset 160.  fp16 (the reference op casts its codes to a.dtype, rwkv_next/kernels/int6_gemm.py:144-147): 1024 + u,
// high bytes 0x64, offset 1056; the products stay exact in the fp32 accumulators.
struct ActBF16 {
    static constexpr uint32_t kCodeHi = 0x43434343u;
    static constexpr uint32_t kBias = 0xC320C320u;  // (-160, -160)
    static constexpr uint32_t kOnes = 0x3F803F80u;  // (1, 1)
    static constexpr float kOffset = 160.f;
    __device__ static f4 mma(u4 a, u4 b, f4 c) { return mfma(__builtin_bit_cast(bf8, a), __builtin_bit_cast(bf8, b), c); }
    __device__ static float dot2(uint32_t a, uint32_t b, float c) {
        return __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf2, a), __builtin_bit_cast(bf2, b), c, false);
    }
};
struct ActF16 {
    static constexpr uint32_t kCodeHi = 0x64646464u;
    static constexpr uint32_t kBias = 0xE420E420u;  // (-1056, -1056)
    static constexpr uint32_t kOnes = 0x3C003C00u;  // (1, 1)
    static constexpr float kOffset = 1056.f;
    __device__ static f4 mma(u4 a, u4 b, f4 c) {
        return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(h8, a), __builtin_bit_cast(h8, b), c, 0, 0, 0);
    }
    __device__ static float dot2(uint32_t a, uint32_t b, float c) {
        return __builtin_amdgcn_fdot2(__builtin_bit_cast(h2, a), __builtin_bit_cast(h2, b), c, false);
    }
};

// Orders LDS traffic between the lanes of one wavefront (its LDS instructions execute in issue order).
__device__ __forceinline__ void wave_lds_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// 4 codes u (one per byte) -> 4 operand values 2^e + u as two dwords.
template <class A>
__device__ __forceinline__ void codes_to_op(uint32_t u, uint32_t& lo2, uint32_t& hi2) {
    lo2 = __builtin_amdgcn_perm(A::kCodeHi, u, 0x04010400u);  // bytes: u0, hi, u1, hi
    hi2 = __builtin_amdgcn_perm(A::kCodeHi, u, 0x04030402u);  // bytes: u2, hi, u3, hi
}

__device__ __forceinline__ void store8(__bf16* dst, const float (&v)[8]) {
    uint32_t o[4];
#pragma unroll
    for (int e = 0; e < 4; ++e)
        o[e] = (uint32_t)__builtin_bit_cast(uint16_t, (__bf16)v[2 * e]) |
               (uint32_t)__builtin_bit_cast(uint16_t, (__bf16)v[2 * e + 1]) << 16;
    *reinterpret_cast<u4*>(dst) = u4{o[0], o[1], o[2], o[3]};
}

__device__ __forceinline__ void store8(_Float16* dst, const float (&v)[8]) {
    uint32_t o[4];
#pragma unroll
    for (int e = 0; e < 4; ++e)
        o[e] = (uint32_t)__builtin_bit_cast(uint16_t, (_Float16)v[2 * e]) |
               (uint32_t)__builtin_bit_cast(uint16_t, (_Float16)v[2 * e + 1]) << 16;
    *reinterpret_cast<u4*>(dst) = u4{o[0], o[1], o[2], o[3]};
}

__device__ __forceinline__ void store8(float* dst, const float (&v)[8]) {
    *reinterpret_cast<f4*>(dst) = f4{v[0], v[1], v[2], v[3]};
    *reinterpret_cast<f4*>(dst + 4) = f4{v[4], v[5], v[6], v[7]};
}

// Output element o of the call as its out_dtype, in kernels instantiated apart for fp16 outputs (F16) and for bf16 /
// fp32 ones.
template <bool F16>
__device__ __forceinline__ void put_out(const Args& p, int64_t o, float v) {
    if constexpr (F16)
        reinterpret_cast<_Float16*>(p.out)[o] = (_Float16)v;
    else if (p.out_dtype == W6A16_OUT_F32)
        reinterpret_cast<float*>(p.out)[o] = v;
    else
        reinterpret_cast<__bf16*>(p.out)[o] = (__bf16)v;
}

// Device-coherent accesses to the split-K partials: relaxed atomics at agent scope, which the compiler emits as
// plain stores / loads that bypass the caches that are not coherent across the chip (sc1).
__device__ __forceinline__ void coherent_store(float* p, float v) {
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

__device__ __forceinline__ float2 coherent_load2(const float* p) {
    const uint64_t u = __hip_atomic_load(reinterpret_cast<const uint64_t*>(p), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    return __builtin_bit_cast(float2, u);
}

// ---------------------------------------------------------------------------------------------------------------
// Packed layout: the same 6 bits per weight and fp16 scales, re-laid out once (w6a16_pack) so that each wavefront's
// 64-row chunk of a 128-column strip is one contiguous 6 KB block already in MFMA operand order.  Block (b, strip,
// chunk) lies at ((b * strips + strip) * chunks + chunk) * 6144; load instruction k (0..5) of lane l reads bytes
// k * 1024 + 16 l .. + 15, i.e. dwords 4 k .. 4 k + 3 of lane l's 24-dword record R.  For lane (i, q) = (l & 15,
// l >> 4) and tile t (column n = 128 strip + 16 t + i):
//   R[2 t], R[2 t + 1]  bytes e = 0..7: lo plane row chunk * 32 + 8 q + e (low nibble: row 8 q + e of the chunk,
//                       high nibble: row 32 + 8 q + e)
//   R[16 + t]           byte e' = 0..3: the top 2 bits of rows 8 q + e', 32 + 8 q + e', 8 q + 4 + e',
//                       32 + 8 q + 4 + e' at bits 0-1, 2-3, 4-5, 6-7
// Scales: block (b, strip, group) of 128 fp16 at ((b * strips + strip) * groups + group) * 128, ordered [i][t], so
// lane (i, q) reads its eight columns' scales as one 16-byte load.  Columns past N hold zero codes and scales.
using wkv7::unroll;  // f(integral_constant<0>), .., f(integral_constant<N - 1>)

// A raw buffer over [base, base + bytes) (capped at 2 GB).  The base and size are passed through readfirstlane so that
// the descriptor is provably wave-uniform: a descriptor the compiler cannot prove uniform is used through a per-lane
// loop.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t rsrc(uint64_t base, int64_t bytes) {
    const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)base);
    const uint32_t hi = __builtin_amdgcn_readfirstlane((uint32_t)(base >> 32));
    const int n = __builtin_amdgcn_readfirstlane(bytes < 0x7FFFFFFF ? (int)bytes : 0x7FFFFFFF);
    return __builtin_amdgcn_make_buffer_rsrc(reinterpret_cast<void*>(((uint64_t)hi << 32) | lo), 0, n,
                                             0x00020000 /* raw 32-bit buffer, gfx9 family */);
}

// A wave-uniform scalar offset (held in an SGPR, as buffer instructions need it).
__device__ __forceinline__ int soff(int x) { return __builtin_amdgcn_readfirstlane(x); }

// x s + a per element, written as a whole vector (stores into the components of an accumulator passed by reference
// kept the accumulators in scratch memory)
__device__ __forceinline__ f4 fma4(const f4 x, float s, const f4 a) {
    return f4{fmaf(x[0], s, a[0]), fmaf(x[1], s, a[1]), fmaf(x[2], s, a[2]), fmaf(x[3], s, a[3])};
}

// ---------------------------------------------------------------------------------------------------------------
// Tile kernel.  K is shared by `parts` wavefronts (part g takes the chunks g, g + parts, ..), which run in one
// workgroup or, `parts` / ks to a workgroup, in ks of them; their partial tiles are summed by quarters of the parts, in
// order within a quarter and then (q0 + q1) + (q2 + q3), so the result depends on `parts` alone and not on how they
// are placed: planes and packed weights give the same bits with different tiles.
//
// What bounds it: per-CU loads.  Every byte a workgroup reads passes its CU's vector L1, in order: a run of L2 hits (A)
// behind HBM misses (weights) gets about 20 bytes a clock through (measured with a load-only kernel: weights alone
// 8 B/clk at 5 TB/s over the chip, 1 : 2 mixed with L2 hits 19, 1 : 4 24), and a load instruction occupies the L1 for 2
// clocks per 128-byte line or 4 lanes, whichever is more.  Hence: A's rows by whole lines (17 clocks an instruction;
// loaded directly in operand order, 16 rows x 64 bytes, 65 clocks), the widest loads the layout allows (a 4-byte load
// at a 16-byte stride takes 32 clocks, an 8-byte one 17), 64 columns to a workgroup wherever that still gives every CU
// one, and no re-reading of A by narrower tiles.  No barrier in the loop and no LDS for the weights: the wavefronts
// drift apart and their loads, LDS turns and MFMAs overlap.
// Measured against the kernels it replaced (a strip-wide split-K kernel with a release fence per workgroup up to 32
// rows, above them a kernel of 128-column workgroups in lock-step with a row-sum pass before it), us per call, packed /
// planes: K = N = 4096, M = 1 11.5 / 11.6 -> 7.0 / 8.6, M = 16 26.1 / 26.1 -> 8.6 / 10.0, M = 64 17.6 / 18.4 -> 10.8 / 13.9; K =
// 4096, N = 16384, M = 1 12.5 / 17.0 -> 12.6 / 16.9, M = 64 27.0 / 29.9 -> 23.0 / 26.1; K = 2560, N = 10240, M = 203 52 / 62 -> 36
// / 41; K = 10240, N = 2560, M = 203 57 / 67 -> 28 / 34.  Where the old ones stayed ahead: wide_call (w6a16_plan.h), and 0.2 us
// of 4.5 at K = 512, N = 16384, 8 and 16 rows packed.
// Counters at K = 4096, N = 16384 (packed / planes): M = 1 MfmaUtil 5 / 4 %, VALUBusy 16 / 17 %; M = 64 16 / 14 and 23 / 23; M =
// 128 24 / 21 and 34 / 35, LDS under 13 %: no unit is near its limit; the wavefronts wait for loads.

// The weights of one chunk in one lane's registers.  Packed: the lane's record of its NT tiles (tile t: column
// n0 + 16 t + i); one tile takes the 8-byte pair its top bits lie in.
template <int NT, bool PACKED>
struct TileW {
    uint32_t lo[2 * NT], hd[NT < 2 ? 2 : NT], sc[2];
};
// Planes: lane (i, q) holds lo-plane rows 8 q + e (e = 0..7) and hi-plane rows 8 (q & 1) + 4 (q >> 1) + e (e = 0..3) of
// columns n0 + NT i .. + NT - 1, NT / 4 words a row, which are its columns of tiles 0..NT - 1 (tile t: columns n0 + NT i + t).
template <int NT>
struct TileW<NT, false> {
    uint32_t lo[2 * NT], hd[NT], sc[NT / 2];
};

// The wavefront's loads: wave-uniform 64-bit bases (moved from chunk to chunk on the scalar unit) and 32-bit per-lane
// offsets fixed for the call, through raw buffers.  A's buffer ends with its last valid row: rows past M read zeros.
// FAR, for planes whose 32 rows span 2 GB and for rows of A so far apart that a workgroup's 64 do: 64-bit lane offsets of
// the planes and their scales, 64-bit addresses of A's rows (rows past M read the last one; they only feed outputs that
// are not stored).
struct TileSrc {
    uint64_t a, lo, hi, sc;
    int na;  // bytes from the first row's start to the last valid row's end
    uint32_t va, vlo, vhi, vsc;
    int64_t flo, fhi, fsc;
    uint64_t fa[2];
};

template <int MT, int NT, bool PACKED, bool FAR>
__device__ __forceinline__ TileSrc tile_src(const Args& p, int b, int m0, int tile, int row0) {
    const int lane = threadIdx.x & 63, i = lane & 15, q = lane >> 4;
    TileSrc s;
    if constexpr (FAR) {
        static_assert(MT == 1, "two groups of eight rows");
#pragma unroll
        for (int e = 0; e < 2; ++e) {
            const int m = min(m0 + row0 + 8 * e + (lane >> 3), p.M - 1);
            s.fa[e] = reinterpret_cast<uint64_t>(p.a + (int64_t)b * p.sa_b + (int64_t)m * p.sa_m) + 16 * (lane & 7);
        }
    } else {
        s.a = reinterpret_cast<uint64_t>(p.a + (int64_t)b * p.sa_b + (int64_t)m0 * p.sa_m);
        s.na = (int)(((int64_t)(min(p.M - m0, 16 * MT) - 1) * p.sa_m + p.K) * 2);
        s.va = (uint32_t)(row0 + (lane >> 3)) * (uint32_t)p.sa_m * 2 + 16 * (lane & 7);
    }
    if constexpr (PACKED) {
        const int strip = tile >> 3, t = tile & 7;
        const uint64_t blk =
            reinterpret_cast<uint64_t>(p.lo + (int64_t)b * p.sl_b + (int64_t)strip * (p.K / 64) * kPackBytes);
        s.lo = blk + 1024 * (t >> 1) + 8 * (t & 1);
        s.hi = blk + 1024 * (4 + (t >> 2)) + 4 * (t & 2);
        s.sc = reinterpret_cast<uint64_t>(p.sc + (int64_t)b * p.ss_b + (int64_t)strip * p.groups * kTileN + (t & 4));
        s.vlo = s.vhi = 16 * lane;
        s.vsc = 16 * i;
    } else {
        const uint32_t n = min(16u * tile + (uint32_t)NT * i, (uint32_t)p.N - NT);  // (unsigned: N up to 2^31 - 16)
        const int hrow = 8 * (q & 1) + 4 * (q >> 1);
        s.lo = reinterpret_cast<uint64_t>(p.lo + (int64_t)b * p.sl_b);
        s.hi = reinterpret_cast<uint64_t>(p.hi + (int64_t)b * p.sh_b);
        s.sc = reinterpret_cast<uint64_t>(p.sc + (int64_t)b * p.ss_b);
        if constexpr (FAR) {
            s.flo = (int64_t)(8 * q) * p.N + n;
            s.fhi = (int64_t)hrow * p.N + n;
            s.fsc = 2 * (int64_t)n;
        } else {
            s.vlo = (uint32_t)(8 * q) * p.N + n;
            s.vhi = (uint32_t)hrow * p.N + n;
            s.vsc = 2 * n;
        }
    }
    return s;
}

__device__ __forceinline__ __amdgpu_buffer_rsrc_t tile_rsrc(uint64_t base, int bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(reinterpret_cast<void*>(base), 0, bytes, 0x00020000);
}

template <int NT, bool PACKED, bool FAR>
__device__ __forceinline__ void tile_load_w(const Args& p, const TileSrc& src, int c, TileW<NT, PACKED>& s) {
    constexpr int kAll = 0x7FFFFFFF;
    const uint32_t g = quotient((uint32_t)c, p.group);  // the chunk's scale group
    if constexpr (PACKED) {
        const __amdgpu_buffer_rsrc_t lo = tile_rsrc(src.lo + (uint64_t)c * kPackBytes, kAll),
                                     hi = tile_rsrc(src.hi + (uint64_t)c * kPackBytes, kAll),
                                     sc = tile_rsrc(src.sc + (uint64_t)g * (2 * kTileN), kAll);
        if constexpr (NT == 1) {
            const uint2 x = __builtin_bit_cast(uint2, __builtin_amdgcn_raw_buffer_load_b64(lo, src.vlo, 0, 0));
            s.lo[0] = x.x, s.lo[1] = x.y;
        } else {
#pragma unroll
            for (int k = 0; k < NT / 2; ++k) {
                const u4 x = __builtin_amdgcn_raw_buffer_load_b128(lo, src.vlo + 1024 * k, 0, 0);
#pragma unroll
                for (int d = 0; d < 4; ++d) s.lo[4 * k + d] = x[d];
            }
        }
        if constexpr (NT == 4) {
            const u4 y = __builtin_amdgcn_raw_buffer_load_b128(hi, src.vhi, 0, 0);
#pragma unroll
            for (int d = 0; d < 4; ++d) s.hd[d] = y[d];
        } else {
            const uint2 y = __builtin_bit_cast(uint2, __builtin_amdgcn_raw_buffer_load_b64(hi, src.vhi, 0, 0));
            s.hd[0] = y.x, s.hd[1] = y.y;
        }
        const uint2 z = __builtin_bit_cast(uint2, __builtin_amdgcn_raw_buffer_load_b64(sc, src.vsc, 0, 0));
        s.sc[0] = z.x, s.sc[1] = z.y;
    } else {
        const uint64_t lo = src.lo + (uint64_t)c * 32 * (uint64_t)p.N, hi = src.hi + (uint64_t)c * 16 * (uint64_t)p.N;
        const uint64_t sc = src.sc + (uint64_t)g * 2 * (uint64_t)p.N;
        if constexpr (FAR) {
            static_assert(NT == 4, "far: 64 columns to a workgroup");
            typedef const __attribute__((address_space(1))) uint32_t* Words;
#pragma unroll
            for (int e = 0; e < 8; ++e) s.lo[e] = *reinterpret_cast<Words>(lo + (uint64_t)(src.flo + (int64_t)e * p.N));
#pragma unroll
            for (int e = 0; e < 4; ++e) s.hd[e] = *reinterpret_cast<Words>(hi + (uint64_t)(src.fhi + (int64_t)e * p.N));
#pragma unroll
            for (int d = 0; d < 2; ++d) s.sc[d] = reinterpret_cast<Words>(sc + (uint64_t)src.fsc)[d];  // (4-byte aligned)
        } else if constexpr (NT == 4) {
#pragma unroll
            for (int e = 0; e < 8; ++e)
                s.lo[e] = __builtin_amdgcn_raw_buffer_load_b32(tile_rsrc(lo, kAll), src.vlo, e * p.N, 0);
#pragma unroll
            for (int e = 0; e < 4; ++e)
                s.hd[e] = __builtin_amdgcn_raw_buffer_load_b32(tile_rsrc(hi, kAll), src.vhi, e * p.N, 0);
            const uint2 z = __builtin_bit_cast(uint2, __builtin_amdgcn_raw_buffer_load_b64(tile_rsrc(sc, kAll), src.vsc, 0, 0));
            s.sc[0] = z.x, s.sc[1] = z.y;
        } else {
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const uint2 x = __builtin_bit_cast(
                    uint2, __builtin_amdgcn_raw_buffer_load_b64(tile_rsrc(lo, kAll), src.vlo, e * p.N, 0));
                s.lo[2 * e] = x.x, s.lo[2 * e + 1] = x.y;
            }
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const uint2 x = __builtin_bit_cast(
                    uint2, __builtin_amdgcn_raw_buffer_load_b64(tile_rsrc(hi, kAll), src.vhi, e * p.N, 0));
                s.hd[2 * e] = x.x, s.hd[2 * e + 1] = x.y;
            }
            const u4 z = __builtin_amdgcn_raw_buffer_load_b128(tile_rsrc(sc, kAll), src.vsc, 0, 0);
#pragma unroll
            for (int d = 0; d < 4; ++d) s.sc[d] = z[d];
        }
    }
}

// NA groups of 8 rows of A's chunk (128 bytes per row).  The rows' offsets are lane offsets: those are what a raw buffer's
// bound covers by its definition, and it is the bound that keeps rows past M from being read.  Eight groups go through two
// buffers: eight lane offsets put registers of the loop into scratch memory (planes, four row tiles, K = 4096, N = 16384, M =
// 64: 30.9 us, 26.1 without).
template <int NA, bool FAR>
__device__ __forceinline__ void tile_load_a(const Args& p, const TileSrc& src, int c, u4 (&a)[NA]) {
    if constexpr (FAR) {
        static_assert(NA == 2, "two groups of eight rows");
#pragma unroll
        for (int e = 0; e < NA; ++e)
            a[e] = *reinterpret_cast<const __attribute__((address_space(1))) u4*>(src.fa[e] + (uint64_t)c * 128);
    } else {
        constexpr int kGroup = NA == 8 ? 4 : NA;  // row groups to a buffer
#pragma unroll
        for (int e0 = 0; e0 < NA; e0 += kGroup) {
            const int off = 16 * e0 * (int)p.sa_m, left = src.na - c * 128 - off;
            const __amdgpu_buffer_rsrc_t r = tile_rsrc(src.a + (uint64_t)c * 128 + (uint64_t)off, e0 == 0 ? left : max(left, 0));
#pragma unroll
            for (int e = e0; e < e0 + kGroup; ++e)
                a[e] = __builtin_amdgcn_raw_buffer_load_b128(r, src.va + 16 * (e - e0) * (uint32_t)p.sa_m, 0, 0);
        }
    }
}

// 16-byte piece j (k = 8 j ..) of row r of the chunk's rows of A in LDS: the 16 rows of one operand read (one j) fall in
// 16 different 16-byte bank groups, and so do the writes.
__device__ __forceinline__ int a_slot(int r, int j) { return 8 * r + (j ^ ((r >> 1) & 7)); }

// Column tile t's weight operands (rows 8 q .. and 32 + 8 q .. of the chunk) and scale.  u0, u1: the planes' codes of
// rows 8 q + e and 32 + 8 q + e, NT / 4 words of four columns each.
template <class A, int NT, bool PACKED>
__device__ __forceinline__ void tile_dequant(const TileW<NT, PACKED>& s, const uint32_t (&u0)[2 * NT], const uint32_t (&u1)[2 * NT],
                                             int t, int tsel, u4& w0, u4& w1, float& sv) {
    uint32_t o0[4], o1[4];
    uint32_t sw;
    if constexpr (PACKED) {
        const uint32_t L0 = s.lo[2 * t], L1 = s.lo[2 * t + 1], Hd = NT == 1 ? (tsel & 1 ? s.hd[1] : s.hd[0]) : s.hd[t];
        codes_to_op<A>((L0 & 0x0F0F0F0Fu) | ((Hd & 0x03030303u) << 4), o0[0], o0[1]);         // rows 8 q + 0..3
        codes_to_op<A>((L1 & 0x0F0F0F0Fu) | (Hd & 0x30303030u), o0[2], o0[3]);                // rows 8 q + 4..7
        codes_to_op<A>(((L0 >> 4) & 0x0F0F0F0Fu) | ((Hd & 0x0C0C0C0Cu) << 2), o1[0], o1[1]);  // rows 32 + 8 q ..
        codes_to_op<A>(((L1 >> 4) & 0x0F0F0F0Fu) | ((Hd >> 2) & 0x30303030u), o1[2], o1[3]);
        if constexpr (NT == 4) sw = s.sc[t >> 1] >> (16 * (t & 1));
        else if constexpr (NT == 2) sw = (tsel & 2 ? s.sc[1] : s.sc[0]) >> (16 * t);
        else sw = (tsel & 2 ? s.sc[1] : s.sc[0]) >> (16 * (tsel & 1));
    } else {
        // rows 2 d, 2 d + 1 of column t: the two rows' bytes interleaved, then each beside the constant high byte
        constexpr uint32_t kPair[2] = {0x05010400u, 0x07030602u};  // columns 0, 1 and 2, 3
#pragma unroll
        for (int d = 0; d < 4; ++d) {
            constexpr int C = NT / 4;
            const int r0 = 2 * d * C + (t >> 2), r1 = r0 + C;
            const uint32_t x = __builtin_amdgcn_perm(u0[r1], u0[r0], kPair[(t >> 1) & 1]);
            const uint32_t y = __builtin_amdgcn_perm(u1[r1], u1[r0], kPair[(t >> 1) & 1]);
            o0[d] = __builtin_amdgcn_perm(A::kCodeHi, x, t & 1 ? 0x04030402u : 0x04010400u);
            o1[d] = __builtin_amdgcn_perm(A::kCodeHi, y, t & 1 ? 0x04030402u : 0x04010400u);
        }
        sw = s.sc[t >> 1] >> (16 * (t & 1));
    }
    sv = h2f((uint16_t)sw);
    w0 = u4{o0[0], o0[1], o0[2], o0[3]};
    w1 = u4{o1[0], o1[1], o1[2], o1[3]};
}

// One chunk: per (M tile, column tile) two MFMAs started at the M tile's bias, scaled into acc.  Software-pipelined over
// the column tiles: tile t's MFMAs are issued between the dequantisation of tile t + 1 and the scaling of tile t - 1
// (left to itself the compiler reused one accumulator and waited out each MFMA pair's latency).
template <class A, int MT, int NT, bool PACKED>
__device__ __forceinline__ void tile_work(const TileW<NT, PACKED>& s, const uint8_t* const (&ra)[2], int tsel,
                                          f4 (&acc)[MT][NT]) {
    const int q = (threadIdx.x & 63) >> 4;
    const u4 bias = u4{A::kBias, A::kBias, A::kBias, A::kBias};  // -(2^e + 32)
    f4 corr[MT], tc[2][MT];
    u4 a[MT][2], w[2][2];
    float sv[2];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int h = 0; h < 2; ++h) a[mt][h] = *reinterpret_cast<const u4*>(ra[h] + 2048 * mt);
    uint32_t u0[2 * NT], u1[2 * NT];
    if constexpr (!PACKED) {
        const int sel = 2 * (q >> 1);  // the hi plane's field of rows 8 q ..
        uint32_t hd[2 * NT];           // hi-plane rows 8 (q & 1) + e: the lower half-wavefront's four, then the upper's
#pragma unroll
        for (int e = 0; e < NT; ++e) {
            const auto x = __builtin_amdgcn_permlane32_swap(s.hd[e], s.hd[e], false, false);
            hd[e] = x[0];
            hd[NT + e] = x[1];
        }
#pragma unroll
        for (int e = 0; e < 2 * NT; ++e) {
            const uint32_t L = s.lo[e], H = hd[e] >> sel;
            u0[e] = (L & 0x0F0F0F0Fu) | ((H & 0x03030303u) << 4);
            u1[e] = ((L >> 4) & 0x0F0F0F0Fu) | (H & 0x30303030u);
        }
    }
    tile_dequant<A, NT, PACKED>(s, u0, u1, 0, tsel, w[0][0], w[0][1], sv[0]);
    if constexpr (MT > 1) __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) corr[mt] = A::mma(a[mt][0], bias, f4{0.f, 0.f, 0.f, 0.f});
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) corr[mt] = A::mma(a[mt][1], bias, corr[mt]);
#pragma unroll
    for (int t = 0; t < NT; ++t) {
        const int k = t & 1;
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) tc[k][mt] = A::mma(a[mt][0], w[k][0], corr[mt]);
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) tc[k][mt] = A::mma(a[mt][1], w[k][1], tc[k][mt]);
        float nsv = 0.f;
        if (t + 1 < NT) tile_dequant<A, NT, PACKED>(s, u0, u1, t + 1, tsel, w[k ^ 1][0], w[k ^ 1][1], nsv);
        if (t > 0) {
#pragma unroll
            for (int mt = 0; mt < MT; ++mt) acc[mt][t - 1] = fma4(tc[k ^ 1][mt], sv[k ^ 1], acc[mt][t - 1]);
        }
        sv[k ^ 1] = nsv;
        if constexpr (MT > 1) {
#pragma unroll
            for (int x = 0; x < 2 * MT; ++x) {
                __builtin_amdgcn_sched_group_barrier(8, 1, 0);                // an MFMA,
                __builtin_amdgcn_sched_group_barrier(2, MT == 4 ? 5 : 7, 0);  // then VALU work of the two other tiles
            }
            __builtin_amdgcn_sched_barrier(0);
        }
    }
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) acc[mt][NT - 1] = fma4(tc[(NT - 1) & 1][mt], sv[(NT - 1) & 1], acc[mt][NT - 1]);
}

// The sum of the W partials of one element, at x, by the quarters of the parts that the workgroup holds (4 / ks).
__device__ __forceinline__ float tile_sum(const float* x, int stride, int W, int ks) {
    auto sum = [&](int w0, int w1) __attribute__((always_inline)) {
        float y = 0.f;
        for (int w = w0; w < min(w1, W); ++w) y += x[w * stride];
        return y;
    };
    if (ks == 4) return sum(0, W);
    const int n = ks == 2 ? W >> 1 : (W + 3) >> 2;  // parts per quarter
    const float s = sum(0, n) + sum(n, 2 * n);
    return ks == 2 ? s : s + (sum(2 * n, 3 * n) + sum(3 * n, 4 * n));
}

// The same of four rows, whole f4 at x (single rows of them meet in a quarter of the banks), Q = 4 / ks quarters at a time.
template <int Q>
__device__ __forceinline__ f4 tile_sum4(const f4* x, int stride, int W) {
    const int n = (W + Q - 1) / Q;  // parts per quarter
    f4 s[Q];
#pragma unroll
    for (int q = 0; q < Q; ++q) s[q] = f4{0.f, 0.f, 0.f, 0.f};
    for (int w = 0; w < n; ++w)
#pragma unroll
        for (int q = 0; q < Q; ++q)
            if (q == 0 || q * n + w < W) s[q] += x[(q * n + w) * stride];
    if constexpr (Q == 4) return (s[0] + s[1]) + (s[2] + s[3]);
    else if constexpr (Q == 2) return s[0] + s[1];
    else return s[0];
}

// LDS of a wavefront: its rows of A, then its partial tile.
constexpr int tile_lds(int MT, int NA, int NT) { return 1024 * (MT * NT > NA ? MT * NT : NA); }

// NA: groups of 8 rows of A a K part stages (1: M <= 8).  D chunks of weights and DA of A are in flight.  CW: wavefronts
// side by side in a K part, 16 NT columns each, sharing its rows of A; with two, each loads half of them, the rows are
// double-buffered and the workgroup meets at one barrier per chunk.
template <class A, int MT, int NA, int NT, int CW, int D, int DA, int MAXW, bool PACKED, bool FAR>
__global__ __launch_bounds__(64 * MAXW) void w6a16_tile_kernel(const Args p) {
    static_assert(PACKED ? NT <= 4 : NT == 4 || NT == 8, "packed: up to four column tiles; planes: four or eight");
    static_assert(!FAR || (MT == 1 && NT == 4 && CW == 1), "far: 16 rows, 64 columns to a workgroup");
    static_assert(D % DA == 0, "stage rings");
    static_assert(CW == 1 || (CW == 2 && D == 2 && DA == 1 && NA % 2 == 0), "one or two column wavefronts");
    constexpr int kA = 1024 * NA;  // bytes of a chunk's rows of A (CW = 2: two buffers a K part)
    constexpr int NW = NA / CW;    // row groups this wavefront loads
    extern __shared__ __attribute__((aligned(16))) uint8_t lds[];  // tile_lds bytes a wavefront
    __shared__ uint32_t completed;
    const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int W = (blockDim.x >> 6) / CW, ks = gridDim.z, split = blockIdx.z;  // W: K parts in the workgroup
    const int cw = CW == 1 ? 0 : wv & 1, kp = CW == 1 ? wv : wv >> 1;
    const TilePos pos = tile_pos(p.grid, blockIdx.x);
    const int wtile = (int)pos.column * NT * CW, tile = wtile + cw * NT;
    const int mg = (int)pos.mg, m0 = mg * 16 * MT, b = blockIdx.y;
    if (wtile >= p.N / 16) return;  // uniform over the workgroup
    // this wavefront's chunks g, g + parts, ..
    const int g = split * W + kp, nchunks = p.K / 64;
    const int n = p.per_part - (g + p.parts * (p.per_part - 1) >= nchunks ? 1 : 0);  // >= 1: parts <= chunks
    // The chunk's rows of A lie at a_slot(row, piece) of the wavefront's buffer; the swizzle repeats every 16 rows, so
    // two addresses serve all writes (row groups this wavefront loads, even and odd) and two all reads (k halves of row i).
    uint8_t* const abuf = lds + kp * CW * kA;
    const int odd = 8 * (cw & NW);  // a wavefront that starts at an odd row group (NW odd, its second half)
    uint8_t* const wa[2] = {abuf + 16 * a_slot((lane >> 3) + odd, lane & 7) - 16 * 8 * odd,
                            abuf + 16 * a_slot(8 - odd + (lane >> 3), lane & 7) - 16 * 8 * (8 - odd)};
    const int ri = NA == 1 ? lane & 7 : lane & 15;
    const uint8_t* const ra[2] = {abuf + 16 * a_slot(ri, lane >> 4), abuf + 16 * a_slot(ri, 4 + (lane >> 4))};

    const TileSrc src = tile_src<MT, NT, PACKED, FAR>(p, b, m0, tile, 8 * NW * cw);
    f4 acc[MT][NT];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int t = 0; t < NT; ++t) acc[mt][t] = f4{0.f, 0.f, 0.f, 0.f};
    TileW<NT, PACKED> w[D];
    u4 a[DA][NW];
    // past the end: the last chunk again (a cache hit), so that every load is unconditional
    auto chunk = [&](int j) __attribute__((always_inline)) { return g + p.parts * min(j, n - 1); };
    auto write = [&](const u4 (&x)[NW], int buf) __attribute__((always_inline)) {
#pragma unroll
        for (int e = 0; e < NW; ++e) {
            *reinterpret_cast<u4*>(wa[e & 1] + 1024 * (e + NW * cw) + buf * kA) = x[e];
        }
    };
    auto work = [&](const TileW<NT, PACKED>& x, int buf) __attribute__((always_inline)) {
        const uint8_t* const rb[2] = {ra[0] + buf * kA, ra[1] + buf * kA};
        tile_work<A, MT, NT, PACKED>(x, rb, tile, acc);
    };
#pragma unroll
    for (int j = 0; j < D; ++j) {
        tile_load_w<NT, PACKED, FAR>(p, src, chunk(j), w[j]);
        if (j < DA) tile_load_a<NW, FAR>(p, src, chunk(j), a[j]);
    }
    __builtin_amdgcn_sched_barrier(0);
    int base = 0;
    if constexpr (CW == 1) {
        auto stage = [&](const u4 (&x)[NW]) __attribute__((always_inline)) {
            wave_lds_sync();  // the previous chunk's reads are issued before these writes
            write(x, 0);
            wave_lds_sync();
        };
        for (; base + D < n; base += D)
#pragma unroll
            for (int j = 0; j < D; ++j) {
                stage(a[j % DA]);
                tile_load_a<NW, FAR>(p, src, chunk(base + j + DA), a[j % DA]);
                __builtin_amdgcn_sched_barrier(0);
                work(w[j], 0);
                tile_load_w<NT, PACKED, FAR>(p, src, chunk(base + D + j), w[j]);
                __builtin_amdgcn_sched_barrier(0);
            }
#pragma unroll
        for (int j = 0; j < D; ++j)
            if (base + j < n) {
                stage(a[j % DA]);
                if (j + DA < D) tile_load_a<NW, FAR>(p, src, chunk(base + j + DA), a[j % DA]);
                __builtin_amdgcn_sched_barrier(0);
                work(w[j], 0);
            }
    } else {
        // chunk j's rows lie in buffer j & 1; the next chunk's are written beside its work and met at the barrier
        write(a[0], 0);
        tile_load_a<NW, FAR>(p, src, chunk(1), a[0]);
        __syncthreads();
        const int steps = p.per_part;  // uniform over the workgroup; a part with a chunk less skips its last one
        for (; base + D < steps; base += D)
#pragma unroll
            for (int j = 0; j < D; ++j) {
                write(a[0], (j + 1) & 1);
                tile_load_a<NW, FAR>(p, src, chunk(base + j + 2), a[0]);
                __builtin_amdgcn_sched_barrier(0);
                work(w[j], j & 1);
                tile_load_w<NT, PACKED, FAR>(p, src, chunk(base + D + j), w[j]);
                __builtin_amdgcn_sched_barrier(0);
                __syncthreads();
            }
#pragma unroll
        for (int j = 0; j < D; ++j) {
            if (j + 1 < D) write(a[0], (j + 1) & 1);
            if (base + j < n) work(w[j], j & 1);
            __syncthreads();
        }
    }

    __syncthreads();  // the staging buffers are dead: the partial tiles reuse the LDS
    const int tid = threadIdx.x;
    f4* const part = reinterpret_cast<f4*>(lds) + tid / 64 * MT * NT * 64 + tid % 64;  // [K part][column wavefront]
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int t = 0; t < NT; ++t) part[(mt * NT + t) * 64] = acc[mt][t];
    __syncthreads();
    // A thread takes one column of every step-th row, or, with more than one row to a thread, of every step-th four rows.
    constexpr int NC = 16 * NT * CW;
    const int rows = min(16 * MT, p.M - m0), n0 = 16 * wtile;
    const int col = tid % NC, step = blockDim.x / NC;
    auto each_sum = [&](auto sink) __attribute__((always_inline)) {
        const int c = col % (16 * NT), t = PACKED ? c >> 4 : c % NT, i = PACKED ? c & 15 : c / NT;
        const f4* const sums = reinterpret_cast<const f4*>(lds) + (col / (16 * NT) * MT * NT + t) * 64 + i;
        constexpr int kPart = CW * MT * NT * 64;
        auto four = [&](int r4) __attribute__((always_inline)) { return sums + (r4 >> 2) * NT * 64 + 16 * (r4 & 3); };
        auto fours = [&](auto quarters) __attribute__((always_inline)) {
            for (int r4 = tid / NC; 4 * r4 < rows; r4 += step) {
                const f4 y = tile_sum4<decltype(quarters)::value>(four(r4), kPart, W);
#pragma unroll
                for (int v = 0; v < 4; ++v)
                    if (4 * r4 + v < rows) sink(4 * r4 + v, y[v]);
            }
        };
        if (rows < 2 * step) {
            for (int r = tid / NC; r < rows; r += step)
                sink(r, tile_sum(reinterpret_cast<const float*>(four(r >> 2)) + (r & 3), 4 * kPart, W, ks));
        } else if (ks == 1) {
            fours(std::integral_constant<int, 4>{});
        } else if (ks == 2) {
            fours(std::integral_constant<int, 2>{});
        } else {
            fours(std::integral_constant<int, 1>{});
        }
    };
    auto store = [&](int r, int c, float x) __attribute__((always_inline)) {
        const int64_t o = (int64_t)b * p.so_b + (int64_t)(m0 + r) * p.so_m + n0 + c;
        if (p.out_dtype == W6A16_OUT_F16) put_out<true>(p, o, x);
        else put_out<false>(p, o, x);
    };
    if (ks == 1) {
        if (col < p.N - n0) each_sum([&](int r, float x) __attribute__((always_inline)) { store(r, col, x); });
        return;
    }
    // K split over ks workgroups.  The partial tile goes out in agent-scope atomic stores (written through to where every
    // XCD sees them), each wavefront waits until its own have completed, and the barrier puts all of them before the
    // arrival count; the workgroup that counts in last reads the partials by agent-scope atomic loads, past the caches.
    // No release or acquire fence at agent scope: a fence writes back or invalidates the XCD's whole L2, and nothing here
    // is cached there (with one fence per workgroup a call of 256 workgroups took 1 us longer, one of 512 4 us).
    // The language alone does not order this: relaxed accesses on either side of a relaxed count promise nothing.  What
    // does is this target: a store counts in vmcnt until it is done, at the place that agent-scope accesses of every XCD go
    // to, so s_waitcnt 0 and the barrier put the stores before the count, and the loads are issued after it by the
    // workgroup's second barrier.  A target that counts stores apart, or keeps agent-scope stores in a cache, would need
    // release and acquire at agent scope around the count.
#if defined(__HIP_DEVICE_COMPILE__) && !defined(__gfx950__)
#error "the hand-off of the partial tiles is ordered by gfx950's store counter and write-through stores"
#endif
    constexpr int kTileFloats = 16 * MT * NC;
    const int64_t id = ((int64_t)b * p.grid.m_groups + mg) * ((p.N / 16 + NT * CW - 1) / (NT * CW)) + wtile / (NT * CW);
    float* const part0 = p.part + id * ks * kTileFloats;
    each_sum([&](int r, float x) __attribute__((always_inline)) { coherent_store(part0 + split * kTileFloats + r * NC + col, x); });
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
    __builtin_amdgcn_s_waitcnt(0);  // this wavefront's partial stores have completed
    __syncthreads();
    if (threadIdx.x == 0) {
        const bool done =
            __hip_atomic_fetch_add(p.cnt + id, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == (uint32_t)ks - 1;
        if (done) __hip_atomic_store(p.cnt + id, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        completed = done ? 1u : 0u;
    }
    __syncthreads();
    if (!completed) return;
    for (int e = 2 * tid; e < rows * NC; e += 2 * blockDim.x) {
        float2 x[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) x[k] = coherent_load2(part0 + min(k, ks - 1) * kTileFloats + e);
        float2 sum = float2{x[0].x + x[1].x, x[0].y + x[1].y};
        if (ks == 4) sum = float2{sum.x + (x[2].x + x[3].x), sum.y + (x[2].y + x[3].y)};
        const int c = e % NC;
        if (c >= p.N - n0) continue;  // (both columns of a pair, or neither)
        store(e / NC, c, sum.x);
        store(e / NC, c + 1, sum.y);
    }
}

// Eight codes (one per byte of u) of eight columns with scales sc: s q, exact in fp32 (11 x 6 bit product).
__device__ __forceinline__ void dequant8(const uint2 u, const u4 sc, float (&v)[8]) {
#pragma unroll
    for (int e = 0; e < 8; ++e) {
        const uint32_t word = e < 4 ? u.x : u.y;
        v[e] = h2f((uint16_t)(sc[e >> 1] >> (16 * (e & 1)))) * ((float)((word >> (8 * (e & 3))) & 0xFF) - 32.f);
    }
}

template <typename OutT>
__device__ __forceinline__ void store_row8(OutT* dst, const float (&v)[8], bool vec) {
    if (vec) {
        store8(dst, v);
    } else {
#pragma unroll
        for (int e = 0; e < 8; ++e) dst[e] = (OutT)v[e];
    }
}

// ---------------------------------------------------------------------------------------------------------------
// Wide kernel: 145 to 256 rows over so many columns that 64 x 128 tiles go at least twice around the CUs (wide_call).  A
// workgroup of four wavefronts covers 128 columns for 64 rows, wavefront cp column tiles 2 cp and 2 cp + 1 for all of them,
// over all of K: each dequantised weight operand serves four row tiles, and each A operand two column tiles.  The tile
// kernel waits on its own chains there (64 accumulators a lane against 32, a scaling per chunk, a bias product per chunk
// and row tile): K = 4096, N = 16384, M = 256, us, planes / packed, 63.0 / 59.2 against 60.4 / 49.7 here; K = 1024, N =
// 65536, M = 256 91.1 / 79.0 against 76.9 / 66.8.
//   * A's chunk ([64 rows][64 k]) is staged in LDS, double-buffered, one workgroup barrier a step; piece j of row r lies at
//     a_slot.  Packed weights go straight to registers, four steps ahead; planes are staged with A (48 rows x 128 columns)
//     and read back transposed (ds_read_b64_tr_b8).
//   * Chains: the products of CG chunks (two where the quantisation group holds two) accumulate in one MFMA chain, which
//     starts at the bias -(2^e + 32) sum_k A[m][k] (row sums of a pass before it), and are scaled once.
constexpr int kWideMT = 4, kWideRows = 16 * kWideMT;
constexpr int kPitch = 136;                // LDS row pitch of the planes: the 8 rows of one transposing read differ in bank
constexpr int kScaleOff = 48 * kPitch;     // the chunk's 128 scales follow 32 lo and 16 hi rows
constexpr int kWideA = kWideRows * 128;    // bytes of A in a stage; the chain's row sums follow, then the planes

template <bool PACKED>
constexpr int wide_stage() { return kWideA + kWideRows * 4 + (PACKED ? 0 : kScaleOff + 2 * kTileN); }

// (1, 1) as an activation pair held in a register (an empty asm keeps the compiler from folding the pair into an
// inline constant, which the packed dot product would read differently).
template <class A>
__device__ __forceinline__ uint32_t ones_x2() {
    uint32_t bits = A::kOnes;
    asm("" : "+v"(bits));
    return bits;
}

template <class A>
__device__ __forceinline__ float sum8(const u4 v, uint32_t one) {
    float x = 0.f;
#pragma unroll
    for (int d = 0; d < 4; ++d) {
        // the element is copied out first: bit-casting a vector element in place (v[d]) compiled to a read of
        // element 0 for every d
        const uint32_t word = v[d];
        x = A::dot2(word, one, x);
    }
    return x;
}

template <int CTRL>
__device__ __forceinline__ float dpp_add(float x) {  // x + x of the lane DPP control CTRL selects (all lanes active)
    return x + __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), CTRL, 0xF, 0xF, false));
}

// Row sums of A per chain of chain_k k: rsum[b][chain][m] = -(2^e + 32) sum A[b][m][chain's k], zero for rows M <= m <
// mpad.  One wavefront per (row, 512-element segment of K; 8 elements per lane, coalesced); the lanes of a chain add
// their sums with DPP in a fixed order.
template <class A>
__global__ __launch_bounds__(256) void w6a16_rowsum_kernel(const Args p) {
    const int lane = threadIdx.x & 63;
    const int m = blockIdx.x * 4 + (threadIdx.x >> 6), k = blockIdx.y * 512 + 8 * lane, b = blockIdx.z;
    if (m >= p.mpad) return;  // uniform over the wavefront
    const int lanes_per_chain = p.chain_k / 8;  // 8 or 16
    const uint16_t* const row = p.a + (int64_t)b * p.sa_b + (int64_t)min(m, p.M - 1) * p.sa_m;
    // K is a multiple of the chain: a chain's lanes are all inside K or all past it
    float x = (m < p.M && k < p.K) ? sum8<A>(*reinterpret_cast<const u4*>(row + k), ones_x2<A>()) : 0.f;
    x = dpp_add<0xB1>(x);   // lanes ^ 1
    x = dpp_add<0x4E>(x);   // lanes ^ 2: each lane holds its quad's sum
    x = dpp_add<0x141>(x);  // half-row mirror: lane 7 - l of the 8-lane group, in the other quad
    if (lanes_per_chain == 16) x = dpp_add<0x140>(x);  // row mirror: lane 15 - l, in the other half
    if ((lane & (lanes_per_chain - 1)) == 0 && k < p.K)
        p.rsum[((int64_t)b * p.nchains + k / p.chain_k) * p.mpad + m] = -A::kOffset * x;
}

// What one thread loads per step into the LDS stage: two pieces of A, four row sums (threads 0..15) and (planes) 16 bytes
// of a lo-plane row, 16 bytes of a hi-plane row (threads 0..127) or two scales (threads 128..191).
struct WideLds {
    u4 a[2], rs, pl[2];
    uint32_t sc;
};

// Buffer bases and sizes (wave-uniform) and per-lane offsets of the loads, fixed for the call; the chunk goes into the
// instructions' scalar offset.  Every range is below 2 GB (wide_call; of A the workgroup's 64 rows, which at row strides of
// 2^24 elements and more, FAR, have 64-bit addresses instead).
struct WideSrc {
    uint64_t a, rs, lo, hi, sc, fa[2];
    int64_t na, nrs, nlo, nhi, nsc;
    uint32_t va[2], vrs, vlo, vhi, vsc;
};

template <bool PACKED, bool FAR>
__device__ __forceinline__ WideSrc wide_src(const Args& p, int b, int m0, int strip) {
    const int t = threadIdx.x, lane = t & 63, i = lane & 15, cp = t >> 6, n0 = strip * kTileN;
    WideSrc x;
    const uint16_t* const a = p.a + (int64_t)b * p.sa_b + (int64_t)m0 * p.sa_m;
    x.a = reinterpret_cast<uint64_t>(a);
    const int last = min(p.M - m0, kWideRows) - 1;  // of the workgroup's rows; those past it take it again
    x.na = ((int64_t)last * p.sa_m + p.K) * 2;
#pragma unroll
    for (int e = 0; e < 2; ++e) {
        const int piece = t + 256 * e;
        const int64_t off = (min(piece >> 3, last) * p.sa_m + 8 * (piece & 7)) * 2;
        if constexpr (FAR) x.fa[e] = x.a + (uint64_t)off;
        else x.va[e] = (uint32_t)off;
    }
    x.rs = reinterpret_cast<uint64_t>(p.rsum + (int64_t)b * p.nchains * p.mpad);
    x.nrs = (int64_t)p.nchains * p.mpad * 4;
    x.vrs = (m0 + 4 * min(t, kWideRows / 4 - 1)) * 4;
    if constexpr (PACKED) {
        const int nchunks = p.K / 64;
        x.lo = reinterpret_cast<uint64_t>(p.lo + (int64_t)b * p.sl_b + (int64_t)strip * nchunks * kPackBytes);
        x.nlo = (int64_t)nchunks * kPackBytes;
        x.vlo = 16 * lane + 1024 * cp;
        x.vhi = 4096 + 1024 * (cp >> 1) + 8 * (cp & 1) + 16 * lane;
        x.sc = reinterpret_cast<uint64_t>(p.sc + (int64_t)b * p.ss_b + (int64_t)strip * p.groups * kTileN);
        x.nsc = (int64_t)p.groups * kTileN * 2;
        x.vsc = (8 * i + 2 * cp) * 2;
    } else {
        const int row = t >> 3, n = min(n0 + 16 * (t & 7), p.N - 16);  // lo row 0..31; hi row (row & 15)
        x.lo = reinterpret_cast<uint64_t>(p.lo + (int64_t)b * p.sl_b);
        x.nlo = (int64_t)(p.K / 2) * p.N;
        x.vlo = row * p.N + n;
        x.hi = reinterpret_cast<uint64_t>(p.hi + (int64_t)b * p.sh_b);
        x.nhi = (int64_t)(p.K / 4) * p.N;
        x.vhi = (row & 15) * p.N + n;
        x.sc = reinterpret_cast<uint64_t>(p.sc + (int64_t)b * p.ss_b);
        x.nsc = (int64_t)p.groups * p.N * 2;
        x.vsc = min(n0 + 2 * (t & 63), p.N - 2) * 2;
    }
    return x;
}

template <int CG, bool PACKED, bool FAR>
__device__ __forceinline__ void wide_load_lds(const Args& p, const WideSrc& src, int c, WideLds& x) {
#pragma unroll
    for (int e = 0; e < 2; ++e) {
        if constexpr (FAR)
            x.a[e] = *reinterpret_cast<const __attribute__((address_space(1))) u4*>(src.fa[e] + (uint64_t)c * 128);
        else
            x.a[e] = __builtin_amdgcn_raw_buffer_load_b128(rsrc(src.a, src.na), src.va[e], soff(c * 128), 0);
    }
    x.rs = __builtin_amdgcn_raw_buffer_load_b128(rsrc(src.rs, src.nrs), src.vrs, soff((c / CG) * p.mpad * 4), 0);
    if constexpr (!PACKED) {
        x.pl[0] = __builtin_amdgcn_raw_buffer_load_b128(rsrc(src.lo, src.nlo), src.vlo, soff(c * 32 * p.N), 0);
        x.pl[1] = __builtin_amdgcn_raw_buffer_load_b128(rsrc(src.hi, src.nhi), src.vhi, soff(c * 16 * p.N), 0);
        x.sc = __builtin_amdgcn_raw_buffer_load_b32(rsrc(src.sc, src.nsc), src.vsc,
                                                    soff((int)quotient((uint32_t)c, p.group) * p.N * 2), 0);
    }
}

template <bool PACKED>
__device__ __forceinline__ void wide_store_lds(const WideLds& x, uint8_t* st) {
    const int t = threadIdx.x;
#pragma unroll
    for (int e = 0; e < 2; ++e) {
        const int piece = t + 256 * e;
        *reinterpret_cast<u4*>(st + 16 * a_slot(piece >> 3, piece & 7)) = x.a[e];
    }
    if (t < kWideRows / 4) *reinterpret_cast<u4*>(st + kWideA + 16 * t) = x.rs;
    if constexpr (!PACKED) {
        uint8_t* const pl = st + kWideA + kWideRows * 4;
        uint8_t* dst = pl + (t >> 3) * kPitch + 16 * (t & 7);
        *reinterpret_cast<uint2*>(dst) = uint2{x.pl[0][0], x.pl[0][1]};
        *reinterpret_cast<uint2*>(dst + 8) = uint2{x.pl[0][2], x.pl[0][3]};
        if (t < 128) {
            dst += 32 * kPitch;
            *reinterpret_cast<uint2*>(dst) = uint2{x.pl[1][0], x.pl[1][1]};
            *reinterpret_cast<uint2*>(dst + 8) = uint2{x.pl[1][2], x.pl[1][3]};
        } else if (t < 192) {
            *reinterpret_cast<uint32_t*>(pl + kScaleOff + 4 * (t & 63)) = x.sc;
        }
    }
}

// The packed weights of one chunk in one lane's registers: the lo dwords of the wavefront's two column tiles, their hi
// dwords and their scales of column i.
struct WideW {
    u4 lo;
    uint2 hd;
    uint32_t sc;
};

__device__ __forceinline__ void wide_load_w(const Args& p, const WideSrc& src, int c, WideW& w) {
    const __amdgpu_buffer_rsrc_t lo = rsrc(src.lo, src.nlo);
    const int off = soff(c * kPackBytes);
    w.lo = __builtin_amdgcn_raw_buffer_load_b128(lo, src.vlo, off, 0);
    w.hd = __builtin_bit_cast(uint2, __builtin_amdgcn_raw_buffer_load_b64(lo, src.vhi, off, 0));
    w.sc = __builtin_amdgcn_raw_buffer_load_b32(rsrc(src.sc, src.nsc), src.vsc,
                                                soff((int)quotient((uint32_t)c, p.group) * kTileN * 2), 0);
}

// The wavefront's two column tiles of one chunk as B operands w0 (rows 0..31 of the chunk) and w1 (rows 32..63), and their
// scales.
template <class A, bool PACKED>
__device__ __forceinline__ void wide_dequant(const uint8_t* st, const WideW& w, u4 (&w0)[2], u4 (&w1)[2], float (&sv)[2]) {
    const int lane = threadIdx.x & 63, cp = threadIdx.x >> 6, i = lane & 15, q = lane >> 4;
    if constexpr (PACKED) {
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int tt = 0; tt < 2; ++tt) {
            const uint32_t L0 = w.lo[2 * tt], L1 = w.lo[2 * tt + 1], Hd = tt ? w.hd.y : w.hd.x;
            uint32_t o0[4], o1[4];
            codes_to_op<A>((L0 & 0x0F0F0F0Fu) | ((Hd & 0x03030303u) << 4), o0[0], o0[1]);         // rows 8 q + 0..3
            codes_to_op<A>((L1 & 0x0F0F0F0Fu) | (Hd & 0x30303030u), o0[2], o0[3]);                // rows 8 q + 4..7
            codes_to_op<A>(((L0 >> 4) & 0x0F0F0F0Fu) | ((Hd & 0x0C0C0C0Cu) << 2), o1[0], o1[1]);  // rows 32 + 8 q ..
            codes_to_op<A>(((L1 >> 4) & 0x0F0F0F0Fu) | ((Hd >> 2) & 0x30303030u), o1[2], o1[3]);
            w0[tt] = u4{o0[0], o0[1], o0[2], o0[3]};
            w1[tt] = u4{o1[0], o1[1], o1[2], o1[3]};
            sv[tt] = h2f((uint16_t)(w.sc >> (16 * tt)));
        }
    } else {
        const uint8_t* const pl = st + kWideA + kWideRows * 4;
        const int sel = 2 * (q >> 1), off = (i >> 1) * kPitch + 8 * (i & 1);
        v2i lo_t[2], hi_t[2];
        uint16_t sh[2];
#pragma unroll
        for (int tt = 0; tt < 2; ++tt) {
            const int t = 2 * cp + tt;
            lo_t[tt] = __builtin_amdgcn_ds_read_tr8_b64_v2i32((lds_v2i*)(pl + (8 * q) * kPitch + off + 16 * t));
            hi_t[tt] = __builtin_amdgcn_ds_read_tr8_b64_v2i32((lds_v2i*)(pl + (32 + 8 * (q & 1)) * kPitch + off + 16 * t));
            sh[tt] = *reinterpret_cast<const uint16_t*>(pl + kScaleOff + 2 * (16 * t + i));
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int tt = 0; tt < 2; ++tt) {
            uint32_t o0[4], o1[4];
#pragma unroll
            for (int d = 0; d < 2; ++d) {
                const uint32_t L = (uint32_t)lo_t[tt][d], Hs = (uint32_t)hi_t[tt][d] >> sel;
                codes_to_op<A>((L & 0x0F0F0F0Fu) | ((Hs & 0x03030303u) << 4), o0[2 * d], o0[2 * d + 1]);  // rows 8 q + e
                codes_to_op<A>(((L >> 4) & 0x0F0F0F0Fu) | (Hs & 0x30303030u), o1[2 * d], o1[2 * d + 1]);  // 32 + 8 q + e
            }
            w0[tt] = u4{o0[0], o0[1], o0[2], o0[3]};
            w1[tt] = u4{o1[0], o1[1], o1[2], o1[3]};
            sv[tt] = h2f(sh[tt]);
        }
    }
}

// One chunk: two MFMAs per (row tile, column tile) into the chain accumulators tc; FIRST starts the chain at the row
// sums' bias, LAST scales it into acc.  The LDS reads are issued ahead of the dequantisation that hides them (left to
// itself the compiler reused a few operand registers and waited on the LDS once per row tile).
template <class A, bool PACKED, bool FIRST, bool LAST>
__device__ __forceinline__ void wide_compute(const uint8_t* st, const WideW& w, f4 (&tc)[kWideMT][2], f4 (&acc)[kWideMT][2]) {
    const int lane = threadIdx.x & 63, i = lane & 15, q = lane >> 4;
    const float* const rsum = reinterpret_cast<const float*>(st + kWideA);
    u4 a0[kWideMT], a1[kWideMT], w0[2], w1[2];
    f4 nc[kWideMT];
    float sv[2];
#pragma unroll
    for (int mt = 0; mt < kWideMT; ++mt) {
        a0[mt] = *reinterpret_cast<const u4*>(st + 16 * a_slot(16 * mt + i, q));
        a1[mt] = *reinterpret_cast<const u4*>(st + 16 * a_slot(16 * mt + i, 4 + q));
        if constexpr (FIRST) nc[mt] = *reinterpret_cast<const f4*>(rsum + 16 * mt + 4 * q);  // rows 16 mt + 4 q + v
    }
    wide_dequant<A, PACKED>(st, w, w0, w1, sv);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int mt = 0; mt < kWideMT; ++mt)
#pragma unroll
        for (int tt = 0; tt < 2; ++tt) {
            const f4 c = A::mma(a0[mt], w0[tt], FIRST ? nc[mt] : tc[mt][tt]);
            tc[mt][tt] = A::mma(a1[mt], w1[tt], c);
        }
    if constexpr (LAST) {
#pragma unroll
        for (int mt = 0; mt < kWideMT; ++mt)
#pragma unroll
            for (int tt = 0; tt < 2; ++tt) acc[mt][tt] = fma4(tc[mt][tt], sv[tt], acc[mt][tt]);
    }
}

// lane (i, q) of wavefront cp holds C[m0 + 16 mt + 4 q + v][n0 + 16 (2 cp + tt) + i]
template <bool F16>
__device__ __forceinline__ void wide_store(const Args& p, int b, int m0, int n0, const f4 (&acc)[kWideMT][2]) {
    const int lane = threadIdx.x & 63, cp = threadIdx.x >> 6, i = lane & 15, q = lane >> 4;
#pragma unroll
    for (int mt = 0; mt < kWideMT; ++mt)
#pragma unroll
        for (int tt = 0; tt < 2; ++tt) {
            const int n = n0 + 16 * (2 * cp + tt) + i;
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const int m = m0 + 16 * mt + 4 * q + v;
                if (n >= p.N || m >= p.M) continue;
                put_out<F16>(p, (int64_t)b * p.so_b + (int64_t)m * p.so_m + n, acc[mt][tt][v]);
            }
        }
}

template <class A, int CG, bool PACKED, bool FAR>
__global__ __launch_bounds__(256, 2) void w6a16_wide_kernel(const Args p) {
    constexpr int kStage = wide_stage<PACKED>(), D = 4;  // loads D steps ahead
    static_assert(D % CG == 0 && D % 2 == 0, "a group of D steps holds whole chains and buffer pairs");
    __shared__ __attribute__((aligned(16))) uint8_t lds[2 * kStage];
    const TilePos pos = tile_pos(p.grid, blockIdx.x);
    const int strip = (int)pos.column, n0 = strip * kTileN, m0 = (int)pos.mg * kWideRows, b = blockIdx.z;
    if (strip >= p.n_strips) return;  // uniform over the workgroup
    const int steps = p.K / 64;
    const WideSrc src = wide_src<PACKED, FAR>(p, b, m0, strip);
    f4 acc[kWideMT][2], tc[kWideMT][2];
#pragma unroll
    for (int mt = 0; mt < kWideMT; ++mt) acc[mt][0] = acc[mt][1] = f4{0.f, 0.f, 0.f, 0.f};
    // The LDS stage of step s is written in step s - 1 (after its reads of the other buffer have passed that step's
    // barrier) from a ring of D register stages.  Loads past the last chunk take it again (a cache hit), so every load is
    // unconditional; whole groups of D steps run unconditionally with a scheduling barrier after each step's loads, and
    // the remainder (already loaded, whole chains) follows.
    WideLds ls[D];
    WideW ws[D];
    auto chunk = [&](int s) __attribute__((always_inline)) { return min(s, steps - 1); };
#pragma unroll
    for (int j = 0; j < D; ++j) wide_load_lds<CG, PACKED, FAR>(p, src, chunk(j), ls[j]);
    if constexpr (PACKED) {
#pragma unroll
        for (int j = 0; j < D; ++j) wide_load_w(p, src, chunk(j), ws[j]);
    }
    wide_store_lds<PACKED>(ls[0], lds);
    wide_load_lds<CG, PACKED, FAR>(p, src, chunk(D), ls[0]);
    __builtin_amdgcn_sched_barrier(0);
    __syncthreads();
    auto step = [&](int base, auto J) __attribute__((always_inline)) {
        constexpr int j = decltype(J)::value;  // every register index is a constant (else the stages go to scratch memory)
        // (always so here; as a branch it keeps the step apart from its neighbours' loads: without it the planes' form had
        // 364 registers)
        if (base + j < steps)
            wide_compute<A, PACKED, j % CG == 0, j % CG == CG - 1>(lds + (j & 1) * kStage, ws[j], tc, acc);
        if constexpr (PACKED) wide_load_w(p, src, chunk(base + j + D), ws[j]);
        wide_store_lds<PACKED>(ls[(j + 1) % D], lds + ((j + 1) & 1) * kStage);
        wide_load_lds<CG, PACKED, FAR>(p, src, chunk(base + j + 1 + D), ls[(j + 1) % D]);
        __builtin_amdgcn_sched_barrier(0);
        __syncthreads();
    };
    const int full = steps / D * D;
    for (int base = 0; base < full; base += D) unroll<D>([&](auto J) __attribute__((always_inline)) { step(base, J); });
    unroll<D - 1>([&](auto J) __attribute__((always_inline)) {
        if (full + decltype(J)::value < steps) step(full, J);
    });
    if (p.out_dtype == W6A16_OUT_F16) wide_store<true>(p, b, m0, n0, acc);
    else wide_store<false>(p, b, m0, n0, acc);
}

// Dequantise the packed layout: one wavefront per (b, strip, chunk).  HBM-bound (0.75 byte read and 2 written per weight
// for bf16) once the stores are whole lines: the block's codes, one column's rows per lane, are turned in LDS -- by
// ds_read_b64_tr_b8 from [column][row] to eight columns of a row, then into row order -- so that 16 lanes store 256
// bytes of a row.  K = 4096, N = 16384, bf16, weights cycled: 49.4 us with 2-byte stores of 16 columns -> 34.9
// (185 MB).
constexpr int kDqCol = 72, kDqRow = 136;  // byte pitches of the two turns: 64 rows or 128 columns, and 8
constexpr int kDqWave = kTileN * kDqCol + 2 * kTileN;

template <typename OutT>
__global__ __launch_bounds__(256) void w6a16_dequant_packed_kernel(const uint8_t* pk, const uint16_t* psc, OutT* w,
                                                                   int32_t K, int32_t N, int32_t group_k,
                                                                   int32_t strips, int64_t sw_b, bool vec) {
    __shared__ __attribute__((aligned(16))) uint8_t lds[4 * kDqWave];
    static_assert(64 * kDqRow <= kTileN * kDqCol, "the second turn reuses the first one's bytes");
    const int nchunks = K / 64, groups = K / group_k;
    const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int64_t x = (int64_t)blockIdx.x * 4 + wv;  // strip * nchunks + c
    const int b = blockIdx.y;
    if (x >= (int64_t)strips * nchunks) return;  // uniform over the wavefront; no barrier follows
    const int c = (int)(x % nchunks), strip = (int)(x / nchunks);
    const int i = lane & 15, q = lane >> 4;
    uint8_t* const buf = lds + wv * kDqWave;
    uint8_t* const scl = buf + kTileN * kDqCol;  // the chunk's 128 scales in column order
    const uint8_t* const blk = pk + ((int64_t)b * strips * nchunks + x) * kPackBytes + 16 * lane;
    u4 R[6];
#pragma unroll
    for (int k = 0; k < 6; ++k) R[k] = *reinterpret_cast<const u4*>(blk + 1024 * k);
    const int g = (c * 64) / group_k;
    const u4 sv = *reinterpret_cast<const u4*>(psc + ((int64_t)b * strips * groups + (int64_t)strip * groups + g) * kTileN +
                                               8 * i);
#pragma unroll
    for (int t = 0; t < kTiles; ++t) {
        const uint32_t L0 = R[t >> 1][2 * (t & 1)], L1 = R[t >> 1][2 * (t & 1) + 1], Hd = R[4 + (t >> 2)][t & 3];
        uint8_t* const col = buf + (16 * t + i) * kDqCol + 8 * q;
        *reinterpret_cast<uint2*>(col) = uint2{(L0 & 0x0F0F0F0Fu) | ((Hd & 0x03030303u) << 4),
                                               (L1 & 0x0F0F0F0Fu) | (Hd & 0x30303030u)};
        *reinterpret_cast<uint2*>(col + 32) = uint2{((L0 >> 4) & 0x0F0F0F0Fu) | ((Hd & 0x0C0C0C0Cu) << 2),
                                                    ((L1 >> 4) & 0x0F0F0F0Fu) | ((Hd >> 2) & 0x30303030u)};
        if (q == 0) *reinterpret_cast<uint16_t*>(scl + 2 * (16 * t + i)) = (uint16_t)(sv[t >> 1] >> (16 * (t & 1)));
    }
    wave_lds_sync();
    // lane i of group q: row 16 k + i, columns 8 (4 m + q) .. + 7
    v2i u[4][4];
#pragma unroll
    for (int k = 0; k < 4; ++k)
#pragma unroll
        for (int m = 0; m < 4; ++m)
            u[k][m] = __builtin_amdgcn_ds_read_tr8_b64_v2i32(
                (lds_v2i*)(buf + (8 * (4 * m + q) + (i >> 1)) * kDqCol + 16 * k + 8 * (i & 1)));
    wave_lds_sync();
#pragma unroll
    for (int k = 0; k < 4; ++k)
#pragma unroll
        for (int m = 0; m < 4; ++m) *reinterpret_cast<v2i*>(buf + (16 * k + i) * kDqRow + 8 * (4 * m + q)) = u[k][m];
    wave_lds_sync();
    // 16 bytes a lane: eight columns of four rows an instruction, in fp32 four columns of two
    if constexpr (sizeof(OutT) == 2) {
        const int n = strip * kTileN + 8 * i;
        if (n >= N) return;
        const u4 sc = *reinterpret_cast<const u4*>(scl + 16 * i);
        OutT* const dst = w + b * sw_b + ((int64_t)c * 64 + q) * N + n;
#pragma unroll
        for (int y = 0; y < 16; ++y) {
            float v[8];
            dequant8(*reinterpret_cast<const uint2*>(buf + (4 * y + q) * kDqRow + 8 * i), sc, v);
            store_row8(dst + (int64_t)(4 * y) * N, v, vec);
        }
    } else {
        const int h = lane >> 5, k = lane & 31, n = strip * kTileN + 4 * k;
        if (n >= N) return;
        const uint2 sc = *reinterpret_cast<const uint2*>(scl + 8 * k);
        OutT* const dst = w + b * sw_b + ((int64_t)c * 64 + h) * N + n;
#pragma unroll
        for (int y = 0; y < 32; ++y) {
            float v[8];
            const uint32_t u = *reinterpret_cast<const uint32_t*>(buf + (2 * y + h) * kDqRow + 4 * k);
            dequant8(uint2{u, 0}, u4{sc.x, sc.y, 0, 0}, v);
            OutT* const d = dst + (int64_t)(2 * y) * N;
            if (vec)
                *reinterpret_cast<f4*>(d) = f4{v[0], v[1], v[2], v[3]};
            else
#pragma unroll
                for (int e = 0; e < 4; ++e) d[e] = v[e];
        }
    }
}

// Repack: one thread per (b, strip, chunk, lane) writes the lane's 24-dword record.
__global__ __launch_bounds__(256) void w6a16_pack_kernel(const uint8_t* lo, const uint8_t* hi, uint8_t* out, int32_t K,
                                                         int32_t N, int32_t strips, int64_t sl_b, int64_t sh_b) {
    const int nchunks = K / 64;
    const int64_t x = (int64_t)blockIdx.x * 256 + threadIdx.x;  // ((strip * nchunks + c) * 64 + lane) within batch
    const int b = blockIdx.y;
    if (x >= (int64_t)strips * nchunks * 64) return;
    const int lane = (int)(x & 63);
    const int64_t sc = x >> 6;
    const int c = (int)(sc % nchunks), strip = (int)(sc / nchunks);
    const int i = lane & 15, q = lane >> 4;
    const uint8_t* const L = lo + b * sl_b;
    const uint8_t* const H = hi + b * sh_b;
    uint32_t R[24];
#pragma unroll
    for (int t = 0; t < kTiles; ++t) {
        const int n = strip * kTileN + 16 * t + i;
        uint32_t l0 = 0, l1 = 0, hd = 0;
        if (n < N) {
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                l0 |= (uint32_t)L[((int64_t)c * 32 + 8 * q + e) * N + n] << (8 * e);
                l1 |= (uint32_t)L[((int64_t)c * 32 + 8 * q + 4 + e) * N + n] << (8 * e);
            }
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int rows[4] = {8 * q + e, 32 + 8 * q + e, 8 * q + 4 + e, 32 + 8 * q + 4 + e};
                uint32_t byte = 0;
#pragma unroll
                for (int f = 0; f < 4; ++f) {
                    const int r = rows[f];
                    const uint32_t top = (H[((int64_t)c * 16 + (r & 15)) * N + n] >> (2 * (r >> 4))) & 3u;
                    byte |= top << (2 * f);
                }
                hd |= byte << (8 * e);
            }
        }
        R[2 * t] = l0;
        R[2 * t + 1] = l1;
        R[16 + t] = hd;
    }
    uint8_t* const blk = out + ((int64_t)b * strips * nchunks + sc) * kPackBytes + 16 * lane;
#pragma unroll
    for (int k = 0; k < 6; ++k) *reinterpret_cast<u4*>(blk + 1024 * k) = u4{R[4 * k], R[4 * k + 1], R[4 * k + 2], R[4 * k + 3]};
}

// Repack the scales: one thread per (b, strip, group, i) writes the eight scales of columns 128 strip + 16 t + i.
__global__ __launch_bounds__(256) void w6a16_pack_scales_kernel(const uint16_t* sc, uint16_t* out, int32_t groups,
                                                                int32_t N, int32_t strips, int64_t ss_b) {
    const int64_t x = (int64_t)blockIdx.x * 256 + threadIdx.x;  // ((strip * groups + g) * 16 + i) within batch
    const int b = blockIdx.y;
    if (x >= (int64_t)strips * groups * 16) return;
    const int i = (int)(x & 15);
    const int64_t sg = x >> 4;
    const int g = (int)(sg % groups), strip = (int)(sg / groups);
    uint32_t o[4];
#pragma unroll
    for (int h = 0; h < 4; ++h) {
        uint32_t v[2];
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            const int n = strip * kTileN + 16 * (2 * h + u) + i;
            v[u] = n < N ? sc[b * ss_b + (int64_t)g * N + n] : 0u;
        }
        o[h] = v[0] | v[1] << 16;
    }
    *reinterpret_cast<u4*>(out + ((int64_t)b * strips * groups + sg) * kTileN + 8 * i) = u4{o[0], o[1], o[2], o[3]};
}

// Dequantise: w[b][k][n] = s q as bf16, fp16 or fp32 (the large-M path hands the result to a library GEMM).  Grid
// (ceil(N / 2048), K / 16, B): one thread per (four hi rows, 8 columns); hi row j's four fields and lo rows j and j + 16
// give rows j, j + 16, j + 32 and j + 48 of the chunk, stored as whole lines (a wavefront 1 KB of a row in bf16).
// K = 4096, N = 16384, bf16, weights cycled: 52.3 us with two 16-byte stores at 32 bytes from lane to lane -> 32.4.
template <typename OutT>
__global__ __launch_bounds__(256) void w6a16_dequant_kernel(const uint8_t* lo, const uint8_t* hi, const uint16_t* sc,
                                                            OutT* w, int32_t K, int32_t N, int32_t group_k,
                                                            int64_t sl_b, int64_t sh_b, int64_t ss_b, int64_t sw_b) {
    const int64_t n = ((int64_t)blockIdx.x * 256 + threadIdx.x) * 8;
    if (n >= N) return;
    const int c = blockIdx.y >> 2, j0 = 4 * (blockIdx.y & 3), b = blockIdx.z;
    const uint8_t* const L = lo + b * sl_b + ((int64_t)c * 32 + j0) * N + n;
    const uint8_t* const H = hi + b * sh_b + ((int64_t)c * 16 + j0) * N + n;
    const u4 s = *reinterpret_cast<const u4*>(sc + b * ss_b + (int64_t)(c * 64 / group_k) * N + n);
    OutT* const dst = w + b * sw_b + ((int64_t)c * 64 + j0) * N + n;
    uint2 l[4][2], h[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        l[j][0] = *reinterpret_cast<const uint2*>(L + (int64_t)j * N);
        l[j][1] = *reinterpret_cast<const uint2*>(L + (int64_t)(16 + j) * N);
        h[j] = *reinterpret_cast<const uint2*>(H + (int64_t)j * N);
    }
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int f = 0; f < 4; ++f) {  // row j0 + j + 16 f: nibble f >> 1 of lo row j0 + j + 16 (f & 1), field f of the hi row
            const uint2 x = l[j][f & 1];
            const int nib = 4 * (f >> 1);
            const uint2 u = uint2{((x.x >> nib) & 0x0F0F0F0Fu) | (((h[j].x >> (2 * f)) & 0x03030303u) << 4),
                                  ((x.y >> nib) & 0x0F0F0F0Fu) | (((h[j].y >> (2 * f)) & 0x03030303u) << 4)};
            float v[8];
            dequant8(u, s, v);
            store8(dst + (int64_t)(16 * f + j) * N, v);
        }
}

// ---------------------------------------------------------------------------------------------------------------
// Large-M kernel (M > kBigMinM, prefill-sized M, packed weights): C = A W~ with W~ = s q rounded to A's type -- the
// values w6a16_dequantize writes, so the result is that of dequantising and multiplying, in one kernel with no
// workspace.  A workgroup of eight wavefronts (two per SIMD) computes a 256 x 256 tile of C.  Per 64-row chunk of K it
// stages A's 256 x 64 slice and W~'s 64 x 256 slice (dequantised once per workgroup and stored transposed: LDS row n
// holds the 64 k of column n) in LDS, double-buffered with one barrier per chunk.  Wavefront (wm, wn) multiplies a
// 128 x 64 eighth: 32 MFMA tiles, 128 fp32 accumulators a lane, in 16 blocks (k half, 16-row tile) whose A operand is
// read one block ahead.  In the MFMAs' shadow, a quarter of the next chunk's weight share (loaded one chunk earlier)
// is dequantised and stored after every fourth block, A's next chunk (loaded at the chunk's start) is stored at its
// end, and the weight bytes of the chunk after that are loaded; scheduler fences keep this order.  The MFMA's A
// operand is a W~^T tile (rows n), its B operand an A^T tile (columns m), so lane (i, q) of tile (mt, nt) ends
// holding C[m0 + 16 mt + i][n0 + 16 nt + 4 q .. + 3]: four adjacent outputs, stored together.
constexpr int kBigTile = 256;                  // rows of A and columns of W per workgroup
constexpr int kBigStage = 2 * kBigTile * 128;  // bytes per stage: A rows, then W~^T rows, 64 elements each

// 16-byte piece p (k = 8 p .. 8 p + 7) of LDS row r (128-byte rows): piece slots XOR-swizzled by (r >> 1) & 7, so the
// 16 rows of one operand read (one p) fall in 16 different 16-byte bank groups.
__device__ __forceinline__ int big_slot(int r, int p) { return r * 128 + 16 * (p ^ ((r >> 1) & 7)); }

// Two values as a pair of A's element type (round to nearest even).
template <class A>
__device__ __forceinline__ uint32_t pack_act(float x, float y) {
    if constexpr (std::is_same_v<A, ActF16>)
        return (uint32_t)__builtin_bit_cast(uint16_t, (_Float16)x) |
               (uint32_t)__builtin_bit_cast(uint16_t, (_Float16)y) << 16;
    else
        return (uint32_t)__builtin_bit_cast(uint16_t, (__bf16)x) | (uint32_t)__builtin_bit_cast(uint16_t, (__bf16)y)
                                                                      << 16;
}

// s (u - 32) of the four codes u in the bytes of `u`, as A's type: the fp32 product of an 11-bit scale and a 6-bit
// integer is exact, so the one rounding is the conversion (the dequantisation kernel's values, bit for bit).
template <class A>
__device__ __forceinline__ void dequant4(uint32_t u, float s, float s32, uint32_t& d0, uint32_t& d1) {
    const float v0 = __builtin_fmaf((float)(u & 0xFF), s, s32), v1 = __builtin_fmaf((float)((u >> 8) & 0xFF), s, s32);
    const float v2 = __builtin_fmaf((float)((u >> 16) & 0xFF), s, s32), v3 = __builtin_fmaf((float)(u >> 24), s, s32);
    d0 = pack_act<A>(v0, v1);
    d1 = pack_act<A>(v2, v3);
}

// One chunk's weight bytes, per thread: the packed weight's share of wavefront w (strip w >> 2 of the tile, tiles
// 2 (w & 3) and 2 (w & 3) + 1 -- their lo dwords, one 16-byte lane load of the block, their two hi dwords and their
// two scales).  A's rows go from memory straight into LDS (big_copy_a).
struct BigW {
    u4 w;
    uint2 h;
    uint32_t sc;
};

// Where a thread's loads go, fixed for the call: raw buffers over A's batch slice, the packed weight's and its scales
// (wave-uniform descriptors), the lane's 32-bit offsets, and the wavefront's strip offsets; per chunk only a scalar
// offset changes.  (With 64-bit per-lane addresses the compiler placed the next chunk's address registers where the
// previous chunk's weight bytes were still arriving and waited for those loads first.)
struct BigSrc {
    __amdgpu_buffer_rsrc_t ra, rw, rs;
    int va[4];        // A row 8 w + 64 j + (lane >> 3) of the tile, the piece its LDS slot lane & 7 holds (+ 128
                      // bytes per chunk)
    int vw, vh, vs;   // the lane's offsets into a weight block (lo dwords, hi dwords) and a scale block
    int sw, ss;       // the wavefront's strip: byte offsets of its first weight block and first scale block
};

__device__ __forceinline__ BigSrc big_src(const Args& p, int b, int m0, int n0) {
    BigSrc d;
    const int t = threadIdx.x, wv = t >> 6, lane = t & 63, i = lane & 15, w4 = wv & 3;
    const int nchunks = p.K / 64, groups = p.K / p.group_k;
    d.ra = rsrc((uint64_t)(p.a + (int64_t)b * p.sa_b), ((int64_t)(p.M - 1) * p.sa_m + p.K) * 2);
    d.rw = rsrc((uint64_t)(p.lo + (int64_t)b * p.sl_b), (int64_t)p.n_strips * nchunks * kPackBytes);
    d.rs = rsrc((uint64_t)(p.sc + (int64_t)b * p.ss_b), (int64_t)p.n_strips * groups * kTileN * 2);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const int r = 8 * wv + 64 * j + (lane >> 3), piece = (lane & 7) ^ ((r >> 1) & 7);  // big_slot's swizzle
        d.va[j] = min(m0 + r, p.M - 1) * (int)p.sa_m * 2 + 16 * piece;
    }
    const int strip = min(n0 / kTileN + (wv >> 2), p.n_strips - 1);
    d.vw = 1024 * w4 + 16 * lane;                                  // R[4 w4 .. 4 w4 + 3]
    d.vh = 1024 * (4 + (w4 >> 1)) + 8 * (w4 & 1) + 16 * lane;     // R[16 + 2 w4], R[17 + 2 w4]
    d.vs = (8 * i + 2 * w4) * 2;
    d.sw = strip * nchunks * kPackBytes;
    d.ss = strip * groups * kTileN * 2;
    return d;
}

__device__ __forceinline__ void vmem_wait() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }

// A's 256 x 64 slice of chunk c into a stage, straight from memory (buffer_load ... lds): wavefront w's load j fills
// the stage's 1 KB of rows 8 w + 64 j .. + 7, lane l the 16-byte slot l & 7 of row 8 w + 64 j + (l >> 3), with the
// piece big_slot places there.  The two stages are separate LDS arrays, so the compiler sees that these writes do
// not alias the current stage's operand reads and waits for them only at the barrier.
__device__ __forceinline__ void big_copy_a(const BigSrc& d, int c, uint8_t* stage) {
    const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
#pragma unroll
    for (int j = 0; j < 4; ++j)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(d.ra, (__attribute__((address_space(3))) void*)(stage + (8 * wv + 64 * j) * 128),
                                                 16, d.va[j], soff(128 * c), 0, 0);
}

__device__ __forceinline__ void big_load_w(const Args& p, const BigSrc& d, int c, BigW& g) {
    const int blk = soff(d.sw + c * kPackBytes);
    g.w = __builtin_bit_cast(u4, __builtin_amdgcn_raw_buffer_load_b128(d.rw, d.vw, blk, 0));
    g.h = __builtin_bit_cast(uint2, __builtin_amdgcn_raw_buffer_load_b64(d.rw, d.vh, blk, 0));
    g.sc = __builtin_amdgcn_raw_buffer_load_b32(d.rs, d.vs, soff(d.ss + ((c * 64) / p.group_k) * kTileN * 2), 0);
}

// Piece e (0..3) of the wavefront's weight share, dequantised into the stage: tile t = 2 (w & 3) + (e >> 1), rows
// 8 q .. + 7 (e even) or 32 + 8 q .. + 7 (e odd) of column 128 (w >> 2) + 16 t + i.
template <class A>
__device__ __forceinline__ void big_store_w(uint8_t* stage, const BigW& g, int e) {
    const int wv = threadIdx.x >> 6, lane = threadIdx.x & 63, i = lane & 15, q = lane >> 4, w4 = wv & 3;
    const int tt = e >> 1;
    const uint32_t L0 = g.w[2 * tt], L1 = g.w[2 * tt + 1], Hd = tt ? g.h.y : g.h.x;
    uint32_t ua, ub;
    if (e & 1) {
        ua = ((L0 >> 4) & 0x0F0F0F0Fu) | ((Hd & 0x0C0C0C0Cu) << 2);  // rows 32 + 8 q + 0..3
        ub = ((L1 >> 4) & 0x0F0F0F0Fu) | ((Hd >> 2) & 0x30303030u);  // rows 32 + 8 q + 4..7
    } else {
        ua = (L0 & 0x0F0F0F0Fu) | ((Hd & 0x03030303u) << 4);  // rows 8 q + 0..3
        ub = (L1 & 0x0F0F0F0Fu) | (Hd & 0x30303030u);         // rows 8 q + 4..7
    }
    const float s = h2f((uint16_t)(g.sc >> (16 * tt))), s32 = -32.f * s;
    uint32_t d[4];
    dequant4<A>(ua, s, s32, d[0], d[1]);
    dequant4<A>(ub, s, s32, d[2], d[3]);
    const int r = kBigTile + 128 * (wv >> 2) + 16 * (2 * w4 + tt) + i;
    *reinterpret_cast<u4*>(stage + big_slot(r, (e & 1) * 4 + q)) = u4{d[0], d[1], d[2], d[3]};
}

// Tile index -> (M tile, N tile).  Workgroup x runs on XCD x % 8; when the tiles divide evenly, XCD x takes the x-th
// eighth of the tiles in bands of 8 N tiles, M tile by M tile, so the workgroups resident on one XCD at a time share
// A's rows and W's columns in that XCD's L2.
__device__ __forceinline__ void big_tile(int tiles_m, int tiles_n, int& tm, int& tn) {
    const int T = tiles_m * tiles_n, x = blockIdx.x;
    const int L = (T % 8 == 0) ? (x % 8) * (T / 8) + x / 8 : x;
    constexpr int kBand = 8;
    const int band = L / (tiles_m * kBand), idx = L - band * tiles_m * kBand;
    const int width = min(kBand, tiles_n - band * kBand);
    tm = idx / width;
    tn = band * kBand + idx % width;
}

// The wavefront's 128 x 64 outputs, lane row m0 + 16 mt, columns n0 + 16 nt .. + 3: ES = 4 (fp32) or 2 (bf16 / fp16,
// out_dtype) bytes an element in one vector store, or (VEC false) element by element as out_dtype.
template <int ES, bool VEC>
__device__ __forceinline__ void big_store_out(const Args& p, int b, int m0, int n0, const f4 (&acc)[8][4]) {
    const bool f16 = p.out_dtype == W6A16_OUT_F16;
#pragma unroll
    for (int mt = 0; mt < 8; ++mt) {
        const int m = m0 + 16 * mt;
        if (m >= p.M) continue;
#pragma unroll
        for (int nt = 0; nt < 4; ++nt) {
            const int n = n0 + 16 * nt;
            if (n >= p.N) continue;
            const int64_t o = (int64_t)b * p.so_b + (int64_t)m * p.so_m + n;
            const f4 v = acc[mt][nt];
            if constexpr (VEC && ES == 4) {
                *reinterpret_cast<f4*>(reinterpret_cast<float*>(p.out) + o) = v;
            } else if constexpr (VEC) {
                *reinterpret_cast<uint2*>(reinterpret_cast<uint16_t*>(p.out) + o) =
                    f16 ? uint2{pack_act<ActF16>(v[0], v[1]), pack_act<ActF16>(v[2], v[3])}
                        : uint2{pack_act<ActBF16>(v[0], v[1]), pack_act<ActBF16>(v[2], v[3])};
            } else {
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    if (p.out_dtype == W6A16_OUT_F32)
                        reinterpret_cast<float*>(p.out)[o + e] = v[e];
                    else if (f16)
                        reinterpret_cast<_Float16*>(p.out)[o + e] = (_Float16)v[e];
                    else
                        reinterpret_cast<__bf16*>(p.out)[o + e] = (__bf16)v[e];
                }
            }
        }
    }
}

// One chunk of the large-M kernel: the MFMAs over stage `cur`; the next chunk's weights dequantised into the other
// stage's weight rows (`nxt_w`) during the first two MFMA blocks, then A's next chunk copied into its A rows (`nxt_a`,
// the same stage base: the two touch disjoint bytes).  The stages come in as restrict pointers, so that after
// inlining their accesses carry alias scopes and the compiler's wait insertion sees that the copies do not alias the
// operand reads of `cur`; no LDS store follows the copies within the step (the compiler would wait for them before
// one), so the only wait for them is at the barrier.
template <class A>
__device__ __forceinline__ void big_step(const Args& p, const BigSrc& src, int c, int nch,
                                         const uint8_t* __restrict__ cur, uint8_t* __restrict__ nxt_a,
                                         uint8_t* __restrict__ nxt_w, const BigW& ws, BigW& wl, f4 (&acc)[8][4]) {
    const int wv = threadIdx.x >> 6, lane = threadIdx.x & 63, i = lane & 15, q = lane >> 4;
    const int wm = wv & 1, wn = wv >> 1;
    big_load_w(p, src, min(c + 2, nch - 1), wl);
    u4 wo[4], ao[2];
    ao[0] = *reinterpret_cast<const u4*>(cur + big_slot(128 * wm + i, q));
#pragma unroll
    for (int blk = 0; blk < 16; ++blk) {
        const int kh = blk >> 3, mt = blk & 7;
        if (mt == 0) {
#pragma unroll
            for (int nt = 0; nt < 4; ++nt)
                wo[nt] = *reinterpret_cast<const u4*>(cur + kBigTile * 128 + big_slot(64 * wn + 16 * nt + i, 4 * kh + q));
        }
        if (blk + 1 < 16) {
            const int kn = (blk + 1) >> 3, mn = (blk + 1) & 7;
            ao[(blk + 1) & 1] = *reinterpret_cast<const u4*>(cur + big_slot(128 * wm + 16 * mn + i, 4 * kn + q));
        }
#pragma unroll
        for (int nt = 0; nt < 4; ++nt) acc[mt][nt] = A::mma(wo[nt], ao[blk & 1], acc[mt][nt]);
        if (blk < 2) {
#pragma unroll
            for (int e = 2 * blk; e < 2 * blk + 2; ++e) big_store_w<A>(nxt_w, ws, e);
        }
        if (blk == 1) big_copy_a(src, min(c + 1, nch - 1), nxt_a);  // after the last weight store (the last steps
                                                                       // copy the last chunk again, unused)
        __builtin_amdgcn_sched_barrier(0);
    }
    vmem_wait();
    __syncthreads();
}

template <class A>
__global__ __launch_bounds__(512, 1) void w6a16_big_kernel(const Args p) {
    __shared__ __attribute__((aligned(16))) uint8_t lds0[kBigStage];
    __shared__ __attribute__((aligned(16))) uint8_t lds1[kBigStage];
    const int wv = threadIdx.x >> 6, lane = threadIdx.x & 63, i = lane & 15, q = lane >> 4;
    const int wm = wv & 1, wn = wv >> 1;  // rows 128 wm .., columns 64 wn ..
    const int tiles_m = (p.M + kBigTile - 1) / kBigTile, tiles_n = (p.N + kBigTile - 1) / kBigTile;
    int tm, tn;
    big_tile(tiles_m, tiles_n, tm, tn);
    const int b = blockIdx.z, m0 = tm * kBigTile, n0 = tn * kBigTile;
    const int nch = p.K / 64;
    f4 acc[8][4];
#pragma unroll
    for (int mt = 0; mt < 8; ++mt)
#pragma unroll
        for (int nt = 0; nt < 4; ++nt) acc[mt][nt] = f4{0.f, 0.f, 0.f, 0.f};
    const BigSrc src = big_src(p, b, m0, n0);
    BigW w0, w1;
    big_copy_a(src, 0, lds0);
    big_load_w(p, src, 0, w0);
    big_load_w(p, src, min(1, nch - 1), w1);
#pragma unroll
    for (int e = 0; e < 4; ++e) big_store_w<A>(lds0, w0, e);
    vmem_wait();  // this wavefront's copies into the stage have landed (the barrier does not wait for them)
    __syncthreads();
    // chunk c: its stage is c & 1 (lds0 / lds1, fixed per unrolled step); ws holds chunk c + 1's weight bytes, wl
    // receives chunk c + 2's
    auto step = [&](auto odd, int c, const BigW& ws, BigW& wl) {
        if constexpr (decltype(odd)::value)
            big_step<A>(p, src, c, nch, lds1, lds0, lds0, ws, wl, acc);
        else
            big_step<A>(p, src, c, nch, lds0, lds1, lds1, ws, wl, acc);
    };
    for (int c = 0; c < nch; c += 2) {
        step(std::false_type{}, c, w1, w0);
        if (c + 1 < nch) step(std::true_type{}, c + 1, w0, w1);
    }
    // lane (i, q) of tile (mt, nt): C[m0 + 128 wm + 16 mt + i][n0 + 64 wn + 16 nt + 4 q .. + 3] (N % 16 == 0: the
    // four columns are all inside or all outside)
    if (p.out_vec && p.out_dtype == W6A16_OUT_F32)
        big_store_out<4, true>(p, b, m0 + 128 * wm + i, n0 + 64 * wn + 4 * q, acc);
    else if (p.out_vec)
        big_store_out<2, true>(p, b, m0 + 128 * wm + i, n0 + 64 * wn + 4 * q, acc);
    else
        big_store_out<0, false>(p, b, m0 + 128 * wm + i, n0 + 64 * wn + 4 * q, acc);
}

int cu_count() { return wkv7::device_cu_count(); }

bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; }

int validate(const w6a16_args* a) {
    if (!a) return WKV7_ERR_NULL;
    if (a->B < 1 || a->M < 0 || a->N < 1 || a->K < 64 || a->K % 64 || a->N % 16) return WKV7_ERR_SHAPE;
    if (a->group_k < 64 || a->group_k % 64 || a->K % a->group_k) return WKV7_ERR_SHAPE;
    if (a->split_k < 1 || a->split_k > 256) return WKV7_ERR_ARG;
    if (a->out_dtype != W6A16_OUT_BF16 && a->out_dtype != W6A16_OUT_F16 && a->out_dtype != W6A16_OUT_F32)
        return WKV7_ERR_ARG;
    if (a->a_dtype != W6A16_IN_BF16 && a->a_dtype != W6A16_IN_F16) return WKV7_ERR_ARG;
    if (a->M == 0) return WKV7_OK;
    if (a->format != W6A16_FORMAT_PLANES && a->format != W6A16_FORMAT_PACKED) return WKV7_ERR_ARG;
    const bool packed = a->format == W6A16_FORMAT_PACKED;
    if (!a->a || !a->lo || (!packed && !a->hi) || !a->scales || !a->out) return WKV7_ERR_NULL;
    if (!aligned16(a->a) || !aligned16(a->lo) || a->a_row_stride % 8 || a->a_batch_stride % 8 ||
        a->lo_batch_stride % 16)
        return WKV7_ERR_ALIGN;
    if (packed ? (!aligned16(a->scales) || a->scales_batch_stride % 8)
               : (!aligned16(a->hi) || (reinterpret_cast<uintptr_t>(a->scales) & 3) || a->hi_batch_stride % 16 ||
                  a->scales_batch_stride % 2))
        return WKV7_ERR_ALIGN;
    if (a->a_row_stride < a->K || a->out_row_stride < a->N) return WKV7_ERR_SHAPE;
    const Layout l = layout(a, cu_count());
    if (l.big) {  // grid (tiles, 1, B)
        const int64_t tiles = (int64_t)((a->M + kBigTile - 1) / kBigTile) * ((a->N + kBigTile - 1) / kBigTile);
        return (a->B > 65535 || tiles > 0x7FFFFFFF) ? WKV7_ERR_SHAPE : WKV7_OK;
    }
    const bool small = a->M <= kSmallM;
    if ((int64_t)a->B * (small ? l.m_groups : 1) > 65535) return WKV7_ERR_SHAPE;  // (B: grid y, at most 65535)
    if (!small && (int64_t)l.m_groups * ((l.n_strips + 7) / 8) * 8 > 0x7FFFFFFF) return WKV7_ERR_SHAPE;
    if (a->split_k > 1 && l.tiles * 4 > kCounterRegion) return WKV7_ERR_SHAPE;  // more tiles than counters
    if (l.total_bytes) {
        if (!a->workspace || a->workspace_bytes < l.total_bytes) return WKV7_ERR_WORKSPACE;
        if (reinterpret_cast<uintptr_t>(a->workspace) % kCounterAlign) return WKV7_ERR_ALIGN;
    }
    return WKV7_OK;
}

template <class A, int MT, int NA, int NT, int CW, int D, int DA, int MAXW, bool PACKED, bool FAR = false>
int launch_tile(Args& p, const TilePlan& t, hipStream_t s) {
    const int chunks = p.K / 64;
    const uint64_t wgs = tile_grid(p.N / 16, (p.M + 16 * MT - 1) / (16 * MT), NT * CW, p.grid);
    if (wgs >> 34) return WKV7_ERR_SHAPE;
    p.group = divisor(p.group_k / 64);
    p.parts = t.parts;
    p.per_part = (chunks + t.parts - 1) / t.parts;
    p.groups = p.K / p.group_k;
    const uint32_t block = 64 * CW * t.parts / t.ks, most = launch_limit(block);
    if (block < 16 * NT * CW || block > 64 * MAXW) return WKV7_ERR_SHAPE;  // (no plan: the outputs take a thread a column)
    for (uint64_t x = 0; x < wgs; x += most) {
        p.grid.first = (uint32_t)(x / 8);
        hipLaunchKernelGGL((w6a16_tile_kernel<A, MT, NA, NT, CW, D, DA, MAXW, PACKED, FAR>),
                           dim3((unsigned)std::min<uint64_t>(wgs - x, most), p.B, t.ks), dim3(block),
                           block / 64 * tile_lds(MT, NA, NT), s, p);
    }
    return WKV7_OK;
}

// D chunks of weights and DA of A in flight: as many as the registers of MAXW wavefronts allow.
template <class A, int NA, bool PACKED>
int launch_tile_one(Args& p, const TilePlan& t, hipStream_t s) {  // one row tile
    if constexpr (PACKED) {
        if (t.nt == 1) return launch_tile<A, 1, NA, 1, 1, 4, 4, 16, true>(p, t, s);
        if (t.nt == 2) return launch_tile<A, 1, NA, 2, 1, 4, 4, 16, true>(p, t, s);
    } else {
        if (t.nt == 8) return launch_tile<A, 1, NA, 8, 1, 2, 2, 8, false>(p, t, s);
    }
    if (t.parts / t.ks > 8) return launch_tile<A, 1, NA, 4, 1, 2, 2, 16, PACKED>(p, t, s);
    return launch_tile<A, 1, NA, 4, 1, 4, 4, 8, PACKED>(p, t, s);
}

template <class A, bool PACKED>
int launch_tile_plan(Args& p, const TilePlan& t, hipStream_t s) {
    if (t.far) return launch_tile<A, 1, 2, 4, 1, 2, 2, 16, PACKED, true>(p, t, s);
    if (t.mt == 1) return p.M <= 8 ? launch_tile_one<A, 1, PACKED>(p, t, s) : launch_tile_one<A, 2, PACKED>(p, t, s);
    if (t.mt == 2) {
        if constexpr (PACKED) {
            if (t.nt == 1) return launch_tile<A, 2, 4, 1, 1, 2, 2, 16, true>(p, t, s);
            if (t.nt == 2) return launch_tile<A, 2, 4, 2, 1, 2, 2, 8, true>(p, t, s);
        }
        return launch_tile<A, 2, 4, 4, 1, 2, 2, 8, PACKED>(p, t, s);
    }
    if (t.mt == 3)
        return t.cw == 2 ? launch_tile<A, 3, 6, 4, 2, 2, 1, 8, PACKED>(p, t, s) : launch_tile<A, 3, 6, 4, 1, 2, 1, 8, PACKED>(p, t, s);
    return t.cw == 2 ? launch_tile<A, 4, 8, 4, 2, 2, 1, 8, PACKED>(p, t, s) : launch_tile<A, 4, 8, 4, 1, 2, 1, 8, PACKED>(p, t, s);
}

template <class A, bool PACKED>
int launch_wide(Args& p, const w6a16_args* a, const Layout& l, hipStream_t s) {
    const uint64_t wgs = tile_grid(p.N / 16, l.m_groups, kTiles, p.grid);  // (K N < 2^32: within one launch)
    p.group = divisor(p.group_k / 64);
    p.groups = p.K / p.group_k;
    p.chain_k = p.group_k % 128 == 0 ? 128 : 64;
    p.nchains = l.nchains;
    p.mpad = l.m_groups * kWideRows;
    p.rsum = reinterpret_cast<float*>(static_cast<char*>(a->workspace) + kCounterRegion + l.partial_bytes);
    hipLaunchKernelGGL(w6a16_rowsum_kernel<A>, dim3(p.mpad / 4, (p.K + 511) / 512, p.B), dim3(256), 0, s, p);
    auto run = [&](auto two, auto far) {
        hipLaunchKernelGGL((w6a16_wide_kernel<A, decltype(two)::value ? 2 : 1, PACKED, decltype(far)::value>),
                           dim3((unsigned)wgs, 1, p.B), dim3(256), 0, s, p);
    };
    const bool two = p.chain_k == 128, far = p.sa_m >= (1 << 24);
    if (two) far ? run(std::true_type{}, std::true_type{}) : run(std::true_type{}, std::false_type{});
    else far ? run(std::false_type{}, std::true_type{}) : run(std::false_type{}, std::false_type{});
    return WKV7_OK;
}

// The kernel for the call's shape and layout, with activations of type A.
template <class A>
int launch_matmul(Args& p, const w6a16_args* a, const Layout& l, hipStream_t s) {
    const bool packed = a->format == W6A16_FORMAT_PACKED;
    if (l.big) {
        const int tiles = ((p.M + kBigTile - 1) / kBigTile) * ((p.N + kBigTile - 1) / kBigTile);
        hipLaunchKernelGGL(w6a16_big_kernel<A>, dim3(tiles, 1, p.B), dim3(512), 0, s, p);
        return WKV7_OK;
    }
    if (wide_call(a, l, cu_count())) return packed ? launch_wide<A, true>(p, a, l, s) : launch_wide<A, false>(p, a, l, s);
    const TilePlan t = tile_plan(a, l, packed, cu_count());
    return packed ? launch_tile_plan<A, true>(p, t, s) : launch_tile_plan<A, false>(p, t, s);
}

}  // namespace
}  // namespace w6

extern "C" {

size_t w6a16_args_size(void) { return sizeof(w6a16_args); }

int w6a16_workspace_size(const w6a16_args* a, size_t* bytes) {
    if (!a || !bytes) return WKV7_ERR_NULL;
    const bool none = a->M <= 0 || a->B < 1 || a->N < 1 || a->K < 64 || a->group_k < 64;
    *bytes = none ? 0 : w6::layout(a, w6::cu_count()).total_bytes;
    return WKV7_OK;
}

int w6a16_plan_split(int32_t B, int32_t M, int32_t N, int32_t K) {
    return B < 1 || M < 1 || N < 1 || K < 64 ? 1 : w6::plan_split(B, M, N, K, w6::cu_count());
}

int w6a16_plan_split_packed(int32_t B, int32_t M, int32_t N, int32_t K) {
    return B < 1 || M < 1 || N < 1 || K < 64 ? 1 : w6::plan_split_packed(B, M, N, K, w6::cu_count());
}

int w6a16_matmul(const w6a16_args* a, void* stream) {
    const int rc = w6::validate(a);
    if (rc != WKV7_OK || a->M == 0) return rc;
    const w6::Layout l = w6::layout(a, w6::cu_count());
    w6::Args p{};
    p.a = a->a;
    p.sa_b = a->a_batch_stride;
    p.sa_m = a->M > 1 ? a->a_row_stride : a->K;
    p.lo = a->lo;
    p.hi = a->hi;
    p.sl_b = a->lo_batch_stride;
    p.sh_b = a->hi_batch_stride;
    p.sc = a->scales;
    p.ss_b = a->scales_batch_stride;
    p.out = a->out;
    p.so_b = a->out_batch_stride;
    p.so_m = a->out_row_stride;
    p.cnt = static_cast<uint32_t*>(a->workspace);  // used only where the plan splits K over workgroups
    p.part = reinterpret_cast<float*>(static_cast<char*>(a->workspace) + w6::kCounterRegion);
    p.B = a->B;
    p.M = a->M;
    p.N = a->N;
    p.K = a->K;
    p.group_k = a->group_k;
    p.out_dtype = a->out_dtype;
    p.n_strips = l.n_strips;
    p.out_vec = w6::aligned16(a->out) && a->out_row_stride % 8 == 0 && a->out_batch_stride % 8 == 0;
    const hipStream_t s = static_cast<hipStream_t>(stream);
    if (const int bad = a->a_dtype == W6A16_IN_F16 ? w6::launch_matmul<w6::ActF16>(p, a, l, s)
                                                   : w6::launch_matmul<w6::ActBF16>(p, a, l, s))
        return bad;
    return static_cast<int>(hipGetLastError());
}

int w6a16_dequantize_packed(const void* packed, const uint16_t* packed_scales, void* w, int32_t B, int32_t K,
                            int32_t N, int32_t group_k, int64_t w_batch_stride, int32_t out_dtype, void* stream) {
    if (!packed || !packed_scales || !w) return WKV7_ERR_NULL;
    if (B < 1 || N < 16 || N % 16 || K < 64 || K % 64 || group_k < 64 || group_k % 64 || K % group_k)
        return WKV7_ERR_SHAPE;
    if (out_dtype != W6A16_OUT_BF16 && out_dtype != W6A16_OUT_F16 && out_dtype != W6A16_OUT_F32) return WKV7_ERR_ARG;
    if (!w6::aligned16(packed) || !w6::aligned16(packed_scales)) return WKV7_ERR_ALIGN;
    if (B > 65535) return WKV7_ERR_SHAPE;
    const int strips = (N + w6::kTileN - 1) / w6::kTileN;
    const dim3 grid((unsigned)(((int64_t)strips * (K / 64) + 3) / 4), B);
    const bool vec = w6::aligned16(w) && w_batch_stride % 8 == 0;  // fp32: 8 elements are two 16-byte stores
    const hipStream_t s = static_cast<hipStream_t>(stream);
    const uint8_t* pk = static_cast<const uint8_t*>(packed);
    if (out_dtype == W6A16_OUT_F32)
        hipLaunchKernelGGL(w6::w6a16_dequant_packed_kernel<float>, grid, dim3(256), 0, s, pk, packed_scales,
                           static_cast<float*>(w), K, N, group_k, strips, w_batch_stride, vec);
    else if (out_dtype == W6A16_OUT_F16)
        hipLaunchKernelGGL(w6::w6a16_dequant_packed_kernel<_Float16>, grid, dim3(256), 0, s, pk, packed_scales,
                           static_cast<_Float16*>(w), K, N, group_k, strips, w_batch_stride, vec);
    else
        hipLaunchKernelGGL(w6::w6a16_dequant_packed_kernel<__bf16>, grid, dim3(256), 0, s, pk, packed_scales,
                           static_cast<__bf16*>(w), K, N, group_k, strips, w_batch_stride, vec);
    return static_cast<int>(hipGetLastError());
}

int w6a16_packed_size(int32_t B, int32_t K, int32_t N, int32_t group_k, size_t* weight_bytes, size_t* scale_bytes) {
    if (!weight_bytes || !scale_bytes) return WKV7_ERR_NULL;
    if (B < 1 || N < 16 || N % 16 || K < 64 || K % 64 || group_k < 64 || group_k % 64 || K % group_k)
        return WKV7_ERR_SHAPE;
    const size_t strips = (N + w6::kTileN - 1) / w6::kTileN;
    *weight_bytes = (size_t)B * strips * (K / 64) * w6::kPackBytes;
    *scale_bytes = (size_t)B * strips * (K / group_k) * w6::kTileN * 2;
    return WKV7_OK;
}

int w6a16_pack(const uint8_t* lo, const uint8_t* hi, const uint16_t* scales, int32_t B, int32_t K, int32_t N,
               int32_t group_k, int64_t lo_batch_stride, int64_t hi_batch_stride, int64_t scales_batch_stride,
               void* packed, uint16_t* packed_scales, void* stream) {
    size_t wb = 0, sb = 0;
    const int rc = w6a16_packed_size(B, K, N, group_k, &wb, &sb);
    if (rc != WKV7_OK) return rc;
    if (!lo || !hi || !scales || !packed || !packed_scales) return WKV7_ERR_NULL;
    if (!w6::aligned16(packed) || !w6::aligned16(packed_scales)) return WKV7_ERR_ALIGN;
    if (B > 65535) return WKV7_ERR_SHAPE;
    const int strips = (N + w6::kTileN - 1) / w6::kTileN, groups = K / group_k;
    const hipStream_t s = static_cast<hipStream_t>(stream);
    const int64_t nw = (int64_t)strips * (K / 64) * 64, ns = (int64_t)strips * groups * 16;
    hipLaunchKernelGGL(w6::w6a16_pack_kernel, dim3((unsigned)((nw + 255) / 256), B), dim3(256), 0, s, lo, hi,
                       static_cast<uint8_t*>(packed), K, N, strips, lo_batch_stride, hi_batch_stride);
    hipLaunchKernelGGL(w6::w6a16_pack_scales_kernel, dim3((unsigned)((ns + 255) / 256), B), dim3(256), 0, s, scales,
                       packed_scales, groups, N, strips, scales_batch_stride);
    return static_cast<int>(hipGetLastError());
}

int w6a16_dequantize(const uint8_t* lo, const uint8_t* hi, const uint16_t* scales, void* w, int32_t B, int32_t K,
                     int32_t N, int32_t group_k, int64_t lo_batch_stride, int64_t hi_batch_stride,
                     int64_t scales_batch_stride, int64_t w_batch_stride, int32_t out_dtype, void* stream) {
    if (!lo || !hi || !scales || !w) return WKV7_ERR_NULL;
    if (B < 1 || N < 16 || N % 16 || K < 64 || K % 64 || group_k < 64 || group_k % 64 || K % group_k)
        return WKV7_ERR_SHAPE;
    if (out_dtype != W6A16_OUT_BF16 && out_dtype != W6A16_OUT_F16 && out_dtype != W6A16_OUT_F32) return WKV7_ERR_ARG;
    if (!w6::aligned16(lo) || !w6::aligned16(hi) || !w6::aligned16(scales) || !w6::aligned16(w) ||
        lo_batch_stride % 16 || hi_batch_stride % 16 || scales_batch_stride % 8 || w_batch_stride % 8)
        return WKV7_ERR_ALIGN;
    if (K / 2 > 65535 || B > 65535) return WKV7_ERR_SHAPE;  // grid y and z
    const dim3 grid((N / 8 + 255) / 256, K / 16, B);
    const hipStream_t s = static_cast<hipStream_t>(stream);
    if (out_dtype == W6A16_OUT_F32)
        hipLaunchKernelGGL(w6::w6a16_dequant_kernel<float>, grid, dim3(256), 0, s, lo, hi, scales,
                           static_cast<float*>(w), K, N, group_k, lo_batch_stride, hi_batch_stride,
                           scales_batch_stride, w_batch_stride);
    else if (out_dtype == W6A16_OUT_F16)
        hipLaunchKernelGGL(w6::w6a16_dequant_kernel<_Float16>, grid, dim3(256), 0, s, lo, hi, scales,
                           static_cast<_Float16*>(w), K, N, group_k, lo_batch_stride, hi_batch_stride,
                           scales_batch_stride, w_batch_stride);
    else
        hipLaunchKernelGGL(w6::w6a16_dequant_kernel<__bf16>, grid, dim3(256), 0, s, lo, hi, scales,
                           static_cast<__bf16*>(w), K, N, group_k, lo_batch_stride, hi_batch_stride,
                           scales_batch_stride, w_batch_stride);
    return static_cast<int>(hipGetLastError());
}

}  // extern "C"
