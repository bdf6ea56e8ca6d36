// SGEMM stage 10: fp32 GEMM from three bf16 matrix-core products.
//
// Numerics. Each fp32 operand x is split as hi = bf16(x), lo = bf16(x - hi)
// (both round-to-nearest-even; x - hi is exact in fp32), so x = hi + lo up to
// 2^-16 |x|. The product a*b is taken as hi_a*hi_b + hi_a*lo_b + lo_a*hi_b,
// dropping lo_a*lo_b (<= 2^-16 |ab|). Each bf16 x bf16 product is exact in
// fp32 and accumulation is fp32 on v_mfma_f32_32x32x16_bf16, so the result is
// the split's exact value up to fp32 summation of 3K terms: a few 2^-17 per
// product against the exact product, an order of magnitude better than the
// TF32 stage it stands in for (src/kernels/k09_tensorcore.cu:119-128 rounds
// to 10 mantissa bits). Three bf16 MFMAs (8 passes each) cost 96 cycles per
// 32x32x16 step against 512 for the fp32 MFMA, so the ceiling is a third of
// the bf16 peak: 833 TFLOP/s of fp32-equivalent work.
//
// MFMA operand layout (v_mfma_f32_32x32x16_bf16): lane l supplies 8
// consecutive-k bf16 of row (A) or column (B) l % 32, k = 8 * (l / 32) + 0..7;
// the D layout matches v_mfma_f32_32x32x2_f32.
//
// Tiles. 256x256 (8 waves of 128x64), 128x256 (8 waves of 64x64), 128x128
// (4 waves of 64x64) and 64x64 (4 waves of 32x32) outputs, K in stages of 32
// (two 16-k MFMA steps); for few tiles, workgroups whose wave groups each take
// every S-th stage (bf16x3_ks_k: 128x64, 64x64 and 32x32 outputs); and a
// split of K into ranges whose fp32 partials one reduce adds in range order
// (deterministic). A planner picks tile and split per shape, as gemm() does
// for the fp32 MFMA path: the 256x256 tile alone leaves most CUs idle below
// N = 4096 (16 workgroups at N = 1024).
//
// LDS: per stage four bf16 planes (A hi, A lo, B hi, B lo), each stored
// [row][k] with k contiguous (row = m for A, n for B), so every fragment is
// one 128-bit read. Rows are 64 bytes with their 16-byte chunks XOR-swizzled
// by row (lds_off), so neither the fragment reads nor the staging stores
// conflict on banks. How an operand gets there (OpStage) depends on whether
// k or m/n is contiguous in memory.
//
// Schedule: double-buffered LDS stages with register prefetch; one barrier
// per stage. While a stage is consumed, the next one is split and stored from
// registers and the global loads for the stage after it are issued. In the
// interior steady state (step0_fused) the split and its LDS stores are cut
// into pieces (one float4 chunk, or one column of a 4 x 4 block) placed
// between the first 16-k step's MFMAs behind scheduling fences, and each
// piece's registers are refilled by the next loads as soon as it is stored.
// Left to the compiler, the first step's MFMAs went out back to back and the
// conversion ran after them, so the two waves of a SIMD, kept in phase by the
// barrier, converted at the same time while the matrix core idled. The fenced
// order is 1-5% faster on the GPT-2 shapes and 2% at N = 4096, bit-identical.
//
// What bounds it. With the device full of 128- or 256-wide tiles: power. On
// N(0, 1) data at N = 4096 the matrix cores are busy 71% of a launch's cycles
// while the clock falls to 1.74 GHz; zeros run the same cycles at 2.44 GHz (315
// and 221 us), so what counts is the energy of everything around the MFMAs.
// Taking instructions out of the staging (split4 on pairs, loads without
// address arithmetic, two stages per loop turn) gave 4-5% on 256 x 256 and
// 6-9% on 128-wide tiles (per 32-k stage and CU: 2.50 -> 2.37 us, 1.42 ->
// 1.33, 1.62 -> 1.48 for two 128 x 128). With few tiles: the latency chain of
// a stage (0.4 us for a lone 64 x 64 workgroup against 0.09 of MFMAs), which
// more resident workgroups overlap and a deeper prefetch does not shorten.
#include <math.h>
#include <stdio.h>
#include <stdlib.h>

#include <algorithm>
#include <map>
#include <mutex>
#include <optional>
#include <tuple>
#include <type_traits>

#include "common.hpp"
#include "gemm_fused.hpp"
#include "mfma_gemm.hpp"
#include "../../include/kernels.h"
#include "launch.hpp"
#include "workspace.hpp"

namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
using bmb::f32x16;

constexpr int BK = 32;   // k per LDS stage: two 16-k MFMA steps
constexpr int LDK = BK;  // bf16 per LDS row (64 bytes, no padding: see lds_off)

template <int BM_, int BN_, int WAVES_M_, int WAVES_N_>
struct B3Tile {
    static constexpr int BM = BM_, BN = BN_, WAVES_M = WAVES_M_, WAVES_N = WAVES_N_;
    static constexpr int NT = 64 * WAVES_M * WAVES_N;
    static constexpr int WM = BM / WAVES_M, WN = BN / WAVES_N;
    static constexpr int FM = WM / 32, FN = WN / 32;
    static constexpr int A_PLANE = BM * LDK, B_PLANE = BN * LDK;  // bf16 elements
    static constexpr int STAGE = 2 * A_PLANE + 2 * B_PLANE;
    static constexpr size_t SMEM_BYTES = 2 * (size_t)STAGE * sizeof(__bf16);
    static_assert(WM % 32 == 0 && WN % 32 == 0, "wave tile is whole 32x32 blocks");
};

using TileL = B3Tile<256, 256, 2, 4>;
using TileM = B3Tile<128, 128, 2, 2>;
using TileS = B3Tile<64, 64, 2, 2>;
using TileT = B3Tile<128, 256, 2, 4>;
using TileH = B3Tile<128, 64, 2, 2>;  // k-sliced kernels only
using TileXS = B3Tile<32, 32, 1, 1>;  // one wave (k-sliced kernels only)

// Offset (in bf16) of element k (a multiple of 4) of LDS row `row`. Rows are
// 64 bytes (four 16-byte chunks); row r is stored in slot p = r ^ ((r >> 2)
// & 1) (rows swap pairwise in every other group of four), and chunk k / 8 of
// it at position chunk ^ ((r >> 3) & 3).
//
// gfx950's LDS has 64 four-byte banks. Measured with SQ_LDS_BANK_CONFLICT
// on single-pattern probes:
// - A 128-bit read is served in four cycles of 16 lanes each, and the
//   groups are not consecutive lanes: {0-3, 12-15, 20-27}, {4-11, 16-19,
//   28-31} and the same two shapes over lanes 32-63. A group is conflict-free
//   when its 16 addresses fall in 16 distinct 16-byte slots modulo 256 bytes.
//   A fragment read covers rows 0-31 of a 32-row block at one chunk. The
//   rows of the first group, 0-3, 12-15, 20-23 and 24-27, occupy four slot
//   pairs (row slot mod 4) and take the XORs 0, 1, 2, 3; so do those of the
//   second group.
// - A 64-bit write is served in groups of 16 consecutive lanes. A stores
//   (two rows x eight 8-byte units per 16 lanes) and the B planes' transposed
//   stores (rows 4m + c of eight consecutive column blocks m, two 8-byte
//   units each) land in 16 distinct 8-byte slots under this mapping.
// The bf16x3 kernel reads no conflict cycle at all (N = 4096), down from
// 2.5e7 per launch for the XOR ((r >> 2) ^ (r >> 4)) & 3, which assumed 16
// consecutive lanes per read cycle. A padded 80-byte row made the transposed
// stores 16-way conflicted.
__device__ __forceinline__ int lds_off(int row, int k) {
    const int p = row ^ ((row >> 2) & 1);
    return p * LDK + 8 * ((k >> 3) ^ ((row >> 3) & 3)) + (k & 7);
}

// The largest float that rounds to a finite bfloat16 (0x7F7F7FFF): above it
// round-to-nearest gives infinity, although x is finite.
constexpr float BF16_FINITE_MAX = 0x1.fefffep+127f;

// x -> (hi, lo) = (bf16(c), bf16(x - hi)) for four values, with c = x clamped
// to +-BF16_FINITE_MAX (one v_med3_f32). For |x| <= BF16_FINITE_MAX, c = x.
// Above it (finite x up to FLT_MAX, or +-inf) hi is bf16's largest finite
// value with x's sign and x - hi is exact (Sterbenz) or +-inf, so a huge
// finite x still splits exactly instead of into (inf, -inf), and an infinite
// x gives (+-3.39e38, +-inf), whose products with a nonzero b are +-inf and
// with b = 0 NaN, as in fp32. NaN stays NaN in lo.
//
// Written on pairs: one v_cvt_pk_bf16_f32 rounds two values, and its result is
// widened again with a shift and a mask (12 instructions per four values
// beside the clamps; asked for one value at a time the compiler converted
// every hi twice, 20 in all).
__device__ __forceinline__ void split4(const float (&x)[4], bf16x4 &hi, bf16x4 &lo) {
#pragma unroll
    for (int i = 0; i < 4; i += 2) {
        const f32x2 c = {__builtin_amdgcn_fmed3f(x[i], -BF16_FINITE_MAX, BF16_FINITE_MAX),
                         __builtin_amdgcn_fmed3f(x[i + 1], -BF16_FINITE_MAX, BF16_FINITE_MAX)};
        const bf16x2 h = __builtin_convertvector(c, bf16x2);
        const unsigned u = __builtin_bit_cast(unsigned, h);
        const f32x2 r = {x[i] - __builtin_bit_cast(float, u << 16),
                         x[i + 1] - __builtin_bit_cast(float, u & 0xffff0000u)};
        const bf16x2 l = __builtin_convertvector(r, bf16x2);
        hi[i] = h[0];
        hi[i + 1] = h[1];
        lo[i] = l[0];
        lo[i + 1] = l[1];
    }
}

// f(integral_constant<int, i>) for i = I .. N - 1.
template <int I, int N, class F>
__device__ __forceinline__ void static_for(F &&f) {
    if constexpr (I < N) {
        f(std::integral_constant<int, I>{});
        static_for<I + 1, N>(f);
    }
}

// A buffer descriptor over an operand from p on (uniform). The staging loads
// go through it because they then take a uniform base that the scalar unit
// advances per stage and a loop-invariant 32-bit offset per lane; with plain
// pointers every load cost two 64-bit vector adds per stage. The loads stay
// inside the operand by their offsets, so the descriptor's size does not
// bound them.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t operand(const float *p) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(p), 0, 0xffffffff, 0x00027000);
}

// Staging of one operand's tile per stage: ROWS rows (m of A, n of B) x BK k,
// into a hi and a lo plane. KCONT: k is the contiguous axis of the stored
// operand (A not transposed, B transposed): 128-bit loads of four k, split,
// one 64-bit store per plane. Otherwise rows are contiguous (A transposed, B
// not): blocks of 4 k x W rows (a wave covers 32 consecutive blocks of two k
// rows), transposed in registers, one 64-bit store of four k per row and
// plane. W is 4, or 2 where a tile has fewer 4 x 4 blocks than the workgroup
// has lanes (64 rows on 256 lanes; see also Bf16x3Gemm::PAIR).
//
// IN (interior): all ROWS rows lie inside the operand. An edge tile loads
// from clamped rows instead of checking bounds: LDS rows past the operand's
// last one then hold copies of other rows, which only reach outputs that are
// not stored. (A block that straddles the last row is loaded from further
// back and shifted into place when it is split.) So edge tiles run the same
// branch-free loop as interior ones; only a last stage with fewer than BK k
// (load_tail) fills with zeros. Every path loads whole vectors and selects
// from them afterwards: where a branch joined vectors loaded at once with
// vectors loaded element by element, the compiler (ROCm 7.2) reused registers
// of the former that were still live. That needs stored rows of at least four
// elements and byte offsets below 2^32.
//
// SHORT: stored rows may be shorter (a K below 4 with k contiguous, an M or N
// below 4 otherwise), down to four elements in the whole operand. A vector then
// runs on into the next stored row, whose elements are masked (k) or only reach
// outputs that are not stored (rows); near the operand's end it is loaded from
// further back and shifted into place (load_tail, which also takes a whole
// stage with fewer than SHORT_K k behind its first). SINGLE: every element is
// loaded by itself.
enum Stage { VECTOR, SHORT, SINGLE };
constexpr int SHORT_K = BK + 3;  // loads of a whole stage stay inside the operand
template <int ROWS, int NT, bool KCONT, bool IN, Stage MODE = VECTOR>
struct OpStage {
    static constexpr int CH = ROWS * BK / 4 / NT;  // KCONT: chunks per lane
    static constexpr int W = !KCONT && ROWS * BK / 16 < NT ? 2 : 4;
    static constexpr int BLK = BK * ROWS / (4 * W);    // otherwise: blocks per stage
    static constexpr int PER_T = (BLK + NT - 1) / NT;  // blocks per lane
    static constexpr int NLD = KCONT ? CH : 4 * PER_T;
    static_assert(!KCONT || (ROWS * BK / 4) % NT == 0, "staging splits evenly over the lanes");
    static_assert(KCONT || BLK % NT == 0 || BLK < NT, "blocks split evenly over the lanes");
    struct Vec {
        float f[W];
    };
    Vec v[NLD];
    // Byte offsets of this lane's loads from the stage's first element (row
    // row0(), k 0), and how many rows before its place each block is loaded:
    // loop-invariant.
    unsigned o[NLD];
    int shift[KCONT || IN || MODE != VECTOR ? 1 : PER_T];

    __device__ static __forceinline__ bool skip(int j, int tid) {
        return !KCONT && BLK % NT != 0 && tid + j * NT >= BLK;
    }
    // Chunk e (KCONT): row r, k c..c+3.
    __device__ static __forceinline__ void chunk(int e, int &r, int &c) {
        r = e / (BK / 4);
        c = (e % (BK / 4)) * 4;
    }
    // Block e: k rows 4kb..4kb+3, rows W*m..W*m+W-1. Neighbouring lanes take
    // the two halves of a 16-byte k chunk (kb even, odd) of one row block.
    __device__ static __forceinline__ void block(int e, int &kb, int &row) {
        const int m = (e >> 1) % (ROWS / W);
        kb = 2 * ((e >> 1) / (ROWS / W)) + (e & 1);
        row = W * m;
    }
    // The row that offsets count from: the tile's first, or 0 where a clamped
    // block may start before the tile.
    __device__ static __forceinline__ int row0(int r0) {
        return (IN && MODE != SHORT) || KCONT ? r0 : 0;
    }
    // R rows in all, ld: the stored row stride, r0: the tile's first row.
    __device__ __forceinline__ void setup(int R, int ld, int r0, int tid) {
        if constexpr (KCONT) {
#pragma unroll
            for (int i = 0; i < NLD; ++i) {
                int r, c;
                chunk(tid + i * NT, r, c);
                if (!IN) r = min(r, R - 1 - r0);
                o[i] = 4u * ((unsigned)r * (unsigned)ld + (unsigned)c);
            }
        } else {
#pragma unroll
            for (int j = 0; j < PER_T; ++j) {
                int kb, rb;
                block(min(tid + j * NT, BLK - 1), kb, rb);
                if (MODE == SHORT) {
                    rb = min(rb, R - 1 - r0);
                } else if (!IN) {
                    shift[j] = rb - min(rb, R - r0 - W);
                    rb -= shift[j];
                }
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    o[4 * j + i] = 4u * ((unsigned)(4 * kb + i) * (unsigned)ld +
                                         (unsigned)(rb + r0 - row0(r0)));
            }
        }
    }
    __device__ static __forceinline__ Vec ldv(__amdgpu_buffer_rsrc_t p, unsigned off) {
        Vec x;
        if constexpr (W == 4) {
            const auto t = __builtin_amdgcn_raw_buffer_load_b128(p, (int)off, 0, 0);
            __builtin_memcpy(&x, &t, sizeof(x));
        } else {
            const auto t = __builtin_amdgcn_raw_buffer_load_b64(p, (int)off, 0, 0);
            __builtin_memcpy(&x, &t, sizeof(x));
        }
        return x;
    }
    // Elements n, n + 1, ... of x in its first places (n < W; what follows the
    // last element is unspecified).
    __device__ static __forceinline__ Vec shifted(const Vec &x, int n) {
        Vec y;
#pragma unroll
        for (int c = 0; c < W; ++c) {
            y.f[c] = x.f[c];
#pragma unroll
            for (int q = c + 1; q < W; ++q) y.f[c] = n == q - c ? x.f[q] : y.f[c];
        }
        return y;
    }
    __device__ __forceinline__ void load(__amdgpu_buffer_rsrc_t p, int tid) {
#pragma unroll
        for (int i = 0; i < NLD; ++i)
            if (!skip(i / 4, tid)) v[i] = ldv(p, o[i]);
    }
    // SINGLE: every element (row, k) by itself; rows past the last of R repeat it,
    // k from rem (> 0) on are zeros. p: the stage's (row 0 of the operand,
    // k 0) element.
    __device__ __forceinline__ void load_single(const float *p, int R, int ld, int r0, int rem,
                                                int tid) {
        const auto at = [&](int r, int c) {
            const size_t row = min(r0 + r, R - 1), k = min(c, rem - 1);
            const float x = p[KCONT ? row * ld + k : k * ld + row];
            return c < rem ? x : 0.0f;
        };
#pragma unroll
        for (int i = 0; i < NLD; ++i) {
            int r, c;
            if (KCONT) {
                chunk(tid + i * NT, r, c);
            } else {
                block(tid + i / 4 * NT, c, r);
                c = 4 * c + i % 4;
            }
#pragma unroll
            for (int e = 0; e < W; ++e) v[i].f[e] = KCONT ? at(r, c + e) : at(r + e, c);
        }
    }
    // A stage of which only the first rem (0 < rem < BK) k exist; the others
    // become zero. p: the descriptor of the stage's base (KCONT: of the four
    // elements before it; a chunk with fewer than four k is loaded as the
    // stage's last four and shifted).
    // SHORT: p is the descriptor of the four elements before the stage's base,
    // end the stored elements from that base to the operand's (or K range's)
    // last one, and rem may be any positive number.
    __device__ __forceinline__ void load_tail(__amdgpu_buffer_rsrc_t p, int ld, int rem, int tid,
                                              long long end = 0) {
        const unsigned last = (unsigned)min(4LL * (end - W + 4), 0xffffffffLL);
#pragma unroll
        for (int i = 0; i < NLD; ++i) {
            if (skip(i / 4, tid)) continue;
            if constexpr (MODE == SHORT) {
                int k, row;
                if (KCONT) {
                    chunk(tid + i * NT, row, k);
                } else {
                    block(tid + i / 4 * NT, k, row);
                    k = 4 * k + i % 4;
                }
                const unsigned at = min(o[i] + 16u, last);
                v[i] = shifted(ldv(p, at), (int)((o[i] + 16u - at) / 4u));
#pragma unroll
                for (int e = 0; e < W; ++e)
                    v[i].f[e] = k + (KCONT ? e : 0) < rem ? v[i].f[e] : 0.0f;
            } else if constexpr (KCONT) {
                int r, c;
                chunk(tid + i * NT, r, c);
                const int n = c - min(c, rem - 4);
                v[i] = shifted(ldv(p, o[i] + 16u - 4u * (unsigned)n), n);
#pragma unroll
                for (int e = 0; e < 4; ++e) v[i].f[e] = c + e < rem ? v[i].f[e] : 0.0f;
            } else {
                int kb, row;
                block(tid + i / 4 * NT, kb, row);
                const int k = 4 * kb + i % 4;
                v[i] = ldv(p, o[i] - 4u * (unsigned)(k - min(k, rem - 1)) * (unsigned)ld);
#pragma unroll
                for (int c = 0; c < W; ++c) v[i].f[c] = k < rem ? v[i].f[c] : 0.0f;
            }
        }
    }
    __device__ __forceinline__ void zero() {
#pragma unroll
        for (int i = 0; i < NLD; ++i) v[i] = Vec{};
    }
    // The split and its LDS stores in pieces: chunk P (KCONT), or row P % W of
    // block P / W.
    static constexpr int NPIECE = KCONT ? NLD : W * PER_T;
    template <int P>
    __device__ __forceinline__ void store_piece(__bf16 *hi, __bf16 *lo, int tid) const {
        bf16x4 h, l;
        if constexpr (KCONT) {
            int r, c;
            chunk(tid + P * NT, r, c);
            split4(v[P].f, h, l);
            *reinterpret_cast<bf16x4 *>(hi + lds_off(r, c)) = h;
            *reinterpret_cast<bf16x4 *>(lo + lds_off(r, c)) = l;
        } else {
            constexpr int j = P / W, c = P % W;
            if (skip(j, tid)) return;
            int kb, row;
            block(tid + j * NT, kb, row);
            float x[4];
#pragma unroll
            for (int i = 0; i < 4; ++i)
                x[i] = IN || MODE != VECTOR ? v[4 * j + i].f[c]
                                            : shifted(v[4 * j + i], shift[j]).f[c];
            split4(x, h, l);
            *reinterpret_cast<bf16x4 *>(hi + lds_off(row + c, 4 * kb)) = h;
            *reinterpret_cast<bf16x4 *>(lo + lds_off(row + c, 4 * kb)) = l;
        }
    }
    __device__ __forceinline__ void store(__bf16 *hi, __bf16 *lo, int tid) const {
        static_for<0, NPIECE>([&](auto pc) { store_piece<decltype(pc)::value>(hi, lo, tid); });
    }
    // The loads into the registers that piece P was the last to read.
    template <int P>
    __device__ __forceinline__ void load_after_piece(__amdgpu_buffer_rsrc_t p, int tid) {
        if constexpr (KCONT) {
            v[P] = ldv(p, o[P]);
        } else if constexpr (P % W == W - 1) {
            constexpr int j = P / W;
            if (skip(j, tid)) return;
#pragma unroll
            for (int i = 0; i < 4; ++i) v[4 * j + i] = ldv(p, o[4 * j + i]);
        }
    }
};

// op(A) is M x K, op(B) K x N; stored A is M x K (lda = K) or, TA, K x M
// (lda = M); stored B is K x N (ldb = N) or, TB, N x K (ldb = K). C is M x N.
template <class Tl, bool TA, bool TB>
struct Bf16x3Gemm {
    static constexpr int BM = Tl::BM, BN = Tl::BN, NT = Tl::NT;
    static constexpr int FM = Tl::FM, FN = Tl::FN;
    // PAIR: both operands are staged in 4 x 4 blocks and each has half as many
    // as the workgroup has lanes (64 x 64 tiles of A^T B): the lower half of
    // the workgroup then stages A and the upper half B, every lane one block
    // with 128-bit loads (blocks half as wide, on all lanes for both
    // operands, halve the bytes per load).
    static constexpr bool PAIR = TA && !TB && BM == BN && BM * BK / 16 * 2 == NT;
    template <bool IN, Stage MODE>
    using StageA = OpStage<BM, PAIR ? NT / 2 : NT, !TA, IN, MODE>;
    template <bool IN, Stage MODE>
    using StageB = OpStage<BN, PAIR ? NT / 2 : NT, TB, IN, MODE>;

    // One 16-k step of MFMAs on stage `st`: for every 32 x 32 block,
    // acc += lo_a hi_b, then hi_a lo_b, then hi_a hi_b (small terms first).
    __device__ static __forceinline__ void step(const __bf16 *st, int kk, int wm, int wn, int lane,
                                                f32x16 (&acc)[FM][FN]) {
        const int l32 = lane & 31, koff = kk * 16 + 8 * (lane >> 5);
        bf16x8 ah[FM], al[FM], bh[FN], bl[FN];
#pragma unroll
        for (int fi = 0; fi < FM; ++fi) {
            const int off = lds_off(wm + fi * 32 + l32, koff);
            ah[fi] = *reinterpret_cast<const bf16x8 *>(st + off);
            al[fi] = *reinterpret_cast<const bf16x8 *>(st + Tl::A_PLANE + off);
        }
#pragma unroll
        for (int fn = 0; fn < FN; ++fn) {
            const int off = 2 * Tl::A_PLANE + lds_off(wn + fn * 32 + l32, koff);
            bh[fn] = *reinterpret_cast<const bf16x8 *>(st + off);
            bl[fn] = *reinterpret_cast<const bf16x8 *>(st + Tl::B_PLANE + off);
        }
#pragma unroll
        for (int fi = 0; fi < FM; ++fi)
#pragma unroll
            for (int fn = 0; fn < FN; ++fn) {
                acc[fi][fn] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(al[fi], bh[fn], acc[fi][fn], 0, 0, 0);
                acc[fi][fn] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ah[fi], bl[fn], acc[fi][fn], 0, 0, 0);
                acc[fi][fn] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ah[fi], bh[fn], acc[fi][fn], 0, 0, 0);
            }
    }

    // MFMA MI of a step in round-robin order over the accumulators: every
    // lo_a hi_b term, then every hi_a lo_b, then every hi_a hi_b. Each
    // accumulator takes its three terms in step()'s order.
    template <int MI>
    __device__ static __forceinline__ void mfma_rr(const bf16x8 (&ah)[FM], const bf16x8 (&al)[FM],
                                                   const bf16x8 (&bh)[FN], const bf16x8 (&bl)[FN],
                                                   f32x16 (&acc)[FM][FN]) {
        constexpr int round = MI / (FM * FN), idx = MI % (FM * FN), fi = idx / FN, fn = idx % FN;
        if constexpr (round == 0)
            acc[fi][fn] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(al[fi], bh[fn], acc[fi][fn], 0, 0, 0);
        else if constexpr (round == 1)
            acc[fi][fn] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ah[fi], bl[fn], acc[fi][fn], 0, 0, 0);
        else
            acc[fi][fn] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ah[fi], bh[fn], acc[fi][fn], 0, 0, 0);
    }

    // Step 0 of stage st with the next stage's split and LDS stores (into nx)
    // between its MFMAs: piece P follows MFMAs [P NM / NP, (P + 1) NM / NP)
    // behind a scheduling fence, and is followed by the loads that refill its
    // registers. piece(P): store and refill.
    template <int NP, class F>
    __device__ static __forceinline__ void step0_fused(const __bf16 *st, int wm, int wn, int lane,
                                                       f32x16 (&acc)[FM][FN], F &&piece) {
        const int l32 = lane & 31, koff = 8 * (lane >> 5);
        bf16x8 ah[FM], al[FM], bh[FN], bl[FN];
#pragma unroll
        for (int fi = 0; fi < FM; ++fi) {
            const int off = lds_off(wm + fi * 32 + l32, koff);
            ah[fi] = *reinterpret_cast<const bf16x8 *>(st + off);
            al[fi] = *reinterpret_cast<const bf16x8 *>(st + Tl::A_PLANE + off);
        }
#pragma unroll
        for (int fn = 0; fn < FN; ++fn) {
            const int off = 2 * Tl::A_PLANE + lds_off(wn + fn * 32 + l32, koff);
            bh[fn] = *reinterpret_cast<const bf16x8 *>(st + off);
            bl[fn] = *reinterpret_cast<const bf16x8 *>(st + Tl::B_PLANE + off);
        }
        constexpr int NM = FM * FN * 3;
        static_for<0, NP>([&](auto pc) {
            constexpr int P = decltype(pc)::value;
            static_for<P * NM / NP, (P + 1) * NM / NP>([&](auto mc) {
                mfma_rr<decltype(mc)::value>(ah, al, bh, bl, acc);
            });
            piece(pc);
            __builtin_amdgcn_sched_barrier(0);
        });
    }

    // One output tile over k in [0, K) (A, B positioned at that range's
    // start). INTERIOR: the tile lies inside M x N. TAIL: K need not be a
    // whole number of stages (a last stage of fewer k is filled with zeros).
    // EPI: what the epilogue stores (bmb::Epi; EPI_PARTIAL: the raw
    // sums). C's rows (and those of ep.act, ep.pre) are ldc floats apart.
    // KS > 1: the workgroup is KS k-slices of NT lanes (bf16x3_ks_k); this
    // slice's stages are at smem, K is its range's length (<= 0: none of its
    // stages holds data) and every slice runs kloop stages, so that all of
    // them meet at the same barriers. The slices' sums are then added in LDS,
    // in slice order, and slice 0 runs the epilogue.
    // MODE: how both operands are staged (OpStage; TAIL unless VECTOR).
    template <bool INTERIOR, int EPI, bool TAIL, int KS = 1, Stage MODE = VECTOR>
    __device__ static __forceinline__ void run(int M, int N, int K, int lda, int ldb, float alpha,
                                               const float *__restrict__ A,
                                               const float *__restrict__ B, float beta, float *C,
                                               int ldc, int m0, int n0, __bf16 *smem,
                                               const bmb::EpiArgs &ep, int kloop = 0) {
        const int tid = KS > 1 ? (int)(threadIdx.x % NT) : (int)threadIdx.x;
        const int wave = tid >> 6, lane = tid & 63;
        const int wm = (wave / Tl::WAVES_N) * Tl::WM, wn = (wave % Tl::WAVES_N) * Tl::WN;

        f32x16 acc[FM][FN];
#pragma unroll
        for (int fi = 0; fi < FM; ++fi)
#pragma unroll
            for (int fn = 0; fn < FN; ++fn)
#pragma unroll
                for (int r = 0; r < 16; ++r) acc[fi][fn][r] = 0.0f;

        const int nkt = KS > 1 ? kloop : (K + BK - 1) / BK;
        using SA = StageA<INTERIOR, MODE>;
        using SB = StageB<INTERIOR, MODE>;
        SA ga;
        SB gb;
        // PAIR: this half's operand in ga (uniform over a wave).
        const bool up = PAIR && __builtin_amdgcn_readfirstlane(tid) >= NT / 2;
        const int stid = PAIR ? tid % (NT / 2) : tid;
        const int lda1 = up ? ldb : lda, a0 = up ? n0 : m0;
        ga.setup(up ? N : M, lda1, a0, stid);
        if (!PAIR) gb.setup(N, ldb, n0, tid);
        // Stage kt's first elements (uniform).
        auto a_at = [&](int kt) {
            const size_t r = ga.row0(a0), k = (size_t)kt * BK;
            return (up ? B : A) + (TA ? k * lda1 + r : r * lda1 + k);
        };
        auto b_at = [&](int kt) {
            const size_t r = gb.row0(n0), k = (size_t)kt * BK;
            return TB ? B + r * ldb + k : B + k * ldb + r;
        };
        auto load = [&](int kt) {
            const int rem = K - kt * BK;
            if (MODE == SINGLE) {
                const size_t k = (size_t)kt * BK;
                ga.load_single((up ? B : A) + (TA ? k * lda1 : k), up ? N : M, lda1, a0, rem,
                               stid);
                if (!PAIR) gb.load_single(B + (TB ? k : k * ldb), N, ldb, n0, rem, tid);
            } else if (!TAIL || rem >= (MODE == SHORT ? SHORT_K : BK)) {
                ga.load(operand(a_at(kt)), stid);
                if (!PAIR) gb.load(operand(b_at(kt)), tid);
            } else if (MODE == SHORT && rem > 0) {
                // Elements from each stage's base to the end of its operand's K
                // range: whole rows of k from row0 on, or whole k of rows.
                const auto left = [&](bool kcont, int R, int ld, int r) {
                    return kcont ? (R - 1LL - r) * ld + rem : (rem - 1LL) * ld + R;
                };
                ga.load_tail(operand(a_at(kt) - 4), lda1, rem, stid,
                             left(!TA, up ? N : M, lda1, ga.row0(a0)));
                if (!PAIR)
                    gb.load_tail(operand(b_at(kt) - 4), ldb, rem, tid, left(TB, N, ldb, gb.row0(n0)));
            } else if (rem > 0) {
                ga.load_tail(operand(a_at(kt) - (TA ? 0 : 4)), lda1, rem, stid);
                if (!PAIR) gb.load_tail(operand(b_at(kt) - (TB ? 4 : 0)), ldb, rem, tid);
            } else {
                ga.zero();
                if (!PAIR) gb.zero();
            }
        };
        auto store = [&](__bf16 *st) {
            __bf16 *sa = st + (up ? 2 * Tl::A_PLANE : 0);
            ga.store(sa, sa + Tl::A_PLANE, stid);
            if (!PAIR) gb.store(st + 2 * Tl::A_PLANE, st + 2 * Tl::A_PLANE + Tl::B_PLANE, tid);
        };
        if (nkt > 0) {
            load(0);
            store(smem);
            if (nkt > 1) load(1);
        }
        __syncthreads();
        // Stages with a next stage to store and a whole one after it to load,
        // two per turn where the LDS addresses of both stages are in reach of
        // constant offsets (no address arithmetic is left; the 256 x 256
        // tile's 128 KB would need a second set of address registers, which
        // spilled 24-34 of them).
        constexpr int UNROLL = Tl::SMEM_BYTES <= 98304 ? 2 : 1;
        int kt0 = 0;
        constexpr int SPARE = MODE == SHORT ? SHORT_K - BK : 0;  // k behind a whole stage
        const int whole = MODE == SINGLE ? 0 : (K - SPARE) / BK;
        for (; kt0 + 1 + UNROLL < whole; kt0 += UNROLL)
            static_for<0, UNROLL>([&](auto uc) {
                const int kt = kt0 + uc, h = UNROLL == 2 ? (int)uc : kt & 1;
                const __bf16 *st = smem + h * Tl::STAGE;
                __bf16 *nx = smem + (1 - h) * Tl::STAGE, *na = nx + (up ? 2 * Tl::A_PLANE : 0);
                const auto an = operand(a_at(kt + 2)), bn = operand(b_at(kt + 2));
                constexpr int NPA = SA::NPIECE;
                constexpr int NP = NPA + (PAIR ? 0 : SB::NPIECE);
                step0_fused<NP>(st, wm, wn, lane, acc, [&](auto pc) {
                    constexpr int P = decltype(pc)::value;
                    if constexpr (P < NPA) {
                        ga.template store_piece<P>(na, na + Tl::A_PLANE, stid);
                        ga.template load_after_piece<P>(an, stid);
                    } else {
                        gb.template store_piece<P - NPA>(nx + 2 * Tl::A_PLANE,
                                                         nx + 2 * Tl::A_PLANE + Tl::B_PLANE, tid);
                        gb.template load_after_piece<P - NPA>(bn, tid);
                    }
                });
                step(st, 1, wm, wn, lane, acc);
                __syncthreads();
            });
        for (int kt = kt0; kt < nkt; ++kt) {
            const __bf16 *st = smem + (kt & 1) * Tl::STAGE;
            step(st, 0, wm, wn, lane, acc);
            if (kt + 1 < nkt) {
                // The other stage was last read before the previous barrier.
                store(smem + ((kt + 1) & 1) * Tl::STAGE);
                if (kt + 2 < nkt) load(kt + 2);
            }
            step(st, 1, wm, wn, lane, acc);
            __syncthreads();
        }

        if constexpr (KS > 1) {
            // Slices 1 .. KS-1 leave their sums in LDS (over the stages, which
            // every slice has finished reading at the loop's last barrier);
            // slice 0 adds them in slice order.
            const int slice = (int)(threadIdx.x / NT);
            float *red = reinterpret_cast<float *>(smem - (size_t)slice * 2 * Tl::STAGE);
            static_assert((size_t)(KS - 1) * FM * FN * 16 * NT * sizeof(float) <=
                              (size_t)KS * Tl::SMEM_BYTES,
                          "the slices' sums fit in the workgroup's stages");
            if (slice > 0) {
#pragma unroll
                for (int fi = 0; fi < FM; ++fi)
#pragma unroll
                    for (int fn = 0; fn < FN; ++fn)
#pragma unroll
                        for (int r = 0; r < 16; ++r)
                            red[((((size_t)slice - 1) * FM + fi) * FN + fn) * 16 * NT + r * NT + tid] =
                                acc[fi][fn][r];
            }
            __syncthreads();
            if (slice > 0) return;
#pragma unroll 1
            for (int sl = 1; sl < KS; ++sl)
#pragma unroll
                for (int fi = 0; fi < FM; ++fi)
#pragma unroll
                    for (int fn = 0; fn < FN; ++fn)
#pragma unroll
                        for (int r = 0; r < 16; ++r)
                            acc[fi][fn][r] +=
                                red[((((size_t)sl - 1) * FM + fi) * FN + fn) * 16 * NT + r * NT + tid];
        }

        // Epilogue: lanes 0-31 of a register cover 32 consecutive columns.
        // Whatever a row of FN blocks reads (C for beta != 0, the GELU input)
        // is gathered before any result is stored: 16 * FN loads in flight.
        const int l32 = lane & 31, half = lane >> 5;
        const bool reads = (EPI == bmb::EPI_BLAS && beta != 0.0f) || EPI == bmb::EPI_GELU_GRAD;
        float sums[FN] = {};  // of this lane's rows, per column (EPI_GELU_GRAD)
        float bias[FN];
        if (EPI == bmb::EPI_BIAS || EPI == bmb::EPI_BIAS_GELU) {
#pragma unroll
            for (int fn = 0; fn < FN; ++fn) {
                const int col = n0 + wn + fn * 32 + l32;
                bias[fn] = (INTERIOR || col < N) ? ep.bias[col] : 0.0f;
            }
        }
#pragma unroll
        for (int fi = 0; fi < FM; ++fi) {
            float in[FN][16];
            if (reads) {
                const float *src = EPI == bmb::EPI_GELU_GRAD ? ep.pre : C;
#pragma unroll
                for (int fn = 0; fn < FN; ++fn) {
                    const int col = n0 + wn + fn * 32 + l32;
#pragma unroll
                    for (int r = 0; r < 16; ++r) {
                        const int row = m0 + wm + fi * 32 + 8 * (r >> 2) + 4 * half + (r & 3);
                        in[fn][r] = (INTERIOR || (row < M && col < N))
                                        ? src[(size_t)row * ldc + col] : 0.0f;
                    }
                }
            }
#pragma unroll
            for (int fn = 0; fn < FN; ++fn) {
                const int col = n0 + wn + fn * 32 + l32;
                if (!INTERIOR && col >= N) continue;
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    const int row = m0 + wm + fi * 32 + 8 * (r >> 2) + 4 * half + (r & 3);
                    if (!INTERIOR && row >= M) continue;
                    const float a = acc[fi][fn][r];
                    const size_t idx = (size_t)row * ldc + col;
                    if (EPI == bmb::EPI_PARTIAL) {
                        C[idx] = a;
                    } else if (EPI == bmb::EPI_BLAS) {
                        C[idx] = reads ? bmb::fma_rn(alpha, a, beta * in[fn][r]) : alpha * a;
                    } else if (EPI == bmb::EPI_GELU_GRAD) {
                        const float v = bmb::gelu_grad(in[fn][r], a);
                        C[idx] = v;
                        sums[fn] += v;
                    } else {
                        const float v = a + bias[fn];
                        C[idx] = v;
                        if (EPI == bmb::EPI_BIAS_GELU) ep.act[idx] = bmb::gelu(v);
                    }
                }
            }
        }
        if (EPI == bmb::EPI_GELU_GRAD && ep.colsum != nullptr) {
            const size_t w = (size_t)(m0 / BM) * Tl::WAVES_M + wave / Tl::WAVES_N;
#pragma unroll
            for (int fn = 0; fn < FN; ++fn) {
                const int col = n0 + wn + fn * 32 + l32;
                const float t = sums[fn] + __shfl_xor(sums[fn], 32, 64);
                if (half == 0 && (INTERIOR || col < N)) ep.colsum[w * N + col] = t;
            }
        }
    }
};

// Grid: x = output tiles (XCD-remapped, grouped), y = K range s, covering
// k in [s*kchunk, min(K, (s+1)*kchunk)) (kchunk a multiple of BK when
// gridDim.y > 1). EPI_PARTIAL: write the range's raw sums to C + s*M*N
// (packed rows). lda, ldb, ldc: the row strides of the stored A (at least M
// when TA, K otherwise), B (at least K when TB, N otherwise) and C (at least
// N), so that a block of rows and columns of a larger problem (its operands
// offset to its first row and column) runs as a problem of its own.
// KT: K is not a whole number of stages. (A separate instantiation: the last
// stage's loads cost the 256 x 256 kernels spilled registers, which the other
// shapes need not pay.) MODE: OpStage's; SHORT only with KT.
template <class Tl, bool TA, bool TB, int EPI, bool KT, Stage MODE = VECTOR>
__global__ __launch_bounds__(Tl::NT) void bf16x3_k(int M, int N, int K, int kchunk, float alpha,
                                                   const float *__restrict__ A, int lda,
                                                   const float *__restrict__ B, int ldb,
                                                   float beta, float *C, int ldc, int tiles_m,
                                                   int tiles_n, bmb::EpiArgs ep) {
    extern __shared__ __bf16 lds[];
    using G = Bf16x3Gemm<Tl, TA, TB>;
    int tm, tn;
    bmb::group_tile(bmb::xcd_remap(blockIdx.x, tiles_m * tiles_n), tiles_m, tiles_n, 8, tm, tn);
    const int m0 = tm * Tl::BM, n0 = tn * Tl::BN;
    const int kb = blockIdx.y * kchunk, klen = min(K, kb + kchunk) - kb;
    const float *Ak = TA ? A + (size_t)kb * lda : A + kb;
    const float *Bk = TB ? B + kb : B + (size_t)kb * ldb;
    float *Cs = EPI == bmb::EPI_PARTIAL ? C + (size_t)blockIdx.y * M * N : C;
    const int ldcs = EPI == bmb::EPI_PARTIAL ? N : ldc;
    if (m0 + Tl::BM <= M && n0 + Tl::BN <= N)
        G::template run<true, EPI, KT, 1, MODE>(M, N, klen, lda, ldb, alpha, Ak, Bk, beta, Cs,
                                                ldcs, m0, n0, lds, ep);
    else
        G::template run<false, EPI, KT, 1, MODE>(M, N, klen, lda, ldb, alpha, Ak, Bk, beta, Cs,
                                                 ldcs, m0, n0, lds, ep);
}

// The same tile as KS k-slices of Tl::NT lanes each: every slice runs per =
// ceil(stages / KS) stages of the workgroup's K range, slice s those from
// s * per on, in its own KS-th of the LDS, and the slices' sums meet in LDS
// (Bf16x3Gemm::run). For problems with too few output tiles to fill the
// device, where split-K alone would need a second launch for its reduce or
// many more ranges (and partials) for the same number of waves.
// KT: some slice's range is not `per` whole stages.
template <class Tl, bool TA, bool TB, int EPI, int KS, bool KT, Stage MODE = VECTOR>
__global__ __launch_bounds__(Tl::NT * KS) void bf16x3_ks_k(int M, int N, int K, int kchunk,
                                                           float alpha,
                                                           const float *__restrict__ A, int lda,
                                                           const float *__restrict__ B, int ldb,
                                                           float beta, float *C, int ldc,
                                                           int tiles_m, int tiles_n,
                                                           bmb::EpiArgs ep) {
    extern __shared__ __bf16 lds[];
    using G = Bf16x3Gemm<Tl, TA, TB>;
    int tm, tn;
    bmb::group_tile(bmb::xcd_remap(blockIdx.x, tiles_m * tiles_n), tiles_m, tiles_n, 8, tm, tn);
    const int m0 = tm * Tl::BM, n0 = tn * Tl::BN;
    const int kr = blockIdx.y * kchunk, kend = min(K, kr + kchunk);
    // (Uniform over a wave, which the compiler cannot see; the descriptors of
    // the staging loads need it in a scalar register.)
    const int slice = __builtin_amdgcn_readfirstlane((int)(threadIdx.x / Tl::NT));
    const int per = ((kend - kr + BK - 1) / BK + KS - 1) / KS;
    const int kb = min(kr + slice * per * BK, kend);
    const int klen = min(kend - kb, per * BK);  // 0: a slice past the range
    const float *Ak = TA ? A + (size_t)kb * lda : A + kb;
    const float *Bk = TB ? B + kb : B + (size_t)kb * ldb;
    float *Cs = EPI == bmb::EPI_PARTIAL ? C + (size_t)blockIdx.y * M * N : C;
    const int ldcs = EPI == bmb::EPI_PARTIAL ? N : ldc;
    __bf16 *st = lds + (size_t)slice * 2 * Tl::STAGE;
    if (m0 + Tl::BM <= M && n0 + Tl::BN <= N)
        G::template run<true, EPI, KT, KS, MODE>(M, N, klen, lda, ldb, alpha, Ak, Bk, beta, Cs,
                                                 ldcs, m0, n0, st, ep, per);
    else
        G::template run<false, EPI, KT, KS, MODE>(M, N, klen, lda, ldb, alpha, Ak, Bk, beta, Cs,
                                                  ldcs, m0, n0, st, ep, per);
}

// Problems that no other kernel takes (SINGLE): 64 x 64 tiles whose
// operands are loaded element by element.
template <bool TA, bool TB, int EPI>
__global__ __launch_bounds__(TileS::NT) void bf16x3_narrow_k(int M, int N, int K, int kchunk,
                                                             float alpha,
                                                             const float *__restrict__ A, int lda,
                                                             const float *__restrict__ B, int ldb,
                                                             float beta, float *C, int ldc,
                                                             int tiles_m, int tiles_n,
                                                             bmb::EpiArgs ep) {
    extern __shared__ __bf16 lds[];
    int tm, tn;
    bmb::group_tile(bmb::xcd_remap(blockIdx.x, tiles_m * tiles_n), tiles_m, tiles_n, 8, tm, tn);
    const int kb = blockIdx.y * kchunk, klen = min(K, kb + kchunk) - kb;
    const float *Ak = TA ? A + (size_t)kb * lda : A + kb;
    const float *Bk = TB ? B + kb : B + (size_t)kb * ldb;
    float *Cs = EPI == bmb::EPI_PARTIAL ? C + (size_t)blockIdx.y * M * N : C;
    Bf16x3Gemm<TileS, TA, TB>::template run<false, EPI, true, 1, SINGLE>(
        M, N, klen, lda, ldb, alpha, Ak, Bk, beta, Cs, EPI == bmb::EPI_PARTIAL ? N : ldc,
        tm * TileS::BM, tn * TileS::BN, lds, ep);
}

// ------------------------------------------------------------- host side

// Tile and split choice. A work item is one output tile over one K range. A
// CU that holds r items of a tile at once takes
//   c + d r + stages (a + b r) (1 + mis u) t
// us for them (t: nt or tn by transposes, 1 for A B): per 32-k stage a part that residents overlap (a, the latency
// chain of a stage) and one that they share (b, the CU's LDS, VALU and matrix
// cores), a prologue c and an epilogue d. u is the share of the staged bytes
// whose rows are not a multiple of 16 bytes apart. The device runs cus x
// occupancy items per round; the last, partial round is charged between its
// mean and its fullest CU. A split adds the partials' round trip, the reduce
// launch and a term per range (each reduce lane adds its ranges one after
// the other), every plan its launch and the write of C. The constants are a
// least-squares fit (on log time) to 13,000 timed plans of 331 problems on
// one MI355X: every tile x slices x split below over the linear layers of
// GPTs of width 256-1024 at 64-16384 rows in all three transposes, squares of
// 192-4608 and random shapes (M, N, K of 64-8192, a third of them odd). On
// those the model's plan is 1.8% slower than the best measured one on average
// (6% at the 90th percentile); the model before it, fitted to the GPT-2
// layers and squares alone, 3.1% (16%), and up to 1.9x on problems of few
// tiles or short K.
//
// Row bands. A tile count just above a whole number of rounds (4097^2 on
// 256 x 256: 289 tiles on 256 CUs; 6144^2: 576 tiles, 2.25 rounds; the GPT-2
// QKV forward, 8192 x 2304: 288 tiles) leaves most CUs idle for a whole
// extra tile time. A plan may therefore run C as two bands of full-width
// rows, one launch each on the same stream: rows [0, m1) on one tile with
// whole K, sized to whole rounds, and rows [m1, M) on the plan (tile and
// split) that suits that remainder, typically a smaller tile or a K split
// that spreads it over every CU.
struct B3Cand {
    int bm, bn, ks;  // tile, and k-slices per workgroup (bf16x3_ks_k)
    double a, b, c, d, mis;
    double nt, tn;  // stages of A B^T and of A^T B (and A^T B^T) against A B
};
constexpr B3Cand CANDS[] = {
    {256, 256, 1, 0.000, 2.316, 3.82, 1.02, 0.06, 0.95, 0.97},
    {128, 128, 1, 0.251, 0.572, 2.07, 0.22, 0.11, 0.98, 1.04},
    {64, 64, 1, 0.158, 0.234, 1.01, 0.04, 0.16, 0.89, 0.99},
    {128, 256, 1, 0.019, 1.263, 1.19, 2.37, 0.08, 0.95, 1.02},
    {64, 64, 2, 0.134, 0.498, 1.15, 0.00, 0.19, 0.89, 0.98},
    {64, 64, 4, 0.118, 1.093, 0.76, 1.10, 0.20, 0.86, 0.95},
    {32, 32, 4, 0.225, 0.331, 0.91, 0.00, 0.35, 0.94, 1.09},
    {32, 32, 8, 0.300, 0.588, 0.14, 1.22, 0.42, 0.96, 1.11},
    {128, 64, 2, 0.180, 0.785, 2.14, 0.00, 0.14, 0.94, 1.11},
};
constexpr int N_CANDS = 9;
constexpr int NARROW = N_CANDS;  // bf16x3_narrow_k, planned as the 64 x 64 tile
constexpr int MIN_DIM = 4;       // the least M and N of a band (vector loads of its rows)
// The 32 x 32 tile is only taken up to XS_MAX_OUTPUTS outputs, and every
// slice keeps at least MIN_SLICE_K of k.
constexpr long long XS_MAX_OUTPUTS = 1LL << 20;
constexpr int MIN_SLICE_K = 64;
// Split counts that are not powers of two fill the device in one round where
// {2, 4, 8} do not (36 tiles of 256 x 256 in 7 ranges on 256 CUs).
constexpr int SPLITS[] = {1, 2, 3, 4, 5, 6, 7, 8, 10, 12, 14, 16};
constexpr double LAUNCH_US = 3.5;                 // one launch, timed back to back
constexpr double C_BYTES_PER_US = 13.0e6;         // the write of C
constexpr double PARTIALS_BYTES_PER_US = 11.0e6;  // the partials' round trip
constexpr double REDUCE_US = 1.1, RANGE_US = 0.24;  // the reduce, and each range in it
constexpr double FULLEST = 0.65;  // a partial round: the weight of its fullest CU
// A second band: its launch and the drain between the bands. Bands are only
// tried for K >= MIN_BAND_K, with K ranges of at least MIN_BAND_SPLIT_K in a
// split remainder band, and taken when modelled 3% faster than one band:
// measured on MI355X, bands gained 15-18% at N = 4097 and 6144 and on the
// GPT-2 LM-head weight gradient (K = 8192), and 4.5% on the GPT-2 QKV
// forward (8192 x 2304 x 768: 7168 rows on 256 x 256 tiles in two whole
// rounds, the last 1024 on 128 x 128). Without the bound on the remainder's
// K ranges they lost 3-7% on the K = 768 and 3072 GPT-2 GEMMs, whose short
// split ranges the model undercharges; with it, no other GPT-2 or square
// sweep shape changes plan. Corner plans (below) are tried for
// K >= MIN_CORNER_K only, the range they were measured on.
constexpr double BAND_US = 9.0;
constexpr double BAND_GAIN = 0.97;
constexpr int MIN_BAND_K = 768;
constexpr int MIN_CORNER_K = 4096;
constexpr int MIN_BAND_SPLIT_K = 512;
constexpr int MIN_SPLIT_K = 64;  // two stages
constexpr long long MAX_SPLIT_FLOATS = 64LL << 20;  // 256 MiB of partials

template <class Kern>
int occupancy_of(Kern kern, int threads, size_t smem) {
    int n = 0;
    bmb::allow_smem(kern, smem);
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, kern, threads, smem) != hipSuccess) {
        (void)hipGetLastError();
        n = 1;
    }
    return n < 1 ? 1 : n;
}
template <class Tl>
int occupancy_of() {
    return occupancy_of(bf16x3_k<Tl, false, false, bmb::EPI_BLAS, false>, Tl::NT, Tl::SMEM_BYTES);
}
template <class Tl, int KS>
int ks_occupancy_of() {
    return occupancy_of(bf16x3_ks_k<Tl, false, false, bmb::EPI_BLAS, KS, false>, Tl::NT * KS,
                        KS * Tl::SMEM_BYTES);
}

// One band's launch: tile candidate, K ranges, the K per range, and the
// staging of the operands.
struct Part {
    int tile, splits, kchunk;
    Stage mode;
};

// Rows [0, m1) run on part[0], rows [m1, M) on part[1] (m1 == M: one band).
// A corner plan (edges) instead runs rows [0, m1) x columns [0, n1) on
// part[0], a block of whole tiles, and the at most EDGE_MAX columns right of
// it and rows below it on the edge kernels (edge_gemm.hip): 4097^2 as
// 4096^2 on 256 x 256 tiles plus a 4096 x 1 and a 1 x 4097 edge, where a
// plan of tiles alone computes 289 tiles (13% more than C) or runs a second
// band.
struct Plan {
    Part part[2];
    int m1, n1;
    bool edges;
};

struct Device {
    int occ[N_CANDS], cus;
};

const Device &device_info(int dev) {
    static std::once_flag once[64];
    static Device info[64];
    std::call_once(once[dev], [&] {
        Device &d = info[dev];
        d.occ[0] = occupancy_of<TileL>();
        d.occ[1] = occupancy_of<TileM>();
        d.occ[2] = occupancy_of<TileS>();
        d.occ[3] = occupancy_of<TileT>();
        d.occ[4] = ks_occupancy_of<TileS, 2>();
        d.occ[5] = ks_occupancy_of<TileS, 4>();
        d.occ[6] = ks_occupancy_of<TileXS, 4>();
        d.occ[7] = ks_occupancy_of<TileXS, 8>();
        d.occ[8] = ks_occupancy_of<TileH, 2>();
        int c = 0;
        if (hipDeviceGetAttribute(&c, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess ||
            c <= 0) {
            (void)hipGetLastError();
            c = 256;
        }
        d.cus = c;
    });
    return info[dev];
}

// What a plan depends on besides M, N and K: the transposes, whether an
// operand's rows are not 16-byte aligned, and the stored row strides (a band's
// operands keep those of the whole problem).
struct Layout {
    bool ta, tb, mis_a, mis_b;
    int lda, ldb;
};

// Whether the staging loads' byte offsets within a tile (OpStage::o) stay
// below 2^32: they span the tile's rows of an operand with contiguous k, BK
// rows of one with contiguous m or n.
bool reaches(const B3Cand &c, const Layout &lo) {
    return (lo.ta ? BK + 1LL : c.bm) * lo.lda < 1LL << 30 &&
           (lo.tb ? (long long)c.bn : BK + 1LL) * lo.ldb < 1LL << 30;
}

// Modelled time (us) of an M x N x K band on tile t with K split s ways;
// false if that split is not allowed (may_split, max_floats caps splits * M *
// N).
bool part_time(const Device &dv, int M, int N, int K, int t, int s, Layout lo, bool may_split,
               long long max_floats, Part &out, double &time) {
    const B3Cand &c = CANDS[t];
    int splits = 1, kchunk = K;
    if (c.ks > 1) {
        if (K / s < c.ks * MIN_SLICE_K) return false;
        if (c.bm == 32 && (long long)M * N > XS_MAX_OUTPUTS) return false;
    }
    if (s > 1) {
        if (!may_split || K < 2 * MIN_SPLIT_K) return false;
        kchunk = (K + s - 1) / s;
        kchunk = (kchunk + BK - 1) / BK * BK;
        if (kchunk < MIN_SPLIT_K) return false;
        splits = (K + kchunk - 1) / kchunk;
        if (splits < 2 || (long long)splits * M * N > max_floats) return false;
        if (splits != s) return false;  // (another entry of SPLITS)
    }
    const double mn = (double)M * N;
    const long long items =
        (long long)bmb::ceil_div(M, c.bm) * bmb::ceil_div(N, c.bn) * splits;
    const int occ = dv.occ[t], cus = dv.cus;
    const double stages = bmb::ceil_div(bmb::ceil_div(kchunk, BK), c.ks);
    const double share = (double)c.bm / (c.bm + c.bn);  // of the staged bytes, A's
    const double mis = 1.0 + c.mis * ((lo.mis_a ? share : 0.0) + (lo.mis_b ? 1.0 - share : 0.0));
    const double rate = mis * (lo.ta ? c.tn : lo.tb ? c.nt : 1.0);
    auto round = [&](double r) { return c.c + c.d * r + stages * (c.a + c.b * r) * rate; };
    const long long slots = (long long)cus * occ, rem = items % slots;
    time = (items / slots) * round(occ) + LAUNCH_US + mn * 4.0 / C_BYTES_PER_US;
    if (rem)
        time += FULLEST * round((double)((rem + cus - 1) / cus)) +
                (1.0 - FULLEST) * round((double)rem / cus);
    if (splits > 1)
        time += (2.0 * splits + 1.0) * mn * 4.0 / PARTIALS_BYTES_PER_US + REDUCE_US +
                splits * RANGE_US;
    out = Part{t, splits, kchunk, VECTOR};
    return true;
}

// How an M x N x K problem's operands can be staged. Vector loads need stored
// rows of four elements; shorter ones take the SHORT kernels (short_ok: the
// epilogue has them) down to four elements in the whole operand. An operand
// that is smaller still, or an empty product, is loaded element by element.
// (An M or N below four is no short row where k is contiguous. With every
// dimension below four loaded by element, in us, against now: 1 x 768 x 768 of
// A B^T 9.4 and 5.9, 3 x 50257 x 768 72 and 30; SHORT: 8192 x 1 x 768 of A B
// 14.2 and 8.3, 768 x 1 x 8192 27.0 and 11.3, 4096 x 4096 x 1 of A^T B 24.3 and
// 14.9.)
Stage staging(int M, int N, int K, Layout lo, bool short_ok) {
    if (std::min(lo.lda, lo.ldb) >= MIN_DIM) return VECTOR;
    const bool flat = (long long)M * K >= MIN_DIM && (long long)N * K >= MIN_DIM;
    return short_ok && flat ? SHORT : SINGLE;
}

// The tiles that have a SHORT kernel.
bool short_tile(int t) { return t == 1 || t == 2 || t == 5 || t == 7; }

// The fastest single-band plan of an M x N x K band (split K ranges of at
// least min_split_k; k-sliced tiles only if ks_ok). Where no tile reaches, the
// narrow kernel.
double best_part(const Device &dv, int M, int N, int K, Layout lo, Stage mode, bool may_split,
                 long long max_floats, Part &best, int min_split_k = 0, bool ks_ok = false) {
    const auto usable = [&](int t) {
        return (CANDS[t].ks == 1 || ks_ok) && (mode != SHORT || short_tile(t)) &&
               reaches(CANDS[t], lo);
    };
    bool any = false;
    for (int t = 0; t < N_CANDS; ++t) any |= usable(t);
    if (!any) mode = SINGLE;
    double best_t = -1.0;
    best = Part{NARROW, 1, K, SINGLE};
    for (int t = 0; t < N_CANDS; ++t)
        for (int s : SPLITS) {
            if (mode == SINGLE ? t != 2 : !usable(t)) continue;
            Part p;
            double tm;
            if (part_time(dv, M, N, K, t, s, lo, may_split, max_floats, p, tm) &&
                (p.splits == 1 || p.kchunk >= min_split_k) && (best_t < 0 || tm < best_t)) {
                best_t = tm;
                best = p;
                best.mode = mode;
                if (mode == SINGLE) best.tile = NARROW;
            }
        }
    return best_t;
}

Plan plan_for(int dev, int M, int N, int K, Layout lo, bool may_split, long long max_floats,
              bool edges_ok, bool short_ok) {
    const Device &dv = device_info(dev);
    const Stage mode = staging(M, N, K, lo, short_ok);
    Plan best{{Part{0, 1, K, VECTOR}, Part{0, 1, K, VECTOR}}, M, N, false};
    const double single_t =
        best_part(dv, M, N, K, lo, mode, may_split, max_floats, best.part[0], 0, true);
    double best_t = single_t;
    // Two bands: the first whole rounds of one tile, the rest on its own plan.
    for (int t = 0; mode == VECTOR && K >= MIN_BAND_K && t < N_CANDS; ++t) {
        const B3Cand &c = CANDS[t];
        if (c.ks > 1 || !reaches(c, lo)) continue;
        const long long tiles_n = bmb::ceil_div(N, c.bn);
        const long long slots = (long long)dv.cus * dv.occ[t];
        for (long long k = 1;; ++k) {
            const long long rows = k * slots / tiles_n;  // tile rows in k whole rounds
            if (rows <= 0) continue;
            if (rows * c.bm >= M) break;
            const int m1 = (int)(rows * c.bm);
            if (M - m1 < MIN_DIM) continue;
            Part p0, p1;
            double t0, t1;
            if (!part_time(dv, m1, N, K, t, 1, lo, false, 0, p0, t0)) continue;
            t1 = best_part(dv, M - m1, N, K, lo, mode, may_split, max_floats, p1,
                           MIN_BAND_SPLIT_K);
            const double tm = t0 + t1 + BAND_US;
            if (tm < BAND_GAIN * single_t && tm < best_t) {
                best_t = tm;
                best = Plan{{p0, p1}, m1, N, false};
            }
        }
    }
    // Corner plans: whole tiles of one candidate over [0, m1) x [0, n1), the
    // edges on the edge kernels (row-major A and B, BLAS epilogue; their
    // scratch only where K may be split).
    for (int t = 0; mode == VECTOR && edges_ok && may_split && K >= MIN_CORNER_K && t < N_CANDS;
         ++t) {
        const B3Cand &c = CANDS[t];
        if (c.ks > 1 || !reaches(c, lo)) continue;
        const int m1 = M / c.bm * c.bm, n1 = N / c.bn * c.bn;
        if (m1 == 0 || n1 == 0 || (m1 == M && n1 == N) || M - m1 > bmb::EDGE_MAX ||
            N - n1 > bmb::EDGE_MAX || bmb::edge_partial_floats(M - m1, N - n1, N, K) > max_floats)
            continue;
        Part p0;
        double t0;
        if (!part_time(dv, m1, n1, K, t, 1, lo, false, 0, p0, t0)) continue;
        const double tm = t0 + 1e6 * bmb::edge_model_s(m1, N - n1, M - m1, N, K);
        if (tm < BAND_GAIN * single_t && tm < best_t) {
            best_t = tm;
            best = Plan{{p0, Part{0, 1, K, VECTOR}}, m1, n1, true};
        }
    }
    if (getenv("BMB_GEMM_PLAN_TRACE") != nullptr)
        fprintf(stderr, "bf16x3 gemm plan %dx%dx%d: m1 %d n1 %d edges %d parts (%d,%d,%d) "
                        "(%d,%d,%d) model %.1f us (one band %.1f us)\n",
                M, N, K, best.m1, best.n1, (int)best.edges, best.part[0].tile,
                best.part[0].splits, best.part[0].kchunk, best.part[1].tile, best.part[1].splits,
                best.part[1].kchunk, best_t, single_t);
    return best;
}

// Plans are memoised per (device, shape, layout, split permission and cap):
// the search above costs tens of microseconds, a GEMM call in a training step
// a few hundred. Each host thread keeps its last plans in a table of its own
// in front of the shared map, so that a repeated call neither locks nor walks
// the map.
struct PlanKey {
    int dev, M, N, K;
    Layout lo;
    bool may_split, edges_ok, short_ok;
    long long max_floats;
    auto tie() const { return std::tie(dev, M, N, K, lo.ta, lo.tb, lo.mis_a, lo.mis_b, may_split,
                                       edges_ok, short_ok, max_floats); }
    bool operator<(const PlanKey &o) const { return tie() < o.tie(); }
    bool operator==(const PlanKey &o) const { return tie() == o.tie(); }
};

Plan pick(int M, int N, int K, Layout lo, bool may_split, long long max_floats, bool edges_ok,
          bool short_ok) {
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) dev = 0;
    const PlanKey key{dev, M, N, K, lo, may_split, edges_ok, short_ok, max_floats};
    struct Entry {
        PlanKey key;
        Plan plan;
    };
    static thread_local Entry recent[64] = {};  // (M = 0 is never planned)
    const unsigned h = ((unsigned)M * 2654435761u) ^ ((unsigned)N * 40503u) ^ (unsigned)K * 97u ^
                       (lo.ta ? 5u : 0u) ^ (lo.tb ? 10u : 0u);
    Entry &e = recent[(h ^ (h >> 13)) % 64];
    if (e.key == key) return e.plan;
    static std::mutex mu;
    static std::map<PlanKey, Plan> memo;
    {
        std::lock_guard<std::mutex> lock(mu);
        const auto it = memo.find(key);
        if (it != memo.end()) {
            e = Entry{key, it->second};
            return e.plan;
        }
    }
    const Plan p = plan_for(dev, M, N, K, lo, may_split, max_floats, edges_ok, short_ok);
    std::lock_guard<std::mutex> lock(mu);
    if (memo.size() > 4096) memo.clear();
    memo.emplace(key, p);
    e = Entry{key, p};
    return p;
}

// The row strides of a launch's operands (see bf16x3_k).
struct Strides {
    int lda, ldb, ldc;
};

// Whether a tile (in KS k-slices) has a SHORT kernel (short_tile), and for this
// epilogue: short rows are planned for gemm() only.
template <class Tl, int KS, int EPI>
constexpr bool HAS_SHORT =
    (EPI == bmb::EPI_BLAS || EPI == bmb::EPI_PARTIAL) &&
    ((KS == 1 && (std::is_same<Tl, TileM>::value || std::is_same<Tl, TileS>::value)) ||
     (KS == 4 && std::is_same<Tl, TileS>::value) || (KS == 8 && std::is_same<Tl, TileXS>::value));

template <class Tl, bool TA, bool TB, int EPI>
void launch(int M, int N, int K, const Part &p, float alpha, const float *A, const float *B,
            float beta, float *C, const Strides &ld, hipStream_t stream, bmb::EpiArgs ep) {
    const int tiles_m = bmb::ceil_div(M, Tl::BM), tiles_n = bmb::ceil_div(N, Tl::BN);
    auto go = [&](auto kern) {
        bmb::allow_smem(kern, Tl::SMEM_BYTES);
        bmb::launch(kern, dim3(tiles_m * tiles_n, p.splits), dim3(Tl::NT), Tl::SMEM_BYTES, stream,
                    M, N, K, p.kchunk, alpha, A, ld.lda, B, ld.ldb, beta, C, ld.ldc, tiles_m,
                    tiles_n, ep);
    };
    if constexpr (HAS_SHORT<Tl, 1, EPI>)
        if (p.mode == SHORT) return go(bf16x3_k<Tl, TA, TB, EPI, true, SHORT>);
    if (K % BK != 0) go(bf16x3_k<Tl, TA, TB, EPI, true>);
    else go(bf16x3_k<Tl, TA, TB, EPI, false>);
}

// The k-sliced launch: one workgroup of KS slices per tile and K range.
template <class Tl, bool TA, bool TB, int EPI, int KS>
void launch_ks(int M, int N, int K, const Part &p, float alpha, const float *A, const float *B,
               float beta, float *C, const Strides &ld, hipStream_t stream, bmb::EpiArgs ep) {
    const int tiles_m = bmb::ceil_div(M, Tl::BM), tiles_n = bmb::ceil_div(N, Tl::BN);
    const size_t smem = (size_t)KS * Tl::SMEM_BYTES;
    auto go = [&](auto kern) {
        bmb::allow_smem(kern, smem);
        bmb::launch(kern, dim3(tiles_m * tiles_n, p.splits), dim3(Tl::NT * KS), smem, stream, M,
                    N, K, p.kchunk, alpha, A, ld.lda, B, ld.ldb, beta, C, ld.ldc, tiles_m,
                    tiles_n, ep);
    };
    if constexpr (HAS_SHORT<Tl, KS, EPI>)
        if (p.mode == SHORT) return go(bf16x3_ks_k<Tl, TA, TB, EPI, KS, true, SHORT>);
    if (p.kchunk % (BK * KS) != 0 || K % p.kchunk != 0) go(bf16x3_ks_k<Tl, TA, TB, EPI, KS, true>);
    else go(bf16x3_ks_k<Tl, TA, TB, EPI, KS, false>);
}

template <bool TA, bool TB, int EPI>
void launch_tile(int M, int N, int K, const Part &p, float alpha, const float *A, const float *B,
                 float beta, float *C, const Strides &ld, hipStream_t stream, bmb::EpiArgs ep) {
    switch (p.tile) {
    case 0: launch<TileL, TA, TB, EPI>(M, N, K, p, alpha, A, B, beta, C, ld, stream, ep); break;
    case 1: launch<TileM, TA, TB, EPI>(M, N, K, p, alpha, A, B, beta, C, ld, stream, ep); break;
    case 2: launch<TileS, TA, TB, EPI>(M, N, K, p, alpha, A, B, beta, C, ld, stream, ep); break;
    case 3: launch<TileT, TA, TB, EPI>(M, N, K, p, alpha, A, B, beta, C, ld, stream, ep); break;
    case 4: launch_ks<TileS, TA, TB, EPI, 2>(M, N, K, p, alpha, A, B, beta, C, ld, stream, ep); break;
    case 5: launch_ks<TileS, TA, TB, EPI, 4>(M, N, K, p, alpha, A, B, beta, C, ld, stream, ep); break;
    case 6: launch_ks<TileXS, TA, TB, EPI, 4>(M, N, K, p, alpha, A, B, beta, C, ld, stream, ep); break;
    case 7: launch_ks<TileXS, TA, TB, EPI, 8>(M, N, K, p, alpha, A, B, beta, C, ld, stream, ep); break;
    case 8: launch_ks<TileH, TA, TB, EPI, 2>(M, N, K, p, alpha, A, B, beta, C, ld, stream, ep); break;
    default:
        bmb::launch(bf16x3_narrow_k<TA, TB, EPI>,
                    dim3(bmb::ceil_div(M, TileS::BM) * bmb::ceil_div(N, TileS::BN), p.splits),
                    dim3(TileS::NT), TileS::SMEM_BYTES, stream, M, N, K, p.kchunk, alpha, A,
                    ld.lda, B, ld.ldb, beta, C, ld.ldc, bmb::ceil_div(M, TileS::BM),
                    bmb::ceil_div(N, TileS::BN), ep);
    }
}

// One band: one launch with the epilogue, or the split partials (EPI_PARTIAL
// into P) and the shared reduce with the epilogue.
template <bool TA, bool TB, int EPI>
void run_band(const Part &p, int M, int N, int K, float alpha, const float *A, const float *B,
              float beta, float *C, const Strides &ld, float *P, hipStream_t stream,
              bmb::EpiArgs ep) {
    if (p.splits > 1) {
        launch_tile<TA, TB, bmb::EPI_PARTIAL>(M, N, K, p, 1.0f, A, B, 0.0f, P, ld, stream, ep);
        bmb::splitk_reduce_epi(EPI, C, P, p.splits, (long long)M * N, N, ld.ldc, alpha, beta,
                               stream, ep.bias, ep.act, ep.pre);
    } else {
        launch_tile<TA, TB, EPI>(M, N, K, p, alpha, A, B, beta, C, ld, stream, ep);
    }
}

// Rows of partial column sums that a part of M rows writes (EpiArgs::colsum).
int sum_rows(const Part &p, int M) {
    if (p.tile == NARROW) return bmb::ceil_div(M, TileS::BM) * TileS::WAVES_M;
    const int bm = CANDS[p.tile].bm;
    return bmb::ceil_div(M, bm) * (bm == 32 ? TileXS::WAVES_M : TileS::WAVES_M);
}
static_assert(TileL::WAVES_M == TileS::WAVES_M && TileM::WAVES_M == TileS::WAVES_M &&
                  TileT::WAVES_M == TileS::WAVES_M && TileH::WAVES_M == TileS::WAVES_M,
              "sum_rows");

// Both bands of a plan, in row order on one stream (the second band's split
// partials reuse P after the first band's reduce has read it).
template <bool TA, bool TB, int EPI>
void run_plan(const Plan &p, int M, int N, int K, float alpha, const float *A, const float *B,
              float beta, float *C, float *P, hipStream_t stream, bmb::EpiArgs ep) {
    const Strides ld{TA ? M : K, TB ? K : N, N};
    run_band<TA, TB, EPI>(p.part[0], p.m1, p.n1, K, alpha, A, B, beta, C, ld, P, stream, ep);
    if (p.edges) {
        bmb::gemm_edges(true, M, N, K, p.m1, p.n1, alpha, A, ld.lda, B, ld.ldb, beta, C, ld.ldc,
                        P, stream);
        return;
    }
    if (p.m1 >= M) return;
    const size_t r = (size_t)p.m1;
    bmb::EpiArgs e1 = ep;
    if (e1.act) e1.act += r * N;
    if (e1.pre) e1.pre += r * N;
    if (e1.colsum) e1.colsum += (size_t)sum_rows(p.part[0], p.m1) * N;
    // A band of rows starts r rows (TA: r columns of the stored K x M) in.
    const float *A1 = TA ? A + r : A + r * K;
    run_band<TA, TB, EPI>(p.part[1], M - p.m1, N, K, alpha, A1, B, beta, C + r * N, ld, P, stream,
                          e1);
}

long long partial_floats(const Plan &p, int M, int N, int K) {
    long long f = 0;
    if (p.edges) return bmb::edge_partial_floats(M - p.m1, N - p.n1, N, K);
    if (p.part[0].splits > 1) f = (long long)p.part[0].splits * p.m1 * N;
    if (p.m1 < M && p.part[1].splits > 1)
        f = std::max(f, (long long)p.part[1].splits * (M - p.m1) * N);
    return f;
}

}  // namespace

// The bf16x3 GEMM behind gemm(), gemm_noalloc() and the GPT's fused linear
// layers (gemm_fused.hpp). Split-K partials go to `fixed` (at most
// fixed_floats), or else to scratch leased for `stream` (its reuse is ordered
// by the lease's event), except under graph capture, where a lease could
// allocate: there K is not split. The epilogue is one of
// EPI_BLAS (any transposes), EPI_BIAS / EPI_BIAS_GELU (A @ W^T) and
// EPI_GELU_GRAD (A @ B). Returns false, with nothing launched, for another
// combination.
bool bmb::bf16x3_gemm(bool ta, bool tb, int M, int N, int K, float alpha, const float *A,
                      const float *B, float beta, float *C, hipStream_t stream, int epi,
                      const float *bias, float *act, const float *pre, float *fixed,
                      long long fixed_floats, float *colsum, int *colsum_rows) {
    if (M <= 0 || N <= 0) return true;
    bmb::EpiArgs ep{bias, act, pre, nullptr};
    const bool may_split = fixed != nullptr || !bmb::stream_capturing(stream);
    const bool edges_ok = !ta && !tb && epi == bmb::EPI_BLAS;
    // (Every epilogue has the kernels of stored rows of at least four elements,
    // so a fused linear layer and gemm() plus the separate bias/GELU pass plan
    // such a shape alike and give the same bits.)
    const bool short_ok = epi == bmb::EPI_BLAS;
    const Layout lo{ta, tb, (ta ? M : K) % 4 != 0 || ((uintptr_t)A & 15) != 0,
                    (tb ? K : N) % 4 != 0 || ((uintptr_t)B & 15) != 0, ta ? M : K, tb ? K : N};
    Plan p = pick(M, N, K, lo, may_split, fixed ? fixed_floats : MAX_SPLIT_FLOATS,
                  edges_ok, short_ok);
    float *P = fixed;
    std::optional<bmb::ScratchLease> lease;
    const long long pf = partial_floats(p, M, N, K);
    if (pf > 0 && fixed == nullptr) {
        lease.emplace(bmb::SCRATCH_GEMM, (size_t)pf * sizeof(float), stream);
        P = static_cast<float *>(lease->get());
        if (P == nullptr) p = pick(M, N, K, lo, false, 0, edges_ok, short_ok);  // no scratch: no split
    }
    const bool banded = p.m1 < M;
    if (colsum != nullptr && p.part[0].splits == 1 && (!banded || p.part[1].splits == 1)) {
        ep.colsum = colsum;
        *colsum_rows = sum_rows(p.part[0], p.m1) + (banded ? sum_rows(p.part[1], M - p.m1) : 0);
    }
#define BMB_B3(TA_, TB_, EPI_)                                                              \
    run_plan<TA_, TB_, EPI_>(p, M, N, K, alpha, A, B, beta, C, P, stream, ep);              \
    return true;
    if (epi == bmb::EPI_BLAS) {
        if (!ta && !tb) { BMB_B3(false, false, bmb::EPI_BLAS) }
        if (!ta && tb) { BMB_B3(false, true, bmb::EPI_BLAS) }
        if (ta && !tb) { BMB_B3(true, false, bmb::EPI_BLAS) }
        BMB_B3(true, true, bmb::EPI_BLAS)
    }
    if (epi == bmb::EPI_BIAS && !ta && tb) { BMB_B3(false, true, bmb::EPI_BIAS) }
    if (epi == bmb::EPI_BIAS_GELU && !ta && tb) { BMB_B3(false, true, bmb::EPI_BIAS_GELU) }
    if (epi == bmb::EPI_GELU_GRAD && !ta && !tb) { BMB_B3(false, false, bmb::EPI_GELU_GRAD) }
#undef BMB_B3
    return false;
}

extern "C" void sgemm_mfma_bf16x3(int M, int N, int K, float alpha,
                                  const float *A, const float *B, float beta,
                                  float *C) {
    bmb::bf16x3_gemm(false, false, M, N, K, alpha, A, B, beta, C, nullptr, bmb::EPI_BLAS,
                     nullptr, nullptr, nullptr, nullptr, 0);
}
