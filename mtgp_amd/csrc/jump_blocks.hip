// jump_blocks.hip -- jump-ahead on the matrix cores in coefficient blocks.
//
// A jump replaces a window by new[j] = XOR_{k : c_k = 1} w[k + j] over the
// generator's own sequence w (mtgp32-fast-jump.c:51-79 computes the same by
// stepping and adding).  The polynomial is cut into blocks of kJbBlock
// coefficients (jump_blocks.hpp):
//  * jump_tiles_kernel: every (jump, block) pair of a base window is one
//    column of a GF(2) product with the same short sequence w[0, N +
//    kJbBlock), so a few jumps already fill the 32 columns of the
//    matrix-core product.  Rows are the 32 bits of a window word, the sum
//    runs over the block's coefficients: bits as fp4 0 and 1.0, exact fp32
//    counts, the parity of a count is the bit.
//  * jump_folds_kernel: one workgroup per jump advances the last block's
//    partial window by kJbBlock numbers, XORs the block before it, and so on
//    (Horner's rule in the generator's step).
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "common.hpp"
#include "jump_blocks.hpp"
#include "kernels.hpp"
// Angle brackets: the kernel emulation build substitutes its own copies.
#include <gfx950_ops.hpp>
#include <jump_ops.hpp>

namespace mtgp {
namespace {

#define GMEM __attribute__((address_space(1)))
typedef GMEM uint32_t gu32;
typedef GMEM uint64_t gu64;
typedef uint32_t v4u __attribute__((ext_vector_type(4)));
typedef uint32_t v2u __attribute__((ext_vector_type(2)));
typedef int v4i __attribute__((ext_vector_type(4)));
typedef GMEM v2u gu2;
typedef GMEM v4u gu4;

constexpr int kWave = 64;
constexpr uint32_t kOnes = 0x22222222u;  // fp4 1.0 in every nibble

struct Rec {
    int n, pos, sh1, sh2;
    uint32_t mask_hi, mask_lo;
};

__device__ __forceinline__ Rec rec_of(const DevParam &D) {
    return Rec{D.n, D.pos, D.sh1, D.sh2, D.mask_hi, D.mask_lo};
}

// The word after window word i of the 32-bit sequence h (MTGP32), or of the
// planes h (high) and l (low) (MTGP64): mtgp32-fast.h:149-159 and
// mtgp64-fast.h:148-169 (only the high half of a table entry is non-zero).
template <int BITS>
__device__ __forceinline__ void next_word(Rec p, const uint32_t *tbl, const uint32_t *h, const uint32_t *l, int i,
                                          uint32_t &rh, uint32_t &rl) {
    if (BITS == 32) {
        const uint32_t x = (h[i] & p.mask_lo) ^ h[i + 1];
        const uint32_t y = xor3(x, x << p.sh1, h[i + p.pos] >> p.sh2);
        rh = y ^ tbl[y & 15];
        rl = 0;
    } else {
        const uint32_t xh = (h[i] & p.mask_hi) ^ h[i + 1];
        const uint32_t xl = (l[i] & p.mask_lo) ^ l[i + 1];
        const uint32_t nh = xor3(xl, xl << p.sh1, h[i + p.pos] >> p.sh2);
        rl = xor3(xh, xh << p.sh1, l[i + p.pos] >> p.sh2);
        rh = nh ^ tbl[rl & 15];
    }
}

// Bits 4 q + r of v as fp4 0 / 1.0 in nibble q of dword r.
__device__ __forceinline__ v4u fp4_expand(uint32_t v) {
    return v4u{(v << 1) & kOnes, v & kOnes, (v >> 1) & kOnes, (v >> 2) & kOnes};
}

// The 32 x 32 bit transpose of each group of 32 lanes: row t in lane t,
// returns column l to lane l.  Round D: lanes l and l ^ D swap the off-diagonal
// D x D blocks of their 2 D x 2 D block: keep[D] of one's own bits, the rest
// from the partner's word rotated by D towards them.
struct Transpose {
    uint32_t keep[5], rot[5];  // for D = 16, 8, 4, 2, 1
    __device__ __forceinline__ Transpose() {
        const uint32_t lo[5] = {0x0000ffffu, 0x00ff00ffu, 0x0f0f0f0fu, 0x33333333u, 0x55555555u};
#pragma unroll
        for (int i = 0; i < 5; i++) {
            const bool up = threadIdx.x >> (4 - i) & 1u;
            keep[i] = up ? ~lo[i] : lo[i];
            rot[i] = up ? 16u >> i : 32u - (16u >> i);
        }
    }
    template <int I>
    __device__ __forceinline__ uint32_t round(uint32_t v) const {
        const uint32_t p = lane_xor<(16 >> I)>(v);
        return (v & keep[I]) | (funnel32(p, p, rot[I]) & ~keep[I]);
    }
    __device__ __forceinline__ uint32_t operator()(uint32_t v) const {
        return round<4>(round<3>(round<2>(round<1>(round<0>(v)))));
    }
};

// ---------------------------------------------------------------- products
// One workgroup of kTileWaves waves per JumpShare.  For each of its tiles (A
// only where the base window or plane changes) the base's sequence is
// generated in LDS (kJbBlock numbers past the window), one 32-bit plane of it
// transposed to bit planes and expanded to fp4 operands (A: bit p of 32
// consecutive positions is 16 bytes), the tile's coefficients expanded to B.
// Then each wave takes word groups: kTileWords consecutive window words, an
// accumulator each per column tile (4 or 8).  The operand of word j is the bit planes from position j on: dword
// r of it holds the bits at offsets 4 q + r, so word j + 1's is the same
// four dwords moved on by one with one new dword (a funnel shift of the
// expanded planes).
constexpr int kTileWaves = 4;
constexpr int kTileThreads = kWave * kTileWaves;
constexpr int kSteps = kJbBlock / 64;  // products per word and tile

// One product step is 64 coefficients of kTileWords words and CT column tiles
// of 32.  Its operands as they lie in LDS: two expanded plane rows from the
// words' first position on, the coefficients.
constexpr int kTileWords = 4;
template <int CT>
struct Loaded {
    v4u m0, m1, b[CT];
    __device__ __forceinline__ Loaded(const v4u *a, const v4u *bt, int ks) {
        m0 = a[64 * ks];
        m1 = a[64 * ks + 32];
#pragma unroll
        for (int c = 0; c < CT; c++)
            b[c] = bt[kWave * (CT * ks + c)];
    }
};
// The matrix operands.  u[0][i], nibble q: the plane's bit at offset sh + i +
// 4 q (sh: the first word's offset in its row); word jj's operand is u[jj ..
// jj + 3] in consecutive registers from an even one on, so the odd words have
// a set of their own, u[1] (made from sh1, which the compiler does not know
// to equal sh: it would copy one set to the other).  EDGE: sh == 28, where
// offsets from sh + 4 on begin the next row.
template <int CT, bool EDGE>
struct Operands {
    uint32_t u[2][kTileWords + 3];
    v4u b[CT];
    __device__ __forceinline__ Operands(const Loaded<CT> &x, uint32_t sh, uint32_t sh1) {
#pragma unroll
        for (int o = 0; o < 2; o++)
#pragma unroll
            for (int i = o; i < kTileWords + 2 + o; i++) {
                const int r = i & 3;
                const uint32_t s = o ? sh1 : sh;
                u[o][i] = i < 4 ? funnel32(x.m1[r], x.m0[r], s) : EDGE ? x.m1[r] : funnel32(x.m1[r], x.m0[r], s + 4u);
            }
#pragma unroll
        for (int c = 0; c < CT; c++)
            b[c] = x.b[c];
    }
    __device__ __forceinline__ void multiply(const mfma_v16f (&in)[CT][kTileWords],
                                             mfma_v16f (&out)[CT][kTileWords]) const {
#pragma unroll
        for (int jj = 0; jj < kTileWords; jj++) {
            const uint32_t *v = &u[jj & 1][jj];
            const mfma_v8i af = {(int)v[0], (int)v[1], (int)v[2], (int)v[3], 0, 0, 0, 0};
#pragma unroll
            for (int c = 0; c < CT; c++) {
                const v4i w = (v4i)b[c];
                out[c][jj] = mfma_bits_32x32x64(af, __builtin_shufflevector(w, w, 0, 1, 2, 3, -1, -1, -1, -1), in[c][jj]);
            }
        }
    }
};

// All kSteps product steps.  While one step's products run, the next step's
// operands are made and the one after's are loaded (interleave_step keeps the
// three mixed, so the matrix cores wait for neither).
template <int CT, bool EDGE>
__device__ __forceinline__ void products(const v4u *a, const v4u *b, uint32_t sh, const mfma_v16f &bias,
                                         mfma_v16f (&acc)[CT][kTileWords]) {
    const uint32_t sh1 = opaque(wave_uniform(sh));
    typedef Operands<CT, EDGE> Op;
    Loaded<CT> next(a, b, 1);
    Op x(Loaded<CT>(a, b, 0), sh, sh1);
    {
        mfma_v16f first[CT][kTileWords];
#pragma unroll
        for (int c = 0; c < CT; c++)
#pragma unroll
            for (int jj = 0; jj < kTileWords; jj++)
                first[c][jj] = bias;
        const Loaded<CT> l2(a, b, 2);
        const Op y(next, sh, sh1);
        x.multiply(first, acc);
        interleave_step<CT>();
        x = y;
        next = l2;
    }
    static_assert(kSteps % 2 == 0, "first and last step, pairs between");
#pragma nounroll
    for (int ks = 1; ks + 2 < kSteps; ks += 2) {
        const Loaded<CT> l2(a, b, ks + 2);
        const Op y(next, sh, sh1);
        x.multiply(acc, acc);
        interleave_step<CT>();
        // (the last pair's second load is not used: the last step again)
        const Loaded<CT> l3(a, b, ks + 3 < kSteps ? ks + 3 : kSteps - 1);
        const Op z(l2, sh, sh1);
        y.multiply(acc, acc);
        interleave_step<CT>();
        x = z;
        next = l3;
    }
    x.multiply(acc, acc);
}

// The products of one wave: CT column tiles, kTileWords words at a time.
template <int BITS, int CT>
__device__ __forceinline__ void tile_products(const v4u *A, const v4u *B, const JumpBlocks &G, const JumpTile &I, int g0, int g1,
                                              int pw) {
    const int l = threadIdx.x & (kWave - 1), wv = (int)wave_uniform(threadIdx.x / kWave);
    const int ncols = G.ncols, plane = I.plane;
    gu32 *P = reinterpret_cast<gu32 *>(G.parts) + plane * pw;
    mfma_v16f bias;
#pragma unroll
    for (int i = 0; i < 16; i++)
        bias[i] = 8388608.0f;  // 2^23: a count's parity is the sum's lowest mantissa bit
    static_assert(kJbGroup == kTileWaves * kTileWords, "a word group is one pass of the workgroup");
    for (int g = g0; g < g1; g++) {
        const int j0 = kJbGroup * g + kTileWords * wv;
        const v4u *a = A + (j0 >> 5) * 32 + l, *b = B + l;
        const uint32_t sh = (uint32_t)j0 & 31u;
        mfma_v16f acc[CT][kTileWords];
        wave_priority<2>();
        if (sh == 32 - kTileWords)
            products<CT, true>(a, b, sh, bias, acc);
        else
            products<CT, false>(a, b, sh, bias, acc);
        wave_priority<0>();
        // Lane L's accumulator r of word jj: bit 8 (r / 4) + 4 (L / 32) + r % 4
        // of the word, column L % 32.  Pack the 16 parities (bits 8 i + 4 + q),
        // exchange halves between words jj and jj + 2, and merge: the lower
        // lanes then hold words 0 and 1, the upper ones words 2 and 3.
#pragma unroll
        for (int c = 0; c < CT; c++) {
            uint32_t w[kTileWords];
#pragma unroll
            for (int jj = 0; jj < kTileWords; jj++) {
                uint32_t v = 0;
#pragma unroll
                for (int r = 0; r < 16; r++) {
                    if (r && r % 4 == 0)
                        v >>= 4;
                    v = funnel32(__float_as_uint(acc[c][jj][r]), v, 1);
                }
                w[jj] = v;
            }
#pragma unroll
            for (int jj = 0; jj < 2; jj++) {
                swap_halves(w[jj], w[jj + 2]);
                w[jj] = ((w[jj] >> 4) & 0x0f0f0f0fu) | (w[jj + 2] & 0xf0f0f0f0u);
            }
            const int col = I.c0 + 32 * c + (l & 31);
            if (col < ncols)
                *reinterpret_cast<gu2 *>(P + (uint64_t)col * (uint64_t)(BITS / 32 * pw) + (uint64_t)(j0 + 2 * (l >> 5))) =
                    v2u{w[0], w[1]};
        }
    }
}

template <int BITS, int NMAX>
__global__ __launch_bounds__(kTileThreads, 2) void jump_tiles_kernel(const JumpBlocks *__restrict__ groups,
                                                                     const JumpTile *__restrict__ tiles,
                                                                     const JumpShare *__restrict__ shares,
                                                                     const DevParam *__restrict__ params) {
    // 32-position rows the products read
    constexpr int ROWS = (((NMAX + kJbGroup - 1) / kJbGroup * kJbGroup - kTileWords) >> 5) + 2 * kSteps + 1;
    constexpr int SEQ = NMAX + kJbBlock;
    constexpr int SEQ_WORDS = BITS / 32 * SEQ, B_WORDS = kSteps * kWave * 4 * kJbCols / 32;
    __shared__ v4u A[ROWS * 32];
    // the sequence first, then (once A is made) the coefficients
    __shared__ __attribute__((aligned(16))) uint32_t R[SEQ_WORDS > B_WORDS ? SEQ_WORDS : B_WORDS];
    __shared__ uint32_t tbl[16];
    const int t = threadIdx.x, l = t & (kWave - 1), wv = t / kWave;
    const JumpShare S = shares[blockIdx.x];
    for (int ti = S.tile0; ti <= S.tile1; ti++) {
        const JumpTile I = ti == S.tile0 ? S.first : tiles[ti];
        const JumpBlocks &G = groups[I.group];
        const DevParam &D = params[I.param];
        const Rec p = rec_of(D);
        const bool make_a = ti == S.tile0 || I.c0 == 0;  // another base window or plane
        const int ncols = G.ncols;
        const int ct = ncols - I.c0 > 32 ? 2 : 1;
        // Loads first: the window (its last use comes before the
        // coefficients'), then this thread's coefficient words 4 cq + k of
        // columns cc + 32 i (i < ct), 16 bytes each (8 lanes of a wave share
        // cq, so that their stores of an operand are 128 bytes).
        const int cq = l >> 3, cc = 8 * wv + (l & 7);
        constexpr int NJ = (NMAX + kTileThreads - 1) / kTileThreads;
        uint32_t wh[NJ], wl[NJ];
        if (make_a) {
#pragma unroll
            for (int m = 0; m < NJ; m++) {
                const int j = t + kTileThreads * m;
                wh[m] = wl[m] = 0;
                if (BITS == 32) {
                    if (j < p.n)
                        wh[m] = reinterpret_cast<const gu32 *>(G.state_in)[j];
                } else if (j < p.n) {
                    const uint64_t v = reinterpret_cast<const gu64 *>(G.state_in)[j];
                    wh[m] = (uint32_t)(v >> 32);
                    wl[m] = (uint32_t)v;
                }
            }
        }
        v4u cw[kJbCols / 32];
#pragma unroll
        for (int i = 0; i < kJbCols / 32; i++) {
            const int c = I.c0 + 32 * i + cc;
            cw[i] = v4u{0, 0, 0, 0};
            if (c < ncols)
                cw[i] = reinterpret_cast<const gu4 *>(G.coef)[(uint64_t)c * (kJbWords / 4) + (uint64_t)cq];
        }
        if (ti != S.tile0)
            __syncthreads();  // the last tile's products
        if (make_a) {
            uint32_t *hi = R, *lo = R + (BITS == 64 ? SEQ : 0);
            if (t < 16)
                tbl[t] = D.tbl[t];
#pragma unroll
            for (int m = 0; m < NJ; m++) {
                const int j = t + kTileThreads * m;
                if (j < p.n) {
                    hi[j] = wh[m];
                    if (BITS == 64)
                        lo[j] = wl[m];
                }
            }
            __syncthreads();
            const int step = p.n - p.pos >= kTileThreads ? kTileThreads : kTileThreads / 2;
            for (int k = 0; k < kJbBlock; k += step) {
                if (t < step) {
                    uint32_t rh, rl;
                    next_word<BITS>(p, tbl, hi, lo, k + t, rh, rl);
                    hi[p.n + k + t] = rh;
                    if (BITS == 64)
                        lo[p.n + k + t] = rl;
                }
                __syncthreads();
            }
            // (positions past the sequence only meet words past the window's end)
            const uint32_t *src = BITS == 64 && I.plane ? lo : hi;
            const Transpose transpose;
            constexpr int PAIRS = (ROWS + 1) / 2, PER = (PAIRS + kTileWaves - 1) / kTileWaves;
#pragma unroll 4
            for (int m = 0; m < PER; m++) {
                const int x = 64 * (wv + kTileWaves * m) + l;
                const v4u e = fp4_expand(transpose(x < p.n + kJbBlock ? src[x] : 0u));
                if (x < 32 * ROWS)
                    A[x] = e;
            }
        }
        __syncthreads();
        // coefficient word w = 2 ks + kg of column 32 c + l is operand (ks, c),
        // lane 32 kg + l
        v4u *B = reinterpret_cast<v4u *>(R);
#pragma unroll
        for (int i = 0; i < kJbCols / 32; i++)
#pragma unroll
            for (int k = 0; k < 4; k++) {
                const int w = 4 * cq + k;
                if (i < ct)
                    B[((w >> 1) * ct + i) * kWave + 32 * (w & 1) + cc] = fp4_expand(cw[i][k]);
            }
        __syncthreads();
        const int pw = (p.n + kJbGroup - 1) / kJbGroup * kJbGroup;
        const int g0 = ti == S.tile0 ? S.g0 : 0, g1 = ti == S.tile1 ? S.g1 : pw / kJbGroup;
        if (ct == 2)
            tile_products<BITS, 2>(A, B, G, I, g0, g1, pw);
        else
            tile_products<BITS, 1>(A, B, G, I, g0, g1, pw);
    }
}

// ------------------------------------------------------------------- folds
// One workgroup per JumpFold: T threads, S numbers per step.  The chain of a
// block is 1 to 4 steps (8 in the narrow class), about as long as a load of its part can take (the
// tiles wrote it from any XCD, so it misses the L2), so parts are loaded
// kFoldAhead blocks ahead (one and four ahead, one jump: MTGP32-11213 8.8 and
// 7.6 us, MTGP64-23209 19.8 and 16.9, MTGP64-44497 28.5 and 24.4, MTGP64-
// 110503 70 and 60).
constexpr int kFoldAhead = 4;
template <int BITS, int NMAX, int S, int T>
__global__ __launch_bounds__(T) void jump_folds_kernel(const JumpBlocks *__restrict__ groups,
                                                       const JumpFold *__restrict__ folds,
                                                       const DevParam *__restrict__ params) {
    constexpr int NJ = (NMAX + T - 1) / T;
    constexpr int PL = BITS / 32;
    __shared__ uint32_t buf[PL][NMAX + kJbBlock];
    __shared__ uint32_t tbl[16];
    const int t = threadIdx.x;
    const JumpFold I = folds[blockIdx.x];
    const JumpBlocks &G = groups[I.group];
    const DevParam &D = params[G.param];
    const Rec p = rec_of(D);
    const int pw = (p.n + kJbGroup - 1) / kJbGroup * kJbGroup;
    const gu32 *P = reinterpret_cast<const gu32 *>(G.parts) + (uint64_t)I.b * (uint64_t)G.ch * (uint64_t)(PL * pw);
    if (t < 16)
        tbl[t] = D.tbl[t];
    // (lanes beyond the window repeat its last word)
    int at[NJ];
#pragma unroll
    for (int m = 0; m < NJ; m++)
        at[m] = t + T * m < p.n ? t + T * m : p.n - 1;
    uint32_t part[PL][NJ], ring[kFoldAhead][PL][NJ];
    const auto load = [&](uint32_t(&r)[PL][NJ], int a) {
        const gu32 *q = P + (uint64_t)(a > 0 ? a : 0) * (uint64_t)(PL * pw);
#pragma unroll
        for (int m = 0; m < NJ; m++)
#pragma unroll
            for (int h = 0; h < PL; h++)
                r[h][m] = q[h * pw + at[m]];
    };
    load(part, G.ch - 1);
#pragma unroll
    for (int i = 0; i < kFoldAhead; i++)
        load(ring[i], G.ch - 2 - i);
    for (int a = G.ch - 2; a >= 0;) {
#pragma unroll
        for (int i = 0; i < kFoldAhead; i++) {
            if (a < 0)
                break;
#pragma unroll
            for (int m = 0; m < NJ; m++)
#pragma unroll
                for (int h = 0; h < PL; h++)
                    buf[h][at[m]] = part[h][m];
            __syncthreads();
            for (int k = 0; k < kJbBlock; k += S) {
                uint32_t rh[S / T], rl[S / T];
#pragma unroll
                for (int i2 = 0; i2 < S / T; i2++)
                    next_word<BITS>(p, tbl, buf[0], buf[PL - 1], k + t + T * i2, rh[i2], rl[i2]);
#pragma unroll
                for (int i2 = 0; i2 < S / T; i2++) {
                    buf[0][p.n + k + t + T * i2] = rh[i2];
                    if (BITS == 64)
                        buf[PL - 1][p.n + k + t + T * i2] = rl[i2];
                }
                __syncthreads();
            }
#pragma unroll
            for (int m = 0; m < NJ; m++)
#pragma unroll
                for (int h = 0; h < PL; h++)
                    part[h][m] = ring[i][h][m] ^ buf[h][kJbBlock + at[m]];
            load(ring[i], a - kFoldAhead);
            a--;
            if (NMAX > kJbBlock)  // the window's old and new places overlap
                __syncthreads();
        }
    }
    if (BITS == 32) {
        gu32 *o = reinterpret_cast<gu32 *>(G.out + (uint64_t)I.b * G.out_stride);
#pragma unroll
        for (int m = 0; m < NJ; m++)
            if (t + T * m < p.n)
                o[t + T * m] = part[0][m];
    } else {
        gu64 *o = reinterpret_cast<gu64 *>(G.out + (uint64_t)I.b * G.out_stride);
#pragma unroll
        for (int m = 0; m < NJ; m++)
            if (t + T * m < p.n)
                o[t + T * m] = ((uint64_t)part[0][m] << 32) | part[PL - 1][m];
    }
}

template <class F>
auto with_class(int bits, int cls, F &&f) {
    if (bits == 32)
        return cls == 0   ? f.template operator()<32, 351>()
               : cls == 1 ? f.template operator()<32, 726>()
                          : f.template operator()<32, 1391>();
    return cls == 0   ? f.template operator()<64, 363>()
           : cls == 1 ? f.template operator()<64, 696>()
           : cls == 2 ? f.template operator()<64, 1727>()
                      : f.template operator()<64, 176>();
}

template <int BITS, int NMAX, int S>
hipError_t launch_fold(const JumpBlocks *groups, const JumpFold *folds, int n, const DevParam *params, hipStream_t s) {
    constexpr int T = S;
    hipLaunchKernelGGL((jump_folds_kernel<BITS, NMAX, S, T>), dim3(n), dim3(T), 0, s, groups, folds, params);
    return hipGetLastError();
}

}  // namespace

int jb_step(int bits, int cls, int n, int pos) {
    // the widest step with kernels for the class (128 in the narrow class)
    const int widest = bits == 64 && cls == 3 ? 128 : cls == 2 ? 1024 : cls == 1 ? 512 : 256;
    int step = widest;
    while (step > 128 && n - pos < step)
        step /= 2;
    return step;
}

hipError_t launch_jump_tiles(int bits, int cls, const JumpBlocks *groups, const JumpTile *tiles,
                             const JumpShare *shares, int n_shares, const DevParam *params, hipStream_t s) {
    if (n_shares <= 0)
        return hipSuccess;
    return with_class(bits, cls, [&]<int BITS, int NMAX>() {
        hipLaunchKernelGGL((jump_tiles_kernel<BITS, NMAX>), dim3(n_shares), dim3(kTileThreads), 0, s, groups, tiles,
                           shares, params);
        return hipGetLastError();
    });
}

hipError_t launch_jump_folds(int bits, int cls, int step, const JumpBlocks *groups, const JumpFold *folds, int n_folds,
                             const DevParam *params, hipStream_t s) {
    if (n_folds <= 0)
        return hipSuccess;
    return with_class(bits, cls, [&]<int BITS, int NMAX>() {
        if constexpr (NMAX > 726)
            if (step == 1024)
                return launch_fold<BITS, NMAX, 1024>(groups, folds, n_folds, params, s);
        if constexpr (NMAX > 363)
            if (step >= 512)
                return launch_fold<BITS, NMAX, 512>(groups, folds, n_folds, params, s);
        if constexpr (NMAX > 176)
            if (step >= 256)
                return launch_fold<BITS, NMAX, 256>(groups, folds, n_folds, params, s);
        if constexpr (NMAX == 176)
            return launch_fold<BITS, NMAX, 128>(groups, folds, n_folds, params, s);
        return hipErrorLaunchFailure;
    });
}

}  // namespace mtgp
