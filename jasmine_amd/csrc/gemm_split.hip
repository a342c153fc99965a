// The GEMM behind mat_dot_t / weight_net_t::forward and the runner's prefill: fp32 products
// on the bf16 matrix cores.
//
// Reference: mat_dot_t::operator() (mat_express_t.hpp:730-736), a scalar triple loop with
// sequential-k accumulation, reached from weight_net_t::forward (mat_net_t.hpp:38-49).
//
// v_mfma_f32_16x16x32_bf16 does 16 times the work of v_mfma_f32_16x16x4_f32 per cycle.  An
// fp32 number is exactly the sum of three bf16 numbers, x = h + m + l (each the rest rounded
// to nearest even: 8 significant bits of 24 each, |m| <= 2^-9 |x|, |l| <= 2^-18 |x|), and a
// product of two bf16 numbers is exact in fp32.  So
//   a b = hh + (hm + mh) + (mm + hl + lh) + (ml + lm + ll),
// and the six products of the first three groups leave out at most 2^-26 |a b| -- a quarter
// of the rounding of one fp32 multiplication.  All six accumulate in fp32, the small ones
// first; six MFMAs take 96 cycles where the fp32 ones take 256.  Weights stored as bf16 are
// their own h, and three products are exact (small ones first as well: prompt logits of a
// four-layer GPT-2-width model 4.8e-7 from 64 bits, 5.0e-7 with the large one first).
//
// The split happens once per element and workgroup, between the global load and LDS: slabs
// of 32 k are loaded to registers a slab ahead, split, and written to LDS as three planes
// of bf16 in MFMA operand order, so that every fragment read is one ds_read_b128.  (Small
// products skip LDS: gemm_split_k_kernel.)
//
// Lane l of a wave (r16 = l % 16, g = l / 16) holds slots j = 0..7 of row r16 in both
// operands: k = 4 g + j for j < 4 and 16 + 4 g + j - 4 above -- a permutation of the slab's k
// applied to A and B alike, and the one the packed weight layouts already have.
//
// Numbers outside the split's range.  Infinities, NaN and magnitudes that round to infinity
// in bf16 make the six-product sum non-finite.  Magnitudes below 2^-110 lose the bits of m and
// l under bf16's smallest step, below 2^-134 all of h too: at most 2^-134 per element, so an
// error of at most K 2^-134 (max|A| + max|B|) in a sum -- more than 2^-24 of it only if the sum
// is below K 2^-110 (max|A| + max|B|), which a sum of zero always is.  The rows and columns of a few
// such sums, or a tile with many, are looked over for operands below 2^-110 that are not zero; a tile
// that has one, or a sum that is not finite, is computed again on the fp32 matrix cores (SplitRange).
// MI355X: 1024^3, 22 us, 32 where every tile is looked over (zeros in each), 55 where every one is
// computed again; 4096 x 4096 x 1024, 205 us: 211 with a row of zeros in each tile, 670 computed again;
// 4096^3, 667 us: 700 with one sum that cancels to zero.  Beside packed bf16 weights, which need no split, the
// activations are split times 2^16, which loses nothing, and only sums that are not finite count.
#include "gemm.hpp"
#include "split.hpp"

#include <cfloat>
#include <type_traits>
#include <utility>

namespace jas {

typedef float f32x4u __attribute__((ext_vector_type(4), aligned(4)));  // rows need not be aligned
typedef float f32x2u __attribute__((ext_vector_type(2), aligned(4)));

// Extremes of a lane's six-product sums, and what they call for
struct SplitRange {
    float hi = 0.f, lo = INFINITY;
    __device__ __forceinline__ void add(floatx4 v)
    {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            hi = __builtin_elementwise_maximum(hi, fabsf(v[r]));  // propagates NaN
            lo = fminf(lo, fabsf(v[r]));
        }
    }
    enum : int { OK = 0, LOOK = 1, REDO = 2 };
    // sums below this, of operands up to `largest`, may have lost too much
    __device__ __forceinline__ static float bound(float largest, int K) { return 2.f * (float)K * 0x1p-110f * largest; }
    // limit: the largest number, or less where further sums follow
    __device__ __forceinline__ int check(float limit, float largest, int K) const
    {
        return !(hi <= limit) ? REDO : lo < bound(largest, K) ? LOOK : OK;
    }
};

// the largest of lanes r16, r16 + 16, r16 + 32 and r16 + 48
__device__ __forceinline__ float max_over_g(float v)
{
    v = fmaxf(v, __shfl_xor(v, 16, WAVE));
    return fmaxf(v, __shfl_xor(v, 32, WAVE));
}

// One operand X(o, k) of a workgroup: its T x 32 slabs from memory to registers to LDS.  SCALED: its
// planes are those of 2^16 X, exact for every magnitude up to 2^111 (beside bf16 weights, whose
// magnitudes are not tracked).
// A wave moves units of 16 rows (32 outer-contiguous ones); unit u belongs to wave u % NW.
template <int MODE, int T, int NW, bool SCALED = false>
struct SplitLoader {
    static constexpr int OW = MODE == SM_OC ? 32 : 16, UNITS = T / OW, UPW = (UNITS + NW - 1) / NW;
    static constexpr int NR = MODE == SM_OC ? 16 : MODE == SM_PKB ? 4 : 8;
    static constexpr int PL = MODE == SM_PKB ? 1 : 3, NB = T / 16;  // planes, 16-row blocks
    typedef float regs_t[UPW][NR];
    static constexpr int R = MODE == SM_OC ? 2 : 1;  // rows per lane and unit
    typedef float max_t[UPW * R];                    // largest magnitude in each of them

    const float *X;
    long so, sk;
    int K, Olim;
    int o[UPW], ou[UPW];    // this lane's (first) outer index, unclamped; its unit's first
    const float *base[UPW]; // its address at k = 4 g (packed: the tile array)
    long rt[UPW], RG;       // packed: row tile, row tiles

    __device__ __forceinline__ static bool mine(int w, int q) { return UNITS % NW == 0 || w + q * NW < UNITS; }

    __device__ __forceinline__ void init(const float *X_, const float *X2, long so_, long sk_, int o0, int Olim_, int K_,
                                         int w, int lane)
    {
        X = X_, so = so_, sk = sk_, K = K_, Olim = Olim_;
        const int i = lane & 15, g = lane >> 4;
#pragma unroll
        for (int q = 0; q < UPW; ++q) {
            const int u = w + q * NW;
            if constexpr (MODE == SM_PK || MODE == SM_PKB) {
                RG = (Olim + 15) >> 4;
                long t = min((long)(o0 >> 4) + u, RG - 1);
                const float *Xm = X;
                if (X2) {  // SwiGLU: virtual row tile 2f is gate tile f, 2f + 1 up tile f
                    Xm = t & 1 ? X2 : X;
                    t >>= 1;
                    RG >>= 1;
                }
                rt[q] = t;
                base[q] = Xm;
            } else if constexpr (MODE == SM_OC) {
                ou[q] = o0 + 32 * u;
                o[q] = ou[q] + 2 * i;
                base[q] = X + min(o[q], max(Olim - 2, 0)) + 4 * g * sk;
            } else {
                o[q] = min(o0 + 16 * u + i, Olim - 1);
                base[q] = X + o[q] * so + 4 * g * sk;
            }
        }
    }

    // slab [k0, k0 + 32), inside K (packed bf16: inside K padded to 32)
    __device__ __forceinline__ void load(regs_t &r, int k0, int w, int lane) const
    {
#pragma unroll
        for (int q = 0; q < UPW; ++q) {
            if (!mine(w, q)) continue;
            if constexpr (MODE == SM_KC) {
                const f32x4u a = *(const f32x4u *)(base[q] + k0), b = *(const f32x4u *)(base[q] + k0 + 16);
#pragma unroll
                for (int e = 0; e < 4; ++e) r[q][e] = a[e], r[q][4 + e] = b[e];
            } else if constexpr (MODE == SM_OC) {
                if (ou[q] + 32 <= Olim) {  // whole unit inside (wave-uniform)
#pragma unroll
                    for (int j = 0; j < 8; ++j) {
                        const f32x2u v = *(const f32x2u *)(base[q] + (long)(k0 + j + (j < 4 ? 0 : 12)) * sk);
                        r[q][2 * j] = v[0], r[q][2 * j + 1] = v[1];
                    }
                } else {
                    load_edge(r, q, k0, lane);
                }
            } else if constexpr (MODE == SM_GEN) {
#pragma unroll
                for (int j = 0; j < 8; ++j) r[q][j] = base[q][(long)(k0 + j + (j < 4 ? 0 : 12)) * sk];
            } else if constexpr (MODE == SM_PK) {
                const int kb = k0 >> 4;
                const floatx4 a = *(const floatx4 *)(base[q] + weight_tile_offset(rt[q], kb, K >> 4, RG) + lane * 4);
                const floatx4 b = *(const floatx4 *)(base[q] + weight_tile_offset(rt[q], kb + 1, K >> 4, RG) + lane * 4);
#pragma unroll
                for (int e = 0; e < 4; ++e) r[q][e] = a[e], r[q][4 + e] = b[e];
            } else {
                const floatx4 a = *(const floatx4 *)((const uint16_t *)(const void *)base[q] +
                                                     weight_tile_offset_b(rt[q], k0 >> 5, k32_of(K), RG) + lane * 8);
#pragma unroll
                for (int e = 0; e < 4; ++e) r[q][e] = a[e];
            }
        }
    }

    // outer-contiguous unit that crosses the last row, or the last, partial slab: one element
    // at a time, rows clamped, zeros from K on
    __device__ __forceinline__ void load_edge(regs_t &r, int q, int k0, int lane) const
    {
        const int g = lane >> 4;
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const int k = k0 + 4 * g + j + (j < 4 ? 0 : 12), kc = k < K ? k : 0;
            if constexpr (MODE == SM_OC) {
#pragma unroll
                for (int e = 0; e < 2; ++e) {
                    const float v = X[min(o[q] + e, Olim - 1) + kc * sk];
                    r[q][2 * j + e] = k < K ? v : 0.f;
                }
            } else {
                const float v = X[o[q] * so + kc * sk];
                r[q][j] = k < K ? v : 0.f;
            }
        }
    }

    __device__ __forceinline__ void load_tail(regs_t &r, int k0, int w, int lane) const
    {
        if constexpr (MODE == SM_PKB) {  // zero-padded to 32
            load(r, k0, w, lane);
        } else {
#pragma unroll
            for (int q = 0; q < UPW; ++q) {
                if (!mine(w, q)) continue;
                if constexpr (MODE == SM_PK) {  // K % 16 == 0: the first half slab exists
                    const floatx4 a = *(const floatx4 *)(base[q] + weight_tile_offset(rt[q], k0 >> 4, K >> 4, RG) + lane * 4);
#pragma unroll
                    for (int e = 0; e < 4; ++e) r[q][e] = a[e], r[q][4 + e] = 0.f;
                } else {
                    load_edge(r, q, k0, lane);
                }
            }
        }
    }

    // operand registers of this lane for its q-th unit (K-contiguous, general or packed)
    __device__ __forceinline__ static void planes(const regs_t &r, int q, float &mx, bf16x8 (&pl)[PL])
    {
        if constexpr (MODE == SM_PKB) {
            pl[0] = __builtin_bit_cast(bf16x8, floatx4{r[q][0], r[q][1], r[q][2], r[q][3]});
        } else {
            float x[8];
#pragma unroll
            for (int j = 0; j < 8; ++j) x[j] = r[q][j];
            if constexpr (!SCALED) track_max(mx, x);
            u32x4 h, m, l;
            split8<SCALED>(x, h, m, l);
            pl[0] = __builtin_bit_cast(bf16x8, h);
            pl[1] = __builtin_bit_cast(bf16x8, m);
            pl[2] = __builtin_bit_cast(bf16x8, l);
        }
    }

    // planes of the slab in registers -> LDS: plane pl, 16-row block b, lane slot: [(pl * NB + b)
    // * 64 + slot].  Lanes 8..15 of a 16-row group swap pairs (slot ^ 1), which keeps the stores
    // of outer-contiguous units (two rows per lane, every other slot) off each other's banks.
    __device__ __forceinline__ static int slot_of(int r16, int g) { return (r16 + 16 * g) ^ (r16 >> 3); }

    __device__ __forceinline__ void store(const regs_t &r, u32x4 *lds, int w, int lane, max_t &mx) const
    {
        const int i = lane & 15, g = lane >> 4;
#pragma unroll
        for (int q = 0; q < UPW; ++q) {
            if (!mine(w, q)) continue;
            const int u = w + q * NW;
            if constexpr (MODE == SM_PKB) {
                lds[u * 64 + slot_of(i, g)] = __builtin_bit_cast(u32x4, floatx4{r[q][0], r[q][1], r[q][2], r[q][3]});
            } else {
#pragma unroll
                for (int e = 0; e < R; ++e) {
                    float x[8];
#pragma unroll
                    for (int j = 0; j < 8; ++j) x[j] = r[q][R * j + e];
                    u32x4 h, m, l;
                    if constexpr (!SCALED) track_max(mx[q * R + e], x);
                    split8<SCALED>(x, h, m, l);
                    const int row = MODE == SM_OC ? 2 * (i & 7) + e : i, blk = MODE == SM_OC ? 2 * u + (i >> 3) : u;
                    u32x4 *d = lds + blk * 64 + slot_of(row, g);
                    d[0] = h;
                    d[NB * 64] = m;
                    d[2 * NB * 64] = l;
                }
            }
        }
    }

    // over all slabs a wave has moved: one value for all its lanes' rows, and each row's into out[row]
    __device__ __forceinline__ static float largest(const max_t &mx)
    {
        float v = 0.f;
#pragma unroll
        for (int q = 0; q < UPW * R; ++q) v = fmaxf(v, mx[q]);
        return v;
    }
    __device__ __forceinline__ static void store_max(const max_t &mx, float *out, int w, int lane)
    {
#pragma unroll
        for (int q = 0; q < UPW; ++q) {
            if (!mine(w, q)) continue;
#pragma unroll
            for (int e = 0; e < R; ++e) {
                const float v = max_over_g(mx[q * R + e]);
                if (lane < 16) out[(w + q * NW) * OW + R * lane + e] = v;
            }
        }
    }

    // whether a slab in registers has a nonzero value below 2^-110 (bf16 weights need no split)
    __device__ __forceinline__ static bool has_tiny(const regs_t &r, int w)
    {
        bool tiny = false;
        if constexpr (MODE != SM_PKB) {
#pragma unroll
            for (int q = 0; q < UPW; ++q)
                if (mine(w, q)) {
#pragma unroll
                    for (int e = 0; e < NR; ++e) tiny |= 2 * __float_as_uint(r[q][e]) - 1 < 2 * __float_as_uint(0x1p-110f) - 1;
                }
        }
        return tiny;
    }

    // one element (the fp32 recomputation); zero from K on
    __device__ __forceinline__ static float element(const float *X, const float *X2, long so, long sk, int o, int k, int Olim,
                                                    int K)
    {
        if (k >= K) return 0.f;
        if constexpr (MODE == SM_PK || MODE == SM_PKB) {
            long RG = (Olim + 15) >> 4;
            const float *Xm = X;
            if (X2) {
                const int t = o >> 4;
                Xm = t & 1 ? X2 : X;
                o = (t >> 1) * 16 + (o & 15);
                RG >>= 1;
            }
            if (MODE == SM_PK) return Xm[weight_pack_offset(o, k, K, RG)];
            return bf16_to_f32(((const uint16_t *)(const void *)Xm)[weight_pack_offset_b(o, k, K, RG)]);
        }
        return X[o * so + k * sk];
    }
};

// acc += A B over k = first + g, first + stride + g, ... below K on the fp32 matrix cores, operands
// element by element: blocks of 16 rows from m on and 16 columns from n on
template <typename LA, typename LB, int NBI, int NBJ>
__device__ __forceinline__ void multiply_fp32(const SplitArgs &p, const float *A, const float *B, int m, int n, int first,
                                              int stride, int lane, floatx4 (&acc)[NBI][NBJ])
{
    // addresses of its own: those of the main loop would otherwise be kept in registers throughout
    asm volatile("" : "+v"(lane));
    const int r16 = lane & 15, g = lane >> 4;
#pragma unroll 1
    for (int k = first; k < p.K; k += stride) {  // (the same count for every lane; element() is zero from K on)
        float av[NBI], bv[NBJ];
#pragma unroll
        for (int i = 0; i < NBI; ++i)
            av[i] = LA::element(A, p.fz.A2, p.as0, p.as1, min(m + 16 * i + r16, p.M - 1), k + g, p.M, p.K);
#pragma unroll
        for (int j = 0; j < NBJ; ++j)
            bv[j] = LB::element(B, nullptr, p.bs1, p.bs0, min(n + 16 * j + r16, p.N - 1), k + g, p.N, p.K);
#pragma unroll
        for (int i = 0; i < NBI; ++i)
#pragma unroll
            for (int j = 0; j < NBJ; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(av[i], bv[j], acc[i][j], 0, 0, 0);
    }
}

// Whether slabs first, first + step, ... of a tile hold a nonzero operand below 2^-110, in wave wa's
// units of A and wave wb's of B
template <typename LA, typename LB>
__device__ __forceinline__ bool tiny_operand(const SplitArgs &p, const float *A, const float *B, int m0, int n0, int first,
                                             int step, int wa, int wb, int lane)
{
    asm volatile("" : "+v"(lane));  // (as above)
    LA la;
    LB lb;
    la.init(A, p.fz.A2, p.as0, p.as1, m0, p.M, p.K, wa, lane);
    lb.init(B, nullptr, p.bs1, p.bs0, n0, p.N, p.K, wb, lane);
    bool tiny = false;
#pragma unroll 1
    for (int k0 = first * 32; k0 < p.K; k0 += step * 32) {
        typename LA::regs_t ra;
        typename LB::regs_t rb;
        if (k0 + 32 <= p.K) {
            la.load(ra, k0, wa, lane);
            lb.load(rb, k0, wb, lane);
        } else {
            la.load_tail(ra, k0, wa, lane);
            lb.load_tail(rb, k0, wb, lane);
        }
        tiny |= LA::has_tiny(ra, wa) || LB::has_tiny(rb, wb);
    }
    return tiny;
}

// The same for the rows and columns of a wave's sums below `bound` alone, if there are at most eight
// (`many`: there are more); blocks of 16 rows from m on and 16 columns from n on.  Sums of ordinary
// numbers cancel to zero now and then (one of 10^8 at K = 4096), and one tile looked over as a whole is
// 95 us of a 4096^3 product's 667 (its row and column 30).  Sums of a row or column of zeros (rm, cm:
// the largest magnitudes) are zero rightly: 4096^3 with a zero row in every tile 890 us when those were
// looked over, 667 without.
template <typename LA, typename LB, int NBI, int NBJ, typename RM, typename CM>
__device__ __forceinline__ bool tiny_lines(const SplitArgs &p, const float *A, const float *B, int m, int n, int first, int step,
                                           int lane, const floatx4 (&acc)[NBI][NBJ], RM rm, CM cm, float bound, bool &many)
{
    asm volatile("" : "+v"(lane));  // (as above)
    static_assert(NBI * NBJ <= 16, "a bit per sum");
    uint64_t bits = 0;
#pragma unroll
    for (int i = 0; i < NBI; ++i)
#pragma unroll
        for (int j = 0; j < NBJ; ++j)
#pragma unroll
            for (int r = 0; r < 4; ++r)
                if (fabsf(acc[i][j][r]) < bound && rm(i, r) > 0.f && cm(j) > 0.f) bits |= 1ull << (4 * (i * NBJ + j) + r);
    many = wave_sum((float)__popcll(bits)) > 8.f;
    if (many) return false;
    bool tiny = false;
    for (uint64_t lanes = __builtin_amdgcn_ballot_w64(bits != 0); lanes; lanes = __builtin_amdgcn_ballot_w64(bits != 0)) {
        const int l = __builtin_ctzll(lanes);
        const uint64_t b = (uint64_t)(unsigned)__builtin_amdgcn_readlane((int)(bits >> 32), l) << 32 |
                           (unsigned)__builtin_amdgcn_readlane((int)bits, l);
        const int at = __builtin_ctzll(b), blk = at / 4;
        const int row = min(m + 16 * (blk / NBJ) + 4 * (l >> 4) + at % 4, p.M - 1), col = min(n + 16 * (blk % NBJ) + (l & 15), p.N - 1);
        if (lane == l) bits &= bits - 1;
#pragma unroll 8
        for (int k0 = first * 32; k0 < p.K; k0 += step * 32) {  // a slab of the row in lanes 0..31, of the column above
            const int k = k0 + (lane & 31);
            const float v = lane < 32 ? LA::element(A, p.fz.A2, p.as0, p.as1, row, k, p.M, p.K)
                                      : LB::element(B, nullptr, p.bs1, p.bs0, col, k, p.N, p.K);
            tiny |= 2 * __float_as_uint(v) - 1 < 2 * __float_as_uint(0x1p-110f) - 1;
        }
    }
    return tiny;
}

// Workgroup ids are remapped so that each of the 8 XCDs (ids go round-robin over them)
// works on a contiguous range of tiles, walked 4 tile rows at a time: the A rows and B
// columns its workgroups share stay in that XCD's L2.
__device__ __forceinline__ void tile_of_workgroup(int &bx, int &by)
{
    constexpr int XG = 4;
    const int gx = gridDim.x, nt = gx * gridDim.y, per = nt / 8;
    const int id = blockIdx.y * gx + blockIdx.x;
    // a permutation of the ids: the first 8 * per go XCD-contiguous, the rest stay
    const int lid = id < 8 * per ? (id % 8) * per + id / 8 : id;
    const int grp = lid / (XG * gx), gy0 = grp * XG, rows = min(XG, (int)gridDim.y - gy0);
    const int in = lid - grp * XG * gx;
    by = gy0 + in % rows;
    bx = in / rows;
}

// What the plain epilogue adds to output rows m .. m + 3 of column n: bias and residual (rows
// past M: the last row's, not stored).
struct EpiOperands {
    float bias[4], resid[4];
    __device__ __forceinline__ void load(const SplitArgs &p, const float *b, int m, int n)
    {
        const int mc = min(m, p.M - 1), nc = min(n, p.N - 1);
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int mr = min(mc + r, p.M - 1);
            bias[r] = b ? b[p.bias_mode == 1 ? mr : nc] : 0.f;
            resid[r] = p.resid ? p.resid[(long)mr * p.rs0 + (long)nc * p.rs1] : 0.f;
        }
    }
};

// Output rows m .. m + 3, column n, from their sums a (SwiGLU: the gate sums, u the up sums of
// the same outputs; m counts gate and up rows in alternating tiles of 16).
__device__ __forceinline__ void split_epilogue(const SplitArgs &p, float *C, const float *bias, const EpiOperands &eo, int m,
                                               int n, floatx4 a, floatx4 u)
{
    if (n >= p.N || m >= p.M) return;
    if (p.fz.mode == FZ_SWIGLU) {
        const int f = (m >> 5) * 16 + (m & 15);  // output feature of this lane's first row
        *(float4 *)(C + f + (long)n * p.cs1) =
            make_float4(silu_f(a[0]) * u[0], silu_f(a[1]) * u[1], silu_f(a[2]) * u[2], silu_f(a[3]) * u[3]);
        return;
    }
    if (p.fz.mode == FZ_QKV) {
        // rows [0, d) q, [d, 2d) k, [2d, 3d) v of token n: bias, rotary on q and k (pairs
        // (2i, 2i+1) of a head are (0, 1) and (2, 3) here), the row, and k / v into the KV
        // cache at the token's position
        const PrefillFused &zf = p.fz;
        float v[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) v[r] = bias ? a[r] + bias[m + r] : a[r];
        const int sec = m / zf.d, e = m % zf.dh, hh = (m % zf.d) / zf.dh;
        const int t = zf.pos[n];
        if (zf.rope && sec < 2) {
#pragma unroll
            for (int pr = 0; pr < 2; ++pr) {
                const double2 cs = zf.rope_tab[(long)t * (zf.dh / 2) + (e >> 1) + pr];
                const float x0 = v[2 * pr], x1 = v[2 * pr + 1];
                v[2 * pr] = (float)(x0 * cs.x - x1 * cs.y);
                v[2 * pr + 1] = (float)(x0 * cs.y + x1 * cs.x);
            }
        }
        *(float4 *)(C + m + (long)n * p.cs1) = make_float4(v[0], v[1], v[2], v[3]);
        if (sec >= 1) {
            const int bseq = n / zf.P;
            const long dst = (((long)bseq * zf.H + hh) * zf.ctx + t) * zf.dh + e;
            *(float4 *)((sec == 1 ? zf.kc : zf.vc) + dst) = make_float4(v[0], v[1], v[2], v[3]);
        }
        return;
    }
    const int nv = min(4, p.M - m);
    float *cp = C + (long)m * p.cs0 + (long)n * p.cs1;
    float v[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        float x = a[r];
        if (bias) x = x + eo.bias[r];
        x = apply_act(x, p.act);
        if (p.resid) x = x + eo.resid[r];
        v[r] = p.accumulate ? cp[min(r, nv - 1) * p.cs0] + x : x;
    }
    if (p.cs0 == 1 && nv == 4) {
        *(f32x4u *)cp = f32x4u{v[0], v[1], v[2], v[3]};
    } else {
#pragma unroll
        for (int r = 0; r < 4; ++r)
            if (r < nv) cp[r * p.cs0] = v[r];
    }
}

// Large products.  TM x TN tile, NW waves in a WGM x (NW / WGM) grid, two slabs of LDS.  A
// workgroup splits each element once; per slab and CU a 256 x 128 tile needs 3072 cycles of
// matrix core, about 900 of vector ALU, 2100 of LDS.  MI355X, 4096^3: 1083 us on the fp32
// matrix cores (127 TFLOP/s), 690 us here (199 TFLOP/s of fp32 products, 1.2 PFLOP/s of bf16
// ones, the rate a plain bf16 product of this size reaches).  A slab takes about 6400 cycles: the
// waves leave its barrier together, and their phases add up rather than overlap (matrix cores busy
// 0.48).
//
// SUMS (where tiles compete with waves that split K): a slab's six products add up by themselves,
// then to the sum, so a slab rounds the long sum once and not six times: the error is that of four
// waves' sums or less.  SUMS_FEW: and the last slab is not loaded again (see below).
enum SlabSums : int { PLAIN = 0, SUMS = 1, SUMS_FEW = 2 };
template <int AM, int BM, int TM, int TN, int NW, int WGM, int FORM = PLAIN>
__global__ void __launch_bounds__(NW * 64, 2) gemm_split_kernel(const SplitArgs p)
{
    constexpr int WGN = NW / WGM, NBI = TM / WGM / 16, NBJ = TN / WGN / 16;
    constexpr bool TWO = FORM != PLAIN;
    using LA = SplitLoader<AM, TM, NW>;
    using LB = SplitLoader<BM, TN, NW, AM == SM_PKB>;
    constexpr int PA = LA::PL, SA = PA * TM * 4, SB = 3 * TN * 4;  // 16-byte units per stage
    static_assert(LB::PL == 3, "B is fp32");
    __shared__ u32x4 lds[2 * (SA + SB)];
    const int tid = threadIdx.x, lane = tid & 63;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = w / WGN, wn = w % WGN, r16 = lane & 15, g = lane >> 4;

    int bx, by;
    tile_of_workgroup(bx, by);
    const int m0 = by * TM, n0 = bx * TN;
    const long bz = blockIdx.z;
    const float *A = p.A + bz * p.abs_;
    const float *B = p.B + bz * p.bbs;
    const int K = p.K, nk = K / 32;

    LA la;
    LB lb;
    const int wb = NW - 1 - w;  // B's units start from the last wave: small tiles use all waves
    la.init(A, p.fz.A2, p.as0, p.as1, m0, p.M, K, w, lane);
    lb.init(B, nullptr, p.bs1, p.bs0, n0, p.N, K, wb, lane);

    floatx4 acc[NBI][NBJ];
#pragma unroll
    for (int i = 0; i < NBI; ++i)
#pragma unroll
        for (int j = 0; j < NBJ; ++j) acc[i][j] = floatx4{0.f, 0.f, 0.f, 0.f};
    const int rslot = LA::slot_of(r16, g);
    auto compute = [&](const u32x4 *sa) {
        const u32x4 *pa = sa + wm * NBI * 64 + rslot, *pb = sa + SA + wn * NBJ * 64 + rslot;
        bf16x8 b[NBJ][3];
#pragma unroll
        for (int j = 0; j < NBJ; ++j)
#pragma unroll
            for (int pl = 0; pl < 3; ++pl) b[j][pl] = __builtin_bit_cast(bf16x8, pb[(pl * LB::NB + j) * 64]);
#pragma unroll
        for (int i = 0; i < NBI; ++i) {
            bf16x8 a[PA];
#pragma unroll
            for (int pl = 0; pl < PA; ++pl) a[pl] = __builtin_bit_cast(bf16x8, pa[(pl * LA::NB + i) * 64]);
            floatx4 slab[NBJ];  // TWO
#pragma unroll
            for (int j = 0; j < NBJ; ++j) slab[j] = floatx4{0.f, 0.f, 0.f, 0.f};
            // small products first; the NBJ accumulators innermost
            auto mul = [&](int ia, int ib) {
#pragma unroll
                for (int j = 0; j < NBJ; ++j) {
                    floatx4 &d = TWO ? slab[j] : acc[i][j];
                    d = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[ia], b[j][ib], d, 0, 0, 0);
                }
            };
            if constexpr (PA == 3) {
                mul(2, 0);
                mul(0, 2);
                mul(1, 1);
                mul(1, 0);
                mul(0, 1);
                mul(0, 0);
            } else {
                mul(0, 2);
                mul(0, 1);
                mul(0, 0);
            }
            if constexpr (TWO) {
#pragma unroll
                for (int j = 0; j < NBJ; ++j) acc[i][j] += slab[j];
            }
        }
    };

    typename LA::max_t mxa = {};
    typename LB::max_t mxb = {};
    typename LA::regs_t ra;
    typename LB::regs_t rb;
    auto fetch = [&](int k0) {
        la.load(ra, k0, w, lane);
        lb.load(rb, k0, wb, lane);
    };
    // Slab s goes to stage s % 2, which was last read two slabs ago, before the barrier of the
    // slab in between: one barrier per slab.  The loads of the next slab are issued whether or
    // not it exists (past the last one: the last again), so the wait counts do not depend on
    // the path.  Where there are few slabs, one load more is dearer than the waits (3072 x 509 x 64
    // 8.4 us with it, 7.7 without; 1024^2 x 768 20.8 and 22.7).
    auto step = [&](int s, bool more) {
        u32x4 *sa = lds + (s & 1) * (SA + SB);
        la.store(ra, sa, w, lane, mxa);
        lb.store(rb, sa + SA, wb, lane, mxb);
        if (more && (FORM != SUMS_FEW || s + 1 < nk)) fetch(min(s + 1, nk - 1) * 32);
        __syncthreads();
        compute(sa);
    };
    if (nk > 0) fetch(0);
    for (int s = 0; s < nk; ++s) step(s, true);
    if (nk * 32 < K) {  // partial last slab
        la.load_tail(ra, nk * 32, w, lane);
        lb.load_tail(rb, nk * 32, wb, lane);
        step(nk, false);
    }

    // a sum outside the split's range anywhere in the tile: compute the tile again in fp32
    __shared__ float smax[NW];
    const float mx = wave_max(fmaxf(LA::largest(mxa), LB::largest(mxb)));
    if (lane == 0) smax[w] = mx;
    __syncthreads();
    float largest = smax[0];
#pragma unroll
    for (int k = 1; k < NW; ++k) largest = fmaxf(largest, smax[k]);
    SplitRange range;
#pragma unroll
    for (int i = 0; i < NBI; ++i)
#pragma unroll
        for (int j = 0; j < NBJ; ++j) range.add(acc[i][j]);
    const int need = range.check(FLT_MAX, largest, K);
    float unscale = AM == SM_PKB ? SPLIT_UNSCALE : 1.f;
    if (__syncthreads_or(need)) {
        bool redo = need == SplitRange::REDO;
        float *lines = (float *)lds;  // (every wave has read its last operands)
        LA::store_max(mxa, lines, w, lane);
        LB::store_max(mxb, lines + TM, wb, lane);
        if (!__syncthreads_or(redo)) {
            bool many;
            auto rm = [&](int i, int r) { return lines[(wm * NBI + i) * 16 + 4 * g + r]; };
            auto cm = [&](int j) { return lines[TM + (wn * NBJ + j) * 16 + r16]; };
            redo = tiny_lines<LA, LB>(p, A, B, m0 + wm * NBI * 16, n0 + wn * NBJ * 16, 0, 1, lane, acc, rm, cm,
                                      SplitRange::bound(largest, K), many);
            if (__syncthreads_or(many)) redo = tiny_operand<LA, LB>(p, A, B, m0, n0, 0, 1, w, wb, lane);
        }
        if (__syncthreads_or(redo)) {
            unscale = 1.f;
#pragma unroll
            for (int i = 0; i < NBI; ++i)
#pragma unroll
                for (int j = 0; j < NBJ; ++j) acc[i][j] = floatx4{0.f, 0.f, 0.f, 0.f};
            multiply_fp32<LA, LB>(p, A, B, m0 + wm * NBI * 16, n0 + wn * NBJ * 16, 0, 4, lane, acc);
        }
    }

    if constexpr (AM == SM_PKB) {
#pragma unroll
        for (int i = 0; i < NBI; ++i)
#pragma unroll
            for (int j = 0; j < NBJ; ++j) acc[i][j] *= unscale;
    }
    // epilogue: block (i, j) of a lane holds rows 4 g .. 4 g + 3, column r16
    float *C = p.C + bz * p.cbs;
    const float *bias = p.bias ? p.bias + bz * p.biasbs : nullptr;
    const int mw = m0 + wm * NBI * 16 + 4 * g, nw = n0 + wn * NBJ * 16 + r16;
    if (p.fz.mode == FZ_SWIGLU) {
#pragma unroll
        for (int i = 0; i + 1 < NBI; i += 2)
#pragma unroll
            for (int j = 0; j < NBJ; ++j)
                split_epilogue(p, C, bias, EpiOperands{}, mw + 16 * i, nw + 16 * j, acc[i][j], acc[i + 1][j]);
        return;
    }
#pragma unroll
    for (int i = 0; i < NBI; ++i)
#pragma unroll
        for (int j = 0; j < NBJ; ++j) {
            EpiOperands eo;
            eo.load(p, bias, mw + 16 * i, nw + 16 * j);
            split_epilogue(p, C, bias, eo, mw + 16 * i, nw + 16 * j, acc[i][j], acc[i][j]);
        }
}

// Small products: a workgroup's tile is 16 NBI x 16 NBJ, and its NW waves split K -- wave w
// takes slabs w, w + NW, ... and holds the whole tile.  Operands go from memory straight to
// the lanes that need them (no LDS, no barrier in the loop), so a short K is about one memory
// round trip; the waves' sums meet in LDS and are added in wave order.
template <int AM, int BM, int NBI, int NBJ, int NW, int PD>
__global__ void __launch_bounds__(NW * 64, 2) gemm_split_k_kernel(const SplitArgs p)
{
    constexpr int TM = 16 * NBI, TN = 16 * NBJ, NBLK = NBI * NBJ;
    constexpr bool TWO = NW == 2;  // (as above: two waves' sums would be longer than four's)
    using LA = SplitLoader<AM, TM, 1>;
    using LB = SplitLoader<BM, TN, 1, AM == SM_PKB>;
    constexpr int PA = LA::PL;
    __shared__ floatx4 red[NW][NBLK][64];
    __shared__ int need[NW];
    const int tid = threadIdx.x, lane = tid & 63;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int r16 = lane & 15, g = lane >> 4;
    int bx, by;
    tile_of_workgroup(bx, by);
    const int m0 = by * TM, n0 = bx * TN;
    const long bz = blockIdx.z;
    const float *A = p.A + bz * p.abs_;
    const float *B = p.B + bz * p.bbs;
    const int K = p.K;

    LA la;
    LB lb;
    la.init(A, p.fz.A2, p.as0, p.as1, m0, p.M, K, 0, lane);
    lb.init(B, nullptr, p.bs1, p.bs0, n0, p.N, K, 0, lane);
    // this wave's first output block; its bias and residual are requested with the operands
    const float *bias = p.bias ? p.bias + bz * p.biasbs : nullptr;
    EpiOperands eo;
    if (w < NBLK) eo.load(p, bias, m0 + 16 * (w / NBJ) + 4 * g, n0 + 16 * (w % NBJ) + r16);
    floatx4 acc[NBI][NBJ];
#pragma unroll
    for (int i = 0; i < NBI; ++i)
#pragma unroll
        for (int j = 0; j < NBJ; ++j) acc[i][j] = floatx4{0.f, 0.f, 0.f, 0.f};
    float mx = 0.f;  // largest magnitude this wave has split
    auto compute = [&](const typename LA::regs_t &ra, const typename LB::regs_t &rb) {
        bf16x8 b[NBJ][3];
#pragma unroll
        for (int j = 0; j < NBJ; ++j) LB::planes(rb, j, mx, b[j]);
#pragma unroll
        for (int i = 0; i < NBI; ++i) {
            bf16x8 a[PA];
            LA::planes(ra, i, mx, a);
            floatx4 slab[NBJ];  // TWO
#pragma unroll
            for (int j = 0; j < NBJ; ++j) slab[j] = floatx4{0.f, 0.f, 0.f, 0.f};
            auto mul = [&](int ia, int ib) {
#pragma unroll
                for (int j = 0; j < NBJ; ++j) {
                    floatx4 &d = TWO ? slab[j] : acc[i][j];
                    d = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[ia], b[j][ib], d, 0, 0, 0);
                }
            };
            if constexpr (PA == 3) {
                mul(2, 0);
                mul(0, 2);
                mul(1, 1);
                mul(1, 0);
                mul(0, 1);
                mul(0, 0);
            } else {
                mul(0, 2);
                mul(0, 1);
                mul(0, 0);
            }
            if constexpr (TWO) {
#pragma unroll
                for (int j = 0; j < NBJ; ++j) acc[i][j] += slab[j];
            }
        }
    };
    const int nk = (K + 31) / 32;  // slabs; the last one may be partial
    auto fetch = [&](int s, typename LA::regs_t &xa, typename LB::regs_t &xb) {
        if (s * 32 + 32 <= K) {
            la.load(xa, s * 32, 0, lane);
            lb.load(xb, s * 32, 0, lane);
        } else {
            la.load_tail(xa, s * 32, 0, lane);
            lb.load_tail(xb, s * 32, 0, lane);
        }
    };
    if constexpr (PD == 0) {
        // The next slab's operands are in flight while one is multiplied, then move over: one
        // copy of the arithmetic in the code.  A short product executes it once or twice per
        // wave, and fetching unrolled copies costs more than the moves (512 x 512 x 512: 8.0 us
        // unrolled, 7.0 us so).
        typename LA::regs_t ra, na;
        typename LB::regs_t rb, nb;
        if (w < nk) fetch(w, ra, rb);
#pragma unroll 1
        for (int s = w; s < nk; s += NW) {
            if (s + NW < nk) fetch(s + NW, na, nb);
            compute(ra, rb);
#pragma unroll
            for (int q = 0; q < LA::UPW; ++q)
#pragma unroll
                for (int e = 0; e < LA::NR; ++e) ra[q][e] = na[q][e];
#pragma unroll
            for (int q = 0; q < LB::UPW; ++q)
#pragma unroll
                for (int e = 0; e < LB::NR; ++e) rb[q][e] = nb[q][e];
        }
    } else {
        // PD slabs of registers in flight, the loop unrolled over them; past the wave's last
        // whole slab the last one is loaded again (path-independent wait counts)
        constexpr int R = PD > 0 ? PD : 1;
        typename LA::regs_t ra[R];
        typename LB::regs_t rb[R];
        const int nf = K / 32, ns = w < nf ? (nf - w + NW - 1) / NW : 0, kl = (w + (ns - 1) * NW) * 32;
        auto refill = [&](int u, int t) {
            const int k0 = min((w + t * NW) * 32, kl);
            la.load(ra[u], k0, 0, lane);
            lb.load(rb[u], k0, 0, lane);
        };
        if (ns > 0) {
#pragma unroll
            for (int u = 0; u < R; ++u) refill(u, u);
        }
        int t = 0;
        for (; t + R <= ns; t += R) {
#pragma unroll
            for (int u = 0; u < R; ++u) {
                compute(ra[u], rb[u]);
                refill(u, t + u + R);
            }
        }
#pragma unroll
        for (int u = 0; u < R - 1; ++u)
            if (t + u < ns) compute(ra[u], rb[u]);
        if (nf < nk && w == nf % NW) {
            fetch(nf, ra[0], rb[0]);
            compute(ra[0], rb[0]);
        }
    }
    // the bound on a sum holds for each wave's part of K, and eight sums of up to 2^124 add up in range
    SplitRange range;
#pragma unroll
    for (int i = 0; i < NBI; ++i)
#pragma unroll
        for (int j = 0; j < NBJ; ++j) {
            red[w][i * NBJ + j][lane] = acc[i][j];
            range.add(acc[i][j]);
        }
    mx = wave_max(mx);
    const int mine = range.check(0x1p124f, mx, K);
    const bool redo_w = __builtin_amdgcn_ballot_w64(mine == SplitRange::REDO), look_w = __builtin_amdgcn_ballot_w64(mine);
    if (lane == 0) need[w] = redo_w ? SplitRange::REDO : look_w ? SplitRange::LOOK : SplitRange::OK;
    __syncthreads();
    int any = 0;
#pragma unroll
    for (int k = 0; k < NW; ++k) any |= need[k];
    float unscale = AM == SM_PKB ? SPLIT_UNSCALE : 1.f;
    if (any) {
        bool redo = any & SplitRange::REDO;
        if (!redo && need[w]) {
            bool many;
            // (the magnitude of each row and column would cost the loop registers, and a wave per SIMD)
            auto unknown = [](auto...) { return 1.f; };
            redo = tiny_lines<LA, LB>(p, A, B, m0, n0, w, NW, lane, acc, unknown, unknown, SplitRange::bound(mx, K), many);
            if (many) redo = tiny_operand<LA, LB>(p, A, B, m0, n0, w, NW, 0, 0, lane);
        }
        if (__syncthreads_or(redo)) {  // (red is read after the barrier below)
            unscale = 1.f;
#pragma unroll
            for (int i = 0; i < NBI; ++i)
#pragma unroll
                for (int j = 0; j < NBJ; ++j) acc[i][j] = floatx4{0.f, 0.f, 0.f, 0.f};
            multiply_fp32<LA, LB>(p, A, B, m0, n0, 4 * w, 4 * NW, lane, acc);
#pragma unroll
            for (int i = 0; i < NBI; ++i)
#pragma unroll
                for (int j = 0; j < NBJ; ++j) red[w][i * NBJ + j][lane] = acc[i][j];
            __syncthreads();
        }
    }
    float *C = p.C + bz * p.cbs;
    const bool pairs = p.fz.mode == FZ_SWIGLU;  // gate block i with up block i + 1
    const int n_items = pairs ? NBLK / 2 : NBLK;
    for (int b = w; b < n_items; b += NW) {
        const int i = pairs ? 2 * (b / NBJ) : b / NBJ, j = b % NBJ;
        const int m = m0 + 16 * i + 4 * g, n = n0 + 16 * j + r16;
        auto total = [&](int ii) {
            floatx4 v = red[0][ii * NBJ + j][lane];
#pragma unroll
            for (int k = 1; k < NW; ++k) v += red[k][ii * NBJ + j][lane];
            if constexpr (AM == SM_PKB) v *= unscale;
            return v;
        };
        if (b != w) eo.load(p, bias, m, n);
        const floatx4 v = total(i);
        split_epilogue(p, C, bias, eo, m, n, v, pairs ? total(min(i + 1, NBI - 1)) : v);
    }
}

template <int AM, int BM, int TM, int TN, int NW, int WGM, int FORM = PLAIN>
static void launch_tile(const SplitArgs &p, int batch, hipStream_t s)
{
    hipLaunchKernelGGL((gemm_split_kernel<AM, BM, TM, TN, NW, WGM, FORM>), dim3(ceil_div(p.N, TN), ceil_div(p.M, TM), batch),
                       dim3(NW * 64), 0, s, p);
}
template <int AM, int BM, int NBI, int NBJ, int NW, int PD>
static void launch_wave_split(const SplitArgs &p, int batch, hipStream_t s)
{
    // outer-contiguous operands load element by element here (16 rows of a slab per lane group)
    constexpr int AD = AM == SM_OC ? (int)SM_GEN : AM, BD = BM == SM_OC ? (int)SM_GEN : BM;
    hipLaunchKernelGGL((gemm_split_k_kernel<AD, BD, NBI, NBJ, NW, PD>),
                       dim3(ceil_div(p.N, 16 * NBJ), ceil_div(p.M, 16 * NBI), batch), dim3(NW * 64), 0, s, p);
}

// Unpacked operands, each K-contiguous (KC below), outer-contiguous (OC) or of general strides:
// the products that launch_split's geometries, chosen for weights and a long K, serve badly; false:
// none of them.  Waves that split K read KC rows 16 apart in memory and OC rows element by element,
// and four of them have little to do for a K of a few slabs: tiles in LDS are ahead from the size at
// which they fill the chip.  t64, t32: tiles of 64 x 64 (three workgroups per CU: 768 at a time) and
// 32 x 32.  MI355X, us per product (M x N x K, operands A x B; launch_split's form -> here; the
// former fp32-MFMA kernels):
//   128 x 64, eight waves, past one round of 64 x 64: 2048^2 x 64 OC x KC 18.8 -> 11.7 (14.7),
//     2048^2 x 128 KC x KC 26.1 -> 15.2 (19.4).  Four waves where both are OC (pieces of 32 rows: half
//     of eight waves would stage nothing): 2048^2 x 64 19.3 -> 14.9 (13.9; eight waves 17.6); from
//     K = 96 on four waves that split K are ahead.  Four waves too from K = 256 on for KC x KC:
//     2048^2 x 512 47.2 -> 36.4 (46.1)
//   64 x 64, four waves, from 448 of them on: 1500^2 x 128 OC x OC 18.5 -> 13.7 (15.7), 1500^2 x 200
//     OC x KC 23.3 -> 19.9 (22.6); past K = 320 with OC in A, splitting K is ahead again.  KC x KC at
//     every K and from 224 of them on: 1500^2 x 1024 71.7 -> 50.4 (63.8), 1024^2 x 768 26.5 -> 20.8
//     (20.3).  Eight waves hide more where there is little K: KC x KC 768 x 4096 x 64 17.8 -> 11.8
//     (12.9; in plain sums 10.2, by four waves 10.6), OC x KC 753 x 2592 x 110 13.5 -> 11.8 (11.9;
//     by four 12.2)
//   64 x 32, four waves, OC x OC under 448: 3072 x 509 x 64 12.8 -> 7.7 (9.6)
//   32 x 32 by two waves, a few slabs: 1024^2 x 64 OC x KC 7.5 -> 6.2 (6.6), OC x OC 9.1 -> 6.5 (6.3);
//     four waves: 1024 x 512 x 192 KC x OC 8.4 -> 6.8 (6.2), 1024^2 x 256 KC x OC 13.4 -> 10.9 (10.2)
//   64 x 32, four waves, one slab ahead: 1024 x 512 x 384 KC x KC 11.3 -> 10.1 (8.5)
//   general strides, each operand in its own mode: 1000^3 with every second element of B's K
//     105.7 -> 41.1 (33.8), 2048^2 x 512 with both such 80.1 -> 60.0 (81.0); still behind by up to a
//     third: 1000^2 x 64 one such 13.1 -> 9.0 (6.4), 2000 x 1500 x 100 28.3 -> 23.2 (14.6)
// Errors against 64 bits over 11 sizes, 10 K from 32 to 2048 and four layouts: nowhere above those
// of launch_split's forms, and below the fp32 kernels'.
template <int AM, int BM>
static bool launch_unpacked(const SplitArgs &p, long t64, long t32, int batch, hipStream_t s)
{
    const int K = p.K;
    constexpr bool kk = AM == SM_KC && BM == SM_KC, oo = AM == SM_OC && BM == SM_OC, ko = AM == SM_KC && BM == SM_OC;
    constexpr bool ok = AM == SM_OC && BM == SM_KC;
    if constexpr (AM > SM_GEN || BM > SM_GEN) {
        return false;
    } else if constexpr (AM == SM_GEN || BM == SM_GEN) {
        if constexpr (AM == SM_OC || BM == SM_OC)
            if (t64 > 192 && t64 <= 512 && K >= 512) {
                launch_wave_split<AM, BM, 4, 2, 4, 2>(p, batch, s);
                return true;
            }
        if (t64 > 512) launch_tile<AM, BM, 128, 64, 4, 2, SUMS>(p, batch, s);
        else if (t64 > 192) launch_tile<AM, BM, 64, 64, 4, 2, SUMS>(p, batch, s);
        else if (K <= 128 || t32 > 256) launch_wave_split<AM, BM, 2, 2, 4, 0>(p, batch, s);
        else if (t32 > 128) launch_wave_split<AM, BM, 2, 2, 8, 0>(p, batch, s);
        else launch_wave_split<AM, BM, 2, 1, 8, 0>(p, batch, s);
        return true;
    } else if (t64 > 768) {
        if constexpr (oo) {
            if (K >= 96) return false;
            launch_tile<AM, BM, 128, 64, 4, 2, SUMS_FEW>(p, batch, s);
            return true;
        }
        if (K >= (kk ? 1024 : 256)) return false;
        if constexpr (!oo)
            if (K < 256) launch_tile<AM, BM, 128, 64, 8, 4, SUMS_FEW>(p, batch, s);
        if constexpr (kk)
            if (K >= 256) launch_tile<AM, BM, 128, 64, 4, 2, SUMS>(p, batch, s);
        return true;
    } else if (t64 >= 448 || (kk && t64 >= 224)) {
        if (!kk && K > (ko ? 1000 : 320)) return false;
        if constexpr (kk || ok)
            if (kk ? K < (t64 >= 448 ? 96 : 129) : t64 <= 512 && K <= 128) {
                launch_tile<AM, BM, 64, 64, 8, 4, SUMS_FEW>(p, batch, s);
                return true;
            }
        launch_tile<AM, BM, 64, 64, 4, 2, kk || ko ? SUMS : SUMS_FEW>(p, batch, s);
        return true;
    } else {
        if constexpr (oo)
            if (t64 > 300) {
                if (K > 160) return false;
                launch_tile<AM, BM, 64, 32, 4, 2, SUMS_FEW>(p, batch, s);
                return true;
            }
        if constexpr (!kk)
            if (K <= (oo ? 256 : 160) && (t64 >= 224 || (oo && t32 > 512))) {
                launch_wave_split<AM, BM, 2, 2, 2, 0>(p, batch, s);
                return true;
            }
        if (K <= 128 || t32 < 400 || (ko ? K >= 1024 : t64 >= 224 || (K > 256 && !kk))) return false;
        if constexpr (kk)
            if (K > 256) {
                launch_wave_split<AM, BM, 4, 2, 4, 0>(p, batch, s);
                return true;
            }
        launch_wave_split<AM, BM, 2, 2, 4, 0>(p, batch, s);
        return true;
    }
}

// Geometry by the number of tiles (256 CUs) and K, for packed weights and what launch_unpacked leaves;
// MI355X, us per product (M x N x K):
//   256 x 128 tiles when their rounds over the CUs are at least four fifths full: 12288 x 2048
//     x 4096 1075 (128 x 64: 1320, 64 x 64: 1250); but 2304 x 4096 x 768, 288 tiles, 166 (123)
//   128 x 64 for a long K with two tiles per CU: 2048^3 109 (64 x 64: 153, 256 x 128: 175)
//   64 x 64, four waves on K: 768 x 4096 x 768 and x 3072 138 (128 x 64: 171, 64 x 32: 146)
//     (128 x 64 in one LDS stage is 7-13 % faster for a short K with many tiles, but the error
//     of its one long chain does not average out over the keys that attention sums:
//     GPT-2-small decode logits 6.0e-7 from 64 bits, against 5.1e-7 here and on fp32 MFMA)
//   64 x 32, four waves: 3072 x 509 x 768 28 (64 x 64: 37, 32 x 32: 38); 1024^3 22 (35, 32)
//   64 x 32, eight waves, when that leaves CUs idle but 32 x 32 would need a second round:
//     2304 x 100 x 768 12.4 (four waves 13.8, 32 x 32 16.2)
//   32 x 32, eight waves: 512^3 7.0 (64 x 32: 8.4); four waves for K <= 128 (two slabs or less
//     per wave: 8 x 192 x 512 x 64 7.0, eight waves 10.6)
//   32 x 16, eight waves, when 32 x 32 would leave half the CUs idle: 12 GPT-2-small layers of
//     100 tokens, all products, 880 (32 x 32: 960)
template <int AM, int BM>
static void launch_split(const SplitArgs &p, int batch, hipStream_t s)
{
    auto tiles = [&](int a, int b) { return (long)ceil_div(p.M, a) * ceil_div(p.N, b) * batch; };
    if (launch_unpacked<AM, BM>(p, tiles(64, 64), tiles(32, 32), batch, s)) return;
    if constexpr (AM != SM_GEN && BM != SM_GEN) {
        const long big = tiles(256, 128);
        if (big >= 256 && big * 5 >= (big + 255) / 256 * 256 * 4) launch_tile<AM, BM, 256, 128, 8, 4>(p, batch, s);
        else if (tiles(128, 64) >= 512 && p.K >= 1024) launch_tile<AM, BM, 128, 64, 4, 2>(p, batch, s);
        else if (tiles(64, 64) >= 768) launch_wave_split<AM, BM, 4, 4, 4, 1>(p, batch, s);
        else if (p.K <= 128) launch_wave_split<AM, BM, 2, 2, 4, 0>(p, batch, s);
        else if (tiles(64, 32) >= 256) launch_wave_split<AM, BM, 4, 2, 4, 2>(p, batch, s);
        else if (tiles(32, 32) > 256) launch_wave_split<AM, BM, 4, 2, 8, 0>(p, batch, s);
        else if (tiles(32, 32) > 128) launch_wave_split<AM, BM, 2, 2, 8, 0>(p, batch, s);
        else launch_wave_split<AM, BM, 2, 1, 8, 0>(p, batch, s);
    }
}

template <int MODE>
using mode_c = std::integral_constant<int, MODE>;

// staging mode of operand X(o, k) = X[o * so + k * sk]
static int split_mode(long so, long sk) { return sk == 1 ? SM_KC : so == 1 ? SM_OC : SM_GEN; }

jas_status gemm_split(SplitArgs p, bool a_packed, bool a_bf16, int batch, hipStream_t s)
{
    int am = a_packed ? (a_bf16 ? SM_PKB : SM_PK) : split_mode(p.as0, p.as1);
    if (!a_packed && p.cs0 != 1 && p.cs1 == 1) {
        // row-major C: the transposed product, whose lanes hold four consecutive elements
        std::swap(p.M, p.N);
        const float *A = p.A;
        p.A = p.B, p.B = A;
        const long a0 = p.as0, a1 = p.as1;
        p.as0 = p.bs1, p.as1 = p.bs0, p.bs0 = a1, p.bs1 = a0;
        std::swap(p.abs_, p.bbs);
        std::swap(p.cs0, p.cs1);
        std::swap(p.rs0, p.rs1);
        if (p.bias_mode) p.bias_mode = 3 - p.bias_mode;
        am = split_mode(p.as0, p.as1);
    }
    int bm = split_mode(p.bs1, p.bs0);
    if (a_packed) {
        JAS_CHECK(bm == SM_KC, JAS_ERR_INVALID, "gemm: packed weights take K-contiguous activations");
        if (a_bf16) launch_split<SM_PKB, SM_KC>(p, batch, s);
        else launch_split<SM_PK, SM_KC>(p, batch, s);
    } else {
        auto go = [&](auto a, auto b) { launch_split<decltype(a)::value, decltype(b)::value>(p, batch, s); };
        auto with_b = [&](auto a) {
            if (bm == SM_KC) go(a, mode_c<SM_KC>());
            else if (bm == SM_OC) go(a, mode_c<SM_OC>());
            else go(a, mode_c<SM_GEN>());
        };
        if (am == SM_KC) with_b(mode_c<SM_KC>());
        else if (am == SM_OC) with_b(mode_c<SM_OC>());
        else with_b(mode_c<SM_GEN>());
    }
    JAS_LAUNCH_CHECK();
    return JAS_OK;
}

} // namespace jas
