// fp32 GEMMs on the CDNA4 matrix cores.
//
// Reference: mat_dot_t::operator() (mat_express_t.hpp:730-736) is a scalar triple loop
// with sequential-k accumulation, reached from weight_net_t::forward (mat_net_t.hpp:38-49)
// for every projection and from mat_head_gen_t::forward (mat_mha_t.hpp:53,71).
//
// Here: skinny_kernel for N <= 16 tokens (decode) -- the weight matrix is streamed from HBM
// straight into MFMA A-operand registers (no LDS), one 16-row tile per wave set, the K range
// split across the waves of a workgroup and reduced through LDS, with the layer's elementwise
// tail fused into the epilogue (bias, GELU, residual add, SwiGLU, RoPE + KV-cache append) --
// the packed weight layouts, and the fp64 GEMM.  Larger products are in gemm_split.hip.
//
// MFMA 16x16x4 f32 operand layout (lane l of 64): A[i = l%16][kslot = l/16],
// B[kslot = l/16][j = l%16], D rows 4*(l/16)+r (r = 0..3), column l%16.  Each lane loads
// a float4 along K; sub-step t of 4 feeds element t, so k-slot s of sub-step t is
// k = 4s + t -- a permutation of K applied identically to A and B.
#include "gemm.hpp"

namespace jas {

typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

__device__ __forceinline__ floatx4 mfma4(float a, float b, floatx4 c)
{
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

static bool al16(const void *p) { return ((uintptr_t)p & 15) == 0; }

jas_status gemm_prefill_fused(int M, int N, int K, const void *A, bool a_bf16, const float *X, float *C, long ldc,
                              const float *bias, const PrefillFused &fz, hipStream_t s)
{
    // SwiGLU: M virtual rows = 2 x the output features (gate / up tiles interleaved)
    JAS_CHECK(fz.mode != FZ_SWIGLU || (M % 32 == 0 && fz.A2 && !bias), JAS_ERR_INVALID, "prefill GEMM: bad SwiGLU shape");
    JAS_CHECK(fz.mode != FZ_QKV || (fz.d % 16 == 0 && fz.dh % 16 == 0 && M == 3 * fz.d && fz.pos && (!fz.rope || fz.rope_tab)),
              JAS_ERR_INVALID, "prefill GEMM: bad QKV shape");
    JAS_CHECK(al16(A) && al16(X) && al16(C) && K % 16 == 0 && ldc % 4 == 0, JAS_ERR_INVALID, "prefill GEMM: bad operands");
    SplitArgs p{(const float *)A, X, C, bias, K, 1, 1, K, 1, ldc, 0, 0, 0, 0, M, N, K, bias ? 1 : 0, JAS_ACT_NONE, 0};
    p.fz = fz;
    return gemm_split(p, true, a_bf16, 1, s);
}

// ---------------------------------------------------------------- prefill GEMM into a bf16 KV cache
// C[n][m] of packed weights A [M][K] and token-major X [N][K] on the fp32 matrix cores: the
// QKV product of a model whose KV cache holds bf16.  A cached key or value is its fp32 sum
// rounded to 8 bits, so a sum that differs in its last bits now and then rounds to the other
// neighbour, 2^-8 away, and the logits move by about 1e-4 to 2e-3.  Sums by fp32 products (k
// ascending by 16, within that k = 4 g + t for t = 0..3) fall to the same side as the fp32
// oracle's often enough for its comparison (1e-3) to hold at d 2048, 16 sequences; by the split
// they reach 1.15e-3 there.  That is this kernel's only ground.  It keeps the cache entries that
// products of this order always gave in layer 0 alone, since the inputs of the layers above come
// out of split products, and it is not the more exact form: decode logits' relative distance from
// 64 bits, mean of 8 seeds, bf16 weights and cache, 1 / 2 / 4 layers: d 1024 LLaMA form 5.9 / 5.3 /
// 5.1e-5 (split: 3.1 / 3.0 / 2.7e-5), d 768 GPT-2 form 2.0 / 1.8 / 1.7e-5 (1.1 / 1.0 / 0.9e-5).
// In time the split with the cache write in its epilogue is ahead too: a prefill of one layer at
// 7B width, 4 x 512 tokens, 3.37 ms here and 2.35 with it.
//
// 32-wide K slabs, a slab ahead in registers, two in LDS in MFMA operand order (lane (r, g) of
// a 16-row block holds k = 4 g .. 4 g + 3 of each 16), so every fragment read is one 16-byte
// read; bf16 weights stay bf16 until then (half the LDS bytes) and widen by a shift or a mask.
// Eight waves of 64 x 64 per workgroup: MFMA-bound.  12288 x 2048 x 4096, bf16 weights, MI355X:
// 1.64 ms, 126 TFLOP/s (1.90 with 128 x 128 tiles of four waves and 16-wide slabs).
template <int AM, int TM, int TN, int NW, int WGM>
__global__ void __launch_bounds__(NW * 64, 2)
gemm_fp32_kernel(int M, int N, int K, const float *__restrict__ A, const float *__restrict__ X, float *__restrict__ C,
                 long ldc, const float *__restrict__ bias)
{
    constexpr int WGN = NW / WGM, NBI = TM / WGM / 16, NBJ = TN / WGN / 16;
    constexpr int PA = AM == SM_PKB ? 1 : 2;                     // 16-byte pieces of a lane's A row and slab
    constexpr int SA = PA * TM * 4, SB = 2 * TN * 4;             // 16-byte units per stage
    constexpr int UA = TM / 16 / NW, UB = TN / 16 / NW;          // 16-row blocks staged per wave
    static_assert(TM % (16 * NW) == 0 && TN % (16 * NW) == 0, "blocks spread evenly over the waves");
    __shared__ floatx4 lds[2][SA + SB];
    const int tid = threadIdx.x, lane = tid & 63, r16 = lane & 15, g = lane >> 4;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6), wm = w / WGN, wn = w % WGN;
    const int m0 = blockIdx.y * TM, n0 = blockIdx.x * TN;
    const long RG = (M + 15) >> 4;

    long rt[UA];
    const float *xr[UB];
#pragma unroll
    for (int q = 0; q < UA; ++q) rt[q] = min((long)(m0 >> 4) + w + q * NW, RG - 1);
#pragma unroll
    for (int q = 0; q < UB; ++q) xr[q] = X + (long)min(n0 + 16 * (w + q * NW) + r16, N - 1) * K + 4 * g;
    floatx4 ra[UA][PA], rb[UB][2];
    // the slab at k0; `whole`: both of its 16-wide halves lie inside K (K % 16 == 0)
    auto fetch = [&](int k0, bool whole) {
#pragma unroll
        for (int q = 0; q < UA; ++q) {
            if constexpr (AM == SM_PKB) {
                ra[q][0] = *(const floatx4 *)((const uint16_t *)(const void *)A +
                                              weight_tile_offset_b(rt[q], k0 >> 5, k32_of(K), RG) + lane * 8);
            } else {
                ra[q][0] = *(const floatx4 *)(A + weight_tile_offset(rt[q], k0 >> 4, K >> 4, RG) + lane * 4);
                if (whole) ra[q][1] = *(const floatx4 *)(A + weight_tile_offset(rt[q], (k0 >> 4) + 1, K >> 4, RG) + lane * 4);
            }
        }
#pragma unroll
        for (int q = 0; q < UB; ++q) {
            rb[q][0] = *(const floatx4 *)(xr[q] + k0);
            if (whole) rb[q][1] = *(const floatx4 *)(xr[q] + k0 + 16);
        }
    };
    floatx4 acc[NBI][NBJ];
#pragma unroll
    for (int i = 0; i < NBI; ++i)
#pragma unroll
        for (int j = 0; j < NBJ; ++j) acc[i][j] = floatx4{0.f, 0.f, 0.f, 0.f};
    const int nk = K / 32;
    // slab s: into stage s % 2, which was last read two slabs ago, before the barrier in between
    auto step = [&](int s, bool whole) {
        floatx4 *sa = lds[s & 1], *sb = sa + SA;
#pragma unroll
        for (int q = 0; q < UA; ++q)
#pragma unroll
            for (int h = 0; h < PA; ++h) sa[(h * (TM / 16) + w + q * NW) * 64 + lane] = ra[q][h];
#pragma unroll
        for (int q = 0; q < UB; ++q)
#pragma unroll
            for (int h = 0; h < 2; ++h) sb[(h * (TN / 16) + w + q * NW) * 64 + lane] = rb[q][h];
        if (whole) fetch(min(s + 1, nk - 1) * 32, true);  // (past the last whole slab: it again)
        __syncthreads();
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            if (h == 1 && !whole) break;
            floatx4 a[NBI], b[NBJ];
#pragma unroll
            for (int i = 0; i < NBI; ++i) {
                a[i] = sa[((AM == SM_PKB ? 0 : h) * (TM / 16) + wm * NBI + i) * 64 + lane];
                if constexpr (AM == SM_PKB) {
                    const u32x4 u = __builtin_bit_cast(u32x4, a[i]);
                    a[i] = widen_bf16x4(u32x2{u[2 * h], u[2 * h + 1]});
                }
            }
#pragma unroll
            for (int j = 0; j < NBJ; ++j) b[j] = sb[(h * (TN / 16) + wn * NBJ + j) * 64 + lane];
#pragma unroll
            for (int t = 0; t < 4; ++t)
#pragma unroll
                for (int i = 0; i < NBI; ++i)
#pragma unroll
                    for (int j = 0; j < NBJ; ++j) acc[i][j] = mfma4(a[i][t], b[j][t], acc[i][j]);
        }
    };
    if (nk > 0) fetch(0, true);
    for (int s = 0; s < nk; ++s) step(s, true);
    if (nk * 32 < K) {
        fetch(nk * 32, false);
        step(nk, false);
    }

    // lane holds rows m = 4g + r of each 16 x 16 block, column n = r16 (M % 16 == 0)
#pragma unroll
    for (int i = 0; i < NBI; ++i)
#pragma unroll
        for (int j = 0; j < NBJ; ++j) {
            const int m = m0 + (wm * NBI + i) * 16 + 4 * g, n = n0 + (wn * NBJ + j) * 16 + r16;
            if (n >= N || m >= M) continue;
            floatx4 v = acc[i][j];
            if (bias) v += *(const floatx4 *)(bias + m);
            *(floatx4 *)(C + m + (long)n * ldc) = v;
        }
}

jas_status gemm_prefill_fp32(int M, int N, int K, const void *A, bool a_bf16, const float *X, float *C, long ldc,
                             const float *bias, hipStream_t s)
{
    JAS_CHECK(M % 16 == 0 && K % 16 == 0 && ldc % 4 == 0 && al16(A) && al16(X) && al16(C) && (!bias || al16(bias)),
              JAS_ERR_INVALID, "prefill GEMM: bad operands");
    // 256 x 128 tiles when they give every CU one, else 64 x 64
    const bool big = (long)ceil_div(N, 128) * ceil_div(M, 256) >= 256;
#define JAS_PF(AM, TM, TN, NW, WGM)                                                                                 \
    hipLaunchKernelGGL((gemm_fp32_kernel<AM, TM, TN, NW, WGM>), dim3(ceil_div(N, TN), ceil_div(M, TM)), dim3(64 * NW), 0, s, \
                       M, N, K, (const float *)A, X, C, ldc, bias)
    if (a_bf16 && big) JAS_PF(SM_PKB, 256, 128, 8, 4);
    else if (a_bf16) JAS_PF(SM_PKB, 64, 64, 4, 2);
    else if (big) JAS_PF(SM_PK, 256, 128, 8, 4);
    else JAS_PF(SM_PK, 64, 64, 4, 2);
#undef JAS_PF
    JAS_LAUNCH_CHECK();
    return JAS_OK;
}

jas_status gemm_general(int M, int N, int K, const void *A, long as0, long as1, const float *B, long bs0, long bs1,
                        float *C, long cs0, long cs1, const float *bias, int bias_mode, int act, int accumulate,
                        int batch, long abs_, long bbs, long cbs, long biasbs, hipStream_t s, bool a_packed,
                        bool a_bf16)
{
    JAS_CHECK(!a_bf16 || a_packed, JAS_ERR_INVALID, "gemm: bf16 A only in the packed layout");
    JAS_CHECK(!a_packed || (K % 16 == 0 && batch == 1 && al16(A)), JAS_ERR_INVALID, "gemm: packed A needs K % 16 == 0");
    const SplitArgs p{(const float *)A, B,    C,   bias_mode ? bias : nullptr, as0, as1, bs0, bs1, cs0,       cs1, abs_,
                      bbs,              cbs,  biasbs, M,                       N,   K,   bias_mode, act, accumulate};
    return gemm_split(p, a_packed, a_bf16, batch, s);
}

// first maximum (ties to the lowest index) over the four 16-lane rows of a wave: lanes l,
// l ^ 16, l ^ 32, l ^ 48 end with the same pair (gfx950 permlane swaps, no LDS round trip)
__device__ __forceinline__ void argmax_rows(float &bv, int &bi)
{
    auto step = [&](bool rows32) {
        const unsigned vb = __float_as_uint(bv), ib = (unsigned)bi;
        const auto pv = rows32 ? __builtin_amdgcn_permlane32_swap(vb, vb, false, false)
                               : __builtin_amdgcn_permlane16_swap(vb, vb, false, false);
        const auto pi = rows32 ? __builtin_amdgcn_permlane32_swap(ib, ib, false, false)
                               : __builtin_amdgcn_permlane16_swap(ib, ib, false, false);
        float av = __uint_as_float(pv[0]), ov = __uint_as_float(pv[1]);
        int ai = (int)pi[0], oi = (int)pi[1];
        if (ov > av || (ov == av && oi < ai)) { av = ov; ai = oi; }
        bv = av;
        bi = ai;
    };
    step(true);
    step(false);
}

// ---------------------------------------------------------------- skinny (decode) GEMM
// One workgroup per row group of 16 rows (NT tiles of 16 rows for NT > 1; DUAL: tile 0 from
// W, tile 1 from W2 at the same 16 rows).  Its WPB waves interleave over the K chunks of 64
// and are reduced through LDS, then the fused epilogue runs.  No cross-workgroup reduction:
// on MI355X each XCD has its own L2, so a device-scope release/acquire inside the kernel
// would write back and invalidate L2 -- far costlier than the parallelism it buys.
//
// PACKED weights (weight_pack_offset): each wave-wide load is one contiguous 1 KB block
// holding exactly the A-operand float4s of 64 lanes, so a workgroup streams its rows as
// long contiguous runs instead of 16 rows x 64 B scattered 4*K bytes apart.
//
// WB (packed only): the weights are bf16 -- the same layout at 2 bytes per element, so one
// wave-wide load is a contiguous 512-byte block.  They feed v_mfma_f32_16x16x32_bf16
// directly: the activations are split exactly into three bf16 parts (x = hi + mid + lo,
// 8 significant bits each, so every bf16 x bf16 product is exact in fp32) and each weight
// fragment is multiplied by all three, accumulating in fp32.  The K order within a 32-wide
// step is permuted identically in both operands: slot j of lane group g is k = 16q + 4g + j
// for j < 4 (block q) and 16(q+1) + 4g + j - 4 for j >= 4 (block q+1) -- exactly what the
// packed weight and activation layouts put in that lane.  One such MFMA does the work of
// eight fp32 16x16x4 ones, so halving the weight bytes does not make the kernel
// matrix-core bound.
//
// EPI: the epilogue (SkinnyEpi; SE_HEAD is EPI_STORE plus the workgroup's greedy picks) is a
// template parameter: a GPT-2-size launch runs each instruction once, and what it fetches of
// a 20 KB body with every epilogue in it (tanh, the row maxima) cost more than its arithmetic.
template <int NT, int WPB, int DEPTH, bool DUAL, bool PACKED, bool WB, int EPI>
__global__ void __launch_bounds__(WPB * 64)
skinny_kernel(const void *__restrict__ W, const void *__restrict__ W2, const float *__restrict__ X, long ldx, int M,
              int N, int K, const SkinnyEpiArgs epi)
{
    static_assert(!WB || PACKED, "bf16 weights are packed");
    using WT = typename std::conditional<WB, uint16_t, float>::type;
    // one lane's weights of a 16-wide block (fp32) or of a 32-wide pair tile (bf16, slots 0-1)
    using WR = typename std::conditional<WB, u32x4, floatx4>::type;
    __shared__ floatx4 red[WPB][NT][64];
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    const int r16 = lane & 15, g = lane >> 4;
    // DUAL: tiles 0..NT/2-1 are gate rows, NT/2..NT-1 the up rows of the same 16-row blocks
    constexpr int NH = DUAL ? NT / 2 : NT;
    static_assert(!DUAL || NT % 2 == 0, "dual tiles come in (gate, up) pairs");
    const int m0 = blockIdx.x * NH * 16;
    const int K16 = K >> 4;

    const long RG = (M + 15) >> 4;  // row tiles of the packed layout
    const WT *wp[NT];
    long wrt[NT];  // packed: this tile's row-tile index
#pragma unroll
    for (int t = 0; t < NT; ++t) {
        const WT *base = (const WT *)((DUAL && t >= NH) ? W2 : W);
        const int tt = t % NH;  // 16-row block of this tile within the workgroup's rows
        if (PACKED) {
            // tiles past the last row tile (M not a multiple of NH*16) re-read the last one;
            // their rows are >= M and the epilogue discards them
            wrt[t] = min((long)(m0 / 16 + tt), RG - 1);
            wp[t] = base + lane * (WB ? 8 : 4);
        } else {
            int row = m0 + tt * 16 + r16;
            row = row < M ? row : M - 1;  // clamped rows are computed and discarded
            wp[t] = base + (long)row * K + 4 * g;
        }
    }
    // token rows >= N feed only output columns >= N, which the epilogue discards, so the
    // activation loads need no predicate (row 0 stands in for them)
    const float *xp = PACKED ? X + (long)lane * 4 : X + (long)(r16 < N ? r16 : 0) * ldx + 4 * g;

    floatx4 acc[NT];
#pragma unroll
    for (int t = 0; t < NT; ++t) acc[t] = floatx4{0.f, 0.f, 0.f, 0.f};

    // K split (PARTIAL mode): this workgroup owns chunks [c_begin, c_end).  The streaming
    // loop covers the full 64-wide chunks; a partial last chunk (K % 64 != 0) is done once
    // at the end with predicated loads.
    const int c_begin = blockIdx.y * epi.cpb;
    const int c_end = min((K + 63) >> 6, c_begin + epi.cpb);
    const int c_full = min(K >> 6, c_end);
    // chunk index of this wave's i-th chunk: cs + i * WPB.  w is made wave-uniform so every
    // bound below is a scalar branch and the loads in the steady state carry no predicate
    // (a predicated load puts a branch around it, and the wait before the MFMAs then drains
    // the whole pipeline).
    const int wu = __builtin_amdgcn_readfirstlane(w);
    const int cs = c_begin + wu;
    const int nw = cs < c_full ? (c_full - cs + WPB - 1) / WPB : 0;
    WR wb[DEPTH][NT][4];
    float4 xb[DEPTH][4];
    const int K32 = k32_of(K);
    auto load = [&](int c, WR (&wv)[NT][4], float4 (&xv)[4]) {
        const int k = c * 64;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
#pragma unroll
            for (int t = 0; t < NT; ++t) {
                if constexpr (WB) {
                    if (q < 2)  // pair tiles 2c, 2c+1
                        wv[t][q] = __builtin_nontemporal_load(
                            (const u32x4 *)(wp[t] + weight_tile_offset_b(wrt[t], 2 * c + q, K32, RG)));
                } else if (PACKED)
                    wv[t][q] = __builtin_nontemporal_load(
                        (const floatx4 *)(wp[t] + weight_tile_offset(wrt[t], 4 * c + q, K16, RG)));
                else
                    wv[t][q] = __builtin_nontemporal_load((const floatx4 *)(wp[t] + k + 16 * q));
            }
            if (PACKED)  // contiguous 1 KB per wave
                xv[q] = *(const float4 *)(xp + (long)(4 * c + q) * 256);
            else
                xv[q] = *(const float4 *)(xp + k + 16 * q);
        }
    };
    auto compute = [&](const WR (&wv)[NT][4], const float4 (&xv)[4]) {
        if constexpr (WB) {
#pragma unroll
            for (int pr = 0; pr < 2; ++pr) {  // blocks 2pr, 2pr+1: one 32-wide MFMA step
                const float4 a = xv[2 * pr], b = xv[2 * pr + 1];
                const float x8[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
                bf16x8 xh, xm, xl;
#pragma unroll
                for (int j = 0; j < 8; ++j) {
                    const __bf16 h = (__bf16)x8[j];
                    const float r1 = x8[j] - (float)h;   // exact
                    const __bf16 m = (__bf16)r1;
                    const float r2 = r1 - (float)m;      // exact, at most 8 significant bits
                    xh[j] = h;
                    xm[j] = m;
                    xl[j] = (__bf16)r2;                  // exact
                }
#pragma unroll
                for (int t = 0; t < NT; ++t) {
                    const bf16x8 wf = __builtin_bit_cast(bf16x8, wv[t][pr]);
                    acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf, xl, acc[t], 0, 0, 0);
                    acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf, xm, acc[t], 0, 0, 0);
                    acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf, xh, acc[t], 0, 0, 0);
                }
            }
        } else {
#pragma unroll
            for (int q = 0; q < 4; ++q)
#pragma unroll
                for (int t = 0; t < NT; ++t) {
                    acc[t] = mfma4(wv[t][q][0], xv[q].x, acc[t]);
                    acc[t] = mfma4(wv[t][q][1], xv[q].y, acc[t]);
                    acc[t] = mfma4(wv[t][q][2], xv[q].z, acc[t]);
                    acc[t] = mfma4(wv[t][q][3], xv[q].w, acc[t]);
                }
        }
    };
#pragma unroll
    for (int j = 0; j < DEPTH - 1; ++j)
        if (j < nw) load(cs + j * WPB, wb[j], xb[j]);
    int i = 0;
    // steady state: DEPTH chunks per trip, every load in range
    for (; i + 2 * DEPTH - 2 < nw; i += DEPTH) {
#pragma unroll
        for (int j = 0; j < DEPTH; ++j) {
            load(cs + (i + j + DEPTH - 1) * WPB, wb[(j + DEPTH - 1) % DEPTH], xb[(j + DEPTH - 1) % DEPTH]);
            compute(wb[j], xb[j]);
        }
    }
    // drain (i % DEPTH == 0 here, so the ring slots are compile-time indices)
#pragma unroll
    for (int j = 0; j < 2 * DEPTH - 1; ++j) {
        if (i + j < nw) {
            if (i + j + DEPTH - 1 < nw)
                load(cs + (i + j + DEPTH - 1) * WPB, wb[(j + DEPTH - 1) % DEPTH], xb[(j + DEPTH - 1) % DEPTH]);
            compute(wb[j % DEPTH], xb[j % DEPTH]);
        }
    }
    // partial last chunk: the wave whose stride reaches it; blocks (packed) or lanes
    // (row-major) past K read as zero
    if (c_full < c_end && (c_full - c_begin) % WPB == wu) {
        const int c = c_full, k = c * 64;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const bool in = PACKED ? (4 * c + q) < K16 : (k + 16 * q + 4 * g) < K;
#pragma unroll
            for (int t = 0; t < NT; ++t) {
                if constexpr (WB) {
                    if (q % 2 == 0)  // a pair tile whose first block is in range (its padding is zero)
                        wb[0][t][q / 2] = in ? *(const u32x4 *)(wp[t] + weight_tile_offset_b(wrt[t], 2 * c + q / 2, K32, RG))
                                             : u32x4{0u, 0u, 0u, 0u};
                } else if (PACKED)
                    wb[0][t][q] = in ? *(const floatx4 *)(wp[t] + weight_tile_offset(wrt[t], 4 * c + q, K16, RG))
                                     : floatx4{0.f, 0.f, 0.f, 0.f};
                else
                    wb[0][t][q] = in ? *(const floatx4 *)(wp[t] + k + 16 * q) : floatx4{0.f, 0.f, 0.f, 0.f};
            }
            if (PACKED)
                xb[0][q] = in ? *(const float4 *)(xp + (long)(4 * c + q) * 256) : make_float4(0.f, 0.f, 0.f, 0.f);
            else
                xb[0][q] = in ? *(const float4 *)(xp + k + 16 * q) : make_float4(0.f, 0.f, 0.f, 0.f);
        }
        compute(wb[0], xb[0]);
    }
#pragma unroll
    for (int t = 0; t < NT; ++t) red[w][t][lane] = acc[t];
    __syncthreads();

    // epilogue: thread (t, ln) owns rows m..m+3 of tile t for token n = ln % 16
    const int n_items = NH * 64;
    const int t = tid / 64, ln = tid % 64;
    const int n = ln & 15;
    const int m = m0 + t * 16 + 4 * (ln >> 4);
    const bool live = tid < n_items && n < N && m < M;
    float v[4] = {0.f, 0.f, 0.f, 0.f};
    const int nv = live ? min(4, M - m) : 0;
    if (live) {
        floatx4 s0 = red[0][t][ln];
#pragma unroll
        for (int ww = 1; ww < WPB; ++ww) s0 += red[ww][t][ln];
        v[0] = s0[0], v[1] = s0[1], v[2] = s0[2], v[3] = s0[3];
    }
    if constexpr (EPI == SE_HEAD) {
        {  // first maximum of the stored values over this workgroup's rows
            __shared__ float sbv[NH * 16];
            __shared__ int sbi[NH * 16];
            float bv = -INFINITY;
            int bi = 0x7fffffff;
            for (int r = 0; r < nv; ++r) {
                const float x = epi.bias ? v[r] + epi.bias[m + r] : v[r];
                if (x > bv) { bv = x; bi = m + r; }
            }
            // the four lanes of a token in each wave (ln, ln ^ 16, ln ^ 32, ln ^ 48) combine in
            // registers, then the tile waves' winners through LDS (ties to the lowest index)
            argmax_rows(bv, bi);
            if (tid < n_items && ln < 16) { sbv[t * 16 + ln] = bv; sbi[t * 16 + ln] = bi; }
            __syncthreads();
            if (tid < 16) {
                for (int k = 1; k < NH; ++k) {
                    const float ov = sbv[k * 16 + tid];
                    const int oi = sbi[k * 16 + tid];
                    if (ov > bv || (ov == bv && oi < bi)) { bv = ov; bi = oi; }
                }
                epi.amax_v[(long)tid * gridDim.x + blockIdx.x] = bv;
                epi.amax_i[(long)tid * gridDim.x + blockIdx.x] = bi;
            }
        }
    }
    if (!live) return;

    if constexpr (EPI == EPI_PARTIAL) {  // raw split-K partial, [split][16][M]; the consumer reduces
        float *o = epi.out + ((long)blockIdx.y * 16 + n) * M + m;
        if (nv == 4 && (M & 3) == 0) *(float4 *)o = make_float4(v[0], v[1], v[2], v[3]);
        else
            for (int r = 0; r < nv; ++r) o[r] = v[r];
        return;
    }
    if constexpr (EPI == EPI_SWIGLU) {  // silu(gate) * up
        floatx4 s1 = red[0][t + NH][ln];
#pragma unroll
        for (int ww = 1; ww < WPB; ++ww) s1 += red[ww][t + NH][ln];
        if (epi.out_packed && nv == 4) {
            *(float4 *)(epi.out + packed_b_offset(n, m)) =
                make_float4(silu_f(v[0]) * s1[0], silu_f(v[1]) * s1[1], silu_f(v[2]) * s1[2], silu_f(v[3]) * s1[3]);
            return;
        }
        float *o = epi.out + (long)n * epi.ldo + m;
        for (int r = 0; r < nv; ++r) o[r] = silu_f(v[r]) * s1[r];
    }
    if constexpr (EPI != EPI_PARTIAL && EPI != EPI_SWIGLU) {
        if (epi.bias)
            for (int r = 0; r < nv; ++r) v[r] = v[r] + epi.bias[m + r];
    }
    if constexpr (EPI == EPI_STORE || EPI == SE_GELU || EPI == SE_HEAD) {
        auto act = [&](float x) { return EPI == EPI_STORE ? apply_act(x, epi.act) : EPI == SE_GELU ? gelu_f(x) : x; };
        if (epi.out_packed && nv == 4) {
            *(float4 *)(epi.out + packed_b_offset(n, m)) = make_float4(act(v[0]), act(v[1]), act(v[2]), act(v[3]));
            return;
        }
        float *o = epi.out + (long)n * epi.ldo + m;
        for (int r = 0; r < nv; ++r) o[r] = act(v[r]);
    }
    if constexpr (EPI == EPI_QKV) {  // (m % 4 == 0, d % 16 == 0, dh even: the 4 rows share a section and head)
        const int sec = m / epi.d, e = m - sec * epi.d, h = e / epi.dh, ee = e - h * epi.dh;
        const int pos = epi.pos[n];
        if (epi.rope_tab && sec < 2) {
#pragma unroll
            for (int pr = 0; pr < 2; ++pr) {
                const double2 cst = epi.rope_tab[(long)pos * (epi.dh / 2) + (ee + 2 * pr) / 2];
                const double cs = cst.x, sn = cst.y, x0 = v[2 * pr], x1 = v[2 * pr + 1];
                v[2 * pr] = (float)(x0 * cs - x1 * sn);
                v[2 * pr + 1] = (float)(x0 * sn + x1 * cs);
            }
        }
        if (sec == 0) {
            *(float4 *)(epi.q_out + (long)n * epi.d + e) = make_float4(v[0], v[1], v[2], v[3]);
        } else {
            const long ce = (long)n * epi.kv_sb + (long)h * epi.kv_sh + (long)pos * epi.dh + ee;
            float *cache = sec == 1 ? epi.k_cache : epi.v_cache;
            if (epi.kv_bf16)
                *(u32x2 *)((uint16_t *)cache + ce) =
                    u32x2{(uint32_t)f32_to_bf16(v[0]) | ((uint32_t)f32_to_bf16(v[1]) << 16),
                          (uint32_t)f32_to_bf16(v[2]) | ((uint32_t)f32_to_bf16(v[3]) << 16)};
            else
                *(float4 *)(cache + ce) = make_float4(v[0], v[1], v[2], v[3]);
        }
    }
}

template <int NT, int WPB, int DEPTH, bool DUAL, bool PACKED, bool WB, int EPI>
static void launch_skinny(const void *W, const void *W2, const float *X, long ldx, int M, int N, int K,
                          const SkinnyEpiArgs &epi, hipStream_t s)
{
    const int rows = DUAL ? 16 * (NT / 2) : NT * 16;
    const int ks = EPI == EPI_PARTIAL ? std::max(1, epi.ksplit) : 1;
    hipLaunchKernelGGL((skinny_kernel<NT, WPB, DEPTH, DUAL, PACKED, WB, EPI>), dim3((M + rows - 1) / rows, ks),
                       dim3(WPB * 64), 0, s, W, W2, X, ldx, M, N, K, epi);
}

// Geometry per decode shape, from a cold-weight sweep on MI355X (16 tokens, packed weights).
// More row tiles per workgroup amortise each activation chunk (read from L2) over more
// weight bytes, best when the workgroup count lands on the 256 CUs (the QKV projection:
// three tiles); small matrices (GPT-2 widths) are latency-bound and keep one tile and
// 8 waves so that more workgroups are in flight.
SkinnyTuning skinny_default_tuning(int M, int K, bool dual, bool split, bool wbf16)
{
    SkinnyTuning t;
    const int rt = (M + 15) / 16;
    if (wbf16) {  // bf16 weights (cold-weight sweep): half the bytes per tile, deeper rings
        if (dual && rt >= 512) { t.nt = 6; t.wpb = 4; t.depth = 2; }  // one round (fp32 note below)
        else if (dual) { t.nt = 2; t.wpb = 4; t.depth = 3; }
        else if (split && rt >= 256) {
            if (K >= 8192) { t.nt = 4; t.wpb = 4; t.depth = 4; }
            else { t.nt = 2; t.wpb = 8; t.depth = 2; }
        } else if (split) { t.nt = 2; t.wpb = 8; t.depth = 2; }
        else if (rt >= 1536 && K >= 2048) { t.nt = 4; t.wpb = 4; t.depth = 2; }
        else if (rt >= 1536) { t.nt = 4; t.wpb = 4; t.depth = 3; }
        else if (rt >= 512) { t.nt = 3; t.wpb = 4; t.depth = 4; }
        else { t.nt = 1; t.wpb = 8; t.depth = 3; }
        return t;
    }
    if (dual) {                      // SwiGLU gate/up pairs
        // three pairs per workgroup at LLaMA-7B width: 688 row tiles in 230 workgroups, one
        // round on 256 CUs instead of 2.7 (236 VGPRs; one 4-wave workgroup per CU keeps
        // ~100 KB in flight): GEMM time per step -4 %.  One pair otherwise.
        if (rt >= 512) { t.nt = 6; t.wpb = 4; t.depth = 2; }
        else { t.nt = 2; t.wpb = 4; t.depth = 3; }
    } else if (split) {              // split-K residual projections
        // (two tiles: four would need twice the K splits, and the norm kernel that sums
        // the split partials then reads twice as much)
        if (rt >= 256) { t.nt = 2; t.wpb = 4; t.depth = K >= 8192 ? 2 : 3; }
        else { t.nt = 2; t.wpb = 8; t.depth = 2; }
    } else if (rt >= 1536) {         // LM head (short K: more waves share each row tile's chunks)
        if (K >= 2048) { t.nt = 4; t.wpb = 4; t.depth = 3; }
        else { t.nt = 2; t.wpb = 8; t.depth = 2; }
    } else if (rt >= 512) {          // QKV at LLaMA-7B width: 768 row tiles, 3 per workgroup
        t.nt = 3; t.wpb = 4; t.depth = 2;  // = 256 workgroups, one per CU (4 tiles: 192, 15 % slower)
    } else {
        t.nt = 1; t.wpb = 8; t.depth = 3;
    }
    return t;
}

// K splits of a split-K residual projection: enough splits for about 256 workgroups with
// the split geometry above, at most 8 and at least two 64-wide chunks per split
int skinny_row_groups(int M, int K, bool dual, bool split, bool wbf16)
{
    const SkinnyTuning tu = skinny_default_tuning(M, K, dual, split, wbf16);
    const int nt = dual && (tu.nt < 2 || tu.nt % 2) ? 2 : tu.nt;
    const int rows = (dual ? nt / 2 : nt) * 16;
    return (M + rows - 1) / rows;
}

int skinny_pick_ksplit(int M, int K, bool wbf16)
{
    const int nt = skinny_default_tuning(M, K, false, true, wbf16).nt;
    const int wgs = ((M + 15) / 16 + nt - 1) / nt, nchunk = (K + 63) / 64;
    int ks = std::max(1, std::min({(256 + wgs - 1) / wgs, nchunk / 2, 8}));
    const int cpb = (nchunk + ks - 1) / ks;
    return (nchunk + cpb - 1) / cpb;  // every split non-empty
}

jas_status skinny_gemm(const void *W, const void *W2, const float *X, long ldx, int M, int N, int K,
                       const SkinnyEpiArgs &epi, hipStream_t s, bool packed, bool wbf16)
{
    JAS_CHECK(!wbf16 || packed, JAS_ERR_INVALID, "skinny_gemm: bf16 weights only in the packed layout");
    JAS_CHECK(N >= 1 && N <= 16 && M > 0 && K > 0 && K % 4 == 0 && ldx % 4 == 0, JAS_ERR_INVALID,
              "skinny_gemm: unsupported shape");
    JAS_CHECK(!packed || K % 16 == 0, JAS_ERR_INVALID, "skinny_gemm: packed weights need K % 16 == 0");
    JAS_CHECK(!epi.out_packed || (M % 16 == 0 && (epi.mode == EPI_STORE || epi.mode == EPI_SWIGLU)), JAS_ERR_INVALID,
              "skinny_gemm: packed output needs M % 16 == 0");
    JAS_CHECK(al16(W) && al16(X) && (!W2 || al16(W2)), JAS_ERR_INVALID, "skinny_gemm: operands must be 16B aligned");
    const bool dual = epi.mode == EPI_SWIGLU;
    if (epi.mode == EPI_QKV)
        JAS_CHECK(epi.d % 16 == 0 && epi.dh % 4 == 0 && M == 3 * epi.d, JAS_ERR_INVALID, "skinny_gemm: bad QKV shape");
    if (dual) JAS_CHECK(W2 != nullptr, JAS_ERR_INVALID, "skinny_gemm: SwiGLU needs both weights");
    // row-major weights serve jas_gemm's few-token products only (store with any activation)
    JAS_CHECK(packed || (epi.mode == EPI_STORE && !epi.amax_v), JAS_ERR_INVALID, "skinny_gemm: packed weights only");
    JAS_CHECK(!epi.amax_v || (epi.mode == EPI_STORE && epi.act == JAS_ACT_NONE), JAS_ERR_INVALID, "skinny_gemm: bad LM head");
    SkinnyTuning tu = skinny_default_tuning(M, K, dual, epi.mode == EPI_PARTIAL, wbf16);
    if (!packed && tu.nt > 2) tu.nt = 2;  // more tiles: packed weights only
    SkinnyEpiArgs ep = epi;
    const int nchunk = (K + 63) / 64;
    if (ep.mode == EPI_PARTIAL) {
        JAS_CHECK(!dual && ep.ksplit >= 1 && ep.out, JAS_ERR_INVALID, "skinny_gemm: bad split-K partial request");
        ep.cpb = (nchunk + ep.ksplit - 1) / ep.ksplit;
        ep.ksplit = (nchunk + ep.cpb - 1) / ep.cpb;  // splits actually used (all non-empty)
        JAS_CHECK(ep.ksplit == epi.ksplit, JAS_ERR_INVALID, "skinny_gemm: K too short for the requested split");
    } else {
        ep.cpb = nchunk;
        ep.ksplit = 1;
    }
    const int kind = epi.amax_v ? (int)SE_HEAD : epi.mode == EPI_STORE && packed && epi.act == JAS_ACT_GELU ? (int)SE_GELU : epi.mode;
    // the geometries that skinny_default_tuning picks, each with the epilogues that reach it
#define JAS_SK(NTV, WPBV, DEP, DV, PV, WBV, EPIV)                                                          \
    if (tu.nt == NTV && tu.wpb == WPBV && tu.depth == DEP && packed == PV && wbf16 == WBV && kind == EPIV) { \
        launch_skinny<NTV, WPBV, DEP, DV, PV, WBV, EPIV>(W, W2, X, ldx, M, N, K, ep, s);                   \
        JAS_LAUNCH_CHECK();                                                                                \
        return JAS_OK;                                                                                     \
    }
    // whole projections: QKV, FC (GELU), LM head, and plain stores (jas_lm_project)
#define JAS_SK_W(NTV, WPBV, DEP, WBV)                                                                       \
    JAS_SK(NTV, WPBV, DEP, false, true, WBV, EPI_QKV) JAS_SK(NTV, WPBV, DEP, false, true, WBV, SE_GELU)     \
    JAS_SK(NTV, WPBV, DEP, false, true, WBV, SE_HEAD) JAS_SK(NTV, WPBV, DEP, false, true, WBV, EPI_STORE)
#define JAS_SK_P(NTV, WPBV, DEP, WBV) JAS_SK(NTV, WPBV, DEP, false, true, WBV, EPI_PARTIAL)
#define JAS_SK_D(NTV, WPBV, DEP, WBV) JAS_SK(NTV, WPBV, DEP, true, true, WBV, EPI_SWIGLU)
    JAS_SK_W(1, 8, 3, false) JAS_SK_W(2, 8, 2, false) JAS_SK_W(3, 4, 2, false) JAS_SK_W(4, 4, 3, false)
    JAS_SK_P(2, 8, 2, false) JAS_SK_P(2, 4, 2, false) JAS_SK_P(2, 4, 3, false)
    JAS_SK_D(2, 4, 3, false) JAS_SK_D(6, 4, 2, false)
    JAS_SK_W(1, 8, 3, true) JAS_SK_W(3, 4, 4, true) JAS_SK_W(4, 4, 2, true) JAS_SK_W(4, 4, 3, true)
    JAS_SK_P(2, 8, 2, true) JAS_SK_P(4, 4, 4, true)
    JAS_SK_D(2, 4, 3, true) JAS_SK_D(6, 4, 2, true)
    // row-major weights (nt clamped to two)
    JAS_SK(1, 8, 3, false, false, false, EPI_STORE) JAS_SK(2, 8, 2, false, false, false, EPI_STORE)
    JAS_SK(2, 4, 2, false, false, false, EPI_STORE) JAS_SK(2, 4, 3, false, false, false, EPI_STORE)
#undef JAS_SK_D
#undef JAS_SK_P
#undef JAS_SK_W
#undef JAS_SK
    return fail(JAS_ERR_INVALID, "skinny_gemm: unsupported tuning");
}

// ---------------------------------------------------------------- packed weight layout
// BF: the bf16 pair-tile layout (weight_pack_offset_b), K padded to a multiple of 32
template <bool BF>
__global__ void weight_pack_kernel(const void *__restrict__ src, void *__restrict__ dst, int M, int Mp, int K,
                                   int unpack)
{
    long p = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= (long)Mp * (BF ? k32_of(K) : K)) return;
    int r, k;
    if (BF) weight_pack_coords_b(p, K, Mp >> 4, &r, &k);
    else weight_pack_coords(p, K, Mp >> 4, &r, &k);
    const bool real = r < M && k < K;
    if (unpack) {
        const float v = BF ? bf16_to_f32(((const uint16_t *)src)[p]) : ((const float *)src)[p];
        if (real) ((float *)dst)[(long)r * K + k] = v;
    } else {
        const float v = real ? ((const float *)src)[(long)r * K + k] : 0.0f;
        if (BF) ((uint16_t *)dst)[p] = f32_to_bf16(v);
        else ((float *)dst)[p] = v;
    }
}

template <bool BF>
__global__ void fill_normal_packed_kernel(void *x, int M, int Mp, int K, uint64_t key, float mean, float std)
{
    long stride = (long)gridDim.x * blockDim.x;
    for (long p = (long)blockIdx.x * blockDim.x + threadIdx.x; p < (long)Mp * (BF ? k32_of(K) : K); p += stride) {
        int r, k;
        if (BF) weight_pack_coords_b(p, K, Mp >> 4, &r, &k);
        else weight_pack_coords(p, K, Mp >> 4, &r, &k);
        float v = 0.0f;
        if (r < M && k < K) {
            uint64_t i = (uint64_t)r * K + k;  // the row-major element index drives the generator
            uint64_t a = splitmix64(key + 2 * i), b = splitmix64(key + 2 * i + 1);
            double u1 = ((double)(a >> 11) + 1.0) * (1.0 / 9007199254740992.0);
            double u2 = (double)(b >> 11) * (1.0 / 9007199254740992.0);
            double z = sqrt(-2.0 * log(u1)) * cos(6.283185307179586 * u2);
            v = (float)((double)mean + (double)std * z);
        }
        if (BF) ((uint16_t *)x)[p] = f32_to_bf16(v);
        else ((float *)x)[p] = v;
    }
}

jas_status weight_pack(const void *src, void *dst, int M, int K, bool unpack, hipStream_t s, bool bf16)
{
    JAS_CHECK(K % 16 == 0, JAS_ERR_INVALID, "weight_pack: K must be a multiple of 16");
    const int Mp = (M + 15) / 16 * 16;
    long n = (long)Mp * (bf16 ? k32_of(K) : K);
    if (bf16)
        hipLaunchKernelGGL(weight_pack_kernel<true>, dim3(ceil_div(n, 256)), dim3(256), 0, s, src, dst, M, Mp, K,
                           unpack ? 1 : 0);
    else
        hipLaunchKernelGGL(weight_pack_kernel<false>, dim3(ceil_div(n, 256)), dim3(256), 0, s, src, dst, M, Mp, K,
                           unpack ? 1 : 0);
    JAS_LAUNCH_CHECK();
    return JAS_OK;
}

jas_status fill_normal_packed(void *x, int M, int K, uint64_t seed, uint64_t stream_id, float mean, float std,
                              hipStream_t s, bool bf16)
{
    JAS_CHECK(K % 16 == 0, JAS_ERR_INVALID, "fill_normal_packed: K must be a multiple of 16");
    const int Mp = (M + 15) / 16 * 16;
    unsigned nb = (unsigned)std::min<long>(((long)Mp * (bf16 ? k32_of(K) : K) + 255) / 256, 65536);
    if (bf16)
        hipLaunchKernelGGL(fill_normal_packed_kernel<true>, dim3(nb), dim3(256), 0, s, x, M, Mp, K,
                           stream_key(seed, stream_id), mean, std);
    else
        hipLaunchKernelGGL(fill_normal_packed_kernel<false>, dim3(nb), dim3(256), 0, s, x, M, Mp, K,
                           stream_key(seed, stream_id), mean, std);
    JAS_LAUNCH_CHECK();
    return JAS_OK;
}

// ---------------------------------------------------------------- fp64 GEMM
// 64x64 tile, K step 8, 256 threads (4 waves as 2x2 of 32x32): v_mfma_f64_16x16x4_f64 with
// A[i = l%16][k = l/16], B[k = l/16][j = l%16]; result register r of lane l holds
// D[i = l/16 + 4r][j = l%16] (the fp64 form interleaves rows, unlike the fp32 16x16x4).
typedef double doublex4 __attribute__((ext_vector_type(4)));

__global__ void __launch_bounds__(256)
gemm_f64_kernel(int M, int N, int K, const double *__restrict__ A, long as0, long as1, const double *__restrict__ B,
                long bs0, long bs1, double *__restrict__ C, long cs0, long cs1, const double *__restrict__ bias,
                int bias_mode)
{
    __shared__ double As[64][9];
    __shared__ double Bs[64][9];
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6, r16 = lane & 15, g = lane >> 4;
    const int wm = w >> 1, wn = w & 1;
    const int m0 = blockIdx.y * 64, n0 = blockIdx.x * 64;
    doublex4 acc[2][2];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) acc[i][j] = doublex4{0.0, 0.0, 0.0, 0.0};
    for (int k0 = 0; k0 < K; k0 += 8) {
        __syncthreads();
#pragma unroll
        for (int q = 0; q < 2; ++q) {  // 64 x 8 tiles of A and B, 512 elements each
            int idx = tid + q * 256, o = idx >> 3, k = idx & 7;
            int gm = m0 + o, gn = n0 + o, gk = k0 + k;
            As[o][k] = (gm < M && gk < K) ? A[(long)gm * as0 + (long)gk * as1] : 0.0;
            Bs[o][k] = (gn < N && gk < K) ? B[(long)gk * bs0 + (long)gn * bs1] : 0.0;
        }
        __syncthreads();
#pragma unroll
        for (int kk = 0; kk < 8; kk += 4)
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int j = 0; j < 2; ++j)
                    acc[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(As[wm * 32 + i * 16 + r16][kk + g],
                                                                     Bs[wn * 32 + j * 16 + r16][kk + g], acc[i][j], 0,
                                                                     0, 0);
    }
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                int m = m0 + wm * 32 + i * 16 + g + 4 * r, n = n0 + wn * 32 + j * 16 + r16;
                if (m >= M || n >= N) continue;
                double v = acc[i][j][r];
                if (bias_mode == 1) v = v + bias[m];
                else if (bias_mode == 2) v = v + bias[n];
                C[(long)m * cs0 + (long)n * cs1] = v;
            }
}

} // namespace jas

using namespace jas;

extern "C" jas_status jas_gemm_f64(int M, int N, int K, const double *A, long as0, long as1, const double *B, long bs0,
                                   long bs1, double *C, long cs0, long cs1, const double *bias, int bias_mode,
                                   jas_stream_t stream)
{
    JAS_CHECK(M >= 0 && N >= 0 && K >= 0 && A && B && C, JAS_ERR_INVALID, "jas_gemm_f64: bad arguments");
    JAS_CHECK(bias_mode >= 0 && bias_mode <= 2 && (bias_mode == 0 || bias), JAS_ERR_INVALID, "jas_gemm_f64: bad bias");
    if (M == 0 || N == 0) return JAS_OK;
    hipLaunchKernelGGL(gemm_f64_kernel, dim3(ceil_div(N, 64), ceil_div(M, 64)), dim3(256), 0, stream_or_default(stream),
                       M, N, K, A, as0, as1, B, bs0, bs1, C, cs0, cs1, bias, bias_mode);
    JAS_LAUNCH_CHECK();
    return JAS_OK;
}

extern "C" jas_status jas_gemm(int M, int N, int K, const float *A, long as0, long as1, const float *B, long bs0,
                               long bs1, float *C, long cs0, long cs1, const float *bias, int bias_mode, int act,
                               int accumulate, int batch, long abs_, long bbs, long cbs, long biasbs,
                               jas_stream_t stream)
{
    JAS_CHECK(M >= 0 && N >= 0 && K >= 0 && batch >= 1, JAS_ERR_INVALID, "jas_gemm: negative size");
    JAS_CHECK(A && B && C, JAS_ERR_INVALID, "jas_gemm: null operand");
    JAS_CHECK(bias_mode >= 0 && bias_mode <= 2 && (bias_mode == 0 || bias), JAS_ERR_INVALID, "jas_gemm: bad bias");
    JAS_CHECK(act >= JAS_ACT_NONE && act <= JAS_ACT_SIGMOID, JAS_ERR_INVALID, "jas_gemm: bad activation");
    if (M == 0 || N == 0) return JAS_OK;
    hipStream_t s = stream_or_default(stream);
    // decode shape: weights [M][K] row-major, tokens K-contiguous, token-major output
    if (batch == 1 && N <= 16 && as1 == 1 && bs0 == 1 && cs0 == 1 && K % 4 == 0 && as0 == K && bs1 % 4 == 0 &&
        al16(A) && al16(B) && bias_mode != 2 && !accumulate && K > 0) {
        SkinnyEpiArgs e;
        e.mode = EPI_STORE;
        e.act = act;
        e.bias = bias_mode == 1 ? bias : nullptr;
        e.out = C;
        e.ldo = cs1;
        return skinny_gemm(A, nullptr, B, bs1, M, N, K, e, s, false);
    }
    return gemm_general(M, N, K, A, as0, as1, B, bs0, bs1, C, cs0, cs1, bias, bias_mode, act, accumulate, batch, abs_,
                        bbs, cbs, biasbs, s, false);
}

extern "C" jas_status jas_gemm_residual(int M, int N, int K, const float *A, long as0, long as1, const float *B,
                                        long bs0, long bs1, float *C, long cs0, long cs1, const float *bias,
                                        int bias_mode, int act, const float *R, long rs0, long rs1,
                                        jas_stream_t stream)
{
    JAS_CHECK(M >= 0 && N >= 0 && K >= 0, JAS_ERR_INVALID, "jas_gemm_residual: negative size");
    JAS_CHECK(A && B && C && R, JAS_ERR_INVALID, "jas_gemm_residual: null operand");
    JAS_CHECK(bias_mode >= 0 && bias_mode <= 2 && (bias_mode == 0 || bias), JAS_ERR_INVALID,
              "jas_gemm_residual: bad bias");
    JAS_CHECK(act >= JAS_ACT_NONE && act <= JAS_ACT_SIGMOID, JAS_ERR_INVALID, "jas_gemm_residual: bad activation");
    if (M == 0 || N == 0) return JAS_OK;
    SplitArgs p{A, B, C, bias_mode ? bias : nullptr, as0, as1, bs0, bs1, cs0, cs1, 0, 0, 0, 0, M, N, K, bias_mode, act, 0};
    p.resid = R, p.rs0 = rs0, p.rs1 = rs1;
    return gemm_split(p, false, false, 1, stream_or_default(stream));
}
