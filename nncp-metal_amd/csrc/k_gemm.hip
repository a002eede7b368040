// GEMM for gfx950 (MI355X): column-major C = act(alpha*op(A)*op(B) + beta*C + bias) [+ addend].
//
// A workgroup of WM x WN wavefronts (times KW k groups) owns a BM x BN tile of C.  A and B
// tiles of depth BK are staged through LDS (double buffered, PF register sets of tiles in
// flight from global memory, k-major rows so a wavefront reads 32 consecutive floats), and
// every wavefront accumulates its part with v_mfma_f32_32x32x2_f32.  The MFMA is issued as
// D[n][m] = sum_k B[k][n]*A[k][m] so that the 32 lanes of a half-wavefront hold 32
// consecutive m of one column: the epilogue stores are 128-byte coalesced in column-major C.
//
// Tile classes (chosen from the shape only): 128x128x32 with 8 wavefronts, 128x64x32 with 8
// wavefronts, 64x64x32 with two k groups of 4 wavefronts (KW = 2: the groups split every
// 32-deep slab, C = chain0 + chain1).  Inside a class a C element is a fixed sequence of MFMA
// accumulations that does not depend on m, n or the number of columns; products with few tiles
// of the 64x64 class go to gemm_small_kernel, which issues the same sums.  The width-invariant
// class (NCHIP_GEMM_WIDTH_INVARIANT: 64x64x32, KW = 2, two accumulator sets per group = four
// chains per element, no split-K) is used by encoder and decoder alike when a column computed
// alone must equal the same column computed inside a larger matrix (bit-exact decode);
// gemm_skinny_nn issues the same sequence for products of a few columns.
//
// precision 1 rounds both operands to bf16 (nearest-even) while they are written to LDS and
// feeds v_mfma_f32_32x32x16_bf16 (fp32 accumulate); large products go through bf16 copies of
// the operands instead (cast_bf16_kernel + gemm_dma_kernel).
#include <hip/hip_runtime.h>
#include <hip/hip_ext.h>
#include <stdint.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>
#include <type_traits>
#include <vector>
#include "../../include/nchip_kernels.h"
#include "k_addrspace.h"
#include "k_bf16.h"
#include "k_act.h"
#include "k_norm_inline.h"
#include "k_lds_dma.h"

typedef float floatx16 __attribute__((ext_vector_type(16)));
typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef float floatx4_u __attribute__((ext_vector_type(4), aligned(4)));
typedef float floatx2_u __attribute__((ext_vector_type(2), aligned(4)));
typedef short shortx8 __attribute__((ext_vector_type(8)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4))); // a first-class value, unlike the uint4 struct

// (operand loads and result stores go through global-address-space pointers: k_addrspace.h)
namespace {

constexpr int KALIGN = 16; // split-K chunk granularity
constexpr int PAD = 4;   // keeps 16-byte alignment of LDS rows, staggers banks
constexpr int NXCD = 8;

#ifdef NCHIP_GEMM_CLOCKS
// debug builds: shader-clock and wall-clock span of the k loop of workgroup 0
__device__ long long *g_gemm_clk = nullptr;
#endif

struct GemmArgs {
    const float *A, *B;
    float *C;
    const float *bias;
    const float *add; // same layout as C, added after the activation (may be NULL)
    const float *dpre; // same layout as C: the result is multiplied by act'(dpre) (may be NULL)
    int dact;
    float *pre;
    float *ws;
    uint16_t *c16; // the result once more, rounded to bf16, laid out like C (may be NULL; gemm_dma_kernel only)
    int64_t lda, ldb, ldc, sa, sb, sc;   // outer batch strides
    int64_t sa_in, sb_in, sc_in;         // inner batch strides
    int batch_in;                        // batch index z -> (z / batch_in, z % batch_in)
    int M, N, K, batch, ksplit, kchunk;
    float alpha, beta;
    int act;
    int tiles_m, tiles_n;
    int gm; // tile rows per band of the tile order (see the kernel)
    int dbg;
    const NchipGemmProblem *grp; // grouped launch: one problem per table row
    int n_grp;
    int grp_chunk; // grouped launch: consecutive tiles of the list handed to one XCD at a time
    float *rowsum; // activation-gradient epilogue only: partial row sums of the result, one row per (tile column, wavefront column, lane half)
    // second product of a few-column pair launch (gemm_skinny_nn, blockIdx.z = 1): same B, N, K
    const float *A_1, *bias_1;
    float *C_1;
    int64_t lda_1, ldc_1;
    int M_1;
    // few-column kernel that normalises B on the way in (gemm_fewcol_mfma with NV > 0): gain and
    // bias (both or neither), the normalised columns written to ln_out (leading dimension
    // ld_ln) by the first row tile when it is not NULL
    const float *ln_w, *ln_b;
    float *ln_out;
    int64_t ld_ln;
    float ln_eps;
    int ln_avg;
};

__device__ __forceinline__ float gelu_tanh(float x) { return nchip_gelu(x); } // k_act.h

// GELU of the products that round their operands to bf16: the launchers turn NCHIP_ACT_GELU
// into this code when the precision argument is not fp32 (k_act.h says why there are two)
constexpr int ACT_GELU_FAST = 3;
static_assert(ACT_GELU_FAST != NCHIP_ACT_NONE && ACT_GELU_FAST != NCHIP_ACT_GELU && ACT_GELU_FAST != NCHIP_ACT_RELU, "");
inline int act_for_precision(int act, int precision) { return (act == NCHIP_ACT_GELU && precision != 0) ? ACT_GELU_FAST : act; }

__device__ __forceinline__ float act_grad(float x, int act)
{
    if (act == NCHIP_ACT_GELU) return nchip_gelu_grad(x);
    if (act == ACT_GELU_FAST) return nchip_gelu_grad_fast(x);
    if (act == NCHIP_ACT_RELU) return x > 0.0f ? 1.0f : 0.0f;
    return 1.0f;
}

__device__ __forceinline__ float apply_act(float v, int act)
{
    if (act == NCHIP_ACT_GELU) return gelu_tanh(v);
    if (act == ACT_GELU_FAST) return nchip_gelu_fast(v);
    if (act == NCHIP_ACT_RELU) return v > 0.0f ? v : 0.0f;
    return v;
}

__device__ __forceinline__ unsigned short f32_to_bf16(float f)
{
    unsigned int u = __float_as_uint(f);
    u += 0x7fffu + ((u >> 16) & 1u);
    return (unsigned short)(u >> 16);
}

__device__ __forceinline__ void wait_for_loads()
{
#if defined(__HIP_DEVICE_COMPILE__)
    __builtin_amdgcn_s_waitcnt(0);
#endif
}

// Loads a BT x BK tile (BT = BM or BN) of an operand into registers.
// MAJOR = 1: the tile's long axis (m or n) is contiguous in memory
//            (A with ta = 0, B with tb = 1);  element (i, k) at p[i + k*ld].
// MAJOR = 0: k is contiguous (A with ta = 1, B with tb = 0); (i, k) at p[k + i*ld].
//
// A k-contiguous tile is fetched row by row: BK / 4 consecutive lanes take one
// row's BK floats (whole 128-byte lines when BK = 32), so a wavefront touches
// 64 * 4 / BK rows instead of 64 - one cache line per lane was what bound these
// tiles.  Its LDS rows are BT + 1 floats apart (FPAD_K): the four transposing
// writes of a lane then fall on banks 4*(k/4) + e + i, distinct over the 32
// lanes served together.
constexpr int FPAD_K = 1;
template <int BT, int BK, int MAJOR, int NT>
struct TileLoader {
    static constexpr int NV = BT * BK / 4 / NT; // float4 per thread
    static constexpr int RS = BT + (MAJOR ? PAD : FPAD_K); // LDS row stride
    static_assert(NV >= 1 && NV * NT * 4 == BT * BK, "tile must divide evenly over the threads");
    floatx4 r[NV];

    __device__ __forceinline__ static void coords(int idx, int &i, int &k)
    {
        if (MAJOR) { i = (idx % (BT / 4)) * 4; k = idx / (BT / 4); }
        else       { i = idx / (BK / 4);       k = (idx % (BK / 4)) * 4; }
    }

    __device__ __forceinline__ void load(const float *p, int64_t ld, int i0, int k0,
                                         int imax, int kmax, bool fast, int t)
    {
#pragma unroll
        for (int v = 0; v < NV; v++) {
            int idx = t + v * NT;
            int i, k;
            coords(idx, i, k);
            if (fast) {
                const int ii = min(i0 + i, imax - 1); // (see whole_stages)
                const float *src = MAJOR ? p + (int64_t)(k0 + k) * ld + ii : p + (int64_t)ii * ld + (k0 + k);
                r[v] = *reinterpret_cast<const floatx4_u NCHIP_GLOBAL *>(as_global(src));
            } else {
                floatx4 tmp;
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    int ii = MAJOR ? i + e : i, kk = MAJOR ? k : k + e;
                    float val = 0.0f;
                    if (i0 + ii < imax && k0 + kk < kmax)
                        val = MAJOR ? as_global(p)[(int64_t)(k0 + kk) * ld + (i0 + ii)]
                                    : as_global(p)[(int64_t)(i0 + ii) * ld + (k0 + kk)];
                    tmp[e] = val;
                }
                r[v] = tmp;
            }
        }
    }

    // fp32 LDS tile: rows are k, RS floats each
    __device__ __forceinline__ void store_f32(float *lds, int t) const
    {
#pragma unroll
        for (int v = 0; v < NV; v++) {
            int i, k;
            coords(t + v * NT, i, k);
            if (MAJOR) {
                *reinterpret_cast<floatx4 *>(lds + k * RS + i) = r[v];
            } else {
#pragma unroll
                for (int e = 0; e < 4; e++)
                    lds[(k + e) * RS + i] = r[v][e];
            }
        }
    }
};

// bf16 variant of the loader.  LDS holds 32-bit words of two bf16 values that
// are consecutive in k: word (kp, i) = (x[i][2kp], x[i][2kp+1]), rows kp of
// BT + PAD words.  A lane of v_mfma_f32_32x32x16_bf16 (row i, k group kg) reads
// the 4 words kp = kb*8 + kg*4 .. +3 of column i: 8 consecutive k, lanes on
// consecutive banks.  Operands whose long axis is contiguous in memory are
// fetched as 2 columns x 2 rows (k, k+1) and stored as one 8-byte LDS write;
// k-contiguous operands give two words per float4.  Rounding is to nearest
// even (v_cvt_pk_bf16_f32).
// (pack_bf16: k_bf16.h)

template <int BT, int BK, int MAJOR, int NT>
struct TileLoaderBf16 {
    static constexpr int NV = BT * BK / 4 / NT; // 4-float units per thread
    static_assert(NV >= 1 && NV * NT * 4 == BT * BK, "tile must divide evenly over the threads");
    floatx4 r[NV];

    // MAJOR = 1: a unit is 2 columns x 2 consecutive k rows, r = (x[i][k], x[i+1][k], x[i][k+1], x[i+1][k+1]);
    // MAJOR = 0: a unit is 4 consecutive k of one column
    __device__ __forceinline__ static void coords(int v, int t, int &i, int &k)
    {
        int idx = t + v * NT;
        if (MAJOR) { i = (idx % (BT / 2)) * 2; k = (idx / (BT / 2)) * 2; }
        else       { i = idx % BT;             k = (idx / BT) * 4; }
    }

    __device__ __forceinline__ void load(const float *p, int64_t ld, int i0, int k0,
                                         int imax, int kmax, bool fast, int t)
    {
#pragma unroll
        for (int v = 0; v < NV; v++) {
            int i, k;
            coords(v, t, i, k);
            if (fast) {
                const int ii = min(i0 + i, imax - 1);
                if (MAJOR) {
                    const float *src = p + (int64_t)(k0 + k) * ld + ii;
                    floatx2_u a = *reinterpret_cast<const floatx2_u NCHIP_GLOBAL *>(as_global(src));
                    floatx2_u b = *reinterpret_cast<const floatx2_u NCHIP_GLOBAL *>(as_global(src) + ld);
                    r[v] = floatx4{ a[0], a[1], b[0], b[1] };
                } else {
                    r[v] = *reinterpret_cast<const floatx4_u NCHIP_GLOBAL *>(as_global(p) + (int64_t)ii * ld + (k0 + k));
                }
            } else {
                floatx4 tmp;
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    int ii = MAJOR ? i + (e & 1) : i, kk = MAJOR ? k + (e >> 1) : k + e;
                    float val = 0.0f;
                    if (i0 + ii < imax && k0 + kk < kmax)
                        val = MAJOR ? as_global(p)[(int64_t)(k0 + kk) * ld + (i0 + ii)]
                                    : as_global(p)[(int64_t)(i0 + ii) * ld + (k0 + kk)];
                    tmp[e] = val;
                }
                r[v] = tmp;
            }
        }
    }

    __device__ __forceinline__ void store(uint32_t *lds, int t) const
    {
#pragma unroll
        for (int v = 0; v < NV; v++) {
            int i, k;
            coords(v, t, i, k);
            if (MAJOR) {
                uint2 w = make_uint2(pack_bf16(r[v][0], r[v][2]), pack_bf16(r[v][1], r[v][3]));
                *reinterpret_cast<uint2 *>(lds + (k >> 1) * (BT + PAD) + i) = w;
            } else {
                lds[(k >> 1) * (BT + PAD) + i] = pack_bf16(r[v][0], r[v][1]);
                lds[((k >> 1) + 1) * (BT + PAD) + i] = pack_bf16(r[v][2], r[v][3]);
            }
        }
    }
};

// Epilogue of one 32x32 accumulator tile: acc[r] is C[m][nb + (r/4)*8 + r%4] (nb already
// holds the lane's (lane/32)*4).  The 16 values go to 16 columns of C.  Everything read here
// (addend, beta*C) is fetched for all 16 first, so the loads are in flight together, and the
// uniform option tests sit outside the element loops: a branch per element with a load
// behind it costs one memory round trip each.  Kernels that end here, and gemm_dma_kernel with the
// same steps in its own layout, write the same bits for the same accumulators.
__device__ __forceinline__ void epilogue_tile(const GemmArgs &g, const floatx16 &acc, int m, int nb,
                                              float NCHIP_GLOBAL *C, float NCHIP_GLOBAL *P,
                                              const float NCHIP_GLOBAL *Radd, const float NCHIP_GLOBAL *Dp,
                                              bool full, bool plain, float NCHIP_GLOBAL *rowsum = nullptr)
{
    if (!full && m >= g.M) return;
    float NCHIP_GLOBAL *Cp = C + (int64_t)nb * g.ldc + m; // element r lives at Cp + nofs(r)*ldc
    auto nofs = [](int r) { return (r >> 2) * 8 + (r & 3); };
    if (plain && full) {
#pragma unroll
        for (int r = 0; r < 16; r++) Cp[(int64_t)nofs(r) * g.ldc] = g.alpha * acc[r];
        return;
    }
    bool ok[16];
#pragma unroll
    for (int r = 0; r < 16; r++) ok[r] = full || nb + nofs(r) < g.N;
    float extra[16]; // beta*C + addend
#pragma unroll
    for (int r = 0; r < 16; r++) extra[r] = 0.0f;
    if (Radd) {
        const float NCHIP_GLOBAL *Ap = Radd + (int64_t)nb * g.ldc + m;
#pragma unroll
        for (int r = 0; r < 16; r++) extra[r] = ok[r] ? Ap[(int64_t)nofs(r) * g.ldc] : 0.0f;
    }
    float prev[16];
    const bool has_beta = g.beta != 0.0f;
    if (has_beta) {
#pragma unroll
        for (int r = 0; r < 16; r++) prev[r] = ok[r] ? Cp[(int64_t)nofs(r) * g.ldc] : 0.0f;
    }
    const float bv = g.bias ? as_global(g.bias)[m] : 0.0f;
    float v[16];
#pragma unroll
    for (int r = 0; r < 16; r++) {
        v[r] = g.alpha * acc[r];
        if (has_beta) v[r] += g.beta * prev[r];
        v[r] += bv;
    }
    if (P) {
        float NCHIP_GLOBAL *Pp = P + (int64_t)nb * g.ldc + m;
#pragma unroll
        for (int r = 0; r < 16; r++)
            if (ok[r]) Pp[(int64_t)nofs(r) * g.ldc] = v[r];
    }
    if (g.act == NCHIP_ACT_GELU) {
#pragma unroll
        for (int r = 0; r < 16; r++) v[r] = gelu_tanh(v[r]);
    } else if (g.act == ACT_GELU_FAST) {
#pragma unroll
        for (int r = 0; r < 16; r++) v[r] = nchip_gelu_fast(v[r]);
    } else if (g.act == NCHIP_ACT_RELU) {
#pragma unroll
        for (int r = 0; r < 16; r++) v[r] = v[r] > 0.0f ? v[r] : 0.0f;
    }
    if (Dp) { // gradient through an activation: times act'(pre-activation)
        const float NCHIP_GLOBAL *Dq = Dp + (int64_t)nb * g.ldc + m;
        float pz[16];
#pragma unroll
        for (int r = 0; r < 16; r++) pz[r] = ok[r] ? Dq[(int64_t)nofs(r) * g.ldc] : 0.0f;
#pragma unroll
        for (int r = 0; r < 16; r++) v[r] = (v[r] + extra[r]) * act_grad(pz[r], g.dact);
#pragma unroll
        for (int r = 0; r < 16; r++)
            if (ok[r]) Cp[(int64_t)nofs(r) * g.ldc] = v[r];
        if (rowsum) { // this lane's 16 columns of row m, in column order: one entry of a partial row
            float sum = 0.0f;
#pragma unroll
            for (int r = 0; r < 16; r++) sum += ok[r] ? v[r] : 0.0f;
            rowsum[m] = sum;
        }
        return;
    }
#pragma unroll
    for (int r = 0; r < 16; r++) v[r] += extra[r];
#pragma unroll
    for (int r = 0; r < 16; r++)
        if (ok[r]) Cp[(int64_t)nofs(r) * g.ldc] = v[r];
}

// Product with a few token columns for the width-invariant class: C (M x N, 32 columns per
// workgroup column) = A (M x K, m contiguous, M a multiple of 32) * B (K x N, k contiguous),
// fp32, K a multiple of 32, operand columns 16-byte aligned.  Per output element it issues
// exactly the MFMA sequence of the four-chain 64x64x32 tile kernel (gemm_kernel with
// NACC = 2: chain c takes k%32 in [8c, 8c+8), two k per v_mfma_f32_32x32x2_f32 in increasing
// order; C = (c0 + c1) + (c2 + c3); the same epilogue), so its columns are bit-identical to
// those of a wide product.  What differs is the plumbing.  A workgroup is one 32-row tile
// and its four wavefronts are the four chains, one per SIMD: the product then runs at the
// speed of one dependent MFMA chain of K/8 instructions, the least this arithmetic allows
// on one CU.  There is nothing to share between wavefronts, so the k loop has no barrier:
// a wavefront fetches its 8 k of every slab with ONE 16-byte load per lane and operand
// (8 x 32 rows of A, 32 columns x 8 k of B), PFD slabs ahead - at 2 microseconds of
// latency and 256 cycles of MFMA per slab the loads of 16 slabs must be in flight - and
// turns them into MFMA fragments through a private corner of LDS (in order within a
// wavefront, so a write followed by a read needs no barrier).  Columns past the edge read
// a clamped address and are never stored.
template <int PFD>
__global__ __launch_bounds__(256) void gemm_skinny_nn(GemmArgs g)
{
    static_assert(PFD % 2 == 0, "fragment registers alternate by slab parity");
    constexpr int AST = 36, BST = 12; // row strides of the staged slabs: A [8 k][32 m], B [32 n][8 k]
    __shared__ __attribute__((aligned(16))) float stage[4][8 * AST + 32 * BST];
    __shared__ float red[3][16 * 64];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    if (blockIdx.z == 1) { // the pair's second product: its own A, C, bias and row count
        g.A = g.A_1; g.C = g.C_1; g.bias = g.bias_1; g.lda = g.lda_1; g.ldc = g.ldc_1; g.M = g.M_1;
    }
    const int m0 = blockIdx.x * 32, n0 = blockIdx.y * 32;
    if (m0 >= g.M) return; // (uniform: the grid covers the taller of the two products)
    const int kh = lane >> 5;
    const int ak = lane >> 3, am = (lane & 7) * 4; // this lane's k row and first of four rows m of the A slab
    const int bn = lane >> 1, bk = (lane & 1) * 4; // this lane's column and first of four k of the B slab
    const int bcol = n0 + bn < g.N ? n0 + bn : g.N - 1;
    const floatx4 NCHIP_GLOBAL *Ag = reinterpret_cast<const floatx4 NCHIP_GLOBAL *>(
        as_global(g.A) + (int64_t)(8 * w + ak) * g.lda + m0 + am);
    const floatx4 NCHIP_GLOBAL *Bg = reinterpret_cast<const floatx4 NCHIP_GLOBAL *>(
        as_global(g.B) + (int64_t)bcol * g.ldb + 8 * w + bk);
    const int64_t a_step = 8 * g.lda; // 32 k rows, in 16-byte units
    float *As = stage[w], *Bs = As + 8 * AST;
    floatx4 *aw = reinterpret_cast<floatx4 *>(As + ak * AST + am);
    floatx4 *bw = reinterpret_cast<floatx4 *>(Bs + bn * BST + bk);
    const float *ar = As + kh * AST + (lane & 31); // MFMA step s reads k = 2s + kh
    const float *br = Bs + (lane & 31) * BST + kh;
    const int nslab = g.K / 32;
    floatx4 ra[PFD], rb[PFD];
    // (register sets and fragment sets are passed by reference: every index below is a
    // constant once the loops are unrolled, so the arrays stay in registers)
    auto load = [&](floatx4 &a, floatx4 &b, int slab) {
        slab = slab < nslab ? slab : nslab - 1; // past the end: the last slab again, never used
        a = Ag[slab * a_step];
        b = Bg[slab * 8];
    };
    float fa[2][4], fb[2][4];
    auto stage_slab = [&](const floatx4 &a, const floatx4 &b, float (&xa)[4], float (&xb)[4]) { // registers -> LDS -> fragments
        *aw = a;
        *bw = b;
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int s4 = 0; s4 < 4; s4++) {
            xa[s4] = ar[2 * s4 * AST];
            xb[s4] = br[2 * s4];
        }
        __builtin_amdgcn_wave_barrier();
    };
#pragma unroll
    for (int j = 0; j < PFD; j++) {
        load(ra[j], rb[j], j);
        __builtin_amdgcn_sched_barrier(0); // oldest slab first, as on the back edge
    }
    floatx16 acc;
#pragma unroll
    for (int r = 0; r < 16; r++) acc[r] = 0.0f;
    stage_slab(ra[0], rb[0], fa[0], fb[0]);
    load(ra[0], rb[0], PFD);
    for (int slab0 = 0; slab0 < nslab; slab0 += PFD) {
#pragma unroll
        for (int j = 0; j < PFD; j++) {
            // fragments of the next slab while the MFMAs of this one run
            stage_slab(ra[(j + 1) % PFD], rb[(j + 1) % PFD], fa[(j + 1) & 1], fb[(j + 1) & 1]);
            load(ra[(j + 1) % PFD], rb[(j + 1) % PFD], slab0 + j + 1 + PFD);
            __builtin_amdgcn_sched_barrier(0);
            if (slab0 + j < nslab) { // uniform
#pragma unroll
                for (int s4 = 0; s4 < 4; s4++)
                    acc = __builtin_amdgcn_mfma_f32_32x32x2f32(fb[j & 1][s4], fa[j & 1][s4], acc, 0, 0, 0);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
    }
    if (w > 0) {
#pragma unroll
        for (int r = 0; r < 16; r++) red[w - 1][r * 64 + lane] = acc[r];
    }
    __syncthreads();
    if (w > 0) return;
#pragma unroll
    for (int r = 0; r < 16; r++) acc[r] = (acc[r] + red[0][r * 64 + lane]) + (red[1][r * 64 + lane] + red[2][r * 64 + lane]);
    const bool full = n0 + 32 <= g.N;
    float NCHIP_GLOBAL *P = g.pre ? as_global(g.pre) : nullptr;
    const float NCHIP_GLOBAL *Radd = g.add ? as_global(g.add) : nullptr;
    const float NCHIP_GLOBAL *Dp = g.dpre ? as_global(g.dpre) : nullptr;
    const bool plain = !g.bias && !P && !Radd && !Dp && g.beta == 0.0f && g.act == NCHIP_ACT_NONE;
    epilogue_tile(g, acc, m0 + (lane & 31), n0 + kh * 4, as_global(g.C), P, Radd, Dp, full, plain);
}

// The same few-column product on the vector ALUs.  An fp32 MFMA accumulates its k values
// one after the other with fused multiply-adds, in increasing k (checked bit for bit against
// v_mfma_f32_32x32x2_f32 chains, denormal products included), so an output element of the
// width-invariant class is four chains of K/4 dependent v_fma_f32 - chain c takes k%32 in
// [8c, 8c+8) - summed as (c0 + c1) + (c2 + c3).  A thread is one chain of one element: a
// workgroup of 256 threads owns an 8 x 8 tile of C (4 chains each), so a 512 x 32 product
// spreads over 256 workgroups instead of 16 and a chain costs K/4 FMAs (0.3 microseconds at
// K = 512) instead of K/8 MFMAs of 64 cycles.  Its 8 rows of A and 8 columns of B pass
// through LDS in chunks of 256 k ([row][k] with k contiguous, two buffers, one barrier per
// chunk); the loads of up to PF chunks are in flight from the start (K = 2048 whole), since
// one memory round trip is longer than all the arithmetic.  Bias and addend are fetched
// before the k loop.  alpha = 1, beta = 0, no activation gradient; M a multiple of 8.
// Row tile of workgroup x of a few-column kernel.  Consecutive workgroups go to the eight XCDs
// in turn, each with an L2 of its own, and a 128-byte line of A (32 rows of one k) spans R
// row tiles: the R tiles that share lines are given to workgroups of one XCD (x, x + 8, ...),
// so that a line is fetched into one L2 and not into R of them.
__device__ __forceinline__ int fewcol_row_tile(int x, int ntiles, int R)
{
    const int span = 8 * R, group = x / span;
    if ((group + 1) * span > ntiles) return x; // a last, partial group keeps its order
    const int in = x - group * span, xcd = in & 7, r = in >> 3;
    return group * span + xcd * R + r;
}

constexpr int FC_KC = 256, FC_RS = FC_KC + 4;
template <int PF>
__global__ __launch_bounds__(256) void gemm_fewcol_fma(GemmArgs g)
{
    __shared__ __attribute__((aligned(16))) float tile[2][16 * FC_RS]; // rows 0-7: A rows, 8-15: B columns
    const int t = threadIdx.x;
    if (blockIdx.z == 1) { // the pair's second product: its own A, C, bias and row count
        g.A = g.A_1; g.C = g.C_1; g.bias = g.bias_1; g.lda = g.lda_1; g.ldc = g.ldc_1; g.M = g.M_1;
    }
    const int m0 = fewcol_row_tile(blockIdx.x, gridDim.x, 4) * 8, n0 = blockIdx.y * 8;
    if (m0 >= g.M) return; // (uniform: the grid covers the taller of the two products)
    const int ch = t & 3, ei = (t >> 2) & 7, ej = t >> 5; // chain, row and column of this thread's element
    const int nslab = g.K / 32, nch = (g.K + FC_KC - 1) / FC_KC;
    // A chunk: 256 k x 8 rows = 512 16-byte pieces (k = piece / 2, four rows each);
    // B chunk: 8 columns x 256 k = 512 pieces (column = piece / 64, four k each)
    const int ak[2] = { t >> 1, (t + 256) >> 1 }, ah = (t & 1) * 4;
    const int bj[2] = { t >> 6, (t + 256) >> 6 }, bk = (t & 63) * 4;
    const float NCHIP_GLOBAL *Ab = as_global(g.A) + m0 + ah;
    const float NCHIP_GLOBAL *Bb[2];
#pragma unroll
    for (int u = 0; u < 2; u++) {
        const int col = n0 + bj[u] < g.N ? n0 + bj[u] : g.N - 1;
        Bb[u] = as_global(g.B) + (int64_t)col * g.ldb;
    }
    floatx4 ra[PF][2], rb[PF][2];
    auto load = [&](floatx4 (&a)[2], floatx4 (&b)[2], int q) { // past the end: clamped, never used
#pragma unroll
        for (int u = 0; u < 2; u++) {
            int ka = q * FC_KC + ak[u], kb = q * FC_KC + bk;
            ka = ka < g.K ? ka : g.K - 1;
            kb = kb < g.K ? kb : g.K - 4;
            a[u] = *reinterpret_cast<const floatx4 NCHIP_GLOBAL *>(Ab + (int64_t)ka * g.lda);
            b[u] = *reinterpret_cast<const floatx4 NCHIP_GLOBAL *>(Bb[u] + kb);
        }
    };
#pragma unroll
    for (int j = 0; j < PF; j++) {
        load(ra[j], rb[j], j);
        __builtin_amdgcn_sched_barrier(0); // oldest chunk first
    }
    const int row = m0 + ei, col = n0 + ej;
    const bool ok = col < g.N;
    float NCHIP_GLOBAL *P = g.pre ? as_global(g.pre) : nullptr;
    const float NCHIP_GLOBAL *Radd = g.add ? as_global(g.add) : nullptr;
    const bool plain = !g.bias && !P && !Radd && g.act == NCHIP_ACT_NONE;
    const float bv = g.bias ? as_global(g.bias)[row] : 0.0f;
    const float extra = (Radd && ok) ? Radd[(int64_t)col * g.ldc + row] : 0.0f;
    auto park = [&](const floatx4 (&a)[2], const floatx4 (&b)[2], float *dst) { // registers -> [row][k]
#pragma unroll
        for (int u = 0; u < 2; u++) {
#pragma unroll
            for (int r = 0; r < 4; r++) dst[(ah + r) * FC_RS + ak[u]] = a[u][r];
            *reinterpret_cast<floatx4 *>(dst + (8 + bj[u]) * FC_RS + bk) = b[u];
        }
    };
    float acc = 0.0f;
    for (int q0 = 0; q0 < nch; q0 += PF) {
#pragma unroll
        for (int j = 0; j < PF; j++) {
            const int q = q0 + j;
            if (q < nch) { // uniform
                float *buf = tile[q & 1];
                park(ra[j], rb[j], buf);
                load(ra[j], rb[j], q + PF);
                __syncthreads();
                const float *wr = buf + ei * FC_RS + 8 * ch, *xr = buf + (8 + ej) * FC_RS + 8 * ch;
                const int ns = nslab - 8 * q < 8 ? nslab - 8 * q : 8;
                auto slab = [&](int s) {
                    const floatx4 w0 = *reinterpret_cast<const floatx4 *>(wr + 32 * s);
                    const floatx4 w1 = *reinterpret_cast<const floatx4 *>(wr + 32 * s + 4);
                    const floatx4 x0 = *reinterpret_cast<const floatx4 *>(xr + 32 * s);
                    const floatx4 x1 = *reinterpret_cast<const floatx4 *>(xr + 32 * s + 4);
#pragma unroll
                    for (int r = 0; r < 4; r++) acc = __builtin_fmaf(x0[r], w0[r], acc);
#pragma unroll
                    for (int r = 0; r < 4; r++) acc = __builtin_fmaf(x1[r], w1[r], acc);
                };
                if (ns == 8) { // a whole chunk, unrolled: the LDS reads run ahead of the chain
#pragma unroll
                    for (int s = 0; s < 8; s++) slab(s);
                } else {
                    for (int s = 0; s < ns; s++) slab(s);
                }
            }
        }
    }
    // (c0 + c1) + (c2 + c3): the four chains of an element sit in four neighbouring lanes
    float v = acc + __shfl_xor(acc, 1, 64);
    v = v + __shfl_xor(v, 2, 64);
    if (ch != 0 || !ok) return;
    float NCHIP_GLOBAL *Cp = as_global(g.C) + (int64_t)col * g.ldc + row;
    if (plain) {
        *Cp = g.alpha * v;
        return;
    }
    v = g.alpha * v + bv;
    if (P) P[(int64_t)col * g.ldc + row] = v;
    v = apply_act(v, g.act);
    *Cp = v + extra;
}

// The few-column product with v_mfma_f32_16x16x4_f32.  That instruction accumulates its
// four k in increasing order like the 32x32x2 one its two, at a quarter of the chain latency
// per k (a 16x16 tile: 8 passes per 4 k instead of 16 passes per 2 k), so chain c of a slab
// is two of them (k%32 = 8c..8c+3, 8c+4..8c+7) and the result is again the bits of the tile
// kernel.  A workgroup is a 16 x 16 tile of C and its four wavefronts are the four chains
// (combined as (c0 + c1) + (c2 + c3) through LDS at the end); a wavefront fetches only the
// 8 k per slab of its own chain - 16 rows of A and 16 columns of B, in chunks of 256 k, up
// to PF chunks in flight - into a private corner of LDS and reads its fragments from there,
// so the k loop has no workgroup barrier.  Against the vector-ALU kernel: a quarter of the
// workgroups, but 1 KB of LDS reads per slab and wavefront for 256 outputs instead of 4 KB
// for 16, which is what bounds that kernel on the taller products.  alpha = 1, beta = 0.
//
// NV > 0: B holds K = 64 NV raw features per column and the product is taken with their
// layer norm (or RMS norm) - the arithmetic of norm_fwd_reg, wavefront c normalising columns
// 4c..4c+3 of the tile before the k loop, the result kept whole in LDS (every workgroup
// repeats it for its 16 columns, which costs less than a launch of its own); the first row
// tile also writes the normalised columns out for the later consumers of that tensor.
//
// TR = 8: tiles of 8 x 8 outputs on the same instruction (rows and columns 8-15 of the MFMA
// tile repeat 0-7 and are not stored): four times the workgroups, for a long reduction and for
// products that would otherwise leave most CUs idle.  What bounds these kernels is not the
// chain (0.85 microseconds per 1024 k) but the 128-byte lines a workgroup must bring in, at
// about 0.4 lines per nanosecond and CU, with warm or cold weights alike: a launch costs about
// 2.6 microseconds plus 2.3 nanoseconds per line of its busiest workgroup.  With A stored
// rows-contiguous that is one line of A per k whatever the tile height up to 32 rows.
//
// AK = 1: A is stored with k contiguous (lda between rows: a k-major copy of a weight matrix).
// The lines a workgroup brings in for A are then TR x K/32 instead of K, which is what the
// kernel is bound by; the arithmetic is the same.
template <int PF, int NV = 0, int TR = 16, int AK = 0>
__global__ __launch_bounds__(256) void gemm_fewcol_mfma(GemmArgs g)
{
    static_assert(TR == 16 || (TR == 8 && NV == 0), "8 x 8 tiles: plain products only");
    constexpr int NU = TR / 4; // 16-byte pieces per lane, chunk and operand
    constexpr int BST = 68, ASZ = AK ? TR * BST : 64 * TR; // per wavefront: A [64 k][TR rows] (AK: [TR rows][64 k]), B [TR columns][64 k]
    constexpr int WSZ = ASZ + (NV ? 0 : TR * BST);
    constexpr int XS = 64 * NV + 4;
    __shared__ __attribute__((aligned(16))) float stage[4][WSZ];
    __shared__ float red[4][4 * 64];
    __shared__ float xn[NV ? 16 * XS : 1]; // normalised B: [16 columns][K]
    const int lane = threadIdx.x & 63, c = threadIdx.x >> 6; // wavefront = chain
    if (blockIdx.z == 1) { // the pair's second product: its own A, C, bias and row count
        g.A = g.A_1; g.C = g.C_1; g.bias = g.bias_1; g.lda = g.lda_1; g.ldc = g.ldc_1; g.M = g.M_1;
    }
    const int m0 = fewcol_row_tile(blockIdx.x, gridDim.x, 32 / TR) * TR, n0 = blockIdx.y * TR;
    if (m0 >= g.M) return; // (uniform: the grid covers the taller of the two products)
    const int il = lane & 15, gq = lane >> 4, it = il & (TR - 1); // (it: this lane's row / column of the tile)
    const int nslab = g.K / 32, nch = (g.K + 255) / 256;
    float *As = stage[c], *Bs = As + ASZ;
    // this lane's NU 16-byte pieces of A (k_local = piece / NU, four rows) and of B
    // (column = piece / 16, slab = (piece % 16) / 2, half a chain's 8 k)
    const float NCHIP_GLOBAL *Ab = as_global(g.A) + m0 + (lane & (NU - 1)) * 4;
    const float NCHIP_GLOBAL *Ar[NU]; // AK: the row of each piece (pieces laid out as those of B)
    const float NCHIP_GLOBAL *Bb[NU];
    int a_k[NU], b_k[NU];
#pragma unroll
    for (int u = 0; u < NU; u++) {
        const int pa = lane + 64 * u, kl = pa / NU;
        a_k[u] = 32 * (kl >> 3) + 8 * c + (kl & 7);
        const int pb = lane + 64 * u, colb = pb >> 4, kq = pb & 15;
        const int col = n0 + colb < g.N ? n0 + colb : g.N - 1;
        Bb[u] = as_global(g.B) + (int64_t)col * g.ldb;
        b_k[u] = 32 * (kq >> 1) + 8 * c + 4 * (kq & 1);
        Ar[u] = as_global(g.A) + (int64_t)(m0 + colb) * g.lda;
    }
    floatx4 ra[PF][NU], rb[NV ? 1 : PF][NU];
    auto load = [&](floatx4 (&a)[NU], floatx4 (&b)[NU], int q) { // past the end: clamped, never used
#pragma unroll
        for (int u = 0; u < NU; u++) {
            int ka = q * 256 + a_k[u], kb = q * 256 + b_k[u];
            ka = ka < g.K ? ka : g.K - 1;
            kb = kb < g.K ? kb : g.K - 4;
            if (AK) a[u] = *reinterpret_cast<const floatx4 NCHIP_GLOBAL *>(Ar[u] + kb);
            else a[u] = *reinterpret_cast<const floatx4 NCHIP_GLOBAL *>(Ab + (int64_t)ka * g.lda);
            if (NV == 0) b[u] = *reinterpret_cast<const floatx4 NCHIP_GLOBAL *>(Bb[u] + kb);
        }
    };
    // the raw columns first: they are needed first
    float xv[NV ? 4 : 1][NV ? NV : 1], lw[NV ? NV : 1], lb[NV ? NV : 1];
    if (NV > 0) {
#pragma unroll
        for (int cc = 0; cc < 4; cc++) {
            const int colb = 4 * c + cc, gcol = n0 + colb < g.N ? n0 + colb : g.N - 1;
            const float NCHIP_GLOBAL *xc = as_global(g.B) + (int64_t)gcol * g.ldb + lane;
#pragma unroll
            for (int v = 0; v < NV; v++) xv[cc][v] = xc[64 * v];
        }
        if (g.ln_w) {
#pragma unroll
            for (int v = 0; v < NV; v++) { lw[v] = as_global(g.ln_w)[lane + 64 * v]; lb[v] = as_global(g.ln_b)[lane + 64 * v]; }
        }
        __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
    for (int j = 0; j < PF; j++) {
        load(ra[j], rb[NV ? 0 : j], j);
        __builtin_amdgcn_sched_barrier(0); // oldest chunk first
    }
    if constexpr (NV > 0) {
        float hh[4][NV], yy[4][NV], rr[4];
        norm_columns_reg<NV, 4>(xv, lw, lb, g.ln_w != nullptr, g.ln_eps, g.ln_avg, hh, yy, rr);
#pragma unroll
        for (int cc = 0; cc < 4; cc++) {
            const int colb = 4 * c + cc;
#pragma unroll
            for (int v = 0; v < NV; v++) xn[colb * XS + lane + 64 * v] = yy[cc][v];
            if (g.ln_out && blockIdx.x == 0 && blockIdx.z == 0 && n0 + colb < g.N) {
                float NCHIP_GLOBAL *yo = as_global(g.ln_out) + (int64_t)(n0 + colb) * g.ld_ln + lane;
#pragma unroll
                for (int v = 0; v < NV; v++) yo[64 * v] = yy[cc][v];
            }
        }
        __syncthreads();
    }
    // epilogue operands, fetched before the k loop: wavefront c finishes row 4 gq + c of the
    // four rows a lane holds (the four chains of an element meet through LDS either way, and
    // bias, activation and addend then take a quarter of the time on each wavefront)
    const int col = n0 + il, row = m0 + 4 * gq + c;
    const bool ok = col < g.N && il < TR && gq < TR / 4; // (8 x 8 tiles: the repeated rows and columns are not stored)
    float NCHIP_GLOBAL *P = g.pre ? as_global(g.pre) : nullptr;
    const float NCHIP_GLOBAL *Radd = g.add ? as_global(g.add) : nullptr;
    const bool plain = !g.bias && !P && !Radd && g.act == NCHIP_ACT_NONE;
    const float bv = (g.bias && gq < TR / 4) ? as_global(g.bias)[row] : 0.0f;
    const float extra = (Radd && ok) ? Radd[(int64_t)col * g.ldc + row] : 0.0f;
    floatx4 acc = { 0, 0, 0, 0 };
    for (int q0 = 0; q0 < nch; q0 += PF) {
#pragma unroll
        for (int j = 0; j < PF; j++) {
            const int q = q0 + j;
            if (q < nch) { // uniform
#pragma unroll
                for (int u = 0; u < NU; u++) {
                    const int pa = lane + 64 * u;
                    if (AK) *reinterpret_cast<floatx4 *>(As + (pa >> 4) * BST + (pa & 15) * 4) = ra[j][u];
                    else *reinterpret_cast<floatx4 *>(As + (pa / NU) * TR + (pa & (NU - 1)) * 4) = ra[j][u];
                    if (NV == 0) *reinterpret_cast<floatx4 *>(Bs + (pa >> 4) * BST + (pa & 15) * 4) = rb[j][u];
                }
                load(ra[j], rb[NV ? 0 : j], q + PF);
                __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
                __builtin_amdgcn_wave_barrier();
                __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
                float fa[16], fb[16];
#pragma unroll
                for (int e = 0; e < 16; e++) { // MFMA e of the chunk: slab e / 2, k_local = 4 e + gq
                    fa[e] = AK ? As[it * BST + 4 * e + gq] : As[(4 * e + gq) * TR + it];
                    int kx = 256 * q + 32 * (e >> 1) + 8 * c + 4 * (e & 1) + gq;
                    kx = kx < g.K ? kx : g.K - 1; // (past a short last chunk: read, never used)
                    fb[e] = NV ? xn[il * XS + kx] : Bs[it * BST + 4 * e + gq];
                }
                __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
                __builtin_amdgcn_wave_barrier(); // the fragments are in registers: the corner may be rewritten
                const int ne = (nslab - 8 * q < 8 ? nslab - 8 * q : 8) * 2;
                if (ne == 16) {
#pragma unroll
                    for (int e = 0; e < 16; e++) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(fa[e], fb[e], acc, 0, 0, 0);
                } else {
#pragma unroll
                    for (int e = 0; e < 16; e++)
                        if (e < ne) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(fa[e], fb[e], acc, 0, 0, 0);
                }
            }
        }
    }
#pragma unroll
    for (int r = 0; r < 4; r++) red[c][r * 64 + lane] = acc[r];
    __syncthreads();
    if (!ok) return;
    // lane (il, gq) of wavefront c finishes row m0 + 4 gq + c of column n0 + il: (c0 + c1) + (c2 + c3)
    const float sum = (red[0][c * 64 + lane] + red[1][c * 64 + lane]) + (red[2][c * 64 + lane] + red[3][c * 64 + lane]);
    float NCHIP_GLOBAL *Cp = as_global(g.C) + (int64_t)col * g.ldc + row;
    if (plain) {
        *Cp = g.alpha * sum;
        return;
    }
    float v = g.alpha * sum + bv;
    if (P) P[(int64_t)col * g.ldc + row] = v;
    v = apply_act(v, g.act);
    *Cp = v + extra;
}

// The tile of this workgroup and, in a grouped launch, the problem that owns it (g receives that
// problem's operands and extents; A2 / B2 its second k range, from k1 on).
template <int BM, int BN>
__device__ __forceinline__ void find_tile(GemmArgs &g, int &tile_m, int &tile_n, const float *&A2, const float *&B2, int &k1)
{
    // XCD-aware tile order: the hardware deals consecutive workgroup ids round
    // robin over the 8 XCDs; give each XCD a contiguous run of tiles so tiles
    // that share an A/B panel also share an L2.
    int bid = blockIdx.x;
    A2 = B2 = nullptr;
    k1 = 0x7fffffff;
    if (g.grp) {
        // grouped launch: consecutive workgroup ids go to the XCDs in turn; hand each XCD
        // GC consecutive tiles of the list at a time (neighbours in a tile column, which share
        // a B panel in that XCD's L2) while the turn-taking keeps the XCDs' work balanced
        {
            const int GC = g.grp_chunk;
            const int total = gridDim.x, span = NXCD * GC;
            if (GC > 1 && (bid / span + 1) * span <= total) {
                const int in = bid % span, x = in % NXCD, slot = in / NXCD;
                bid = (bid / span) * span + x * GC + slot;
            }
        }
        // find the problem that owns this workgroup
        int lo = 0, hi = g.n_grp; // grp[lo].tile_start <= bid < grp[hi].tile_start
        while (hi - lo > 1) {
            int mid = (lo + hi) >> 1;
            if (g.grp[mid].tile_start <= bid) lo = mid; else hi = mid;
        }
        const NchipGemmProblem pr = g.grp[lo];
        bid -= pr.tile_start;
        g.A = pr.A; g.B = pr.B; g.C = pr.C;
        g.M = pr.m; g.N = pr.n; g.K = pr.k + pr.k2;
        if (pr.k2 > 0) { A2 = pr.A2; B2 = pr.B2; k1 = pr.k; }
        g.lda = pr.lda; g.ldb = pr.ldb; g.ldc = pr.ldc;
        g.alpha = pr.alpha;
        g.kchunk = pr.k + pr.k2;
        g.tiles_m = (pr.m + BM - 1) / BM;
        g.tiles_n = (pr.n + BN - 1) / BN;
    }
    int ntiles = g.tiles_m * g.tiles_n;
    if (!g.grp && ntiles % NXCD == 0)
        bid = (bid % NXCD) * (ntiles / NXCD) + bid / NXCD;
    // Tile order inside an XCD's run: bands of gm tile rows, column by column
    // inside a band, so the workgroups in flight on one XCD form a block about
    // as wide as it is tall and share both A and B panels in that XCD's L2.
    if (g.gm > 1) {
        const int band = g.gm * g.tiles_n, bi = bid / band, first = bi * g.gm;
        const int rows = min(g.tiles_m - first, g.gm), r = bid - bi * band;
        tile_m = first + r % rows;
        tile_n = r / rows;
    } else {
        tile_m = bid % g.tiles_m;
        tile_n = bid / g.tiles_m;
    }
}

// f(0), f(1), ... with constants: arrays indexed by them stay in registers whatever the unroller's limits
template <typename F, int... I>
__device__ __forceinline__ void each_constant(F f, std::integer_sequence<int, I...>)
{
    (f(std::integral_constant<int, I>()), ...);
}

// Products of operands that are bf16 in memory, staged by DMA: global memory to LDS without a
// register in between, ST stages of 64 k in flight, so that a stage is asked for ST - 1 stages
// before it is read and a wavefront's registers hold accumulators and fragments only (256 x 256
// tiles fit).  An element is one chain of v_mfma_f32_32x32x16_bf16 over increasing k or, with NACC = 2,
// two of them - k % 32 below 16, and from 16 on - that are added (see bf16_two_chains).
//
// A stage holds each operand as it lies in memory, in units of 16 bytes.  k contiguous: rows of 64 k,
// unit c of row i in place c ^ (i / 2 & 7), a fragment is one 16-byte read.  Long axis contiguous: rows
// of one k, and a fragment is two transposing reads of 4 k x 16 each; 32-byte granules (16 values)
// are stored in place q ^ f(k) so that the four rows of a read lie in different banks.  The
// swizzles are applied to the global address, a DMA being linear in LDS.
//
// Bound by the matrix units and LDS together (a 128 x 64 wavefront tile reads 6 KB for 8 MFMAs) on
// large shapes: 16384 x 1024 x 4096 227 us with register staging, 122 now (1.12 PFLOP/s); on small ones
// by one memory round trip and the epilogue: 512 x 2048 x 512 6.8 -> 5.0 us.
//
// The stage of step it + 1 is waited for before the last quarter of step it, whose MFMAs cover the
// barrier and the first fragment reads of the next; that barrier also says that stage it has
// been read, and its place is refilled at once.
//
// F32: the same for fp32 operands, stages of 32 k.  v_mfma_f32_32x32x2_f32 takes one value a lane, k = 2 u +
// lane / 32 of step u: rows of one k are stored with their odd rows' halves of 64 exchanged, so that the
// two halves of a wavefront read different banks.  KW = 2 as in gemm_kernel, whose classes' sums
// these are.  Bound by the matrix pipe (64 cycles a step) but for first loads and epilogue:
// us before -> now, 512 x 2048 x 512 16.7 -> 14.5, 2048 x 2048 x 512 48.5 -> 42.0, the grouped weight
// gradients of 12 layers of 512 over 2048 tokens 1571 -> 1361 (133 TFLOP/s).
constexpr int BOX_LD = 36; // words between the columns of an accumulator tile in LDS
template <int F32, int BM, int BN, int WM, int WN, int KW, int ST, int TA, int TB, int NACC = 1, int FAR = 0>
__global__ __launch_bounds__(64 * WM * WN * KW) void gemm_dma_kernel(GemmArgs g0)
{
    GemmArgs g = g0;
    constexpr int NG = WM * WN, NT = 64 * NG * KW;
    constexpr int TM = BM / (32 * WM), TN = BN / (32 * WN), WTM = BM / WM, WTN = BN / WN;
    constexpr int E = F32 ? 4 : 2, V = 16 / E, BK = 128 / E; // bytes of an element, elements of a unit, k of a stage
    constexpr int NVA = BM * 8 / NT, NVB = BN * 8 / NT, NL = NVA + NVB; // 16-byte loads a lane and stage
    constexpr int STAGE = (BM + BN) * 64, NP = KW == 2 ? 2 : 4, NC = F32 ? NP : 1; // a stage in 16-bit words; parts its k is read in, chunks it is asked for in
    static_assert(KW == 1 || (F32 && KW == 2 && TM * TN == 1), "k groups: fp32, one accumulator tile a wavefront");
    static_assert(NACC == 1 || (!F32 && NACC == 2), "two accumulator sets: bf16");
    static_assert(NVA * NT == BM * 8 && NVB * NT == BN * 8, "whole loads");
    static_assert(ST >= 2 && ST <= 4 && (ST - 1) * NL <= 63, "arrive()'s counts; the memory counter has six bits");
    static_assert(NG * KW * 32 * BOX_LD * 4 <= ST * STAGE * 2, "the epilogue's corners fit where the stages were");
    extern __shared__ __attribute__((aligned(16))) uint16_t stages_lds[];
    uint16_t NCHIP_LDS *const stages = (uint16_t NCHIP_LDS *)stages_lds;
    const int t = threadIdx.x, lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6);
    const int kg = wave / NG, wm = wave % NG % WM, wn = wave % NG / WM, hi = lane >> 5;

    int tile_m, tile_n;
    const float *A2, *B2;
    int k1;
    find_tile<BM, BN>(g, tile_m, tile_n, A2, B2, k1);
    const int m0 = tile_m * BM, n0 = tile_n * BN;
    int kbeg = 0, kend = g.K;
    int64_t off_a = 0, off_b = 0;
    if constexpr (F32) { // batch entry and k chunk
        const int b = blockIdx.y / g.ksplit, kz = blockIdx.y % g.ksplit, out = b / g.batch_in, in = b % g.batch_in;
        if (!g.grp) { kbeg = kz * g.kchunk; kend = min(g.K, kbeg + g.kchunk); }
        off_a = out * g.sa + in * g.sa_in;
        off_b = out * g.sb + in * g.sb_in;
        const int64_t off_c = out * g.sc + in * g.sc_in;
        if (g.ksplit > 1) { // the chunk's sum alone, for gemm_splitk_reduce
            g.C = g.ws + ((int64_t)kz * g.batch + b) * g.M * g.N;
            g.ldc = g.M;
            g.bias = g.add = g.dpre = nullptr;
            g.pre = g.rowsum = nullptr;
            g.alpha = 1.0f; g.beta = 0.0f; g.act = NCHIP_ACT_NONE;
        } else {
            g.C += off_c;
            if (g.pre) g.pre += off_c;
            if (g.add) g.add += off_c;
            if (g.dpre) g.dpre += off_c;
        }
    }
    const int nk = (kend - kbeg) / BK, it2 = k1 / BK;

    // this lane's byte offsets inside a stage's panel of an operand (64 bits with FAR, for rows that far apart);
    // rows and units past the edge repeat the last one (their results are not stored)
    using Off = std::conditional_t<FAR != 0, uint64_t, uint32_t>;
    auto offsets = [&](auto &off, auto kcontig, auto extent, int64_t ld, int i0, int imax) {
        constexpr int BT = decltype(extent)::value, NV = BT * 8 / NT;
#pragma unroll
        for (int v = 0; v < NV; v++) {
            const int p = t + v * NT;
            if constexpr (decltype(kcontig)::value) {
                const int i = p / 8, row = i0 + i < imax ? i : imax - 1 - i0;
                off[v] = (Off)(E * (row * ld + ((p ^ i >> 1) & 7) * V));
            } else {
                constexpr int U = BT / V, SH = BT >= 128 ? 1 : 0;
                const int k = p / U, u = p % U;
                const int i = F32 ? (u ^ (k & 1) << 3) * V : (((u >> 1) ^ ((k & 3) << SH)) * 2 + (u & 1)) * V;
                off[v] = (Off)(E * (k * ld + (i0 + i + V <= imax ? i : imax - V - i0)));
            }
        }
    };
    Off oa[NVA], ob[NVB];
    // (a long axis that is no multiple of V lies in a copy whose columns are padded to one)
    offsets(oa, std::integral_constant<bool, TA != 0>(), std::integral_constant<int, BM>(), g.lda, m0, TA ? g.M : (g.M + V - 1) & ~(V - 1));
    offsets(ob, std::integral_constant<bool, TB == 0>(), std::integral_constant<int, BN>(), g.ldb, n0, TB ? (g.N + V - 1) & ~(V - 1) : g.N);
    const int64_t ea = E * (TA ? m0 * g.lda : m0), eb = E * (TB ? n0 : n0 * g.ldb);
    const int64_t sa = E * (TA ? BK : BK * g.lda), sb = E * (TB ? BK * g.ldb : BK); // bytes from stage to stage
    const char *pa = reinterpret_cast<const char *>(g.A) + E * (off_a + (TA ? kbeg : kbeg * g.lda)) + ea;
    const char *pb = reinterpret_cast<const char *>(g.B) + E * (off_b + (TB ? kbeg * g.ldb : kbeg)) + eb;
    int to = 0, asked = 0; // where the next stage goes, its number
    // chunk c of NC of the next stage's loads
    auto issue = [&](auto chunk, auto piece) { // piece: an index into the chunk
        constexpr int c = decltype(chunk)::value, v = c * NL / NC + decltype(piece)::value;
        if (v == 0 && asked == it2) {
            pa = reinterpret_cast<const char *>(A2) + ea;
            pb = reinterpret_cast<const char *>(B2) + eb;
        }
        uint16_t NCHIP_LDS *dst = stages + to * STAGE + wave * 512;
        if constexpr (v < NVA) lds_dma16(dst + v * NT * 8, pa, oa[v < NVA ? v : 0]);
        else lds_dma16(dst + BM * 64 + (v - NVA) * NT * 8, pb, ob[v < NVA ? 0 : v - NVA]);
        if constexpr (v == NL - 1) {
            pa += sa; pb += sb;
            asked++;
            to = to + 1 < ST ? to + 1 : 0;
        }
    };
    auto issue_chunk = [&](auto chunk) {
        constexpr int c = decltype(chunk)::value;
        each_constant([&](auto piece) { issue(chunk, piece); }, std::make_integer_sequence<int, (c + 1) * NL / NC - c * NL / NC>());
    };

    // fragments of part u of a stage's panel (bf16: 16 k; fp32: four steps of 2): offsets of lane and
    // tile, then constants
    auto fragment = [&](const uint16_t NCHIP_LDS *panel, auto kcontig, auto extent, int at, int j, int u) -> u32x4 {
        constexpr int BT = decltype(extent)::value;
        if constexpr (F32) {
            const uint32_t NCHIP_LDS *p = (const uint32_t NCHIP_LDS *)panel;
            const int i = at + j * 32 + (lane & 31), kb = (KW == 2 ? kg * 16 : 0) + u * 8;
            u32x4 r;
#pragma unroll
            for (int s = 0; s < 4; s++) {
                if constexpr (decltype(kcontig)::value) r[s] = p[i * 32 + (((kb / 4 + (s >> 1)) ^ (lane >> 1 & 7)) * 4) + 2 * (s & 1) + hi];
                else r[s] = p[(kb + 2 * s + hi) * BT + (i ^ hi << 5)];
            }
            return r;
        } else if constexpr (decltype(kcontig)::value) {
            return *reinterpret_cast<const u32x4 NCHIP_LDS *>(panel + (at + j * 32 + (lane & 31)) * 64 + (((u * 2 + hi) ^ (lane >> 1 & 7)) * 8));
        } else {
            constexpr int SH = BT >= 128 ? 1 : 0;
            const int k = u * 16 + hi * 8 + ((lane & 15) >> 2);
            const int q = (at / 16 + j * 2 + ((lane >> 4) & 1)) ^ ((k & 3) << SH);
            const uint16_t NCHIP_LDS *r = panel + k * BT + q * 16 + (lane & 3) * 4;
            const uint2 lo = lds_read_columns(r), up = lds_read_columns(r + 4 * BT);
            return u32x4{ lo.x, lo.y, up.x, up.y };
        }
    };
    floatx16 acc[TN][TM], acc2[NACC == 2 ? TN : 1][NACC == 2 ? TM : 1];
#pragma unroll
    for (int i = 0; i < TN; i++)
#pragma unroll
        for (int j = 0; j < TM; j++)
#pragma unroll
            for (int r = 0; r < 16; r++) {
                acc[i][j][r] = 0.0f;
                if constexpr (NACC == 2) acc2[i][j][r] = 0.0f;
            }
    u32x4 fa[2][TM], fb[2][TN];
    auto fetch = [&](int stage, int u, int set) {
        const uint16_t NCHIP_LDS *s = stages + stage * STAGE;
#pragma unroll
        for (int j = 0; j < TM; j++)
            fa[set][j] = fragment(s, std::integral_constant<bool, TA != 0>(), std::integral_constant<int, BM>(), wm * WTM, j, u);
#pragma unroll
        for (int i = 0; i < TN; i++)
            fb[set][i] = fragment(s + BM * 64, std::integral_constant<bool, TB == 0>(), std::integral_constant<int, BN>(), wn * WTN, i, u);
    };
    // the MFMAs of a part (its parity names the fragments' set and the chain), with the loads of a chunk between them
    // where `on`: a load waits its turn at the CU's address unit, and the MFMAs in front of it go on
    // (fp32, whose MFMAs are long, gains 5-8 %; bf16 loses as much by asking later)
    auto multiply = [&](auto parity, auto chunk, auto on) {
        typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
        constexpr int set = decltype(parity)::value & 1, c = decltype(chunk)::value, NM = (F32 ? 4 : 1) * TM * TN;
        constexpr int n = c < NC && NC > 1 ? (c + 1) * NL / NC - c * NL / NC : 0;
        each_constant([&](auto index) {
            constexpr int q = decltype(index)::value, s = q / (TM * TN), i = q % (TM * TN) / TM, j = q % TM;
            if constexpr (F32) {
                acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(__uint_as_float(fb[set][i][s]), __uint_as_float(fa[set][j][s]), acc[i][j], 0, 0, 0);
            } else {
                floatx16 &chain = *(NACC == 2 && set == 1 ? &acc2[NACC == 2 ? i : 0][NACC == 2 ? j : 0] : &acc[i][j]);
                chain = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, fb[set][i]),
                                                                __builtin_bit_cast(bf16x8, fa[set][j]), chain, 0, 0, 0);
            }
            each_constant([&](auto piece) {
                constexpr int x = decltype(piece)::value;
                if constexpr ((x + 1) * NM / (n + 1) == q || ((x + 1) * NM / (n + 1) >= NM && q == NM - 1)) {
                    if (on()) {
                        __builtin_amdgcn_sched_barrier(0);
                        issue(chunk, piece);
                        __builtin_amdgcn_sched_barrier(0);
                    }
                }
            }, std::make_integer_sequence<int, n>());
        }, std::make_integer_sequence<int, NM>());
    };
    // waits until `younger` stages, at most ST - 2, are in flight
    auto arrive = [&](int younger) {
        if (ST > 2 && younger >= ST - 2) { lds_dma_barrier<(ST - 2) * NL>(); return; }
        if (ST > 3 && younger == 1) { lds_dma_barrier<NL>(); return; }
        lds_dma_barrier<0>(); // (from here on: everything)
    };

    // ahead of step it: the stages up to it + ST - 2 and the first chunk of it + ST - 1, whose place
    // step it - 1 has left
    using chunks = std::make_integer_sequence<int, NP>;
    using const0 = std::integral_constant<int, 0>;
    using const1 = std::integral_constant<int, 1>;
    if (nk > 0) { // uniform; an empty k range (a chunk past the end, k = 0) has asked for nothing and adds nothing
#pragma unroll
        for (int s = 0; s < ST - 1; s++)
            if (s < nk) each_constant(issue_chunk, std::make_integer_sequence<int, NC>());
        if (ST - 1 < nk) issue_chunk(const0());
        // (with fewer stages than ST all of them are waited for)
        if (nk >= ST) lds_dma_barrier<(ST - 2) * NL + NL / NC>(); else lds_dma_barrier<0>();
        fetch(0, 0, 0);
        int at = 0; // the stage being read
        auto no = [] { return false; };
        auto body = [&](auto more, int it) {
            constexpr bool steady = decltype(more)::value;
            each_constant([&](auto part) {
                constexpr int u = decltype(part)::value;
                if constexpr (u < NP - 1) {
                    fetch(at, u + 1, (u + 1) & 1);
                    __builtin_amdgcn_sched_barrier(0);
                    multiply(part, std::integral_constant<int, u + 1>(), [&] { return steady || it + ST - 1 < nk; });
                    __builtin_amdgcn_sched_barrier(0);
                }
            }, chunks());
            if constexpr (steady) lds_dma_barrier<(ST - 2) * NL>();
            else arrive(nk - 2 - it);
            at = at + 1 < ST ? at + 1 : 0;
            if (NC == 1 && (steady || it + ST < nk)) issue_chunk(const0());
            fetch(at, 0, 0);
            __builtin_amdgcn_sched_barrier(0);
            multiply(const1(), const0(), [&] { return steady || it + ST < nk; });
            __builtin_amdgcn_sched_barrier(0);
        };
        int it = 0;
        for (; it + ST < nk; it++) body(std::true_type(), it);
        for (; it + 1 < nk; it++) body(std::false_type(), it);
        each_constant([&](auto part) {
            constexpr int u = decltype(part)::value;
            if constexpr (u + 1 < NP) fetch(at, u + 1, (u + 1) & 1);
            multiply(part, const0(), no);
        }, chunks());
        if constexpr (NACC == 2) {
#pragma unroll
            for (int i = 0; i < TN; i++)
#pragma unroll
                for (int j = 0; j < TM; j++)
#pragma unroll
                    for (int r = 0; r < 16; r++) acc[i][j][r] += acc2[i][j][r];
        }
    }

    // Epilogue.  Every 32 x 32 accumulator tile passes through a corner of LDS (the stages are dead)
    // so that a lane holds four consecutive rows m of columns nl, nl + 8, nl + 16, nl + 24 and moves
    // them 16 bytes at a time, and what the next tile reads is on its way while this one is
    // finished: a tile that loads, computes and stores alone is a memory round trip of its own.  Two k
    // groups add their sums (group 0's first) on the way and finish half of the columns each.
    lds_dma_barrier<0>();
    float NCHIP_LDS *const box = (float NCHIP_LDS *)stages + wave * (32 * BOX_LD), *const box0 = (float NCHIP_LDS *)stages + wave % NG * (32 * BOX_LD);
    const int ml = (lane & 7) * 4, nl = lane >> 3;
    const bool full = (m0 + BM <= g.M) && (n0 + BN <= g.N); // uniform
    const bool wide = ((g.M | g.ldc) & 3) == 0 && (((uintptr_t)g.C | (uintptr_t)g.pre | (uintptr_t)g.add | (uintptr_t)g.dpre | (uintptr_t)g.bias | (uintptr_t)g.rowsum | (uintptr_t)(2 * (uintptr_t)g.c16)) & 15) == 0;
    // what a tile reads besides its accumulators: beta C or the addend (never both), else the
    // pre-activation (with an addend that one is read where it is used)
    const float *const first = g.beta != 0.0f ? g.C : g.add, *const operand = first ? first : g.dpre;
    constexpr int NQ = 4 / KW; // 8-column steps a wavefront finishes
    floatx4 next[NQ], bias_next;
    auto load4 = [&](const float *p, int64_t at, int left) -> floatx4 { // left: rows of the matrix from here on
        floatx4 v = { 0.0f, 0.0f, 0.0f, 0.0f };
        if (left <= 0) return v;
        if (wide) return *reinterpret_cast<const floatx4 NCHIP_GLOBAL *>(as_global(p) + at);
#pragma unroll
        for (int e = 0; e < 4; e++) v[e] = e < left ? as_global(p)[at + e] : 0.0f;
        return v;
    };
    auto store4 = [&](float *p, int64_t at, int left, const floatx4 &v) {
        if (wide) { *reinterpret_cast<floatx4 NCHIP_GLOBAL *>(as_global(p) + at) = v; return; }
#pragma unroll
        for (int e = 0; e < 4; e++)
            if (e < left) as_global(p)[at + e] = v[e];
    };
    auto ask = [&](int tile) {
        const int m = m0 + wm * WTM + tile % TM * 32 + ml, nb = n0 + wn * WTN + tile / TM * 32 + nl + kg * NQ * 8;
        if (g.bias) bias_next = load4(g.bias, m, g.M - m);
        if (operand) {
#pragma unroll
            for (int q = 0; q < NQ; q++) next[q] = load4(operand, (int64_t)(nb + 8 * q) * g.ldc + m, full || nb + 8 * q < g.N ? g.M - m : 0);
        }
    };
    bias_next = floatx4{ 0.0f, 0.0f, 0.0f, 0.0f };
#pragma unroll
    for (int q = 0; q < NQ; q++) next[q] = bias_next;
    ask(0);
#pragma unroll 1
    for (int tile = 0; tile < TM * TN; tile++) { // (one copy of this code: unrolled it would not fit the instruction cache)
        each_constant([&](auto index) {
            constexpr int t0 = decltype(index)::value;
            if (tile == t0) {
#pragma unroll
                for (int r = 0; r < 16; r++) box[((r >> 2) * 8 + (r & 3) + hi * 4) * BOX_LD + (lane & 31)] = acc[t0 / TM][t0 % TM][r];
            }
        }, std::make_integer_sequence<int, TM * TN>());
        if constexpr (KW == 2) __syncthreads(); else __builtin_amdgcn_wave_barrier();
        floatx4 x[NQ], y[NQ];
        const floatx4 bv = bias_next;
#pragma unroll
        for (int q = 0; q < NQ; q++) {
            const float NCHIP_LDS *from = box + (nl + 8 * q) * BOX_LD + ml;
            if constexpr (KW == 2) {
                from = box0 + (nl + 8 * (q + kg * NQ)) * BOX_LD + ml;
                x[q] = *reinterpret_cast<const floatx4 NCHIP_LDS *>(from) + *reinterpret_cast<const floatx4 NCHIP_LDS *>(from + NG * (32 * BOX_LD));
            } else {
                x[q] = *reinterpret_cast<const floatx4 NCHIP_LDS *>(from);
            }
            y[q] = next[q];
        }
        __builtin_amdgcn_wave_barrier();
        if (tile + 1 < TM * TN) ask(tile + 1);
        const int m = m0 + wm * WTM + tile % TM * 32 + ml, nb = n0 + wn * WTN + tile / TM * 32 + nl + kg * NQ * 8;
        int left[NQ];
        const int64_t at0 = (int64_t)nb * g.ldc + m;
        auto at = [&](int q) { return at0 + 8 * q * g.ldc; };
#pragma unroll
        for (int q = 0; q < NQ; q++) {
            left[q] = full || nb + 8 * q < g.N ? g.M - m : 0;
#pragma unroll
            for (int e = 0; e < 4; e++) {
                x[q][e] = g.alpha * x[q][e];
                if (g.beta != 0.0f) x[q][e] += g.beta * y[q][e];
                x[q][e] += bv[e];
            }
        }
        if (g.pre) {
#pragma unroll
            for (int q = 0; q < NQ; q++)
                if (left[q] > 0) store4(g.pre, at(q), left[q], x[q]);
        }
        if (g.act == (F32 ? NCHIP_ACT_GELU : ACT_GELU_FAST)) {
#pragma unroll
            for (int q = 0; q < NQ; q++)
#pragma unroll
                for (int e = 0; e < 4; e++) x[q][e] = F32 ? nchip_gelu(x[q][e]) : nchip_gelu_fast(x[q][e]);
        } else if (g.act == NCHIP_ACT_RELU) {
#pragma unroll
            for (int q = 0; q < NQ; q++)
#pragma unroll
                for (int e = 0; e < 4; e++) x[q][e] = x[q][e] > 0.0f ? x[q][e] : 0.0f;
        }
        if (g.add) {
#pragma unroll
            for (int q = 0; q < NQ; q++)
#pragma unroll
                for (int e = 0; e < 4; e++) x[q][e] += y[q][e];
        }
        if (g.dpre) { // gradient through an activation: times act'(pre-activation)
            if (first) {
#pragma unroll
                for (int q = 0; q < NQ; q++) y[q] = load4(g.dpre, at(q), left[q]);
            }
            if (g.dact == (F32 ? NCHIP_ACT_GELU : ACT_GELU_FAST)) {
#pragma unroll
                for (int q = 0; q < NQ; q++)
#pragma unroll
                    for (int e = 0; e < 4; e++) x[q][e] *= F32 ? nchip_gelu_grad(y[q][e]) : nchip_gelu_grad_fast(y[q][e]);
            } else if (g.dact == NCHIP_ACT_RELU) {
#pragma unroll
                for (int q = 0; q < NQ; q++)
#pragma unroll
                    for (int e = 0; e < 4; e++) x[q][e] *= y[q][e] > 0.0f ? 1.0f : 0.0f;
            }
        }
#pragma unroll
        for (int q = 0; q < NQ; q++)
            if (left[q] > 0) store4(g.C, at(q), left[q], x[q]);
        if (g.c16) {
#pragma unroll
            for (int q = 0; q < NQ; q++) {
                uint16_t NCHIP_GLOBAL *h = as_global(g.c16) + at(q);
                if (wide && left[q] > 0) {
                    *reinterpret_cast<uint2 NCHIP_GLOBAL *>(h) = make_uint2(pack_bf16(x[q][0], x[q][1]), pack_bf16(x[q][2], x[q][3]));
                } else {
#pragma unroll
                    for (int e = 0; e < 4; e++)
                        if (e < left[q]) h[e] = f32_to_bf16_rne(x[q][e]);
                }
            }
        }
        if (g.rowsum) { // one partial row per wavefront and half of its columns (n % 8 below 4, from 4 on)
            floatx4 sum = { 0.0f, 0.0f, 0.0f, 0.0f };
#pragma unroll
            for (int q = 0; q < NQ; q++)
#pragma unroll
                for (int e = 0; e < 4; e++) sum[e] += left[q] > 0 ? x[q][e] : 0.0f;
#pragma unroll
            for (int e = 0; e < 4; e++) {
                sum[e] += __shfl_xor(sum[e], 8, 64);
                sum[e] += __shfl_xor(sum[e], 16, 64);
            }
            if ((lane & 24) == 0 && m < g.M)
                store4(g.rowsum, (int64_t)((((tile_n * WN + wn) * TN + tile / TM) * 2 + hi) * KW + kg) * g.M + m, g.M - m, sum);
        }
    }
}

// KW = 2 doubles the wavefronts of a workgroup without shrinking its tile: the
// two groups of WM x WN wavefronts share the LDS tiles and split every 32-deep
// k slab, group 0 taking k%32 < 16 and group 1 the rest; group 1 hands its
// accumulators over through LDS at the end (C = chain0 + chain1, fixed order).
// NACC = 2 (the width-invariant class): each k group keeps two accumulator sets and gives
// the first four MFMA steps of every 32-deep slab to one, the last four to the other, so a
// product is four chains - chain c takes k%32 in [8c, 8c+8) - summed as (c0 + c1) + (c2 + c3).
// The products are the same; the order of the additions is what a kernel with four
// wavefronts per row tile can reproduce (gemm_skinny_nn).
template <int BM, int BN, int BK, int WM, int WN, int TA, int TB, int BF16, int KW = 1, int PF = 2, int NACC = 1, int FRAG = 0>
__global__ __launch_bounds__(64 * WM * WN * KW) void gemm_kernel(GemmArgs g0)
{
    GemmArgs g = g0;
    static_assert(NACC == 1 || (NACC == 2 && BF16 == 0 && KW == 2 && BK == 32), "two accumulator sets: fp32 64-wide class only");
    static_assert(KW == 1 || (KW == 2 && BK % 32 == 0), "k groups split 32-deep slabs");
    constexpr int NT = 64 * WM * WN * KW;                 // threads: KW groups of WM x WN wavefronts
    constexpr int TM = BM / (32 * WM), TN = BN / (32 * WN); // 32x32 MFMA tiles per wavefront
    constexpr int WTM = BM / WM, WTN = BN / WN;           // wavefront tile
    // fp32 row strides of the LDS tiles (see TileLoader)
    constexpr int RSA = BM + (TA ? FPAD_K : PAD), RSB = BN + (TB ? PAD : FPAD_K);
    constexpr int LDS_A = BF16 ? (BK / 2) * (BM + PAD) : BK * RSA; // in 32-bit words
    constexpr int LDS_B = BF16 ? (BK / 2) * (BN + PAD) : BK * RSB;
    static_assert(KW == 1 || BM * BN <= 2 * (LDS_A + LDS_B), "accumulator hand-over must fit in the tile buffers");
    // tile buffers above the 64 KiB a static array may take come from the
    // launch's dynamic allocation instead
    constexpr bool BIG_LDS = 2 * (LDS_A + LDS_B) * 4 > 65536;
    __shared__ __attribute__((aligned(16))) float smem_static[BIG_LDS ? 4 : 2 * (LDS_A + LDS_B)];
    extern __shared__ __attribute__((aligned(16))) float smem_dynamic[];
    float *const smem = BIG_LDS ? smem_dynamic : smem_static;

    const int t = threadIdx.x, lane = t & 63;
    const int kg = (t >> 6) / (WM * WN), wave = (t >> 6) % (WM * WN);
    const int wm = wave % WM, wn = wave / WM;

    int tile_m, tile_n;
    // second k range of a grouped problem: k tiles from k1 on read A2 / B2
    const float *A2, *B2;
    int k1;
    find_tile<BM, BN>(g, tile_m, tile_n, A2, B2, k1);
    const int bz = blockIdx.y;
    const int b = bz / g.ksplit, kz = bz % g.ksplit;
    const int m0 = tile_m * BM, n0 = tile_n * BN;
    const int kbeg = kz * g.kchunk;
    const int kend = min(g.K, kbeg + g.kchunk);

    const int b_out = b / g.batch_in, b_in = b % g.batch_in;
    const float *A = g.A + (int64_t)b_out * g.sa + (int64_t)b_in * g.sa_in;
    const float *B = g.B + (int64_t)b_out * g.sb + (int64_t)b_in * g.sb_in;

    // Stages of BK k: nk1 of the first k range, then those of the second; only a range's last stage
    // may be partial.  The first whole_stages() of a range need no guards: loads of 16 bytes at any
    // 4-byte alignment, from row / column imax - 1 at the latest (what lies past the edge lands in
    // results that are not stored).  With the long axis contiguous such a load runs past the edge by up
    // to 3 values, into the next k: the stage with the range's last k is then left to the guarded loads.
    // Guarding every value of partial or unaligned tiles made a stage a serial chain of memory round trips
    // (3.8 us); 777 x 481 x 352 in the 64x64 class 19.8 -> 16.1 us.
    const bool two = g.grp && A2; // uniform
    const int end1 = two ? k1 : kend, end2 = kend - k1; // where the ranges end (the second counts from 0)
    const int nk1 = (end1 - kbeg + BK - 1) / BK, nk = nk1 + (two ? (end2 + BK - 1) / BK : 0);
    auto whole_stages = [&](int len) {
        const int la_len = (TA || m0 + BM <= g.M) ? len : len - (g.lda >= 3 ? 1 : 3);
        const int lb_len = (!TB || n0 + BN <= g.N) ? len : len - (g.ldb >= 3 ? 1 : 3);
        const int l = min(la_len, lb_len);
        return l > 0 ? l / BK : 0;
    };
    const int whole1 = whole_stages(end1 - kbeg), whole2 = two ? nk1 + whole_stages(end2) : 0;

    // PF register sets: while tile it is computed, tiles it+1 .. it+PF are landing
    // or in flight, so a load has PF compute phases to arrive.  Two sets are
    // enough for the wide classes; the 64x64 class, whose tiles are consumed in
    // half the time, keeps four.
    using LoaderA = std::conditional_t<BF16 == 1, TileLoaderBf16<BM, BK, TA ? 0 : 1, NT>, TileLoader<BM, BK, TA ? 0 : 1, NT>>;
    using LoaderB = std::conditional_t<BF16 == 1, TileLoaderBf16<BN, BK, TB ? 1 : 0, NT>, TileLoader<BN, BK, TB ? 1 : 0, NT>>;
    LoaderA la[PF];
    LoaderB lb[PF];

    floatx16 acc[TN][TM], acc2[TN][TM]; // acc2: second chain of a k group (NACC = 2)
#pragma unroll
    for (int i = 0; i < TN; i++)
#pragma unroll
        for (int j = 0; j < TM; j++)
#pragma unroll
            for (int r = 0; r < 16; r++)
                acc[i][j][r] = acc2[i][j][r] = 0.0f;

    // One pipeline step: write the register set holding tile `it` to LDS buffer
    // it&1, barrier, refill that set with tile it+PF (when there is one), then
    // the MFMAs of tile `it`.  One barrier per tile is enough because a buffer
    // is rewritten only two tiles later.  The steady-state loop carries no
    // guarded-load code: the guarded path shares registers with the vector
    // loads and the compiler then serialises every prefetch behind an
    // s_waitcnt vmcnt(0).
    // the MFMAs of the tile held in LDS at sa / sb
    auto compute = [&](const float *sa, const float *sb) {
        if constexpr (BF16 != 0) {
            // one 32x32x16 MFMA per tile pair per 16 k; group kg takes every KW-th block
            const uint32_t *wa = reinterpret_cast<const uint32_t *>(sa) + (lane >> 5) * 4 * (BM + PAD) + wm * WTM + (lane & 31);
            const uint32_t *wb = reinterpret_cast<const uint32_t *>(sb) + (lane >> 5) * 4 * (BN + PAD) + wn * WTN + (lane & 31);
#pragma unroll
            for (int u = 0; u < BK / 16 / KW; u++) {
                const int row0 = (u * KW + kg) * 8; // word row of this 16-k block
                u32x4 fa[TM], fb[TN];
#pragma unroll
                for (int j = 0; j < TM; j++) {
                    const uint32_t *q = wa + row0 * (BM + PAD) + j * 32;
                    fa[j] = u32x4{ q[0], q[BM + PAD], q[2 * (BM + PAD)], q[3 * (BM + PAD)] };
                }
#pragma unroll
                for (int i = 0; i < TN; i++) {
                    const uint32_t *q = wb + row0 * (BN + PAD) + i * 32;
                    fb[i] = u32x4{ q[0], q[BN + PAD], q[2 * (BN + PAD)], q[3 * (BN + PAD)] };
                }
#pragma unroll
                for (int i = 0; i < TN; i++)
#pragma unroll
                    for (int j = 0; j < TM; j++)
                        acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
                            __builtin_bit_cast(__attribute__((ext_vector_type(8))) __bf16, fb[i]),
                            __builtin_bit_cast(__attribute__((ext_vector_type(8))) __bf16, fa[j]),
                            acc[i][j], 0, 0, 0);
            }
        } else {
            // The k-steps of a tile go in chunks of CH: the fragments of chunk c+1 are read
            // from LDS (into the other half of fa / fb) before the MFMAs of chunk c are issued,
            // and a scheduling fence keeps them there - left alone, the scheduler sinks every
            // read next to its use and each MFMA pair then waits a full LDS round trip.
            // LDS row of step u: 2u (KW = 1), or the u-th pair of this group's half of each
            // 32-deep slab (KW = 2).
            constexpr int NSTEP = BK / 2 / KW;
            auto krow = [](int u) { return KW == 1 ? 2 * u : (u >> 3) * 32 + 2 * (u & 7); };
            constexpr int CH = NSTEP < 4 ? NSTEP : 4, NCH = NSTEP / CH;
            static_assert(NSTEP % CH == 0, "whole chunks");
            float fa[2][CH][TM], fb[2][CH][TN];
            const float *pa = sa + ((lane >> 5) + kg * 16) * RSA + wm * WTM + (lane & 31);
            const float *pb = sb + ((lane >> 5) + kg * 16) * RSB + wn * WTN + (lane & 31);
            // Issue order: with two accumulator sets the steps of the two chains alternate
            // (chain A's step p, chain B's step p, ...), so consecutive MFMAs never depend on
            // each other; each chain still sees its own steps in increasing k order.
            auto stepof = [](int v) { return NACC == 2 ? (v & 1) * 4 + (v >> 1) : v; };
            auto fetch_chunk = [&](int c, int buf) {
#pragma unroll
                for (int u = 0; u < CH; u++) {
#pragma unroll
                    for (int j = 0; j < TM; j++) fa[buf][u][j] = pa[krow(stepof(c * CH + u)) * RSA + j * 32];
#pragma unroll
                    for (int i = 0; i < TN; i++) fb[buf][u][i] = pb[krow(stepof(c * CH + u)) * RSB + i * 32];
                }
            };
            if constexpr (FRAG == 1) {
                // rolling window instead of chunks: the fragments of step u+3 are read while
                // the MFMAs of step u run, and the scheduler is left to place them (wavefronts
                // that own two or more accumulator tiles have enough MFMA time per step)
                static_assert(NACC == 1, "the rolling window feeds one accumulator set");
                constexpr int FD = NSTEP < 4 ? NSTEP : 4;
                float ga[FD][TM], gb[FD][TN];
#pragma unroll
                for (int u = 0; u < FD - 1; u++) {
#pragma unroll
                    for (int j = 0; j < TM; j++) ga[u][j] = pa[krow(u) * RSA + j * 32];
#pragma unroll
                    for (int i = 0; i < TN; i++) gb[u][i] = pb[krow(u) * RSB + i * 32];
                }
#pragma unroll
                for (int u = 0; u < NSTEP; u++) {
                    const int cur = u % FD, nxt = (u + FD - 1) % FD;
                    if (u + FD - 1 < NSTEP) {
#pragma unroll
                        for (int j = 0; j < TM; j++) ga[nxt][j] = pa[krow(u + FD - 1) * RSA + j * 32];
#pragma unroll
                        for (int i = 0; i < TN; i++) gb[nxt][i] = pb[krow(u + FD - 1) * RSB + i * 32];
                    }
#pragma unroll
                    for (int i = 0; i < TN; i++)
#pragma unroll
                        for (int j = 0; j < TM; j++)
                            acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(gb[cur][i], ga[cur][j], acc[i][j], 0, 0, 0);
                }
                return;
            }
            fetch_chunk(0, 0);
#pragma unroll
            for (int c = 0; c < NCH; c++) {
                if (c + 1 < NCH) fetch_chunk(c + 1, (c + 1) & 1);
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int u = 0; u < CH; u++)
#pragma unroll
                    for (int i = 0; i < TN; i++)
#pragma unroll
                        for (int j = 0; j < TM; j++) {
                            if (NACC == 2 && stepof(c * CH + u) >= 4) // steps 4..7 of the slab: the group's second chain
                                acc2[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(fb[c & 1][u][i], fa[c & 1][u][j], acc2[i][j], 0, 0, 0);
                            else
                                acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(fb[c & 1][u][i], fa[c & 1][u][j], acc[i][j], 0, 0, 0);
                        }
                __builtin_amdgcn_sched_barrier(0);
            }
        }
    };

    // stage s without guards, from a range whose stage s starts at k = k0 + s BK
    auto load_whole = [&](const float *As, const float *Bs, int k0, int s, auto &la, auto &lb) {
        la.load(As, g.lda, m0, k0 + s * BK, g.M, 0, true, t);
        lb.load(Bs, g.ldb, n0, k0 + s * BK, g.N, 0, true, t);
    };
    auto load = [&](int s, auto &la, auto &lb) {
        const bool second = s >= nk1, whole = s < (second ? whole2 : whole1); // uniform
        const int k0 = second ? (s - nk1) * BK : kbeg + s * BK, ke = second ? end2 : end1;
        la.load(second ? A2 : A, g.lda, m0, k0, g.M, ke, whole, t);
        lb.load(second ? B2 : B, g.ldb, n0, k0, g.N, ke, whole, t);
    };
    auto step = [&](int it, auto next, auto &la, auto &lb) {
        float *sa = smem + (it & 1) * (LDS_A + LDS_B);
        float *sb = sa + LDS_A;
        if constexpr (BF16 != 0) {
            la.store(reinterpret_cast<uint32_t *>(sa), t);
            lb.store(reinterpret_cast<uint32_t *>(sb), t);
        } else {
            la.store_f32(sa, t);
            lb.store_f32(sb, t);
        }
        __syncthreads();
        next(it + PF, la, lb);
        // keep the prefetch ahead of the MFMAs: without this fence the
        // scheduler sinks the global loads below the compute block and their
        // latency is paid in full at the next LDS write
        __builtin_amdgcn_sched_barrier(0);
        compute(sa, sb);
    };

#ifdef NCHIP_GEMM_CLOCKS
    long long dbg_c0 = clock64(), dbg_w0 = wall_clock64();
#endif
    int it = 0;
    // The first PF stages are fetched by the same straight-line vector loads as inside the steady
    // loop: the compiler then sees one and the same sequence of outstanding loads on entry and on
    // the back edge and waits for the oldest register set only (s_waitcnt vmcnt(n)) instead of for
    // everything in flight.
    if (2 * PF <= whole1) {
#pragma unroll
        for (int j = 0; j < PF; j++) {
            load_whole(A, B, kbeg, j, la[j], lb[j]);
            __builtin_amdgcn_sched_barrier(0); // oldest tile first, as on the back edge
        }
    } else {
#pragma unroll
        for (int j = 0; j < PF; j++)
            if (j < nk) load(j, la[j], lb[j]);
        wait_for_loads();
    }
    for (;;) {
        // steady state: the stages asked for, it + PF .. it + 2 PF - 1, are whole ones of one range
        const bool second = it + PF >= nk1; // uniform
        const float *As = second ? A2 : A, *Bs = second ? B2 : B;
        const int k0 = second ? -nk1 * BK : kbeg, last = (second ? whole2 : whole1) - 2 * PF;
        for (; it <= last; it += PF) {
#pragma unroll
            for (int j = 0; j < PF; j++)
                step(it + j, [&](int s, auto &la, auto &lb) { load_whole(As, Bs, k0, s, la, lb); }, la[j], lb[j]);
        }
        if (it >= nk) break;
        // around a range's end
#pragma unroll
        for (int j = 0; j < PF; j++)
            if (it + j < nk) step(it + j, [&](int s, auto &la, auto &lb) { if (s < nk) load(s, la, lb); }, la[j], lb[j]);
        it += PF;
        if (it >= nk) break;
        wait_for_loads(); // (the steady loop's waits then count its own loads only)
    }

#ifdef NCHIP_GEMM_CLOCKS
    if (g_gemm_clk && blockIdx.y == 0 && t == 0) {
        if (blockIdx.x == 0) {
            g_gemm_clk[0] = clock64() - dbg_c0;       // shader cycles of the k loop
            g_gemm_clk[1] = wall_clock64() - dbg_w0;  // 100 MHz ticks of the same span
        }
        g_gemm_clk[4 + 3 * blockIdx.x] = dbg_w0;          // per workgroup: start,
        g_gemm_clk[5 + 3 * blockIdx.x] = wall_clock64();  // end of the k loop
    }
#endif
    if constexpr (NACC == 2) {
        static_assert(NACC == 1 || (BK / 2 / KW == 8), "chunks of four steps: one chunk per chain");
#pragma unroll
        for (int i = 0; i < TN; i++)
#pragma unroll
            for (int j = 0; j < TM; j++)
#pragma unroll
                for (int r = 0; r < 16; r++) acc[i][j][r] += acc2[i][j][r];
    }
    if (KW == 2) {
        // group 1 parks its accumulators in LDS (the tiles are dead), group 0 adds them
        __syncthreads();
        float *red = smem + (size_t)wave * (TN * TM * 16 * 64) + lane;
        if (kg == 1) {
#pragma unroll
            for (int i = 0; i < TN; i++)
#pragma unroll
                for (int j = 0; j < TM; j++)
#pragma unroll
                    for (int r = 0; r < 16; r++) red[((i * TM + j) * 16 + r) * 64] = acc[i][j][r];
        }
        __syncthreads();
        if (kg == 1) return;
#pragma unroll
        for (int i = 0; i < TN; i++)
#pragma unroll
            for (int j = 0; j < TM; j++)
#pragma unroll
                for (int r = 0; r < 16; r++) acc[i][j][r] += red[((i * TM + j) * 16 + r) * 64];
    }

    // epilogue.  acc[i][j][r] is C[m][n] with
    //   m = m0 + wm*BM/2 + j*32 + lane%32
    //   n = n0 + wn*BN/2 + i*32 + (r/4)*8 + (lane/32)*4 + r%4
    const int mm_base = m0 + wm * WTM + (lane & 31);
    const int nn_base = n0 + wn * WTN + (lane >> 5) * 4;
    if (g.ksplit > 1) {
        float NCHIP_GLOBAL *ws = as_global(g.ws + ((int64_t)(kz * g.batch + b)) * g.M * g.N);
#pragma unroll
        for (int i = 0; i < TN; i++)
#pragma unroll
            for (int j = 0; j < TM; j++) {
                int m = mm_base + j * 32;
                if (m >= g.M) continue;
#pragma unroll
                for (int r = 0; r < 16; r++) {
                    int n = nn_base + i * 32 + (r >> 2) * 8 + (r & 3);
                    if (n < g.N)
                        ws[(int64_t)n * g.M + m] = acc[i][j][r];
                }
            }
        return;
    }
    const int64_t coff = (int64_t)b_out * g.sc + (int64_t)b_in * g.sc_in;
    float NCHIP_GLOBAL *C = as_global(g.C + coff);
    float NCHIP_GLOBAL *P = g.pre ? as_global(g.pre + coff) : nullptr;
    const float NCHIP_GLOBAL *Radd = g.add ? as_global(g.add + coff) : nullptr;
    const bool full = (m0 + BM <= g.M) && (n0 + BN <= g.N); // uniform
    const float NCHIP_GLOBAL *Dp = g.dpre ? as_global(g.dpre + coff) : nullptr;
    const bool plain = !g.bias && !P && !Radd && !Dp && g.beta == 0.0f && g.act == NCHIP_ACT_NONE;
#pragma unroll
    for (int i = 0; i < TN; i++)
#pragma unroll
        for (int j = 0; j < TM; j++) {
            float NCHIP_GLOBAL *rs = nullptr;
            if (g.rowsum) // partial row of this (tile column, wavefront column, accumulator column, lane half)
                rs = as_global(g.rowsum) + (int64_t)((((tile_n * WN + wn) * TN + i) * 2) + (lane >> 5)) * g.M;
            epilogue_tile(g, acc[i][j], mm_base + j * 32, nn_base + i * 32, C, P, Radd, Dp, full, plain, rs);
        }
#ifdef NCHIP_GEMM_CLOCKS
    if (g_gemm_clk && blockIdx.y == 0 && t == 0) g_gemm_clk[6 + 3 * blockIdx.x] = wall_clock64(); // stores issued
#endif
}

// Small fp32 products: a 16 x 16 tile of C per workgroup and batch entry, with the bits of the
// 64x64x32 class (KW = 2) that the shape would otherwise take.  That class gives every element
// two chains per k chunk - chain 0 the first 16 k of each 32-deep slab, chain 1 the rest - and
// with split-K adds the chunks' (chain 0 + chain 1) in order; a wavefront here is one such chain,
// issued as v_mfma_f32_16x16x4_f32, which accumulates its four k in increasing order like the
// 32x32x2 form its two.  No operand is shared between tiles, which is what the tile kernel's LDS
// stages are for: when the output has fewer 64 x 64 tiles than a chip fills, those stages are a
// serial chain of memory round trips; here a wavefront holds PF blocks of 16 k of both operands in
// registers, so that one round trip covers K = 32 PF (per chunk, with SPLIT: 2 g.ksplit chains,
// NW of them at a time).
// VA / VB: the operand is contiguous along k (K at least 4), and a lane reads four k at once, at any
// 4-byte alignment.  It then holds k = 4 (lane / 16) + s where the matrix instruction wants
// k = 4 s + lane / 16: transpose_k4 exchanges the four 16-lane rows, four swaps for 16 k.
__device__ __forceinline__ void transpose_k4(floatx4 &v)
{
    uint32_t r[4];
#pragma unroll
    for (int s = 0; s < 4; s++) r[s] = __float_as_uint(v[s]);
#pragma unroll
    for (int s = 0; s < 2; s++) { // upper 32 lanes of r[s] against lower 32 of r[s + 2]
        const auto x = __builtin_amdgcn_permlane32_swap(r[s], r[s + 2], false, false);
        r[s] = x[0]; r[s + 2] = x[1];
    }
#pragma unroll
    for (int s = 0; s < 4; s += 2) { // odd 16-lane rows of r[s] against even ones of r[s + 1]
        const auto x = __builtin_amdgcn_permlane16_swap(r[s], r[s + 1], false, false);
        r[s] = x[0]; r[s + 1] = x[1];
    }
#pragma unroll
    for (int s = 0; s < 4; s++) v[s] = __uint_as_float(r[s]);
}

constexpr int SMALL_KSPLIT = 16; // nchip_gemm_pick_ksplit's limit

template <int NW, int PF, int VA, int VB, int SPLIT>
__global__ __launch_bounds__(64 * NW) void gemm_small_kernel(GemmArgs g, int64_t am, int64_t ak, int64_t bn, int64_t bk)
{
    __shared__ float red[SPLIT ? 2 * SMALL_KSPLIT : 2][256];
    // (w in a scalar register: the branches around the matrix instructions, which ignore the
    // execution mask, have to be scalar ones)
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), il = lane & 15, kq = lane >> 4;
    const int m0 = blockIdx.x * 16, n0 = blockIdx.y * 16, bo = blockIdx.z / g.batch_in, bi = blockIdx.z % g.batch_in;
    // (am, ak / bn, bk: strides of A along m and k, of B along n and k; byte offsets from the tile's
    // first row fit 32 bits, so an address is a scalar base and one register)
    const char NCHIP_GLOBAL *A0 = (const char NCHIP_GLOBAL *)(as_global(g.A) + bo * g.sa + bi * g.sa_in + m0 * am);
    const char NCHIP_GLOBAL *B0 = (const char NCHIP_GLOBAL *)(as_global(g.B) + bo * g.sb + bi * g.sb_in + n0 * bn);
    const uint32_t ma = 4 * (uint32_t)(m0 + il < g.M ? il : g.M - 1 - m0) * (uint32_t)am, ka = 4 * (uint32_t)ak;
    const uint32_t nb = 4 * (uint32_t)(n0 + il < g.N ? il : g.N - 1 - n0) * (uint32_t)bn, kb = 4 * (uint32_t)bk;
    const int K = g.K, chains = SPLIT ? 2 * g.ksplit : 2;
    // 16 k from k0 on.  A block that passes the end reads clamped addresses, so that every block
    // issues the same loads; keep() clears what lies past it
    const uint32_t aoff = ma + (VA ? 16 : ka) * kq, boff = nb + (VB ? 16 : kb) * kq; // this lane's first k of a block
    auto fetch = [&](floatx4 &v, const char NCHIP_GLOBAL *p, uint32_t row, uint32_t off, uint32_t step, int k0, auto vec) {
        constexpr bool V = decltype(vec)::value;
        if (k0 + 16 <= K) { // uniform
            const char NCHIP_GLOBAL *q = p + (V ? 4 : step) * (uint32_t)k0;
            if constexpr (V) {
                v = *reinterpret_cast<const floatx4_u NCHIP_GLOBAL *>(q + off);
            } else {
#pragma unroll
                for (int s = 0; s < 4; s++) v[s] = *reinterpret_cast<const float NCHIP_GLOBAL *>(q + s * 4 * step + off);
            }
        } else if constexpr (V) {
            const int k = k0 + 4 * kq;
            v = *reinterpret_cast<const floatx4_u NCHIP_GLOBAL *>(p + (row + 4 * (uint32_t)(k < K - 4 ? k : K - 4)));
        } else {
#pragma unroll
            for (int s = 0; s < 4; s++) {
                const int k = k0 + 4 * s + kq;
                v[s] = *reinterpret_cast<const float NCHIP_GLOBAL *>(p + (row + step * (uint32_t)(k < K ? k : K - 1)));
            }
        }
    };
    auto keep = [&](floatx4 &v, int k0, int kend, auto vec) {
        if constexpr (decltype(vec)::value) {
            if (k0 + 16 > kend) { // v was read from K - 4 where four k from k on pass the end: d of them are to go
                const int k = k0 + 4 * kq, d = k < K - 4 ? 0 : k - (K - 4);
                v = d & 1 ? floatx4{ v[1], v[2], v[3], 0.0f } : v;
                v = d & 2 ? floatx4{ v[2], v[3], 0.0f, 0.0f } : v;
                v = d > 3 ? floatx4{ 0.0f, 0.0f, 0.0f, 0.0f } : v;
            }
            transpose_k4(v);
        } else if (k0 + 16 > kend) {
#pragma unroll
            for (int s = 0; s < 4; s++) v[s] = k0 + 4 * s + kq < kend ? v[s] : 0.0f;
        }
    };
    // this thread's elements of the tile, and what the epilogue reads for them: fetched before the
    // operands, it costs no round trip of its own at the end
    constexpr int NE = NW >= 4 ? 1 : 4 / NW;
    bool ok[NE];
    int64_t off[NE];
    float extra[NE], prev[NE], bv[NE];
#pragma unroll
    for (int i = 0; i < NE; i++) {
        const int e = threadIdx.x + i * 64 * NW, tm = m0 + (e & 15), tn = n0 + (e >> 4);
        ok[i] = e < 256 && tm < g.M && tn < g.N;
        off[i] = bo * g.sc + bi * g.sc_in + (int64_t)tn * g.ldc + tm;
        extra[i] = g.add && ok[i] ? as_global(g.add)[off[i]] : 0.0f;
        prev[i] = g.beta != 0.0f && ok[i] ? as_global(g.C)[off[i]] : 0.0f;
        bv[i] = g.bias && ok[i] ? as_global(g.bias)[tm] : 0.0f;
    }
    for (int c = w; c < chains; c += NW) {
        const int kbeg = (c >> 1) * g.kchunk, kend = kbeg + g.kchunk < K ? kbeg + g.kchunk : K;
        floatx4 acc = { 0.0f, 0.0f, 0.0f, 0.0f };
        for (int k0 = kbeg + 16 * (c & 1); k0 < kend; k0 += 32 * PF) {
            floatx4 a[PF], b[PF];
#pragma unroll
            for (int p = 0; p < PF; p++) {
                fetch(b[p], B0, nb, boff, kb, k0 + 32 * p, std::integral_constant<bool, VB>());
                fetch(a[p], A0, ma, aoff, ka, k0 + 32 * p, std::integral_constant<bool, VA>());
            }
            __builtin_amdgcn_sched_barrier(0); // every load is out before the first is waited for
#pragma unroll
            for (int p = 0; p < PF; p++) {
                if (k0 + 32 * p >= kend) break; // uniform
                keep(b[p], k0 + 32 * p, kend, std::integral_constant<bool, VB>());
                keep(a[p], k0 + 32 * p, kend, std::integral_constant<bool, VA>());
#pragma unroll
                for (int s = 0; s < 4; s++) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(b[p][s], a[p][s], acc, 0, 0, 0);
            }
        }
#pragma unroll
        for (int r = 0; r < 4; r++) red[c][(4 * kq + r) * 16 + il] = acc[r]; // [n][m]
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < NE; i++) {
        if (!ok[i]) continue;
        const int e = threadIdx.x + i * 64 * NW;
        float sum = red[0][e] + red[1][e];
        if (SPLIT)
            for (int z = 1; z < g.ksplit; z++) sum += red[2 * z][e] + red[2 * z + 1][e];
        float v = g.alpha * sum;
        if (g.beta != 0.0f) v += g.beta * prev[i];
        v += bv[i];
        if (g.pre) as_global(g.pre)[off[i]] = v;
        as_global(g.C)[off[i]] = apply_act(v, g.act) + extra[i];
    }
}

// sums the ksplit partial tiles in increasing k order, then the same epilogue
__global__ __launch_bounds__(256) void gemm_splitk_reduce(GemmArgs g)
{
    int64_t total = (int64_t)g.M * g.N;
    int b = blockIdx.y;
    const int64_t coff = (int64_t)(b / g.batch_in) * g.sc + (int64_t)(b % g.batch_in) * g.sc_in;
    float *C = g.C + coff;
    float *P = g.pre ? g.pre + coff : nullptr;
    const float *Radd = g.add ? g.add + coff : nullptr;
    for (int64_t e = (int64_t)blockIdx.x * 256 + threadIdx.x; e < total; e += (int64_t)gridDim.x * 256) {
        int m = (int)(e % g.M);
        int64_t n = e / g.M;
        float s = 0.0f;
        for (int kz = 0; kz < g.ksplit; kz++)
            s += g.ws[((int64_t)(kz * g.batch + b)) * total + e];
        int64_t off = n * g.ldc + m;
        float v = g.alpha * s;
        if (g.beta != 0.0f) v += g.beta * C[off];
        if (g.bias) v += g.bias[m];
        if (P) P[off] = v;
        v = apply_act(v, g.act);
        if (Radd) v += Radd[off];
        if (g.dpre) v *= act_grad(g.dpre[coff + off], g.dact);
        C[off] = v;
    }
}

// Rounds a column-major fp32 matrix (rows x cols, leading dimension ld_src) to
// bf16 (nearest even) in the same layout, padded with zeros to rows_pad x
// cols_pad (rows_pad a multiple of 8 = the leading dimension of the copy).
// One thread per 8 consecutive rows of one column.
__global__ __launch_bounds__(256) void cast_bf16_kernel(const float *src, uint16_t *dst, int rows, int cols,
                                                        int64_t ld_src, int rows_pad, int cols_pad, int vec)
{
    const int units = rows_pad / 8;
    const int64_t total = (int64_t)units * cols_pad;
    for (int64_t e = (int64_t)blockIdx.x * 256 + threadIdx.x; e < total; e += (int64_t)gridDim.x * 256) {
        const int u = (int)(e % units), c = (int)(e / units), r0 = u * 8;
        float f[8];
        if (c < cols && vec && r0 + 8 <= rows) {
            const floatx4 *q = reinterpret_cast<const floatx4 *>(src + (int64_t)c * ld_src + r0);
            floatx4 a = q[0], b = q[1];
            f[0] = a[0]; f[1] = a[1]; f[2] = a[2]; f[3] = a[3];
            f[4] = b[0]; f[5] = b[1]; f[6] = b[2]; f[7] = b[3];
        } else {
#pragma unroll
            for (int j = 0; j < 8; j++)
                f[j] = (c < cols && r0 + j < rows) ? src[(int64_t)c * ld_src + r0 + j] : 0.0f;
        }
        uint4 w = make_uint4(pack_bf16(f[0], f[1]), pack_bf16(f[2], f[3]), pack_bf16(f[4], f[5]), pack_bf16(f[6], f[7]));
        *reinterpret_cast<uint4 *>(dst + (int64_t)c * rows_pad + r0) = w;
    }
}

// dst[i] = bf16(src[i]) for i < n, 8 elements per thread and step (two 16-byte loads, one
// 16-byte store); both pointers 16-byte aligned
__global__ __launch_bounds__(256) void cast_bf16_flat_kernel(const float *src, uint16_t *dst, int64_t n)
{
    const int64_t units = n / 8, stride = (int64_t)gridDim.x * 256;
    const floatx4 NCHIP_GLOBAL *s4 = reinterpret_cast<const floatx4 NCHIP_GLOBAL *>(as_global(src));
    u32x4 NCHIP_GLOBAL *d4 = reinterpret_cast<u32x4 NCHIP_GLOBAL *>(as_global(dst));
    for (int64_t u = (int64_t)blockIdx.x * 256 + threadIdx.x; u < units; u += stride) {
        const floatx4 a = s4[2 * u], b = s4[2 * u + 1];
        d4[u] = u32x4{ pack_bf16(a[0], a[1]), pack_bf16(a[2], a[3]), pack_bf16(b[0], b[1]), pack_bf16(b[2], b[3]) };
    }
    if (blockIdx.x == 0) // the last n % 8 elements
        for (int64_t i = units * 8 + threadIdx.x; i < n; i += 256) as_global(dst)[i] = f32_to_bf16_rne(as_global(src)[i]);
}

// dst[i] = float(bf16 src[i]) for i < n (exact): one streaming pass
__global__ __launch_bounds__(256) void widen_bf16_flat_kernel(const uint16_t *src, float *dst, int64_t n)
{
    const int64_t stride = (int64_t)gridDim.x * 256;
    const uint16_t NCHIP_GLOBAL *s = as_global(src);
    float NCHIP_GLOBAL *d = as_global(dst);
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += stride)
        d[i] = __builtin_bit_cast(float, (uint32_t)s[i] << 16);
}

// ---- optional per-launch timing (HIP events on the launch stream) ----------
struct ProfRec {
    hipEvent_t start, stop;
    int variant;
    double flops;
};
bool g_prof_on = false;
int g_force_cfg = getenv("NCHIP_GEMM_CFG") ? atoi(getenv("NCHIP_GEMM_CFG")) : 0;
int g_skinny = 3; // width-invariant products with <= 64 columns: 3 = the 16x16x4 MFMA kernel, 2 = the vector-ALU kernel, 1 = the 32x32x2 MFMA kernel, 0 = tiles

// chunks of 256 k in flight: as many as the product has, up to 8
static void launch_fewcol_fma(const GemmArgs &g, dim3 grid, hipStream_t st)
{
    const int nch = (g.K + FC_KC - 1) / FC_KC;
    if (nch <= 2) hipLaunchKernelGGL(gemm_fewcol_fma<2>, grid, dim3(256), 0, st, g);
    else if (nch <= 4) hipLaunchKernelGGL(gemm_fewcol_fma<4>, grid, dim3(256), 0, st, g);
    else hipLaunchKernelGGL(gemm_fewcol_fma<8>, grid, dim3(256), 0, st, g);
}

// 16 x 16 tiles; 8 x 8 tiles from K = 1280 on (up to 8 chunks in flight) and, with a k-major A,
// whenever 16 x 16 tiles would leave most CUs without a workgroup (mmax: the taller product
// of the launch, nz: 1 or 2 products, ak: A is k-major)
static void launch_fewcol_mfma(const GemmArgs &g, int mmax, int nz, hipStream_t st, bool ak = false)
{
    const int nch = (g.K + 255) / 256;
    const dim3 grid16(mmax / 16, (g.N + 15) / 16, nz), grid8(mmax / 8, (g.N + 7) / 8, nz);
    const bool small = nch > 4 || (ak && grid16.x * grid16.y * grid16.z < 192);
    if (!ak) {
        if (small) hipLaunchKernelGGL((gemm_fewcol_mfma<8, 0, 8>), grid8, dim3(256), 0, st, g);
        else if (nch <= 2) hipLaunchKernelGGL(gemm_fewcol_mfma<2>, grid16, dim3(256), 0, st, g);
        else hipLaunchKernelGGL(gemm_fewcol_mfma<4>, grid16, dim3(256), 0, st, g);
    } else if (small) {
        if (nch <= 2) hipLaunchKernelGGL((gemm_fewcol_mfma<2, 0, 8, 1>), grid8, dim3(256), 0, st, g);
        else if (nch <= 4) hipLaunchKernelGGL((gemm_fewcol_mfma<4, 0, 8, 1>), grid8, dim3(256), 0, st, g);
        else hipLaunchKernelGGL((gemm_fewcol_mfma<8, 0, 8, 1>), grid8, dim3(256), 0, st, g);
    } else {
        if (nch <= 2) hipLaunchKernelGGL((gemm_fewcol_mfma<2, 0, 16, 1>), grid16, dim3(256), 0, st, g);
        else hipLaunchKernelGGL((gemm_fewcol_mfma<4, 0, 16, 1>), grid16, dim3(256), 0, st, g);
    }
}
int g_force_gm = -1;
std::vector<ProfRec> g_prof;
int g_bf16ops_cls = getenv("NCHIP_GEMM_BF16OPS_CLASS") ? atoi(getenv("NCHIP_GEMM_BF16OPS_CLASS")) : 0;


// With `rec` the kernel's own start / stop timestamps are bound to the record's
// events (hipExtLaunchKernelGGL), so the measured time is the dispatch alone,
// as a kernel trace reports it, without the marker packets of hipEventRecord.
// bytes of the two tile buffer pairs when they exceed what a static array may hold (else 0)
template <int BM, int BN, int BK, int TA, int TB, int BF16>
constexpr size_t lds_dynamic_bytes()
{
    constexpr size_t a = BF16 ? (BK / 2) * (BM + PAD) : BK * (BM + (TA ? FPAD_K : PAD));
    constexpr size_t b = BF16 ? (BK / 2) * (BN + PAD) : BK * (BN + (TB ? PAD : FPAD_K));
    constexpr size_t bytes = 2 * (a + b) * sizeof(float);
    static_assert(bytes <= 160 * 1024, "tile buffers exceed LDS");
    return bytes > 65536 ? bytes : 0;
}

template <int BM, int BN, int BK, int WM, int WN, int BF16, int KW = 1, int PF = 2, int NACC = 1, int FRAG = 0>
void launch_tile(hipStream_t st, int ta, int tb, GemmArgs &g, ProfRec *rec, int grouped_tiles = 0)
{
    g.tiles_m = (g.M + BM - 1) / BM;
    g.tiles_n = (g.N + BN - 1) / BN;
    g.gm = g_force_gm >= 0 ? g_force_gm : 8;
    g.dbg = 0;
    dim3 grid(grouped_tiles ? grouped_tiles : g.tiles_m * g.tiles_n, g.batch * g.ksplit), block(64 * WM * WN * KW);
#define LAUNCH(TA, TB)                                                                                     \
    do {                                                                                                   \
        constexpr size_t dyn = lds_dynamic_bytes<BM, BN, BK, TA, TB, BF16>();                              \
        if (dyn) {                                                                                         \
            static const bool ok = hipFuncSetAttribute(                                                    \
                reinterpret_cast<const void *>(gemm_kernel<BM, BN, BK, WM, WN, TA, TB, BF16, KW, PF, NACC, FRAG>),     \
                hipFuncAttributeMaxDynamicSharedMemorySize, (int)dyn) == hipSuccess;                       \
            if (!ok) { fprintf(stderr, "nchip_gemm: cannot reserve %zu bytes of LDS\n", dyn); abort(); }  \
        }                                                                                                  \
        if (rec) hipExtLaunchKernelGGL((gemm_kernel<BM, BN, BK, WM, WN, TA, TB, BF16, KW, PF, NACC, FRAG>), grid, block, dyn, \
                                       st, rec->start, rec->stop, 0, g);                                   \
        else hipLaunchKernelGGL((gemm_kernel<BM, BN, BK, WM, WN, TA, TB, BF16, KW, PF, NACC, FRAG>), grid, block, dyn, st, g); \
    } while (0)
    if (!ta && !tb) LAUNCH(0, 0);
    else if (ta && !tb) LAUNCH(1, 0);
    else if (!ta && tb) LAUNCH(0, 1);
    else LAUNCH(1, 1);
#undef LAUNCH
}

// (0, or -2 with a message where the stages' LDS is refused)
template <int F32, int BM, int BN, int WM, int WN, int KW, int ST, int NACC = 1, int FAR = 0>
int launch_dma(hipStream_t st, int ta, int tb, GemmArgs &g, ProfRec *rec, int grouped_tiles = 0)
{
    g.tiles_m = (g.M + BM - 1) / BM;
    g.tiles_n = (g.N + BN - 1) / BN;
    g.gm = g_force_gm >= 0 ? g_force_gm : 8;
    constexpr size_t dyn = (size_t)(BM + BN) * 64 * 2 * ST;
    static_assert(dyn <= 160 * 1024, "stages exceed LDS");
    dim3 grid(grouped_tiles ? grouped_tiles : g.tiles_m * g.tiles_n, g.batch * g.ksplit), block(64 * WM * WN * KW);
#define LAUNCH(TA, TB)                                                                                     \
    do {                                                                                                   \
        static const bool ok = hipFuncSetAttribute(                                                        \
            reinterpret_cast<const void *>(gemm_dma_kernel<F32, BM, BN, WM, WN, KW, ST, TA, TB, NACC, FAR>),                    \
            hipFuncAttributeMaxDynamicSharedMemorySize, (int)dyn) == hipSuccess;                           \
        if (!ok) { fprintf(stderr, "nchip_gemm: cannot reserve %zu bytes of LDS\n", dyn); return -2; }    \
        if (rec) hipExtLaunchKernelGGL((gemm_dma_kernel<F32, BM, BN, WM, WN, KW, ST, TA, TB, NACC, FAR>), grid, block, dyn, st, rec->start, rec->stop, 0, g); \
        else hipLaunchKernelGGL((gemm_dma_kernel<F32, BM, BN, WM, WN, KW, ST, TA, TB, NACC, FAR>), grid, block, dyn, st, g);   \
    } while (0)
    if (!ta && !tb) LAUNCH(0, 0);
    else if (ta && !tb) LAUNCH(1, 0);
    else if (!ta && tb) LAUNCH(0, 1);
    else LAUNCH(1, 1);
#undef LAUNCH
    return 0;
}

// The widest leading dimension of bf16 operands whose 256 rows or 64 k of a stage are within 32 bits.
constexpr int64_t DMA_LD = 1 << 23;

// Tile class of a product of bf16 operands, from the tile counts.  One 256 x 256 tile fills a CU
// (128 KB of stages, 256 registers): it is taken when its rounds of 256 workgroups are at least
// seven eighths full; below that two workgroups of 128 x 128 and two stages share a CU as long as
// there are that many; a single round gets 8 wavefronts a tile and four stages; then smaller tiles
// until the chip is covered.  Measured, us (m x n x k; classes 4 / 1 / 5 / 2 / 3; before = tiles
// staged through registers, best class):
//   16384 x 4096 x 1024   155 / 162 / 207 / 197 / 246   before 204
//   4096 x 4096 x 1024     44 /  46 /  59 /  58 /  69   before  56
//   2048 x 4096 x 1024     32 /  24 /  29 /  31 /  36   before  31
//   1024 x 4096 x 4096     96 /  59 /  43 /  53 /  64   before  52
//   1024 x 2048 x 3072     71 /  39 /  30 /  24 /  28   before  33
//   512 x 2048 x 2048      47 /  21 /  19 /  13 /  10   before  13
// (class 6: rows too far apart for 32-bit offsets; two chains: no room for the second accumulators in 256 x 256 tiles, nor twice a CU in classes of 64 x 64 a wavefront)
static int dma_class(const GemmArgs &g, bool two_chains)
{
    const int m = g.M, n = g.N;
    if (g.lda > DMA_LD || g.ldb > DMA_LD) return 6;
    auto tiles = [&](int bm, int bn) { return (int64_t)((m + bm - 1) / bm) * ((n + bn - 1) / bn); };
    const int64_t t256 = tiles(256, 256), t128 = tiles(128, 128);
    if (!two_chains && 8 * t256 >= 7 * 256 * ((t256 + 255) / 256)) return 4;
    if (!two_chains && t128 >= 448) return 1;
    if (t128 >= 224) return 5;
    return tiles(128, 64) >= 224 && m >= 128 ? 2 : 3;
}

static int launch_dma_class(hipStream_t st, int cls, bool two_chains, int ta, int tb, GemmArgs &g, ProfRec *rec)
{
    if (two_chains) {
        if (cls == 6) return launch_dma<0, 64, 64, 2, 2, 1, 4, 2, 1>(st, ta, tb, g, rec);
        if (cls == 1 || cls == 5) return launch_dma<0, 128, 128, 2, 4, 1, 4, 2>(st, ta, tb, g, rec);
        if (cls == 2) return launch_dma<0, 128, 64, 2, 2, 1, 3, 2>(st, ta, tb, g, rec);
        return launch_dma<0, 64, 64, 2, 2, 1, 4, 2>(st, ta, tb, g, rec);
    }
    if (cls == 6) return launch_dma<0, 64, 64, 2, 2, 1, 4, 1, 1>(st, ta, tb, g, rec);
    if (cls == 4) return launch_dma<0, 256, 256, 2, 4, 1, 2>(st, ta, tb, g, rec);
    if (cls == 1) return launch_dma<0, 128, 128, 2, 2, 1, 2>(st, ta, tb, g, rec);
    if (cls == 5) return launch_dma<0, 128, 128, 2, 4, 1, 4>(st, ta, tb, g, rec);
    if (cls == 2) return launch_dma<0, 128, 64, 2, 2, 1, 3>(st, ta, tb, g, rec);
    return launch_dma<0, 64, 64, 2, 2, 1, 4>(st, ta, tb, g, rec);
}

template <int NW, int PF, int SPLIT>
void launch_small(hipStream_t st, int ta, int tb, const GemmArgs &g, ProfRec *rec)
{
    const dim3 grid((g.M + 15) / 16, (g.N + 15) / 16, g.batch), block(64 * NW);
    const bool va = ta && g.K >= 4, vb = !tb && g.K >= 4;
    const int64_t am = ta ? g.lda : 1, ak = ta ? 1 : g.lda, bn = tb ? 1 : g.ldb, bk = tb ? g.ldb : 1;
#define LAUNCH(VA, VB)                                                                                     \
    do {                                                                                                   \
        if (rec) hipExtLaunchKernelGGL((gemm_small_kernel<NW, PF, VA, VB, SPLIT>), grid, block, 0, st, rec->start, rec->stop, 0, g, am, ak, bn, bk); \
        else hipLaunchKernelGGL((gemm_small_kernel<NW, PF, VA, VB, SPLIT>), grid, block, 0, st, g, am, ak, bn, bk); \
    } while (0)
    if (!va && !vb) LAUNCH(0, 0);
    else if (va && !vb) LAUNCH(1, 0);
    else if (!va && vb) LAUNCH(0, 1);
    else LAUNCH(1, 1);
#undef LAUNCH
}

// Device scratch for the bf16 copies of one product's operands, one buffer per
// stream: successive products on a stream reuse it in stream order.  It grows
// on demand and lives until the process ends.
struct CastScratch { hipStream_t st; uint16_t *ptr; size_t cap; };
std::vector<CastScratch> g_cast;
int g_bf16src = getenv("NCHIP_GEMM_BF16SRC") ? atoi(getenv("NCHIP_GEMM_BF16SRC")) : 1;
double g_bf16src_min_flops = getenv("NCHIP_GEMM_BF16SRC_FLOPS") ? atof(getenv("NCHIP_GEMM_BF16SRC_FLOPS")) : 8e9;

uint16_t *cast_scratch(hipStream_t st, size_t elems)
{
    for (CastScratch &c : g_cast)
        if (c.st == st) {
            if (c.cap >= elems) return c.ptr;
            (void)hipStreamSynchronize(st);
            (void)hipFree(c.ptr);
            c.ptr = nullptr; c.cap = 0;
            size_t cap = elems + elems / 4;
            if (hipMalloc((void **)&c.ptr, cap * sizeof(uint16_t)) != hipSuccess) { (void)hipGetLastError(); return nullptr; }
            c.cap = cap;
            return c.ptr;
        }
    CastScratch c = { st, nullptr, 0 };
    if (hipMalloc((void **)&c.ptr, elems * sizeof(uint16_t)) != hipSuccess) { (void)hipGetLastError(); return nullptr; }
    c.cap = elems;
    g_cast.push_back(c);
    return c.ptr;
}

// copy of a column-major rows x cols operand; k_is_rows says which extent is k
// (padded to kpad); returns the leading dimension of the copy
int64_t cast_operand(hipStream_t st, const float *src, int rows, int cols, int64_t ld, bool k_is_rows,
                     int kpad, uint16_t *dst)
{
    const int rows_pad = k_is_rows ? kpad : (rows + 7) / 8 * 8;
    const int cols_pad = k_is_rows ? cols : kpad;
    const int vec = (ld % 4 == 0) && (((uintptr_t)src & 15) == 0);
    int64_t total = (int64_t)(rows_pad / 8) * cols_pad;
    int nb = (int)((total + 255) / 256 < 8192 ? (total + 255) / 256 : 8192);
    hipLaunchKernelGGL(cast_bf16_kernel, dim3(nb), dim3(256), 0, st, src, dst, rows, cols, ld, rows_pad, cols_pad, vec);
    return rows_pad;
}

size_t cast_elems(int rows, int cols, bool k_is_rows, int kpad)
{
    const size_t rows_pad = k_is_rows ? kpad : (rows + 7) / 8 * 8;
    const size_t cols_pad = k_is_rows ? cols : kpad;
    return (rows_pad * cols_pad + 127) / 128 * 128;
}

} // namespace

extern "C" int nchip_gemm_pick_ksplit(int m, int n, int k, int batch)
{
    // Aim at >= 512 workgroups (2 per CU on 256 CUs) when the output is small
    // and the reduction long (the weight-gradient GEMMs: k = tokens).
    int64_t tiles = (int64_t)((m + 63) / 64) * ((n + 63) / 64) * batch;
    if (tiles >= 256 || k < 1024)
        return 1;
    int s = (int)((512 + tiles - 1) / tiles);
    int smax = k / 256;
    if (s > smax) s = smax;
    if (s > 16) s = 16;
    return s < 1 ? 1 : s;
}

// Tile class of an fp32 or bf16-rounding product (nb: batch entries times split-K chunks), from the
// shape alone.  Measured on MI355X (fp32): small outputs want the most workgroups and the most
// wavefronts per workgroup (10: 64x64x32, two k groups of 4 wavefronts, four register sets of
// tiles in flight); once 128x64 tiles still give >= 256 workgroups, 8 wavefronts of 32x32 on a
// 128x64x32 tile win (4); very large problems use 128x128x32 with 8 wavefronts (7).
static int gemm_class(int m, int n, int64_t nb)
{
    const int64_t tm = (m + 127) / 128;
    if (tm * ((n + 127) / 128) * nb >= 512 && m >= 128 && n >= 128) return 7;
    if (tm * ((n + 63) / 64) * nb >= 256 && m >= 128 && n >= 64) return 4;
    return 10;
}

// Whether a product with operands rounded to bf16 rounds them in memory first: below that the extra
// pass over them costs more than the tiles save.
static bool rounds_in_memory(int m, int n, int k)
{
    return k > 0 && (g_bf16src == 2 || (g_bf16src == 1 && m >= 128 && n >= 128 && k >= 256 && 2.0 * m * n * (double)k >= g_bf16src_min_flops));
}

// Chains over k of an element of such a product: two, added, where the output has few tiles - fewer than
// 512 of 128x128 from rounded copies, the 64x64 class where the tile loader rounds - and one
// elsewhere.  Precision, not time, keeps the two: their rms error is 0.70 times that of one chain
// (k = 1000 to 10000), at the same speed up to 447 tiles and 0.91 times it above (2000 x 3500 x 1000 34.2
// us in one chain, 37.7 in two).
static bool bf16_two_chains(int m, int n, int k)
{
    if (!rounds_in_memory(m, n, k)) return gemm_class(m, n, 1) == 10;
    if (g_force_cfg == 7 || g_force_cfg == 11 || g_force_cfg == 13) return g_force_cfg == 11; // tuning aid
    return (int64_t)((m + 127) / 128) * ((n + 127) / 128) < 512;
}

extern "C" int nchip_gemm_is_64x64(int m, int n, int k, int precision)
{
    return (precision != 1 || !rounds_in_memory(m, n, k)) && gemm_class(m, n, 1) == 10;
}

// Whether an fp32 product of the 64x64 class is issued by gemm_small_kernel (the same sums; this is
// about time only).  That kernel reads each operand once per 16 rows or columns, 128 bytes per tile
// and k from the caches, where the 64x64 class waits for a memory round trip per 32 or 64 k.
// Measured under a kernel trace, 64x64 class -> this, us (A and B plain / A transposed / B transposed):
//   256 x 16 x 512      18.2 / 17.8 / 19.0 -> 5.6 / 5.8 / 5.9     128 x 80 x 128   7.3 / 7.1 / 7.8 -> 4.1 / 3.6 / 3.6
//   352 x 481 x 352     15.8 / 14.9 / 17.0 -> 7.7 / 8.2 / 7.6     352 x 481 x 777 32.8 / 34.1 / 31.8 -> 11.9 / 12.3 / 13.0
//   512 x 512 x 512     13.7 / 13.2 / 14.1 -> 9.3 / 11.4 / 8.9    512 x 512 x 1000 24.4 / 23.8 / 24.7 -> 14.1 / 18.3 / 14.9
//   512 x 576 x 777     29.1 / 34.4 / 19.9 -> 15.9 / 18.4 / 21.0  640 x 512 x 640 16.3 / 15.8 / 16.7 -> 16.2 / 21.2 / 20.5
//   512 x 768 x 256      9.2 / 8.7 / 9.4 -> 8.2 / 9.4 / 8.2       512 x 768 x 512 13.9 / 13.5 / 14.4 -> 12.0 / 15.4 / 15.4
//   512 of 32 x 32 x 64 10.2 / 10.3 / 10.9 -> 5.0 / 5.5 / 5.2     512 x 1024 x 192 9.3 / 9.0 / 9.5 -> 8.9 / 10.2 / 8.6
// and split over k, where one workgroup walks all chunks of its tile and no second launch adds them:
//   512 x 83 x 2048     16.0 / 15.6 / 17.2 -> 9.4 / 10.5 / 9.2    512 x 192 x 2048 16.1 / 15.5 / 16.6 -> 15.6 / 18.6 / 15.8
//   64 x 64 x 3072      15.1 / 15.9 / 15.3 -> 11.2 / 13.4 / 10.2  512 x 256 x 1500 16.9 / 16.7 / 17.2 -> 17.4 / 17.8 / 18.8
static bool gemm_is_small(int m, int n, int k, int batch, int ksplit)
{
    const int64_t tiles = (int64_t)((m + 15) / 16) * ((n + 15) / 16) * batch;
    return tiles <= 2048 && (k < 1024 ? tiles <= 1152 || tiles * k <= 3 << 17 : k <= 3072 && tiles * k <= 3 << 18) && gemm_class(m, n, (int64_t)batch * ksplit) == 10;
}

// Whether an fp32 product of class 7, 4 or 10 is issued by gemm_dma_kernel (the same sums; this is about
// time only): whole stages of 32 k, 16-byte units, 32-bit offsets inside a stage.  The single-chain
// classes gain everywhere; of the 64x64 class, more tiles than CUs and operands that need no reads across
// rows (both K-contiguous reads of a step hit two banks twice); partial tiles, whose rows this kernel
// repeats and the other moves to the edge, and short reductions make up for one such operand.  Speed against
// the 64x64 class, K = 128 / 352 / 512 / 1024 / 2048 / 4096:
//   512 x 2112 (264 tiles)   1.23 / 1.22 / 1.12 / 1.11 / 1.11 / 1.10   A transposed 1.15 / 1.15 / 1.08 / 1.07 / 1.05 / 1.04
//   1028 x 1028 (289)        1.35 / 1.27 / 1.22 / 1.18 / 1.14 / 1.11   A transposed 1.23 / 1.19 / 1.11 / 1.08 / 1.06 / 1.04
//   512 x 2048 (256)         1.08 / 1.08 / 1.01 / 1.01; 43.9 us against 42.5 at 2048 (kept out), B transposed 1.11 / 1.12 / 1.06 / 1.08 / 1.10 / 1.10
//   1000 x 1000 (256)        1.16 / 1.13 / 1.16 / 1.10 / 1.08 / 1.05   A transposed 1.10 / 1.04 / 0.95 / 0.95 / 0.93 / 0.92
//   352 x 1068 (102)         K = 352 1.16, A transposed 1.05, B transposed 1.22; 512 1.17, 0.98, 1.23
//   128 of 100 x 100 (512)   B transposed 1.41 / 1.26 / 1.23 / 1.09 / 0.97 / 0.95, the others 1.07 and up
// class 4: 2048 x 2048 x 512 48.5 -> 42.0, 1024 x 2048 x 512 24.9 -> 23.7, 256 of 320 x 64 x 128 31.0 -> 24.8
// class 7: 4096 x 4096 x 1024 300 -> 261, A transposed 291 -> 267, B transposed (4096 x 1024 x 4096) 303 -> 249
static bool dma_fits_f32(const GemmArgs &g, int ta, int tb)
{
    const int64_t any = g.lda | g.ldb | g.sa | g.sb | g.sa_in | g.sb_in | (ta ? 0 : g.M) | (tb ? g.N : 0);
    return g.K > 0 && g.K % 32 == 0 && (g.ksplit == 1 || g.kchunk % 32 == 0) && any % 4 == 0 &&
           (((uintptr_t)g.A | (uintptr_t)g.B) & 15) == 0 && g.lda < 1 << 22 && g.ldb < 1 << 22;
}
static bool dma_gains_f32(const GemmArgs &g, int cfg, int ta, int tb)
{
    if (cfg != 10) return cfg == 7 || cfg == 4;
    const int64_t tiles = (int64_t)((g.M + 63) / 64) * ((g.N + 63) / 64) * g.batch * g.ksplit;
    const bool partial = g.M % 64 || g.N % 64;
    return tiles > 256 || tb || (ta ? partial && g.K <= 384 : partial || g.K <= 1024);
}

extern "C" int nchip_gemm_is_small(int m, int n, int k, int batch)
{
    return !g_force_cfg && gemm_is_small(m, n, k, batch, nchip_gemm_pick_ksplit(m, n, k, batch));
}

static int gemm2_impl(void *stream, int ta, int tb, int m, int n, int k, float alpha,
                      const float *A, int64_t lda, int64_t sa_out, int64_t sa_in,
                      const float *B, int64_t ldb, int64_t sb_out, int64_t sb_in,
                      float beta, float *C, int64_t ldc, int64_t sc_out, int64_t sc_in,
                      int batch, int batch_in,
                      const float *bias, int act, float *pre, const float *addend, int precision,
                      int ksplit, float *workspace, const float *dpre = nullptr, int dact = 0,
                      float *rowsum = nullptr, int *rowsum_rows = nullptr)
{
    if (rowsum_rows) *rowsum_rows = 0;
    if (m <= 0 || n <= 0 || batch <= 0)
        return 0;
    if (k < 0 || !A || !B || !C || lda < (ta ? k : m) || ldb < (tb ? n : k) || ldc < m || batch_in < 1) {
        fprintf(stderr, "nchip_gemm: bad arguments (m=%d n=%d k=%d lda=%ld ldb=%ld ldc=%ld)\n",
                m, n, k, (long)lda, (long)ldb, (long)ldc);
        return -1;
    }
    const bool invariant = (precision & NCHIP_GEMM_WIDTH_INVARIANT) != 0;
    precision &= 0xff;
    if (ksplit < 1 || invariant) ksplit = 1;
    if (ksplit > 1 && !workspace) {
        fprintf(stderr, "nchip_gemm: ksplit=%d needs a workspace\n", ksplit);
        return -1;
    }
    if ((int64_t)batch * ksplit > 65535) {
        fprintf(stderr, "nchip_gemm: batch*ksplit=%ld exceeds the grid limit\n", (long)batch * ksplit);
        return -1;
    }
    GemmArgs g;
    memset(&g, 0, sizeof(g));
    g.A = A; g.B = B; g.C = C; g.bias = bias; g.add = addend; g.pre = pre; g.ws = workspace;
    g.dpre = dpre; g.dact = act_for_precision(dact, precision);
    g.rowsum = nullptr;
    g.lda = lda; g.ldb = ldb; g.ldc = ldc; g.sa = sa_out; g.sb = sb_out; g.sc = sc_out;
    g.sa_in = sa_in; g.sb_in = sb_in; g.sc_in = sc_in; g.batch_in = batch_in;
    g.M = m; g.N = n; g.K = k; g.batch = batch; g.ksplit = ksplit;
    g.kchunk = ((k + ksplit - 1) / ksplit + KALIGN - 1) / KALIGN * KALIGN;
    if (g.kchunk < KALIGN) g.kchunk = KALIGN;
    g.alpha = alpha; g.beta = beta; g.act = act_for_precision(act, precision);
    g.grp = nullptr; g.n_grp = 0;
    hipStream_t st = (hipStream_t)stream;
    ProfRec rec;
    if (g_prof_on) {
        (void)hipEventCreate(&rec.start);
        (void)hipEventCreate(&rec.stop);
        rec.variant = -1;
        rec.flops = 2.0 * m * n * (double)k * batch;
    }
    ProfRec *pr = g_prof_on ? &rec : nullptr;
    if (invariant && g_skinny == 3 && ta && !tb && batch == 1 && precision == 0 && n <= 64 && k >= 32 && k % 32 == 0 &&
        m % 32 == 0 && lda % 4 == 0 && ldb % 4 == 0 && (((uintptr_t)A | (uintptr_t)B) & 15) == 0 && beta == 0.0f &&
        alpha == 1.0f && !dpre && !g_prof_on) {
        // a few token columns against a k-major A (a weight matrix's transposed copy): same chains
        launch_fewcol_mfma(g, m, 1, st, true);
        hipError_t e = hipGetLastError();
        if (e != hipSuccess) {
            fprintf(stderr, "nchip_gemm: launch failed: %s\n", hipGetErrorString(e));
            return -2;
        }
        return 0;
    }
    if (invariant && g_skinny && !ta && !tb && batch == 1 && precision == 0 && n <= 64 && k >= 32 && k % 32 == 0 &&
        m % 32 == 0 && lda % 4 == 0 && ldb % 4 == 0 && (((uintptr_t)A | (uintptr_t)B) & 15) == 0 && beta == 0.0f && !g_prof_on) {
        // a few token columns: the same arithmetic without the tile pipeline
        if (g_skinny == 3 && alpha == 1.0f && !dpre)
            launch_fewcol_mfma(g, m, 1, st);
        else if (g_skinny >= 2 && alpha == 1.0f && !dpre)
            launch_fewcol_fma(g, dim3(m / 8, (n + 7) / 8), st);
        else
            hipLaunchKernelGGL(gemm_skinny_nn<16>, dim3(m / 32, (n + 31) / 32), dim3(256), 0, st, g);
        hipError_t e = hipGetLastError();
        if (e != hipSuccess) {
            fprintf(stderr, "nchip_gemm: launch failed: %s\n", hipGetErrorString(e));
            return -2;
        }
        return 0;
    }
    const bool small_fits = precision == 0 && !dpre && ksplit <= SMALL_KSPLIT && (k + 16) * (lda > ldb ? lda : ldb) < 1 << 29; // (32-bit byte offsets)
    const bool small = !invariant && !g_force_cfg && small_fits && gemm_is_small(m, n, k, batch, ksplit);
    int cfg = invariant ? 30 : g_force_cfg; // tuning aid: 0 = choose from the shape
    if (cfg == 40 && !small_fits) cfg = 10;
    if (!cfg) cfg = small ? 40 : gemm_class(m, n, (int64_t)batch * ksplit);
    // Large bf16 products are bound by operand traffic from L2, not by the MFMA
    // rate: round both operands to bf16 in memory first (one streaming pass
    // each) and let the tiles load half the bytes.  The rounded values are
    // the ones the conversion inside the tile loader would produce, so the
    // result is the same either way.
    bool from_bf16 = false;
    if (precision == 1 && batch == 1 && ksplit == 1 && !invariant && rounds_in_memory(m, n, k)) {
        const int kpad = (k + 63) / 64 * 64;
        const size_t ea = cast_elems(ta ? k : m, ta ? m : k, ta != 0, kpad);
        const size_t eb = cast_elems(tb ? n : k, tb ? k : n, tb == 0, kpad);
        uint16_t *buf = cast_scratch(st, ea + eb);
        if (buf) {
            g.lda = cast_operand(st, A, ta ? k : m, ta ? m : k, lda, ta != 0, kpad, buf);
            g.ldb = cast_operand(st, B, tb ? n : k, tb ? k : n, ldb, tb == 0, kpad, buf + ea);
            g.A = reinterpret_cast<const float *>(buf);
            g.B = reinterpret_cast<const float *>(buf + ea);
            g.K = kpad; g.kchunk = kpad;
            from_bf16 = true;
        }
    }
    const bool dma = precision == 0 && !g_force_cfg && dma_fits_f32(g, ta, tb) && dma_gains_f32(g, cfg, ta, tb);
    // partial row sums of the result (activation-gradient epilogue): one row per 16 columns of the
    // padded column range, 8 in two k groups staged by DMA; only the plain tile classes write them
    if (rowsum && rowsum_rows && dpre && ksplit == 1 && batch == 1 && !from_bf16 &&
        (cfg == 7 || cfg == 4 || cfg == 10 || cfg == 30)) {
        const int bn = cfg == 7 && !(dma && tb) ? 128 : 64;
        g.rowsum = rowsum;
        *rowsum_rows = (n + bn - 1) / bn * bn / (dma && cfg == 10 ? 8 : 16);
    }
    if (from_bf16) {
        const bool two_chains = bf16_two_chains(m, n, k);
        const int cls = dma_class(g, two_chains);
        rec.variant = (two_chains ? 92 : 64) + cls * 4 + (ta ? 2 : 0) + (tb ? 1 : 0);
        if (launch_dma_class(st, cls, two_chains, ta, tb, g, pr)) return -2;
    } else if (precision == 1) {
        if (cfg == 7) launch_tile<128, 128, 32, 4, 2, 1>(st, ta, tb, g, pr);
        else if (cfg == 4) launch_tile<128, 64, 32, 4, 2, 1>(st, ta, tb, g, pr);
        else if (cfg == 9) launch_tile<64, 64, 64, 2, 2, 1, 2>(st, ta, tb, g, pr);
        else launch_tile<64, 64, 32, 2, 2, 1, 2>(st, ta, tb, g, pr);
    } else if (dma) {
        if (cfg == 10 ? launch_dma<1, 64, 64, 2, 2, 2, 4>(st, ta, tb, g, pr)
            : cfg == 7 && !tb ? launch_dma<1, 128, 128, 2, 2, 1, 2>(st, ta, tb, g, pr)
                              : launch_dma<1, 128, 64, 4, 2, 1, 3>(st, ta, tb, g, pr))
            return -2;
    } else if (cfg == 40) {
        // (wavefronts: the two chains, or as many of the 2 ksplit; blocks in flight: one round trip's)
        if (ksplit > 4) launch_small<16, 8, 1>(st, ta, tb, g, pr);
        else if (ksplit > 1) launch_small<8, 8, 1>(st, ta, tb, g, pr);
        else if (k <= 32) launch_small<2, 1, 0>(st, ta, tb, g, pr);
        else if (k <= 64) launch_small<2, 2, 0>(st, ta, tb, g, pr);
        else if (k <= 128) launch_small<2, 4, 0>(st, ta, tb, g, pr);
        else if (k <= 256) launch_small<2, 8, 0>(st, ta, tb, g, pr);
        else if (k <= 384) launch_small<2, 12, 0>(st, ta, tb, g, pr);
        else launch_small<2, 16, 0>(st, ta, tb, g, pr);
    } else if (cfg == 1) {
        launch_tile<128, 128, 16, 2, 2, 0>(st, ta, tb, g, pr);
    } else if (cfg == 2) {
        launch_tile<128, 128, 16, 4, 2, 0>(st, ta, tb, g, pr);
    } else if (cfg == 3) {
        launch_tile<128, 64, 16, 2, 2, 0>(st, ta, tb, g, pr);
    } else if (cfg == 4) {
        launch_tile<128, 64, 32, 4, 2, 0>(st, ta, tb, g, pr);
    } else if (cfg == 6) {
        launch_tile<64, 128, 16, 2, 2, 0>(st, ta, tb, g, pr);
    } else if (cfg == 7) {
        launch_tile<128, 128, 32, 4, 2, 0, 1, 2, 1, 1>(st, ta, tb, g, pr); // rolling fragment window: two accumulator tiles per wavefront
    } else if (cfg == 8) {
        launch_tile<64, 64, 32, 2, 2, 0, 2>(st, ta, tb, g, pr);
    } else if (cfg == 9) {
        launch_tile<64, 64, 64, 2, 2, 0, 2>(st, ta, tb, g, pr);
    } else if (cfg == 10) {
        launch_tile<64, 64, 32, 2, 2, 0, 2, 4>(st, ta, tb, g, pr);
    } else if (cfg == 30) { // the width-invariant class: four chains per element
        launch_tile<64, 64, 32, 2, 2, 0, 2, 4, 2>(st, ta, tb, g, pr);
    } else {
        launch_tile<64, 64, 16, 2, 2, 0>(st, ta, tb, g, pr);
    }
    if (g_prof_on) {
        int tile = cfg == 40 ? 6 : cfg == 7 ? 2 : (cfg == 4 ? 1 : ((cfg == 8 || cfg == 10 || cfg == 30) ? 3 : 0));
        if (!from_bf16) rec.variant = tile * 8 + (ta ? 4 : 0) + (tb ? 2 : 0) + (precision == 1 ? 1 : 0);
        if (dma) rec.variant = 120 + (cfg == 10 ? 12 : (cfg == 7 && !tb ? 4 : 8)) + (ta ? 2 : 0) + (tb ? 1 : 0);
        g_prof.push_back(rec);
    }
    if (ksplit > 1 && cfg != 40) {
        int64_t total = (int64_t)m * n;
        int nb = (int)((total + 255) / 256);
        if (nb > 2048) nb = 2048;
        hipLaunchKernelGGL(gemm_splitk_reduce, dim3(nb, batch), dim3(256), 0, st, g);
    }
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) {
        fprintf(stderr, "nchip_gemm: launch failed: %s\n", hipGetErrorString(e));
        return -2;
    }
    return 0;
}

extern "C" int nchip_gemm2(void *stream, int ta, int tb, int m, int n, int k, float alpha,
                           const float *A, int64_t lda, int64_t sa_out, int64_t sa_in,
                           const float *B, int64_t ldb, int64_t sb_out, int64_t sb_in,
                           float beta, float *C, int64_t ldc, int64_t sc_out, int64_t sc_in,
                           int batch, int batch_in,
                           const float *bias, int act, float *pre, int precision,
                           int ksplit, float *workspace)
{
    return gemm2_impl(stream, ta, tb, m, n, k, alpha, A, lda, sa_out, sa_in, B, ldb, sb_out, sb_in,
                      beta, C, ldc, sc_out, sc_in, batch, batch_in, bias, act, pre, nullptr, precision,
                      ksplit, workspace);
}

extern "C" int nchip_gemm_add(void *stream, int ta, int tb, int m, int n, int k, float alpha,
                              const float *A, int64_t lda, int64_t stride_a,
                              const float *B, int64_t ldb, int64_t stride_b,
                              float *C, int64_t ldc, int64_t stride_c, int batch,
                              const float *bias, int act, float *pre, const float *addend,
                              int precision, int ksplit, float *workspace)
{
    return gemm2_impl(stream, ta, tb, m, n, k, alpha, A, lda, stride_a, 0, B, ldb, stride_b, 0,
                      0.0f, C, ldc, stride_c, 0, batch, 1, bias, act, pre, addend, precision, ksplit,
                      workspace);
}

extern "C" int nchip_gemm_dact(void *stream, int ta, int tb, int m, int n, int k, float alpha,
                               const float *A, int64_t lda, const float *B, int64_t ldb,
                               float *C, int64_t ldc, const float *pre_act, int act,
                               int precision, int ksplit, float *workspace)
{
    return gemm2_impl(stream, ta, tb, m, n, k, alpha, A, lda, 0, 0, B, ldb, 0, 0, 0.0f, C, ldc, 0, 0, 1, 1,
                      nullptr, 0, nullptr, nullptr, precision, ksplit, workspace, pre_act, act);
}

// nchip_gemm_dact that also leaves partial row sums of C: rowsum holds nchip_gemm_rowsum_rows(n)
// rows of m floats, of which *rows_written are written, each over 8 or 16 columns of C (0 when this
// product's kernel does not write them: the caller then sums C itself)
extern "C" int nchip_gemm_rowsum_rows(int n) { return (n + 255) / 256 * 32; } // (the widest tile's, two k groups)

extern "C" int nchip_gemm_dact_rowsum(void *stream, int ta, int tb, int m, int n, int k, float alpha,
                                      const float *A, int64_t lda, const float *B, int64_t ldb,
                                      float *C, int64_t ldc, const float *pre_act, int act,
                                      int precision, int ksplit, float *workspace,
                                      float *rowsum, int *rows_written)
{
    return gemm2_impl(stream, ta, tb, m, n, k, alpha, A, lda, 0, 0, B, ldb, 0, 0, 0.0f, C, ldc, 0, 0, 1, 1,
                      nullptr, 0, nullptr, nullptr, precision, ksplit, workspace, pre_act, act, rowsum, rows_written);
}

extern "C" int nchip_gemm(void *stream, int ta, int tb, int m, int n, int k, float alpha,
                          const float *A, int64_t lda, int64_t stride_a,
                          const float *B, int64_t ldb, int64_t stride_b,
                          float beta, float *C, int64_t ldc, int64_t stride_c, int batch,
                          const float *bias, int act, float *pre, int precision,
                          int ksplit, float *workspace)
{
    return nchip_gemm2(stream, ta, tb, m, n, k, alpha, A, lda, stride_a, 0, B, ldb, stride_b, 0,
                       beta, C, ldc, stride_c, 0, batch, 1, bias, act, pre, precision, ksplit,
                       workspace);
}

// tuning aid: forces tile configuration `cfg` for every later call (0 = automatic)
extern "C" void nchip_gemm_force_config(int cfg)
{
    g_force_cfg = cfg;
}

// testing aid: 0 sends width-invariant products of a few columns through the tile
// kernel again, 1 through the 32x32x2 MFMA few-column kernel, 2 through the vector-ALU
// kernel, 3 (default) through the 16x16x4 MFMA kernel (same bits, by construction: the
// tests compare the four)
extern "C" void nchip_gemm_few_columns_kernel(int on)
{
    g_skinny = on;
}

// Two width-invariant few-column products with one operand in common, in ONE launch:
// C0 (m0 x n) = A0 B + bias0 and C1 (m1 x n) = A1 B + bias1 (bias pointers may be NULL),
// the decoder's query and key/value projections of a timestep.  Same kernel and the same
// bits as two nchip_gemm calls in width-invariant mode.  Returns 1 when the shapes are not
// the few-column kernel's (nothing launched: the caller issues the two products itself).
extern "C" int nchip_gemm_pair_few_columns(void *stream, int m0, int m1, int n, int k,
                                           const float *A0, int64_t lda0, const float *A1, int64_t lda1,
                                           const float *B, int64_t ldb,
                                           float *C0, int64_t ldc0, float *C1, int64_t ldc1,
                                           const float *bias0, const float *bias1, int a_k_major)
{
    if (m0 <= 0 || m1 <= 0 || n <= 0 || !A0 || !A1 || !B || !C0 || !C1) return -1;
    if (a_k_major && g_skinny != 3) return 1;
    if (!g_skinny || g_prof_on || n > 64 || k < 32 || k % 32 || m0 % 32 || m1 % 32 || lda0 % 4 || lda1 % 4 || ldb % 4 ||
        lda0 < (a_k_major ? k : m0) || lda1 < (a_k_major ? k : m1) || ldb < k || ldc0 < m0 || ldc1 < m1 ||
        (((uintptr_t)A0 | (uintptr_t)A1 | (uintptr_t)B) & 15) != 0)
        return 1;
    GemmArgs g;
    memset(&g, 0, sizeof(g));
    g.A = A0; g.B = B; g.C = C0; g.bias = bias0; g.lda = lda0; g.ldb = ldb; g.ldc = ldc0;
    g.M = m0; g.N = n; g.K = k; g.batch = 1; g.batch_in = 1; g.ksplit = 1; g.alpha = 1.0f;
    g.A_1 = A1; g.C_1 = C1; g.bias_1 = bias1; g.lda_1 = lda1; g.ldc_1 = ldc1; g.M_1 = m1;
    const int mmax = m0 > m1 ? m0 : m1;
    if (g_skinny == 3)
        launch_fewcol_mfma(g, mmax, 2, (hipStream_t)stream, a_k_major != 0);
    else if (g_skinny == 2)
        launch_fewcol_fma(g, dim3(mmax / 8, (n + 7) / 8, 2), (hipStream_t)stream);
    else
        hipLaunchKernelGGL(gemm_skinny_nn<16>, dim3(mmax / 32, (n + 31) / 32, 2), dim3(256), 0, (hipStream_t)stream, g);
    if (hipGetLastError() != hipSuccess) {
        fprintf(stderr, "nchip_gemm_pair_few_columns: launch failed\n");
        return -2;
    }
    return 0;
}

// One or two width-invariant few-column products of the layer norm (avg = 1) or RMS norm
// (avg = 0) of B's columns, in ONE launch: C0 (m0 x n) = act0(A0 norm(B) + bias0) and, when
// m1 > 0, C1 (m1 x n) = A1 norm(B) + bias1.  B holds k = 128, 256 or 512 raw features per
// column; ln_w / ln_b are the gain and bias (both or neither); the normalised columns are
// also written to ln_out (leading dimension ld_ln) when it is not NULL.  The bits are those
// of nchip_norm_fwd followed by the products in width-invariant mode.  Returns 1 when the
// shapes are not this kernel's (nothing launched: the caller issues the steps itself).
extern "C" int nchip_norm_gemm_few_columns(void *stream, const float *ln_w, const float *ln_b, float eps, int avg,
                                           float *ln_out, int64_t ld_ln, int m0, int m1, int n, int k,
                                           const float *A0, int64_t lda0, const float *A1, int64_t lda1,
                                           const float *B, int64_t ldb, float *C0, int64_t ldc0,
                                           float *C1, int64_t ldc1, const float *bias0, const float *bias1, int act0,
                                           int a_k_major)
{
    if (m0 <= 0 || m1 < 0 || n <= 0 || !A0 || !B || !C0 || (m1 > 0 && (!A1 || !C1)) || (ln_w == nullptr) != (ln_b == nullptr))
        return -1;
    if (g_skinny != 3 || g_prof_on || n > 64 || (k != 128 && k != 256 && k != 512) || m0 % 32 || m1 % 32 || lda0 % 4 ||
        (m1 > 0 && lda1 % 4) || lda0 < (a_k_major ? k : m0) || (m1 > 0 && lda1 < (a_k_major ? k : m1)) || ldb < k || ldc0 < m0 || (m1 > 0 && ldc1 < m1) ||
        (ln_out && ld_ln < k) || (((uintptr_t)A0 | (uintptr_t)A1) & 15) != 0 ||
        (act0 != NCHIP_ACT_NONE && act0 != NCHIP_ACT_GELU && act0 != NCHIP_ACT_RELU))
        return 1;
    GemmArgs g;
    memset(&g, 0, sizeof(g));
    g.A = A0; g.B = B; g.C = C0; g.bias = bias0; g.lda = lda0; g.ldb = ldb; g.ldc = ldc0; g.act = act0;
    g.M = m0; g.N = n; g.K = k; g.batch = 1; g.batch_in = 1; g.ksplit = 1; g.alpha = 1.0f;
    g.A_1 = A1; g.C_1 = C1; g.bias_1 = bias1; g.lda_1 = lda1; g.ldc_1 = ldc1; g.M_1 = m1;
    g.ln_w = ln_w; g.ln_b = ln_b; g.ln_out = ln_out; g.ld_ln = ld_ln; g.ln_eps = eps; g.ln_avg = avg;
    const int mmax = m0 > m1 ? m0 : m1;
    const dim3 grid(mmax / 16, (n + 15) / 16, m1 > 0 ? 2 : 1);
    hipStream_t st = (hipStream_t)stream;
    if (a_k_major) {
        if (k == 128) hipLaunchKernelGGL((gemm_fewcol_mfma<2, 2, 16, 1>), grid, dim3(256), 0, st, g);
        else if (k == 256) hipLaunchKernelGGL((gemm_fewcol_mfma<2, 4, 16, 1>), grid, dim3(256), 0, st, g);
        else hipLaunchKernelGGL((gemm_fewcol_mfma<2, 8, 16, 1>), grid, dim3(256), 0, st, g);
    } else if (k == 128) hipLaunchKernelGGL((gemm_fewcol_mfma<2, 2>), grid, dim3(256), 0, st, g);
    else if (k == 256) hipLaunchKernelGGL((gemm_fewcol_mfma<2, 4>), grid, dim3(256), 0, st, g);
    else hipLaunchKernelGGL((gemm_fewcol_mfma<2, 8>), grid, dim3(256), 0, st, g);
    if (hipGetLastError() != hipSuccess) {
        fprintf(stderr, "nchip_norm_gemm_few_columns: launch failed\n");
        return -2;
    }
    return 0;
}

// 0: bf16 products always round their operands inside the tile loader;
// 1: large ones go through bf16 copies of the operands (default);
// 2: every unbatched bf16 product does (testing aid)
extern "C" void nchip_gemm_bf16_source(int mode)
{
    g_bf16src = mode;
}

extern "C" void nchip_gemm_force_band(int gm)
{
    g_force_gm = gm;
}

extern "C" int nchip_cast_bf16(void *stream, const float *src, uint16_t *dst, int64_t n)
{
    if (n <= 0) return 0;
    if (!src || !dst || (((uintptr_t)src | (uintptr_t)dst) & 15) != 0) {
        fprintf(stderr, "nchip_cast_bf16: 16-byte aligned buffers expected\n");
        return -1;
    }
    int64_t nb = (n / 8 + 255) / 256;
    if (nb < 1) nb = 1;
    if (nb > 4096) nb = 4096;
    hipLaunchKernelGGL(cast_bf16_flat_kernel, dim3((unsigned)nb), dim3(256), 0, (hipStream_t)stream, src, dst, n);
    if (hipGetLastError() != hipSuccess) { fprintf(stderr, "nchip_cast_bf16: launch failed\n"); return -2; }
    return 0;
}

extern "C" int nchip_widen_bf16(void *stream, const uint16_t *src, float *dst, int64_t n)
{
    if (n <= 0) return 0;
    int64_t nb = (n + 255) / 256;
    if (nb > 8192) nb = 8192;
    hipLaunchKernelGGL(widen_bf16_flat_kernel, dim3((unsigned)nb), dim3(256), 0, (hipStream_t)stream, src, dst, n);
    if (hipGetLastError() != hipSuccess) { fprintf(stderr, "nchip_widen_bf16: launch failed\n"); return -2; }
    return 0;
}

// Product whose operands are already bf16 in memory (the rounded copies of the fp32 matrices,
// element for element in the same column-major layout: no padding).  Unguarded 16-byte loads
// throughout, so the shapes must fit: k a multiple of 64; an operand whose long axis is
// contiguous (A with ta = 0, B with tb = 1) a multiple of 64 along it; leading dimensions
// multiples of 8 elements; 16-byte aligned bases.  Returns 1 when they do not (nothing launched: the caller takes another
// route).  Epilogue options as in the fp32-operand calls; c16, when given, receives the
// result rounded to bf16 next to C.
extern "C" int nchip_gemm_bf16_operands(void *stream, const NchipGemmBf16Args *a)
{
    if (a->rows_written) *a->rows_written = 0;
    const int m = a->m, n = a->n, k = a->k, ta = a->ta != 0, tb = a->tb != 0;
    if (m <= 0 || n <= 0) return 0;
    if (!a->A16 || !a->B16 || !a->C || k <= 0 || a->lda < (ta ? k : m) || a->ldb < (tb ? n : k) || a->ldc < m) {
        fprintf(stderr, "nchip_gemm_bf16_operands: bad arguments (m=%d n=%d k=%d)\n", m, n, k);
        return -1;
    }
    if (k % 64 || a->lda % 8 || a->ldb % 8 || (!ta && m % 64) || (tb && n % 64) || (((uintptr_t)a->A16 | (uintptr_t)a->B16) & 15) != 0)
        return 1;
    GemmArgs g;
    memset(&g, 0, sizeof(g));
    g.A = reinterpret_cast<const float *>(a->A16); g.B = reinterpret_cast<const float *>(a->B16);
    g.C = a->C; g.c16 = a->C16; g.bias = a->bias; g.add = a->addend; g.pre = a->pre;
    g.dpre = a->dpre; g.dact = act_for_precision(a->dact, 2);
    g.lda = a->lda; g.ldb = a->ldb; g.ldc = a->ldc;
    g.batch_in = 1; g.M = m; g.N = n; g.K = k; g.batch = 1; g.ksplit = 1; g.kchunk = k;
    g.alpha = a->alpha; g.beta = 0.0f; g.act = act_for_precision(a->act, 2);
    hipStream_t st = (hipStream_t)stream;
    // One chain where the operands whose long axis is contiguous fill the tiles that cover the chip (128x128 from
    // 224 of them on, then 128x64, else 64x64); elsewhere the sums of nchip_gemm with precision 1.
    const int64_t t128 = (int64_t)((m + 127) / 128) * ((n + 127) / 128), t128x64 = (int64_t)((m + 127) / 128) * ((n + 63) / 64);
    const int bm = t128 >= 224 || (t128x64 >= 224 && m >= 128) ? 128 : 64, bn = t128 >= 224 ? 128 : 64;
    const bool whole = (ta || m % bm == 0) && (!tb || n % bn == 0), two_chains = !whole && bf16_two_chains(m, n, k);
    int cls = dma_class(g, two_chains);
    if (cls != 6 && g_bf16ops_cls >= 1 && g_bf16ops_cls <= 5 && !(two_chains && g_bf16ops_cls == 4)) cls = g_bf16ops_cls;
    if (a->rowsum && a->rows_written && a->dpre) {
        const int bn = cls == 4 ? 256 : (cls == 1 || cls == 5 ? 128 : 64);
        g.rowsum = a->rowsum;
        *a->rows_written = (n + bn - 1) / bn * bn / 16;
    }
    ProfRec rec;
    if (g_prof_on) {
        (void)hipEventCreate(&rec.start);
        (void)hipEventCreate(&rec.stop);
        rec.flops = 2.0 * m * n * (double)k;
        rec.variant = (two_chains ? 92 : 64) + cls * 4 + ta * 2 + tb;
    }
    ProfRec *pr = g_prof_on ? &rec : nullptr;
    if (launch_dma_class(st, cls, two_chains, ta, tb, g, pr)) return -2;
    if (g_prof_on) g_prof.push_back(rec);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) {
        fprintf(stderr, "nchip_gemm_bf16_operands: launch failed: %s\n", hipGetErrorString(e));
        return -2;
    }
    return 0;
}

// tuning aid: 0 = choose the bf16-operand tile class from the shape, 1 = 128x128, 2 = 128x64, 3 = 64x64, 4 = 256x256,
// 5 = 128x128 with 8 wavefronts
extern "C" void nchip_gemm_bf16_operands_class(int cls) { g_bf16ops_cls = cls; }

// ---- profiling entry points ---------------------------------------------------
extern "C" void nchip_gemm_profile_enable(int on)
{
    g_prof_on = on != 0;
}

extern "C" int nchip_gemm_profile_read(int max_variants, char (*names)[48], int64_t *launches,
                                       double *flops, double *seconds)
{
    constexpr int NVAR = 136;
    double fl[NVAR] = { 0 }, sec[NVAR] = { 0 };
    int64_t cnt[NVAR] = { 0 };
    for (ProfRec &r : g_prof) {
        float ms = 0.0f;
        (void)hipEventSynchronize(r.stop);
        (void)hipEventElapsedTime(&ms, r.start, r.stop);
        if (r.variant >= 0 && r.variant < NVAR) {
            fl[r.variant] += r.flops;
            sec[r.variant] += ms * 1e-3;
            cnt[r.variant]++;
        }
        (void)hipEventDestroy(r.start);
        (void)hipEventDestroy(r.stop);
    }
    g_prof.clear();
    static const char *tiles_f32[4] = { "64,64,16,2,2", "128,64,32,4,2", "128,128,32,4,2", "64,64,32,2,2" };
    static const char *tiles_bf16[4] = { "64,64,32,2,2", "128,64,32,4,2", "128,128,32,4,2", "64,64,32,2,2" };
    static const char *tiles_ops[7] = { "256,256,2,4,1,2", "128,128,2,2,1,2", "128,64,2,2,1,3", "64,64,2,2,1,4", "256,256,2,4,1,2", "128,128,2,4,1,4", "64,64,2,2,1,4" }; // 0: grouped; 6: 64-bit offsets
    static const char *tiles_f32_dma[4] = { "128,128,4,2,1,4", "128,128,2,2,1,2", "128,64,4,2,1,3", "64,64,2,2,2,4" }; // 0: grouped
    int n = 0;
    for (int v = 0; v < NVAR && n < max_variants; v++) {
        if (!cnt[v]) continue;
        if (v >= 120) { // fp32 operands staged by DMA
            snprintf(names[n], 48, "gemm_dma_kernel<1,%s,%d,%d%s>", tiles_f32_dma[(v - 120) / 4], (v >> 1) & 1, v & 1, v < 124 ? ",grouped" : "");
        } else if (v >= 92) { // bf16, two chains
            snprintf(names[n], 48, "gemm_dma_kernel<0,%s,%d,%d,2>", tiles_ops[(v - 92) / 4], (v >> 1) & 1, v & 1);
        } else if (v >= 64) { // operands read as bf16: gemm_dma_kernel<tile, wavefronts, stages, ta, tb>
            snprintf(names[n], 48, "gemm_dma_kernel<0,%s,%d,%d%s>", tiles_ops[(v - 64) / 4], (v >> 1) & 1, v & 1,
                     v < 68 ? ",grouped" : "");
        } else if (v >= 48) {
            snprintf(names[n], 48, "gemm_small_kernel<%d,%d>", (v >> 2) & 1, (v >> 1) & 1);
        } else if (v >= 32) { // the grouped launch in 128 x 128 tiles
            snprintf(names[n], 48, "gemm_dma_kernel<0,128,128,2,2,1,2,%d,%d,grouped>", (v >> 1) & 1, v & 1);
        } else {
            const bool two_groups = v / 8 == 3 || ((v & 1) && v / 8 == 0);
            snprintf(names[n], 48, "gemm_kernel<%s,%d,%d,%d%s>", (v & 1) ? tiles_bf16[v / 8] : tiles_f32[v / 8],
                     (v >> 2) & 1, (v >> 1) & 1, v & 1, two_groups ? ",2" : "");
        }
        launches[n] = cnt[v]; flops[n] = fl[v]; seconds[n] = sec[v];
        n++;
    }
    return n;
}

// ---- grouped launch ---------------------------------------------------------------
extern "C" int nchip_gemm_grouped_tiles(int m, int n)
{
    return ((m + 127) / 128) * ((n + 127) / 128);
}

extern "C" int nchip_gemm_grouped_tiles256(int m, int n)
{
    return ((m + 255) / 256) * ((n + 255) / 256);
}

extern "C" int nchip_gemm_grouped_tiles64(int m, int n)
{
    return ((m + 63) / 64) * ((n + 63) / 64);
}

extern "C" int nchip_gemm_grouped(void *stream, int ta, int tb, const NchipGemmProblem *dev_table,
                                  int n_problems, int total_tiles, int precision, double total_flops)
{
    if (n_problems <= 0 || total_tiles <= 0) return 0;
    GemmArgs g;
    memset(&g, 0, sizeof(g));
    g.grp = dev_table; g.n_grp = n_problems;
    // 16 tiles per turn: measured at C3 (1156 tiles), FETCH_SIZE of the launch 3.18 GB at 1 (plain
    // round robin), 2.67 at 8, 2.13 at 16, duration 1574 / 1555 / 1563 us; from 32 on the runs
    // are long enough for the XCDs to finish apart (1692 us)
    { static const int gc = getenv("NCHIP_GRP_CHUNK") ? atoi(getenv("NCHIP_GRP_CHUNK")) : 16; g.grp_chunk = gc; }
    g.batch = 1; g.batch_in = 1; g.ksplit = 1;
    g.beta = precision >= 5 ? 1.0f : 0.0f; g.act = 0;
    hipStream_t st = (hipStream_t)stream;
    dim3 grid(total_tiles, 1), block(512);
    ProfRec rec;
    if (g_prof_on) {
        (void)hipEventCreate(&rec.start);
        (void)hipEventCreate(&rec.stop);
        rec.variant = precision >= 5 ? 3 * 8 + (ta ? 4 : 0) + (tb ? 2 : 0) + (precision == 6 ? 1 : 0)
                    : precision >= 2 ? (precision == 4 ? 120 : precision == 3 ? 64 : 32) + (ta ? 2 : 0) + (tb ? 1 : 0)
                                     : 2 * 8 + (ta ? 4 : 0) + (tb ? 2 : 0) + (precision == 1 ? 1 : 0);
        rec.flops = total_flops;
    }
#define GRP_LAUNCH(KERNEL, BK_, TA, TB, BF)                                                                \
    do {                                                                                                   \
        constexpr size_t dyn = lds_dynamic_bytes<128, 128, BK_, TA, TB, BF>();                             \
        if (dyn) {                                                                                         \
            static const bool ok = hipFuncSetAttribute(reinterpret_cast<const void *>(KERNEL),             \
                hipFuncAttributeMaxDynamicSharedMemorySize, (int)dyn) == hipSuccess;                       \
            if (!ok) { fprintf(stderr, "nchip_gemm_grouped: cannot reserve %zu bytes of LDS\n", dyn); return -2; } \
        }                                                                                                  \
        if (g_prof_on) hipExtLaunchKernelGGL(KERNEL, grid, block, dyn, st, rec.start, rec.stop, 0, g);     \
        else hipLaunchKernelGGL(KERNEL, grid, block, dyn, st, g);                                          \
    } while (0)
#define GRP(TA, TB, BF) GRP_LAUNCH((gemm_kernel<128, 128, 32, 4, 2, TA, TB, BF, 1, 2, 1, (BF == 0)>), 32, TA, TB, BF)
    if (precision == 6) {
        launch_tile<64, 64, 32, 2, 2, 1, 2>(st, ta, tb, g, g_prof_on ? &rec : nullptr, total_tiles);
    } else if (precision == 5) {
        launch_tile<64, 64, 32, 2, 2, 0, 2, 4>(st, ta, tb, g, g_prof_on ? &rec : nullptr, total_tiles);
    } else if (precision == 4) {
        if (launch_dma<1, 128, 128, 4, 2, 1, 4>(st, ta, tb, g, g_prof_on ? &rec : nullptr, total_tiles)) return -2;
    } else if (precision == 3) {
        if (launch_dma<0, 256, 256, 2, 4, 1, 2>(st, ta, tb, g, g_prof_on ? &rec : nullptr, total_tiles)) return -2;
    } else if (precision == 2) {
        if (launch_dma<0, 128, 128, 2, 2, 1, 2>(st, ta, tb, g, g_prof_on ? &rec : nullptr, total_tiles)) return -2;
    } else if (precision == 1) {
        if (!ta && !tb) GRP(0, 0, 1); else if (ta && !tb) GRP(1, 0, 1); else if (!ta && tb) GRP(0, 1, 1); else GRP(1, 1, 1);
    } else {
        if (!ta && !tb) GRP(0, 0, 0); else if (ta && !tb) GRP(1, 0, 0); else if (!ta && tb) GRP(0, 1, 0); else GRP(1, 1, 0);
    }
#undef GRP
#undef GRP_LAUNCH
    if (g_prof_on) g_prof.push_back(rec);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) {
        fprintf(stderr, "nchip_gemm_grouped: launch failed: %s\n", hipGetErrorString(e));
        return -2;
    }
    return 0;
}
