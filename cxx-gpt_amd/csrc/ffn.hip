// ffn.hip -- the two-stage block's expander FFNs: two bias-free Linear
// layers with the exact GELU between them, forward and backward, as FP32
// GEMMs with the elementwise work in their epilogues.
//
// Replaces the call sequence (per expander, two_stage_gpt.hpp:86-99 and
// :177-195; Linear::forward/backward at gpt_gpt.hpp:86-112):
//   forward   pre = X W1^T; act = gelu(pre); Y = act W2^T
//   backward  dP = dY W2; dact = dP * gelu'(G); dW2 += dY^T act;
//             dX = dact W1; dW1 += dact^T X
// X [M][E], W1 [F][E], W2 [E][F], row-major.  G is the tensor the caller
// evaluates gelu' at: the expanders pass their GELU output, the final FFN its
// pre-activation (:141, :179).
//
// One GEMM kernel C[M][N] = sum_k A(i,k) B(k,j) covers all six products:
//   AK: A(i,k) at A[i*lda + k] (k contiguous), else at A[k*lda + i];
//   BK: B(k,j) at B[j*ldb + k], else at B[k*ldb + j].
// Bound by the matrix unit and the card's power: the FP32 product runs as six
// bf16 MFMAs on exactly split operands (bf3.hpp).  A workgroup of 8 waves, two
// a SIMD, computes a 256 x 128 tile of C (128 x 128 where rows are few), each
// wave 64 x 64 as 2 x 2 blocks of v_mfma_f32_32x32x16_bf16 with a main and a
// cross accumulator, over k-tiles of 32.  Operands are split once per k-tile
// on their way from registers to LDS: a 256 x 128 tile takes 1.04 k splits of
// pairs a k-tile against 192 MFMAs' worth of matrix time, where splitting the
// fragments as they are read would repeat each four times.  Measured on gfx950:
// a SIMD issues about four VALU instructions in the shadow of one 32-cycle
// MFMA, and none in that of the next if they come in a block, so a quarter of a
// pair's split (two or three instructions) follows every MFMA, in program order
// (sched_barrier).  Two LDS stages (147 KB), one barrier a k-tile, fragments
// requested one product ahead; the loads of the k-tile after next refill the
// registers as they are split.
// The MFMA takes the B fragment as its first operand, so a lane's accumulator
// holds four consecutive columns of one row of C and every epilogue access is
// 16 bytes.
// M = 2048, E = 768, F = 6144, six products: 106 us each (184 TFLOP/s) at 2.0
// GHz, which the power limit leaves of 2.4, with 58% of cycles on the matrix
// unit; on v_mfma_f32_16x16x4_f32 in 128 x 128 tiles 167 us (116 TFLOP/s, 74%
// of that instruction's peak).  The step 1099 -> 720 us.
// Work is cut into P equal runs of (tile, k-tile) units in tile-major order
// (gemm_plan: one run a tile, several, or one a compute unit, so that a tile
// count just above the unit count does not leave most units idle for a second
// round).  A run computes whole tiles straight into C with the epilogue; a tile
// cut by a run boundary is left as partial tiles in the workspace (at most two
// per run, no waiting on other workgroups) and a fix-up kernel sums them in run
// order and applies the epilogue.
//
// A batch of same-shape products with element strides between them shares
// one launch: its tiles are numbered product-major and the runs cut across
// products like any other tiles.
//
// Requires E, F multiples of 4 and 16-byte aligned tensors (checked at the C
// ABI); any M.  Callers with other shapes (GPT's score matrices, whose
// sequence length S need not be a multiple of 4) store into padded rows and
// bound the operand reads separately (FfnGemm::Mc, Nc, Kc).
#include "bf3.hpp"
#include "common.hpp"
#include "gelu_dev.hpp"
#include "launch.hpp"

#include <algorithm>

namespace cxg {

constexpr int GT = 128;                 // tile rows and columns
constexpr int GKT = 32;                 // k-tile

struct GemmArgs {
    const float* A;
    const float* B;
    float* C;
    const float* G;
    float* pre;
    float* part;       // 2 * P partial tiles (slot 0, 1 per workgroup)
    long lda, ldb, ldc;
    int M, N, K;
    int Mc, Nc, Kc;    // read extents (FfnGemm)
    int tn;            // tiles along N
    int Tb;            // tiles per product of the batch
    long sA, sB, sC;   // batch strides (elements)
    int T;             // tiles (all products)
    int KT;            // k-tiles per tile
    int P;             // workgroups
    long U;            // T * KT units
};

// Stream-K partition: the U (tile, k-tile) units, tile-major, are cut into P
// contiguous runs of equal length; run w is [sk_begin(w), sk_begin(w + 1)).
__host__ __device__ inline long sk_begin(long U, int P, int w) { return U * w / P; }

// The workgroup whose run holds unit u.
__device__ inline int sk_owner(long U, int P, long u)
{
    int w = (int)(u * P / U);
    while (w + 1 < P && sk_begin(U, P, w + 1) <= u)
        w++;
    while (w > 0 && sk_begin(U, P, w) > u)
        w--;
    return w;
}

// Epilogue for four consecutive columns of one row of C at element offset off.
template <int EPI>
__device__ __forceinline__ void epi_apply(f4 v, long off, float* C, const float* G, float* pre)
{
    if (EPI == FFN_EPI_STORE) {
        *reinterpret_cast<f4*>(C + off) = v;
    } else if (EPI == FFN_EPI_GELU) {
        if (pre != nullptr)
            *reinterpret_cast<f4*>(pre + off) = v;
#pragma unroll
        for (int e = 0; e < 4; e++)
            v[e] = gelu_f(v[e]);
        *reinterpret_cast<f4*>(C + off) = v;
    } else if (EPI == FFN_EPI_DGELU) {
        const f4 g = *reinterpret_cast<const f4*>(G + off);
#pragma unroll
        for (int e = 0; e < 4; e++)
            v[e] *= gelu_d(g[e]);
        *reinterpret_cast<f4*>(C + off) = v;
    } else {   // FFN_EPI_ACCUM
        const f4 c = *reinterpret_cast<const f4*>(C + off);
        *reinterpret_cast<f4*>(C + off) = c + v;
    }
}

// Staging: an operand's k-tile of 64 * 2^RB rows x 32 k goes from memory to
// registers (8 * 2^(RB-1) floats a thread), is split there and written to LDS
// as three planes (h, m, l) of [row][32 k] bf16.
//   KC: element (row, k) at P[row*ld + k]; a thread takes eight consecutive k
//       of rows t / 4 (+ 128): two 16-byte loads, one 16-byte write a plane.
//   else: element (row, k) at P[k*ld + row]; a thread takes four consecutive
//       k of R consecutive rows (R = 4 with 256 rows, 2 with 128), lane pairs
//       the two halves of a k-chunk: four loads of R floats, an 8-byte write a
//       row and plane.
// Rows past `rows` are clamped onto the last row (KC) or the last R rows (their
// products land in C rows/columns that are never stored, or are multiplied by
// zeros of the other operand); k past K is zeroed as it is split; addresses
// stay below K (KC) or Kc k-rows.
//
// A row sits at slot_row(row) of its plane, its 16-byte k-chunk c at c ^ x(row):
// the four rows of a group rotate with the group number, so that the 16 rows
// of a fragment read, and each kind of staging write, cover all 64 banks once.
__device__ __forceinline__ int slot_at(int row, int c)
{
    const int i = row >> 2;
    return ((row & ~3) | ((row + i) & 3)) * (GKT * 2) + ((c ^ (i & 3)) << 4);
}

template <bool KC, int RB>
struct Stage {
    static constexpr int ROWS = 64 << RB;          // 128 or 256
    static constexpr int R = RB == 2 ? 4 : 2;      // rows a thread (row-contiguous)
    static constexpr int NP = 2 << RB;             // pairs of k a thread
    static constexpr int UP = KC ? 4 : 2;          // pairs of one write (a row's k-chunk or half)
    static constexpr int UL = KC ? 4 : NP;         // pairs of one group of loads
    static constexpr int PLANE = ROWS * GKT * 2;   // bytes
    const float* p[KC ? RB : 1];                   // this thread's rows (KC) or its row group
    float v[2 * NP];
    unsigned h[UP], m[UP], l[UP];

    __device__ __forceinline__ void begin(const float* __restrict__ P, long ld, int r0, int rows)
    {
        const int t = threadIdx.x;
        if constexpr (KC) {
#pragma unroll
            for (int q = 0; q < RB; q++)
                p[q] = P + (long)min(r0 + (t >> 2) + 128 * q, rows - 1) * ld;
        } else {
            const int lane = t & 63;
            p[0] = P + min(r0 + (t >> 8) * (ROWS / 2) + (lane >> 1) * R, rows - R) +
                   (long)(lane & 1) * 4 * ld;
        }
    }
    // load group q (pairs UL q .. UL q + UL - 1) of the k-tile at k0
    __device__ __forceinline__ void fetch(int q, int k0, long ld, int K, int Kc)
    {
        const int t = threadIdx.x;
        if constexpr (KC) {
            const int k = k0 + (t & 3) * 8;
            const f4 x = *reinterpret_cast<const f4*>(p[q] + min(k, K - 4));
            const f4 y = *reinterpret_cast<const f4*>(p[q] + min(k + 4, K - 4));
#pragma unroll
            for (int e = 0; e < 4; e++) {
                v[8 * q + e] = x[e];
                v[8 * q + 4 + e] = y[e];
            }
        } else {
            typedef float fR __attribute__((ext_vector_type(R)));
            const int kw = k0 + 8 * (__builtin_amdgcn_readfirstlane(t >> 6) & 3);
#pragma unroll
            for (int j = 0; j < 4; j++) {
                // k-rows kw + j (even lanes) and kw + 4 + j (odd, from p[0]),
                // both kept below Kc
                const long e0 = (long)min(kw + j, Kc - 1) * ld;
                const long e1 = (long)(min(kw + 4 + j, Kc - 1) - 4) * ld;
                const fR x = *reinterpret_cast<const fR*>(p[0] + ((t & 1) ? e1 : e0));
#pragma unroll
                for (int r = 0; r < R; r++)
                    v[4 * r + j] = x[r];
            }
        }
    }
    __device__ __forceinline__ void fetch_all(int k0, long ld, int K, int Kc)
    {
#pragma unroll
        for (int q = 0; q < NP / UL; q++)
            fetch(q, k0, ld, K, Kc);
    }
    // zero the k's at or past K (called for the last k-tile only)
    __device__ __forceinline__ void tail(int k0, int K)
    {
        const int t = threadIdx.x;
#pragma unroll
        for (int e = 0; e < 2 * NP; e++) {
            const int k = KC ? (t & 3) * 8 + (e & 7) : 8 * ((t >> 6) & 3) + 4 * (t & 1) + (e & 3);
            v[e] = k0 + k < K ? v[e] : 0.0f;
        }
    }
    // split pair x, quarter by quarter
    __device__ __forceinline__ void split(int x, int quarter)
    {
        bf3_split2_part(quarter, v[2 * x], v[2 * x + 1], h[x % UP], m[x % UP], l[x % UP]);
    }
    // pair x is split: the last pair of a write stores it
    __device__ __forceinline__ void put(int x, char* L)
    {
        const int t = threadIdx.x, w = x / UP;
        if (x % UP != UP - 1)
            return;
        if constexpr (KC) {
            const int at = slot_at((t >> 2) + 128 * w, t & 3);
            *reinterpret_cast<u4*>(L + at) = (u4){h[0], h[1], h[2], h[3]};
            *reinterpret_cast<u4*>(L + PLANE + at) = (u4){m[0], m[1], m[2], m[3]};
            *reinterpret_cast<u4*>(L + 2 * PLANE + at) = (u4){l[0], l[1], l[2], l[3]};
        } else {
            const int at = slot_at((t >> 8) * (ROWS / 2) + ((t & 63) >> 1) * R + w, (t >> 6) & 3) +
                           8 * (t & 1);
            *reinterpret_cast<u2*>(L + at) = (u2){h[0], h[1]};
            *reinterpret_cast<u2*>(L + PLANE + at) = (u2){m[0], m[1]};
            *reinterpret_cast<u2*>(L + 2 * PLANE + at) = (u2){l[0], l[1]};
        }
    }
};

// A workgroup of 8 waves computes a (128 MI) x 128 tile of C, wave w rows
// 32 MI (w / 2) .. and columns 64 (w % 2) ..
template <bool AK, bool BK, int EPI, int MI>
__global__ __launch_bounds__(512, 2) void ffn_gemm_kernel(GemmArgs a)
{
    constexpr int TM = 128 * MI;
    typedef Stage<AK, MI> SA;
    typedef Stage<BK, 1> SB;
    constexpr int STAGE = 3 * (SA::PLANE + SB::PLANE);
    __shared__ __attribute__((aligned(16))) char lds[2 * STAGE];   // 2 stages of [A, B]

    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int l32 = lane & 31, g = lane >> 5;
    const int wm = (wave >> 1) * 32 * MI, wn = (wave & 1) * 64;
    // this lane's slot of a fragment's row, k-chunks g and 2 + g; the other
    // 32-row blocks follow at multiples of 2 KB
    const int fs[2] = {slot_at(l32, g), slot_at(l32, 2 + g)};

    const long ub = sk_begin(a.U, a.P, blockIdx.x);
    const long ue = sk_begin(a.U, a.P, blockIdx.x + 1);
    for (long u = ub; u < ue;) {
        // segment: k-tiles [ka, kb) of tile t
        const int t = (int)(u / a.KT);
        const int ka = (int)(u - (long)t * a.KT);
        const int kb = (int)min((long)a.KT, (long)ka + (ue - u));
        const int bt = t / a.Tb, tl = t - bt * a.Tb;   // product of the batch, its tile
        const int m0 = (tl / a.tn) * TM;
        const int n0 = (tl % a.tn) * GT;
        const int nkt = kb - ka;
        const long cb = bt * a.sC;

        f16 acc[MI][2], crs[MI][2];
#pragma unroll
        for (int i = 0; i < MI; i++)
#pragma unroll
            for (int j = 0; j < 2; j++)
#pragma unroll
                for (int e = 0; e < 16; e++)
                    acc[i][j][e] = crs[i][j][e] = 0.0f;

        // (LDS is free here: the previous segment's last reads precede its
        // final barrier.)
        SA sa;
        SB sb;
        sa.begin(a.A + bt * a.sA, a.lda, m0, a.Mc);
        sb.begin(a.B + bt * a.sB, a.ldb, n0, a.Nc);
        int k0 = ka * GKT;   // first k of the tile in registers
        sa.fetch_all(k0, a.lda, a.K, a.Kc);
        sb.fetch_all(k0, a.ldb, a.K, a.Kc);
        auto tail = [&]() {
            if (k0 + GKT > a.K) {
                sa.tail(k0, a.K);
                sb.tail(k0, a.K);
            }
        };
        // pair x of the tile in registers to LDS stage L; a load group whose
        // last pair has gone is refilled from the next k-tile
        auto split = [&](int x, int quarter) {
            if (x < SA::NP)
                sa.split(x, quarter);
            else if (x < SA::NP + SB::NP)
                sb.split(x - SA::NP, quarter);
        };
        auto put = [&](int x, char* L) {
            if (x < SA::NP) {
                sa.put(x, L);
                if ((x + 1) % SA::UL == 0)
                    sa.fetch(x / SA::UL, k0 + GKT, a.lda, a.K, a.Kc);
            } else if (x < SA::NP + SB::NP) {
                sb.put(x - SA::NP, L + 3 * SA::PLANE);
                if ((x - SA::NP + 1) % SB::UL == 0)
                    sb.fetch((x - SA::NP) / SB::UL, k0 + GKT, a.ldb, a.K, a.Kc);
            }
        };
        tail();
#pragma unroll
        for (int x = 0; x < 12; x++) {
#pragma unroll
            for (int q = 0; q < 4; q++)
                split(x, q);
            put(x, lds);
        }
        k0 += GKT;
        __syncthreads();

        for (int kt = 0; kt < nkt; kt++) {
            const char* LA = lds + (kt & 1) * STAGE + wm * (GKT * 2);
            const char* LB = lds + (kt & 1) * STAGE + 3 * SA::PLANE + wn * (GKT * 2);
            char* LN = lds + ((kt & 1) ^ 1) * STAGE;
            tail();
            b8 fa[2][3][MI], fb[2][3][2];
            auto read_a = [&](int s, int p) {
#pragma unroll
                for (int i = 0; i < MI; i++)
                    fa[s][p][i] = *reinterpret_cast<const b8*>(LA + p * SA::PLANE + i * 2048 + fs[s]);
            };
            auto read_b = [&](int s, int p) {
#pragma unroll
                for (int j = 0; j < 2; j++)
                    fb[s][p][j] = *reinterpret_cast<const b8*>(LB + p * SB::PLANE + j * 2048 + fs[s]);
            };
            read_a(0, 0);
            read_b(0, 0);
            // Twelve stages (two 16-wide k-steps, six products each): a
            // stage's MFMAs, one pair of the next tile's split between them,
            // and the fragments that the following stages need requested.
#pragma unroll
            for (int x = 0; x < 12; x++) {
                const int s = x / 6, y = x % 6;
                constexpr int pa[6] = {0, 1, 2, 0, 1, 0}, pb[6] = {0, 0, 0, 1, 1, 2};
                if (y < 2) {
                    read_a(s, y + 1);
                } else if (y < 4) {
                    read_b(s, y - 1);
                } else if (y == 4 && s == 0) {
                    read_a(1, 0);
                    read_b(1, 0);
                }
#pragma unroll
                for (int q = 0; q < 2 * MI; q++) {
                    f16& d = y == 0 ? acc[q >> 1][q & 1] : crs[q >> 1][q & 1];
                    d = mfma32b(fb[s][pb[y]][q & 1], fa[s][pa[y]][q >> 1], d);
                    split(x, MI == 2 ? q : 2 * q);
                    if (MI == 1)
                        split(x, 2 * q + 1);
                    __builtin_amdgcn_sched_barrier(0);
                }
                put(x, LN);
            }
            k0 += GKT;
            __syncthreads();
        }

        // lane (l32, g), accumulator (i, j), group q: tile row wm + 32i + l32,
        // columns wn + 32j + 8q + 4g .. +3.  A piece of a tile shared with
        // neighbouring runs goes to slot 0 if it opens this run, else slot 1
        // (then it closes the run).
#pragma unroll
        for (int q = 0; q < 2 * MI; q++) {
            settle(acc[q >> 1][q & 1]);
            settle(crs[q >> 1][q & 1]);
        }
        const bool whole = ka == 0 && kb == a.KT;
        float* P = a.part + ((long)2 * blockIdx.x + (u == ub ? 0 : 1)) * (TM * GT);
#pragma unroll
        for (int i = 0; i < MI; i++) {
            const int tr = wm + 32 * i + l32;
#pragma unroll
            for (int j = 0; j < 2; j++)
#pragma unroll
                for (int q = 0; q < 4; q++) {
                    const int tc = wn + 32 * j + 8 * q + 4 * g;
                    f4 v;
#pragma unroll
                    for (int e = 0; e < 4; e++)
                        v[e] = bf3_join(acc[i][j][4 * q + e], crs[i][j][4 * q + e]);
                    if (!whole)
                        *reinterpret_cast<f4*>(P + tr * GT + tc) = v;
                    else if (m0 + tr < a.M && n0 + tc < a.N)
                        epi_apply<EPI>(v, cb + (long)(m0 + tr) * a.ldc + n0 + tc, a.C, a.G, a.pre);
                }
        }
        u += nkt;
    }
}

// Tiles whose units span more than one run: sum the pieces in run order and
// apply the epilogue.  Four workgroups per 128 rows (32 rows each, four float4
// per thread, so the pieces' loads of many tiles are in flight at once);
// whole tiles return at once.
template <int EPI, int MI>
__global__ __launch_bounds__(256) void ffn_fixup_kernel(GemmArgs a)
{
    constexpr int TM = 128 * MI;
    const int t = (int)(blockIdx.x / (4 * MI)), part = (int)(blockIdx.x % (4 * MI));
    const long u0 = (long)t * a.KT;
    const int wa = sk_owner(a.U, a.P, u0);
    const int wb = sk_owner(a.U, a.P, u0 + a.KT - 1);
    if (wa == wb)
        return;
    // thread's float4s: q = 1024 part + threadIdx.x + 256 e: tile row q / 32,
    // column 4 (q % 32)
    constexpr int NE = 4;
    f4 v[NE];
#pragma unroll
    for (int e = 0; e < NE; e++)
        v[e] = f4zero();
#pragma unroll 4
    for (int w = wa; w <= wb; w++) {   // (P <= U: no run is empty)
        const long b = sk_begin(a.U, a.P, w);
        const float* src = a.part + ((long)2 * w + (b >= u0 ? 0 : 1)) * (TM * GT) + (long)part * 4096;
        f4 x[NE];
#pragma unroll
        for (int e = 0; e < NE; e++)
            x[e] = *reinterpret_cast<const f4*>(src + (threadIdx.x + 256 * e) * 4);
#pragma unroll
        for (int e = 0; e < NE; e++)
            v[e] += x[e];
    }
    const int bt = t / a.Tb, tl = t - bt * a.Tb;
    const int m0 = (tl / a.tn) * TM;
    const int n0 = (tl % a.tn) * GT;
    const long cb = bt * a.sC;
#pragma unroll
    for (int e = 0; e < NE; e++) {
        const int q = part * 1024 + threadIdx.x + 256 * e;
        const int row = m0 + (q >> 5), col = n0 + (q & 31) * 4;
        if (row < a.M && col < a.N)
            epi_apply<EPI>(v[e], cb + (long)row * a.ldc + col, a.C, a.G, a.pre);
    }
}

static int dev_cus()
{
    int cus = 256, dev = 0;
    if (hipGetDevice(&dev) == hipSuccess)
        (void)hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev);
    return cus;
}

// How one product (or a batch of them) is cut: tile height 128 mi, P runs.
struct GemmPlan {
    int mi, P;
    bool split;   // some tile is cut by a run boundary
};

// The cheapest of: 256- and 128-row tiles, each as one run a tile, as equal
// runs on every compute unit, and as s runs a tile.  Costs in microseconds,
// fitted to MI355X timings of this kernel: a k-tile 2.6 (256 rows) or 1.5,
// each tile a run touches 3 (first loads, epilogue), a fix-up launch 4 plus
// its pieces' write and read at 6 TB/s and 0.4 for each piece of one tile,
// which it adds one after another.  (Always one equal run a compute unit: a
// [40][128] x [128][512] FFN step cut its 4-k-tile products into 64 KB pieces
// of one k-tile each.)
static GemmPlan gemm_plan(int M, int N, int K, int batch)
{
    const long cus = dev_cus();
    const long KT = (K + GKT - 1) / GKT;
    GemmPlan best = {2, 1, false};
    double cost = 1e30;
    for (int mi = 1; mi <= 2; mi++) {
        const long TM = 128 * mi;
        const long T = (long)std::max(batch, 1) * ((M + TM - 1) / TM) * ((N + GT - 1) / GT);
        const double unit = mi == 2 ? 2.6 : 1.5, piece = TM * GT * 4 * 2 / 6e6;
        auto consider = [&](long P, double busy, long pieces, long per_tile) {
            const double c = busy + (pieces ? 4.0 + pieces * piece + 0.4 * per_tile : 0.0);
            if (c < cost) {
                cost = c;
                best = {mi, (int)P, pieces != 0};
            }
        };
        if (T <= 0x7fffffff)
            consider(T, (double)((T + cus - 1) / cus) * (KT * unit + 3.0), 0, 0);
        for (long s = 2; s <= KT && T * s <= cus; s++)
            consider(T * s, (double)((KT + s - 1) / s) * unit + 3.0, T * s, s);
        if (T * KT > cus && T * KT % (cus * KT) != 0) {
            const long L = (T * KT + cus - 1) / cus;
            const long touched = L / KT + 1 + (L % KT != 0);
            long pieces = 0, last = -1;   // one a cut, one more a tile that is cut
            for (int w = 1; w < cus; w++) {
                const long b = sk_begin(T * KT, (int)cus, w);
                if (b % KT != 0) {
                    pieces += 1 + (b / KT != last);
                    last = b / KT;
                }
            }
            consider(cus, L * unit + 3.0 * touched, pieces, (KT + L - 1) / L + 1);
        }
    }
    return best;
}

// Room for any plan of these sizes: two pieces a run, a run for every compute
// unit or unit of work.  (It grows with the batch, so one sized for a group of
// products also serves a smaller last group.)
size_t ffn_gemm_ws_floats(int M, int N, int K, int batch)
{
    const long KT = (K + GKT - 1) / GKT, tn = (N + GT - 1) / GT;
    long fl = 0;
    for (long TM = 128; TM <= 256; TM += 128) {
        const long U = (long)std::max(batch, 1) * ((M + TM - 1) / TM) * tn * KT;
        fl = std::max(fl, 2 * std::min<long>(dev_cus(), U) * TM * GT);
    }
    return (size_t)fl;
}

template <bool AK, bool BK, int EPI, int MI>
static void launch_main(dim3 grid, hipStream_t st, const GemmArgs& a)
{
    CXG_LAUNCH((ffn_gemm_kernel<AK, BK, EPI, MI>), grid, dim3(512), 0, st, a);
}

template <int EPI, int MI>
static void launch_layout(const FfnGemm& op, dim3 grid, hipStream_t st, const GemmArgs& a)
{
    if (op.ak && op.bk)
        launch_main<true, true, EPI, MI>(grid, st, a);
    else if (op.ak)
        launch_main<true, false, EPI, MI>(grid, st, a);
    else
        launch_main<false, false, EPI, MI>(grid, st, a);
}

template <int EPI>
static hipError_t launch_gemm(const FfnGemm& op, hipStream_t st, const GemmArgs& a,
                              const GemmPlan& plan)
{
    const int mi = plan.mi;
    {
        ProfScope ps(st, "ffn_gemm");
        const dim3 grid((unsigned)a.P);
        if (mi == 2)
            launch_layout<EPI, 2>(op, grid, st, a);
        else
            launch_layout<EPI, 1>(op, grid, st, a);
    }
    hipError_t e = hipGetLastError();
    if (e != hipSuccess)
        return e;
    if (!plan.split)
        return hipSuccess;
    ProfScope ps(st, "ffn_fixup");
    const dim3 grid((unsigned)(a.T * 4 * mi));
    if (mi == 2)
        CXG_LAUNCH((ffn_fixup_kernel<EPI, 2>), grid, dim3(256), 0, st, a);
    else
        CXG_LAUNCH((ffn_fixup_kernel<EPI, 1>), grid, dim3(256), 0, st, a);
    return hipGetLastError();
}

hipError_t ffn_gemm_launch(const FfnGemm& op, float* ws, hipStream_t st)
{
    if (op.M <= 0 || op.N <= 0 || op.K <= 0)
        return hipSuccess;
    const GemmPlan plan = gemm_plan(op.M, op.N, op.K, op.batch);
    if ((!op.ak && op.bk) || ws == nullptr)
        return hipErrorInvalidValue;   // no caller needs A row-contiguous with B k-contiguous
    const int TM = 128 * plan.mi;
    GemmArgs a;
    a.A = op.A;
    a.B = op.B;
    a.C = op.C;
    a.G = op.G;
    a.pre = op.pre;
    a.part = ws;
    a.lda = op.lda;
    a.ldb = op.ldb;
    a.ldc = op.ldc;
    a.M = op.M;
    a.N = op.N;
    a.K = op.K;
    a.Mc = op.Mc > 0 ? op.Mc : op.M;
    a.Nc = op.Nc > 0 ? op.Nc : op.N;
    a.Kc = op.Kc > 0 ? op.Kc : op.K;
    a.tn = (op.N + GT - 1) / GT;
    a.Tb = ((op.M + TM - 1) / TM) * a.tn;
    a.sA = op.sA;
    a.sB = op.sB;
    a.sC = op.sC;
    a.T = std::max(op.batch, 1) * a.Tb;
    a.KT = (op.K + GKT - 1) / GKT;
    a.U = (long)a.T * a.KT;
    a.P = plan.P;
    switch (op.epi) {
    case FFN_EPI_GELU: return launch_gemm<FFN_EPI_GELU>(op, st, a, plan);
    case FFN_EPI_DGELU: return launch_gemm<FFN_EPI_DGELU>(op, st, a, plan);
    case FFN_EPI_ACCUM: return launch_gemm<FFN_EPI_ACCUM>(op, st, a, plan);
    default: return launch_gemm<FFN_EPI_STORE>(op, st, a, plan);
    }
}

} // namespace cxg
