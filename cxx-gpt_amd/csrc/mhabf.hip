// mhabf.hip -- causal softmax multi-head attention with its FP32 products on
// the bf16 matrix unit (split operands, bf3.hpp).
//
// The same functions as mha.hip's tile kernels for heads of 17 to 96 columns
// (16-byte aligned rows, no RoPE); mha.hip's dispatch says which shapes come
// here.  Tensors (B*S, H*Dh) row-major, head h of row r at [(r*H + h)*Dh, +Dh);
// lse, Di [B*H][S].
//
// LDS.  A streamed tile (K and V rows forward, Q and dO rows backward) is split
// once, on its way from registers to LDS, into three planes of bf16 rows.  Each
// plane serves both as a product's row operand and, through the transposing
// read, as its column operand (bf3.hpp), so no second, transposed copy is
// formed.
//
// MFMA 32x32x16: lane (l32 = l % 32, g = l / 32) holds A[l32][8g + e], B[8g + e]
// [l32] and D[8 (r / 4) + 4g + r % 4][l32].  A score accumulator's registers
// 8t .. 8t+7 are the B operand of the next product's k-step t as they stand if
// that k-step's slot (g, e) is row 16t + 8 (e / 4) + 4g + e % 4: the transposing
// reads take rows in that order.
#include "bf3.hpp"
#include "common.hpp"
#include "launch.hpp"

#include <math.h>

namespace cxg {

constexpr float kLazy = 8.0f;   // log2 units a score may exceed its row's reference by
constexpr float kBig = 3.0e38f;

// A cross sum that an infinity or NaN in an operand has made NaN: any finite
// value, since the main sum is then not finite and stands (bf3.hpp).
__device__ __forceinline__ float tame(float x) { return __builtin_amdgcn_fmed3f(x, -kBig, kBig); }

// ROWS rows of one head held in registers between load and split: thread t of
// NT takes 8-column chunks t, t + NT, ... (2 NK a row).
template <int NK, int ROWS, int NT>
struct RowTile {
    static constexpr int DHP = NK <= 2 ? 32 : NK <= 4 ? 64 : NK <= 6 ? 96 : 128;
    static constexpr int CPR = 2 * NK;                        // chunks a row
    static constexpr int U = (ROWS * CPR + NT - 1) / NT;      // chunks a thread
    static constexpr bool FULL = ROWS * CPR % NT == 0;
    static constexpr int PL = ROWS * DHP * 2;                 // bytes of a plane
    float v[U][8];

    // voff[u]: byte offsets of the thread's chunks in the tile (past the
    // descriptor's range where the columns are past Dh: read as 0)
    __device__ __forceinline__ static void offsets(unsigned (&voff)[U][2], int ld, int Dh)
    {
#pragma unroll
        for (int u = 0; u < U; u++) {
            const int i = threadIdx.x + u * NT, row = i / CPR, c = 8 * (i % CPR);
            const bool in = FULL || row < ROWS;
#pragma unroll
            for (int q = 0; q < 2; q++)
                voff[u][q] = in && c + 4 * q < Dh ? (unsigned)(row * ld + c + 4 * q) * 4u : kDropOffset;
        }
    }
    __device__ __forceinline__ void load(__amdgpu_buffer_rsrc_t r, const unsigned (&voff)[U][2],
                                         unsigned soff)
    {
#pragma unroll
        for (int u = 0; u < U; u++)
#pragma unroll
            for (int q = 0; q < 2; q++) {
                const f4 x = buffer_load_f4s(r, voff[u][q], soff);
#pragma unroll
                for (int e = 0; e < 4; e++)
                    v[u][4 * q + e] = x[e];
            }
    }
    __device__ __forceinline__ void put(char* L) const
    {
#pragma unroll
        for (int u = 0; u < U; u++) {
            const int i = threadIdx.x + u * NT, row = i / CPR, c = i % CPR;
            if (!FULL && row >= ROWS)
                break;
            b8 h, m, l;
            split8(v[u], h, m, l);
            char* at = L + chunk_off<DHP>(row, c);
            *reinterpret_cast<b8*>(at) = h;
            *reinterpret_cast<b8*>(at + PL) = m;
            *reinterpret_cast<b8*>(at + 2 * PL) = l;
        }
    }
};

// ---------------------------------------------------------------------------
// forward
// ---------------------------------------------------------------------------
// A workgroup owns 32 NQ query rows of one head; wave (qg, ks) owns queries
// 32 qg .. +31 and keys 32 ks .. +31 of every 32 NS-key tile, with its own
// online-softmax state (merged through LDS at the end).  Scores transposed
// (S^T = K Q^T), so a lane holds one query; Q scaled to log2 units and split
// into registers once.  DB: two LDS stages and one barrier a tile, else one
// stage and two.
template <int NK, int NQ, int NS, bool DB, bool WRITE_O>
__global__ __launch_bounds__(64 * NQ * NS) void mhabf_fwd_kernel(
    const float* __restrict__ Q, const float* __restrict__ K, const float* __restrict__ V,
    float* __restrict__ O, float* __restrict__ lse, int S, int H, int Dh, int BH, int nqb,
    float qscale)
{
    constexpr int NT = 64 * NQ * NS, KT = 32 * NS, BM = 32 * NQ;
    typedef RowTile<NK, KT, NT> T;
    constexpr int DHP = T::DHP, PL = T::PL, NO = (NK + 1) / 2;
    constexpr int STAGE = (WRITE_O ? 6 : 3) * PL;
    constexpr int REC = WRITE_O ? 16 * NO + 2 : 2;   // floats a lane: O, m, l
    constexpr int MERGE = NS * NQ * REC * 64 * 4;
    constexpr int LDS = (DB ? 2 : 1) * STAGE > MERGE ? (DB ? 2 : 1) * STAGE : MERGE;
    __shared__ __attribute__((aligned(16))) char lds[LDS];

    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int l32 = lane & 31, g = lane >> 5;
    const int qg = wave % NQ, ks = wave / NQ;

    const int job = blockIdx.x, qb = nqb - 1 - job / BH, bh = job % BH;
    const int b = bh / H, h = bh % H, ld = H * Dh;
    const long base = ((long)b * S * H + h) * Dh;
    const unsigned range = (unsigned)(((long)(S - 1) * ld + Dh) * 4);
    const __amdgpu_buffer_rsrc_t rq = buf_rsrc_n(Q + base, range), rk = buf_rsrc_n(K + base, range),
                                 rv = buf_rsrc_n((WRITE_O ? V : K) + base, range);
    const int q0 = qb * BM, qw = q0 + 32 * qg;   // workgroup's, wave's first query
    const int nkt = (min(q0 + BM, S) + KT - 1) / KT;

    unsigned voff[T::U][2];
    T::offsets(voff, ld, Dh);
    T tk, tv;
    tk.load(rk, voff, 0);
    if (WRITE_O)
        tv.load(rv, voff, 0);
    // Q as B operand: k-step k: columns 16k + 8g .. +7 of this lane's query
    b8 fq[NK][3];
    {
        float x[NK][8];
#pragma unroll
        for (int k = 0; k < NK; k++)
#pragma unroll
            for (int q = 0; q < 2; q++) {
                const int c = 16 * k + 8 * g + 4 * q;
                const f4 y = buffer_load_f4(rq, c < Dh ? (unsigned)((qw + l32) * ld + c) * 4u : kDropOffset);
#pragma unroll
                for (int e = 0; e < 4; e++)
                    x[k][4 * q + e] = y[e] * qscale;
            }
#pragma unroll
        for (int k = 0; k < NK; k++)
            split8(x[k], fq[k][0], fq[k][1], fq[k][2]);
    }

    f16 o[NO], oc[NO];   // O^T: column 32 ob + 8 (r/4) + 4g + r%4 of this lane's query
#pragma unroll
    for (int i = 0; i < NO; i++)
        o[i] = oc[i] = f16zero();
    float m = 0.0f, l = 0.0f;   // reference (log2 units), this lane's part of the sum
    bool fresh = true;          // no block seen: the reference is not set yet

    auto put = [&](char* L) {
        tk.put(L);
        if (WRITE_O)
            tv.put(L + 3 * PL);
    };
    auto load = [&](int kt) {
        const unsigned so = (unsigned)(kt * KT * ld) * 4u;
        tk.load(rk, voff, so);
        if (WRITE_O)
            tv.load(rv, voff, so);
    };
    if (DB) {
        put(lds);
        if (nkt > 1)
            load(1);
        __syncthreads();
    }
    for (int kt = 0; kt < nkt; kt++) {
        char* L = lds + (DB ? (kt & 1) * STAGE : 0);
        if (!DB) {
            put(L);
            __syncthreads();
            if (kt + 1 < nkt)
                load(kt + 1);
        }
        const int k0 = kt * KT + 32 * ks;   // wave's first key
        if (k0 <= qw && qw < S) {           // else wholly above the diagonal
            // products before the other waves' splitting ([2, 4096, 12, 64] 299 -> 287 us)
            __builtin_amdgcn_s_setprio(1);
            const int row = 32 * ks + l32;
            f16 s = f16zero();
            b8 kh[NK];
#pragma unroll
            for (int k = 0; k < NK; k++) {
                b8 fk[3];
#pragma unroll
                for (int p = 0; p < 3; p++)
                    fk[p] = read_row<DHP>(L + p * PL, row, 2 * k + g);
                kh[k] = fk[0];
#pragma unroll
                for (int x = 0; x < 5; x++)
                    s = mfma32b(fk[kPa[x]], fq[k][kPb[x]], s);
            }
            settle(s);
#pragma unroll
            for (int r = 0; r < 16; r++)
                s[r] = tame(s[r]) - m;
#pragma unroll
            for (int k = 0; k < NK; k++)
                s = mfma32b(kh[k], fq[k][0], s);
            settle(s);
            if (k0 == qw) {   // the diagonal block
#pragma unroll
                for (int r = 0; r < 16; r++)
                    s[r] = 8 * (r >> 2) + 4 * g + (r & 3) <= l32 ? s[r] : -INFINITY;
            }
            float mx = fmaxf(s[0], s[1]);
#pragma unroll
            for (int r = 2; r < 16; r += 2)
                mx = fmaxf(fmaxf(mx, s[r]), s[r + 1]);
            if (fresh || __any(mx > kLazy)) {
                mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
                float d = fresh ? mx : fmaxf(mx, 0.0f);
                d = d == -INFINITY ? 0.0f : d;
                const float f = fast_exp2(-d);
                m += d;
                l *= f;
#pragma unroll
                for (int r = 0; r < 16; r++)
                    s[r] -= d;
                if (!fresh) {
#pragma unroll
                    for (int i = 0; i < NO; i++)
#pragma unroll
                        for (int r = 0; r < 16; r++) {
                            o[i][r] *= f;
                            oc[i][r] *= f;
                        }
                }
                fresh = false;
            }
#pragma unroll
            for (int r = 0; r < 16; r++)
                s[r] = fast_exp2(s[r]);
#pragma unroll
            for (int r = 0; r < 16; r++)
                l += s[r];
            if (WRITE_O) {
#pragma unroll
                for (int t = 0; t < 2; t++) {
                    float pv[8];
#pragma unroll
                    for (int e = 0; e < 8; e++)
                        pv[e] = s[8 * t + e];
                    b8 fp[3];
                    split8(pv, fp[0], fp[1], fp[2]);
#pragma unroll
                    for (int i = 0; i < NO; i++) {
                        b8 fv[3];
#pragma unroll
                        for (int p = 0; p < 3; p++)
                            fv[p] = read_tr<DHP>(L + (3 + p) * PL, 32 * ks + 16 * t, 32 * i, lane);
                        o[i] = mfma32b(fv[0], fp[0], o[i]);
#pragma unroll
                        for (int x = 0; x < 5; x++)
                            oc[i] = mfma32b(fv[kPa[x]], fp[kPb[x]], oc[i]);
                    }
                }
            }
        }
        __builtin_amdgcn_s_setprio(0);
        if (DB && kt + 1 < nkt) {
            put(lds + ((kt & 1) ^ 1) * STAGE);
            if (kt + 2 < nkt)
                load(kt + 2);
        }
        __syncthreads();
    }

    // merge the NS states: every wave leaves its own, then takes 1 / NS of the
    // columns of its queries
#pragma unroll
    for (int i = 0; i < NO; i++) {
        settle(o[i]);
        settle(oc[i]);
    }
    l += __shfl_xor(l, 32, 64);
    float* rec = reinterpret_cast<float*>(lds);
    auto slot = [&](int k, int grp) { return rec + ((k * NQ + qg) * REC * 64) + grp * 256 + lane * 4; };
    auto stat = [&](int k, int i) { return rec + ((k * NQ + qg) * REC + (REC - 2) + i) * 64 + lane; };
    *stat(ks, 0) = fresh ? -INFINITY : m;
    *stat(ks, 1) = l;
    if (WRITE_O) {
#pragma unroll
        for (int i = 0; i < NO; i++)
#pragma unroll
            for (int q = 0; q < 4; q++) {
                f4 v;
#pragma unroll
                for (int e = 0; e < 4; e++)
                    v[e] = bf3_join(o[i][4 * q + e], oc[i][4 * q + e]);
                *reinterpret_cast<f4*>(slot(ks, 4 * i + q)) = v;
            }
    }
    __syncthreads();
    float M = *stat(0, 0);
#pragma unroll
    for (int k = 1; k < NS; k++)
        M = fmaxf(M, *stat(k, 0));
    float w[NS], Ls = 0.0f;
#pragma unroll
    for (int k = 0; k < NS; k++) {
        const float mk = *stat(k, 0);
        w[k] = mk == -INFINITY ? 0.0f : fast_exp2(mk - M);   // a split that saw no key
        Ls += w[k] * *stat(k, 1);
    }
    const int t = qw + l32;
    if (t >= S)
        return;
    if (lse != nullptr && ks == 0 && g == 0)
        lse[(long)bh * S + t] = (M + fast_log2(Ls)) * kLn2;
    if (!WRITE_O)
        return;
    const float inv = 1.0f / Ls;
    float* orow = O + base + (long)t * ld;
#pragma unroll
    for (int j = 0; j < 4 * NO / NS; j++) {
        const int grp = ks * (4 * NO / NS) + j, c = 8 * grp + 4 * g;
        f4 v = f4zero();
#pragma unroll
        for (int k = 0; k < NS; k++)
            if (w[k] != 0.0f)
                v += *reinterpret_cast<const f4*>(slot(k, grp)) * w[k];
        if (c < Dh)
            *reinterpret_cast<f4*>(orow + c) = v * inv;
    }
}

template <int NK, int NQ, int NS, bool DB>
static hipError_t fwd_go(const float* Q, const float* K, const float* V, float* O, float* lse,
                         int B, int S, int H, int Dh, hipStream_t st)
{
    constexpr int BM = 32 * NQ;
    const int BH = B * H, nqb = (S + BM - 1) / BM;
    const float qscale = (1.0f / sqrtf((float)Dh)) * kLog2e;
    const dim3 grid((unsigned)((long)nqb * BH)), block(64 * NQ * NS);
    if (O != nullptr) {
        ProfScope ps(st, "mha_fwd");
        CXG_LAUNCH((mhabf_fwd_kernel<NK, NQ, NS, DB, true>), grid, block, 0, st, Q, K, V, O, lse, S, H,
                   Dh, BH, nqb, qscale);
    } else {
        ProfScope ps(st, "mha_stats");
        CXG_LAUNCH((mhabf_fwd_kernel<NK, NQ, NS, DB, false>), grid, block, 0, st, Q, K, V, O, lse, S,
                   H, Dh, BH, nqb, qscale);
    }
    return hipGetLastError();
}

static inline bool al16(const void* p) { return ((uintptr_t)p & 15u) == 0; }

static bool mhabf_ok(int S, int H, int Dh, const float* Q, const float* K, const float* V, const float* O)
{
    return Dh > 16 && Dh <= 96 && Dh % 4 == 0 && (long)S * H * Dh * 4 < (1L << 31) - 64 &&
           al16(Q) && al16(K) && al16(V) && al16(O);
}

// Which forward, by 64-row query tiles against compute units (time in us, this
// file's kernel against mha.hip's, MI355X):
//   heads past 64 columns: all but very short, many sequences ([4, 333, 10, 80]
//     23.4 / 35.3; [32, 64, 16, 96] 19.7 / 18.1);
//   at most one tile a unit: 64 queries a workgroup, keys over four waves, so
//     that a unit's four SIMDs share one tile ([1, 256, 8, 64] 11.3 / 12.4,
//     [1, 4096, 4, 64] 94.8 / 137.4, [2, 1000, 8, 32] 19.1 / 21.8; below 96
//     rows there is nothing to share);
//   more than two rounds and 256 rows or more: 128 queries a workgroup, so
//     that a key tile is split once for twice the products ([2, 4096, 12, 64]
//     287 / 402, [16, 384, 12, 64] 42.6 / 45.2, [16, 512, 12, 32] 30.3 / 37.7;
//     shorter ones lose: [32, 128, 16, 64] 25.7 / 22.9);
//   between one and two rounds mha.hip's paired jobs are the faster
//     ([8, 256, 12, 64] 16.8 / 15.0).
enum { BF_NONE = 0, BF_SHARED, BF_LONG };

static int fwd_kind(int B, int S, int H, int Dh)
{
    const long tiles = (long)B * H * ((S + 63) / 64), cus = mha_device_cus();
    if (Dh > 64)
        return S > 64 || tiles <= cus ? BF_SHARED : BF_NONE;
    if (tiles <= cus)
        return S >= 96 ? BF_SHARED : BF_NONE;
    return tiles > 2 * cus && S >= 256 ? BF_LONG : BF_NONE;
}

bool mhabf_fwd_use(int B, int S, int H, int Dh, const float* Q, const float* K, const float* V,
                   const float* O)
{
    return mhabf_ok(S, H, Dh, Q, K, V, O) && fwd_kind(B, S, H, Dh) != BF_NONE;
}

hipError_t mhabf_fwd_launch(const float* Q, const float* K, const float* V, float* O, float* lse,
                            int B, int S, int H, int Dh, hipStream_t st)
{
    const bool lng = fwd_kind(B, S, H, Dh) == BF_LONG;
    if (Dh > 64)
        return fwd_go<6, 2, 2, false>(Q, K, V, O, lse, B, S, H, Dh, st);
    if (Dh > 32)
        return lng ? fwd_go<4, 4, 2, true>(Q, K, V, O, lse, B, S, H, Dh, st)
                   : fwd_go<4, 2, 4, false>(Q, K, V, O, lse, B, S, H, Dh, st);
    return lng ? fwd_go<2, 4, 2, true>(Q, K, V, O, lse, B, S, H, Dh, st)
               : fwd_go<2, 2, 4, false>(Q, K, V, O, lse, B, S, H, Dh, st);
}

// ---------------------------------------------------------------------------
// backward
// ---------------------------------------------------------------------------
// A workgroup owns 32 NKB key rows of one head and streams 32 NQB-row query
// tiles; wave (kb, qs) owns the 32 x 32 block of keys 32 kb, queries 32 qs of
// each: S and dP (a lane per key), P = exp2(S - lse), dS = P (dP - Di), then
// dV^T += dO^T P and dK^T += Q^T dS in registers, P and dS being the products'
// operands as they stand.  dS goes to LDS as planes of [key][query]; after a
// barrier every wave takes its share of dQ = dS K (both operands through the
// transposing read) into float atomics, and splits its part of the next query
// tile.  dQ is zero and Di ready before the launch.
template <int NK, int NKB, int NQB, bool ALIAS>
__global__ __launch_bounds__(64 * NKB * NQB, ALIAS ? 2 : 1) void mhabf_bwd_kernel(
    const float* __restrict__ Q, const float* __restrict__ K, const float* __restrict__ V,
    const float* __restrict__ dO, const float* __restrict__ lse, const float* __restrict__ Di,
    float* __restrict__ dQ, float* __restrict__ dK, float* __restrict__ dV, int S, int H, int Dh,
    int BH, float scale)
{
    constexpr int NW = NKB * NQB, NT = 64 * NW, BN = 32 * NKB, BM = 32 * NQB;
    static_assert(BM == 64, "the dS planes' rows");
    typedef RowTile<NK, BM, NT> T;
    typedef RowTile<NK, BN, NT> TK;
    constexpr int DHP = T::DHP, PQ = T::PL, PK = TK::PL, PS = BN * BM * 2, NO = (NK + 1) / 2;
    // ALIAS: dS takes dO's place while dQ is formed
    constexpr int OFF_DO = 3 * PQ, DOB = ALIAS && PS > PQ ? 3 * PS : 3 * PQ;
    constexpr int OFF_K = OFF_DO + DOB, OFF_ST = OFF_K + 3 * PK;
    constexpr int OFF_DS = ALIAS ? OFF_DO : OFF_ST + 2 * BM * 4;
    constexpr int END = ALIAS ? OFF_ST + 2 * BM * 4 : OFF_DS + 3 * PS;
    constexpr int REC = 2 * NO * 16 * 64;   // floats a wave leaves for the reduction
    constexpr int LDS = END > NW * REC * 4 ? END : NW * REC * 4;
    __shared__ __attribute__((aligned(16))) char lds[LDS];
    float* const st = reinterpret_cast<float*>(lds + OFF_ST);   // lse (log2), Di (scaled)

    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int l32 = lane & 31, g = lane >> 5;
    const int kb = wave % NKB, qs = wave / NKB;

    const int job = blockIdx.x, bh = job % BH, k0 = job / BH * BN;
    const int b = bh / H, h = bh % H, ld = H * Dh;
    const long base = ((long)b * S * H + h) * Dh;
    const unsigned range = (unsigned)(((long)(S - 1) * ld + Dh) * 4);
    const __amdgpu_buffer_rsrc_t rq = buf_rsrc_n(Q + base, range), rk = buf_rsrc_n(K + base, range),
                                 rv = buf_rsrc_n(V + base, range), rdo = buf_rsrc_n(dO + base, range),
                                 rdq = buf_rsrc_n(dQ + base, range);
    const int qt0 = k0 / BM, nqt = (S + BM - 1) / BM;

    unsigned voff[T::U][2];
    T::offsets(voff, ld, Dh);
    T tq, tdo;
    float st0 = 0.0f;   // threads below 2 BM: this tile's lse or Di
    auto load = [&](int qt) {
        const unsigned so = (unsigned)(qt * BM * ld) * 4u;
        tq.load(rq, voff, so);
        tdo.load(rdo, voff, so);
        if (threadIdx.x < 2 * BM) {
            const int t = qt * BM + (threadIdx.x & (BM - 1));
            const float* src = threadIdx.x < BM ? lse : Di;
            st0 = t < S ? src[(long)bh * S + t] : (threadIdx.x < BM ? 1e30f : 0.0f);
        }
    };
    auto put = [&]() {
        tq.put(lds);
        tdo.put(lds + OFF_DO);
        if (threadIdx.x < 2 * BM)
            st[threadIdx.x] = st0 * (threadIdx.x < BM ? kLog2e : scale);
    };
    load(qt0);
    {   // K planes, once
        TK t;
        unsigned vk[TK::U][2];
        TK::offsets(vk, ld, Dh);
        t.load(rk, vk, (unsigned)(k0 * ld) * 4u);
        t.put(lds + OFF_K);
    }
    // V rows as B operand, scaled: k-step k: columns 16k + 8g .. +7 of the key
    b8 fv[NK][3];
#pragma unroll
    for (int k = 0; k < NK; k++) {
        float x[8];
#pragma unroll
        for (int q = 0; q < 2; q++) {
            const int c = 16 * k + 8 * g + 4 * q;
            const f4 y = buffer_load_f4(
                rv, c < Dh ? (unsigned)((k0 + 32 * kb + l32) * ld + c) * 4u : kDropOffset);
#pragma unroll
            for (int e = 0; e < 4; e++)
                x[4 * q + e] = y[e] * scale;
        }
        split8(x, fv[k][0], fv[k][1], fv[k][2]);
    }
    put();
    if (!ALIAS && qt0 + 1 < nqt)
        load(qt0 + 1);
    __syncthreads();

    f16 dk[NO], dv[NO];   // column 32 i + 8 (r/4) + 4g + r%4 of this lane's key
#pragma unroll
    for (int i = 0; i < NO; i++)
        dk[i] = dv[i] = f16zero();
    const float c2 = scale * kLog2e;

    for (int qt = qt0; qt < nqt; qt++) {
        const int qb = qt * BM + 32 * qs, kk = k0 + 32 * kb;   // the block's first query, key
        b8 fd[2][3];
        if (kk <= qb) {
            const int row = 32 * qs + l32;
            f16 s = f16zero(), dp = f16zero();
            {
                f16 sc = f16zero();
#pragma unroll
                for (int k = 0; k < NK; k++) {
                    b8 fq[3], fk[3];
#pragma unroll
                    for (int p = 0; p < 3; p++) {
                        fq[p] = read_row<DHP>(lds + p * PQ, row, 2 * k + g);
                        fk[p] = read_row<DHP>(lds + OFF_K + p * PK, 32 * kb + l32, 2 * k + g);
                    }
                    s = mfma32b(fq[0], fk[0], s);
#pragma unroll
                    for (int x = 0; x < 5; x++)
                        sc = mfma32b(fq[kPa[x]], fk[kPb[x]], sc);
                }
                settle(s);
                settle(sc);
#pragma unroll
                for (int q = 0; q < 4; q++) {
                    const f4 ls = *reinterpret_cast<const f4*>(st + 32 * qs + 8 * q + 4 * g);
#pragma unroll
                    for (int e = 0; e < 4; e++)
                        s[4 * q + e] = fast_exp2(
                            __builtin_fmaf(s[4 * q + e] + tame(sc[4 * q + e]), c2, -ls[e]));
                }
            }
            {
                f16 dc = f16zero();
#pragma unroll
                for (int k = 0; k < NK; k++) {
                    b8 fo[3];
#pragma unroll
                    for (int p = 0; p < 3; p++)
                        fo[p] = read_row<DHP>(lds + OFF_DO + p * PQ, row, 2 * k + g);
                    dp = mfma32b(fo[0], fv[k][0], dp);
#pragma unroll
                    for (int x = 0; x < 5; x++)
                        dc = mfma32b(fo[kPa[x]], fv[k][kPb[x]], dc);
                }
                settle(dp);
                settle(dc);
                dp += dc;
            }
            if (kk == qb) {   // the diagonal block
#pragma unroll
                for (int r = 0; r < 16; r++)
                    s[r] = l32 <= 8 * (r >> 2) + 4 * g + (r & 3) ? s[r] : 0.0f;
            }
#pragma unroll
            for (int q = 0; q < 4; q++) {
                const f4 d = *reinterpret_cast<const f4*>(st + BM + 32 * qs + 8 * q + 4 * g);
#pragma unroll
                for (int e = 0; e < 4; e++)
                    dp[4 * q + e] = s[4 * q + e] * (dp[4 * q + e] - d[e]);
            }
#pragma unroll
            for (int t = 0; t < 2; t++) {
                float x[8];
                b8 fp[3];
#pragma unroll
                for (int e = 0; e < 8; e++)
                    x[e] = dp[8 * t + e];
                split8(x, fd[t][0], fd[t][1], fd[t][2]);
#pragma unroll
                for (int e = 0; e < 8; e++)
                    x[e] = s[8 * t + e];
                split8(x, fp[0], fp[1], fp[2]);
#pragma unroll
                for (int i = 0; i < NO; i++) {
                    b8 fo[3], fq[3];
#pragma unroll
                    for (int p = 0; p < 3; p++) {
                        fo[p] = read_tr<DHP>(lds + OFF_DO + p * PQ, 32 * qs + 16 * t, 32 * i, lane);
                        fq[p] = read_tr<DHP>(lds + p * PQ, 32 * qs + 16 * t, 32 * i, lane);
                    }
#pragma unroll
                    for (int x5 = 0; x5 < 5; x5++) {
                        dv[i] = mfma32b(fo[kPa[x5]], fp[kPb[x5]], dv[i]);
                        dk[i] = mfma32b(fq[kPa[x5]], fd[t][kPb[x5]], dk[i]);
                    }
                    dv[i] = mfma32b(fo[0], fp[0], dv[i]);
                    dk[i] = mfma32b(fq[0], fd[t][0], dk[i]);
                }
            }
        }
        if (ALIAS) {
            if (qt + 1 < nqt)
                load(qt + 1);
            __syncthreads();
        }
        if (kk <= qb) {
            // this lane's key row, queries 32 qs + 16 t + 8 u + 4 g .. +3
#pragma unroll
            for (int t = 0; t < 2; t++)
#pragma unroll
                for (int u = 0; u < 2; u++) {
                    const int q = 32 * qs + 16 * t + 8 * u + 4 * g;
                    char* at = lds + OFF_DS + chunk_off<64>(32 * kb + l32, q >> 3) + 8 * g;
#pragma unroll
                    for (int p = 0; p < 3; p++) {
                        const u4 w = __builtin_bit_cast(u4, fd[t][p]);
                        *reinterpret_cast<u2*>(at + p * PS) = (u2){w[2 * u], w[2 * u + 1]};
                    }
                }
        }
        __syncthreads();
        if (!ALIAS && qt + 1 < nqt) {
            put();
            if (qt + 2 < nqt)
                load(qt + 2);
        }
        // dQ: units (query block, 32 columns, share of the keys)
        constexpr int KSPL = (NQB * NO) % NW == 0 ? 1 : (2 * NQB * NO) % NW == 0 ? 2 : 4;
        static_assert(NQB * NO * KSPL % NW == 0 && NKB % KSPL == 0, "dQ shares");
#pragma unroll
        for (int n = 0; n < NQB * NO * KSPL / NW; n++) {
            const int u = wave + n * NW, i = u % NO, qd = u / NO % NQB, ksp = u / (NO * NQB);
            const int qbd = qt * BM + 32 * qd;
            f16 acc = f16zero();
            bool any = false;
#pragma unroll
            for (int j = 0; j < NKB / KSPL; j++) {
                const int kbd = ksp * (NKB / KSPL) + j;
                if (k0 + 32 * kbd > qbd)
                    continue;
                any = true;
#pragma unroll
                for (int t = 0; t < 2; t++) {
                    b8 fa[3], fb[3];
#pragma unroll
                    for (int p = 0; p < 3; p++) {
                        fa[p] = read_tr<64>(lds + OFF_DS + p * PS, 32 * kbd + 16 * t, 32 * qd, lane);
                        fb[p] = read_tr<DHP>(lds + OFF_K + p * PK, 32 * kbd + 16 * t, 32 * i, lane);
                    }
#pragma unroll
                    for (int x = 0; x < 5; x++)
                        acc = mfma32b(fa[kPa[x]], fb[kPb[x]], acc);
                    acc = mfma32b(fa[0], fb[0], acc);
                }
            }
            settle(acc);
            if (any) {   // lane: column 32 i + l32, queries qbd + 8 (r/4) + 4g + r%4
                const unsigned vo = 32 * i + l32 < Dh ? (unsigned)(4 * g * ld + 32 * i + l32) * 4u
                                                      : kDropOffset;
#pragma unroll
                for (int r = 0; r < 16; r++)
                    buffer_atomic_add_f32s(rdq, vo, (unsigned)((qbd + 8 * (r >> 2) + (r & 3)) * ld) * 4u,
                                           acc[r]);
            }
        }
        __syncthreads();
        if (ALIAS && qt + 1 < nqt) {
            put();
            __syncthreads();
        }
    }

    // the query splits' partial dK, dV through LDS: a wave takes 1 / NQB of its
    // key block's columns
    float* rec = reinterpret_cast<float*>(lds);
#pragma unroll
    for (int i = 0; i < NO; i++) {
        settle(dk[i]);
        settle(dv[i]);
    }
#pragma unroll
    for (int i = 0; i < NO; i++)
#pragma unroll
        for (int q = 0; q < 4; q++) {
            float* at = rec + wave * REC + (4 * i + q) * 256 + lane * 4;
            *reinterpret_cast<f4*>(at) = f4{dk[i][4 * q], dk[i][4 * q + 1], dk[i][4 * q + 2], dk[i][4 * q + 3]};
            *reinterpret_cast<f4*>(at + 4 * NO * 256) =
                f4{dv[i][4 * q], dv[i][4 * q + 1], dv[i][4 * q + 2], dv[i][4 * q + 3]};
        }
    __syncthreads();
    const int key = k0 + 32 * kb + l32;
    if (key >= S)
        return;
#pragma unroll
    for (int j = 0; j < 8 * NO / NQB; j++) {
        const int grp = qs * (8 * NO / NQB) + j, c = 8 * (grp % (4 * NO)) + 4 * g;
        f4 v = f4zero();
#pragma unroll
        for (int k = 0; k < NQB; k++)
            v += *reinterpret_cast<const f4*>(rec + (kb + k * NKB) * REC + grp * 256 + lane * 4);
        if (c < Dh)
            *reinterpret_cast<f4*>((grp < 4 * NO ? dK : dV) + base + (long)key * ld + c) = v;
    }
}

template <int NK, int NKB, int NQB, bool ALIAS>
static hipError_t bwd_go(const float* Q, const float* K, const float* V, const float* dO,
                         const float* lse, const float* Di, float* dQ, float* dK, float* dV, int B,
                         int S, int H, int Dh, hipStream_t st)
{
    constexpr int BN = 32 * NKB;
    const int BH = B * H, nkb = (S + BN - 1) / BN;
    ProfScope ps(st, "mha_bwd");
    CXG_LAUNCH((mhabf_bwd_kernel<NK, NKB, NQB, ALIAS>), dim3((unsigned)((long)nkb * BH)),
               dim3(64 * NKB * NQB), 0, st, Q, K, V, dO, lse, Di, dQ, dK, dV, S, H, Dh, BH,
               1.0f / sqrtf((float)Dh));
    return hipGetLastError();
}

// Which backward (times as above, the pre-pass included):
//   heads past 64 columns: all ([4, 333, 10, 80] 56.3 / 111.6 us, [32, 64, 16,
//     96] 50.6 / 58.5);
//   33 to 64 columns, at most one 64-key tile a compute unit and 128 rows or
//     more, or at most two and 384 rows: one workgroup of four waves a unit,
//     with room to split the next query tile beside the products of this one
//     ([2, 512, 8, 64] 45.0 / 50.8, [4, 333, 10, 40] 35.9 / 41.5, [8, 512, 8,
//     64] 60.9 / 64.0; [3, 90, 12, 64] 18.0 / 17.8, [5, 300, 16, 64] 39.7 /
//     38.9);
//   more tiles and 256 rows or more: two workgroups a unit, dS taking dO's
//     place in LDS ([2, 4096, 12, 64] 816 / 1040, [16, 384, 12, 64] 99.7 /
//     118.2; [32, 128, 16, 64] 56.1 / 52.9);
//   narrower heads: none ([4, 1000, 12, 32] 96.2 / 94.4).
static int bwd_kind(int B, int S, int H, int Dh)
{
    const long tiles = (long)B * H * ((S + 63) / 64), cus = mha_device_cus();
    if (Dh > 64)
        return BF_SHARED;
    if (Dh <= 32)
        return BF_NONE;
    if (tiles <= 2 * cus)
        return S >= (tiles <= cus ? 128 : 384) ? BF_SHARED : BF_NONE;
    return S >= 256 ? BF_LONG : BF_NONE;
}

bool mhabf_bwd_use(int B, int S, int H, int Dh, const float* Q, const float* K, const float* V,
                   const float* dO, const float* dK, const float* dV)
{
    return mhabf_ok(S, H, Dh, Q, K, V, dO) && al16(dK) && al16(dV) &&
           bwd_kind(B, S, H, Dh) != BF_NONE;
}

hipError_t mhabf_bwd_launch(const float* Q, const float* K, const float* V, const float* dO,
                            const float* lse, const float* Di, float* dQ, float* dK, float* dV,
                            int B, int S, int H, int Dh, hipStream_t st)
{
    if (Dh > 64)
        return bwd_go<6, 2, 2, false>(Q, K, V, dO, lse, Di, dQ, dK, dV, B, S, H, Dh, st);
    if (bwd_kind(B, S, H, Dh) == BF_LONG)
        return bwd_go<4, 2, 2, true>(Q, K, V, dO, lse, Di, dQ, dK, dV, B, S, H, Dh, st);
    return bwd_go<4, 2, 2, false>(Q, K, V, dO, lse, Di, dQ, dK, dV, B, S, H, Dh, st);
}

}  // namespace cxg
