// pk_chain4.h - exact weight GEMMs on the four-deep fp32 matrix instruction.
//
// v_mfma_f32_16x16x4_f32 adds four products per output, one after another in
// ascending k, each as a correctly rounded fused multiply-add: bit for bit the
// chain c = fma(a[k], w[k], c) that the K = 1 forms of pk_gemm_tiles.h take
// four instructions for (subnormals, infinities and signed zeros included).
// Measured on MI355X, a dependent instruction takes 14.9 ns, 3.7 ns per k step,
// where the 4x4x1 form takes 6.3 and the 32x32x1 form 27.8, and one wave alone
// on a SIMD reaches 141 of the 157 TFLOP/s peak.  So a chain needs neither
// wide tiles nor many waves to run at rate, and the unit of work is 16 x 16
// outputs: small enough to share a GEMM of a few hundred rows out evenly.
//
// A workgroup owns BM x BN = 16 R NWM x 16 C NWN outputs.  NWM x NWN waves
// multiply R x C units each, NP producer waves stage the operands.  fp32 MFMA
// and VALU instructions share a SIMD and do not overlap (a VALU instruction
// between two of a wave's MFMAs costs about 5 ns, the next ones 1.5-2.3), so
// the multiplying waves hold none: every LDS address is a register plus an
// instruction offset, operands are read 16 k at a time, and the conversions
// run in the producers.  What bounds the GEMMs after that: the producers'
// VALU time (int4: 24 instructions per 8 weights), the last round of
// workgroups, and the start and end of a launch.  Against the K = 1 tiles
// (time in us on one MI355X, hot weights):
//   int4   375 x 4096 x 1024   38.3 -> 30.9     375 x 1024 x 4096   51.1 -> 35.0
//   int4  1656 x 4096 x 1024  163.4 -> 124.0   1656 x 1024 x 4096  144.5 -> 132.2
//   int8  1656 x 3072 x 1024  109.2 -> 89.9     375 x 3072 x 1024   35.2 -> 28.4
//   fp32   500 x 4096 x 1024   43.6 -> 34.9     500 x 1024 x 4096   53.8 -> 35.4
//   fp32  1656 x 2048 x 1024   75.3 -> 61.6    int4 16 x 1024 x 4096 41.1 -> 17.2
// A GEMM that fills the chip (2048 x 4096 x 4096, fp32) runs at 145 TFLOP/s.
#pragma once

#include "pk_gemm_tiles.h"

namespace pkgpu {
namespace chain4 {

using tiles::KArgs;
using tiles::v4f;
using tiles::v4u;

// Lane l = j + 16 g supplies A[row j][k + g] and B[k + g][column j]; the result
// holds rows 4 g + v (v = 0..3) of column j.
__device__ __forceinline__ v4f step(float a, float b, v4f c)
{
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

// Weights are staged in units of 8 consecutive columns of one k row.
template <int WK> struct Unit8;

template <> struct Unit8<W_F32> {
    static constexpr int BYTES = 32;
    struct Raw { v4u w[2]; };
    __device__ static Raw load(__amdgpu_buffer_rsrc_t rb, __amdgpu_buffer_rsrc_t, uint32_t off, uint32_t)
    {
        return Raw{{tiles::ld_v4(rb, off), tiles::ld_v4(rb, off + 16)}};
    }
    __device__ static void dequant(const KArgs&, const Raw& r, float (&w)[8])
    {
#pragma unroll
        for (int e = 0; e < 8; ++e) w[e] = __uint_as_float(r.w[e >> 2][e & 3]);
    }
};

template <> struct Unit8<W_I8> {
    static constexpr int BYTES = 8;
    typedef uint32_t v2u __attribute__((ext_vector_type(2)));
    struct Raw { v2u w; };
    __device__ static Raw load(__amdgpu_buffer_rsrc_t rb, __amdgpu_buffer_rsrc_t, uint32_t off, uint32_t)
    {
        return Raw{__builtin_amdgcn_raw_buffer_load_b64(rb, (int)off, 0, 0)};
    }
    __device__ static void dequant(const KArgs& p, const Raw& r, float (&w)[8])
    {
#pragma unroll
        for (int e = 0; e < 8; ++e) w[e] = __fmul_rn((float)(int8_t)(r.w[e >> 2] >> (8 * (e & 3))), p.scale);
    }
};

template <> struct Unit8<W_I4> {
    static constexpr int BYTES = 4;
    struct Raw { uint32_t w; float s; };
    __device__ static Raw load(__amdgpu_buffer_rsrc_t rb, __amdgpu_buffer_rsrc_t rs, uint32_t off, uint32_t soff)
    {
        return Raw{tiles::ld_u32(rb, off), tiles::ld_f32(rs, soff)};
    }
    __device__ static void dequant(const KArgs& p, const Raw& r, float (&w)[8])
    {
        tiles::WStage<W_I4>::dequant_unit(p, tiles::WStage<W_I4>::Unit{r.w, r.s}, w);
    }
};

// LDS position of step k of a chunk: each run of 16 k is kept as 4 groups of 4,
// group g holding k = g, 4 + g, 8 + g, 12 + g.  Lane group g's operands of four
// successive instructions are then one b128 read.
__host__ __device__ constexpr int kpos(int k) { return (k & ~15) + 4 * (k & 3) + ((k >> 2) & 3); }

template <int WK, int R, int C, int NWM, int NWN, int NP, int KT>
struct Tile {
    using US = Unit8<WK>;
    static constexpr int NT = 64 * NP;                // staging threads
    static constexpr int BM = 16 * R * NWM, BN = 16 * C * NWN;
    // Rows (of A, and columns of W) are S floats apart in LDS, and W has 4
    // more floats after every 8 columns.  Laid out for 32 banks of 4 bytes, b128
    // accesses of 8 lanes and b32 ones of 32 a cycle: the operand reads (8
    // rows, one group) and both kinds of stores (4 rows x 8 units of A; 8
    // units of W at 4 steps k, k + 4, ...) then each touch every bank once.
    // The counter still reads 0.33 conflict cycles for each cycle of LDS work,
    // in every tile and format, which is 0.16 to 0.37 of a launch's.
    static constexpr int S = KT + 4;
    static constexpr int A_LDS = BM * S, B_LDS = BN * S + BN / 2, BUF = A_LDS + B_LDS;
    static constexpr int NQ = BN / 8, NQL = NQ < 8 ? NQ : 8, K16 = KT / 16;
    static constexpr int A_TOTAL = BM * KT / 4, B_TOTAL = NQ * KT;
    static constexpr int A_ITEMS = (A_TOTAL + NT - 1) / NT, B_ITEMS = (B_TOTAL + NT - 1) / NT;
    static_assert(KT % 32 == 0 && A_TOTAL % 64 == 0 && B_TOTAL % 64 == 0, "wave-uniform staging");
    static_assert(NQ == 4 || NQ % 8 == 0, "column units");

    struct Raw {
        v4u a[A_ITEMS];
        typename US::Raw b[B_ITEMS];
    };

    uint32_t a_off[A_ITEMS], b_off[B_ITEMS], s_off[WK == W_I4 ? B_ITEMS : 1];
    uint32_t a_step, b_step, s_step;     // bytes per chunk (uniform)
    int last;                            // the last chunk

    // Unit e of A: 8 consecutive units lie along k (128 bytes of one row).
    __device__ static int a_row(int e) { return (e >> 3) % BM; }
    __device__ static int a_kq(int e) { return (e & 7) + 8 * ((e >> 3) / BM); }
    __device__ static int b_nq(int e) { return NQ < 8 ? e % NQ : (e & 7) + 8 * ((e >> 5) % (NQ / 8)); }
    __device__ static int b_k(int e)
    {
        const int r = NQ < 8 ? e / (4 * NQL) : (e >> 5) / (NQ / 8);     // which 16 k and k % 4
        return 16 * (r % K16) + 4 * ((e / NQL) & 3) + r / K16;
    }

    __device__ Tile(const KArgs& p, int tid, int m0, int n0)
    {
        constexpr int UB = US::BYTES;                                   // bytes of 8 columns
        const uint32_t row_bytes = (uint32_t)p.ldb * (WK == W_F32 ? 4u : 1u);
#pragma unroll
        for (int i = 0; i < A_ITEMS; ++i) {
            const int e = tid + i * NT;
            a_off[i] = ((uint32_t)(m0 + a_row(e)) * p.lda + 4 * a_kq(e)) * 4u;
        }
#pragma unroll
        for (int i = 0; i < B_ITEMS; ++i) {
            const int e = tid + i * NT, n = n0 + 8 * b_nq(e);
            b_off[i] = (uint32_t)b_k(e) * row_bytes + (uint32_t)(n / 8) * UB;
            if constexpr (WK == W_I4) s_off[i] = ((uint32_t)b_k(e) * p.n_groups + (n >> 5)) * 4u;
        }
        a_step = 4u * KT;
        b_step = row_bytes * KT;
        s_step = 4u * KT * p.n_groups;
        last = (p.K - 1) / KT;
    }
    // Chunk c's raw operands, or the last chunk's again when there is no c.  The
    // chunk's start goes into the descriptors (scalar work): their ranges end
    // where the operands do, so what lies past them reads 0.
    __device__ void load(Raw& r, const KArgs& p, int c, int tid) const
    {
        const uint32_t q = (uint32_t)min(c, last);
        const uint32_t sa = q * a_step, sb = q * b_step, ss = q * s_step;
        const auto rsA = tiles::make_rsrc(reinterpret_cast<const char*>(p.A) + sa, p.a_bytes - sa);
        const auto rsB = tiles::make_rsrc(static_cast<const char*>(p.B) + sb, p.b_bytes - sb);
        const auto rsS = WK == W_I4 ? tiles::make_rsrc(reinterpret_cast<const char*>(p.scales) + ss, p.s_bytes - ss)
                                    : rsB;
#pragma unroll
        for (int i = 0; i < A_ITEMS; ++i) {
            if (A_TOTAL % NT != 0 && tid + i * NT >= A_TOTAL) continue;
            r.a[i] = tiles::ld_v4(rsA, a_off[i]);
        }
#pragma unroll
        for (int i = 0; i < B_ITEMS; ++i) {
            if (B_TOTAL % NT != 0 && tid + i * NT >= B_TOTAL) continue;
            r.b[i] = US::load(rsB, rsS, b_off[i], s_off[WK == W_I4 ? i : 0]);
        }
    }
    __device__ void store(const Raw& r, const KArgs& p, int tid, float* lds) const
    {
#pragma unroll
        for (int i = 0; i < A_ITEMS; ++i) {
            const int e = tid + i * NT;
            if (A_TOTAL % NT != 0 && e >= A_TOTAL) continue;
            float* d = lds + a_row(e) * S + kpos(4 * a_kq(e));
#pragma unroll
            for (int j = 0; j < 4; ++j) d[4 * j] = __uint_as_float(r.a[i][j]);
        }
        float* Bs = lds + A_LDS;
#pragma unroll
        for (int i = 0; i < B_ITEMS; ++i) {
            const int e = tid + i * NT;
            if (B_TOTAL % NT != 0 && e >= B_TOTAL) continue;
            float w[8];
            US::dequant(p, r.b[i], w);
            float* d = Bs + b_nq(e) * (8 * S + 4) + kpos(b_k(e));
#pragma unroll
            for (int q = 0; q < 8; ++q) d[q * S] = w[q];
        }
    }
};

// The fused output step of NV consecutive columns of one row.
template <int NV>
__device__ __forceinline__ void store_row(const KArgs& p, const float (&v)[NV], int row, int col, bool vec)
{
    if (row >= p.M) return;
    if (vec && col + NV <= p.N) {
        typedef float vn __attribute__((ext_vector_type(NV)));
        float o[NV];
        float* c = p.C + (size_t)row * p.ldc + col;
        vn old, bs, res;
        const bool residual = p.epi == EPI_HALF_RESIDUAL || p.epi == EPI_RESIDUAL;
        if (residual) old = *reinterpret_cast<const vn*>(c);
        if (p.bias) bs = *reinterpret_cast<const vn*>(p.bias + col);
#pragma unroll
        for (int q = 0; q < NV; ++q) {
            float x = v[q];
            if (p.bias) x = __fadd_rn(x, bs[q]);
            if (p.epi == EPI_SWISH) x = swish_f(x);
            else if (p.epi == EPI_HALF_RESIDUAL) x = __fmaf_rn(x, 0.5f, old[q]);
            else if (p.epi == EPI_RESIDUAL) x = __fadd_rn(old[q], x);
            else if (p.epi == EPI_RELU) x = x > 0.0f ? x : 0.0f;
            o[q] = x;
        }
#pragma unroll
        for (int q = 0; q < NV; ++q) res[q] = o[q];
        *reinterpret_cast<vn*>(c) = res;
        return;
    }
#pragma unroll
    for (int q = 0; q < NV; ++q)
        if (col + q < p.N) tiles::store_c(p, v[q], row, col + q);
}

// W is the instruction's row operand and A its column operand (the products are
// the same), so that a lane ends with 4 consecutive columns of one row.
template <int WK, int R, int C, int NWM, int NWN, int NP, int KT>
__global__ __launch_bounds__(64 * (NWM * NWN + NP), 2) void gemm(KArgs p)
{
    using T = Tile<WK, R, C, NWM, NWN, NP, KT>;
    constexpr int NC = NWM * NWN;                     // multiplying waves
    constexpr int S = T::S, NB = KT / 16;
    constexpr int D = R * C <= 2 ? 3 : 1;             // blocks of 16 k that operands are read ahead
    constexpr int SETS = D + 1;
    static_assert(NB % SETS == 0, "operand sets");
    __shared__ __attribute__((aligned(16))) float lds[2][T::BUF];

    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int j = lane & 15, g = lane >> 4;
    const int wm = wave / NWN, wn = wave % NWN;
    int m0, n0;
    tiles::tile_origin(p, T::BM, T::BN, m0, n0);
    const int npair = p.K / (2 * KT);
    const int rem0 = 2 * npair * KT;                  // what is left of K: less than two chunks

    if (wave >= NC) {
        // Producer: converts chunk ch + 1 while chunk ch is multiplied.
        const int ptid = tid - 64 * NC;
        const T st(p, ptid, m0, n0);
        typename T::Raw raw;
        st.load(raw, p, 0, ptid);
        st.store(raw, p, ptid, lds[0]);
        st.load(raw, p, 1, ptid);
        __syncthreads();
        for (int c = 0; c < npair; ++c) {
            st.store(raw, p, ptid, lds[1]);
            st.load(raw, p, 2 * c + 2, ptid);
            __syncthreads();
            st.store(raw, p, ptid, lds[0]);
            st.load(raw, p, 2 * c + 3, ptid);
            __syncthreads();
        }
        if (rem0 + KT < p.K) {
            __syncthreads();
            st.store(raw, p, ptid, lds[0]);
            __syncthreads();
        }
        return;
    }

    const int wrow = 16 * R * wm, wcol = 16 * C * wn;
    // Output element (r, c, v) of this lane.
    auto row_of = [&](int r) { return m0 + wrow + 16 * r + j; };
    auto col_of = [&](int c) { return n0 + wcol + 16 * c + 4 * g; };

    v4f acc[R][C];
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
        for (int c = 0; c < C; ++c) acc[r][c] = v4f{0.f, 0.f, 0.f, 0.f};
    if (p.beta != 0.0f || p.chain_bias) {
#pragma unroll
        for (int r = 0; r < R; ++r)
#pragma unroll
            for (int c = 0; c < C; ++c)
#pragma unroll
                for (int v = 0; v < 4; ++v) acc[r][c][v] = tiles::beta_c(p, row_of(r), col_of(c) + v);
    }
    __syncthreads();

    const int a_off = (wrow + j) * S + 4 * g;
    const int b_off = T::A_LDS + (wcol + j) * S + 4 * ((wcol + j) >> 3) + 4 * g;
    constexpr int BC = 16 * S + 8;                    // 16 columns on
    v4f a[SETS][R], b[SETS][C];                       // the operands of 16 k
    auto fetch = [&](int set, int buf, int blk) {
#pragma unroll
        for (int r = 0; r < R; ++r) a[set][r] = *reinterpret_cast<const v4f*>(lds[buf] + a_off + 16 * blk + 16 * S * r);
#pragma unroll
        for (int c = 0; c < C; ++c) b[set][c] = *reinterpret_cast<const v4f*>(lds[buf] + b_off + 16 * blk + BC * c);
    };
    // A chunk lies in lds[buf] and its first D blocks of operands are in
    // registers.  The barrier after block NB - D - 1 says both that the next
    // chunk is staged and that this one has been read by all: the multiplies
    // on both sides of it wait for nothing.
    auto chunk = [&](auto J) {
        constexpr int buf = decltype(J)::value;
#pragma unroll
        for (int blk = 0; blk < NB; ++blk) {
            if (blk == NB - D) __syncthreads();
            fetch((blk + D) % SETS, blk + D < NB ? buf : buf ^ 1, (blk + D) % NB);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int u = 0; u < 4; ++u)
#pragma unroll
                for (int r = 0; r < R; ++r)
#pragma unroll
                    for (int c = 0; c < C; ++c)
                        acc[r][c] = step(b[blk % SETS][c][u], a[blk % SETS][r][u], acc[r][c]);
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    if (npair) {
#pragma unroll
        for (int q = 0; q < D; ++q) fetch(q, 0, q);
    }
    for (int c = 0; c < npair; ++c) {
        chunk(std::integral_constant<int, 0>{});
        chunk(std::integral_constant<int, 1>{});
    }
    // What is left of K: its first chunk is staged.
    for (int k0 = rem0; k0 < p.K; k0 += KT) {
        if (k0 != rem0) {
            __syncthreads();
            __syncthreads();
        }
        const int kn = min(KT, p.K - k0);
        const float* as = lds[0] + a_off;
        const float* bs = lds[0] + b_off;
        int k = 0;
        for (; k + 4 <= kn; k += 4) {
            const int kp = kpos(k);
#pragma unroll
            for (int r = 0; r < R; ++r)
#pragma unroll
                for (int c = 0; c < C; ++c) acc[r][c] = step(bs[kp + BC * c], as[kp + 16 * S * r], acc[r][c]);
        }
        // the last K % 4 steps: a product with zeros instead would turn -0 into +0
        for (; k < kn; ++k) {
            const float* a1 = lds[0] + (wrow + j) * S + kpos(k);
            const float* b1 = lds[0] + T::A_LDS + (wcol + 4 * g) * S + 4 * ((wcol + 4 * g) >> 3) + kpos(k);
#pragma unroll
            for (int r = 0; r < R; ++r)
#pragma unroll
                for (int c = 0; c < C; ++c)
#pragma unroll
                    for (int v = 0; v < 4; ++v)
                        acc[r][c][v] = __fmaf_rn(a1[16 * S * r], b1[BC * c + S * v], acc[r][c][v]);
        }
    }

    const bool vec = (p.ldc % 4 == 0) && ((reinterpret_cast<uintptr_t>(p.C) & 15) == 0) &&
                     ((reinterpret_cast<uintptr_t>(p.bias) & 15) == 0);
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
        for (int c = 0; c < C; ++c) {
            const float o[4] = {acc[r][c][0], acc[r][c][1], acc[r][c][2], acc[r][c][3]};
            store_row<4>(p, o, row_of(r), col_of(c), vec);
        }
}

// The tiles: R, C, NWM, NWN, NP, KT.  Deeper chunks and more blocks ahead where a
// wave holds one or two chains, whose 60 ns per 16 k are shorter than an LDS
// read under load.  48 x 32 puts its two producers on the two SIMDs that hold
// one multiplying wave.
#define PK_CHAIN4_TILES(X)                                                                       \
    X(0, 1, 1, 1, 2, 2, 128)  /*  16 x 32 */                                                     \
    X(1, 1, 1, 2, 2, 4, 64)   /*  32 x 32 */                                                     \
    X(2, 1, 1, 3, 2, 2, 64)   /*  48 x 32 */                                                     \
    X(3, 2, 1, 2, 2, 4, 64)   /*  64 x 32 */                                                     \
    X(4, 2, 2, 2, 2, 4, 32)   /*  64 x 64 */                                                     \
    X(5, 4, 2, 2, 2, 4, 32)   /* 128 x 64 */

struct Chain4Tile { int bm, bn, threads; };
#define PK_CHAIN4_ENTRY(i, r, c, wm, wn, np, kt) {16 * r * wm, 16 * c * wn, 64 * (wm * wn + np)},
static constexpr Chain4Tile kTiles[] = {PK_CHAIN4_TILES(PK_CHAIN4_ENTRY)};
#undef PK_CHAIN4_ENTRY
constexpr int kNumTiles = sizeof(kTiles) / sizeof(kTiles[0]);

template <int WK>
hipError_t launch(int tile, const KArgs& a, hipStream_t s)
{
    if (tile < 0 || tile >= kNumTiles) return hipErrorInvalidValue;
    const Chain4Tile& t = kTiles[tile];
    const dim3 grid((a.N + t.bn - 1) / t.bn, (a.M + t.bm - 1) / t.bm), block(t.threads);
#define PK_CHAIN4_CASE(i, r, c, wm, wn, np, kt)                                                  \
    case i: hipLaunchKernelGGL((gemm<WK, r, c, wm, wn, np, kt>), grid, block, 0, s, a); break;
    switch (tile) { PK_CHAIN4_TILES(PK_CHAIN4_CASE) }
#undef PK_CHAIN4_CASE
    return hipGetLastError();
}

// Launchers of one weight format each (defined in pk_chain4_{f32,i8,i4}.hip).
// Operands: 16-byte aligned A rows, weight rows as the vector form of the
// K = 1 tiles takes them (KArgs::vec_a, vec_b), alpha = 1.
hipError_t launch_f32(int tile, const KArgs& a, hipStream_t s);
hipError_t launch_i8(int tile, const KArgs& a, hipStream_t s);
hipError_t launch_i4(int tile, const KArgs& a, hipStream_t s);

}  // namespace chain4
}  // namespace pkgpu
