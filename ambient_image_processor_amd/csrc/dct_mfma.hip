// Separable DCT-II / DCT-III passes as dense per-axis matrix products on the
// gfx950 matrix cores.
//
// Reference: cuda_image_operations/cosine_transform.cu:142-223 and
// inverse_cosine_transform.cu:79-164 evaluate every output with an O(n) loop
// of FP64 cospi calls; here each axis pass is out = C * in along that axis,
// with C the n x n cosine matrix (host FP64, rounded once):
//   forward  C[k][m] = cos(pi (m + 1/2) k / n)
//   inverse  C[k][m] = w_m cos(pi (k + 1/2) m / n), w_0 = 1, w_m = 2 (the
//            reference's "X[0] + 2 sum_{m>=1}" folded into the matrix)
// The last pass (z, or y or x where the axes after it have one voxel and no pass)
// applies the reference's *8 (forward) or 1/(W*H*D*8) (inverse), and can fuse the
// Poisson eigenvalue divide of solve_poisson_in_cosine_domain.cu:42-53 into its epilogue.
//
// Precisions:
//   F32     v_mfma_f32_16x16x4_f32, FP32 operands, FP32 accumulate
//   BF16X3  v_mfma_f32_16x16x32_bf16 on hi/lo bf16 splits of both operands:
//           C_hi*X_hi + C_hi*X_lo + C_lo*X_hi, FP32 accumulate (the lo*lo
//           term is below the split's own rounding)
//
// Every pass is a product D[i][j] = sum_m X[i][m] Y[m][j]:
//   column pass (y, z): X = C[k][m] (table), Y = in[o][m][s], D = out[o][k][s]
//   row pass (x):       X = in[r][m],       Y[m][k] = C[k][m], D = out[r][k]
// Operand k-slots are assigned identically for X and Y, so the products do not
// depend on the hardware's k order within a slot group.
#include "amb_internal.hpp"

#include <algorithm>
#include <type_traits>

namespace amb {
namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

// Poisson eigenvalue divide of the coefficient v at (x, y, z), linear index idx
// (the same arithmetic as poisson_kernel in dct.hip,
// solve_poisson_in_cosine_domain.cu:42-53; with the index quirk the coordinates
// are recovered from the linear index through float arithmetic as the
// reference does).
__device__ __forceinline__ float poisson_apply(float v, int x, int y, int z, size_t idx,
                                               const Geometry& g, int quirk, const float* cx,
                                               const float* cy, const float* cz) {
    if (quirk) {
        const unsigned wh = unsigned(g.w) * unsigned(g.h);
        const unsigned i = unsigned(idx);
        const float zf = floorf(float(i / wh));
        int rest = int(float(int(i)) - zf * float(wh));
        const float yf = floorf(float(unsigned(rest) / unsigned(g.w)));
        rest = int(float(rest) - yf * float(unsigned(g.w)));
        x = rest; y = int(yf); z = int(zf);
    }
    if (x == 0 && y == 0 && z == 0) return 0.0f;
    const double den =
        g.d == 1 ? 4.0 - 2.0 * double(cx[x]) - 2.0 * double(cy[y])   // the 2-D kernel
                 : 6.0 - 2.0 * double(cx[x]) - 2.0 * double(cy[y]) - 2.0 * double(cz[z]);
    return float(double(v) / den);
}

// four floats at any 4-byte aligned address (global memory takes them unaligned)
typedef float f32x4u __attribute__((ext_vector_type(4), aligned(4)));

// ---------------------------------------------------------------------------
// F32 kernel: 128 x 128 output tiles, 4 waves of 64 x 64, 32-deep K chunks
// ---------------------------------------------------------------------------
constexpr int BM = 128, BN = 128, BK = 32;
constexpr int PF32 = BK + 4;          // LDS row pitch (floats), K contiguous
constexpr int GEMM_THREADS = 256;

struct GemmArgs {
    const float* data;      // FP32 volume (X in the row pass, Y in the column pass)
    const float* t32;       // FP32 table [k][m]
    float* out;
    int M, N, K;            // output rows, output columns, summed extent
    int O;                  // outer count (column pass: planes above the axis)
    int axis;
    float scale;
    int poisson, quirk;
    Geometry g;
    const float* cx;
    const float* cy;
    const float* cz;
};

__device__ __forceinline__ float poisson_at(float v, int i, int j, const GemmArgs& a) {
    // the last pass: z over (y, x) columns, or along y or x where z has one voxel
    const int hi = a.axis == 2 ? j / a.g.w : i;
    const int x = a.axis == 2 ? j - hi * a.g.w : j, z = a.axis == 2 ? i : 0;
    return poisson_apply(v, x, hi, z, size_t(i) * a.N + j, a.g, a.quirk, a.cx, a.cy, a.cz);
}

// LDS tiles X [BM][pitch], Y [BN][pitch].  The column pass keeps its data tile Y
// as loaded, [k][j] with a pitch of BN + 16 floats (the 16 lanes of a fragment
// read consecutive j; the four k rows of a read are 16 banks apart).
struct GemmLds {
    float x[BM][PF32];
    float y[BN][PF32];
};
constexpr int PYK = BN + 16;
static_assert(BK * PYK == BN * PF32, "column-pass Y tile reuses the Y array");

// Staging registers of a thread: 4 pieces of 4 values per operand.  The global
// loads of chunk c + 2 are issued before the MFMAs of chunk c.
struct Piece {
    float v[4][4];
};

// Operand with K contiguous in memory (the table; the data of the row pass):
// thread e loads rows r0 + e / 8 + 32 q, columns m0 + 4 (e % 8) .. + 4.
__device__ __forceinline__ void load_kc(Piece& R, const float* src, int rows, int r0, int m0, int K) {
    const int e = threadIdx.x, m = m0 + (e % 8) * 4;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const int rg = r0 + e / 8 + 32 * q;
        if (rg < rows && m + 3 < K) {
            const f32x4u t = *reinterpret_cast<const f32x4u*>(src + size_t(rg) * K + m);
#pragma unroll
            for (int c = 0; c < 4; ++c) R.v[q][c] = t[c];
        } else {
#pragma unroll
            for (int c = 0; c < 4; ++c)
                R.v[q][c] = (rg < rows && m + c < K) ? src[size_t(rg) * K + m + c] : 0.0f;
        }
    }
}

// Data operand of the column pass (N contiguous in memory): thread e loads rows
// m0 + 4 (e / 32) + q at columns j0 + 4 (e % 32) .. + 4.
__device__ __forceinline__ void load_nc(Piece& R, const float* src, int N, int K, int j0, int m0) {
    const int e = threadIdx.x, kq = (e / 32) * 4, j = j0 + (e % 32) * 4;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const int m = m0 + kq + q;
        if (m < K && j + 3 < N) {
            const f32x4u t = *reinterpret_cast<const f32x4u*>(src + size_t(m) * N + j);
#pragma unroll
            for (int c = 0; c < 4; ++c) R.v[q][c] = t[c];
        } else {
#pragma unroll
            for (int c = 0; c < 4; ++c)
                R.v[q][c] = (m < K && j + c < N) ? src[size_t(m) * N + j + c] : 0.0f;
        }
    }
}

__device__ __forceinline__ void put_kc(float (*tile)[PF32], const Piece& R) {
    const int e = threadIdx.x, c4 = (e % 8) * 4;
#pragma unroll
    for (int q = 0; q < 4; ++q)
        *reinterpret_cast<float4*>(&tile[e / 8 + 32 * q][c4]) =
            make_float4(R.v[q][0], R.v[q][1], R.v[q][2], R.v[q][3]);
}

__device__ __forceinline__ void put_nc(float* y, const Piece& R) {
    const int e = threadIdx.x, k4 = (e / 32) * 4, j = (e % 32) * 4;
#pragma unroll
    for (int q = 0; q < 4; ++q)
        *reinterpret_cast<float4*>(y + (k4 + q) * PYK + j) =
            make_float4(R.v[q][0], R.v[q][1], R.v[q][2], R.v[q][3]);
}

template <int ROW>
__global__ __launch_bounds__(GEMM_THREADS) void dct_gemm_kernel(GemmArgs a) {
    __shared__ __align__(16) GemmLds L;
    const int M = a.M, N = a.N, K = a.K;
    const int tm = (M + BM - 1) / BM, tn = (N + BN - 1) / BN;
    // tile order: the tiles sharing a data panel are adjacent, and each XCD
    // takes a contiguous range of tiles, so a panel is fetched from HBM once
    // into one XCD's L2 instead of once per XCD its tiles land on
    int bid = int(xcd_contiguous(blockIdx.x, gridDim.x));
    int it, jt, o;
    if (ROW) {                  // data panel = rows it; j tiles fastest
        jt = bid % tn; bid /= tn; it = bid % tm; o = bid / tm;
    } else {                    // data panel = columns jt; i tiles fastest
        it = bid % tm; bid /= tm; jt = bid % tn; o = bid / tn;
    }
    const int i0 = it * BM, j0 = jt * BN;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int li = lane & 15, lg = lane >> 4;
    const int wi = (wave >> 1) * 64, wj = (wave & 1) * 64;
    const size_t obase = size_t(o) * size_t(M) * size_t(N);

    f32x4 acc[4][4];
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int u = 0; u < 4; ++u) acc[t][u] = f32x4{0.f, 0.f, 0.f, 0.f};

    const float* dsrc = ROW ? a.data : a.data + size_t(o) * size_t(K) * size_t(N);
    Piece R0, R1, T0, T1;
    auto load = [&](Piece& R, Piece& T, int m0) {
        if (ROW) {
            load_kc(R, dsrc, M, i0, m0, K);
            load_kc(T, a.t32, N, j0, m0, K);
        } else {
            load_kc(T, a.t32, M, i0, m0, K);
            load_nc(R, dsrc, N, K, j0, m0);
        }
    };
    auto chunk = [&](Piece& R, Piece& T, int m0) {
        if (ROW) {
            put_kc(L.x, R);
            put_kc(L.y, T);
        } else {
            put_kc(L.x, T);
            put_nc(&L.y[0][0], R);
        }
        __syncthreads();
        if (m0 + 2 * BK < K) load(R, T, m0 + 2 * BK);
#pragma unroll
        for (int kk = 0; kk < BK / 4; ++kk) {
            const int kc = 4 * kk + lg;
            float xf[4], yf[4];
#pragma unroll
            for (int t = 0; t < 4; ++t) xf[t] = L.x[wi + t * 16 + li][kc];
#pragma unroll
            for (int u = 0; u < 4; ++u)
                yf[u] = ROW ? L.y[wj + u * 16 + li][kc] : (&L.y[0][0])[kc * PYK + wj + u * 16 + li];
#pragma unroll
            for (int t = 0; t < 4; ++t)
#pragma unroll
                for (int u = 0; u < 4; ++u)
                    acc[t][u] = __builtin_amdgcn_mfma_f32_16x16x4f32(xf[t], yf[u], acc[t][u], 0, 0, 0);
        }
        __syncthreads();
    };
    load(R0, T0, 0);
    if (BK < K) load(R1, T1, BK);
    for (int m0 = 0; m0 < K; m0 += 2 * BK) {
        chunk(R0, T0, m0);
        if (m0 + BK < K) chunk(R1, T1, m0 + BK);
    }
    // lane holds D rows 4*lg + r, column li of each 16 x 16 tile
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int u = 0; u < 4; ++u)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int i = i0 + wi + t * 16 + 4 * lg + r;
                const int j = j0 + wj + u * 16 + li;
                if (i < M && j < N) {
                    const size_t idx = obase + size_t(i) * N + j;
                    float v = acc[t][u][r] * a.scale;
                    if (a.poisson) v = poisson_at(v, i, j, a);
                    a.out[idx] = v;
                }
            }
}

// 4 floats -> packed bf16 hi and lo (2 x 64 bits): hi = rne(x), lo = rne(x - hi),
// two values per conversion instruction
__device__ __forceinline__ void split4(const float (&x)[4], uint2& hi, uint2& lo) {
    const uint32_t h01 = StoreBF16::rne2(x[0], x[1]), h23 = StoreBF16::rne2(x[2], x[3]);
    hi = make_uint2(h01, h23);
    lo = make_uint2(StoreBF16::rne2(x[0] - __uint_as_float(h01 << 16),
                                    x[1] - __uint_as_float(h01 & 0xffff0000u)),
                    StoreBF16::rne2(x[2] - __uint_as_float(h23 << 16),
                                    x[3] - __uint_as_float(h23 & 0xffff0000u)));
}

// ---------------------------------------------------------------------------
// BF16x3 panel kernel.
//
// An item is a panel of columns (lines of the axis) and a group of up to 16 output tiles of 16
// rows: axes of up to 256 values have one group, longer ones load and split each panel once
// per group (512: twice).  A block of 8 waves walks through its items, 64
// summed indices (a stage) at a time: the stage's data lie in LDS as bf16 hi/lo
// splits, two buffers, and each wave multiplies them with its two 16-row tiles
// of the table (x 16 CT columns).  The table's fragments come straight from L2 in
// fragment order (coalesced 1 KB loads, no LDS).  Everything the next stage
// needs - its table fragments and its data - is loaded into registers before the
// products of this one and split into the other buffer after them: one barrier
// per stage, and the loads' latency lies behind the products.  One block per CU
// (up to 256 registers), which goes on to its next panel without draining.
// Every output sums the same products in the same order as a 32-deep chunked
// product (per chunk X_hi Y_hi, X_hi Y_lo, X_lo Y_hi with X the table in the
// column passes and the data in the row pass).
//
// Measured at 512 x 512 x 256 (us per pass; 128 x 128 output tiles with 32-deep
// chunks staged through LDS before): x 298 -> 265, y 325 -> 258, z 190 -> 157,
// z with the eigenvalue divide 325 -> 237.  The matrix products alone need 104 us
// of an n = 512 pass at the 1.9 GHz the card runs them at, its bytes 110 us at
// the rate of a large copy; what is left is the part of the two, of the table's
// 1 GB from L2 and of the splits that does not overlap.  Two blocks of 64
// columns per CU (2 GB of table reads) took 235 - 280 us, 4-wave blocks with four
// tiles per wave 264 - 280 us.
// ---------------------------------------------------------------------------
constexpr int PANEL_THREADS = 512;
constexpr int PANEL_WAVES = PANEL_THREADS / 64, TT = 2;   // output tiles per wave
constexpr int PANEL_K = 64;           // summed indices per stage

struct PanelArgs {
    const float* in;
    float* out;
    const uint4* tab;     // table fragments [tile][chunk][hi, lo][64 lanes]
    int n;                // extent of the axis
    int axis;
    uint32_t N;           // column passes: columns per plane (the axis' stride)
    uint32_t quads;       // column passes: groups of four columns per plane
    uint32_t cols;        // columns (four per group) or rows in all
    uint32_t total;       // elements of the volume
    int chunks;           // 32-deep chunks of the axis
    int tiles, tg;        // 16-row output tiles in all and per group
    int groups;
    unsigned items;       // panels x groups
    float scale;
    int quirk;
    Geometry g;
    const float* cx;
    const float* cy;
    const float* cz;
};

// Bank swizzle of a panel row's eight 16-byte blocks: the 16 columns of a
// fragment read cover all 64 banks, and the transposing writes (columns four
// apart) spread over all blocks.
__device__ __forceinline__ int panel_swz(int col) { return ((col >> 1) ^ (col >> 4)) & 7; }

__device__ __forceinline__ void split8(const float (&x)[8], uint4& hi, uint4& lo) {
    const float a[4] = {x[0], x[1], x[2], x[3]}, b[4] = {x[4], x[5], x[6], x[7]};
    uint2 ha, la, hb, lb;
    split4(a, ha, la);
    split4(b, hb, lb);
    hi = make_uint4(ha.x, ha.y, hb.x, hb.y);
    lo = make_uint4(la.x, la.y, lb.x, lb.y);
}

// Column group of the column passes: planes are cut into groups of four columns
// (the last one of a plane may reach past it; those columns are never stored).
struct Quad {
    uint32_t o, s;   // plane, first column in it
    size_t base;     // its element 0
    __device__ __forceinline__ Quad(const PanelArgs& a, uint32_t q) {
        o = a.axis == 2 ? 0u : q / a.quads;
        s = (q - o * a.quads) * 4;
        base = size_t(o) * a.N * uint32_t(a.n) + s;
    }
};

// v / den as the FP64 division gives it (one Newton step on the FP32 reciprocal
// and one residual correction: the last bit of the FP64 quotient may differ),
// rounded to float; den is an eigenvalue, a normal float's range.
__device__ __forceinline__ float divide_eigenvalue(float v, double den) {
    double r = double(__builtin_amdgcn_rcpf(float(den)));
    r = fma(fma(-den, r, 1.0), r, r);
    double q = double(v) * r;
    q = fma(fma(-den, q, double(v)), r, q);
    return float(q);
}

// The Poisson eigenvalue divide of coefficient v at (x, y, z), linear index idx
__device__ __forceinline__ float panel_poisson(const PanelArgs& a, float v, int x, int y, int z,
                                               size_t idx) {
    if (a.quirk) return poisson_apply(v, x, y, z, idx, a.g, 1, a.cx, a.cy, a.cz);
    if ((x | y | z) == 0) return 0.0f;
    double den = (a.g.d == 1 ? 4.0 : 6.0) - 2.0 * double(a.cx[x]) - 2.0 * double(a.cy[y]);
    if (a.g.d > 1) den -= 2.0 * double(a.cz[z]);
    return divide_eigenvalue(v, den);
}

template <int ROW, int WI, int CT, int POI>
__global__ __launch_bounds__(PANEL_THREADS, 2) void dct_panel_bf16x3(PanelArgs a) {
    constexpr int NCOLS = 16 * CT * (PANEL_WAVES / WI);   // columns per panel
    constexpr int KB = PANEL_K / 8;                   // 16-byte blocks per panel row
    constexpr int LO = NCOLS * KB;                    // the lo half's first block
    constexpr int BUF = 2 * LO;                       // blocks per buffer
    constexpr int UH = CT < 4 ? CT : 4;               // column tiles multiplied at a time
    extern __shared__ __align__(16) uint4 panel[];    // [2][hi, lo][NCOLS][KB]
    const int tid = int(threadIdx.x), lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int li = lane & 15, lg = lane >> 4;
    const int wi = wave % WI, wc = (wave / WI) * 16 * CT;          // row tile, first column
    const int stages = (a.n + PANEL_K - 1) / PANEL_K;
    const unsigned first = xcd_contiguous(blockIdx.x, gridDim.x);  // a panel's groups adjacent
    const unsigned items = a.items;

    // data of one stage: the row pass loads units of 8 k of a row, the column passes
    // units of 4 columns x 4 k
    constexpr int NU = ROW ? (NCOLS * KB + PANEL_THREADS - 1) / PANEL_THREADS : 1;
    constexpr int UF = ROW ? 8 : 16;
    constexpr bool ALL = ROW ? NCOLS * KB % PANEL_THREADS == 0 : NCOLS == 128;
    float v[NU][UF];
    // column passes: 16 quads x 4 k-groups per wave
    const int cq = (tid & 15) + (NCOLS == 128 ? ((tid >> 6) & 1) * 16 : 0);
    const int kq = ((tid >> 4) & 3) + 4 * (NCOLS == 128 ? tid >> 7 : tid >> 6);
    const bool stager = ALL || (ROW ? tid < NCOLS * KB : kq < 16 && cq < NCOLS / 4);
    auto load_data = [&](unsigned item, int k0) {
        if (!stager) return;
        const uint32_t c0 = (item / unsigned(a.groups)) * uint32_t(NCOLS);
        if (ROW) {
#pragma unroll
            for (int q = 0; q < NU; ++q) {
                const int u = tid + q * PANEL_THREADS, k = k0 + (u % KB) * 8;
                const uint32_t r = min(c0 + uint32_t(u / KB), a.cols - 1);
                const float* src = a.in + size_t(r) * uint32_t(a.n) + k;
                if (k + 7 < a.n) {
                    const f32x4u x = *reinterpret_cast<const f32x4u*>(src);
                    const f32x4u y = *reinterpret_cast<const f32x4u*>(src + 4);
#pragma unroll
                    for (int e = 0; e < 4; ++e) { v[q][e] = x[e]; v[q][4 + e] = y[e]; }
                } else {
#pragma unroll
                    for (int e = 0; e < 8; ++e) v[q][e] = k + e < a.n ? src[e] : 0.0f;
                }
            }
        } else {
            const int k = k0 + kq * 4;
            const size_t i0 = Quad(a, min(c0 / 4 + uint32_t(cq), a.cols / 4 - 1)).base + size_t(k) * a.N;
            if (i0 + size_t(3) * a.N + 3 < a.total) {
                const float* src = a.in + i0;
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const f32x4u x = *reinterpret_cast<const f32x4u*>(src + size_t(q) * a.N);
#pragma unroll
                    for (int e = 0; e < 4; ++e) v[0][4 * q + e] = x[e];
                }
            } else {   // at the volume's end
#pragma unroll
                for (int q = 0; q < 4; ++q)
#pragma unroll
                    for (int e = 0; e < 4; ++e)
                        v[0][4 * q + e] = a.in[min(i0 + size_t(q) * a.N + e, size_t(a.total) - 1)];
            }
        }
    };
    auto store_data = [&](int buf, int k0) {
        if (!stager) return;
        uint4* const dst = panel + buf * BUF;
        if (ROW) {
#pragma unroll
            for (int q = 0; q < NU; ++q) {
                const int u = tid + q * PANEL_THREADS, col = u / KB;
                uint4 h, l;
                split8(*reinterpret_cast<const float(*)[8]>(&v[q][0]), h, l);
                const int i = col * KB + ((u % KB) ^ panel_swz(col));
                dst[i] = h;
                dst[LO + i] = l;
            }
        } else {
            const int k = k0 + kq * 4;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                float x[4];
#pragma unroll
                for (int q = 0; q < 4; ++q) x[q] = k + q < a.n ? v[0][4 * q + e] : 0.0f;
                uint2 h, l;
                split4(x, h, l);
                const int col = cq * 4 + e, i = col * KB + ((kq >> 1) ^ panel_swz(col));
                reinterpret_cast<uint2*>(dst + i)[kq & 1] = h;
                reinterpret_cast<uint2*>(dst + LO + i)[kq & 1] = l;
            }
        }
    };
    // this wave's table fragments of one stage: two chunks x two tiles, hi and lo
    auto tile_of = [&](unsigned item, int t) {
        return min(int(item % unsigned(a.groups)) * a.tg + wi + t * WI, a.tiles - 1);
    };
    uint4 th[2][TT], tl[2][TT];   // [chunk][tile]
    auto load_table = [&](unsigned item, int k0, int c) {
#pragma unroll
        for (int t = 0; t < TT; ++t) {
            const uint4* p = a.tab + (size_t(tile_of(item, t)) * a.chunks +
                                      min(k0 / 32 + c, a.chunks - 1)) * 128 + lane;
            th[c][t] = p[0];
            tl[c][t] = p[64];
        }
    };

    f32x4 acc[TT][CT];
    if (first < items) {
        load_data(first, 0);
        load_table(first, 0, 0);
        load_table(first, 0, 1);
        store_data(0, 0);
        __syncthreads();
    }
    int buf = 0;
    for (unsigned item = first; item < items; item += gridDim.x) {
        const int t0 = int(item % unsigned(a.groups)) * a.tg + wi;
        const int tend = min(int(item % unsigned(a.groups)) * a.tg + a.tg, a.tiles);
        const int nt = (tend - t0 + WI - 1) / WI;   // this wave's tiles, at most TT
#pragma unroll
        for (int t = 0; t < TT; ++t)
#pragma unroll
            for (int u = 0; u < CT; ++u) acc[t][u] = f32x4{0.f, 0.f, 0.f, 0.f};
        for (int st = 0; st < stages; ++st) {
            // the next stage: of this panel, or the first one of the next
            const bool last = st + 1 == stages;
            const unsigned nitem = last ? item + gridDim.x : item;
            const int nk = last ? 0 : (st + 1) * PANEL_K;
            const bool more = nitem < items;
            if (more) load_data(nitem, nk);
            __builtin_amdgcn_sched_barrier(0);   // the loads stay ahead of the products
            const uint4* const src = panel + buf * BUF;
            auto multiply = [&](auto NTC, auto CC) {
                constexpr int NT = decltype(NTC)::value, c = decltype(CC)::value;
                {
#pragma unroll
                    for (int u0 = 0; u0 < CT; u0 += UH) {
                        bf16x8 xh[UH], xl[UH];
#pragma unroll
                        for (int u = 0; u < UH; ++u) {
                            const int col = wc + (u0 + u) * 16 + li;
                            const int i = col * KB + ((c * 4 + lg) ^ panel_swz(col));
                            xh[u] = __builtin_bit_cast(bf16x8, src[i]);
                            xl[u] = __builtin_bit_cast(bf16x8, src[LO + i]);
                        }
                        // column passes: rows of D are columns of the volume (four
                        // consecutive ones per lane), row pass: outputs k
                        auto mma = [&](const uint4 (&tf)[TT], const bf16x8 (&xf)[UH]) {
#pragma unroll
                            for (int t = 0; t < NT; ++t)
#pragma unroll
                                for (int u = 0; u < UH; ++u) {
                                    const bf16x8 tb = __builtin_bit_cast(bf16x8, tf[t]);
                                    f32x4& d = acc[t][u0 + u];
                                    d = ROW ? __builtin_amdgcn_mfma_f32_16x16x32_bf16(tb, xf[u], d, 0, 0, 0)
                                            : __builtin_amdgcn_mfma_f32_16x16x32_bf16(xf[u], tb, d, 0, 0, 0);
                                }
                        };
                        mma(th[c], xh);
                        if (ROW) { mma(tl[c], xh); mma(th[c], xl); }
                        else { mma(th[c], xl); mma(tl[c], xh); }
                    }
                }
            };
            auto chunk = [&](auto CC) {
                constexpr int c = decltype(CC)::value;
                if (st * 2 + c < a.chunks) {
                    if (nt == 2) multiply(std::integral_constant<int, 2>{}, CC);
                    else if (nt > 0) multiply(std::integral_constant<int, 1>{}, CC);
                }
                __builtin_amdgcn_sched_barrier(0);
                if (more) load_table(nitem, nk, c);
                __builtin_amdgcn_sched_barrier(0);
            };
            chunk(std::integral_constant<int, 0>{});
            chunk(std::integral_constant<int, 1>{});
            if (last) break;
            store_data(buf ^ 1, nk);   // read last one stage ago
            buf ^= 1;
            __syncthreads();
        }
        const uint32_t c0 = (item / unsigned(a.groups)) * uint32_t(NCOLS);
#pragma unroll
        for (int u = 0; u < CT; ++u) {
            if (ROW) {   // lane: row r, outputs k .. k + 3
                const uint32_t r = c0 + uint32_t(wc + u * 16 + li);
                if (r >= a.cols) continue;
#pragma unroll
                for (int t = 0; t < TT; ++t) {
                    const int k = (t0 + t * WI) * 16 + 4 * lg;
                    if (t >= nt || k >= a.n) continue;
                    const size_t b = size_t(r) * uint32_t(a.n) + uint32_t(k);
                    f32x4u o;
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        o[e] = acc[t][u][e] * a.scale;
                        if (POI) {
                            const int x = min(k + e, a.n - 1);
                            o[e] = panel_poisson(a, o[e], x, int(r % uint32_t(a.g.h)),
                                                 int(r / uint32_t(a.g.h)), b + uint32_t(x - k));
                        }
                    }
                    if (k + 3 < a.n) {
                        *reinterpret_cast<f32x4u*>(a.out + b) = o;
                    } else {
                        a.out[b] = o[0];
                        if (k + 1 < a.n) a.out[b + 1] = o[1];
                        if (k + 2 < a.n) a.out[b + 2] = o[2];
                    }
                }
            } else {     // lane: output k, columns c .. c + 3
                const uint32_t c = c0 + uint32_t(wc + u * 16 + 4 * lg);
                if (c >= a.cols) continue;
                const Quad co(a, c / 4);
                // POI: along z, or along y where the volume has one plane; the
                // eigenvalues' part from x and (along z) y, once per column
                double dxy[4];
                int xs[4], ys[4];
                if (POI) {
                    int x = int(co.s), y = 0;
                    if (a.axis == 2) { y = x / a.g.w; x -= y * a.g.w; }
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        if (co.s + e >= a.N) { x = 0; y = 0; }   // never stored
                        xs[e] = x;
                        ys[e] = y;
                        dxy[e] = (a.g.d == 1 ? 4.0 : 6.0) - 2.0 * double(a.cx[x]);
                        if (a.axis == 2) dxy[e] -= 2.0 * double(a.cy[y]);
                        if (++x == a.g.w) { x = 0; ++y; }
                    }
                }
#pragma unroll
                for (int t = 0; t < TT; ++t) {
                    const int k = (t0 + t * WI) * 16 + li;
                    if (t >= nt || k >= a.n) continue;
                    const size_t row = size_t(k) * a.N;
                    const double dk = POI ? 2.0 * double(a.axis == 2 ? (a.g.d > 1 ? a.cz[k] : 0.0f) : a.cy[k]) : 0.0;
                    f32x4u o;
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        o[e] = acc[t][u][e] * a.scale;
                        if (POI) {
                            if (a.quirk)
                                o[e] = poisson_apply(o[e], xs[e], a.axis == 2 ? ys[e] : k,
                                                     a.axis == 2 ? k : 0, row + co.s + e, a.g, 1,
                                                     a.cx, a.cy, a.cz);
                            else
                                o[e] = (xs[e] | ys[e] | k) == 0
                                           ? 0.0f : divide_eigenvalue(o[e], dxy[e] - dk);
                        }
                    }
                    float* dst = a.out + co.base + row;
                    if (co.s + 3 < a.N) {
                        *reinterpret_cast<f32x4u*>(dst) = o;
                    } else {
                        dst[0] = o[0];
                        if (co.s + 1 < a.N) dst[1] = o[1];
                        if (co.s + 2 < a.N) dst[2] = o[2];
                    }
                }
            }
        }
        if (item + gridDim.x < items) {   // the next panel's first stage
            store_data(buf ^ 1, 0);
            buf ^= 1;
            __syncthreads();
        }
    }
}

// One BF16x3 pass.  WI waves share a panel's columns: as few as give every output
// tile of a group a wave's slot.  128 columns per panel, or fewer while that
// leaves CUs without one.
template <int ROW, int WI, int CT, int POI>
hipError_t panel_launch(hipStream_t s, PanelArgs a, int cus) {
    constexpr int NCOLS = 16 * CT * (PANEL_WAVES / WI);
    const size_t items = (size_t(a.cols) + NCOLS - 1) / NCOLS * size_t(a.groups);
    if constexpr (CT > 1 && (WI < 8 || CT > 2)) {
        if (items < size_t(cus)) return panel_launch<ROW, WI, CT / 2, POI>(s, a, cus);
    }
    if (items > 0x7fffffffu) return hipErrorInvalidValue;
    a.items = unsigned(items);
    const size_t lds = size_t(NCOLS) * PANEL_K * 4 * 2;
    auto kern = dct_panel_bf16x3<ROW, WI, CT, POI>;
    const hipError_t e = ensure_dynamic_lds(reinterpret_cast<const void*>(kern), lds);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(kern, dim3(unsigned(std::min(items, size_t(cus)))), dim3(PANEL_THREADS), lds,
                       s, a);
    return hipGetLastError();
}

template <int ROW, int POI>
hipError_t panel_pass(hipStream_t s, PanelArgs a) {
    int dev = 0, cus = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return e;
    e = hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev);
    if (e != hipSuccess) return e;
    a.chunks = (a.n + 31) / 32;
    a.tiles = (a.n + 15) / 16;
    a.groups = (a.tiles + 15) / 16;
    a.tg = (a.tiles + a.groups - 1) / a.groups;
    return a.tg > 8   ? panel_launch<ROW, 8, 8, POI>(s, a, cus)
           : a.tg > 4 ? panel_launch<ROW, 4, 4, POI>(s, a, cus)
           : a.tg > 2 ? panel_launch<ROW, 2, 2, POI>(s, a, cus)
                      : panel_launch<ROW, 1, 1, POI>(s, a, cus);
}

}  // namespace

int dct_mfma_max_extent() { return 4096; }

hipError_t launch_dct_mfma_pass(hipStream_t s, const float* in, float* out, const void* table,
                                Geometry g, int axis, float scale, int precision,
                                const float* eig_x, const float* eig_y, const float* eig_z,
                                int fuse_poisson, int quirk) {
    if (precision == 2) {
        PanelArgs p{};
        p.in = in; p.out = out; p.tab = static_cast<const uint4*>(table);
        p.axis = axis;
        p.n = axis == 0 ? g.w : axis == 1 ? g.h : g.d;
        p.N = axis == 0 ? 1u : axis == 1 ? uint32_t(g.w) : uint32_t(g.w) * uint32_t(g.h);
        p.total = uint32_t(g.n());
        p.quads = (p.N + 3) / 4;
        p.cols = axis == 0 ? p.total / uint32_t(p.n)
                           : p.total / (p.N * uint32_t(p.n)) * p.quads * 4;
        p.scale = scale;
        p.quirk = quirk;
        p.g = g; p.cx = eig_x; p.cy = eig_y; p.cz = eig_z;
        if (axis == 0) return fuse_poisson ? panel_pass<1, 1>(s, p) : panel_pass<1, 0>(s, p);
        return fuse_poisson ? panel_pass<0, 1>(s, p) : panel_pass<0, 0>(s, p);
    }
    GemmArgs a;
    a.data = in; a.out = out; a.t32 = static_cast<const float*>(table);
    a.g = g; a.cx = eig_x; a.cy = eig_y; a.cz = eig_z;
    a.quirk = quirk;
    a.poisson = fuse_poisson;
    if (axis == 0) {           // rows r of length W
        a.M = g.h * g.d; a.N = g.w; a.K = g.w; a.O = 1;
    } else if (axis == 1) {    // per plane: out[z][k][x] = sum_m C[k][m] in[z][m][x]
        a.M = g.h; a.N = g.w; a.K = g.h; a.O = g.d;
    } else {                   // out[k][s] = sum_m C[k][m] in[m][s], s over the plane
        a.M = g.d; a.N = g.w * g.h; a.K = g.d; a.O = 1;
    }
    a.axis = axis;
    a.scale = scale;
    const long tm = (a.M + BM - 1) / BM, tn = (a.N + BN - 1) / BN;
    const long blocks = tm * tn * a.O;
    if (blocks > 0x7fffffffL) return hipErrorInvalidValue;
    const dim3 grid{static_cast<unsigned>(blocks), 1, 1};
    if (axis == 0) hipLaunchKernelGGL(dct_gemm_kernel<1>, grid, dim3(GEMM_THREADS), 0, s, a);
    else hipLaunchKernelGGL(dct_gemm_kernel<0>, grid, dim3(GEMM_THREADS), 0, s, a);
    return hipGetLastError();
}

}  // namespace amb
